// Plans random passes of one-qubit matrices and sign gates with the
// library's layerPass and planPass and applies the planned programs -- op by
// op, with a restatement of LAYER, DENSE1, SIGNS, PHASES, GROUP and DIAG1 over
// whole states -- against the gates in queue order.  The matrices are unitaries
// of every kind and others, the ones that a layer leaves out among them.
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "qa_tile.hpp"

using namespace qa::fuse;
typedef std::complex<double> cx;

static cx at(const double* f, int i) { return cx(f[2 * i], f[2 * i + 1]); }
static void dense1(std::vector<cx>& v, int q, const double* m) {
    for (size_t i = 0; i < v.size(); i++) {
        if ((i >> q) & 1) continue;
        const cx a = v[i], b = v[i | (1ull << q)];
        v[i] = at(m, 0) * a + at(m, 1) * b;
        v[i | (1ull << q)] = at(m, 2) * a + at(m, 3) * b;
    }
}

// One matrix, planned with a frame on a state of its own: the program must
// apply the matrix that was given, to a few ulp of FP64, whether or not it is
// exactly unitary.
static bool oneMatrix(const cx (&m)[4], const char* what) {
    const int n = 4;
    GOp g;
    g.kind = F_DENSE1;
    g.t1 = 2;
    for (int k = 0; k < 4; k++) g.f[2 * k] = m[k].real(), g.f[2 * k + 1] = m[k].imag();
    LayerFrame frame;
    frame.finish = true;
    TileArgs a;
    std::vector<TOp> prog;
    planPass(&g, 1, n, (1ull << n) - 1, 0, a, prog, true, &frame);
    // each column of the product of the program's ops on the one qubit
    double worst = 0;
    for (int col = 0; col < 2; col++) {
        cx v[2] = {col == 0 ? 1.0 : 0.0, col == 1 ? 1.0 : 0.0};
        int reg = -1;  // the qubit's register bit
        for (const TOp& t : prog) {
            const double* b = reinterpret_cast<const double*>(t.b);
            if (t.h.kind == F_GROUP) {
                for (int r = 0; r < RB; r++)
                    if (a.localPos[reinterpret_cast<const int*>(t.b)[r]] == g.t1) reg = r;
            } else if (t.h.kind == F_DENSE1) {
                const cx x = v[0], y = v[1];
                v[0] = at(b, 0) * x + at(b, 1) * y;
                v[1] = at(b, 2) * x + at(b, 3) * y;
            } else if (t.h.kind == F_DIAG1) {
                v[1] *= at(b, 1);
                if (!t.h.pad) v[0] *= at(b, 0);
            } else if (t.h.kind == F_LAYER) {
                const LayerBody<double>& body = *reinterpret_cast<const LayerBody<double>*>(t.b);
                for (int r = 0; r < 2; r++) {
                    const int w = r << reg;
                    v[r] *= cx(body.factor[2 * w], body.factor[2 * w + 1]);
                }
                const cx x = v[0], y = v[1];
                v[0] = x - body.t[reg] * y;
                v[1] = body.t[reg] * x + y;
            } else {
                std::printf("FAIL: %s: op kind %d\n", what, t.h.kind);
                return false;
            }
        }
        for (int r = 0; r < 2; r++) {
            const double off = std::abs(v[r] - m[2 * r + col]);
            worst = std::isnan(off) ? INFINITY : std::max(worst, off);
        }
    }
    if (worst <= 8 * 2.3e-16) return true;
    std::printf("FAIL: %s: an element is off by %.3e\n", what, worst);
    return false;
}

static bool layersOnly(const std::vector<GOp>& ops) {
    for (const GOp& g : ops)
        if (!(g.kind == F_DENSE1 && !g.cMask) && !(g.kind == F_DIAG1 && g.f[2] == -1.0)) return false;
    return true;
}

// queues of rotations go as layers, those with many matrices that do not split
// (here X) or with other gates do not
static bool choices() {
    for (int prec : {QA_FP64, QA_FP32})
        for (int x : {0, 1, 2, 10, 32}) {
            std::vector<GOp> ops;
            for (int i = 0; i < 32; i++) {
                GOp g;
                g.kind = F_DENSE1;
                g.t1 = i % 5;
                const double th = i < x ? M_PI : 0.1 * i;
                const double m[8] = {std::cos(th / 2), 0, 0, -std::sin(th / 2), 0, -std::sin(th / 2), std::cos(th / 2), 0};
                std::memcpy(g.f, m, sizeof m);
                ops.push_back(g);
                GOp cz;
                cz.kind = F_DIAG1;
                cz.t1 = i % 5;
                cz.cMask = cz.cVal = (1ull << cz.t1) | (1ull << ((i + 1) % 5));
                cz.f[0] = 1;
                cz.f[2] = -1;
                ops.push_back(cz);
            }
            if (layerable(ops.data(), ops.size(), prec) != (x <= 2))
                return std::printf("FAIL: layers chosen wrongly for %d of 32 matrices\n", x), false;
            ops[40].cMask = 1ull << 7;
            ops[40].cVal = 1ull << 7;
            if (layerable(ops.data(), ops.size(), prec))
                return std::printf("FAIL: layers chosen for a controlled matrix\n"), false;
        }
    return true;
}

static bool matrices() {
    const double h = std::sqrt(0.5), nan = std::nan("");
    const cx e = std::polar(1.0, 2.45), f = std::polar(1.0, -0.7);
    for (double th : {5e-324, 2e-323, 1e-322, 1e-320, 1e-318, 1e-300, 1e-160, 0.3}) {
        const double c = std::cos(th), s = std::sin(th);
        // a rotation, then a phase
        const cx m[4] = {c, -s, e * s, e * c};
        if (!oneMatrix(m, "small angle")) return false;
    }
    for (double d : {4e-14, 1e-14, 3e-15}) {
        const cx b[4] = {0.6 * f, -0.8 * (1 + d), 0.8 * f * e, 0.6 * e}, a[4] = {h, h, h, -h * (1 - d)};
        if (!oneMatrix(b, "nearly unitary") || !oneMatrix(a, "nearly unitary")) return false;
    }
    for (int k = 0; k < 4; k++) {
        cx m[4] = {h, h, h, -h};
        m[k] = cx(nan, 0);
        LayerFrame frame;
        frame.finish = true;
        GOp g;
        g.kind = F_DENSE1;
        g.t1 = 2;
        for (int i = 0; i < 4; i++) g.f[2 * i] = m[i].real(), g.f[2 * i + 1] = m[i].imag();
        TileArgs a;
        std::vector<TOp> prog;
        planPass(&g, 1, 4, 15, 0, a, prog, true, &frame);
        // a matrix that is no unitary goes as it is
        bool kept = false;
        for (const TOp& t : prog)
            if (t.h.kind == F_DENSE1) kept = std::isnan(reinterpret_cast<const double*>(t.b)[2 * k]);
        if (!kept) return std::printf("FAIL: a NaN element of a matrix is lost\n"), false;
    }
    return true;
}

int main(int argc, char** argv) {
    if (!matrices() || !choices()) return 1;
    const int rounds = argc > 1 ? std::atoi(argv[1]) : 200;
    std::mt19937_64 rng(argc > 2 ? std::strtoull(argv[2], nullptr, 0) : 1);
    auto below = [&](int n) { return (int)(rng() % (uint64_t)n); };
    auto uniform = [&] { return 2.0 * (double)(rng() >> 11) / 9007199254740992.0 - 1; };
    long signOps = 0, layerOps = 0;
    for (int round = 0; round < rounds; round++) {
        const int n = 4 + below(6), kMax = 4 + below(n - 3), low = below(std::min(kMax, 3) + 1);
        LayerFrame frame;
        std::vector<GOp> ops;
        const int num = 1 + below(60);
        for (int i = 0; i < num; i++) {
            GOp g;
            if (below(3)) {
                g.kind = F_DENSE1;
                g.t1 = below(n);
                for (int k = 0; k < 8; k++) g.f[k] = uniform();
                if (below(8)) {
                    // e^{ia} [[c, -s e^{il}], [s e^{ip}, c e^{i(l+p)}]]: any angle, or a (nearly) diagonal or
                    // antidiagonal one
                    const double special[] = {0, 1e-12, 1e-7, M_PI / 2, M_PI / 2 - 1e-5, M_PI, 0.78539816339744828,
                                              5e-324, 2e-323, 1e-322, 1e-320, 1e-318, 1e-300, 1e-160, 1e-140};
                    const double th = below(3) ? M_PI * uniform() : special[below(15)];
                    const double a = M_PI * uniform(), l = below(4) ? M_PI * uniform() : 0, p = below(4) ? M_PI * uniform() : 0;
                    const cx m[4] = {std::polar(1.0, a) * std::cos(th), -std::polar(1.0, a + l) * std::sin(th),
                                     std::polar(1.0, a + p) * std::sin(th), std::polar(1.0, a + l + p) * std::cos(th)};
                    for (int k = 0; k < 4; k++) g.f[2 * k] = m[k].real(), g.f[2 * k + 1] = m[k].imag();
                }
            } else {
                // a sign gate: any controls, in any states, its target among them
                g.kind = F_DIAG1;
                g.t1 = below(n);
                for (int c = below(4); c > 0; c--) {
                    const int q = below(n);
                    g.cMask |= 1ull << q;
                    if (below(4)) g.cVal |= 1ull << q;
                }
                g.cMask |= 1ull << g.t1;
                g.cVal = (g.cVal & g.cMask) | (1ull << g.t1);
                g.f[0] = 1;
                g.f[2] = -1;
            }
            ops.push_back(g);
        }
        std::vector<cx> want(1ull << n), got;
        for (cx& x : want) x = cx(uniform(), uniform());
        got = want;
        for (const GOp& g : ops) {
            if (g.kind == F_DENSE1) dense1(want, g.t1, g.f);
            else
                for (size_t i = 0; i < want.size(); i++)
                    if ((i & g.cMask) == g.cVal) want[i] = -want[i];
        }
        std::vector<uint32_t> picked;
        std::vector<GOp> pass, rest, layers;
        while (!ops.empty()) {
            uint64_t L = 0;
            picked.clear();
            pickPass(ops.data(), ops.size(), n, kMax, low, L, picked);
            if (picked.empty()) return std::printf("FAIL: nothing picked\n"), 1;
            pass.clear();
            rest.clear();
            size_t p = 0;
            for (size_t i = 0; i < ops.size(); i++)
                if (p < picked.size() && picked[p] == i) pass.push_back(ops[i]), p++;
                else rest.push_back(ops[i]);
            if (!layersOnly(pass)) return std::printf("FAIL: not layerable\n"), 1;
            layers.clear();
            layerPass(pass.data(), pass.size(), (1ull << low) - 1, layers);
            if (layers.size() != pass.size()) return std::printf("FAIL: %zu of %zu ops\n", layers.size(), pass.size()), 1;
            TileArgs a;
            std::vector<TOp> prog;
            frame.finish = rest.empty();
            planPass(layers.data(), layers.size(), n, L, low, a, prog, true, &frame);
            int slots[RB] = {0, 0, 0, 0};
            for (const TOp& t : prog) {
                auto qubit = [&](int b) { return a.localPos[slots[b]]; };
                const double* b = reinterpret_cast<const double*>(t.b);
                switch (t.h.kind) {
                    case F_GROUP: std::memcpy(slots, t.b, sizeof(slots)); break;
                    case F_DENSE1: dense1(got, qubit(t.h.rb1), b); break;
                    case F_SIGNS: case F_LAYER: case F_PHASES: case F_DIAG1: {
                        const LayerBody<double>& body = *reinterpret_cast<const LayerBody<double>*>(t.b);
                        const bool layer = t.h.kind == F_LAYER;
                        const SignTerm* st = layer ? body.terms : reinterpret_cast<const SignTerm*>(t.b);
                        const int numSigns = layer ? (int)t.h.rm1 : t.h.kind == F_SIGNS ? t.h.rb1 : 0;
                        for (uint64_t i = 0; i < got.size(); i++) {
                            const uint64_t base = i & a.nonLocalMask;
                            uint32_t v = 0, j = 0;
                            for (int s = 0; s < a.k; s++) j |= (uint32_t)((i >> a.localPos[s]) & 1) << s;
                            for (int r = 0; r < RB; r++) {
                                v |= ((j >> slots[r]) & 1u) << r;
                                j &= ~(1u << slots[r]);
                            }
                            bool flip = false;
                            for (int k = 0; k < numSigns; k++) {
                                if (k < t.h.rb2 && st[k].jm) return std::printf("FAIL: term order\n"), 1;
                                if ((base & st[k].gm) == st[k].gv && (j & st[k].jm) == st[k].jv)
                                    flip ^= (st[k].regs >> v) & 1;
                            }
                            if (flip) got[i] = -got[i];
                            if (layer) got[i] *= cx(body.factor[2 * v], body.factor[2 * v + 1]);
                            if (t.h.kind == F_PHASES) {
                                const PhaseTerm* pt = reinterpret_cast<const PhaseTerm*>(t.b);
                                for (int k = 0; k < t.h.rb1; k++)
                                    if ((v & pt[k].rm) == pt[k].rv && (j & pt[k].jm) == pt[k].jv &&
                                        (base & pt[k].gm) == pt[k].gv)
                                        got[i] *= cx(pt[k].fre, pt[k].fim);
                            }
                            if (t.h.kind == F_DIAG1) {
                                const bool one = t.h.rb1 >= 0 ? (v >> t.h.rb1) & 1 : ((j & t.b[4]) | (base & t.b[5])) != 0;
                                if ((v & t.h.rcMask) == t.h.rcVal && (j & t.h.jcMask) == t.h.jcVal &&
                                    (base & t.h.gcMask) == t.h.gcVal && !(t.h.pad && !one))
                                    got[i] *= at(b, one ? 1 : 0);
                            }
                        }
                        if (layer) {
                            const double* rot = body.t;
                            for (int r = 0; r < RB; r++) {
                                if (!((t.h.rb1 >> r) & 1)) continue;
                                const double m[8] = {1, 0, -rot[r], 0, rot[r], 0, 1, 0};
                                dense1(got, qubit(r), m);
                            }
                            layerOps++;
                        }
                        signOps += numSigns != 0;
                        break;
                    }
                    default: return std::printf("FAIL: op kind %d\n", t.h.kind), 1;
                }
            }
            ops.swap(rest);
        }
        double err = 0, norm = 0;
        for (size_t i = 0; i < want.size(); i++) err += std::norm(got[i] - want[i]), norm += std::norm(want[i]);
        if (!(std::sqrt(err / norm) <= 1e-12)) {
            std::printf("FAIL: round %d n %d tile %d low %d: error %.3e\n", round, n, kMax, low, std::sqrt(err / norm));
            return 1;
        }
    }
    std::printf("ok: %d queues, %ld sign ops, %ld layer ops\n", rounds, signOps, layerOps);
    return signOps && layerOps ? 0 : 1;
}
