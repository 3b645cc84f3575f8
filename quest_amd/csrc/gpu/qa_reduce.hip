// FP64 reductions (probabilities, purity, Pauli expectations, inner
// products, fidelities) replacing the Thrust transform_reduce calls of
// quest/src/gpu/gpu_thrust.cuh:745-1005 and gpu_subroutines.cpp:1440-1723.
//
// Deterministic for a given problem size:
//  1. a fixed-size grid (at most RED_BLOCKS workgroups) sweeps the terms in a
//     grid-stride loop, 4 independent loads in flight per lane; each lane
//     keeps a compensated (Neumaier) FP64 sum, waves combine lanes with
//     cross-lane shuffles and a two-sum merge, workgroups combine their 4
//     waves through LDS and write one (sum, compensation) pair;
//  2. one workgroup merges the partials in a fixed order.  A reduction that
//     one workgroup holds writes its value straight away.
// The value goes straight to a slot of pinned host memory, with a flag behind
// it that the caller's thread watches: at small sizes a reduction is all round
// trip, and a copy and a stream synchronisation cost more than the sums (10
// qubits: 18 us with both, see land()).
// Amplitudes are widened to FP64 before squaring, so FP32 states reduce in
// FP64 too.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <vector>

#include "qa_common.hpp"
#include "qa_fused.hpp"
#include "qa_sum.hpp"

namespace qa {
namespace {

constexpr int RED_BLOCKS = 1024;

// ---- results on the host ------------------------------------------------------
//
// Slots of pinned, coherent host memory, taken in turn: a kernel writes a
// slot's values, then its ticket.  A slot comes round again after LAND_SLOTS
// reductions, each of which its caller has waited for.
constexpr int LAND_SLOTS = 256;
constexpr int LAND_VALUES = 20;
struct LandSlot {
    double v[LAND_VALUES];
    uint64_t ticket;
    uint64_t pad[11];
};
LandSlot* g_land = nullptr;
std::atomic<uint64_t> g_ticket{0};

struct Ticket {
    LandSlot* slot;
    uint64_t number;
};
Ticket takeTicket() {
    const uint64_t t = g_ticket.fetch_add(1, std::memory_order_relaxed) + 1;
    return Ticket{g_land + t % LAND_SLOTS, t};
}

// the device side: n values by one thread
__device__ __forceinline__ void landValues(const Ticket& t, const double* v, int n) {
    for (int i = 0; i < n; i++) t.slot->v[i] = v[i];
    __hip_atomic_store(&t.slot->ticket, t.number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The host side: waits for the ticket's values.  Watching the slot answers a
// few microseconds sooner than the stream's synchronisation, which remains
// for long reductions (the watch ends after 100 us) and reports a failed
// launch.
int land(const Ticket& t, double* out, int n) {
    uint64_t* const seen = &t.slot->ticket;
    if (__atomic_load_n(seen, __ATOMIC_ACQUIRE) != t.number) {
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(100);
        bool here = false;
        while (!here && std::chrono::steady_clock::now() < until)
            for (int i = 0; i < 64 && !here; i++) here = __atomic_load_n(seen, __ATOMIC_ACQUIRE) == t.number;
        if (!here) {
            QA_HIP(hipStreamSynchronize(stream()));
            if (__atomic_load_n(seen, __ATOMIC_ACQUIRE) != t.number) {
                setError("reduction ended without a result");
                return QA_ERR_HIP;
            }
        }
    }
    for (int i = 0; i < n; i++) out[i] = t.slot->v[i];
    return QA_OK;
}

// workgroups for numWork terms
int reduceBlocks(uint64_t numWork) {
    const uint64_t want = (numWork + (uint64_t)BLOCK * 4 - 1) / ((uint64_t)BLOCK * 4);
    return (int)(want < 1 ? 1 : (want > RED_BLOCKS ? RED_BLOCKS : want));
}

// the compensated sums of NV values over numWork terms by `blocks`
// workgroups; `single`: the only workgroup lands them, else they go to
// partials[(block * NV + value) * 2]
template <int NV, typename F>
__device__ __forceinline__ void reduceTerms(const F& f, uint64_t numWork, unsigned block, unsigned blocks,
                                            double* __restrict__ partials, bool single, const Ticket& ticket) {
    KB acc[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] = KB{0, 0};
    const uint64_t stride = (uint64_t)blocks * BLOCK;
    uint64_t n = (uint64_t)block * BLOCK + threadIdx.x;
    for (; n + 3 * stride < numWork; n += 4 * stride) {
        double t[4][NV];
#pragma unroll
        for (int u = 0; u < 4; u++) f(n + (uint64_t)u * stride, t[u]);
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int v = 0; v < NV; v++) kadd(acc[v], t[u][v]);
    }
    for (; n < numWork; n += stride) {
        double t[NV];
        f(n, t);
#pragma unroll
        for (int v = 0; v < NV; v++) kadd(acc[v], t[v]);
    }
    blockMerge<NV>(acc);
    if (threadIdx.x != 0) return;
    if (single) {
        double out[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) out[v] = acc[v].s + acc[v].c;
        landValues(ticket, out, NV);
        return;
    }
#pragma unroll
    for (int v = 0; v < NV; v++) {
        partials[(block * NV + v) * 2] = acc[v].s;
        partials[(block * NV + v) * 2 + 1] = acc[v].c;
    }
}

template <int NV, typename F>
__global__ void __launch_bounds__(BLOCK) k_reduce(F f, uint64_t numWork, double* __restrict__ partials,
                                                 Ticket ticket) {
    reduceTerms<NV>(f, numWork, blockIdx.x, gridDim.x, partials, gridDim.x == 1, ticket);
}

// merges numParts partials of nv <= LAND_VALUES values (a wave per value, in
// a fixed order) and lands them; pairs: a value as (s, c), all s first
__device__ __forceinline__ void mergePartials(const double* __restrict__ partials, int numParts, int nv,
                                              const Ticket& ticket, bool pairs = false) {
    __shared__ double out[LAND_VALUES];
    const int lane = threadIdx.x & 63;
    for (int v = threadIdx.x >> 6; v < nv; v += BLOCK / 64) {
        KB acc = {0, 0};
        for (int p = lane; p < numParts; p += 64)
            kmerge(acc, KB{partials[(p * nv + v) * 2], partials[(p * nv + v) * 2 + 1]});
        waveMerge(acc);
        if (lane == 0) {
            out[v] = pairs ? acc.s : acc.s + acc.c;
            if (pairs) out[nv + v] = acc.c;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) landValues(ticket, out, pairs ? 2 * nv : nv);
}

__global__ void __launch_bounds__(BLOCK) k_finalize(const double* __restrict__ partials, int numParts, int nv,
                                                   Ticket ticket) {
    mergePartials(partials, numParts, nv, ticket);
}

template <int NV, typename F>
int runReduce(F f, uint64_t numWork, double* out) {
    static_assert(NV <= LAND_VALUES, "values of one reduction");
    double* scratch = devScratch((size_t)RED_BLOCKS * NV * 2);
    if (!scratch || !g_land) {
        setError("reduction scratch unavailable");
        return QA_ERR_OOM;
    }
    const int blocks = reduceBlocks(numWork);
    const Ticket ticket = takeTicket();
    k_reduce<NV, F><<<blocks, BLOCK, 0, stream()>>>(f, numWork, scratch, ticket);
    QA_LAUNCH_CHECK();
    if (blocks > 1) {
        k_finalize<<<1, BLOCK, 0, stream()>>>(scratch, blocks, NV, ticket);
        QA_LAUNCH_CHECK();
    }
    return land(ticket, out, NV);
}

template <typename T>
__device__ __forceinline__ cd ldd(const T* __restrict__ a, uint64_t i) {
    ct<T> v = ld(a, i);
    return cd{(double)v.re, (double)v.im};
}
__device__ __forceinline__ double norm2(cd a) { return a.re * a.re + a.im * a.im; }

// ---- term functors --------------------------------------------------------

// both outcome probabilities of PQ qubits q0..q0+PQ-1 in one read of the
// state: |a_n|^2 goes to o[b] when qubit q0 + b is 0 in n, to o[PQ + b]
// when it is 1, so each outcome is the compensated sum of its own terms
// (never a difference of two sums, which would lose a small probability).
// Ten qubits a read: states of 33 to 40 qubits are read 4 times, states of
// fewer than 10 once.
constexpr int PQ = 10;
static_assert(2 * PQ <= LAND_VALUES, "a read's values land in one slot");
template <typename T>
struct FProbsOfQubits {
    const T* a;
    int q0;
    __device__ void operator()(uint64_t n, double* o) const {
        const double p = norm2(ldd(a, n));
#pragma unroll
        for (int b = 0; b < PQ; b++) {
            const bool one = (n >> (q0 + b)) & 1ull;
            o[b] = one ? 0.0 : p;
            o[PQ + b] = one ? p : 0.0;
        }
    }
};

// Both outcome probabilities of every qubit of a statevector of 10..PQALL
// qubits in one read.  A wave reads 1024-amplitude chunks, lane l the
// amplitudes chunk*1024 + 64 i + l (i < 16), so in each amplitude's index
// bits 0-5 are the lane's, bits 6-9 are i's and the higher bits the
// chunk's.  Each lane keeps: its total (bits 0-5 are constant for the lane;
// the workgroup merge splits the totals by lane bit), the zero- and
// one-sums of bits 6-9 (sums of 8 of its 16 terms per chunk), and for each
// higher bit the zero- and one-sums of its chunk totals.  Every outcome is
// a sum of its own terms, never a difference.  The merges are compensated;
// a lane's chunk totals for the high bits are plain FP64 sums (at most a
// few hundred per lane).
// Below about 24 qubits the merges are what it costs, so a wave merges 16
// values at a time by halving: in each of 4 steps a lane hands half of its
// values to the lane across and merges the other half, 17 merges instead of
// the 96 of a butterfly per value, and one workgroup merges all partials
// (19 qubits complex64: 7.8 + 4.3 us, 80 us with a butterfly and a
// launch for every 8 values).
constexpr int PQALL = 32;
// NHI: the qubits above the tenth that the kernel provides for; value 2q + o
// is qubit q's outcome o
template <typename T, int NHI>
__global__ void __launch_bounds__(BLOCK) k_probsOfEveryQubit(const T* __restrict__ a, uint64_t numChunks,
                                                             double* __restrict__ partials) {
    constexpr int NVAL = 20 + 2 * NHI;
    static_assert(NVAL % 16 == 0, "values merge 16 at a time");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t waves = (uint64_t)gridDim.x * (BLOCK / 64);
    KB tot = {0, 0};
    KB mid[8];
#pragma unroll
    for (int j = 0; j < 8; j++) mid[j] = KB{0, 0};
    double hi[2 * NHI];
#pragma unroll
    for (int j = 0; j < 2 * NHI; j++) hi[j] = 0;
    for (uint64_t c = (uint64_t)blockIdx.x * (BLOCK / 64) + wave; c < numChunks; c += waves) {
        const uint64_t base = (c << 10) | (uint64_t)lane;
        double p[16];
#pragma unroll
        for (int i = 0; i < 16; i++) p[i] = norm2(ldd(a, base + 64 * i));
        double g = 0;
#pragma unroll
        for (int i = 0; i < 16; i++) g += p[i];
        kadd(tot, g);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            double z = 0, o = 0;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                if ((i >> b) & 1) o += p[i];
                else z += p[i];
            }
            kadd(mid[2 * b], z);
            kadd(mid[2 * b + 1], o);
        }
#pragma unroll
        for (int b = 0; b < NHI; b++) {
            const bool one = (c >> b) & 1ull;
            hi[2 * b] += one ? 0.0 : g;
            hi[2 * b + 1] += one ? g : 0.0;
        }
    }
    __shared__ KB sh[BLOCK / 64][NVAL];
#pragma unroll
    for (int batch = 0; batch < NVAL; batch += 16) {
        KB t[16];
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int val = batch + v, q = val >> 1, o = val & 1;
            if (q < 6) t[v] = (((lane >> q) & 1) == o) ? tot : KB{0, 0};
            else if (q < 10) t[v] = mid[2 * (q - 6) + o];
            else t[v] = KB{hi[2 * (q - 10) + o], 0};
        }
        // step with lane bit s: the lane keeps the values whose bit s is its own
#pragma unroll
        for (int s = 3; s >= 0; s--) {
            const bool up = (lane >> s) & 1;
#pragma unroll
            for (int v = 0; v < (1 << s); v++) {
                const KB lo = t[v], hiV = t[v + (1 << s)];
                KB give = {up ? lo.s : hiV.s, up ? lo.c : hiV.c};
                KB keep = {up ? hiV.s : lo.s, up ? hiV.c : lo.c};
                give.s = __shfl_xor(give.s, 1 << s, 64);
                give.c = __shfl_xor(give.c, 1 << s, 64);
                kmerge(keep, give);
                t[v] = keep;
            }
        }
#pragma unroll
        for (int s = 16; s <= 32; s <<= 1) {
            KB o;
            o.s = __shfl_xor(t[0].s, s, 64);
            o.c = __shfl_xor(t[0].c, s, 64);
            kmerge(t[0], o);
        }
        if (lane < 16) sh[wave][batch + lane] = t[0];
    }
    __syncthreads();
    if (threadIdx.x < NVAL) {
        KB acc = sh[0][threadIdx.x];
        for (int w = 1; w < BLOCK / 64; w++) kmerge(acc, sh[w][threadIdx.x]);
        partials[((size_t)blockIdx.x * NVAL + threadIdx.x) * 2] = acc.s;
        partials[((size_t)blockIdx.x * NVAL + threadIdx.x) * 2 + 1] = acc.c;
    }
}

// Merges the workgroups' partials into out[0..nval): thread (v, w) of a
// 1024-thread workgroup takes value v of every 1024/nval-th workgroup (each
// read covers a workgroup's whole row), then one thread per value merges
// those in order.
__global__ void __launch_bounds__(1024) k_finalizeProbs(const double* __restrict__ partials, int blocks, int nval,
                                                       double* __restrict__ out) {
    __shared__ KB sh[1024];
    const int v = threadIdx.x % nval, rows = 1024 / nval;
    KB acc = {0, 0};
    // (1024 is no multiple of 48: the last threads have no row)
    for (int b = threadIdx.x / nval; b < blocks && (int)threadIdx.x < rows * nval; b += rows) {
        const double* p = partials + ((size_t)b * nval + v) * 2;
        kmerge(acc, KB{p[0], p[1]});
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    if ((int)threadIdx.x < nval) {
        for (int w = 1; w < rows; w++) kmerge(acc, sh[w * nval + threadIdx.x]);
        out[threadIdx.x] = acc.s + acc.c;
    }
}

template <typename T>
struct FNormAll {  // |a_n|^2
    const T* a;
    __device__ void operator()(uint64_t n, double* o) const { o[0] = norm2(ldd(a, n)); }
};
template <typename T>
struct FNormOutcome {  // |a_i|^2, i = n with outcome bits inserted
    const T* a;
    InsertSpec ins;
    __device__ void operator()(uint64_t n, double* o) const { o[0] = norm2(ldd(a, insertBits(n, ins))); }
};
template <typename T>
struct FDiagReal {  // Re rho_rr, r = n with outcome bits inserted
    const T* a;
    InsertSpec ins;
    uint64_t diagStride;  // 2^N + 1
    __device__ void operator()(uint64_t n, double* o) const {
        o[0] = ldd(a, insertBits(n, ins) * diagStride).re;
    }
};
template <typename T>
struct FExpecZ {
    const T* a;
    uint64_t mask;
    __device__ void operator()(uint64_t n, double* o) const {
        double v = norm2(ldd(a, n));
        o[0] = parity64(n & mask) ? -v : v;
    }
};
template <typename T>
struct FDensExpecZ {
    const T* a;
    uint64_t mask, diagStride;
    __device__ void operator()(uint64_t n, double* o) const {
        cd v = ldd(a, n * diagStride);
        double s = parity64(n & mask) ? -1.0 : 1.0;
        o[0] = s * v.re;
        o[1] = s * v.im;
    }
};
// One Pauli string or several that share their X/Y mask, in one read of the
// state.  An amplitude pair (n, j = n ^ maskXY), n with the top X/Y bit
// clear, contributes sign(j) conj(a_n) a_j + sign(n) conj(a_j) a_n, whose
// second product is the first's conjugate: with an even number of Y the
// signs agree and the pair gives 2 sign Re(conj(a_n) a_j), with an odd number
// they differ and it gives 2i sign Im(conj(a_n) a_j), so one value per string
// is summed (the doubling and the factors of i are left to the caller).
// Without X or Y a term is sign |a_n|^2.  A string's sum is bitwise the same
// alone or in a group read by itself.
constexpr int GROUP_STRINGS = 8;
constexpr int GROUP_VALUES = GROUP_STRINGS + 2;  // of one partial, at most
struct PauliGroup {
    uint64_t maskXY, topLow;  // topLow: the bits below the top X/Y bit
    uint64_t maskYZ[GROUP_STRINGS];
    uint64_t odd;             // bit t: maskXY and string t's maskYZ share an odd number of bits
    uint64_t numWork;
    int blocks, numStrings;
    int nv;                   // values of one partial: numStrings, or more
    int pairs;                // a shared read: values land as (s, c), all s first
    Ticket ticket;
};
template <typename T, int NT>
struct FPauliGroup {
    const T* a;
    PauliGroup g;
    __device__ __forceinline__ void operator()(uint64_t w, double* o) const {
        double re, im;
        uint64_t n = w;
        if (g.maskXY) {
            n = ((w & ~g.topLow) << 1) | (w & g.topLow);
            const cd x = ldd(a, n), y = ldd(a, n ^ g.maskXY);
            re = fmaT(x.re, y.re, x.im * y.im);
            im = fmaT(x.re, y.im, -(x.im * y.re));
        } else {
            const cd x = ldd(a, n);
            re = fmaT(x.re, x.re, x.im * x.im);
            im = 0;
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const bool odd = (g.odd >> t) & 1ull;
            const double c = odd ? im : re;
            o[t] = (parity64(n & g.maskYZ[t]) != 0) != odd ? -c : c;
        }
    }
};

constexpr int MAX_GROUPS = 24;  // in one launch: their descriptions fit a kernel's arguments
struct PauliGroups {
    PauliGroup g[MAX_GROUPS];
};
template <typename T, int NT>
__global__ void __launch_bounds__(BLOCK) k_pauliGroups(const T* __restrict__ a, PauliGroups gs,
                                                      double* __restrict__ partials) {
    const PauliGroup& g = gs.g[blockIdx.y];
    if ((int)blockIdx.x >= g.blocks) return;
    FPauliGroup<T, NT> f;
    f.a = a;
    f.g = g;
    reduceTerms<NT>(f, g.numWork, blockIdx.x, (unsigned)g.blocks,
                    partials + (size_t)blockIdx.y * RED_BLOCKS * GROUP_VALUES * 2, g.blocks == 1, g.ticket);
}
__global__ void __launch_bounds__(BLOCK) k_finalizeGroups(PauliGroups gs, const double* __restrict__ partials) {
    const PauliGroup& g = gs.g[blockIdx.x];
    if (g.blocks == 1) return;
    mergePartials(partials + (size_t)blockIdx.x * RED_BLOCKS * GROUP_VALUES * 2, g.blocks, g.nv, g.ticket, g.pairs);
}

// G = 2..4 groups with linearly independent X/Y masks in one read of the
// state: a thread takes the 2^G amplitudes n ^ (masks selected by v), n having
// the masks' pivot bits clear, and finds every group's pairs among them, v and
// v with bit g flipped.  Group after group the state would be read G times,
// which is all that such a sum costs on a state larger than the caches.  The
// terms are those of FPauliGroup, bit for bit (the first of a pair is the one
// with the mask's top bit, a pivot, clear), and each is added compensated.
// A string's sum (s, c) goes to the host as it is, with the sum of its terms'
// magnitudes: see settled().  Bound by arithmetic where groups have several
// strings, 9 FP64 operations a pair and string: 25 qubits complex128, four
// groups of 5 strings 193 us, of one 119 us (a read for each group: 4 x 92).
__device__ __forceinline__ double flipIf(double x, uint32_t signBit) {
    return __longlong_as_double(__double_as_longlong(x) ^ (long long)((uint64_t)signBit << 32));
}
// kadd of sign * v, sign being 1 or -1
__device__ __forceinline__ void kaddSigned(KB& a, double v, double sign) {
    const double t = fmaT(v, sign, a.s), bb = t - a.s;
    a.c += (a.s - (t - bb)) + fmaT(v, sign, -bb);
    a.s = t;
}
struct PauliSpan {
    PauliGroup g[4];
    uint64_t signs[4];  // byte t: bit p the sign of string t's pair p against the thread's own
    uint32_t swapped[4];  // bit p: the second of pair p has the top bit clear
    InsertSpec pivots;
    uint64_t numWork;
};
template <typename T, int G, int NT>
__global__ void __launch_bounds__(BLOCK, 2) k_pauliSpan(const T* __restrict__ a, PauliSpan s,
                                                    double* __restrict__ partials) {
    constexpr int V = 1 << G;
    KB acc[G][NT];
    double magnitude[G][2];  // of the even and the odd strings' terms
#pragma unroll
    for (int g = 0; g < G; g++) {
        magnitude[g][0] = magnitude[g][1] = 0;
#pragma unroll
        for (int t = 0; t < NT; t++) acc[g][t] = KB{0, 0};
    }
    uint64_t at[V];
#pragma unroll
    for (int v = 0; v < V; v++) {
        at[v] = 0;
#pragma unroll
        for (int g = 0; g < G; g++)
            if ((v >> g) & 1) at[v] ^= s.g[g].maskXY;
    }
    for (uint64_t w = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; w < s.numWork; w += (uint64_t)gridDim.x * BLOCK) {
        const uint64_t n = insertBits(w, s.pivots);
        cd x[V];
#pragma unroll
        for (int v = 0; v < V; v++) x[v] = ldd(a, n ^ at[v]);
#pragma unroll
        for (int g = 0; g < G; g++) {
            double re[V / 2], im[V / 2];
#pragma unroll
            for (int p = 0; p < V / 2; p++) {
                const int v = ((p >> g) << (g + 1)) | (p & ((1 << g) - 1));
                const cd y = x[v], z = x[v | (1 << g)];
                re[p] = fmaT(y.re, z.re, y.im * z.im);
                const double yz = fmaT(y.re, z.im, -(y.im * z.re)), zy = fmaT(z.re, y.im, -(z.im * y.re));
                im[p] = (s.swapped[g] >> p) & 1u ? zy : yz;
                magnitude[g][0] += fabs(re[p]);
                magnitude[g][1] += fabs(im[p]);
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                // the thread's own sign is taken by the accumulator, which
                // leaves the pairs' signs uniform: operands of the additions
                const uint32_t signs = (uint32_t)(s.signs[g] >> (8 * t));
                const uint32_t own = parity64(n & s.g[g].maskYZ[t]) ? 0x80000000u : 0u;
                KB sum = {flipIf(acc[g][t].s, own), flipIf(acc[g][t].c, own)};
                const bool odd = (s.g[g].odd >> t) & 1ull;
#pragma unroll
                for (int p = 0; p < V / 2; p++)
                    kaddSigned(sum, odd ? im[p] : re[p], (signs >> p) & 1u ? -1.0 : 1.0);
                acc[g][t] = KB{flipIf(sum.s, own), flipIf(sum.c, own)};
            }
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        KB sums[NT + 2];
#pragma unroll
        for (int t = 0; t < NT; t++) sums[t] = acc[g][t];
        sums[NT] = KB{magnitude[g][0], 0};
        sums[NT + 1] = KB{magnitude[g][1], 0};
        blockMerge<NT + 2>(sums);
        if (threadIdx.x == 0) {
            double* dst =
                partials + (size_t)g * RED_BLOCKS * GROUP_VALUES * 2 + (size_t)blockIdx.x * (NT + 2) * 2;
#pragma unroll
            for (int t = 0; t < NT + 2; t++) {
                dst[2 * t] = sums[t].s;
                dst[2 * t + 1] = sums[t].c;
            }
        }
        __syncthreads();  // the next group's merge reuses the workgroup's LDS
    }
}

// The value of a sum that a shared read left as (s, c), if it is certain that
// the string's own read gives the same double.
// Both add the same terms, exactly but for the rounding of the compensations:
// an accumulator of k terms holds a compensation of at most k u A (u = 2^-53, A
// the sum of its terms' magnitudes), rounded k times, and D merges round the
// sums of compensations twice each, so that s + c is within 2 (k + D)^2 u^2 A
// of the exact sum of the terms.  The two are then apart by at most delta =
// 4 (k + D)^2 u^2 A, k being the longer chain's, here taken twice, and round to
// the same double when the interval around s + c does.  A sum that is zero but
// for rounding is not settled, nor is one with infinities or NaN.
bool settled(double s, double c, double magnitude, uint64_t chain, double& value) {
    constexpr double MERGES = 48;  // 6 over a wave, 3 waves, 16 partials a lane, 6 more, and some
    const double k = (double)chain + MERGES, delta = 8 * k * k * 0x1p-106 * magnitude;
    const double lo = s + (c - delta), hi = s + (c + delta);
    value = hi;
    return lo == hi;
}

template <typename T>
struct FDensExpecPauli {  // column n, row i = n ^ maskXY: sign(i & maskYZ) rho_{i,n}
    const T* a;
    uint64_t maskXY, maskYZ;
    int N;
    __device__ void operator()(uint64_t n, double* o) const {
        uint64_t i = n ^ maskXY;
        cd v = ldd(a, i + (n << N));
        double s = parity64(i & maskYZ) ? -1.0 : 1.0;
        o[0] = s * v.re;
        o[1] = s * v.im;
    }
};
template <typename T>
struct FInner {
    const T* a;
    const T* b;
    __device__ void operator()(uint64_t n, double* o) const {
        cd t = cmul(cconj(ldd(a, n)), ldd(b, n));
        o[0] = t.re;
        o[1] = t.im;
    }
};
template <typename T>
struct FHSDist {
    const T* a;
    const T* b;
    __device__ void operator()(uint64_t n, double* o) const {
        cd x = ldd(a, n), y = ldd(b, n);
        o[0] = norm2(cd{x.re - y.re, x.im - y.im});
    }
};
template <typename T>
struct FFidelity {  // cpu_densmatr_calcFidelityWithPureState_sub
    const T* rho;
    const T* psi;
    int N, conj;
    __device__ void operator()(uint64_t n, double* o) const {
        uint64_t r = n & ((1ull << N) - 1), c = n >> N;
        cd rv = ldd(rho, n), pr = ldd(psi, r), pc = ldd(psi, c);
        if (conj) {
            rv = cconj(rv);
            pc = cconj(pc);
        } else {
            pr = cconj(pr);
        }
        cd t = cmul(cmul(rv, pr), pc);
        o[0] = t.re;
        o[1] = t.im;
    }
};
__device__ __forceinline__ cd diagElem(const double* __restrict__ e, uint64_t k, int powMode, double xr,
                                       double xi) {
    double er = e[2 * k], ei = e[2 * k + 1];
    if (powMode == 1) return cpowD(er, ei, xr, xi);
    if (powMode == 2) return cd{pow(er, xr), 0};
    return cd{er, ei};
}
template <typename T>
struct FExpecDiag {
    const T* a;
    const double* e;
    int powMode;
    double xr, xi;
    __device__ void operator()(uint64_t n, double* o) const {
        cd t = cscale(diagElem(e, n, powMode, xr, xi), norm2(ldd(a, n)));
        o[0] = t.re;
        o[1] = t.im;
    }
};
template <typename T>
struct FDensExpecDiag {
    const T* a;
    const double* e;
    int powMode;
    double xr, xi;
    uint64_t diagStride;
    __device__ void operator()(uint64_t n, double* o) const {
        cd t = cmul(diagElem(e, n, powMode, xr, xi), ldd(a, n * diagStride));
        o[0] = t.re;
        o[1] = t.im;
    }
};

// Tables of all outcomes of `num` qubits.  A wave reads runs of 64
// consecutive terms (lanes are index bits 0-5, whatever the table's qubits):
// wave (h, c) sums, compensated, the runs whose table qubits above bit 5 hold
// h and whose other high bits r satisfy r = c (mod R), so every lane has one
// accumulator, for the outcome that h and the lane's own table bits make.
// Lanes that differ in other bits are merged, and the R sums of an outcome by
// a wave in k_mergeOutcomes.  Bound by reading the state once, every line
// whole (25 qubits complex128: 98 us and 7 for the merge, 3 qubits or 9; a register
// bin per outcome and a thread per outcome measured 500 and 490 us).  The order of
// every sum depends on the sizes and qubits only.
struct OutcomeShape {
    int laneBits = 0;   // index bits of a run
    int numHigh = 0;    // table qubits above them
    int logRest = 0;    // other high bits
    int logR = 0;
    size_t partials = 0;
};

OutcomeShape outcomeShape(uint64_t numTerms, const int* qubits, int num) {
    OutcomeShape s;
    int n = 0;
    while ((1ull << n) < numTerms) n++;
    s.laneBits = std::min(n, 6);
    for (int i = 0; i < num; i++) s.numHigh += qubits[i] >= s.laneBits;
    s.logRest = n - s.laneBits - s.numHigh;
    // about 2^13 waves, each with at least 4 runs
    s.logR = std::max(0, std::min(s.logRest - 2, 13 - s.numHigh));
    s.partials = s.logR ? ((size_t)2 << num) << s.logR : 0;
    return s;
}

template <typename T>
__global__ void __launch_bounds__(BLOCK) k_outcomeSums(const T* __restrict__ a, InsertSpec high, TargSpec highBit,
                                                      TargSpec low, TargSpec lowBit, OutcomeShape s, uint64_t diagStride,
                                                      double* __restrict__ dst) {
    const uint64_t wave = blockId() * (BLOCK / 64) + (threadIdx.x >> 6);
    if (wave >> (s.numHigh + s.logR)) return;
    const int lane = threadIdx.x & 63;
    const bool active = lane < (1 << s.laneBits);
    const uint64_t h = wave >> s.logR, c = wave & ((1ull << s.logR) - 1ull), R = 1ull << s.logR;
    uint64_t bits = 0, outcome = 0;
    for (int k = 0; k < high.num; k++) {
        const uint64_t one = (h >> k) & 1ull;
        bits |= one << high.pos[k];
        outcome |= one << highBit.targ[k];
    }
    uint32_t tableLanes = 0;
    for (int k = 0; k < low.num; k++) {
        tableLanes |= 1u << low.targ[k];
        outcome |= (uint64_t)((lane >> low.targ[k]) & 1) << lowBit.targ[k];
    }
    auto term = [&](uint64_t r) {
        const uint64_t n = insertBits(r << s.laneBits, high) | bits | (uint64_t)(active ? lane : 0);
        return diagStride ? ldd(a, n * diagStride).re : norm2(ldd(a, n));
    };
    KB acc = {0, 0};
    const uint64_t rest = 1ull << s.logRest;
    uint64_t r = c;
    for (; r + 3 * R < rest; r += 4 * R) {
        double t[4];
#pragma unroll
        for (int u = 0; u < 4; u++) t[u] = term(r + (uint64_t)u * R);
#pragma unroll
        for (int u = 0; u < 4; u++) kadd(acc, t[u]);
    }
    for (; r < rest; r += R) kadd(acc, term(r));
    for (int b = 0; b < s.laneBits; b++) {
        if ((tableLanes >> b) & 1u) continue;
        KB o;
        o.s = __shfl_xor(acc.s, 1 << b, 64);
        o.c = __shfl_xor(acc.c, 1 << b, 64);
        kmerge(acc, o);
    }
    if (!active || (lane & ~tableLanes)) return;
    if (s.logR) {
        dst[2 * ((outcome << s.logR) + c)] = acc.s;
        dst[2 * ((outcome << s.logR) + c) + 1] = acc.c;
    } else {
        dst[outcome] = acc.s + acc.c;
    }
}

__global__ void __launch_bounds__(BLOCK) k_mergeOutcomes(const double* __restrict__ partials, int logR, uint64_t nb,
                                                        double* __restrict__ out) {
    const uint64_t b = (uint64_t)blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    if (b >= nb) return;
    const int lane = threadIdx.x & 63, R = 1 << logR;
    const double* p = partials + 2 * (b << logR);
    KB acc = {0, 0};
    for (int c = lane; c < R; c += 64) kmerge(acc, KB{p[2 * c], p[2 * c + 1]});
    waveMerge(acc);
    if (lane == 0) out[b] = acc.s + acc.c;
}

// the launches of an outcome table on the library stream: partial sums in
// `scratch` (at least shape.partials doubles, every one written before it
// is read), the 2^num probabilities into the device array `res`
template <typename T>
int launchAllOutcomes(double* res, double* scratch, const OutcomeShape& s, const T* a, const int* qubits, int num,
                      uint64_t diagStride) {
    const uint64_t nb = 1ull << num;
    // the table's qubits below and above the lanes' bits, each with its bit of
    // the outcome; the high ones ascending, as zeros to insert into an index
    InsertSpec high;
    TargSpec highBit, low, lowBit;
    high.num = highBit.num = low.num = lowBit.num = 0;
    high.valueMask = 0;
    int order[MAXQ];
    for (int i = 0; i < num; i++) order[i] = i;
    std::sort(order, order + num, [&](int x, int y) { return qubits[x] < qubits[y]; });
    for (int i = 0; i < num; i++) {
        const int q = qubits[order[i]];
        if (q < s.laneBits) {
            low.targ[low.num++] = q;
            lowBit.targ[lowBit.num++] = order[i];
        } else {
            high.pos[high.num++] = q;
            highBit.targ[highBit.num++] = order[i];
        }
    }
    const uint64_t waves = 1ull << (s.numHigh + s.logR);
    k_outcomeSums<T><<<gridFor(waves * 64, 1), BLOCK, 0, stream()>>>(
        a, high, highBit, low, lowBit, s, diagStride, s.logR ? scratch : res);
    QA_LAUNCH_CHECK();
    if (s.logR) {
        k_mergeOutcomes<<<(unsigned)((nb + 3) / 4), BLOCK, 0, stream()>>>(scratch, s.logR, nb, res);
        QA_LAUNCH_CHECK();
    }
    return QA_OK;
}

template <typename T>
int allOutcomes(double* out, const T* a, uint64_t numTerms, const int* qubits, int num, uint64_t diagStride) {
    const uint64_t nb = 1ull << num;
    const OutcomeShape s = outcomeShape(numTerms, qubits, num);
    // small tables are written to pinned memory by the kernel itself
    const bool small = num <= 12;
    double* scratch = devScratch(s.partials + (small ? 1 : (size_t)nb));
    double* host = small ? hostScratch(nb) : nullptr;
    if (!scratch || (small && !host)) return QA_ERR_OOM;
    double* res = small ? host : scratch + s.partials;
    int rc = launchAllOutcomes<T>(res, scratch, s, a, qubits, num, diagStride);
    if (rc != QA_OK) return rc;
    if (small) {
        QA_HIP(hipStreamSynchronize(stream()));
        for (uint64_t b = 0; b < nb; b++) out[b] = host[b];
        return QA_OK;
    }
    QA_HIP(hipMemcpyAsync(out, res, nb * sizeof(double), hipMemcpyDeviceToHost, stream()));
    QA_HIP(hipStreamSynchronize(stream()));
    trimDevScratch();
    return QA_OK;
}

// ---- outcome tables without allocation -----------------------------------
//
// Scratch of qa_statevec_calcProbsOfAllMultiQubitOutcomesNoAlloc: a
// file-scope device array, one copy per device for the life of the
// process.  Its largest use is 2 * 2^19 doubles (2^13 waves of at most 64
// outcomes, one compensated pair each), so every table the allocating entry
// point accepts (1..24 qubits) fits, with the same launch shape and therefore
// the same sums.  Host code reaches it only through the address that
// hipGetSymbolAddress gives, taken once per device by qa_init.
constexpr size_t NOALLOC_SCRATCH_DOUBLES = (size_t)1 << 21;  // 16 MiB
constexpr int NOALLOC_MAX_DEVICES = 64;
__device__ __align__(256) double scratch[NOALLOC_SCRATCH_DOUBLES];
double* g_scratchPtr[NOALLOC_MAX_DEVICES] = {};

}  // namespace

int initLanding() {
    if (g_land) return QA_OK;
    void* p = nullptr;
    QA_HIP(hipHostMalloc(&p, LAND_SLOTS * sizeof(LandSlot), hipHostMallocCoherent | hipHostMallocMapped));
    g_land = static_cast<LandSlot*>(p);
    std::fill_n(reinterpret_cast<unsigned char*>(g_land), LAND_SLOTS * sizeof(LandSlot), (unsigned char)0);
    return QA_OK;
}
void freeLanding() {
    if (g_land) (void)hipHostFree(g_land);
    g_land = nullptr;
}

// called by qa_init with `device` current
int initNoAllocScratch(int device) {
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) {
        setError("qa_init: device %d beyond the %d devices of the no-allocation scratch table", device,
                 NOALLOC_MAX_DEVICES);
        return QA_ERR_ARG;
    }
    if (g_scratchPtr[device]) return QA_OK;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        setError("qa_init: hipGetSymbolAddress of the no-allocation scratch failed: %s", hipGetErrorString(e));
        return QA_ERR_HIP;
    }
    g_scratchPtr[device] = static_cast<double*>(p);
    return QA_OK;
}

namespace {

bool checkArgs(const void* a, int prec, int nq, const char* caller) {
    if (!a || (prec != QA_FP32 && prec != QA_FP64) || nq < 1 || nq > 62) {
        setError("%s: bad qureg arguments", caller);
        return false;
    }
    return true;
}

bool outcomeSpec(InsertSpec& s, int nq, const int* qubits, const int* outcomes, int num, const char* caller) {
    if (num < 0 || num > nq || num > MAXQ) {
        setError("%s: bad number of qubits", caller);
        return false;
    }
    int idx[MAXQ];
    for (int i = 0; i < num; i++) idx[i] = i;
    // insertion sort by qubit
    for (int i = 1; i < num; i++)
        for (int j = i; j > 0 && qubits[idx[j]] < qubits[idx[j - 1]]; j--) {
            int t = idx[j];
            idx[j] = idx[j - 1];
            idx[j - 1] = t;
        }
    s.num = num;
    s.valueMask = 0;
    for (int i = 0; i < num; i++) {
        int q = qubits[idx[i]];
        if (q < 0 || q >= nq || (i && q == s.pos[i - 1])) {
            setError("%s: bad qubit %d", caller, q);
            return false;
        }
        s.pos[i] = q;
        if (outcomes && outcomes[idx[i]]) s.valueMask |= 1ull << q;
    }
    return true;
}

#define QA_DISPATCH(prec, ...)   \
    do {                         \
        if ((prec) == QA_FP64) { \
            typedef double T;    \
            __VA_ARGS__;         \
        } else {                 \
            typedef float T;     \
            __VA_ARGS__;         \
        }                        \
    } while (0)

}  // namespace
}  // namespace qa

using namespace qa;

extern "C" {

int qa_statevec_calcTotalProb(const void* amps, int prec, int nq, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<1>(FNormAll<T>{(const T*)amps}, 1ull << nq, out));
    return rc;
}

int qa_statevec_calcProbsOfEveryQubit(const void* amps, int prec, int nq, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    QA_ARG_CHECK(out, "%s: NULL output", __func__);
    if (nq >= 10 && nq <= PQALL) {
        // every qubit in one read (k_probsOfEveryQubit)
        const uint64_t chunks = 1ull << (nq - 10);
        const int blocks = (int)std::min<uint64_t>(RED_BLOCKS, (chunks + BLOCK / 64 - 1) / (BLOCK / 64));
        const int nval = nq <= 16 ? 32 : nq <= 24 ? 48 : 64;
        double* scratch = devScratch((size_t)blocks * nval * 2);
        double* host = hostScratch((size_t)nval);
        if (!scratch || !host) {
            setError("reduction scratch unavailable");
            return QA_ERR_OOM;
        }
#define QA_PROBS(NHI) \
    QA_DISPATCH(prec, (k_probsOfEveryQubit<T, NHI><<<blocks, BLOCK, 0, stream()>>>((const T*)amps, chunks, scratch)))
        if (nval == 32) QA_PROBS(6);
        else if (nval == 48) QA_PROBS(14);
        else QA_PROBS(22);
#undef QA_PROBS
        QA_LAUNCH_CHECK();
        k_finalizeProbs<<<1, 1024, 0, stream()>>>(scratch, blocks, nval, host);
        QA_LAUNCH_CHECK();
        QA_HIP(hipStreamSynchronize(stream()));
        for (int q = 0; q < nq; q++) {
            out[2 * q] = host[2 * q];
            out[2 * q + 1] = host[2 * q + 1];
        }
        return QA_OK;
    }
    for (int q0 = 0; q0 < nq; q0 += PQ) {
        double v[2 * PQ];
        int rc;
        QA_DISPATCH(prec, rc = runReduce<2 * PQ>(FProbsOfQubits<T>{(const T*)amps, q0}, 1ull << nq, v));
        if (rc != QA_OK) return rc;
        for (int b = 0; b < PQ && q0 + b < nq; b++) {
            out[2 * (q0 + b)] = v[b];
            out[2 * (q0 + b) + 1] = v[PQ + b];
        }
    }
    return QA_OK;
}

int qa_densmatr_calcTotalProb(const void* amps, int prec, int N, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, 2 * N, __func__)) return QA_ERR_ARG;
    InsertSpec none;
    none.num = 0;
    none.valueMask = 0;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<1>(FDiagReal<T>{(const T*)amps, none, (1ull << N) + 1}, 1ull << N, out));
    return rc;
}

int qa_statevec_calcProbOfMultiQubitOutcome(const void* amps, int prec, int nq, const int* qubits,
                                            const int* outcomes, int num, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    InsertSpec ins;
    if (!outcomeSpec(ins, nq, qubits, outcomes, num, __func__)) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<1>(FNormOutcome<T>{(const T*)amps, ins}, 1ull << (nq - num), out));
    return rc;
}

int qa_densmatr_calcProbOfMultiQubitOutcome(const void* amps, int prec, int N, const int* qubits,
                                            const int* outcomes, int num, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, 2 * N, __func__)) return QA_ERR_ARG;
    InsertSpec ins;
    if (!outcomeSpec(ins, N, qubits, outcomes, num, __func__)) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<1>(FDiagReal<T>{(const T*)amps, ins, (1ull << N) + 1}, 1ull << (N - num), out));
    return rc;
}

int qa_statevec_calcProbsOfAllMultiQubitOutcomes(double* out, const void* amps, int prec, int nq,
                                                 const int* qubits, int num) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    InsertSpec chk;
    if (!outcomeSpec(chk, nq, qubits, nullptr, num, __func__)) return QA_ERR_ARG;
    QA_ARG_CHECK(num >= 1 && num <= 24, "%s: %d qubits unsupported", __func__, num);
    int rc;
    QA_DISPATCH(prec, rc = allOutcomes<T>(out, (const T*)amps, 1ull << nq, qubits, num, 0));
    return rc;
}

int qa_statevec_calcProbsOfAllMultiQubitOutcomesNoAlloc(double* devOutProbs, const void* amps, int prec, int nq,
                                                        const int* qubits, int num) {
    QA_REQUIRE_INIT_RO();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    QA_ARG_CHECK(devOutProbs, "%s: NULL output", __func__);
    InsertSpec chk;
    if (!outcomeSpec(chk, nq, qubits, nullptr, num, __func__)) return QA_ERR_ARG;
    QA_ARG_CHECK(num >= 1 && num <= 24, "%s: %d qubits unsupported", __func__, num);
    // a flush could allocate the fusion program ring: the caller flushes first
    QA_ARG_CHECK(!fuse::pending(amps), "%s: gates are queued for this state; call qa_flush(amps) first", __func__);
    const int dev = device();
    double* sp = (dev >= 0 && dev < NOALLOC_MAX_DEVICES) ? g_scratchPtr[dev] : nullptr;
    if (!sp) {
        setError("%s: no scratch address for device %d", __func__, dev);
        return QA_ERR_NOT_INIT;
    }
    const OutcomeShape s = outcomeShape(1ull << nq, qubits, num);
    QA_ARG_CHECK(s.partials <= NOALLOC_SCRATCH_DOUBLES,
                 "%s: a %d-qubit table of a %d-qubit state needs %zu doubles of scratch, more than the %zu of the "
                 "no-allocation scratch", __func__, num, nq, s.partials, NOALLOC_SCRATCH_DOUBLES);
    int rc;
    QA_DISPATCH(prec, rc = launchAllOutcomes<T>(devOutProbs, sp, s, (const T*)amps, qubits, num, 0));
    return rc;
}

int qa_densmatr_calcProbsOfAllMultiQubitOutcomes(double* out, const void* amps, int prec, int N,
                                                 const int* qubits, int num) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, 2 * N, __func__)) return QA_ERR_ARG;
    InsertSpec chk;
    if (!outcomeSpec(chk, N, qubits, nullptr, num, __func__)) return QA_ERR_ARG;
    QA_ARG_CHECK(num >= 1 && num <= 24, "%s: %d qubits unsupported", __func__, num);
    int rc;
    QA_DISPATCH(prec, rc = allOutcomes<T>(out, (const T*)amps, 1ull << N, qubits, num, (1ull << N) + 1));
    return rc;
}

int qa_statevec_calcInnerProduct(const void* a, const void* b, int prec, int nq, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(a, prec, nq, __func__) || !b) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<2>(FInner<T>{(const T*)a, (const T*)b}, 1ull << nq, out));
    return rc;
}

int qa_densmatr_calcHilbertSchmidtDistance(const void* a, const void* b, int prec, int N, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(a, prec, 2 * N, __func__) || !b) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<1>(FHSDist<T>{(const T*)a, (const T*)b}, 1ull << (2 * N), out));
    return rc;
}

int qa_densmatr_calcFidelityWithPureState(const void* rho, const void* psi, int prec, int N, int conj,
                                          double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(rho, prec, 2 * N, __func__) || !psi) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<2>(FFidelity<T>{(const T*)rho, (const T*)psi, N, conj}, 1ull << (2 * N), out));
    return rc;
}

int qa_statevec_calcExpecAnyTargZ(const void* amps, int prec, int nq, uint64_t mask, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<1>(FExpecZ<T>{(const T*)amps, mask}, 1ull << nq, out));
    return rc;
}

int qa_densmatr_calcExpecAnyTargZ(const void* amps, int prec, int N, uint64_t mask, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, 2 * N, __func__)) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<2>(FDensExpecZ<T>{(const T*)amps, mask, (1ull << N) + 1}, 1ull << N, out));
    return rc;
}

}  // extern "C"

namespace qa {
namespace {

void timesPowerOfI(double* v, int k) {
    for (int i = 0; i < (k & 3); i++) {
        double re = v[0], im = v[1];
        v[0] = -im;
        v[1] = re;
    }
}

// one launch of groups gs.g[from, to), each its own read
template <typename T>
int launchGroups(const T* a, PauliGroups& gs, int from, int to, double* scratch) {
    int most = 1, maxBlocks = 1;
    PauliGroups sub;
    for (int i = from; i < to; i++) most = std::max(most, gs.g[i].numStrings);
    for (int i = from; i < to; i++) {
        gs.g[i].nv = most;
        gs.g[i].pairs = 0;
        sub.g[i - from] = gs.g[i];
        maxBlocks = std::max(maxBlocks, gs.g[i].blocks);
    }
    double* dst = scratch + (size_t)from * RED_BLOCKS * GROUP_VALUES * 2;
    const dim3 grid((unsigned)maxBlocks, (unsigned)(to - from), 1);
    switch (most) {
#define QA_NV(NV) \
    case NV: k_pauliGroups<T, NV><<<grid, BLOCK, 0, stream()>>>(a, sub, dst); break
        QA_NV(1); QA_NV(2); QA_NV(3); QA_NV(4); QA_NV(5); QA_NV(6); QA_NV(7); QA_NV(8);
#undef QA_NV
    }
    QA_LAUNCH_CHECK();
    return QA_OK;
}

// one launch of groups gs.g[from, from + num), num = 2..4 with independent
// masks, in one read; chain: the most terms that one accumulator adds
template <typename T>
int launchSpanGroups(const T* a, int nq, PauliGroups& gs, int from, int num, double* scratch, uint64_t& chain) {
    PauliSpan s;
    // the first amplitude of pair p of group g, against the thread's own: the
    // masks selected by p with a zero inserted at bit g
    auto firstOf = [&](int g, int p) {
        const int v = ((p >> g) << (g + 1)) | (p & ((1 << g) - 1));
        uint64_t at = 0;
        for (int b = 0; b < num; b++)
            if ((v >> b) & 1) at ^= s.g[b].maskXY;
        return at;
    };
    int most = 1;
    for (int i = 0; i < num; i++) most = std::max(most, gs.g[from + i].numStrings);
    // each mask less the pivots (highest bits) of those before it
    uint64_t lead[4], pivots = 0;
    for (int i = 0; i < num; i++) {
        uint64_t m = gs.g[from + i].maskXY;
        for (int j = 0; j < i; j++)
            if ((m >> (63 - __builtin_clzll(lead[j]))) & 1ull) m ^= lead[j];
        lead[i] = m;
        pivots |= 1ull << (63 - __builtin_clzll(m));
    }
    s.pivots.num = 0;
    s.pivots.valueMask = 0;
    for (int q = 0; q < nq; q++)
        if ((pivots >> q) & 1ull) s.pivots.pos[s.pivots.num++] = q;
    s.numWork = 1ull << (nq - num);
    // as many workgroups as are resident (2 waves per SIMD)
    const int blocks = (int)std::min<uint64_t>(RED_BLOCKS / 2, (s.numWork + BLOCK - 1) / BLOCK);
    for (int i = 0; i < num; i++) {
        gs.g[from + i].nv = most + 2;
        gs.g[from + i].pairs = 1;
        gs.g[from + i].blocks = blocks;
        s.g[i] = gs.g[from + i];
    }
    chain = (s.numWork / ((uint64_t)blocks * BLOCK) + 1) << (num - 1);
    for (int g = 0; g < num; g++) {
        s.signs[g] = 0;
        s.swapped[g] = 0;
        const uint64_t top = s.g[g].topLow + 1;
        for (int p = 0; p < (1 << num) / 2; p++)
            s.swapped[g] |= (firstOf(g, p) & top) ? 1u << p : 0u;
        for (int t = 0; t < s.g[g].numStrings; t++) {
            const uint64_t odd = (s.g[g].odd >> t) & 1ull;
            for (int p = 0; p < (1 << num) / 2; p++) {
                // an even string's sign is that of either amplitude, an odd one's
                // that of the amplitude with the top bit set
                const uint64_t par = (uint64_t)(__builtin_popcountll(firstOf(g, p) & s.g[g].maskYZ[t]) & 1);
                const uint64_t swapped = (s.swapped[g] >> p) & 1u;
                s.signs[g] |= (par ^ (odd & ~swapped)) << (8 * t + p);
            }
        }
    }
    double* dst = scratch + (size_t)from * RED_BLOCKS * GROUP_VALUES * 2;
    switch (num * 16 + most) {
#define QA_SPAN(G, NT) \
    case G * 16 + NT: k_pauliSpan<T, G, NT><<<blocks, BLOCK, 0, stream()>>>(a, s, dst); break
#define QA_SPANS(G)                                             \
    QA_SPAN(G, 1); QA_SPAN(G, 2); QA_SPAN(G, 3); QA_SPAN(G, 4); \
    QA_SPAN(G, 5); QA_SPAN(G, 6); QA_SPAN(G, 7); QA_SPAN(G, 8)
        QA_SPANS(2); QA_SPANS(3); QA_SPANS(4);
#undef QA_SPANS
#undef QA_SPAN
    }
    QA_LAUNCH_CHECK();
    return QA_OK;
}

// whether mask is no XOR of some of masks[0, num)
bool independent(const uint64_t* masks, int num, uint64_t mask) {
    for (int v = 0; v < (1 << num); v++) {
        uint64_t x = mask;
        for (int g = 0; g < num; g++)
            if ((v >> g) & 1) x ^= masks[g];
        if (!x) return false;
    }
    return true;
}

// Sums over states of at least this many qubits read the state once for up to
// 4 groups (k_pauliSpan).  One call, a read per four groups against a read per
// group (us, random states; groups x strings):
//   complex128   2x1        4x1        4x4        4x5        4x8        8x4
//   20 qubits    18 / 16    19 / 20    28 / 26    31 / 29    43 / 33    44 / 32
//   21           18 / 25    22 / 34    35 / 36    39 / 45    58 / 50    60 / 53
//   22           26 / 35    29 / 47    46 / 52    50 / 61    73 / 69    77 / 90
//   23           35 / 48    41 / 84    62 / 90    69 / 98    104 / 115  107 / 168
//   24           52 / 88    58 / 164   92 / 187   106 / 185  168 / 197  177 / 332
//   complex64
//   21           18 / 20    22 / 26    35 / 32    38 / 40    54 / 48    56 / 46
//   22           22 / 25    26 / 31    43 / 43    48 / 53    70 / 67    72 / 68
//   23           29 / 33    35 / 47    60 / 65    67 / 78    99 / 104   104 / 115
//   24           41 / 51    48 / 79    90 / 107   106 / 131  161 / 182  172 / 193
// A group with a sum that is not settled (zero but for rounding, which
// symmetries of a state bring about) is read once more: at worst the two
// add up, 26 qubits complex128 4x5 strings of zero sum 1057 us, alone 715.
constexpr int SPAN_MIN_QUBITS = 22;

// The values of numTerms Pauli strings, (re, im) each, in vals: strings are
// grouped by X/Y mask (of at most GROUP_STRINGS, in ascending mask order, each
// in term order), and each group is one read of the state or shares one with
// up to three others; where a shared read leaves a last bit open, the group is
// read by itself too, so that a string's value is that of its own read
// whatever it is summed with.  Up to MAX_GROUPS groups are launched together and then
// waited for.
template <typename T>
int expecStrings(const T* a, int nq, int64_t numTerms, const uint64_t* maskX, const uint64_t* maskY,
                 const uint64_t* maskZ, double* vals) {
    std::vector<int64_t> order((size_t)numTerms);
    for (int64_t t = 0; t < numTerms; t++) order[t] = t;
    std::stable_sort(order.begin(), order.end(), [&](int64_t x, int64_t y) {
        return (maskX[x] | maskY[x]) < (maskX[y] | maskY[y]);
    });
    struct Group {
        uint64_t mxy;
        int64_t first;
        int num;
    };
    std::vector<Group> alone, rest, later;
    for (int64_t at = 0; at < numTerms;) {
        Group g{maskX[order[at]] | maskY[order[at]], at, 0};
        while (at < numTerms && (maskX[order[at]] | maskY[order[at]]) == g.mxy && g.num < GROUP_STRINGS) {
            at++;
            g.num++;
        }
        (g.mxy && nq >= SPAN_MIN_QUBITS ? rest : alone).push_back(g);
    }
    double* scratch = nullptr;
    while (!alone.empty() || !rest.empty()) {
        PauliGroups gs;
        int64_t first[MAX_GROUPS];
        uint64_t chains[MAX_GROUPS];
        int num = 0, rc = QA_OK;
        auto take = [&](const Group& x) {
            PauliGroup& g = gs.g[num];
            first[num++] = x.first;
            g.maskXY = x.mxy;
            g.topLow = x.mxy ? (1ull << (63 - __builtin_clzll(x.mxy))) - 1ull : 0;
            g.odd = 0;
            g.numStrings = x.num;
            for (int t = 0; t < GROUP_STRINGS; t++) g.maskYZ[t] = 0;
            for (int t = 0; t < x.num; t++) {
                const int64_t term = order[x.first + t];
                g.maskYZ[t] = maskY[term] | maskZ[term];
                // as many bits in both as there are Y; a single string may also
                // have X and Z on one qubit, whose product it then is
                g.odd |= (uint64_t)(__builtin_popcountll(x.mxy & g.maskYZ[t]) & 1) << t;
            }
            g.numWork = 1ull << (x.mxy ? nq - 1 : nq);
            g.blocks = reduceBlocks(g.numWork);
            g.ticket = takeTicket();
        };
        if (!scratch) {
            const size_t groups = std::min<size_t>(MAX_GROUPS, alone.size() + rest.size());
            scratch = devScratch(groups * RED_BLOCKS * GROUP_VALUES * 2);
            if (!scratch || !g_land) {
                setError("reduction scratch unavailable");
                return QA_ERR_OOM;
            }
        }
        while (!rest.empty() && num + 4 <= MAX_GROUPS) {
            uint64_t masks[4];
            int n = 0;
            const int from = num;
            later.clear();
            for (const Group& g : rest) {
                if (n < 4 && independent(masks, n, g.mxy)) {
                    masks[n++] = g.mxy;
                    take(g);
                } else {
                    later.push_back(g);
                }
            }
            rest.swap(later);
            uint64_t chain = 0;
            rc = n > 1 ? launchSpanGroups(a, nq, gs, from, n, scratch, chain) : launchGroups(a, gs, from, num, scratch);
            if (rc != QA_OK) return rc;
            for (int i = from; i < num; i++) chains[i] = chain;
        }
        const int from = num;
        while (!alone.empty() && num < MAX_GROUPS) {
            take(alone.back());
            alone.pop_back();
        }
        if (num > from) rc = launchGroups(a, gs, from, num, scratch);
        if (rc != QA_OK) return rc;
        bool merge = false;
        for (int i = 0; i < num; i++) merge = merge || gs.g[i].blocks > 1;
        if (merge) {
            k_finalizeGroups<<<(unsigned)num, BLOCK, 0, stream()>>>(gs, scratch);
            QA_LAUNCH_CHECK();
        }
        for (int i = 0; i < num; i++) {
            const PauliGroup& g = gs.g[i];
            double res[LAND_VALUES];
            rc = land(g.ticket, res, g.pairs ? 2 * g.nv : g.numStrings);
            if (rc != QA_OK) return rc;
            if (g.pairs) {
                const double* const c = res + g.nv;
                const uint64_t own = g.numWork / ((uint64_t)reduceBlocks(g.numWork) * BLOCK) + 1;
                bool all = true;
                for (int t = 0; t < g.numStrings; t++) {
                    const int mag = g.nv - 2 + (int)((g.odd >> t) & 1ull);
                    all &= settled(res[t], c[t], res[mag] + c[mag], std::max(own, chains[i]), res[t]);
                }
                if (!all) {
                    alone.push_back(Group{g.maskXY, first[i], g.numStrings});
                    continue;
                }
            }
            for (int t = 0; t < g.numStrings; t++) {
                const int64_t term = order[first[i] + t];
                const double x = g.maskXY ? 2 * res[t] : res[t];
                const bool odd = (g.odd >> t) & 1ull;
                vals[2 * term] = odd ? 0 : x;
                vals[2 * term + 1] = odd ? x : 0;
                timesPowerOfI(vals + 2 * term, __builtin_popcountll(maskY[term]));
            }
        }
    }
    return QA_OK;
}

}  // namespace
}  // namespace qa

extern "C" {

int qa_statevec_calcExpecPauliStr(const void* amps, int prec, int nq, uint64_t maskX, uint64_t maskY,
                                  uint64_t maskZ, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    const uint64_t all = nq >= 64 ? ~0ull : ((1ull << nq) - 1ull);
    QA_ARG_CHECK(((maskX | maskY) & ~all) == 0, "%s: Pauli beyond register", __func__);
    int rc;
    QA_DISPATCH(prec, rc = expecStrings<T>((const T*)amps, nq, 1, &maskX, &maskY, &maskZ, out));
    return rc;
}

int qa_statevec_calcExpecPauliStrSum(const void* amps, int prec, int nq, int64_t numTerms, const uint64_t* maskX,
                                     const uint64_t* maskY, const uint64_t* maskZ, const double* coeffs,
                                     double* termValues, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__)) return QA_ERR_ARG;
    QA_ARG_CHECK(numTerms >= 0 && (numTerms == 0 || (maskX && maskY && maskZ && coeffs)),
                 "%s: bad term arrays", __func__);
    const uint64_t all = nq >= 64 ? ~0ull : ((1ull << nq) - 1ull);
    for (int64_t t = 0; t < numTerms; t++)
        QA_ARG_CHECK(((maskX[t] | maskY[t] | maskZ[t]) & ~all) == 0 && !(maskX[t] & maskY[t]) &&
                         !(maskX[t] & maskZ[t]) && !(maskY[t] & maskZ[t]),
                     "%s: term %lld is not a Pauli string on the qureg", __func__, (long long)t);
    std::vector<double> vals(2 * (size_t)numTerms);
    int rc = QA_OK;
    QA_DISPATCH(prec, rc = expecStrings<T>((const T*)amps, nq, numTerms, maskX, maskY, maskZ, vals.data()));
    if (rc != QA_OK) return rc;
    // sum of coefficient x value, in term order
    double re = 0, im = 0;
    for (int64_t t = 0; t < numTerms; t++) {
        const double cr = coeffs[2 * t], ci = coeffs[2 * t + 1], vr = vals[2 * t], vi = vals[2 * t + 1];
        re += cr * vr - ci * vi;
        im += cr * vi + ci * vr;
    }
    if (termValues)
        for (int64_t t = 0; t < 2 * numTerms; t++) termValues[t] = vals[t];
    out[0] = re;
    out[1] = im;
    return QA_OK;
}

int qa_densmatr_calcExpecPauliStr(const void* amps, int prec, int N, uint64_t maskX, uint64_t maskY,
                                  uint64_t maskZ, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, 2 * N, __func__)) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<2>(FDensExpecPauli<T>{(const T*)amps, maskX | maskY, maskY | maskZ, N},
                                        1ull << N, out));
    if (rc == QA_OK) timesPowerOfI(out, __builtin_popcountll(maskY));
    return rc;
}

int qa_statevec_calcExpecFullStateDiagMatr(const void* amps, int prec, int nq, const void* e, int powMode,
                                           double xr, double xi, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, nq, __func__) || !e) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<2>(FExpecDiag<T>{(const T*)amps, (const double*)e, powMode, xr, xi},
                                        1ull << nq, out));
    return rc;
}

int qa_densmatr_calcExpecFullStateDiagMatr(const void* amps, int prec, int N, const void* e, int powMode,
                                           double xr, double xi, double* out) {
    QA_REQUIRE_INIT_RO();
    QA_FLUSH_ALL();
    if (!checkArgs(amps, prec, 2 * N, __func__) || !e) return QA_ERR_ARG;
    int rc;
    QA_DISPATCH(prec, rc = runReduce<2>(FDensExpecDiag<T>{(const T*)amps, (const double*)e, powMode, xr, xi,
                                                          (1ull << N) + 1},
                                        1ull << N, out));
    return rc;
}

}  // extern "C"
