// Compensated FP64 accumulation shared by the reductions (qa_reduce.hip)
// and the serving engine's batched expectations (qa_serve.hip).
#pragma once

#include "qa_common.hpp"

namespace qa {

struct KB {  // compensated accumulator
    double s, c;
};

// the rounding error of t = a + b, exact (Knuth's two-sum): the value
// Neumaier's larger-minus-smaller form gives, in 6 operations without the
// comparison and its four selects
__device__ __forceinline__ double sumError(double a, double b, double t) {
    const double bb = t - a;
    return (a - (t - bb)) + (b - bb);
}
__device__ __forceinline__ void kadd(KB& a, double v) {
    const double t = a.s + v;
    a.c += sumError(a.s, v, t);
    a.s = t;
}
// symmetric in a and b, so that a merge gives both lanes of a pair the same
__device__ __forceinline__ void kmerge(KB& a, KB b) {
    const double t = a.s + b.s;
    a.c = (a.c + b.c) + sumError(a.s, b.s, t);
    a.s = t;
}
// the lanes' accumulators merged; every lane ends holding the result
__device__ __forceinline__ void waveMerge(KB& acc) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        KB o;
        o.s = __shfl_xor(acc.s, off, 64);
        o.c = __shfl_xor(acc.c, off, 64);
        kmerge(acc, o);
    }
}

// reduce NV compensated accumulators across the workgroup; thread 0 ends
// holding the result.  Lanes are paired at distances 32, 16, .. 1; while more
// than one value is left, a pair splits them (each lane hands over one half
// and merges the other), so a wave makes NV + 4 or so merges rather than
// 6 NV.  The pairing does not depend on NV, so neither does a value's sum.
template <int NV>
__device__ void blockMerge(KB (&acc)[NV]) {
    constexpr int H = NV <= 1 ? 0 : NV <= 2 ? 1 : NV <= 4 ? 2 : NV <= 8 ? 3 : NV <= 16 ? 4 : 5, P = 1 << H;
    static_assert(NV <= 32, "values of one merge");
    __shared__ KB sh[BLOCK / 64][P];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    KB t[P];
#pragma unroll
    for (int v = 0; v < P; v++) t[v] = v < NV ? acc[v] : KB{0, 0};
#pragma unroll
    for (int h = 0; h < H; h++) {
        const int half = P >> (h + 1), dist = 32 >> h;
        const bool up = lane & dist;
#pragma unroll
        for (int v = 0; v < half; v++) {
            const KB lo = t[v], hi = t[v + half];
            KB give = {up ? lo.s : hi.s, up ? lo.c : hi.c};
            KB keep = {up ? hi.s : lo.s, up ? hi.c : lo.c};
            give.s = __shfl_xor(give.s, dist, 64);
            give.c = __shfl_xor(give.c, dist, 64);
            kmerge(keep, give);
            t[v] = keep;
        }
    }
#pragma unroll
    for (int dist = 32 >> H; dist >= 1; dist >>= 1) {
        KB o;
        o.s = __shfl_xor(t[0].s, dist, 64);
        o.c = __shfl_xor(t[0].c, dist, 64);
        kmerge(t[0], o);
    }
    constexpr int LANES = 64 >> H;  // lanes that hold the same value
    if (lane % LANES == 0) sh[wave][lane / LANES] = t[0];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            acc[v] = sh[0][v];
            for (int w = 1; w < BLOCK / 64; w++) kmerge(acc[v], sh[w][v]);
        }
    }
}

}  // namespace qa
