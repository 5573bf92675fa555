// Device helpers shared by the fused evolution kernel (kernels.hip) and the
// split generation loop (split_kernels.hip): member rows, jDE controls, trial
// vectors, chi^2 sums and the reference's non-fused dot product.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace deac {

namespace {

// Chain of one (member, row) pair in the order of the reference's inlined
// matrix_multiply_MxN_by_Nx1 (deac.cpp:102-108): rounded products added one at
// a time, except the last element of each sign when G is odd, which is fused.
__device__ double fold_row(const double *x, const double *row, int Kc, int G)
{
    constexpr int kBatch = 16;
    double acc = 0.0;
    const bool godd = (G & 1) != 0;
    for (int k0 = 0; k0 < Kc; k0 += kBatch) {
        double xv[kBatch], rv[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int k = k0 + u;
            xv[u] = k < Kc ? x[k] : 0.0;
            rv[u] = k < Kc ? row[k] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int k = k0 + u;
            if (k >= Kc) break;
            if (godd && (k == G - 1 || k == Kc - 1)) acc = fma(xv[u], rv[u], acc);
            else acc = acc + xv[u] * rv[u];
        }
    }
    return acc;
}

// Genome row of member i that the chain phase reads: the current genome for
// the initial fitness, the trial (in the spare buffer) otherwise.
__device__ __forceinline__ const double *chain_row(const EvoArgs &a, int i, bool init)
{
    const int c = i < a.P ? a.cur[i] : 0;
    const bool second = init ? c != 0 : c == 0;
    return (second ? a.pop1 : a.pop0) + static_cast<size_t>(i) * a.stride;
}

// Two doubles as a native vector: plain 16-byte loads and stores that stay
// in registers (HIP's double2 struct is copied through memory).
typedef double dvec2 __attribute__((ext_vector_type(2)));
typedef uint64_t uvec2 __attribute__((ext_vector_type(2)));

// The state of the members as one workgroup sees it: in its LDS, where every
// workgroup repeats the selection (EvoArgs::local), or in global memory.
struct Members {
    double *fitness, *cr, *f;  // [P], [P][nsign], [P][nsign]
    int *cur;                  // [P]
};

__device__ __forceinline__ const double *row_of(const EvoArgs &a, const int *cur, int i, bool spare)
{
    return ((cur[i] != 0) != spare ? a.pop1 : a.pop0) + static_cast<size_t>(i) * a.stride;
}

// CR and F of member i in a generation, per sign (the second repeats the first
// where there is one sign): redrawn or the member's own.  Both are loaded
// whichever holds, so that a member costs one memory latency and not one per
// value.
struct Controls {
    double cr[2] = {0.0, 0.0}, f[2] = {0.0, 0.0};
    __device__ __forceinline__ Controls() {}
    __device__ __forceinline__ Controls(const EvoArgs &a, const Members &s, const MemberCtl &c, int i)
    {
        const int j = i * a.nsign, j1 = j + a.nsign - 1, two = a.nsign - 1;
        const double c0 = s.cr[j], c1 = s.cr[j1], f0 = s.f[j], f1 = s.f[j1];
        const double n0 = c.cr_value[0], n1 = c.cr_value[1], m0 = c.f_value[0], m1 = c.f_value[1];
        const uint32_t flags = c.flags;
        cr[0] = flags & 1 ? n0 : c0;
        f[0] = flags & 2 ? m0 : f0;
        cr[1] = !two ? cr[0] : flags & 4 ? n1 : c1;
        f[1] = !two ? f[0] : flags & 8 ? m1 : f1;
    }
};

// u < cr for the draw u = r 2^-53, as r < ceil(cr 2^53) in whole numbers
__device__ __forceinline__ uint64_t cross_limit(double cr)
{
    return !(cr > 0.0) ? 0 : cr >= 1.0 ? UINT64_C(1) << 53 : static_cast<uint64_t>(ceil(cr * 0x1.0p53));
}

// A member's trial vector (deac.cpp:1261-1308), in blocks of 128 genome
// positions, two per lane: load() fetches a block's parent, donor and draw
// values, form() the trial values, zero past the genome.  The values are all
// loaded, whichever the crossover keeps, so the loads issue together instead
// of behind the comparison.
struct Trial {
    const EvoArgs &a;
    const uint64_t *raw;
    const double *r1, *r2, *r3, *rp;
    double *out;  // the member's spare row
    double f0, f1;
    uint64_t lim0, lim1;
    struct Load {
        uvec2 u;
        dvec2 x1, x2, x3, xp;
    };
    __device__ __forceinline__ Trial(const EvoArgs &ea, const Members &s, const int *cur, const MemberCtl &c,
                                     const uint64_t *draws, int i)
        : a(ea), raw(draws)
    {
        r1 = row_of(a, cur, c.mutant[0], false);
        r2 = row_of(a, cur, c.mutant[1], false);
        r3 = row_of(a, cur, c.mutant[2], false);
        rp = row_of(a, cur, i, false);
        out = const_cast<double *>(row_of(a, cur, i, true));
        const Controls k(a, s, c, i);
        f0 = k.f[0];
        f1 = k.f[1];
        lim0 = cross_limit(k.cr[0]);
        lim1 = cross_limit(k.cr[1]);
    }
    static __device__ __forceinline__ int position(int b) { return b * kChunk + 2 * (threadIdx.x & 63); }
    __device__ __forceinline__ void load(int b, Load &v) const
    {
        const int k = position(b);
        if (k < a.Kc) v.u = *reinterpret_cast<const uvec2 *>(raw + k);
        v.x1 = *reinterpret_cast<const dvec2 *>(r1 + k);
        v.x2 = *reinterpret_cast<const dvec2 *>(r2 + k);
        v.x3 = *reinterpret_cast<const dvec2 *>(r3 + k);
        v.xp = *reinterpret_cast<const dvec2 *>(rp + k);
    }
    __device__ __forceinline__ double value(bool neg, uint64_t r, double d1, double d2, double d3, double p) const
    {
        const double w = fma(neg ? f1 : f0, d2 - d3, d1);
        return r < (neg ? lim1 : lim0) ? (a.allow_neg ? w : fabs(w)) : p;
    }
    __device__ __forceinline__ dvec2 form(int b, const Load &v) const
    {
        const int k = position(b);
        dvec2 o = {0.0, 0.0};
        if (k < a.Kc) o.x = value(k >= a.G, v.u.x, v.x1.x, v.x2.x, v.x3.x, v.xp.x);
        if (k + 1 < a.Kc) o.y = value(k + 1 >= a.G, v.u.y, v.x1.y, v.x2.y, v.x3.y, v.xp.y);
        // the negative sign's zero frequency repeats the positive one's
        if (a.nsign == 2 && (k == a.G || k + 1 == a.G)) {
            const double z = value(false, raw[0], r1[0], r2[0], r3[0], rp[0]);
            if (k == a.G) o.x = z;
            else o.y = z;
        }
        return o;
    }
    __device__ __forceinline__ void store(int b, const dvec2 &o) const
    {
        *reinterpret_cast<dvec2 *>(out + position(b)) = o;
    }
};

// Sums d[0..n) squared in tau order from LDS, the last one fused when fused
// is set (deac.cpp:120-126); 8 reads ahead of the adds.
__device__ __forceinline__ double chi_sum(const double *d, int n, bool fused, double acc)
{
    const int m = fused ? n - 1 : n;
    int t = 0;
    for (; t + 8 <= m; t += 8) {
        double v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = d[t + e];
#pragma unroll
        for (int e = 0; e < 8; e++) acc = acc + v[e] * v[e];
    }
    for (; t < m; t++) acc = acc + d[t] * d[t];
    if (fused) acc = fma(d[n - 1], d[n - 1], acc);
    return acc;
}

}  // namespace

}  // namespace deac
