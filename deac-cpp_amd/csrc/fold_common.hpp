// Sequential folds on the matrix cores, shared by the kernels that need the
// reference's non-fused dot product (matrix_multiply_MxN_by_Nx1 as its build
// inlines it, deac.cpp:102-108): rounded products added one at a time in
// position order, the last element of each sign fused when the genome length
// is odd.
//
// v_mfma_f64_4x4x4_4b_f64 is four fused multiply-adds in ascending k for every
// output, so with rounded products p in A and ones in B it is four additions in
// order: fma(p, 1, acc) rounds p + acc once.  8.8 ns per MFMA are 2.2 ns per
// position, and one instruction in four: a wavefront issues one instruction
// every five cycles or so, and a chain of v_add_f64 needs one per position and
// half a load (5.3 ns per position through LDS, 5.0 by DPP row_newbcast).
#pragma once

#include <hip/hip_runtime.h>

namespace deac {

namespace {

typedef double fold_pair __attribute__((ext_vector_type(2)));

// Blocks of 128 positions, two per lane; units of 8 positions, two MFMAs each;
// units read ahead from LDS; LDS of one wave_fold: two blocks of products.
constexpr int kFoldBlock = 128;
constexpr int kFoldUnits = kFoldBlock / 8;
constexpr int kFoldAhead = 8;
constexpr int kFoldLds = 2 * kFoldBlock;

// The fused elements of a fold: positions within the block, second factors
// (their first factors stand in LDS in place of the products).
struct FoldFused {
    int k[2];
    double w[2];
};

// Adds one block; v holds the units about to be added and is refilled
// kFoldAhead units on (past the block's end from the next one).
template <bool FUSED>
__device__ __forceinline__ void fold_block(double &acc, fold_pair (&v)[kFoldAhead], const double *here,
                                           const double *next, const FoldFused &f)
{
    const int q = (threadIdx.x & 63) >> 4;
    auto second = [&](int k) __attribute__((always_inline)) {
        return !FUSED ? 1.0 : k == f.k[0] ? f.w[0] : k == f.k[1] ? f.w[1] : 1.0;
    };
#pragma unroll
    for (int u = 0; u < kFoldUnits; u++) {
        const fold_pair p = v[u % kFoldAhead];
        const int j = u + kFoldAhead;
        const double *s = j < kFoldUnits ? here + 8 * j : next + 8 * (j - kFoldUnits);
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(p.x, second(8 * u + q), acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        v[u % kFoldAhead] = fold_pair{s[0], s[4]};
        __builtin_amdgcn_sched_barrier(0);
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(p.y, second(8 * u + 4 + q), acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// sum over k < Kc of x[k] w[k] in the reference's order, by one whole
// wavefront; every lane returns the sum.  buf: kFoldLds doubles of LDS, owned
// by this wavefront; x, w and buf are 16-byte aligned, and x[Kc], w[Kc] can be
// read where Kc is odd.
//
// The lanes form a block's products together (coalesced 16-byte loads three
// blocks ahead, the products one block ahead in LDS); every row of the MFMA
// then takes the same four positions.  Bound: the chain of MFMAs.
// Positions past Kc add +0.0, which changes no sum that started from +0.0.
__device__ __forceinline__ double wave_fold(const double *x, const double *w, int Kc, int G, double *buf)
{
    const int lane = threadIdx.x & 63;
    const int nblk = (Kc + kFoldBlock - 1) / kFoldBlock;
    const int klast = (Kc - 1) & ~1;
    const bool godd = (G & 1) != 0;
    struct Pairs {
        fold_pair x, w;
    };
    auto load = [&](int b, Pairs &v) __attribute__((always_inline)) {
        const int k = min(b * kFoldBlock + 2 * lane, klast);
        v.x = *reinterpret_cast<const fold_pair *>(x + k);
        v.w = *reinterpret_cast<const fold_pair *>(w + k);
    };
    auto publish = [&](int b, const Pairs &v) __attribute__((always_inline)) {
        const int k = b * kFoldBlock + 2 * lane;
        fold_pair p = v.x * v.w;
        if (godd) {  // a fused element's first factor in place of its product
            if (k == G - 1 || k == Kc - 1) p.x = v.x.x;
            if (k + 1 == G - 1 || k + 1 == Kc - 1) p.y = v.x.y;
        }
        if (k >= Kc) p.x = 0.0;
        if (k + 1 >= Kc) p.y = 0.0;
        reinterpret_cast<fold_pair *>(buf + (b & 1) * kFoldBlock)[lane] = p;
    };
    // the lanes of one wavefront run in step and LDS keeps their order: only
    // the compiler has to be held
    auto settle = []() __attribute__((always_inline)) { asm volatile("" ::: "memory"); };
    FoldFused f = {{-1, -1}, {1.0, 1.0}};
    if (godd) {
        f.w[0] = w[G - 1];
        f.w[1] = w[Kc - 1];
    }
    Pairs p0, p1;
    load(0, p0);
    load(1, p1);
    publish(0, p0);
    load(2, p0);
    settle();
    const double *even = buf + (lane >> 4), *odd = even + kFoldBlock;
    fold_pair v[kFoldAhead];
#pragma unroll
    for (int u = 0; u < kFoldAhead; u++) v[u] = fold_pair{even[8 * u], even[8 * u + 4]};
    double acc = 0.0;
    auto block = [&](int b, Pairs &p, const double *here, const double *next) __attribute__((always_inline)) {
        publish(b + 1, p);
        load(b + 3, p);
        settle();
        f.k[0] = godd ? G - 1 - b * kFoldBlock : -1;
        f.k[1] = godd ? Kc - 1 - b * kFoldBlock : -1;
        const bool fused = (f.k[0] >= 0 && f.k[0] < kFoldBlock) || (f.k[1] >= 0 && f.k[1] < kFoldBlock);
        if (fused) fold_block<true>(acc, v, here, next, f);
        else fold_block<false>(acc, v, here, next, f);
        settle();  // the buffer of this block is refilled in the next turn
    };
    for (int b = 0;; b += 2) {
        block(b, p1, even, odd);
        if (b + 1 >= nblk) break;
        block(b + 1, p0, odd, even);
        if (b + 2 >= nblk) break;
    }
    return acc;
}

// ---- rounded-product folds of K rows with one member (bdsf contraction)

// Units of K in flight (one 16-byte load each) and LDS of a wavefront: two
// blocks of the member's row.
constexpr int kFoldRing = kFoldUnits;
constexpr int kFoldTaskLds = 2 * kFoldBlock;

// One block of a fold_task: kr holds its K units and is refilled with the next
// block's; sr holds the member's units about to be used, p the current unit's
// products.
template <bool FUSED>
__device__ __forceinline__ void fold_units(double &acc, fold_pair &p, fold_pair (&kr)[kFoldRing],
                                           fold_pair (&sr)[kFoldAhead], const fold_pair *&ka, const double *here,
                                           const double *next, int fused)
{
    const int q = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int i = 0; i < kFoldUnits; i++) {
        // a fused element goes into the MFMA by its factors
        const fold_pair k = kr[i], s = sr[i % kFoldAhead];
        const bool f0 = FUSED && 8 * i + q == fused, f1 = FUSED && 8 * i + 4 + q == fused;
        const int j = i + kFoldAhead;
        const double *t = j < kFoldUnits ? here + 8 * j : next + 8 * (j - kFoldUnits);
        const fold_pair kn = kr[(i + 1) % kFoldRing], sn = sr[(i + 1) % kFoldAhead];
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(f0 ? k.x : p.x, f0 ? s.x : 1.0, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        sr[i % kFoldAhead] = fold_pair{t[0], t[4]};
        p.x = kn.x * sn.x;
        __builtin_amdgcn_sched_barrier(0);
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(f1 ? k.y : p.y, f1 ? s.y : 1.0, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        kr[i] = ka[i * 64];
        p.y = kn.y * sn.y;
        __builtin_amdgcn_sched_barrier(0);
    }
    ka += kFoldUnits * 64;
}

// Model ISF of one member at 16 timeslices on one wavefront as the
// detailed-balance (bdsf) reference build sums it (its loop inlines
// matrix_multiply_LxM_by_MxN, deac.cpp:110-118, 1389-1390, as a fold of
// rounded products, the last of an odd count fused).  Lane l returns timeslice
// 4 ((l >> 2) & 3) + (l >> 4).  ktile: the tau block's K in the chains' operand
// order, kFoldRing units past its end readable; row: the member's; nblk: blocks
// of 128 positions; buf: kFoldTaskLds doubles of LDS of this wavefront.
//
// Bound: the chain of MFMAs, one per 4 positions, and the eight instructions
// per 8 positions around them.  The four columns of an MFMA repeat each other
// (a product belongs to one member): 4 members per wavefront on v_mul_f64 and
// v_add_f64 took 36 us for 4096 positions, this 13.
__device__ __forceinline__ double fold_task(const double *ktile, const double *row, int nblk, int Kc, bool odd,
                                            double *buf)
{
    const int lane = threadIdx.x & 63;
    const fold_pair *ka = reinterpret_cast<const fold_pair *>(ktile) + lane;
    auto load = [&](int b) __attribute__((always_inline)) {
        return *reinterpret_cast<const fold_pair *>(row + min(b, nblk - 1) * kFoldBlock + 2 * lane);
    };
    auto put = [&](int b, const fold_pair &v) __attribute__((always_inline)) {
        reinterpret_cast<fold_pair *>(buf + (b & 1) * kFoldBlock)[lane] = v;
    };
    auto settle = []() __attribute__((always_inline)) { asm volatile("" ::: "memory"); };
    const double *even = buf + (lane >> 4), *oddb = even + kFoldBlock;
    fold_pair s0 = load(0), s1 = load(1);
    fold_pair kr[kFoldRing], sr[kFoldAhead];
#pragma unroll
    for (int i = 0; i < kFoldRing; i++) kr[i] = ka[i * 64];
    ka += kFoldRing * 64;
    __builtin_amdgcn_sched_barrier(0);
    put(0, s0);
    s0 = load(2);
    settle();
#pragma unroll
    for (int j = 0; j < kFoldAhead; j++) sr[j] = fold_pair{even[8 * j], even[8 * j + 4]};
    fold_pair p = kr[0] * sr[0];
    double acc = 0.0;
    const int last = odd ? Kc - 1 : -1;
    for (int b = 0;; b += 2) {
        put(b + 1, s1);
        s1 = load(b + 3);
        settle();
        int fused = last - b * kFoldBlock;
        if (fused >= 0 && fused < kFoldBlock) fold_units<true>(acc, p, kr, sr, ka, even, oddb, fused);
        else fold_units<false>(acc, p, kr, sr, ka, even, oddb, -1);
        settle();
        if (b + 1 >= nblk) break;
        put(b + 2, s0);
        s0 = load(b + 4);
        settle();
        fused = last - (b + 1) * kFoldBlock;
        if (fused >= 0 && fused < kFoldBlock) fold_units<true>(acc, p, kr, sr, ka, oddb, even, fused);
        else fold_units<false>(acc, p, kr, sr, ka, oddb, even, -1);
        settle();
        if (b + 2 >= nblk) break;
    }
    return acc;
}

}  // namespace

}  // namespace deac
