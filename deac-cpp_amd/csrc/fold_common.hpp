// Sequential folds on one wavefront, shared by the kernels that need the
// reference's non-fused dot product (matrix_multiply_MxN_by_Nx1 as its build
// inlines it, deac.cpp:102-108): rounded products added one at a time in
// position order, the last element of each sign fused when the genome length
// is odd.
#pragma once

#include <hip/hip_runtime.h>

namespace deac {

namespace {

// Positions per block of wave_fold (two per lane), LDS of one wave_fold (two
// blocks of products), and product pairs read ahead of the adds.
constexpr int kFoldBlock = 128;
constexpr int kFoldLds = 2 * kFoldBlock;
constexpr int kFoldAhead = 16;

typedef double fold_pair __attribute__((ext_vector_type(2)));

// The fused elements of a fold: positions within the current block, values.
struct FoldFused {
    int k[2];
    double x[2], w[2];
};

// Adds one block's products in order; v holds the pairs about to be added and
// is refilled kFoldAhead pairs on (past the block's end from the next one).
template <bool FUSED>
__device__ __forceinline__ void fold_block(double &acc, fold_pair (&v)[kFoldAhead], const double *here,
                                           const double *next, const FoldFused &f)
{
#pragma unroll
    for (int u = 0; u < kFoldBlock / 2; u++) {
        const fold_pair p = v[u % kFoldAhead];
        const int j = u + kFoldAhead;
        v[u % kFoldAhead] = *reinterpret_cast<const fold_pair *>(j < kFoldBlock / 2 ? here + 2 * j
                                                                                    : next + (2 * j - kFoldBlock));
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const double sum = acc + (e ? p.y : p.x);
            if (FUSED) {
                const int k = 2 * u + e;
                const double f0 = fma(f.x[0], f.w[0], acc), f1 = fma(f.x[1], f.w[1], acc);
                acc = k == f.k[0] ? f0 : k == f.k[1] ? f1 : sum;
            } else {
                acc = sum;
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the adds
    }
}

// sum over k < Kc of x[k] w[k] in the reference's order, by one whole
// wavefront; every lane returns the sum.  buf: kFoldLds doubles of LDS, owned
// by this wavefront; x, w and buf are 16-byte aligned, and x[Kc], w[Kc] can be
// read where Kc is odd.
//
// Bound: the chain of dependent adds (2.5 ns each).  The lanes form a block's
// products together (coalesced 16-byte loads two blocks ahead, the products
// one block ahead in LDS), then every lane adds them in order from broadcast
// LDS reads 16 pairs ahead.  4096 positions: 64 us with the reads 3 pairs
// ahead, 800 us with one lane loading from memory.
// Positions past Kc add +0.0, which changes no sum that started from +0.0.
__device__ __forceinline__ double wave_fold(const double *x, const double *w, int Kc, int G, double *buf)
{
    const int lane = threadIdx.x & 63;
    const int nblk = (Kc + kFoldBlock - 1) / kFoldBlock;
    const int klast = (Kc - 1) & ~1;
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
        if (k >= Kc) p.x = 0.0;
        if (k + 1 >= Kc) p.y = 0.0;
        reinterpret_cast<fold_pair *>(buf + (b & 1) * kFoldBlock)[lane] = p;
    };
    // the lanes of one wavefront run in step and LDS keeps their order: only
    // the compiler has to be held
    auto settle = []() __attribute__((always_inline)) { asm volatile("" ::: "memory"); };
    const bool godd = (G & 1) != 0;
    FoldFused f = {{-1, -1}, {0.0, 0.0}, {0.0, 0.0}};
    if (godd) {
        f.x[0] = x[G - 1];
        f.w[0] = w[G - 1];
        f.x[1] = x[Kc - 1];
        f.w[1] = w[Kc - 1];
    }
    Pairs p0, p1;
    load(0, p0);
    load(1, p1);
    publish(0, p0);
    load(2, p0);
    settle();
    fold_pair v[kFoldAhead];
#pragma unroll
    for (int u = 0; u < kFoldAhead; u++) v[u] = *reinterpret_cast<const fold_pair *>(buf + 2 * u);
    double acc = 0.0;
    auto block = [&](int b, Pairs &p) __attribute__((always_inline)) {
        publish(b + 1, p);
        load(b + 3, p);
        settle();
        const double *here = buf + (b & 1) * kFoldBlock, *next = buf + (~b & 1) * kFoldBlock;
        f.k[0] = godd ? G - 1 - b * kFoldBlock : -1;
        f.k[1] = godd ? Kc - 1 - b * kFoldBlock : -1;
        const bool fused = (f.k[0] >= 0 && f.k[0] < kFoldBlock) || (f.k[1] >= 0 && f.k[1] < kFoldBlock);
        if (fused) fold_block<true>(acc, v, here, next, f);
        else fold_block<false>(acc, v, here, next, f);
        settle();  // the buffer of this block is refilled in the next turn
    };
    for (int b = 0;; b += 2) {
        block(b, p1);
        if (b + 1 >= nblk) break;
        block(b + 1, p0);
        if (b + 2 >= nblk) break;
    }
    return acc;
}

}  // namespace

}  // namespace deac
