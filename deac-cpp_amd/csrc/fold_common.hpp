// Sequential folds on one wavefront, shared by the kernels that need the
// reference's non-fused dot product (matrix_multiply_MxN_by_Nx1 as its build
// inlines it, deac.cpp:102-108): rounded products added one at a time in
// position order, the last element of each sign fused when the genome length
// is odd.
#pragma once

#include <hip/hip_runtime.h>

namespace deac {

namespace {

// Positions per block of wave_fold: two per lane.
constexpr int kFoldBlock = 128;
// LDS of one wave_fold: two blocks of products.
constexpr int kFoldLds = 2 * kFoldBlock;

typedef double fold_pair __attribute__((ext_vector_type(2)));

// sum over k of x[k] w[k] in the reference's order, by one whole wavefront;
// every lane returns the sum.  buf: kFoldLds doubles of LDS, 16-byte aligned,
// owned by this wavefront.  x and w: 16-byte aligned, Kc readable positions.
//
// Bound: the chain of dependent adds (2.5 ns each).  The lanes form a block's
// products together (coalesced 16-byte loads, one block ahead of the adds in
// LDS and two in registers), then every lane adds the block's products in
// order from broadcast LDS reads.  One lane loading 16 positions at a time
// from memory, the products in the chain, took 170 ns per position.
// Positions past Kc add +0.0, which changes no sum that started from +0.0.
__device__ __forceinline__ double wave_fold(const double *x, const double *w, int Kc, int G, double *buf)
{
    const int lane = threadIdx.x & 63;
    const int nblk = (Kc + kFoldBlock - 1) / kFoldBlock;
    const bool godd = (G & 1) != 0;
    auto load = [&](int b, fold_pair &xv, fold_pair &wv) __attribute__((always_inline)) {
        const int k = b * kFoldBlock + 2 * lane;
        xv = fold_pair{0.0, 0.0};
        wv = fold_pair{0.0, 0.0};
        if (k + 1 < Kc) {
            xv = *reinterpret_cast<const fold_pair *>(x + k);
            wv = *reinterpret_cast<const fold_pair *>(w + k);
        } else if (k < Kc) {
            xv.x = x[k];
            wv.x = w[k];
        }
    };
    auto publish = [&](int b, const fold_pair &xv, const fold_pair &wv) __attribute__((always_inline)) {
        reinterpret_cast<fold_pair *>(buf + (b & 1) * kFoldBlock)[lane] = fold_pair{xv.x * wv.x, xv.y * wv.y};
    };
    auto settle = []() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    fold_pair x1, w1;
    load(0, x1, w1);
    publish(0, x1, w1);
    load(1, x1, w1);
    double acc = 0.0;
    for (int b = 0; b < nblk; b++) {
        publish(b + 1, x1, w1);
        load(b + 2, x1, w1);
        settle();
        const double *p = buf + (b & 1) * kFoldBlock;
        const int k0 = b * kFoldBlock;
        const bool fused = godd && ((k0 <= G - 1 && G - 1 < k0 + kFoldBlock) || k0 + kFoldBlock >= Kc);
        if (!fused) {
#pragma unroll
            for (int u = 0; u < kFoldBlock; u += 2) {
                const fold_pair v = *reinterpret_cast<const fold_pair *>(p + u);
                acc = acc + v.x;
                acc = acc + v.y;
            }
        } else {
            const int n = min(kFoldBlock, Kc - k0);
            for (int u = 0; u < n; u++) {
                const int k = k0 + u;
                if (k == G - 1 || k == Kc - 1) acc = fma(x[k], w[k], acc);
                else acc = acc + p[u];
            }
        }
        settle();  // this block's buffer is refilled in the next turn
    }
    return acc;
}

}  // namespace

}  // namespace deac
