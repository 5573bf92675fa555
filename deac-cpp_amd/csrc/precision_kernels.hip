// Model ISF E = K.S of a stack of genomes at three K.S precisions, on the
// gfx950 matrix cores (the precision sweep of the K.S contraction):
//
//   FP64    v_mfma_f64_16x16x4f64, one accumulator per output tile over the
//           whole genome in ascending position order: each output element is
//           the reference's sequential FMA chain (deac.cpp:110-118), bit for
//           bit, as in the batch kernel;
//   FP32    K (scaled per tau row by a power of two) and S rounded to FP32,
//           v_mfma_f32_16x16x4f32 with FP32 accumulation over slices of the
//           genome, slices summed in FP32;
//   BF16x3  K = Kh + Kl and S = Sh + Sl split into bfloat16 pairs,
//           Kl.Sh + Kh.Sl + Kh.Sh per 32 positions on v_mfma_f32_16x16x32_bf16,
//           FP32 accumulation as above.
//
// Operands arrive in MFMA lane order (pack_kernels.hip), one coalesced
// load per wave and k-block:
//   16x16x4  (FP64, FP32): A[mt][kb][lane] = K[16 mt + lane%16][4 kb + lane/16],
//                          B[nt][kb][lane] = S[16 nt + lane%16][4 kb + lane/16];
//   16x16x32 (BF16):       A[mt][kb][lane][e] = K[16 mt + lane%16][32 kb + 8 (lane/16) + e],
//                          B likewise with S.
// Outputs: FP64 E[n][t] directly; FP32/BF16 partial tiles [slice][Npad][Mpad]
// reduced in slice order by reduce_slices.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "precision_kernels.hpp"

namespace deac {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int kDepth = kSweepDepth;      // k-blocks in flight, 16x16x4 operands
constexpr int kDepth16 = kSweepDepth16;  // k-blocks in flight, 16x16x32 operands

// One wave per (tau tile, genome tile); the four waves of a workgroup take
// four genome tiles.
__global__ __launch_bounds__(256) void ks_fp64_kernel(const double *__restrict__ A, const double *__restrict__ B,
                                                      double *__restrict__ E, int T, int N, int Mt, int Nt, int Kb,
                                                      const int *halt)
{
    if (halt && *halt) return;
    const int lane = threadIdx.x & 63;
    const int mt = blockIdx.x, nt = blockIdx.y * 4 + static_cast<int>(threadIdx.x >> 6);
    if (mt >= Mt || nt >= Nt) return;
    const double *a = A + static_cast<size_t>(mt) * Kb * 64 + lane;
    const double *b = B + static_cast<size_t>(nt) * Kb * 64 + lane;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    // operands of the next kDepth k-blocks in flight (Kb is a multiple of
    // kDepth; the refill past the end re-reads the last block, unused)
    double ra[kDepth], rb[kDepth];
#pragma unroll
    for (int i = 0; i < kDepth; i++) {
        ra[i] = a[static_cast<size_t>(i) * 64];
        rb[i] = b[static_cast<size_t>(i) * 64];
    }
    for (int kb = 0; kb < Kb; kb += kDepth) {
#pragma unroll
        for (int i = 0; i < kDepth; i++) {
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ra[i], rb[i], acc, 0, 0, 0);
            const size_t nk = static_cast<size_t>(min(kb + i + kDepth, Kb - 1)) * 64;
            ra[i] = a[nk];
            rb[i] = b[nk];
        }
    }
    // lane l holds rows 4v + l/16 of the tile, column l%16
    const int n = nt * 16 + (lane & 15);
    for (int v = 0; v < 4; v++) {
        const int t = mt * 16 + 4 * v + (lane >> 4);
        if (t < T && n < N) E[static_cast<size_t>(n) * T + t] = acc[v];
    }
}

__device__ __forceinline__ void store_partial(float *part, int slice, int Mpad, int Npad, int mt, int nt, int lane,
                                              f4 acc)
{
    // lane l holds rows 4 (l/16) + v of the tile, column l%16
    float *p = part + (static_cast<size_t>(slice) * Npad + nt * 16 + (lane & 15)) * Mpad + mt * 16 + 4 * (lane >> 4);
    *reinterpret_cast<f4 *>(p) = acc;
}

// What one wavefront contracts: MB tau tiles x NB genome tiles over one slice.  The workgroups (one wavefront each) of an XCD, which they go to in
// turn, take a range of (slice, genome tiles, tau tiles), tau tiles fastest,
// so that a slice's genomes come through one L2.
constexpr int kXcds = 8;
template <int MB, int NB>
struct SliceTask {
    int slice, mt[MB], nt[NB];
    bool mine;
    __device__ __forceinline__ SliceTask(int Mt, int Nt, int slices)
    {
        const int mp = (Mt + MB - 1) / MB, ng = (Nt + NB - 1) / NB;
        const int task = blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds;
        slice = task / (mp * ng);
        mine = slice < slices;
        // past the last tile: the last one again
        for (int m = 0; m < MB; m++) mt[m] = min(task % mp * MB + m, Mt - 1);
        for (int n = 0; n < NB; n++) nt[n] = min(task / mp % ng * NB + n, Nt - 1);
    }
    __device__ __forceinline__ void store(float *part, int Mt, int Nt, const f4 (&acc)[MB][NB]) const
    {
        for (int m = 0; m < MB; m++)
            for (int n = 0; n < NB; n++)
                if ((m == 0 || mt[m] != mt[m - 1]) && (n == 0 || nt[n] != nt[n - 1]))
                    store_partial(part, slice, Mt * 16, Nt * 16, mt[m], nt[n], threadIdx.x, acc[m][n]);
    }
};

// FP32: two tau tiles per wavefront or one, whichever gives the fullest SIMD
// fewer tiles (one reads more, 320 bytes per MFMA instead of 192 at NB = 4): T =
// 257, 64 genomes, 114 slices make 1026 wavefronts of two, 22.8 us, or 1938 of
// one, 16.0.
constexpr int kSimds = 1024;
inline int slice_tasks(int MB, int NB, int Mt, int Nt, int slices)
{
    return slices * ((Mt + MB - 1) / MB) * ((Nt + NB - 1) / NB);
}
inline bool two_tau_tiles(int NB, int Mt, int Nt, int slices)
{
    auto fullest = [&](int MB) { return (slice_tasks(MB, NB, Mt, Nt, slices) + kSimds - 1) / kSimds * MB; };
    return fullest(2) <= fullest(1);
}

// Bound: the matrix cores (32 cycles per MFMA) and the operands from L2.  T =
// 257, 64 genomes of 32768 positions: 16.0 us (71 TFLOP/s); one output tile per
// wavefront (512 bytes per MFMA) 24.8.
template <int MB, int NB>
__global__ __launch_bounds__(64) void ks_fp32_kernel(const float *__restrict__ A, const float *__restrict__ B,
                                                     float *__restrict__ part, int Mt, int Nt, int Kb, int kb_per_slice,
                                                     int slices, const int *halt)
{
    if (halt && *halt) return;
    const SliceTask<MB, NB> t(Mt, Nt, slices);
    if (!t.mine) return;
    // a slice's length is a multiple of kDepth
    const int kb0 = t.slice * kb_per_slice, turns = (min(kb0 + kb_per_slice, Kb) - kb0) / kDepth;
    const float *a[MB], *b[NB];
    for (int m = 0; m < MB; m++) a[m] = A + (static_cast<size_t>(t.mt[m]) * Kb + kb0) * 64 + threadIdx.x;
    for (int n = 0; n < NB; n++) b[n] = B + (static_cast<size_t>(t.nt[n]) * Kb + kb0) * 64 + threadIdx.x;
    f4 acc[MB][NB] = {};
    float ra[kDepth][MB], rb[kDepth][NB];
    // (the scheduler would gather the loads in front of their use)
    auto load = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MB; m++) ra[i][m] = a[m][i * 64];
#pragma unroll
        for (int n = 0; n < NB; n++) rb[i][n] = b[n][i * 64];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto advance = [&]() __attribute__((always_inline)) {
        for (int m = 0; m < MB; m++) a[m] += kDepth * 64;
        for (int n = 0; n < NB; n++) b[n] += kDepth * 64;
    };
    auto contract = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int m = 0; m < MB; m++)
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[i][m], rb[i][n], acc[m][n], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < kDepth; i++) load(i);
    for (int turn = 1; turn < turns; turn++) {
        advance();
#pragma unroll
        for (int i = 0; i < kDepth; i++) {
            contract(i);
            load(i);
        }
    }
#pragma unroll
    for (int i = 0; i < kDepth; i++) contract(i);
    t.store(part, Mt, Nt, acc);
}

template <int MB, int NB>
__global__ __launch_bounds__(64) void ks_bf16x3_kernel(const bf8 *__restrict__ Ah, const bf8 *__restrict__ Al,
                                                       const bf8 *__restrict__ Bh, const bf8 *__restrict__ Bl,
                                                       float *__restrict__ part, int Mt, int Nt, int Kb,
                                                       int kb_per_slice, int slices, const int *halt)
{
    if (halt && *halt) return;
    const SliceTask<MB, NB> t(Mt, Nt, slices);
    if (!t.mine) return;
    // a slice's length is a multiple of kDepth16
    const int kb0 = t.slice * kb_per_slice, turns = (min(kb0 + kb_per_slice, Kb) - kb0) / kDepth16;
    size_t a[MB], b[NB];
    for (int m = 0; m < MB; m++) a[m] = (static_cast<size_t>(t.mt[m]) * Kb + kb0) * 64 + threadIdx.x;
    for (int n = 0; n < NB; n++) b[n] = (static_cast<size_t>(t.nt[n]) * Kb + kb0) * 64 + threadIdx.x;
    f4 acc[MB][NB] = {};
    bf8 ah[kDepth16][MB], al[kDepth16][MB], bh[kDepth16][NB], bl[kDepth16][NB];
    auto load = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MB; m++) ah[i][m] = Ah[a[m] + i * 64], al[i][m] = Al[a[m] + i * 64];
#pragma unroll
        for (int n = 0; n < NB; n++) bh[i][n] = Bh[b[n] + i * 64], bl[i][n] = Bl[b[n] + i * 64];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto advance = [&]() __attribute__((always_inline)) {
        for (int m = 0; m < MB; m++) a[m] += kDepth16 * 64;
        for (int n = 0; n < NB; n++) b[n] += kDepth16 * 64;
    };
    // one product of the three for every tile, small terms first
    auto product = [&](const bf8 (&x)[MB], const bf8 (&y)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int m = 0; m < MB; m++)
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[m], y[n], acc[m][n], 0, 0, 0);
    };
    auto contract = [&](int i) __attribute__((always_inline)) {
        product(al[i], bh[i]);
        product(ah[i], bl[i]);
        product(ah[i], bh[i]);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < kDepth16; i++) load(i);
    for (int turn = 1; turn < turns; turn++) {
        advance();
#pragma unroll
        for (int i = 0; i < kDepth16; i++) {
            contract(i);
            load(i);
        }
    }
#pragma unroll
    for (int i = 0; i < kDepth16; i++) contract(i);
    t.store(part, Mt, Nt, acc);
}

// E32[n][m] = sum over slices (in order, FP32) of part[slice][n][m]
__global__ __launch_bounds__(256) void reduce_slices_kernel(const float *__restrict__ part, float *__restrict__ out,
                                                            int slices, size_t mn)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= mn) return;
    float s = 0.0f;
#pragma unroll 8
    for (int k = 0; k < slices; k++) s += part[static_cast<size_t>(k) * mn + i];
    out[i] = s;
}

}  // namespace

hipError_t launch_ks_fp64(const double *A, const double *B, double *E, int T, int N, int Mt, int Nt, int Kb,
                          hipStream_t s, hipEvent_t start, hipEvent_t stop, const int *halt)
{
    hipExtLaunchKernelGGL(ks_fp64_kernel, dim3(Mt, (Nt + 3) / 4), dim3(256), 0, s, start, stop, 0, A, B, E, T, N, Mt,
                          Nt, Kb, halt);
    return hipGetLastError();
}

hipError_t launch_ks_fp32(const float *A, const float *B, float *part, int Mt, int Nt, int Kb, int kb_per_slice,
                          int slices, hipStream_t s, hipEvent_t start, hipEvent_t stop, const int *halt)
{
    auto go = [&](auto kernel, int MB, int NB) {
        const unsigned grid = (slice_tasks(MB, NB, Mt, Nt, slices) + kXcds - 1) / kXcds * kXcds;
        hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, s, start, stop, 0, A, B, part, Mt, Nt, Kb, kb_per_slice,
                              slices, halt);
        return hipGetLastError();
    };
    const bool two = two_tau_tiles(std::min(Nt, 4), Mt, Nt, slices);
    if (Nt == 1) return two ? go(ks_fp32_kernel<2, 1>, 2, 1) : go(ks_fp32_kernel<1, 1>, 1, 1);
    if (Nt == 2) return two ? go(ks_fp32_kernel<2, 2>, 2, 2) : go(ks_fp32_kernel<1, 2>, 1, 2);
    if (Nt == 3) return two ? go(ks_fp32_kernel<2, 3>, 2, 3) : go(ks_fp32_kernel<1, 3>, 1, 3);
    return two ? go(ks_fp32_kernel<2, 4>, 2, 4) : go(ks_fp32_kernel<1, 4>, 1, 4);
}

hipError_t launch_ks_bf16x3(const void *Ah, const void *Al, const void *Bh, const void *Bl, float *part, int Mt,
                            int Nt, int Kb, int kb_per_slice, int slices, hipStream_t s, hipEvent_t start,
                            hipEvent_t stop, const int *halt)
{
    auto go = [&](auto kernel, int MB, int NB) {
        const unsigned grid = (slice_tasks(MB, NB, Mt, Nt, slices) + kXcds - 1) / kXcds * kXcds;
        hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, s, start, stop, 0, static_cast<const bf8 *>(Ah),
                              static_cast<const bf8 *>(Al), static_cast<const bf8 *>(Bh), static_cast<const bf8 *>(Bl),
                              part, Mt, Nt, Kb, kb_per_slice, slices, halt);
        return hipGetLastError();
    };
    // (two genome tiles at most: their operands of four k-blocks take 128
    // registers.  Two tau tiles always: one, where it fills the SIMDs better,
    // reads 6 KB per three MFMAs instead of 4, 30.4 and 32.0 ms for 600
    // generations at T = 257 and 64 genomes of 32768 positions.)
    return Nt == 1 ? go(ks_bf16x3_kernel<2, 1>, 2, 1) : go(ks_bf16x3_kernel<2, 2>, 2, 2);
}

hipError_t launch_reduce_slices(const float *part, float *out, int slices, size_t mn, hipStream_t s, hipEvent_t start,
                                hipEvent_t stop)
{
    const unsigned blocks = static_cast<unsigned>((mn + 255) / 256);
    hipExtLaunchKernelGGL(reduce_slices_kernel, dim3(blocks), dim3(256), 0, s, start, stop, 0, part, out, slices, mn);
    return hipGetLastError();
}

}  // namespace deac
