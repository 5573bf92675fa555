// gfx950 kernels of the operand layouts.  Each is one pass over rows that are
// in L2 or coming from HBM; on the host the same gathers took most of
// deac_model_isf (1024 genomes of 8192 positions: 50 of 90 ms) and of an
// engine's or a batch's first mixed-precision run.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pack_kernels.hpp"

namespace deac {

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ size_t grid_thread() { return static_cast<size_t>(blockIdx.x) * kThreads + threadIdx.x; }
__device__ __forceinline__ size_t grid_threads() { return static_cast<size_t>(gridDim.x) * kThreads; }

__device__ __forceinline__ double value(const PackArgs &a, int row, int k)
{
    const double v = a.rows[static_cast<size_t>(row) * a.L + k];
    return a.ex ? ldexp(v, -a.ex[row]) : v;
}

template <class Out>
__global__ __launch_bounds__(kThreads) void pack_kernel(PackArgs a, Out pad, Out *out)
{
    const size_t slots = static_cast<size_t>(a.tiles) * a.Kb * 64;
    for (size_t s = grid_thread(); s < slots; s += grid_threads()) {
        const int l = static_cast<int>(s & 63);
        const int kb = static_cast<int>((s >> 6) % a.Kb), row = static_cast<int>((s >> 6) / a.Kb) * 16 + (l & 15);
        const int k = 4 * kb + (l >> 4);
        out[s] = row < a.n && k < a.L ? static_cast<Out>(value(a, row, k)) : pad;
    }
}

// Round-to-nearest-even FP32 -> bfloat16 bits (finite inputs).
__device__ __forceinline__ uint32_t bf16_rne(float x)
{
    uint32_t u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}

// x = hi + lo: hi = bf16(x), lo = bf16(x - hi), the remainder taken in FP32.
__global__ __launch_bounds__(kThreads) void pack_bf16x3_kernel(PackArgs a, uint4 *hi, uint4 *lo)
{
    const size_t slots = static_cast<size_t>(a.tiles) * a.Kb * 64;
    for (size_t s = grid_thread(); s < slots; s += grid_threads()) {
        const int l = static_cast<int>(s & 63);
        const int kb = static_cast<int>((s >> 6) % a.Kb), row = static_cast<int>((s >> 6) / a.Kb) * 16 + (l & 15);
        uint32_t h[4] = {0, 0, 0, 0}, r[4] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int k = 32 * kb + 8 * (l >> 4) + e;
            if (row < a.n && k < a.L) {
                const float f = static_cast<float>(value(a, row, k));
                const uint32_t hb = bf16_rne(f), lb = bf16_rne(f - __uint_as_float(hb << 16));
                h[e >> 1] |= hb << (16 * (e & 1));
                r[e >> 1] |= lb << (16 * (e & 1));
            }
        }
        const uint4 hv = make_uint4(h[0], h[1], h[2], h[3]), lv = make_uint4(r[0], r[1], r[2], r[3]);
        if (lo) {
            hi[s] = hv;
            lo[s] = lv;
        } else {
            hi[2 * s] = hv;
            hi[2 * s + 1] = lv;
        }
    }
}

__global__ __launch_bounds__(kThreads) void pack_units_kernel(PackArgs a, float4 *out)
{
    const size_t slots = static_cast<size_t>(a.tiles) * a.Kb * 64;
    for (size_t s = grid_thread(); s < slots; s += grid_threads()) {
        const int l = static_cast<int>(s & 63);
        const int kb = static_cast<int>((s >> 6) % a.Kb), row = static_cast<int>((s >> 6) / a.Kb) * 16 + (l & 15);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = 16 * kb + 4 * e + (l >> 4);
            v[e] = row < a.n && k < a.L ? static_cast<float>(value(a, row, k)) : 0.0f;
        }
        out[s] = make_float4(v[0], v[1], v[2], v[3]);
    }
}

__global__ __launch_bounds__(kThreads) void pack_transposed_kernel(PackArgs a, int width, int positions, double *out)
{
    // consecutive threads take consecutive positions of one row
    const size_t total = static_cast<size_t>(width) * positions;
    for (size_t i = grid_thread(); i < total; i += grid_threads()) {
        const int row = static_cast<int>(i / positions), k = static_cast<int>(i % positions);
        out[static_cast<size_t>(k) * width + row] = row < a.n && k < a.L ? value(a, row, k) : 0.0;
    }
}

unsigned grid_for(size_t work)
{
    return static_cast<unsigned>(std::clamp<size_t>((work + kThreads - 1) / kThreads, 1, 16384));
}

size_t slots_of(const PackArgs &a) { return static_cast<size_t>(a.tiles) * a.Kb * 64; }

}  // namespace

hipError_t launch_pack_fp64(const PackArgs &a, double pad, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(pack_kernel<double>, dim3(grid_for(slots_of(a))), dim3(kThreads), 0, s, a, pad, out);
    return hipGetLastError();
}

hipError_t launch_pack_fp32(const PackArgs &a, float *out, hipStream_t s)
{
    hipLaunchKernelGGL(pack_kernel<float>, dim3(grid_for(slots_of(a))), dim3(kThreads), 0, s, a, 0.0f, out);
    return hipGetLastError();
}

hipError_t launch_pack_bf16x3(const PackArgs &a, void *hi, void *lo, hipStream_t s)
{
    hipLaunchKernelGGL(pack_bf16x3_kernel, dim3(grid_for(slots_of(a))), dim3(kThreads), 0, s, a,
                       static_cast<uint4 *>(hi), static_cast<uint4 *>(lo));
    return hipGetLastError();
}

hipError_t launch_pack_fp32_units(const PackArgs &a, float *out, hipStream_t s)
{
    hipLaunchKernelGGL(pack_units_kernel, dim3(grid_for(slots_of(a))), dim3(kThreads), 0, s, a,
                       reinterpret_cast<float4 *>(out));
    return hipGetLastError();
}

hipError_t launch_pack_transposed(const PackArgs &a, int width, int positions, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(pack_transposed_kernel, dim3(grid_for(static_cast<size_t>(width) * positions)), dim3(kThreads),
                       0, s, a, width, positions, out);
    return hipGetLastError();
}

}  // namespace deac
