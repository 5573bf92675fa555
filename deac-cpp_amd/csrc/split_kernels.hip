// Split generation loop of the plain engine: one generation of the fused
// evolution kernel (kernels.hip) as a sequence of kernels on one stream, so
// that the model ISF can come from the K.S contraction kernels at any of
// their precisions (precision_kernels.hip) while the trial vectors, chi^2,
// the selection, the statistics and every constraint stay FP64 in the
// reference's order.  Per generation g of a batch (deac.cpp:1145-1572):
//
//   split_trial_kernel    best fitness, statistics, stop test (workgroup 0),
//                         trial vectors into each member's spare buffer
//   split_renorm_*        per-generation renormalization, when enabled
//   split_pack_*          rows into the contraction's operand layout: at FP64,
//                         where the trials are renormalized, and for the
//                         initial fitness (the trial kernel packs the rest)
//   ks_*_kernel           the contraction: FP64 exact chains straight into
//                         the model ISF, or FP32 / BF16x3 genome slices
//   split_fold_kernel     (bdsf at FP64, in place of the two above) the
//                         reference build's rounded-product fold
//   split_moment_kernel   first / third moment rows, when used
//   split_select_kernel   the FP32 slices summed in slice order and scaled back
//                         per tau row into the FP64 model ISF; chi^2 and greedy
//                         selection
//
// A stop found at the top of generation g sets status[0]; every later kernel
// (of this batch and of any batch queued behind it) reads it first and
// returns, leaving the state of the stop.
// The file is compiled with -ffp-contract=off: every fused multiply-add is
// written as fma().
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.hpp"
#include "evolve_common.hpp"
#include "fold_common.hpp"
#include "split_kernels.hpp"

namespace deac {

namespace {

constexpr int kThreads = 256;
constexpr int kWave = 64;

__device__ __forceinline__ bool stopped(const EvoArgs &a) { return a.status[0] != 0; }

__device__ __forceinline__ size_t grid_thread() { return static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; }
__device__ __forceinline__ size_t grid_threads() { return static_cast<size_t>(gridDim.x) * blockDim.x; }

// Top of generation g: best fitness, statistics, stop test (deac.cpp:1145-1166),
// scanned by thread 0 in the reference's order from fit(i).
template <class Fit>
__device__ void top_scan(const EvoArgs &a, int g, Fit fit)
{
    double mn = fit(0);
    for (int i = 0; i < a.P; i++)
        if (fit(i) < mn) mn = fit(i);
    const long ii = (a.iter ? a.iter[0] : a.gen0) + g;
    if (a.track_stats) {
        double s = 0.0;
        for (int i = 0; i < a.P; i++) s += fit(i);
        double q = 0.0;
        const int p4 = a.P & ~3;
        for (int i = 0; i < a.P; i++) {
            const double v = fit(i);
            if (i < p4) q = q + v * v;
            else q = fma(v, v, q);
        }
        a.stats[ii] = s / static_cast<double>(a.P);
        a.stats[a.stats_len + ii] = mn;
        a.stats[2 * a.stats_len + ii] = q / static_cast<double>(a.P);
    }
    if (mn <= a.stop) {
        a.status[0] = 1;
        a.status[1] = g;
    }
}

// Run by every thread of one workgroup: the fitnesses are staged in LDS by
// one coalesced load (up to kTopLds of them), so the sequential scans do not
// wait on a load each.
constexpr int kTopLds = 512;
constexpr int kSelectLds = 4096;  // residuals staged per member at a time (32 KB)

__device__ void top_of_generation(const EvoArgs &a, int g)
{
    __shared__ double fs[kTopLds];
    if (a.P <= kTopLds) {
        for (int i = threadIdx.x; i < a.P; i += blockDim.x) fs[i] = a.fitness[i];
        __syncthreads();
        if (threadIdx.x == 0) top_scan(a, g, [&](int i) { return fs[i]; });
    } else if (threadIdx.x == 0) {
        top_scan(a, g, [&](int i) { return a.fitness[i]; });
    }
}

// Round-to-nearest-even FP32 -> bfloat16 bits (finite inputs).
__device__ __forceinline__ uint32_t bf16_rne(float x)
{
    uint32_t u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}

// x = hi + lo with hi = bf16(x) and lo = bf16(x - hi), the remainder taken in
// FP32, into half e of word e/2.
__device__ __forceinline__ void bf16_split(float x, int e, uint32_t (&hi)[4], uint32_t (&lo)[4])
{
    const uint32_t h = bf16_rne(x);
    const uint32_t r = bf16_rne(x - __uint_as_float(h << 16));
    hi[e >> 1] |= h << (16 * (e & 1));
    lo[e >> 1] |= r << (16 * (e & 1));
}

// Trial vectors of generation g into each member's spare buffer
// (deac.cpp:1261-1308; the padding stays zero), and into the contraction's
// operand B (Bl: the BF16x3 remainders) where its precision is PACK, in the
// layout that the pack kernels below write (they fill what the genomes do not
// reach, once, for the initial fitness).  Workgroup 0 runs the top of the
// generation: it reads only the fitnesses, which no trial writes, and if its
// stop test fires the trials are never selected (every later kernel of the
// generation returns).  The others take 128 positions of a member per wavefront:
// with an operand 16 members each, four per wavefront, so that rows and operand
// are both whole lines; without one a member per wavefront, whose records and
// rows are waited for one after the other.
//
// Bound: memory (40 bytes read, 12 written per position).  64 members of 32768
// positions: 19.3 us; with a kernel of its own for the operand 17.4 and 9.7.
// Without an operand, one member per wavefront and four: 4 members of 600
// positions 3.8 us and 5.5, 20 members 4.2 and 8.7, 64 members of 32768 13.2 and
// 16.7, 300 members of 16384 27.3 and 32.0.
constexpr int kTileMembers = 16;
constexpr int trial_members(int pack) { return pack == DEAC_PRECISION_FP64 ? kThreads / kWave : kTileMembers; }
constexpr int kTileRow = kChunk + 4;  // floats: the operand's readers meet no bank twice
template <int PACK>
__global__ __launch_bounds__(kThreads) void split_trial_kernel(EvoArgs a, int g, void *B, void *Bl, int Kb)
{
    constexpr int kWaves = kThreads / kWave, kMembers = trial_members(PACK), kEach = kMembers / kWaves;
    __shared__ __attribute__((aligned(16))) float tile[PACK == DEAC_PRECISION_FP64 ? 1 : kTileMembers][kTileRow];
    if (stopped(a)) return;
    if (a.iter) g = static_cast<int>(a.iter[1]);
    if (blockIdx.x == 0) {
        // (the selection reads the generation here and moves the counter on)
        if (a.iter && threadIdx.x == 0) a.iter[2] = g;
        top_of_generation(a, g);
        return;
    }
    const int nblk = a.stride / kChunk;
    const int nt = (blockIdx.x - 1) / nblk, b = (blockIdx.x - 1) % nblk;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const Members s = {a.fitness, a.cr_old, a.f_old, a.cur};
    const MemberCtl *ctlg = a.ctl + static_cast<size_t>(g) * a.P;
    const uint64_t *rawg = a.raw + static_cast<size_t>(g) * a.P * a.rstride;
    auto member = [&](int j) { return nt * kMembers + wid + j * kWaves; };
    auto trial = [&](int j) {
        const int i = min(member(j), a.P - 1);
        return Trial(a, s, a.cur, ctlg[i], rawg + static_cast<size_t>(i) * a.rstride, i);
    };
    static_assert(kEach == 1 || kEach == 4);
    const Trial t[4] = {trial(0), trial(1 % kEach), trial(2 % kEach), trial(3 % kEach)};
    Trial::Load v[kEach] = {};
#pragma unroll
    for (int j = 0; j < kEach; j++) t[j].load(b, v[j]);
#pragma unroll
    for (int j = 0; j < kEach; j++) {
        const bool in = member(j) < a.P;
        const dvec2 o = in ? t[j].form(b, v[j]) : dvec2{0.0, 0.0};
        if (in) t[j].store(b, o);
        if constexpr (PACK != DEAC_PRECISION_FP64)
            *reinterpret_cast<float2 *>(&tile[wid + j * kWaves][2 * lane]) =
                make_float2(static_cast<float>(o.x), static_cast<float>(o.y));
    }
    if constexpr (PACK == DEAC_PRECISION_FP32) {
        __syncthreads();
        const int per = kChunk / 4;  // k-blocks of a tile, 64 values each
        float4 *to = reinterpret_cast<float4 *>(static_cast<float *>(B) + (static_cast<size_t>(nt) * Kb + b * per) * 64);
        for (int u = threadIdx.x; u < per * 16; u += kThreads) {
            const int kb = u >> 4, k = 4 * kb + ((u >> 2) & 3), m = 4 * (u & 3);
            if (b * per + kb < Kb) to[u] = make_float4(tile[m][k], tile[m + 1][k], tile[m + 2][k], tile[m + 3][k]);
        }
    } else if constexpr (PACK == DEAC_PRECISION_BF16X3) {
        __syncthreads();
        const int per = kChunk / 32, kb = threadIdx.x / kWave;
        static_assert(kThreads / kWave == kChunk / 32, "a k-block per wavefront");
        uint32_t hi[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};
        const float *x = &tile[lane & 15][32 * kb + 8 * (lane >> 4)];
        for (int e = 0; e < 8; e++) bf16_split(x[e], e, hi, lo);
        if (b * per + kb < Kb) {
            const size_t slot = (static_cast<size_t>(nt) * Kb + b * per + kb) * 64 + lane;
            static_cast<uint4 *>(B)[slot] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
            static_cast<uint4 *>(Bl)[slot] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        }
    }
}

// Per-generation renormalization (deac.cpp:1342-1364): zeroth moment of each
// trial, one thread per member, then every position scaled.
__global__ __launch_bounds__(kWave) void split_renorm_sum_kernel(EvoArgs a)
{
    if (stopped(a)) return;
    const int i = static_cast<int>(grid_thread());
    if (i >= a.P) return;
    const double *src = (a.cur[i] ? a.pop0 : a.pop1) + static_cast<size_t>(i) * a.stride;
    a.mom[i * 4 + 0] = fold_row(src, a.nterm, a.Kc, a.G);
}

__global__ __launch_bounds__(kThreads) void split_renorm_scale_kernel(EvoArgs a)
{
    if (stopped(a)) return;
    const int half = a.stride / 2;
    const size_t items = static_cast<size_t>(a.P) * half;
    for (size_t it = grid_thread(); it < items; it += grid_threads()) {
        const int i = static_cast<int>(it / half);
        const int kp = static_cast<int>(it % half);
        double *dst = (a.cur[i] ? a.pop0 : a.pop1) + static_cast<size_t>(i) * a.stride;
        double2 *p2 = reinterpret_cast<double2 *>(dst + 2 * kp);
        double2 v = *p2;
        const double scale = a.zeroth / a.mom[i * 4 + 0];
        v.x *= scale;
        v.y *= scale;
        *p2 = v;
    }
}

// Genome operand of the contraction, 16x16x4 lane order:
// B[nt][kb][lane] = row(16 nt + lane%16)[4 kb + lane/16], padded with +0.0.
// The rows are the trials, or the current genomes for the initial fitness.
template <class Out>
__global__ __launch_bounds__(kThreads) void split_pack_kernel(EvoArgs a, int init, Out *B, int Nt, int Kb)
{
    if (stopped(a)) return;
    const size_t slots = static_cast<size_t>(Nt) * Kb * 64;
    for (size_t s = grid_thread(); s < slots; s += grid_threads()) {
        const int l = static_cast<int>(s & 63);
        const size_t kb = (s >> 6) % Kb;
        const int n = static_cast<int>((s >> 6) / Kb) * 16 + (l & 15);
        const size_t k = 4 * kb + (l >> 4);
        double v = 0.0;
        if (n < a.P && k < static_cast<size_t>(a.Kc)) v = chain_row(a, n, init != 0)[k];
        B[s] = static_cast<Out>(v);
    }
}

// Genome operand, 16x16x32 lane order, each value split into hi and lo: slot
// (nt, kb, lane) holds positions 32 kb + 8 (lane/16) + e, e = 0..7.
__global__ __launch_bounds__(kThreads) void split_pack_bf16x3_kernel(EvoArgs a, int init, uint4 *Bh, uint4 *Bl,
                                                                      int Nt, int Kb)
{
    if (stopped(a)) return;
    const size_t slots = static_cast<size_t>(Nt) * Kb * 64;
    for (size_t s = grid_thread(); s < slots; s += grid_threads()) {
        const int l = static_cast<int>(s & 63);
        const size_t kb = (s >> 6) % Kb;
        const int n = static_cast<int>((s >> 6) / Kb) * 16 + (l & 15);
        const size_t k0 = 32 * kb + 8 * static_cast<size_t>(l >> 4);
        const double *row = n < a.P ? chain_row(a, n, init != 0) : nullptr;
        uint32_t hi[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};
        for (int e = 0; e < 8; e++) {
            const size_t k = k0 + e;
            if (row && k < static_cast<size_t>(a.Kc)) bf16_split(static_cast<float>(row[k]), e, hi, lo);
        }
        Bh[s] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        Bl[s] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
}

// The trials' model ISF as the detailed-balance (bdsf) reference build sums
// it, straight into emod: one wavefront per member and 16 timeslices.
__global__ __launch_bounds__(kWave) void split_fold_kernel(EvoArgs a, int first)
{
    if (stopped(a)) return;
    __shared__ __attribute__((aligned(16))) double buf[kFoldTaskLds];
    const int task = first + static_cast<int>(blockIdx.x), tb = task % a.TB, i = task / a.TB;
    const int lane = threadIdx.x;
    const double e = fold_task(a.ktile + static_cast<size_t>(tb) * a.stride * kChainTau, chain_row(a, i, false),
                               a.stride / kFoldBlock, a.Kc, (a.G & 1) != 0, buf);
    const int t = tb * kChainTau + 4 * ((lane >> 2) & 3) + (lane >> 4);
    if ((lane & 3) == 0 && t < a.T) a.emod[static_cast<size_t>(i) * a.T + t] = e;
}

// First and third moment rows of the contraction's genomes, one thread per
// (member, moment) (deac.cpp:1420-1476).
__global__ __launch_bounds__(kWave) void split_moment_kernel(EvoArgs a, int init)
{
    if (stopped(a)) return;
    const int idx = static_cast<int>(grid_thread());
    const int i = idx >> 1, rr = idx & 1;
    if (i >= a.P) return;
    const bool used = rr == 0 ? a.use_first : a.use_third;
    if (!used) return;
    const double *row = rr == 0 ? a.fterm : a.tterm;
    a.mom[i * 4 + 1 + rr] = fold_row(chain_row(a, i, init != 0), row, a.Kc, a.G);
}

// Fitness and greedy selection, one workgroup per member (deac.cpp:1539-1572;
// the initial fitness, deac.cpp:957-976).  The workgroup forms the weighted
// residuals; thread 0 adds their squares in tau order, the last one fused when
// T is odd.
//
// MODEL: the model ISF from the contraction's slices part [slices][Npad][Mpad]
// first, emod[i][t] = 2^ex[t] * (sum over slices, in slice order, in FP32).  A
// thread takes four timeslices of a run of slices, which it loads at once; the
// runs then take over each other's sums in order.
//
// Bound: latency: loads, one barrier per run, thread 0's sum.  257 timeslices,
// 114 slices, 64 members: 11.6 us in a kernel trace (15.0 with a test around each
// load); as two kernels, with a part of each sum's loads in flight, 9.2 and 7.5
// by themselves and the gap between them.
constexpr int kSliceRun = 8;  // slices a thread loads at once
constexpr int kSelectThreads = 1024;

// Runs of slices: as many as the threads hold, but none of fewer slices than a
// thread loads at once (a turn with its barrier costs 0.15 us among 1024 threads:
// with all the runs that fit, FP32, 8 members, G = 4096, a generation took 181 us
// at 2 timeslices, 134 at 8, 70 at 17 and 38 at 65; 22.6, 22.5, 23.0 and 25.3 with
// this).
__host__ __device__ __forceinline__ int slice_runs(int cols, int slices, int threads)
{
    const int held = threads / cols, full = (slices + kSliceRun - 1) / kSliceRun;
    return held < full ? held : full;
}

template <bool MODEL>
__global__ __launch_bounds__(MODEL ? kSelectThreads : kWave) void split_select_kernel(EvoArgs a, int g, int init,
                                                                                      const float *part, int slices,
                                                                                      int Npad, int Mpad, const int *ex,
                                                                                      int first)
{
    constexpr int kTauEach = 4;
    const int i = first + static_cast<int>(blockIdx.x);
    if (stopped(a)) return;
    if (a.iter && !init) {
        g = static_cast<int>(a.iter[2]);
        if (i == 0 && threadIdx.x == 0) a.iter[1] = g + 1;
    }
    extern __shared__ __attribute__((aligned(16))) double dsh[];  // a window of residuals, and MODEL their sums
    const Members s = {a.fitness, a.cr_old, a.f_old, a.cur};
    Controls next;  // loaded ahead of their use
    double old = 0.0;
    if (threadIdx.x == 0 && !init) {
        old = a.fitness[i];
        next = Controls(a, s, a.ctl[static_cast<size_t>(g) * a.P + i], i);
    }
    double chi = 0.0;
    for (int t0 = 0; t0 < a.T; t0 += kSelectLds) {
        const int n = min(kSelectLds, a.T - t0);
        if constexpr (MODEL) {
            const int cols = (n + kTauEach - 1) / kTauEach, runs = slice_runs(cols, slices, blockDim.x);
            const int col = threadIdx.x % cols, run = threadIdx.x / cols;
            const int each = (slices + runs - 1) / runs, k0 = run * each, k1 = min(k0 + each, slices);
            const float4 *from = reinterpret_cast<const float4 *>(part + static_cast<size_t>(i) * Mpad + t0) + col;
            const size_t step = static_cast<size_t>(Npad) * Mpad / 4;
            float4 *sums = reinterpret_cast<float4 *>(dsh + (min(kSelectLds, a.T) + 1) / 2 * 2);
            float4 v[kSliceRun];
            // past the run the last slice again, as zeros: a sum that starts
            // from +0 is never -0, so that they leave it as it is
            auto load = [&](int k) {
#pragma unroll
                for (int u = 0; u < kSliceRun; u++) v[u] = from[min(k + u, slices - 1) * step];
#pragma unroll
                for (int u = 0; u < kSliceRun; u++)
                    if (k + u >= k1) v[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            };
            load(k0);
            for (int r = 0; r < runs; r++) {
                if (run == r) {
                    float4 x = r ? sums[col] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    for (int k = k0; k < k1; k += kSliceRun) {
                        if (k > k0) load(k);
#pragma unroll
                        for (int u = 0; u < kSliceRun; u++) {
                            x.x += v[u].x;
                            x.y += v[u].y;
                            x.z += v[u].z;
                            x.w += v[u].w;
                        }
                    }
                    sums[col] = x;
                }
                __syncthreads();
            }
        }
        for (int u = threadIdx.x; u < n; u += blockDim.x) {
            const int t = t0 + u;
            double e;
            if constexpr (MODEL) {
                const float *sums = reinterpret_cast<const float *>(dsh + (min(kSelectLds, a.T) + 1) / 2 * 2);
                e = ldexp(static_cast<double>(sums[u]), ex[t]);
                a.emod[static_cast<size_t>(i) * a.T + t] = e;
            } else {
                e = a.emod[static_cast<size_t>(i) * a.T + t];
            }
            dsh[u] = (a.obs[t] - e) / a.sig[t];
        }
        __syncthreads();
        if (threadIdx.x == 0) chi = chi_sum(dsh, n, (a.T & 1) && t0 + n == a.T, chi);
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    double fit = chi / static_cast<double>(a.T);
    if (a.use_nfm) {  // deac.cpp:961-965, 1398-1416, 1543-1547
        const double mi = fold_row(a.emod + static_cast<size_t>(i) * a.T, a.nfm_dt, a.T, a.T);
        const double q = (a.nfm_value - mi) / a.nfm_error;
        fit = fma(q, q, fit);
    }
    if (a.use_first) {
        const double d = a.mom[i * 4 + 1] - a.first_moment;
        fit += (d * d) / a.first_moment;
    }
    if (a.use_third) {
        const double q = (a.third_moment - a.mom[i * 4 + 2]) / a.third_moment_error;
        fit = fma(q, q, fit);
    }
    if (init) {
        a.fitness[i] = fit;
    } else if (fit <= old) {
        a.fitness[i] = fit;
        a.cur[i] ^= 1;
        for (int sg = 0; sg < a.nsign; sg++) {
            a.cr_old[i * a.nsign + sg] = sg ? next.cr[1] : next.cr[0];
            a.f_old[i * a.nsign + sg] = sg ? next.f[1] : next.f[0];
        }
    }
}

// The generation counter of a captured batch, from the batch's first
// generation on.
__global__ void split_iter_kernel(long *iter, long gen0)
{
    iter[0] = gen0;
    iter[1] = 0;
}

unsigned grid_for(size_t work, unsigned threads)
{
    const size_t blocks = (work + threads - 1) / threads;
    return static_cast<unsigned>(std::max<size_t>(1, std::min<size_t>(blocks, 4096)));
}

// go(first, grid) for all items, a workgroup each: a dispatch holds fewer than
// 2^32 threads, which a selection of 4 million members or a fold of 67 million
// tasks exceeds.
template <class F>
void in_dispatches(size_t items, unsigned threads, F go)
{
    const size_t most = UINT32_MAX / threads;
    for (size_t first = 0; first < items; first += most)
        go(static_cast<int>(first), static_cast<unsigned>(std::min(most, items - first)));
}

}  // namespace

hipError_t launch_split_trial(const EvoArgs &a, int g, int pack, void *B, void *Bl, int Kb, hipStream_t s)
{
    const int members = trial_members(pack);
    const size_t tiles = static_cast<size_t>((a.P + members - 1) / members) * (a.stride / kChunk);
    const dim3 grid(static_cast<unsigned>(tiles) + 1), threads(kThreads);
    if (pack == DEAC_PRECISION_FP32)
        hipLaunchKernelGGL(split_trial_kernel<DEAC_PRECISION_FP32>, grid, threads, 0, s, a, g, B, Bl, Kb);
    else if (pack == DEAC_PRECISION_BF16X3)
        hipLaunchKernelGGL(split_trial_kernel<DEAC_PRECISION_BF16X3>, grid, threads, 0, s, a, g, B, Bl, Kb);
    else
        hipLaunchKernelGGL(split_trial_kernel<DEAC_PRECISION_FP64>, grid, threads, 0, s, a, g, B, Bl, Kb);
    return hipGetLastError();
}

hipError_t launch_split_renorm(const EvoArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(split_renorm_sum_kernel, dim3(grid_for(a.P, kWave)), dim3(kWave), 0, s, a);
    const size_t items = static_cast<size_t>(a.P) * (a.stride / 2);
    hipLaunchKernelGGL(split_renorm_scale_kernel, dim3(grid_for(items, kThreads)), dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_split_pack_fp64(const EvoArgs &a, int init, double *B, int Nt, int Kb, hipStream_t s)
{
    const size_t slots = static_cast<size_t>(Nt) * Kb * 64;
    hipLaunchKernelGGL(split_pack_kernel<double>, dim3(grid_for(slots, kThreads)), dim3(kThreads), 0, s, a, init, B,
                       Nt, Kb);
    return hipGetLastError();
}

hipError_t launch_split_pack_fp32(const EvoArgs &a, int init, float *B, int Nt, int Kb, hipStream_t s)
{
    const size_t slots = static_cast<size_t>(Nt) * Kb * 64;
    hipLaunchKernelGGL(split_pack_kernel<float>, dim3(grid_for(slots, kThreads)), dim3(kThreads), 0, s, a, init, B,
                       Nt, Kb);
    return hipGetLastError();
}

hipError_t launch_split_pack_bf16x3(const EvoArgs &a, int init, void *Bh, void *Bl, int Nt, int Kb, hipStream_t s)
{
    const size_t slots = static_cast<size_t>(Nt) * Kb * 64;
    hipLaunchKernelGGL(split_pack_bf16x3_kernel, dim3(grid_for(slots, kThreads)), dim3(kThreads), 0, s, a, init,
                       static_cast<uint4 *>(Bh), static_cast<uint4 *>(Bl), Nt, Kb);
    return hipGetLastError();
}

hipError_t launch_split_fold(const EvoArgs &a, hipStream_t s)
{
    in_dispatches(static_cast<size_t>(a.P) * a.TB, kWave, [&](int first, unsigned grid) {
        hipLaunchKernelGGL(split_fold_kernel, dim3(grid), dim3(kWave), 0, s, a, first);
    });
    return hipGetLastError();
}

hipError_t launch_split_moments(const EvoArgs &a, int init, hipStream_t s)
{
    hipLaunchKernelGGL(split_moment_kernel, dim3(grid_for(static_cast<size_t>(a.P) * 2, kWave)), dim3(kWave), 0, s, a,
                       init);
    return hipGetLastError();
}

hipError_t launch_split_select(const EvoArgs &a, int g, int init, hipStream_t s)
{
    const size_t lds = static_cast<size_t>(std::min(a.T, kSelectLds)) * sizeof(double);
    in_dispatches(a.P, kWave, [&](int first, unsigned grid) {
        hipLaunchKernelGGL(split_select_kernel<false>, dim3(grid), dim3(kWave), lds, s, a, g, init, nullptr, 0, 0, 0,
                           nullptr, first);
    });
    return hipGetLastError();
}

hipError_t launch_split_model_select(const EvoArgs &a, int g, int init, const float *part, int slices, int Npad, int Mpad,
                                     const int *ex, hipStream_t s)
{
    const size_t window = static_cast<size_t>(std::min(a.T, kSelectLds));
    const size_t lds = (window + 1) / 2 * 2 * sizeof(double) + (window + 3) / 4 * sizeof(float4);
    const int cols = (static_cast<int>(window) + 3) / 4;
    // the wavefronts that have slices to add, and one per 64 residuals
    const int used = std::max(cols * slice_runs(cols, slices, kSelectThreads), std::min(a.T, kSelectThreads));
    const unsigned threads = static_cast<unsigned>((used + kWave - 1) / kWave * kWave);
    in_dispatches(a.P, threads, [&](int first, unsigned grid) {
        hipLaunchKernelGGL(split_select_kernel<true>, dim3(grid), dim3(threads), lds, s, a, g, init, part, slices, Npad,
                           Mpad, ex, first);
    });
    return hipGetLastError();
}

hipError_t launch_split_iter(long *iter, long gen0, hipStream_t s)
{
    hipLaunchKernelGGL(split_iter_kernel, dim3(1), dim3(1), 0, s, iter, gen0);
    return hipGetLastError();
}

}  // namespace deac
