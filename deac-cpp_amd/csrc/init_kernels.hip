// gfx950 kernels of the engines' set-up: jump tables, and the initial
// populations (deac.cpp:430-458, 584-602): the draws of every member in
// parallel, then the normalization.  The host only
// computes the random state at each member's first draw (one GF(2) jump per
// member).  Compiled with -ffp-contract=off.
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "fold_common.hpp"
#include "init_kernels.hpp"

namespace deac {

namespace {

constexpr int kThreads = 256;
constexpr int kWave = 64;

// One thread per sub-stream of a member's nsign*G draws: it jumps to its
// first draw with a nibble table and steps sublen draws.  The draws
// interleave the signs gene by gene; the negative sign's zero frequency
// repeats the positive one's.  Bound: the 8-byte stores, which a lane makes
// at consecutive positions of its own run (the cache lines fill in L2).  On
// host threads with a pageable upload the same populations took 150 ms for
// 256 instances of 32 members at G = 4096; here 1 ms.
__global__ __launch_bounds__(kThreads) void init_draw_kernel(InitArgs a)
{
    const long item = static_cast<long>(blockIdx.x) * kThreads + threadIdx.x;
    const long row = item / a.nsub;
    const int sub = static_cast<int>(item % a.nsub);
    if (row >= a.rows) return;
    const uint64_t *st = a.start + row * 4;
    uint64_t s[4] = {st[0], st[1], st[2], st[3]};
    if (a.lane_tab) {
        lane_jump(a.tab, s, s);
    } else if (sub > 0) {
        const uint64_t *tab = a.tab + static_cast<size_t>(sub - 1) * (64 * 16 * 4);
        uint64_t o[4] = {0, 0, 0, 0};
#pragma unroll 4
        for (int n = 0; n < 64; n++) {
            const int v = static_cast<int>((s[n >> 4] >> ((n & 15) * 4)) & 15);
            const uint64_t *e = tab + (n * 16 + v) * 4;
            o[0] ^= e[0];
            o[1] ^= e[1];
            o[2] ^= e[2];
            o[3] ^= e[3];
        }
        for (int w = 0; w < 4; w++) s[w] = o[w];
    }
    const long inst = row / a.P, member = row % a.P;
    double *x = a.pop + (a.offset ? a.offset[inst] : 0) + static_cast<size_t>(member) * a.stride;
    const int Kc = a.nsign * a.G;
    const int d0 = sub * a.sublen, d1 = min(d0 + a.sublen, Kc);
    for (int d = d0; d < d1; d++) {
        double u = to_unit(xnext(s));
        if (a.allow_neg) u -= 0.5;
        const int j = a.nsign == 2 ? d >> 1 : d;
        if (a.nsign == 1 || !(d & 1)) {
            x[j] = u;
            if (a.nsign == 2 && j == 0) x[a.G] = u;
        } else if (j > 0) {
            x[a.G + j] = u;
        }
    }
    if (sub == a.nsub - 1)
        for (int k = Kc; k < a.stride; k++) x[k] = 0.0;
}

// One wavefront per member: the zeroth moment as the reference folds it,
// then every position scaled.  Bound: the fold's chain of adds.
__global__ __launch_bounds__(kThreads) void init_normalize_kernel(InitArgs a)
{
    __shared__ __attribute__((aligned(16))) double buf[kThreads / kWave][kFoldLds];
    const int wid = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const long row = static_cast<long>(blockIdx.x) * (kThreads / kWave) + wid;
    if (row >= a.rows) return;
    const long inst = row / a.P, member = row % a.P;
    double *x = a.pop + (a.offset ? a.offset[inst] : 0) + static_cast<size_t>(member) * a.stride;
    const int Kc = a.nsign * a.G;
    const double scale = a.zeroth / wave_fold(x, a.nterm, Kc, a.G, buf[wid]);
    for (int k = lane; k < Kc; k += kWave) x[k] *= scale;
}

// One workgroup per matrix: thread b carries column b of M^l from power to
// power by nibble lookups in LDS, and every power's 16 sums of four columns go
// out to the lane's place.  (On the host a set of tables took 2 ms.)
__global__ __launch_bounds__(kThreads) void lane_tables_kernel(LaneTabArgs a)
{
    typedef uint64_t pair __attribute__((ext_vector_type(2)));
    struct State {
        pair h[2];
    };
    __shared__ State step[64][16];  // nibble table of M
    __shared__ State col[256];
    const int b = threadIdx.x, n = b >> 2, v0 = (b & 3) * 4;
    uint64_t *out = a.tab[blockIdx.x];
    // the 4 of a nibble's 16 sums of columns that this thread forms
    auto sums = [&](State (&s)[4]) {
        const State c0 = col[4 * n], c1 = col[4 * n + 1], c2 = col[4 * n + 2], c3 = col[4 * n + 3];
        for (int h = 0; h < 2; h++) {
            pair base = {0, 0};
            if (v0 & 4) base ^= c2.h[h];
            if (v0 & 8) base ^= c3.h[h];
            s[0].h[h] = base;
            s[1].h[h] = base ^ c0.h[h];
            s[2].h[h] = base ^ c1.h[h];
            s[3].h[h] = s[1].h[h] ^ c1.h[h];
        }
    };
    const pair *m = reinterpret_cast<const pair *>(a.columns) + (static_cast<size_t>(blockIdx.x) * 256 + b) * 2;
    col[b].h[0] = m[0];
    col[b].h[1] = m[1];
    __syncthreads();
    State s[4];
    sums(s);
    for (int j = 0; j < 4; j++) step[n][v0 + j] = s[j];
    State c;  // column b of M^l, from the identity on
    for (int h = 0; h < 2; h++)
        c.h[h] = pair{b >> 6 == 2 * h ? UINT64_C(1) << (b & 63) : 0, b >> 6 == 2 * h + 1 ? UINT64_C(1) << (b & 63) : 0};
    for (int l = 0; l < 64; l++) {
        __syncthreads();
        col[b] = c;
        __syncthreads();
        sums(s);
        for (int j = 0; j < 4; j++)
            for (int h = 0; h < 2; h++)
                reinterpret_cast<pair *>(out)[((n * 16 + v0 + j) * 2 + h) * 64 + l] = s[j].h[h];
        const uint64_t w[4] = {c.h[0].x, c.h[0].y, c.h[1].x, c.h[1].y};
        pair o0 = {0, 0}, o1 = {0, 0};
#pragma unroll
        for (int q = 0; q < 64; q++) {
            const State &e = step[q][(w[q >> 4] >> ((q & 15) * 4)) & 15];
            o0 ^= e.h[0];
            o1 ^= e.h[1];
        }
        c.h[0] = o0;
        c.h[1] = o1;
    }
}

// One workgroup per instance.  (A copy per instance from the host took 25 us.)
__global__ __launch_bounds__(kThreads) void gather_best_kernel(const long *table, const double *fitness, int pitch,
                                                               const double *pop, double *out)
{
    const long *t = table + static_cast<size_t>(blockIdx.x) * 5;
    const double *fit = fitness + static_cast<size_t>(blockIdx.x) * pitch;
    int best = 0;
    double minimum = fit[0];
    for (int k = 0; k < t[2]; k++)
        if (fit[k] < minimum) {
            minimum = fit[k];
            best = k;
        }
    const double *row = pop + t[1] + best * t[4];
    for (long k = threadIdx.x; k < t[3]; k += kThreads) out[t[0] + k] = row[k];
}

}  // namespace

hipError_t launch_gather_best(const long *table, size_t n, const double *fitness, int pitch, const double *pop,
                              double *out, hipStream_t s)
{
    hipLaunchKernelGGL(gather_best_kernel, dim3(static_cast<unsigned>(n)), dim3(kThreads), 0, s, table, fitness, pitch,
                       pop, out);
    return hipGetLastError();
}

hipError_t launch_lane_tables(const LaneTabArgs &a, int sets, hipStream_t s)
{
    hipLaunchKernelGGL(lane_tables_kernel, dim3(sets), dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_initial_population(const InitArgs &a, hipStream_t s)
{
    const long items = a.rows * a.nsub;
    hipLaunchKernelGGL(init_draw_kernel, dim3(static_cast<unsigned>((items + kThreads - 1) / kThreads)), dim3(kThreads),
                       0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !a.nterm) return e;
    constexpr long per = kThreads / kWave;
    hipLaunchKernelGGL(init_normalize_kernel, dim3(static_cast<unsigned>((a.rows + per - 1) / per)), dim3(kThreads), 0,
                       s, a);
    return hipGetLastError();
}

}  // namespace deac
