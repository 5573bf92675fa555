// gfx950 kernels of the DEAC engine, plain FP64 form.
//
// One generation of the reference loop (deac.cpp:1138-1573) is split in
// two independent parts:
//   * the random choices, which depend only on the xoshiro256+ stream:
//       walk         - one wavefront walks the sequential, data-dependent
//                      part of the stream (jDE F/CR redraws, rejection-
//                      sampled donor indices) and skips each member's 2G
//                      crossover-mask draws with GF(2) jumps;
//       mask draws   - one wavefront per member regenerates them: lane l
//                      jumps to draw l*chunk with a nibble table and steps
//                      chunk draws;
//   * evolve_kernel - a persistent kernel (all workgroups co-resident) that runs a batch of
//     generations: best-fitness/stats/stop test, trial vectors (DE/rand/1,
//     binomial crossover, |.|, zero-frequency match), the model ISF
//     E = K.S as exact FP64 FMA chains (4x4x4 FP64 MFMAs), chi^2 in the reference's summation
//     order, greedy selection.  Grid barriers separate the phases.
// The file is compiled with -ffp-contract=off: every fused multiply-add is
// written as fma().
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.hpp"
#include "evolve_common.hpp"
#include "fold_common.hpp"
#include "kernels.hpp"

namespace deac {

namespace {

constexpr int kWave = 64;
constexpr int kEvoWaves = kEvoThreads / kWave;

// Status words for the host, by one thread: it reads them after the dispatch's
// own stop event, which does not release at system scope, so this does, and the
// stores have arrived in host memory before the wave ends.
__device__ __forceinline__ void tell_host(int *status, int word, int value)
{
    __hip_atomic_store(status + word, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
}

// Grid-wide barrier of the persistent evolution kernel.  The wait is
// bounded: after kBarrierSpins polls the workgroup records a failure and every
// caller leaves the kernel, so a broken launch cannot hang the device.
constexpr unsigned kBarrierSpins = 1u << 24;

// Where many workgroups take part (kXcdBarrierWgs), those of an XCD, which share
// its L2, arrive together: the last of them writes the L2 back for all.  The
// write-backs of an XCD's workgroups queue: with three barriers a generation,
// 248 workgroups, T = 257, G = 16384, 64 members took 168 us a generation with
// one each and 141 this way, 512 members G = 4096 147 and 112; with 52 workgroups
// (two barriers) 43.3 and 43.1; below 32 it makes no difference.
constexpr int kXcdBarrierWgs = 32;
struct GridBarrier {
    unsigned *bar;          // arrivals
    unsigned *xcd = nullptr;  // arrivals of this XCD's workgroups, or null: one by one
    unsigned mine = 0;      // of them, per barrier
    unsigned arrivals;      // at bar, per barrier
    unsigned epoch = 0, target = 0;
    const EvoArgs &a;

    __device__ __forceinline__ GridBarrier(const EvoArgs &ea)
        : bar(ea.bar), arrivals(ea.nwg), a(ea)
    {
    }

    // Each wave drains its own memory operations (the wait alone is no memory
    // fence to the compiler: the one in front holds the stores there; where
    // an XCD's workgroups arrive together, nothing else stands between the
    // stores of all but the last and their arrival); then one thread per
    // workgroup publishes the workgroup's stores at agent scope (L2 write-back,
    // visible to the other XCDs), arrives, waits, and invalidates this CU's
    // caches for what the other workgroups wrote.
    __device__ __forceinline__ bool wait()
    {
        __shared__ int timed_out;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        target += arrivals;
        epoch++;
        if (threadIdx.x == 0) {
            timed_out = 0;
            bool last = true;
            if (xcd)
                last = __hip_atomic_fetch_add(xcd, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == mine * epoch;
            if (last) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
                __hip_atomic_fetch_add(bar, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            unsigned spins = 0;
            while (__hip_atomic_load(bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
                __builtin_amdgcn_s_sleep(1);
                if (++spins == kBarrierSpins) {
                    timed_out = 1;
                    __hip_atomic_store(a.status + 2, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    tell_host(a.host_status, 2, 1);
                    break;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();
        return timed_out == 0;
    }

    // Counts the workgroups per XCD: by the number the hardware gives, which
    // says whose L2 a workgroup's stores are in.
    __device__ __forceinline__ bool by_xcd()
    {
        __shared__ unsigned counted[2];
        constexpr int kXccId = 20 | 3 << 11;  // HW_REG_XCC_ID, 4 bits
        unsigned *here = a.xbar + (__builtin_amdgcn_s_getreg(kXccId) % kXcds) * kXcdWords;
        if (threadIdx.x == 0) __hip_atomic_fetch_add(here + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!wait()) return false;
        if (threadIdx.x == 0) {
            unsigned n = 0;
            for (int x = 0; x < kXcds; x++)
                n += __hip_atomic_load(a.xbar + x * kXcdWords + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
            counted[0] = __hip_atomic_load(here + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            counted[1] = n;
        }
        __syncthreads();
        xcd = here;
        mine = counted[0];
        arrivals = counted[1];
        epoch = 0;
        return true;
    }
};

// The walk's stream is wave-uniform: its step as scalar (SALU) operations,
// the rotate as two 64-bit shifts (the funnel-shift form of xnext would put
// it on the VALU and bring it back with v_readfirstlane on every draw).
__device__ __forceinline__ uint64_t xnext_uniform(uint64_t (&s)[4])  // rng.hpp:25-39
{
    const uint64_t s0 = s[0], s1 = s[1], s2 = s[2], s3 = s[3];
    const uint64_t out = s0 + s3;
    const uint64_t t = s1 << 17;
    const uint64_t n3 = s3 ^ s1;
    s[1] = s1 ^ s2 ^ s0;
    s[0] = s0 ^ n3;
    s[2] = s2 ^ s0 ^ t;
    s[3] = (n3 << 45) | (n3 >> 19);
    return out;
}

// mod_p for a wave-uniform draw: the remainder before the correction is
// below 2P < 2^32, so the correction compares 32-bit words (SALU)
__device__ __forceinline__ uint32_t mod_p_uniform(uint64_t x, uint64_t magic, uint32_t P)
{
    const uint64_t q = __umul64hi(x, magic);
    uint32_t r = static_cast<uint32_t>(x - q * P);
    if (r >= P) r -= P;
    return r;
}

// s <- M s from M's nibble table: 64 lookups of 32 bytes.
__device__ __forceinline__ void nibble_jump(const uint64_t *tab, uint64_t (&s)[4])
{
    uint64_t o[4] = {0, 0, 0, 0};
#pragma unroll 16
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

// Lane q's copy of a state, in every lane (q uniform).
__device__ __forceinline__ void lane_state(const uint64_t (&s)[4], int q, uint64_t (&out)[4])
{
    for (int w = 0; w < 4; w++) {
        const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(s[w]), q);
        const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(s[w] >> 32), q);
        out[w] = (static_cast<uint64_t>(hi) << 32) | lo;
    }
}

// u < p for the draw x, u = (x >> 11) 2^-53, in whole numbers: x < below, or
// all draws.
struct DrawLimit {
    uint64_t below;
    bool all;
};

__device__ __forceinline__ DrawLimit draw_limit(double p)
{
    if (!(p > 0.0)) return {0, false};
    if (p >= 1.0) return {0, true};
    return {static_cast<uint64_t>(ceil(p * 0x1.0p53)) << 11, false};
}

__device__ __forceinline__ bool passes(const DrawLimit &l, uint64_t x) { return l.all || x < l.below; }

}  // namespace

// ---------------------------------------------------------------- walk

namespace {

// Whether the batch that runs beside these draws has met its stop test (the
// walk looks every few generations): what they make is then not used.
constexpr int kWalkPoll = 16;

__device__ __forceinline__ bool stopped(const int *halt)
{
    return halt && __hip_atomic_load(halt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

// Which of a window's 64 draws are values: bit i where draw i belongs to a test
// before it that passed its limit (bit i of passed: draw i is under the limit).
// Among draws under the limit tests and values alternate, a test first, so a
// draw is a value where the run of them that ends in front of it is odd; every
// lane measures its own.  carry: whether draw 0 is a value (which ends a run,
// whatever its size); set to whether the draw behind the window is.  By the whole
// wavefront.
__device__ __forceinline__ uint64_t value_bits(uint64_t passed, bool &carry)
{
    const int lane = threadIdx.x & (kWave - 1);
    const uint64_t first = carry ? 1 : 0, failed = ~passed | first;
    // the failed draws in front of the lane's, the nearest at the top
    const int zeros = lane ? __clzll(failed << (kWave - lane)) : 0;
    carry = __clzll(failed) & 1;
    return __ballot(min(zeros, lane) & 1) | first;
}

// Walk of a.ngen generations by one wavefront (deac.cpp:1180-1240): the
// sequential, data-dependent part of the stream -- which draws are F/CR
// redraws, how many draws each member's rejection-sampled donors take -- with
// the draws themselves made in parallel.
//
// jDE controls (CR+, F+, CR-, F- per member, a test draw each and a value
// draw where the test passes): lane l jumps to draw l*c1 of the generation
// and makes c1 draws into LDS; windows of 64 draws are then told apart into
// tests and values at once.  Donors: lane l jumps to where member m0+l starts
// if every member before it takes exactly 3 donor draws (its crossover draws
// are skipped in the same jump); e, the draws really taken beyond that, is
// uniform, so all lanes try their member at offset e, the lanes up to the
// first one that rejects a draw are right, and the rest try again from there.
// The lane behind the last member is where the next block, or the next
// generation, starts.
//
// Bound: latency of one wavefront, mostly the jumps' table loads (128 of 1 KB
// each, from L2).  Walking member by member took 0.7 us per member: per
// generation 356 us at 512 members, 45 at 64.
__device__ void walk_wide(const WalkArgs &a, uint64_t *lds)
{
    const int lane = threadIdx.x & (kWave - 1);
    uint64_t *draws = lds;                                                   // [kWave][c1 | 1]
    uint32_t *res = reinterpret_cast<uint32_t *>(lds + kWave * (a.c1 | 1));  // [kWalkDraws][kWave]
    uint32_t *flags = res + kWalkDraws * kWave;                              // [P]
    const int c1 = a.c1, pitch = a.c1 | 1;
    const uint32_t P = static_cast<uint32_t>(a.P);
    const int tests = 2 * a.nsign * a.P;
    const DrawLimit lim = draw_limit(a.tau_cr);  // tau_f is the same (walk_is_wide)
    // lanes that usually cover a generation's controls
    const int n1 = min(kWave, (tests + tests / 4 + 8 + c1 - 1) / c1);
    uint64_t s[4] = {a.state[0], a.state[1], a.state[2], a.state[3]};  // uniform: where the next draw is
    for (int g = 0; g < a.ngen; g++) {
        if (g % kWalkPoll == 0 && stopped(a.halt)) return;
        if (lane < 4) a.gen_start[static_cast<size_t>(g) * 4 + lane] = s[lane & 3];
        MemberCtl *ctl = a.ctl + static_cast<size_t>(g) * a.P;
        for (int i = lane; i < a.P; i += kWave) flags[i] = 0;

        int k0 = 0;          // tests before the current window
        bool carry = false;  // the window's first draw is a value
        int end = -1;        // draw behind the last control, of the current round
        while (end < 0) {
            uint64_t start[4] = {s[0], s[1], s[2], s[3]};
            if (lane < n1) {
                lane_jump(a.tab1, s, start);
                uint64_t t[4] = {start[0], start[1], start[2], start[3]};
                for (int j = 0; j < c1; j++) draws[lane * pitch + j] = xnext(t);
            }
            asm volatile("" ::: "memory");
            const int avail = n1 * c1;
            for (int w = 0; w < avail && end < 0; w += kWave) {
                const int o = w + lane;
                const uint64_t x = o < avail ? draws[o / c1 * pitch + o % c1] : 0;
                const bool in = o < avail;
                const uint64_t valid = __ballot(in);
                const uint64_t passed = __ballot(in && passes(lim, x));
                const uint64_t values = value_bits(passed, carry) & valid;
                const uint64_t below = (UINT64_C(1) << lane) - 1;
                const uint64_t test_bits = valid & ~values;
                // the test of this draw, or the one its value belongs to
                const int k = k0 + __popcll(test_bits & below) - ((values >> lane) & 1 ? 1 : 0);
                if (((values >> lane) & 1) && k < tests) {
                    const int i = k / (2 * a.nsign), sg = (k / 2) % a.nsign;
                    if (k & 1) ctl[i].f_value[sg] = 2.0 * to_unit(x);
                    else ctl[i].cr_value[sg] = to_unit(x);
                    __hip_atomic_fetch_or(&flags[i], (k & 1 ? 2u : 1u) << (2 * sg), __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                // the first draw that is a test past the last one ends the controls
                const uint64_t past = __ballot(in && !((values >> lane) & 1) && k >= tests);
                if (past) end = w + __builtin_ctzll(past);
                k0 += __popcll(test_bits);
                if (w + kWave > avail) carry = (passed & test_bits) >> (avail - w - 1) & 1;
            }
            if (end < 0 && k0 == tests && !carry) end = avail;
            // on to the next round, or to the draw behind the controls
            const int to = end < 0 ? avail : end;
            const int q = min(to / c1, n1 - 1);
            lane_state(start, q, s);
            for (int j = q * c1; j < to; j++) (void)xnext_uniform(s);
        }

        for (int m0 = 0; m0 < a.P;) {
            const int cnt = min(kWave - 1, a.P - m0);  // members tried in this block
            uint64_t start[4] = {s[0], s[1], s[2], s[3]};
            if (lane <= cnt) lane_jump(a.tab2, s, start);
            uint64_t t[4] = {start[0], start[1], start[2], start[3]};
            int made = 0;
            auto more = [&]() {
#pragma unroll 2
                for (int j = 0; j < 4; j++) res[(made + j) * kWave + lane] = mod_p(xnext(t), a.mod_magic, P);
                made += 4;
                asm volatile("" ::: "memory");
            };
            const uint32_t i = static_cast<uint32_t>(m0 + lane);
            int cur = 0, e = 0;
            bool room = true;
            while (cur < cnt && room) {
                while (made < e + 4 && made + 4 <= kWalkDraws) more();
                // donor indices (deac.cpp:200-216) from draw e on
                uint32_t m[3] = {i, i, i};
                int got = 0, d = e;
                while (got < 3 && d < made) {
                    const uint32_t r = res[d++ * kWave + lane];
                    if (r == i || (got > 0 && r == m[0]) || (got > 1 && r == m[1])) continue;
                    if (got == 0) m[0] = r;
                    else if (got == 1) m[1] = r;
                    else m[2] = r;
                    got++;
                }
                const bool mine = lane >= cur && lane < cnt;
                const uint64_t bad = __ballot(mine && (got < 3 || d - e > 3));
                const int f = bad ? __builtin_ctzll(bad) : cnt;
                const bool whole = f < cnt && __builtin_amdgcn_readlane(static_cast<uint32_t>(got), f) == 3;
                if (mine && (lane < f || (lane == f && whole))) {
                    MemberCtl &c = ctl[i];
                    c.flags = flags[i];
                    c.mutant[0] = m[0];
                    c.mutant[1] = m[1];
                    c.mutant[2] = m[2];
                    c.mask_steps = static_cast<uint32_t>(d);
                    for (int w = 0; w < 4; w++) c.mask_state[w] = start[w];
                }
                cur = f;
                if (whole) {
                    e = static_cast<int>(__builtin_amdgcn_readlane(static_cast<uint32_t>(d), f)) - 3;
                    cur = f + 1;
                } else if (f < cnt) {  // this member needs more draws than were made
                    if (made + 4 <= kWalkDraws) more();
                    else room = false;  // a new block starts at it
                }
            }
            // a member that one block cannot settle at its start would need
            // more than kWalkDraws draws for three donors: walked one by one
            if (cur == 0) {
                uint32_t m[3] = {static_cast<uint32_t>(m0), static_cast<uint32_t>(m0), static_cast<uint32_t>(m0)};
                const uint32_t i0 = static_cast<uint32_t>(m0);
                uint64_t first[4] = {s[0], s[1], s[2], s[3]};
                uint32_t steps = 0;
                for (int got = 0; got < 3; steps++) {
                    const uint32_t r = mod_p_uniform(xnext_uniform(s), a.mod_magic, P);
                    if (r == i0 || (got > 0 && r == m[0]) || (got > 1 && r == m[1])) continue;
                    m[got++] = r;
                }
                if (lane == 0) {
                    MemberCtl &c = ctl[m0];
                    c.flags = flags[m0];
                    for (int w = 0; w < 3; w++) c.mutant[w] = m[w];
                    c.mask_steps = steps;
                    for (int w = 0; w < 4; w++) c.mask_state[w] = first[w];
                }
                nibble_jump(a.skip_tab, s);
                m0 += 1;
                continue;
            }
            lane_state(start, cur, s);
            for (int j = 0; j < e; j++) (void)xnext_uniform(s);
            m0 += cur;
        }
    }
    if (lane < 4) a.state[lane] = s[lane & 3];
}

// The same member by member.
__device__ void walk_serial(const WalkArgs &a, uint64_t *rows)
{
    const int lane = threadIdx.x & (kWave - 1);
    for (int k = lane; k < 256 * 4; k += kWave) rows[k] = a.skip_rows[k];
    asm volatile("" ::: "memory");
    // Every lane carries the same state; lane 0 writes the records.
    uint64_t s[4] = {a.state[0], a.state[1], a.state[2], a.state[3]};
    const uint32_t P = static_cast<uint32_t>(a.P);
    const DrawLimit lim_cr = draw_limit(a.tau_cr), lim_f = draw_limit(a.tau_f);
    for (int g = 0; g < a.ngen; g++) {
        if (g % kWalkPoll == 0 && stopped(a.halt)) return;
        if (lane == 0)
            for (int w = 0; w < 4; w++) a.gen_start[static_cast<size_t>(g) * 4 + w] = s[w];
        MemberCtl *ctl = a.ctl + static_cast<size_t>(g) * a.P;
        // jDE control redraws, deac.cpp:1180-1213: CR+, F+, CR-, F- per member.
        for (int i = 0; i < a.P; i++) {
            uint32_t flags = 0;
            double crv[2] = {0.0, 0.0}, fv[2] = {0.0, 0.0};
            for (int sg = 0; sg < a.nsign; sg++) {
                if (passes(lim_cr, xnext_uniform(s))) {
                    flags |= 1u << (2 * sg);
                    crv[sg] = to_unit(xnext_uniform(s));
                }
                if (passes(lim_f, xnext_uniform(s))) {
                    flags |= 2u << (2 * sg);
                    fv[sg] = 2.0 * to_unit(xnext_uniform(s));
                }
            }
            if (lane == 0) {
                ctl[i].flags = flags;
                ctl[i].cr_value[0] = crv[0];
                ctl[i].cr_value[1] = crv[1];
                ctl[i].f_value[0] = fv[0];
                ctl[i].f_value[1] = fv[1];
            }
        }
        // Donor indices (deac.cpp:200-216), then skip the member's masks.
        for (int i = 0; i < a.P; i++) {
            const uint32_t i0 = static_cast<uint32_t>(i);
            uint32_t m0 = i0, m1 = i0, m2 = i0;
            while (m0 == i0) m0 = mod_p_uniform(xnext_uniform(s), a.mod_magic, P);
            while (m1 == i0 || m1 == m0) m1 = mod_p_uniform(xnext_uniform(s), a.mod_magic, P);
            while (m2 == i0 || m2 == m0 || m2 == m1) m2 = mod_p_uniform(xnext_uniform(s), a.mod_magic, P);
            if (lane == 0) {
                ctl[i].mutant[0] = m0;
                ctl[i].mutant[1] = m1;
                ctl[i].mutant[2] = m2;
                ctl[i].mask_steps = 0;
                for (int w = 0; w < 4; w++) ctl[i].mask_state[w] = s[w];
            }
            // s <- T^(nsign*G) s: lane l forms output bits l, 64+l, 128+l,
            // 192+l as parities of (row & s); ballots assemble the words.
            // (r & s) ^ acc is one v_bitop3 per 32-bit half (truth table
            // 0x6a over the inputs 0xf0, 0xcc, 0xaa).
            uint64_t out[4];
            for (int w = 0; w < 4; w++) {
                const uint64_t *r = rows + (w * 64 + lane) * 4;
                uint32_t lo = static_cast<uint32_t>(r[0]) & static_cast<uint32_t>(s[0]);
                uint32_t hi = static_cast<uint32_t>(r[0] >> 32) & static_cast<uint32_t>(s[0] >> 32);
                for (int k = 1; k < 4; k++) {
                    lo = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(r[k]), static_cast<uint32_t>(s[k]), lo, 0x6a);
                    hi = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(r[k] >> 32), static_cast<uint32_t>(s[k] >> 32),
                                                     hi, 0x6a);
                }
                out[w] = __ballot(__popc(lo ^ hi) & 1);
            }
            for (int w = 0; w < 4; w++) s[w] = out[w];
        }
    }
    if (lane == 0)
        for (int w = 0; w < 4; w++) a.state[w] = s[w];
}

// One wavefront.
__device__ __forceinline__ void walk(const WalkArgs &a, uint64_t *lds)
{
    if (a.wide) walk_wide(a, lds);
    else walk_serial(a, lds);
}

}  // namespace

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 1))) void walk_kernel(WalkArgs a)
{
    extern __shared__ uint64_t walk_lds[];
    walk(a, walk_lds);
}

// ---------------------------------------------------------------- masks

namespace {

// Crossover-mask draws: one wavefront per member of a generation, lane l makes
// draws l*chunk on.  first, step: the wavefront's members; buf: kMaskLds
// doubles of LDS of this wavefront.
//
// Bound: alone on the chip the stores (8 bytes per draw); beside an evolution
// one wavefront's instruction issue.  Rounds of 16 draws per lane go
// through LDS, so that 8 lanes together store one line of 128 bytes.  Lane by
// lane, 64 lines per store, 512 members of 8192 draws took 22 us, 64 members
// of 32768 draws 37.
__device__ void mask_draws(const MaskArgs &a, size_t first, size_t step, double *buf)
{
    typedef uint64_t pair __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & (kWave - 1);
    uint64_t *mine = reinterpret_cast<uint64_t *>(buf) + lane * kMaskRow;
    const pair *from = reinterpret_cast<const pair *>(buf) + (lane >> 3) * (kMaskRow / 2) + (lane & 7);
    for (size_t wave = first; wave < static_cast<size_t>(a.ngen) * a.P; wave += step) {
        if (stopped(a.halt)) return;
        const MemberCtl &c = a.ctl[wave];
        uint64_t s[4] = {c.mask_state[0], c.mask_state[1], c.mask_state[2], c.mask_state[3]};
        for (uint32_t k = 0; k < c.mask_steps; k++) (void)xnext(s);
        lane_jump(a.lane_tab, s, s);  // T^(lane*chunk)
        uint64_t *raw = a.raw + wave * a.rstride;
        for (int c0 = 0; c0 < a.chunk; c0 += kMaskRound) {
            const int n = min(kMaskRound, a.chunk - c0);
            for (int j = 0; j < n; j++) mine[j] = xnext(s) >> 11;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // 8 lanes' draws at a time, a pair per lane
            int k = (lane >> 3) * a.chunk + c0 + 2 * (lane & 7);
            const bool in = 2 * (lane & 7) < n;
            for (int r = 0; r < 8; r++, k += 8 * a.chunk)
                if (in && k < a.Kc) *reinterpret_cast<pair *>(raw + k) = from[r * 8 * (kMaskRow / 2)];
            __builtin_amdgcn_wave_barrier();
        }
    }
}

}  // namespace

template <bool WALK>
__global__ __launch_bounds__(256) void mask_kernel(MaskArgs a, WalkArgs next)
{
    extern __shared__ __attribute__((aligned(16))) double mask_lds[];
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int block = blockIdx.x;
    if constexpr (WALK) {
        if (block == 0) {
            if (wid == 0) walk(next, reinterpret_cast<uint64_t *>(mask_lds));
            return;
        }
        block--;
    }
    const size_t waves = static_cast<size_t>(a.ngen) * a.P;
    mask_draws(a, static_cast<size_t>(block) * kEvoWaves + wid, waves, mask_lds + wid * kMaskLds);
}

// ---------------------------------------------------------------- evolution

namespace {

// Chains: units of 8 positions, chunks of 16 units; K units in flight per
// wavefront (one 16-byte load each, 17.6 ns a unit), genome units read ahead
// from LDS, and the LDS of a wavefront: two chunks of 4 genome rows, padded
// so that the rows start 8 banks apart.
constexpr int kChunkUnits = kChunk / kUnit;
constexpr int kRing = 2 * kChunkUnits;
constexpr int kReadAhead = 4;
constexpr int kSRow = kChunk + 4;
constexpr int kChainLds = 2 * kChainRows * kSRow;
static_assert(kChainLds >= kFoldLds && kChainLds >= kFoldTaskLds, "a wave's LDS serves its folds as well");
static_assert(kKtilePad >= kRing && kKtilePad >= kFoldRing, "the K rings read past the last unit");
static_assert((kEvoWaves * kChainLds + kResidLds) * sizeof(double) <= kEvoLds, "chains and members' state fit in LDS");

// A tau block's K units from a moving chunk on, as buffer loads: the base is
// scalar and the unit an immediate offset from one of four lane offsets, so a
// load is one instruction with one address register (with 64-bit lane
// addresses a unit took 28 ns, 24.5 this way, with the genome's loads still in
// front of the MFMAs; 17.6 now).
struct KUnits {
    static_assert(kChunkUnits == 16, "four lane offsets, four units each");
    const char *base;
    int vo[4];
    __device__ __forceinline__ KUnits(const double *p)
        : base(reinterpret_cast<const char *>(p))
    {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            vo[k] = (threadIdx.x & (kWave - 1)) * 16 + k * 4096;
            asm("" : "+v"(vo[k]));  // a register each
        }
    }
    __device__ __forceinline__ dvec2 load(int i) const
    {
        const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base), 0, kChunkUnits * 1024, 0x00020000);
        return __builtin_bit_cast(dvec2, __builtin_amdgcn_raw_buffer_load_b128(r, vo[i >> 2] + (i & 3) * 1024, 0, 0));
    }
    __device__ __forceinline__ void advance() { base += kChunkUnits * 1024; }
};

// Positions in front of a chunk: rows may be longer than the 4 GiB that a buffer
// load's own offset reaches, so that the base moves.
__host__ __device__ constexpr size_t chunk_offset(int chunk) { return static_cast<size_t>(chunk) * kChunk; }
static_assert(chunk_offset((1 << 30) / kChunk) * sizeof(double) == size_t(8) << 30, "rows of 2^30 positions");

// A member group's four genome rows, read the same way, 128 positions a load.
struct GenomeRows {
    const double *row[kChainRows];
    int vo;  // this lane's two positions, bytes
    __device__ __forceinline__ dvec2 load(int m, int chunk) const
    {
        const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(row[m] + chunk_offset(chunk)), 0, kChunk * 8,
                                                         0x00020000);
        return __builtin_bit_cast(dvec2, __builtin_amdgcn_raw_buffer_load_b128(r, vo, 0, 0));
    }
};

// One chunk of the chains: kr[h .. h+15] hold its K units and are refilled
// with those two chunks on; sr holds the genome units about to be used.  st,
// the genome rows of the next chunk, goes to its place in LDS (to) and is
// refilled from chunk `ahead`.  Every instruction beside the MFMAs has its
// place behind one, whose result the next one waits for.
template <int H>
__device__ __forceinline__ void chain_chunk(double &acc, dvec2 (&kr)[kRing], dvec2 (&sr)[kReadAhead], KUnits &ku,
                                            const double *here, const double *next, dvec2 (&st)[kChainRows],
                                            const GenomeRows &rows, double *to, int ahead)
{
#pragma unroll
    for (int i = 0; i < kChunkUnits; i++) {
        const dvec2 k = kr[H + i], s = sr[i % kReadAhead];
        const int j = i + kReadAhead;
        const double *p = j < kChunkUnits ? here + j * kUnit : next + (j - kChunkUnits) * kUnit;
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(k.x, s.x, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        sr[i % kReadAhead] = dvec2{p[0], p[4]};
        __builtin_amdgcn_sched_barrier(0);
        if (i < kChainRows) *reinterpret_cast<dvec2 *>(to + i * kSRow) = st[i % kChainRows];
        __builtin_amdgcn_sched_barrier(0);
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(k.y, s.y, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        kr[H + i] = ku.load(i);
        if (i >= kChainRows && i < 2 * kChainRows) st[i % kChainRows] = rows.load(i % kChainRows, ahead);
        __builtin_amdgcn_sched_barrier(0);
    }
    ku.advance();
}

// Model ISF E[i][t] of one (tau block, member group) task on one wavefront:
// E = sum over the concatenated genome (positive sign, then negative sign)
// as one sequential FMA chain per (member, tau) starting from zero
// (matrix_multiply_LxM_by_MxN called twice, deac.cpp:1386-1394), 64 chains
// (16 tau x 4 members) advanced 4 positions per v_mfma_f64_4x4x4_4b_f64, which
// is bit for bit four fused multiply-adds in ascending position order: block b
// holds tau rows 4b..4b+3 of the task, every block the same 4 members.  A:
// lane l holds tau row l&15 at position l>>4 of the MFMA's four; B: member l&3
// at the same position (the same for the four blocks).  buf: kChainLds
// doubles of LDS of this wavefront.
//
// Bound: the chain, 8.8 ns per dependent MFMA (18 us at 8192 positions).  The
// wavefront brings its own operands: K, tiled in operand order, straight
// into a ring of registers, the genome rows by coalesced loads through LDS,
// which puts them in operand order.  Nothing is shared between wavefronts, so
// no barrier sits in the chain.  Measured per 8 positions: the MFMAs alone
// 17.2 ns, genome operands loaded lane by lane from the rows 25 (75 with four
// wavefronts on the CU, the L1 takes 45 cycles for such a load), 16-byte genome
// loads put in order by v_permlane swaps 45, chunks staged by helper
// wavefronts with a barrier per 128 positions 34.
__device__ __forceinline__ void chain_task(const EvoArgs &a, const GenomeRows &rows, int tb, int mg, double *buf)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int nchunk = a.stride / kChunk;
    KUnits ku(a.ktile + static_cast<size_t>(tb) * nchunk * kChunkUnits * (2 * kWave));
    double *to_even = buf + 2 * lane, *to_odd = to_even + kChainRows * kSRow;
    const double *even = buf + (lane & 3) * kSRow + (lane >> 4), *odd = even + kChainRows * kSRow;
    dvec2 s0[kChainRows], s1[kChainRows];
    dvec2 kr[kRing], sr[kReadAhead];
    auto load = [&](int c, dvec2 (&st)[kChainRows]) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < kChainRows; m++) st[m] = rows.load(m, min(c, nchunk - 1));
        __builtin_amdgcn_sched_barrier(0);
    };
    // the loads in about the order of the loop, whose waits hold for its first
    // turn as well
    auto fill = [&](int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kChunkUnits; i++) {
            kr[h + i] = ku.load(i);
            __builtin_amdgcn_sched_barrier(0);
        }
        ku.advance();
    };
    load(0, s0);
    load(1, s1);
    fill(0);
#pragma unroll
    for (int m = 0; m < kChainRows; m++) *reinterpret_cast<dvec2 *>(to_even + m * kSRow) = s0[m];
    load(2, s0);
    fill(kChunkUnits);
#pragma unroll
    for (int j = 0; j < kReadAhead; j++) sr[j] = dvec2{even[j * kUnit], even[j * kUnit + 4]};
    double acc = 0.0;
    // two chunks a turn and an odd one behind the loop: with an exit between
    // the two the waits let 19 loads stay in flight, not 39
    for (int c = 0; c + 1 < nchunk; c += 2) {
        chain_chunk<0>(acc, kr, sr, ku, even, odd, s1, rows, to_odd, min(c + 3, nchunk - 1));
        chain_chunk<kChunkUnits>(acc, kr, sr, ku, odd, even, s0, rows, to_even, min(c + 4, nchunk - 1));
    }
    if (nchunk & 1) chain_chunk<0>(acc, kr, sr, ku, even, odd, s1, rows, to_odd, nchunk - 1);
    // 4x4x4_4b output: lane l holds row l>>4 of block (l>>2)&3, column l&3
    const int i = mg * kChainRows + (lane & 3), t = tb * kChainTau + 4 * ((lane >> 2) & 3) + (lane >> 4);
    if (i < a.P && t < a.T) a.emod[static_cast<size_t>(i) * a.T + t] = acc;
}

// ---- chains whose genome rows the workgroup forms as they run

__device__ __forceinline__ unsigned uniform(unsigned x) { return __builtin_amdgcn_readfirstlane(x); }

// Three wavefronts form the trial vectors of the group's members, every third
// chunk each, into a ring of chunks in LDS; the chain's wavefront follows.
// ready[slot] is the chunk in a slot of the ring, counted since the launch
// began, plus one; used the chunks that the chain is done with.
constexpr int kFedSlots = 8;
constexpr int kFeeders = kEvoWaves - 1;
constexpr int kFedAhead = 2;  // chunks whose loads a feeder has in flight
constexpr int kFedChunk = kChainRows * kSRow;
static_assert(kFedSlots * kFedChunk <= kEvoWaves * kChainLds, "the ring fits in front of the members' state");
struct Feed {
    double *ring;
    unsigned *ready, *used;
    __device__ __forceinline__ double *slot(unsigned n) const { return ring + n % kFedSlots * kFedChunk; }
    static __device__ __forceinline__ unsigned read(const unsigned *p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    static __device__ __forceinline__ void write(unsigned *p, unsigned v)
    {
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

// Until *p is at least need; there: what it held a while ago.  One piece of
// assembly, so that the chain around it stays one block of code (as a loop in
// the source it cost register copies and a wait for all loads in flight).  The
// feeders never wait for anything but chunks used, so that the wait ends.
__device__ __forceinline__ void await(const unsigned *p, unsigned there, unsigned need)
{
    typedef const __attribute__((address_space(3))) unsigned *Lds;
    const unsigned at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((Lds)p));
    unsigned v, u;
    asm volatile("s_cmp_ge_u32 %2, %3\n\t"
                 "s_cbranch_scc1 2f\n"
                 "1:\n\t"
                 "ds_read_b32 %0, %4\n\t"
                 "s_waitcnt lgkmcnt(0)\n\t"
                 "v_readfirstlane_b32 %1, %0\n\t"
                 "s_cmp_ge_u32 %1, %3\n\t"
                 "s_cbranch_scc0 1b\n"
                 "2:"
                 : "=&v"(v), "=&s"(u)
                 : "s"(there), "s"(need), "v"(at)
                 : "scc", "memory");
}

// chain_chunk on the ring: chunk n of the launch; more: another one follows.
template <int H>
__device__ __forceinline__ void fed_chunk(double &acc, dvec2 (&kr)[kRing], dvec2 (&sr)[kReadAhead], KUnits &ku,
                                          const Feed &f, unsigned n, int offset, bool more)
{
    const double *here = f.slot(n) + offset, *next = f.slot(n + 1) + offset;
    const unsigned need = more ? n + 2 : 0;
    unsigned there = 0;
#pragma unroll
    for (int i = 0; i < kChunkUnits; i++) {
        const dvec2 k = kr[H + i], s = sr[i % kReadAhead];
        const int j = i + kReadAhead;
        const double *p = j < kChunkUnits ? here + j * kUnit : next + (j - kChunkUnits) * kUnit;
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(k.x, s.x, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (i == kChunkUnits - 2 * kReadAhead) there = Feed::read(f.ready + (n + 1) % kFedSlots);
        if (j == kChunkUnits) {  // from here on the reads are of the next chunk
            await(f.ready + (n + 1) % kFedSlots, uniform(there), need);
            Feed::write(f.used, n + 1);
        }
        sr[i % kReadAhead] = dvec2{p[0], p[4]};
        __builtin_amdgcn_sched_barrier(0);
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(k.y, s.y, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        kr[H + i] = ku.load(i);
        __builtin_amdgcn_sched_barrier(0);
    }
    ku.advance();
}

// chain_task on the ring, from chunk n0 of the launch on.
__device__ __forceinline__ void fed_chain(const EvoArgs &a, double *emod, int tb, int mg, const Feed &f, unsigned n0)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int nchunk = a.stride / kChunk, offset = (lane & 3) * kSRow + (lane >> 4);
    KUnits ku(a.ktile + static_cast<size_t>(tb) * nchunk * kChunkUnits * (2 * kWave));
    dvec2 kr[kRing], sr[kReadAhead];
#pragma unroll
    for (int h = 0; h < kRing; h += kChunkUnits) {
#pragma unroll
        for (int i = 0; i < kChunkUnits; i++) {
            kr[h + i] = ku.load(i);
            __builtin_amdgcn_sched_barrier(0);
        }
        ku.advance();
    }
    await(f.ready + n0 % kFedSlots, n0, n0 + 1);
    const double *first = f.slot(n0) + offset;
#pragma unroll
    for (int j = 0; j < kReadAhead; j++) sr[j] = dvec2{first[j * kUnit], first[j * kUnit + 4]};
    double acc = 0.0;
    for (int c = 0; c + 1 < nchunk; c += 2) {
        fed_chunk<0>(acc, kr, sr, ku, f, n0 + c, offset, true);
        fed_chunk<kChunkUnits>(acc, kr, sr, ku, f, n0 + c + 1, offset, c + 2 < nchunk);
    }
    if (nchunk & 1) fed_chunk<0>(acc, kr, sr, ku, f, n0 + nchunk - 1, offset, false);
    const int i = mg * kChainRows + (lane & 3), t = tb * kChainTau + 4 * ((lane >> 2) & 3) + (lane >> 4);
    if (i < a.P && t < a.T) emod[static_cast<size_t>(i) * a.T + t] = acc;
}

typedef unsigned raw_quad __attribute__((ext_vector_type(4)));

// Chunks feeder, feeder + 3, ... of the group's trial vectors (deac.cpp:
// 1261-1308) into the ring, from chunk n0 of the launch on, and into the spare
// rows where this workgroup writes them.  ctl: the members' records; raw: the
// generation's draws.
//
// Bound: the operands (36 KB a chunk with the chain's: 407 ns, the chain alone
// needs 281), and a feeder's instruction issue, so what a sign's or the genome's
// end needs stands aside (8 members, G = 4096, T = 65: 34.1 us a generation;
// 35.3 with a step of 390 instructions in place of 190; 39.5 with the barrier's
// fences replaced by loads and stores past the caches; 38.6 with flat
// addresses).  Rows are byte offsets from pop0 (both populations are one allocation) in buffer operations:
// flat ones would have to be waited for at every LDS operation.
__device__ __forceinline__ void feed_chain(const EvoArgs &a, const Members &s, const MemberCtl (&ctl)[kChainRows],
                                           const uint64_t *raw, int mg, bool write, int feeder, const Feed &f, unsigned n0)
{
    const int lane = threadIdx.x & (kWave - 1), nchunk = a.stride / kChunk;
    if (feeder >= nchunk) return;
    const auto pop = __builtin_amdgcn_make_buffer_rsrc(a.pop0, 0, -1, 0x00020000);
    const auto draws = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint64_t *>(raw), 0, -1, 0x00020000);
    const unsigned span = static_cast<unsigned>(reinterpret_cast<uintptr_t>(a.pop1) - reinterpret_cast<uintptr_t>(a.pop0));
    struct Row {
        unsigned r1, r2, r3, rp, out, u;  // byte offsets
        double f0, f1;
        uint64_t lim0, lim1;
    } row[kChainRows];
    auto offset_of = [&](unsigned i, bool spare) __attribute__((always_inline)) {
        const unsigned j = uniform(i);
        return ((uniform(static_cast<unsigned>(s.cur[j])) != 0) != spare ? span : 0) + j * static_cast<unsigned>(a.stride) * 8;
    };
#pragma unroll
    for (int m = 0; m < kChainRows; m++) {
        const int i = min(mg * kChainRows + m, a.P - 1);
        Row &r = row[m];
        r.r1 = offset_of(ctl[m].mutant[0], false);
        r.r2 = offset_of(ctl[m].mutant[1], false);
        r.r3 = offset_of(ctl[m].mutant[2], false);
        r.rp = offset_of(i, false);
        r.out = offset_of(i, true);
        r.u = static_cast<unsigned>(i) * static_cast<unsigned>(a.rstride) * 8;
        const Controls c(a, s, ctl[m], i);
        r.f0 = c.f[0];
        r.f1 = c.f[1];
        r.lim0 = cross_limit(c.cr[0]);
        r.lim1 = cross_limit(c.cr[1]);
    }
    const unsigned sign_mask = a.allow_neg ? ~0u : 0x7fffffffu;
    auto value = [&](double fm, uint64_t lim, uint64_t u, double d1, double d2, double d3, double p)
                     __attribute__((always_inline)) {
        const uint64_t w = __builtin_bit_cast(uint64_t, fma(fm, d2 - d3, d1));
        const uint64_t x = static_cast<uint64_t>(static_cast<unsigned>(w >> 32) & sign_mask) << 32 | static_cast<unsigned>(w);
        return u < lim ? __builtin_bit_cast(double, x) : p;
    };
    const int vo = lane * 16, last = ((a.Kc - 1) & ~1) * 8;
    auto load = [&](int m, int c, Trial::Load &v) __attribute__((always_inline)) {
        const int so = min(c, nchunk - 1) * (kChunk * 8);
        auto pair = [&](unsigned r) __attribute__((always_inline)) {
            return __builtin_bit_cast(dvec2, __builtin_amdgcn_raw_buffer_load_b128(pop, vo, r + so, 0));
        };
        v.u = __builtin_bit_cast(uvec2, __builtin_amdgcn_raw_buffer_load_b128(draws, min(so + vo, last), row[m].u, 0));
        v.x1 = pair(row[m].r1);
        v.x2 = pair(row[m].r2);
        v.x3 = pair(row[m].r3);
        v.xp = pair(row[m].rp);
    };
    // the trial's value at the zero frequency, which the negative sign repeats
    double zero[kChainRows];
    {
        double x[kChainRows][4];
        uint64_t u[kChainRows];
        auto one = [&](unsigned r) __attribute__((always_inline)) {
            return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(pop, 0, r, 0));
        };
#pragma unroll
        for (int m = 0; m < kChainRows; m++) {
            u[m] = __builtin_bit_cast(uint64_t, __builtin_amdgcn_raw_buffer_load_b64(draws, 0, row[m].u, 0));
            x[m][0] = one(row[m].r1);
            x[m][1] = one(row[m].r2);
            x[m][2] = one(row[m].r3);
            x[m][3] = one(row[m].rp);
        }
#pragma unroll
        for (int m = 0; m < kChainRows; m++)
            zero[m] = value(row[m].f0, row[m].lim0, u[m], x[m][0], x[m][1], x[m][2], x[m][3]);
    }
    Trial::Load v[kFedAhead][kChainRows];
#pragma unroll
    for (int u = 0; u < kFedAhead; u++)
#pragma unroll
        for (int m = 0; m < kChainRows; m++) load(m, feeder + u * kFeeders, v[u][m]);
    auto step = [&](Trial::Load (&x)[kChainRows], int c) __attribute__((always_inline)) {
        const unsigned n = n0 + c;
        while (static_cast<int>(n - uniform(Feed::read(f.used))) >= kFedSlots) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
        const bool neg = c * kChunk >= a.G;
        dvec2 o[kChainRows];
#pragma unroll
        for (int m = 0; m < kChainRows; m++) {
            const double fm = neg ? row[m].f1 : row[m].f0;
            const uint64_t lim = neg ? row[m].lim1 : row[m].lim0;
            o[m].x = value(fm, lim, x[m].u.x, x[m].x1.x, x[m].x2.x, x[m].x3.x, x[m].xp.x);
            o[m].y = value(fm, lim, x[m].u.y, x[m].x1.y, x[m].x2.y, x[m].x3.y, x[m].xp.y);
        }
        if ((c * kChunk <= a.G && (c + 1) * kChunk > a.G) || (c + 1) * kChunk > a.Kc) {
            // where a sign begins inside the chunk, or the genome ends
            const int k = Trial::position(c);
#pragma unroll
            for (int m = 0; m < kChainRows; m++) {
                const Row &r = row[m];
                if (k >= a.G) o[m].x = value(r.f1, r.lim1, x[m].u.x, x[m].x1.x, x[m].x2.x, x[m].x3.x, x[m].xp.x);
                if (k + 1 >= a.G) o[m].y = value(r.f1, r.lim1, x[m].u.y, x[m].x1.y, x[m].x2.y, x[m].x3.y, x[m].xp.y);
                if (k == a.G) o[m].x = zero[m];
                if (k + 1 == a.G) o[m].y = zero[m];
                if (k >= a.Kc) o[m].x = 0.0;
                if (k + 1 >= a.Kc) o[m].y = 0.0;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < kChainRows; m++) load(m, c + kFedAhead * kFeeders, x[m]);
        __builtin_amdgcn_sched_barrier(0);
        dvec2 *to = reinterpret_cast<dvec2 *>(f.slot(n)) + lane;
#pragma unroll
        for (int m = 0; m < kChainRows; m++) to[m * (kSRow / 2)] = o[m];
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // the rows are in LDS (lgkmcnt 0, the other counters as they are)
        Feed::write(f.ready + n % kFedSlots, n + 1);
        if (write) {
#pragma unroll
            for (int m = 0; m < kChainRows; m++)
                if (mg * kChainRows + m < a.P)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(raw_quad, o[m]), pop, vo,
                                                           row[m].out + c * (kChunk * 8), 0);
        }
    };
    // (two chunks a turn and an odd one behind: an exit between them costs
    // copies of the loads in flight)
    static_assert(kFedAhead == 2);
    int c = feeder;
    for (; c + kFeeders < nchunk; c += 2 * kFeeders) {
        step(v[0], c);
        step(v[1], c + kFeeders);
    }
    if (c < nchunk) step(v[0], c);
}

// Blocks [b0, b1) of a trial vector into the spare row, two blocks' loads
// ahead of the two being formed.
// Bound: memory (40 bytes read and 8 written per position): 512 members of
// 8192 positions take 46 us with the top of the generation and the barrier
// (4.4 TB/s; a large copy reaches 4.7).  With a cache write-back per workgroup at
// the barrier it was 67, with runs of 8 blocks and nothing read ahead 96.
__device__ __forceinline__ void trial_blocks(const Trial &t, int b0, int b1)
{
    typedef Trial::Load Load;
    Load v0 = {}, v1 = {}, w0 = {}, w1 = {};
    auto two = [&](int b, Load &x, Load &y) __attribute__((always_inline)) {
        if (b < b1) t.load(b, x);
        if (b + 1 < b1) t.load(b + 1, y);
    };
    auto put = [&](int b, const Load &x, const Load &y) __attribute__((always_inline)) {
        t.store(b, t.form(b, x));
        if (b + 1 < b1) t.store(b + 1, t.form(b + 1, y));
    };
    two(b0, v0, v1);
    for (int b = b0;; b += 4) {
        two(b + 2, w0, w1);
        put(b, v0, v1);
        if (b + 2 >= b1) break;
        two(b + 4, v0, v1);
        put(b + 2, w0, w1);
        if (b + 4 >= b1) break;
    }
}

// A trial vector and its zeroth moment (deac.cpp:1342-1352) by one workgroup:
// waves 1 to 3 form the blocks of one stage, store them and leave their products
// in LDS while wave 0 folds the stage before.  Returns the moment in wave 0.
// buf: 2 stages in LDS.
// Bound: the fold's chain of MFMAs, 9 us at 4096 positions.  The trial phase
// took 25 us there with trial, fold and scaling one after the other, 29 with
// the fold's wave forming the trial as it went; 20.5 this way.
constexpr int kStageBlocks = 9;
constexpr int kStage = kStageBlocks * kChunk;
static_assert(kStageBlocks % (kEvoWaves - 1) == 0 && kFoldBlock == kChunk);
static_assert(2 * kStage <= kEvoWaves * kChainLds, "the stages fit in front of the members' state");

__device__ __forceinline__ double trial_fold(const Trial &t, const double *w, int nblk, double *buf)
{
    constexpr int kEach = kStageBlocks / (kEvoWaves - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    const int Kc = t.a.Kc, G = t.a.G, nstage = (nblk + kStageBlocks - 1) / kStageBlocks;
    const bool godd = (G & 1) != 0;
    double acc = 0.0;
    for (int c = -1; c < nstage; c++) {
        if (wid == 0 && c >= 0) {
            FoldFused f = {{-1, -1}, {1.0, 1.0}};
            if (godd) {
                f.w[0] = w[G - 1];
                f.w[1] = w[Kc - 1];
            }
            const double *here = buf + (c & 1) * kStage + (lane >> 4);
            fold_pair v[kFoldAhead];
#pragma unroll
            for (int u = 0; u < kFoldAhead; u++) v[u] = fold_pair{here[8 * u], here[8 * u + 4]};
            const int b0 = c * kStageBlocks, b1 = min(b0 + kStageBlocks, nblk);
            for (int b = b0; b < b1; b++, here += kChunk) {
                // (a stage's last block reads ahead into its own start)
                const double *next = b + 1 < b1 ? here + kChunk : here;
                f.k[0] = godd ? G - 1 - b * kChunk : -1;
                f.k[1] = godd ? Kc - 1 - b * kChunk : -1;
                const bool fused = (f.k[0] >= 0 && f.k[0] < kChunk) || (f.k[1] >= 0 && f.k[1] < kChunk);
                if (fused) fold_block<true>(acc, v, here, next, f);
                else fold_block<false>(acc, v, here, next, f);
            }
        }
        if (wid != 0 && c + 1 < nstage) {
            Trial::Load v[kEach] = {};
            dvec2 wk[kEach];
            const int j0 = (wid - 1) * kEach, b0 = (c + 1) * kStageBlocks + j0;
#pragma unroll
            for (int j = 0; j < kEach; j++)
                if (b0 + j < nblk) {
                    t.load(b0 + j, v[j]);
                    wk[j] = *reinterpret_cast<const dvec2 *>(w + min(Trial::position(b0 + j), (Kc - 1) & ~1));
                }
#pragma unroll
            for (int j = 0; j < kEach; j++)
                if (b0 + j < nblk) {
                    const int k = Trial::position(b0 + j);
                    const dvec2 x = t.form(b0 + j, v[j]);
                    t.store(b0 + j, x);
                    dvec2 p = x * wk[j];
                    if (godd) {  // a fused element's first factor in place of its product
                        if (k == G - 1 || k == Kc - 1) p.x = x.x;
                        if (k + 1 == G - 1 || k + 1 == Kc - 1) p.y = x.y;
                    }
                    if (k >= Kc) p.x = 0.0;
                    if (k + 1 >= Kc) p.y = 0.0;
                    reinterpret_cast<dvec2 *>(buf + ((c + 1) & 1) * kStage + (j0 + j) * kChunk)[lane] = p;
                }
        }
        if (c == nstage - 1) __builtin_amdgcn_s_waitcnt(0);  // the trial, before it is scaled
        __syncthreads();
    }
    return acc;
}

// Blocks [b0, b1) of a row times a factor.
__device__ __forceinline__ void scale_blocks(double *x, double scale, int b0, int b1)
{
    dvec2 *p = reinterpret_cast<dvec2 *>(x) + (threadIdx.x & (kWave - 1));
#pragma unroll 8
    for (int b = b0; b < b1; b++) p[b * (kChunk / 2)] = p[b * (kChunk / 2)] * scale;
}

// Lowest fitness as the reference's scan finds it (deac.cpp:128-138: the first
// of equal ones, no value but the first may be NaN), by one whole wavefront.
__device__ __forceinline__ double lowest(const double *fit, int P)
{
    double mn = fit[0];
    if (P <= 32) {  // (64 values take 0.4 us in a row, 0.6 in parallel)
        for (int i = 1; i < P; i++) mn = fit[i] < mn ? fit[i] : mn;
        return mn;
    }
    const double first = mn;
    int at = 0;
    for (int i = threadIdx.x & (kWave - 1); i < P; i += kWave) {
        const double v = fit[i];
        if (v < mn) {
            mn = v;
            at = i;
        }
    }
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
        const double v = __shfl_xor(mn, m);
        const int i = __shfl_xor(at, m);
        if (v < mn || (v == mn && i < at)) {
            mn = v;
            at = i;
        }
    }
    return first != first ? first : mn;
}

// Mean and squared mean of the fitnesses of generation g in the reference's
// order (deac.cpp:1145-1160), by one wavefront: staged in its LDS (kChainLds
// doubles), 8 values read ahead.
__device__ __forceinline__ void statistics(const EvoArgs &a, const double *fit, int g, double mn, double *buf)
{
    const int lane = threadIdx.x & (kWave - 1);
    constexpr int kWindow = kChainLds & ~7;
    double sum = 0.0, sq = 0.0;
    const int p4 = a.P & ~3;
    for (int w0 = 0; w0 < a.P; w0 += kWindow) {
        const int n = min(kWindow, a.P - w0);
        for (int i = lane; i < n; i += kWave) buf[i] = fit[w0 + i];
        asm volatile("" ::: "memory");  // (one wavefront: LDS keeps its order)
        for (int i0 = 0; i0 < n; i0 += 8) {
            double v[8];
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = buf[min(i0 + e, n - 1)];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (i0 + e >= n) break;
                sum = sum + v[e];
                sq = w0 + i0 + e < p4 ? sq + v[e] * v[e] : fma(v[e], v[e], sq);
            }
        }
        asm volatile("" ::: "memory");
    }
    const long ii = a.gen0 + g;
    if (lane == 0) {
        a.stats[ii] = sum / static_cast<double>(a.P);
        a.stats[a.stats_len + ii] = mn;
        a.stats[2 * a.stats_len + ii] = sq / static_cast<double>(a.P);
    }
}

// acc + the products w[0..n) added in tau order from LDS: the -1st moment
// (deac.cpp:1398-1416), whose last product is fused where T is odd.
__device__ __forceinline__ double product_sum(const EvoArgs &a, const double *w, int i, int t0, int n, double acc)
{
    const bool fused = (a.T & 1) && t0 + n == a.T;
    const int m = fused ? n - 1 : n;
    int t = 0;
    for (; t + 8 <= m; t += 8) {
        double v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = w[t + e];
#pragma unroll
        for (int e = 0; e < 8; e++) acc = acc + v[e];
    }
    for (; t < m; t++) acc = acc + w[t];
    if (fused) acc = fma(a.emod[static_cast<size_t>(i) * a.T + a.T - 1], a.nfm_dt[a.T - 1], acc);
    return acc;
}

// The greedy selection of a member (deac.cpp:1556-1571), by one lane: what it
// needs beside the new fitness is loaded ahead of the sums.
struct Selection {
    const EvoArgs &a;
    const Members &s;
    int i;
    bool init;
    double old, first, third;
    Controls next;
    __device__ __forceinline__ Selection(const EvoArgs &ea, const Members &members, int g, int member, bool initial)
        : a(ea), s(members), i(member), init(initial), old(s.fitness[i]), first(a.use_first ? a.mom[i * 4 + 1] : 0.0),
          third(a.use_third ? a.mom[i * 4 + 2] : 0.0)
    {
        // (the initial fitness has no control records)
        if (!init) next = Controls(a, s, a.ctl[static_cast<size_t>(g) * a.P + i], i);
    }
    // from the chi^2 sum and the -1st moment (deac.cpp:957-976, 1539-1555)
    __device__ __forceinline__ void take(double chi, double nfm) const
    {
        double fit = chi / static_cast<double>(a.T);
        if (a.use_nfm) {
            const double q = (a.nfm_value - nfm) / a.nfm_error;
            fit = fma(q, q, fit);
        }
        if (a.use_first) {
            const double d = first - a.first_moment;
            fit += (d * d) / a.first_moment;
        }
        if (a.use_third) {
            const double q = (a.third_moment - third) / a.third_moment_error;
            fit = fma(q, q, fit);
        }
        if (init) {
            s.fitness[i] = fit;
        } else if (fit <= old) {
            s.fitness[i] = fit;
            s.cur[i] ^= 1;
            for (int sg = 0; sg < a.nsign; sg++) {
                s.cr[i * a.nsign + sg] = sg ? next.cr[1] : next.cr[0];
                s.f[i * a.nsign + sg] = sg ? next.f[1] : next.f[0];
            }
        }
    }
};

}  // namespace

// Phase timestamps (s_memtime) of workgroup 0, compiled in only for
// profiling builds: slot 0 top of generation, 1 after the trial barrier,
// 2 after the chain barrier, 3 after the selection.
#ifdef DEAC_PHASE_TIMERS
__device__ unsigned long long deac_phase_clock[4];
#define DEAC_PHASE(slot)                                                                      \
    do {                                                                                      \
        if (blockIdx.x == 0 && threadIdx.x == 0 && !init) {                                   \
            const unsigned long long now = clock64();                                         \
            if (slot == 0) phase_t0 = now;                                                     \
            else atomicAdd(&deac_phase_clock[slot], now - phase_t0), phase_t0 = now;           \
        }                                                                                     \
    } while (0)
#else
#define DEAC_PHASE(slot) \
    do {                 \
    } while (0)
#endif

// Per generation: trial vectors, barrier, chains and moment rows, barrier,
// selection.  Where the population's residuals fit in LDS (a.local) every
// workgroup repeats the whole selection and keeps the members' state itself,
// which saves the third barrier: a grid barrier costs 1 us, a repeated selection
// of 8 members 1.3 us.  One workgroup per CU is launched
// (evolve_max_workgroups); a second handle's workgroup still fits beside it.
// FOLD: the trials' model ISF as rounded-product folds (bdsf; its initial
// population goes through the chains of the other form, deac.cpp:860).
// FED (EvoArgs::fed): a workgroup per contraction task, and one for the
// statistics, which forms the trial vectors of its members beside their chains:
// no trial phase, one barrier per generation.
enum Form { kChains, kFold, kFed };
template <Form FORM>
__global__ __launch_bounds__(kEvoThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void evolve_kernel(EvoArgs a, WalkArgs next,
                                                                                              MaskArgs masks)
{
#ifdef DEAC_PHASE_TIMERS
    unsigned long long phase_t0 = 0;
#endif
    constexpr bool FOLD = FORM == kFold, FED = FORM == kFed;
    extern __shared__ __attribute__((aligned(16))) double lds[];
    __shared__ double minimum, scale;
    const int lane = threadIdx.x & (kWave - 1);
    // the wave index as a scalar: what depends on it alone is then uniform
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int nwg = a.nwg;
    if (blockIdx.x >= nwg) {
        // the workgroups behind the evolution's draw for the batches to come
        // and take no part in the barriers: the walk, then the masks
        const int behind = blockIdx.x - nwg - (next.ngen > 0 ? 1 : 0);
        if (behind >= 0)
            mask_draws(masks, static_cast<size_t>(wid) * masks.nwg + behind,
                       static_cast<size_t>(masks.nwg) * kEvoWaves, lds + wid * kMaskLds);
        else if (wid == 0)
            walk(next, reinterpret_cast<uint64_t *>(lds));
        return;
    }
    if (blockIdx.x == 0 && a.clear)
        for (int i = threadIdx.x; i < kSyncWords; i += kEvoThreads) a.clear[i] = 0;
    const int total_waves = nwg * kEvoWaves;
    // Waves are numbered wave-slot-major so that consecutive tasks land on
    // different workgroups (and CUs).
    const int gwave = wid * nwg + blockIdx.x;
    GridBarrier barrier(a);
    if (a.xbar && nwg >= kXcdBarrierWgs && !barrier.by_xcd()) return;
    // The contraction's tasks and the moment folds of this workgroup's XCD
    // (workgroups go to the XCDs in turn), in equal ranges: neighbouring tasks
    // share a tau block's K or a member group's rows in its L2.
    const int nx = min(kXcds, nwg), xcd = blockIdx.x % nx;
    const int xwg = (nwg - xcd + nx - 1) / nx, xwave = wid * xwg + blockIdx.x / nx;  // workgroups here, this wave
    const int before = xcd * (nwg / nx) + min(xcd, nwg % nx);                        // workgroups of lower XCDs
    const int groups = FOLD ? a.P : a.MG;
    const int nmom = a.use_first + a.use_third;  // moment folds per member
    auto share = [&](int all, int wgs) { return static_cast<int>(static_cast<long>(all) * wgs / nwg); };
    const int ks0 = share(groups * a.TB, before), nks = share(groups * a.TB, before + xwg) - ks0;
    const int mom0 = share(nmom * a.P, before), nmoms = share(nmom * a.P, before + xwg) - mom0;
    const int nblk = a.stride / kChunk;
    // This wave's share of the trials' blocks: equal shares, across members.
    // (In runs of 8 blocks of one member, 4096 of them for 992 waves, the fifth
    // round was nearly empty.)
    const size_t blocks = static_cast<size_t>(a.P) * nblk;
    const int share0 = static_cast<int>(gwave * blocks / total_waves);
    const int nshare = static_cast<int>((gwave + 1) * blocks / total_waves) - share0;
    const int share_i = share0 / nblk, share_b = share0 % nblk;
    const int Tp = a.T | 1;  // odd row stride: lanes of different members read different banks

    Members s = {a.fitness, a.cr_old, a.f_old, a.cur};
    // Where each member's current genome is: a copy in LDS of the members' state
    // in global memory where it fits.
    const bool copy = !a.local && a.P <= 2 * kResidLds;
    // [P][Tp] residuals and -1st-moment products (a.local), behind the chains' buffers
    double *resid = lds + kEvoWaves * kChainLds;
    double *moment = resid + static_cast<size_t>(a.P) * Tp;
    if (a.local) {
        s.fitness = moment + (a.use_nfm ? static_cast<size_t>(a.P) * Tp : 0);
        s.cr = s.fitness + a.P;
        s.f = s.cr + a.P * a.nsign;
        s.cur = reinterpret_cast<int *>(s.f + a.P * a.nsign);
        for (int i = threadIdx.x; i < a.P; i += kEvoThreads) {
            s.cur[i] = a.cur[i];
            s.fitness[i] = a.fitness[i];
            for (int sg = 0; sg < a.nsign; sg++) {
                s.cr[i * a.nsign + sg] = a.cr_old[i * a.nsign + sg];
                s.f[i * a.nsign + sg] = a.f_old[i * a.nsign + sg];
            }
        }
    }
    const int *cur = s.cur;
    __shared__ unsigned fed_ready[kFedSlots], fed_used;
    const Feed feed = {lds, fed_ready, &fed_used};
    // FED: this workgroup's task; one workgroup has none.  The members' records
    // are put into LDS a generation ahead.
    const int fed_task = ks0 + static_cast<int>(blockIdx.x) / nx;
    const int fed_tb = a.by_tau ? fed_task / groups : fed_task % a.TB, fed_mg = a.by_tau ? fed_task % groups : fed_task / a.TB;
    const bool fed_mine = static_cast<int>(blockIdx.x) / nx < nks;
    __shared__ MemberCtl fed_ctl[2][kChainRows];
    auto records = [&](int g) {
        constexpr int kWords = sizeof(MemberCtl) / sizeof(uint64_t);
        static_assert(kChainRows * kWords <= kWave);
        const int m = lane / kWords;
        const MemberCtl *from = a.ctl + static_cast<size_t>(min(g, a.ngen - 1)) * a.P;
        if (m < kChainRows)
            reinterpret_cast<uint64_t *>(fed_ctl[g & 1])[lane] =
                reinterpret_cast<const uint64_t *>(from + min(fed_mg * kChainRows + m, a.P - 1))[lane % kWords];
    };
    if constexpr (FED) {
        if (threadIdx.x < kFedSlots) fed_ready[threadIdx.x] = 0;
        if (threadIdx.x == 0) fed_used = 0;
        if (wid == 1) records(0);
    }
    __syncthreads();

    for (int g = 0; g <= a.ngen; g++) {
        const bool init = !FOLD && a.init_mode != 0;
        if (!init) {
            if (g == a.ngen) break;
            DEAC_PHASE(0);
            // Top of the generation: best fitness and stop test
            // (deac.cpp:1145-1166); the statistics are left to the chains'
            // phase, which one wave's scan does not lengthen.
            if (copy) {
                int *to = reinterpret_cast<int *>(resid);
                for (int i = threadIdx.x; i < a.P; i += kEvoThreads) to[i] = a.cur[i];
                cur = to;
            }
            if (wid == 0) {
                const double mn = lowest(s.fitness, a.P);
                if (lane == 0) minimum = mn;
            }
            __syncthreads();
            if (minimum <= a.stop) {
                if (blockIdx.x == 0 && wid == 0) {
                    if (a.track_stats) statistics(a, s.fitness, g, minimum, lds);
                    if (lane == 0) {
                        a.status[1] = g;
                        __hip_atomic_store(a.status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        tell_host(a.host_status, 1, g);
                        tell_host(a.host_status, 0, 1);
                    }
                }
                break;
            }

            // Trial vectors into each member's spare buffer.
            const MemberCtl *ctlg = a.ctl + static_cast<size_t>(g) * a.P;
            const uint64_t *rawg = a.raw + static_cast<size_t>(g) * a.P * a.rstride;
            if constexpr (FED) {
                // beside the chains, below
            } else if (!a.renorm) {
                for (int i = share_i, b0 = share_b, left = nshare; left > 0; i++, b0 = 0) {
                    const int n = min(nblk - b0, left);
                    trial_blocks(Trial(a, s, cur, ctlg[i], rawg + static_cast<size_t>(i) * a.rstride, i), b0, b0 + n);
                    left -= n;
                }
            } else {
                // With per-generation renormalization (deac.cpp:1342-1364) a
                // workgroup takes whole members, or where there are more
                // members than workgroups every wave has one of its own.
                const bool alone = a.P > nwg;
                for (int i = alone ? gwave : static_cast<int>(blockIdx.x); i < a.P; i += alone ? total_waves : nwg) {
                    const Trial t(a, s, cur, ctlg[i], rawg + static_cast<size_t>(i) * a.rstride, i);
                    if (alone) {
                        trial_blocks(t, 0, nblk);
                        __builtin_amdgcn_s_waitcnt(0);
                        scale_blocks(t.out, a.zeroth / wave_fold(t.out, a.nterm, a.Kc, a.G, lds + wid * kChainLds), 0,
                                     nblk);
                        continue;
                    }
                    const double norm = trial_fold(t, a.nterm, nblk, lds);
                    if (threadIdx.x == 0) scale = a.zeroth / norm;
                    __syncthreads();
                    const int share = (nblk + kEvoWaves - 1) / kEvoWaves;
                    scale_blocks(t.out, scale, min(wid * share, nblk), min((wid + 1) * share, nblk));
                    __syncthreads();
                }
            }
            if constexpr (!FED) {
                if (!barrier.wait()) return;
                DEAC_PHASE(1);
            }
        }

        // FED: a workgroup may still select from a generation's model ISF while
        // the next one's chains end.
        double *const emod = FED && (g & 1) ? a.emod + static_cast<size_t>(a.P) * a.T : a.emod;
        if constexpr (FED) {
            const unsigned n0 = static_cast<unsigned>(g) * nblk;
            if (fed_mine) {
                if (wid == 0) {
                    fed_chain(a, emod, fed_tb, fed_mg, feed, n0);
                } else {
                    feed_chain(a, s, fed_ctl[g & 1], a.raw + static_cast<size_t>(g) * a.P * a.rstride, fed_mg, fed_tb == 0, wid - 1,
                               feed, n0);
                    if (wid == 1) records(g + 1);
                }
            } else if (wid == 0 && a.track_stats) {
                statistics(a, s.fitness, g, minimum, lds);
            }
        }
        // Model ISF chains and moment rows, one wave per task: of the trials,
        // or of the current genomes for the initial fitness.
        for (int n = FED ? nks + nmoms : xwave; n < nks + nmoms; n += xwg * kEvoWaves) {
            double *buf = lds + wid * kChainLds;
            if (n < nks) {
                const int task = ks0 + n;
                const int tb = a.by_tau ? task / groups : task % a.TB, mg = a.by_tau ? task % groups : task / a.TB;
                if constexpr (FOLD) {
                    const double e = fold_task(a.ktile + static_cast<size_t>(tb) * a.stride * kChainTau,
                                               row_of(a, cur, mg, true), nblk, a.Kc, (a.G & 1) != 0, buf);
                    const int t = tb * kChainTau + 4 * ((lane >> 2) & 3) + (lane >> 4);
                    if ((lane & 3) == 0 && t < a.T) a.emod[static_cast<size_t>(mg) * a.T + t] = e;
                } else {
                    GenomeRows rows;
                    const int first = mg * kChainRows;
                    const int c = cur[min(first + (lane & (kChainRows - 1)), a.P - 1)];
#pragma unroll
                    for (int m = 0; m < kChainRows; m++) {
                        const bool second = (__builtin_amdgcn_readlane(c, m) != 0) == init;
                        rows.row[m] = (second ? a.pop1 : a.pop0) + static_cast<size_t>(min(first + m, a.P - 1)) * a.stride;
                    }
                    rows.vo = lane * 16;
                    chain_task(a, rows, tb, mg, buf);
                }
            } else {
                const int task = mom0 + n - nks, i = task / nmom;
                const bool third = !a.use_first || task % nmom != 0;
                const double m = wave_fold(row_of(a, cur, i, !init), third ? a.tterm : a.fterm, a.Kc, a.G, buf);
                if (lane == 0) a.mom[i * 4 + (third ? 2 : 1)] = m;
            }
        }
        if (!FED && gwave == total_waves - 1 && a.track_stats && !init)
            statistics(a, s.fitness, g, minimum, lds + wid * kChainLds);
        if (!barrier.wait()) return;
        DEAC_PHASE(2);

        // Fitness and greedy selection.
        if (a.local) {
            const int total = a.P * a.T;
            for (int idx = threadIdx.x; idx < total; idx += kEvoThreads) {
                const int i = idx / a.T, t = idx % a.T;
                const double e = emod[idx];
                resid[i * Tp + t] = (a.obs[t] - e) / a.sig[t];
                if (a.use_nfm) moment[i * Tp + t] = e * a.nfm_dt[t];
            }
            __syncthreads();
            for (int i = threadIdx.x; i < a.P; i += kEvoThreads) {
                const Selection sel(a, s, g, i, init);
                const double chi = chi_sum(resid + i * Tp, a.T, a.T & 1, 0.0);
                const double nfm = a.use_nfm ? product_sum(a, moment + i * Tp, i, 0, a.T, 0.0) : 0.0;
                sel.take(chi, nfm);
            }
            __syncthreads();
        } else if constexpr (!FED) {
            // one wavefront per member, residuals in windows
            const int window = a.use_nfm ? kResidWave / 2 : kResidWave;
            double *d = lds + wid * kResidWave, *p = d + window;
            for (int i = gwave; i < a.P; i += total_waves) {
                const Selection sel(a, s, g, i, init);
                double chi = 0.0, nfm = 0.0;
                for (int t0 = 0; t0 < a.T; t0 += window) {
                    const int n = min(window, a.T - t0);
                    for (int u = lane; u < n; u += kWave) {
                        const double e = a.emod[static_cast<size_t>(i) * a.T + t0 + u];
                        d[u] = (a.obs[t0 + u] - e) / a.sig[t0 + u];
                        if (a.use_nfm) p[u] = e * a.nfm_dt[t0 + u];
                    }
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    chi = chi_sum(d, n, (a.T & 1) && t0 + n == a.T, chi);
                    if (a.use_nfm) nfm = product_sum(a, p, i, t0, n, nfm);
                    __builtin_amdgcn_wave_barrier();
                }
                if (lane == 0) sel.take(chi, nfm);
            }
            if (!barrier.wait()) return;
        }
        DEAC_PHASE(3);
        if (init) break;
    }
    if (a.local && blockIdx.x == 0)
        for (int i = threadIdx.x; i < a.P; i += kEvoThreads) {
            a.cur[i] = s.cur[i];
            a.fitness[i] = s.fitness[i];
            for (int sg = 0; sg < a.nsign; sg++) {
                a.cr_old[i * a.nsign + sg] = s.cr[i * a.nsign + sg];
                a.f_old[i * a.nsign + sg] = s.f[i * a.nsign + sg];
            }
        }
}

// K rows [T][Kc] into operand order: [tau block][unit of 8 positions][lane][2],
// lane l holding tau row l&15 at positions l>>4 and (l>>4)+4 of the unit.  Past
// T and Kc -0.0: with genomes padded with +0.0 the products are -0.0 and leave
// every sum exactly as it is.
__global__ __launch_bounds__(256) void ktile_kernel(const double *rows, double *ktile, int T, int Kc, int TB, int nunit)
{
    const size_t total = (static_cast<size_t>(TB) * nunit + kKtilePad) * kWave * 2;
    for (size_t o = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; o < total;
         o += static_cast<size_t>(gridDim.x) * 256) {
        const int e = static_cast<int>(o & 1), l = static_cast<int>((o >> 1) & (kWave - 1));
        const size_t tu = o >> 7;
        const int t = static_cast<int>(tu / nunit) * kChainTau + (l & 15);  // past T in the units of padding
        const int k = static_cast<int>(tu % nunit) * kUnit + (l >> 4) + 4 * e;
        ktile[o] = t < T && k < Kc ? rows[static_cast<size_t>(t) * Kc + k] : -0.0;
    }
}

__global__ void zero_u32_kernel(unsigned *p, size_t n)
{
    const size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------- launchers

hipError_t launch_walk(const WalkArgs &a, hipStream_t s)
{
    hipLaunchKernelGGL(walk_kernel, dim3(1), dim3(64), walk_lds_bytes(a), s, a);
    return hipGetLastError();
}

hipError_t launch_mask(const MaskArgs &a, const WalkArgs &next, hipStream_t s)
{
    const size_t waves = static_cast<size_t>(a.ngen) * a.P;
    const unsigned blocks = static_cast<unsigned>((waves + kEvoWaves - 1) / kEvoWaves);
    const size_t lds = kEvoWaves * kMaskLds * sizeof(double);
    if (next.ngen > 0)
        hipLaunchKernelGGL(mask_kernel<true>, dim3(blocks + 1), dim3(kEvoThreads), std::max(lds, walk_lds_bytes(next)), s,
                           a, next);
    else
        hipLaunchKernelGGL(mask_kernel<false>, dim3(blocks), dim3(kEvoThreads), lds, s, a, next);
    return hipGetLastError();
}

// A regular launch: the device holds one cooperative queue, which one
// process keeps once it has used it, so cooperative launches from a second
// process fail.  The evolution's workgroups never exceed the co-resident limit
// that evolve_max_workgroups reports (one workgroup per CU, bounded by LDS) and
// are dispatched first, so on an otherwise idle device every one of them is
// resident; if one is not, the bounded grid barrier reports a timeout instead
// of hanging.
hipError_t launch_evolve(const EvoArgs &a, const WalkArgs &next, const MaskArgs &masks, hipStream_t s, hipEvent_t start,
                         hipEvent_t stop)
{
    if (next.ngen > 0 && walk_lds_bytes(next) > kEvoLds) return hipErrorInvalidValue;
    const bool fed = a.fed && !a.init_mode;
    hipExtLaunchKernelGGL(fed ? evolve_kernel<kFed> : a.fold_ks && !a.init_mode ? evolve_kernel<kFold> : evolve_kernel<kChains>,
                          dim3(a.nwg + (next.ngen > 0 ? 1 : 0) + (masks.ngen > 0 ? masks.nwg : 0)), dim3(kEvoThreads),
                          kEvoLds, s, start, stop, 0, a, next, masks);
    return hipGetLastError();
}

hipError_t launch_ktile(const double *rows, double *ktile, int T, int Kc, int TB, int stride, hipStream_t s)
{
    const size_t total = ktile_doubles(TB, stride);
    const unsigned blocks = static_cast<unsigned>(std::min<size_t>((total + 255) / 256, 8192));
    hipLaunchKernelGGL(ktile_kernel, dim3(blocks), dim3(256), 0, s, rows, ktile, T, Kc, TB, stride / kUnit);
    return hipGetLastError();
}

hipError_t launch_zero_u32(unsigned *p, size_t n, hipStream_t s)
{
    hipLaunchKernelGGL(zero_u32_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

int evolve_max_workgroups(int device)
{
    int per_cu = 1, cus = 0;
    for (const void *k : {reinterpret_cast<const void *>(evolve_kernel<kChains>),
                          reinterpret_cast<const void *>(evolve_kernel<kFold>),
                          reinterpret_cast<const void *>(evolve_kernel<kFed>)}) {
        int n = 0;
        if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kEvoLds) != hipSuccess) return 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, kEvoThreads, kEvoLds) != hipSuccess) return 0;
        per_cu = std::min(per_cu, n);
    }
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 0;
    // One workgroup per CU: the grid barrier needs every workgroup resident,
    // and a second one per CU is not guaranteed to be even where the
    // occupancy estimate allows it.
    return per_cu * cus;
}

}  // namespace deac
