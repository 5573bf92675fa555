// Device helpers shared by the gfx950 kernels: the xoshiro256+ step, its
// exact uniform, the modulo of the donor draws, GF(2) parity and the
// s_waitcnt forms the pipelines use.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace deac {

__device__ __forceinline__ uint64_t xnext(uint64_t (&s)[4])  // rng.hpp:25-39
{
    // The reference's five in-place xors, written as three-input xors of the
    // old state (v_xor3_b32) and a rotate by two funnel shifts.
    const uint64_t s0 = s[0], s1 = s[1], s2 = s[2], s3 = s[3];
    const uint64_t out = s0 + s3;
    const uint64_t t = s1 << 17;
    const uint64_t n3 = s3 ^ s1;
    s[1] = s1 ^ s2 ^ s0;
    s[0] = s0 ^ n3;
    s[2] = s2 ^ s0 ^ t;
    const uint32_t lo = static_cast<uint32_t>(n3), hi = static_cast<uint32_t>(n3 >> 32);
    // rotl(n3, 45) = rotr(n3, 19)
    const uint32_t rlo = __builtin_amdgcn_alignbit(hi, lo, 19), rhi = __builtin_amdgcn_alignbit(lo, hi, 19);
    s[3] = (static_cast<uint64_t>(rhi) << 32) | rlo;
    return out;
}

// (x >> 11) * 2^-53, exact (deac.cpp:437)
__device__ __forceinline__ double to_unit(uint64_t x) { return static_cast<double>(x >> 11) * 0x1.0p-53; }

// x % P for P < 2^32 with magic = floor((2^64-1)/P): the quotient estimate is
// low by at most one, fixed by one conditional subtraction.
__device__ __forceinline__ uint32_t mod_p(uint64_t x, uint64_t magic, uint32_t P)
{
    const uint64_t q = __umul64hi(x, magic);
    uint64_t r = x - q * P;
    if (r >= P) r -= P;
    return static_cast<uint32_t>(r);
}

__device__ __forceinline__ int parity64(uint64_t x)
{
    return __popc(static_cast<uint32_t>(x) ^ static_cast<uint32_t>(x >> 32)) & 1;
}

// The lane's jump M^lane s of a state s that all 64 lanes share, from the
// interleaved tables of launch_lane_tables (init_kernels.hpp): 128 coalesced 1 KB loads
// a wavefront.  (The same tables one after another, each lane gathering its
// 32-byte entries, took four times as long.)
__device__ __forceinline__ void lane_jump(const uint64_t *tab, const uint64_t (&s)[4], uint64_t (&out)[4])
{
    typedef uint32_t quad __attribute__((ext_vector_type(4)));
    const int voff = (threadIdx.x & 63) * 16;
    uint32_t u[8];
    for (int w = 0; w < 4; w++) {
        u[2 * w] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s[w]));
        u[2 * w + 1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s[w] >> 32));
    }
    // the entry's address is scalar (buffer loads take it as one offset), 24 loads in flight
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint64_t *>(tab), 0, 64 * 16 * 2048, 0x00020000);
    constexpr int kHold = 12;
    quad e0[kHold], e1[kHold], lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
    auto load = [&](int n) __attribute__((always_inline)) {
        const uint32_t v = (u[n >> 3] >> ((n & 7) * 4)) & 15;
        const int off = static_cast<int>((n * 16 + v) * 2048);
        e0[n % kHold] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, off, 0);
        e1[n % kHold] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + 1024, off, 0);
    };
#pragma unroll
    for (int n = 0; n < kHold; n++) load(n);
#pragma unroll
    for (int n = 0; n < 64; n++) {
        lo ^= e0[n % kHold];
        hi ^= e1[n % kHold];
        // (the sums stay here, so that the entries' registers are free again)
        asm volatile("" : "+v"(lo), "+v"(hi));
        if (n + kHold < 64) load(n + kHold);
        __builtin_amdgcn_sched_barrier(0);
    }
    out[0] = (static_cast<uint64_t>(lo.y) << 32) | lo.x;
    out[1] = (static_cast<uint64_t>(lo.w) << 32) | lo.z;
    out[2] = (static_cast<uint64_t>(hi.y) << 32) | hi.x;
    out[3] = (static_cast<uint64_t>(hi.w) << 32) | hi.z;
}

}  // namespace deac

// s_waitcnt with vmcnt <= n (n < 64) and the other counters unconstrained.
#define DEAC_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))
// s_waitcnt lgkmcnt(0) (LDS operations retired), other counters unconstrained.
#define DEAC_WAIT_LDS() __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4))
