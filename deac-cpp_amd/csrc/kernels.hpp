// Device-side interface of the DEAC engine: argument blocks and launchers of
// the gfx950 kernels in kernels.hip.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace deac {

// Exact FP64 model-ISF contraction: one wavefront holds 4 members x 16
// timeslices, one sequential FMA chain per output on v_mfma_f64_4x4x4_4b_f64,
// its operands loaded in units of 8 positions.  Rows are padded to kChunk.
constexpr int kChainRows = 4;
constexpr int kChainTau = 16;
constexpr int kUnit = 8;
constexpr int kChunk = 128;
constexpr int kKtilePad = 32;  // units past the last, which the chains load ahead and do not use

// Evolution kernel: 4 wavefronts per workgroup; its registers and LDS leave
// room for a second workgroup on the CU (another handle's).
constexpr int kEvoThreads = 256;
constexpr size_t kEvoLds = 78 * 1024;
constexpr int kResidLds = 5632;   // doubles of LDS for residuals and the members' state
constexpr int kResidWave = 1024;  // residuals per wave and window, where a wave selects a member
static_assert(kEvoThreads / 64 * kResidWave <= kResidLds, "the waves' windows fit in LDS");
// Every workgroup repeats the selection while that is at most this many
// residuals, 16 per thread.
constexpr int kLocalResid = 4096;

constexpr int kXcds = 8;
// Words of a launch's synchronization: barrier counter [0], status [4..6], and
// from kXcdSync on a line of kXcdWords per XCD.
constexpr int kXcdSync = 32;
constexpr int kXcdWords = 32;
constexpr int kSyncWords = kXcdSync + kXcds * kXcdWords;

// Random choices of one member in one generation, produced by walk_kernel.
struct MemberCtl {
    uint64_t mask_state[4];  // xoshiro256+ state mask_steps draws before the member's first crossover-mask draw
    uint32_t mutant[3];      // donor indices r1, r2, r3 (deac.cpp:200-216)
    uint32_t flags;          // bit 2s: CR of sign s redrawn; bit 2s+1: F of sign s redrawn
    double cr_value[2];      // redrawn CR per sign
    double f_value[2];       // redrawn F per sign
    uint32_t mask_steps;
};

struct WalkArgs {
    uint64_t *state;             // in/out, 4 words
    uint64_t *gen_start;         // [ngen][4] state at the top of each generation
    MemberCtl *ctl;              // [ngen][P]
    const uint64_t *skip_rows;   // rows of T^(nsign*G), 256 x 4 words (serial walk)
    const uint64_t *tab1;        // lane_tables of T^c1 (wide walk)
    const uint64_t *tab2;        // lane_tables of T^(nsign*G+3) (wide walk)
    const uint64_t *skip_tab;    // nibble table of T^(nsign*G) (wide walk)
    int wide, c1;
    const int *halt;             // status of the batch that evolves beside the walk, or null
    int ngen, P, nsign;
    uint64_t mod_magic;          // floor((2^64-1)/P)
    double tau_cr, tau_f;
};

struct MaskArgs {
    const MemberCtl *ctl;        // [ngen][P]
    const uint64_t *lane_tab;    // lane_tables of T^chunk
    uint64_t *raw;               // [ngen][P][rstride] 53-bit draws (x >> 11)
    const int *halt;             // status of the batch that evolves beside the draws, or null
    int ngen, P, Kc, rstride;
    int chunk;                   // draws per lane, even
    int nwg;                     // workgroups (beside the evolution)
};
// LDS of a wavefront that makes mask draws: rounds of 16 per lane.
constexpr int kMaskRound = 16;
constexpr int kMaskRow = kMaskRound + 2;
constexpr int kMaskLds = 64 * kMaskRow;  // doubles
static_assert(kEvoThreads / 64 * kMaskLds * sizeof(double) <= kEvoLds, "mask draws fit beside the evolution");

struct EvoArgs {
    int P, T, G, nsign, Kc;
    int stride;                  // row stride of K and of the populations: Kc padded to kChunk
    int rstride;                 // row stride of the draws: Kc padded to whole 16-byte pairs
    int local;                   // every workgroup repeats the selection (evolve_local)
    int fed;                     // trial vectors formed beside the chains (evolve_fed)
    int MG, TB;                  // member groups of kChainRows, tau blocks of kChainTau
    int by_tau;                  // contraction tasks in order of tau blocks, else of member groups (evolve_by_tau)
    int use_first, use_third, renorm, allow_neg, init_mode, track_stats;
    double stop, zeroth, first_moment, third_moment, third_moment_error;
    int use_nfm;                 // -1st-moment term of the fitness (bdsf): weights nfm_dt [T]
    double nfm_value, nfm_error;
    const double *nfm_dt;
    int fold_ks;                 // the trials' model ISF as a rounded-product fold (bdsf)
    const double *ktile;         // K in the chains' and folds' operand order (launch_ktile)
    const double *nterm, *fterm, *tterm;   // [Kc] or null
    const double *obs, *sig;     // [T]
    double *pop0, *pop1;         // [MG*4][stride] each, one allocation, member-major rows, zero padded
    int *cur;                    // [P] buffer holding each member's current genome
    double *fitness;             // [P]
    double *cr_old, *f_old;      // [P][nsign]
    double *emod;                // [2][P][T] (the second where fed)
    double *mom;                 // [P][4]: normalization, first, third moment
    const MemberCtl *ctl;        // [ngen][P]
    const uint64_t *raw;         // [ngen][P][rstride]
    double *stats;               // [3][stats_len]: mean, minimum, squared mean
    size_t stats_len;
    unsigned *bar;               // grid barrier counter, zero at launch
    unsigned *xbar;              // [kXcds][kXcdWords] the same per XCD, or null (split loop)
    int *status;                 // [0] stopped, [1] generation index within the batch, [2] barrier timeout
    int *host_status;            // the same in pinned host memory, or null (split loop)
    unsigned *clear;             // the next launch's words (kSyncWords), or null
    long gen0;                   // generation index of the batch's first generation
    int ngen;
    int nwg;                     // workgroups that evolve
    long *iter;                  // split loop under graph capture: [0] gen0, [1] generation within the batch
                                 // (read in place of gen0 and the kernels' g; the selection reads [2]), or null
};

// Wide walk: draws per lane and round for the jDE controls, donor draws per
// member that one block looks ahead, members it holds flags of.
constexpr int kWalkControls = 33;
constexpr int kWalkDraws = 48;
constexpr int kWalkMaxP = 4096;
// The wide walk from here on (us per generation, serial and wide: 16 members
// 11.4 and 14.3, 24 members 16.7 and 14.4, 64 members 43 and 19, 512 members
// 340 and 65); its one test per control needs equal redraw probabilities.
constexpr int kWalkWideP = 20;
inline bool walk_is_wide(int P, double tau_cr, double tau_f)
{
    return P >= kWalkWideP && P <= kWalkMaxP && tau_cr == tau_f;
}
inline int walk_c1(int P, int nsign)
{
    const int tests = 2 * nsign * P;
    const int c = (tests + tests / 4 + 8 + 63) / 64;
    return c < 4 ? 4 : c > kWalkControls ? kWalkControls : c;
}
inline size_t walk_lds_bytes(const WalkArgs &a)
{
    if (!a.wide) return 256 * 4 * sizeof(uint64_t);
    return (64 * static_cast<size_t>(a.c1 | 1)) * sizeof(uint64_t) +
           (static_cast<size_t>(kWalkDraws) * 64 + a.P) * sizeof(uint32_t);
}
hipError_t launch_walk(const WalkArgs &a, hipStream_t s);
// Mask draws, and where next.ngen > 0 a walk on one more workgroup.
hipError_t launch_mask(const MaskArgs &a, const WalkArgs &next, hipStream_t s);
// Whether the evolution kernel's workgroups repeat the selection: the
// residuals are few, and they and the members' state fit in LDS.
inline int evolve_local(int P, int T, int nsign, int use_nfm)
{
    const long resid = static_cast<long>(P) * (T | 1);
    return resid <= kLocalResid && resid * (1 + use_nfm) + static_cast<long>(P) * (2 + 2 * nsign) <= kResidLds;
}
// Whether a workgroup per contraction task forms the trial vectors of its
// members itself, beside their chains: where the tasks have a CU each, the
// selection is every workgroup's own, nothing but the chains reads whole trials,
// and 32-bit offsets reach the populations.  (us a generation without and with:
// 8 members G = 512, T = 33 13.6 and 12.7; G = 4096, T = 65 and 8 members 35.2
// and 34.1, 16 39.8 and 36.7, 32 48.8 and 42.0, 62 66.1 and 49.8; 31 members G =
// 2048, T = 129 38.2 and 33.4; 200 members G = 6000, T = 17 102 and 80.)
inline int evolve_fed(const EvoArgs &a, int maxwg)
{
    return a.local && !a.renorm && !a.use_first && !a.use_third && !a.use_nfm && !a.fold_ks && a.MG * a.TB + 1 <= maxwg &&
           static_cast<size_t>(a.MG) * kChainRows * a.stride * 16 < (size_t(1) << 31);
}
// Whether an XCD's range of contraction tasks reads fewer rows in order of tau
// blocks (16 K rows each) than in order of member groups (`rows` genome rows).
inline int evolve_by_tau(int groups, int rows, int TB)
{
    const long n = (static_cast<long>(groups) * TB + kXcds - 1) / kXcds;
    const long tau = kChainTau * ((n - 1) / groups + 2) + rows * (n < groups ? n : groups);
    const long member = kChainTau * (n < TB ? n : TB) + rows * ((n - 1) / TB + 2);
    return tau < member;
}
// Doubles of the K operand of TB tau blocks.
inline size_t ktile_doubles(int TB, int stride)
{
    return (static_cast<size_t>(TB) * (stride / kUnit) + kKtilePad) * 64 * 2;
}
hipError_t launch_ktile(const double *rows, double *ktile, int T, int Kc, int TB, int stride, hipStream_t s);
// The evolution of a batch and beside it the mask draws of the next one and
// the walk of the one after, where they have generations.  start, stop: events
// that the dispatch itself records, or null (recorded in the stream on its two
// sides they cost the gap between two launches 6 us).
hipError_t launch_evolve(const EvoArgs &a, const WalkArgs &next, const MaskArgs &masks, hipStream_t s, hipEvent_t start,
                         hipEvent_t stop);
hipError_t launch_zero_u32(unsigned *p, size_t n, hipStream_t s);
// Workgroups of the evolution kernel that are co-resident on the device: one
// per CU.
int evolve_max_workgroups(int device);

}  // namespace deac
