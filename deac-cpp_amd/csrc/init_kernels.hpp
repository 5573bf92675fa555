// Device set-up and readback of the engines: initial populations (deac.cpp:430-458,
// 584-602), for the single-instance engine and the batch, and jump tables.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace deac {

struct InitArgs {
    const uint64_t *start;   // [rows][4]: random state at each member's first draw
    const long *offset;      // [rows / P] offset of each instance's population from pop, or null (0)
    double *pop;             // member rows of `stride` doubles
    const uint64_t *tab;     // lane_tab: lane_tables of T^sublen (64 sub-streams, one wavefront per member);
                             // else nibble tables of T^(k*sublen) for sub-streams k = 1 .. nsub-1
    const double *nterm;     // [Kc] normalization weights, or null: populations are not normalized
    long rows;               // members of all instances
    int P, G, nsign, stride;
    int nsub, sublen;        // sub-streams per member and draws of each
    bool lane_tab;
    int allow_neg;
    double zeroth;
};

// Nibble tables of M^0 .. M^63, interleaved by lane: tab[n][v][half][l][2] is
// half (words 0-1, 2-3) of M^l * (v << 4n), so that 64 lanes that jump one
// common state by different powers load side by side (lane_jump).
constexpr size_t kLaneTabWords = 64 * 16 * 4 * 64;
constexpr int kLaneTabSets = 3;
struct LaneTabArgs {
    const uint64_t *columns;         // [sets][256][4]: the columns of each M
    uint64_t *tab[kLaneTabSets];
};
hipError_t launch_lane_tables(const LaneTabArgs &a, int sets, hipStream_t s);

// Draws every member's genome, then normalizes it when nterm is given.
hipError_t launch_initial_population(const InitArgs &a, hipStream_t s);

// Best member of each of n instances (the first of the lowest fitnesses,
// deac.cpp:128-138) into out; table: per instance 5 values, its offset in out
// and in pop, members, genome length, row stride; fitness rows of `pitch`.
hipError_t launch_gather_best(const long *table, size_t n, const double *fitness, int pitch, const double *pop,
                              double *out, hipStream_t s);

}  // namespace deac
