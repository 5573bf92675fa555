// Initial populations on the device (deac.cpp:430-458, 584-602), for the
// single-instance engine and the batch.
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

// Draws every member's genome, then normalizes it when nterm is given.
hipError_t launch_initial_population(const InitArgs &a, hipStream_t s);

}  // namespace deac
