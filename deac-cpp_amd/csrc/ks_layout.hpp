// Operand layouts of the K.S contraction kernels (precision_kernels.hip): the
// kernel matrix and, for deac_model_isf, the stack of genomes, packed from
// plain rows by pack_kernels.hip.  The split generation loop packs its trial
// genomes into the same layout (split_kernels.hip).
//
// Lane order, one coalesced load per wave and k-block:
//   FP64, FP32  slot (tile, kb, lane)     = X[16 tile + lane%16][4 kb + lane/16]
//   BF16X3      slot (tile, kb, lane, e)  = X[16 tile + lane%16][32 kb + 8 (lane/16) + e]
// with X = K (tiles of 16 timeslices) or S (tiles of 16 genomes).
#pragma once

#include <algorithm>
#include <cmath>
#include <vector>

#include "deac_engine.h"
#include "host_model.hpp"
#include "precision_kernels.hpp"

namespace deac {

struct KsLayout {
    int precision = DEAC_PRECISION_FP64;
    size_t T = 0, N = 0, L = 0;        // timeslices, genomes, genome length
    int Mt = 0, Nt = 0;                // tiles of 16 timeslices and of 16 genomes
    size_t kblock = 4;                 // positions per k-block: 4, or 32 for BF16X3
    size_t per = 1;                    // values per lane and k-block: 1, or 8 for BF16X3
    size_t Kb = 0;                     // k-blocks, a multiple of the kernels' prefetch depth
    int kb_per_slice = 0, slices = 1;  // genome slices (FP32, BF16X3)
    std::vector<int> ex;               // K row t is scaled by 2^-ex[t] (FP32, BF16X3)

    size_t mpad() const { return static_cast<size_t>(Mt) * 16; }
    size_t npad() const { return static_cast<size_t>(Nt) * 16; }
    size_t a_count() const { return static_cast<size_t>(Mt) * Kb * 64 * per; }
    size_t b_count() const { return static_cast<size_t>(Nt) * Kb * 64 * per; }
};

inline KsLayout ks_layout(const Model &m, int precision, size_t count)
{
    KsLayout y;
    y.precision = precision;
    y.T = m.T;
    y.N = count;
    y.L = m.Kc;
    y.Mt = static_cast<int>((m.T + 15) / 16);
    y.Nt = static_cast<int>((count + 15) / 16);
    const bool bf = precision == DEAC_PRECISION_BF16X3;
    y.kblock = bf ? 32 : 4;
    y.per = bf ? 8 : 1;
    const size_t depth = bf ? kSweepDepth16 : kSweepDepth;
    y.Kb = (y.L + y.kblock * depth - 1) / (y.kblock * depth) * depth;  // zero padded
    if (precision != DEAC_PRECISION_FP64) {
        // K row t scaled by 2^-e_t (exact), e_t the exponent of its largest
        // magnitude, so every row's largest entry lies in [1, 2)
        y.ex.assign(m.T, 0);
        for (size_t t = 0; t < m.T; t++) {
            double mx = 0.0;
            for (size_t k = 0; k < y.L; k++) mx = std::fmax(mx, std::fabs(m.kernel[t * y.L + k]));
            y.ex[t] = mx > 0.0 ? std::ilogb(mx) : 0;
        }
        // genome slices: enough workgroups (about 2048) to fill the device,
        // at least 8 k-blocks per slice.  (Fewer, longer slices are cheaper
        // to sum but longer FP32 accumulations: capping them at 32 at
        // T=257, G=16384, P=64 raised the model-ISF error 100-fold.)
        const size_t tiles = static_cast<size_t>(y.Mt) * ((y.Nt + 3) / 4);
        const size_t want =
            std::max<size_t>(1, std::min<size_t>((2048 + tiles - 1) / tiles, std::max<size_t>(y.Kb / 8, 1)));
        y.kb_per_slice = static_cast<int>(((y.Kb + want - 1) / want + depth - 1) / depth * depth);
        y.slices = static_cast<int>((y.Kb + y.kb_per_slice - 1) / y.kb_per_slice);
    }
    return y;
}

}  // namespace deac
