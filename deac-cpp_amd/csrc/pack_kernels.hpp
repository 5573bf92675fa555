// Operand layouts made on the device from plain rows: the kernel matrix of
// the K.S contractions and the genome stack of deac_model_isf.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace deac {

struct PackArgs {
    const double *rows;  // [n][L]
    const int *ex;       // row r is scaled by 2^-ex[r] (exact), or null
    int n, L;
    int tiles, Kb;       // tiles of 16 rows, k-blocks per tile
};

// 16x16x4 operands (KsLayout): out[tile][kb][lane] = row(16 tile + lane%16)
// [4 kb + lane/16]; pad past the rows and past L.
hipError_t launch_pack_fp64(const PackArgs &a, double pad, double *out, hipStream_t s);
hipError_t launch_pack_fp32(const PackArgs &a, float *out, hipStream_t s);
// 16x16x32 operands: 8 values per lane, positions 32 kb + 8 (lane/16) + e, each
// split x = hi + lo into bfloat16; hi and lo apart, or 8 hi then 8 lo per lane
// in hi when lo is null (the batch's K tiles).
hipError_t launch_pack_bf16x3(const PackArgs &a, void *hi, void *lo, hipStream_t s);
// The batch's FP32 K tiles: [tile][kb][lane][4], positions 16 kb + 4 e + lane/16.
hipError_t launch_pack_fp32_units(const PackArgs &a, float *out, hipStream_t s);
// K rows position-major: out[k][width], zero past n and past L, for k < positions.
hipError_t launch_pack_transposed(const PackArgs &a, int width, int positions, double *out, hipStream_t s);

}  // namespace deac
