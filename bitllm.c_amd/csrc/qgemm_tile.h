// qgemm_tile.h -- the register-tiled int8-MFMA GEMM of large token batches (qgemm_tile.hip).
#pragma once

#include "hip_common.h"

namespace eif {

// One linear on prepped rows: y[m, r] = epilogue of sum_k w[r, k] xq[m, k] (the contract of eif_hip_qlinear).
struct TileGemm {
    const uint8_t *W;      // resident layout (qlinear.hip), rows padded to 64
    const float *scales;   // grouped [rows / 16][G][16]; row-scaled [N] or NULL
    const int8_t *xq;      // [M, ldq]
    const float *xs;       // [M]
    const float *bias;     // [N] or NULL
    float *y;              // [M, ldy]
    const float *res;      // [M, ldr] added to the outputs (may be y itself), or NULL
    int ldr;
    int fmt, ud, grouped;  // EIF_HIP_W_*, group / 32 (4 for row-scaled ternary), group scales
    int wld, rows_pad, G, ldq, ldy, M, N, nsteps;
    int ks;                // splits along K (>= 1)
    float *part;           // ks > 1: their partial sums,
    int *cnt;              // and one arrival counter per tile, zero between launches
};

// Whether the form takes this shape (with g.ks splits; g.part and g.cnt are not read), its output tiles and the bytes
// of partial sums that its splits leave.
bool gemm_tile_takes(const TileGemm &g, int *tiles, size_t *part_bytes);
int launch_gemm_tile(const TileGemm &g, hipStream_t st);

}  // namespace eif
