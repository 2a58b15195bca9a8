// prep_batch.h -- the activation prep of a batch of many token rows (prep_batch.hip).
#pragma once

#include "hip_common.h"

namespace eif {

struct PrepBatch {
    const float *x;           // [M, ldx] rows, 16-byte aligned
    int ldx;
    const float *signs, *nw;  // [K] or NULL
    int K, block;
    float norm, eps;
    int pre;                  // EIF_HIP_PRE_*
    int8_t *xq;               // [M, ldq], 16-byte aligned, ldq a multiple of 16
    int ldq;
    float *xs;                // [M]
    int M;
};

// The prep of eif_hip_prep_spec_rows, one wave a row; 1 when the shape is left to the kernel of one workgroup a row.
int launch_prep_batch(const PrepBatch &p, hipStream_t st);

}  // namespace eif
