// mxh_gemm_f16.h — arguments shared by the fp16 matrix-core GEMMs over
// quantized rows.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mxh_plan.h"

namespace mxh {

// out[m x n] (row stride ldo) = a . W^T (+ res), a as fp16 hi / lo of a 2^e
// per row (row stride lda), s: split sums of every 32-element sub-block (row
// stride lds), rscale = 2^-e.  W's rows hold row_blocks 256-element blocks, the
// first k / 256 of them real.  K is cut into `splits` ranges of `blocks`
// blocks; with more than one, split z writes its partial tile to
// part[z][m][n].
struct CodesArgs {
    const uint16_t *a_hi, *a_lo, *s_hi, *s_lo;
    const float* rscale;
    const uint8_t* w;
    float* out;
    const float* res;
    float* part;
    int lda, lds, ldo, m, n, k, form, row_blocks, blocks, splits;
};

int gemm_codes_launch(GemmFmt f, GemmTile t, const CodesArgs& a, hipStream_t st);

}  // namespace mxh
