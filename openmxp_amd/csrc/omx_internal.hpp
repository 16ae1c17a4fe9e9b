// omx_internal.hpp -- launches that the solver makes of several entry points'
// work at once (not part of the C ABI): the column and the row panel of a step
// packed, or multiplied, in one launch instead of two that wait for each
// other.  Results are those of the single calls bit for bit.
#pragma once

#include <stdint.h>

#define OMX_HIDDEN __attribute__((visibility("hidden")))

// one panel to pack, as omx_pack_f16 / omx_pack_f16_window (unscaled) or
// omx_pack_f8_window with its tile maxima given (exps, tile_max, headroom)
struct omx_pack_job {
    int64_t rows, k;
    const float *src;
    int64_t rs, ls;
    int mask;
    void *P;
    int64_t ldk, k0;
    int headroom;
    int32_t *exps;
    const float *tile_max;
};

// one product, as omx_gemm_f16_packed_tri / omx_gemm_f16_packed_window
// (unscaled) or omx_gemm_f8_packed_window
struct omx_gemm_job {
    int64_t m, n, k;
    const void *X;
    const int32_t *xexp;
    int64_t x_row0, x_ldk, x_k0;
    const void *Y;
    const int32_t *yexp;
    int64_t y_row0, y_ldk, y_k0;
    float *C;
    int64_t ldc;
    int tri;
    float *tile_max;
};

// up to four FP16 / two FP8 panels of equal k
OMX_HIDDEN int omx_pack_f16_jobs(int count, const omx_pack_job *jobs, void *stream);
OMX_HIDDEN int omx_pack_f8_jobs(int count, const omx_pack_job *jobs, void *stream);
// C_i = beta C_i + alpha X_i Y_i^T, i = 0, 1 (FP8: beta = 1); both with rows
// and columns
OMX_HIDDEN int omx_gemm_f16_pair(const omx_gemm_job *jobs, float alpha, float beta, void *stream);
OMX_HIDDEN int omx_gemm_f8_pair(const omx_gemm_job *jobs, float alpha, void *stream);
