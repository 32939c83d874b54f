// Fused dequant-GEMV of several tokens on the matrix cores (gemv_mm.hip).
#pragma once

#include "nsx_common.h"

// Bytes of workspace nsx_gemv_mm needs for this call; 0: it does not take it.
int64_t nsx_gemv_mm_workspace(int ggml_type, int64_t n_rows, int64_t K, int64_t T);
// Whether nsx_gemv_mm takes this call and is the faster path for it.
int nsx_gemv_mm_takes(int ggml_type, int64_t n_rows, int64_t K, int64_t T);
// y[t, r] = resid[t, r] + (sum_k x[t, k] dequant(raw)[r, k] + bias[r]), as nsx_fused_gemv_ex; ws 16-byte aligned.
int nsx_gemv_mm(int ggml_type, const void* raw, int64_t n_rows, int64_t K, const void* x, int x_dtype, int64_t T,
                float* y, const float* bias, const float* resid, void* ws, hipStream_t st);
