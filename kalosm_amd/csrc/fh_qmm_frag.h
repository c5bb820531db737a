// Quantized matmul for prompts through fragment-ordered operands (fh_qmm_frag.hip).
#pragma once
#include "fh_internal.h"

bool fh_qmm_frag_supports(const fh_qmatrix *q);
bool fh_qmm_frag_pays(const fh_qmatrix *q, int x_is_bf16, int m); // and where it is the faster way
// y[m, n] = x[m, k] . deq(q)^T; x f32 or bf16, rows contiguous and 16-byte aligned.
fh_status fh_launch_qmm_frag(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y);
// (More than 16 rows.)  y[m, n / 2] = silu(x . deq(rows 0 ..)^T) * (x . deq(rows n / 2 ..)^T); FH_ERR_UNSUPPORTED where two launches are the faster way.
fh_status fh_qmm_frag_swiglu(const fh_qmatrix *q, const float *x, int m, float *y);
