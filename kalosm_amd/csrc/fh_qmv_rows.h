// Quantized matmul for a few rows of f32 activations in one launch (fh_qmv_rows.hip).
#pragma once
#include "fh_internal.h"

bool fh_qmv_rows_supports(const fh_qmatrix *q, const float *x, int m);
bool fh_qmv_rows_pays(const fh_qmatrix *q, const float *x, int m); // and where it is the faster way
// y[m, n] = x[m, k] . deq(q)^T; FH_ERR_UNSUPPORTED where the memory for parts of k cannot be had
fh_status fh_launch_qmv_rows(const fh_qmatrix *q, const float *x, int m, float *y);
