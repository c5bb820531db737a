// Quantized matmul for prompts through fragment-ordered operands (fh_qmm_frag.hip).
#pragma once
#include "fh_internal.h"

bool fh_qmm_frag_supports(const fh_qmatrix *q);
bool fh_qmm_frag_pays(const fh_qmatrix *q, int x_is_bf16, int m); // and where it is the faster way
double fh_qmm_frag_us(const fh_qmatrix *q, int x_is_bf16, int m, int *parts); // (more than FH_SHORT_PROMPT rows) how long it would take, in how many parts of k
double fh_qmm_tile_us(const fh_qmatrix *q, int x_is_bf16, int m);             // the tile kernels; 1e30 where they are far from filling the device
// y[m, n] = x[m, k] . deq(q)^T; x f32 or bf16, rows contiguous and 16-byte aligned.  FH_ERR_UNSUPPORTED where the memory for the
// fragments cannot be had.
fh_status fh_launch_qmm_frag(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y);
// A decoder's prompts of up to this many tokens keep the sums of the tile kernels (k_qmm_short: 37 tokens and 64 sampled ones through four
// layers of width 2048 in 9.3 ms, the tiles 11.1).  The fragments are closer (against 64 bits 4e-6 of the logits, the tiles 1e-5),
// but the cache they leave differs in its last bits: of 1200 sampled continuations of 64 tokens two came to a draw that those bits
// decide and went another way from there.
enum { FH_SHORT_PROMPT = 64 };
// (More than FH_SHORT_PROMPT rows.)  y[m, n / 2] = silu(x . deq(rows 0 ..)^T) * (x . deq(rows n / 2 ..)^T); FH_ERR_UNSUPPORTED where two launches are the faster way.
fh_status fh_qmm_frag_swiglu(const fh_qmatrix *q, const float *x, int m, float *y);
// y[i] = part[i] + part[stride + i] + .., count of them, 16 planes at most, added in pairs
fh_status fh_frag_sum(fh_device *dev, const float *part, int parts, int64_t stride, int64_t count, float *y);

// The same for fewer rows, weights decoded in registers (fh_qmm_reg.hip); memory and results as above.  planes: the tile kernels, which take
// the call where the memory cannot be had, find theirs.
bool fh_qmm_reg_supports(const fh_qmatrix *q);
bool fh_qmm_reg_pays(const fh_qmatrix *q, int x_is_bf16, int m);
fh_status fh_launch_qmm_reg(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y, bool planes);
bool fh_qmm_reg_swiglu_pays(const fh_qmatrix *q, int m); // (where fh_qmm_reg_pays)
fh_status fh_qmm_reg_swiglu(const fh_qmatrix *q, const float *x, int m, float *y);
