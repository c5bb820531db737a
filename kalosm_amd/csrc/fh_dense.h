// Device helpers and host launchers for dense bf16 weights (FH_BF16) with bf16 or f32 activations: the products of the
// layer-list decoders (fh_hybrid.hip).  Weight rows are row-major with a stride of k rounded up to 64 elements, the
// rows are rounded up to 16, and all padding is zero; activation rows use the same stride, so no kernel has an edge
// along k.
#pragma once
#include "fh_internal.h"

typedef __bf16 fh_bf;
typedef __bf16 fh_bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 fh_bf4 __attribute__((ext_vector_type(4)));
typedef float fh_f4 __attribute__((ext_vector_type(4)));
struct fh_f8 { float v[8]; };

static inline int64_t fh_pad64(int64_t k) { return (k + 63) / 64 * 64; }

__device__ __forceinline__ float fh_bf_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ uint16_t fh_f32_bf(float f) {
    const fh_bf b = (fh_bf)f;
    uint16_t u;
    __builtin_memcpy(&u, &b, 2);
    return u;
}
// low / high half of a 32-bit word of two bf16
__device__ __forceinline__ float fh_bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float fh_bf_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }

template <typename T> __device__ __forceinline__ T fh_to(float f);
template <> __device__ __forceinline__ float fh_to<float>(float f) { return f; }
template <> __device__ __forceinline__ uint16_t fh_to<uint16_t>(float f) { return fh_f32_bf(f); }
__device__ __forceinline__ float fh_up(float f) { return f; }
__device__ __forceinline__ float fh_up(uint16_t b) { return fh_bf_f32(b); }

// The sum over the wavefront, in every lane: of lanes 32 apart, 16, 8, 4, 2, 1.  (By register moves: through the LDS, as __shfl_xor has it, the same sum is six
// round trips, and a matvec of 32768 rows of 512, one such sum each, took 11.0 us instead of 8.9.)
__device__ __forceinline__ float fh_wave_sum(float v) {
    typedef uint32_t pair __attribute__((ext_vector_type(2)));
    const auto both = [](const pair &r) { return __uint_as_float(r[0]) + __uint_as_float(r[1]); };
    v = both(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    v = both(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true)); // row_ror:8
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xF, 0xF, true)); // row_ror:4
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));  // quad_perm 2 3 0 1
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));  // quad_perm 1 0 3 2
    return v;
}
__device__ __forceinline__ float fh_wave_max(float v) {
    typedef uint32_t pair __attribute__((ext_vector_type(2)));
    const auto both = [](const pair &r) { return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])); };
    v = both(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    v = both(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xF, 0xF, true)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true)));
    return fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true)));
}
// silu, softplus and the logistic function with the full-precision exponential
__device__ __forceinline__ float fh_silu_f(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float fh_softplus_f(float z) { return fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float fh_sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }

// Eight k-values of an MFMA operand in the layout of v_mfma_f32_16x16x32_bf16 (lane l: row l % 16, k = 8 (l / 16) .. + 7)
// and one 16 x 16 x 32 step on them.  f32 operands keep the same layout: eight v_mfma_f32_16x16x4_f32, each with one of
// the lane's values, add up to the same 32 of k in true f32.
template <typename T> struct FhFrag;
template <> struct FhFrag<uint16_t> { typedef fh_bf8 type; };
template <> struct FhFrag<float> { typedef fh_f8 type; };
__device__ __forceinline__ void fh_frag_load(fh_bf8 &f, const uint16_t *p) {
    const uint4 r = *(const uint4 *)p;
    __builtin_memcpy(&f, &r, 16);
}
__device__ __forceinline__ void fh_frag_load(fh_f8 &f, const float *p) {
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
    f.v[0] = a.x, f.v[1] = a.y, f.v[2] = a.z, f.v[3] = a.w;
    f.v[4] = b.x, f.v[5] = b.y, f.v[6] = b.z, f.v[7] = b.w;
}
__device__ __forceinline__ fh_f4 fh_mma32(const fh_bf8 &a, const fh_bf8 &b, fh_f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ fh_f4 fh_mma32(const fh_f8 &a, const fh_f8 &b, fh_f4 c) {
#pragma unroll
    for (int e = 0; e < 8; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[e], b.v[e], c, 0, 0, 0);
    return c;
}

// A barrier behind LDS writes that leaves requests to memory on their way.
__device__ __forceinline__ void fh_lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 16 bytes that are read once.  Decoders take the hint whatever their size: where the last cache keeps the weights, the launch that reads most of them can be slower with it,
// but what lies in the second cache for the launches around it stays there.  us a step, plainly / with the hint, output launches and the rest: 512 wide, eight experts of
// 2048 (201 MB) 59.6 + 65.1 / 67.2 + 66.2; 512 wide, an always-on one of 8192 (100 MB) 54.6 + 58.4 / 58.6 + 54.6; 1024 wide, the same (201 MB) 61.4 + 68.3 / 64.3 + 66.2;
// 1024 wide, four experts and an always-on one of 512 29.7 + 54.3 / 30.3 + 51.5; 2048 wide, eight of 2048 (805 MB) 91.0 + 141.3 / 86.8 + 135.4.  ms of 33 + 64 tokens: Fidasun
// 1024 wide (169 MB) 8.96 / 8.71, 1536 wide (363 MB) 11.03 / 10.87, Zovovik 1024 wide (137 MB) 8.77 / 8.90, 1536 wide (245 MB) 10.06 / 10.51, 2048 wide (295 MB) 10.30 / 10.30.
__device__ __forceinline__ uint4 fh_load_once(const uint16_t *p) {
    typedef uint32_t words __attribute__((ext_vector_type(4)));
    const words v = __builtin_nontemporal_load((const words *)p);
    return make_uint4(v[0], v[1], v[2], v[3]);
}
// Values at .. at + 7 of a row of kp (in a scalar register), zeros past its end: it is a buffer of its own, and what lies past a buffer is not read.  (The row's last
// eight values again, whose products with zeros are dropped, would have to be told from others: an infinity among them makes NaN.  us of 32768 x 1024 / 16384 x 1280 /
// 4096 x 4096: without that, 13.0 / 9.4 / 8.2, with that choice in the code 13.5 / 9.5 / 8.4, so 13.4 / 9.3 / 8.1.)
__device__ __forceinline__ uint4 fh_load_row_once(const uint16_t *row, int kp, int at) {
    typedef uint32_t words __attribute__((ext_vector_type(4)));
    const words v = __builtin_amdgcn_raw_buffer_load_b128(__builtin_amdgcn_make_buffer_rsrc((void *)row, 0, kp * 2, 0x00027000), at * 2, 0, 2); // (2: not read again)
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ float fh_dot8(const uint4 &w, const float4 &a, const float4 &b, float acc) {
    acc = fmaf(fh_bf_lo(w.x), a.x, acc);
    acc = fmaf(fh_bf_hi(w.x), a.y, acc);
    acc = fmaf(fh_bf_lo(w.y), a.z, acc);
    acc = fmaf(fh_bf_hi(w.y), a.w, acc);
    acc = fmaf(fh_bf_lo(w.z), b.x, acc);
    acc = fmaf(fh_bf_hi(w.z), b.y, acc);
    acc = fmaf(fh_bf_lo(w.w), b.z, acc);
    return fmaf(fh_bf_hi(w.w), b.w, acc);
}

// The rows of a matrix that one wavefront goes through, one after the other: `count` rows `hop` elements apart, in pieces of 512 (a lane:
// eight values, 16 bytes) with AHEAD pieces on their way.  Requests past the last row repeat it, and none is under a condition.
// A compute unit answers its requests in their order, so what is on the way is also what the launch's own input waits behind: a launch
// has one workgroup of eight wavefronts a compute unit, each with 4 KB on its way - 8 MB over the device, the rate of the memory
// times its latency.  us of 14336 x 4096 / 32768 x 4096 / 4096 x 14336: 19.9 / 40.9 / 20.0 (plain reads of the bytes 19.6 / 42.5 / 19.6); 3 KB 20.0 /
// 40.8 / 20.3, 2 KB 23.3 / 49.2 / 22.9, 8 KB 21.4 / 43.5 / 21.0, two such workgroups 22.7 / 45.7 / 22.0; without the hint that the weights are not
// read again 20.7 / 44.4 / 22.0; as many workgroups as there are rows for, two rows and 8 KB a wavefront, 22.4 / 44.4 / 22.3, four rows and 16 KB 29.5 / 62.0 / 26.5.
// The input lies in the LDS in two planes, so that neighbouring lanes read neighbouring 16 bytes.
struct FhRowInput {
    float *xs; // [2][plane]: the first and the second four of every eight values; zeros up to whole pieces
    int plane; // pieces * 256
    __device__ __forceinline__ float4 &quad(int q) const { return *(float4 *)(xs + (q & 1) * plane + (q >> 1) * 4); } // values 4 q ..
    __device__ __forceinline__ float &at(int i) const { return xs[((i >> 2) & 1) * plane + (i >> 3) * 4 + (i & 3)]; }
};
__host__ __device__ static inline int fh_row_pieces(int kp) { return (kp + 511) / 512; }
template <int AHEAD = 4>
struct FhRowDeal {
    const uint16_t *row; // of the next request
    int64_t hop;
    int kp, pieces, count, left, piece, lane8;
    uint4 u[AHEAD];
    __device__ __forceinline__ void fetch(int slot) {
        u[slot] = fh_load_row_once(row, kp, piece * 512 + lane8);
        const bool end = ++piece == pieces;
        piece = end ? 0 : piece;
        left -= end;
        row += end && left > 0 ? hop : 0;
    }
    // rows first, first + step, .. of n (first: the wavefront's, in a scalar register)
    __device__ __forceinline__ void start(const uint16_t *w, int kp_, int first, int step, int n) {
        kp = kp_, pieces = fh_row_pieces(kp), lane8 = (threadIdx.x & 63) * 8, piece = 0;
        left = count = first < n ? (n - first + step - 1) / step : 0;
        row = w + (int64_t)(first < n ? first : n - 1) * kp, hop = (int64_t)step * kp;
#pragma unroll
        for (int i = 0; i < AHEAD; i++) fetch(i);
    }
    // done(i, row i . x) for each of them, in all lanes
    template <typename F>
    __device__ __forceinline__ void run(const FhRowInput &x, F done) {
        float acc = 0.f;
        int p = 0, i = 0;
        const int total = count * pieces;
        for (int t = 0; t < total; t += AHEAD) {
#pragma unroll
            for (int s = 0; s < AHEAD; s++) {
                const float *at = x.xs + p * 256 + (lane8 >> 1);
                const float4 a = *(const float4 *)at, b = *(const float4 *)(at + x.plane);
                acc = fh_dot8(u[s], a, b, acc);
                fetch(s);
                if (++p == pieces) {
                    acc = fh_wave_sum(acc);
                    if (i < count) done(i, acc); // (what is behind the last row is the last piece again)
                    acc = 0.f, p = 0, i++;
                }
            }
        }
    }
};
// Several matrices in one launch of at most `most` workgroups: as few rows a workgroup as that allows; tiles[i]: workgroups of matrix i.
static inline int fh_row_share(const int *n, int count, int most, int *tiles) {
    int64_t total = 0;
    for (int i = 0; i < count; i++) total += n[i];
    for (int64_t per = (total + most - 1) / most;; per++) {
        int64_t sum = 0;
        for (int i = 0; i < count; i++) sum += tiles[i] = (int)((n[i] + per - 1) / per);
        if (sum <= most || per >= total) return (int)sum;
    }
}

// ---------------------------------------------------------------- host launchers
// Storage of activations between kernels: FH_F32, or FH_BF16_ACT for decoders that serve in bf16.
enum { FH_BF16_ACT = 2 };
static inline size_t fh_act_size(int dtype) { return dtype == FH_BF16_ACT ? 2 : 4; }

// Row groups of a grouped product: tile i covers rows [row0, row0 + rows) that all belong to group `group`.
// A tile is number `at` of `of` (8 at most) neighbours of its group whose products are worked on together.
struct FhTile { int group, row0, rows; short at, of; };
// Tile j of a group of `rows` rows: row tiles of more than 128 rows share them out evenly, in steps of 32.
__host__ __device__ static inline int fh_tiles_of(int rows, int tile_rows) { return (rows + tile_rows - 1) / tile_rows; }
__host__ __device__ static inline FhTile fh_tile(int group, int row0, int rows, int j, int tile_rows) {
    const int n = fh_tiles_of(rows, tile_rows), steps = (rows + 31) / 32, of = n - (j & ~7);
    const int from = tile_rows > 128 ? (int)((int64_t)steps * j / n) * 32 : j * tile_rows;
    const int to = tile_rows > 128 ? (int)((int64_t)steps * (j + 1) / n) * 32 : from + tile_rows;
    return FhTile{group, row0 + from, (to < rows ? to : rows) - from, (short)(j & 7), (short)(of < 8 ? of : 8)};
}

enum {
    FH_GEMM_F32 = 0,        // y f32 [m, ldy]
    FH_GEMM_ACT = 1,        // y in the activation type [m, ldy]
    FH_GEMM_ACT_T = 2,      // y in the activation type, transposed: [n, ldy], ldy >= m
    FH_GEMM_SWIGLU = 3,     // weight rows in alternating groups of 16 (gate, up): y = silu(gate) * up, activation type [m, ldy]
    FH_GEMM_RELU2 = 4       // y = max(x, 0)^2, activation type [m, ldy]
};
struct FhGemm {
    const uint16_t *w = nullptr; // [n, kp]
    int64_t w_group = 0;         // elements between the weights of two groups
    const void *x = nullptr;     // [rows, kp]
    const int *gather = nullptr; // row of x behind row i (NULL: i)
    void *y = nullptr;
    int64_t ldy = 0;
    int n = 0, kp = 0, m = 0;    // n: weight rows of a group
    const FhTile *tiles = nullptr; // grouped: device table and its fill count
    const int *n_tiles = nullptr;
    int max_tiles = 0, tile_rows = 64; // rows an entry may cover: 64, or with bf16 activations 128 or a multiple of 32 up to 320
};
fh_status fh_gemm(fh_device *dev, int dtype, int epi, const FhGemm &g);

// y[seg][row] = W_seg[row, :] . n(x), n(x) = x / rms(x) * w (w NULL: x as it is).  norm_out (optional, with w) receives n(x), kp values.
struct FhMvSeg { const uint16_t *w; float *y; int n; };
fh_status fh_matvec_norm(fh_device *dev, const float *x, int k, const float *w, float eps, const FhMvSeg *segs, int n_segs,
                         float *norm_out);
int fh_head_rows_from(int k, int n); // from how many rows on the pass below is faster than a matvec for each
// y[place[i]] [n] = W . n(x row row[i]) for `count` rows that share the pass over the weights; norm_out: n(the last row), kp values.
fh_status fh_head_rows(fh_device *dev, const float *x, int k, const float *w, float eps, const uint16_t *out, int n, const int *row,
                       const int *place, int count, float *y, int64_t ldy, float *norm_out);
// f32 rows -> activation rows of stride kp: plain copy, or RMS norm with weight w (w NULL: copy)
fh_status fh_rows_to_act(fh_device *dev, int dtype, const float *x, int64_t ldx, int rows, int k, const float *w, float eps,
                         void *y, int kp);

// The row table of a product whose `groups` groups have s rows each, group after group (FhGemm::tiles, n_tiles).
static inline int fh_group_tile_rows(const fh_device *dev, int dtype, int groups, int s, int n) {
    // tiles of up to 256 rows where their rounds of workgroups cost less than those of 128 rows (fh_gemm): four groups of 2048 rows,
    // 4096 x 4096 253 us (300)
    const int64_t opt = dev->opt_matmul_kernel, cus = dev->compute_units, wn = (n + 255) / 256;
    const int64_t t256 = groups * wn * ((s + 255) / 256), t128 = groups * wn * ((s + 127) / 128);
    const bool tall = t256 * 4 >= cus * 3 && (t128 + cus - 1) / cus * 2 >= (t256 + cus - 1) / cus * 3;
    if (dtype != FH_F32 && opt != 3 && opt != 14 && (opt == 4 || tall)) return 256;
    return dtype != FH_F32 && (int64_t)groups * ((s + 127) / 128) * ((n + 127) / 128) >= dev->compute_units ? 128 : 64;
}
fh_status fh_group_tiles(fh_device *dev, int groups, int s, int tile_rows, FhTile *tiles, int *n_tiles);

// ---------------------------------------------------------------- residual streams that are normed at a sublayer's end
// x_out = x + y / rms(y) * w per row, and (act not NULL) x_out as activation rows of stride kp; x_out may be x.
fh_status fh_add_normed(fh_device *dev, int dtype, const float *x, const float *y, int rows, int k, const float *w, float eps,
                        float *x_out, void *act, int kp);
// x[t] = table row ids[t] + pos row (pos + t, or *pos_dev for one token); pos_table NULL: without.  Also activation rows.
fh_status fh_embed_at(fh_device *dev, int dtype, const fh_qmatrix *table, const fh_qmatrix *pos_table, const uint32_t *ids, int s,
                      int pos, const int *pos_dev, float *x, void *act, int kp);

// Token shift: mixture n of token t is x_t + (x_(t-1) - x_t) * mu_n.  The row ahead of the portion is kept in a state of two
// rows (position p in row p % 2; nothing is read at position 0).
enum { FH_SHIFT_MAX = 6 };
struct FhShift {
    int n = 0;
    const float *mu[FH_SHIFT_MAX] = {};
    void *y[FH_SHIFT_MAX] = {};   // [s, kp]
    int f32[FH_SHIFT_MAX] = {};   // rows in f32 whatever the activation type
};
// y = tanh(W x) in 32 bits, W [n, kp] for a small n: x [rows, kp] f32, y [rows, ldy] f32 with zeros from n on.
fh_status fh_low_rank_tanh(fh_device *dev, const float *x, int kp, int rows, const uint16_t *w, int n, float *y, int ldy);
fh_status fh_token_shift(fh_device *dev, int dtype, const FhShift &m, const float *x, int s, int k, int pos, float *state, int kp);

// Decode: x' = x + y / rms(y) * w (y NULL: x), then up to FH_MV_MAX matrices on mixtures of x' (mu NULL: x' itself).  One
// workgroup stores x' (x_out, not x) and, with a state, the row of this position.
// With a gate: x' = x / rms(x) * w * silu(gate) * scale, the norm over `groups` equal groups of x (w NULL: without).
enum { FH_MV_ACT_NONE = 0, FH_MV_ACT_RELU2 = 1, FH_MV_ACT_TANH = 2, FH_MV_MAX = 6 };
struct FhMvMix { const uint16_t *w; const float *mu; float *y; int n, act; };
struct FhMvAdd {
    const float *x = nullptr, *y = nullptr, *w = nullptr;
    const float *norm = nullptr;  // x' = x / rms(x) * norm instead (fh_matvec_norm)
    float eps = 0.f;
    float *x_out = nullptr;
    float *state = nullptr;       // [2][k]
    const int *pos_dev = nullptr;
    const float *gate = nullptr;
    int groups = 0, w_len = 0;
    float scale = 1.f;
};
fh_status fh_matvec_mix(fh_device *dev, const FhMvAdd &in, int k, const FhMvMix *segs, int n_segs);

#ifdef __HIPCC__
// Dimension i of a head after rotation: pairs (2i, 2i + 1), or (i, i + pairs) with `halves`, of the first 2 pairs dimensions;
// at(i) gives dimension i before it, ct / st the row of the position.
template <typename F>
__device__ __forceinline__ float fh_rotated(F at, int i, int pairs, int halves, const float *ct, const float *st) {
    const float v = at(i);
    if (i >= 2 * pairs) return v;
    if (halves) return i < pairs ? v * ct[i] - at(i + pairs) * st[i] : v * ct[i - pairs] + at(i - pairs) * st[i - pairs];
    const int p = i >> 1;
    return i & 1 ? v * ct[p] + at(i - 1) * st[p] : v * ct[p] - at(i + 1) * st[p];
}
#endif
