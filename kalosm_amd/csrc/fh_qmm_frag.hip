// Quantized matmul for prompts: Y[m, n] = X[m, k] . deq(W)[n, k]^T with both operands laid out once per call in the order
// the matrix cores take them ("fragments"), and a product that does nothing but move and multiply fragments.
//
// A fragment is the operand of one v_mfma_f32_32x32x16_f16: 32 rows x 16 of k, 1 KB, lane l = row l % 32, k 8 (l / 32) .. + 8.
// Operands are stored [row group of 32][k / 16][1 KB]: an LDS-direct load of a wavefront takes one whole fragment from 1 KB of
// consecutive memory to 1 KB of consecutive LDS, a later operand read is lane * 16 plus a constant - no swizzle, no bank
// conflicts, no address arithmetic.
//
// Weights are written as integer codes that an f16 holds exactly, so the block scale is applied to f32 sums:
//   Q4_K / Q5_K  sc * q (at most 945 / 1953), d per 256; the offsets dmin * m are ordinary columns behind the codes (below)
//   Q6_K         sc * (q - 32) = hi + lo, hi its f16 rounding and lo what that leaves (-1, 0, 1), d per 256
//   Q8_0, Q4_0, Q5_0   the code, d per 32
// Activations are the planes of the other tile kernels: a power of two per row, hi + lo (f32 input) or one exact term (bf16).
// Products: w x_hi (+ w x_lo), for Q6_K hi x_hi (+ hi x_lo) + lo x_hi.  With f32 input Q6_K drops lo x_lo, at most 2^-22 of
// the largest product, the residue the split form of the tile kernels has as well.
//
// Offsets: y -= sum over sub-blocks s of dmin m_s * (sum of the 32 activations of s).  With w = -64 dmin m_s (a power of two per
// row brings it into the f16 range) = wh + wl and the activation sums / 64 = sh + sl these are k / 32 columns more:
// [wh | wl] against planes [sh | sh], [sl | sl] (two activation planes), or [wh | wl | wh] against [sh | sh | sl] (one).
//
// Why two passes: the tile kernels that decode inside the product decode every weight once per 256 rows of activations and
// put it through vector ALU, LDS write and barrier each time; here the decode is one pass over memory.
#include "fh_blocks.h"
#include "fh_qmm_frag.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// ------------------------------------------------------------------------------ activations
// Columns behind the codes' (k / 16 fragments): what the offsets take, rounded up to 128.
static int frag_ext(int k, int planes) { return (k / 32 * (planes == 2 ? 2 : 3) + 127) / 128 * 128; }

// One workgroup: eight rows, one of gridDim.y runs of k.  IN: 0 f32, 1 bf16.  A wavefront finds the maximum of one row; then a
// thread converts eight consecutive values of row t % 8, so that a wavefront reads 256 bytes of each row and writes whole
// 128-byte runs.  sums: [8][run / 32] floats of dynamic LDS when ext > 0.  Eight requests of a row on their way: 2048 rows of an 8B prompt's
// widths take 29.9 us a call (34.3 with the loops as they come).
template <int IN>
__global__ __launch_bounds__(512) void k_frag_x(const void *__restrict__ xin, int m, int k, int ext, uint8_t *__restrict__ out,
                                                 int64_t plane, float *__restrict__ rs) {
    extern __shared__ float sums[];
    __shared__ float s_sc[8];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int row0 = (int)blockIdx.x * 8;
    {
        const int row = row0 + wave < m ? row0 + wave : m - 1;
        float amax = 0.f;
        if (IN == 1) {
            const uint16_t *p = (const uint16_t *)xin + (int64_t)row * k;
#pragma unroll 8
            for (int c = lane * 8; c < k; c += 512) {
                const uint4 u = *(const uint4 *)(p + c);
                const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int e = 0; e < 4; e++)
                    amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(w[e] << 16)), fabsf(__uint_as_float(w[e] & 0xFFFF0000u))));
            }
        } else {
            const float *p = (const float *)xin + (int64_t)row * k;
#pragma unroll 8
            for (int c = lane * 4; c < k; c += 256) {
                const float4 a = *(const float4 *)(p + c);
                amax = fmaxf(amax, fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))));
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
        int e = 141 - (int)((__float_as_uint(amax) >> 23) & 0xFFu); // 14 - floor(log2 amax); zero / inf / nan clamp
        e = e > 100 ? 100 : (e < -100 ? -100 : e);
        const bool infrow = amax == INFINITY; // finite values vanish next to an infinity, which is carried as +-32768
        if (lane == 0) {
            s_sc[wave] = infrow ? -__uint_as_float((uint32_t)(e + 127) << 23) : __uint_as_float((uint32_t)(e + 127) << 23);
            if (blockIdx.y == 0 && row0 + wave < m) rs[row0 + wave] = infrow ? INFINITY : __uint_as_float((uint32_t)(127 - e) << 23);
        }
    }
    __syncthreads();
    const int r = tid & 7, row = row0 + r;
    const bool live = row < m, infrow = s_sc[r] < 0.f;
    const float sc = fabsf(s_sc[r]);
    const int kf = (k + ext) >> 4;
    uint8_t *dst = out + ((int64_t)(row >> 5) * kf) * 1024 + (row & 31) * 16;
    const int parts = (int)gridDim.y, span = ((k + parts - 1) / parts + 511) / 512 * 512, ns = k >> 5;
    const int from = (int)blockIdx.y * span, to = from + span < k ? from + span : k; // (whole 512s, so whole runs of 8 sums)
    for (int at = from; at < to; at += 512) {
        const int c = at + (tid >> 3) * 8;
        float v[8];
        if (live && c < to) {
            if (IN == 1) {
                const uint4 u = *(const uint4 *)((const uint16_t *)xin + (int64_t)row * k + c);
                const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int e = 0; e < 4; e++) v[2 * e] = __uint_as_float(w[e] << 16), v[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
            } else {
                const float4 a = *(const float4 *)((const float *)xin + (int64_t)row * k + c);
                const float4 b = *(const float4 *)((const float *)xin + (int64_t)row * k + c + 4);
                v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = 0.f;
        }
        _Float16 h[8], l[8];
        float t = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float w = v[e] * sc;
            if (infrow && fabsf(w) == INFINITY) w = copysignf(32768.f, w);
            h[e] = (_Float16)w;
            const float d = w - (float)h[e];
            l[e] = (_Float16)(d == d ? d : 0.f); // a NaN stays in the hi plane alone
            t += w;
        }
        if (live && c < to) {
            uint8_t *p = dst + (int64_t)(c >> 4) * 1024 + ((c >> 3) & 1) * 512;
            uint4 u;
            __builtin_memcpy(&u, h, 16);
            *(uint4 *)p = u;
            if (IN != 1) {
                __builtin_memcpy(&u, l, 16);
                *(uint4 *)(p + plane) = u;
            }
        }
        if (ext) { // sums of 32: four threads eight lanes apart
            t += __shfl_xor(t, 8, 64);
            t += __shfl_xor(t, 16, 64);
            if (c < to && (lane & 24) == 0) sums[r * (span >> 5) + ((c - from) >> 5)] = t * 0.015625f;
        }
    }
    if (!ext) return;
    __syncthreads();
    // the run's sums, eight columns a thread, into every place they have; the columns behind them are zero
    auto put = [&](int col, const _Float16 *a, const _Float16 *b) {
        uint8_t *p = dst + (int64_t)((k + col) >> 4) * 1024 + ((col >> 3) & 1) * 512;
        uint4 u;
        __builtin_memcpy(&u, a, 16);
        *(uint4 *)p = u;
        if (IN != 1) {
            __builtin_memcpy(&u, b, 16);
            *(uint4 *)(p + plane) = u;
        }
    };
    if (!live) return;
    for (int c = (from >> 5) + (tid >> 3) * 8; c < (to >> 5); c += 512) {
        _Float16 sh[8], sl[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float s = sums[r * (span >> 5) + c - (from >> 5) + e];
            sh[e] = (_Float16)s;
            sl[e] = (_Float16)(s - (float)sh[e]);
        }
        put(c, sh, sl);
        put(c + ns, sh, sl);
        if (IN == 1) put(c + 2 * ns, sl, sl);
    }
    const _Float16 z[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (blockIdx.y == 0)
        for (int c = ns * (IN == 1 ? 3 : 2) + (tid >> 3) * 8; c < ext; c += 512) put(c, z, z);
}

// ------------------------------------------------------------------------------ weights
__device__ __forceinline__ void frag_store(uint8_t *p, const _Float16 *h) {
    uint4 u;
    __builtin_memcpy(&u, h, 16);
    *(uint4 *)p = u;
}

// One workgroup: a tile of 16 rows of the tiled layout, its wavefronts share out the 256-runs of k; lane = (lane group g, row j)
// of the layout.  `d` receives the scales [k / 256 (+ 1)] (formats with one per 256; the last one belongs to the offsets) or
// [k / 32], n_pad apart.  ext columns as in k_frag_x; plane: distance of the second weight plane (Q6_K).
// half > 0 (a multiple of 32): rows i and half + i belong together (gate and up); their groups of 32 are stored in turn, so that a
// wavefront of the product holds both.
template <int T>
__global__ __launch_bounds__(512) void k_frag_w(QView q, int64_t tile0, int ext, int xplanes, uint8_t *__restrict__ out,
                                                 int64_t plane, float *__restrict__ d, int64_t n_pad, int half) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int64_t tile = tile0 + blockIdx.x;
    const int k = (int)q.k, kf = (k + ext) >> 4;
    int row = (int)blockIdx.x * 16;
    if (half) row = row < half ? (row & ~31) * 2 + (row & 31) : ((row - half) & ~31) * 2 + 32 + ((row - half) & 31);
    row += j;
    uint8_t *dst = out + ((int64_t)(row >> 5) * kf) * 1024 + (row & 31) * 16;
    const uint8_t *recs = q.data + tile * q.recs * q.rec_bytes;
    const int runs = (k + 255) >> 8;
    float dscale = 1.f;
    if (T == FH_Q4_K || T == FH_Q5_K) { // the power of two of the row's offsets
        __shared__ float s_max[8][16];
        float top = 0.f;
        for (int b = tid >> 4; b < runs; b += 32)
            top = fmaxf(top, fabsf(fh_h2f(fh_ld16(recs + (int64_t)b * q.rec_bytes + 16 * j + 2))));
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        if (lane < 16) s_max[wave][lane] = top;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; i++) top = fmaxf(top, s_max[i][j]);
        int e = 135 - (int)((__float_as_uint(top) >> 23) & 0xFFu); // dmin * 63 below 2^15
        e = e > 100 ? 100 : (e < -100 ? -100 : e);
        dscale = __uint_as_float((uint32_t)(e + 127) << 23);
        if (wave == 0 && g == 0)
            for (int i = 0; i < (ext + 255) >> 8; i++) d[(int64_t)(runs + i) * n_pad + row] = -64.f * __uint_as_float((uint32_t)(127 - e) << 23);
    }
    for (int b = wave; b < runs; b += 8) {
        uint8_t *pb = dst + (int64_t)b * 16 * 1024;
        if (T == FH_Q4_K || T == FH_Q5_K) {
            const uint8_t *rec = recs + (int64_t)b * (T == FH_Q5_K ? 2816 : 2304);
            const uint4 h = *(const uint4 *)(rec + 16 * j);
            uint2 hb = make_uint2(0, 0);
            if (T == FH_Q5_K) hb = *(const uint2 *)(rec + 2304 + lane * 8);
            const uint32_t sc[2] = {h.y & 0x3F3F3F3Fu, (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u)};
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const uint4 c = *(const uint4 *)(rec + 256 + p * 1024 + lane * 16);
                const uint32_t cw[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int hn = 0; hn < 2; hn++) {
                        const int sb = 4 * p + 2 * u + hn; // sub-block: elements 32 sb + 8 g ..
                        const _Float16 s = (_Float16)(float)((sc[p] >> (8 * (sb & 3))) & 0xFFu);
                        _Float16 w[8];
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            uint32_t v = (cw[2 * u + (i >> 2)] >> (8 * (i & 3) + 4 * hn)) & 15u;
                            if (T == FH_Q5_K) v += (((i < 4 ? hb.x : hb.y) >> (8 * (i & 3) + sb)) & 1u) << 4;
                            w[i] = (_Float16)(float)v * s;
                        }
                        frag_store(pb + (2 * sb + (g >> 1)) * 1024 + (g & 1) * 512, w);
                    }
            }
            if (g == 0) d[(int64_t)b * n_pad + row] = fh_h2f((uint16_t)(h.x & 0xFFFF));
            // the block's eight offsets: lane group 0 writes the hi columns, 1 the lo columns, 2 (one activation plane) hi again
            const float dm = fh_h2f((uint16_t)(h.x >> 16)) * dscale;
            const uint32_t mn[2] = {h.z & 0x3F3F3F3Fu, ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)};
            _Float16 w[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float o = dm * (float)((mn[i >> 2] >> (8 * (i & 3))) & 0xFFu);
                const _Float16 oh = (_Float16)o;
                w[i] = g == 1 ? (_Float16)(o - (float)oh) : oh;
            }
            const int col = k + g * (k >> 5) + 8 * b;
            if (g < (xplanes == 2 ? 2 : 3)) frag_store(dst + (int64_t)(col >> 4) * 1024 + ((col >> 3) & 1) * 512, w);
        } else if (T == FH_Q6_K) {
            const uint8_t *rec = recs + (int64_t)b * 3360;
            uint4 lw[2];
            lw[0] = *(const uint4 *)(rec + lane * 16);
            lw[1] = *(const uint4 *)(rec + 1024 + lane * 16);
            const uint4 hw4 = *(const uint4 *)(rec + 2048 + lane * 16);
            const uint32_t hws[4] = {hw4.x, hw4.y, hw4.z, hw4.w};
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const uint4 l4 = lw[t >> 2];
                const uint32_t l = (t & 3) == 0 ? l4.x : (t & 3) == 1 ? l4.y : (t & 3) == 2 ? l4.z : l4.w, hw = hws[t >> 1];
                const int sc = (int)(int8_t)rec[q6k_sc_off(j, 2 * t + (g >> 1))];
                _Float16 hi[8], lo[8];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int pp = i >> 1, odd = i & 1;
                    const int nib = (int)((l >> (4 * (pp + 4 * odd))) & 15u), two = (int)((hw >> (q6k_hbit(t, pp) + 16 * odd)) & 3u);
                    const float v = (float)(sc * (((two << 4) | nib) - 32));
                    hi[i] = (_Float16)v;
                    lo[i] = (_Float16)(v - (float)hi[i]);
                }
                uint8_t *p = pb + (2 * t + (g >> 1)) * 1024 + (g & 1) * 512;
                frag_store(p, hi);
                frag_store(p + plane, lo);
            }
            if (g == 0) d[(int64_t)b * n_pad + row] = fh_h2f(fh_ld16(rec + q6k_d_off(j)));
        } else { // a scale per 32: eight blocks (as many as there are)
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int blk = 8 * b + u;
                if (blk * 32 >= k) break;
                uint8_t *p = dst + (int64_t)blk * 2048;
                if (T == FH_Q8_0) {
                    const uint8_t *rec = recs + (int64_t)(blk >> 1) * 1088;
                    const uint2 c = *(const uint2 *)(rec + lane * 16 + 8 * (u & 1));
                    _Float16 w[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) w[i] = (_Float16)(float)(int)(int8_t)((i < 4 ? c.x : c.y) >> (8 * (i & 3)));
                    frag_store(p + (g >> 1) * 1024 + (g & 1) * 512, w);
                    if (g == 0) d[(int64_t)blk * n_pad + row] = fh_h2f(fh_ld16(rec + 1024 + 4 * j + 2 * (u & 1)));
                } else { // nibble order: bytes 4 g .. of the block are elements 4 g .. and 16 + 4 g ..
                    const uint8_t *rec = recs + (int64_t)(blk >> 2) * (T == FH_Q5_0 ? 1408 : 1152);
                    const uint32_t c = *(const uint32_t *)(rec + lane * 16 + 4 * (u & 3));
                    const uint32_t hb = T == FH_Q5_0 ? rec[q50_qh_off(j, u & 3, g)] : 0u;
                    _Float16 a[4], e[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        int lo = (int)((c >> (8 * i)) & 15u), hi = (int)((c >> (8 * i + 4)) & 15u);
                        if (T == FH_Q5_0) lo |= (int)((hb >> i) & 1u) << 4, hi |= (int)((hb >> (4 + i)) & 1u) << 4;
                        a[i] = (_Float16)(float)(lo - (T == FH_Q5_0 ? 16 : 8));
                        e[i] = (_Float16)(float)(hi - (T == FH_Q5_0 ? 16 : 8));
                    }
                    uint2 u0, u1;
                    __builtin_memcpy(&u0, a, 8);
                    __builtin_memcpy(&u1, e, 8);
                    *(uint2 *)(p + (g >> 1) * 512 + (g & 1) * 8) = u0;
                    *(uint2 *)(p + 1024 + (g >> 1) * 512 + (g & 1) * 8) = u1;
                    if (g == 0) d[(int64_t)blk * n_pad + row] = fh_h2f(fh_ld16(rec + 1024 + 8 * j + 2 * (u & 3)));
                }
            }
        }
    }
    if ((T == FH_Q4_K || T == FH_Q5_K)) { // columns behind the offsets are zero
        const int used = (k >> 5) * (xplanes == 2 ? 2 : 3);
        const uint4 z = make_uint4(0, 0, 0, 0);
        for (int c = k + used + (tid >> 4) * 8; c < k + ext; c += 256)
            *(uint4 *)(dst + (int64_t)(c >> 4) * 1024 + ((c >> 3) & 1) * 512) = z;
    }
}

// ------------------------------------------------------------------------------ product
struct FragArgs {
    const uint8_t *w, *x;
    int64_t w_plane, x_plane;
    const float *d;  // scales, n_pad apart
    int64_t n_pad;
    const float *rs;
    float *y;
    int64_t ldy;     // outputs of a row of y
    int m, n, n0;    // rows, weight rows of this launch, first of them in y
    int kf, tiles_w, tiles_x, parts;
    float *part;         // partial planes of a split k,
    int64_t part_stride; // so many floats apart
    int half;            // > 0: y[:, i] = silu(row i) * (row half + i)
};

// NW / NX: weight and activation planes; SC: k per scale (32 or 256); a wavefront owns FW x FX tiles of 32 x 32, the eight
// wavefronts of a workgroup are 8 / WGX along the weight rows x WGX along the activation rows.
// A step is 16 of k, one fragment per row group and plane; as many stages in the LDS as fit, up to six.  The wait ahead of the
// barrier of step s is for stage s + 1, so the operands of step s are already in registers and the matrix cores never wait for
// the LDS behind a barrier; the stages behind s + 1 stay on their way.
// The loop runs over 256 of k (straight-line), with 128 left over at most: scales are requested a round ahead, and without a
// condition in between the compiler knows how many requests are younger and waits for none of them.
template <int NW, int NX, int FW, int FX, int WGX>
struct FragTile {
    static constexpr int TW = 8 / WGX * FW * 32, TX = WGX * FX * 32;
    static constexpr int UW = NW * TW / 32, UX = NX * TX / 32, PIECES = UW + UX; // fragments (1 KB) of a stage
    static constexpr int STAGE = PIECES * 1024, FIT = 163840 / STAGE, STAGES = FIT > 6 ? 6 : FIT;
    static constexpr int PW = (PIECES + 7) / 8;                                  // requests of a wavefront per stage
    static_assert(STAGES >= 4, "four stages at least");
};

template <int NW, int NX, int SC, int FW, int FX, int WGX>
__global__ __launch_bounds__(512) void k_qmm_frag(FragArgs g) {
    typedef FragTile<NW, NX, FW, FX, WGX> Tile;
    constexpr int TW = Tile::TW, TX = Tile::TX, UW = Tile::UW, PW = Tile::PW, STAGE = Tile::STAGE, STAGES = Tile::STAGES;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31;
    const int ww = wave / WGX, wx = wave % WGX;
    // Workgroups go to the eight dies in turn.  A die takes a run of tiles, in groups of eight weight tiles by all activation
    // tiles, weight tiles first: what runs on it at a time is about 8 x 4 tiles that share their operands in its L2.
    const int total = g.tiles_w * g.tiles_x * g.parts, per = total >> 3, more = total & 7, die = (int)blockIdx.x & 7;
    int lin = ((int)blockIdx.x >> 3) + die * per + (die < more ? die : more);
    const int part = lin / (g.tiles_w * g.tiles_x);
    lin -= part * g.tiles_w * g.tiles_x;
    const int group = lin / (8 * g.tiles_x), in = lin - group * 8 * g.tiles_x;
    const int gw = g.tiles_w - group * 8 < 8 ? g.tiles_w - group * 8 : 8;
    const int tw = group * 8 + in % gw, tx = in / gw;
    const int rounds = (g.kf + 15) >> 4; // of 256 of k
    const int s0 = rounds * part / g.parts * 16, s_end = rounds * (part + 1) / g.parts * 16;
    const int s1 = s_end < g.kf ? s_end : g.kf; // steps of this workgroup
    // this wavefront's fragments of a stage: wave + 8 i.  (Past the last one, where they do not divide: the last one again, the
    // same bytes to the same place.)
    const uint8_t *src[PW];
    int at[PW];
#pragma unroll
    for (int i = 0; i < PW; i++) {
        const int u = wave + 8 * i < Tile::PIECES ? wave + 8 * i : Tile::PIECES - 1;
        const uint8_t *base = u < UW ? g.w + (u / (TW / 32)) * g.w_plane + ((int64_t)(tw * (TW / 32) + u % (TW / 32)) * g.kf) * 1024
                                     : g.x + ((u - UW) / (TX / 32)) * g.x_plane +
                                           ((int64_t)(tx * (TX / 32) + (u - UW) % (TX / 32)) * g.kf) * 1024;
        src[i] = base;
        at[i] = u * 1024;
    }
    auto fetch = [&](int s, int buf) { // step s into the buffer at byte `buf`; past the end a repeat, so that the counts stay equal
        const int o = (s < s1 ? s : s1 - 1) * 1024;
#pragma unroll
        for (int i = 0; i < PW; i++)
            fh_buffer_to_lds(src[i], g.kf * 1024, smem + buf + at[i], lane * 16, o);
    };
    half8 fw[2][NW][FW], fx[2][NX][FX];
    auto read = [&](int set, int buf) {
        const uint8_t *b = smem + buf + lane * 16;
#pragma unroll
        for (int p = 0; p < NW; p++)
#pragma unroll
            for (int a = 0; a < FW; a++) fw[set][p][a] = *(const half8 *)(b + (p * (TW / 32) + ww * FW + a) * 1024);
#pragma unroll
        for (int p = 0; p < NX; p++)
#pragma unroll
            for (int c = 0; c < FX; c++) fx[set][p][c] = *(const half8 *)(b + (UW + p * (TX / 32) + wx * FX + c) * 1024);
    };
    floatx16 acc[FW][FX], sum[FW][FX];
    const floatx16 zero = {0.f};
#pragma unroll
    for (int a = 0; a < FW; a++)
#pragma unroll
        for (int c = 0; c < FX; c++) {
            acc[a][c] = zero;
            if (SC == 32) sum[a][c] = zero;
        }
    // neighbouring products belong to different tiles, so that none waits for the one before it
    auto mul = [&](int set, int a0, int a1, bool first) {
#pragma unroll
        for (int t = 0; t < (NW == 2 ? NX + 1 : NX); t++)
#pragma unroll
            for (int a = a0; a < a1; a++)
#pragma unroll
                for (int c = 0; c < FX; c++)
                    sum[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fx[set][t < NX ? t : 0][c], fw[set][t < NX ? 0 : NW - 1][a],
                                                                       first && t == 0 ? zero : sum[a][c], 0, 0, 0);
    };
    const float *dp = g.d + tw * TW + ww * FW * 32 + li;
    constexpr int ND = SC == 32 ? 4 : 2; // scales on their way: of four 32s, of two 256s
    float dv[ND][FW];
    const int d_last = SC == 32 ? (s1 - 1) >> 1 : (s1 - 1) >> 4;
    auto load_d = [&](int slot, int i) {
        const int at_ = i < d_last ? i : d_last;
#pragma unroll
        for (int a = 0; a < FW; a++) dv[slot][a] = dp[(int64_t)at_ * g.n_pad + a * 32];
    };
    auto scale = [&](int slot, int a0, int a1) {
#pragma unroll
        for (int a = a0; a < a1; a++)
#pragma unroll
            for (int c = 0; c < FX; c++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[a][c][r] = fmaf(sum[a][c][r], dv[slot][a], acc[a][c][r]);
    };
    int cur = 0;
    // e: s within its round.  With a scale per 32 the second half of the tiles is scaled between the products of the next
    // step, the first half behind those of its own: the vector ALU works while the matrix cores do.
    auto step = [&](int s, int e) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 3) * PW) : "memory"); // stage s + 1 has landed ...
        __builtin_amdgcn_s_barrier();                                            // ... everywhere; the buffer of s - 1 is free
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int nxt = cur + STAGE == STAGES * STAGE ? 0 : cur + STAGE;
        const int i = e >> 1;
        if (SC == 32 && (e & 1) == 0) load_d((i + 2) & 3, (s >> 1) + 2);
        read((e + 1) & 1, nxt);
        fetch(s + STAGES - 1, cur == 0 ? (STAGES - 1) * STAGE : cur - STAGE);
        if (SC == 256) mul(e & 1, 0, FW, e == 0);
        else if ((e & 1) == 0) {
            mul(0, 0, FW / 2, true);
            scale((i + 3) & 3, FW / 2, FW);
            mul(0, FW / 2, FW, true);
        } else {
            mul(1, 0, FW, false);
            scale(i & 3, 0, FW / 2);
        }
        if (SC == 32) // an operand read and some of the scaling behind every product
#pragma unroll
            for (int p = 0; p < FW * FX * NX; p++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 8 / NX, 0);
            }
        cur = nxt;
    };
    if (SC == 32) { // (the sums ahead of the first 32 are zero)
        load_d(0, s0 >> 1);
        load_d(1, (s0 >> 1) + 1);
#pragma unroll
        for (int a = 0; a < FW; a++) dv[ND - 1][a] = 0.f;
    } else {
        load_d(0, s0 >> 4);
    }
#pragma unroll
    for (int i = 0; i < STAGES - 1; i++) fetch(s0 + i, i * STAGE);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * PW) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    int s = s0;
    for (; s + 16 <= s1; s += 16) {
        if (SC == 256) {
#pragma unroll
            for (int a = 0; a < FW; a++) dv[1][a] = dv[0][a];
            load_d(0, (s >> 4) + 1);
        }
#pragma unroll
        for (int e = 0; e < 16; e++) step(s + e, e);
        if (SC == 256) scale(1, 0, FW);
    }
    if (s < s1) { // 128 of k left
#pragma unroll
        for (int e = 0; e < 8; e++) step(s + e, e);
        if (SC == 256) scale(0, 0, FW);
    }
    if (SC == 32) scale(3, FW / 2, FW); // (a multiple of four 32s: the last one's scale is in the last place)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // no LDS-direct load outlives the workgroup's LDS
    // The rows' factors ahead of all stores: a load between them would wait for the stores before it (one counter for both).
    float rs[FX][16];
#pragma unroll
    for (int c = 0; c < FX; c++)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            const float4 v = *(const float4 *)(g.rs + tx * TX + (wx * FX + c) * 32 + 2 * r + 4 * (lane >> 5));
            rs[c][r] = v.x, rs[c][r + 1] = v.y, rs[c][r + 2] = v.z, rs[c][r + 3] = v.w;
        }
    float *y = g.y + part * g.part_stride;
    if (g.half) { // (FW is 2: gate and up)
        const int nn = (tw * (TW / 64) + ww) * 32 + li;
        if (nn >= g.half) return;
#pragma unroll
        for (int c = 0; c < FX; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int mm = tx * TX + (wx * FX + c) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (mm >= g.m) continue;
                const float gate = acc[0][c][r] * rs[c][r], up = acc[1][c][r] * rs[c][r];
                y[(int64_t)mm * g.ldy + nn] = (gate / (expf(-gate) + 1.0f)) * up;
            }
        return;
    }
#pragma unroll
    for (int a = 0; a < FW; a++) {
        const int nn = tw * TW + (ww * FW + a) * 32 + li;
        if (nn >= g.n) continue;
#pragma unroll
        for (int c = 0; c < FX; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int mm = tx * TX + (wx * FX + c) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (mm < g.m) y[(int64_t)mm * g.ldy + g.n0 + nn] = acc[a][c][r] * rs[c][r];
            }
    }
}

// Planes added in pairs, pairs of pairs ..: one after the other 16 planes of one 256 of k each are as inexact as one chain along k (1024 x 4096,
// 20 bf16 rows, against 64 bits 1.0e-7 in Q4_K and 1.23e-7 in Q6_K; in pairs 8.5e-8 and 1.11e-7, and all planes asked for at once: 16.0 us / 13.3).  MAX: planes at most.
template <int MAX>
__global__ void k_frag_sum(const float *__restrict__ part, int parts, int64_t stride, int64_t count, float *__restrict__ y) {
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= count) return;
    if (i + 3 < count && (stride & 3) == 0 && ((uintptr_t)y & 15) == 0) {
        float4 v[MAX];
#pragma unroll
        for (int p = 0; p < MAX; p++) v[p] = *(const float4 *)(part + (p < parts ? p : 0) * stride + i);
#pragma unroll
        for (int h = 1; h < MAX; h *= 2)
#pragma unroll
            for (int p = 0; p < MAX; p += 2 * h)
                if (p + h < parts) v[p] = make_float4(v[p].x + v[p + h].x, v[p].y + v[p + h].y, v[p].z + v[p + h].z, v[p].w + v[p + h].w);
        *(float4 *)(y + i) = v[0];
        return;
    }
    for (int64_t e = i; e < count && e < i + 4; e++) {
        float v[MAX];
#pragma unroll
        for (int p = 0; p < MAX; p++) v[p] = part[(p < parts ? p : 0) * stride + e];
#pragma unroll
        for (int h = 1; h < MAX; h *= 2)
#pragma unroll
            for (int p = 0; p < MAX; p += 2 * h)
                if (p + h < parts) v[p] += v[p + h];
        y[e] = v[0];
    }
}

// ------------------------------------------------------------------------------ launches
fh_status fh_frag_sum(fh_device *dev, const float *part, int parts, int64_t stride, int64_t count, float *y) {
    const dim3 grid((unsigned)((count + 1023) / 1024));
    if (parts <= 2) k_frag_sum<2><<<grid, 256, 0, dev->stream>>>(part, parts, stride, count, y);
    else if (parts <= 4) k_frag_sum<4><<<grid, 256, 0, dev->stream>>>(part, parts, stride, count, y);
    else if (parts <= 8) k_frag_sum<8><<<grid, 256, 0, dev->stream>>>(part, parts, stride, count, y);
    else k_frag_sum<16><<<grid, 256, 0, dev->stream>>>(part, parts, stride, count, y);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

struct FragAsk {
    int parts;                     // of k
    int64_t rounds, steps;         // of workgroups, 128s of k in all of them
    double sum;                    // us for partial planes
};
template <int NW, int NX, int SC, int FW, int FX, int WGX>
static fh_status frag_product(fh_device *dev, FragArgs g, FragAsk *ask) { // ask: only how it would be cut
    typedef FragTile<NW, NX, FW, FX, WGX> Tile;
    constexpr int TW = Tile::TW, TX = Tile::TX, LDS = Tile::STAGES * Tile::STAGE;
    g.tiles_w = (g.n + TW - 1) / TW;
    g.tiles_x = (g.m + TX - 1) / TX;
    // parts of k: the fewest rounds of workgroups by their length, against writing and adding the partial planes.  A step of 128
    // of k takes about 2.5 us, starting and storing a tile as long as 1.5 of them.
    const int quads = g.kf >> 3;
    const int64_t tiles = (int64_t)g.tiles_w * g.tiles_x;
    double best = 1e30;
    int parts = 1;
    FragAsk cut{1, 0, 0, 0.0};
    const int most = g.n == g.ldy || g.half ? 8 : 1; // (weight rows in several launches: whole)
    for (int p = 1; p <= most && p * 2 <= quads; p++) {
        const int64_t rounds = (tiles * p + dev->compute_units - 1) / dev->compute_units;
        const double sum = p > 1 ? 4.0 + (2.0 * p + 1.0) * g.m * (double)g.n * 4.0 / 4e6 : 0.0;
        const double t = (double)rounds * ((double)((quads + p - 1) / p) + 1.5) * 2.5 + sum;
        if (t < best * 0.97) best = t, parts = p, cut = FragAsk{p, rounds, rounds * ((quads + p - 1) / p), sum};
    }
    if (ask) {
        *ask = cut;
        return FH_OK;
    }
    g.parts = parts;
    float *y = g.y;
    if (parts > 1) { // whole planes [m][n] of this launch's weight rows
        g.y = g.part;
        g.part_stride = (int64_t)g.m * g.n;
    }
    FH_TRY(fh_kernel_lds(dev, (const void *)k_qmm_frag<NW, NX, SC, FW, FX, WGX>, (size_t)LDS));
    k_qmm_frag<NW, NX, SC, FW, FX, WGX><<<dim3((unsigned)(tiles * parts)), 512, LDS, dev->stream>>>(g);
    FH_HIP(hipGetLastError());
    return parts > 1 ? fh_frag_sum(dev, g.part, parts, g.part_stride, (int64_t)g.m * g.n, y) : FH_OK;
}

bool fh_qmm_frag_supports(const fh_qmatrix *q) {
    switch (q->type) {
    case FH_Q4_0: case FH_Q8_0: case FH_Q5_0: return q->k % 128 == 0;
    case FH_Q4_K: case FH_Q5_K: case FH_Q6_K: return q->k % 256 == 0;
    }
    return false;
}

// Where the fragments pay for being written, against the tile kernels that decode inside the product (the rows and matrices that
// fh_qmm_reg.hip takes are not asked about: of those up to 64, only k below 1024, above 16384 or no multiple of 256 is left).  Both were timed for 13 - 64
// rows of 12 matrices and 129 - 3000 rows of 23, in every format; us, fragments / tiles, at the lines:
//   Up to 64 rows a tile kernel takes the same time for any matrix whose tiles of 128 rows fit the device at once (32768 rows), the
//     fragments as long as they are: Q4_K f32, 32 rows, 11008 x 4096 55 / 150, 32768 x 4096 145 / 158, 128256 x 4096 595 / 294;
//     Q4_0 22528 x 4096 97 / 142, 28672 x 4096 160 / 141; Q6_K, two planes, 16384 x 4096 128 / 166, 28672 x 4096 232 / 166.
//   Above, they cost 52 us for a 28672 x 4096 matrix whatever the rows (250 MB), and two launches more: narrow matrices need rows
//     for that (640 rows, Q8_0 f32, 512 x 2048 39 / 33, 1024 x 4096 53 / 59, 2048 x 2048 45 / 55), unless their n is no multiple of
//     four, which the tile kernels cannot split k for (Q4_0 130 x 14336: 117 / 434).
//   Few rows (Q4_K f32 257 - 512, Q5_0 129 - 256) are worth it where the tiles leave the device idle: `fill` is what they keep busy
//     of it, with what they spend on rows past m against tiles of 128.  Q4_K f32, 512 rows: 14336 x 4096 150 / 166,
//     4096 x 14336 190 / 172; Q5_0 f32, 192 rows: 6144 x 4096 69 / 89, 4096 x 14336 131 / 128.
//   The 5-bit formats, which the tiles multiply as split f32 values, gain most (Q5_K f32, 4096 x 14336, 512 rows: 190 / 255); one activation
//     plane halves the products but not the fragments (Q4_K bf16, 14336 x 4096: 768 rows 182 / 180, 2048 rows 369 / 415).
//   Left on the tiles although the fragments are up to 1.8 times as fast there: 129 - 512 rows of Q4_0, Q8_0 and Q6_K, f32 (6144 x 4096;
//     4096 x 14336 0.75 - 1.3), 129 - 256 of Q4_K (0.75 - 1.4).  bf16 rows of Q6_K (2048 x 4096 x 14336: 463 / 480, too little) and of
//     Q8_0 (bound by its scaling, 475 / 364) stay there as well.
static double tile_fill(const fh_qmatrix *q, int m) {
    const int64_t cus = q->dev->compute_units, rows = (m + 255) / 256;
    int64_t tiles = (q->n + 127) / 128 * rows, parts = 1, steps = q->k / 32;
    while (tiles * parts * 5 < cus * 4 && parts < 8 && steps % (parts * 4) == 0 && steps / (parts * 2) >= 16) parts *= 2; // (as qmm_launch_t)
    tiles *= parts;
    return (double)tiles / (double)((tiles + cus - 1) / cus * cus) * (double)((m + 127) / 128) / (double)(2 * rows);
}

bool fh_qmm_frag_pays(const fh_qmatrix *q, int x_is_bf16, int m) {
    if (!fh_qmm_frag_supports(q)) return false;
    const int64_t n = q->n, k = q->k, fits = (int64_t)q->dev->compute_units * 128;
    const bool four = q->type == FH_Q4_K || q->type == FH_Q5_K; // one plane, a scale per 256
    if (m <= 64) {
        if (m <= 12 || k < 512) return false;
        if (four) return n <= fits;
        return q->type == FH_Q6_K ? n <= fits * 9 / 16 : n <= (k <= 2048 ? fits : fits * 11 / 16);
    }
    const bool any = n % 4 != 0, wide = n >= 2048 || (n >= 1024 && k >= 4096), rows = m > 1024 && (n >= 1024 || (n >= 512 && k >= 4096));
    switch (q->type) {
    case FH_Q5_K: return m > 128 && (any || n >= 3072 || (m > 256 && n >= 1024) || (m > 512 && n >= 512) || m > 1024);
    case FH_Q5_0:
        if (m <= 256) return m > 128 && (any || (n >= 3072 && n <= fits / 2 && tile_fill(q, m) < 0.9));
        return any || (m <= 512 ? n >= 3072 : wide || rows);
    case FH_Q4_K:
        if (x_is_bf16) return m > 768 && (any || (m <= 1024 ? n >= 2048 && n <= fits / 2 : n >= 512));
        if (m <= 512) return m > 256 && (any || (n >= 2048 && tile_fill(q, m) < 0.9));
        return any || n >= (m <= 1024 ? 1024 : 512);
    }
    return !x_is_bf16 && m > 512 && (any || wide || rows);
}

#define FRAG_GO(NW_, NX_, SC_, WGX_) \
    (m <= 64 ? frag_product<NW_, NX_, SC_, 2, 1, 2>(dev, g, ask) : frag_product<NW_, NX_, SC_, 2, 2, WGX_>(dev, g, ask))
static fh_status frag_go(fh_device *dev, const FragArgs &g, int sc, int wp, int xp, FragAsk *ask) {
    const int m = g.m;
    if (sc == 32) return xp == 2 ? FRAG_GO(1, 2, 32, 2) : FRAG_GO(1, 1, 32, 2);
    if (wp == 2) return xp == 2 ? FRAG_GO(2, 2, 256, 4) : FRAG_GO(2, 1, 256, 4);
    return xp == 2 ? FRAG_GO(1, 2, 256, 2) : FRAG_GO(1, 1, 256, 2);
}
#undef FRAG_GO

struct FragPlan {
    FragArgs g;
    FragAsk cut;             // of a launch
    int ext;                 // columns of offsets
    int64_t rows, row_bytes; // weight rows of a launch
};
static fh_status frag_plan(const fh_qmatrix *q, int x_is_bf16, int m, int half, FragPlan *p) {
    const int k = (int)q->k, xp = x_is_bf16 ? 1 : 2, wp = q->type == FH_Q6_K ? 2 : 1, sc = fh_block_elems(q->type);
    const int ext = q->type == FH_Q4_K || q->type == FH_Q5_K ? frag_ext(k, xp) : 0, kf = (k + ext) / 16;
    // weights: as many rows at a time as 512 MB of fragments and their scales hold (less where the device's scratch is bounded)
    const int64_t rows_all = (q->n + 255) / 256 * 256, scales = sc == 32 ? k / 32 : k / 256 + (ext ? (ext + 255) / 256 : 0);
    const int64_t row_bytes = (int64_t)kf * 32 * wp + scales * 4, bound = q->dev->opt_scratch_limit;
    int64_t rows = (bound > 0 && bound < (512 << 20) ? bound : 512 << 20) / row_bytes / 256 * 256;
    rows = rows < 256 ? 256 : (rows > rows_all ? rows_all : rows);
    p->g = FragArgs{};
    p->g.m = m, p->g.n = (int)(rows < q->n ? rows : q->n), p->g.ldy = half ? half : q->n, p->g.kf = kf, p->g.half = half;
    p->ext = ext, p->rows = rows, p->row_bytes = row_bytes;
    return frag_go(q->dev, p->g, sc, wp, xp, &p->cut);
}
// us, fitted to 2428 products of 65 - 2048 rows (standard deviation 8 %): fragments of the weights and the activations, the rounds of workgroups and the 128s of
// k in them, the sums' bytes, partial planes.
double fh_qmm_frag_us(const fh_qmatrix *q, int x_is_bf16, int m, int *parts) {
    FragPlan p;
    if (frag_plan(q, x_is_bf16, m, 0, &p) != FH_OK) return 1e30;
    if (parts) *parts = p.cut.parts;
    double step = 0.0; // 128 of k
    switch (q->type) {
    case FH_Q4_K: step = x_is_bf16 ? 1.47 : 2.4; break;
    case FH_Q5_K: step = x_is_bf16 ? 1.47 : 2.5; break;
    case FH_Q5_0: step = x_is_bf16 ? 1.96 : 2.9; break;
    case FH_Q6_K: step = 4.05; break; // (bf16 rows of the last two are not asked about)
    default: step = 3.05;
    }
    const double n = (double)q->n, k = (double)q->k, launches = (double)((q->n + p.rows - 1) / p.rows);
    return 6.0 + 0.62 * n * k / 1e6 + (x_is_bf16 ? 1.95 : 3.5) * m * k / 1e6 + launches * (8.0 * p.cut.rounds + step * p.cut.steps) + 0.36 * m * n / 1e6 + 0.5 * p.cut.sum;
}

static fh_status qmm_frag(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y, int half) {
    fh_device *dev = q->dev;
    FragPlan plan;
    FH_TRY(frag_plan(q, x_is_bf16, m, half, &plan));
    FragArgs &g = plan.g;
    const int k = (int)q->k, xp = x_is_bf16 ? 1 : 2, wp = q->type == FH_Q6_K ? 2 : 1, sc = fh_block_elems(q->type), ext = plan.ext, kf = g.kf, parts = plan.cut.parts;
    const int64_t rows = plan.rows, row_bytes = plan.row_bytes;
    if (half && (rows < q->n || parts > 1)) return FH_ERR_UNSUPPORTED; // all rows at once, k in one part
    // activations: rows up to a multiple of the largest tile (rows past m are multiplied and never stored)
    const int64_t mp = ((int64_t)m + 255) / 256 * 256, xplane = mp * kf * 32, wplane = rows * kf * 32;
    const size_t part_at = ((size_t)(xplane * xp + mp * 4) + 255) & ~(size_t)255, x_bytes = part_at + (parts > 1 ? (size_t)parts * m * g.n * 4 : 0);
    // The tile kernels need less, so what cannot be had is no error.  Their planes are there too: a captured product takes them where the
    // fragments do not fit.  (The growth of one of frag_x and frag_buf may give the other back.)
    (void)fh_dev_scratch_try(dev, &dev->act_buf, &dev->act_cap, fh_qmatmul_tile_planes(q, x_is_bf16, m));
    if (!fh_dev_scratch_try(dev, &dev->frag_x, &dev->frag_x_cap, x_bytes) ||
        !fh_dev_scratch_try(dev, &dev->frag_buf, &dev->frag_cap, (size_t)(rows * row_bytes)) || dev->frag_x_cap < x_bytes)
        return FH_ERR_UNSUPPORTED;
    dev->frag_used = true;
    uint8_t *xf = (uint8_t *)dev->frag_x;
    float *rs = (float *)(xf + xplane * xp);
    g.part = (float *)(xf + part_at);
    int runs = 1;
    while (runs < 8 && (m + 7) / 8 * runs < dev->compute_units && k / (runs * 2) >= 1024) runs *= 2;
    while (ext && ((k + runs - 1) / runs + 511) / 512 * 512 > 32768) runs *= 2; // the sums of a run: at most 32 KB of LDS
    const size_t lds = ext ? (size_t)(((k + runs - 1) / runs + 511) / 512 * 512 / 32) * 32 : 0; // 8 rows of f32 sums of a run
    if (x_is_bf16) {
        FH_TRY(fh_kernel_lds(dev, (const void *)k_frag_x<1>, lds));
        k_frag_x<1><<<dim3((unsigned)((m + 7) / 8), (unsigned)runs), 512, lds, dev->stream>>>(x, m, k, ext, xf, xplane, rs);
    } else {
        FH_TRY(fh_kernel_lds(dev, (const void *)k_frag_x<0>, lds));
        k_frag_x<0><<<dim3((unsigned)((m + 7) / 8), (unsigned)runs), 512, lds, dev->stream>>>(x, m, k, ext, xf, xplane, rs);
    }
    FH_HIP(hipGetLastError());
    uint8_t *wf = (uint8_t *)dev->frag_buf;
    float *d = (float *)(wf + wplane * wp);
    QView v = fh_view(q);
    for (int64_t n0 = 0; n0 < q->n; n0 += rows) {
        const int64_t n = q->n - n0 < rows ? q->n - n0 : rows;
        const dim3 grid((unsigned)((n + 15) / 16));
#define FRAG_W(T_) k_frag_w<T_><<<grid, 512, 0, dev->stream>>>(v, n0 / 16, ext, xp, wf, wplane, d, rows, half)
        switch (q->type) {
        case FH_Q4_0: FRAG_W(FH_Q4_0); break;
        case FH_Q8_0: FRAG_W(FH_Q8_0); break;
        case FH_Q5_0: FRAG_W(FH_Q5_0); break;
        case FH_Q4_K: FRAG_W(FH_Q4_K); break;
        case FH_Q5_K: FRAG_W(FH_Q5_K); break;
        case FH_Q6_K: FRAG_W(FH_Q6_K); break;
        default: FH_FAIL(FH_ERR_UNSUPPORTED, "unsupported type %u", q->type);
        }
#undef FRAG_W
        FH_HIP(hipGetLastError());
        g.w = wf, g.x = xf, g.w_plane = wplane, g.x_plane = xplane, g.d = d, g.n_pad = rows, g.rs = rs, g.y = y, g.n = (int)n, g.n0 = (int)n0;
        FH_TRY(frag_go(dev, g, sc, wp, xp, nullptr));
    }
    return FH_OK;
}

fh_status fh_launch_qmm_frag(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y) { return qmm_frag(q, x, x_is_bf16, m, y, 0); }

// In the epilogue of the product SwiGLU saves writing and reading 2 n floats a row and a launch: 2048 rows of a 28672 x 4096 matrix
// take 835 us and no 77 of a SwiGLU launch (7 % of a layer was writing and reading what one store now holds).
fh_status fh_qmm_frag_swiglu(const fh_qmatrix *q, const float *x, int m, float *y) {
    const int64_t opt = q->dev->opt_matmul_kernel;
    if (q->n % 64 == 0 && ((uintptr_t)x & 15) == 0 && (opt == 0 ? m > FH_SHORT_PROMPT && fh_qmm_reg_pays(q, 0, m) : opt >= 14 && opt <= 16 && fh_qmm_reg_supports(q)))
        return opt || fh_qmm_reg_swiglu_pays(q, m) ? fh_qmm_reg_swiglu(q, x, m, y) : FH_ERR_UNSUPPORTED;
    if (q->n % 64 || ((uintptr_t)x & 15) || m <= 16 || !(opt == 0 ? m > FH_SHORT_PROMPT && fh_qmm_frag_pays(q, 0, m) : opt == 13 && fh_qmm_frag_supports(q)))
        return FH_ERR_UNSUPPORTED;
    return qmm_frag(q, x, 0, m, y, (int)(q->n / 2));
}
