// Weights of the tiled layout decoded in a lane's registers into operands of the matrix cores (fh_qmm_reg.hip, fh_qmv_rows.hip).
#pragma once
#include "fh_blocks.h"
#include "fh_mv_lanes.h"

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

static constexpr __host__ __device__ bool reg_sums(int t) { return t == FH_Q4_K || t == FH_Q5_K; }
// order of the eight k of a lane: 0 ascending, 1 (0 2 1 3, 4 6 5 7), 2 the same of 4 g .. and 16 + 4 g ..
static constexpr __host__ __device__ int reg_order(int t) { return reg_sums(t) ? 1 : t == FH_Q4_0 || t == FH_Q5_0 ? 2 : 0; }

__device__ __forceinline__ half2v reg_h2(uint32_t u) {
    half2v h;
    __builtin_memcpy(&h, &u, 4);
    return h;
}
__device__ __forceinline__ half2v reg_splat(float v) { return half2v{(_Float16)v, (_Float16)v}; }

__device__ __forceinline__ half8 reg_cat(const half2v (&r)[4]) {
    half8 out;
#pragma unroll
    for (int i = 0; i < 4; i++) out[2 * i] = r[i][0], out[2 * i + 1] = r[i][1];
    return out;
}
// bytes B and B + 1 (or B twice) of w under the byte 0x64: the f16 pair 1024 + byte
template <int A, int B>
__device__ __forceinline__ half2v reg_bytes(uint32_t w) {
    return reg_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | A | B << 16));
}

// A row tile's 256 of k for v_mfma_f32_16x16x32_f16 as a wavefront holds them, lane = (lane group g, row j) of the layout: what is asked for with the first half
// (ask_a, for the next 256 while this one's second half is multiplied) and with the second (ask_b), begin() in between.
// get: block sb's operands, one = 0x64006400 in a vector register; scale: of block sb (formats with one per 32), of the 256.
template <int T>
struct RegW;

template <int T>
struct RegK { // Q4_K, Q5_K
    static constexpr int REC = T == FH_Q5_K ? 2816 : 2304, QA = T == FH_Q5_K ? 3 : 2, QB = 1, NW = 1;
    uint4 next, cod[2];
    uint2 next5, five;
    uint32_t dm, sc[2], mn[2];
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_a(const uint8_t *rec, int lane) {
        next = fh_ld_weights<ONCE, uint4>(rec + (lane & 15) * 16);
        cod[0] = fh_ld_weights<ONCE, uint4>(rec + 256 + lane * 16);
        if (T == FH_Q5_K) next5 = fh_ld_weights<ONCE, uint2>(rec + 2304 + lane * 8);
    }
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_b(const uint8_t *rec, int lane) { cod[1] = fh_ld_weights<ONCE, uint4>(rec + 1280 + lane * 16); }
    __device__ __forceinline__ void begin() {
        dm = next.x, five = next5;
        sc[0] = next.y & 0x3F3F3F3Fu, sc[1] = (next.w & 0x0F0F0F0Fu) | ((next.y >> 2) & 0x30303030u);
        mn[0] = next.z & 0x3F3F3F3Fu, mn[1] = ((next.w >> 4) & 0x0F0F0F0Fu) | ((next.z >> 2) & 0x30303030u);
    }
    // sc q, exact: a nibble (and its fifth bit) under the byte 0x64 is the f16 1024 + q, high nibbles 1024 + 16 q; one fma per two
    __device__ __forceinline__ void get(int sb, uint32_t one, half8 (&out)[1]) const {
        const int p = sb >> 2, u = (sb >> 1) & 1, hn = sb & 1;
        const uint4 c = cod[p];
        const uint32_t w[2] = {u ? c.z : c.x, u ? c.w : c.y}, h[2] = {five.x, five.y};
        const half2v s = reg_h2(__builtin_amdgcn_perm(0x64646464u, sc[p], 0x04000400u + (uint32_t)(sb & 3) * 0x00010001u)) - reg_splat(1024.f);
        const half2v a = hn ? s * reg_splat(0.0625f) : s, b = s * reg_splat(hn ? -64.f : -1024.f);
        half2v r[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t v = (((i & 1) ? w[i >> 1] >> 8 : w[i >> 1]) & (hn ? 0x00F000F0u : 0x000F000Fu)) | one;
            if (T == FH_Q5_K) {
                const int from = sb + 8 * (i & 1), to = hn ? 8 : 4;
                v |= (from > to ? h[i >> 1] >> (from - to) : h[i >> 1] << (to - from)) & (hn ? 0x01000100u : 0x00100010u);
            }
            r[i] = __builtin_elementwise_fma(reg_h2(v), a, b);
        }
        out[0] = reg_cat(r);
    }
    __device__ __forceinline__ float scale(int) const { return fh_h2f((uint16_t)(dm & 0xFFFFu)); }
    __device__ __forceinline__ float offset() const { return -64.f * fh_h2f((uint16_t)(dm >> 16)); }
    __device__ __forceinline__ half8 offsets() const {
        const half2v k = reg_splat(1024.f), r[4] = {reg_bytes<0, 1>(mn[0]) - k, reg_bytes<2, 3>(mn[0]) - k, reg_bytes<0, 1>(mn[1]) - k, reg_bytes<2, 3>(mn[1]) - k};
        return reg_cat(r);
    }
    __device__ __forceinline__ half8 block_offset(int sb) const { // m of block sb, for all of its k
        const half2v h = reg_h2(__builtin_amdgcn_perm(0x64646464u, mn[sb >> 2], 0x04000400u + (uint32_t)(sb & 3) * 0x00010001u)) - reg_splat(1024.f), r[4] = {h, h, h, h};
        return reg_cat(r);
    }
};
template <>
struct RegW<FH_Q4_K> : RegK<FH_Q4_K> {};
template <>
struct RegW<FH_Q5_K> : RegK<FH_Q5_K> {};

template <>
struct RegW<FH_Q6_K> {
    static constexpr int REC = 3360, QA = 4, QB = 1, NW = 2;
    uint4 lo[2], next_hi, hi;
    uint32_t next_sc, sc[4], at;
    uint16_t next_d, dv;
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_a(const uint8_t *rec, int lane) {
        lo[0] = fh_ld_weights<ONCE, uint4>(rec + lane * 16);
        next_hi = fh_ld_weights<ONCE, uint4>(rec + 2048 + lane * 16);
        next_sc = fh_ld_weights<ONCE, uint32_t>(rec + 3072 + lane * 4);
        next_d = fh_ld16(rec + 3328 + (lane & 15) * 2);
    }
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_b(const uint8_t *rec, int lane) { lo[1] = fh_ld_weights<ONCE, uint4>(rec + 1024 + lane * 16); }
    __device__ __forceinline__ void begin() {
        hi = next_hi, dv = next_d;
        const int lane = (int)threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < 4; q++) // groups 2 q, 2 q + 1 of both halves are in lane group q; bytes 0 and 2: the one of this lane's k
            sc[q] = ((uint32_t)__builtin_amdgcn_ds_bpermute((q * 16 + (lane & 15)) * 4, (int)next_sc) ^ 0x80808080u) >> ((lane >> 5) * 8);
    }
    // sc (q - 32) = its f16 rounding and what that leaves (-1, 0 or 1)
    __device__ __forceinline__ void get(int sb, uint32_t one, half8 (&out)[2]) const {
        const uint4 l4 = lo[sb >> 2];
        const uint32_t l = (sb & 3) == 0 ? l4.x : (sb & 3) == 1 ? l4.y : (sb & 3) == 2 ? l4.z : l4.w;
        const uint32_t h = (sb >> 1) == 0 ? hi.x : (sb >> 1) == 1 ? hi.y : (sb >> 1) == 2 ? hi.z : hi.w;
        const half2v s = (sb < 4 ? reg_bytes<0, 0>(sc[sb & 3]) : reg_bytes<2, 2>(sc[sb & 3])) - reg_splat(1152.f);
        half2v a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int from = q6k_hbit(sb, i);
            const uint32_t v = (((l >> (4 * i)) & 0x000F000Fu) | one) | ((from > 4 ? h >> (from - 4) : h << (4 - from)) & 0x00300030u);
            const half2v q = reg_h2(v) - reg_splat(1056.f);
            a[i] = q * s;
            b[i] = __builtin_elementwise_fma(q, s, -a[i]);
        }
        out[0] = reg_cat(a), out[1] = reg_cat(b);
    }
    __device__ __forceinline__ float scale(int) const { return fh_h2f(dv); }
};

template <>
struct RegW<FH_Q8_0> {
    static constexpr int REC = 4352, QA = 4, QB = 4, NW = 1;
    uint4 cod[2][2];
    uint32_t dd[2][2];
    template <bool ONCE = false>
    __device__ __forceinline__ void ask(int p, const uint8_t *rec, int lane) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            cod[p][r] = fh_ld_weights<ONCE, uint4>(rec + (2 * p + r) * 1088 + lane * 16);
            dd[p][r] = fh_ld_weights<ONCE, uint32_t>(rec + (2 * p + r) * 1088 + 1024 + (lane & 15) * 4);
        }
    }
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_a(const uint8_t *rec, int lane) { ask<ONCE>(0, rec, lane); }
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_b(const uint8_t *rec, int lane) { ask<ONCE>(1, rec, lane); }
    __device__ __forceinline__ void begin() {}
    __device__ __forceinline__ void get(int sb, uint32_t, half8 (&out)[1]) const {
        const uint4 c = cod[sb >> 2][(sb >> 1) & 1];
        const uint32_t x = (sb & 1 ? c.z : c.x) ^ 0x80808080u, y = (sb & 1 ? c.w : c.y) ^ 0x80808080u;
        const half2v k = reg_splat(1152.f), r[4] = {reg_bytes<0, 1>(x) - k, reg_bytes<2, 3>(x) - k, reg_bytes<0, 1>(y) - k, reg_bytes<2, 3>(y) - k};
        out[0] = reg_cat(r);
    }
    __device__ __forceinline__ float scale(int sb) const { return fh_h2f((uint16_t)(dd[sb >> 2][(sb >> 1) & 1] >> (16 * (sb & 1)))); }
};

template <int T>
struct Reg4 { // Q4_0, Q5_0
    static constexpr int HALF = T == FH_Q5_0 ? 1408 : 1152, REC = 2 * HALF, QA = T == FH_Q5_0 ? 3 : 2, QB = QA, NW = 1;
    uint4 cod[2];
    uint2 dd[2];
    uint32_t five[2];
    template <bool ONCE = false>
    __device__ __forceinline__ void ask(int p, const uint8_t *rec, int lane) {
        cod[p] = fh_ld_weights<ONCE, uint4>(rec + p * HALF + lane * 16);
        dd[p] = fh_ld_weights<ONCE, uint2>(rec + p * HALF + 1024 + (lane & 15) * 8);
        if (T == FH_Q5_0) five[p] = fh_ld_weights<ONCE, uint32_t>(rec + p * HALF + 1152 + lane * 4);
    }
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_a(const uint8_t *rec, int lane) { ask<ONCE>(0, rec, lane); }
    template <bool ONCE = false>
    __device__ __forceinline__ void ask_b(const uint8_t *rec, int lane) { ask<ONCE>(1, rec, lane); }
    __device__ __forceinline__ void begin() {}
    // q - 8 (q - 16) from 1024 + q, high nibbles from 1024 + 16 q
    __device__ __forceinline__ void get(int sb, uint32_t one, half8 (&out)[1]) const {
        const int p = sb >> 2, u = sb & 3;
        const uint4 c = cod[p];
        const uint32_t w = u == 0 ? c.x : u == 1 ? c.y : u == 2 ? c.z : c.w, lo5 = (five[p] >> (8 * u)) & 15u, hi5 = (five[p] >> (8 * u + 4)) & 15u;
        const float off = T == FH_Q5_0 ? 16.f : 8.f;
        half2v r[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t a = ((i ? w >> 8 : w) & 0x000F000Fu) | one, b = ((i ? w >> 8 : w) & 0x00F000F0u) | one;
            if (T == FH_Q5_0) { // bits i and i + 2 of four
                a |= (lo5 * (i ? 0x20008u : 0x40010u)) & 0x00100010u;
                b |= (hi5 * (i ? 0x200080u : 0x400100u)) & 0x01000100u;
            }
            r[i] = reg_h2(a) - reg_splat(1024.f + off);
            r[2 + i] = __builtin_elementwise_fma(reg_h2(b), reg_splat(0.0625f), reg_splat(-64.f - off));
        }
        out[0] = reg_cat(r);
    }
    __device__ __forceinline__ float scale(int sb) const { return fh_h2f((uint16_t)((sb & 2 ? dd[sb >> 2].y : dd[sb >> 2].x) >> (16 * (sb & 1)))); }
};
template <>
struct RegW<FH_Q4_0> : Reg4<FH_Q4_0> {};
template <>
struct RegW<FH_Q5_0> : Reg4<FH_Q5_0> {};

// Two row tiles' (32 rows') 256 of k for v_mfma_f32_32x32x16_f16.  The tiles' registers [A0 A1 A2 A3], [B0 B1 B2 B3] (16 lanes each, k in
// eights) become [A0 B0 A2 B2], [A1 B1 A3 B3] by one v_permlane16_swap each: operands of 32 rows with eights 0 and 2, 1 and 3 of a block.
// Slots are what a request brings: SL of them are a 256, two are held.  A lane's row is lane % 32, its header, scales and sums that row's.
__device__ __forceinline__ void reg_swap(uint32_t &a, uint32_t &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}
__device__ __forceinline__ void reg_swap(uint4 &a, uint4 &b) { reg_swap(a.x, b.x), reg_swap(a.y, b.y), reg_swap(a.z, b.z), reg_swap(a.w, b.w); }

template <int T>
struct WideW {
    static constexpr bool K4 = T == FH_Q4_K || T == FH_Q5_K, Q6 = T == FH_Q6_K, Q8 = T == FH_Q8_0;
    static constexpr int REC = T == FH_Q4_K ? 2304 : T == FH_Q5_K ? 2816 : Q6 ? 3360 : Q8 ? 4352 : T == FH_Q5_0 ? 2816 : 2304;
    static constexpr int SL = Q8 ? 4 : 2, NW = Q6 ? 2 : 1; // slots of a 256
    static constexpr int SLOT = K4 || Q6 ? 0 : REC / SL;   // bytes of one (formats with a scale per 32)
    // requests of a slot, and those of a 256's header
    static constexpr int QS = K4 || Q6 ? 2 : T == FH_Q5_0 ? 5 : 3, QH = T == FH_Q4_K ? 1 : T == FH_Q5_K ? 3 : Q6 ? 7 : 0;
    uint4 cod[2][2];
    uint32_t five[2][2]; // Q5_0: a slot's fifth bits
    uint2 dd[2];         // scales of a slot's blocks
    uint4 head, hi[2], next_hi[2];
    uint2 five_k[2], next5[2]; // Q5_K: a 256's
    uint32_t dm, sc[4], next_sc[4], mn[2];
    uint16_t next_d;

    // a, b: the tiles' records of a 256, own: the one of this lane's row
    __device__ __forceinline__ void ask(int s, const uint8_t *a, const uint8_t *b, int lane) {
        const int o = K4 ? 256 + s * 1024 : Q6 ? s * 1024 : s * SLOT;
        cod[s & 1][0] = *(const uint4 *)(a + o + lane * 16);
        cod[s & 1][1] = *(const uint4 *)(b + o + lane * 16);
        if (K4 || Q6) return;
        if (T == FH_Q5_0) {
            five[s & 1][0] = *(const uint32_t *)(a + o + 1152 + lane * 4);
            five[s & 1][1] = *(const uint32_t *)(b + o + 1152 + lane * 4);
        }
        const uint8_t *own = (lane & 16 ? b : a) + o + 1024;
        if (Q8) dd[s & 1].x = *(const uint32_t *)(own + (lane & 15) * 4);
        else dd[s & 1] = *(const uint2 *)(own + (lane & 15) * 8);
    }
    __device__ __forceinline__ void ask_head(const uint8_t *a, const uint8_t *b, int lane) {
        const uint8_t *own = lane & 16 ? b : a;
        if (K4) head = *(const uint4 *)(own + (lane & 15) * 16);
        if (T == FH_Q5_K) next5[0] = *(const uint2 *)(a + 2304 + lane * 8), next5[1] = *(const uint2 *)(b + 2304 + lane * 8);
        if (Q6) {
            next_hi[0] = *(const uint4 *)(a + 2048 + lane * 16), next_hi[1] = *(const uint4 *)(b + 2048 + lane * 16);
#pragma unroll
            for (int q = 0; q < 4; q++) next_sc[q] = *(const uint32_t *)(own + 3072 + (q * 16 + (lane & 15)) * 4);
            next_d = fh_ld16(own + 3328 + (lane & 15) * 2);
        }
    }
    __device__ __forceinline__ void begin_head(int lane) {
        if (K4) {
            dm = head.x;
            sc[0] = head.y & 0x3F3F3F3Fu, sc[1] = (head.w & 0x0F0F0F0Fu) | ((head.y >> 2) & 0x30303030u);
            mn[0] = head.z & 0x3F3F3F3Fu, mn[1] = ((head.w >> 4) & 0x0F0F0F0Fu) | ((head.z >> 2) & 0x30303030u);
        }
        if (T == FH_Q5_K) {
            five_k[0] = next5[0], five_k[1] = next5[1];
            reg_swap(five_k[0].x, five_k[1].x), reg_swap(five_k[0].y, five_k[1].y);
        }
        if (Q6) {
            hi[0] = next_hi[0], hi[1] = next_hi[1], dm = next_d;
            reg_swap(hi[0], hi[1]);
#pragma unroll
            for (int q = 0; q < 4; q++) sc[q] = (next_sc[q] ^ 0x80808080u) >> ((lane >> 5) * 8); // bytes 0 and 2: the one of this lane's k
        }
    }
    __device__ __forceinline__ void begin(int s) {
        reg_swap(cod[s & 1][0], cod[s & 1][1]);
        if (T == FH_Q5_0) reg_swap(five[s & 1][0], five[s & 1][1]);
    }
    // block e's operand h (eights 0 and 2, or 1 and 3)
    __device__ __forceinline__ void get(int e, int h, uint32_t one, half8 (&out)[NW]) const {
        const int s = e * SL / 8, u = e % (8 / SL);
        const uint4 c = cod[s & 1][h];
        half2v r[4], r2[4];
        if (K4) {
            const int hn = e & 1;
            const uint32_t w[2] = {e & 2 ? c.z : c.x, e & 2 ? c.w : c.y}, f[2] = {five_k[h].x, five_k[h].y};
            const half2v k = reg_h2(__builtin_amdgcn_perm(0x64646464u, sc[e >> 2], 0x04000400u + (uint32_t)(e & 3) * 0x00010001u)) - reg_splat(1024.f);
            const half2v a = hn ? k * reg_splat(0.0625f) : k, b = k * reg_splat(hn ? -64.f : -1024.f);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t v = (((i & 1) ? w[i >> 1] >> 8 : w[i >> 1]) & (hn ? 0x00F000F0u : 0x000F000Fu)) | one;
                if (T == FH_Q5_K) {
                    const int from = e + 8 * (i & 1), to = hn ? 8 : 4;
                    v |= (from > to ? f[i >> 1] >> (from - to) : f[i >> 1] << (to - from)) & (hn ? 0x01000100u : 0x00100010u);
                }
                r[i] = __builtin_elementwise_fma(reg_h2(v), a, b);
            }
        } else if (Q6) {
            const uint32_t l = (e & 3) == 0 ? c.x : (e & 3) == 1 ? c.y : (e & 3) == 2 ? c.z : c.w;
            const uint32_t t = (e >> 1) == 0 ? hi[h].x : (e >> 1) == 1 ? hi[h].y : (e >> 1) == 2 ? hi[h].z : hi[h].w;
            const half2v k = (e < 4 ? reg_bytes<0, 0>(sc[e & 3]) : reg_bytes<2, 2>(sc[e & 3])) - reg_splat(1152.f);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int from = q6k_hbit(e, i);
                const uint32_t v = (((l >> (4 * i)) & 0x000F000Fu) | one) | ((from > 4 ? t >> (from - 4) : t << (4 - from)) & 0x00300030u);
                const half2v q = reg_h2(v) - reg_splat(1056.f);
                r[i] = q * k;
                r2[i] = __builtin_elementwise_fma(q, k, -r[i]);
            }
            out[NW - 1] = reg_cat(r2);
        } else if (Q8) {
            const uint32_t x = (u ? c.z : c.x) ^ 0x80808080u, y = (u ? c.w : c.y) ^ 0x80808080u;
            const half2v k = reg_splat(1152.f);
            r[0] = reg_bytes<0, 1>(x) - k, r[1] = reg_bytes<2, 3>(x) - k, r[2] = reg_bytes<0, 1>(y) - k, r[3] = reg_bytes<2, 3>(y) - k;
        } else {
            const uint32_t w = u == 0 ? c.x : u == 1 ? c.y : u == 2 ? c.z : c.w, f = five[s & 1][h];
            const uint32_t lo5 = (f >> (8 * u)) & 15u, hi5 = (f >> (8 * u + 4)) & 15u;
            const float off = T == FH_Q5_0 ? 16.f : 8.f;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                uint32_t a = ((i ? w >> 8 : w) & 0x000F000Fu) | one, b = ((i ? w >> 8 : w) & 0x00F000F0u) | one;
                if (T == FH_Q5_0) {
                    a |= (lo5 * (i ? 0x20008u : 0x40010u)) & 0x00100010u;
                    b |= (hi5 * (i ? 0x200080u : 0x400100u)) & 0x01000100u;
                }
                r[i] = reg_h2(a) - reg_splat(1024.f + off);
                r[2 + i] = __builtin_elementwise_fma(reg_h2(b), reg_splat(0.0625f), reg_splat(-64.f - off));
            }
        }
        out[0] = reg_cat(r);
    }
    __device__ __forceinline__ float scale(int e) const { // of block e (formats with one per 32), of the 256
        if (K4 || Q6) return fh_h2f((uint16_t)(dm & 0xFFFFu));
        const int s = e * SL / 8, u = e % (8 / SL);
        return fh_h2f((uint16_t)((u & 2 ? dd[s & 1].y : dd[s & 1].x) >> (16 * (u & 1))));
    }
    __device__ __forceinline__ float offset() const { return -64.f * fh_h2f((uint16_t)(dm >> 16)); }
    __device__ __forceinline__ half8 offsets() const {
        const half2v k = reg_splat(1024.f), r[4] = {reg_bytes<0, 1>(mn[0]) - k, reg_bytes<2, 3>(mn[0]) - k, reg_bytes<0, 1>(mn[1]) - k, reg_bytes<2, 3>(mn[1]) - k};
        return reg_cat(r);
    }
};
