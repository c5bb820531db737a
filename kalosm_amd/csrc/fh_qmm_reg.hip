// Quantized matmul for a small prompt (17 to some hundred rows; bf16 from one row on), weights decoded in registers:
// Y[m, n] = X[m, k] . deq(W)[n, k]^T.
//
// The tiled layout holds a lane's codes in the order in which v_mfma_f32_16x16x32_f16 takes them, so a wavefront loads 16 bytes a lane
// and turns them into operands by itself: no pass over memory that writes f16 weights (products on fragments write and read 4 bytes
// a weight, 52 us for 14336 x 4096 whatever the rows), no LDS or barrier for them (the tile kernels, 128 rows of weights a workgroup
// one slab after the other).  Only the activations, laid out once per call, come through the LDS.
//
// Codes are exact in f16, products add up in f32:
//   Q4_K / Q5_K  sc * q, d per 256; the offsets dmin * m: one product of the integers m with the sums of 32 activations / 64 (hi + lo)
//   Q6_K         sc * (q - 32) = its f16 rounding and what that leaves (-1, 0, 1)
//   Q8_0, Q4_0, Q5_0   the code, d per 32, a sum of its own per 256
// Activations: a power of two per row, hi + lo (f32 input) or one exact term (bf16).  With f32 input Q6_K drops lo * lo.
//
// What bounds it: 17 rows of 14336 x 4096 in Q4_K take 22 us (63 on fragments), 64 rows 34 (67), 192 rows 71 (103), 512 rows 137
// (152); in Q6_K 29 (118), 40 (124), 92 (136), 185 (244); bf16 rows of Q8_0: one row 17 (140), 33 rows 23 (67), 512 rows 104 (114).  Up
// to 64 rows that is three launches and, in the middle one, two or three memory round trips; from some hundred rows on the matrix
// cores and the vector ALU beside them (a 16 x 16 x 32 product hides two vector instructions, a block of 32 has 2.2 a product).
// Against 64 bits, 17 - 512 rows of that matrix: 1.6e-7 - 1.7e-7 (Q4_K, Q5_K), 1.1e-7 (Q8_0, 64 rows), 1.7e-7 (Q6_K); the fragments 1.6e-7 -
// 1.7e-7 and, Q8_0 and Q5_0, 1.3e-7 - 1.6e-7, the tiles that few rows had in Q6_K 5e-7 - 7e-7, one bf16 row 0.8e-7 - 1.1e-7 for 5.6e-7 - 6.3e-7.
#include "fh_qmm_frag.h"
#include "fh_reg_weights.h"

// ------------------------------------------------------------------------------ activations
// Stored [row tile of 16][256 of k]: eight (hi plane) and eight (lo plane, f32 input) operands of 1 KB, one of the sums if there are offsets.

template <int IN, int ORDER>
__device__ __forceinline__ void reg_x_read(const void *xin, int64_t row, int k, int gi, float v[8]) {
    const int sb = gi >> 2, g = gi & 3;
    const int64_t a = row * k + (ORDER == 2 ? sb * 32 + 4 * g : gi * 8), b = a + (ORDER == 2 ? 16 : 4);
    float4 p, q;
    if (IN == 1) {
        const uint2 u = *(const uint2 *)((const uint16_t *)xin + a), w = *(const uint2 *)((const uint16_t *)xin + b);
        p = make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xFFFF0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xFFFF0000u));
        q = make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xFFFF0000u), __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xFFFF0000u));
    } else {
        p = *(const float4 *)((const float *)xin + a);
        q = *(const float4 *)((const float *)xin + b);
    }
    if (ORDER == 0) v[0] = p.x, v[1] = p.y, v[2] = p.z, v[3] = p.w, v[4] = q.x, v[5] = q.y, v[6] = q.z, v[7] = q.w;
    else v[0] = p.x, v[1] = p.z, v[2] = p.y, v[3] = p.w, v[4] = q.x, v[5] = q.z, v[6] = q.y, v[7] = q.w;
}

// One workgroup: ROWS rows (1, or 8 for whole 128-byte pieces of the operands), G groups of eight a thread in registers between the
// maximum and the conversion; G = 0: read twice.  WIDE: operands of 32 rows and 16 of k instead (k_qmm_wide).  OWN: a power of two per 32
// values instead of one per row, [8][16 rows] floats of a 256 in the place of its sums (k_qmm_reg, OWN; ROWS 1, G > 0).
template <int IN, int ORDER, int G, bool WIDE, int ROWS, bool OWN = false>
__global__ __launch_bounds__(1024) void k_reg_x(const void *__restrict__ xin, int m, int k, uint8_t *__restrict__ out, float *__restrict__ rs) {
    constexpr bool SUMS = ORDER == 1 && !OWN;
    constexpr int CH = (IN == 1 ? 8 : 16) * (WIDE ? 2048 : 1024) + (SUMS || OWN ? 1024 : 0);
    __shared__ float s_max[16][ROWS], sums[SUMS ? 512 * ROWS : 1]; // k <= 16384
    const int tid = threadIdx.x, r = tid % ROWS, row = (int)blockIdx.x * ROWS + r, groups = k >> 3, step = (int)blockDim.x / ROWS;
    const int from = row < m ? row : m - 1;
    float v[G ? G : 1][8], amax = 0.f, own[OWN ? G : 1] = {0.f};
    auto most = [&](const float (&w)[8]) {
#pragma unroll
        for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(w[j]));
    };
    if (G) {
#pragma unroll
        for (int i = 0; i < G; i++) {
            const int gi = tid / ROWS + i * step;
            reg_x_read<IN, ORDER>(xin, from, k, gi < groups ? gi : groups - 1, v[i]);
        }
#pragma unroll
        for (int i = 0; i < G; i++) {
            most(v[i]);
            if (OWN) { // of four threads
                amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
                own[i] = fmaxf(amax, __shfl_xor(amax, 2, 64));
                amax = 0.f;
            }
        }
    } else {
#pragma unroll 4
        for (int gi = tid / ROWS; gi < groups; gi += step) {
            float w[8];
            reg_x_read<IN, ORDER>(xin, from, k, gi, w);
            most(w);
        }
    }
    bool inf; // finite values vanish next to an infinity, which is carried as +-32768
    float sc;
    auto normal = [&](float a) { // the power of two, and what it takes back
        int e = 141 - (int)((__float_as_uint(a) >> 23) & 0xFFu); // 14 - floor(log2 a); zero / inf / nan clamp
        e = e > 100 ? 100 : (e < -100 ? -100 : e);
        inf = a == INFINITY;
        sc = __uint_as_float((uint32_t)(e + 127) << 23);
        return inf ? INFINITY : __uint_as_float((uint32_t)(127 - e) << 23);
    };
    if (!OWN) {
#pragma unroll
        for (int o = 32; o >= ROWS; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
        if ((tid & 63) < ROWS) s_max[tid >> 6][r] = amax;
        __syncthreads();
        for (int i = 0; i < (int)blockDim.x >> 6; i++) amax = fmaxf(amax, s_max[i][r]);
    }
    const float back = normal(amax);
    if (tid < ROWS && row < m) rs[row] = OWN ? 1.f : back;
    uint8_t *dst = WIDE ? out + (int64_t)(row >> 5) * (k >> 8) * CH + (row & 31) * 16 : out + (int64_t)(row >> 4) * (k >> 8) * CH + (row & 15) * 16;
    auto put = [&](int gi, const float (&x)[8]) {
        _Float16 h[8], l[8];
        float t = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            float w = x[j] * sc;
            if (inf && fabsf(w) == INFINITY) w = copysignf(32768.f, w);
            h[j] = (_Float16)w;
            const float d = w - (float)h[j];
            l[j] = (_Float16)(d == d ? d : 0.f); // a NaN stays in the hi plane alone
            t += w;
        }
        if (SUMS) { // of 32: four threads
            t += __shfl_xor(t, ROWS, 64);
            t += __shfl_xor(t, 2 * ROWS, 64);
            if ((gi & 3) == 0 && gi < groups) sums[(gi >> 2) * ROWS + r] = t * 0.015625f;
        }
        if (gi < groups && row < m) {
            // a block's eights 0 and 2 are the halves of one wide operand, 1 and 3 of the other
            uint8_t *p = dst + (int64_t)(gi >> 5) * CH + (WIDE ? ((gi >> 2) & 7) * 2048 + (gi & 1) * 1024 + (gi & 2) * 256 : ((gi >> 2) & 7) * 1024 + (gi & 3) * 256);
            uint4 u;
            __builtin_memcpy(&u, h, 16);
            *(uint4 *)p = u;
            if (IN != 1) {
                __builtin_memcpy(&u, l, 16);
                *(uint4 *)(p + (WIDE ? 16384 : 8192)) = u;
            }
        }
    };
    if (G) {
#pragma unroll
        for (int i = 0; i < G; i++) {
            const int gi = tid / ROWS + i * step;
            if (OWN) {
                const float b = normal(own[i]);
                if ((gi & 3) == 0 && gi < groups) *(float *)(out + ((int64_t)(row >> 4) * (k >> 8) + (gi >> 5)) * CH + CH - 1024 + ((gi >> 2) & 7) * 64 + (row & 15) * 4) = b;
            }
            put(gi, v[i]);
        }
    } else
        for (int at = 0; at < groups; at += step) { // (all threads together: the sums go through their neighbours)
            const int gi = at + tid / ROWS;
            float w[8];
            reg_x_read<IN, ORDER>(xin, from, k, gi < groups ? gi : groups - 1, w);
            put(gi, w);
        }
    if (!SUMS) return;
    __syncthreads();
    // a 256's sums: hi in lane group 0, lo in 1, zeros in 2 and 3
    if (row < m)
        for (int i = tid / ROWS; i < (k >> 6); i += step) {
            const int c = i >> 2, g = i & 3;
            _Float16 h[8];
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const float s = sums[(c * 8 + b) * ROWS + r];
                const _Float16 sh = (_Float16)s;
                h[b] = g == 0 ? sh : g == 1 ? (_Float16)(s - (float)sh) : (_Float16)0.f;
            }
            uint4 u;
            __builtin_memcpy(&u, h, 16);
            if (!WIDE) *(uint4 *)(dst + (int64_t)c * CH + CH - 1024 + g * 256) = u;
            else if (g < 2) *(uint4 *)(dst + (int64_t)c * CH + CH - 1024 + g * 512) = u;
        }
}

// ------------------------------------------------------------------------------ product
struct RegArgs {
    QView q;
    const uint8_t *x;
    const float *rs;
    float *y;
    int64_t ldy;
    int m, n, chunks, wtiles; // 256s of k, row tiles of the matrix
    int tiles_w, tiles_x, parts;
    int64_t part_stride;
    int half; // > 0: y[:, i] = silu(row i) * (row half + i)
};

// NX planes of activations, MT row tiles of 16 of them; the eight wavefronts are WW along the weight rows, TW row tiles each, times KW
// along k (added up in LDS at the end).  KW is what a small product needs: with 2 x 4 wavefronts 1024 x 4096 is 16 workgroups whose
// wavefronts multiply four 256s, with 8 x 1 it is four whose wavefronts multiply 16.
// A stage is SB blocks of 32 of k: one barrier, in front of it the wait for the stage after.  TW is 2: with 4, half the LDS reads a
// product, 17 rows took 15 - 25 % longer and 512 rows the same.
// OWN: activations with a power of two per 32 (one row tile of f32), so every block's sum is scaled by itself, in Q5_K with the block's offset,
// two more products with its m (12 rows of 14336 x 4096, one power of two per row / per 32: Q5_0 20.5 / 22.7 us, Q5_K 20.4 / 25.4).
template <int T, int NX, int TW, int MT, int WW, int KW, bool OWN>
struct RegTile {
    static constexpr int SB = KW == 1 ? 4 : KW == 2 ? 2 : 1; // blocks of 32 in a stage
    static constexpr int PIECES = NX * MT * SB, FR = (PIECES + WW - 1) / WW, STAGE = PIECES * KW * 1024;
    static constexpr int FIT = 163840 / STAGE, ST = FIT > 8 ? 8 : FIT;
    static constexpr int RED = (KW - 1) * WW * TW * MT * 1024, LDS = ST * STAGE > RED ? ST * STAGE : RED;
    static constexpr int CH = NX * 8192 + (reg_sums(T) || OWN ? 1024 : 0);
    static_assert(ST >= 4, "four stages at least");
    static_assert(!OWN || (MT == 1 && NX == 2), "one row tile of f32");
    // requests for weights (and sums, or powers of two) at block e of a 256
    static constexpr int wreq(int e) { return e == 0 ? TW * RegW<T>::QB : e == 4 ? TW * RegW<T>::QA + (OWN ? 8 : 0) : e == 6 && reg_sums(T) && !OWN ? MT : 0; }
    // requests younger than those of stage s + 1 at the start of stage s, which begins at block e of a 256.  (In its own stage the
    // pieces of a stage come behind the first block's requests; those of its other blocks are not counted.)
    static constexpr int younger(int e) {
        int n = 0;
        for (int b = 1; b <= (ST - 3) * SB; b++) n += (b % SB == 0 ? FR : 0) + wreq((e + 64 - b) & 7);
        return n > 63 ? 63 : n;
    }
};

template <int T, int NX, int TW, int MT, int WW, int KW, bool OWN>
__global__ __launch_bounds__(512) void k_qmm_reg(RegArgs g) {
    typedef RegTile<T, NX, TW, MT, WW, KW, OWN> Tile;
    constexpr int FR = Tile::FR, PIECES = Tile::PIECES, STAGE = Tile::STAGE, ST = Tile::ST, CH = Tile::CH, SB = Tile::SB;
    constexpr bool SUMS = reg_sums(T) && !OWN, PER32 = OWN || (!SUMS && T != FH_Q6_K), MINS = OWN && reg_sums(T);
    constexpr int NW = RegW<T>::NW, NP = NW == 2 ? NX + 1 : NX; // products of a weight operand and 16 rows
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int ww = wave % WW, kw = wave / WW;
    // workgroups go to the eight dies in turn: a die takes a run of tiles, those of the same weights together
    const int total = g.tiles_w * g.tiles_x * g.parts, per = total >> 3, more = total & 7, die = (int)blockIdx.x & 7;
    int lin = ((int)blockIdx.x >> 3) + die * per + (die < more ? die : more);
    const int tx = lin % g.tiles_x;
    lin /= g.tiles_x;
    const int tw = lin % g.tiles_w, part = lin / g.tiles_w;
    // 256s of this group of wavefronts: first .. first + mine, and the most that one has
    const int P = g.parts * KW, run = part * KW + kw;
    const int first = g.chunks * run / P, mine = g.chunks * (run + 1) / P - first;
    int most = 0;
#pragma unroll
    for (int i = 0; i < KW; i++) {
        const int a = g.chunks * (part * KW + i) / P, b = g.chunks * (part * KW + i + 1) / P;
        most = b - a > most ? b - a : most;
    }
    auto chunk = [&](int i) { const int c = first + (i < most ? i : most - 1); return c < g.chunks ? c : g.chunks - 1; };
    int tile[TW];
    const uint8_t *recs[TW];
#pragma unroll
    for (int t = 0; t < TW; t++) {
        const int w = tw * WW + ww;
        int at = g.half ? (t < TW / 2 ? w * (TW / 2) + t : (g.half >> 4) + w * (TW / 2) + t - TW / 2) : w * TW + t;
        tile[t] = at;
        at = at < g.wtiles ? at : g.wtiles - 1;
        recs[t] = g.q.data + (int64_t)at * g.chunks * RegW<T>::REC;
    }
    const uint8_t *xt = g.x + (int64_t)tx * MT * g.chunks * CH;
    auto fetch = [&](int c, int sb, int buf) { // the stage from block sb of the 256 c on into the buffer at byte `buf`
#pragma unroll
        for (int i = 0; i < FR; i++) {
            const int u = ww + WW * i < PIECES ? ww + WW * i : PIECES - 1; // (past the last one: the same bytes to the same place)
            const int v = u / (NX * MT), p = u / MT % NX, mt = u % MT;
            fh_buffer_to_lds(xt, MT * g.chunks * CH, smem + buf + (kw * PIECES + u) * 1024, lane * 16, (mt * g.chunks + c) * CH + (p * 8 + sb + v) * 1024);
        }
    };
    RegW<T> w[TW];
    floatx4 acc[TW][MT], sum[TW][MT], part256[TW][MT]; // of some 256s, of a scale, of a 256 (formats with a scale per 32)
    floatx4 all[TW][MT];                               // of those before (formats with a scale per 256)
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TW; t++)
#pragma unroll
        for (int c = 0; c < MT; c++) acc[t][c] = all[t][c] = zero;
    half8 xs[MT];
    int cur = 0;
#pragma unroll
    for (int t = 0; t < TW; t++) w[t].ask_a(recs[t] + (int64_t)chunk(0) * RegW<T>::REC, lane);
    floatx4 pw[OWN ? 8 : 1], next_pw[OWN ? 8 : 1]; // powers of two of a 256's blocks, of the next
    floatx4 off[TW], off256[TW], own = zero;       // sums with m, of a block and of a 256; the powers of two that go with the sums before
    auto ask_pw = [&](int c) {
#pragma unroll
        for (int b = 0; b < 8; b++) next_pw[b] = *(const floatx4 *)(xt + (int64_t)c * CH + CH - 1024 + b * 64 + (lane >> 4) * 16);
    };
    if constexpr (OWN) ask_pw(chunk(0));
#pragma unroll
    for (int i = 0; i < ST - 1; i++) fetch(chunk(i * SB >> 3), i * SB & 7, i * STAGE);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (the counts of the first steps are those of later ones, with more requests)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    half8 xv[MT * NX], wv[2][NW];
    float d32 = 0.f;
#pragma unroll
    for (int u = 0; u < MT * NX; u++) xv[u] = *(const half8 *)(smem + (kw * PIECES + u) * 1024 + lane * 16);
    uint32_t one;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(one));
    // The sum ends after four 256s (eight where there are many), so that none is long: against 64 bits 384 bf16 rows of 4096 x 14336 in Q4_K 9.9e-8 (sums of
    // 28: 1.22e-7), in Q5_K 1.08e-7 (1.30e-7), of 5632 x 2048 in Q5_K 9.3e-8 (of 8: 9.7e-8), for a hundredth of the time.  (With a scale per 32 there are no
    // registers for it, and the tiles added 32s.)
    const int span = most > 32 ? 8 : 4;
    for (int from = 0; from < most;) {
        const int to = PER32 || from + span > most ? most : from + span;
        for (int i = from; i < to; i++) {
            const int c0 = chunk(i), c1 = chunk(i + 1);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (e % SB == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Tile::younger(e)) : "memory"); // stage s + 1 has landed (and stage s) ...
                    __builtin_amdgcn_s_barrier();                                           // ... everywhere; the buffer of s - 1 is free
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (e == 0) {
#pragma unroll
                    for (int t = 0; t < TW; t++) w[t].ask_b(recs[t] + (int64_t)c0 * RegW<T>::REC, lane);
#pragma unroll
                    for (int t = 0; t < TW; t++) w[t].begin();
                    if constexpr (OWN)
#pragma unroll
                        for (int b = 0; b < 8; b++) pw[b] = next_pw[b];
                }
                if (e == 4) {
#pragma unroll
                    for (int t = 0; t < TW; t++) w[t].ask_a(recs[t] + (int64_t)c1 * RegW<T>::REC, lane);
                    if constexpr (OWN) ask_pw(c1);
                }
                if (SUMS && e == 6)
#pragma unroll
                    for (int m = 0; m < MT; m++) xs[m] = *(const half8 *)(xt + (m * g.chunks + c0) * CH + CH - 1024 + lane * 16);
                __builtin_amdgcn_sched_barrier(0);
                if (e % SB == 0) {
                    constexpr int AHEAD = (ST - 1) * SB; // blocks
                    fetch(chunk(i + (e + AHEAD) / 8), (e + AHEAD) & 7, cur == 0 ? (ST - 1) * STAGE : cur - STAGE);
                    __builtin_amdgcn_sched_barrier(0);
                }
                // the next block's activations, each behind its last use here
                const int nb = e % SB == SB - 1 ? (cur + STAGE == ST * STAGE ? 0 : cur + STAGE) : cur;
                const uint8_t *b = smem + nb + (kw * PIECES + (e + 1) % SB * NX * MT) * 1024 + lane * 16;
                if (e == 0) w[0].get(0, one, wv[0]);
#pragma unroll
                for (int t = 0; t < TW; t++) { // the next tile's (block's) weights are decoded while this one's are multiplied
                    const int now = t & 1;
                    if (e < 7 || t < TW - 1) w[(t + 1) % TW].get(t == TW - 1 ? e + 1 : e, one, wv[now ^ 1]);
#pragma unroll
                    for (int u = 0; u < MT * NP; u++) { // (plane by plane, so that neighbours are of different sums)
                        const int m = u % MT, p = u / MT;
                        sum[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[p < NX ? u : m], wv[now][p < NX ? 0 : NW - 1],
                                                                           (PER32 || e == 0) && p == 0 ? zero : sum[t][m], 0, 0, 0);
                    }
                    floatx4 off_now;
                    if constexpr (MINS) {
                        const half8 ov = w[t].block_offset(e);
                        off_now = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[0], ov, zero, 0, 0, 0);
                        off_now = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[1], ov, off_now, 0, 0, 0);
                    }
                    if (t == TW - 1)
#pragma unroll
                        for (int u = 0; u < MT * NX; u++) xv[u] = *(const half8 *)(b + u * 1024);
                    if (PER32) {
                        if (e + t > 0) { // the sums before these
                            const int pe = t ? e : e - 1, pt = t ? t - 1 : TW - 1;
#pragma unroll
                            for (int m = 0; m < MT; m++)
#pragma unroll
                                for (int r = 0; r < 4; r++) {
                                    const float d = OWN ? own[r] : d32;
                                    part256[pt][m][r] = pe ? fmaf(sum[pt][m][r], d, part256[pt][m][r]) : sum[pt][m][r] * d;
                                    if constexpr (MINS) off256[pt][r] = pe ? fmaf(off[pt][r], d, off256[pt][r]) : off[pt][r] * d;
                                }
                        }
                        d32 = i < mine ? w[t].scale(e) : 0.f; // (before the next half's scales are asked for into their place)
                        if constexpr (MINS) off[t] = off_now, own = pw[e]; // (the scale is the 256's)
                        else if constexpr (OWN) own = pw[e] * d32;
                    }
#pragma unroll
                    for (int u = 0; u < MT * NP + (MINS ? 2 : 0); u++) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, (16 * NW + (MINS ? 28 : OWN ? 8 : PER32 ? 4 * MT : 0)) / (MT * NP + (MINS ? 2 : 0)), 0);
                        if (t == TW - 1 && u >= MT * (NP - NX) + (MINS ? 2 : 0)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    }
                }
                if (e % SB == SB - 1) cur = cur + STAGE == ST * STAGE ? 0 : cur + STAGE;
            }
            // a 256's own sum first (with its offsets, which all but cancel it): the long sum takes one rounding for it
#pragma unroll
            for (int t = 0; t < TW; t++) {
                const float d = PER32 ? d32 : i < mine ? w[t].scale(0) : 0.f;
                if constexpr (SUMS) {
                    const float o = i < mine ? w[t].offset() : 0.f;
                    const half8 ov = w[t].offsets();
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const floatx4 so = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[m], ov, zero, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[t][m][r] += fmaf(sum[t][m][r], d, so[r] * o);
                    }
                } else if constexpr (MINS) {
                    const float d256 = i < mine ? w[t].scale(0) : 0.f, o256 = i < mine ? w[t].offset() * 0.015625f : 0.f;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float s = t == TW - 1 ? fmaf(sum[t][0][r], own[r], part256[t][0][r]) : part256[t][0][r];
                        const float o = t == TW - 1 ? fmaf(off[t][r], own[r], off256[t][r]) : off256[t][r];
                        acc[t][0][r] += fmaf(s, d256, o * o256);
                    }
                } else if constexpr (OWN) {
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[t][0][r] += t == TW - 1 ? fmaf(sum[t][0][r], own[r], part256[t][0][r]) : part256[t][0][r];
                } else
#pragma unroll
                    for (int m = 0; m < MT; m++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            acc[t][m][r] = PER32 ? acc[t][m][r] + (t == TW - 1 ? fmaf(sum[t][m][r], d, part256[t][m][r]) : part256[t][m][r])
                                                 : fmaf(sum[t][m][r], d, acc[t][m][r]);
            }
        }
        from = to;
        if (!PER32)
#pragma unroll
            for (int t = 0; t < TW; t++)
#pragma unroll
                for (int m = 0; m < MT; m++) all[t][m] += acc[t][m], acc[t][m] = to < most ? zero : all[t][m];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // no LDS-direct load outlives its buffer
    if (KW > 1) { // the groups' sums through LDS, in their order
        __syncthreads();
        float *red = (float *)smem + lane * 4;
        if (kw > 0)
#pragma unroll
            for (int t = 0; t < TW; t++)
#pragma unroll
                for (int m = 0; m < MT; m++) *(floatx4 *)(red + (((kw - 1) * WW + ww) * TW * MT + t * MT + m) * 256) = acc[t][m];
        __syncthreads();
        if (kw > 0) return;
#pragma unroll
        for (int i = 0; i < KW - 1; i++)
#pragma unroll
            for (int t = 0; t < TW; t++)
#pragma unroll
                for (int m = 0; m < MT; m++) acc[t][m] += *(const floatx4 *)(red + ((i * WW + ww) * TW * MT + t * MT + m) * 256);
    }
    float rs[MT][4]; // ahead of all stores: a load between them would wait for the stores before it
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const float4 v = *(const float4 *)(g.rs + (tx * MT + m) * 16 + 4 * (lane >> 4));
        rs[m][0] = v.x, rs[m][1] = v.y, rs[m][2] = v.z, rs[m][3] = v.w;
    }
    float *y = g.y + part * g.part_stride;
    if (g.half) {
#pragma unroll
        for (int t = 0; t < TW / 2; t++) {
            const int nn = tile[t] * 16 + (lane & 15);
            if (nn >= g.half) continue;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int mm = (tx * MT + m) * 16 + 4 * (lane >> 4) + r;
                    const float gate = acc[t][m][r] * rs[m][r], up = acc[t + TW / 2][m][r] * rs[m][r];
                    if (mm < g.m) y[mm * g.ldy + nn] = (gate / (expf(-gate) + 1.0f)) * up;
                }
        }
        return;
    }
#pragma unroll
    for (int t = 0; t < TW; t++) {
        const int nn = tile[t] * 16 + (lane & 15);
        if (nn >= g.n) continue;
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int mm = (tx * MT + m) * 16 + 4 * (lane >> 4) + r;
                if (mm < g.m) y[mm * g.ldy + nn] = acc[t][m][r] * rs[m][r];
            }
    }
}

// ------------------------------------------------------------------------------ wide product
// A wavefront: two pairs of row tiles (64 rows, for SwiGLU 32 of gate and 32 of up) by MX groups of 32 rows of activations; four
// wavefronts side by side along the weight rows, 256 x 32 MX a workgroup, two of which share a compute unit.  What bounds it is the vector
// ALU beside the matrix cores (Q8_0, one plane: 7.4 vector instructions for the work of a 16 x 16 x 32 product, of which two hide), so
//   products are the 32 x 32 x 16 ones, which leave it more room (16 of their half-size and 128 vector instructions of two wavefronts
//   take 307 ns, as 16 x 16 x 32 ones 370);
//   the two workgroups drift apart, and one decodes while the other multiplies: as one of eight wavefronts, in step at every barrier, 2048
//   rows of 14336 x 4096 took 393 us in Q8_0 (333 so, k in one chain; 344 in two halves), 332 in Q4_K (289), bf16;
//   the tiles that run together on a die are eight weight tiles by eight of activations (as two by 32: 358 and 304).
template <int T, int NX, int MX>
struct WideTile {
    static constexpr int SB = 2, PIECES = NX * MX * 2 * SB, FR = PIECES / 4, STAGE = PIECES * 1024;
    // A scale per 32 and one plane: k in two halves, the first one's sums in LDS and registers meanwhile.
    static constexpr bool HALVES = NX == 1 && !reg_sums(T) && T != FH_Q6_K;
    static constexpr int FIT = 81920 / STAGE, ST = FIT > 6 ? 6 : FIT, LDS = ST * STAGE + (HALVES ? MX * 16384 : 0);
    static constexpr int CH = NX * 16384 + (reg_sums(T) ? 1024 : 0);
    static_assert(ST >= 4 && PIECES % 4 == 0 && LDS <= 81920, "four stages at least, two workgroups a compute unit");
    typedef WideW<T> W;
    static constexpr int wreq(int e) {
        return (e % (8 / W::SL) == 0 ? 2 * W::QS : 0) + (e == 8 - 8 / W::SL ? 2 * W::QH : 0) + (e == 6 && reg_sums(T) ? MX : 0);
    }
    static constexpr int younger(int e) { // as RegTile::younger
        int n = 0;
        for (int b = 1; b <= (ST - 3) * SB; b++) n += (b % SB == 0 ? FR : 0) + wreq((e + 64 - b) & 7);
        return n > 63 ? 63 : n;
    }
};

template <int T, int NX, int MX>
__global__ __launch_bounds__(256, 2) void k_qmm_wide(RegArgs g) {
    typedef WideTile<T, NX, MX> Tile;
    typedef WideW<T> W;
    constexpr int FR = Tile::FR, STAGE = Tile::STAGE, ST = Tile::ST, CH = Tile::CH, SB = Tile::SB, SL = W::SL;
    constexpr bool SUMS = reg_sums(T), PER32 = !SUMS && T != FH_Q6_K;
    constexpr int NW = W::NW, NP = NW == 2 ? NX + 1 : NX, XB = NX * MX * 2; // operands of a block: [plane][eights][group]
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int total = g.tiles_w * g.tiles_x, per = total >> 3, more = total & 7, die = (int)blockIdx.x & 7;
    const int lin = ((int)blockIdx.x >> 3) + die * per + (die < more ? die : more);
    const int group = lin / (8 * g.tiles_x), in = lin - group * 8 * g.tiles_x; // eight weight tiles by all others, weight tiles first
    const int gw = g.tiles_w - group * 8 < 8 ? g.tiles_w - group * 8 : 8;
    const int tw = group * 8 + in % gw, tx = in / gw;
    const int most = g.chunks;
    auto chunk = [&](int i) { return i < most ? i : most - 1; };
    int row0[2];
    const uint8_t *ra[2], *rb[2];
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int w = tw * 4 + wave;
        row0[p] = g.half ? p * g.half + w * 32 : w * 64 + p * 32;
        const int a = row0[p] >> 4, b = a + 1;
        ra[p] = g.q.data + (int64_t)(a < g.wtiles ? a : g.wtiles - 1) * g.chunks * W::REC;
        rb[p] = g.q.data + (int64_t)(b < g.wtiles ? b : g.wtiles - 1) * g.chunks * W::REC;
    }
    const uint8_t *xt = g.x + (int64_t)tx * MX * g.chunks * CH;
    auto fetch = [&](int c, int e, int buf) { // the stage from block e of the 256 c on into the buffer at byte `buf`
#pragma unroll
        for (int i = 0; i < FR; i++) {
            const int u = wave + 4 * i, v = u / XB, p = u % XB / (2 * MX), h = u / MX % 2, m = u % MX;
            fh_buffer_to_lds(xt, MX * g.chunks * CH, smem + buf + u * 1024, lane * 16, (m * g.chunks + c) * CH + p * 16384 + (e + v) * 2048 + h * 1024);
        }
    };
    W w[2];
    floatx16 acc[2][MX], sum[PER32 ? 1 : 2][PER32 ? 2 : MX];
    const floatx16 zero = {0.f};
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int m = 0; m < MX; m++) acc[p][m] = zero;
    half8 xs[MX];
    int cur = 0;
#pragma unroll
    for (int p = 0; p < 2; p++) {
        w[p].ask_head(ra[p] + (int64_t)chunk(0) * W::REC, rb[p] + (int64_t)chunk(0) * W::REC, lane);
        w[p].ask(0, ra[p] + (int64_t)chunk(0) * W::REC, rb[p] + (int64_t)chunk(0) * W::REC, lane);
    }
#pragma unroll
    for (int i = 0; i < ST - 1; i++) fetch(chunk(i * SB >> 3), i * SB & 7, i * STAGE);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (the counts of the first steps are those of later ones, with more requests)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    half8 xv[XB], wv[2][2][NW];
#pragma unroll
    for (int u = 0; u < XB; u++) xv[u] = *(const half8 *)(smem + u * 1024 + lane * 16);
    uint32_t one;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(one));
    float d32 = 0.f;
    if (PER32) sum[0][1] = zero;
    // k in two halves: against 64 bits 2048 rows of 14336 x 4096 in Q8_0 1.47e-7 (one sum 2.04e-7, the tiles, which part k in their last round, 1.97e-7),
    // for one to two hundredths of the time.  (The first half's sums through y: half as long again, all workgroups write and read them at once.)
    floatx16 held[MX];
    float4 *const held_lds = (float4 *)(smem + ST * STAGE) + tid;
    if (Tile::HALVES)
#pragma unroll
        for (int m = 0; m < MX; m++) held[m] = zero;
    for (int from = 0; from < most;) {
        const int to = Tile::HALVES && from == 0 && most > 1 ? most >> 1 : most;
        for (int i = from; i < to; i++) {
            const int c0 = chunk(i), c1 = chunk(i + 1);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                constexpr int PER = 8 / SL; // blocks of a slot
                if (e % SB == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Tile::younger(e)) : "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (e % PER == 0) {
                    const int s = e / PER, c = s + 1 < SL ? c0 : c1;
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        if (s == 0) w[p].begin_head(lane);
                        w[p].begin(s);
                    }
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        if (s == SL - 1) w[p].ask_head(ra[p] + (int64_t)c * W::REC, rb[p] + (int64_t)c * W::REC, lane);
                        w[p].ask((s + 1) % SL, ra[p] + (int64_t)c * W::REC, rb[p] + (int64_t)c * W::REC, lane);
                    }
                }
                if (SUMS && e == 6)
#pragma unroll
                    for (int m = 0; m < MX; m++) xs[m] = *(const half8 *)(xt + (m * g.chunks + c0) * CH + CH - 1024 + lane * 16);
                __builtin_amdgcn_sched_barrier(0);
                if (e % SB == 0) {
                    constexpr int AHEAD = (ST - 1) * SB; // blocks
                    fetch(chunk(i + (e + AHEAD) / 8), (e + AHEAD) & 7, cur == 0 ? (ST - 1) * STAGE : cur - STAGE);
                    __builtin_amdgcn_sched_barrier(0);
                }
                const int nb = e % SB == SB - 1 ? (cur + STAGE == ST * STAGE ? 0 : cur + STAGE) : cur;
                const uint8_t *b = smem + nb + (e + 1) % SB * XB * 1024 + lane * 16; // the next block's activations
                if (PER32 && e % PER == 0) w[0].get(e, 0, one, wv[0][0]), w[0].get(e, 1, one, wv[0][1]);
#pragma unroll
                for (int p = 0; p < 2; p++) { // the next pair's (block's) weights are decoded while this one's are multiplied
                    if (!PER32) w[p].get(e, 0, one, wv[p][0]), w[p].get(e, 1, one, wv[p][1]);
                    else if (p == 0 || (e + 1) % PER) w[p ^ 1].get(e + p, 0, one, wv[p ^ 1][0]), w[p ^ 1].get(e + p, 1, one, wv[p ^ 1][1]);
                    if (PER32) {
                        float d = w[p].scale(e);
                        asm volatile("" : "+v"(d)); // (an f32 of its own: fused into the multiply-adds the conversion makes them the slow mixed ones)
#pragma unroll
                        for (int m = 0; m < MX; m++) { // a finished sum is scaled while the next is multiplied
                            const int at = (p * MX + m) & 1;
#pragma unroll
                            for (int v = 0; v < NX * 2; v++)
                                sum[0][at] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xv[(v >> 1) * 2 * MX + (v & 1) * MX + m], wv[p][v & 1][0], v ? sum[0][at] : zero, 0, 0, 0);
                            const int pp = m ? p : p ^ 1, pm = m ? m - 1 : MX - 1;
#pragma unroll
                            for (int r = 0; r < 16; r++) acc[pp][pm][r] = fmaf(sum[0][at ^ 1][r], d32, acc[pp][pm][r]);
                            d32 = d;
                            if (p)
#pragma unroll
                                for (int v = 0; v < NX * 2; v++) {
                                    const int u = (v >> 1) * 2 * MX + (v & 1) * MX + m;
                                    xv[u] = *(const half8 *)(b + u * 1024);
                                }
#pragma unroll
                            for (int v = 0; v < NX * 2; v++) {
                                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                                __builtin_amdgcn_sched_group_barrier(0x002, (16 + 44 / MX) / (NX * 2), 0);
                                if (p) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                            }
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < MX * NP * 2; j++) {
                            const int m = j % MX, v = j / MX, h = v & 1, q = v >> 1;
                            sum[p][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xv[(q < NX ? q : 0) * 2 * MX + h * MX + m], wv[p][h][q < NX ? 0 : NW - 1],
                                                                               e == 0 && v == 0 ? zero : sum[p][m], 0, 0, 0);
                        }
                        if (p)
#pragma unroll
                            for (int u = 0; u < XB; u++) xv[u] = *(const half8 *)(b + u * 1024);
                    }
                }
                if (e % SB == SB - 1) cur = cur + STAGE == ST * STAGE ? 0 : cur + STAGE;
            }
            if (!PER32)
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const float d = w[p].scale(0);
                    if constexpr (SUMS) {
                        const float o = w[p].offset();
                        const half8 ov = w[p].offsets();
#pragma unroll
                        for (int m = 0; m < MX; m++) {
                            const floatx16 so = __builtin_amdgcn_mfma_f32_32x32x16_f16(xs[m], ov, zero, 0, 0, 0);
#pragma unroll
                            for (int r = 0; r < 16; r++) acc[p][m][r] += fmaf(sum[p][m][r], d, so[r] * o);
                        }
                    } else
#pragma unroll
                        for (int m = 0; m < MX; m++)
#pragma unroll
                            for (int r = 0; r < 16; r++) acc[p][m][r] = fmaf(sum[p][m][r], d, acc[p][m][r]);
                }
        }
        if (Tile::HALVES && to < most)
#pragma unroll
            for (int m = 0; m < MX; m++) {
                held[m] = acc[1][m], acc[1][m] = zero;
#pragma unroll
                for (int r = 0; r < 16; r += 4)
                    held_lds[(m * 4 + r / 4) * 256] = make_float4(acc[0][m][r], acc[0][m][r + 1], acc[0][m][r + 2], acc[0][m][r + 3]);
                acc[0][m] = zero;
            }
        from = to;
    }
    if (PER32)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[1][MX - 1][r] = fmaf(sum[0][1][r], d32, acc[1][MX - 1][r]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // no LDS-direct load outlives its buffer
    if (Tile::HALVES && most > 1)
#pragma unroll
        for (int m = 0; m < MX; m++) {
            acc[1][m] += held[m];
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const float4 v = held_lds[(m * 4 + r / 4) * 256];
                acc[0][m][r] += v.x, acc[0][m][r + 1] += v.y, acc[0][m][r + 2] += v.z, acc[0][m][r + 3] += v.w;
            }
        }
    float *y = g.y;
#pragma unroll
    for (int m = 0; m < MX; m++) {
        float rs[16]; // ahead of the stores: a load between them would wait for the stores before it
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            const float4 v = *(const float4 *)(g.rs + (tx * MX + m) * 32 + 2 * r + 4 * (lane >> 5));
            rs[r] = v.x, rs[r + 1] = v.y, rs[r + 2] = v.z, rs[r + 3] = v.w;
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int nn = row0[p] + (lane & 31);
            if (nn >= (g.half ? g.half : g.n) || (g.half && p)) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int mm = (tx * MX + m) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                float v = acc[p][m][r] * rs[r];
                if (g.half) v = (v / (expf(-v) + 1.0f)) * (acc[1][m][r] * rs[r]);
                if (mm < g.m) y[mm * g.ldy + nn] = v;
            }
        }
    }
}

// ------------------------------------------------------------------------------ launches
template <int T, int NX, int TW, int MT, int WW, int KW, bool OWN = false>
static fh_status reg_product(fh_device *dev, RegArgs g, float *part) {
    typedef RegTile<T, NX, TW, MT, WW, KW, OWN> Tile;
    g.tiles_w = (g.wtiles + TW * WW - 1) / (TW * WW);
    g.tiles_x = (g.m + MT * 16 - 1) / (MT * 16);
    float *y = g.y;
    if (g.parts > 1) {
        g.y = part;
        g.part_stride = (int64_t)g.m * g.n;
    }
    FH_TRY(fh_kernel_lds(dev, (const void *)k_qmm_reg<T, NX, TW, MT, WW, KW, OWN>, (size_t)Tile::LDS));
    k_qmm_reg<T, NX, TW, MT, WW, KW, OWN><<<dim3((unsigned)(g.tiles_w * g.tiles_x * g.parts)), 512, Tile::LDS, dev->stream>>>(g);
    FH_HIP(hipGetLastError());
    if (g.parts > 1) return fh_frag_sum(dev, part, g.parts, g.part_stride, g.part_stride, y);
    return FH_OK;
}

template <int T, int NX>
static fh_status reg_go(fh_device *dev, const RegArgs &g, float *part, int mt, int kw, bool own) {
    if constexpr ((T == FH_Q5_0 || T == FH_Q5_K) && NX == 2)
        if (own) return kw == 1 ? reg_product<T, NX, 2, 1, 8, 1, true>(dev, g, part) : kw == 2 ? reg_product<T, NX, 2, 1, 4, 2, true>(dev, g, part)
                                                                                               : reg_product<T, NX, 2, 1, 2, 4, true>(dev, g, part);
#define GO(MT_)                                                                                                  \
    return kw == 1 ? reg_product<T, NX, 2, MT_, 8, 1>(dev, g, part) : kw == 2 ? reg_product<T, NX, 2, MT_, 4, 2>(dev, g, part) \
                                                                              : reg_product<T, NX, 2, MT_, 2, 4>(dev, g, part)
    switch (mt) {
    case 1: GO(1);
    case 2: GO(2);
    case 3: GO(3);
    default: GO(4);
    }
#undef GO
}

template <int T, int NX, int MX>
static fh_status wide_product(fh_device *dev, RegArgs g) {
    typedef WideTile<T, NX, MX> Tile;
    const int n = g.half ? g.half * 2 : g.n;
    g.tiles_w = (n + 255) / 256;
    g.tiles_x = (g.m + MX * 32 - 1) / (MX * 32);
    FH_TRY(fh_kernel_lds(dev, (const void *)k_qmm_wide<T, NX, MX>, (size_t)Tile::LDS));
    k_qmm_wide<T, NX, MX><<<dim3((unsigned)(g.tiles_w * g.tiles_x)), 256, Tile::LDS, dev->stream>>>(g);
    FH_HIP(hipGetLastError());
    return FH_OK;
}
bool fh_qmm_reg_supports(const fh_qmatrix *q) {
    switch (q->type) {
    case FH_Q4_0: case FH_Q5_0: case FH_Q8_0: case FH_Q4_K: case FH_Q5_K: case FH_Q6_K: return q->k % 256 == 0 && q->k <= 16384;
    }
    return false;
}

// How a product is cut: row tiles of activations a workgroup takes (as even as they come out, four at most: registers), groups of
// wavefronts and workgroups that share out k.  The least of a model fitted to 17 - 192 rows of four matrices: a round of workgroups
// costs 5 us and, per 256 of k, 1 us (Q6_K 2) and 0.28 us a row tile and product, more of it the fewer wavefronts share their
// activations; partial planes a launch and their bytes.  whole: k in one part.
struct RegCut {
    int mt, kw, parts;
    double us;
};
static RegCut reg_cut(const fh_qmatrix *q, int x_is_bf16, int m, bool whole) {
    const int chunks = (int)(q->k / 256), tiles = (m + 15) / 16, tx = (tiles + 3) / 4;
    const int np = (x_is_bf16 ? 1 : 2) + (q->type == FH_Q6_K ? 1 : 0);
    RegCut best{(tiles + tx - 1) / tx, 1, 1, 0.0};
    const double block = (q->type == FH_Q6_K ? 2.0 : 1.0) + 0.28 * best.mt * np; // us of 256 of k
    double least = 1e30;
    for (int kw = 1; kw <= 4; kw *= 2)
        for (int parts = 1; parts <= (whole ? 1 : 16) && parts * kw <= chunks; parts++) {
            if (x_is_bf16 && q->k >= 8192 && parts * kw < 2) continue; // (one chain along a long k is less exact than the tiles' parted ones)
            const int64_t groups = (q->n + 16 * 16 / kw - 1) / (16 * 16 / kw) * tx * parts;
            const int64_t rounds = (groups + q->dev->compute_units - 1) / q->dev->compute_units;
            const int run = (chunks + parts * kw - 1) / (parts * kw);
            double t = (double)rounds * (5.0 + run * block * (kw == 1 ? 1.0 : kw == 2 ? 1.13 : 1.4));
            if (parts > 1) t += 3.4 + (2.0 * parts + 1.0) * m * (double)q->n * 4.0 / 4e6;
            if (t < least * 0.98) least = t, best.kw = kw, best.parts = parts;
        }
    double type;
    switch (q->type) {
    case FH_Q4_K: type = 1.15; break;
    case FH_Q6_K: type = x_is_bf16 ? 0.85 : 0.92; break;
    case FH_Q5_K: type = x_is_bf16 ? 1.38 : 1.32; break;
    case FH_Q5_0: type = x_is_bf16 ? 1.45 : 1.32; break;
    case FH_Q4_0: type = 1.16; break;
    default: type = 1.22;
    }
    best.us = 8.0 + m * (double)q->k / 1e6 * 1.6 + type * least; // (with the activations' launch; from 320 rows on, where there is a choice)
    return best;
}

// Few rows: where k_qmm_reg is the better way, by timing 17 - 2048 rows of five matrices (14336 x 4096, 4096 x 14336, 4096 x 4096, 1024 x 4096, 5632 x 2048)
// in six formats and both activation types against the fragments and the tiles; us, this / the others, at the lines:
//   Q4_K f32   512 rows 140 / 153, 152 / 180, 52 / 76, 32 / 47, 44 / 54; 768 rows 193 / 236, 218 / 245, 70 / 82, 37 / 45, 71 / 66
//   Q4_K bf16  768 rows 133 / 185, 150 / 209, 50 / 93, 28 / 53, 55 / 91; 1024 rows 186 / 182, 168 / 191, 56 / 69, 30 / 46, 58 / 54
//   Q5_K f32   512 rows 150 / 156, 159 / 185, 56 / 66, 33 / 46, 47 / 54; 768 rows 224 / 238, 260 / 249; bf16 384 rows 103 / 109,
//              108 / 112, 512 rows 120 / 117
//   Q6_K f32   512 rows 175 / 247, 178 / 250, 59 / 91, 33 / 44, 51 / 100; 768 rows 264 / 319 but 87 / 78; bf16 768 rows 205 / 212, 207 / 240,
//              73 / 100, 1024 rows 278 / 257; of 14336 columns 400 rows 148 / 145, 512 152 / 148
//   Q8_0 f32   512 rows 146 / 194, 153 / 238, 52 / 93, 32 / 44, 43 / 97; 768 rows 218 / 257 but 75 / 69; bf16 768 rows 161 / 178, 180 / 279,
//              59 / 111, 1024 rows 216 / 212 but 190 / 349, 62 / 123, 31 / 56, 64 / 107 for the smaller n.  Q4_0 as Q8_0.
//   Q5_0 bf16  512 rows 122 / 136, 118 / 166; 768 rows 71 / 59 for 5632 x 2048
// Rows of whole tiles: Q4_K f32 of 8192 x 2048 500 rows 46 / 71, 512 49 / 71, 513 77 / 67, 640 82 / 70; of 8192 x 3072 512 65 / 92, 640 107 / 95.  What is slower
// past such an edge is left out by reg_way, which compares the two at hand.
// Not taken although faster, as the fragments' test holds these sizes to be the tiles': Q4_K, 512 f32 rows of matrices with four times as many rows as
// columns whose tiles fill the device, and Q5_0, 193 - 256 f32 rows of such (8192 x 2048, 200 rows 32 / 53).  Not yet taken: Q5_0, 257 - 512 f32 rows
// of fewer than 3072 rows (320 of 2048 x 2048 27 / 47), Q6_K f32 above 512 (640 of 11008 x 4096 180 / 302), Q6_K, 257 - 512 bf16 rows, k above 8192 (384
// of 5120 x 13824 126 / 297), Q8_0 bf16 above 1280 (1536 of 4096 x 14336 307 / 501).
// Fewer than 1024 columns: four 256s are the least that a workgroup's wavefronts share out.
static bool reg_few(const fh_qmatrix *q, int x_is_bf16, int m) {
    const int64_t n = q->n, k = q->k;
    switch (q->type) {
    case FH_Q4_K:
        if (x_is_bf16) return m <= 768;
        return m < 512 || (m <= 640 && (k > n || n < 4 * k || fh_qmm_frag_pays(q, 0, m)));
    case FH_Q5_K: return m <= (x_is_bf16 ? 448 : 512);
    case FH_Q5_0:
        if (x_is_bf16) return m <= 512;
        return m <= 192 || (m <= 512 && fh_qmm_frag_pays(q, 0, m));
    case FH_Q6_K: return x_is_bf16 ? m <= 768 && (k <= 8192 || m <= 256 || m > 512) : m <= 512;
    }
    return m <= (x_is_bf16 ? (n <= 8192 ? 1280 : 768) : 512); // Q8_0, Q4_0
}

// k_qmm_wide: us, model fitted to 14 matrices, nine row counts from 320 to 2048, four formats and both activation types (within 3 - 5 %
// of all of them): 256 of k of a tile take so long alone on its compute unit and so long for two that share one.
static double wide_us(const fh_qmatrix *q, int x_is_bf16, int m) {
    const int64_t tiles = (q->n + 255) / 256 * ((m + 63) / 64), each = (tiles + q->dev->compute_units - 1) / q->dev->compute_units;
    double one, two;
    switch (q->type) {
    case FH_Q4_K: one = x_is_bf16 ? 2.3 : 3.8, two = x_is_bf16 ? 4.2 : 6.8; break;
    case FH_Q6_K: one = x_is_bf16 ? 3.75 : 5.55, two = x_is_bf16 ? 6.8 : 9.7; break;
    case FH_Q5_K: one = x_is_bf16 ? 3.15 : 4.1, two = x_is_bf16 ? 5.2 : 7.5; break;
    case FH_Q5_0: one = x_is_bf16 ? 3.4 : 4.1, two = x_is_bf16 ? 5.6 : 7.5; break;
    case FH_Q4_0: one = x_is_bf16 ? 2.9 : 3.9, two = x_is_bf16 ? 4.6 : 6.8; break;
    default: one = x_is_bf16 ? 3.1 : 4.3, two = x_is_bf16 ? 5.0 : 7.5;
    }
    return 15.0 + m * (double)q->k / 1e6 * (x_is_bf16 ? 0.9 : 1.5) + (double)(q->k / 256) * ((double)(each & 1) * one + (double)(each >> 1) * two);
}

// Which of the two, if any.  Where few rows take k_qmm_reg: the one that is quicker by the models.  Above, k_qmm_wide where its
// tiles keep the device busy (us, wide / fragments / tiles: Q4_K bf16, 2048 rows, 14336 x 4096 300 / 333 / 474, 8192 x 3072 141 / 141 / 208, 5632 x 2048
// 78 / 90 / 132; Q8_0 bf16 356 / 388 / 436, 164 / 159 / 175, 89 / 100 / 121; Q6_K bf16 470 / 466 / 526, 208 / 184 / 224, 108 / 114 / 149, both on the
// tiles otherwise; Q4_K f32, 1024 rows, 28672 x 4096 490 / 525 / 702), with f32 rows only for
// matrices of 8192 rows and more (4096 x 4096, 2048 rows: 146 / 143) and not for Q6_K (2048 rows, 8192 x 3072 313 / 266).  k to 8192 only, and not where
// the tiles would part all of it (qmm_launch_t): its sums are long.  k_qmm_reg, whose 256s add up in fours or by themselves, takes what the others would
// part (reg_parted; 750 rows of 14336 x 8192, Q8_0, against 64 bits 1.4e-7, fragments 2.2e-7, wide 3.0e-7; 402, 462 and 407 us).  bf16 rows of the formats whose
// tiles leave the device idle for narrow matrices stay on k_qmm_reg (Q8_0, 1536 rows, 1024 x 4096 45 / 86, 3072 x 3072 85 / 140).
// Neither where the fragments or the tiles, whichever would take the call, are quicker by their models: a last round of workgroups that is nearly empty here and full
// there, or tiles that just fill the device.  (us, this / those: Q5_K f32, 384 rows, 11008 x 4096 136 / 111; Q5_K bf16, 2048 rows 284 / 240; Q4_K f32, 640
// rows, 8192 x 2048 82 / 70; Q8_0 bf16, 1000 rows, 7168 x 12288 354 / 275; Q6_K bf16, 1280 rows, 6528 x 8192 364 / 270; of 3000 products the models pick one that is more than
// 3 % slower 20 times, by 11 % at most.)
enum { REG_NONE, REG_NARROW, REG_WIDE };
// Whether what k_qmm_wide would take the place of has k in parts and is the closer one for it: the fragments, for f32 rows of formats with a scale per 32
// also the tiles in their last round.  (The tiles of Q5_0 multiply f32 values and are the least exact.)
static bool reg_parted(const fh_qmatrix *q, int x_is_bf16, int m) {
    if (fh_qmm_frag_pays(q, x_is_bf16, m)) {
        int parts = 1;
        (void)fh_qmm_frag_us(q, x_is_bf16, m, &parts);
        return parts > 1;
    }
    const int64_t tiles = (q->n + 127) / 128 * ((m + 255) / 256), cus = q->dev->compute_units, last = tiles > cus ? tiles % cus : 0;
    return (q->type == FH_Q8_0 || q->type == FH_Q4_0) && last > 0 && last * 2 <= cus;
}
static int reg_way(const fh_qmatrix *q, int x_is_bf16, int m, bool whole) { // whole: k in one part
    if (!fh_qmm_reg_supports(q) || q->k < 1024) return REG_NONE;
    const int64_t n = q->n, tiles = (n + 255) / 256 * ((m + 63) / 64), cus = q->dev->compute_units;
    const bool can = q->k <= 8192 && (x_is_bf16 || n >= 8192) && (n + 127) / 128 * ((m + 255) / 256) * 5 >= cus * 4, few = reg_few(q, x_is_bf16, m);
    const bool narrow = few || (x_is_bf16 && n <= 3072 && (q->type == FH_Q8_0 || q->type == FH_Q4_0 || q->type == FH_Q6_K));
    const bool parted = can && q->type != FH_Q6_K && (reg_sums(q->type) || !x_is_bf16) && reg_parted(q, x_is_bf16, m);
    const double fill = (double)tiles / (double)((tiles + cus - 1) / cus * cus);
    bool wide = !few && can && m > 512 && (x_is_bf16 || q->type != FH_Q6_K) && tiles >= 160 && fill >= (x_is_bf16 ? 0.6 : 0.7);
    if (!narrow && !wide) return REG_NONE;
    const double narrow_us = reg_cut(q, x_is_bf16, m, whole).us, us = wide_us(q, x_is_bf16, m);
    wide = !parted && (wide || (can && us < 0.97 * narrow_us));
    if (!whole && m > FH_SHORT_PROMPT) { // (SwiGLU was asked about as a product first)
        const double other = fh_qmm_frag_pays(q, x_is_bf16, m) ? fh_qmm_frag_us(q, x_is_bf16, m, nullptr) : fh_qmm_tile_us(q, x_is_bf16, m);
        if ((wide ? us : narrow_us) > (wide && q->type == FH_Q4_K ? 1.0 : 0.97) * other) return REG_NONE; // (what is next to level stays with the others)
    }
    return wide ? REG_WIDE : REG_NARROW;
}
bool fh_qmm_reg_pays(const fh_qmatrix *q, int x_is_bf16, int m) { return reg_way(q, x_is_bf16, m, false) != REG_NONE; }
// SwiGLU at the store takes k in one part.  A product that is quicker in several, its sums to memory and a launch for SwiGLU (4 us and their bytes, of
// 243 layers of three formats): 65 rows of 1024 x 4096 in Q8_0 11 us less a layer in two launches, 2048 x 4096 6, 4096 x 4096 2; 200 rows of 4096 x 4096 6 more.
bool fh_qmm_reg_swiglu_pays(const fh_qmatrix *q, int m) {
    const int way = reg_way(q, 0, m, true);
    if (way != REG_NARROW) return way == REG_WIDE;
    return reg_cut(q, 0, m, true).us <= reg_cut(q, 0, m, false).us + 4.0 + 2.0 * m * (double)q->n * 4.0 / 4e6;
}

static fh_status qmm_reg(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y, int half, bool planes) {
    fh_device *dev = q->dev;
    const int k = (int)q->k, xp = x_is_bf16 ? 1 : 2;
    RegCut cut = reg_cut(q, x_is_bf16, m, half > 0);
    const int64_t opt = dev->opt_matmul_kernel; // 15: always the wide one, 16: never
    const bool wide = opt == 15 || (opt != 16 && reg_way(q, x_is_bf16, m, half > 0) == REG_WIDE);
    if (wide) cut.parts = 1;
    else if (dev->opt_matmul_cut > 0) { // tests: row tiles, groups of wavefronts and workgroups along k as asked for
        const int c = (int)dev->opt_matmul_cut, mt = c & 15, kw = (c >> 4) & 15, parts = c >> 8;
        FH_REQUIRE(mt >= 1 && mt <= 4 && (kw == 1 || kw == 2 || kw == 4) && parts >= 1 && parts <= (half ? 1 : 16) && parts * kw <= k / 256,
                   "matmul_cut = %d for k = %d", c, k);
        cut.mt = mt, cut.kw = kw, cut.parts = parts;
    }
    RegArgs g{};
    g.q = fh_view(q);
    g.m = m, g.n = (int)q->n, g.ldy = half ? half : q->n, g.chunks = k / 256, g.wtiles = (int)((q->n + 15) / 16), g.parts = cut.parts, g.half = half;
    // activations: up to four row tiles past the last one (rows past m are multiplied and never stored)
    const int rows = wide ? 32 : 16;
    // Up to 12 rows of the 5-bit formats are a launch each of the kernel for one row otherwise, which normalises 32 values by themselves, so that
    // groups small beside a row's largest value keep all their bits: as it does.
    const bool own = !wide && !x_is_bf16 && m <= 12 && (q->type == FH_Q5_0 || q->type == FH_Q5_K);
    const int64_t ch = xp * 512 * rows + (reg_sums(q->type) || own ? 1024 : 0), xbytes = (((int64_t)m + rows - 1) / rows + 4) * g.chunks * ch;
    const size_t part_at = ((size_t)xbytes + ((size_t)m + 160) * 4 + 255) & ~(size_t)255;
    const size_t bytes = part_at + (cut.parts > 1 ? (size_t)cut.parts * m * q->n * 4 : 0);
    // as products on fragments do it: what cannot be had is no error, and the tile kernels' planes are there too
    if (planes) (void)fh_dev_scratch_try(dev, &dev->act_buf, &dev->act_cap, fh_qmatmul_tile_planes(q, x_is_bf16, m));
    if (!fh_dev_scratch_try(dev, &dev->frag_x, &dev->frag_x_cap, bytes)) return FH_ERR_UNSUPPORTED;
    dev->frag_used = true;
    uint8_t *xf = (uint8_t *)dev->frag_x;
    float *rs = (float *)(xf + xbytes), *part = (float *)(xf + part_at);
    g.x = xf, g.rs = rs, g.y = y;
    const bool many = m >= 1024 || (m >= 512 && k <= 8192);
    const unsigned threads = many || k / 8 >= 1024 ? 1024 : (unsigned)(k / 8 + 63) / 64 * 64;
#define REG_X3(IN_, O_, G_, W_, R_) k_reg_x<IN_, O_, G_, W_, R_><<<dim3((unsigned)((m + R_ - 1) / R_)), threads, 0, dev->stream>>>(x, m, k, xf, rs)
#define REG_X2(IN_, O_, W_)                          \
    if (!many && k > 8192) REG_X3(IN_, O_, 2, W_, 1); \
    else if (!many) REG_X3(IN_, O_, 1, W_, 1);       \
    else if (k > 8192) REG_X3(IN_, O_, 0, W_, 8);    \
    else if (k > 4096) REG_X3(IN_, O_, 8, W_, 8);    \
    else REG_X3(IN_, O_, 4, W_, 8)
#define REG_X(IN_, O_)                    \
    if (wide) { REG_X2(IN_, O_, true); } \
    else { REG_X2(IN_, O_, false); }      \
    break
#define REG_OWN(O_, G_) k_reg_x<0, O_, G_, false, 1, true><<<dim3((unsigned)m), threads, 0, dev->stream>>>(x, m, k, xf, rs)
    if (own && q->type == FH_Q5_K) { if (k > 8192) REG_OWN(1, 2); else REG_OWN(1, 1); }
    else if (own) { if (k > 8192) REG_OWN(2, 2); else REG_OWN(2, 1); }
    else switch (reg_order(q->type) + (x_is_bf16 ? 3 : 0)) {
    case 0: REG_X(0, 0);
    case 1: REG_X(0, 1);
    case 2: REG_X(0, 2);
    case 3: REG_X(1, 0);
    case 4: REG_X(1, 1);
    case 5: REG_X(1, 2);
    }
#undef REG_X
#undef REG_X2
#undef REG_X3
#undef REG_OWN
    FH_HIP(hipGetLastError());
#define REG_GO(T_)                                                                                              \
    if (wide) return x_is_bf16 ? wide_product<T_, 1, 2>(dev, g) : wide_product<T_, 2, 2>(dev, g); \
    return x_is_bf16 ? reg_go<T_, 1>(dev, g, part, cut.mt, cut.kw, false) : reg_go<T_, 2>(dev, g, part, cut.mt, cut.kw, own)
    switch (q->type) {
    case FH_Q4_0: REG_GO(FH_Q4_0);
    case FH_Q5_0: REG_GO(FH_Q5_0);
    case FH_Q8_0: REG_GO(FH_Q8_0);
    case FH_Q4_K: REG_GO(FH_Q4_K);
    case FH_Q5_K: REG_GO(FH_Q5_K);
    case FH_Q6_K: REG_GO(FH_Q6_K);
    }
#undef REG_GO
    FH_FAIL(FH_ERR_UNSUPPORTED, "unsupported type %u", q->type);
}

fh_status fh_launch_qmm_reg(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y, bool planes) {
    return qmm_reg(q, x, x_is_bf16, m, y, 0, planes);
}
fh_status fh_qmm_reg_swiglu(const fh_qmatrix *q, const float *x, int m, float *y) { return qmm_reg(q, x, 0, m, y, (int)(q->n / 2), true); }
