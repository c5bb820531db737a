// Quantized matmul for a few rows of f32 activations (2 .. 16), one launch: Y[m, n] = X[m, k] . deq(W)[n, k]^T.
//
// What bounds it: the phases of a launch, one after the other (about 2 us to its first bytes, 1 for the operands, 1.5 - 2.5 a tile of sixteen wavefronts, of
// which the vector ALU is busy most, 3 for the parts of k).  Two launches, one that writes operands and one that reads 17 KB of them for every 256 in each of its
// workgroups, are bound by those reads: a workgroup here reads KC 256s of the activations only.  (All of k a workgroup, so that nothing is parted, reads 256 KB for
// 4096 columns: 11.3 us for 4096 x 4096, 8.4 so.)
//
// A workgroup of sixteen wavefronts takes KC 256s of k and 16 / KC times TT row tiles.  Its wavefronts ask for the weights of their first two
// tiles (HBM) and turn the activations into f16 hi + lo operands in LDS while those are on their way; then each multiplies one 256 with TT
// tiles.  The 256s' sums are added through LDS.  k longer than that is in parts over workgroups: each writes its sums past the L2 and counts
// itself in, and the last of a group adds the parts in their order.  (Nobody waits for anybody: a workgroup that is not the last ends.)
//
// Codes are exact in f16 (RegW), products add up in f32, a power of two per row and 256 of k brings the activations into the f16 range - per 32 of k
// for the 5-bit formats, whose rows were a launch each of the kernel for one row and are normalised so there: groups small beside a row's
// largest value keep all their bits.
#include "fh_qmv_rows.h"
#include "fh_reg_weights.h"

typedef float floatx2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float rows_max(float top, float a, float b) { // (fmaxf would first make every operand canonical)
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(top), "v"(a), "v"(b));
    return r;
}
template <int CTRL>
__device__ __forceinline__ float rows_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// A 256's operands in LDS: [block][hi, lo][1 KB], the sums [hi, lo][1 KB] of Q4_K, the rows' factors (of each block).  Row r of lane group g
// lies in slot g 16 + (r + 4 g) % 16, so that four rows written together cover all banks.
template <int T>
struct RowsX {
    static constexpr bool OWN = T == FH_Q5_0 || T == FH_Q5_K, SUMS = T == FH_Q4_K; // OWN: a power of two per block
    static constexpr int SUM_AT = 16384, FAC_AT = SUM_AT + (SUMS ? 2048 : 0), BYTES = FAC_AT + (OWN ? 512 : 64);
};

// Four rows of a 256, one a row of 16 lanes: lane i has k 64 s + 4 i .. of its row in v[s].
template <int T>
__device__ __forceinline__ void rows_put(uint8_t *img, int row, int i, float4 (&v)[4]) {
    typedef RowsX<T> X;
    constexpr int NF = X::OWN ? 4 : 1;
    // The largest power of two: per 32 its inverse times a scale (2^-24 and more) has to be a normal number.  Per 256 any value may be normalised; at 100, Q4_K's
    // sums / 64 of activations of 1e-34 had lost so much that outputs were 3.8e-4 off (the kernels ahead of this one 1.4e-4, now 1.2e-7).
    constexpr int MOST = X::OWN ? 100 : 126;
    float sc[NF], top[NF];
    const bool first = (i & (X::OWN ? 7 : 15)) == 0; // of a factor's lanes
    auto quads = [&](float t) {                      // of eight lanes
        t = fmaxf(t, rows_dpp<0xB1>(t));
        t = fmaxf(t, rows_dpp<0x4E>(t));
        return fmaxf(t, rows_dpp<0x141>(t));
    };
    float *fac = (float *)(img + X::FAC_AT) + row + (X::OWN ? (i >> 3) * 16 : 0);
    if constexpr (X::OWN) {
#pragma unroll
        for (int s = 0; s < 4; s++) top[s] = quads(rows_max(rows_max(0.f, v[s].x, v[s].y), v[s].z, v[s].w));
    } else {
        float t = 0.f;
#pragma unroll
        for (int s = 0; s < 4; s++) t = rows_max(rows_max(t, v[s].x, v[s].y), v[s].z, v[s].w);
        t = quads(t);
        top[0] = fmaxf(t, rows_dpp<0x140>(t)); // of sixteen
    }
    float most = top[0];
#pragma unroll
    for (int s = 0; s < NF; s++) {
        int e = 141 - (int)((__float_as_uint(top[s]) >> 23) & 0xFFu); // 14 - floor(log2 top); zero / inf / nan clamp
        e = e > MOST ? MOST : (e < -100 ? -100 : e);
        sc[s] = __uint_as_float((uint32_t)(e + 127) << 23);
        if (first) fac[s * 32] = __uint_as_float((uint32_t)(127 - e) << 23);
        most = fmaxf(most, top[s]);
    }
    // An infinity is carried as +-2^15 with an infinite factor, so that the row's outputs are infinities of its weights' signs (its hi + lo would be a NaN).
    // One branch for all values, out of the way: with one a quad of them launches of 512 x 2048 took 5 % longer.
    if (__builtin_expect(__any(most == INFINITY), 0)) {
        auto carry = [&](float &u) { u = fabsf(u) == INFINITY ? copysignf(0x1p115f, u) : u; }; // (times 2^-100)
#pragma unroll
        for (int s = 0; s < 4; s++) carry(v[s].x), carry(v[s].y), carry(v[s].z), carry(v[s].w);
#pragma unroll
        for (int s = 0; s < NF; s++)
            if (first && top[s] == INFINITY) fac[s * 32] = INFINITY;
    }
    const int qi = i & 7, g = reg_order(T) == 2 ? qi & 3 : qi >> 1, half = reg_order(T) == 2 ? qi >> 2 : qi & 1;
    const int slot = (g * 16 + ((row + 4 * g) & 15)) * 16;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int b = 2 * s + (i >> 3);
        const float4 u = v[s];
        const float f = sc[X::OWN ? s : 0];
        const floatx2 p0 = {u.x * f, (reg_order(T) ? u.z : u.y) * f}, p1 = {(reg_order(T) ? u.y : u.z) * f, u.w * f};
        const half2v h[2] = {__builtin_convertvector(p0, half2v), __builtin_convertvector(p1, half2v)};
        const floatx2 r0 = {p0[0] - (float)h[0][0], p0[1] - (float)h[0][1]}, r1 = {p1[0] - (float)h[1][0], p1[1] - (float)h[1][1]};
        const half2v l[2] = {__builtin_convertvector(r0, half2v), __builtin_convertvector(r1, half2v)};
        uint2 w;
        __builtin_memcpy(&w, h, 8);
        *(uint2 *)(img + b * 2048 + slot + half * 8) = w;
        __builtin_memcpy(&w, l, 8);
        *(uint2 *)(img + b * 2048 + 1024 + slot + half * 8) = w;
        if (X::SUMS) { // of a lane's eight, / 64; the product with the offsets adds the lane groups'
            float t = (p0[0] + p0[1]) + (p1[0] + p1[1]);
            t = (t + rows_dpp<0xB1>(t)) * 0.015625f;
            const _Float16 th = (_Float16)t;
            if (half == 0) {
                *(_Float16 *)(img + X::SUM_AT + slot + b * 2) = th;
                *(_Float16 *)(img + X::SUM_AT + 1024 + slot + b * 2) = (_Float16)(t - (float)th);
            }
        }
    }
}

template <int T, int KC, int TT>
struct RowsTile {
    static constexpr int TILES = 16 / KC * TT, IMG = KC * RowsX<T>::BYTES, RED = 16 * TT * 272 * 4, LDS = IMG > RED ? IMG : RED;
};

template <int T, int KC, int TT, bool ONCE>
__global__ __launch_bounds__(1024) void k_qmv_rows(const uint8_t *data, const float *__restrict__ x, int n, int k, int m, int wtiles, int parts, float *__restrict__ part,
                                                   uint32_t *__restrict__ arrived, float *__restrict__ y) {
    const QView q{data, n, k, 0, 0, 0}; // (plain values: in registers when the kernel starts)
    constexpr bool OWN = RowsX<T>::OWN, SUMS = RowsX<T>::SUMS, PER32 = OWN || (!SUMS && T != FH_Q6_K), MINS = T == FH_Q5_K; // MINS: offsets block by block
    constexpr int REC = RegW<T>::REC, NW = RegW<T>::NW, PITCH = 272, TILES = RowsTile<T, KC, TT>::TILES;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ uint32_t s_last;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int chunks = (int)(q.k >> 8), group = (int)blockIdx.x / parts, p = (int)blockIdx.x - group * parts;
    const int kc = wave % KC, tg = wave / KC, mine = chunks - p * KC < KC ? chunks - p * KC : KC;
    const int c = kc < mine ? p * KC + kc : chunks - 1;
    float4 v[KC / 4][4];
#pragma unroll
    for (int r = 0; r < KC / 4; r++) {
        const int row = (tg * (KC / 4) + r) * 4 + g;
        const float *xr = x + (int64_t)(row < m ? row : m - 1) * q.k + c * 256 + j * 4;
#pragma unroll
        for (int s = 0; s < 4; s++) v[r][s] = *(const float4 *)(xr + 64 * s);
    }
    __builtin_amdgcn_sched_barrier(0); // the activations are asked for ahead of the weights
    RegW<T> w[TT > 1 ? 2 : 1];
    auto ask = [&](int s, int t) {
        int at = (group * (16 / KC) + tg) * TT + t;
        at = at < wtiles ? at : wtiles - 1;
        const uint8_t *rec = q.data + ((int64_t)at * chunks + c) * REC;
        w[s].template ask_a<ONCE>(rec, lane);
        w[s].template ask_b<ONCE>(rec, lane);
    };
    ask(0, 0);
    if (TT > 1) ask(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    uint8_t *img = smem + kc * RowsX<T>::BYTES;
#pragma unroll
    for (int r = 0; r < KC / 4; r++) rows_put<T>(img, (tg * (KC / 4) + r) * 4 + g, j, v[r]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (the weights stay on their way)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint8_t *at = img + (g * 16 + ((j + 4 * g) & 15)) * 16;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    const float *fac = (const float *)(img + RowsX<T>::FAC_AT) + 4 * g; // of the rows this lane's sums are of
    const floatx4 back = OWN ? zero : *(const floatx4 *)fac;
    uint32_t one;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(one));
    floatx4 sum[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) {
        RegW<T> &ww = w[t & 1];
        ww.begin();
        floatx4 a = zero, b = zero, out = zero;
#pragma unroll
        for (int sb = 0; sb < 8; sb++) {
            const half8 xh = *(const half8 *)(at + sb * 2048), xl = *(const half8 *)(at + sb * 2048 + 1024);
            half8 o[NW];
            ww.get(sb, one, o);
            a = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, o[0], PER32 ? zero : a, 0, 0, 0);
            if (PER32) {
                a = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, o[0], a, 0, 0, 0);
                const float d = MINS ? ww.scale(0) : ww.scale(sb);
                floatx4 f;
                if (OWN) f = *(const floatx4 *)(fac + 16 * sb);
                if constexpr (MINS) {
                    const half8 ov = ww.block_offset(sb);
                    b = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, ov, zero, 0, 0, 0);
                    b = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, ov, b, 0, 0, 0);
                    const float off = ww.offset() * 0.015625f;
#pragma unroll
                    for (int i = 0; i < 4; i++) out[i] = fmaf(fmaf(a[i], d, b[i] * off), f[i], out[i]);
                } else
#pragma unroll
                    for (int i = 0; i < 4; i++) out[i] = fmaf(a[i], OWN ? d * f[i] : d, out[i]);
            } else {
                b = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, o[0], b, 0, 0, 0);
                if (NW == 2) b = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, o[NW - 1], b, 0, 0, 0);
            }
        }
        if (!PER32) {
            const float d = ww.scale(0);
            if constexpr (SUMS) {
                const half8 sh = *(const half8 *)(at + RowsX<T>::SUM_AT), sl = *(const half8 *)(at + RowsX<T>::SUM_AT + 1024), ov = ww.offsets();
                floatx4 so = __builtin_amdgcn_mfma_f32_16x16x32_f16(sh, ov, zero, 0, 0, 0);
                so = __builtin_amdgcn_mfma_f32_16x16x32_f16(sl, ov, so, 0, 0, 0);
                const float off = ww.offset();
#pragma unroll
                for (int i = 0; i < 4; i++) out[i] = fmaf(a[i] + b[i], d, so[i] * off);
            } else
#pragma unroll
                for (int i = 0; i < 4; i++) out[i] = (a[i] + b[i]) * d;
        }
        sum[t] = OWN ? out : out * back;
        if (OWN) __builtin_amdgcn_sched_barrier(0); // (two tiles side by side would not fit the registers)
        if (t + 2 < TT) ask(t & 1, t + 2);
    }
    __syncthreads(); // the sums take the operands' place: [wavefront][tile][16 rows of 17]
    float *red = (float *)smem;
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[(wave * TT + t) * PITCH + (4 * g + i) * 17 + j] = sum[t][i];
    __syncthreads();
    auto total = [&](int e) { // element e of the workgroup's tiles: tile, row, weight row; the 256s in pairs
        const float *r = red + (e >> 8) / TT * (KC * TT * PITCH) + (e >> 8) % TT * PITCH + ((e >> 4) & 15) * 17 + (e & 15);
        float s[KC];
#pragma unroll
        for (int i = 0; i < KC; i++) s[i] = i < mine ? r[i * TT * PITCH] : 0.f;
#pragma unroll
        for (int h = 1; h < KC; h *= 2)
#pragma unroll
            for (int i = 0; i < KC; i += 2 * h) s[i] += s[i + h];
        return s[0];
    };
    auto store = [&](int e, float s) {
        const int64_t n = ((int64_t)group * TILES + (e >> 8)) * 16 + (e & 15);
        const int row = (e >> 4) & 15;
        if (row < m && n < q.n) y[row * q.n + n] = s;
    };
    if (parts == 1) {
        for (int e = tid; e < TILES * 256; e += 1024) store(e, total(e));
        return;
    }
    float *own = part + (int64_t)blockIdx.x * (TILES * 256);
    for (int e = tid; e < TILES * 256; e += 1024) __hip_atomic_store(own + e, total(e), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // written before this workgroup counts itself in
    __syncthreads();
    if (tid == 0) s_last = __hip_atomic_fetch_add(arrived + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_last != (uint32_t)parts - 1) return;
    if (tid == 0) __hip_atomic_store(arrived + group, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); // as it was found
    const float *all = part + (int64_t)group * parts * (TILES * 256);
    for (int e = tid; e < TILES * 256; e += 1024) {
        float s[4] = {0.f, 0.f, 0.f, 0.f}; // (four short sums: one of 14 parts is a tenth less exact)
        for (int i = 0; i < parts; i += 4)
#pragma unroll
            for (int h = 0; h < 4; h++)
                if (i + h < parts) s[h] += __hip_atomic_load(all + (i + h) * (TILES * 256) + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        store(e, (s[0] + s[1]) + (s[2] + s[3]));
    }
}

template <int T, int KC, int TT>
static fh_status rows_go(const fh_qmatrix *q, const float *x, int m, float *y) {
    typedef RowsTile<T, KC, TT> Tile;
    fh_device *dev = q->dev;
    const int chunks = (int)(q->k / 256), parts = (chunks + KC - 1) / KC, tiles = (int)((q->n + 15) / 16), groups = (tiles + Tile::TILES - 1) / Tile::TILES;
    float *part = nullptr;
    if (parts > 1) {
        if (!fh_dev_scratch_try(dev, (void **)&dev->ksplit_buf, &dev->ksplit_cap, (size_t)groups * parts * Tile::TILES * 1024)) return FH_ERR_UNSUPPORTED;
        part = dev->ksplit_buf;
    }
    const auto kern = fh_weights_once(q) ? k_qmv_rows<T, KC, TT, true> : k_qmv_rows<T, KC, TT, false>;
    FH_TRY(fh_kernel_lds(dev, (const void *)kern, (size_t)Tile::LDS));
    kern<<<dim3((unsigned)(groups * parts)), 1024, Tile::LDS, dev->stream>>>(q->data, x, (int)q->n, (int)q->k, m, tiles, parts, part, dev->arrived, y);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// Row tiles a wavefront and 256s a workgroup: the least of a model fitted to 16 matrices in each format (us: of a launch, of a round of workgroups, of a
// tile in it; of 128 - 11264 rows by 256 - 16384 columns the cut picked is 0.5 % slower than the best of the eight on average).  Up to four 256s there is nothing
// for eight to a workgroup to do (512 x 1024 in Q6_K 5.5 us, by eight 6.5); more than four parts of four 256s cost what the last of a group reads, a
// quarter of a microsecond a part and tile (1408 x 16384 in Q4_0, sixteen parts of two tiles 17.6 us, eight parts of eight 256s 11.1; 4096 x 11008 in Q4_K, eleven of
// three tiles 18.8, six of eight 256s 15.4).
struct RowsCut {
    int kc, tt;
    int64_t rounds;
    double us;
};
static RowsCut rows_cut(const fh_qmatrix *q) {
    const int64_t tiles = (q->n + 15) / 16, chunks = q->k / 256, cus = q->dev->compute_units;
    static const double of[6][2][3] = {{{0.9, 2.4, 2.56}, {-1.2, 5.3, 1.54}}, {{1.5, 1.2, 3.8}, {-1.0, 5.5, 2.56}}, {{0.6, 3.4, 2.76}, {-1.7, 5.5, 2.0}},
                                       {{1.1, 2.6, 2.52}, {-1.0, 5.75, 1.67}}, {{1.3, 1.8, 4.5}, {-0.8, 5.6, 3.2}}, {{1.2, 2.1, 3.8}, {-1.2, 4.7, 3.3}}};
    const int type = q->type == FH_Q4_0 ? 0 : q->type == FH_Q5_0 ? 1 : q->type == FH_Q8_0 ? 2 : q->type == FH_Q4_K ? 3 : q->type == FH_Q5_K ? 4 : 5;
    RowsCut best{4, 1, 0, 1e30};
    for (int kc = 4; kc <= (chunks > 4 ? 8 : 4); kc += 4)
        for (int tt = 1; tt <= 4; tt++) {
            const double *c = of[type][kc == 8];
            const int64_t parts = (chunks + kc - 1) / kc, groups = (tiles * kc + 16 * tt - 1) / (16 * tt), rounds = (groups * parts + cus - 1) / cus;
            const double sum = parts == 1 ? 0.0 : kc == 8 ? 2.3 : 1.0 + 0.07 * tt * tt * (double)(parts > 4 ? parts - 4 : 0);
            const double us = c[0] + sum + (double)rounds * (c[1] + c[2] * tt);
            if (us < best.us) best = RowsCut{kc, tt, rounds, us};
        }
    return best;
}

bool fh_qmv_rows_supports(const fh_qmatrix *q, const float *x, int m) {
    if (m < 2 || m > 16 || q->k % 256 || ((uintptr_t)x & 15) || q->n > 16 * FH_ARRIVED) return false;
    switch (q->type) {
    case FH_Q4_0: case FH_Q5_0: case FH_Q8_0: case FH_Q4_K: case FH_Q5_K: case FH_Q6_K: return true;
    }
    return false;
}
// Where one round of workgroups does it, against what took the call (k_qb_prep and k_qmv_direct, 5-bit formats k_qmm_reg, the tiles or a launch a row).  Replayed
// graphs of 70 random products a format, 100 - 30000 rows, 256 - 16384 columns, 5 - 16 activation rows, those that come here: Q4_0 0.83 of the time, Q8_0 0.83, Q4_K
// 0.85, Q6_K 0.86, Q5_0 0.49, Q5_K 0.52 (geometric means; 16 of 2048 x 8192 in Q4_K 11.0 / 9.4 us, 11008 x 4096 in Q8_0 18.2 / 13.5, 4096 x 11008 in Q6_K 24.4 / 19.5,
// 5 of 4096 x 4096 in Q5_K 13.8 / 9.9).  In two rounds 0.94 - 1.24, for a workgroup's own phases do not overlap the next one's.
// Left to the others, us there / here:
// - Q4_K from 3.5 row tiles a compute unit on and up to 4096 columns, where k_qmv_direct has four tiles a wavefront: 14336 x 4096 (224 workgroups here, one round)
//   14.7 / 14.8, 14336 x 3072 13.0 / 13.1, 16384 x 3072 13.1 / 14.5.  The line takes in some that would be quicker here (14336 x 2048 10.4 / 8.6, 20480 x 3072
//   20.2 / 15.5).  Q4_0 likewise of 2304 - 3072 columns: 14336 x 2560 11.6 / 12.3 (12288 x 2560 12.7 / 11.2, 16000 x 4096 15.0 / 13.9).
// - Q4_K of five to seven 256s and few rows: 512 x 1536 5.9 / 6.2.
// - More than 24576 rows of few columns: 10 of 30848 x 256 in Q6_K 7.9 / 9.1; of 256 columns in Q6_K and Q8_0 more than 16384: 5 of 22528 x 256 7.3 / 8.5 and
//   6.2 / 6.7 (16000 x 256 7.1 / 6.0 and 6.0 / 4.9).
// - 13 - 16 rows of Q5_K where a wavefront has four tiles, in parts: 16326 x 2304 17.0 / 20.2, 8192 x 5376 19.4 / 20.4 (4096 x 14336 24.2 / 23.3).
// - Up to 65536 weights of the 5-bit formats, although 64 x 1024 is 9.7 / 5.3: there k_qmm_reg's own line, five rows of 1024 columns, can be seen.
// - 2 - 4 rows, which are the single-row kernel's row variant (4096 x 4096, four rows 6.8 / 8.6); Q6_K, which has none, only from 3 rows on and with one tile a
//   wavefront (3 rows of 4096 x 4096 9.8 / 9.5, of 8192 x 3072 12.6 / 13.1).  The 5-bit formats, which have none either and take a launch a row, from 3 rows on where a
//   launch is more than its own start, that is beyond 2^20 weights: three rows of 4096 x 4096 in Q5_0 11.6 / 9.4 and in Q5_K 11.6 / 10.3, of 14336 x 4096 25.8 / 18.0 and
//   26.4 / 20.7, four rows 33.8 / 17.8 and 34.6 / 20.8, of 8192 x 3072 17.9 / 12.2 and 18.1 / 13.6 (512 x 2048 9.7 / 6.7, two rows 5.0 / 6.6).
//   Not where no single-row kernel shares their 256s out: those rows are f32 sums element by element, which take activations of any size as they are (here
//   those below 2^-86 lose bits: 1.4e-4 of 1e-34).
bool fh_qmv_rows_pays(const fh_qmatrix *q, const float *x, int m) {
    const bool five = q->type == FH_Q5_0 || q->type == FH_Q5_K;
    const int64_t kb = q->k / 256;
    const bool even = kb <= 16 || (kb <= 32 && kb % 2 == 0) || (kb <= 64 && kb % 4 == 0); // 1, 2 or 4 blocks a wavefront, 16 wavefronts
    if (!fh_qmv_rows_supports(q, x, m) || m < (q->type == FH_Q6_K || (five && even && q->n * q->k > 1 << 20) ? 3 : 5)) return false;
    const int64_t tiles = (q->n + 15) / 16, cus = q->dev->compute_units;
    if (five && q->n * q->k <= 65536) return false;
    if (q->type == FH_Q4_K && q->k > 1024 && q->k < 2048 && q->n <= 2816) return false;
    if (tiles * 2 >= 7 * cus && ((q->type == FH_Q4_K && q->k <= 4096) || (q->type == FH_Q4_0 && q->k > 2048 && q->k <= 3072))) return false;
    if (tiles > ((q->type == FH_Q6_K || q->type == FH_Q8_0) && q->k <= 256 ? 4 : 6) * cus) return false;
    const RowsCut cut = rows_cut(q);
    if (q->type == FH_Q5_K && m > 12 && cut.tt == 4 && q->k > 256 * cut.kc && q->k < 8192) return false;
    return cut.rounds == 1 && (m >= 5 || five || cut.tt == 1);
}

fh_status fh_launch_qmv_rows(const fh_qmatrix *q, const float *x, int m, float *y) {
    RowsCut cut = rows_cut(q);
    const int force = (int)q->dev->opt_matvec_tiles; // tests: tiles + 8 for eight 256s a workgroup
    if (force) cut.kc = force & 8 ? 8 : 4, cut.tt = force & 7;
    FH_REQUIRE(cut.tt >= 1 && cut.tt <= 4, "matvec_tiles = %d", force);
#define ROWS_TT(T_)                                                                                                \
    switch (cut.tt) {                                                                                              \
    case 1: return cut.kc == 4 ? rows_go<T_, 4, 1>(q, x, m, y) : rows_go<T_, 8, 1>(q, x, m, y);                    \
    case 2: return cut.kc == 4 ? rows_go<T_, 4, 2>(q, x, m, y) : rows_go<T_, 8, 2>(q, x, m, y);                    \
    case 3: return cut.kc == 4 ? rows_go<T_, 4, 3>(q, x, m, y) : rows_go<T_, 8, 3>(q, x, m, y);                    \
    default: return cut.kc == 4 ? rows_go<T_, 4, 4>(q, x, m, y) : rows_go<T_, 8, 4>(q, x, m, y);                   \
    }
    switch (q->type) {
    case FH_Q4_0: ROWS_TT(FH_Q4_0)
    case FH_Q5_0: ROWS_TT(FH_Q5_0)
    case FH_Q8_0: ROWS_TT(FH_Q8_0)
    case FH_Q4_K: ROWS_TT(FH_Q4_K)
    case FH_Q5_K: ROWS_TT(FH_Q5_K)
    case FH_Q6_K: ROWS_TT(FH_Q6_K)
    }
#undef ROWS_TT
    FH_FAIL(FH_ERR_UNSUPPORTED, "unsupported type %u", q->type);
}
