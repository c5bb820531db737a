// Prefill attention on the matrix cores: softmax(Q . K^T * scale [causal]) . V for many query rows, grouped-query
// heads, head_dim 64 or 128.
// Reference: fusor-ml/fusor/src/composite/flash_attention.rs:58-236 (semantics; causal mask as MaskKind::Causal
// with the queries aligned to the END of the keys), fusor-ml/core/src/row_program.rs:1210-1382 (the fused kernel).
//
// grid (q heads / HW, query blocks of 128, batch); 4 x HW wavefronts, each owning 32 query rows of one head: the HW
// (1, or 2 of f32 keys) heads of a workgroup share a KV head, so a KV tile is fetched and staged once for 128 x HW query rows.
// KV tiles of 64 keys go through LDS as f16, both as [key][d] rows written with 16-byte stores; the V^T operand
// of the second product is read with the transposing LDS load of gfx950 (ds_read_b64_tr_b16: the 16 lanes of a
// group supply 4 keys x 16 dims and receive, per lane, one dim of the 4 keys).  Two LDS buffers and one barrier per
// tile: tile t+1 is written to the other buffer right after the first product of tile t (its LDS writes and the
// request for tile t+2 then run under the softmax arithmetic).
// KS = 2 (prompts whose workgroups are no more than two rounds): eight wavefronts per query block, the second four take every
// other key tile with running statistics of their own, and the two halves are merged through LDS at the end - half the tile steps per
// workgroup.  (k_attn_prefill has it for f32 operands rounded to f16 only, attn_kernel = 2.)
// Of f16 keys and values k_attn_prefill has the launches of at most 128 keys; all others are k_attn_ahead's.
// QW = 2 (k_attn_ahead, shorter still: every workgroup of 64 query rows finds a compute unit of its own): two wavefronts per key
// group, so a SIMD runs one wavefront's chain of a step instead of two.
// What bounds the loop (measured per stage): the first product is matrix-core bound, the softmax vector-ALU bound
// (both wavefronts of a SIMD are in it together) and the second product bound by the transposing LDS loads, which
// run at half the rate of plain 16-byte loads.  So the softmax is kept to what a score needs (some 160 vector instructions for a wavefront's 2048; with
// address arithmetic for the requests, cleared accumulators and output rescaled in most tiles they were 310): a request is a buffer load from a
// descriptor that moves with the tile, and split operands, whose weights lose nothing by it, move their reference only where a maximum is 2^8
// above it.  The denominator is the sum of the f32 weights, whatever the products take them as: weights below 2^-25 of the largest are zero in f16, and
// many of them still count (16384 keys 2^25.5 below one: 3.5e-4 of the output).  (Added up in pairs from the rounded weights it saved 16 of the
// instructions and no time in k_attn_ahead: 2048 tokens 51.9 us against 52.0.)  Rows of V are 64 bytes apart in the banks (ap_v_row), so that the 16
// lanes of a transposing load cover them once.  Heads that share a workgroup (four wavefronts each) are half a step apart, one in the softmax while
// the other multiplies.  Replayed graphs of ten calls, causal, 32 / 8 heads of 128, before all that (and k_attn_ahead) and now, us: f16 1024 tokens
// 28.3 / 26.1, 2048 64 / 59, 3000 114 / 104, 4096 178 / 172, 8192 604 / 585 (940 TFLOP/s); f32 2048 146 / 143, 4096 390 / 358.
// Both products are computed TRANSPOSED with
// v_mfma_f32_32x32x16_f16 so that a lane always stands for ONE query (the accumulator column):
//   S^T (keys x queries) = K . Q^T      A = K rows, B = Q^T kept in registers for the whole kernel
//   O^T (d x queries)    = V^T . P^T    A = V^T rows, B = P^T = the S^T accumulator, exponentiated, as f16
// The online-softmax statistics (running max, running sum, rescale factor) are then per-lane scalars, and the row
// maximum is a reduction over the lane's own registers plus one exchange with lane + 32.  MFMA row i of the K
// operand reads key 16*(i/16) + 8*((i/4)%2) + 4*((i/8)%2) + i%4 of the tile: with that order the 16 accumulator
// registers of a lane are keys 8g .. 8g+7 and 16 + 8g .. 16 + 8g+7 (g = lane / 32), which is exactly the k-slot
// order of the B operand of the second product - P^T never leaves the registers.
// Inputs may be f32 or f16; operands are rounded to f16, all accumulation and the softmax are f32.
// SPLIT (f32 Q, K and V): every operand is the exact two-term f16 split hi + lo of the f32 value (2^-22 relative;
// the values must lie within the f16 range of +-65504) and both products are the three MFMAs
// hi.hi + lo.hi + hi.lo, so the result keeps f32 accuracy at three times the matrix-core work.  Its tiles fill the LDS: one workgroup a
// compute unit, for head_dim 128 and one head a workgroup one wavefront a SIMD, which nothing covers while it waits for an operand - so pairs are
// requested four ahead (head_dim 64, two wavefronts: two) and the wavefront may have all registers (32 / 8 heads, 2048 tokens, causal: 152 us,
// 190 with each pair requested in front of its products; 16 / 4 heads of 64, 3000 tokens 102 / 107).
#include "fh_blocks.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void ap_load8(const float *p, fh_half *o) {
    float x[8];
    __builtin_memcpy(x, p, 32);
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (fh_half)x[e];
}
__device__ __forceinline__ void ap_load8(const fh_half *p, fh_half *o) { __builtin_memcpy(o, p, 16); } // (any address)
// 16 bytes of a buffer, zeros past its end
__device__ __forceinline__ uint4 ap_buffer16(__amdgpu_buffer_rsrc_t b, int offset) {
    const auto u = __builtin_amdgcn_raw_buffer_load_b128(b, offset, 0, 0);
    return make_uint4(u[0], u[1], u[2], u[3]);
}
__device__ __forceinline__ float ap_swap32_max(float v) {
    const uint32_t u = __float_as_uint(v);
    auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float ap_swap32_sum(float v) {
    const uint32_t u = __float_as_uint(v);
    auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
__device__ __forceinline__ void ap_store4(float *p, float a, float b, float c, float d) {
    *(float4 *)p = make_float4(a, b, c, d);
}
__device__ __forceinline__ void ap_store4(fh_half *p, float a, float b, float c, float d) {
    const fh_half h[4] = {(fh_half)a, (fh_half)b, (fh_half)c, (fh_half)d};
    uint2 u;
    __builtin_memcpy(&u, h, 8);
    *(uint2 *)p = u;
}

__device__ __forceinline__ void ap_split8(const float *x, fh_half *hi, fh_half *lo) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        hi[e] = (fh_half)x[e];
        lo[e] = (fh_half)(x[e] - (float)hi[e]);
    }
}

typedef short short4v __attribute__((ext_vector_type(4)));
// Eight halfs of the V^T operand: keys k .. k+7 of the dim this lane stands for (two transposing loads of 4 keys).
__device__ __forceinline__ half8 ap_vt8(const fh_half *p, int row_stride) {
    const short4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(uintptr_t)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p);
    const short4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(uintptr_t)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)(p + 4 * row_stride));
    half8 r;
    __builtin_memcpy(&r, &a, 8);
    __builtin_memcpy((char *)&r + 8, &b, 8);
    return r;
}

// The second group of wavefronts hands its statistics and output over: [value][query wavefront][lane] floats in the tile buffers (the barrier
// that ended the last step has passed: nobody reads them any more).
template <int D, int QW>
__device__ __forceinline__ void ap_merge(float *sm, int wave, int lane, int kset, float &m_run, float &l_run, floatx16 (&acc)[D / 32]) {
    constexpr int NQ = 64 * QW, DT = D / 32;
    const int slot = (wave % QW) * 64 + lane;
    if (kset == 1) {
        sm[slot] = m_run;
        sm[NQ + slot] = l_run;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) sm[(2 + dt * 16 + r) * NQ + slot] = acc[dt][r];
    }
    __syncthreads();
    if (kset == 1) return;
    const float m1 = sm[slot], l1 = sm[NQ + slot];
    const float mm = fmaxf(m_run, m1), ref = mm == -INFINITY ? 0.f : mm;
    const float f0 = __builtin_amdgcn_exp2f(m_run - ref), f1 = __builtin_amdgcn_exp2f(m1 - ref);
    l_run = l_run * f0 + l1 * f1;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[dt][r] = acc[dt][r] * f0 + sm[(2 + dt * 16 + r) * NQ + slot] * f1;
}
// Halfs of a row of V in LDS: 64 bytes past a multiple of the banks, or 32 where that many more would leave a compute unit one workgroup of split operands
// instead of two (head_dim 64: 32 / 4 heads, causal, 3000 tokens 161 us with 64 bytes, 144 with 32).
template <int D, bool SPLIT, int HW>
constexpr int ap_v_row = SPLIT && D == 64 && HW == 1 ? D + 16 : D + 32;

// lane = query, register r of d-tile dt is d = 32 dt + 8 (r / 4) + 4 g + r % 4
template <int D, typename TQ>
__device__ __forceinline__ void ap_store(TQ *op, int g, float inv, const floatx16 (&acc)[D / 32]) {
#pragma unroll
    for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++)
            ap_store4(op + 32 * dt + 8 * r4 + 4 * g, acc[dt][4 * r4] * inv, acc[dt][4 * r4 + 1] * inv, acc[dt][4 * r4 + 2] * inv,
                      acc[dt][4 * r4 + 3] * inv);
}

// ANY: K and V through plain loads of 64-bit addresses instead of buffer requests, for views that those do not take (fh_attention_prefill_mfma).
template <typename TQ, typename TKV, int D, bool SPLIT = false, int HW = 1, int KS = 1, bool ANY = false>
__global__ __launch_bounds__(256 * HW * KS) __attribute__((amdgpu_waves_per_eu(SPLIT && D == 128 && HW == 1 ? 1 : 2, SPLIT && D == 128 && HW == 1 ? 1 : 2))) void k_attn_prefill(const TQ *__restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_st,
                                                       const TKV *__restrict__ k, const TKV *__restrict__ v,
                                                       int64_t kv_sb, int64_t kv_sh, int64_t kv_st, int hq, int hkv,
                                                       int sq, int skv, float scale, int causal, int by_row, TQ *__restrict__ out) {
    constexpr int BN = 64, KS_ = D + 8, VS = ap_v_row<D, SPLIT, HW>, DT = D / 32, KSTEPS = D / 16, CH = D / 8; // CH: 8-element chunks per row
    constexpr int NP = SPLIT ? 2 : 1; // operand planes: hi (, lo)
    static_assert(HW * KS <= 2 && !(SPLIT && KS == 2), "eight wavefronts at most; split operands leave no room for two tiles");
    constexpr int QB = 128, NTH = 256 * HW * KS, KBUF = NP * BN * KS_, VBUF = NP * BN * VS, TILE = KBUF + VBUF; // halfs per staged tile
    extern __shared__ __attribute__((aligned(16))) fh_half ap_lds[]; // [2 buffers][K planes | V planes]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31, g = lane >> 5;
    const int kset = KS == 2 ? wave / 4 : 0; // which key tiles of a step this wavefront multiplies
    // The wavefronts of two heads are half a step apart: those of one are in the first product and the softmax while those of the other are in the
    // second product.
    constexpr bool APART = HW == 2;
    const int head = wave >> 2;
    const int h = (int)blockIdx.x * HW + (HW == 2 ? wave >> 2 : 0), bi = blockIdx.z, kh = (int)blockIdx.x * HW / (hq / hkv);
    // causal: the last query blocks see the most keys; with the block index on the slow grid axis ALL heads of the
    // longest block are dispatched first and the short blocks fill the tail
    const int qb0 = (causal ? (int)(gridDim.y - 1 - blockIdx.y) : (int)blockIdx.y) * QB;
    const int qi = qb0 + (wave % 4) * 32 + li; // this lane's query row (KS = 2: both groups have the same rows)
    const int off = skv - sq;                  // causal: query i sees keys 0 .. i + off
    const TKV *kb = k + bi * kv_sb + kh * kv_sh, *vb = v + bi * kv_sb + kh * kv_sh;

    // Q^T operand, once: lane (query li, k-slots 8g .. 8g+7 of every 16-wide step of d)
    half8 qf[KSTEPS], ql[SPLIT ? KSTEPS : 1];
    {
        const TQ *qp = q + bi * q_sb + h * q_sh + (int64_t)(qi < sq ? qi : sq - 1) * q_st + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ks++) {
            fh_half t[8];
            if constexpr (SPLIT) {
                const float4 a = *(const float4 *)(qp + 16 * ks), b = *(const float4 *)(qp + 16 * ks + 4);
                const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
                fh_half lo[8];
                ap_split8(x, t, lo);
                __builtin_memcpy(&ql[ks], lo, 16);
            } else {
                ap_load8(qp + 16 * ks, t);
            }
            __builtin_memcpy(&qf[ks], t, 16);
        }
    }
    const int prow = 16 * (li >> 4) + 8 * ((li >> 2) & 1) + 4 * ((li >> 3) & 1) + (li & 3); // key read by MFMA row li
    const float sc2 = scale * 1.4426950408889634f;                                        // scores in the log2 domain
    float m_run = -INFINITY, l_run = 0.f;
    floatx16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[dt][r] = 0.f;

    int kend = skv;
    if (causal) {
        const int last = (qb0 + QB - 1 < sq ? qb0 + QB - 1 : sq - 1) + off + 1;
        kend = last < skv ? last : skv;
    }
    // A KV tile waits in registers (as f16; SPLIT: as the f32 values) from one tile before it is written to LDS.
    // Piece c = tid + NTH i of a tile: key c / CH, d chunk c % CH - consecutive threads along d, K and V alike.
    constexpr int NCH = KS * BN * CH / NTH;
    uint4 kreg[SPLIT ? 1 : NCH], vreg[SPLIT ? 1 : NCH];
    float4 kraw[SPLIT ? 2 * NCH : 1], vraw[SPLIT ? 2 * NCH : 1];
    // Requested through buffer descriptors that begin at the step's first key, so that a request is one instruction; rows past the last key
    // are zeros (their scores are masked and their P is 0).
    const int row_bytes = (int)(kv_st * sizeof(TKV));
    int piece[NCH]; // bytes from the step's first key
#pragma unroll
    for (int i = 0; i < NCH; i++) {
        const int c = tid + NTH * i;
        piece[i] = c / CH * row_bytes + 8 * (c % CH) * (int)sizeof(TKV); // key 0 .. KS * BN - 1: the KS tiles of a step
    }
    auto fetch = [&](int t0) {
        if constexpr (ANY) { // (rows past the last key repeat it)
#pragma unroll
            for (int i = 0; i < NCH; i++) {
                const int c = tid + NTH * i, row = t0 + c / CH;
                const int64_t at = (int64_t)(row < skv ? row : skv - 1) * kv_st + 8 * (c % CH);
                if constexpr (SPLIT) {
                    __builtin_memcpy(&kraw[2 * i], kb + at, 32);
                    __builtin_memcpy(&vraw[2 * i], vb + at, 32);
                } else {
                    fh_half t[16];
                    ap_load8(kb + at, t);
                    ap_load8(vb + at, t + 8);
                    __builtin_memcpy(&kreg[i], t, 16);
                    __builtin_memcpy(&vreg[i], t + 8, 16);
                }
            }
            return;
        }
        const int64_t end = (int64_t)(skv - t0 - 1) * row_bytes + D * (int)sizeof(TKV);
        const int bytes = end < 0x7FFFFFFF ? (int)end : 0x7FFFFFFF;
        const auto bk = __builtin_amdgcn_make_buffer_rsrc((void *)(kb + t0 * kv_st), 0, bytes, 0x00027000);
        const auto bv = __builtin_amdgcn_make_buffer_rsrc((void *)(vb + t0 * kv_st), 0, bytes, 0x00027000);
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            if constexpr (sizeof(TKV) == 2) {
                kreg[i] = ap_buffer16(bk, piece[i]);
                vreg[i] = ap_buffer16(bv, piece[i]);
            } else {
                const uint4 u[4] = {ap_buffer16(bk, piece[i]), ap_buffer16(bk, piece[i] + 16), ap_buffer16(bv, piece[i]), ap_buffer16(bv, piece[i] + 16)};
                if constexpr (SPLIT) {
                    __builtin_memcpy(&kraw[2 * i], &u[0], 32);
                    __builtin_memcpy(&vraw[2 * i], &u[2], 32);
                } else {
                    float x[16];
                    __builtin_memcpy(x, u, 64);
                    fh_half t[16];
#pragma unroll
                    for (int e = 0; e < 16; e++) t[e] = (fh_half)x[e];
                    __builtin_memcpy(&kreg[i], t, 16);
                    __builtin_memcpy(&vreg[i], t + 8, 16);
                }
            }
        }
    };
    auto stash = [&](int buf) { // K tile -> sK[key][d], V tile -> sV[key][d]
#pragma unroll
        for (int i = 0; i < NCH; i++) {
            const int c = tid + NTH * i, kk = c / CH, key = kk % BN, dc = c % CH;
            fh_half *sK = ap_lds + (buf * KS + kk / BN) * TILE, *sV = sK + KBUF;
            if constexpr (SPLIT) {
                const float kx[8] = {kraw[2 * i].x, kraw[2 * i].y, kraw[2 * i].z, kraw[2 * i].w,
                                     kraw[2 * i + 1].x, kraw[2 * i + 1].y, kraw[2 * i + 1].z, kraw[2 * i + 1].w};
                fh_half hi[8], lo[8];
                ap_split8(kx, hi, lo);
                uint4 uh, ul;
                __builtin_memcpy(&uh, hi, 16);
                __builtin_memcpy(&ul, lo, 16);
                *(uint4 *)(sK + key * KS_ + 8 * dc) = uh;
                *(uint4 *)(sK + BN * KS_ + key * KS_ + 8 * dc) = ul;
                const float vx[8] = {vraw[2 * i].x, vraw[2 * i].y, vraw[2 * i].z, vraw[2 * i].w,
                                     vraw[2 * i + 1].x, vraw[2 * i + 1].y, vraw[2 * i + 1].z, vraw[2 * i + 1].w};
                ap_split8(vx, hi, lo);
                __builtin_memcpy(&uh, hi, 16);
                __builtin_memcpy(&ul, lo, 16);
                *(uint4 *)(sV + key * VS + 8 * dc) = uh;
                *(uint4 *)(sV + BN * VS + key * VS + 8 * dc) = ul;
            } else {
                *(uint4 *)(sK + key * KS_ + 8 * dc) = kreg[i];
                *(uint4 *)(sV + key * VS + 8 * dc) = vreg[i];
            }
        }
    };
    // V^T operand addressing: the 16 lanes of a group supply keys (8 g + s / 4) and dims (16 * (group & 1) + 4 * (s % 4))
    // .. +3 and receive dim 16 * (group & 1) + s of keys 8 g .. 8 g + 3
    const int vt_off = (8 * g + ((lane & 15) >> 2)) * VS + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    // The Q loads must have landed before the loop: a wait for them inside the loop would also wait, every tile, for
    // the KV loads issued after them (the memory counter is in order).
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
        asm volatile("" ::"v"(qf[ks]));
        if constexpr (SPLIT) asm volatile("" ::"v"(ql[ks]));
    }
    const int lim = causal ? (qi + off < skv - 1 ? qi + off : skv - 1) : skv - 1; // this query's last visible key
    if (kend > 0) {
        fetch(0);
        stash(0);
        if (KS * BN < kend) fetch(KS * BN);
    }
    __syncthreads();
    auto bar = [&]() { // (requests for the tile after next stay on their way)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (APART && head == 1) bar();

    const float ninf = -INFINITY;
    for (int ts = 0, it = 0; ts < kend; ts += KS * BN, it++) { // a step: KS tiles, one per group of four wavefronts
        const int t0 = ts + kset * BN;
        // a group without a tile in the last step multiplies the staged rows (behind the last key: zeros) with every key masked
        const int lim_t = (KS == 1 || t0 < kend) ? lim : -1;
        const fh_half *sK = ap_lds + ((it & 1) * KS + kset) * TILE, *sV = sK + KBUF;
        // ---- S^T = K . Q^T for the two 32-key halves of the tile
        const floatx16 zero = {0.f};
        floatx16 st[2];
        if constexpr (!SPLIT) {
            // product i: key half i % 2, d step i / 2; the K operands are requested eight products ahead
            const fh_half *ap = sK + prow * KS_ + 8 * g;
            constexpr int NI = 2 * KSTEPS, AHEAD = 8;
            half8 ka[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) ka[i] = *(const half8 *)(ap + (i & 1) * 32 * KS_ + 16 * (i >> 1));
#pragma unroll
            for (int i = 0; i < NI; i++) {
                st[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[i % AHEAD], qf[i >> 1], i < 2 ? zero : st[i & 1], 0, 0, 0);
                if (i + AHEAD < NI) ka[i % AHEAD] = *(const half8 *)(ap + (i & 1) * 32 * KS_ + 16 * ((i + AHEAD) >> 1));
            }
            __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
            for (int i = 0; i < NI - AHEAD; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
        } else {
            // three products an operand pair (hi.hi, lo.hi, hi.lo); pairs are requested four (two) ahead
            const fh_half *ap = sK + prow * KS_ + 8 * g;
            constexpr int NI = 2 * KSTEPS, AHEAD = D == 128 ? 4 : 2;
            half8 kh_[AHEAD], kl_[AHEAD];
            auto read = [&](int i) {
                kh_[i % AHEAD] = *(const half8 *)(ap + (i & 1) * 32 * KS_ + 16 * (i >> 1));
                kl_[i % AHEAD] = *(const half8 *)(ap + (BN + (i & 1) * 32) * KS_ + 16 * (i >> 1));
            };
#pragma unroll
            for (int i = 0; i < AHEAD; i++) read(i);
#pragma unroll
            for (int i = 0; i < NI; i++) {
                st[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh_[i % AHEAD], qf[i >> 1], i < 2 ? zero : st[i & 1], 0, 0, 0);
                st[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl_[i % AHEAD], qf[i >> 1], st[i & 1], 0, 0, 0);
                st[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh_[i % AHEAD], ql[i >> 1], st[i & 1], 0, 0, 0);
                if (i + AHEAD < NI) read(i + AHEAD);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * AHEAD, 0);
#pragma unroll
            for (int i = 0; i < NI - AHEAD; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 3 * AHEAD, 0);
        }
        // ---- tile t+1 goes into the other buffer (last read before the barrier that ended the previous tile) and
        // tile t+2 is requested: the LDS writes and the loads run under the softmax arithmetic
        // (the scheduler may not mix the stages: the operands prefetched for one product and the tile in flight would
        // otherwise be live together with the scores)
        __builtin_amdgcn_sched_barrier(0);
        auto next = [&]() {
            if (ts + KS * BN < kend) stash((it + 1) & 1);
            if (ts + 2 * KS * BN < kend) fetch(ts + 2 * KS * BN);
        };
        if (!APART || head == 1) next(); // (both heads in the same half step: neither has a wavefront in the other buffer then)
        __builtin_amdgcn_sched_barrier(0);
        // ---- mask, running max: register r of half kt is key t0 + 32 kt + 16 (r / 8) + 8 g + r % 8
        // Only a tile that reaches past some query's last visible key pays for the compares (one branch for the
        // wavefront); the select works in place, so the common path has no register copies at the join.
        if (__any(t0 + BN - 1 > lim_t)) {
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = t0 + 32 * kt + 16 * (r >> 3) + 8 * g + (r & 7);
                    asm volatile("v_cmp_le_i32 vcc, %1, %2\n\tv_cndmask_b32 %0, %3, %0, vcc"
                                 : "+v"(st[kt][r])
                                 : "v"(key), "v"(lim_t), "v"(ninf)
                                 : "vcc");
                }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int r = 0; r < 16; r++) mx = fmaxf(mx, st[kt][r]);
        // the scale (> 0) is applied inside the exponent: p = 2^(s * sc2 - m), one multiply-add per score
        mx = ap_swap32_max(mx) * sc2;
        // The reference of the exponents.  Split operands: it moves only where a maximum is more than 2^8 above it, so that the output is rescaled
        // in the first tiles and then hardly ever.  (Weights rounded to f16: where one key has most of the weight that is 1, exact; against 64 bits
        // 2048 tokens with scores of four times the usual spread 2.13e-4, with a reference of its own 2.25e-4.)
        const bool moves = mx > m_run + (SPLIT ? 8.f : 0.f), move = __any(moves); // (each row's by its own scores, so that its bits do not depend on its neighbours)
        float alpha = 1.f;
        if (move) {
            const float m_new = moves ? mx : m_run;
            alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new); // (nothing visible yet: only queries past the end)
            m_run = m_new;
        }
        const float m_sub = m_run == -INFINITY ? 0.f : -m_run; // dead rows: 2^(-inf - 0) = 0
        float ps = 0.f;
        half8 pb[2][2], pl[SPLIT ? 2 : 1][2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++) {
                fh_half t[8], tl[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(st[kt][8 * s2 + e], sc2, m_sub)); // arguments <= 0, split operands <= 8 (weights up to 2^8)
                    ps += p;
                    t[e] = (fh_half)p;
                    if constexpr (SPLIT) tl[e] = (fh_half)(p - (float)t[e]);
                }
                __builtin_memcpy(&pb[kt][s2], t, 16);
                if constexpr (SPLIT) __builtin_memcpy(&pl[kt][s2], tl, 16);
            }
        l_run = l_run * alpha + (SPLIT ? ps : ap_swap32_sum(ps)); // (split operands: of this lane's keys)
        // ---- O^T = O^T * alpha + V^T . P^T
        __builtin_amdgcn_sched_barrier(0);
        if (APART) {
            bar();
            if (head == 0) next();
            __builtin_amdgcn_sched_barrier(0);
        }
        if (move) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[dt][r] *= alpha;
        }
        if constexpr (!SPLIT) {
            // product j: d tile j % DT, key step j / DT (= 2 kt + s2): consecutive products go to different
            // accumulators; the V^T operand is requested eight products ahead
            const fh_half *vp = sV + vt_off;
            constexpr int NJ = 4 * DT, AHEAD = 8;
            half8 va[AHEAD];
#pragma unroll
            for (int j = 0; j < AHEAD; j++) va[j] = ap_vt8(vp + 32 * (j % DT) + 16 * (j / DT) * VS, VS);
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int c = j / DT;
                acc[j % DT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[j % AHEAD], pb[c >> 1][c & 1], acc[j % DT], 0, 0, 0);
                if (j + AHEAD < NJ) va[j % AHEAD] = ap_vt8(vp + 32 * ((j + AHEAD) % DT) + 16 * ((j + AHEAD) / DT) * VS, VS);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * AHEAD, 0);
#pragma unroll
            for (int j = 0; j < NJ - AHEAD; j++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
        } else {
            const fh_half *vp = sV + vt_off;
            constexpr int NJ = 4 * DT, AHEAD = D == 128 ? 4 : 2;
            half8 vh_[AHEAD], vl_[AHEAD];
            auto read = [&](int j) {
                vh_[j % AHEAD] = ap_vt8(vp + 32 * (j % DT) + 16 * (j / DT) * VS, VS);
                vl_[j % AHEAD] = ap_vt8(vp + BN * VS + 32 * (j % DT) + 16 * (j / DT) * VS, VS);
            };
#pragma unroll
            for (int j = 0; j < AHEAD; j++) read(j);
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int c = j / DT, dt = j % DT;
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh_[j % AHEAD], pb[c >> 1][c & 1], acc[dt], 0, 0, 0);
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl_[j % AHEAD], pb[c >> 1][c & 1], acc[dt], 0, 0, 0);
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh_[j % AHEAD], pl[c >> 1][c & 1], acc[dt], 0, 0, 0);
                if (j + AHEAD < NJ) read(j + AHEAD);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 4 * AHEAD, 0);
#pragma unroll
            for (int j = 0; j < NJ - AHEAD; j++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 3 * AHEAD, 0);
        }
        if (APART) bar();
        else __syncthreads(); // tile t+1 is staged, and nobody reads this tile's buffer any more
    }
    if (APART && head == 0) bar(); // (as many barriers as the other)
    if constexpr (SPLIT) l_run = ap_swap32_sum(l_run);
    if constexpr (KS == 2) {
        ap_merge<D, 4>((float *)ap_lds, wave, lane, kset, m_run, l_run, acc);
        if (kset == 1) return;
    }
    if (qi < sq) ap_store<D>(out + (by_row ? ((int64_t)bi * sq + qi) * hq + h : ((int64_t)bi * hq + h) * sq + qi) * D, g, 1.0f / l_run, acc);
}

// f16 keys and values, one head a workgroup (KS as above).  The first product of the next tile and the softmax of this one are one stretch of code,
// so that the matrix cores work beside the vector ALU; K is a tile ahead of V for it.  Two sets of scores leave no registers for tiles on their way:
// those go straight into LDS, in rows without padding whose 16-byte pieces are swapped on the memory side (K: 16 rows' pieces of one number, V:
// 4 rows' 64 bytes cover the banks once).  What is left is the chain of a step in one wavefront (with the two key groups half a step apart, one in
// the softmax and one in the second product, it is longer: 2048 tokens 56 us).  Replayed graphs, causal, us, k_attn_prefill in the same shape and this: 8 heads of 64, 3000
// tokens 37.5 / 34.9; 16 / 4 of 64, 777 13.5 / 12.3; 32 / 8 of 128, 512 15.1 / 14.7, 2048 61.8 / 61.1, 3000 113 / 108.
template <typename TQ, int D, int KS, int QW>
__global__ __launch_bounds__(64 * QW * KS) __attribute__((amdgpu_waves_per_eu(QW == 4 ? 2 : 1, 2))) void k_attn_ahead(
    const TQ *__restrict__ q, int64_t q_sb, int64_t q_sh, int64_t q_st, const fh_half *__restrict__ k, const fh_half *__restrict__ v, int64_t kv_sb,
    int64_t kv_sh, int64_t kv_st, int hq, int hkv, int sq, int skv, float scale, int causal, int by_row, TQ *__restrict__ out) {
    constexpr int BN = 64, DT = D / 32, KSTEPS = D / 16, CH = D / 8, TILE = BN * D, NW = QW * KS, NP = TILE * KS * 2 / 1024 / NW; // NP: 1 KB pieces of K a wavefront
    extern __shared__ __attribute__((aligned(16))) fh_half ap_lds[]; // [2 buffers][KS tiles of K, KS of V]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31, g = lane >> 5;
    const int kset = KS == 2 ? wave / QW : 0;
    const int h = (int)blockIdx.x, bi = blockIdx.z, kh = h / (hq / hkv);
    const int qb0 = (causal ? (int)(gridDim.y - 1 - blockIdx.y) : (int)blockIdx.y) * 32 * QW;
    const int qi = qb0 + (wave % QW) * 32 + li, off = skv - sq;
    const fh_half *kb = k + bi * kv_sb + kh * kv_sh, *vb = v + bi * kv_sb + kh * kv_sh;
    int kend = skv;
    if (causal) {
        const int last = (qb0 + 32 * QW - 1 < sq ? qb0 + 32 * QW - 1 : sq - 1) + off + 1;
        kend = last < skv ? last : skv;
    }
    const int steps = (kend + KS * BN - 1) / (KS * BN);
    // Piece i of this wavefront: rows row + i RSTEP of a step's KS tiles; a lane brings one 16-byte piece of a row to its place.
    constexpr int RSTEP = NW * 64 / CH;
    static_assert(RSTEP % 16 == 0, "the same swap in all of a lane's rows");
    const int row_bytes = (int)(kv_st * 2), row = (wave * 64 + lane) / CH, piece = lane % CH;
    const int kc = (piece ^ (D == 128 ? row & 15 : (row >> 1) & 7)) * 16, vc = (piece ^ (D == 128 ? (row & 3) << 2 : ((row >> 1) & 1) << 2)) * 16;
    auto fetch = [&](const fh_half *base, int c, int it, int plane) { // step `it` of K (plane 0) or V (1) into its buffer
        const int t0 = it * KS * BN;
        fh_half *to = ap_lds + ((it & 1) * 2 + plane) * KS * TILE + wave * 512;
        const fh_half *from = base + t0 * kv_st;
        if (t0 + KS * BN <= skv) {
#pragma unroll
            for (int i = 0; i < NP; i++) fh_buffer_to_lds(from, 0x7FFFFFFF, to + NW * i * 512, row * row_bytes + c, i * RSTEP * row_bytes);
        } else {
#pragma unroll
            for (int i = 0; i < NP; i++) { // rows past the last key repeat it: their scores are masked and their P is 0
                const int r = row + i * RSTEP, end = skv - 1 - t0;
                fh_buffer_to_lds(from, 0x7FFFFFFF, to + NW * i * 512, (r < end ? r : end) * row_bytes + c, 0);
            }
        }
    };
    auto landed = [&]() { // this wavefront's pieces, and everybody's behind the barrier
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (steps > 0) fetch(kb, kc, 0, 0), fetch(vb, vc, 0, 1);
    half8 qf[KSTEPS];
    {
        const TQ *qp = q + bi * q_sb + h * q_sh + (int64_t)(qi < sq ? qi : sq - 1) * q_st + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ks++) {
            fh_half t[8];
            ap_load8(qp + 16 * ks, t);
            __builtin_memcpy(&qf[ks], t, 16);
        }
    }
    const int prow = 16 * (li >> 4) + 8 * ((li >> 2) & 1) + 4 * ((li >> 3) & 1) + (li & 3); // key read by MFMA row li
    const uint32_t k_at = kset * TILE * 2 + prow * D * 2 + (g ^ (D == 128 ? prow & 15 : (prow >> 1) & 7)) * 16; // bytes
    // keys 8 g + s / 4 (and 4 more) of a step of 16, dims 16 (lane / 16 % 2) + 4 (s % 4) .. of a tile of 32
    const int vrow = 8 * g + ((lane & 15) >> 2), vpiece = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
    const uint32_t v_at = (KS + kset) * TILE * 2 + vrow * D * 2 + (vpiece ^ (D == 128 ? (vrow & 3) << 2 : ((vrow >> 1) & 1) << 2)) * 16 + 8 * (lane & 1);
    const float sc2 = scale * 1.4426950408889634f, ninf = -INFINITY;
    const int lim = causal ? (qi + off < skv - 1 ? qi + off : skv - 1) : skv - 1;
    float m_run = -INFINITY, l_run = 0.f;
    floatx16 acc[DT], sa[2], sb[2];
    const floatx16 zero = {0.f};
#pragma unroll
    for (int dt = 0; dt < DT; dt++) acc[dt] = zero;

    auto scores = [&](int it, floatx16 (&to)[2]) { // S^T of step `it`
        uint32_t at = k_at + (uint32_t)(it & 1) * (4 * KS * TILE); // (swapped pieces are an exclusive or on the address, one instruction where it is used)
        asm volatile("" : "+v"(at));
        constexpr int NI = 2 * KSTEPS, AHEAD = 4;
        half8 ka[AHEAD];
        auto read = [&](int i) { ka[i % AHEAD] = *(const half8 *)((const uint8_t *)ap_lds + (at ^ (uint32_t)((i >> 1) * 32)) + (i & 1) * 64 * D); };
#pragma unroll
        for (int i = 0; i < AHEAD; i++) read(i);
#pragma unroll
        for (int i = 0; i < NI; i++) {
            to[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[i % AHEAD], qf[i >> 1], i < 2 ? zero : to[i & 1], 0, 0, 0);
            if (i + AHEAD < NI) read(i + AHEAD);
        }
    };
    auto mask = [&](int it, floatx16 (&to)[2]) {
        const int t0 = (it * KS + kset) * BN, lim_t = KS == 1 || t0 < kend ? lim : -1; // (a group without a tile in the last step: all of it)
        if (__any(t0 + BN - 1 > lim_t))
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = t0 + 32 * kt + 16 * (r >> 3) + 8 * g + (r & 7);
                    asm volatile("v_cmp_le_i32 vcc, %1, %2\n\tv_cndmask_b32 %0, %3, %0, vcc"
                                 : "+v"(to[kt][r])
                                 : "v"(key), "v"(lim_t), "v"(ninf)
                                 : "vcc");
                }
    };
    auto step = [&](int it, floatx16 (&st)[2], floatx16 (&next)[2], bool last) {
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int r = 0; r < 16; r++) mx = fmaxf(mx, st[kt][r]);
        mx = ap_swap32_max(mx) * sc2;
        if (__any(mx > m_run)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new, l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[dt][r] *= alpha;
        }
        const float m_sub = m_run == -INFINITY ? 0.f : -m_run; // dead rows: 2^(-inf - 0) = 0
        if (it + 2 < steps) fetch(kb, kc, it + 2, 0);
        if (!last) fetch(vb, vc, it + 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        if (!last) scores(it + 1, next);
        half8 pb[2][2];
        float ps = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++) {
                fh_half t[8];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(st[kt][8 * s2 + e], sc2, m_sub)); // arguments <= 0
                    ps += p;
                    t[e] = (fh_half)p;
                }
                __builtin_memcpy(&pb[kt][s2], t, 16);
            }
        l_run += ap_swap32_sum(ps);
        if (!last) {
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int i = 0; i < 2 * KSTEPS; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (i < 2 * KSTEPS - 4) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 80 / (2 * KSTEPS), 0);
                __builtin_amdgcn_sched_group_barrier(0x400, 32 / (2 * KSTEPS), 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!last) mask(it + 1, next);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t at = v_at + (uint32_t)(it & 1) * (4 * KS * TILE);
        asm volatile("" : "+v"(at));
        constexpr int NJ = 4 * DT, AHEAD = 8;
        half8 va[AHEAD];
        auto read = [&](int j) { va[j % AHEAD] = ap_vt8((const fh_half *)((const uint8_t *)ap_lds + (at ^ (uint32_t)(j % DT * 64))) + 16 * (j / DT) * D, D); };
#pragma unroll
        for (int j = 0; j < AHEAD; j++) read(j);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int c = j / DT;
            acc[j % DT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[j % AHEAD], pb[c >> 1][c & 1], acc[j % DT], 0, 0, 0);
            if (j + AHEAD < NJ) read(j + AHEAD);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * AHEAD, 0);
#pragma unroll
        for (int j = 0; j < NJ - AHEAD; j++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
        landed();
    };
    if (steps > 0) {
        landed();
        if (steps > 1) fetch(kb, kc, 1, 0);
        scores(0, sa);
        mask(0, sa);
        landed(); // (K of step 1; the place of step 0's is free)
        int t = 0;
        for (; t + 2 < steps; t += 2) {
            step(t, sa, sb, false);
            step(t + 1, sb, sa, false);
        }
        if (t + 2 == steps) {
            step(t, sa, sb, false);
            step(t + 1, sb, sa, true);
        } else
            step(t, sa, sb, true);
    }
    if constexpr (KS == 2) ap_merge<D, QW>((float *)ap_lds, wave, lane, kset, m_run, l_run, acc);
    if (KS == 2 && kset == 1) return;
    if (qi < sq) ap_store<D>(out + (by_row ? ((int64_t)bi * sq + qi) * hq + h : ((int64_t)bi * hq + h) * sq + qi) * D, g, 1.0f / l_run, acc);
}

template <typename TQ, typename TKV, int D, bool SPLIT, int HW, int KS = 1, bool ANY = false>
static fh_status ap_launch_k(fh_device *dev, const void *q, int64_t q_sb, int64_t q_sh, int64_t q_st, const void *k,
                             const void *v, int64_t kv_sb, int64_t kv_sh, int64_t kv_st, int b, int hq, int hkv, int sq,
                             int skv, float scale, int causal, int by_row, void *out) {
    constexpr int LDS = 2 * KS * (SPLIT ? 2 : 1) * 64 * (D + 8 + ap_v_row<D, SPLIT, HW>) * 2; // two buffers of KS tiles (K and V planes), bytes
    static_assert(KS == 1 || LDS >= (2 + (D / 32) * 16) * 256 * 4, "the merge of the key groups reuses the tile buffers");
    static_assert(!(SPLIT && D == 64 && HW == 1) || 2 * LDS <= 160 * 1024, "two workgroups a compute unit");
    static_assert(LDS <= 160 * 1024, "KV tiles exceed the LDS of a compute unit");
    auto kern = k_attn_prefill<TQ, TKV, D, SPLIT, HW, KS, ANY>;
    FH_TRY(fh_kernel_lds(dev, (const void *)kern, LDS)); // allow more than 64 KB of dynamic LDS
    dim3 grid((unsigned)(hq / HW), (unsigned)((sq + 127) / 128), (unsigned)b);
    kern<<<grid, 256 * HW * KS, LDS, dev->stream>>>((const TQ *)q, q_sb, q_sh, q_st, (const TKV *)k, (const TKV *)v, kv_sb,
                                               kv_sh, kv_st, hq, hkv, sq, skv, scale, causal, by_row, (TQ *)out);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

template <typename TQ, int D, int KS, int QW = 4>
static fh_status ap_launch_ahead(fh_device *dev, const void *q, int64_t q_sb, int64_t q_sh, int64_t q_st, const void *k, const void *v, int64_t kv_sb,
                                 int64_t kv_sh, int64_t kv_st, int b, int hq, int hkv, int sq, int skv, float scale, int causal, int by_row, void *out) {
    constexpr int LDS = 2 * 2 * KS * 64 * D * 2, MERGE = KS == 2 ? (2 + D / 2) * 64 * QW * 4 : 0, BYTES = LDS > MERGE ? LDS : MERGE;
    FH_TRY(fh_kernel_lds(dev, (const void *)k_attn_ahead<TQ, D, KS, QW>, BYTES));
    k_attn_ahead<TQ, D, KS, QW><<<dim3((unsigned)hq, (unsigned)((sq + 32 * QW - 1) / (32 * QW)), (unsigned)b), 64 * QW * KS, BYTES, dev->stream>>>(
        (const TQ *)q, q_sb, q_sh, q_st, (const fh_half *)k, (const fh_half *)v, kv_sb, kv_sh, kv_st, hq, hkv, sq, skv, scale, causal, by_row, (TQ *)out);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

template <typename TQ, typename TKV, bool SPLIT = false>
static fh_status ap_launch(fh_device *dev, const void *q, int64_t q_sb, int64_t q_sh, int64_t q_st, const void *k,
                           const void *v, int64_t kv_sb, int64_t kv_sh, int64_t kv_st, int b, int hq, int hkv, int sq,
                           int skv, int d, float scale, int causal, int by_row, void *out) {
    const long wgs = (long)hq * ((sq + 127) / 128) * b;
    // attn_kernel = 6 / 7 / 8 / 9 force the workgroup shape (two heads, f32 keys only / two key groups / plain / 64-row query blocks
    // with two key groups) whatever the size: tests
    const int64_t force = dev->opt_attn_kernel;
#define FH_AP(D, HW, KS, ...) ap_launch_k<TQ, TKV, D, SPLIT, HW, KS, ##__VA_ARGS__>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, scale, causal, by_row, out)
    // A request of 16 bytes, straight into LDS above all, is made for an address of its multiple, and a step's 128 rows lie within the 2^31 bytes
    // of a buffer.  Other views are read as they lie by the plain form (32 / 8 heads of 128, causal, us: K and V of f16 one element off 149, aligned 55, a row a
    // workgroup 8600; of f32 128, 134, 6400).
    if (((uintptr_t)k | (uintptr_t)v) & 15 || kv_st < 0 || kv_st >= 1 << 21) return d == 128 ? FH_AP(128, 1, 1, true) : FH_AP(64, 1, 1, true);
    if constexpr (!SPLIT) {
        // up to two rounds of workgroups (one a compute unit at a time: its tiles are 128 KB of LDS for head_dim 128), the longest first, so that a long and a short
        // one follow each other: a workgroup's key tiles are shared out over two groups of wavefronts
        const bool halves = force == 7 || force == 9 || (force != 6 && force != 8 && wgs <= 2L * dev->compute_units && skv > 128);
        if constexpr (sizeof(TKV) == 2) {
            // shorter still: query blocks of 64 rows, four wavefronts, while one workgroup per compute unit holds (nearly) all
            // of them - a SIMD then runs one wavefront's chain of a step instead of two (512 tokens: 15.0 against 16.8 us)
            const long wgs64 = (long)hq * ((sq + 63) / 64) * b;
            const bool rows64 = force == 9 || (force == 0 && halves && 4 * wgs64 <= 5L * dev->compute_units);
#define FH_AH(D, KS) ap_launch_ahead<TQ, D, KS>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, scale, causal, by_row, out)
            if (rows64)
                return d == 128 ? ap_launch_ahead<TQ, 128, 2, 2>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, scale, causal, by_row, out)
                                : ap_launch_ahead<TQ, 64, 2, 2>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, scale, causal, by_row, out);
            if (halves) return d == 128 ? FH_AH(128, 2) : FH_AH(64, 2);
            // Up to two key tiles a query there is little to overlap, and the longer code costs more than it gives (32 / 8 heads of 128:
            // 65 tokens 6.74 us for 6.55, 128 tokens 7.85 for 7.71; from 129 on, in two key groups, 7.5 for 8.4).  Two heads a workgroup are not quicker in any number of
            // workgroups (causal, us, two heads in k_attn_prefill / this: 8 x 8 / 2 of 64, 2048 tokens 104 / 73; 4 x 32 / 8 of 128, 1024 75 / 62; 32 / 8 of 128, 8000
            // 570 / 566; 128 x 8 / 2 of 64, 65 tokens 17.6 / 14.6, 32 x 32 / 8 of 128, 128 level).
            if (skv > 128 || force == 8) return d == 128 ? FH_AH(128, 1) : FH_AH(64, 1);
#undef FH_AH
            return d == 128 ? FH_AP(128, 1, 1) : FH_AP(64, 1, 1);
        } else {
            if (halves) return d == 128 ? FH_AP(128, 1, 2) : FH_AP(64, 1, 2);
        }
    }
    if constexpr (sizeof(TKV) == 4) {
        // Two heads of one KV group share the staged tiles when the launch still has enough workgroups without the
        // split: short prompts are bound by the longest workgroup and by how many compute units have one at all.
        const bool pair = (hq / hkv) % 2 == 0 && (force == 6 || (force != 7 && force != 8 && wgs >= 1024));
        if (d == 128) return pair ? FH_AP(128, 2, 1) : FH_AP(128, 1, 1);
        return pair ? FH_AP(64, 2, 1) : FH_AP(64, 1, 1);
    }
#undef FH_AP
}

// out [b][hq][sq][d], or with by_row [b][sq][hq][d], the rows that the product behind it takes: a decoder's prompt of 2048 (32 heads of 128)
// saves the 21 us a layer of turning the one into the other.
// FH_ERR_UNSUPPORTED when the shape is not one this kernel is written for (the caller keeps the generic kernel).
fh_status fh_attention_prefill_mfma(fh_device *dev, int q_dtype, int kv_dtype, const void *q, int64_t q_sb,
                                    int64_t q_sh, int64_t q_st, const void *k, const void *v, int64_t kv_sb,
                                    int64_t kv_sh, int64_t kv_st, int b, int hq, int hkv, int sq, int skv, int d,
                                    float scale, int mask_kind, bool by_row, void *out) {
    if ((d != 128 && d != 64) || hq % hkv || (mask_kind != FH_MASK_NONE && mask_kind != FH_MASK_CAUSAL)) return FH_ERR_UNSUPPORTED;
    if (q_st % 8 || q_sh % 8 || q_sb % 8 || kv_st % 8 || kv_sh % 8 || kv_sb % 8 || (sq + 127) / 128 > 65535 || b > 65535) return FH_ERR_UNSUPPORTED;
    if (mask_kind == FH_MASK_CAUSAL && skv < sq) return FH_ERR_UNSUPPORTED;
    const int causal = mask_kind == FH_MASK_CAUSAL;
    if (q_dtype == FH_F16 && kv_dtype == FH_F16)
        return ap_launch<fh_half, fh_half>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, d, scale, causal, by_row, out);
    if (q_dtype == FH_F32 && kv_dtype == FH_F16)
        return ap_launch<float, fh_half>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, d, scale, causal, by_row, out);
    if (q_dtype == FH_F32 && kv_dtype == FH_F32 && dev->opt_attn_kernel != 2) // all f32: split operands, f32 accuracy
        return ap_launch<float, float, true>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, d, scale, causal, by_row, out);
    if (q_dtype == FH_F32 && kv_dtype == FH_F32)
        return ap_launch<float, float>(dev, q, q_sb, q_sh, q_st, k, v, kv_sb, kv_sh, kv_st, b, hq, hkv, sq, skv, d, scale, causal, by_row, out);
    return FH_ERR_UNSUPPORTED;
}
