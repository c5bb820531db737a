// Decode step kernels of the layer-list decoders (fh_step.h).
#include "fh_step.h"
#include <algorithm>

static constexpr float FH_LOG2E = 1.4426950408889634f;


// One step of a recurrence: workgroup b takes 16 columns of one head's state, RPT rows per lane as in the prefill scan.
template <int RPT>
__device__ __forceinline__ void rec_step(const FhStep &st, int b, float *lds) {
    const FhRecurrent &r = st.rec;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, rg = lane & 15;
    const int ncb = (r.vdim + 15) / 16, h = b / ncb, cb = b % ncb, d = r.dim, rep = r.heads / r.kv_heads, kh = h / rep;
    const int nq = r.kv_heads * d, channels = 2 * nq + r.heads * r.vdim, pos = *st.pos_dev;
    const int col = cb * 16 + wave * 4 + (lane >> 4), i0 = rg * RPT;
    const bool live = col < r.vdim;
    const int c = live ? col : r.vdim - 1;
    float *sp = st.rec_state.s + ((int64_t)h * r.vdim + c) * d;
    float S[RPT];
#pragma unroll
    for (int i = 0; i < RPT; i++) S[i] = pos > 0 && i0 + i < d ? sp[i0 + i] : 0.f;
    float *qk = lds, *vv = lds + 2 * d, *f = vv + 16; // [2 d], [16], [2]
    float *slot = st.rec_state.conv + (int64_t)(pos % r.taps) * channels; // not among the rows the convolution reads
    const bool keep = cb == 0 && h % rep == 0;        // one workgroup per key head stores its projections
    for (int i = tid; i < 2 * d; i += 256) {
        const int ch = i < d ? kh * d + i : nq + kh * d + i - d;
        qk[i] = fh_rec_conv(r, ch, st.proj, 0, 0, pos, st.rec_state.conv, channels);
        if (keep) slot[ch] = st.proj[i < d ? r.col_q + kh * d + i : r.col_k + kh * d + i - d];
    }
    if (tid < 16 && cb * 16 + tid < r.vdim) {
        const int vc = h * r.vdim + cb * 16 + tid;
        vv[tid] = fh_rec_conv(r, 2 * nq + vc, st.proj, 0, 0, pos, st.rec_state.conv, channels);
        slot[2 * nq + vc] = st.proj[r.col_v + vc];
    }
    __syncthreads();
    if (wave < 2) {
        float g = 1.f;
        if (r.delta()) {
            float ss = 0.f;
            for (int i = lane; i < d; i += 64) ss = fmaf(qk[wave * d + i], qk[wave * d + i], ss);
            g = 1.0f / sqrtf(fh_wave_sum(ss) + 1e-6f);
        }
        if (lane == 0) f[wave] = wave == 0 ? g * r.q_scale : g;
    }
    const float sp_ = fh_softplus_f(st.proj[r.col_a + h] + r.dt_bias[h]);
    const float g = expf(-expf(r.a_log[h]) * sp_), be = r.delta() ? fh_sigmoid_f(st.proj[r.col_b + h]) : sp_;
    __syncthreads();
    const float v = vv[live ? wave * 4 + (lane >> 4) : 0];
    float k[RPT], dot = 0.f, o = 0.f;
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        k[i] = i0 + i < d ? qk[d + i0 + i] * f[1] : 0.f;
        S[i] *= g;
        dot = fmaf(S[i], k[i], dot);
    }
    const float u = r.delta() ? be * (v - fh_row16_sum(dot)) : be * v;
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        S[i] = fmaf(k[i], u, S[i]);
        o = fmaf(S[i], i0 + i < d ? qk[i0 + i] * f[0] : 0.f, o);
        if (live && i0 + i < d) sp[i0 + i] = S[i];
    }
    o = fh_row16_sum(o);
    if (rg == 0 && live) st.o[h * r.vdim + col] = o + (r.d_skip ? r.d_skip[h] * v : 0.f);
}

// Absorbed queries of latent attention: workgroup b < heads * chunks takes 128 latent dimensions of one head, the last one
// appends this position's cache row.
template <typename T>
__device__ __forceinline__ void latent_step(const FhStep &st, T *ring, int cap, int b, float *lds) {
    const FhLatent &a = st.lat;
    const int tid = threadIdx.x, chunks = (a.r8 + 127) / 128, pos = *st.pos_dev, row = a.r8 + a.drp;
    const float *ct = a.cos_t + (int64_t)pos * a.pairs, *sn = a.sin_t + (int64_t)pos * a.pairs;
    if (b == a.heads * chunks) {
        const float *p = st.proj + a.col_kv;
        float ss = 0.f;
        for (int c = tid; c < a.rank; c += 256) ss = fmaf(p[c], p[c], ss);
        ss = fh_wave_sum(ss);
        if ((tid & 63) == 0) lds[tid >> 6] = ss;
        __syncthreads();
        const float inv = 1.0f / sqrtf((lds[0] + lds[1] + lds[2] + lds[3]) / (float)a.rank + a.eps);
        T *dst = ring + (int64_t)(pos % cap) * row;
        for (int c = tid; c < row; c += 256) {
            float v = 0.f;
            if (c < a.rank) v = p[c] * inv * a.c_norm[c];
            else if (c >= a.r8 && c - a.r8 < a.dr) {
                const int i = c - a.r8, pr = i >> 1;
                v = p[a.rank + i];
                if (pr < a.pairs) {
                    const float o = p[a.rank + (i ^ 1)];
                    v = (i & 1) ? v * ct[pr] + o * sn[pr] : v * ct[pr] - o * sn[pr];
                }
            }
            dst[c] = fh_to<T>(v);
        }
        return;
    }
    const int h = b / chunks, c0 = (b % chunks) * 128, sub = tid & 15, dg = tid >> 4, c = c0 + sub * 8;
    const float sc = a.scale * FH_LOG2E;
    const float *q = st.proj + a.col_q + h * (a.dn + a.dr);
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = 0.f;
    if (c < a.rp)
        for (int d = dg; d < a.dn; d += 16) {
            const uint4 w = *(const uint4 *)(a.uk + (int64_t)(h * a.dnp + d) * a.rp + c);
            const float x = q[d];
            acc[0] = fmaf(fh_bf_lo(w.x), x, acc[0]);
            acc[1] = fmaf(fh_bf_hi(w.x), x, acc[1]);
            acc[2] = fmaf(fh_bf_lo(w.y), x, acc[2]);
            acc[3] = fmaf(fh_bf_hi(w.y), x, acc[3]);
            acc[4] = fmaf(fh_bf_lo(w.z), x, acc[4]);
            acc[5] = fmaf(fh_bf_hi(w.z), x, acc[5]);
            acc[6] = fmaf(fh_bf_lo(w.w), x, acc[6]);
            acc[7] = fmaf(fh_bf_hi(w.w), x, acc[7]);
        }
#pragma unroll
    for (int e = 0; e < 8; e++) lds[dg * 128 + sub * 8 + e] = acc[e];
    __syncthreads();
    float *dst = st.qa + (int64_t)h * row;
    if (tid < 128 && c0 + tid < a.r8) {
        float v = 0.f;
#pragma unroll
        for (int g = 0; g < 16; g++) v += lds[g * 128 + tid];
        dst[c0 + tid] = v * sc;
    }
    if (c0 == 0)
        for (int i = tid; i < a.drp; i += 256) {
            const int pr = i >> 1;
            float v = i < a.dr ? q[a.dn + i] : 0.f;
            if (i < a.dr && pr < a.pairs) {
                const float o = q[a.dn + (i ^ 1)];
                v = (i & 1) ? v * ct[pr] + o * sn[pr] : v * ct[pr] - o * sn[pr];
            }
            dst[a.r8 + i] = v * sc;
        }
}

// Gate and up products of the chosen experts, dealt out over `blocks` workgroups of four wavefronts: a wavefront takes one activation after
// the other, its gate and its up row together, in pieces of 512 with 4 KB on their way (FhRowDeal has the reason).  The chosen experts have
// to be known first, so every workgroup works them out.  us of the launch in a step of width 2048, top 6 of 64 experts of 1024 (50 MB: a plain read takes 9.0):
// beside latent attention 14.9 / 12.9, beside a recurrence 15.5 / 13.8 (workgroups of eight activations, 16 KB a wavefront on their way / now).
__device__ __forceinline__ void expert_step(const FhStep &st, int b, int blocks, float *lds) {
    constexpr int AHEAD = 2, NX = 4;
    const FhMoe &m = st.moe;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lane8 = lane * 8;
    const int kp = st.kp, pieces = fh_row_pieces(kp), total = m.top * m.ff, step = blocks * 4, first = wave * blocks + b;
    const FhRowInput xs{lds, pieces * 256};
    int *who = (int *)(lds + 2 * xs.plane);
    float4 x[NX]; // requested beside the router's logits
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int i = (tid + 256 * j) * 4;
        x[j] = *(const float4 *)(st.hn + (i < kp ? i : 0));
    }
    if (wave == 0)
        fh_moe_route(st.proj + m.col_z, m.experts, m.scale, m.top, [&](int n, int e, float w) {
            if (lane == 0) {
                who[n] = e;
                if (b == 0) st.ids[n] = e, st.wts[n] = w;
            }
        });
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int i = (tid + 256 * j) * 4;
        float4 v = x[j];
        if (i >= kp) v.x = v.y = v.z = v.w = 0.f;
        if (i < 2 * xs.plane) xs.quad(i >> 2) = v;
    }
    for (int i = (tid + 256 * NX) * 4; i < 2 * xs.plane; i += 1024) {
        float4 v = zero;
        if (i < kp) v = *(const float4 *)(st.hn + i);
        xs.quad(i >> 2) = v;
    }
    fh_lds_barrier();
    const int count = first < total ? (total - first + step - 1) / step : 0;
    struct At { int slot, p; }; // activation p of a chosen expert
    auto ahead = [&](At a, int by) {
        a.p += by;
        while (a.p >= m.ff) a.p -= m.ff, a.slot++;
        return a;
    };
    auto gate = [&](const At &a) { // (its up row is the 16th behind it)
        return m.gate_up + (int64_t)__builtin_amdgcn_readfirstlane(who[a.slot]) * m.gu_stride + (int64_t)(a.p / 16 * 32 + a.p % 16) * kp;
    };
    At next = ahead(At{0, 0}, count ? first : 0), now = next;
    const uint16_t *row = gate(next);
    int left = count, piece = 0;
    uint4 g[AHEAD], u[AHEAD];
    auto fetch = [&](int s) {
        g[s] = fh_load_row_once(row, kp, piece * 512 + lane8);
        u[s] = fh_load_row_once(row + (int64_t)16 * kp, kp, piece * 512 + lane8);
        if (++piece == pieces) {
            piece = 0, left--;
            if (left > 0) next = ahead(next, step), row = gate(next);
        }
    };
#pragma unroll
    for (int s = 0; s < AHEAD; s++) fetch(s);
    float ag = 0.f, au = 0.f;
    int p = 0, i = 0;
    for (int t = 0; t < count * pieces; t += AHEAD) {
#pragma unroll
        for (int s = 0; s < AHEAD; s++) {
            const float *at = xs.xs + p * 256 + lane * 4;
            const float4 a = *(const float4 *)at, c = *(const float4 *)(at + xs.plane);
            ag = fh_dot8(g[s], a, c, ag);
            au = fh_dot8(u[s], a, c, au);
            fetch(s);
            if (++p == pieces) {
                ag = fh_wave_sum(ag), au = fh_wave_sum(au);
                if (i < count && lane == 0) st.act[(int64_t)now.slot * m.ffp + now.p] = fh_silu_f(ag) * au;
                ag = au = 0.f, p = 0;
                if (++i < count) now = ahead(now, step);
            }
        }
    }
}

template <int RPT>
__global__ __launch_bounds__(256) void k_step_recurrent(FhStep st, int n_mix) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    if ((int)blockIdx.x < n_mix) rec_step<RPT>(st, blockIdx.x, lds);
    else expert_step(st, (int)blockIdx.x - n_mix, (int)gridDim.x - n_mix, lds);
}
template <typename T>
__global__ __launch_bounds__(256) void k_step_latent(FhStep st, T *ring, int cap, int n_mix) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    if ((int)blockIdx.x < n_mix) latent_step<T>(st, ring, cap, blockIdx.x, lds);
    else expert_step(st, (int)blockIdx.x - n_mix, (int)gridDim.x - n_mix, lds);
}

fh_status fh_step_middle(fh_device *dev, int dtype, const FhStep &st, fh_kvcache *cache) {
    const FhMoe &m = st.moe;
    // two workgroups of four wavefronts a compute unit, if there is an activation for every wavefront
    const int n_exp = m.experts ? std::min(2 * dev->compute_units, (m.top * m.ff + 3) / 4) : 0;
    size_t lds = m.experts ? (size_t)(fh_row_pieces(st.kp) * 512 + m.top) * 4 : 0;
    if (st.kind == FH_MIX_RECURRENT) {
        const int n_mix = st.rec.heads * ((st.rec.vdim + 15) / 16), rpt = (st.rec.dim + 15) / 16;
        const size_t need = (size_t)(2 * st.rec.dim + 32) * 4;
        lds = lds > need ? lds : need;
        FH_REQUIRE(rpt <= 16, "recurrent state of %d rows (at most 256)", st.rec.dim);
        const dim3 grid((unsigned)(n_mix + n_exp));
#define STEP_RECURRENT(RPT_)                                                                                     \
    do {                                                                                                         \
        if (lds > 48 * 1024) FH_TRY(fh_kernel_lds(dev, (const void *)k_step_recurrent<RPT_>, lds));              \
        k_step_recurrent<RPT_><<<grid, 256, lds, dev->stream>>>(st, n_mix);                                      \
    } while (0)
        if (rpt <= 2) STEP_RECURRENT(2);
        else if (rpt <= 4) STEP_RECURRENT(4);
        else if (rpt <= 8) STEP_RECURRENT(8);
        else STEP_RECURRENT(16);
#undef STEP_RECURRENT
    } else {
        const int n_mix = st.lat.heads * ((st.lat.r8 + 127) / 128) + 1;
        const size_t need = (size_t)16 * 128 * 4;
        lds = lds > need ? lds : need;
        const dim3 grid((unsigned)(n_mix + n_exp));
#define STEP_LATENT(T_)                                                                                          \
    do {                                                                                                         \
        if (lds > 48 * 1024) FH_TRY(fh_kernel_lds(dev, (const void *)k_step_latent<T_>, lds));                   \
        k_step_latent<T_><<<grid, 256, lds, dev->stream>>>(st, (T_ *)cache->k, cache->capacity, n_mix);          \
    } while (0)
        if (dtype == FH_F32) STEP_LATENT(float);
        else STEP_LATENT(uint16_t);
#undef STEP_LATENT
    }
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// ------------------------------------------------------------------------------ output launch
// Rows of the residual stream, dealt out over workgroups of eight wavefronts, one a compute unit.  A row's weights - of the output projection, of
// the chosen experts and of the always-on one - are one list of pieces of 512, and a wavefront has 4 KB of them on their way (FhRowDeal has the
// reason).  The inputs and the experts' numbers are requested first, so that they do not wait behind weights, then the first pieces of the output
// projection, whose places are known.  us of the launch in a step of width 2048, seven experts of 1024: behind latent attention (38 MB, a plain read 7.2) 12.6 /
// 11.5, a delta rule 15.7 / 13.0, a state space (46 MB, 8.4) 20.1 / 14.2 (one row a wavefront with 8 KB on their way / now; with a table of the
// pieces in the LDS, a round trip for every piece, 14.4 / 16.4 / 16.5).  Narrow streams gain nothing here, long rows of few wavefronts lose (512 wide, eight experts of 2048
// 14.9 / 16.9, of which the hint of fh_load_once is all; 1024 wide 17.6 / 17.9): 8 KB on the way 16.9, the experts' numbers in a register instead of the LDS 17.1, the next
// piece's inputs asked for ahead 17.2.
// NO, NE, NS: fours of values of the mixer, of the experts and of the always-on one that a thread holds in registers, requested ahead of the weights;
// NO = 0: mixers whose length or groups are no multiple of 4, and longer inputs, are read as they are staged.  PRE: the output projection has four pieces or more.
template <int NO, int NE, int NS, bool PRE>
__global__ __launch_bounds__(512) void k_step_out(FhStep st) {
    constexpr int AHEAD = 4;
    constexpr bool EARLY = NO > 0;
    extern __shared__ __attribute__((aligned(16))) float lds[]; // [kpo | top * ffp | sffp | norm groups | kpo / 4 (EARLY, recurrent) | top]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lane8 = lane * 8;
    const FhMoe &m = st.moe;
    const int n_e = m.experts ? m.top : 0, n_s = m.sff ? m.sffp : 0, n_in = st.kpo + n_e * m.ffp + n_s;
    const bool recurrent = st.kind == FH_MIX_RECURRENT;
    const int n_g = recurrent ? (st.rec.norm_groups + 3) / 4 * 4 : 0, e0 = st.kpo, s0 = e0 + n_e * m.ffp;
    const FhRowInput in{lds, n_in / 2}; // (all lengths are multiples of 64)
    float *ginv = lds + n_in, *sums = ginv + n_g;
    int *who = (int *)(sums + (EARLY && recurrent ? st.kpo / 4 : 0));
    const int inner = recurrent ? st.rec.heads * st.rec.vdim : st.lat.heads * st.lat.dv;
    const float *gate = recurrent ? st.proj + st.rec.col_g : st.o;
    const bool gate_first = recurrent && st.rec.gate_first;
    const int blocks = (int)gridDim.x, step = 8 * blocks, first = wave * blocks + (int)blockIdx.x;
    const int count = first < st.width ? (st.width - first + step - 1) / step : 0;
    const int expert = (n_e ? st.ids : (const int *)st.o)[tid < n_e ? tid : 0]; // (what is not there is read from the mixer's output and dropped)
    float ew[EARLY ? NE : 1];
    float4 o[EARLY ? NO : 1], g[EARLY ? NO : 1], ev[EARLY ? NE : 1], sg[EARLY ? NS : 1], su[EARLY ? NS : 1], nw[EARLY ? NO : 1];
    const float *acts = n_e ? st.act : st.o, *weights = n_e ? st.wts : st.o, *shared = n_s ? st.s_gu : st.o, *norm = recurrent ? st.rec.norm : st.o;
    if constexpr (EARLY) {
#pragma unroll
        for (int j = 0; j < NO; j++) {
            const int i = (tid + 512 * j) * 4, at = i < inner ? i : 0;
            o[j] = *(const float4 *)(st.o + at);
            g[j] = *(const float4 *)(gate + at);
            nw[j] = *(const float4 *)(norm + (recurrent && st.rec.norm_len != inner ? at % st.rec.norm_len : at));
        }
#pragma unroll
        for (int j = 0; j < NE; j++) {
            const int i = (tid + 512 * j) * 4;
            ev[j] = *(const float4 *)(acts + (i < n_e * m.ffp ? i : 0));
            ew[j] = weights[i < n_e * m.ffp ? i / m.ffp : 0];
        }
#pragma unroll
        for (int j = 0; j < NS; j++) { // (gate and up in alternating groups of 16)
            const int i = (tid + 512 * j) * 4, at = i < n_s ? i / 16 * 32 + i % 16 : 0;
            sg[j] = *(const float4 *)(shared + at);
            su[j] = *(const float4 *)(shared + (n_s ? at + 16 : 0));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    uint4 u[AHEAD];
    // A row's stretches: the output projection, the experts, the always-on one; a place is k values into one, whose inputs begin at `from`.
    const int n_seg = 1 + n_e + (n_s ? 1 : 0);
    struct Place { int seg, k, kp, from; };
    auto advance = [&](Place &a) { // true: to the next row
        a.k += 512;
        if (a.k < a.kp) return false;
        a.k = 0, a.from += a.kp, a.seg++;
        const bool end = a.seg == n_seg;
        if (end) a.seg = a.from = 0;
        a.kp = a.seg == 0 ? st.kpo : a.seg <= n_e ? m.ffp : m.sffp;
        return end;
    };
    Place next{0, 0, st.kpo, 0}, now = next;
    int row = first < st.width ? first : st.width - 1, left = count;
    const uint16_t *w = st.wo + (int64_t)row * st.kpo;
    auto fetch = [&](int s) { // (a lane past the end of a short piece repeats its last eight values)
        const int c = next.k + lane8;
        u[s] = fh_load_once(w + (c < next.kp ? c : next.kp - 8));
        if (advance(next)) row += --left > 0 ? step : 0;
        if (next.k == 0) {
            const uint16_t *base = next.seg == 0 ? st.wo : next.seg > n_e ? m.s_down : m.down + (int64_t)__builtin_amdgcn_readfirstlane(who[next.seg - 1]) * m.down_stride;
            w = base + (int64_t)row * next.kp;
        }
    };
    if (PRE)
#pragma unroll
        for (int s = 0; s < AHEAD; s++) { // (the last one's place is worked out behind the barrier, where the experts are known)
            const int c = s * 512 + lane8;
            u[s] = fh_load_once(w + (c < st.kpo ? c : st.kpo - 8));
        }
    __builtin_amdgcn_sched_barrier(0);
    if (tid < n_e) who[tid] = expert;
    for (int i = tid + 512; i < n_e; i += 512) who[i] = st.ids[i]; // (a token has as many as there are, up to 1024)
    auto put = [&](int i, float4 v, float w) {
        const int c = i % m.ffp;
        v.x = c < m.ff ? w * v.x : 0.f, v.y = c + 1 < m.ff ? w * v.y : 0.f, v.z = c + 2 < m.ff ? w * v.z : 0.f, v.w = c + 3 < m.ff ? w * v.w : 0.f;
        in.quad((e0 + i) >> 2) = v;
    };
    if constexpr (EARLY) {
#pragma unroll
        for (int j = 0; j < NO; j++) {
            const int q = tid + 512 * j, i = q * 4;
            if (gate_first) o[j] = make_float4(o[j].x * fh_silu_f(g[j].x), o[j].y * fh_silu_f(g[j].y), o[j].z * fh_silu_f(g[j].z), o[j].w * fh_silu_f(g[j].w));
            if (i >= inner) o[j].x = o[j].y = o[j].z = o[j].w = 0.f;
            if (!recurrent && i < st.kpo) in.quad(q) = o[j];
            if (recurrent && i < st.kpo) sums[q] = fmaf(o[j].x, o[j].x, fmaf(o[j].y, o[j].y, fmaf(o[j].z, o[j].z, o[j].w * o[j].w)));
        }
#pragma unroll
        for (int j = 0; j < NE; j++)
            if ((tid + 512 * j) * 4 < n_e * m.ffp) put((tid + 512 * j) * 4, ev[j], ew[j]);
#pragma unroll
        for (int j = 0; j < NS; j++) {
            const int i = (tid + 512 * j) * 4;
            if (i < n_s)
                in.quad((s0 + i) >> 2) = make_float4(fh_silu_f(sg[j].x) * su[j].x, fh_silu_f(sg[j].y) * su[j].y, fh_silu_f(sg[j].z) * su[j].z, fh_silu_f(sg[j].w) * su[j].w);
        }
    } else {
        for (int i = tid; i < st.kpo; i += 512) {
            float v = i < inner ? st.o[i] : 0.f;
            if (gate_first && i < inner) v *= fh_silu_f(gate[i]);
            in.at(i) = v;
        }
        for (int i = tid * 4; i < n_e * m.ffp; i += 2048) put(i, *(const float4 *)(st.act + i), st.wts[i / m.ffp]);
        for (int i = tid; i < n_s; i += 512) {
            const int at = i / 16 * 32 + i % 16;
            in.at(s0 + i) = fh_silu_f(st.s_gu[at]) * st.s_gu[at + 16];
        }
    }
    fh_lds_barrier();
    if (PRE) { // where the requests above left off
        next.k = (AHEAD - 1) * 512;
        if (advance(next)) row += --left > 0 ? step : 0;
        if (next.k == 0)
            w = (next.seg == 0 ? st.wo : next.seg > n_e ? m.s_down : m.down + (int64_t)__builtin_amdgcn_readfirstlane(who[next.seg - 1]) * m.down_stride) + (int64_t)row * next.kp;
    } else
#pragma unroll
        for (int i = 0; i < AHEAD; i++) fetch(i);
    if (recurrent) {
        const FhRecurrent &rc = st.rec;
        const int gl = inner / rc.norm_groups;
        for (int n = wave; n < rc.norm_groups; n += 8) {
            float ss = 0.f;
            if (EARLY)
                for (int i = lane; i < gl >> 2; i += 64) ss += sums[n * (gl >> 2) + i];
            else
                for (int i = lane; i < gl; i += 64) ss = fmaf(in.at(n * gl + i), in.at(n * gl + i), ss);
            ss = fh_wave_sum(ss);
            if (lane == 0) ginv[n] = 1.0f / sqrtf(ss / (float)gl + rc.eps);
        }
        fh_lds_barrier();
        if constexpr (EARLY) {
#pragma unroll
            for (int j = 0; j < NO; j++) {
                const int q = tid + 512 * j, i = q * 4;
                const float inv = ginv[i < inner ? i / gl : 0];
                float4 v = make_float4(o[j].x * inv * nw[j].x, o[j].y * inv * nw[j].y, o[j].z * inv * nw[j].z, o[j].w * inv * nw[j].w);
                if (!gate_first) v = make_float4(v.x * fh_silu_f(g[j].x), v.y * fh_silu_f(g[j].y), v.z * fh_silu_f(g[j].z), v.w * fh_silu_f(g[j].w));
                if (i >= inner) v.x = v.y = v.z = v.w = 0.f;
                if (i < st.kpo) in.quad(q) = v;
            }
        } else {
            for (int i = tid; i < inner; i += 512) {
                float v = in.at(i) * ginv[i / gl] * rc.norm[rc.norm_len == inner ? i : i % rc.norm_len];
                if (!gate_first) v *= fh_silu_f(gate[i]);
                in.at(i) = v;
            }
        }
        fh_lds_barrier();
    }
    float acc = 0.f;
    for (int i = 0; i < count;) {
#pragma unroll
        for (int s = 0; s < AHEAD; s++) {
            const bool in_row = now.k + lane8 < now.kp;
            const float *at = in.xs + ((now.from + now.k) >> 1) + (in_row ? lane * 4 : 0);
            const float more = fh_dot8(u[s], *(const float4 *)at, *(const float4 *)(at + in.plane), acc);
            acc = in_row ? more : acc;
            fetch(s);
            if (advance(now)) {
                acc = fh_wave_sum(acc);
                if (i < count && lane == 0) st.x[first + i * step] += acc;
                acc = 0.f, i++;
            }
        }
    }
}

fh_status fh_step_out(fh_device *dev, const FhStep &st) {
    const FhMoe &m = st.moe;
    const int n_e = m.experts ? m.top : 0, n_s = m.sff ? m.sffp : 0;
    const bool recurrent = st.kind == FH_MIX_RECURRENT;
    const size_t need = (size_t)(st.kpo + n_e * m.ffp + n_s + (recurrent ? (st.rec.norm_groups + 3) / 4 * 4 : 0) + n_e) * 4;
    FH_REQUIRE(need <= 156 * 1024, "a decode step stages at most 156 KB of inputs (%zu bytes needed)", need);
    const int inner = recurrent ? st.rec.heads * st.rec.vdim : st.lat.heads * st.lat.dv;
    bool quads = inner % 4 == 0 && need + st.kpo <= 156 * 1024 && ((uintptr_t)st.o & 15) == 0;
    if (recurrent) quads = quads && inner / st.rec.norm_groups % 4 == 0 && st.rec.norm_len % 4 == 0 && ((uintptr_t)(st.proj + st.rec.col_g) & 15) == 0;
    const dim3 grid((unsigned)std::min(dev->compute_units, (st.width + 7) / 8));
#define STEP_OUT(NO_, NE_, NS_, PRE_)                                                                                         \
    do {                                                                                                                      \
        const size_t lds = need + (NO_ && recurrent ? st.kpo : 0);                                                            \
        if (lds > 48 * 1024) FH_TRY(fh_kernel_lds(dev, (const void *)k_step_out<NO_, NE_, NS_, PRE_>, lds));                  \
        k_step_out<NO_, NE_, NS_, PRE_><<<grid, 512, lds, dev->stream>>>(st);                                                 \
    } while (0)
    if (!quads || st.kpo > 8192 || n_e * m.ffp > 8192 || n_s > 2048) STEP_OUT(0, 1, 1, false);
    else if (st.kpo <= 1536 && n_e * m.ffp <= 2048) STEP_OUT(1, 1, 1, false);
    else if (st.kpo <= 1536) STEP_OUT(1, 4, 1, false);
    else if (st.kpo <= 2048 && n_e * m.ffp <= 4096) STEP_OUT(1, 2, 1, true);
    else if (st.kpo <= 4096) STEP_OUT(2, 4, 1, true);
    else STEP_OUT(4, 4, 1, true);
#undef STEP_OUT
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// ------------------------------------------------------------------------------ mixers of sublayers normed at their end
// RPT consecutive values from i0 on, those past d repeat the last one.
template <int RPT>
__device__ __forceinline__ void rec_load(float *v, const float *p, int i0, int d, bool full) {
    constexpr int N = RPT < 4 ? RPT : 4;
    if (full) {
#pragma unroll
        for (int i = 0; i < RPT; i += N) __builtin_memcpy(v + i, p + i0 + i, N * 4);
    } else {
#pragma unroll
        for (int i = 0; i < RPT; i++) v[i] = p[i0 + i < d ? i0 + i : d - 1];
    }
}

// One step of a recurrence without a short convolution: workgroup b takes 16 columns of one head's state.
template <int RPT>
__device__ __forceinline__ void linear_step(const FhMixStep &st, int pos, int b, float *lds) {
    const FhRecurrent &r = st.r;
    const int tid = threadIdx.x, lane = tid & 63, rg = lane & 15, d = r.dim;
    const int ncb = (r.vdim + 15) / 16, h = b / ncb, col = b % ncb * 16 + (tid >> 4), i0 = rg * RPT;
    const bool live = col < r.vdim;
    float *sp = st.state.s + ((int64_t)h * r.vdim + (live ? col : r.vdim - 1)) * d;
    float S[RPT];
    const bool full = d == 16 * RPT; // whole rows in float4s
    rec_load<RPT>(S, sp, i0, d, full);
#pragma unroll
    for (int i = 0; i < RPT; i++) S[i] = pos > 0 ? S[i] : 0.f;
    const float *q = st.proj + r.col_q + h * d, *k = st.proj + r.col_k + h * d;
    const float v = st.proj[r.col_v + h * r.vdim + (live ? col : r.vdim - 1)];
    float o = 0.f;
    if (r.kind == FH_REC_CHANNEL) {
        float *g = lds, *t1 = lds + 256; // [d], [rp]
        // every request goes out before the first wait
        uint4 w2[RPT];
        float kk[RPT], qq[RPT], uu[RPT], w0[RPT];
#pragma unroll
        for (int i = 0; i < RPT; i++) { // the 16 lanes of a DPP row share a channel: 16 i + tid / 16
            const int c = 16 * i + (tid >> 4);
            const int64_t cc = h * d + (c < d ? c : d - 1);
            w2[i] = *(const uint4 *)(r.w2 + cc * r.rp + (rg * 8 < r.rp ? rg * 8 : 0));
            w0[i] = r.w0[cc];
        }
        rec_load<RPT>(kk, k, i0, d, full);
        rec_load<RPT>(qq, q, i0, d, full);
        rec_load<RPT>(uu, r.bonus + h * d, i0, d, full);
#pragma unroll
        for (int i = 0; i < RPT; i++) // rows past the end read nothing out
            if (i0 + i >= d) kk[i] = 0.f, qq[i] = 0.f;
        for (int i = tid; i < r.rp; i += 256) t1[i] = i < r.rank ? st.proj[r.col_a + i] : 0.f;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            const int c = 16 * i + (tid >> 4);
            float z = rg * 8 < r.rp ? fh_dot8(w2[i], *(const float4 *)(t1 + rg * 8), *(const float4 *)(t1 + rg * 8 + 4), 0.f) : 0.f;
            if (c < d)
                for (int x = rg * 8 + 128; x < r.rp; x += 128) z = fh_dot8(*(const uint4 *)(r.w2 + (int64_t)(h * d + c) * r.rp + x), *(const float4 *)(t1 + x), *(const float4 *)(t1 + x + 4), z);
            z = fh_row16_sum(z);
            if (rg == 0 && c < d) g[c] = expf(fh_rec_la(z + w0[i]));
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            const float kv = kk[i] * v;
            o = fmaf(fmaf(uu[i], kv, S[i]), qq[i], o);
            S[i] = fmaf(S[i], g[i0 + i], kv);
        }
    } else {
        const float g = expf(r.log_decay[h]), *ct = r.cos_t + (int64_t)pos * r.pairs, *sn = r.sin_t + (int64_t)pos * r.pairs;
        float *qk = lds; // [2][16 RPT], zeros from d on
        for (int i = tid; i < 32 * RPT; i += 256) {
            const bool key = i >= 16 * RPT;
            const int c0 = i % (16 * RPT), c = c0 < d ? c0 : d - 1, p = r.halves ? c < r.pairs ? c : c - r.pairs : c >> 1;
            const bool second = r.halves ? c >= r.pairs : c & 1, turn = c < 2 * r.pairs;
            const float *x = key ? k : q;
            const float y = x[c], z = x[!turn ? c : !r.halves ? c ^ 1 : second ? c - r.pairs : c + r.pairs];
            const float co = ct[turn ? p : 0], si = sn[turn ? p : 0];
            qk[i] = c0 < d ? (turn ? y * co + (second ? z * si : -z * si) : y) * (key ? r.k_scale : r.q_scale) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            S[i] = fmaf(qk[16 * RPT + i0 + i], v, S[i] * g);
            o = fmaf(S[i], qk[i0 + i], o);
        }
    }
    o = fh_row16_sum(o);
    if (!live) return;
    if (full)
#pragma unroll
        for (int i = 0; i < RPT; i += RPT < 4 ? RPT : 4) __builtin_memcpy(sp + i0 + i, S + i, (RPT < 4 ? RPT : 4) * 4);
    else
        for (int i = 0; i < RPT; i++)
            if (i0 + i < d) sp[i0 + i] = S[i];
    if (rg == 0) st.o[h * r.vdim + col] = o;
}

template <typename T, int NP, int RPT>
__global__ __launch_bounds__(256) void k_step_mixers(FhMixStep st, T *ring, int cap, int splits, int n_attn) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int pos = *st.pos_dev;
    if ((int)blockIdx.x < n_attn) fh_gqa_step<T, NP>(st.gqa, st.proj, ring, cap, pos, splits, blockIdx.x, st.part, lds);
    else linear_step<RPT>(st, pos, (int)blockIdx.x - n_attn, lds);
}

template <typename T, int NP>
static fh_status step_mixers_t(fh_device *dev, const FhMixStep &st, fh_kvcache *cache) {
    const int splits = st.attn ? fh_gqa_splits(cache) : 1, n_attn = st.attn ? fh_gqa_blocks(st.gqa, splits) : 0;
    const int n_rec = st.rec ? st.r.heads * ((st.r.vdim + 15) / 16) : 0, rpt = st.rec ? (st.r.dim + 15) / 16 : 1;
    size_t lds = st.attn ? fh_gqa_lds(st.gqa) : 0;
    const size_t need = !st.rec ? 0 : (size_t)(st.r.kind == FH_REC_CHANNEL ? 256 + st.r.rp : 512) * 4;
    lds = lds > need ? lds : need;
    FH_REQUIRE(lds <= 60 * 1024 && rpt <= 16, "mixers too wide for a decode step (%zu bytes of LDS)", lds);
    const dim3 grid((unsigned)(n_attn + n_rec));
    T *ring = cache ? (T *)cache->k : nullptr;
    const int cap = cache ? cache->capacity : 1;
    if (rpt <= 2) k_step_mixers<T, NP, 2><<<grid, 256, lds, dev->stream>>>(st, ring, cap, splits, n_attn);
    else if (rpt <= 4) k_step_mixers<T, NP, 4><<<grid, 256, lds, dev->stream>>>(st, ring, cap, splits, n_attn);
    else if (rpt <= 8) k_step_mixers<T, NP, 8><<<grid, 256, lds, dev->stream>>>(st, ring, cap, splits, n_attn);
    else k_step_mixers<T, NP, 16><<<grid, 256, lds, dev->stream>>>(st, ring, cap, splits, n_attn);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

fh_status fh_step_mixers(fh_device *dev, int dtype, const FhMixStep &st, fh_kvcache *cache) {
    FH_REQUIRE(!st.attn || (cache && st.gqa.dnp <= 256 && st.gqa.dvp <= 256), "attention heads of a decode step have at most 256 dimensions");
    const bool one = !st.attn || (st.gqa.dnp <= 128 && st.gqa.dvp <= 128);
    if (dtype == FH_F32) return one ? step_mixers_t<float, 1>(dev, st, cache) : step_mixers_t<float, 2>(dev, st, cache);
    return one ? step_mixers_t<uint16_t, 1>(dev, st, cache) : step_mixers_t<uint16_t, 2>(dev, st, cache);
}

// One wavefront per attention head, then one per norm group of the recurrence.
__global__ __launch_bounds__(64) void k_step_mix_out(FhMixStep st, int splits) {
    const int lane = threadIdx.x, na = st.attn ? st.gqa.heads : 0, b = blockIdx.x;
    if (b < na) {
        const FhGqa &a = st.gqa;
        fh_gqa_merge(a, st.part, splits, b, st.act + b * a.vdim);
        if (b == na - 1)
            for (int i = a.heads * a.vdim + lane; i < st.kpl; i += 64) st.act[i] = 0.f;
        return;
    }
    const FhRecurrent &r = st.r;
    const int g = b - na, inner = r.heads * r.vdim, gl = inner / r.norm_groups;
    const float *o = st.o + g * gl, *gate = st.proj + r.col_g + g * gl;
    float ss = 0.f;
    for (int i = lane; i < gl; i += 64) ss = fmaf(o[i], o[i], ss);
    const float inv = 1.0f / sqrtf(fh_wave_sum(ss) / (float)gl + r.eps);
    for (int i = lane; i < gl; i += 64) {
        float v = o[i] * inv;
        if (r.norm) v *= r.norm[r.norm_len == inner ? g * gl + i : i % r.norm_len];
        st.act[st.kpl + g * gl + i] = v * fh_silu_f(gate[i]) * r.out_scale;
    }
}

fh_status fh_step_mix_out(fh_device *dev, const FhMixStep &st, const fh_kvcache *cache) {
    FH_REQUIRE(!st.rec || !st.r.gate_first, "this step gates behind the norm");
    const int blocks = (st.attn ? st.gqa.heads : 0) + (st.rec ? st.r.norm_groups : 0);
    k_step_mix_out<<<dim3((unsigned)blocks), 64, 0, dev->stream>>>(st, st.attn ? fh_gqa_splits(cache) : 1);
    FH_HIP(hipGetLastError());
    return FH_OK;
}
