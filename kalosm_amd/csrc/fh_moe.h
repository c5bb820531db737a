// Mixture-of-experts feed-forward: softmax router, the `top` best experts of a token weighted by scale times their score,
// and optionally one more expert that is always on.  Expert weights are stacked: gate | up rows in
// alternating groups of 16, [experts][2 ffp][kp], and down [experts][dp][ffp], with ffp = ff rounded up to 64 (zero rows)
// and dp = the width rounded up to 16.
#pragma once
#include "fh_dense.h"

enum { FH_MOE_MAX_EXPERTS = 1024 };
struct FhMoe {
    int experts = 0, top = 0, ff = 0, ffp = 0;   // experts 0: no routed part
    float scale = 1.f;
    int col_z = 0;                               // router logits in a projection row
    const uint16_t *gate_up = nullptr, *down = nullptr;
    int64_t gu_stride = 0, down_stride = 0;      // elements per expert
    int sff = 0, sffp = 0;                       // the always-on expert (0: none)
    const uint16_t *s_gate_up = nullptr, *s_down = nullptr;
};
// Work arrays of a prefill portion.
struct FhMoeWork {
    int *ids;       // [t, top] chosen experts
    float *wts;     // [t, top]
    int *src;       // [t * top] token behind a sorted assignment
    int *inv;       // [t, top] sorted place of an assignment
    FhTile *tiles;  // fh_moe_max_tiles
    int *n_tiles;
    void *act;      // [t * top, ffp] activation rows
    float *y;       // [t * top, width]
    void *s_act;    // [t, sffp]
    float *s_y;     // [t, width]
};
// rows per tile: the larger ones where an expert has rows to fill them on average.  Of more than 128 rows an expert is one tile of up to
// 320, so that its weights cross into the LDS once; with fewer there is nothing to save, and with few tiles the compute units
// share out better by 128.  32 experts of 4096 x 4096 / 4096 x 2048, top 4, tiles of 320 (and of 128): 1800 tokens 281 / 177 us (331 / 193),
// 1300 tokens 250 / 161 (282 / 176), 1000 tokens 236 / 153 (243 / 148).
static inline int fh_moe_tile_rows(const fh_device *dev, const FhMoe &m, int dtype, int s, int width) {
    const int64_t opt = dev->opt_matmul_kernel, rows = (int64_t)s * m.top, narrow = 2 * m.ffp < width ? 2 * m.ffp : width;
    const bool tall = rows >= (int64_t)m.experts * 144 && m.experts * ((narrow + 255) / 256) >= dev->compute_units;
    if (dtype != FH_F32 && opt != 3 && opt != 14 && (opt == 4 || tall)) return 320;
    return dtype != FH_F32 && rows >= (int64_t)m.experts * 96 ? 128 : 64;
}
static inline int fh_moe_max_tiles(const FhMoe &m, int s, int tile_rows) { return s * m.top / tile_rows + m.experts; }
// x [s, width] += mix [s, width] + the feed-forward of the activation rows h [s, kp]
fh_status fh_moe_prefill(fh_device *dev, int dtype, const FhMoe &m, const void *h, int kp, const float *proj, int64_t ldp,
                         int s, int width, const FhMoeWork &w, const float *mix, float *x);

#ifdef __HIPCC__
// The n-th best expert of one token and its weight, for all n < count, by one wavefront: every lane keeps the logits
// e = lane + 64 i, i < PER.  Ties go to the smaller index.  pick(n, expert, weight) runs in every lane.
template <int PER, typename F>
__device__ __forceinline__ void fh_moe_route_per(const float *z, int experts, float scale, int count, F pick) {
    const int lane = threadIdx.x & 63;
    float v[PER];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int e = lane + 64 * i;
        v[i] = z[e < experts ? e : 0];
        v[i] = e < experts ? v[i] : -INFINITY;
        mx = fmaxf(mx, v[i]);
    }
    mx = fh_wave_max(mx);
    float den = 0.f;
#pragma unroll
    for (int i = 0; i < PER; i++) den += v[i] == -INFINITY ? 0.f : expf(v[i] - mx);
    den = fh_wave_sum(den);
    float best = mx;
    for (int n = 0; n < count; n++) {
        int e = -1; // of those with the best logit the first
#pragma unroll
        for (int i = PER - 1; i >= 0; i--) {
            const uint64_t who = __ballot(v[i] == best);
            e = who ? 64 * i + __builtin_ctzll(who) : e;
        }
        if (e < 0 || best == -INFINITY) e = 0; // only when no logit is a number
        pick(n, e, expf(best - mx) / den * scale);
        best = -INFINITY;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            v[i] = e == lane + 64 * i ? -INFINITY : v[i];
            best = fmaxf(best, v[i]);
        }
        best = fh_wave_max(best);
    }
}
template <typename F>
__device__ __forceinline__ void fh_moe_route(const float *z, int experts, float scale, int count, F pick) {
    if (experts <= 64) fh_moe_route_per<1>(z, experts, scale, count, pick);
    else if (experts <= 256) fh_moe_route_per<4>(z, experts, scale, count, pick);
    else fh_moe_route_per<FH_MOE_MAX_EXPERTS / 64>(z, experts, scale, count, pick);
}
#endif
