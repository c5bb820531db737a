// Dense bf16 weights: prefill products on the matrix cores (plain and grouped by expert), the decode matvec with the
// RMS norm of its input, and the norm that writes activation rows.
#include "fh_dense.h"
#include <type_traits>

// ------------------------------------------------------------------------------ prefill product
// y[m, n] = x[m, :] . W[n, :].  The weights are the A operand (accumulator rows), the activations the B operand
// (accumulator columns), so a lane holds four neighbouring outputs of one activation row; for the transposed output the
// operands change places and a lane holds four neighbouring activation rows of one output.
//
// bf16: 128 weight rows x BM activation rows per workgroup, four wavefronts, 64 of k per step.  Both operands go from
// memory straight into the LDS (LDS-direct loads, double buffered, one barrier per step).  An LDS row is 128 bytes =
// eight 16-byte pieces; piece c of row r sits at position c ^ ((r / 2) % 8), so that the 16 rows an operand read touches
// at one c cover the 64 banks once.  The swizzle is applied on the memory side of the loads.
template <int EPI, typename T>
__device__ __forceinline__ void gemm_store(void *y, int64_t ldy, int m_row, int n_row, const fh_f4 &v, int m, int n) {
    // EPI F32 / ACT: outputs n_row .. n_row + 3 of row m_row.  ACT_T: rows m_row .. m_row + 3 of output n_row.
    if (EPI == FH_GEMM_ACT_T) {
        if (n_row >= n) return;
        T *p = (T *)y + (int64_t)n_row * ldy + m_row;
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (m_row + r < m) p[r] = fh_to<T>(v[r]);
        return;
    }
    if (m_row >= m) return;
    if (EPI == FH_GEMM_F32) {
        float *p = (float *)y + (int64_t)m_row * ldy + n_row;
        if (n_row + 3 < n && (ldy & 3) == 0) *(float4 *)p = make_float4(v[0], v[1], v[2], v[3]);
        else
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (n_row + r < n) p[r] = v[r];
    } else {
        T *p = (T *)y + (int64_t)m_row * ldy + n_row;
        T t[4];
#pragma unroll
        for (int r = 0; r < 4; r++) t[r] = fh_to<T>(v[r]);
        if (n_row + 3 < n && (ldy & 3) == 0) {
            struct alignas(4 * sizeof(T)) V4 { T t[4]; };
            *(V4 *)p = V4{{t[0], t[1], t[2], t[3]}};
        } else
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (n_row + r < n) p[r] = t[r];
    }
}

__device__ __forceinline__ fh_f4 relu2(fh_f4 v) {
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = fmaxf(v[e], 0.f) * fmaxf(v[e], 0.f);
    return v;
}

__device__ __forceinline__ int gemm_sw(int row) { return (row >> 1) & 7; }

template <int BM, int EPI>
__global__ __launch_bounds__(256) void k_gemm_bf16(FhGemm g) {
    constexpr int BN = 128, LDK = 64;
    constexpr int WM = BM >= 128 ? 2 : 1, WN = 4 / WM;        // wavefronts along m and n
    constexpr int FN = BN / WN / 16, FM = BM / WM / 16;       // 16 x 16 tiles of a wavefront
    constexpr int BUF = (BN + BM) * LDK;
    __shared__ __attribute__((aligned(16))) uint16_t smem[2 * BUF];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wn = wave / WM, wm = wave % WM, li = lane & 15, gq = lane >> 4;
    int row0, m_end;
    const uint16_t *w = g.w;
    if (g.tiles) {
        if ((int)blockIdx.y >= *g.n_tiles) return;
        const FhTile t = g.tiles[blockIdx.y];
        row0 = t.row0;
        m_end = t.row0 + t.rows;
        w += (int64_t)t.group * g.w_group;
    } else {
        row0 = (int)blockIdx.y * BM;
        m_end = g.m;
    }
    const int n0 = (int)blockIdx.x * BN;
    const uint16_t *x = (const uint16_t *)g.x;
    // LDS-direct loads: a wavefront's request fills eight rows; lane l supplies row l / 8, position l % 8
    constexpr int NL_W = BN / 32, NL_X = BM / 32;
    const uint16_t *wp[NL_W], *xp[NL_X];
    const int rl = tid >> 3, pos = tid & 7;
#pragma unroll
    for (int i = 0; i < NL_W; i++) {
        const int r = rl + 32 * i, n = n0 + r < g.n ? n0 + r : g.n - 1; // rows past the end repeat the last one, never stored
        wp[i] = w + (int64_t)n * g.kp + (pos ^ gemm_sw(r)) * 8;
    }
#pragma unroll
    for (int i = 0; i < NL_X; i++) {
        const int r = rl + 32 * i;
        int m = row0 + r < m_end ? row0 + r : m_end - 1;
        if (g.gather) m = g.gather[m];
        xp[i] = x + (int64_t)m * g.kp + (pos ^ gemm_sw(r)) * 8;
    }
    auto fetch = [&](int ks) {
        uint16_t *dst = smem + (ks & 1) * BUF + wave * 8 * LDK;
#pragma unroll
        for (int i = 0; i < NL_W; i++)
            __builtin_amdgcn_global_load_lds((const uint32_t *)(wp[i] + ks * 64),
                                             (__attribute__((address_space(3))) uint32_t *)(dst + i * 32 * LDK), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < NL_X; i++)
            __builtin_amdgcn_global_load_lds((const uint32_t *)(xp[i] + ks * 64),
                                             (__attribute__((address_space(3))) uint32_t *)(dst + (BN + i * 32) * LDK), 16, 0, 0);
    };
    fh_f4 acc[FN][FM];
#pragma unroll
    for (int a = 0; a < FN; a++)
#pragma unroll
        for (int b = 0; b < FM; b++) acc[a][b] = fh_f4{0.f, 0.f, 0.f, 0.f};
    const int steps = g.kp / 64;
    fetch(0);
    for (int ks = 0; ks < steps; ks++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // this wavefront's pieces of step ks have landed
        __syncthreads();                                  // everybody's have, and nobody reads the other buffer any more
        if (ks + 1 < steps) fetch(ks + 1);
        const uint16_t *bw = smem + (ks & 1) * BUF, *bx = bw + BN * LDK;
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            fh_bf8 fw[FN], fx[FM];
#pragma unroll
            for (int a = 0; a < FN; a++) {
                const int r = wn * FN * 16 + a * 16 + li;
                fh_frag_load(fw[a], bw + r * LDK + ((kk * 4 + gq) ^ gemm_sw(r)) * 8);
            }
#pragma unroll
            for (int b = 0; b < FM; b++) {
                const int r = wm * FM * 16 + b * 16 + li;
                fh_frag_load(fx[b], bx + r * LDK + ((kk * 4 + gq) ^ gemm_sw(r)) * 8);
            }
#pragma unroll
            for (int a = 0; a < FN; a++)
#pragma unroll
                for (int b = 0; b < FM; b++)
                    acc[a][b] = EPI == FH_GEMM_ACT_T ? fh_mma32(fx[b], fw[a], acc[a][b]) : fh_mma32(fw[a], fx[b], acc[a][b]);
        }
    }
#pragma unroll
    for (int b = 0; b < FM; b++) {
#pragma unroll
        for (int a = 0; a < FN; a += EPI == FH_GEMM_SWIGLU ? 2 : 1) {
            const int nb = n0 + wn * FN * 16 + a * 16, mb = row0 + wm * FM * 16 + b * 16;
            if (EPI == FH_GEMM_SWIGLU) {
                fh_f4 v;
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = fh_silu_f(acc[a][b][r]) * acc[a + 1 < FN ? a + 1 : a][b][r];
                gemm_store<FH_GEMM_ACT, uint16_t>(g.y, g.ldy, mb + li, nb / 2 + gq * 4, v, m_end, g.n / 2);
            } else if (EPI == FH_GEMM_RELU2) {
                gemm_store<FH_GEMM_ACT, uint16_t>(g.y, g.ldy, mb + li, nb + gq * 4, relu2(acc[a][b]), m_end, g.n);
            } else if (EPI == FH_GEMM_ACT_T) {
                gemm_store<EPI, uint16_t>(g.y, g.ldy, mb + gq * 4, nb + li, acc[a][b], m_end, g.n);
            } else {
                gemm_store<EPI, uint16_t>(g.y, g.ldy, mb + li, nb + gq * 4, acc[a][b], m_end, g.n);
            }
        }
    }
}

// Large products: 256 weight rows x 256 or 128 activation rows per workgroup of eight wavefronts, on v_mfma_f32_32x32x16_bf16.
// What bounds the 128 x 128 kernel above is what a compute unit gets from its L2 - 32 KB per 64 of k and 128 x 128 outputs, 78 B/ns
// at the rate of the matrix cores - and that every step waits for the step just requested.  256 x 256 halves the bytes, and
// the clock, which the matrix cores bring down to 1.7 GHz, becomes the bound: 2048 x 14336 x 4096 in 231 us (1.04 PFLOP/s, 331 us
// before), 2048 x 4096 x 14336 with 128 rows per tile in 211 us (1.14 PFLOP/s).  Products grouped by expert: 32 experts of 4096 x 4096 and
// 8192 rows 305 us with tiles of up to 320 rows where no expert has more, 364 over uneven ones (382 with 128 rows; reading 1.07 GB takes 230 us).  Their
// row tiles are of any height: a wavefront multiplies only the 32-column tiles that have rows (without that, and with a weight tile's row tiles
// on several dies, the 128-row form took 447), and the two wavefronts of a SIMD take the two halves of the columns.
// 64 of k (a slab) per barrier; the barrier sits ahead of the slab's last quarter, whose operands are in registers already, so
// the next slab's first operands are read and the requests of the slab after it go out while that quarter is multiplied.
// SLABS buffers: two of 64 KB, three of 48 KB with 128 activation rows (fewer rows), or two of 72 KB with up to 320 (groups of rows).
template <int TX>
struct WideTile {
    static constexpr int TW = 256, WGX = TX == 256 ? 4 : 2, FW = TX == 256 ? 4 : 2, FX = TX / 32 / WGX; // a wavefront: FW x FX tiles of 32 x 32
    static constexpr int NLW = TW / 64, NLX = TX / 64, NL = NLW + NLX;                                  // requests of a wavefront per slab
    static constexpr int SLAB = (TW + TX) * 128, SLABS = TX == 128 ? 3 : 2;
    static constexpr bool COUNT_VARIES = TX == 320; // rows that are not there are not requested: two slabs, of which none may be on its way
};

template <int TX, int EPI>
__global__ __launch_bounds__(512) void k_gemm_bf16_wide(FhGemm g) {
    typedef WideTile<TX> Tile;
    typedef float f16v __attribute__((ext_vector_type(16)));
    constexpr int TW = Tile::TW, WGX = Tile::WGX, FW = Tile::FW, FX = Tile::FX, SLAB = Tile::SLAB, SLABS = Tile::SLABS;
    constexpr bool W_ROWS = EPI == FH_GEMM_SWIGLU || EPI == FH_GEMM_ACT_T; // weight rows along the registers of the result, else along its lanes
    extern __shared__ __attribute__((aligned(16))) uint8_t wide_smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 31;
    constexpr int WGW = 8 / WGX;
    const int ww = wave % WGW, wx = wave / WGW;
    // The eight dies take runs of tiles.  Without groups: eight weight tiles by all row tiles, weight tiles first.  With groups: up
    // to eight row tiles of a group by all weight tiles, row tiles first, so that they read a weight tile from one die's L2 together.
    const int tn = (g.n + TW - 1) / TW, die = (int)blockIdx.x & 7, idx = (int)blockIdx.x >> 3;
    int row0, m_end, n0;
    const uint16_t *w = g.w;
    if (g.tiles) {
        const int total = *g.n_tiles * tn, per = total >> 3, more = total & 7;
        if (idx >= per + (die < more ? 1 : 0)) return;
        const int lin = idx + die * per + (die < more ? die : more), i = lin / tn;
        const int of = g.tiles[i].of, at = g.tiles[i].at, l = lin - (i - at) * tn;
        const FhTile t = g.tiles[i - at + l % of];
        n0 = l / of * TW;
        row0 = t.row0;
        m_end = t.row0 + t.rows;
        w += (int64_t)t.group * g.w_group;
    } else {
        const int ty = (g.m + TX - 1) / TX, total = tn * ty, per = total >> 3, more = total & 7;
        if (idx >= per + (die < more ? 1 : 0)) return;
        const int lin = idx + die * per + (die < more ? die : more);
        const int grp = lin / (8 * ty), in = lin - grp * 8 * ty, gw = tn - grp * 8 < 8 ? tn - grp * 8 : 8;
        n0 = (grp * 8 + in % gw) * TW;
        row0 = in / gw * TX;
        m_end = g.m;
    }
    // LDS-direct loads: a wavefront's request fills eight rows of 128 bytes; lane l supplies row l / 8, position l % 8 (swizzle
    // as above, on the memory side)
    const uint16_t *wp[Tile::NLW], *xp[Tile::NLX];
    const int rl = tid >> 3, piece = ((tid & 7) ^ gemm_sw(rl)) * 8;
#pragma unroll
    for (int i = 0; i < Tile::NLW; i++) {
        const int n = n0 + rl + 64 * i < g.n ? n0 + rl + 64 * i : g.n - 1; // rows past the end repeat the last one, never stored
        wp[i] = w + (int64_t)n * g.kp + piece;
    }
#pragma unroll
    for (int i = 0; i < Tile::NLX; i++) {
        int m = row0 + rl + 64 * i < m_end ? row0 + rl + 64 * i : m_end - 1;
        if (g.gather) m = g.gather[m];
        xp[i] = (const uint16_t *)g.x + (int64_t)m * g.kp + piece;
    }
    // the 32-column tiles that have rows; with two wavefronts along them they are shared out evenly
    const int cols = m_end - row0 < TX ? (m_end - row0 + 31) / 32 : TX / 32;
    const int c0 = WGX > 2 ? wx * FX : wx ? (cols + 1) / 2 : 0, mine = WGX > 2 ? cols - c0 < FX ? cols - c0 : FX : wx ? cols / 2 : (cols + 1) / 2;
    const int slabs = g.kp / 64;
    auto fetch = [&](int s, int at) { // slab s into the buffer at byte `at`; past the end a repeat, so that the counts stay equal
        const int64_t o = (int64_t)(s < slabs ? s : slabs - 1) * 64;
        uint8_t *dst = wide_smem + at + wave * 1024;
#pragma unroll
        for (int i = 0; i < Tile::NLW; i++)
            __builtin_amdgcn_global_load_lds((const uint32_t *)(wp[i] + o),
                                             (__attribute__((address_space(3))) uint32_t *)(dst + i * 8192), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < Tile::NLX; i++)
            if (!Tile::COUNT_VARIES || i * 2 < cols) __builtin_amdgcn_global_load_lds((const uint32_t *)(xp[i] + o),
                                             (__attribute__((address_space(3))) uint32_t *)(dst + (Tile::NLW + i) * 8192), 16, 0, 0);
    };
    const int sw = gemm_sw(li), rw = (ww * FW * 32 + li) * 128, rx = (TW + c0 * 32 + li) * 128; // (tiles start at multiples of 32 rows)
    f16v acc[FW][FX];
#pragma unroll
    for (int a = 0; a < FW; a++)
#pragma unroll
        for (int c = 0; c < FX; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][c][r] = 0.f;
#pragma unroll
    for (int i = 0; i < SLABS; i++) fetch(i, i * SLAB);
    auto all = [&](auto have) { // so many of the wavefront's FX column tiles; the barriers are the same ones for every number
        constexpr int C = decltype(have)::value;
        fh_bf8 fw[2][FW], fx[2][FX];
        auto read = [&](int set, int at, int q) { // quarter q (16 of k) of the slab at byte `at`
            if (!C) return;
            const uint8_t *b = wide_smem + at + ((2 * q + (lane >> 5)) ^ sw) * 16;
#pragma unroll
            for (int a = 0; a < FW; a++) fw[set][a] = *(const fh_bf8 *)(b + rw + a * 4096);
#pragma unroll
            for (int c = 0; c < C; c++) fx[set][c] = *(const fh_bf8 *)(b + rx + c * 4096);
        };
        auto mul = [&](int set) {
#pragma unroll
            for (int a = 0; a < FW; a++)
#pragma unroll
                for (int c = 0; c < C; c++)
                    acc[a][c] = W_ROWS ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[set][a], fx[set][c], acc[a][c], 0, 0, 0)
                                       : __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[set][c], fw[set][a], acc[a][c], 0, 0, 0);
        };
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Tile::COUNT_VARIES ? 0 : (SLABS - 1) * Tile::NL) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read(0, 0, 0);
        int cur = 0;
        for (int s = 0; s < slabs; s++) {
            const int nxt = cur + SLAB == SLABS * SLAB ? 0 : cur + SLAB;
            read(1, cur, 1);
            mul(0);
            __builtin_amdgcn_sched_barrier(0);
            read(0, cur, 2);
            mul(1);
            __builtin_amdgcn_sched_barrier(0);
            read(1, cur, 3);
            mul(0);
            __builtin_amdgcn_sched_barrier(0);
            // the last quarter's operands are here: this wavefront is done with the slab's buffer; and slab s + 1 has landed
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((SLABS - 2) * Tile::NL) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            read(0, nxt, 0);
            fetch(s + SLABS, cur);
            mul(1);
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
        }
    };
    if (mine >= FX) all(std::integral_constant<int, FX>{});
    else if (FX > 4 && mine == 4) all(std::integral_constant<int, (FX > 4 ? 4 : 0)>{});
    else if (FX > 3 && mine == 3) all(std::integral_constant<int, (FX > 3 ? 3 : 0)>{});
    else if (FX > 2 && mine == 2) all(std::integral_constant<int, (FX > 2 ? 2 : 0)>{});
    else if (mine == 1) all(std::integral_constant<int, 1>{});
    else all(std::integral_constant<int, 0>{}); // its requests only
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // no LDS-direct load outlives the workgroup's LDS
    const int nb = n0 + ww * FW * 32, mb = row0 + c0 * 32, h4 = 4 * (lane >> 5);
#pragma unroll
    for (int a = 0; a < FW; a++)
#pragma unroll
        for (int c = 0; c < FX; c++) {
            if (c >= mine) break;
            if (EPI == FH_GEMM_SWIGLU) { // rows 0 .. 15 of a tile are gates, 16 .. 31 the same outputs' up rows
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    fh_f4 v;
#pragma unroll
                    for (int r = 0; r < 4; r++) v[r] = fh_silu_f(acc[a][c][4 * q + r]) * acc[a][c][8 + 4 * q + r];
                    gemm_store<FH_GEMM_ACT, uint16_t>(g.y, g.ldy, mb + c * 32 + li, (nb + a * 32) / 2 + 8 * q + h4, v, m_end, g.n / 2);
                }
            } else {
                const int nl = nb + a * 32, ml = mb + c * 32;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int o = 8 * (r >> 2) + h4 + (r & 3);
                    const int n = W_ROWS ? nl + o : nl + li, m = W_ROWS ? ml + li : ml + o;
                    if (n >= g.n || m >= m_end) continue;
                    const float v = acc[a][c][r];
                    if (EPI == FH_GEMM_F32) ((float *)g.y)[(int64_t)m * g.ldy + n] = v;
                    else if (EPI == FH_GEMM_ACT_T) ((uint16_t *)g.y)[(int64_t)n * g.ldy + m] = fh_to<uint16_t>(v);
                    else if (EPI == FH_GEMM_RELU2) ((uint16_t *)g.y)[(int64_t)m * g.ldy + n] = fh_to<uint16_t>(fmaxf(v, 0.f) * fmaxf(v, 0.f));
                    else ((uint16_t *)g.y)[(int64_t)m * g.ldy + n] = fh_to<uint16_t>(v);
                }
            }
        }
}

template <int TX>
static fh_status gemm_wide(fh_device *dev, int epi, const FhGemm &g) {
    constexpr int LDS = WideTile<TX>::SLAB * WideTile<TX>::SLABS;
    const int64_t ty = g.tiles ? g.max_tiles : (g.m + TX - 1) / TX, total = (g.n + 255) / 256 * ty;
    FH_REQUIRE(total <= 0x7FFFFF00, "product too large for one launch");
    const dim3 grid((unsigned)((total + 7) / 8 * 8));
#define WIDE_GO(E_)                                                                           \
    do {                                                                                      \
        FH_TRY(fh_kernel_lds(dev, (const void *)k_gemm_bf16_wide<TX, E_>, (size_t)LDS));      \
        k_gemm_bf16_wide<TX, E_><<<grid, 512, LDS, dev->stream>>>(g);                         \
    } while (0)
    switch (epi) {
    case FH_GEMM_F32: WIDE_GO(FH_GEMM_F32); break;
    case FH_GEMM_ACT: WIDE_GO(FH_GEMM_ACT); break;
    case FH_GEMM_ACT_T: // (never grouped)
        if constexpr (TX != 320) WIDE_GO(FH_GEMM_ACT_T);
        break;
    case FH_GEMM_RELU2: WIDE_GO(FH_GEMM_RELU2); break;
    default: WIDE_GO(FH_GEMM_SWIGLU); break;
    }
#undef WIDE_GO
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// f32 activations: 64 x 64 outputs per workgroup, 32 of k per step, true f32 products (v_mfma_f32_16x16x4_f32) of the
// widened weights.
template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_f32(FhGemm g) {
    constexpr int BN = 64, BM = 64, LD = 36;
    __shared__ __attribute__((aligned(16))) float sw_[BN * LD], sx_[BM * LD];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, wn = wave >> 1, wm = wave & 1, li = lane & 15, gq = lane >> 4;
    int row0, m_end;
    const uint16_t *w = g.w;
    if (g.tiles) {
        if ((int)blockIdx.y >= *g.n_tiles) return;
        const FhTile t = g.tiles[blockIdx.y];
        row0 = t.row0;
        m_end = t.row0 + t.rows;
        w += (int64_t)t.group * g.w_group;
    } else {
        row0 = (int)blockIdx.y * BM;
        m_end = g.m;
    }
    const int n0 = (int)blockIdx.x * BN, r = tid >> 2, c = (tid & 3) * 8;
    const int n = n0 + r < g.n ? n0 + r : g.n - 1;
    int m = row0 + r < m_end ? row0 + r : m_end - 1;
    if (g.gather) m = g.gather[m];
    const uint16_t *wp = w + (int64_t)n * g.kp + c;
    const float *xp = (const float *)g.x + (int64_t)m * g.kp + c;
    fh_f4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) acc[a][b] = fh_f4{0.f, 0.f, 0.f, 0.f};
    uint4 rw = *(const uint4 *)wp;
    float4 rx0 = *(const float4 *)xp, rx1 = *(const float4 *)(xp + 4);
    for (int k = 0; k < g.kp; k += 32) {
        float *d = sw_ + r * LD + c;
        *(float4 *)d = make_float4(fh_bf_lo(rw.x), fh_bf_hi(rw.x), fh_bf_lo(rw.y), fh_bf_hi(rw.y));
        *(float4 *)(d + 4) = make_float4(fh_bf_lo(rw.z), fh_bf_hi(rw.z), fh_bf_lo(rw.w), fh_bf_hi(rw.w));
        *(float4 *)(sx_ + r * LD + c) = rx0;
        *(float4 *)(sx_ + r * LD + c + 4) = rx1;
        __syncthreads();
        if (k + 32 < g.kp) {
            rw = *(const uint4 *)(wp + k + 32);
            rx0 = *(const float4 *)(xp + k + 32);
            rx1 = *(const float4 *)(xp + k + 36);
        }
        fh_f8 fw[2], fx[2];
#pragma unroll
        for (int a = 0; a < 2; a++) {
            fh_frag_load(fw[a], sw_ + (wn * 32 + a * 16 + li) * LD + gq * 8);
            fh_frag_load(fx[a], sx_ + (wm * 32 + a * 16 + li) * LD + gq * 8);
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++)
                acc[a][b] = EPI == FH_GEMM_ACT_T ? fh_mma32(fx[b], fw[a], acc[a][b]) : fh_mma32(fw[a], fx[b], acc[a][b]);
        __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const int mb = row0 + wm * 32 + b * 16;
        if (EPI == FH_GEMM_SWIGLU) {
            fh_f4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = fh_silu_f(acc[0][b][e]) * acc[1][b][e];
            gemm_store<FH_GEMM_ACT, float>(g.y, g.ldy, mb + li, (n0 + wn * 32) / 2 + gq * 4, v, m_end, g.n / 2);
        } else {
#pragma unroll
            for (int a = 0; a < 2; a++) {
                const int nb = n0 + wn * 32 + a * 16;
                if (EPI == FH_GEMM_ACT_T) gemm_store<EPI, float>(g.y, g.ldy, mb + gq * 4, nb + li, acc[a][b], m_end, g.n);
                else if (EPI == FH_GEMM_RELU2) gemm_store<FH_GEMM_ACT, float>(g.y, g.ldy, mb + li, nb + gq * 4, relu2(acc[a][b]), m_end, g.n);
                else gemm_store<EPI, float>(g.y, g.ldy, mb + li, nb + gq * 4, acc[a][b], m_end, g.n);
            }
        }
    }
}

fh_status fh_gemm(fh_device *dev, int dtype, int epi, const FhGemm &g) {
    FH_REQUIRE(g.w && g.x && g.y && g.n > 0 && g.kp > 0 && g.kp % 64 == 0, "bad product");
    FH_REQUIRE(g.tiles ? g.max_tiles > 0 && g.n_tiles : g.m > 0, "product without rows");
    FH_REQUIRE(epi != FH_GEMM_SWIGLU || g.n % 32 == 0, "gate and up rows come in groups of 16");
    FH_REQUIRE(!g.tiles || g.tile_rows == 64 || (g.tile_rows >= 128 && g.tile_rows <= 320 && g.tile_rows % 32 == 0 && dtype != FH_F32), "row tiles of %d", g.tile_rows);
    FH_REQUIRE(epi != FH_GEMM_ACT_T || !g.tiles, "a grouped product has no transposed form");
    hipStream_t s = dev->stream;
#define FH_GEMM_EPI(K_, GRID_)                                              \
    switch (epi) {                                                          \
    case FH_GEMM_F32: K_(FH_GEMM_F32)<<<GRID_, 256, 0, s>>>(g); break;      \
    case FH_GEMM_ACT: K_(FH_GEMM_ACT)<<<GRID_, 256, 0, s>>>(g); break;      \
    case FH_GEMM_ACT_T: K_(FH_GEMM_ACT_T)<<<GRID_, 256, 0, s>>>(g); break;  \
    case FH_GEMM_RELU2: K_(FH_GEMM_RELU2)<<<GRID_, 256, 0, s>>>(g); break;  \
    default: K_(FH_GEMM_SWIGLU)<<<GRID_, 256, 0, s>>>(g); break;            \
    }
    if (dtype == FH_F32) {
        const int ty = g.tiles ? g.max_tiles : (g.m + 63) / 64;
        FH_REQUIRE(ty <= 65535, "too many rows for one launch");
        const dim3 grid((unsigned)((g.n + 63) / 64), (unsigned)ty);
#define FH_K_(E_) k_gemm_f32<E_>
        FH_GEMM_EPI(FH_K_, grid)
#undef FH_K_
    } else {
        const int64_t cus = dev->compute_units, wn = (g.n + 255) / 256;
        // The wide kernel from three quarters of a workgroup per compute unit on (below, the 128 x 128 and 128 x 64 tiles have more of
        // them): prompts of 2048 / 1000 / 512 tokens through the four Zovovik layers of width 4096 took 5.9 / 4.3 / 3.2 ms with
        // this line and 7.2 / 4.7 / 3.4 ms without the kernel.  matmul_kernel = 3: never, 4: always where its row tiles fit, 14: the form with
        // 128 activation rows.
        const int64_t opt = dev->opt_matmul_kernel;
        if (g.tiles && g.tile_rows > 128) return gemm_wide<320>(dev, epi, g);
        if (opt != 3) {
            // A round of workgroups with 128 activation rows takes two thirds of one with 256 (67 / 101 us at 4096 columns), so they
            // are the better ones where the tiles of 256 just miss a round: 14336 x 4096, 1025 rows 139 / 202 us (128 x 128: 156).
            const int64_t t256 = wn * ((g.m + 255) / 256), t128 = wn * ((g.m + 127) / 128);
            const bool tall = t256 * 4 >= cus * 3 && (t128 + cus - 1) / cus * 2 >= (t256 + cus - 1) / cus * 3;
            if (!g.tiles && opt != 14 && (opt == 4 || tall)) return gemm_wide<256>(dev, epi, g);
            if (g.tiles ? g.tile_rows == 128 && (opt == 4 || opt == 14 || wn * g.max_tiles >= cus) : opt == 14 || t128 * 4 >= cus * 3)
                return gemm_wide<128>(dev, epi, g);
        }
        const int tn = (g.n + 127) / 128;
        // small row tiles where the large ones would leave compute units without work
        const bool big = g.tiles ? g.tile_rows == 128 : (int64_t)tn * ((g.m + 127) / 128) >= dev->compute_units;
        const int ty = g.tiles ? g.max_tiles : big ? (g.m + 127) / 128 : (g.m + 63) / 64;
        FH_REQUIRE(ty <= 65535, "too many rows for one launch");
        const dim3 grid((unsigned)tn, (unsigned)ty);
        if (big) {
#define FH_K_(E_) k_gemm_bf16<128, E_>
            FH_GEMM_EPI(FH_K_, grid)
#undef FH_K_
        } else {
#define FH_K_(E_) k_gemm_bf16<64, E_>
            FH_GEMM_EPI(FH_K_, grid)
#undef FH_K_
        }
    }
#undef FH_GEMM_EPI
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// ------------------------------------------------------------------------------ rows -> activation rows
template <typename T>
__global__ __launch_bounds__(256) void k_rows_to_act(const float *__restrict__ x, int64_t ldx, int k, const float *__restrict__ w,
                                                     float eps, T *__restrict__ y, int kp) {
    __shared__ float red[4];
    const float *xr = x + (int64_t)blockIdx.x * ldx;
    T *yr = y + (int64_t)blockIdx.x * kp;
    float inv = 1.f;
    if (w) {
        float ss = 0.f;
        for (int i = threadIdx.x; i < k; i += 256) ss = fmaf(xr[i], xr[i], ss);
        ss = fh_wave_sum(ss);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
        __syncthreads();
        inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)k + eps);
    }
    for (int i = threadIdx.x; i < kp; i += 256) {
        float v = i < k ? xr[i] : 0.f;
        if (w && i < k) v = v * inv * w[i];
        yr[i] = fh_to<T>(v);
    }
}

fh_status fh_rows_to_act(fh_device *dev, int dtype, const float *x, int64_t ldx, int rows, int k, const float *w, float eps,
                         void *y, int kp) {
    if (dtype == FH_F32)
        k_rows_to_act<float><<<dim3((unsigned)rows), 256, 0, dev->stream>>>(x, ldx, k, w, eps, (float *)y, kp);
    else
        k_rows_to_act<uint16_t><<<dim3((unsigned)rows), 256, 0, dev->stream>>>(x, ldx, k, w, eps, (uint16_t *)y, kp);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// Sums of squares of a row: fours of values (single ones where their number is no multiple of 4) dealt out to 512 threads, eight wavefronts' sums in pairs.  A
// workgroup of four wavefronts has two of those threads' chains a thread (ss[1]: those of threads 256 on), so a row's norm has the same bits in every launch.
template <int WAVES>
__device__ __forceinline__ void row_sums(const float (&ss)[8 / WAVES], float *red) {
#pragma unroll
    for (int h = 0; h < 8 / WAVES; h++) {
        const float s = fh_wave_sum(ss[h]);
        if ((threadIdx.x & 63) == 0) red[h * WAVES + (threadIdx.x >> 6)] = s;
    }
}
__device__ __forceinline__ float row_sum(const float *red) { return ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7])); }

// ------------------------------------------------------------------------------ the output matrix for several rows
// Bound by the weights, which the matvec reads again for every row (16 rows of 4096 and a matrix of 32768: 16 x 45 us), so up to 16
// rows share one pass over them on the matrix cores.  The rows stay f32: each value is cut into three bf16 numbers of 8 bits (24
// in all: without a remainder), whose products with a bf16 weight are exact.  Each of the four wavefronts of a workgroup takes every fourth 64 of k and
// sums the first terms of even and odd steps and the others apart, so a sum has an eighth of the chain: against 64 bits 1.4e-7 of the root
// mean square at k = 4096, the matvec 1.6e-7.  With the launch that norms and cuts the rows 14 + 70 us at the size above.
enum { HEAD_ROWS = 16 };

// A small matrix is a few workgroups' work here, one after the other through its k, whatever the rows, and a matvec of it is short.  Both
// launches here / one matvec, us (k x n): 1024 x 512 12.7 / 3.4, 2048 x 512 17.5 / 4.4, 2048 x 4096 17.4 / 4.8, 2048 x 16384 20 / 18, 4096 x 512
// 28 / 5.5, 4096 x 4096 30 / 8.3, 4096 x 8192 31 / 14, 4096 x 12000 32 / 18, 8192 x 512 49 / 6.8, 8192 x 4096 53 / 14, 8192 x 6144 53 / 19.
int fh_head_rows_from(int k, int n) {
    if (n >= 6000) return n >= 12000 ? 2 : 3;
    if (n >= 3500) return k < 2048 ? 3 : 4;
    return 3 + std::min((k + 1024) / 2048, n >= 2048 ? 2 : 4);
}
struct HeadRows { int row[HEAD_ROWS], place[HEAD_ROWS], n; };

// Final norm of the rows (the arithmetic of k_matvec_mix, addition for addition: the normed row that a pass gives back has the same
// bits however many rows it has) and their three terms in the order of the MFMA operand: 64 of k: two
// steps of 32: three terms: lane l (row l % 16, k = 8 (l / 16) .. + 7): 16 bytes.  Rows that are not there are zeros.
__global__ __launch_bounds__(256) void k_head_x(const float *__restrict__ x, int k, int kp, const float *__restrict__ nw, float eps,
                                                HeadRows rows, uint16_t *__restrict__ xf, float *__restrict__ norm_out) {
    __shared__ float red[8];
    const int tid = threadIdx.x, r = blockIdx.x;
    const bool there = r < rows.n;
    const float *xr = x + (int64_t)rows.row[there ? r : 0] * k;
    float ss[2] = {0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (!(k & 3))
            for (int i = (tid + 256 * h) * 4; i < k; i += 2048) {
                const float4 v = *(const float4 *)(xr + i);
                ss[h] = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ss[h]))));
            }
        else
            for (int i = tid + 256 * h; i < k; i += 512) ss[h] = fmaf(xr[i], xr[i], ss[h]);
    row_sums<4>(ss, red);
    __syncthreads();
    const float inv = 1.0f / sqrtf(row_sum(red) / (float)k + eps);
    for (int i = tid; i < kp; i += 256) {
        const float v = there && i < k ? xr[i] * inv * nw[i] : 0.f;
        if (r == rows.n - 1) norm_out[i] = v;
        // cut, not rounded: nothing overflows; an infinity or a NaN is the first term's alone
        const uint32_t u = __float_as_uint(v);
        const bool finite = (u & 0x7F800000u) != 0x7F800000u;
        uint16_t t[3] = {(uint16_t)(u >> 16), 0, 0};
        if (finite) {
            const float v1 = v - __uint_as_float(u & 0xFFFF0000u);
            const uint32_t u1 = __float_as_uint(v1);
            t[1] = (uint16_t)(u1 >> 16);
            t[2] = (uint16_t)(__float_as_uint(v1 - __uint_as_float(u1 & 0xFFFF0000u)) >> 16);
        } else if (u & 0x007FFFFFu)
            t[0] |= 0x40u;
        const int step = i >> 5, lane = (i >> 3 & 3) * 16 + r;
#pragma unroll
        for (int e = 0; e < 3; e++) xf[(((int64_t)step * 3 + e) * 64 + lane) * 8 + (i & 7)] = t[e];
    }
}

__global__ __launch_bounds__(256, 2) void k_head_rows(const uint16_t *__restrict__ w, int n, int kp, const uint16_t *__restrict__ xf,
                                                      HeadRows rows, float *__restrict__ y, int64_t ldy) {
    constexpr int STAGES = 3; // 64 of k each: 8 KB of weights and 6 KB of rows a wavefront
    __shared__ fh_f4 red[4][4][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, row0 = blockIdx.x * 64;
    const int blocks = kp >> 6, mine = (blocks - wave + 3) >> 2;
    const uint16_t *wp[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int row = row0 + 16 * t + (lane & 15);
        wp[t] = w + (int64_t)(row < n ? row : n - 1) * kp + (lane >> 4) * 8;
    }
    fh_bf8 a[STAGES][2][4], b[STAGES][2][3];
    const auto fetch = [&](int s, int i) { // (no request under a condition; past the end the last block again)
        const int blk = min(4 * min(i, mine - 1) + wave, blocks - 1);
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int t = 0; t < 4; t++) fh_frag_load(a[s][h][t], wp[t] + blk * 64 + h * 32);
#pragma unroll
            for (int e = 0; e < 3; e++) fh_frag_load(b[s][h][e], xf + (((int64_t)blk * 2 + h) * 3 + e) * 512 + lane * 8);
        }
    };
    fh_f4 acc[4][3] = {}; // of the first term in the even and the odd steps, of the two others
    const auto use = [&](int s) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int e = 0; e < 3; e++) acc[t][e ? 2 : h] = fh_mma32(a[s][h][t], b[s][h][e], acc[t][e ? 2 : h]);
    };
    if (mine > 0) {
#pragma unroll
        for (int s = 0; s < STAGES; s++) fetch(s, s);
        int i = 0;
        for (; i + STAGES < mine; i += STAGES) {
#pragma unroll
            for (int s = 0; s < STAGES; s++) {
                use(s);
                fetch(s, i + s + STAGES);
            }
        }
#pragma unroll
        for (int s = 0; s < STAGES; s++)
            if (i + s < mine) use(s);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        fh_f4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) { // (a weight that is infinite leaves a NaN in the terms that are 0)
            const float hi = acc[t][0][e] + acc[t][1][e];
            v[e] = (__float_as_uint(hi) & 0x7F800000u) != 0x7F800000u ? hi + acc[t][2][e] : hi;
        }
        red[wave][t][lane] = v;
    }
    __syncthreads();
    const fh_f4 v = (red[0][wave][lane] + red[1][wave][lane]) + (red[2][wave][lane] + red[3][wave][lane]);
    const int r = lane & 15, at = row0 + 16 * wave + 4 * (lane >> 4);
    if (r >= rows.n) return;
    float *yr = y + rows.place[r] * ldy;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (at + e < n) yr[at + e] = v[e];
}

fh_status fh_head_rows(fh_device *dev, const float *x, int k, const float *w, float eps, const uint16_t *out, int n, const int *row,
                       const int *place, int count, float *y, int64_t ldy, float *norm_out) {
    const int kp = (int)fh_pad64(k);
    FH_REQUIRE((size_t)kp * 3 * HEAD_ROWS * 2 <= FH_FIXED_BYTES, "k = %d too long for the output matrix", k);
    uint16_t *xf = (uint16_t *)dev->fixed_buf;
    for (int at = 0; at < count; at += HEAD_ROWS) {
        HeadRows rows = {};
        rows.n = std::min<int>(count - at, HEAD_ROWS);
        for (int i = 0; i < rows.n; i++) rows.row[i] = row[at + i], rows.place[i] = place[at + i];
        k_head_x<<<dim3(HEAD_ROWS), 256, 0, dev->stream>>>(x, k, kp, w, eps, rows, xf, norm_out);
        k_head_rows<<<dim3((unsigned)((n + 63) / 64)), 256, 0, dev->stream>>>(out, n, kp, xf, rows, y, ldy);
        FH_HIP(hipGetLastError());
    }
    return FH_OK;
}

// ------------------------------------------------------------------------------ residual streams normed at a sublayer's end
__global__ void k_group_tiles(int groups, int s, int tile_rows, FhTile *tiles, int *n_tiles) {
    const int per = fh_tiles_of(s, tile_rows);
    for (int i = threadIdx.x; i < groups * per; i += blockDim.x) tiles[i] = fh_tile(i / per, i / per * s, s, i % per, tile_rows);
    if (threadIdx.x == 0) *n_tiles = groups * per;
}

fh_status fh_group_tiles(fh_device *dev, int groups, int s, int tile_rows, FhTile *tiles, int *n_tiles) {
    k_group_tiles<<<1, 256, 0, dev->stream>>>(groups, s, tile_rows, tiles, n_tiles);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

template <typename T>
__global__ __launch_bounds__(256) void k_add_normed(const float *__restrict__ x, const float *__restrict__ y, int k,
                                                    const float *__restrict__ w, float eps, float *__restrict__ x_out,
                                                    T *__restrict__ act, int kp) {
    constexpr int R = 16; // values of a thread that are requested at once; longer rows are read twice
    __shared__ float red[4];
    const int64_t row = (int64_t)blockIdx.x * k;
    float xv[R], yv[R], wv[R], ss = 0.f;
#pragma unroll
    for (int j = 0; j < R; j++) {
        const int i = threadIdx.x + 256 * j;
        const bool ok = i < k;
        yv[j] = ok ? y[row + i] : 0.f;
        xv[j] = ok ? x[row + i] : 0.f;
        wv[j] = ok ? w[i] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < R; j++) ss = fmaf(yv[j], yv[j], ss);
    for (int i = threadIdx.x + 256 * R; i < k; i += 256) ss = fmaf(y[row + i], y[row + i], ss);
    ss = fh_wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)k + eps);
    T *ar = act + (int64_t)blockIdx.x * kp;
#pragma unroll
    for (int j = 0; j < R; j++) {
        const int i = threadIdx.x + 256 * j;
        const float v = xv[j] + yv[j] * inv * wv[j];
        if (i < k) x_out[row + i] = v;
        if (act && i < kp) ar[i] = fh_to<T>(v); // zeros from k on
    }
    for (int i = threadIdx.x + 256 * R; i < kp; i += 256) {
        float v = 0.f;
        if (i < k) x_out[row + i] = v = x[row + i] + y[row + i] * inv * w[i];
        if (act) ar[i] = fh_to<T>(v);
    }
}

fh_status fh_add_normed(fh_device *dev, int dtype, const float *x, const float *y, int rows, int k, const float *w, float eps,
                        float *x_out, void *act, int kp) {
    const dim3 grid((unsigned)rows);
    if (dtype == FH_F32) k_add_normed<float><<<grid, 256, 0, dev->stream>>>(x, y, k, w, eps, x_out, (float *)act, kp);
    else k_add_normed<uint16_t><<<grid, 256, 0, dev->stream>>>(x, y, k, w, eps, x_out, (uint16_t *)act, kp);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

template <typename T>
__global__ __launch_bounds__(256) void k_embed_at(const uint16_t *__restrict__ table, int n, const uint16_t *__restrict__ pos_table,
                                                  int positions, const uint32_t *__restrict__ ids, int pos,
                                                  const int *__restrict__ pos_dev, int k, float *__restrict__ x, T *__restrict__ act, int kp) {
    const int t = blockIdx.y, c = (int)blockIdx.x * 256 + threadIdx.x;
    if (c >= kp) return;
    const uint32_t id = ids[t];
    int p = (pos_dev ? *pos_dev : pos) + t;
    p = p < positions ? p : positions - 1; // the host refuses positions behind the table
    float v = 0.f;
    if (c < k) {
        v = fh_bf_f32(table[(int64_t)(id < (uint32_t)n ? id : 0) * kp + c]);
        if (pos_table) v += fh_bf_f32(pos_table[(int64_t)p * kp + c]);
        x[(int64_t)t * k + c] = v;
    }
    if (act) act[(int64_t)t * kp + c] = fh_to<T>(v);
}

fh_status fh_embed_at(fh_device *dev, int dtype, const fh_qmatrix *table, const fh_qmatrix *pos_table, const uint32_t *ids, int s,
                      int pos, const int *pos_dev, float *x, void *act, int kp) {
    FH_REQUIRE(table->type == FH_BF16 && table->recs == kp && (!pos_table || (pos_table->type == FH_BF16 && pos_table->recs == kp)),
               "embedding tables are bf16 rows of one stride");
    const dim3 grid((unsigned)((kp + 255) / 256), (unsigned)s);
    const uint16_t *tb = (const uint16_t *)table->data, *pt = pos_table ? (const uint16_t *)pos_table->data : nullptr;
    const int n = (int)table->n, np = pos_table ? (int)pos_table->n : 1 << 30, k = (int)table->k;
    if (dtype == FH_F32) k_embed_at<float><<<grid, 256, 0, dev->stream>>>(tb, n, pt, np, ids, pos, pos_dev, k, x, (float *)act, kp);
    else k_embed_at<uint16_t><<<grid, 256, 0, dev->stream>>>(tb, n, pt, np, ids, pos, pos_dev, k, x, (uint16_t *)act, kp);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

template <typename T>
__global__ __launch_bounds__(256) void k_token_shift(FhShift m, const float *__restrict__ x, int k, int pos,
                                                     const float *__restrict__ state, int kp) {
    const int t = blockIdx.y, c = (int)blockIdx.x * 256 + threadIdx.x;
    if (c >= kp) return;
    float v = 0.f, d = 0.f;
    if (c < k) {
        v = x[(int64_t)t * k + c];
        d = (t > 0 ? x[(int64_t)(t - 1) * k + c] : pos > 0 ? state[((pos - 1) & 1) * k + c] : 0.f) - v;
    }
#pragma unroll
    for (int n = 0; n < FH_SHIFT_MAX; n++) {
        if (n >= m.n) break;
        const float y = c < k ? fmaf(d, m.mu[n][c], v) : 0.f;
        const int64_t o = (int64_t)t * kp + c;
        if (m.f32[n]) ((float *)m.y[n])[o] = y;
        else ((T *)m.y[n])[o] = fh_to<T>(y);
    }
}

fh_status fh_token_shift(fh_device *dev, int dtype, const FhShift &m, const float *x, int s, int k, int pos, float *state, int kp) {
    const dim3 grid((unsigned)((kp + 255) / 256), (unsigned)s);
    if (dtype == FH_F32) k_token_shift<float><<<grid, 256, 0, dev->stream>>>(m, x, k, pos, state, kp);
    else k_token_shift<uint16_t><<<grid, 256, 0, dev->stream>>>(m, x, k, pos, state, kp);
    FH_HIP(hipGetLastError());
    // after every reader of the old rows
    return fh_copy(dev, state + (int64_t)((pos + s - 1) & 1) * k, x + (int64_t)(s - 1) * k, (size_t)k * 4);
}

// A workgroup takes 16 rows of x and 16 of W; its four wavefronts share out k.  True f32 products on the widened weights.
__global__ __launch_bounds__(256) void k_low_rank_tanh(const float *__restrict__ x, int kp, int rows, const uint16_t *__restrict__ w, int n,
                                                       float *__restrict__ y, int ldy) {
    __shared__ float red[4][256];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, g = lane >> 4, m0 = (int)blockIdx.x * 16, n0 = (int)blockIdx.y * 16;
    const float *xp = x + (int64_t)(m0 + li < rows ? m0 + li : rows - 1) * kp + 8 * g;
    const uint16_t *wp = w + (int64_t)(n0 + li < n ? n0 + li : n - 1) * kp + 8 * g;
    fh_f4 acc = fh_f4{0.f, 0.f, 0.f, 0.f};
    for (int k = 32 * wave; k < kp; k += 128) {
        const uint4 u = *(const uint4 *)(wp + k);
        const fh_f8 fw = {{fh_bf_lo(u.x), fh_bf_hi(u.x), fh_bf_lo(u.y), fh_bf_hi(u.y), fh_bf_lo(u.z), fh_bf_hi(u.z), fh_bf_lo(u.w), fh_bf_hi(u.w)}};
        fh_f8 fx;
        fh_frag_load(fx, xp + k);
        acc = fh_mma32(fw, fx, acc); // a lane: W rows 4 g .. + 3 of x row li
    }
#pragma unroll
    for (int e = 0; e < 4; e++) red[wave][lane * 4 + e] = acc[e];
    __syncthreads();
    const int r = m0 + (tid >> 2) % 16, c = n0 + 4 * (tid >> 6) + (tid & 3); // lane tid / 4, element tid % 4
    const float v = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
    if (r < rows && c < ldy) y[(int64_t)r * ldy + c] = c < n ? tanhf(v) : 0.f;
}

fh_status fh_low_rank_tanh(fh_device *dev, const float *x, int kp, int rows, const uint16_t *w, int n, float *y, int ldy) {
    FH_REQUIRE(n > 0 && ldy >= n && kp % 64 == 0, "bad low-rank product");
    k_low_rank_tanh<<<dim3((unsigned)((rows + 15) / 16), (unsigned)((ldy + 15) / 16)), 256, 0, dev->stream>>>(x, kp, rows, w, n, y, ldy);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// A workgroup of eight wavefronts, one a compute unit, works its input out once, into the LDS, and goes through its share of one matrix's rows
// (FhRowDeal).  The input is requested ahead of the first weights, for requests are answered in their order, and under no condition.  What bounds
// it is the memory: 1.9 us of a launch, the bytes at 7.1 TB/s (a plain read) and one to two us for the input.  Replayed graphs over 1 GB of matrices,
// us, as many workgroups as there are rows for (two or four rows a wavefront, up to 16 KB on their way) / now:
//   normed    2880 x 2048 5.6 / 4.5, 8288 x 2048 10.7 / 7.6, 32768 x 2048 28.1 / 21.5, 4096 x 4096 10.3 / 8.0, 32768 x 4096 47.2 / 41.0
//   as it is  4096 x 14336 22.8 / 19.7;  a sublayer added  14336 x 4096 26.6 / 19.8, 16384 x 4096 29.7 / 22.1
//   gated     4096 x 4096 16.0 / 9.6;   six matrices, five of them on mixtures with the token before, 14336 x 4096 together 28.2 / 21.9
// (Before, the input's branches alone cost a third of that: with them in the code, though not taken, 4096 x 4096 took 9.7 us for 8.0.)
struct MvMixes { FhMvMix s[FH_MV_MAX]; int tiles[FH_MV_MAX]; int n; };

__device__ __forceinline__ float4 mv_if(bool c, float4 v) { // (v or zeros: as one choice of two float4 it would be one of addresses, in scratch memory)
    return make_float4(c ? v.x : 0.f, c ? v.y : 0.f, c ? v.z : 0.f, c ? v.w : 0.f);
}

// x' into the LDS, mixed with the token before it where the matrix wants that; start() asks for the first weights.
// XQ: fours of consecutive values of each vector that a thread holds, all requested at once (k a multiple of 4, 256 WAVES XQ at most); 0: any k, in
// fours or value by value.  MODE: what a launch has of this, so that one without a norm has no requests and registers for it.
enum { MV_PLAIN = 0, MV_NORM = 1, MV_ADD = 2, MV_SHIFT = 3, MV_GATED = 4 };
typedef float mv_four __attribute__((ext_vector_type(4), aligned(4))); // (of a vector that may begin anywhere)
template <int WAVES, int XQ, int MODE, typename F>
__device__ __forceinline__ void mv_input(const FhMvAdd &in, const float *mu, int k, int kp, const FhRowInput &xs, float *red, F start) {
    constexpr int NT = WAVES * 64;
    const int tid = threadIdx.x, end = 2 * xs.plane; // (whole pieces)
    constexpr bool NORM = MODE == MV_NORM, SHIFT = MODE == MV_SHIFT, ADD = MODE == MV_ADD || SHIFT;
    if (!SHIFT) mu = nullptr;
    const bool add = MODE == MV_ADD || (SHIFT && in.y), normed = NORM || add, one = blockIdx.x == 0;
    float *state = SHIFT ? in.state : nullptr;
    const int pos = state ? *in.pos_dev : 0;
    const float *before = state + ((pos - 1) & 1) * k;
    float *here = state + (pos & 1) * k;
    const bool shift = mu && pos > 0;
    const int out = NORM ? kp : k; // values of x_out
    float ss[8 / WAVES] = {0.f};
    const auto scale = [&]() { // of the norm, from the threads' sums of squares
        row_sums<WAVES>(ss, red);
        fh_lds_barrier();
        return 1.0f / sqrtf(row_sum(red) / (float)k + in.eps);
    };
    if constexpr (XQ > 0) {
        float4 x[XQ], y[ADD ? XQ : 1], w[MODE ? XQ : 1], m[SHIFT ? XQ : 1], b[SHIFT ? XQ : 1];
        // (what is not there is read from x and dropped: behind a condition the compiler no longer knows how many requests are on their way)
        const float *nw = NORM ? in.norm : add ? in.w : in.x, *yp = add ? in.y : in.x, *mp = mu ? mu : in.x, *bp = shift ? before : in.x;
#pragma unroll
        for (int j = 0; j < XQ; j++) {
            const int i = (tid + NT * j) * 4, at = i < k ? i : 0; // (past the end: the first values again, dropped below)
            x[j] = *(const float4 *)(in.x + at);
            if (ADD) y[j] = *(const float4 *)(yp + at);
            if (MODE) w[j] = *(const float4 *)(nw + at);
            if (SHIFT) m[j] = *(const float4 *)(mp + at), b[j] = *(const float4 *)(bp + at);
        }
        __builtin_amdgcn_sched_barrier(0);
        start();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < XQ; j++) {
            const bool past = (tid + NT * j) * 4 >= k;
            x[j] = mv_if(!past, x[j]);
            if (ADD) y[j] = mv_if(!past && add, y[j]);
            if (SHIFT) b[j] = mv_if(shift, b[j]);
        }
        float inv = 0.f;
        if (normed) {
#pragma unroll
            for (int j = 0; j < XQ; j++) {
                const float4 v = NORM ? x[j] : y[j];
                float &t = ss[j % (8 / WAVES)];
                t = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, t))));
            }
            inv = scale();
        }
#pragma unroll
        for (int j = 0; j < XQ; j++) {
            const int i = (tid + NT * j) * 4;
            if (i >= end) break;
            float4 v = x[j];
            if (NORM) v = make_float4(v.x * inv * w[j].x, v.y * inv * w[j].y, v.z * inv * w[j].z, v.w * inv * w[j].w);
            else if (add) v = make_float4(v.x + y[j].x * inv * w[j].x, v.y + y[j].y * inv * w[j].y, v.z + y[j].z * inv * w[j].z, v.w + y[j].w * inv * w[j].w);
            if (one) {
                if (in.x_out && i < out) *(float4 *)(in.x_out + i) = mv_if(i < k, v);
                if (state && i < k) *(float4 *)(here + i) = v;
            }
            if (mu)
                v = make_float4(fmaf(b[j].x - v.x, m[j].x, v.x), fmaf(b[j].y - v.y, m[j].y, v.y), fmaf(b[j].z - v.z, m[j].z, v.z),
                                fmaf(b[j].w - v.w, m[j].w, v.w));
            xs.quad(i >> 2) = mv_if(i < k, v);
        }
    } else if (!(k & 3)) { // longer than that, or from anywhere: in fours as well, dealt out alike, so that a norm has the same bits
        float inv = 0.f;
        if (normed) {
            const float *from = NORM ? in.x : in.y;
#pragma unroll
            for (int h = 0; h < 8 / WAVES; h++)
                for (int i = (tid + NT * h) * 4; i < k; i += 2048) {
                    const mv_four v = *(const mv_four *)(from + i);
                    ss[h] = fmaf(v[0], v[0], fmaf(v[1], v[1], fmaf(v[2], v[2], fmaf(v[3], v[3], ss[h]))));
                }
            inv = scale();
        }
#pragma unroll 2
        for (int i = tid * 4; i < end; i += NT * 4) {
            mv_four v = {0.f, 0.f, 0.f, 0.f};
            if (i < k) {
                v = *(const mv_four *)(in.x + i);
                if (NORM) v = v * inv * *(const mv_four *)(in.norm + i);
                else if (add) v += *(const mv_four *)(in.y + i) * inv * *(const mv_four *)(in.w + i);
                if (one) {
                    if (in.x_out) *(mv_four *)(in.x_out + i) = v;
                    if (state) *(mv_four *)(here + i) = v;
                }
                if (mu) {
                    const mv_four m = *(const mv_four *)(mu + i);
                    mv_four b = {0.f, 0.f, 0.f, 0.f};
                    if (shift) b = *(const mv_four *)(before + i);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = fmaf(b[e] - v[e], m[e], v[e]);
                }
            } else if (one && in.x_out && i < out) *(mv_four *)(in.x_out + i) = v;
            xs.quad(i >> 2) = make_float4(v[0], v[1], v[2], v[3]);
        }
        start();
    } else {
        float inv = 0.f;
        if (normed) {
            const float *v = NORM ? in.x : in.y;
            for (int i = tid; i < k; i += 512)
#pragma unroll
                for (int h = 0; h < 8 / WAVES; h++)
                    if (i + NT * h < k) ss[h] = fmaf(v[i + NT * h], v[i + NT * h], ss[h]);
            inv = scale();
        }
#pragma unroll 4
        for (int i = tid; i < end; i += NT) {
            float v = 0.f;
            if (i < k) {
                v = in.x[i];
                if (NORM) v = v * inv * in.norm[i];
                else if (add) v += in.y[i] * inv * in.w[i];
                if (one) {
                    if (in.x_out) in.x_out[i] = v;
                    if (state) here[i] = v;
                }
                if (mu) v = fmaf((shift ? before[i] : 0.f) - v, mu[i], v);
            } else if (one && in.x_out && i < out) in.x_out[i] = 0.f;
            xs.at(i) = v;
        }
        start();
    }
}

// Normed group by group and gated.  sums: k / 4 floats (XQ > 0: groups of a multiple of four values).
template <int WAVES, int XQ, typename F>
__device__ __forceinline__ void mv_gated(const FhMvAdd &in, int k, const FhRowInput &xs, float *ginv, float *sums, F start) {
    constexpr int NT = WAVES * 64;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, gl = k / in.groups, end = 2 * xs.plane;
    if constexpr (XQ > 0) {
        float4 x[XQ], g[XQ], w[XQ];
#pragma unroll
        for (int j = 0; j < XQ; j++) {
            const int i = (tid + NT * j) * 4, at = i < k ? i : 0;
            x[j] = *(const float4 *)(in.x + at);
            g[j] = *(const float4 *)(in.gate + at);
            w[j] = *(const float4 *)(in.w ? in.w + (in.w_len == k ? at : at % in.w_len) : in.gate + at);
        }
        __builtin_amdgcn_sched_barrier(0);
        start();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < XQ; j++) {
            const int q = tid + NT * j;
            if (q * 4 < k) sums[q] = fmaf(x[j].x, x[j].x, fmaf(x[j].y, x[j].y, fmaf(x[j].z, x[j].z, x[j].w * x[j].w)));
        }
        fh_lds_barrier();
        for (int n = wave; n < in.groups; n += WAVES) {
            float ss = 0.f;
            for (int i = lane; i < gl >> 2; i += 64) ss += sums[n * (gl >> 2) + i];
            ss = fh_wave_sum(ss);
            if (lane == 0) ginv[n] = 1.0f / sqrtf(ss / (float)gl + in.eps) * in.scale;
        }
        fh_lds_barrier();
#pragma unroll
        for (int j = 0; j < XQ; j++) {
            const int i = (tid + NT * j) * 4;
            const float s = ginv[i < k ? i / gl : 0];
            if (!in.w) w[j].x = w[j].y = w[j].z = w[j].w = 1.f;
            const float4 v = make_float4(x[j].x * s * w[j].x * fh_silu_f(g[j].x), x[j].y * s * w[j].y * fh_silu_f(g[j].y),
                                         x[j].z * s * w[j].z * fh_silu_f(g[j].z), x[j].w * s * w[j].w * fh_silu_f(g[j].w));
            if (i < end) xs.quad(i >> 2) = mv_if(i < k, v);
        }
    } else {
#pragma unroll 4
        for (int i = tid; i < end; i += NT) xs.at(i) = i < k ? in.x[i] : 0.f;
        start();
        fh_lds_barrier();
        for (int n = wave; n < in.groups; n += WAVES) {
            float ss = 0.f;
            for (int i = lane; i < gl; i += 64) ss = fmaf(xs.at(n * gl + i), xs.at(n * gl + i), ss);
            ss = fh_wave_sum(ss);
            if (lane == 0) ginv[n] = 1.0f / sqrtf(ss / (float)gl + in.eps) * in.scale;
        }
        fh_lds_barrier();
#pragma unroll 4
        for (int i = tid; i < k; i += NT) {
            float v = xs.at(i) * ginv[i / gl];
            if (in.w) v *= in.w[i % in.w_len];
            xs.at(i) = v * fh_silu_f(in.gate[i]);
        }
    }
}

template <int WAVES, int AHEAD, int XQ, int MODE>
__global__ __launch_bounds__(WAVES * 64) void k_matvec_mix(FhMvAdd in, int k, int kp, MvMixes segs) {
    extern __shared__ __attribute__((aligned(16))) float lds[]; // [kp in whole pieces | groups | k / 4 (gated)]
    __shared__ float red[8];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int tile = blockIdx.x, si = 0;
    while (si + 1 < segs.n && tile >= segs.tiles[si]) tile -= segs.tiles[si++];
    const FhMvMix seg = segs.s[si];
    const int nt = segs.tiles[si], first = wave * nt + tile, step = WAVES * nt;
    const FhRowInput xs{lds, fh_row_pieces(kp) * 256};
    FhRowDeal<AHEAD> rows;
    const auto start = [&]() { rows.start(seg.w, kp, first, step, seg.n); };
    if constexpr (MODE == MV_GATED) mv_gated<WAVES, XQ>(in, k, xs, lds + 2 * xs.plane, lds + 2 * xs.plane + in.groups, start);
    else mv_input<WAVES, XQ, MODE>(in, seg.mu, k, kp, xs, red, start);
    fh_lds_barrier();
    rows.run(xs, [&](int i, float v) {
        if (seg.act == FH_MV_ACT_RELU2) v = fmaxf(v, 0.f) * fmaxf(v, 0.f);
        else if (seg.act == FH_MV_ACT_TANH) v = tanhf(v);
        if (lane == 0) seg.y[first + i * step] = v;
    });
}

template <int WAVES, int AHEAD, int XQ, int MODE>
static fh_status matvec_mix_go(fh_device *dev, const FhMvAdd &in, int k, const MvMixes &ms, int tiles) {
    const int kp = (int)fh_pad64(k);
    const size_t lds = (size_t)(fh_row_pieces(kp) * 512 + (MODE == MV_GATED ? in.groups + (XQ ? k / 4 : 0) : 0)) * 4;
    if (lds > 48 * 1024) FH_TRY(fh_kernel_lds(dev, (const void *)k_matvec_mix<WAVES, AHEAD, XQ, MODE>, lds));
    k_matvec_mix<WAVES, AHEAD, XQ, MODE><<<dim3((unsigned)tiles), WAVES * 64, lds, dev->stream>>>(in, k, kp, ms);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// Few rows: workgroups of four wavefronts, a row each, with up to 8 KB on their way (every workgroup reads the whole input, so there are no more of them than
// that).  us, eight wavefronts / four: 128 x 1024 2.9 / 2.5, 512 x 2048 4.1 / 3.0, 1024 x 4096 5.3 / 4.4, 2048 x 1024 3.9 / 3.0, 4096 x 1024 4.4 / 4.0; the other way
// round 7000 x 1000 5.6 / 6.9, 2048 x 2048 4.0 / 4.1.  Inputs of 4097 values and more with nothing or a norm on their way in: 1024 x 14336 9.3 / 8.4.
static fh_status matvec_mix(fh_device *dev, const FhMvAdd &in, int k, const FhMvMix *segs, int n_segs) {
    MvMixes ms{};
    int n[FH_MV_MAX], total = 0;
    bool shift = in.state;
    ms.n = n_segs;
    for (int i = 0; i < n_segs; i++) ms.s[i] = segs[i], total += n[i] = segs[i].n, shift = shift || segs[i].mu;
    const int mode = in.gate ? MV_GATED : in.norm ? MV_NORM : shift ? MV_SHIFT : in.y ? MV_ADD : in.x_out ? MV_SHIFT : MV_PLAIN;
    const bool few = total <= (k <= 1024 ? 16 : 4) * dev->compute_units && (k <= 4096 || mode == MV_PLAIN || mode == MV_NORM);
    const int tiles = fh_row_share(n, n_segs, few ? (total + 3) / 4 + n_segs - 1 : dev->compute_units, ms.tiles);
    auto aligned = [](const void *p) { return !((uintptr_t)p & 15); };
    bool quads = !(k & 3) && k <= 16384 && aligned(in.x) && aligned(in.y) && aligned(in.w) && aligned(in.norm) && aligned(in.x_out) && aligned(in.state) && aligned(in.gate);
    for (int i = 0; i < n_segs; i++) quads = quads && aligned(segs[i].mu);
    if (in.gate) quads = quads && !(k / in.groups & 3) && !(in.w && (in.w_len & 3));
#define MV_MIX(W_, A_, XQ_)                                                                 \
    switch (mode) {                                                                         \
    case MV_PLAIN: return matvec_mix_go<W_, A_, XQ_, MV_PLAIN>(dev, in, k, ms, tiles);      \
    case MV_NORM: return matvec_mix_go<W_, A_, XQ_, MV_NORM>(dev, in, k, ms, tiles);        \
    case MV_ADD: return matvec_mix_go<W_, A_, XQ_, MV_ADD>(dev, in, k, ms, tiles);          \
    case MV_SHIFT: return matvec_mix_go<W_, A_, XQ_, MV_SHIFT>(dev, in, k, ms, tiles);      \
    default: return matvec_mix_go<W_, A_, XQ_, MV_GATED>(dev, in, k, ms, tiles);            \
    }
    if (few) {
        if (!quads) MV_MIX(4, 4, 0)
        if (k <= 1024) MV_MIX(4, 2, 1)
        if (k <= 2048) MV_MIX(4, 4, 2)
        if (k <= 4096) MV_MIX(4, 8, 4)
        if (mode == MV_PLAIN) return k <= 8192 ? matvec_mix_go<4, 8, 8, MV_PLAIN>(dev, in, k, ms, tiles) : matvec_mix_go<4, 8, 16, MV_PLAIN>(dev, in, k, ms, tiles);
        return k <= 8192 ? matvec_mix_go<4, 8, 8, MV_NORM>(dev, in, k, ms, tiles) : matvec_mix_go<4, 8, 16, MV_NORM>(dev, in, k, ms, tiles);
    }
    if (!quads) MV_MIX(8, 4, 0)
    if (k <= 2048) MV_MIX(8, 4, 1)
    if (k <= 4096) MV_MIX(8, 4, 2)
    if (k <= 8192) MV_MIX(8, 4, 4)
    MV_MIX(8, 4, 8)
#undef MV_MIX
}

fh_status fh_matvec_mix(fh_device *dev, const FhMvAdd &in, int k, const FhMvMix *segs, int n_segs) {
    FH_REQUIRE(n_segs >= 1 && n_segs <= FH_MV_MAX, "1 to %d matrices per launch", FH_MV_MAX);
    FH_REQUIRE(in.x && in.x != in.x_out && (!in.y || in.w) && (!in.state || in.pos_dev) && !in.norm, "bad input of a decode product");
    FH_REQUIRE(!in.gate || (!in.y && !in.state && in.groups > 0 && k % in.groups == 0), "bad gated input of a decode product");
    FH_REQUIRE((fh_pad64(k) + (in.gate ? in.groups : 0)) * 4 <= 150 * 1024, "k = %d too long for the matvec", k);
    return matvec_mix(dev, in, k, segs, n_segs);
}

fh_status fh_matvec_norm(fh_device *dev, const float *x, int k, const float *w, float eps, const FhMvSeg *segs, int n_segs,
                         float *norm_out) {
    FH_REQUIRE(n_segs >= 1 && n_segs <= 3, "1 to 3 matrices per matvec launch");
    FH_REQUIRE(w || !norm_out, "a normed row to give back needs a norm");
    FH_REQUIRE(fh_pad64(k) * 4 <= 120 * 1024, "k = %d too long for the matvec", k);
    FhMvMix ms[3];
    for (int i = 0; i < n_segs; i++) ms[i] = FhMvMix{segs[i].w, nullptr, segs[i].y, segs[i].n, FH_MV_ACT_NONE};
    FhMvAdd in;
    in.x = x, in.norm = w, in.eps = eps, in.x_out = norm_out;
    return matvec_mix(dev, in, k, ms, n_segs);
}

// ------------------------------------------------------------------------------ fh_qmatmul on bf16 rows
__global__ __launch_bounds__(256) void k_pad_bf16_rows(const uint16_t *__restrict__ x, int k, uint16_t *__restrict__ y, int kp) {
    for (int i = threadIdx.x; i < kp; i += 256) y[(int64_t)blockIdx.x * kp + i] = i < k ? x[(int64_t)blockIdx.x * k + i] : 0;
}

// ROWS weight rows of one wavefront, streamed in pieces of 512 (a lane: eight values, 16 bytes) with AHEAD pieces on their way.
// No request is under a condition - a lane past the end of the rows repeats the last eight values, a piece past the last one the
// last piece: with a branch around a request the compiler can no longer count what is younger and waits for everything.
template <int ROWS, int AHEAD>
struct RowStream {
    const uint16_t *w[ROWS];
    uint4 u[AHEAD][ROWS];
    int kp, pieces, lane8;
    __device__ __forceinline__ void fetch(int slot, int piece) {
        const int c = piece * 512 + lane8, at = c < kp ? c : kp - 8;
#pragma unroll
        for (int r = 0; r < ROWS; r++) u[slot][r] = *(const uint4 *)(w[r] + at);
    }
    __device__ __forceinline__ void start(int kp_) {
        kp = kp_, pieces = fh_row_pieces(kp), lane8 = (threadIdx.x & 63) * 8;
#pragma unroll
        for (int i = 0; i < AHEAD; i++) fetch(i, i < pieces ? i : pieces - 1);
    }
    __device__ __forceinline__ void use(int slot, int piece, const float *x, float *acc) const {
        const int c = piece * 512 + lane8;
        if (c >= kp) return;
        const float4 a = *(const float4 *)(x + c), b = *(const float4 *)(x + c + 4);
#pragma unroll
        for (int r = 0; r < ROWS; r++) acc[r] = fh_dot8(u[slot][r], a, b, acc[r]);
    }
    // acc[r] += rows . x (x: kp values in the LDS), not yet summed over the lanes
    __device__ __forceinline__ void run(const float *x, float *acc) {
        int p = 0;
        for (; p + AHEAD < pieces; p += AHEAD) {
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                use(i, p + i, x, acc);
                fetch(i, p + i + AHEAD < pieces ? p + i + AHEAD : pieces - 1);
            }
        }
#pragma unroll
        for (int i = 0; i < AHEAD; i++)
            if (p + i < pieces) use(i, p + i, x, acc);
    }
};

// The product by itself where dealing the rows out (FhRowDeal, k_matvec_mix) costs more than it gives: as many workgroups of four wavefronts as there are rows for,
// each with all that it reads on its way; the same sums.  XV: 16-byte pieces of the input a thread holds, requested ahead of the first weights (k a multiple
// of four); 0: the input goes to the LDS in a loop ahead of them.
template <int ROWS, int XV>
__global__ __launch_bounds__(256, XV ? 1 : 8) void k_matvec_rows(const float *__restrict__ x, const uint16_t *__restrict__ w, int k, int kp, int n, float *__restrict__ y) {
    extern __shared__ __attribute__((aligned(16))) float xs[]; // [kp]
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, row0 = ((int)blockIdx.x * 4 + wave) * ROWS;
    RowStream<ROWS, XV == 0 ? 8 / ROWS : XV == 1 ? 2 : 8> rows;
#pragma unroll
    for (int r = 0; r < ROWS; r++) rows.w[r] = w + (int64_t)(row0 + r < n ? row0 + r : n - 1) * kp;
    if (XV && !(k & 3)) { // (k is at most 1024 XV)
        constexpr int NX = XV ? XV : 1;
        mv_four v[NX];
#pragma unroll
        for (int j = 0; j < NX; j++) {
            const int i = (tid + 256 * j) * 4;
            v[j] = *(const mv_four *)(x + (i < k ? i : 0));
        }
        __builtin_amdgcn_sched_barrier(0);
        rows.start(kp);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NX; j++) {
            const int i = (tid + 256 * j) * 4;
            if (i < kp) *(float4 *)(xs + i) = mv_if(i < k, make_float4(v[j][0], v[j][1], v[j][2], v[j][3]));
        }
    } else {
        if (!(k & 3)) {
#pragma unroll 8
            for (int i = tid * 4; i < kp; i += 1024) {
                mv_four v = {0.f, 0.f, 0.f, 0.f};
                if (i < k) v = *(const mv_four *)(x + i);
                *(float4 *)(xs + i) = make_float4(v[0], v[1], v[2], v[3]);
            }
        } else {
#pragma unroll 8
            for (int i = tid; i < kp; i += 256) xs[i] = i < k ? x[i] : 0.f;
        }
        rows.start(kp);
    }
    __syncthreads();
    float acc[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) acc[r] = 0.f;
    rows.run(xs, acc);
#pragma unroll
    for (int r = 0; r < ROWS; r++) acc[r] = fh_wave_sum(acc[r]);
    if (lane == 0)
#pragma unroll
        for (int r = 0; r < ROWS; r++)
            if (row0 + r < n) y[row0 + r] = acc[r];
}

template <int ROWS, int XV>
static fh_status matvec_rows_go(const fh_qmatrix *q, const float *x, float *y) {
    fh_device *dev = q->dev;
    const int n = (int)q->n, kp = (int)q->recs;
    const size_t lds = (size_t)kp * 4;
    if (lds > 48 * 1024) FH_TRY(fh_kernel_lds(dev, (const void *)k_matvec_rows<ROWS, XV>, lds));
    k_matvec_rows<ROWS, XV><<<dim3((unsigned)((n + 4 * ROWS - 1) / (4 * ROWS))), 256, lds, dev->stream>>>(x, (const uint16_t *)q->data, (int)q->k, kp, n, y);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// Where that is.  Times of the rows dealt out over those here, one matrix again and again / 420 MB of them:
// - long inputs and few rows, of which a wavefront has one: 512 x 14336 1.4 / 1.25, 512 x 8192 1.2 / 1.05, 512 x 28672 1.8 / 1.8, 1024 x 28672 1.4 / 1.3, but 1024 x 14336 1.3 / 1.0 and
//   1024 x 16384 1.25 / 0.9 (1536 x 14336 0.87 / 0.95, 512 x 4096 1.0 / 0.8);
// - rows of one piece, whose sum over the lanes is all there is to wait for: k = 512 1.2 to 1.5 / 1.1 to 1.3; of two pieces (k = 1024) 4096 rows 1.36 / 1.0, 16384 rows
//   1.5 / 1.0 (512 rows 1.13 / 0.94), and of three where the dealt out ones come out uneven: k = 1536 6144 rows 1.5 / 1.25, 4096 rows 1.4 / 1.05 (3072 rows / 0.98);
// - k up to 3072 and 2048 to 6144 rows that stay in the last cache: 4096 x 2048 4.0 us / 3.1, 3072 x 2048 1.29 (/ 0.95; 16384 x 2048 0.76 / 0.8).
static bool matvec_rows_pay(const fh_device *dev, int n, int k) {
    const bool stream = fh_matrices_stream(dev);
    if (k > 4096) return n <= (stream && k <= 16384 ? 512 : 1024);
    if (k <= 512 || (k <= 1536 && n >= 4096 && n < 8192)) return true;
    return !stream && (k <= 1024 || (k <= 3072 && n >= 2048 && n <= 6144) || (k <= 2048 && n >= 2048 && n <= 8192));
}
static fh_status matvec_rows(const fh_qmatrix *q, const float *x, float *y) {
    const int64_t k = q->k, waves = (int64_t)q->dev->compute_units * 4;
    if (q->n >= waves * 8) return matvec_rows_go<4, 0>(q, x, y);
    if (q->n >= waves * 2) return k <= 1024 ? matvec_rows_go<2, 1>(q, x, y) : matvec_rows_go<2, 0>(q, x, y);
    if (k <= 1024) return matvec_rows_go<1, 1>(q, x, y);
    return k <= 16384 ? matvec_rows_go<1, 16>(q, x, y) : matvec_rows_go<1, 0>(q, x, y);
}

// f32 activations are multiplied in true f32, bf16 ones on the bf16 matrix cores.
fh_status fh_launch_bf16_matmul(const fh_qmatrix *q, const void *x, int x_is_bf16, int m, float *y) {
    fh_device *dev = q->dev;
    const int k = (int)q->k, kp = (int)q->recs;
    if (m == 1 && !x_is_bf16 && (size_t)kp * 4 <= 120 * 1024) {
        if (matvec_rows_pay(dev, (int)q->n, k)) return matvec_rows(q, (const float *)x, y);
        const FhMvSeg s{(const uint16_t *)q->data, y, (int)q->n};
        return fh_matvec_norm(dev, (const float *)x, k, nullptr, 0.f, &s, 1, nullptr);
    }
    const int dt = x_is_bf16 ? FH_BF16_ACT : FH_F32;
    FH_TRY(fh_dev_scratch(dev, &dev->act_buf, &dev->act_cap, (size_t)m * kp * fh_act_size(dt)));
    if (x_is_bf16) {
        k_pad_bf16_rows<<<dim3((unsigned)m), 256, 0, dev->stream>>>((const uint16_t *)x, k, (uint16_t *)dev->act_buf, kp);
        FH_HIP(hipGetLastError());
    } else FH_TRY(fh_rows_to_act(dev, FH_F32, (const float *)x, k, m, k, nullptr, 0.f, dev->act_buf, kp));
    FhGemm g;
    g.w = (const uint16_t *)q->data, g.x = dev->act_buf, g.y = y, g.ldy = q->n, g.n = (int)q->n, g.kp = kp, g.m = m;
    return fh_gemm(dev, dt, FH_GEMM_F32, g);
}
