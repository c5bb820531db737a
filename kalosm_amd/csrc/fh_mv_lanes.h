// Lane-level helpers shared by the single-row MFMA matvec kernels (Q4_K, Q6_K).
#pragma once
#include "fh_internal.h"

// Cross-lane moves inside a row of 16 lanes as DPP modifiers (one VALU op, no LDS round trip).
#define DPP_XOR1 0xB1        // quad_perm [1,0,3,2]
#define DPP_XOR2 0x4E        // quad_perm [2,3,0,1]
#define DPP_HALF_MIRROR 0x141 // lane i <- lane 7-i within each group of 8
#define DPP_ROW_MIRROR 0x140  // lane i <- lane 15-i within each row of 16
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
// sum over the four rows of 16 lanes of a wavefront (lane i of every row gets it): two register swaps, no LDS
__device__ __forceinline__ float rows_sum(float a) {
    const uint32_t u = __float_as_uint(a);
    auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    a = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
    const uint32_t w = __float_as_uint(a);
    auto s32 = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
}
// LDS addresses as 32-bit integers, so that a per-lane choice between two of them is one v_cndmask on a constant
// lane mask held in scalar registers.
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 lds_read16(uint32_t a) {
    const u32x4 v = *(__attribute__((address_space(3))) const u32x4 *)(uintptr_t)a;
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint32_t sel_lanes(uint64_t mask, uint32_t yes, uint32_t no) {
    uint32_t r;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(no), "v"(yes), "s"(mask));
    return r;
}


// Weights of a product of one or a few rows are read by one wavefront each and not again in this launch.  Where more than the 256 MB of the last cache passes
// before the next step reads them, they are read with the hint that they are streamed.  A decoder knows whether it does; a matrix by itself is taken for a part
// of a larger whole from 16 MB on, if the matrices on the device are more than that cache.  us, plainly / with the hint: 8B, 512 + 128 tokens 197017 / 188284 (only the
// matrices of 16 MB and more 196240), a 2048-wide decoder of 193 MB 8904 / 9052; one row of Q4_K 28672 x 4096, one of them 12.4 / 12.9, four (264 MB) 12.4 / 13.8, seven (462 MB)
// 14.8 / 14.0, of 65536 x 4096, one (151 MB) 23.2 / 26.1, two 28.0 / 26.7; sixteen rows of Q8_0 14336 x 4096, four (250 MB) 17.0 / 18.2, seven 19.3 / 18.5.
template <bool ONCE, typename T>
__device__ __forceinline__ T fh_ld_weights(const uint8_t *p) {
    if constexpr (!ONCE) return *(const T *)p;
    typedef uint32_t words __attribute__((ext_vector_type(sizeof(T) / 4)));
    const words v = __builtin_nontemporal_load((const words *)p);
    T r;
    __builtin_memcpy(&r, &v, sizeof(T));
    return r;
}
static inline bool fh_weights_once(const fh_qmatrix *q) { return q->streamed < 0 ? q->bytes >= (size_t)16 << 20 && fh_matrices_stream(q->dev) : q->streamed != 0; }
