// What the kernels of four waves with 128x128 outputs share (gemm_quad.h, bgemm_quad.h): products on the accumulation registers, and a wave's way from there to whole rows.
#pragma once
#include "common.h"

constexpr int QUAD_PANEL = 16384, QUAD_STAGE = 4 * QUAD_PANEL, QUAD_SMEM = 2 * QUAD_STAGE;
__host__ __device__ constexpr int64_t quad_share(int64_t K, int ksplit) { return ((K + 63) / 64 + 2 * ksplit - 1) / (2 * ksplit) * 2; }  // K-tiles of one of ksplit shares of K, an even number; the last one's are what is left

// Sums in the accumulation registers: left to itself the compiler moves part of 256 of them back and forth.  B's fragment is the first operand: a lane holds C[row lane & 15][4 (lane >> 4) + e].
// first: the sum starts at the constant 0 (no accumulator is cleared anywhere)
__device__ __forceinline__ void quad_mma_first(f32x4& c, const bf16x8& a, const bf16x8& b) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(b), "v"(a)); }
__device__ __forceinline__ void quad_mma(f32x4& c, const bf16x8& a, const bf16x8& b) { asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a)); }

// A sum, moved where it is used (left to the compiler those of many blocks are moved out at once, and spilled).  Behind the products' last way through the pipe: the caller waits.
__device__ __forceinline__ float quad_value(const f32x4& c, int e) {
    float x;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(c[e]));
    return x;
}
__device__ __forceinline__ void quad_swap(unsigned x, unsigned y, unsigned& lo, unsigned& hi) {
    const auto s = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    lo = s[0], hi = s[1];
}
// rows 0-7 (half 0) or 8-15 of 16: a's in the lanes of bit 3 clear, b's in the others
__device__ __forceinline__ unsigned quad_rows(unsigned a, unsigned b, int half) {
    return (unsigned)(half == 0 ? __builtin_amdgcn_update_dpp((int)a, (int)b, 0x128, 0xf, 0xc, false) : __builtin_amdgcn_update_dpp((int)b, (int)a, 0x128, 0xf, 0x3, false));
}
// A 16 x 64 block as eight rows at a time, o[half]: lane & 7 is the row, bits 3, 4, 5 of the lane are its columns' group of 32, of 16 and of 8.  As bf16 ...
__device__ __forceinline__ void quad_packed(const f32x4 (&c)[4], u32x4 (&o)[2]) {
    unsigned a[4], b[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        quad_swap(pack_bf2(quad_value(c[0], 2 * e), quad_value(c[0], 2 * e + 1)), pack_bf2(quad_value(c[1], 2 * e), quad_value(c[1], 2 * e + 1)), a[e], a[2 + e]);
        quad_swap(pack_bf2(quad_value(c[2], 2 * e), quad_value(c[2], 2 * e + 1)), pack_bf2(quad_value(c[3], 2 * e), quad_value(c[3], 2 * e + 1)), b[e], b[2 + e]);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[half][e] = quad_rows(a[e], b[e], half);
}
// ... and in fp32
__device__ __forceinline__ void quad_spread(const f32x4 (&c)[4], float (&o)[2][8]) {
    unsigned a[8], b[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        quad_swap(__float_as_uint(quad_value(c[0], e)), __float_as_uint(quad_value(c[1], e)), a[e], a[4 + e]);
        quad_swap(__float_as_uint(quad_value(c[2], e)), __float_as_uint(quad_value(c[3], e)), b[e], b[4 + e]);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int e = 0; e < 8; ++e) o[half][e] = __uint_as_float(quad_rows(a[e], b[e], half));
}
