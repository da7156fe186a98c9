// What the chunked recurrences share (gdr_chunk.hip: training of the hybrid text stack; delta_chunk.hip: ragged serving steps): chunks of 64 tokens of heads 128 | 128 as
// products on v_mfma_f32_32x32x2_f32 (lane l supplies A[m = l % 32][k = l / 32] and B[k][n = l % 32]), decays in fp64 logarithms, the unit triangle's inverse.
#pragma once
#include "common.h"
#include "lane_sums.h"

constexpr int GC = 64, GD = 128, GV = 32;  // tokens of a chunk, head width (keys and values), value columns of a scan's workgroup

__device__ __forceinline__ f32x16 mfma2(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 widen4(u32x2 w) {
    return f32x4{__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16), __uint_as_float(w[1] & 0xffff0000u)};
}
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int e = 0; e < 16; ++e) z[e] = 0.f;
    return z;
}
// accumulator register e of lane (ln, hf) holds row c_row(e, hf), column ln of a 32 x 32 tile
__device__ __forceinline__ constexpr int c_row(int e, int hf) { return 8 * (e >> 2) + 4 * hf + (e & 3); }
__device__ __forceinline__ float half_sum(float v) {  // sum over the 32 lanes of a half wave
    v = lanes_sum<16>(v);
    return v + __shfl_xor(v, 16, 64);
}
// the decay as its logarithm is taken of it: what is below 1e-30 counts as 1e-30, a NaN stays one
__device__ __forceinline__ float decay_at_least(float a) { return a < 1e-30f ? 1e-30f : a; }
// logarithms of 64 decays, cumulated over the lanes of one wave in fp64: a difference of two large sums keeps its digits
__device__ __forceinline__ double cumulated_log64(float a) {
    double g = log((double)a);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double u = __shfl_up(g, o, 64);
        if (lane >= o) g += u;
    }
    return g;
}

// exp of a sum of log decays: expf takes the rounded sum, the first power of what was cut off comes back behind it (of -20 fp32 keeps two parts in 10^6)
__device__ __forceinline__ float exp_of(double g) {
    const float r = (float)g, e = expf(r);
    return fmaf(e, (float)(g - (double)r), e);
}
__device__ __forceinline__ void add16(f32x16& to, f32x16& from) {  // a chain's sum so far to its total, and the chain begins anew: half the length, 0.7 of its error
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        to[e] += from[e];
        from[e] = 0.f;
    }
}

// ---- fp32 products on the bf16 matrix pipe: a number is the sum of three bf16 parts (24 bits: 8 and 8 and the rest, exactly), a product the sum of the parts' products, exact in fp32.  Of two split
// operands the six largest are taken -- what is left out is 2^-26 of the product -- the first parts' by themselves in one accumulator, the others in a second: a sum over 128 rounds eight times at its
// own size where a chain of fp32 products rounds 64 times.  32 clocks for 32 x 32 x 16 and 16 of a part against 512 on the fp32 pipe.  An infinity or a NaN makes the sum a NaN.
// Not all 24 bits near the ends of the range: below some 2^-110 the third part is subnormal, or nothing; and what lies within half a step of bf16 of the largest number has an infinite first part, so
// its sums are NaN (the forward's scan then takes the recurrence).
struct Parts8 { bf16x8 p[3]; };  // eight consecutive k of a fragment's row
__device__ __forceinline__ void parts_of(float a, float b, unsigned (&w)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        w[i] = pack_bf2(a, b);
        a -= __uint_as_float(w[i] << 16);
        b -= __uint_as_float(w[i] & 0xffff0000u);
    }
}
__device__ __forceinline__ Parts8 parts8(const f32x4& a, const f32x4& b) {
    unsigned w[4][3];
    parts_of(a[0], a[1], w[0]), parts_of(a[2], a[3], w[1]), parts_of(b[0], b[1], w[2]), parts_of(b[2], b[3], w[3]);
    Parts8 r;
#pragma unroll
    for (int i = 0; i < 3; ++i) r.p[i] = __builtin_bit_cast(bf16x8, u32x4{w[0][i], w[1][i], w[2][i], w[3][i]});
    return r;
}
__device__ __forceinline__ f32x16 mfma16(const bf16x8& a, const bf16x8& b, const f32x16& c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ void mfma_parts(const Parts8& a, const Parts8& b, f32x16& hi, f32x16& lo) {
    lo = mfma16(a.p[2], b.p[0], lo);
    lo = mfma16(a.p[0], b.p[2], lo);
    lo = mfma16(a.p[1], b.p[1], lo);
    lo = mfma16(a.p[1], b.p[0], lo);
    lo = mfma16(a.p[0], b.p[1], lo);
    hi = mfma16(a.p[0], b.p[0], hi);
}
__device__ __forceinline__ void mfma_parts(const bf16x8& a, const Parts8& b, f32x16& hi, f32x16& lo) {  // a: a bf16 operand
    lo = mfma16(a, b.p[2], lo);
    lo = mfma16(a, b.p[1], lo);
    hi = mfma16(a, b.p[0], hi);
}
// the three parts of [rows][ld] in LDS, a plane each: the fragment at `at` (elements), and four values of it written
template <int PLANE>
__device__ __forceinline__ Parts8 parts_at(const bf16_t* planes, int at) {
    Parts8 r;
#pragma unroll
    for (int i = 0; i < 3; ++i) r.p[i] = *reinterpret_cast<const bf16x8*>(planes + i * PLANE + at);
    return r;
}
template <int PLANE>
__device__ __forceinline__ void put_parts(bf16_t* planes, int at, float a, float b, float c, float d) {
    unsigned w0[3], w1[3];
    parts_of(a, b, w0), parts_of(c, d, w1);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2*>(planes + i * PLANE + at) = u32x2{w0[i], w1[i]};
}
// whether any of 16 values is infinite or NaN
__device__ __forceinline__ bool lost16(const f32x16& v) {
    float z = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) z = fmaf(v[e], 0.f, z);
    return z != z;
}

// T = (I + tril(N, -1))^-1, both [64][68] in LDS, by the four waves of a workgroup (N's upper right quarter is scratch): the two diagonal 32 x 32 blocks by forward
// substitution (lane = column), the block below them as -R22 (N21 R11).
__device__ __forceinline__ void invert_unit_lower64(float (&N)[GC][GC + 4], float (&T)[GC][GC + 4]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5;
    if (wave < 2) {  // R of the two diagonal 32 x 32 blocks: lane = column, forward substitution down the rows
        if (lane < 32) {
            float r[32];
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                float s = i == ln ? 1.f : 0.f;
#pragma unroll
                for (int m = 0; m < i; ++m) s = fmaf(-N[32 * wave + i][32 * wave + m], r[m], s);
                r[i] = s;
                T[32 * wave + i][32 * wave + ln] = s;
            }
        }
    } else {
        for (int idx = tid - 128; idx < 32 * 32; idx += 128) T[idx >> 5][32 + (idx & 31)] = 0.f;
    }
    __syncthreads();
    if (wave == 0) {  // R21 = -R22 (A21 R11): the inner product parks above N's diagonal
        f32x16 y = zero16();
#pragma unroll
        for (int kb = 0; kb < 32; kb += 8) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(&N[32 + ln][kb + 4 * hf]);
#pragma unroll
            for (int j = 0; j < 4; ++j) y = mfma2(a[j], T[kb + 4 * hf + j][ln], y);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) N[c_row(e, hf)][32 + ln] = y[e];
    }
    __syncthreads();
    if (wave == 0) {
        f32x16 y = zero16();
#pragma unroll
        for (int kb = 0; kb < 32; kb += 8) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(&T[32 + ln][32 + kb + 4 * hf]);
#pragma unroll
            for (int j = 0; j < 4; ++j) y = mfma2(a[j], N[kb + 4 * hf + j][32 + ln], y);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) T[32 + c_row(e, hf)][ln] = -y[e];
    }
    __syncthreads();
}
