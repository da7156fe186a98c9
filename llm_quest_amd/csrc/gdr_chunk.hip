// Gated delta rule in chunks of 64 tokens on the fp32 matrix pipe (gfx950 only), forward and backward, for heads of 128 | 128.
//
// The token-by-token recurrence of qwen35.hip (S <- a S + b (v - a S k) k^T, o = S q / sqrt(dk)) is one dependent chain per token: at 8 x 708 tokens x 16 heads its
// forward takes 565 us and its backward 1 470 us a layer, whatever the chip could multiply.  Inside a chunk the recurrence is linear algebra (rows are tokens,
// g = cumulated log decay, D_ij = exp(g_i - g_j), gam = exp(g), Gp_j = exp(g_63 - g_j)):
//     A = tril(diag(b) K K^T . D, -1),  R = (I + A)^-1,  T = R diag(b),  P = scale tril(Q K^T . D),  Uv = T V,  Kw = T (gam K)      -- no state: one workgroup per chunk
//     U = Uv - Kw S^T,  O = scale gam (Q S^T) + P U,  S <- gam_63 S + (Gp U)^T K                                                    -- the chain: one step per chunk
// and the adjoint splits the same way: only dS crosses chunks (dU = P^T dO + Gp (K dS^T), dS <- gam_63 dS + (scale gam dO)^T Q - dU^T Kw), everything else is one
// workgroup per chunk afterwards.  Four kernels: prep, scan, reverse scan (both per 32 value rows of the state: a row never meets another), and the rest.
// All sums are fp32 FMAs on v_mfma_f32_32x32x2_f32 (the two products of bf16 operands alone, K K^T and Q K^T, on the bf16 shape: exact); the log decays are cumulated
// in fp64, so a difference of two large ones keeps its digits.  d(alpha) is taken from sums over the pairs that span a token -- never as a difference of
// larger sums, so it keeps its digits where alpha is tiny (below 1e-30 alpha counts as 1e-30); d(beta) as what reaches u times u / beta.
// A matrix pipe's chain of 128 products rounds 128 times at its size where lanes sum 16 and meet in a tree; so the chains that show are cut (add16) and the state's gradient
// gathers its terms from the last token to the first.  Distance to 64 bits, token-by-token kernels | here, 256 tokens, geometric mean of four draws: outputs, d(q), d(k), d(v)
// 1.65e-3 | 1.65e-3 (their bf16); fp32: state 7.4e-8 | 8.6e-8, d(state) 9.0e-8 | 9.5e-8 (2.9e-7 from the first token on), d(beta) 1.5e-7 | 1.8e-7 (2.6e-7 with whole chains), d(alpha)
// 1.7e-7 | 2.1e-7 (2.5e-7); decays near one 4.4e-7 | 3.6e-7, 5.0e-7 | 4.9e-7; nearly parallel keys 1.5e-7 | 2.3e-7, 2.1e-7 | 4.4e-7.  Cutting d(q)'s and d(k)'s chains as well:
// d(alpha) 1.9e-7 for 50 us of a backward of 680 (registers spill).
// Bound: the fp32 matrix pipe (256 FLOP a clock and CU).  The products of one 64-token chunk of one head: 37 MFLOP forward and backward together.
#include "gdr_chunk.h"

#define ST(s) ((hipStream_t)(s))

namespace {

// one chunk of one head in the saved buffer (floats): Kw [64][128], U [64][128], P [64][64], gam [64], Gp [64] (C_: from Kw on); for a backward the state at its start
// [128 dv][128 dk] lies in front of them and R [64][64] behind (G_: from there on)
constexpr int C_U = GC * GD, C_P = C_U + GC * GD, C_GAM = C_P + GC * GC, C_R = C_GAM + 2 * GC, G_SMALL = C_R, G_KW = GD * GD, G_U = G_KW + C_U, G_P = G_KW + C_P, G_GAM = G_KW + C_GAM,
              G_R = G_KW + C_R, G_BLOCK = G_R + GC * GC;
constexpr int64_t SPAN_BYTES = 256 << 20;  // of a forward that keeps nothing: what one span of chunks takes at most, if that holds four (a prompt of any length, bounded scratch)
constexpr int W_DU = GD * GD, W_BLOCK = W_DU + GC * GD;  // backward workspace of a chunk: dS at its end, dU

// four consecutive bf16 of row `r` of a [tokens, ld] operand, zeros beyond the sequence
__device__ __forceinline__ u32x2 row4(const bf16_t* p, int64_t ld, int r, int cnt, int c) {
    return r < cnt ? *reinterpret_cast<const u32x2*>(p + r * ld + c) : u32x2{0u, 0u};
}
__device__ __forceinline__ float one(const bf16_t* p, int64_t ld, int r, int cnt, int c) { return r < cnt ? bf2f(p[r * ld + c]) : 0.f; }

__device__ __forceinline__ double cumulated_log(const float* alpha, int64_t idx, bool in, float& a_out) {
    a_out = decay_at_least(in ? alpha[idx] : 1.f);
    return cumulated_log64(a_out);
}
// a token's beta; zero counts as 1e-30 (as the decays' floor: nothing that is kept changes, and u / beta is v minus what the state already holds)
__device__ __forceinline__ float beta_of(const float* beta, int64_t idx, bool in) { return in ? decay_at_least(beta[idx]) : 0.f; }

// The scans' workgroups: the four value ranges of a head read the same Kw / P / Q / K, so they go to one XCD (workgroups are dealt to the eight XCDs in turn), side by side.
__device__ __forceinline__ bool scan_place(int heads, int& head, int& v0) {
    const int id = blockIdx.x;
    head = (id >> 5) * 8 + (id & 7);
    v0 = ((id >> 3) & 3) * GV;
    return head < heads;
}
static_assert(GD / GV == 4, "four value ranges to a head");

// ------------------------------------------------------------------------------------------- prep: everything of a chunk that needs no state
__global__ __launch_bounds__(256, 2) void gdrc_prep_kernel(int S, int n0, int keep, int Hqk, int Hv, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                                                           const bf16_t* __restrict__ v, int64_t ldv, const float* __restrict__ beta, const float* __restrict__ alpha,
                                                           float* __restrict__ saved, float qscale) {
    __shared__ __attribute__((aligned(16))) bf16_t Ks[GC][GD + 8];
    __shared__ __attribute__((aligned(16))) bf16_t Vs[GC][GD + 8];
    __shared__ __attribute__((aligned(16))) float N[GC][GC + 4];
    __shared__ __attribute__((aligned(16))) float T[GC][GC + 4];
    __shared__ double gd[GC];
    __shared__ float be[GC], gam[GC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5;
    const int n = blockIdx.x, h = blockIdx.y, b = blockIdx.z, hq = h / (Hv / Hqk), t0 = (n0 + n) * GC, cnt = min(GC, S - t0);
    const int64_t tok0 = (int64_t)b * S + t0, ldqk = (int64_t)Hqk * GD;
    const bf16_t *qp = q + tok0 * ldqk + hq * GD, *kp = k + tok0 * ldqk + hq * GD, *vp = v + tok0 * ldv + (int64_t)h * GD;
    float* blk = saved + (((int64_t)b * Hv + h) * gridDim.x + n) * (keep ? G_BLOCK : G_SMALL) + (keep ? G_KW : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int idx = tid + 256 * i, r = idx >> 4, c = (idx & 15) * 8;
        u32x4 kv = {0u, 0u, 0u, 0u}, vv = {0u, 0u, 0u, 0u};
        if (r < cnt) {
            kv = *reinterpret_cast<const u32x4*>(kp + r * ldqk + c);
            vv = *reinterpret_cast<const u32x4*>(vp + r * ldv + c);
        }
        *reinterpret_cast<u32x4*>(&Ks[r][c]) = kv;
        *reinterpret_cast<u32x4*>(&Vs[r][c]) = vv;
    }
    if (wave == 0) {
        float a;
        const double g = cumulated_log(alpha, (tok0 + lane) * Hv + h, lane < cnt, a);
        const double g63 = __shfl(g, 63, 64);
        gd[lane] = g;
        be[lane] = beta_of(beta, (tok0 + lane) * Hv + h, lane < cnt);
        gam[lane] = exp_of(g);
        blk[C_GAM + lane] = exp_of(g);
        blk[C_GAM + GC + lane] = exp_of(g63 - g);
    }
    __syncthreads();
    {  // K K^T and Q K^T: wave = tile (ti, tj); the tile above the diagonal is zero
        const int ti = wave >> 1, tj = wave & 1;
        f32x16 kk = zero16(), qk = zero16();
        if (wave != 1) {
            const int qr = 32 * ti + ln;
#pragma unroll
            for (int c = 0; c < GD; c += 16) {
                const u32x4 qw = qr < cnt ? *reinterpret_cast<const u32x4*>(qp + qr * ldqk + c + 8 * hf) : u32x4{0u, 0u, 0u, 0u};
                const bf16x8 af = *reinterpret_cast<const bf16x8*>(&Ks[32 * ti + ln][c + 8 * hf]), bf = *reinterpret_cast<const bf16x8*>(&Ks[32 * tj + ln][c + 8 * hf]);
                kk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf, kk, 0, 0, 0);
                qk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, qw), bf, qk, 0, 0, 0);
            }
        }
        const int j = 32 * tj + ln;
        const double gj = gd[j];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = 32 * ti + c_row(e, hf);
            const float D = i >= j ? exp_of(gd[i] - gj) : 0.f;
            N[i][j] = i > j ? be[i] * kk[e] * D : 0.f;
            blk[C_P + i * GC + j] = i >= j ? qscale * qk[e] * D : 0.f;
        }
    }
    __syncthreads();
    invert_unit_lower64(N, T);
    if (keep) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 4, c = (idx & 15) * 4;
            *reinterpret_cast<f32x4*>(blk + C_R + r * GC + c) = *reinterpret_cast<const f32x4*>(&T[r][c]);
        }
    }
    {  // Uv = R (b V), Kw = R (b gam K): wave = 32 columns, both row halves (the upper one ends at token 32)
        f32x16 u0 = zero16(), u1 = zero16(), w0 = zero16(), w1 = zero16(), ut = zero16(), wt = zero16();
        const int col = 32 * wave + ln;
#pragma unroll
        for (int kb = 0; kb < GC; kb += 8) {
            const f32x4 a1 = *reinterpret_cast<const f32x4*>(&T[32 + ln][kb + 4 * hf]);
            f32x4 a0 = {0.f, 0.f, 0.f, 0.f};
            if (kb < 32) a0 = *reinterpret_cast<const f32x4*>(&T[ln][kb + 4 * hf]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int t = kb + 4 * hf + j;
                const float bv = bf2f(Vs[t][col]) * be[t], bk = bf2f(Ks[t][col]) * (be[t] * gam[t]);
                u1 = mfma2(a1[j], bv, u1);
                w1 = mfma2(a1[j], bk, w1);
                if (kb < 32) {
                    u0 = mfma2(a0[j], bv, u0);
                    w0 = mfma2(a0[j], bk, w0);
                }
            }
            if (kb == 24) add16(ut, u1), add16(wt, w1);
        }
        add16(u1, ut);
        add16(w1, wt);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int r = c_row(e, hf);
            blk[C_U + r * GD + col] = u0[e];
            blk[C_U + (32 + r) * GD + col] = u1[e];
            blk[r * GD + col] = w0[e];
            blk[(32 + r) * GD + col] = w1[e];
        }
    }
}

// ------------------------------------------------------------------------------------------- scan: the state chunk by chunk, 32 value rows per workgroup
// Waves 0, 1 take Kw S^T (row halves), waves 2, 3 Q S^T and then P U; the state's four 32-column tiles go one to a wave.  Bound: the chain
// of chunks -- reads in flight, then two products behind two barriers.  Everything a chunk reads first is requested at its top, all at once: 172 us at 8 x 708 tokens x 16
// heads (167 before its chains were cut, and so measured: requested a chunk ahead 189, the registers spill; in two halves 187; the value ranges of a head on different XCDs 177).
__global__ __launch_bounds__(256, 2) void gdrc_scan_kernel(int heads, int S, int n0, int NC, int Hqk, int Hv, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                                                           const bf16_t* __restrict__ v, int64_t ldv, const float* __restrict__ beta, const float* __restrict__ alpha, float* __restrict__ saved,
                                                           bf16_t* __restrict__ o, const float* initial_state, float* final_state, int keep, float qscale) {
    __shared__ __attribute__((aligned(16))) float Ss[GV][GD + 4];
    __shared__ __attribute__((aligned(16))) float Us[GC][GV + 8];
    __shared__ __attribute__((aligned(16))) bf16_t Ks[GC][GD + 8];
    __shared__ float gg[2 * GC];
    __shared__ int lost[2];  // a chunk's flag: set by its U, cleared a chunk later
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5, rh = wave & 1;
    int at, v0;
    if (!scan_place(heads, at, v0)) return;
    const int h = at % Hv, b = at / Hv, hq = h / (Hv / Hqk);
    const bool qside = wave >= 2;
    const int64_t ldqk = (int64_t)Hqk * GD, head = at;
    const bf16_t *qp = q + (int64_t)b * S * ldqk + hq * GD, *kp = k + (int64_t)b * S * ldqk + hq * GD;
    const int64_t block = keep ? G_BLOCK : G_SMALL;
    float* base = saved + head * NC * block + (keep ? G_KW : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int idx = tid + 256 * i, r = idx >> 5, c = (idx & 31) * 4;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        if (initial_state) s = *reinterpret_cast<const f32x4*>(initial_state + (head * GD + v0 + r) * GD + c);
        *reinterpret_cast<f32x4*>(&Ss[r][c]) = s;
    }
    if (tid < 2) lost[tid] = 0;
    int n = 0;
    for (; n < NC; ++n) {
        float* blk = base + n * block;
        const int t0 = (n0 + n) * GC, cnt = min(GC, S - t0);
        // a Kw row (waves 0, 1) or, in half the words, a Q row (waves 2, 3) in fragment form, all of it in flight at once
        const int row = 32 * rh + ln;
        const float* kw = blk + row * GD + 4 * hf;
        f32x4 fr[16];
        if (!qside) {
#pragma unroll
            for (int i = 0; i < 16; ++i) fr[i] = *reinterpret_cast<const f32x4*>(kw + 8 * i);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const u32x2 w0 = row4(qp + t0 * ldqk, ldqk, row, cnt, 16 * i + 4 * hf), w1 = row4(qp + t0 * ldqk, ldqk, row, cnt, 16 * i + 8 + 4 * hf);
                fr[i] = f32x4{__uint_as_float(w0[0]), __uint_as_float(w0[1]), __uint_as_float(w1[0]), __uint_as_float(w1[1])};
            }
        }
        u32x4 kr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 4, c = (idx & 15) * 8;
            kr[i] = r < cnt ? *reinterpret_cast<const u32x4*>(kp + (t0 + r) * ldqk + c) : u32x4{0u, 0u, 0u, 0u};
        }
        const float gr = tid < 2 * GC ? blk[C_GAM + tid] : 0.f;
        __syncthreads();  // the state is whole, the last chunk's K and U are read
        if (tid < 2 * GC) gg[tid] = gr;
        if (tid == 0) lost[(n + 1) & 1] = 0;
        if (keep) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int idx = tid + 256 * i, r = idx >> 5, c = (idx & 31) * 4;
                *reinterpret_cast<f32x4*>(blk - G_KW + (v0 + r) * GD + c) = *reinterpret_cast<const f32x4*>(&Ss[r][c]);
            }
        }
        f32x16 uv = zero16(), acc = zero16();
        if (!qside) {
#pragma unroll
            for (int e = 0; e < 16; ++e) uv[e] = blk[C_U + (32 * rh + c_row(e, hf)) * GD + v0 + ln];
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const f32x4 s = *reinterpret_cast<const f32x4*>(&Ss[ln][8 * i + 4 * hf]);
            f32x4 a;
            if (!qside) a = fr[i];
            else a = widen4(i & 1 ? u32x2{__float_as_uint(fr[i >> 1][2]), __float_as_uint(fr[i >> 1][3])} : u32x2{__float_as_uint(fr[i >> 1][0]), __float_as_uint(fr[i >> 1][1])});
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = mfma2(a[j], s[j], acc);
            if (i == 7) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    uv[e] -= acc[e];
                    acc[e] = 0.f;
                }
            }
            if (i % 4 == 3) asm volatile("" ::: "memory");  // keep the state reads of later steps where they are: all sixteen at once cost more registers than there are
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 4, c = (idx & 15) * 8;
            *reinterpret_cast<u32x4*>(&Ks[r][c]) = kr[i];
        }
        f32x4 pr[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) pr[i] = qside ? *reinterpret_cast<const f32x4*>(blk + C_P + (32 * rh + ln) * GC + 8 * i + 4 * hf) : f32x4{0.f, 0.f, 0.f, 0.f};
        if (!qside) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = 32 * rh + c_row(e, hf);
                acc[e] = uv[e] - acc[e];
                Us[r][ln] = acc[e];
                blk[C_U + r * GD + v0 + ln] = acc[e];
            }
            if (__any(lost16(acc)) && lane == 0) lost[n & 1] = 1;
        }
        __syncthreads();
        const int gone = lost[n & 1];
        if (qside) {
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = (acc[e] - uv[e]) * (gg[32 * rh + c_row(e, hf)] * qscale);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (rh == 0 && i >= 4) break;  // P is lower triangular
#pragma unroll
                for (int j = 0; j < 4; ++j) acc = mfma2(pr[i][j], Us[8 * i + 4 * hf + j][ln], acc);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = 32 * rh + c_row(e, hf);
                if (r < cnt) o[((int64_t)b * S + t0 + r) * Hv * GD + (int64_t)h * GD + v0 + ln] = f2bf(acc[e]);
            }
        }
        if (gone) break;  // (the same for the whole workgroup)
        f32x16 s;
        const float gC = gg[GC - 1];
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = gC * Ss[c_row(e, hf)][32 * wave + ln];
#pragma unroll 2
        for (int kb = 0; kb < GC; kb += 8)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int t = kb + 4 * hf + j;
                s = mfma2(Us[t][ln] * gg[GC + t], bf2f(Ks[t][32 * wave + ln]), s);
            }
#pragma unroll
        for (int e = 0; e < 16; ++e) Ss[c_row(e, hf)][32 * wave + ln] = s[e];  // read by this wave alone since the last barrier
    }
    // A chunk whose U is not finite, and all behind it: the recurrence itself, eight lanes to a value row.  (In a chunk the triangles' zeros are multiplied, not skipped: a token's key,
    // value, decay or beta that is not finite reaches U and with it the rows before it.  A query reaches its own row alone.)
    if (n < NC) {
        __threadfence();
        __syncthreads();  // what the chunk wrote of its outputs and U lies below what comes
        const int r = tid >> 3, c = (tid & 7) * 16;
        float st[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) st[i] = Ss[r][c + i];
        for (int t = (n0 + n) * GC; t < min(S, (n0 + NC) * GC); ++t) {
            float* blk = base + (t / GC - n0) * block;
            if (keep && t % GC == 0) {
#pragma unroll
                for (int i = 0; i < 16; ++i) (blk - G_KW)[(v0 + r) * GD + c + i] = st[i];
            }
            const int64_t at_ = ((int64_t)b * S + t) * Hv + h;
            const float a = alpha[at_];
            float u = 0.f, x = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                st[i] *= a;
                u = fmaf(st[i], bf2f(kp[t * ldqk + c + i]), u);
            }
            u = beta[at_] * (bf2f(v[((int64_t)b * S + t) * ldv + (int64_t)h * GD + v0 + r]) - lanes_sum<8>(u));
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                st[i] = fmaf(u, bf2f(kp[t * ldqk + c + i]), st[i]);
                x = fmaf(st[i], bf2f(qp[t * ldqk + c + i]), x);
            }
            x = lanes_sum<8>(x) * qscale;
            if (c == 0) {
                o[at_ * GD + v0 + r] = f2bf(x);
                blk[C_U + t % GC * GD + v0 + r] = u;
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) Ss[r][c + i] = st[i];
    }
    if (final_state) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 5, c = (idx & 31) * 4;
            *reinterpret_cast<f32x4*>(final_state + (head * GD + v0 + r) * GD + c) = *reinterpret_cast<const f32x4*>(&Ss[r][c]);
        }
    }
}

// ------------------------------------------------------------------------------------------- reverse scan: the state's gradient, 32 value rows per workgroup
__global__ __launch_bounds__(256, 2) void gdrc_rscan_kernel(int heads, int S, int NC, int Hqk, int Hv, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const float* __restrict__ saved,
                                                            const bf16_t* __restrict__ d_o, float* __restrict__ ws, const float* d_final, float* d_initial, float qscale) {
    __shared__ __attribute__((aligned(16))) float Ss[GV][GD + 4];
    __shared__ float Us[GC][GV + 4];
    __shared__ __attribute__((aligned(16))) float Ws[GC][GD + 4];
    __shared__ __attribute__((aligned(16))) bf16_t Qs[GC][GD + 8];
    __shared__ __attribute__((aligned(16))) bf16_t Os[GC][GV];  // (unpadded: two workgroups of this kernel fill a CU's LDS to the byte)
    __shared__ float gg[2 * GC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5, rh = wave & 1, kh = wave >> 1;
    int at, v0;
    if (!scan_place(heads, at, v0)) return;
    const int h = at % Hv, b = at / Hv, hq = h / (Hv / Hqk);
    const int64_t ldqk = (int64_t)Hqk * GD, ldo = (int64_t)Hv * GD, head = at;
    const bf16_t *qp = q + (int64_t)b * S * ldqk + hq * GD, *kp = k + (int64_t)b * S * ldqk + hq * GD, *gp = d_o + (int64_t)b * S * ldo + (int64_t)h * GD + v0;
    const float* base = saved + head * NC * G_BLOCK;
    float* wbase = ws + head * NC * W_BLOCK;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int idx = tid + 256 * i, r = idx >> 5, c = (idx & 31) * 4;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        if (d_final) s = *reinterpret_cast<const f32x4*>(d_final + (head * GD + v0 + r) * GD + c);
        *reinterpret_cast<f32x4*>(&Ss[r][c]) = s;
    }
    f32x4 wr[8];
    u32x4 qr[4], gr;
    float gv = 0.f;
    auto request = [&](int n) {
        const float* blk = base + (int64_t)n * G_BLOCK;
        const int t0 = n * GC, cnt = min(GC, S - t0);
#pragma unroll
        for (int i = 0; i < 8; ++i) wr[i] = *reinterpret_cast<const f32x4*>(blk + G_KW + (tid + 256 * i) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 4, c = (idx & 15) * 8;
            qr[i] = r < cnt ? *reinterpret_cast<const u32x4*>(qp + (t0 + r) * ldqk + c) : u32x4{0u, 0u, 0u, 0u};
        }
        const int r = tid >> 2, c = (tid & 3) * 8;
        gr = r < cnt ? *reinterpret_cast<const u32x4*>(gp + (t0 + r) * ldo + c) : u32x4{0u, 0u, 0u, 0u};
        if (tid < 2 * GC) gv = blk[G_GAM + tid];
    };
    request(NC - 1);
    for (int n = NC - 1; n >= 0; --n) {
        const float* blk = base + (int64_t)n * G_BLOCK;
        float* wblk = wbase + (int64_t)n * W_BLOCK;
        const int t0 = n * GC, cnt = min(GC, S - t0);
        __syncthreads();  // dS is whole, the last chunk's operands are read
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = tid + 256 * i, r = idx >> 5, c = (idx & 31) * 4;
            *reinterpret_cast<f32x4*>(&Ws[r][c]) = wr[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 4, c = (idx & 15) * 8;
            *reinterpret_cast<u32x4*>(&Qs[r][c]) = qr[i];
        }
        {
            const int r = tid >> 2, c = (tid & 3) * 8;
            *reinterpret_cast<u32x4*>(&Os[r][c]) = gr;
        }
        if (tid < 2 * GC) gg[tid] = gv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 5, c = (idx & 31) * 4;
            *reinterpret_cast<f32x4*>(wblk + (v0 + r) * GD + c) = *reinterpret_cast<const f32x4*>(&Ss[r][c]);
        }
        __syncthreads();
        // dU = P^T dO + Gp (K dS^T): wave = (row half, half of the contraction); the two halves of a contraction meet in LDS
        f32x16 u = zero16(), ut = zero16(), pt = zero16();
        {
            f32x4 kf[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) kf[i] = widen4(row4(kp + t0 * ldqk, ldqk, 32 * rh + ln, cnt, 64 * kh + 8 * i + 4 * hf));
            float pf[16];
            const bool some = !(rh == 1 && kh == 0);  // P[i][j] with i < 32 <= j is zero
            if (some) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) pf[4 * i + j] = blk[G_P + (32 * kh + 8 * i + 4 * hf + j) * GC + 32 * rh + ln];
            }
            if (n > 0) request(n - 1);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const f32x4 s = *reinterpret_cast<const f32x4*>(&Ss[ln][64 * kh + 8 * i + 4 * hf]);
#pragma unroll
                for (int j = 0; j < 4; ++j) u = mfma2(kf[i][j], s[j], u);
                if (i == 3) add16(ut, u);
            }
            add16(u, ut);
            if (some) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) pt = mfma2(pf[4 * i + j], bf2f(Os[32 * kh + 8 * i + 4 * hf + j][ln]), pt);
            }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) u[e] = fmaf(gg[GC + 32 * rh + c_row(e, hf)], u[e], pt[e]);
        if (kh == 1) {
#pragma unroll
            for (int e = 0; e < 16; ++e) Us[32 * rh + c_row(e, hf)][ln] = u[e];
        }
        __syncthreads();
        if (kh == 0) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = 32 * rh + c_row(e, hf);
                const float d = u[e] + Us[r][ln];
                Us[r][ln] = d;
                wblk[W_DU + r * GD + v0 + ln] = d;
            }
        }
        __syncthreads();
        f32x16 s;
        const float gC = gg[GC - 1];
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = gC * Ss[c_row(e, hf)][32 * wave + ln];
        // from the last token to the first: what reaches the chunk's start grows that way (the other way around the large terms come first and every later sum rounds at their size)
#pragma unroll 2
        for (int kb = GC - 8; kb >= 0; kb -= 8)
#pragma unroll
            for (int j = 3; j >= 0; --j) {
                const int t = kb + 4 * hf + j;
                s = mfma2(bf2f(Os[t][ln]) * (gg[t] * qscale), bf2f(Qs[t][32 * wave + ln]), s);
                s = mfma2(-Us[t][ln], Ws[t][32 * wave + ln], s);
            }
#pragma unroll
        for (int e = 0; e < 16; ++e) Ss[c_row(e, hf)][32 * wave + ln] = s[e];  // read by this wave alone since the barrier behind dU
    }
    if (d_initial) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + 256 * i, r = idx >> 5, c = (idx & 31) * 4;
            *reinterpret_cast<f32x4*>(d_initial + (head * GD + v0 + r) * GD + c) = *reinterpret_cast<const f32x4*>(&Ss[r][c]);
        }
    }
}

// ------------------------------------------------------------------------------------------- the rest of the backward: one workgroup per chunk and head
__global__ __launch_bounds__(256, 2) void gdrc_bwd_kernel(int S, int NC, int Hqk, int Hv, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
                                                          int64_t ldv, const float* __restrict__ beta, const float* __restrict__ alpha, const float* __restrict__ saved,
                                                          const float* __restrict__ ws, const bf16_t* __restrict__ d_o, bf16_t* __restrict__ dq, bf16_t* __restrict__ dk,
                                                          bf16_t* __restrict__ dv, int64_t lddv, float* __restrict__ dbeta, float* __restrict__ dalpha, float* __restrict__ pdq,
                                                          float* __restrict__ pdk, float qscale) {
    constexpr int LM = GC + 4, LZ = GC + 2;
    __shared__ __attribute__((aligned(16))) float Z[GC][GD + 4];   // -dU S0; later Y, then d(Q K^T) (first half), and the pairs' decay terms (second half)
    __shared__ __attribute__((aligned(16))) float M1[GC][LM];      // dR; later d(K K^T) + its transpose
    __shared__ __attribute__((aligned(16))) float M2[GC][LM];      // R
    __shared__ double gd[GC];
    __shared__ float be[GC], al[GC], gam[GC], gp[GC], redG[4][GC], redP[4][GC], redB[4][GC], dss[4];
    float(*M3)[LZ] = reinterpret_cast<float(*)[LZ]>(&Z[0][0]);
    float(*ME)[LZ] = reinterpret_cast<float(*)[LZ]>(&Z[0][0] + GC * LZ);
    static_assert(2 * GC * LZ <= GC * (GD + 4), "both late matrices fit the early one's space");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5;
    const int n = blockIdx.x, h = blockIdx.y, b = blockIdx.z, hq = h / (Hv / Hqk), t0 = n * GC, cnt = min(GC, S - t0);
    const int64_t tok0 = (int64_t)b * S + t0, ldqk = (int64_t)Hqk * GD, ldo = (int64_t)Hv * GD, head = (int64_t)b * Hv + h;
    const bf16_t *qp = q + tok0 * ldqk + hq * GD, *kp = k + tok0 * ldqk + hq * GD, *vp = v + tok0 * ldv + (int64_t)h * GD, *op = d_o + tok0 * ldo + (int64_t)h * GD;
    const float* blk = saved + (head * NC + n) * G_BLOCK;
    const float *dS = ws + (head * NC + n) * W_BLOCK, *dU = dS + W_DU, *Up = blk + G_U;
    const int col = 32 * wave + ln;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int idx = tid + 256 * i, r = idx >> 4, c = (idx & 15) * 4;
        *reinterpret_cast<f32x4*>(&M2[r][c]) = *reinterpret_cast<const f32x4*>(blk + G_R + r * GC + c);
    }
    if (wave == 0) {
        float a;
        gd[lane] = cumulated_log(alpha, (tok0 + lane) * Hv + h, lane < cnt, a);
        al[lane] = a;
        be[lane] = beta_of(beta, (tok0 + lane) * Hv + h, lane < cnt);
        gam[lane] = blk[G_GAM + lane];
        gp[lane] = blk[G_GAM + GC + lane];
    }
    {  // Z = -dU S0: wave = 32 columns, both row halves, contraction over the value rows straight from memory (a state row's 32 columns are one line)
        f32x16 z[2] = {zero16(), zero16()};
        f32x4 du[2];
        float s0[4];
        auto request = [&](int kb) {
#pragma unroll
            for (int r = 0; r < 2; ++r) du[r] = *reinterpret_cast<const f32x4*>(dU + (32 * r + ln) * GD + kb + 4 * hf);
#pragma unroll
            for (int j = 0; j < 4; ++j) s0[j] = blk[(kb + 4 * hf + j) * GD + col];
        };
        request(0);
#pragma unroll 2
        for (int kb = 0; kb < GD; kb += 8) {
            const f32x4 c0 = -du[0], c1 = -du[1], cs = {s0[0], s0[1], s0[2], s0[3]};
            if (kb + 8 < GD) request(kb + 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                z[0] = mfma2(c0[j], cs[j], z[0]);
                z[1] = mfma2(c1[j], cs[j], z[1]);
            }
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int e = 0; e < 16; ++e) Z[32 * r + c_row(e, hf)][col] = z[r][e];
    }
    __syncthreads();
    // the 64 x 64 matrices: wave = tile (ti, tj)
    const int ti = wave >> 1, tj = wave & 1, j0 = 32 * tj + ln;
    f32x16 lkk, e1, dqk;
    {
        f32x16 kk = zero16(), qk = zero16(), dP = zero16(), dT = zero16(), tz = zero16(), dPt = zero16();
        if (wave != 1) {
            const int ri = 32 * ti + ln, rj = 32 * tj + ln;
#pragma unroll
            for (int c = 0; c < GD; c += 16) {
                const u32x4 z4 = {0u, 0u, 0u, 0u};
                const u32x4 qi = ri < cnt ? *reinterpret_cast<const u32x4*>(qp + ri * ldqk + c + 8 * hf) : z4, ki = ri < cnt ? *reinterpret_cast<const u32x4*>(kp + ri * ldqk + c + 8 * hf) : z4,
                            kj = rj < cnt ? *reinterpret_cast<const u32x4*>(kp + rj * ldqk + c + 8 * hf) : z4;
                kk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ki), __builtin_bit_cast(bf16x8, kj), kk, 0, 0, 0);
                qk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, qi), __builtin_bit_cast(bf16x8, kj), qk, 0, 0, 0);
            }
#pragma unroll 2
            for (int kb = 0; kb < GD; kb += 8) {
                const f32x4 oi = widen4(row4(op, ldo, ri, cnt, kb + 4 * hf)), uj = *reinterpret_cast<const f32x4*>(Up + rj * GD + kb + 4 * hf);
                const f32x4 di = *reinterpret_cast<const f32x4*>(dU + ri * GD + kb + 4 * hf), vj = widen4(row4(vp, ldv, rj, cnt, kb + 4 * hf));
                const f32x4 zi = *reinterpret_cast<const f32x4*>(&Z[ri][kb + 4 * hf]), kj = widen4(row4(kp, ldqk, rj, cnt, kb + 4 * hf));
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    dP = mfma2(oi[j], uj[j], dP);
                    dT = mfma2(di[j], vj[j], dT);
                    tz = mfma2(zi[j], kj[j], tz);
                }
                if ((kb & 24) == 24) add16(dPt, dP);
            }
            add16(dP, dPt);
        }
        const double gj = gd[j0];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = 32 * ti + c_row(e, hf);
            const bool in = i >= j0;
            const float D = in ? exp_of(gd[i] - gj) : 0.f, t = in ? dT[e] + gam[j0] * tz[e] : 0.f, p = in ? qscale * dP[e] : 0.f;
            lkk[e] = i > j0 ? kk[e] * D : 0.f;
            e1[e] = p * (qk[e] * D);
            dqk[e] = p * D;
            M1[i][j0] = t * be[j0];
        }
    }
    __syncthreads();
    f32x16 w[2];  // dK, from here on
    {  // dV = T^T dU, d(gam K) = T^T Z: wave = 32 columns
        f32x16 a[2] = {zero16(), zero16()}, g[2] = {zero16(), zero16()}, at = zero16(), gt = zero16();
#pragma unroll 2
        for (int kb = 0; kb < GC; kb += 8) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = kb + 4 * hf + j;
                const float bu = dU[i * GD + col], bz = Z[i][col], r0 = M2[i][ln], r1 = M2[i][32 + ln];
                a[0] = mfma2(r0, bu, a[0]);
                g[0] = mfma2(r0, bz, g[0]);
                if (kb >= 32) {  // R is lower triangular
                    a[1] = mfma2(r1, bu, a[1]);
                    g[1] = mfma2(r1, bz, g[1]);
                }
            }
            if (kb == 24) add16(at, a[0]), add16(gt, g[0]);
        }
        add16(a[0], at);
        add16(g[0], gt);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int i = 32 * r + c_row(e, hf);
                // d(beta): what reaches u = beta (v - the state's answer to k) times that difference, which is u / beta
                const float sb = half_sum(a[r][e] * Up[i * GD + col]);
                if (ln == 0) redB[wave][i] = sb;
                if (i < cnt) dv[(tok0 + i) * lddv + (int64_t)h * GD + col] = f2bf(be[i] * a[r][e]);
                const float d = be[i] * g[r][e];
                w[r][e] = gam[i] * d;
                const float sg = half_sum(d * one(kp, ldqk, i, cnt, col));
                if (ln == 0) redG[wave][i] = sg;
            }
    }
    __syncthreads();  // Z is done with
    {  // Y = dR R^T
        f32x16 y = zero16();
        const int kend = ti && tj ? GC : 32;
        for (int kb = 0; kb < kend; kb += 8) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(&M1[32 * ti + ln][kb + 4 * hf]), r = *reinterpret_cast<const f32x4*>(&M2[32 * tj + ln][kb + 4 * hf]);
#pragma unroll
            for (int j = 0; j < 4; ++j) y = mfma2(a[j], r[j], y);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) M3[32 * ti + c_row(e, hf)][j0] = y[e];
    }
    __syncthreads();
    f32x16 dn = zero16();
    if (wave != 1) {  // dN = -R^T Y
        for (int kb = 32 * ti; kb < GC; kb += 8)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = kb + 4 * hf + j;
                dn = mfma2(M2[i][32 * ti + ln], M3[i][32 * tj + ln], dn);
            }
    }
    __syncthreads();  // dR and Y are done with
    if (wave != 1) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = 32 * ti + c_row(e, hf);
            const float d = i > j0 ? -dn[e] : 0.f;
            const float dl = be[i] * d, D = i > j0 ? exp_of(gd[i] - gd[j0]) : 0.f;
            if (i > j0) M1[i][j0] = M1[j0][i] = dl * D;
            else if (i == j0) M1[i][i] = 0.f;
            M3[i][j0] = dqk[e];
            ME[i][j0] = fmaf(dl, lkk[e], e1[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = c_row(e, hf);
            M3[i][j0] = 0.f;
            ME[i][j0] = 0.f;
        }
    }
    __syncthreads();
    // dQ = scale gam (dO S0), dK += Gp (U dS): contraction over the value rows, straight from memory as above
    f32x16 x[2] = {zero16(), zero16()};
    {
        f32x16 y[2] = {zero16(), zero16()};
        float sds = 0.f;
        u32x2 ox[2];
        f32x4 ur[2];
        float s0[4], s1[4];
        auto request = [&](int kb) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                ox[r] = row4(op, ldo, 32 * r + ln, cnt, kb + 4 * hf);
                ur[r] = *reinterpret_cast<const f32x4*>(Up + (32 * r + ln) * GD + kb + 4 * hf);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s0[j] = blk[(kb + 4 * hf + j) * GD + col];
                s1[j] = dS[(kb + 4 * hf + j) * GD + col];
            }
        };
        request(0);
#pragma unroll 2
        for (int kb = 0; kb < GD; kb += 8) {
            const f32x4 a0 = widen4(ox[0]), a1 = widen4(ox[1]), u0 = ur[0], u1 = ur[1], c0 = {s0[0], s0[1], s0[2], s0[3]}, c1 = {s1[0], s1[1], s1[2], s1[3]};
            if (kb + 8 < GD) request(kb + 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sds = fmaf(c0[j], c1[j], sds);
                x[0] = mfma2(a0[j], c0[j], x[0]);
                x[1] = mfma2(a1[j], c0[j], x[1]);
                y[0] = mfma2(u0[j], c1[j], y[0]);
                y[1] = mfma2(u1[j], c1[j], y[1]);
            }
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int i = 32 * r + c_row(e, hf);
                const float qx = qscale * x[r][e];
                const float sg = half_sum(qx * one(qp, ldqk, i, cnt, col)), sp = half_sum(y[r][e] * one(kp, ldqk, i, cnt, col));
                if (ln == 0) {
                    redG[wave][i] += sg;
                    redP[wave][i] = sp;
                }
                x[r][e] = gam[i] * qx;
                w[r][e] = fmaf(gp[i], y[r][e], w[r][e]);
            }
        sds = half_sum(sds);
        sds += __shfl_xor(sds, 32, 64);
        if (lane == 0) dss[wave] = sds;
    }
    // dK += (dKK + dKK^T) K + dQK^T Q, dQ += dQK K
#pragma unroll 2
    for (int kb = 0; kb < GC; kb += 8) {
        const f32x4 s0 = *reinterpret_cast<const f32x4*>(&M1[ln][kb + 4 * hf]), s1 = *reinterpret_cast<const f32x4*>(&M1[32 + ln][kb + 4 * hf]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = kb + 4 * hf + j;
            const float kf = one(kp, ldqk, t, cnt, col), qf = one(qp, ldqk, t, cnt, col);
            w[0] = mfma2(s0[j], kf, w[0]);
            w[1] = mfma2(s1[j], kf, w[1]);
            w[0] = mfma2(M3[t][ln], qf, w[0]);
            x[1] = mfma2(M3[32 + ln][t], kf, x[1]);
            if (kb >= 32) w[1] = mfma2(M3[t][32 + ln], qf, w[1]);
            else x[0] = mfma2(M3[ln][t], kf, x[0]);
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = 32 * r + c_row(e, hf);
            if (i >= cnt) continue;
            if (pdq) {  // several value heads share a q / k head: per value head, summed afterwards
                const int64_t at = (head * S + t0 + i) * GD + col;
                pdq[at] = x[r][e];
                pdk[at] = w[r][e];
            } else {
                dq[(tok0 + i) * ldqk + hq * GD + col] = f2bf(x[r][e]);
                dk[(tok0 + i) * ldqk + hq * GD + col] = f2bf(w[r][e]);
            }
        }
    // d(log alpha_t): every pair (i, j) with j < t <= i, what reaches token i >= t from the chunk's first state, what token j < t leaves in its last, and the state passing through
    if (tid < GC) {
        double run = 0.;
        float row[GC];
#pragma unroll
        for (int j = 0; j < GC; ++j) row[j] = ME[tid][j];
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            const float c = row[j];
            ME[tid][j] = (float)run;  // sum over the columns before j
            run += c;
        }
    }
    __syncthreads();
    if (tid < cnt) {
        const int t = tid;
        double s = gam[GC - 1] * ((dss[0] + dss[1]) + (dss[2] + dss[3]));
        for (int i = 0; i < GC; ++i) {
            if (i >= t) s += ME[i][t] + gam[i] * ((redG[0][i] + redG[1][i]) + (redG[2][i] + redG[3][i]));
            else s += gp[i] * ((redP[0][i] + redP[1][i]) + (redP[2][i] + redP[3][i]));
        }
        dalpha[(tok0 + t) * Hv + h] = (float)s / al[t];
        dbeta[(tok0 + t) * Hv + h] = ((redB[0][t] + redB[1][t]) + (redB[2][t] + redB[3][t])) / be[t];
    }
}

// dq / dk of a q / k head: the sum over its value heads, in order
__global__ __launch_bounds__(256) void gdrc_heads_kernel(int S, int Hqk, int Hv, const float* __restrict__ pdq, const float* __restrict__ pdk, bf16_t* __restrict__ dq,
                                                         bf16_t* __restrict__ dk, int64_t total) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    const int j = (int)(idx % GD), hq = (int)((idx / GD) % Hqk), rep = Hv / Hqk;
    const int64_t tok = idx / ((int64_t)GD * Hqk), b = tok / S, t = tok % S;
    float sq = 0.f, sk = 0.f;
    for (int h = hq * rep; h < (hq + 1) * rep; ++h) {
        const int64_t at = ((b * Hv + h) * S + t) * GD + j;
        sq += pdq[at];
        sk += pdk[at];
    }
    dq[idx] = f2bf(sq);
    dk[idx] = f2bf(sk);
}

}  // namespace

static int check_gdrc(const char* who, int B, int S, int Hqk, int Hv) {
    MI355_REQUIRE(B > 0 && S > 0 && Hqk > 0 && Hv > 0 && Hv % Hqk == 0, "%s: value heads (%d) must be a multiple of q/k heads (%d)", who, Hv, Hqk);
    MI355_REQUIRE(Hv <= 65535 && B <= 65535 && (int64_t)B * Hv <= (1 << 28), "%s: grid limits", who);
    return 0;
}

extern "C" int64_t mi355_gdr_chunked_saved_bytes(int B, int S, int Hv) { return B > 0 && S > 0 && Hv > 0 ? (int64_t)B * Hv * (((int64_t)S + GC - 1) / GC) * G_BLOCK * 4 : 0; }

static int span_chunks(int B, int S, int Hv) {
    const int64_t all = ((int64_t)S + GC - 1) / GC, fit = SPAN_BYTES / ((int64_t)B * Hv * G_SMALL * 4);
    return (int)(fit >= all ? all : fit < 4 ? (all < 4 ? all : 4) : fit);
}
extern "C" int64_t mi355_gdr_chunked_scratch_bytes(int B, int S, int Hv) {
    if (B <= 0 || S <= 0 || Hv <= 0) return 0;
    const int64_t span = span_chunks(B, S, Hv);
    return (int64_t)B * Hv * 4 * (span * G_SMALL + (span * GC < S ? GD * GD : 0));
}

extern "C" int64_t mi355_gdr_chunked_bwd_workspace_bytes(int B, int S, int Hqk, int Hv) {
    if (B <= 0 || S <= 0 || Hqk <= 0 || Hv <= 0) return 0;
    const int64_t blocks = (int64_t)B * Hv * (((int64_t)S + GC - 1) / GC) * W_BLOCK;
    return 4 * (blocks + (Hv > Hqk ? 2 * (int64_t)B * Hv * S * GD : 0));
}

extern "C" int mi355_gdr_chunked_fwd(int B, int S, int Hqk, int Hv, const void* q, const void* k, const void* v, int64_t ldv, const float* beta, const float* alpha, void* o,
                                     float* saved, int64_t saved_bytes, int keep, const float* initial_state, float* final_state, void* stream) {
    if (check_gdrc("gdr_chunked_fwd", B, S, Hqk, Hv)) return 1;
    MI355_REQUIRE(q && k && v && beta && alpha && o && saved && ldv >= (int64_t)Hv * GD && ldv % 8 == 0, "gdr_chunked_fwd: null pointer, or v's row pitch too small or no multiple of 8");
    MI355_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)saved | (uintptr_t)initial_state | (uintptr_t)final_state) & 15) == 0, "gdr_chunked_fwd: operands must be 16-byte aligned");
    MI355_REQUIRE(saved_bytes >= (keep ? mi355_gdr_chunked_saved_bytes(B, S, Hv) : mi355_gdr_chunked_scratch_bytes(B, S, Hv)), "gdr_chunked_fwd: saved buffer too small (%lld bytes)",
                  (long long)saved_bytes);
    const int all = (S + GC - 1) / GC, span = keep ? all : span_chunks(B, S, Hv);
    const float qs = 1.0f / sqrtf((float)GD);
    // several spans: the state travels through final_state, or behind the blocks where nobody asks for it
    float* carry = final_state ? final_state : saved + (int64_t)B * Hv * span * G_SMALL;
    for (int n0 = 0; n0 < all; n0 += span) {
        const int nc = all - n0 < span ? all - n0 : span;
        gdrc_prep_kernel<<<dim3(nc, Hv, B), 256, 0, ST(stream)>>>(S, n0, keep, Hqk, Hv, (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, beta, alpha, saved, qs);
        MI355_LAUNCH_CHECK("gdr_chunked_fwd(prep)");
        gdrc_scan_kernel<<<(B * Hv + 7) / 8 * 32, 256, 0, ST(stream)>>>(B * Hv, S, n0, nc, Hqk, Hv, (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, beta, alpha, saved, (bf16_t*)o,
                                                                          n0 ? carry : initial_state, n0 + nc < all ? carry : final_state, keep, qs);
        MI355_LAUNCH_CHECK("gdr_chunked_fwd");
    }
    return 0;
}

extern "C" int mi355_gdr_chunked_bwd(int B, int S, int Hqk, int Hv, const void* q, const void* k, const void* v, int64_t ldv, const float* beta, const float* alpha, const float* saved,
                                     int64_t saved_bytes, const void* d_o, void* dq, void* dk, void* dv, int64_t lddv, float* dbeta, float* dalpha, void* workspace, int64_t workspace_bytes,
                                     const float* d_final_state, float* d_initial_state, void* stream) {
    if (check_gdrc("gdr_chunked_bwd", B, S, Hqk, Hv)) return 1;
    MI355_REQUIRE(q && k && v && beta && alpha && saved && d_o && dq && dk && dv && dbeta && dalpha && workspace, "gdr_chunked_bwd: null pointer");
    MI355_REQUIRE(ldv >= (int64_t)Hv * GD && ldv % 8 == 0 && lddv >= (int64_t)Hv * GD, "gdr_chunked_bwd: row pitch too small, or v's no multiple of 8");
    MI355_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)saved | (uintptr_t)d_o | (uintptr_t)workspace | (uintptr_t)d_final_state | (uintptr_t)d_initial_state) & 15) == 0,
                  "gdr_chunked_bwd: operands must be 16-byte aligned");
    MI355_REQUIRE(saved_bytes >= mi355_gdr_chunked_saved_bytes(B, S, Hv) && workspace_bytes >= mi355_gdr_chunked_bwd_workspace_bytes(B, S, Hqk, Hv), "gdr_chunked_bwd: saved buffer or workspace too small");
    const int NC = (S + GC - 1) / GC;
    const float qs = 1.0f / sqrtf((float)GD);
    float* ws = (float*)workspace;
    float* pdq = Hv > Hqk ? ws + (int64_t)B * Hv * NC * W_BLOCK : nullptr;
    float* pdk = pdq ? pdq + (int64_t)B * Hv * S * GD : nullptr;
    gdrc_rscan_kernel<<<(B * Hv + 7) / 8 * 32, 256, 0, ST(stream)>>>(B * Hv, S, NC, Hqk, Hv, (const bf16_t*)q, (const bf16_t*)k, saved, (const bf16_t*)d_o, ws, d_final_state, d_initial_state, qs);
    MI355_LAUNCH_CHECK("gdr_chunked_bwd(scan)");
    gdrc_bwd_kernel<<<dim3(NC, Hv, B), 256, 0, ST(stream)>>>(S, NC, Hqk, Hv, (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, beta, alpha, saved, ws, (const bf16_t*)d_o, (bf16_t*)dq,
                                                             (bf16_t*)dk, (bf16_t*)dv, lddv, dbeta, dalpha, pdq, pdk, qs);
    MI355_LAUNCH_CHECK("gdr_chunked_bwd");
    if (pdq) {
        const int64_t total = (int64_t)B * S * Hqk * GD;
        gdrc_heads_kernel<<<(unsigned)((total + 255) / 256), 256, 0, ST(stream)>>>(S, Hqk, Hv, pdq, pdk, (bf16_t*)dq, (bf16_t*)dk, total);
        MI355_LAUNCH_CHECK("gdr_chunked_bwd(heads)");
    }
    return 0;
}
