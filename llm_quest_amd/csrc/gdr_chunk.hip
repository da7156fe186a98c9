// Gated delta rule in chunks of 64 tokens on the fp32 matrix pipe (gfx950 only), forward and backward, for heads of 128 | 128.
//
// The token-by-token recurrence of qwen35.hip (S <- a S + b (v - a S k) k^T, o = S q / sqrt(dk)) is one dependent chain per token: at 8 x 708 tokens x 16 heads its
// forward takes 565 us and its backward 1 470 us a layer, whatever the chip could multiply.  Inside a chunk the recurrence is linear algebra (rows are tokens,
// g = cumulated log decay, D_ij = exp(g_i - g_j), gam = exp(g), Gp_j = exp(g_63 - g_j)):
//     A = tril(diag(b) K K^T . D, -1),  R = (I + A)^-1,  T = R diag(b),  P = scale tril(Q K^T . D),  Uv = T V,  Kw = T (gam K)      -- no state: one workgroup per chunk
//     U = Uv - Kw S^T,  O = scale gam (Q S^T) + P U,  S <- gam_63 S + (Gp U)^T K                                                    -- the chain: one step per chunk
// and the adjoint splits the same way: only dS crosses chunks (dU = P^T dO + Gp (K dS^T), dS <- gam_63 dS + (scale gam dO)^T Q - dU^T Kw), everything else is one
// workgroup per chunk afterwards.  Four kernels: prep, scan, reverse scan (both per 32 value rows of the state: a row never meets another), and the rest.
// All sums are fp32 FMAs on v_mfma_f32_32x32x2_f32 (the two products of bf16 operands alone, K K^T and Q K^T, on the bf16 shape: exact; the scans' products with the state, U, dO of three bf16 parts to an
// fp32 number, which is all of it); the log decays are cumulated
// in fp64, so a difference of two large ones keeps its digits.  d(alpha) is taken from sums over the pairs that span a token -- never as a difference of
// larger sums, so it keeps its digits where alpha is tiny (below 1e-30 alpha counts as 1e-30); d(beta) as what reaches u times u / beta.
// A matrix pipe's chain of 128 products rounds 128 times at its size where lanes sum 16 and meet in a tree; so the chains that show are cut (add16) and the state's gradient
// gathers its terms from the last token to the first.  Distance to 64 bits, token-by-token kernels | here, 256 tokens, geometric mean of four draws: outputs, d(q), d(k), d(v)
// 1.65e-3 | 1.65e-3 (their bf16); fp32: state 7.4e-8 | 8.6e-8, d(state) 9.0e-8 | 9.5e-8 (2.9e-7 from the first token on), d(beta) 1.5e-7 | 1.8e-7 (2.6e-7 with whole chains), d(alpha)
// 1.7e-7 | 2.1e-7 (2.5e-7); decays near one 4.4e-7 | 3.6e-7, 5.0e-7 | 4.9e-7; nearly parallel keys 1.5e-7 | 2.3e-7, 2.1e-7 | 4.4e-7.  Cutting d(q)'s and d(k)'s chains as well:
// d(alpha) 1.9e-7 for 50 us of a backward of 680 (registers spill).
// Three-part products in the scans against fp32 ones there, 64 draws of gates: state 1.41e-7 -> 1.37e-7, d(state) 2.44e-7 -> 2.43e-7, d(beta) 2.67e-7 -> 2.28e-7, d(alpha) 4.82e-7 -> 4.69e-7.
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

__device__ __forceinline__ double cumulated_log(const float* alpha, int64_t idx, bool in, float& a_out) {
    a_out = decay_at_least(in ? alpha[idx] : 1.f);
    return cumulated_log64(a_out);
}
// a token's beta; zero counts as 1e-30 (as the decays' floor: nothing that is kept changes, and u / beta is v minus what the state already holds)
__device__ __forceinline__ float beta_of(const float* beta, int64_t idx, bool in) { return in ? decay_at_least(beta[idx]) : 0.f; }

// four consecutive bf16 of row `r`, or of the last row where `r` lies beyond the sequence (its reader puts zeros there): a load without a branch, which can be under way
__device__ __forceinline__ u32x2 held4(const bf16_t* p, int64_t ld, int r, int cnt, int c) { return *reinterpret_cast<const u32x2*>(p + min(r, cnt - 1) * ld + c); }
__device__ __forceinline__ u32x4 held8(const bf16_t* p, int64_t ld, int r, int cnt, int c) { return *reinterpret_cast<const u32x4*>(p + min(r, cnt - 1) * ld + c); }
// requests stay in front of the products that hide them (short of registers, the compiler moves them down to where they are used)
__device__ __forceinline__ void in_order() { __builtin_amdgcn_sched_barrier(0); }
// a lane's 16 features of a row (transposed accumulators: c_row(4 c, hf) on); wide: the rows lie on 8-byte words
__device__ __forceinline__ void put16(bf16_t* p, const f32x4 (&v)[4], int hf, bool wide) {
    if (wide) {
#pragma unroll
        for (int c = 0; c < 4; ++c) *reinterpret_cast<u32x2*>(p + c_row(4 * c, hf)) = u32x2{pack_bf2(v[c][0], v[c][1]), pack_bf2(v[c][2], v[c][3])};
    } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) p[c_row(e, hf)] = f2bf(v[e >> 2][e & 3]);
    }
}
__device__ __forceinline__ float both_halves(float v) {  // the sum over a lane and its other half's
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

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
// Waves 0, 1 take Kw S^T (row halves), waves 2, 3 Q S^T and then P U; the state's four 32-column tiles go one to a wave, which holds its tile in registers (lane = value row) and leaves
// its three bf16 parts in LDS for the next chunk's products; so does U, for P U.  The state's own sum, S <- gam_63 S + (Gp U)^T K, stays on the fp32 pipe: on the bf16 pipe a chain's
// roundings differ, and where decays are strong the state is one such rounding from exact (4.4e-8 against 5.2e-8 from 64 bits; as it is 4.3e-8), for no time gained.  Bound: the chain of chunks
// and the bytes (8 x 708 tokens x 16 heads: 344 MB, 70 us): two products behind two barriers, every operand of the next chunk requested under this one's second half.
// 172 -> 148 us at 8 x 708 tokens x 16 heads, 58 -> 45 at 333 tokens (the state in fp32 in LDS, read by both sides' fp32 products, a chunk's operands requested at its own top) -> 136 and 37 with a
// loop for each side.
constexpr int SP = GV * (GD + 8), UP = GV * (GC + 8);  // planes of S [32 v][128 k] and U^T [32 v][64 t]
__global__ __launch_bounds__(256, 2) void gdrc_scan_kernel(int heads, int S, int n0, int NC, int Hqk, int Hv, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                                                           const bf16_t* __restrict__ v, int64_t ldv, const float* __restrict__ beta, const float* __restrict__ alpha, float* __restrict__ saved,
                                                           bf16_t* __restrict__ o, const float* initial_state, float* final_state, int keep, float qscale) {
    __shared__ __attribute__((aligned(16))) bf16_t Sp[3 * SP];
    __shared__ __attribute__((aligned(16))) bf16_t Ut[3 * UP];
    __shared__ __attribute__((aligned(16))) float Ug[GV][GC + 4];  // Gp U
    __shared__ __attribute__((aligned(16))) bf16_t Ks[GC][GD + 8];
    __shared__ __attribute__((aligned(16))) float gg[2][256];  // gam and Gp (a word a thread: a condition would take the request with it, to where it is used)
    __shared__ int lost[2];  // a chunk's flag: set by its U, cleared a chunk later
    static_assert(GV * (GD + 4) * 4 <= 3 * SP * 2, "the recurrence's state lies where the planes were");
    float(*Ss)[GD + 4] = reinterpret_cast<float(*)[GD + 4]>(Sp);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 31, hf = lane >> 5, rh = wave & 1;
    int at, v0;
    if (!scan_place(heads, at, v0)) return;
    const int h = at % Hv, b = at / Hv, hq = h / (Hv / Hqk);
    const int64_t ldqk = (int64_t)Hqk * GD, head = at;
    const bf16_t *qp = q + (int64_t)b * S * ldqk + hq * GD, *kp = k + (int64_t)b * S * ldqk + hq * GD;
    const int64_t block = keep ? G_BLOCK : G_SMALL;
    float* base = saved + head * NC * block + (keep ? G_KW : 0);
    const int row = 32 * rh + ln, col = 32 * wave + 4 * hf;  // the lane's row of a fragment; its first column of the state
    f32x16 s;  // S[v0 + ln][32 wave + c_row(e, hf)]
    auto put_state = [&]() {
#pragma unroll
        for (int c = 0; c < 4; ++c) put_parts<SP>(Sp, ln * (GD + 8) + col + 8 * c, s[4 * c], s[4 * c + 1], s[4 * c + 2], s[4 * c + 3]);
    };
    if (tid < 2) lost[tid] = 0;
    int n = 0;
    // The two sides' waves run loops of their own (the barriers are counted by wave, not by place): in one loop a wait for a chunk's operands cannot be counted over the other side's
    // requests and stores and becomes a wait for every store before it.
    auto chunks = [&](auto side) {
        constexpr bool Q = decltype(side)::value;
        // what a chunk reads: a Kw row, or a Q row and a P row, in fragment form; K; U before the state's part; its decays.  (Loads carry no condition: rows beyond the sequence are its
        // last; of queries they give rows that are not written, keys are dropped where they are used.)
        f32x4 fr[16];
        u32x4 kr[4];
        float uv[16], gr;
        auto request = [&](int n) {
            const float* blk = base + n * block;
            const int t0 = (n0 + n) * GC, last = min(GC, S - t0) - 1;
#pragma unroll
            for (int i = 0; i < 4; ++i) kr[i] = *reinterpret_cast<const u32x4*>(kp + t0 * ldqk + (min((tid >> 4) + 16 * i, last) * (unsigned)ldqk + (tid & 15) * 8));
            gr = blk[C_GAM + min(tid, 2 * GC - 1)];
            if (Q) {
#pragma unroll
                for (int i = 0; i < 8; ++i) fr[i] = *reinterpret_cast<const f32x4*>(qp + t0 * ldqk + (min(row, last) * (unsigned)ldqk + 8 * hf) + 16 * i);
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) fr[i] = *reinterpret_cast<const f32x4*>(blk + row * GD + 8 * hf + 16 * (i >> 1) + 4 * (i & 1));
#pragma unroll
                for (int e = 0; e < 16; ++e) uv[e] = (blk + C_U + v0)[(32 * rh + c_row(e, hf)) * GD + ln];
            }
        };
        auto request_p = [&](int n) {
#pragma unroll
            for (int i = 0; i < 8; ++i) fr[8 + i] = *reinterpret_cast<const f32x4*>(base + n * block + C_P + row * GC + 8 * hf + 16 * (i >> 1) + 4 * (i & 1));
        };
        auto put_out = [&](int t0, int cnt, const f32x16& x) {  // rows beyond the sequence: beyond the buffer, dropped
            auto rs = __builtin_amdgcn_make_buffer_rsrc(o + (((int64_t)b * S + t0) * Hv + h) * GD + v0, 0, 0x7fffffff, 0x00020000);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = 32 * rh + c_row(e, hf);
                __builtin_amdgcn_raw_buffer_store_b16(f2bf(x[e]), rs, r < cnt ? (r * Hv * GD + ln) * 2 : -1, 0, 0);
            }
        };
        request(0);
        if (Q) request_p(0);
#pragma unroll
        for (int c = 0; c < 4; ++c) {  // (behind the first chunk's requests: one latency for both)
            f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if (initial_state) x = *reinterpret_cast<const f32x4*>(initial_state + (head * GD + v0 + ln) * GD + col + 8 * c);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[4 * c + e] = x[e];
        }
        put_state();
        if (Q) {
#pragma unroll
            for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(fr[i])::"memory");  // (landed before the loop, where only its own requests are then waited for)
            put_out(n0 * GC, 0, s);  // (dropped whole: sixteen stores behind P's request from either way in)
        }
        gg[0][tid] = gr;
        for (; n < NC; ++n) {
            float* blk = base + n * block;
            const int t0 = (n0 + n) * GC, cnt = min(GC, S - t0);
            const float* g = gg[n & 1];
            __syncthreads();  // the state is whole, the last chunk's K and U are read
            if (tid == 0) lost[(n + 1) & 1] = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = (tid >> 4) + 16 * i;
                *reinterpret_cast<u32x4*>(&Ks[r][(tid & 15) * 8]) = r < cnt ? kr[i] : u32x4{0u, 0u, 0u, 0u};
            }
            f32x16 hi = zero16(), lo = zero16();
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const Parts8 sp = parts_at<SP>(Sp, ln * (GD + 8) + 16 * i + 8 * hf);
                if (Q) mfma_parts(__builtin_bit_cast(bf16x8, fr[i]), sp, hi, lo);
                else mfma_parts(parts8(fr[2 * i], fr[2 * i + 1]), sp, hi, lo);
            }
            if (!Q) {
                f32x16 u;
#pragma unroll
                for (int e = 0; e < 16; ++e) u[e] = uv[e] - (hi[e] + lo[e]);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int t = 32 * rh + 8 * c + 4 * hf;
                    const f32x4 G = *reinterpret_cast<const f32x4*>(g + GC + t);
                    put_parts<UP>(Ut, ln * (GC + 8) + t, u[4 * c], u[4 * c + 1], u[4 * c + 2], u[4 * c + 3]);
                    *reinterpret_cast<f32x4*>(&Ug[ln][t]) = f32x4{u[4 * c] * G[0], u[4 * c + 1] * G[1], u[4 * c + 2] * G[2], u[4 * c + 3] * G[3]};
                }
                if (__any(lost16(u)) && lane == 0) lost[n & 1] = 1;
#pragma unroll
                for (int e = 0; e < 16; ++e) (blk + C_U + v0)[(32 * rh + c_row(e, hf)) * GD + ln] = u[e];
            }
            if (keep) {
#pragma unroll
                for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4*>(blk - G_KW + v0 * GD + ln * GD + col + 8 * c) = f32x4{s[4 * c], s[4 * c + 1], s[4 * c + 2], s[4 * c + 3]};
            }
            __syncthreads();
            const int gone = lost[n & 1];
            request(min(n + 1, NC - 1));  // (the last chunk's own once more: nothing here hangs on a condition)
            if (Q) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float f = g[32 * rh + c_row(e, hf)] * qscale;
                    hi[e] *= f;
                    lo[e] *= f;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (rh == 0 && i >= 2) break;  // P is lower triangular
                    mfma_parts(parts8(fr[8 + 2 * i], fr[9 + 2 * i]), parts_at<UP>(Ut, ln * (GC + 8) + 16 * i + 8 * hf), hi, lo);
                }
                request_p(min(n + 1, NC - 1));
                asm volatile("" ::: "memory");  // (the stores behind the requests: waits for those then leave the stores alone)
#pragma unroll
                for (int e = 0; e < 16; ++e) hi[e] += lo[e];
                put_out(t0, cnt, hi);
            }
            if (gone) break;  // (the same for the whole workgroup)
            const float gC = g[GC - 1];
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] *= gC;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const f32x4 d = *reinterpret_cast<const f32x4*>(&Ug[ln][8 * i + 4 * hf]);
#pragma unroll
                for (int j = 0; j < 4; ++j) s = mfma2(bf2f(Ks[8 * i + 4 * hf + j][32 * wave + ln]), d[j], s);
            }
            put_state();
            gg[(n + 1) & 1][tid] = gr;
        }
    };
    if (wave >= 2) chunks(std::true_type{});
    else chunks(std::false_type{});
    if (n == NC && final_state) {
#pragma unroll
        for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4*>(final_state + (head * GD + v0 + ln) * GD + col + 8 * c) = f32x4{s[4 * c], s[4 * c + 1], s[4 * c + 2], s[4 * c + 3]};
    }
    // A chunk whose U is not finite, and all behind it: the recurrence itself, eight lanes to a value row.  (In a chunk the triangles' zeros are multiplied, not skipped: a token's key,
    // value, decay or beta that is not finite reaches U and with it the rows before it.  A query reaches its own row alone.)
    if (n < NC) {
#pragma unroll
        for (int e = 0; e < 16; ++e) Ss[ln][32 * wave + c_row(e, hf)] = s[e];  // (the planes are read no more)
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
        for (int i = 0; i < 16; ++i)
            if (final_state) final_state[(head * GD + v0 + r) * GD + c + i] = st[i];
    }
}

// ------------------------------------------------------------------------------------------- reverse scan: the state's gradient, 32 value rows per workgroup
// dU = P^T dO + Gp (K dS^T): a wave takes 16 tokens, both products over their whole sums, of three bf16 parts to dS and P (two tiles of 16 x 16).  dS <- gam_63 dS + (scale gam dO)^T Q - dU^T Kw stays on the
// fp32 pipe, as the scan's: the state's four tiles of 32 key channels go one to a wave, in registers (lane = value row), their three parts in LDS for the next chunk.  Bound: the chain of chunks and the
// bytes; every operand is requested a chunk ahead, without conditions (rows beyond the sequence are its last, made zero where they are used).  8 x 708 tokens x 16
// heads 159 -> 120 us, 333 tokens 57 -> 40 (fp32 products of halves of a sum that met in LDS, K and P requested where they were used).
__global__ __launch_bounds__(256, 2) void gdrc_rscan_kernel(int heads, int S, int NC, int Hqk, int Hv, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const float* __restrict__ saved,
                                                            const bf16_t* __restrict__ d_o, float* __restrict__ ws, const float* d_final, float* d_initial, float qscale) {
    __shared__ __attribute__((aligned(16))) bf16_t Sp[3 * SP];
    __shared__ __attribute__((aligned(16))) bf16_t Qs[GC][GD + 8];
    __shared__ __attribute__((aligned(16))) bf16_t Os[GC][GV + 8];
    __shared__ __attribute__((aligned(16))) float Og[GV][GC + 4], Ug[GV][GC + 4];  // scale gam dO and dU, [value row][token]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 31, hf = lane >> 5;
    const int l16 = lane & 15, g = lane >> 4, q4 = (lane >> 2) & 3, p4 = lane & 3;
    int at, v0;
    if (!scan_place(heads, at, v0)) return;
    const int h = at % Hv, b = at / Hv, hq = h / (Hv / Hqk), col = 32 * wave + 4 * hf, orow = tid >> 2, ocol = (tid & 3) * 8;
    const int64_t ldqk = (int64_t)Hqk * GD, ldo = (int64_t)Hv * GD, head = at;
    const bf16_t *qp = q + (int64_t)b * S * ldqk + hq * GD, *kp = k + (int64_t)b * S * ldqk + hq * GD, *gp = d_o + (int64_t)b * S * ldo + (int64_t)h * GD + v0;
    const float* base = saved + head * NC * G_BLOCK;
    float* wbase = ws + head * NC * W_BLOCK;
    // what a chunk reads: 16 rows of K and 16 columns of P in fragment form; the wave's 32 columns of Kw; Q; dO; decays
    u32x4 kr[4], qr[4], gr;
    float pr[16], wr[32], gam, last;
    f32x4 Gp;
    auto request = [&](int n) {
        const float* blk = base + (int64_t)n * G_BLOCK;
        const int t0 = n * GC, end = min(GC, S - t0) - 1;
        gr = *reinterpret_cast<const u32x4*>(gp + t0 * ldo + min(orow, end) * ldo + ocol);
        gam = blk[G_GAM + orow];
#pragma unroll
        for (int i = 0; i < 4; ++i) qr[i] = *reinterpret_cast<const u32x4*>(qp + t0 * ldqk + (min((tid >> 4) + 16 * i, end) * (unsigned)ldqk + (tid & 15) * 8));
#pragma unroll
        for (int i = 0; i < 4; ++i) kr[i] = *reinterpret_cast<const u32x4*>(kp + t0 * ldqk + (min(16 * wave + l16, end) * (unsigned)ldqk + 8 * g) + 32 * i);
#pragma unroll
        for (int i = 0; i < 16; ++i) pr[i] = (blk + G_P)[(32 * (i >> 3) + 8 * g + (i & 7)) * GC + 16 * wave + l16];
        Gp = *reinterpret_cast<const f32x4*>(blk + G_GAM + GC + 16 * wave + 4 * g);
        last = blk[G_GAM + GC - 1];
    };
    auto request_w = [&](int n) {
#pragma unroll
        for (int i = 0; i < 32; ++i) wr[i] = (base + (int64_t)n * G_BLOCK + G_KW)[(8 * (i >> 2) + 4 * hf + (i & 3)) * GD + 32 * wave + ln];
    };
    f32x16 s;  // dS[v0 + ln][32 wave + c_row(e, hf)]
    auto put_state = [&]() {
#pragma unroll
        for (int c = 0; c < 4; ++c) put_parts<SP>(Sp, ln * (GD + 8) + col + 8 * c, s[4 * c], s[4 * c + 1], s[4 * c + 2], s[4 * c + 3]);
    };
    request(NC - 1);
    request_w(NC - 1);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        f32x4 x = {0.f, 0.f, 0.f, 0.f};
        if (d_final) x = *reinterpret_cast<const f32x4*>(d_final + (head * GD + v0 + ln) * GD + col + 8 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[4 * c + e] = x[e];
    }
    put_state();
    for (int n = NC - 1; n >= 0; --n) {
        float* wblk = wbase + (int64_t)n * W_BLOCK;
        const int cnt = min(GC, S - n * GC);
        const float gC = last;
        __syncthreads();  // dS is whole, the last chunk's operands are read
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = (tid >> 4) + 16 * i;
            *reinterpret_cast<u32x4*>(&Qs[r][(tid & 15) * 8]) = r < cnt ? qr[i] : u32x4{0u, 0u, 0u, 0u};
        }
        {
            const u32x4 x = orow < cnt ? gr : u32x4{0u, 0u, 0u, 0u};
            const float f = gam * qscale;
            *reinterpret_cast<u32x4*>(&Os[orow][ocol]) = x;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                Og[ocol + 2 * e][orow] = __uint_as_float(x[e] << 16) * f;
                Og[ocol + 2 * e + 1][orow] = __uint_as_float(x[e] & 0xffff0000u) * f;
            }
        }
        f32x4 hi[2], lo[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) hi[j] = lo[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bf16x8 kf = __builtin_bit_cast(bf16x8, kr[i]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const Parts8 sp = parts_at<SP>(Sp, (16 * j + l16) * (GD + 8) + 32 * i + 8 * g);
                lo[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, sp.p[2], lo[j], 0, 0, 0);
                lo[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, sp.p[1], lo[j], 0, 0, 0);
                hi[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, sp.p[0], hi[j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4*>(wblk + v0 * GD + ln * GD + col + 8 * c) = f32x4{s[4 * c], s[4 * c + 1], s[4 * c + 2], s[4 * c + 3]};
        Parts8 pp[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) pp[i] = parts8(f32x4{pr[8 * i], pr[8 * i + 1], pr[8 * i + 2], pr[8 * i + 3]}, f32x4{pr[8 * i + 4], pr[8 * i + 5], pr[8 * i + 6], pr[8 * i + 7]});
        __syncthreads();  // dO lies
        f32x4 u[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f32x4 ph = {0.f, 0.f, 0.f, 0.f}, pl = ph;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (i == 0 && wave >= 2) continue;  // P is lower triangular, and its zeros are not multiplied: a dO that is not finite reaches no later token but those of its own 32
                const bf16_t* o = &Os[32 * i + 8 * g + q4][16 * j + 4 * p4];
                const bf16x4 o0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)(o)), o1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)(o + 4 * (GV + 8)));
                const bf16x8 of = __builtin_shufflevector(o0, o1, 0, 1, 2, 3, 4, 5, 6, 7);
                pl = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pp[i].p[2], of, pl, 0, 0, 0);
                pl = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pp[i].p[1], of, pl, 0, 0, 0);
                ph = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pp[i].p[0], of, ph, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) u[j][e] = 16 * wave + 4 * g + e < cnt ? fmaf(Gp[e], hi[j][e] + lo[j][e], ph[e] + pl[e]) : 0.f;
            *reinterpret_cast<f32x4*>(&Ug[16 * j + l16][16 * wave + 4 * g]) = u[j];
        }
        __syncthreads();
        request(n > 0 ? n - 1 : 0);  // (the first chunk's own once more: nothing here hangs on a condition)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) (wblk + W_DU + v0)[(16 * wave + 4 * g + e) * GD + 16 * j + l16] = u[j][e];
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] *= gC;
        // from the last token to the first: what reaches the chunk's start grows that way (the other way around the large terms come first and every later sum rounds at their size)
#pragma unroll
        for (int i = 7; i >= 0; --i) {
            const f32x4 o4 = *reinterpret_cast<const f32x4*>(&Og[ln][8 * i + 4 * hf]), u4 = *reinterpret_cast<const f32x4*>(&Ug[ln][8 * i + 4 * hf]);
#pragma unroll
            for (int j = 3; j >= 0; --j) {
                s = mfma2(bf2f(Qs[8 * i + 4 * hf + j][32 * wave + ln]), o4[j], s);
                s = mfma2(wr[4 * i + j], -u4[j], s);
            }
        }
        request_w(n > 0 ? n - 1 : 0);
        put_state();
    }
    if (d_initial) {
#pragma unroll
        for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4*>(d_initial + (head * GD + v0 + ln) * GD + col + 8 * c) = f32x4{s[4 * c], s[4 * c + 1], s[4 * c + 2], s[4 * c + 3]};
    }
}

// ------------------------------------------------------------------------------------------- the rest of the backward: one workgroup per chunk and head
// Bound: the fp32 matrix pipe (130 us of 8 x 708 tokens x 16 heads) and the chunk's blocks from memory (0.5 GB, 105 us), with eight waves a CU to overlap them; so
// nothing may stand between the products.  542 -> 287 us (96 chunks, one a CU: 110 -> 50): sums over a token's features meet in a lane, since results are taken transposed (half-wave
// sums, one row after the other, were a quarter of the time); loads carry no condition (rows beyond the sequence are its last, and what they give is dropped) and stand two stages
// ahead, held there by in_order(); the first product's operands are requested all at once; the pairs' decay sums go by 256 threads and scans instead of 64 chains (25 000 clocks -> 5 000).
// Requests three stages ahead: 293 us (registers spill); the two workgroups of a CU set off apart: 370 against 366 at that time.
__global__ __launch_bounds__(256, 2) void gdrc_bwd_kernel(int S, int NC, int Hqk, int Hv, const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
                                                          int64_t ldv, const float* __restrict__ beta, const float* __restrict__ alpha, const float* __restrict__ saved,
                                                          const float* __restrict__ ws, const bf16_t* __restrict__ d_o, bf16_t* __restrict__ dq, bf16_t* __restrict__ dk,
                                                          bf16_t* __restrict__ dv, int64_t lddv, float* __restrict__ dbeta, float* __restrict__ dalpha, float* __restrict__ pdq,
                                                          float* __restrict__ pdk, float qscale, int wide) {
    constexpr int LM = GC + 4, LZ = GC + 2;
    __shared__ __attribute__((aligned(16))) float Z[GC][GD + 4];   // -dU S0; later Y, then d(Q K^T) (first half), and the pairs' decay terms (second half)
    __shared__ __attribute__((aligned(16))) float M12[2 * GC * LM];  // dU; later the next two
    float(*M1)[LM] = reinterpret_cast<float(*)[LM]>(M12);            // dR; later d(K K^T) + its transpose
    float(*M2)[LM] = reinterpret_cast<float(*)[LM]>(M12 + GC * LM);  // R
    float(*Ud)[GD + 4] = reinterpret_cast<float(*)[GD + 4]>(M12);
    static_assert(GC * (GD + 4) <= 2 * GC * LM, "dU fits the space of the two matrices");
    __shared__ double gd[GC];
    __shared__ float be[GC], al[GC], gam[GC], gp[GC], redG[4][GC], redP[4][GC], redB[4][GC], dss[4];
    __shared__ double pairs[4][GC];
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
    // Everything of the first product is requested at once: dU, which the next phase reads too, goes to LDS, a lane's share of the first state stays in registers.
    f32x4 ud[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) ud[i] = *reinterpret_cast<const f32x4*>(dU + 4 * (tid + 256 * i));
    float st[GD / 2];
#pragma unroll
    for (int j = 0; j < GD / 2; ++j) st[j] = blk[(8 * (j >> 2) + 4 * hf + (j & 3)) * GD + col];
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(&Ud[(tid + 256 * i) >> 5][((tid + 256 * i) & 31) * 4]) = ud[i];
    __syncthreads();
    {  // Z = -dU S0: wave = 32 columns, both row halves
        f32x16 z[2] = {zero16(), zero16()};
#pragma unroll
        for (int kb = 0; kb < GD; kb += 8) {
            const f32x4 d0 = *reinterpret_cast<const f32x4*>(&Ud[ln][kb + 4 * hf]), d1 = *reinterpret_cast<const f32x4*>(&Ud[32 + ln][kb + 4 * hf]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                z[0] = mfma2(st[kb / 2 + j], -d0[j], z[0]);
                z[1] = mfma2(st[kb / 2 + j], -d1[j], z[1]);
            }
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int e = 0; e < 16; e += 4) *reinterpret_cast<f32x4*>(&Z[32 * r + ln][32 * wave + c_row(e, hf)]) = f32x4{z[r][e], z[r][e + 1], z[r][e + 2], z[r][e + 3]};
    }
    __syncthreads();
    // the 64 x 64 matrices: wave = tile (ti, tj)
    const int ti = wave >> 1, tj = wave & 1, j0 = 32 * tj + ln;
    f32x16 lkk, e1, dqk;
    f32x4 rr[4];
    float un[32];  // dU once more, by columns
    {
        f32x16 kk = zero16(), qk = zero16(), dP = zero16(), dT = zero16(), tz = zero16(), dPt = zero16();
        if (wave != 1) {
            const int ri = 32 * ti + ln, rj = 32 * tj + ln;
            const float* ur = Up + rj * GD + 8 * hf;
            struct Stage {  // 16 features, a half wave's eight of them together
                u32x4 o, v, k, qi, ki;
                f32x4 u[2];
            };
            auto request = [&](Stage& t, int kb) {
                t.o = held8(op, ldo, ri, cnt, kb + 8 * hf), t.v = held8(vp, ldv, rj, cnt, kb + 8 * hf), t.k = held8(kp, ldqk, rj, cnt, kb + 8 * hf);
                t.qi = held8(qp, ldqk, ri, cnt, kb + 8 * hf), t.ki = held8(kp, ldqk, ri, cnt, kb + 8 * hf);
#pragma unroll
                for (int c = 0; c < 2; ++c) t.u[c] = *reinterpret_cast<const f32x4*>(ur + kb + 4 * c);
                in_order();
            };
            auto work = [&](const Stage& t, int kb) {
                const u32x4 &o = t.o, &v8 = t.v, &k8 = t.k;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const f32x4 of = widen4(u32x2{o[2 * c], o[2 * c + 1]}), vf = widen4(u32x2{v8[2 * c], v8[2 * c + 1]}), kf = widen4(u32x2{k8[2 * c], k8[2 * c + 1]});
                    const f32x4 zi = *reinterpret_cast<const f32x4*>(&Z[ri][kb + 8 * hf + 4 * c]), di = *reinterpret_cast<const f32x4*>(&Ud[ri][kb + 8 * hf + 4 * c]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        dP = mfma2(of[j], t.u[c][j], dP);
                        dT = mfma2(di[j], vf[j], dT);
                        tz = mfma2(zi[j], kf[j], tz);
                    }
                }
                kk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, t.ki), __builtin_bit_cast(bf16x8, k8), kk, 0, 0, 0);
                qk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, t.qi), __builtin_bit_cast(bf16x8, k8), qk, 0, 0, 0);
            };
            Stage x, y;
            request(x, 0);
            for (int kb = 0; kb < GD - 32; kb += 32) {
                request(y, kb + 16);
                work(x, kb);
                request(x, kb + 32);
                work(y, kb + 16);
                add16(dPt, dP);
            }
            request(y, GD - 16);
            work(x, GD - 32);
            work(y, GD - 16);
            add16(dPt, dP);
            add16(dP, dPt);
        } else {  // (the upper right tiles are empty)
            float a;
            gd[lane] = cumulated_log(alpha, (tok0 + lane) * Hv + h, lane < cnt, a);
            al[lane] = a;
            be[lane] = beta_of(beta, (tok0 + lane) * Hv + h, lane < cnt);
            gam[lane] = blk[G_GAM + lane];
            gp[lane] = blk[G_GAM + GC + lane];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) rr[i] = *reinterpret_cast<const f32x4*>(blk + G_R + 4 * (tid + 256 * i));
#pragma unroll
        for (int j = 0; j < 32; ++j) un[j] = dU[(8 * (j >> 2) + 4 * hf + (j & 3)) * GD + col];
        __syncthreads();  // dU's place is free
        const double gj = gd[j0];
        const float gaj = gam[j0], bj = be[j0];
#pragma unroll
        for (int e = 0; e < 16; ++e) {  // (no branch: what lies above the diagonal is computed and dropped)
            const int i = 32 * ti + c_row(e, hf);
            const bool in = i >= j0 && i < cnt;  // (the operands' rows beyond the sequence are its last)
            const float x = exp_of(gd[i] - gj), D = in ? x : 0.f, t = in ? dT[e] + gaj * tz[e] : 0.f, p = in ? qscale * dP[e] : 0.f;
            lkk[e] = in && i > j0 ? kk[e] * D : 0.f;
            e1[e] = in ? p * (qk[e] * D) : 0.f;
            dqk[e] = p * D;
            M1[i][j0] = t * bj;
            if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (four at a time: the registers)
        }
        asm volatile("" : "+v"(lkk), "+v"(e1), "+v"(dqk));  // (here and not where they are first used: three products' sums would stay instead)
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4*>(&M2[(tid + 256 * i) >> 4][((tid + 256 * i) & 15) * 4]) = rr[i];
    }
    __syncthreads();
    // From here on results are taken transposed (the operands change places, the products and their order stay): a lane holds 16 features of one token, four neighbours at a time, so
    // what a token sums over its features meets in the lane and its other half, and rows are read and written four features at a time.
    f32x16 w[2];  // dK, from here on
    {  // dV = T^T dU, d(gam K) = T^T Z: wave = 32 columns
        f32x16 a[2] = {zero16(), zero16()}, g[2] = {zero16(), zero16()};
#pragma unroll
        for (int kb = 0; kb < 32; kb += 8)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = kb + 4 * hf + j;
                const float r0 = M2[i][ln];
                a[0] = mfma2(un[kb / 2 + j], r0, a[0]);
                g[0] = mfma2(Z[i][col], r0, g[0]);
            }
        f32x16 at = zero16(), gt = zero16();
        add16(at, a[0]), add16(gt, g[0]);
#pragma unroll
        for (int kb = 32; kb < GC; kb += 8)  // R is lower triangular
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = kb + 4 * hf + j;
                const float bz = Z[i][col], r0 = M2[i][ln], r1 = M2[i][32 + ln];
                a[0] = mfma2(un[kb / 2 + j], r0, a[0]);
                g[0] = mfma2(bz, r0, g[0]);
                a[1] = mfma2(un[kb / 2 + j], r1, a[1]);
                g[1] = mfma2(bz, r1, g[1]);
            }
        add16(a[0], at);
        add16(g[0], gt);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int i = 32 * r + ln;
            const bool in = i < cnt;
            const float bi = be[i], ga = gam[i];
            bf16_t* out = dv + (tok0 + i) * lddv + (int64_t)h * GD + 32 * wave;
            f32x4 u4[4];
            u32x2 k4[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                u4[c] = *reinterpret_cast<const f32x4*>(Up + i * GD + 32 * wave + c_row(4 * c, hf));
                k4[c] = held4(kp, ldqk, i, cnt, 32 * wave + c_row(4 * c, hf));
            }
            float sb[4], sg[4];
            f32x4 ov[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const f32x4 kf = widen4(k4[c]);
                float o[4], pb[4], pg[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float av = a[r][4 * c + j], d = bi * g[r][4 * c + j];
                    // d(beta): what reaches u = beta (v - the state's answer to k) times that difference, which is u / beta
                    pb[j] = av * u4[c][j];
                    o[j] = bi * av;
                    w[r][4 * c + j] = ga * d;
                    pg[j] = d * kf[j];
                }
                sb[c] = (pb[0] + pb[1]) + (pb[2] + pb[3]);
                sg[c] = (pg[0] + pg[1]) + (pg[2] + pg[3]);
                ov[c] = {o[0], o[1], o[2], o[3]};
            }
            const float b1 = both_halves((sb[0] + sb[1]) + (sb[2] + sb[3])), g1 = both_halves((sg[0] + sg[1]) + (sg[2] + sg[3]));
            if (hf == 0) redB[wave][i] = b1, redG[wave][i] = in ? g1 : 0.f;
            if (in) put16(out, ov, hf, wide);
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
    auto dn_rows = [&](int k0) {
#pragma unroll
        for (int kb = k0; kb < k0 + 32; kb += 8)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = kb + 4 * hf + j;
                dn = mfma2(M2[i][32 * ti + ln], M3[i][32 * tj + ln], dn);
            }
    };
    if (wave != 1) {  // dN = -R^T Y
        if (ti == 0) dn_rows(0);
        dn_rows(32);
    }
    __syncthreads();  // dR and Y are done with
    if (wave != 1) {
        double gj = gd[j0];
        asm volatile("" : "+v"(gj));  // (once more, and not kept in registers from above)
        float* spare = &M1[ln][GC];  // (the rows' padding takes what is not below the diagonal)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = 32 * ti + c_row(e, hf);
            const bool in = i > j0;
            const float x = exp_of(gd[i] - gj), D = in ? x : 0.f, dl = be[i] * (in ? -dn[e] : 0.f), m = dl * D;
            *(in ? &M1[i][j0] : spare) = m;
            *(in ? &M1[j0][i] : spare) = m;
            M3[i][j0] = dqk[e];
            ME[i][j0] = fmaf(dl, lkk[e], e1[e]);
            if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        M1[lane][lane] = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = c_row(e, hf);
            M3[i][j0] = 0.f;
            ME[i][j0] = 0.f;
        }
    }
    // the last large products' first operands, under way from here on
    struct Late {
        u32x4 o[2];
        f32x4 u[2][2];
        float s0[8], s1[8];
    };
    auto request_late = [&](Late& t, int kb) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            t.o[r] = held8(op, ldo, 32 * r + ln, cnt, kb + 8 * hf);
#pragma unroll
            for (int c = 0; c < 2; ++c) t.u[r][c] = *reinterpret_cast<const f32x4*>(Up + (32 * r + ln) * GD + kb + 8 * hf + 4 * c);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            t.s0[j] = blk[(kb + 8 * hf + j) * GD + col];
            t.s1[j] = dS[(kb + 8 * hf + j) * GD + col];
        }
        in_order();
    };
    Late now, next;
    request_late(now, 0);
    __syncthreads();
    // dQ = scale gam (dO S0), dK += Gp (U dS): contraction over the value rows, straight from memory as above
    f32x16 x[2] = {zero16(), zero16()};
    {
        f32x16 y[2] = {zero16(), zero16()};
        float sds = 0.f;
        auto work = [&](const Late& t) {
            const u32x4 &o0 = t.o[0], &o1 = t.o[1];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const f32x4 a0 = widen4(u32x2{o0[2 * c], o0[2 * c + 1]}), a1 = widen4(u32x2{o1[2 * c], o1[2 * c + 1]});
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float c0 = t.s0[4 * c + j], c1 = t.s1[4 * c + j];
                    sds = fmaf(c0, c1, sds);
                    x[0] = mfma2(c0, a0[j], x[0]);
                    x[1] = mfma2(c0, a1[j], x[1]);
                    y[0] = mfma2(c1, t.u[0][c][j], y[0]);
                    y[1] = mfma2(c1, t.u[1][c][j], y[1]);
                }
            }
        };
        for (int kb = 0; kb < GD - 32; kb += 32) {  // (no request behind a condition: where the paths meet, a wait is for either's)
            request_late(next, kb + 16);
            work(now);
            request_late(now, kb + 32);
            work(next);
        }
        request_late(next, GD - 16);
        work(now);
        work(next);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int i = 32 * r + ln;
            const bool in = i < cnt;
            const float ga = gam[i], gi = gp[i];
            u32x2 q4[4], k4[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                q4[c] = held4(qp, ldqk, i, cnt, 32 * wave + c_row(4 * c, hf));
                k4[c] = held4(kp, ldqk, i, cnt, 32 * wave + c_row(4 * c, hf));
            }
            float sg[4], sp[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const f32x4 qf = widen4(q4[c]), kf = widen4(k4[c]);
                float pg[4], pp[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float qx = qscale * x[r][4 * c + j], yv = y[r][4 * c + j];
                    pg[j] = qx * qf[j];
                    pp[j] = yv * kf[j];
                    x[r][4 * c + j] = ga * qx;
                    w[r][4 * c + j] = fmaf(gi, yv, w[r][4 * c + j]);
                }
                sg[c] = (pg[0] + pg[1]) + (pg[2] + pg[3]);
                sp[c] = (pp[0] + pp[1]) + (pp[2] + pp[3]);
            }
            const float g1 = both_halves((sg[0] + sg[1]) + (sg[2] + sg[3])), p1 = both_halves((sp[0] + sp[1]) + (sp[2] + sp[3]));
            if (hf == 0) redG[wave][i] += in ? g1 : 0.f, redP[wave][i] = in ? p1 : 0.f;
        }
        sds = half_sum(sds);
        sds += __shfl_xor(sds, 32, 64);
        if (lane == 0) dss[wave] = sds;
    }
    // dK += (dKK + dKK^T) K + dQK^T Q, dQ += dQK K
    {
        bf16_t kn[2][8], qn[2][8];
        const int ld = (int)ldqk, first = 8 * hf * ld, last = (cnt - 1) * ld;
        auto request = [&](int b16) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const unsigned at = 2u * (unsigned)(min(first + (16 * b16 + j) * ld, last) + col);
                kn[b16 & 1][j] = *reinterpret_cast<const bf16_t*>(reinterpret_cast<const char*>(kp) + at);
                qn[b16 & 1][j] = *reinterpret_cast<const bf16_t*>(reinterpret_cast<const char*>(qp) + at);
            }
            in_order();
        };
        request(0);
#pragma unroll
        for (int b16 = 0; b16 < 4; ++b16) {
            if (b16 < 3) request(b16 + 1);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k0 = 16 * b16 + 8 * hf + 4 * c;
                const f32x4 s0 = *reinterpret_cast<const f32x4*>(&M1[ln][k0]), s1 = *reinterpret_cast<const f32x4*>(&M1[32 + ln][k0]);
                const f32x2 x1a = *reinterpret_cast<const f32x2*>(&M3[32 + ln][k0]), x1b = *reinterpret_cast<const f32x2*>(&M3[32 + ln][k0 + 2]);
                const f32x2 x0a = *reinterpret_cast<const f32x2*>(&M3[ln][k0]), x0b = *reinterpret_cast<const f32x2*>(&M3[ln][k0 + 2]);
                const float x1[4] = {x1a[0], x1a[1], x1b[0], x1b[1]}, x0[4] = {x0a[0], x0a[1], x0b[0], x0b[1]};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool in = k0 + j < cnt;
                    const float kf = bf2f(in ? kn[b16 & 1][4 * c + j] : (bf16_t)0), qf = bf2f(in ? qn[b16 & 1][4 * c + j] : (bf16_t)0);
                    w[0] = mfma2(kf, s0[j], w[0]);
                    w[1] = mfma2(kf, s1[j], w[1]);
                    w[0] = mfma2(qf, M3[k0 + j][ln], w[0]);
                    x[1] = mfma2(kf, x1[j], x[1]);
                    if (b16 >= 2) w[1] = mfma2(qf, M3[k0 + j][32 + ln], w[1]);
                    else x[0] = mfma2(kf, x0[j], x[0]);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int i = 32 * r + ln;
        if (i >= cnt) continue;
        f32x4 dx[4], dw[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            dx[c] = f32x4{x[r][4 * c], x[r][4 * c + 1], x[r][4 * c + 2], x[r][4 * c + 3]};
            dw[c] = f32x4{w[r][4 * c], w[r][4 * c + 1], w[r][4 * c + 2], w[r][4 * c + 3]};
        }
        if (pdq) {  // several value heads share a q / k head: per value head, summed afterwards
            const int64_t at = (head * S + t0 + i) * GD + 32 * wave;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                *reinterpret_cast<f32x4*>(pdq + at + c_row(4 * c, hf)) = dx[c];
                *reinterpret_cast<f32x4*>(pdk + at + c_row(4 * c, hf)) = dw[c];
            }
        } else {
            put16(dq + (tok0 + i) * ldqk + hq * GD + 32 * wave, dx, hf, wide);
            put16(dk + (tok0 + i) * ldqk + hq * GD + 32 * wave, dw, hf, wide);
        }
    }
    // d(log alpha_t): every pair (i, j) with j < t <= i, what reaches token i >= t from the chunk's first state, what token j < t leaves in its last, and the state passing through.
    // Row i's sums over the columns before each t by four lanes, then column t's over the rows from t on by one lane of each wave; all in fp64.
    {
        const int i = tid >> 2, c = 16 * (tid & 3);
        float row[16];
        double mine = 0.;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            row[j] = ME[i][c + j];
            mine += row[j];
        }
        double run = 0.;
#pragma unroll
        for (int o = 1; o < 4; ++o) {
            const double v = __shfl_up(mine, o, 4);
            if ((tid & 3) >= o) run += v;
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            ME[i][c + j] = (float)run;
            run += row[j];
        }
    }
    __syncthreads();
    {
        double s = 0.;
#pragma unroll
        for (int o = 0; o < 16; ++o) {
            const int i = 16 * wave + o;
            const float m = ME[i][lane];
            s += i >= lane ? m : 0.f;
        }
        pairs[wave][lane] = s;
    }
    __syncthreads();
    if (wave == 0) {
        const int t = lane;
        double from = gam[t] * ((redG[0][t] + redG[1][t]) + (redG[2][t] + redG[3][t]));  // summed over the tokens from t on
        const double leaves = gp[t] * ((redP[0][t] + redP[1][t]) + (redP[2][t] + redP[3][t]));
        double left = leaves;  // summed over the tokens up to t
#pragma unroll
        for (int o = 1; o < GC; o <<= 1) {
            const double f = __shfl_down(from, o, 64), l = __shfl_up(left, o, 64);
            if (t + o < GC) from += f;
            if (t >= o) left += l;
        }
        const double before = __shfl_up(left, 1, 64);
        const double s = (double)(gam[GC - 1] * ((dss[0] + dss[1]) + (dss[2] + dss[3]))) + ((pairs[0][t] + pairs[1][t]) + (pairs[2][t] + pairs[3][t])) + from + (t ? before : 0.);
        if (t < cnt) {
            dalpha[(tok0 + t) * Hv + h] = (float)s / al[t];
            dbeta[(tok0 + t) * Hv + h] = ((redB[0][t] + redB[1][t]) + (redB[2][t] + redB[3][t])) / be[t];
        }
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
                                                             (bf16_t*)dk, (bf16_t*)dv, lddv, dbeta, dalpha, pdq, pdk, qs, (((uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) & 7) == 0 && lddv % 4 == 0);
    MI355_LAUNCH_CHECK("gdr_chunked_bwd");
    if (pdq) {
        const int64_t total = (int64_t)B * S * Hqk * GD;
        gdrc_heads_kernel<<<(unsigned)((total + 255) / 256), 256, 0, ST(stream)>>>(S, Hqk, Hv, pdq, pdk, (bf16_t*)dq, (bf16_t*)dk, total);
        MI355_LAUNCH_CHECK("gdr_chunked_bwd(heads)");
    }
    return 0;
}
