// KV-cache decoding on the step's right edge: the per-token path of generate_loop_kv_cache
// (llm_quest/generate.py:97-151) through Qwen3 with utils.KVCache (utils.py:409-531).  One new token per sequence makes every
// linear layer a matrix-VECTOR product and attention one query row against the cache: both are HBM-bound byte streams (weights,
// resp. cached K/V read exactly once per token), so the kernels here are bandwidth kernels, not MFMA kernels.
//   gemv            y[m, :] = x[m, :] W^T (+ residual), m < 8 rows: 16 weight rows at a time on the matrix pipe (one operand row: a wave per weight row), fp32 accumulate
//   attn_decode     one query per (batch, head) over `len` cached keys: 4 waves split the keys (flash-decoding), scores with the
//                   key on the lane, P V with the feature on the lane, combined through LDS; reference mask semantics (finite fill)
//   gemv_pro        the same weight stream with the row operation that feeds it folded in (PRO 1: RMSNorm of x, PRO 2: SwiGLU of a gate-up row): every
//                   workgroup rebuilds the <= 8 operand rows (a few KB) instead of a launch of its own writing them
//   attn_decode_qkv the same attention started from the fused QKV stream's raw row: QK-RMSNorm + RoPE of the head's query and of its kv head's new key inside the launch,
//                   key and value head written to the cache row at the device-side position (qknorm_rope_fwd + kv_append + attn_decode in one launch)
//   argmax_rows     greedy sampling: first index of the row maximum (torch.argmax tie rule on ties is unspecified; first is used)
#include "common.h"
#include "lane_sums.h"

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float MASK_T = -2.0e38f;  // finite "masked" score in the log2 domain (finfo(bf16).min / 2 semantics: exp -> 0, uniform if all masked)

__device__ __forceinline__ void unpack8(const u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        f[2 * e] = __uint_as_float(v[e] << 16);
        f[2 * e + 1] = __uint_as_float(v[e] & 0xffff0000u);
    }
}

// ------------------------------------------------------------------------------------------- skinny GEMM (NT), M <= 8
// A workgroup takes 16 weight rows (ROWS: or 8) at a time; its NW waves share k out in consecutive runs of `steps` x 32.  A weight row is an A row of v_mfma_f32_16x16x32_bf16, an operand row a
// B column (eight of the sixteen stay idle: the pipe has nothing else to do), the waves' sums meet in LDS and are added in wave order -- which sums a result is made of
// depends on N and K alone, for two to eight rows: one row goes through gemv_one_kernel, which sums in another order.  The operand rows go straight to fragments, finished there by the row operation that feeds the stream: PRO 1 RMSNorm(x[m]) * nw in the arithmetic
// and summation order of rmsnorm_fwd_generic (norm_rope.hip; == rmsnorm_fwd_kernel<2> at width 1024), PRO 2 x holds gate-up rows [M, 2K] (up | gate, as the fused
// lin1 | lin_gate projection writes them), swiglu_act(up, gate) as swiglu_fwd_kernel rounds it: fused == the two launches bit for bit.  GLU: W holds 2N rows (up | gate) and the
// activation is the epilogue -- eight up rows and their gate rows make a group; every activation is worked out once, not once a workgroup.
// Bound: a launch of a few MB is a chain of memory round trips (operand rows, row sums, weights, results), so the weights' trip runs under the operands': loads return in
// order, hence operand loads first, weights behind them, and the next 16 rows' weights under this one's products.
// EVEN: the waves' runs are whole chunks of T steps and end with K: no load has a condition (a branch, a select and an address of its own each: 28 of them in front of the first
// product were 1 us of a launch), what rows past the last one give is not stored.  us, six rows, weights from memory, before -> EVEN: RMSNorm + 4096 x
// 1024 6.9 -> 5.8, RMSNorm + SwiGLU of 6144 x 1024 7.9 -> 7.5, 1024 x 3072 5.3 -> 4.9, 1024 x 2048 4.6 -> 4.2.  One row (gemv_one_kernel, T strips of 512 k): 4.9 -> 4.4, 5.2 -> 4.6,
// 3.8 -> 3.5.  T 4 or 8: chunks of 7 steps (K = 3584) gain nothing, nor do 384 workgroups for 384 groups.
// Lanes past the last operand row stay out of its loads (one branch; the row again, REPEAT, is as many requests as sixteen rows: eight rows, 4096 x 2048 7.0 us against 6.5, 3072 x 3072 8.3 / 7.3).  REPEAT where
// the row sums come first and the weights of a group are eight rows: three rows, RMSNorm + 1024 x 2048 5.1 / 5.8.
constexpr int OUT_BF16 = 0, OUT_F32 = 1, OUT_BF16_BIAS = 2;  // what is stored, and what `res` is: bf16 rows of a residual, or one fp32 row
constexpr int GEMV_STEPS = 8;  // of 32 k in flight per wave: 8 x 16 bytes a lane
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = pack_bf2(f[2 * e], f[2 * e + 1]);
    return o;
}
__device__ __forceinline__ float rbf(float x) { return bf2f(f2bf(x)); }

template <int NW, int PRO, int OUT, bool GLU, int ROWS, int T, bool EVEN>
__global__ __launch_bounds__(64 * NW) void gemv_kernel(int M, int64_t N, int K, int steps, const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ nw, float eps,
                                                       const bf16_t* __restrict__ W, int64_t ldw, void* __restrict__ y, int64_t ldy, const void* __restrict__ res, int64_t ldr) {
    static_assert(!EVEN || (PRO != 2 && NW * T % 16 == 0), "whole strips of 512 k");
    constexpr bool REPEAT = PRO == 1 && ROWS == 8;  // lanes past the last operand row: that row again, else one branch around the loads
    __shared__ float rs[8];
    __shared__ __attribute__((aligned(16))) float part[2][NW][8][16];
    __shared__ __attribute__((aligned(16))) bf16_t act[PRO == 2 ? NW : 1][8][PRO == 2 ? 32 * T + 8 : 8];  // PRO 2: a wave's run of the activated rows
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, kg = (lane >> 4) * 8;
    const int nvec = K >> 3, chunks = (steps + T - 1) / T;
    const int k_lo = wave * steps * 32, k_hi = min(K, k_lo + steps * 32);
    constexpr int GN = GLU ? 8 : ROWS;  // columns of a group
    const bool on = GLU || r16 < ROWS;  // lanes that hold a weight row
    const int64_t groups = (N + GN - 1) / GN;
    const u32x4 z4 = {0u, 0u, 0u, 0u};
    u32x4 xf[T], gf[PRO ? T : 1], w0[T], w1[T];
    auto request_x = [&](int c) {
        if constexpr (PRO == 2) {  // whole rows dealt to the lanes: an activation costs ~ 100 clocks, fragments have eight or more lanes of sixteen idle
#pragma unroll
            for (int t = 0; t < T / 2; ++t) {
                const int m = 2 * t + (lane >> 5), k = k_lo + c * T * 32 + (lane & 31) * 8;
                const bool in = m < M && k < k_hi;
                xf[t] = in ? *reinterpret_cast<const u32x4*>(x + m * ldx + k) : z4;
                gf[t] = in ? *reinterpret_cast<const u32x4*>(x + m * ldx + K + k) : z4;
            }
        } else if constexpr (EVEN) {
            const int m = REPEAT ? min(r16, M - 1) : r16;
            if (m >= M) return;
            const bf16_t *row = x + m * ldx + k_lo + c * T * 32 + kg, *g = nw + k_lo + c * T * 32 + kg;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                xf[t] = *reinterpret_cast<const u32x4*>(row + t * 32);
                if constexpr (PRO == 1) gf[t] = *reinterpret_cast<const u32x4*>(g + t * 32);
            }
        } else {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int k = k_lo + (c * T + t) * 32 + kg;
                const bool in = r16 < M && k < k_hi;
                xf[t] = in ? *reinterpret_cast<const u32x4*>(x + r16 * ldx + k) : z4;
                if constexpr (PRO == 1) gf[t] = in ? *reinterpret_cast<const u32x4*>(nw + k) : z4;
            }
        }
    };
    auto request_w = [&](u32x4 (&w)[T], int64_t g, int c) {
        const int64_t n = g * GN + (r16 & (GN - 1));
        const bf16_t* row = W + ((n < N ? n : N - 1) + (GLU && r16 >= 8 ? N : 0)) * ldw;
        if constexpr (EVEN) {
            if (!on) return;
            row += k_lo + c * T * 32 + kg;
#pragma unroll
            for (int t = 0; t < T; ++t) w[t] = *reinterpret_cast<const u32x4*>(row + t * 32);
            return;
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int k = k_lo + (c * T + t) * 32 + kg;
            w[t] = on && k < k_hi ? *reinterpret_cast<const u32x4*>(row + k) : z4;
        }
    };
    float r = 0.f;  // PRO 1: 1 / rms of the lane's operand row
    auto finish_x = [&]() {
        if constexpr (PRO == 1) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                float a[8], b[8], o[8];
                unpack8(xf[t], a);
                unpack8(gf[t], b);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = a[e] * r * b[e];
                xf[t] = EVEN || r16 < M ? pack8(o) : z4;
            }
        } else if constexpr (PRO == 2) {
#pragma unroll
            for (int t = 0; t < T / 2; ++t) {
                if (2 * t >= M) break;
                float a[8], b[8], o[8];
                unpack8(xf[t], a);
                unpack8(gf[t], b);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = swiglu_act(a[e], b[e]);
                *reinterpret_cast<u32x4*>(&act[wave][2 * t + (lane >> 5)][(lane & 31) * 8]) = pack8(o);
            }
            __builtin_amdgcn_wave_barrier();  // written and read by this wave alone, in order
#pragma unroll
            for (int t = 0; t < T; ++t) xf[t] = r16 < M ? *reinterpret_cast<const u32x4*>(&act[wave][r16 & 7][t * 32 + kg]) : z4;
            __builtin_amdgcn_wave_barrier();
        }
    };
    int64_t g = blockIdx.x;
    if constexpr (EVEN) {  // what no load writes
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if constexpr (!REPEAT) xf[t] = z4;
            if constexpr (!REPEAT && PRO == 1) gf[t] = z4;
            if constexpr (ROWS == 8) w0[t] = w1[t] = z4;
        }
    }
    if constexpr (PRO == 1) {  // row sums: rows wave, wave + NW
        u32x4 v0[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v0[i] = wave < M && (EVEN ? 0 : lane) + 64 * i < nvec ? *reinterpret_cast<const u32x4*>(x + wave * ldx + (lane + 64 * i) * 8) : z4;
        request_x(0);
        request_w(w0, g, 0);
        for (int m = wave; m < M; m += NW) {
            float ss = 0.f, v[8];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if ((EVEN ? 0 : lane) + 64 * i < nvec) {
                    unpack8(m == wave ? v0[i] : *reinterpret_cast<const u32x4*>(x + m * ldx + (lane + 64 * i) * 8), v);
#pragma unroll
                    for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
                }
            for (int i = lane + 256; i < nvec; i += 64) {
                unpack8(*reinterpret_cast<const u32x4*>(x + m * ldx + i * 8), v);
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
            }
            ss = wave_sum(ss);
            if (lane == 0) rs[m] = rsqrtf(ss / (float)K + eps);
        }
        __syncthreads();
        r = rs[r16 & 7];
    } else {
        request_x(0);
        request_w(w0, g, 0);
    }
    finish_x();
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int c = 0, flip = 0;
    // one chunk of one group: the next one's weights are requested first
    auto work = [&](u32x4 (&now)[T], u32x4 (&next)[T]) {
        int64_t gn = g;
        int cn = c + 1;
        const int m = threadIdx.x >> 4;
        const int64_t n = g * GN + r16;
        float add = 0.f;
        if (cn == chunks) {
            cn = 0, gn += gridDim.x;
            if (res && m < M && n < N && r16 < GN) add = OUT ? ((const float*)res)[n] : bf2f(((const bf16_t*)res)[m * ldr + n]);
        }
        if (gn < groups) request_w(next, gn, cn);
#pragma unroll
        for (int t = 0; t < T; ++t)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, now[t]), __builtin_bit_cast(bf16x8, xf[t]), acc, 0, 0, 0);
        if (cn == 0) {
            if (r16 < 8) *reinterpret_cast<f32x4*>(&part[flip][wave][r16][lane >> 4 << 2]) = acc;
            __syncthreads();
            if (m < M && n < N && r16 < GN) {
                float s = part[flip][0][m][r16];
#pragma unroll
                for (int i = 1; i < NW; ++i) s += part[flip][i][m][r16];
                if constexpr (GLU) {
                    float gate = part[flip][0][m][8 + (r16 & 7)];
#pragma unroll
                    for (int i = 1; i < NW; ++i) gate += part[flip][i][m][8 + (r16 & 7)];
                    ((bf16_t*)y)[m * ldy + n] = f2bf(swiglu_act(rbf(s), rbf(gate)));
                } else if constexpr (OUT == OUT_F32) ((float*)y)[m * ldy + n] = res ? s + add : s;
                else ((bf16_t*)y)[m * ldy + n] = f2bf(res ? s + add : s);
            }
            flip ^= 1;  // (the next group's sums go beside these: its barrier is behind every read of them)
            acc = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        if (chunks > 1 && gn < groups) {
            request_x(cn);
            finish_x();
        }
        g = gn, c = cn;
    };
    while (g < groups) {
        work(w0, w1);
        if (g >= groups) break;
        work(w1, w0);
    }
}

// One operand row: a matrix pipe with one column at work gains nothing, and a row fits the registers of every wave in the layout of the weights' strips (512 k, 8 per lane), so
// there is neither an image nor a barrier between the loads and the products (PRO 2 alone shares its activations through LDS: each costs ~ 100 clocks).  One wave = one
// column (GLU: an up column and its gate column), the workgroups walk the columns.  Arithmetic of the prologues and of GLU as above; a sum is a lane's strips in order, then wave_sum.
// PRO 3: the row is a context that the decode attention left in `fold.S` splits; every workgroup folds it, as attn_decode_combine_kernel would (the same bits), into LDS -- S x 8 KB
// from L2 under the weights' flight against a launch of its own: at 590 keys in five splits 3.3 us and the gap behind it.
struct SplitRow {
    const float* ws; int D, S;
};
__device__ __forceinline__ void fold_splits8(const SplitRow& fold, int k, float (&o)[8]) {  // features k .. k + 7 (of one head)
    const int head = k / fold.D, i = k - head * fold.D, pitch = fold.D + 2;
    const float* src = fold.ws + (int64_t)head * fold.S * pitch;
    constexpr int AT = 8;  // splits requested at a time
    float ms[AT], ls[AT];
    f32x2 v[AT][4];
    auto request = [&](int s0) {
#pragma unroll
        for (int j = 0; j < AT; ++j) {
            const float* p = src + min(s0 + j, fold.S - 1) * pitch;
            ms[j] = p[fold.D], ls[j] = p[fold.D + 1];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j][e] = *reinterpret_cast<const f32x2*>(p + i + 2 * e);
        }
    };
    request(0);
    float mg = -__builtin_huge_valf();
#pragma unroll
    for (int j = 0; j < AT; ++j) mg = fmaxf(mg, ms[j]);
    for (int s = AT; s < fold.S; ++s) mg = fmaxf(mg, src[s * pitch + fold.D]);
    float lg = 0.f, out[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = 0.f;
    for (int s0 = 0; s0 < fold.S; s0 += AT) {
        if (s0) request(s0);
#pragma unroll
        for (int j = 0; j < AT; ++j) {
            if (s0 + j >= fold.S) break;
            const float f = ms[j] == -__builtin_huge_valf() ? 0.f : exp2f(ms[j] - mg);  // (a split without keys)
            lg += ls[j] * f;
#pragma unroll
            for (int e = 0; e < 8; ++e) out[e] += v[j][e >> 1][e & 1] * f;
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = out[e] / lg;
}
template <int T, int PRO, int OUT, bool GLU, bool EVEN>
__global__ __launch_bounds__(256) void gemv_one_kernel(int64_t N, int K, const bf16_t* __restrict__ x, const bf16_t* __restrict__ nw, float eps, const bf16_t* __restrict__ W, int64_t ldw,
                                                       void* __restrict__ y, const void* __restrict__ res, SplitRow fold) {
    extern __shared__ __attribute__((aligned(16))) bf16_t act[];  // PRO 2, 3: [K]
    constexpr int C = GLU ? 2 : 1;  // columns of a wave; T strips in registers (the smallest of 2, 4, 8 that holds the row; longer rows go through eight at a time)
    const int lane = threadIdx.x & 63, its = EVEN ? T : (K + 511) >> 9;
    const u32x4 z4 = {0u, 0u, 0u, 0u};
    u32x4 xr[T], nr[PRO == 1 ? T : 1], w[C][T];
    auto request_x = [&](int base) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int k = (base + t) * 512 + lane * 8;
            xr[t] = EVEN || k < K ? *reinterpret_cast<const u32x4*>((PRO >= 2 ? act : x) + k) : z4;
            if constexpr (PRO == 1) nr[t] = EVEN || k < K ? *reinterpret_cast<const u32x4*>(nw + k) : z4;
        }
    };
    auto request_w = [&](int64_t n, int base) {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int k = (base + t) * 512 + lane * 8;
                w[c][t] = EVEN || k < K ? *reinterpret_cast<const u32x4*>(W + (n + c * N) * ldw + k) : z4;
            }
    };
    float r = 0.f;
    auto finish_x = [&]() {
        if constexpr (PRO == 1) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                float a[8], b[8], o[8];
                unpack8(xr[t], a);
                unpack8(nr[t], b);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = a[e] * r * b[e];
                xr[t] = pack8(o);
            }
        }
    };
    const int64_t stride = (int64_t)gridDim.x * 4;
    int64_t n = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if constexpr (PRO == 2) {
        for (int k = threadIdx.x * 8; k < K; k += 2048) {
            float u[8], g[8], o[8];
            unpack8(*reinterpret_cast<const u32x4*>(x + k), u);
            unpack8(*reinterpret_cast<const u32x4*>(x + K + k), g);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = swiglu_act(u[e], g[e]);
            *reinterpret_cast<u32x4*>(act + k) = pack8(o);
        }
        __syncthreads();
    }
    if constexpr (PRO == 3) {
        request_w(n < N ? n : N - 1, 0);
        for (int k = threadIdx.x * 8; k < K; k += 2048) {
            float o[8];
            fold_splits8(fold, k, o);
            *reinterpret_cast<u32x4*>(act + k) = pack8(o);
        }
        __syncthreads();
    }
    if (n >= N) return;  // (no barrier behind this)
    request_x(0);
    if constexpr (PRO != 3) request_w(n, 0);
    if constexpr (PRO == 1) {
        float ss = 0.f, v[8];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            unpack8(xr[t], v);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
        }
        for (int k = T * 512 + lane * 8; !EVEN && k < K; k += 512) {
            unpack8(*reinterpret_cast<const u32x4*>(x + k), v);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
        }
        r = rsqrtf(wave_sum(ss) / (float)K + eps);
    }
    finish_x();
    for (bool first = true; n < N; n += stride) {
        float acc[C];
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] = 0.f;
        float add = 0.f;
        if (res) add = OUT ? ((const float*)res)[n] : bf2f(((const bf16_t*)res)[n]);
        for (int base = 0; base < its; base += T) {
            if (!first) {
                if (its > T) request_x(base);
                request_w(n, base);
                if (its > T) finish_x();
            }
            first = false;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if (base + t >= its) break;
                float xf[8], wf[8];
                unpack8(xr[t], xf);
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    unpack8(w[c][t], wf);
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[c] = fmaf(wf[e], xf[e], acc[c]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] = wave_sum(acc[c]);
        if (lane == 0) {
            if constexpr (GLU) ((bf16_t*)y)[n] = f2bf(swiglu_act(rbf(acc[0]), rbf(acc[C - 1])));
            else if constexpr (OUT == OUT_F32) ((float*)y)[n] = res ? acc[0] + add : acc[0];
            else ((bf16_t*)y)[n] = f2bf(res ? acc[0] + add : acc[0]);
        }
    }
}

// ------------------------------------------------------------------------------------------- decode attention
// grid (Hq, B), WAVES waves; chunks of CK keys go round the waves (chunk c to wave c % WAVES).  D = 32 .. 256.
// POST: the launch starts from the fused QKV stream's raw row instead of finished q rows and a finished cache row -- QK-RMSNorm + RoPE of this head's query (to LDS, never to
// memory) and of its kv head's new key, which goes with the value head into cache row *write_pos, exactly as qknorm_rope_fwd_kernel (norm_rope.hip) computes them: fp32 norm
// rounded to bf16, bf16-rounded cos / sin, every product rounded.  The query heads of one kv head all write the same bytes to the same row; each workgroup reads back its own.
struct QkvPost {
    const bf16_t* qkv; int64_t ldqkv; const bf16_t* qw; const bf16_t* kw; const float* cosT; const float* sinT; const int32_t* pos; const int32_t* write_pos; int capacity; float eps;
};

// Sums and maxima over lanes on the VALU: a ds_bpermute (what __shfl_xor compiles to) is an LDS round trip, and a one-token step's attention is a chain of them.
__device__ __forceinline__ float other16(float v, bool max) {  // with the lane whose number differs in bit 4
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return max ? fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) : __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float other32(float v, bool max) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return max ? fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) : __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int CH>
__device__ __forceinline__ float chunk_sum(float v) {  // over the CH lanes that hold a key's features
    if constexpr (CH <= 16) return lanes_sum<CH>(v);
    else return other16(lanes_sum<16>(v), false);
}
template <int CH>
__device__ __forceinline__ float across_groups(float v, bool max) {  // over the 64 / CH lanes of one chunk
#pragma unroll
    for (int o = CH; o < 16; o <<= 1) {
        const float w = __shfl_xor(v, o, 64);
        v = max ? fmaxf(v, w) : v + w;
    }
    if constexpr (CH <= 16) v = other16(v, max);
    return other32(v, max);
}

// QK-RMSNorm + RoPE of one head in two stages (request the operands; later, finish): lane i < D / 2 holds features i and D / 2 + i.  The bits of qknorm_rope_fwd_kernel
// (norm_rope.hip), whose lanes hold eight features of each half: the sum of squares is taken in that order -- eight neighbours one after the other, then the groups of eight in a
// tree -- but an element's arithmetic runs once, not eight times over (a wave's whole norm and rotation 1 500 -> 500 clocks, at the head of a one-token step's chain).
struct HeadOperands {
    bf16_t w1, w2, x1, x2;
    float c1, s1, c2, s2;
    template <int D>
    __device__ __forceinline__ void load(const bf16_t* __restrict__ src, const bf16_t* __restrict__ w, const float* __restrict__ cosT, const float* __restrict__ sinT, int64_t p, int lane) {
        constexpr int HALF = D / 2;
        const int i = lane % HALF;
        x1 = src[i], x2 = src[HALF + i], w1 = w[i], w2 = w[HALF + i];
        c1 = cosT[p * D + i], s1 = sinT[p * D + i], c2 = cosT[p * D + HALF + i], s2 = sinT[p * D + HALF + i];
    }
    template <int D>
    __device__ __forceinline__ void finish(float eps, float& y1, float& y2) const {
        const float xf1 = bf2f(x1), xf2 = bf2f(x2), t = xf1 * xf1 + xf2 * xf2;
        float ss = 0.f;  // of eight lanes, at the first of them (row_shl:k brings the value of the lane k further on)
        ss += t;
        ss += dpp_f<0x101>(t), ss += dpp_f<0x102>(t), ss += dpp_f<0x103>(t), ss += dpp_f<0x104>(t), ss += dpp_f<0x105>(t), ss += dpp_f<0x106>(t), ss += dpp_f<0x107>(t);
        if constexpr (D == 128) ss = other32(ss, false);
        ss = other16(ss, false);
        ss += dpp_f<0x128>(ss);  // row_ror:8
        ss = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(ss)));
        const float r = rsqrtf(ss / (float)D + eps);
        const float n1 = rbf(xf1 * r * bf2f(w1)), n2 = rbf(xf2 * r * bf2f(w2));
        y1 = rbf(rbf(rbf(c1) * n1) + rbf(rbf(s1) * (-n2)));
        y2 = rbf(rbf(rbf(c2) * n2) + rbf(rbf(s2) * n1));
    }
};

template <int D, int WAVES, bool POST>
__global__ __launch_bounds__(64 * WAVES) void attn_decode_kernel(int Hq, int Hkv, const bf16_t* __restrict__ q, const bf16_t* kc, const bf16_t* vc, int64_t batch_stride,
                                                                 int64_t ld, int len, const int32_t* __restrict__ len_dev, const uint8_t* __restrict__ key_mask, int64_t ldm,
                                                                 bf16_t* __restrict__ o, float scale_log2, QkvPost post, float* __restrict__ ws) {
    // One mapping for both products: lane = (key group kg, 16-byte feature chunk ch); a load instruction covers KG whole key rows, coalesced.  Scores: 8 features per lane,
    // folded over the CH lanes of a key; P V: the key groups are folded at the end.  Rows of the new token never come back from memory (POST: they are used from LDS, the cache
    // row is written for the later steps only).
    // Bound: one wave's chain -- arguments, position, angles, norm and rotation; cache rows; scores, softmax, P V -- of which the arithmetic was the longer half (a wave's vector
    // instruction takes four clocks whatever it does): few keys per wave, no per-lane branch round a load, the new token's norm and rotation on waves without keys.  Eight keys a
    // lane and everything behind the position's load -> now: 1 sequence x 100 keys 8.2 -> 5.4 us, 6 x 80 8.3 -> 5.5, 590 keys in three splits 9.5 -> 6.7, in five 5.8.  (Sixteen waves
    // instead of a second round: 7.3 for the 6.7.)
    constexpr int CH = D / 8, KG = 64 / CH;
    constexpr int NT = 4;        // keys per lane and chunk: 2 x NT 16-byte rows in flight per lane
    constexpr int CK = NT * KG;  // keys per chunk; chunk c belongs to split c % S (blockIdx.z of S = gridDim.z), there to wave (c / S) % WAVES
    // S > 1 (long caches): every split leaves its un-normalised context, maximum and sum in `ws` ([B, Hq, S, D + 2] floats), folded in split order by who reads them.
    __shared__ float qs[D];
    __shared__ __attribute__((aligned(16))) bf16_t ksn[POST ? D : 8], vsn[POST ? D : 8];
    __shared__ float part[WAVES][D + 2];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = lane / CH, ch = lane % CH;
    const int h = blockIdx.x, b = blockIdx.y, hk = h / (Hq / Hkv);
    const int S = gridDim.z, sp = blockIdx.z;
    const int c0 = sp + S * wave, cstep = S * WAVES;
    // A wave's first rows are requested by the bound that the host knows, in front of what the device alone knows (the length, the new token's row and position: a memory round
    // trip), where the bound is no longer than four rounds of the workgroups; what is read past the length is dropped below.  POST: the row at the bound's end is left out, for
    // where the host knows the length it is the new token's, being written now by the heads that share it.
    const bool early = len <= 4 * CK * WAVES * S;
    const int bound = len;
    int first = POST ? max(bound - 1, 1) : bound;
    if (!early && len_dev) first = min(bound, *len_dev);
    int wp = -1;  // POST: the cache row of the new token (its key / value are taken from LDS)
    const bf16_t* kb = kc + b * batch_stride + (int64_t)hk * D + ch * 8;
    const bf16_t* vb = vc + b * batch_stride + (int64_t)hk * D + ch * 8;
    u32x4 kraw[NT], vraw[NT];
    auto request = [&](u32x4 (&r)[NT], const bf16_t* from, int base, int bound) {  // (rows past the bound: the last one; the new token's row, being written now, is read and not used)
        if (base >= bound) return;
#pragma unroll
        for (int t = 0; t < NT; ++t) r[t] = *reinterpret_cast<const u32x4*>(from + (int64_t)min(base + t * KG + kg, bound - 1) * ld);
    };
    if constexpr (POST) {
        static_assert(D == 64 || D == 128, "QK-norm + RoPE geometry: 8 features per lane and half");
        constexpr int HALF = D / 2;
        const bf16_t* row = post.qkv + b * post.ldqkv;
        // The last waves, which short caches leave without keys, finish the query, the new key and the new value.  Loads return in order: their operands are requested in front
        // of their cache rows, and their arithmetic runs under the rows' flight.
        HeadOperands hop;
        u32x4 vnew = {0u, 0u, 0u, 0u};
        const int role = WAVES - 1 - wave;
        if (role < 2) hop.load<D>(row + (int64_t)(role == 0 ? h : Hq + hk) * D, role == 0 ? post.qw : post.kw, post.cosT, post.sinT, post.pos[b], lane);
        else if (role == 2 && lane < D / 8) vnew = *reinterpret_cast<const u32x4*>(row + (int64_t)(Hq + Hkv + hk) * D + lane * 8);
        request(kraw, kb, c0 * CK, first);
        request(vraw, vb, c0 * CK, first);
        wp = *post.write_pos;
        len = min(len, *len_dev);
        const bool room = wp >= 0 && wp < post.capacity;  // never write outside the cache
        if (early && len == bound && wp != bound - 1) {   // (the row that was left out is an old one)
            request(kraw, kb, c0 * CK, bound);
            request(vraw, vb, c0 * CK, bound);
        }
        if (role < 2) {
            float y1, y2;
            hop.finish<D>(post.eps, y1, y2);
            if (lane < HALF) {
                if (role == 0) {
                    qs[lane] = y1, qs[HALF + lane] = y2;
                } else {
                    const bf16_t p1 = f2bf(y1), p2 = f2bf(y2);
                    ksn[lane] = p1, ksn[HALF + lane] = p2;
                    if (room) {
                        bf16_t* dst = const_cast<bf16_t*>(kc) + b * batch_stride + (int64_t)wp * ld + (int64_t)hk * D;
                        dst[lane] = p1, dst[HALF + lane] = p2;
                    }
                }
            }
        } else if (role == 2 && lane < D / 8) {
            *reinterpret_cast<u32x4*>(vsn + lane * 8) = vnew;
            if (room) *reinterpret_cast<u32x4*>(const_cast<bf16_t*>(vc) + b * batch_stride + (int64_t)wp * ld + (int64_t)hk * D + lane * 8) = vnew;
        }
    } else {
        for (int i = threadIdx.x; i < D; i += 64 * WAVES) qs[i] = bf2f(q[((int64_t)b * Hq + h) * D + i]);
        request(kraw, kb, c0 * CK, first);
        request(vraw, vb, c0 * CK, first);
        if (len_dev) len = min(len, *len_dev);  // graph replay: the current length lives on the device, `len` is the capacity bound
    }
    __syncthreads();
    const uint8_t* km = key_mask ? key_mask + b * ldm : nullptr;
    float qf[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) qf[e] = qs[ch * 8 + e];
    float m = -__builtin_huge_valf(), l = 0.f, acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    for (int base = c0 * CK; base < len; base += cstep * CK) {
        const int nb = base + cstep * CK;
        u32x4 kn = {0u, 0u, 0u, 0u}, vn = kn;
        if constexpr (POST) kn = *reinterpret_cast<const u32x4*>(ksn + ch * 8), vn = *reinterpret_cast<const u32x4*>(vsn + ch * 8);
#pragma unroll
        for (int t = 0; t < NT; ++t) {  // (selects, no branches: cold code would cost the one wave that meets the new token or the end more than these cost all)
            const int j = base + t * KG + kg;
            if constexpr (POST) kraw[t] = j == wp ? kn : kraw[t], vraw[t] = j == wp ? vn : vraw[t];
            vraw[t] = j < len ? vraw[t] : u32x4{0u, 0u, 0u, 0u};  // (a probability of 0 times whatever lies there)
        }
        float sc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float kf[8];
            unpack8(kraw[t], kf);
            float d = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) d = fmaf(kf[e], qf[e], d);
            sc[t] = chunk_sum<CH>(d) * scale_log2;
        }
        if (nb < len) request(kraw, kb, nb, len);  // the next round's rows travel under this round's arithmetic
        if (km) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (!km[min(base + t * KG + kg, len - 1)]) sc[t] = MASK_T;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) sc[t] = base + t * KG + kg < len ? sc[t] : -__builtin_huge_valf();  // keys beyond the cache do not exist
        float mc = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
        mc = across_groups<CH>(mc, true);
        const float mn = fmaxf(m, mc);
        const float alpha = __builtin_amdgcn_exp2f(m - mn);  // m = -inf on the first chunk -> 0
        float psum = 0.f;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            sc[t] = __builtin_amdgcn_exp2f(sc[t] - mn);  // -inf -> 0
            psum += sc[t];
        }
        psum = across_groups<CH>(psum, false);
        l = l * alpha + psum;
        m = mn;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] *= alpha;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float vf[8];
            unpack8(vraw[t], vf);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] = fmaf(sc[t], vf[e], acc[e]);
        }
        if (nb < len) request(vraw, vb, nb, len);
    }
    // fold the key groups of the wave (lanes with the same chunk), then combine the waves' key ranges
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = across_groups<CH>(acc[e], false);
    if (kg == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) part[wave][ch * 8 + e] = acc[e];
    }
    if (lane == 0) {
        part[wave][D] = m;
        part[wave][D + 1] = l;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < D; i += 64 * WAVES) {
        float mw[WAVES], mg = -__builtin_huge_valf();
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mg = fmaxf(mg, mw[w] = part[w][D]);
        float lg = 0.f, out = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float f = mw[w] == -__builtin_huge_valf() ? 0.f : __builtin_amdgcn_exp2f(mw[w] - mg);
            lg += part[w][D + 1] * f;
            out += part[w][i] * f;
        }
        if (S == 1) {
            o[((int64_t)b * Hq + h) * D + i] = f2bf(out / lg);
        } else {
            float* dst = ws + (((int64_t)b * Hq + h) * S + sp) * (D + 2);
            dst[i] = out;
            if (i == 0) { dst[D] = mg; dst[D + 1] = lg; }
        }
    }
}

// The splits of one (sequence, head) folded in split order: grid (Hq, B), D threads.
__global__ void attn_decode_combine_kernel(int Hq, int D, int S, const float* __restrict__ ws, bf16_t* __restrict__ o) {
    const int h = blockIdx.x, b = blockIdx.y, i = threadIdx.x;
    const float* src = ws + ((int64_t)b * Hq + h) * S * (D + 2);
    float mg = -__builtin_huge_valf();
    for (int s = 0; s < S; ++s) mg = fmaxf(mg, src[s * (D + 2) + D]);
    float lg = 0.f, out = 0.f;
    for (int s = 0; s < S; ++s) {
        const float ms = src[s * (D + 2) + D];
        const float f = ms == -__builtin_huge_valf() ? 0.f : exp2f(ms - mg);  // a split without keys
        lg += src[s * (D + 2) + D + 1] * f;
        out += src[s * (D + 2) + i] * f;
    }
    o[((int64_t)b * Hq + h) * D + i] = f2bf(out / lg);
}

// The tail of a greedy step: the chosen ids become the next input ids, every counter of the device-side bookkeeping moves on by one (one launch instead of four).
__global__ void decode_advance_kernel(int B, const int64_t* __restrict__ next, int64_t* __restrict__ tok, int32_t* __restrict__ rope_pos, int32_t* __restrict__ write_pos,
                                      int32_t* __restrict__ length) {
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i < B) {
        tok[i] = next[i];
        rope_pos[i] += 1;
    }
    if (i == 0) {
        *write_pos += 1;
        *length += 1;
    }
}

// cache[b, pos[0], :] = rows[b, :] for K and V: the KVCache append of one decoded token with the position read from the device
__global__ void kv_append_kernel(int B, int width, const bf16_t* __restrict__ k_rows, int64_t ldk, const bf16_t* __restrict__ v_rows, int64_t ldv,
                                 bf16_t* __restrict__ kc, bf16_t* __restrict__ vc, int64_t batch_stride, int64_t ld, int capacity,
                                 const int32_t* __restrict__ pos) {
    const int vec = width >> 3;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)B * vec) return;
    const int b = (int)(idx / vec), c = (int)(idx % vec);
    const int p = *pos;
    if (p < 0 || p >= capacity) return;  // never write outside the cache
    *reinterpret_cast<u32x4*>(kc + b * batch_stride + (int64_t)p * ld + c * 8) = *reinterpret_cast<const u32x4*>(k_rows + b * ldk + c * 8);
    *reinterpret_cast<u32x4*>(vc + b * batch_stride + (int64_t)p * ld + c * 8) = *reinterpret_cast<const u32x4*>(v_rows + b * ldv + c * 8);
}

// cache[b, start + s, :] = rows[b * S + s, :] for K and V, position known on the host: the whole append in one launch instead of one strided copy per sequence and
// operand (6 sequences: 12 launches a layer; a one-token step of 28 layers spent 8 400 of its 13 700 launches on them).  Launch-bound at one token per sequence,
// a plain 16-byte copy stream for a prompt.
__global__ __launch_bounds__(256) void kv_append_rows_kernel(int64_t total, int S, int wvec, const char* __restrict__ k_rows, int64_t ldk, const char* __restrict__ v_rows, int64_t ldv,
                                                             char* __restrict__ kc, char* __restrict__ vc, int64_t batch_stride, int64_t ld, int start) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / wvec, c = (i - row * wvec) * 16;
        const int64_t b = row / S, s = row - b * S;
        const int64_t dst = b * batch_stride + (start + s) * ld + c;
        *reinterpret_cast<u32x4*>(kc + dst) = *reinterpret_cast<const u32x4*>(k_rows + row * ldk + c);
        *reinterpret_cast<u32x4*>(vc + dst) = *reinterpret_cast<const u32x4*>(v_rows + row * ldv + c);
    }
}

// two stages so that a handful of rows still fills the chip: stage 1 = ARG_SPLIT column ranges per row, stage 2 = merge
constexpr int ARG_SPLIT = 64;
__device__ __forceinline__ void argmax_merge(float& best, int64_t& idx, float ov, int64_t oi) {
    if (ov > best || (ov == best && oi < idx)) {
        best = ov;
        idx = oi;
    }
}
__device__ __forceinline__ float argmax_load(const bf16_t* p) { return bf2f(*p); }
__device__ __forceinline__ float argmax_load(const float* p) { return *p; }
template <typename T>
__global__ __launch_bounds__(256) void argmax_part_kernel(int64_t V, const T* __restrict__ x, int64_t ld, float* __restrict__ pv, int64_t* __restrict__ pi) {
    __shared__ float bv[4];
    __shared__ int64_t bi[4];
    const T* r = x + (int64_t)blockIdx.y * ld;
    const int64_t span = (V + ARG_SPLIT - 1) / ARG_SPLIT, c0 = blockIdx.x * span, c1 = c0 + span < V ? c0 + span : V;
    float best = -__builtin_huge_valf();
    int64_t idx = 0x7fffffffffffffffll;
    for (int64_t i = c0 + threadIdx.x; i < c1; i += 256) {
        const float v = argmax_load(r + i);
        if (v > best) {
            best = v;
            idx = i;
        }
    }
    for (int o = 32; o > 0; o >>= 1) argmax_merge(best, idx, __shfl_xor(best, o, 64), __shfl_xor(idx, o, 64));
    if ((threadIdx.x & 63) == 0) {
        bv[threadIdx.x >> 6] = best;
        bi[threadIdx.x >> 6] = idx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) argmax_merge(best, idx, bv[w], bi[w]);
        pv[(int64_t)blockIdx.y * ARG_SPLIT + blockIdx.x] = best;
        pi[(int64_t)blockIdx.y * ARG_SPLIT + blockIdx.x] = idx;
    }
}
__global__ __launch_bounds__(64) void argmax_merge_kernel(const float* __restrict__ pv, const int64_t* __restrict__ pi, int64_t* __restrict__ out) {
    float best = pv[(int64_t)blockIdx.x * ARG_SPLIT + threadIdx.x];
    int64_t idx = pi[(int64_t)blockIdx.x * ARG_SPLIT + threadIdx.x];
    for (int o = 32; o > 0; o >>= 1) argmax_merge(best, idx, __shfl_xor(best, o, 64), __shfl_xor(idx, o, 64));
    if (threadIdx.x == 0) out[blockIdx.x] = idx;
}

}  // namespace

#define ST(s) ((hipStream_t)(s))

// One row: gemv_one_kernel.  Two to eight: eight waves and at most a workgroup for each CU; four waves and two workgroups a CU where they walk many groups (a table of 151 936
// rows: 56 us so, 64 with eight waves and 59 with four workgroups; 6144 x 1024: 7.9 us with eight waves, 8.7 with four; sixteen waves spill under a prologue).  Twelve waves where
// eight would take a second chunk and half of it empty (K of 2 049 to 3 072): its operands are only requested behind the first one's products.  Groups of eight weight rows, not
// sixteen, while those leave half the CUs without one: a CU's loads, 64 bytes a clock, are what a group takes longest for.  Both together: 1024 x 2048 and 1024 x 3072, six rows, 5.7
// us in the mean of the two (by the profiler's clock) -> 4.4 and 5.4.  How many waves share a sum depends on N and K alone, so a product with its prologue keeps the bits of the two launches.
// us of one launch, weights from memory, before (a column per wave on the vector pipe for up to eight rows) -> the matrix pipe in groups of 16 (without EVEN, whose figures stand at the kernel):   N x K      1 row          6 rows
//     RMSNorm + 4096 x 1024    4.9 -> 4.5     9.0 -> 6.2          |   1024 x 3072 (from activated rows)    4.6 -> 3.5     7.9 -> 5.8
//     RMSNorm + 6144 x 1024    6.6 -> 5.7    11.3 -> 7.9          |   1024 x 2048                          3.8 -> 2.9     6.3 -> 4.5
//     RMSNorm + 151936 x 1024   52 -> 52      152 -> 56           |   3072 x 4096                          8.5 -> 7.1    14.0 -> 9.0
template <int PRO, int OUT, bool GLU = false>
static void gemv_launch(int M, int64_t N, int K, const void* x, int64_t ldx, const void* nw, float eps, const void* W, int64_t ldw, void* y, int64_t ldy, const void* res, int64_t ldr, void* stream, SplitRow fold = {}) {
    if (M == 1) {
        const int64_t blocks = (N + 3) / 4;
#define GEMV(T) (K == T * 512 ? gemv_one_kernel<T, PRO, OUT, GLU, true> : gemv_one_kernel<T, PRO, OUT, GLU, false>)<<<(int)(blocks < 2048 ? blocks : 2048), 256, PRO >= 2 ? (size_t)K * 2 : 0, ST(stream)>>>(N, K, (const bf16_t*)x, (const bf16_t*)nw, eps, (const bf16_t*)W, ldw, y, res, fold)
        if (K <= 1024) GEMV(2); else if (K <= 2048) GEMV(4); else if (K <= 3072) GEMV(6); else GEMV(8);
#undef GEMV
        return;
    }
    if constexpr (PRO != 3) {
        const int all = (K + 31) / 32;
        const int64_t groups = ((GLU ? 2 * N : N) + 15) / 16;
        const int waves = groups >= 1024 ? 4 : all > 8 * GEMV_STEPS && all <= 12 * GEMV_STEPS ? 12 : 8, most = waves == 4 ? 512 : 256;
        const bool half = !GLU && groups <= 128;
        const int64_t work = half ? (N + 7) / 8 : groups;
        const int grid = (int)(work < most ? work : most), steps = (all + waves - 1) / waves;
        const bool even = PRO != 2 && K == steps * waves * 32;
        constexpr int T4 = PRO == 2 ? GEMV_STEPS : 4;
#define GEMV(NW, R) \
    (even && steps % GEMV_STEPS == 0       ? gemv_kernel<NW, PRO, OUT, GLU, R, GEMV_STEPS, PRO != 2> \
     : even && steps == 4                  ? gemv_kernel<NW, PRO, OUT, GLU, R, T4, PRO != 2> \
                                           : gemv_kernel<NW, PRO, OUT, GLU, R, GEMV_STEPS, false>)<<<grid, 64 * NW, 0, ST(stream)>>>(M, N, K, steps, (const bf16_t*)x, ldx, (const bf16_t*)nw, eps, (const bf16_t*)W, ldw, (void*)y, ldy, res, ldr)
        if (waves == 4) GEMV(4, 16);
        else if (half && !GLU) {
            if (waves == 12) GEMV(12, GLU ? 16 : 8); else GEMV(8, GLU ? 16 : 8);
        } else if (waves == 12) GEMV(12, 16);
        else GEMV(8, 16);
#undef GEMV
    }
}

extern "C" int mi355_gemv_bf16(int M, int64_t N, int K, const void* x, int64_t ldx, const void* W, int64_t ldw, void* y, int64_t ldy,
                               const void* residual, int64_t ldr, void* stream) {
    MI355_REQUIRE(M >= 1 && M <= 8, "gemv_bf16: 1..8 rows (got %d); larger batches go through mi355_gemm_bf16", M);
    MI355_REQUIRE(N > 0 && K > 0 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= K && ldw >= K && ldy >= N, "gemv_bf16: K and the leading dimensions of x / W must be multiples of 8");
    MI355_REQUIRE(x && W && y && (!residual || ldr >= N), "gemv_bf16: null pointer or residual pitch too small");
    gemv_launch<0, OUT_BF16>(M, N, K, x, ldx, nullptr, 0.f, W, ldw, y, ldy, residual, ldr, stream);
    MI355_LAUNCH_CHECK("gemv_bf16");
    return 0;
}

extern "C" int mi355_gemv_bf16_f32out(int M, int64_t N, int K, const void* x, int64_t ldx, const void* W, int64_t ldw, float* y, int64_t ldy, const float* bias,
                                      void* stream) {
    MI355_REQUIRE(M >= 1 && M <= 8, "gemv_bf16_f32out: 1..8 rows (got %d)", M);
    MI355_REQUIRE(N > 0 && K > 0 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= K && ldw >= K && ldy >= N, "gemv_bf16_f32out: K and the leading dimensions of x / W must be multiples of 8");
    MI355_REQUIRE(x && W && y, "gemv_bf16_f32out: null pointer");
    gemv_launch<0, OUT_F32>(M, N, K, x, ldx, nullptr, 0.f, W, ldw, y, ldy, bias, 0, stream);
    MI355_LAUNCH_CHECK("gemv_bf16_f32out");
    return 0;
}

// bgemm.hip's products of one to eight bf16 rows with a bias, results in bf16
extern "C" __attribute__((visibility("hidden"))) void mi355_gemv_bias_part(int M, int64_t N, int K, const void* x, int64_t ldx, const void* W, int64_t ldw, void* y, int64_t ldy, const float* bias, void* stream) {
    gemv_launch<0, OUT_BF16_BIAS>(M, N, K, x, ldx, nullptr, 0.f, W, ldw, y, ldy, bias, 0, stream);
}

extern "C" int mi355_gemv_bf16_pro(int M, int64_t N, int K, const void* x, int64_t ldx, int prologue, const void* norm_w, float eps, const void* W, int64_t ldw,
                                   void* y, int64_t ldy, const void* residual, int64_t ldr, void* stream) {
    MI355_REQUIRE(M >= 1 && M <= 8, "gemv_bf16_pro: 1..8 rows (got %d)", M);
    MI355_REQUIRE(prologue == 1 || prologue == 2, "gemv_bf16_pro: prologue 1 (RMSNorm of x) or 2 (SwiGLU of gate-up rows), got %d", prologue);
    MI355_REQUIRE(N > 0 && K > 0 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= (prologue == 2 ? 2 * K : K) && ldw >= K && ldy >= N,
                  "gemv_bf16_pro: K and the leading dimensions must be multiples of 8 (x rows hold 2K elements under prologue 2)");
    // Where the entry ends, and ops_decode.fused_rows with it; beyond, the row operation has a launch of its own.  Only one row's activations (prologue 2) are in LDS as a whole; the line
    // is where an earlier image of all rows ended, and is kept because it decides which launches, and so which bits, a step of that size has.
    MI355_REQUIRE((int64_t)M * K * 2 + 32 <= 65536, "gemv_bf16_pro: takes operand rows (here %d x %d bf16) up to 64 KiB less 32 bytes", M, K);
    MI355_REQUIRE(x && W && y && (!residual || ldr >= N) && (prologue != 1 || norm_w), "gemv_bf16_pro: null pointer or residual pitch too small");
    if (prologue == 1) gemv_launch<1, OUT_BF16>(M, N, K, x, ldx, norm_w, eps, W, ldw, y, ldy, residual, ldr, stream);
    else gemv_launch<2, OUT_BF16>(M, N, K, x, ldx, nullptr, 0.f, W, ldw, y, ldy, residual, ldr, stream);
    MI355_LAUNCH_CHECK("gemv_bf16_pro");
    return 0;
}

extern "C" int mi355_kv_append(int B, int width, const void* k_rows, int64_t ldk, const void* v_rows, int64_t ldv, void* k_cache, void* v_cache,
                               int64_t batch_stride, int64_t ld, int capacity, const int32_t* pos, void* stream) {
    MI355_REQUIRE(B > 0 && width > 0 && width % 8 == 0 && ldk % 8 == 0 && ldv % 8 == 0 && ld % 8 == 0, "kv_append: width and pitches must be multiples of 8 elements");
    MI355_REQUIRE(k_rows && v_rows && k_cache && v_cache && pos && capacity > 0 && ld >= width && batch_stride >= (int64_t)capacity * ld, "kv_append: bad arguments");
    kv_append_kernel<<<(int)(((int64_t)B * (width / 8) + 255) / 256), 256, 0, ST(stream)>>>(B, width, (const bf16_t*)k_rows, ldk, (const bf16_t*)v_rows, ldv, (bf16_t*)k_cache, (bf16_t*)v_cache, batch_stride, ld, capacity, pos);
    MI355_LAUNCH_CHECK("kv_append");
    return 0;
}

extern "C" int mi355_kv_append_rows(int B, int S, int64_t width_bytes, const void* k_rows, int64_t ldk_bytes, const void* v_rows, int64_t ldv_bytes, void* k_cache, void* v_cache,
                                    int64_t batch_stride_bytes, int64_t ld_bytes, int start, int capacity, void* stream) {
    MI355_REQUIRE(B > 0 && S > 0 && width_bytes > 0 && start >= 0 && capacity > 0 && (int64_t)start + S <= capacity, "kv_append_rows: rows [%d, %lld) of a cache of %d", start, (long long)start + S, capacity);
    MI355_REQUIRE(k_rows && v_rows && k_cache && v_cache, "kv_append_rows: null pointer");
    MI355_REQUIRE(((width_bytes | ldk_bytes | ldv_bytes | batch_stride_bytes | ld_bytes | (int64_t)(uintptr_t)k_rows | (int64_t)(uintptr_t)v_rows | (int64_t)(uintptr_t)k_cache |
                    (int64_t)(uintptr_t)v_cache) & 15) == 0, "kv_append_rows: addresses, pitches and the row width must be multiples of 16 bytes");
    MI355_REQUIRE(width_bytes <= (1 << 30) && ldk_bytes >= width_bytes && ldv_bytes >= width_bytes && ld_bytes >= width_bytes && batch_stride_bytes / ld_bytes >= capacity,
                  "kv_append_rows: a pitch is smaller than what it spans");
    const int wvec = (int)(width_bytes >> 4);
    const int64_t total = (int64_t)B * S * wvec, blocks = (total + 255) / 256;
    kv_append_rows_kernel<<<(int)(blocks < 2048 ? blocks : 2048), 256, 0, ST(stream)>>>(total, S, wvec, (const char*)k_rows, ldk_bytes, (const char*)v_rows, ldv_bytes, (char*)k_cache, (char*)v_cache,
                                                                                       batch_stride_bytes, ld_bytes, start);
    MI355_LAUNCH_CHECK("kv_append_rows");
    return 0;
}

static int attn_decode_launch(const char* who, int B, int Hq, int Hkv, int D, const void* q, const void* k_cache, const void* v_cache, int64_t batch_stride, int64_t ld, int len,
                              const int32_t* len_dev, const uint8_t* key_mask, int64_t ldm, void* o, float scale, const QkvPost* post, int splits, float* workspace,
                              void* stream, bool combine = true) {
    MI355_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && len > 0, "%s: bad sizes", who);
    MI355_REQUIRE(k_cache && v_cache && o && ld >= (int64_t)Hkv * D && ld % 8 == 0 && batch_stride >= (int64_t)len * ld, "%s: cache pitch / stride too small", who);
    MI355_REQUIRE(!key_mask || ldm >= len, "%s: key mask pitch smaller than the cache length", who);
    MI355_REQUIRE(B <= 65535, "%s: grid limits", who);
    MI355_REQUIRE(splits >= 1 && splits <= 64 && (splits == 1 || workspace), "%s: 1..64 splits, and a workspace of B * Hq * splits * (D + 2) floats for more than one", who);
    dim3 grid(Hq, B, splits);
    const QkvPost none = {};
#define LAUNCH(DD, WV, PP) attn_decode_kernel<DD, WV, PP><<<grid, 64 * WV, 0, ST(stream)>>>(Hq, Hkv, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, batch_stride, ld, len, len_dev, key_mask, ldm, (bf16_t*)o, scale * LOG2E, PP ? *post : none, workspace)
    if (post) {
        if (D == 64) LAUNCH(64, 8, true); else LAUNCH(128, 8, true);
    } else {
        if (D == 32) LAUNCH(32, 8, false); else if (D == 64) LAUNCH(64, 8, false); else if (D == 128) LAUNCH(128, 8, false); else LAUNCH(256, 8, false);
    }
#undef LAUNCH
    if (splits > 1 && combine) attn_decode_combine_kernel<<<dim3(Hq, B), D, 0, ST(stream)>>>(Hq, D, splits, workspace, (bf16_t*)o);
    return 0;
}

extern "C" int mi355_attn_decode(int B, int Hq, int Hkv, int D, const void* q, const void* k_cache, const void* v_cache, int64_t batch_stride,
                                 int64_t ld, int len, const int32_t* len_dev, const uint8_t* key_mask, int64_t ldm, void* o, float scale, int splits, float* workspace,
                                 void* stream) {
    MI355_REQUIRE(D == 32 || D == 64 || D == 128 || D == 256, "attn_decode: head_dim %d not built (32, 64, 128, 256)", D);
    MI355_REQUIRE(q != nullptr, "attn_decode: null query");
    if (int rc = attn_decode_launch("attn_decode", B, Hq, Hkv, D, q, k_cache, v_cache, batch_stride, ld, len, len_dev, key_mask, ldm, o, scale, nullptr, splits, workspace, stream)) return rc;
    MI355_LAUNCH_CHECK("attn_decode");
    return 0;
}

static int attn_decode_qkv(int B, int Hq, int Hkv, int D, const void* qkv, int64_t ldqkv, const void* q_norm_w, const void* k_norm_w, const float* cos,
                                     const float* sin, const int32_t* pos, void* k_cache, void* v_cache, int64_t batch_stride, int64_t ld, int capacity,
                                     const int32_t* write_pos, const int32_t* len_dev, const uint8_t* key_mask, int64_t ldm, void* o, float scale, float eps, int splits,
                           float* workspace, void* stream, bool combine) {
    MI355_REQUIRE(D == 128 || D == 64, "attn_decode_qkv: head_dim must be 64 or 128 (got %d)", D);
    MI355_REQUIRE(Hq > 0 && Hkv > 0 && ldqkv >= (int64_t)(Hq + 2 * Hkv) * D && ldqkv % 8 == 0, "attn_decode_qkv: the qkv row holds (Hq + 2 Hkv) * D elements, pitch a multiple of 8");
    MI355_REQUIRE(qkv && q_norm_w && k_norm_w && cos && sin && pos && write_pos && len_dev, "attn_decode_qkv: null pointer (the write position and the length live on the device)");
    const QkvPost post = {(const bf16_t*)qkv, ldqkv, (const bf16_t*)q_norm_w, (const bf16_t*)k_norm_w, cos, sin, pos, write_pos, capacity, eps};
    if (int rc = attn_decode_launch("attn_decode_qkv", B, Hq, Hkv, D, nullptr, k_cache, v_cache, batch_stride, ld, capacity, len_dev, key_mask, ldm, o, scale, &post, splits, workspace, stream, combine)) return rc;
    MI355_LAUNCH_CHECK("attn_decode_qkv");
    return 0;
}

extern "C" int mi355_attn_decode_qkv(int B, int Hq, int Hkv, int D, const void* qkv, int64_t ldqkv, const void* q_norm_w, const void* k_norm_w, const float* cos,
                                     const float* sin, const int32_t* pos, void* k_cache, void* v_cache, int64_t batch_stride, int64_t ld, int capacity,
                                     const int32_t* write_pos, const int32_t* len_dev, const uint8_t* key_mask, int64_t ldm, void* o, float scale, float eps, int splits,
                                     float* workspace, void* stream) {
    return attn_decode_qkv(B, Hq, Hkv, D, qkv, ldqkv, q_norm_w, k_norm_w, cos, sin, pos, k_cache, v_cache, batch_stride, ld, capacity, write_pos, len_dev, key_mask, ldm, o, scale, eps,
                           splits, workspace, stream, true);
}

// One layer of a one-token step (M = B <= 8 rows): the step's launches behind one call.  A launch costs the host 3.5 us and its Python around it as much again and more (checks,
// an allocation, parameter look-ups): 28 layers x 5 launches of ~ 8 us were 2.4 ms of host time a token beside 1.3 ms of kernels.
namespace {
constexpr int64_t pad8(int64_t n) { return (n + 7) / 8 * 8; }
}  // namespace

extern "C" int64_t mi355_decode_block_scratch_bytes(int B, int d, int F, int Hq, int Hkv, int D, int splits) {
    if (B < 1 || d < 1 || F < 1 || Hq < 1 || Hkv < 1 || D < 1 || splits < 1) return 0;
    const int64_t rows = pad8((int64_t)(Hq + 2 * Hkv) * D) + pad8((int64_t)Hq * D) + pad8(d) + pad8(F);
    return B * rows * 2 + (splits > 1 ? (int64_t)B * Hq * splits * (D + 2) * 4 : 0);
}

extern "C" int mi355_decode_block(int B, int d, int F, int Hq, int Hkv, int D, const void* h, const void* norm1_w, const void* w_qkv, const void* q_norm_w, const void* k_norm_w,
                                  const float* cos, const float* sin, const int32_t* pos, void* k_cache, void* v_cache, int64_t batch_stride, int64_t ld, int capacity,
                                  const int32_t* write_pos, const int32_t* len_dev, const uint8_t* key_mask, int64_t ldm, const void* w_out, const void* norm2_w,
                                  const void* w_gate_up, const void* w_down, float scale, float eps, int splits, void* scratch, int64_t scratch_bytes, void* out, void* stream) {
    MI355_REQUIRE(B >= 1 && B <= 8 && d > 0 && F > 0 && Hq > 0 && Hkv > 0 && D > 0 && scratch && out && out != h && splits >= 1, "decode_block: bad arguments");
    MI355_REQUIRE(scratch_bytes >= mi355_decode_block_scratch_bytes(B, d, F, Hq, Hkv, D, splits) && ((uintptr_t)scratch & 15) == 0, "decode_block: scratch too small (%lld bytes) or not 16-byte aligned",
                  (long long)scratch_bytes);
    const int64_t nq = (int64_t)(Hq + 2 * Hkv) * D, lq = pad8(nq), nc = (int64_t)Hq * D, lc = pad8(nc), l1 = pad8(d), la = pad8(F);
    bf16_t *qkv = (bf16_t*)scratch, *ctx = qkv + B * lq, *h1 = ctx + B * lc, *act = h1 + B * l1;
    MI355_REQUIRE(lc == nc && norm2_w && w_gate_up && w_down, "decode_block: Hq * D must be a multiple of 8; null pointer");
    if (int rc = mi355_gemv_bf16_pro(B, nq, d, h, d, 1, norm1_w, eps, w_qkv, d, qkv, lq, nullptr, 0, stream)) return rc;
    float* parts = (float*)(act + B * la);
    const bool fold = B == 1 && splits > 1 && nc <= 32768;  // (two rows and more go through the matrix pipe, whose operands have no image to fold into; 64 KiB of LDS)
    if (int rc = attn_decode_qkv(B, Hq, Hkv, D, qkv, lq, q_norm_w, k_norm_w, cos, sin, pos, k_cache, v_cache, batch_stride, ld, capacity, write_pos, len_dev, key_mask, ldm, ctx,
                                 scale, eps, splits, parts, stream, !fold)) return rc;
    if (fold) {
        MI355_REQUIRE(w_out, "decode_block: null pointer");
        gemv_launch<3, OUT_BF16>(1, d, (int)nc, ctx, nc, nullptr, 0.f, w_out, nc, h1, l1, h, d, stream, SplitRow{parts, D, splits});
        MI355_LAUNCH_CHECK("decode_block(out)");
    } else if (int rc = mi355_gemv_bf16(B, d, (int)nc, ctx, nc, w_out, nc, h1, l1, h, d, stream)) return rc;
    gemv_launch<1, OUT_BF16, true>(B, F, d, h1, l1, norm2_w, eps, w_gate_up, d, act, la, nullptr, 0, stream);
    MI355_LAUNCH_CHECK("decode_block(gate, up)");
    return mi355_gemv_bf16(B, d, F, act, la, w_down, F, out, d, h1, l1, stream);
}

extern "C" int mi355_decode_blocks(int layers, const int64_t* table, int B, int d, int F, int Hq, int Hkv, int D, const void* h, const float* cos, const float* sin, const int32_t* pos,
                                   const int32_t* write_pos, const int32_t* len_dev, const uint8_t* key_mask, int64_t ldm, float scale, float eps, int splits, void* scratch,
                                   int64_t scratch_bytes, void* rows_a, void* rows_b, void* stream) {
    MI355_REQUIRE(layers >= 1 && table && rows_a && rows_b && rows_a != rows_b && h != rows_a, "decode_blocks: bad arguments");
    for (int i = 0; i < layers; ++i, table += 13) {
        void* out = i & 1 ? rows_b : rows_a;
        const auto at = [&](int j) { return reinterpret_cast<void*>(static_cast<uintptr_t>(table[j])); };
        MI355_REQUIRE(table[12] > 0 && table[12] <= 0x7fffffff, "decode_blocks: bad capacity");
        if (int rc = mi355_decode_block(B, d, F, Hq, Hkv, D, h, at(0), at(1), at(2), at(3), cos, sin, pos, at(4), at(5), table[10], table[11], (int)table[12], write_pos, len_dev, key_mask, ldm,
                                        at(6), at(7), at(8), at(9), scale, eps, splits, scratch, scratch_bytes, out, stream)) return rc;
        h = out;
    }
    return 0;
}

extern "C" int mi355_decode_advance(int B, const int64_t* next_ids, int64_t* tok, int32_t* rope_pos, int32_t* write_pos, int32_t* length, void* stream) {
    MI355_REQUIRE(B > 0 && next_ids && tok && rope_pos && write_pos && length, "decode_advance: bad arguments");
    decode_advance_kernel<<<(B + 63) / 64, 64, 0, ST(stream)>>>(B, next_ids, tok, rope_pos, write_pos, length);
    MI355_LAUNCH_CHECK("decode_advance");
    return 0;
}

extern "C" int mi355_argmax_rows(int64_t rows, int64_t V, const void* logits, int64_t ld, int64_t* out, void* workspace, void* stream) {
    MI355_REQUIRE(rows > 0 && rows <= 65535 && V > 0 && logits && out && workspace && ld >= V, "argmax_rows: bad arguments (workspace: rows * 64 * 12 bytes)");
    static_assert(ARG_SPLIT == 64, "the merge kernel is one wave");
    float* pv = (float*)workspace;
    int64_t* pi = (int64_t*)((char*)workspace + ((rows * ARG_SPLIT * 4 + 7) / 8) * 8);
    argmax_part_kernel<bf16_t><<<dim3(ARG_SPLIT, (unsigned)rows), 256, 0, ST(stream)>>>(V, (const bf16_t*)logits, ld, pv, pi);
    MI355_LAUNCH_CHECK("argmax_rows(part)");
    argmax_merge_kernel<<<(int)rows, 64, 0, ST(stream)>>>(pv, pi, out);
    MI355_LAUNCH_CHECK("argmax_rows");
    return 0;
}

extern "C" int mi355_argmax_rows_f32(int64_t rows, int64_t V, const float* logits, int64_t ld, int64_t* out, void* workspace, void* stream) {
    MI355_REQUIRE(rows > 0 && rows <= 65535 && V > 0 && logits && out && workspace && ld >= V, "argmax_rows_f32: bad arguments (workspace: rows * 64 * 12 bytes)");
    float* pv = (float*)workspace;
    int64_t* pi = (int64_t*)((char*)workspace + ((rows * ARG_SPLIT * 4 + 7) / 8) * 8);
    argmax_part_kernel<float><<<dim3(ARG_SPLIT, (unsigned)rows), 256, 0, ST(stream)>>>(V, logits, ld, pv, pi);
    MI355_LAUNCH_CHECK("argmax_rows_f32(part)");
    argmax_merge_kernel<<<(int)rows, 64, 0, ST(stream)>>>(pv, pi, out);
    MI355_LAUNCH_CHECK("argmax_rows_f32");
    return 0;
}
