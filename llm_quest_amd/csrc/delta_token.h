// The gated delta rule of a ragged batch token by token: what a workgroup does, for seqrec.hip (steps of single tokens and short portions) and delta_chunk.hip (the short sequences of
// a step whose long ones go in chunks: the same arithmetic, so the same bits).
#pragma once
#include "common.h"
#include "lane_sums.h"

__device__ __forceinline__ float ldr_dt(const void* p, int dt, int64_t i) { return dt == MI355_DT_F32 ? ((const float*)p)[i] : bf2f(((const bf16_t*)p)[i]); }

// Per value head h a state S [dk, dv] (fp32, carried per sequence slot); its query / key head is h / (H / G).  Per token:
//   k^ = k / sqrt(sum k^2 + 1e-6), q^ = q / sqrt(sum q^2 + 1e-6) * qscale   (unit vectors; raw q / k rows come in)
//   beta = sigmoid(b), g = exp(-exp(A_log[h]) * softplus(a + dt_bias[h]))
//   S <- g S;  u = beta (v - S^T k^);  S <- S + k^ u^T;  o = S^T q^
// Column c of S obeys its own recurrence, so columns are spread over lanes and the time loop stays inside: DR_LPR lanes share a column (CPL key
// channels each, in registers), the two dot products of a step close with lane sums -- no LDS, no barrier.  The per-token scalars (g, beta and the two
// unit-vector factors, which multiply the dot products instead of the rows) are prepared once per (token, head) by delta_prep_kernel; the operands of
// step t + 1 are requested before step t's arithmetic.
#define DR_LPR 8
struct DeltaArgs {
    const int *seq_off, *slot;
    const void *q, *k, *v, *b, *a;
    const float *A_log, *dt_bias;
    float *state, *o;
    f32x4* ws;  // [tokens, H]: g, beta, key factor, query factor * qscale
    int64_t ldq, ldk, ldv, ldb, lda;
    int H, G, dk, dv, qk_dt, v_dt, ba_dt;
    float qscale;
};

// the columns col0 .. col0 + 64 / DR_LPR - 1 of head h over the rows t0 .. t1 - 1, one wave; S: that head's state from column c0 on, entry (channel, column) at
// channel * s_ch + (column - c0) * s_col; no block-level synchronisation.  RULE false: linear attention with the decay, key and query factors `fixed` of every token.
template <int CPL, bool VEC, bool RULE = true>
__device__ __forceinline__ void delta_rule_columns(const DeltaArgs& p, int h, int col0, int t0, int t1, float* S, int64_t s_ch, int64_t s_col, int c0 = 0, f32x4 fixed = {}) {
    const int lane = threadIdx.x & 63;
    const int col = col0 + lane / DR_LPR, cg = lane % DR_LPR, ch0 = cg * CPL;
    const bool col_ok = col < p.dv;
    const int hq = h / (p.H / p.G), dk = p.dk;
    float st[CPL];
#pragma unroll
    for (int i = 0; i < CPL; ++i) st[i] = (col_ok && ch0 + i < dk) ? S[(ch0 + i) * s_ch + (col - c0) * s_col] : 0.f;
    struct In {
        float k[CPL], q[CPL];
        f32x4 sc;
        float v;
    };
    auto load_in = [&](In& in, int t) {
        const int64_t ko = (int64_t)t * p.ldk + (int64_t)hq * dk + ch0, qo = (int64_t)t * p.ldq + (int64_t)hq * dk + ch0;
        if (VEC) {
#pragma unroll
            for (int i = 0; i < CPL; i += 4) {
                f32x4 kv = {0.f, 0.f, 0.f, 0.f}, qv = {0.f, 0.f, 0.f, 0.f};
                if (ch0 + i < dk) {
                    kv = *(const f32x4*)((const float*)p.k + ko + i);
                    qv = *(const f32x4*)((const float*)p.q + qo + i);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) in.k[i + e] = kv[e], in.q[i + e] = qv[e];
            }
        } else {
#pragma unroll
            for (int i = 0; i < CPL; ++i) {
                const bool ok = ch0 + i < dk;
                in.k[i] = ok ? ldr_dt(p.k, p.qk_dt, ko + i) : 0.f;
                in.q[i] = ok ? ldr_dt(p.q, p.qk_dt, qo + i) : 0.f;
            }
        }
        in.sc = RULE ? p.ws[(int64_t)t * p.H + h] : fixed;
        in.v = col_ok ? ldr_dt(p.v, p.v_dt, (int64_t)t * p.ldv + (int64_t)h * p.dv + col) : 0.f;
    };
    auto step = [&](const In& in, int t) {
        const float a = in.sc[0], b = in.sc[1], kn = in.sc[2], qn = in.sc[3];
        float u0 = 0.f, u1 = 0.f;
#pragma unroll
        for (int i = 0; i < CPL; i += 2) {
            st[i] *= a;
            st[i + 1] *= a;
            u0 = fmaf(st[i], in.k[i], u0);
            u1 = fmaf(st[i + 1], in.k[i + 1], u1);
        }
        const float u = RULE ? lanes_sum<DR_LPR>(u0 + u1) * kn : 0.f;
        const float c = b * (in.v - u) * kn;
        float o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int i = 0; i < CPL; i += 2) {
            st[i] = fmaf(c, in.k[i], st[i]);
            st[i + 1] = fmaf(c, in.k[i + 1], st[i + 1]);
            o0 = fmaf(st[i], in.q[i], o0);
            o1 = fmaf(st[i + 1], in.q[i + 1], o1);
        }
        const float oo = lanes_sum<DR_LPR>(o0 + o1) * qn;
        if (cg == 0 && col_ok) p.o[(int64_t)t * p.H * p.dv + (int64_t)h * p.dv + col] = oo;
    };
    In inA, inB;
    if (t0 < t1) load_in(inA, t0);
    for (int t = t0; t < t1; t += 2) {
        if (t + 1 < t1) load_in(inB, t + 1);
        step(inA, t);
        if (t + 1 < t1) {
            if (t + 2 < t1) load_in(inA, t + 2);
            step(inB, t + 1);
        }
    }
#pragma unroll
    for (int i = 0; i < CPL; ++i)
        if (col_ok && ch0 + i < dk) S[(ch0 + i) * s_ch + (col - c0) * s_col] = st[i];
}
