// Linear recurrences of served decoders over the new tokens of a ragged batch, in chunks of 64 tokens on the fp32 matrix pipe (gfx950 only), heads of 128 | 128:
// the gated delta rule (unit keys, decay and beta per token) and retention (one decay per head, no correction).  The mathematics of a chunk is that of gdr_chunk.hip;
// here operands are fp32 rows of a packed batch, the state is [dk][dv] per slot, and nothing is kept for a backward pass.
//     delta:      U = R (b V) - Kw S,  O = gam q S + P U,  S <- gam_63 S + (Gp K)^T U
//     retention:  U = V,               the same
// Which sequences of a step go this way is their own number of new tokens' affair (`from`): beside a long prompt, a short one and a single token
// get the bits that they get alone -- of the delta rule inside the scan's launch, whose long chains hide them; of retention by mi355_gla_fwd_below.
// A prompt's tokens through the token-by-token kernels are one dependent chain: six prompts of 900 tokens, 16 heads, 921 us a delta layer and 504 us of retention whatever
// the chip could multiply; the chunks take 318 us and 179 us.  Bound: the scan's chain of chunks (two products behind two barriers each), not the
// pipe.
// Chains of 128 products on the matrix pipe are cut (add16): outputs' distance to 64 bits, token by token | here with whole chains | here: 1.29e-7 | 2.32e-7 | 1.73e-7, decays near zero
// 1.19e-7 | 2.27e-7 | 1.45e-7, nearly parallel keys 1.29e-7 | 2.67e-7 | 1.90e-7, decays near one 4.7e-7 | 5.0e-7 | 4.7e-7, retention 3.1e-7 | 3.0e-7 | 2.6e-7; 6 of the 363 us that the six prompts took.
// A chunk whose U is not finite and all behind it go token by token inside the scan: the triangles' zeros are multiplied, not skipped, and a token's key, value, decay or beta that
// is not finite would reach the rows before it.  (A query reaches its own row alone, a key under retention the rows behind it.)
#include "delta_token.h"
#include "gdr_chunk.h"

#define ST(s) ((hipStream_t)(s))

namespace {

// one chunk of one head in the workspace (floats): Kw [64][128], Uv [64][128] (delta only), P [64][64], then per token gam x query factor, Gp x key factor, and the chunk's decay
constexpr int D_KW = 0, D_U = GC * GD, D_P = 2 * GC * GD, D_G = D_P + GC * GC, D_BLOCK = D_G + 2 * GC + 4;

struct DChunkArgs {
    const int *seq_off, *slot;
    const float *q, *k, *v;
    int64_t ldq, ldk, ldv;
    const f32x4* tok;         // delta: [tokens, H] decay, beta, key factor, query factor
    const float* head_decay;  // retention: [H]
    float qscale, kscale;     // retention
    int H, G, heads;  // heads: of all sequences
    int from;         // sequences with fewer new tokens: retention leaves them alone, the delta rule goes token by token
    int by_tokens;    // where a sequence's chunks lie (chunk_block)
    float *state, *o, *ws;
};

// Chunks are packed: those of sequence s start at seq_off[s] / 64 + s, never less than the chunks of the sequences before it.  Where most sequences are short ones (501 sequences of 564
// tokens: 660 MB for the one that has chunks) at 2 seq_off[s] / 64: a sequence of 64 tokens and more has no more chunks than twice its tokens hold.
__host__ __device__ __forceinline__ bool by_tokens(int64_t tokens, int n_seq, int from) { return from >= GC && tokens * 2 / GC < tokens / GC + n_seq; }
__device__ __forceinline__ float* chunk_block(const DChunkArgs& p, int s, int h, int n) {
    return p.ws + ((int64_t)((p.by_tokens ? p.seq_off[s] * 2 / GC : p.seq_off[s] / GC + s) + n) * p.H + h) * D_BLOCK;
}

template <bool DELTA>
__global__ __launch_bounds__(256, 2) void dchunk_prep_kernel(DChunkArgs p) {
    __shared__ __attribute__((aligned(16))) float Ks[GC][GD + 4];
    __shared__ __attribute__((aligned(16))) float N[DELTA ? GC : 1][GC + 4];
    __shared__ __attribute__((aligned(16))) float T[DELTA ? GC : 1][GC + 4];
    __shared__ double gd[GC];
    __shared__ float be[GC], gam[GC], qf[GC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5;
    const int n = blockIdx.x, h = blockIdx.y, s = blockIdx.z, hq = h / (p.H / p.G), t0 = p.seq_off[s] + n * GC, cnt = min(GC, p.seq_off[s + 1] - t0);
    if (cnt <= 0 || p.seq_off[s + 1] - p.seq_off[s] < p.from) return;
    const float *qp = p.q + (int64_t)t0 * p.ldq + (int64_t)hq * GD, *kp = p.k + (int64_t)t0 * p.ldk + (int64_t)hq * GD, *vp = p.v + (int64_t)t0 * p.ldv + (int64_t)h * GD;
    float* blk = chunk_block(p, s, h, n);
    // Everything is requested before it is needed, one latency for each: keys and their factors, queries in fragment form (tile (ti, tj) of Q K^T), and, once those are used, a column of
    // values: six prompts of 900 tokens, 16 heads, 135 -> 105 us (retention 38 -> 35).  (No conditions: rows beyond the sequence are its last, dropped where they are used.)
    const int ti = wave >> 1, tj = wave & 1, last = cnt - 1;
    f32x4 kr[8], qr[16];
    float kf[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = min((tid >> 5) + 8 * i, last);
        kr[i] = *reinterpret_cast<const f32x4*>(kp + r * p.ldk + (tid & 31) * 4);
        kf[i] = DELTA ? p.tok[((int64_t)t0 + r) * p.H + h][2] : p.kscale;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) qr[i] = *reinterpret_cast<const f32x4*>(qp + min(32 * ti + ln, last) * p.ldq + 8 * i + 4 * hf);
    if (wave == 0) {
        f32x4 c = {1.f, 0.f, 0.f, 0.f};
        if (lane < cnt) {
            if (DELTA) c = p.tok[((int64_t)t0 + lane) * p.H + h];
            else c = f32x4{p.head_decay[h], 1.f, p.kscale, p.qscale};
        }
        const double g = cumulated_log64(decay_at_least(c[0])), g63 = __shfl(g, 63, 64);
        gd[lane] = g;
        be[lane] = c[1];
        gam[lane] = exp_of(g);
        qf[lane] = c[3];
        blk[D_G + lane] = exp_of(g) * c[3];
        blk[D_G + GC + lane] = exp_of(g63 - g) * c[2];
        if (lane == 0) blk[D_G + 2 * GC] = exp_of(g63);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // keys, made unit vectors (resp. scaled) on the way
        const int r = (tid >> 5) + 8 * i;
        *reinterpret_cast<f32x4*>(&Ks[r][(tid & 31) * 4]) = r < cnt ? kr[i] * kf[i] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();
    [[maybe_unused]] float vr[32];
    {  // K K^T and Q K^T: wave = tile (ti, tj); the tile above the diagonal is zero
        f32x16 kk = zero16(), qk = zero16(), kkt = zero16(), qkt = zero16();
        if (wave != 1) {
#pragma unroll
            for (int c = 0; c < GD; c += 8) {
                const f32x4 qv = 32 * ti + ln < cnt ? qr[c / 8] : f32x4{0.f, 0.f, 0.f, 0.f};
                const f32x4 bv = *reinterpret_cast<const f32x4*>(&Ks[32 * tj + ln][c + 4 * hf]);
                const f32x4 av = *reinterpret_cast<const f32x4*>(&Ks[32 * ti + ln][c + 4 * hf]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    qk = mfma2(qv[j], bv[j], qk);
                    if (DELTA) kk = mfma2(av[j], bv[j], kk);
                }
                if ((c & 24) == 24) {
                    add16(qkt, qk);
                    if (DELTA) add16(kkt, kk);
                }
            }
            qk = qkt, kk = kkt;
        }
        if (DELTA) {
#pragma unroll
            for (int i = 0; i < 32; ++i) vr[i] = vp[min(8 * (i >> 2) + 4 * hf + (i & 3), last) * p.ldv + 32 * wave + ln];
        }
        const int j = 32 * tj + ln;
        const double gj = gd[j];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int i = 32 * ti + c_row(e, hf);
            const float D = i >= j ? exp_of(gd[i] - gj) : 0.f;
            if (DELTA) N[i][j] = i > j ? be[i] * kk[e] * D : 0.f;
            blk[D_P + i * GC + j] = i >= j ? qf[i] * qk[e] * D : 0.f;
        }
    }
    if constexpr (DELTA) {
        __syncthreads();
        invert_unit_lower64(N, T);
        // Uv = R (b V), Kw = R (b gam K): wave = 32 columns, both row halves (the upper one ends at token 32)
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
                const float bv = t < cnt ? vr[kb / 2 + j] * be[t] : 0.f, bk = Ks[t][col] * (be[t] * gam[t]);
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
            blk[D_U + r * GD + col] = u0[e];
            blk[D_U + (32 + r) * GD + col] = u1[e];
            blk[D_KW + r * GD + col] = w0[e];
            blk[D_KW + (32 + r) * GD + col] = w1[e];
        }
    }
}

// One workgroup per sequence, head and 32 value columns, chunk by chunk.  Waves 0, 1 take Kw S (row halves), waves 2, 3 q S and then P U; the state's four tiles of 32 key
// channels go one to a wave.  Every operand of a chunk is requested a chunk ahead, by each side for itself: six prompts of 900 tokens, 16 heads, 219 -> 184 us (retention 180 -> 158), one of 2 000
// 266 -> 236 with its prep; in one loop for both sides 230 (registers spill, and waits count every store).
template <bool DELTA>
__global__ __launch_bounds__(256, 2) void dchunk_scan_kernel(DChunkArgs p) {
    __shared__ __attribute__((aligned(16))) float Ss[GV][GD + 4];  // [value column][key channel]
    __shared__ __attribute__((aligned(16))) float Us[GC][GV + 8];
    __shared__ __attribute__((aligned(16))) float Ks[GC][GD + 4];
    __shared__ float gg[2][256];  // gam, Gp and the chunk's decay (a word a thread: a condition would take the request with it, to where it is used)
    __shared__ int lost[2];  // a chunk's flag: set by its U, cleared a chunk later
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 31, hf = lane >> 5, rh = wave & 1;
    // the four value ranges of a head read the same rows: to one XCD (workgroups are dealt to the eight XCDs in turn), side by side
    const int id = blockIdx.x, at = (id >> 5) * 8 + (id & 7), v0 = ((id >> 3) & 3) * GV;
    if (at >= p.heads) return;
    const int h = at % p.H, s = at / p.H, hq = h / (p.H / p.G), s0 = p.seq_off[s], len = p.seq_off[s + 1] - s0, NC = (len + GC - 1) / GC;
    const float *qp = p.q + (int64_t)s0 * p.ldq + (int64_t)hq * GD, *kp = p.k + (int64_t)s0 * p.ldk + (int64_t)hq * GD, *vp = p.v + (int64_t)s0 * p.ldv + (int64_t)h * GD + v0;
    float* state = p.state + ((int64_t)p.slot[s] * p.H + h) * GD * GD + v0;
    if (NC <= 0) return;
    auto by_token = [&](int ta, int tb, float* S, int64_t s_ch, int64_t s_col) {  // S: from this workgroup's first column on
        DeltaArgs d = {};
        d.q = p.q, d.k = p.k, d.v = p.v, d.ldq = p.ldq, d.ldk = p.ldk, d.ldv = p.ldv, d.ws = const_cast<f32x4*>(p.tok), d.o = p.o;
        d.H = p.H, d.G = p.G, d.dk = d.dv = GD, d.qk_dt = d.v_dt = MI355_DT_F32;
        static_assert(GV == 4 * (64 / DR_LPR) && GD == 16 * DR_LPR, "a workgroup's columns and a lane's channels there and here");
        f32x4 fixed = {};
        if (!DELTA) fixed = f32x4{p.head_decay[h], 1.f, p.kscale, p.qscale};
        delta_rule_columns<16, true, DELTA>(d, h, v0 + wave * (64 / DR_LPR), ta, tb, S, s_ch, s_col, v0, fixed);
    };
    if (len < p.from) {
        if (DELTA) by_token(s0, s0 + len, state, GD, 1);
        return;
    }
    const int row = 32 * rh + ln;
    const float* first = chunk_block(p, s, h, 0);
    const int64_t block = (int64_t)p.H * D_BLOCK;
    if (tid < 2) lost[tid] = 0;
    int n = 0;
    // The two sides' waves run loops of their own (the barriers are counted by wave, not by place): in one loop a wait for a chunk's operands cannot be counted over the other side's
    // requests and stores and becomes a wait for all of them, and both sides' registers are live at once.
    auto chunks = [&](auto side) {
        constexpr bool Q = decltype(side)::value;
        // what a chunk reads: a Kw row, or a q row and a P row, in fragment form; keys; U before the state's part; its decays.  (Loads carry no condition: rows beyond the sequence are its
        // last; of queries they give rows that are not written, keys and values are dropped where they are used.)
        f32x4 fr[16], kr[8], pr[8];
        float uv[16], gr;
        auto request = [&](int n) {
            const float* blk = first + n * block;
            const int t0 = n * GC, last = min(GC, len - t0) - 1;
#pragma unroll
            for (int i = 0; i < 8; ++i) kr[i] = *reinterpret_cast<const f32x4*>(kp + t0 * p.ldk + min((tid >> 5) + 8 * i, last) * p.ldk + (tid & 31) * 4);
            gr = blk[D_G + min(tid, 2 * GC)];
            if (Q || DELTA) {
                const float* src = Q ? qp + t0 * p.ldq + min(row, last) * p.ldq + 4 * hf : blk + D_KW + row * GD + 4 * hf;
#pragma unroll
                for (int i = 0; i < 16; ++i) fr[i] = *reinterpret_cast<const f32x4*>(src + 8 * i);
            }
            if (!Q) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int r = 32 * rh + c_row(e, hf);
                    uv[e] = DELTA ? (blk + D_U + v0)[r * GD + ln] : (vp + t0 * p.ldv)[min(r, last) * p.ldv + ln];
                }
            }
        };
        auto request_p = [&](int n) {
#pragma unroll
            for (int i = 0; i < 8; ++i) pr[i] = *reinterpret_cast<const f32x4*>(first + n * block + D_P + row * GC + 4 * hf + 8 * i);
        };
        auto put_out = [&](int t0, int cnt, const f32x16& x) {  // rows beyond the sequence: beyond the buffer, dropped
            auto rs = __builtin_amdgcn_make_buffer_rsrc(p.o + ((int64_t)s0 + t0) * p.H * GD + (int64_t)h * GD + v0, 0, 0x7fffffff, 0x00020000);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = 32 * rh + c_row(e, hf);
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[e]), rs, r < cnt ? (r * p.H * GD + ln) * 4 : -1, 0, 0);
            }
        };
        request(0);
        if (Q) request_p(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {  // (behind the first chunk's requests: one latency for both)
            const int idx = tid + 256 * i, r = idx >> 5, c = idx & 31;
            Ss[c][r] = state[(int64_t)r * GD + c];
        }
        if (Q) {
#pragma unroll
            for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(fr[i])::"memory");  // (landed before the loop, where only its own requests are then waited for)
            put_out(0, 0, zero16());  // (dropped whole: sixteen stores behind P's request from either way in)
        }
        gg[0][tid] = gr;
        for (; n < NC; ++n) {
            const int t0 = n * GC, cnt = min(GC, len - t0);
            const float* g = gg[n & 1];
            __syncthreads();  // the state is whole, the last chunk's keys and U are read
            if (tid == 0) lost[(n + 1) & 1] = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int r = (tid >> 5) + 8 * i;
                *reinterpret_cast<f32x4*>(&Ks[r][(tid & 31) * 4]) = r < cnt ? kr[i] : f32x4{0.f, 0.f, 0.f, 0.f};
            }
            f32x16 acc = zero16(), half = zero16();
            if (DELTA || Q) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const f32x4 c = *reinterpret_cast<const f32x4*>(&Ss[ln][8 * i + 4 * hf]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc = mfma2(fr[i][j], c[j], acc);
                    if (i == 7) add16(half, acc);
                }
            }
            if (!Q) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float v = DELTA || 32 * rh + c_row(e, hf) < cnt ? uv[e] : 0.f;
                    acc[e] = (v - half[e]) - acc[e];
                    Us[32 * rh + c_row(e, hf)][ln] = acc[e];
                }
                if (__any(lost16(acc)) && lane == 0) lost[n & 1] = 1;
            }
            __syncthreads();
            const int gone = lost[n & 1];
            request(min(n + 1, NC - 1));  // (the last chunk's own once more: nothing here hangs on a condition)
            if (Q) {
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[e] = (acc[e] + half[e]) * g[32 * rh + c_row(e, hf)];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (rh == 0 && i >= 4) break;  // P is lower triangular
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc = mfma2(pr[i][j], Us[8 * i + 4 * hf + j][ln], acc);
                }
                request_p(min(n + 1, NC - 1));
                asm volatile("" ::: "memory");  // (the stores behind the requests: waits for those then leave the stores alone)
                put_out(t0, cnt, acc);
            }
            if (gone) break;  // (the same for the whole workgroup)
            f32x16 c;
            const float gC = g[2 * GC];
#pragma unroll
            for (int e = 0; e < 16; ++e) c[e] = gC * Ss[c_row(e, hf)][32 * wave + ln];
#pragma unroll
            for (int kb = 0; kb < GC; kb += 8)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int t = kb + 4 * hf + j;
                    c = mfma2(Us[t][ln] * g[GC + t], Ks[t][32 * wave + ln], c);
                }
#pragma unroll
            for (int e = 0; e < 16; ++e) Ss[c_row(e, hf)][32 * wave + ln] = c[e];  // read by this wave alone since the last barrier
            gg[(n + 1) & 1][tid] = gr;
        }
    };
    if (wave >= 2) chunks(std::true_type{});
    else chunks(std::false_type{});
    if (n < NC) {
        __threadfence();
        __syncthreads();  // what the chunk wrote of its outputs lies below what comes
        by_token(s0 + n * GC, s0 + len, &Ss[0][0], 1, GD + 4);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int idx = tid + 256 * i, r = idx >> 5, c = idx & 31;
        state[(int64_t)r * GD + c] = Ss[c][r];
    }
}

}  // namespace

extern "C" int64_t mi355_delta_chunked_workspace_bytes(int64_t tokens, int n_seq, int H, int from) {
    return tokens > 0 && n_seq > 0 && H > 0 ? (by_tokens(tokens, n_seq, from) ? tokens * 2 / GC : tokens / GC + n_seq) * (int64_t)H * D_BLOCK * 4 : 0;
}

extern "C" int mi355_delta_chunked(int64_t tokens, int n_seq, int max_new, int from, const int* seq_off, const int* slot, int H, int G, const float* q, int64_t ldq, const float* k, int64_t ldk,
                                   const float* v, int64_t ldv, const float* tok, const float* head_decay, float qscale, float kscale, float* state, float* o, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
    MI355_REQUIRE(tokens > 0 && tokens < (1 << 30) && n_seq > 0 && n_seq <= 65535 && (int64_t)n_seq * H <= (1 << 26) && max_new > 0 && seq_off && slot && H > 0 && H <= 65535 && G > 0 && H % G == 0 && q && k && v && state && o && workspace &&
                      (tok != nullptr) != (head_decay != nullptr),
                  "delta_chunked: bad arguments (either a decay per head or four numbers per token and head)");
    MI355_REQUIRE(ldq >= (int64_t)G * GD && ldk >= (int64_t)G * GD && ldv >= (int64_t)H * GD && ldq % 4 == 0 && ldk % 4 == 0, "delta_chunked: rows too short, or query / key pitches no multiple of 4");
    MI355_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)tok | (uintptr_t)workspace) & 15) == 0, "delta_chunked: queries, keys and the workspace must be 16-byte aligned");
    MI355_REQUIRE(workspace_bytes >= mi355_delta_chunked_workspace_bytes(tokens, n_seq, H, from), "delta_chunked: workspace too small (%lld bytes)", (long long)workspace_bytes);
    DChunkArgs p;
    p.seq_off = seq_off, p.slot = slot, p.q = q, p.k = k, p.v = v, p.ldq = ldq, p.ldk = ldk, p.ldv = ldv, p.tok = (const f32x4*)tok, p.head_decay = head_decay;
    p.qscale = qscale, p.kscale = kscale, p.H = H, p.G = G, p.heads = n_seq * H, p.from = from, p.by_tokens = by_tokens(tokens, n_seq, from), p.state = state, p.o = o, p.ws = (float*)workspace;
    const dim3 prep((max_new + GC - 1) / GC, H, n_seq), scan((unsigned)((n_seq * (int64_t)H + 7) / 8 * 32));
    if (tok) {
        dchunk_prep_kernel<true><<<prep, 256, 0, ST(stream)>>>(p);
        MI355_LAUNCH_CHECK("delta_chunked(prep)");
        dchunk_scan_kernel<true><<<scan, 256, 0, ST(stream)>>>(p);
    } else {
        dchunk_prep_kernel<false><<<prep, 256, 0, ST(stream)>>>(p);
        MI355_LAUNCH_CHECK("delta_chunked(prep)");
        dchunk_scan_kernel<false><<<scan, 256, 0, ST(stream)>>>(p);
    }
    MI355_LAUNCH_CHECK("delta_chunked");
    return 0;
}
