// Batched / grouped matrix products with general strides (gfx950 only).
//
//   C[b][m, n] = epi( sum_k A[b][m, k] * B[b][n, k] )        b < batch
//
// A element (m, k) of batch b:  A[b * a_bs + row(m) * lda + k]
// B element (n, k) of batch b:  B[b * b_bs + n * sbn + k * sbk]      (sbk == 1: weight stored [out, in]; sbn == 1: stored [in, out])
// C element (m, n) of batch b:  C[b * c_bs + crow(m) * ldc + n]
//
// Uses: the per-head products of latent attention with the key / value up-projections folded onto the query and the output side;
// the experts of a mixture (batch = expert, a batch's rows given by device-side offsets, A rows gathered through a dispatch list,
// C rows scattered back and scaled by the routing weight); and every linear layer of the true-fp32 mode (fp32 activations,
// weights kept in bf16, exact products, fp32 accumulation in a fixed k order, so a row's result does not depend on which other rows share its tile).
//
// Compute paths:
//   * FMA: 64 x 64 tile, 256 threads, 4 x 4 outputs per thread, k in steps of 16 through LDS (any operand type and stride);
//   * fp32 A, bf16 B stored [out, in] in 16-byte words: an fp32 number as three bf16 numbers, v_mfma_f32_32x32x16_bf16, tile or weight stream;
//   * MFMA (bf16 A and B): the same tile, four waves of 32 x 32 on v_mfma_f32_32x32x8_bf16_1k, k in steps of 32; a 128 x 128 tile on v_mfma_f32_32x32x16_bf16 for
//     weights stored [out, in]; and, for few rows in all groups together, a stream of the weights that deals k to the waves of a workgroup.
#include <type_traits>

#include "common.h"
#include "quad.h"

#define ST(s) ((hipStream_t)(s))

struct BgemmArgs {
    const void* A;
    const void* B;
    void* C;
    int64_t lda, a_bs, sbn, sbk, b_bs, ldc, c_bs;
    int M, N, K;
    const int* grp_offs;     // [batch + 1] or null: rows of batch b are the sorted rows [grp_offs[b], grp_offs[b+1]) (then M is the tile bound)
    const int* a_rows;       // or null: sorted row r reads A row a_rows[r] / a_div
    int a_div;
    const int* c_rows;       // or null: sorted row r writes C row c_rows[r]
    const float* row_scale;  // or null: C row (after c_rows) is multiplied by row_scale[that row]
    const float* bias;       // or null: bias[n] is added to column n before the epilogue
    int epi;                 // 0 none, 1 relu(x)^2, 2 / 3 / 4 gated (see gated_act): B's rows come in blocks of 64 = [32 gate rows | 32 up rows], C has n_out columns
    float limit;
    int n_out;
    int a_dt, b_dt, c_dt;
    bool rows_last;          // row tiles are the grid's slowest index (see row_tile_of)
};

// Gated activations of a feed-forward's [gate | up] product.  2: g = min(gate, limit), u = clamp(up, -limit, limit), g sigmoid(1.702 g) (u + 1).
// 3: gelu_tanh(gate) * up.  4: silu(gate) * up.
__device__ __forceinline__ float gated_act(int epi, float g, float u, float limit) {
    if (epi == 2) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    if (epi == 4) return g / (1.0f + expf(-g)) * u;
    return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
}

__device__ __forceinline__ float ldx(const void* p, int dt, int64_t i) { return dt == MI355_DT_F32 ? ((const float*)p)[i] : bf2f(((const bf16_t*)p)[i]); }

#define BM 64
#define BN 64
#define BK 16

// A workgroup's matrix (or group) and row tile.  With groups M counts all groups' rows, so most of a group's row tiles are empty, and between the groups' first ones they hold those up: row tiles are
// then the slowest index (450 fp32 tokens on 2 of 16 experts, 1 024 -> 1 792, 56 rows an expert in 15 tiles of 64: 46 -> 34 us; on 4 of 64 45 -> 33).  Not where groups have several tiles and the
// weights are more than the caches hold, which every row tile would then read again (3 000 tokens on 16 experts of 2 048 -> 7 168: 643 -> 693 us); nor without groups.  (Of 128 groups of 190 - 400 fp32
// rows, whose empty tiles are most of the launch either way, it is 2 048 -> 256 913 -> 300 us, 1 024 -> 512 600 -> 352, but 512 -> 1 024 471 -> 516.)
__device__ __forceinline__ int batch_of(const BgemmArgs& p) { return p.rows_last ? blockIdx.y : blockIdx.z; }
__device__ __forceinline__ int row_tile_of(const BgemmArgs& p) { return p.rows_last ? blockIdx.z : blockIdx.y; }
static dim3 tile_grid(const BgemmArgs& p, int64_t cols, int64_t rows, int batch) { return p.rows_last ? dim3((unsigned)cols, (unsigned)batch, (unsigned)rows) : dim3((unsigned)cols, (unsigned)rows, (unsigned)batch); }
__global__ __launch_bounds__(256) void bgemm_fma_kernel(BgemmArgs p) {
    __shared__ float As[BK][BM + 4];
    __shared__ float Bs[BK][BN + 4];
    const int b = batch_of(p);
    int row0 = 0, rows = p.M;
    if (p.grp_offs) {
        row0 = p.grp_offs[b];
        rows = p.grp_offs[b + 1] - row0;
    }
    const int m0 = row_tile_of(p) * BM, n0 = blockIdx.x * BN;
    if (m0 >= rows) return;
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    // loader roles: A element (m = tid / 4 + {0}, k = (tid % 4) * 4 .. +4): 64 rows x 16 k
    const int am = tid >> 2, ak = (tid & 3) * 4;
    int64_t a_base = -1;
    if (m0 + am < rows) {
        const int r = row0 + m0 + am;
        const int64_t arow = p.a_rows ? p.a_rows[r] / p.a_div : r;
        a_base = (int64_t)b * p.a_bs + arow * p.lda;
    }
    // B loader: if sbk == 1 the same (n = tid / 4, k chunk) shape as A; if sbn == 1, n runs fastest: (k = tid / 16, n = (tid % 16) * 4 .. +4)
    const bool b_kfast = p.sbk == 1;
    const int bn = b_kfast ? tid >> 2 : (tid & 15) * 4, bk = b_kfast ? (tid & 3) * 4 : tid >> 4;
    const int64_t b_base = (int64_t)b * p.b_bs;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < p.K; k0 += BK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = k0 + ak + i;
            As[ak + i][am] = (a_base >= 0 && k < p.K) ? ldx(p.A, p.a_dt, a_base + k) : 0.f;
        }
        if (b_kfast) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = k0 + bk + i, n = n0 + bn;
                Bs[bk + i][bn] = (n < p.N && k < p.K) ? ldx(p.B, p.b_dt, b_base + (int64_t)n * p.sbn + k) : 0.f;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = k0 + bk, n = n0 + bn + i;
                Bs[bk][bn + i] = (n < p.N && k < p.K) ? ldx(p.B, p.b_dt, b_base + (int64_t)n * p.sbn + (int64_t)k * p.sbk) : 0.f;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; ++k) {
            float a[4], bb[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i], bb[i] = Bs[k][(i >> 1) * 32 + tx * 2 + (i & 1)];  // columns 2 tx, 2 tx + 1 and the same + 32: a gate and its up
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], bb[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= rows) continue;
        const int r = row0 + m;
        const int64_t crow = p.c_rows ? p.c_rows[r] : r;
        const float sc = p.row_scale ? p.row_scale[crow] : 1.0f;
        const int64_t cb = (int64_t)b * p.c_bs + crow * p.ldc;
        if (p.epi >= 2) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int n = (n0 >> 1) + tx * 2 + j;  // gate column n0 + 2 tx + j, up column 32 further
                if (n >= p.n_out) continue;
                const float v = gated_act(p.epi, acc[i][j], acc[i][j + 2], p.limit) * sc;
                if (p.c_dt == MI355_DT_F32) ((float*)p.C)[cb + n] = v;
                else ((bf16_t*)p.C)[cb + n] = f2bf(v);
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + (j >> 1) * 32 + tx * 2 + (j & 1);
            if (n >= p.N) continue;
            float v = acc[i][j] + (p.bias ? p.bias[n] : 0.f);
            if (p.epi == 1) v = v > 0.f ? v * v : 0.f;
            v *= sc;
            if (p.c_dt == MI355_DT_F32) ((float*)p.C)[cb + n] = v;
            else ((bf16_t*)p.C)[cb + n] = f2bf(v);
        }
    }
}

// ---- MFMA path: bf16 A and B.  LDS tiles [64][32 + 8] bf16 (k contiguous; the 16-byte pad keeps the 8-byte fragment reads off one bank group).
// Wave w computes the 32 x 32 block (w / 2, w % 2).  v_mfma_f32_32x32x8_bf16_1k: lane l supplies A[m = l % 32][k = 4 * (l / 32) .. +4] and
// B[n = l % 32][same k]; accumulator register 4 * g + i of lane l is C[m = 8 * g + 4 * (l / 32) + i][n = l % 32].
#define MK 32
#define MPAD 8
__global__ __launch_bounds__(256) void bgemm_mfma_kernel(BgemmArgs p) {
    __shared__ bf16_t As[BM][MK + MPAD];
    __shared__ bf16_t Bs[BN][MK + MPAD];
    const int b = batch_of(p);
    int row0 = 0, rows = p.M;
    if (p.grp_offs) {
        row0 = p.grp_offs[b];
        rows = p.grp_offs[b + 1] - row0;
    }
    const int m0 = row_tile_of(p) * BM, n0 = blockIdx.x * BN;
    if (m0 >= rows) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bf16_t* A = (const bf16_t*)p.A;
    const bf16_t* B = (const bf16_t*)p.B;
    // loaders: 64 rows x 32 k = 2048 elements, 8 per thread: (row = tid / 4, k = (tid % 4) * 8 .. +8)
    const int lr = tid >> 2, lk = (tid & 3) * 8;
    int64_t a_base = -1;
    if (m0 + lr < rows) {
        const int r = row0 + m0 + lr;
        const int64_t arow = p.a_rows ? p.a_rows[r] / p.a_div : r;
        a_base = (int64_t)b * p.a_bs + arow * p.lda;
    }
    const bool b_kfast = p.sbk == 1;
    const int64_t b_base = (int64_t)b * p.b_bs;
    const bool a_vec = (p.lda % 8 == 0) && (p.a_bs % 8 == 0) && (((uintptr_t)p.A & 15) == 0);
    const bool b_vec = b_kfast && (p.sbn % 8 == 0) && (p.b_bs % 8 == 0) && (((uintptr_t)p.B & 15) == 0);
    f32x16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    for (int k0 = 0; k0 < p.K; k0 += MK) {
        // A tile
        if (a_base >= 0 && a_vec && k0 + lk + 8 <= p.K) {
            *(u32x4*)&As[lr][lk] = *(const u32x4*)(A + a_base + k0 + lk);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) As[lr][lk + i] = (a_base >= 0 && k0 + lk + i < p.K) ? A[a_base + k0 + lk + i] : (bf16_t)0;
        }
        // B tile
        if (b_kfast) {
            const int n = n0 + lr;
            if (n < p.N && b_vec && k0 + lk + 8 <= p.K) {
                *(u32x4*)&Bs[lr][lk] = *(const u32x4*)(B + b_base + (int64_t)n * p.sbn + k0 + lk);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) Bs[lr][lk + i] = (n < p.N && k0 + lk + i < p.K) ? B[b_base + (int64_t)n * p.sbn + k0 + lk + i] : (bf16_t)0;
            }
        } else {  // n runs fastest in memory: thread (k = tid / 8, n = (tid % 8) * 8 .. +8)
            const int k = k0 + (tid >> 3), nb = (tid & 7) * 8;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int n = n0 + nb + i;
                Bs[nb + i][tid >> 3] = (n < p.N && k < p.K) ? B[b_base + (int64_t)n * p.sbn + (int64_t)k * p.sbk] : (bf16_t)0;
            }
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < MK; kk += 8) {
            const bf16x4 a = *(const bf16x4*)&As[wm + (lane & 31)][kk + 4 * (lane >> 5)];
            const bf16x4 bb = *(const bf16x4*)&Bs[wn + (lane & 31)][kk + 4 * (lane >> 5)];
            acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, bb, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    const int n = n0 + wn + (lane & 31);
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = m0 + wm + 8 * g + 4 * (lane >> 5) + i;
            if (m >= rows || n >= p.N) continue;
            const int r = row0 + m;
            const int64_t crow = p.c_rows ? p.c_rows[r] : r;
            const float sc = p.row_scale ? p.row_scale[crow] : 1.0f;
            float v = acc[4 * g + i] + (p.bias ? p.bias[n] : 0.f);
            if (p.epi == 1) v = v > 0.f ? v * v : 0.f;
            v *= sc;
            const int64_t ci = (int64_t)b * p.c_bs + crow * p.ldc + n;
            if (p.c_dt == MI355_DT_F32) ((float*)p.C)[ci] = v;
            else ((bf16_t*)p.C)[ci] = f2bf(v);
        }
}

// ---- MFMA path, 128 x 128 tile: four waves of 64 x 64 (2 x 2 blocks of v_mfma_f32_32x32x16_bf16: lane l supplies A[m = l % 32][k = 8 * (l / 32) .. +8] and B[n = l % 32]
// [same k]), k in steps of 64; the next step's operands are fetched into registers while the current step multiplies from LDS (one LDS stage, two barriers per step).
// Four LDS fragment reads feed four MFMAs.
#define TM 128
#define TK 64
// VEC: both operands in 16-byte words (K and every stride a multiple of 8, B stored [out, in]).
template <bool VEC>
__global__ __launch_bounds__(256) void bgemm_mfma128_kernel(BgemmArgs p) {
    __shared__ __attribute__((aligned(16))) bf16_t As[TM][TK + MPAD];
    __shared__ __attribute__((aligned(16))) bf16_t Bs[TM][TK + MPAD];
    const int b = batch_of(p);
    int row0 = 0, rows = p.M;
    if (p.grp_offs) {
        row0 = p.grp_offs[b];
        rows = p.grp_offs[b + 1] - row0;
    }
    const int m0 = row_tile_of(p) * TM, n0 = blockIdx.x * TM;
    if (m0 >= rows) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5;
    const bf16_t* A = (const bf16_t*)p.A;
    const bf16_t* B = (const bf16_t*)p.B;
    const bool b_kfast = p.sbk == 1;
    const int64_t b_base = (int64_t)b * p.b_bs;
    const bool a_vec = (p.lda % 8 == 0) && (p.a_bs % 8 == 0) && (((uintptr_t)p.A & 15) == 0);
    const bool b_vec = b_kfast && (p.sbn % 8 == 0) && (p.b_bs % 8 == 0) && (((uintptr_t)p.B & 15) == 0);
    // loader roles: chunk c = tid + 256 i (i < 4): row c / 8, k offset (c % 8) * 8
    int64_t a_base[4];
    const int lr0 = tid >> 3, lk = (tid & 7) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        a_base[i] = -1;
        if (m0 + lr0 + 32 * i < rows) {
            const int r = row0 + m0 + lr0 + 32 * i;
            const int64_t arow = p.a_rows ? p.a_rows[r] / p.a_div : r;
            a_base[i] = (int64_t)b * p.a_bs + arow * p.lda;
        }
    }
    u32x4 ra[4], rb[4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            u32x4 va = {0u, 0u, 0u, 0u}, vb = {0u, 0u, 0u, 0u};
            if (a_base[i] >= 0) {
                if (VEC) {
                    if (k0 + lk < p.K) va = *(const u32x4*)(A + a_base[i] + k0 + lk);
                } else if (a_vec && k0 + lk + 8 <= p.K) va = *(const u32x4*)(A + a_base[i] + k0 + lk);
                else {
                    bf16_t e[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) e[j] = k0 + lk + j < p.K ? A[a_base[i] + k0 + lk + j] : (bf16_t)0;
                    va = u32x4{(unsigned)e[0] | ((unsigned)e[1] << 16), (unsigned)e[2] | ((unsigned)e[3] << 16), (unsigned)e[4] | ((unsigned)e[5] << 16), (unsigned)e[6] | ((unsigned)e[7] << 16)};
                }
            }
            const int n = n0 + lr0 + 32 * i;
            if (n < p.N) {
                if (VEC) {
                    if (k0 + lk < p.K) vb = *(const u32x4*)(B + b_base + (int64_t)n * p.sbn + k0 + lk);
                } else if (b_vec && k0 + lk + 8 <= p.K) vb = *(const u32x4*)(B + b_base + (int64_t)n * p.sbn + k0 + lk);
                else {
                    bf16_t e[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) e[j] = k0 + lk + j < p.K ? B[b_base + (int64_t)n * p.sbn + (int64_t)(k0 + lk + j) * p.sbk] : (bf16_t)0;
                    vb = u32x4{(unsigned)e[0] | ((unsigned)e[1] << 16), (unsigned)e[2] | ((unsigned)e[3] << 16), (unsigned)e[4] | ((unsigned)e[5] << 16), (unsigned)e[6] | ((unsigned)e[7] << 16)};
                }
            }
            ra[i] = va, rb[i] = vb;
        }
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    fetch(0);
    for (int k0 = 0; k0 < p.K; k0 += TK) {
        __syncthreads();  // the previous step's fragments are read
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *(u32x4*)&As[lr0 + 32 * i][lk] = ra[i];
            *(u32x4*)&Bs[lr0 + 32 * i][lk] = rb[i];
        }
        __syncthreads();
        if (k0 + TK < p.K) fetch(k0 + TK);
#pragma unroll
        for (int kk = 0; kk < TK; kk += 16) {
            const bf16x8 a0 = *(const bf16x8*)&As[wm + ln][kk + 8 * hf], a1 = *(const bf16x8*)&As[wm + 32 + ln][kk + 8 * hf];
            const bf16x8 b0 = *(const bf16x8*)&Bs[wn + ln][kk + 8 * hf], b1 = *(const bf16x8*)&Bs[wn + 32 + ln][kk + 8 * hf];
            acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b1, acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b0, acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b1, acc[1][1], 0, 0, 0);
        }
    }
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + wm + 32 * bi + 8 * g + 4 * hf + i;
                if (m >= rows) continue;
                const int r = row0 + m;
                const int64_t crow = p.c_rows ? p.c_rows[r] : r;
                const float sc = p.row_scale ? p.row_scale[crow] : 1.0f;
                const int64_t cb = (int64_t)b * p.c_bs + crow * p.ldc;
                if (p.epi >= 2) {  // this wave's 64 columns are one [32 gates | 32 ups] block: the lane holds a gate (bj = 0) and its up (bj = 1)
                    const int n = ((n0 + wn) >> 1) + ln;
                    if (n < p.n_out) {
                        const float v = gated_act(p.epi, acc[bi][0][4 * g + i], acc[bi][1][4 * g + i], p.limit) * sc;
                        if (p.c_dt == MI355_DT_F32) ((float*)p.C)[cb + n] = v;
                        else ((bf16_t*)p.C)[cb + n] = f2bf(v);
                    }
                    continue;
                }
#pragma unroll
                for (int bj = 0; bj < 2; ++bj) {
                    const int n = n0 + wn + 32 * bj + ln;
                    if (n >= p.N) continue;
                    float v = acc[bi][bj][4 * g + i] + (p.bias ? p.bias[n] : 0.f);
                    if (p.epi == 1) v = v > 0.f ? v * v : 0.f;
                    v *= sc;
                    if (p.c_dt == MI355_DT_F32) ((float*)p.C)[cb + n] = v;
                    else ((bf16_t*)p.C)[cb + n] = f2bf(v);
                }
            }
}

// ---- MFMA path, 256 x 256 tile: eight waves of 128 x 64 (4 x 2 blocks of v_mfma_f32_32x32x16_bf16), k in steps of 64, operands HBM -> LDS by DMA (16 bytes a lane, rows gathered by
// the lanes' addresses), two stages of 64 KiB: the next step's DMA is in flight while this one multiplies, one barrier a step.  A wave's six LDS fragments feed eight MFMAs (the
// 128 x 128 kernel's four feed four, behind writes through registers: LDS-bound).  The DMA writes lanes in order, so rows of 128 bytes are swizzled on the source address:
// 16-byte word c of row r lies at c ^ ((r >> 1) & 7).  Groups: a group's rows are dealt evenly over its ceil(rows / 256) tiles, blocks of 32 rows beyond a tile's end are
// not multiplied; the grid holds what M sorted rows can need at most and a workgroup finds its tile from the offsets (a grid of row tiles x groups would be
// mostly empty: 114 688 workgroups for 16 groups of 16 384 rows).  Tiles are walked rows first, then columns, then groups, an XCD in one piece: what the tiles of an XCD
// share stays in its L2.  The write-out goes through LDS: a value by value one (a row look-up and a 2-byte store each) cost as much as 2048 k of products.
// 16 384 rows in 16 groups, us, before -> now: 2048 -> 2 x 3584 gated 816 -> 644 (750 TFLOP/s), 3584 -> 2048 402 -> 318; 2 048 rows 165 -> 148, 110 -> 89.  What is left: half of
// the steps' time is not products (one workgroup a CU: fragments are read and DMA waited for behind every barrier), and the gated activation's exponentials run alone (90 us).
// 128 x 256 tiles, three stages of 32 k, two workgroups a CU: 726 and 360 (64-byte rows: twice the requests per byte); turning each column panel's k by some steps: the same.
constexpr int WTM = 256, WTN = 256, WK = 64, WSTAGES = 2, WSTAGE = (WTM + WTN) * WK * 2;
__global__ __launch_bounds__(512, 2) void bgemm_wide_kernel(BgemmArgs p, int batch, int tn) {
    __shared__ __attribute__((aligned(16))) char lds[WSTAGES * WSTAGE + WTM * 8];  // (ONE object: beside others, hipcc waits for every DMA in front of each fragment read)
    int* to_row = (int*)(lds + WSTAGES * WSTAGE);
    float* scale = (float*)(to_row + WTM);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 31, hf = lane >> 5;
    // tiles in all groups; then this workgroup's group, and its tile there
    auto group_tiles = [&](int b) { return b < batch ? ((p.grp_offs ? p.grp_offs[b + 1] - p.grp_offs[b] : p.M) + WTM - 1) / WTM : 0; };
    auto scan = [&](int v) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(v, o, 64);
            if (lane >= o) v += u;
        }
        return v;
    };
    int all = 0;
    for (int b0 = 0; b0 < batch; b0 += 64) all += __shfl(scan(group_tiles(b0 + lane)), 63, 64);
    const int useful = __builtin_amdgcn_readfirstlane(all) * tn;
    auto tile = [&](int id) __attribute__((always_inline)) {
        const int q = useful >> 3, r8 = useful & 7, xcd = id & 7;
        const int at = (xcd < r8 ? xcd * (q + 1) : r8 * (q + 1) + (xcd - r8) * q) + (id >> 3);
        int b = 0, before = 0, mine = 1;
        for (int b0 = 0; b0 < batch; b0 += 64) {
            const int n = group_tiles(b0 + lane), incl = before + scan(n);
            const unsigned long long hit = __ballot(incl * tn > at);
            if (hit) {
                const int l = __ffsll(hit) - 1;
                b = b0 + l;
                mine = __shfl(n, l, 64);
                before = __shfl(incl, l, 64) - mine;
                break;
            }
            before = __shfl(incl, 63, 64);
        }
        b = __builtin_amdgcn_readfirstlane(b);
        mine = __builtin_amdgcn_readfirstlane(mine);
        const int local = at - __builtin_amdgcn_readfirstlane(before) * tn, tm = local % mine, n0 = local / mine * WTN;
        const int row0 = p.grp_offs ? p.grp_offs[b] : 0, rows = p.grp_offs ? p.grp_offs[b + 1] - row0 : p.M;
        const int per = ((rows + mine - 1) / mine + 31) & ~31, m0 = tm * per, cnt = __builtin_amdgcn_readfirstlane(min(per, rows - m0));
        if (cnt <= 0) return;  // (rounding up to 32 rows can leave the last tile without any)
        // this wave's share of a stage: four pieces of A and four of B, eight rows of 128 bytes each (rows beyond the tile: the last one again, their results are not stored)
        const char* src[8];
        auto piece = [&](int i) { return wave * 4 + (i & 3); };
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = piece(i) * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
            if (i < 4) {
                const int ar = row0 + m0 + min(r, cnt - 1);
                src[i] = (const char*)((const bf16_t*)p.A + (int64_t)b * p.a_bs + (int64_t)(p.a_rows ? p.a_rows[ar] / p.a_div : ar) * p.lda + c * 8);
            } else {
                src[i] = (const char*)((const bf16_t*)p.B + (int64_t)b * p.b_bs + (int64_t)min(n0 + r, p.N - 1) * p.sbn + c * 8);
            }
        }
        auto issue = [&](int t, int stage, int lo, int hi) {  // (lo, hi: 0, 4 the A pieces, 4, 8 the B pieces)
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (i >= lo && i < hi)
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + (int64_t)t * (WK * 2)),
                                                 (__attribute__((address_space(3))) void*)(lds + stage * WSTAGE + (i < 4 ? 0 : WTM * WK * 2) + piece(i) * 1024), 16, 0, 0);
        };
        const int wm = (wave >> 2) * 128, wn = (wave & 3) * 64, nt = p.K / WK;
        auto frag = [&](const char* tile, int r, int kk) { return *(const bf16x8*)(tile + r * 128 + (((kk * 2 + hf) ^ ((r >> 1) & 7)) << 4)); };
        auto rows_of_tile = [&]() {  // where the tile's rows go, and what they are multiplied by
            if (tid < cnt) {
                const int r = row0 + m0 + tid, c = p.c_rows ? p.c_rows[r] : r;
                to_row[tid] = c;
                scale[tid] = p.row_scale ? p.row_scale[c] : 1.0f;
            }
        };
        auto run = [&](auto nb) {
            constexpr int NB = decltype(nb)::value;  // blocks of 32 rows
            f32x16 acc[NB ? NB : 1][2];
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
            issue(0, 0, 0, 8);
            rows_of_tile();
            for (int t = 0; t < nt; ++t) {
                // this wave's pieces of the step have landed and its reads of the step before are done -- behind the barrier everyone's
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if constexpr (NB > 0) {
                    const char *sa = lds + (t & 1) * WSTAGE, *sb = sa + WTM * WK * 2;
                    bf16x8 fa[2][NB], fb[2][2];  // the fragments of the next 16 k are requested in front of the products of this one
                    auto read = [&](int kk) {
#pragma unroll
                        for (int j = 0; j < 2; ++j) fb[kk & 1][j] = frag(sb, wn + 32 * j + ln, kk);
#pragma unroll
                        for (int i = 0; i < NB; ++i) fa[kk & 1][i] = frag(sa, wm + 32 * i + ln, kk);
                    };
                    read(0);  // (in front of the DMA's issue, and that in two parts: with all of it first 8192^3 takes 1 020 us instead of 944)
                    if (t + 1 < nt) issue(t + 1, (t + 1) & 1, 0, 4);
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) {
                        if (kk < 3) read(kk + 1);
                        if (kk == 1 && t + 1 < nt) issue(t + 1, (t + 1) & 1, 4, 8);
#pragma unroll
                        for (int i = 0; i < NB; ++i)
#pragma unroll
                            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kk & 1][i], fb[kk & 1][j], acc[i][j], 0, 0, 0);
                    }
                } else if (t + 1 < nt) issue(t + 1, (t + 1) & 1, 0, 8);
            }
            // write-out through the stages' LDS, which nobody reads any more: 64 rows of a wave at a time as fp32, then whole 4-column words of a row to a lane
            __syncthreads();
            float* mine = (float*)(lds + wave * 16384);
            const bool glu = p.epi >= 2;
            const int cols = glu ? 32 : 64, lanes = cols / 4, cq = (lane & (lanes - 1)) * 4, nq = glu ? ((n0 + wn) >> 1) + cq : n0 + wn + cq, n_end = glu ? p.n_out : p.N;
            float bias[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) bias[j] = p.bias && nq + j < n_end ? p.bias[nq + j] : 0.f;
            const bool words = nq + 4 <= n_end && p.ldc % 4 == 0 && p.c_bs % 4 == 0 && ((uintptr_t)p.C & 15) == 0;
#pragma unroll
            for (int h = 0; h < (NB + 1) / 2; ++h) {
#pragma unroll
                for (int i = 0; i < (NB - 2 * h < 2 ? NB - 2 * h : 2); ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) mine[(32 * i + 8 * (e >> 2) + 4 * hf + (e & 3)) * 64 + 32 * j + ln] = acc[2 * h + i][j][e];
                __builtin_amdgcn_wave_barrier();  // (a wave's LDS accesses are in order)
                for (int r = lane / lanes; r < 64; r += 64 / lanes) {
                    const int m = wm + 64 * h + r;
                    if (m >= cnt) break;
                    const float sc = scale[m];
                    const int64_t at = (int64_t)b * p.c_bs + (int64_t)to_row[m] * p.ldc + nq;
                    f32x4 v = *(const f32x4*)(mine + r * 64 + cq);
                    if (glu) {
                        const f32x4 u = *(const f32x4*)(mine + r * 64 + 32 + cq);
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[j] = gated_act(p.epi, v[j], u[j], p.limit) * sc;
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            v[j] += bias[j];
                            if (p.epi == 1) v[j] = v[j] > 0.f ? v[j] * v[j] : 0.f;
                            v[j] *= sc;
                        }
                    }
                    if (words) {
                        if (p.c_dt == MI355_DT_F32) *(f32x4*)((float*)p.C + at) = v;
                        else *(u32x2*)((bf16_t*)p.C + at) = u32x2{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (nq + j < n_end) {
                                if (p.c_dt == MI355_DT_F32) ((float*)p.C)[at + j] = v[j];
                                else ((bf16_t*)p.C)[at + j] = f2bf(v[j]);
                            }
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
        };
        if (cnt - wm > 96) run(std::integral_constant<int, 4>{});
        else if (cnt - wm > 64) run(std::integral_constant<int, 3>{});
        else if (cnt > wm) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 0>{});
    };
    if ((int)blockIdx.x < useful) tile(blockIdx.x);
    for (int id = blockIdx.x + gridDim.x; id < useful; id += gridDim.x) {  // only where M counts the rows of one group, not of all
        __syncthreads();  // the last tile's write-out has left the LDS
        tile(id);
    }
}

#include "bgemm_quad.h"

// ---- fp32 A times bf16 B on the matrix pipe, with the fp32 product's accuracy.  An fp32 number is the sum of three bf16 numbers exactly (its 24 significant bits cut into three
// runs of 8 by truncation: no rounding, no overflow; what is lost lies below 2^-133), a product of two bf16 numbers is exact in fp32, and the accumulator is fp32 -- so three
// products (lo, mid, hi) stand for one fp32 product, and what rounds is the sum, as in an FMA chain.  K is cut into SW runs of 16-steps that are summed one by one and
// then joined in order, in EVERY kernel of this path: a row's bits depend neither on the rows beside it nor on which of the kernels its row count takes.
// Against the FMA kernel (64 x 64 tile, scalar fp32: VALU-bound, and at few rows a chain of uncached 2-byte loads): a fp32 replay of three 150-token prompts and four
// single tokens through four layers with experts 19.9 -> 6.0 ms, its logits' error against 64 bits 4.9e-6 -> 2.1e-6
// (fewer roundings per sum).  An infinite weight may meet a zero part, which would make NaN of an infinity: a result that is not finite is summed again the plain way.
#define SW 8
struct Split8 { u32x4 hi, mid, lo; };
struct FragF32 { f32x4 a, b; };  // eight consecutive k of a row
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned& hi, unsigned& mid, unsigned& lo) {
    const unsigned u0 = __float_as_uint(x0), u1 = __float_as_uint(x1), h0 = u0 & 0xffff0000u, h1 = u1 & 0xffff0000u;
    const bool f0 = (u0 & 0x7f800000u) != 0x7f800000u, f1 = (u1 & 0x7f800000u) != 0x7f800000u;  // infinities and NaN stay whole in `hi` (a NaN keeps a set top bit below)
    const float r0 = f0 ? x0 - __uint_as_float(h0) : 0.f, r1 = f1 ? x1 - __uint_as_float(h1) : 0.f;
    const unsigned m0 = __float_as_uint(r0) & 0xffff0000u, m1 = __float_as_uint(r1) & 0xffff0000u;
    const float s0 = r0 - __uint_as_float(m0), s1 = r1 - __uint_as_float(m1);
    const unsigned n0 = !f0 && (u0 & 0x007fffffu) ? h0 | 0x00400000u : h0, n1 = !f1 && (u1 & 0x007fffffu) ? h1 | 0x00400000u : h1;
    hi = (n0 >> 16) | n1;
    mid = (m0 >> 16) | m1;
    lo = (__float_as_uint(s0) >> 16) | (__float_as_uint(s1) & 0xffff0000u);
}
// the same parts of finite numbers in 11 instructions instead of 25; a part of an infinity or NaN is NaN, and so is every sum it reaches: for kernels that sum those again (`settled`)
__device__ __forceinline__ void split_finite(float x0, float x1, unsigned& hi, unsigned& mid, unsigned& lo) {
    const unsigned u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
    const float r0 = x0 - __uint_as_float(u0 & 0xffff0000u), r1 = x1 - __uint_as_float(u1 & 0xffff0000u);
    const unsigned m0 = __float_as_uint(r0), m1 = __float_as_uint(r1);
    const float s0 = r0 - __uint_as_float(m0 & 0xffff0000u), s1 = r1 - __uint_as_float(m1 & 0xffff0000u);
    hi = __builtin_amdgcn_perm(u1, u0, 0x07060302u);  // the upper halves side by side
    mid = __builtin_amdgcn_perm(m1, m0, 0x07060302u);
    lo = __builtin_amdgcn_perm(__float_as_uint(s1), __float_as_uint(s0), 0x07060302u);
}
__device__ __forceinline__ Split8 split8(const f32x4 a, const f32x4 b) {
    Split8 r;
    unsigned h, m, l;
    split_pair(a[0], a[1], h, m, l); r.hi[0] = h; r.mid[0] = m; r.lo[0] = l;
    split_pair(a[2], a[3], h, m, l); r.hi[1] = h; r.mid[1] = m; r.lo[1] = l;
    split_pair(b[0], b[1], h, m, l); r.hi[2] = h; r.mid[2] = m; r.lo[2] = l;
    split_pair(b[2], b[3], h, m, l); r.hi[3] = h; r.mid[3] = m; r.lo[3] = l;
    return r;
}

__device__ __forceinline__ float settled(const BgemmArgs& p, float v, int b, int r, int n) {  // sorted row r, column n
    if (v - v == 0.f || n >= p.N) return v;
    const float* a = (const float*)p.A + (int64_t)b * p.a_bs + (int64_t)(p.a_rows ? p.a_rows[r] / p.a_div : r) * p.lda;
    const bf16_t* w = (const bf16_t*)p.B + (int64_t)b * p.b_bs + (int64_t)n * p.sbn;
    v = 0.f;
    for (int k = 0; k < p.K; ++k) v = fmaf(a[k], bf2f(w[k]), v);
    return v;
}

// Tile of 64 WM rows x 128 columns, four waves of 32 WM x 64 (2 x 2): k in steps of 32 through two LDS stages that take turns (A as three bf16 planes, split once per tile), one barrier a
// step, operands requested DEPTH steps ahead into registers.  VALU (the split) and matrix pipe are level at WM = 1; WM = 2 halves the split's and B's share where there are rows for it.
// With one stage and requests one step ahead a step was the weights' way from memory: 1.1 - 1.5 us, its products 0.16.  450 fp32 rows, us, before -> now: 2048 -> 1024 74 -> 49, 1024 -> 8256 86 -> 49; 3 000 rows
// 1024 -> 4096 218 -> 115; 900 rows over 16 experts 1792 -> 1024 83 -> 62 (now 40).  The split in front of the last step's products instead of behind them: experts 42 / 57, but 204 registers leave two
// workgroups to a CU (1024 -> 8256: 60); interleaved with the products it spills; eight steps ahead too.
// HALVES = 2: eight waves, for products whose tiles leave CUs idle -- one workgroup then fills a CU where two would have.  The shares of a sum (SW of them, added in order) go to the two groups of four
// waves in turn; the second group hands its share over in LDS, and the first adds both in their order: the same bits.  450 rows, 2048 -> 1024: 47.6 -> 39.9 us.
#define FK 32
template <int WM, int HALVES>
__global__ __launch_bounds__(256 * HALVES, 2 / HALVES) void bgemm_f32_tile_kernel(BgemmArgs p) {
    constexpr int R = 64 * WM, AP = R / 32;  // A: 8 threads per row of 32 fp32, 32 rows per pass; B: 4 threads per row of 32 bf16, 64 rows per pass
    constexpr int DEPTH = WM == 1 ? 4 : 2;   // (sums and running sums of WM = 2 take 128 registers)
    __shared__ __attribute__((aligned(16))) bf16_t Asm[HALVES][2][3][R][FK + MPAD];
    __shared__ __attribute__((aligned(16))) bf16_t Bsm[HALVES][2][128][FK + MPAD];
    __shared__ __attribute__((aligned(16))) f32x4 swap[HALVES > 1 ? 256 * WM * 8 : 1];
    const int b = batch_of(p);
    int row0 = 0, rows = p.M;
    if (p.grp_offs) {
        row0 = p.grp_offs[b];
        rows = p.grp_offs[b + 1] - row0;
    }
    const int m0 = row_tile_of(p) * R, n0 = blockIdx.x * 128;
    if (m0 >= rows) return;
    const int half = HALVES > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, ln = lane & 31, hf = lane >> 5;
    bf16_t(&As)[2][3][R][FK + MPAD] = Asm[half];
    bf16_t(&Bs)[2][128][FK + MPAD] = Bsm[half];
    const float* a_row[AP];  // rows and columns beyond the end: the last one again, their results are not stored
    const int ar = tid >> 3, ak = (tid & 7) * 4, br = tid >> 2, bk = (tid & 3) * 8;
#pragma unroll
    for (int i = 0; i < AP; ++i) {
        const int r = row0 + min(m0 + ar + 32 * i, rows - 1);
        a_row[i] = (const float*)p.A + (int64_t)b * p.a_bs + (int64_t)(p.a_rows ? p.a_rows[r] / p.a_div : r) * p.lda;
    }
    const bf16_t* b_row[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) b_row[i] = (const bf16_t*)p.B + (int64_t)b * p.b_bs + (int64_t)min(n0 + br + 64 * i, p.N - 1) * p.sbn;
    f32x4 ra[DEPTH][AP];
    u32x4 rb[DEPTH][2];
    auto fetch = [&](f32x4 (&x)[AP], u32x4 (&w)[2], int k0) {  // K is a multiple of 8: a 16-byte word lies inside or outside as a whole; outside: the row's first one, replaced by zeros below
        int ka = k0 + ak, kb = k0 + bk;
        if (k0 + FK > p.K) ka = ka < p.K ? ka : 0, kb = kb < p.K ? kb : 0;
#pragma unroll
        for (int i = 0; i < AP; ++i) x[i] = *(const f32x4*)(a_row[i] + ka);
#pragma unroll
        for (int i = 0; i < 2; ++i) w[i] = *(const u32x4*)(b_row[i] + kb);
    };
    f32x16 acc[WM][2], tot[WM][2];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = tot[i][j][e] = 0.f;
    const int steps = (p.K + 15) / 16, per = (steps + SW - 1) / SW;
    int left = per;
    const int wm = (wave >> 1) * 32 * WM, wn = (wave & 1) * 64;
    auto stage = [&](f32x4 (&x)[AP], u32x4 (&w)[2], int k0, int st) {
        if (k0 + FK > p.K) {
            if (k0 + ak >= p.K)
#pragma unroll
                for (int i = 0; i < AP; ++i) x[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
            if (k0 + bk >= p.K) w[0] = w[1] = (u32x4){0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < AP; ++i) {
            u32x2 h, m, l;
            unsigned hi, mid, lo;
            split_finite(x[i][0], x[i][1], hi, mid, lo); h[0] = hi; m[0] = mid; l[0] = lo;
            split_finite(x[i][2], x[i][3], hi, mid, lo); h[1] = hi; m[1] = mid; l[1] = lo;
            *(u32x2*)&As[st][0][ar + 32 * i][ak] = h;
            *(u32x2*)&As[st][1][ar + 32 * i][ak] = m;
            *(u32x2*)&As[st][2][ar + 32 * i][ak] = l;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) *(u32x4*)&Bs[st][br + 64 * i][bk] = w[i];
    };
    auto step = [&](f32x4 (&x)[AP], u32x4 (&w)[2], int k0, int st, int next, int end) {
        stage(x, w, k0, st);
        __builtin_amdgcn_sched_barrier(0);
        fetch(x, w, next);
        // this wave's rows of the step are written, and its reads of the stage (two steps ago) are done -- behind the barrier everyone's; requests stay under way
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < FK; kk += 16) {
            if (k0 + kk < end) {
                bf16x8 bf[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) bf[j] = *(const bf16x8*)&Bs[st][wn + 32 * j + ln][kk + 8 * hf];
#pragma unroll
                for (int s = 2; s >= 0; --s)
#pragma unroll
                    for (int i = 0; i < WM; ++i) {
                        const bf16x8 af = *(const bf16x8*)&As[st][s][wm + 32 * i + ln][kk + 8 * hf];
#pragma unroll
                        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf[j], acc[i][j], 0, 0, 0);
                    }
                if (HALVES == 1 && --left == 0) {
                    left = per;
#pragma unroll
                    for (int i = 0; i < WM; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
#pragma unroll
                            for (int e = 0; e < 16; ++e) {
                                tot[i][j][e] += acc[i][j][e];
                                acc[i][j][e] = 0.f;
                            }
                }
            }
        }
    };
    if constexpr (HALVES == 1) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) fetch(ra[d], rb[d], d * FK);
        for (int k0 = 0; k0 < p.K; k0 += DEPTH * FK)  // (steps past K: zeros written, nothing multiplied)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) step(ra[d], rb[d], k0 + d * FK, d & 1, k0 + (d + DEPTH) * FK, p.K);
    } else {
        const int in_share = (per + 1) / 2, all = SW / 2 * in_share;  // steps of FK; a share that is no whole number of them ends within its last
        auto share_at = [&](int share) { return (2 * share + half) * per * 16; };
        int fs = 0, fp = 0;  // the next step to request: share, place in it
        auto requested = [&]() {
            const int at = share_at(fs) + fp * FK;
            if (++fp == in_share) fp = 0, ++fs;
            return min(at, p.K);  // (from K on: nothing is read beyond the rows' first words)
        };
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) fetch(ra[d], rb[d], requested());
        int share = 0, place = 0;
        for (int t = 0; t < all; t += DEPTH)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                if (t + d >= all) break;  // (the same for the whole workgroup)
                const int begin = share_at(share);
                step(ra[d], rb[d], min(begin + place * FK, p.K), d & 1, requested(), min(p.K, begin + per * 16));
                if (++place < in_share) continue;
                if (half == 1) {
#pragma unroll
                    for (int i = 0; i < WM * 8; ++i) swap[i * 256 + tid] = f32x4{acc[i / 8][i / 4 % 2][4 * (i % 4)], acc[i / 8][i / 4 % 2][4 * (i % 4) + 1], acc[i / 8][i / 4 % 2][4 * (i % 4) + 2], acc[i / 8][i / 4 % 2][4 * (i % 4) + 3]};
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (as in a step: requests stay under way)
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                const bool first = 2 * share * per * 16 < p.K, second = (2 * share + 1) * per * 16 < p.K;  // a share beyond K is none
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            if (half == 0) {
                                const f32x4 x = swap[((i * 2 + j) * 4 + g) * 256 + tid];
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    float v = tot[i][j][4 * g + e];
                                    v = first ? v + acc[i][j][4 * g + e] : v;
                                    tot[i][j][4 * g + e] = second ? v + x[e] : v;
                                }
                            }
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[i][j][4 * g + e] = 0.f;
                        }
                place = 0, ++share;
            }
        if (half == 1) return;
    }
    if (HALVES == 1 && left != per) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) tot[i][j][e] += acc[i][j][e];
    }
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) z = fmaf(tot[i][j][e], 0.f, z);
    if (__any(z != z)) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * hf + (e & 3);
                if (m < rows) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) tot[i][j][e] = settled(p, tot[i][j][e], b, row0 + m, n0 + wn + 32 * j + ln);
                }
            }
    }
#pragma unroll
    for (int bi = 0; bi < WM; ++bi)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + wm + 32 * bi + 8 * g + 4 * hf + i;
                if (m >= rows) continue;
                const int r = row0 + m;
                const int64_t crow = p.c_rows ? p.c_rows[r] : r;
                const float sc = p.row_scale ? p.row_scale[crow] : 1.0f;
                const int64_t cb = (int64_t)b * p.c_bs + crow * p.ldc;
                if (p.epi >= 2) {  // this wave's 64 columns are one [32 gates | 32 ups] block
                    const int n = ((n0 + wn) >> 1) + ln;
                    if (n < p.n_out) {
                        const float v = gated_act(p.epi, tot[bi][0][4 * g + i], tot[bi][1][4 * g + i], p.limit) * sc;
                        if (p.c_dt == MI355_DT_F32) ((float*)p.C)[cb + n] = v;
                        else ((bf16_t*)p.C)[cb + n] = f2bf(v);
                    }
                    continue;
                }
#pragma unroll
                for (int bj = 0; bj < 2; ++bj) {
                    const int n = n0 + wn + 32 * bj + ln;
                    if (n >= p.N) continue;
                    float v = tot[bi][bj][4 * g + i] + (p.bias ? p.bias[n] : 0.f);
                    if (p.epi == 1) v = v > 0.f ? v * v : 0.f;
                    v *= sc;
                    if (p.c_dt == MI355_DT_F32) ((float*)p.C)[cb + n] = v;
                    else ((bf16_t*)p.C)[cb + n] = f2bf(v);
                }
            }
}

// ---- MFMA path for few rows per group (one-token steps through a mixture's experts): bound by the stream of the weights.  A workgroup is eight waves on 32 rows x 32
// columns (GLU: the 32 gate and the 32 up columns of one block); the waves deal the k range among themselves, read both operands straight from memory in
// fragment form -- 16 bytes per lane, two stages of SU steps of 16 in flight -- and their partial sums meet in LDS.  A workgroup lives for a few memory round trips, so what
// depends on nothing goes first: the weights in front of the row list that says which operand rows meet them, and where the results go is looked up under the stream.
// (One stage held the other up: its registers were copied, and so waited for, before the next was requested: six rows of 16 experts, 1024 x 1792 gated 13.3 -> 11.0 us,
// 896 x 1024 9.0 -> 8.4; 24 rows 26.7 -> 21.2, 18.1 -> 16.3.  Eight steps a stage: 8.9 and 17.8.)
#define SU 4
#define F32_STREAM_ROWS 128  // fp32 A: beyond this many rows the tile kernel's one split per 128 columns beats the stream's one per 32 (450 rows: a third of the time)
#define STREAM_ROWS 256  // up to this many sorted rows in all groups together
// F32: A is fp32, split into three bf16 fragments in registers (see above: the waves' k runs are that path's runs).
template <bool GLU, bool F32>
__global__ __launch_bounds__(64 * SW) void bgemm_stream_kernel(BgemmArgs p) {
    constexpr int NB = GLU ? 2 : 1;
    using elem_t = std::conditional_t<F32, float, bf16_t>;
    using frag_t = std::conditional_t<F32, FragF32, u32x4>;
    __shared__ float red[SW][NB][16][64];
    const int b = batch_of(p), row0 = p.grp_offs ? p.grp_offs[b] : 0, rows = p.grp_offs ? p.grp_offs[b + 1] - row0 : p.M;
    const int m0 = row_tile_of(p) * 32, n0 = blockIdx.x * 32 * NB;
    if (m0 >= rows) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 31, hf = lane >> 5;
    const int steps = (p.K + 15) / 16, per = (steps + SW - 1) / SW, s0 = min(wave * per, steps), s1 = min(s0 + per, steps);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    struct Stage {
        frag_t a[SU];
        u32x4 b[SU][NB];
    };
    Stage x, y;
    const bf16_t* b_row[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) b_row[j] = (const bf16_t*)p.B + (int64_t)b * p.b_bs + (int64_t)min(n0 + 32 * j + ln, p.N - 1) * p.sbn + 8 * hf;  // (columns past N are not stored)
    auto request_b = [&](Stage& t, int st) {
        if (st + SU <= s1 && (st + SU) * 16 <= p.K) {
#pragma unroll
            for (int u = 0; u < SU; ++u)
#pragma unroll
                for (int j = 0; j < NB; ++j) t.b[u][j] = *(const u32x4*)(b_row[j] + (st + u) * 16);
        } else {
#pragma unroll
            for (int u = 0; u < SU; ++u) {
                const bool in = st + u < s1 && (st + u) * 16 + 8 * hf < p.K;  // K is a multiple of 8
#pragma unroll
                for (int j = 0; j < NB; ++j) t.b[u][j] = in ? *(const u32x4*)(b_row[j] + (st + u) * 16) : zero;
            }
        }
    };
    request_b(x, s0);
    const elem_t* a_row = nullptr;
    if (m0 + ln < rows) {
        const int r = row0 + m0 + ln;
        a_row = (const elem_t*)p.A + (int64_t)b * p.a_bs + (int64_t)(p.a_rows ? p.a_rows[r] / p.a_div : r) * p.lda;
    }
    auto request_a = [&](Stage& t, int st) {
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            const int k = (st + u) * 16 + 8 * hf;
            const bool in = a_row && st + u < s1 && k < p.K;
            if constexpr (F32) {
                t.a[u].a = in ? *(const f32x4*)(a_row + k) : (f32x4){0.f, 0.f, 0.f, 0.f};
                t.a[u].b = in ? *(const f32x4*)(a_row + k + 4) : (f32x4){0.f, 0.f, 0.f, 0.f};
            } else {
                t.a[u] = in ? *(const u32x4*)(a_row + k) : zero;
            }
        }
    };
    request_a(x, s0);
    // this thread's results: rows m0 + 8 (e >> 2) + 4 hf + (e & 3), e = wave * 16 / SW + q
    int64_t crow[16 / SW];
    float scale[16 / SW];
#pragma unroll
    for (int q = 0; q < 16 / SW; ++q) {
        const int e = wave * (16 / SW) + q, r = row0 + min(m0 + 8 * (e >> 2) + 4 * hf + (e & 3), rows - 1);
        crow[q] = p.c_rows ? p.c_rows[r] : r;
    }
    f32x16 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
    auto work = [&](Stage& now, Stage& next, int st) {
        if (st + SU < s1) {
            request_b(next, st + SU);
            request_a(next, st + SU);
        }
#pragma unroll
        for (int u = 0; u < SU; ++u) {
            if constexpr (F32) {
                const Split8 t = split8(now.a[u].a, now.a[u].b);
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const bf16x8 w = __builtin_bit_cast(bf16x8, now.b[u][j]);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, t.lo), w, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, t.mid), w, acc[j], 0, 0, 0);
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, t.hi), w, acc[j], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int j = 0; j < NB; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, now.a[u]), __builtin_bit_cast(bf16x8, now.b[u][j]), acc[j], 0, 0, 0);
            }
        }
    };
    for (int st = s0; st < s1; st += 2 * SU) {
        work(x, y, st);
        if (st + SU < s1) work(y, x, st + SU);
    }
#pragma unroll
    for (int q = 0; q < 16 / SW; ++q) scale[q] = p.row_scale ? p.row_scale[crow[q]] : 1.0f;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) red[wave][j][e][lane] = acc[j][e];
    __syncthreads();
    const int n = n0 / NB + ln;
#pragma unroll
    for (int q = 0; q < 16 / SW; ++q) {
        const int e = wave * (16 / SW) + q, m = m0 + 8 * (e >> 2) + 4 * hf + (e & 3);
        float v[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            v[j] = 0.f;
#pragma unroll
            for (int w = 0; w < SW; ++w) v[j] += red[w][j][e][lane];
        }
        if (m >= rows || n >= (GLU ? p.n_out : p.N)) continue;
        if constexpr (F32) {
#pragma unroll
            for (int j = 0; j < NB; ++j) v[j] = settled(p, v[j], b, row0 + m, n0 + 32 * j + ln);
        }
        float o;
        if constexpr (GLU) {
            o = gated_act(p.epi, v[0], v[NB - 1], p.limit);
        } else {
            o = v[0] + (p.bias ? p.bias[n] : 0.f);
            if (p.epi == 1) o = o > 0.f ? o * o : 0.f;
        }
        o *= scale[q];
        const int64_t ci = (int64_t)b * p.c_bs + crow[q] * p.ldc + n;
        if (p.c_dt == MI355_DT_F32) ((float*)p.C)[ci] = o;
        else ((bf16_t*)p.C)[ci] = f2bf(o);
    }
}

// The same product of fp32 rows where few rows meet the weights: in the kernel above every wave splits its operand fragments in registers, for 32 rows whether they exist or not
// (90 vector instructions a step of 16: 12 us of a 2048 x 1024 product of three rows).  Here the workgroup splits the rows that exist once, into three bf16 planes in LDS, under the
// weights' flight; a lane without a row reads a row of zeros.  The same parts meet the same weights in the same order: the bits are those of the other kernels of this path.
// Three rows, K x N: 2048 x 1024 12.4 -> 6.7 us, 1024 x 4096 9.2 -> 6.1, 1024 x 8256 16.5 -> 8.7, 1024 x 32000 32.9 -> 17.1 (the kernel above as it is now: 11.8, 8.4, 14.4, 28.5); one row
// 1024 x 512 7.7 -> 4.6; 32 rows 1024 x 1024 10.1 -> 9.4 (the kernel above: 9.4); six rows of 16 experts 1792 x 1024 13.1 -> 10.5 (above: 11.9).  Gated epilogues stay above: two
// accumulators want the registers of the second stage (six rows of 16 experts, 1024 x 1792: 12.7 here, 11.0 there).
// Columns a workgroup: 32 is what a product of the matrix pipe holds; fewer idle its lanes, and pay while the workgroups with work leave CUs without any.  8 / 16 / 32 columns, by tiles
// of 32: 16 tiles 4.6 / 4.9 / 5.2 us, 32 tiles 6.7 / 7.3 / 8.3; 128 tiles 7.1 / 6.0 / 6.3; 192 tiles with 1792 deep 12.3 / 10.5 / 12.0, 896 deep 9.4 / 7.3 / 6.4; 258 tiles 13.2 / 10.1 / 8.8.
#define F32_ROWS_LDS (144 * 1024)
#define F32_ROWS_HALF 192
static inline int64_t f32_rows_pitch(int64_t K) { return (K + 15) / 16 * 16 + 8; }  // (8: rows start in different banks)
template <int COLS>
__global__ __launch_bounds__(64 * SW) void bgemm_f32_rows_kernel(BgemmArgs p, int cap, int pitch) {
    constexpr int RU = 8;  // steps of a stage: two stages hold a wave's run up to K = 2048
    extern __shared__ __attribute__((aligned(16))) char smem[];  // planes [3][cap + 1][pitch]; then the waves' sums [SW][16][64]
    bf16_t* planes = (bf16_t*)smem;
    float* red = (float*)smem;
    const int b = blockIdx.z, row0 = p.grp_offs ? p.grp_offs[b] : 0, rows = p.grp_offs ? min(p.grp_offs[b + 1] - row0, cap) : p.M;
    const int n0 = blockIdx.x * COLS;
    if (rows <= 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 31, hf = lane >> 5;
    const int steps = (p.K + 15) / 16, per = (steps + SW - 1) / SW, s0 = min(wave * per, steps), s1 = min(s0 + per, steps);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    u32x4 x[RU], y[RU];
    const bf16_t* b_row = (const bf16_t*)p.B + (int64_t)b * p.b_bs + (int64_t)min(n0 + ln, p.N - 1) * p.sbn + 8 * hf;  // (columns past N are not stored)
    auto request = [&](u32x4 (&t)[RU], int st) {
        if (COLS < 32 && ln >= COLS) return;
        if (st + RU <= s1 && (st + RU) * 16 <= p.K) {
#pragma unroll
            for (int u = 0; u < RU; ++u) t[u] = *(const u32x4*)(b_row + (st + u) * 16);
        } else {
#pragma unroll
            for (int u = 0; u < RU; ++u) {
                const bool in = st + u < s1 && (st + u) * 16 + 8 * hf < p.K;  // K is a multiple of 8
                t[u] = in ? *(const u32x4*)(b_row + (st + u) * 16) : zero;
            }
        }
    };
    if constexpr (COLS < 32) {
#pragma unroll
        for (int u = 0; u < RU; ++u) x[u] = y[u] = zero;
    }
    request(x, s0);
    if (s0 + RU < s1) request(y, s0 + RU);
    const int words = (pitch - 8) / 8, plane = (cap + 1) * pitch;  // 8 k at a time
    for (int c = tid; c < (rows + 1) * words; c += 64 * SW) {
        const int i = c / words, k = (c - i * words) * 8;
        Split8 t = {zero, zero, zero};
        if (i < rows && k < p.K) {
            const int r = row0 + i;
            const float* a = (const float*)p.A + (int64_t)b * p.a_bs + (int64_t)(p.a_rows ? p.a_rows[r] / p.a_div : r) * p.lda + k;
            t = split8(*(const f32x4*)a, *(const f32x4*)(a + 4));
        }
        bf16_t* to = planes + i * pitch + k;  // (row `rows` is the row of zeros)
        *(u32x4*)to = t.hi;
        *(u32x4*)(to + plane) = t.mid;
        *(u32x4*)(to + 2 * plane) = t.lo;
    }
    int64_t crow[16 / SW];
#pragma unroll
    for (int q = 0; q < 16 / SW; ++q) {
        const int e = wave * (16 / SW) + q, r = row0 + min(8 * (e >> 2) + 4 * hf + (e & 3), rows - 1);
        crow[q] = p.c_rows ? p.c_rows[r] : r;
    }
    __syncthreads();
    const bf16_t* a_row = planes + min(ln, rows) * pitch + 8 * hf;
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
    auto work = [&](u32x4 (&t)[RU], int st) {
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            if (st + u >= s1) break;
            const bf16x8 hi = *(const bf16x8*)(a_row + (st + u) * 16), mid = *(const bf16x8*)(a_row + plane + (st + u) * 16), lo = *(const bf16x8*)(a_row + 2 * plane + (st + u) * 16);
            const bf16x8 w = __builtin_bit_cast(bf16x8, t[u]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, w, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mid, w, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, w, acc, 0, 0, 0);
        }
        if (st + 2 * RU < s1) request(t, st + 2 * RU);
    };
    for (int st = s0; st < s1; st += 2 * RU) {
        work(x, st);
        if (st + RU < s1) work(y, st + RU);
    }
    float scale[16 / SW];
#pragma unroll
    for (int q = 0; q < 16 / SW; ++q) scale[q] = p.row_scale ? p.row_scale[crow[q]] : 1.0f;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 16; ++e) red[(wave * 16 + e) * 64 + lane] = acc[e];
    __syncthreads();
    const int n = n0 + ln;
#pragma unroll
    for (int q = 0; q < 16 / SW; ++q) {
        const int e = wave * (16 / SW) + q, m = 8 * (e >> 2) + 4 * hf + (e & 3);
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < SW; ++w) v += red[(w * 16 + e) * 64 + lane];
        if (m >= rows || ln >= COLS || n >= p.N) continue;
        float o = settled(p, v, b, row0 + m, n) + (p.bias ? p.bias[n] : 0.f);
        if (p.epi == 1) o = o > 0.f ? o * o : 0.f;
        o *= scale[q];
        const int64_t ci = (int64_t)b * p.c_bs + crow[q] * p.ldc + n;
        if (p.c_dt == MI355_DT_F32) ((float*)p.C)[ci] = o;
        else ((bf16_t*)p.C)[ci] = f2bf(o);
    }
}

extern "C" __attribute__((visibility("hidden"))) void mi355_gemv_bias_part(int M, int64_t N, int K, const void* x, int64_t ldx, const void* W, int64_t ldw, void* y, int64_t ldy, const float* bias, void* stream);

extern "C" int mi355_bgemm(int batch, int M, int N, int K, const void* A, int a_dt, int64_t lda, int64_t a_bs, const void* B, int b_dt, int64_t sbn, int64_t sbk,
                           int64_t b_bs, void* C, int c_dt, int64_t ldc, int64_t c_bs, const int* grp_offs, const int* a_rows, int a_div, const int* c_rows,
                           const float* row_scale, int epi, int use_mfma, const float* bias, float limit, int n_out, void* stream) {
    MI355_REQUIRE(batch > 0 && batch <= 65535 && M > 0 && N > 0 && K > 0 && A && B && C, "bgemm: bad arguments");
    MI355_REQUIRE((a_dt == MI355_DT_BF16 || a_dt == MI355_DT_F32) && (b_dt == MI355_DT_BF16 || b_dt == MI355_DT_F32) && (c_dt == MI355_DT_BF16 || c_dt == MI355_DT_F32),
                  "bgemm: bad dtype");
    MI355_REQUIRE(epi >= 0 && epi <= 4, "bgemm: bad epilogue");
    MI355_REQUIRE(epi < 2 || (N % 64 == 0 && n_out > 0 && n_out <= N / 2 && !bias), "bgemm: a gated epilogue takes B rows in [32 gate | 32 up] blocks (N a multiple of 64), n_out <= N / 2 columns, no bias");
    MI355_REQUIRE(!a_rows || a_div >= 1, "bgemm: gathered rows need a divisor >= 1");
    MI355_REQUIRE(sbn >= 1 && sbk >= 1 && (sbn == 1 || sbk == 1), "bgemm: one of B's strides must be 1");
    MI355_REQUIRE(!use_mfma || (a_dt == MI355_DT_BF16 && b_dt == MI355_DT_BF16), "bgemm: the MFMA path takes bf16 operands");
    BgemmArgs p;
    p.A = A, p.B = B, p.C = C;
    p.lda = lda, p.a_bs = a_bs, p.sbn = sbn, p.sbk = sbk, p.b_bs = b_bs, p.ldc = ldc, p.c_bs = c_bs;
    p.M = M, p.N = N, p.K = K;
    p.grp_offs = grp_offs, p.a_rows = a_rows, p.a_div = a_rows ? a_div : 1, p.c_rows = c_rows, p.row_scale = row_scale;
    p.bias = bias;
    p.limit = limit, p.n_out = n_out;
    p.epi = epi, p.a_dt = a_dt, p.b_dt = b_dt, p.c_dt = c_dt;
    p.rows_last = grp_offs && (M <= 64 * (int64_t)batch || (int64_t)batch * N * K <= 64 << 20);
    const bool vec = sbk == 1 && K % 8 == 0 && lda % 8 == 0 && a_bs % 8 == 0 && sbn % 8 == 0 && b_bs % 8 == 0 && ((uintptr_t)A & 15) == 0 && ((uintptr_t)B & 15) == 0;
    // one to eight rows with a bias: the weight streams of decode.hip (1024 x 1024, six rows, 24.4 -> 3.8 us; 128-column tiles leave all but eight CUs idle)
    if (use_mfma && batch == 1 && M <= 8 && bias && c_dt == MI355_DT_BF16 && vec && epi == 0 && !grp_offs && !a_rows && !c_rows && !row_scale) {
        mi355_gemv_bias_part(M, N, K, A, lda, B, sbn, C, ldc, bias, stream);
        MI355_LAUNCH_CHECK("bgemm(few rows)");
        return 0;
    }
    if (use_mfma && grp_offs && M <= STREAM_ROWS && K >= 256 && vec) {
        const dim3 grid = tile_grid(p, (N + (epi >= 2 ? 63 : 31)) / (epi >= 2 ? 64 : 32), (M + 31) / 32, batch);
        if (epi >= 2) bgemm_stream_kernel<true, false><<<grid, 64 * SW, 0, ST(stream)>>>(p);
        else bgemm_stream_kernel<false, false><<<grid, 64 * SW, 0, ST(stream)>>>(p);
        MI355_LAUNCH_CHECK("bgemm(stream)");
        return 0;
    }
    if (use_mfma && ((sbk == 1 && N >= 128 && K >= 64) || epi >= 2)) {  // (a gated epilogue needs a gate and its up in one lane: this kernel's 64 columns per wave)  // the large tile: weights stored [out, in], enough columns to fill it
        const int64_t wide_tn = (N + WTN - 1) / WTN, wide_tiles = (grp_offs ? (int64_t)M / WTM + batch : batch * (((int64_t)M + WTM - 1) / WTM)) * wide_tn;
        // where the line lies, us, wide / small tiles, K = 1024: 2048 x 4096 (128 wide tiles: half the chip) 40 / 36, 4096 x 4096 46 / 70.  With groups the small kernel's grid is
        // mostly empty and its tiles are no fuller: 640 rows in 16 groups, N = 1024, K = 1792 (72 tiles at most) 32 / 38
        if (vec && K % WK == 0 && wide_tiles >= (grp_offs ? 64 : 160) && wide_tiles <= (1 << 30)) {
            const int64_t words = c_dt == MI355_DT_F32 ? 4 : 8;  // of 16 bytes
            // four waves where they can -- K in pairs of K-tiles, two pairs at least; a panel's weights within a descriptor; the groups in the tables; columns and rows of C in whole 16 bytes -- and are faster: all
            // products of one matrix; groups from the K on where a tile's products outweigh its look-ups and a write-out with nothing beside it.  Four waves / eight, mean over 4 - 64 groups and 300 - 16 000 rows
            // (single ones up to 0.1 beside it): plain and squared 256 1.05 - 1.13, 512 1.00 - 1.05, 640 0.95 - 1.03, 768 0.94 - 1.01, 1 024 0.93 - 1.00, 2 048 0.86 - 0.91; SiLU 256 0.96 - 1.02, 512 0.91 - 0.97, 1 024
            // 0.90 - 0.94; the longer activations 256 1.07 - 1.10, 640 1.00 - 1.07, 768 0.99 - 1.03, 1 024 0.97 - 0.99 (single ones 1.15), 1 280
            // 0.94 - 0.97, 2 048 0.89 - 0.97.  One matrix: 256 0.54 - 0.79, 1 024 0.65 - 0.85
            const int least = !grp_offs ? 256 : epi == 4 ? 512 : epi >= 2 ? 1280 : 768;
            if (K % 128 == 0 && K >= least && batch <= QUAD_GROUPS && sbn * 2 * 512 < 0x7fffffffLL && (epi >= 2 ? n_out : N) % 8 == 0 && ldc % words == 0 && c_bs % words == 0 && ((uintptr_t)C & 15) == 0) {
                const unsigned grid = (unsigned)(wide_tiles < 256 ? wide_tiles : 256), lds = QUAD_SMEM + (2 * 256 + 2 * (QUAD_GROUPS + 1)) * 4;
                if (epi >= 2) bgemm_quad_kernel<true><<<grid, 256, lds, ST(stream)>>>(p, batch, (int)wide_tn);
                else bgemm_quad_kernel<false><<<grid, 256, lds, ST(stream)>>>(p, batch, (int)wide_tn);
                MI355_LAUNCH_CHECK("bgemm(four waves)");
                return 0;
            }
            bgemm_wide_kernel<<<(unsigned)wide_tiles, 512, 0, ST(stream)>>>(p, batch, (int)wide_tn);
            MI355_LAUNCH_CHECK("bgemm(wide)");
            return 0;
        }
        const int64_t my128 = ((int64_t)M + TM - 1) / TM;
        MI355_REQUIRE(my128 <= 65535, "bgemm: too many row tiles");
        const dim3 grid = tile_grid(p, (N + TM - 1) / TM, my128, batch);
        if (vec) bgemm_mfma128_kernel<true><<<grid, 256, 0, ST(stream)>>>(p);
        else bgemm_mfma128_kernel<false><<<grid, 256, 0, ST(stream)>>>(p);
        MI355_LAUNCH_CHECK("bgemm");
        return 0;
    }
    // fp32 rows times bf16 weights stored [out, in], in 16-byte words: three bf16 products for one.  The choice looks at types, strides and K only, never at M: a row's
    // bits do not depend on the batch.  Among the kernels: few rows stream the weights, more take the tile; 128-row tiles once they fill the chip.
    const bool f32_split = !use_mfma && a_dt == MI355_DT_F32 && b_dt == MI355_DT_BF16 && sbk == 1 && K % 8 == 0 && lda % 4 == 0 && a_bs % 4 == 0 && sbn % 8 == 0 && b_bs % 8 == 0 &&
                           ((uintptr_t)A & 15) == 0 && ((uintptr_t)B & 15) == 0;
    if (f32_split) {
        const int64_t ty = ((int64_t)M + 63) / 64;
        MI355_REQUIRE(ty <= 65535, "bgemm: too many row tiles");
        if (M <= F32_STREAM_ROWS) {
            const dim3 grid = tile_grid(p, (N + (epi >= 2 ? 63 : 31)) / (epi >= 2 ? 64 : 32), (M + 31) / 32, batch);
            const int64_t pitch = f32_rows_pitch(K), planes = 6 * (M + 1) * pitch, sums = SW * 16 * 64 * 4;
            if (epi < 2 && M <= 32 && planes <= F32_ROWS_LDS) {  // (M bounds the rows of every group)
                const unsigned lds = (unsigned)(planes > sums ? planes : sums);
                // (a group without rows is no work)
                const int64_t tiles = (int64_t)grid.x * (grp_offs && M < batch ? M : batch);
#define ROWS(C) bgemm_f32_rows_kernel<C><<<dim3((N + C - 1) / C, 1, batch), 64 * SW, lds, ST(stream)>>>(p, M, (int)pitch)
                if (tiles <= 32) ROWS(8); else if (tiles <= F32_ROWS_HALF) ROWS(16); else ROWS(32);
#undef ROWS
            } else if (epi >= 2) bgemm_stream_kernel<true, true><<<grid, 64 * SW, 0, ST(stream)>>>(p);
            else bgemm_stream_kernel<false, true><<<grid, 64 * SW, 0, ST(stream)>>>(p);
        } else {
            const int64_t tn = (N + 127) / 128, tiles = (grp_offs ? 1 : batch) * tn * ((M + 127) / 128);
            // Eight waves to a tile while every tile has a CU: 450 rows 2048 -> 1024 (64 tiles) 47.6 -> 39.9 us, 1024 -> 1536 29.5 -> 26.8; 304 tiles 38.5 | 53, 376 67 | 84; at K = 512 level.  Of groups a
            // tile for half of them is counted beside the full ones.
            const int64_t few = tn * (grp_offs ? ty + batch / 2 : ty * batch);
            if (tiles >= 512) bgemm_f32_tile_kernel<2, 1><<<tile_grid(p, tn, (M + 127) / 128, batch), 256, 0, ST(stream)>>>(p);
            else if (few <= 256 && K >= 1024) bgemm_f32_tile_kernel<1, 2><<<tile_grid(p, tn, ty, batch), 512, 0, ST(stream)>>>(p);
            else bgemm_f32_tile_kernel<1, 1><<<tile_grid(p, tn, ty, batch), 256, 0, ST(stream)>>>(p);
        }
        MI355_LAUNCH_CHECK("bgemm(f32)");
        return 0;
    }
    const int64_t my = ((int64_t)M + BM - 1) / BM;
    MI355_REQUIRE(my <= 65535, "bgemm: too many row tiles");
    const dim3 grid = tile_grid(p, (N + BN - 1) / BN, my, batch);
    if (use_mfma) bgemm_mfma_kernel<<<grid, 256, 0, ST(stream)>>>(p);
    else bgemm_fma_kernel<<<grid, 256, 0, ST(stream)>>>(p);
    MI355_LAUNCH_CHECK("bgemm");
    return 0;
}
