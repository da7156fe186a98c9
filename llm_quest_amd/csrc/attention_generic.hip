// Attention for head dims the tuned kernels of attention.hip do not cover (d_h = 256 of the Qwen3.5 gated-attention layers;
// 32 for the tiny fixtures), with the mask semantics of F.scaled_dot_product_attention as the reference calls it
// (qwen3_next_attention.py:238-254, qwen3_5_text_model.py:244-259): boolean mask, True = attend, everything else -inf.
//   allowed(i, j) = j <= i  OR  key j is padding        <- upstream ORs the inverted padding mask into the ALLOW mask,
//                                                           which un-masks padded keys for every query; reproduced.
// Same data flow as the tuned forward: S^T = K Q^T with the query on the MFMA lane (mfma_f32_32x32x16_bf16, A = K rows from
// LDS, B = Q rows in registers), lane-local online softmax, P^T packed from the accumulators as the B operand of
// O^T += V^T P^T, V consumed K-strided through ds_read_b64_tr_b16.
// Backward: query-major dQ (its prologue leaves delta = rowsum(dO * O)), then key-major dK / dV, no atomics.
// What bounds them: the products alone take 7 us of a forward at 8 sequences of 708 tokens, 8 heads of 256 over 2 key heads (17 700 pairs of 32 queries and 32 keys, 32 products
// of 32 clocks each), so a pair is a chain of LDS reads, products and softmax arithmetic of one wave, and its workgroup's tiles must already be there: tiles arrive through
// registers two ahead into two stages of swizzled LDS images, one barrier a tile, fragments four ahead of their products, masks as bits that tiles seen whole skip.
// Workgroups are up to four neighbouring (head, query tile) pairs of one kv head, or 32 keys, the long ones first: at 128 queries / keys each, a key-major grid was 96 workgroups.
// us, one tile per pair of barriers, loads exposed -> now (key-major: 1.5 times the products, to fit its accumulators -> a pair of waves, one product each):
//     8 x 708, 8 heads of 256 over 2: forward 195 -> 52, backward 729 -> 184;  1 x 333: 46 -> 22, 231 -> 91;  2 x 1 024 with a key mask (all keys walked): 193 -> 65, 858 -> 257;
//     3 x 100, 6 heads of 128 over 2: 13 -> 8.5, 59 -> 25;  2 x 77, 4 heads of 64: 8.5 -> 6.0, 22 -> 13 (the launches).
//
// PLAIN = true is the second semantics built on the same kernels (mi355_attn_dropout_fwd / _bwd): softmax over all keys or
// plain causal (no key mask, no quirk), with nn.Dropout(p) on the NORMALISED weights as ViTMultiHeadAttention applies it
// (vit_attention.py:79): O = ((P o M) / (1 - p)) V / l with l from the un-dropped P.  The mask is never stored: element
// (b, h, query, key) keeps iff Philox4x32-10(seed; key / 4, (b Hq + h) S + query, offset)[key % 4] >= round(p 2^32), and the
// backward regenerates it (dV += (P o M / keep)^T dO, dP = (dO V^T) o M / keep, dS = P (dP - delta), delta = rowsum(dO o O)).
#include "common.h"

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;
#define NEG_INF (-__builtin_huge_valf())

struct DropArgs {
    int causal;       // PLAIN only: 1 = keys <= query, 0 = every key
    unsigned thresh;  // 0 = no dropout
    float inv_keep;
    unsigned k0, k1, o0, o1;
};
// keep multipliers (0 or 1 / (1 - p)) of the four consecutive keys key4 .. key4+3 (key4 % 4 == 0) of attention row `row`
__device__ __forceinline__ void drop4(const DropArgs& da, unsigned row, int key4, float (&mul)[4]) {
    unsigned bits[4];
    philox4x32_10((unsigned)key4 >> 2, row, da.o0, da.o1, da.k0, da.k1, bits);
#pragma unroll
    for (int e = 0; e < 4; ++e) mul[e] = bits[e] >= da.thresh ? da.inv_keep : 0.f;
}

// the same bits where a lane holds one key and 16 queries (x = 4 g + e: row(x)): a draw is four keys of one query, and four neighbouring lanes hold those keys, so each of them draws
// for one query of every four and the bits go round by DPP -- 4 draws for 16.  Drawn per element, by both waves of a pair, they were more than the products: 128 x 197, 12 heads of 64, all keys seen, backward
// 552 -> 430 us (one draw per element by one wave for both, before the pair: 480); 8 x 708, 8 heads of 256 over 2, causal 340 -> 246.
template <class Row>
__device__ __forceinline__ void drop_bits(const DropArgs& da, int key, Row row, unsigned (&kept)[4]) {
    const int j = key & 3;
    unsigned mine = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        unsigned bits[4];
        philox4x32_10((unsigned)key >> 2, row(4 * g + j), da.o0, da.o1, da.k0, da.k1, bits);
#pragma unroll
        for (int w = 0; w < 4; ++w) mine |= (unsigned)(bits[w] >= da.thresh) << (4 * g + w);
    }
    kept[0] = (unsigned)__builtin_amdgcn_mov_dpp((int)mine, 0x00, 0xf, 0xf, true) >> j;  // quad_perm: lane e of the four
    kept[1] = (unsigned)__builtin_amdgcn_mov_dpp((int)mine, 0x55, 0xf, 0xf, true) >> j;
    kept[2] = (unsigned)__builtin_amdgcn_mov_dpp((int)mine, 0xaa, 0xf, 0xf, true) >> j;
    kept[3] = (unsigned)__builtin_amdgcn_mov_dpp((int)mine, 0xff, 0xf, 0xf, true) >> j;
}

template <int D>
struct GA {
    static constexpr int ROWB = D * 2;       // bytes per LDS row
    static constexpr int CH = D / 8;         // 16-byte chunks per row
    static constexpr int KS = D / 16;        // k-steps over d
    static constexpr int DT = D / 32;        // 32-row tiles of a transposed [d x 32] accumulator
    static constexpr int IMG = 32 * ROWB;    // one 32-row image
    static constexpr int PIECES = IMG / 1024;
};
// bank swizzle of a row image: chunk ^ the two 2-bit fields of row & 15, swapped.  The 16 rows that a ds_read_b128 serves together meet 16 different chunks of 256 bytes, and
// the four rows of a transposing read four different groups of four.
template <int D>
__device__ __forceinline__ int swz(int row) { return (((row & 3) << 2) | ((row >> 2) & 3)) & (GA<D>::CH - 1); }

// 32 rows x D bf16 on their way to a row image through the registers of NT threads (thread t): requested a tile ahead, put into LDS when the stage they go to is free.  Not by
// LDS-DMA: hipcc has every ds_read_b64_tr_b16 wait for a DMA under way, and a read from an asm statement of its own must not be left in flight.
template <int D, int NT>
struct Rows {
    static constexpr int N = 32 * GA<D>::CH / NT > 0 ? 32 * GA<D>::CH / NT : 1;
    u32x4 r[N];
    __device__ __forceinline__ void request(const bf16_t* base, int64_t ld, int rows_valid, int t) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int c = t + i * NT, row = c / GA<D>::CH;
            r[i] = u32x4{0u, 0u, 0u, 0u};
            if (row < rows_valid && (32 * GA<D>::CH % NT == 0 || row < 32)) r[i] = *reinterpret_cast<const u32x4*>(base + row * ld + c % GA<D>::CH * 8);
        }
    }
    __device__ __forceinline__ void put(char* img, int t) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int c = t + i * NT, row = c / GA<D>::CH;
            if (32 * GA<D>::CH % NT == 0 || row < 32) *reinterpret_cast<u32x4*>(img + row * GA<D>::ROWB + ((c % GA<D>::CH ^ swz<D>(row)) << 4)) = r[i];
        }
    }
};
// A operand (32 rows x 16 k) from a row image: row = lane & 31, k = 16 ks + 8 (lane >> 5) ..
template <int D>
__device__ __forceinline__ bf16x8 frag_rows(const char* img, int ks, int lane) {
    const int r = lane & 31;
    return *reinterpret_cast<const bf16x8*>(img + r * GA<D>::ROWB + (((2 * ks + (lane >> 5)) ^ swz<D>(r)) << 4));
}
// A operands of the TRANSPOSE of a row image: rows of A = image columns 32 dt .. + 31, k = image rows in the order in which an accumulator tile packs into a B operand: element
// j <-> image row k0 + 8 (j >> 2) + 4 (lane >> 5) + (j & 3).
// (the chunk of a column tile: bits 2, 3 meet the swizzle, bit 4 is an offset of 256 bytes; 8 rows further down the swizzle's low field differs by 2)
template <int D>
struct ColOff {
    static constexpr int N = GA<D>::DT < 4 ? GA<D>::DT : 4;
    int at[N];
};
template <int D>
__device__ __forceinline__ void col_offsets(ColOff<D>& o, int lane) {
    const int g = lane >> 4, q4 = (lane >> 2) & 3, p = lane & 3, row = 4 * (g >> 1) + q4;
#pragma unroll
    for (int dt = 0; dt < ColOff<D>::N; ++dt) o.at[dt] = row * GA<D>::ROWB + (((4 * dt + 2 * (g & 1) + (p >> 1)) ^ swz<D>(row)) << 4) + (p & 1) * 8;
}
template <int D>
__device__ __forceinline__ bf16x8 frag_cols(const char* img, const ColOff<D>& o, int dt, int k0) {
    const int at = o.at[dt & 3], imm = k0 * GA<D>::ROWB + (dt >> 2) * 256;
    bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)(img + at + imm));
    bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) bf16x4*)(img + (at ^ 0x20) + imm + 8 * GA<D>::ROWB));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// Fragments go to the products AHEAD at a time: the empty statement keeps the reads of a later group in front of the products of an earlier one, where hipcc, short of registers, reads
// each operand right before its product and waits a whole LDS latency there.
__device__ __forceinline__ void reads_stay() { asm volatile("" ::: "memory"); }
// s = (rows of the image) x (32 rows in registers)^T
template <int D>
__device__ __forceinline__ f32x16 dot_rows(const char* img, const bf16x8 (&b)[GA<D>::KS], int lane) {
    constexpr int AHEAD = GA<D>::KS < 4 ? GA<D>::KS : 4;
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    bf16x8 f[GA<D>::KS];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) f[i] = frag_rows<D>(img, i, lane);
#pragma unroll
    for (int g = 0; g < GA<D>::KS; g += AHEAD) {
#pragma unroll
        for (int i = g + AHEAD; i < g + 2 * AHEAD && i < GA<D>::KS; ++i) f[i] = frag_rows<D>(img, i, lane);
        reads_stay();
#pragma unroll
        for (int i = g; i < g + AHEAD; ++i) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[i], b[i], s, 0, 0, 0);
    }
    return s;
}
// acc[dt] += (image columns 32 dt ..)^T x (32 rows of the image, packed in p0 | p1)
// HOME: which file carries the tiles round the loop, 'a' or 'v' by an asm statement (left to itself, hipcc copies 128 registers from one to the other and back every trip), 0: hipcc's choice
template <int D, char HOME, int NDT>
__device__ __forceinline__ void add_cols(f32x16 (&acc)[NDT], const char* img, const ColOff<D>& o, const bf16x8& p0, const bf16x8& p1) {
    constexpr int N = 2 * NDT, AHEAD = N < 4 ? N : 4;
    bf16x8 f[N];
    auto read = [&](int i) { f[i] = frag_cols<D>(img, o, i % NDT, i < NDT ? 0 : 16); };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) read(i);
#pragma unroll
    for (int g = 0; g < N; g += AHEAD) {
#pragma unroll
        for (int i = g + AHEAD; i < g + 2 * AHEAD && i < N; ++i) read(i);
        reads_stay();
#pragma unroll
        for (int i = g; i < g + AHEAD; ++i) {
            f32x16& t = acc[i % NDT];
            const bf16x8& p = i < NDT ? p0 : p1;
            if constexpr (HOME == 'v') asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(t) : "v"(f[i]), "v"(p));
            else if constexpr (HOME == 'a') asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(t) : "v"(f[i]), "v"(p));
            else t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[i], p, t, 0, 0, 0);
        }
    }
}
// the last products of add_cols are written before the tiles are read
template <char HOME, int NDT>
__device__ __forceinline__ void settle(f32x16 (&acc)[NDT]) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
        if constexpr (HOME == 'v') asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[dt]));
        else if constexpr (HOME == 'a') asm volatile("s_nop 15\n\ts_nop 3" : "+a"(acc[dt]));
    }
}
// To stand right behind a chain of products: the tile is moved to VGPRs in the block that computed it.  hipcc pads the wait states between a product and the first read of its
// tile only there -- behind a branch the tile was read too early (wrong scores wherever no key mask was loaded in between).
__device__ __forceinline__ void land(f32x16& s) { asm volatile("" : "+v"(s)); }
// 32 bits, one a key of the tile from key0 on: visible to the query (existing, and not after it or padded -- quirk -- or every one of them); pad: the tile's padded keys
__device__ __forceinline__ unsigned visible_keys(int query, int key0, int S, bool every, unsigned pad) {
    const int n = S - key0, c = query - key0;
    const unsigned exist = n >= 32 ? ~0u : (1u << n) - 1u, past = c >= 31 ? ~0u : c < 0 ? 0u : (2u << c) - 1u;
    return exist & (every ? ~0u : past | pad);
}
__device__ __forceinline__ unsigned padded_keys(const uint8_t* km, int key0, int S, int lane) {
    if (!km) return 0u;
    const int key = key0 + (lane & 31);
    return (unsigned)__ballot(key < S && !km[min(key, S - 1)]);
}
// bit of accumulator register i in a mask of 32 rows that was moved down by 4 (lane >> 5)
__device__ __forceinline__ bool row_bit(unsigned bits, int i) { return bits >> (8 * (i >> 2) + (i & 3)) & 1u; }
__device__ __forceinline__ bf16x8 pack_frag(const f32x16& x, int s) {
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = pack_bf2(x[8 * s + 2 * e], x[8 * s + 2 * e + 1]);
    return __builtin_bit_cast(bf16x8, o);
}
// B operand fragments of a row held on the lane (row = lane & 31 of the wave's 32 rows)
template <int D>
__device__ __forceinline__ void load_row_frags(const bf16_t* rowptr, bool valid, int lane, bf16x8 (&f)[GA<D>::KS]) {
#pragma unroll
    for (int ks = 0; ks < GA<D>::KS; ++ks) {
        u32x4 v = {0, 0, 0, 0};
        if (valid) v = *reinterpret_cast<const u32x4*>(rowptr + 16 * ks + 8 * (lane >> 5));
        f[ks] = __builtin_bit_cast(bf16x8, v);
    }
}
// accumulator tile [32 d x 32 rows-on-lane] -> token-major bf16 rows (4 consecutive d per 8-byte store)
template <int NDT>
__device__ __forceinline__ void store_t_tiles(const f32x16 (&acc)[NDT], float mul, bf16_t* rowptr, bool valid, int lane) {
    if (!valid) return;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            u32x2 w;
            w[0] = pack_bf2(acc[dt][4 * i4] * mul, acc[dt][4 * i4 + 1] * mul);
            w[1] = pack_bf2(acc[dt][4 * i4 + 2] * mul, acc[dt][4 * i4 + 3] * mul);
            *reinterpret_cast<u32x2*>(rowptr + 32 * dt + 8 * i4 + 4 * (lane >> 5)) = w;
        }
}
template <int N>
__device__ __forceinline__ void zero_tiles(f32x16 (&acc)[N]) {
#pragma unroll
    for (int dt = 0; dt < N; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;
}

// The grid is (blocks of one (sequence, kv head), Hkv, B); under the causal mask a block's work grows with its index, so the numbers are dealt out anew: the last blocks of
// every (sequence, kv head) run first.
__device__ __forceinline__ void heavy_first(int& blk, int& hkv, int& b) {
    const int64_t heads = (int64_t)gridDim.y * gridDim.z, id = blockIdx.x + (int64_t)gridDim.x * (blockIdx.y + (int64_t)gridDim.y * blockIdx.z);
    blk = (int)(id / heads);
    const int bh = (int)(id - blk * heads);
    hkv = bh % (int)gridDim.y, b = bh / (int)gridDim.y;
}

// Query-major passes: an item is (query head of the group, 32 queries), heads fastest; a wave takes an item, a workgroup `per` neighbours, four as a rule -- the four heads of a group at
// one query tile, where a group has four -- that share every key / value tile.  Two stages of tiles, and a third tile on its way in registers under the products.
struct QItem {
    int h, q0, ntiles, b, hkv;
    bool on;
};
__device__ __forceinline__ QItem query_item(int S, int rep, bool all_keys, int wave, int per = 4) {  // per: items of a workgroup
    QItem it;
    int blk;
    heavy_first(blk, it.hkv, it.b);
    blk = (int)gridDim.x - 1 - blk;
    const int nqt = (S + 31) / 32, items = rep * nqt, i = blk * per + wave, last = min(blk * per + per - 1, items - 1);
    it.on = wave < per && i < items;
    const int c = it.on ? i : items - 1;
    it.h = it.hkv * rep + c % rep, it.q0 = c / rep * 32;
    it.ntiles = all_keys ? nqt : last / rep + 1;
    return it;
}

template <int D, bool PLAIN, bool DROP>
__global__ __launch_bounds__(256) void ga_fwd_kernel(int B, int S, int Hq, int Hkv, const bf16_t* __restrict__ q, int64_t ldq,
                                                     const bf16_t* __restrict__ k, int64_t ldk, const bf16_t* __restrict__ v, int64_t ldv,
                                                     bf16_t* __restrict__ o, int64_t ldo, float* __restrict__ lse,
                                                     const uint8_t* __restrict__ key_mask, float scale_log2, DropArgs da, int per) {
    using C = GA<D>;
    __shared__ __attribute__((aligned(1024))) char smem[4 * C::IMG];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool all_keys = PLAIN ? !da.causal : key_mask != nullptr;  // every key tile is walked
    const QItem it = query_item(S, Hq / Hkv, all_keys, wave, per);
    const int query = it.q0 + (lane & 31);
    const bool qvalid = it.on && query < S;
    const int64_t tok0 = (int64_t)it.b * S;
    const bf16_t *kb = k + tok0 * ldk + (int64_t)it.hkv * D, *vb = v + tok0 * ldv + (int64_t)it.hkv * D;
    Rows<D, 256> kn, vn;  // the tile behind the one that is put next
    auto request = [&](int kt) {
        kn.request(kb + (int64_t)kt * 32 * ldk, ldk, S - kt * 32, threadIdx.x);
        vn.request(vb + (int64_t)kt * 32 * ldv, ldv, S - kt * 32, threadIdx.x);
    };
    auto put = [&](int kt) {
        char* st = smem + (kt & 1) * 2 * C::IMG;
        kn.put(st, threadIdx.x);
        vn.put(st + C::IMG, threadIdx.x);
    };
    request(0);
    bf16x8 qf[C::KS];
    load_row_frags<D>(q + (tok0 + query) * ldq + (int64_t)it.h * D, qvalid, lane, qf);
    ColOff<D> co;
    col_offsets<D>(co, lane);
    f32x16 acc[C::DT];
    zero_tiles(acc);
    float m = NEG_INF, l = 0.f;
    const uint8_t* km = (!PLAIN && key_mask) ? key_mask + tok0 : nullptr;
    const unsigned drow = (unsigned)(((int64_t)it.b * Hq + it.h) * S + query);
    put(0);
    if (it.ntiles > 1) request(1);
    for (int kt = 0; kt < it.ntiles; ++kt) {
        const int key0 = kt * 32;
        __syncthreads();
        if (kt + 1 < it.ntiles) put(kt + 1);
        if (kt + 2 < it.ntiles) request(kt + 2);
        if (!it.on || (!all_keys && key0 > it.q0 + 31)) continue;  // no item, or a tile entirely above this wave's diagonal
        const char* kimg = smem + (kt & 1) * 2 * C::IMG;
        f32x16 s = dot_rows<D>(kimg, qf, lane);
        land(s);
        float mx = NEG_INF;
        const unsigned vis = visible_keys(query, key0, S, PLAIN && !da.causal, padded_keys(km, key0, S, lane));
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] *= scale_log2;
        if (!__all(vis == ~0u)) {
            const unsigned bits = vis >> 4 * (lane >> 5);
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = row_bit(bits, i) ? s[i] : NEG_INF;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m, mx);
        const float m_use = m_new == NEG_INF ? 0.f : m_new;
        if (__any(m_new > m)) {
            const float alpha = __builtin_amdgcn_exp2f(m - m_use);
            l *= alpha;
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[dt][i] *= alpha;
        }
        float rs = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = __builtin_amdgcn_exp2f(s[i] - m_use);
            rs += s[i];
        }
        rs += __shfl_xor(rs, 32, 64);
        l += rs;
        m = m_new;
        if (DROP && da.thresh) {  // (DROP is a template parameter: the p = 0 kernels of the Qwen3.5 training path carry no Philox code)  // dropout on the weights that multiply V; the row sum above keeps every key
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float mul[4];
                drop4(da, drow, key0 + 8 * g + 4 * (lane >> 5), mul);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[4 * g + e] *= mul[e];
            }
        }
        add_cols<D, D == 256 ? 'v' : 0>(acc, kimg + C::IMG, co, pack_frag(s, 0), pack_frag(s, 1));
    }
    settle<D == 256 ? 'v' : 0>(acc);
    store_t_tiles<C::DT>(acc, 1.f / l, o + (tok0 + query) * ldo + (int64_t)it.h * D, qvalid, lane);
    if (lane < 32 && qvalid) lse[((int64_t)it.b * Hq + it.h) * S + query] = (m + log2f(l)) * LN2;
}

// dQ; its prologue leaves delta[b, h, s] = sum_d dO * O for the key-major pass behind it.
template <int D, bool PLAIN, bool DROP>
__global__ __launch_bounds__(256) void ga_bwd_dq_kernel(int B, int S, int Hq, int Hkv, const bf16_t* __restrict__ q, int64_t ldq,
                                                        const bf16_t* __restrict__ k, int64_t ldk, const bf16_t* __restrict__ v, int64_t ldv,
                                                        const bf16_t* __restrict__ o, int64_t ldo, const bf16_t* __restrict__ d_o, int64_t lddo,
                                                        const float* __restrict__ lse, float* __restrict__ delta, bf16_t* __restrict__ dq, int64_t lddq,
                                                        const uint8_t* __restrict__ key_mask, float scale, DropArgs da) {
    using C = GA<D>;
    __shared__ __attribute__((aligned(1024))) char smem[4 * C::IMG];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool all_keys = PLAIN ? !da.causal : key_mask != nullptr;
    const QItem it = query_item(S, Hq / Hkv, all_keys, wave);
    const int query = it.q0 + (lane & 31);
    const bool qvalid = it.on && query < S;
    const int64_t tok0 = (int64_t)it.b * S;
    const bf16_t *kb = k + tok0 * ldk + (int64_t)it.hkv * D, *vb = v + tok0 * ldv + (int64_t)it.hkv * D;
    Rows<D, 256> kn, vn;  // the tile behind the one that is put next
    auto request = [&](int kt) {
        kn.request(kb + (int64_t)kt * 32 * ldk, ldk, S - kt * 32, threadIdx.x);
        vn.request(vb + (int64_t)kt * 32 * ldv, ldv, S - kt * 32, threadIdx.x);
    };
    auto put = [&](int kt) {
        char* st = smem + (kt & 1) * 2 * C::IMG;
        kn.put(st, threadIdx.x);
        vn.put(st + C::IMG, threadIdx.x);
    };
    request(0);
    bf16x8 qf[C::KS], gf[C::KS];
    load_row_frags<D>(d_o + (tok0 + query) * lddo + (int64_t)it.h * D, qvalid, lane, gf);
    load_row_frags<D>(o + (tok0 + query) * ldo + (int64_t)it.h * D, qvalid, lane, qf);
    const float lse_q = qvalid ? lse[((int64_t)it.b * Hq + it.h) * S + query] * LOG2E : 0.f;
    float delta_q = 0.f;
#pragma unroll
    for (int ks = 0; ks < C::KS; ++ks)
#pragma unroll
        for (int e = 0; e < 8; ++e) delta_q = fmaf(bf2f((bf16_t)gf[ks][e]), bf2f((bf16_t)qf[ks][e]), delta_q);
    delta_q += __shfl_xor(delta_q, 32, 64);
    if (lane < 32 && qvalid) delta[((int64_t)it.b * Hq + it.h) * S + query] = delta_q;
    load_row_frags<D>(q + (tok0 + query) * ldq + (int64_t)it.h * D, qvalid, lane, qf);
    const float scale_log2 = scale * LOG2E;
    ColOff<D> co;
    col_offsets<D>(co, lane);
    f32x16 acc[C::DT];
    zero_tiles(acc);
    const uint8_t* km = (!PLAIN && key_mask) ? key_mask + tok0 : nullptr;
    const unsigned drow = (unsigned)(((int64_t)it.b * Hq + it.h) * S + query);
    put(0);
    if (it.ntiles > 1) request(1);
    auto next_tile = [&](int kt) {
        __syncthreads();
        if (kt + 1 < it.ntiles) put(kt + 1);
        if (kt + 2 < it.ntiles) request(kt + 2);
    };
    // A wave without an item, or above its diagonal, multiplies nothing: a weight of zero times a later token that is not finite would be NaN.  Those tiles are its last ones, so they
    // have a loop of their own (a branch around the products costs every trip 256 register copies).
    const int seen = !it.on ? 0 : all_keys ? it.ntiles : it.q0 / 32 + 1;
    for (int kt = 0; kt < seen; ++kt) {
        const int key0 = kt * 32;
        next_tile(kt);
        const char* kimg = smem + (kt & 1) * 2 * C::IMG;
        const char* vimg = kimg + C::IMG;
        f32x16 s = dot_rows<D>(kimg, qf, lane), dp = dot_rows<D>(vimg, gf, lane);
        land(s), land(dp);
        if (DROP && da.thresh) {  // (DROP is a template parameter: the p = 0 kernels of the Qwen3.5 training path carry no Philox code)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float mul[4];
                drop4(da, drow, key0 + 8 * g + 4 * (lane >> 5), mul);
#pragma unroll
                for (int e = 0; e < 4; ++e) dp[4 * g + e] *= mul[e];
            }
        }
        const unsigned vis = qvalid ? visible_keys(query, key0, S, PLAIN && !da.causal, padded_keys(km, key0, S, lane)) : 0u;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(s[i] * scale_log2 - lse_q);
        if (!__all(vis == ~0u)) {
            const unsigned bits = vis >> 4 * (lane >> 5);
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = row_bit(bits, i) ? s[i] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = s[i] * (dp[i] - delta_q) * scale;
        add_cols<D, D == 256 ? 'a' : 0>(acc, kimg, co, pack_frag(s, 0), pack_frag(s, 1));
    }
    settle<D == 256 ? 'a' : 0>(acc);
    for (int kt = seen; kt < it.ntiles; ++kt) next_tile(kt);
    store_t_tiles<C::DT>(acc, 1.f, dq + (tok0 + query) * lddq + (int64_t)it.h * D, qvalid, lane);
}

// Key-major pass: a workgroup owns 32 keys of one kv head; the (query head, query tile) pairs from the diagonal on go round two streams of two waves.  The first wave of a stream
// works out P and dV, the second dP and dK -- one wave's registers do not hold both gradients and the key and value rows at D = 256 -- and P passes between them through LDS.
// Two stages of tiles per stream, a third pair's on its way in registers under the products; the streams' sums meet in LDS at the end, stream 0's first.
template <int D, bool PLAIN, bool DROP>
__global__ __launch_bounds__(256) void ga_bwd_dkv_kernel(int B, int S, int Hq, int Hkv, const bf16_t* __restrict__ q, int64_t ldq,
                                                         const bf16_t* __restrict__ k, int64_t ldk, const bf16_t* __restrict__ v, int64_t ldv,
                                                         const bf16_t* __restrict__ d_o, int64_t lddo, const float* __restrict__ lse,
                                                         const float* __restrict__ delta, bf16_t* __restrict__ dk, int64_t lddk,
                                                         bf16_t* __restrict__ dv, int64_t lddv, const uint8_t* __restrict__ key_mask, float scale,
                                                         DropArgs da) {
    using C = GA<D>;
    __shared__ __attribute__((aligned(1024))) char smem[8 * C::IMG];  // [stream][stage][query rows | dO rows]
    __shared__ __attribute__((aligned(16))) f32x4 probs[2][4][64];
    __shared__ __attribute__((aligned(16))) float stats[2][4][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), stream = wave >> 1;
    const bool second = wave & 1;
    int kb, hkv, b;
    heavy_first(kb, hkv, b);  // (the first keys have the most queries)
    const int rep = Hq / Hkv, k0 = kb * 32, key = k0 + (lane & 31);
    const bool kvalid = key < S;
    const int64_t tok0 = (int64_t)b * S;
    const bool all_queries = PLAIN ? !da.causal : key_mask != nullptr;  // every query tile is walked
    const int qt0 = all_queries ? 0 : kb, items = rep * ((S + 31) / 32 - qt0), rounds = (items + 1) / 2;
    auto row_of = [&](int r, int& h, int& qs) {  // the stream's item of a round; past the last one, that one again, of which nothing is then seen
        const int i = min(2 * r + stream, items - 1);
        h = hkv * rep + i % rep, qs = (qt0 + i / rep) * 32;
        return 2 * r + stream < items;
    };
    float st_next = 0.f;  // the first wave: lse, the second: delta of the queries of the item that is put next
    Rows<D, 64> rn;
    auto request = [&](int r) {
        int h, qs;
        row_of(r, h, qs);
        const int qi = qs + (lane & 31);
        st_next = qi < S ? (second ? delta : lse)[((int64_t)b * Hq + h) * S + qi] : 0.f;
        rn.request((second ? d_o + (tok0 + qs) * lddo : q + (tok0 + qs) * ldq) + (int64_t)h * D, second ? lddo : ldq, S - qs, lane);
    };
    auto put = [&](int r) {
        rn.put(smem + (stream * 2 + (r & 1)) * 2 * C::IMG + (second ? C::IMG : 0), lane);
        if (lane < 32) stats[r & 1][wave][lane] = second ? st_next : st_next * LOG2E;
    };
    request(0);
    bf16x8 kvf[C::KS];
    if (second) load_row_frags<D>(v + (tok0 + key) * ldv + (int64_t)hkv * D, kvalid, lane, kvf);
    else load_row_frags<D>(k + (tok0 + key) * ldk + (int64_t)hkv * D, kvalid, lane, kvf);
    const bool padded = !PLAIN && key_mask && kvalid && !key_mask[tok0 + key];
    const float scale_log2 = scale * LOG2E;
    ColOff<D> co;
    col_offsets<D>(co, lane);
    f32x16 acc[C::DT];
    zero_tiles(acc);
    put(0);
    if (rounds > 1) request(1);
    for (int r = 0; r < rounds; ++r) {
        int h, qs;
        const bool on = row_of(r, h, qs);
        __syncthreads();
        if (r + 1 < rounds) put(r + 1);
        if (r + 2 < rounds) request(r + 2);
        const char *qimg = smem + (stream * 2 + (r & 1)) * 2 * C::IMG, *gimg = qimg + C::IMG, *rows = second ? gimg : qimg;
        f32x16 s = dot_rows<D>(rows, kvf, lane);  // the first wave's scores, the second's dP
        land(s);
        if (!second) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 ls = *reinterpret_cast<const f32x4*>(&stats[r & 1][wave][8 * g + 4 * (lane >> 5)]);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[4 * g + e] = __builtin_amdgcn_exp2f(s[4 * g + e] * scale_log2 - ls[e]);
            }
            const int n = S - qs, c = key - qs;  // queries of the tile: n exist, those from c on are not before the key
            const unsigned exist = n >= 32 ? ~0u : (1u << n) - 1u, after = c <= 0 ? ~0u : c > 31 ? 0u : ~0u << c;
            const unsigned vis = kvalid && on ? exist & ((PLAIN && !da.causal) || padded ? ~0u : after) : 0u;
            if (!__all(vis == ~0u)) {
                const unsigned bits = vis >> 4 * (lane >> 5);
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = row_bit(bits, i) ? s[i] : 0.f;
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) probs[stream][g][lane] = f32x4{s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
        }
        __syncthreads();
        unsigned kept[4] = {~0u, ~0u, ~0u, ~0u};  // per query of a group of four: bit 4 g, this lane's key
        // (DROP is a template parameter: the p = 0 kernels of the Qwen3.5 training path carry no Philox code)
        if (DROP && da.thresh) drop_bits(da, key, [&](int x) { return (unsigned)(((int64_t)b * Hq + h) * S + qs + 8 * (x >> 2) + 4 * (lane >> 5) + (x & 3)); }, kept);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 dl = *reinterpret_cast<const f32x4*>(&stats[r & 1][wave][8 * g + 4 * (lane >> 5)]), p = probs[stream][g][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int x = 4 * g + e;
                const float keep = DROP && da.thresh ? (kept[e] >> 4 * g & 1u ? da.inv_keep : 0.f) : 1.f;
                if (second) s[x] = p[e] * (s[x] * keep - dl[e]) * scale;
                else s[x] *= keep;
            }
        }
        add_cols<D, D == 256 ? 'a' : 0>(acc, second ? qimg : gimg, co, pack_frag(s, 0), pack_frag(s, 1));
    }
    settle<D == 256 ? 'a' : 0>(acc);
    __syncthreads();
    f32x4* other = reinterpret_cast<f32x4*>(smem + (wave & 1) * 2 * C::IMG);  // D / 32 tiles of fp32 take two images
    if (stream == 1) {
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) other[(dt * 4 + i4) * 64 + lane] = f32x4{acc[dt][4 * i4], acc[dt][4 * i4 + 1], acc[dt][4 * i4 + 2], acc[dt][4 * i4 + 3]};
    }
    __syncthreads();
    if (stream == 1) return;
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
            const f32x4 t = other[(dt * 4 + i4) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[dt][4 * i4 + e] += t[e];
        }
    store_t_tiles<C::DT>(acc, 1.f, second ? dk + (tok0 + key) * lddk + (int64_t)hkv * D : dv + (tok0 + key) * lddv + (int64_t)hkv * D, kvalid, lane);
}

dim3 query_grid(int B, int S, int Hq, int Hkv, int per = 4) { return dim3((Hq / Hkv * ((S + 31) / 32) + per - 1) / per, Hkv, B); }
// Items of a workgroup in the forward pass: four waves on a CU share its LDS, so while CUs are without a workgroup an item has one of its own (its other three waves fetch), or two have.  us with 1 / 2 / 4,
// head dim 256, 8 heads over 2: 20 tokens 6.9 / 7.9 / 9.8, 333 23 / 24 / 26, 2 000 (504 items) 119 / 108 / 111, 3 x 708 (552) 58 / 45 / 47; 8 x 708 (1 472) 137 / 81 / 51.  Heads of 32 and 64
// gain nothing from two (2 000 tokens, 8 heads of 32 over 2: 47 / 50 / 48).
int items_per_workgroup(int B, int S, int Hq, int Hkv, int D) {
    const int64_t items = (int64_t)Hq / Hkv * ((S + 31) / 32), groups = (int64_t)Hkv * B;
    return items * groups <= 256 ? 1 : D >= 128 && (items + 1) / 2 * groups <= 256 ? 2 : 4;
}

int check_ga(int B, int S, int Hq, int Hkv, int D, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo) {
    MI355_REQUIRE(B > 0 && S > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0, "attn_generic: query heads (%d) must be a multiple of kv heads (%d)", Hq, Hkv);
    MI355_REQUIRE(D == 32 || D == 64 || D == 128 || D == 256, "attn_generic: head_dim %d not built (32, 64, 128, 256)", D);
    MI355_REQUIRE(ldq >= (int64_t)Hq * D && ldo >= (int64_t)Hq * D && ldk >= (int64_t)Hkv * D && ldv >= (int64_t)Hkv * D, "attn_generic: leading dimension smaller than heads*head_dim");
    MI355_REQUIRE(ldq % 8 == 0 && ldk % 8 == 0 && ldv % 8 == 0 && ldo % 8 == 0, "attn_generic: leading dimensions must be multiples of 8 elements");
    MI355_REQUIRE(B <= 65535 && Hq <= 65535, "attn_generic: grid limits");
    return 0;
}

}  // namespace

#define ST(s) ((hipStream_t)(s))

extern "C" int mi355_attn_generic_fwd(int B, int S, int Hq, int Hkv, int D, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v,
                                      int64_t ldv, void* o, int64_t ldo, float* lse, const uint8_t* key_mask, float scale, void* stream) {
#define GA_DROP false
    if (check_ga(B, S, Hq, Hkv, D, ldq, ldk, ldv, ldo)) return 1;
    MI355_REQUIRE(q && k && v && o && lse, "attn_generic_fwd: null pointer");
    const int per = items_per_workgroup(B, S, Hq, Hkv, D);
    const dim3 grid = query_grid(B, S, Hq, Hkv, per);
    const DropArgs da = {};
#define LAUNCH(DD) ga_fwd_kernel<DD, false, GA_DROP><<<grid, 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (bf16_t*)o, ldo, lse, key_mask, scale * LOG2E, da, per)
    switch (D) {
        case 32: LAUNCH(32); break;
        case 64: LAUNCH(64); break;
        case 128: LAUNCH(128); break;
        default: LAUNCH(256); break;
    }
#undef LAUNCH
    MI355_LAUNCH_CHECK("attn_generic_fwd");
#undef GA_DROP
    return 0;
}

extern "C" int mi355_attn_generic_bwd(int B, int S, int Hq, int Hkv, int D, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v,
                                      int64_t ldv, const void* o, int64_t ldo, const void* d_o, int64_t lddo, const float* lse, float* delta,
                                      void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv, int64_t lddv, const uint8_t* key_mask,
                                      float scale, void* stream) {
#define GA_DROP false
    if (check_ga(B, S, Hq, Hkv, D, ldq, ldk, ldv, ldo)) return 1;
    if (check_ga(B, S, Hq, Hkv, D, lddq, lddk, lddv, lddo)) return 1;
    MI355_REQUIRE(q && k && v && o && d_o && lse && delta && dq && dk && dv, "attn_generic_bwd: null pointer");
    const dim3 gq = query_grid(B, S, Hq, Hkv);
    const DropArgs da = {};
#define LAUNCH_DQ(DD) ga_bwd_dq_kernel<DD, false, GA_DROP><<<gq, 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (const bf16_t*)o, ldo, (const bf16_t*)d_o, lddo, lse, delta, (bf16_t*)dq, lddq, key_mask, scale, da)
#define LAUNCH_DKV(DD) ga_bwd_dkv_kernel<DD, false, GA_DROP><<<dim3((S + 31) / 32, Hkv, B), 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (const bf16_t*)d_o, lddo, lse, delta, (bf16_t*)dk, lddk, (bf16_t*)dv, lddv, key_mask, scale, da)
    switch (D) {
        case 32: LAUNCH_DQ(32); LAUNCH_DKV(32); break;
        case 64: LAUNCH_DQ(64); LAUNCH_DKV(64); break;
        case 128: LAUNCH_DQ(128); LAUNCH_DKV(128); break;
        default: LAUNCH_DQ(256); LAUNCH_DKV(256); break;
    }
#undef LAUNCH_DQ
#undef LAUNCH_DKV
    MI355_LAUNCH_CHECK("attn_generic_bwd");
#undef GA_DROP
    return 0;
}

// ---- PLAIN semantics: full or plain-causal softmax with dropout on the weights (ViTMultiHeadAttention in train mode) -------------
static int make_drop_args(const char* who, int B, int S, int Hq, int causal, float p, uint64_t seed, uint64_t offset, DropArgs* da) {
    MI355_REQUIRE(p >= 0.f && p < 1.f, "%s: p must be in [0, 1) (got %f)", who, (double)p);
    MI355_REQUIRE((int64_t)B * Hq * S < (int64_t)1 << 32, "%s: B * Hq * S must fit 32 bits (dropout counter)", who);
    da->causal = causal != 0;
    da->thresh = p > 0.f ? mi355_dropout_threshold(p) : 0u;
    da->inv_keep = 1.0f / (1.0f - p);
    da->k0 = (unsigned)seed, da->k1 = (unsigned)(seed >> 32), da->o0 = (unsigned)offset, da->o1 = (unsigned)(offset >> 32);
    return 0;
}

extern "C" int mi355_attn_dropout_fwd(int B, int S, int Hq, int Hkv, int D, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v,
                                      int64_t ldv, void* o, int64_t ldo, float* lse, int causal, float scale, float p, uint64_t seed, uint64_t offset,
                                      void* stream) {
    if (check_ga(B, S, Hq, Hkv, D, ldq, ldk, ldv, ldo)) return 1;
    MI355_REQUIRE(q && k && v && o && lse, "attn_dropout_fwd: null pointer");
    DropArgs da;
    if (make_drop_args("attn_dropout_fwd", B, S, Hq, causal, p, seed, offset, &da)) return 1;
    const int per = items_per_workgroup(B, S, Hq, Hkv, D);
    const dim3 grid = query_grid(B, S, Hq, Hkv, per);
#define LAUNCH(DD) ga_fwd_kernel<DD, true, true><<<grid, 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (bf16_t*)o, ldo, lse, nullptr, scale * LOG2E, da, per)
    switch (D) {
        case 32: LAUNCH(32); break;
        case 64: LAUNCH(64); break;
        case 128: LAUNCH(128); break;
        default: LAUNCH(256); break;
    }
#undef LAUNCH
    MI355_LAUNCH_CHECK("attn_dropout_fwd");
    return 0;
}

extern "C" int mi355_attn_dropout_bwd(int B, int S, int Hq, int Hkv, int D, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v,
                                      int64_t ldv, const void* o, int64_t ldo, const void* d_o, int64_t lddo, const float* lse, float* delta,
                                      void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv, int64_t lddv, int causal, float scale, float p,
                                      uint64_t seed, uint64_t offset, void* stream) {
    if (check_ga(B, S, Hq, Hkv, D, ldq, ldk, ldv, ldo)) return 1;
    if (check_ga(B, S, Hq, Hkv, D, lddq, lddk, lddv, lddo)) return 1;
    MI355_REQUIRE(q && k && v && o && d_o && lse && delta && dq && dk && dv, "attn_dropout_bwd: null pointer");
    DropArgs da;
    if (make_drop_args("attn_dropout_bwd", B, S, Hq, causal, p, seed, offset, &da)) return 1;
    const dim3 gq = query_grid(B, S, Hq, Hkv);
#define LAUNCH_DQ(DD) ga_bwd_dq_kernel<DD, true, true><<<gq, 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (const bf16_t*)o, ldo, (const bf16_t*)d_o, lddo, lse, delta, (bf16_t*)dq, lddq, nullptr, scale, da)
#define LAUNCH_DKV(DD) ga_bwd_dkv_kernel<DD, true, true><<<dim3((S + 31) / 32, Hkv, B), 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (const bf16_t*)d_o, lddo, lse, delta, (bf16_t*)dk, lddk, (bf16_t*)dv, lddv, nullptr, scale, da)
    switch (D) {
        case 32: LAUNCH_DQ(32); LAUNCH_DKV(32); break;
        case 64: LAUNCH_DQ(64); LAUNCH_DKV(64); break;
        case 128: LAUNCH_DQ(128); LAUNCH_DKV(128); break;
        default: LAUNCH_DQ(256); LAUNCH_DKV(256); break;
    }
#undef LAUNCH_DQ
#undef LAUNCH_DKV
    MI355_LAUNCH_CHECK("attn_dropout_bwd");
    return 0;
}

// ---- the reference's SDPA call WITH dropout_p and a padding mask (GatedAttention in training mode on padded batches, qwen3_next_attention.py:240-253):
// the quirk-mask kernels (PLAIN = false) with the dropout arguments set -- Philox masks on the normalised weights, regenerated by the backward.
extern "C" int mi355_attn_generic_dropout_fwd(int B, int S, int Hq, int Hkv, int D, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v,
                                              int64_t ldv, void* o, int64_t ldo, float* lse, const uint8_t* key_mask, float scale, float p, uint64_t seed,
                                              uint64_t offset, void* stream) {
#define GA_DROP true
    if (check_ga(B, S, Hq, Hkv, D, ldq, ldk, ldv, ldo)) return 1;
    MI355_REQUIRE(q && k && v && o && lse, "attn_generic_dropout_fwd: null pointer");
    DropArgs da;
    if (make_drop_args("attn_generic_dropout_fwd", B, S, Hq, 1, p, seed, offset, &da)) return 1;
    const int per = items_per_workgroup(B, S, Hq, Hkv, D);
    const dim3 grid = query_grid(B, S, Hq, Hkv, per);
#define LAUNCH(DD) ga_fwd_kernel<DD, false, GA_DROP><<<grid, 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (bf16_t*)o, ldo, lse, key_mask, scale * LOG2E, da, per)
    switch (D) {
        case 32: LAUNCH(32); break;
        case 64: LAUNCH(64); break;
        case 128: LAUNCH(128); break;
        default: LAUNCH(256); break;
    }
#undef LAUNCH
    MI355_LAUNCH_CHECK("attn_generic_dropout_fwd");
#undef GA_DROP
    return 0;
}

extern "C" int mi355_attn_generic_dropout_bwd(int B, int S, int Hq, int Hkv, int D, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v,
                                              int64_t ldv, const void* o, int64_t ldo, const void* d_o, int64_t lddo, const float* lse, float* delta,
                                              void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv, int64_t lddv, const uint8_t* key_mask, float scale,
                                              float p, uint64_t seed, uint64_t offset, void* stream) {
#define GA_DROP true
    if (check_ga(B, S, Hq, Hkv, D, ldq, ldk, ldv, ldo)) return 1;
    if (check_ga(B, S, Hq, Hkv, D, lddq, lddk, lddv, lddo)) return 1;
    MI355_REQUIRE(q && k && v && o && d_o && lse && delta && dq && dk && dv, "attn_generic_dropout_bwd: null pointer");
    DropArgs da;
    if (make_drop_args("attn_generic_dropout_bwd", B, S, Hq, 1, p, seed, offset, &da)) return 1;
    const dim3 gq = query_grid(B, S, Hq, Hkv);
#define LAUNCH_DQ(DD) ga_bwd_dq_kernel<DD, false, GA_DROP><<<gq, 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (const bf16_t*)o, ldo, (const bf16_t*)d_o, lddo, lse, delta, (bf16_t*)dq, lddq, key_mask, scale, da)
#define LAUNCH_DKV(DD) ga_bwd_dkv_kernel<DD, false, GA_DROP><<<dim3((S + 31) / 32, Hkv, B), 256, 0, ST(stream)>>>(B, S, Hq, Hkv, (const bf16_t*)q, ldq, (const bf16_t*)k, ldk, (const bf16_t*)v, ldv, (const bf16_t*)d_o, lddo, lse, delta, (bf16_t*)dk, lddk, (bf16_t*)dv, lddv, key_mask, scale, da)
    switch (D) {
        case 32: LAUNCH_DQ(32); LAUNCH_DKV(32); break;
        case 64: LAUNCH_DQ(64); LAUNCH_DKV(64); break;
        case 128: LAUNCH_DQ(128); LAUNCH_DKV(128); break;
        default: LAUNCH_DQ(256); LAUNCH_DKV(256); break;
    }
#undef LAUNCH_DQ
#undef LAUNCH_DKV
    MI355_LAUNCH_CHECK("attn_generic_dropout_bwd");
#undef GA_DROP
    return 0;
}
