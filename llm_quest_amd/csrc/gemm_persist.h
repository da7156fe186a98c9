// Short sums over many tiles, NT form: one workgroup of eight waves (128x64 outputs each, gemm_tile's) per CU, walking its share of the 256x256 tiles (included by gemm.hip).
//
// What bounds it: the results' way to memory.  Two waves per SIMD fill each other's waits in a write-out, which gemm_quad.h's one wave cannot, and K-tiles are 64 (an odd number of them is made even by one
// of zeros there): short_nt has the line.  us, gemm_quad.h (K <= 192, which it does not take: gemm_tile) -> here: 70 000 x 1 536, K = 128 68 -> 46, 256 73 -> 66, 320 91 -> 78; 25 216 x 2 304, K = 320 54 -> 45, 576 77 -> 68,
// 704 85 -> 79, 832 94 / 95; SwiGLU forward of 2 x 1 152 columns, K = 128 58 -> 40, 448 75 -> 68, 832 104 / 105.
//   * the K-tile stream runs across tile boundaries (the last two barriers of a tile request the next tile's first two K-tiles), so there is no prologue, no
//     retire wait and no workgroup turnover;
//   * the write-out stages through a 32-KiB region BESIDE the two stages (4 KiB per wave: 32 rows x 64 columns of packed bf16 at a time, swizzled, not padded), so it
//     needs no barrier and does not collide with the stream; the B fragment is the MFMA's first operand, so a lane holds four consecutive columns of a row and
//     packs them itself: a quarter of the LDS bytes of gemm_tile's fp32 staging.
//   * more than 128 column panels (vocabulary-wide heads): WALK.  us, without -> with: 2 048 x 151 936, K = 256 229 -> 185, 512 359 -> 306, 1 024 x 248 320, K = 512 311 -> 249; 4 096 x 32 000, 512 125 / 130.
// The bits of gemm_bf16_kernel (same MFMA sequence per output, same rounding).  bf16 output, K % 64 == 0, K >= 128, N % 8 == 0, no bias.
template <int KIND, bool RES, bool WALK>  // KIND: MI355_EPI_NONE (RES: + bf16 residual, added in fp32 before the rounding), MI355_EPI_SWIGLU_FWD, MI355_EPI_SWIGLU_BWD (see gemm_tile's epilogue for both)
__global__ __launch_bounds__(512, 2) void gemm_nt_persist_kernel(GemmParams p, int ntiles) {
    using T = Cfg256;
    constexpr int BK = 64, HM = T::FM / 2;
    static_assert(T::A_PPW == 4 && T::B_PPW == 4 && T::FM == 8 && T::FN == 4 && T::NS == 2, "written for 8 waves of 128x64 on two 64-KiB stages");
    __shared__ __attribute__((aligned(16))) char smem[2 * T::STAGE + 32768];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    char* const stg = smem + 2 * T::STAGE + wave * 4096;
    const int wr0 = (wave / T::WN) * T::WTM, wc0 = (wave % T::WN) * T::WTN;
    const int nt = (int)(p.K / BK);
    const int G = gridDim.x;

    // The walk: tile blockIdx.x + j G of the XCD-chunked order in 6-row groups.  WALK: weight-stationary per XCD -- column panels four at a time, an XCD owns a contiguous run of (column group, row
    // panel) pairs, its 32 workgroups are 4 column panels x 8 row streams, stream r takes the run's pairs r, r + 8, ...  A column group's missing panels (N / 256 not a multiple of 4) are walked as empty
    // tiles (everything beyond the matrix: zero operands, no stores).  Needs the full grid of 256.  Stores with the non-temporal hint there: a tile is written once and next read by another kernel.
    constexpr int CAUX = WALK ? 2 : 0;
    const int wk_xcd = blockIdx.x & 7, wk_l = blockIdx.x >> 3, wk_ci = wk_l & 3;
    const int64_t wk_pairs = (int64_t)((p.tiles_n + 3) >> 2) * p.tiles_m;
    const int wk_lo = (int)(wk_pairs * wk_xcd / 8) + (wk_l >> 2), wk_hi = (int)(wk_pairs * (wk_xcd + 1) / 8);
    const int wk_J = wk_hi > wk_lo ? (wk_hi - wk_lo + 7) / 8 : 0;
    const int qend = WALK ? (int)blockIdx.x + wk_J * G : ntiles;  // this workgroup's tiles: q = blockIdx.x + j G < qend
    auto origin = [&](int q, int64_t& m0, int64_t& n0) {
        if constexpr (WALK) {
            const int pp = wk_lo + 8 * ((q - (int)blockIdx.x) / G);
            const int cg = pp / p.tiles_m;
            m0 = (int64_t)(pp - cg * p.tiles_m) * T::BM;
            n0 = (int64_t)(cg * 4 + wk_ci) * T::BN;
            return;
        }
        const int pid = xcd_chunked(q, ntiles);
        constexpr int GROUP_M = 6;
        const int in_group = GROUP_M * p.tiles_n;
        const int first_m = (pid / in_group) * GROUP_M;
        const int gsz = min(p.tiles_m - first_m, GROUP_M);
        m0 = (int64_t)(first_m + (pid % in_group) % gsz) * T::BM;
        n0 = (int64_t)((pid % in_group) / gsz) * T::BN;
    };
    // ---- the request side of the stream: tile qi, K-tile ti, element number si (stage si & 1).  The LDS-DMA requests of a SIMD's two waves (w and w + 4) are divided by
    // OPERAND, not by wave: wave w requests the A-panel pieces of both (8 per K-tile), right behind the barrier that frees the stage; wave w + 4 requests the B-panel
    // pieces of both (weights: they come from L2) a phase later, under its partner's MFMAs.  Issued symmetrically (every wave its own 4 + 4 behind the barrier), both waves
    // of a SIMD stand in the CU's one address unit's queue at the same time and the matrix pipe idles; with the two request bursts half a K-tile apart, one wave of every
    // SIMD always multiplies.  (All 16 requests on wave w, none on w + 4: between the two -- the requesting wave's burst plus its own 64 MFMAs is the K-tile's critical path.)
    // The SwiGLU-backward form keeps all 16 requests on wave w (BY_OPERAND false): with the second request point in the K-tile its register allocation spills 72 values.
    constexpr bool BY_OPERAND = KIND != MI355_EPI_SWIGLU_BWD;
    const bool a_side = wave < 4;
    const int wlo = wave & 3;
    unsigned voff[2 * T::A_PPW];  // this wave's operand: pieces of waves wlo (0-3) and wlo + 4 (4-7)
    [[maybe_unused]] unsigned voff2[2 * T::B_PPW];  // !BY_OPERAND: wave w's B-panel pieces
    static_assert(T::A_PPW == T::B_PPW, "one offset array serves either operand");
    const bf16_t* baseX = p.A;
    [[maybe_unused]] const bf16_t* baseY = p.B;
    auto plan = [&](int q) {
        int64_t m0, n0;
        origin(q, m0, n0);
        int l = lane;
        asm volatile("" : "+v"(l));  // recomputed from the lane number once per tile: hoisted, the per-piece rows and chunks would occupy 16 registers across the main loop
        if (a_side) {  // (wave-uniform)
            baseX = uniform_ptr(p.A + m0 * p.lda);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                unsigned v[T::A_PPW];
                int unused[T::A_PPW];
                piece_offsets<false, T::BM, BK, T::A_PPW>(wlo + 4 * h, l, p.lda, p.M - m0, v, unused);
#pragma unroll
                for (int j = 0; j < T::A_PPW; ++j) voff[h * T::A_PPW + j] = v[j];
                if constexpr (!BY_OPERAND) {
                    piece_offsets<false, T::BN, BK, T::B_PPW>(wlo + 4 * h, l, p.ldb, p.N - n0, v, unused);
#pragma unroll
                    for (int j = 0; j < T::B_PPW; ++j) voff2[h * T::B_PPW + j] = v[j];
                }
            }
            if constexpr (!BY_OPERAND) baseY = uniform_ptr(p.B + n0 * p.ldb);
        } else if constexpr (BY_OPERAND) {
            baseX = KIND == MI355_EPI_SWIGLU_FWD ? uniform_ptr(p.B) : uniform_ptr(p.B + n0 * p.ldb);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int w = wlo + 4 * h;
                unsigned v[T::B_PPW];
                if constexpr (KIND == MI355_EPI_SWIGLU_FWD) {
                    // every 64 output columns of the tile are [32 lin1 rows | the 32 lin_gate rows of the SAME hidden units] of the fused weight (see gemm_tile)
                    const int64_t nh = p.N >> 1;
#pragma unroll
                    for (int j = 0; j < T::B_PPW; ++j) {
                        const int r = (w * T::B_PPW + j) * 8 + l / 8;
                        const int c = swz_rowk<BK>(l % 8, r);
                        const int64_t hid = (n0 >> 1) + (r >> 6) * 32 + (r & 31);
                        v[j] = hid < nh ? (unsigned)((((r >> 5) & 1) * nh + hid) * p.ldb * 2 + c * 16) : OOB;
                    }
                } else {
                    int unused[T::B_PPW];
                    piece_offsets<false, T::BN, BK, T::B_PPW>(w, l, p.ldb, p.N - n0, v, unused);
                }
#pragma unroll
                for (int j = 0; j < T::B_PPW; ++j) voff[h * T::B_PPW + j] = v[j];
            }
        }
    };
    int qi = blockIdx.x, ti = 0, si = 0;
    auto request_next = [&]() {  // this wave's operand of element si
        if (qi < qend) {
            char* dst = smem + (si & 1) * T::STAGE + (a_side ? 0 : T::A_BYTES) + wlo * T::A_PPW * 1024;
            const bf16_t* px = baseX + (int64_t)ti * BK;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < T::A_PPW; ++j) dma_piece(px, voff[h * T::A_PPW + j], dst + (h * 4 * T::A_PPW + j) * 1024);
            if constexpr (!BY_OPERAND) {
                const bf16_t* py = baseY + (int64_t)ti * BK;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int j = 0; j < T::B_PPW; ++j) dma_piece(py, voff2[h * T::B_PPW + j], dst + T::A_BYTES + (h * 4 * T::B_PPW + j) * 1024);
            }
            if (++ti == nt) {
                ti = 0;
                qi += G;
                if (qi < qend) plan(qi);
            }
        }
        ++si;
    };

    int qc = blockIdx.x, sc = 0;  // the multiplying side: tile qc, element number sc
    if (qc >= qend) return;
    plan(qi);
    f32x4 acc[T::FM][T::FN];
    bf16x8 aE[HM], aO[HM], b0[T::FN], b1[T::FN];
    auto loadA = [&](bf16x8 (&a)[HM], const char* sA, int kk, int mh) {
#pragma unroll
        for (int i = 0; i < HM; ++i) a[i] = frag_rowk<BK>(sA, wr0 + (mh * HM + i) * 16, kk, lane);
    };
    auto loadB = [&](bf16x8 (&b)[T::FN], const char* sB, int kk) {
#pragma unroll
        for (int j = 0; j < T::FN; ++j) b[j] = frag_rowk<BK>(sB, wc0 + j * 16, kk, lane);
    };
    // B fragment first: the lane holds C[row lane & 15][4 (lane >> 4) + e].  ZERO: the tile's first k-step starts from the constant 0 (no accumulator is cleared anywhere)
    auto mma = [&](bool zero, const bf16x8 (&a)[HM], const bf16x8 (&b)[T::FN], int mh) {
        if (zero) {  // wave-uniform
#pragma unroll
            for (int i = 0; i < HM; ++i)
#pragma unroll
                for (int j = 0; j < T::FN; ++j) acc[mh * HM + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < HM; ++i)
#pragma unroll
                for (int j = 0; j < T::FN; ++j) acc[mh * HM + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[mh * HM + i][j], 0, 0, 0);
        }
    };
    bool more_tiles = false;
    auto kstep = [&](int t) {  // one element of the stream: 64 MFMAs in four phases (k-step, row half), the next element's first fragments requested under the last
        const char* sA = smem + (sc & 1) * T::STAGE;
        const char* sB = sA + T::A_BYTES;
        loadA(aO, sA, 0, 1);
        mma(t == 0, aE, b0, 0);
        if (BY_OPERAND && !a_side && sc > 0) request_next();  // the B panels of element sc + 1 (its A panels were requested behind the last barrier; elements 0 and 1: before the loop)
        loadB(b1, sB, 1);
        loadA(aE, sA, 1, 0);
        mma(t == 0, aO, b0, 1);
        loadA(aO, sA, 1, 1);
        mma(false, aE, b1, 0);
        const bool last = t + 1 == nt;
        if (!last || more_tiles) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's reads of the element are complete ...
            wait_vmcnt<0>();                                    // ... its share of the next element has landed (and the previous tile's stores have retired)
            __builtin_amdgcn_s_barrier();                       // ... for every wave
            if (a_side) request_next();                         // the A panels of element sc + 2 into the stage just left: at the end of a tile that is the NEXT tile's stream
            if (!last) {
                const char* nA = smem + ((sc + 1) & 1) * T::STAGE;
                loadB(b0, nA + T::A_BYTES, 0);
                loadA(aE, nA, 0, 0);
            }
        }
        mma(false, aO, b1, 1);
        ++sc;
    };
    if (BY_OPERAND || a_side) request_next();  // elements 0 and 1: both operands
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    if (BY_OPERAND || a_side) request_next();
    loadB(b0, smem + T::A_BYTES, 0);
    loadA(aE, smem, 0, 0);
    for (;;) {
        more_tiles = qc + G < qend;
        for (int t = 0; t < nt; ++t) kstep(t);
        // ---- write-out of tile qc: 4 sub-blocks of 32 rows x 64 columns per wave; packed bf16 through this wave's own 4 KiB.  LDS operations of a wave execute in
        // order, so sub-block sb + 1 is staged right behind the row reads of sub-block sb, whose stores go out while it is being packed; rows and columns beyond the
        // matrix are dropped by the buffer range check (offset OOB), so the passes have no branches.
        int le = lane;
        asm volatile("" : "+v"(le));  // derived per tile, not kept across the main loop
        const int g = le >> 4, r16 = le & 15;
        // staging addresses of this lane.  Write side: row r = ii * 16 + r16 of a 32 x 64 sub-block (128-byte rows), 16-byte chunk (2 j + g / 2) ^ (r & 7), 8-byte half
        // (g & 1) ^ (r >> 3 & 1): the 16 rows one store instruction covers hit 32 distinct banks.  Read side: row pass * 8 + lane / 8, chunk (lane & 7) ^ (row & 7).
        const int wr_off = r16 * 128 + ((((g & 1) ^ (r16 >> 3)) & 1) << 3), wr_x = r16 & 7;
        const int rd_row = le >> 3, rd_ch = le & 7;
        const int rd_off = rd_row * 128 + ((rd_ch ^ (rd_row & 7)) << 4);  // (pass * 8 + rd_row) & 7 == rd_row & 7
        int64_t m0, n0;
        origin(qc, m0, n0);
        const int64_t rows_left = p.M - m0 - wr0;
        u32x4 rd[4];
        [[maybe_unused]] u32x2 rres[2][T::FN];   // RES: the residual of a sub-block in the accumulators' layout (8-byte loads)
        [[maybe_unused]] u32x4 uv[4], gv[4];     // SwiGLU backward: the forward's gate-up pair of a sub-block's rows (16-byte loads)
        [[maybe_unused]] u32x2 partner[4];       // SwiGLU forward: the other operand of the four units this lane activates
        [[maybe_unused]] float psum[4][4];       // attention delta: this wave's half-head row sums (sub-block, pass), complete in every lane of the row's eight
        const int hi4 = rd_ch >> 2;
        // column base of this wave in C (and R), validity of this lane's 8 columns
        int64_t cbase, cbase2 = 0;
        bool col_ok;
        if constexpr (KIND == MI355_EPI_SWIGLU_FWD) {
            const int64_t nh = p.N >> 1, hid = (n0 >> 1) + (wc0 >> 6) * 32 + (rd_ch & 3) * 8;
            col_ok = hid < nh;
            cbase = (hi4 ? nh : 0) + hid;  // gate-up output: u into [:, hid], g into [:, N/2 + hid]
            cbase2 = hid + 4 * hi4;        // activation output (R): four units per lane
        } else {
            cbase = n0 + wc0 + rd_ch * 8;
            col_ok = cbase < p.N;
        }
        auto rsrc_c = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<bf16_t*>(p.C) + (m0 + wr0) * p.ldc, 0, 0x7fffffff, 0x00020000);
        auto rsrc_r = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(reinterpret_cast<const bf16_t*>(p.R)) + (m0 + wr0) * p.ldr, 0, 0x7fffffff, 0x00020000);
        auto fetch_res = [&](int sb) {  // residual of sub-block sb, requested a sub-block before it is packed
            if constexpr (RES) {
#pragma unroll
                for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                    for (int j = 0; j < T::FN; ++j) {
                        const int row = sb * 32 + ii * 16 + r16;
                        const int64_t col = n0 + wc0 + j * 16 + 4 * g;
                        rres[ii][j] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc_r, (row < rows_left && col < p.N) ? (unsigned)((row * p.ldr + col) * 2) : OOB, 0, 0));
                    }
            }
        };
        auto fetch_ug = [&](int sb) {  // gate-up rows of sub-block sb, requested when it is staged, used a sub-block later (after the stores of sb - 1 have consumed theirs)
            if constexpr (KIND == MI355_EPI_SWIGLU_BWD || KIND == MI355_EPI_ATTN_DELTA) {
#pragma unroll
                for (int pass = 0; pass < 4; ++pass) {
                    const int row = sb * 32 + pass * 8 + rd_row;
                    const bool ok = col_ok && row < rows_left;
                    uv[pass] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, ok ? (unsigned)((row * p.ldr + cbase) * 2) : OOB, 0, 0));  // delta: the forward's ctx
                    if constexpr (KIND == MI355_EPI_SWIGLU_BWD)
                        gv[pass] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, ok ? (unsigned)((row * p.ldr + cbase + p.N) * 2) : OOB, 0, 0));
                }
            }
        };
        auto stores = [&](int sb) {
#pragma unroll
            for (int pass = 0; pass < 4; ++pass) {
                const u32x4 o = (pass & 1) ? (u32x4){rd[pass][2], rd[pass][3], rd[pass][0], rd[pass][1]} : rd[pass];  // rows 8-15 of a 16-row tile were written with their halves exchanged
                const int row = sb * 32 + pass * 8 + rd_row;
                const bool ok = col_ok && row < rows_left;
                if constexpr (KIND == MI355_EPI_SWIGLU_BWD) {
                    // o = d(act) of hidden units cbase..+7, rounded to bf16: d(gate-up) = [d * g sig(g) | d * u sig(g) (1 + g (1 - sig(g)))] into C[:, unit], C[:, N + unit] (ldc = 2N)
                    u32x4 o0, o1;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float du[2], dg[2];
#pragma unroll
                        for (int hlf = 0; hlf < 2; ++hlf) {
                            const float d_ = hlf ? __uint_as_float(o[e] & 0xffff0000u) : __uint_as_float(o[e] << 16);
                            const float u_ = hlf ? __uint_as_float(uv[pass][e] & 0xffff0000u) : __uint_as_float(uv[pass][e] << 16);
                            const float g_ = hlf ? __uint_as_float(gv[pass][e] & 0xffff0000u) : __uint_as_float(gv[pass][e] << 16);
                            swiglu_grads(d_, u_, g_, du[hlf], dg[hlf]);
                        }
                        o0[e] = pack_bf2(du[0], du[1]);
                        o1[e] = pack_bf2(dg[0], dg[1]);
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(o0, rsrc_c, ok ? (unsigned)((row * p.ldc + cbase) * 2) : OOB, 0, CAUX);
                    __builtin_amdgcn_raw_buffer_store_b128(o1, rsrc_c, ok ? (unsigned)((row * p.ldc + cbase + p.N) * 2) : OOB, 0, CAUX);
                } else {
                    __builtin_amdgcn_raw_buffer_store_b128(o, rsrc_c, ok ? (unsigned)((row * p.ldc + cbase) * 2) : OOB, 0, CAUX);
                    if constexpr (KIND == MI355_EPI_ATTN_DELTA) {
                        // o = d(ctx), rounded; uv = ctx: the row's dot product over this lane's 8 columns, folded over the row's eight lanes = half a head (the wave's 64 columns)
                        float dsum = 0.f;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            dsum += __uint_as_float(o[e] << 16) * __uint_as_float(uv[pass][e] << 16) + __uint_as_float(o[e] & 0xffff0000u) * __uint_as_float(uv[pass][e] & 0xffff0000u);
                        dsum += __shfl_xor(dsum, 1, 64);
                        dsum += __shfl_xor(dsum, 2, 64);
                        dsum += __shfl_xor(dsum, 4, 64);
                        psum[sb][pass] = dsum;
                    }
                    if constexpr (KIND == MI355_EPI_SWIGLU_FWD) {
                        // this lane's 8 columns are u (chunks 0-3) or g (chunks 4-7) of 8 hidden units; it activates four of them: units 0-3 (u lanes) resp. 4-7 (g lanes),
                        // the other operand = the partner lane's chunk, read back from the staging rows; a = u * silu(g) on the ROUNDED operands, as mi355_swiglu_fwd sees them
                        // (operands are picked with selects, word by word: written as `hi4 ? act(other, mine) : act(mine, other)` on an indexed `o[2 * hi4 + ..]`, every lane
                        // ran both sides of a divergent branch -- twice the exponentials -- behind a chain of compares for the index)
                        const u32x2 pv = partner[pass];
                        const unsigned own0 = hi4 ? o[2] : o[0], own1 = hi4 ? o[3] : o[1];
                        const unsigned uw[2] = {hi4 ? pv[0] : own0, hi4 ? pv[1] : own1}, gw[2] = {hi4 ? own0 : pv[0], hi4 ? own1 : pv[1]};
                        float a4[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float u_ = (e & 1) ? __uint_as_float(uw[e >> 1] & 0xffff0000u) : __uint_as_float(uw[e >> 1] << 16);
                            const float g_ = (e & 1) ? __uint_as_float(gw[e >> 1] & 0xffff0000u) : __uint_as_float(gw[e >> 1] << 16);
                            a4[e] = swiglu_act(u_, g_);
                        }
                        const u32x2 av = {pack_bf2(a4[0], a4[1]), pack_bf2(a4[2], a4[3])};
                        __builtin_amdgcn_raw_buffer_store_b64(av, rsrc_r, ok ? (unsigned)((row * p.ldr + cbase2) * 2) : OOB, 0, 0);
                    }
                }
            }
        };
        fetch_res(0);
#pragma unroll
        for (int sb = 0; sb < 4; ++sb) {
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < T::FN; ++j) {
                    f32x4 v = acc[sb * 2 + ii][j];
                    if constexpr (RES) {
                        v[0] += __uint_as_float(rres[ii][j][0] << 16);
                        v[1] += __uint_as_float(rres[ii][j][0] & 0xffff0000u);
                        v[2] += __uint_as_float(rres[ii][j][1] << 16);
                        v[3] += __uint_as_float(rres[ii][j][1] & 0xffff0000u);
                    }
                    const u32x2 pk = {pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])};
                    *reinterpret_cast<u32x2*>(stg + ii * 2048 + wr_off + (((2 * j + (g >> 1)) ^ wr_x) << 4)) = pk;
                }
            if (sb > 0) stores(sb - 1);
            if (sb < 3) fetch_res(sb + 1);
            fetch_ug(sb);
#pragma unroll
            for (int pass = 0; pass < 4; ++pass) {
                rd[pass] = *reinterpret_cast<const u32x4*>(stg + pass * 1024 + rd_off);
                if constexpr (KIND == MI355_EPI_SWIGLU_FWD) {
                    // partner chunk rd_ch ^ 4 of the same row, its half hi4 (units 4-7 of the partner's eight for g lanes, 0-3 for u lanes); odd passes hold rows whose halves are exchanged
                    const int prow = rd_row;  // (pass * 8 + rd_row) & 7
                    partner[pass] = *reinterpret_cast<const u32x2*>(stg + pass * 1024 + rd_row * 128 + ((((rd_ch ^ 4) ^ (prow & 7))) << 4) + (((hi4 ^ pass) & 1) << 3));
                }
            }
        }
        stores(3);
        if constexpr (KIND == MI355_EPI_ATTN_DELTA) {
            // a head's two halves sit in two neighbouring waves: every wave parks its 128 row sums in its own staging region (behind its last row reads: LDS operations
            // execute in order), one barrier, then one thread per (row, head) adds the halves in a fixed order and writes the attention backward's three row constants.
            // The regions are next written in the following tile's write-out, which every wave reaches only through that tile's K-loop barriers.
            static_assert(T::NTHREADS == 512 && T::WN == 4 && T::WTN == 64, "delta write-out: 2 x 4 waves of 128 x 64 on a 256 x 256 tile");
            float* part = reinterpret_cast<float*>(stg);
#pragma unroll
            for (int sb = 0; sb < 4; ++sb)
#pragma unroll
                for (int pass = 0; pass < 4; ++pass)
                    if (rd_ch == 0) part[sb * 32 + pass * 8 + rd_row] = psum[sb][pass];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            const int t_ = threadIdx.x, row = t_ & 255, hsel = t_ >> 8;
            const float* p0 = reinterpret_cast<const float*>(smem + 2 * T::STAGE + ((row >> 7) * 4 + 2 * hsel) * 4096);
            const float sum = p0[row & 127] + p0[1024 + (row & 127)];
            const int64_t gm = m0 + row, head = (n0 >> 7) + hsel;
            if (gm < p.M && head < p.ad_Hq) {
                const int64_t bb = gm / p.ad_S, sq = gm - bb * p.ad_S;
                const int64_t di = (bb * p.ad_Hq + head) * p.ad_S + sq;
                p.ad_delta[di] = sum;
                p.ad_ndl[di] = -sum;
                p.ad_nl2[di] = -p.ad_lse[di] * 1.4426950408889634f;
            }
        }
        qc += G;
        if (qc >= qend) break;
        const char* nA = smem + (sc & 1) * T::STAGE;
        loadB(b0, nA + T::A_BYTES, 0);
        loadA(aE, nA, 0, 0);
    }
}

int launch_persist(GemmParams p, hipStream_t s) {
    using T = Cfg256;
    p.tiles_m = (int)((p.M + T::BM - 1) / T::BM);
    p.tiles_n = (int)((p.N + T::BN - 1) / T::BN);
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
    MI355_REQUIRE(tiles < 0x7fffffffLL / 16, "mi355_gemm_bf16: grid too large");
    const dim3 grid((unsigned)(tiles < 256 ? tiles : 256)), block(T::NTHREADS);  // one workgroup per CU
#define PERSIST_LAUNCH(KIND_, RES_, WALK_) hipLaunchKernelGGL((gemm_nt_persist_kernel<KIND_, RES_, WALK_>), grid, block, 0, s, p, (int)tiles)
    if (p.epilogue == MI355_EPI_SWIGLU_FWD) PERSIST_LAUNCH(MI355_EPI_SWIGLU_FWD, false, false);
    else if (p.epilogue == MI355_EPI_SWIGLU_BWD) PERSIST_LAUNCH(MI355_EPI_SWIGLU_BWD, false, false);
    else if (p.epilogue == MI355_EPI_ATTN_DELTA) PERSIST_LAUNCH(MI355_EPI_ATTN_DELTA, false, false);
    else if (p.R) PERSIST_LAUNCH(MI355_EPI_NONE, true, false);
    else if (p.N > 32768 && tiles >= 256) PERSIST_LAUNCH(MI355_EPI_NONE, false, true);
    else PERSIST_LAUNCH(MI355_EPI_NONE, false, false);
#undef PERSIST_LAUNCH
    MI355_LAUNCH_CHECK("mi355_gemm_bf16(persistent)");
    return 0;
}
