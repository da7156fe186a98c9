// Products on 256x256 tiles by four waves of 128x128 outputs each (included by gemm.hip).
//
// What bounds it: the matrix pipe under the board's power cap (8 192^3: 1 590 TFLOP/s on random operands, 2 040 on zeros), and beside short sums the result's way to memory.  Eight waves of 128x64 on the
// same tile (gemm_tile) read 96 + 96 KiB of fragments a K-tile of 64 where 64 + 64 are enough here, drain their requests once a K-tile and reached 1 306 / 1 420; four waves on K-tiles of 32 (Cfg256w) fetch
// half lines, 1 269 / 1 464.
//   * One wave per SIMD: 256 accumulators in the accumulation registers (products from asm: left to itself the compiler moves part of them), two halves of either operand's fragments in the others.
//   * A stage (64 KiB, two of them) is four panels of 128 rows x 64: A0, A1, B0, B1.  A wave's 128x128 outputs are four quadrants of 64x64, a K-tile four phases of 32 products in the order (A0 B0),
//     (A0 B1), (A1 B1), (A1 B0): each phase needs one fragment half that the one before it did not have, 8 reads, and reads it one phase ahead.  A panel's place is free as soon as its fragments are
//     read, so the request for the same panel two K-tiles on goes out there: 5 - 6 phases (1.7 - 2.1 us) in front of its use, four of them a phase, and the wait is a counted one that leaves 16 in flight.
//   * Two barriers a K-tile.  Behind the one after phase 2 the places of A0, B0 (read in phases 3 and 4 of the K-tile before) hold the next K-tile for every wave; behind the one after phase 4 those
//     of B1, A1 do.  Requests of phases 1, 2 (3, 4) go into places whose last reads lie in front of the barrier before them.
//   * The stream of K-tiles runs on over a workgroup's tiles: while one is written out the next one's first two K-tiles are under way.
//   * Edges: rows (NT) or K (TN) past the end lie beyond num_records of the stream's buffer descriptor, columns (TN) past the end get the offset OOB: both load zeros.  An odd number of
//     K-tiles is made even by one of zeros.
//   * NN: A as in the NT form, B's panels as in the TN form, fragments by transposing reads.  us, copy of the weight + NT -> NN: 16 384 x 1 024, K = 3 072 78.7 -> 73.6, 6 144 146 -> 140.5; 5 664 x 3 584,
//     K = 1 024 60 -> 50; eight waves' tile -> here in shares of K: 602 x 1 024, K = 151 936 292 -> 182, 1 300 x 1 024, K = 20 032 90 -> 63.
//   * Write-out from the registers: B's fragment is the product's first operand, so a lane holds four consecutive columns of a row; v_permlane16_swap makes eight of them, a rotation by eight lanes makes
//     whole rows of 128 bytes, and no LDS is touched.  Whole lines with the non-temporal hint leave the L2 to the operands: 16 384 x 4 096, K = 1 024 107.0 -> 103.9 us (segments of 64 bytes 109.7).
//     Rows that start inside a line (a pitch or a corner that is no multiple of 128 bytes) go without it: two waves' parts of a line meet in the L2.  us, with it -> without: 12 288 x 5 000, K = 1 024 132 -> 103,
//     17 016 x 2 056 in fp32, K = 512 89 -> 56, 8 224 x 3 080 in fp32 from 640 tokens 60 -> 49.
//     (Beside the products of the last and the next K-tile instead of between them: level.  Stores left out: 91.8.)
// The sum of every output runs over K in the order of gemm_tile's: the same bits.

constexpr int QUAD_RES = 16, QUAD_BIAS = 32;  // added to KIND (MI355_EPI_NONE): residual, bias
constexpr int QUAD_SPLIT = 64;                // alone: p.ksplit shares of K, each with its own fp32 [M, N] of p.ws (splitk_reduce_kernel adds them up)

// q, q + G, ... < ntiles: the tiles (SPLIT: and shares of K, those of one share after each other) of this workgroup (CHUNK: in a numbering that deals them over the XCDs).  FORM: which operands are K-strided, none (NT), B (NN) or both (TN).  More than three K-tiles.
template <int FORM, int OUT_DT, int KIND_, bool CHUNK = true>
__device__ __forceinline__ void quad_tiles(const GemmParams& p, int q, const int G, const int ntiles, char* smem) {
    constexpr int KIND = KIND_ & 15, ADD = KIND_ & ~15;
    constexpr bool TA = FORM == MI355_GEMM_TN, TB = FORM != MI355_GEMM_NT;
    static_assert(!TB || KIND != MI355_EPI_SWIGLU_FWD);
    constexpr bool B16 = OUT_DT == MI355_DT_BF16, SPLIT = ADD == QUAD_SPLIT;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int nt_all = (int)((p.K + 63) >> 6), nt_even = nt_all + (nt_all & 1), per = SPLIT ? (int)quad_share(p.K, p.ksplit) : 0;
    constexpr int ESZ = B16 ? 2 : 4;

    // tile number -> its corner and first K-tile: XCD-chunked, row groups under every column panel (six NT and NN, three TN: see gemm_tile)
    auto origin = [&](int t, int& m0, int& n0, int& k0) {
        constexpr int GROUP_M = TA ? 3 : 6;
        int pid = CHUNK ? xcd_chunked(t, ntiles) : t;
        k0 = 0;
        if constexpr (SPLIT) {
            const int tiles = p.tiles_m * p.tiles_n, share = pid / tiles;
            pid -= share * tiles, k0 = share * per;
        }
        const int in_group = GROUP_M * p.tiles_n, first_m = (pid / in_group) * GROUP_M, gsz = min(p.tiles_m - first_m, GROUP_M);
        m0 = (first_m + (pid % in_group) % gsz) * 256;
        n0 = ((pid % in_group) / gsz) * 256;
    };

    // ---- requests: a wave asks for four of a panel's sixteen KiB.  A panel's rows (NT; TN: columns) r are the tile's (r / 64) 128 + 64 h + r % 64: a wave's 128 are 64 of panel 0 and 64 of panel 1.
    // SwiGLU forward: B0 holds 128 rows of lin1, B1 the lin_gate rows of the same units, so that a lane holds both operands of an activation.
    unsigned vA[2][4], vB[2][4];
    auto plan = [&](int m0, int n0) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // K-strided: [64 k][128 columns], swizzled as in piece_offsets
                const int k = wave * 16 + j * 4 + (lane >> 4), ck = (lane & 15) ^ (tr_f(k) << 1), col = (ck >> 3) * 128 + h * 64 + (ck & 7) * 8;
                // K-contiguous: [128 rows][64 k]
                const int r = wave * 32 + j * 8 + (lane >> 3), c = swz_rowk<64>(lane & 7, r) * 16, row = (r >> 6) * 128 + h * 64 + (r & 63);
                if constexpr (TA) vA[h][j] = col < p.M - m0 ? (unsigned)((k * p.lda + col) * 2) : OOB;
                else vA[h][j] = (unsigned)(row * p.lda * 2 + c);
                if constexpr (TB) vB[h][j] = col < p.N - n0 ? (unsigned)((k * p.ldb + col) * 2) : OOB;
                else vB[h][j] = (unsigned)((KIND == MI355_EPI_SWIGLU_FWD ? h * (p.N >> 1) + r : row) * p.ldb * 2 + c);
            }
    };
    const char *baseA, *baseB;  // the K-tile requested next, its number, its buffers' sizes (K-contiguous: to the end of the tile's last row; K-strided: of the K-tile's last row)
    int kreq = 0, recA = 0, recB = 0;
    int tailA = 0, tailB = 0;
    const int tail_at = TA && (p.K & 63) ? nt_all - 1 : -1;  // the K-tile that K ends in
    const int64_t stepA = TA ? 128 * p.lda : 128, stepB = TB ? 128 * p.ldb : 128;
    auto open = [&](int m0, int n0, int k0) {
        kreq = k0;
        const int64_t bn0 = KIND == MI355_EPI_SWIGLU_FWD ? n0 >> 1 : n0;
        baseA = (const char*)uniform_ptr(TA ? p.A + m0 : p.A + m0 * p.lda), baseB = (const char*)uniform_ptr(TB ? p.B + n0 : p.B + bn0 * p.ldb);
        recA = (int)(TA ? 128 * p.lda : min((int64_t)256, p.M - m0) * p.lda * 2);
        recB = (int)(TB ? 128 * p.ldb : (KIND == MI355_EPI_SWIGLU_FWD ? p.N - bn0 : min((int64_t)256, p.N - bn0)) * p.ldb * 2);
        if constexpr (TA) tailA = (int)(((p.K & 63) * p.lda - m0) * 2), tailB = (int)(((p.K & 63) * p.ldb - n0) * 2);
        if constexpr (TB) plan(m0, n0);
        if constexpr (SPLIT) baseA += k0 * stepA, baseB += k0 * stepB;
    };
    auto advance = [&]() {
        ++kreq;
        baseA += stepA, baseB += stepB;
    };
    auto request = [&](int stage, int panel, int j) {  // panels 0, 1: A0, A1; 2, 3: B0, B1
        const int rec = TA && kreq == tail_at ? (panel < 2 ? tailA : tailB) : panel < 2 ? recA : recB;
        dma_piece(panel < 2 ? baseA : baseB, panel < 2 ? vA[panel & 1][j] : vB[panel & 1][j], smem + stage * QUAD_STAGE + panel * QUAD_PANEL + wave * 4096 + j * 1024, kreq < nt_all ? rec : 0);
    };

    // ---- fragments: fa, fb[panel or register set][k-step][16 rows]
    bf16x8 fa[2][2][4], fb[2][2][4];
    const int r16 = lane & 15;
    const int off0 = r16 * 128 + (swz_rowk<64>(lane >> 4, r16) << 4);  // the swizzle of a row goes by its last four bits: one lane offset a k-step serves every fragment
    [[maybe_unused]] unsigned offA[4], offB[4];
    if constexpr (TB) {  // the XOR of a lane's row reaches into the column bits: one lane offset per column tile (frag_tr)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int g = lane >> 4, kq = (lane >> 2) & 3, fx = (kq | ((g & 1) << 2)) << 1, row = (8 * g + kq) * 256 + (lane & 1) * 8;
            offA[i] = (unsigned)(uintptr_t)LDS_PTR(smem) + row + (((wm * 8 + 2 * i + ((lane & 3) >> 1)) ^ fx) << 4);
            offB[i] = (unsigned)(uintptr_t)LDS_PTR(smem) + row + (((wn * 8 + 2 * i + ((lane & 3) >> 1)) ^ fx) << 4);
        }
    }
    TrHalves halves[2][4];
    auto read_frag = [&](bf16x8 (&f)[2][4], auto stage_c, auto panel_c, int n) __attribute__((always_inline)) {  // n: 4 k-step + row tile
        TrHalves(&h)[2][4] = halves;
        constexpr int STAGE = decltype(stage_c)::value, PANEL = decltype(panel_c)::value;
        const int kk = n >> 2, i = n & 3;
        if constexpr (PANEL < 2 ? TA : TB) {
            const unsigned addr = (PANEL < 2 ? offA[i] : offB[i]) + STAGE * QUAD_STAGE;
            if (kk == 0) asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%c3\n\tds_read_b64_tr_b16 %1, %2 offset:%c4" : "=&v"(h[0][i].lo), "=&v"(h[0][i].hi) : "v"(addr), "i"(PANEL * QUAD_PANEL), "i"(PANEL * QUAD_PANEL + 1024));
            else asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%c3\n\tds_read_b64_tr_b16 %1, %2 offset:%c4" : "=&v"(h[1][i].lo), "=&v"(h[1][i].hi) : "v"(addr), "i"(PANEL * QUAD_PANEL + 8192), "i"(PANEL * QUAD_PANEL + 9216));
        } else {
            f[kk][i] = *reinterpret_cast<const bf16x8*>(smem + STAGE * QUAD_STAGE + PANEL * QUAD_PANEL + (PANEL < 2 ? wm : wn) * 8192 + i * 2048 + (off0 ^ (kk * 64)));
        }
    };
    auto join = [&](bf16x8 (&f)[2][4], auto panel_c) __attribute__((always_inline)) {  // a K-strided panel's reads: waits for those of a phase
        if constexpr (decltype(panel_c)::value < 2 ? TA : TB) {
            TrHalves(&h)[2][4] = halves;
            asm volatile("s_waitcnt lgkmcnt(0)" : TRH(h[0][0]), TRH(h[0][1]), TRH(h[0][2]), TRH(h[0][3]), TRH(h[1][0]), TRH(h[1][1]), TRH(h[1][2]), TRH(h[1][3])::"memory");
#pragma unroll
            for (int n = 0; n < 8; ++n) f[n >> 2][n & 3] = tr_join(h[n >> 2][n & 3]);
        }
    };
    using std::integral_constant;
    using I0 = integral_constant<int, 0>;
    using I1 = integral_constant<int, 1>;
    using I2 = integral_constant<int, 2>;
    using I3 = integral_constant<int, 3>;

    f32x4 acc[2][2][4][4];  // [A half][B half][row tile][column tile]
    // 32 products of a quadrant; a read behind each of the first eight, a request in every quarter.  WAIT >= 0: the barrier behind it, with that many of this wave's requests and stores in flight
    auto phase = [&](auto first_c, f32x4 (&c)[4][4], const bf16x8 (&a)[2][4], const bf16x8 (&b)[2][4], bf16x8 (&next)[2][4], auto rstage, auto rpanel, int qstage, int qpanel, auto wait_c) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value;
        constexpr int WAIT = decltype(wait_c)::value;
#pragma unroll
        for (int s = 0; s < 32; ++s) {
            const int kk = s >> 4, i = (s >> 2) & 3, j = s & 3;
            if (FIRST && kk == 0) quad_mma_first(c[i][j], a[kk][i], b[kk][j]);
            else quad_mma(c[i][j], a[kk][i], b[kk][j]);
            if ((s & 1) == 0 && s < 16) read_frag(next, rstage, rpanel, s >> 1);
            if ((s & 7) == 5) request(qstage, qpanel, s >> 3);
            __builtin_amdgcn_sched_barrier(0);
        }
        join(next, rpanel);
        if constexpr (WAIT >= 0) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WAIT) : "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // K-tile t in stage PAR = t & 1; its requests are K-tile t + 2's.  B0's fragments are in set PAR, B1's come into the other one
    auto ktile = [&](auto par, auto first_c, auto wait_c) __attribute__((always_inline)) {
        constexpr int S = decltype(par)::value;
        using Here = integral_constant<int, S>;
        using There = integral_constant<int, S ^ 1>;
        using None = integral_constant<int, -1>;
        phase(first_c, acc[0][0], fa[0], fb[S], fb[S ^ 1], Here{}, I3{}, S, 0, None{});
        phase(first_c, acc[0][1], fa[0], fb[S ^ 1], fa[1], Here{}, I1{}, S, 2, wait_c);
        phase(first_c, acc[1][1], fa[1], fb[S ^ 1], fa[0], There{}, I0{}, S, 3, None{});
        phase(first_c, acc[1][0], fa[1], fb[S], fb[S ^ 1], There{}, I2{}, S, 1, wait_c);
        advance();
    };

    int m0, n0, k0;
    origin(q, m0, n0, k0);
    if constexpr (!TB) plan(m0, n0);
    open(m0, n0, k0);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
        for (int n = 0; n < 16; ++n) request(st, n < 4 ? 0 : n < 8 ? 2 : n < 12 ? 3 : 1, n & 3);
        advance();
    }
    asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int n = 0; n < 8; ++n) read_frag(fa[0], I0{}, I0{}, n);
    join(fa[0], I0{});
#pragma unroll
    for (int n = 0; n < 8; ++n) read_frag(fb[0], I0{}, I2{}, n);
    join(fb[0], I2{});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);

    // ---- write-out.  Eight rows x 128 bytes at a time: lane & 7 is the row; bf16: bits 3, 4, 5 of the lane are the columns' group of 32, of 16 and of 8 of a 64-column half; fp32: bit 3 the group of 16, bits 4
    // and 5 the groups of 4 of a 32-column quarter
    constexpr bool RES = ADD & QUAD_RES, BIAS = ADD & QUAD_BIAS, SW_FWD = KIND == MI355_EPI_SWIGLU_FWD, SW_BWD = KIND == MI355_EPI_SWIGLU_BWD, DELTA = KIND == MI355_EPI_ATTN_DELTA;
    constexpr int STORES = SW_FWD ? 48 : SW_BWD || !B16 ? 64 : 32;            // a wave's, at least
    constexpr int QW = B16 ? 1 : 2, WORDS = SW_BWD ? 2 : QW;                   // 16-byte groups of a lane's row of a half; those read with it
    constexpr int LOADS = RES || SW_BWD || DELTA ? 4 * WORDS : 0;              // of a block of 16 rows: residual (SwiGLU backward: the forward's [u | g]; attention delta: its ctx)
    [[maybe_unused]] u32x4 rv[2][2][2][WORDS];
    unsigned vc[2][QW], vr[2][QW];
    int ldc, ldr, rows;
    int64_t mw, nw;
    auto place = [&](int m, int n) {  // of the tile at (m, n): this wave's corner, its lanes' offsets
        int le = lane;
        asm volatile("" : "+v"(le));  // derived per tile, not kept across the products
        mw = m + wm * 128, nw = SW_FWD ? (n >> 1) + wn * 64 : n + wn * 128;
        rows = (int)max((int64_t)0, min((int64_t)128, p.M - mw));
        const int cols = (int)min((int64_t)128, (SW_FWD ? p.N >> 1 : p.N) - nw);
        ldc = (int)(SPLIT ? p.N : p.ldc) * ESZ, ldr = (int)p.ldr * ESZ;
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
#pragma unroll
            for (int w = 0; w < QW; ++w) {
                const int col = (SW_FWD ? 0 : hb * 64) + (B16 ? ((le >> 3) & 1) * 32 + ((le >> 4) & 1) * 16 + (le >> 5) * 8 : w * 32 + ((le >> 3) & 1) * 16 + (le >> 4) * 4);
                vc[hb][w] = col < cols ? (unsigned)((le & 7) * ldc + col * ESZ) : OOB;
                vr[hb][w] = col < cols ? (unsigned)((le & 7) * ldr + col * ESZ) : OOB;
            }
    };
    // rows past the end are beyond num_records
    auto corner_of = [&](const void* x, int64_t ld) { return (char*)uniform_ptr((const bf16_t*)((const char*)x + (mw * ld + nw) * ESZ)); };
    auto fetch = [&](int blk, bool res) __attribute__((always_inline)) {
        if constexpr (LOADS > 0) {
            const auto rr = __builtin_amdgcn_make_buffer_rsrc(corner_of(p.R, p.ldr), 0, res ? rows * ldr : 0, 0x00020000);
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                for (int half = 0; half < 2; ++half)
#pragma unroll
                    for (int w = 0; w < WORDS; ++w)
                        rv[blk & 1][hb][half][w] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rr, vr[hb][SW_BWD ? 0 : w] + (unsigned)((blk * 16 + half * 8) * ldr + (SW_BWD ? w * (int)p.N * 2 : 0)), 0, 0));
        }
    };
    auto corner_c = [&]() { return corner_of(SPLIT ? p.ws + (int64_t)(k0 / max(per, 1)) * p.M * p.N : p.C, SPLIT ? p.N : p.ldc); };
    auto write_out = [&](auto res_c) __attribute__((always_inline)) {  // (grouped: residual or none, every problem its own)
        constexpr bool ADD_R = decltype(res_c)::value;
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products' way through the pipe: the compiler does not know that the statements above are products (quad_value stays behind this one: both are volatile)
        const auto rc = __builtin_amdgcn_make_buffer_rsrc(corner_c(), 0, rows * ldc, 0x00020000);
        // non-temporal: whole lines only (SwiGLU: of both halves of C's columns)
        const bool whole = (((unsigned)(uintptr_t)corner_c() | (unsigned)ldc | (SW_FWD || SW_BWD ? (unsigned)p.N * (SW_FWD ? 1 : 2) : 0u)) & 127) == 0;
        auto put = [&](const u32x4& o, unsigned at) __attribute__((always_inline)) {
            if (whole) __builtin_amdgcn_raw_buffer_store_b128(o, rc, at, 0, 2);
            else __builtin_amdgcn_raw_buffer_store_b128(o, rc, at, 0, 0);
        };
        constexpr int BW = B16 ? 8 : 4;  // consecutive columns of a lane
        [[maybe_unused]] float bias[2][QW][BW];
        if constexpr (BIAS) {
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                for (int w = 0; w < QW; ++w) {
                    const float* at = p.bias + nw + (vc[hb][w] == OOB ? 0 : ((int)vc[hb][w] - (lane & 7) * ldc) / ESZ);  // (a column past the end is not stored)
#pragma unroll
                    for (int e = 0; e < BW; ++e) bias[hb][w][e] = nw < p.N ? at[e] : 0.f;
                }
        }
        [[maybe_unused]] float dot[8][2];
#pragma unroll
        for (int blk = 0; blk < 8; ++blk) {
            const int ha = blk >> 2, i = blk & 3;
            __builtin_amdgcn_sched_barrier(0);
            if (blk < 7) fetch(blk + 1, ADD_R || !RES);
            if constexpr (SW_FWD) {
                // column half 0 is u, half 1 the same units' g: u into C[:, unit], g into C[:, N/2 + unit], u silu(g) of the rounded operands into R[:, unit]
                const auto ra = __builtin_amdgcn_make_buffer_rsrc(corner_of(p.R, p.ldr), 0, rows * ldr, 0x00020000);
                u32x4 u[2], g[2];
                quad_packed(acc[ha][0][i], u);
                quad_packed(acc[ha][1][i], g);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    u32x4 act;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        act[e] = pack_bf2(swiglu_act(__uint_as_float(u[half][e] << 16), __uint_as_float(g[half][e] << 16)), swiglu_act(__uint_as_float(u[half][e] & 0xffff0000u), __uint_as_float(g[half][e] & 0xffff0000u)));
                    const unsigned at = vc[0][0] + (unsigned)((blk * 16 + half * 8) * ldc);
                    put(u[half], at);
                    put(g[half], at + (unsigned)p.N);
                    __builtin_amdgcn_raw_buffer_store_b128(act, ra, vr[0][0] + (unsigned)((blk * 16 + half * 8) * ldr), 0, 0);
                }
                continue;
            }
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
                if constexpr (!B16) {
#pragma unroll
                    for (int w = 0; w < 2; ++w) {
                        float a[4], b[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) a[e] = quad_value(acc[ha][hb][i][2 * w], e), b[e] = quad_value(acc[ha][hb][i][2 * w + 1], e);
#pragma unroll
                        for (int half = 0; half < 2; ++half) {
                            u32x4 o;
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                float v = __uint_as_float(quad_rows(__float_as_uint(a[e]), __float_as_uint(b[e]), half));
                                if constexpr (BIAS) v += bias[hb][w][e];
                                if constexpr (ADD_R) v += __uint_as_float(rv[blk & 1][hb][half][w][e]);
                                o[e] = __float_as_uint(v);
                            }
                            put(o, vc[hb][w] + (unsigned)((blk * 16 + half * 8) * ldc));
                        }
                    }
                } else if constexpr (BIAS || ADD_R) {
                    float v[2][8];
                    quad_spread(acc[ha][hb][i], v);
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            if constexpr (BIAS) v[half][e] += bias[hb][0][e];
                            if constexpr (ADD_R) v[half][e] += __uint_as_float(e & 1 ? rv[blk & 1][hb][half][0][e >> 1] & 0xffff0000u : rv[blk & 1][hb][half][0][e >> 1] << 16);
                        }
                        const u32x4 o = {pack_bf2(v[half][0], v[half][1]), pack_bf2(v[half][2], v[half][3]), pack_bf2(v[half][4], v[half][5]), pack_bf2(v[half][6], v[half][7])};
                        put(o, vc[hb][0] + (unsigned)((blk * 16 + half * 8) * ldc));
                    }
                } else {
                    u32x4 o[2];
                    quad_packed(acc[ha][hb][i], o);
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const unsigned at = vc[hb][0] + (unsigned)((blk * 16 + half * 8) * ldc);
                        if constexpr (SW_BWD) {
                            // o = d(act), rounded; d(gate-up) = [d g sig(g) | d u sig(g) (1 + g (1 - sig(g)))] into C[:, unit], C[:, N + unit]
                            const u32x4 u = rv[blk & 1][hb][half][0], g = rv[blk & 1][hb][half][WORDS - 1];
                            u32x4 o0, o1;
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                float du[2], dg[2];
                                swiglu_grads(__uint_as_float(o[half][e] << 16), __uint_as_float(u[e] << 16), __uint_as_float(g[e] << 16), du[0], dg[0]);
                                swiglu_grads(__uint_as_float(o[half][e] & 0xffff0000u), __uint_as_float(u[e] & 0xffff0000u), __uint_as_float(g[e] & 0xffff0000u), du[1], dg[1]);
                                o0[e] = pack_bf2(du[0], du[1]), o1[e] = pack_bf2(dg[0], dg[1]);
                            }
                            put(o0, at);
                            put(o1, at + (unsigned)(p.N * 2));
                        } else {
                            put(o[half], at);
                            if constexpr (DELTA) {
                                // o = d(ctx), rounded: its product with ctx over the half head's 64 columns, folded over the row's eight lanes from their lowest column bit up
                                const u32x4 cv = rv[blk & 1][hb][half][0];
                                float d = 0.f;
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    d += __uint_as_float(o[half][e] << 16) * __uint_as_float(cv[e] << 16) + __uint_as_float(o[half][e] & 0xffff0000u) * __uint_as_float(cv[e] & 0xffff0000u);
                                unsigned x, y;
                                const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(d), __float_as_uint(d), false, false);
                                d = __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
                                quad_swap(__float_as_uint(d), __float_as_uint(d), x, y);
                                d = __uint_as_float(x) + __uint_as_float(y);
                                d += wave_dpp<0x128>(d);
                                dot[blk][half] = hb == 0 ? d : dot[blk][half] + d;
                            }
                        }
                    }
                }
            }
        }
        if constexpr (DELTA) {  // a wave's 128 columns are one head: lane's row of 64 = its eight lanes' group of eight rows
            const int64_t head = nw >> 7;
#pragma unroll
            for (int ha = 0; ha < 2; ++ha) {
                float d = dot[ha * 4][0];
#pragma unroll
                for (int g = 1; g < 8; ++g) d = (lane >> 3) == g ? dot[ha * 4 + (g >> 1)][g & 1] : d;
                const int64_t gm = mw + ha * 64 + lane;
                if (gm < p.M && head < p.ad_Hq) {
                    const int64_t bb = gm / p.ad_S, at = (bb * p.ad_Hq + head) * p.ad_S + gm - bb * p.ad_S;
                    p.ad_delta[at] = d;
                    p.ad_ndl[at] = -d;
                    p.ad_nl2[at] = -p.ad_lse[at] * 1.4426950408889634f;
                }
            }
        }
    };

    using Cold = integral_constant<int, 16>;
    using Behind = integral_constant<int, 16 + STORES < 63 ? 16 + STORES : 63>;  // a write-out's stores are younger than the K-tile that its successor starts with
    ktile(I0{}, std::true_type{}, Cold{});
    ktile(I1{}, std::false_type{}, Cold{});
    for (;;) {
        const int nt = SPLIT ? min(per, nt_even - k0) : nt_even;
        for (int t = 4; t < nt; t += 2) {
            ktile(I0{}, std::false_type{}, Cold{});
            ktile(I1{}, std::false_type{}, Cold{});
        }
        const int next = q + G;  // the last two K-tiles request the next tile's first two (none: a K-tile past the end, zeros)
        int m1 = m0, n1 = n0, k1 = k0;
        if (next < ntiles) {
            origin(next, m1, n1, k1);
            open(m1, n1, k1);
        } else {
            kreq = nt_all;
        }
        place(m0, n0);
        ktile(I0{}, std::false_type{}, Cold{});
        // the first block's residual rows go out a K-tile ahead; that K-tile's requests are younger
        fetch(0, CHUNK || p.R != nullptr);
        __builtin_amdgcn_sched_barrier(0);
        ktile(I1{}, std::false_type{}, integral_constant<int, 16 + LOADS>{});
        if constexpr (!CHUNK && RES) {
            if (p.R) write_out(std::true_type{});
            else write_out(std::false_type{});
        } else {
            write_out(integral_constant<bool, RES>{});
        }
        if (next >= ntiles) break;
        q = next, m0 = m1, n0 = n1, k0 = k1;
        ktile(I0{}, std::true_type{}, Behind{});
        ktile(I1{}, std::false_type{}, Cold{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the zeros past the end must not reach the LDS of a workgroup that follows
}

template <int FORM, int OUT_DT, int KIND>
__global__ __launch_bounds__(256, 1) void gemm_quad_kernel(GemmParams p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    quad_tiles<FORM, OUT_DT, KIND>(p, blockIdx.x, gridDim.x, p.tiles_m * p.tiles_n * (KIND == QUAD_SPLIT ? p.ksplit : 1), smem);
}

// several problems of the TN form in one launch, a workgroup per tile, or per tile and share of K (see gemm_grouped_kernel)
template <int OUT_DT, bool SPLIT>
__global__ __launch_bounds__(256, 1) void gemm_quad_grouped_kernel(GroupTable tbl) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tiles = tbl.start[tbl.count];
    int v = xcd_chunked(blockIdx.x, gridDim.x), share = 0;
    if constexpr (SPLIT) share = v / tiles, v -= share * tiles;
    int g = 0;
#pragma unroll
    for (int i = 1; i < MAX_GROUP; ++i)
        if (i < tbl.count && v >= tbl.start[i]) g = i;
    const GemmParams p = tbl.g[g];
    quad_tiles<MI355_GEMM_TN, OUT_DT, SPLIT ? QUAD_SPLIT : QUAD_RES, false>(p, v - tbl.start[g] + share * p.tiles_m * p.tiles_n, 1 << 30, p.tiles_m * p.tiles_n * (SPLIT ? p.ksplit : 1), smem);
}

// C = the sum of a problem's shares, in their order (+ R).  U groups of four columns a thread, start[i] the first block of problem i.  Four shares' loads go out before the first is added.
template <int OUT_DT, int U>
__global__ __launch_bounds__(256) void quad_fold_kernel(GroupTable tbl) {
    int g = 0;
#pragma unroll
    for (int i = 1; i < MAX_GROUP; ++i)
        if (i < tbl.count && (int)blockIdx.x >= tbl.start[i]) g = i;
    const GemmParams p = tbl.g[g];
    const int64_t all = p.M * p.N, at = ((int64_t)(blockIdx.x - tbl.start[g]) * (256 * U) + threadIdx.x) * 4;
    f32x4 acc[U];
    int64_t from[U];  // (past the end: the last group again)
#pragma unroll
    for (int u = 0; u < U; ++u) {
        from[u] = min(at + u * 1024, all - 4);
        acc[u] = *reinterpret_cast<const f32x4*>(p.ws + from[u]);
    }
    int share = 1;
    for (; share + 4 <= p.ksplit; share += 4) {
        f32x4 v[4][U];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int u = 0; u < U; ++u) v[s][u] = *reinterpret_cast<const f32x4*>(p.ws + (share + s) * all + from[u]);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int u = 0; u < U; ++u) acc[u] += v[s][u];
    }
    for (; share < p.ksplit; ++share)
#pragma unroll
        for (int u = 0; u < U; ++u) acc[u] += *reinterpret_cast<const f32x4*>(p.ws + share * all + from[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (at + u * 1024 >= all) continue;
        const int64_t m = (at + u * 1024) / p.N, n = at + u * 1024 - m * p.N;
        if constexpr (OUT_DT == MI355_DT_BF16) {
            if (p.R) {
                const u32x2 r = *reinterpret_cast<const u32x2*>((const bf16_t*)p.R + m * p.ldr + n);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[u][e] += __uint_as_float(e & 1 ? r[e >> 1] & 0xffff0000u : r[e >> 1] << 16);
            }
            *reinterpret_cast<u32x2*>((bf16_t*)p.C + m * p.ldc + n) = u32x2{pack_bf2(acc[u][0], acc[u][1]), pack_bf2(acc[u][2], acc[u][3])};
        } else {
            if (p.R) acc[u] += *reinterpret_cast<const f32x4*>((const float*)p.R + m * p.ldr + n);
            *reinterpret_cast<f32x4*>((float*)p.C + m * p.ldc + n) = acc[u];
        }
    }
}
