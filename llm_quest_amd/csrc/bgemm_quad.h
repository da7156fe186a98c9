// bgemm on 256 x 256 tiles by four waves of 128 x 128 outputs, bf16 operands, weights stored [out, in], K a multiple of 128 (included by bgemm.hip).  The ring of panels, the phases and the waits are
// gemm_quad.h's NT form; what differs:
//   * A workgroup finds its tile's group from the device-side offsets (as bgemm_wide_kernel), and walks tiles id, id + grid, ...: the next one's place and its rows' sources are looked up while the
//     current one multiplies, and its first K-tiles requested beside the last of that one.
//   * A group's rows are dealt evenly over its ceil(rows / 256) tiles and a tile's evenly over the two waves of a column half, in blocks of 16; blocks that a wave does not have are not multiplied (NA of
//     them: 4 or fewer leave the second half of A out).  Rows beyond a wave's are the tile's last one again, and not stored.
//   * A's rows are gathered, so every lane's source is a pointer of its own; B's panels come by descriptor.  Gated: panel B0 holds 128 gate rows, B1 the same units' up rows, a lane both operands.
//   * Rows are scattered and scaled by the tables to_row and scale in LDS behind the ring: looked up two steps ahead, one look-up behind the other, so that none is waited for.
// 16 378 rows in 16 groups, us, bgemm_wide_kernel -> here: 2 048 -> 2 x 3 584 gated 557 -> 469 (1 026 TFLOP/s), 3 584 -> 2 048 303 -> 255; 6 000 rows, 1 024 -> 2 x 1 792 86 -> 75, 1 792 -> 1 024
// 50 -> 44; 640 rows 33 -> 30 and 32 -> 25.  Numbers of blocks without a variant of their own (5, 3, 1) take the next larger one's: with 8, 7 and 4 alone it is 486 and 257, 163 and 97, 34 and 28;
// with a run-time count 528 and 293.  What is left beside the products: the write-out, in which the matrix cores idle, and 2.25 tiles a workgroup at 3 584 -> 2 048.
constexpr int QUAD_GROUPS = 256;  // at most
template <bool GLU>
__global__ __launch_bounds__(256, 1) void bgemm_quad_kernel(BgemmArgs p, int batch, int tn) {
    extern __shared__ __attribute__((aligned(16))) char quad_lds[];
    char* const smem = quad_lds;
    int* const to_row = (int*)(smem + QUAD_SMEM);  // [256]
    float* const scale = (float*)(to_row + 256);  // [256]
    int* const offs = to_row + 512;               // [batch + 1] first sorted row of a group
    int* const tiles = offs + QUAD_GROUPS + 1;    // [batch + 1] row tiles in the groups before
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    for (int i = tid; i <= batch; i += 256) offs[i] = p.grp_offs ? p.grp_offs[i] : i * p.M;
    __syncthreads();
    if (wave == 0) {
        int before = 0;
        for (int b0 = 0; b0 < batch; b0 += 64) {
            int v = b0 + lane < batch ? (offs[b0 + lane + 1] - offs[b0 + lane] + 255) / 256 : 0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(v, o, 64);
                if (lane >= o) v += u;
            }
            if (b0 + lane < batch) tiles[b0 + lane + 1] = before + v;
            before += __shfl(v, 63, 64);
        }
        if (lane == 0) tiles[0] = 0;
    }
    __syncthreads();
    const int useful = __builtin_amdgcn_readfirstlane(tiles[batch]) * tn;
    struct Tile {
        int b, first, cnt, per, n0;  // group, first sorted row, rows, rows of a wave (a multiple of 16), first column
    };
    auto find = [&](int id) {
        const int q = useful >> 3, r8 = useful & 7, xcd = id & 7;
        const int at = (xcd < r8 ? xcd * (q + 1) : r8 * (q + 1) + (xcd - r8) * q) + (id >> 3);
        int b = 0;  // groups that end at this tile or before
        for (int b0 = 0; b0 < batch; b0 += 64) b += __popcll(__ballot(b0 + lane < batch && tiles[b0 + lane + 1] * tn <= at));
        b = __builtin_amdgcn_readfirstlane(b);
        const int before = __builtin_amdgcn_readfirstlane(tiles[b]), mine = __builtin_amdgcn_readfirstlane(tiles[b + 1]) - before, local = at - before * tn, tm = local % mine;
        const int row0 = p.grp_offs ? __builtin_amdgcn_readfirstlane(offs[b]) : 0, rows = __builtin_amdgcn_readfirstlane(offs[b + 1]) - __builtin_amdgcn_readfirstlane(offs[b]);
        const int share = (rows + mine - 1) / mine, m0 = tm * share;  // (share <= 256 and 256 (mine - 1) < rows: no tile is without rows)
        Tile t;
        t.b = b, t.n0 = local / mine * 256;
        t.first = row0 + m0;
        t.cnt = min(share, rows - m0);
        t.per = ((t.cnt + 1) / 2 + 15) & ~15;
        return t;
    };
    // ---- requests: pieces as in gemm_quad.h; a wave's rows of panel h are its own 64 h + (0 .. 63)
    const char *srcA[2][4], *baseB, *nextB;
    int next_row[2][4], next_to = 0, to = 0;  // the following tile's rows in A, the row in C of its row number tid; this tile's
    unsigned vB[2][4];
    int recB, next_recB;
    const int pr = wave * 32 + (lane >> 3);  // (piece j: + 8 j)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = pr + j * 8, c = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
            const int row = GLU ? (r >> 5) * 64 + h * 32 + (r & 31) : (r >> 6) * 128 + h * 64 + (r & 63);
            vB[h][j] = (unsigned)(row * p.sbn * 2 + c);
        }
    const int* const a_list = p.a_rows ? p.a_rows : (const int*)p.A;  // (no list: one word of A, not used)
    const int* const c_list = p.c_rows ? p.c_rows : (const int*)p.A;
    const float* const scales = p.row_scale ? p.row_scale : (const float*)p.A;
    // What the following tile needs, all requests at once; settled two K-tiles later, when they have come.
    auto look_up = [&](const Tile& t) {
        int l = lane;
        asm volatile("" : "+v"(l));  // what follows from the lane is derived per tile: kept across the products it would cost registers, and fragments that are moved about in front of products from asm
        const int pr = wave * 32 + (l >> 3), tid = wave * 64 + l;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = pr + j * 8, own = h * 64 + (r & 63), row = t.first + min((own < t.per ? (r >> 6) * t.per + own : t.cnt), t.cnt - 1);
                next_row[h][j] = a_list[p.a_rows ? row : 0];
                if (!p.a_rows) next_row[h][j] = row;
            }
        const unsigned long long at = (unsigned long long)((const bf16_t*)p.B + (int64_t)t.b * p.b_bs + (int64_t)t.n0 * p.sbn);
        nextB = (const char*)(((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(at >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((unsigned)at));
        next_recB = (int)(min(256, p.N - t.n0) * p.sbn * 2);
        const int row = t.first + min(tid, t.cnt - 1);
        next_to = c_list[p.c_rows ? row : 0];
        if (!p.c_rows) next_to = row;
    };
    auto settle = [&]() {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) next_row[h][j] = p.a_rows ? next_row[h][j] / p.a_div : next_row[h][j];
        asm volatile("" : "+v"(next_to));
    };
    int kreq = 0;
    auto open = [&](const Tile& t) {
        int l = lane;
        asm volatile("" : "+v"(l));
        const int pr = wave * 32 + (l >> 3);
        const char* const a = (const char*)((const bf16_t*)p.A + (int64_t)t.b * p.a_bs);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) srcA[h][j] = a + (int64_t)next_row[h][j] * p.lda * 2 + ((l & 7) ^ (((pr + j * 8) >> 1) & 7)) * 16;
        baseB = nextB, recB = next_recB, kreq = 0;
        to = next_to;
    };
    auto request = [&](int stage, int panel, int j) {
        char* dst = smem + stage * QUAD_STAGE + panel * QUAD_PANEL + wave * 4096 + j * 1024;
        if (panel < 2) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(srcA[panel & 1][j] + (int64_t)kreq * 128), (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
        } else {
            auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(baseB + (int64_t)kreq * 128), 0, recB, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS_PTR(dst), 16, vB[panel & 1][j], 0, 0, 0);
        }
    };
    // ---- fragments (gemm_quad.h)
    bf16x8 fa[2][2][4], fb[2][2][4];
    const int r16 = lane & 15, off0 = r16 * 128 + (((lane >> 4) ^ ((r16 >> 1) & 7)) << 4);
    auto read_frag = [&](bf16x8 (&f)[2][4], auto stage_c, auto panel_c, int n) __attribute__((always_inline)) {
        constexpr int STAGE = decltype(stage_c)::value, PANEL = decltype(panel_c)::value;
        const int kk = n >> 2, i = n & 3;
        f[kk][i] = *reinterpret_cast<const bf16x8*>(smem + STAGE * QUAD_STAGE + PANEL * QUAD_PANEL + (PANEL < 2 ? wm : wn) * 8192 + i * 2048 + (off0 ^ (kk * 64)));
    };
    using std::integral_constant;
    using I0 = integral_constant<int, 0>;
    using I1 = integral_constant<int, 1>;
    using I2 = integral_constant<int, 2>;
    using I3 = integral_constant<int, 3>;
    const int nt = p.K >> 6;  // even, at least four
    int id = blockIdx.x;
    bool more = false;
    Tile t, tnext;

    auto run = [&](auto na_c) __attribute__((always_inline)) {
        constexpr int NA = decltype(na_c)::value;  // blocks of 16 rows of a wave
        f32x4 acc[NA > 4 ? 2 : 1][2][4][4];
        // 8 NI products of a quadrant, one half of a K-tile's reads and requests beside them
        auto phase = [&](auto first_c, auto ni_c, f32x4 (&c)[4][4], const bf16x8 (&a)[2][4], const bf16x8 (&b)[2][4], bf16x8 (&next)[2][4], auto rstage, auto rpanel, int qstage, int qpanel, auto wait_c) __attribute__((always_inline)) {
            constexpr bool FIRST = decltype(first_c)::value;
            constexpr int NI = decltype(ni_c)::value, WAIT = decltype(wait_c)::value, P = NI > 0 ? NI * 8 : 8;
#pragma unroll
            for (int s = 0; s < P; ++s) {
                if constexpr (NI > 0) {
                    const int kk = s / (4 * NI), i = (s >> 2) % NI, j = s & 3;
                    if (FIRST && kk == 0) quad_mma_first(c[i][j], a[kk][i], b[kk][j]);
                    else quad_mma(c[i][j], a[kk][i], b[kk][j]);
                }
                if (s < 8 && !(NA <= 4 && decltype(rpanel)::value == 1)) read_frag(next, rstage, rpanel, s);
                if (s % (P / 4) == P / 4 - 1) request(qstage, qpanel, s / (P / 4));
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (WAIT >= 0) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WAIT) : "memory");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto ktile = [&](auto par, auto first_c) __attribute__((always_inline)) {
            constexpr int S = decltype(par)::value, N0 = NA < 4 ? NA : 4, N1 = NA > 4 ? NA - 4 : 0;
            using Here = integral_constant<int, S>;
            using There = integral_constant<int, S ^ 1>;
            using None = integral_constant<int, -1>;
            using Wait = integral_constant<int, 16>;
            phase(first_c, integral_constant<int, N0>{}, acc[0][0], fa[0], fb[S], fb[S ^ 1], Here{}, I3{}, S, 0, None{});
            phase(first_c, integral_constant<int, N0>{}, acc[0][1], fa[0], fb[S ^ 1], fa[1], Here{}, I1{}, S, 2, Wait{});
            phase(first_c, integral_constant<int, N1>{}, acc[NA > 4 ? 1 : 0][1], fa[1], fb[S ^ 1], fa[0], There{}, I0{}, S, 3, None{});
            phase(first_c, integral_constant<int, N1>{}, acc[NA > 4 ? 1 : 0][0], fa[1], fb[S], fb[S ^ 1], There{}, I2{}, S, 1, Wait{});
            ++kreq;
        };
        float factor_of_row = scales[p.row_scale ? to : 0];
        more = id + (int)gridDim.x < useful;
        tnext = more ? find(id + gridDim.x) : t;
        look_up(tnext);
        __builtin_amdgcn_sched_barrier(0);
        // (the compiler may have moved fragments about at the end of the last tile; products from asm read a register two wait states after it was written at the earliest)
        asm volatile("s_nop 1" : "+v"(fa[0][0][0]), "+v"(fa[0][0][1]), "+v"(fa[0][0][2]), "+v"(fa[0][0][3]), "+v"(fa[0][1][0]), "+v"(fa[0][1][1]), "+v"(fa[0][1][2]), "+v"(fa[0][1][3]),
                     "+v"(fb[0][0][0]), "+v"(fb[0][0][1]), "+v"(fb[0][0][2]), "+v"(fb[0][0][3]), "+v"(fb[0][1][0]), "+v"(fb[0][1][1]), "+v"(fb[0][1][2]), "+v"(fb[0][1][3]));
        ktile(I0{}, std::true_type{});
        ktile(I1{}, std::false_type{});
        if (!p.row_scale) factor_of_row = 1.0f;
        to_row[tid] = to, scale[tid] = factor_of_row;  // (every wave has written the tile before out)
        settle();
        for (int k = 4; k < nt; k += 2) {
            ktile(I0{}, std::false_type{});
            ktile(I1{}, std::false_type{});
        }
        if (more) open(tnext);
        else kreq = 0;  // (no tile follows: the first K-tiles again, which nobody reads)
        ktile(I0{}, std::false_type{});
        ktile(I1{}, std::false_type{});
        // ---- write-out: eight rows x 64 columns at a time (quad.h)
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products' way through the pipe
        int le = lane;
        asm volatile("" : "+v"(le));
        const int lcol = ((le >> 3) & 1) * 32 + ((le >> 4) & 1) * 16 + (le >> 5) * 8, n = GLU ? (t.n0 >> 1) + wn * 64 + lcol : t.n0 + wn * 128 + lcol, n_end = GLU ? p.n_out : p.N;
        const int* const rows_at = to_row + wm * t.per;
        const float* const scale_at = scale + wm * t.per;
        const int own_end = min(t.per, t.cnt - wm * t.per);
        const int64_t base = (int64_t)t.b * p.c_bs;
        auto store = [&](const float (&o)[8], int64_t at) __attribute__((always_inline)) {
            if (p.c_dt == MI355_DT_F32) {
                *(f32x4*)((float*)p.C + at) = f32x4{o[0], o[1], o[2], o[3]};
                *(f32x4*)((float*)p.C + at + 4) = f32x4{o[4], o[5], o[6], o[7]};
            } else {
                *(u32x4*)((bf16_t*)p.C + at) = u32x4{pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]), pack_bf2(o[4], o[5]), pack_bf2(o[6], o[7])};
            }
        };
#pragma unroll
        for (int blk = 0; blk < NA; ++blk) {
            __builtin_amdgcn_sched_barrier(0);
            float v[2][2][8];
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) quad_spread(acc[blk >> 2][hb][blk & 3], v[hb]);
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int own = blk * 16 + half * 8 + (le & 7);
                const float factor = scale_at[own];  // (beyond the tile's rows: the last one's, not used)
                const int64_t at = base + (int64_t)rows_at[own] * p.ldc + n;
                if constexpr (GLU) {
                    if (p.epi == 4) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[0][half][e] = gated_act(4, v[0][half][e], v[1][half][e], p.limit) * factor;
                    } else if (p.epi == 3) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[0][half][e] = gated_act(3, v[0][half][e], v[1][half][e], p.limit) * factor;
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[0][half][e] = gated_act(2, v[0][half][e], v[1][half][e], p.limit) * factor;
                    }
                } else {
#pragma unroll
                    for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            float x = v[hb][half][e];
                            if (p.bias) x += p.bias[min(n + hb * 64, n_end - 8) + e];
                            if (p.epi == 1) x = x > 0.f ? x * x : 0.f;
                            v[hb][half][e] = x * factor;
                        }
                }
                if (own < own_end) {
                    if (n < n_end) store(v[0][half], at);
                    if (!GLU && n + 64 < n_end) store(v[1][half], at + 64);
                }
            }
        }
    };

    if (id >= useful) return;
    t = find(id);
    look_up(t);
    settle();
    open(t);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
        for (int n = 0; n < 16; ++n) request(st, n < 4 ? 0 : n < 8 ? 2 : n < 12 ? 3 : 1, n & 3);
        ++kreq;
    }
    asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int n = 0; n < 8; ++n) {
        read_frag(fa[0], I0{}, I0{}, n);
        read_frag(fb[0], I0{}, I2{}, n);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    for (;;) {
        if (t.per > 112) run(integral_constant<int, 8>{});
        else if (t.per > 96) run(integral_constant<int, 7>{});
        else if (t.per > 64) run(integral_constant<int, 6>{});
        else if (t.per > 32) run(integral_constant<int, 4>{});
        else run(integral_constant<int, 2>{});
        if (!more) break;
        t = tnext, id += gridDim.x;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the requests that nobody reads must not reach the LDS of a workgroup that follows
}
