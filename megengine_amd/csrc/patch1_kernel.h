// The text of patch1_kernel, included by conv_patch1.hip into a namespace for each of its forms (a common device function costs layers of one
// stage 1 to 2 %).  KS: groups of four waves; two take every other stage each, with stage buffers of their own, their sums meet in LDS, and each
// finishes half of the channels.
template <int MT, int NT, int T>
__global__ __launch_bounds__(256 * KS, 2) void patch1_kernel(P1Args a) {
    static_assert(KS == 1 || (KS == 2 && MT * NT == 1), "each of two groups finishes half of one block");
    constexpr int QN = 4 / KS;
    constexpr int NPI = P1_NPI;
    constexpr bool ZPRE = MT * NT <= 2;  // the residual is asked for ahead of the products (the largest tile has no registers for it)
    constexpr int BM = MT * 32, GS = p1_gs(T), F = p1_f(T), E = GS * T, EP = (E + 1) & ~1, STEPS = EP / 2, BMP = p1_bmp(MT);
    constexpr int TPG = 256 / GS;                          // threads per channel group of the patch
    constexpr int QPR = 4 * GS;                            // channel quads of a filter row and stage
    constexpr int FI = (BM * QPR + 255) / 256;             // filter items per thread and stage
    constexpr int A_VECS = EP * BMP;
    extern __shared__ __attribute__((aligned(16))) v4i lds_all[];
    __shared__ __attribute__((aligned(16))) int sBias_all[KS][BM];
    // everything up to the first operands in one batch of scalar loads, and a word of each line that the epilogue reads
    asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.dst), "s"(a.IC), "s"(a.IH), "s"(a.IW), "s"(a.IHW), "s"(a.OC), "s"(a.N),
                 "s"(a.sh), "s"(a.sw), "s"(a.ph), "s"(a.pw), "s"(a.src_sn), "s"(a.kbytes), "s"(a.flt_bytes), "s"(a.has_bias), "s"(a.nstages),
                 "s"(a.NI), "s"(a.TH), "s"(a.TW), "s"(a.tile_px), "s"(a.run), "s"(a.PWC), "s"(a.PX), "s"(a.PXQ), "s"(a.tiles_m));
    asm volatile("" ::"s"(a.tiles_n), "s"(a.tiles_img), "s"(a.tiles_w), "s"(a.div_tiles_m.m), "s"(a.div_tiles_img.m), "s"(a.div_tiles_w.m),
                 "s"(a.div_pqi.m), "s"(a.div_pqi.s2), "s"(a.div_pqw.m), "s"(a.div_pqw.s2), "s"(a.div_tile_px.m), "s"(a.div_tw.m), "s"(a.epi.s_b),
                 "s"(a.epi.lin_lo));
    const int t = threadIdx.x & 255, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31, lh = lane >> 5;
    const int kg = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    const int stage_vecs = A_VECS + GS * a.PX;
    int* const sBias = sBias_all[kg];
    v4i* const lds = lds_all + kg * 2 * stage_vecs;

    // tile: contiguous pixel tiles per XCD (workgroup b runs on XCD b % 8), channel tiles of a pixel tile side by side
    int tm, tn;
    {
        const int per = (a.tiles_n + 7) >> 3, x = blockIdx.x & 7, i = blockIdx.x >> 3;
        const int r = (int)fdiv(i, a.div_tiles_m);
        tm = i - r * a.tiles_m;
        tn = x * per + r;
        if (r >= per || tn >= a.tiles_n) return;
    }
    const P1Tile o = p1_tile_at(a, tn);
    const int n0 = o.n0, oc0 = tm * BM, oh0 = o.oh0, ow0 = o.ow0;
    const int iw_lo = (ow0 * a.sw - a.pw) & ~3;  // the patch starts at a column that is a multiple of four: a quad that starts
                                                 // inside a row starts at one of its columns

    // Patch quads of this thread.  Waves of a group of TPG threads share a channel group, so a channel's plane is a scalar base.
    const int g = GS == 1 ? 0 : wave / (TPG / 64), tg = t & (TPG - 1);
    uint32_t p_sel[NPI][4];
    int p_off[NPI], p_lds[NPI];
    const int turn = (tg >> 1) & 3;
#pragma unroll
    for (int k = 0; k < NPI; ++k) {
        const uint32_t pq = tg + k * TPG, im = fdiv(pq, a.div_pqi), r = pq - im * (uint32_t)(a.PXI >> 2);
        const uint32_t pr = fdiv(r, a.div_pqw), pc = (r - pr * (uint32_t)(a.PWC >> 2)) * 4;
        const int ih = oh0 * a.sh - a.ph + (int)pr, iw = iw_lo + (int)pc, n = n0 + (int)im;
        const bool ok = ((int)pq < a.PXQ) & (n < a.N) & ((unsigned)ih < (unsigned)a.IH) & ((unsigned)iw < (unsigned)a.IW);
        const int back = iw + 4 > a.IW ? iw + 4 - a.IW : 0;  // the row ends inside the quad: loaded `back` columns further left
        p_off[k] = ok ? n * a.src_sn + ih * a.IW + iw - back : SENT;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int p = ((j + turn) & 3) + back;  // byte of the loaded dword that is this pixel
            p_sel[k][j] = ok && p < 4 ? 0x00000400u | (uint32_t)(p | p << 8) : 0x0c0cu;
            p_sel[k][j] |= 0x0c0c0000u;
        }
        p_lds[k] = (int)pq < a.PXQ ? A_VECS + g * a.PX + (int)pq * 4 : -1;
    }
    // filter items of this thread: four channels of a row
    const int f_quad = t & (QPR - 1), f_row = t / QPR;
    constexpr int ROWS_PER_PASS = 256 / QPR;
    int f_off[FI];
#pragma unroll
    for (int k = 0; k < FI; ++k) {
        const int row = f_row + k * ROWS_PER_PASS;
        f_off[k] = row < BM && oc0 + row < a.OC ? (oc0 + row) * a.kbytes + f_quad * 4 * T : -1;
    }

    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes), rs_flt = make_rsrc(a.flt, (uint32_t)a.flt_bytes);
    const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias && kg == 0 ? a.OC * 4 : 0);
    uint32_t xp[NPI][16], xf[FI][T];
    const bool two = a.PXQ > TPG;  // a second quad per thread
    auto fetch = [&](int st) __attribute__((always_inline)) {
        const int c0 = (st * GS + g) * 16;
#pragma unroll
        for (int k = 0; k < FI; ++k) {
            // (a quad past the last channel is not loaded; one whose bytes pass the end of the filter is loaded whole channels further
            // left, and turned back in store)
            const int at = f_off[k] + st * GS * 16 * T;
            const bool in = (f_off[k] >= 0) & (st * GS * 16 + f_quad * 4 < a.IC);
            const int v0 = in ? min(at, a.flt_bytes - 4 * T) : SENT;
#pragma unroll
            for (int v = 0; v + 4 <= T; v += 4) {
                const v4i y = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, v0 + 4 * v, 0, 0);
                xf[k][v] = y[0]; xf[k][v + 1] = y[1]; xf[k][v + 2] = y[2]; xf[k][v + 3] = y[3];
            }
            if constexpr (T % 4 != 0) xf[k][T - 1] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_flt, v0 + 4 * (T - 1), 0, 0);
        }
        // (channels past the last one meet zero filter bytes; the scalar offset never leads out of the image)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            xp[0][i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_src, p_off[0], min(c0 + i, a.IC - 1) * a.IHW, 0);
        if (two)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                xp[NPI - 1][i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_src, p_off[NPI - 1], min(c0 + i, a.IC - 1) * a.IHW, 0);
    };
    auto store = [&](int st, int buf) __attribute__((always_inline)) {
        v4i* s = lds + buf * stage_vecs;
        uint32_t* sw = reinterpret_cast<uint32_t*>(s);
#pragma unroll
        for (int k = 0; k < FI; ++k) {
            const int row = f_row + k * ROWS_PER_PASS, left = a.IC - (st * GS * 16 + f_quad * 4);  // channels from here on
            // Channels that exist, and the quads at the filter's end, which may be those of its last three rows: loaded one to three
            // channels further left.  One selector does both.  (Loading such a quad byte by byte, 4 T loads of one lane, held up the last
            // channel tile: 5x5 59 -> 63 at 79 x 22, batch 4: 13.3 us.)
            const int over = f_off[k] + st * GS * 16 * T + 4 * T - a.flt_bytes;
            const int turned = over <= 0 ? 0 : over <= T ? 1 : over <= 2 * T ? 2 : 3;
            const uint32_t there = left >= 4 ? 0xffffffffu : left > 0 ? (1u << (8 * left)) - 1 : 0u;
            const uint32_t keep = ((0x03020100u + 0x01010101u * (uint32_t)turned) & there) | (0x0c0c0c0cu & ~there);
            if (BM * QPR >= 256 || row < BM)
#pragma unroll
                for (int tap = 0; tap < T; ++tap)
                    sw[(((f_quad >> 2) * T + tap) * BMP + row) * 4 + (f_quad & 3)] = __builtin_amdgcn_perm(0u, p1_tap<T>(xf[k], tap), keep);
        }
#pragma unroll
        for (int k = 0; k < NPI; ++k) {
            if (k == 1 && !two) break;
            if (p_lds[k] >= 0)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v4i turned;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const uint32_t lo = __builtin_amdgcn_perm(xp[k][4 * c + 1], xp[k][4 * c], p_sel[k][j]);
                        const uint32_t hi = __builtin_amdgcn_perm(xp[k][4 * c + 3], xp[k][4 * c + 2], p_sel[k][j]);
                        turned[c] = (int)(lo | hi << 16);
                    }
                    s[p_lds[k] + ((j + turn) & 3)] = turned;
                }
        }
    };
    const int bias_v = __builtin_amdgcn_raw_buffer_load_b32(rs_bias, (oc0 + (t & (BM - 1))) * 4, 0, 0);
    fetch(kg);

    // the filter entry that fills up an odd number stays zero, and the bias
    if (EP != E)
        for (int u = t; u < 2 * BM; u += 256) lds[(u / BM) * stage_vecs + E * BMP + u % BM] = v4i{0, 0, 0, 0};
    if (t < BM) sBias[t] = bias_v;

    // B operands: patch vector of each of this lane's pixels, and of each step's entry relative to it
    int b_px[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const uint32_t p = (wave * NT + j) * 32 + l32;
        const uint32_t im = fdiv(p, a.div_tile_px), r = p - im * (uint32_t)a.tile_px + o.skip, oh = fdiv(r, a.div_tw), ow = r - oh * a.TW;
        b_px[j] = (((int)im < a.NI) & ((int)oh < a.TH)) ? (int)(im * a.PXI + oh * a.sh * a.PWC) + ((int)ow + ow0) * a.sw - a.pw - iw_lo : 0;
    }
    int offs[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
        const int e0 = 2 * k, e1 = 2 * k + 1 < E ? 2 * k + 1 : 0;  // (the filling entry multiplies any vector by zero)
        const int o0 = (e0 / T) * a.PX + ((e0 % T) / F) * a.PWC + (e0 % T) % F, o1 = (e1 / T) * a.PX + ((e1 % T) / F) * a.PWC + (e1 % T) % F;
        offs[k] = A_VECS + (lh ? o1 : o0);
    }
    // Where the residual lies is worked out while the first operands are on their way, and its loads stand ahead of the next stage's, which are
    // waited for first.  (Both inside the branch, behind those: 300 drawn layers with a residual 1.025 of the time.  Without the branch sixteen loads
    // of no bytes: 300 without a residual 1.01 to 1.03.)
    P1Residual z_at[NT];
    if constexpr (ZPRE)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            z_at[j] = p1_residual_at(a, p1_out(a, o, (wave * NT + j) * 32 + (l32 & ~3), 4 * lh + (l32 & 3)));
            asm volatile("" : "+v"(z_at[j].off));
        }
    store(kg, 0);
    __builtin_amdgcn_s_waitcnt(P1_VMCNT0);  // (the compiler knows: a stage's products do not wait for the next stage's loads)
    uint32_t zq[NT][MT][QN];
    if (ZPRE && a.epi.has_z) p1_residual<MT, NT, QN>(a, zq, z_at, oc0 + kg * 16, 4 * lh + (l32 & 3));
    if (kg + KS < a.nstages) fetch(kg + KS);
    __syncthreads();
    v16i acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4i b = *reinterpret_cast<const v4i*>(sBias + i * 32 + 8 * q + 4 * lh);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                acc[i][j][4 * q] = b[0]; acc[i][j][4 * q + 1] = b[1]; acc[i][j][4 * q + 2] = b[2]; acc[i][j][4 * q + 3] = b[3];
            }
        }
    const int groups = (a.IC + 15) >> 4;
    auto products = [&](int st, int buf) __attribute__((always_inline)) {
        const v4i* s = lds + buf * stage_vecs;
        const v4i* pa = s + lh * BMP + l32;
        auto load = [&](int k, v4i (&fa)[MT], v4i (&fb)[NT]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i) fa[i] = pa[k * 2 * BMP + i * 32];
#pragma unroll
            for (int j = 0; j < NT; ++j) fb[j] = s[offs[k] + b_px[j]];
        };
        constexpr int AHEAD = 2;  // steps whose operands are read ahead
        v4i fa[AHEAD + 1][MT], fb[AHEAD + 1][NT];
#pragma unroll
        for (int k = 0; k < AHEAD && k < STEPS; ++k) load(k, fa[k], fb[k]);
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
            // (an incomplete last stage: nothing of the groups past the last one; wave-uniform)
            if (k > 0 && (2 * k) % T < 2 && st * GS + (2 * k) / T >= groups) break;
            if (k + AHEAD < STEPS) load(k + AHEAD, fa[(k + AHEAD) % (AHEAD + 1)], fb[(k + AHEAD) % (AHEAD + 1)]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[k % (AHEAD + 1)][i], fb[k % (AHEAD + 1)][j], acc[i][j], 0, 0, 0);
        }
    };
    for (int st = kg;; st += KS) {  // (as many rounds for either group)
        if (KS == 1 || st < a.nstages) products(st, (st / KS) & 1);
        if (st - kg + KS >= a.nstages) break;
        if (KS == 1 || st + KS < a.nstages) {
            store(st + KS, (st / KS + 1) & 1);
            if (st + 2 * KS < a.nstages) fetch(st + 2 * KS);
        }
        __syncthreads();
    }
    if constexpr (KS == 2) {
        // group 0 finishes the first sixteen channels of the block and group 1 the others: each hands the other's over
        v16i& c = acc[0][0];
        const v4i give[2] = {kg ? v4i{c[0], c[1], c[2], c[3]} : v4i{c[8], c[9], c[10], c[11]},
                             kg ? v4i{c[4], c[5], c[6], c[7]} : v4i{c[12], c[13], c[14], c[15]}};
        __syncthreads();
        v4i* x = lds_all + kg * 512 + t;
        x[0] = give[0];
        x[256] = give[1];
        __syncthreads();
        const v4i* y = lds_all + (kg ^ 1) * 512 + t;
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = (kg ? c[8 + i] : c[i]) + y[(i >> 2) * 256][i & 3];
    }

    // (the largest tile has registers for it once the products are done: all of it at once, where each dword used to be waited for behind the
    // store before it; 3x3 7 -> 210 at 63 x 84, batch 42: 75.4 -> 61.2 us)
    if constexpr (ZPRE) {
        if (a.epi.has_z && a.OHW < 4) p1_residual_bytes<MT, NT, QN>(a, zq, o, oc0 + kg * 16, wave, l32, lh);
    } else if (a.epi.has_z) {
        p1_residual_late<MT, NT, QN>(a, zq, o, oc0, wave, l32, lh);
    }
#define MI355_P1(NL, HZ) p1_epilogue<MT, NT, QN, NL, HZ>(a, acc, zq, o, oc0 + kg * 16, wave, l32, lh)
    if (a.epi.lin) {
        MI355_P1(NL_LIN, false);
    } else if (a.epi.has_z) {
        switch (a.epi.nonline) {
            case NL_RELU: MI355_P1(NL_RELU, true); break;
            case NL_H_SWISH: MI355_P1(NL_H_SWISH, true); break;
            default: MI355_P1(NL_IDENTITY, true); break;
        }
    } else {
        switch (a.epi.nonline) {
            case NL_RELU: MI355_P1(NL_RELU, false); break;
            case NL_H_SWISH: MI355_P1(NL_H_SWISH, false); break;
            default: MI355_P1(NL_IDENTITY, false); break;
        }
    }
#undef MI355_P1
}
