// The text of patch4_kernel, included by conv_patch4.hip into a namespace for each of its forms (behind a common device function the compiler
// schedules the loops of all of them worse, up to 8 % of a layer).  The namespace says
//   KS      groups of four waves; two take every other stage each, with stage buffers of their own, and their sums meet in LDS;
//   TAPS25  a stage is one channel group of 25 taps: thirteen steps, compiled in.  Otherwise FORM is the number of matrix steps of a stage
//           where it is known (9: nine taps, two channel groups), or 0: from the arguments.
template <int MT, int NT, int FORM>
__global__ __launch_bounds__(256 * KS, 2) void patch4_kernel(P4Args a) {
    constexpr int STEPS = TAPS25 ? 13 : FORM;
    static_assert(KS == 1 || (KS == 2 && MT * NT == 1), "each of two groups finishes half of one block");
    constexpr int BM = MT * 32, TAPS = STEPS == 9 ? 9 : STEPS == 13 ? 25 : 0, GROUPS = STEPS == 9 ? 2 : 1, RPI = STEPS ? 256 / (GROUPS * TAPS) : 1;
    constexpr int KAN = (BM + RPI - 1) / RPI;
    // vectors from one entry to the next: the rows its passes store, made odd so that the stores of a row spread over the banks
    const int kan = STEPS ? KAN : a.kan, rpi = STEPS ? RPI : a.rpi, BMP = (kan * rpi) | 1;
    extern __shared__ __attribute__((aligned(16))) v4i lds_all[];
    const int t = threadIdx.x & 255, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31, lh = lane >> 5;
    const int kg = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    const int T = STEPS ? TAPS : a.T, GS = STEPS ? GROUPS : a.GS;
    const int E = GS * T, EP = (E + 1) & ~1;              // entries of a stage, of a whole number of steps
    const int a_vecs = EP * BMP, stage_vecs = a_vecs + GS * a.PX;
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
    const int ig = (int)fdiv(tn, a.div_tiles_img), ti = tn - ig * a.tiles_img;
    const int th = (int)fdiv(ti, a.div_tiles_w), tw = ti - th * a.tiles_w;
    const int n0 = ig * a.NI, oh0 = th * a.TH, ow0 = tw * a.TW, oc0 = tm * BM;

    // patch pixels of this thread: source offset of the first channel block, SENT outside the image
    int p_off[P4_NPK];
#pragma unroll
    for (int k = 0; k < P4_NPK; ++k) {
        if (k >= a.pkn) break;
        const uint32_t px = t + k * 256, im = fdiv(px, a.div_pxi), r = px - im * a.PXI, pr = fdiv(r, a.div_pwc), pc = r - pr * a.PWC;
        const int ih = oh0 * a.sh - a.ph + (int)pr, iw = ow0 * a.sw - a.pw + (int)pc, n = n0 + (int)im;
        const bool ok = (int)px < a.PX && n < a.N && (unsigned)ih < (unsigned)a.IH && (unsigned)iw < (unsigned)a.IW;
        p_off[k] = ok ? n * a.src_sn + (ih * a.IW + iw) * 4 : SENT;
    }
    // filter vectors of this thread: the same 16 bytes of every rpi-th row; dword d of a row is tap d % T of channel block
    // d / T (rows past the last channel lie past the end of the buffer: zero)
    const int vr = STEPS ? GROUPS * TAPS : a.vr;
    const int f_row = STEPS ? t / (GROUPS * (TAPS ? TAPS : 1)) : (int)fdiv(t, a.div_vr), f_first = (t - f_row * vr) * 4;
    int f_off[P4_NKA];
#pragma unroll
    for (int k = 0; k < P4_NKA; ++k) {
        if (k >= kan) break;
        f_off[k] = f_row < rpi ? (oc0 + f_row + k * rpi) * a.kbytes + f_first * 4 : SENT;
    }
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes), rs_flt = make_rsrc(a.flt, a.flt_bytes);
    v4i xp[P4_NPK], xf[P4_NKA];
    const int row_words = a.icb * T;
    // The patch's channel blocks are a scalar offset: those past the last one are the last one's again (they meet zero filter
    // bytes), so that the scalar offset never leads out of the image.  The filter's stage is part of the lane's offset, which
    // the descriptor's bounds check covers.
    const uint32_t last_cb = (uint32_t)(a.icb - 1) * a.src_scb;
    auto fetch = [&](int st) __attribute__((always_inline)) {
        const int cb0 = st * GS * 4, left = row_words - cb0 * T;  // filter words left in a row
        const int fo = cb0 * T * 4;
#pragma unroll
        for (int k = 0; k < P4_NKA; ++k) {
            if (k >= kan) break;
            xf[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, f_off[k] + fo, 0, 0);
        }
        int so[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) so[i] = (int)min((uint32_t)(cb0 + i) * a.src_scb, last_cb);
#pragma unroll
        for (int k = 0; k < P4_NPK; ++k) {
            if (k >= a.pkn) break;
#pragma unroll
            for (int i = 0; i < 4; ++i) xp[k][i] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_src, p_off[k], so[i], 0);
            if (k < P4_NPK / 2 && GS == 2) {
#pragma unroll
                for (int i = 0; i < 4; ++i) xp[P4_NPK / 2 + k][i] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_src, p_off[k], so[4 + i], 0);
            }
        }
        if (left < vr * 4) {  // the last stage, incomplete: words past the row's end are the next row's
#pragma unroll
            for (int k = 0; k < P4_NKA; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) xf[k][i] = f_first + i < left ? xf[k][i] : 0;
        }
    };
    fetch(kg);

    int f_lds[4];
    {
        uint32_t cb = STEPS ? f_first / (TAPS ? TAPS : 1) : fdiv(f_first, a.div_t), tap = f_first - cb * T;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f_lds[i] = (int)((((cb >> 2) * T + tap) * BMP + f_row) * 4 + (cb & 3));
            if (++tap == (uint32_t)T) {
                tap = 0;
                ++cb;
            }
        }
    }
    auto store = [&](int buf) __attribute__((always_inline)) {
        v4i* s = lds + buf * stage_vecs;
        int* sw = reinterpret_cast<int*>(s);
        if (f_row < rpi) {
#pragma unroll
            for (int k = 0; k < P4_NKA; ++k) {
                if (k >= kan) break;
#pragma unroll
                for (int i = 0; i < 4; ++i) sw[f_lds[i] + k * rpi * 4] = xf[k][i];
            }
        }
#pragma unroll
        for (int k = 0; k < P4_NPK; ++k) {
            if (k >= a.pkn) break;
            if (t + k * 256 < a.PX) {
                s[a_vecs + t + k * 256] = xp[k];
                if (k < P4_NPK / 2 && GS == 2) s[a_vecs + a.PX + t + k * 256] = xp[P4_NPK / 2 + k];
            }
        }
    };

    // B operands: patch vector of each of this lane's pixels, and of each entry relative to it
    int b_px[NT], d_px[NT], z_px[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const uint32_t p = (wave * NT + j) * 32 + l32;
        const uint32_t im = fdiv(p, a.div_tile_px), r = p - im * (uint32_t)(a.TH * a.TW), oh = fdiv(r, a.div_tw), ow = r - oh * a.TW;
        const bool ok = (int)im < a.NI && n0 + (int)im < a.N && oh0 + (int)oh < a.OH && ow0 + (int)ow < a.OW;
        b_px[j] = (int)im < a.NI ? (int)(im * a.PXI + oh * a.sh * a.PWC + ow * a.sw) : 0;
        const int at = ((oh0 + (int)oh) * a.OW + ow0 + (int)ow) * 4;
        d_px[j] = ok ? (n0 + (int)im) * a.dst_sn + at : -1;
        z_px[j] = (n0 + (int)im) * a.z_sn + at;
    }
    int* tab = reinterpret_cast<int*>(lds_all + KS * 2 * stage_vecs);
    for (int e = threadIdx.x; e < EP; e += 256 * KS) {
        const int g = (int)fdiv(e, a.div_t), tap = e - g * a.T, fh = tap / a.FW, fw = tap - fh * a.FW;
        tab[e] = e < E ? a_vecs + g * a.PX + fh * a.PWC + fw : a_vecs;
    }
    // the filter entry that fills up an odd number stays zero
    if (EP != E && t < 2 * BM) lds[(t / BM) * stage_vecs + E * BMP + t % BM] = v4i{0, 0, 0, 0};
    v16i acc[MT][NT];
    {
        const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias && kg == 0 ? a.OC * 4 : 0);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            v16i b;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4i v = __builtin_amdgcn_raw_buffer_load_b128(rs_bias, (oc0 + i * 32 + 8 * q + 4 * lh) * 4, 0, 0);
                b[4 * q] = v[0]; b[4 * q + 1] = v[1]; b[4 * q + 2] = v[2]; b[4 * q + 3] = v[3];
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = b;
        }
    }
    store(0);
    __syncthreads();
    const int steps = EP / 2;
    int offs[STEPS ? STEPS : 1];
    if constexpr (STEPS != 0) {
#pragma unroll
        for (int k = 0; k < STEPS; ++k) offs[k] = tab[2 * k + lh];
    }
    for (int st = kg; st - kg < a.nstages; st += KS) {  // (as many rounds for either group)
        if (st + KS < a.nstages) fetch(st + KS);
        const v4i* s = lds + ((st / KS) & 1) * stage_vecs;
        const v4i* pa = s + lh * BMP + l32;
        auto load = [&](int k, int off, v4i (&fa)[MT], v4i (&fb)[NT]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i) fa[i] = pa[k * 2 * BMP + i * 32];
#pragma unroll
            for (int j = 0; j < NT; ++j) fb[j] = s[off + b_px[j]];
        };
        auto mult = [&](const v4i (&fa)[MT], const v4i (&fb)[NT]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
        };
        if (KS > 1 && st >= a.nstages) {
        } else if constexpr (STEPS != 0) {
            constexpr int AHEAD = 2;  // steps whose operands are read ahead
            v4i fa[AHEAD + 1][MT], fb[AHEAD + 1][NT];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) load(k, offs[k], fa[k], fb[k]);
#pragma unroll
            for (int k = 0; k < STEPS; ++k) {
                if (k + AHEAD < STEPS) load(k + AHEAD, offs[k + AHEAD], fa[(k + AHEAD) % (AHEAD + 1)], fb[(k + AHEAD) % (AHEAD + 1)]);
                __builtin_amdgcn_sched_barrier(0);
                mult(fa[k % (AHEAD + 1)], fb[k % (AHEAD + 1)]);
            }
        } else {
            // two steps' operands, and the table entries of the two after them, are read ahead (past the last step: its own)
            v4i fa[3][MT], fb[3][NT];
            const int last = steps - 1;
            load(0, tab[lh], fa[0], fb[0]);
            load(min(1, last), tab[2 * min(1, last) + lh], fa[1], fb[1]);
            int o0 = tab[2 * min(2, last) + lh], o1 = tab[2 * min(3, last) + lh], o2 = tab[2 * min(4, last) + lh];
            for (int k = 0; k < steps; k += 3) {
                load(min(k + 2, last), o0, fa[2], fb[2]);
                o0 = tab[2 * min(k + 5, last) + lh];
                mult(fa[0], fb[0]);
                if (k + 1 >= steps) break;
                load(min(k + 3, last), o1, fa[0], fb[0]);
                o1 = tab[2 * min(k + 6, last) + lh];
                mult(fa[1], fb[1]);
                if (k + 2 >= steps) break;
                load(min(k + 4, last), o2, fa[1], fb[1]);
                o2 = tab[2 * min(k + 7, last) + lh];
                mult(fa[2], fb[2]);
            }
        }
        if (st + KS < a.nstages) store((st / KS + 1) & 1);
        __syncthreads();
    }

    if constexpr (KS == 2) {
        // Group 0 finishes the first two quads of channels of the block and group 1 the others: each hands the other's over.
        v16i& c = acc[0][0];
        const v4i give[2] = {kg ? v4i{c[0], c[1], c[2], c[3]} : v4i{c[8], c[9], c[10], c[11]},
                             kg ? v4i{c[4], c[5], c[6], c[7]} : v4i{c[12], c[13], c[14], c[15]}};
        v4i* x = lds_all + kg * 512 + t;
        x[0] = give[0];
        x[256] = give[1];
        __syncthreads();
        const v4i* y = lds_all + (kg ^ 1) * 512 + t;
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = (kg ? c[8 + i] : c[i]) + y[(i >> 2) * 256][i & 3];
        p4_finish<MT, NT, 2>(a, acc, oc0 + kg * 16, d_px, z_px, lh);
    } else {
        p4_finish(a, acc, oc0, d_px, z_px, lh);
    }
}
