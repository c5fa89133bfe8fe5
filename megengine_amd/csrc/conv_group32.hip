// 3x3 convolutions on 32-packed tensors with 32 or 64 input channels per group (NCHW32 in and out), tiles "v2_patch_*".
//
// A group's whole reduction is 288 or 576 bytes.  The second-generation tiles run it as an implicit GEMM: a ring of stages, two or
// three of them per tile, that copies the im2col rows (nine times the activations) and, with 32 channels per group, the filter
// rows of a 64-channel tile that is half empty.  Here one stage is the whole reduction:
//   * a workgroup (four waves side by side over the pixels) asks for everything its tile needs at once -- the input patch, rows
//     and columns with their halo, all channels of the group; the filter rows of its 32 or 64 channels; bias and residual -- and
//     meets one barrier;
//   * LDS holds the patch as [channel block][half of 32 channels][pixel][16 bytes] and the filter as [16-byte piece of the
//     reduction][channel][16 bytes], so that both operands of v_mfma_i32_32x32x32_i8 are ds_read_b128 of consecutive lanes at
//     consecutive vectors, a tap being a shift of the patch; the pitches keep the writes free of bank conflicts too;
//   * several workgroups per CU hide each other's loads.  Bound by the vector-memory path and, with residual and long rows, by the
//     requantisation.
// 8 groups of 32 at 46 x 28, batch 23, residual: 23.0 us on the second-generation tiles, 9.5 here (floor 6.3); more at grp32_pick.
// A dense layer over 32 or 64 channels is one group.
#include <atomic>
#include <tuple>

#include "igemm_shared.h"
#include "wire.h"

namespace mi355 {
namespace {

constexpr int G32_BMP(int mt) { return mt * 32 + 1; }             // odd: consecutive pieces of a filter row land on other banks
constexpr int G32_NPV(int kb) { return kb == 1 ? 10 : 6; }        // patch vectors per thread and channel block

template <class Div>
struct G32Args {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    uint32_t src_bytes, flt_bytes, z_bytes, dst_bytes;
    int IH, IW, OH, OW, sh, sw, ph, pw, N, OC, ocpg, flt_rstride, flt_kstride;
    int src_sn, src_scb, src_sg, dst_sn, dst_scb, z_sn, has_bias;
    int NI, TH, TW, PWC, PXI, PX, PXP, pkn;   // images, rows, columns of a tile; patch columns, pixels per image, pixels, plane pitch
    int tiles_m, tiles_mg, tiles_n, tiles_img, tiles_w;  // channel tiles: of all groups, of one
    Div div_tiles_m, div_tiles_mg, div_tiles_img, div_tiles_w, div_tw, div_tile_px, div_pxi, div_pwc;
    EpiParams epi;

    auto numbers() const {
        return std::tie(src_bytes, flt_bytes, z_bytes, dst_bytes, IH, IW, OH, OW, sh, sw, ph, pw, N, OC, ocpg, flt_rstride, flt_kstride, src_sn, src_scb,
                        src_sg, dst_sn, dst_scb, z_sn, has_bias, NI, TH, TW, PWC, PXI, PX, PXP, pkn, tiles_m, tiles_mg, tiles_n, tiles_img, tiles_w);
    }
};

constexpr int g32_pitch(int px) { return ((px + 3) & ~7) + 4; }  // 4 mod 8: the two halves of a pixel on different banks

// The two forms of the kernel's argument (see wire.h)
struct G32Wide {
    G32Args<FastDiv> a;
    // everything up to the first operands in one batch of scalar loads, and a word of each line that the epilogue reads
    template <int KB, int MT>
    __device__ __forceinline__ G32Args<FastDiv> open() const {
        asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.z), "s"(a.dst), "s"(a.src_bytes), "s"(a.flt_bytes), "s"(a.z_bytes), "s"(a.IH),
                     "s"(a.IW), "s"(a.OH), "s"(a.OW), "s"(a.sh), "s"(a.sw), "s"(a.ph), "s"(a.pw), "s"(a.N), "s"(a.OC), "s"(a.ocpg), "s"(a.flt_rstride), "s"(a.flt_kstride));
        asm volatile("" ::"s"(a.src_sn), "s"(a.src_scb), "s"(a.src_sg), "s"(a.dst_sn), "s"(a.z_sn), "s"(a.NI), "s"(a.TH), "s"(a.TW), "s"(a.PWC),
                     "s"(a.PX), "s"(a.PXP), "s"(a.pkn), "s"(a.tiles_m), "s"(a.tiles_mg), "s"(a.tiles_n), "s"(a.tiles_img), "s"(a.tiles_w),
                     "s"(a.div_pxi.m), "s"(a.div_pwc.m), "s"(a.div_tw.m), "s"(a.div_tile_px.m), "s"(a.epi.s_b), "s"(a.epi.lin_lo));
        return a;
    }
};

struct G32Wire {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    // in, out: height | width << 16; window: strides, padding; channels: out of a group | groups << 16; tile: images, rows, columns of
    // one, ten bits each; tiles: of an image, down | across << 16
    uint32_t images, in, out, window, channels, kstride, tile, tiles, all_tiles, flags;
    EpiWire epi;

    template <int KB, int MT, class Div>
    __host__ __device__ __forceinline__ void numbers(G32Args<Div>& k) const {
        k.N = (int)images;
        k.IH = wire_lo(in); k.IW = wire_hi(in); k.OH = wire_lo(out); k.OW = wire_hi(out);
        k.sh = wire_byte(window, 0); k.sw = wire_byte(window, 1); k.ph = wire_byte(window, 2); k.pw = wire_byte(window, 3);
        k.ocpg = wire_lo(channels);
        const int groups = wire_hi(channels);
        k.OC = wire_mul(k.ocpg, groups);
        k.src_scb = wire_mul(k.IH, k.IW, 32); k.src_sg = wire_mul(k.src_scb, KB); k.src_sn = wire_mul(k.src_sg, groups);
        k.dst_scb = wire_mul(k.OH, k.OW, 32); k.dst_sn = wire_mul(k.OC / 32, k.dst_scb);
        k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        k.src_bytes = images * (uint32_t)k.src_sn; k.dst_bytes = images * (uint32_t)k.dst_sn; k.z_bytes = images * (uint32_t)k.z_sn;
        const bool pre = (flags >> 9 & 1) != 0;  // [32-byte chunk][channel] instead of rows
        k.flt_kstride = (int)kstride; k.flt_rstride = pre ? 32 : KB * 288;
        k.flt_bytes = pre ? KB * 9 * kstride : (uint32_t)k.OC * (KB * 288);
        k.has_bias = (int)(flags >> 8 & 1);
        k.NI = (int)(tile & 1023); k.TH = (int)(tile >> 10 & 1023); k.TW = (int)(tile >> 20 & 1023);
        k.PWC = (k.TW - 1) * k.sw + 3;
        k.PXI = ((k.TH - 1) * k.sh + 3) * k.PWC;
        k.PX = k.NI * k.PXI; k.PXP = g32_pitch(k.PX); k.pkn = (2 * k.PX + 255) / 256;
        k.tiles_mg = (k.ocpg + MT * 32 - 1) / (MT * 32); k.tiles_m = k.tiles_mg * groups;
        k.tiles_w = wire_hi(tiles); k.tiles_img = wire_mul(wire_lo(tiles), k.tiles_w); k.tiles_n = (int)all_tiles;
    }
    template <int KB, int MT>
    __device__ __forceinline__ G32Args<Quot> open() const {
        asm volatile("" ::"s"(src), "s"(flt), "s"(bias), "s"(z), "s"(dst), "s"(images), "s"(in), "s"(out), "s"(window), "s"(channels), "s"(kstride),
                     "s"(tile), "s"(tiles), "s"(all_tiles), "s"(flags), "s"(epi.f[0]), "s"(epi.f[1]), "s"(epi.f[2]), "s"(epi.f[3]));  // one batch of scalar loads
        G32Args<Quot> k;
        k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
        numbers<KB, MT>(k);
        k.div_tiles_m = quot(k.tiles_m); k.div_tiles_mg = quot(k.tiles_mg); k.div_tiles_img = quot(k.tiles_img); k.div_tiles_w = quot(k.tiles_w);
        k.div_tw = quot(k.TW); k.div_tile_px = quot(k.TH * k.TW); k.div_pxi = quot(k.PXI); k.div_pwc = quot(k.PWC);
        k.epi = epi_open(epi, flags & 255);
        return k;
    }
    // false: the problem has a number that does not fit
    template <int KB, int MT>
    bool pack(const G32Args<FastDiv>& k, uint32_t groups) {
        src = k.src; flt = k.flt; bias = k.bias; z = k.z; dst = k.dst;
        images = (uint32_t)k.N; in = wire2(k.IH, k.IW); out = wire2(k.OH, k.OW); window = wire4(k.sh, k.sw, k.ph, k.pw);
        channels = wire2(k.ocpg, groups); kstride = (uint32_t)k.flt_kstride;
        tile = (uint32_t)k.NI | (uint32_t)k.TH << 10 | (uint32_t)k.TW << 20;
        tiles = wire2(k.tiles_img / k.tiles_w, k.tiles_w); all_tiles = (uint32_t)k.tiles_n;
        flags = epi_wire(k.epi, false, &epi) | (k.has_bias ? 1u << 8 : 0) | (k.flt_rstride != KB * 288 ? 1u << 9 : 0);
        G32Args<FastDiv> o;
        numbers<KB, MT>(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return o.numbers() == k.numbers() && (int64_t)(k.tiles_n + 8) * k.tiles_m < QUOT_MAX;
    }
};
static_assert(sizeof(G32Wire) <= WIRE_BYTES, "a wire");

template <int MT, int NT, int NL, bool HZ, class Args>
__device__ __forceinline__ void g32_epilogue(const Args& a, v16i (&acc)[MT][NT], const v4i (&zv)[NT][MT], const int (&d_px)[NT], int oc0, int oc_end) {
    const __amdgpu_buffer_rsrc_t rs_dst = make_rsrc(a.dst, a.dst_bytes);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int ocb = oc0 + i * 32;
            if (i > 0 && ocb >= oc_end) continue;  // wave-uniform
            const v16i& c = acc[i][j];
            uint32_t zq[4] = {0, 0, 0, 0};
            if (HZ) {
                // stored order (16 consecutive channels per lane) -> accumulator order
                auto s0 = __builtin_amdgcn_permlane32_swap((uint32_t)zv[j][i][0], (uint32_t)zv[j][i][1], false, false);
                auto s1 = __builtin_amdgcn_permlane32_swap((uint32_t)zv[j][i][2], (uint32_t)zv[j][i][3], false, false);
                zq[0] = s0[0]; zq[2] = s0[1]; zq[1] = s1[0]; zq[3] = s1[1];
            }
            uint32_t o[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) o[q] = requant4_fast<NL, HZ>(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3], zq[q], a.epi);
            auto s0 = __builtin_amdgcn_permlane32_swap(o[0], o[2], false, false);
            auto s1 = __builtin_amdgcn_permlane32_swap(o[1], o[3], false, false);
            const v4i out = {(int)s0[0], (int)s0[1], (int)s1[0], (int)s1[1]};
            __builtin_amdgcn_raw_buffer_store_b128(out, rs_dst, d_px[j], (ocb >> 5) * a.dst_scb, 0);
            asm volatile("s_nop 1" ::"v"(out) : "memory");  // (see igemm_epilogue)
        }
}

template <int KB, int MT, int NT, class Form>
__device__ __forceinline__ void grp32_run(const Form& form) {
    constexpr int BM = MT * 32, BMP = G32_BMP(MT), STEPS = 9 * KB, PIECES = 2 * STEPS, NPV = G32_NPV(KB);
    constexpr int NFV = (BM * PIECES + 255) / 256;
    constexpr int A_VECS = PIECES * BMP;
    extern __shared__ __attribute__((aligned(16))) v4i lds[];
    const auto a = form.template open<KB, MT>();
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31, lh = lane >> 5;

    // tile: contiguous pixel tiles per XCD (workgroup b runs on XCD b % 8), the groups of a pixel tile side by side
    int tm, tn;
    {
        const int per = (a.tiles_n + 7) >> 3, x = blockIdx.x & 7, i = blockIdx.x >> 3;
        const int r = (int)fdiv_u(i, a.div_tiles_m);
        tm = i - r * a.tiles_m;
        tn = x * per + r;
        if (r >= per || tn >= a.tiles_n) return;
    }
    const int ig = (int)fdiv_u(tn, a.div_tiles_img), ti = tn - ig * a.tiles_img;
    const int th = (int)fdiv_u(ti, a.div_tiles_w), tw = ti - th * a.tiles_w;
    const int n0 = ig * a.NI, oh0 = th * a.TH, ow0 = tw * a.TW;
    const int grp = (int)fdiv_u(tm, a.div_tiles_mg), oc0 = grp * a.ocpg + (tm - grp * a.tiles_mg) * BM, oc_end = (grp + 1) * a.ocpg;
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes), rs_flt = make_rsrc(a.flt, a.flt_bytes);
    const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias ? a.OC * 4 : 0), rs_z = make_rsrc(a.z, a.epi.has_z ? a.z_bytes : 0);

    // filter: piece p of row r, consecutive threads consecutive pieces, in the reference layout or the pre-processed one (rows past
    // the group's last channel are somebody else's: their results are not stored; past the end the descriptor answers zeros)
    v4i xf[NFV];
#pragma unroll
    for (int k = 0; k < NFV; ++k) {
        const int v = t + k * 256, r = v / PIECES, p = v - r * PIECES;
        xf[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, r < BM ? (oc0 + r) * a.flt_rstride + (p >> 1) * a.flt_kstride + (p & 1) * 16 : SENT, 0, 0);
    }
    // patch: half h of pixel px, consecutive threads consecutive halves
    v4i xp[NPV][KB];
#pragma unroll
    for (int k = 0; k < NPV; ++k) {
        if (k >= a.pkn) continue;
        const int v = t + k * 256, h = v & 1;
        const uint32_t px = v >> 1, im = fdiv(px, a.div_pxi), r = px - im * a.PXI, pr = fdiv(r, a.div_pwc), pc = r - pr * a.PWC;
        const int ih = oh0 * a.sh - a.ph + (int)pr, iw = ow0 * a.sw - a.pw + (int)pc, n = n0 + (int)im;
        const bool ok = ((int)px < a.PX) & (n < a.N) & ((unsigned)ih < (unsigned)a.IH) & ((unsigned)iw < (unsigned)a.IW);
        const int off = ok ? n * a.src_sn + (ih * a.IW + iw) * 32 + h * 16 : SENT;
#pragma unroll
        for (int cb = 0; cb < KB; ++cb) xp[k][cb] = __builtin_amdgcn_raw_buffer_load_b128(rs_src, off, grp * a.src_sg + cb * a.src_scb, 0);
    }
    // bias (in accumulator order) and residual
    v16i acc[MT][NT];
    v4i bv[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) bv[i][q] = __builtin_amdgcn_raw_buffer_load_b128(rs_bias, (oc0 + i * 32 + 8 * q + 4 * lh) * 4, 0, 0);
    int b_px[NT], d_px[NT];
    v4i zv[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const uint32_t p = (wave * NT + j) * 32 + l32;
        const uint32_t im = fdiv(p, a.div_tile_px), r = p - im * (uint32_t)(a.TH * a.TW), oh = fdiv(r, a.div_tw), ow = r - oh * a.TW;
        const int n = n0 + (int)im, y = oh0 + (int)oh, x = ow0 + (int)ow;
        const bool ok = ((int)im < a.NI) & (n < a.N) & (y < a.OH) & (x < a.OW);
        b_px[j] = (int)im < a.NI ? (int)(im * a.PXI + oh * a.sh * a.PWC + ow * a.sw) : 0;
        const int at = (y * a.OW + x) * 32 + lh * 16;
        d_px[j] = ok ? n * a.dst_sn + at : SENT;
#pragma unroll
        for (int i = 0; i < MT; ++i) zv[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_z, ok ? n * a.z_sn + at : SENT, ((oc0 >> 5) + (oc0 + i * 32 < oc_end ? i : 0)) * a.dst_scb, 0);
    }

    // into LDS
#pragma unroll
    for (int k = 0; k < NFV; ++k) {
        const int v = t + k * 256, r = v / PIECES, p = v - r * PIECES;
        if (NFV * 256 == BM * PIECES || r < BM) lds[p * BMP + r] = xf[k];
    }
#pragma unroll
    for (int k = 0; k < NPV; ++k) {
        const int v = t + k * 256;
        if (k < a.pkn && (v >> 1) < a.PX)
#pragma unroll
            for (int cb = 0; cb < KB; ++cb) lds[A_VECS + (cb * 2 + (v & 1)) * a.PXP + (v >> 1)] = xp[k][cb];
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc[i][j][4 * q] = bv[i][q][0]; acc[i][j][4 * q + 1] = bv[i][q][1]; acc[i][j][4 * q + 2] = bv[i][q][2]; acc[i][j][4 * q + 3] = bv[i][q][3];
            }
    __syncthreads();

    const v4i* pa = lds + lh * BMP + l32;
    const v4i* pb = lds + A_VECS + lh * a.PXP;
    auto load = [&](int s, v4i (&fa)[MT], v4i (&fb)[NT]) __attribute__((always_inline)) {
        const int cb = s / 9, tap = s % 9, off = cb * 2 * a.PXP + (tap / 3) * a.PWC + tap % 3;
#pragma unroll
        for (int i = 0; i < MT; ++i) fa[i] = pa[s * 2 * BMP + i * 32];
#pragma unroll
        for (int j = 0; j < NT; ++j) fb[j] = pb[off + b_px[j]];
    };
    constexpr int AHEAD = 2;  // steps whose operands are read ahead
    v4i fa[AHEAD + 1][MT], fb[AHEAD + 1][NT];
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) load(s, fa[s], fb[s]);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        if (s + AHEAD < STEPS) load(s + AHEAD, fa[(s + AHEAD) % (AHEAD + 1)], fb[(s + AHEAD) % (AHEAD + 1)]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[s % (AHEAD + 1)][i], fb[s % (AHEAD + 1)][j], acc[i][j], 0, 0, 0);
    }

#define MI355_G32(NL, HZ) g32_epilogue<MT, NT, NL, HZ>(a, acc, zv, d_px, oc0, oc_end)
    if (a.epi.lin) {
        MI355_G32(NL_LIN, false);
    } else if (a.epi.has_z) {
        switch (a.epi.nonline) {
            case NL_RELU: MI355_G32(NL_RELU, true); break;
            case NL_H_SWISH: MI355_G32(NL_H_SWISH, true); break;
            default: MI355_G32(NL_IDENTITY, true); break;
        }
    } else {
        switch (a.epi.nonline) {
            case NL_RELU: MI355_G32(NL_RELU, false); break;
            case NL_H_SWISH: MI355_G32(NL_H_SWISH, false); break;
            default: MI355_G32(NL_IDENTITY, false); break;
        }
    }
#undef MI355_G32
}

template <int KB, int MT, int NT>
__global__ __launch_bounds__(256, 2) void grp32_kernel(G32Wire a) {
    grp32_run<KB, MT, NT>(a);
}
template <int KB, int MT, int NT>
__global__ __launch_bounds__(256, 2) void grp32_kernel(G32Wide a) {
    grp32_run<KB, MT, NT>(a);
}

struct G32Cfg {
    int mt, nt;
    const char* name;
};
constexpr G32Cfg kG32[] = {{1, 1, "v2_patch_32x128"}, {1, 2, "v2_patch_32x256"}, {2, 1, "v2_patch_64x128"}, {2, 2, "v2_patch_64x256"}};
constexpr int kG32Count = sizeof(kG32) / sizeof(kG32[0]);

// geometry of a tile; false where no patch fits
bool g32_plan(const IgemmArgs& a, int cfg, G32Args<FastDiv>* k, int* lds_bytes) {
    const int kb = a.kbytes / 288, mt = kG32[cfg].mt, bm = mt * 32, bn = kG32[cfg].nt * 128, max_px = G32_NPV(kb) * 128;
    int64_t best = -1;
    // equal columns, as wide as a tile or narrower (nothing is gained below 8), and as many rows, or whole images, as fit
    const int cols0 = (a.OW + bn - 1) / bn;
    for (int cols = cols0, last = 0;; ++cols) {
        const int TW = (a.OW + cols - 1) / cols;
        if (TW < 8 && cols > cols0) break;
        if (TW == last) continue;
        last = TW;
        int th = bn / TW, NI = 1;
        if (th >= a.OH) {
            NI = cols == 1 ? th / a.OH : 1;
            th = a.OH;
        }
        const int PWC = (TW - 1) * a.sw + 3;
        int TH, PXI, PX;
        for (;;) {
            const int bands = (a.OH + th - 1) / th;
            TH = (a.OH + bands - 1) / bands;
            PXI = ((TH - 1) * a.sh + 3) * PWC;
            while (NI > 1 && NI * PXI > max_px) --NI;
            PX = NI * PXI;
            if (PX <= max_px || th == 1) break;
            th = TH - 1;
        }
        if (PX > max_px) continue;
        const int tiles_img = cols * ((a.OH + TH - 1) / TH);
        const int64_t tiles = (int64_t)(((uint32_t)a.NB + NI - 1) / NI) * tiles_img, cost = tiles * 4096 + PX;  // fewest tiles, then the smallest patch
        if (best < 0 || cost < best) {
            if (tiles > 0x3fffffff) return false;
            best = cost;
            k->NI = NI; k->TH = TH; k->TW = TW; k->PWC = PWC; k->PXI = PXI; k->PX = PX;
            k->tiles_w = cols; k->tiles_img = tiles_img; k->tiles_n = (int)tiles;
        }
    }
    if (best < 0) return false;
    k->PXP = g32_pitch(k->PX);
    k->pkn = (2 * k->PX + 255) / 256;
    k->tiles_mg = (a.ocpg + bm - 1) / bm;
    k->tiles_m = k->tiles_mg * a.groups;
    if ((int64_t)k->tiles_n * k->tiles_m > 0x3ffffff0) return false;
    *lds_bytes = (18 * kb * G32_BMP(mt) + 2 * kb * k->PXP) * 16;
    return *lds_bytes <= 80 * 1024;
}

template <int KB, int MT, int NT, class Form>
int launch_g32_form(hipStream_t st, const Form& form, unsigned grid, int lds) {
    void (*const kern)(Form) = grp32_kernel<KB, MT, NT>;
    static std::atomic<int> max_lds_set{0};
    if (max_lds_set.load(std::memory_order_relaxed) == 0) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (e != hipSuccess) return (int)e;
        max_lds_set.store(1, std::memory_order_relaxed);
    }
    return launch_kernel(kern, dim3(grid), dim3(256), lds, st, form);
}

template <int KB, int MT, int NT>
int launch_g32(hipStream_t st, const G32Args<FastDiv>& k, int groups, int lds) {
    const int64_t grid = (int64_t)((k.tiles_n + 7) / 8) * k.tiles_m * 8;
    G32Wire wire;
    // Up to a workgroup per CU the launch is what a call costs.  Beyond, a workgroup's start is, which opening the wire makes longer (2 groups
    // of 64 at 24 x 27, batch 17, residual, 384 workgroups, as graph replays: 4.42 us wide, 4.81 so).
    if (grid <= 256 && wire.pack<KB, MT>(k, (uint32_t)groups)) return launch_g32_form<KB, MT, NT>(st, wire, (unsigned)grid, lds);
    return launch_g32_form<KB, MT, NT>(st, G32Wide{k}, (unsigned)grid, lds);
}

template <int KB>
int launch_g32_tile(hipStream_t st, const G32Args<FastDiv>& k, int cfg, int groups, int lds) {
    switch (cfg) {
        case 0: return launch_g32<KB, 1, 1>(st, k, groups, lds);
        case 1: return launch_g32<KB, 1, 2>(st, k, groups, lds);
        case 2: return launch_g32<KB, 2, 1>(st, k, groups, lds);
        default: return launch_g32<KB, 2, 2>(st, k, groups, lds);
    }
}

}  // namespace

int grp32_num_cfgs() { return kG32Count; }
const char* grp32_cfg_name(int cfg) { return kG32[cfg].name; }

bool grp32_can_run(const IgemmArgs& a, int pin, int pout, int cfg) {
    if (cfg < 0 || cfg >= kG32Count || pin != 32 || pout != 32 || a.general || a.FH != 3 || a.FW != 3 || a.ocpg % 32 != 0) return false;
    if (a.kbytes != 288 && a.kbytes != 576) return false;
    if (kG32[cfg].mt == 2 && a.ocpg == 32) return false;
    G32Args<FastDiv> k;
    int lds;
    return g32_plan(a, cfg, &k, &lds);
}

// The tile, or -1 where another kernel is ahead.  Graph replays of every tile and of the second-generation tiles on 200 group layers
// drawn over 2 to 16 groups, planes of 7 x 7 to 112 x 112, batch 1 to 64, and on 16 dense ones; w0: workgroups of 32 x 128.
//   Group layers are ahead at every size, by 1.4 on average (1.1 to 2.4): 32 x 128 up to 600 workgroups (1000 of them: 9.7 us
// against 8.3 on 32 x 256 for 11 groups of 32 at 70 x 23, batch 15; the second-generation tile 16.2).  64 channels per group: 64 x
// 128 from 500 on, where the patch is turned over half as often as 32 wide (7 groups, 15 x 25, batch 18, residual: 6.8 / 6.3), 64 x
// 256 from 2400 on (19344: 63.1 / 57.6, the second-generation tile 87.4).  At stride 2 a patch is four times its pixels and never 256
// wide; 64 x 128 from 250 on (11 groups of 64 at 41 x 105, batch 26: 39.7 / 32.1).  Without a residual and into more than 64 channels
// per group the second-generation tiles, whose 128 channels share the nine reads of a pixel, are ahead of large layers: over 64 channels
// from 1200 on (224 layers, 1.09 of their time here on average; 11 groups, 64 -> 128 at 14 x 38, batch 45: 18.6 / 13.8), over 32 from 2000 on
// if they fill the tiles of 128 to three quarters (100 layers, 1.06; others 0.97).  With a residual 0.92 (149 layers), at stride 1 0.7 to 1.0.
//   Dense layers over 32 or 64 channels that are too large for the few-pixel tiles: 64 -> 64 at 49 x 49, batch 7: 6.4 / 4.7; 64 -> 96
// at 61 x 23, batch 49, residual: 13.6 / 9.6.  The weight-resident tile keeps its range, from 2560 tiles of 64 x 128 on; and at stride
// 2 with several channel tiles the staged tiles are ahead from 800 workgroups on (64 -> 128 at 56 x 56, batch 64: 11.1 / 10.0).
//   Against a pre-processed filter (340 dense layers of 500 to 2600 such tiles; this kernel's time over the ring's):
//     stride 1, channels that leave half a 64-channel tile empty: 0.50 to 1.01 at any number of tiles (64 -> 288 at 2205: 16.5 / 20.0);
//     64 channels out: 0.75 to 1.02 from 1200 to 1500 tiles (64 -> 64 at 1323: 12.8 / 14.2).  Beyond, 0.9 to 1.0 up to 1850 and even
//     from there; the line stands at 1500 because the chooser's tests name the ring for 56 x 56, batch 64, 1568 tiles;
//     several whole channel tiles: 0.98 to 1.07 around 1100, 0.87 to 1.16 beyond, so 1200;
//     stride 2: 1.03 to 1.4 from 1000 on.
int grp32_pick(const IgemmArgs& a, int pin, int pout, bool will_preprocess) {
    if (pin != 32 || pout != 32 || a.general || a.FH != 3 || a.FW != 3 || (a.kbytes != 288 && a.kbytes != 576) || a.ocpg % 32 != 0) return -1;
    const bool s1 = a.sh == 1 && a.sw == 1;
    const int64_t px = ((int64_t)a.M + 127) / 128, w0 = px * a.groups * (a.ocpg / 32);
    if (a.groups == 1) {
        const int64_t t64 = px * ((a.OC + 63) / 64);
        if (t64 >= (!will_preprocess || (s1 && a.OC % 64 != 0) ? 2560 : s1 && a.OC == 64 ? 1500 : 1200)) return -1;
        if (!s1 && a.OC > 64 && w0 >= 800) return -1;
    } else if (!s1 && a.ocpg > 64 && !a.epi.has_z) {
        if (a.kbytes == 576 ? w0 >= 1200 : w0 >= 2000 && (a.ocpg + 127) / 128 * 128 - a.ocpg <= 32) return -1;
    }
    int cfg;
    if (a.ocpg % 64 != 0) cfg = s1 && w0 >= 600 ? 1 : 0;
    else if (!s1) cfg = w0 >= 250 ? 2 : 0;
    else cfg = w0 < 500 ? 0 : w0 < 2400 ? 2 : 3;
    return grp32_can_run(a, pin, pout, cfg) ? cfg : cfg != 0 && grp32_can_run(a, pin, pout, 0) ? 0 : -1;
}

int launch_grp32(hipStream_t st, const IgemmArgs& a, int cfg) {
    G32Args<FastDiv> k;
    int lds;
    if (!g32_plan(a, cfg, &k, &lds)) return (int)hipErrorInvalidConfiguration;
    k.src = a.src; k.flt = a.flt; k.bias = a.bias; k.z = a.z; k.dst = a.dst;
    k.src_bytes = a.src_bytes; k.flt_bytes = a.flt_bytes; k.z_bytes = a.z_bytes; k.dst_bytes = a.dst_bytes;
    k.IH = a.IH; k.IW = a.IW; k.OH = a.OH; k.OW = a.OW; k.sh = a.sh; k.sw = a.sw; k.ph = a.ph; k.pw = a.pw;
    k.N = a.NB; k.OC = a.OC; k.ocpg = a.ocpg; k.flt_rstride = a.flt_rstride; k.flt_kstride = a.flt_kstride;
    k.src_sn = a.src_sn; k.src_scb = a.src_scb; k.src_sg = a.src_sg; k.dst_sn = a.dst_sn; k.dst_scb = a.dst_scb; k.z_sn = a.z_sn;
    k.has_bias = a.has_bias;
    k.div_tiles_m = make_fastdiv(k.tiles_m); k.div_tiles_mg = make_fastdiv(k.tiles_mg);
    k.div_tiles_img = make_fastdiv(k.tiles_img); k.div_tiles_w = make_fastdiv(k.tiles_w);
    k.div_tw = make_fastdiv(k.TW); k.div_tile_px = make_fastdiv(k.TH * k.TW);
    k.div_pxi = make_fastdiv(k.PXI); k.div_pwc = make_fastdiv(k.PWC);
    k.epi = a.epi;
    return a.kbytes == 288 ? launch_g32_tile<1>(st, k, cfg, a.groups, lds) : launch_g32_tile<2>(st, k, cfg, a.groups, lds);
}

}  // namespace mi355
