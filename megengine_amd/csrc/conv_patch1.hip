// Plain NCHW convolutions in one launch, no workspace: the input patch and the filter are turned on their way into LDS.
//
// The matrix cores want sixteen reduction bytes side by side, and an NCHW tensor keeps every channel in a plane of its own.
// Packing it in a launch ahead of the convolution (conv_nchw.hip) costs that launch, the gap behind it, a round trip through
// memory and the padding of 75 channels to 96.  Here a workgroup stages the patch of its tile -- rows and columns with their halo, sixteen
// channels at a time -- as [group of 16 channels][patch pixel][16 bytes], as the 4-packed patch kernel does (conv_patch4.hip),
// so that the operand of a tap is one ds_read_b128 at a shifted pixel:
//   * A thread takes four neighbouring pixels of sixteen channels: sixteen dword loads at any address, consecutive lanes
//     consecutive dwords of a row, and turns them with v_perm into four 16-byte vectors.  The selectors of v_perm are per lane
//     and made once per tile: they put zeros where a column lies outside the image, move the bytes of a dword that was loaded
//     further left because the row ends inside it, and turn the order of the four pixels by lane, so that the 16-byte writes of
//     eight lanes meet eight different bank groups.
//   * The filter's rows are [channel][tap] bytes: a thread takes four channels of a row, 4 T contiguous bytes, and T times three
//     v_perm with constant selectors make the T dwords (four channels of one tap) that an operand is made of.
//   * A tile is rows and columns, or a run of pixels in the order of memory (p1_run says where), whose rows end wherever they do.
//   * Two stages in LDS, the next one's loads in registers while the current one is multiplied, one barrier per stage.
//   * Bound by LDS, as the 4-packed patch tiles are, and by the latency of a stage where tiles are few.
// Filters of 1x1, 3x3 and 5x5; others go through the
// workspace.  Graph replays: 75 -> 150 channels, 3x3 at 61 x 45, batch 6, with a residual: 16.6 us packed, 11.1 here (four waves of
// 1200 vector instructions for 23 products each, a third of their time waiting for a stage's loads); more at p1_tile.
#include <algorithm>
#include <atomic>

#include "igemm_shared.h"
#include "relayout_parts.h"

namespace mi355 {
namespace {

constexpr int P1_NPI = 2;          // pixel quads per thread and stage
constexpr int P1_VMCNT0 = 0x0f70;  // s_waitcnt vmcnt(0), the other counters at their maxima

constexpr int p1_gs(int t) { return t == 1 ? 4 : t == 9 ? 2 : 1; }  // channel groups of a stage
constexpr int p1_f(int t) { return t == 1 ? 1 : t == 9 ? 3 : 5; }
constexpr int p1_bmp(int mt) { return mt * 32 + 1; }  // odd: the dword writes of a filter row spread over the banks

struct P1Args {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    int IC, IH, IW, IHW, OC, OH, OW, OHW, N, sh, sw, ph, pw;
    int src_sn, dst_sn, z_sn, kbytes, flt_bytes, has_bias, nstages;
    uint32_t src_bytes, dst_bytes, z_bytes;
    int NI, TH, TW, tile_px, PWC, PXI, PX, PXQ;  // images, rows, columns of a tile; its pixels of an image; patch columns (a multiple of 4), pixels per image, pixels, quads
    int tiles_m, tiles_n, tiles_img, tiles_w;
    int run;  // not zero: a tile is that many pixels in the order of memory (TW = OW), zero: TH rows of TW columns
    FastDiv div_tiles_m, div_tiles_img, div_tiles_w, div_tw, div_tile_px, div_pqi, div_pqw;
    EpiParams epi;
};

typedef uint32_t u32_at __attribute__((aligned(1)));

// byte b of 4 T contiguous bytes
template <int T>
__device__ __forceinline__ uint32_t p1_tap(const uint32_t (&x)[T], int tap) {
    const int b0 = tap, b1 = T + tap, b2 = 2 * T + tap, b3 = 3 * T + tap;
    const uint32_t lo = __builtin_amdgcn_perm(x[b1 >> 2], x[b0 >> 2], (uint32_t)(0x0c0c0400 | (b0 & 3) | (b1 & 3) << 8));
    const uint32_t hi = __builtin_amdgcn_perm(x[b3 >> 2], x[b2 >> 2], (uint32_t)(0x04000c0c | (b2 & 3) << 16 | (b3 & 3) << 24));
    return lo | hi;
}

// where a tile begins: image, row and column out; skip: columns of the first row that are the tile's before
struct P1Tile {
    int n0, oh0, ow0, skip;
};
__host__ __device__ __forceinline__ P1Tile p1_tile_at(const P1Args& a, int tn) {
    const int ig = (int)fdiv(tn, a.div_tiles_img), ti = tn - ig * a.tiles_img;
    const bool is_run = a.run != 0;
    const int at = is_run ? ti * a.run : ti, th = (int)fdiv(at, a.div_tiles_w), tw = at - th * a.tiles_w;  // (a run: row and column)
    return {ig * a.NI, is_run ? th : th * a.TH, is_run ? 0 : tw * a.TW, is_run ? tw : 0};
}

// where four neighbouring lanes put (and find the residual of) their four columns: offset of channel ch = 4 lh + l32 % 4 of the
// first eight channels, and the columns from there to the end of the row, or of the image for a run (0: nothing)
struct P1Out {
    int d0, z0, cols;
};
__host__ __device__ __forceinline__ P1Out p1_out(const P1Args& a, const P1Tile& o, int p, int ch) {
    const uint32_t im = fdiv(p, a.div_tile_px), r = p - im * (uint32_t)a.tile_px + o.skip, oh = fdiv(r, a.div_tw), ow = r - oh * a.TW;
    const bool in = ((int)im < a.NI) & (o.n0 + (int)im < a.N) & (o.oh0 + (int)oh < a.OH);
    const int at = (o.oh0 + (int)oh) * a.OW + o.ow0 + (int)ow, px = at + ch * a.OHW;
    return {(o.n0 + (int)im) * a.dst_sn + px, (o.n0 + (int)im) * a.z_sn + px, in ? a.run ? a.OHW - at : a.OW - (o.ow0 + (int)ow) : 0};
}

// Where a lane loads the residual of its four columns, and how far it turns the dword: a group that the row's end cuts short is loaded as the
// dword that ends there, or begins with the plane, and not byte by byte, three loads to be waited for behind the store before them.  Of 300
// drawn layers those with a residual take 0.944 of the time, the others the same (1x1 27 -> 37 at 83 x 93, stride 2, batch 14: 7.40 -> 6.02 us;
// 3x3 11 -> 41 at 70 x 13, stride 2, batch 10: 5.43 -> 4.58).  (Planes of fewer than four bytes hold no dword: p1_residual_across on the largest tile,
// which has many, p1_residual_bytes on the others.)
struct P1Residual {
    int off, turn;
};
__host__ __device__ __forceinline__ P1Residual p1_residual_at(const P1Args& a, const P1Out& w) {
    const int at = w.cols >= 4 ? w.z0 : max(w.z0 + w.cols - 4, 0);
    const bool in = (w.cols > 0) & (a.OHW >= 4);
    return {in ? at : SENT, in ? (w.z0 - at) * 8 : 0};
}
// What an access to channel oc8 + ch passes beside its offset of the first eight channels, by the rule at SENT: SENT, to be or'ed to that offset, in
// a lane without a channel, and a scalar offset that does not lead out of the tensor.  (One minimum and no selection: with the scalar offset
// chosen and a mask for each store, 200 drawn layers without a residual took 1.006 of the time.)
struct P1Access {
    int lane, scalar;
};
__host__ __device__ __forceinline__ P1Access p1_access(const P1Args& a, int oc8, int ch) {
    const int oc = min(oc8, a.OC);
    int left = a.OC - oc;
#ifdef __HIP_DEVICE_COMPILE__
    asm("" : "+s"(left));  // (or the masks of a whole tile are made at once and kept, and scalar registers spill)
#endif
    return {ch < left ? 0 : SENT, oc * a.OHW};
}
// The residual in planes of fewer than four bytes, which hold no dword, in a tensor that does: the dword that ends with the group or begins with
// the tensor, by the whole offset, which the lane's part does not tell.
__host__ __device__ __forceinline__ P1Residual p1_residual_across(const P1Out& w, const P1Access& at) {
    const int off = w.z0 + at.scalar, start = max(off + w.cols - 4, 0);
    return {w.cols > 0 ? at.lane | start : SENT, (off - start) * 8 & 31};
}
template <int MT, int NT, int QN>
__device__ __forceinline__ void p1_residual_bytes(const P1Args& a, uint32_t (&zq)[NT][MT][QN], const P1Tile& o, int oc0, int wave, int l32, int lh) {
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z, a.z_bytes);
    const int ch = 4 * lh + (l32 & 3);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const P1Out w = p1_out(a, o, (wave * NT + j) * 32 + (l32 & ~3), ch);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < QN; ++q) {
                const P1Access at = p1_access(a, oc0 + i * 32 + 8 * q, ch);
                zq[j][i][q] = 0;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const int off = k < w.cols ? w.z0 + k : SENT;
                    zq[j][i][q] |= (uint32_t)(uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rs_z, at.lane | off, at.scalar, 0) << (8 * k);
                }
            }
    }
}

// the residual of a wave's outputs, in flight at once; ch: the lane's channel of eight
template <int MT, int NT, int QN>
__device__ __forceinline__ void p1_residual(const P1Args& a, uint32_t (&zq)[NT][MT][QN], const P1Residual (&z)[NT], int oc0, int ch) {
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z, a.z_bytes);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < QN; ++q) {
                const P1Access at = p1_access(a, oc0 + i * 32 + 8 * q, ch);
                zq[j][i][q] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_z, at.lane | z[j].off, at.scalar, 0);
            }
}
// The same for the largest tile, where it is asked for behind the products.  (Planes of fewer than four bytes: 8192 images of 64 channels, 3 x 4
// -> 256, 3x3, take 66 us by single bytes, 80 on the smaller tiles, 52 so.)
template <int MT, int NT, int QN>
__device__ __forceinline__ void p1_residual_late(const P1Args& a, uint32_t (&zq)[NT][MT][QN], const P1Tile& o, int oc0, int wave, int l32, int lh) {
    const int ch = 4 * lh + (l32 & 3);
    P1Out w[NT];
    P1Residual z[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        w[j] = p1_out(a, o, (wave * NT + j) * 32 + (l32 & ~3), ch);
        z[j] = p1_residual_at(a, w[j]);
    }
    if (a.OHW >= 4) return p1_residual<MT, NT, QN>(a, zq, z, oc0, ch);
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z, a.z_bytes);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < QN; ++q) {
                const P1Residual at = p1_residual_across(w[j], p1_access(a, oc0 + i * 32 + 8 * q, ch));
                zq[j][i][q] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_z, at.off, 0, 0) >> at.turn;
            }
}

// QN: eights of channels of each block of 32 that are in acc (all four, or two)
template <int MT, int NT, int QN, int NL, bool HZ>
__device__ __forceinline__ void p1_epilogue(const P1Args& a, v16i (&acc)[MT][NT], const uint32_t (&zq)[NT][MT][QN], const P1Tile& o, int oc0,
                                            int wave, int l32, int lh) {
    const __amdgpu_buffer_rsrc_t rs_dst = make_rsrc(a.dst, a.dst_bytes);
    const int lane4 = l32 & 3, ch = 4 * lh + lane4;  // after the exchange a lane holds four columns of channel ch of every eight
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const P1Out w = p1_out(a, o, (wave * NT + j) * 32 + (l32 & ~3), ch);
        const int d0 = w.d0, cols = w.cols, turn = p1_residual_at(a, w).turn;
        const bool part = (cols > 0) & (cols < 4), split = __builtin_amdgcn_ballot_w64(part) != 0;
        const int four = cols >= 4 ? d0 : SENT, two = (part & (cols >= 2)) ? d0 : SENT,
                  one = (part & ((cols & 1) != 0)) ? d0 + (cols & 2) : SENT;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < QN; ++q) {
                const int oc8 = oc0 + i * 32 + 8 * q;  // wave-uniform
                uint32_t zw = 0;
                if (HZ) {
                    zw = zq[j][i][q] >> turn;
                    zw = quad_transpose(zw, lane4);
                }
                const v16i& c = acc[i][j];
                const uint32_t y = quad_transpose(requant4_fast<NL, HZ>(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3], zw, a.epi), lane4);
                const P1Access to = p1_access(a, oc8, ch);
                __builtin_amdgcn_raw_buffer_store_b32((int)y, rs_dst, to.lane | four, to.scalar, 0);
                if (split) {
                    __builtin_amdgcn_raw_buffer_store_b16((uint16_t)y, rs_dst, to.lane | two, to.scalar, 0);
                    __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(cols == 3 ? y >> 16 : y), rs_dst, to.lane | one, to.scalar, 0);
                }
            }
    }
}

namespace one {
constexpr int KS = 1;
#include "patch1_kernel.h"
}  // namespace one
namespace two {
constexpr int KS = 2;
#include "patch1_kernel.h"
}  // namespace two

constexpr int kP1Tiles[][2] = {{1, 1}, {1, 2}, {2, 2}, {2, 1}};  // 32 x 128, 32 x 256, 64 x 256, 64 x 128

// geometry of a tile; false where no patch fits
bool p1_plan(const ConvProblem& p, int tile, P1Args* k, int* lds_bytes) {
    const mi355_conv_desc& d = p.d;
    const int T = (int)(d.fh * d.fw), F = (int)d.fw, GS = p1_gs(T), mt = kP1Tiles[tile][0], bm = mt * 32, bn = kP1Tiles[tile][1] * 128;
    const int OH = (int)p.oh, OW = (int)p.ow, sh = (int)d.stride_h, sw = (int)d.stride_w, max_q = P1_NPI * (256 / GS);
    const int G = ((int)d.ic + 15) / 16;
    k->nstages = (G + GS - 1) / GS;
    int64_t best = -1;
    // equal columns of whole quads, as wide as the tile or narrower; rows (of whole images where one is small) as they fit
    const int cols0 = (OW + bn - 1) / bn;
    for (int parts = cols0, last = 0;; ++parts) {
        const int TW = ((OW + parts - 1) / parts + 3) & ~3, cols = (OW + TW - 1) / TW;
        if (TW < 16 && parts > cols0) break;
        if (TW == last) continue;
        last = TW;
        // patch columns: the first is rounded down to a multiple of four, whatever the tile's position
        const int PWC = ((TW - 1) * sw + F + 3 + 3) & ~3;
        int th = bn / TW, NI = 1;
        if (th >= OH) {
            NI = TW >= OW ? th / OH : 1;
            th = OH;
        }
        int TH, PXI, PXQ;
        for (;;) {
            const int bands = (OH + th - 1) / th;
            TH = (OH + bands - 1) / bands;
            PXI = ((TH - 1) * sh + F) * PWC;
            while (NI > 1 && NI * PXI / 4 > max_q) --NI;
            PXQ = NI * PXI / 4;
            if (PXQ <= max_q || th == 1) break;
            th = TH - 1;
        }
        if (PXQ <= max_q) {
            const int64_t tiles = ((int64_t)d.n + NI - 1) / NI * cols * ((OH + TH - 1) / TH);
            // fewest tiles; among those the smallest patch
            const int64_t cost = tiles * 4096 + PXQ;
            if (best < 0 || cost < best) {
                best = cost;
                k->NI = NI; k->TH = TH; k->TW = TW; k->PWC = PWC; k->PXI = PXI; k->PX = PXQ * 4; k->PXQ = PXQ;
                k->tiles_w = cols;
                k->tiles_img = cols * ((OH + TH - 1) / TH);
                k->tile_px = TH * TW;
                k->run = 0;
                if (tiles > 0x3fffffff) return false;
                k->tiles_n = (int)tiles;
            }
        }
    }
    if (best < 0) return false;
    k->tiles_m = ((int)d.oc + bm - 1) / bm;
    if ((int64_t)k->tiles_n * k->tiles_m > 0x3ffffff0) return false;
    const int E = GS * T, EP = (E + 1) & ~1;
    *lds_bytes = 2 * (EP * p1_bmp(mt) + GS * k->PX) * 16;
    return *lds_bytes <= 150 * 1024;
}

// The same tile as a run of pixels in the order of memory where that is ahead of the rows and columns of p1_plan.
// Rows that end inside a group of four columns cost rows-and-columns tiles a group of its own in each row, two more stores for its outputs of
// every channel (six more memory instructions, all of single bytes, when this rule was made), and columns of the tile that hold nothing; a run has
// one such group at an image's end.  Its patch is all columns of the rows that it touches.  231 drawn layers with such rows, graph replays:
// 0.97 of the time since this rule takes runs for some (3x3 121 -> 251 at 45 x 10, batch 54: 29.2 -> 18.6 us; 3x3 75 -> 150 at 61 x 45, batch 6,
// residual: 12.4 -> 11.3).  What a run needs to know costs layers with rows of whole groups up to 3 % of a launch of 4 us.
// Not where a run's patch asks more of a thread or leaves fewer workgroups to a CU (3x3 at stride 2, 202 -> 106 at 60 x 91, batch 14: 24.5 ->
// 37.4), nor, where every workgroup has a CU for itself, for a patch that takes longer to turn (5x5 5 -> 180 at 14 x 43, batch 2: 4.8 -> 6.4).
void p1_run(const ConvProblem& p, int tile, int cu_count, P1Args* k, int* lds_bytes) {
    const mi355_conv_desc& d = p.d;
    const int T = (int)(d.fh * d.fw), F = (int)d.fw, GS = p1_gs(T), TPG = 256 / GS, bm = kP1Tiles[tile][0] * 32, bn = kP1Tiles[tile][1] * 128;
    const int OH = (int)p.oh, OW = (int)p.ow, sh = (int)d.stride_h, sw = (int)d.stride_w;
    if (OW % 4 == 0 || (int64_t)OH * OW > 0x3fffff00) return;
    const int ohw4 = (OH * OW + 3) & ~3;
    int NI = ohw4 < bn ? bn / ohw4 : 1, run = ohw4, runs = 1;
    if (NI == 1) {
        runs = (ohw4 + bn - 1) / bn;
        run = ((ohw4 + runs - 1) / runs + 3) & ~3;
        runs = (ohw4 + run - 1) / run;
    }
    const int64_t pwc = ((int64_t)(OW - 1) * sw + F + 3 + 3) & ~3;
    if (pwc > 0xffff) return;
    const int PWC = (int)pwc, TH = std::min((run + OW - 2) / OW + 1, OH);
    const int64_t pxi = (int64_t)((TH - 1) * sh + F) * PWC, pxq = NI * pxi / 4;
    const int threads_had = (k->PXQ + TPG - 1) / TPG;  // quads of a thread
    if (pxq > (int64_t)threads_had * TPG) return;
    const int64_t tiles = ((int64_t)d.n + NI - 1) / NI * runs;
    const int lds = *lds_bytes + 2 * GS * ((int)pxq * 4 - k->PX) * 16;
    if (tiles > k->tiles_n || lds > 150 * 1024 || std::min(3, 160 * 1024 / lds) < std::min(3, 160 * 1024 / *lds_bytes)) return;
    if (tiles * pxq * 5 > (int64_t)k->tiles_n * k->PXQ * 8) return;
    if (tiles * ((d.oc + bm - 1) / bm) <= cu_count && pxq * 10 > (int64_t)k->PXQ * 13) return;
    k->NI = NI; k->TH = TH; k->TW = OW; k->PWC = PWC; k->PXI = (int)pxi; k->PX = (int)pxq * 4; k->PXQ = (int)pxq;
    k->tiles_w = OW;  // (what a run's first pixel is divided by)
    k->tiles_img = runs;
    k->tile_px = k->run = run;
    k->tiles_n = (int)tiles;
    *lds_bytes = lds;
}

typedef void (*P1Kernel)(P1Args);
template <P1Kernel kern>
int launch_p1(hipStream_t st, const P1Args& k, int threads, int lds) {
    static std::atomic<int> max_lds_set{0};
    if (max_lds_set.load(std::memory_order_relaxed) == 0) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 152 * 1024);
        if (e != hipSuccess) return (int)e;
        max_lds_set.store(1, std::memory_order_relaxed);
    }
    const int64_t grid = (int64_t)((k.tiles_n + 7) / 8) * k.tiles_m * 8;
    return launch_kernel(kern, dim3((unsigned)grid), dim3(threads), lds, st, k);
}

// LDS of the form with two groups of waves, or 0 where one is better.  Where every workgroup has a CU to itself a layer is its chain of stages, and
// two groups halve it (us, graph replays of one group / two): 5x5, 129 workgroups, 27.0 / 20.6; 3x3, 88 workgroups, eight stages, 13.6 / 11.0;
// 1x1 230 -> 16 at 17 x 105, batch 14, four stages, 7.6 / 6.6.  Not two stages (68 layers: 0.987 on average, up to 1.034), nor more than one workgroup to a CU, where
// registers and LDS keep the second one out: 1.04 to 1.4 times as long on 12 of 13 such layers.
int p1_split_lds(const P1Args& k, int lds, int cu_count) {
    const int both = std::max(2 * lds, 16 * 1024);  // (16 KiB: the sums that the groups exchange)
    return k.nstages >= 3 && (int64_t)((k.tiles_n + 7) / 8) * k.tiles_m <= cu_count / 8 && both <= 150 * 1024 ? both : 0;
}

template <int T>
int launch_p1_tile(hipStream_t st, const P1Args& k, int tile, int lds, int cu_count) {
    switch (tile) {
        case 0: {
            const int lds2 = p1_split_lds(k, lds, cu_count);
            return lds2 ? launch_p1<two::patch1_kernel<1, 1, T>>(st, k, 512, lds2) : launch_p1<one::patch1_kernel<1, 1, T>>(st, k, 256, lds);
        }
        case 1: return launch_p1<one::patch1_kernel<1, 2, T>>(st, k, 256, lds);
        case 2: return launch_p1<one::patch1_kernel<2, 2, T>>(st, k, 256, lds);
        default: return launch_p1<one::patch1_kernel<2, 1, T>>(st, k, 256, lds);
    }
}

}  // namespace

bool patch1_usable(const ConvProblem& p) {
    const mi355_conv_desc& d = p.d;
    if (d.format != MI355_FMT_NCHW || p.dw4 || d.group != 1) return false;
    if (d.dst_dtype != MI355_DT_QS8 || d.bias_mode == MI355_BIAS_FULL || !p.epi.fast) return false;
    if (d.mode != MI355_MODE_CROSS_CORRELATION || d.dilate_h != 1 || d.dilate_w != 1) return false;
    if (d.fh != d.fw || (d.fh != 1 && d.fh != 3 && d.fh != 5)) return false;
    // a row holds a quad; the filter holds one item; paddings and strides that keep a tile's coordinates small
    if (d.iw < 4 || (uint64_t)d.oc * d.ic < 4 || d.pad_h > 0xfff || d.pad_w > 0xfff || d.stride_h > 64 || d.stride_w > 64) return false;
    const int64_t lim = (int64_t)1 << 31, n1 = (int64_t)d.n - 1;
    const int64_t src_b = n1 * p.src_sn + (int64_t)d.ic * d.ih * d.iw, out = (int64_t)d.oc * p.oh * p.ow;
    if (src_b >= lim || n1 * p.dst_sn + out >= lim || n1 * p.z_sn + out >= lim || (int64_t)d.oc * d.ic * d.fh * d.fw >= lim / 2) return false;
    return d.n > 0 && out > 0;
}

// The tile, or -1 where packing in a launch of its own is ahead.  Graph replays of every tile and of the packed path on 220
// sizes drawn over 3 to 256 channels in, 8 to 256 out, planes of 7 x 7 to 112 x 112 and batch 1 to 64; w0: workgroups of 32 x 128.
//   The packed path takes 6 to 9 us however few the tiles -- two launches, but its few-pixel kernel splits the reduction -- where
// this kernel walks the stages one after the other at 0.9 us each (1.7 with 25 taps): up to half a workgroup per CU a long
// reduction goes there (3x3 130 -> 44 at 12 x 12, five stages: 8.6 us here, 6.9 there; 48 -> 12, two: 5.0 / 6.4).  With more tiles
// it is the other way round: 3x3 45 -> 12 at 22 x 22, batch 47: 5.3 / 9.4; 1x1 20 -> 149 at 96 x 78: 24.1 / 34.3; 5x5 46 -> 45,
// 168640 pixels: 25.4 / 41.4.  A caller without a workspace has no packed path (packed = false).
//   (These figures are of one group of waves.  With two, p1_split_lds, the lines for few tiles and long chains still lie right: of 240 drawn layers that go to the
// packed path and that two groups would share here, one launch is ahead on 27, and takes 1.04 of the packed path's time on average with 1x1,
// 1.19 with 3x3, 1.41 with 5x5.)
//   Below 64 workgroups and from 2^24 multiply-adds on the packed path stays, 5 to 25 % behind on one or two stages: a workspace of
// the size that it needs is written there, which the interface's tests hold (24 -> 40 at 28 x 28, batch 4, among them).
//   Tiles: the smallest up to 400 workgroups of it (5x5: 256), where a stage's latency is all there is; beyond that 32 x 256 (3x3
// 14 -> 19, 202800 pixels: 15.6 us against 18.5), and 64 x 256, which turns a patch for twice the channels, once those are two per
// CU (3x3 8 -> 189, 61950 pixels: 15.6 against 18.9 and 20.1).  At strides a patch is several times its pixels: 64 x 128 (3x3 38 ->
// 97, stride 2, 588 workgroups: 14.0 against 18.3).
//   At strides every tile of 64 channels turns that patch again, so from three of them on (tm) packing once gets ahead on filters of 1x1 and
// 3x3 as their workgroups (w) grow.  Of 7315 layers at stride 2, this kernel over the packed path (two launches), us:
//     w >= 4 per CU, tm >= 4: 1.14 on average without a residual (3x3 6 -> 193 at 69 x 65, batch 64: 34.7 / 23.2), with one only 3x3 with
//       rows out that are not whole quads (1.04; 1x1 0.94, whole quads 0.84);
//     w >= 1200, tm = 3: 1.03 without a residual, rows out that are not whole quads;
//     another round of chains of three and more stages, w of 1 to 1.6 or 2 to 2.5 per CU, tm >= 3: 1.04 (1x1 219 -> 207 at 106 x 28, batch
//       20, w = 640: 22.6 / 16.4).
//   744 of the 7315 were more than 3 % behind packing in one launch and 485 more than 10 %; with these lines 235 and 108.
//   5x5 with two and more stages at strides of 1 and 2, against the packed path: by what each takes, see p1_behind_packed.
// (k: the geometry of some tile; *chosen: the workgroups of the one that is returned)
static int p1_tile(const ConvProblem& p, bool packed, int cu_count, P1Args& k, int64_t* chosen) {
    int lds;
    auto wgs = [&](int tile) { return p1_plan(p, tile, &k, &lds) ? (int64_t)k.tiles_n * k.tiles_m : (int64_t)-1; };
    const int64_t w0 = wgs(0);
    *chosen = w0;
    auto take = [&](int tile, int64_t w) {
        *chosen = w;
        return tile;
    };
    const int T = (int)(p.d.fh * p.d.fw);
    if (w0 < 0) return -1;
    const uint64_t macs = (uint64_t)p.d.n * p.d.oc * p.oh * p.ow * p.icpg * p.d.fh * p.d.fw;
    if (packed && w0 < 64 && macs >= (1u << 24)) return -1;
    if (packed && w0 < 128 && k.nstages >= (T == 1 ? 4 : T == 9 ? 3 : 2)) return -1;
    if (w0 <= (T == 25 ? 256 : 400)) return 0;
    if (p.d.stride_h > 1 || p.d.stride_w > 1) {
        if (p.d.oc <= 32) return 0;
        const int64_t w = wgs(3), cu = cu_count;
        if (packed && p.d.oc > 128 && T <= 9) {
            const bool ragged = p.ow % 4 != 0, z = p.d.has_z != 0;
            if (p.d.oc > 192 ? w >= 4 * cu && (!z || (T == 9 && ragged)) : 256 * w >= 1200 * cu && !z && ragged) return -1;
            if (k.nstages >= 3 && ((w > cu && 5 * w <= 8 * cu) || (w > 2 * cu && 2 * w <= 5 * cu))) return -1;
        }
        return w > 0 ? take(3, w) : 0;
    }
    const int64_t w2 = p.d.oc > 32 ? wgs(2) : 0;
    if (w2 >= 512) return take(2, w2);
    const int64_t w1 = wgs(1);
    return w1 > 0 ? take(1, w1) : 0;
}

// 5x5 in two and more stages: whether the packed path is ahead of this kernel on its tile, by prices on a device of 256 CUs in us and, of
// reductions, us per stage or per 1024 packed bytes.  This kernel walks its stages one after the other, so workgroups that begin another
// round over the device -- of one or two to a CU -- cost a whole chain more; the packed path splits few tiles' reductions and deals
// many tiles out smoothly.  (Prices of one group of waves and of tiles of rows and columns: two groups and runs take less than this says.)  Fitted to graph replays of 2397 layers over 17 to 256 channels on both; of these 213 were more than 3 %
// behind the packed path and 117 more than 10 % (5x5 209 -> 33 at 26 x 7, batch 38: 24.2 / 13.3; 183 -> 164 at 41 x 85, batch 5:
// 56.4 / 36.8); with the prices 40 and 12.  On 591 others 70 and 44 before, 9 and 1 now, 0.70 and 0.69 of the packed path on average.
static bool p1_behind_packed(const ConvProblem& p, int tile, int64_t workgroups, int nstages, int cu_count) {
    struct One {
        float launch, stage, round2_stage, round_stage, share;
    };
    static const One one[4] = {{2.907f, 0.716f, 0.178f, 0.457f, 0.981f},   // 32 x 128
                               {3.431f, 0.046f, 1.065f, 0.460f, 1.673f},   // 32 x 256
                               {5.295f, 0.710f, 0.615f, 1.079f, 2.326f},   // 64 x 256
                               {2.954f, 0.303f, 1.051f, 0.647f, 1.806f}};  // 64 x 128
    struct Packed {
        float launch, k, round_k, share_k, share, strided_k, round2_k;
    };
    static const Packed packed[2] = {{5.747f, 1.533f, 0.000f, 3.430f, 0.000f, 1.973f, 0.000f},   // tiles of 64 x 128 for a quarter of the CUs
                                     {7.846f, 0.155f, 1.474f, 0.277f, 1.204f, 2.086f, 1.357f}};
    const uint32_t cu = (uint32_t)cu_count, wgs = (uint32_t)workgroups, r1 = (wgs + cu - 1) / cu;
    const One& a = one[tile];
    const float this_us = a.launch + (float)nstages * (a.stage + a.round2_stage * (float)((r1 + 1) / 2) + a.round_stage * (float)r1) +
                          a.share * ((float)wgs / (float)cu);
    const uint64_t px = (uint64_t)p.d.n * p.oh * p.ow, tiles = (px + 127) / 128 * ((p.d.oc + 63) / 64), rounds = (tiles + cu - 1) / cu;
    const float share = (float)tiles / (float)cu, kb = (float)((p.d.ic + 31) / 32 * 32 * 25) / 1024.0f;
    const Packed& b = packed[share > 0.25f];
    const float packed_us = b.launch + b.share * share + kb * (b.k + b.round_k * (float)rounds + b.share_k * share + b.round2_k * (float)((rounds + 1) / 2) +
                                                               (p.d.stride_h * p.d.stride_w > 1 ? b.strided_k * share : 0.0f));
    return this_us > 0.97f * packed_us;
}

int patch1_pick(const ConvProblem& p, bool packed, int cu_count) {
    if (!patch1_usable(p)) return -1;
    P1Args k;
    int64_t wgs;
    const int tile = p1_tile(p, packed, cu_count, k, &wgs);
    if (tile < 0 || !packed || p.d.fh != 5 || p.d.ic <= 16 || p.d.stride_h > 2 || p.d.stride_w > 2) return tile;
    return p1_behind_packed(p, tile, wgs, k.nstages, cu_count) ? -1 : tile;
}

int launch_patch1(hipStream_t st, const ConvProblem& p, int tile, int cu_count, const int8_t* src, const int8_t* flt, const int32_t* bias, const int8_t* z,
                  int8_t* dst) {
    const mi355_conv_desc& d = p.d;
    P1Args k;
    int lds;
    if (!p1_plan(p, tile, &k, &lds)) return (int)hipErrorInvalidConfiguration;
    p1_run(p, tile, cu_count, &k, &lds);
    k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
    k.IC = d.ic; k.IH = d.ih; k.IW = d.iw; k.IHW = d.ih * d.iw;
    k.OC = d.oc; k.OH = p.oh; k.OW = p.ow; k.OHW = p.oh * p.ow; k.N = d.n;
    k.sh = d.stride_h; k.sw = d.stride_w; k.ph = d.pad_h; k.pw = d.pad_w;
    k.src_sn = (int)p.src_sn; k.dst_sn = (int)p.dst_sn; k.z_sn = (int)p.z_sn;
    k.src_bytes = (uint32_t)((d.n - 1) * p.src_sn + (int64_t)d.ic * k.IHW);
    k.dst_bytes = (uint32_t)((d.n - 1) * p.dst_sn + (int64_t)d.oc * k.OHW);
    k.z_bytes = (uint32_t)((d.n - 1) * p.z_sn + (int64_t)d.oc * k.OHW);
    k.kbytes = d.ic * d.fh * d.fw;
    k.flt_bytes = k.kbytes * d.oc;
    k.has_bias = d.bias_mode == MI355_BIAS_BROADCAST_CHANNEL;
    k.div_tiles_m = make_fastdiv(k.tiles_m); k.div_tiles_img = make_fastdiv(k.tiles_img); k.div_tiles_w = make_fastdiv(k.tiles_w);
    k.div_tw = make_fastdiv(k.TW); k.div_tile_px = make_fastdiv(k.tile_px);
    k.div_pqi = make_fastdiv(k.PXI >> 2); k.div_pqw = make_fastdiv(k.PWC >> 2);
    k.epi = p.epi;
    const int T = (int)(d.fh * d.fw);
    return T == 1 ? launch_p1_tile<1>(st, k, tile, lds, cu_count) : T == 9 ? launch_p1_tile<9>(st, k, tile, lds, cu_count) : launch_p1_tile<25>(st, k, tile, lds, cu_count);
}

}  // namespace mi355
