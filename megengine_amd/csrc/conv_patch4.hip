// Windowed convolutions on 4-packed tensors (NCHW4 in and out), tiles "patch4_*".
//
// An im2col operand of a 4-packed tensor comes in pieces of 4 bytes -- the channels of a pixel lie in planes -- so a tiled
// implicit GEMM loads every byte of a 3x3 layer nine times, a dword at a time, through a per-unit table of offsets: 3x3
// 64 -> 64 at 56 x 56, batch 16, took 12.4 us where its bytes and products allow 1.5, and the vector-memory path was what
// it waited for.  Here the input patch of a tile is loaded once and turned on its way into LDS: sixteen channels of a pixel
// side by side, [group of 16 channels][patch pixel][16 bytes], so that every tap's operand is one ds_read_b128 at a shifted
// pixel, consecutive lanes consecutive pixels, free of bank conflicts.  The filter is turned with it: entry (channel group,
// tap) of a stage holds 16 bytes per output channel, [entry][channel][16 bytes]; a step of v_mfma_i32_32x32x32_i8 is two
// entries, one per half wave.
//   * A workgroup is four waves side by side over the pixels; each multiplies all BM = 32 or 64 channels of the tile by its
//     32 or 64 pixels.  A stage is GS channel groups (two for 3x3, one for larger filters); two stages are in LDS, the
//     next one's global loads are in registers while the current one is multiplied, one barrier per stage.
//   * Tiles are TH x TW pixels of one image, or of NI whole images where one is small; sizes chosen on the host so that the
//     last tiles of a row and column are as full as the others.
//   * Channel blocks past the last one meet zero filter bytes.
//   * What bounds it: LDS, which a wave of 32 x 64 outputs reads three times for two matrix instructions, and the latency of a
//     stage where tiles are few.  A wave of 64 x 64 (four reads for four) is ahead only where it still fills the chip twice: it
//     costs a third of the occupancy.  Loads two stages ahead, tried, cost more occupancy than they hid (7.5 us against 6.9 at
//     56 x 56 below); reading one step's operands ahead instead of two, or computing a descriptor per channel block instead of
//     a scalar offset (157 scalar instructions per stage instead of 64), cost up to a quarter of the time.
//   * Where there is a workgroup to a CU or fewer, it has two groups of four waves that take every other stage each (p4_split_lds).
//   * 3x3 over at most 64 channels has a kernel of its own with one stage (patch4_one_kernel), ahead at every size and tile: 64 -> 64 at
//     56 x 56, batch 16: 7.5 -> 7.0 us; 28 -> 20 at 29 x 28, stride 2, batch 34: 4.6 -> 3.9; 48 -> 148 at 97 x 107, batch 7: 20.7 -> 14.3;
//     56 -> 480 at 82 x 94, batch 10: 50 -> 41; 30 drawn layers on each tile: 1.05 to 1.25 times as fast.
// Graph replays of the layer, here and below: 3x3 64 -> 64 at 56 x 56, batch 16: 12.4 -> 6.9 us, batch 64: 31.7 -> 17.0; 256 ->
// 256 at 14 x 14, batch 16: 15.5 -> 8.3; 32 -> 32 at 112 x 112, batch 64: 52 -> 26.8; 5x5 100 -> 132 at 33 x 35, batch 20: 50 -> 22.5.
// 5x5 has its thirteen steps compiled in as nine taps have: in the general form's loop the compiler reads a step's operands next to the product that
// waits for them (80 -> 228 at 15 x 52, batch 30: 28.3 -> 22.6 us; 220 -> 88 at 65 x 102, batch 9: 82 -> 68).
#include <atomic>
#include <algorithm>

#include "igemm_shared.h"

namespace mi355 {
namespace {

constexpr int P4_NPK = 4;   // patch vectors per thread and stage
constexpr int P4_NKA = 7;   // filter vectors per thread and stage

// vectors between the planes of a patch: 4 mod 8, so that the two halves of a wave read from other banks
__host__ __device__ constexpr int p4_pitch(int px) { return ((px + 3) & ~7) + 4; }

struct P4Args {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    uint32_t src_bytes, flt_bytes;
    int IH, IW, OH, OW, FW, T, sh, sw, ph, pw;
    int OC, N, icb, GS, nstages, kbytes;
    int src_sn, src_scb, dst_sn, dst_scb, z_sn, has_bias;
    int NI, TH, TW, PWC, PXI, PX;     // images, rows, columns of a tile; patch columns, pixels per image, pixels
    int pkn, rpi, kan;                // patch pixels per thread; filter rows per pass of the workgroup, passes
    int tiles_m, tiles_n, vr;         // vr: filter vectors per output channel and stage
    FastDiv div_tiles_m, div_tiles_img, div_tiles_w, div_tw, div_tile_px, div_pxi, div_pwc, div_vr, div_t;
    int tiles_img, tiles_w;           // tiles per image group, tiles per row
    EpiParams epi;
};

// QN: quads of channels of each block of 32 that are in acc (all four of the sixteen sums, or the first two)
template <int MT, int NT, int QN, int NL, bool HZ>
__device__ __forceinline__ void p4_epilogue(const P4Args& a, v16i (&acc)[MT][NT], int oc0, const int (&d_px)[NT], const int (&z_px)[NT], int lh) {
    uint32_t zw[NT][MT][QN];
    if (HZ) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < QN; ++q) {
                    const int oc4 = oc0 + i * 32 + 8 * q + 4 * lh;
                    zw[j][i][q] = d_px[j] >= 0 && oc4 < a.OC ? *reinterpret_cast<const uint32_t*>(a.z + z_px[j] + (int64_t)(oc4 >> 2) * a.dst_scb) : 0u;
                }
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < QN; ++q) {
                const int oc4 = oc0 + i * 32 + 8 * q + 4 * lh;
                const v16i& c = acc[i][j];
                const uint32_t o = requant4_fast<NL, HZ>(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3], HZ ? zw[j][i][q] : 0u, a.epi);
                if (d_px[j] >= 0 && oc4 < a.OC) *reinterpret_cast<uint32_t*>(a.dst + d_px[j] + (int64_t)(oc4 >> 2) * a.dst_scb) = o;
            }
}

template <int MT, int NT, int QN = 4>
__device__ __forceinline__ void p4_finish(const P4Args& a, v16i (&acc)[MT][NT], int oc0, const int (&d_px)[NT], const int (&z_px)[NT], int lh) {
#define MI355_P4(NL, HZ) p4_epilogue<MT, NT, QN, NL, HZ>(a, acc, oc0, d_px, z_px, lh)
    if (a.epi.lin) {
        MI355_P4(NL_LIN, false);
    } else if (a.epi.has_z) {
        switch (a.epi.nonline) {
            case NL_RELU: MI355_P4(NL_RELU, true); break;
            case NL_H_SWISH: MI355_P4(NL_H_SWISH, true); break;
            default: MI355_P4(NL_IDENTITY, true); break;
        }
    } else {
        switch (a.epi.nonline) {
            case NL_RELU: MI355_P4(NL_RELU, false); break;
            case NL_H_SWISH: MI355_P4(NL_H_SWISH, false); break;
            default: MI355_P4(NL_IDENTITY, false); break;
        }
    }
#undef MI355_P4
}

// the kernel, by groups of waves and taps of a stage
namespace one {
constexpr int KS = 1;
constexpr bool TAPS25 = false;
#include "patch4_kernel.h"
}  // namespace one
namespace two {
constexpr int KS = 2;
constexpr bool TAPS25 = false;
#include "patch4_kernel.h"
}  // namespace two
namespace one25 {
constexpr int KS = 1;
constexpr bool TAPS25 = true;
#include "patch4_kernel.h"
}  // namespace one25
namespace two25 {
constexpr int KS = 2;
constexpr bool TAPS25 = true;
#include "patch4_kernel.h"
}  // namespace two25

// 3x3 over at most 32 KB channels: the whole reduction in one stage.  All of a workgroup's loads are in flight at once and one barrier
// stands between them and the products, where the kernel above waits for a stage's latency per 32 channels.  LDS: [step][half of 32
// channels][output channel] and [group of 16 channels][patch pixel], 16 bytes each.
template <int KB, int MT, int NT>
__global__ __launch_bounds__(256, 2) void patch4_one_kernel(P4Args a) {
    constexpr int BM = MT * 32, BMP = BM + 1, G = 2 * KB, STEPS = 9 * KB, VR = 18 * KB, RPI = 256 / VR, KAN = (BM + RPI - 1) / RPI;
    constexpr int A_VECS = 2 * STEPS * BMP, NPX = 2;
    const int PXP = p4_pitch(a.PX);
    extern __shared__ __attribute__((aligned(16))) v4i lds[];
    // everything up to the first operands in one batch of scalar loads, and a word of each line that the epilogue reads
    asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.z), "s"(a.dst), "s"(a.src_bytes), "s"(a.flt_bytes), "s"(a.IH), "s"(a.IW),
                 "s"(a.OH), "s"(a.OW), "s"(a.sh), "s"(a.sw), "s"(a.ph), "s"(a.pw), "s"(a.OC), "s"(a.N), "s"(a.icb), "s"(a.kbytes), "s"(a.src_sn),
                 "s"(a.src_scb), "s"(a.has_bias), "s"(a.NI), "s"(a.TH), "s"(a.TW), "s"(a.PWC), "s"(a.PXI), "s"(a.PX), "s"(a.tiles_m));
    asm volatile("" ::"s"(a.tiles_n), "s"(a.tiles_img), "s"(a.tiles_w), "s"(a.dst_sn), "s"(a.dst_scb), "s"(a.z_sn), "s"(a.div_tiles_m.m),
                 "s"(a.div_tiles_img.m), "s"(a.div_tiles_w.m), "s"(a.div_tw.m), "s"(a.div_tile_px.m), "s"(a.div_pxi.m), "s"(a.div_pwc.m),
                 "s"(a.epi.s_b), "s"(a.epi.lin_lo));
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31, lh = lane >> 5;
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
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes), rs_flt = make_rsrc(a.flt, a.flt_bytes);

    // filter: the same 16 bytes of every RPI-th row; what lies past a row's end is the next row's, and becomes zero
    const int f_row = t / VR, f_first = (t - f_row * VR) * 4, f_left = a.icb * 9 - f_first;
    v4i xf[KAN];
#pragma unroll
    for (int k = 0; k < KAN; ++k)
        xf[k] = __builtin_amdgcn_raw_buffer_load_b128(
                rs_flt, ((f_row < RPI) & (f_left > 0)) ? (oc0 + f_row + k * RPI) * a.kbytes + f_first * 4 : SENT, 0, 0);
    // patch: a pixel's channel blocks are a scalar offset (blocks past the last one: the last one again, they meet zero filter bytes)
    v4i xp[NPX][G];
    const uint32_t last_cb = (uint32_t)(a.icb - 1) * a.src_scb;
#pragma unroll
    for (int k = 0; k < NPX; ++k) {
        const uint32_t px = t + k * 256, im = fdiv(px, a.div_pxi), r = px - im * a.PXI, pr = fdiv(r, a.div_pwc), pc = r - pr * a.PWC;
        const int ih = oh0 * a.sh - a.ph + (int)pr, iw = ow0 * a.sw - a.pw + (int)pc, n = n0 + (int)im;
        const bool ok = ((int)px < a.PX) & (n < a.N) & ((unsigned)ih < (unsigned)a.IH) & ((unsigned)iw < (unsigned)a.IW);
        const int off = ok ? n * a.src_sn + (ih * a.IW + iw) * 4 : SENT;
#pragma unroll
        for (int c = 0; c < G * 4; ++c)
            xp[k][c / 4][c % 4] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_src, off, (int)min((uint32_t)c * a.src_scb, last_cb), 0);
    }
    v4i bv[MT][4];
    {
        const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias ? a.OC * 4 : 0);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) bv[i][q] = __builtin_amdgcn_raw_buffer_load_b128(rs_bias, (oc0 + i * 32 + 8 * q + 4 * lh) * 4, 0, 0);
    }
    int b_px[NT], d_px[NT], z_px[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const uint32_t p = (wave * NT + j) * 32 + l32;
        const uint32_t im = fdiv(p, a.div_tile_px), r = p - im * (uint32_t)(a.TH * a.TW), oh = fdiv(r, a.div_tw), ow = r - oh * a.TW;
        const bool ok = ((int)im < a.NI) & (n0 + (int)im < a.N) & (oh0 + (int)oh < a.OH) & (ow0 + (int)ow < a.OW);
        b_px[j] = (int)im < a.NI ? (int)(im * a.PXI + oh * a.sh * a.PWC + ow * a.sw) : 0;
        const int at = ((oh0 + (int)oh) * a.OW + ow0 + (int)ow) * 4;
        d_px[j] = ok ? (n0 + (int)im) * a.dst_sn + at : -1;
        z_px[j] = (n0 + (int)im) * a.z_sn + at;
    }

    // into LDS: word (channel block, tap) of the row goes to step (block / 8, tap), half (block / 4) % 2, word block % 4
    int f_lds[4];
    {
        int cb = f_first / 9, tap = f_first - cb * 9;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f_lds[i] = (((((cb >> 3) * 9 + tap) * 2 + ((cb >> 2) & 1)) * BMP + f_row) << 2) + (cb & 3);
            if (++tap == 9) {
                tap = 0;
                ++cb;
            }
        }
    }
    if (f_row < RPI) {
        int* w = reinterpret_cast<int*>(lds);
#pragma unroll
        for (int k = 0; k < KAN; ++k)
            if (BM % RPI == 0 || k + 1 < KAN || f_row + k * RPI < BM)
#pragma unroll
                for (int i = 0; i < 4; ++i) w[f_lds[i] + k * RPI * 4] = i < f_left ? xf[k][i] : 0;
    }
#pragma unroll
    for (int k = 0; k < NPX; ++k)
        if (t + k * 256 < a.PX)
#pragma unroll
            for (int g = 0; g < G; ++g) lds[A_VECS + g * PXP + t + k * 256] = xp[k][g];
    v16i acc[MT][NT];
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
    const v4i* pb = lds + A_VECS + lh * PXP;
    auto load = [&](int s, v4i (&fa)[MT], v4i (&fb)[NT]) __attribute__((always_inline)) {
        const int cb = s / 9, tap = s % 9, off = cb * 2 * PXP + (tap / 3) * a.PWC + tap % 3;
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
    p4_finish(a, acc, oc0, d_px, z_px, lh);
}

struct P4Cfg {
    int mt, nt;
    const char* name;
};
constexpr P4Cfg kP4[] = {{1, 1, "patch4_32x128"}, {1, 2, "patch4_32x256"}, {2, 2, "patch4_64x256"}};
constexpr int kP4Count = sizeof(kP4) / sizeof(kP4[0]);

// geometry of a tile; false where no patch fits
bool p4_plan(const IgemmArgs& a, int cfg, bool one, P4Args* k, int* lds_bytes) {
    const int bm = kP4[cfg].mt * 32, bn = kP4[cfg].nt * 128;
    const int FH = a.FH, FW = a.FW;
    k->icb = a.kbytes / (4 * a.T);
    const int G = (k->icb + 3) / 4;
    if (one && (FH != 3 || FW != 3 || G > 4)) return false;
    k->GS = one ? (G > 2 ? 4 : 2) : a.T <= 9 && G > 1 ? 2 : 1;
    k->nstages = (G + k->GS - 1) / k->GS;
    k->vr = k->GS * a.T;
    if (k->vr > 256) return false;
    k->rpi = 256 / k->vr;
    k->kan = (bm + k->rpi - 1) / k->rpi;
    if (!one && k->kan > P4_NKA) return false;
    const int max_px = one ? 512 : P4_NPK / k->GS * 256;
    // whole images while they fit several times, else rows; a wide image is split into equal columns
    int tiles_w = 1;
    for (;; ++tiles_w) {
        k->TW = (a.OW + tiles_w - 1) / tiles_w;
        if (k->TW > bn) continue;
        int th = bn / k->TW;
        k->NI = 1;
        if (th >= a.OH) {
            k->NI = tiles_w == 1 ? th / a.OH : 1;
            th = a.OH;
        }
        for (;;) {
            const int bands = (a.OH + th - 1) / th;
            k->TH = (a.OH + bands - 1) / bands;
            k->PWC = (k->TW - 1) * a.sw + FW;
            k->PXI = ((k->TH - 1) * a.sh + FH) * k->PWC;
            while (k->NI > 1 && k->NI * k->PXI > max_px) --k->NI;
            k->PX = k->NI * k->PXI;
            if (k->PX <= max_px || th == 1) break;
            th = k->TH - 1;
        }
        if (k->PX <= max_px) break;
        if (k->TW == 1) return false;
    }
    k->pkn = (k->PX + 255) / 256;
    k->tiles_w = (a.OW + k->TW - 1) / k->TW;
    k->tiles_img = k->tiles_w * ((a.OH + k->TH - 1) / k->TH);
    const int64_t tn = (int64_t)((a.NB + k->NI - 1) / k->NI) * k->tiles_img;
    k->tiles_m = (a.OC + bm - 1) / bm;
    if (tn * k->tiles_m > 0x3ffffff0) return false;
    k->tiles_n = (int)tn;
    const int E = k->GS * a.T, EP = (E + 1) & ~1;
    if (one) {
        *lds_bytes = (E * (bm + 1) + k->GS * p4_pitch(k->PX)) * 16;
        return *lds_bytes <= 80 * 1024;
    }
    *lds_bytes = 2 * (EP * ((k->kan * k->rpi) | 1) + k->GS * k->PX) * 16 + EP * 4;
    return *lds_bytes <= 160 * 1024;
}

// LDS of the form with two groups of waves, or 0 where one is better.  Where every workgroup has a CU to itself a layer is its chain of stages,
// each as long as its loads and its way through LDS, and two groups halve it (us, graph replays, one group / two): 5x5 356 -> 24 at 76 x 108, stride
// 2, batch 9, 23 stages: 40.8 / 29.5; 3x3 424 -> 220 at 12 x 10, batch 60, 14: 17.2 / 14.0; 72 -> 28 at 24 x 33, batch 8, three: 5.0 / 4.6.  104 drawn
// layers with no more workgroups to an XCD than it has CUs: 0.70 to 0.98.  With one more the second form has two to a CU, which its LDS seldom
// allows: 76 such layers 0.86 to 1.36, all but two behind.
int p4_split_lds(const P4Args& k, int lds, int cu_count) {
    const int tab = ((k.GS * k.T + 1) & ~1) * 4, both = std::max(2 * (lds - tab) + tab, 16 * 1024);  // (16 KiB: the sums that the groups exchange)
    return k.nstages >= 2 && (int64_t)((k.tiles_n + 7) / 8) * k.tiles_m <= cu_count / 8 && both <= 160 * 1024 ? both : 0;
}

template <int KB, int MT, int NT>
int launch_one(hipStream_t st, const P4Args& k, int lds) {
    auto kern = patch4_one_kernel<KB, MT, NT>;
    static std::atomic<int> max_lds_set{0};
    if (max_lds_set.load(std::memory_order_relaxed) == 0) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (e != hipSuccess) return (int)e;
        max_lds_set.store(1, std::memory_order_relaxed);
    }
    const int64_t grid = (int64_t)((k.tiles_n + 7) / 8) * k.tiles_m * 8;
    return launch_kernel(kern, dim3((unsigned)grid), dim3(256), lds, st, k);
}

typedef void (*P4Kernel)(P4Args);
template <P4Kernel kern>
int launch_form(hipStream_t st, const P4Args& k, int threads, int lds) {
    static std::atomic<int> max_lds_set{0};
    if (max_lds_set.load(std::memory_order_relaxed) == 0) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        max_lds_set.store(1, std::memory_order_relaxed);
    }
    const int64_t grid = (int64_t)((k.tiles_n + 7) / 8) * k.tiles_m * 8;
    return launch_kernel(kern, dim3((unsigned)grid), dim3(threads), lds, st, k);
}

template <int MT, int NT>
int launch_p4(hipStream_t st, const P4Args& k, int lds, int lds2 = 0) {
    // two groups of nine taps, and not one group of eighteen (3x6, 2x9, ...): the stage has as many entries, the filter rows
    // and the patch of the two differ
    const bool nine = k.GS == 2 && k.T == 9, five = k.GS == 1 && k.T == 25;
    if constexpr (MT * NT == 1) {
        if (lds2)
            return nine   ? launch_form<two::patch4_kernel<1, 1, 9>>(st, k, 512, lds2)
                   : five ? launch_form<two25::patch4_kernel<1, 1, 0>>(st, k, 512, lds2)
                          : launch_form<two::patch4_kernel<1, 1, 0>>(st, k, 512, lds2);
    }
    return nine   ? launch_form<one::patch4_kernel<MT, NT, 9>>(st, k, 256, lds)
           : five ? launch_form<one25::patch4_kernel<MT, NT, 0>>(st, k, 256, lds)
                  : launch_form<one::patch4_kernel<MT, NT, 0>>(st, k, 256, lds);
}

}  // namespace

int patch4_num_cfgs() { return kP4Count; }
const char* patch4_cfg_name(int cfg) { return kP4[cfg].name; }

// the whole reduction in one stage
bool patch4_one_stage(const IgemmArgs& a, int pin, int pout) {
    P4Args k;
    int lds;
    return patch4_can_run(a, pin, pout, 0) && p4_plan(a, 0, true, &k, &lds);
}

bool patch4_can_run(const IgemmArgs& a, int pin, int pout, int cfg) {
    if (cfg < 0 || cfg >= kP4Count || pin != 4 || pout != 4 || a.groups != 1 || a.general || a.T < 2) return false;
    P4Args k;
    int lds;
    return p4_plan(a, cfg, false, &k, &lds);
}

// Which tile, several stages: a workgroup of 32 x 256 once those are more than one per CU (64 -> 64 at 56 x 56, batch 16, 448 of them: 6.9 us
// against 7.5 on 32 x 128; 100 -> 132 at 33 x 35 with a 5x5 filter: 22.5 against 29.7), or 64 x 256 once those are two (128 -> 128
// at 28 x 28, batch 64: 13.8 us against 16.3); below, the smallest tile, because a stage's latency is all there is (256 -> 256 at
// 14 x 14, batch 16, 128 workgroups of 32 x 256: 9.7 us against 8.3).  At strides a tile's patch is several times its pixels:
// the smallest tile (64 -> 128 at 56 x 56, stride 2, batch 16: 6.8 us against 7.6 on 32 x 256), and with many output channels
// and pixels the 128 x 128 tiles of the general kernel, whose operand traffic shrinks with the stride (the same at batch 64:
// 14.7 us against 18.1; 128 -> 128 at 56 x 56, batch 32: 14.2 against 16.2).
// One stage: 32 x 256 from 350 workgroups of it on (20 -> 228 at 95 x 110, batch 1, 330 of them: 5.9 us against 5.6 on 32 x 128; 20 ->
// 192 at 62 x 22, batch 12, 384: 6.4 / 6.7) and at any number of channels (48 -> 148 at 97 x 107, batch 7: 14.3 us, on 64 x 256 17.5);
// at strides 32 x 128 up to 600 tiles of 128 x 128 of the general kernel (16 -> 88, 36960 pixels, 289 of them: 6.9 / 10.9; 12 -> 160,
// 534: 9.0 / 9.6; 28 -> 168, 1054: 22.6 / 18.4).
int patch4_pick(const IgemmArgs& a, int pin, int pout) {
    if (!patch4_can_run(a, pin, pout, 0)) return -1;
    P4Args k;
    int lds;
    const bool one = p4_plan(a, 1, true, &k, &lds);
    if (a.sh > 1 || a.sw > 1) return a.OC > 64 && (int64_t)((a.OC + 127) / 128) * ((a.M + 127) / 128) >= (one ? 600 : 150) ? -1 : 0;
    if (one) return (int64_t)k.tiles_n * k.tiles_m >= 350 ? 1 : 0;
    auto wgs = [&](int cfg) { return p4_plan(a, cfg, false, &k, &lds) ? (int64_t)k.tiles_n * k.tiles_m : 0; };
    if (a.OC > 64 && wgs(2) >= 512) return 2;
    return wgs(1) >= 300 ? 1 : 0;
}

int launch_patch4(hipStream_t st, const IgemmArgs& a, int cfg, int cu_count) {
    P4Args k;
    int lds;
    const bool one = p4_plan(a, cfg, true, &k, &lds);
    if (!one && !p4_plan(a, cfg, false, &k, &lds)) return (int)hipErrorInvalidConfiguration;
    k.src = a.src; k.flt = a.flt; k.bias = a.bias; k.z = a.z; k.dst = a.dst;
    k.src_bytes = a.src_bytes; k.flt_bytes = a.flt_bytes;
    k.IH = a.IH; k.IW = a.IW; k.OH = a.OH; k.OW = a.OW; k.FW = a.FW; k.T = a.T;
    k.sh = a.sh; k.sw = a.sw; k.ph = a.ph; k.pw = a.pw;
    k.OC = a.OC; k.N = a.NB; k.kbytes = a.kbytes;
    k.src_sn = a.src_sn; k.src_scb = a.src_scb; k.dst_sn = a.dst_sn; k.dst_scb = a.dst_scb; k.z_sn = a.z_sn;
    k.has_bias = a.has_bias;
    k.div_tiles_m = make_fastdiv(k.tiles_m); k.div_tiles_img = make_fastdiv(k.tiles_img); k.div_tiles_w = make_fastdiv(k.tiles_w);
    k.div_tw = make_fastdiv(k.TW); k.div_tile_px = make_fastdiv(k.TH * k.TW);
    k.div_pxi = make_fastdiv(k.PXI); k.div_pwc = make_fastdiv(k.PWC);
    k.div_vr = make_fastdiv(k.vr); k.div_t = make_fastdiv(a.T);
    k.epi = a.epi;
    if (one && k.GS == 2) return cfg == 0 ? launch_one<1, 1, 1>(st, k, lds) : cfg == 1 ? launch_one<1, 1, 2>(st, k, lds) : launch_one<1, 2, 2>(st, k, lds);
    if (one) return cfg == 0 ? launch_one<2, 1, 1>(st, k, lds) : cfg == 1 ? launch_one<2, 1, 2>(st, k, lds) : launch_one<2, 2, 2>(st, k, lds);
    switch (cfg) {
        case 0: return launch_p4<1, 1>(st, k, lds, p4_split_lds(k, lds, cu_count));
        case 1: return launch_p4<1, 2>(st, k, lds);
        default: return launch_p4<2, 2>(st, k, lds);
    }
}

}  // namespace mi355
