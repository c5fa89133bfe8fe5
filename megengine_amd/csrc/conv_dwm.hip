// Channel-wise convolution on the matrix cores (4-packed activations, filters up to 32 blocks of a window, any stride).
//
// A channel-wise layer has no contraction over channels, but it has one over the pixels of a window, and the layout
// (n, c/4, h, w, 4) lays that out for the matrix cores as it stands: 16 bytes in memory are four pixels of four channels.
// v_mfma_i32_16x16x64_i8 takes four such blocks of a window as its K dimension,
//   B (64 x 16): column = a quad of four output pixels, its K = blocks of four input pixels, read from LDS as they lie;
//   A (16 x 64): row = (output pixel j of the quad, channel c), K = (input pixel, channel): the filter tap that connects input
//                pixel and output pixel where the channels agree, zero elsewhere,
// so the transposes, byte alignments and dot products of the vector form (conv_dw.hip) all fall away: a wave's 64 pixels of four
// channels take ceil(rows x blocks / 4) matrix instructions -- 2 for 3x3, 3 for 5x5, 6 for 7x7 at stride 1 -- of which a sixth to
// a third is useful, still several times the rate of byte dot products.  A lane ends with the four channels of one pixel.
//
// A workgroup computes a band of output rows of one channel block: the padded input rows go to LDS in one pass (a row, or several
// narrow ones, per wave instruction, no register stage), so a pixel is read from memory once, and everything outside the image
// is zero there.  Bound by the vector instructions: the requantisation of 8 values per lane and iteration and the set-up of
// a workgroup (350 instructions per wave), not by the matrix instructions (5x5 stride 2, 240 channels at 57 x 57, batch 16:
// 8.4 us, of which the copy rate accounts for 3.2; the byte dot products took 9.4).
#include <tuple>

#include "lds_copy.h"
#include "wire.h"

namespace mi355 {
namespace {

constexpr int DWM_LDS_PX = 8192;  // most pixels of a band's patch

// division of 24-bit numbers up to a known bound by one full-rate multiplication and a shift
struct SmallDiv {
    uint32_t m, s;
};
SmallDiv small_div(uint32_t d, uint32_t most) {  // most < 32768
    SmallDiv v = {0, 0};
    while (((uint64_t)1 << v.s) <= (uint64_t)most * d) ++v.s;
    v.m = (uint32_t)(((uint64_t)1 << v.s) / d + 1);
    return v;
}
__device__ __forceinline__ int sdiv(int x, const SmallDiv& d) { return (int)(__umul24((uint32_t)x, d.m) >> d.s); }
__device__ __forceinline__ int mad24(int a, int b, int c) { return (int)(__umul24((uint32_t)a, (uint32_t)b) + (uint32_t)c); }

// (Div: of the divisions that a workgroup needs once)
template <class Div, class Small>
struct DwmArgs {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    int IH, IW, OH, OW, FH, FW, sh, sw, ph, pw;
    int TH, PH, PW, NB;  // output rows of a band, patch rows of an image, patch columns, 4-pixel blocks of a quad's window
    int rpw, waves;      // patch rows of one copy instruction, waves of the workgroup
    int part;            // blocks of a patch row that lie together
    int QW, tab_w, tab, tab_at;  // quads of an output row; columns of the filter table and its entries (whole runs of 64), and where it starts
    int CG, bands, taps, has_bias;
    uint32_t grid;
    int64_t src_sn, dst_sn, z_sn;
    Div div_bands, div_cg, div_tab;
    SmallDiv div_qw;
    Small div_pw, div_nb, div_part, div_sw;
    EpiParams epi;

    auto numbers() const {
        return std::tie(IH, IW, OH, OW, FH, FW, sh, sw, ph, pw, TH, PH, PW, NB, rpw, waves, part, QW, tab_w, tab, tab_at, CG, bands, taps, has_bias, grid,
                        src_sn, dst_sn, z_sn, div_qw.m, div_qw.s);
    }
};
__device__ __forceinline__ int sdiv(int x, const Quot& d) { return (int)fdiv((uint32_t)x, d); }

// The two forms of the kernel's argument (see wire.h)
struct DwmWide {
    DwmArgs<FastDiv, SmallDiv> a;
    __device__ __forceinline__ DwmArgs<FastDiv, SmallDiv> open() const {
        asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.z), "s"(a.dst), "s"(a.IH), "s"(a.IW), "s"(a.OH), "s"(a.OW), "s"(a.FH), "s"(a.FW),
                     "s"(a.sh), "s"(a.sw), "s"(a.ph), "s"(a.pw), "s"(a.TH), "s"(a.PH), "s"(a.PW), "s"(a.NB), "s"(a.rpw), "s"(a.waves), "s"(a.part),
                     "s"(a.CG), "s"(a.bands), "s"(a.grid));
        asm volatile("" ::"s"(a.taps), "s"(a.has_bias), "s"(a.src_sn), "s"(a.dst_sn), "s"(a.z_sn), "s"(a.QW), "s"(a.tab_w), "s"(a.tab), "s"(a.tab_at),
                     "s"(a.div_bands.m), "s"(a.div_cg.m), "s"(a.div_tab.m), "s"(a.div_qw.m), "s"(a.div_pw.m), "s"(a.div_nb.m), "s"(a.epi.s_b),
                     "s"(a.epi.lin_lo));
        return a;
    }
};

struct DwmWire {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    // in, out: height | width << 16; window: its height, width, strides; pads: padding, rows per copy, waves; bands: output rows of a
    // band | bands << 16; more: channel blocks | entries of the filter table << 16; qw: its SmallDiv; part: blocks of a row together
    uint32_t grid, in, out, window, pads, bands, more, qw, part, flags;
    EpiWire epi;

    template <class Div, class Small>
    __host__ __device__ __forceinline__ void numbers(DwmArgs<Div, Small>& k) const {
        k.IH = wire_lo(in); k.IW = wire_hi(in); k.OH = wire_lo(out); k.OW = wire_hi(out);
        k.FH = wire_byte(window, 0); k.FW = wire_byte(window, 1); k.sh = wire_byte(window, 2); k.sw = wire_byte(window, 3);
        k.ph = wire_byte(pads, 0); k.pw = wire_byte(pads, 1); k.rpw = wire_byte(pads, 2); k.waves = wire_byte(pads, 3);
        k.TH = wire_lo(bands); k.bands = wire_hi(bands);
        k.CG = wire_lo(more); k.tab = wire_hi(more);
        k.part = (int)part; k.PW = wire_mul(k.part, 4, k.sw);
        k.PH = (k.TH - 1) * k.sh + k.FH;
        k.NB = (3 * k.sw + k.FW + 3) / 4;
        k.tab_w = k.NB * 4 + 3 * k.sw; k.tab_at = k.PH * k.PW + k.NB * 4;
        k.QW = (k.OW + 3) / 4;
        k.taps = k.FH * k.FW;
        k.has_bias = (int)(flags >> 8 & 1);
        k.grid = grid;
        k.src_sn = (uint32_t)wire_mul(k.CG, k.IH, k.IW * 4); k.dst_sn = (uint32_t)wire_mul(k.CG, k.OH, k.OW * 4);
        k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        k.div_qw.m = qw & 0xffffff; k.div_qw.s = qw >> 24;
    }
    __device__ __forceinline__ DwmArgs<Quot, Quot> open() const {
        asm volatile("" ::"s"(src), "s"(flt), "s"(bias), "s"(z), "s"(dst), "s"(grid), "s"(in), "s"(out), "s"(window), "s"(pads), "s"(bands), "s"(more),
                     "s"(qw), "s"(part), "s"(flags), "s"(epi.f[0]), "s"(epi.f[1]), "s"(epi.f[2]), "s"(epi.f[3]));  // one batch of scalar loads
        DwmArgs<Quot, Quot> k;
        k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
        numbers(k);
        k.div_bands = quot(k.bands); k.div_cg = quot(k.CG); k.div_tab = quot(k.tab_w);
        k.div_pw = quot(k.PW); k.div_nb = quot(k.NB); k.div_part = quot(k.part); k.div_sw = quot(k.sw);
        k.epi = epi_open(epi, flags & 255);
        return k;
    }
    // false: the problem has a number that does not fit
    bool pack(const DwmArgs<FastDiv, SmallDiv>& k) {
        src = k.src; flt = k.flt; bias = k.bias; z = k.z; dst = k.dst;
        grid = k.grid; in = wire2(k.IH, k.IW); out = wire2(k.OH, k.OW);
        window = wire4(k.FH, k.FW, k.sh, k.sw); pads = wire4(k.ph, k.pw, k.rpw, k.waves);
        bands = wire2(k.TH, k.bands); more = wire2(k.CG, k.tab);
        qw = k.div_qw.m | k.div_qw.s << 24; part = (uint32_t)k.part;
        flags = epi_wire(k.epi, false, &epi) | (k.has_bias ? 1u << 8 : 0);
        DwmArgs<FastDiv, SmallDiv> o;
        numbers(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return o.numbers() == k.numbers() && grid < QUOT_MAX;
    }
};
static_assert(sizeof(DwmWire) <= WIRE_BYTES, "a wire");

template <int STEPS, bool HZ, class Form>
__device__ __forceinline__ void dwm_run(const Form& form) {
    extern __shared__ __attribute__((aligned(16))) v4i lds_dwm[];  // patch, filter table
    const auto a = form.open();
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l16 = lane & 15, kq = lane >> 4;
    const uint32_t item = xcd_block(a.grid);
    const uint32_t i1 = fdiv_u(item, a.div_bands), band = item - i1 * a.bands;
    const uint32_t n = fdiv_u(i1, a.div_cg), cg = i1 - n * a.CG;
    const int oh0 = (int)band * a.TH, th = a.OH - oh0 < a.TH ? a.OH - oh0 : a.TH;
    const int plane = a.IH * a.IW * 4, oplane = a.OH * a.OW * 4;
    const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)lds_dwm);

    // Filter table: row by row, with 3 sw zeros in front (the later pixels of a quad start further on) and zeros behind
    {
        const v4i rs = uniform_rsrc(a.flt, (uint32_t)(a.CG * a.taps) * 4);
        for (int e = wave * 64; e < a.tab; e += a.waves * 64) {
            const int r = (int)fdiv(e + lane, a.div_tab), tap = e + lane - r * a.tab_w - 3 * a.sw;
            const bool ok = (r < a.FH) & ((unsigned)tap < (unsigned)a.FW);
            lds_copy64x4(lds0 + (uint32_t)(a.tab_at + e) * 4, ok ? ((int)cg * a.taps + r * a.FW + tap) * 4 : SENT, rs);
        }
    }
    const v4i bv = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(a.bias, a.has_bias ? a.CG * 16 : 0), (int)cg * 16, 0, 0);
    // the patch: lanes are the columns of `rpw` rows, or of 64 columns of one row
    {
        const v4i rs = uniform_rsrc(a.src + n * a.src_sn + (int64_t)cg * plane, (uint32_t)plane);
        const int r0 = a.PW < 64 ? sdiv(lane, a.div_pw) : 0, rows = a.PH;
        const int ih0 = oh0 * a.sh - a.ph, rstep = a.waves * a.rpw;
        for (int c = lane - r0 * a.PW, cb = 0; cb < a.PW; cb += 64, c += 64) {
            // every sw-th block of a row lies together: the windows of consecutive quads start at consecutive blocks, at any stride
            const int blk = c >> 2, part = sdiv(blk, a.div_part), iw = ((blk - part * a.part) * a.sw + part) * 4 + (c & 3) - a.pw;
            const bool in = (r0 < a.rpw) & (c < a.PW);
            // an invalid column is an invalid row from the start
            const int r_in = in ? r0 : 0x40000000;
            int ih = (unsigned)iw < (unsigned)a.IW ? ih0 + wave * a.rpw + r0 : 0x40000000;
            int off = ((ih0 + wave * a.rpw + r0) * a.IW + iw) * 4;
            for (int r = wave * a.rpw; r < rows; r += rstep) {
                if (r_in < rows - r) lds_copy64x4(lds0 + (uint32_t)(r * a.PW + cb) * 4, (unsigned)ih < (unsigned)a.IH ? off : SENT, rs);
                ih += rstep;
                off += rstep * a.IW * 4;
            }
        }
    }
    // while the copies run: where this lane finds its operands, and its first two units
    int boff[STEPS], woff[STEPS];
    const int mask = 0xff << (8 * (l16 & 3));
    {
        const int at = a.tab_at + (3 - (l16 >> 2)) * a.sw;
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            const int b = st * 4 + kq, row = sdiv(b, a.div_nb), q = b - mad24(row, a.NB, 0), turn = sdiv(q, a.div_sw);
            boff[st] = row < a.FH ? mad24(row, a.PW >> 2, mad24(q - mad24(turn, a.sw, 0), a.part, turn)) : 0;
            woff[st] = mad24(row, a.tab_w, q * 4) + at;
        }
    }
    const __amdgpu_buffer_rsrc_t rs_dst = make_rsrc(a.dst + n * a.dst_sn + (int64_t)cg * oplane, (uint32_t)oplane);
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z + n * a.z_sn + (int64_t)cg * oplane, HZ ? (uint32_t)oplane : 0u);
    const int quads = th * a.QW, out0 = oh0 * a.OW * 4, kq4 = out0 + kq * 4, x_end = a.OW - kq;
    struct Unit {
        int src, dst;  // first block of the window in LDS; byte offset of this lane's pixel, out of range if it has none
    };
    const int row_blk = a.sh * a.PW >> 2, row_b = a.OW * 4;
    auto unit = [&](int u) __attribute__((always_inline)) {
        const int qi = u + l16, qc = qi < quads ? qi : quads - 1;
        const int r = sdiv(qc, a.div_qw), q = qc - mad24(r, a.QW, 0);
        Unit o;
        o.src = mad24(r, row_blk, q);
        o.dst = ((qi < quads) & (q * 4 < x_end)) ? mad24(r, row_b, q * 16 + kq4) : SENT;
        return o;
    };
    const int step = a.waves * 32;
    Unit un[2];
    uint32_t zn[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        un[k] = unit(wave * 32 + k * 16);
        if (HZ) zn[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_z, un[k].dst, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<0>();
    __syncthreads();
    v4i fa[STEPS];
#pragma unroll
    for (int st = 0; st < STEPS; ++st)
#pragma unroll
        for (int p = 0; p < 4; ++p) fa[st][p] = reinterpret_cast<const int*>(lds_dwm)[woff[st] + p] & mask;
    // One loop per requantisation form: chosen inside it the form was a dozen branches per step (5x5, 60 channels at 76 x 22, batch 21, with a
    // residual: 6.99 -> 5.81 us; 240 channels at 57 x 57, stride 2, batch 16, H_SWISH: 7.41 -> 6.67).  Without branches the compiler reads a
    // step's operands further ahead: four steps take 73 to 95 registers, five and six waves per SIMD, where they took 49 to 70, five to eight, with
    // the choice inside.  They are bounded to five (unbounded: 544 channels at 95 x 100, stride 2, batch 22: 45.9 -> 52.0 us).  Longer windows would
    // spill then and keep the choice inside.
    auto multiply = [&](auto form_of) __attribute__((always_inline)) {
        constexpr int NL = decltype(form_of)::value;
        for (int u = wave * 32; u < quads; u += step) {
            v4i fb[2][STEPS];
            uint32_t zw[2] = {zn[0], zn[1]};
            int d[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
#pragma unroll
                for (int st = 0; st < STEPS; ++st) fb[k][st] = lds_dwm[un[k].src + boff[st]];
                d[k] = un[k].dst;
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                un[k] = unit(u + step + k * 16);
                if (HZ) zn[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_z, un[k].dst, 0, 0);
            }
            v4i acc[2] = {bv, bv};
#pragma unroll
            for (int st = 0; st < STEPS; ++st)
#pragma unroll
                for (int k = 0; k < 2; ++k) acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[st], fb[k][st], acc[k], 0, 0, 0);
            requant8_as<NL, HZ>(acc[0], acc[1], zw, a.epi);
#pragma unroll
            for (int k = 0; k < 2; ++k) __builtin_amdgcn_raw_buffer_store_b32(zw[k], rs_dst, d[k], 0, 0);
        }
    };
    if constexpr (STEPS <= 4) with_requant_form<HZ>(a.epi, multiply);
    else multiply(std::integral_constant<int, NL_ANY>());
}

template <int STEPS, bool HZ>
__global__ __launch_bounds__(256, 5) void dwm_kernel(DwmWire a) {
    dwm_run<STEPS, HZ>(a);
}
template <int STEPS, bool HZ>
__global__ __launch_bounds__(256, 5) void dwm_kernel(DwmWide a) {
    dwm_run<STEPS, HZ>(a);
}

template <int STEPS, class Form>
int launch_form(hipStream_t st, dim3 grid, dim3 block, int lds, const Form& form, bool hz) {
    typedef void (*Kernel)(Form);
    return launch_kernel(hz ? (Kernel)dwm_kernel<STEPS, true> : (Kernel)dwm_kernel<STEPS, false>, grid, block, lds, st, form);
}
template <int STEPS>
int launch_steps(hipStream_t st, dim3 grid, dim3 block, int lds, const DwmArgs<FastDiv, SmallDiv>& a, bool hz) {
    // Up to four workgroups per CU; beyond, opening the wire in each of them costs more than the launch gains (5x5, 1132 channels at 73 x 5,
    // batch 28, 7924 workgroups, as graph replays: 21.3 us wide, 22.7 so)
    DwmWire wire;
    return a.grid <= 1024 && wire.pack(a) ? launch_form<STEPS>(st, grid, block, lds, wire, hz) : launch_form<STEPS>(st, grid, block, lds, DwmWide{a}, hz);
}

int dwm_blocks(const ConvProblem& p) { return (3 * p.d.stride_w + (int)p.d.fw + 3) / 4; }

// whole blocks, as many for each of the sw parts
int dwm_columns(const ConvProblem& p) {
    const int sw = p.d.stride_w, cols = ((int)p.ow - 1) * sw + (int)p.d.fw;
    return (cols + 4 * sw - 1) / (4 * sw) * (4 * sw);
}

}  // namespace

bool dwm_usable(const ConvProblem& p) {
    const mi355_conv_desc& d = p.d;
    if (!depthwise_usable(p) || d.stride_w > 4 || d.stride_h > 64) return false;
    // matrix instructions of a quad, one output row's patch, and 24-bit products of rows and bytes
    return (int)d.fh * dwm_blocks(p) <= 32 && p.ow < 65536 && (int64_t)dwm_columns(p) * d.fh <= DWM_LDS_PX;
}

// Bands: as much of the patch as 16 KiB hold, so that eight workgroups share a CU; fewer rows where that leaves CUs without one.
DwmBands dwm_bands(const ConvProblem& p) {
    const mi355_conv_desc& d = p.d;
    const int QW = ((int)p.ow + 3) / 4, FH = d.fh, sh = d.stride_h;
    DwmBands b;
    b.PW = dwm_columns(p);
    const int64_t most = (4096 / b.PW - FH) / sh + 1;
    b.TH = most < 1 ? 1 : most < (int64_t)p.oh ? (int)most : (int)p.oh;
    while (b.TH > 1 && b.TH * QW > 64 && (int64_t)d.n * (d.ic / 4) * ((p.oh + b.TH - 1) / b.TH) < 256) b.TH = (b.TH + 1) / 2;
    b.bands = ((int)p.oh + b.TH - 1) / b.TH;
    b.TH = ((int)p.oh + b.bands - 1) / b.bands;  // even bands
    b.PH = (b.TH - 1) * sh + FH;
    b.rpw = b.PW < 64 ? 64 / b.PW : 1;
    const int units = (b.TH * QW + 15) / 16;
    b.waves = units > 4 ? 4 : units > 2 ? 2 : 1;
    return b;
}

int launch_dwm(hipStream_t st, const ConvProblem& p, const int8_t* src, const int8_t* flt, const int32_t* bias, const int8_t* z,
               int8_t* dst) {
    const mi355_conv_desc& d = p.d;
    DwmArgs<FastDiv, SmallDiv> a;
    a.src = src; a.flt = flt; a.bias = bias; a.z = z; a.dst = dst;
    a.IH = d.ih; a.IW = d.iw; a.OH = p.oh; a.OW = p.ow; a.FH = d.fh; a.FW = d.fw; a.sh = d.stride_h; a.sw = d.stride_w;
    a.ph = d.pad_h; a.pw = d.pad_w;
    const DwmBands b = dwm_bands(p);
    a.NB = dwm_blocks(p); a.PW = b.PW; a.part = a.PW / 4 / a.sw;
    a.CG = d.ic / 4; a.taps = d.fh * d.fw; a.QW = ((int)p.ow + 3) / 4;
    a.has_bias = d.bias_mode == MI355_BIAS_BROADCAST_CHANNEL;
    a.TH = b.TH; a.bands = b.bands; a.PH = b.PH; a.rpw = b.rpw; a.waves = b.waves;
    const int steps = (a.FH * a.NB + 3) / 4;
    a.tab_w = a.NB * 4 + 3 * a.sw;
    a.tab = (((steps * 4 - 1) / a.NB + 1) * a.tab_w + 63) / 64 * 64;
    a.tab_at = a.PH * a.PW + a.NB * 4;  // the window of a row's last quad may end past its columns
    a.src_sn = p.src_sn; a.dst_sn = p.dst_sn; a.z_sn = p.z_sn;
    a.div_bands = make_fastdiv(a.bands); a.div_cg = make_fastdiv(a.CG); a.div_tab = make_fastdiv(a.tab_w);
    a.div_qw = small_div(a.QW, a.TH * a.QW); a.div_pw = small_div(a.PW, 64); a.div_nb = small_div(a.NB, 32);
    a.div_part = small_div(a.part, a.PW / 4 + 16); a.div_sw = small_div(a.sw, 32);
    a.epi = p.epi;
    const int64_t items = (int64_t)d.n * a.CG * a.bands;
    if (items > 0x7fffffff) return (int)hipErrorInvalidValue;
    a.grid = (uint32_t)items;
    const int lds = (a.tab_at + a.tab) * 4;
    const dim3 grid((unsigned)items), block(64 * a.waves);
    switch (steps) {
        case 1: return launch_steps<1>(st, grid, block, lds, a, d.has_z);
        case 2: return launch_steps<2>(st, grid, block, lds, a, d.has_z);
        case 3: return launch_steps<3>(st, grid, block, lds, a, d.has_z);
        case 4: return launch_steps<4>(st, grid, block, lds, a, d.has_z);
        case 5: return launch_steps<5>(st, grid, block, lds, a, d.has_z);
        case 6: return launch_steps<6>(st, grid, block, lds, a, d.has_z);
        case 7: return launch_steps<7>(st, grid, block, lds, a, d.has_z);
        default: return launch_steps<8>(st, grid, block, lds, a, d.has_z);
    }
}

}  // namespace mi355
