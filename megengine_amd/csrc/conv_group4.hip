// NCHW4 group convolutions with few channels per group, in one launch (tile "grp4_dot4": dot products in general, the matrix
// cores for the usual grouped bottleneck).
//
// Such a layer is G small convolutions.  As G launches of the dense tiles it costs G launch latencies, and a matrix tile of
// 32 channels is mostly empty when a group has 4, 8 or 16: 32 groups of 4 channels, 3x3 at 56 x 56, batch 16, took 165 us.
// Here a thread computes 4 or 8 channels of one group for two rows (3x3 filters; otherwise one) of one output column, one
// byte dot product per 4 input channels and tap:
//   * a wave's lanes are consecutive output columns of one group of one image: its loads and stores are contiguous runs of
//     4-byte pixels, and its filter words are the same for all lanes, so they are scalar loads and cost no vector memory;
//   * two output rows share the input rows between them (12 loads for 8 or 16 outputs at stride 1);
//   * what lies outside the image is an out-of-range offset of a buffer descriptor that spans the group's planes.
// Bound by the dot products (9 per 4 channels in and output) and the instructions around its loads.
//
// The usual grouped bottleneck -- 3x3, as many channels out of a group as into it, 4, 8 or 16 -- goes to the matrix cores
// all the same, sixteen channels at a time (one group of 16, two of 8, four of 4): the filter of the slab is a 16 x 16
// matrix per tap, block-diagonal where several groups share it, and sixteen channels of a pixel are exactly the 16 bytes
// a lane of v_mfma_i32_16x16x64_i8 holds, so a step is four taps and 3x3 is three steps, zeros of the block diagonal
// included a third of the time of the dot products.  A workgroup stages a band of input rows in LDS as [pixel][16
// channels] (NCHW4 keeps them in four planes), so every operand is one conflict-free ds_read_b128; the filter stays in
// twelve registers.  A workgroup is one band, with no band in flight behind it: other workgroups on the CU hide more than a second band's pixels
// in sixteen registers did (six of 77 to 80 registers fit, four of 100 to 104 with those).
// 32 groups of 4 at 56 x 56, batch 16 (13 MB): 165 us as 32 launches, 9.8 with dot products, 5.9 here; 32 groups of 16
// (51 MB): 50 us with dot products, 17 here; 47 groups of 16 at 78 x 8, batch 60: 20.7 with bands in a row,
// 16.8 one to a workgroup.  Small layers are a chain: with the filter staged beside the first band instead of
// gathered dword by dword ahead of it, and the next operands read while results are requantised, 55 groups of 16 at 8 x 47,
// stride 2, batch 4 went from 6.2 to 4.2 us, 5 groups of 16 at 33 x 100, stride 2, batch 64 from 9.8 to 8.4.
#include <tuple>

#include "igemm_shared.h"
#include "wire.h"

namespace mi355 {
namespace {

constexpr int GRP4_MAX_IC = 16;  // beyond, a group is worth a matrix tile of its own

template <class Div>
struct Grp4Args {
    const int8_t* src;
    const int* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    int IH, IW, OH, OW, FH, FW, sh, sw, ph, pw;
    int icb, ocpg, src_scb, dst_scb, has_bias;
    int64_t src_sn, dst_sn, z_sn;
    uint32_t items;
    Div div_ow, div_ocpg;
    EpiParams epi;

    auto numbers() const {
        return std::tie(IH, IW, OH, OW, FH, FW, sh, sw, ph, pw, icb, ocpg, src_scb, dst_scb, has_bias, src_sn, dst_sn, z_sn, items);
    }
};

// The two forms of the kernel's argument (see wire.h)
struct Grp4Wide {
    Grp4Args<FastDiv> a;
    template <int R>
    __device__ __forceinline__ const Grp4Args<FastDiv>& open() const { return a; }
};

struct Grp4Wire {
    const int8_t* src;
    const int* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    // in, out: height | width << 16; window: its height, width, strides; pads: padding, channel blocks into a group; channels: out of a
    // group | groups << 16
    uint32_t in, out, window, pads, channels, flags;
    EpiWire epi;

    template <int R, class Div>
    __host__ __device__ __forceinline__ void numbers(Grp4Args<Div>& k) const {
        k.IH = wire_lo(in); k.IW = wire_hi(in); k.OH = wire_lo(out); k.OW = wire_hi(out);
        k.FH = wire_byte(window, 0); k.FW = wire_byte(window, 1); k.sh = wire_byte(window, 2); k.sw = wire_byte(window, 3);
        k.ph = wire_byte(pads, 0); k.pw = wire_byte(pads, 1); k.icb = wire_byte(pads, 2);
        k.ocpg = wire_lo(channels);
        k.src_scb = wire_mul(k.IH, k.IW, 4); k.dst_scb = wire_mul(k.OH, k.OW, 4);
        k.src_sn = (uint32_t)wire_mul(wire_hi(channels), k.icb, k.src_scb);
        k.dst_sn = (uint32_t)wire_mul(wire_hi(channels), k.ocpg / 4, k.dst_scb);
        k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        k.items = (uint32_t)wire_mul((k.OH + R - 1) / R, k.OW);
        k.has_bias = (int)(flags >> 8 & 1);
    }
    template <int R>
    __device__ __forceinline__ Grp4Args<Quot> open() const {
        // (no asm statement to batch the loads: behind one the filter's words are no scalar loads any more)
        Grp4Args<Quot> k;
        k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
        numbers<R>(k);
        k.div_ow = quot(k.OW); k.div_ocpg = quot(k.ocpg);
        k.epi = epi_open(epi, flags & 255);
        return k;
    }
    // false: the problem has a number that does not fit
    template <int R>
    bool pack(const Grp4Args<FastDiv>& k, uint32_t groups) {
        src = k.src; flt = k.flt; bias = k.bias; z = k.z; dst = k.dst;
        in = wire2(k.IH, k.IW); out = wire2(k.OH, k.OW);
        window = wire4(k.FH, k.FW, k.sh, k.sw); pads = wire4(k.ph, k.pw, k.icb, 0); channels = wire2(k.ocpg, groups);
        flags = epi_wire(k.epi, false, &epi) | (k.has_bias ? 1u << 8 : 0);
        Grp4Args<FastDiv> o;
        numbers<R>(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return o.numbers() == k.numbers() && groups < 65536 && k.items < QUOT_MAX && (int64_t)groups * k.ocpg < QUOT_MAX;
    }
};
static_assert(sizeof(Grp4Wire) <= WIRE_BYTES, "a wire");

// OQ: output channel quads per thread; F = 3: 3x3 filter, stride ST, two output rows per thread; F = 0: any filter, one row
template <int OQ, int F, int ST, class Form>
__device__ __forceinline__ void grp4_run(const Form& form) {
    constexpr int R = F == 3 ? 2 : 1;
    const auto a = form.template open<R>();
    const uint32_t it = blockIdx.x * 256 + threadIdx.x;
    const bool live = it < a.items;
    const uint32_t ohs = fdiv(live ? it : 0, a.div_ow), ow = (live ? it : 0) - ohs * a.OW;
    const int oh0 = (int)ohs * R, oc0 = blockIdx.y * OQ * 4, g = (int)fdiv_u(oc0, a.div_ocpg);
    const int64_t n = blockIdx.z;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.src + n * a.src_sn + (int64_t)g * a.icb * a.src_scb, (uint32_t)(a.icb * a.src_scb));
    const int ih0 = oh0 * a.sh - a.ph, iw0 = (int)ow * a.sw - a.pw;
    const int T = F == 3 ? 9 : a.FH * a.FW;
    const int* __restrict__ w = a.flt + (int64_t)oc0 * a.icb * T;

    int acc[R][OQ * 4];
#pragma unroll
    for (int o = 0; o < OQ * 4; ++o)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][o] = a.has_bias ? a.bias[oc0 + o] : 0;

    // the residual is in flight while the sums are made
    const int64_t plane = n * a.dst_sn + (int64_t)(oc0 / 4) * a.dst_scb, zplane = n * a.z_sn + (int64_t)(oc0 / 4) * a.dst_scb;
    uint32_t zw[R][OQ] = {};
    if (a.epi.has_z) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int q = 0; q < OQ; ++q)
                if (live && oh0 + r < a.OH)
                    zw[r][q] = *reinterpret_cast<const uint32_t*>(a.z + zplane + (int64_t)q * a.dst_scb + ((oh0 + r) * a.OW + (int)ow) * 4);
    }

    for (int ib = 0; ib < a.icb; ++ib) {
        const int base = ib * a.src_scb;
        if constexpr (F == 3) {
            constexpr int ROWS = (R - 1) * ST + 3;
            int x[ROWS][3];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const int row = live && (unsigned)(ih0 + r) < (unsigned)a.IH ? ((ih0 + r) * a.IW + iw0) * 4 : SENT;
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    x[r][c] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (unsigned)(iw0 + c) < (unsigned)a.IW ? row + c * 4 : SENT, base, 0);
            }
#pragma unroll
            for (int o = 0; o < OQ * 4; ++o)
#pragma unroll
                for (int t = 0; t < 9; ++t) {
                    const int f = w[(o * a.icb + ib) * 9 + t];
#pragma unroll
                    for (int r = 0; r < R; ++r) acc[r][o] = __builtin_amdgcn_sdot4(x[r * ST + t / 3][t % 3], f, acc[r][o], false);
                }
        } else {
            for (int fh = 0; fh < a.FH; ++fh)
                for (int fw = 0; fw < a.FW; ++fw) {
                    const bool ok = live && (unsigned)(ih0 + fh) < (unsigned)a.IH && (unsigned)(iw0 + fw) < (unsigned)a.IW;
                    const int x = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, ok ? base + ((ih0 + fh) * a.IW + iw0 + fw) * 4 : SENT, 0, 0);
#pragma unroll
                    for (int o = 0; o < OQ * 4; ++o)
                        acc[0][o] = __builtin_amdgcn_sdot4(x, w[(o * a.icb + ib) * T + fh * a.FW + fw], acc[0][o], false);
                }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < OQ; ++q) {
            const uint32_t o = requant4(acc[r][4 * q], acc[r][4 * q + 1], acc[r][4 * q + 2], acc[r][4 * q + 3], zw[r][q], a.epi);
            if (live && oh0 + r < a.OH)
                *reinterpret_cast<uint32_t*>(a.dst + plane + (int64_t)q * a.dst_scb + ((oh0 + r) * a.OW + (int)ow) * 4) = o;
        }
}

template <int OQ, int F, int ST>
__global__ __launch_bounds__(256) void grp4_kernel(Grp4Wire a) {
    grp4_run<OQ, F, ST>(a);
}
template <int OQ, int F, int ST>
__global__ __launch_bounds__(256) void grp4_kernel(Grp4Wide a) {
    grp4_run<OQ, F, ST>(a);
}

template <int OQ, int F, int ST>
int launch_grp4_kernel(hipStream_t st, dim3 grid, const Grp4Args<FastDiv>& a, uint32_t groups) {
    Grp4Wire wire;
    // Up to two workgroups per CU the launch is what a call costs; beyond, opening the wire in every workgroup is.  Graph replays, wire / wide by
    // workgroups: to 255 1.01 .. 1.02 (0.05 us of kernels of 3, where a launch that is waited for gains 0.6), to 511 1.02 .. 1.04 (0.1 of 3.9),
    // to 1023 1.02 .. 1.03 (of 5), beyond 1.04 .. 1.06 (9 groups of 4 at 57 x 61, batch 20, 1260 workgroups: 4.43 us wide, 4.70 so).
    if ((uint64_t)grid.x * grid.y * grid.z <= 512 && wire.pack<F == 3 ? 2 : 1>(a, groups))
        return launch_kernel((void (*)(Grp4Wire))grp4_kernel<OQ, F, ST>, grid, dim3(256), 0, st, wire);
    return launch_kernel((void (*)(Grp4Wide))grp4_kernel<OQ, F, ST>, grid, dim3(256), 0, st, Grp4Wide{a});
}

constexpr int64_t G16_BANDS = 1 << 24;  // bands of a batch (256 times as many threads in a grid's first dimension)
constexpr int G16_PX = 1024;  // pixels of a staged band (16 KiB), four per thread

template <class Div>
struct G16Args {
    const int8_t* src;
    const int* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    int IH, IW, OH, OW, s, ph, pw;
    int TH, PW, bands, items;  // output rows of a band, padded input columns, bands per image, bands of the batch
    int log_icpg, src_scb, dst_scb, has_bias;
    int slabs;  // blocks of 16 channels
    int64_t src_sn, dst_sn, z_sn;
    Div div_pw, div_ow, div_bands;
    EpiParams epi;

    auto numbers() const {
        return std::tie(IH, IW, OH, OW, s, ph, pw, TH, PW, bands, items, log_icpg, src_scb, dst_scb, has_bias, slabs, src_sn, dst_sn, z_sn);
    }
};

struct G16Wide {
    G16Args<FastDiv> a;
    // everything up to the first operands in one batch of scalar loads, and a word of each line that the epilogue reads
    __device__ __forceinline__ G16Args<FastDiv> open() const {
        asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.z), "s"(a.dst), "s"(a.IH), "s"(a.IW), "s"(a.OH), "s"(a.OW), "s"(a.s), "s"(a.ph),
                     "s"(a.pw), "s"(a.TH), "s"(a.PW), "s"(a.bands), "s"(a.items), "s"(a.log_icpg), "s"(a.src_scb), "s"(a.dst_scb), "s"(a.has_bias),
                     "s"(a.slabs), "s"(a.src_sn), "s"(a.div_pw.m), "s"(a.div_bands.m), "s"(a.div_ow.m), "s"(a.epi.s_b), "s"(a.epi.lin_lo));
        return a;
    }
};

struct G16Wire {
    const int8_t* src;
    const int* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    // in, out: height | width << 16; window: stride, padding, log of a group's channels; bands: output rows of one | slabs << 16
    uint32_t N, in, out, window, bands, per_image, flags;
    EpiWire epi;

    template <class Div>
    __host__ __device__ __forceinline__ void numbers(G16Args<Div>& k) const {
        k.IH = wire_lo(in); k.IW = wire_hi(in); k.OH = wire_lo(out); k.OW = wire_hi(out);
        k.s = wire_byte(window, 0); k.ph = wire_byte(window, 1); k.pw = wire_byte(window, 2); k.log_icpg = wire_byte(window, 3);
        k.TH = wire_lo(bands); k.slabs = wire_hi(bands); k.PW = (k.OW - 1) * k.s + 3;
        k.bands = (int)per_image; k.items = wire_mul((int)N, k.bands);
        k.src_scb = wire_mul(k.IH, k.IW, 4); k.dst_scb = wire_mul(k.OH, k.OW, 4);
        k.src_sn = (uint32_t)wire_mul(k.slabs, 4, k.src_scb); k.dst_sn = (uint32_t)wire_mul(k.slabs, 4, k.dst_scb);
        k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        k.has_bias = (int)(flags >> 8 & 1);
    }
    __device__ __forceinline__ G16Args<Quot> open() const {
        asm volatile("" ::"s"(src), "s"(flt), "s"(bias), "s"(z), "s"(dst), "s"(N), "s"(in), "s"(out), "s"(window), "s"(bands), "s"(per_image),
                     "s"(flags), "s"(epi.f[0]), "s"(epi.f[1]), "s"(epi.f[2]), "s"(epi.f[3]));  // one batch of scalar loads
        G16Args<Quot> k;
        k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
        numbers(k);
        k.div_pw = quot(k.PW); k.div_ow = quot(k.OW); k.div_bands = quot(k.bands);
        k.epi = epi_open(epi, flags & 255);
        return k;
    }
    // false: the problem has a number that does not fit
    bool pack(const G16Args<FastDiv>& k, uint32_t n) {
        src = k.src; flt = k.flt; bias = k.bias; z = k.z; dst = k.dst;
        N = n; in = wire2(k.IH, k.IW); out = wire2(k.OH, k.OW); window = wire4(k.s, k.ph, k.pw, k.log_icpg);
        bands = wire2(k.TH, k.slabs); per_image = (uint32_t)k.bands;
        flags = epi_wire(k.epi, false, &epi) | (k.has_bias ? 1u << 8 : 0);
        G16Args<FastDiv> o;
        numbers(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return o.numbers() == k.numbers() && k.items < QUOT_MAX;
    }
};
static_assert(sizeof(G16Wire) <= WIRE_BYTES, "a wire");

struct G16Lane {
    int ow[2], at[2];  // of the lane's two pixels of a band's first step: column out, byte of the staged band
    int OW, step, wrap, cols, last;  // (uniform) columns out; 128 pixels on: bytes, bytes where the row ends, columns; the last pixel's byte
    int tap[3];        // byte of the lane's tap of each matrix step, relative to the pixel
    int out, p;        // byte of the first pixel in the planes of the slab; the pixel
};

// The two offsets of unit k of step u, pixels from p = l.p + u + 16 k on, in the four planes of a slab.  first: the wave's first pixel.  (Past the
// wave's last step nothing is loaded, and the scalar offset would lead out of planes of few pixels: by the rule at SENT it is zero there.)
struct G16Access {
    int lane, scalar;
};
__host__ __device__ __forceinline__ G16Access g16_access(const G16Lane& l, int k, int u, int first, int pixels, int base) {
    return {l.p + u + k * 16 < pixels ? l.out + k * 64 : SENT, first + u < pixels ? base + u * 4 : 0};
}

// The pixels of one staged band, two units of 16 per wave and step; the operands and the residual of the next step are read while this
// one is requantised.
template <int NL, bool HZ>
__device__ __forceinline__ void grp16_band(const EpiParams& epi, const G16Lane& l, const v4i* sm, const v4i (&fa)[3], v4i bv,
                                           __amdgpu_buffer_rsrc_t rs_dst, __amdgpu_buffer_rsrc_t rs_z, int base, int pixels, int first) {
    v4i fb[2][3];
    uint32_t zn[2] = {0, 0};
    int ow[2] = {l.ow[0], l.ow[1]}, at[2] = {l.at[0], l.at[1]};
    const char* band = reinterpret_cast<const char*>(sm);
    auto operands = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int here = at[k] < l.last ? at[k] : l.last;  // (past the band: any pixel of it)
#pragma unroll
            for (int st = 0; st < 3; ++st) fb[k][st] = *reinterpret_cast<const v4i*>(band + here + l.tap[st]);
            ow[k] += l.cols;
            at[k] += l.step;
            const bool over = ow[k] >= l.OW;
            ow[k] -= over ? l.OW : 0;
            at[k] += over ? l.wrap : 0;
        }
    };
    auto residual = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const G16Access at = g16_access(l, k, u, first, pixels, base);
            zn[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_z, at.lane, at.scalar, 0);
        }
    };
    if (HZ) residual(0);
    operands();
    for (int u = 0; first + u < pixels; u += 128) {
        uint32_t zw[2] = {zn[0], zn[1]};
        v4i acc[2] = {bv, bv};
#pragma unroll
        for (int st = 0; st < 3; ++st)
#pragma unroll
            for (int k = 0; k < 2; ++k) acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[st], fb[k][st], acc[k], 0, 0, 0);
        operands();
        if (HZ) residual(u + 128);
        __builtin_amdgcn_sched_barrier(0);
        requant8_as<NL, HZ>(acc[0], acc[1], zw, epi);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const G16Access to = g16_access(l, k, u, first, pixels, base);
            __builtin_amdgcn_raw_buffer_store_b32((int)zw[k], rs_dst, to.lane, to.scalar, 0);
        }
    }
}

template <bool HZ, class Form>
__device__ __forceinline__ void grp16_run(const Form& form) {
    __shared__ __attribute__((aligned(16))) v4i sm[G16_PX], sf[144];
    const auto a = form.open();
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l16 = lane & 15, kq = lane >> 4, slab = blockIdx.y;
    const int PH = (a.TH - 1) * a.s + 3, patch = PH * a.PW;

    // The slab's filter is one contiguous piece, at most 2304 bytes: 16 bytes per thread into LDS, ahead of the band's pixels, and
    // from there each lane takes its dwords.  (Taken from memory, 48 gathers of 64 scattered dwords per workgroup cost more of the
    // vector-memory path than everything else.)
    const int icb = 1 << (a.log_icpg - 2), f_vecs = 36 * icb;
    const __amdgpu_buffer_rsrc_t rs_flt = make_rsrc(a.flt, (uint32_t)(a.slabs * f_vecs) * 16);
    const v4i f_vec = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, t < f_vecs ? (slab * f_vecs + t) * 16 : SENT, 0, 0);
    const v4i bv = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(a.bias, a.has_bias ? a.slabs * 64 : 0), (slab * 16 + kq * 4) * 4, 0, 0);
    const int item = blockIdx.x, n = (int)fdiv_u(item, a.div_bands), oh0 = (item - n * a.bands) * a.TH;
    {
        v4i x[G16_PX / 256];
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.src + n * a.src_sn + (int64_t)slab * 4 * a.src_scb, (uint32_t)a.src_scb * 4);
#pragma unroll
        for (int k = 0; k < G16_PX / 256; ++k) {
            const uint32_t p = t + k * 256, pr = fdiv(p, a.div_pw), pc = p - pr * a.PW;
            const int ih = oh0 * a.s - a.ph + (int)pr, iw = (int)pc - a.pw;
            const bool ok = (int)p < patch && (unsigned)ih < (unsigned)a.IH && (unsigned)iw < (unsigned)a.IW;
            const int off = ok ? (ih * a.IW + iw) * 4 : SENT;
#pragma unroll
            for (int b = 0; b < 4; ++b) x[k][b] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, off, b * a.src_scb, 0);
        }
        if (t < f_vecs) sf[t] = f_vec;
#pragma unroll
        for (int k = 0; k < G16_PX / 256; ++k) sm[t + k * 256] = x[k];
    }
    __syncthreads();
    // filter rows: lane = output channel, 16 bytes of tap 4 step + kq = its 16 input channels, zero outside its group
    v4i fa[3];
    int tap_off[3];
    const int first = (l16 >> a.log_icpg) * icb;  // first channel block of the lane's group
#pragma unroll
    for (int st = 0; st < 3; ++st) {
        const int tap = st * 4 + kq;
        tap_off[st] = tap < 9 ? tap / 3 * a.PW + tap % 3 : 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const bool in = (tap < 9) & (b >= first) & (b < first + icb);
            const int w = reinterpret_cast<const int*>(sf)[in ? (l16 * icb + b - first) * 9 + tap : 0];
            fa[st][b] = in ? w : 0;
        }
    }
    // Where a lane's two pixels of a step lie: column out and byte of the staged band.  Every band begins with the same, and 128 pixels
    // further on is a sum and a wrap (a division per pixel and step, with its quarter-rate multiplications, was a third of the loop's
    // vector instructions).
    const uint32_t rows128 = fdiv_u(128, a.div_ow);
    const int cols128 = 128 - (int)rows128 * a.OW;
    G16Lane l;
    l.step = ((int)rows128 * a.PW + cols128) * a.s * 16;
    l.wrap = (a.PW - a.OW) * a.s * 16;
    l.cols = cols128;
    l.OW = a.OW;
    l.last = (((a.TH - 1) * a.PW + a.OW - 1) * a.s) * 16;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int p = wave * 32 + k * 16 + l16, oh = (int)fdiv(p, a.div_ow);
        l.ow[k] = p - oh * a.OW;
        l.at[k] = (oh * a.PW + l.ow[k]) * a.s * 16;
    }
#pragma unroll
    for (int st = 0; st < 3; ++st) l.tap[st] = tap_off[st] * 16;
    l.out = kq * a.dst_scb + (wave * 32 + l16) * 4;
    l.p = wave * 32 + l16;
    const int pixels = (a.OH - oh0 < a.TH ? a.OH - oh0 : a.TH) * a.OW;
    const __amdgpu_buffer_rsrc_t rs_dst = make_rsrc(a.dst + n * a.dst_sn + (int64_t)slab * 4 * a.dst_scb, (uint32_t)a.dst_scb * 4);
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z + (HZ ? n * a.z_sn + (int64_t)slab * 4 * a.dst_scb : 0), HZ ? (uint32_t)a.dst_scb * 4 : 0);
    // one loop per requantisation form: with the choice inside it a step was a dozen branches longer and the kernel held 116 registers
    with_requant_form<HZ>(a.epi, [&](auto form_of) __attribute__((always_inline)) {
        grp16_band<decltype(form_of)::value, HZ>(a.epi, l, sm, fa, bv, rs_dst, rs_z, oh0 * a.OW * 4, pixels, wave * 32);
    });
}

template <bool HZ>
__global__ __launch_bounds__(256, 6) void grp16_kernel(G16Wire a) {
    grp16_run<HZ>(a);
}
template <bool HZ>
__global__ __launch_bounds__(256, 6) void grp16_kernel(G16Wide a) {
    grp16_run<HZ>(a);
}

template <class Form>
int launch_g16_form(hipStream_t st, dim3 grid, const Form& form, bool hz) {
    typedef void (*Kernel)(Form);
    return launch_kernel(hz ? (Kernel)grp16_kernel<true> : (Kernel)grp16_kernel<false>, grid, dim3(256), 0, st, form);
}

// output rows of a band: the largest number whose input patch fits; 0: not even one row fits
int g16_rows(const ConvProblem& p) {
    const int s = p.d.stride_h, pw = ((int)p.ow - 1) * s + 3;
    const int rows = (int)(G16_PX / pw);
    return rows < 3 ? 0 : (rows - 3) / s + 1;
}

// Output rows of a band, one band to a workgroup: equal bands (oh = 87 in rows of 44, not 76 and 11), as many as cost least.  A workgroup
// takes 0.29 us of its CU and 0.06 per step of 128 pixels, beside 0.09 per step of its own chain and 0.12 of memory; W: workgroups of the
// busiest CU, w: on average.  Fitted to graph replays of every band of 160 drawn layers: 0.3 % behind the best band on average, 6 % at most,
// where fewer rows until there were 240 or 512 workgroups was 5.4 % behind (8 groups of 16 at 46 x 30, batch 42: 6.91 -> 5.69 us).
int g16_band_rows(const ConvProblem& p, int cu_count) {
    const int rows = g16_rows(p), oh = (int)p.oh, ow = (int)p.ow, cu = cu_count > 0 ? cu_count : 256;
    int best = 0;
    float least = 0.f;
    for (int bands = (oh + rows - 1) / rows;;) {
        const int th = (oh + bands - 1) / bands, steps = (th * ow + 127) / 128;
        const int64_t items = (int64_t)p.d.n * ((oh + th - 1) / th), wgs = items * (p.d.oc / 16);
        const float W = (float)((wgs + cu - 1) / cu), w = (float)wgs / (float)cu;
        const float cost = (float)steps * (0.091f + 0.117f * w + 0.059f * W) + 0.287f * W;
        if (best == 0 || (cost < least && items < G16_BANDS)) {
            best = th;
            least = cost;
        }
        if (th == 1 || steps == 1) return best;
        bands = (oh + th - 2) / (th - 1);  // the next smaller band
    }
}

bool g16_usable(const ConvProblem& p) {
    const mi355_conv_desc& d = p.d;
    return d.fh == 3 && d.fw == 3 && d.stride_h == d.stride_w && d.stride_h <= 2 && p.icpg == p.ocpg &&
           (p.icpg == 4 || p.icpg == 8 || p.icpg == 16) && d.oc % 16 == 0 && p.ow < G16_PX && g16_rows(p) > 0 &&
           (int64_t)d.ih * d.iw * 16 < (1ll << 31) && (int64_t)p.oh * p.ow * 16 < (1ll << 31) &&
           (int64_t)d.n * ((p.oh + g16_rows(p) - 1) / g16_rows(p)) < G16_BANDS;
}

int launch_g16(hipStream_t st, const ConvProblem& p, int cu_count, const int8_t* src, const int8_t* flt, const int32_t* bias, const int8_t* z,
               int8_t* dst) {
    const mi355_conv_desc& d = p.d;
    G16Args<FastDiv> a;
    a.src = src; a.flt = reinterpret_cast<const int*>(flt); a.bias = bias; a.z = z; a.dst = dst;
    a.IH = d.ih; a.IW = d.iw; a.OH = p.oh; a.OW = p.ow; a.s = d.stride_h; a.ph = d.pad_h; a.pw = d.pad_w;
    const int slabs = d.oc / 16;
    a.TH = g16_band_rows(p, cu_count);
    a.PW = ((int)p.ow - 1) * a.s + 3;
    a.bands = ((int)p.oh + a.TH - 1) / a.TH;
    const int64_t items = (int64_t)d.n * a.bands;
    a.items = (int)items;
    a.log_icpg = p.icpg == 4 ? 2 : p.icpg == 8 ? 3 : 4; a.src_scb = d.ih * d.iw * 4; a.dst_scb = p.oh * p.ow * 4;
    a.has_bias = d.bias_mode == MI355_BIAS_BROADCAST_CHANNEL;
    a.src_sn = p.src_sn; a.dst_sn = p.dst_sn; a.z_sn = p.z_sn;
    a.div_pw = make_fastdiv(a.PW); a.div_ow = make_fastdiv(p.ow); a.div_bands = make_fastdiv(a.bands);
    a.epi = p.epi;
    a.slabs = slabs;
    const dim3 grid((unsigned)items, slabs);
    G16Wire wire;
    return wire.pack(a, d.n) ? launch_g16_form(st, grid, wire, d.has_z) : launch_g16_form(st, grid, G16Wide{a}, d.has_z);
}

}  // namespace

// Whether one launch is ahead of a dense launch per group.  The matrix form always is (165 sizes of 2 to 64 groups, batch 1 to
// 64, 7 x 7 to 112 x 112), and 3x3 dot products at stride 2 almost always.  The others lose where a group is large -- the
// dense patch tiles run on the matrix cores -- or has many taps: without the unrolled 3x3 form a thread loads and waits for
// one tap after the other.  The two sides in us, fitted to graph replays of 1775 sizes of 4 to 16 channels into a group and
// 4 to 128 out of it, filters 1x1 to 7x7, 1x7 and 3x6, with outputs, dot products and matrix steps in millions:
//   one launch      3x3: 4 + 0.5 outputs + 0.04 dot products
//                   others: 3 + 0.145 per tap and channel block (in a row, for any size) + 1 outputs + 0.22 dot products
//   each group      3.6 + 0.05 matrix steps (pixels x taps x output channels in 32s x input channels in 16s)
//   all groups      0.1 outputs, with a residual 0.5
// One launch is kept up to a quarter more, which G submissions cost the host.  Of the 1775, 435 go group by group for it, one
// launch against those: 2.6 times faster on average (2 groups 16 -> 116, 7x7 at 33 x 39, batch 51: 590 us / 46; 4 groups 16 ->
// 120, 3x3 at 90 x 67, batch 38: 173 / 81; 6 groups 16 -> 76, 7x7 at 8 x 14, batch 12: 77 / 29; 3 groups 12 -> 100, 1x1 at 57 x
// 79, batch 44: 114 / 42), none of them more than a fifth slower; of what stays, 29 are behind by more than a quarter, at most by
// 2.2 times (34 groups 8 -> 108, 7x7 stride 2 at 31 x 8).  On 250 other sizes 44 change sides and are 2.2 times faster on average.
bool grp4_pick(const ConvProblem& p) {
    const mi355_conv_desc& d = p.d;
    if (!grp4_usable(p)) return false;
    if (g16_usable(p)) return true;
    const bool f3 = d.fh == 3 && d.fw == 3 && d.stride_h == d.stride_w;
    if (f3 && d.stride_h == 2) return true;
    const double pixels = (double)d.n * p.oh * p.ow * 1e-6, outputs = pixels * d.oc;
    const double taps = (double)d.fh * d.fw, serial = taps * (p.icpg / 4), dots = outputs * serial;
    const double steps = pixels * taps * ((p.ocpg + 31) / 32 * 32) * ((p.icpg + 15) / 16);
    const double one = f3 && d.stride_h == 1 ? 4 + 0.5 * outputs + 0.04 * dots : 3 + 0.145 * serial + outputs + 0.22 * dots;
    const double groups = d.group * (3.6 + 0.05 * steps) + (d.has_z ? 0.5 : 0.1) * outputs;
    return one <= 1.25 * groups;
}

bool grp4_usable(const ConvProblem& p) {
    const mi355_conv_desc& d = p.d;
    return d.format == MI355_FMT_NCHW4 && d.group > 1 && !p.dw4 && p.icpg % 4 == 0 && p.ocpg % 4 == 0 && p.icpg <= GRP4_MAX_IC &&
           d.n <= 65535 && d.oc / 4 <= 65535 && (uint64_t)p.oh * p.ow < (1u << 28);
}

int launch_grp4(hipStream_t st, const ConvProblem& p, int cu_count, const int8_t* src, const int8_t* flt, const int32_t* bias, const int8_t* z,
                int8_t* dst) {
    const mi355_conv_desc& d = p.d;
    if (d.n == 0 || p.oh == 0 || p.ow == 0) return 0;
    if (g16_usable(p)) return launch_g16(st, p, cu_count, src, flt, bias, z, dst);
    Grp4Args<FastDiv> a;
    a.src = src; a.flt = reinterpret_cast<const int*>(flt); a.bias = bias; a.z = z; a.dst = dst;
    a.IH = d.ih; a.IW = d.iw; a.OH = p.oh; a.OW = p.ow; a.FH = d.fh; a.FW = d.fw;
    a.sh = d.stride_h; a.sw = d.stride_w; a.ph = d.pad_h; a.pw = d.pad_w;
    a.icb = p.icpg / 4; a.ocpg = p.ocpg;
    a.src_scb = d.ih * d.iw * 4; a.dst_scb = p.oh * p.ow * 4;
    a.has_bias = d.bias_mode == MI355_BIAS_BROADCAST_CHANNEL;
    a.src_sn = p.src_sn; a.dst_sn = p.dst_sn; a.z_sn = p.z_sn;
    a.div_ow = make_fastdiv(p.ow); a.div_ocpg = make_fastdiv(p.ocpg);
    a.epi = p.epi;
    const bool f3 = d.fh == 3 && d.fw == 3 && d.stride_h == d.stride_w && d.stride_h <= 2;
    const bool wide = p.ocpg % 8 == 0;  // 8 channels per thread halve the loads per output
    a.items = (f3 ? (p.oh + 1) / 2 : p.oh) * p.ow;
    const dim3 grid((a.items + 255) / 256, d.oc / (wide ? 8 : 4), d.n);
    if (f3 && d.stride_h == 1) return wide ? launch_grp4_kernel<2, 3, 1>(st, grid, a, d.group) : launch_grp4_kernel<1, 3, 1>(st, grid, a, d.group);
    if (f3) return wide ? launch_grp4_kernel<2, 3, 2>(st, grid, a, d.group) : launch_grp4_kernel<1, 3, 2>(st, grid, a, d.group);
    return wide ? launch_grp4_kernel<2, 0, 1>(st, grid, a, d.group) : launch_grp4_kernel<1, 0, 1>(st, grid, a, d.group);
}

}  // namespace mi355
