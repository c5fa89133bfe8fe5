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
// twelve registers; the next band is in flight while this one is multiplied.
// 32 groups of 4 at 56 x 56, batch 16 (13 MB): 165 us as 32 launches, 9.8 with dot products, 6.6 here; 32 groups of 16
// (51 MB): 50 us with dot products, 17 here.  Small layers are a chain: with the filter staged beside the first band instead of
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
    int slabs, step;  // blocks of 16 channels; workgroups per slab
    int64_t src_sn, dst_sn, z_sn;
    Div div_pw, div_ow, div_bands;
    EpiParams epi;

    auto numbers() const {
        return std::tie(IH, IW, OH, OW, s, ph, pw, TH, PW, bands, items, log_icpg, src_scb, dst_scb, has_bias, slabs, step, src_sn, dst_sn, z_sn);
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
    uint32_t N, in, out, window, bands, per_image, step, flags;
    EpiWire epi;

    template <class Div>
    __host__ __device__ __forceinline__ void numbers(G16Args<Div>& k) const {
        k.IH = wire_lo(in); k.IW = wire_hi(in); k.OH = wire_lo(out); k.OW = wire_hi(out);
        k.s = wire_byte(window, 0); k.ph = wire_byte(window, 1); k.pw = wire_byte(window, 2); k.log_icpg = wire_byte(window, 3);
        k.TH = wire_lo(bands); k.slabs = wire_hi(bands); k.PW = (k.OW - 1) * k.s + 3;
        k.bands = (int)per_image; k.items = wire_mul((int)N, k.bands); k.step = (int)step;
        k.src_scb = wire_mul(k.IH, k.IW, 4); k.dst_scb = wire_mul(k.OH, k.OW, 4);
        k.src_sn = (uint32_t)wire_mul(k.slabs, 4, k.src_scb); k.dst_sn = (uint32_t)wire_mul(k.slabs, 4, k.dst_scb);
        k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        k.has_bias = (int)(flags >> 8 & 1);
    }
    __device__ __forceinline__ G16Args<Quot> open() const {
        asm volatile("" ::"s"(src), "s"(flt), "s"(bias), "s"(z), "s"(dst), "s"(N), "s"(in), "s"(out), "s"(window), "s"(bands), "s"(per_image), "s"(step),
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
        bands = wire2(k.TH, k.slabs); per_image = (uint32_t)k.bands; step = (uint32_t)k.step;
        flags = epi_wire(k.epi, false, &epi) | (k.has_bias ? 1u << 8 : 0);
        G16Args<FastDiv> o;
        numbers(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return o.numbers() == k.numbers() && k.items < QUOT_MAX;
    }
};
static_assert(sizeof(G16Wire) <= WIRE_BYTES, "a wire");

template <bool HZ, class Form>
__device__ __forceinline__ void grp16_run(const Form& form) {
    __shared__ __attribute__((aligned(16))) v4i sm[G16_PX], sf[144];
    const auto a = form.open();
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l16 = lane & 15, kq = lane >> 4, slab = blockIdx.y;
    const int PH = (a.TH - 1) * a.s + 3, patch = PH * a.PW;

    v4i x[G16_PX / 256];
    auto fetch = [&](int item) __attribute__((always_inline)) {
        const int n = (int)fdiv_u(item, a.div_bands), oh0 = (item - n * a.bands) * a.TH;
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
    };

    // The slab's filter is one contiguous piece, at most 2304 bytes: 16 bytes per thread into LDS, ahead of the band's pixels, and
    // from there each lane takes its dwords.  (Taken from memory, 48 gathers of 64 scattered dwords per workgroup cost more of the
    // vector-memory path than everything else.)
    const int icb = 1 << (a.log_icpg - 2), f_vecs = 36 * icb;
    const __amdgpu_buffer_rsrc_t rs_flt = make_rsrc(a.flt, (uint32_t)(a.slabs * f_vecs) * 16);
    const v4i f_vec = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, t < f_vecs ? (slab * f_vecs + t) * 16 : SENT, 0, 0);
    const v4i bv = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(a.bias, a.has_bias ? a.slabs * 64 : 0), (slab * 16 + kq * 4) * 4, 0, 0);
    int item = blockIdx.x;
    fetch(item);
    if (t < f_vecs) sf[t] = f_vec;
#pragma unroll
    for (int k = 0; k < G16_PX / 256; ++k) sm[t + k * 256] = x[k];
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
    for (;;) {
        const int next = item + a.step;
        if (next < a.items) fetch(next);  // lands during the multiplies
        const int n = (int)fdiv_u(item, a.div_bands), oh0 = (item - n * a.bands) * a.TH;
        const int pixels = (a.OH - oh0 < a.TH ? a.OH - oh0 : a.TH) * a.OW;
        const int64_t at = (int64_t)(slab * 4 + kq) * a.dst_scb + (int64_t)oh0 * a.OW * 4;
        int8_t* dst = a.dst + n * a.dst_sn + at;
        const int8_t* z = a.z + n * a.z_sn + at;
        // two units of 16 pixels at a time; the operands of the next two are read while these are requantised
        v4i fb[2][3];
        auto operands = [&](int u) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int p = u + k * 16 + l16, pp = p < pixels ? p : 0;
                const int oh = (int)fdiv(pp, a.div_ow), ow = pp - oh * a.OW;
                const v4i* px = sm + (oh * a.PW + ow) * a.s;
#pragma unroll
                for (int st = 0; st < 3; ++st) fb[k][st] = px[tap_off[st]];
            }
        };
        operands(wave * 32);
        for (int u = wave * 32; u < pixels; u += 128) {
            uint32_t zw[2] = {0, 0};
            v4i acc[2] = {bv, bv};
            if (HZ)
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int p = u + k * 16 + l16;
                    zw[k] = *reinterpret_cast<const uint32_t*>(z + (p < pixels ? p : 0) * 4);
                }
#pragma unroll
            for (int st = 0; st < 3; ++st)
#pragma unroll
                for (int k = 0; k < 2; ++k) acc[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[st], fb[k][st], acc[k], 0, 0, 0);
            operands(u + 128);
            __builtin_amdgcn_sched_barrier(0);
            requant8(acc[0], acc[1], zw, a.epi);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int p = u + k * 16 + l16;
                if (p < pixels) *reinterpret_cast<uint32_t*>(dst + p * 4) = zw[k];
            }
        }
        if (next >= a.items) break;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < G16_PX / 256; ++k) sm[t + k * 256] = x[k];
        __syncthreads();
        item = next;
    }
}

template <bool HZ>
__global__ __launch_bounds__(256) void grp16_kernel(G16Wire a) {
    grp16_run<HZ>(a);
}
template <bool HZ>
__global__ __launch_bounds__(256) void grp16_kernel(G16Wide a) {
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

bool g16_usable(const ConvProblem& p) {
    const mi355_conv_desc& d = p.d;
    return d.fh == 3 && d.fw == 3 && d.stride_h == d.stride_w && d.stride_h <= 2 && p.icpg == p.ocpg &&
           (p.icpg == 4 || p.icpg == 8 || p.icpg == 16) && d.oc % 16 == 0 && p.ow < G16_PX && g16_rows(p) > 0 &&
           (int64_t)d.ih * d.iw * 16 < (1ll << 31);
}

int launch_g16(hipStream_t st, const ConvProblem& p, const int8_t* src, const int8_t* flt, const int32_t* bias, const int8_t* z,
               int8_t* dst) {
    const mi355_conv_desc& d = p.d;
    G16Args<FastDiv> a;
    a.src = src; a.flt = reinterpret_cast<const int*>(flt); a.bias = bias; a.z = z; a.dst = dst;
    a.IH = d.ih; a.IW = d.iw; a.OH = p.oh; a.OW = p.ow; a.s = d.stride_h; a.ph = d.pad_h; a.pw = d.pad_w;
    const int slabs = d.oc / 16;
    a.TH = g16_rows(p);
    if (a.TH > (int)p.oh) a.TH = p.oh;
    // Fewer rows per band while that leaves CUs without one, or with one long one: a workgroup's fixed part is worth about 200
    // pixels (8 groups of 16 at 11 x 10, batch 30, 240 workgroups: 4.3 us, 5.0 with twice as many; 6 groups of 16 at 20 x 70, batch
    // 18, H_SWISH and a residual: 7.8 with bands of 420 pixels, 6.9 with 210).
    while (a.TH > 1) {
        const int64_t wgs = (int64_t)slabs * d.n * ((p.oh + a.TH - 1) / a.TH);
        if (wgs >= (a.TH * (int)p.ow > 400 ? 512 : 240)) break;
        a.TH = (a.TH + 1) / 2;
    }
    a.PW = ((int)p.ow - 1) * a.s + 3;
    a.bands = ((int)p.oh + a.TH - 1) / a.TH;
    const int64_t items = (int64_t)d.n * a.bands;
    if (items > 0x3fffffff) return (int)hipErrorInvalidValue;
    a.items = (int)items;
    a.log_icpg = p.icpg == 4 ? 2 : p.icpg == 8 ? 3 : 4; a.src_scb = d.ih * d.iw * 4; a.dst_scb = p.oh * p.ow * 4;
    a.has_bias = d.bias_mode == MI355_BIAS_BROADCAST_CHANNEL;
    a.src_sn = p.src_sn; a.dst_sn = p.dst_sn; a.z_sn = p.z_sn;
    a.div_pw = make_fastdiv(a.PW); a.div_ow = make_fastdiv(p.ow); a.div_bands = make_fastdiv(a.bands);
    a.epi = p.epi;
    int64_t per_slab = (2048 + slabs - 1) / slabs;  // eight workgroups per CU over all slabs
    if (per_slab > items) per_slab = items;
    a.slabs = slabs; a.step = (int)per_slab;
    const dim3 grid((unsigned)per_slab, slabs);
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

int launch_grp4(hipStream_t st, const ConvProblem& p, const int8_t* src, const int8_t* flt, const int32_t* bias, const int8_t* z,
                int8_t* dst) {
    const mi355_conv_desc& d = p.d;
    if (d.n == 0 || p.oh == 0 || p.ow == 0) return 0;
    if (g16_usable(p)) return launch_g16(st, p, src, flt, bias, z, dst);
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
