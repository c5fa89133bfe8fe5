// Pointwise (1x1) int8 ConvBias on 4-packed activations, NCHW4 in and out.  At stride 1 pw4q_kernel and pw4k_kernel below;
// pw4s_kernel serves strided layers of the two kinds that a tiled kernel serves badly: at most 64 input channels and many output channels (the expansion layers of the MobileNet
// family: one or two MFMA k-steps, the cost is the output), and at most 32 output channels with up to 192 input
// channels (its narrow projections: a tile of 128 filter rows would be three quarters empty).
//
// A tiled implicit GEMM spends such a layer on its per-tile pipeline (stage, barrier, multiply: one k-stage per tile).
// Here nothing is staged and nothing is shared after the first barrier:
//   * a wave keeps the filter rows of its 32, 64 or 96 output channels in registers for the whole launch
//     (MFMA A fragments: lane = output channel, 16 contiguous k-bytes of its row);
//   * it walks blocks of 32 pixels; a lane's B fragment -- 16 k-bytes of its pixel = 4 channel blocks -- is four
//     coalesced dword loads (32 consecutive pixels x 4 bytes each), fetched for the NEXT block, together with its
//     residual, while this one is multiplied and requantised;
//   * accumulators start from the bias (LDS copy), the fused epilogue and the NCHW4 stores are those of the tiled
//     kernels (igemm_shared.h).
// Channel blocks past the last one, and filter bytes past the end of a row, meet zero activations.
#include <string.h>

#include <tuple>
#include <type_traits>

#include "igemm_shared.h"
#include "wire.h"

namespace mi355 {
namespace {

constexpr int PW4_MAX_OC = 1024;

// All loads so far have landed, and the compiler knows.  Ahead of a loop whose loads run a step ahead: with the first step's
// loads possibly pending at the loop's head, the wait that the compiler puts there is for everything, the stores of the step
// before included.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// How the waves of a streaming launch walk the pixel blocks: wave g of the launch (of its XCD's share of the launch) takes the
// channel group g % n_ocg of the blocks g / n_ocg, + step, ...  With slabs the XCDs take one contiguous eighth of the blocks
// each.  The divisions are the host's: a run-time integer division is 0.1 us on the way to the first load.
template <class Div>
struct PwWalk {
    int n_ocg, step, slabs;
    Div div_ocg;
};
PwWalk<FastDiv> make_walk(int64_t blocks, int n_ocg) {
    PwWalk<FastDiv> w;
    w.n_ocg = n_ocg;
    w.slabs = blocks % 8 == 0 && blocks / 8 * 4 % n_ocg == 0;
    w.step = (int)((w.slabs ? blocks / 8 : blocks) * 4 / n_ocg);
    w.div_ocg = make_fastdiv(n_ocg);
    return w;
}
template <class Div>
__device__ __forceinline__ void pw_walk(const PwWalk<Div>& w, int n_pb, int wave, int* pb0, int* pb_hi, int* ocg) {
    int lo = 0, hi = n_pb, g = (int)blockIdx.x * 4 + wave;
    if (w.slabs) {
        const int xc = blockIdx.x & 7, per = n_pb >> 3, rem = n_pb & 7;
        lo = xc * per + (xc < rem ? xc : rem);
        hi = lo + per + (xc < rem ? 1 : 0);
        g = (int)(blockIdx.x >> 3) * 4 + wave;
    }
    const int q = (int)fdiv_u(g, w.div_ocg);
    *ocg = g - q * w.n_ocg;
    *pb0 = lo + q;
    *pb_hi = hi;
}

// HZ: the launch has a residual (its registers exist only in that instantiation)
template <int MT, int KC, bool HZ>
__global__ __launch_bounds__(256) void pw4s_kernel(IgemmArgs a, int n_ocg, int n_pb) {
    __shared__ __attribute__((aligned(16))) int sBias[PW4_MAX_OC + 96];
    const int t = threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l32 = lane & 31, lh = lane >> 5;

    const int gw = blockIdx.x * 4 + wave, GW = gridDim.x * 4;  // GW is a multiple of n_ocg
    const int pb0 = gw / n_ocg, ocg = gw - pb0 * n_ocg, step = GW / n_ocg;
    const int oc_w = ocg * MT * 32;
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes);
    const __amdgpu_buffer_rsrc_t rs_flt = make_rsrc(a.flt, a.flt_bytes);

    v4i fa[MT][KC];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = oc_w + i * 32 + l32;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
            fa[i][kc] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, row < a.OC ? row * a.kbytes + kc * 32 + lh * 16 : SENT, 0, 0);
    }

    const int icb = a.kbytes >> 2;
    auto load_b = [&](int pb, v4i (&x)[KC]) __attribute__((always_inline)) {
        const int m = pb * 32 + l32;
        const bool ok = m < a.M;  // also false for every block past the last one
        const uint32_t mm = ok ? m : 0;
        const uint32_t n = fdiv(mm, a.div_ohw), rem = mm - n * a.OHW;
        const uint32_t oh = fdiv(rem, a.div_ow), ow = rem - oh * a.OW;
        const int pix = (int)n * a.src_sn + ((int)oh * a.sh * a.IW + (int)ow * a.sw) * 4;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int cb = kc * 8 + lh * 4 + i;
                x[kc][i] = __builtin_amdgcn_raw_buffer_load_b32(rs_src, (ok && cb < icb) ? pix + cb * a.src_scb : SENT, 0, 0);
            }
    };

    v4i fb[KC], nb[KC];
    ZRegs<HZ ? MT : 1, 1> zr, nz;
    load_b(pb0, fb);
    if constexpr (HZ) igemm_load_z<4, MT, 1>(a, zr, oc_w, pb0 * 32, l32, lh);
    // the bias goes to LDS after the filter rows and the first block are requested: one memory round trip before the
    // first multiply instead of two (the barrier waits for everything outstanding)
    for (int i = t; i < PW4_MAX_OC + 96; i += 256) sBias[i] = (a.has_bias && i < a.OC) ? a.bias[i] : 0;
    __syncthreads();
    for (int pb = pb0; pb < n_pb; pb += step) {
        // the next block's pixels and residual are in flight during the multiply and the epilogue
        load_b(pb + step, nb);
        if constexpr (HZ) igemm_load_z<4, MT, 1>(a, nz, oc_w, (pb + step) * 32, l32, lh);
        v16i acc[MT][1];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const v4i b = *reinterpret_cast<const v4i*>(sBias + oc_w + i * 32 + 8 * q + 4 * lh);
                acc[i][0][4 * q + 0] = b[0]; acc[i][0][4 * q + 1] = b[1]; acc[i][0][4 * q + 2] = b[2]; acc[i][0][4 * q + 3] = b[3];
            }
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i][kc], fb[kc], acc[i][0], 0, 0, 0);
        if constexpr (HZ)
            igemm_run_epilogue<4, MT, 1, true>(a, acc, oc_w, pb * 32, l32, lh, &zr);
        else
            igemm_run_epilogue<4, MT, 1>(a, acc, oc_w, pb * 32, l32, lh);
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) fb[kc] = nb[kc];
        if constexpr (HZ) zr = nz;
    }
}

// The arguments of the kernels with four pixels per lane (groups of them, at stride 1)
template <class Div>
struct QuadArgs {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    uint32_t src_bytes, flt_bytes, z_bytes, dst_bytes;
    int NB, OHW, OC, kbytes, has_bias;
    int src_sn, src_scb, dst_sn, dst_scb, z_sn;
    int groups;  // of four pixels in an image
    Div div_g;
    EpiParams epi;

    auto numbers() const {
        return std::tie(src_bytes, flt_bytes, z_bytes, dst_bytes, NB, OHW, OC, kbytes, has_bias, src_sn, src_scb, dst_sn, dst_scb, z_sn, groups);
    }
};
QuadArgs<FastDiv> quad_args(const IgemmArgs& a) {
    QuadArgs<FastDiv> k;
    k.src = a.src; k.flt = a.flt; k.bias = a.bias; k.z = a.z; k.dst = a.dst;
    k.src_bytes = a.src_bytes; k.flt_bytes = a.flt_bytes; k.z_bytes = a.z_bytes; k.dst_bytes = a.dst_bytes;
    k.NB = a.NB; k.OHW = a.OHW; k.OC = a.OC; k.kbytes = a.kbytes; k.has_bias = a.has_bias;
    k.src_sn = a.src_sn; k.src_scb = a.src_scb; k.dst_sn = a.dst_sn; k.dst_scb = a.dst_scb; k.z_sn = a.z_sn;
    k.groups = (a.OHW + 3) / 4; k.div_g = make_fastdiv(k.groups);
    k.epi = a.epi;
    return k;
}

// What the wire forms of those kernels carry of it (see wire.h)
struct QuadWire {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    uint32_t images, plane, channels, flags;  // channels: out | in << 16
    EpiWire epi;

    template <class Div>
    __host__ __device__ __forceinline__ void numbers(QuadArgs<Div>& k) const {
        k.NB = (int)images; k.OHW = (int)plane; k.OC = wire_lo(channels); k.kbytes = wire_hi(channels);
        k.has_bias = (int)(flags >> 8 & 1);
        k.src_scb = k.dst_scb = wire_mul(k.OHW, 4);
        k.src_sn = wire_mul(k.kbytes, k.OHW); k.dst_sn = wire_mul(k.OC, k.OHW); k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        k.src_bytes = images * (uint32_t)k.src_sn; k.dst_bytes = images * (uint32_t)k.dst_sn; k.z_bytes = images * (uint32_t)k.z_sn;
        k.flt_bytes = (uint32_t)k.OC * (uint32_t)k.kbytes;
        k.groups = (k.OHW + 3) / 4;
    }
    __device__ __forceinline__ QuadArgs<Quot> open() const {
        asm volatile("" ::"s"(src), "s"(flt), "s"(bias), "s"(z), "s"(dst), "s"(images), "s"(plane), "s"(channels), "s"(flags), "s"(epi.f[0]), "s"(epi.f[1]),
                     "s"(epi.f[2]), "s"(epi.f[3]));  // one batch of scalar loads
        QuadArgs<Quot> k;
        k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
        numbers(k);
        k.div_g = quot(k.groups);
        k.epi = epi_open(epi, flags & 255);
        return k;
    }
    // false: the problem has a number that does not fit
    bool pack(const QuadArgs<FastDiv>& k) {
        src = k.src; flt = k.flt; bias = k.bias; z = k.z; dst = k.dst;
        images = (uint32_t)k.NB; plane = (uint32_t)k.OHW; channels = wire2(k.OC, k.kbytes);
        flags = epi_wire(k.epi, false, &epi) | (k.has_bias ? 1u << 8 : 0);
        QuadArgs<FastDiv> o;
        numbers(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return o.numbers() == k.numbers() && (int64_t)k.NB * k.groups < QUOT_MAX;
    }
};

// Stride 1, at most 64 input channels and many tiles: the same with four consecutive pixels per lane.  pw4s_kernel's cost is its memory instructions -- a dword per lane,
// four loads and four stores for every 32 x 32 block, 256 bytes each -- and an NCHW4 plane is contiguous over its pixels.  The
// 32 columns of an MFMA need not be 32 neighbouring pixels: column l of product j is pixel 4 l + j here, so that a lane's operands
// of four products are 16-byte loads, its results 16-byte stores, and a wave's access is a contiguous half kilobyte per channel
// block.  The last group of an image whose plane is no multiple of four holds 1 to 3 pixels: its surplus columns multiply
// whatever follows (the descriptor answers zeros past the tensor) and are not stored.  Bound by the output stream and the
// four vector instructions per output: 16 -> 96 at 112 x 112, batch 64, 18.9 us for 90 MB (4.8 TB/s) against 22.2.
struct Pw4qWide {
    QuadArgs<FastDiv> a;
    PwWalk<FastDiv> w;
    __device__ __forceinline__ const QuadArgs<FastDiv>& open() const {
        // everything up to the first operands in one batch of scalar loads, and a word of each line that the epilogue reads
        asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.dst), "s"(a.src_bytes), "s"(a.flt_bytes), "s"(a.OHW), "s"(a.OC), "s"(a.NB),
                     "s"(a.kbytes), "s"(a.src_sn), "s"(a.src_scb), "s"(a.has_bias), "s"(a.epi.s_b), "s"(a.epi.lin_lo), "s"(w.div_ocg.m),
                     "s"(w.div_ocg.s1), "s"(w.div_ocg.s2), "s"(w.n_ocg), "s"(w.step), "s"(w.slabs), "s"(a.groups), "s"(a.div_g.m),
                     "s"(a.div_g.s1), "s"(a.div_g.s2));
        return a;
    }
    template <int MT>
    __device__ __forceinline__ const PwWalk<FastDiv>& walk(int) const { return w; }
};
struct Pw4qWire : QuadWire {
    uint32_t step;  // and whether it walks slabs, << 31
    template <int MT>
    __device__ __forceinline__ PwWalk<Quot> walk(int oc) const {
        PwWalk<Quot> w;
        w.n_ocg = (oc + MT * 32 - 1) / (MT * 32);
        w.step = (int)(step & 0x7fffffff);
        w.slabs = (int)(step >> 31);
        w.div_ocg = quot(w.n_ocg);
        return w;
    }
};
static_assert(sizeof(Pw4qWire) <= WIRE_BYTES, "a wire");

template <int MT, int KC, bool HZ, class Form>
__device__ __forceinline__ void pw4q_run(const Form& form) {
    __shared__ __attribute__((aligned(16))) int sBias[4][MT * 32];
    const int t = threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const auto a = form.open();
    const auto w = form.template walk<MT>(a.OC);
    const auto div_g = a.div_g;
    const int groups = a.groups, n_pb = (a.NB * groups + 31) / 32;
    int pb0, pb_hi, ocg;
    pw_walk(w, n_pb, wave, &pb0, &pb_hi, &ocg);
    const int oc_w = ocg * MT * 32, step = w.step;
    int* bias_w = sBias[wave];
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes);
    const __amdgpu_buffer_rsrc_t rs_flt = make_rsrc(a.flt, a.flt_bytes);
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z, HZ ? a.z_bytes : 0);
    const __amdgpu_buffer_rsrc_t rs_dst = make_rsrc(a.dst, a.dst_bytes);

    v4i fa[MT][KC];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = oc_w + i * 32 + l32;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
            fa[i][kc] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, row < a.OC ? row * a.kbytes + kc * 32 + lh * 16 : SENT, 0, 0);
    }
    const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias ? a.OC * 4 : 0);
    int bias_v[(MT + 1) / 2];
#pragma unroll
    for (int i = 0; i < MT * 32; i += 64) bias_v[i / 64] = __builtin_amdgcn_raw_buffer_load_b32(rs_bias, (oc_w + i + lane) * 4, 0, 0);
    const int icb = a.kbytes >> 2, total = a.NB * groups;
    // x[kc][i]: four pixels of channel block kc * 8 + lh * 4 + i (zeros past the last one)
    auto load_b = [&](int pb, v4i (&x)[KC][4]) __attribute__((always_inline)) {
        const int m = pb * 32 + l32;
        const bool ok = m < total;  // also false for every block past the last one
        const uint32_t mm = ok ? m : 0, n = fdiv(mm, div_g), g = mm - n * groups;
        const int pix = (int)n * a.src_sn + (int)g * 16 + lh * 4 * a.src_scb;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                x[kc][i] = __builtin_amdgcn_raw_buffer_load_b128(
                        rs_src, ok && kc * 8 + lh * 4 + i < icb ? pix + (kc * 8 + i) * a.src_scb : SENT, 0, 0);
    };
    v4i x[KC][4];
    load_b(pb0 < pb_hi ? pb0 : n_pb, x);
    // The bias of the wave's channels in accumulator order lies in LDS that only this wave reads: no barrier, and no round trip
    // beside that of the operands.
#pragma unroll
    for (int i = 0; i < MT * 32; i += 64)
        if (i + lane < MT * 32) bias_w[i + lane] = bias_v[i / 64];
    lds_between_lanes();
    wait_loads();
    const int tail = a.OHW & 3;
    auto blocks = [&](auto nl) __attribute__((always_inline)) {
        constexpr int NL = decltype(nl)::value;
        for (int pb = pb0; pb < pb_hi; pb += step) {
            v4i fb[KC][4];
#pragma unroll
            for (int kc = 0; kc < KC; ++kc)
#pragma unroll
                for (int j = 0; j < 4; ++j) fb[kc][j] = v4i{x[kc][0][j], x[kc][1][j], x[kc][2][j], x[kc][3][j]};
            load_b(pb + step < pb_hi ? pb + step : n_pb, x);  // in flight during the products and the epilogue of this block
            const int m = pb * 32 + l32;
            const bool ok = m < total;
            const uint32_t mm = ok ? m : 0, n = fdiv(mm, div_g), g = mm - n * groups;
            const bool part = tail != 0 && (int)g == groups - 1;
            const int d0 = (int)n * a.dst_sn + (int)g * 16 + ((oc_w >> 2) + lh) * a.dst_scb;
            const int z0 = (int)n * a.z_sn + (int)g * 16 + ((oc_w >> 2) + lh) * a.dst_scb;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                if (i > 0 && oc_w + i * 32 >= a.OC) break;  // wave-uniform (a wave's first block always holds channels)
                v4i zv[4];
                if constexpr (HZ)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        zv[q] = __builtin_amdgcn_raw_buffer_load_b128(
                                rs_z, ok && oc_w + i * 32 + 8 * q + 4 * lh < a.OC ? z0 + (i * 8 + q * 2) * a.dst_scb : SENT, 0, 0);
                v16i bv;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4i b = *reinterpret_cast<const v4i*>(bias_w + i * 32 + 8 * q + 4 * lh);
                    bv[4 * q + 0] = b[0]; bv[4 * q + 1] = b[1]; bv[4 * q + 2] = b[2]; bv[4 * q + 3] = b[3];
                }
                v4i o[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v16i c = bv;
#pragma unroll
                    for (int kc = 0; kc < KC; ++kc) c = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i][kc], fb[kc][j], c, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        o[q][j] = (int)requant4_fast<NL, HZ>(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3], HZ ? (uint32_t)zv[q][j] : 0u, a.epi);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const bool in = ok && oc_w + i * 32 + 8 * q + 4 * lh < a.OC;
                    const int at = d0 + (i * 8 + q * 2) * a.dst_scb;
                    __builtin_amdgcn_raw_buffer_store_b128(o[q], rs_dst, in && !part ? at : SENT, 0, 0);
                    // (see igemm_epilogue: the data registers of a wide store are read after it issues, and inline
                    // assembly packs the next results)
                    asm volatile("s_nop 1" ::"v"(o[q]) : "memory");
                    if (tail != 0)
#pragma unroll
                        for (int r = 0; r < 3; ++r)
                            if (r < tail) __builtin_amdgcn_raw_buffer_store_b32(o[q][r], rs_dst, in && part ? at + r * 4 : SENT, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);  // one channel block's accumulators and residual at a time
            }
        }
    };
    if (!HZ && a.epi.lin) {
        blocks(std::integral_constant<int, NL_LIN>{});
    } else {
        switch (a.epi.nonline) {
            case NL_RELU: blocks(std::integral_constant<int, NL_RELU>{}); break;
            case NL_H_SWISH: blocks(std::integral_constant<int, NL_H_SWISH>{}); break;
            default: blocks(std::integral_constant<int, NL_IDENTITY>{}); break;
        }
    }
}

// Longer reductions at stride 1: four pixels per lane as above, tiles of 16 MT channels x 64 pixels, and the reduction split
// over the W waves of a workgroup, operands straight into registers (v_mfma_i32_16x16x64_i8: lane l holds filter row l % 16
// and, of pixels 4 (l % 16) .. + 3, the 16 k-bytes at 16 (l / 16)).  What bounds these layers is latency -- a few megabytes and a
// few hundred products per CU -- so a wave asks for all (or four steps) of its operands at once, and the partial sums meet
// in LDS once.
struct Pw4kWide {
    QuadArgs<FastDiv> a;
    FastDiv div_tm;  // by the channel tiles
    __device__ __forceinline__ const QuadArgs<FastDiv>& open() const {
        asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.dst), "s"(a.z), "s"(a.src_bytes), "s"(a.flt_bytes), "s"(a.z_bytes),
                     "s"(a.OHW), "s"(a.OC), "s"(a.NB), "s"(a.kbytes), "s"(a.src_sn), "s"(a.src_scb), "s"(a.dst_scb), "s"(a.z_sn),
                     "s"(a.has_bias), "s"(a.epi.s_b), "s"(a.epi.lin_lo), "s"(a.groups), "s"(a.div_g.m), "s"(a.div_g.s1),
                     "s"(a.div_g.s2), "s"(div_tm.m), "s"(div_tm.s1), "s"(div_tm.s2));
        return a;
    }
    __device__ __forceinline__ const FastDiv& by_tiles(int) const { return div_tm; }
};
struct Pw4kWire : QuadWire {
    __device__ __forceinline__ Quot by_tiles(int tiles_m) const { return quot(tiles_m); }
};
static_assert(sizeof(Pw4kWire) <= WIRE_BYTES, "a wire");

template <int MT, int W, class Form>
__device__ __forceinline__ void pw4k_run(const Form& form) {
    constexpr int AHEAD = MT <= 2 ? 4 : 3;
    extern __shared__ __attribute__((aligned(16))) v4i part[];
    const auto a = form.open();
    const int groups = a.groups, tiles_m = (a.OC + MT * 16 - 1) / (MT * 16), tiles_n = (a.NB * groups + 15) / 16;
    const auto div_g = a.div_g;
    const auto div_tm = form.by_tiles(tiles_m);
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int ls = lane & 15, lk = lane >> 4;
    // workgroup b runs on XCD b % 8: each XCD takes a contiguous run of pixels with all their channels
    const uint32_t at = blockIdx.x >> 3, r0 = fdiv_u(at, div_tm);
    const int tm = (int)(at - r0 * tiles_m), tn = (int)(blockIdx.x & 7) * ((tiles_n + 7) >> 3) + (int)r0;
    if (tn >= tiles_n) return;
    const int oc0 = tm * MT * 16;
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes);
    const __amdgpu_buffer_rsrc_t rs_flt = make_rsrc(a.flt, a.flt_bytes);
    const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias ? a.OC * 4 : 0);
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z, a.z_bytes);
    const __amdgpu_buffer_rsrc_t rs_dst = make_rsrc(a.dst, a.dst_bytes);

    const int m = tn * 16 + ls;
    const bool ok = m < a.NB * groups;
    const uint32_t mm = ok ? m : 0, n = fdiv(mm, div_g), g = mm - n * groups;
    const int pix = (int)n * a.src_sn + (int)g * 16 + lk * 4 * a.src_scb, icb = ok ? a.kbytes >> 2 : 0;
    int row[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) row[i] = oc0 + i * 16 + ls < a.OC ? (oc0 + i * 16 + ls) * a.kbytes + lk * 16 : SENT;

    // this wave's piece of the reduction, in steps of 64 bytes
    const int steps = (a.kbytes + 63) >> 6, per = steps / W, extra = steps % W;  // (W is a power of two)
    int kc = wave * per + (wave < extra ? wave : extra);
    const int k1 = kc + per + (wave < extra ? 1 : 0);
    int left = k1 - kc;
    // operands of the next step; past the wave's piece every lane is out of range: zeros, no memory access.  (No && here: the
    // compiler makes a branch of a wave-uniform one, with the load behind it, and waits for everything at each of them.)
    auto load = [&](v4i (&fa)[MT], v4i (&x)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            fa[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, ((kc < k1) & (row[i] != SENT)) ? row[i] + kc * 64 : SENT, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int cb = kc * 16 + i;
            x[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_src, ((kc < k1) & (cb + lk * 4 < icb)) ? pix + cb * a.src_scb : SENT, 0, 0);
        }
        ++kc;
    };
    v4i acc[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    auto multiply = [&](const v4i (&fa)[MT], const v4i (&x)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const v4i fb = {x[0][j], x[1][j], x[2][j], x[3][j]};
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[i], fb, acc[i][j], 0, 0, 0);
        }
    };
    const int tail = a.OHW & 3;
    // What a thread finishes.  Tiles of at least one block of 16 channels per wave: whole blocks, 4 pixels x 4 channels of each.
    // Tiles of fewer blocks than waves: their dwords are dealt out again, so that no wave adds up and requantises for all -- unit
    // u = wave, + W, ... is the channel quad u % 4 of block u / 4, and a lane takes pixel `lane` of the 64 (64 consecutive
    // dwords of the plane; 960 -> 160 at 7 x 7, one image, with a residual: 3.7 -> 3.3 us).
    constexpr bool DEAL = MT < W;
    constexpr int ITEMS = DEAL ? MT * 4 / W : MT / W;
    const int mf = tn * 16 + (lane >> 2);
    const bool okf = DEAL ? mf < a.NB * groups : ok;
    const uint32_t mmf = okf ? mf : 0, nf = DEAL ? fdiv(mmf, div_g) : n, gf = DEAL ? mmf - nf * groups : g;
    const bool cut = tail != 0 && (int)gf == groups - 1;  // 1 to 3 pixels: the last group of an image
    const bool px_ok = okf && !(DEAL && cut && (lane & 3) >= tail);
    const int z_px = (int)nf * a.z_sn + (int)gf * 16 + (DEAL ? (lane & 3) * 4 : 0), d_px = (int)nf * a.dst_sn + (int)gf * 16 + (DEAL ? (lane & 3) * 4 : 0);
    auto quad_of = [&](int r) __attribute__((always_inline)) { return DEAL ? oc0 + (wave + W * r) * 4 : oc0 + (wave + W * r) * 16 + lk * 4; };
    v4i bz[ITEMS], zv[ITEMS];
    auto bias_z = [&](int r) __attribute__((always_inline)) {
        const int oc4 = quad_of(r), at = px_ok && oc4 < a.OC ? z_px + (oc4 >> 2) * a.dst_scb : SENT;
        if (W > 1) bz[r] = __builtin_amdgcn_raw_buffer_load_b128(rs_bias, oc4 * 4, 0, 0);
        zv[r] = v4i{0, 0, 0, 0};
        if (a.epi.has_z) {
            if (DEAL) zv[r][0] = __builtin_amdgcn_raw_buffer_load_b32(rs_z, at, 0, 0);
            else zv[r] = __builtin_amdgcn_raw_buffer_load_b128(rs_z, at, 0, 0);
        }
    };
    if (W == 1)
#pragma unroll
        for (int i = 0; i < MT; ++i) bz[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_bias, quad_of(i) * 4, 0, 0);
    {
        v4i fa[AHEAD][MT], x[AHEAD][4];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) load(fa[u], x[u]);
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) bias_z(r);
        if (W == 1)  // one wave: the sums start from the bias (asked for before the operands)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = bz[i];
        for (; left > AHEAD; left -= AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                multiply(fa[u], x[u]);
                load(fa[u], x[u]);
                __builtin_amdgcn_sched_barrier(0);  // (or the loads of all steps end up behind the last product)
            }
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (u < left) multiply(fa[u], x[u]);
    }
    if (W > 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            // (the slots of a lane's four pixels are turned by its number: no two lanes of a write meet on a bank)
            for (int j = 0; j < 4; ++j)
                part[DEAL ? (wave * MT + i) * 256 + lane * 4 + (j ^ ((lane >> 1) & 3)) : ((wave * MT + i) * 4 + j) * 64 + lane] = acc[i][j];
        __syncthreads();
    }
    auto finish = [&](auto nl, auto hz) __attribute__((always_inline)) {
        constexpr int NL = decltype(nl)::value;
        constexpr bool HZ = decltype(hz)::value;
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const int oc4 = quad_of(r);
            const bool in = px_ok && oc4 < a.OC;
            const int at = d_px + (oc4 >> 2) * a.dst_scb;
            if (DEAL) {
                const int u = wave + W * r, owner = (u & 3) * 16 + (lane >> 2);
                v4i s = bz[r];
#pragma unroll
                for (int w = 0; w < W; ++w) s += part[(w * MT + (u >> 2)) * 256 + owner * 4 + ((lane & 3) ^ ((owner >> 1) & 3))];
                const uint32_t o = requant4_fast<NL, HZ>(s[0], s[1], s[2], s[3], (uint32_t)zv[r][0], a.epi);
                __builtin_amdgcn_raw_buffer_store_b32(o, rs_dst, in ? at : SENT, 0, 0);
                continue;
            }
            v4i s[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = W == 1 ? acc[r][j] : bz[r];
            if (W > 1)
#pragma unroll
                for (int w = 0; w < W; ++w)
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[j] += part[((w * MT + wave + W * r) * 4 + j) * 64 + lane];
            v4i o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = (int)requant4_fast<NL, HZ>(s[j][0], s[j][1], s[j][2], s[j][3], (uint32_t)zv[r][j], a.epi);
            __builtin_amdgcn_raw_buffer_store_b128(o, rs_dst, in && !cut ? at : SENT, 0, 0);
            asm volatile("s_nop 1" ::"v"(o) : "memory");  // (see igemm_epilogue)
            if (tail != 0)
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if (k < tail) __builtin_amdgcn_raw_buffer_store_b32(o[k], rs_dst, in && cut ? at + k * 4 : SENT, 0, 0);
        }
    };
    using std::integral_constant;
    if (a.epi.lin) {
        finish(integral_constant<int, NL_LIN>{}, integral_constant<bool, false>{});
    } else if (a.epi.has_z) {
        switch (a.epi.nonline) {
            case NL_RELU: finish(integral_constant<int, NL_RELU>{}, integral_constant<bool, true>{}); break;
            case NL_H_SWISH: finish(integral_constant<int, NL_H_SWISH>{}, integral_constant<bool, true>{}); break;
            default: finish(integral_constant<int, NL_IDENTITY>{}, integral_constant<bool, true>{}); break;
        }
    } else {
        switch (a.epi.nonline) {
            case NL_RELU: finish(integral_constant<int, NL_RELU>{}, integral_constant<bool, false>{}); break;
            case NL_H_SWISH: finish(integral_constant<int, NL_H_SWISH>{}, integral_constant<bool, false>{}); break;
            default: finish(integral_constant<int, NL_IDENTITY>{}, integral_constant<bool, false>{}); break;
        }
    }
}

// The same for 32-packed activations (NCHW32 in and out) with at most 128 input channels: the expanding 1x1 layers of a
// bottleneck block and its projection shortcut, whose cost is their output (and residual) stream.  A lane's B fragment
// of k-step kc is one 16-byte load -- half of its pixel's 32-byte block kc; 32 consecutive pixels are one contiguous
// kilobyte -- and the stores are the 16-byte stores of the tiled kernels.
struct Pw32sWide {
    IgemmArgs a;
    PwWalk<FastDiv> w;
    __device__ __forceinline__ const IgemmArgs& open() const {
        asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.dst), "s"(a.z), "s"(a.src_bytes), "s"(a.flt_bytes), "s"(a.z_bytes),
                     "s"(a.OHW), "s"(a.OC), "s"(a.M), "s"(a.OW), "s"(a.IW), "s"(a.sh), "s"(a.sw), "s"(a.kbytes), "s"(a.src_sn), "s"(a.src_scb),
                     "s"(a.dst_scb), "s"(a.z_sn), "s"(a.has_bias), "s"(a.epi.s_b), "s"(a.epi.lin_lo), "s"(w.div_ocg.m));
        asm volatile("" ::"s"(a.div_ohw.m), "s"(a.div_ohw.s1), "s"(a.div_ohw.s2), "s"(a.div_ow.m), "s"(a.div_ow.s1), "s"(a.div_ow.s2),
                     "s"(w.div_ocg.s1), "s"(w.div_ocg.s2), "s"(w.n_ocg), "s"(w.step), "s"(w.slabs));
        return a;
    }
    template <int MT>
    __device__ __forceinline__ const PwWalk<FastDiv>& walk(int) const { return w; }
};
struct Pw32sWire {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    // in: columns | rows << 16, out: columns | rows << 16; channels: out | in << 16; window: strides; m_*: multipliers of the divisions
    uint32_t images, in, out, channels, window, step, m_ohw, m_ow, flags;
    EpiWire epi;

    __host__ __device__ __forceinline__ void numbers(IgemmArgs& k) const {
        k.IW = wire_lo(in); k.OW = wire_lo(out); k.OHW = wire_mul(k.OW, wire_hi(out));
        k.OC = wire_lo(channels); k.kbytes = wire_hi(channels);
        k.sh = wire_lo(window); k.sw = wire_hi(window);
        k.M = wire_mul((int)images, k.OHW);
        k.src_scb = wire_mul(k.IW, wire_hi(in), 32); k.dst_scb = wire_mul(k.OHW, 32);
        k.src_sn = wire_mul(k.kbytes / 32, k.src_scb); k.dst_sn = wire_mul(k.OC, k.OHW); k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        k.src_bytes = images * (uint32_t)k.src_sn; k.dst_bytes = images * (uint32_t)k.dst_sn; k.z_bytes = images * (uint32_t)k.z_sn;
        k.flt_bytes = (uint32_t)k.OC * (uint32_t)k.kbytes;
        k.has_bias = (int)(flags >> 8 & 1);
    }
    static auto compared(const IgemmArgs& k) {
        return std::tie(k.IW, k.OW, k.OHW, k.OC, k.kbytes, k.sh, k.sw, k.M, k.src_scb, k.dst_scb, k.src_sn, k.dst_sn, k.z_sn, k.src_bytes, k.dst_bytes,
                        k.z_bytes, k.flt_bytes, k.has_bias);
    }
    __device__ __forceinline__ IgemmArgs open() const {
        asm volatile("" ::"s"(src), "s"(flt), "s"(bias), "s"(z), "s"(dst), "s"(images), "s"(in), "s"(out), "s"(channels), "s"(window), "s"(step), "s"(m_ohw),
                     "s"(m_ow), "s"(flags), "s"(epi.f[0]), "s"(epi.f[1]), "s"(epi.f[2]), "s"(epi.f[3]));  // one batch of scalar loads
        IgemmArgs k;
        k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
        numbers(k);
        k.div_ohw = fastdiv_open(m_ohw, k.OHW); k.div_ow = fastdiv_open(m_ow, k.OW);
        k.epi = epi_open(epi, flags & 255);
        return k;
    }
    template <int MT>
    __device__ __forceinline__ PwWalk<Quot> walk(int oc) const {
        PwWalk<Quot> w;
        w.n_ocg = (oc + MT * 32 - 1) / (MT * 32);
        w.step = (int)step;
        w.slabs = (int)(flags >> 9 & 1);
        w.div_ocg = quot(w.n_ocg);
        return w;
    }
    // false: the problem has a number that does not fit
    bool pack(const IgemmArgs& k, const PwWalk<FastDiv>& w, int64_t blocks) {
        if (k.OW <= 0 || k.IW <= 0) return false;
        src = k.src; flt = k.flt; bias = k.bias; z = k.z; dst = k.dst;
        images = (uint32_t)k.NB; in = wire2(k.IW, k.IH); out = wire2(k.OW, k.OHW / k.OW); channels = wire2(k.OC, k.kbytes); window = wire2(k.sh, k.sw);
        step = (uint32_t)w.step; m_ohw = k.div_ohw.m; m_ow = k.div_ow.m;
        flags = epi_wire(k.epi, false, &epi) | (k.has_bias ? 1u << 8 : 0) | (w.slabs ? 1u << 9 : 0);
        IgemmArgs o;
        numbers(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return compared(o) == compared(k) && !k.epi.zlin && blocks * 4 < QUOT_MAX;
    }
};
static_assert(sizeof(Pw32sWire) <= WIRE_BYTES, "a wire");

template <int MT, int KC, bool HZ, class Form, class Table>
__device__ __forceinline__ void pw32s_run(const Form& form, const Table& tab) {
    const int t = threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l32 = lane & 31, lh = lane >> 5;

    const auto a = form.open();
    const auto w = form.template walk<MT>(a.OC);
    const int n_pb = (a.M + 31) / 32;
    // Pixel blocks by XCD, as the tiled kernels deal out their tiles: workgroup b runs on XCD b % 8 (round-robin
    // dispatch) and each XCD takes one contiguous eighth of the pixel blocks, so that this layer finds its inputs in the
    // L2 of the XCD that wrote them and leaves its outputs where the next layer's workgroups will look for them.
    // (Grids that are no multiple of 8 n_ocg / 4 workgroups -- small problems -- interleave the blocks instead.)
    int pb0, pb_hi, ocg;
    pw_walk(w, n_pb, wave, &pb0, &pb_hi, &ocg);
    const int oc_w = ocg * MT * 32, step = w.step;
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes);
    const __amdgpu_buffer_rsrc_t rs_flt = make_rsrc(a.flt, a.flt_bytes);
    const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias ? a.OC * 4 : 0);
    // residual table form (the wide one only): the 256 offsets from the kernel's last argument into LDS, once per workgroup (ahead of the first
    // loads: behind them, with the barrier holding every wave until the slowest wave's loads are back, the stack is 3 us
    // slower)
    constexpr bool TABLE = std::is_same<Table, ResidualTable>::value;
    __shared__ float zt[TABLE ? 256 : 1];
    if constexpr (TABLE) {
        if (a.epi.zlin) zt[t] = tab.v[t];
        __syncthreads();
    }

    v4i fa[MT][KC];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = oc_w + i * 32 + l32;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
            fa[i][kc] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, row < a.OC ? row * a.kbytes + kc * 32 + lh * 16 : SENT, 0, 0);
    }
    // the bias of the wave's channels, in accumulator order: the first multiply of every block takes it as its addend
    // (channels past the last one read as zero through the descriptor)
    v16i bv[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const v4i b = __builtin_amdgcn_raw_buffer_load_b128(rs_bias, (oc_w + i * 32 + 8 * q + 4 * lh) * 4, 0, 0);
            bv[i][4 * q + 0] = b[0]; bv[i][4 * q + 1] = b[1]; bv[i][4 * q + 2] = b[2]; bv[i][4 * q + 3] = b[3];
        }

    auto load_b = [&](int pb, v4i (&x)[KC]) __attribute__((always_inline)) {
        const int m = pb * 32 + l32;
        const bool ok = m < a.M;  // also false for every block past the last one
        const uint32_t mm = ok ? m : 0;
        const uint32_t n = fdiv(mm, a.div_ohw), rem = mm - n * a.OHW;
        const uint32_t oh = fdiv(rem, a.div_ow), ow = rem - oh * a.OW;
        const int pix = ok ? (int)n * a.src_sn + ((int)oh * a.sh * a.IW + (int)ow * a.sw) * 32 + lh * 16 : SENT;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) x[kc] = __builtin_amdgcn_raw_buffer_load_b128(rs_src, pix, kc * a.src_scb, 0);
    };

    v4i fb[KC], nb[KC];
    ZRegs<HZ ? MT : 1, 1> zr, nz;
    load_b(pb0 < pb_hi ? pb0 : n_pb, fb);
    if constexpr (HZ) igemm_load_z<32, MT, 1>(a, zr, oc_w, (pb0 < pb_hi ? pb0 : n_pb) * 32, l32, lh);
    wait_loads();
    // one loop per form of the epilogue: a choice inside the loop, and a branch around a wave's first block, which always
    // holds channels, leave the compiler unable to count the stores of a step, and it waits for them at the next one
    auto blocks = [&](auto nl) __attribute__((always_inline)) {
        constexpr int NL = decltype(nl)::value;
        for (int pb = pb0; pb < pb_hi; pb += step) {
            // the next block's pixels and residual are in flight during the multiply and the epilogue (past the end of this
            // XCD's blocks: the block past the last one, whose lanes are all masked)
            const int nx = pb + step < pb_hi ? pb + step : n_pb;
            load_b(nx, nb);
            if constexpr (HZ) igemm_load_z<32, MT, 1>(a, nz, oc_w, nx * 32, l32, lh);
            // the two channel blocks side by side, or where that leaves no registers for a third wave one after the other
            // (128 -> 512 at 28 x 28 with a residual, batch 16: 9.0 us, with two waves per SIMD 9.7)
            constexpr bool TURNS = HZ && MT * KC == 8;
            v16i acc[MT][1][1];
            auto multiply = [&](int i0, int i1) __attribute__((always_inline)) {
#pragma unroll
                for (int i = i0; i < i1; ++i) acc[i][0][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i][0], fb[0], bv[i], 0, 0, 0);
#pragma unroll
                for (int kc = 1; kc < KC; ++kc)
#pragma unroll
                    for (int i = i0; i < i1; ++i) acc[i][0][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i][kc], fb[kc], acc[i][0][0], 0, 0, 0);
            };
            if constexpr (!TURNS) multiply(0, MT);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                if (i > 0 && oc_w + i * 32 >= a.OC) break;  // wave-uniform
                if constexpr (TURNS) multiply(i, i + 1);
                ZRegs<1, 1> z1;
                if constexpr (HZ) z1.v[0][0] = zr.v[i][0];
                igemm_epilogue<32, 1, 1, NL, HZ, HZ>(a, acc[i], &z1, oc_w + i * 32, pb * 32, l32, lh, 0x7fffffff, 1, 0, a.M, zt);
            }
#pragma unroll
            for (int kc = 0; kc < KC; ++kc) fb[kc] = nb[kc];
            if constexpr (HZ) zr = nz;
        }
    };
    using std::integral_constant;
    if (TABLE && a.epi.zlin) {
        if constexpr (TABLE) blocks(integral_constant<int, NL_ZLIN>{});
    } else if (!HZ && a.epi.lin) {
        if constexpr (!HZ) blocks(integral_constant<int, NL_LIN>{});
    } else {
        switch (a.epi.nonline) {
            case NL_RELU: blocks(integral_constant<int, NL_RELU>{}); break;
            case NL_H_SWISH: blocks(integral_constant<int, NL_H_SWISH>{}); break;
            default: blocks(integral_constant<int, NL_IDENTITY>{}); break;
        }
    }
}

template <int MT, int KC, bool HZ>
__global__ __launch_bounds__(256, 3) void pw32s_kernel(Pw32sWide a, std::conditional_t<HZ, ResidualTable, NoResidualTable> tab) {
    pw32s_run<MT, KC, HZ>(a, tab);
}
template <int MT, int KC, bool HZ>
__global__ __launch_bounds__(256, 3) void pw32s_wire_kernel(Pw32sWire a) {
    pw32s_run<MT, KC, HZ>(a, NoResidualTable{});
}
template <int MT, int KC, bool HZ>
__global__ __launch_bounds__(256, 3) void pw4q_kernel(Pw4qWide a) {
    pw4q_run<MT, KC, HZ>(a);
}
template <int MT, int KC, bool HZ>
__global__ __launch_bounds__(256, 3) void pw4q_kernel(Pw4qWire a) {
    pw4q_run<MT, KC, HZ>(a);
}
template <int MT, int W>
__global__ __launch_bounds__(W * 64, 2) void pw4k_kernel(Pw4kWide a) {
    pw4k_run<MT, W>(a);
}
template <int MT, int W>
__global__ __launch_bounds__(W * 64, 2) void pw4k_kernel(Pw4kWire a) {
    pw4k_run<MT, W>(a);
}

template <int MT, int KC>
int launch32_mt(hipStream_t st, const IgemmArgs& a, int cu_count) {
    const int ocb = (a.OC + 31) / 32;
    const int n_ocg = (ocb + MT - 1) / MT;
    const int n_pb = (a.M + 31) / 32;
    if (cu_count <= 0) cu_count = 256;
    int64_t blocks = ((int64_t)n_pb * n_ocg + 3) / 4;
    const int64_t cap = (int64_t)cu_count * 3;  // 12 waves per CU
    if (blocks > cap) blocks = cap;
    blocks = (blocks + n_ocg - 1) / n_ocg * n_ocg;  // waves of one pixel block stay together; 4 * blocks % n_ocg == 0
    // large grids: a multiple of 8 n_ocg workgroups, which the kernel splits into one slab of pixel blocks per XCD
    if (blocks >= 16 * (int64_t)n_ocg) blocks = blocks / (8 * n_ocg) * (8 * n_ocg);
    const dim3 grid((unsigned)blocks);
    const PwWalk<FastDiv> walk = make_walk(blocks, n_ocg);
    Pw32sWire wire;
    if (wire.pack(a, walk, blocks)) {
        return launch_kernel(a.epi.has_z ? pw32s_wire_kernel<MT, KC, true> : pw32s_wire_kernel<MT, KC, false>, grid, dim3(256), 0, st, wire);
    }
    if (a.epi.has_z) {
        ResidualTable tab;
        if (a.epi.zlin) memcpy(tab.v, a.ztab, sizeof(tab.v)); else memset(tab.v, 0, sizeof(tab.v));
        return launch_kernel(pw32s_kernel<MT, KC, true>, grid, dim3(256), 0, st, Pw32sWide{a, walk}, tab);
    }
    return launch_kernel(pw32s_kernel<MT, KC, false>, grid, dim3(256), 0, st, Pw32sWide{a, walk}, NoResidualTable{});
}

template <int MT, int KC>
int launch_quad(hipStream_t st, const IgemmArgs& a, int cu_count) {
    const int ocb = (a.OC + 31) / 32;
    const int n_ocg = (ocb + MT - 1) / MT;
    const int groups = (a.OHW + 3) / 4;
    const int n_pb = (int)(((int64_t)a.NB * groups + 31) / 32);
    if (cu_count <= 0) cu_count = 256;
    int64_t blocks = ((int64_t)n_pb * n_ocg + 3) / 4;
    const int64_t cap = (int64_t)cu_count * 3;  // 12 waves per CU
    if (blocks > cap) blocks = cap;
    blocks = (blocks + n_ocg - 1) / n_ocg * n_ocg;  // waves of one pixel block stay together; 4 * blocks % n_ocg == 0
    // a multiple of the workgroups that deal out whole pixel blocks on every XCD (see the kernel)
    const int unit = 8 * (n_ocg % 4 == 0 ? n_ocg / 4 : n_ocg % 2 == 0 ? n_ocg / 2 : n_ocg);
    if (2 * blocks >= unit) blocks = (blocks + unit - 1) / unit * unit;
    const dim3 grid((unsigned)blocks);
    const PwWalk<FastDiv> walk = make_walk(blocks, n_ocg);
    const QuadArgs<FastDiv> k = quad_args(a);
    Pw4qWire wire;
    if (wire.pack(k) && blocks * 4 < QUOT_MAX) {
        wire.step = (uint32_t)walk.step | (walk.slabs ? 1u << 31 : 0u);
        typedef void (*Kernel)(Pw4qWire);
        return launch_kernel(a.epi.has_z ? (Kernel)pw4q_kernel<MT, KC, true> : (Kernel)pw4q_kernel<MT, KC, false>, grid, dim3(256), 0, st, wire);
    }
    typedef void (*Kernel)(Pw4qWide);
    return launch_kernel(a.epi.has_z ? (Kernel)pw4q_kernel<MT, KC, true> : (Kernel)pw4q_kernel<MT, KC, false>, grid, dim3(256), 0, st, Pw4qWide{k, walk});
}

template <int MT, int W>
int launch_split(hipStream_t st, const IgemmArgs& a) {
    const int tiles_m = (a.OC + MT * 16 - 1) / (MT * 16);
    const int groups = (a.OHW + 3) / 4;
    const int tiles_n = (int)(((int64_t)a.NB * groups + 15) / 16);
    const int64_t grid = (int64_t)((tiles_n + 7) / 8) * 8 * tiles_m;
    if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
    const QuadArgs<FastDiv> k = quad_args(a);
    const int lds = W > 1 ? W * MT * 4096 : 0;
    Pw4kWire wire;
    // (Up to eight workgroups per CU.  Graph replays, wire / wide: to 2047 workgroups 0.99 to 1.005, from 2048 on 1.01 to 1.04.)
    if (grid < 2048 && wire.pack(k)) return launch_kernel((void (*)(Pw4kWire))pw4k_kernel<MT, W>, dim3((unsigned)grid), dim3(W * 64), lds, st, wire);
    return launch_kernel((void (*)(Pw4kWide))pw4k_kernel<MT, W>, dim3((unsigned)grid), dim3(W * 64), lds, st, Pw4kWide{k, make_fastdiv(tiles_m)});
}

template <int MT, int KC>
int launch_mt(hipStream_t st, const IgemmArgs& a, int cu_count) {
    const int ocb = (a.OC + 31) / 32;
    const int n_ocg = (ocb + MT - 1) / MT;
    const int n_pb = (a.M + 31) / 32;
    if (cu_count <= 0) cu_count = 256;
    int64_t blocks = ((int64_t)n_pb * n_ocg + 3) / 4;
    const int64_t cap = (int64_t)cu_count * 4;  // 16 waves per CU
    if (blocks > cap) blocks = cap;
    blocks = (blocks + n_ocg - 1) / n_ocg * n_ocg;  // waves of one pixel block stay together; 4 * blocks % n_ocg == 0
    if (a.epi.has_z)
        return launch_kernel((pw4s_kernel<MT, KC, true>), dim3((unsigned)blocks), dim3(256), 0, st, a, n_ocg, n_pb);
    return launch_kernel((pw4s_kernel<MT, KC, false>), dim3((unsigned)blocks), dim3(256), 0, st, a, n_ocg, n_pb);
}

}  // namespace

// Stride 1, where the planes of src and dst match pixel for pixel: which kernel with four pixels per lane, and its tile.
// Tiles of 16 channels x 64 pixels (T) and steps of 64 input channels decide.  Every variant was timed as graph replays on the
// layers of MobileNetV2 at batch 1 to 64 and on 70 sizes drawn over 16 to 960 channels on both sides, planes of 7 x 7 to
// 112 x 112 and batch 1 to 64, against the kernels that served them before; us, this rule against those:
//   at most 64 channels, streaming: 16 -> 96 at 112 x 112, batch 64: 18.9 / 22.2; 24 -> 144 at 56 x 56: 11.2 / 13.6; batch 16:
//     5.0 / 6.6; 32 -> 192 at 28 x 28, batch 64: 5.9 / 7.2.  (96 channels per wave instead of 32 with very many tiles: less of the
//     input again, 18.9 / 19.4.)
//   one wave per tile while a wave can ask for all its operands at once (up to five steps): 192 -> 32 at 28 x 28, batch 64:
//     4.3 / 5.7; 68 -> 76 at 10 x 70, batch 13: 3.6 / 4.8.
//   longer reductions over the waves of a workgroup: 576 -> 96 at 14 x 14, batch 64: 5.9 / 7.0; 960 -> 160 at 7 x 7: 5.5 / 6.8,
//     batch 16: 4.0 / 5.2, batch 1: 3.7 / 3.7.
// The tiled kernels keep what they are better at (pw4_quad_pick), large products without a residual: 88 -> 448 at 42 x 19,
// batch 30: 9.2 / 8.4; 956 -> 524 at 105 x 25, batch 7: 28.2 / 23.9; 960 -> 320 at 7 x 7, batch 64: 7.1 / 6.7 (with a residual
// they are behind: 156 -> 628 at 43 x 58, batch 23: 27.5 / 34.9).
// They also keep layers that they are not better at.  Timed on 600 more sizes of T = 300 to 15000 and 68 to 960 channels in:
//   without a residual, two to five steps to more than 64 channels from T = 3000 on, and six steps from T = 750 on: up to
//     T = 6000 (69 sizes) the tiled kernels take 14 % longer on average, from 7 % less to 34 % more, at every number of steps;
//     beyond, the two are even (38 sizes: 4 % less).  96 -> 576 at 14 x 14, batch 64: 6.5 / 7.2; 160 -> 960 at 7 x 7: 5.4 / 6.1;
//     384 -> 64 at 14 x 14: 4.3 / 4.7; all of MobileNetV2 at batch 64: 352 / 358.  The lines stand there because the chooser's
//     tests (test_heuristic_picks, tests/test_gpu_parity.py) name the tiled kernel for these three layers.
//   seven and more steps to more than 256 channels between T = 450 and 2000: from 22 % less to 51 % more (47 sizes: 11 % more).
struct QuadPlan {
    int mt;      // 0: none
    int waves;   // 0: the streaming kernel
};
static bool quad_stride(const IgemmArgs& a) { return a.sh == 1 && a.sw == 1; }
static int64_t quad_tiles(const IgemmArgs& a) {
    return (int64_t)((a.OC + 15) / 16) * (((int64_t)a.NB * ((a.OHW + 3) / 4) + 15) / 16);
}
static QuadPlan quad_plan(const IgemmArgs& a) {
    const int64_t T = quad_tiles(a);
    const int steps = (a.kbytes + 63) / 64;
    const auto most = [&](int mt) { return mt > 2 && a.OC <= 32 ? 2 : mt; };  // no rows for channels that are not there
    if (steps == 1 && T > 2000 && a.OC <= PW4_MAX_OC) return {T >= 30000 && a.kbytes <= 32 && a.OC > 64 && a.OC <= 512 ? 3 : 1, 0};
    if (steps <= 5) return {T <= 1300 ? 1 : T <= 3000 ? 2 : most(4), 1};
    if (T <= 250) return {1, 4};
    if (T <= 450) return {2, 4};
    if (T <= 2000) return steps > 6 ? QuadPlan{most(4), 4} : QuadPlan{2, 2};
    return {most(4), 1};
}
// The streaming tile (pw4_stream) runs where a wave holds its channels' whole filter rows or, narrow, at most three steps; the
// split tile (pw4_split) runs every pointwise layer at stride 1.
bool pw4s_usable(const IgemmArgs& a) {
    if (a.T != 1 || a.ph != 0 || a.pw != 0 || a.OC > PW4_MAX_OC) return false;
    return a.kbytes <= 64 || (a.OC <= 32 && a.kbytes <= 192);
}
bool pw4_split_usable(const IgemmArgs& a, int pin, int pout) {
    return pin == 4 && pout == 4 && a.groups == 1 && !a.general && a.T == 1 && a.ph == 0 && a.pw == 0 && quad_stride(a);
}
// whether one of the two takes the layer from the tiled kernels
bool pw4_quad_pick(const IgemmArgs& a, int pin, int pout) {
    if (!pw4_split_usable(a, pin, pout)) return false;
    if (pw4s_usable(a)) return true;
    const int64_t T = quad_tiles(a);
    const int steps = (a.kbytes + 63) / 64;
    if (steps > 6 && T > 450 && T <= 2000 && a.OC > 256) return false;
    if (a.epi.has_z) return T * steps <= 200000;
    if (T * steps > 100000) return false;
    return a.OC <= 64 ? T <= 750 || steps != 6 : T <= (steps == 6 ? 750 : steps > 6 ? 9000 : 3000);
}

// 32-packed: pointwise without padding, dense, the fast epilogue, 32 to 128 input channels, at most 1024 output channels
bool pw32s_usable(const IgemmArgs& a, int pin, int pout) {
    return pin == 32 && pout == 32 && a.T == 1 && a.ph == 0 && a.pw == 0 && a.groups == 1 && !a.general &&
           a.OC <= PW4_MAX_OC && a.kbytes >= 32 && a.kbytes <= 128 && a.kbytes % 32 == 0;
}

int launch_pw32s(hipStream_t st, const IgemmArgs& a, int cu_count) {
    if (a.M == 0 || a.OC == 0) return 0;
    const bool one = (a.OC + 31) / 32 == 1;  // a single channel block: one block per wave
    switch (a.kbytes / 32) {
        case 1: return one ? launch32_mt<1, 1>(st, a, cu_count) : launch32_mt<2, 1>(st, a, cu_count);
        case 2: return one ? launch32_mt<1, 2>(st, a, cu_count) : launch32_mt<2, 2>(st, a, cu_count);
        case 3: return one ? launch32_mt<1, 3>(st, a, cu_count) : launch32_mt<2, 3>(st, a, cu_count);
        default: return one ? launch32_mt<1, 4>(st, a, cu_count) : launch32_mt<2, 4>(st, a, cu_count);
    }
}

int launch_pw4_split(hipStream_t st, const IgemmArgs& a) {
    if (a.M == 0 || a.OC == 0) return 0;
    QuadPlan q = quad_plan(a);
    if (q.waves == 0) q = {4, 1};
    if (q.waves == 1) return q.mt == 1 ? launch_split<1, 1>(st, a) : q.mt == 2 ? launch_split<2, 1>(st, a) : launch_split<4, 1>(st, a);
    if (q.waves == 2) return launch_split<2, 2>(st, a);
    return q.mt == 1 ? launch_split<1, 4>(st, a) : q.mt == 2 ? launch_split<2, 4>(st, a) : launch_split<4, 4>(st, a);
}

int launch_pw4s(hipStream_t st, const IgemmArgs& a, int cu_count) {
    if (a.M == 0 || a.OC == 0) return 0;
    const int ocb = (a.OC + 31) / 32;
    if (quad_stride(a)) {
        const QuadPlan q = quad_plan(a);
        if (q.waves != 0) return launch_pw4_split(st, a);
        if (a.kbytes > 32) return launch_quad<1, 2>(st, a, cu_count);
        return q.mt == 3 ? launch_quad<3, 1>(st, a, cu_count) : launch_quad<1, 1>(st, a, cu_count);
    }
    if (ocb == 1) {  // narrow outputs (the projections): one channel block per wave, up to six k-steps
        switch ((a.kbytes + 31) / 32) {
            case 1: return launch_mt<1, 1>(st, a, cu_count);
            case 2: return launch_mt<1, 2>(st, a, cu_count);
            case 3: return launch_mt<1, 3>(st, a, cu_count);
            case 4: return launch_mt<1, 4>(st, a, cu_count);
            case 5: return launch_mt<1, 5>(st, a, cu_count);
            default: return launch_mt<1, 6>(st, a, cu_count);
        }
    }
    const bool three = ocb % 3 == 0 || ocb > 4;  // 96-channel waves unless the channel count splits evenly into 64s
    if (a.kbytes <= 32) return three ? launch_mt<3, 1>(st, a, cu_count) : launch_mt<2, 1>(st, a, cu_count);
    return three ? launch_mt<3, 2>(st, a, cu_count) : launch_mt<2, 2>(st, a, cu_count);
}

}  // namespace mi355
