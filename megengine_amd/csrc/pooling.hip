// QuantizedS8 Pooling forward: MAX, AVERAGE (padding counts as zeros) and AVERAGE_COUNT_EXCLUDE_PADDING over
// NCHW, NCHW4 / NCHW44 and NCHW32 tensors, with the arithmetic of the reference's naive operator
// (dnn/src/naive/pooling/opr_impl.cpp:16-36 MaxPooler, :107-127 MeanIncludeRoundedPooler for dt_qint8,
// :237-268 MeanExcludeRoundedPooler, :270-289 the window walk): the mean is roundf(float(sum) / count), one
// correctly rounded float division and a round-half-away.
//
// A pure streaming kernel.  One thread produces one vector of VB output bytes -- 16 channels of an NCHW32
// pixel (two threads per pixel), the 4 channels of an NCHW4 pixel, one NCHW element -- so that a wave's loads
// and stores cover whole, consecutive pixels.  Overlapping windows are re-read through the vector cache; HBM sees
// every input byte about once.  The window is clipped to the image up front, so the inner loops carry no
// bounds tests.  MAX compares four bytes with two packed 16-bit maxima: bytes 1 and 3 of a word are
// compared in place (as the high bytes of the two 16-bit lanes), bytes 0 and 2 after a shift.
#include "common.h"

namespace mi355 {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef short s2 __attribute__((ext_vector_type(2)));

struct PoolArgs {
    const int8_t* src;
    int8_t* dst;
    uint32_t units, grid;  // output vectors, workgroups
    int IH, IW, OH, OW, ph, pw, sh, sw, fh, fw;
    FastDiv div_ow, div_oh;
};

enum { POOL_MAX = 0, POOL_AVG = 1, POOL_AVG_EXCL = 2 };

__device__ __forceinline__ uint32_t pk_max_i16(uint32_t a, uint32_t b) {
    const s2 r = __builtin_elementwise_max(__builtin_bit_cast(s2, a), __builtin_bit_cast(s2, b));
    return __builtin_bit_cast(uint32_t, r);
}

// running maximum of the four signed bytes of a word, kept as 2 + 2 sixteen-bit lanes.  The byte that counts is a lane's high one; the
// low one is whatever came with it and only ever decides between equal high bytes.
struct Max4 {
    uint32_t odd, even;  // bytes 1, 3 | bytes 0, 2
    __device__ __forceinline__ void init() { odd = even = 0x80008000u; }
    __device__ __forceinline__ void feed(uint32_t w) {
        odd = pk_max_i16(odd, w);
        even = pk_max_i16(even, w << 8);
    }
    __device__ __forceinline__ void join(const Max4& m) {
        odd = pk_max_i16(odd, m.odd);
        even = pk_max_i16(even, m.even);
    }
    __device__ __forceinline__ uint32_t get() const { return (odd & 0xff00ff00u) | (even >> 8 & 0x00ff00ffu); }
};

struct Sum4 {
    int s[4];
    __device__ __forceinline__ void init() { s[0] = s[1] = s[2] = s[3] = 0; }
    __device__ __forceinline__ void feed(uint32_t w) {
        const int x = (int)w;
        s[0] += (x << 24) >> 24;
        s[1] += (x << 16) >> 24;
        s[2] += (x << 8) >> 24;
        s[3] += x >> 24;
    }
    __device__ __forceinline__ uint32_t get(float count) const {
        uint32_t r = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int v = (int)roundf((float)s[q] / count);
            r |= ((uint32_t)v & 0xffu) << (8 * q);
        }
        return r;
    }
};

template <int VB>
struct VecIO;
template <>
struct VecIO<1> {
    uint32_t w[1];
    __device__ __forceinline__ void load(const int8_t* p) { w[0] = (uint8_t)*p; }
};
template <>
struct VecIO<4> {
    uint32_t w[1];
    __device__ __forceinline__ void load(const int8_t* p) { w[0] = *reinterpret_cast<const uint32_t*>(p); }
    __device__ __forceinline__ void store(int8_t* p) const { *reinterpret_cast<uint32_t*>(p) = w[0]; }
};
template <>
struct VecIO<16> {
    uint32_t w[4];
    __device__ __forceinline__ void load(const int8_t* p) {
        const v4i x = *reinterpret_cast<const v4i*>(p);
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = (uint32_t)x[q];
    }
    __device__ __forceinline__ void store(int8_t* p) const {
        v4i o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = (int)w[q];
        *reinterpret_cast<v4i*>(p) = o;
    }
};

// Windows of a size known at compile time (2x2, 3x3): every tap is loaded -- from a clamped address when it falls
// outside the image -- so all loads of a thread are in flight together.  With run-time loop bounds they would be
// issued one at a time and the kernel would be bound by memory latency.
template <int PACK, int VB, int MODE, int FH, int FW>
__global__ __launch_bounds__(256) void pooling_static_kernel(PoolArgs a) {
    constexpr int UPP = PACK / VB;
    constexpr int W = VB / 4;
    const XcdRun<uint32_t> run = xcd_run<uint32_t>(a.units, a.grid);
    for (uint32_t u = run.at; u < run.end; u += run.step) {
        const uint32_t sub = UPP == 1 ? 0 : u % UPP, pix = UPP == 1 ? u : u / UPP;
        const uint32_t t = fdiv(pix, a.div_ow), ow = pix - t * a.OW;
        const uint32_t plane = fdiv(t, a.div_oh), oh = t - plane * a.OH;
        const int ih0 = (int)oh * a.sh - a.ph, iw0 = (int)ow * a.sw - a.pw;
        const int8_t* base = a.src + ((size_t)plane * a.IH * a.IW) * PACK + sub * VB;
        VecIO<VB> x[FH][FW];
        // row and column offsets once per window; a coordinate outside the image is clamped into it.  For MAX that is
        // all: the window meets the image, so the clamped tap is another tap of the same window.  The sums replace
        // such a tap by zero
        int roff[FH], coff[FW];
        bool rok[FH], cok[FW];
#pragma unroll
        for (int fh = 0; fh < FH; ++fh) {
            const int ih = ih0 + fh;
            rok[fh] = (unsigned)ih < (unsigned)a.IH;
            roff[fh] = (ih < 0 ? 0 : ih >= a.IH ? a.IH - 1 : ih) * a.IW * PACK;
        }
#pragma unroll
        for (int fw = 0; fw < FW; ++fw) {
            const int iw = iw0 + fw;
            cok[fw] = (unsigned)iw < (unsigned)a.IW;
            coff[fw] = (iw < 0 ? 0 : iw >= a.IW ? a.IW - 1 : iw) * PACK;
        }
        int inside = 0;
#pragma unroll
        for (int fh = 0; fh < FH; ++fh)
#pragma unroll
            for (int fw = 0; fw < FW; ++fw) {
                x[fh][fw].load(base + (uint32_t)(roff[fh] + coff[fw]));
                if (MODE != POOL_MAX) {
                    const bool ok = rok[fh] && cok[fw];
                    inside += ok;
                    if (!ok) {
#pragma unroll
                        for (int q = 0; q < W; ++q) x[fh][fw].w[q] = 0u;
                    }
                }
            }
        VecIO<VB> o;
        if (MODE == POOL_MAX) {
            Max4 acc[W];
#pragma unroll
            for (int q = 0; q < W; ++q) acc[q].init();
#pragma unroll
            for (int fh = 0; fh < FH; ++fh)
#pragma unroll
                for (int fw = 0; fw < FW; ++fw)
#pragma unroll
                    for (int q = 0; q < W; ++q) acc[q].feed(x[fh][fw].w[q]);
#pragma unroll
            for (int q = 0; q < W; ++q) o.w[q] = acc[q].get();
        } else {
            Sum4 acc[W];
#pragma unroll
            for (int q = 0; q < W; ++q) acc[q].init();
#pragma unroll
            for (int fh = 0; fh < FH; ++fh)
#pragma unroll
                for (int fw = 0; fw < FW; ++fw)
#pragma unroll
                    for (int q = 0; q < W; ++q) acc[q].feed(x[fh][fw].w[q]);
            const float count = MODE == POOL_AVG ? (float)(FH * FW) : (float)inside;
#pragma unroll
            for (int q = 0; q < W; ++q) o.w[q] = acc[q].get(count);
        }
        o.store(a.dst + (size_t)u * VB);
    }
}

typedef int v4i_dwords __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t v2u_dwords __attribute__((ext_vector_type(2), aligned(4)));

// MAX over 3 x 3 at stride 2 of an NCHW4 image of four and more columns, with a column of padding: the pool behind the first layer of a
// network.  A thread makes two outputs side by side, of columns 4 j - 1 .. 4 j + 3, from one pixel and one 16-byte load in each of three
// rows, where the kernel above has nine loads of four bytes to an output.  A row or column outside the image gives way to another of the
// same window; at the right edge of a row that is not WHOLE vectors the last one moves back into the row and its columns are moved up.
// 64 channels, batch 64: 112 x 112 18.1 -> 10.9 us (13.0 without WHOLE), 113 x 113 19.3 -> 12.8; 112 x 112 at batch 8 4.2 -> 3.3.
template <bool WHOLE>
__global__ __launch_bounds__(256) void pooling_max3s2_kernel(PoolArgs a) {
    const XcdRun<uint32_t> run = xcd_run<uint32_t>(a.units, a.grid);
    for (uint32_t u = run.at; u < run.end; u += run.step) {
        const uint32_t t = fdiv(u, a.div_ow), pair = u - t * a.div_ow.d;  // (pairs of outputs)
        const uint32_t plane = fdiv(t, a.div_oh), oh = t - plane * a.OH;
        const int ih0 = (int)oh * 2 - a.ph, col = (int)pair * 4;
        const int at = WHOLE || col + 4 <= a.IW ? col : a.IW - 4, up = col - at;
        const int8_t* base = a.src + (size_t)plane * a.IH * a.IW * 4;
        uint32_t left[3];
        v4i x[3];
#pragma unroll
        for (int fh = 0; fh < 3; ++fh) {
            const int ih = ih0 + fh;
            const int row = (ih < 0 ? 0 : ih >= a.IH ? a.IH - 1 : ih) * a.IW;
            x[fh] = *reinterpret_cast<const v4i_dwords*>(base + (uint32_t)(row + at) * 4);
            left[fh] = *reinterpret_cast<const uint32_t*>(base + (uint32_t)(row + (col ? col - 1 : 0)) * 4);
        }
        Max4 first, m[4];  // the left output, and the columns of the vector
        first.init();
#pragma unroll
        for (int q = 0; q < 4; ++q) m[q].init();
        if (WHOLE) {
#pragma unroll
            for (int fh = 0; fh < 3; ++fh) {
                m[1].feed((uint32_t)x[fh][1]);
                first.feed(left[fh]);
                first.feed((uint32_t)x[fh][0]);
            }
            first.join(m[1]);
#pragma unroll
            for (int fh = 0; fh < 3; ++fh) {
                m[1].feed((uint32_t)x[fh][2]);
                m[1].feed((uint32_t)x[fh][3]);
            }
        } else {
#pragma unroll
            for (int fh = 0; fh < 3; ++fh) {
                first.feed(left[fh]);
#pragma unroll
                for (int q = 0; q < 4; ++q) m[q].feed((uint32_t)x[fh][q]);
            }
            if (up) {  // (at most 3: the last pair begins inside the row)
                if (up & 1) { m[0] = m[1]; m[1] = m[2]; m[2] = m[3]; }
                if (up & 2) { m[0] = m[2]; m[1] = m[3]; m[2] = m[3]; }
            }
            first.join(m[0]);
            first.join(m[1]);
            m[1].join(m[2]);
            m[1].join(m[3]);
        }
        int8_t* out = a.dst + ((size_t)t * a.OW + 2 * pair) * 4;
        if (WHOLE || 2 * pair + 1 < (uint32_t)a.OW)
            *reinterpret_cast<v2u_dwords*>(out) = v2u_dwords{first.get(), m[1].get()};
        else
            *reinterpret_cast<uint32_t*>(out) = first.get();
    }
}

// PACK = channel pack of the layout, VB = bytes per thread (PACK = 1: VB = 1; PACK = 4: VB = 4; PACK = 32: VB = 16)
template <int PACK, int VB, int MODE>
__global__ __launch_bounds__(256) void pooling_kernel(PoolArgs a) {
    constexpr int UPP = PACK / VB;  // threads per pixel
    constexpr int W = VB >= 4 ? VB / 4 : 1;
    const XcdRun<uint32_t> run = xcd_run<uint32_t>(a.units, a.grid);
    for (uint32_t u = run.at; u < run.end; u += run.step) {
        const uint32_t sub = UPP == 1 ? 0 : u % UPP, pix = UPP == 1 ? u : u / UPP;
        const uint32_t t = fdiv(pix, a.div_ow), ow = pix - t * a.OW;
        const uint32_t plane = fdiv(t, a.div_oh), oh = t - plane * a.OH;
        const int ih0 = (int)oh * a.sh - a.ph, iw0 = (int)ow * a.sw - a.pw;
        const int h_lo = ih0 < 0 ? -ih0 : 0, h_hi = ih0 + a.fh > a.IH ? a.IH - ih0 : a.fh;
        const int w_lo = iw0 < 0 ? -iw0 : 0, w_hi = iw0 + a.fw > a.IW ? a.IW - iw0 : a.fw;
        const int8_t* base = a.src + ((size_t)plane * a.IH * a.IW) * PACK + sub * VB;
        int8_t* out = a.dst + (size_t)u * VB;
        float count = (float)(a.fh * a.fw);
        if (MODE == POOL_AVG_EXCL) {
            const int nh = h_hi > h_lo ? h_hi - h_lo : 0, nw = w_hi > w_lo ? w_hi - w_lo : 0;
            count = (float)(nh * nw);
        }
        if (VB == 1) {
            int m = -128, s = 0;
            for (int fh = h_lo; fh < h_hi; ++fh)
                for (int fw = w_lo; fw < w_hi; ++fw) {
                    const int x = base[(size_t)(ih0 + fh) * a.IW + (iw0 + fw)];
                    m = x > m ? x : m;
                    s += x;
                }
            out[0] = MODE == POOL_MAX ? (int8_t)m : (int8_t)(int)roundf((float)s / count);
        } else if (MODE == POOL_MAX) {
            Max4 acc[W];
#pragma unroll
            for (int q = 0; q < W; ++q) acc[q].init();
            for (int fh = h_lo; fh < h_hi; ++fh) {
                const int8_t* row = base + ((size_t)(ih0 + fh) * a.IW + iw0) * PACK;
                for (int fw = w_lo; fw < w_hi; ++fw) {
                    if (VB == 16) {
                        const v4i x = *reinterpret_cast<const v4i*>(row + fw * PACK);
#pragma unroll
                        for (int q = 0; q < W; ++q) acc[q].feed((uint32_t)x[q]);
                    } else {
                        acc[0].feed(*reinterpret_cast<const uint32_t*>(row + fw * PACK));
                    }
                }
            }
            if (VB == 16) {
                v4i o;
#pragma unroll
                for (int q = 0; q < W; ++q) o[q] = (int)acc[q].get();
                *reinterpret_cast<v4i*>(out) = o;
            } else {
                *reinterpret_cast<uint32_t*>(out) = acc[0].get();
            }
        } else {
            Sum4 acc[W];
#pragma unroll
            for (int q = 0; q < W; ++q) acc[q].init();
            for (int fh = h_lo; fh < h_hi; ++fh) {
                const int8_t* row = base + ((size_t)(ih0 + fh) * a.IW + iw0) * PACK;
                for (int fw = w_lo; fw < w_hi; ++fw) {
                    if (VB == 16) {
                        const v4i x = *reinterpret_cast<const v4i*>(row + fw * PACK);
#pragma unroll
                        for (int q = 0; q < W; ++q) acc[q].feed((uint32_t)x[q]);
                    } else {
                        acc[0].feed(*reinterpret_cast<const uint32_t*>(row + fw * PACK));
                    }
                }
            }
            if (VB == 16) {
                v4i o;
#pragma unroll
                for (int q = 0; q < W; ++q) o[q] = (int)acc[q].get(count);
                *reinterpret_cast<v4i*>(out) = o;
            } else {
                *reinterpret_cast<uint32_t*>(out) = acc[0].get(count);
            }
        }
    }
}

// Large windows over few outputs (the global mean at the end of a network): one thread per output vector would walk the
// window in a chain of dependent-latency loads while most of the chip idles (7 x 7 over 2048 channels: 20 us at batch 1 as
// at batch 64).  Sixteen lanes share a window, lane k takes taps k, k + 16, ..., and a butterfly adds the partial sums up:
// in each of its first steps a lane hands half of its channels to its partner and keeps the other half, so 16 channels
// cost 15 exchanges and every lane ends with one channel, whose byte it writes.
// 7 x 7 x 2048 in NCHW4: 2.6 us at batch 1, 5.0 us at batch 64.  The next kernel has taken over where it is ahead; what is left here are
// windows of an NCHW4 tensor that are short or many (launch_mode has the lines), and planes of 2 GiB and more in either layout, whose
// offsets that kernel does not hold.
constexpr int POOL_LANES = 16;
template <int PACK, int VB, int MODE>
__global__ __launch_bounds__(256) void pooling_split_kernel(PoolArgs a, FastDiv div_fw) {
    constexpr int UPP = PACK / VB;  // vectors per pixel: neighbouring lanes, then the sixteen shares of the window
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    const uint32_t sub = id % UPP, share = id / UPP % POOL_LANES, pix_raw = id / (UPP * POOL_LANES);
    const uint32_t pixels = a.units / UPP;
    const bool live = pix_raw < pixels;
    const uint32_t pix = live ? pix_raw : pixels - 1;  // every lane takes part in the exchanges
    const uint32_t t = fdiv(pix, a.div_ow), ow = pix - t * a.OW;
    const uint32_t plane = fdiv(t, a.div_oh), oh = t - plane * a.OH;
    const int ih0 = (int)oh * a.sh - a.ph, iw0 = (int)ow * a.sw - a.pw;
    const int8_t* base = a.src + ((size_t)plane * a.IH * a.IW) * PACK + sub * VB;
    int v[VB];
#pragma unroll
    for (int q = 0; q < VB; ++q) v[q] = MODE == POOL_MAX ? -128 : 0;
    const uint32_t taps = (uint32_t)(a.fh * a.fw);
    // four taps at a time, loaded from a clamped address when they lie outside, so that their loads are in flight together
    for (uint32_t k0 = share; k0 < taps; k0 += 4 * POOL_LANES) {
        VecIO<VB> x[4];
        bool ok[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t k = k0 + j * POOL_LANES;
            const uint32_t fh = fdiv(k, div_fw), fw = k - fh * a.fw;
            const int ih = ih0 + (int)fh, iw = iw0 + (int)fw;
            ok[j] = k < taps && (unsigned)ih < (unsigned)a.IH && (unsigned)iw < (unsigned)a.IW;
            x[j].load(base + (ok[j] ? ((size_t)ih * a.IW + iw) * PACK : 0));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < VB; ++q) {
                const int b = (int)(x[j].w[q / 4] << (24 - 8 * (q % 4))) >> 24;
                if (MODE == POOL_MAX)
                    v[q] = ok[j] && b > v[q] ? b : v[q];
                else
                    v[q] += ok[j] ? b : 0;
            }
    }
    // halves while there are channels to hand over, then plain exchanges
    int mine = 0;  // the channel this lane ends with
    int n = VB;
#pragma unroll
    for (int bit = POOL_LANES / 2; bit >= 1; bit /= 2) {
        const int mask = bit * UPP;
        if (n > 1) {
            n /= 2;
            const bool up = (share & bit) != 0;
#pragma unroll
            for (int q = 0; q < VB / 2; ++q) {
                if (q < n) {
                    const int give = up ? v[q] : v[q + n], keep = up ? v[q + n] : v[q];
                    const int got = __shfl_xor(give, mask);
                    v[q] = MODE == POOL_MAX ? (got > keep ? got : keep) : keep + got;
                }
            }
            mine += up ? n : 0;
        } else {
            const int got = __shfl_xor(v[0], mask);
            v[0] = MODE == POOL_MAX ? (got > v[0] ? got : v[0]) : v[0] + got;
        }
    }
    if (!live || (share & (POOL_LANES / VB - 1))) return;  // after plain exchanges several lanes hold one channel
    int r = v[0];
    if (MODE != POOL_MAX) {
        float count = (float)(a.fh * a.fw);
        if (MODE == POOL_AVG_EXCL) {
            const int h_lo = ih0 < 0 ? 0 : ih0, h_hi = ih0 + a.fh > a.IH ? a.IH : ih0 + a.fh;
            const int w_lo = iw0 < 0 ? 0 : iw0, w_hi = iw0 + a.fw > a.IW ? a.IW : iw0 + a.fw;
            count = (float)((h_hi > h_lo ? h_hi - h_lo : 0) * (w_hi > w_lo ? w_hi - w_lo : 0));
        }
        r = (int)roundf((float)r / count);
    }
    a.dst[((size_t)pix * UPP + sub) * VB + mine] = (int8_t)r;
}

// The same with a wave or several to a window.  Four channels to a lane: the 32 channels of an NCHW32 pixel are eight lanes, so a wave
// loads eight taps, 256 bytes, at a time (NCHW4: 64 taps) and eight such loads are in flight.  A lane sums its four channels with one
// byte dot product each (taps outside the window or the image are zeros), and the shares of a wave are added up in registers, 32 lanes
// apart, 16, 8 and so on: in the first two exchanges a lane gives half of its channels for the other half of its partner's, so that it
// ends with one channel to divide and to write.  Short code matters as much as the few exchanges: in a network it comes cold from
// memory.  Several waves meet in LDS.  Against the kernel above:
// NCHW32, 7 x 7 over 2048 channels: batch 1 5.1 -> 2.5 us, batch 64 6.9 -> 3.9; 4 x 4 at 32 x 32 over 256, batch 16: 10.5 -> 5.7; 28 x 28
// over 512, batch 1: 11.4 -> 3.6; 56 x 56 over 256, batch 64: 48.7 -> 12.7.  NCHW4, 56 x 56 over 256, batch 1: 18.8 -> 3.2.
template <int PACK, int MODE, int WAVES>
__global__ __launch_bounds__(WAVES == 1 ? 256 : WAVES * 64) void pooling_wave_kernel(PoolArgs a, FastDiv div_fw) {
    constexpr int UPP = PACK / 4, SHARES = 64 / UPP, STEP = WAVES * 8 * SHARES;
    __shared__ int part[WAVES][WAVES == 1 ? 1 : PACK];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t pix = WAVES == 1 ? blockIdx.x * 4 + wave : blockIdx.x;
    if (pix >= a.units / (PACK == 32 ? 2 : 1)) return;  // (all of a wave; of a workgroup where its waves meet)
    const uint32_t lane = threadIdx.x & 63, sub = lane % UPP, share = lane / UPP;
    const uint32_t t = fdiv(pix, a.div_ow), ow = pix - t * a.OW;
    const uint32_t plane = fdiv(t, a.div_oh), oh = t - plane * a.OH;
    const int ih0 = (int)oh * a.sh - a.ph, iw0 = (int)ow * a.sw - a.pw;
    const int8_t* base = a.src + (size_t)plane * a.IH * a.IW * PACK;
    const uint32_t taps = (uint32_t)(a.fh * a.fw);
    Max4 most;
    most.init();
    int sum[4] = {0, 0, 0, 0};
    for (uint32_t k0 = WAVES == 1 ? 0 : wave * (8 * SHARES); k0 < taps; k0 += STEP) {
        uint32_t x[8];
        bool ok[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t k = k0 + j * SHARES + share;
            const uint32_t fh = fdiv(k, div_fw), fw = k - fh * a.fw;
            const int ih = ih0 + (int)fh, iw = iw0 + (int)fw;
            ok[j] = k < taps && (unsigned)ih < (unsigned)a.IH && (unsigned)iw < (unsigned)a.IW;
            x[j] = *reinterpret_cast<const uint32_t*>(base + ((ok[j] ? (uint32_t)(ih * a.IW + iw) * PACK : 0u) + sub * 4));
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (MODE == POOL_MAX) {
                most.feed(ok[j] ? x[j] : 0x80808080u);
            } else {
                const int w = ok[j] ? (int)x[j] : 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) sum[q] = __builtin_amdgcn_sdot4(w, 1 << (8 * q), sum[q], false);
            }
        }
    }
    int8_t* out = a.dst + (size_t)pix * PACK;
    if (MODE == POOL_MAX) {
        uint32_t m[2] = {most.odd, most.even};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const auto h = __builtin_amdgcn_permlane32_swap(m[q], m[q], false, false);
            m[q] = pk_max_i16(h[0], h[1]);
            const auto r = __builtin_amdgcn_permlane16_swap(m[q], m[q], false, false);
            m[q] = pk_max_i16(r[0], r[1]);
            // rotations of a row of 16 lanes
            m[q] = pk_max_i16(m[q], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m[q], 0x128, 0xf, 0xf, false));
            if (UPP == 1) {
                m[q] = pk_max_i16(m[q], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m[q], 0x124, 0xf, 0xf, false));
                m[q] = pk_max_i16(m[q], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m[q], 0x122, 0xf, 0xf, false));
                m[q] = pk_max_i16(m[q], (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m[q], 0x121, 0xf, 0xf, false));
            }
        }
        if (WAVES > 1) {
            if (share == 0) {
                part[wave][2 * sub] = (int)m[0];
                part[wave][2 * sub + 1] = (int)m[1];
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < WAVES; ++i) {
                m[0] = pk_max_i16(m[0], (uint32_t)part[i][2 * sub]);
                m[1] = pk_max_i16(m[1], (uint32_t)part[i][2 * sub + 1]);
            }
        }
        most.odd = m[0];
        most.even = m[1];
        if ((WAVES == 1 || wave == 0) && share == 0) reinterpret_cast<uint32_t*>(out)[sub] = most.get();
        return;
    }
    const auto h0 = __builtin_amdgcn_permlane32_swap((uint32_t)sum[0], (uint32_t)sum[2], false, false);
    const auto h1 = __builtin_amdgcn_permlane32_swap((uint32_t)sum[1], (uint32_t)sum[3], false, false);
    const auto r = __builtin_amdgcn_permlane16_swap(h0[0] + h0[1], h1[0] + h1[1], false, false);
    int s = (int)(r[0] + r[1]);
    s += __builtin_amdgcn_update_dpp(0, s, 0x128, 0xf, 0xf, false);
    if (UPP == 1) {
        s += __builtin_amdgcn_update_dpp(0, s, 0x124, 0xf, 0xf, false);
        s += __builtin_amdgcn_update_dpp(0, s, 0x122, 0xf, 0xf, false);
        s += __builtin_amdgcn_update_dpp(0, s, 0x121, 0xf, 0xf, false);
    }
    const uint32_t channel = sub * 4 + (lane >> 5) * 2 + (lane >> 4 & 1);
    const bool first = (lane & 15) < UPP;  // one of the lanes that hold a channel
    if (WAVES > 1) {
        if (first) part[wave][channel] = s;
        __syncthreads();
        s = 0;
#pragma unroll
        for (int i = 0; i < WAVES; ++i) s += part[i][channel];
    }
    if (!first || (WAVES > 1 && wave != 0)) return;
    float count = (float)taps;
    if (MODE == POOL_AVG_EXCL) {
        const int h_lo = ih0 < 0 ? 0 : ih0, h_hi = ih0 + a.fh > a.IH ? a.IH : ih0 + a.fh;
        const int w_lo = iw0 < 0 ? 0 : iw0, w_hi = iw0 + a.fw > a.IW ? a.IW : iw0 + a.fw;
        count = (float)((h_hi > h_lo ? h_hi - h_lo : 0) * (w_hi > w_lo ? w_hi - w_lo : 0));
    }
    out[channel] = (int8_t)(int)roundf((float)s / count);
}

template <int PACK, int WAVES>
int launch_wave(hipStream_t st, const PoolArgs& a, int mode, FastDiv dfw) {
    const uint32_t pixels = a.units / (PACK == 32 ? 2 : 1);
    const dim3 grid(WAVES == 1 ? (pixels + 3) / 4 : pixels), block(WAVES == 1 ? 256 : WAVES * 64);
    switch (mode) {
        case POOL_MAX: return launch_kernel((pooling_wave_kernel<PACK, POOL_MAX, WAVES>), grid, block, 0, st, a, dfw);
        case POOL_AVG: return launch_kernel((pooling_wave_kernel<PACK, POOL_AVG, WAVES>), grid, block, 0, st, a, dfw);
        default: return launch_kernel((pooling_wave_kernel<PACK, POOL_AVG_EXCL, WAVES>), grid, block, 0, st, a, dfw);
    }
}

template <int PACK, int VB, int FH, int FW>
int launch_static(hipStream_t st, const PoolArgs& a, int mode, unsigned blocks) {
    switch (mode) {
        case POOL_MAX:
            return launch_kernel((pooling_static_kernel<PACK, VB, POOL_MAX, FH, FW>), dim3(blocks), dim3(256), 0, st, a);
        case POOL_AVG:
            return launch_kernel((pooling_static_kernel<PACK, VB, POOL_AVG, FH, FW>), dim3(blocks), dim3(256), 0, st, a);
        default:
            return launch_kernel((pooling_static_kernel<PACK, VB, POOL_AVG_EXCL, FH, FW>), dim3(blocks), dim3(256), 0, st, a);
    }
}

template <int PACK, int VB>
int launch_mode(hipStream_t st, const PoolArgs& a, int mode, unsigned blocks) {
    if constexpr (VB >= 4) {
        // the static kernels address a plane with 32-bit offsets
        if ((uint64_t)a.IH * (uint64_t)a.IW * PACK >= (1ull << 31)) goto generic;
        if (a.fh == 2 && a.fw == 2) return launch_static<PACK, VB, 2, 2>(st, a, mode, blocks);
        if (a.fh == 3 && a.fw == 3) return launch_static<PACK, VB, 3, 3>(st, a, mode, blocks);
    }
generic:
    // sixteen lanes per window where one thread per output vector leaves the chip less than half full and there are taps
    // for all of them
    if (a.fh * a.fw >= POOL_LANES && a.units < 131072u) {
        const uint32_t threads = a.units * POOL_LANES;
        const dim3 grid((threads + 255) / 256);
        const FastDiv dfw = make_fastdiv((uint32_t)a.fw);
        if constexpr (PACK > 1) {
            const uint32_t taps = (uint32_t)(a.fh * a.fw), pixels = a.units / (PACK == 32 ? 2 : 1);
            if ((uint64_t)a.IH * (uint64_t)a.IW * PACK < (1ull << 31)) {  // (32-bit offsets in a plane)
                // NCHW32: always.  One wave where it has a window's taps in flight at once, or where the windows alone fill the chip and
                // are not long (2048 windows of 81 taps 3.8 us with one wave, 4.1 with four; of 400 9.1 and 8.1)
                if (PACK == 32) {
                    if (taps <= 64 || (pixels > 1024 && taps <= 256)) return launch_wave<PACK, 1>(st, a, mode, dfw);
                    return taps <= 512 ? launch_wave<PACK, 4>(st, a, mode, dfw) : launch_wave<PACK, 16>(st, a, mode, dfw);
                }
                // NCHW4: where sixteen lanes to a window leave the chip idle (512 windows of 81 taps 2.6 us, 2.9 with sixteen lanes; 2048
                // of 784 4.0 and 6.8; but 8192 of 576 10.4 and 6.8, 8192 of 196 5.4 and 4.4)
                if (pixels <= 1024 ? taps > 64 : pixels <= 4096 && taps > 512) {
                    if (taps <= 512) return launch_wave<PACK, 1>(st, a, mode, dfw);
                    return taps <= 4096 ? launch_wave<PACK, 4>(st, a, mode, dfw) : launch_wave<PACK, 16>(st, a, mode, dfw);
                }
            }
        }
        switch (mode) {
            case POOL_MAX: return launch_kernel(pooling_split_kernel<PACK, VB, POOL_MAX>, grid, dim3(256), 0, st, a, dfw);
            case POOL_AVG: return launch_kernel(pooling_split_kernel<PACK, VB, POOL_AVG>, grid, dim3(256), 0, st, a, dfw);
            default: return launch_kernel(pooling_split_kernel<PACK, VB, POOL_AVG_EXCL>, grid, dim3(256), 0, st, a, dfw);
        }
    }
    switch (mode) {
        case POOL_MAX:
            return launch_kernel((pooling_kernel<PACK, VB, POOL_MAX>), dim3(blocks), dim3(256), 0, st, a);
        case POOL_AVG:
            return launch_kernel((pooling_kernel<PACK, VB, POOL_AVG>), dim3(blocks), dim3(256), 0, st, a);
        default:
            return launch_kernel((pooling_kernel<PACK, VB, POOL_AVG_EXCL>), dim3(blocks), dim3(256), 0, st, a);
    }
}

}  // namespace

// pack: 1, 4 or 32; the caller has checked the descriptor (every window meets the image where the mode needs it,
// fewer than 2^31 output vectors)
int launch_pooling(hipStream_t st, const mi355_pooling_desc& d, int pack, uint32_t oh, uint32_t ow, const int8_t* src,
                   int8_t* dst, int cu_count) {
    PoolArgs a;
    a.src = src;
    a.dst = dst;
    a.IH = (int)d.ih; a.IW = (int)d.iw; a.OH = (int)oh; a.OW = (int)ow;
    a.ph = (int)d.pad_h; a.pw = (int)d.pad_w; a.sh = (int)d.stride_h; a.sw = (int)d.stride_w;
    a.fh = (int)d.window_h; a.fw = (int)d.window_w;
    a.div_ow = make_fastdiv(ow);
    a.div_oh = make_fastdiv(oh);
    const uint64_t pixels = (uint64_t)d.n * (d.c / (uint32_t)pack) * oh * ow;
    const uint64_t units = pack == 32 ? pixels * 2 : pixels;
    if (units == 0) return 0;
    a.units = (uint32_t)units;
    if (cu_count <= 0) cu_count = 256;
    const bool max3s2 = pack == 4 && d.mode == MI355_POOL_MAX && a.fh == 3 && a.fw == 3 && a.sh == 2 && a.sw == 2 && a.pw == 1 &&
                        a.IW >= 4 && (uint64_t)d.ih * d.iw * 4 < (1ull << 31);  // (32-bit offsets in a plane)
    if (max3s2) {
        a.units = (uint32_t)(units / ow * ((ow + 1) / 2));
        a.div_ow = make_fastdiv((ow + 1) / 2);
    }
    uint64_t blocks = (a.units + 255ull) / 256;
    const uint64_t cap = (uint64_t)cu_count * 64;
    if (blocks > cap) blocks = cap;
    blocks = xcd_grid(blocks);
    a.grid = (uint32_t)blocks;
    if (max3s2 && a.IW % 4 == 0) return launch_kernel(pooling_max3s2_kernel<true>, dim3(a.grid), dim3(256), 0, st, a);
    if (max3s2) return launch_kernel(pooling_max3s2_kernel<false>, dim3(a.grid), dim3(256), 0, st, a);
    if (pack == 32) return launch_mode<32, 16>(st, a, (int)d.mode, (unsigned)blocks);
    if (pack == 4) return launch_mode<4, 4>(st, a, (int)d.mode, (unsigned)blocks);
    return launch_mode<1, 1>(st, a, (int)d.mode, (unsigned)blocks);
}

}  // namespace mi355
