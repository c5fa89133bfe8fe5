// Pieces of the byte-transposing layout conversions, shared by RelayoutFormat (relayout.hip) and by the preparation pass of
// plain-NCHW convolutions (conv_nchw.hip).
#pragma once
#include "common.h"

namespace mi355 {
namespace {

// ---- 4x4 byte transpose in registers: rows r0..r3 (4 bytes each) -> columns ----
__device__ __forceinline__ void transpose4x4(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3, uint32_t& c0,
                                             uint32_t& c1, uint32_t& c2, uint32_t& c3) {
    // t01_lo = r0.b0 r1.b0 r0.b1 r1.b1 ; t01_hi = r0.b2 r1.b2 r0.b3 r1.b3
    uint32_t t01_lo = __builtin_amdgcn_perm(r1, r0, 0x05010400u);
    uint32_t t01_hi = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
    uint32_t t23_lo = __builtin_amdgcn_perm(r3, r2, 0x05010400u);
    uint32_t t23_hi = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
    c0 = __builtin_amdgcn_perm(t23_lo, t01_lo, 0x05040100u);
    c1 = __builtin_amdgcn_perm(t23_lo, t01_lo, 0x07060302u);
    c2 = __builtin_amdgcn_perm(t23_hi, t01_hi, 0x05040100u);
    c3 = __builtin_amdgcn_perm(t23_hi, t01_hi, 0x07060302u);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(1)));  // 16 bytes at any address
typedef uint32_t u32u __attribute__((aligned(1)));

__device__ __forceinline__ u32x4 load16u(const int8_t* p) { return *reinterpret_cast<const u32x4u*>(p); }
__device__ __forceinline__ void store16u(int8_t* p, u32x4 v) { *reinterpret_cast<u32x4u*>(p) = v; }
__device__ __forceinline__ uint32_t load4u(const int8_t* p) { return *reinterpret_cast<const u32u*>(p); }
__device__ __forceinline__ void store4u(int8_t* p, uint32_t v) { *reinterpret_cast<u32u*>(p) = v; }

// `have` (>= 1) bytes from p, the rest zero; the sixteen bytes before p + have exist.  (One load that ends where they do, turned to the front: byte by
// byte the end of a plane was fifteen loads more for every wave that held one: into
// NCHW32 416 x 49 x 78 at batch 29 33.0 -> 18.4 us, 300 drawn conversions 0.84 of the time, back 0.93.)
__device__ __forceinline__ u32x4 load16_tail(const int8_t* p, uint32_t have) {
    if (have >= 16) return load16u(p);
    const uint32_t skip = 16 - have;
    const u32x4 x = load16u(p - skip);
    uint32_t y[5];  // by whole dwords, then by bytes
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        y[i] = x[i];
#pragma unroll
        for (uint32_t d = 1; d < 4; ++d) y[i] = skip >> 2 == d ? (i + d < 4 ? x[(i + d) & 3] : 0u) : y[i];
    }
    y[4] = 0;
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_alignbyte(y[i + 1], y[i], skip & 3);
    return r;
}
// the first `have` bytes: sixteen, or eight, four, two and one
__device__ __forceinline__ void store16_tail(int8_t* p, u32x4 v, uint32_t have) {
    typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(1)));
    typedef uint16_t u16u __attribute__((aligned(1)));
    if (have >= 16) return store16u(p, v);
    uint32_t a = v[0], b = v[1], at = 0;
    if (have & 8) {
        *reinterpret_cast<u32x2u*>(p) = u32x2u{a, b};
        a = v[2];
        b = v[3];
        at = 8;
    }
    if (have & 4) {
        store4u(p + at, a);
        a = b;
        at += 4;
    }
    if (have & 2) {
        *reinterpret_cast<u16u*>(p + at) = (uint16_t)a;
        a >>= 16;
        at += 2;
    }
    if (have & 1) p[at] = (int8_t)a;
}

// NCHW -> NCHW4 / NCHW32 for small planes (filters, 7 x 7 images): one thread per 4 output channels of a pixel, channels
// past the last one are zero.
struct SmallPlanes {
    uint32_t C, CB, HW, log_quads, items;
    FastDiv hw, cb;
};
static inline SmallPlanes make_small_planes(uint32_t n, uint32_t c, uint32_t hw, uint32_t pack) {
    SmallPlanes g;
    g.C = c;
    g.CB = (c + pack - 1) / pack;
    g.HW = hw;
    g.log_quads = pack == 32 ? 3 : 0;
    g.items = n * g.CB * hw * (pack / 4);
    g.hw = make_fastdiv(hw);
    g.cb = make_fastdiv(g.CB);
    return g;
}
// `images` (not zero): not image by image, but [channel block][pixel][image][pack channels], the order of a pre-processed filter
__device__ __forceinline__ void small_planes_quad(const int8_t* __restrict__ src, uint32_t* __restrict__ dst, const SmallPlanes& g,
                                                  uint32_t it, uint32_t images = 0) {
    if (it >= g.items) return;
    const uint32_t k = it & ((1u << g.log_quads) - 1), t = it >> g.log_quads;
    const uint32_t b = fdiv(t, g.hw), px = t - b * g.HW;
    const uint32_t n = fdiv(b, g.cb), c0 = ((b - n * g.CB) << (g.log_quads + 2)) + k * 4;
    const int8_t* s = src + ((int64_t)n * g.C + c0) * g.HW + px;
    uint32_t w = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q)
        if (c0 + q < g.C) w |= (uint32_t)(uint8_t)s[(int64_t)q * g.HW] << (8 * q);
    dst[images ? (((((b - n * g.CB) * g.HW + px) * images + n) << g.log_quads) + k) : it] = w;
}

}  // namespace
}  // namespace mi355
