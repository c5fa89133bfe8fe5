// Kernel arguments in at most 112 bytes.
//
// What a launch costs the host goes by the bytes of its arguments: on a stream that runs dry up to 112 of them cost 2.6 to 2.8 us, 116
// and more 3.2 to 3.8 (empty kernels, 16 to 512 bytes; hidden arguments such as gridDim count, they lie behind the others).  A call whose
// kernel takes three microseconds is paced by that.  So kernels of such calls do not take the launch code's view of the problem -- strides,
// tile counts, division constants, 200 to 500 bytes -- but a "wire" struct of the numbers those follow from, and open() computes them
// again, in a few scalar instructions that run while nothing else could.
//
// Not everything fits: sides of 65536 and more, gaps between the images of a batch.  The launch code packs a wire, opens it on the
// host and compares; if anything differs, the wide form of the kernel takes the arguments as they are.
#pragma once
#include "common.h"

namespace mi355 {

constexpr size_t WIRE_BYTES = 112;

// Division by d through its reciprocal: floor((x + 1/2) rcp(d)).  v_rcp_f32 is within an ulp and the product is rounded once, so the
// relative error stays below 2^-22; (x + 1/2) / d is at least 1 / (2 d) away from an integer, so the quotient is exact for x < 2^21.
struct Quot {
    float r;
};
constexpr int64_t QUOT_MAX = 1 << 21;
__device__ __forceinline__ Quot quot(uint32_t d) { return {__builtin_amdgcn_rcpf((float)d)}; }
__device__ __forceinline__ uint32_t fdiv(uint32_t x, const Quot& q) { return (uint32_t)(((float)x + 0.5f) * q.r); }
// Of a value that all lanes share, into a scalar register.  (Where the compiler sees that all lanes share the value it drops the builtin,
// keeps the value in a vector register and makes a loop of every load that takes it as a scalar: the empty statement hides it.  The
// instruction itself stays the compiler's, which puts the wait state behind the vector instruction that it reads from.)
__device__ __forceinline__ uint32_t fdiv_u(uint32_t x, const Quot& q) {
    uint32_t v = fdiv(x, q);
    asm("" : "+v"(v));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ uint32_t fdiv_u(uint32_t x, const FastDiv& f) { return fdiv(x, f); }

// The constants of a FastDiv from its multiplier and the divisor
__device__ __forceinline__ FastDiv fastdiv_open(uint32_t m, uint32_t d) {
    FastDiv f;
    f.m = m;
    f.s1 = d > 1;
    f.s2 = d > 1 ? 31 - (uint32_t)__builtin_clz(d - 1) : 0;
    return f;
}

// The requantisation: four floats and eight bits.  Each form reads its own of the floats (literal: the forms with the divide).
constexpr uint32_t EPI_WIRE_BITS = 8;
struct EpiWire {
    float f[4];
};
static inline uint32_t epi_wire(const EpiParams& e, bool literal, EpiWire* w) {
    if (e.lin && !literal) *w = {{e.lin_c, e.lin_d, e.lin_lo, 0.f}};
    else if (e.fast && !literal) *w = {{e.s_b, e.s_z, e.y_hi, e.y_lo}};
    else *w = {{e.s_b, e.s_z, e.s_d, 0.f}};
    return (uint32_t)e.nonline | (e.has_z ? 8u : 0u) | (e.fast && !literal ? 16u : 0u) | (e.lin && !literal ? 32u : 0u);
}
__host__ __device__ __forceinline__ EpiParams epi_open(const EpiWire& w, uint32_t bits) {
    EpiParams e;
    e.s_b = e.lin_c = w.f[0];
    e.s_z = e.lin_d = w.f[1];
    e.s_d = e.y_hi = e.lin_lo = w.f[2];
    e.y_lo = w.f[3];
    e.nonline = (int)(bits & 7);
    e.has_z = (int)(bits >> 3 & 1);
    e.fast = (int)(bits >> 4 & 1);
    e.lin = (int)(bits >> 5 & 1);
    e.zlin = 0;
    return e;
}

// two sixteen-bit numbers, four eight-bit ones
static inline uint32_t wire2(uint32_t lo, uint32_t hi) { return (lo & 0xffff) | hi << 16; }
static inline uint32_t wire4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return (a & 255) | (b & 255) << 8 | (c & 255) << 16 | d << 24; }
__host__ __device__ __forceinline__ int wire_lo(uint32_t w) { return (int)(w & 0xffff); }
__host__ __device__ __forceinline__ int wire_hi(uint32_t w) { return (int)(w >> 16); }
// products that wrap where a number was cut off (another of the numbers tells)
__host__ __device__ __forceinline__ int wire_mul(int a, int b) { return (int)((uint32_t)a * (uint32_t)b); }
__host__ __device__ __forceinline__ int wire_mul(int a, int b, int c) { return wire_mul(wire_mul(a, b), c); }
__host__ __device__ __forceinline__ int wire_byte(uint32_t w, int i) { return (int)(w >> (8 * i) & 255); }

}  // namespace mi355
