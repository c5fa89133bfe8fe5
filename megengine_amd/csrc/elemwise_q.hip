// ElemwiseMultiType quantized modes with one to three inputs (dnn/src/naive/elemwise_multi_type/opr_impl_3.cpp:11-60,
// opr_impl_4.cpp:11-66, opr_impl_5.cpp:11-45): per element, dequantize every input with its own scale, run the mode's
// float kernel (dnn/src/common/elemwise/kern_defs.cuh:166-313), quantize with dst's scale.  Streaming: sixteen elements
// per thread step, 16-byte accesses; 2-13 bytes per element, bound by HBM.
//
// What kept it from that bound was arithmetic: the IEEE divide of the quantization (about twelve instructions per element)
// and a switch over the modes per element.  Now
//   * the mode is chosen once per kernel, around the loop;
//   * where the host can bound the result of the mode and has proved the divide-free quotient for the scale of dst
//     (epilogue.h; the same proof the convolutions use), a multiply and a fused multiply-add replace the divide;
//   * a unary mode from QuantizedS8 to QuantizedS8 is a function of a byte: every workgroup evaluates it -- literally --
//     on the 256 bytes, and the tensor goes through that table in LDS.  256 bytes are the 64 banks once, so any mix of
//     indexes is read without conflict.
// 6.4 M elements: FUSE_MUL_ADD3 10.4 -> 7.2 us, H_SWISH 10.0 -> 4.7 us.
//
// Every operation below is one individually rounded IEEE binary32 operation (the file is compiled without contraction
// and with the correctly rounded divide), in the order the reference's expressions evaluate them, so the bits of the
// result are defined; FUSE_MUL_ADD3 is a multiply followed by an add, as the reference's x86 build without FMA code
// generation computes it.  min and max are the reference's std::min / std::max: max(a, b) = a < b ? b : a.
#include "common.h"

namespace mi355 {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float std_max(float a, float b) { return a < b ? b : a; }
__device__ __forceinline__ float std_min(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float hswish(float x) { return x * std_min(std_max(x + 3.f, 0.f), 6.f) * (1.f / 6.f); }

__device__ __forceinline__ float ew_apply(uint32_t mode, float x, float y, float z) {
    switch (mode) {
        case MI355_EW_RELU: return x <= 0.f ? 0.f : x;
        case MI355_EW_ABS: return __builtin_fabsf(x);
        case MI355_EW_CEIL: return __builtin_ceilf(x);
        case MI355_EW_FLOOR: return __builtin_floorf(x);
        case MI355_EW_NEGATE: return -x;
        case MI355_EW_ROUND: return __builtin_roundf(x);
        case MI355_EW_FAST_TANH: return x * (27.f + x * x) / (27.f + 9.f * x * x);
        case MI355_EW_H_SWISH: return hswish(x);
        case MI355_EW_ABS_GRAD: return x > 0.f ? y : -y;
        case MI355_EW_ADD: return x + y;
        case MI355_EW_FLOOR_DIV: return __builtin_floorf(x / y);
        case MI355_EW_MAX: return x > y ? x : y;
        case MI355_EW_MIN: return x < y ? x : y;
        case MI355_EW_MUL: return x * y;
        case MI355_EW_SIGMOID_GRAD: return x * (1.f - x) * y;
        case MI355_EW_SUB: return x - y;
        case MI355_EW_SWITCH_GT0: return x > 0.f ? y : 0.f;
        case MI355_EW_TANH_GRAD: return (1.f - x * x) * y;
        case MI355_EW_TRUE_DIV: return x / y;
        case MI355_EW_LT: return x < y ? 1.f : 0.f;
        case MI355_EW_LEQ: return x <= y ? 1.f : 0.f;
        case MI355_EW_EQ: return x == y ? 1.f : 0.f;
        case MI355_EW_FUSE_ADD_RELU: return (x + y) <= 0.f ? 0.f : (x + y);
        case MI355_EW_FAST_TANH_GRAD: {
            const float x2 = x * x, deno = 3.f + x2;
            return ((-48.f * x2) / deno + 27.f + x2) / (deno * 9.f) * y;
        }
        case MI355_EW_H_SWISH_GRAD: return x < -3.f ? 0.f : (x > 3.f ? y : (2.f * x + 3.f) / 6.f * y);
        case MI355_EW_FUSE_ADD_H_SWISH: return hswish(x + y);
        case MI355_EW_COND_LEQ_MOV: return x <= y ? z : 0.f;
        case MI355_EW_COND_LT_MOV: return x < y ? z : 0.f;
        case MI355_EW_FUSE_MUL_ADD3: return x * y + z;
        default: return 0.f;
    }
}

// DTypeParamImpl<dt_qint8>::quantize / <dt_qint32>::quantize (dnn/include/megdnn/dtype.h:845-853, :887-896); fmaxf drops
// a NaN, as the reference's fmax does
template <bool DST32>
__device__ __forceinline__ int ew_quantize(float r, float scale) {
    float v = r / scale;
    v = __builtin_roundf(v);
    if (DST32) return (int)fminf(fmaxf(-2147483648.f, v), 2147483520.f);
    return (int)fminf(fmaxf(-128.f, v), 127.f);
}

// the quotient as r (y_hi + y_lo), rounded like epilogue.h's form without RELU
__device__ __forceinline__ int ew_quantize_fast(float r, float y_hi, float y_lo) {
    const float t = r * y_lo;
    float q = __builtin_fmaf(r, y_hi, t);
    q = __builtin_amdgcn_fmed3f(q, -128.f, 127.f);
    return (int)(q + __builtin_copysignf(0.49999997f, q));
}

struct EwArgs {
    const void* src[3];
    void* dst;
    float scale[3];
    float scale_dst, y_hi, y_lo;
    uint64_t blocks16, count;
    uint32_t mode, grid;
};

typedef int v4iu __attribute__((ext_vector_type(4), aligned(4)));  // QuantizedS8 tensors are 4-byte aligned

// four elements from dword `i` of an int8 tensor, or element quad `i` of an int32 tensor
__device__ __forceinline__ void ew_unpack(int w, int (&v)[4]) {
    v[0] = (w << 24) >> 24; v[1] = (w << 16) >> 24; v[2] = (w << 8) >> 24; v[3] = w >> 24;
}

template <bool SRC32>
__device__ __forceinline__ int ew_load1(const void* p, uint64_t j) {
    return SRC32 ? reinterpret_cast<const int32_t*>(p)[j] : (int)reinterpret_cast<const int8_t*>(p)[j];
}

template <int MODE, int ARITY, bool SRC32, bool DST32, bool FAST>
__device__ __forceinline__ int ew_one(const EwArgs& a, int v0, int v1, int v2, uint32_t mode) {
    const float x = (float)v0 * a.scale[0];
    const float y = ARITY > 1 ? (float)v1 * a.scale[1] : 0.f;
    const float z = ARITY > 2 ? (float)v2 * a.scale[2] : 0.f;
    const float r = ew_apply(MODE >= 0 ? (uint32_t)MODE : mode, x, y, z);
    return FAST ? ew_quantize_fast(r, a.y_hi, a.y_lo) : ew_quantize<DST32>(r, a.scale_dst);
}

template <int MODE, int ARITY, bool SRC32, bool DST32, bool FAST>
__device__ __forceinline__ void ew_run(const EwArgs& a) {
    const XcdRun<uint64_t> run = xcd_run<uint64_t>(a.blocks16, a.grid);
    for (uint64_t i = run.at; i < run.end; i += run.step) {
        v4i in[ARITY][SRC32 ? 4 : 1];
#pragma unroll
        for (int s = 0; s < ARITY; ++s)
#pragma unroll
            for (int k = 0; k < (SRC32 ? 4 : 1); ++k)
                in[s][k] = SRC32 ? reinterpret_cast<const v4i*>(a.src[s])[i * 4 + k] : (v4i)reinterpret_cast<const v4iu*>(a.src[s])[i];
        v4i out[DST32 ? 4 : 1];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int v[3][4] = {}, q[4];
#pragma unroll
            for (int s = 0; s < ARITY; ++s) {
                if (SRC32) {
                    v[s][0] = in[s][SRC32 ? k : 0][0]; v[s][1] = in[s][SRC32 ? k : 0][1];
                    v[s][2] = in[s][SRC32 ? k : 0][2]; v[s][3] = in[s][SRC32 ? k : 0][3];
                } else {
                    ew_unpack(in[s][0][k], v[s]);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) q[e] = ew_one<MODE, ARITY, SRC32, DST32, FAST>(a, v[0][e], v[1][e], v[2][e], a.mode);
            if (DST32)
                out[DST32 ? k : 0] = v4i{q[0], q[1], q[2], q[3]};
            else
                out[0][k] = (int)pack4(q[0], q[1], q[2], q[3]);
        }
        if (DST32) {
#pragma unroll
            for (int k = 0; k < 4; ++k) reinterpret_cast<v4i*>(a.dst)[i * 4 + k] = out[DST32 ? k : 0];
        } else {
            reinterpret_cast<v4iu*>(a.dst)[i] = out[0];
        }
    }
    // ragged tail (count % 16 elements): the first lanes of the first workgroup, an element each
    const uint64_t j = a.blocks16 * 16 + threadIdx.x;
    if (blockIdx.x == 0 && j < a.count) {
        const int q = ew_one<MODE, ARITY, SRC32, DST32, FAST>(a, ew_load1<SRC32>(a.src[0], j), ARITY > 1 ? ew_load1<SRC32>(a.src[1], j) : 0,
                                                              ARITY > 2 ? ew_load1<SRC32>(a.src[2], j) : 0, a.mode);
        if (DST32)
            reinterpret_cast<int32_t*>(a.dst)[j] = q;
        else
            reinterpret_cast<int8_t*>(a.dst)[j] = (int8_t)q;
    }
}

template <int ARITY, bool SRC32, bool DST32>
__global__ __launch_bounds__(256) void elemwise_q_kernel(EwArgs a) {
    ew_run<-1, ARITY, SRC32, DST32, false>(a);
}

// the modes whose result the host can bound (ew_bound below), with the divide-free quotient
template <int ARITY, bool SRC32>
__global__ __launch_bounds__(256) void elemwise_q_fast_kernel(EwArgs a) {
#define MI355_EW_CASE(M) case M: ew_run<M, ARITY, SRC32, false, true>(a); break
    if constexpr (ARITY == 1) {
        switch (a.mode) {
            MI355_EW_CASE(MI355_EW_RELU);
            MI355_EW_CASE(MI355_EW_ABS);
            MI355_EW_CASE(MI355_EW_NEGATE);
            MI355_EW_CASE(MI355_EW_H_SWISH);
        }
    } else if constexpr (ARITY == 2) {
        switch (a.mode) {
            MI355_EW_CASE(MI355_EW_ADD);
            MI355_EW_CASE(MI355_EW_SUB);
            MI355_EW_CASE(MI355_EW_MUL);
            MI355_EW_CASE(MI355_EW_MAX);
            MI355_EW_CASE(MI355_EW_MIN);
            MI355_EW_CASE(MI355_EW_SWITCH_GT0);
            MI355_EW_CASE(MI355_EW_FUSE_ADD_RELU);
            MI355_EW_CASE(MI355_EW_FUSE_ADD_H_SWISH);
        }
    } else {
        switch (a.mode) {
            MI355_EW_CASE(MI355_EW_FUSE_MUL_ADD3);
            MI355_EW_CASE(MI355_EW_COND_LEQ_MOV);
            MI355_EW_CASE(MI355_EW_COND_LT_MOV);
        }
    }
#undef MI355_EW_CASE
}

// an upper bound of |mode(x, y, z)| for |x| <= b[0] ..., or 0 for a mode without one here (a division, a gradient)
double ew_bound(uint32_t mode, const double (&b)[3]) {
    const double hs[2] = {b[0], b[0] + b[1]};
    switch (mode) {
        case MI355_EW_RELU: case MI355_EW_ABS: case MI355_EW_NEGATE: return b[0];
        case MI355_EW_H_SWISH: return hs[0] * 6.;
        case MI355_EW_FUSE_ADD_H_SWISH: return hs[1] * 6.;
        case MI355_EW_ADD: case MI355_EW_SUB: case MI355_EW_FUSE_ADD_RELU: return b[0] + b[1];
        case MI355_EW_MUL: return b[0] * b[1];
        case MI355_EW_MAX: case MI355_EW_MIN: return b[0] > b[1] ? b[0] : b[1];
        case MI355_EW_SWITCH_GT0: return b[1];
        case MI355_EW_FUSE_MUL_ADD3: return b[0] * b[1] + b[2];
        case MI355_EW_COND_LEQ_MOV: case MI355_EW_COND_LT_MOV: return b[2];
        default: return 0.;
    }
}

// unary, QuantizedS8 to QuantizedS8
__global__ __launch_bounds__(256) void elemwise_q_table_kernel(EwArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t table[256];  // by the byte as an unsigned value
    const int t = threadIdx.x;
    table[t] = (uint8_t)ew_one<-1, 1, false, false, false>(a, (int)(int8_t)t, 0, 0, a.mode);
    __syncthreads();
    const XcdRun<uint64_t> run = xcd_run<uint64_t>(a.blocks16, a.grid);
    for (uint64_t i = run.at; i < run.end; i += run.step) {
        const v4i x = reinterpret_cast<const v4iu*>(a.src[0])[i];
        v4i o;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t w = (uint32_t)x[k];
            o[k] = (int)pack4(table[w & 255], table[(w >> 8) & 255], table[(w >> 16) & 255], table[w >> 24]);
        }
        reinterpret_cast<v4iu*>(a.dst)[i] = o;
    }
    const uint64_t j = a.blocks16 * 16 + t;
    if (blockIdx.x == 0 && j < a.count) reinterpret_cast<uint8_t*>(a.dst)[j] = table[reinterpret_cast<const uint8_t*>(a.src[0])[j]];
}

template <int ARITY>
int launch_arity(hipStream_t st, const EwArgs& a, bool src32, bool dst32, bool fast, unsigned blocks) {
    if (fast) {
        if (src32) return launch_kernel(elemwise_q_fast_kernel<ARITY, true>, dim3(blocks), dim3(256), 0, st, a);
        return launch_kernel(elemwise_q_fast_kernel<ARITY, false>, dim3(blocks), dim3(256), 0, st, a);
    }
    if (src32 && dst32) return launch_kernel(elemwise_q_kernel<ARITY, true, true>, dim3(blocks), dim3(256), 0, st, a);
    if (src32) return launch_kernel(elemwise_q_kernel<ARITY, true, false>, dim3(blocks), dim3(256), 0, st, a);
    if (dst32) return launch_kernel(elemwise_q_kernel<ARITY, false, true>, dim3(blocks), dim3(256), 0, st, a);
    return launch_kernel(elemwise_q_kernel<ARITY, false, false>, dim3(blocks), dim3(256), 0, st, a);
}

}  // namespace

// number of inputs of a served mode, 0 for a mode that is not served
int elemwise_q_arity(uint32_t mode) {
    switch (mode) {
        case MI355_EW_RELU: case MI355_EW_ABS: case MI355_EW_CEIL: case MI355_EW_FLOOR: case MI355_EW_NEGATE:
        case MI355_EW_ROUND: case MI355_EW_FAST_TANH: case MI355_EW_H_SWISH:
            return 1;
        case MI355_EW_ABS_GRAD: case MI355_EW_ADD: case MI355_EW_FLOOR_DIV: case MI355_EW_MAX: case MI355_EW_MIN:
        case MI355_EW_MUL: case MI355_EW_SIGMOID_GRAD: case MI355_EW_SUB: case MI355_EW_SWITCH_GT0:
        case MI355_EW_TANH_GRAD: case MI355_EW_TRUE_DIV: case MI355_EW_LT: case MI355_EW_LEQ: case MI355_EW_EQ:
        case MI355_EW_FUSE_ADD_RELU: case MI355_EW_FAST_TANH_GRAD: case MI355_EW_H_SWISH_GRAD:
        case MI355_EW_FUSE_ADD_H_SWISH:
            return 2;
        case MI355_EW_COND_LEQ_MOV: case MI355_EW_COND_LT_MOV: case MI355_EW_FUSE_MUL_ADD3:
            return 3;
        default:
            return 0;
    }
}

int launch_elemwise_q(hipStream_t st, const mi355_elemwise_desc& d, const void* s0, const void* s1, const void* s2, void* dst,
                      int cu_count) {
    if (d.count == 0) return 0;
    EwArgs a;
    a.src[0] = s0; a.src[1] = s1; a.src[2] = s2;
    a.dst = dst;
    for (int i = 0; i < 3; ++i) a.scale[i] = d.scale_src[i];
    a.scale_dst = d.scale_dst;
    a.blocks16 = d.count / 16;
    a.count = d.count;
    a.mode = d.mode;
    if (cu_count <= 0) cu_count = 256;
    uint64_t blocks = (a.blocks16 + 255) / 256;
    const uint64_t cap = (uint64_t)cu_count * 16;
    if (blocks > cap) blocks = cap;
    if (blocks == 0) blocks = 1;
    blocks = xcd_grid(blocks);
    a.grid = (uint32_t)blocks;
    const bool src32 = d.src_dtype == MI355_DT_QS32, dst32 = d.dst_dtype == MI355_DT_QS32;
    if (d.arity == 1 && !src32 && !dst32) return launch_kernel(elemwise_q_table_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a);
    // the divide-free quotient: QuantizedS8 dst, a bounded result that stays far from overflow on the way to the clamp, a
    // scale with a proof
    bool fast = false;
    if (!dst32) {
        double b[3];
        bool sane = true;
        for (uint32_t i = 0; i < d.arity; ++i) {
            sane = sane && d.scale_src[i] >= 0x1p-60f && d.scale_src[i] <= 0x1p40f;
            b[i] = (double)d.scale_src[i] * (src32 ? 0x1p31 : 128.);
        }
        for (uint32_t i = d.arity; i < 3; ++i) b[i] = 0.;
        const double bound = ew_bound(d.mode, b);
        fast = sane && bound > 0. && epi_quotient(d.scale_dst, &a.y_hi, &a.y_lo) && bound * (double)a.y_hi < 0x1p100 && bound < 0x1p100;
    }
    switch (d.arity) {
        case 1: return launch_arity<1>(st, a, src32, dst32, fast, (unsigned)blocks);
        case 2: return launch_arity<2>(st, a, src32, dst32, fast, (unsigned)blocks);
        case 3: return launch_arity<3>(st, a, src32, dst32, fast, (unsigned)blocks);
        default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace mi355
