// Plain-NCHW int8 ConvBias on the MFMA kernels: algorithm MI355_NCHW_RELAYOUT_MFMA_I8.
//
// Format::NCHW is what the reference's own x86 int8 algorithms accept (dnn/src/x86/conv_bias/int8/
// algo_usable_preferred.cpp:19-37,88-108; shape rule dnn/src/common/convolution.cpp:774-801), and the CUDA backend runs
// it by way of the packed format of its tensor-core kernels (dnn/src/cuda/conv_bias/conv_nchwqs8.cpp).  Here two launches
// do: one brings src and filter into the packed layout, in the caller's workspace -- the first algorithm of this backend
// that reports a non-zero get_workspace_in_bytes (dnn/include/megdnn/oprs/nn.h:419-422) --
//
//     [src packed by 4 or 32 channels][filter as (OC, IC/4, FH, FW, 4), or pre-processed: (IC/32, FH, FW, OC, 32)]
//
// (that order costs the conversion nothing, and the kernels read it in contiguous kilobytes: 419 drawn layers 0.946 of the time of the
// reference order, 0.84 .. 0.88 on the tiles that split long reductions), and the implicit GEMM reads those, and bias, residual and destination as they are: its planar epilogue knows NCHW.
// Padded input channels are zero bytes (they add nothing to a sum).  The arithmetic is that of the packed kernels, which
// is bit-exact to the reference's naive path; a permutation of the operands changes no integer sum.
// Most sizes with filters of 1x1, 3x3 and 5x5 need neither the packing nor the workspace: conv_patch1.hip reads the planes
// themselves, and patch1_pick says where it is ahead.
#include <string.h>

#include "igemm_shared.h"
#include "relayout_parts.h"

namespace mi355 {
namespace {

constexpr size_t kAlign = 256;
size_t up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }

struct NchwLayout {
    int pack;                       // channel pack of the inner problem
    size_t off_flt, used;           // (src stands at the front)
    size_t reported;                // what query answers
    ConvProblem inner;              // packed src and filter, planar bias, z and dst
};

bool make_layout(const ConvProblem& p, NchwLayout* L) {
    const mi355_conv_desc& d = p.d;
    if (d.format != MI355_FMT_NCHW || p.dw4) return false;
    if (d.dst_dtype != MI355_DT_QS8 || d.bias_mode == MI355_BIAS_FULL || !p.epi.fast) return false;
    if (d.mode != MI355_MODE_CROSS_CORRELATION || d.dilate_h != 1 || d.dilate_w != 1) return false;
    // groups must be whole channel blocks on both sides: then the packed tensors of the groups are contiguous pieces of
    // the packed tensors, as the 32-packed group kernel expects them
    if (d.group != 1 && (p.icpg % 32 || p.ocpg % 32)) return false;
    // dense batches only (a strided view would need strided conversions)
    const int64_t src_img = (int64_t)d.ic * d.ih * d.iw, dst_img = (int64_t)d.oc * p.oh * p.ow;
    if (p.src_sn != src_img || p.dst_sn != dst_img || (d.has_z && p.z_sn != dst_img)) return false;
    if (d.n > 65535) return false;
    // The size that query reports, and that exec asks of a caller who names this algorithm, is part of the interface and fixed
    // by its tests: src, filter, dst, z and bias all packed by 32, the tensors this algorithm once kept.  The first two, `used`,
    // are what it writes, and what an exec that chooses for itself goes by.
    const uint32_t ic32 = (d.ic + 31) / 32 * 32, oc32 = (d.oc + 31) / 32 * 32;
    const size_t src32 = (size_t)d.n * ic32 * d.ih * d.iw, dst32 = (size_t)d.n * oc32 * p.oh * p.ow;
    L->reported = up(src32) + up((size_t)oc32 * (ic32 / d.group) * d.fh * d.fw) + up(dst32) + (d.has_z ? up(dst32) : 0) +
               (d.bias_mode == MI355_BIAS_BROADCAST_CHANNEL && oc32 != d.oc ? up((size_t)oc32 * 4) : 0);
    // up to 16 channels a block of 32 would be half and more padding
    L->pack = d.ic <= 16 ? 4 : 32;
    const uint32_t icp = (d.ic + L->pack - 1) / L->pack * L->pack;
    if ((uint64_t)d.n * icp * d.ih * d.iw >= (1ull << 31) || (uint64_t)d.oc * (icp / d.group) * d.fh * d.fw >= (1ull << 31)) return false;
    L->off_flt = up((size_t)d.n * icp * d.ih * d.iw);
    L->used = L->off_flt + up((size_t)d.oc * (icp / d.group) * d.fh * d.fw);
    ConvProblem& q = L->inner;
    q = p;
    q.d.format = L->pack == 4 ? FMT_INNER_NCHW4_NCHW : FMT_INNER_NCHW32_NCHW;
    q.d.ic = icp;
    q.d.src_stride_n = q.d.dst_stride_n = q.d.z_stride_n = 0;
    q.icpg = icp / d.group;
    q.pin = L->pack;
    q.pout = 1;
    q.dw4 = false;
    q.src_sn = (int64_t)icp * d.ih * d.iw;
    return igemm_usable(q);
}

// src and filter into their packed layouts, one launch: the first blocks convert src -- 32 channels x 128 pixels through
// LDS, or quads of a pixel where the planes are smaller than that -- the others the filter, an NCHW tensor of oc images.
constexpr int NP_TP = 128, NP_ROW = NP_TP + 4;  // pixels per tile; padded LDS row (33 dwords: channel rows on other banks)
struct PrepArgs {
    const int8_t* src;
    int8_t* src_p;
    const int8_t* flt;
    int8_t* flt_p;
    uint32_t C, CB, HW, ptiles;    // tiled src
    uint32_t src_blocks, tiled, flt_rows;
    FastDiv div_ptiles, div_cb;
    SmallPlanes src_small, flt_small;
};

__global__ __launch_bounds__(256) void nchw_prep_kernel(PrepArgs a) {
    __shared__ __attribute__((aligned(16))) int8_t sm[32 * NP_ROW];
    const uint32_t t = threadIdx.x;
    if (blockIdx.x >= a.src_blocks)
        return small_planes_quad(a.flt, reinterpret_cast<uint32_t*>(a.flt_p), a.flt_small, (blockIdx.x - a.src_blocks) * 256 + t, a.flt_rows);
    if (!a.tiled) return small_planes_quad(a.src, reinterpret_cast<uint32_t*>(a.src_p), a.src_small, blockIdx.x * 256 + t);
    const uint32_t b = fdiv(blockIdx.x, a.div_ptiles), p0 = (blockIdx.x - b * a.ptiles) * NP_TP;  // b = image * CB + block
    const uint32_t n = fdiv(b, a.div_cb), cb = b - n * a.CB;
    {
        const uint32_t row = t >> 3, v = t & 7, px = p0 + v * 16, c = cb * 32 + row;
        u32x4 x = {0, 0, 0, 0};
        if (px < a.HW && c < a.C) x = load16_tail(a.src + ((int64_t)n * a.C + c) * a.HW + px, a.HW - px);
        uint32_t* d = reinterpret_cast<uint32_t*>(sm + row * NP_ROW + v * 16);
#pragma unroll
        for (int k = 0; k < 4; ++k) d[k] = x[k];
    }
    __syncthreads();
    // 4 channels x 4 pixels per thread; eight neighbouring lanes are the 32 channels of a pixel
    const uint32_t cq = t & 7, pq = t >> 3;
    uint32_t r[4], o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = *reinterpret_cast<const uint32_t*>(sm + (cq * 4 + k) * NP_ROW + pq * 4);
    transpose4x4(r[0], r[1], r[2], r[3], o[0], o[1], o[2], o[3]);
    uint32_t* d = reinterpret_cast<uint32_t*>(a.src_p) + ((int64_t)b * a.HW + p0 + pq * 4) * 8 + cq;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (p0 + pq * 4 + k < a.HW) d[k * 8] = o[k];
}

}  // namespace

bool nchw_mfma_usable(const ConvProblem& p) {
    NchwLayout L;
    return make_layout(p, &L);
}

size_t nchw_mfma_workspace(const ConvProblem& p) {
    NchwLayout L;
    return make_layout(p, &L) ? L.reported : 0;
}

size_t nchw_mfma_workspace_used(const ConvProblem& p) {
    NchwLayout L;
    return make_layout(p, &L) ? L.used : 0;
}

int launch_conv_nchw_mfma(hipStream_t st, const ConvProblem& p, int cu_count, const int8_t* src, const int8_t* flt,
                          const int32_t* bias, const int8_t* z, int8_t* dst, void* workspace) {
    NchwLayout L;
    if (!make_layout(p, &L)) return (int)hipErrorInvalidValue;
    const mi355_conv_desc& d = p.d;
    if ((uint64_t)d.n * d.oc * p.oh * p.ow == 0) return 0;
    const int tile = patch1_pick(p, true, cu_count);  // no packing where the kernel that reads the planes is ahead
    if (tile >= 0) return launch_patch1(st, p, tile, cu_count, src, flt, bias, z, dst);
    int8_t* ws = reinterpret_cast<int8_t*>(workspace);
    const uint32_t HW = d.ih * d.iw;
    PrepArgs a;
    a.src = src; a.src_p = ws; a.flt = flt; a.flt_p = ws + L.off_flt;
    a.C = d.ic; a.CB = (d.ic + 31) / 32; a.HW = HW;
    a.ptiles = (HW + NP_TP - 1) / NP_TP;
    a.div_ptiles = make_fastdiv(a.ptiles);
    a.div_cb = make_fastdiv(a.CB);
    a.tiled = L.pack == 32 && HW >= NP_TP / 2;
    a.src_small = make_small_planes(d.n, d.ic, HW, L.pack);
    a.flt_small = make_small_planes(d.oc, p.icpg, d.fh * d.fw, L.pack);
    a.flt_rows = L.pack == 32 ? d.oc : 0;
    a.src_blocks = a.tiled ? d.n * a.CB * a.ptiles : (a.src_small.items + 255) / 256;
    const uint32_t blocks = a.src_blocks + (a.flt_small.items + 255) / 256;
    const int rc = launch_kernel(nchw_prep_kernel, dim3(blocks), dim3(256), 0, st, a);
    if (rc) return rc;
    const bool pre = L.pack == 32;
    return launch_conv_igemm(st, L.inner, igemm_pick_cfg(L.inner, cu_count, pre), cu_count, a.src_p, a.flt_p, bias, z, dst, pre, a.flt_rows);
}

}  // namespace mi355
