// Which launches an exec of the heuristic's choice makes (no GPU: the runtime's calls that would need one are answered here, and
// a launch is only noted).  One layer per line of the input: format (0 NCHW, else as in the interface), n, ic, ih, iw, oc, filter,
// stride, group, residual; one line of the output for each: the number of launches, and dynamic LDS and threads of the last one.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>

#include "../../include/mi355_convbias.h"

static int g_launches;
static unsigned g_lds, g_threads;
extern "C" {
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3 block, void**, size_t lds, hipStream_t) {
    ++g_launches;
    g_lds = (unsigned)lds;
    g_threads = block.x;
    return hipSuccess;
}
}

int main() {
    unsigned fmt, n, ic, ih, iw, oc, f, stride, group, z;
    while (scanf("%u %u %u %u %u %u %u %u %u %u", &fmt, &n, &ic, &ih, &iw, &oc, &f, &stride, &group, &z) == 10) {
        mi355_conv_desc d;
        memset(&d, 0, sizeof(d));
        d.format = fmt;
        d.sparse = group > 1 ? MI355_SPARSE_GROUP : MI355_SPARSE_DENSE;
        d.n = n; d.ic = ic; d.oc = oc; d.ih = ih; d.iw = iw; d.group = group;
        d.fh = d.fw = f;
        d.pad_h = d.pad_w = f / 2;
        d.stride_h = d.stride_w = stride;
        d.dilate_h = d.dilate_w = 1;
        d.bias_mode = MI355_BIAS_BROADCAST_CHANNEL;
        d.nonline = MI355_NL_RELU;
        d.has_z = z;
        d.dst_dtype = MI355_DT_QS8;
        d.scale_bias = 2e-4f;
        d.scale_z = d.scale_dst = 0.05f;
        mi355_algo a;
        size_t ws = 0;
        int8_t* const t = reinterpret_cast<int8_t*>(0x1000000);  // device addresses that nothing on the host reads
        g_launches = 0;
        int st = mi355_convbias_s8_query(&d, MI355_ALGO_HEURISTIC, &a, &ws);
        if (!st) st = mi355_convbias_s8_exec(nullptr, &d, &a, t, t, reinterpret_cast<int32_t*>(t), z ? t : nullptr, t, t, ws);
        if (st) {
            printf("status %d: %s\n", st, mi355_last_error());
            return 1;
        }
        printf("%d %u %u\n", g_launches, g_lds, g_threads);
    }
    return 0;
}
