// The tile of a dense 32-packed layer on devices of different sizes (no GPU: the two calls of the runtime that say what the device
// is are answered here).  Choices that go by rounds of tiles over the CUs make the same choice for n images on half a device as
// for 2n images on a whole one, wherever the tiles of n images are half those of 2n.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>

#include "../../include/mi355_convbias.h"

static const int kCus[] = {256, 128};  // CUs of device 0 and 1
static int g_device = 0;
extern "C" hipError_t hipGetDevice(int* d) {
    *d = g_device;
    return hipSuccess;
}
extern "C" hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int d) {  // (the header names the current form of the struct)
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = kCus[d];
    return hipSuccess;
}

static int pick(uint32_t n, uint32_t ic, uint32_t oc, uint32_t f, uint32_t stride, int z, int device) {
    mi355_conv_desc d;
    memset(&d, 0, sizeof(d));
    d.format = MI355_FMT_NCHW32;
    d.n = n;
    d.ic = ic;
    d.oc = oc;
    d.group = 1;
    d.ih = d.iw = 32 * stride;  // 32 x 32 outputs: pixels of an image are a multiple of every tile
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
    size_t ws;
    g_device = device;
    const int st = mi355_convbias_s8_query(&d, MI355_ALGO_HEURISTIC, &a, &ws);
    if (st || a.id != 1) {
        printf("query: %s\n", mi355_last_error());
        return -1;
    }
    return a.tile_cfg;
}

int main() {
    int layers = 0, bad = 0, seen[256] = {0};
    for (uint32_t ic : {128u, 160u, 256u, 512u, 832u})
        for (uint32_t oc : {64u, 128u, 192u, 320u, 512u})
            for (uint32_t f : {3u, 5u})
                for (uint32_t stride : {1u, 2u})
                    for (int z : {0, 1})
                        for (uint32_t n : {24u, 27u, 34u, 47u, 64u}) {
                            // (that many pixels: no layer goes to the few-pixel tiles, whose line is not one of rounds)
                            int t[2];
                            for (int dev = 0; dev < 2; ++dev) t[dev] = pick(n << (1 - dev), ic, oc, f, stride, z, dev);
                            ++layers;
                            if (t[0] < 0 || t[1] < 0) return 1;
                            ++seen[t[0] & 255];
                            if (t[0] != t[1] && bad++ < 5)
                                printf("%u -> %u, %ux%u, stride %u, z %d: %u images on 256 CUs take tile %d, %u on 128 tile %d\n", ic, oc, f, f, stride, z, 2 * n, t[0],
                                       n, t[1]);
                        }
    int kinds = 0;
    for (int s : seen) kinds += s > 0;
    printf("%d layers, %d tiles, %d differ\n", layers, kinds, bad);
    if (bad || kinds < 4) return 1;
    printf("ALL OK\n");
    return 0;
}
