// A host that runs out of memory while a call is bound (no GPU): mi355_convbias_s8_bind reports it, returns no call, throws
// nothing through the C interface, and leaves the thread as it was -- an exec after it goes to the device (which is not
// there, so it fails) instead of being noted down as part of the call that was not bound.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <new>

#include "../../include/mi355_convbias.h"

static thread_local int g_left = -1;  // allocations until one fails; negative: none does
void* operator new(size_t n) {
    if (g_left >= 0 && g_left-- == 0) throw std::bad_alloc();
    void* p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void* operator new(size_t n, const std::nothrow_t&) noexcept { return g_left >= 0 && g_left-- == 0 ? nullptr : malloc(n ? n : 1); }
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

int main() {
    mi355_conv_desc d;
    memset(&d, 0, sizeof(d));
    d.format = MI355_FMT_NCHW4;  // channel-wise
    d.sparse = MI355_SPARSE_GROUP;
    d.n = 2;
    d.ic = d.oc = d.group = 16;
    d.ih = d.iw = 9;
    d.fh = d.fw = 3;
    d.pad_h = d.pad_w = d.stride_h = d.stride_w = d.dilate_h = d.dilate_w = 1;
    d.scale_bias = 2e-4f;
    d.scale_z = d.scale_dst = 0.05f;
    d.bias_mode = MI355_BIAS_BROADCAST_CHANNEL;
    mi355_algo a;
    size_t ws;
    int8_t* const t = reinterpret_cast<int8_t*>(0x1000000);  // device addresses that nothing on the host reads
    if (mi355_convbias_s8_query(&d, MI355_ALGO_HEURISTIC, &a, &ws) != MI355_OK) return printf("query: %s\n", mi355_last_error()), 1;
    int refused = 0, bound = 0;
    for (int k = 0; k < 32 && bound < 2; ++k) {
        mi355_bound_call* b = nullptr;
        g_left = k;
        const int st = mi355_convbias_s8_bind(&d, &a, t, t, 0, reinterpret_cast<int32_t*>(t), nullptr, t, nullptr, 0, &b);
        g_left = -1;
        (st == MI355_OK ? bound : refused)++;
        if ((st == MI355_OK) != (b != nullptr)) return printf("allocation %d: status %d, call %p\n", k, st, (void*)b), 1;
        const int ex = mi355_convbias_s8_exec(nullptr, &d, &a, t, t, reinterpret_cast<int32_t*>(t), nullptr, t, nullptr, 0);
        if (ex != MI355_ERR_LAUNCH) return printf("allocation %d: exec without a device answers %d\n", k, ex), 1;
        mi355_bound_call_destroy(b);
    }
    if (refused < 3 || bound < 2) return printf("%d refused, %d bound\n", refused, bound), 1;
    printf("ALL OK\n");
    return 0;
}
