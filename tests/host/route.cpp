// Which kernels an exec launches (no GPU: the runtime's calls that would need one are answered here, and a launch is only noted).
// One exec per line of the input: the descriptor's bytes in hexadecimal, an algorithm (a number: by that name; -1: the heuristic's
// choice, named; -2: none, exec chooses for itself), its tile (-1: the query's), and whether there is a workspace.  One line of the
// output for each: the number of launches, dynamic LDS, threads, and workgroups in the first dimension of the last one, and the kernels, separated by
// tabs.
// A descriptor of a layout conversion or of a pooling, told apart by its size, is executed as such.
#include <cxxabi.h>
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>

#include "../../include/mi355_convbias.h"

static std::map<const void*, std::string>& kernels() {  // (filled by the library's constructors, ahead of this file's)
    static std::map<const void*, std::string> m;
    return m;
}
static std::string g_names;
static int g_launches;
static unsigned g_lds, g_threads, g_grid;
extern "C" {
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    int st;
    char* s = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    kernels()[host] = s ? s : name;
    free(s);
}
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
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t lds, hipStream_t) {
    ++g_launches;
    g_lds = (unsigned)lds;
    g_threads = block.x;
    g_grid = grid.x;
    g_names += "\t" + (kernels().count(f) ? kernels()[f] : "?");
    return hipSuccess;
}
}

int main() {
    static char hex[2 * sizeof(mi355_conv_desc) + 2];
    char format[32];
    snprintf(format, sizeof(format), "%%%zus %%d %%d %%d", sizeof(hex) - 1);
    int algo, tile, room;
    while (scanf(format, hex, &algo, &tile, &room) == 4) {
        unsigned char bytes[sizeof(mi355_conv_desc)];
        const size_t size = strlen(hex) / 2;
        unsigned b;
        for (size_t i = 0; i < size; ++i) {
            if (sscanf(hex + 2 * i, "%2x", &b) != 1) return 1;
            bytes[i] = (unsigned char)b;
        }
        int8_t* const t = reinterpret_cast<int8_t*>(0x1000000);  // device addresses that nothing on the host reads
        g_launches = 0;
        g_names.clear();
        int st;
        if (size == sizeof(mi355_conv_desc)) {
            mi355_conv_desc d;
            memcpy(&d, bytes, size);
            mi355_algo a;
            size_t ws = 0;
            st = mi355_convbias_s8_query(&d, algo < 0 ? MI355_ALGO_HEURISTIC : algo, &a, &ws);
            if (tile >= 0) a.tile_cfg = tile;
            if (!st)
                st = mi355_convbias_s8_exec(nullptr, &d, algo == -2 ? nullptr : &a, t, t, reinterpret_cast<int32_t*>(t), d.has_z ? t : nullptr,
                                            t, room ? t : nullptr, room ? ws : 0);
        } else if (size == sizeof(mi355_relayout_desc)) {
            mi355_relayout_desc d;
            memcpy(&d, bytes, size);
            st = mi355_relayout_exec(nullptr, &d, t, t);
        } else if (size == sizeof(mi355_pooling_desc)) {
            mi355_pooling_desc d;
            memcpy(&d, bytes, size);
            st = mi355_pooling_s8_exec(nullptr, &d, t, t);
        } else {
            printf("a descriptor of %zu bytes\n", size);
            return 1;
        }
        if (st) {
            printf("status %d: %s\n", st, mi355_last_error());
            return 1;
        }
        printf("%d %u %u %u%s\n", g_launches, g_lds, g_threads, g_grid, g_names.c_str());
    }
    return 0;
}
