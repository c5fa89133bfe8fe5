// Where the residual loads and the stores of plain NCHW layers in one launch and of grouped layers on the matrix cores lead (no GPU).
// conv_patch1.hip and conv_group4.hip are compiled into this program, a launch is noted with its arguments, and the offsets of every lane of
// every wave are made by the kernel's own functions.  By the rule at SENT (igemm_shared.h) a lane either passes SENT or stays inside the tensor
// with its scalar offset added, and the scalar offset alone does too.
// One descriptor per line of the input, in hexadecimal; one line of the output for each: the tile (blocks of 32 channels, of 128 pixels; 0 0 for
// grouped layers), the accesses that were looked at, and those that break the rule.
#include <cxxabi.h>
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>

#include "../../megengine_amd/csrc/common.h"
namespace mi355 {
__host__ static inline uint32_t fdiv(uint32_t x, const FastDiv& f) {
    const uint32_t t = (uint32_t)((uint64_t)x * f.m >> 32);
    return (t + ((x - t) >> f.s1)) >> f.s2;
}
}  // namespace mi355
#pragma GCC visibility push(hidden)  // (the library's launch code runs, not this copy of it)
#include "../../megengine_amd/csrc/conv_patch1.hip"
#include "../../megengine_amd/csrc/conv_group4.hip"
#pragma GCC visibility pop

namespace mi355 {
static int g_mt, g_nt;  // of the last launch
static P1Args g_args;
static G16Args<FastDiv> g_grouped;
static long g_seen, g_broken;

// `size` bytes at the two offsets, in a tensor of `bytes`
static void look(int lane, int scalar, int size, uint32_t bytes) {
    ++g_seen;
    const bool scalar_in = scalar >= 0 && (uint32_t)scalar <= bytes;
    const bool lane_in = lane < 0 || (int64_t)lane + scalar + size <= bytes;  // (SENT, whatever is or'ed to it)
    if (!scalar_in || !lane_in) ++g_broken;
}

static void walk(const P1Args& a) {
    for (int tm = 0; tm < a.tiles_m; ++tm)
        for (int tn = 0; tn < a.tiles_n; ++tn) {
            const P1Tile o = p1_tile_at(a, tn);
            for (int px = 0; px < 128 * g_nt; px += 4)
                for (int ch = 0; ch < 8; ++ch) {
                    const P1Out w = p1_out(a, o, px, ch);
                    const P1Residual z = p1_residual_at(a, w);
                    for (int oc8 = tm * g_mt * 32; oc8 < (tm + 1) * g_mt * 32; oc8 += 8) {
                        const P1Access at = p1_access(a, oc8, ch);
                        if (a.epi.has_z) {
                            look(at.lane | z.off, at.scalar, 4, a.z_bytes);
                            if (a.OHW < 4 && g_mt * g_nt > 2) look(p1_residual_across(w, at).off, 0, 4, a.z_bytes);
                            if (a.OHW < 4 && g_mt * g_nt <= 2)
                                for (int k = 0; k < 3; ++k) look(at.lane | (k < w.cols ? w.z0 + k : SENT), at.scalar, 1, a.z_bytes);
                        }
                        look(at.lane | (w.cols > 0 ? w.d0 : SENT), at.scalar, w.cols < 4 ? w.cols : 4, a.dst_bytes);
                    }
                }
        }
}

static void look(const G16Access& at, uint32_t bytes) { look(at.lane, at.scalar, 4, bytes); }
static void walk(const G16Args<FastDiv>& a) {
    const uint32_t bytes = (uint32_t)a.dst_scb * 4;
    for (int band = 0; band < a.bands; ++band) {
        const int oh0 = band * a.TH, pixels = (a.OH - oh0 < a.TH ? a.OH - oh0 : a.TH) * a.OW, base = oh0 * a.OW * 4;
        for (int t = 0; t < 256; ++t) {
            G16Lane l;
            l.p = (t >> 6) * 32 + (t & 15);
            l.out = (t >> 4 & 3) * a.dst_scb + l.p * 4;
            const int first = (t >> 6) * 32;
            for (int k = 0; k < 2; ++k) {
                if (a.epi.has_z) look(g16_access(l, k, 0, first, pixels, base), bytes);
                for (int u = 0; first + u < pixels; u += 128) {
                    if (a.epi.has_z) look(g16_access(l, k, u + 128, first, pixels, base), bytes);
                    look(g16_access(l, k, u, first, pixels, base), bytes);
                }
            }
        }
    }
}

static std::map<const void*, std::string>& kernels() {  // (filled ahead of this file's constructors)
    static std::map<const void*, std::string> m;
    return m;
}
}  // namespace mi355

extern "C" {
char __hip_fatbin[16];  // (compiled for the host alone: no kernels to register)
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    int st;
    char* s = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    mi355::kernels()[host] = s ? s : name;
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
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    const std::string& name = mi355::kernels()[f];
    mi355::g_mt = mi355::g_nt = 0;
    if (name.find("grp16_kernel<") != std::string::npos) {
        if (name.find("G16Wide") != std::string::npos) {
            mi355::g_grouped = static_cast<mi355::G16Wide*>(args[0])->a;
        } else {
            static_cast<mi355::G16Wire*>(args[0])->numbers(mi355::g_grouped);
            mi355::g_grouped.epi.has_z = static_cast<mi355::G16Wire*>(args[0])->flags >> 3 & 1;
        }
        return hipSuccess;
    }
    const size_t at = name.find("patch1_kernel<");
    if (at == std::string::npos || sscanf(name.c_str() + at, "patch1_kernel<%d, %d", &mi355::g_mt, &mi355::g_nt) != 2) return hipErrorInvalidValue;
    memcpy(&mi355::g_args, args[0], sizeof(mi355::g_args));
    return hipSuccess;
}
}

int main() {
    static char hex[2 * sizeof(mi355_conv_desc) + 2];
    char format[32];
    snprintf(format, sizeof(format), "%%%zus", sizeof(hex) - 1);
    while (scanf(format, hex) == 1) {
        mi355_conv_desc d;
        unsigned b;
        for (size_t i = 0; i < sizeof(d); ++i) {
            if (sscanf(hex + 2 * i, "%2x", &b) != 1) return 1;
            reinterpret_cast<unsigned char*>(&d)[i] = (unsigned char)b;
        }
        int8_t* const t = reinterpret_cast<int8_t*>(0x1000000);  // device addresses that nothing on the host reads
        const int st = mi355_convbias_s8_exec(nullptr, &d, nullptr, t, t, reinterpret_cast<int32_t*>(t), d.has_z ? t : nullptr, t, nullptr, 0);
        if (st) {
            printf("status %d: %s\n", st, mi355_last_error());
            return 1;
        }
        mi355::g_seen = mi355::g_broken = 0;
        mi355::g_mt ? mi355::walk(mi355::g_args) : mi355::walk(mi355::g_grouped);
        printf("%d %d %ld %ld\n", mi355::g_mt, mi355::g_nt, mi355::g_seen, mi355::g_broken);
    }
    return 0;
}
