// RelayoutFormat kernels: NCHW <-> NCHW4 / NCHW32, NCHW4 <-> NCHW32, conv weight packing.
// Semantics: naive::RelayoutFormatImpl::exec (dnn/src/naive/relayout_format/opr_impl.cpp:486-773):
// zero-filled destination, permuted copy, per-group channel padding, optional crop on the way
// back, and for QuantizedS8 -> QuantizedS8 with different scales quantize(dequantize(x)).
//
// Two tiers:
//   * relayout_generic_kernel: one thread per destination element, any mode / element size.
//   * byte-transposing kernels for the int8 pure permutations, any channel count and image size;
//     16-byte vectors, coalesced on both sides (HBM bound).
#include "relayout_parts.h"

namespace mi355 {
namespace {

struct RelayoutArgs {
    const void* src;
    void* dst;
    uint32_t mode;
    uint32_t s[7];   // src shape
    uint32_t o[7];   // dst shape
    uint32_t group;
    uint32_t elem_bytes;
    int requant;
    float s_src, s_dst;
    int64_t total;   // dst elements
};

__device__ __forceinline__ int8_t requant_s8(int8_t v, float ss, float sd) {
    float x = (float)v * ss;
    float q = x / sd;
    q = __builtin_roundf(q);
    q = fminf(fmaxf(-128.f, q), 127.f);
    return (int8_t)q;
}

__global__ __launch_bounds__(256) void relayout_generic_kernel(RelayoutArgs a) {
    int64_t di = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (di >= a.total) return;
    int64_t si = -1;
    const uint32_t g = a.group;
    switch (a.mode) {
        case MI355_RL_NCHW_NCHW4_IC_SMALL:
        case MI355_RL_NCHW_NCHW4:
        case MI355_RL_NCHW_NCHW32: {
            const int64_t p = a.o[4], C = a.s[1], H = a.s[2], W = a.s[3], CB = a.o[1];
            const int64_t gg = a.mode == MI355_RL_NCHW_NCHW4_IC_SMALL ? 1 : g;
            const int64_t icpg = C / gg, cpb = CB / gg;
            int64_t t = di;
            int64_t k = t % p; t /= p;
            int64_t w = t % W; t /= W;
            int64_t h = t % H; t /= H;
            int64_t cbg = t % CB;
            int64_t n = t / CB;
            int64_t gi = cbg / cpb, cb = cbg % cpb;
            int64_t cin = cb * p + k;
            if (cin < icpg) si = ((n * C + gi * icpg + cin) * H + h) * W + w;
            break;
        }
        case MI355_RL_NCHW4_NCHW:
        case MI355_RL_NCHW32_NCHW: {
            const int64_t p = a.s[4], CB = a.s[1], H = a.s[2], W = a.s[3], C = a.o[1];
            const int64_t ocpg = C / g, cpb = CB / g;
            int64_t t = di;
            int64_t w = t % W; t /= W;
            int64_t h = t % H; t /= H;
            int64_t c = t % C;
            int64_t n = t / C;
            int64_t gi = c / ocpg, ci = c % ocpg;
            int64_t pc = gi * cpb * p + ci;
            si = (((n * CB + pc / p) * H + h) * W + w) * p + pc % p;
            break;
        }
        case MI355_RL_NCHW_NCHW4_WEIGHT: {
            const int grp = a.o[5] ? 1 : 0;  // 6-dim dst => group
            const int64_t OC = a.s[grp], IC = a.s[grp + 1], FH = a.s[grp + 2], FW = a.s[grp + 3];
            const int64_t OCp = a.o[grp], ICb = a.o[grp + 1];
            int64_t t = di;
            int64_t k = t % 4; t /= 4;
            int64_t fw = t % FW; t /= FW;
            int64_t fh = t % FH; t /= FH;
            int64_t ib = t % ICb; t /= ICb;
            int64_t oc = t % OCp;
            int64_t gi = t / OCp;
            int64_t ic = ib * 4 + k;
            if (oc < OC && ic < IC) si = (((gi * OC + oc) * IC + ic) * FH + fh) * FW + fw;
            break;
        }
        case MI355_RL_NCHW4_NCHW32:
        case MI355_RL_NCHW32_NCHW4: {
            const int64_t ps = a.s[4], pd = a.o[4], H = a.s[2], W = a.s[3], C = (int64_t)a.s[1] * ps;
            int64_t t = di;
            int64_t k = t % pd; t /= pd;
            int64_t w = t % W; t /= W;
            int64_t h = t % H; t /= H;
            int64_t cb = t % (C / pd);
            int64_t n = t / (C / pd);
            int64_t c = cb * pd + k;
            si = (((n * (C / ps) + c / ps) * H + h) * W + w) * ps + c % ps;
            break;
        }
        default:
            break;
    }
    if (a.elem_bytes == 4) {
        reinterpret_cast<int32_t*>(a.dst)[di] = si < 0 ? 0 : reinterpret_cast<const int32_t*>(a.src)[si];
    } else {
        int8_t v = si < 0 ? (int8_t)0 : reinterpret_cast<const int8_t*>(a.src)[si];
        if (a.requant) v = requant_s8(v, a.s_src, a.s_dst);
        reinterpret_cast<int8_t*>(a.dst)[di] = v;
    }
}

// Planes of a plain tensor start at any byte when the image has an odd size: their 16-byte accesses are unaligned ones
// (the memory pipe takes them at full rate as long as a wave's run is contiguous).  The last 16 pixels of a plane start
// at HW - 16, so they overlap the run before them and both write the same bytes: no tail code, every lane does the same.
//
// NCHW -> NCHW4 (C any: missing channels are zero), HW >= 4 (the dispatch sends planes from 16 pixels on).  A step is 4 pixels of 4 channels: a wave loads 256 consecutive bytes of
// each channel and stores one contiguous kilobyte.  (With 16 pixels to a thread the loads are four times as wide, but a store covers a
// quarter of 64 lines, and small images leave the chip idle.)  A thread takes STEPS of them, 64 steps apart, whose loads are in flight
// together (see four_steps).  The last step of a plane ends with it: its first pixels are written twice, with the same bytes.
// grid.x covers CB * ceil(HW / 4) steps per image, grid.y = N.  3 x 224 x 224 (the image of a first layer), against
// 16 pixels to a thread: batch 1 2.55 -> 2.29 us, 16 3.36 -> 2.70, 64 7.50 -> 4.48; 256 x 64 x 64, batch 32: 16.6 -> 11.2 (6 TB/s).
template <int STEPS>
__global__ __launch_bounds__(256) void nchw_to_nchw4_kernel(const int8_t* __restrict__ src, int8_t* __restrict__ dst,
                                                            uint32_t C, uint32_t HW, uint32_t steps, FastDiv pq) {
    const uint32_t first = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 * STEPS) + (threadIdx.x & 63);
    const uint32_t CB = (C + 3) / 4;
    const int8_t* image = src + (int64_t)blockIdx.y * C * HW;
    int8_t* out = dst + (int64_t)blockIdx.y * CB * HW * 4;
    uint32_t r[STEPS][4];
    int64_t at[STEPS];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        const uint32_t it = first + i * 64 < steps ? first + i * 64 : steps - 1;
        const uint32_t cg = fdiv(it, pq), pb = it - cg * pq.d;
        const uint32_t px = pb * 4 + 4 <= HW ? pb * 4 : HW - 4;
        const int8_t* s = image + (int64_t)cg * 4 * HW + px;
        const uint32_t have = C - cg * 4;
        at[i] = ((int64_t)cg * HW + px) * 4;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            r[i][k] = 0;
            if (k < have) r[i][k] = load4u(s + (int64_t)k * HW);
        }
    }
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        if (first + i * 64 >= steps) return;
        uint32_t c0, c1, c2, c3;
        transpose4x4(r[i][0], r[i][1], r[i][2], r[i][3], c0, c1, c2, c3);
        store16u(out + at[i], u32x4{c0, c1, c2, c3});
    }
}

// 4 steps to a thread: from four workgroups for every CU to thirty-two, where few lanes of an image's last workgroup lack a step.  Against one
// step, by the share of lanes that have one: two workgroups to an image and more 0.94 .. 0.98 of the time from 0.88 on, 1.05 to 1.4 below;
// one workgroup 0.84 .. 0.94 from 0.69 on, 1.0 to 2.2 below (2873 images of 364 steps 1.3); beyond thirty-two 1.02 and more.
static bool four_steps(uint64_t steps, uint32_t N, int cu) {
    const uint64_t all = steps * N, few = 4096ull * cu, lanes = (steps + 1023) / 1024 * 1024;
    return all >= few && all < 8 * few && (steps <= 1024 ? steps >= 704 : steps * 8 >= lanes * 7);
}

// NCHW4 -> NCHW (the first C channels), HW >= 4: the same steps the other way round, one to a thread (four are 1.0 to 1.25 times as long).
__global__ __launch_bounds__(256) void nchw4_to_nchw_kernel(const int8_t* __restrict__ src, int8_t* __restrict__ dst,
                                                            uint32_t C, uint32_t HW, uint32_t steps, FastDiv pq) {
    const uint32_t it = blockIdx.x * 256 + threadIdx.x;
    if (it >= steps) return;
    const uint32_t cg = fdiv(it, pq), pb = it - cg * pq.d;
    const uint32_t px = pb * 4 + 4 <= HW ? pb * 4 : HW - 4;
    const uint32_t CB = (C + 3) / 4;
    const u32x4 v = load16u(src + (((int64_t)blockIdx.y * CB + cg) * HW + px) * 4);  // 4 pixels x 4 channels
    uint32_t o[4];
    transpose4x4(v[0], v[1], v[2], v[3], o[0], o[1], o[2], o[3]);
    int8_t* d = dst + ((int64_t)blockIdx.y * C + cg * 4) * HW + px;
    const uint32_t have = C - cg * 4;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (k < have) store4u(d + (int64_t)k * HW, o[k]);
}

// The same with 16 pixels to a thread, HW >= 16: a quarter of the workgroups, whose dispatch is what many small images cost.
__global__ __launch_bounds__(256) void nchw4_to_nchw16_kernel(const int8_t* __restrict__ src, int8_t* __restrict__ dst,
                                                              uint32_t C, uint32_t HW, uint32_t items, FastDiv pq) {
    const uint32_t it = blockIdx.x * 256 + threadIdx.x;
    if (it >= items) return;
    const uint32_t cg = fdiv(it, pq), pb = it - cg * pq.d;
    const uint32_t px = pb * 16 + 16 <= HW ? pb * 16 : HW - 16;
    const uint32_t CB = (C + 3) / 4;
    const int8_t* s = src + (((int64_t)blockIdx.y * CB + cg) * HW + px) * 4;
    u32x4 o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const u32x4 v = load16u(s + j * 16);  // 4 pixels x 4 channels
        uint32_t c0, c1, c2, c3;
        transpose4x4(v[0], v[1], v[2], v[3], c0, c1, c2, c3);
        o[0][j] = c0; o[1][j] = c1; o[2][j] = c2; o[3][j] = c3;
    }
    int8_t* d = dst + ((int64_t)blockIdx.y * C + cg * 4) * HW + px;
    const uint32_t have = C - cg * 4;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (k < have) store16u(d + (int64_t)k * HW, o[k]);
}

// Which of the two.  16 pixels: where an image is one workgroup of those and more of the others, if there are two for every CU (4 pixels take
// 1.02 to 1.2 times as long, 770 images of 280 steps 1.3); where it is three workgroups and more, from four of the others for every CU on
// (1.0 to 1.07); where it is two, if those are nearly full and there are sixteen (1.02 to 1.07).  Elsewhere 4 pixels: of two workgroups the
// second half empty 0.76 to 0.96, small tensors 0.95 to 1.0.
static bool sixteen_pixels(uint64_t steps, uint64_t items, uint32_t N, int cu) {
    const uint64_t all = steps * N;
    if (items <= 256) return steps > 256 && all >= 512ull * cu;
    return items <= 512 ? items >= 448 && all >= 4096ull * cu : all >= 1024ull * cu;
}

// NCHW4 <-> NCHW32: dwords change places.  Two threads per pixel of a 32-channel block, each moves 16 channels: on the
// NCHW32 side a wave covers one contiguous kilobyte, on the other side two runs of 128 bytes per access.
// 16 blocks of 4 at 56 x 56, batch 64: 53 us one byte per thread, 5.8 here.
template <bool TO32>
__global__ __launch_bounds__(256) void nchw4_nchw32_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                           uint32_t HW, uint32_t items, FastDiv hw) {
    const uint32_t it = blockIdx.x * 256 + threadIdx.x;
    if (it >= items) return;
    const uint32_t half = it & 1, t = it >> 1;
    const uint32_t blk = fdiv(t, hw), px = t - blk * HW;      // blk = image * channel blocks of 32 + block
    const int64_t at4 = ((int64_t)blk * 8 + half * 4) * HW + px;
    const int64_t at32 = (int64_t)it * 4;
    if (TO32) {
        u32x4 v;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = src[at4 + (int64_t)k * HW];
        *reinterpret_cast<u32x4*>(dst + at32) = v;
    } else {
        const u32x4 v = *reinterpret_cast<const u32x4*>(src + at32);
#pragma unroll
        for (int k = 0; k < 4; ++k) dst[at4 + (int64_t)k * HW] = v[k];
    }
}

__global__ __launch_bounds__(256) void nchw_to_packed_small_kernel(const int8_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                                   SmallPlanes g) {
    small_planes_quad(src, dst, g, blockIdx.x * 256 + threadIdx.x);
}

// NCHW <-> NCHW32 through LDS.  Tile = 32 channels x 512 pixels (16 KiB).  The LDS image keeps
// the NCHW order (channel rows of 512 bytes, padded to 520 so that rows c and c+16 are 32 banks
// apart); global accesses on both sides are 16-byte vectors over contiguous runs, unaligned ones on the plain side when
// the image has an odd size.  C any: missing channels are zero on the way in and dropped on the way out.
constexpr int RL_TP = 512;           // pixels per tile
constexpr int RL_WAVE = 128;         // of a tile that is one wave (see RlWave)
constexpr int rl_row(int tp) { return tp + 8; }  // padded channel row (bytes): 16 rows = 8320 = 32*256 + 128, or 2176 = 8*256 + 128

// Where 16-byte unit u of a wave's 128 pixels (two units each) lies in LDS: lanes that write units 8 apart and lanes that read consecutive ones
// meet different banks.
__device__ __forceinline__ uint32_t rl_slot(uint32_t u) { return u ^ ((u >> 3 & 3) << 1); }

// Whole lines: from two workgroups to a CU on, if their tiles are three quarters full, and half full from four on.  Bound by bytes there:
// 256 x 64 x 64 at batch 128 46.0 -> 41.3 us (5.8 -> 6.5 TB/s), 64 x 112 x 112 at batch 64 19.7 -> 17.0; 220 drawn conversions 0.84 .. 0.97 of the
// time on this side of the line, 1.03 .. 1.08 with fewer workgroups, where the second meeting in LDS is one more step of a chain, and 1.06 on
// emptier tiles (512 x 14 x 14 at batch 128: 9.5 / 10.1).
static bool whole_lines(uint64_t workgroups, uint64_t tiles_of_plane, uint32_t HW, int cu) {
    const uint64_t room = tiles_of_plane * RL_TP;
    return workgroups >= 4 * (uint64_t)cu ? 2ull * HW >= room : workgroups >= 2 * (uint64_t)cu && 4ull * HW >= 3 * room;
}

// LINES: stores of whole lines, see below
template <bool LINES, int TP>
__device__ __forceinline__ void nchw_to_nchw32(const int8_t* __restrict__ src, int8_t* __restrict__ dst, uint32_t C, uint32_t CB, uint32_t HW) {
    constexpr int RL_ROW = rl_row(TP);
    constexpr uint32_t VECS = TP / 16;  // of a row; a pass of the workgroup (TP / 2 threads) takes eight rows
    __shared__ __attribute__((aligned(16))) int8_t sm[32 * RL_ROW];
    const uint32_t t = threadIdx.x;
    const uint32_t ptiles = (HW + TP - 1) / TP;
    const uint32_t cb = blockIdx.x / ptiles, pt = blockIdx.x % ptiles;
    const uint32_t p0 = pt * TP;
    const int64_t n = blockIdx.y;
    // load: 32 rows of VECS vectors; thread t -> vector t % VECS, rows t / VECS + 8 i
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t row = t / VECS + 8 * i, v = t % VECS;
        uint32_t px = p0 + v * 16;
        u32x4 x = {0, 0, 0, 0};
        if (px < HW && cb * 32 + row < C) x = load16_tail(src + (n * C + cb * 32 + row) * HW + px, HW - px);
        *reinterpret_cast<u32x4*>(sm + row * RL_ROW + v * 16) = x;
    }
    __syncthreads();
    // item: pixel quad pq = t / 2 (4 pixels), half = t % 2 (16 channels)
    const uint32_t pq = t >> 1, half = t & 1;
    uint32_t rows[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
        rows[k] = *reinterpret_cast<const uint32_t*>(sm + (half * 16 + k) * RL_ROW + pq * 4);
    u32x4 out[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t c0, c1, c2, c3;
        transpose4x4(rows[4 * q], rows[4 * q + 1], rows[4 * q + 2], rows[4 * q + 3], c0, c1, c2, c3);
        out[0][q] = c0; out[1][q] = c1; out[2][q] = c2; out[3][q] = c3;
    }
    if constexpr (!LINES) {
        const uint32_t px = p0 + pq * 4;
        int8_t* d = dst + ((n * CB + cb) * HW + px) * 32 + half * 16;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (px + i < HW) *reinterpret_cast<u32x4*>(d + i * 32) = out[i];
        return;
    }
    // A wave's 128 pixels are four contiguous kilobytes of dst: turned once more in LDS, so that a store writes one of them and not 32 bytes of
    // every 128 of all four.
    __syncthreads();
    u32x4* mine = reinterpret_cast<u32x4*>(sm) + (t >> 6) * 256;
    const uint32_t lane = t & 63;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) mine[rl_slot((lane >> 1) * 8 + i * 2 + half)] = out[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t px = p0 + (t >> 6) * 128 + (lane >> 1);
    int8_t* d = dst + ((n * CB + cb) * HW + px) * 32 + half * 16;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i)
        if (px + i * 32 < HW) *reinterpret_cast<u32x4*>(d + i * 1024) = mine[rl_slot(i * 64 + lane)];
}

template <int TP>
__device__ __forceinline__ void nchw32_to_nchw(const int8_t* __restrict__ src, int8_t* __restrict__ dst, uint32_t C, uint32_t CB, uint32_t HW) {
    constexpr int RL_ROW = rl_row(TP);
    constexpr uint32_t VECS = TP / 16;
    __shared__ __attribute__((aligned(16))) int8_t sm[32 * RL_ROW];
    const uint32_t t = threadIdx.x;
    const uint32_t ptiles = (HW + TP - 1) / TP;
    const uint32_t cb = blockIdx.x / ptiles, pt = blockIdx.x % ptiles;
    const uint32_t p0 = pt * TP;
    const int64_t n = blockIdx.y;
    const uint32_t pq = t >> 1, half = t & 1;
    const uint32_t px = p0 + pq * 4;
    u32x4 in[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        in[i] = u32x4{0, 0, 0, 0};
        if (px + i < HW) in[i] = *reinterpret_cast<const u32x4*>(src + ((n * CB + cb) * HW + px + i) * 32 + half * 16);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t c0, c1, c2, c3;
        // rows = pixels, bytes = channels 4q..4q+3  ->  columns = channels, bytes = pixels
        transpose4x4(in[0][q], in[1][q], in[2][q], in[3][q], c0, c1, c2, c3);
        uint32_t base = (half * 16 + 4 * q) * RL_ROW + pq * 4;
        *reinterpret_cast<uint32_t*>(sm + base) = c0;
        *reinterpret_cast<uint32_t*>(sm + base + RL_ROW) = c1;
        *reinterpret_cast<uint32_t*>(sm + base + 2 * RL_ROW) = c2;
        *reinterpret_cast<uint32_t*>(sm + base + 3 * RL_ROW) = c3;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t row = t / VECS + 8 * i, v = t % VECS;
        uint32_t p = p0 + v * 16;
        if (p < HW && cb * 32 + row < C) {
            u32x4 x = *reinterpret_cast<const u32x4*>(sm + row * RL_ROW + v * 16);
            store16_tail(dst + (n * C + cb * 32 + row) * HW + p, x, HW - p);
        }
    }
}

template <bool LINES>
__global__ __launch_bounds__(256) void nchw_to_nchw32_kernel(const int8_t* __restrict__ src, int8_t* __restrict__ dst, uint32_t C, uint32_t CB,
                                                             uint32_t HW) {
    nchw_to_nchw32<LINES, RL_TP>(src, dst, C, CB, HW);
}
__global__ __launch_bounds__(256) void nchw32_to_nchw_kernel(const int8_t* __restrict__ src, int8_t* __restrict__ dst, uint32_t C, uint32_t CB,
                                                             uint32_t HW) {
    nchw32_to_nchw<RL_TP>(src, dst, C, CB, HW);
}

// The form with tiles of one wave, four times as many: where workgroups of the other are few, into NCHW32 up to three for four CUs (130 drawn
// conversions 0.91 of the time on average, beyond, to 384, 0.97 .. 1.04; 128 x 54 x 33 at batch 2 3.96 -> 3.47 us), back up to one for two (93 drawn ones
// 0.94, beyond 0.99 .. 1.05; 128 x 27 x 22 at batch 2 3.05 -> 2.88).  From 400 on it loses to shorter runs of a plane: 1.02 .. 1.4.
struct RlWave {
    const int8_t* src;
    int8_t* dst;
    uint32_t C, CB, HW;
};
template <bool LINES>
__global__ __launch_bounds__(64) void nchw_to_nchw32_kernel(RlWave a) {
    nchw_to_nchw32<LINES, RL_WAVE>(a.src, a.dst, a.C, a.CB, a.HW);
}
__global__ __launch_bounds__(64) void nchw32_to_nchw_kernel(RlWave a) {
    nchw32_to_nchw<RL_WAVE>(a.src, a.dst, a.C, a.CB, a.HW);
}

}  // namespace

int launch_relayout(hipStream_t st, const mi355_relayout_desc& d, const uint32_t* oshape, uint32_t ondim,
                    const void* src, void* dst, bool allow_fast, int cu_count) {
    int64_t total = 1;
    if (cu_count <= 0) cu_count = 256;
    for (uint32_t i = 0; i < ondim; ++i) total *= oshape[i];
    if (total == 0) return 0;
    const bool requant = d.elem_bytes == 1 && d.scale_src != d.scale_dst;
    const uint32_t g = d.group ? d.group : 1;
    // byte permutations without channel groups: kernels that move vectors.  What is left to the generic kernel -- rescaling
    // conversions, group padding, 32-bit elements, weights with padded output channels -- runs once per model or not at all.
    // Their tensors may have any size (offsets are 64 bits wide); what is 32 bits wide is the number of a thread.  (33 images of
    // 256 x 512 x 512, 2.2 GB: 0.8 to 0.9 ms in either direction and packing, 7.7 to 8.5 one byte per thread.)
    const uint64_t HW64 = d.ndim >= 4 ? (uint64_t)d.shape[2] * d.shape[3] : 0;
    auto numbered = [](uint64_t threads) { return threads <= 0xffffff00ull; };
    if (allow_fast && d.elem_bytes == 1 && !requant && g == 1 && d.shape[0] <= 65535 && HW64 < (1ull << 31)) {
        const uint32_t N = d.shape[0], HW = (uint32_t)HW64;
        const int8_t* s8 = (const int8_t*)src;
        int8_t* d8 = (int8_t*)dst;
        const uint32_t ptiles = (HW + RL_TP - 1) / RL_TP;
        switch (d.mode) {
            case MI355_RL_NCHW_NCHW4:
            case MI355_RL_NCHW_NCHW4_IC_SMALL:
            case MI355_RL_NCHW_NCHW32: {
                const uint32_t C = d.shape[1], CB = oshape[1];
                const uint32_t pq = (HW + 3) / 4;
                if (oshape[4] == 4 && HW >= 16 && numbered((uint64_t)CB * pq + 1024)) {
                    const uint32_t steps = CB * pq;
                    if (four_steps(steps, N, cu_count))
                        return launch_kernel(nchw_to_nchw4_kernel<4>, dim3((steps + 1023) / 1024, N), dim3(256), 0, st, s8, d8, C, HW,
                                             steps, make_fastdiv(pq));
                    return launch_kernel(nchw_to_nchw4_kernel<1>, dim3((steps + 255) / 256, N), dim3(256), 0, st, s8, d8, C, HW, steps,
                                         make_fastdiv(pq));
                }
                // planes of a quarter of the LDS tile and more: below, most of a tile's threads would find no pixel
                if (oshape[4] == 32 && HW >= RL_TP / 4 && numbered((uint64_t)CB * ptiles * 256)) {
                    typedef void (*Tile)(const int8_t*, int8_t*, uint32_t, uint32_t, uint32_t);
                    if (4ull * N * CB * ptiles <= 3ull * cu_count)
                        return launch_kernel((void (*)(RlWave))nchw_to_nchw32_kernel<false>, dim3(CB * ((HW + RL_WAVE - 1) / RL_WAVE), N), dim3(64), 0, st,
                                             RlWave{s8, d8, C, CB, HW});
                    const Tile tile = whole_lines((uint64_t)N * CB * ptiles, ptiles, HW, cu_count) ? (Tile)nchw_to_nchw32_kernel<true> : (Tile)nchw_to_nchw32_kernel<false>;
                    return launch_kernel(tile, dim3(CB * ptiles, N), dim3(256), 0, st, s8, d8, C, CB, HW);
                }
                if (!numbered((uint64_t)total / 4)) break;
                const SmallPlanes g = make_small_planes(N, C, HW, oshape[4]);
                return launch_kernel(nchw_to_packed_small_kernel, dim3((g.items + 255) / 256), dim3(256), 0, st, s8,
                                     reinterpret_cast<uint32_t*>(dst), g);
            }
            case MI355_RL_NCHW4_NCHW:
                if (HW >= 16 && numbered((uint64_t)d.shape[1] * ((HW + 3) / 4) + 256)) {
                    const uint32_t C = oshape[1], pq = (HW + 3) / 4, steps = d.shape[1] * pq;
                    const uint32_t p16 = (HW + 15) / 16, items = d.shape[1] * p16;
                    if (sixteen_pixels(steps, items, N, cu_count))
                        return launch_kernel(nchw4_to_nchw16_kernel, dim3((items + 255) / 256, N), dim3(256), 0, st, s8, d8, C, HW, items,
                                             make_fastdiv(p16));
                    return launch_kernel(nchw4_to_nchw_kernel, dim3((steps + 255) / 256, N), dim3(256), 0, st, s8, d8, C, HW, steps,
                                         make_fastdiv(pq));
                }
                break;
            case MI355_RL_NCHW32_NCHW:
                if (!numbered((uint64_t)d.shape[1] * ptiles * 256)) break;
                if (2ull * N * d.shape[1] * ptiles <= (uint64_t)cu_count)
                    return launch_kernel((void (*)(RlWave))nchw32_to_nchw_kernel, dim3(d.shape[1] * ((HW + RL_WAVE - 1) / RL_WAVE), N), dim3(64), 0, st,
                                         RlWave{s8, d8, oshape[1], d.shape[1], HW});
                return launch_kernel((void (*)(const int8_t*, int8_t*, uint32_t, uint32_t, uint32_t))nchw32_to_nchw_kernel, dim3(d.shape[1] * ptiles, N),
                                     dim3(256), 0, st, s8, d8, oshape[1], d.shape[1], HW);
            case MI355_RL_NCHW4_NCHW32:
            case MI355_RL_NCHW32_NCHW4: {
                if (!numbered((uint64_t)total / 16)) break;
                const uint32_t items = (uint32_t)(total / 16);
                const uint32_t* sw = (const uint32_t*)src;
                uint32_t* dw = (uint32_t*)dst;
                if (d.mode == MI355_RL_NCHW4_NCHW32)
                    return launch_kernel(nchw4_nchw32_kernel<true>, dim3((items + 255) / 256), dim3(256), 0, st, sw, dw, HW, items,
                                         make_fastdiv(HW));
                return launch_kernel(nchw4_nchw32_kernel<false>, dim3((items + 255) / 256), dim3(256), 0, st, sw, dw, HW, items,
                                     make_fastdiv(HW));
            }
            default:
                break;
        }
    }
    RelayoutArgs a;
    a.src = src; a.dst = dst; a.mode = d.mode;
    for (int i = 0; i < 7; ++i) {
        a.s[i] = i < (int)d.ndim ? d.shape[i] : 0;
        a.o[i] = i < (int)ondim ? oshape[i] : 0;
    }
    a.group = g;
    a.elem_bytes = d.elem_bytes;
    a.requant = requant ? 1 : 0;
    a.s_src = d.scale_src; a.s_dst = d.scale_dst;
    a.total = total;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 0x7fffffff) return (int)hipErrorInvalidValue;
    return launch_kernel(relayout_generic_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a);
}

}  // namespace mi355
