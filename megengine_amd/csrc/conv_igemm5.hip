// Implicit GEMM for convolutions with few output pixels (tiles "v2_ks_*" for 32-packed
// inputs, "ks4_*" for 4-packed ones): the reduction of one small output tile is split
// over the waves of a workgroup, and operands go from global memory straight into registers.
//
// A layer of one image leaves a tiled kernel two bad choices: its tiles are too few for the chip, and one tile is a serial
// chain of LDS stages (copy, barrier, multiply) as long as the reduction -- 3x3 over 512 channels at 7 x 7 took 11 us on
// 16 workgroups, 36 stages of 0.3 us each, whatever the tile.  What bounds such a layer is latency, so this kernel has
// next to none of its own:
//   * tile = 16 to 64 channels x 16 or 32 pixels, so that the tiles of a layer reach more of the 256 CUs;
//   * the waves of a workgroup take contiguous pieces of the reduction.  An MFMA operand of a 32-byte k-chunk is one
//     16-byte load per lane (32 filter rows, or 32 pixels of a 32-packed tensor: one contiguous kilobyte); a wave keeps
//     several chunks of both operands in flight, sixteen waves therefore most of the tile's operands, and memory is
//     waited for about once instead of once per stage;
//   * no staging, no barrier before the partial sums meet in LDS; there the quads of an accumulator block are dealt out
//     over the waves again, each adds up its quad, adds the bias, requantises and stores.
// The price is operand traffic (2 KB per MFMA of a 32 x 32 tile, through a path of 64 bytes per clock and CU): with enough
// pixels to fill the chip the staged tiles win, see the chooser.
//
// 4-packed inputs: a lane's 16 k-bytes are four dwords of its pixel, one per (channel block, tap) unit of the filter's own
// order; a table in LDS says where each unit lies.
#include <atomic>
#include <tuple>

#include "igemm_shared.h"
#include "wire.h"

namespace mi355 {
namespace {

// MFMA steps whose operands a wave keeps in flight
constexpr int ks_ahead(int s, int mt) { return s == 16 ? 6 : mt == 1 ? 8 : 4; }
// 16-byte vectors between the rows of partial sums in LDS (a row: 4 channels of the S pixels of a block): both ways of
// reading them back -- a row by consecutive lanes, or all rows of a pixel by consecutive lanes -- then meet every bank once
// per pass
constexpr int ks_row(int s) { return s == 32 ? 34 : 20; }
// vectors of a wave's share of LDS: its partial sums, and before them (TURN) a stage of the filter, 128 bytes of each row of the tile
constexpr int ks_wave_vecs(int s, int mt, bool turn) {
    const int sums = mt * (s / 4) * ks_row(s), stage = mt * s * 8;
    return turn && stage > sums ? stage : sums;
}

template <class Div>
struct KsArgs {
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    uint32_t src_bytes, flt_bytes, z_bytes, dst_bytes;
    int IH, IW, OHW, OW, FW, T;
    int sh, sw, ph, pw;
    int OC, M, KC, entries;
    int src_sn, src_scb, dst_sn, dst_scb, z_sn;
    int flt_rstride, flt_kstride;
    int tiles_m, tiles_n, by_m;
    int FH, steps, per_wave, extra;  // steps of the reduction: per_wave for every wave, one more for the first `extra`
    int log_pout, has_bias, dst_s32;
    Div div_tile;                    // by tiles_n (by_m) or tiles_m
    Div div_ohw, div_ow, div_t, div_fw;
    EpiParams epi;

    auto numbers() const {
        return std::tie(src_bytes, flt_bytes, z_bytes, dst_bytes, IH, IW, OHW, OW, FW, T, sh, sw, ph, pw, OC, M, KC, entries, src_sn, src_scb,
                        dst_sn, dst_scb, z_sn, flt_rstride, flt_kstride, tiles_m, tiles_n, by_m, FH, steps, per_wave, extra, log_pout, has_bias,
                        dst_s32);
    }
};

// The two forms of the kernel's argument (see wire.h)
struct KsWide {
    static constexpr bool WIRE = false;
    KsArgs<FastDiv> a;
    template <int PIN, int S, int MT, int W>
    __device__ __forceinline__ KsArgs<FastDiv> open() const { return a; }
};

struct KsWire {
    static constexpr bool WIRE = true;
    const int8_t* src;
    const int8_t* flt;
    const int32_t* bias;
    const int8_t* z;
    int8_t* dst;
    uint32_t N, in, out, channels, window, flags, kstride;  // in, out: height | width << 16; channels: out | blocks in << 16
    EpiWire epi;

    template <int PIN, int S, int MT, int W, class Div>
    __host__ __device__ __forceinline__ void numbers(KsArgs<Div>& k) const {
        k.IH = wire_lo(in); k.IW = wire_hi(in);
        k.OW = wire_hi(out); k.OHW = wire_mul(wire_lo(out), k.OW);
        k.sh = wire_byte(window, 0); k.sw = wire_byte(window, 1); k.ph = wire_byte(window, 2); k.pw = wire_byte(window, 3);
        k.FH = wire_byte(flags, 2); k.FW = wire_byte(flags, 3); k.T = k.FH * k.FW;
        k.OC = wire_lo(channels);
        k.M = wire_mul((int)N, k.OHW);
        k.entries = wire_mul(wire_hi(channels), k.T);
        k.KC = PIN == 32 ? k.entries : (k.entries + 7) / 8;
        k.src_scb = wire_mul(k.IH, k.IW, PIN); k.src_sn = wire_mul(wire_hi(channels), k.src_scb);
        k.log_pout = (int)(flags >> 8 & 7); k.has_bias = (int)(flags >> 11 & 1); k.dst_s32 = (int)(flags >> 12 & 1);
        k.dst_scb = wire_mul(k.OHW, 1 << k.log_pout); k.dst_sn = wire_mul(k.OC, k.OHW);
        k.z_sn = (flags >> 3 & 1) ? k.dst_sn : 0;
        const uint32_t el = k.dst_s32 ? 4 : 1;
        k.src_bytes = N * (uint32_t)k.src_sn; k.dst_bytes = N * (uint32_t)k.dst_sn * el; k.z_bytes = N * (uint32_t)k.z_sn * el;
        const bool pre = (flags >> 13 & 1) != 0;  // [32-byte chunk][channel] instead of rows
        k.flt_kstride = (int)kstride;
        k.flt_rstride = pre ? 32 : wire_mul(k.entries, PIN);
        k.flt_bytes = pre ? (uint32_t)k.KC * kstride : (uint32_t)k.OC * (uint32_t)k.flt_rstride;
        k.tiles_m = (k.OC + MT * S - 1) / (MT * S);
        k.tiles_n = (k.M + S - 1) / S;
        k.by_m = k.tiles_m >= 8;
        k.steps = S == 32 ? k.KC : (k.KC + 1) / 2;
        k.per_wave = k.steps / W;
        k.extra = k.steps % W;
    }
    template <int PIN, int S, int MT, int W>
    __device__ __forceinline__ KsArgs<Quot> open() const {
        asm volatile("" ::"s"(src), "s"(flt), "s"(bias), "s"(z), "s"(dst), "s"(N), "s"(in), "s"(out), "s"(channels), "s"(window), "s"(flags),
                     "s"(kstride), "s"(epi.f[0]), "s"(epi.f[1]), "s"(epi.f[2]), "s"(epi.f[3]));  // one batch of scalar loads
        KsArgs<Quot> k;
        k.src = src; k.flt = flt; k.bias = bias; k.z = z; k.dst = dst;
        numbers<PIN, S, MT, W>(k);
        k.div_tile = quot(k.by_m ? k.tiles_n : k.tiles_m);
        k.div_ohw = quot(k.OHW); k.div_ow = quot(k.OW);
        k.div_t = quot(k.T); k.div_fw = quot(k.FW);
        k.epi = epi_open(epi, flags & 255);
        return k;
    }
    // false: the problem has a number that does not fit
    template <int PIN, int S, int MT, int W>
    bool pack(const KsArgs<FastDiv>& k, uint32_t n) {
        src = k.src; flt = k.flt; bias = k.bias; z = k.z; dst = k.dst;
        N = n; in = wire2(k.IH, k.IW); out = wire2(k.OW ? k.OHW / k.OW : 0, k.OW);
        channels = wire2(k.OC, k.T ? k.entries / k.T : 0);
        window = wire4(k.sh, k.sw, k.ph, k.pw);
        kstride = (uint32_t)k.flt_kstride;
        flags = epi_wire(k.epi, k.dst_s32, &epi) | (uint32_t)k.log_pout << 8 | (k.has_bias ? 1u << 11 : 0) | (k.dst_s32 ? 1u << 12 : 0) |
                (k.flt_rstride != wire_mul(k.entries, PIN) ? 1u << 13 : 0) | wire4(0, 0, k.FH, k.FW);
        KsArgs<FastDiv> o;
        numbers<PIN, S, MT, W>(o);
        if (!k.epi.has_z) o.z_sn = k.z_sn;  // (nothing reads it)
        return o.numbers() == k.numbers() && k.M < QUOT_MAX && (int64_t)k.entries + 16 < QUOT_MAX && (int64_t)(k.tiles_m + 8) * (k.tiles_n + 8) < QUOT_MAX;
    }
};
static_assert(sizeof(KsWire) <= WIRE_BYTES, "a wire");

// S = 32: v_mfma_i32_32x32x32_i8, a step is one 32-byte k-chunk; S = 16: v_mfma_i32_16x16x64_i8, a step is two of them.
// Lane l holds filter row (pixel) l % S and 16 bytes at 16 (l / S) of the step.
template <int S>
struct KsAcc;
template <>
struct KsAcc<32> {
    v16i v;
    __device__ __forceinline__ void clear() { v = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}; }
    __device__ __forceinline__ void mfma(v4i a, v4i b) { v = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, v, 0, 0, 0); }
    // quad q: channels 8 q + 4 (lane / 32) .. + 3, a row of its own in LDS
    __device__ __forceinline__ v4i quad(int q) const { return v4i{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]}; }
};
template <>
struct KsAcc<16> {
    v4i v;
    __device__ __forceinline__ void clear() { v = v4i{0, 0, 0, 0}; }
    __device__ __forceinline__ void mfma(v4i a, v4i b) { v = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, v, 0, 0, 0); }
    __device__ __forceinline__ v4i quad(int) const { return v; }  // channels 4 (lane / 16) .. + 3
};

// TURN: long rows of a filter in the reference layout.  Loaded as operands, where neighbouring lanes hold different rows, 16 bytes per
// lane take the address path 64 clocks instead of the 16 of a contiguous kilobyte, and that path is what the kernel is then bound by.
// Here an instruction loads 128 bytes of each of eight rows, and LDS that only this wave uses turns them into operands (no barrier, but
// see lds_between_lanes).  A stage costs its LDS round trip, so short pieces do not take it: see ks_turns.
template <int PIN, int S, int MT, int W, bool PW, bool TURN, class Form>
__device__ __forceinline__ void ks_run(const Form& form) {
    constexpr int ROWS = S / 4;           // channel quads of a block
    constexpr int PARTS = S == 32 ? 4 : 1;  // a block's quads over its pixels, 64 at a time
    constexpr int ROWP = ks_row(S), WP = ks_wave_vecs(S, MT, TURN);  // vectors per row, per wave
    constexpr int CH = S == 32 ? 1 : 2;   // 32-byte chunks per step
    constexpr int AHEAD = ks_ahead(S, MT);
    extern __shared__ __attribute__((aligned(16))) v4i red[];
    // Every argument on the way to the operands in one batch of scalar loads (left alone, the compiler asks for them where they
    // are first used, behind the early exit: a second round trip), and one word of each line that the epilogue reads.
    const auto a = form.template open<PIN, S, MT, W>();
    if constexpr (!Form::WIRE) {
        asm volatile("" ::"s"(a.src), "s"(a.flt), "s"(a.bias), "s"(a.z), "s"(a.src_bytes), "s"(a.flt_bytes), "s"(a.OHW), "s"(a.OW), "s"(a.IW),
                     "s"(a.IH), "s"(a.sh), "s"(a.sw), "s"(a.ph), "s"(a.pw), "s"(a.OC), "s"(a.M), "s"(a.src_sn), "s"(a.src_scb),
                     "s"(a.flt_rstride), "s"(a.flt_kstride), "s"(a.tiles_m), "s"(a.tiles_n), "s"(a.by_m), "s"(a.KC));
        asm volatile("" ::"s"(a.steps), "s"(a.per_wave), "s"(a.extra), "s"(a.div_tile.m), "s"(a.div_tile.s1), "s"(a.div_tile.s2),
                     "s"(a.div_ohw.m), "s"(a.div_ohw.s1), "s"(a.div_ohw.s2), "s"(a.div_ow.m), "s"(a.div_ow.s1), "s"(a.div_ow.s2),
                     "s"(a.log_pout), "s"(a.has_bias), "s"(a.epi.s_b), "s"(a.epi.lin_lo));
        if (!PW)
            asm volatile("" ::"s"(a.div_t.m), "s"(a.div_t.s1), "s"(a.div_t.s2), "s"(a.div_fw.m), "s"(a.div_fw.s1), "s"(a.div_fw.s2), "s"(a.T),
                         "s"(a.FW), "s"(a.FH));
    }
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int ls = lane & (S - 1), lk = lane / S;

    // Workgroup b runs on XCD b % 8.  Layers with eight and more channel tiles give each XCD channel tiles of its own (the
    // filter, the larger operand there, enters one L2 only); the others give each XCD a contiguous run of pixels.
    int tm, tn;
    {
        const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
        if (a.by_m) {
            const int r = (int)fdiv_u(i, a.div_tile);
            tm = r * 8 + x;
            tn = i - r * a.tiles_n;
            if (tm >= a.tiles_m) return;
        } else {
            const int per = (a.tiles_n + 7) >> 3, r = (int)fdiv_u(i, a.div_tile);
            tm = i - r * a.tiles_m;
            tn = x * per + r;
            if (tn >= a.tiles_n) return;
        }
    }
    const int oc0 = tm * MT * S, px0 = tn * S;
    const __amdgpu_buffer_rsrc_t rs_src = make_rsrc(a.src, a.src_bytes);
    const __amdgpu_buffer_rsrc_t rs_flt = make_rsrc(a.flt, a.flt_bytes);

    // this wave's piece of the reduction, in steps
    const int k0 = wave * a.per_wave + (wave < a.extra ? wave : a.extra), k1 = k0 + a.per_wave + (wave < a.extra ? 1 : 0);

    KEntry* tab = reinterpret_cast<KEntry*>(red + W * WP);
    if (PIN == 4 && !PW) {
        for (int u = t; u < a.steps * CH * 8; u += W * 64) {
            const uint32_t cb = fdiv(u, a.div_t), tap = u - cb * a.T, fh = fdiv(tap, a.div_fw), fw = tap - fh * a.FW;
            tab[u] = u < a.entries ? KEntry{(int)cb * a.src_scb + ((int)fh * a.IW + (int)fw) * 4, (int)(fh | fw << 16)}
                                   : KEntry{0, 0x4000};
        }
    }

    int arow[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = oc0 + i * S + ls;
        arow[i] = row < a.OC ? row * a.flt_rstride + (S == 32 ? lk * 16 : (lk >> 1) * a.flt_kstride + (lk & 1) * 16) : SENT;
    }
    int pix, ih0, iw0;
    {
        const int m = px0 + ls;
        const bool ok = m < a.M;
        const uint32_t mm = ok ? m : 0;
        const uint32_t n = fdiv(mm, a.div_ohw), rem = mm - n * a.OHW;
        const uint32_t oh = fdiv(rem, a.div_ow), ow = rem - oh * a.OW;
        ih0 = ok ? (int)oh * a.sh - a.ph : -0x10000;  // no tap of a pixel past the last one lies inside
        iw0 = (int)ow * a.sw - a.pw;
        pix = (int)n * a.src_sn + ((int)oh * a.sh - a.ph) * a.IW * PIN + iw0 * PIN + (PIN == 32 ? (lk & 1) * 16 : 0);
        if (PW && !ok) pix = SENT;
    }
    if (PIN == 4 && !PW) __syncthreads();

    // load cursor: step kc; for 32-packed inputs and one chunk per step its channel block and tap (wave-uniform)
    int kc = k0, cb = 0, fh = 0, fw = 0;
    if (PIN == 32 && !PW && S == 32) {
        cb = (int)fdiv_u(k0, a.div_t);
        const int tap = k0 - cb * a.T;
        fh = (int)fdiv_u(tap, a.div_fw);
        fw = tap - fh * a.FW;
    }
    // Operands of the next step.  Past the wave's piece every lane is out of the buffers' range: zeros, no memory access
    // (an unconditional load keeps the number of loads in flight known to the compiler, and with it the waits short).
    // A 4-packed row may end inside its last chunk, so there the whole offset stands where the descriptor checks it.
    auto load_filter = [&](v4i (&fa)[MT]) __attribute__((always_inline)) {
        const bool in = kc < k1;
        const int kf = kc * CH * a.flt_kstride;
        const bool half_in = S == 32 || kc * 2 + (lk >> 1) < a.KC;  // an odd number of chunks: no second one in the last step
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const bool ok = in && half_in && arow[i] != SENT;
            fa[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, ok ? arow[i] + kf : SENT, 0, 0);
        }
    };
    auto load_pixels = [&](v4i& fb) __attribute__((always_inline)) {
        const bool in = kc < k1;
        const bool half_in = S == 32 || kc * 2 + (lk >> 1) < a.KC;
        if (PIN == 32 && PW) {
            const int c = S == 32 ? 0 : (lk >> 1) * a.src_scb;
            fb = __builtin_amdgcn_raw_buffer_load_b128(rs_src, in && half_in && pix != SENT ? pix + c : SENT, (in ? kc : 0) * CH * a.src_scb, 0);
        } else if (PIN == 32 && S == 32) {
            const bool ok = in && (unsigned)(ih0 + fh) < (unsigned)a.IH && (unsigned)(iw0 + fw) < (unsigned)a.IW;
            // (not the block's offset as the instruction's scalar one: where the compiler keeps the cursor in a vector register, that
            // makes a loop of the load)
            fb = __builtin_amdgcn_raw_buffer_load_b128(rs_src, ok ? pix + (fh * a.IW + fw) * 32 + cb * a.src_scb : SENT, 0, 0);
        } else if (PIN == 32) {
            const uint32_t c = kc * 2 + (lk >> 1), b = fdiv(c, a.div_t), tap = c - b * a.T, h = fdiv(tap, a.div_fw), w = tap - h * a.FW;
            const bool ok = in && half_in && (unsigned)(ih0 + (int)h) < (unsigned)a.IH && (unsigned)(iw0 + (int)w) < (unsigned)a.IW;
            fb = __builtin_amdgcn_raw_buffer_load_b128(rs_src, ok ? pix + ((int)h * a.IW + (int)w) * 32 + (int)b * a.src_scb : SENT, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int u = kc * CH * 8 + lk * 4 + i;
                if (PW) {
                    fb[i] = __builtin_amdgcn_raw_buffer_load_b32(rs_src, in && u < a.entries && pix != SENT ? pix + u * a.src_scb : SENT, 0, 0);
                } else {
                    const KEntry e = tab[in ? u : 0];
                    const bool ok = in && (unsigned)(ih0 + (e.fhfw & 0xffff)) < (unsigned)a.IH &&
                                    (unsigned)(iw0 + (e.fhfw >> 16)) < (unsigned)a.IW;
                    fb[i] = __builtin_amdgcn_raw_buffer_load_b32(rs_src, ok ? pix + e.off : SENT, 0, 0);
                }
            }
        }
        ++kc;
        if (PIN == 32 && !PW && S == 32) {
            if (++fw == a.FW) {
                fw = 0;
                if (++fh == a.FH) {
                    fh = 0;
                    ++cb;
                }
            }
        }
    };

    KsAcc<S> acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i].clear();

    // The partial sums of a block are dealt out over the waves in parts of 64 quads: by rows where the destination keeps
    // four channels of a pixel together (consecutive pixels are contiguous), by pixels where it keeps 32.
    const __amdgpu_buffer_rsrc_t rs_z = make_rsrc(a.z, a.z_bytes);
    const __amdgpu_buffer_rsrc_t rs_bias = make_rsrc(a.bias, a.has_bias ? a.OC * 4 : 0);
    const __amdgpu_buffer_rsrc_t rs_dst = make_rsrc(a.dst, a.dst_bytes);
    int d_off = SENT, z_off = SENT, at_red = 0, left = 0;
    v4i bv = {0, 0, 0, 0};
    uint32_t zw = 0;
    auto fetch = [&](int u) __attribute__((always_inline)) {
        const int i = u / PARTS, part = u % PARTS;
        const int row = a.log_pout == 5 ? lane % ROWS : part * (64 / S) + lk;  // channels 4 row .. + 3 of the block
        const int px = a.log_pout == 5 ? part * (64 / ROWS) + lane / ROWS : ls;
        at_red = (i * ROWS + row) * ROWP + px;
        const int oc4 = oc0 + i * S + row * 4, m = px0 + px;
        const bool ok = m < a.M && oc4 < a.OC && u < MT * PARTS;
        const uint32_t mm = m < a.M ? m : 0;
        const uint32_t n = fdiv(mm, a.div_ohw), rem = mm - n * a.OHW;
        const int at = (oc4 >> a.log_pout) * a.dst_scb + ((int)rem << a.log_pout) + (oc4 & ((1 << a.log_pout) - 1));
        d_off = ok ? (int)n * a.dst_sn + at : SENT;
        z_off = ok ? (int)n * a.z_sn + at : SENT;
        bv = __builtin_amdgcn_raw_buffer_load_b128(rs_bias, ok ? oc4 * 4 : SENT, 0, 0);
        zw = 0;
        if (a.log_pout == 0) {
            // planar: four channels of a pixel lie OHW apart
            left = ok ? a.OC - oc4 : 0;
            if (a.epi.has_z)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < left) zw |= (uint32_t)(uint8_t)a.z[z_off + r * a.OHW] << (8 * r);
        } else if (a.epi.has_z && !a.dst_s32) zw = __builtin_amdgcn_raw_buffer_load_b32(rs_z, z_off, 0, 0);
    };

    if constexpr (TURN) {
        // A stage is 128 bytes of every row: load j of a wave holds rows 8 j + lane / 8.  In LDS a row's 16-byte pieces change places
        // by its number, so that neither the writes (a row by eight lanes) nor the reads (a piece of sixteen rows) meet on a bank.
        constexpr int LOADS = MT * S / 8, STEPS = S == 32 ? 4 : 2, STEP_BYTES = 128 / STEPS;
        v4i* mine = red + wave * WP;
        int off[LOADS], at_w[LOADS], at_r[MT];
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int row = j * 8 + (lane >> 3), piece = lane & 7;
            off[j] = oc0 + row < a.OC ? (oc0 + row) * a.flt_rstride + piece * 16 : SENT;
            at_w[j] = row * 8 + (piece ^ ((row >> 1) & 7));
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) at_r[i] = (i * S + ls) * 8;
        const int turn = (ls >> 1) & 7;
        v4i xf[2][LOADS], fb[2][STEPS];
        int kf = k0, left = k1 - k0;
        const int tail = a.flt_rstride - (lane & 7) * 16;  // bytes of the row from this lane's piece on
        auto load_f = [&](int buf) __attribute__((always_inline)) {
            // (nothing past the wave's piece of the reduction, whose last stage may be cut short, or past the row's end)
            const bool in = kf * STEP_BYTES + (lane & 7) * 16 < k1 * STEP_BYTES && kf * STEP_BYTES < tail;
#pragma unroll
            for (int j = 0; j < LOADS; ++j) xf[buf][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_flt, in && off[j] != SENT ? off[j] + kf * STEP_BYTES : SENT, 0, 0);
            kf += STEPS;
        };
        auto load_p = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < STEPS; ++b) load_pixels(fb[buf][b]);
        };
        auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < LOADS; ++j) mine[at_w[j]] = xf[buf][j];
            lds_between_lanes();
            load_f(buf);
            v4i fa[STEPS][MT];
#pragma unroll
            for (int b = 0; b < STEPS; ++b)
#pragma unroll
                for (int i = 0; i < MT; ++i) fa[b][i] = mine[at_r[i] + ((b * (8 / STEPS) + lk) ^ turn)];
            lds_between_lanes();  // (the next stage, and the sums behind the last, overwrite what is read here)
#pragma unroll
            for (int b = 0; b < STEPS; ++b)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[i].mfma(fa[b][i], fb[buf][b]);  // (steps past the piece: zeros)
            load_p(buf);
        };
        if (left > 0) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                load_f(b);
                load_p(b);
            }
        }
        fetch(wave);
        for (; left > 0; left -= 2 * STEPS) {
            stage(0);
            if (left <= STEPS) break;
            stage(1);
        }
    } else {
        v4i fa[AHEAD][MT], fb[AHEAD];
        if (k0 < k1)  // (waves beyond the number of steps have nothing to add)
#pragma unroll
            for (int g = 0; g < AHEAD; ++g) {
                load_filter(fa[g]);
                load_pixels(fb[g]);
            }
        fetch(wave);  // behind the first operands, so that bias and residual cost no round trip of their own
        auto multiply = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i].mfma(fa[g][i], fb[g]);
        };
        int left = k1 - k0;
        for (; left > AHEAD; left -= AHEAD) {
#pragma unroll
            for (int g = 0; g < AHEAD; ++g) {
                multiply(g);
                load_filter(fa[g]);
                load_pixels(fb[g]);
            }
        }
#pragma unroll
        for (int g = 0; g < AHEAD; ++g)
            if (g < left) multiply(g);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int q = 0; q < PARTS; ++q) red[wave * WP + (i * ROWS + q * (64 / S) + lk) * ROWP + ls] = acc[i].quad(q);
    __syncthreads();
    for (int u = wave; u < MT * PARTS; u += W) {
        if (u != wave) fetch(u);
        v4i s = bv;
#pragma unroll
        for (int w = 0; w < W; ++w) s += red[w * WP + at_red];
        if (a.dst_s32) {
            // four elements of an int32 dst: element offset d_off, a residual of the same type and its own batch stride
            if (a.epi.has_z || a.epi.nonline != NL_IDENTITY) {
                v4i zv = {0, 0, 0, 0};
                if (a.epi.has_z) zv = __builtin_amdgcn_raw_buffer_load_b128(rs_z, z_off != SENT ? z_off * 4 : SENT, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) s[r] = requant_s32_exact(s[r], a.epi.has_z != 0, zv[r], a.epi);
            }
            __builtin_amdgcn_raw_buffer_store_b128(s, rs_dst, d_off != SENT ? d_off * 4 : SENT, 0, 0);
        } else {
            const uint32_t o = requant4(s[0], s[1], s[2], s[3], zw, a.epi);
            if (a.log_pout == 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < left) a.dst[d_off + r * a.OHW] = (int8_t)(o >> (8 * r));
            } else {
                __builtin_amdgcn_raw_buffer_store_b32(o, rs_dst, d_off, 0, 0);
            }
        }
    }
}

template <int PIN, int S, int MT, int W, bool PW>
__global__ __launch_bounds__(W * 64) void ks_kernel(KsWire a) {
    ks_run<PIN, S, MT, W, PW, false>(a);
}
template <int PIN, int S, int MT, int W, bool PW>
__global__ __launch_bounds__(W * 64) void ks_kernel(KsWide a) {
    ks_run<PIN, S, MT, W, PW, false>(a);
}
template <int PIN, int S, int MT, int W, bool PW>
__global__ __launch_bounds__(W * 64) void ks_turn_kernel(KsWire a) {
    ks_run<PIN, S, MT, W, PW, true>(a);
}
template <int PIN, int S, int MT, int W, bool PW>
__global__ __launch_bounds__(W * 64) void ks_turn_kernel(KsWide a) {
    ks_run<PIN, S, MT, W, PW, true>(a);
}

struct KsCfg {
    int pin, s, mt, waves;
    const char* name;
};
constexpr KsCfg kKs[] = {
        {32, 16, 1, 8, "v2_ks_16x16w8"}, {32, 16, 1, 4, "v2_ks_16x16w4"}, {32, 32, 1, 8, "v2_ks_32x32w8"},
        {32, 32, 1, 4, "v2_ks_32x32w4"}, {32, 32, 2, 8, "v2_ks_64x32w8"}, {32, 32, 2, 4, "v2_ks_64x32w4"},
        {4, 16, 1, 8, "ks4_16x16w8"},    {4, 16, 1, 4, "ks4_16x16w4"},    {4, 32, 1, 8, "ks4_32x32w8"},
        {4, 32, 1, 4, "ks4_32x32w4"},    {4, 32, 2, 8, "ks4_64x32w8"},    {4, 32, 2, 4, "ks4_64x32w4"}};
constexpr int kKsCount = sizeof(kKs) / sizeof(kKs[0]);

// Whether the filter goes through LDS (see ks_run): rows in the reference layout, and pieces of them from which on it pays.  Graph replays,
// new / old by bytes of a row per wave, means over drawn layers: 64x32w8 256 to 383: 1.02 .. 1.07, 384 to 511: 0.93, 512 to 767: 0.86, from
// 768 on 0.67 .. 0.84 (3x3 over 864 channels, 192 tiles: 14.5 -> 12.4 us); 16x16w4 256 to 511: 1.04 .. 1.14, 512 to 767: 0.99, from 768
// on 0.89; 16x16w8 256 to 383: 1.07, 384 to 767: 0.93 .. 1.0, from 768 on 0.86.  The 32 x 32 tile of four waves has twice the
// workgroups to a CU that cover its loads for each other: 1.16 to 1.31 with it at any length, and 4-packed rows 1.0 to 1.25.  Nor the
// 64 x 32 tile with half of its rows missing (32 channels: 1.12 .. 1.19).
constexpr bool ks_can_turn(int pin, int s, int mt, int waves) { return pin == 32 && (s == 16 || waves == 8); }
bool ks_turns(const IgemmArgs& a, const KsCfg& c) {
    return ks_can_turn(c.pin, c.s, c.mt, c.waves) && (c.mt == 1 || a.OC > 32) && a.flt_rstride == a.kbytes && a.kbytes >= (c.s == 32 ? 384 : 640) * c.waves;
}
int ks_lds(const IgemmArgs& a, const KsCfg& c, bool pw) {
    return c.waves * ks_wave_vecs(c.s, c.mt, ks_turns(a, c)) * 16 + (c.pin == 4 && !pw ? (a.KC + 1) * 8 * 8 : 0);
}

template <int PIN, int S, int MT, int W, bool PW, bool TURN, class Form>
int launch_ks_form(hipStream_t st, const Form& form, unsigned grid, int lds) {
    void (*kern)(Form);
    if constexpr (TURN) kern = ks_turn_kernel<PIN, S, MT, W, PW>;
    else kern = ks_kernel<PIN, S, MT, W, PW>;
    static std::atomic<int> max_lds_set{0};
    if (lds > max_lds_set.load(std::memory_order_relaxed)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
        max_lds_set.store(160 * 1024, std::memory_order_relaxed);
    }
    return launch_kernel(kern, dim3(grid), dim3(W * 64), lds, st, form);
}

template <int PIN, int S, int MT, int W, bool PW>
int launch_ks(hipStream_t st, const KsArgs<FastDiv>& k, uint32_t n, int lds, bool turn) {
    const int64_t grid = igemm5_workgroups(k.tiles_m, k.tiles_n);
    if (grid > 0x7fffffff) return (int)hipErrorInvalidValue;
    KsWire wire;
    // Windowed 32 x 32 tiles up to two workgroups per CU: beyond, opening the wire costs more than the launch gains.  Graph replays, wire /
    // wide: to 256 workgroups 1.01 (0.04 us of 4, where a launch that is waited for gains 0.6), to 512 1.02, beyond 1.035 .. 1.04 (0.27 us of 6
    // to 11; 3x3 160 -> 32 at 90 x 15, batch 12, 512 workgroups: 5.16 us wide, 5.73 so).  Pointwise ones take 3 to 4 us at any number, and one
    // image of ResNet-50 0.8 % longer with them wide from 256 on.  The others: 16 x 16 0.98 .. 1.0, 64 x 32 1.0 .. 1.01.
    const bool fits = (PW || S != 32 || MT != 1 || grid <= 512) && wire.pack<PIN, S, MT, W>(k, n);
    if constexpr (ks_can_turn(PIN, S, MT, W))
        if (turn) return fits ? launch_ks_form<PIN, S, MT, W, PW, true>(st, wire, (unsigned)grid, lds) : launch_ks_form<PIN, S, MT, W, PW, true>(st, KsWide{k}, (unsigned)grid, lds);
    return fits ? launch_ks_form<PIN, S, MT, W, PW, false>(st, wire, (unsigned)grid, lds) : launch_ks_form<PIN, S, MT, W, PW, false>(st, KsWide{k}, (unsigned)grid, lds);
}

}  // namespace

int igemm5_num_cfgs() { return kKsCount; }
const char* igemm5_cfg_name(int cfg) { return kKs[cfg].name; }

// The tile for a 4-packed problem, or -1 where the staged tiles are the better ones (32-packed ones go by prices, conv_igemm.hip).  The
// line between them is the number of workgroups a tile would make: up to about one per CU this kernel hides what the staged tiles wait
// for, beyond that its operand traffic costs more.  (At batch 1 the layers of ResNet-50 sum to 178 us instead of 255 with these tiles, 3x3
// over 512 channels at 7 x 7: 11.0 -> 4.2 us; over 256 at 14 x 14: 7.2 -> 3.4; the pointwise layers of MobileNetV2 to 115 instead of 140.)
static int ks_id(int pin, int s, int mt, int waves) {
    for (int i = 0; i < kKsCount; ++i)
        if (kKs[i].pin == pin && kKs[i].s == s && kKs[i].mt == mt && kKs[i].waves == waves) return i;
    return -1;
}
int igemm5_pick(const IgemmArgs& a, int pin, int pout) {
    auto tiles = [&](int bm, int bn) { return (int64_t)((a.OC + bm - 1) / bm) * ((a.M + bn - 1) / bn); };
    if (pin != 4) return -1;
    const int64_t g16 = tiles(16, 16), g32 = tiles(32, 32), g64 = tiles(64, 32);
    const int K = a.kbytes;
    const bool window = a.T > 1;
    int id = -1;
    if (window) {
        // Against the 4-packed patch tiles: they pay a fixed price per 32 input channels, this kernel one per pixel and tap.
        // Graph replays of every tile, us, ks against patch: 128 -> 128 at 28 x 28, batch 1 (g16 = 392): 5.4 / 5.9, batch 4:
        // 6.8 / 6.0; 232 -> 72 at 40 x 16, stride 2, batch 12: 8.9 / 10.8; 5x5 64 -> 64 at 32 x 32, batch 8: 8.0 / 8.9;
        // 512 -> 512 at 7 x 7, batch 16: 16.1 / 17.9.
        // 3x3 over at most 32 channels: the patch tile that has one stage too is ahead at any number of pixels (32 -> 20, 1980 pixels:
        // 3.75 us / 4.5; 24 -> 12, 112 pixels: 3.5 / 4.1); over 64 the two meet at about 200 tiles of 16 x 16.
        if (K <= 288 && patch4_one_stage(a, pin, pout)) return -1;
        const bool patch = patch4_can_run(a, pin, pout, 0), few_taps = a.T <= 9 && a.sh == 1 && a.sw == 1;
        if (K >= 128 && g16 <= 300) id = ks_id(4, 16, 1, K >= 1024 ? 8 : 4);
        else if (K >= 1024 && g16 <= 450) id = ks_id(4, 16, 1, 4);
        else if (K >= 1024 && g32 <= (patch && few_taps && K < 4096 ? 200 : 256)) id = ks_id(4, 32, 1, 8);
        else if (g64 <= 256 && (!patch || a.T > 9 || K >= 4096)) id = ks_id(4, 32, 2, 8);
    } else {
        if (K >= 128 && g16 <= 300) id = ks_id(4, 16, 1, K >= 1024 ? 8 : 4);
        else if (g64 <= 256) id = ks_id(4, 32, 2, K <= 192 ? 8 : 4);
    }
    return id >= 0 && igemm5_can_run(a, pin, pout, id) ? id : -1;
}

bool igemm5_can_run(const IgemmArgs& a, int pin, int pout, int cfg) {
    if (cfg < 0 || cfg >= kKsCount || kKs[cfg].pin != pin || a.groups != 1 || (pout != 1 && pout != 4 && pout != 32)) return false;
    if (pout == 1 && (a.dst_f32 || a.bias_full || !a.epi.fast)) return false;  // planar: the fast int8 forms
    // of the general epilogue only the int32 result, below 2 GiB
    if (a.general && !(a.dst_s32 && !a.bias_full && a.dst_bytes < (1u << 29) && a.z_bytes < (1u << 29))) return false;
    const bool pw = a.T == 1 && a.ph == 0 && a.pw == 0;
    return ks_lds(a, kKs[cfg], pw) <= 160 * 1024;
}

int launch_igemm5(hipStream_t st, const IgemmArgs& a, int pin, int pout, int cfg) {
    if (!igemm5_can_run(a, pin, pout, cfg)) return (int)hipErrorInvalidConfiguration;
    const KsCfg& c = kKs[cfg];
    KsArgs<FastDiv> k;
    k.src = a.src; k.flt = a.flt; k.bias = a.bias; k.z = a.z; k.dst = a.dst;
    k.src_bytes = a.src_bytes; k.flt_bytes = a.flt_bytes; k.z_bytes = a.z_bytes; k.dst_bytes = a.dst_bytes;
    k.IH = a.IH; k.IW = a.IW; k.OHW = a.OHW; k.OW = a.OW; k.FW = a.FW; k.T = a.T;
    k.sh = a.sh; k.sw = a.sw; k.ph = a.ph; k.pw = a.pw;
    k.OC = a.OC; k.M = a.M; k.KC = a.KC; k.entries = a.entries;
    k.src_sn = a.src_sn; k.src_scb = a.src_scb; k.dst_sn = a.dst_sn; k.dst_scb = a.dst_scb; k.z_sn = a.z_sn;
    k.flt_rstride = a.flt_rstride; k.flt_kstride = a.flt_kstride;
    k.tiles_m = (a.OC + c.s * c.mt - 1) / (c.s * c.mt);
    k.tiles_n = (a.M + c.s - 1) / c.s;
    k.by_m = k.tiles_m >= 8;
    k.div_tile = make_fastdiv(k.by_m ? k.tiles_n : k.tiles_m);
    k.FH = a.FH;
    k.steps = c.s == 32 ? a.KC : (a.KC + 1) / 2;
    k.per_wave = k.steps / c.waves;
    k.extra = k.steps % c.waves;
    k.log_pout = pout == 32 ? 5 : pout == 4 ? 2 : 0;
    k.has_bias = a.has_bias;
    k.dst_s32 = a.dst_s32;
    if (a.dst_s32) {  // bytes of int32 tensors
        k.dst_bytes = a.dst_bytes * 4;
        k.z_bytes = a.z_bytes * 4;
    }
    k.div_ohw = a.div_ohw; k.div_ow = a.div_ow; k.div_t = a.div_t; k.div_fw = a.div_fw;
    k.epi = a.epi;
    const bool pw = a.T == 1 && a.ph == 0 && a.pw == 0;
    const int lds = ks_lds(a, c, pw);
    const bool turn = ks_turns(a, c);
#define MI355_KS(PIN, S, MT) \
    (pw ? c.waves == 8 ? launch_ks<PIN, S, MT, 8, true>(st, k, a.NB, lds, turn) : launch_ks<PIN, S, MT, 4, true>(st, k, a.NB, lds, turn) \
        : c.waves == 8 ? launch_ks<PIN, S, MT, 8, false>(st, k, a.NB, lds, turn) : launch_ks<PIN, S, MT, 4, false>(st, k, a.NB, lds, turn))
    if (pin == 32) {
        if (c.s == 16) return MI355_KS(32, 16, 1);
        return c.mt == 1 ? MI355_KS(32, 32, 1) : MI355_KS(32, 32, 2);
    }
    if (c.s == 16) return MI355_KS(4, 16, 1);
    return c.mt == 1 ? MI355_KS(4, 32, 1) : MI355_KS(4, 32, 2);
#undef MI355_KS
}

}  // namespace mi355
