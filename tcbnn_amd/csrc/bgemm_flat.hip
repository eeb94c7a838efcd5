// FP4 matrix-core kernel of the bit convolutions and bit products whose batch is not a multiple of 32 images wide or
// whose whole work is small: the columns of the product are (pixel, image) pairs numbered through,
// column = pixel * batch + image, so a 32-column MFMA tile is full whatever the batch is.  (The kernels that give a
// tile 32 images of ONE pixel multiply 32 / batch times too much at a batch below 32.)
//
//   tile      = MT x 32 columns by NT x 32 output channels, one wave; with 2x2 OR-pooling a column is a window, and its
//               four pixels are either the MT = 4 column tiles (the window is reduced in the lane's own registers) or,
//               where that leaves too few waves, four groups of 8 lanes of one tile;
//   K         = the words of the filter row, (tap, input word) numbered through.  A group is 8 words: lane half h owns
//               words 8g + 4h .. + 3, one 128-bit load per channel tile straight from the packed filter rows, and the
//               matching four activation words; step i multiplies word 8g + 4h + i.  Cin = 32 or 96 costs no padding;
//   borders   : a lane's invalid taps are bits of a mask; such an activation is not loaded (its offset lies outside the
//               buffer) and enters as FP4 zero, the reference's "exclude" rule (kernel.cuh:752-768).  Where an
//               activation word of the group lies relative to the column's first tap, and which tap it belongs to, is
//               a table in LDS, filled once per workgroup;
//   small work: K is split over the waves of a workgroup (up to 8) so that a launch of few tiles still spreads over
//               the machine; the partial sums, exact integers, meet in LDS.
//
// The finish of a tile stays in fp32 (whole numbers): sums start from minus what the pad bits add, a bit is the sign of sum -
// threshold shifted in, and what lies past the last channel is masked once.  Small launches end with one wave's finish, and
// with conversions, compares and selects per value it was a fifth of their time: ResNet-18 at batch 1 / 8 113.1 -> 105.3 / 117.4 ->
// 112.3 us a pass, VGG-16 at batch 8 212 -> 180, AlexNet at batch 150 175 -> 168.  (Shared by two waves instead, eight channels of a
// lane each: 1 % slower than by one.)
//
// What bounds it, with counters (from before that): the small launches latency, one or two memory round trips and the launch itself (3x3
// layers at batch 8, 5.6-6.3 us: waves wait for memory 52-64 % of their time, VALU busy 20-33 %, matrix cores 4 %).  The larger ones
// instruction issue: expanding the operands takes 7 VALU instructions per fragment, plus 5 per column tile and step for
// address and border, against 32 cycles per MFMA (AlexNet's 5x5 layer at batch 256, 50 us: VALU 63 %, matrix cores 27 %, of
// the same issue slots).
#include <algorithm>
#include <initializer_list>
#include <utility>

#include "common.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

using namespace mfma;

typedef float v4f __attribute__((ext_vector_type(4)));

// what happens to the sums
constexpr int FM_BITS = 0;    // threshold, packed bits
constexpr int FM_RES = 1;     // residual injected from a source of the same size and / or saved; threshold
constexpr int FM_RESPOOL = 2; // residual injected as the 2x2 maximum of a source twice the size
constexpr int FM_RAW = 3;     // int32 dot products
// 2x2 OR-pooling: none; the window's four pixels in lanes 8 apart of one column tile; in the four column tiles of a wave
constexpr int FW_NONE = 0, FW_LANES = 1, FW_TILES = 2;

constexpr int kTapNone = 31;  // tap number of a word past K: its mask bit is always "invalid"
constexpr int kMaxWords = 4096;

// Everything the kernel reads, and nothing else: it is fetched in one go at the start (see fetch_now).
struct FlatArgs {
    const uint32_t* act;
    const uint32_t* wgt;
    const float* bn;
    const int32_t* res_in;
    uint32_t* out_bits;
    int32_t* out_i32;
    int32_t* res_out;
    long long bits_pix_stride, raw_pix_stride, raw_b_stride;
    FastDiv by_batch, by_row, by_cw, by_s, by_groups;  // columns per item, items per row, words per tap, taps per filter row
    int B, cw, H, W, R, S, stride_h, stride_w, pad_h, pad_w, PW, N, k_tap, nan_bit, bits_row_words;
    int res_in_ch, res_out_fmt, res_lim;
    int cols, n_groups, kw_tot, groups, per_slice, slices;
    int total;         // tiles (column groups x channel groups) of the launch
    int wgs, per_xcd;  // workgroups with work, and how many of them an XCD gets
    unsigned act_bytes, wgt_bytes;
};

constexpr int raw_pitch(int nt) { return 32 * nt + 4; }  // words; an odd multiple of 4: conflict-free both ways
constexpr int max_waves(int mt, int nt) { return mt * nt == 1 ? 8 : 4; }
// groups of operand words in flight per wave (registers)
constexpr int ring_depth(int mt, int nt, int fm) { return mt * nt >= 8 ? 1 : (mt * nt >= 4 || fm == FM_RESPOOL ? 2 : 4); }

template <typename T>
__device__ __forceinline__ void fetch_one(T v) {
    asm volatile("" ::"s"(v));
}

// Sixteen sums less their thresholds, the signs shifted in (MSB first).  Lane l of each row of 16 holds threshold l of its half: one
// request for all of them, and a subtraction takes its threshold by DPP.  (Every lane of the wave is active here.)
template <int V>
__device__ __forceinline__ float row_lane(float t) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(t), 0x150 + V, 0xf, 0xf, true));  // row_newbcast:V
}
template <int... V>
__device__ __forceinline__ uint32_t signs(const float (&sum)[16], float t, std::integer_sequence<int, V...>) {
    uint32_t hw = 0;
    ((hw = __builtin_amdgcn_alignbit(hw, __float_as_uint(sum[V] - row_lane<V>(t)), 31)), ...);
    return hw;
}

template <int MT, int NT, int FM, int RF, int WIN>
__global__ __launch_bounds__(64 * max_waves(MT, NT)) __attribute__((amdgpu_waves_per_eu(MT * NT == 1 ? (FM == FM_RESPOOL ? 3 : 4) : 2))) void
bgemm_flat_f4_kernel(const FlatArgs p) {
    static_assert(WIN == FW_NONE || (FM == FM_BITS && MT == (WIN == FW_TILES ? 4 : 1)), "see FW_*");
    static_assert(FM != FM_RESPOOL || MT == 1, "four source pixels per column");
    constexpr bool kRes = FM == FM_RES || FM == FM_RESPOOL;
    constexpr int D = ring_depth(MT, NT, FM);
    // Left to the compiler, an argument is a scalar load right before its first use: four round trips one after the
    // other before the first activation is asked for.
    auto fetch_now = [](auto... v) __attribute__((always_inline)) { (void)std::initializer_list<int>{(fetch_one(v), 0)...}; };
    fetch_now(p.act, p.wgt, p.by_batch.mul, p.by_row.mul, p.by_cw.mul, p.by_s.mul, p.by_groups.mul, p.B, p.cw, p.H, p.W, p.R,
              p.S, p.stride_h, p.stride_w, p.pad_h, p.pad_w, p.PW, p.N, p.k_tap, p.cols, p.kw_tot, p.groups, p.slices, p.wgs,
              p.act_bytes, p.wgt_bytes);
    if constexpr (FM == FM_RAW) fetch_now(p.out_i32, p.raw_pix_stride, p.raw_b_stride);
    else fetch_now(p.bn, p.out_bits, p.bits_pix_stride, p.nan_bit, p.bits_row_words);
    if constexpr (kRes) fetch_now(p.res_in, p.res_out, p.res_in_ch, p.res_out_fmt, p.res_lim);
    extern __shared__ v4i lds_dyn[];
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int waves = blockDim.x >> 6;
    // Tiles are dealt so that each XCD (workgroups go to the 8 of them in turn) gets a contiguous run: neighbouring
    // pixels share activation rows, and the channel groups of a column tile all of them.
    const int per_wg = p.slices > 1 ? 1 : waves;
    const int wg = (int)(blockIdx.x & 7) * p.per_xcd + (int)(blockIdx.x >> 3);
    const int slice = p.slices > 1 ? wave : 0;
    const int tile = p.slices > 1 ? wg : wg * waves + wave;
    const bool live = wg < p.wgs && tile < p.total;  // (uniform per wave)
    const int ct = live ? (int)div_by((unsigned)tile, p.by_groups) : 0, ng = live ? tile - ct * p.n_groups : 0;
    const int n0 = ng * (32 * NT);

    v4f* red = reinterpret_cast<v4f*>(lds_dyn);                                   // [slices - 1][MT * NT][4][64]
    int* raw_area = reinterpret_cast<int*>(red + (size_t)(p.slices - 1) * MT * NT * 256);
    constexpr int kRawWords = FM == FM_RAW ? 32 * raw_pitch(NT) + 64 : 0;         // per tile of the workgroup
    int2* tab = reinterpret_cast<int2*>(raw_area + per_wg * kRawWords);           // [8 * groups]

    const int g_begin = slice * p.per_slice, g_end = live ? min(p.groups, g_begin + p.per_slice) : 0;

    // ---- weights: lane (j, h) reads words 8g + 4h .. + 3 of its channel's row (past the last row: zeros; past the end
    // of a row: the next row's words, which meet activations that are zero)
    const __amdgpu_buffer_rsrc_t r_wgt =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.wgt), 0, (int)p.wgt_bytes, 0x00020000);
    unsigned wvoff[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
        wvoff[nt] = ((unsigned)(n0 + nt * 32 + row_to_channel(j)) * (unsigned)p.kw_tot + 4u * (unsigned)h) * 4u;
    v4i aw[D][NT];
    auto request_w = [&](int slot, int g) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            aw[slot][nt] = __builtin_amdgcn_raw_buffer_load_b128(r_wgt, (int)wvoff[nt], g * 32, 0);
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (g_begin + d < g_end) request_w(d, g_begin + d);

    // ---- columns
    const unsigned row_b = (unsigned)p.B * 4u, pix_b = (unsigned)p.cw * row_b;
    unsigned base[MT], inval[MT];  // byte offset of the column's first tap (may be "negative"); mask of its invalid taps
    int cpix[WIN == FW_TILES ? 1 : MT], cb[WIN == FW_TILES ? 1 : MT], cy[MT], cx[MT];
    bool cok[WIN == FW_TILES ? 1 : MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        constexpr bool tiles = WIN == FW_TILES;
        const int sub = tiles ? mt : j >> 3;  // pixel of the window
        if (!tiles || mt == 0) {
            const unsigned col = WIN == FW_LANES ? (unsigned)ct * 8u + (unsigned)(j & 7)
                                                 : (unsigned)(tiles ? ct : ct * MT + mt) * 32u + (unsigned)j;
            const unsigned cc = min(col, (unsigned)p.cols - 1u);
            const unsigned item = div_by(cc, p.by_batch);
            cok[mt] = live && col < (unsigned)p.cols;
            cpix[mt] = (int)item;
            cb[mt] = (int)(cc - item * p.by_batch.d);
        }
        const int k = tiles ? 0 : mt;
        const unsigned iy = div_by((unsigned)cpix[k], p.by_row), ix = (unsigned)cpix[k] - iy * p.by_row.d;
        cy[mt] = WIN != FW_NONE ? 2 * (int)iy + (sub >> 1) : (int)iy;
        cx[mt] = WIN != FW_NONE ? 2 * (int)ix + (sub & 1) : (int)ix;
        const int ay0 = cy[mt] * p.stride_h - p.pad_h, ax0 = cx[mt] * p.stride_w - p.pad_w;
        base[mt] = (unsigned)(ay0 * p.W + ax0) * pix_b + (unsigned)cb[k] * 4u;
        // valid taps: rows lo_y .. hi_y, columns lo_x .. hi_x
        const int lo_x = max(0, -ax0), hi_x = min(p.S, p.W - ax0);
        const unsigned run = hi_x > lo_x ? ((1u << hi_x) - 1u) & ~((1u << lo_x) - 1u) : 0u;
        unsigned ok = 0;
        for (int r = 0; r < p.R; ++r)
            if (ay0 + r >= 0 && ay0 + r < p.H) ok |= run << (r * p.S);
        inval[mt] = cok[k] ? ~ok : 0xffffffffu;
    }

    // ---- operands of the epilogue, requested ahead of K
    const bool fin = live && slice == 0;  // (uniform) this wave finishes the tile
    float thr[NT];
    constexpr int NRAW = RF == TCBNN_RES_I12 ? 6 : (RF == TCBNN_RES_I16 ? 8 : 16);
    constexpr int NSRC = FM == FM_RESPOOL ? 4 : 1;
    int rraw[kRes ? MT * NT : 1][NSRC][NRAW];
    if (FM != FM_RAW && fin) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) thr[nt] = p.bn[min(n0 + nt * 32 + 16 * h + (lane & 15), p.N - 1)];
    }
    if constexpr (kRes) {
        if (fin && p.res_lim > 0) {
            const unsigned G = (unsigned)(p.res_in_ch + (int)residual_group_channels(RF) - 1) / (unsigned)residual_group_channels(RF);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int b = cb[mt];
#pragma unroll
                for (int s = 0; s < NSRC; ++s) {
                    const size_t spix = FM == FM_RESPOOL
                                            ? (size_t)(2 * cy[mt] + (s >> 1)) * (size_t)(2 * p.PW) + (size_t)(2 * cx[mt] + (s & 1))
                                            : (size_t)cy[mt] * p.PW + cx[mt];
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const int cbase = n0 + nt * 32 + 16 * h;
                        int* dst = rraw[mt * NT + nt][s];
                        if constexpr (RF == TCBNN_RES_I12) {
                            if (cbase < p.res_in_ch) {
                                const uint32_t* w = reinterpret_cast<const uint32_t*>(p.res_in) + (spix * G + cbase / 16) * (size_t)p.B * 6;
                                const v4i a = *reinterpret_cast<const v4i*>(w + (size_t)b * 4);
                                const int2 c = *reinterpret_cast<const int2*>(w + (size_t)p.B * 4 + (size_t)b * 2);
                                dst[0] = a[0], dst[1] = a[1], dst[2] = a[2], dst[3] = a[3], dst[4] = c.x, dst[5] = c.y;
                            }
                        } else {
                            constexpr int kCh = (int)residual_group_channels(RF);
#pragma unroll
                            for (int g = 0; g < 16 / kCh; ++g)
                                if (cbase + kCh * g < p.res_in_ch) {
                                    const v4i a = reinterpret_cast<const v4i*>(p.res_in)[(spix * G + cbase / kCh + g) * (size_t)p.B + b];
                                    dst[4 * g] = a[0], dst[4 * g + 1] = a[1], dst[4 * g + 2] = a[2], dst[4 * g + 3] = a[3];
                                }
                        }
                    }
                }
            }
        }
    }

    // ---- the table of K: byte offset of word k's activation from the column's first tap, and its tap
    for (int k = tid; k < 8 * p.groups; k += blockDim.x) {
        const unsigned tap = div_by((unsigned)k, p.by_cw), w = (unsigned)k - tap * p.by_cw.d;
        const unsigned r = div_by(tap, p.by_s), s = tap - r * p.by_s.d;
        tab[k] = k < p.kw_tot ? make_int2((int)((r * (unsigned)p.W + s) * pix_b + w * row_b), (int)tap) : make_int2(0, kTapNone);
    }
    __syncthreads();

    const __amdgpu_buffer_rsrc_t r_act =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.act), 0, (int)p.act_bytes, 0x00020000);
    uint32_t bw[D][MT][4];
    int tp[D][4];
    auto request_b = [&](int slot, int g) __attribute__((always_inline)) {
        const v4i* t = reinterpret_cast<const v4i*>(tab + 8 * g + 4 * h);
        const v4i t0 = t[0], t1 = t[1];
        const int off[4] = {t0[0], t0[2], t1[0], t1[2]};
        tp[slot][0] = t0[1], tp[slot][1] = t0[3], tp[slot][2] = t1[1], tp[slot][3] = t1[3];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                // all ones where the tap is invalid: the offset then lies outside the buffer, the load returns 0
                const unsigned m = (unsigned)__builtin_amdgcn_sbfe((int)inval[mt], (unsigned)tp[slot][i], 1u);
                bw[slot][mt][i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r_act, (int)((base[mt] + (unsigned)off[i]) | m), 0, 0);
            }
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (g_begin + d < g_end) request_b(d, g_begin + d);

    // A tap's pad bits are 0 in both operands: each adds +1, which the sums (of the wave that finishes) start below 0 by.
    v16f acc[MT][NT];
    const int padbits = 32 * p.cw - p.k_tap;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const float from = slice == 0 ? 0.0f - (float)(padbits * (p.R * p.S - __popc(inval[mt] & ((1u << (p.R * p.S)) - 1u)))) : 0.0f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[mt][nt][v] = from;
    }

    // +-1 in FP4 as in expand_f4, zero where the tap is invalid (its word was returned as 0)
    auto expand_col = [&](uint32_t x, unsigned c) __attribute__((always_inline)) {
        v4i r;
        auto bfi = [&](uint32_t shifted) __attribute__((always_inline)) {
            int d;
            asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(d) : "s"(0x88888888u), "v"(shifted), "v"(c));
            return d;
        };
        r[0] = bfi(x << 3);
        r[1] = bfi(x << 2);
        r[2] = bfi(x << 1);
        r[3] = bfi(x);
        return r;
    };
    for (int g0 = g_begin; g0 < g_end; g0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int g = g0 + d;
            if (g < g_end) {  // (uniform)
                const int left = p.kw_tot - 8 * g;  // steps past the row's last word in both halves are not multiplied
                v4i a[NT];
                uint32_t x[MT][4];
                int tq[4];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) a[nt] = aw[d][nt];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    tq[i] = tp[d][i];
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) x[mt][i] = bw[d][mt][i];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (i < left) {
                        v4i bf[MT], af[NT];
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) {
                            const unsigned m = (unsigned)__builtin_amdgcn_sbfe((int)inval[mt], (unsigned)tq[i], 1u);
                            bf[mt] = expand_col(x[mt][i], ~m & 0x22222222u);
                        }
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) af[nt] = expand_f4((uint32_t)a[nt][i]);
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                            for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = Acc<FMT_F4>::mma(af[nt], bf[mt], acc[mt][nt]);
                    }
                if (g + D < g_end) {
                    request_w(d, g + D);
                    request_b(d, g + D);
                }
            }
        }
    }

    // ---- the slices' sums meet in LDS; wave 0 of the workgroup finishes the tile
    if (p.slices > 1) {
        if (slice > 0) {
#pragma unroll
            for (int t = 0; t < MT * NT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v16f& s = acc[t / NT][t % NT];
                    red[(((slice - 1) * MT * NT + t) * 4 + q) * 64 + lane] = v4f{s[4 * q], s[4 * q + 1], s[4 * q + 2], s[4 * q + 3]};
                }
        }
        __syncthreads();
        if (slice > 0) return;
    }
    if (!live) return;

    const int ow = (p.N + 31) / 32;
    const float never = p.nan_bit ? -INFINITY : INFINITY;  // (a threshold that is no number)
    uint32_t orw[NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int k = WIN == FW_TILES ? 0 : mt;
        const int b = cb[k];
        const bool ok = cok[k];
        const size_t pix = (size_t)cy[mt] * p.PW + cx[mt];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int cbase = n0 + nt * 32 + 16 * h;
            float sum[16];  // (whole numbers below 2^24)
#pragma unroll
            for (int v = 0; v < 16; ++v) sum[v] = acc[mt][nt][v];
            for (int s = 1; s < p.slices; ++s)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const v4f o = red[(((s - 1) * MT * NT + mt * NT + nt) * 4 + q) * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[4 * q + e] += o[e];
                }
            if constexpr (FM == FM_RAW) {
                int* mine = raw_area + (p.slices > 1 ? 0 : wave) * kRawWords;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<v4i*>(mine + j * raw_pitch(NT) + nt * 32 + 16 * h + 4 * q) =
                        v4i{(int)sum[4 * q], (int)sum[4 * q + 1], (int)sum[4 * q + 2], (int)sum[4 * q + 3]};
                continue;
            }
            int whole[16];
            if constexpr (kRes && RF == TCBNN_RES_I32) {
#pragma unroll
                for (int v = 0; v < 16; ++v) whole[v] = (int)sum[v];
            }
            if constexpr (kRes) {
                if (p.res_lim > 0) {
                    int rv[16];
#pragma unroll
                    for (int s = 0; s < NSRC; ++s) {
                        const int* w = rraw[mt * NT + nt][s];
                        int t[16];
                        if constexpr (RF == TCBNN_RES_I12) {
                            i12_unpack8((uint32_t)w[0], (uint32_t)w[1], (uint32_t)w[2], t);
                            i12_unpack8((uint32_t)w[3], (uint32_t)w[4], (uint32_t)w[5], t + 8);
                        } else if constexpr (RF == TCBNN_RES_I16) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) t[2 * e] = (w[e] << 16) >> 16, t[2 * e + 1] = w[e] >> 16;
                        } else {
#pragma unroll
                            for (int v = 0; v < 16; ++v) t[v] = w[v];
                        }
#pragma unroll
                        for (int v = 0; v < 16; ++v) rv[v] = s == 0 ? t[v] : max(rv[v], t[v]);
                    }
                    if (n0 + nt * 32 + 32 > p.res_lim)  // (uniform)
#pragma unroll
                        for (int v = 0; v < 16; ++v) rv[v] = cbase + v < p.res_lim ? rv[v] : 0;
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        if constexpr (RF == TCBNN_RES_I32) whole[v] += rv[v], sum[v] = (float)whole[v];  // (any number)
                        else sum[v] += (float)rv[v];
                    }
                }
            }
            // bits, MSB first: the inverted sign of sum - threshold
            uint32_t hw = signs(sum, thr[nt] == thr[nt] ? thr[nt] : never, std::make_integer_sequence<int, 16>{});
            hw = ~hw & 0xffffu & (0xffff0000u >> min(max(p.N - cbase, 0), 16));
            if constexpr (kRes) {
                if (p.res_out != nullptr) {
                    if (ok && cbase < p.N) {
                        int rs[16];
#pragma unroll
                        for (int v = 0; v < 16; ++v) rs[v] = RF == TCBNN_RES_I32 ? whole[v] : (int)sum[v];
                        if (n0 + nt * 32 + 32 > p.N)  // (uniform)
#pragma unroll
                            for (int v = 0; v < 16; ++v) rs[v] = cbase + v < p.N ? rs[v] : 0;  // (0 past N inside a group)
                        if (p.res_out_fmt == TCBNN_RES_I12) {
                            residual_store_group16(p.res_out, TCBNN_RES_I12, pix, p.N, cbase / 16, p.B, b, rs);
                        } else if (p.res_out_fmt == TCBNN_RES_I16) {
                            v4i* dst = reinterpret_cast<v4i*>(p.res_out) + (pix * (size_t)((p.N + 7) / 8) + cbase / 8) * p.B + b;
#pragma unroll
                            for (int g = 0; g < 2; ++g)
                                if (cbase + 8 * g < p.N)
                                    dst[(size_t)g * p.B] = v4i{(rs[8 * g] & 0xffff) | (rs[8 * g + 1] << 16),
                                                               (rs[8 * g + 2] & 0xffff) | (rs[8 * g + 3] << 16),
                                                               (rs[8 * g + 4] & 0xffff) | (rs[8 * g + 5] << 16),
                                                               (rs[8 * g + 6] & 0xffff) | (rs[8 * g + 7] << 16)};
                        } else {
                            v4i* dst = reinterpret_cast<v4i*>(p.res_out) + (pix * (size_t)((p.N + 3) / 4) + cbase / 4) * p.B + b;
#pragma unroll
                            for (int g = 0; g < 4; ++g)
                                if (cbase + 4 * g < p.N)
                                    dst[(size_t)g * p.B] = v4i{rs[4 * g], rs[4 * g + 1], rs[4 * g + 2], rs[4 * g + 3]};
                        }
                    }
                }
            }
            // the half word of lane + 32 completes the word of lane j
            const uint32_t other = __builtin_amdgcn_permlane32_swap(hw, hw, false, false)[1];
            uint32_t word = (hw << 16) | other;
            if constexpr (WIN == FW_TILES) {
                orw[nt] = mt == 0 ? word : orw[nt] | word;
                if (mt < MT - 1) continue;
                word = orw[nt];
            }
            if constexpr (WIN == FW_LANES) {
                word |= (uint32_t)__shfl_xor((int)word, 8);
                word |= (uint32_t)__shfl_xor((int)word, 16);
            }
            if ((WIN == FW_LANES ? lane < 8 : h == 0) && ok) {
                const size_t opix = WIN != FW_NONE ? (size_t)cpix[0] : pix;
                uint32_t* dst = p.out_bits + opix * (size_t)p.bits_pix_stride + b;
                const int w = ng * NT + nt;
                if (w < p.bits_row_words) dst[(size_t)w * p.B] = word;
                if (ng == p.n_groups - 1 && nt == NT - 1)  // the pixel's padding words
                    for (int z = max(ow, p.n_groups * NT); z < p.bits_row_words; ++z) dst[(size_t)z * p.B] = 0;
            }
        }
        if constexpr (FM == FM_RAW) {
            // int32 output: a lane holds 16 channels of one column; through LDS (the same wave writes and reads) a
            // store instruction covers whole channel runs of its columns instead of 64 pieces of 16 bytes
            int* mine = raw_area + (p.slices > 1 ? 0 : wave) * kRawWords;
            long long* start = reinterpret_cast<long long*>(mine + 32 * raw_pitch(NT));
            const long long at = (long long)pix * p.raw_pix_stride + (long long)b * p.raw_b_stride + n0;
            if (h == 0) start[j] = ok ? at : -1;
            const int chans = min(32 * NT, p.N - n0);
            const bool vec = chans == 32 * NT && p.raw_pix_stride % 4 == 0 && p.raw_b_stride % 4 == 0 &&
                             (reinterpret_cast<uintptr_t>(p.out_i32) & 15) == 0;  // (uniform)
            if (vec) {
                constexpr int kCols = 8 * NT, kRows = 64 / kCols;
                const int rl = lane / kCols, cl = lane % kCols;
#pragma unroll
                for (int r = 0; r < 32; r += kRows) {
                    const v4i q = *reinterpret_cast<const v4i*>(mine + (r + rl) * raw_pitch(NT) + 4 * cl);
                    const long long to = start[r + rl];
                    if (to >= 0) *reinterpret_cast<v4i*>(p.out_i32 + to + 4 * cl) = q;
                }
            } else {
                constexpr int kCols = 32, kRows = 2;
                const int rl = lane / kCols, cl = lane % kCols;
                for (int r = 0; r < 32; r += kRows) {
                    const long long to = start[r + rl];
                    for (int c = cl; c < chans; c += kCols)
                        if (to >= 0) p.out_i32[to + c] = mine[(r + rl) * raw_pitch(NT) + c];
                }
            }
        }
    }
}

struct FlatPlan {
    int mt, nt, slices, win;
};

int flat_mode(const BgemmParams& p) {
    if (p.mode == EPI_RAW) return FM_RAW;
    if (p.res_in == nullptr && p.res_out == nullptr) return FM_BITS;
    return p.res_in != nullptr && p.res_pool ? FM_RESPOOL : FM_RES;
}

// column tiles (of MT x 32, or of 32 windows) times channel groups
long long flat_tiles(const BgemmParams& p, int mt, int nt, int win) {
    const long long items = win != FW_NONE ? (long long)(p.PH / 2) * (p.PW / 2) : (long long)p.PH * p.PW;
    const long long per = win == FW_LANES ? 8 : (win == FW_TILES ? 32 : 32LL * mt);
    return (items * p.B + per - 1) / per * ((p.N + 32 * nt - 1) / (32 * nt));
}

// The largest tile that still gives each of the 1024 SIMDs a wave (every expanded fragment then feeds more MFMAs); tiles
// of one MFMA are split along K until the SIMDs are busy or a slice is one group.  Measured on the 8 x 8 .. 56 x 56
// layers of the networks at batch 1 .. 64: eight slices 5.9 us against 8.3 us unsplit for 512 -> 512 channels at 7 x 7,
// batch 8; more than eight gained nothing (the one wave that adds the sums up takes as long as it saves).
FlatPlan flat_plan(const BgemmParams& p) {
    const int groups = (p.R * p.S * p.cw + 7) / 8;
    const int fm = flat_mode(p);
    constexpr int kSimds = 1024;
    FlatPlan f = {1, 1, 1, p.pool_h == 2 ? FW_LANES : FW_NONE};
    if (f.win != FW_NONE) {
        if (flat_tiles(p, 4, 2, FW_TILES) >= kSimds) f = {4, 2, 1, FW_TILES};
        else if (flat_tiles(p, 4, 1, FW_TILES) >= kSimds) f = {4, 1, 1, FW_TILES};
    } else if (fm != FM_RESPOOL) {  // (with a residual a 4 x 2 tile does not fit the registers)
        if (fm != FM_RES && flat_tiles(p, 4, 2, FW_NONE) >= kSimds) f.mt = 4, f.nt = 2;
        else if (flat_tiles(p, 2, 2, FW_NONE) >= kSimds) f.mt = 2, f.nt = 2;
    }
    if (f.mt * f.nt == 1) {
        const long long tiles = flat_tiles(p, 1, 1, f.win);
        while (f.slices < max_waves(1, 1) && tiles * f.slices < kSimds && 2 * f.slices <= groups) f.slices *= 2;
    }
    return f;
}

// LDS of a workgroup: the sums of the slices, the staging area of int32 output, the table of K.  A workgroup gets 64 KiB
// of it; a long K of int32 output can need more (above 4000 words where it is split over eight waves, above 3712 where
// four waves stage a 2 x 2 tile each), and such a problem is left to the generic kernel.
constexpr size_t kLdsMost = 64 * 1024;
int flat_waves(const FlatPlan& pl) { return pl.slices > 1 ? pl.slices : 4; }
int flat_tiles_per_wg(const FlatPlan& pl) { return pl.slices > 1 ? 1 : 4; }
size_t flat_lds_bytes(const BgemmParams& p, const FlatPlan& pl) {
    const size_t raw = p.mode == EPI_RAW ? (size_t)flat_tiles_per_wg(pl) * (32 * raw_pitch(pl.nt) + 64) * 4 : 0;
    return (size_t)(pl.slices - 1) * pl.mt * pl.nt * 4096 + raw + (size_t)((p.R * p.S * p.cw + 7) / 8) * 64;
}

template <int MT, int NT, int FM, int RF, int WIN>
int launch(const BgemmParams& p, const FlatPlan& pl, hipStream_t stream) {
    FlatArgs f{};
    const int row = WIN != FW_NONE ? p.PW / 2 : p.PW;
    const long long items = WIN != FW_NONE ? (long long)(p.PH / 2) * (p.PW / 2) : (long long)p.PH * p.PW;
    f.act = p.act, f.wgt = p.wgt, f.bn = p.bn, f.res_in = p.res_in;
    f.out_bits = p.out_bits, f.out_i32 = p.out_i32, f.res_out = p.res_out;
    f.bits_pix_stride = p.bits_pix_stride, f.raw_pix_stride = p.raw_pix_stride, f.raw_b_stride = p.raw_b_stride;
    f.n_groups = (p.N + 32 * NT - 1) / (32 * NT);
    f.by_batch = fast_div((uint32_t)p.B);
    f.by_row = fast_div((uint32_t)row);
    f.by_cw = fast_div((uint32_t)p.cw);
    f.by_s = fast_div((uint32_t)p.S);
    f.by_groups = fast_div((uint32_t)f.n_groups);
    f.B = p.B, f.cw = p.cw, f.H = p.H, f.W = p.W, f.R = p.R, f.S = p.S;
    f.stride_h = p.stride_h, f.stride_w = p.stride_w, f.pad_h = p.pad_h, f.pad_w = p.pad_w;
    f.PW = p.PW, f.N = p.N, f.k_tap = p.k_tap, f.nan_bit = p.nan_bit, f.bits_row_words = p.bits_row_words;
    f.res_in_ch = p.res_in_ch, f.res_out_fmt = p.res_out_fmt;
    f.res_lim = p.res_in != nullptr ? std::min(std::min(p.res_limit, p.res_in_ch), p.N) : 0;
    f.cols = (int)(items * p.B);
    f.kw_tot = p.R * p.S * p.cw;
    f.groups = (f.kw_tot + 7) / 8;
    f.per_slice = (f.groups + pl.slices - 1) / pl.slices;
    f.slices = pl.slices;
    const long long total = flat_tiles(p, MT, NT, WIN);
    f.total = (int)total;
    f.act_bytes = (unsigned)(4LL * p.H * p.W * p.cw * p.B);
    f.wgt_bytes = (unsigned)(4LL * pad32(p.N) * f.kw_tot);
    const int waves = flat_waves(pl), per_wg = flat_tiles_per_wg(pl);
    const long long wgs = (total + per_wg - 1) / per_wg, blocks = (wgs + 7) / 8 * 8;
    f.wgs = (int)wgs;
    f.per_xcd = (int)(blocks / 8);
    const size_t lds = flat_lds_bytes(p, pl);
    if (blocks <= 0 || blocks > 0x7fffffffLL || lds > kLdsMost) return fail(TCBNN_EINVAL, "bgemm_flat: launch too large");
    hipLaunchKernelGGL((bgemm_flat_f4_kernel<MT, NT, FM, RF, WIN>), dim3((unsigned)blocks), dim3(64 * waves), lds, stream, f);
    TCBNN_LAUNCH_CHECK("bgemm_flat_f4_kernel");
    return TCBNN_OK;
}

template <int MT, int NT>
int launch_res(const BgemmParams& p, const FlatPlan& pl, hipStream_t stream) {
    const int fmt = p.res_in != nullptr ? p.res_in_fmt : TCBNN_RES_I32;
    if (fmt == TCBNN_RES_I12) return launch<MT, NT, FM_RES, TCBNN_RES_I12, FW_NONE>(p, pl, stream);
    if (fmt == TCBNN_RES_I16) return launch<MT, NT, FM_RES, TCBNN_RES_I16, FW_NONE>(p, pl, stream);
    return launch<MT, NT, FM_RES, TCBNN_RES_I32, FW_NONE>(p, pl, stream);
}

}  // namespace

bool bgemm_flat_applicable(const BgemmParams& p) {
    if (p.ksplit > 1 || (p.mode != EPI_THRESH && p.mode != EPI_RAW)) return false;
    const int kw_tot = p.R * p.S * p.cw;
    if (p.R * p.S >= kTapNone || kw_tot > kMaxWords - 8) return false;
    const bool res = p.res_in != nullptr || p.res_out != nullptr;
    const bool pool1 = p.pool_h == 1 && p.pool_w == 1;
    const bool pool2 = p.pool_h == 2 && p.pool_w == 2 && p.PH % 2 == 0 && p.PW % 2 == 0 && !res && p.mode == EPI_THRESH;
    if (!pool1 && !pool2) return false;
    if (p.res_out_pool) return false;
    const long long cols = (long long)p.PH * p.PW * p.B;
    return cols < (1LL << 30) && 4LL * p.H * p.W * p.cw * p.B < (1LL << 31) && 4LL * (p.N + 64) * kw_tot < (1LL << 31) &&
           flat_lds_bytes(p, flat_plan(p)) <= kLdsMost;
}

// Both kernels serve the 3x3 layers of conv3x3_mfma.hip: which is faster?  An estimate of both launches in microseconds,
// fitted to 623 measured pairs (all layers of five networks at batch 1 .. 200, and int32 convolutions with 64 .. 512
// input channels, 64 .. 512 output channels, 8 x 8 .. 56 x 56 pixels, batch 2 .. 200): choosing by it costs 0.5 % over
// choosing by measurement, always taking the persistent kernel 20 %.  (Measured with eight waves to a large workgroup and the
// image tiles of conv3x3_mfma_image_tiles: where the persistent kernel has got faster since, the estimate charges it too much.)
bool bgemm_flat_preferred(const BgemmParams& p) {
    if (!conv3x3_mfma_applicable(p) || !bgemm_flat_applicable(p)) return false;
    const double steps = 9.0 * p.cw / 2, pix = (double)p.PH * p.PW, n_tiles = (p.N + 31) / 32;
    const bool raw = p.mode == EPI_RAW, res = p.res_in != nullptr || p.res_out != nullptr, pool = p.pool_h == 2;
    // Outside what was measured, or where nothing is to be gained, the persistent kernel stays: partial channel tiles
    // (its other instantiations), un-pooled layers of 32 images and more (multiples of 32 fill their tiles there too; for
    // others the estimate was not fitted), and pooled ones of fewer windows than fill two tiles.
    const int res_lim = p.res_in != nullptr ? std::min(std::min(p.res_limit, p.res_in_ch), p.N) : 0;
    if (!raw && (p.N % 64 != 0 || res_lim % 32 != 0 || (p.B >= 32 && !pool))) return false;
    if (pool && (long long)p.OH * p.OW * p.B < 16) return false;
    const int mt = conv3x3_mfma_image_tiles(p);
    const double b_groups = (p.B + 32 * mt - 1) / (32 * mt);
    const double mib = raw ? 4e-6 * pix * p.B * p.N : 0.0;  // output, MB
    // persistent kernel: staging the weights, then the longer of one work item's MFMAs and the whole machine's
    const double item = 0.0175 * steps * 2 * mt * (pool ? 4 : 1);
    const double all = 23e-6 * pix * b_groups * mt * n_tiles * steps;
    const double t_persistent = 4.0 + 0.02 * steps + std::max(item, all) + (res ? 1.2 : 0.0) + 0.24 * mib;
    // this kernel: full tiles, but operands expanded for every tile and a prologue per tile (the share of short K)
    const double mfmas = (double)(((long long)p.PH * p.PW * p.B + 31) / 32) * n_tiles * steps;
    // (The fit is from before the finish in fp32, which launches of few tiles gain from by up to 1.2 us: with that, ResNet-18 at batch 8
    // 111.9 -> 107.4 us a pass and at 10 117.0 -> 113.8.  As much for all launches: batch 25 of the textbook wiring 1.7 % slower.)
    const double few = 1.2 * std::max(0.0, 1.0 - mfmas / 23000.0);
    const double t_flat = 4.4 - few + 1e-6 * mfmas * (40.0 + 380.0 / steps) + 0.015 * steps + (res ? 0.5 : 0.0) + 0.16 * mib;
    return t_flat < t_persistent;
}

void bgemm_flat_kernel_name(const BgemmParams& p, char* buf, size_t len) {
    const FlatPlan f = flat_plan(p);
    const int fm = flat_mode(p);
    const int rf = (fm == FM_RES || fm == FM_RESPOOL) && p.res_in != nullptr ? p.res_in_fmt : TCBNN_RES_I32;
    snprintf(buf, len, "bgemm_flat_f4_kernel<%d, %d, %d, %d, %d>", f.mt, f.nt, fm, rf, f.win);
}

int launch_bgemm_flat(const BgemmParams& p, hipStream_t stream) {
    const FlatPlan pl = flat_plan(p);
    const int fm = flat_mode(p);
    if (pl.win == FW_LANES) return launch<1, 1, FM_BITS, TCBNN_RES_I32, FW_LANES>(p, pl, stream);
    if (pl.win == FW_TILES)
        return pl.nt == 2 ? launch<4, 2, FM_BITS, TCBNN_RES_I32, FW_TILES>(p, pl, stream)
                          : launch<4, 1, FM_BITS, TCBNN_RES_I32, FW_TILES>(p, pl, stream);
    if (fm == FM_RESPOOL) {
        if (p.res_in_fmt == TCBNN_RES_I12) return launch<1, 1, FM_RESPOOL, TCBNN_RES_I12, FW_NONE>(p, pl, stream);
        if (p.res_in_fmt == TCBNN_RES_I16) return launch<1, 1, FM_RESPOOL, TCBNN_RES_I16, FW_NONE>(p, pl, stream);
        return launch<1, 1, FM_RESPOOL, TCBNN_RES_I32, FW_NONE>(p, pl, stream);
    }
    if (fm == FM_RES)
        return pl.mt == 1 ? launch_res<1, 1>(p, pl, stream) : launch_res<2, 2>(p, pl, stream);
    if (fm == FM_RAW)
        return pl.mt == 1 ? launch<1, 1, FM_RAW, TCBNN_RES_I32, FW_NONE>(p, pl, stream)
                          : (pl.mt == 2 ? launch<2, 2, FM_RAW, TCBNN_RES_I32, FW_NONE>(p, pl, stream)
                                        : launch<4, 2, FM_RAW, TCBNN_RES_I32, FW_NONE>(p, pl, stream));
    return pl.mt == 1 ? launch<1, 1, FM_BITS, TCBNN_RES_I32, FW_NONE>(p, pl, stream)
                      : (pl.mt == 2 ? launch<2, 2, FM_BITS, TCBNN_RES_I32, FW_NONE>(p, pl, stream)
                                    : launch<4, 2, FM_BITS, TCBNN_RES_I32, FW_NONE>(p, pl, stream));
}

}  // namespace tcbnn
