// FP4 matrix-core kernel of 1x1 bit convolutions that save their sums as a residual (the shortcuts of the textbook wiring:
// 64 .. 256 channels in, stride 2).  K is one to four products long, so everything but the epilogue is done once per wave and
// kept: a wave owns 64 output channels, holds their weights as FP4 fragments and their thresholds in registers, and walks a
// strided list of 32-column tiles (column = pixel * batch + image, full whatever the batch), asking for the next tile's words
// before it finishes the present one.
//
// The sums start from 1.5 * 2^23: the bit pattern of a finished sum is then 0x4B400000 + s, whose low bits are stored without
// a conversion, and one subtraction of 1.5 * 2^23 + ceil(threshold) gives the output bit by its sign.
//
// What bounds it: the stores, and at the start of a launch the way of the words.  bgemm_flat.hip's kernel, which serves the other
// 1x1 forms, spends most of such a launch on each tile's prologue.  The three shortcuts of ResNet-18, launched on end, us, there
// -> here: batch 256 64 -> 128 channels at 28x28 19.8 -> 9.9 (48 MB, 4.8 TB/s), 128 -> 256 at 14x14 13.3 -> 7.0, 256 -> 512 at 7x7
// 7.9 -> 6.0; batch 64 7.5 -> 5.0, 5.7 -> 4.6, 4.7 -> 4.5; batch 8 and fewer level (4.1 .. 4.4).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

using namespace mfma;

typedef int v2i __attribute__((ext_vector_type(2)));

constexpr int kWaves = 4;
constexpr int kNT = 2;  // channel tiles of a wave
constexpr int kCus = 256;
constexpr int resident(int ks) { return ks == 4 ? 3 : 4; }  // workgroups a compute unit holds (registers)
constexpr float kMagic = 12582912.0f;          // 1.5 * 2^23
constexpr uint32_t kMagicBits = 0x4B400000u;
constexpr float kThrLimit = 2097152.0f;        // 2^21: beyond every sum

struct Conv1x1Args {
    const uint32_t* act;
    const uint32_t* wgt;
    const float* bn;
    uint32_t* out_bits;
    int32_t* res_out;
    long long bits_pix_stride;
    FastDiv by_batch, by_row;
    int B, W, PW, N, stride_h, stride_w, nan_bit;
    int cols, tiles, streams, n_groups;
    unsigned act_bytes;
};

// KS = 64-channel k-steps; FMT = format of the saved residual
template <int KS, int FMT>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(resident(KS)))) void conv1x1_mfma_f4_kernel(const Conv1x1Args p) {
    constexpr int cw = 2 * KS;
    const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
    const int id = __builtin_amdgcn_readfirstlane((int)blockIdx.x * kWaves + (int)(threadIdx.x >> 6));
    const int stream = id / p.n_groups, n0 = (id - stream * p.n_groups) * (32 * kNT);
    if (stream >= p.streams) return;

    const __amdgpu_buffer_rsrc_t r_act = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.act), 0, (int)p.act_bytes, 0x00020000);
    struct Column {
        unsigned pix, b;
    };
    auto column = [&](int tile) __attribute__((always_inline)) {  // (past the last column: the last one, not stored)
        const unsigned col = min((unsigned)tile * 32u + (unsigned)j, (unsigned)p.cols - 1u);
        Column c;
        c.pix = div_by(col, p.by_batch);
        c.b = col - c.pix * (unsigned)p.B;
        return c;
    };
    auto request = [&](const Column& c, uint32_t (&x)[KS]) __attribute__((always_inline)) {
        const unsigned y = div_by(c.pix, p.by_row), px = c.pix - y * (unsigned)p.PW;
        const unsigned at = (((y * (unsigned)p.stride_h * (unsigned)p.W + px * (unsigned)p.stride_w) * cw + (unsigned)(KS * h)) * (unsigned)p.B + c.b) * 4u;
#pragma unroll
        for (int s = 0; s < KS; ++s)  // lane half h multiplies words KS h + s, which lie together in a row of weights
            x[s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r_act, (int)at, s * 4 * p.B, 0);
    };
    int tile = stream;
    Column now = column(tile);
    uint32_t x[KS];
    request(now, x);

    const __amdgpu_buffer_rsrc_t r_wgt = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.wgt), 0, p.N * cw * 4, 0x00020000);
    uint32_t wword[KS][kNT];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
        const int at = ((n0 + 32 * nt + row_to_channel(j)) * cw + KS * h) * 4;
        if constexpr (KS == 1) {
            wword[0][nt] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r_wgt, at, 0, 0);
        } else if constexpr (KS == 2) {
            const v2i q = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(r_wgt, at, 0, 0));
            wword[0][nt] = (uint32_t)q[0], wword[1][nt] = (uint32_t)q[1];
        } else {
            const v4i q = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r_wgt, at, 0, 0));
#pragma unroll
            for (int s = 0; s < 4; ++s) wword[s][nt] = (uint32_t)q[s];
        }
    }
    // One request for the thresholds of 64 channels, and through LDS (written and read by this wave only) to the lanes' sixteen
    // of each channel tile: the address unit takes 17 cycles for a request (a channel at a time, 32 requests a wave: 11.3 us for 9.9,
    // 8.7 for 7.4; weights by the word instead of the row's part: 8.9 for 6.2 at 256 channels).
    __shared__ __align__(16) float par[kWaves][32 * kNT];
    float* const mine = par[threadIdx.x >> 6];
    const float t = p.bn[n0 + lane];
    // s < t is s < ceil(t) for a whole number s
    mine[lane] = kMagic + (t == t ? fminf(fmaxf(ceilf(t), -kThrLimit), kThrLimit) : (p.nan_bit ? -kThrLimit : kThrLimit));
    // (what other lanes wrote is read below: the order within the wave is said, not left to what the compiler cannot prove)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    v4i w[KS][kNT];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
#pragma unroll
        for (int s = 0; s < KS; ++s) w[s][nt] = expand_f4(wword[s][nt]);
    }
    float thr[kNT][16];
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
        for (int v = 0; v < 16; ++v) thr[nt][v] = mine[32 * nt + 16 * h + v];

    for (; tile < p.tiles; tile += p.streams) {
        v16f acc[kNT];
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[nt][v] = kMagic;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const v4i y = expand_f4(x[s]);
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt) acc[nt] = Acc<FMT_F4>::mma(w[s][nt], y, acc[nt]);
        }
        const Column c = now;
        const bool ok = tile * 32 + j < p.cols;
        if (tile + p.streams < p.tiles) {  // (uniform)
            now = column(tile + p.streams);
            request(now, x);
        }
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) {
            uint32_t hw = 0;
#pragma unroll
            for (int v = 0; v < 16; ++v) hw = __builtin_amdgcn_alignbit(hw, __float_as_uint(acc[nt][v] - thr[nt][v]), 31);
            hw = ~hw & 0xffffu;
            // the half word of lane + 32 completes the word of lane j
            const uint32_t other = __builtin_amdgcn_permlane32_swap(hw, hw, false, false)[1];
            if (h == 0 && ok)
                p.out_bits[(size_t)c.pix * (size_t)p.bits_pix_stride + (size_t)(n0 / 32 + nt) * p.B + c.b] = (hw << 16) | other;
            if (ok) {
                int s[16];
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = __float_as_int(acc[nt][v]);
                const int cbase = n0 + 32 * nt + 16 * h;
                if constexpr (FMT == TCBNN_RES_I12) {  // (takes the low 12 bits)
                    residual_store_group16(p.res_out, TCBNN_RES_I12, c.pix, p.N, cbase / 16, p.B, (int)c.b, s);
                } else if constexpr (FMT == TCBNN_RES_I16) {
                    v4i* dst = reinterpret_cast<v4i*>(p.res_out) + ((size_t)c.pix * (size_t)(p.N / 8) + cbase / 8) * p.B + c.b;
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        v4i o;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[e] = (int)__builtin_amdgcn_perm((uint32_t)s[8 * g + 2 * e + 1], (uint32_t)s[8 * g + 2 * e], 0x05040100u);
                        dst[(size_t)g * p.B] = o;
                    }
                } else {
                    v4i* dst = reinterpret_cast<v4i*>(p.res_out) + ((size_t)c.pix * (size_t)(p.N / 4) + cbase / 4) * p.B + c.b;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        v4i o;
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = s[4 * g + e] - (int)kMagicBits;
                        dst[(size_t)g * p.B] = o;
                    }
                }
            }
        }
    }
}

template <int KS, int FMT>
int launch(const BgemmParams& p, hipStream_t stream) {
    Conv1x1Args a{};
    a.act = p.act, a.wgt = p.wgt, a.bn = p.bn, a.out_bits = p.out_bits, a.res_out = p.res_out;
    a.bits_pix_stride = p.bits_pix_stride;
    a.by_batch = fast_div((uint32_t)p.B), a.by_row = fast_div((uint32_t)p.PW);
    a.B = p.B, a.W = p.W, a.PW = p.PW, a.N = p.N, a.stride_h = p.stride_h, a.stride_w = p.stride_w, a.nan_bit = p.nan_bit;
    a.cols = p.PH * p.PW * p.B;
    a.tiles = (a.cols + 31) / 32;
    a.n_groups = p.N / (32 * kNT);
    a.act_bytes = (unsigned)(4LL * p.H * p.W * p.cw * p.B);
    // all workgroups resident, fewer where there are not as many tiles
    const long long waves = std::min((long long)a.tiles * a.n_groups, (long long)resident(KS) * kCus * kWaves);
    a.streams = (int)std::max(1LL, waves / a.n_groups);
    const long long wgs = ((long long)a.streams * a.n_groups + kWaves - 1) / kWaves;
    hipLaunchKernelGGL((conv1x1_mfma_f4_kernel<KS, FMT>), dim3((unsigned)wgs), dim3(64 * kWaves), 0, stream, a);
    TCBNN_LAUNCH_CHECK("conv1x1_mfma_f4_kernel");
    return TCBNN_OK;
}

}  // namespace

bool conv1x1_mfma_applicable(const BgemmParams& p) {
    if (p.mode != EPI_THRESH || p.ksplit > 1 || p.R * p.S != 1 || p.pad_h != 0 || p.pad_w != 0 || p.pool_h * p.pool_w != 1) return false;
    if (p.res_in != nullptr || p.res_out == nullptr || p.res_out_pool) return false;
    // whole words of 64, 128 or 256 channels, whole pairs of channel tiles, no padding words
    if ((p.cw != 2 && p.cw != 4 && p.cw != 8) || p.k_tap != 32 * p.cw || p.N % (32 * kNT) != 0 || p.bits_row_words != p.N / 32) return false;
    // windows inside the frame, and 32-bit offsets
    if ((p.PH - 1) * (long long)p.stride_h >= p.H || (p.PW - 1) * (long long)p.stride_w >= p.W) return false;
    // Int32 residuals, whose stores are nearly all of a launch: a persistent grid's waves drift apart and scatter the lines that they
    // write, where bgemm_flat.hip's workgroups, dealt in order, keep together.  us, there -> here (MB of input and outputs): 256
    // channels, 256 outputs at 21x21, batch 166 18.3 -> 15.3 (80 MB); from 120 MB on level within 5 %, even batches a little
    // shorter, odd ones longer (192 outputs at 49x49, batch 69 25.3 -> 26.4, 137 MB); shorter again where the other launch has just
    // left the 256 MiB memory-side cache (384 at 37x37, batch 136 68.7 -> 51.6, 301 MB); longer beyond (512 at 54x54, batch 185
    // 245 -> 389).  Narrow residuals take 0.5 .. 0.9 of the time at all sizes to 1.5 GB.
    const long long pixels = (long long)p.PH * p.PW * p.B;
    if (p.res_out_fmt == TCBNN_RES_I32) {
        const long long bytes = 4LL * p.N * pixels + 4LL * p.bits_row_words * pixels + 4LL * p.H * p.W * p.cw * p.B;
        if (bytes > 120000000LL && (bytes < 268000000LL || bytes > 320000000LL)) return false;
    }
    return pixels < (1LL << 30) && 4LL * p.H * p.W * p.cw * p.B < (1LL << 31);
}

void conv1x1_mfma_kernel_name(const BgemmParams& p, char* buf, size_t len) {
    snprintf(buf, len, "conv1x1_mfma_f4_kernel<%d, %d>", p.cw / 2, p.res_out_fmt);
}

int launch_conv1x1_mfma(const BgemmParams& p, hipStream_t stream) {
    auto by_format = [&](auto ks) {
        constexpr int KS = decltype(ks)::value;
        if (p.res_out_fmt == TCBNN_RES_I12) return launch<KS, TCBNN_RES_I12>(p, stream);
        if (p.res_out_fmt == TCBNN_RES_I16) return launch<KS, TCBNN_RES_I16>(p, stream);
        return launch<KS, TCBNN_RES_I32>(p, stream);
    };
    if (p.cw == 2) return by_format(std::integral_constant<int, 1>{});
    if (p.cw == 4) return by_format(std::integral_constant<int, 2>{});
    return by_format(std::integral_constant<int, 4>{});
}

}  // namespace tcbnn
