// FP4 matrix-core kernel for small fully connected layers (Fc128LayerFMT / Out128LayerFMT,
// kernel.cuh:174-280) at inference batch sizes: a few hundred images times a few hundred
// neurons is only some hundred 32 x 32 output tiles, far too few to fill 1024 SIMDs when one
// wave walks the whole K of a tile, and K can be long (25088 for the first FC of ResNet-18).
//
//   workgroup = one 32-image x 32-neuron output tile, up to 16 waves;
//   wave      = a contiguous slice of K: it requests its activation and weight words (128-bit
//               weight loads: the K order inside a group of 8 words is chosen so that a lane
//               owns 4 consecutive words), multiplies them, and adds its partial tile into LDS
//               with integer atomics (the partial sums are exact integers);
//   wave 0    = epilogue: threshold + pack (FC) or scale + bias (output layer).
// No split-K workspace in HBM, no clearing or finishing launch.
// Launches of few tiles take 16 x 16 ones: fc_mfma_f4_small_kernel below.
// The last wave's work is on every launch's way: a bit is the sign of sum - threshold, shifted in (with compares and selects per
// value CIFAR VGG's pass at batch 1 took 39.7 us, now 38.8, AlexNet's at batch 150 169.6, now 165.6: three such layers each).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

using namespace mfma;

constexpr int kMaxWaves = 16;
constexpr int FC_THRESH = 0, FC_AFFINE = 1;

// PRE > 0: the wave's K slice is at most PRE groups and is requested whole before the first multiply.  STAGED: activations are
// requested sixteen bytes a lane and turned in LDS (fc_plan says when).
template <int MODE, int PRE, bool STAGED>
__global__ __launch_bounds__(64 * kMaxWaves) void fc_mfma_f4_kernel(
    const BgemmParams p, const uint32_t* __restrict__ act, const uint32_t* __restrict__ wgt,
    const float* __restrict__ bnp, const float* __restrict__ bias, int n_tiles, int groups_per_wave) {
    __shared__ int red[16 * 64];
    extern __shared__ __align__(16) v4i stage[];  // [wave][2][64]: a group's activations on their way from rows to lanes
    __shared__ float par[64];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int j = lane & 31;
    const int h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kwaves = blockDim.x >> 6;
    const int nt = blockIdx.x % n_tiles, bt = blockIdx.x / n_tiles;
    const int n0 = nt * 32, b0 = bt * 32;
    const int b = b0 + j;
    const int cw = p.cw;  // words per image / per neuron; a multiple of 4
    // The weights in lane order (after the [NPAD32][cw] rows): a group is 64 lanes x 4 words, contiguous; rows >= N
    // and words >= cw hold zeros (their outputs are discarded / they multiply activation words that read as 0).
    const int groups = (cw + 7) / 8;
    const v4i* __restrict__ wlane = reinterpret_cast<const v4i*>(wgt + fc_weight_row_words(n_tiles * 32, cw)) +
                                    (size_t)nt * groups * 64 + lane;

    // K order: group g = words 8g .. 8g+7; step 4g+i multiplies words 8g+i (lanes 0-31) and 8g+4+i
    // (lanes 32-63) of both operands.
    const int g_begin = wave * groups_per_wave, g_end = min(groups, g_begin + groups_per_wave);

    // Activations.  STAGED: eight words of 32 images are one request of 16 bytes per lane (lane l: word l / 8, images 4 (l % 8) ..), a
    // quarter of the address unit's time of four words per lane; through LDS each lane gets its image's words.  Past the tensor:
    // zeros, images past the batch: whatever is there (discarded).
    const __amdgpu_buffer_rsrc_t r_act = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(act), 0, cw * p.B * 4, 0x00020000);
    const int act_lane = STAGED ? ((lane >> 3) * p.B + b0 + 4 * (lane & 7)) * 4 : (4 * h * p.B + min(b, p.B - 1)) * 4;
    uint32_t* const mine = reinterpret_cast<uint32_t*>(stage + wave * 128);
    auto load_group = [&](int g, v4i& a, v4i& bw) {
        a = wlane[(size_t)g * 64];  // (one contiguous 1 KB request per wave)
        const int at = act_lane + g * 32 * p.B;
        if constexpr (STAGED) {
            bw = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r_act, at, 0, 0));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) bw[i] = (int)__builtin_amdgcn_raw_buffer_load_b32(r_act, at + i * 4 * p.B, 0, 0);
        }
    };
    v16f acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    auto compute_group = [&](int g, int turn, const v4i& a, const v4i& words) {
        uint32_t bw[4];
        if constexpr (STAGED) {
            uint32_t* const at = mine + turn * 256;
            reinterpret_cast<v4i*>(at)[lane] = words;  // (written and read by this wave only)
#pragma unroll
            for (int i = 0; i < 4; ++i) bw[i] = at[(4 * h + i) * 32 + j];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) bw[i] = (uint32_t)words[i];
        }
        const int w0 = 8 * g + 4 * h;
        if (32 * (8 * g + 8) <= p.k_tap) {  // uniform: every bit of the group is a true input
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = Acc<FMT_F4>::mma(expand_f4((uint32_t)a[i]), expand_f4(bw[i]), acc);
        } else {  // K tail: pad bits (and words past cw) must multiply as 0, not as +1
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int nbits = p.k_tap - 32 * (w0 + i);
                const uint32_t valid = nbits >= 32 ? 0xffffffffu : (nbits <= 0 ? 0u : 0xffffffffu << (32 - nbits));
                acc = Acc<FMT_F4>::mma(expand_f4_masked((uint32_t)a[i], valid), expand_f4(bw[i]), acc);
            }
        }
    };

    // Epilogue parameters (thresholds, or scales and biases) of the tile's 32 neurons: one per lane, requested here,
    // ahead of the K loop, so that their round trip hides behind the operands'.  Neurons past N read the last valid
    // entry and are discarded.  Wave 0 passes them through LDS into the epilogue's layout (16 neurons per lane).
    const float my_thr = bnp[min(n0 + j, p.N - 1)];
    const float my_bias = MODE == FC_AFFINE ? bias[min(n0 + j, p.N - 1)] : 0.0f;

    if constexpr (PRE > 0) {
        // short slice: every operand word of the wave is requested before the first multiply (one round trip)
        v4i a[PRE];
        v4i bw[PRE];
#pragma unroll
        for (int u = 0; u < PRE; ++u)
            if (g_begin + u < g_end) load_group(g_begin + u, a[u], bw[u]);
#pragma unroll
        for (int u = 0; u < PRE; ++u)
            if (g_begin + u < g_end) compute_group(g_begin + u, u & 1, a[u], bw[u]);
    } else {
        // two groups (8 k-steps) per stage, double-buffered in registers
        v4i a0[2], a1[2];
        v4i w0[2], w1[2];
        auto load_stage = [&](int g, v4i (&a)[2], v4i (&bw)[2]) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (g + u < g_end) load_group(g + u, a[u], bw[u]);
        };
        auto compute_stage = [&](int g, v4i (&a)[2], v4i (&bw)[2]) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (g + u < g_end) compute_group(g + u, u, a[u], bw[u]);
        };
        int g = g_begin;
        if (g < g_end) load_stage(g, a0, w0);
        while (g < g_end) {
            if (g + 2 < g_end) load_stage(g + 2, a1, w1);
            compute_stage(g, a0, w0);
            g += 2;
            if (g >= g_end) break;
            if (g + 2 < g_end) load_stage(g + 2, a0, w0);
            compute_stage(g, a1, w1);
            g += 2;
        }
    }

    // ---- sum the K slices of the waves (exact integers) in LDS
    int dot[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) dot[v] = (int)acc[v];
    if (wave == 0) {
        par[j] = MODE == FC_THRESH && my_thr != my_thr ? (p.nan_bit ? -INFINITY : INFINITY) : my_thr;
        if constexpr (MODE == FC_AFFINE) par[32 + j] = my_bias;
    }
    if (kwaves > 1) {
        if (wave == 0) {
#pragma unroll
            for (int v = 0; v < 16; ++v) red[v * 64 + lane] = dot[v];
        }
        __syncthreads();
        if (wave != 0) {
#pragma unroll
            for (int v = 0; v < 16; ++v) atomicAdd(&red[v * 64 + lane], dot[v]);
        }
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int v = 0; v < 16; ++v) dot[v] = red[v * 64 + lane];
    } else {
        __syncthreads();
    }

    // ---- epilogue (wave 0): the lane holds neurons cbase + v of image b
    const int cbase = n0 + 16 * h;
    float thr[16], bia[MODE == FC_AFFINE ? 16 : 1];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        thr[v] = par[16 * h + v];
        if constexpr (MODE == FC_AFFINE) bia[v] = par[32 + 16 * h + v];
    }
    if constexpr (MODE == FC_THRESH) {
        uint32_t hw = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) hw = __builtin_amdgcn_alignbit(hw, __float_as_uint((float)dot[v] - thr[v]), 31);
        hw = ~hw & 0xffffu & (0xffff0000u >> min(max(p.N - cbase, 0), 16));
        const uint32_t other = (uint32_t)__shfl_xor((int)hw, 32);
        if (h == 0 && b < p.B) {
            if (nt < p.bits_row_words) p.out_bits[(size_t)nt * p.B + b] = (hw << 16) | other;
            if (nt == n_tiles - 1)  // padding words of the 128-padded feature axis
                for (int w = n_tiles; w < p.bits_row_words; ++w) p.out_bits[(size_t)w * p.B + b] = 0;
        }
    } else {
        if (b < p.B) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int c = cbase + v;
                // the +-1 dot product equals (float)K - (float)popc*2.0f exactly (kernel.cuh:258-270)
                if (c < p.N) p.out_f32[(size_t)b * p.N + c] = __fadd_rn(__fmul_rn((float)dot[v], thr[v]), bia[v]);
            }
        }
    }
}

// A tile of 16 images x 16 neurons, for launches that leave compute units out (thresholds and bits only; fc_plan says when): four
// times the workgroups of the kernel above, each with half the expansions, which are what its waves wait for each other with
// (14 VALU instructions to a product of 32 cycles there, to two of 16 here).  Operands are the same words: lane (i, q) multiplies
// words 8g + 4 (q & 1) + 2 (q >> 1) + s of group g in step s, of neuron and image i of the tile.  A workgroup writes half words.
template <int PRE>
__global__ __launch_bounds__(64 * kMaxWaves) void fc_mfma_f4_small_kernel(
    const BgemmParams p, const uint32_t* __restrict__ act, const uint32_t* __restrict__ wgt, const float* __restrict__ bnp, int n_tiles,
    int groups_per_wave) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef int v2i __attribute__((ext_vector_type(2)));
    __shared__ int red[4 * 64];

    const int tid = threadIdx.x;
    const int lane = tid & 63, i = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = blockIdx.x & 1, nt = (blockIdx.x >> 1) % n_tiles, bt = (blockIdx.x >> 1) / n_tiles;
    const int n0 = nt * 32 + 16 * half, b = bt * 16 + i;
    const int cw = p.cw, groups = (cw + 7) / 8;
    // neuron 16 half + i of the tile is row 8 (i / 4) + 4 half + i % 4 of the lane order (row_to_channel)
    const int row = 32 * (q & 1) + 8 * (i >> 2) + 4 * half + (i & 3), first = 4 * (q & 1) + 2 * (q >> 1);
    const v2i* __restrict__ wlane = reinterpret_cast<const v2i*>(wgt + fc_weight_row_words(n_tiles * 32, cw)) +
                                    ((size_t)nt * groups * 64 + row) * 2 + (q >> 1);
    const __amdgpu_buffer_rsrc_t r_act = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(act), 0, cw * p.B * 4, 0x00020000);
    const int act_lane = (first * p.B + min(b, p.B - 1)) * 4;
    const int g_begin = wave * groups_per_wave, g_end = min(groups, g_begin + groups_per_wave);

    // every word of the wave is requested before the first multiply
    v2i a[PRE];
    uint32_t x[PRE][2];
#pragma unroll
    for (int u = 0; u < PRE; ++u)
        if (g_begin + u < g_end) {
            a[u] = wlane[(size_t)(g_begin + u) * 128];
#pragma unroll
            for (int s = 0; s < 2; ++s)
                x[u][s] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r_act, act_lane + ((g_begin + u) * 8 + s) * 4 * p.B, 0, 0);
        }
    float thr[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) thr[v] = bnp[min(n0 + 4 * q + v, p.N - 1)];
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    auto product = [&](v4i w, v4i y) __attribute__((always_inline)) {
        const v8i w8 = {w[0], w[1], w[2], w[3], 0, 0, 0, 0}, y8 = {y[0], y[1], y[2], y[3], 0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w8, y8, acc, 4, 4, 0, 0, 0, 0);
    };
#pragma unroll
    for (int u = 0; u < PRE; ++u)
        if (g_begin + u < g_end) {
            const int g = g_begin + u;
            if (32 * (8 * g + 8) <= p.k_tap) {  // (uniform)
#pragma unroll
                for (int s = 0; s < 2; ++s) product(expand_f4((uint32_t)a[u][s]), expand_f4(x[u][s]));
            } else {  // K tail: pad bits (and words past cw) must multiply as 0, not as +1
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int nbits = p.k_tap - 32 * (8 * g + first + s);
                    const uint32_t valid = nbits >= 32 ? 0xffffffffu : (nbits <= 0 ? 0u : 0xffffffffu << (32 - nbits));
                    product(expand_f4_masked((uint32_t)a[u][s], valid), expand_f4(x[u][s]));
                }
            }
        }

    // ---- sum the slices (exact integers) in LDS
    int dot[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) dot[v] = (int)acc[v];
    if (blockDim.x > 64) {
        if (wave == 0) {
#pragma unroll
            for (int v = 0; v < 4; ++v) red[v * 64 + lane] = dot[v];
        }
        __syncthreads();
        if (wave != 0) {
#pragma unroll
            for (int v = 0; v < 4; ++v) atomicAdd(&red[v * 64 + lane], dot[v]);
        }
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int v = 0; v < 4; ++v) dot[v] = red[v * 64 + lane];
    }
    // ---- lane (i, q) holds neurons n0 + 4q + v of image b: its four bits, then the half word of the four lanes of an image
    uint32_t bits = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float t = thr[v] != thr[v] ? (p.nan_bit ? -INFINITY : INFINITY) : thr[v];
        bits = __builtin_amdgcn_alignbit(bits, __float_as_uint((float)dot[v] - t), 31);
    }
    bits = (~bits & 15u) << (12 - 4 * q);
    bits |= (uint32_t)__shfl_xor((int)bits, 16);
    bits |= (uint32_t)__shfl_xor((int)bits, 32);
    bits &= 0xffff0000u >> min(max(p.N - n0, 0), 16);
    if (q == 0 && b < p.B) {
        if (nt < p.bits_row_words) reinterpret_cast<uint16_t*>(p.out_bits + (size_t)nt * p.B + b)[1 - half] = (uint16_t)bits;
        if (nt == n_tiles - 1 && half == 0)  // padding words of the 128-padded feature axis
            for (int w = n_tiles; w < p.bits_row_words; ++w) p.out_bits[(size_t)w * p.B + b] = 0;
    }
}

}  // namespace

bool fc_mfma_applicable(const BgemmParams& p) {
    // (a 1 x 1 convolution on a 1 x 1 frame has this shape too, but its filter buffer holds no copy in lane order)
    if (!p.wgt_lane_copy) return false;
    if (p.PH * p.PW != 1 || p.R * p.S != 1 || p.res_in != nullptr || p.res_out != nullptr) return false;
    if (p.mode != EPI_THRESH && p.mode != EPI_AFFINE) return false;
    if (p.cw % 4 != 0 || p.k_tap > 32 * p.cw || 4LL * p.B * (p.cw + 4) >= (1LL << 31)) return false;
    // larger problems fill the machine with one wave per tile and are served by the generic kernel
    const long long tiles = (long long)((p.B + 31) / 32) * ((p.N + 31) / 32);
    return tiles <= 16384;
}

namespace {
constexpr int kCus = 256;       // compute units
constexpr int kSimdWaves = 4;   // waves of these kernels that one of a compute unit's four SIMDs holds (120 registers)
// Split of K over the waves of a workgroup: waves per tile, 8-word groups per wave, and how many groups the
// kernel requests ahead of its first multiply (0: a streaming loop).
struct FcPlan {
    int n_tiles, b_tiles, kwaves, gpw, pre;
    bool staged, small;
};
FcPlan fc_plan(const BgemmParams& p) {
    FcPlan f;
    f.n_tiles = (p.N + 31) / 32;
    f.b_tiles = (p.B + 31) / 32;
    const int groups = (p.cw + 7) / 8;
    // Tiles of 16 x 16 while a compute unit has no more than one of them, slices as long as a wave requests whole, at least three
    // groups each (13 waves are faster than 16 where both hold: sums of fewer).  us, tiles of 32 x 32 -> 16 x 16: 25088 inputs, 512
    // outputs, batch 1 .. 64 7.4 -> 5.1, 128 7.3 -> 5.3, above the line 192 7.3 -> 7.3, 256 7.6 -> 7.7; 32768 -> 512, batch 77 8.3 ->
    // 6.3; 9216 -> 4096, batch 16 4.6 -> 3.9, above 17 4.6 -> 4.7; 8192 -> 1024, batch 64 4.1 -> 3.6, above 100 4.1 -> 4.2.  Under 32
    // such tiles (fewer than 512 outputs at batches to 16) nothing was measured and the kernel of 32 x 32 stays.
    const long long small_tiles = 2LL * f.n_tiles * ((p.B + 15) / 16);
    f.small = p.mode == EPI_THRESH && small_tiles >= 32 && small_tiles <= kCus && groups <= 8 * kMaxWaves;
    if (f.small) {
        f.b_tiles = (p.B + 15) / 16;
        f.gpw = std::max(3, (groups + 12) / 13);
        if (f.gpw > 8) f.gpw = (groups + kMaxWaves - 1) / kMaxWaves;
        f.kwaves = (groups + f.gpw - 1) / f.gpw;
        f.pre = f.gpw <= 4 ? 4 : 8;
        f.staged = false;
        return f;
    }
    // Waves per tile: at least 4 groups (16 k-steps) each, and no more than let every workgroup be resident at once (the kernels hold
    // four waves per SIMD): a second round of workgroups pays for its start and its sums again, while four waves a SIMD keep the VALU
    // busy, which is what binds (14 of its instructions to a product).  Four waves are taken all the same: they end at different times
    // and follow one another.  9216 inputs, 4096 outputs, batch 200: 9 waves in four rounds 13.6 us, 4 in one 9.3 (batch 128: 7.9 ->
    // 5.9, 384: 16.1 -> 12.2 with four waves in two rounds, 14.8 with two in one); 25088 -> 4096, batch 224: 27.0 -> 19.3;
    // 32768 -> 512, batch 544: 16.0 -> 13.7; 16384 -> 2048, batch 256: 10.4 -> 8.9.  A workgroup's waves are counted in fours,
    // one to a SIMD: a fifth is a second wave of one SIMD, which then has as much again to do (513 .. 768 tiles with five waves,
    // three workgroups a compute unit -> four waves, 35 layers: 0.75 .. 0.91 of the time; 8825 -> 3484, batch 212: 10.2 -> 8.3).
    const long long tiles = (long long)f.n_tiles * f.b_tiles;
    int kwaves = std::max(1, std::min(kMaxWaves, groups / 4));
    while (kwaves > 4 && tiles > kCus * (kSimdWaves / ((kwaves + 3) / 4))) --kwaves;
    while (kwaves > 1 && tiles * kwaves > 8192) --kwaves;
    f.gpw = (groups + kwaves - 1) / kwaves;
    f.kwaves = (groups + f.gpw - 1) / f.gpw;
    f.pre = f.gpw <= 2 ? 2 : (f.gpw <= 7 ? 7 : 0);
    // Requests of sixteen bytes a lane where the address units are busy: long slices (25088 inputs, batch 256, 4096 outputs: 32.5 ->
    // 27.7 us; 32768 inputs, 512 outputs, batch 77: 13.2 -> 12.3) and many waves in large workgroups (16384 inputs, 2048 outputs, batch
    // 128, 4096 waves: 5.65 -> 5.5).  With few, the way through LDS only adds to the chain (8192 inputs, 1024 outputs, batch 256, 2048
    // waves: 8.2 -> 8.4), and four workgroups of four waves a CU hide it less (4096 inputs and outputs, batch 200: 5.5 -> 5.8).
    f.staged = f.pre == 0 || (f.pre == 7 && f.kwaves > 4 && tiles * f.kwaves >= 3072);
    return f;
}
}  // namespace

void fc_mfma_kernel_name(const BgemmParams& p, char* buf, size_t len) {
    const FcPlan f = fc_plan(p);
    if (f.small) snprintf(buf, len, "fc_mfma_f4_small_kernel<%d>", f.pre);
    else snprintf(buf, len, "fc_mfma_f4_kernel<%d, %d, %s>", p.mode == EPI_AFFINE ? FC_AFFINE : FC_THRESH, f.pre, f.staged ? "true" : "false");
}

int launch_fc_mfma(const BgemmParams& p, hipStream_t stream) {
    const FcPlan f = fc_plan(p);
    const int n_tiles = f.n_tiles, b_tiles = f.b_tiles, kwaves = f.kwaves, gpw = f.gpw;
    const dim3 grid((unsigned)(n_tiles * b_tiles * (f.small ? 2 : 1))), block(64 * kwaves);
    if (f.small) {
        auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, stream, p, p.act, p.wgt, p.bn, n_tiles, gpw); };
        if (f.pre == 4) launch(fc_mfma_f4_small_kernel<4>);
        else launch(fc_mfma_f4_small_kernel<8>);
        TCBNN_LAUNCH_CHECK("fc_mfma_f4_small_kernel");
        return TCBNN_OK;
    }
    auto launch = [&](auto mode, auto pre, auto staged) {
        constexpr int MODE = decltype(mode)::value, PRE = decltype(pre)::value;
        constexpr bool STAGED = decltype(staged)::value;
        hipLaunchKernelGGL((fc_mfma_f4_kernel<MODE, PRE, STAGED>), grid, block, STAGED ? kwaves * 2048 : 0, stream, p, p.act, p.wgt,
                           MODE == FC_AFFINE ? p.bn_scale : p.bn, MODE == FC_AFFINE ? p.bn_bias : p.bn, n_tiles, gpw);
    };
    auto by_slice = [&](auto mode) {
        if (f.pre == 2) launch(mode, std::integral_constant<int, 2>{}, std::false_type{});
        else if (f.pre == 0) launch(mode, std::integral_constant<int, 0>{}, std::true_type{});
        else if (f.staged) launch(mode, std::integral_constant<int, 7>{}, std::true_type{});
        else launch(mode, std::integral_constant<int, 7>{}, std::false_type{});
    };
    if (p.mode == EPI_AFFINE) by_slice(std::integral_constant<int, FC_AFFINE>{});
    else by_slice(std::integral_constant<int, FC_THRESH>{});
    TCBNN_LAUNCH_CHECK("fc_mfma_f4_kernel");
    return TCBNN_OK;
}

}  // namespace tcbnn
