// A chain of fully connected layers (In128LayerFMT, Fc128LayerFMT, Out128LayerFMT; kernel.cuh:153-280) in one launch.
//
// Launched one by one, the layers of the MLP (784 - 1024 - 1024 - 1024 - 10) are bound by what a launch costs before and after its
// few hundred cycles of products: launch gap, weights' way from L2, one staging of operands, an epilogue, and the activations' way
// through memory.  Images do not meet in such layers, so a workgroup takes 32 images through all of them:
//   - the activations stay in LDS, expanded to FP4 once, when they are made (a fragment is one 16-byte read per lane);
//   - a wave multiplies two tiles of 32 neurons over the whole of K; their weights come from L2 as bits, in the lane
//     order that tcbnn_pack_fc_weight writes (a contiguous KB per 256 of K), four requests ahead, those of the next layer
//     requested before the epilogue of this one;
//   - neurons are the rows of a product and images its columns: a lane finishes an image's sums, and what a sum is too large by
//     (below) is one number per lane;
//   - every layer's output is written, as the layers do it alone.
// The weights are the operand that is expanded on the way (expand_rows_f4: four instructions a word), so the activations are
// expanded as its counterpart, and a sum starts from the negative of the image's constant.
// What binds it: the matrix and vector pipes of a SIMD in turn (they overlap little here).  A 1024 x 1024 layer's 512 products and
// as many expansions per workgroup are 2.6 us, epilogues and starts of tiles 1.2 us more; the signs of the input take 4 us from
// the launch on.  MLP, batch 8192: 42.6 -> 21.4 us a pass (256 workgroups, one per compute unit; 257, at batch 8200: 60.3 -> 36.8).
#include <algorithm>
#include <atomic>

#include "common.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

using namespace mfma;

constexpr int kWaves = 16, kImages = 32;
constexpr int kMaxLayers = 8;
constexpr int kMaxWidth = 2048;  // inputs and outputs of a layer: two layers' activations are 64 KB of LDS
constexpr int kAhead = 4;        // groups (256 of K) of weights requested ahead

struct ChainLayer {
    const v4i* weights;    // in lane order
    const float* scale;    // thresholds, or the output layer's scales
    const float* bias;     // null: thresholds
    void* out;             // bits [KW128(n)][B], or floats [B][n]
    int k, n;
};
struct ChainArgs {
    const float* x;        // first layer's floats [B][k], or null
    const uint32_t* bits;  // ... or its bits [KW128(k)][B]
    uint32_t* x_bits;      // where the floats' signs go
    int B, n_layers, steps;  // steps: K steps of 64 of the widest layer
    ChainLayer layer[kMaxLayers];
};

__host__ __device__ constexpr int groups_of(int k) { return (kw128(k) + 7) / 8; }

typedef float v4f __attribute__((ext_vector_type(4)));

// bits of word w that are among n
__device__ __forceinline__ uint32_t valid_bits(int n, int w) {
    const int left = n - 32 * w;
    return left >= 32 ? ~0u : (left <= 0 ? 0u : ~0u << (32 - left));
}

__global__ __launch_bounds__(64 * kWaves) void fc_chain_kernel(const ChainArgs args) {
    extern __shared__ __align__(16) char lds[];
    v4i* const frags = reinterpret_cast<v4i*>(lds);                      // [2][steps][64]
    int* const shift = reinterpret_cast<int*>(lds + 2 * args.steps * 1024);  // [layer][image]: what its sums are too large by
    float* const par = reinterpret_cast<float*>(shift + kMaxLayers * kImages);          // [wave][thresholds, scales, biases][64]
    uint32_t* const rows = reinterpret_cast<uint32_t*>(par + kWaves * 192);             // [word][33]: the input's signs

    const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b0 = (int)blockIdx.x * kImages, B = args.B;

    // Waves exchange LDS contents only: what they wait for is that, not the outputs' way to memory or the weights' from it.
    auto barrier = [] __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // A layer's weights as a wave requests them: two tiles of 32 neurons, a group (256 of K) of each at a time.  (Always loads, beyond
    // the buffer where there is nothing to load: a load under a condition makes the compiler copy the registers where the
    // paths meet, and wait for the load to do so.)
    struct Source {
        __amdgpu_buffer_rsrc_t rsrc;
        int n_tiles, groups;
    };
    auto source = [](const ChainLayer& l) __attribute__((always_inline)) -> Source {
        const int n_tiles = (l.n + 31) / 32, groups = groups_of(l.k);
        return {__builtin_amdgcn_make_buffer_rsrc(const_cast<v4i*>(l.weights), 0, n_tiles * groups * 1024, 0x00020000), n_tiles, groups};
    };
    v4i w[kAhead][2];
    float scale[2], bias[2];  // of neuron 32 (tile + m) + j
    auto request_group = [&](const Source& l, int tile, int g, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const bool some = g < l.groups && tile + m < l.n_tiles;  // uniform
            w[slot][m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(l.rsrc, (int)((unsigned)(lane * 16) | (some ? 0u : 0x80000000u)),
                                                                                       some ? ((tile + m) * l.groups + g) * 1024 : 0, 0));
        }
    };
    auto request_parameters = [&](const ChainLayer& l, int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int c = min((tile + m) * 32 + j, l.n - 1);
            scale[m] = l.scale[c];
            bias[m] = (l.bias != nullptr ? l.bias : l.scale)[c];
        }
    };
    auto request = [&](const ChainLayer& l) __attribute__((always_inline)) {  // this wave's first two tiles
        const Source of = source(l);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) request_group(of, 2 * wave, u, u);
        request_parameters(l, 2 * wave);
    };
    // A word of activations (neurons or inputs 32 w ...) of an image to the fragments that layer `of` multiplies
    auto put_word = [&](int of, int width, int wi, int image, uint32_t x) __attribute__((always_inline)) {
        const uint32_t valid = valid_bits(width, wi);
        v4i f = expand_weights_f4(x);
        if (valid != ~0u) {
#pragma unroll
            for (int c = 0; c < 4; ++c) f[c] &= (int)((((valid << (3 - c)) & 0x88888888u) >> 3) * 15u);
        }
        const int step = 4 * (wi >> 3) + (wi & 3), half = wi >> 2 & 1;
        frags[((of & 1) * args.steps + step) * 64 + half * 32 + image] = f;
        const uint32_t s = x & valid;
        const int sum = 2 * (5 * __popc(s & 0x11111111u) + 3 * __popc(s & 0x22222222u) + __popc(s & 0x44444444u)) -
                        (5 * __popc(valid & 0x11111111u) + 3 * __popc(valid & 0x22222222u) + __popc(valid & 0x44444444u));
        atomicAdd(&shift[of * kImages + image], sum);
    };

    if (tid < kMaxLayers * kImages) shift[tid] = 0;
    const int k0 = args.layer[0].k, words0 = 8 * groups_of(k0);
    if (args.x != nullptr) {  // uniform
        // signs of two images' rows, 32 words of each at a time; a lane's four inputs are a nibble, eight lanes make a word
        const bool vectors = k0 % 4 == 0 && (reinterpret_cast<uintptr_t>(args.x) & 15u) == 0;
        for (int c = 0; 32 * c < words0; ++c) {
            v4f v[2][4];
            const float* const row[2] = {args.x + (size_t)min(b0 + wave, B - 1) * k0, args.x + (size_t)min(b0 + wave + kWaves, B - 1) * k0};
            const int first = 1024 * c + 4 * lane;
            if (vectors) {  // uniform
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int s = 0; s < 4; ++s) v[i][s] = *reinterpret_cast<const v4f*>(row[i] + min(first + 256 * s, k0 - 4));
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[i][s][e] = row[i][min(first + 256 * s + e, k0 - 1)];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int at = first + 256 * s, wi = 32 * c + 8 * s + (lane >> 3);
                    uint32_t nibble = 0u;
#pragma unroll
                    for (int e = 0; e < 4; ++e) nibble |= at + e < k0 && v[i][s][e] >= 0.0f ? 8u >> e : 0u;
                    uint32_t word = nibble << (28 - 4 * (lane & 7));
                    word |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)word, 0xb1, 0xf, 0xf, false);   // the neighbour's,
                    word |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)word, 0x4e, 0xf, 0xf, false);   // the other pair's,
                    word |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)word, 0x141, 0xf, 0xf, false);  // the other quad's
                    if ((lane & 7) == 0 && wi < words0) rows[wi * 33 + wave + i * kWaves] = word;
                }
        }
    }
    request(args.layer[0]);  // (no sooner: registers)
    barrier();
    for (int e = tid; e < words0 * kImages; e += 64 * kWaves) {
        const int image = e & 31, wi = e >> 5, b = b0 + image;
        uint32_t x = 0u;
        if (args.x != nullptr) {
            x = rows[wi * 33 + image];
            if (wi < kw128(k0) && b < B) args.x_bits[(size_t)wi * B + b] = x;
        } else if (wi < kw128(k0)) {
            x = args.bits[(size_t)wi * B + min(b, B - 1)];
        }
        put_word(0, k0, wi, image, x);
    }
    barrier();

#pragma unroll 1
    for (int l = 0; l < args.n_layers; ++l) {
        const ChainLayer& layer = args.layer[l];
        const int n = layer.n;
        const bool last = l + 1 == args.n_layers, affine = layer.bias != nullptr;  // uniform
        const v4i* const mine = frags + (l & 1) * args.steps * 64 + lane;
        const ChainLayer& next = args.layer[last ? l : l + 1];
        const Source own = source(layer), follows = source(next);
        const int n_tiles = own.n_tiles, groups = own.groups;
#pragma unroll 1
        for (int tile = 2 * wave; tile < n_tiles; tile += 2 * kWaves) {
            const bool more = tile + 2 * kWaves < n_tiles;
            // What the registers of used weights are for: these tiles' further groups, then the wave's next tiles, or the next layer's.
            Source after = more ? own : follows;
            after.n_tiles = more || !last ? after.n_tiles : 0;
            const int after_tile = more ? tile + 2 * kWaves : 2 * wave;
            v16f acc[2];
            // Sums are whole numbers: at or above a threshold is at or above the whole number that it is rounded up to, and one
            // beyond any sum serves for those that are further off (no number: above all).  Sums start from its negative: a bit
            // is a sum's sign.
            {
                // (this wave's own: written and read in order)
                float* const p = par + wave * 192;
                const float t = h ? scale[1] : scale[0];
                const float above = t == t ? __builtin_fminf(__builtin_fmaxf(__builtin_ceilf(t), -2.0f * kMaxWidth), 2.0f * kMaxWidth) : 2.0f * kMaxWidth;
                p[lane] = affine ? 0.0f : above;
                p[64 + lane] = t;
                p[128 + lane] = h ? bias[1] : bias[0];
            }
            const float first = -(float)shift[l * kImages + j];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const v4f* const tp = reinterpret_cast<const v4f*>(par + wave * 192 + 32 * m + 16 * h);
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[m][v] = first - tp[v >> 2][v & 3];
            }
            v4i ahead[4];  // the next group's activations
#pragma unroll
            for (int i = 0; i < 4; ++i) ahead[i] = mine[i * 64];
#pragma unroll 1
            for (int g0 = 0; g0 < groups; g0 += kAhead) {
                const bool final = g0 + kAhead >= groups;  // uniform
#pragma unroll
                for (int u = 0; u < kAhead; ++u) {
                    if (g0 + u < groups) {  // uniform
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const v4i b = ahead[i];
                            ahead[i] = mine[(4 * min(g0 + u + 1, groups - 1) + i) * 64];
#pragma unroll
                            for (int m = 0; m < 2; ++m) acc[m] = Acc<FMT_F4>::mma(expand_rows_f4((uint32_t)w[u][m][i]), b, acc[m]);
                        }
                    }
                    request_group(final ? after : own, final ? after_tile : tile, final ? u : g0 + kAhead + u, u);
                    __builtin_amdgcn_sched_barrier(0);  // (registers)
                }
            }
            if (more || !last) request_parameters(more ? layer : next, after_tile);  // uniform
            if (!affine) {
                // bits, MSB first
                uint32_t word[2];
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    uint32_t below = 0u;
#pragma unroll
                    for (int v = 0; v < 16; ++v) below = __builtin_amdgcn_alignbit(below, __float_as_uint(acc[m][v]), 31);
                    word[m] = ~below & 0xffffu;
                }
                const auto sw = __builtin_amdgcn_permlane32_swap(word[0], word[1], false, false);
                uint32_t full = (sw[0] << 16) | sw[1];  // half m: the word of tile m
                const int wi = tile + h, b = b0 + j;
                if (wi < n_tiles) {
                    full &= valid_bits(n, wi);
                    if (b < B) static_cast<uint32_t*>(layer.out)[(size_t)wi * B + b] = full;
                    if (!last) put_word(l + 1, n, wi, j, full);
                }
            } else {
                const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(static_cast<float*>(layer.out) + (size_t)b0 * n, 0, min(kImages, B - b0) * n * 4, 0x00020000);
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    if (tile + m >= n_tiles) break;  // uniform
                    const v4f* const p = reinterpret_cast<const v4f*>(par + wave * 192 + 64 + 32 * m + 16 * h);
                    const int c = (tile + m) * 32 + 16 * h;
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(__fadd_rn(__fmul_rn(acc[m][v], p[v >> 2][v & 3]), p[16 + (v >> 2)][v & 3])), rsrc,
                                                              c + v < n ? (j * n + c + v) * 4 : (int)0x80000000u, 0, 0);
                }
            }
        }
        // waves without a tile of this layer may have one of the next
        if (2 * wave >= n_tiles && !last) request(next);
        if (!affine) {  // words past the last tile's: 0, and nothing in the next layer's sums
            const int words = 8 * groups_of(n);
            for (int e = n_tiles * kImages + tid; e < words * kImages; e += 64 * kWaves) {
                const int image = e & 31, wi = e >> 5, b = b0 + image;
                if (wi < kw128(n) && b < B) static_cast<uint32_t*>(layer.out)[(size_t)wi * B + b] = 0u;
                if (!last) frags[(((l + 1) & 1) * args.steps + 4 * (wi >> 3) + (wi & 3)) * 64 + (wi >> 2 & 1) * 32 + image] = v4i{0, 0, 0, 0};
            }
        }
        barrier();
    }
}

bool fits(int batch, int k, int n) { return batch > 0 && k > 0 && n > 0 && k <= kMaxWidth && n <= kMaxWidth; }

// Whether one launch is faster than one per layer, by what it saves (us), fitted to both sides' times of 380 runs (1 to 5 layers,
// 10 to 2048 wide, batch 1 to 16384, launched on end; the layers' own launches have got faster since, with tiles of 16 x 16 and
// large outputs four values a request).  A launch of its own costs a layer 1.75 us more than its share of this one, the
// input's signs 0.7 and more where there is more to read, and this launch has 3.6 of its own.  A workgroup does a layer's products
// for its 32 images on one compute unit, 1.85 us longer for 1024 x 1024 of them than all units together where there are few images, and
// less where there are many; a layer of 4096 tiles or more is 2.4 us slower by itself; an output layer stores a number at a
// time (14 us for 1000 of 32 images); and beyond 8192 images workgroups wait for a compute unit.
// us, a launch per layer and here: the MLP, batch 1 / 256 / 8192: 17.5 / 19.5 / 45.1 and 17.6 / 18.0 / 20.5; 1408 wide, batch 256 /
// 1024 / 1536: 21.5 / 25.1 / 28.5 and 25.4 / 25.4 / 25.5; 2048 wide, batch 256 / 1536 / 2048: 21.2 / 32.2 / 40.6 and 36.3 / 36.6 / 37.0;
// the last two layers of CIFAR VGG (1024 x 1024, 1024 x 10), batch 256 / 1024 / 2048 / 4096: 7.2 / 7.4 / 8.1 / 12.6 and 8.8 / 8.9 / 9.0 / 9.2.
struct Work {
    int inputs;           // of the signs; 0: none
    int layers;           // besides the signs
    double products;      // in 1024 x 1024
    int large;            // layers of 4096 tiles or more
    int numbers;          // outputs that are numbers
};
bool pays(const Work& w, int batch) {
    const double x = std::min(batch, 8192) / 1024.0, read = (double)w.inputs * batch / (1024 * 1024);
    const double saved = 1.75 * w.layers + (w.inputs > 0 ? 0.7 + 0.0029 * w.inputs : 0.0) - 3.6 + w.products * (0.48 * x - 1.85) + 2.4 * w.large -
                         0.014 * w.numbers * std::min(batch, 16) / 16 * std::max(0.0, 1.0 - x / 6);
    return saved + (batch > 8192 ? 1.1 * read - 7.0 : 0.0) >= 0.0;
}

// The memory of a run's layers.  Launched one by one, a layer may write where an earlier one has read or written (two buffers in
// turn); in one launch nothing orders the waves and workgroups of different layers but LDS, so every output has to be apart
// from all else that the run reads and writes, except as the input of the layer that follows.
class Memory {
   public:
    // A layer that reads `n` ranges besides the output of the one before it; false: it has to have a launch of its own
    struct Range {
        const void* at;
        size_t bytes;
    };
    bool add(const Range* reads, int n, const Range& write) {
        bool apart = true;
        for (int i = 0; i < n; ++i) apart &= !meets(reads[i], writes_, n_writes_) && !meets(reads[i], &write, 1);
        apart &= !meets(write, reads_, n_reads_) && !meets(write, writes_, n_writes_);
        if (!apart) return false;
        for (int i = 0; i < n; ++i) reads_[n_reads_++] = reads[i];
        writes_[n_writes_++] = write;
        return true;
    }

   private:
    static bool meets(const Range& r, const Range* of, int n) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(r.at);
        for (int i = 0; i < n; ++i) {
            const uintptr_t b = reinterpret_cast<uintptr_t>(of[i].at);
            if (a < b ? b - a < r.bytes : a - b < of[i].bytes) return true;
        }
        return false;
    }
    Range reads_[3 * kMaxLayers + 1], writes_[kMaxLayers + 1];
    int n_reads_ = 0, n_writes_ = 0;
};

// The layers from fc[0] on that one launch can take (0: none, or the chain is not worth one)
int chain_length(const tcbnn_in128_desc* in, const tcbnn_fc128_desc* fc, int n_fc, const tcbnn_out128_desc* out, bool* with_out) {
    *with_out = false;
    auto usable = [](const void* a, const void* b, const void* c, const void* d) { return a != nullptr && b != nullptr && c != nullptr && d != nullptr; };
    auto bits = [](const void* at, int batch, int n) { return Memory::Range{at, 4 * tcbnn_fc_act_words(batch, n)}; };
    auto weights = [](const void* at, int k, int n) { return Memory::Range{at, 4 * tcbnn_fc_weight_words(k, n)}; };
    auto floats = [](const void* at, int rows, int n) { return Memory::Range{at, (size_t)4 * rows * n}; };
    Memory memory;
    if (in != nullptr) {
        if (in->input == nullptr || in->output != fc[0].input || in->input_height != fc[0].input_height || in->input_width != fc[0].input_width ||
            !fits(in->input_height, in->input_width, 1))
            return 0;
        const Memory::Range x = floats(in->input, in->input_height, in->input_width);
        if (!memory.add(&x, 1, bits(in->output, in->input_height, in->input_width))) return 0;
    }
    int n = 0;
    for (; n < n_fc && n < kMaxLayers; ++n) {
        const tcbnn_fc128_desc& f = fc[n];
        if (!usable(f.input, f.weight, f.bn, f.output) || !fits(f.input_height, f.input_width, f.weight_width) ||
            resolve_variant(f.variant) != TCBNN_VARIANT_MFMA_F4)
            break;
        if (n > 0 && (f.input != fc[n - 1].output || f.input_height != fc[0].input_height || f.input_width != fc[n - 1].weight_width)) break;
        const Memory::Range reads[3] = {weights(f.weight, f.input_width, f.weight_width), floats(f.bn, 1, f.weight_width), bits(f.input, f.input_height, f.input_width)};
        if (!memory.add(reads, n == 0 && in == nullptr ? 3 : 2, bits(f.output, f.input_height, f.weight_width))) break;
    }
    if (n == 0) return 0;
    const int batch = fc[0].input_height;
    Work work{in != nullptr ? in->input_width : 0, 0, 0.0, 0, 0};
    auto count = [&](int k, int outputs) {
        ++work.layers;
        work.products += (double)k * outputs / (1024 * 1024);
        work.large += (long long)((batch + 31) / 32) * ((outputs + 31) / 32) >= 4096;
    };
    for (int i = 0; i < n; ++i) count(fc[i].input_width, fc[i].weight_width);
    *with_out = out != nullptr && n == n_fc && n < kMaxLayers && usable(out->input, out->weight, out->bn_scale, out->output) && out->bn_bias != nullptr &&
                fits(out->input_height, out->input_width, out->weight_width) && resolve_variant(out->variant) == TCBNN_VARIANT_MFMA_F4 &&
                out->input == fc[n - 1].output && out->input_height == fc[0].input_height && out->input_width == fc[n - 1].weight_width;
    if (*with_out) {
        const Memory::Range reads[3] = {weights(out->weight, out->input_width, out->weight_width), floats(out->bn_scale, 1, out->weight_width), floats(out->bn_bias, 1, out->weight_width)};
        *with_out = memory.add(reads, 3, floats(out->output, out->input_height, out->weight_width));
    }
    if (*with_out) {
        count(out->input_width, out->weight_width);
        work.numbers = out->weight_width;
    }
    return work.layers + (in != nullptr ? 1 : 0) >= 2 && pays(work, batch) ? n : 0;
}

int launch_chain(const tcbnn_in128_desc* in, const tcbnn_fc128_desc* fc, int n_fc, const tcbnn_out128_desc* out, hipStream_t stream) {
    ChainArgs a{};
    int widest = 0;
    auto lanes = [](const uint32_t* weight, int k, int n) { return reinterpret_cast<const v4i*>(weight + fc_weight_row_words(pad32(n), kw128(k))); };
    for (int i = 0; i < n_fc; ++i) {
        a.layer[i] = {lanes(fc[i].weight, fc[i].input_width, fc[i].weight_width), fc[i].bn, nullptr, fc[i].output, fc[i].input_width, fc[i].weight_width};
        widest = std::max(widest, std::max(fc[i].input_width, fc[i].weight_width));
    }
    a.n_layers = n_fc;
    if (out != nullptr) a.layer[a.n_layers++] = {lanes(out->weight, out->input_width, out->weight_width), out->bn_scale, out->bn_bias, out->output, out->input_width, out->weight_width};
    a.x = in != nullptr ? in->input : nullptr;
    a.x_bits = in != nullptr ? in->output : nullptr;
    a.bits = fc[0].input;
    a.B = fc[0].input_height;
    a.steps = 4 * groups_of(widest);
    const size_t bytes = (size_t)2 * a.steps * 1024 + kMaxLayers * kImages * 4 + kWaves * 192 * 4 + (in != nullptr ? (size_t)8 * groups_of(fc[0].input_width) * 33 * 4 : 0);
    if (bytes > 64 * 1024) {
        constexpr int kMaxDevices = 64;
        static std::atomic<bool> ready[kMaxDevices];  // (setting the limit twice does no harm)
        int dev = 0;
        if (int rc = check_hip(hipGetDevice(&dev), "hipGetDevice")) return rc;
        if (dev < 0 || dev >= kMaxDevices) return fail(TCBNN_EUNSUPPORTED, "fc_chain: device ordinal %d", dev);
        if (!ready[dev].load(std::memory_order_acquire)) {
            if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&fc_chain_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024),
                                   "hipFuncSetAttribute(MaxDynamicSharedMemorySize)"))
                return rc;
            ready[dev].store(true, std::memory_order_release);
        }
    }
    hipLaunchKernelGGL(fc_chain_kernel, dim3((unsigned)((a.B + kImages - 1) / kImages)), dim3(64 * kWaves), bytes, stream, a);
    TCBNN_LAUNCH_CHECK("fc_chain_kernel");
    return TCBNN_OK;
}

// The launches of a run, in order: chain(in, fc, n_fc, out) for one of several layers, single(in, fc, out), one of them not null
template <typename Chain, typename Single>
int each_launch(const tcbnn_in128_desc* in, const tcbnn_fc128_desc* fc, int n_fc, const tcbnn_out128_desc* out, const Chain& chain, const Single& single) {
    TCBNN_REQUIRE(n_fc >= 0 && (n_fc == 0 || fc != nullptr), "fc_chain: no layers");
    bool with_out = false;
    for (int i = 0; i <= n_fc;) {
        const tcbnn_in128_desc* const first = i == 0 ? in : nullptr;
        const int n = i < n_fc ? chain_length(first, fc + i, n_fc - i, out, &with_out) : 0;
        if (n > 0) {
            if (int rc = chain(first, fc + i, n, with_out ? out : nullptr)) return rc;
            i += n;
            if (with_out) return TCBNN_OK;
            continue;
        }
        if (first != nullptr)
            if (int rc = single(first, nullptr, nullptr)) return rc;
        if (i < n_fc) {
            if (int rc = single(nullptr, fc + i, nullptr)) return rc;
        } else if (out != nullptr) {
            return single(nullptr, nullptr, out);
        }
        ++i;
    }
    return TCBNN_OK;
}

}  // namespace
}  // namespace tcbnn

using namespace tcbnn;

extern "C" int tcbnn_fc_chain_forward(const tcbnn_in128_desc* in, const tcbnn_fc128_desc* fc, int n_fc, const tcbnn_out128_desc* out, void* stream) {
    return each_launch(
        in, fc, n_fc, out,
        [&](const tcbnn_in128_desc* i, const tcbnn_fc128_desc* f, int n, const tcbnn_out128_desc* o) { return launch_chain(i, f, n, o, (hipStream_t)stream); },
        [&](const tcbnn_in128_desc* i, const tcbnn_fc128_desc* f, const tcbnn_out128_desc* o) {
            return i != nullptr ? tcbnn_in128_forward(i, stream) : (f != nullptr ? tcbnn_fc128_forward(f, stream) : tcbnn_out128_forward(o, stream));
        });
}

extern "C" int tcbnn_fc_chain_plan(const tcbnn_in128_desc* in, const tcbnn_fc128_desc* fc, int n_fc, const tcbnn_out128_desc* out, int* layers, int* n_launches) {
    TCBNN_REQUIRE(layers != nullptr && n_launches != nullptr, "fc_chain: NULL pointer");
    int n = 0;
    const int rc = each_launch(
        in, fc, n_fc, out,
        [&](const tcbnn_in128_desc* i, const tcbnn_fc128_desc*, int n_layers, const tcbnn_out128_desc* o) {
            layers[n++] = n_layers + (i != nullptr) + (o != nullptr);
            return (int)TCBNN_OK;
        },
        [&](const tcbnn_in128_desc*, const tcbnn_fc128_desc*, const tcbnn_out128_desc*) {
            layers[n++] = 1;
            return (int)TCBNN_OK;
        });
    *n_launches = n;
    return rc;
}
