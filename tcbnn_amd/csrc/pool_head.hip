// Layers of the textbook ResNet wiring that the reference's drivers do not have: overlapping
// OR / max pooling of a packed activation tensor with its residual, and the global-average-pool +
// fp32 fully connected head.  The pooling is one pass over its input; the head is latency (below).
#include <algorithm>

#include "common.h"

namespace tcbnn {
namespace {

constexpr int kThreads = 256;

struct PoolParams {
    const uint32_t* in;
    uint32_t* out;
    const int32_t* rin;
    int32_t* rout;
    int H, W, C, B, OH, OW, cw, groups;  // groups = 16-byte residual groups per pixel
    int window, stride, pad, fmt;
};

// One thread per (output pixel, word or residual group, image); the image index runs fastest,
// so a wavefront reads and writes contiguous runs.
__global__ __launch_bounds__(kThreads) void pool128_kernel(const PoolParams p) {
    const long long per_pix = (long long)(p.cw + p.groups) * p.B;
    const long long idx = (long long)blockIdx.x * kThreads + threadIdx.x;
    if (idx >= per_pix * p.OH * p.OW) return;
    const int opix = (int)(idx / per_pix);
    const int rem = (int)(idx % per_pix);
    const int u = rem / p.B, b = rem % p.B;  // unit (word, then group) and image
    const int oy = opix / p.OW, ox = opix % p.OW;
    const int y0 = oy * p.stride - p.pad, x0 = ox * p.stride - p.pad;
    if (u < p.cw) {  // OR of the window's words
        uint32_t acc = 0;
        for (int r = 0; r < p.window; ++r)
            for (int s = 0; s < p.window; ++s) {
                const int y = y0 + r, x = x0 + s;
                if (y >= 0 && y < p.H && x >= 0 && x < p.W) acc |= p.in[(((size_t)y * p.W + x) * p.cw + u) * p.B + b];
            }
        p.out[((size_t)opix * p.cw + u) * p.B + b] = acc;
        return;
    }
    const int g = u - p.cw;  // maximum of the window's residual groups
    if (p.fmt == TCBNN_RES_I12) {  // groups of 16 channels, unpacked to ints and packed again
        int m[16], v[16];
        bool none = true;
        for (int r = 0; r < p.window; ++r)
            for (int s = 0; s < p.window; ++s) {
                const int y = y0 + r, x = x0 + s;
                if (y < 0 || y >= p.H || x < 0 || x >= p.W) continue;
                residual_load_group16(p.rin, p.fmt, (size_t)y * p.W + x, p.C, g, p.B, b, v);
#pragma unroll
                for (int e = 0; e < 16; ++e) m[e] = none ? v[e] : max(m[e], v[e]);
                none = false;
            }
        if (none)
#pragma unroll
            for (int e = 0; e < 16; ++e) m[e] = 0;
        residual_store_group16(p.rout, p.fmt, (size_t)opix, p.C, g, p.B, b, m);
        return;
    }
    const int4* __restrict__ src = reinterpret_cast<const int4*>(p.rin);
    int4 m;
    bool first = true;
    for (int r = 0; r < p.window; ++r)
        for (int s = 0; s < p.window; ++s) {
            const int y = y0 + r, x = x0 + s;
            if (y < 0 || y >= p.H || x < 0 || x >= p.W) continue;
            const int4 v = src[(((size_t)y * p.W + x) * p.groups + g) * p.B + b];
            if (first) {
                m = v;
                first = false;
            } else if (p.fmt == TCBNN_RES_I16) {  // two int16 per word
                auto max2 = [](int a, int c) {
                    const int lo = max((int)(short)(a & 0xffff), (int)(short)(c & 0xffff));
                    const int hi = max(a >> 16, c >> 16);
                    return (lo & 0xffff) | (hi << 16);
                };
                m = make_int4(max2(m.x, v.x), max2(m.y, v.y), max2(m.z, v.z), max2(m.w, v.w));
            } else {
                m = make_int4(max(m.x, v.x), max(m.y, v.y), max(m.z, v.z), max(m.w, v.w));
            }
        }
    if (first) m = make_int4(0, 0, 0, 0);  // window entirely outside the frame (cannot happen: padding < window)
    reinterpret_cast<int4*>(p.rout)[((size_t)opix * p.groups + g) * p.B + b] = m;
}

// ---- 3x3 window, stride 2 (the textbook wiring's only pooling layer) -------------------------------------------------
// A 12-bit residual's maximum is taken on packed 16-bit halves that hold a value each in their upper 12 bits; whatever
// lies in the lower four only decides between equal values.
typedef short v2s __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t max2x16(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(v2s, a), __builtin_bit_cast(v2s, b)));
}
// words w0..w2 of eight 12-bit values -> four pairs, and back
__device__ __forceinline__ void i12_to_pairs(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t* q) {
    constexpr uint32_t kLow = 0x0000ffffu;
    auto pair = [](uint32_t low_at_4, uint32_t high_at_20) { return (low_at_4 & kLow) | (high_at_20 & ~kLow); };
    q[0] = pair(w0 << 4, w0 << 8);
    q[1] = pair(__builtin_amdgcn_alignbit(w1, w0, 20), w1 << 16);
    q[2] = pair(w1 >> 12, __builtin_amdgcn_alignbit(w2, w1, 8));
    q[3] = pair(w2 >> 4, w2);
}
__device__ __forceinline__ void i12_from_pairs(const uint32_t* q, uint32_t& w0, uint32_t& w1, uint32_t& w2) {
    int v[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[2 * k] = (int)(q[k] >> 4);
        v[2 * k + 1] = (int)(q[k] >> 20);
    }
    i12_pack8(v, w0, w1, w2);
}

// A thread takes one unit (word of bits, or residual group) of one image and a few output pixels of a column: of the three input
// rows of a window the last is the next window's first.  A pixel's address is scalar and a lane's place in it 32 bits.
// Neighbouring windows share a column and runs of outputs a row, and an XCD's L2 has what they share where the XCD takes them all:
// asked for by several XCDs it came from memory again.  Workgroups are dealt
//   TURN          in turn, an output pixel's units first, as many rows a thread as leave every SIMD eight waves (8 at most).  With a
//                 multiple of eight workgroups a pixel an XCD has the same units of every pixel, all that they share with it: us, dealt
//                 as below -> in turn, 256 channels at 27x27, batch 256, 16-bit 23.4 -> 20.4, 56x56 in 32 bits 215 -> 205.  Few
//                 outputs (under four waves a SIMD), whose input the caches have: 32 channels in 12 bits at 56x56, batch 8 5.9 -> 3.9.
//                 Bits alone, a word a thread, to which the division of the shares and a short walk cost more than they save: 64
//                 channels at 112x112, batch 256 10.6 -> 8.2;
//   ROWS          the others in runs of neighbours to an XCD, two rows a thread (more: fewer, longer chains): whole rows of outputs,
//                 an XCD reads what no other one does;
//   COLUMNS       a part of each row, all XCDs at the same row: better where the launch's bytes are more than the memory-side cache has
//                 room for beside its producer's (us in the textbook wiring's pass, batch 64 / 90 / 110 / 128 / 200 / 256: 17.7 / 28.4 / 39.1 /
//                 45.6 / 74.1 / 99.0 in ROWS, 19.7 / 29.7 / 37.9 / 42.3 / 69.7 / 94.0 in COLUMNS);
//   COLUMNS_BACK  the same, last rows first, where the input alone is more than that cache (256 MiB): what was written last is still
//                 in it (batch 256 91.3; 200, whose input fits, 70.7).
// (The lines between the last three are from that pass: 64 channels, 12 bits, a producer that goes down the rows.)
// In the pass, with eight rows a thread and all dealt in turn -> here: batch 32 14.8 -> 10.2, 64 26.3 -> 17.7, 128 49.4 -> 42.3, 256
// 97.8 -> 91.3 (417 MB, while the producer's last stores are on their way: on its own 79, 5.3 TB/s).  What binds it: memory.
// (Asking for the next output's words while one is reduced: 3 % slower below batch 256, 4 % faster there.)
enum PoolOrder : int { ROWS = 0, COLUMNS = 1, COLUMNS_BACK = 2, TURN = 3 };
constexpr int kPoolRows = 2;             // output rows a thread takes in the orders but TURN
constexpr long long kPoolFew = 1 << 18;  // outputs' units: four waves for each of 1024 SIMDs
template <int FMT>
__global__ __launch_bounds__(kThreads) void pool3x3s2_kernel(const PoolParams p, int units, int per_xcd, PoolOrder order, int rows) {
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    int bx, ox, pair;  // workgroup of a pixel, column, run of rows
    if (order == TURN) {
        bx = (int)blockIdx.x, ox = (int)blockIdx.y, pair = (int)blockIdx.z;
    } else {
        // workgroup i of an XCD's share of turn z (a row of the grid's last dimension); units, then columns, then pairs of rows
        const int xcd = (int)blockIdx.x & 7, i = (int)(blockIdx.x >> 3) + (int)(gridDim.x >> 3) * (int)blockIdx.y, z = (int)blockIdx.z;
        if (i >= per_xcd) return;
        const int pairs = (int)gridDim.z, share = (order == ROWS ? xcd * pairs + z : xcd) * per_xcd + i;
        const int col = uniform(share / units), row = order == ROWS ? uniform(col / p.OW) : 0;
        bx = share - col * units, ox = col - row * p.OW;
        pair = order == ROWS ? row : (order == COLUMNS ? z : pairs - 1 - z);
        if (ox >= p.OW || pair >= pairs) return;  // (shares are rounded up)
    }
    const int oy0 = pair * rows, oy1 = min(p.OH, oy0 + rows);
    const unsigned rem = (unsigned)bx * kThreads + threadIdx.x;
    if (rem >= (unsigned)((p.cw + p.groups) * p.B)) return;
    const unsigned u = rem / (unsigned)p.B, b = rem - u * (unsigned)p.B;
    const int x0 = ox * 2 - p.pad;
    // columns outside the frame repeat one inside it (padding < window: there is one)
    int xs[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) xs[s] = min(max(x0 + s, max(x0, 0)), min(x0 + 2, p.W - 1));
    if (u < (unsigned)p.cw) {  // OR of the window's words
        const unsigned at = u * (unsigned)p.B + b;
        const size_t px = (size_t)p.cw * p.B;
        auto row = [&](int y) {
            uint32_t v = 0u;
            if (y >= 0 && y < p.H)
#pragma unroll
                for (int s = 0; s < 3; ++s) v |= (p.in + ((size_t)y * p.W + xs[s]) * px)[at];
            return v;
        };
        uint32_t last = row(oy0 * 2 - p.pad);
        for (int oy = oy0; oy < oy1; ++oy) {
            const int y = oy * 2 - p.pad;
            const uint32_t mid = row(y + 1), next = row(y + 2);
            (p.out + ((size_t)oy * p.OW + ox) * px)[at] = last | mid | next;
            last = next;
        }
        return;
    }
    const unsigned g = u - (unsigned)p.cw;
    constexpr bool kI12 = FMT == TCBNN_RES_I12;
    constexpr int kQ = kI12 ? 8 : 4;  // registers of a group: pairs, or the four words
    // a lane's bytes of a pixel: sixteen, and eight more of twelve-bit groups
    const unsigned at = kI12 ? (g * 6u * (unsigned)p.B + b * 4u) * 4u : (g * (unsigned)p.B + b) * 16u;
    const unsigned at8 = (g * 6u * (unsigned)p.B + (unsigned)p.B * 4u + b * 2u) * 4u;
    const size_t px = (size_t)p.groups * p.B * (kI12 ? 24 : 16);
    struct Words {  // three pixels of a row, as they lie in memory
        uint4 a[3];
        uint2 c[kI12 ? 3 : 1];
    };
    struct Group {
        uint32_t q[kQ];
    };
    auto most = [](const Group& a, const Group& c) __attribute__((always_inline)) {
        Group m;
#pragma unroll
        for (int k = 0; k < kQ; ++k)
            m.q[k] = FMT == TCBNN_RES_I32 ? (uint32_t)max((int)a.q[k], (int)c.q[k]) : max2x16(a.q[k], c.q[k]);
        return m;
    };
    // (rows outside the frame repeat the nearest row inside, which is in the window: padding < window)
    auto request = [&](int y, int oy, Words& w) __attribute__((always_inline)) {
        const int yc = min(max(y, max(0, oy * 2 - p.pad)), min(p.H - 1, oy * 2 - p.pad + 2));
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const char* const pix = reinterpret_cast<const char*>(p.rin) + ((size_t)yc * p.W + xs[s]) * px;
            w.a[s] = *reinterpret_cast<const uint4*>(pix + at);
            if constexpr (kI12) w.c[s] = *reinterpret_cast<const uint2*>(pix + at8);
        }
    };
    auto reduce = [&](const Words& w) __attribute__((always_inline)) {
        Group r[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            if constexpr (kI12) {
                i12_to_pairs(w.a[s].x, w.a[s].y, w.a[s].z, r[s].q);
                i12_to_pairs(w.a[s].w, w.c[s].x, w.c[s].y, r[s].q + 4);
            } else {
                r[s].q[0] = w.a[s].x, r[s].q[1] = w.a[s].y, r[s].q[2] = w.a[s].z, r[s].q[3] = w.a[s].w;
            }
        }
        return most(most(r[0], r[1]), r[2]);
    };
    Words first;
    request(oy0 * 2 - p.pad, oy0, first);
    Group last = reduce(first);
    for (int oy = oy0; oy < oy1; ++oy) {
        const int y = oy * 2 - p.pad;
        Words mid, next;
        request(y + 1, oy, mid);
        request(y + 2, oy, next);
        const Group upper = most(last, reduce(mid));
        last = reduce(next);
        const Group m = most(upper, last);
        char* const pix = reinterpret_cast<char*>(p.rout) + ((size_t)oy * p.OW + ox) * px;
        if constexpr (kI12) {
            uint32_t d[6];
            i12_from_pairs(m.q, d[0], d[1], d[2]);
            i12_from_pairs(m.q + 4, d[3], d[4], d[5]);
            *reinterpret_cast<uint4*>(pix + at) = make_uint4(d[0], d[1], d[2], d[3]);
            *reinterpret_cast<uint2*>(pix + at8) = make_uint2(d[4], d[5]);
        } else {
            *reinterpret_cast<uint4*>(pix + at) = make_uint4(m.q[0], m.q[1], m.q[2], m.q[3]);
        }
    }
}

struct HeadParams {
    const int32_t* rin;
    const float* w;
    const float* bias;
    float* out;
    int P, C, B, N, groups, fmt;  // P = pixels
};

constexpr int kHeadImages = 8;     // images per workgroup
constexpr int kHeadOutputs = 128;  // outputs per workgroup: a thread takes one of them for two of the images
constexpr int kHeadThreads = kHeadOutputs * kHeadImages / 2;
constexpr int kHeadMaxC = 512;
constexpr int kHeadChunk = 32;     // channels whose weights are laid out in LDS at a time
constexpr int kHeadAhead = 2;      // chunks requested ahead

// Sixteen channels of a thread's output and two images: means lie one channel per lane of each row of 16 (all rows the same), and
// a multiply-add takes its channel's by DPP.  (As asm because the compiler moves the lane's value first, in an instruction of
// its own; the wait states are those between a write of m and a DPP read of it.)
#define TCBNN_HEAD_CHANNEL(K, LANE)                                                        \
    "v_fmac_f32_dpp %0, %2, %" #K " row_newbcast:" #LANE " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %1, %3, %" #K " row_newbcast:" #LANE " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void head_channels(const float2& m, const float (&w)[16], float (&acc)[2]) {
    asm("s_nop 1\n\t" TCBNN_HEAD_CHANNEL(4, 0) TCBNN_HEAD_CHANNEL(5, 1) TCBNN_HEAD_CHANNEL(6, 2) TCBNN_HEAD_CHANNEL(7, 3)
            TCBNN_HEAD_CHANNEL(8, 4) TCBNN_HEAD_CHANNEL(9, 5) TCBNN_HEAD_CHANNEL(10, 6) TCBNN_HEAD_CHANNEL(11, 7)
                TCBNN_HEAD_CHANNEL(12, 8) TCBNN_HEAD_CHANNEL(13, 9) TCBNN_HEAD_CHANNEL(14, 10) TCBNN_HEAD_CHANNEL(15, 11)
                    TCBNN_HEAD_CHANNEL(16, 12) TCBNN_HEAD_CHANNEL(17, 13) TCBNN_HEAD_CHANNEL(18, 14) TCBNN_HEAD_CHANNEL(19, 15)
        : "+&v"(acc[0]), "+&v"(acc[1])
        : "v"(m.x), "v"(m.y), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]),
          "v"(w[10]), "v"(w[11]), "v"(w[12]), "v"(w[13]), "v"(w[14]), "v"(w[15]));
}

// Workgroup = 8 images x 128 outputs.  Phase 1: the means of the 8 images, all channels, into LDS.  Phase 2: a thread
// takes one output of two images: per channel a weight from LDS and two fused multiply-adds, channels in ascending order.
// Everything here is latency: a chain of C multiply-adds behind the pixels' way from memory and the fetch of the code, which runs
// once.  So the grid is as many workgroups as CUs at batch 256, two waves to a SIMD (with one, 256 threads and four images each,
// the means took 10 us and the products 11), and the pixels' loop is rolled (all 49 of a 7x7 map unrolled: 27.7 us for 23.8).
// Weights come from memory sixteen bytes a lane, two channels a request, two chunks of 32 channels ahead, and are shared through
// LDS: the address unit takes 17 cycles for a request whatever its size, and eight waves that each ask for a channel's 256 bytes
// at a time would keep it busy for 30 us.  A group of 16 channels' means is one read, a channel to a lane of each row of 16, and a
// multiply-add takes its lane's by DPP: read per channel they would keep LDS busy for 7 us.
// 7x7x512 -> 1000, events around one launch in a pass, us, 256 threads with weights straight from memory -> here: batch 1 23.6 -> 18.8,
// 50 29.1 -> 22.4, 128 27.5 -> 21.0, 256 30.5 -> 23.8.
template <int FMT>
__global__ __launch_bounds__(kHeadThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void avgpool_fc_kernel(const HeadParams p) {
    constexpr int kPer = (int)residual_group_channels(FMT);
    constexpr int kPixels = 17;  // requested together (integer sums: the order does not matter)
    __shared__ __align__(16) float mean[kHeadMaxC][kHeadImages];
    const int tid = threadIdx.x;
    const int b0 = blockIdx.x * kHeadImages;
    const int n = blockIdx.y * kHeadOutputs + (tid & (kHeadOutputs - 1)), i0 = tid / kHeadOutputs * 2;
    __shared__ __align__(16) float weights[2][kHeadChunk][kHeadOutputs];
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    // A chunk: 32 threads to a channel's 128 outputs (past the last one: the next channel's, or zeros; not stored).  Past the last
    // channel: zeros.  A buffer is one chunk (128 N bytes: 2^31 is out of reach of a grid's second dimension).
    const int w_at = ((tid >> 5) * p.N + (int)blockIdx.y * kHeadOutputs + (tid & 31) * 4) * 4;
    v4u ahead[kHeadAhead][2];
    float* next = const_cast<float*>(p.w);
    int left = p.C;
    auto request = [&](int slot) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc(next, 0, min(kHeadChunk, max(0, left)) * p.N * 4, 0x00020000);
        next += (size_t)kHeadChunk * p.N;
        left -= kHeadChunk;
#pragma unroll
        for (int q = 0; q < 2; ++q) ahead[slot][q] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, w_at + q * 16 * p.N * 4, 0, 0);
    };
    auto lay_out = [&](int chunk, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 2; ++q) *reinterpret_cast<v4u*>(&weights[chunk & 1][(tid >> 5) + 16 * q][(tid & 31) * 4]) = ahead[slot][q];
    };
#pragma unroll
    for (int k = 0; k < kHeadAhead; ++k) request(k);

    const float npix = (float)p.P;
    const size_t pixel_b = (size_t)p.groups * residual_group_bytes(FMT) * p.B;
    for (int u = tid; u < p.groups * kHeadImages; u += kHeadThreads) {
        const int g = u / kHeadImages, i = u % kHeadImages;  // image fastest: 128-byte runs
        const unsigned bb = (unsigned)min(b0 + i, p.B - 1);
        const unsigned lane = (unsigned)g * (unsigned)residual_group_bytes(FMT) * (unsigned)p.B + bb * 16u;
        const unsigned lane8 = (unsigned)g * 24u * (unsigned)p.B + (unsigned)p.B * 16u + bb * 8u;
        int sum[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) sum[k] = 0;
#pragma unroll 1
        for (int pix0 = 0; pix0 < p.P; pix0 += kPixels) {
            uint4 v[kPixels];
            uint2 v2[FMT == TCBNN_RES_I12 ? kPixels : 1];
            const char* at = reinterpret_cast<const char*>(p.rin) + (size_t)pix0 * pixel_b;
#pragma unroll
            for (int q = 0; q < kPixels; ++q) {
                v[q] = *reinterpret_cast<const uint4*>(at + lane);
                if constexpr (FMT == TCBNN_RES_I12) v2[q] = *reinterpret_cast<const uint2*>(at + lane8);
                if (pix0 + q + 1 < p.P) at += pixel_b;  // (past the last pixel: the last one again, not added)
            }
            auto add = [&](int q) {
                if constexpr (FMT == TCBNN_RES_I12) {
                    int e[16];
                    i12_unpack8(v[q].x, v[q].y, v[q].z, e);
                    i12_unpack8(v[q].w, v2[q].x, v2[q].y, e + 8);
#pragma unroll
                    for (int k = 0; k < kPer; ++k) sum[k] += e[k];
                } else {
                    const int wv[4] = {(int)v[q].x, (int)v[q].y, (int)v[q].z, (int)v[q].w};
#pragma unroll
                    for (int k = 0; k < kPer; ++k)
                        sum[k] += FMT == TCBNN_RES_I32 ? wv[k % 4] : (k % 2 == 0 ? (int)(short)(wv[k / 2] & 0xffff) : wv[k / 2] >> 16);
                }
            };
#pragma unroll
            for (int q = 0; q < kPixels; ++q)
                if (pix0 + q < p.P) add(q);  // uniform
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            if (g * kPer + k < p.C) mean[g * kPer + k][i] = (float)sum[k] / npix;
    }
    float acc[2] = {0.0f, 0.0f};
    const int col = tid & (kHeadOutputs - 1), chunks = (p.C + kHeadChunk - 1) / kHeadChunk;
    for (int k0 = 0; k0 < chunks; k0 += kHeadAhead) {
#pragma unroll
        for (int k = 0; k < kHeadAhead; ++k) {
            const int chunk = k0 + k;
            if (chunk >= chunks) break;  // uniform
            lay_out(chunk, k);  // (the buffer's last readers have passed the barrier of the chunk before)
            request(k);
            __syncthreads();
#pragma unroll
            for (int g = 0; g < kHeadChunk; g += 16) {
                const int c0 = chunk * kHeadChunk + g;
                if (c0 + 16 <= p.C) {  // uniform
                    float w[16];
#pragma unroll
                    for (int c = 0; c < 16; ++c) w[c] = weights[chunk & 1][g + c][col];
                    head_channels(*reinterpret_cast<const float2*>(&mean[c0 + (tid & 15)][i0]), w, acc);
                } else {
                    for (int c = c0; c < p.C; ++c) {
                        const float weight = weights[chunk & 1][c - chunk * kHeadChunk][col];
                        acc[0] = __fmaf_rn(mean[c][i0], weight, acc[0]);
                        acc[1] = __fmaf_rn(mean[c][i0 + 1], weight, acc[1]);
                    }
                }
            }
        }
    }
    if (n >= p.N) return;
    const float bias = p.bias[n];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (b0 + i0 + i < p.B) p.out[(size_t)(b0 + i0 + i) * p.N + n] = __fadd_rn(acc[i], bias);
}

}  // namespace
}  // namespace tcbnn

using namespace tcbnn;

extern "C" int tcbnn_pool_out(int in_size, int window, int stride, int padding) {
    if (window <= 0 || stride <= 0 || padding < 0 || in_size + 2 * padding < window) return 0;
    return (in_size + 2 * padding - window) / stride + 1;
}

extern "C" int tcbnn_pool128_forward(const tcbnn_pool128_desc* d, void* stream) {
    TCBNN_NOTNULL(d);
    TCBNN_NOTNULL(d->input);
    TCBNN_NOTNULL(d->output);
    TCBNN_REQUIRE(d->input_height > 0 && d->input_width > 0 && d->channels > 0 && d->batch > 0 && d->window > 0 &&
                      d->stride > 0 && d->padding >= 0 && d->padding < d->window,
                  "pool128: bad shape");
    TCBNN_REQUIRE((d->input_residual == nullptr) == (d->output_residual == nullptr),
                  "pool128: input_residual and output_residual go together");
    TCBNN_REQUIRE(d->input_residual == nullptr || residual_format_known(d->residual_format),
                  "pool128: unknown residual_format");
    TCBNN_REQUIRE(d->input_residual == nullptr || d->residual_format != TCBNN_RES_I12 || d->batch % 2 == 0,
                  "pool128: a 12-bit residual needs an even batch");
    PoolParams p;
    p.in = d->input;
    p.out = d->output;
    p.rin = d->input_residual;
    p.rout = d->output_residual;
    p.H = d->input_height;
    p.W = d->input_width;
    p.C = d->channels;
    p.B = d->batch;
    p.OH = tcbnn_pool_out(p.H, d->window, d->stride, d->padding);
    p.OW = tcbnn_pool_out(p.W, d->window, d->stride, d->padding);
    TCBNN_REQUIRE(p.OH > 0 && p.OW > 0, "pool128: empty output");
    p.cw = step32(p.C);
    p.fmt = d->residual_format;
    p.groups = p.rin == nullptr ? 0 : (int)((p.C + residual_group_channels(p.fmt) - 1) / residual_group_channels(p.fmt));
    p.window = d->window;
    p.stride = d->stride;
    p.pad = d->padding;
    const long long total = (long long)(p.cw + p.groups) * p.B * p.OH * p.OW;
    const long long blocks = (total + kThreads - 1) / kThreads;
    TCBNN_REQUIRE(blocks <= 0x7fffffffLL, "pool128: grid too large");
    const long long per_pixel = (long long)(p.cw + p.groups) * p.B;
    const long long units = (per_pixel + kThreads - 1) / kThreads;
    const bool in_turn = p.groups == 0 || units % 8 == 0 || total < kPoolFew;
    const int rows = in_turn ? (int)std::min(8LL, std::max(1LL, total / (8192LL * 64))) : kPoolRows;
    const int runs = (p.OH + rows - 1) / rows;
    // (32 bits hold a lane's bytes within a pixel and a workgroup's number, rounded up)
    if (p.window == 3 && p.stride == 2 && runs <= 65535 && (!in_turn || p.OW <= 65535) && per_pixel * 24 < (1LL << 32) - 24 * kThreads &&
        (units * p.OW + 8) * runs < (1LL << 31)) {
        const long long pixel = 4LL * p.cw * p.B + (p.fmt == TCBNN_RES_I12 ? 24LL : 16LL) * p.groups * p.B;
        const long long in_bytes = pixel * p.H * p.W, bytes = in_bytes + pixel * p.OH * p.OW;
        const PoolOrder order = in_turn ? TURN : (bytes < 165LL << 20 ? ROWS : (in_bytes <= 256LL << 20 ? COLUMNS : COLUMNS_BACK));
        const int per_xcd = (int)((units * p.OW + 7) / 8), across = std::min(per_xcd, 1 << 18);
        const dim3 grid = in_turn ? dim3((unsigned)units, (unsigned)p.OW, (unsigned)runs)
                                  : dim3((unsigned)across * 8, (unsigned)((per_xcd + across - 1) / across), (unsigned)runs);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, (hipStream_t)stream, p, (int)units, per_xcd, order, rows);
        };
        if (p.fmt == TCBNN_RES_I12)
            launch(pool3x3s2_kernel<TCBNN_RES_I12>);
        else if (p.fmt == TCBNN_RES_I16)
            launch(pool3x3s2_kernel<TCBNN_RES_I16>);
        else
            launch(pool3x3s2_kernel<TCBNN_RES_I32>);
        TCBNN_LAUNCH_CHECK("pool3x3s2_kernel");
        return TCBNN_OK;
    }
    hipLaunchKernelGGL(pool128_kernel, dim3((unsigned)blocks), dim3(kThreads), 0, (hipStream_t)stream, p);
    TCBNN_LAUNCH_CHECK("pool128_kernel");
    return TCBNN_OK;
}

extern "C" int tcbnn_avgpool_fc_forward(const tcbnn_avgpool_fc_desc* d, void* stream) {
    TCBNN_NOTNULL(d);
    TCBNN_NOTNULL(d->input_residual);
    TCBNN_NOTNULL(d->weight);
    TCBNN_NOTNULL(d->bias);
    TCBNN_NOTNULL(d->output);
    TCBNN_REQUIRE(d->input_height > 0 && d->input_width > 0 && d->channels > 0 && d->batch > 0 && d->out_features > 0,
                  "avgpool_fc: bad shape");
    TCBNN_REQUIRE(d->channels <= kHeadMaxC, "avgpool_fc: at most 512 channels");
    TCBNN_REQUIRE(residual_format_known(d->residual_format), "avgpool_fc: unknown residual_format");
    TCBNN_REQUIRE(d->residual_format != TCBNN_RES_I12 || d->batch % 2 == 0,
                  "avgpool_fc: a 12-bit residual needs an even batch");
    HeadParams p;
    p.rin = d->input_residual;
    p.w = d->weight;
    p.bias = d->bias;
    p.out = d->output;
    p.P = d->input_height * d->input_width;
    p.C = d->channels;
    p.B = d->batch;
    p.N = d->out_features;
    p.fmt = d->residual_format;
    const int per_group = (int)residual_group_channels(p.fmt);
    p.groups = (p.C + per_group - 1) / per_group;
    const dim3 grid((unsigned)((p.B + kHeadImages - 1) / kHeadImages), (unsigned)((p.N + kHeadOutputs - 1) / kHeadOutputs));
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kHeadThreads), 0, (hipStream_t)stream, p); };
    if (p.fmt == TCBNN_RES_I12)
        launch(avgpool_fc_kernel<TCBNN_RES_I12>);
    else if (p.fmt == TCBNN_RES_I16)
        launch(avgpool_fc_kernel<TCBNN_RES_I16>);
    else
        launch(avgpool_fc_kernel<TCBNN_RES_I32>);
    TCBNN_LAUNCH_CHECK("avgpool_fc_kernel");
    return TCBNN_OK;
}
