// First-layer convolution (fp32 3-channel NCHW input, +-1 filters; InConv128LayerFMT, kernel.cuh:578-672) on the
// matrix cores, with the bits and residuals of the reference's own fp32 order of additions
//     acc = 0; for r, for s (in-frame taps): acc += ((+-f0) + (+-f1)) + (+-f2);  bit = !(acc < bn);  residual = (int)acc.
// On the VALU that order costs one dependent fp32 add per (tap, channel, pixel): 73 us at the very least for ResNet-18's
// first layer at batch 256, 121-138 us in practice.  Here it is computed as a filtered predicate:
//   1. every input is split into two fp16 numbers, x = hi + lo (22-23 bits), and S = sum of +-hi + sum of +-lo runs on
//      v_mfma_f32_32x32x16_f16: products are exact, sums are fp32;
//   2. a bound E of |S - acc| is known per pixel (below), so wherever S is further than E from the threshold, and from
//      every integer where a residual is saved, the bit and the residual of S are those of acc;
//   3. the few values within E (0.1 % with a residual, a few in 10^5 without) are put on a list and recomputed in the
//      reference's order by the same wave, which then repairs the stored bit and residual;
//   4. where that is not few (flat areas, large magnitudes), a wave leaves the list for passes that cost a bounded factor.
// The results are therefore the reference's, bit for bit, for every input; only the time depends on the data, and by a
// small factor (below).
//
// The bound.  u = 2^-24, A = sum of |x| under the window, A_k = what of it has been multiplied up to step k.  A rounding of a
// running sum is at most u times that sum, and the sum is at most A_k: there is one rounding per tap in the reference's order,
// and there are four per step here (an MFMA adds its 16 products in two halves of eight and rounds each once; lo, then hi;
// tests/test_gpu_matrix_core.py holds the instruction to this).  Added to these: 2 u A inside the reference's taps; 2 u A that
// the split drops (and 2^-25 per input where fp16 runs out of exponents); and what lies below u times a half's largest product
// M, which is lost of each product and of the sum they are added to: an fp16 number has 11 bits, so only products below
// 2^-13 M lose anything, with the sum at most 8 u M, and the M of all halves are at most A (those of lo 2^-11 of that).
// E = u (sum of n_k A_k + 13.5 A), n_k roundings of sums up to step k; 2 % cover the bound's own roundings.  For 7-row filters
// with a residual the A_k are summed up as the window passes (1.9 doubtful values per 32 pixels x 64 channels instead of 2.8
// with A for each); the others, which have few doubtful values, take A for every A_k.
// Where a residual is saved, -E itself enters the sum as one more product (a place that no tap uses; 7x8 at strides 2 and 4 has none:
// taken off at the end, one more rounding), so the accumulators hold S - E: a bit is certainly 1 where S - E >= bn, certainly 0 below bn - 2E.  Where none is saved, sums start from -bn: the
// bit is the sign, in doubt where |S - bn| <= E (partial sums are then at most what is still to come and |S - bn|: A again).
// Inputs outside the fp16 range, infinities and NaN make NaN of the sums or an infinity of E: all values of such a window are
// recomputed, as are those of windows whose neighbouring rows (multiplied by zeros) hold them.
//
// Many values in doubt.  A saved residual puts every sum ON an integer in doubt, and images have areas of such sums: bars of
// +-1 after scaling to [-1, 1], saturated white, bytes, a flat grey of 0.2 (every fifth channel); and E grows with the
// magnitudes: bytes less a mean leave 7 % of the sums in doubt, values in the thousands all of them.
//   grid    : sums of a window whose inputs are multiples of 1/256 (bytes, bytes / 128 - 1, +-1) with a sum of |x| below 2^16
//             are exact in both orders: every partial sum is a multiple of 1/256 below 2^24 / 256, and the two halves hold
//             inputs below 2^15 (a lane's |x| of a step add up to less than that).  E is 0.  (Sums that start from -bn: below 2^15,
//             if all thresholds are such multiples too.  With 2^15 for all, windows of bytes above 223 were in doubt: 7x7/4
//             293 us for 113, 7x7/2 1110 for 351.)
//   check   : a wave looks whether its inputs are on that grid (120 VALU instructions per item of 7-row filters) as long as all
//             have been; other inputs pay for their first item.  From an item with many values in doubt on it always looks.
//   ordered : from an item that has many even so, sums in the reference's order, 32 columns x 64 channels at a time, as fp32
//             products on the matrix cores (ordered_sums): no values in doubt but those that are no numbers.  It lasts to the
//             end of the wave's rows (left as soon as few would be in doubt, the common pass is reached from two places, and
//             the registers that takes cost 7x7/2 288 -> 328 us on ordinary images).
// ResNet-18's first layer at batch 256, launched on end, us: normal data 83, bytes and bytes / 128 - 1 73, images in [-1, 1] with a bar
// and patches of +-1 87, bytes of 195 to 255 113, bytes / 255 119, a bar and patches of 0.2 grey 360, bytes less a mean 313, normal x
// 1000 320.
//
// Work split.  A tile is 32 columns = NI images x 32/NI neighbouring pixels of a row (so small batches fill their tiles) by 64
// channels.  A wave walks down the rows of one column of tiles, a step per output row: the A (stride) input rows that are new
// are loaded straight into registers, split there, and multiplied at once for every output row that they are part of.
// sets_of(R, A) sums are under way; the first product of a step reads the next younger set's registers and writes its own, so
// they move on without copies.  Compared with a ring of split rows in LDS (of which a CU holds eight waves' worth, at 240
// registers a wave): no LDS traffic but the weights, which four waves share, no barrier, three waves per SIMD for 3x3 and 7x7/4
// (two for the rest), and 8 places for a row's 7 taps in one channel, not 32 for its 21.  The next step's rows are requested as the
// present ones are used up.  A workgroup's waves are neighbouring columns of tiles; an XCD has whole image tiles (3x3 with large
// residuals: neighbouring image tiles, see choose()).
// Eight images per tile: their residuals of a pixel are a whole 128-byte line.  Sixteen (64 bytes of output words) where no
// residual is saved and a wave has 32 items or more: VGG-16 217 -> 206 us; below that fewer units fill the machine worse
// (CIFAR VGG 16.7 -> 18.0 us).
//
// What binds it: memory traffic and the waits for it.  ResNet-18's layer at batch 256 fetches 289 MB for 154 MB of images (a doubtful
// value's window comes back from HBM, 21 rows of 128 bytes; without the recomputations 178 MB) and writes 90 MB, 3.7 TB/s; the VALU is
// busy 30 % of the time, the matrix cores 15 %.  Recomputing a value at once finds its rows in L2 no more often (an XCD's waves bring
// in 4 MB per step) and costs a trip to memory per item (a tenth slower).
// Measured, us within the network's pass at batch 256 (kernel trace, medians; adds on the VALU -> ring in LDS -> here): ResNet-18 7x7/4
// 127 -> 121 -> 103, 7x7/2 423 -> 315 -> 296, VGG-16 3x3 399 -> 207 -> 200, AlexNet 11x11/4 310 -> 137 -> 102, CIFAR VGG 23 -> 18.0 -> 14.8,
// CIFAR ResNet 27.4 -> 27.1 -> 25.9.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

#include "inconv.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

constexpr int kListCap = 64;   // doubtful values a wave keeps
constexpr int kBatch = 16;     // ... and recomputes at a time
// What counts as many values in doubt: one lane with this many (of its column's 32; a flat area), or this many lanes (of 64)
// with any; the second for windows already checked for the grid.
constexpr int kManyInLane = 8, kManyLanes = 28, kManyLanesChecked = 32;

// A wave walks down the input, A rows (the stride) at a time, and an input row is multiplied for every output row that it is
// part of while it is in registers: sets_of(R, A) sums are under way, the oldest of which is finished by the step.  A = R: a step
// loads the window of its output row whole, and the next one's begins a stride (of any size) further down.
constexpr int sets_of(int r, int a) { return (r + a - 1) / a; }
// The K order of a step.  A "pair" is one of its rows in one channel: 3 A of them, the even ones for lane half 0, the odd ones
// for half 1.  A lane loads a pair's T taps at once and gives each pair slots_of(T) places of its stream; every eight places
// are one fragment.  T = 7: a fragment is a pair; T = 3: places 0-2, 3-5; T = 11: 12 places.
constexpr int pairs_of(int a) { return (3 * a + 1) / 2; }
constexpr int slots_of(int t) { return t == 7 ? 8 : (t == 11 ? 12 : t); }
constexpr int steps_of(int a, int t) { return (pairs_of(a) * slots_of(t) + 7) / 8; }
// Place (of the step's last fragment, lane half 1) through which -E enters: none of the taps'.
constexpr int kBoundPlace = 7;
constexpr bool bound_place_free(int a, int t) {
    const int slot = 8 * (steps_of(a, t) - 1) + kBoundPlace, pair = 2 * (slot / slots_of(t)) + 1;
    return pair >= 3 * a || slot % slots_of(t) >= t;
}
// What E counts (top of this file).
template <int R, int T, int A>
struct Order {
    static constexpr int P = slots_of(T), D = sets_of(R, A), KS = steps_of(A, T);
    // Whether a pair's row is part of the oldest set's windows, or has zero weights there (3-row filters: all count)
    static constexpr bool in_old(int pair) { return pair < 3 * A && (P % 2 != 0 || pair / 3 < R - (D - 1) * A); }
    // Roundings of sums that hold what has been multiplied up to step k (a pair each of both lane halves): two halves of lo
    // and of hi, and a row's T taps with its last pair.
    static constexpr int roundings(int k, bool old) {
        int n = !old || in_old(2 * k) ? 4 : 0;
        for (int at = 2; at < 3 * A; at += 3)
            if ((!old || in_old(at)) && at / 2 == k) n += T;
        return n;
    }
    static constexpr int roundings(bool old) {
        int n = 0;
        for (int k = 0; k < KS; ++k) n += roundings(k, old);
        return n;
    }
};
// Registers: sums of sets_of() rows x 64 channels, taps of the next rows
constexpr int waves_per_simd(int r, int t, int a) { return r == 3 || (t == 7 && sets_of(r, a) == 2) ? 3 : 2; }
constexpr int waves_of(int r) { return r > 7 ? 8 : 4; }  // of a workgroup: they share the LDS copy of the weight fragments
constexpr int MT = 2;  // channel tiles of 32 that a wave multiplies

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v3f __attribute__((ext_vector_type(3)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// Saved residual: none, 12 bits, or 16 / 32 bits (looked up at run time).
enum Residual : int { RES_NONE = 0, RES_12 = 1, RES_WIDE = 2 };

// What neighbouring work units differ in (after the first: in this order), and whether a workgroup's waves go down their rows in step
enum Units : int { COLUMNS_BANDS_IMAGES = 0, IMAGES_COLUMNS_BANDS_IN_STEP = 1, IMAGES_BANDS_COLUMNS_IN_STEP = 2 };

struct Geometry {
    int ni_log2;             // images per tile
    int groups;              // tiles across a row
    int bands, band_rows;    // bands of convolution rows
    int rows;                // convolution rows
    int cgroups;             // channel groups (of 64)
    int total, per_xcd;      // waves' work units (image tile, band, column group), and those of an XCD
    Units units;             // their order
    int img_tiles;
    int rs_taps;
    float bound_parts;       // E = bound_parts * (the sum of |x| before each rounding) + bound_sum * (the sum of |x|) + bound_add
    float bound_sum;
    float bound_add;
};

// The kernel's argument.  Code that seldom runs reads it anew from the argument segment (seldom_args): fields that
// only such code needs are then not kept in scalar registers, and spilled, all the way through the common one.  (The
// segment's address is a register of the kernel itself: taken in a function that is not inlined it would be 0.)
struct KernelArgs {
    InConvParams p;
    Geometry q;
    const uint32_t* pats;
    unsigned out_bytes, res_bytes;
};
typedef const KernelArgs __attribute__((address_space(4))) * SeldomArgs;
__device__ __forceinline__ SeldomArgs seldom_args(SeldomArgs a) {
    asm volatile("" : "+s"(a));
    return a;
}

// x - (float)pair[I], exact: one multiply-add with a half-precision operand
template <int I>
__device__ __forceinline__ float minus_half(float x, h2 pair) {
    float d;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[%3,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(pair), "v"(x), "n"(I));
    return d;
}

// 16 channels of one image and pixel: 12 bits each, 16 bytes at `at` and 8 at `at8`; 16 or 32 bits, 16-byte pieces
// `piece` bytes apart from `at` on.  Ordinary stores: a tile's eight images are whole 128-byte lines only if the batch is a
// multiple of 8, and otherwise the cache has to join the halves (CIFAR ResNet at batch 170: 33.9 us with non-temporal
// stores, 23.0 us with these; at batch 256 28.5 and 27.7 us).  Lanes without a value pass offsets
// beyond the tensor and store nothing.  (No scalar offset register on these stores: a 128-bit buffer store with one,
// directly followed by a VALU write of its data, can store the new value.)
template <int RES>
__device__ __forceinline__ void store_residual_group(__amdgpu_buffer_rsrc_t rsrc, int fmt, unsigned at, unsigned at8, unsigned piece,
                                                     const int* v) {
    if constexpr (RES == RES_12) {
        uint32_t d[6];
        i12_pack8(v, d[0], d[1], d[2]);
        i12_pack8(v + 8, d[3], d[4], d[5]);
        __builtin_amdgcn_raw_buffer_store_b128(v4u{d[0], d[1], d[2], d[3]}, rsrc, (int)at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b64(v2u{d[4], d[5]}, rsrc, (int)at8, 0, 0);
    } else if (fmt == TCBNN_RES_I16) {
#pragma unroll
        for (int e = 0; e < 16; e += 8)
            __builtin_amdgcn_raw_buffer_store_b128(v4u{(uint32_t)((v[e] & 0xffff) | (v[e + 1] << 16)), (uint32_t)((v[e + 2] & 0xffff) | (v[e + 3] << 16)),
                                                       (uint32_t)((v[e + 4] & 0xffff) | (v[e + 5] << 16)), (uint32_t)((v[e + 6] & 0xffff) | (v[e + 7] << 16))},
                                                   rsrc, (int)(at + (unsigned)(e / 8) * piece), 0, 0);
    } else {
#pragma unroll
        for (int e = 0; e < 16; e += 4)
            __builtin_amdgcn_raw_buffer_store_b128(v4u{(uint32_t)v[e], (uint32_t)v[e + 1], (uint32_t)v[e + 2], (uint32_t)v[e + 3]}, rsrc,
                                                   (int)(at + (unsigned)(e / 4) * piece), 0, 0);
    }
}

// The sum of v over the lane halves
__device__ __forceinline__ float both_halves(float v) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
// acc + lane T of m's quad
template <int T>
__device__ __forceinline__ float add_quad_lane(float acc, float m) {
    return acc + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m), 0x55 * T, 0xf, 0xf, false));
}

// Taps t = 0 .. N - 1 from byte offset `at` (+ a uniform one): the address unit takes 16 cycles for 64 lanes' 4 to 16 bytes
// each, whatever their alignment to 4, and 30 for single words that are not neighbours.
template <int N>
__device__ __forceinline__ void load_taps(__amdgpu_buffer_rsrc_t rsrc, unsigned at, unsigned base, float* f) {
    if constexpr (N >= 4) {
        const v4f v = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)at, (int)base, 0));
        f[0] = v[0], f[1] = v[1], f[2] = v[2], f[3] = v[3];
        if constexpr (N > 4) load_taps<N - 4>(rsrc, at + 16u, base, f + 4);
    } else {
        static_assert(N == 3, "");
        const v3f v = __builtin_bit_cast(v3f, __builtin_amdgcn_raw_buffer_load_b96(rsrc, (int)at, (int)base, 0));
        f[0] = v[0], f[1] = v[1], f[2] = v[2];
    }
}

template <int R, int T, int A, int RES, int POOL>
__global__ __launch_bounds__(64 * waves_of(R)) __attribute__((amdgpu_waves_per_eu(waves_per_simd(R, T, A)))) void inconv_mfma_kernel(
    const KernelArgs args) {
    const SeldomArgs args_at = (SeldomArgs)__builtin_amdgcn_kernarg_segment_ptr();
    const InConvParams& p = args.p;
    const Geometry& q = args.q;
    static_assert(!(RES != RES_NONE && POOL > 1), "residuals of un-pooled layers only");
    constexpr int kWaves = waves_of(R), kPairs = pairs_of(A), P = slots_of(T), KS = steps_of(A, T), D = sets_of(R, A);
    constexpr int kRing = (R == 3 || A == 2 || D == 1 ? kPairs : 3);  // pairs in registers
    static_assert(kPairs % kRing == 0, "a pair's place does not depend on the step");
    constexpr unsigned kOutOfRange = 0x80000000u;
    constexpr int kChannels = 32 * MT;
    // Where no residual is saved the sums start from the threshold's negative: the bit is the sum's sign.
    constexpr bool kFromThreshold = RES == RES_NONE;
    constexpr bool kBoundInSum = !kFromThreshold && bound_place_free(A, T);  // (else -E is added at the end)
    using order = Order<R, T, A>;
    constexpr bool kParts = T == 7 && !kFromThreshold;  // E by the sums before each rounding
    extern __shared__ __align__(16) char lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // LDS: weight fragments, thresholds of the channel group, lists, signs
    v4i* const frags = reinterpret_cast<v4i*>(lds);
    float* const thr = reinterpret_cast<float*>(lds + D * KS * MT * 1024);
    uint32_t* const list = reinterpret_cast<uint32_t*>(lds + D * KS * MT * 1024 + MT * 128) + wave * 2 * kListCap;
    uint8_t* const signs = reinterpret_cast<uint8_t*>(lds + D * KS * MT * 1024 + MT * 128 + kWaves * 8 * kListCap);

    const int slot = (int)blockIdx.x >> 3, cg = slot % q.cgroups, in_xcd = slot / q.cgroups * kWaves + wave;
    int work = ((int)blockIdx.x & 7) * q.per_xcd + in_xcd;
    const bool idle = in_xcd >= q.per_xcd || work >= q.total;
    const int tile0 = cg * MT;  // first channel tile

    if (idle) work = 0;  // (such a wave helps with the weights and leaves)

    constexpr bool kOrders = R == 3 && A == 1 && RES != RES_NONE;  // units in other orders (choose())
    const bool in_step = kOrders && q.units != COLUMNS_BANDS_IMAGES;  // uniform
    int g, band, it;
    if (in_step) {
        it = work % q.img_tiles;
        work /= q.img_tiles;
        if (q.units == IMAGES_COLUMNS_BANDS_IN_STEP) g = work % q.groups, band = work / q.groups;
        else band = work % q.bands, g = work / q.bands;
    } else {
        g = work % q.groups;
        work /= q.groups;
        band = work % q.bands, it = work / q.bands;
    }
    const int advance = D == 1 ? p.stride_h : A;  // input rows from one output row's to the next one's
    int cy = band * q.band_rows;  // convolution row
    const int cy_end = min(cy + q.band_rows, q.rows);
    const int NI = 1 << q.ni_log2, NX = 32 >> q.ni_log2, b0 = it << q.ni_log2;
    const int xcols = POOL > 1 ? POOL * p.OW : p.PW;
    const unsigned plane_b = (unsigned)(p.H * p.W) * 4u, row_b = (unsigned)p.W * 4u;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.in + (size_t)b0 * 3 * p.H * p.W), 0,
                                                                          (int)((unsigned)min(NI, p.B - b0) * 3u * plane_b), 0x00020000);
    const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)args.out_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t res_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.res, 0, (int)args.res_bytes, 0x00020000);
    auto threshold = [&](int i) __attribute__((always_inline)) { return kFromThreshold ? -thr[i] : thr[i]; };
    const unsigned uB = (unsigned)p.B, group_b = (RES == RES_12 ? 24u : (p.res_fmt == TCBNN_RES_I16 ? 32u : 64u)) * uB;
    const unsigned pixel_b = (unsigned)(p.O / 16) * group_b;
    // Where lane ln stores, relative to the item (uniform): its output word, its 16 residuals (12-bit: the 8-byte part
    // apart); beyond the tensors for an image past the batch.
    auto place_word = [&](int ln) __attribute__((always_inline)) {
        const unsigned px = (unsigned)((ln & 31) >> q.ni_log2), h = (unsigned)ln >> 5, b = (unsigned)(b0 + (ln & (NI - 1)));
        return b < uB && (POOL == 1 || (px & 1u) == 0u) ? ((px / POOL * (unsigned)p.ow + h) * uB + b) * 4u : kOutOfRange;
    };
    const unsigned word_place = kFromThreshold ? place_word(lane) : 0u;  // (where registers allow)
    auto place_residual = [&](int ln) __attribute__((always_inline)) {
        const unsigned px = (unsigned)((ln & 31) >> q.ni_log2), h = (unsigned)ln >> 5, b = (unsigned)(b0 + (ln & (NI - 1)));
        return px * pixel_b + h * group_b + b * 16u;
    };
    auto place_residual8 = [&](int ln) __attribute__((always_inline)) { return place_residual(ln) + uB * 16u - (unsigned)(b0 + (ln & (NI - 1))) * 8u; };

    // ---- loading: pair 2 i + h of a step's rows into ring place i % kRing
    // Where this lane reads: its pixel's window relative to the step's first one, and which of two pairs is this half's.
    unsigned from_a, from_b;  // channels c, c + 1 of a row; channel 2 of a row and channel 0 of the next
    unsigned outside = 0u;    // taps that are not inside the frame's columns (columns of the tile that are none: all)
    const int ax_first = g * NX * p.stride_w - p.pad_w;
    const bool columns_inside = p.S == T && ax_first >= 0 && ax_first + (NX - 1) * p.stride_w + T <= p.W && (g + 1) * NX <= xcols;
    {
        const int px = (lane & 31) >> q.ni_log2, h = lane >> 5, img = lane & (NI - 1), ax = ax_first + px * p.stride_w;
        const int from = min(max(-ax, 0), 31), to = min(max(min(p.W - ax, p.S), 0), 31);
        const bool none = (b0 + img >= p.B) | (g * NX + px >= xcols);
        outside = none ? ~0u : ((1u << from) - 1u) | (~0u << to);
        const unsigned first = b0 + img < p.B ? (unsigned)img * 3u * plane_b + (unsigned)(px * p.stride_w) * 4u : kOutOfRange;
        from_a = first + (h ? plane_b : 0u);
        from_b = first + (h ? row_b : 2u * plane_b);
    }
    float x[kRing][T];
    // How a step's rows (`ay`: the first) are loaded: all inside the frame; rows outside it; columns outside it, which are masked
    // when the taps are used (not in the first and last rows: what is in front of the first one's taps, or behind the last
    // one's, need not be the tensor's); tap by tap.
    enum Path : int { INSIDE, ROWS, COLUMNS, TAPS };
    const bool columns_masked = p.W >= T;
    auto path_of = [&](int ay) __attribute__((always_inline)) -> int {
        if (columns_inside) return ay >= 0 && ay + A <= p.H ? INSIDE : ROWS;
        return columns_masked && ay > 0 && ay + A < p.H ? COLUMNS : TAPS;
    };
    auto load = [&](int ay, int path, int i) __attribute__((always_inline)) {
        float* const f = x[i % kRing];
        const int r0 = 2 * i / 3, c0 = 2 * i % 3, r1 = (2 * i + 1) / 3;
        const bool last = 2 * i + 1 >= 3 * A;  // half 1 has none
        unsigned step_b = row_b;
        asm volatile("" : "+v"(from_a), "+v"(from_b), "+s"(step_b));  // (sums with them are made when used, not kept)
        const unsigned at = (unsigned)(ay * p.W + ax_first) * 4u + (unsigned)r0 * step_b + (c0 == 1 ? plane_b : 0u);
        const unsigned from = c0 == 2 ? from_b : from_a;
        if (path == INSIDE || path == COLUMNS) {  // uniform
            load_taps<T>(rsrc, last && lane >= 32 ? kOutOfRange : from, at, f);
        } else {
            // rows outside the frame (and taps, and columns that are none): offsets beyond the tensor, zeros.  An offset can be
            // negative where a window begins in front of its image; those of taps inside are not.
            const unsigned row0 = (unsigned)(ay + r0) < (unsigned)p.H ? 0u : ~0u, row1 = !last && (unsigned)(ay + r1) < (unsigned)p.H ? 0u : ~0u;
            const unsigned out = lane >= 32 ? row1 : row0;
            if (path == ROWS) {
                load_taps<T>(rsrc, out != 0u ? kOutOfRange : from + at, 0u, f);
            } else {
#pragma unroll
                for (int t = 0; t < T; ++t)
                    f[t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                         rsrc, (int)(((out | outside) << (31 - t) & kOutOfRange) | (from + at + 4u * t)), 0, 0));
            }
        }
    };

    // ---- The first rows are on their way while the weights are laid out.
#pragma unroll
    for (int i = 0; i < kRing; ++i) load(cy * advance - p.pad_h, path_of(cy * advance - p.pad_h), i);
    // ---- signs of the channel group's filters (pattern 4 neg0 + 2 neg1 + neg2 of a tap; four channels to a load), thresholds (NaN:
    // -infinity, the bit is 1 either way)
    bool steps_256 = true;  // every threshold a multiple of 1/256 (below 2^15), or infinite: exact sums stay exact less these
    {
        constexpr int kLoads = (R * T * kChannels / 4 + 64 * kWaves - 1) / (64 * kWaves);
        v4u sign[kLoads];
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int e = i * 64 * kWaves + tid;
            sign[i] = *reinterpret_cast<const v4u*>(args.pats + (unsigned)(min(e / (kChannels / 4), q.rs_taps - 1) * p.opad + tile0 * 32 + e % (kChannels / 4) * 4));
        }
        const float t = p.bn[tile0 * 32 + min(lane, kChannels - 1)];  // (every wave looks at all of them)
        const float known = t != t ? -INFINITY : t;
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            if (i * 64 * kWaves + tid < R * T * kChannels / 4)
                reinterpret_cast<uint32_t*>(signs)[i * 64 * kWaves + tid] = sign[i][0] | sign[i][1] << 8 | sign[i][2] << 16 | sign[i][3] << 24;
        if (tid < kChannels) thr[tid] = kFromThreshold ? 0.0f - known : known;  // (a threshold of 0: sums start from +0)
        steps_256 = __ballot(!(__builtin_fabsf(t) <= 32768.0f) ? __builtin_fabsf(t) < INFINITY : __builtin_amdgcn_fractf(t * 256.0f) != 0.0f) == 0;
    }
    __syncthreads();
    // ---- +-1 fragments: lane (row n, half h) of set d's step k holds places 8 k .. 8 k + 7 of channel row_to_channel(n), half h
    {
        constexpr int kFrags = (D * KS * MT + kWaves - 1) / kWaves;  // of a wave
        const int h = lane >> 5, n = mfma::row_to_channel(lane & 31);
#pragma unroll 2
        for (int i = 0; i < kFrags; ++i) {
            const int e = i * kWaves + wave, d = e / (KS * MT), k = e / MT % KS;
            if (e >= D * KS * MT) break;  // uniform
            uint32_t half[8], pt[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int place = 8 * k + j, tap = place % P, r = d * A + (2 * (place / P) + h) / 3;
                pt[j] = signs[(min(r, R - 1) * p.S + min(tap, p.S - 1)) * kChannels + e % MT * 32 + n];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int place = 8 * k + j, pair = 2 * (place / P) + h, tap = place % P, row = pair / 3;
                const bool used = (tap < p.S) & (tap < T) & (pair < 3 * A) & (d * A + row < R);
                half[j] = used ? 0x3c00u | (pt[j] << (13 + pair - 3 * row) & 0x8000u) : 0u;
                if (kBoundInSum && j == kBoundPlace && d == D - 1 && k == KS - 1 && h == 1) half[j] = 0x3c00u;
            }
            v4i f;
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = (int)(half[2 * j] | half[2 * j + 1] << 16);
            frags[e * 64 + lane] = f;
        }
    }
    __syncthreads();
    if (idle) return;

    // ---- doubtful values: recomputed in the reference's order, 4 lanes per value (lane t of a quad: rows t, t + 4, ...), the
    // list's last sixteen at a time.  What the residual's words hold is asked for with the inputs.
    int count = 0;  // entries on this wave's list (uniform)
    auto recompute = [&]() __attribute__((always_inline)) {
        const SeldomArgs a = seldom_args(args_at);
        const auto& p = a->p;
        constexpr int kTurns = (R + 3) / 4;  // rows of a lane
        const int pending = min(count, kBatch);
        count -= pending;
        int ln = lane;
        asm volatile("" : "+v"(ln));  // (nothing derived from it is kept outside)
        const int t4 = ln & 3, e = count + min(ln >> 2, pending - 1);
        const uint32_t ex = list[2 * e], ey = list[2 * e + 1];
        const int ay0 = (int)(ex >> 16) * p.stride_h - p.pad_h, ax0 = (int)(ex & 0xffffu) * p.stride_w - p.pad_w;
        const int o = (int)(ey & 0xffffu);
        const unsigned im = (ey >> 16) * 3u * plane_b;
        const bool active = (ln >> 2) < pending;
        const int bb = b0 + (int)(ey >> 16);
        const unsigned pix = (ex >> 16) / POOL * (unsigned)p.OW + (ex & 0xffffu) / POOL;  // (host: tensors below 2 GiB)
        // Bits [fix_shift, ...) of the 32-bit word fix_at, under fix_mask, are the value's from bit fix_drop on; only this lane
        // changes them, neighbours in the same word are left alone (exclusive or with what differs).
        uint32_t* const residual = reinterpret_cast<uint32_t*>(p.res);
        size_t fix_at = 0;
        int fix_shift = 0, fix_drop = 0;
        uint32_t fix_mask = 0u, old = 0u;
        if constexpr (RES == RES_12) {
            const int bit = 12 * (o & 15), here = min(12, 32 - (bit & 31));
            const bool second = t4 == 1;
            fix_shift = second ? 0 : bit & 31;
            fix_drop = second ? here : 0;
            fix_mask = t4 < 2 ? (1u << (second ? 12 - here : here)) - 1u : 0u;
            fix_at = i12_word_index(pix, (size_t)((p.O + 15) / 16), o >> 4, p.B, bb, (bit >> 5) + (second ? 1 : 0));
        } else if constexpr (RES == RES_WIDE) {
            fix_at = residual_index(p.res_fmt, pix, p.O, o, p.B, bb);
            if (p.res_fmt == TCBNN_RES_I16) {
                fix_shift = (int)(fix_at & 1) * 16;
                fix_mask = t4 == 0 ? 0xffffu : 0u;
                fix_at >>= 1;
            }
        }
        const bool fix = active && fix_mask != 0u;
        if (RES != RES_NONE && fix) old = __hip_atomic_load(residual + fix_at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool whole = p.S == T && __ballot((ax0 < 0) | (ax0 + T > p.W)) == 0;  // uniform: every window inside the frame's columns
        float acc = 0.0f;
#pragma unroll(kTurns <= 2 ? kTurns : 1)
        for (int turn = 0; turn < kTurns; ++turn) {
            const int r = 4 * turn + t4, ay = ay0 + r;
            const bool row = (r < R) & (ay >= 0) & (ay < p.H);  // (else zeros, which add nothing)
            const unsigned at = im + (unsigned)(ay * p.W + ax0) * 4u;
            float f[3][T];
            if (whole) {
#pragma unroll
                for (int ch = 0; ch < 3; ++ch) load_taps<T>(rsrc, row ? at : kOutOfRange, ch * plane_b, f[ch]);
            } else {
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const bool inside = row & (t < p.S) & (ax0 + t >= 0) & (ax0 + t < p.W);
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch)
                        f[ch][t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(inside ? at + 4u * t : kOutOfRange), (int)(ch * plane_b), 0));
                }
            }
            const uint8_t* const row_signs = signs + min(r, R - 1) * p.S * kChannels + (o - tile0 * 32);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const uint32_t pt = row_signs[min(t, p.S - 1) * kChannels];
                const float f0 = __uint_as_float(__float_as_uint(f[0][t]) ^ (pt << 29 & 0x80000000u));
                const float f1 = __uint_as_float(__float_as_uint(f[1][t]) ^ (pt << 30 & 0x80000000u));
                const float f2 = __uint_as_float(__float_as_uint(f[2][t]) ^ (pt << 31));
                f[0][t] = (f0 + f1) + f2;
            }
#pragma unroll
            for (int t = 0; t < T; ++t) acc = add_quad_lane<0>(acc, f[0][t]);
#pragma unroll
            for (int t = 0; t < T; ++t) acc = add_quad_lane<1>(acc, f[0][t]);
#pragma unroll
            for (int t = 0; t < T; ++t) acc = add_quad_lane<2>(acc, f[0][t]);
            if (kTurns * 4 == R || turn + 1 < kTurns) {
#pragma unroll
                for (int t = 0; t < T; ++t) acc = add_quad_lane<3>(acc, f[0][t]);
            }
        }
        // (the quad's lanes all hold the sum: lane 2 sets the bit, lanes 0 and 1 repair the one or two words)
        if (active && t4 == 2 && !(acc < threshold(o - tile0 * 32)))
            __hip_atomic_fetch_or(p.out + ((pix * (unsigned)p.ow + (unsigned)(o >> 5)) * (unsigned)p.B + (unsigned)bb), 0x80000000u >> (o & 31), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (RES != RES_NONE) {
            const uint32_t v = (uint32_t)(int)acc;
            const uint32_t d = ((old >> fix_shift ^ v >> fix_drop) & fix_mask) << fix_shift;
            if (fix && d != 0u) __hip_atomic_fetch_xor(residual + fix_at, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (RES == RES_WIDE && active && t4 == 0 && p.res_fmt == TCBNN_RES_I32) residual[fix_at] = v;
        }
    };

    // ---- a whole item in the reference's order: words, residuals; in doubt stay sums that are no numbers.
    // A tap's eight possible values are four and their negatives, so adding one of them to 32 x 32 sums is a product with a
    // matrix of one +-1 and three 0 per row: two v_mfma_f32_32x32x2_f32, each one fp32 addition per sum (adding the zeros
    // changes nothing; tests/test_gpu_matrix_core.py).
    auto ordered_sums = [&](int cy, uint32_t* word) __attribute__((always_inline)) -> uint32_t {
        const SeldomArgs a = seldom_args(args_at);
        const auto& p = a->p;
        int ln = lane;
        asm volatile("" : "+v"(ln));  // (nothing derived from it is kept outside)
        const int h = ln >> 5, img = ln & (NI - 1), xc = g * NX + ((ln & 31) >> a->q.ni_log2);
        const bool valid = b0 + img < p.B && xc < xcols;
        const int ax0 = xc * p.stride_w - p.pad_w, ay0 = cy * advance - p.pad_h, r_end = min(R, p.H - ay0);
        const unsigned im = (unsigned)img * 3u * plane_b, flip = (unsigned)h << 31;
        uint32_t undecided = 0u;
        const bool whole = p.S == T && __ballot(valid & ((ax0 < 0) | (ax0 + T > p.W))) == 0;  // uniform
        v16f acc[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
        // a filter row at a time, requested two rows ahead; out of the frame: zeros, which add nothing
        float next[2][3][T];
        auto request = [&](int r, int slot) __attribute__((always_inline)) {
            const unsigned at0 = im + (unsigned)((ay0 + r) * p.W + ax0) * 4u;
            if (whole) {
#pragma unroll
                for (int ch = 0; ch < 3; ++ch) load_taps<T>(rsrc, valid ? at0 : kOutOfRange, ch * plane_b, next[slot][ch]);
            } else {
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const bool inside = valid & (t < p.S) & (ax0 + t >= 0) & (ax0 + t < p.W);
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch)
                        next[slot][ch][t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(inside ? at0 + 4u * t : kOutOfRange), (int)(ch * plane_b), 0));
                }
            }
        };
        const int r_begin = max(0, -ay0);
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (r_begin + u < r_end) request(r_begin + u, u);
#pragma unroll 1
        for (int r0 = r_begin; r0 < r_end; r0 += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int r = r0 + u;
                if (r >= r_end) break;  // uniform
                float f[3][T];
                uint32_t pt[T][MT];
                const uint8_t* const row_signs = signs + (unsigned)(r * p.S * kChannels) + mfma::row_to_channel(ln & 31);
#pragma unroll
                for (int t = 0; t < T; ++t) {
#pragma unroll
                    for (int m = 0; m < MT; ++m) pt[t][m] = row_signs[min(t, p.S - 1) * kChannels + 32 * m];
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch) f[ch][t] = next[u][ch][t];
                }
                if (r + 2 < r_end) request(r + 2, u);
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    if (T == 3 || t < T - 2 || t < p.S) {  // uniform (narrower filters than that: zeros)
                        const float f2 = __uint_as_float(__float_as_uint(f[2][t]) ^ flip);
                        const float same = (f[0][t] + f[1][t]) + f2, other = (f[0][t] - f[1][t]) + f2;
                        // pattern 4 neg0 + 2 neg1 + neg2; a pattern from 4 on is the negative of the inverted one
                        uint32_t c[MT], one[MT];
#pragma unroll
                        for (int m = 0; m < MT; ++m) {
                            const uint32_t neg = (uint32_t)((int)(pt[t][m] << 29) >> 31);
                            c[m] = (pt[t][m] ^ neg) & 3u;
                            one[m] = 0x3f800000u | (neg & 0x80000000u);
                        }
#pragma unroll
                        for (int m = 0; m < MT; ++m)
                            acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(c[m] == (uint32_t)h ? one[m] : 0u), same, acc[m], 0, 0, 0);
#pragma unroll
                        for (int m = 0; m < MT; ++m)
                            acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(c[m] == (uint32_t)h + 2u ? one[m] : 0u), other, acc[m], 0, 0, 0);
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const v4f* const tp = reinterpret_cast<const v4f*>(thr + m * 32 + 16 * h);
            uint32_t w = 0u;
            float zero = 0.0f;  // an infinity or NaN among a tap's values makes NaN of it, times 0, in every sum
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                w = __builtin_amdgcn_alignbit(w, __float_as_uint(kFromThreshold ? acc[m][i] + tp[i >> 2][i & 3] : acc[m][i] - tp[i >> 2][i & 3]), 31);
                zero = __builtin_fmaf(acc[m][i], 0.0f, zero);
            }
            const bool bad = !(zero == 0.0f);
            w = bad ? 0u : ~w & 0xffffu;
            undecided |= (bad && valid ? 0xffffu : 0u) << (16 * m);
            word[m] |= w;
            if constexpr (RES != RES_NONE) {
                int v[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = (int)acc[m][i];
                const unsigned item = (unsigned)(cy * p.PW + g * NX) * pixel_b + (unsigned)((tile0 + m) * 2) * group_b;
                store_residual_group<RES>(res_rsrc, p.res_fmt, valid ? place_residual(ln) + item : kOutOfRange,
                                          RES == RES_12 ? (valid ? place_residual8(ln) + item : kOutOfRange) : 0u, uB * 16u, v);
            }
        }
        return undecided;
    };

    // ---- the wave's rows.  An item (a row) with many values in doubt is done again with its windows checked for the grid, as
    // are all that follow; one that still has many, and all that follow, in the reference's order.
    bool check = !kFromThreshold, keep_checking = false, loaded = true;  // (sums that start from -bn are seldom in doubt)
    auto pass = [&](auto ordered) __attribute__((always_inline)) {
        constexpr bool kOrdered = decltype(ordered)::value;
        v16f acc[D][MT];
        float sum[D], parts[D], off[D];
        const int first_row = cy;
        int block = cy;  // of A input rows; the oldest set's output row is block - D + 1
        if constexpr (!kOrdered) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                sum[d] = parts[d] = off[d] = 0.0f;
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[d][m][i] = 0.0f;
            }
            if (!loaded) {  // uniform
#pragma unroll
                for (int i = 0; i < kRing; ++i) load(block * advance - p.pad_h, path_of(block * advance - p.pad_h), i);
            }
            loaded = false;
        }
        v4i weights[MT];  // of the set and step that is multiplied next
        auto read_weights = [&](int d, int k) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < MT; ++m) weights[m] = frags[((d * KS + k) * MT + m) * 64 + lane];
        };
        if constexpr (!kOrdered) read_weights(D - 1, 0);
        uint32_t word[MT], doubt[POOL];
#pragma unroll
        for (int m = 0; m < MT; ++m) word[m] = 0u;
#pragma unroll
        for (int py = 0; py < POOL; ++py) doubt[py] = 0u;
#pragma unroll 1
        while (cy < cy_end) {
            // A lane's place (column of the tile: image and pixel; half of the channels) is worked out anew from a lane
            // index the compiler cannot carry over: kept across the multiplication, the addresses made from it spill.
            int ln = lane;
            asm volatile("" : "+v"(ln));
            uint32_t undecided = 0u;
            // (Waves that have ended are not waited for, and every wave gets on without the others or ends.)
            if (in_step) __builtin_amdgcn_s_barrier();
            if constexpr (!kOrdered) {
                const int ay = block * advance - p.pad_h, done = block - (D - 1);  // (uniform)
                const bool more = done + 1 < cy_end;
                const int path = path_of(ay), next_path = path_of(ay + advance);
                // Sums of |x| (and what is off the grid): of the step's rows, and of those that the oldest set has weights for; and
                // these sums before each rounding, added up.
                float step_sum = 0.0f, step_off = 0.0f, step_parts = 0.0f, old_sum = 0.0f, old_off = 0.0f, old_parts = 0.0f, two_e = 0.0f;
                [[maybe_unused]] float lowered = 0.0f;  // E, where it is not one of the products
                bool bad = false, small = false;  // small: |S| and |acc| are below 1/2, the residual is 0
#pragma unroll
                for (int k = 0; k < KS; ++k) {
                    if (!columns_inside) {  // uniform
                        unsigned in = ~outside;
                        asm volatile("" : "+v"(in));  // (nothing derived from it is kept outside)
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const int at = 8 * k + j;
                            if (at / P >= kPairs || at % P >= T) continue;
                            float& f = x[at / P % kRing][at % P < T ? at % P : 0];
                            f = __uint_as_float(__float_as_uint(f) & (unsigned)((int)(in << (31 - at % P)) >> 31));
                        }
                    }
                    // eight places: hi and lo
                    v4i hi, lo;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int p0 = 8 * k + 2 * j, p1 = p0 + 1;
                        const bool u0 = p0 / P < kPairs && p0 % P < T, u1 = p1 / P < kPairs && p1 % P < T;
                        const float f0 = u0 ? x[p0 / P % kRing][p0 % P < T ? p0 % P : 0] : 0.0f, f1 = u1 ? x[p1 / P % kRing][p1 % P < T ? p1 % P : 0] : 0.0f;
                        const h2 v = __builtin_convertvector(v2f{f0, f1}, h2);
                        const h2 w = __builtin_convertvector(v2f{u0 ? minus_half<0>(f0, v) : 0.0f, u1 ? minus_half<1>(f1, v) : 0.0f}, h2);
                        hi[j] = __builtin_bit_cast(int, v);
                        lo[j] = __builtin_bit_cast(int, w);
                    }
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int at = 8 * k + j;
                        if (at / P >= kPairs || at % P >= T) continue;
                        step_sum += __builtin_fabsf(x[at / P % kRing][at % P < T ? at % P : 0]);
                        if (order::in_old(2 * (at / P)) && order::in_old(2 * (at / P) + 1)) old_sum = step_sum;
                        else if (order::in_old(2 * (at / P)) && (at % P == T - 1 || j == 7)) old_sum = lane < 32 ? step_sum : old_sum;
                    }
                    if constexpr (kParts) {
                        step_parts = __builtin_fmaf(step_sum, (float)order::roundings(k, false), step_parts);
                        old_parts = __builtin_fmaf(old_sum, (float)order::roundings(k, true), old_parts);
                    }
                    if (check) {  // uniform
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const int at = 8 * k + j;
                            if (at / P < kPairs && at % P < T) step_off = __builtin_fmaxf(step_off, __builtin_amdgcn_fractf(x[at / P % kRing][at % P < T ? at % P : 0] * 256.0f));
                            if (order::in_old(2 * (at / P)) && order::in_old(2 * (at / P) + 1)) old_off = step_off;
                            else if (order::in_old(2 * (at / P))) old_off = lane < 32 ? step_off : old_off;
                        }
                    }
                    // the pairs that are used up make room
#pragma unroll
                    for (int i = 8 * k / P; i < (k == KS - 1 ? kPairs : 8 * (k + 1) / P); ++i) {
                        if (i + kRing < kPairs)
                            load(ay, path, i + kRing);
                        else if (more)  // uniform
                            load(ay + advance, next_path, i + kRing - kPairs);
                    }
                    if (k == KS - 1) {
                        if (check) {  // uniform; an input of 2^15 or more can have more bits than the halves hold
                            step_off = step_sum < 32768.0f ? step_off : 1.0f;
                            old_off = old_sum < 32768.0f ? old_off : 1.0f;
                        }
#pragma unroll
                        for (int d = D - 1; d > 0; --d) {
                            const bool old = d == D - 1;
                            if constexpr (kParts) parts[d] = __builtin_fmaf(sum[d - 1], (float)order::roundings(old), parts[d - 1]) + (old ? old_parts : step_parts);
                            sum[d] = sum[d - 1] + (old ? old_sum : step_sum);
                            off[d] = __builtin_fmaxf(off[d - 1], old ? old_off : step_off);
                        }
                        parts[0] = step_parts, sum[0] = step_sum, off[0] = step_off;
                        const float all = both_halves(sum[D - 1]);
                        small = all < 0.49f;
                        const float e = __builtin_fmaf(all, q.bound_sum, kParts ? __builtin_fmaf(both_halves(parts[D - 1]), q.bound_parts, q.bound_add) : q.bound_add);
                        bad = !(e < 3.0e4f);
                        _Float16 eh = (_Float16)e;
                        bool exact = false;
                        if (check) {  // uniform
                            const auto so = __builtin_amdgcn_permlane32_swap(__float_as_uint(off[D - 1]), __float_as_uint(off[D - 1]), false, false);
                            exact = (so[0] | so[1]) == 0u;
                            if (!keep_checking && done >= cy && __ballot(!exact) != 0) check = false;
                            exact = exact & (kFromThreshold ? (all < 3.2e4f) & steps_256 : all < 6.5e4f);  // (with a threshold: below 2^16 together)
                        }
                        if (exact | bad) eh = (_Float16)0.0f;  // (bad: nothing infinite may meet the other sets' zeros)
                        if constexpr (kFromThreshold) {
                            two_e = exact ? 0.0f : e;
                        } else {
                            lowered = (float)eh;
                            two_e = 2.002f * lowered;
                            if (kBoundInSum && lane >= 32) hi[kBoundPlace / 2] |= (int)((uint32_t)(__builtin_bit_cast(uint16_t, eh) | 0x8000u) << 16);
                        }
                    }
                    // lo, then hi; the first product of a step moves a set's sums on to the next.  A set's weights are read while the
                    // one before it is multiplied.  (7x7/4: the test for rows of other bands costs it registers that it does not have:
                    // 111 us -> 151; elsewhere 2 to 6 % less.)
#pragma unroll
                    for (int d = D - 1; d >= 0; --d) {
                        v4i a[MT];
#pragma unroll
                        for (int m = 0; m < MT; ++m) a[m] = weights[m];
                        read_weights(d > 0 ? d - 1 : D - 1, d > 0 ? k : (k + 1) % KS);
                        if (D > 1 && (R != 7 || (A == 2 && T == 7)) && (block - d < first_row || block - d >= cy_end)) continue;  // uniform: not a row of this band
#pragma unroll
                        for (int m = 0; m < MT; ++m) {
                            v16f c = acc[d][m];
                            if (k == 0) {
                                if (d > 0) {
                                    c = acc[d > 0 ? d - 1 : 0][m];
                                } else if (kFromThreshold) {
                                    const v4f* const tp = reinterpret_cast<const v4f*>(thr + m * 32 + (lane >> 5) * 16);
#pragma unroll
                                    for (int i = 0; i < 16; ++i) c[i] = tp[i >> 2][i & 3];
                                } else {
#pragma unroll
                                    for (int i = 0; i < 16; ++i) c[i] = 0.0f;
                                }
                            }
                            acc[d][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a[m]), __builtin_bit_cast(h8, lo), c, 0, 0, 0);
                        }
#pragma unroll
                        for (int m = 0; m < MT; ++m)
                            acc[d][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a[m]), __builtin_bit_cast(h8, hi), acc[d][m], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                ++block;
                if (done < cy) continue;  // the first rows' sums are not complete
                // (An input outside the fp16 range has an infinity in hi and another in lo: no sum of its window is a number then,
                // and none of a window whose rows only met zero weights with it.)
                bad |= acc[D - 1][0][0] != acc[D - 1][0][0];
                if constexpr (!kFromThreshold && !kBoundInSum) {
#pragma unroll
                    for (int m = 0; m < MT; ++m)
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[D - 1][m][i] -= lowered;
                }
                // ---- bits (MSB first; the sign of S - E - bn, inverted), residual, doubtful values
                asm volatile("" : "+v"(ln));
                const int h = ln >> 5;
                const bool valid = b0 + (ln & (NI - 1)) < p.B && g * NX + ((ln & 31) >> q.ni_log2) < xcols;
                if constexpr (kFromThreshold) {
                    // the sums are S - bn: their signs are the bits, and those within E of 0 are in doubt (rare: the nearest tells)
                    float nearest[MT];
                    uint32_t bits[MT];
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        uint32_t w = 0u;
                        nearest[m] = INFINITY;
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            w = __builtin_amdgcn_alignbit(w, __float_as_uint(acc[D - 1][m][i]), 31);
                            nearest[m] = __builtin_fminf(nearest[m], __builtin_fabsf(acc[D - 1][m][i]));
                        }
                        bits[m] = ~w & 0xffffu;
                    }
                    const float least = __builtin_fminf(nearest[0], nearest[1]);
                    if (__ballot(bad | !(least > two_e)) != 0) {  // uniform
#pragma unroll
                        for (int m = 0; m < MT; ++m) {
                            uint32_t dm = 0u;
#pragma unroll
                            for (int i = 0; i < 16; ++i) dm = __builtin_amdgcn_alignbit(dm, __builtin_fabsf(acc[D - 1][m][i]) > two_e ? 0u : 0x80000000u, 31);
                            dm = bad ? 0xffffu : (two_e == 0.0f ? 0u : dm & 0xffffu);
                            undecided |= (valid ? dm : 0u) << (16 * m);
                            bits[m] &= ~dm;  // (a bit in doubt is 0 here: the recomputation only ever sets it)
                        }
                    }
#pragma unroll
                    for (int m = 0; m < MT; ++m) word[m] |= bits[m];
                } else {
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        const v4f* const tp = reinterpret_cast<const v4f*>(thr + m * 32 + 16 * h);
                        // Signs are collected MSB first (bit 15 - i: channel i).  w: S - E < bn, dm: values in doubt.  Integers
                        // within E are common (in every other tile) and collected like the bits; thresholds within E are
                        // rare: the tile's nearest distance below a threshold tells whether to look for them.
                        uint32_t w = 0u, dm = 0u;
                        int nearest = INT32_MAX;
                        {
                            const v4f th[4] = {tp[0], tp[1], tp[2], tp[3]};
#pragma unroll
                            for (int i = 0; i < 16; ++i) {
                                const float d = acc[D - 1][m][i] - th[i >> 2][i & 3];
                                w = __builtin_amdgcn_alignbit(w, __float_as_uint(d), 31);
                                nearest = min(nearest, __float_as_int(d));
                                dm = __builtin_amdgcn_alignbit(dm, __float_as_uint(__builtin_amdgcn_fractf(-acc[D - 1][m][i]) - two_e), 31);
                            }
                        }
                        dm = small ? 0u : dm;
                        // (NaN: `bad` is set)
                        if (__ballot(bad | (nearest <= (int)(0x80000000u | __float_as_uint(two_e)))) != 0) {
                            uint32_t w2 = 0u;
#pragma unroll
                            for (int i = 0; i < 16; ++i) {
                                float a = acc[D - 1][m][i];
                                asm volatile("" : "+v"(a));  // (evaluated again here: not kept from above)
                                const float d = a - tp[i >> 2][i & 3];
                                w2 = __builtin_amdgcn_alignbit(w2, __float_as_uint(d + two_e), 31);
                            }
                            dm = bad ? 0xffffu : (w & ~w2) | dm;
                            w = bad ? 0xffffu : w;
                        }
                        undecided |= (valid ? dm & 0xffffu : 0u) << (16 * m);
                        word[m] |= ~w & 0xffffu;  // (a bit in doubt is 0 here: the recomputation only ever sets it)
                        int v[16];
#pragma unroll
                        for (int i = 0; i < 16; ++i) v[i] = (int)acc[D - 1][m][i];
                        const unsigned item = (unsigned)(done * p.PW + g * NX) * pixel_b + (unsigned)((tile0 + m) * 2) * group_b;
                        store_residual_group<RES>(res_rsrc, p.res_fmt, valid ? place_residual(ln) + item : kOutOfRange,
                                                  RES == RES_12 ? (valid ? place_residual8(ln) + item : kOutOfRange) : 0u, uB * 16u, v);
                        __builtin_amdgcn_sched_barrier(0);  // (one tile at a time: registers)
                    }
                }
            } else {
                undecided = ordered_sums(cy, word);
            }
            const bool last = cy + 1 == cy_end;
            if (POOL > 1 && (cy & 1) == 0) {
                doubt[0] = undecided;
                ++cy;
                continue;
            }
            doubt[POOL - 1] = undecided;
            // ---- output words: two tiles: lane half h stores the word of tile h; one tile: half 0 stores
            asm volatile("" : "+v"(ln));
            const int h = ln >> 5, img = ln & (NI - 1), xc = g * NX + ((ln & 31) >> q.ni_log2);
            const auto sw = __builtin_amdgcn_permlane32_swap(word[0], word[MT - 1], false, false);
            uint32_t full = (sw[0] << 16) | sw[1];
            if constexpr (POOL > 1) full |= (uint32_t)__shfl_xor((int)full, NI);  // the window's other column
            const unsigned item_word = ((unsigned)(cy / POOL * p.OW + g * NX / POOL) * (unsigned)p.ow + (unsigned)tile0) * uB * 4u;
            __builtin_amdgcn_raw_buffer_store_b32(full, out_rsrc, (int)(xc < xcols ? (kFromThreshold ? word_place : place_word(ln)) + item_word : kOutOfRange), 0, 0);
#pragma unroll
            for (int m = 0; m < MT; ++m) word[m] = 0u;
            // ---- doubtful values of this item go on the list, one per lane at a time.  Recomputed are those of earlier
            // items (their stores are older than this item's, so nothing of this item is waited for), sixteen at a time, and
            // all that are there where the list is full and after the wave's last item.
            const uint32_t any = doubt[0] | doubt[POOL - 1];
            const unsigned long long lanes = __ballot(any != 0u);
            if (!kOrdered && lanes != 0) {  // uniform
                if (__builtin_popcountll(lanes) >= (check ? kManyLanesChecked : kManyLanes) ||
                    __ballot(__builtin_popcount(doubt[0]) >= kManyInLane || (POOL > 1 && __builtin_popcount(doubt[POOL - 1]) >= kManyInLane)) != 0) {
                    cy -= POOL - 1;  // (what is stored of this item is stored again)
                    return;
                }
            }
            bool go = count >= kBatch;
            if (go) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(RES != RES_NONE ? 2 * MT + 1 : 1) : "memory");
            if (go || lanes != 0 || last) {
                for (;;) {
                    if (go) recompute();
                    bool full_list = false;
#pragma unroll
                    for (int py = 0; py < POOL; ++py) {
                        unsigned long long who = __ballot(doubt[py] != 0u);
                        int c;
                        while ((c = __builtin_amdgcn_readfirstlane(__popcll(who))) != 0 && count + c <= kListCap) {
                            if (doubt[py] != 0u) {
                                const int bit = __ffs(doubt[py]) - 1;
                                doubt[py] &= doubt[py] - 1u;
                                const int at = count + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u));
                                list[2 * at] = (uint32_t)(cy - (POOL - 1) + py) << 16 | (uint32_t)xc;
                                list[2 * at + 1] = (uint32_t)((tile0 + (bit >> 4)) * 32 + 16 * h + 15 - (bit & 15)) | (uint32_t)img << 16;
                            }
                            count += c;
                            who = __ballot(doubt[py] != 0u);
                        }
                        full_list |= c != 0;
                    }
                    if (!full_list && (!last || count == 0)) break;
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    go = true;
                }
            }
            ++cy;
        }
    };
    for (;;) {
        pass(std::false_type{});
        if (cy >= cy_end) return;
        if (check) break;
        check = keep_checking = true;
    }
    pass(std::true_type{});
}

// ---------------------------------------------------------------- host side
struct Choice {
    int r, t, a, pool, res;
    Geometry q;
    size_t lds_bytes;
    int grid;
    long long out_bytes, res_bytes;
};

// The instantiation for a problem's form, if there is one: what the networks' first layers need (3- and 7-row filters with strides of 1
// and 2, 2 and 4), and for other strides of such filters one that loads each window whole.  (For other forms, 5x5 filters, pooled
// 3x3, 32-channel 7x7 layers, there is none and nothing has been measured: the kernels of inconv.hip serve them.)  Filters
// narrower than the instantiation's row have the taps beyond masked, like columns outside the frame (loaded tap by tap the
// 7x6/4 layer took 32.6 us for 26.3, 7x5/2 58 for 52).
// Windows loaded whole, 64 channels, 224x224, batch 64, us, inconv.hip -> here, without and with a residual: 3x3/3 26.1 -> 13.8, 29.5 ->
// 21.4; 3x3/5 16.1 -> 8.9, 17.6 -> 13.8; 3x4/2 44 -> 24.7, 52 -> 41.2; 7x7/3 82 -> 41.7, 84 -> 52; 7x7/1 400 -> 274, 415 -> 327; 7x8/3 91 -> 43,
// 93 -> 56; batch 8, 3x3/3 29.8 -> 6.2.  7x8 filters at strides 2 and 4 share rows: 152 -> 64, 155 -> 90 and 53 -> 25.6, 56 -> 37 (windows
// loaded whole 83, 107, 30, 41).
bool instantiated(const InConvParams& p, int cus, Choice* out) {
    Choice& c = *out;
    c.r = p.R;
    c.a = p.stride_h;
    c.res = p.res == nullptr ? RES_NONE : (p.res_fmt == TCBNN_RES_I12 ? RES_12 : RES_WIDE);
    const bool pooled = p.pool_h != 1 || p.pool_w != 1;
    if (p.O % 64 != 0) return false;
    if (p.R == 3 && p.S <= 4 && !pooled) {
        c.t = p.S <= 3 ? 3 : 4, c.pool = 1;
        if (c.a > 2 || (c.a == 2 && c.t == 4)) c.a = 3;
    } else if (p.R == 7 && p.S <= 8 && !pooled) {
        c.t = p.S <= 7 ? 7 : 8, c.pool = 1;
        if (c.a != 2 && c.a != 4) c.a = 7;
    } else if (p.R == 11 && p.S <= 11 && p.pool_h == 2 && p.pool_w == 2 && c.res == RES_NONE && c.a == 4) {
        // Thirteen tiles of a row per compute unit or more: below that, and for 32 channels, the ring in LDS is faster
        // (inconv_mfma_ring.hip has both sides' times).
        if (4LL * p.OH * p.OW * p.B * (p.O / 64) < 13LL * 32 * cus) return false;
        c.t = 11, c.pool = 2;
    } else {
        return false;
    }
    return true;
}

// How a launch is split; false for sizes that the kernel does not take.  `cus`: compute units.
bool choose(const InConvParams& p, int cus, Choice* out) {
    Choice c{};
    if (!instantiated(p, cus, &c)) return false;
    Geometry& q = c.q;
    if (p.PH > 32767 || p.PW > 32767 || p.O > 65535) return false;
    // (32-bit buffer offsets)
    c.out_bytes = 4LL * p.OH * p.OW * p.ow * p.B;
    c.res_bytes = p.res != nullptr ? (long long)tcbnn_residual_bytes(p.PH, p.PW, p.O, p.B, p.res_fmt) : 0;
    if (c.out_bytes >= (1LL << 31) || c.res_bytes >= (1LL << 31)) return false;
    const long long bytes = 12LL * p.H * p.W * p.B + c.out_bytes + c.res_bytes;
    // Residuals of more than the memory-side cache holds (256 MiB with the rest) at few products a byte: the VALU kernel, whose waves
    // store 64 images side by side (3x3/3 at 224x224, batch 128 / 256 / 512: there 43 / 78 / 158 us, here 36 / 93 / 182; 3x4/2, batch 256: 162
    // and 201; 3x3/4, batch 512: 90 and 119).
    if (c.r == 3 && sets_of(c.r, c.a) == 1 && c.res != RES_NONE && bytes > 256LL << 20 && p.B % 64 == 0) return false;
    q.rs_taps = p.R * p.S;
    const int waves = waves_of(c.r), xcols = c.pool > 1 ? c.pool * p.OW : p.PW, sets = sets_of(c.r, c.a), steps = sets * steps_of(c.a, c.t);
    q.cgroups = p.O / (32 * MT);
    q.rows = c.pool * p.OH;

    // Images per 32-column tile.  Fewer than eight are stored in pieces shorter than what memory takes at once, which shows where the
    // launch's bytes are not at home in the memory-side cache with what the network does between two passes: VGG-16's layer
    // within a pass, us: batch 148 in fours 178, 133 in ones 208, 150 in twos 239; in sixteens 125-150.  (Batch 100 in
    // fours 94, in sixteens 95; the 7x7/2 layer at batch 28 in fours 42.3, in eights 47.8.)
    constexpr double kFewer[4] = {2.2, 1.65, 1.25, 1.06};
    const bool large = bytes >= 96LL << 20;
    double best = 1e30;
    int imgtiles = 0;
    const long long target = std::max(1LL, (long long)cus * 4 * waves_per_simd(c.r, c.t, c.a) / q.cgroups);  // resident waves
    const int most = c.res == RES_NONE && c.pool == 1 && (long long)p.B * xcols * q.rows / 32 >= 32 * target ? 4 : 3;
    for (int ni_log2 = most; ni_log2 >= 0; --ni_log2) {
        const int NI = 1 << ni_log2, NX = 32 >> ni_log2;
        if ((long long)NI * 3 * p.H * p.W * 4 >= (1LL << 31)) continue;
        const int tiles = (p.B + NI - 1) >> ni_log2, groups = (xcols + NX - 1) / NX;
        const double cost = (double)tiles * groups * (ni_log2 == most ? 1.0 : (large ? kFewer[ni_log2] : 1.06));
        if (cost < best) {
            best = cost;
            q.ni_log2 = ni_log2;
            q.groups = groups;
            imgtiles = tiles;
        }
    }
    if (best >= 1e30) return false;
    c.lds_bytes = (size_t)steps * MT * 1024 + MT * 128 + (size_t)waves * kListCap * 8 + (size_t)c.r * c.t * MT * 32;

    // Bands of rows: whole rounds of resident waves; a band begins with sets - 1 steps whose rows are only read (0.6 of one)
    const long long per = (long long)imgtiles * q.groups;
    double best_t = 1e30;
    for (int bands = 1; bands <= p.OH; ++bands) {
        const int br = (p.OH + bands - 1) / bands;
        if ((p.OH + br - 1) / br != bands) continue;
        const double t = (double)((per * bands + target - 1) / target) * (br * c.pool + 0.6 * (sets - 1) + 0.5);
        if (t < best_t * 0.999) {
            best_t = t;
            q.bands = bands;
            q.band_rows = br * c.pool;
        }
    }
    const long long total = per * q.bands;
    // 11x11: a launch that leaves a third of the machine's waves out is slower than the ring in LDS too (AlexNet, batch 48 / 64, 1176 and
    // 1568 of 2048 waves with two pooled rows: 44.0 / 46.4 us; there 40.7 / 49.7)
    if (c.r == 11 && total * 10 < target * 7) return false;
    if (total * q.cgroups > 0x0fffffffLL) return false;
    q.total = (int)total;
    q.img_tiles = imgtiles;
    q.units = COLUMNS_BANDS_IMAGES;
    // Large residuals of 3x3 filters.  Waves that drift apart scatter the 128-byte lines that they write over memory; four tiles of images
    // that go down the same rows in step write 512 bytes side by side.  Worth it where the launch's bytes nearly fill the
    // memory-side cache (256 MiB; us within the network's pass, 32x32, 128 channels, batch 768 / 800 / 896 / 1024 / 1100: 64.6 / 72 / 79.6 /
    // 87.5 / 88 -> 65.6 / 69 / 76.5 / 79.6 / 87), beyond it where the 512 bytes are whole pieces of memory (batch 1600 / 2048: 131 / 172 -> 120 /
    // 158; others there have no rule: 1200 / 1300 / 3000: 110 / 102 / 244 -> 113.5 / 113 / 247), and, with the bands in front of the
    // columns, beyond it where frames are wide (on end, 64 channels, 224x224, batch 64 / 128: 150 / 284 -> 131 / 255, 112x112, batch 512:
    // 289 -> 250, 64x64, batch 1024: 192 -> 177; below it 64x64, batch 512 85 -> 90).
    if (c.r == 3 && c.a == 1 && c.res != RES_NONE) {
        if (q.groups < 16 && bytes >= 170LL << 20 && (bytes <= 256LL << 20 || p.B % 32 == 0)) q.units = IMAGES_COLUMNS_BANDS_IN_STEP;
        if (q.groups >= 16 && bytes > 256LL << 20) q.units = IMAGES_BANDS_COLUMNS_IN_STEP;
    }
    q.per_xcd = (q.total + 7) / 8;
    c.grid = 8 * ((q.per_xcd + waves - 1) / waves) * q.cgroups;
    // E (see the top of this file)
    const double T = q.rs_taps, u = std::ldexp(1.0, -24) * 1.02;
    q.bound_parts = (float)u;
    q.bound_sum = (float)((13.5 + (bound_place_free(c.a, c.t) ? 0.0 : 1.0) + (c.t == 7 && c.res != RES_NONE ? 0.0 : T + 4.0 * steps)) * u);
    q.bound_add = (float)(3.0 * T * std::ldexp(1.0, -24) + std::ldexp(1.0, -22));
    *out = c;
    return true;
}

int device_info(int* dev, int* cus) {
    static std::atomic<int> cu_count[kInConvDevices];
    if (int rc = check_hip(hipGetDevice(dev), "hipGetDevice")) return rc;
    if (*dev < 0 || *dev >= kInConvDevices) return fail(TCBNN_EUNSUPPORTED, "inconv: device ordinal %d", *dev);
    int n = cu_count[*dev].load(std::memory_order_acquire);
    if (n == 0) {
        if (int rc = check_hip(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, *dev),
                               "hipDeviceGetAttribute(MultiprocessorCount)"))
            return rc;
        n = std::max(1, n);
        cu_count[*dev].store(n, std::memory_order_release);
    }
    *cus = n;
    return TCBNN_OK;
}

template <int R, int T, int A, int RES, int POOL>
int launch(const InConvParams& p, const Choice& c, int dev, hipStream_t stream) {
    if (c.lds_bytes > 64 * 1024) {
        static std::atomic<bool> ready[kInConvDevices];  // (setting the limit twice does no harm)
        if (!ready[dev].load(std::memory_order_acquire)) {
            const void* fn = reinterpret_cast<const void*>(&inconv_mfma_kernel<R, T, A, RES, POOL>);
            if (int rc = check_hip(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)c.lds_bytes), "hipFuncSetAttribute(MaxDynamicSharedMemorySize)"))
                return rc;
            ready[dev].store(true, std::memory_order_release);
        }
    }
    const uint32_t* pats = reinterpret_cast<const uint32_t*>(p.masks) + (size_t)p.R * p.S * p.opad * 4;
    hipLaunchKernelGGL((inconv_mfma_kernel<R, T, A, RES, POOL>), dim3((unsigned)c.grid), dim3(64 * waves_of(R)),
                       c.lds_bytes, stream, KernelArgs{p, c.q, pats, (unsigned)c.out_bytes, (unsigned)c.res_bytes});
    TCBNN_LAUNCH_CHECK("inconv_mfma_kernel");
    return TCBNN_OK;
}

}  // namespace

bool inconv_mfma_kernel_name(const InConvParams& p, char* buf, size_t len) {
    Choice c;
    if (!choose(p, 256, &c)) {
        if (!inconv_mfma_ring_serves(p)) return false;
        snprintf(buf, len, "inconv_mfma_ring_kernel");
        return true;
    }
    snprintf(buf, len, "inconv_mfma_kernel<%d, %d, %d, %d, %d>", c.r, c.t, c.a, c.res, c.pool);
    return true;
}

int launch_inconv_mfma(const InConvParams& p, hipStream_t stream, bool* served) {
    Choice c{};
    *served = p.O % 32 == 0 && (p.R == 3 || p.R == 7 || p.R == 11);
    if (!*served) return TCBNN_OK;
    int dev = 0, cus = 0;
    if (int rc = device_info(&dev, &cus)) return rc;
    if (!choose(p, cus, &c)) return launch_inconv_mfma_ring(p, dev, cus, stream, served);
    auto with_residual = [&](auto go) { return c.res == RES_12 ? go(std::integral_constant<int, RES_12>{}) : (c.res == RES_WIDE ? go(std::integral_constant<int, RES_WIDE>{}) : go(std::integral_constant<int, RES_NONE>{})); };
    if (c.r == 3)
        return with_residual([&](auto res) {
            constexpr int RES = decltype(res)::value;
            if (c.t == 4) return c.a == 1 ? launch<3, 4, 1, RES, 1>(p, c, dev, stream) : launch<3, 4, 3, RES, 1>(p, c, dev, stream);
            return c.a == 1 ? launch<3, 3, 1, RES, 1>(p, c, dev, stream) : (c.a == 2 ? launch<3, 3, 2, RES, 1>(p, c, dev, stream) : launch<3, 3, 3, RES, 1>(p, c, dev, stream));
        });
    if (c.r == 7)
        return with_residual([&](auto res) {
            constexpr int RES = decltype(res)::value;
            if (c.t == 8) return c.a == 4 ? launch<7, 8, 4, RES, 1>(p, c, dev, stream) : (c.a == 2 ? launch<7, 8, 2, RES, 1>(p, c, dev, stream) : launch<7, 8, 7, RES, 1>(p, c, dev, stream));
            return c.a == 4 ? launch<7, 7, 4, RES, 1>(p, c, dev, stream) : (c.a == 2 ? launch<7, 7, 2, RES, 1>(p, c, dev, stream) : launch<7, 7, 7, RES, 1>(p, c, dev, stream));
        });
    return launch<11, 11, 4, RES_NONE, 2>(p, c, dev, stream);
}

}  // namespace tcbnn
