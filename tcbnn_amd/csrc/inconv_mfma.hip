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
// The bound.  u = 2^-24, A = sum of |x| under the window, T = R*S taps.  A rounding of a running sum is at most u times
// that sum, which is at most what has been added so far and at most |S| plus what is still to come: (A + |S|) / 2.  The
// ordered sum has T such roundings and 2 u A more inside its taps; the split drops at most 2 u |x| per input (and 2^-25
// where fp16 runs out of exponents).  An MFMA adds its 16 products in two halves of eight (six, without the fourth channel).
// A half rounds its result once, and what lies below u times its largest product M is lost, of each product and of the sum
// that they are added to (tests/test_gpu_matrix_core.py holds the instruction to this).  An fp16 number has 11 bits, so
// only products below 2^-13 M lose anything: m of them and the sum, (m + 1) u M at most, where the sum is below M.
// The lo steps run first, on sums below 2^-10 A.  For A stands sqrt(3 T sum of hi^2), whose squares are one v_dot2 per
// loaded dword and which such small values hardly enter: by Cauchy and Schwarz the losses of all halves add the most to
// the rest of the bound where m = 0, and then 2 R NQ / (3 T) < 0.25 u A; 2.25 roundings are taken per step, not 2.  From
// 7 rows on E is taken for |S| <= A/2 (partial sums below 3/4 A); a lane with a larger sum looks again with the full
// bound.  -E itself enters the sum as one more product (the fourth channel of the last tap, unused otherwise), so the
// accumulators hold S - E: a bit is certainly 1 where S - E >= bn, certainly 0 below bn - 2E.
// Inputs outside the fp16 range, infinities and NaN make E infinite: all values of such a window are recomputed.
//
// Many values in doubt.  A saved residual puts every sum ON an integer in doubt, and images have areas of such sums: bars of
// +-1 after scaling to [-1, 1], saturated white, bytes, a flat grey of 0.2 (every fifth channel); and E grows with the
// magnitudes: bytes less a mean leave 7 % of the sums in doubt, values in the thousands all of them.  One by one (four at a
// time, a trip to memory and 49 dependent additions) a tile full of them takes 512 rounds, a hundred multiplications' time.
//   grid    : while every row a wave has staged is multiples of 1/256 (bytes, bytes / 128 - 1, +-1), sums of windows with
//             a sum of |x| below 2^16 are exact: every partial sum is a multiple of 1/256 below 2^24 / 256, in both orders.
//             E is 0.  Rows are checked as long as that holds; other inputs pay for the first window.
//   COMMON  : a wave's first pass; it ends at an item with many values in doubt (kManyInLane, kManyLanesCommon; where no
//             residual is saved: at a full list).  The test and the exit cost it 1.5 %; what the later passes do cost 3-9 %
//             inside its loop, by its registers.
//   MARKED  : the window is staged again, and rows from then on, with a mark at every column that is off that grid (the
//             fourth channel of the lo plane).  An item looks at its windows' marks first; E is 0 where there is none.
//   ORDERED : where that still leaves many, sums in the reference's order, 32 columns x 64 channels at a time, as fp32
//             products on the matrix cores (ordered_sums): no values in doubt but those that are no numbers.
// A single wave that leaves the common pass takes 80 us longer (code that no other wave has fetched), and the launch with
// it: the lines lie where none of 25000 items of bytes / 255 (0.6 % in doubt) reaches them.
// ResNet-18's first layer at batch 256, us, in brackets with the list alone: normal data 107 (111), bytes / 128 - 1 92 (245),
// images in [-1, 1] with bars and patches of +-1 over a third 117 (7690), bytes / 255 147 (163), a third of 0.2 grey 271
// (1490), bytes less a mean 326 (1404), normal x 1000 336 (14150); the additions on the VALU (inconv.hip) take 138 for any.
//
// Work split.  A team owns NI images x a strip of xo output columns x a band of output rows, and walks down the rows:
// the input rows of the window stay in LDS (a ring; stride_h new rows per output row, every input row is read and split
// once per strip), as fp16 [row][image][column][4] for hi and the same for lo, image pitch an odd number of 16-byte units
// (conflict-free).  A multiplication is 32 columns = NI images x 32/NI neighbouring pixels (so small batches fill their
// tiles) by 32 MT channels whose +-1 fragments stay in registers; the next rows are requested before it and written
// after it.  A team is ONE wave where its ring fits an eighth (2-wave registers) or twelfth to sixteenth of a CU's LDS:
// waves then never wait for each other (with four waves to a ring and two barriers a row, every row waited for the
// slowest wave's recomputation: ResNet-18's first layer at batch 256 took 170-180 us instead of 105 without doubtful
// values).  11-row filters, whose rings are larger, share one among the four waves of a workgroup.  The four waves of a
// workgroup are neighbouring strips; work of one image tile goes to one XCD.
//
// What binds it: nothing by itself.  At ResNet-18's layer (batch 256, 12-bit residual; 950 VALU instructions and 56 MFMAs per
// 32 columns x 64 channels) the VALU is busy 38 % of the time and the matrix cores 18 %; a wave waits 31 % of its time for
// counters (memory, LDS) and 28 % for its turn to issue: 1792 waves, under two per SIMD, do not hide one another's waits.
// In a network's pass, where the images come from HBM and not from the memory-side cache, the first of these grows.  HBM
// would allow 40 us; the launch fetches 336 MB, 2.2 times the images: a strip's rows are 80 bytes, and lines that neighbouring
// strips share come more than once.
// Measured, us, VALU adds (inconv.hip) -> here.  A launch within the network's pass, kernel trace, batch 256: ResNet-18 7x7/4
// 127 -> 121 (launch after launch on one batch 121 -> 98), 7x7/2 423 -> 315, VGG-16 3x3 399 -> 207, AlexNet 11x11/4 310 -> 137,
// CIFAR ResNet 3x3 27 -> 27, CIFAR VGG (no residual) 23 -> 18.  Events around 20 launches: ResNet-18 batch 8 52 -> 14; 7x7/2
// batch 20 151 -> 38; VGG-16 batch 5 129 -> 14; CIFAR ResNet batch 77 26 -> 18; AlexNet batch 200 403 -> 134, batch 3 137 -> 16.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

#include "inconv.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

constexpr int kThreads = 256;
constexpr int rounds_of(int r) { return r == 3 ? 3 : 5; }  // staging units (column pairs) per thread and step, at most
// Whether E is taken for sums up to A/2: sums of 27 terms pass that in every fortieth value.
constexpr bool bound_for_half(int r) { return r > 3; }
constexpr bool ring_shared(int r) { return r > 7; }          // four waves to a ring, else one
constexpr int kListCap = 64;   // doubtful values a wave keeps
// A wave's passes (top of this file), and what counts as many values in doubt: one lane with this many (of its column's 32;
// a flat area), or this many lanes (of 64) with any.
enum Mode : int { COMMON, MARKED, ORDERED };
constexpr int kManyInLane = 8, kManyLanesCommon = 28, kManyLanesMarked = 32;

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h8u __attribute__((ext_vector_type(8), aligned(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// Saved residual: none, 12 bits, or 16 / 32 bits (looked up at run time).
enum Residual : int { RES_NONE = 0, RES_12 = 1, RES_WIDE = 2 };

// How a staged image row lies in LDS: column pairs of 16 bytes.  A multiplication's 64 lanes read 16 bytes each, half h of
// them pair 2j + h of their pixel's window.  Strides that are multiples of four: even pairs, then odd ones, so that
// neighbouring pixels are neighbouring units (with an image pitch of 2 modulo 4 units the lanes fall into different banks).
// Other even strides: pairs in order, odd pitch.  Odd strides: the same, windows begin inside a pair (8-byte reads).
enum Pairs : int { PAIRS_ANY = 0, PAIRS_EVEN = 1, PAIRS_SPLIT = 2 };

// Workgroups a CU is to hold (one wave of each per SIMD): what the registers allow.
constexpr int workgroups_per_cu(int r) { return r == 3 ? 4 : 2; }

struct Geometry {
    int ni_log2;             // images per tile
    int xo;                  // convolution columns per strip
    int np, pp;              // staged column pairs per image row, and their odd pitch
    int odd_pairs;           // PAIRS_SPLIT: where the odd pairs begin
    int rounds;              // units per lane and step
    int ring;                // input rows in LDS
    int adv;                 // input rows a step moves on by
    int strips, bands, band_rows, imgtiles, cgroups, waves_c;  // waves_c: waves of a workgroup side by side over channels
    int total, per_xcd;
    int rows;                // output rows (pooled)
    int rs_taps;
    unsigned s_magic;        // tap / S == tap * s_magic >> 16 for every tap
    float bound_scale;       // E = bound_scale * sqrt(sum of hi^2) + bound_add for |S| <= half_scale * sqrt(sum of hi^2)
    float bound_scale_full;  // ... and for any S
    float half_scale;
    float bound_add;
    float small_squares;     // sum of hi^2 below which the sum of |x| is below 1/2
    float exact_squares;     // ... below which sums of multiples of 1/256 are exact
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

#define TCBNN_ROW_BCAST(v, t) \
    __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 | (t), 0xf, 0xf, false))

// acc += m of lane T, T + 1, ... N - 1 of each row of 16 lanes, in this order; all N of them, or while taps are left
template <int T, int N, bool ALL>
__device__ __forceinline__ float add_row_taps(float acc, float m, int left) {
    if constexpr (T < N) {
        if (ALL || T < left) {  // uniform
            acc = acc + TCBNN_ROW_BCAST(m, T);
            return add_row_taps<T + 1, N, ALL>(acc, m, left);
        }
    }
    return acc;
}

template <int R, int NQ, int MT, int RES, int POOL, int PAIRS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(workgroups_per_cu(R)))) void inconv_mfma_kernel(
    const KernelArgs args) {
    const SeldomArgs args_at = (SeldomArgs)__builtin_amdgcn_kernarg_segment_ptr();
    const InConvParams& p = args.p;
    const Geometry& q = args.q;
    static_assert(MT * POOL <= 2 && !(RES != RES_NONE && POOL > 1), "doubtful values of an item are 32 bits of a register");
    static_assert(!(ring_shared(R) && RES != RES_NONE), "a wave of a shared ring cannot leave its pass at an item");
    constexpr int NK = R * NQ;  // MFMA steps: four taps (of one filter row) x four channels each
    constexpr int kRounds = rounds_of(R);
    constexpr unsigned kOutOfRange = 0x80000000u;
    extern __shared__ __align__(16) char lds[];

    constexpr bool kShared = ring_shared(R);
    constexpr bool kHalf = bound_for_half(R);
    constexpr int kTeam = kShared ? 4 : 1;  // waves to a ring
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int member = kShared ? wave : 0;
    const int slot_x = (int)blockIdx.x >> 3;
    int work = ((int)blockIdx.x & 7) * q.per_xcd + (kShared ? slot_x : slot_x * 4 + wave);
    const bool idle = (kShared ? slot_x : slot_x * 4 + wave) >= q.per_xcd || work >= q.total;
    if (kShared && idle) return;  // whole workgroup
    if (idle) work = 0;           // (such a wave helps with the thresholds and leaves)
    const int strip = work % q.strips;
    work /= q.strips;
    const int band = work % q.bands;
    work /= q.bands;
    const int cg = work % q.cgroups, it = work / q.cgroups;
    const int NI = 1 << q.ni_log2, NX = 32 >> q.ni_log2;
    const int b0 = it << q.ni_log2;
    const int x0 = strip * q.xo;
    const int oy_begin = band * q.band_rows, oy_end = min(q.rows, oy_begin + q.band_rows);
    const int wc = kShared ? wave % q.waves_c : 0, wg0 = kShared ? wave / q.waves_c : 0, wg_step = kShared ? 4 / q.waves_c : 1;
    const int tile0 = (cg * q.waves_c + wc) * MT;  // first channel tile of this wave
    const int xcols = POOL > 1 ? POOL * p.OW : p.PW;
    const int n_groups = (min(q.xo, xcols - x0) + NX - 1) >> (5 - q.ni_log2);

    // LDS: thresholds of all channels, lists, a flag, then the rings: hi rows, lo rows
    const int row_bytes = (q.pp * 16) << q.ni_log2;
    const int plane = q.ring * row_bytes;
    float* const thr = reinterpret_cast<float*>(lds);
    uint32_t* const list = reinterpret_cast<uint32_t*>(lds) + p.O + wave * 2 * kListCap;
    int* const flags = reinterpret_cast<int*>(lds) + p.O + 4 * 2 * kListCap;  // kShared: rows off the grid; many doubts
    char* const rows = lds + (p.O + 4 * 2 * kListCap + 4) * 4 + (kShared ? 0 : wave * 2 * plane);

    // ---- thresholds (NaN: -infinity, the bit is 1 either way)
    for (int i = tid; i < p.O; i += kThreads) {
        const float t = p.bn[i];
        thr[i] = t != t ? -INFINITY : t;
    }
    if (tid < 2) flags[tid] = 0;
    __syncthreads();
    if (idle) return;

    // ---- +-1 fragments: lane (row n, half h) holds taps 4j + 2h, 4j + 2h + 1 of channel row_to_channel(n), 4 channels each
    v4i wf[NK][MT];
    {
    const int n = lane & 31, h = lane >> 5;
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int o = (tile0 + m) * 32 + mfma::row_to_channel(n);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int s = 4 * (k % NQ) + 2 * h + t;
                const uint32_t pt = args.pats[(size_t)((k / NQ) * p.S + min(s, p.S - 1)) * p.opad + o];
                uint32_t d0 = 0x3c003c00u | ((pt & 4u) << 13) | (pt << 30 & 0x80000000u), d1 = 0x3c00u | ((pt & 1u) << 15);
                if (s >= p.S) d0 = d1 = 0u;
                if (k == NK - 1 && t == 0) d1 |= h == 0 ? 0x3c000000u : 0u;  // the slot that -E enters through
                wf[k][m][2 * t] = (int)d0;
                wf[k][m][2 * t + 1] = (int)d1;
            }
        }
    }

    // ---- staging: units of one column pair x three channels, numbered over (row, image, pair)
    const unsigned plane_b = (unsigned)(p.H * p.W) * 4u;
    const int ax_first = x0 * p.stride_w - p.pad_w;
    const bool edge = ax_first < 0 || ax_first + 2 * q.np > p.W;  // uniform
    __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.in + (size_t)b0 * 3 * p.H * p.W), 0,
                                                                    (int)((unsigned)min(NI, p.B - b0) * 3u * plane_b), 0x00020000);
    unsigned voff[kRounds];  // byte offset of the left column (out of range: no such image)
    unsigned cell[kRounds];  // cell in a row | left column in the frame << 16 | right one << 17 | row << 20
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
        const int e = (member + kTeam * k) * 64 + lane, e2 = e / q.np, pr = e - e2 * q.np, im = e2 & (NI - 1), row = e2 >> q.ni_log2;
        const int ax = ax_first + 2 * pr;
        const bool used = row < q.adv && b0 + im < p.B;
        voff[k] = used ? (unsigned)im * 3u * plane_b + (unsigned)((row * p.W + ax) * 4) : kOutOfRange;
        cell[k] = (unsigned)(im * q.pp + (PAIRS == PAIRS_SPLIT ? (pr >> 1) + (pr & 1) * q.odd_pairs : pr)) | (used && ax >= 0 && ax < p.W ? 1u << 16 : 0u) |
                  (used && ax + 1 >= 0 && ax + 1 < p.W ? 1u << 17 : 0u) | (unsigned)row << 20;
    }
    const int rounds = q.rounds;
    v2f x[kRounds][3];
    auto fetch = [&](int ay_first, int n_rows) __attribute__((always_inline)) {
        const int row_b = ay_first * p.W * 4;
        const bool inner = !edge && ay_first >= 0 && ay_first + q.adv <= p.H;  // uniform (units past n_rows read what nobody uses)
#pragma unroll
        for (int k = 0; k < kRounds; ++k) {
            if (k >= rounds) break;  // uniform
            if (inner) {
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    x[k][c] = __builtin_bit_cast(v2f, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)voff[k], (int)((unsigned)row_b + c * plane_b), 0));
            } else {
                asm volatile("" : "+v"(cell[k]));  // (what is decoded from it is not kept across the multiplication)
                // (an offset can be negative in front of the first image: the row's is part of the lane's here)
                const int row = (int)(cell[k] >> 20), ay = ay_first + row;
                const bool ok = row < n_rows && ay >= 0 && ay < p.H;
                const unsigned oa = ok && (cell[k] >> 16 & 1u) ? voff[k] + (unsigned)row_b : kOutOfRange;
                const unsigned ob = ok && (cell[k] >> 17 & 1u) ? voff[k] + (unsigned)row_b + 4u : kOutOfRange;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    x[k][c][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)oa, (int)(c * plane_b), 0));
                    x[k][c][1] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)ob, (int)(c * plane_b), 0));
                }
            }
        }
    };
    bool grid = true;  // every row staged so far is multiples of 1/256 (rows are checked as long as that holds)
    // marks: the fourth channel of the lo plane says which columns are not multiples of 1/256
    auto split_and_store = [&](auto marks, int n_rows, int slot0) __attribute__((always_inline)) {
        bool on_grid = true;
#pragma unroll
        for (int k = 0; k < kRounds; ++k) {
            if (k >= rounds) break;  // uniform
            const float f[6] = {x[k][0][0], x[k][1][0], x[k][2][0], x[k][0][1], x[k][1][1], x[k][2][1]};
            v4u hi, lo;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const h2 a = __builtin_convertvector(v2f{f[3 * t], f[3 * t + 1]}, h2);
                const h2 c = __builtin_convertvector(v2f{f[3 * t + 2], 0.0f}, h2);
                const h2 al = __builtin_convertvector(v2f{minus_half<0>(f[3 * t], a), minus_half<1>(f[3 * t + 1], a)}, h2);
                const h2 cl = __builtin_convertvector(v2f{minus_half<0>(f[3 * t + 2], c), 0.0f}, h2);
                hi[2 * t] = __builtin_bit_cast(uint32_t, a);
                hi[2 * t + 1] = __builtin_bit_cast(uint32_t, c);
                lo[2 * t] = __builtin_bit_cast(uint32_t, al);
                lo[2 * t + 1] = __builtin_bit_cast(uint32_t, cl);
            }
            if constexpr (decltype(marks)::value) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    float off = 0.0f;
#pragma unroll
                    for (int c = 0; c < 3; ++c) off = __builtin_fmaxf(off, __builtin_amdgcn_fractf(f[3 * t + c] * 256.0f));
                    lo[2 * t + 1] |= off > 0.0f ? 0x10000u : 0u;
                }
            }
            asm volatile("" : "+v"(cell[k]));
            const unsigned row = cell[k] >> 20;
            if (row < (unsigned)n_rows) {
                const unsigned s = (unsigned)slot0 + row, slot = min(s, s - (unsigned)q.ring);  // (ring: the smaller as unsigned)
                char* const dst = rows + slot * (unsigned)row_bytes + (cell[k] & 0xffffu) * 16u;
                *reinterpret_cast<v4u*>(dst) = hi;
                *reinterpret_cast<v4u*>(dst + plane) = lo;
            }
            if (grid) {  // uniform
#pragma unroll
                for (int t = 0; t < 6; ++t) on_grid = on_grid & ((__builtin_amdgcn_fractf(f[t] * 256.0f) == 0.0f) | (row >= (unsigned)n_rows));
            }
        }
        if (grid) {
            const bool mine = __ballot(!on_grid) == 0;
            if constexpr (kShared) {
                if (!mine && lane == 0) flags[0] = 1;
            } else {
                grid = mine;
            }
        }
    };

    // ---- doubtful values: recomputed in the reference's order, 16 lanes per value (lane t of a row: tap 16 c + t), the
    // list's last four at a time.  One trip to memory: inputs, signs and the residual's words are asked for together (the
    // words after the sums, and the threshold from memory: two more trips, 111 us for 107, bytes / 255 163 for 147)
    int count = 0;  // entries on this wave's list (uniform)
    constexpr int NC = (R * 4 * NQ + 15) / 16;
    auto recompute = [&]() __attribute__((always_inline)) {
        const SeldomArgs a = seldom_args(args_at);
        const auto& p = a->p;
        const auto& q = a->q;
        const uint32_t* const pats = a->pats;
        float f[NC][3];
        uint32_t pt[NC];
        const int pending = min(count, 4);
        count -= pending;
        int t16 = lane & 15;
        int taps = q.rs_taps;
        asm volatile("" : "+v"(t16), "+s"(taps));  // (nothing derived from them is kept outside)
        const int e = count + min(lane >> 4, pending - 1);
        const uint32_t ex = list[2 * e], ey = list[2 * e + 1];
        const int ay0 = (int)(ex >> 16) * p.stride_h - p.pad_h, ax0 = (int)(ex & 0xffffu) * p.stride_w - p.pad_w;
        const int o = (int)(ey & 0xffffu);
        const unsigned im = (ey >> 16) * 3u * plane_b;
        const bool active = (lane >> 4) < pending;
        const int bb = b0 + (int)(ey >> 16);
        const unsigned pix = (ex >> 16) / POOL * (unsigned)p.OW + (ex & 0xffffu) / POOL;  // (host: tensors below 2 GiB)
        // What the residual's words hold is asked for now, with the inputs.  Bits [fix_shift, ...) of the 32-bit word fix_at,
        // under fix_mask, are the value's from bit fix_drop on; only this lane changes them, neighbours in the same word are
        // left alone (exclusive or with what differs).
        uint32_t* const residual = reinterpret_cast<uint32_t*>(p.res);
        size_t fix_at = 0;
        int fix_shift = 0, fix_drop = 0;
        uint32_t fix_mask = 0u, old = 0u;
        if constexpr (RES == RES_12) {
            const int bit = 12 * (o & 15), here = min(12, 32 - (bit & 31));
            const bool second = t16 == 1;
            fix_shift = second ? 0 : bit & 31;
            fix_drop = second ? here : 0;
            fix_mask = t16 < 2 ? (1u << (second ? 12 - here : here)) - 1u : 0u;
            fix_at = i12_word_index(pix, (size_t)((p.O + 15) / 16), o >> 4, p.B, bb, (bit >> 5) + (second ? 1 : 0));
        } else if constexpr (RES == RES_WIDE) {
            fix_at = residual_index(p.res_fmt, pix, p.O, o, p.B, bb);
            if (p.res_fmt == TCBNN_RES_I16) {
                fix_shift = (int)(fix_at & 1) * 16;
                fix_mask = t16 == 0 ? 0xffffu : 0u;
                fix_at >>= 1;
            }
        }
        const bool fix = active && fix_mask != 0u;
        if (RES != RES_NONE && fix) old = __hip_atomic_load(residual + fix_at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int tap = 16 * c + t16, r = (int)((unsigned)tap * q.s_magic >> 16), s = tap - r * p.S;
            const int ay = ay0 + r, ax = ax0 + s;
            const bool inside = (tap < taps) & (ay >= 0) & (ay < p.H) & (ax >= 0) & (ax < p.W);  // (else zeros, which add nothing)
            const unsigned at = inside ? im + (unsigned)(ay * p.W + ax) * 4u : kOutOfRange;
#pragma unroll
            for (int ch = 0; ch < 3; ++ch)
                f[c][ch] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)at, (int)(ch * plane_b), 0));
            pt[c] = pats[(unsigned)(min(tap, taps - 1) * p.opad + o)];
        }
        {
            float acc = 0.0f;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const float f0 = __uint_as_float(__float_as_uint(f[c][0]) ^ ((pt[c] & 4u) << 29));
                const float f1 = __uint_as_float(__float_as_uint(f[c][1]) ^ ((pt[c] & 2u) << 30));
                const float f2 = __uint_as_float(__float_as_uint(f[c][2]) ^ ((pt[c] & 1u) << 31));
                const float m = (f0 + f1) + f2;
                if (16 * c + 16 <= taps)  // uniform
                    acc = add_row_taps<0, 16, true>(acc, m, 16);
                else
                    acc = add_row_taps<0, 16, false>(acc, m, taps - 16 * c);
            }
            // (the row's 16 lanes all hold the sum: lane 2 sets the bit, lanes 0 and 1 repair the one or two words)
            if (active && t16 == 2 && !(acc < thr[o]))
                __hip_atomic_fetch_or(p.out + ((pix * (unsigned)p.ow + (unsigned)(o >> 5)) * (unsigned)p.B + (unsigned)bb), 0x80000000u >> (o & 31), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
            if constexpr (RES != RES_NONE) {
                const uint32_t v = (uint32_t)(int)acc;
                const uint32_t d = ((old >> fix_shift ^ v >> fix_drop) & fix_mask) << fix_shift;
                if (fix && d != 0u) __hip_atomic_fetch_xor(residual + fix_at, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (RES == RES_WIDE && active && t16 == 0 && p.res_fmt == TCBNN_RES_I32) residual[fix_at] = v;
            }
        }
    };

    // ---- the window
    int ay0 = oy_begin * POOL * p.stride_h - p.pad_h;  // first input row of the step's window
    int s0 = 0;                                        // its ring slot
    auto stage_window = [&](auto marks) __attribute__((always_inline)) {
        for (int done = 0; done < q.ring; done += q.adv) {
            const int n = min(q.adv, q.ring - done), slot = s0 + done;
            fetch(ay0 + done, n);
            split_and_store(marks, n, slot >= q.ring ? slot - q.ring : slot);
        }
    };
    stage_window(std::false_type{});

    const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)args.out_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t res_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.res, 0, (int)args.res_bytes, 0x00020000);
    // Where this lane stores, relative to the item (uniform): its output word, its 16 residuals (12-bit: the 8-byte part
    // apart); beyond the tensors for an image past the batch.
    const unsigned uB = (unsigned)p.B, group_b = (RES == RES_12 ? 24u : (p.res_fmt == TCBNN_RES_I16 ? 32u : 64u)) * uB;
    const unsigned pixel_b = (unsigned)(p.O / 16) * group_b;
    unsigned place_word, place_res = 0u, place_res8 = 0u;
    {
        const unsigned px = (unsigned)((lane & 31) >> q.ni_log2), h = (unsigned)lane >> 5, b = (unsigned)(b0 + (lane & (NI - 1)));
        const bool image = b < uB;
        place_word = image && (MT == 2 || h == 0u) && (POOL == 1 || (px & 1u) == 0u)
                         ? ((px / POOL * (unsigned)p.ow + (MT == 2 ? h : 0u)) * uB + b) * 4u : kOutOfRange;
        if constexpr (RES != RES_NONE) {
            place_res = image ? px * pixel_b + h * group_b + b * 16u : kOutOfRange;
            place_res8 = image ? px * pixel_b + h * group_b + uB * 16u + b * 8u : kOutOfRange;
        }
    }

    // ---- a whole item in the reference's order: words, residuals; in doubt stay sums that are no numbers.
    // A tap's eight possible values are four and their negatives, so adding one of them to 32 x 32 sums is a product with a
    // matrix of one +-1 and three 0 per row: two v_mfma_f32_32x32x2_f32, each one fp32 addition per sum (adding the zeros
    // changes nothing; tests/test_gpu_matrix_core.py).
    auto ordered_sums = [&](int oy, int g, uint32_t* word, uint32_t& doubt) __attribute__((always_inline)) {
        const SeldomArgs a = seldom_args(args_at);
        const auto& p = a->p;
        const uint32_t* const pats = a->pats;
        int ln = lane;
        asm volatile("" : "+v"(ln));  // (nothing derived from it is kept outside)
        const int h = ln >> 5, img = ln & (NI - 1), xc = x0 + g * NX + ((ln & 31) >> a->q.ni_log2);
        const bool valid = b0 + img < p.B && xc < xcols;
        const int ax0 = xc * p.stride_w - p.pad_w, o0 = tile0 * 32 + mfma::row_to_channel(ln & 31);
        const unsigned im = (unsigned)img * 3u * plane_b, flip = (unsigned)h << 31;
        doubt = 0u;
#pragma unroll
        for (int m = 0; m < MT; ++m) word[m] = 0u;
#pragma unroll 1
        for (int py = 0; py < POOL; ++py) {
            const int ay0 = (oy * POOL + py) * p.stride_h - p.pad_h, r_end = min(R, p.H - ay0);
            v16f acc[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
            // a filter row at a time, requested one row ahead; out of the frame: zeros, which add nothing
            constexpr int kTaps = 4 * NQ;
            float next[kTaps][3];
            uint32_t next_pt[kTaps][MT];
            auto request = [&](int r) __attribute__((always_inline)) {
                const unsigned at0 = im + (unsigned)((ay0 + r) * p.W + ax0) * 4u;
#pragma unroll
                for (int j = 0; j < NQ; ++j) {
                    const int ax = ax0 + 4 * j;
                    const unsigned at = at0 + 16u * j;
                    if (__ballot(valid & ((ax < 0) | (ax + 4 > p.W))) == 0) {  // uniform
#pragma unroll
                        for (int ch = 0; ch < 3; ++ch) {
                            const v4f v = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(valid ? at : kOutOfRange), (int)(ch * plane_b), 0));
#pragma unroll
                            for (int t = 0; t < 4; ++t) next[4 * j + t][ch] = v[t];
                        }
                    } else {
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const bool inside = valid & (ax + t >= 0) & (ax + t < p.W);
#pragma unroll
                            for (int ch = 0; ch < 3; ++ch)
                                next[4 * j + t][ch] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(inside ? at + 4u * t : kOutOfRange), (int)(ch * plane_b), 0));
                        }
                    }
                }
                const uint32_t* const row = pats + (unsigned)(r * p.S * p.opad);  // (uniform)
#pragma unroll
                for (int t = 0; t < kTaps; ++t)
#pragma unroll
                    for (int m = 0; m < MT; ++m) next_pt[t][m] = row[(unsigned)(min(t, p.S - 1) * p.opad + o0 + 32 * m)];
            };
            const int r_begin = max(0, -ay0);
            if (r_begin < r_end) request(r_begin);
#pragma unroll 1
            for (int r = r_begin; r < r_end; ++r) {
                float f[kTaps][3];
                uint32_t pt[kTaps][MT];
#pragma unroll
                for (int t = 0; t < kTaps; ++t) {
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch) f[t][ch] = next[t][ch];
#pragma unroll
                    for (int m = 0; m < MT; ++m) pt[t][m] = next_pt[t][m];
                }
                if (r + 1 < r_end) request(r + 1);
#pragma unroll
                for (int t = 0; t < kTaps; ++t) {
                    if (t >= p.S) break;  // uniform
                    const float f2 = __uint_as_float(__float_as_uint(f[t][2]) ^ flip);
                    const float same = (f[t][0] + f[t][1]) + f2, other = (f[t][0] - f[t][1]) + f2;
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        // pattern 4 neg0 + 2 neg1 + neg2; a pattern from 4 on is the negative of the inverted one
                        const uint32_t neg = (uint32_t)((int)(pt[t][m] << 29) >> 31), c = (pt[t][m] ^ neg) & 3u;
                        const uint32_t one = 0x3f800000u | (neg & 0x80000000u);
                        acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(c == (uint32_t)h ? one : 0u), same, acc[m], 0, 0, 0);
                        acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(c == (uint32_t)h + 2u ? one : 0u), other, acc[m], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const v4f* const tp = reinterpret_cast<const v4f*>(thr + (tile0 + m) * 32 + 16 * h);
                uint32_t w = 0u;
                float zero = 0.0f;  // an infinity or NaN among a tap's values makes NaN of it, times 0, in every sum
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    w = __builtin_amdgcn_alignbit(w, __float_as_uint(acc[m][i] - tp[i >> 2][i & 3]), 31);
                    zero = __builtin_fmaf(acc[m][i], 0.0f, zero);
                }
                const bool bad = !(zero == 0.0f);
                word[m] |= bad ? 0u : ~w & 0xffffu;
                doubt |= (bad && valid ? 0xffffu : 0u) << (16 * (POOL > 1 ? py : m));
                if constexpr (RES != RES_NONE) {
                    int v[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i) v[i] = (int)acc[m][i];
                    const unsigned item = (unsigned)(oy * p.PW + x0 + g * NX) * pixel_b + (unsigned)((tile0 + m) * 2) * group_b;
                    store_residual_group<RES>(res_rsrc, p.res_fmt, valid ? place_res + item : kOutOfRange,
                                              RES == RES_12 ? (valid ? place_res8 + item : kOutOfRange) : 0u, uB * 16u, v);
                    __builtin_amdgcn_sched_barrier(0);  // (one tile at a time: registers)
                }
            }
        }
    };

    // ---- the band's items, in up to three passes.  The common one ends at an item with many values in doubt.  That item and
    // the rest of the band are then done with marks (common sums, exact where a window has none), and from an item on where
    // that still leaves many, in the reference's order.  (A shared ring is left by all its waves together, before the next
    // row, and for ordered sums.)
    int oy = oy_begin, g = wg0;
    bool many = false;
    auto pass = [&](auto mode) __attribute__((always_inline)) {
        constexpr bool kMarked = decltype(mode)::value == MARKED, kOrdered = decltype(mode)::value == ORDERED;
        constexpr int kManyLanes = kMarked ? kManyLanesMarked : kManyLanesCommon;
        // Few sums are ever in doubt where no residual is saved: that there are many is seen by the list, and the pass ends
        // with the row, which costs its loop less.
        constexpr bool kRowExit = RES == RES_NONE && !kShared;
        int first_g = n_groups;
        many = false;
        for (; oy < oy_end; ++oy) {
            const bool more = oy + 1 < oy_end;  // uniform
            if constexpr (kShared && !kOrdered) {
                __syncthreads();
                if (grid) grid = __builtin_amdgcn_readfirstlane(flags[0]) == 0;
                if (__builtin_amdgcn_readfirstlane(flags[1]) != 0) return;  // (written between the two barriers only)
            }
            if (!kOrdered && more) fetch(ay0 + q.ring, q.adv);
            while (g < n_groups) {
                uint32_t word[MT];
                uint32_t doubt = 0u;
                // A lane's place (column of the tile: image and pixel; half of the channels) is worked out anew from a lane
                // index the compiler cannot carry over: kept across the multiplication, the addresses made from it spill.
                int ln = lane;
                asm volatile("" : "+v"(ln));
#pragma unroll
                for (int m = 0; m < MT; ++m) word[m] = 0u;
                if constexpr (!kOrdered) {
#pragma unroll 1
                    for (int py = 0; py < POOL; ++py) {
                        v16f acc[MT];
#pragma unroll
                        for (int m = 0; m < MT; ++m)
#pragma unroll
                            for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
                        const int first_col = (g * NX + ((ln & 31) >> q.ni_log2)) * p.stride_w;
                        const int lane_at = (ln & (NI - 1)) * q.pp * 16 + (PAIRS == PAIRS_SPLIT ? (first_col >> 2) * 16 + (ln >> 5) * q.odd_pairs * 16
                                                                                               : first_col * 8 + (ln >> 5) * 16);
                        auto fragment = [&](int r, int j, int plane_off) -> v4i {
                            int slot = s0 + py * p.stride_h + r;
                            slot = slot >= q.ring ? slot - q.ring : slot;
                            const char* const at = rows + (slot * row_bytes + plane_off) + lane_at + j * (PAIRS == PAIRS_SPLIT ? 16 : 32);
                            if constexpr (PAIRS != PAIRS_ANY)
                                return __builtin_bit_cast(v4i, *reinterpret_cast<const h8*>(at));
                            else
                                return __builtin_bit_cast(v4i, static_cast<h8>(*reinterpret_cast<const h8u*>(at)));
                        };
                        bool exact = false;  // this lane's window has no mark
                        if constexpr (kMarked) {
                            uint32_t marks = 0u;
#pragma unroll 2
                            for (int k = 0; k < NK; ++k) {
                                const v4i v = fragment(k / NQ, k % NQ, plane);
                                const int s = 4 * (k % NQ) + 2 * (ln >> 5);
                                marks |= (s < p.S ? (uint32_t)v[1] : 0u) | (s + 1 < p.S ? (uint32_t)v[3] : 0u);
                            }
                            const auto sw = __builtin_amdgcn_permlane32_swap(marks, marks, false, false);
                            exact = (sw[0] | sw[1]) < 0x10000u;
                        }
                        // lo steps, then hi steps; a step's fragment is requested kAhead steps ahead
                        constexpr int kAhead = 4;
                        v4i ahead[kAhead];
#pragma unroll
                        for (int k = 0; k < kAhead; ++k) ahead[k] = fragment(k % NK / NQ, k % NK % NQ, k < NK ? plane : 0);
                        float sq = 0.0f, two_e = 0.0f, half_a = 0.0f, wide_shift = 0.0f, wide_two_e = 0.0f;
                        bool bad = false, small = false;  // small: |S| and |acc| are below 1/2, the residual is 0
#pragma unroll
                        for (int k = 0; k < 2 * NK; ++k) {
                            v4i v = ahead[k % kAhead];
                            if (k + kAhead < 2 * NK)
                                ahead[k % kAhead] = fragment((k + kAhead) % NK / NQ, (k + kAhead) % NK % NQ, k + kAhead < NK ? plane : 0);
                            if (k >= NK) {
#pragma unroll
                                for (int d = 0; d < 4; ++d) {
                                    const int two = v[d];
                                    sq = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, two), __builtin_bit_cast(h2, two), sq, false);
                                }
                            }
                            if (kMarked && k == NK - 1 && lane < 32) v[1] &= 0xffff;  // (a mark where -E will enter)
                            if (k == 2 * NK - 1) {
                                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(sq), __float_as_uint(sq), false, false);
                                const float all = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
                                const float root = __builtin_amdgcn_sqrtf(all), full = root * q.bound_scale_full + q.bound_add;
                                small = all < q.small_squares;
                                bad = !(all < 4.0e9f) || !(full < 3.0e4f);
                                _Float16 eh = (_Float16)(root * q.bound_scale + q.bound_add);
                                half_a = root * q.half_scale;
                                wide_two_e = 2.002f * full;
                                if ((grid | exact) & (all < q.exact_squares)) {
                                    eh = (_Float16)0.0f;
                                    half_a = INFINITY;
                                }
                                two_e = 2.002f * (float)eh;
                                wide_shift = (float)eh - full;
                                if (lane < 32) v[1] |= (int)((uint32_t)(__builtin_bit_cast(uint16_t, eh) | 0x8000u) << 16);
                            }
#pragma unroll
                            for (int m = 0; m < MT; ++m)
                                acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, wf[k % NK][m]), __builtin_bit_cast(h8, v), acc[m], 0, 0, 0);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        // ---- bits (MSB first; the sign of S - E - bn, inverted), residual, doubtful values
                        asm volatile("" : "+v"(ln));
                        const int h = ln >> 5;
                        const bool valid = b0 + (ln & (NI - 1)) < p.B && x0 + g * NX + ((ln & 31) >> q.ni_log2) < xcols;
#pragma unroll
                        for (int m = 0; m < MT; ++m) {
                            const v4f* const tp = reinterpret_cast<const v4f*>(thr + (tile0 + m) * 32 + 16 * h);
                            // Signs are collected MSB first (bit 15 - i: channel i).  w: S - E < bn, dm: values in doubt.  Integers
                            // within E are common (in every other tile) and collected like the bits; thresholds within E and sums
                            // above A/2 (E is less than a bound for those) are rare: the tile's nearest distance below a threshold
                            // and its largest |S| tell whether to look for them.
                            uint32_t w = 0u, dm = 0u;
                            int nearest = INT32_MAX;
                            float most = 0.0f;
                            {
                                const v4f th[4] = {tp[0], tp[1], tp[2], tp[3]};
#pragma unroll
                                for (int i = 0; i < 16; ++i) {
                                    const float d = acc[m][i] - th[i >> 2][i & 3];
                                    w = __builtin_amdgcn_alignbit(w, __float_as_uint(d), 31);
                                    nearest = min(nearest, __float_as_int(d));
                                    if constexpr (kHalf) most = __builtin_fmaxf(most, __builtin_fabsf(acc[m][i]));
                                    if constexpr (RES != RES_NONE)
                                        dm = __builtin_amdgcn_alignbit(dm, __float_as_uint(__builtin_amdgcn_fractf(-acc[m][i]) - two_e), 31);
                                }
                            }
                            if constexpr (RES != RES_NONE) dm = small ? 0u : dm;
                            // (NaN: `bad` is set)
                            if (__ballot(bad | (kHalf & !(most <= half_a)) | (nearest <= (int)(0x80000000u | __float_as_uint(two_e)))) != 0) {
                                const bool wide = kHalf & !(most <= half_a);  // this lane's sums with the full bound
                                const float shift = wide ? wide_shift : 0.0f, two = wide ? wide_two_e : two_e;
                                uint32_t w2 = 0u, r = 0u;
                                w = 0u;
#pragma unroll
                                for (int i = 0; i < 16; ++i) {
                                    float a = acc[m][i];
                                    asm volatile("" : "+v"(a));  // (evaluated again here: not kept from above)
                                    a += shift;
                                    const float d = a - tp[i >> 2][i & 3];
                                    w = __builtin_amdgcn_alignbit(w, __float_as_uint(d), 31);
                                    w2 = __builtin_amdgcn_alignbit(w2, __float_as_uint(d + two), 31);
                                    if constexpr (RES != RES_NONE) r = __builtin_amdgcn_alignbit(r, __float_as_uint(__builtin_amdgcn_fractf(-a) - two), 31);
                                }
                                w = bad ? 0xffffu : w;
                                dm = bad ? 0xffffu : (w & ~w2) | (wide || !small ? r : 0u);
                            }
                            doubt |= (valid ? dm & 0xffffu : 0u) << (16 * (POOL > 1 ? py : m));
                            word[m] |= ~w & 0xffffu;  // (a bit in doubt is 0 here: the recomputation only ever sets it)
                            if constexpr (RES != RES_NONE) {
                                int v[16];
#pragma unroll
                                for (int i = 0; i < 16; ++i) v[i] = (int)acc[m][i];
                                const unsigned item = (unsigned)(oy * p.PW + x0 + g * NX) * pixel_b + (unsigned)((tile0 + m) * 2) * group_b;
                                store_residual_group<RES>(res_rsrc, p.res_fmt, valid ? place_res + item : kOutOfRange,
                                                          RES == RES_12 ? (valid ? place_res8 + item : kOutOfRange) : 0u, uB * 16u, v);
                                __builtin_amdgcn_sched_barrier(0);  // (one tile at a time: registers)
                            }
                        }
                    }
                }
                if constexpr (kOrdered) ordered_sums(oy, g, word, doubt);
                // ---- output words: two tiles: lane half h stores the word of tile h; one tile: half 0 stores
                asm volatile("" : "+v"(ln));
                const int h = ln >> 5, img = ln & (NI - 1), xc = x0 + g * NX + ((ln & 31) >> q.ni_log2);
                const auto sw = __builtin_amdgcn_permlane32_swap(word[0], word[MT - 1], false, false);
                uint32_t full = (sw[0] << 16) | sw[1];
                if constexpr (POOL > 1) full |= (uint32_t)__shfl_xor((int)full, NI);  // the window's other column
                const unsigned item_word = ((unsigned)(oy * p.OW + (x0 + g * NX) / POOL) * (unsigned)p.ow + (unsigned)tile0) * uB * 4u;
                __builtin_amdgcn_raw_buffer_store_b32(full, out_rsrc, (int)(xc < xcols ? place_word + item_word : kOutOfRange), 0, 0);
                // ---- doubtful values of this item go on the list, one per lane at a time.  Recomputed are those of earlier
                // items (their stores are older than this item's, so nothing of this item is waited for), four at a time, and
                // all that are there where the list is full and after the wave's last item.
                const bool last = !more && g + wg_step >= n_groups;
                if (count >= 4) {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(RES != RES_NONE ? 2 * MT + 1 : 1) : "memory");
                    recompute();
                }
                unsigned long long who = __ballot(doubt != 0u);
                const int earlier = count;
                if (!kOrdered && RES != RES_NONE && who != 0) {  // uniform
                    many = __builtin_popcountll(who) >= kManyLanes || __ballot(__builtin_popcount(doubt) >= kManyInLane) != 0;
                    if (many) who = 0;  // (what is stored of this item is stored again)
                }
                if (!kOrdered && kRowExit && many) who = 0;
                for (;;) {
                    int c;
                    while ((c = __builtin_amdgcn_readfirstlane(__popcll(who))) != 0 && count + c <= kListCap) {
                        if (doubt != 0u) {
                            const int bit = __ffs(doubt) - 1;
                            doubt &= doubt - 1u;
                            const int at = count + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u));
                            const int py = POOL > 1 ? bit >> 4 : 0, m = POOL > 1 ? 0 : bit >> 4;
                            list[2 * at] = (uint32_t)(oy * POOL + py) << 16 | (uint32_t)xc;
                            list[2 * at + 1] = (uint32_t)((tile0 + m) * 32 + 16 * h + 15 - (bit & 15)) | (uint32_t)img << 16;
                        }
                        count += c;
                        who = __ballot(doubt != 0u);
                    }
                    if (c == 0 && (!last || count == 0 || (!kShared && many))) break;
                    if (!kOrdered && RES == RES_NONE && c != 0) {  // the list is full
                        many = true;
                        if constexpr (kRowExit) {
                            first_g = g;
                            count = earlier;
                            break;
                        }
                    }
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    do recompute();
                    while (count > kListCap / 2);
                }
                if (RES != RES_NONE && many) return;
                g += wg_step;
            }
            if (kRowExit && many) {
                g = first_g;
                return;
            }
            g = wg0;
            if constexpr (kShared && !kOrdered) {
                __syncthreads();
                if (many && lane == 0) flags[1] = 1;
            }
            if (!kOrdered && more) split_and_store(std::bool_constant<kMarked>{}, q.adv, s0);
            ay0 += q.adv;
            s0 += q.adv;
            s0 = s0 >= q.ring ? s0 - q.ring : s0;
        }
    };
    pass(std::integral_constant<Mode, COMMON>{});
    if (!kShared && oy < oy_end) {
        stage_window(std::true_type{});
        pass(std::integral_constant<Mode, MARKED>{});
    }
    if (oy < oy_end) pass(std::integral_constant<Mode, ORDERED>{});
}

// ---------------------------------------------------------------- host side
constexpr int kMaxDevices = 64;
constexpr int kLdsPerCu = 160 * 1024;

struct Choice {
    int r, nq, mt, pool;
    int res, pairs;
    int wg_per_cu;
    Geometry q;
    size_t lds_bytes;
    int grid;
    long long out_bytes, res_bytes;
};

size_t lds_extra(int channels) { return (size_t)(channels + 4 * 2 * kListCap + 4) * 4; }

// The instantiation for a problem's form, if there is one: what the networks' first layers need.  (For other forms, 5x5
// filters, pooled 3x3, 32-channel or odd-stride 7x7 layers, there is none and nothing has been measured: the kernels of
// inconv.hip serve them.)
bool instantiated(const InConvParams& p, Choice* out) {
    Choice& c = *out;
    c.r = p.R;
    c.nq = (p.S + 3) / 4;
    c.res = p.res == nullptr ? RES_NONE : (p.res_fmt == TCBNN_RES_I12 ? RES_12 : RES_WIDE);
    c.pairs = p.stride_w % 4 == 0 ? PAIRS_SPLIT : (p.stride_w % 2 == 0 ? PAIRS_EVEN : PAIRS_ANY);
    const bool pooled = p.pool_h != 1 || p.pool_w != 1;
    if (p.R == 3 && c.nq == 1 && !pooled && p.O % 64 == 0 && c.pairs != PAIRS_SPLIT) {
        c.mt = 2, c.pool = 1;
    } else if (p.R == 7 && c.nq == 2 && !pooled && p.O % 64 == 0 && c.pairs != PAIRS_ANY) {
        c.mt = 2, c.pool = 1;
    } else if (p.R == 11 && c.nq == 3 && p.pool_h == 2 && p.pool_w == 2 && p.O % 32 == 0 && c.pairs == PAIRS_SPLIT) {
        c.mt = 1, c.pool = 2;
    } else {
        return false;
    }
    return true;
}

// How a launch is split; false for sizes that the kernel does not take.  `cus`: compute units.
bool choose(const InConvParams& p, int cus, Choice* out) {
    Choice c{};
    if (!instantiated(p, &c)) return false;
    c.wg_per_cu = workgroups_per_cu(c.r);
    Geometry& q = c.q;
    q.adv = c.pool * p.stride_h;
    q.ring = p.R + (c.pool - 1) * p.stride_h;
    if (q.adv > q.ring) return false;
    if (p.PH > 32767 || p.PW > 32767 || p.O > 65535) return false;
    // (32-bit buffer offsets)
    c.out_bytes = 4LL * p.OH * p.OW * p.ow * p.B;
    c.res_bytes = p.res != nullptr ? (long long)tcbnn_residual_bytes(p.PH, p.PW, p.O, p.B, p.res_fmt) : 0;
    if (c.out_bytes >= (1LL << 31) || c.res_bytes >= (1LL << 31)) return false;
    q.rows = p.OH;
    q.rs_taps = p.R * p.S;
    const bool shared = ring_shared(c.r);
    const int teams = shared ? 1 : 4;  // per workgroup
    const int chp = p.O / (32 * c.mt);
    q.waves_c = !shared ? 1 : (chp % 4 == 0 ? 4 : (chp % 2 == 0 ? 2 : 1));
    q.cgroups = chp / q.waves_c;
    const size_t extra = lds_extra(p.O), share = (size_t)kLdsPerCu / c.wg_per_cu;
    if (extra >= share) return false;
    const size_t lds_limit = (share - extra) / teams;
    q.s_magic = 65536u / (unsigned)p.S + 1u;
    for (int t = 0; t < q.rs_taps; ++t)
        if ((int)((unsigned)t * q.s_magic >> 16) != t / p.S) return false;

    // Images per 32-column tile and columns per strip: the cheapest over the batch and the width, in rough cycles of a
    // wave: items (multiplication and epilogue) and staging rounds.  At most eight images (eight images' residuals of a
    // pixel are a whole 128-byte line; more would leave no room for a strip), fewer than that only where it is worth an
    // eighth; a pooled layer needs neighbouring pixels in one tile and stores little.
    const int xcols = c.pool > 1 ? c.pool * p.OW : p.PW;
    const int item = p.R == 3 ? 900 : (p.R == 7 ? 2300 : 3200) * c.pool;
    double best = 1e30;
    int most_images = 3;
    while (most_images > 0 && (1 << (most_images - 1)) >= p.B) --most_images;
    for (int ni_log2 = most_images; ni_log2 >= std::max(0, most_images - 2); --ni_log2) {
        const int NI = 1 << ni_log2, NX = 32 >> ni_log2, step = std::max(NX, c.pool), imgtiles = (p.B + NI - 1) >> ni_log2;
        if ((long long)NI * 3 * p.H * p.W * 4 >= (1LL << 31)) continue;
        for (int xo = step; xo < xcols + step; xo += step) {
            const int np = ((xo - 1) * p.stride_w + 4 * c.nq + 1) / 2, odd = (np + 1) / 2;
            const int pp = c.pairs == PAIRS_SPLIT ? 2 * odd + (odd % 2 == 0 ? 2 : 0) : np | 1;
            const int per_round = shared ? 256 : 64, units = (np * NI * q.adv + per_round - 1) / per_round;
            const size_t bytes = (size_t)2 * q.ring * NI * pp * 16;
            if (units > rounds_of(p.R) || bytes > lds_limit || NI * pp > 0xffff) break;
            const int groups = xo / NX, strips = (xcols + xo - 1) / xo;
            const int rounds = shared ? (groups * q.waves_c + 3) / 4 : groups;
            const double cost = (double)imgtiles * strips * (rounds * (double)item + 200.0 * units + (shared ? 500.0 : 100.0)) *
                                (ni_log2 < most_images && c.pool == 1 ? 1.125 : 1.0);
            if (cost < best * 0.999) {
                best = cost;
                q.ni_log2 = ni_log2;
                q.imgtiles = imgtiles;
                q.xo = xo;
                q.np = np;
                q.pp = pp;
                q.odd_pairs = odd;
                q.rounds = units;
                q.strips = strips;
            }
        }
    }
    if (best >= 1e30) return false;
    c.lds_bytes = (size_t)2 * q.ring * ((size_t)q.pp << q.ni_log2) * 16 * teams + extra;

    // Bands of rows: one round of resident workgroups where the width and the batch leave a choice; a band's first
    // window is staged whole (counted as 0.7 of a row's work).
    const long long per = (long long)q.imgtiles * q.cgroups * q.strips, target = (long long)cus * c.wg_per_cu * teams;
    double best_t = 1e30;
    for (int bands = 1; bands <= q.rows; ++bands) {
        const int br = (q.rows + bands - 1) / bands;
        if ((q.rows + br - 1) / br != bands) continue;
        const double t = (double)((per * bands + target - 1) / target) * (br + 0.7);
        if (t < best_t * 0.999) {
            best_t = t;
            q.bands = bands;
            q.band_rows = br;
        }
    }
    const long long total = per * q.bands;
    if (total > 0x0fffffffLL) return false;
    q.total = (int)total;
    q.per_xcd = (q.total + 7) / 8;  // (teams)
    c.grid = 8 * ((q.per_xcd + teams - 1) / teams);
    // E (see the top of this file): the roundings of sums, T of the reference's and 2 per hi step and for -E (2.25 taken:
    // what the halves lose) with partial sums below (A + |S|) / 2 <= 0.75 A (or A); 2 u A for the additions in a tap, 2 u A for the split, and
    // 0.5 u A for the lo steps.  2 % cover the roundings of the bound itself.
    const double T = q.rs_taps, u = std::ldexp(1.0, -24), sums = T + 2.25 * (p.R * c.nq + 1), a_scale = std::sqrt(3.0 * T);
    q.bound_scale = (float)(((bound_for_half(p.R) ? 0.75 : 1.0) * sums + 4.5) * u * 1.02 * a_scale);
    q.bound_scale_full = (float)((sums + 4.5) * u * 1.02 * a_scale);
    q.half_scale = (float)(0.49 * a_scale);
    q.bound_add = (float)(3.0 * T * std::ldexp(1.0, -24) + std::ldexp(1.0, -22));
    q.small_squares = (float)(0.2 / (3.0 * T));
    q.exact_squares = (float)(60000.0 * 60000.0 / (3.0 * T));  // (sum of |x| below 2^16 = 2^24 / 256)
    *out = c;
    return true;
}

int device_info(int* dev, int* cus) {
    static std::atomic<int> cu_count[kMaxDevices];
    if (int rc = check_hip(hipGetDevice(dev), "hipGetDevice")) return rc;
    if (*dev < 0 || *dev >= kMaxDevices) return fail(TCBNN_EUNSUPPORTED, "inconv: device ordinal %d", *dev);
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

template <int R, int NQ, int MT, int RES, int POOL, int PAIRS>
int launch(const InConvParams& p, const Choice& c, int dev, hipStream_t stream) {
    static std::atomic<bool> ready[kMaxDevices];  // (setting the limit twice does no harm)
    if (!ready[dev].load(std::memory_order_acquire)) {
        const void* fn = reinterpret_cast<const void*>(&inconv_mfma_kernel<R, NQ, MT, RES, POOL, PAIRS>);
        if (int rc = check_hip(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsPerCu / workgroups_per_cu(R)),
                               "hipFuncSetAttribute(MaxDynamicSharedMemorySize)"))
            return rc;
        ready[dev].store(true, std::memory_order_release);
    }
    const uint32_t* pats = reinterpret_cast<const uint32_t*>(p.masks) + (size_t)p.R * p.S * p.opad * 4;
    hipLaunchKernelGGL((inconv_mfma_kernel<R, NQ, MT, RES, POOL, PAIRS>), dim3((unsigned)c.grid), dim3(kThreads),
                       c.lds_bytes, stream, KernelArgs{p, c.q, pats, (unsigned)c.out_bytes, (unsigned)c.res_bytes});
    TCBNN_LAUNCH_CHECK("inconv_mfma_kernel");
    return TCBNN_OK;
}

}  // namespace

bool inconv_mfma_kernel_name(const InConvParams& p, char* buf, size_t len) {
    Choice c;
    if (!choose(p, 256, &c)) return false;
    snprintf(buf, len, "inconv_mfma_kernel<%d, %d, %d, %d, %d, %d>", c.r, c.nq, c.mt, c.res, c.pool, c.pairs);
    return true;
}

int launch_inconv_mfma(const InConvParams& p, hipStream_t stream, bool* served) {
    Choice c{};
    *served = instantiated(p, &c);
    if (!*served) return TCBNN_OK;
    int dev = 0, cus = 0;
    if (int rc = device_info(&dev, &cus)) return rc;
    *served = choose(p, cus, &c);
    if (!*served) return TCBNN_OK;
    auto with_residual = [&](auto go) { return c.res == RES_12 ? go(std::integral_constant<int, RES_12>{}) : (c.res == RES_WIDE ? go(std::integral_constant<int, RES_WIDE>{}) : go(std::integral_constant<int, RES_NONE>{})); };
    if (c.r == 3)
        return with_residual([&](auto res) {
            return c.pairs == PAIRS_EVEN ? launch<3, 1, 2, decltype(res)::value, 1, PAIRS_EVEN>(p, c, dev, stream) : launch<3, 1, 2, decltype(res)::value, 1, PAIRS_ANY>(p, c, dev, stream);
        });
    if (c.r == 7)
        return with_residual([&](auto res) {
            return c.pairs == PAIRS_SPLIT ? launch<7, 2, 2, decltype(res)::value, 1, PAIRS_SPLIT>(p, c, dev, stream) : launch<7, 2, 2, decltype(res)::value, 1, PAIRS_EVEN>(p, c, dev, stream);
        });
    return launch<11, 3, 1, RES_NONE, 2, PAIRS_SPLIT>(p, c, dev, stream);
}

}  // namespace tcbnn
