// First layer (fp32 3-channel NCHW input, +-1 filters; InConv128LayerFMT, kernel.cuh:578-672) on the matrix cores for 11-row
// filters with 2x2 pooling where there are few rows, or 32 channels: a ring of split rows in LDS.  Results, the split of the inputs
// and the recomputation of values in doubt are those of inconv_mfma.hip (the reference's bits, for every input), whose kernel walks
// down rows that it loads into registers.  At 11x11 that kernel lays out 54 KB of weights per workgroup before its first row, and a
// pooled row of a wave takes four dependent steps of 216 products; here the four waves of a workgroup share a window that they
// stage once, and a wave holds its weights in registers.  AlexNet's layer, launched on end, batch 8 / 16 / 26 / 32 / 40 / 80, us: here
// 16.9 / 21.0 / 31.1 / 31.3 / 39.3 / 60.7, there 30.5 / 31.6 / 32.7 / 33.2 / 34 / 47.5.  (There with 32 channels to a wave, or
// with the sets of a row multiplied by waves side by side: 23 and 35 at batch 8.)
//
// The bound E.  u = 2^-24, A = sum of |x| under the window, T = R*S taps.  A rounding of a running sum is at most u times
// that sum, which is at most what has been added so far and at most |S| plus what is still to come: (A + |S|) / 2.  The
// ordered sum has T such roundings and 2 u A more inside its taps; the split drops at most 2 u |x| per input (and 2^-25
// where fp16 runs out of exponents).  An MFMA adds its 16 products in two halves of eight (six, without the fourth channel).
// A half rounds its result once, and what lies below u times its largest product M is lost, of each product and of the sum
// that they are added to (tests/test_gpu_matrix_core.py holds the instruction to this).  An fp16 number has 11 bits, so
// only products below 2^-13 M lose anything: m of them and the sum, (m + 1) u M at most, where the sum is below M.
// The lo steps run first, on sums below 2^-10 A.  For A stands sqrt(3 T sum of hi^2), whose squares are one v_dot2 per
// loaded dword and which such small values hardly enter: by Cauchy and Schwarz the losses of all halves add the most to
// the rest of the bound where m = 0, and then 2 R NQ / (3 T) < 0.25 u A; 2.25 roundings are taken per step, not 2.  E is
// taken for |S| <= A/2 (partial sums below 3/4 A); a lane with a larger sum looks again with the full bound.  -E itself
// enters the sum as one more product (the fourth channel of the last tap, unused otherwise), so the accumulators hold
// S - E: a bit is certainly 1 where S - E >= bn, certainly 0 below bn - 2E.  Inputs outside the fp16 range, infinities and
// NaN make E infinite: all values of such a window are recomputed.  While every row that a workgroup has staged is multiples of
// 1/256 below 2^15 (23 bits, which the halves hold), windows with a sum of |x| below 2^16 are exact, and E is 0.  (Bytes, batch 8 /
// 32: 13.5 / 27.1 us; with sums below 2^15 16.6 / 31.3.)
// A wave's list of values in doubt that fills up ends the common pass for the workgroup, before the next row: the rest of
// the band is summed in the reference's order, as fp32 products on the matrix cores (ordered_sums).
//
// Work split.  A workgroup owns NI images x a strip of xo convolution columns x a band of output rows, and walks down the rows:
// the input rows of the window stay in LDS (a ring; every input row is read and split once per strip), as fp16
// [row][image][column][4] for hi and the same for lo, image pitch an odd number of 16-byte units (conflict-free).  A
// multiplication is 32 columns = NI images x 32/NI neighbouring pixels (so small batches fill their tiles) by 32 channels.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

#include "inconv.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

constexpr int kThreads = 256;
constexpr int kRounds = 5;  // staging units (column pairs) per thread and step, at most
constexpr int kR = 11, kNQ = 3, kPool = 2;  // filter rows, fragments to a filter row, pooling window
constexpr int kListCap = 64;   // doubtful values a wave keeps
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// A staged image row lies in LDS as column pairs of 16 bytes, even pairs first, then odd ones.  A multiplication's 64 lanes read
// 16 bytes each, half h of them pair 2j + h of their pixel's window: strides are multiples of four, so neighbouring pixels are
// neighbouring units (with an image pitch of 2 modulo 4 units the lanes fall into different banks).

constexpr int kWorkgroupsPerCu = 2;  // one wave of each per SIMD: what the registers allow

struct Geometry {
    int ni_log2;             // images per tile
    int xo;                  // convolution columns per strip
    int np, pp;              // staged column pairs per image row, and their pitch
    int odd_pairs;           // where the odd pairs begin
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
    float exact_squares;     // ... below which sums of multiples of 1/256 are exact
};

// The kernel's argument.  Code that seldom runs reads it anew from the argument segment (seldom_args): fields that
// only such code needs are then not kept in scalar registers, and spilled, all the way through the common one.  (The
// segment's address is a register of the kernel itself: taken in a function that is not inlined it would be 0.)
struct KernelArgs {
    InConvParams p;
    Geometry q;
    const uint32_t* pats;
    unsigned out_bytes;
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

__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kWorkgroupsPerCu))) void inconv_mfma_ring_kernel(
    const KernelArgs args) {
    const SeldomArgs args_at = (SeldomArgs)__builtin_amdgcn_kernarg_segment_ptr();
    const InConvParams& p = args.p;
    const Geometry& q = args.q;
    constexpr int R = kR, NQ = kNQ, POOL = kPool;
    constexpr int NK = R * NQ;  // MFMA steps: four taps (of one filter row) x four channels each
    constexpr unsigned kOutOfRange = 0x80000000u;
    extern __shared__ __align__(16) char lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slot_x = (int)blockIdx.x >> 3;
    int work = ((int)blockIdx.x & 7) * q.per_xcd + slot_x;
    if (slot_x >= q.per_xcd || work >= q.total) return;  // whole workgroup
    const int strip = work % q.strips;
    work /= q.strips;
    const int band = work % q.bands;
    work /= q.bands;
    const int cg = work % q.cgroups, it = work / q.cgroups;
    const int NI = 1 << q.ni_log2, NX = 32 >> q.ni_log2;
    const int b0 = it << q.ni_log2;
    const int x0 = strip * q.xo;
    const int oy_begin = band * q.band_rows, oy_end = min(q.rows, oy_begin + q.band_rows);
    const int wc = wave % q.waves_c, wg0 = wave / q.waves_c, wg_step = 4 / q.waves_c;
    const int tile = cg * q.waves_c + wc;  // this wave's channel tile
    const int xcols = POOL * p.OW;
    const int n_groups = (min(q.xo, xcols - x0) + NX - 1) >> (5 - q.ni_log2);

    // LDS: thresholds of all channels, lists, flags, then the ring: hi rows, lo rows
    const int row_bytes = (q.pp * 16) << q.ni_log2;
    const int plane = q.ring * row_bytes;
    float* const thr = reinterpret_cast<float*>(lds);
    uint32_t* const list = reinterpret_cast<uint32_t*>(lds) + p.O + wave * 2 * kListCap;
    int* const flags = reinterpret_cast<int*>(lds) + p.O + 4 * 2 * kListCap;  // rows off the grid; many doubts
    char* const rows = lds + (p.O + 4 * 2 * kListCap + 4) * 4;

    // ---- thresholds (NaN: -infinity, the bit is 1 either way)
    for (int i = tid; i < p.O; i += kThreads) {
        const float t = p.bn[i];
        thr[i] = t != t ? -INFINITY : t;
    }
    if (tid < 2) flags[tid] = 0;
    __syncthreads();

    // ---- +-1 fragments: lane (row n, half h) holds taps 4j + 2h, 4j + 2h + 1 of channel row_to_channel(n), 4 channels each
    v4i wf[NK];
    {
    const int n = lane & 31, h = lane >> 5;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
            const int o = tile * 32 + mfma::row_to_channel(n);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int s = 4 * (k % NQ) + 2 * h + t;
                const uint32_t pt = args.pats[(size_t)((k / NQ) * p.S + min(s, p.S - 1)) * p.opad + o];
                uint32_t d0 = 0x3c003c00u | ((pt & 4u) << 13) | (pt << 30 & 0x80000000u), d1 = 0x3c00u | ((pt & 1u) << 15);
                if (s >= p.S) d0 = d1 = 0u;
                if (k == NK - 1 && t == 0) d1 |= h == 0 ? 0x3c000000u : 0u;  // the slot that -E enters through
                wf[k][2 * t] = (int)d0;
                wf[k][2 * t + 1] = (int)d1;
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
        const int e = (wave + 4 * k) * 64 + lane, e2 = e / q.np, pr = e - e2 * q.np, im = e2 & (NI - 1), row = e2 >> q.ni_log2;
        const int ax = ax_first + 2 * pr;
        const bool used = row < q.adv && b0 + im < p.B;
        voff[k] = used ? (unsigned)im * 3u * plane_b + (unsigned)((row * p.W + ax) * 4) : kOutOfRange;
        cell[k] = (unsigned)(im * q.pp + (pr >> 1) + (pr & 1) * q.odd_pairs) | (used && ax >= 0 && ax < p.W ? 1u << 16 : 0u) |
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
    bool grid = true;  // every row staged so far is multiples of 1/256 below 2^15 (rows are checked as long as that holds)
    auto split_and_store = [&](int n_rows, int slot0) __attribute__((always_inline)) {
        bool on_grid = true;
        float most = 0.0f;
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
#pragma unroll
                for (int t = 0; t < 6; ++t) most = __builtin_fmaxf(most, __builtin_fabsf(f[t]));
            }
        }
        if (grid) {
            if (__ballot(!on_grid | !(most < 32768.0f)) != 0 && lane == 0) flags[0] = 1;
        }
    };

    // ---- doubtful values: recomputed in the reference's order, 16 lanes per value (lane t of a row: tap 16 c + t), the
    // list's last four at a time.  Inputs and signs are one trip to memory.
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
            // (the row's 16 lanes all hold the sum)
            if (active && t16 == 0 && !(acc < thr[o]))
                __hip_atomic_fetch_or(p.out + ((pix * (unsigned)p.ow + (unsigned)(o >> 5)) * (unsigned)p.B + (unsigned)bb), 0x80000000u >> (o & 31), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        }
    };

    // ---- the window
    int ay0 = oy_begin * POOL * p.stride_h - p.pad_h;  // first input row of the step's window
    int s0 = 0;                                        // its ring slot
    for (int done = 0; done < q.ring; done += q.adv) {
        const int n = min(q.adv, q.ring - done);
        fetch(ay0 + done, n);
        split_and_store(n, done);
    }

    const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)args.out_bytes, 0x00020000);
    // Where this lane stores its output word, relative to the item (uniform); beyond the tensor for an image past the batch
    const unsigned uB = (unsigned)p.B;
    unsigned place_word;
    {
        const unsigned px = (unsigned)((lane & 31) >> q.ni_log2), h = (unsigned)lane >> 5, b = (unsigned)(b0 + (lane & (NI - 1)));
        place_word = b < uB && h == 0u && (px & 1u) == 0u ? (px / POOL * (unsigned)p.ow * uB + b) * 4u : kOutOfRange;
    }

    // ---- a whole item in the reference's order: words; in doubt stay sums that are no numbers.
    // A tap's eight possible values are four and their negatives, so adding one of them to 32 x 32 sums is a product with a
    // matrix of one +-1 and three 0 per row: two v_mfma_f32_32x32x2_f32, each one fp32 addition per sum (adding the zeros
    // changes nothing; tests/test_gpu_matrix_core.py).
    auto ordered_sums = [&](int oy, int g, uint32_t& word, uint32_t& doubt) __attribute__((always_inline)) {
        const SeldomArgs a = seldom_args(args_at);
        const auto& p = a->p;
        const uint32_t* const pats = a->pats;
        int ln = lane;
        asm volatile("" : "+v"(ln));  // (nothing derived from it is kept outside)
        const int h = ln >> 5, img = ln & (NI - 1), xc = x0 + g * NX + ((ln & 31) >> a->q.ni_log2);
        const bool valid = b0 + img < p.B && xc < xcols;
        const int ax0 = xc * p.stride_w - p.pad_w, o0 = tile * 32 + mfma::row_to_channel(ln & 31);
        const unsigned im = (unsigned)img * 3u * plane_b, flip = (unsigned)h << 31;
        doubt = word = 0u;
#pragma unroll 1
        for (int py = 0; py < POOL; ++py) {
            const int ay0 = (oy * POOL + py) * p.stride_h - p.pad_h, r_end = min(R, p.H - ay0);
            v16f acc;
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
            // a filter row at a time, requested one row ahead; out of the frame: zeros, which add nothing
            constexpr int kTaps = 4 * NQ;
            float next[kTaps][3];
            uint32_t next_pt[kTaps];
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
                    next_pt[t] = row[(unsigned)(min(t, p.S - 1) * p.opad + o0)];
            };
            const int r_begin = max(0, -ay0);
            if (r_begin < r_end) request(r_begin);
#pragma unroll 1
            for (int r = r_begin; r < r_end; ++r) {
                float f[kTaps][3];
                uint32_t pt[kTaps];
#pragma unroll
                for (int t = 0; t < kTaps; ++t) {
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch) f[t][ch] = next[t][ch];
                    pt[t] = next_pt[t];
                }
                if (r + 1 < r_end) request(r + 1);
#pragma unroll
                for (int t = 0; t < kTaps; ++t) {
                    if (t >= p.S) break;  // uniform
                    const float f2 = __uint_as_float(__float_as_uint(f[t][2]) ^ flip);
                    const float same = (f[t][0] + f[t][1]) + f2, other = (f[t][0] - f[t][1]) + f2;
                    {
                        // pattern 4 neg0 + 2 neg1 + neg2; a pattern from 4 on is the negative of the inverted one
                        const uint32_t neg = (uint32_t)((int)(pt[t] << 29) >> 31), c = (pt[t] ^ neg) & 3u;
                        const uint32_t one = 0x3f800000u | (neg & 0x80000000u);
                        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(c == (uint32_t)h ? one : 0u), same, acc, 0, 0, 0);
                        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(c == (uint32_t)h + 2u ? one : 0u), other, acc, 0, 0, 0);
                    }
                }
            }
            {
                const v4f* const tp = reinterpret_cast<const v4f*>(thr + tile * 32 + 16 * h);
                uint32_t w = 0u;
                float zero = 0.0f;  // an infinity or NaN among a tap's values makes NaN of it, times 0, in every sum
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    w = __builtin_amdgcn_alignbit(w, __float_as_uint(acc[i] - tp[i >> 2][i & 3]), 31);
                    zero = __builtin_fmaf(acc[i], 0.0f, zero);
                }
                const bool bad = !(zero == 0.0f);
                word |= bad ? 0u : ~w & 0xffffu;
                doubt |= (bad && valid ? 0xffffu : 0u) << (16 * py);
            }
        }
    };

    // ---- the band's items: sums with a bound, and from the row on after which a list was full, in the reference's order
    int oy = oy_begin, g = wg0;
    bool many = false;
    auto pass = [&](auto ordered) __attribute__((always_inline)) {
        constexpr bool kOrdered = decltype(ordered)::value;
        for (; oy < oy_end; ++oy) {
            const bool more = oy + 1 < oy_end;  // uniform
            if constexpr (!kOrdered) {
                __syncthreads();
                if (grid) grid = __builtin_amdgcn_readfirstlane(flags[0]) == 0;
                if (__builtin_amdgcn_readfirstlane(flags[1]) != 0) return;  // (written between the two barriers only)
            }
            if (!kOrdered && more) fetch(ay0 + q.ring, q.adv);
            while (g < n_groups) {
                uint32_t word = 0u, doubt = 0u;
                // A lane's place (column of the tile: image and pixel; half of the channels) is worked out anew from a lane
                // index the compiler cannot carry over: kept across the multiplication, the addresses made from it spill.
                int ln = lane;
                asm volatile("" : "+v"(ln));
                if constexpr (!kOrdered) {
#pragma unroll 1
                    for (int py = 0; py < POOL; ++py) {
                        v16f acc;
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
                        const int first_col = (g * NX + ((ln & 31) >> q.ni_log2)) * p.stride_w;
                        const int lane_at = (ln & (NI - 1)) * q.pp * 16 + (first_col >> 2) * 16 + (ln >> 5) * q.odd_pairs * 16;
                        auto fragment = [&](int r, int j, int plane_off) -> v4i {
                            int slot = s0 + py * p.stride_h + r;
                            slot = slot >= q.ring ? slot - q.ring : slot;
                            const char* const at = rows + (slot * row_bytes + plane_off) + lane_at + j * 16;
                            return __builtin_bit_cast(v4i, *reinterpret_cast<const h8*>(at));
                        };
                        // lo steps, then hi steps; a step's fragment is requested kAhead steps ahead
                        constexpr int kAhead = 4;
                        v4i ahead[kAhead];
#pragma unroll
                        for (int k = 0; k < kAhead; ++k) ahead[k] = fragment(k % NK / NQ, k % NK % NQ, k < NK ? plane : 0);
                        float sq = 0.0f, two_e = 0.0f, half_a = 0.0f, wide_shift = 0.0f, wide_two_e = 0.0f;
                        bool bad = false;
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
                            if (k == 2 * NK - 1) {
                                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(sq), __float_as_uint(sq), false, false);
                                const float all = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
                                const float root = __builtin_amdgcn_sqrtf(all), full = root * q.bound_scale_full + q.bound_add;
                                bad = !(all < 4.0e9f) || !(full < 3.0e4f);
                                _Float16 eh = (_Float16)(root * q.bound_scale + q.bound_add);
                                half_a = root * q.half_scale;
                                wide_two_e = 2.002f * full;
                                if (grid & (all < q.exact_squares)) {
                                    eh = (_Float16)0.0f;
                                    half_a = INFINITY;
                                }
                                two_e = 2.002f * (float)eh;
                                wide_shift = (float)eh - full;
                                if (lane < 32) v[1] |= (int)((uint32_t)(__builtin_bit_cast(uint16_t, eh) | 0x8000u) << 16);
                            }
                            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, wf[k % NK]), __builtin_bit_cast(h8, v), acc, 0, 0, 0);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        // ---- bits (MSB first; the sign of S - E - bn, inverted), residual, doubtful values
                        asm volatile("" : "+v"(ln));
                        const int h = ln >> 5;
                        const bool valid = b0 + (ln & (NI - 1)) < p.B && x0 + g * NX + ((ln & 31) >> q.ni_log2) < xcols;
                        {
                            const v4f* const tp = reinterpret_cast<const v4f*>(thr + tile * 32 + 16 * h);
                            // Signs are collected MSB first (bit 15 - i: channel i).  w: S - E < bn, dm: values in doubt.  Thresholds
                            // within E and sums above A/2 (E is less than a bound for those) are rare: the tile's nearest distance
                            // below a threshold and its largest |S| tell whether to look for them.
                            uint32_t w = 0u, dm = 0u;
                            int nearest = INT32_MAX;
                            float most = 0.0f;
                            {
                                const v4f th[4] = {tp[0], tp[1], tp[2], tp[3]};
#pragma unroll
                                for (int i = 0; i < 16; ++i) {
                                    const float d = acc[i] - th[i >> 2][i & 3];
                                    w = __builtin_amdgcn_alignbit(w, __float_as_uint(d), 31);
                                    nearest = min(nearest, __float_as_int(d));
                                    most = __builtin_fmaxf(most, __builtin_fabsf(acc[i]));
                                }
                            }
                            // (NaN: `bad` is set)
                            if (__ballot(bad | !(most <= half_a) | (nearest <= (int)(0x80000000u | __float_as_uint(two_e)))) != 0) {
                                const bool wide = !(most <= half_a);  // this lane's sums with the full bound
                                const float shift = wide ? wide_shift : 0.0f, two = wide ? wide_two_e : two_e;
                                uint32_t w2 = 0u;
                                w = 0u;
#pragma unroll
                                for (int i = 0; i < 16; ++i) {
                                    float a = acc[i];
                                    asm volatile("" : "+v"(a));  // (evaluated again here: not kept from above)
                                    a += shift;
                                    const float d = a - tp[i >> 2][i & 3];
                                    w = __builtin_amdgcn_alignbit(w, __float_as_uint(d), 31);
                                    w2 = __builtin_amdgcn_alignbit(w2, __float_as_uint(d + two), 31);
                                }
                                w = bad ? 0xffffu : w;
                                dm = bad ? 0xffffu : w & ~w2;
                            }
                            doubt |= (valid ? dm & 0xffffu : 0u) << (16 * py);
                            word |= ~w & 0xffffu;  // (a bit in doubt is 0 here: the recomputation only ever sets it)
                        }
                    }
                }
                if constexpr (kOrdered) ordered_sums(oy, g, word, doubt);
                // ---- output words: half 0 stores
                asm volatile("" : "+v"(ln));
                const int h = ln >> 5, img = ln & (NI - 1), xc = x0 + g * NX + ((ln & 31) >> q.ni_log2);
                const auto sw = __builtin_amdgcn_permlane32_swap(word, word, false, false);
                uint32_t full = (sw[0] << 16) | sw[1];
                full |= (uint32_t)__shfl_xor((int)full, NI);  // the window's other column
                const unsigned item_word = ((unsigned)(oy * p.OW + (x0 + g * NX) / POOL) * (unsigned)p.ow + (unsigned)tile) * uB * 4u;
                __builtin_amdgcn_raw_buffer_store_b32(full, out_rsrc, (int)(xc < xcols ? place_word + item_word : kOutOfRange), 0, 0);
                // ---- doubtful values of this item go on the list, one per lane at a time.  Recomputed are those of earlier
                // items (their stores are older than this item's, so nothing of this item is waited for), four at a time, and
                // all that are there where the list is full and after the wave's last item.
                const bool last = !more && g + wg_step >= n_groups;
                if (count >= 4) {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(1) : "memory");
                    recompute();
                }
                unsigned long long who = __ballot(doubt != 0u);
                for (;;) {
                    int c;
                    while ((c = __builtin_amdgcn_readfirstlane(__popcll(who))) != 0 && count + c <= kListCap) {
                        if (doubt != 0u) {
                            const int bit = __ffs(doubt) - 1;
                            doubt &= doubt - 1u;
                            const int at = count + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(who >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who, 0u));
                            const int py = bit >> 4;
                            list[2 * at] = (uint32_t)(oy * POOL + py) << 16 | (uint32_t)xc;
                            list[2 * at + 1] = (uint32_t)(tile * 32 + 16 * h + 15 - (bit & 15)) | (uint32_t)img << 16;
                        }
                        count += c;
                        who = __ballot(doubt != 0u);
                    }
                    if (c == 0 && (!last || count == 0)) break;
                    if (c != 0) many = true;  // the list is full
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    do recompute();
                    while (count > kListCap / 2);
                }
                g += wg_step;
            }
            g = wg0;
            if constexpr (!kOrdered) {
                __syncthreads();
                if (many && lane == 0) flags[1] = 1;
            }
            if (!kOrdered && more) split_and_store(q.adv, s0);
            ay0 += q.adv;
            s0 += q.adv;
            s0 = s0 >= q.ring ? s0 - q.ring : s0;
        }
    };
    pass(std::false_type{});
    if (oy < oy_end) pass(std::true_type{});
}

// ---------------------------------------------------------------- host side
constexpr int kLdsPerCu = 160 * 1024;

struct Choice {
    Geometry q;
    size_t lds_bytes;
    int grid;
    long long out_bytes;
};

size_t lds_extra(int channels) { return (size_t)(channels + 4 * 2 * kListCap + 4) * 4; }

// What the kernel serves: pooled 11-row filters of 9 to 12 taps a row.
bool serves(const InConvParams& p) {
    return p.R == kR && (p.S + 3) / 4 == kNQ && p.pool_h == kPool && p.pool_w == kPool && p.O % 32 == 0 && p.stride_w % 4 == 0 && p.res == nullptr;
}

// How a launch is split; false for sizes that the kernel does not take.  `cus`: compute units.
bool choose(const InConvParams& p, int cus, Choice* out) {
    Choice c{};
    if (!serves(p)) return false;
    Geometry& q = c.q;
    q.adv = kPool * p.stride_h;
    q.ring = p.R + (kPool - 1) * p.stride_h;
    if (q.adv > q.ring) return false;
    if (p.PH > 32767 || p.PW > 32767 || p.O > 65535) return false;
    // (32-bit buffer offsets)
    c.out_bytes = 4LL * p.OH * p.OW * p.ow * p.B;
    if (c.out_bytes >= (1LL << 31)) return false;
    q.rows = p.OH;
    q.rs_taps = p.R * p.S;
    const int chp = p.O / 32;
    q.waves_c = chp % 4 == 0 ? 4 : (chp % 2 == 0 ? 2 : 1);
    q.cgroups = chp / q.waves_c;
    const size_t extra = lds_extra(p.O), share = (size_t)kLdsPerCu / kWorkgroupsPerCu;
    if (extra >= share) return false;
    const size_t lds_limit = share - extra;
    q.s_magic = 65536u / (unsigned)p.S + 1u;
    for (int t = 0; t < q.rs_taps; ++t)
        if ((int)((unsigned)t * q.s_magic >> 16) != t / p.S) return false;

    // Images per 32-column tile and columns per strip: the cheapest over the batch and the width, in rough cycles of a
    // wave: items (multiplication and epilogue) and staging rounds.  At most eight images.
    const int xcols = kPool * p.OW;
    const int item = 3200 * kPool;
    double best = 1e30;
    int most_images = 3;
    while (most_images > 0 && (1 << (most_images - 1)) >= p.B) --most_images;
    for (int ni_log2 = most_images; ni_log2 >= std::max(0, most_images - 2); --ni_log2) {
        const int NI = 1 << ni_log2, NX = 32 >> ni_log2, step = std::max(NX, kPool), imgtiles = (p.B + NI - 1) >> ni_log2;
        if ((long long)NI * 3 * p.H * p.W * 4 >= (1LL << 31)) continue;
        for (int xo = step; xo < xcols + step; xo += step) {
            const int np = ((xo - 1) * p.stride_w + 4 * kNQ + 1) / 2, odd = (np + 1) / 2;
            const int pp = 2 * odd + (odd % 2 == 0 ? 2 : 0);
            const int units = (np * NI * q.adv + kThreads - 1) / kThreads;
            const size_t bytes = (size_t)2 * q.ring * NI * pp * 16;
            if (units > kRounds || bytes > lds_limit || NI * pp > 0xffff) break;
            const int groups = xo / NX, strips = (xcols + xo - 1) / xo;
            const int rounds = (groups * q.waves_c + 3) / 4;
            const double cost = (double)imgtiles * strips * (rounds * (double)item + 200.0 * units + 500.0);
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
    c.lds_bytes = (size_t)2 * q.ring * ((size_t)q.pp << q.ni_log2) * 16 + extra;

    // Bands of rows: one round of resident workgroups where the width and the batch leave a choice; a band's first
    // window is staged whole (counted as 0.7 of a row's work).
    const long long per = (long long)q.imgtiles * q.cgroups * q.strips, target = (long long)cus * kWorkgroupsPerCu;
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
    q.per_xcd = (q.total + 7) / 8;
    c.grid = 8 * q.per_xcd;
    // E (see the top of this file): the roundings of sums, T of the reference's and 2 per hi step and for -E (2.25 taken:
    // what the halves lose) with partial sums below (A + |S|) / 2 <= 0.75 A (or A); 2 u A for the additions in a tap, 2 u A for the split, and
    // 0.5 u A for the lo steps.  2 % cover the roundings of the bound itself.
    const double T = q.rs_taps, u = std::ldexp(1.0, -24), sums = T + 2.25 * (kR * kNQ + 1), a_scale = std::sqrt(3.0 * T);
    q.bound_scale = (float)((0.75 * sums + 4.5) * u * 1.02 * a_scale);
    q.bound_scale_full = (float)((sums + 4.5) * u * 1.02 * a_scale);
    q.half_scale = (float)(0.49 * a_scale);
    q.bound_add = (float)(3.0 * T * std::ldexp(1.0, -24) + std::ldexp(1.0, -22));
    q.exact_squares = (float)(65000.0 * 65000.0 / (3.0 * T));  // (sum of |x| below 2^16)
    *out = c;
    return true;
}

}  // namespace

bool inconv_mfma_ring_serves(const InConvParams& p) {
    Choice c;
    return choose(p, 256, &c);
}

int launch_inconv_mfma_ring(const InConvParams& p, int dev, int cus, hipStream_t stream, bool* served) {
    Choice c{};
    *served = choose(p, cus, &c);
    if (!*served) return TCBNN_OK;
    static std::atomic<bool> ready[kInConvDevices];  // (setting the limit twice does no harm)
    if (!ready[dev].load(std::memory_order_acquire)) {
        const void* fn = reinterpret_cast<const void*>(&inconv_mfma_ring_kernel);
        if (int rc = check_hip(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsPerCu / kWorkgroupsPerCu),
                               "hipFuncSetAttribute(MaxDynamicSharedMemorySize)"))
            return rc;
        ready[dev].store(true, std::memory_order_release);
    }
    const uint32_t* pats = reinterpret_cast<const uint32_t*>(p.masks) + (size_t)p.R * p.S * p.opad * 4;
    hipLaunchKernelGGL(inconv_mfma_ring_kernel, dim3((unsigned)c.grid), dim3(kThreads), c.lds_bytes, stream,
                       KernelArgs{p, c.q, pats, (unsigned)c.out_bytes});
    TCBNN_LAUNCH_CHECK("inconv_mfma_ring_kernel");
    return TCBNN_OK;
}

}  // namespace tcbnn
