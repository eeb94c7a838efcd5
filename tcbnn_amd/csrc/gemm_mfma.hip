// FP4 matrix-core kernel for LARGE bit-GEMMs: the stand-alone bit matrix product (BMMAS_new,
// tensorcore_kernel.cu:336-356: C = K - 2 popc(A xor B)) and fully connected layers at large batch
// (Fc128LayerFMT / Out128LayerFMT, kernel.cuh:174-280; e.g. the 1024 -> 1024 layers of the MLP at batch
// 8192).  The generic implicit-GEMM kernel serves the same problems, but pays for its generality in every k-step (tap
// bookkeeping, frame and range tests, weights expanded with masks behind two barriers per block).
//
//   workgroup = 4 waves = (4 x MT x 32 rows of the batch / of A) x 64 output columns;
//   wave      = MT image tiles x 2 column tiles: 2 MT MFMAs (32 x 32 x 64, FP4) per k-step;
//   weights   : the 64 columns' words are expanded to MFMA "A" fragments in LDS, 8 or 16 k-steps at a time,
//               double-buffered: the words of the next block, 16 bytes a thread with four threads to a row, are
//               requested before the current block is multiplied and expanded into the other buffer after it, one
//               barrier per block;
//   rows      : a lane's words, of MT neighbouring images in one request, come straight from memory through buffer
//               addressing (a per-lane constant offset, the k-step in the scalar offset), eight k-steps ahead of their use.
// Bound by the matrix pipe and by power: with operands like these the MFMA alone reaches 8.1 P (constants: 9.8), this kernel 5.8
// on 8 192^3, of whose time a tenth is the output's.  Before (a row of the weights per lane, a request per image tile, one block
// size): 8 192^3 223 us, 5 000 x 3 104 x 7 200 59, 3 072 x 3 072 x 8 192 53, 1 500 x 8 192 x 4 096 31.4; now 189, 47.4, 37.4, 24.0.
// Operand roles, fragment order and the accumulator layout are those of bgemm_mfma.hip.
#include "common.h"
#include "mfma_util.h"

namespace tcbnn {
namespace {

using namespace mfma;

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kNT = 2;     // 32-column tiles per wave
// k-steps of weights per LDS buffer (kNT KiB each): with two image tiles per wave the registers hold three workgroups in a CU, and
// so does the LDS
constexpr int blk_of(int mt) { return mt == 2 ? 8 : 16; }
constexpr int kAhead = 8;  // k-steps a row word is requested ahead of its use; divides blk_of()
constexpr int kOutOfRange = (int)0x80000000u;  // (a request there touches no memory and returns 0)
static_assert(kThreads == 4 * 32 * kNT, "four threads stage a column");
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v4f_word __attribute__((ext_vector_type(4), aligned(4)));  // sixteen bytes at any word

// Row words are expanded without shifts (expand_rows_f4 in mfma_util.h): the accumulator ends as the dot product
// plus a per-column constant, which the staging lanes count as they go and the epilogue takes off.
// TAIL: rows that are no whole 128-bit units (the stand-alone product alone has them): the last unit's words past the row
// are the next row's.
template <int MT, int EPI, bool TAIL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(MT == 2 ? 3 : 2))) void gemm_mfma_f4_kernel(
    const BgemmParams p, const uint32_t* __restrict__ act, const uint32_t* __restrict__ wgt,
    const float* __restrict__ bnp, const float* __restrict__ bias, int n_groups) {
    constexpr int kBlk = blk_of(MT);
    constexpr int kUnits = kBlk / 8;  // 16-byte units of a column's row that a thread stages per block: two k-steps each, four threads
    constexpr int kRawInts = kNT * 32 + kWaves * 32 * (32 * kNT + 4);  // int32 output on its way (below)
    __shared__ v4i lds_all[(2 * kBlk * kNT * 64 * 4 > kRawInts || EPI != EPI_RAW ? 2 * kBlk * kNT * 64 * 4 : kRawInts) / 4];
    v4i(*const lds_w)[kBlk * kNT * 64] = reinterpret_cast<v4i(*)[kBlk * kNT * 64]>(lds_all);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int j = lane & 31;  // image within a 32-image tile
    const int h = lane >> 5;  // k half (operands) / column half (accumulator)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ng = blockIdx.x % n_groups, rb = blockIdx.x / n_groups;
    const int n0 = ng * (32 * kNT);
    const int b0 = (rb * kWaves + wave) * (32 * MT);
    // 64-bit k-steps, run in whole groups of kAhead.  Nothing is masked: a pad bit is 0 in both operands (the layouts'
    // convention), and so is every bit of a word past K: the upper half of the last step of an odd cw, and the steps
    // that fill up the group (rows: outside the descriptor's range; weights: staged as 0).  A 0 bit expands to +1.0 on
    // both sides, so each such position adds exactly +1 to the dot product, and the known count is taken off in the
    // epilogue.
    const int steps = (p.cw + 2 * kAhead - 1) / (2 * kAhead) * kAhead;
    const int corr = 64 * steps - p.k_tap + 2 * steps * class_sum(0u);  // (with what a column of zeros adds, see set0)

    // ---- weights: this thread stages 16-byte units sc and sc + 4 (two k-steps each) of one of the 64 columns' rows.  Fragments
    // lie in LDS with the low bits of their lane exchanged by the unit, so eight neighbouring threads (two columns, four
    // units) write to different banks; a reading wave covers whole runs of 64 slots either way.
    const int sj = tid >> 2 & 31, snt = tid >> 7, sc = tid & 3;
    // a row past N (stand-alone product: the rows do not exist) reads the last row; its results are discarded
    const int srow = min(n0 + snt * 32 + row_to_channel(sj), p.N - 1) - n0;
    const __amdgpu_buffer_rsrc_t r_wgt = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(wgt + (size_t)n0 * p.cw), 0, min(32 * kNT, p.N - n0) * p.cw * 4, 0x00020000);
    const int woff = (srow * p.cw + 4 * sc) * 4;
    v4i wx[kUnits];
    auto stage_load = [&](int q0) {
#pragma unroll
        for (int i = 0; i < kUnits; ++i) {
            const int w = 2 * q0 + 16 * i + 4 * sc;  // the unit's first word
            wx[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r_wgt, w < p.cw ? woff + (2 * q0 + 16 * i) * 4 : kOutOfRange, 0, 0));
        }
    };
    // this thread's share of its column's constant C, counted by class (words past K are zeros and count nothing)
    int set0 = 0, set1 = 0, set2 = 0;
    auto stage_store = [&](int buf, int q0) {
#pragma unroll
        for (int i = 0; i < kUnits; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int ql = 8 * i + 2 * sc + (t >> 1);
                uint32_t word = (uint32_t)wx[i][t];
                if (TAIL && 2 * (q0 + ql) + (t & 1) >= p.cw) word = 0u;
                lds_w[buf][(ql * kNT + snt) * 64 + ((32 * (t & 1) + sj) ^ (sc << 1))] = expand_weights_f4(word);
                set0 += __popc(word & 0x11111111u);
                set1 += __popc(word & 0x22222222u);
                set2 += __popc(word & 0x44444444u);
            }
    };
    int rlane[4];  // where the lane's fragment of k-step q lies in its run of 64: rlane[q / 2 % 4]
#pragma unroll
    for (int c = 0; c < 4; ++c) rlane[c] = lane ^ (c << 1);

    // ---- rows: words [cw][B]; lane (j, h) reads word 2 q + h of its MT neighbouring images in one request.  Images past B:
    // the next word's, or 0 behind the tensor; their results are discarded.
    const int b_lane = b0 + MT * j;
    const int voff = (h * p.B + b_lane) * 4;
    const __amdgpu_buffer_rsrc_t r_act =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(act), 0, p.cw * p.B * 4, 0x00020000);
    const int step_bytes = 2 * p.B * 4;
    uint32_t ring[kAhead][MT];
    int lq = 0;  // next k-step to request
    // no test for the end of K: a request past it lies outside the descriptor's range, touches no memory and
    // returns 0 (such words are never multiplied), and the k-steps stay free of branches
    auto request = [&](uint32_t* dst) {
        static_assert(MT == 2 || MT == 4, "one request holds the lane's images");
        if constexpr (MT == 4) {
            const v4i v = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r_act, voff, lq * step_bytes, 0));
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) dst[mt] = (uint32_t)v[mt];
        } else {
            const v2i v = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(r_act, voff, lq * step_bytes, 0));
            dst[0] = (uint32_t)v[0];
            dst[1] = (uint32_t)v[1];
        }
        ++lq;
    };

    v16f acc[MT][kNT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[mt][nt][v] = 0.0f;

#pragma unroll
    for (int d = 0; d < kAhead; ++d) request(ring[d]);
    stage_load(0);
    __builtin_amdgcn_sched_barrier(0);  // (everything is requested before anything is waited for)
    stage_store(0, 0);
    __syncthreads();

    // Software pipeline, one k-step deep: while step q is multiplied, the weight fragments of step q + 1 are on
    // their way from LDS and its row words are expanded (their ring slot is then asked for step q + 9).  Step q's
    // words sit in ring slot q % kAhead; kBlk is a multiple of kAhead, so the slot of step ql + d of a block is d.
    v4i anext[kNT], bnext[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) bnext[mt] = expand_rows_f4(ring[0][mt]);
    request(ring[0]);

    auto run = [&](const v4i* __restrict__ wl, int ql) __attribute__((always_inline)) {  // kAhead steps of a block
#pragma unroll
        for (int d = 0; d < kAhead; ++d) {
            v4i acur[kNT], bcur[MT];
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt) acur[nt] = anext[nt];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) bcur[mt] = bnext[mt];
            const int qn = min(ql + d + 1, kBlk - 1);  // after a block's last step: read again, not used
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt) anext[nt] = wl[(qn * kNT + nt) * 64 + rlane[(d + 1) / 2 % 4]];
            const int dn = (d + 1) % kAhead;  // a constant once the loop over d is unrolled
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) bnext[mt] = expand_rows_f4(ring[dn][mt]);
            request(ring[dn]);
#pragma unroll
            for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[mt][nt] = Acc<FMT_F4>::mma(acur[nt], bcur[mt], acc[mt][nt]);
            // issue order of the step: fragment reads first, then each MFMA followed by a few of the next
            // step's expansion instructions (they run while the matrix pipeline is busy), the row requests
            // in the middle
            __builtin_amdgcn_sched_group_barrier(0x100, kNT, 0);  // LDS reads
#pragma unroll
            for (int i = 0; i < kNT * MT; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, (4 * MT + kNT * MT - 1) / (kNT * MT), 0);  // VALU
                if (i == kNT * MT / 2) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // row request
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto first_fragments = [&](const v4i* __restrict__ wl) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < kNT; ++nt) anext[nt] = wl[nt * 64 + rlane[0]];
    };
    // Whole blocks that another one follows, without a branch from the next weights' request to their staging: with one (a
    // request only where there are more, a loop over the block's steps) the compiler cannot count what is outstanding
    // and waits for every row request twice a block (8 192 x 448 x 8 192 23.1 us, so 19.1; 200 x 8 192 x 8 192 18.7 / 16.5;
    // 2 048 x 4 096 x 8 192 31.9 / 30.5; level where two workgroups in a CU cover for each other).
    int buf = 0, q0 = 0;
    for (; q0 + kBlk < steps; q0 += kBlk) {
        stage_load(q0 + kBlk);
        first_fragments(lds_w[buf]);
#pragma unroll
        for (int ql = 0; ql < kBlk; ql += kAhead) run(lds_w[buf], ql);
        // the other buffer was last read in the previous block, which every wave left before the barrier below
        stage_store(buf ^ 1, q0 + kBlk);
        __syncthreads();
        buf ^= 1;
    }
    first_fragments(lds_w[buf]);
    for (int ql = 0; ql < steps - q0; ql += kAhead) run(lds_w[buf], ql);
    __syncthreads();

    // ---- the columns' constants: four threads staged each column's words.  The weight
    // buffers are free now (every wave has passed the loop's last barrier).
    int* colc = reinterpret_cast<int*>(&lds_w[0][0]);  // [kNT * 32]
    if (tid < kNT * 32) colc[tid] = 0;
    __syncthreads();
    atomicAdd(&colc[snt * 32 + row_to_channel(sj)], 2 * (5 * set0 + 3 * set1 + set2));
    __syncthreads();

    // int32 output, all 64 columns of the group exist and every row's run of them is 16-byte aligned (uniform): the
    // sums leave through LDS, a row at a time (below)
    const bool raw_rows = EPI == EPI_RAW && n0 + 32 * kNT <= p.N && p.raw_b_stride % 4 == 0 &&
                          (reinterpret_cast<uintptr_t>(p.out_i32) & 15) == 0;

    // ---- epilogue: the lane holds columns cbase + v of image b_lane + mt
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
        const int cbase = n0 + nt * 32 + 16 * h;
        int off[16];  // what the accumulator holds beyond the dot product
#pragma unroll
        for (int v = 0; v < 16; ++v) off[v] = corr + colc[nt * 32 + 16 * h + v];
        float thr[16], bia[EPI == EPI_AFFINE ? 16 : 1];
        if constexpr (EPI != EPI_RAW) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                thr[v] = bnp[min(cbase + v, p.N - 1)];
                if constexpr (EPI == EPI_AFFINE) bia[v] = bias[min(cbase + v, p.N - 1)];
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int b = b_lane + mt;
            const bool b_ok = b < p.B;
            if constexpr (EPI == EPI_THRESH) {
                uint32_t hw = 0;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const uint32_t bit = cbase + v < p.N ? thresh_bit((int)acc[mt][nt][v] - off[v], thr[v], p.nan_bit) : 0u;
                    hw = hw + hw + bit;
                }
                const uint32_t other = (uint32_t)__shfl_xor((int)hw, 32);
                const int w = ng * kNT + nt;
                if (h == 0 && b_ok) {
                    if (w < p.bits_row_words) p.out_bits[(size_t)w * p.B + b] = (hw << 16) | other;
                    if (ng == n_groups - 1 && nt == kNT - 1)  // padding words of the 128-padded feature axis
                        for (int z = max((p.N + 31) / 32, n_groups * kNT); z < p.bits_row_words; ++z)
                            p.out_bits[(size_t)z * p.B + b] = 0;
                }
            } else if constexpr (EPI == EPI_AFFINE) {
                // Sixteen bytes a request: a lane's row is another one than its neighbour's, so every word asked for by itself is
                // a line of its own, and that is what such a layer takes its time for (us, a word at a time -> here: 14 792 x 528 of
                // 167 inputs 47.9 -> 17.3, 15 660 x 508 of 1 273 54.1 -> 25.0, 8 192 x 1 000 of 1 024 44.3 -> 16.8).
                if (b_ok) {
                    // the +-1 dot product equals (float)K - (float)popc*2.0f exactly (kernel.cuh:258-270)
                    auto y = [&](int v) { return __fadd_rn(__fmul_rn((float)((int)acc[mt][nt][v] - off[v]), thr[v]), bia[v]); };
                    float* const dst = p.out_f32 + (size_t)b * p.N + cbase;
                    if (cbase + 16 <= p.N) {
#pragma unroll
                        for (int v = 0; v < 16; v += 4) *reinterpret_cast<v4f_word*>(dst + v) = v4f_word{y(v), y(v + 1), y(v + 2), y(v + 3)};
                    } else {
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            if (cbase + v < p.N) dst[v] = y(v);
                    }
                }
            } else if (raw_rows) {
                // (int32 output of whole, aligned column groups: written further down, a row at a time)
            } else {
                if (b_ok) {
                    int32_t* dst = p.out_i32 + (size_t)b * p.raw_b_stride + cbase;
                    // a lane's 16 values are consecutive in memory: four 128-bit stores where the run is whole
                    // and aligned
                    if (cbase + 16 <= p.N && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
#pragma unroll
                        for (int g = 0; g < 4; ++g)
                            reinterpret_cast<int4*>(dst)[g] =
                                make_int4((int)acc[mt][nt][4 * g] - off[4 * g], (int)acc[mt][nt][4 * g + 1] - off[4 * g + 1],
                                          (int)acc[mt][nt][4 * g + 2] - off[4 * g + 2],
                                          (int)acc[mt][nt][4 * g + 3] - off[4 * g + 3]);
                    } else {
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            if (cbase + v < p.N) dst[v] = (int)acc[mt][nt][v] - off[v];
                    }
                }
            }
        }
    }

    // int32 output [rows][N] (BMMAS_new, tensorcore_kernel.cu:355): in the accumulator a lane holds 16 columns of ONE
    // row, so a direct store scatters 16-byte pieces over 64 different rows per instruction (the product writes
    // 4 M N bytes: a quarter of the 8192^3 launch was this).  The sums of a 32-row tile go through a per-wave LDS
    // area instead (row = image, pitch 68 words: conflict-free both ways; the weight buffers are free by now) and
    // leave as 128-bit stores in which 16 consecutive lanes cover one row's whole run of 64 columns (4 runs of
    // 256 bytes per instruction).
    if constexpr (EPI == EPI_RAW) {
        if (raw_rows) {
            constexpr int kPitch = 32 * kNT + 4;
            // (behind the column constants, which stay where they are)
            int* mine = reinterpret_cast<int*>(&lds_w[0][0]) + kNT * 32 + wave * (32 * kPitch);
            const int rl = lane >> 4, cl = lane & 15;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
                for (int nt = 0; nt < kNT; ++nt) {
                    int off[16];
#pragma unroll
                    for (int v = 0; v < 16; ++v) off[v] = corr + colc[nt * 32 + 16 * h + v];
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<v4i*>(mine + j * kPitch + nt * 32 + 16 * h + 4 * g) =
                            v4i{(int)acc[mt][nt][4 * g] - off[4 * g], (int)acc[mt][nt][4 * g + 1] - off[4 * g + 1],
                                (int)acc[mt][nt][4 * g + 2] - off[4 * g + 2], (int)acc[mt][nt][4 * g + 3] - off[4 * g + 3]};
                }
                // (same wave writes and reads: program order and the wait for LDS are all the synchronisation)
#pragma unroll
                for (int part = 0; part < 2; ++part) {
                    v4i q[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) q[k] = *reinterpret_cast<const v4i*>(mine + (16 * part + 4 * k + rl) * kPitch + 4 * cl);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int row = b0 + MT * (16 * part + 4 * k + rl) + mt;
                        if (row < p.B)
                            *reinterpret_cast<v4i*>(p.out_i32 + (size_t)row * p.raw_b_stride + n0 + 4 * cl) = q[k];
                    }
                }
            }
        }
    }
}

// Image tiles per wave: two, whose smaller workgroups leave less of a last round empty and of which a compute unit runs three
// (3 072 x 3 072 x 8 192 37.4 us against 44.3 with four, 8 000 x 2 080 x 6 016 48.0 / 54.6, 1 500 x 8 192 x 4 096 24.0 / 27.5); four, which multiply
// every weight fragment twice as often, where they come out even over the compute units, at two workgroups in each or more,
// and K is long (5 000 x 3 104 x 7 200 49.0 us with two, 47.3 with four; 8 192^3 200 / 184; 8 192 x 8 192 x 512 45.2 / 48.2).  Over 66
// products the pick is at most 2.4 % slower than the other number of tiles.
int gemm_mt(const BgemmParams& p) {
    constexpr int kCus = 256, kLongK = 64;  // (words)
    const long long n_groups = (p.N + 32 * kNT - 1) / (32 * kNT);
    auto a_cu = [&](int mt) {  // image tiles that the busiest compute unit's waves take
        return mt * ((((p.B + 32 * mt * kWaves - 1) / (32 * mt * kWaves)) * n_groups + kCus - 1) / kCus);
    };
    return p.cw >= kLongK && a_cu(4) >= 8 && a_cu(4) <= a_cu(2) ? 4 : 2;
}

}  // namespace

bool gemm_mfma_applicable(const BgemmParams& p) {
    if (p.PH * p.PW != 1 || p.R * p.S != 1 || p.pool_h * p.pool_w != 1) return false;
    // the rows are the frame's first pixel: with a padding the one output pixel lies elsewhere in the frame (a stride beyond
    // the frame makes it negative) or outside
    if (p.pad_h != 0 || p.pad_w != 0) return false;
    if (p.res_in != nullptr || p.res_out != nullptr) return false;
    if (p.mode != EPI_THRESH && p.mode != EPI_AFFINE && p.mode != EPI_RAW) return false;
    if (p.k_tap > 32 * p.cw || (p.cw % 4 != 0 && p.mode != EPI_RAW)) return false;
    // The sums hold up to 13/4 of a count for each position of K, words past it included (1, 2, 4 and 6 on the four classes of
    // expand_rows_f4), and fp32 is exact to 2^24: to K = 5.1 million.  A longer one goes to the kernels that multiply +-1.
    if (13LL * 64 / 4 * ((p.cw + 2 * kAhead - 1) / (2 * kAhead) * kAhead) > (1LL << 24)) return false;
    // 32-bit buffer offsets: all rows' words, 64 columns' words
    if ((long long)p.cw * p.B * 4 >= (1LL << 31) || (long long)p.cw * 32 * kNT * 4 >= (1LL << 31)) return false;
    // Large enough to give every CU a workgroup with two image tiles per wave; smaller problems are bound by launch and fill and
    // stay with the kernels written for them, but for int32 products that take those kernels' waves, one 32 x 32 tile each, more than
    // one round of 1 024: the second one is as long as the first for however few tiles.  Two rounds from K = 3 840 on (332 x 4 224 x
    // 3 872 10.8 us there, 10.5 here; 200 x 8 192 x 8 192 24.6 / 17.0; shorter ones 264 x 6 976 x 1 728 7.0 / 8.0, 2 450 x 608 x 2 592
    // 8.3 / 9.2), more rounds at 100 000 words of tiles (8 192 x 448 x 8 192 30.3 / 19.5, 1 500 x 1 504 x 1 504 8.4 / 7.7, 2 433 x 1 312 x
    // 1 696 10.4 / 8.8; below the line 1 812 x 1 312 x 864 6.3 / 6.8).  Over 800 products to either side of the lines none takes more
    // than 3 % longer than with the other kernel.
    const long long wgs = (long long)((p.B + 32 * 2 * kWaves - 1) / (32 * 2 * kWaves)) * ((p.N + 32 * kNT - 1) / (32 * kNT));
    const long long tiles = (long long)((p.B + 31) / 32) * ((p.N + 31) / 32);
    return wgs >= 256 || (p.mode == EPI_RAW && ((tiles > 1024 && p.cw >= 120) || (tiles > 2048 && tiles * p.cw >= 100000)));
}

void gemm_mfma_kernel_name(const BgemmParams& p, char* buf, size_t len) {
    snprintf(buf, len, "gemm_mfma_f4_kernel<%d, %d, %s>", gemm_mt(p), p.mode, p.cw % 4 != 0 ? "true" : "false");
}

template <int MT>
static int launch_gemm_mt(const BgemmParams& p, hipStream_t stream) {
    const int n_groups = (p.N + 32 * kNT - 1) / (32 * kNT);
    const long long row_blocks = (p.B + 32 * MT * kWaves - 1) / (32 * MT * kWaves);
    const long long blocks = row_blocks * n_groups;
    if (blocks <= 0 || blocks > 0x7fffffffLL) return fail(TCBNN_EINVAL, "gemm grid too large");
    const dim3 grid((unsigned)blocks), block(kThreads);
    const bool tail = p.cw % 4 != 0;
    TCBNN_REQUIRE(!tail || p.mode == EPI_RAW, "gemm: rows that are no whole 128-bit units");
    switch (p.mode) {
        case EPI_THRESH:
            hipLaunchKernelGGL((gemm_mfma_f4_kernel<MT, EPI_THRESH, false>), grid, block, 0, stream, p, p.act, p.wgt, p.bn,
                               p.bn, n_groups);
            break;
        case EPI_AFFINE:
            hipLaunchKernelGGL((gemm_mfma_f4_kernel<MT, EPI_AFFINE, false>), grid, block, 0, stream, p, p.act, p.wgt,
                               p.bn_scale, p.bn_bias, n_groups);
            break;
        default:
            if (tail)
                hipLaunchKernelGGL((gemm_mfma_f4_kernel<MT, EPI_RAW, true>), grid, block, 0, stream, p, p.act, p.wgt, p.bn,
                                   p.bn, n_groups);
            else
                hipLaunchKernelGGL((gemm_mfma_f4_kernel<MT, EPI_RAW, false>), grid, block, 0, stream, p, p.act, p.wgt, p.bn,
                                   p.bn, n_groups);
    }
    TCBNN_LAUNCH_CHECK("gemm_mfma_f4_kernel");
    return TCBNN_OK;
}

int launch_gemm_mfma(const BgemmParams& p, hipStream_t stream) {
    return gemm_mt(p) == 4 ? launch_gemm_mt<4>(p, stream) : launch_gemm_mt<2>(p, stream);
}

}  // namespace tcbnn
