// Single-step launches: every team of waves takes exactly one row, and the
// hardware's block scheduler walks the rows instead of a loop in the kernel.
// They serve the launches in which a row's latency chain (load, reduce,
// store), not the HBM, sets the time; the walking kernels of rln_device.h
// serve the larger ones. single_forward and single_backward say which.
//
// What bounds a small launch is the time from its first load to its last
// store: an empty kernel in a graph's chain takes 1.9 us per node, a copy
// 2.0-2.2 us, and the walking kernels 4-7 us, most of it in blocks that take
// several rows one after the other on a few of the 256 CUs, behind unrolled
// walks and, with dropout, a Philox chain of 2-4 draws per lane. Here
//  * a row is split over more waves, one to four four-element slots per lane,
//    so a lane holds 36-96 VGPRs (forward) or 57-90 (backward) over all types and
//    alignments, 5-8 waves fit a SIMD, and rows spread over every CU; row sums
//    cross the waves in LDS, in the walking shape's order, so both kernels give a
//    row the same bits;
//  * no loop: one row's loads, sums and stores are the whole kernel;
//  * rows are read through buffer descriptors over exactly the row, so lanes
//    past its end read zeros and store nothing, without a branch;
//  * the waves of a row share its Philox draws: a unit of 64 draws is one
//    wave's, and its ballots are the mask words themselves.
// Measured on MI355X (us per launch in graphs of dependent calls, walking ->
// single-step): forward [10, 768] bf16 in and out 4.0 -> 2.9, [64, 1600] fp16
// 3.9 -> 3.3, [682, 384] fp16 branch with dropout 6.9 -> 4.1, [341, 768] with
// dropout 7.1 -> 4.4, [2048, 1024] with dropout 9.5 -> 7.6.

#ifndef RLN_SINGLE_H
#define RLN_SINGLE_H

#include "rln_device.h"

// Switches for A/B builds (bench.py --ab): 0 keeps a pass on the walking kernels
// at every size; 1 gives 768 columns with 32-bit gradients the line of the others
// (single_backward_most); and the rows of a chunk (single_chunk_rows), 0 = by rule.
#ifndef RLN_FWD_SINGLE_STEP
#define RLN_FWD_SINGLE_STEP 1
#endif
#ifndef RLN_BWD_SINGLE_STEP
#define RLN_BWD_SINGLE_STEP 1
#endif
#ifndef RLN_BWD_SINGLE_STEP_768
#define RLN_BWD_SINGLE_STEP_768 0
#endif
#ifndef RLN_SINGLE_CHUNK_ROWS
#define RLN_SINGLE_CHUNK_ROWS 0
#endif

namespace rln {

// Waves of a row, and of a block, of the single-step kernels.
constexpr int kSingleMaxParts = 8;
constexpr int kSingleMaxWaves = 8;

// Cache policies. Row inputs of the forward are read once: non-temporal
// ([4096, 512] 8.8 -> 8.1 us, [2048, 768] 7.6 -> 7.0 against cached loads).
// Row outputs are written through, as in every launch of this size: with
// plain stores the end of the kernel waits for L2's write-back ([8, 768] 2.9
// against 3.4 us, [1024, 768] 5.3 against 7.7 us).
constexpr int kSingleStreamLoad = 2;
constexpr int kSingleCachedLoad = 0;

// The order in which a row's sums add up, which is that of the walking shape
// the row would run in, so that a row's outputs are the same bits whichever
// kernel computes them: each lane of a part adds its slots in ascending
// order, the lanes add by row_sum, the parts in ascending order (Slots and
// team_sum in rln_device.h; vector j is slot v of lane l of part p with
// j = (v * parts + p) * lanes + l).
struct SumOrder {
    int lanes;
    int vectors;
    int parts;
};

template <Pass kPass>
SumOrder sum_order(int64_t hidden, int64_t rows) {
    const ShapeInfo info = shape_info(hidden, kPass, rows);
    int lanes = kWaveSize / info.rows_per_wave;
    if (kPass == Pass::kForward && specialized_hidden(hidden)) {
        lanes = forward_lanes<float>(hidden);
    }
    const int64_t per_slot = 4 * lanes * info.parts;
    return {lanes, static_cast<int>((hidden + per_slot - 1) / per_slot), info.parts};
}

// How the lanes of a split reach the sum order's lanes.
enum class SumPath {
    kDirect,    // they hold the row as the order does
    kLanes,     // one wave per row, lanes of 16 or 32 in the order: across the wave's halves
    kExchange,  // several waves per row, one part in the order (or two): slot sums through LDS
};

// How a single-step launch splits its rows.
struct SingleSplit {
    int vectors;  // four-element slots per lane
    SumPath path;
    int parts;       // waves per row
    int groups;      // rows per block
    int reciprocal;  // wave / parts == (wave * reciprocal) >> 8 for every wave of a block
    SumOrder order;
    int waves() const { return parts * groups; }
    int threads() const { return kWaveSize * waves(); }
};

// The forward splits rows of up to 2048 columns finer than their sum order:
// two slots per lane (one up to 256 columns, where a second would be idle),
// so more waves share a row's Philox draws and loads ([341, 768] with
// dropout 4.3 us on two waves of two slots, 4.8 on one of three; [512, 1024]
// 4.8 against 5.8; [163, 1600] 4.0 against 4.4). Longer rows keep their order's
// waves ([64, 4096] without dropout 4.3 us either way). The backward splits
// rows of up to 768 columns finer, one slot per lane ([341, 768] 3.6 us on
// three waves of one slot, 3.8 on one of three; [10923, 768] 28.2 against
// 28.8), and keeps the order's waves above.
template <Pass kPass>
SingleSplit single_split(int64_t hidden, int64_t rows) {
    SingleSplit s{};
    s.order = sum_order<kPass>(hidden, rows);
    const int64_t finest = kPass == Pass::kForward ? 2048 : 768;
    if (hidden > finest) {
        s.path = SumPath::kDirect;
        s.vectors = s.order.vectors;
        s.parts = s.order.parts;
    } else {
        s.vectors = kPass == Pass::kForward && hidden > 256 ? 2 : 1;
        const int64_t per_wave = 4 * kWaveSize * s.vectors;
        s.parts = static_cast<int>((hidden + per_wave - 1) / per_wave);
        // One wave of one slot holds the backward's row as its order does (at
        // 128 columns the upper lanes add zeros).
        s.path = s.parts > 1                ? SumPath::kExchange
            : kPass == Pass::kForward ? SumPath::kLanes
                                      : SumPath::kDirect;
    }
    s.groups = s.parts <= 2 ? 4 / s.parts : 1;
    s.reciprocal = (256 + s.parts - 1) / s.parts;
    return s;
}

// The forward runs single-step up to 2^21 elements for rows of at most 1280
// columns and 6144 rows, and up to 2^20 for longer rows; there the walking
// kernels' look-ahead starts to pay ([2731, 768] 10.4 -> 8.8 us with dropout,
// [4139, 768] 11.9 -> 12.1; [4096, 512] 9.4 -> 7.1, [6208, 512] 11.3 -> 11.4;
// [8192, 128] 7.0 -> 7.8; [655, 1600] 5.6 -> 5.1, [993, 1600] 6.2 -> 6.4).
// Without dropout, rows above 4096 columns only for a few rows ([1, 8192]
// 5.0 -> 4.7 us, [32, 8192] 5.3 -> 5.6; with dropout [128, 8192] 7.2 -> 6.7), and
// rows of 128 columns only up to one row step of the walk, 4096 rows ([4096,
// 128] 4.3 -> 4.1, [5792, 128] 4.5 -> 4.9; with dropout [5792, 128] 6.8 -> 6.6).
//
// Misaligned tensors (element accesses) up to 384 K elements (512 K for 512-1024
// columns) of rows of at most 4096 columns: from there four times the access
// instructions per lane cost more than the walk (us, walking -> single-step: [341,
// 768] with dropout 8.3 -> 5.1, [512, 1024] 10.9 -> 7.0, [64, 4096] 7.7 -> 6.4; past
// the lines [257, 2880] fp16 8.7 -> 10.1, [1927, 1088] 18.5 -> 21.9), and above 4096
// columns it gains nothing at any size ([12, 5120] without dropout 5.7 -> 6.2, [64,
// 8192] with it 9.4 -> 10.3).
inline bool single_forward(int64_t rows, int64_t hidden, bool dropout, bool aligned) {
    const int64_t elements = rows * hidden;
    if (!RLN_FWD_SINGLE_STEP) {
        return false;
    }
    if (!aligned) {
        return hidden <= 4096
            && elements <= (hidden >= 512 && hidden <= 1024 ? 512 << 10 : 384 << 10);
    }
    if (hidden > 4096 && !dropout) {
        return elements <= (1 << 17);
    }
    return rows <= (hidden == 128 && !dropout ? 4096 : 6144)
        && elements <= (hidden <= 1280 ? 1 << 21 : 1 << 20);
}

// Orders a block's LDS writes before its reads: a barrier where several waves
// share a row (a property of the launch, so every wave of the block calls
// it), else a handoff within the wave.
__device__ __forceinline__ void row_handoff(int parts) {
    if (parts > 1) {
        __syncthreads();
    } else {
        wave_handoff();
    }
}

// The backward runs single-step up to 12 M elements (2^24 above 6144 columns,
// 2^23 for 256 and 4096-6144, 6 M for 1025-3072, 4 M there with a 32-bit branch
// and gradient, 3 M for 3073-4095, 2^22 for 128), where the
// walking backward's own costs - the fixed part of its row chains, and the
// weight/bias atomics of its up to 256 blocks, which grow with the row length
// and not with the rows - outweigh reading `updated` and grad_normalized a
// second time. Measured (us, walking -> single-step), backward alone: [10, 768]
// 4.2 -> 2.6, [682, 384] 5.8 -> 3.7, [163, 1600] 6.2 -> 3.8, [128, 4096] 9.3 ->
// 4.8, [256, 8192] 35.0 -> 10.8, [4096, 512] 13.2 -> 9.6, [8192, 1024] 30.9 ->
// 28.4, [12291, 384] fp32 20.6 -> 18.8, [2340, 7168] 71.0 -> 65.2; forward and
// backward of the same batch, three or four batches in turn: [1024, 1024] 19.7
// -> 12.3, [4096, 1024] 31.9 -> 28.4, [33111, 384] 77.8 -> 73.8, [2621, 1600]
// 35.6 -> 32.9, [1024, 4096] 36.6 -> 30.2; and where the lines lie [32768, 128]
// 32.1 -> 31.5, [61445, 128] fp16 out 47.2 -> 48.5, [32768, 256] 53.2 -> 50.6,
// [52119, 256] fp32 branch 84.2 -> 85.0, [16555, 768] 77.4 -> 75.7, [21845, 768]
// 95.8 -> 96.9, [3973, 1600] 45.0 -> 43.6, [2207, 2880] 45.2 -> 45.9, [2048,
// 4096] 55.4 -> 55.4, [2048, 8192] 116.6 -> 110.9; with a 32-bit branch and gradient,
// backward alone, [2621, 1600] 18.6 -> 18.5, [3707, 1600] 23.4 -> 25.0; [827, 3584] 18.8 -> 16.0,
// [1170, 3584] 20.1 -> 21.4, [1655, 3584] fp16 23.8 -> 25.3.
//
// Rows of 768 columns with a 32-bit grad_normalized and weight/bias sums pass over
// to the walk at 7168 rows already: from there single-step is still faster alone
// ([8192, 768] 23.1 -> 20.2), but a forward right after it takes 1-3 us longer as long
// as the batches that alternate are few enough to stay partly in the 256 MB
// Infinity Cache. Forward and backward, fp16 branch, walking -> single-step, over
// three / four / eight batches: 6656 rows 35.6 -> 34.0 / 36.0 -> 34.8 / 38.5 -> 35.9;
// 7168 35.6 -> 36.4 / 35.9 -> 36.9 / 38.1 -> 37.1; 7936 38.9 -> 40.4 / 39.5 -> 40.2 /
// 41.6 -> 40.4; 8192 39.3 -> 40.7 / 39.5 -> 41.2 / 41.8 -> 40.9; 9217 44.6 -> 45.5 /
// 45.3 -> 46.4 / 46.5 -> 46.3; 11264 52.3 -> 52.3 / 52.2 -> 52.6 / 54.0 -> 52.6; 13312
// 59.0 -> 60.4 / 58.8 -> 60.5 / 61.5 -> 60.5; 15360 67.7 -> 68.9 / 67.2 -> 68.8 / 70.0 ->
// 68.9 (fp32 branch: the same signs). So the walk is the choice for programs of a few
// layers, and costs those with many between a forward and its backward 1-3 %.
// Nothing of it shows with 16-bit gradients ([8192, 768] 37.9 -> 36.1 over three), at 640
// and 896 columns (5120-16384 rows, three batches: 0.88-1.01 and 0.91-1.00 of the walk)
// or without the sums.
//
// Misaligned tensors (element accesses) have lines of their own. At 320-768
// columns, whose rows hold one slot per lane, they are the same ([5461, 768] 33.7
// -> 21.8, [6553, 640] 36.5 -> 22.1); elsewhere the slab blocks' second read costs
// four times the instructions. With weight/bias sums: [5792, 128] 11.1 -> 8.8, [772,
// 960] 14.0 -> 8.7, [926, 1600] 17.5 -> 15.5, [252, 4160] 20.8 -> 10.8, [337, 6208] 34.6
// -> 20.9; past the lines [11585, 128] fp32 17.4 -> 19.1, [4369, 960] fp32 40.6 ->
// 49.7, [712, 4160] 29.6 -> 33.4, [675, 6208] fp32 51.1 -> 60.2, [682, 6144] fp32 42.5 ->
// 63.1. Without sums, where only the row chains can gain: [204, 1280] 5.8 -> 4.7,
// [579, 1280] 8.3 -> 9.6, and rows of 2433-6144 columns lose at every size ([21,
// 3072] 4.4 -> 4.6, [482, 3072] 12.2 -> 14.8).
//
// Deterministic launches put partials into the workspace instead of adding
// atomics, so the row chains alone pay for the second read, up to 2 M elements
// for 320-768 columns, 3 M up to 2432, 4 M, 6 M and 12 M for longer rows: [2730, 768]
// 17.0 -> 13.6, [2048, 1024] 13.5 -> 12.0, [1310, 1600] 14.2 -> 13.2, [965, 3072] 19.3 ->
// 16.3, [819, 5120] 26.6 -> 21.9, [827, 7168] 37.6 -> 29.4, [1448, 256] 9.6 -> 6.8; past the
// lines [5461, 768] 19.9 -> 21.4, [13107, 640] 32.6 -> 36.1, [8192, 1024] 31.1 -> 33.1,
// [3707, 1600] 24.8 -> 26.2, [1655, 3584] 27.4 -> 28.7, [1638, 5120] 35.6 -> 38.8, [2702,
// 6208] 72.5 -> 75.9, [5792, 256] 11.1 -> 11.7, [1930, 192] bf16 6.8 -> 7.1, [4096, 128] 7.5 ->
// 8.2. The sums are the same bits for tensors of any alignment, so these lines do
// not ask for it; element accesses alone would walk from 1 M elements ([1310, 1600]
// 21.1 -> 24.3, [682, 6144] fp32 46.2 -> 63.9, [1024, 8192] fp32 93.0 -> 153.8).
struct SingleBackwardCall {
    int64_t rows;
    int64_t hidden;
    int branch_dtype;
    int grad_normalized_dtype;
    bool has_grad_normalized;
    bool sums;      // weight and bias sums, by atomics or ...
    bool partials;  // ... through partials in the workspace
    bool aligned;   // vector accesses
};

inline int64_t single_backward_most(const SingleBackwardCall& c) {
    constexpr int64_t K = 1 << 10;
    constexpr int64_t M = 1 << 20;
    struct Misaligned {
        int64_t hidden;  // rows of up to so many columns
        int64_t sums;    // elements
        int64_t none;
    };
    constexpr Misaligned kMisaligned[] = {
        {256, M, 256 * K},  {768, 12 * M, 12 * M}, {1024, M, 384 * K},           {2432, M, 512 * K},
        {4096, M, 0},       {6144, 1536 * K, 0},   {kMaxHidden, 3 * M, 2 * M},
    };
    if (c.partials) {
        return c.hidden == 128  ? 384 * K
            : c.hidden == 192   ? 256 * K
            : c.hidden == 256   ? 768 * K
            : c.hidden <= 768   ? 2 * M
            : c.hidden <= 2432  ? 3 * M
            : c.hidden < 4096   ? 4 * M
            : c.hidden <= 6144  ? 6 * M
                                : 12 * M;
    }
    if (!c.aligned) {
        for (const Misaligned& line : kMisaligned) {
            if (c.hidden <= line.hidden) {
                return c.sums ? line.sums : line.none;
            }
        }
    }
    const bool wide =
        c.branch_dtype == RLN_DTYPE_F32 && c.grad_normalized_dtype == RLN_DTYPE_F32;
    return c.hidden == 128           ? 4 * M
        : c.hidden == 256            ? 8 * M
        : c.hidden == 768 && c.sums && c.grad_normalized_dtype == RLN_DTYPE_F32
                && !RLN_BWD_SINGLE_STEP_768
            ? 7167 * 768
        : c.hidden <= 1024           ? 12 * M
        : c.hidden <= 3072           ? (wide ? 4 * M : 6 * M)
        : c.hidden < 4096            ? 3 * M
        : c.hidden <= 6144           ? 8 * M
        : c.hidden <= 7936 || c.sums ? 16 * M
        : wide                       ? 3 * M
                                     : 5 * M;
}

// A backward without weight/bias sums (frozen parameters, or no grad_normalized)
// has no atomics to save, and the walk of few rows is short: where its whole
// grid of one block per CU is (nearly) full in its first or second row step,
// single-step blocks lose up to a quarter. Measured (us, walking ->
// single-step), frozen parameters unless said otherwise:
//  * eight-wave rows of 2433-6144 columns (one row per block and step): up to
//    256 rows [241, 3072] 5.1 -> 4.5, above [482, 3072] 7.1 -> 7.7, [512, 4096] 8.1 ->
//    9.1, [682, 6144] fp32 17.2 -> 21.0 (forward and backward [682, 3072] 18.2 ->
//    20.3); without grad_normalized, whose walk is shorter, up to 2^19 elements
//    of 2433-5120 columns too ([42, 3072] 3.1 -> 3.4, [148, 2496] 3.6 -> 3.9; [241,
//    3072] 4.8 -> 4.3, [85, 6144] 5.3 -> 4.7);
//  * four-wave rows of 1217-2048 columns, 768 to a step: [579, 1280] 5.1 -> 5.4,
//    [655, 1600] 5.8 -> 6.3, [724, 2048] 6.8 -> 7.9, [1170, 1792] 9.1 -> 9.7;
//    and beside them [512, 2048] 5.8 -> 5.7, [926, 1600] 8.3 -> 7.3; of 2049-2432
//    columns, 512 to a step, its second: [862, 2432] 9.1 -> 9.4 (forward and
//    backward [609, 2432] 16.3 -> 17.4);
//  * rows of 128-256 columns without grad_normalized in the first step: [4096, 128]
//    3.7 -> 4.0, [5792, 128] 5.3 -> 4.5;
//  * rows of 8000-8192 columns lose from 5 M elements, 3 M with a 32-bit branch and
//    gradient ([362, 8192] 18.1 -> 13.7, [512, 8192] 21.6 -> 18.2, fp32 22.1 -> 25.0, [1448,
//    8192] 45.5 -> 50.8), shorter ones up to 7936 do not ([1170, 7168] 33.5 -> 34.3).
inline bool walk_without_sums(const SingleBackwardCall& c) {
    const ShapeInfo info = shape_info(c.hidden, Pass::kBackward, c.rows);
    const int64_t step = kBackwardMaxBlocks * (info.backward_threads / kWaveSize)
        * info.rows_per_wave / info.parts;
    const int64_t steps = (c.rows + step - 1) / step;
    const int64_t last = c.rows - (steps - 1) * step;
    if (c.hidden > 2432) {
        return c.hidden <= 6144
            && (steps > 1 || (!c.has_grad_normalized && c.hidden <= 5120
                              && c.rows * c.hidden <= (1 << 19)));
    }
    if (c.hidden > 2048) {
        return steps == 2;
    }
    if (c.hidden > 1216) {
        return (steps == 1 && 4 * last > 3 * step) || (steps == 2 && 2 * last > step);
    }
    return c.hidden <= 256 && !c.has_grad_normalized && steps == 1 && 3 * last > 2 * step;
}

inline bool single_backward(const SingleBackwardCall& c) {
    if (!RLN_BWD_SINGLE_STEP) {
        return false;
    }
    return c.rows * c.hidden <= single_backward_most(c) && (c.sums || !walk_without_sums(c));
}

// Rows of one chunk: its blocks run on one XCD, and its slab blocks read again
// from that XCD's L2 what its row blocks read. 64 rows, 32 where a block has
// three waves (513-768 columns: its slab has three quarters of the waves of the
// others', and takes as long for fewer rows), fewer when there are fewer rows than
// eight such chunks, one per XCD, so that every XCD has work. Smaller chunks mean
// more weight/bias atomics, larger ones longer slab blocks, and past L2's size a
// second read from memory: [8192, 768] 21.9 us at 32 rows, 22.7 at 64, 23.5 at 128;
// [8192, 1600] 44.5, 43.2, 43.8; [16384, 128] 16.3, 10.4, 10.6. At 513-768 columns over
// 2^17-2^23 elements, against 32 rows: 64 rows +1 to +14 %, 48 rows (a whole
// unrolled step of three waves) -2 to +2 % but +3 to +10 % at the rows that then leave
// an XCD idle ([482, 768]).
inline int64_t single_chunk_rows(int64_t rows, const SingleSplit& split) {
    const int64_t most = RLN_SINGLE_CHUNK_ROWS ? RLN_SINGLE_CHUNK_ROWS
        : split.waves() == 3                    ? 32
                                                : 64;
    const int64_t spread = (rows + 7) / 8;
    return spread < most ? (spread + 3) / 4 * 4 : most;
}

// Deterministic launches put one group of partials per chunk into a workspace
// of backward_blocks(rows, hidden) groups, so a chunk may have to be larger.
inline int64_t single_partial_rows(int64_t rows, int64_t hidden, const SingleSplit& split) {
    const int64_t groups = backward_blocks(rows, hidden);
    const int64_t least = (rows + groups - 1) / groups;
    const int64_t chunk = single_chunk_rows(rows, split);
    return least > chunk ? least : chunk;
}

// Whether two device ranges share a byte (null: no range).
inline bool ranges_overlap(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
    const uintptr_t first = reinterpret_cast<uintptr_t>(a);
    const uintptr_t second = reinterpret_cast<uintptr_t>(b);
    return a != nullptr && b != nullptr && first < second + static_cast<uintptr_t>(b_bytes)
        && second < first + static_cast<uintptr_t>(a_bytes);
}

// Whether a backward writes grad_x or grad_branch over `updated`,
// grad_normalized, mean or rstd.
inline bool gradients_over_inputs(const BackwardArgs& a, int64_t hidden, int branch_dtype,
                                  int grad_normalized_dtype) {
    const int64_t bytes = a.rows * hidden * 4;
    const auto sized = [&](int dtype) { return dtype == RLN_DTYPE_F32 ? bytes : bytes / 2; };
    const auto written = [&](const void* input, int64_t input_bytes) {
        return ranges_overlap(input, input_bytes, a.grad_x, bytes)
            || ranges_overlap(input, input_bytes, a.grad_branch, sized(branch_dtype));
    };
    return written(a.updated, bytes) || written(a.grad_normalized, sized(grad_normalized_dtype))
        || written(a.mean, a.rows * 4) || written(a.rstd, a.rows * 4);
}

// Whether a backward launch runs single-step. Its slab blocks read `updated`
// and grad_normalized beside the row blocks' stores, so gradients written over
// what they read take the walking kernels, which read each row once, before
// its stores. (The size rules come first: sizes in bytes are then small, while
// the C ABI accepts row counts whose bytes overflow int64.)
inline bool takes_single_backward(const BackwardArgs& a, int64_t hidden, int branch_dtype,
                                  int grad_normalized_dtype, bool aligned) {
    const bool sums = (a.flags & kParameters) != 0;
    const bool partials = (a.flags & kPartials) != 0;
    return single_backward({a.rows, hidden, branch_dtype, grad_normalized_dtype,
                            (a.flags & kHasGradNormalized) != 0, sums, partials, aligned})
        && !(sums && gradients_over_inputs(a, hidden, branch_dtype, grad_normalized_dtype));
}

// A block's LDS array of row sums: its length, where the sums of the block's
// row `group` begin, and how many elements from there its lanes read. Direct:
// one per wave; the lanes read kSingleMaxParts of them in a fixed loop and drop
// those past the row's waves, so the array reaches that far past the last row's
// first. Exchange: one per vector of the block's rows (at most four waves).
constexpr int single_shared_size(SumPath path, int vectors) {
    return path == SumPath::kExchange ? vectors * 4 * kWaveSize
                                      : kSingleMaxWaves + kSingleMaxParts;
}
constexpr int single_shared_first(SumPath path, int vectors, int parts, int group) {
    return group * parts * (path == SumPath::kExchange ? vectors * kWaveSize : 1);
}
constexpr int single_shared_read(SumPath path, int parts, const SumOrder& order) {
    if (path == SumPath::kExchange) {
        return order.vectors * order.parts * order.lanes;
    }
    return parts > 1 ? kSingleMaxParts : 0;  // one wave keeps its sum in registers
}

// `value` of the lanes of the wave's lower (upper) half in `low` (`high`), for
// the lanes of both halves.
__device__ __forceinline__ void split_halves(float value, float& low, float& high) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, value);
    const auto halves = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    low = __builtin_bit_cast(float, static_cast<uint32_t>(halves[0]));
    high = __builtin_bit_cast(float, static_cast<uint32_t>(halves[1]));
}

// Sums over a row of V slots per lane, in the row's sum order; every lane of
// the row's waves gets it. `slots` are the lane's slot sums (zeros past the
// row) and `shared` the row's own LDS floats: one per wave (direct), or one
// per vector (exchange). Every wave of a block of several waves per row calls
// it (it holds a barrier).
template <int V, SumPath Path>
__device__ __forceinline__ float single_sum(const float (&slots)[V], float* shared, int parts,
                                            int part, const SumOrder& order) {
    const int lane = threadIdx.x & (kWaveSize - 1);
    if constexpr (Path == SumPath::kDirect) {
        float partial = 0.0f;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            partial += slots[v];
        }
        partial = row_sum<kWaveSize>(partial);
        if (parts == 1) {
            return partial;
        }
        if (lane == 0) {
            shared[part] = partial;
        }
        __syncthreads();
        float total = shared[0];
#pragma unroll
        for (int other = 1; other < kSingleMaxParts; ++other) {
            const float next = shared[other];
            total = other < parts ? total + next : total;
        }
        return total;
    } else if constexpr (Path == SumPath::kLanes) {
        // Vector j is slot j / lanes of lane j % lanes in the order, and here
        // slot j / 64 of lane j % 64.
        if (order.lanes == 64) {
            float partial = slots[0];
#pragma unroll
            for (int v = 1; v < V; ++v) {
                partial += slots[v];
            }
            return row_sum<64>(partial);
        }
        if (order.lanes == 32) {
            float partial = 0.0f;
#pragma unroll
            for (int v = 0; v < V; ++v) {
                float low;
                float high;
                split_halves(slots[v], low, high);
                partial = (partial + low) + high;
            }
            partial = row16_sum(partial);
            return readlane_f32(partial, 0) + readlane_f32(partial, 16);
        }
        // 16 lanes of two slots (128 columns): lanes l and l + 16.
        const uint32_t bits = __builtin_bit_cast(uint32_t, slots[0]);
        const auto rows = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
        const float partial = row16_sum(__builtin_bit_cast(float, static_cast<uint32_t>(rows[0]))
                                        + __builtin_bit_cast(float, static_cast<uint32_t>(rows[1])));
        return readlane_f32(partial, 0);
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            shared[(v * parts + part) * kWaveSize + lane] = slots[v];
        }
        __syncthreads();
        // Rows of one part of 64 lanes, or two; the split covers every vector
        // of the order, with zeros past the row. Every slot is read before
        // any is added (slots past the order's count again, and not added): a
        // read under a branch would wait for each in turn ([163, 1600] 4.7
        // against 4.0 us).
        const int stride = order.parts * kWaveSize;
        const float* const first = shared + lane;
        const float* const second = first + (order.parts > 1 ? kWaveSize : 0);
        float a[4];
        float b[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int slot = v < order.vectors ? v : 0;
            a[v] = first[slot * stride];
            b[v] = second[slot * stride];
        }
        float partial_a = a[0];
        float partial_b = b[0];
#pragma unroll
        for (int v = 1; v < 4; ++v) {
            partial_a = v < order.vectors ? partial_a + a[v] : partial_a;
            partial_b = v < order.vectors ? partial_b + b[v] : partial_b;
        }
        const float sum_a = row_sum<kWaveSize>(partial_a);
        const float sum_b = row_sum<kWaveSize>(partial_b);
        return order.parts > 1 ? sum_a + sum_b : sum_a;
    }
}

// The backward's two row sums at once, as single_sum: `shared` holds the pair
// of every wave of the row (direct) or of every vector (exchange: one slot per
// lane, one part in the order).
template <int V, SumPath Path>
__device__ __forceinline__ float2 single_pair_sum(const float (&q)[V], const float (&qx)[V],
                                                  float2* shared, int parts, int part,
                                                  const SumOrder& order) {
    const int lane = threadIdx.x & (kWaveSize - 1);
    if constexpr (Path == SumPath::kDirect) {
        float2 partial = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            partial.x += q[v];
            partial.y += qx[v];
        }
        partial.x = row_sum<kWaveSize>(partial.x);
        partial.y = row_sum<kWaveSize>(partial.y);
        if (parts == 1) {
            return partial;
        }
        if (lane == 0) {
            shared[part] = partial;
        }
        __syncthreads();
        float2 total = shared[0];
#pragma unroll
        for (int other = 1; other < kSingleMaxParts; ++other) {
            const float2 next = shared[other];
            total.x = other < parts ? total.x + next.x : total.x;
            total.y = other < parts ? total.y + next.y : total.y;
        }
        return total;
    } else {
        static_assert(V == 1, "one slot per lane");
        shared[part * kWaveSize + lane] = make_float2(q[0], qx[0]);
        __syncthreads();
        // Two or three slots of 64 lanes, or three of 32 (384 columns).
        const float2* const first = shared + (lane & (order.lanes - 1));
        const float2 a = first[0];
        const float2 b = first[order.lanes];
        const float2 c = first[order.vectors > 2 ? 2 * order.lanes : 0];
        float2 partial = make_float2(a.x + b.x, a.y + b.y);
        partial.x = order.vectors > 2 ? partial.x + c.x : partial.x;
        partial.y = order.vectors > 2 ? partial.y + c.y : partial.y;
        partial.x = row16_sum(partial.x);
        partial.y = row16_sum(partial.y);
        const float2 low =
            make_float2(readlane_f32(partial.x, 0) + readlane_f32(partial.x, 16),
                        readlane_f32(partial.y, 0) + readlane_f32(partial.y, 16));
        const float2 high =
            make_float2(readlane_f32(partial.x, 32) + readlane_f32(partial.x, 48),
                        readlane_f32(partial.y, 32) + readlane_f32(partial.y, 48));
        return order.lanes == kWaveSize ? make_float2(low.x + high.x, low.y + high.y) : low;
    }
}

// A descriptor over `count` elements of `tensor` from element `first`, for
// reading (wave-uniform arguments; count * sizeof(T) < 2^31). A count of 0
// makes every read return zero and touch no memory.
template <typename T>
__device__ __forceinline__ rsrc_t input_range(const T* tensor, int64_t first, int64_t count) {
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(static_cast<const void*>(tensor + first)), 0,
        static_cast<int>(count * static_cast<int64_t>(sizeof(T))), kRawBufferWord3);
}

// Four consecutive elements from element `index` of a descriptor in their
// storage type; zeros past its end.
template <typename T, bool Aligned, int Policy>
__device__ __forceinline__ typename Vector4<T>::type input4(rsrc_t r, uint32_t index) {
    using Raw = typename Vector4<T>::type;
    if constexpr (Aligned && sizeof(T) == 4) {
        return __builtin_bit_cast(
            Raw, __builtin_amdgcn_raw_buffer_load_b128(r, index * 4, 0, Policy));
    } else if constexpr (Aligned) {
        return __builtin_bit_cast(
            Raw, __builtin_amdgcn_raw_buffer_load_b64(r, index * 2, 0, Policy));
    } else {
        Raw raw;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (sizeof(T) == 4) {
                const uint32_t bits =
                    __builtin_amdgcn_raw_buffer_load_b32(r, (index + e) * 4, 0, Policy);
                raw[e] = __builtin_bit_cast(T, bits);
            } else {
                const uint16_t bits =
                    __builtin_amdgcn_raw_buffer_load_b16(r, (index + e) * 2, 0, Policy);
                raw[e] = __builtin_bit_cast(T, bits);
            }
        }
        return raw;
    }
}

// What a kernel needs to issue its first loads comes as arguments of its own,
// at most 14 words, which the build has the hardware preload into scalar
// registers at wave launch (-amdgpu-kernarg-preload-count); the rest follows in
// a struct. Scalar loads return out of order, so the first use of one waits
// for every one issued: with all arguments in one struct the first row load
// waited for several cold lines of arguments. Measured (us, one struct ->
// separate words -> preloaded): forward [8, 768] bf16 2.92 -> 2.89 -> 2.79,
// [1024, 384] with dropout 4.29 -> 4.18 -> 4.06, [2048, 768] with dropout 6.67
// -> 6.70 -> 6.24; backward [1024, 384] 3.96 -> 3.98 -> 3.75, [64, 1600] 3.31 ->
// 3.33 -> 3.21.
struct SplitWord {
    uint32_t bits;
    static SplitWord of(const SingleSplit& s) {
        return {static_cast<uint32_t>(s.parts | s.groups << 4 | s.reciprocal << 8
                                      | s.order.parts << 18 | s.order.vectors << 22
                                      | (s.order.lanes / 16) << 25)};
    }
    __device__ __forceinline__ int parts() const { return bits & 15; }
    __device__ __forceinline__ int groups() const { return (bits >> 4) & 15; }
    __device__ __forceinline__ int reciprocal() const { return (bits >> 8) & 1023; }
    __device__ __forceinline__ SumOrder order() const {
        return {static_cast<int>(bits >> 25) * 16, static_cast<int>((bits >> 22) & 7),
                static_cast<int>((bits >> 18) & 15)};
    }
};

// Dropout of a single-step forward: off, or the stream's launch width (0: the
// library's layout) and whether the seed is a device pointer.
struct DropWord {
    uint32_t bits;
    static DropWord of(int dropout, const PhiloxArgs& philox) {
        return {static_cast<uint32_t>((dropout ? 1 : 0) | (philox.seed_ptr ? 2 : 0)
                                      | philox.threads << 2)};
    }
    __device__ __forceinline__ bool on() const { return bits & 1; }
    __device__ __forceinline__ bool captured() const { return bits & 2; }
    __device__ __forceinline__ int threads() const { return bits >> 2; }
};

struct SingleForwardArgs {
    uint32_t threshold;
    float scale;
    const float* weight;
    const float* bias;
    float* updated;
    void* normalized;
    uint32_t* mask;
    float* mean;
    float* rstd;
    float inv_hidden;  // 1.0f / hidden, rounded once on the host
    float eps;
    float* zero_weight;
    float* zero_bias;
};

// One row per team of `parts` waves; slot v of lane l of part p holds columns
// 4 * ((v * parts + p) * 64 + l) .. + 3.
template <int V, SumPath Path, typename B, typename N, bool Aligned>
__global__ __launch_bounds__(kSingleMaxWaves * kWaveSize)
void rln_single_forward_kernel(const float* x_rows, const B* branch_rows, int rows, uint32_t hidden,
                               SplitWord split, DropWord drop,
                               const int64_t* __restrict__ seed_or_value, uint64_t philox_offset,
                               const int64_t* __restrict__ offset_ptr,
                               SingleForwardArgs a) {
    // [0] the mean's sum, [1] the variance's.
    __shared__ float shared[2][single_shared_size(Path, V)];
    // Keep bits of the reference's stream, 64 columns each (at most 1024
    // columns, so at most 16 per row, and at most four rows per block).
    __shared__ uint64_t keep[4][16];
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int parts = split.parts();
    const SumOrder order = split.order();
    const int group = (wave * split.reciprocal()) >> 8;
    const int part = wave - group * parts;
    // A team past the last row reads and writes nothing (empty descriptors),
    // but meets its block's barriers.
    const int team_row = blockIdx.x * split.groups() + group;
    const bool valid = team_row < rows;
    const int64_t row = valid ? team_row : 0;
    const int64_t count = valid ? hidden : 0;
    const int64_t base = row * hidden;
    const int row_shared = single_shared_first(Path, V, parts, group);

    // The Philox key and position first: the draws hang on them, and under
    // graph capture they come from memory.
    uint32_t key0 = 0;
    uint32_t key1 = 0;
    uint64_t position = 0;
    const bool dropout = drop.on();
    if (dropout) {
        const uint64_t seed = drop.captured() ? static_cast<uint64_t>(*seed_or_value)
                                              : reinterpret_cast<uint64_t>(seed_or_value);
        const uint64_t offset =
            philox_offset + (offset_ptr ? static_cast<uint64_t>(*offset_ptr) : 0);
        key0 = static_cast<uint32_t>(seed);
        key1 = static_cast<uint32_t>(seed >> 32);
        position = offset / 4;
    }
    uint32_t column[V];
    f32x4 x[V];
    typename Vector4<B>::type branch[V];
    f32x4 w[V];
    f32x4 b[V];
    const rsrc_t x_in = input_range(x_rows, base, count);
    const rsrc_t branch_in = input_range(branch_rows, base, count);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        column[v] = ((v * parts + part) * kWaveSize + lane) * 4;
        x[v] = input4<float, Aligned, kSingleStreamLoad>(x_in, column[v]);
        branch[v] = input4<B, Aligned, kSingleStreamLoad>(branch_in, column[v]);
    }
    const rsrc_t weight_in = input_range(a.weight, 0, hidden);
    const rsrc_t bias_in = input_range(a.bias, 0, hidden);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        w[v] = input4<float, Aligned, kSingleCachedLoad>(weight_in, column[v]);
        b[v] = input4<float, Aligned, kSingleCachedLoad>(bias_in, column[v]);
    }
    // Zero the weight/bias gradient sums a later backward accumulates into.
    if (a.zero_weight != nullptr) {
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < hidden;
             i += gridDim.x * blockDim.x) {
            a.zero_weight[i] = 0.0f;
            a.zero_bias[i] = 0.0f;
        }
    }

    // Keep bits of each slot in bits 0-3 of `bits`; both layouts of the
    // stream are those of the walking forward (rln_device.h).
    uint32_t bits[V];
    if (dropout && drop.threads() != 0) {
        // The reference's stream: thread t of the row draws `calls` Philox
        // blocks, value `item` of which decides column t + item * threads.
        // 64 consecutive threads and one call are a unit; a ballot over value
        // e of a unit covers 64 consecutive columns, two words of the mask.
        const int threads = drop.threads();
        const int per_item = threads / kWaveSize;
        const int items = (static_cast<int>(hidden) + threads - 1) / threads;
        const int calls = (items + 3) / 4;  // 1 or 2
        const int chunks = hidden / kWaveSize;
        for (int unit = part; unit < per_item * calls; unit += parts) {
            const int k = calls == 2 ? unit >> 1 : unit;
            const int n = calls == 2 ? unit & 1 : 0;
            const uint64_t low = position + n;
            const uint64_t high = static_cast<uint64_t>(row) * threads + k * kWaveSize + lane
                + (low < position ? 1 : 0);
            const uint4 random = philox4x32_10(
                make_uint4(static_cast<uint32_t>(low), static_cast<uint32_t>(low >> 32),
                           static_cast<uint32_t>(high), static_cast<uint32_t>(high >> 32)),
                key0, key1);
            const uint32_t draws[4] = {random.x, random.y, random.z, random.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int item = 4 * n + e;
                const int chunk = item * per_item + k;
                const uint64_t ballot = __ballot(draws[e] >= a.threshold);
                if (item < items && chunk < chunks && lane == 0) {
                    keep[group][chunk] = ballot;
                }
            }
        }
        row_handoff(parts);
        const uint32_t* const words = reinterpret_cast<const uint32_t*>(keep[group]);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            bits[v] = column[v] < hidden ? words[column[v] / 32] >> (column[v] % 32) : 0u;
        }
        if (part == 0 && lane < static_cast<int>(hidden / 32)) {
            output_b32(output_range(a.mask, row * (hidden / 32), count / 32), lane * 4,
                       words[lane], true);
        }
    } else if (dropout) {
        const rsrc_t mask_out = output_range(a.mask, row * (hidden / 32), count / 32);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint64_t quad = static_cast<uint64_t>(row) * (hidden / 4) + column[v] / 4;
            const uint4 random = philox4x32_10(
                make_uint4(static_cast<uint32_t>(position), static_cast<uint32_t>(position >> 32),
                           static_cast<uint32_t>(quad), static_cast<uint32_t>(quad >> 32)),
                key0, key1);
            bits[v] = (random.x >= a.threshold ? 1u : 0u) | (random.y >= a.threshold ? 2u : 0u)
                | (random.z >= a.threshold ? 4u : 0u) | (random.w >= a.threshold ? 8u : 0u);
            // Lanes past the row write past its descriptor: dropped.
            const uint32_t word = or8(bits[v] << (4 * (lane & 7)));
            if ((lane & 7) == 0) {
                output_b32(mask_out, column[v] / 8, word, true);
            }
        }
    }

    const rsrc_t updated_out = output_range(a.updated, base, count);
    f32x4 u[V];
    float slots[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        f32x4 d = widen4<B>(branch[v]);
        if (dropout) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                d[e] = round_to_branch<B>(d[e] * static_cast<float>((bits[v] >> e) & 1u)
                                          * a.scale);
            }
        }
        u[v] = x[v] + d;
        output4<Aligned>(updated_out, column[v] * 4, u[v], true);
        slots[v] = sum4(u[v]);  // lanes past the row hold zeros
    }
    const float mean = single_sum<V, Path>(slots, &shared[0][row_shared], parts, part,
                                             order) * a.inv_hidden;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        u[v] = column[v] < hidden ? u[v] - mean : zero4();
        slots[v] = (u[v].x * u[v].x + u[v].y * u[v].y) + (u[v].z * u[v].z + u[v].w * u[v].w);
    }
    const float variance = single_sum<V, Path>(slots, &shared[1][row_shared], parts, part,
                                                 order) * a.inv_hidden;
    const float rstd = rsqrtf(variance + a.eps);
    if (part == 0 && lane == 0) {
        output_b32(output_range(a.mean, row, valid ? 1 : 0), 0,
                   __builtin_bit_cast(uint32_t, mean), true);
        output_b32(output_range(a.rstd, row, valid ? 1 : 0), 0,
                   __builtin_bit_cast(uint32_t, rstd), true);
    }
    const rsrc_t normalized_out = output_range(static_cast<N*>(a.normalized), base, count);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            y[e] = __builtin_fmaf(u[v][e] * rstd, w[v][e], b[v][e]);
        }
        output_convert4<N, Aligned>(normalized_out, column[v] * sizeof(N), y, true);
    }
}

struct SingleBackwardArgs {
    int row_blocks;  // per chunk
    int slab_waves;  // waves that share a slab's rows
    int slabs;       // slabs of a slab block
    int dropout;
    const float* grad_updated;
    const uint32_t* mask;
    const float* weight;
    float* grad_x;
    void* grad_branch;
    float inv_hidden;
    float scale;
    float* grad_weight;
    float* grad_bias;
    float* partials;  // [chunks][2][hidden], or null for atomics
};

constexpr int kSlabColumns = 64;
constexpr int kSlabUnroll = 4;

// Weight/bias sums of a chunk's rows over the slabs of 64 columns of one slab
// block. They need no row sums (the forward saved mean and rstd), so they run
// beside the chunk's row blocks instead of after them, read what those read
// from the XCD's L2, and leave each block two sums per column to add: one add
// per chunk and column instead of one per walking block, spread over the
// kernel instead of at its end. A wave takes four rows of 16 lanes per step;
// the order of the sums is fixed (steps, then the wave's four row slots, then
// waves), so partials are reproducible bit for bit.
template <typename GY, bool Aligned>
__device__ __forceinline__ void single_slab(const SingleBackwardArgs& a, const float* updated,
                                            const GY* grad_normalized, const float* means_in,
                                            const float* rstds_in, uint32_t hidden, int block,
                                            int64_t chunk, int64_t begin, int count) {
    __shared__ float sums[kSingleMaxWaves][8][16];
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave_in_block = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int waves = a.slab_waves;
    const int slab_in_block = wave_in_block >= waves ? 1 : 0;
    const int wave = wave_in_block - slab_in_block * waves;
    const int first_slab = block * a.slabs;
    const uint32_t column =
        (first_slab + slab_in_block) * kSlabColumns + (lane & 15) * 4;
    // A slab past the row's end reads nothing and stores nothing.
    const int64_t rows = column < hidden ? count : 0;
    const int64_t extent = wave_uniform(rows) * hidden;
    const rsrc_t u_in = input_range(updated, begin * hidden, extent);
    const rsrc_t gy_in =
        input_range(grad_normalized, begin * hidden, extent);
    const rsrc_t mean_in = input_range(means_in, begin, count);
    const rsrc_t rstd_in = input_range(rstds_in, begin, count);
    const int sub = lane / 16;
    const int steps = (count + 4 * waves - 1) / (4 * waves);
    f32x4 acc_w = zero4();
    f32x4 acc_b = zero4();
    float means = 0.0f;
    float rstds = 0.0f;
    for (int step = 0; step < steps; step += kSlabUnroll) {
        if (step % 16 == 0) {
            // Lane i keeps the statistics of the wave's i-th row of 16 steps.
            const uint32_t own = ((step + lane / 4) * waves + wave) * 4 + lane % 4;
            means = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(mean_in, own * 4, 0, 0));
            rstds = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(rstd_in, own * 4, 0, 0));
        }
        f32x4 u[kSlabUnroll];
        typename Vector4<GY>::type gy[kSlabUnroll];
#pragma unroll
        for (int k = 0; k < kSlabUnroll; ++k) {
            // Rows past the chunk's end read zeros: they add nothing.
            const uint32_t row = ((step + k) * waves + wave) * 4 + sub;
            u[k] = input4<float, Aligned, kSingleCachedLoad>(u_in, row * hidden + column);
            gy[k] = input4<GY, Aligned, kSingleCachedLoad>(gy_in, row * hidden + column);
        }
#pragma unroll
        for (int k = 0; k < kSlabUnroll; ++k) {
            const int source = (step % 16 + k) * 4 + sub;
            const float mean = __shfl(means, source);
            const float rstd = __shfl(rstds, source);
            const f32x4 g = widen4<GY>(gy[k]);
            const f32x4 xhat = (u[k] - mean) * rstd;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc_w[e] = __builtin_fmaf(g[e], xhat[e], acc_w[e]);
            }
            acc_b = acc_b + g;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        acc_w[e] += __shfl_xor(acc_w[e], 16);
        acc_w[e] += __shfl_xor(acc_w[e], 32);
        acc_b[e] += __shfl_xor(acc_b[e], 16);
        acc_b[e] += __shfl_xor(acc_b[e], 32);
    }
    if (lane < 16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sums[wave_in_block][e][lane] = acc_w[e];
            sums[wave_in_block][4 + e][lane] = acc_b[e];
        }
    }
    __syncthreads();
    // Two waves per slab: its 64 weight sums and its 64 bias sums.
    const int slab = threadIdx.x / (2 * kSlabColumns);
    const int c = threadIdx.x % kSlabColumns;
    const uint32_t out = (first_slab + slab) * kSlabColumns + c;
    if (slab < a.slabs && out < hidden) {
        const int which = (threadIdx.x / kSlabColumns) & 1;
        float total = 0.0f;
        for (int source = 0; source < waves; ++source) {
            total += sums[slab * waves + source][4 * which + c % 4][c / 4];
        }
        if (a.partials != nullptr) {
            a.partials[(chunk * 2 + which) * hidden + out] = total;
        } else {
            unsafeAtomicAdd((which ? a.grad_bias : a.grad_weight) + out, total);
        }
    }
}

// Input gradients: one row per team, as in the forward; weight/bias sums: slab
// blocks of the same launch. gridDim.x = 8 * (row blocks + slab blocks of a
// chunk) and consecutive blocks go to consecutive XCDs, so chunk 8 * y + x
// runs on XCD x, its slab blocks behind its row blocks. (The placement is a
// matter of speed alone.)
template <int V, SumPath Path, typename B, typename GY, bool Aligned>
__global__ __launch_bounds__(kSingleMaxWaves * kWaveSize)
void rln_single_backward_kernel(const float* updated, const GY* grad_normalized,
                                const float* means, const float* rstds, int rows,
                                uint32_t hidden, SplitWord split, int chunk_rows,
                                SingleBackwardArgs a) {
    const int local = blockIdx.x >> 3;
    const int64_t chunk = static_cast<int64_t>(blockIdx.y) * 8 + (blockIdx.x & 7);
    const int64_t begin = chunk * chunk_rows;
    if (begin >= rows) {
        return;
    }
    const int64_t left = rows - begin;
    const int64_t end = begin + (left < chunk_rows ? left : chunk_rows);
    if (local >= a.row_blocks) {
        single_slab<GY, Aligned>(a, updated, grad_normalized, means, rstds, hidden,
                                 local - a.row_blocks, chunk, begin,
                                 static_cast<int>(end - begin));
        return;
    }
    __shared__ float2 shared[single_shared_size(Path, V)];  // both sums
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int parts = split.parts();
    const int group = (wave * split.reciprocal()) >> 8;
    const int part = wave - group * parts;
    const int64_t team_row = begin + static_cast<int64_t>(local) * split.groups() + group;
    const bool valid = team_row < end;
    const int64_t row = valid ? team_row : 0;
    const int64_t count = valid ? hidden : 0;
    const int64_t base = row * hidden;
    // Absent inputs have empty descriptors: zeros, no memory access.
    const bool has_gy = grad_normalized != nullptr;
    const bool has_gu = a.grad_updated != nullptr;
    const rsrc_t u_in = input_range(updated, base, count);
    const rsrc_t gy_in = input_range(grad_normalized, has_gy ? base : 0, has_gy ? count : 0);
    const rsrc_t gu_in = input_range(a.grad_updated, has_gu ? base : 0, has_gu ? count : 0);
    const rsrc_t mask_in = input_range(a.mask, a.dropout ? row * (hidden / 32) : 0,
                                       a.dropout ? count / 32 : 0);
    const rsrc_t weight_in = input_range(a.weight, 0, hidden);
    const float mean = means[row];
    const float rstd = rstds[row];
    uint32_t column[V];
    f32x4 u[V];
    typename Vector4<GY>::type raw_gy[V];
    f32x4 gu[V];
    f32x4 w[V];
    uint32_t bits[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        // What the slab blocks read again is loaded cached, the rest streams.
        column[v] = ((v * parts + part) * kWaveSize + lane) * 4;
        u[v] = input4<float, Aligned, kSingleCachedLoad>(u_in, column[v]);
        raw_gy[v] = input4<GY, Aligned, kSingleCachedLoad>(gy_in, column[v]);
        w[v] = input4<float, Aligned, kSingleCachedLoad>(weight_in, column[v]);
        gu[v] = input4<float, Aligned, kSingleStreamLoad>(gu_in, column[v]);
        bits[v] = __builtin_amdgcn_raw_buffer_load_b32(mask_in, column[v] / 32 * 4, 0,
                                                       kSingleStreamLoad);
    }
    f32x4 gy[V];
    f32x4 xhat[V];
    float q_slots[V];
    float qx_slots[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        gy[v] = widen4<GY>(raw_gy[v]);
        xhat[v] = column[v] < hidden ? (u[v] - mean) * rstd : zero4();
        const f32x4 q = gy[v] * w[v];
        q_slots[v] = sum4(q);
        qx_slots[v] =
            (q.x * xhat[v].x + q.y * xhat[v].y) + (q.z * xhat[v].z + q.w * xhat[v].w);
    }
    const float2 totals = single_pair_sum<V, Path>(
        q_slots, qx_slots, shared + single_shared_first(Path, V, parts, group), parts, part,
        split.order());
    const float mean_q = totals.x * a.inv_hidden;
    const float mean_qx = totals.y * a.inv_hidden;
    const rsrc_t grad_x_out = output_range(a.grad_x, base, count);
    const rsrc_t grad_branch_out = output_range(static_cast<B*>(a.grad_branch), base, count);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        f32x4 g = gu[v];
        if (has_gy) {
            const f32x4 q = gy[v] * w[v];
            g = g + rstd * ((q - mean_q) - xhat[v] * mean_qx);
        }
        output4<Aligned>(grad_x_out, column[v] * 4, g, true);
        if (a.dropout) {
            const uint32_t nibble = bits[v] >> (column[v] % 32);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                g[e] = g[e] * (static_cast<float>((nibble >> e) & 1u) * a.scale);
            }
        }
        output_convert4<B, Aligned>(grad_branch_out, column[v] * sizeof(B), g, true);
    }
}

// Instantiated in rln_single.hip.
int launch_single_forward(const ForwardArgs& a, int64_t hidden, int branch_dtype,
                          int normalized_dtype, bool aligned);
// With kPartials, one group of partials per single_partial_rows rows.
int launch_single_backward(const BackwardArgs& a, int64_t hidden, int branch_dtype,
                           int grad_normalized_dtype, bool aligned);

}  // namespace rln

#endif  // RLN_SINGLE_H
