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
//    so a lane holds 36-90 VGPRs, 5-8 waves fit a SIMD, and rows spread over
//    every CU; row sums cross the waves in LDS, in the walking shape's order,
//    so both kernels give a row the same bits;
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
// waves ([64, 4096] without dropout 4.3 us either way).
template <Pass kPass>
SingleSplit single_split(int64_t hidden, int64_t rows) {
    SingleSplit s{};
    s.order = sum_order<kPass>(hidden, rows);
    if (hidden > 2048) {
        s.path = SumPath::kDirect;
        s.vectors = s.order.vectors;
        s.parts = s.order.parts;
    } else {
        s.vectors = hidden <= 256 ? 1 : 2;
        const int64_t per_wave = 4 * kWaveSize * s.vectors;
        s.parts = static_cast<int>((hidden + per_wave - 1) / per_wave);
        s.path = s.parts == 1 ? SumPath::kLanes : SumPath::kExchange;
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
// 5.0 -> 4.7 us, [32, 8192] 5.3 -> 5.6; with dropout [128, 8192] 7.2 -> 6.7).
inline bool single_forward(int64_t rows, int64_t hidden, bool dropout) {
    const int64_t elements = rows * hidden;
    if (hidden > 4096 && !dropout) {
        return elements <= (1 << 17);
    }
    return rows <= 6144 && elements <= (hidden <= 1280 ? 1 << 21 : 1 << 20);
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

struct SingleForwardArgs {
    const float* x;
    const void* branch;
    const float* weight;
    const float* bias;
    float* updated;
    void* normalized;
    float* mean;
    float* rstd;
    uint32_t* mask;
    float* zero_weight;
    float* zero_bias;
    int64_t rows;
    int hidden;
    int parts;
    int groups;
    int reciprocal;
    float inv_hidden;  // 1.0f / hidden, rounded once on the host
    float eps;
    int dropout;
    float scale;
    uint32_t threshold;
    SumOrder order;
    PhiloxArgs philox;
};

// One row per team of `parts` waves; slot v of lane l of part p holds columns
// 4 * ((v * parts + p) * 64 + l) .. + 3.
template <int V, SumPath Path, typename B, typename N, bool Aligned>
__global__ __launch_bounds__(kSingleMaxWaves * kWaveSize)
void rln_single_forward_kernel(SingleForwardArgs a) {
    // [0] the mean's sum, [1] the variance's: one float per wave of the row
    // (direct), or one per vector of the block's rows (exchange, at most four
    // waves).
    constexpr int kShared = Path == SumPath::kExchange ? V * 4 * kWaveSize : kSingleMaxParts;
    __shared__ float shared[2][kShared];
    // Keep bits of the reference's stream, 64 columns each (at most 1024
    // columns, so at most 16 per row, and at most four rows per block).
    __shared__ uint64_t keep[4][16];
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    const int group = (wave * a.reciprocal) >> 8;
    const int part = wave - group * a.parts;
    const uint32_t hidden = a.hidden;
    // A team past the last row reads and writes nothing (empty descriptors),
    // but meets its block's barriers.
    const int64_t team_row = static_cast<int64_t>(blockIdx.x) * a.groups + group;
    const bool valid = team_row < a.rows;
    const int64_t row = valid ? team_row : 0;
    const int64_t count = valid ? hidden : 0;
    const int64_t base = row * hidden;
    const int row_shared = Path == SumPath::kExchange ? group * V * a.parts * kWaveSize : 0;

    // The Philox key and position first: the draws hang on them, and under
    // graph capture they come from memory.
    uint32_t key0 = 0;
    uint32_t key1 = 0;
    uint64_t position = 0;
    if (a.dropout) {
        const uint64_t seed = a.philox.seed_ptr ? static_cast<uint64_t>(*a.philox.seed_ptr)
                                                : a.philox.seed;
        const uint64_t offset = a.philox.offset
            + (a.philox.offset_ptr ? static_cast<uint64_t>(*a.philox.offset_ptr) : 0);
        key0 = static_cast<uint32_t>(seed);
        key1 = static_cast<uint32_t>(seed >> 32);
        position = offset / 4;
    }
    uint32_t column[V];
    f32x4 x[V];
    typename Vector4<B>::type branch[V];
    f32x4 w[V];
    f32x4 b[V];
    const rsrc_t x_in = input_range(a.x, base, count);
    const rsrc_t branch_in = input_range(static_cast<const B*>(a.branch), base, count);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        column[v] = ((v * a.parts + part) * kWaveSize + lane) * 4;
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
    if (a.dropout && a.philox.threads != 0) {
        // The reference's stream: thread t of the row draws `calls` Philox
        // blocks, value `item` of which decides column t + item * threads.
        // 64 consecutive threads and one call are a unit; a ballot over value
        // e of a unit covers 64 consecutive columns, two words of the mask.
        const int threads = a.philox.threads;
        const int per_item = threads / kWaveSize;
        const int items = (a.hidden + threads - 1) / threads;
        const int calls = (items + 3) / 4;  // 1 or 2
        const int chunks = a.hidden / kWaveSize;
        for (int unit = part; unit < per_item * calls; unit += a.parts) {
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
        row_handoff(a.parts);
        const uint32_t* const words = reinterpret_cast<const uint32_t*>(keep[group]);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            bits[v] = column[v] < hidden ? words[column[v] / 32] >> (column[v] % 32) : 0u;
        }
        if (part == 0 && lane < a.hidden / 32) {
            output_b32(output_range(a.mask, row * (hidden / 32), count / 32), lane * 4,
                       words[lane], true);
        }
    } else if (a.dropout) {
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
        if (a.dropout) {
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
    const float mean = single_sum<V, Path>(slots, &shared[0][row_shared], a.parts, part,
                                             a.order) * a.inv_hidden;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        u[v] = column[v] < hidden ? u[v] - mean : zero4();
        slots[v] = (u[v].x * u[v].x + u[v].y * u[v].y) + (u[v].z * u[v].z + u[v].w * u[v].w);
    }
    const float variance = single_sum<V, Path>(slots, &shared[1][row_shared], a.parts, part,
                                                 a.order) * a.inv_hidden;
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

// Instantiated in rln_single.hip.
int launch_single_forward(const ForwardArgs& a, int64_t hidden, int branch_dtype,
                          int normalized_dtype, bool aligned);

}  // namespace rln

#endif  // RLN_SINGLE_H
