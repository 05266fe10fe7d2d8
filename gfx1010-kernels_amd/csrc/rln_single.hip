// Launchers of the single-step kernels (rln_single.h). Compiled once per
// pass, with -DRLN_PASSES=<1: forward, 2: backward>, in parallel with the
// walking kernels.
#include "rln_single.h"

namespace rln {
namespace {

#if RLN_PASSES & 1
// Calls `launch.template operator()<V, Path>()` for a forward split.
template <typename Launch>
int with_forward_split(const SingleSplit& split, Launch&& launch) {
    if (split.path == SumPath::kLanes) {
        return split.vectors == 1 ? launch.template operator()<1, SumPath::kLanes>()
                                  : launch.template operator()<2, SumPath::kLanes>();
    }
    if (split.path == SumPath::kExchange) {
        return launch.template operator()<2, SumPath::kExchange>();
    }
    return split.vectors == 3 ? launch.template operator()<3, SumPath::kDirect>()
                              : launch.template operator()<4, SumPath::kDirect>();
}
#endif

#if RLN_PASSES & 2
// The same for a backward split.
template <typename Launch>
int with_backward_split(const SingleSplit& split, Launch&& launch) {
    if (split.path == SumPath::kExchange) {
        return launch.template operator()<1, SumPath::kExchange>();
    }
    switch (split.vectors) {
        case 1: return launch.template operator()<1, SumPath::kDirect>();
        case 2: return launch.template operator()<2, SumPath::kDirect>();
        case 3: return launch.template operator()<3, SumPath::kDirect>();
        default: return launch.template operator()<4, SumPath::kDirect>();
    }
}
#endif

}  // namespace

#if RLN_PASSES & 1
int launch_single_forward(const ForwardArgs& f, int64_t hidden, int branch_dtype,
                          int normalized_dtype, bool aligned) {
    const SingleSplit split = single_split<Pass::kForward>(hidden, f.rows);
    SingleForwardArgs a{};
    a.threshold = f.threshold;
    a.scale = f.scale;
    a.weight = f.weight;
    a.bias = f.bias;
    a.updated = f.updated;
    a.normalized = f.normalized;
    a.mask = f.mask;
    a.mean = f.mean;
    a.rstd = f.rstd;
    a.inv_hidden = 1.0f / static_cast<float>(hidden);
    a.eps = f.eps;
    a.zero_weight = f.zero_weight;
    a.zero_bias = f.zero_bias;
    // A pointer argument either way: the kernel then knows the address space.
    const int64_t* const seed = f.philox.seed_ptr
        ? f.philox.seed_ptr : reinterpret_cast<const int64_t*>(f.philox.seed);
    const dim3 grid(static_cast<unsigned>((f.rows + split.groups - 1) / split.groups));
    const int threads = split.threads();
    return with_dtype(branch_dtype, [&]<typename B>() {
        return with_dtype(normalized_dtype, [&]<typename N>() {
            return with_forward_split(split, [&]<int V, SumPath Path>() {
                const auto kernel = aligned ? &rln_single_forward_kernel<V, Path, B, N, true>
                                            : &rln_single_forward_kernel<V, Path, B, N, false>;
                kernel<<<grid, threads, 0, f.stream>>>(
                    f.x, static_cast<const B*>(f.branch), static_cast<int>(f.rows),
                    static_cast<uint32_t>(hidden), SplitWord::of(split),
                    DropWord::of(f.dropout, f.philox), seed, f.philox.offset,
                    f.philox.offset_ptr, a);
                return check_launch("rln_single_forward_kernel");
            });
        });
    });
}
#endif

#if RLN_PASSES & 2
int launch_single_backward(const BackwardArgs& f, int64_t hidden, int branch_dtype,
                           int grad_normalized_dtype, bool aligned) {
    const SingleSplit split = single_split<Pass::kBackward>(hidden, f.rows);
    const int chunk_rows = static_cast<int>((f.flags & kPartials)
        ? single_partial_rows(f.rows, hidden, split) : single_chunk_rows(f.rows, split));
    SingleBackwardArgs a{};
    a.row_blocks = (chunk_rows + split.groups - 1) / split.groups;
    a.slabs = split.waves() >= 8 ? 2 : 1;
    a.slab_waves = split.waves() / a.slabs;
    a.dropout = (f.flags & kDropout) ? 1 : 0;
    a.grad_updated = f.grad_updated;
    a.mask = f.mask;
    a.weight = f.weight;
    a.grad_x = f.grad_x;
    a.grad_branch = f.grad_branch;
    a.inv_hidden = 1.0f / static_cast<float>(hidden);
    a.scale = f.scale;
    a.grad_weight = f.grad_weight;
    a.grad_bias = f.grad_bias;
    a.partials = (f.flags & kPartials) ? f.partials : nullptr;
    const int64_t slab_columns = static_cast<int64_t>(a.slabs) * kSlabColumns;
    const int64_t slab_blocks =
        (f.flags & kParameters) ? (hidden + slab_columns - 1) / slab_columns : 0;
    const int64_t chunks = (f.rows + chunk_rows - 1) / chunk_rows;
    const dim3 grid(static_cast<unsigned>(8 * (a.row_blocks + slab_blocks)),
                    static_cast<unsigned>((chunks + 7) / 8));
    const int threads = split.threads();
    return with_dtype(branch_dtype, [&]<typename B>() {
        return with_dtype(grad_normalized_dtype, [&]<typename GY>() {
            return with_backward_split(split, [&]<int V, SumPath Path>() {
                const auto kernel = aligned ? &rln_single_backward_kernel<V, Path, B, GY, true>
                                            : &rln_single_backward_kernel<V, Path, B, GY, false>;
                kernel<<<grid, threads, 0, f.stream>>>(
                    f.updated, static_cast<const GY*>(f.grad_normalized), f.mean, f.rstd,
                    static_cast<int>(f.rows), static_cast<uint32_t>(hidden), SplitWord::of(split),
                    chunk_rows, a);
                return check_launch("rln_single_backward_kernel");
            });
        });
    });
}
#endif

}  // namespace rln
