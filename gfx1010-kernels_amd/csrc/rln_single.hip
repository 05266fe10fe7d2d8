// Launchers of the single-step kernels (rln_single.h). Compiled once per
// pass, with -DRLN_PASSES=<1: forward, 2: backward>, in parallel with the
// walking kernels.
#include "rln_single.h"

namespace rln {
namespace {

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

}  // namespace

#if RLN_PASSES & 1
int launch_single_forward(const ForwardArgs& f, int64_t hidden, int branch_dtype,
                          int normalized_dtype, bool aligned) {
    const SingleSplit split = single_split<Pass::kForward>(hidden, f.rows);
    SingleForwardArgs a{};
    a.x = f.x;
    a.branch = f.branch;
    a.weight = f.weight;
    a.bias = f.bias;
    a.updated = f.updated;
    a.normalized = f.normalized;
    a.mean = f.mean;
    a.rstd = f.rstd;
    a.mask = f.mask;
    a.zero_weight = f.zero_weight;
    a.zero_bias = f.zero_bias;
    a.rows = f.rows;
    a.hidden = static_cast<int>(hidden);
    a.parts = split.parts;
    a.groups = split.groups;
    a.reciprocal = split.reciprocal;
    a.inv_hidden = 1.0f / static_cast<float>(hidden);
    a.eps = f.eps;
    a.dropout = f.dropout;
    a.scale = f.scale;
    a.threshold = f.threshold;
    a.order = split.order;
    a.philox = f.philox;
    const dim3 grid(static_cast<unsigned>((f.rows + split.groups - 1) / split.groups));
    const int threads = split.threads();
    return with_dtype(branch_dtype, [&]<typename B>() {
        return with_dtype(normalized_dtype, [&]<typename N>() {
            return with_forward_split(split, [&]<int V, SumPath Path>() {
                if (aligned) {
                    rln_single_forward_kernel<V, Path, B, N, true>
                        <<<grid, threads, 0, f.stream>>>(a);
                } else {
                    rln_single_forward_kernel<V, Path, B, N, false>
                        <<<grid, threads, 0, f.stream>>>(a);
                }
                return check_launch("rln_single_forward_kernel");
            });
        });
    });
}
#endif

}  // namespace rln
