// Prints what the host rules of the single-step kernels (csrc/rln_single.h)
// decide, for tests/test_single_step_rules.py (test infrastructure). Host code
// only, built with the address and undefined-behaviour sanitizers; nothing
// reaches a device. Each input line is a query and its integers, each output
// line its answer:
//
//   lds PASS ROWS HIDDEN    length of the block's array of row sums, and one
//                           past the last element its rows read (PASS 0:
//                           forward, 1: backward)
//   forward ROWS HIDDEN DROPOUT ALIGNED
//                           1 if a forward runs single-step, and 1 if it writes
//                           through
//   backward ROWS HIDDEN BRANCH GRAD_NORMALIZED FLAGS OVER ALIGNED
//                           1 if a backward with these dtypes and flags
//                           (kHasGradUpdated, ... of rln_device.h) runs
//                           single-step; OVER: what shares its memory, 0 nothing,
//                           1 grad_x and updated, 2 grad_x and grad_normalized,
//                           3 grad_branch and updated, 4 grad_branch and mean
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

#include "rln_single.h"

namespace {

template <rln::Pass kPass>
void lds(int64_t rows, int64_t hidden) {
    const rln::SingleSplit s = rln::single_split<kPass>(hidden, rows);
    const int end = rln::single_shared_first(s.path, s.vectors, s.parts, s.groups - 1)
        + rln::single_shared_read(s.path, s.parts, s.order);
    std::printf("%d %d\n", rln::single_shared_size(s.path, s.vectors), end);
}

void* at(int64_t tebibytes) {
    return reinterpret_cast<void*>(static_cast<uintptr_t>(tebibytes) << 40);
}

bool backward(int64_t rows, int64_t hidden, int branch, int grad_normalized, int flags, int over,
              bool aligned) {
    rln::BackwardArgs a{};
    a.rows = rows;
    a.flags = flags;
    a.grad_updated = static_cast<const float*>((flags & rln::kHasGradUpdated) ? at(1) : nullptr);
    a.grad_normalized = (flags & rln::kHasGradNormalized) ? at(2) : nullptr;
    a.updated = static_cast<const float*>(at(3));
    a.weight = static_cast<const float*>(at(4));
    a.mean = static_cast<const float*>(at(5));
    a.rstd = static_cast<const float*>(at(6));
    a.grad_x = static_cast<float*>(at(over == 1 ? 3 : over == 2 ? 2 : 7));
    a.grad_branch = at(over == 3 ? 3 : over == 4 ? 5 : 8);
    return rln::takes_single_backward(a, hidden, branch, grad_normalized, aligned);
}

}  // namespace

int main() {
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string query;
        in >> query;
        if (query == "lds") {
            int64_t pass = 0, rows = 0, hidden = 0;
            in >> pass >> rows >> hidden;
            pass == 0 ? lds<rln::Pass::kForward>(rows, hidden)
                      : lds<rln::Pass::kBackward>(rows, hidden);
        } else if (query == "backward") {
            int64_t rows = 0, hidden = 0;
            int branch = 0, grad_normalized = 0, flags = 0, over = 0;
            bool aligned = true;
            in >> rows >> hidden >> branch >> grad_normalized >> flags >> over >> aligned;
            std::printf("%d\n",
                        backward(rows, hidden, branch, grad_normalized, flags, over, aligned));
        } else if (query == "forward") {
            int64_t rows = 0, hidden = 0;
            bool dropout = false, aligned = true;
            in >> rows >> hidden >> dropout >> aligned;
            std::printf("%d %d\n", rln::single_forward(rows, hidden, dropout, aligned),
                        rln::forward_write_through(rows, hidden, dropout, aligned));
        } else {
            query.clear();
        }
        if (in.fail() || query.empty()) {
            std::fprintf(stderr, "bad query: %s\n", line.c_str());
            return 1;
        }
    }
    return 0;
}
