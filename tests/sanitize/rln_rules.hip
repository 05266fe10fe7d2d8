// Prints what the host rules of the single-step kernels (csrc/rln_single.h)
// decide, for tests/test_single_step_rules.py (test infrastructure). Host code
// only, built with the address and undefined-behaviour sanitizers; nothing
// reaches a device. Each input line is a query and its integers, each output
// line its answer:
//
//   lds PASS ROWS HIDDEN    length of the block's array of row sums, and one
//                           past the last element its rows read (PASS 0:
//                           forward, 1: backward)
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
        }
        if (in.fail() || query.empty()) {
            std::fprintf(stderr, "bad query: %s\n", line.c_str());
            return 1;
        }
    }
    return 0;
}
