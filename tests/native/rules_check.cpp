// The sizes and routes that csrc/kernels.hpp chooses, for tests on the CPU (tests/test_rules.py).
#include "kernels.hpp"

extern "C" {

int32_t rule_lds_count_copies(int64_t total, int32_t n) { return trs::lds_count_copies(total, n); }
int32_t rule_counts_in_lds(int32_t n) { return trs::counts_in_lds(n) ? 1 : 0; }

}
