// The sizes and routes that csrc/kernels.hpp chooses, for tests on the CPU (tests/test_rules.py).
#include "kernels.hpp"

extern "C" {

int32_t rule_lds_count_copies(int64_t total, int32_t n) { return trs::lds_count_copies(total, n); }
// out: task, narrow, piece, full_task, full_piece, row_task, even
void rule_task_sizes(int64_t entries, int64_t nonempty, int32_t longest, int32_t spmm, int32_t split, int32_t task_opt,
                     int32_t piece_opt, int32_t* out) {
  const trs::TaskSizes t = trs::task_sizes(entries, nonempty, longest, spmm != 0, split != 0, true, task_opt, piece_opt);
  const int32_t v[7] = {t.task, t.narrow, t.piece, t.full_task, t.full_piece, t.row_task, t.even ? 1 : 0};
  for (int i = 0; i < 7; ++i) out[i] = v[i];
}
int32_t rule_counts_in_lds(int32_t n) { return trs::counts_in_lds(n) ? 1 : 0; }

}
