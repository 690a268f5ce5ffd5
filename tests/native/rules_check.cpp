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
// plan fields: entries, columns, rows cut into pieces, split part's tasks, task_nnz, row_task, even_rows, staged rows,
// feature_lanes; out: features per lane, lanes per group (0: as many as the width needs)
static trs::DevicePlan plan_of(const int64_t* f) {
  trs::DevicePlan p;
  p.nnz_csr = f[0];
  p.m = p.n = (int32_t)f[1];
  p.nfixups = (int32_t)f[2];
  p.x_ntasks = (int32_t)f[3];
  p.task_nnz = (int32_t)f[4];
  p.row_task = (int32_t)f[5];
  p.even_rows = (int32_t)f[6];
  p.nhot = (int32_t)f[7];
  p.feature_lanes = (int32_t)f[8];
  return p;
}
void rule_spmm_route(const int64_t* f, int32_t K, int32_t aligned, int32_t* out) {
  const trs::Route r = trs::spmm_route(plan_of(f), K, aligned != 0);
  out[0] = r.vec;
  out[1] = r.lanes;
}
int64_t rule_hot_bytes(const int64_t* f, int32_t K, int32_t sddmm) { return trs::hot_buffer_bytes(plan_of(f), K, sddmm != 0); }
int32_t rule_windows_pay(int64_t in_tiles, int64_t entries) { return trs::windows_pay(in_tiles, entries) ? 1 : 0; }
int32_t rule_sddmm_one_pass(const int64_t* f, int32_t K) { return trs::sddmm_one_pass(plan_of(f), K) ? 1 : 0; }
void rule_sddmm_route(const int64_t* f, int32_t K, int32_t* out) {
  const trs::Route r = trs::sddmm_route(plan_of(f), K);
  out[0] = r.vec;
  out[1] = r.lanes;
}
uint32_t rule_entry_ahead(uint32_t p0, int32_t k, int32_t lane, uint32_t e) { return trs::entry_ahead(p0, k, lane, e); }
int32_t rule_window_vec(int32_t K) { return trs::window_vec(K); }
int32_t rule_counts_in_lds(int32_t n) { return trs::counts_in_lds(n) ? 1 : 0; }

}
