// Device kernels of the hybrid SpMM / SDDMM path (gfx950) and their launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace trs {

// Residual task: rows [row_begin, row_end) with their entries [nz_begin, nz_end), or, when
// row_end < 0, a piece [nz_begin, nz_end) of row `row_begin` whose sum goes to partial slot
// ~row_end (a split row, finished by the fixup kernel).
struct Task { int32_t row_begin, row_end, nz_begin, nz_end; };

// A split row: C[row] = sum of partial slots slot_list[slot_begin .. slot_begin + slots) in order.
struct Fixup { int32_t row, slot_begin, slots, pad; };

// Rows per multi-row residual task (the task kernel preloads their row pointers into LDS).
constexpr int kTaskRows = 32;
// Split rows with more slots than this are summed by one workgroup each.
// (A Fixup's slot_begin indexes DevicePlan::slot_list, which names the row's partial slots in
// summation order.)
constexpr int kWideFixupSlots = 16;

// XCDs of an MI355X: workgroup i of a launch runs on XCD i mod kXcds (each XCD has its own L2).
constexpr int kXcds = 8;
// XCD whose L2 serves column c's B row in the SpMM column split: a multiplicative hash spreads hot
// and cold columns evenly over the XCDs.
__host__ __device__ inline int xcd_of_column(int32_t c) { return (int)(((uint32_t)c * 2654435761u) >> 29); }

// Entry of lane `lane` in step k of a wave that walks a row from p0 on, 64 entries a step, or the row's last one past
// its end e (entry indexes run to 2^31 - 1, the steps ahead past that: unsigned).
__host__ __device__ inline uint32_t entry_ahead(uint32_t p0, int k, int lane, uint32_t e) {
  const uint32_t q = p0 + (uint32_t)(k * 64 + lane);
  return q < e ? q : e - 1;
}

// SDDMM split rows, merged: out[e] = xbuf[x_src[k_begin + e - e_begin]] for e in [e_begin, e_end),
// at most kMergeTaskEntries indices per task (a multiple of 256).
struct MergeTask { int32_t e_begin, e_end, k_begin, pad; };
constexpr int32_t kMergeTaskEntries = 4096;

// A window handled by the MFMA window kernel: 16 output rows starting at row0 (rows >= m are
// dropped), dense 16x16 fp16 tiles [tile_begin, tile_end), plus that window's residual rows.
struct MfmaWindow { int32_t row0, tile_begin, tile_end, pad; };

struct DevicePlan {
  int32_t m = 0, n = 0;
  int64_t nnz_csr = 0;
  const int32_t* rowptr = nullptr;   // [m + 1] residual CSR (fp16 values)
  const int32_t* col = nullptr;
  const uint16_t* val = nullptr;
  const Task* tasks = nullptr;
  int32_t ntasks = 0;
  const Fixup* fixups = nullptr;      // split rows with <= kWideFixupSlots slots
  int32_t nfixups = 0;
  const Fixup* wfixups = nullptr;     // split rows with more slots
  int32_t nwfixups = 0;
  int32_t partial_slots = 0;
  const MfmaWindow* mwin = nullptr;
  int32_t nmwin = 0;
  const int32_t* tile_cols = nullptr;  // [tiles][16]
  const uint16_t* tile_a = nullptr;    // [tiles][16 rows][16 cols] fp16 (SpMM)
  int32_t ntiles = 0;
  // SpMM 2:4 quads (sptc_sparse): window i owns quads [win_quad[i], win_quad[i + 1]); quad q covers
  // four 16-column tiles, tile b as columns 16 b .. 16 b + 15 (quad_cols[q][64], -1 = none); lane l
  // of v_smfmac_f32_16x16x64_f16 holds row l % 16 of tile l / 16: quad_a[q][l][8] fp16, two values
  // per group of 4 columns, at the 2-bit column positions packed in quad_idx[q][l] (value j at
  // bits 2j .. 2j + 1).
  const int32_t* win_quad = nullptr;
  const int32_t* quad_cols = nullptr;
  const uint16_t* quad_a = nullptr;
  const uint16_t* quad_idx = nullptr;
  int32_t nquads = 0;
  // SDDMM plans: output index of each residual entry (null = identity; see res_off) and, per tile, its first
  // row and the output index of each of its 256 (row, column) slots (-1 = not stored)
  const int32_t* res_pos = nullptr;
  const int32_t* tile_row0 = nullptr;
  const int32_t* tile_pos = nullptr;
  int32_t feature_lanes = 0;   // lanes per residual lane group (0 = automatic)
  int32_t streaming = 0;       // bit 0: non-temporal A-stream loads, bit 1: non-temporal C stores
  int32_t xcd_run = 1;         // consecutive workgroups per XCD run (1 = hardware round robin)
  int32_t stage = 0;           // staged task streams: 0 automatic, -1 never
  int32_t occupancy = 0;       // waves per SIMD for the residual task kernel: 2..8, 0 automatic, -1 uncapped
  int32_t sddmm_unroll = 0;    // SDDMM residual entries in flight per lane group (4, 8; 0 automatic)
  int32_t split_dispatch = 0;  // 1: main part and XCD split part as two launches (profiling)
  int32_t task_nnz = 0;        // entries per packed residual task
  int32_t row_task = 0;        // ... of a large matrix with these rows (see task_sizes)
  int32_t even_rows = 0;       // 1: no row that tasks walk is longer than that
  int32_t task_max = 0;        // most entries of any residual task (packed rows or a piece)
  const int32_t* slot_list = nullptr;   // partial slots of the split rows, in summation order
  // XCD column split: sub-rows (pieces of long rows by column range, laid out range-major in
  // col / val after the main part) with their own tasks, queue x = x_tasks [xq[x], xq[x + 1]) for
  // XCD x; SpMM sub-row j sums into partial slot j
  const Task* x_tasks = nullptr;
  int32_t x_ntasks = 0;
  int32_t x_task_max = 0;
  const int32_t* x_rowptr = nullptr;
  const int32_t* x_pos = nullptr;       // SDDMM: output index of the split part's entries
  const int32_t* x_sub_row = nullptr;   // SDDMM: the row of sub-row j
  // SDDMM plans with a split part also keep the unsplit task list of all rows, used below
  // kSddmmSplitMinK
  const Task* full_tasks = nullptr;
  int32_t nfull_tasks = 0;
  const Task* narrow_tasks = nullptr;  // SDDMM: the unsplit layout in pieces of S entries, for lane
  int32_t nnarrow_tasks = 0;           // groups of <= 8 lanes (none where no row is longer than S)
  int32_t xq[kXcds + 1] = {};
  // set in the view the launcher builds for the split part (see split_view): tasks come from the
  // per-XCD queues, workgroup i taking queue i mod kXcds; rows are sub-rows
  int32_t xcd_queues = 0;
  const int32_t* sub_row = nullptr;
  int32_t res_off = 0;   // res_pos[q - res_off] is entry q's output index
  // Staged hot rows: hot_col is col with every entry of the nhot most used columns renumbered
  // ~rank (rank 0 = most used), hot_rows[rank] that column.  A call copies those B (Y) rows into a
  // dense buffer and the task kernels then read hot_col, gathering a negative id ~rank from the
  // buffer (hot_b, leading dimension hot_ld: set in the launch view only).
  const int32_t* hot_col = nullptr;
  const int32_t* hot_rows = nullptr;
  int32_t nhot = 0;
  const uint16_t* hot_b = nullptr;
  int32_t hot_ld = 0;
  // SDDMM split part written in its own order: with a buffer from the workspace, sub-row entry q
  // (of the x_entries after the main part) writes xbuf[q - nnz_csr], and a merge pass puts the
  // split rows' outputs in place: merge task i covers output indices [e_begin, e_end), whose
  // values sit at xbuf[x_src[k]] (k counts the split rows' entries in output order)
  const int32_t* x_src = nullptr;
  const MergeTask* merge = nullptr;
  int32_t nmerge = 0;
  int64_t x_entries = 0;
  int32_t out_off = 0;   // set in the view that writes xbuf: entry q writes out[q - out_off]
};

// Whether MFMA windows with `in_tiles` entries in their tiles, of `entries` in all, stay on MFMA: their launch, and
// the residual rows of those windows, each walked by one lane group, cost 8 to 25 us a call whatever their number, and
// an entry in a tile saves as little as 17 us a million at K = 32 and 40 at K = 128.  Kept minus dropped, us at K = 32 /
// 64 / 128 / 256: R-MAT 2^14, 216 of 492K entries in tiles 17 / 18 / 24 / 27; blocks added to R-MAT 2^17, 145K of 3.1M
// (4.6%) 20 / 19 / 20 / 19; to ER of 131,072 nodes, 62K of 2.3M (2.7%) 8 / 8 / 7 / 5, 128K of 2.4M (5.4%) 7 / 7 / 5 / 4, 671K
// of 3.0M (23%) -3 / -1 / -14 / -32; of 524,288 nodes, 249K of 9.2M (2.7%) 0 / 2 / -4 / -15, 513K of 9.5M (5.4%) 4 / -2 /
// -11 / -28; of 2^20 nodes, 498K of 18.4M (2.7%) -2 / - / -13 / -.  Block graphs hold 36% and more of theirs.
constexpr int64_t kMinTileShare = 16, kEnoughTileEntries = 1 << 18;
inline bool windows_pay(int64_t in_tiles, int64_t entries) {
  return in_tiles >= kEnoughTileEntries || in_tiles * kMinTileShare >= entries;
}

// Sizes of residual tasks and pieces.
// A plan of fewer entries than this is small: it splits rows over the XCDs from 512 entries on, not 256, and its
// tasks and pieces shrink (see task_sizes).
constexpr int64_t kSmallEntries = 3 << 20;
// ... and of fewer than this, tiny.
constexpr int64_t kTinyEntries = 3 << 18;
// Tasks that tiny and even plans aim at, and the uneven small ones of SpMM.
constexpr int64_t kMinTasks = 16384;
constexpr int64_t kMinTasksUneven = 65536;

struct TaskSizes {
  int32_t task = 0;     // entries per task of packed rows
  int32_t narrow = 0;   // the same in the list of SDDMM lane groups of <= 8 lanes
  int32_t piece = 0;    // longest piece of a row
  int32_t full_task = 0, full_piece = 0;   // both in the unsplit list of an SDDMM plan with a split part
  int32_t row_task = 0;     // automatic entries per task of a large matrix
  bool even = false;        // no row is longer than such a task
};

// Sizes for `entries` residual entries in `nonempty` rows, the longest row that tasks walk being `longest`; split:
// the long rows are cut by XCD; task_opt, piece_opt: sizes that the caller asks for (0 = automatic).
// Entries per task: about four mean rows, 32 .. 128 (MI355X: 32 for a degree-4 mesh, 128 for R-MAT).  Short rows
// want small tasks (more lane groups in flight, fewer row flushes per group), long rows larger ones.
// Small matrices are bound by the longest chain of batches any lane group walks, one memory round trip after
// another, while the chip has lane groups to spare: their tasks hold 16 entries (tiny) or 32, and pieces of long
// rows 32 or 64.  Measured, us per call at K = 32 / 64 / 128, pieces of 32 / 64 / 128 / 256 entries: R-MAT 2^12
// (123K entries) 18 / 17 / 21, 22 / 23 / 28, 29 / 31 / 42; R-MAT 2^14 (491K) 19 / 20 / 26, 22 / 23 / 33, 36 / 38 /
// 52; R-MAT 2^16 (2.0M; tasks of 32) 32 / 43 / 65, 32 / 41 / 57, 42 / 54 / 66; grid of 800^2 nodes with hubs (3.5M)
// 51 / 80 / 191, 47 / 72 / 177, 50 / 71 / 168, 61 / 73 / 177.
// Where no row is longer than a task (even) there is no long chain to shorten: tasks shrink to 16,384 of them (ER of
// 52,861 nodes, 740K entries, K = 16 / 36 / 80 / 128, tasks of 16 10.7 / 20.7 / 25.2 / 30.1, of 45 10.5 / 14.5 / 21.0
// / 26.8; ER of 60,000 nodes, 1.0M, K = 32 / 64 / 128 / 256, of 48 18.3 / 22.5 / 39.8 / 71.8, of 62 20.7 / 26.1 /
// 35.6 / 68.9).
// SDDMM lane groups of 16 lanes take larger tasks than narrower ones (no row is written per task), which walk a list
// of their own: tiny plans 16,384 tasks (R-MAT 2^14, K = 48 / 64, tasks of 16 19.3 / 19.6, of 30 17.1 / 17.6; ER of
// 42,440 nodes, 552K, 19.3 / 19.2, of 33 17.8 / 17.9; not 17 to 19, three batches of 8 where 16 are two: ER of 40,000 nodes,
// 280K, K = 16 8.8, 7.6), small ones 64 (R-MAT 2^16 with 983K entries K = 64 / 128 / 200:
// of 32 25.2 / 41.9 / 82.5, of 64 26.6 / 36.1 / 78.4); K <= 32 those of SpMM, even tiny plans at most 24 (ER of 28,439
// nodes K = 16 / 32, of 16 9.7 / 10.8, 22 8.0 / 8.5, 30 9.6 / 9.9; of 60,000 nodes, 10 a row 12.3 / 14.2, 11.9 / 13.7,
// 11.2 / 14.0, of 45 13.2 / 18.1).  With a split part that is for those who walk whole rows, K < 128; K >=
// 128 take 16 (R-MAT 2^14 K = 128, of 16 22.4, of 28 27.8).  From 393K on the pieces of those who walk whole rows hold
// 64 (R-MAT 2^14 K = 80 / 96 22.3 / 23.0 with 32, 20.1 / 20.6 with 64; R-MAT 2^13, 150K, K = 64 8.7, 12.1).
// Past kSmallEntries pieces of 128 pay where rows are short, and up to 5M entries, or 6M where the long rows are
// split: a piece is a partial slot, written and summed again at every width (SpMM us, K = 16 / 64 / 128 / 200, pieces
// of 128 / 256: R-MAT 2^19 with 4.9M entries, 20 a row 66 / 98 / 155 / 345, 90 / 106 / 168 / 354, with 5.9M, 22 a row 72
// / 111 / 171 / 380, 80 / 106 / 164 / 369; R-MAT 2^17 with 3.2M, 36 a row 43 / 61 / 85 / 160, 47 / 55 / 72 / 150; R-MAT
// 2^18 with 4.4M 63 / 79 / 117 / 237, 54 / 78 / 112 / 231; grid of 900^2 nodes, 4.5M 54 / - / 221 / 493, 60 / - / 232 /
// 497, of 1000^2, 5.5M 66 / 133 / 247 / 598, 63 / 125 / 241 / 575).  The SDDMM writes no slots: 128 to 6M.
inline TaskSizes task_sizes(int64_t entries, int64_t nonempty, int32_t longest, bool spmm, bool split, bool auto_split,
                            int32_t task_opt, int32_t piece_opt) {
  TaskSizes t;
  const double mean = nonempty > 0 ? (double)entries / (double)nonempty : 1.0;
  t.row_task = (int32_t)(4.0 * mean < 32.0 ? 32.0 : 4.0 * mean > 128.0 ? 128.0 : 4.0 * mean);
  t.even = longest <= t.row_task;
  const bool tiny = entries < kTinyEntries, small = entries < kSmallEntries;
  auto at_most = [](int64_t v, int64_t hi) { return (int32_t)(v < hi ? v : hi); };
  t.task = t.narrow = task_opt > 0 ? task_opt : t.row_task;
  if (task_opt <= 0 && small) {
    const int64_t least = tiny ? 16 : 32, uneven = entries / kMinTasksUneven;
    int64_t shared = entries / kMinTasks;
    if (!spmm && shared < 20) shared = 16;
    t.narrow = at_most(t.even && (spmm || tiny) ? (shared > least ? shared : least) : uneven > least ? uneven : least,
                       t.row_task);
    if (!spmm && tiny && t.narrow > 16) t.narrow = t.narrow < 24 ? 16 : 24;
    t.task = spmm ? t.narrow : tiny ? at_most(shared > 16 ? shared : 16, t.row_task) : at_most(64, t.row_task);
  }
  t.full_task = t.task;
  if (task_opt <= 0 && tiny && split && !spmm) t.task = 16;
  // (pieces of 32 only with the automatic split threshold, which they were measured with)
  int32_t piece = tiny && auto_split && (spmm || split || entries < 3 << 17) ? 32 : 64;
  if (!small) {
    const int64_t line = split || !spmm ? 6ll << 20 : 5'000'000;
    piece = entries < line && (!spmm || 3 * t.row_task <= 2 * 128) ? 128 : 256;
  }
  // ... but a longest row of at most two pieces stays whole: the chain it saves is shorter than the fixup launch that
  // cutting it asks for (ER of 4096 nodes, 17 entries a row, longest 40: 9.7 us with no row cut, 13.2 with a few)
  while (piece < 256 && longest <= 2 * piece) piece *= 2;
  if (piece_opt > 0) piece = piece_opt;
  t.piece = piece > t.task ? piece : t.task;
  // (no slots, no fixups to repeat; pieces twice as long where they were shortened: R-MAT 2^16 with 983K entries
  // K = 64 26.6 -> 23.9 us, 2^17 with 2.9M 56.5 -> 52.6)
  t.full_piece = t.piece;
  const int32_t full = tiny ? 64 : 256;
  if (piece_opt <= 0 && t.piece < full && (!tiny || entries >= 3 << 17)) t.full_piece = at_most(2 * t.piece, full);
  if (t.full_piece < t.full_task) t.full_piece = t.full_task;
  return t;
}

// Features per load that stages B rows for the MFMA windows: 16 bytes from K = 17 on, also where the task kernel takes
// 8-byte loads (K = 40 / 50 / 64 on SBM of 250K nodes: 59 / 70 / 56 us, 62 / 74 / 65 with 8-byte loads), but for odd rows
// of about that width (K = 31 / 33 / 41: 57 / 65 / 69, 55 / 62 / 66) and rows of 33 to 48 features on the 8-byte grid only
// (K = 28 / 36 / 44 / 52, SBM of 20,000 nodes 8.8 / 10.4 / 10.5 / 9.7, 9.1 / 9.2 / 9.3 / 10.4).
inline int window_vec(int K) {
  if (K > 16) return (K % 2 != 0 && K > 24 && K <= 64) || (K > 32 && K <= 48 && K % 8 == 4) ? 4 : 8;
  return K > 8 ? 4 : K > 4 ? 2 : 1;
}

// How a width is run: features per lane (16-, 8-, 4- or 2-byte loads) and lanes per group (0: as many as the width
// needs, at most 16 of 16-byte loads).
struct Route { int vec, lanes; };

// SpMM widths K = 132, 140, .. 252, that 4 divides and 8 does not, in one feature pass: two passes of rows off the
// 16-byte grid cost more than the narrower slices save (us, two passes of 16 lanes of 16 bytes / one of 32 / one of
// 64 lanes of 8 bytes: ER of 907,888 nodes K = 132 / 180 / 244 1458 / 1646 / 1935, 854 / 1071 / 1362, 908 / 1132 /
// 1374; ER of 150,000 nodes, 9 a row 126 / 151 / 182, 86 / 105 / 136, 82 / 100 / 127; R-MAT 2^18 with 7.9M entries 309
// / 306 / 358, 263 / 277 / 321, 384 / 384 / 409; grid of 1300^2 nodes 810 / 1025 / 1264, 691 / 811 / 1013, 726 / 800
// / 917).
// The staged rows serve passes of 16 lanes only.
inline bool spmm_one_pass(int K) { return K > 128 && K <= 256 && K % 4 == 0 && K % 8 != 0; }
// 8-byte loads serve those widths, and K = 100 .. 124, where rows are short and nothing is staged, but for the
// smallest plans (K = 100 / 124, 16 lanes of 16 bytes / 32 of 8: ER of 349,663 nodes, 11 a row 191 / 222, 185 / 218; of
// 80,000 nodes, 9 a row 38.4 / 44.2, 34.7 / 40.3; grid of 1300^2 nodes 454 / 545, 450 / 510; longer rows lose, ER of
// 142,496 nodes, 17 a row 102 / 121, 105 / 124).
inline bool unstaged(const DevicePlan& p) { return p.x_ntasks == 0 && p.nhot == 0; }
// Uneven rows from 786K entries on only (grid of 300^2 nodes with hubs, 495K entries, K = 132 / 244, 32 lanes / 64: 39.6
// / 54.1, 42.7 / 56.5).
inline bool short_rows(const DevicePlan& p) {
  return p.row_task < 64 && unstaged(p) && p.nnz_csr >= (p.even_rows ? 1 << 17 : kTinyEntries);
}

// Even rows, none of them cut into pieces.
inline bool uncut(const DevicePlan& p) { return p.even_rows && p.nfixups + p.nwfixups == 0 && p.x_ntasks == 0; }
// Short rows and a few long ones that are cut into pieces.
inline bool mesh(const DevicePlan& p) { return p.row_task <= 32 && p.nfixups + p.nwfixups > 0 && p.x_ntasks == 0; }

// The route of an SpMM (aligned: rows of B on the 16-byte grid).
// wide loads only where they leave at least 4 lanes per group (whose column/value loads are
// shared): with K <= 8 one or two lanes would stream a task alone (R-MAT K=8: 0.545 ms with one
// 16-byte load per entry, 0.348 with two lanes of 8-byte loads, 0.283 with eight lanes of 2-byte
// loads, 0.273 with four lanes of 4-byte loads (below); K=4 0.515 -> 0.220), and K=16 runs best
// as 4 lanes of 8-byte loads (R-MAT 0.436 ms with 2 lanes of 16-byte loads, 0.324; grid+hubs
// 0.368 -> 0.307)
// Load width by K alone: a row of any alignment is read with whole vectors (see half8_u), the last
// lane taking the row's last VEC features.  16-byte loads from K = 17 on, where 3 lanes of a group
// have work (K = 16 is faster as 4 lanes of 8 bytes: R-MAT 2^20 0.436 -> 0.324 ms, and K = 8 as 4
// lanes of 4 bytes: 0.545 -> 0.273; K = 4 as 4 lanes of 2 bytes: 0.233 -> 0.219).  With narrower
// loads for the widths that 8, 4 or 2 do not divide, and 2-byte ones for odd ones, R-MAT 2^20 took
// (us, narrow -> this): K = 5 310 -> 244, 7 336 -> 262, 13 348 -> 289, 17 580 -> 379, 18 385 ->
// 312, 28 460 -> 371, 31 643 -> 458, 65 1755 -> 643, 97 2198 -> 724, 100 942 -> 661, 127 2425 -> 814,
// 130 2122 -> 1333, 255 4436 -> 1618; SBM 250K nodes K = 17 76 -> 43, 65 169 -> 95, 127 240 -> 132.
// K = 33..64 take 8-byte loads in 16-lane groups, whose staged stream holds more entries in flight than
// 8-lane groups of 16-byte loads held to 2 waves (us, 16-byte / 8-byte, in batches of 8): R-MAT 2^20 K =
// 33 595 / 442, 41 622 / 453, 48 507 / 372, 64 457 / 376; R-MAT 2^18 K = 40 / 48 / 56 / 64 120 / 120 / 127 / 112,
// 110 / 110 / 115 / 109; R-MAT 2^14 K = 64 20.4 / 18.7; ER of 274K nodes K = 40 69.8 / 66.5; grid of 4M nodes
// with hubs K = 64 587 / 564.  On the 16-byte grid the 16-byte loads stay for a mesh whose pieces of a few hub rows are
// far longer than its packed tasks, up to 200 MB of B (K = 40 / 48 / 64, 16-byte / 8-byte: grid of 300^2 nodes, 495K
// entries 17.1 / 17.6 / 17.6, 19.4 / 19.2 / 19.9, of 640K nodes 73 / 74 / 71, 79 / 85 / 85; of 1300^2 nodes K = 48 / 64,
// 162 / 216 MB 200 / 233, 225 / 217; of 145^2 nodes, 115K entries, K = 48 / 64 16.2 / 16.5, 15.6 / 15.8).
// K = 5 and 7 stay on 8 lanes of 2 bytes over short rows (grid of 2M nodes K = 7: 109 us, 127 with 4-byte
// loads; R-MAT, whose tasks are long, 336 / 262)
inline Route spmm_route(const DevicePlan& p, int K, bool aligned) {
  const bool any_lanes = p.feature_lanes <= 0;   // (a plan may ask for fewer lanes)
  if (any_lanes && K > 8 && K <= 32 && uncut(p)) {
    // Rows of one length, none cut: past 2 MB of B (half an XCD's L2) the gathers miss and no hot rows serve them,
    // which the many lanes and uncapped waves of narrow loads in 16-lane groups with a staged stream stand best (us,
    // K = 9 / 16 / 18 / 24 / 31, 4-lane groups of 8 (K <= 16) or 16 bytes / this: ER of 142,496 nodes 35.9 / 37.7 / 43.2
    // / 47.3 / 62.5, 31.7 / 29.6 / 35.3 / 34.6 / 46.5; of 907,888 nodes 308 / 297 / 361 / 363 / 447, 256 / 255 / 324 / 332
    // / 407).  Below, and in tiny plans, 8-lane groups of 8-byte loads for odd widths, and for all in the smallest plans
    // (K = 17 / 24 / 31: ER of 28,439 nodes 12.7 / 9.1 / 12.9, 11.6 / 10.1 / 11.7; of 30,000 nodes, 180K entries 9.7 / 8.0 /
    // 9.8, 7.2 / 6.7 / 7.2).
    if (p.nnz_csr >= kTinyEntries && (int64_t)p.n * K * 2 >= 2'000'000) return {K <= 16 ? 1 : 2, 16};
    if (K > 16 && (K % 2 != 0 || p.nnz_csr < 1 << 18)) return {4, 8};
  }
  if (any_lanes && K > 8 && K <= 32) {
    // The smallest meshes, whose time is the chain of one hub row's pieces and their sum, take narrow loads in 16-lane
    // groups (us, K = 9 / 16 / 17 / 24 / 31, 4-lane groups / this: grid of 120^2 nodes 13.7 / 13.9 / 17.2 / 15.3 / 17.6, 11.8
    // / 11.9 / 12.6 / 12.6 / 13.0; of 200^2, 220K entries 10.9 / 10.6 / 13.5 / 11.8 / 13.7, 10.8 / 10.2 / 11.1 / 10.9 / 11.4;
    // of 250^2, 344K 11.1 / 10.7 / 16.3 / 12.6 / 17.1, 13.3 / 12.2 / 14.1 / 12.8 / 14.6).  Off the 16-byte grid, 8-lane groups
    // of 8-byte loads at odd widths of other tiny ones, and where B is past all L2s (32 MB) and within half the MALL
    // (K = 17 / 28 / 31, 16 bytes / 8: 250^2 16.3 / 13.1 / 17.1, 13.6 / 12.8 / 13.6; 1300^2 169 / 187 / 227, 160 / 172 / 196;
    // 800^2, K = 18 / 22 / 28, 23 / 28 / 36 MB 51 / 57 / 64, 56 / 59 / 62; 2048^2, K = 17 / 20 / 28, 143 .. 235 MB 405 / 381 /
    // 465, 450 / 434 / 508).
    if (mesh(p) && p.nnz_csr < 1 << 18) return {K <= 16 ? 1 : 2, 16};
    const int64_t bytes = (int64_t)p.n * K * 2;
    if (K > 16 && mesh(p) && ((K % 2 != 0 && p.nnz_csr < kTinyEntries) || (K % 8 != 0 && bytes >= 32 << 20 && bytes < 128 << 20)))
      return {4, 8};
    // Tiny plans with split rows are chains of few batches: more lanes with narrower loads (K = 17 / 24 / 32: R-MAT 2^14
    // 22.1 / 19.9 / 20.0, 18.8 / 17.4 / 17.4; R-MAT 2^16 with 614K entries 28.8 / 24.8 / 24.8, 23.2 / 22.8 / 23.1).
    if (K > 16 && p.x_ntasks > 0 && p.nnz_csr < kTinyEntries) return {4, 8};
  }
  if (K <= 8) return {K > 4 && (K % 2 == 0 || p.task_nnz >= 64) ? 2 : 1, 0};
  if (K <= 16) return {4, 0};
  if (K <= 32) return {8, 0};
  if (K <= 64) {
    const bool hub_pieces = mesh(p) && p.nnz_csr >= 1 << 18 && (int64_t)p.n * K * 2 < 200'000'000;
    return {aligned && K % 8 == 0 && hub_pieces ? 8 : 4, 0};
  }
  if (any_lanes && K % 4 == 0 && K % 8 != 0) {
    if (K > 96 && K <= 128 && short_rows(p)) return {4, 32};
    // (past 256 features passes of 256, where nothing is staged: ER of 150,000 nodes K = 300 / 388 231 / 292 us in passes of
    // 128, 203 / 233)
    if (spmm_one_pass(K) || (K > 256 && unstaged(p))) return short_rows(p) ? Route{4, 64} : Route{8, 32};
  }
  return {8, 0};
}

// The route of an SDDMM.
// K <= 8 takes 2-byte loads so that K lanes share a task (R-MAT K=8: 0.747 ms with one lane of
// 16-byte loads per task, 0.331), and up to K=64 8-byte loads are faster than 16-byte ones
// (same-box A/B on R-MAT: K=32 0.468 -> 0.430 ms, K=64 0.550 -> 0.503; K=128 1.038 vs 1.080
// with 8-byte loads, so 16-byte loads from K=72 on)
// Load width by K alone, as in launch_spmm: 8 lanes of 2 bytes to K = 8 and of 4 bytes to K = 16
// (outputs in 32-byte runs; R-MAT 2^20 K = 16 0.418 -> 0.334 ms, K = 12 0.408 -> 0.287), 8-byte loads
// to K = 64 (K = 32 0.468 -> 0.430 against 16-byte loads, K = 64 0.550 -> 0.503; K = 33 598 / 605 us, 52
// 477 / 582), 16-byte loads above.  With narrower loads for the widths that the vector does not
// divide the pattern took (us, narrow -> this): K = 9 393 -> 293, 13 396 -> 303, 17 706 -> 356, 31 712 ->
// 404, 33 702 -> 508, 63 1447 -> 567, 65 1173 -> 724, 97 2003 -> 779, 98 1508 -> 753, 100 905 -> 753,
// 127 2058 -> 944, 130 1657 -> 1484, 255 3692 -> 1809.
// Even rows take narrower loads in more lanes where the gathers miss: 2-byte loads in 16 lanes at K = 9 .. 16 past 12 MB of
// Y, 4-byte ones at K = 17 .. 32 past 6 MB (us, 8 lanes of 4 or 8 bytes / this: ER of 907,888 nodes K = 9 / 15 / 18 / 24 / 32
// 321 / 376 / 378 / 404 / 352, 290 / 340 / 355 / 370 / 323; of 200,000 nodes K = 18 / 24 / 31 70 / 70 / 88, 65 / 67 / 80; of
// 500,000 nodes K = 9 / 15, 9 / 15 MB 92 / 106, 97 / 103; of 142,496 nodes K = 18 / 22, 5.1 / 6.3 MB 44 / 47, 45 / 47), and 8-byte
// ones in 32 lanes at K = 100 .. 124, which need no masks of a ragged tail, but for tiny plans (ER of 907,888 nodes K = 108
// 765 / 737, of 349,663 K = 124 212 / 205, of 60,000 46.1 / 46.7, of 28,439 23.4 / 24.9).
inline Route sddmm_route(const DevicePlan& p, int K) {
  const int64_t bytes = (int64_t)p.n * K * 2;
  const bool even = p.even_rows && p.x_ntasks == 0 && p.feature_lanes <= 0;
  if (K <= 8) return {1, 0};
  if (K <= 16) return even && bytes >= 12'000'000 ? Route{1, 16} : Route{2, 0};
  if (K <= 32) return even && p.nnz_csr >= kTinyEntries && bytes >= 6'000'000 ? Route{2, 16} : Route{4, 0};
  if (K <= 64) return {4, 0};
  return even && p.nnz_csr >= kTinyEntries && K > 96 && K <= 128 && K % 8 == 4 ? Route{4, 32} : Route{8, 0};
}

// Hot-row staging applies to 16-byte gathers of at least this many features (one 16-lane group,
// 256-byte rows: R-MAT 2^20 K = 128 -6%, K = 256 -5%; K = 32 and 64 unchanged or slower).
constexpr int kHotMinK = 128;
// The SDDMM split part writes its own buffer (then merged) from this width on.
constexpr int kSddmmMergeMinK = 128;
// Bytes of that buffer for plan p at width K (0: the plan has no split part, or K is narrower).
inline int64_t merge_buffer_bytes(const DevicePlan& p, int K) {
  return p.nmerge > 0 && K >= kSddmmMergeMinK ? p.x_entries * 4 : 0;
}
// Widths that 8 does not divide stage their hot rows padded to whole cache lines, so that most gathers
// are aligned again.  A staged row pays where an unaligned one is dear: odd widths (rows off the
// 4-byte grid) from the first 16-lane width on, even ones where a row spans three lines, and the
// SDDMM, which waits on its reductions besides, only near 256 bytes.  R-MAT 2^20, unstaged -> staged:
// SpMM K = 65 684 -> 643 us, 81 859 -> 805, 127 1156 -> 817, 100 661 -> 644, 110 734 -> 684 (2^18
// nodes: 65 187 -> 175, 127 224 -> 192, 100 151 -> 157: the copy's own 5 us); SDDMM K = 101 802 ->
// 815, 107 839 -> 828, 121 900 -> 856, 127 1544 -> 945 (2^18: 101 190 -> 201, 121 196 -> 203, 127
// 259 -> 206).
inline bool stages_hot_rows(int K, bool sddmm) {
  if (K % 8 == 0) return K >= kHotMinK;
  return K >= (sddmm ? 121 : K % 2 != 0 ? 65 : 104);
}
// SDDMM K = 129..256 in one pass of 32 lanes where no long rows' columns are there to be read again from the L2s (no
// split part, no staged rows), or the Y rows come from the caches anyway: the pass saves a launch, a walk of the
// entries and the outputs' read and write (us, two passes / one: ER of 907,888 nodes K = 132 / 180 / 256 1283 / 1461 / 1235,
// 871 / 1055 / 1137; of 150,000 nodes K = 228 159 / 116; grid of 1300^2 nodes K = 130 / 244 / 256 696 / 1041 / 765, 556 / 744 /
// 706; SBM of 250,000 nodes K = 180 286 / 207; ER of 6558 nodes K = 256 16.5 / 7.2; R-MAT 2^14 K = 200 47 / 36, 2^16 K = 200
// / 256 123 / 99, 108 / 99, 2^18 400 / 331, 357 / 357).  Rows off the 16-byte grid gain from the staged rows of two passes
// sooner: even widths to 64 MB of Y (R-MAT 2^17 K = 222 174 / 149, 2^18 K = 130 308 / 344), odd ones to 16 MB (R-MAT 2^14 K =
// 145 45 / 44, 2^16 109 / 117).  The staged rows serve two passes only.
inline bool sddmm_one_pass(const DevicePlan& p, int K) {
  if (K <= 128 || K > 256 || p.feature_lanes > 0) return false;
  return unstaged(p) || (int64_t)p.n * K * 2 <= (int64_t)(K % 8 == 0 ? 128 : K % 2 == 0 ? 64 : 16) << 20;
}
inline int hot_row_stride(int K) { return K % 8 == 0 ? K : (K + 63) / 64 * 64; }
// Bytes of the staged-row buffer of plan p at width K (0 when the plan or K does not stage).
inline int64_t hot_buffer_bytes(const DevicePlan& p, int K, bool sddmm) {
  if (p.nhot <= 0 || !stages_hot_rows(K, sddmm)) return 0;
  if (!sddmm && p.feature_lanes <= 0 && spmm_one_pass(K)) return 0;
  // (K = 121 .. 127: the copy and the renumbered walk pay once Y is past the L2s' reach, 48 MB: unstaged -> staged, R-MAT
  // 2^16 with 614K entries K = 124 / 127 26 -> 31, 28 -> 32; 2^17, 33 MB, 84 -> 95, 90 -> 98; 2^18, 66 MB, K = 127 143 -> 123)
  if (sddmm && K % 8 != 0 && K <= 128 && (int64_t)p.n * K * 2 < 48 << 20) return 0;
  return (int64_t)p.nhot * hot_row_stride(K) * 2;
}
// Column histogram of col[0, total) into counts[n] (ids outside [0, n) are skipped), counted in
// `copies` histograms counts[k * n .. (k + 1) * n) and summed into the first (all zeroed by the caller,
// unless counts_in_lds(n): then every counter is written); and the renumbering hot_col[e] = rank[col[e]] >= 0 ? ~rank[col[e]] : col[e].
// Up to 32 ranges of kCountSpan columns are counted in LDS (128 KB a workgroup); the list is read once a
// range, so past that many the global atomics, spread over as many columns, cost less (grid of 4M nodes, 128
// ranges: 23M entries in 293 us with atomics).
constexpr int32_t kCountSpan = 32768;
constexpr int kCountRanges = 32;
inline bool counts_in_lds(int32_t n) { return n <= kCountSpan * kCountRanges; }
// Copies for a list of `total` entries over n columns counted in LDS: a workgroup to every CU, of at least
// 8192 entries each, within a buffer of 1.75 MB, or of 8 copies where that is more (16 past 2^16 columns).  The
// kernel alone would take more copies, but the buffer lives for one plan, and what it costs to get and to give
// back more than that is not won back (us per plan, 73 / 8 copies: ER of 60,000 nodes 1340 / 1016; 120 / 9,
// grid of 223^2 nodes with hubs 1096 / 782, and 280 of the next format build; 128 / 8, R-MAT 2^16 2430 / 2133;
// 32 / 16 / 8, ER of 250,000 nodes 2305 / 2331 / 2657; 2 MB itself is where the steps begin: ER of 16,384 nodes, format,
// plan and product, 32 / 16 copies 2027 / 1282).
inline int lds_count_copies(int64_t total, int32_t n) {
  const int64_t ranges = (n + kCountSpan - 1) / kCountSpan;
  const int64_t held = (int64_t)(7 << 18) / ((int64_t)n * 4), least = n > 1 << 16 ? 16 : 8;
  int64_t copies = held > least ? held : least;
  if (copies > 256 / ranges) copies = 256 / ranges;
  const int64_t fit = total / 8192;
  if (copies > fit) copies = fit;
  return (int)(copies < 1 ? 1 : copies);
}
hipError_t launch_count_columns(const int32_t* col, int64_t total, int32_t n, int32_t* counts, int copies,
                                hipStream_t stream);
hipError_t launch_renumber_hot(const int32_t* col, int64_t total, int32_t n, const int32_t* rank, int32_t* hot_col,
                               hipStream_t stream);
// counts[col[e]] -= 1 for the residual entries e of the nmwin MFMA windows' rows (rowptr [m + 1]):
// the window kernel reads those through the plain ids, so they do not count towards staging.
hipError_t launch_uncount_windows(const MfmaWindow* mwin, int32_t nmwin, int32_t m, const int32_t* rowptr,
                                  const int32_t* col, int32_t n, int32_t* counts, hipStream_t stream);

// SDDMM runs a plan's split part from this feature width on (narrower rows measured faster
// unsplit).
constexpr int kSddmmSplitMinK = 128;

// Device-side plan lowering (the residual of a plan built from the input CSR the format keeps).
// A dense tile's stored entries: rows row0 + r (r < 16), columns cols[k]; bit (r % 4) * 16 + k of
// present[r / 4] marks entry (r, k).
struct TileEntries { int32_t row0; int32_t cols[16]; int32_t pad[3]; uint64_t present[4]; };
// Byte e of the flag words (little-endian) = 1 for every CSR entry e (rows < m, columns ascending)
// that a tile stores; *marked (zeroed by the caller) counts the entries flagged, each once.
// tile_pos (optional, SDDMM): tile_pos[t * 256 + r * 16 + k] = CSR index of stored entry (r, k).
hipError_t launch_mark_tile_entries(const TileEntries* tiles, int32_t ntiles, int32_t m, const int32_t* rowptr,
                                    const int32_t* col, uint32_t* flag_words, uint32_t* marked, int32_t* tile_pos,
                                    hipStream_t stream);
// Entries of CSR rows [0, m) into the plan's entry arrays.  Row r with split_index[r] = i >= 0 is
// scattered by the XCD of each column to cursor[i * kXcds + x] onward (column order kept), with
// x_pos[position - x_base] = CSR index when x_pos is set; compact (SpMM) plans store such a row
// only there.  Every other row -- and in a non-compact (SDDMM) plan every row -- goes, without its
// flagged entries (flag may be null), to main_rowptr[r] onward, with res_pos[position] = CSR index
// when res_pos is set.  Values (val_out set) are rounded to fp16.
struct PlaceEntries {
  int32_t m = 0;
  const int32_t* rowptr = nullptr;
  const int32_t* col = nullptr;
  const float* val = nullptr;
  const uint8_t* flag = nullptr;
  const int32_t* main_rowptr = nullptr;
  const int32_t* split_index = nullptr;
  const int32_t* cursor = nullptr;
  int32_t* col_out = nullptr;
  uint16_t* val_out = nullptr;
  int32_t* res_pos = nullptr;
  int32_t* x_pos = nullptr;
  int64_t x_base = 0;
  int32_t compact = 1;
  // SDDMM: x_src[merge_off[split_index] + offset in the row] = position - x_base (when x_src set)
  const int32_t* merge_off = nullptr;
  int32_t* x_src = nullptr;
};
hipError_t launch_place_entries(const PlaceEntries& a, hipStream_t stream);

// Plans from a device-resident format (trs_dformat): what the host lowering reads of the input
// CSR's columns, computed where they are.
// *first_bad (the caller sets it to ~0ull) = the lowest index e with col[e] outside [0, n).
hipError_t launch_check_columns(const int32_t* col, int64_t total, int32_t n, unsigned long long* first_bad,
                                hipStream_t stream);
// Chunk i of the split-row candidates, entries col[start[i] .. start[i] + len[i]) of candidate
// row[i]: cnt[row[i] * kXcds + x] += its entries of XCD class x (xcd_of_column; cnt zeroed by the
// caller); with seen (n bytes, zeroed by the caller, 4-byte padded) seen[c] = 1 for its columns.
hipError_t launch_split_stats(const int32_t* col, const int32_t* start, const int32_t* len, const int32_t* row,
                              int32_t chunks, int32_t* cnt, uint8_t* seen, hipStream_t stream);
// *out += the nonzero bytes of flags[0, n) (values 0 or 1, n padded to 4 bytes; *out zeroed by
// the caller).
hipError_t launch_count_flags(const uint8_t* flags, int64_t n, unsigned long long* out, hipStream_t stream);
// 2:4 group tiles of a window-16 format (tiles of four groups per window, block_online.cpp:796-841):
// pass[t] = 1 when the stored values of tile t's groups (s_pos >= 0, 32 per group) are at least
// min_fill * 256, the fill rule of the host lowering.
hipError_t launch_group_tile_fill(const int32_t* tile_win, const int32_t* tile_group, const int32_t* s_offsets,
                                  const int8_t* s_pos, int32_t ntiles, float min_fill, uint8_t* pass,
                                  hipStream_t stream);
// The groups of the listed tiles, packed: GroupTile i holds tile ids[i]'s window row, group count,
// s_columns, s_values and s_pos (window 16).
struct GroupTile { int32_t row0, ngroups; int32_t cols[16]; float val[4][32]; int8_t pos[4][32]; };
hipError_t launch_gather_group_tiles(const int32_t* ids, int32_t nids, const int32_t* tile_win,
                                     const int32_t* tile_group, const int32_t* s_offsets, const int32_t* s_col,
                                     const float* s_val, const int8_t* s_pos, GroupTile* out, hipStream_t stream);

// hot: the staged-row buffer (hot_buffer_bytes(p, K) bytes; null = gather every row from B).
// ev (optional): 4 events recorded before the task kernel (and the hot-row copy) and after each of
// the three kernels.
hipError_t launch_spmm(const DevicePlan& p, const uint16_t* B, int64_t ldb, int K, float* C, int64_t ldc,
                       float* partial, uint16_t* hot, hipStream_t stream, hipEvent_t* ev = nullptr);
// The plan's MFMA windows (a part of launch_spmm).
void launch_spmm_windows(const DevicePlan& p, const uint16_t* B, int64_t ldb, int K, float* C, int64_t ldc,
                         hipStream_t stream);
// out[0, n) = 0 with a kernel (not a memset node: callers may capture the stream in a graph).
hipError_t launch_zero_fill(float* out, int64_t n, hipStream_t stream);
// hot: as for launch_spmm, Y rows.  xbuf: the split part's own output buffer
// (merge_buffer_bytes(p, K) bytes; null = the split part writes its outputs in place).  ev
// (optional): 3 events recorded before the residual kernels (and the hot-row copy) and after them
// (and the merge), and after the tile kernel.
hipError_t launch_sddmm(const DevicePlan& p, const uint16_t* X, int64_t ldx, const uint16_t* Y, int64_t ldy,
                        int K, float* out, uint16_t* hot, float* xbuf, hipStream_t stream,
                        hipEvent_t* ev = nullptr);

}  // namespace trs
