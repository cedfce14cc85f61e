// C-ABI launcher of the persistent shard GEMM (include/iris_amd.h).
#include <cstdio>
#include <cstring>
#include <cstdlib>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "gemm_skinny.hpp"

namespace iris_amd {

namespace {

const GemmKernelEntry* entries_for(int dt, int op, int* count) {
  if (dt == IRIS_DTYPE_BF16) {
    switch (op) {
      case OP_STORE16: return gemm_entries_bf16_store16(count);
      case OP_STORE32: return gemm_entries_bf16_store32(count);
      case OP_ATOMIC32: return gemm_entries_bf16_atomic32(count);
      case OP_ATOMIC16: return gemm_entries_bf16_atomic16(count);
    }
  } else if (dt == IRIS_DTYPE_F16) {
    switch (op) {
      case OP_STORE16: return gemm_entries_f16_store16(count);
      case OP_STORE32: return gemm_entries_f16_store32(count);
      case OP_ATOMIC32: return gemm_entries_f16_atomic32(count);
      case OP_ATOMIC16: return gemm_entries_f16_atomic16(count);
    }
  } else if (dt == IRIS_DTYPE_F32) {
    switch (op) {
      case OP_STORE32: return gemm_entries_f32_store32(count);
      case OP_ATOMIC32: return gemm_entries_f32_atomic32(count);
    }
  }
  *count = 0;
  return nullptr;
}

// Tiles behind the table (`variant` does not number them), in three lists: those for a row-major B, those for operands at any
// alignment, and the fp32 ones for a K of at least LONG_STEPS of their K-steps with the gathering ones.
constexpr int LONG_STEPS = 8;
const GemmKernelEntry* rows_entries_for(int dt, int op, int* count) {
  *count = 0;
  if (dt != IRIS_DTYPE_BF16 && dt != IRIS_DTYPE_F16) return nullptr;
  const bool bf16 = dt == IRIS_DTYPE_BF16;
  switch (op) {
    case OP_STORE16: return bf16 ? gemm_entries_bf16_store16_rows(count) : gemm_entries_f16_store16_rows(count);
    case OP_STORE32: return bf16 ? gemm_entries_bf16_store32_rows(count) : gemm_entries_f16_store32_rows(count);
    case OP_ATOMIC32: return bf16 ? gemm_entries_bf16_atomic32_rows(count) : gemm_entries_f16_atomic32_rows(count);
    case OP_ATOMIC16: return bf16 ? gemm_entries_bf16_atomic16_rows(count) : gemm_entries_f16_atomic16_rows(count);
  }
  return nullptr;
}
const GemmKernelEntry* loose_entries_for(int dt, int op, int* count) {
  *count = 0;
  if (dt != IRIS_DTYPE_BF16 && dt != IRIS_DTYPE_F16) return nullptr;
  const bool bf16 = dt == IRIS_DTYPE_BF16;
  switch (op) {
    case OP_STORE16: return bf16 ? gemm_entries_bf16_store16_loose(count) : gemm_entries_f16_store16_loose(count);
    case OP_STORE32: return bf16 ? gemm_entries_bf16_store32_loose(count) : gemm_entries_f16_store32_loose(count);
    case OP_ATOMIC32: return bf16 ? gemm_entries_bf16_atomic32_loose(count) : gemm_entries_f16_atomic32_loose(count);
    case OP_ATOMIC16: return bf16 ? gemm_entries_bf16_atomic16_loose(count) : gemm_entries_f16_atomic16_loose(count);
  }
  return nullptr;
}
const GemmKernelEntry* more_entries_for(int dt, int op, int* count) {
  *count = 0;
  switch (op) {
    case OP_STORE16:
      return dt == IRIS_DTYPE_BF16 ? gemm_entries_bf16_store16_gather(count) : gemm_entries_f16_store16_gather(count);
    case OP_STORE32:
      return dt == IRIS_DTYPE_F32    ? gemm_entries_f32_store32_long(count)
             : dt == IRIS_DTYPE_BF16 ? gemm_entries_bf16_store32_gather(count)
                                     : gemm_entries_f16_store32_gather(count);
    case OP_ATOMIC32:
      return dt == IRIS_DTYPE_F32    ? gemm_entries_f32_atomic32_long(count)
             : dt == IRIS_DTYPE_BF16 ? gemm_entries_bf16_atomic32_gather(count)
                                     : gemm_entries_f16_atomic32_gather(count);
    case OP_ATOMIC16:
      return dt == IRIS_DTYPE_BF16 ? gemm_entries_bf16_atomic16_gather(count) : gemm_entries_f16_atomic16_gather(count);
  }
  return nullptr;
}

// The plain build (every wave fetches its share) of the tile shape of `e`, an
// entry with fetching waves; null if `e` has none or the list holds no such build.
const GemmKernelEntry* plain_twin(const GemmKernelEntry* list, int count, const GemmKernelEntry& e) {
  if (e.fetch_waves == 0 || !e.dma || e.b_rows || e.loose) return nullptr;
  for (int i = 0; i < count; ++i)
    if (list[i].dma && list[i].fetch_waves == 0 && list[i].cm == e.cm && list[i].cn == e.cn && list[i].wm == e.wm &&
        list[i].wn == e.wn)
      return &list[i];
  return nullptr;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Whether every row of both operands (A's K-contiguous, B's along K or across it) starts on a cache line; strides in 16-bit
// units.
bool whole_lines(const iris_gemm_args& a) {
  return a.stride_am % 64 == 0 && (a.stride_bn == 1 ? a.stride_bk : a.stride_bn) % 64 == 0 &&
         ((reinterpret_cast<uintptr_t>(a.a) | reinterpret_cast<uintptr_t>(a.b)) & 127) == 0;
}

// 16-byte vector access on a row-major [rows, cols] view of `es`-byte elements
bool vec_ok(const void* base, int64_t stride_m, int64_t stride_n, int es) {
  return stride_n == 1 && aligned16(base) && ((stride_m * es) % 16) == 0;
}

// (the few-rows kernel's build that reduces) tiles of a launch, and bytes of all ranks' partials of a tile
constexpr int REDUCE_MAX_TILES = 128;
constexpr int64_t REDUCE_MAX_BYTES = 128 << 10;

struct Plan {
  const GemmKernelEntry* entry = nullptr;
  GemmKArgs k{};
  int fused_reduce = 0;  // ONE_SHOT, CONSUME on its own or IRIS_PHASE_TWO_KERNELS: follow with the reduce kernel
  int in_program = 0;    // ONE_SHOT, IRIS_PHASE_FUSED: the build of the kernel that reduces each tile itself
  int one_per_cu = 0;    // (asked for) not two programs of a small tile a CU: they have no fetching waves, and no build that covers
  int parts = 0;         // the launch's tiles lie across the caller's (plan_cover; 2: by plan_across)
  int loose = 0;         // the few-rows kernel's build for operands at any alignment
  int b_rows = 0;        // ... for a row-major B (cells)
  int two_kernels = 0;   // ... or, for such a launch too, what IRIS_PHASE_TWO_KERNELS would run (reduce_in_program)
  // the few-rows kernel instead of a table entry: workgroups along the columns, the rows and K
  GemmKernelFn skinny = nullptr;
  int skinny_grid = 0, skinny_grid_y = 1, skinny_grid_z = 1, skinny_lds = 0;
  int reduces = 0;       // the few-rows kernel's build that reduces, too
  int skinny_arows = 16;
  int skinny_rb = 1, skinny_cb = 1;  // blocks of 16 rows and of 16 columns a workgroup of the few-rows kernel takes
  // a second launch of the entry's split-K build behind the first: the tiles of the last round, K shared out
  // over the programs that round would leave idle
  int last_round = 0;
  GemmKArgs k_last{};
  // the build that numbers its flags in a grid of its own (blocks of the caller's tiles, or a range of its columns)
  int remap_flags = 0;
  // a second plan behind this one: the columns of tiles this one leaves out
  std::shared_ptr<Plan> rest;
};

int dbg() {
  static int v = std::getenv("IRIS_AMD_DEBUG") ? 1 : 0;
  return v;
}

// Workgroups that share the K range of each of `cells` blocks of C in the few-rows kernel, from what bounds it: the
// CU with the most workgroups (`block_us` for a block of K a wave), B at the rate a stream of it reaches (6 TB/s),
// and for a shared range the hand-over (2 us, 0.1 more for every part).  A part keeps 32 blocks, four a wave.  (us a
// pass, by parts: [4,8192] x [8192,192] 9.8 / 9.1 / 8.0 / 8.3 with 1 / 2 / 4 / 8, [16,8192] x [8192,1024] 10.0 / 9.6 /
// 8.9 / 10.2, [6,9344] x [9344,2560] 13.2 unshared and 14.4 in 3.)
int few_rows_parts(int64_t cells, int64_t nb, double block_us, int64_t b_bytes) {
  const int64_t cus = current_cu_count();
  int best = 1;
  double least = 0;
  for (int parts = 1; parts <= SKINNY_MAX_SPLIT && (parts == 1 || parts * 32 <= nb); ++parts) {
    const int64_t share = (nb + parts - 1) / parts;
    if ((parts - 1) * share >= nb) continue;  // (the last part would be empty)
    const double busiest = (double)((cells * parts + cus - 1) / cus * ((share + SKINNY_WAVES - 1) / SKINNY_WAVES)) * block_us;
    const double stream = (double)b_bytes / 6e6;
    const double cost = (busiest > stream ? busiest : stream) + (parts > 1 ? 2 + 0.1 * parts : 0);
    if (parts == 1 || cost < least) best = parts, least = cost;
  }
  return best;
}

// A few rows: the product is a stream over B, and the kernel built for that
// takes it when the operands allow the 16-byte fetches, the logical tile
// covers every row (or whole workgroups of them) and the tiles' arrival counters have a home.  Fills the
// plan and returns true when the launch qualifies.
// `loose`: the operands are not aligned, or K is no multiple of eight (dma_ok says that the kernel's build for those takes them).
bool plan_few_rows(const iris_gemm_args& a, int op, bool dma_ok, bool loose, Plan* plan) {
  GemmKArgs& k = plan->k;
  const int64_t lim = (int64_t)1 << 31;
  // Up to 32 rows: a workgroup per 16 rows x 16 columns, unless B is more than the 16 MB that are as well read
  // twice ([32,4096] x [4096,4096] 12.5 us in blocks of 16 rows and 11.3 in 32, [32,2560] x [2560,8192] 18.5 and 13.8, but
  // [17,4096] x [4096,1376] 8.4 and 9.2).  Up to 64 rows of a long K, where the persistent kernel would split K and
  // pay more for the hand-over: 32 rows x 16 columns a workgroup, as long as one round of workgroups covers the
  // matrix ([64,4096] x [4096,1376]: 172 workgroups, 11.5 us against 12.7).
  const int64_t b_bytes = (int64_t)a.N * a.K * 2;
  const bool mid = a.M > SKINNY_MAX_ROWS;
  const int rb = mid || (a.M > SKINNY_ROWS && a.K >= SKINNY_MID_MIN_K && b_bytes > (16 << 20)) ? 2 : 1;
  const int m_blocks = (a.M + SKINNY_ROWS * rb - 1) / (SKINNY_ROWS * rb);
  const int n_blocks = (a.N + SKINNY_COLS - 1) / SKINNY_COLS;
  const int64_t cells = (int64_t)m_blocks * n_blocks;
  const bool counters = (m_blocks == 1 && (a.block_n <= SKINNY_COLS || a.N <= SKINNY_COLS)) || k.flag_mode == 0 ||
                        (a.locks && k.total_tiles <= a.num_sms);
  // fp32: the matrix cores do a sixteenth of the 16-bit rate and a tile that is half padding costs twice, so it is
  // taken up to 128 rows, above 64 where the workgroups come in (nearly) whole rounds.  (us a pass: [64,512] x
  // [512,1024] 13.8 by the persistent kernel, 8.7 here, [96,4096] x [4096,1024] 23.1 and 17.8, [128,2048] x
  // [2048,2048] 24.2 and 17.3, but [128,4096] x [4096,1376], 344 workgroups, 26.4 and 28.4.)
  const bool f32 = a.ab_dtype == IRIS_DTYPE_F32;
  const int64_t cus = current_cu_count();
  const bool f32_room = a.M <= SKINNY_MID_MAX_ROWS ||
                        (a.M <= SKINNY_F32_MAX_ROWS && (cells <= cus || cells * 4 >= (cells + cus - 1) / cus * cus * 3));
  const bool room = !mid || (f32 && f32_room) || (cells <= (int64_t)current_cu_count() && a.M <= SKINNY_MID_MAX_ROWS && a.K >= SKINNY_MID_MIN_K);
  // 17 to 32 rows of a long K are left to the persistent kernel where the workgroups need a second round, or where
  // rows that start anywhere on a cache line cost more than B's stream ([17..32,16384] x [16384,4776] 40-42 us here and
  // 31.5 there, [27,21136] x [21136,4776] 63 and 39, [32,21136] x [21136,4096] 41 and 36; but at K = 4096 14 and 16.6,
  // [32,16384] x [16384,4096] 28.2 and 30.5, [17,21136] x [21136,4096] 34.2 and 35.6, [32,21136] x [21136,1376] 21 and 23).
  const bool lines = whole_lines(a);
  const bool long_k = a.variant == 0 && !mid && rb == 2 && !f32 &&
                      (cells > cus ? a.K >= 8192 : !lines && a.M > 24 && a.K >= 20480 && b_bytes > (96 << 20));
  // Off the 16 bytes the L1 is the bound earlier, and the tiles no longer gather.  (us a pass, here / there: [9,12977] x
  // [12977,4352] 46 / 35, [15,20993] x [20993,3392] 49 / 43, [24,449] x [449,5824] 11.3 / 7.1, [23,29889] x [29889,2368] 54 / 43,
  // [36,26745] x [26745,1376] 42 / 26, fp32 [43,10433] x [10433,3136] 100 / 70, [115,10753] x [10753,6400] 341 / 177; but [1,23937] x
  // [23937,3584] 37 / 46, [24,15489] x [15489,1600] 16.7 / 18.3, [63,27009] x [27009,528] 23 / 29, fp32 [58,17025] x [17025,192] 18 / 20.)
  const bool off = loose && a.variant == 0;
  const bool off_f32 = off && f32 && (mid ? (cells >= 128 && a.K >= 32768) || (cells > cus && a.K >= 8192) || (cells > 4 * cus && a.K >= 1024)
                                          : a.M > 16 && cells > cus && a.K >= 8192);
  const bool off_16 =
      off && !f32 && (mid        ? (cells >= 72 && a.K >= 16384) || (cells >= 192 && a.K >= 12288)
                      : rb == 2  ? (cells >= 128 && a.K >= 18432) || (cells > cus && a.K >= 6144)
                      : a.M > 16 ? cells > 2 * cus
                                 : (cells > cus && a.K >= (a.M > 8 ? 8192 : 16384)) || (a.M > 8 && b_bytes > (128 << 20)));
  // (the workgroups' rows belong to one tile)
  const bool rows_ok = a.block_m >= a.M || (f32 && a.block_m % (SKINNY_ROWS * rb) == 0);
  const bool ok = room && !long_k && !off_f32 && !off_16 && a.K > 0 && dma_ok && !plan->in_program && rows_ok && (a.block_n % SKINNY_COLS) == 0 &&
                  !a.mm_begin_timestamp && !a.mm_end_timestamp && (a.split_k == 0 || a.split_k == 1) && counters &&
                  ((int64_t)SKINNY_ROWS * rb * a.stride_am + a.K) * 2 < lim &&
                  ((int64_t)SKINNY_COLS * a.stride_bn + a.K) * 2 < lim;
  if (!ok) return false;
  // K shared out: the blocks of C count their parts' arrivals in the words of `locks` behind the tiles' own
  int parts = 1;
  if (a.split_k == 0 && a.partials && aligned16(a.partials) && a.locks && k.total_tiles + cells <= a.num_sms) {
    // a block of K of a workgroup alone on its CU, by what it fetches; rows that do not start on a cache line
    // touch half as many lines again ([31,11800] x [11800,1360] 0.85 us, [40,16384] x [16384,512] 0.48)
    const double block_us = (rb == 2 ? 0.5 : 0.3) * (lines ? 1 : 1.6);
    parts = few_rows_parts(cells, (a.K + 63) / 64, block_us, b_bytes);
    const int64_t elems = cells * rb * (SKINNY_ROWS * SKINNY_COLS);  // of one part's sums
    if (parts * elems > (int64_t)a.num_sms * a.partials_slot_elems) parts = 1;
  }
  plan->skinny = gemm_skinny_kernel_for(a.ab_dtype, op, a.M <= 8 ? 8 : 16, rb, 1, loose, false, false);
  if (!plan->skinny) return false;
  plan->loose = loose;
  plan->skinny_lds = skinny_lds_bytes(rb);
  plan->skinny_grid = n_blocks;
  plan->skinny_grid_y = m_blocks;
  plan->skinny_grid_z = parts;
  plan->skinny_rb = rb;
  plan->skinny_arows = a.M <= 8 ? 8 : 16;
  k.split_k = 1;
  k.locks = a.locks;
  k.partials = a.partials;
  return true;
}

// A small product of more rows in cells of 32 x 32 (gemm_skinny.hpp), where one round of workgroups covers it.  us a pass
// as 64 x 64 tiles, K shared out where that helps, and as cells: [213,624] x [624,320] 7.7 / 6.4, [475,2560] x [2560,480]
// 12.3 / 8.6, [128,4096] x [4096,1376] 12.7 / 9.6, [1239,4288] x [4288,192] 13.9 / 10.0, [100,8192] x [8192,256] 12.3 /
// 9.0; fp32 [475,2560] x [2560,480] 21.7 / 17.6.  In two rounds the second starts from nothing and the tiles are as good
// or better: [728,3072] x [3072,448] 13.8 / 13.8, [1113,832] x [832,393] 8.9 / 10.3.  Only for a launch that owns the
// device and says how many XCDs it has: the cells are dealt to them so that each fetches its own part of an operand.
// Whether it is better than tiles at the launch's K is for plan_small to say.
// `b_rows`: a row-major B, up to 32 rows of A too, which the few-rows kernel does not take with it (us a pass, operands changed
// from call to call, tiles / cells: [1,4096] x [4096,1376] 14.4 / 9.4, [4,1376] x [1376,4096] 12.3 / 8.2, [95,4224] x [4224,1280]
// 14.2 / 11.0, [251,1344] x [1344,384] 10.6 / 7.9; 90 random calls 1.27x).
bool plan_cells(const iris_gemm_args& a, int op, bool dma_ok, bool loose, bool b_rows, Plan* plan) {
  GemmKArgs& k = plan->k;
  const int64_t lim = (int64_t)1 << 31, cus = current_cu_count();
  const int64_t m_cells = (a.M + CELL - 1) / CELL, n_cells = (a.N + CELL - 1) / CELL, cells = m_cells * n_cells;
  const bool counters = k.flag_mode == 0 || (a.locks && k.total_tiles <= a.num_sms);
  const bool ok = a.K > 0 && dma_ok && !plan->in_program && cells <= cus && a.num_sms >= cus && a.num_xcds > 1 && (a.block_m >= a.M || a.block_m % CELL == 0) &&
                  a.block_n % CELL == 0 && !a.mm_begin_timestamp && !a.mm_end_timestamp && (a.split_k == 0 || a.split_k == 1) &&
                  counters && (CELL * a.stride_am + a.K) * 2 < lim && (CELL * a.stride_bn + a.K) * 2 < lim;
  if (!ok) return false;
  const int xcd_per = (int)((cells + a.num_xcds - 1) / a.num_xcds);
  int parts = 1;
  // (K of a row-major B is shared out for one row of cells only: [138,32000] x [32000,128] in twelve parts 24.4 us, 18.0 in tiles)
  if (a.split_k == 0 && a.partials && aligned16(a.partials) && a.locks && k.total_tiles + cells <= a.num_sms && (m_cells == 1 || !b_rows)) {
    // An XCD takes xcd_per workgroups of each part: it is those that have to fit its CUs, not all parts' workgroups the device's.
    // (us a pass with a second round on some XCDs, 35 workgroups on 32 CUs / so: off the 16 bytes [40,18929] x [18929,800] 25.3 /
    // 18.4, [92,32385] x [32385,384] 33.7 / 25.2, row-major [20,26048] x [26048,576] 21.0 / 15.4, fp32 along K [171,21184] x
    // [21184,960] 98.7 / 85.4; 137 random calls 1.21x, one slower than before cells took such operands.)
    // (0.6 us for 64 of K of a workgroup, 1.5 times that with a row-major B: its half lines)
    parts = few_rows_parts(xcd_per * a.num_xcds, (a.K + 63) / 64, b_rows ? 0.9 : 0.6, (int64_t)a.N * a.K * 2);
    if (parts * cells * (CELL * CELL) > (int64_t)a.num_sms * a.partials_slot_elems) parts = 1;
  }
  // (a row-major B with up to 16 rows of A: cells of 16 x 32, which fetch the half or the quarter of A that there is)
  const int rb = b_rows && a.M <= SKINNY_ROWS ? 1 : 2;
  plan->skinny = gemm_skinny_kernel_for(a.ab_dtype, op, rb == 1 && a.M <= 8 ? 8 : 16, rb, 2, loose, b_rows, false);
  if (!plan->skinny) return false;
  k.cells = (int)cells;
  k.cells_by_row = a.M > a.N;
  k.cells_inner = (int)(k.cells_by_row ? n_cells : m_cells);
  k.xcd_per = xcd_per;
  k.div_inner = make_fast_div((uint32_t)k.cells_inner, (uint64_t)cells + 1);
  k.div_xcd = make_fast_div((uint32_t)a.num_xcds, (uint64_t)k.xcd_per * a.num_xcds + 1);
  plan->loose = loose;
  plan->b_rows = b_rows;
  plan->skinny_lds = cells_lds_bytes(rb);
  plan->skinny_grid = k.xcd_per * a.num_xcds;
  plan->skinny_grid_y = 1;
  plan->skinny_grid_z = parts;
  plan->skinny_rb = rb;
  plan->skinny_arows = rb == 1 && a.M <= 8 ? 8 : 16;
  plan->skinny_cb = 2;
  k.split_k = 1;
  k.locks = a.locks;
  k.partials = a.partials;
  return true;
}

// Parts of K for `tiles` tiles of `steps` K-steps of 64 (1: unsplit).  The hand-over of partials costs about as much as ten
// K-steps of a small tile: as many parts as there are idle programs, at least four K-steps each, and a K loop shorter
// than 32 steps is only split in four or more parts (measured on [M, 1376] x [1376, 4096], 22 steps of 128 x 128 tiles:
// 4 parts 16.4 against 19.5 us unsplit at 128 rows, 2 parts 25.9 against 20.2 at 512).
int auto_split(int64_t tiles, int steps, int programs) {
  if (tiles * 2 > programs || steps < 16) return 1;
  int sk = (int)(programs / tiles);
  if (sk > steps / 4) sk = steps / 4;
  if (sk > 16) sk = 16;
  return sk >= 4 || steps >= 32 ? sk : 1;
}

// Split-K and stream-K.  The owner of a tile waits for the programs that hold
// its other parts, so every part needs a program of its own that is resident
// at the same time: no more programs than the device has CUs.
hipError_t plan_split(const iris_gemm_args& a, const GemmKernelEntry& pick, bool in_program, GemmKArgs* kp) {
  GemmKArgs& k = *kp;
  k.split_k = 1;
  k.split_q = k.split_r = 0;
  k.partials = a.partials;
  k.locks = a.locks;
  k.partial_stride = a.partials_slot_elems;
  k.status = a.status;
  k.timeout = a.spin_timeout_ticks ? a.spin_timeout_ticks : 200000000ull;  // 2 s at 100 MHz
  k.stream_k = 0;
  if (a.split_k < 0 && a.split_k != IRIS_GEMM_SPLIT_STREAM_K) return hipErrorInvalidValue;
  if (a.split_handover < IRIS_GEMM_HANDOVER_AUTO || a.split_handover > IRIS_GEMM_HANDOVER_PAIR)
    return hipErrorInvalidValue;
  const int nk = (a.K + pick.bk - 1) / pick.bk;
  // the rules below were measured on K-steps of 64: `d` such steps to one of this tile
  const int d = pick.bk > 64 ? pick.bk / 64 : 1;
  if (in_program) {
    // the program that computes a tile also reduces it: K is never shared out
    return (a.split_k > 1 || a.split_k == IRIS_GEMM_SPLIT_STREAM_K) ? hipErrorInvalidValue : hipSuccess;
  }
  if (a.split_k != 1 && a.partials && a.locks) {
    const bool resident = a.num_sms <= current_cu_count();
    const bool any_way = resident && pick.splitk && pick.fn_split && k.sub_m == 1 && k.sub_n == 1 &&
                         (reinterpret_cast<uintptr_t>(a.partials) & 15) == 0 && (a.partials_slot_elems % 4) == 0;
    // Two parts of a 128-accumulator tile can meet with half a partial tile each (the pair hand-over: each part
    // keeps the accumulators of the waves it owns), so a slot of half a tile is enough for them; that is what a
    // caller who holds tiles half as wide has ([8192,14336] x [14336,448] in 256 x 64 tiles, run as 256 x 128).
    const bool pair_ok = any_way && !pick.split_owner && (pick.wm * pick.wn) % 2 == 0 &&
                         a.partials_slot_elems * 2 >= (int64_t)pick.cm * pick.cn;
    const bool possible = any_way && a.partials_slot_elems >= (int64_t)pick.cm * pick.cn;
    // Stream-K: every program takes the same number of K-steps (within one).
    // A run of at least four steps keeps the parts of a tile few.
    const int64_t steps = (int64_t)k.total_tiles * nk;
    const int run = (int)(steps / a.num_sms);
    const bool stream_ok = possible && pick.split_owner && run * d >= 4 && run >= 1 && steps < ((int64_t)1 << 30) &&
                           (nk + run - 1) / run + 1 <= 32;
    if (a.split_k == IRIS_GEMM_SPLIT_STREAM_K) {
      if (!stream_ok) return hipErrorInvalidValue;
      k.stream_k = 1;
    } else if (a.split_k > 1) {
      if (!(possible || (pair_ok && a.split_k == 2)) || a.split_k > nk || a.split_k > 64 ||
          (int64_t)k.total_tiles * a.split_k > a.num_sms)
        return hipErrorInvalidValue;
      k.split_k = a.split_k;
    } else if (possible || pair_ok) {
      int sk = auto_split(k.total_tiles, nk * d, a.num_sms);
      if (!possible && sk > 2) sk = 2;  // (slots of half a tile: two parts)
      if (sk >= 4 || (sk > 1 && nk * d >= 32)) k.split_k = sk;
      // Stream-K is only taken on request.  With the plain four-wave tiles it beat both the
      // unsplit and the split launch where the tiles left programs idle and the walk was long
      // (132 tiles of 64 steps on 256 programs: -17 %).  The tiles with fetching waves made
      // the K-steps a quarter shorter and left the hand-over as it was: on the same shapes
      // stream-K now ties with split-K (66 tiles: 27.9 against 27.6 us in three parts) or
      // loses (88 tiles: 33.2 against 31.9 in two parts; 132 tiles: 41.0 against 37.6 unsplit;
      // more tiles than programs: 80 against 54).  Nor does it pay where the walk is long and the last round
      // of tiles leaves most programs idle ([8192,36864] x [36864,576] in 288 tiles of 256 x 64 on 256
      // programs: 940 against 805 us): programs that start at different depths of K no longer fetch the
      // panels their neighbours fetch at the same time, and the operands come from HBM several times over.
    }
  } else if (a.split_k > 1 || a.split_k == IRIS_GEMM_SPLIT_STREAM_K) {
    return hipErrorInvalidValue;  // forced, but no workspace
  }
  if (k.split_k > 1) {
    k.split_q = nk / k.split_k;
    k.split_r = nk % k.split_k;
    // Many parts: every part reduces and stores a slice of the tile, instead
    // of the first part reading all the others' partials one after another.
    // Few parts: the owner's way, which has one hand-over less on its critical
    // path (measured on [128, 4096] x [4096, 1376] with 128 x 128 tiles: 16
    // parts 16.6 against 26.7 us, 8 parts 17.2 against 23.4, 4 parts 23.2
    // against 25.1, 2 parts 39 against 33; 64 x 64 tiles in 5 parts 16.2
    // against 14.9): sliced from eight parts up.
    // (the 128-accumulator tiles only have the sliced one)
    if (a.split_handover == IRIS_GEMM_HANDOVER_SLICED && k.split_k > pick.cm) return hipErrorInvalidValue;
    if (a.split_handover == IRIS_GEMM_HANDOVER_OWNER && !pick.split_owner) return hipErrorInvalidValue;
    const bool can_pair = k.split_k == 2 && !pick.split_owner && (pick.wm * pick.wn) % 2 == 0 &&
                          a.partials_slot_elems * 2 >= (int64_t)pick.cm * pick.cn;
    const bool can_slice = a.partials_slot_elems >= (int64_t)pick.cm * pick.cn;
    if (a.split_handover == IRIS_GEMM_HANDOVER_PAIR && !can_pair) return hipErrorInvalidValue;
    if (a.split_handover == IRIS_GEMM_HANDOVER_SLICED && !can_slice) return hipErrorInvalidValue;
    // (two parts of a 128-accumulator tile: the pair hand-over moves half the bytes of the sliced one)
    k.sliced = a.split_handover == IRIS_GEMM_HANDOVER_SLICED  ? 1
               : a.split_handover == IRIS_GEMM_HANDOVER_OWNER ? 0
               : a.split_handover == IRIS_GEMM_HANDOVER_PAIR  ? 2
               : can_pair                                     ? 2
                                                              : (!pick.split_owner || k.split_k >= 8) ? 1 : 0;
  }
  if (k.stream_k) {
    const int64_t steps = (int64_t)k.total_tiles * nk;
    k.split_q = (int)(steps / a.num_sms);
    k.split_r = (int)(steps % a.num_sms);
  }
  return hipSuccess;
}

// The launch's divisors as multiply-high constants, and how its items are dealt to the XCDs.
void launch_constants(const iris_gemm_args& a, const GemmKernelEntry& pick, GemmKArgs* kp) {
  GemmKArgs& k = *kp;
  const int nk = (a.K + pick.bk - 1) / pick.bk;
  const uint64_t items = (uint64_t)k.total_tiles * k.sub_m * k.sub_n + 1;
  k.tile_divs = make_tile_divs(k.num_pid_m, k.num_pid_n, k.G);
  k.div_subs = make_fast_div((uint32_t)(k.sub_m * k.sub_n), items);
  k.div_sub_n = make_fast_div((uint32_t)k.sub_n, items);
  k.div_split = make_fast_div((uint32_t)k.split_k, (uint64_t)a.num_sms + 1);
  k.div_xcd = make_fast_div((uint32_t)a.num_xcds, 2 * (uint64_t)a.num_sms + 1);
  k.div_nk = make_fast_div((uint32_t)(nk > 0 ? nk : 1), (uint64_t)k.total_tiles * (nk > 0 ? nk : 1) + 1);
  // Fewer (tile, part) items than programs: deal them to the XCDs evenly, in
  // consecutive runs, instead of filling the first XCDs and idling the rest.
  // (under stream-K every program has a run: the reference's XCD remap stays)
  const int64_t work = (int64_t)k.total_tiles * k.split_k;
  // parts of 32 K-steps or more: the programs part by part (see GemmKArgs::part_major; the short walks of
  // the decoder shapes were tuned tile by tile and stay so)
  k.part_major = (k.split_k > 1 && !k.stream_k && nk / k.split_k >= 32) ? k.total_tiles : 0;
  k.xcd_per = 0;
  if (!k.stream_k && a.num_xcds > 1 && work < a.num_sms) k.xcd_per = (int)((work + a.num_xcds - 1) / a.num_xcds);
  // L2 prefetch hints for long walks over K (the tiles with fetching waves read them): an XCD's share of a round
  // of tiles is a block of `rows` x `cols` neighbouring tiles, whose CUs share the A panels `cols` ways and the B
  // panels `rows` ways.  They pay on the 64-column tiles, whose K-steps are short enough to be bound by how
  // long a stage takes to arrive from HBM ([8192,14336] x [14336,448] in 256 x 64 tiles: 175 -> 161 us eight
  // steps ahead, 155 sixteen ahead); the wider tiles' steps are bound by the matrix cores' power budget on real
  // data and gain nothing (256 x 128: 427 -> 440 us on N(0, 0.02) data, 408 -> 380 us on zeros).
  // Staggered start (see GemmKArgs::stagger_groups): the unsplit eight-wave 256 x 256 tile, when every program has
  // two tiles or more, so that there are epilogues whose store bursts the stagger keeps apart (a launch of one
  // tile per program would only end later).  Two groups, 8 x 576 clocks = 2 us apart: [8192,1024] x [1024,8192]
  // 90.2 -> 87.6 us on zeros, 113.7 -> 112.0 on N(0, 0.02) data; [8192,1536] x [1536,4096] stored to eight ranks
  // 185.6 -> 182.6; [8192,7168] x [7168,4096] (two tiles a program, 112 K-steps each) unchanged.  Only for walks of
  // at most 64 K-steps: on a long walk the epilogues are little beside the K loop, and programs that fetch the
  // same panels two microseconds apart find less of them in their XCD's L2 ([8192,36864] x [36864,4608]: +2 %).
  k.stagger_groups = k.stagger_sleeps = 0;
  if (pick.cm == 256 && pick.cn == 256 && pick.wm * pick.wn == 8 && pick.fetch_waves == 0 && k.split_k == 1 &&
      !k.stream_k && a.num_xcds > 1 && k.sub_m == 1 && k.sub_n == 1 && k.total_tiles >= 2 * (int64_t)a.num_sms &&
      a.num_sms >= 2 * a.num_xcds && nk <= 64) {
    k.stagger_groups = 2;
    k.stagger_sleeps = 8;
  }
  k.pf_dist = k.pf_sa = k.pf_sb = 0;
  const int pf_dist = 8;
  if (pick.fetch_waves > 0 && pick.cm == 256 && pick.cn == 64 && !pick.b_rows && !pick.loose && !k.stream_k && k.sub_m == 1 && k.sub_n == 1 && nk >= 16 * pf_dist &&
      a.num_xcds > 1) {
    const int64_t per_xcd = k.xcd_per > 0 ? k.xcd_per : (k.num_sms / a.num_xcds);
    int64_t tiles_per_xcd = k.split_k > 1 ? (per_xcd + k.split_k - 1) / k.split_k : per_xcd;
    if (k.part_major > 0) tiles_per_xcd = per_xcd;  // (part by part: an XCD's programs are neighbouring tiles)
    const int g_rows = k.G < k.num_pid_m ? k.G : k.num_pid_m;
    int64_t cols = tiles_per_xcd / (g_rows > 0 ? g_rows : 1);
    if (cols < 1) cols = 1;
    if (cols > k.num_pid_n) cols = k.num_pid_n;
    int64_t rows = tiles_per_xcd / cols;
    if (rows < 1) rows = 1;
    // one touch instruction per operand covers 64 rows of the share: the share must thin the panel out enough
    if (cols * 64 >= pick.cm && rows * 64 >= pick.cn && cols * rows > 1) {
      k.pf_dist = pf_dist;
      k.pf_sa = (int)cols;
      k.pf_sb = (int)rows;
    }
  }
  // The same hints for the eight-wave 256 x 256 tile, whose every wave also loads: they are a build of their own
  // (GemmKernelEntry::fn_touch), taken where a round of tiles streams its operands from HBM.  Looping
  // [8192,14336] x [14336,2048] (294 MB of operands, one tile a program): 358 -> 339 us three steps ahead, 345 four,
  // 352 eight (an XCD's share of eight steps, 3 MB, no longer stays in its 4 MB L2), 411 when every program touches
  // all its lines instead of its share; on zeros 337 -> 296.  [8192,28672] x [28672,4096] (two tiles a program)
  // 1393 -> 1344.  Where the operands stay in the 256 MB last-level cache the touches only add L2 requests:
  // [8192,12288] x [12288,2048] (252 MB) +3 %, [8192,7168] x [7168,4096] +2 %; and an XCD whose tiles are two rows
  // of sixteen (group size 2) fetches half as many lines again per step and is bound by that, not by latency
  // ([8192,36864] x [36864,4608]: +5 %).  So: at least 272 MB of operands per round of tiles, and an XCD block of at
  // least four tiles either way.
  if (a.touch_ahead != IRIS_GEMM_TOUCH_OFF && pick.fn_touch && k.split_k == 1 && !k.stream_k && k.sub_m == 1 && k.sub_n == 1) {
    const int64_t per_xcd = a.num_xcds > 1 ? (k.xcd_per > 0 ? k.xcd_per : (k.num_sms / a.num_xcds)) : k.num_sms;
    const int g_rows = k.G < k.num_pid_m ? k.G : k.num_pid_m;
    int64_t cols = per_xcd / (g_rows > 0 ? g_rows : 1);
    if (cols < 1) cols = 1;
    if (cols > k.num_pid_n) cols = k.num_pid_n;
    int64_t rows = per_xcd / cols;
    if (rows < 1) rows = 1;
    // (the kernel takes its share of a panel's rows with a mask: powers of two)
    int sa = 1, sb = 1;
    while (sa * 2 <= cols && sa < 64) sa *= 2;
    while (sb * 2 <= rows && sb < 64) sb *= 2;
    const int64_t rounds = (k.total_tiles + k.num_sms - 1) / k.num_sms;
    const int64_t operand_bytes = ((int64_t)a.M + a.N) * a.K * 2;
    const bool streams = nk >= 32 && sa >= 4 && sb >= 4 && operand_bytes >= rounds * ((int64_t)272 << 20);
    if (a.touch_ahead == IRIS_GEMM_TOUCH_ON || streams) {
      k.pf_dist = 3;
      k.pf_sa = sa;
      k.pf_sb = sb;
    }
  }
}

// Validate `a` and build the launch plan.  Returns hipSuccess,
// hipErrorInvalidValue, or a pseudo-success with entry == nullptr when there
// is no GEMM work to do.
// `cells`: as cells of 32 x 32, if the launch can be (the caller asks with `skinny_cb`).
hipError_t make_plan_body(const iris_gemm_args& a, Plan* plan, bool cells = false);

// A long GEMM whose tiles are a few more than a multiple of the programs spends a whole round on those few:
// 288 tiles on 256 programs take two rounds for 1.125 rounds of work.  Where a tile's walk over K is long
// and the caller brought the split-K workspace, the plan becomes two launches on the stream: the full rounds
// as they are, then the tiles of the last round with K shared out over the programs it would leave idle
// (every part at the same depths of K as its neighbours', so the operand panels are still fetched together;
// stream-K, which would even out the rounds too, loses that and is slower here).
void split_last_round(const iris_gemm_args& a, Plan* plan) {
  GemmKArgs& k = plan->k;
  const GemmKernelEntry* e = plan->entry;
  plan->last_round = 0;
  if (!e || plan->skinny || plan->in_program || k.split_k != 1 || k.stream_k || k.sub_m != 1 || k.sub_n != 1) return;
  if (k.merge_m * k.merge_n > 1 || plan->remap_flags) return;  // (the second launch would raise flags of its own grid)
  if (a.split_k != 0 || a.variant != 0 || a.mm_begin_timestamp || a.mm_end_timestamp) return;
  if (!a.partials || !a.locks || !e->splitk || !e->fn_split || k.num_sms != a.num_sms) return;
  if (a.num_sms > current_cu_count() || a.partials_slot_elems < (int64_t)e->cm * e->cn) return;
  const int programs = a.num_sms, rounds = k.total_tiles / programs, last = k.total_tiles - rounds * programs;
  if (rounds < 1 || last == 0 || last * 2 > programs) return;
  const int nk = (a.K + e->bk - 1) / e->bk;
  // parts of at least 32 K-steps: the build with fetching waves of a split 128-accumulator tile needs them
  // to pay for its spills, and the second launch's start must be little beside a part's walk
  int parts = programs / last;
  if (parts > 16) parts = 16;
  if (parts > nk / 32) parts = nk / 32;
  if (parts < 2) return;
  iris_gemm_args forced = a;
  forced.split_k = parts;
  GemmKArgs t = k;
  t.tile_base = rounds * programs;
  t.total_tiles = last;
  if (plan_split(forced, *e, false, &t) != hipSuccess || t.split_k != parts) return;
  launch_constants(forced, *e, &t);
  k.total_tiles = rounds * programs;
  launch_constants(a, *e, &k);
  plan->k_last = t;
  plan->last_round = 1;
}

// The plan for the caller's tiles blocked merge_m x merge_n; false when the launcher has no kernel for it.
bool plan_merged(const iris_gemm_args& a, int merge_m, int merge_n, Plan* plan) {
  iris_gemm_args b = a;
  b.block_m = a.block_m * merge_m;
  b.block_n = a.block_n * merge_n;
  Plan merged;
  const hipError_t err = make_plan_body(b, &merged);
  // (only the persistent kernels publish merged tiles: unsplit, or split in parts)
  const bool unsplit = merged.k.split_k == 1 && merged.entry && merged.entry->fn_merged;
  const bool parts = merged.k.split_k > 1 && merged.entry && merged.entry->fn_split_merged;
  if (err != hipSuccess || !merged.entry || merged.skinny || !(unsplit || parts) || merged.k.stream_k || merged.in_program)
    return false;
  *plan = merged;
  plan->remap_flags = 1;
  plan->k.merge_m = merge_m;
  plan->k.merge_n = merge_n;
  plan->k.flag_num_pid_m = (a.M + a.block_m - 1) / a.block_m;
  plan->k.flag_num_pid_n = (a.N + a.block_n - 1) / a.block_n;
  plan->k.flag_pn_base = 0;
  if (merge_m * merge_n > 1) split_last_round(b, plan);
  return true;
}

// `a` restricted to columns [col0, col0 + cols) of B and of the output (whole tiles of the caller).
iris_gemm_args column_range(const iris_gemm_args& a, int64_t col0, int64_t cols) {
  iris_gemm_args b = a;
  b.N = (int32_t)cols;
  b.b = static_cast<const char*>(a.b) + col0 * a.stride_bn * 2;
  if (a.epilogue == IRIS_EPI_ALL_SCATTER) {
    // (the launcher adds cur_rank * N columns to c_global: of the range's N, so the difference goes in here;
    // the pointer is only ever used with that offset added)
    const int64_t shift = (int64_t)a.cur_rank * (a.N - cols) + col0;
    b.c_global = static_cast<char*>(a.c_global) + shift * a.stride_cn_global * dtype_size(a.c_global_dtype);
  } else {
    b.c = static_cast<char*>(a.c) + col0 * a.stride_cn * dtype_size(a.c_dtype);
    b.c_global = static_cast<char*>(a.c_global) + col0 * a.stride_cn_global * dtype_size(a.c_global_dtype);
  }
  return b;
}

// The plan of a launch.  A caller's tile that is narrow or short (the reference scripts' 256 x 64; 128 x 128)
// makes a large GEMM wait for its operands: a 256 x 64 tile fetches 256 rows of A every K-step for 64 columns'
// worth of work.  Where there are enough of them, the launch computes a block of the caller's tiles as one
// 256 x 128 or 256 x 256 tile and raises each one's flag: tile ids and flags are the caller's, which program
// computes a tile was never observable ([8192,8192] x [8192,1024] in 256 x 64 tiles: 739-762 -> 928 TFLOP/s
// over the eight ranks of the reference's 07 benchmark).
hipError_t make_plan_units(const iris_gemm_args& a, Plan* plan);

// fp32 operands (the reference scripts' --datatype fp32; the output is fp32 too): the kernels count K and the
// operands' strides in 16-bit units, two to an element, and everything between this function and the MFMAs
// (loaders, slabs, stages, K tail, the 2 GiB windows of the buffer descriptors) is the 16-bit kernels' as it is.
hipError_t make_plan(const iris_gemm_args& a, Plan* plan) {
  if (a.ab_dtype != IRIS_DTYPE_F32) return make_plan_units(a, plan);
  const int64_t lim = (int64_t)1 << 30;
  if (a.K < 0 || a.K >= lim) return hipErrorInvalidValue;
  iris_gemm_args b = a;
  b.K = 2 * a.K;
  b.stride_am = 2 * a.stride_am;
  b.stride_ak = 2 * a.stride_ak;
  b.stride_bk = 2 * a.stride_bk;
  b.stride_bn = 2 * a.stride_bn;
  return make_plan_units(b, plan);
}

// A plan whose tiles are the caller's.
void own_flags(Plan* plan) {
  GemmKArgs& k = plan->k;
  k.merge_m = k.merge_n = 1;
  k.flag_num_pid_m = k.num_pid_m;
  k.flag_num_pid_n = k.num_pid_n;
  k.flag_pn_base = 0;
}

// Estimated times of a small product's launch, in us: what plan_small compares its plans by.  A CU fetches 108 KB a us
// (its L1), an eighth less when all of them do (L2); rows that start anywhere on a cache line touch a third to a half as
// many lines again, and a gathering tile's fetching waves need three times as long.  A K-step takes as long as its operands, or as
// the matrix cores where those are slower.  Around the K loop: the launch, the arrival counters of parts, the epilogue
// (each rank's copy), and for a shared K the hand-over, which grows with the partials that cross memory.  The constants
// are a fit to 8200 timings of 33 shapes ([24,8192] .. [96,2560] .. [4477,136] .. [1500,1500]) at K from 152 to 36864:
// every tile, cells, up to 16 parts of K, 16-bit and fp32, weights in rows of either direction and at any alignment,
// stores and atomics.  The plan with the least of these times is on average 0.5 % over the fastest one timed, in three
// cases of 200 more than 8 %.
struct TileLaunch {
  int cm, cn;
  int64_t tiles;  // (the caller's, `subs` of these to one, or parts of the caller's)
  int subs, split_k;
  bool sliced, parts;
};
struct Operands {
  bool f32, lines, gather, b_rows, loose, atomic, vec_out;
  int copies;     // of the output
  bool peers;     // other ranks wait for it
  int64_t tile;   // elements of a caller's tile that lie in the output
};
// How much of the operands comes from HBM: none of it up to 60 MB, all from 110 MB on (a program has other data in the 256 MB
// of the last-level cache between two launches).
double streamed(const iris_gemm_args& a) {
  const double of = (((double)a.M + a.N) * a.K * 2e-6 - 60) / 50;
  return of < 0 ? 0 : of > 1 ? 1 : of;
}
double tiles_us(const iris_gemm_args& a, const TileLaunch& t, const Operands& o, int64_t cus) {
  const int64_t items = t.tiles * t.split_k, programs = items < cus ? items : cus;
  const bool split = t.split_k > 1;
  const double cover = programs * 5 > cus * 4 ? 1.0 : 0.0;  // (nearly) every CU fetches
  const double area = (double)t.cm * t.cn / 4096, partials = programs * area / 64;  // tiles of 64 x 64; MB
  const bool deep = t.cm == 64 && t.cn == 64;  // (K-steps of 128: whole lines, mostly)
  const double fetch = (t.cm + t.cn) / (8 * 108.0) * (1 + 0.13 * cover + (split ? 0.17 : 0.0)) *
                       (o.gather ? 2.9 : o.lines ? 1.0 : o.loose ? (deep ? 1.9 : 2.1) : deep ? 1.3 : 1.5) *
                       ((o.b_rows || o.loose) && !split ? 1 + 0.5 * streamed(a) : 1.0);
  const double multiply = o.f32 ? area * 0.452 * (1 + 0.04 * cover) + 0.1 : area * 0.0535;
  const int64_t unit = deep ? 2 : 1, nk = ((int64_t)a.K + 64 * unit - 1) / (64 * unit);
  const int64_t part_steps = (nk + t.split_k - 1) / t.split_k * unit, steps = (items + cus - 1) / cus * t.subs * part_steps;
  const double loop = steps * (fetch > multiply ? fetch : multiply);
  // (from the last-level cache, or from HBM, which a few programs do not keep busy)
  const double mb = ((double)a.M + a.N) * a.K * 2e-6, rate = mb > 200 ? 2 + 3.5 * programs / cus : 5.5;
  const double stream = mb / rate - 6.9;
  double us = 7.4 + 0.005 * programs + 0.1 * area * (o.copies - 1) + (loop > stream ? loop : stream);
  if (o.gather) us += 2.3 + 0.24 * area;
  if (o.atomic) us += 1.5 * area;
  if (t.parts && !o.atomic) {
    const double per_tile = (double)o.tile / (t.cm * t.cn) / 16;  // (the more parts count on one word, the longer it takes)
    us += 0.1 + 0.008 * programs * (per_tile < 1 ? per_tile : 1.0);
  }
  if (!split) {
    us += area > 4 ? 2.4 : 0.1 * area;
    // (more where peers wait for it: us a pass in 64 x 64 / 128 x 64 parts, [4318,576] x [576,192] to four ranks 11.8 / 12.4,
    // [518,256] x [256,928] and its reduce over eight 17.2 / 17.9; [389,512] x [512,2240] alone 10.24 / 10.28)
    if (o.peers && !o.atomic) us += 0.45 * (area - 1);
    if (!o.vec_out) us += area < 4 ? 1.5 * area : 6.0;  // (rows that 16-byte stores don't fit)
  } else {
    us += 3.1 + 0.53 * area + 0.2 * (partials < 16 ? partials : 16) + (partials > 16 ? 0.4 * (partials - 16) : 0.0);
    // (an owner adds the parts of a tile one after another)
    if (!t.sliced && area > 1) us += 0.31 * area * (t.split_k - 1);
    // (a short part pays for the 256 x 64 tile's prefetch hints)
    if (!o.f32 && t.cm == 256 && t.cn == 64 && nk >= 128 && part_steps < 64) us += 5;
  }
  return us;
}
double cells_us(const iris_gemm_args& a, int64_t cells, int parts, const Operands& o, int64_t cus) {
  const int64_t groups = cells * parts, nk = ((int64_t)a.K + 63) / 64;
  const double mb = ((double)a.M + a.N) * a.K * 2e-6;
  // us for 64 of K, operands in whole lines / not: [512,512] 256 cells 0.090 / 0.13; [128,1376] 172 cells 0.083 / 0.11;
  // [200,512] 112 cells 0.048 / 0.066 as long as the L2s hold the operands, 0.07 / 0.08 beyond
  // (a row-major B comes in half lines: 1.5 times the requests' time with the 32 rows of A beside it, and from HBM at half the rate;
  // fitted with both in it.  [28,7936] x [7936,4864] 33.8, in tiles 23.5; with up to 16 rows of A a cell fetches half of A)
  const double lines = o.b_rows ? (a.M <= SKINNY_ROWS ? 1.08 : 1.8) : o.lines ? 1.0 : o.loose ? 2.1 : 1.45;
  const double step = 0.083 * (groups * 5 > cus * 4 ? 1.09 : groups * 2 <= cus && mb <= 30 ? 0.7 : 1.0) *
                      (o.f32 && lines < 1.65 ? 1.65 : lines);
  // (a workgroup's first sixteen blocks of K are in flight together)
  const double loop = ((groups + cus - 1) / cus * ((nk + parts - 1) / parts) - 16) * step;
  const double stream = mb / (o.b_rows ? (mb > 80 ? 3.2 : 4.8) : o.loose ? (mb > 100 ? 3.2 : 6.0) : mb > 200 ? 4.4 : 8.4) - 3, k_time = loop > stream ? loop : stream;
  const double per_tile = o.atomic ? 0.0 : (double)o.tile / (CELL * CELL) / 64;
  return 5.85 + (0.0075 + 0.004 * (per_tile < 1 ? per_tile : 1.0)) * groups + 0.025 * (o.copies - 1) + (parts > 1 ? 0.7 : 0.0) +
         (o.atomic ? 0.4 : 0.0) + (k_time > 0 ? k_time : 0.0);
}

// Whether `e` fetches the operands by the loader of `own`, or by a faster one: the DMA, the gathering loads, single elements.
bool no_slower_loader(const GemmKernelEntry& e, const GemmKernelEntry& own) {
  return e.dma || (!own.dma && (e.gather || !own.gather));
}

// Words of the caller's locks in which its `tiles` tiles count arrivals, one each (pack 0) or four to a word (2).
int64_t arrival_words(int64_t tiles, int pack) { return pack ? (tiles + 3) / 4 : tiles; }

// Whether tiles of cm x cn may lie across the caller's, whose arrivals are counted in words (pack 0) or bytes (2): no more of
// them to one of the caller's than a byte counts, and no more of the caller's to one of them than its publication, which takes
// them one after another, walks in MOST_TOUCHED round trips of an atomic.
constexpr int MOST_TOUCHED = 64;
bool can_cover(const iris_gemm_args& a, int cm, int cn, int pack) {
  const int64_t touched = ((int64_t)(cm - 1) / a.block_m + 2) * ((cn - 1) / a.block_n + 2);
  const int64_t parts = ((int64_t)(a.block_m - 1) / cm + 2) * ((a.block_n - 1) / cn + 2);
  return touched <= MOST_TOUCHED && (pack == 0 || parts <= 255);
}

// The launch in tiles of cm x cn, K shared out in split_k.  A caller's tile is the unit of a flag, not of work: the tiles that share
// one of the caller's count their arrivals in the caller's locks (the last `words` of them), and the last one raises its flag.
bool plan_cover(const iris_gemm_args& a, int cm, int cn, int split_k, int64_t words, int pack, Plan* plan) {
  iris_gemm_args b = a;
  b.block_m = cm;
  b.block_n = cn;
  b.variant = IRIS_GEMM_VARIANT_PERSISTENT;
  b.split_k = split_k;
  // (slots of this tile's size, as many as the workspace holds)
  const int64_t items = ((int64_t)a.M + cm - 1) / cm * (((int64_t)a.N + cn - 1) / cn) * split_k;
  // (and the parts of a tile's K count in the locks, too)
  if (words > a.num_sms || (split_k > 1 && items + words > a.num_sms)) return false;
  if (split_k > 1 && a.partials && a.partials_slot_elems < (int64_t)cm * cn)
    b.partials_slot_elems = (int64_t)a.num_sms * a.partials_slot_elems / items & ~(int64_t)3;
  plan->one_per_cu = 1;
  if (make_plan_body(b, plan) != hipSuccess) return false;
  GemmKArgs& k = plan->k;
  if (!plan->entry || plan->entry->cm != cm || plan->entry->cn != cn || k.sub_m != 1 || k.sub_n != 1 || k.num_sms != a.num_sms ||
      plan->in_program)
    return false;
  own_flags(plan);
  k.flag_num_pid_m = (a.M + a.block_m - 1) / a.block_m;
  k.flag_num_pid_n = (a.N + a.block_n - 1) / a.block_n;
  if (words > 0) {
    const GemmKernelEntry* e = plan->entry;
    const bool small = cm <= 128 && cn <= 128 && e->fetch_waves != 0;
    if (!small && !(split_k > 1 ? e->fn_split_merged : e->fn_merged)) return false;
    if (cm == 256 && cn == 128 && split_k == 1 && (e->b_rows || e->loose)) return false;  // (`covers`)
    plan->remap_flags = small ? 0 : 1;
    k.cover_bm = a.block_m;
    k.cover_bn = a.block_n;
    k.arrive_pack = pack;
    k.div_cover_m = make_fast_div((uint32_t)a.block_m, (uint64_t)a.M);
    k.div_cover_n = make_fast_div((uint32_t)a.block_n, (uint64_t)a.N);
    k.tile_arrivals = a.locks + (a.num_sms - words);
  }
  plan->parts = 1;
  return true;
}

// A small product: the caller's tiles, cells of 32 x 32, or parts of the caller's tiles, whichever is expected to finish
// first, each with K shared out as its own rule has it, parts also without.  Returns false for the caller's
// tiles.  us a pass, the caller's tiles / the best parts / cells:
//   [1000,1504] x [1504,999] in 256 x 64 tiles  21.6 (K in four) / 10.7 / -
//   [512,512] in 256 x 128 tiles                K 1024 12.3 / 10.2 / 9.0   16384 26.6 / 25.8 / 28.8   36864 33.5 / 33.3 / 61
//   [256,2048] in 128 x 128 tiles               K 2048 17.8 / 13.3 / -     8192 25.7 / 24.8 / -       36864 48 / 65 / -
// Small tiles fill the chip and fetch more for the work they do: their K-steps are many times as many as those of a
// large tile whose K is shared out, so they lose to it from some K on.  What the few-rows kernel takes is its;
// parts for a launch that owns the device and leaves tile and split to the launcher.
bool plan_small(const iris_gemm_args& a, Plan* plan) {
  const int64_t cus = current_cu_count();
  if (a.variant != 0 || (a.split_k != 0 && a.split_k != 1) || a.mm_begin_timestamp || a.mm_end_timestamp) return false;
  if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.block_m <= 0 || a.block_n <= 0 || a.num_sms < cus) return false;
  if (a.epilogue == IRIS_EPI_ONE_SHOT && (a.phase == IRIS_PHASE_FUSED || a.phase == IRIS_PHASE_CONSUME)) return false;
  auto tiles_of = [&](int cm, int cn) { return ((int64_t)a.M + cm - 1) / cm * (((int64_t)a.N + cn - 1) / cn); };
  if (tiles_of(128, 128) > a.num_sms) return false;
  Plan whole;
  if (make_plan_body(a, &whole) != hipSuccess) return false;
  if (whole.skinny) {  // few rows
    own_flags(&whole);
    *plan = whole;
    return true;
  }
  if (!whole.entry) return false;
  const GemmKArgs& w = whole.k;
  const Operands o{a.ab_dtype == IRIS_DTYPE_F32, whole_lines(a), !whole.entry->dma, whole.entry->b_rows, whole.entry->loose,
                   a.epilogue == IRIS_EPI_ATOMIC_ADD, w.vec_out != 0, w.dest_all ? a.world_size : 1, a.world_size > 1,
                   (int64_t)(a.block_m < a.M ? a.block_m : a.M) * (a.block_n < a.N ? a.block_n : a.N)};
  double least = tiles_us(a, TileLaunch{whole.entry->cm, whole.entry->cn, w.total_tiles, w.sub_m * w.sub_n, w.split_k,
                                        w.sliced != 0, false}, o, cus);
  bool found = false;
  if (tiles_of(CELL, CELL) <= cus) {
    Plan cells;
    if (make_plan_body(a, &cells, true) == hipSuccess && cells.skinny_cb == 2) {
      const double us = cells_us(a, cells.k.cells, cells.skinny_grid_z, o, cus);
      if (us < least) {
        least = us;
        own_flags(&cells);
        *plan = cells;
        found = true;
      }
    }
  }
  // (fp32 operands, K in 16-bit units here: the tiles for longer K)
  if (a.split_k != 0 || a.num_sms != cus || (a.ab_dtype == IRIS_DTYPE_F32 && a.K < 1024)) return found;
  const bool flags = a.epilogue == IRIS_EPI_ALL_SCATTER ? a.notify != 0 : a.epilogue == IRIS_EPI_ONE_SHOT && a.world_size > 1;
  const int64_t words = flags ? tiles_of(a.block_m, a.block_n) : 0;
  if (words > 0 && (!a.locks || words > a.num_sms)) return found;
  // (the last part raises the flag for all: where it is a release, only its own stores would be covered, see publish_tile)
  if (words > 0 && a.flag_sem == IRIS_FLAG_SEM_RELEASE_ACQUIRE) return found;
  // Where K of the caller's tiles is shared out, parts larger than 64 x 64 are taken up to this K only: they fetch no less
  // than the shared tiles do, and the longer the K the less their hand-over weighs.  (us a pass, the caller's tiles / parts:
  // 256 x 256 tiles [2534,1664] x [1664,896] 35.5 / 19.1, [667,5888] x [5888,4160] 72 / 58, [1669,30872] x [30872,320] 91 /
  // 95; 256 x 128 [3319,1792] x [1792,312] 24.3 / 17.0, [7069,13376] x [13376,512] 117 / 138; 256 x 64 [797,2048] x
  // [2048,1856] 32.1 / 27.6, [786,25064] x [25064,1368] 154 / 232; 128 x 128 tiles [1024,2048] x [2048,1376] keep theirs.)
  const int whole_k = a.ab_dtype == IRIS_DTYPE_F32 || a.block_m < 256 ? 0 : a.block_n >= 256 ? 6144 : 2560;
  static const int shapes[4][2] = {{64, 64}, {128, 64}, {64, 128}, {128, 128}};
  TileLaunch list[8];
  double times[8];
  int count = 0;
  for (const auto& s : shapes) {
    if (a.block_m % s[0] != 0 || a.block_n % s[1] != 0 || !can_cover(a, s[0], s[1], 0)) continue;
    const int64_t tiles = tiles_of(s[0], s[1]);
    if (tiles > a.num_sms) continue;
    if (s[0] == a.block_m && s[1] == a.block_n) break;  // (the caller's tile is the smallest that fits)
    if (s[0] * s[1] > 64 * 64 && w.split_k > 1 && a.K > whole_k) break;
    const int bk = s[0] == 64 && s[1] == 64 ? 128 : 64;  // (the 64 x 64 tile's K-step)
    int sk = a.partials && a.locks ? auto_split(tiles, (int)(((int64_t)a.K + bk - 1) / bk) * (bk / 64), a.num_sms) : 1;
    // (the parts of a part's K use the locks, too)
    if (tiles * sk + words > a.num_sms) sk = (int)((a.num_sms - words) / tiles);
    for (int split_k = 1;; split_k = sk) {
      const TileLaunch t{s[0], s[1], tiles, 1, split_k, split_k >= 8, true};
      list[count] = t;
      times[count++] = tiles_us(a, t, o, cus);
      if (split_k >= sk) break;
    }
    // (the gathering tiles' times scatter more: the first shape that fits, unless another is clearly ahead of it)
    if (o.gather && s[0] * s[1] == 64 * 64) times[count - 1] *= 0.9;
  }
  // the best of them that there is a kernel for
  for (;;) {
    int best = -1;
    for (int i = 0; i < count; ++i)
      if (times[i] < least && (best < 0 || times[i] < times[best])) best = i;
    if (best < 0) return found;
    Plan parts;
    if (plan_cover(a, list[best].cm, list[best].cn, list[best].split_k, words, 0, &parts) &&
        no_slower_loader(*parts.entry, *whole.entry)) {
      *plan = parts;
      return true;
    }
    times[best] = 1e30;
  }
}

// Whether a launch of IRIS_PHASE_FUSED is better off reducing inside the program than behind it, `producer` being the
// plan of the same launch without the reduce.  Inside, a tile is one program's from its first K-step to its last
// strip: K is not shared out, the caller's tiles are not blocked, the fetching waves' registers are not there, and
// CUs whose tiles are done do not help with the others' reduces.  Behind, a kernel boundary is paid, 4 us.  So inside
// for one round of small tiles with a short K, whose producer would run the same way (us a pass, inside / behind:
// K-shard [785,216] x [216,2752], 8 fp32 partials, 256 x 64 tiles 25.3 / 28; 64^3 8.9 / 12); behind otherwise
// ([1999,1376] x [1376,4096] in 256 x 128 tiles 67 / 54, in 256 x 256 tiles 78 / 62, 25 tiles of K = 29408 741 / 103).
// Where the producer would run in smaller units than the caller's tiles, those win from a shorter K on: [64,K] x [K,640],
// 8 bf16 partials, 256 x 64 tiles 11.6 / 13.5 at K = 128, 12.4 / 13.5 at 320, 13.9 / 14.0 at 640, 16.7 / 14.6 at 1376;
// [128,K] x [K,4096] 13.1 / 17.2 at 128, 17.2 / 18.9 at 640; [128,K] x [K,320] 13.2 / 12.7 at 128 (5 tiles: 5 CUs);
// [2000,320] x [320,640], 2 fp32 partials 18.0 / 21.4; [16,K] x [K,4096] 10.8 / 12.2 at 128, 11.9 / 12.0 at 320.
// A launch that shares the device with its peers' (fewer programs than CUs) stays inside: every program's CU is counted
// there.
bool reduce_in_program(const iris_gemm_args& a, const Plan& producer) {
  if (a.num_sms < current_cu_count() || a.variant != 0 || a.split_k != 0 || a.mm_begin_timestamp || a.mm_end_timestamp) return true;
  if (!producer.entry && !producer.skinny) return true;  // (nothing to compute)
  const GemmKArgs& k = producer.k;
  const int steps = (a.K + 63) / 64;
  const int64_t tiles = ((int64_t)a.M + a.block_m - 1) / a.block_m * (((int64_t)a.N + a.block_n - 1) / a.block_n);
  const int64_t inside = (int64_t)(a.block_m < a.M ? a.block_m : a.M) * (a.block_n < a.N ? a.block_n : a.N);
  const int64_t strips = inside * a.world_size * dtype_size(a.c_dtype);  // bytes that a program's tile is reduced from
  // (inside, operands at any alignment and a row-major B are gathered)
  const bool rows = producer.skinny ? producer.b_rows != 0 : producer.entry->b_rows;
  const bool loose = producer.skinny ? producer.loose != 0 : producer.entry->loose;
  if (tiles <= a.num_sms && k.vec_out && !rows && !loose && (producer.skinny || producer.entry->dma)) {
    const bool few = producer.skinny && producer.skinny_cb == 1;
    if (inside <= 64 * 64 && (few ? steps <= 2 && a.block_n <= 64 : steps <= 10)) return true;
    if (!few && tiles >= 16 && a.block_n <= 64 && steps <= 5 && (inside <= 128 * 64 || strips <= (128 << 10))) return true;
  }
  // (few rows off the 16 bytes: [16,133] x [133,4096] of 8 bf16 partials 12.0 / 13.2, K 389 12.9 / 13.2, 637 14.7 / 13.2)
  if (loose && producer.skinny && tiles <= a.num_sms && k.vec_out && inside <= 64 * 64 && a.block_n <= 64 && steps <= 7)
    return true;
  // (parts of those, for what is behind them: row-major [3587,K] x [K,448] in 256 x 64 tiles of 4, K 128 15.2 / 17.1, fp32 19.2 / 21.5, 256
  // 18.1 / 18.0, fp32 21.3 / 22.4, 384 20.8 / 19.0; of 8, bf16, K 128 19.7 / 18.6)
  const bool wide = a.c_dtype == IRIS_DTYPE_F32;
  if ((rows || loose) && producer.parts && tiles <= a.num_sms && k.vec_out && a.block_m * a.block_n <= 128 * 128 && steps <= 4 &&
      strips < (wide ? (256 << 10) + 1 : 256 << 10))
    return true;
  if ((producer.skinny && producer.skinny_cb == 1) || producer.last_round || producer.rest || producer.parts == 1) return false;
  // (a producer that runs faster across the caller's tiles: inside, those are back, in a round for every num_sms of them.  us a pass,
  // inside / behind: 30 random calls of more tiles than programs 1.22x, [1330,552] x [552,3560] of 4, 64 x 128 tiles 46.4 / 35.4; one
  // round of 256 x 256 tiles [2550,344] x [344,2376] of 8 58.8 / 39.6, fp32 in 128 x 128 [418,256] x [256,760] 30.2 / 22.4, 256 x 64
  // 1.09x; of 128 x 64, fp32 [748,256] x [256,1504] of 4 23.0 / 27.1, row-major [580,227] x [227,2880] 16.9 / 22.3, 24 calls 0.92x)
  if (producer.parts == 2 && (tiles > a.num_sms || a.block_m * a.block_n > 128 * 64)) return false;
  // (cells: the caller's tiles inside, when they are as small as the parts they would be run in)
  if (producer.skinny && a.block_m * a.block_n > 64 * 64) return false;
  if (k.split_k > 1 || k.merge_m * k.merge_n > 1 || k.total_tiles > a.num_sms || !k.vec_out) return false;
  // Behind, those operands go through the DMA, so they stay inside for less: up to fewer K-steps the larger the tile, and not
  // where a program has 256 KB to reduce.  (us a pass, inside / behind, bf16 partials; row-major B, 64 x 64 tiles [1000,1024] of 8,
  // K 1024 17.9 / 19.7, 1504 21.7 / 20.9; cells [16,4096] of 8, K 256 11.6 / 13.8, 520 14.7 / 13.2; 128 x 128 tiles [2048,2048] of 2,
  // K 392 21.4 / 24.1, 1288 37.8 / 27.6, of 8, K 1024 37.3 / 31.0; 256 x 128 [4096,2048] of 2, K 136 28.2 / 30.0, 392 35.7 / 31.5;
  // along K off the 16 bytes, 128 x 128 tiles of 2, K 709 24.2 / 27.7, 1285 34.8 / 31.7; 256 x 64 [4096,1024] of 8, K 1501 48.7 / 43.6.)
  if (rows || loose) {
    const int area = a.block_m * a.block_n;
    // (a short shard, inside / behind: along K off the 16 bytes, 128 x 128 tiles [2048,2048] of 8, bf16, K 129 27.0 / 28.5, 385 30.5 /
    // 30.9, of 8, fp32, 37.2 / 40.2, 41.0 / 42.7, of 4, fp32, 26.2 / 32.2, 29.7 / 34.5, 641 33.3 / 37.1; row-major, of 8, bf16, K 128 25.5 /
    // 27.3, 384 29.5 / 28.9, of 4, fp32, 24.4 / 31.0, 512 30.3 / 33.7; 256 x 128 tiles, fp32, 144 tiles of 4, 34 / 42, 41 / 46.5, 256 tiles
    // 46.5 / 46.0, 54 / 50.4; bf16 there, and 256 x 64 tiles [2580,185] x [185,1000] of 8 29.1 / 24.3, as the line below)
    const int few = loose ? (!wide ? 6 : strips > (256 << 10) ? 7 : 12) : strips > (256 << 10) ? (wide ? 4 : 0) : wide ? 8 : 4;
    if (steps <= few && strips <= (512 << 10) && area <= 128 * 128 && a.block_m <= 128) return true;
    if (steps <= (loose ? 7 : 8) && wide && area > 128 * 128 && area <= 256 * 128 && tiles * 4 <= (int64_t)a.num_sms * 3) return true;
    const int most = area > 128 * 128 ? 4 : area > 64 * 64 ? (rows ? 8 : 12) : rows ? (producer.skinny ? 7 : 16) : 24;
    return steps <= most && (area <= 64 * 64 || strips < (256 << 10));
  }
  return steps <= 8 || (steps <= 24 && a.block_m * a.block_n <= 128 * 128);
}

// Times of a launch in large tiles, by which plan_blocks compares its plans: us = fixed + rounds of tiles * (tile + K-steps
// of a part * step), a step being dearer by `cover` when every CU takes one (the board's power, the L2s), by `off_lines`
// where rows do not start on cache lines, by `streamed` where the operands come from HBM (none of it up to 50 MB, all from
// 150 MB on: a program has other data in the 256 MB of the last-level cache between two launches).  Fitted to two thirds of
// 7000 random calls ([256 .. 8192, 128 .. 36864] x [.., 128 .. 8192], weights in rows of either direction and at any alignment,
// up to eight copies of the output, operands changed from launch to launch); on the other third the error is 7.4 % rms.
// (128 x 64 from an earlier fit.)
struct BlockTime {
  int cm, cn, split;
  double fixed, tile, step, cover, off_lines, streamed;
};
constexpr BlockTime BLOCK_TIMES[] = {
    {128, 64, 1, 4.4, 2.0, 0.249, 0.03, 0.45, 0.45},  {128, 128, 1, 4.1, 2.3, 0.375, 0.12, 0.26, 0.33},
    {256, 64, 1, 4.0, 2.2, 0.464, 0.00, 0.39, 0.41},  {256, 128, 1, 3.7, 4.1, 0.634, 0.07, 0.29, 0.22},
    {256, 128, 2, 8.9, 4.6, 0.505, 0.31, 0.36, 0.34}, {256, 256, 1, 2.9, 5.5, 0.999, 0.23, 0.20, 0.20},
    {256, 256, 2, 9.4, 4.9, 0.977, 0.37, 0.17, 0.21},
};
// A launch in tiles of cm x cn as plan_split and split_last_round make it, before there is a plan of it: K in `split` parts, or
// the last `last_tiles` tiles in `last_parts`.  (The plan is asked whether that is what it is: as_expected.)
struct BlockLaunch {
  int cm, cn, split;
  int64_t tiles;
  int last_tiles, last_parts;
};
BlockLaunch block_launch(const iris_gemm_args& a, int cm, int cn, bool callers, int cus) {
  BlockLaunch l{cm, cn, 1, ((int64_t)a.M + cm - 1) / cm * (((int64_t)a.N + cn - 1) / cn), 0, 0};
  const int nk = (a.K + 63) / 64;
  if (!a.partials || !a.locks || a.num_sms > cus) return l;
  const bool slots = a.partials_slot_elems >= (int64_t)cm * cn;
  if (slots || (cm * cn >= 256 * 128 && a.partials_slot_elems * 2 >= (int64_t)cm * cn)) {
    int sk = auto_split(l.tiles, nk, a.num_sms);
    if (!slots && sk > 2) sk = 2;
    if (sk >= 4 || (sk > 1 && nk >= 32)) l.split = sk;
  }
  if (callers && slots && l.split == 1) {
    const int64_t last = l.tiles % a.num_sms;
    int parts = last > 0 && l.tiles > a.num_sms && last * 2 <= a.num_sms ? (int)(a.num_sms / last) : 1;
    if (parts > 16) parts = 16;
    if (parts > nk / 32) parts = nk / 32;
    if (parts >= 2) {
      l.last_tiles = (int)last;
      l.last_parts = parts;
      l.tiles -= last;
    }
  }
  return l;
}
bool as_expected(const BlockLaunch& l, const Plan& plan) {
  const GemmKArgs& k = plan.k;
  return plan.entry && !plan.skinny && !k.stream_k && k.sub_m == 1 && k.sub_n == 1 && plan.entry->bk == 64 && plan.entry->cm == l.cm &&
         plan.entry->cn == l.cn && k.split_k == l.split && k.total_tiles == l.tiles && plan.last_round == (l.last_parts > 0) &&
         (!plan.last_round || (plan.k_last.split_k == l.last_parts && plan.k_last.total_tiles == l.last_tiles));
}

// The launch's time in us, or a negative number for one that the table does not know.
double block_us(const iris_gemm_args& a, const BlockLaunch& l, int cus) {
  const bool lines = whole_lines(a);
  double streamed = (((double)a.M + a.N) * a.K * 2e-6 - 50) / 100;
  streamed = streamed < 0 ? 0 : streamed > 1 ? 1 : streamed;
  const int nk = (a.K + 63) / 64;
  const bool along = a.stride_ak == 1 && a.stride_bk == 1;
  const bool loose = along && ((a.K | a.stride_am | a.stride_bn) % 8 != 0 || !aligned16(a.a) || !aligned16(a.b));
  const bool scatter = a.epilogue == IRIS_EPI_ALL_SCATTER, wide = (scatter ? a.c_global_dtype : a.c_dtype) == IRIS_DTYPE_F32;
  for (const BlockTime& t : BLOCK_TIMES) {
    if (t.cm != l.cm || t.cn != l.cn || t.split != l.split) continue;
    const int64_t items = l.tiles * t.split, rounds = (items + a.num_sms - 1) / a.num_sms;
    const double busy = (double)(rounds > 1 ? a.num_sms : items) / cus;
    const double step = t.step * (1 + t.cover * busy) * (lines ? 1.0 : 1 + t.off_lines) * (1 + t.streamed * streamed) * (loose ? 1.23 : 1.0);
    // (the other copies of the output, or its wider elements: 6.5 TB/s of stores on all CUs, a third of them hidden behind the
    // next round's products)
    const double copies = (scatter ? a.world_size : 1) * (wide ? 2 : 1), store = (copies - 1) * t.cm * t.cn * 2 / 25400.0 / t.split;
    const double us = t.fixed + rounds * (t.tile + (nk + t.split - 1) / t.split * step) +
                      store * (busy > 0.37 ? busy : 0.37) * (1 + (rounds - 1) * 0.67);
    if (l.last_parts == 0) return us;
    // the tiles of a last round that are shared out over all programs, as a launch of their own
    return us + 17.7 + t.tile + store * 0.37 + (nk + l.last_parts - 1) / l.last_parts * step;
  }
  return -1;
}

// Columns of the blocks (256 rows high) that a large launch is run in by number of tiles alone, 0 for the caller's tiles: blocks
// that give seven programs in eight one, by rounds of them and a tile's time (a 256 x 256 tile does twice the work at 1.25
// times the rate), or every other one with K in two.
int blocks_by_count(const iris_gemm_args& a, int64_t tiles_n) {
  const int64_t rows = ((int64_t)a.M + 255) / 256;
  const int mm = 256 / a.block_m;
  double best = 0;
  int found = 0;
  for (int width = 256; width >= 128; width /= 2) {
    const int mn = width / a.block_n;
    const int64_t tiles = rows * ((tiles_n + mn - 1) / mn);
    if (mm * mn == 1 || tiles * 8 < (int64_t)a.num_sms * 7) continue;
    const double cost = (double)((tiles + a.num_sms - 1) / a.num_sms) * (width == 256 ? 1.6 : 1.0);
    if (!found || cost < best) best = cost, found = width;
  }
  if (found || !a.partials || !a.locks || a.K < 4096) return found;
  for (int width = 256; width >= 128; width /= 2) {
    const int mn = width / a.block_n;
    const int64_t tiles = rows * ((tiles_n + mn - 1) / mn);
    if (mm * mn > 1 && tiles * 2 <= a.num_sms && tiles * 16 >= (int64_t)a.num_sms * 7 && a.partials_slot_elems * 2 >= (int64_t)256 * width)
      return width;
  }
  return 0;
}

// A large launch in the caller's tiles or in blocks of them, as 256 x 128 or 256 x 256 tiles; K shared by two programs a block
// where half of them suffice for the blocks and the caller's workspace has the slots; or the columns of tiles that block well
// first and the rest as a launch of their own.  What blocks_by_count says, unless another is expected to be faster by more than
// 5 % (2 % where it says the caller's tiles): the times above are not good for less, nor for as much on fewer programs than CUs,
// which they were not taken on, so 10 % there.  (us, [8192,K] x [K,N] in 256 x 64 tiles, the caller's / 256 x 128 / 256 x 256: N 576,
// K 1024 23 / 16 / 24; N 704, K 4128 98 / 53 / -; N 1152, K 12288 337 / 299 / 263; N 1344, K 4096 100 / 100 / 82.  6000 random calls,
// on average over the fastest plan timed: by count alone 9 % for a weight along K and 14 to 17 % for others, so 0.3 %; slower than
// by count by more than 3 %: 79 by the times alone, 45 so.  2000 calls on 16 to 248 programs, time by count / so 1.012 on average; slower
// than by count by more than 3 % 10 at 5 %, 4 at 10 %.)  The plans are weighed first, and only the one that is taken is made.
bool plan_blocks(const iris_gemm_args& a, Plan* plan) {
  if (a.ab_dtype == IRIS_DTYPE_F32) return false;
  const int cus = current_cu_count();
  const BlockLaunch own = block_launch(a, a.block_m, a.block_n, true, cus);
  const double own_us = block_us(a, own, cus);
  if (own_us < 0) return false;  // (K of the caller's tiles shared out, or no such tile)
  auto blocks = [&](const iris_gemm_args& b, int width) { return block_launch(b, 256, width, false, cus); };
  auto blocks_us = [&](const iris_gemm_args& b, int width) {
    const int mm = 256 / b.block_m, mn = width / b.block_n;
    if (mn < 1 || mm * mn == 1) return -1.0;
    const BlockLaunch l = blocks(b, width);
    // (a launch on fewer programs than CUs leaves room for others: none of its own stays idle for a larger block)
    if (b.num_sms < cus && l.tiles * l.split * 8 < (int64_t)b.num_sms * 7) return -1.0;
    return block_us(b, l, cus);
  };
  struct Candidate {
    double us;
    int width;       // of the blocks; 0: the caller's tiles
    int64_t main_n;  // columns of tiles in blocks, the others apart
  };
  const int64_t tiles_n = ((int64_t)a.N + a.block_n - 1) / a.block_n;
  Candidate list[5] = {{own_us, 0, tiles_n}};
  int count = 1, by_count = blocks_by_count(a, tiles_n), first = 0;
  for (int width = 256; width >= 128; width /= 2) {
    const double us = blocks_us(a, width);
    if (us <= 0) continue;
    if (width == by_count) first = count;
    list[count++] = {us, width, tiles_n};
  }
  // The columns of tiles may be one or a few too many for blocks that fill the programs: [8192,36864] x [36864,576] is nine
  // columns of 256 x 64 tiles, eight of which make 128 blocks with K in two parts.  (For a K that can be shared out.)
  const bool two_kernels = a.epilogue == IRIS_EPI_ONE_SHOT && a.phase != IRIS_PHASE_PRODUCE;
  if (a.N % a.block_n == 0 && a.K >= 4096 && a.partials && a.locks && !two_kernels) {
    for (int width = 256; width >= 128; width /= 2) {
      const int mn = width / a.block_n;
      if (mn < 2) continue;
      const int64_t main_n = tiles_n / mn * mn, rest_n = tiles_n - main_n;
      if (main_n == 0 || rest_n == 0 || rest_n * 4 > main_n) continue;
      const iris_gemm_args am = column_range(a, 0, main_n * a.block_n);
      const double wide_us = blocks_us(am, 256), half_us = blocks_us(am, 128);
      if (wide_us < 0 && half_us < 0) continue;
      const bool half = wide_us < 0 || (half_us > 0 && half_us < wide_us);
      // K of the rest shared out so far that A streams through again
      const double rest_us = 12.8 + ((double)a.M + (double)rest_n * a.block_n) * a.K * 2e-6 / 3.3;
      if (by_count == 0 && first == 0 && blocks_by_count(am, main_n) > 0) first = count;
      list[count++] = {(half ? half_us : wide_us) + rest_us, half ? 128 : 256, main_n};
    }
  }
  // (blocks that share K are a plan like the others)
  if (first == 0)
    list[0].us *= 0.98;
  else if (list[first].main_n < tiles_n || blocks(a, by_count).split == 1)
    list[first].us *= a.num_sms < cus ? 0.9 : 0.95;
  // the least of them that there is a kernel for
  for (;;) {
    Candidate* c = &list[0];
    for (int i = 1; i < count; ++i)
      if (list[i].us < c->us) c = &list[i];
    if (c->width == 0) break;
    const iris_gemm_args am = c->main_n < tiles_n ? column_range(a, 0, c->main_n * a.block_n) : a;
    Plan blocked;
    if (plan_merged(am, 256 / a.block_m, c->width / a.block_n, &blocked) && as_expected(blocks(am, c->width), blocked)) {
      // (the remaining columns as the caller's tiles; their flags sit at their place in the caller's grid)
      bool found = true;
      if (c->main_n < tiles_n) {
        const iris_gemm_args ar = column_range(a, c->main_n * a.block_n, (tiles_n - c->main_n) * a.block_n);
        blocked.rest = std::make_shared<Plan>();
        found = plan_merged(ar, 1, 1, blocked.rest.get());
        blocked.k.flag_num_pid_n = blocked.rest->k.flag_num_pid_n = (int)tiles_n;
        blocked.rest->k.flag_pn_base = (int)c->main_n;
      }
      if (found) {
        *plan = std::move(blocked);
        return true;
      }
    }
    c->us = 1e30;
  }
  return false;
}

// Whether `p_bytes` from p on and `q_bytes` from q on share any.
bool overlap(const void* p, int64_t p_bytes, const void* q, int64_t q_bytes) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(p), y = reinterpret_cast<uintptr_t>(q);
  return x < y + (uint64_t)q_bytes && y < x + (uint64_t)p_bytes;
}

// Few rows and cells with a reduce behind them: the reduce in the same kernel (gemm_skinny.hpp, REDUCE), where a tile is small
// enough for one workgroup to reduce it should its peers be late, and there are few enough tiles for that.
// One workgroup has 32 KB of partials in flight, so a late tile of REDUCE_MAX_BYTES is four round trips to memory, about what a reduce
// kernel's launch and chain take.  Waiting workgroups hold LDS that a peer on this device needs: late_tiles.hpp says how many of
// them wait at a time, of however many ranks; the others leave their tiles to those, up to REDUCE_MAX_TILES (of eight ranks one
// on a shader engine waits, on 32: four tiles one after the other).  The words for that, one an engine, are the last of the
// caller's locks.  Up to eight ranks (a wave each fetches their strips), of which late_most has one wait.  Not for
// a launch that shares the device with its peers' by its number of programs (fewer than CUs).
// Only for a result that shares no memory with what the kernel reads or stores besides: behind the product, one in the operands'
// or the partials' own buffer is as good as any other.
bool reduce_in_few_rows(const iris_gemm_args& a, Plan* plan) {
  GemmKArgs& k = plan->k;
  if (!plan->skinny || !plan->fused_reduce || a.epilogue != IRIS_EPI_ONE_SHOT || a.world_size < 2) return false;
  if (a.num_sms < current_cu_count() || !k.row_out || a.stride_cn_global != 1 || k.som < a.N || a.stride_cm_global < a.N) return false;
  const int gdt = a.c_global_dtype, ies = dtype_size(a.c_dtype), oes = dtype_size(gdt);
  if (gdt != IRIS_DTYPE_F32 && gdt != IRIS_DTYPE_F16 && gdt != IRIS_DTYPE_BF16) return false;
  const int64_t lim = (int64_t)1 << 31, rows = a.block_m < a.M ? a.block_m : a.M, cols = a.block_n < a.N ? a.block_n : a.N;
  if (((int64_t)a.block_m + 64) * k.som * ies >= lim || ((int64_t)a.block_m + 64) * a.stride_cm_global * oes >= lim) return false;
  if (k.total_tiles > REDUCE_MAX_TILES || rows * cols * ies * a.world_size > REDUCE_MAX_BYTES) return false;
  // (operands of fp32: K and strides in 16-bit units, make_plan)
  const int unit = a.ab_dtype == IRIS_DTYPE_F32 ? 2 : 1;
  const int64_t result = ((a.M - 1) * a.stride_cm_global + a.N) * oes, last_k = a.K / unit - 1;
  if (overlap(a.c_global, result, a.a, ((a.M - 1) * a.stride_am + last_k * a.stride_ak + unit) * 2) ||
      overlap(a.c_global, result, a.b, (last_k * a.stride_bk + (a.N - 1) * a.stride_bn + unit) * 2) ||
      overlap(a.c_global, result, a.c, ((a.M - 1) * a.stride_cm + a.N) * ies))
    return false;
  const GemmKernelFn fn = gemm_skinny_kernel_for(a.ab_dtype, a.c_dtype == IRIS_DTYPE_F32 ? OP_STORE32 : OP_STORE16, plan->skinny_arows,
                                                 plan->skinny_rb, plan->skinny_cb, plan->loose != 0, plan->b_rows != 0, true);
  if (!fn) return false;
  const int most = late_most(a.world_size);
  if (most < 1 || a.world_size > SKINNY_WAVES) return false;
  if (k.total_tiles > most) {
    const int64_t counters = k.total_tiles + (plan->skinny_grid_z > 1 ? (int64_t)plan->skinny_grid * plan->skinny_grid_y : 0);
    if (!a.locks || counters + LATE_ENGINES > a.num_sms) return false;
    k.tile_arrivals = a.locks + (a.num_sms - LATE_ENGINES);
  }
  plan->skinny = fn;
  plan->fused_reduce = 0;
  plan->reduces = 1;
  k.cg = static_cast<char*>(a.c_global);
  k.sgm = a.stride_cm_global;
  k.sgn = a.stride_cn_global;
  k.cg_dt = gdt;
  k.fused_vec = k.vec_out && vec_ok(k.cg, k.sgm, k.sgn, oes) && a.block_n % (16 / ies) == 0 && (a.block_n * oes) % 16 == 0;
  k.status = a.status;
  k.timeout = a.spin_timeout_ticks ? a.spin_timeout_ticks : 200000000ull;  // 2 s at 100 MHz
  return true;
}

hipError_t make_plan_tiles(const iris_gemm_args& a, Plan* plan);

hipError_t make_plan_units(const iris_gemm_args& a, Plan* plan) {
  const hipError_t err = make_plan_tiles(a, plan);
  if (err == hipSuccess) reduce_in_few_rows(a, plan);
  return err;
}

// A launch with atomics has no flags, so nothing shows which tiles it ran in: any tile will do, not only one that divides the
// caller's, and with fp32 atomics K may be shared out over programs that each add their own sums, with no hand-over and
// nobody waiting.  (16-bit atomics would round every part's sum on its way in: they keep whole sums.  So do launches whose
// ranks are other GPUs: each part's sums would cross the links, and the rate below is the one GPU's.)
//
// Times of such a launch in us: fixed + the first tile + the others, each as long as its K loop or its atomics (the chip adds
// 331 G a second, a CU a 64 x 64 tile in 1.1 us) + the last tile's atomics; `step`: 64 units of K of a tile, dearer by the same
// three things as BlockTime's.  Fitted to 6500 timings of 390 random calls ([33 .. 8192, 128 .. 36864] x [.., 128 .. 8192], 16-bit and
// fp32, weights in rows of either direction and at any alignment, K in up to 16 parts), rms 11 % on a third kept apart.
struct AtomicTime {
  int cm, cn;
  double tile, step, step_f32;  // (0: no such tile)
};
constexpr AtomicTime ATOMIC_TIMES[] = {
    {64, 64, 0.78, 0.149, 0.512},  {128, 64, 1.51, 0.234, 0},  {64, 128, 1.98, 0.245, 0.934}, {128, 128, 5.14, 0.333, 1.773},
    {256, 64, 4.46, 0.403, 1.832}, {256, 128, 10.3, 0.514, 0}, {128, 256, 9.20, 0.519, 0},
};
struct AtomicLaunch {
  double streamed;  // how much of the operands comes from HBM
  double each;      // us that the chip takes for all atomics of one part of K
  double contend;   // ... by which it takes longer for each part that adds to the same sums
  double kind;      // of the loader
  bool f32, lines;
};
// (`last_parts`: K of the last round's tiles in as many, as split_last_round leaves them, at 20 us for their launch and hand-over.)
double atomic_us(const iris_gemm_args& a, const AtomicTime& t, int parts, const AtomicLaunch& l, int last_parts = 1) {
  const int64_t items = ((int64_t)a.M + t.cm - 1) / t.cm * (((int64_t)a.N + t.cn - 1) / t.cn) * parts;
  const int64_t rounds = (items + a.num_sms - 1) / a.num_sms, nk = ((int64_t)a.K + 63) / 64, steps = (nk + parts - 1) / parts;
  const double busy = rounds > 1 ? 1.0 : (double)items / a.num_sms;
  const double step = (l.f32 ? t.step_f32 * (1 + 0.043 * busy) : t.step * (1 + 0.148 * busy) * (1 + 0.399 * l.streamed)) *
                      (l.lines ? 1.0 : 1.19) * l.kind;
  const double loop = t.tile + steps * step, cu = 0.518 * t.cm * t.cn / 4096;
  const double chip = 0.537 * l.each * parts / rounds * (1 + l.contend * (parts - 1));
  const double adds = chip > cu ? chip : cu, next = loop + 1.083 * adds;
  const double spared = last_parts > 1 ? steps * step * (1 - 1.0 / last_parts) - 20 : 0;
  return 6.82 + 1.09 * busy + loop + (rounds - 1) * (next > adds ? next : adds) + adds - (spared > 0 ? spared : 0);
}

// K of an unsplit plan with fp32 atomics in `parts`, each of which adds its own sums.
bool split_direct(const iris_gemm_args& a, int parts, Plan* plan) {
  GemmKArgs& k = plan->k;
  const GemmKernelEntry* e = plan->entry;
  const int nk = (a.K + e->bk - 1) / e->bk;
  if (e->op != OP_ATOMIC32 || !e->fn_split || k.split_k != 1 || k.stream_k || k.sub_m != 1 || k.sub_n != 1 || parts > nk ||
      (int64_t)k.total_tiles * parts > a.num_sms)
    return false;
  k.num_sms = a.num_sms;
  k.split_k = parts;
  k.split_q = nk / parts;
  k.split_r = nk % parts;
  k.sliced = SPLIT_DIRECT;
  launch_constants(a, *e, &k);
  return true;
}

// Replaces the plan of a launch with atomics where another tile, or (fp32 atomics) another number of parts of K, is expected to be
// faster by more than an eighth, a quarter where K is short and the atomics are most of the time; less the times above are not
// good for.  (us, in the caller's tiles or what plan_small made of
// them / so: [828,20672] x [20672,2688] in 256 x 64 tiles 208 / 109, 128 x 256 in three parts; [2023,22656] x [22656,192] in 256 x 128
// 54 / 36; fp32 [904,1024] x [1024,4224] in 128 x 128 140 / 77, 64 x 128; fp32 [1171,456] x [456,258] 41 / 15; row-major
// [494,9968] x [9968,4480] with 16-bit atomics in 64 x 64 98 / 68.  Of 353 random calls in tiles 96 change, 1.07x on average
// over all of them; four slower by 4 to 7 %, all in more than four rounds of tiles, which are left out.  The rules on
// more than two copies and on a last round whose K is shared out change the plans of 55 of 320 random calls of up to eight copies:
// 0.93 of the time in the caller's tiles without them, 18 of the 55 slower by more than 3 %, and 0.89 with them, three slower.)
void plan_atomics(const iris_gemm_args& a, Plan* plan) {
  const GemmKernelEntry* own = plan->entry;
  if (a.epilogue != IRIS_EPI_ATOMIC_ADD || !own || plan->skinny || plan->k.stream_k) return;
  if (a.variant != 0 || a.split_k != 0 || a.mm_begin_timestamp || a.mm_end_timestamp || a.num_sms != current_cu_count() || a.K <= 0) return;
  const bool wide = a.c_global_dtype == IRIS_DTYPE_F32, handed = plan->k.split_k > 1;
  // (To more than two copies, parts that hand over add their own slices of a tile to each, which is faster than all of it: of
  // 23 random calls of four and eight 0.95x so, [39,3816] x [3816,287] of eight 18 us and 28.)
  const bool parts_add = wide && (a.scope != IRIS_SCOPE_SYSTEM || a.world_size <= 1) && !(handed && a.world_size > 2);
  if (!parts_add && handed) return;
  AtomicLaunch l;
  const double mb = ((double)a.M + a.N) * a.K * 2e-6;
  l.streamed = mb < 50 ? 0 : mb > 150 ? 1 : (mb - 50) / 100;
  l.each = (double)a.M * a.N * a.world_size / 331e3 * (wide ? 1.0 : 0.5);
  l.contend = a.world_size > 2 ? 0.15 : 0;
  l.kind = !own->dma ? 1.9 : own->loose ? 1.24 : 1.0;
  l.f32 = a.ab_dtype == IRIS_DTYPE_F32;
  l.lines = whole_lines(a);
  constexpr int TILES = sizeof(ATOMIC_TIMES) / sizeof(ATOMIC_TIMES[0]);
  double own_us = -1;
  for (const AtomicTime& t : ATOMIC_TIMES)
    if (t.cm == own->cm && t.cn == own->cn) {
      // (a hand-over: 6 us, and the parts' sums are added up once)
      AtomicLaunch whole = l;
      whole.each /= plan->k.split_k;
      whole.contend = 0;
      own_us = atomic_us(a, t, plan->k.split_k, whole, plan->last_round ? plan->k_last.split_k : 1) + (handed ? 6 : 0);
    }
  if (own_us < 12) return;  // (another tile than these, or nothing to gain that the search would not cost)
  double best_us[TILES];
  int best_parts[TILES];
  for (int i = 0; i < TILES; ++i) {
    const AtomicTime& t = ATOMIC_TIMES[i];
    best_us[i] = 1e30;
    if (l.f32 && t.step_f32 == 0) continue;
    const int64_t tiles = ((int64_t)a.M + t.cm - 1) / t.cm * (((int64_t)a.N + t.cn - 1) / t.cn);
    if (tiles > 4 * (int64_t)a.num_sms) continue;
    int most = parts_add ? (int)(a.num_sms / tiles) : 1;
    if (most > 16) most = 16;
    if (most > (a.K + 63) / 64 / 3) most = (a.K + 63) / 64 / 3;
    for (int parts = 1; parts == 1 || parts <= most; parts += parts < 4 || parts + 2 > most ? 1 : 2) {
      const double us = atomic_us(a, t, parts, l);
      if (us < best_us[i]) best_us[i] = us, best_parts[i] = parts;
    }
  }
  // the least of them that there is a kernel for
  for (;;) {
    int i = 0;
    for (int j = 1; j < TILES; ++j)
      if (best_us[j] < best_us[i]) i = j;
    const AtomicTime& t = ATOMIC_TIMES[i];
    if (best_us[i] > (a.K < 512 && !l.f32 ? 0.78 : 0.87) * own_us) return;
    if (t.cm == own->cm && t.cn == own->cn && best_parts[i] == 1 && !handed) return;
    iris_gemm_args b = a;
    b.block_m = t.cm;
    b.block_n = t.cn;
    b.variant = IRIS_GEMM_VARIANT_PERSISTENT;
    b.split_k = 1;
    Plan free;
    if (make_plan_body(b, &free) == hipSuccess && free.entry && free.entry->cm == t.cm && free.entry->cn == t.cn &&
        no_slower_loader(*free.entry, *own) && (best_parts[i] == 1 || split_direct(b, best_parts[i], &free))) {
      own_flags(&free);
      *plan = std::move(free);
      return;
    }
    best_us[i] = 1e30;
  }
}

// Times of a launch with flags in us, for tiles that need not divide the caller's: fixed + rounds of tiles + the other copies of the
// output + the hand-over of a shared K, which grows with the partials that cross memory (MB) and with the parts; `step`: 64 units of
// K of a tile, dearer as BlockTime's are.  Fitted to two thirds of 11000 timings of 600 random
// calls ([33 .. 8192, 128 .. 36864] x [.., 128 .. 8192], 16-bit and fp32, weights in rows of either direction and at any alignment, up to eight
// copies, operands changed from launch to launch), rms 13 % on the rest.
struct AcrossTime {
  int cm, cn;
  double tile, step, step_f32;  // (0: no such tile)
};
constexpr AcrossTime ACROSS_TIMES[] = {
    {64, 64, 2.55, 0.153, 0.486}, {128, 64, 2.99, 0.245, 0.000}, {64, 128, 2.72, 0.256, 0.913}, {128, 128, 3.63, 0.343, 1.701},
    {256, 64, 3.75, 0.409, 0.000}, {256, 128, 5.07, 0.528, 0.000}, {256, 256, 6.20, 0.918, 0.000},
};
struct AcrossLaunch {
  double streamed, kind;
  int copies;  // of the output, in 16-bit elements
  bool f32, lines;
  int off;  // copies of rows that 16-byte stores don't fit, or end inside one (the times above know only the others)
};
double across_us(const iris_gemm_args& a, const AcrossTime& t, int parts, const AcrossLaunch& l, bool off = false) {
  const int64_t items = ((int64_t)a.M + t.cm - 1) / t.cm * (((int64_t)a.N + t.cn - 1) / t.cn) * parts;
  const int64_t rounds = (items + a.num_sms - 1) / a.num_sms, nk = ((int64_t)a.K + 63) / 64, steps = (nk + parts - 1) / parts;
  const double busy = rounds > 1 ? 1.0 : (double)items / a.num_sms, area = (double)t.cm * t.cn / 4096;
  const double step = (l.f32 ? t.step_f32 * (1 + 0.059 * busy) : t.step * (1 + 0.112 * busy) * (1 + 0.404 * l.streamed)) * (l.lines ? 1.0 : 1.223) * l.kind;
  const double loop = t.tile + steps * step, store = area / parts * (0.377 * (l.copies - 1) + (off ? 1 + l.off : 0)) * (busy > 0.37 ? busy : 0.37);
  const double mb = items * area / 64, low = mb < 16 ? mb : 16;
  const double hand = parts > 1 ? 3.210 + 0.417 * area + 0.114 * low + 0.092 * (mb - low) + 0.151 * parts : 0;
  return 3.946 + 0.920 * busy + rounds * loop + store * (1 + (rounds - 1) * 0.67) + hand;
}

// Replaces the plan of a launch in tiles where tiles of another size, that lie across the caller's (plan_cover), are expected to be
// faster by more than an eighth.  (us, the caller's tiles or what the plans above made of
// them / so: fp32 [1972,448] x [448,696] in 256 x 256 tiles, whose 128 x 128 ones a program computes in turn, 136 / 25; [2152,22464] x
// [22464,384] in 256 x 256 tiles 105 / 59; [668,16256] x [16256,960] in 256 x 64 55 / 41; [916,2240] x [2240,5184] in 256 x 256 46 / 29;
// [108,27664] x [27664,4032] in 256 x 64 137 / 74.  Of 370 random calls in tiles 45 change, 1.024x on average over all of them; slower
// by more than 3 %: two, by 5 %.  Small tiles two to a CU are not in the fit: only where K is long.)
void plan_across(const iris_gemm_args& a, Plan* plan) {
  const GemmKernelEntry* own = plan->entry;
  if (!own || plan->skinny || plan->in_program || plan->last_round || plan->rest || plan->k.stream_k) return;
  if (a.epilogue == IRIS_EPI_ATOMIC_ADD || a.variant != 0 || a.split_k != 0 || a.mm_begin_timestamp || a.mm_end_timestamp) return;
  if (a.num_sms != current_cu_count() || a.K <= 0) return;
  const bool flags = a.epilogue == IRIS_EPI_ALL_SCATTER ? a.notify != 0 : a.world_size > 1;
  const int64_t own_tiles = flags ? ((int64_t)a.M + a.block_m - 1) / a.block_m * (((int64_t)a.N + a.block_n - 1) / a.block_n) : 0;
  const int64_t least = arrival_words(own_tiles, 2);  // (words that the arrivals need)
  if (flags && (!a.locks || least > a.num_sms || a.flag_sem == IRIS_FLAG_SEM_RELEASE_ACQUIRE)) return;
  const bool scatter = a.epilogue == IRIS_EPI_ALL_SCATTER;
  AcrossLaunch l;
  const double mb = ((double)a.M + a.N) * a.K * 2e-6;
  l.streamed = mb < 50 ? 0 : mb > 150 ? 1 : (mb - 50) / 100;
  l.kind = !own->dma ? 1.368 : own->loose ? 1.177 : own->b_rows ? 1.023 : 1.0;
  l.copies = (scatter ? a.world_size : 1) * ((scatter ? a.c_global_dtype : a.c_dtype) == IRIS_DTYPE_F32 ? 2 : 1);
  l.f32 = a.ab_dtype == IRIS_DTYPE_F32;
  l.lines = whole_lines(a);
  constexpr int TILES = sizeof(ACROSS_TIMES) / sizeof(ACROSS_TIMES[0]);
  double own_us = -1;
  for (const AcrossTime& t : ACROSS_TIMES)
    if (t.cm == own->cm && t.cn == own->cn && !(l.f32 && t.step_f32 == 0)) own_us = across_us(a, t, plan->k.split_k, l);
  if (plan->k.num_sms != a.num_sms && a.K < 2048) return;
  const int own_parts = plan->k.split_k;
  // (what the times above are not good for: K in this many parts, and small tiles that share it, whose operands the L2s hold)
  if (own_parts > 12 || (own_parts > 2 && own->cm * own->cn == 64 * 64)) return;
  if (own_us < 12) return;  // (another tile than these, or nothing to gain that the search would not cost)
  // (one or two K-steps: the stores are most of it, and other tiles than the caller's are 0.99 of the time over 17 random calls,
  // 1.44 at most)
  if (a.K <= 128 && own->dma && plan->k.merge_m * plan->k.merge_n == 1) return;
  const int es = dtype_size(scatter ? a.c_global_dtype : a.c_dtype);
  l.off = !plan->k.vec_out || (int64_t)a.N * es % 16 != 0 ? (scatter ? a.world_size : 1) : 0;
  const AcrossTime* own_time = nullptr;
  for (const AcrossTime& t : ACROSS_TIMES)
    if (t.cm == own->cm && t.cn == own->cn) own_time = &t;
  double best_us[TILES];
  int best_parts[TILES];
  const int64_t room = a.partials && a.locks && aligned16(a.partials) ? a.num_sms * a.partials_slot_elems : 0;
  for (int i = 0; i < TILES; ++i) {
    const AcrossTime& t = ACROSS_TIMES[i];
    best_us[i] = 1e30;
    if ((l.f32 && t.step_f32 == 0) || !can_cover(a, t.cm, t.cn, 0)) continue;
    const int64_t tiles = ((int64_t)a.M + t.cm - 1) / t.cm * (((int64_t)a.N + t.cn - 1) / t.cn), elems = tiles * t.cm * t.cn;
    if (tiles > 4 * (int64_t)a.num_sms) continue;
    int most = (int)((a.num_sms - least) / tiles);
    if (most > 12) most = 12;
    if (most > (a.K + 63) / 64 / 4) most = (a.K + 63) / 64 / 4;
    for (int parts = 1; parts == 1 || parts <= most; parts += parts < 4 || parts + 2 > most ? 1 : 2) {
      // (two parts of a tile of 128 accumulators hand half of it over each)
      const bool half = parts == 2 && t.cm * t.cn >= 256 * 128;
      // (K of a 128 x 128 tile stays shared out rather than the tile cut, as plan_small has it)
      if (parts == 1 && own_parts > 1 && a.block_m < 256 && t.cm * t.cn < own->cm * own->cn) continue;
      if (parts > 1 && elems * parts > room * (half ? 2 : 1)) break;
      const double us = across_us(a, t, parts, l);
      if (us < best_us[i]) best_us[i] = us, best_parts[i] = parts;
    }
  }
  // the least of them that there is a kernel for
  for (;;) {
    int i = 0;
    for (int j = 1; j < TILES; ++j)
      if (best_us[j] < best_us[i]) i = j;
    const AcrossTime& t = ACROSS_TIMES[i];
    if (best_us[i] > 0.87 * own_us) return;
    // (us a pass, the caller's tiles / so, without this: [1034,64] x [64,2135] to eight 31 / 42, [753,467] x [467,3183] 45 / 58; of 541
    // random calls that were planned so 27 keep theirs for it and the line of K above, 1.04x slower so on average)
    if (l.off && across_us(a, t, best_parts[i], l, true) > 0.95 * across_us(a, *own_time, own_parts, l, true)) {
      best_us[i] = 1e30;
      continue;
    }
    // (a word for each of the caller's tiles where they have room beside those of the parts of K)
    const int64_t used = best_parts[i] > 1 ? ((int64_t)a.M + t.cm - 1) / t.cm * (((int64_t)a.N + t.cn - 1) / t.cn) * best_parts[i] : 0;
    const int pack = used + own_tiles <= a.num_sms ? 0 : 2;
    Plan across;
    if (can_cover(a, t.cm, t.cn, pack) && plan_cover(a, t.cm, t.cn, best_parts[i], arrival_words(own_tiles, pack), pack, &across) && across.k.split_k == best_parts[i] && no_slower_loader(*across.entry, *own)) {
      across.parts = 2;
      *plan = std::move(across);
      return;
    }
    best_us[i] = 1e30;
  }
}

hipError_t make_plan_tiles(const iris_gemm_args& a, Plan* plan) {
  if (a.epilogue == IRIS_EPI_ONE_SHOT && a.phase == IRIS_PHASE_FUSED) {
    iris_gemm_args b = a;
    b.phase = IRIS_PHASE_TWO_KERNELS;
    Plan behind;
    if (a.split_k <= 1 && a.split_k != IRIS_GEMM_SPLIT_STREAM_K && make_plan_units(b, &behind) == hipSuccess &&
        (!reduce_in_program(a, behind) || (behind.reduces && !behind.loose && !behind.b_rows && a.variant == 0))) {
      // (inside, few rows and cells of aligned operands are faster than the caller's tiles with their own reduce: us a pass, [125,384] x
      // [384,1216] of 2, 64 x 64 tiles 9.9 / 8.8, [82,128] x [128,4120] of 8 11.3 / 10.8.  A variant that was asked for is not among
      // the programs that reduce, or is one of them.)
      *plan = behind;
      plan->two_kernels = !reduce_in_program(a, behind);
      return hipSuccess;
    }
  }
  if (plan_small(a, plan)) {
    plan_atomics(a, plan);
    plan_across(a, plan);
    return hipSuccess;
  }
  const bool plain = a.variant == 0 && a.split_k == 0 && !a.mm_begin_timestamp && !a.mm_end_timestamp &&
                     !(a.epilogue == IRIS_EPI_ONE_SHOT && a.phase != IRIS_PHASE_PRODUCE && a.phase != IRIS_PHASE_TWO_KERNELS) &&
                     a.epilogue != IRIS_EPI_ATOMIC_ADD && a.num_sms > 0 && (a.block_m == 128 || a.block_m == 256) &&
                     (a.block_n == 64 || a.block_n == 128) && a.M >= 256;
  if (plain && plan_blocks(a, plan)) {
    plan_across(a, plan);
    return hipSuccess;
  }
  const hipError_t err = make_plan_body(a, plan);
  own_flags(plan);
  if (err == hipSuccess) {
    split_last_round(a, plan);
    plan_atomics(a, plan);
    plan_across(a, plan);
  }
  return err;
}

hipError_t make_plan_body(const iris_gemm_args& a, Plan* plan, bool cells) {
  if (a.M < 0 || a.N < 0 || a.K < 0) return hipErrorInvalidValue;
  if (a.block_m <= 0 || a.block_n <= 0 || a.group_size_m <= 0) return hipErrorInvalidValue;
  if (a.num_sms <= 0 || a.num_xcds <= 0 || (a.num_sms % a.num_xcds) != 0) return hipErrorInvalidValue;
  if (a.world_size <= 0 || a.cur_rank < 0 || a.cur_rank >= a.world_size) return hipErrorInvalidValue;
  if (a.world_size > 1 && a.heap_bases == nullptr) return hipErrorInvalidValue;
  if (a.ab_dtype != IRIS_DTYPE_BF16 && a.ab_dtype != IRIS_DTYPE_F16 && a.ab_dtype != IRIS_DTYPE_F32)
    return hipErrorInvalidValue;

  int op, out_dt;
  GemmKArgs& k = plan->k;
  k = GemmKArgs{};
  switch (a.epilogue) {
    case IRIS_EPI_ALL_SCATTER:
      if (!a.c_global) return hipErrorInvalidValue;
      out_dt = a.c_global_dtype;
      op = out_dt == IRIS_DTYPE_F32 ? OP_STORE32 : OP_STORE16;
      k.out = static_cast<char*>(a.c_global) +
              (int64_t)a.cur_rank * a.N * a.stride_cn_global * dtype_size(out_dt);
      k.som = a.stride_cm_global;
      k.son = a.stride_cn_global;
      k.dest_all = 1;
      k.flag_mode = a.notify ? 1 : 0;
      break;
    case IRIS_EPI_ATOMIC_ADD:
      if (!a.c_global) return hipErrorInvalidValue;
      out_dt = a.c_global_dtype;
      op = out_dt == IRIS_DTYPE_F32 ? OP_ATOMIC32 : OP_ATOMIC16;
      k.out = static_cast<char*>(a.c_global);
      k.som = a.stride_cm_global;
      k.son = a.stride_cn_global;
      k.dest_all = 1;
      k.flag_mode = 0;
      break;
    case IRIS_EPI_ONE_SHOT:
      if (!a.c || !a.c_global) return hipErrorInvalidValue;
      if (a.phase != IRIS_PHASE_PRODUCE && a.phase != IRIS_PHASE_CONSUME && a.phase != IRIS_PHASE_FUSED &&
          a.phase != IRIS_PHASE_TWO_KERNELS)
        return hipErrorInvalidValue;
      out_dt = a.c_dtype;
      op = out_dt == IRIS_DTYPE_F32 ? OP_STORE32 : OP_STORE16;
      k.out = static_cast<char*>(a.c);
      k.som = a.stride_cm;
      k.son = a.stride_cn;
      k.dest_all = 0;
      k.flag_mode = 2;
      plan->in_program = a.phase == IRIS_PHASE_FUSED ? 1 : 0;
      plan->fused_reduce = (a.phase == IRIS_PHASE_CONSUME || a.phase == IRIS_PHASE_TWO_KERNELS) ? 1 : 0;
      if (!(a.phase & IRIS_PHASE_PRODUCE)) return hipSuccess;  // consumer only: no GEMM
      if (plan->in_program) {
        const int gdt = a.c_global_dtype;
        if (gdt != IRIS_DTYPE_F32 && gdt != IRIS_DTYPE_F16 && gdt != IRIS_DTYPE_BF16) return hipErrorInvalidValue;
        k.cg = static_cast<char*>(a.c_global);
        k.sgm = a.stride_cm_global;
        k.sgn = a.stride_cn_global;
        k.cg_dt = gdt;
      }
      break;
    default:
      return hipErrorInvalidValue;
  }
  if (out_dt != IRIS_DTYPE_F32 && out_dt != a.ab_dtype) return hipErrorInvalidValue;
  if (a.touch_ahead != IRIS_GEMM_TOUCH_AUTO && a.touch_ahead != IRIS_GEMM_TOUCH_ON && a.touch_ahead != IRIS_GEMM_TOUCH_OFF)
    return hipErrorInvalidValue;
  if (a.flag_sem != IRIS_FLAG_SEM_WRITE_THROUGH && a.flag_sem != IRIS_FLAG_SEM_RELEASE_ACQUIRE)
    return hipErrorInvalidValue;
  if (k.flag_mode != 0 && a.flag_sem == IRIS_FLAG_SEM_RELEASE_ACQUIRE) k.flag_mode |= FLAG_RELEASE;
  if (k.flag_mode != 0 && a.world_size > 1 && !a.tile_completed) return hipErrorInvalidValue;
  if ((k.flag_mode & FLAG_MODE_MASK) == 1 && !a.tile_completed) return hipErrorInvalidValue;
  if (a.M == 0 || a.N == 0) return hipSuccess;  // nothing to compute
  if (!a.a || !a.b) {
    if (a.K > 0) return hipErrorInvalidValue;
  }

  k.a = static_cast<const char*>(a.a);
  k.b = static_cast<const char*>(a.b);
  k.flags = a.tile_completed;
  k.heap_bases = a.heap_bases;
  k.ts_begin = a.mm_begin_timestamp;
  k.ts_end = a.mm_end_timestamp;
  k.sam = a.stride_am;
  k.sak = a.stride_ak;
  k.sbk = a.stride_bk;
  k.sbn = a.stride_bn;
  k.M = a.M;
  k.N = a.N;
  k.K = a.K;
  k.BM = a.block_m;
  k.BN = a.block_n;
  k.G = a.group_size_m;
  k.num_sms = a.num_sms;
  k.num_xcds = a.num_xcds;
  k.cur_rank = a.cur_rank;
  k.ws = a.world_size;
  k.num_pid_m = (a.M + a.block_m - 1) / a.block_m;
  k.num_pid_n = (a.N + a.block_n - 1) / a.block_n;
  k.total_tiles = k.num_pid_m * k.num_pid_n;
  k.sys = a.scope == IRIS_SCOPE_SYSTEM;
  k.row_out = k.son == 1;
  k.vec_out = vec_ok(k.out, k.som, k.son, dtype_size(out_dt)) ? 1 : 0;
  if (plan->in_program) {
    // 16-byte strips in the in-program reduce: aligned rows on both sides, tile
    // origins on strip boundaries, rows at least as long as the matrix is wide
    // and 32-bit offsets inside a tile
    const int ies = dtype_size(out_dt), oes = dtype_size(k.cg_dt), ve = 16 / ies;
    k.fused_vec = k.vec_out && vec_ok(k.cg, k.sgm, k.sgn, oes) && a.block_n % ve == 0 && (a.block_n * oes) % 16 == 0 &&
                  k.som >= a.N && k.sgm >= a.N && ((int64_t)a.block_m + 64) * k.som * ies < (1ll << 31) &&
                  ((int64_t)a.block_m + 64) * k.sgm * oes < (1ll << 31);
  }

  int count = 0;
  const GemmKernelEntry* list = entries_for(a.ab_dtype, op, &count);
  if (!list) return hipErrorInvalidValue;

  // Operands fit the LDS-DMA loader when both are K-contiguous with 16-byte
  // aligned rows and K is a multiple of 8; a compute tile's rows must stay
  // within a 2 GiB window of its buffer descriptor.
  // (an fp32 launch arrives here with K and the operands' strides in 16-bit units: make_plan)
  const int unit = a.ab_dtype == IRIS_DTYPE_F32 ? 2 : 1;
  const bool dma_ok = a.stride_ak == unit && a.stride_bk == unit && (a.stride_am % 8) == 0 && (a.stride_bn % 8) == 0 &&
                      aligned16(a.a) && aligned16(a.b) && (a.K % 8) == 0 && a.stride_am > 0 && a.stride_bn > 0;
  // The gathering loader takes operands that are contiguous in one direction, with at least one 16-byte load of them
  // in it (a load at the edge is moved back inside), a block of eight rows when that direction is across K, and
  // 32-bit offsets inside a tile.
  const bool a_along = a.stride_ak == unit && a.K >= 8, b_along = a.stride_bk == unit && a.K >= 8;
  const bool a_across = !a_along && a.stride_am == unit && a.M >= 8, b_across = !b_along && a.stride_bn == unit && a.N >= 8;
  k.a_across = a_across;
  k.b_across = b_across;
  // A row-major B goes through the LDS-DMA too where its rows are whole aligned 16-byte chunks and all of it, K rows, lies
  // within the 2 GiB window of a descriptor.  (us a pass gathered / so / the same weight along K, 256 x 64 tiles:
  // [2048,4096] x [4096,1376] 81.6 / 34.2 / 34.5, [2697,1936] x [1936,1600] 77.9 / 30.9 / 32.6, [1232,29704] x [29704,512] 129 / 97 /
  // 87; 64 x 64 [50,2752] x [2752,7040] 26.1 / 16.6 / 16.3; cells [42,320] x [320,3968] 8.7 / 6.2 / 6.1.  21 random calls in tiles take
  // 0.87 to 1.12 of the time along K, 0.99 on average; 33 in cells 0.93 to 1.5, 1.15 on average, the more the longer K is.)
  const bool rows_ok = !dma_ok && unit == 1 && a.stride_ak == 1 && a.stride_am > 0 && (a.stride_am % 8) == 0 && (a.K % 8) == 0 &&
                       a.stride_bn == 1 && a.stride_bk > 0 && (a.stride_bk % 8) == 0 && (a.N % 8) == 0 && aligned16(a.a) &&
                       aligned16(a.b) && ((int64_t)256 * a.stride_am + a.K) * 2 < ((int64_t)1 << 31) &&
                       ((int64_t)(a.K > 128 ? a.K : 128) * a.stride_bk + 256) * 2 < ((int64_t)1 << 31);
  // Operands along K at any alignment and of any K from eight on: the same tiles, built to take them (LOAD_DMA_LOOSE; us a
  // pass gathered / so / with one k less, aligned: 256 x 64 tiles [2048,4097] x [4097,1376] 60.1 / 42.8 / 34.5, [2871,4865] x
  // [4865,5952] 409 / 266 / 187, 128 x 128 [3929,1153] x [1153,576] 22.3 / 18.5 / 13.4; 21 random calls in tiles take 1.12 to 1.9 of
  // the aligned time, 1.3 on average, 37 in cells and few rows 1.07 to 1.4, 1.2 on average).  Rows
  // that overlap stay with the gathering tiles: past the edge, a chunk could straddle the end of the descriptor.
  const bool loose_ok = !dma_ok && a.stride_ak == unit && a.stride_bk == unit && a.K >= 8 && a.stride_am >= a.K &&
                        a.stride_bn >= a.K && ((int64_t)256 * a.stride_am + a.K + 8) * 2 < ((int64_t)1 << 31) &&
                        ((int64_t)256 * a.stride_bn + a.K + 8) * 2 < ((int64_t)1 << 31);
  auto gatherable = [&](bool along, bool across, int rows, int bk, int64_t ld_row, int64_t ld_k, int64_t extent) {
    const int64_t lim = (int64_t)1 << 30;  // 16-bit units
    return (along && ld_row >= 0 && rows * ld_row + a.K < lim) ||
           (across && ld_k >= 0 && bk * ld_k + extent * unit < lim);
  };
  auto fits = [&](const GemmKernelEntry& e) {
    if (e.gather)
      return gatherable(a_along, a_across, e.cm, e.bk, a.stride_am, a.stride_ak, a.M) &&
             gatherable(b_along, b_across, e.cn, e.bk, a.stride_bn, a.stride_bk, a.N);
    if (!e.dma) return true;
    if (e.b_rows) return rows_ok;
    if (e.loose) return loose_ok;
    if (!dma_ok) return false;
    const int64_t lim = (int64_t)1 << 31;
    return ((int64_t)e.cm * a.stride_am + a.K) * 2 < lim && ((int64_t)e.cn * a.stride_bn + a.K) * 2 < lim;
  };

  if (a.variant == 0 || a.variant == IRIS_GEMM_VARIANT_FEW_ROWS) {
    // (insisted on, it is for aligned operands)
    const bool any_ok = dma_ok || (loose_ok && a.variant == 0);
    if (plan_few_rows(a, op, any_ok, !dma_ok, plan)) return hipSuccess;
    if (cells && plan_cells(a, op, any_ok || (rows_ok && a.variant == 0), !dma_ok && !rows_ok, rows_ok, plan)) return hipSuccess;
    if (a.variant == IRIS_GEMM_VARIANT_FEW_ROWS) return hipErrorInvalidValue;
  }

  const GemmKernelEntry* pick = nullptr;
  if (a.variant == IRIS_GEMM_VARIANT_PERSISTENT) {
    // the default choice among the persistent kernels
  } else if (a.variant > 0) {
    if (a.variant > count) return hipErrorInvalidValue;
    const GemmKernelEntry& e = list[a.variant - 1];
    if (!fits(e)) return hipErrorInvalidValue;
    pick = &e;
  }
  if (!pick) {
    // first entry whose compute tile divides the logical tile; the rows and
    // columns a small matrix cannot fill are not worth a tall compute tile
    int more = 0, dma = 0;
    const GemmKernelEntry* more_list = more_entries_for(a.ab_dtype, op, &more);
    const GemmKernelEntry* dma_list = rows_ok    ? rows_entries_for(a.ab_dtype, op, &dma)
                                      : loose_ok ? loose_entries_for(a.ab_dtype, op, &dma)
                                                 : nullptr;
    for (int i = -dma; i < more + count && !pick; ++i) {
      const GemmKernelEntry& e = i < 0 ? dma_list[i + dma] : i < more ? more_list[i] : list[i - more];
      if (i < more && a.ab_dtype == IRIS_DTYPE_F32 && a.K < LONG_STEPS * e.bk) continue;
      // (the gathering tiles are for what the DMA does not take, and for the reduce inside the program, of which there are
      // builds for aligned operands along K only)
      if (!fits(e) || (e.gather && (dma_ok || (dma > 0 && !plan->in_program)))) continue;
      if (plan->in_program && !e.fn_fused) continue;
      // (a caller's split needs a K-step per part: a tile with a deeper step may not have them)
      if (a.split_k > 1 && a.split_k > (a.K + e.bk - 1) / e.bk && e.bk > 64) continue;
      if (a.block_m % e.cm != 0 || a.block_n % e.cn != 0) continue;
      // (up to half a tall tile may be padding: its rows cost matrix-core time only, and
      // the tall tiles are the ones whose K range can be shared out over idle programs)
      if (e.cm > 64 && e.cm >= 4 * a.M) continue;
      if (e.cn > 64 && e.cn >= 4 * a.N) continue;
      // (a row-major B, and rows off the 16 bytes, come at no more than half the rate into the half of a tile that is padding)
      if (e.cn > 128 && (e.b_rows || e.loose) && e.cn >= 2 * a.N) continue;
      // An atomic epilogue is bound by the chip's atomic rate (329 G fp32
      // adds a second, 51 us for 4096 x 4096), and while a program walks its
      // K loop it sends none: with two half tiles per logical tile the
      // second's K loop runs while the first's atomics drain (-7 % per launch).
      if ((op == OP_ATOMIC32 || op == OP_ATOMIC16) && e.cm * e.cn > 256 * 128) continue;
      pick = &e;
    }
    // otherwise 64 x 64, with masked sub-tiles: gathered if the operands allow it, else element by element
    for (int i = 0; i < more + count && !pick; ++i) {
      const GemmKernelEntry& e = i < more ? more_list[i] : list[i - more];
      if (i < more && a.ab_dtype == IRIS_DTYPE_F32) continue;
      if (!e.dma && e.cm == 64 && e.cn == 64 && fits(e) && !(plan->in_program && !e.fn_fused)) pick = &e;
    }
  }
  if (!pick) return hipErrorInvalidValue;
  if (plan->in_program && !pick->fn_fused) return hipErrorInvalidValue;
  // compute tiles per logical tile; a matrix smaller than one logical tile
  // has nothing beyond its own edge
  const int span_m = a.block_m < a.M ? a.block_m : a.M, span_n = a.block_n < a.N ? a.block_n : a.N;
  k.sub_m = (span_m + pick->cm - 1) / pick->cm;
  k.sub_n = (span_n + pick->cn - 1) / pick->cn;
  plan->entry = pick;

  const hipError_t err = plan_split(a, *pick, plan->in_program != 0, &k);
  launch_constants(a, *pick, &k);
  // (under stream-K every program has a run: the reference's XCD remap stays)
  if (err != hipSuccess || k.stream_k) return err;
  // A tile whose stages take at most half a CU's LDS runs one wave per SIMD
  // and has every instruction of a K-step on its critical path.  A launch
  // that owns the whole device (one program per CU or more) and has at least
  // two such tiles per program is given two programs per CU, each other's
  // cover: which program computes which tile is not observable, the tiles'
  // flags are.  (64 x 64 tiles, 256 -> 512 programs: [512,1376] x [1376,4096]
  // 25.0 -> 17.8 us, [2048,4096] x [4096,1376] 80 -> 65 us.)
  const int64_t items = (int64_t)k.total_tiles * k.sub_m * k.sub_n;
  // (Two programs of a tile with fetching waves are slower than one, so such a launch takes
  // the plain tile of the same shape: [512,1376] x [1376,4096] 20.6 -> 17.1 us.)
  const GemmKernelEntry* twin = a.variant > 0 ? nullptr : plain_twin(list, count, *pick);
  const bool two_ok = pick->fetch_waves == 0 || twin;
  if (!plan->in_program && !plan->one_per_cu && k.split_k == 1 && two_ok && (twin ? twin : pick)->lds_bytes * 2 <= 160 * 1024 &&
      a.num_sms >= current_cu_count() && a.num_sms <= 2 * current_cu_count() && items >= 2 * (int64_t)a.num_sms &&
      !a.mm_begin_timestamp && !a.mm_end_timestamp) {
    k.num_sms = 2 * a.num_sms;
    if (twin) plan->entry = twin;
  }
  // (A split launch of a 128-accumulator tile runs the `_f4` build too: its split build handles one (tile, part)
  // item per program and keeps nothing live across the epilogue, which leaves it 40 registers to spare.  Before
  // that it spilled around the hand-over, now and then inside the K loop, and such launches took the plain tile:
  // [8192,12288] x [12288,512] as 128 tiles of 256 x 128 in two parts 145 us, against 131 or 181 as the spills fell.)
  return hipSuccess;
}

hipError_t ensure_lds(GemmKernelFn fn, int lds_bytes) {
  // dynamic LDS above 64 KiB must be opted into once per function and device
  static std::mutex m;
  static std::vector<std::pair<int, GemmKernelFn>> done;
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  std::lock_guard<std::mutex> lock(m);
  for (const auto& d : done)
    if (d.first == dev && d.second == fn) return hipSuccess;
  err = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  if (err == hipSuccess) done.emplace_back(dev, fn);
  return err;
}

iris_reduce_args reduce_args_from(const iris_gemm_args& a) {
  iris_reduce_args r{};
  r.c = a.c;
  r.c_global = a.c_global;
  r.tile_completed = a.tile_completed;
  r.heap_bases = a.heap_bases;
  r.status = a.status;
  r.M = a.M;
  r.N = a.N;
  r.stride_cm = a.stride_cm;
  r.stride_cn = a.stride_cn;
  r.stride_cm_global = a.stride_cm_global;
  r.stride_cn_global = a.stride_cn_global;
  r.block_m = a.block_m;
  r.block_n = a.block_n;
  r.group_size_m = a.group_size_m;
  // A launch that owns the device leaves the reduce its own grid, two groups a CU: with one (num_sms programs) HBM is
  // not kept busy (8 x fp32 [8192,8192] 477 us instead of 359).
  r.num_sms = a.num_sms >= current_cu_count() ? 0 : a.num_sms;
  r.num_xcds = a.num_xcds;
  r.cur_rank = a.cur_rank;
  r.world_size = a.world_size;
  r.c_dtype = a.c_dtype;
  r.c_global_dtype = a.c_global_dtype;
  r.scope = a.scope;
  r.wait_flags = 1;
  r.variant = 0;
  r.spin_timeout_ticks = a.spin_timeout_ticks;
  r.flag_sem = a.flag_sem;
  return r;
}

}  // namespace
}  // namespace iris_amd

using namespace iris_amd;

namespace {

// Whether the plan's launch is the build that touches lines of K-steps to come (launch_constants decides; a
// launch that splits K has no such build).
bool plan_touches(const Plan& plan) {
  const GemmKernelEntry* e = plan.entry;
  return e && !plan.skinny && !plan.in_program && plan.k.split_k == 1 && !plan.k.stream_k && plan.k.pf_dist > 0 && e->fn_touch;
}

// The build of the picked kernel that the plan launches.
GemmKernelFn plan_fn(const Plan& plan) {
  const GemmKernelEntry* e = plan.entry;
  if (plan.in_program) return e->fn_fused;
  const bool split = plan.k.split_k > 1 || plan.k.stream_k;
  const bool touch = plan_touches(plan);
  if (plan.remap_flags) return split ? e->fn_split_merged : touch ? e->fn_touch_merged : e->fn_merged;
  return split ? e->fn_split : touch ? e->fn_touch : e->fn;
}

// Enqueue what `plan` describes on `stream`.  (`args` is the caller's launch: only a reduce kernel behind the GEMM
// reads it.)
hipError_t run_plan(const Plan& plan, const iris_gemm_args& args, void* stream) {
  hipError_t err = hipSuccess;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (plan.skinny) {
    if (dbg())
      std::fprintf(stderr, "[iris_amd] gemm few-rows M=%d N=%d K=%d tiles=%d grid=%dx%dx%d\n", plan.k.M, plan.k.N, plan.k.K,
                   plan.k.total_tiles, plan.skinny_grid, plan.skinny_grid_y, plan.skinny_grid_z);
    if (plan.skinny_lds > 64 * 1024) {
      err = ensure_lds(plan.skinny, plan.skinny_lds);
      if (err != hipSuccess) return err;
    }
    hipLaunchKernelGGL(plan.skinny, dim3(plan.skinny_grid, plan.skinny_grid_y, plan.skinny_grid_z), dim3(SKINNY_THREADS), plan.skinny_lds, s,
                       plan.k);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
  } else if (plan.entry) {
    const GemmKernelEntry* e = plan.entry;
    const GemmKernelFn fn = plan_fn(plan);
    if (e->lds_bytes > 64 * 1024) {
      err = ensure_lds(fn, e->lds_bytes);
      if (err != hipSuccess) return err;
    }
    if (dbg())
      std::fprintf(stderr, "[iris_amd] gemm %s%s M=%d N=%d K=%d tiles=%d grid=%d sub=%dx%d lds=%d\n", e->name,
                   plan.in_program ? "+reduce" : "", plan.k.M, plan.k.N, plan.k.K, plan.k.total_tiles, plan.k.num_sms,
                   plan.k.sub_m, plan.k.sub_n, e->lds_bytes);
    hipLaunchKernelGGL(fn, dim3(plan.k.num_sms), dim3(e->threads), e->lds_bytes, s, plan.k);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    if (plan.last_round) {
      if (e->lds_bytes > 64 * 1024) {
        err = ensure_lds(e->fn_split, e->lds_bytes);
        if (err != hipSuccess) return err;
      }
      if (dbg())
        std::fprintf(stderr, "[iris_amd] gemm %s: last round, tiles %d..%d in %d parts\n", e->name,
                     plan.k_last.tile_base, plan.k_last.tile_base + plan.k_last.total_tiles - 1, plan.k_last.split_k);
      hipLaunchKernelGGL(e->fn_split, dim3(plan.k_last.num_sms), dim3(e->threads), e->lds_bytes, s, plan.k_last);
      err = hipGetLastError();
      if (err != hipSuccess) return err;
    }
  }
  if (plan.rest) {
    err = run_plan(*plan.rest, args, stream);
    if (err != hipSuccess) return err;
  }
  if (plan.fused_reduce) {
    // The consumer half of the one-shot epilogue runs as a second kernel on
    // the same stream: it waits for each tile's flag, sums the partials and
    // stores the result, exactly what the tail of the reference program does
    // for that tile (gemm_one_shot_all_reduce.py:220-271).
    const iris_reduce_args r = reduce_args_from(args);
    return static_cast<hipError_t>(iris_one_shot_reduce_launch(&r, stream));
  }
  return hipSuccess;
}

}  // namespace

extern "C" int iris_gemm_launch(const iris_gemm_args* args, void* stream) {
  if (!args) return hipErrorInvalidValue;
  Plan plan;
  hipError_t err = make_plan(*args, &plan);
  if (err != hipSuccess) return err;
  return run_plan(plan, *args, stream);
}

// ---------------------------------------------------------------------------
// The launch that allocates nothing: the split-K / stream-K / few-rows
// workspace (partial tiles and their locks) lives in a device array of this
// library instead of in buffers of the caller.
// ---------------------------------------------------------------------------

namespace {

constexpr size_t NOALLOC_LOCK_BYTES = 4096;  // int32[1024]: one lock per program or tile
constexpr size_t NOALLOC_PARTIAL_BYTES =
    (size_t)IRIS_GEMM_NOALLOC_MAX_PROGRAMS * IRIS_GEMM_NOALLOC_MAX_TILE_ELEMS * sizeof(float);
constexpr size_t NOALLOC_BYTES = NOALLOC_LOCK_BYTES + NOALLOC_PARTIAL_BYTES;

}  // namespace

// locks first, then one partial-tile slot per program.  Every device the
// library runs on holds its own copy until the process ends.
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

namespace {

__global__ __launch_bounds__(256) void fill_i32_kernel(int32_t* p, int32_t v, int n) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = v;
}

// Device address of `scratch` on the current device, looked up once per
// device.  (In host code the array's name is only a handle for this lookup.)
hipError_t scratch_address(unsigned char** out) {
  static std::mutex m;
  static unsigned char* ptr[64] = {};
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(m);
  if (!ptr[dev]) {
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess) return err;
    if (!p) return hipErrorInvalidSymbol;
    ptr[dev] = static_cast<unsigned char*>(p);
  }
  *out = ptr[dev];
  return hipSuccess;
}

}  // namespace

extern "C" int iris_gemm_launch_noalloc(const iris_gemm_args* args, void* stream) {
  if (!args) return hipErrorInvalidValue;
  if (args->num_sms > IRIS_GEMM_NOALLOC_MAX_PROGRAMS) {
    std::fprintf(stderr, "[iris_amd] iris_gemm_launch_noalloc: num_sms %d exceeds the workspace's %d programs\n",
                 args->num_sms, IRIS_GEMM_NOALLOC_MAX_PROGRAMS);
    return hipErrorInvalidValue;
  }
  const int64_t tile_elems = (int64_t)args->block_m * args->block_n;
  const bool forced = args->split_k > 1 || args->split_k == IRIS_GEMM_SPLIT_STREAM_K;
  if (forced && tile_elems > IRIS_GEMM_NOALLOC_MAX_TILE_ELEMS) {
    std::fprintf(stderr,
                 "[iris_amd] iris_gemm_launch_noalloc: a split of K was asked for, and a %d x %d tile exceeds the "
                 "workspace's %d elements per partial tile\n",
                 args->block_m, args->block_n, IRIS_GEMM_NOALLOC_MAX_TILE_ELEMS);
    return hipErrorInvalidValue;
  }
  unsigned char* base = nullptr;
  hipError_t err = scratch_address(&base);
  if (err != hipSuccess) return err;

  iris_gemm_args a = *args;
  a.locks = reinterpret_cast<int32_t*>(base);
  // tiles beyond the slot size run unsplit, exactly as without a workspace
  a.partials = tile_elems <= IRIS_GEMM_NOALLOC_MAX_TILE_ELEMS ? reinterpret_cast<float*>(base + NOALLOC_LOCK_BYTES) : nullptr;
  a.partials_slot_elems = a.partials ? IRIS_GEMM_NOALLOC_MAX_TILE_ELEMS : 0;
  Plan plan;
  err = make_plan(a, &plan);
  if (err != hipSuccess) return err;
  // The array keeps what the last call left: the locks must start at zero (a
  // wait that timed out leaves one raised).  A fill kernel, not a memset, so
  // that the call can be recorded into a HIP graph.
  auto needs_locks = [](const Plan& q) {
    const bool handed = q.k.split_k > 1 && q.k.sliced != SPLIT_DIRECT;
    return (q.skinny && (q.k.flag_mode != 0 || q.skinny_grid_z > 1)) || q.k.cover_bm > 0 || (q.entry && (handed || q.k.stream_k || q.last_round));
  };
  const bool uses_locks = needs_locks(plan) || (plan.rest && needs_locks(*plan.rest));
  if (uses_locks) {
    hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(256), 0, static_cast<hipStream_t>(stream), a.locks, 0,
                       (int)(NOALLOC_LOCK_BYTES / sizeof(int32_t)));
    err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return run_plan(plan, a, stream);
}

extern "C" int iris_gemm_split_k(const iris_gemm_args* args, int* split_k) {
  if (!args || !split_k) return hipErrorInvalidValue;
  Plan plan;
  hipError_t err = make_plan(*args, &plan);
  if (err != hipSuccess) return err;
  *split_k = plan.entry && !plan.skinny ? (plan.k.stream_k ? IRIS_GEMM_SPLIT_STREAM_K : plan.k.split_k) : 1;
  return hipSuccess;
}

extern "C" int iris_gemm_kernel_info(const iris_gemm_args* args, int* n_regs, int* n_spills) {
  if (!args) return hipErrorInvalidValue;
  Plan plan;
  hipError_t err = make_plan(*args, &plan);
  if (err != hipSuccess) return err;
  if (n_regs) *n_regs = 0;
  if (n_spills) *n_spills = 0;
  if (!plan.entry && !plan.skinny) return hipSuccess;
  hipFuncAttributes attr;
  err = hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(plan.skinny ? plan.skinny : plan_fn(plan)));
  if (err != hipSuccess) return err;
  if (n_regs) *n_regs = attr.numRegs;
  if (n_spills) *n_spills = static_cast<int>(attr.localSizeBytes);
  return hipSuccess;
}

extern "C" int iris_gemm_variant_name(int ab_dtype, int out_is_f32, int atomic, int variant, char* buf, size_t len) {
  const int op = atomic ? (out_is_f32 ? OP_ATOMIC32 : OP_ATOMIC16) : (out_is_f32 ? OP_STORE32 : OP_STORE16);
  int count = 0;
  const GemmKernelEntry* list = entries_for(ab_dtype, op, &count);
  if (!list || variant < 1 || variant > count || !buf || len == 0) return hipErrorInvalidValue;
  std::snprintf(buf, len, "%s", list[variant - 1].name);
  return hipSuccess;
}

extern "C" int iris_gemm_plan_name(const iris_gemm_args* args, char* buf, size_t len) {
  if (!args || !buf || len == 0) return hipErrorInvalidValue;
  Plan plan;
  hipError_t err = make_plan(*args, &plan);
  if (err != hipSuccess) return err;
  const char* few = plan.skinny_cb == 2 ? (plan.skinny_rb == 2 ? "cells_32x32" : "cells_16x32") : plan.skinny_rb == 2 ? "few_rows_32xN" : "few_rows_16xN";
  std::snprintf(buf, len, "%s%s%s%s", plan.skinny ? few : plan.entry ? plan.entry->name : "", plan.loose ? "_gather_dma" : plan.b_rows ? "_rows" : "",
                plan.entry && plan.k.stream_k                   ? "+stream_k"
                : plan.entry && plan.in_program                 ? "+reduce"
                : plan.entry && plan.k.num_sms > args->num_sms ? "+two_per_cu"
                                                                : "",
                !plan.entry                            ? ""
                : plan.k.merge_m * plan.k.merge_n == 2 ? "+two_tiles_each"
                : plan.k.merge_m * plan.k.merge_n == 4 ? "+four_tiles_each"
                : plan.k.merge_m * plan.k.merge_n == 8 ? "+eight_tiles_each"
                                                       : "");
  if (plan_touches(plan)) {
    const size_t n = std::strlen(buf);
    std::snprintf(buf + n, len > n ? len - n : 0, "+touch_ahead");
  }
  if (plan.last_round) {
    const size_t n = std::strlen(buf);
    std::snprintf(buf + n, len > n ? len - n : 0, "+last_round_in_%d_parts", plan.k_last.split_k);
  }
  if (plan.rest) {
    const size_t n = std::strlen(buf);
    std::snprintf(buf + n, len > n ? len - n : 0, "+last_%d_columns_apart", plan.rest->k.N);
  }
  if (plan.parts) {
    const size_t n = std::strlen(buf);
    std::snprintf(buf + n, len > n ? len - n : 0, plan.parts == 2 ? "+across_the_tiles" : "+parts_of_tiles");
  }
  if (plan.two_kernels || (plan.reduces && args->phase == IRIS_PHASE_FUSED)) {
    const size_t n = std::strlen(buf);
    std::snprintf(buf + n, len > n ? len - n : 0, plan.two_kernels ? "+kernel+reduce" : "+reduce");
  }
  return hipSuccess;
}

extern "C" int iris_gemm_launch_kernels(const iris_gemm_args* args, int* kernels, int* waiting) {
  if (!args) return hipErrorInvalidValue;
  Plan plan;
  const hipError_t err = make_plan(*args, &plan);
  if (err != hipSuccess) return err;
  auto count = [](const Plan& q) { return q.skinny ? 1 : q.entry ? (q.last_round ? 2 : 1) : 0; };
  // (a reduce of nothing is no kernel)
  const bool behind = plan.fused_reduce && args->M > 0 && args->N > 0;
  if (kernels) *kernels = count(plan) + (plan.rest ? count(*plan.rest) : 0) + (behind ? 1 : 0);
  if (waiting) {
    const int on_all_engines = LATE_ENGINES * late_most(args->world_size);
    const int most = plan.reduces ? on_all_engines : plan.in_program && plan.entry && args->world_size > 1 ? plan.k.num_sms : 0;
    *waiting = most < plan.k.total_tiles ? most : plan.k.total_tiles;
  }
  return hipSuccess;
}

extern "C" int iris_stream_k_schedule_host(int32_t total_tiles, int32_t k_steps, int32_t num_programs, int32_t pid,
                                           int32_t* items, int32_t cap, int32_t* n_items) {
  if (total_tiles <= 0 || k_steps <= 0 || num_programs <= 0 || pid < 0 || pid >= num_programs || !n_items ||
      (int64_t)total_tiles * k_steps >= ((int64_t)1 << 30))
    return hipErrorInvalidValue;
  GemmKArgs k{};
  const int64_t steps = (int64_t)total_tiles * k_steps;
  k.split_q = (int)(steps / num_programs);
  k.split_r = (int)(steps % num_programs);
  if (k.split_q < 1) return hipErrorInvalidValue;  // the kernel is never launched with empty runs
  k.div_nk = make_fast_div((uint32_t)k_steps, (uint64_t)steps + 1);
  const StreamRun sr = stream_run(k, pid, k_steps);
  const int n = stream_items(sr, k_steps);
  *n_items = n;
  for (int i = 0; i < n && i < cap && items; ++i) {
    // the kernel's k_range for a split build, and the owner's count of parts
    const int k_begin = i == 0 ? sr.k0 : 0;
    const int k_end = sr.g1 - (sr.tile0 + i) * k_steps < k_steps ? sr.g1 - (sr.tile0 + i) * k_steps : k_steps;
    items[4 * i + 0] = sr.tile0 + i;
    items[4 * i + 1] = k_begin;
    items[4 * i + 2] = k_end;
    items[4 * i + 3] = k_begin == 0 ? stream_parts(k, pid, k_end, k_steps) : 0;
  }
  return hipSuccess;
}
