// Table of compiled shard-GEMM kernels.  Each instantiation file defines the
// entries of one (operand type, epilogue op) pair; the launcher picks one
// entry per call.
#pragma once

#include "gemm_kernel.hpp"

namespace iris_amd {

using GemmKernelFn = void (*)(const GemmKArgs);

struct GemmKernelEntry {
  int dt;      // operand type: IRIS_DTYPE_F16 | IRIS_DTYPE_BF16 | IRIS_DTYPE_F32
  int op;      // StoreOp
  int cm, cn;  // compute tile
  int bk, wm, wn, stages;  // (bk in 16-bit units: half as many elements of fp32 operands)
  bool dma;    // LDS-DMA loader (needs K-contiguous, 16-byte aligned operands)
  bool b_rows;  // ... of a B whose rows are its k (row-major [K, N], 16-byte aligned rows)
  bool loose;   // ... of operands along K at any alignment and of any K from eight on
  bool gather;  // gathering loader (operands contiguous along K or across it, at any alignment); neither: generic
  bool splitk;  // the kernel can share a tile's K range with other programs
  bool split_owner;  // ... and its first part can add the others' partials itself (needed for stream-K runs)
  int threads;        // launch size: the multiplying waves and the fetching waves (if any)
  int fetch_waves;    // waves that only issue the stage loads (0: every wave fetches its share)
  int lds_bytes;
  GemmKernelFn fn;
  GemmKernelFn fn_split;  // split-K build, or null
  GemmKernelFn fn_fused;  // build with the one-shot reduce inside the program (store epilogues), or null
  GemmKernelFn fn_merged;  // build whose tiles are blocks of the caller's (store epilogues, 256 x 128 and 256 x 256), or null
  GemmKernelFn fn_split_merged;  // ... and its split-K build, or null
  GemmKernelFn fn_touch;         // unsplit build that touches lines of K-steps to come (the eight-wave 256 x 256 tile), or null
  GemmKernelFn fn_touch_merged;  // ... whose tiles are blocks of the caller's
  const char* name;
};

template <class Cfg, int OP, int ODT>
constexpr GemmKernelFn split_fn() {
  if constexpr (Cfg::SPLITK)
    return &gemm_persistent_kernel<Cfg, OP, ODT, true>;
  else
    return nullptr;
}

template <class Cfg, int OP, int ODT>
constexpr GemmKernelFn fused_fn() {
  // (the DMA tiles with fetching waves have no such build: the reduce wants the registers their
  // fetch state takes, and the launcher takes the plain tile of the same shape instead; the gathering tiles, which
  // have no plain twin, have one where the accumulators leave room)
  if constexpr ((OP == OP_STORE16 || OP == OP_STORE32) && !Cfg::B_ROWS && !Cfg::LOOSE && (Cfg::LW == 0 || (Cfg::GATHER && Cfg::IM * Cfg::IN * 4 <= 64)))
    return &gemm_persistent_kernel<Cfg, OP, ODT, false, true>;
  else
    return nullptr;
}

// The launcher only merges the caller's tiles into 256 x 128 and 256 x 256 ones, for the store epilogues, and
// runs them with the table's first tile of either shape.
// (... and, for a range of the caller's columns launched on its own, with the 256 x 64 one as it is)
template <class Cfg>
constexpr bool merged_build = Cfg::CM == 256 && Cfg::DMA && Cfg::BK == 64 &&
                              ((Cfg::CN == 256 && Cfg::LW == 0 && Cfg::NW == 8) || (Cfg::CN == 128 && Cfg::LW == 4) ||
                               (Cfg::CN == 64 && Cfg::LW == 4 && Cfg::S == 3));
template <class Cfg, int OP, int ODT>
constexpr GemmKernelFn merged_fn() {
  if constexpr ((OP == OP_STORE16 || OP == OP_STORE32) && merged_build<Cfg>)
    return &gemm_persistent_kernel<Cfg, OP, ODT, false, false, true>;
  else
    return nullptr;
}

template <class Cfg, int OP, int ODT>
constexpr GemmKernelFn split_merged_fn() {
  if constexpr ((OP == OP_STORE16 || OP == OP_STORE32) && merged_build<Cfg> && Cfg::SPLITK)
    return &gemm_persistent_kernel<Cfg, OP, ODT, true, false, true>;
  else
    return nullptr;
}

// The eight-wave 256 x 256 tile's builds with the touches of Loader::touch (store epilogues).
template <class Cfg>
constexpr bool touch_build = Cfg::CM == 256 && Cfg::CN == 256 && Cfg::DMA && !Cfg::B_ROWS && !Cfg::LOOSE && Cfg::BK == 64 && Cfg::LW == 0 && Cfg::NW == 8 &&
                             Cfg::S == 2 && Cfg::WM == 2;
template <int DT>
using TouchCfg = GemmCfg<DT, 256, 256, 64, 2, 4, 2, true, 0, true>;
template <class Cfg, int OP, int ODT, bool MERGED>
constexpr GemmKernelFn touch_fn() {
  if constexpr ((OP == OP_STORE16 || OP == OP_STORE32) && touch_build<Cfg>)
    return &gemm_persistent_kernel<TouchCfg<Cfg::DT>, OP, ODT, false, false, MERGED>;
  else
    return nullptr;
}

template <class Cfg, int OP>
constexpr GemmKernelEntry make_entry(const char* name) {
  constexpr int ODT = (OP == OP_STORE32 || OP == OP_ATOMIC32) ? IRIS_DTYPE_F32 : Cfg::DT;
  return GemmKernelEntry{Cfg::DT, OP,      Cfg::CM, Cfg::CN, Cfg::BK,        Cfg::WM,
                         Cfg::WN, Cfg::S,  Cfg::DMA, Cfg::B_ROWS, Cfg::LOOSE, Cfg::GATHER, Cfg::SPLITK, Cfg::SPLIT_OWNER, Cfg::THREADS, Cfg::LW, Cfg::LDS_BYTES,
                         &gemm_persistent_kernel<Cfg, OP, ODT, false>, split_fn<Cfg, OP, ODT>(), fused_fn<Cfg, OP, ODT>(),
                         merged_fn<Cfg, OP, ODT>(), split_merged_fn<Cfg, OP, ODT>(), touch_fn<Cfg, OP, ODT, false>(),
                         touch_fn<Cfg, OP, ODT, true>(), name};
}

// The variants, in the launcher's order of preference: the first entry whose
// compute tile divides the logical tile (and whose loader fits the operands)
// wins.  `variant` k > 0 in iris_gemm_args forces entry k-1 (tuning runs).
// Columns: compute tile CM, CN, BK; waves WM x WN; stages; loader (SlabLoad);
// fetching waves; whether the tile also has a split-K build (must equal
// GemmCfg::SPLITK); name.
//
// The four-wave tiles come twice: with one fetching wave per SIMD beside the
// multiplying one (`_f4`: a K-step then costs the longer of fetch and multiply
// instead of their sum; [2048,4096] x [4096,1376] in 128 x 128 tiles 48 -> 40 us)
// and as deep a ring as LDS holds, since a fetching wave cannot refill the
// stage that is being multiplied (256 x 64 tiles in three stages instead of
// two: 57 -> 42 us on the same shape); and plain, which the launcher takes
// where the first loses: with the reduce inside the program (no such build)
// and for two programs per CU.
//
// The generic tile is left for operands that are contiguous neither along K nor across it.
#define IRIS_GEMM_VARIANTS(X, DT, OP)                                     \
  X(DT, OP, 256, 256, 64, 2, 4, 2, LOAD_DMA, 0, 1, "256x256x64_w2x4_s2")         \
  X(DT, OP, 256, 128, 64, 2, 2, 3, LOAD_DMA, 4, 1, "256x128x64_w2x2_s3_f4")      \
  X(DT, OP, 128, 256, 64, 1, 4, 3, LOAD_DMA, 4, 1, "128x256x64_w1x4_s3_f4")      \
  X(DT, OP, 128, 128, 64, 2, 2, 4, LOAD_DMA, 4, 1, "128x128x64_w2x2_s4_f4")      \
  X(DT, OP, 256, 64, 64, 4, 1, 3, LOAD_DMA, 4, 1, "256x64x64_w4x1_s3_f4")        \
  X(DT, OP, 128, 64, 64, 2, 2, 4, LOAD_DMA, 4, 1, "128x64x64_w2x2_s4_f4")        \
  X(DT, OP, 64, 128, 64, 2, 2, 4, LOAD_DMA, 4, 1, "64x128x64_w2x2_s4_f4")        \
  X(DT, OP, 64, 64, 128, 2, 2, 4, LOAD_DMA, 4, 1, "64x64x128_w2x2_s4_f4")        \
  X(DT, OP, 256, 128, 64, 2, 2, 2, LOAD_DMA, 0, 1, "256x128x64_w2x2_s2")         \
  X(DT, OP, 128, 256, 64, 1, 4, 2, LOAD_DMA, 0, 1, "128x256x64_w1x4_s2")         \
  X(DT, OP, 128, 128, 64, 2, 2, 4, LOAD_DMA, 0, 1, "128x128x64_w2x2_s4")         \
  X(DT, OP, 256, 64, 64, 4, 1, 2, LOAD_DMA, 0, 1, "256x64x64_w4x1_s2")           \
  X(DT, OP, 64, 64, 64, 2, 2, 4, LOAD_DMA, 0, 1, "64x64x64_w2x2_s4")             \
  X(DT, OP, 64, 64, 32, 2, 2, 1, LOAD_GENERIC, 0, 0, "64x64x32_w2x2_generic")

// Tiles behind the table, which `variant` does not number.  The `_gather` tiles take what the DMA cannot: operands that
// lie along K at any alignment, or across it (a row-major B, a column-major A).
#define IRIS_GEMM_GATHER_VARIANTS(X, DT, OP)                                \
  X(DT, OP, 256, 128, 64, 2, 2, 2, LOAD_GATHER, 4, 1, "256x128x64_w2x2_gather") \
  X(DT, OP, 128, 128, 64, 2, 2, 2, LOAD_GATHER, 4, 1, "128x128x64_w2x2_gather") \
  X(DT, OP, 256, 64, 64, 4, 1, 2, LOAD_GATHER, 4, 1, "256x64x64_w4x1_gather")   \
  X(DT, OP, 64, 128, 64, 2, 2, 2, LOAD_GATHER, 4, 1, "64x128x64_w2x2_gather")   \
  X(DT, OP, 64, 64, 128, 2, 2, 2, LOAD_GATHER, 4, 1, "64x64x128_w2x2_gather")

// ... and, in a list of their own in front of those, the LDS-DMA tiles for a row-major B (LOAD_DMA_ROWS), the first for the store epilogues only (atomics take half
// tiles).  The gathering tiles transpose such a B in the fetching waves' registers, and a K-step waits for them: a step of
// 128 x 128 x 64 in 1.2 us.  Here the DMA brings the rows as they lie and the transposing LDS read costs what a plain one
// does: 0.45 us, as for a B along K ([2697,1936] x [1936,1600], 275 tiles in two rounds, 66.8 -> 40.1 us a pass).
// The same tiles (LOOSE) for operands along K that the plain ones do not take: rows at any alignment, a K that is no multiple
// of eight.  The DMA brings 16 bytes from any address at little more than the aligned ones' cost; the gathering tiles, which
// shift such rows in registers, are left for what lies across K ([4096,4096] x [4096,4096] on rows 8 bytes off, 256 x 256 tiles:
// 144 us gathered, 116 so, 100 aligned).
#define IRIS_GEMM_DMA_VARIANTS(X, DT, OP, LOAD, SUFFIX)                           \
  X(DT, OP, 256, 128, 64, 2, 2, 3, LOAD, 4, 1, "256x128x64_w2x2_s3_f4" SUFFIX)    \
  X(DT, OP, 128, 128, 64, 2, 2, 4, LOAD, 4, 1, "128x128x64_w2x2_s4_f4" SUFFIX)    \
  X(DT, OP, 256, 64, 64, 4, 1, 3, LOAD, 4, 1, "256x64x64_w4x1_s3_f4" SUFFIX)      \
  X(DT, OP, 128, 64, 64, 2, 2, 4, LOAD, 4, 1, "128x64x64_w2x2_s4_f4" SUFFIX)      \
  X(DT, OP, 64, 128, 64, 2, 2, 4, LOAD, 4, 1, "64x128x64_w2x2_s4_f4" SUFFIX)      \
  X(DT, OP, 64, 64, 128, 2, 2, 4, LOAD, 4, 1, "64x64x128_w2x2_s4_f4" SUFFIX)
#define IRIS_GEMM_DMA_STORE_VARIANTS(X, DT, OP, LOAD, SUFFIX)                     \
  X(DT, OP, 256, 256, 64, 2, 4, 2, LOAD, 0, 1, "256x256x64_w2x4_s2" SUFFIX)       \
  IRIS_GEMM_DMA_VARIANTS(X, DT, OP, LOAD, SUFFIX)
#define IRIS_GEMM_ROWS_VARIANTS(X, DT, OP) IRIS_GEMM_DMA_VARIANTS(X, DT, OP, LOAD_DMA_ROWS, "_rows")
#define IRIS_GEMM_ROWS_STORE_VARIANTS(X, DT, OP) IRIS_GEMM_DMA_STORE_VARIANTS(X, DT, OP, LOAD_DMA_ROWS, "_rows")
#define IRIS_GEMM_LOOSE_VARIANTS(X, DT, OP) IRIS_GEMM_DMA_VARIANTS(X, DT, OP, LOAD_DMA_LOOSE, "_gather_dma")
#define IRIS_GEMM_LOOSE_STORE_VARIANTS(X, DT, OP) IRIS_GEMM_DMA_STORE_VARIANTS(X, DT, OP, LOAD_DMA_LOOSE, "_gather_dma")

// extra variants, compiled for the bf16 store op only (tuning runs, and the
// one-substep stage whose fragment buffers alternate from step to step)
#define IRIS_GEMM_TUNING_VARIANTS(X, DT, OP)                              \
  X(DT, OP, 256, 128, 32, 2, 4, 4, LOAD_DMA, 0, 0, "256x128x32_w2x4_s4")         \
  X(DT, OP, 256, 128, 64, 2, 4, 2, LOAD_DMA, 0, 1, "256x128x64_w2x4_s2")         \
  X(DT, OP, 128, 256, 64, 2, 4, 2, LOAD_DMA, 0, 1, "128x256x64_w2x4_s2")         \
  X(DT, OP, 128, 128, 32, 2, 2, 4, LOAD_DMA, 0, 0, "128x128x32_w2x2_s4")         \
  X(DT, OP, 64, 64, 64, 2, 2, 4, LOAD_DMA, 4, 1, "64x64x64_w2x2_s4_f4")          \
  X(DT, OP, 256, 64, 64, 4, 1, 2, LOAD_DMA, 4, 1, "256x64x64_w4x1_s2_f4")

#define IRIS_GEMM_ENTRY(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW, SPLIT, NAME) \
  make_entry<GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>, OP>(NAME),

// Explicit instantiation of an entry's kernels.  Taking their addresses in
// make_entry should be enough, but with the plain and the split-K build of a
// tile in one translation unit the compiler's host pass has been seen to
// reference one of the two without emitting it.
#define IRIS_GEMM_ODT(DT, OP) (((OP) == OP_STORE32 || (OP) == OP_ATOMIC32) ? IRIS_DTYPE_F32 : (DT))
#define IRIS_GEMM_INSTANTIATE_SPLIT_0(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW) \
  static_assert(!GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>::SPLITK, "split-K column of the variant table");
#define IRIS_GEMM_INSTANTIATE_SPLIT_1(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW)                                  \
  static_assert(GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>::SPLITK, "split-K column of the variant table"); \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>, OP,           \
                                                  IRIS_GEMM_ODT(DT, OP), true>(const GemmKArgs);
#define IRIS_GEMM_INSTANTIATE(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW, SPLIT, NAME)                    \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>, OP,    \
                                                  IRIS_GEMM_ODT(DT, OP), false>(const GemmKArgs); \
  IRIS_GEMM_INSTANTIATE_SPLIT_##SPLIT(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW)
// the store epilogues' build with the one-shot reduce inside the program
#define IRIS_GEMM_INSTANTIATE_FUSED(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW, SPLIT, NAME) \
  IRIS_GEMM_INSTANTIATE_FUSED_##LW(DT, OP, CM, CN, BK, WM, WN, S, DMA)
#define IRIS_GEMM_INSTANTIATE_FUSED_0(DT, OP, CM, CN, BK, WM, WN, S, DMA)                     \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA>, OP, \
                                                  IRIS_GEMM_ODT(DT, OP), false, true>(const GemmKArgs);
#define IRIS_GEMM_INSTANTIATE_FUSED_4(DT, OP, CM, CN, BK, WM, WN, S, DMA)

// the store epilogues' builds whose tiles are blocks of the caller's
#define IRIS_GEMM_INSTANTIATE_MERGED(DT, OP)                                                                        \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, 256, 256, 64, 2, 4, 2, true, 0>, OP,                \
                                                  IRIS_GEMM_ODT(DT, OP), false, false, true>(const GemmKArgs); \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, 256, 128, 64, 2, 2, 3, true, 4>, OP,                \
                                                  IRIS_GEMM_ODT(DT, OP), false, false, true>(const GemmKArgs); \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, 256, 256, 64, 2, 4, 2, true, 0>, OP,                \
                                                  IRIS_GEMM_ODT(DT, OP), true, false, true>(const GemmKArgs);  \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, 256, 128, 64, 2, 2, 3, true, 4>, OP,                \
                                                  IRIS_GEMM_ODT(DT, OP), true, false, true>(const GemmKArgs);  \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, 256, 64, 64, 4, 1, 3, true, 4>, OP,                 \
                                                  IRIS_GEMM_ODT(DT, OP), false, false, true>(const GemmKArgs); \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, 256, 64, 64, 4, 1, 3, true, 4>, OP,                 \
                                                  IRIS_GEMM_ODT(DT, OP), true, false, true>(const GemmKArgs);  \
  template __global__ void gemm_persistent_kernel<TouchCfg<DT>, OP, IRIS_GEMM_ODT(DT, OP), false, false, false>(  \
      const GemmKArgs);                                                                                           \
  template __global__ void gemm_persistent_kernel<TouchCfg<DT>, OP, IRIS_GEMM_ODT(DT, OP), false, false, true>(   \
      const GemmKArgs);

#define IRIS_GEMM_MERGED_KERNEL(DT, OP, CN, WM, WN, S, LOAD, LW, SPLIT)                                      \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, 256, CN, 64, WM, WN, S, LOAD, LW>, OP,         \
                                                  IRIS_GEMM_ODT(DT, OP), SPLIT, false, true>(const GemmKArgs);
#define IRIS_GEMM_INSTANTIATE_MERGED_DMA(DT, OP, LOAD)           \
  IRIS_GEMM_MERGED_KERNEL(DT, OP, 256, 2, 4, 2, LOAD, 0, false)  \
  IRIS_GEMM_MERGED_KERNEL(DT, OP, 256, 2, 4, 2, LOAD, 0, true)   \
  IRIS_GEMM_MERGED_KERNEL(DT, OP, 128, 2, 2, 3, LOAD, 4, false)  \
  IRIS_GEMM_MERGED_KERNEL(DT, OP, 128, 2, 2, 3, LOAD, 4, true)   \
  IRIS_GEMM_MERGED_KERNEL(DT, OP, 64, 4, 1, 3, LOAD, 4, false)   \
  IRIS_GEMM_MERGED_KERNEL(DT, OP, 64, 4, 1, 3, LOAD, 4, true)

// fp32 operands (fp32 output only): a short table.  The tiles are the 16-bit ones' (a stage of BK 16-bit units holds
// BK / 2 elements of K; the names count elements); the matrix cores run fp32 at a sixteenth of the 16-bit rate, so any
// tile that keeps them fed will do, and none is split along K or merged.
// (SPLIT: with a split-K build, which only the tiles behind the table have)
template <class Cfg, int OP, bool SPLIT = false>
constexpr GemmKernelEntry make_entry_f32(const char* name) {
  static_assert(Cfg::DT == IRIS_DTYPE_F32 && (OP == OP_STORE32 || OP == OP_ATOMIC32), "fp32 operands, fp32 output");
  GemmKernelFn split = nullptr;
  if constexpr (SPLIT) split = split_fn<Cfg, OP, IRIS_DTYPE_F32>();
  return GemmKernelEntry{Cfg::DT, OP, Cfg::CM, Cfg::CN, Cfg::BK, Cfg::WM, Cfg::WN, Cfg::S, Cfg::DMA, Cfg::B_ROWS, Cfg::LOOSE, Cfg::GATHER, SPLIT, SPLIT && Cfg::SPLIT_OWNER,
                         Cfg::THREADS, Cfg::LW, Cfg::LDS_BYTES, &gemm_persistent_kernel<Cfg, OP, IRIS_DTYPE_F32, false>,
                         split, fused_fn<Cfg, OP, IRIS_DTYPE_F32>(), nullptr, nullptr, nullptr, nullptr, name};
}
#define IRIS_GEMM_F32_VARIANTS(X, OP)                                                   \
  X(IRIS_DTYPE_F32, OP, 128, 128, 64, 2, 2, 4, LOAD_DMA, 4, "128x128x32_w2x2_s4_f4_fp32")  \
  X(IRIS_DTYPE_F32, OP, 128, 128, 64, 2, 2, 4, LOAD_DMA, 0, "128x128x32_w2x2_s4_fp32")     \
  X(IRIS_DTYPE_F32, OP, 64, 64, 64, 2, 2, 4, LOAD_DMA, 0, "64x64x32_w2x2_s4_fp32")         \
  X(IRIS_DTYPE_F32, OP, 64, 64, 32, 2, 2, 1, LOAD_GENERIC, 0, "64x64x16_w2x2_generic_fp32")
// Tiles behind the fp32 table: the launcher takes them for a K of eight K-steps or more.
// The scripts' 256 x 64 tile as one compute tile ([2048,1024] x [1024,2048]: as four of 64 x 64, fetch-bound, 131 us;
// 70 so), split-K builds, and the gathering loader.
#define IRIS_GEMM_F32_LONG_VARIANTS(X, OP)                                                        \
  X(IRIS_DTYPE_F32, OP, 128, 128, 64, 2, 2, 4, LOAD_DMA, 4, "128x128x32_w2x2_s4_f4_fp32")        \
  X(IRIS_DTYPE_F32, OP, 256, 64, 64, 4, 1, 3, LOAD_DMA, 4, "256x64x32_w4x1_s3_f4_fp32")          \
  X(IRIS_DTYPE_F32, OP, 64, 128, 64, 2, 2, 4, LOAD_DMA, 4, "64x128x32_w2x2_s4_f4_fp32")          \
  X(IRIS_DTYPE_F32, OP, 64, 64, 128, 2, 2, 4, LOAD_DMA, 4, "64x64x64_w2x2_s4_f4_fp32")           \
  X(IRIS_DTYPE_F32, OP, 128, 128, 64, 2, 2, 2, LOAD_GATHER, 4, "128x128x32_w2x2_gather_fp32")    \
  X(IRIS_DTYPE_F32, OP, 256, 64, 64, 4, 1, 2, LOAD_GATHER, 4, "256x64x32_w4x1_gather_fp32")      \
  X(IRIS_DTYPE_F32, OP, 64, 64, 128, 2, 2, 2, LOAD_GATHER, 4, "64x64x64_w2x2_gather_fp32")
#define IRIS_GEMM_F32_LONG_ENTRY(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW, NAME) \
  make_entry_f32<GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>, OP, true>(NAME),
#define IRIS_GEMM_F32_ENTRY(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW, NAME) \
  make_entry_f32<GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>, OP>(NAME),
#define IRIS_GEMM_F32_INSTANTIATE(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW, NAME)                    \
  template __global__ void gemm_persistent_kernel<GemmCfg<DT, CM, CN, BK, WM, WN, S, DMA, LW>, OP, \
                                                  IRIS_DTYPE_F32, false>(const GemmKArgs);
#define IRIS_GEMM_F32_INSTANTIATE_FUSED(DT, OP, CM, CN, BK, WM, WN, S, DMA, LW, NAME) \
  IRIS_GEMM_INSTANTIATE_FUSED_##LW(DT, OP, CM, CN, BK, WM, WN, S, DMA)

#define IRIS_GEMM_DECLARE(TAG) const GemmKernelEntry* gemm_entries_##TAG(int* count);
IRIS_GEMM_DECLARE(f32_store32)
IRIS_GEMM_DECLARE(f32_atomic32)
IRIS_GEMM_DECLARE(f32_store32_long)
IRIS_GEMM_DECLARE(f32_atomic32_long)
IRIS_GEMM_DECLARE(bf16_store16_rows)
IRIS_GEMM_DECLARE(bf16_store32_rows)
IRIS_GEMM_DECLARE(bf16_atomic32_rows)
IRIS_GEMM_DECLARE(bf16_atomic16_rows)
IRIS_GEMM_DECLARE(f16_store16_rows)
IRIS_GEMM_DECLARE(f16_store32_rows)
IRIS_GEMM_DECLARE(f16_atomic32_rows)
IRIS_GEMM_DECLARE(f16_atomic16_rows)
IRIS_GEMM_DECLARE(bf16_store16_loose)
IRIS_GEMM_DECLARE(bf16_store32_loose)
IRIS_GEMM_DECLARE(bf16_atomic32_loose)
IRIS_GEMM_DECLARE(bf16_atomic16_loose)
IRIS_GEMM_DECLARE(f16_store16_loose)
IRIS_GEMM_DECLARE(f16_store32_loose)
IRIS_GEMM_DECLARE(f16_atomic32_loose)
IRIS_GEMM_DECLARE(f16_atomic16_loose)
IRIS_GEMM_DECLARE(bf16_store16_gather)
IRIS_GEMM_DECLARE(bf16_store32_gather)
IRIS_GEMM_DECLARE(bf16_atomic32_gather)
IRIS_GEMM_DECLARE(bf16_atomic16_gather)
IRIS_GEMM_DECLARE(f16_store16_gather)
IRIS_GEMM_DECLARE(f16_store32_gather)
IRIS_GEMM_DECLARE(f16_atomic32_gather)
IRIS_GEMM_DECLARE(f16_atomic16_gather)
IRIS_GEMM_DECLARE(bf16_store16)
IRIS_GEMM_DECLARE(bf16_store32)
IRIS_GEMM_DECLARE(bf16_atomic32)
IRIS_GEMM_DECLARE(bf16_atomic16)
IRIS_GEMM_DECLARE(f16_store16)
IRIS_GEMM_DECLARE(f16_store32)
IRIS_GEMM_DECLARE(f16_atomic32)
IRIS_GEMM_DECLARE(f16_atomic16)

}  // namespace iris_amd
