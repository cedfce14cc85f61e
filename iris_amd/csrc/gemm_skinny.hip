// Instantiations of the few-rows shard GEMM.
#include "gemm_skinny.hpp"

namespace iris_amd {

namespace {

template <int DT, int OP, bool LOOSE, bool REDUCE>
GemmKernelFn pick(int arows, int rb, int cb) {
  constexpr int ODT = (OP == OP_STORE32 || OP == OP_ATOMIC32) ? IRIS_DTYPE_F32 : DT;
  if (cb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2, 2, LOOSE, false, REDUCE>;
  if (rb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2, 1, LOOSE, false, REDUCE>;
  return arows == 8 ? &gemm_skinny_kernel<DT, OP, ODT, 8, 1, 1, LOOSE, false, REDUCE>
                    : &gemm_skinny_kernel<DT, OP, ODT, 16, 1, 1, LOOSE, false, REDUCE>;
}

template <int DT, int OP, bool REDUCE>
GemmKernelFn pick_b_rows(int arows, int rb, int cb) {
  constexpr int ODT = (OP == OP_STORE32 || OP == OP_ATOMIC32) ? IRIS_DTYPE_F32 : DT;
  if (cb != 2) return nullptr;
  if (rb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2, 2, false, true, REDUCE>;
  return arows == 8 ? &gemm_skinny_kernel<DT, OP, ODT, 8, 1, 2, false, true, REDUCE>
                    : &gemm_skinny_kernel<DT, OP, ODT, 16, 1, 2, false, true, REDUCE>;
}

template <int DT, int OP>
GemmKernelFn pick(int arows, int rb, int cb, bool loose, bool b_rows, bool reduce) {
  if constexpr (OP == OP_STORE16 || OP == OP_STORE32) {
    if (reduce) {
      if constexpr (DT != IRIS_DTYPE_F32)
        if (b_rows) return pick_b_rows<DT, OP, true>(arows, rb, cb);
      if (b_rows) return nullptr;
      return loose ? pick<DT, OP, true, true>(arows, rb, cb) : pick<DT, OP, false, true>(arows, rb, cb);
    }
  }
  if (reduce) return nullptr;
  if constexpr (DT != IRIS_DTYPE_F32)
    if (b_rows) return pick_b_rows<DT, OP, false>(arows, rb, cb);
  if (b_rows) return nullptr;
  return loose ? pick<DT, OP, true, false>(arows, rb, cb) : pick<DT, OP, false, false>(arows, rb, cb);
}

}  // namespace

GemmKernelFn gemm_skinny_kernel_for(int dt, int op, int arows, int rb, int cb, bool loose, bool b_rows, bool reduce) {
  if (dt == IRIS_DTYPE_BF16) {
    if (op == OP_STORE16) return pick<IRIS_DTYPE_BF16, OP_STORE16>(arows, rb, cb, loose, b_rows, reduce);
    if (op == OP_STORE32) return pick<IRIS_DTYPE_BF16, OP_STORE32>(arows, rb, cb, loose, b_rows, reduce);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_BF16, OP_ATOMIC32>(arows, rb, cb, loose, b_rows, reduce);
    if (op == OP_ATOMIC16) return pick<IRIS_DTYPE_BF16, OP_ATOMIC16>(arows, rb, cb, loose, b_rows, reduce);
  } else if (dt == IRIS_DTYPE_F16) {
    if (op == OP_STORE16) return pick<IRIS_DTYPE_F16, OP_STORE16>(arows, rb, cb, loose, b_rows, reduce);
    if (op == OP_STORE32) return pick<IRIS_DTYPE_F16, OP_STORE32>(arows, rb, cb, loose, b_rows, reduce);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_F16, OP_ATOMIC32>(arows, rb, cb, loose, b_rows, reduce);
    if (op == OP_ATOMIC16) return pick<IRIS_DTYPE_F16, OP_ATOMIC16>(arows, rb, cb, loose, b_rows, reduce);
  } else if (dt == IRIS_DTYPE_F32) {
    if (op == OP_STORE32) return pick<IRIS_DTYPE_F32, OP_STORE32>(arows, rb, cb, loose, b_rows, reduce);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_F32, OP_ATOMIC32>(arows, rb, cb, loose, b_rows, reduce);
  }
  return nullptr;
}

}  // namespace iris_amd
