// Instantiations of the few-rows shard GEMM.
#include "gemm_skinny.hpp"

namespace iris_amd {

namespace {

template <int DT, int OP, bool LOOSE>
GemmKernelFn pick(int arows, int rb, int cb) {
  constexpr int ODT = (OP == OP_STORE32 || OP == OP_ATOMIC32) ? IRIS_DTYPE_F32 : DT;
  if (cb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2, 2, LOOSE>;
  if (rb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2, 1, LOOSE>;
  return arows == 8 ? &gemm_skinny_kernel<DT, OP, ODT, 8, 1, 1, LOOSE> : &gemm_skinny_kernel<DT, OP, ODT, 16, 1, 1, LOOSE>;
}

template <int DT, int OP>
GemmKernelFn pick(int arows, int rb, int cb, bool loose, bool b_rows) {
  if (b_rows) {
    if constexpr (DT == IRIS_DTYPE_F32) {
      return nullptr;
    } else {
      constexpr int ODT = (OP == OP_STORE32 || OP == OP_ATOMIC32) ? IRIS_DTYPE_F32 : DT;
      if (cb != 2) return nullptr;
      if (rb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2, 2, false, true>;
      return arows == 8 ? &gemm_skinny_kernel<DT, OP, ODT, 8, 1, 2, false, true> : &gemm_skinny_kernel<DT, OP, ODT, 16, 1, 2, false, true>;
    }
  }
  return loose ? pick<DT, OP, true>(arows, rb, cb) : pick<DT, OP, false>(arows, rb, cb);
}

}  // namespace

GemmKernelFn gemm_skinny_kernel_for(int dt, int op, int arows, int rb, int cb, bool loose, bool b_rows) {
  if (dt == IRIS_DTYPE_BF16) {
    if (op == OP_STORE16) return pick<IRIS_DTYPE_BF16, OP_STORE16>(arows, rb, cb, loose, b_rows);
    if (op == OP_STORE32) return pick<IRIS_DTYPE_BF16, OP_STORE32>(arows, rb, cb, loose, b_rows);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_BF16, OP_ATOMIC32>(arows, rb, cb, loose, b_rows);
    if (op == OP_ATOMIC16) return pick<IRIS_DTYPE_BF16, OP_ATOMIC16>(arows, rb, cb, loose, b_rows);
  } else if (dt == IRIS_DTYPE_F16) {
    if (op == OP_STORE16) return pick<IRIS_DTYPE_F16, OP_STORE16>(arows, rb, cb, loose, b_rows);
    if (op == OP_STORE32) return pick<IRIS_DTYPE_F16, OP_STORE32>(arows, rb, cb, loose, b_rows);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_F16, OP_ATOMIC32>(arows, rb, cb, loose, b_rows);
    if (op == OP_ATOMIC16) return pick<IRIS_DTYPE_F16, OP_ATOMIC16>(arows, rb, cb, loose, b_rows);
  } else if (dt == IRIS_DTYPE_F32) {
    if (op == OP_STORE32) return pick<IRIS_DTYPE_F32, OP_STORE32>(arows, rb, cb, loose, b_rows);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_F32, OP_ATOMIC32>(arows, rb, cb, loose, b_rows);
  }
  return nullptr;
}

}  // namespace iris_amd
