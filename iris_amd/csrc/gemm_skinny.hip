// Instantiations of the few-rows shard GEMM.
#include "gemm_skinny.hpp"

namespace iris_amd {

namespace {

template <int DT, int OP>
GemmKernelFn pick(int arows, int rb, int cb) {
  constexpr int ODT = (OP == OP_STORE32 || OP == OP_ATOMIC32) ? IRIS_DTYPE_F32 : DT;
  if (cb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2, 2>;
  if (rb == 2) return &gemm_skinny_kernel<DT, OP, ODT, 16, 2>;
  return arows == 8 ? &gemm_skinny_kernel<DT, OP, ODT, 8> : &gemm_skinny_kernel<DT, OP, ODT, 16>;
}

}  // namespace

GemmKernelFn gemm_skinny_kernel_for(int dt, int op, int arows, int rb, int cb) {
  if (dt == IRIS_DTYPE_BF16) {
    if (op == OP_STORE16) return pick<IRIS_DTYPE_BF16, OP_STORE16>(arows, rb, cb);
    if (op == OP_STORE32) return pick<IRIS_DTYPE_BF16, OP_STORE32>(arows, rb, cb);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_BF16, OP_ATOMIC32>(arows, rb, cb);
    if (op == OP_ATOMIC16) return pick<IRIS_DTYPE_BF16, OP_ATOMIC16>(arows, rb, cb);
  } else if (dt == IRIS_DTYPE_F16) {
    if (op == OP_STORE16) return pick<IRIS_DTYPE_F16, OP_STORE16>(arows, rb, cb);
    if (op == OP_STORE32) return pick<IRIS_DTYPE_F16, OP_STORE32>(arows, rb, cb);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_F16, OP_ATOMIC32>(arows, rb, cb);
    if (op == OP_ATOMIC16) return pick<IRIS_DTYPE_F16, OP_ATOMIC16>(arows, rb, cb);
  } else if (dt == IRIS_DTYPE_F32) {
    if (op == OP_STORE32) return pick<IRIS_DTYPE_F32, OP_STORE32>(arows, rb, cb);
    if (op == OP_ATOMIC32) return pick<IRIS_DTYPE_F32, OP_ATOMIC32>(arows, rb, cb);
  }
  return nullptr;
}

}  // namespace iris_amd
