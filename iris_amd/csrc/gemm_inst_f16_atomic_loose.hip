// Shard-GEMM kernel instantiations: fp16 operands, the tiles for operands along K at any alignment, atomic epilogues.
#include "gemm_registry.hpp"

namespace iris_amd {

IRIS_GEMM_LOOSE_VARIANTS(IRIS_GEMM_INSTANTIATE, IRIS_DTYPE_F16, OP_ATOMIC32)
static const GemmKernelEntry k_atomic32[] = {IRIS_GEMM_LOOSE_VARIANTS(IRIS_GEMM_ENTRY, IRIS_DTYPE_F16, OP_ATOMIC32)};
const GemmKernelEntry* gemm_entries_f16_atomic32_loose(int* count) {
  *count = (int)(sizeof(k_atomic32) / sizeof(k_atomic32[0]));
  return k_atomic32;
}

IRIS_GEMM_LOOSE_VARIANTS(IRIS_GEMM_INSTANTIATE, IRIS_DTYPE_F16, OP_ATOMIC16)
static const GemmKernelEntry k_atomic16[] = {IRIS_GEMM_LOOSE_VARIANTS(IRIS_GEMM_ENTRY, IRIS_DTYPE_F16, OP_ATOMIC16)};
const GemmKernelEntry* gemm_entries_f16_atomic16_loose(int* count) {
  *count = (int)(sizeof(k_atomic16) / sizeof(k_atomic16[0]));
  return k_atomic16;
}

}  // namespace iris_amd
