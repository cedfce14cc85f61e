// Shard-GEMM kernel instantiations: bf16 operands, the tiles for a row-major B, store epilogues.
#include "gemm_registry.hpp"

namespace iris_amd {

IRIS_GEMM_ROWS_STORE_VARIANTS(IRIS_GEMM_INSTANTIATE, IRIS_DTYPE_BF16, OP_STORE16)
IRIS_GEMM_INSTANTIATE_MERGED_DMA(IRIS_DTYPE_BF16, OP_STORE16, LOAD_DMA_ROWS)
static const GemmKernelEntry k_store16[] = {IRIS_GEMM_ROWS_STORE_VARIANTS(IRIS_GEMM_ENTRY, IRIS_DTYPE_BF16, OP_STORE16)};
const GemmKernelEntry* gemm_entries_bf16_store16_rows(int* count) {
  *count = (int)(sizeof(k_store16) / sizeof(k_store16[0]));
  return k_store16;
}

IRIS_GEMM_ROWS_STORE_VARIANTS(IRIS_GEMM_INSTANTIATE, IRIS_DTYPE_BF16, OP_STORE32)
IRIS_GEMM_INSTANTIATE_MERGED_DMA(IRIS_DTYPE_BF16, OP_STORE32, LOAD_DMA_ROWS)
static const GemmKernelEntry k_store32[] = {IRIS_GEMM_ROWS_STORE_VARIANTS(IRIS_GEMM_ENTRY, IRIS_DTYPE_BF16, OP_STORE32)};
const GemmKernelEntry* gemm_entries_bf16_store32_rows(int* count) {
  *count = (int)(sizeof(k_store32) / sizeof(k_store32[0]));
  return k_store32;
}

}  // namespace iris_amd
