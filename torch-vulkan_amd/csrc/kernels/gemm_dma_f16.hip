// The direct-to-LDS matrix-core GEMM for f16 operands (one file per type, so that they compile in parallel).
#include "gemm_dma_kernel.h"

namespace hk {
template bool dma_queue<F16>(const hrt_mm_args&, GemmTile, int64_t, hipStream_t);
template bool dma_queue_dq8<F16>(const hrt_mm_dq8_args&, GemmTile, uint64_t, int64_t, int64_t, hipStream_t);
}  // namespace hk
