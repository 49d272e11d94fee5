// The direct-to-LDS matrix-core GEMM (gemm_dma_kernel.h): which operands it takes, its tile shapes, and the
// launch functions, instantiated per element type in gemm_dma_bf16.hip and gemm_dma_f16.hip.
#pragma once

#include "../hrt/registry.h"
#include "device_common.h"

namespace hk {

constexpr int GBK = 64;  // K elements per step

enum GemmTile { T256x256, T128x256, T256x128, T128x192, T128x128, T64x128, T64x64, kGemmTiles };
struct TileShape {
  int bm, bn;
};
constexpr TileShape kTileShape[kGemmTiles] = {{256, 256}, {128, 256}, {256, 128}, {128, 192}, {128, 128}, {64, 128}, {64, 64}};

// How the kernel can take a product with a bm x bn tile.  atr / btr: the operand is contiguous along M (N)
// instead of K.  exact: whole tiles and K steps and a C of 16-byte aligned rows; otherwise the EDGE form, which
// masks.  Both need 16-byte aligned operand rows; the EDGE form also whole 16-byte chunks along the contiguous
// axis (K % 8 == 0 for an operand contiguous along K, its M or N % 8 == 0 otherwise).
struct DmaForm {
  bool ok, exact, atr, btr;
};
DmaForm dma_form(const hrt_mm_args& a, int bm, int bn);

// Queues c = alpha a b + beta bias on `tile`; the caller has checked dma_form(...).ok.  HRT_MM_F32_OUT writes
// fp32 products; kslice > 0 (a multiple of 64, HRT_MM_F32_OUT only): the batch index is a slice of K, slice z
// covers [z kslice, min(K, (z + 1) kslice)).  False: no kernel for this combination (nothing queued).
template <typename T>
bool dma_queue(const hrt_mm_args& a, GemmTile tile, int64_t kslice, hipStream_t s);

// The fused int8 linear: y = alpha x deq(q)^T + beta bias as A = x, B = q read as [N][K] int8 rows with one scale
// per 64 columns (K % 64 == 0, 16-byte aligned q).  ws != 0: fp32 partial products over `splits` slices of kslice.
template <typename T>
bool dma_queue_dq8(const hrt_mm_dq8_args& d, GemmTile tile, uint64_t ws, int64_t splits, int64_t kslice, hipStream_t s);
// The GEMM whose operands those are (b: int8, strides in bytes).
hrt_mm_args dq8_as_mm(const hrt_mm_dq8_args& d);

}  // namespace hk
