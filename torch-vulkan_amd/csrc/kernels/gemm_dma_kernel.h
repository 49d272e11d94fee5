// Direct-to-LDS matrix-core GEMM of the bf16 / f16 products and of the fused int8 linear: operands copied
// global -> LDS directly, v_mfma_f32_32x32x16.  Included by gemm_dma_{bf16,f16}.hip, which instantiate it for one
// element type each.
//
// C tile BM x BN per workgroup of (BM / WM) x (BN / WN) wavefronts; each wavefront owns a WM x WN sub-tile as
// (WM / 32) x (WN / 32) v_mfma_f32_32x32x16 accumulators.  Eight wavefronts (two per SIMD) of 64 x 64, 32 x 96 or
// 32 x 64 sub-tiles on the 128-row and larger tiles, four on 64 x 128 and 64 x 64, which fit a CU two and three
// times; plan_gemm (gemm_mfma.hip) chooses the tile.  128 x 128 tiles run eight wavefronts of 32 x 64: four of
// 64 x 64 leave one per SIMD, whose LDS latency nothing covers (2048^3 NT 25.6 against 22.3 us; 64 x 128 tiles 24.2).
// K advances in steps of 64 through a ring of RING LDS buffers (three; two for 256 x 256 tiles) filled by
// global_load_lds_dwordx4 copies of the operands' raw rows: the copies of step kt + RING - 1 are spread over
// the MFMAs of step kt, so a copy has RING - 1 steps to land (one step of compute is shorter than the L2
// latency plus the transfer of a 48 KiB step), one barrier per step.  An operand whose K axis is contiguous (A [M][K],
// or B given as [N][K]) is staged as [row][k] and read with 128-bit row reads; an operand contiguous along
// M or N (A given as [K][M], B as [K][N]) is staged as [k][row] and read with ds_read_b64_tr_b16 column
// reads, so all four layouts need no register transposes.  Epilogue: alpha * acc + beta * bias in fp32,
// one rounding, transposed through LDS so that C is written as 16-byte row pieces.
//
// EDGE: sizes that are no multiple of the tile or of a K step.  The copies go through a buffer resource whose range
// check returns zeros for the lanes past an edge (edge_lane_offsets), the partial K step comes first, so that the
// loop itself masks nothing, and the epilogue stores what exists.  The products of M = 4020 tokens (2048 x 2048
// weights, cold) took 66 / 89 / 133 us (x W^T, g W, g^T x) in the register-staged general kernel (gemm_mfma.hip) and take
// 37.4 / 38.4 / 44.3 (34.6 / 35.5 / 38.8 from cache).  The exact form stays for whole tiles: 4096 x 4096 x 2048 against
// 4088 x 4088 x 2048 takes 66.3 / 68.1 us (NT), 66.0 / 70.8 (NN), 65.5 / 71.2 (TN), 66.4 / 70.3 (TT); with half the M
// or N the two are within 5% either way.  Tile indices are read back into scalar registers (readfirstlane): from the
// vector registers that their divisions leave them in, every copy was a loop over distinct resources (806 x 4096 x 3840
// 45.8 us so, 41.3 now).
//
// DQ8 (the fused int8 linear y = x deq(q)^T + bias): B is int8 q [N][K] with one bf16 scale per row and
// 64-column block, so a K step covers exactly one scale block.  The raw int8 rows of step kt + 3 are copied
// global -> LDS during step kt (a ring of three int8 tiles: a copy still has two steps to land before it
// is converted); during step kt every thread converts 8-element pieces of step kt + 1's tile to
// deq = round(float(q) * float(scale)) in the input dtype (the exact product, one RNE rounding,
// as the standalone dequant) and writes it into the swizzled B tile of step kt + 1 (two such tiles), which
// the MFMAs then read exactly as a copied B tile.  The step barrier also waits for these LDS writes.
#pragma once

#include <type_traits>
#include <utility>

#include "gemm_dma.h"
#include "lds_stage.h"

namespace hk {
namespace {

// f(std::integral_constant<int, I>()) for I = 0 .. N - 1, unrolled at compile time (ring buffers are separate
// LDS objects picked by a compile-time index)
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>());
}
template <typename T, int BM, int BN, int WM, int WN, bool ATR, bool BTR, bool DQ8, int RING = 3, bool F32OUT = false,
          bool EDGE = false>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void mm_dma(hrt_mm_args p, int tiles_m, int tiles_n, int xbm,
                                                                   uint64_t dq_scale, int64_t dq_nblocks,
                                                                   int64_t kslice) {
  static_assert(!DQ8 || !BTR, "int8 B is staged as [n][k] rows");
  static_assert(RING == 3 || (RING == 2 && !DQ8), "three-buffer ring, or two buffers for the plain GEMM");
  constexpr int WNN = BN / WN;         // wavefronts along n
  constexpr int NW = (BM / WM) * WNN;  // wavefronts
  constexpr int FM = WM / 32, FN = WN / 32;  // 32 x 32 accumulators per wavefront along m, n
  static_assert(BM % WM == 0 && BN % WN == 0 && WM % 32 == 0 && WN % 32 == 0 && NW >= 4, "tile shape");
  constexpr int A_ROWS = ATR ? GBK : BM, A_NCH = ATR ? BM / 8 : GBK / 8;
  constexpr int B_ROWS = BTR ? GBK : BN, B_NCH = BTR ? BN / 8 : GBK / 8;
  constexpr int A_ROWB = A_NCH * 16, B_ROWB = B_NCH * 16;
  constexpr int A_TILE = A_ROWS * A_ROWB, B_TILE = B_ROWS * B_ROWB;
  constexpr int IPA = A_ROWS * A_NCH / 64 / NW, IPB = B_ROWS * B_NCH / 64 / NW;  // copies per wavefront
  static_assert(IPA >= 1 && IPB >= 1 && IPA * NW * 64 == A_ROWS * A_NCH && IPB * NW * 64 == B_ROWS * B_NCH &&
                    IPA + IPB <= 16, "copy split");
  constexpr int RS = 40;                  // epilogue row stride (floats): conflict-free half-wave writes
  constexpr int AREA = WM * RS * 4;       // one wavefront's epilogue area (bytes)
  constexpr int PA = A_TILE / AREA, PB = B_TILE / AREA;  // epilogue areas per A / B tile
  static_assert(2 * PA + 2 * PB >= NW, "epilogue areas fit the tiles");
  // DQ8: int8 tiles of BN rows x 64 bytes (4 chunks, unswizzled); each thread converts CPT 8-element pieces
  // per step, piece c = row c / 8, bf16 chunk c % 8
  constexpr int Q_TILE = DQ8 ? BN * GBK : 16, IPQ = DQ8 ? BN * 4 / 64 / NW : 1, CPT = DQ8 ? BN * 8 / (NW * 64) : 1;
  static_assert(!DQ8 || (IPQ >= 1 && IPA + IPQ <= 16 && CPT * NW * 64 == BN * 8), "int8 copy split");
  // separate LDS objects per buffer, so that reads of one are known not to alias copies into another
  __shared__ __attribute__((aligned(1024))) uint8_t a0_raw[A_TILE], a1_raw[A_TILE], a2_raw[RING >= 3 ? A_TILE : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t b0_raw[B_TILE], b1_raw[B_TILE];
  __shared__ __attribute__((aligned(1024))) uint8_t b2_raw[DQ8 ? Q_TILE : RING >= 3 ? B_TILE : 16];  // DQ8: int8 tile 0
  __shared__ __attribute__((aligned(DQ8 ? 1024 : 16))) uint8_t q1_raw[Q_TILE], q2_raw[Q_TILE];
  HK_L uint8_t* const A0 = (HK_L uint8_t*)a0_raw;
  HK_L uint8_t* const A1 = (HK_L uint8_t*)a1_raw;
  HK_L uint8_t* const B0 = (HK_L uint8_t*)b0_raw;
  auto abuf = [&](auto ic) {
    constexpr int I = decltype(ic)::value;
    return (HK_L uint8_t*)(I == 0 ? a0_raw : I == 1 ? a1_raw : a2_raw);
  };
  auto bbuf = [&](auto ic) {
    constexpr int I = decltype(ic)::value;
    return (HK_L uint8_t*)(I == 0 ? b0_raw : I == 1 ? b1_raw : b2_raw);
  };
  HK_L uint8_t* const Q0 = (HK_L uint8_t*)b2_raw;
  HK_L uint8_t* const Q1 = (HK_L uint8_t*)q1_raw;
  HK_L uint8_t* const Q2 = (HK_L uint8_t*)q2_raw;
  auto qbuf = [&](auto ic) { constexpr int I = decltype(ic)::value; return I == 0 ? Q0 : I == 1 ? Q1 : Q2; };

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WNN, wn = wave % WNN;
  const int l32 = lane & 31, h = lane >> 5, s16 = lane & 15, g2 = (lane >> 4) & 1;
  // Workgroups are dealt to the eight XCDs in turn (workgroup i to XCD i % 8), and each XCD has its own L2.
  // xbm > 0 (a batch of 1, 2, 4 or 8 products whose tile count per product divides into 8 / batch blocks):
  // XCD x takes product x / (8 / batch) and, of its tile grid, one xbm x (count / (8 / batch) / xbm) block,
  // the block shape the launcher chose to minimise the A and B panel bytes each XCD reads (a split-K
  // product's K slices are its batch).  xbm = 0: tiles numbered n-fastest, products one after another.
  const uint32_t tile = blockIdx.x;
  uint32_t tn = tile % (uint32_t)tiles_n, tm = (tile / (uint32_t)tiles_n) % (uint32_t)tiles_m;
  uint32_t bz = tile / ((uint32_t)tiles_n * (uint32_t)tiles_m);
  if (xbm > 0) {
    const uint32_t G = 8 / (uint32_t)p.batch;  // XCDs per product
    const uint32_t bnw = (uint32_t)tiles_m * (uint32_t)tiles_n / G / (uint32_t)xbm, nbn = (uint32_t)tiles_n / bnw;
    const uint32_t x = tile % 8, loc = tile / 8, sub = x % G;
    bz = x / G;
    tm = (sub / nbn) * (uint32_t)xbm + loc / bnw;
    tn = (sub % nbn) * bnw + loc % bnw;
  }
  if constexpr (EDGE) {
    // the divisions leave these in vector registers, and with them every address computed from them; a buffer resource
    // built there is wrapped in a loop over the lanes at each copy (ten instructions and a branch, between the MFMAs)
    tm = __builtin_amdgcn_readfirstlane(tm), tn = __builtin_amdgcn_readfirstlane(tn), bz = __builtin_amdgcn_readfirstlane(bz);
  }
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  // this workgroup's K range: all of it, or slice bz of a product split along K
  int64_t k0 = 0;
  int K = (int)p.K;
  if (F32OUT && kslice > 0) {
    k0 = bz * kslice;
    K = (int)(p.K - k0 < kslice ? p.K - k0 : kslice);
  }
  const int nk = EDGE ? (K + GBK - 1) / GBK : K / GBK;
  // EDGE: K step 0 is the partial one.  The operands are addressed as if K began kskip elements earlier, and
  // the copies of step 0 read zeros there, so every later step is whole and needs no mask.
  const int kskip = EDGE && !DQ8 ? nk * GBK - K : 0;
  k0 -= kskip;

  // copy sources (bytes) of K step 0 and the per-step advance
  const HK_G uint8_t* Ab = reinterpret_cast<const HK_G uint8_t*>(gcptr<uint16_t>(p.a) + bz * p.a_sb +
                                                                 (ATR ? m0 : m0 * p.a_sm) + k0 * p.a_sk);
  // (DQ8: B = q, strides in bytes, one byte per element)
  constexpr int BEL = DQ8 ? 1 : 2;
  const HK_G uint8_t* Bb = DQ8 ? gcptr<uint8_t>(p.b) + n0 * p.b_sn + k0
                               : reinterpret_cast<const HK_G uint8_t*>(gcptr<uint16_t>(p.b) + bz * p.b_sb +
                                                                       (BTR ? n0 : n0 * p.b_sn) + k0 * p.b_sk);
  const uint32_t ass = (uint32_t)((ATR ? p.a_sk : p.a_sm) * 2), bss = (uint32_t)((BTR ? p.b_sk : p.b_sn) * BEL);
  const int64_t astep = ATR ? (int64_t)GBK * p.a_sk * 2 : GBK * 2;
  const int64_t bstep = BTR ? (int64_t)GBK * p.b_sk * BEL : GBK * BEL;
  constexpr int IPBQ = DQ8 ? IPQ : IPB, BQ_NCH = DQ8 ? 4 : B_NCH;
  const DmaLanes alo = EDGE ? DmaLanes{} : dma_lane_offsets<A_NCH>(ass, lane, wave * IPA);
  const DmaLanes blo = EDGE ? DmaLanes{} : dma_lane_offsets<BQ_NCH>(bss, lane, wave * IPBQ);
  // EDGE: lane offsets of whole K steps (aeo, beo) and of step 0 (ae0, be0); rows / columns past M and N read
  // zeros and their outputs are not stored
  uint32_t aeo[IPA], beo[IPBQ], ae0[IPA], be0[IPBQ];
  if constexpr (EDGE) {
    const int ml = p.M - m0 < BM ? (int)(p.M - m0) : BM, nl = p.N - n0 < BN ? (int)(p.N - n0) : BN;
    edge_lane_offsets<A_NCH>(aeo, ass, lane, wave * IPA, 0, ATR ? GBK : ml, 0, ATR ? ml / 8 : A_NCH);
    edge_lane_offsets<BQ_NCH>(beo, bss, lane, wave * IPBQ, 0, BTR ? GBK : nl, 0, BTR ? nl / 8 : BQ_NCH);
    edge_lane_offsets<A_NCH>(ae0, ass, lane, wave * IPA, ATR ? kskip : 0, ATR ? GBK : ml, ATR ? 0 : kskip / 8, ATR ? ml / 8 : A_NCH);
    edge_lane_offsets<BQ_NCH>(be0, bss, lane, wave * IPBQ, BTR ? kskip : 0, BTR ? GBK : nl, BTR ? 0 : kskip / 8,
                              BTR ? nl / 8 : BQ_NCH);
  }
  // copy c of this wavefront's share of K step ks's A tile (B tile; DQ8: int8 tile) into `dst`
  auto copy_a = [&](int ks, HK_L uint8_t* dst, int c) {
    if constexpr (EDGE) edge_copy(edge_rsrc(Ab + ks * astep), dst, wave * IPA + c, ks == 0 ? ae0[c] : aeo[c]);
    else dma_tile_part<A_NCH, A_ROWS, NW>(Ab + ks * astep, ass, dst, wave, alo, c);
  };
  auto copy_b = [&](int ks, HK_L uint8_t* dst, int c) {
    if constexpr (EDGE) edge_copy(edge_rsrc(Bb + ks * bstep), dst, wave * IPBQ + c, ks == 0 ? be0[c] : beo[c]);
    else dma_tile_part<BQ_NCH, DQ8 ? BN : B_ROWS, NW>(Bb + ks * bstep, bss, dst, wave, blo, c);
  };

  // fragment offsets inside a tile for m (n) sub-tile i (j) and 16-wide K slice kk; a transposed operand
  // uses two column reads per fragment (rows 16 kk + 8 h + 4 t + (s >> 2), t = 0, 1: entries kk = 0, 1)
  int aoff[FM][4], boff[FN][4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if constexpr (!ATR) {
        aoff[i][kk] = tile_off<A_NCH>(wm * WM + i * 32 + l32, 2 * kk + h);
      } else {
        const int col = wm * WM + i * 32 + 16 * g2 + 4 * (s16 & 3);
        aoff[i][kk] = kk < 2 ? tile_off<A_NCH>(8 * h + 4 * (kk & 1) + (s16 >> 2), col >> 3) + (s16 & 1) * 8 : 0;
      }
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (!BTR) {
        boff[j][kk] = tile_off<B_NCH>(wn * WN + j * 32 + l32, 2 * kk + h);
      } else {
        const int col = wn * WN + j * 32 + 16 * g2 + 4 * (s16 & 3);
        boff[j][kk] = kk < 2 ? tile_off<B_NCH>(8 * h + 4 * (kk & 1) + (s16 >> 2), col >> 3) + (s16 & 1) * 8 : 0;
      }
    }
  }
  auto afrag = [&](const HK_L uint8_t* At, int i, int kk) -> u32x4 {
    if constexpr (!ATR) {
      return *reinterpret_cast<const HK_L u32x4*>(At + aoff[i][kk]);
    } else {
      const u32x2 lo = lds_tr4(At + aoff[i][0] + kk * 16 * A_ROWB), hi = lds_tr4(At + aoff[i][1] + kk * 16 * A_ROWB);
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };
  auto bfrag = [&](const HK_L uint8_t* Bt, int j, int kk) -> u32x4 {
    if constexpr (!BTR) {
      return *reinterpret_cast<const HK_L u32x4*>(Bt + boff[j][kk]);
    } else {
      const u32x2 lo = lds_tr4(Bt + boff[j][0] + kk * 16 * B_ROWB), hi = lds_tr4(Bt + boff[j][1] + kk * 16 * B_ROWB);
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = zero16();

  // DQ8 conversion: chunk u of this thread in the int8 tile of K step ks (buffer Qt) -> B tile Bt
  const HK_G uint16_t* scl = gcptr<uint16_t>(dq_scale) + (DQ8 ? n0 * dq_nblocks + k0 / GBK : 0);
  auto dq_scales = [&](int ks, float* sv) {
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      int row = (u * NW * 64 + (int)threadIdx.x) >> 3;
      if (EDGE && n0 + row >= p.N) row = (int)(p.N - 1 - n0);  // the column is not stored
      sv[u] = bf16_bits_to_f32(scl[row * dq_nblocks + ks]);
    }
  };
  // 8 int8 -> 8 values of T per piece: the 8 lanes of a group write the 8 chunks of one 128-byte B row
  // (LDS writes are conflict-free when each group of 8 consecutive lanes stays inside one 128-byte row,
  // measured), and the int8 reads are contiguous 8-byte pieces.
  auto dq_convert = [&](const HK_L uint8_t* Qt, HK_L uint8_t* Bt, const float* sv) {
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
      const int c = u * NW * 64 + (int)threadIdx.x, row = c >> 3, ch = c & 7;
      const u32x2 w = *reinterpret_cast<const HK_L u32x2*>(Qt + c * 8);
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = (float)(int8_t)(((i < 4 ? w.x : w.y) >> (8 * (i & 3))) & 0xffu) * sv[u];
      // round to the input dtype: the hardware pack (RNE) when the products are finite, which they are
      // unless the scale is inf or NaN; then the software rounding, which maps NaN to 0x7FC0 like dq8_*
      const u32x4 h = __builtin_isfinite(sv[u]) ? u32x4{cvt2<T>(v[0], v[1]), cvt2<T>(v[2], v[3]), cvt2<T>(v[4], v[5]), cvt2<T>(v[6], v[7])}
                                                 : u32x4{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7])};
      *reinterpret_cast<HK_L u32x4*>(Bt + tile_off<B_NCH>(row, ch)) = h;
    }
  };
  const int k1 = nk > 1 ? 1 : 0, k2 = nk > 2 ? 2 : nk - 1;
  float svq[CPT];  // DQ8: scales of the int8 tile that the next step converts (loaded a step ahead)
  if constexpr (!DQ8 && RING == 2) {
    // step 0; each step then copies the next one into the other buffer and waits for it at its end
#pragma unroll
    for (int c = 0; c < IPA; ++c) copy_a(0, A0, c);
#pragma unroll
    for (int c = 0; c < IPB; ++c) copy_b(0, B0, c);
    barrier_keep_vm_lds<0>();
  } else if constexpr (!DQ8) {
    // steps 0 .. RING - 2 into buffers 0 .. RING - 2 (step min(s, nk - 1): a short K re-copies its last step
    // into buffers nobody reads)
    static_for<RING - 1>([&](auto ic) {
      constexpr int S = decltype(ic)::value;
      const int ks = S < nk ? S : nk - 1;
#pragma unroll
      for (int c = 0; c < IPA; ++c) copy_a(ks, abuf(ic), c);
#pragma unroll
      for (int c = 0; c < IPB; ++c) copy_b(ks, bbuf(ic), c);
      issue_order_fence();
    });
    barrier_keep_vm<(RING - 2) * (IPA + IPB)>();  // step 0 landed everywhere, steps 1 .. RING - 2 in flight
  } else {
    // int8 steps 0, 1, 2 and A steps 0, 1; step 0's int8 tile converted before the loop
    float sv[CPT];
    dq_scales(0, sv);
#pragma unroll
    for (int c = 0; c < IPQ; ++c) copy_b(0, Q0, c);
#pragma unroll
    for (int c = 0; c < IPA; ++c) copy_a(0, A0, c);
    issue_order_fence();
#pragma unroll
    for (int c = 0; c < IPA; ++c) copy_a(k1, A1, c);
#pragma unroll
    for (int c = 0; c < IPQ; ++c) copy_b(k1, Q1, c);
#pragma unroll
    for (int c = 0; c < IPQ; ++c) copy_b(k2, Q2, c);
    barrier_keep_vm<IPA + 2 * IPQ>();  // int8 step 0 and A step 0 landed everywhere
    dq_scales(k1, svq);
    dq_convert(Q0, B0, sv);
    barrier_keep_vm_lds<0>();  // B tile 0 written; the other copies landed
  }

  // K step kt: MFMAs from buffer kt % 3, copies of step min(kt + 2, nk - 1) into buffer (kt + 2) % 3 (read
  // by step kt - 1, whose readers all passed the previous barrier) placed after the first MFMAs; no copy is
  // issued for steps past the end.  Before the barrier that ends
  // the step each wavefront waits for its copies of the previous step only, so step kt + 1's buffer is
  // complete after the barrier while the copies of step kt + 2 stay in flight.  DQ8: B tiles alternate
  // (kt % 2), int8 step min(kt + 3, nk - 1) is copied into int8 buffer kt % 3 (converted during step
  // kt - 1) and int8 step kt + 1 (buffer (kt + 1) % 3, landed at the last barrier) is converted into B
  // tile (kt + 1) % 2 (last read in step kt - 1); steps past the end convert a repeat nobody reads.
  auto step = [&](auto bc, auto bq, int kt) {
    constexpr int BUF = decltype(bc)::value;
    constexpr int NXT = DQ8 ? (BUF + 2) % 3 : (BUF + RING - 1) % RING;
    constexpr int BB = decltype(bq)::value;  // DQ8: B tile kt % 2
    constexpr int AHEAD = RING - 1;          // steps between a copy and its use
    const int kn = kt + AHEAD < nk ? kt + AHEAD : nk - 1;
    const HK_L uint8_t* At = abuf(bc);
    const HK_L uint8_t* Bt = DQ8 ? bbuf(bq) : bbuf(bc);
    const int kq = DQ8 ? (kt + 3 < nk ? kt + 3 : nk - 1) : kn;
    // No copies past the last K step: the ring buffers they would fill are the epilogue's staging areas.
    // (DQ8: A runs AHEAD = 2 steps ahead, the int8 tiles 3.)
    const bool more_a = kt + AHEAD < nk, more_b = DQ8 ? kt + 3 < nk : more_a;
    float sv[CPT];
    if constexpr (DQ8) {
#pragma unroll
      for (int u = 0; u < CPT; ++u) sv[u] = svq[u];
      dq_scales(kt + 2 < nk ? kt + 2 : nk - 1, svq);
    }
    // the same copies for steps after the first (kn, kq >= 1 whenever a copy is issued: no mask along K)
    const HK_G uint8_t* an = Ab + kn * astep;
    const HK_G uint8_t* bn = Bb + kq * bstep;
    auto next_a = [&](HK_L uint8_t* dst, int c) {
      if constexpr (EDGE) edge_copy(edge_rsrc(an), dst, wave * IPA + c, aeo[c]);
      else dma_tile_part<A_NCH, A_ROWS, NW>(an, ass, dst, wave, alo, c);
    };
    auto next_b = [&](HK_L uint8_t* dst, int c) {
      if constexpr (EDGE) edge_copy(edge_rsrc(bn), dst, wave * IPBQ + c, beo[c]);
      else dma_tile_part<BQ_NCH, DQ8 ? BN : B_ROWS, NW>(bn, bss, dst, wave, blo, c);
    };
    // Sub-tiles of at least two accumulators: the fragments of K slice kk + 1 are read while slice kk's
    // MFMAs run (two register sets, each slice fenced by sched_barrier: in the compiler's own order every
    // slice waited for its reads; 1024 x 2048 x 8192 -3%, the fused int8 linear -3%, the DiT stack -2%).
    // 64 x 64 tiles (one MFMA per slice) keep the compiler's order, which measured faster for them.
    constexpr bool AHEAD1 = FM * FN >= 2;
    u32x4 af[2][FM], bf[2][FN];
    auto rdk = [&](int kk) {
#pragma unroll
      for (int i = 0; i < FM; ++i) af[kk & 1][i] = afrag(At, i, kk);
#pragma unroll
      for (int j = 0; j < FN; ++j) bf[kk & 1][j] = bfrag(Bt, j, kk);
    };
    if constexpr (AHEAD1) rdk(0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if constexpr (AHEAD1) {
        __builtin_amdgcn_sched_barrier(0);
        if (kk + 1 < 4) rdk(kk + 1);
      } else {
        rdk(kk);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = Mfma32<T>::mac(af[kk & 1][i], bf[kk & 1][j], acc[i][j]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = kk * 4 + q;
        if (c < IPA) {
          if (more_a) next_a(abuf(std::integral_constant<int, NXT>()), c);
        } else if constexpr (!DQ8) {
          if (c < IPA + IPB && more_b)
            next_b(bbuf(std::integral_constant<int, NXT>()), c - IPA);
        } else {
          if (c < IPA + IPQ && more_b)
            next_b(qbuf(std::integral_constant<int, BUF>()), c - IPA);
        }
      }
      if constexpr (DQ8) {
        if (kk == 1) dq_convert(qbuf(std::integral_constant<int, (BUF + 1) % 3>()), bbuf(std::integral_constant<int, BB ^ 1>()), sv);
      }
    }
    if constexpr (AHEAD1) __builtin_amdgcn_sched_barrier(0);
    // each wavefront lets exactly the copies it issued in this step stay in flight
    if constexpr (DQ8) {
      if (more_b) barrier_keep_vm_lds<IPA + IPQ>();
      else if (more_a) barrier_keep_vm_lds<IPA>();
      else barrier_keep_vm_lds<0>();
    } else if constexpr (RING >= 3) {
      // step kt + 1's copies (issued RING - 1 steps before it) must have landed; those of steps kt + 2 ..
      // min(kt + RING - 1, nk - 1), issued after them, may stay in flight (a count below the true one only
      // waits longer)
      const int last = kt + RING - 1 < nk - 1 ? kt + RING - 1 : nk - 1;
      const int fly = last - (kt + 1) > 0 ? last - (kt + 1) : 0;
      static_for<RING - 1>([&](auto ic) {
        constexpr int F = decltype(ic)::value;
        if (fly == F || (F == RING - 2 && fly > F)) barrier_keep_vm<F * (IPA + IPB)>();
      });
    } else {
      barrier_keep_vm_lds<0>();  // the next step's copies, issued in this one, have landed everywhere
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  if constexpr (!DQ8 && RING == 2) {
    int kt = 0;
    for (; kt + 2 <= nk; kt += 2) {
      step(I0(), I0(), kt);
      step(I1(), I0(), kt + 1);
    }
    if (kt < nk) step(I0(), I0(), kt);
  } else if constexpr (!DQ8) {
    int kt = 0;
    for (; kt + RING <= nk; kt += RING) static_for<RING>([&](auto ic) { step(ic, I0(), kt + decltype(ic)::value); });
    static_for<RING - 1>([&](auto ic) {
      if (kt + decltype(ic)::value < nk) step(ic, I0(), kt + decltype(ic)::value);
    });
  } else {
    // A and int8 buffers rotate by 3, B tiles by 2: blocks of 6 steps, leaving after any step
    for (int kt = 0;; kt += 6) {
      step(I0(), I0(), kt);
      if (kt + 1 >= nk) break;
      step(I1(), I1(), kt + 1);
      if (kt + 2 >= nk) break;
      step(I2(), I0(), kt + 2);
      if (kt + 3 >= nk) break;
      step(I0(), I1(), kt + 3);
      if (kt + 4 >= nk) break;
      step(I1(), I0(), kt + 4);
      if (kt + 5 >= nk) break;
      step(I2(), I1(), kt + 5);
      if (kt + 6 >= nk) break;
    }
  }
  __syncthreads();  // (the last step waited for its copies) the epilogue reuses the tiles

  // ---- epilogue: per n sub-tile j, the WM x 32 fp32 block goes through this wavefront's area as [m][n]
  float* const area = reinterpret_cast<float*>(wave < PA            ? a0_raw + wave * AREA
                                              : wave < 2 * PA        ? a1_raw + (wave - PA) * AREA
                                              : wave < 2 * PA + PB   ? b0_raw + (wave - 2 * PA) * AREA
                                                                     : b1_raw + (wave - 2 * PA - PB) * AREA);
  const bool has_bias = p.has_bias != 0;
  const HK_G uint16_t* bias = gcptr<uint16_t>(p.bias) + bz * p.bias_sb;
  HK_G uint16_t* C = gptr<uint16_t>(p.c) + bz * p.c_sb;
  HK_G float* C32 = gptr<float>(p.c) + bz * p.c_sb;  // F32OUT: unrounded fp32 results (split-K partials)
  constexpr int CAL = F32OUT ? 4 : 8;                // elements of C per 16 bytes
  const bool vec_c = !EDGE || (p.c % 16 == 0 && p.c_sm % CAL == 0 && (p.batch == 1 || p.c_sb % CAL == 0));
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int64_t gn = n0 + wn * WN + j * 32 + l32;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      float bv[16];  // beta * bias, all 16 loads in flight together
      if (has_bias) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
          int64_t bm = m0 + wm * WM + r, bn = gn;
          if constexpr (EDGE) bm = bm < p.M ? bm : p.M - 1, bn = bn < p.N ? bn : p.N - 1;
          bv[e] = p.beta * T::to_f32(bias[bm * p.bias_sm + bn * p.bias_sn]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) bv[e] = 0.f;
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
        area[r * RS + l32] = p.alpha * acc[i][j][e] + bv[e];
      }
    }
    // 4 lanes per 32-wide row, 8 floats each: 16 rows per pass
#pragma unroll
    for (int ps = 0; ps < WM / 16; ++ps) {
      const int r = ps * 16 + (lane >> 2), c8 = (lane & 3) * 8;
      const f32x4 x = *reinterpret_cast<const f32x4*>(area + r * RS + c8);
      const f32x4 y = *reinterpret_cast<const f32x4*>(area + r * RS + c8 + 4);
      const int64_t om = m0 + wm * WM + r, on = n0 + wn * WN + j * 32 + c8;
      const int64_t off = om * p.c_sm + on;
      if constexpr (EDGE) {
        if (om >= p.M || on >= p.N) continue;
        if (!(vec_c && on + 8 <= p.N)) {  // the last columns, or rows of C without 16-byte alignment
          const float o8[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (on + e < p.N) {
              if constexpr (F32OUT) C32[off + e] = o8[e];
              else C[off + e] = T::from_f32(o8[e]);
            }
          continue;
        }
      }
      if constexpr (F32OUT) {
        *reinterpret_cast<HK_G f32x4*>(C32 + off) = x;
        *reinterpret_cast<HK_G f32x4*>(C32 + off + 4) = y;
      } else {
        const float o8[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        *reinterpret_cast<HK_G u32x4*>(C + off) = pack8<T>(o8);
      }
    }
  }
}

// The XCD block of mm_dma for a tm x tn tile grid of each of `batch` products (batch 1, 2, 4 or 8; a
// split-K product's slices): the rows xbm of the block shape xbm x bn (xbm | tm, bn | tn, 8 / batch blocks
// per product, one per XCD) with the fewest panel bytes per XCD, xbm * a_panel + bn * b_panel (a_panel /
// b_panel: bytes of one BM-row A panel / BN-row B panel over K); 0 (n-fastest order) when the grid does not
// split so, or K < 2048 (one product) / 1536 (slices).  For the four K slices of a 1024 x 2048 output on
// 128 x 256 tiles each XCD then reads one slice's A panels and half its B panels instead of every slice's
// A panels: 2.6-4.6% faster (K = 6144 and 8192, slices + reduction 42.2 -> 41.1, 49.9 -> 48.5 us).
// The block order is used only where it reads at least 10% fewer panel bytes than the n-fastest order (which,
// with tn a multiple of 8, gives each XCD tn / 8 B panels and every A panel): where the two read the same,
// as at 1024 x 2048 x 8192 on 128 x 256 tiles, the block order measured ~1.5% slower.  Measured:
// 1024 x 2048 x 2048 on 64 x 64 tiles 15.4-16.1 us against 16.6-18.1 n-fastest (41.9 -> 33.6 MB of panels
// read), 4096 x 2048 x 8192 1.5% faster; but 1024^3 6.65 against 6.45 us although it reads 12.6 instead of
// 18.9 MB, so short reductions keep the n-fastest order.
int xcd_block_rows(int64_t tm, int64_t tn, int64_t batch, int64_t K, double a_panel, double b_panel) {
  if (batch < 1 || batch > 8 || 8 % batch != 0 || tn % 8 != 0) return 0;
  if (K < (batch == 1 ? 2048 : 1536)) return 0;
  const int64_t G = 8 / batch;  // XCDs per product
  if ((tm * tn) % G != 0) return 0;
  const int64_t per = tm * tn / G;
  int best = 0;
  double cost = 0.0;
  for (int64_t bm = 1; bm <= tm; ++bm) {
    if (tm % bm || per % bm) continue;
    const int64_t bn = per / bm;
    if (tn % bn) continue;
    const double c = bm * a_panel + bn * b_panel;
    if (best == 0 || c < cost) best = (int)bm, cost = c;
  }
  // n-fastest order: every XCD reads all A panels and tn / 8 B panels of every product
  const double n_fastest = batch * (tm * a_panel + (tn / 8) * b_panel);
  return best > 0 && cost <= 0.9 * n_fastest ? best : 0;
}

template <typename T, int BM, int BN, int WM, int WN, int RING, bool F32OUT, bool EDGE>
void queue_tile(const hrt_mm_args& a, const DmaForm& f, int64_t kslice, hipStream_t s) {
  const int tm = (int)cdiv(a.M, BM), tn = (int)cdiv(a.N, BN);
  const int64_t K = kslice > 0 ? kslice : a.K;
  const int xbm = xcd_block_rows(tm, tn, a.batch, K, (double)BM * K * 2, (double)BN * K * 2);
  const dim3 g((uint32_t)((int64_t)tm * tn * a.batch)), blk((BM / WM) * (BN / WN) * 64);
  const auto go = [&](auto ac, auto bc) {
    hipLaunchKernelGGL((mm_dma<T, BM, BN, WM, WN, decltype(ac)::value, decltype(bc)::value, false, RING, F32OUT, EDGE>), g, blk, 0,
                       s, a, tm, tn, xbm, (uint64_t)0, (int64_t)0, kslice);
  };
  using Y = std::true_type;
  using N = std::false_type;
  // 128 x 192: the 24-chunk rows of an N-contiguous B have no LDS swizzle
  if constexpr (BN != 192) {
    if (f.btr) {
      if (f.atr) go(Y(), Y());
      else go(N(), Y());
      return;
    }
  }
  if (f.atr) go(Y(), N());
  else go(N(), N());
}

template <typename T, int BM, int BN, int WM, int WN, bool F32OUT, bool EDGE>
void queue_tile_dq8(const hrt_mm_args& a, const DmaForm& f, const hrt_mm_dq8_args& d, int64_t kslice, hipStream_t s) {
  const int tm = (int)cdiv(a.M, BM), tn = (int)cdiv(a.N, BN);
  const int64_t K = kslice > 0 ? kslice : a.K;
  const int xbm = xcd_block_rows(tm, tn, a.batch, K, (double)BM * K * 2, (double)BN * K);
  const dim3 g((uint32_t)((int64_t)tm * tn * a.batch)), blk((BM / WM) * (BN / WN) * 64);
  if (!f.atr)
    hipLaunchKernelGGL((mm_dma<T, BM, BN, WM, WN, false, false, true, 3, F32OUT, EDGE>), g, blk, 0, s, a, tm, tn, xbm, d.scale,
                       d.nblocks, kslice);
  else
    hipLaunchKernelGGL((mm_dma<T, BM, BN, WM, WN, true, false, true, 3, F32OUT, EDGE>), g, blk, 0, s, a, tm, tn, xbm, d.scale,
                       d.nblocks, kslice);
}

}  // namespace

template <typename T>
bool dma_queue(const hrt_mm_args& a, GemmTile tile, int64_t kslice, hipStream_t s) {
  const DmaForm f = dma_form(a, kTileShape[tile].bm, kTileShape[tile].bn);
  if (!f.ok) return false;
  if (a.flags & HRT_MM_F32_OUT) {
    const bool exact = f.exact && (kslice == 0 || a.K % GBK == 0);
    switch (tile) {
      case T128x256:
        if (exact) queue_tile<T, 128, 256, 64, 64, 3, true, false>(a, f, kslice, s);
        else queue_tile<T, 128, 256, 64, 64, 3, true, true>(a, f, kslice, s);
        return true;
      case T128x128: queue_tile<T, 128, 128, 32, 64, 3, true, true>(a, f, kslice, s); return true;
      case T64x128: queue_tile<T, 64, 128, 32, 64, 3, true, true>(a, f, kslice, s); return true;
      case T64x64: queue_tile<T, 64, 64, 32, 32, 3, true, true>(a, f, kslice, s); return true;
      default: return false;
    }
  }
#define HK_TILE(BM, BN, WM, WN, RING)                                       \
  if (f.exact) queue_tile<T, BM, BN, WM, WN, RING, false, false>(a, f, 0, s); \
  else queue_tile<T, BM, BN, WM, WN, RING, false, true>(a, f, 0, s);          \
  return true
  switch (tile) {
    case T256x256: HK_TILE(256, 256, 64, 128, 2);
    case T128x256: HK_TILE(128, 256, 64, 64, 3);
    case T256x128: HK_TILE(256, 128, 64, 64, 3);
    case T128x128: HK_TILE(128, 128, 32, 64, 3);
    case T64x128: HK_TILE(64, 128, 32, 64, 3);
    case T64x64: HK_TILE(64, 64, 32, 32, 3);
    case T128x192:
      if (f.btr) return false;
      HK_TILE(128, 192, 32, 96, 3);
    default: return false;
  }
#undef HK_TILE
}

template <typename T>
bool dma_queue_dq8(const hrt_mm_dq8_args& d, GemmTile tile, uint64_t ws, int64_t splits, int64_t kslice, hipStream_t s) {
  hrt_mm_args a = dq8_as_mm(d);
  const DmaForm f = dma_form(a, kTileShape[tile].bm, kTileShape[tile].bn);
  if (!f.ok || f.btr || d.K % GBK || d.q % 16) return false;
  if (ws) {
    a.c = ws, a.batch = splits, a.c_sb = a.M * a.N, a.alpha = 1.f, a.has_bias = 0, a.flags = HRT_MM_F32_OUT;
    if (tile != T64x64) return false;
    queue_tile_dq8<T, 64, 64, 32, 32, true, true>(a, f, d, kslice, s);
    return true;
  }
#define HK_TILE(BM, BN, WM, WN)                                                  \
  if (f.exact) queue_tile_dq8<T, BM, BN, WM, WN, false, false>(a, f, d, 0, s);   \
  else queue_tile_dq8<T, BM, BN, WM, WN, false, true>(a, f, d, 0, s);            \
  return true
  switch (tile) {
    case T256x128: HK_TILE(256, 128, 64, 64);
    case T128x128: HK_TILE(128, 128, 32, 64);
    case T64x64: HK_TILE(64, 64, 32, 32);
    default: return false;
  }
#undef HK_TILE
}

}  // namespace hk
