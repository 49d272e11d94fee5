// Matrix-core GEMM "mm_mfma_{bf16,f16}" for gfx950:  c = alpha * a @ b + beta * bias, fp32 accumulate.
//
// Same contract as the reference's cooperative-matrix kernel (vkrt/shaders/mm_coop.comp.in:96-208):
// arbitrary strides (transposes and slices read in place), batched, bias broadcast through strides,
// epilogue alpha*acc + beta*bias with one rounding.  Built for CDNA4 instead of translated:
//   * v_mfma_f32_16x16x32 on 64-wide wavefronts; each wavefront owns a (BM/WM) x (BN/WN) sub-tile held
//     in accumulator registers for the whole K loop;
//   * A and B tiles are staged through LDS with K contiguous (+8 halves of row padding against bank
//     conflicts), double-buffered, one barrier per K step; the next tile's global loads are issued
//     before the current tile's MFMAs so HBM/L2 latency overlaps the math;
//   * global loads are 128-bit along the operand's contiguous axis: a K-contiguous operand goes straight
//     to its LDS row, an M-/N-contiguous one (W for dX = dY W, B of a row-major X @ B) is loaded as 8x8
//     blocks and transposed in registers before the 128-bit LDS store — no copies, no strided LDS writes;
//   * odd strides / alignments use a per-element gather loader on the same MMA core;
//   * tiles are numbered N-fastest so the default round-robin placement of workgroups over the 8 XCDs
//     gives each XCD a band of N-panels that it reads once into its own L2.
// This general kernel takes what the direct-to-LDS kernel (gemm_dma_kernel.h) does not: operand rows off 16-byte
// lines, a strided C.  The choice between them, the tile and the K split are made here (plan_gemm).
#include <array>
#include <cstring>
#include <type_traits>
#include <utility>

#include "../hrt/registry.h"
#include "gemm_dma.h"
#include "gemm_skinny.h"
#include "lds_stage.h"

namespace hk {

bool mm_check_operands(const hrt_mm_args& a, uint64_t elem, hrt::LaunchCtx& ctx);
int64_t mm_f32_workspace(const hrt_mm_args& a);  // gemm_f32.hip
void mm_f32_plan(const hrt_mm_args& a, bool may_split, hrt_mm_plan* out);

namespace {

enum LoadMode { KVEC = 0, MNVEC = 1, GATHER = 2 };

constexpr int BK = 64;       // K per LDS stage
constexpr int LDK = BK + 8;  // padded LDS row (halves)

template <int ROWS, int MODE>
struct TileLoader {
  // The ROWS x BK tile of an operand whose element (r, k) is at p[r * s_r + k * s_k]; rows >= nrows and
  // k >= nk read as zero.  load() fills registers, store() writes LDS as [ROWS][LDK] with K contiguous.
  static constexpr int CHUNKS = ROWS * BK / 8;  // 16-byte chunks per tile
  static constexpr int PER_THREAD_V = CHUNKS / 256 > 0 ? CHUNKS / 256 : 1;
  static constexpr int BLOCKS = (ROWS / 8) * (BK / 8);  // 8x8 blocks (MNVEC)
  static constexpr int PER_THREAD_T = BLOCKS / 256 > 0 ? BLOCKS / 256 : 1;
  static constexpr int ELEMS = ROWS * BK / 256;  // GATHER
  static_assert(CHUNKS % 256 == 0 || CHUNKS < 256, "tile/threads mismatch");

  const HK_G uint16_t* p;
  int64_t s_r, s_k, r0, nrows, nk;
  u32x4 v[MODE == KVEC ? PER_THREAD_V : (MODE == MNVEC ? 8 * PER_THREAD_T : 1)];
  uint16_t g[MODE == GATHER ? ELEMS : 1];

  __device__ __forceinline__ void load(int64_t k0) {
    const int t = threadIdx.x;
    if constexpr (MODE == KVEC) {
#pragma unroll
      for (int i = 0; i < PER_THREAD_V; ++i) {
        const int c = t + i * 256;
        const int r = c / (BK / 8), kc = c % (BK / 8);
        const int64_t gr = r0 + r, gk = k0 + kc * 8;
        if (c < CHUNKS && gr < nrows && gk < nk)
          v[i] = *reinterpret_cast<const HK_G u32x4*>(p + gr * s_r + gk);
        else
          v[i] = u32x4{0, 0, 0, 0};
      }
    } else if constexpr (MODE == MNVEC) {
#pragma unroll
      for (int i = 0; i < PER_THREAD_T; ++i) {
        const int b = t + i * 256;
        const int rb = b % (ROWS / 8), kb = b / (ROWS / 8);
        const int64_t gr = r0 + rb * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int64_t gk = k0 + kb * 8 + j;
          if (b < BLOCKS && gr < nrows && gk < nk)
            v[i * 8 + j] = *reinterpret_cast<const HK_G u32x4*>(p + gk * s_k + gr);
          else
            v[i * 8 + j] = u32x4{0, 0, 0, 0};
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < ELEMS; ++i) {
        const int e = t + i * 256;
        const int r = e / BK, k = e % BK;
        const int64_t gr = r0 + r, gk = k0 + k;
        g[i] = (gr < nrows && gk < nk) ? p[gr * s_r + gk * s_k] : (uint16_t)0;
      }
    }
  }

  __device__ __forceinline__ void store(uint16_t* lds) const {
    const int t = threadIdx.x;
    if constexpr (MODE == KVEC) {
#pragma unroll
      for (int i = 0; i < PER_THREAD_V; ++i) {
        const int c = t + i * 256;
        if (c < CHUNKS) {
          const int r = c / (BK / 8), kc = c % (BK / 8);
          *reinterpret_cast<u32x4*>(lds + r * LDK + kc * 8) = v[i];
        }
      }
    } else if constexpr (MODE == MNVEC) {
#pragma unroll
      for (int i = 0; i < PER_THREAD_T; ++i) {
        const int b = t + i * 256;
        if (b < BLOCKS) {
          const int rb = b % (ROWS / 8), kb = b / (ROWS / 8);
          u32x4 o[8];
          transpose8x8(&v[i * 8], o);
#pragma unroll
          for (int m = 0; m < 8; ++m) *reinterpret_cast<u32x4*>(lds + (rb * 8 + m) * LDK + kb * 8) = o[m];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < ELEMS; ++i) {
        const int e = t + i * 256;
        lds[(e / BK) * LDK + (e % BK)] = g[i];
      }
    }
  }
};

// B tile of the fused int8 linear: rows n of the int8 weight q [N, K] (contiguous), dequantized while
// staging: value = round_T(float(q[n, k]) * float(scale[n, k / 64])) — bit-identical to dq8 — so the
// matrix cores see exactly the weights dequant_int8 would have produced, without them touching HBM.
template <int ROWS, typename T>
struct Dq8Loader {
  static constexpr int CHUNKS = ROWS * BK / 8;  // 8 int8 per chunk
  static constexpr int PT = CHUNKS / 256 > 0 ? CHUNKS / 256 : 1;
  const HK_G int8_t* q;
  const HK_G uint16_t* scale;
  int64_t K, nblocks, r0, nrows;
  u32x2 v[PT];
  float sc[PT];

  __device__ __forceinline__ void load(int64_t k0) {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int c = threadIdx.x + i * 256;
      const int r = c / (BK / 8), kc = c % (BK / 8);
      const int64_t gr = r0 + r, gk = k0 + kc * 8;
      if (c < CHUNKS && gr < nrows && gk < K) {
        v[i] = *reinterpret_cast<const HK_G u32x2*>(q + gr * K + gk);
        sc[i] = bf16_bits_to_f32(scale[gr * nblocks + (gk >> 6)]);
      } else {
        v[i] = u32x2{0, 0};
        sc[i] = 0.f;
      }
    }
  }
  __device__ __forceinline__ void store(uint16_t* lds) const {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int c = threadIdx.x + i * 256;
      if (c < CHUNKS) {
        const int r = c / (BK / 8), kc = c % (BK / 8);
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (float)(int8_t)(((e < 4 ? v[i].x : v[i].y) >> (8 * (e & 3))) & 0xffu) * sc[i];
        *reinterpret_cast<u32x4*>(lds + r * LDK + kc * 8) = pack8<T>(f);
      }
    }
  }
};

// Main loop shared by the GEMM kernels: K in steps of BK through double-buffered LDS; acc[i][j] is the
// wavefront's (i, j) 16x16 accumulator tile.
template <typename T, int BM, int BN, int WM, int WN, class LA, class LB>
__device__ __forceinline__ void gemm_mainloop(LA& la, LB& lb, int64_t K, uint16_t (*lds)[(BM + BN) * LDK],
                                              f32x4 (&acc)[BM / WM / 16][BN / WN / 16]) {
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t nk = (K + BK - 1) / BK;
  la.load(0);
  lb.load(0);
  la.store(lds[0]);
  lb.store(lds[0] + BM * LDK);
  __syncthreads();
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  for (int64_t kt = 0; kt < nk; ++kt) {
    const bool more = kt + 1 < nk;
    if (more) {
      la.load((kt + 1) * BK);
      lb.load((kt + 1) * BK);
    }
    const uint16_t* As = lds[kt & 1];
    const uint16_t* Bs = As + BM * LDK;
#pragma unroll
    for (int ks = 0; ks < BK; ks += 32) {
      u32x4 af[TM], bfr[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = *reinterpret_cast<const u32x4*>(As + (wm * WTM + i * 16 + fr) * LDK + ks + fk);
#pragma unroll
      for (int j = 0; j < TN; ++j) bfr[j] = *reinterpret_cast<const u32x4*>(Bs + (wn * WTN + j * 16 + fr) * LDK + ks + fk);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<T>::mac(af[i], bfr[j], acc[i][j]);
    }
    if (more) {
      uint16_t* nxt = lds[(kt + 1) & 1];
      la.store(nxt);
      lb.store(nxt + BM * LDK);
    }
    __syncthreads();
  }
}

// Epilogue: c = alpha * acc + beta * bias, one rounding; lane holds rows 4*(lane/16)+r, column lane%16
// of every 16x16 tile.
// Epilogue: alpha * acc + beta * bias, one rounding (f32out: C is fp32 and takes the unrounded value, the
// split-K partials of HRT_MM_F32_OUT).  Each wavefront's WTM x WTN block goes through LDS in 32-column
// chunks so that a lane writes 8 consecutive outputs of a row (one 16-byte store when C's row is contiguous
// and aligned) instead of 2-byte stores scattered over 4 rows.
constexpr int EPI_RS = 36;  // floats per LDS row of a chunk (conflict-free writes, 16-byte aligned rows)
template <typename T, int BM, int BN, int WM, int WN>
__device__ __forceinline__ void gemm_epilogue(const f32x4 (&acc)[BM / WM / 16][BN / WN / 16], HK_G uint16_t* C, int64_t c_sm,
                                              int64_t c_sn, const HK_G uint16_t* bias, int64_t bias_sm, int64_t bias_sn,
                                              bool has_bias, float alpha, float beta, int64_t m0, int64_t n0, int64_t M,
                                              int64_t N, uint16_t (*lds)[(BM + BN) * LDK], bool f32out = false) {
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  static_assert(WTN % 32 == 0 && WM * WN * WTM * EPI_RS * 4 <= 2 * (BM + BN) * LDK * 2, "epilogue chunks fit the tiles");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;
  float* const area = reinterpret_cast<float*>(&lds[0][0]) + wave * WTM * EPI_RS;
  __syncthreads();  // every wavefront is done with the K loop's tiles
#pragma unroll
  for (int jc = 0; jc < WTN / 32; ++jc) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          area[(i * 16 + (lane >> 4) * 4 + r) * EPI_RS + jj * 16 + (lane & 15)] = acc[i][2 * jc + jj][r];
    // WTM rows x 4 pieces of 8 columns; LDS reads and writes of one wavefront complete in order
#pragma unroll
    for (int ps = 0; ps < WTM / 16; ++ps) {
      const int q = ps * 64 + lane, row = q >> 2, c8 = (q & 3) * 8;
      const f32x4 x = *reinterpret_cast<const f32x4*>(area + row * EPI_RS + c8);
      const f32x4 y = *reinterpret_cast<const f32x4*>(area + row * EPI_RS + c8 + 4);
      const int64_t gm = m0 + wm * WTM + row, gn = n0 + wn * WTN + jc * 32 + c8;
      if (gm >= M || gn >= N) continue;
      float o[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
      const bool full = gn + 8 <= N;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] *= alpha;
      if (has_bias) {
        const HK_G uint16_t* bp = bias + gm * bias_sm + gn * bias_sn;
        if (full && bias_sn == 1 && ((uint64_t)bp & 15) == 0) {  // one 16-byte load of the bias row
          const u32x4 bv = *reinterpret_cast<const HK_G u32x4*>(bp);
#pragma unroll
          for (int w = 0; w < 4; ++w) o[2 * w] += beta * lo16<T>(bv[w]), o[2 * w + 1] += beta * hi16<T>(bv[w]);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (full || gn + e < N) o[e] += beta * T::to_f32(bp[e * bias_sn]);
        }
      }
      if (f32out) {
        HK_G float* c = reinterpret_cast<HK_G float*>(C) + gm * c_sm + gn * c_sn;
        if (full && c_sn == 1 && ((uint64_t)c & 15) == 0) {
          *reinterpret_cast<HK_G f32x4*>(c) = f32x4{o[0], o[1], o[2], o[3]};
          *reinterpret_cast<HK_G f32x4*>(c + 4) = f32x4{o[4], o[5], o[6], o[7]};
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (gn + e < N) c[e * c_sn] = o[e];
        }
      } else {
        HK_G uint16_t* c = C + gm * c_sm + gn * c_sn;
        if (full && c_sn == 1 && ((uint64_t)c & 15) == 0) {
          *reinterpret_cast<HK_G u32x4*>(c) = pack8<T>(o);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (gn + e < N) c[e * c_sn] = T::from_f32(o[e]);
        }
      }
    }
  }
}

template <typename T, int BM, int BN, int WM, int WN, int AMODE, int BMODE>
__global__ __launch_bounds__(256) void mm_mfma(hrt_mm_args p, int64_t tiles_m, int64_t tiles_n) {
  static_assert(WM * WN == 4, "four wavefronts");
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][(BM + BN) * LDK];
  const int64_t tile = blockIdx.x;
  const int64_t tn = tile % tiles_n, tm = (tile / tiles_n) % tiles_m, bz = tile / (tiles_n * tiles_m);
  const int64_t m0 = tm * BM, n0 = tn * BN;
  // A as rows m with K; B as rows n with K.
  TileLoader<BM, AMODE> la;
  la.p = gcptr<uint16_t>(p.a) + bz * p.a_sb;
  la.s_r = p.a_sm, la.s_k = p.a_sk, la.r0 = m0, la.nrows = p.M, la.nk = p.K;
  TileLoader<BN, BMODE> lb;
  lb.p = gcptr<uint16_t>(p.b) + bz * p.b_sb;
  lb.s_r = p.b_sn, lb.s_k = p.b_sk, lb.r0 = n0, lb.nrows = p.N, lb.nk = p.K;
  f32x4 acc[BM / WM / 16][BN / WN / 16];
  gemm_mainloop<T, BM, BN, WM, WN>(la, lb, p.K, lds, acc);
  const bool f32out = (p.flags & HRT_MM_F32_OUT) != 0;
  HK_G uint16_t* const C = f32out ? reinterpret_cast<HK_G uint16_t*>(gptr<float>(p.c) + bz * p.c_sb)
                                  : gptr<uint16_t>(p.c) + bz * p.c_sb;
  gemm_epilogue<T, BM, BN, WM, WN>(acc, C, p.c_sm, p.c_sn, gcptr<uint16_t>(p.bias) + bz * p.bias_sb, p.bias_sm,
                                   p.bias_sn, p.has_bias != 0, p.alpha, p.beta, m0, n0, p.M, p.N, lds, f32out);
}

template <typename T, int BM, int BN, int WM, int WN, int AMODE>
__global__ __launch_bounds__(256) void mm_dq8_mfma(hrt_mm_dq8_args p, int64_t tiles_m, int64_t tiles_n) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][(BM + BN) * LDK];
  const int64_t tile = blockIdx.x;
  const int64_t tn = tile % tiles_n, tm = tile / tiles_n;
  const int64_t m0 = tm * BM, n0 = tn * BN;
  TileLoader<BM, AMODE> la;
  la.p = gcptr<uint16_t>(p.x);
  la.s_r = p.x_sm, la.s_k = p.x_sk, la.r0 = m0, la.nrows = p.M, la.nk = p.K;
  Dq8Loader<BN, T> lb;
  lb.q = gcptr<int8_t>(p.q);
  lb.scale = gcptr<uint16_t>(p.scale);
  lb.K = p.K, lb.nblocks = p.nblocks, lb.r0 = n0, lb.nrows = p.N;
  f32x4 acc[BM / WM / 16][BN / WN / 16];
  gemm_mainloop<T, BM, BN, WM, WN>(la, lb, p.K, lds, acc);
  gemm_epilogue<T, BM, BN, WM, WN>(acc, gptr<uint16_t>(p.y), p.N, 1, gcptr<uint16_t>(p.bias), 0,
                                   1, p.has_bias != 0, p.alpha, p.beta, m0, n0, p.M, p.N, lds);
}

// ---- choice of tile and K split for the direct-to-LDS kernel -----------------------------------------------------
// Cost model of mm_dma, in microseconds, fitted to 3225 products (all layouts, 2e-4 to 140 GFLOP, layers of 256 to 4096
// tokens among them) timed on every tile and split, with operands from HBM (rotated through 600 MB) and from cache: what
// it picks takes 1.8% longer than the best of them on average.  The numbers order the choices; as times they are rough.
// A grid runs in rounds of `slots` tiles (the workgroups that 256 CUs hold at once).  A K step takes step[0] on a nearly
// empty chip, step[i] when i workgroups a CU are at work and what lies between for part-filled rounds (the tiles share
// L2 and power), kMasked times that in masked forms, whose last tiles hold less.  A round also takes its first loads and the
// writing of its outputs.
struct TileCost {
  uint32_t slots;
  double first, step[4];
};
constexpr TileCost kTileCost[kGemmTiles] = {
    {256, 3.12, {1.387, 2.029}},                 // 256 x 256
    {256, 3.031, {0.6527, 1.156}},               // 128 x 256
    {256, 1.854, {0.8738, 1.423}},               // 256 x 128
    {256, 2.695, {0.6901, 0.8706}},              // 128 x 192
    {256, 1.571, {0.4424, 0.7417}},              // 128 x 128
    {512, 0.6518, {0.5139, 0.5901, 2.027}},      // 64 x 128
    {768, 0.1275, {0.3852, 0.4836, 0.7293, 0.9727}}, // 64 x 64
};
constexpr double kMasked = 0.9717, kHalfLines = 1.178;

double tile_us(const TileCost& c, TileShape sh, uint32_t tiles, double steps) {
  const uint32_t full = tiles / c.slots, rest = tiles % c.slots;  // 32 bits: a plan costs a call well under 1 us
  const double out = 5.499 * (c.slots / 256) * sh.bm * sh.bn / 65536;  // a full round's outputs
  double us = full * (c.first + out + steps * c.step[c.slots / 256]);
  if (rest) {
    const uint32_t i = rest / 256;
    const double last = c.step[i] + (c.step[i + 1] - c.step[i]) * (rest - 256 * i) / 256;
    us += c.first + out * rest / c.slots + steps * last;
  }
  return us;
}
// The partial products of a split: their write and read, the second launch and each slice's start.
double split_us(int64_t splits, int64_t M, int64_t N) { return 1.305 + 0.2128 * splits + 1.625 * (double)splits * M * N * 4 / 5e6; }

struct GemmPlan {
  int tile = -1;  // GemmTile, -1: the direct-to-LDS kernel does not take the product
  int64_t splits = 1, kslice = 0;
  double us = 0.0;
};

// The cheapest tile, and for one product (no batch) the cheapest number of K slices when may_split: under-filled
// grids with a long reduction then run several slices per tile, whose fp32 partial products a second kernel adds
// in order.  A split has to promise kSplitGain: its workspace and second launch cost the host a few microseconds, which a
// program of small layers waits for.
constexpr double kSplitGain = 6.43;
GemmPlan search_plan(const hrt_mm_args& a, bool may_split) {
  GemmPlan best, whole;
  const bool f32out = (a.flags & HRT_MM_F32_OUT) != 0;
  const int64_t nk = cdiv(a.K, GBK);
  double best_us = 0.0;
  double whole_us = 0.0;
  static constexpr int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32};
  for (int t = 0; t < kGemmTiles; ++t) {
    const DmaForm f = dma_form(a, kTileShape[t].bm, kTileShape[t].bn);
    if (!f.ok || (t == T128x192 && f.btr)) continue;
    if (t == T256x256 && (nk > 64 || nk < 8)) continue;  // its two-buffer ring waits a step for each copy: slower at 8192^3
    const int64_t tiles = cdiv(a.M, kTileShape[t].bm) * cdiv(a.N, kTileShape[t].bn) * a.batch;
    // a 64-wide tile of an operand contiguous along M or N whose rows start off 128-byte lines touches two lines for
    // each line's worth
    const bool lines = (f.atr && kTileShape[t].bm == 64 && a.a_sk % 64 != 0) || (f.btr && kTileShape[t].bn == 64 && a.b_sk % 64 != 0);
    const double slow = (lines ? kHalfLines : 1.0) * (f.exact ? 1.0 : kMasked);
    const bool slices_ok = t == T128x256 || t >= T128x128;  // tiles with an fp32-output form
    if (f32out && !slices_ok) continue;
    for (int s : kSplits) {
      // slices of at least 4 steps, and none that start a third round of tiles
      if (s > 1 && (!may_split || !slices_ok || a.batch != 1 || nk < 4 * s || tiles * s > 2 * kTileCost[t].slots)) break;
      const uint32_t per = (uint32_t)(nk + s - 1) / s, n = ((uint32_t)nk + per - 1) / per;
      double us = tile_us(kTileCost[t], kTileShape[t], tiles * n, per * slow);
      if (n > 1) us += split_us(n, a.M, a.N);
      const GemmPlan p{t, n, n > 1 ? (int64_t)per * GBK : 0, us};
      if (n == 1 && (whole.tile < 0 || us < whole_us)) whole_us = us, whole = p;
      if (best.tile < 0 || us < best_us) best_us = us, best = p;
    }
  }
  return best.splits > 1 && whole.tile >= 0 && best_us > whole_us - kSplitGain ? whole : best;
}

// The shim asks for a workspace and then queues the same product, and a program's layers come back: the plans of the
// last few dozen products are kept per thread, by the values they depend on (an unsplit choice among splits is the choice
// without them too).  A search takes 0.35 to 0.55 us of the host's 4 per product, a kept plan 0.05.
GemmPlan plan_gemm(const hrt_mm_args& a, bool may_split) {
  struct Kept {
    std::array<int64_t, 17> key{};  // M = 0: no plan yet
    GemmPlan plan;
    bool split = false;
  };
  const std::array<int64_t, 17> key = {a.M, a.N, a.K, a.batch, a.a_sb, a.a_sm, a.a_sk, a.b_sb, a.b_sk, a.b_sn, a.c_sb, a.c_sm, a.c_sn,
                                       (int64_t)(a.a % 16), (int64_t)(a.b % 16), (int64_t)(a.c % 16), (int64_t)a.flags};
  uint64_t h = 0;
  for (const int64_t x : key) h = (h ^ (uint64_t)x) * 0x9e3779b97f4a7c15ull;
  thread_local std::array<Kept, 64> kept;
  Kept& e = kept[h >> 58];
  if (key != e.key || (may_split != e.split && !(e.split && e.plan.splits == 1)))
    e.plan = search_plan(a, may_split), e.key = key, e.split = may_split;
  return e.plan;
}

// Which loader an operand can use.  rows = M (A) or N (B); s_r / s_k its strides.
int pick_mode(uint64_t ptr, int64_t s_b, int64_t s_r, int64_t s_k, int64_t rows, int64_t K, int64_t batch) {
  const bool aligned = ptr % 16 == 0 && (batch == 1 || s_b % 8 == 0);
  if (aligned && s_k == 1 && K % 8 == 0 && (rows == 1 || s_r % 8 == 0)) return KVEC;
  if (aligned && s_r == 1 && rows % 8 == 0 && (K == 1 || s_k % 8 == 0)) return MNVEC;
  return GATHER;
}

template <typename T, int BM, int BN, int WM, int WN, int AM, int BMd>
void queue(const hrt_mm_args& a, hipStream_t s) {
  const int64_t tm = cdiv(a.M, BM), tn = cdiv(a.N, BN);
  hipLaunchKernelGGL((mm_mfma<T, BM, BN, WM, WN, AM, BMd>), dim3((uint32_t)(tm * tn * a.batch)), dim3(256), 0, s, a, tm, tn);
}

template <typename T>
void dispatch_modes(const hrt_mm_args& a, int am, int bm, hipStream_t s) {
  switch (am * 3 + bm) {
    case KVEC * 3 + KVEC: queue<T, 64, 64, 2, 2, KVEC, KVEC>(a, s); break;
    case KVEC * 3 + MNVEC: queue<T, 64, 64, 2, 2, KVEC, MNVEC>(a, s); break;
    case KVEC * 3 + GATHER: queue<T, 64, 64, 2, 2, KVEC, GATHER>(a, s); break;
    case MNVEC * 3 + KVEC: queue<T, 64, 64, 2, 2, MNVEC, KVEC>(a, s); break;
    case MNVEC * 3 + MNVEC: queue<T, 64, 64, 2, 2, MNVEC, MNVEC>(a, s); break;
    case MNVEC * 3 + GATHER: queue<T, 64, 64, 2, 2, MNVEC, GATHER>(a, s); break;
    case GATHER * 3 + KVEC: queue<T, 64, 64, 2, 2, GATHER, KVEC>(a, s); break;
    case GATHER * 3 + MNVEC: queue<T, 64, 64, 2, 2, GATHER, MNVEC>(a, s); break;
    default: queue<T, 64, 64, 2, 2, GATHER, GATHER>(a, s); break;
  }
}

template <typename T>
bool launch_mm_mfma(const void* pp, const uint32_t*, hrt::LaunchCtx& ctx) {
  const auto& a = *static_cast<const hrt_mm_args*>(pp);
  if (!mm_check_operands(a, 2, ctx)) return false;
  if (a.flags & ~HRT_MM_F32_OUT) return ctx.fail("unknown GEMM flags");
  const bool f32out = (a.flags & HRT_MM_F32_OUT) != 0;
  const int am = pick_mode(a.a, a.a_sb, a.a_sm, a.a_sk, a.M, a.K, a.batch);
  const int bm = pick_mode(a.b, a.b_sb, a.b_sn, a.b_sk, a.N, a.K, a.batch);
  const int64_t small = cdiv(a.M, 64) * cdiv(a.N, 64) * a.batch;
  if (small > 0x7fffffffLL) return ctx.fail("GEMM grid too large");
  // a short reduction (K <= 32, a low-rank adapter's up-projection): bound by the output, not the matrix cores
  if (!f32out && a.K <= 32 && skinny::queue_expand<T>(a, ctx.stream)) return hrt::launch_ok(hipGetLastError(), ctx, "mm_expand");
  // a narrow output (M or N <= 16, a low-rank adapter's down-projection and factor gradients, also the
  // fp32 slices of such a product split along K)
  if ((a.M <= 16 || a.N <= 16) && skinny::queue_narrow<T>(a, ctx.stream))
    return hrt::launch_ok(hipGetLastError(), ctx, "mm_narrow");
  // aligned operands: copied global -> LDS directly, on the tile the cost model finds cheapest
  const GemmPlan plan = plan_gemm(a, false);
  if (plan.tile >= 0 && dma_queue<T>(a, (GemmTile)plan.tile, 0, ctx.stream))
    return hrt::launch_ok(hipGetLastError(), ctx, "mm_dma");
  dispatch_modes<T>(a, am, bm, ctx.stream);
  return hrt::launch_ok(hipGetLastError(), ctx, "mm_mfma");
}

template <typename T>
bool launch_mm_reduce(const void* pp, const uint32_t*, hrt::LaunchCtx& ctx);

// Splits of the products that launch_mm_mfma gives to kernels of their own (short K, narrow output) are the
// caller's; "mm_splitk" leaves those whole.
bool own_kernel(const hrt_mm_args& a) { return a.K <= 32 || a.M <= 16 || a.N <= 16; }

template <typename T>
bool launch_mm_splitk(const void* pp, const uint32_t* grid, hrt::LaunchCtx& ctx) {
  const auto& s = *static_cast<const hrt_mm_splitk_args*>(pp);
  const hrt_mm_args& a = s.mm;
  if (a.flags != 0) return ctx.fail("mm_splitk takes no flags");
  if (!mm_check_operands(a, 2, ctx)) return false;
  const GemmPlan plan = own_kernel(a) ? GemmPlan{} : plan_gemm(a, true);
  if (plan.tile < 0 || plan.splits <= 1) return launch_mm_mfma<T>(&a, grid, ctx);
  if (s.ws_floats < plan.splits * a.M * a.N) return ctx.fail("workspace smaller than hrt_mm_workspace says");
  if (!ctx.check(s.ws, (uint64_t)s.ws_floats * 4, "ws")) return false;
  hrt_mm_args part = a;
  part.c = s.ws, part.batch = plan.splits, part.c_sb = a.M * a.N, part.c_sm = a.N, part.c_sn = 1;
  part.a_sb = part.b_sb = 0, part.alpha = 1.f, part.has_bias = 0, part.flags = HRT_MM_F32_OUT;
  if (!dma_queue<T>(part, (GemmTile)plan.tile, plan.kslice, ctx.stream)) return ctx.fail("no split-K kernel");
  if (!hrt::launch_ok(hipGetLastError(), ctx, "mm_splitk")) return false;
  hrt_mm_reduce_args r{};
  r.ws = s.ws, r.c = a.c, r.bias = a.bias, r.M = a.M, r.N = a.N, r.splits = plan.splits;
  r.c_sm = a.c_sm, r.c_sn = a.c_sn, r.bias_sm = a.bias_sm, r.bias_sn = a.bias_sn;
  r.alpha = a.alpha, r.beta = a.beta, r.has_bias = a.has_bias;
  return launch_mm_reduce<T>(&r, nullptr, ctx);
}

template <typename T, int BM, int BN, int AM>
void queue_dq8(const hrt_mm_dq8_args& a, hipStream_t s) {
  const int64_t tm = cdiv(a.M, BM), tn = cdiv(a.N, BN);
  hipLaunchKernelGGL((mm_dq8_mfma<T, BM, BN, 2, 2, AM>), dim3((uint32_t)(tm * tn)), dim3(256), 0, s, a, tm, tn);
}

// The same choice for the fused int8 linear (tile costs, fitted to 237 products, include the conversion of the int8 tile:
// M = 512 at 8192 x 2048 weights 31 us on 128 x 128 tiles, 41 on 256 x 128, 50 on 64 x 64; M = 16 on 64 x 64 12 us in four
// slices, 19 unsplit).  A split keeps its partial products in the optional workspace, which a caller may size for the
// dequantized weights: N K 16-bit elements hold them while 2 splits M <= K.
GemmPlan plan_dq8(const hrt_mm_dq8_args& d, bool may_split) {
  static constexpr struct {
    GemmTile t;
    TileCost c;
  } kTiles[] = {{T256x128, {256, 2.256, {0.7299, 1.526}}}, {T128x128, {256, 0.8656, {0.8287, 1.019}}}, {T64x64, {768, 0.01143, {0.6201, 0.6693, 0.914, 1.166}}}};
  GemmPlan best;
  if (d.K % GBK || d.q % 16 || d.scale % 2) return best;
  const hrt_mm_args a = dq8_as_mm(d);
  const int64_t nk = d.K / GBK;
  double best_us = 0.0;
  for (const auto& k : kTiles) {
    const DmaForm f = dma_form(a, kTileShape[k.t].bm, kTileShape[k.t].bn);
    if (!f.ok || f.btr) continue;
    const int64_t tiles = cdiv(a.M, kTileShape[k.t].bm) * cdiv(a.N, kTileShape[k.t].bn);
    for (int s : {1, 2, 3, 4, 6, 8}) {
      if (s > 1 && (!may_split || k.t != T64x64 || nk < 4 * s || 2 * s * d.M > d.K)) break;
      const int64_t per = cdiv(nk, s), n = cdiv(nk, per);
      double us = tile_us(k.c, kTileShape[k.t], tiles * n, per);
      if (n > 1) us += 3.697 + split_us(n, a.M, a.N);
      if (best.tile < 0 || us < best_us) best_us = us, best = GemmPlan{k.t, n, n > 1 ? per * GBK : 0, us};
    }
  }
  return best;
}

void fill_plan(const hrt_mm_args& a, const GemmPlan& p, hrt_mm_plan* out) {
  if (p.tile < 0) return;
  const TileShape t = kTileShape[p.tile];
  *out = hrt_mm_plan{HRT_MM_DIRECT, t.bm, t.bn, dma_form(a, t.bm, t.bn).exact ? 1 : 0, p.splits};
}

// The product of a dequantize-first call: its B is the workspace (16-byte aligned).
hrt_mm_args dq8_weights_as_mm(const hrt_mm_dq8_args& d) {
  hrt_mm_args m = dq8_as_mm(d);
  m.b = d.ws;
  return m;
}

// Smallest M at which the fused int8 linear may dequantize into the caller's workspace first: the fused kernel
// converts every weight once per 256-row block of x, which costs more than one standalone dequant pass
// beyond a few blocks (M = 4096: 222 us fused vs 153 us dequant + GEMM for 8192 x 2048 weights).
constexpr int64_t kDq8WsMinM = 2048;
// The plan of the product on dequantized weights (ws: their address, 0 = any aligned one) where that is estimated
// faster, with the pass that dequantizes them, than the fused kernel; else tile = -1.  Short reductions stay fused: 2048 x
// 1024 x 320 7.1 us against 8.8, 3120 x 1024 x 320 8.1 / 10.0, 2048 x 2048 x 2048 33.1 / 30.4.
GemmPlan plan_dequant(const hrt_mm_dq8_args& d) {
  if (d.M < kDq8WsMinM || d.K % GBK != 0) return GemmPlan{};
  const GemmPlan whole = plan_gemm(dq8_weights_as_mm(d), false), fused = plan_dq8(d, false);
  return whole.tile >= 0 && (fused.tile < 0 || whole.us + 2.0 < fused.us) ? whole : GemmPlan{};
}

template <typename T>
bool launch_mm_dq8(const void* pp, const uint32_t*, hrt::LaunchCtx& ctx) {
  const auto& a = *static_cast<const hrt_mm_dq8_args*>(pp);
  if (a.M <= 0 || a.N <= 0 || a.K <= 0) return ctx.fail("empty GEMM");
  if (a.nblocks != (a.K + 63) / 64) return ctx.fail("nblocks must equal ceil(K / 64)");
  if (a.x_sm < 0 || a.x_sk < 0) return ctx.fail("negative stride");
  if (a.K % 8 != 0 || a.q % 8 != 0) return ctx.fail("the fused int8 linear needs K % 8 == 0 and an 8-byte aligned q");
  const int64_t xs[2] = {a.M, a.K}, xt[2] = {a.x_sm, a.x_sk};
  if (!ctx.check(a.x, hrt::span_bytes(2, xs, xt, 2), "x") || !ctx.check(a.q, (uint64_t)(a.N * a.K), "q") ||
      !ctx.check(a.scale, (uint64_t)(a.N * a.nblocks) * 2, "scale") || !ctx.check(a.y, (uint64_t)(a.M * a.N) * 2, "y") ||
      (a.has_bias && !ctx.check(a.bias, (uint64_t)a.N * 2, "bias")))
    return false;
  // many rows and a workspace: dequantize once (the dq8 kernel), then the GEMM on the bf16 / f16 weights, where faster
  const bool ws_ok = a.ws && a.ws % 16 == 0;
  if (const GemmPlan plan = ws_ok ? plan_dequant(a) : GemmPlan{}; plan.tile >= 0) {
    const hrt_mm_args m = dq8_weights_as_mm(a);
    if (!ctx.check(a.ws, (uint64_t)(a.N * a.K) * 2, "ws")) return false;
    hrt_dq8_args d{};
    d.q = a.q, d.scale = a.scale, d.out = a.ws, d.rows = a.N, d.cols = a.K, d.nblocks = a.nblocks;
    const char* dq = std::is_same<T, BF16>::value ? "dq8_bf16" : "dq8_f16";
    for (auto& e : hrt::kernel_table())
      if (!strcmp(e.name, dq)) {
        if (!e.launch(&d, nullptr, ctx)) return false;
        if (dma_queue<T>(m, (GemmTile)plan.tile, 0, ctx.stream)) return hrt::launch_ok(hipGetLastError(), ctx, "mm_dq8_ws");
      }
    return ctx.fail("mm_dq8: workspace path unavailable");
  }
  // K in whole steps: dequant fused into the direct-to-LDS GEMM, K split over the workspace where the grid is small
  const GemmPlan plan = plan_dq8(a, ws_ok);
  if (plan.tile >= 0 && plan.splits > 1) {
    if (!ctx.check(a.ws, (uint64_t)(plan.splits * a.M * a.N) * 4, "ws")) return false;
    if (dma_queue_dq8<T>(a, (GemmTile)plan.tile, a.ws, plan.splits, plan.kslice, ctx.stream)) {
      if (!hrt::launch_ok(hipGetLastError(), ctx, "mm_dq8_splitk")) return false;
      hrt_mm_reduce_args r{};
      r.ws = a.ws, r.c = a.y, r.bias = a.bias, r.M = a.M, r.N = a.N, r.splits = plan.splits;
      r.c_sm = a.N, r.c_sn = 1, r.bias_sn = 1, r.alpha = a.alpha, r.beta = a.beta, r.has_bias = a.has_bias;
      return launch_mm_reduce<T>(&r, nullptr, ctx);
    }
  }
  if (plan.tile >= 0 && plan.splits == 1 && dma_queue_dq8<T>(a, (GemmTile)plan.tile, 0, 1, 0, ctx.stream))
    return hrt::launch_ok(hipGetLastError(), ctx, "mm_dq8_dma");
  const int am = pick_mode(a.x, 0, a.x_sm, a.x_sk, a.M, a.K, 1);
  const int64_t big = cdiv(a.M, 128) * cdiv(a.N, 256);
  if (big >= 240) {
    if (am == KVEC) queue_dq8<T, 128, 256, KVEC>(a, ctx.stream);
    else if (am == MNVEC) queue_dq8<T, 128, 256, MNVEC>(a, ctx.stream);
    else queue_dq8<T, 64, 64, GATHER>(a, ctx.stream);
  } else {
    if (am == KVEC) queue_dq8<T, 64, 64, KVEC>(a, ctx.stream);
    else if (am == MNVEC) queue_dq8<T, 64, 64, MNVEC>(a, ctx.stream);
    else queue_dq8<T, 64, 64, GATHER>(a, ctx.stream);
  }
  return hrt::launch_ok(hipGetLastError(), ctx, "mm_dq8");
}

// ---- split-K reduction: c = round(alpha * sum_s ws[s] + beta * bias), splits summed in order ---------------
// Four consecutive outputs (of the flattened [M, N]) per thread, read as 16-byte pieces of each split when
// M N is a multiple of 4; the loads of up to 16 splits are in flight together (the outputs are small: one
// memory round trip per 16 splits bounds the kernel), then summed in split order.
template <typename T>
__global__ __launch_bounds__(256) void mm_reduce(hrt_mm_reduce_args p) {
  const int64_t total = p.M * p.N;
  const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i0 >= total) return;
  const HK_G float* w = gcptr<float>(p.ws);
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (total % 4 == 0) {
    for (int64_t k = 0; k < p.splits; k += 16) {
      f32x4 v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u)  // splits past the end re-read the last one (in range) and are not added
        v[u] = *reinterpret_cast<const HK_G f32x4*>(w + (k + u < p.splits ? k + u : p.splits - 1) * total + i0);
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (k + u < p.splits) s += v[u];
    }
  } else {
    for (int64_t k = 0; k < p.splits; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e < total) s[e] += w[k * total + i0 + e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t i = i0 + e;
    if (i >= total) break;
    const int64_t m = i / p.N, n = i % p.N;
    float o = p.alpha * s[e];
    if (p.has_bias) o += p.beta * T::to_f32(gcptr<uint16_t>(p.bias)[m * p.bias_sm + n * p.bias_sn]);
    gptr<uint16_t>(p.c)[m * p.c_sm + n * p.c_sn] = T::from_f32(o);
  }
}

// Vector form of mm_reduce for the common layout (N % 8 == 0, C rows contiguous and 16-byte aligned, the bias
// absent or with contiguous rows): a thread takes 8 consecutive outputs of one row (one division for the
// row), loads exactly the S slices' two 16-byte pieces (four slices' loads in flight at a time), adds them in
// slice order 0, 1, ... exactly as mm_reduce does (bit-identical results) and writes one 16-byte store.
template <typename T>
__global__ __launch_bounds__(256) void mm_reduce_vec(hrt_mm_reduce_args p, int64_t nvec) {
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= nvec) return;
  const int64_t i0 = v * 8, total = p.M * p.N;
  const int64_t m = i0 / p.N, n = i0 - m * p.N;
  const HK_G f32x4* w = gcptr<f32x4>(p.ws) + i0 / 4;
  const int64_t st = total / 4;  // 16-byte pieces per slice
  f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
  int64_t k = 0;
  for (; k + 4 <= p.splits; k += 4) {
    f32x4 a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = w[(k + u) * st], b[u] = w[(k + u) * st + 1];
#pragma unroll
    for (int u = 0; u < 4; ++u) s0 += a[u], s1 += b[u];
  }
  for (; k < p.splits; ++k) s0 += w[k * st], s1 += w[k * st + 1];
  float o[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = p.alpha * s0[e], o[4 + e] = p.alpha * s1[e];
  if (p.has_bias) {
    const u32x4 bb = *reinterpret_cast<const HK_G u32x4*>(gcptr<uint16_t>(p.bias) + m * p.bias_sm + n);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[2 * e] += p.beta * T::to_f32((uint16_t)(bb[e] & 0xffffu));
      o[2 * e + 1] += p.beta * T::to_f32((uint16_t)(bb[e] >> 16));
    }
  }
  u32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (uint32_t)T::from_f32(o[2 * e]) | ((uint32_t)T::from_f32(o[2 * e + 1]) << 16);
  *reinterpret_cast<HK_G u32x4*>(gptr<uint16_t>(p.c) + m * p.c_sm + n) = r;
}

template <typename T>
bool launch_mm_reduce(const void* pp, const uint32_t*, hrt::LaunchCtx& ctx) {
  const auto& a = *static_cast<const hrt_mm_reduce_args*>(pp);
  if (a.M <= 0 || a.N <= 0 || a.splits <= 0) return ctx.fail("empty split-K reduction");
  if (a.c_sm < 0 || a.c_sn < 0 || a.bias_sm < 0 || a.bias_sn < 0) return ctx.fail("negative stride");
  const int64_t total = a.M * a.N;
  if (cdiv(total, 1024) > 0x7fffffffLL) return ctx.fail("reduction grid too large");
  const int64_t sw[3] = {a.splits, a.M, a.N}, tw[3] = {a.M * a.N, a.N, 1};
  const int64_t sc[2] = {a.M, a.N}, tc[2] = {a.c_sm, a.c_sn}, tb[2] = {a.bias_sm, a.bias_sn};
  if (!ctx.check(a.ws, hrt::span_bytes(3, sw, tw, 4), "ws") || !ctx.check(a.c, hrt::span_bytes(2, sc, tc, 2), "c") ||
      (a.has_bias && !ctx.check(a.bias, hrt::span_bytes(2, sc, tb, 2), "bias")))
    return false;
  const bool vec = a.N % 8 == 0 && a.c_sn == 1 && a.c % 16 == 0 && a.c_sm % 8 == 0 && a.ws % 16 == 0 &&
                   (!a.has_bias || (a.bias_sn == 1 && a.bias % 16 == 0 && a.bias_sm % 8 == 0));
  if (vec) {
    const int64_t nvec = total / 8;
    hipLaunchKernelGGL(mm_reduce_vec<T>, dim3((uint32_t)cdiv(nvec, 256)), dim3(256), 0, ctx.stream, a, nvec);
  } else {
    hipLaunchKernelGGL(mm_reduce<T>, dim3((uint32_t)cdiv(total, 1024)), dim3(256), 0, ctx.stream, a);
  }
  return hrt::launch_ok(hipGetLastError(), ctx, "mm_reduce");
}

HRT_REGISTER("mm_mfma_bf16", hrt_mm_args, launch_mm_mfma<BF16>);
HRT_REGISTER("mm_reduce_bf16", hrt_mm_reduce_args, launch_mm_reduce<BF16>);
HRT_REGISTER("mm_reduce_f16", hrt_mm_reduce_args, launch_mm_reduce<F16>);
HRT_REGISTER("mm_mfma_f16", hrt_mm_args, launch_mm_mfma<F16>);
HRT_REGISTER("mm_splitk_bf16", hrt_mm_splitk_args, launch_mm_splitk<BF16>);
HRT_REGISTER("mm_splitk_f16", hrt_mm_splitk_args, launch_mm_splitk<F16>);
HRT_REGISTER("mm_dq8_bf16", hrt_mm_dq8_args, launch_mm_dq8<BF16>);
HRT_REGISTER("mm_dq8_f16", hrt_mm_dq8_args, launch_mm_dq8<F16>);

}  // namespace

DmaForm dma_form(const hrt_mm_args& a, int bm, int bn) {
  DmaForm f{};
  const auto al = [](uint64_t x) { return x % 16 == 0; };
  const int64_t lim = (int64_t)1 << 31;
  if (!al(a.a) || !al(a.b) || a.c_sn != 1 || (a.batch > 1 && (a.a_sb % 8 || a.b_sb % 8)) || a.K >= lim) return f;
  if (a.a_sk == 1 && a.a_sm % 8 == 0 && a.K % 8 == 0) f.atr = false;
  else if (a.a_sm == 1 && a.a_sk % 8 == 0 && a.M % 8 == 0) f.atr = true;
  else return f;
  if (a.b_sk == 1 && a.b_sn % 8 == 0 && a.K % 8 == 0) f.btr = false;
  else if (a.b_sn == 1 && a.b_sk % 8 == 0 && a.N % 8 == 0) f.btr = true;
  else return f;
  // row offsets inside a tile, workgroup numbers
  if ((f.atr ? a.a_sk : a.a_sm) * 2 * ((f.atr ? GBK : bm) + 1) >= lim || (f.btr ? a.b_sk : a.b_sn) * 2 * ((f.btr ? GBK : bn) + 1) >= lim ||
      cdiv(a.M, bm) * cdiv(a.N, bn) * a.batch >= lim)
    return f;
  f.ok = true;
  f.exact = a.M % bm == 0 && a.N % bn == 0 && a.K % GBK == 0 && al(a.c) && a.c_sm % 8 == 0 && (a.batch == 1 || a.c_sb % 8 == 0);
  return f;
}

hrt_mm_args dq8_as_mm(const hrt_mm_dq8_args& d) {
  hrt_mm_args a{};
  a.a = d.x, a.b = d.q, a.c = d.y, a.bias = d.bias;
  a.M = d.M, a.N = d.N, a.K = d.K, a.batch = 1;
  a.a_sm = d.x_sm, a.a_sk = d.x_sk, a.b_sk = 1, a.b_sn = d.K, a.c_sm = d.N, a.c_sn = 1, a.bias_sn = 1;
  a.alpha = d.alpha, a.beta = d.beta, a.has_bias = d.has_bias;
  return a;
}

}  // namespace hk

extern "C" int64_t hrt_mm_workspace(const hrt_mm_args* a, int32_t dtype) {
  if (a == nullptr || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->batch != 1 || a->flags != 0) return 0;
  if (dtype == HRT_F32) return hk::mm_f32_workspace(*a);
  if ((dtype != HRT_BF16 && dtype != HRT_F16) || hk::own_kernel(*a)) return 0;
  const hk::GemmPlan p = hk::plan_gemm(*a, true);
  return p.tile < 0 ? -1 : p.splits > 1 ? p.splits * a->M * a->N : 0;
}

extern "C" int64_t hrt_mm_dq8_workspace(const hrt_mm_dq8_args* a) {
  if (a == nullptr || a->M <= 0 || a->N <= 0 || a->K <= 0) return 0;
  if (hk::plan_dequant(*a).tile >= 0) return a->N * a->K;
  // not N K: 256 MiB and more is a reservation and a wait for the GPU on every call (16 x 16384 x 8192 340 us, 41 so)
  const int64_t splits = hk::plan_dq8(*a, true).splits;
  return splits > 1 ? 2 * splits * a->M * a->N : 0;  // fp32 partial products in 16-bit elements
}

// Both plans: 0, or -1 for a product that the launches refuse.
extern "C" int hrt_mm_plan_of(const hrt_mm_args* a, int32_t dtype, int32_t may_split, hrt_mm_plan* out) {
  if (a == nullptr || out == nullptr || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->batch <= 0) return -1;
  *out = hrt_mm_plan{HRT_MM_GENERAL, 64, 64, 0, 1};
  if (dtype == HRT_F32) {
    hk::mm_f32_plan(*a, may_split != 0, out);
    return 0;
  }
  if (dtype != HRT_BF16 && dtype != HRT_F16) return -1;
  if (hk::own_kernel(*a)) {
    out->kernel = HRT_MM_NARROW;
    return 0;
  }
  hk::fill_plan(*a, hk::plan_gemm(*a, may_split != 0), out);
  return 0;
}

extern "C" int hrt_mm_dq8_plan_of(const hrt_mm_dq8_args* a, int32_t with_ws, hrt_mm_plan* out) {
  if (a == nullptr || out == nullptr || a->M <= 0 || a->N <= 0 || a->K <= 0) return -1;
  *out = hrt_mm_plan{HRT_MM_GENERAL, 64, 64, 0, 1};
  if (const hk::GemmPlan p = with_ws != 0 ? hk::plan_dequant(*a) : hk::GemmPlan{}; p.tile >= 0) {
    hk::fill_plan(hk::dq8_weights_as_mm(*a), p, out);
    out->kernel = HRT_MM_DEQUANT;
    return 0;
  }
  hk::fill_plan(hk::dq8_as_mm(*a), hk::plan_dq8(*a, with_ws != 0), out);
  return 0;
}
