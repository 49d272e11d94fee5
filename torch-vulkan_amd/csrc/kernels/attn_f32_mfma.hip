// fp32 fused attention on the fp32 matrix cores: "attn_{fwd,dq,dkdv}_fma_f32" wherever a tile's offsets fit 31 bits
// (attn_f32.hip keeps the rest, and bf16 / f16 with the matrix cores switched off).  Logits, P and dS stay fp32 and
// every product is v_mfma_f32_32x32x2_f32 (no rounding of its inputs), as the scalar kernels of
// vkrt/shaders/attn.comp.in:256-395, which this file's predecessor followed one row per lane.
//
// Bound: the fp32 matrix rate (64 cycles per MFMA and SIMD): a 32 x 32 tile of the forward is D MFMAs, of dQ 3 D / 2, of
// dK/dV 2 D, against some 200-300 vector instructions for its softmax.
//   * A workgroup's four wavefronts share 32 G stationary rows (queries; keys for dK/dV), whose operand fragments stay
//     in registers, and split each stage of the streamed rows into KH = 4 / G tiles of 32: G = 1 for D <= 64 (the
//     finest grid: B H S / 32 workgroups over 256 CUs, two of them on a CU so that one's softmax and copies run
//     under the other's MFMAs), G = 2 above, where a stage fills LDS twice over (one workgroup per CU, copies of the
//     next stage under the MFMAs of this one).
//   * The first product has the stationary row in the lane: element 4 j + r of a lane's 16 accumulators is streamed row
//     8 j + 4 h + r (h = lane / 32).  The second product takes its k pairs as rows 8 j + r (h = 0) and 8 j + 4 + r
//     (h = 1), so P and dS are its B operand as they stand: no lane exchange, no LDS round trip.
//   * Row reads are 16 bytes per lane (k pairs d, d + 4), column reads 4 bytes per lane of 32 consecutive d; chunks are
//     XOR-swizzled by row so that both are conflict-free.  Rows past the end and columns past D are zeros by the
//     buffer's range check.
// B1 H16 S2080 D64, forward and backward: 8680 us in the one-row-per-lane kernels (2449 + 2449 + 3759), 915 here (68
// TFLOP/s of the 7 products a step counts; dQ and dK/dV recompute two more), forward 238; S2048 D128 1404 (86).  Errors
// against float64 1.2e-6 before, 7.6e-7 now.
#include <cmath>
#include <type_traits>

#include "../hrt/registry.h"
#include "attn_common.h"

namespace hk {

bool attn_check(const hrt_attn_args& a, bool fwd, bool dkdv, bool dq, uint64_t elem, hrt::LaunchCtx& ctx);
bool attn_f32_mfma(const hrt_attn_args& a, int which, hipStream_t s);

namespace {

// XOR on the 16-byte chunk index: 16 consecutive rows at one chunk fall in distinct chunks of a 256-byte bank line
// (rows of 8 or 24 chunks: two rows share a line), and a run of 8 aligned chunks stays such a run.
template <int NCH>
__device__ __forceinline__ int f32_swz(int row) {
  return NCH % 16 == 0 ? row & 15 : (row >> 1) & 7;
}
template <int NCH>
__device__ __forceinline__ int f32_off(int row, int c) {
  return row * (NCH * 16) + ((c ^ f32_swz<NCH>(row)) << 4);
}

// A ROWS x DP tile copied by the workgroup's four wavefronts, 16 bytes (W16: 16-byte aligned rows, D % 4 == 0) or 4
// bytes per lane.
template <int ROWS, int DP, bool W16>
struct F32Tile {
  static constexpr int NCH = DP / 4, BYTES = ROWS * DP * 4, CB = W16 ? 1024 : 256, IPW = BYTES / CB / 4;
  // rows [0, valid) from `base` on; a copy's lane offset is recomputed (cheap beside the MFMAs), not held
  __device__ __forceinline__ static void copy(const HK_G uint8_t* base, uint32_t ss, int D, int valid, HK_L uint8_t* tile, int wave,
                                              int lane) {
    const __amdgpu_buffer_rsrc_t rs = edge_rsrc(base);
    asm volatile("" : "+v"(lane));  // keeps the lane offsets out of registers between stages
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int j = wave * IPW + i;
      if constexpr (W16) {
        const int ch = j * 64 + lane, row = ch / NCH, c = (ch % NCH) ^ f32_swz<NCH>(row);
        edge_copy(rs, tile, j, row < valid && c * 4 < D ? (uint32_t)row * ss + (uint32_t)(c << 4) : kNoRow);
      } else {
        const int d = j * 64 + lane, row = d / DP, e = (((d % DP) >> 2) ^ f32_swz<NCH>(row)) * 4 + (d & 3);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, tile + j * 256, 4, (int)(row < valid && e < D ? (uint32_t)row * ss + (uint32_t)e * 4 : kNoRow),
                                                 0, 0, 0);
      }
    }
  }
};

// Operand fragments of one stationary row per lane: group g holds d = 8 g + 4 h .. + 3.
template <int DP, bool W16>
__device__ __forceinline__ void load_frags(f32x4 (&f)[DP / 8], const HK_G float* row, bool ok, int D, int h) {
#pragma unroll
  for (int g = 0; g < DP / 8; ++g) {
    const int d = 8 * g + 4 * h;
    f[g] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (ok) {
      if constexpr (W16) {
        if (d < D) f[g] = *reinterpret_cast<const HK_G f32x4*>(row + d);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < D) f[g][e] = row[d + e];
      }
    }
  }
}

__device__ __forceinline__ f32x16 mfma2(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

// Rows r0 .. r0 + 31 of the tile (A) times the stationary fragments (B), over d.  Chunk 2 g + h of row l32 sits at
// (2 g + h) ^ swz: the lane's base address XOR a constant.
template <int DP>
__device__ __forceinline__ f32x16 rows_times(const HK_L uint8_t* T, int r0, const f32x4 (&f)[DP / 8], int l32, int h) {
  f32x16 s = zero16();
  const int row = (r0 + l32) * DP * 4, x = (h ^ f32_swz<DP / 4>(l32)) << 4;
#pragma unroll
  for (int g = 0; g < DP / 8; ++g) {
    const f32x4 a = *reinterpret_cast<const HK_L f32x4*>(T + row + (x ^ (g << 5)));
#pragma unroll
    for (int e = 0; e < 4; ++e) s = mfma2(a[e], f[g][e], s);
  }
  return s;
}
// acc[n] + (columns 32 n .. + 31 of the tile's rows r0 .. r0 + 31)^T times p: d x stationary row.  The swizzle of row
// 8 j + 4 h + r splits into a lane part (four bases) and constants.
template <int DP>
__device__ __forceinline__ void cols_times(f32x16 (&acc)[DP / 32], const HK_L uint8_t* T, int r0, const f32x16& p, int l32, int h) {
  constexpr bool WIDE = (DP / 4) % 16 == 0;
  const HK_L uint8_t* base[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {  // WIDE: k = r; else k = 2 (j & 1) + r / 2
    const int x = WIDE ? 4 * h + k : 4 * (k >> 1) + 2 * h + (k & 1);
    base[k] = T + (r0 + 4 * h) * DP * 4 + (((l32 >> 2) ^ x) << 4) + (l32 & 3) * 4;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int n = 0; n < DP / 32; ++n) {
        const int blk = WIDE ? n ^ (j & 1) : n;
        const float a = *reinterpret_cast<const HK_L float*>(base[WIDE ? r : 2 * (j & 1) + (r >> 1)] + (8 * j + r) * DP * 4 + blk * 128);
        acc[n] = mfma2(a, p[4 * j + r], acc[n]);
      }
}

// d block n of one stationary row per lane: elements 4 j + r are d = 32 n + 8 j + 4 h + r
template <bool W16>
__device__ __forceinline__ void store_block(HK_G float* row, const f32x16& v, float mul, int n, int D, int h) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int d = 32 * n + 8 * j + 4 * h;
    if constexpr (W16) {
      if (d < D) *reinterpret_cast<HK_G f32x4*>(row + d) = f32x4{v[4 * j] * mul, v[4 * j + 1] * mul, v[4 * j + 2] * mul, v[4 * j + 3] * mul};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (d + r < D) row[d + r] = v[4 * j + r] * mul;
    }
  }
}

// WHICH: 0 forward, 1 dK/dV, 2 dQ
template <int WHICH, int DP, bool W16>
struct Shape {
  static constexpr int G = DP <= 64 ? 1 : 2, KH = 4 / G, ST = 32 * KH, NBUF = DP <= 64 ? 1 : 2, DCH = DP / 32;
  static constexpr int NACC = WHICH == 1 ? 2 * DCH : DCH;
  using Tile = F32Tile<ST, DP, W16>;
  static constexpr int XCH = G * (KH - 1) * 64 * (NACC * 16 + (WHICH == 0 ? 2 : 0)) * 4;  // bytes of the merge
  static constexpr int POOL = 2 * NBUF * Tile::BYTES > XCH ? 2 * NBUF * Tile::BYTES : XCH;
};

template <int WHICH, int DP, bool W16>
__global__ __launch_bounds__(256, DP <= 64 ? 2 : 1) void attn_f32_k(hrt_attn_args p, int nblk) {
  using S = Shape<WHICH, DP, W16>;
  constexpr int G = S::G, KH = S::KH, ST = S::ST, DCH = S::DCH, TB = S::Tile::BYTES;
  __shared__ __attribute__((aligned(1024))) uint8_t pool[S::POOL];
  __shared__ float stat[2][2][ST];  // dK/dV: lse (log2 units) and delta of the streamed rows, per buffer
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave % G, kh = wave / G, l32 = lane & 31, h = lane >> 5;
  uint32_t bh32, blk32;
  xcd_map32(blockIdx.x, (uint32_t)nblk * p.B * p.H, nblk, bh32, blk32);
  const int64_t bh = bh32, b = bh32 / (uint32_t)p.H, hh = bh32 % (uint32_t)p.H;
  const int D = p.D, Sq = p.Sq, Sk = p.Sk;
  const int own_n = WHICH == 1 ? Sk : Sq, str_n = WHICH == 1 ? Sq : Sk;
  const int64_t own = (int64_t)blk32 * (32 * G) + 32 * g + l32;  // this lane's stationary row
  const HK_G float* Q = gcptr<float>(p.q) + b * p.q_sb + hh * p.q_sh;
  const HK_G float* K = gcptr<float>(p.k) + b * p.k_sb + hh * p.k_sh;
  const HK_G float* V = gcptr<float>(p.v) + b * p.v_sb + hh * p.v_sh;
  const HK_G float* dO = gcptr<float>(p.dout) + b * p.do_sb + hh * p.do_sh;
  // streamed tensors: K and V, or Q and dO
  const HK_G uint8_t* T0 = reinterpret_cast<const HK_G uint8_t*>(WHICH == 1 ? Q : K);
  const HK_G uint8_t* T1 = reinterpret_cast<const HK_G uint8_t*>(WHICH == 1 ? dO : V);
  const uint32_t s0 = (uint32_t)((WHICH == 1 ? p.q_ss : p.k_ss) * 4), s1 = (uint32_t)((WHICH == 1 ? p.do_ss : p.v_ss) * 4);
  const int nst = (str_n + ST - 1) / ST;
  const float sl2 = p.scale * kLog2e;

  auto copy = [&](int st) {
    HK_L uint8_t* const t = (HK_L uint8_t*)pool + (S::NBUF == 2 ? (st & 1) * 2 * TB : 0);
    const int valid = str_n - st * ST;
    S::Tile::copy(T0 + (int64_t)st * ST * s0, s0, D, valid, t, wave, lane);
    S::Tile::copy(T1 + (int64_t)st * ST * s1, s1, D, valid, t + TB, wave, lane);
    if constexpr (WHICH == 1) {
      if (threadIdx.x < ST) {  // rows past the end: P = exp2(-inf) = 0
        const int64_t q = (int64_t)st * ST + threadIdx.x;
        stat[st & 1][0][threadIdx.x] = q < Sq ? gcptr<float>(p.lse)[bh * Sq + q] * kLog2e : INFINITY;
        stat[st & 1][1][threadIdx.x] = q < Sq ? gcptr<float>(p.delta)[bh * Sq + q] : 0.f;
      }
    }
  };
  copy(0);
  f32x4 f0[DP / 8], f1[WHICH == 0 ? 1 : DP / 8];  // Q; Q, dO; K, V
  const bool own_ok = own < own_n;
  load_frags<DP, W16>(f0, WHICH == 1 ? K + own * p.k_ss : Q + own * p.q_ss, own_ok, D, h);
  if constexpr (WHICH != 0) load_frags<DP, W16>(f1, WHICH == 1 ? V + own * p.v_ss : dO + own * p.do_ss, own_ok, D, h);
  float lse2 = 0.f, dlt = 0.f;
  if constexpr (WHICH == 2) {
    lse2 = own_ok ? gcptr<float>(p.lse)[bh * Sq + own] * kLog2e : INFINITY;
    dlt = own_ok ? gcptr<float>(p.delta)[bh * Sq + own] : 0.f;
  }
  f32x16 acc[S::NACC > DCH ? 2 : 1][DCH];
#pragma unroll
  for (auto& a : acc)
#pragma unroll
    for (int n = 0; n < DCH; ++n) a[n] = zero16();
  float m = -INFINITY, l = 0.f;  // forward: running max in log2 units of the scaled logits, sum

  for (int st = 0; st < nst; ++st) {
    // stage st's copies are complete (every wavefront waits for its own, explicitly: the compiler puts no wait for
    // copies into LDS before __syncthreads() on the loop's back edge); the other buffer is free
    barrier_keep_vm_lds<0>();
    if (S::NBUF == 2 && st + 1 < nst) copy(st + 1);
    const HK_L uint8_t* const t0 = (const HK_L uint8_t*)pool + (S::NBUF == 2 ? (st & 1) * 2 * TB : 0);
    const HK_L uint8_t* const t1 = t0 + TB;
    const int r0 = 32 * kh, left = str_n - st * ST - r0;  // this wavefront's tile: rows r0 .. r0 + 31, `left` of them exist
    if (left > 0) {
      f32x16 s = rows_times<DP>(t0, r0, f0, l32, h);
      if constexpr (WHICH == 0) {
        if (left < 32) {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (8 * (e >> 2) + 4 * h + (e & 3) >= left) s[e] = -INFINITY;
        }
        float mx = fmaxf(s[0], s[1]);
#pragma unroll
        for (int e = 2; e < 16; ++e) mx = fmaxf(mx, s[e]);
        const float mn = fmaxf(m, halfswap_max(mx) * sl2);  // scale > 0: max commutes with the scaling
        if (__any(mn != m)) {
          const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
          l *= alpha;
#pragma unroll
          for (int n = 0; n < DCH; ++n)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[0][n][e] *= alpha;
          m = mn;
        }
        const float nm = m == -INFINITY ? 0.f : -m;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          s[e] = __builtin_amdgcn_exp2f(fmaf(s[e], sl2, nm));
          l += s[e];
        }
        cols_times<DP>(acc[0], t1, r0, s, l32, h);
      } else {
        f32x16 dp = rows_times<DP>(t1, r0, f1, l32, h);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f32x4 ls, de;
          if constexpr (WHICH == 1) {
            ls = *reinterpret_cast<const f32x4*>(&stat[st & 1][0][r0 + 8 * j + 4 * h]);
            de = *reinterpret_cast<const f32x4*>(&stat[st & 1][1][r0 + 8 * j + 4 * h]);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int e = 4 * j + r;
            float pv = __builtin_amdgcn_exp2f(fmaf(s[e], sl2, WHICH == 1 ? -ls[r] : -lse2));
            if (WHICH == 2 && left < 32 && 8 * j + 4 * h + r >= left) pv = 0.f;  // keys past the end
            dp[e] = pv * (dp[e] - (WHICH == 1 ? de[r] : dlt));
            s[e] = pv;
          }
        }
        if constexpr (WHICH == 1) {
          cols_times<DP>(acc[0], t0, r0, dp, l32, h);  // dK^T += Q^T dS
          cols_times<DP>(acc[S::NACC > DCH ? 1 : 0], t1, r0, s, l32, h);  // dV^T += dO^T P
        } else {
          cols_times<DP>(acc[0], t0, r0, dp, l32, h);  // dQ^T += K^T dS^T
        }
      }
    }
    if (S::NBUF == 1 && st + 1 < nst) {
      __syncthreads();  // every wavefront is done with the stage
      copy(st + 1);
    }
  }

  // merge the KH partial results of each stationary group, in stage-tile order, into the wavefront kh = 0
  __syncthreads();
  float* const x = reinterpret_cast<float*>(pool);
  constexpr int NV = S::NACC * 16;  // values per lane
  if (kh > 0) {
    float* const mine = x + (g * (KH - 1) + kh - 1) * 64 * (NV + (WHICH == 0 ? 2 : 0));
#pragma unroll
    for (int k = 0; k < S::NACC; ++k)
#pragma unroll
      for (int e = 0; e < 16; ++e) mine[(k * 16 + e) * 64 + lane] = acc[k / DCH][k % DCH][e];
    if (WHICH == 0) mine[NV * 64 + lane] = m, mine[(NV + 1) * 64 + lane] = l;
  }
  __syncthreads();
  if (kh > 0) return;
  const float* const parts = x + g * (KH - 1) * 64 * (NV + (WHICH == 0 ? 2 : 0));
  constexpr int PS = 64 * (NV + (WHICH == 0 ? 2 : 0));
  if constexpr (WHICH == 0) {
    float mt = m;
#pragma unroll
    for (int k = 0; k < KH - 1; ++k) mt = fmaxf(mt, parts[k * PS + NV * 64 + lane]);
    float w = m == -INFINITY ? 0.f : exp2f(m - mt);
    l *= w;
#pragma unroll
    for (int n = 0; n < DCH; ++n)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[0][n][e] *= w;
#pragma unroll
    for (int k = 0; k < KH - 1; ++k) {
      const float mk = parts[k * PS + NV * 64 + lane];
      w = mk == -INFINITY ? 0.f : exp2f(mk - mt);
      l += w * parts[k * PS + (NV + 1) * 64 + lane];
#pragma unroll
      for (int n = 0; n < DCH; ++n)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[0][n][e] = fmaf(w, parts[k * PS + (n * 16 + e) * 64 + lane], acc[0][n][e]);
    }
    const float lrow = halfswap_sum(l);
    if (!own_ok) return;
    const float inv = lrow > 0.f ? 1.f / lrow : 0.f;
    if (h == 0) gptr<float>(p.lse)[bh * Sq + own] = lrow > 0.f ? (mt + log2f(lrow)) * kLn2 : -INFINITY;
    const int64_t off = ((b * Sq + own) * p.H + hh) * D;
#pragma unroll
    for (int n = 0; n < DCH; ++n) {
      store_block<W16>(gptr<float>(p.o) + off, acc[0][n], inv, n, D, h);
      if (p.o32) store_block<W16>(gptr<float>(p.o32) + off, acc[0][n], inv, n, D, h);
    }
  } else {
#pragma unroll
    for (int k = 0; k < KH - 1; ++k)
#pragma unroll
      for (int v = 0; v < S::NACC; ++v)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[v / DCH][v % DCH][e] += parts[k * PS + (v * 16 + e) * 64 + lane];
    if (!own_ok) return;
    if constexpr (WHICH == 1) {
      HK_G float* const dk = gptr<float>(p.dk) + grad_row(p, b, hh, own, Sk, p.k_sb, p.k_sh, p.k_ss);
      HK_G float* const dv = gptr<float>(p.dv) + grad_row(p, b, hh, own, Sk, p.v_sb, p.v_sh, p.v_ss);
#pragma unroll
      for (int n = 0; n < DCH; ++n) {
        store_block<W16>(dk, acc[0][n], p.scale, n, D, h);
        store_block<W16>(dv, acc[S::NACC > DCH ? 1 : 0][n], 1.f, n, D, h);
      }
    } else {
      HK_G float* const dq = gptr<float>(p.dq) + grad_row(p, b, hh, own, Sq, p.q_sb, p.q_sh, p.q_ss);
#pragma unroll
      for (int n = 0; n < DCH; ++n) store_block<W16>(dq, acc[0][n], p.scale, n, D, h);
    }
  }
}

template <int WHICH, int DP, bool W16>
void queue_f32(const hrt_attn_args& a, hipStream_t s) {
  const int nb = (int)cdiv(WHICH == 1 ? a.Sk : a.Sq, 32 * Shape<WHICH, DP, W16>::G);
  hipLaunchKernelGGL((attn_f32_k<WHICH, DP, W16>), dim3((uint32_t)((int64_t)nb * a.B * a.H)), dim3(256), 0, s, a, nb);
}

template <int WHICH, bool W16>
void queue_d(const hrt_attn_args& a, hipStream_t s) {
  switch ((a.D + 31) / 32) {
    case 1: queue_f32<WHICH, 32, W16>(a, s); break;
    case 2: queue_f32<WHICH, 64, W16>(a, s); break;
    case 3: queue_f32<WHICH, 96, W16>(a, s); break;
    default: queue_f32<WHICH, 128, W16>(a, s); break;
  }
}

}  // namespace

// Queues the kernel (0 forward, 1 dK/dV, 2 dQ); false (nothing queued) when a stage's offsets do not fit 31 bits or the
// grid is too large (the scalar kernels take 64 rows in 64 threads, these 32 in 256).
bool attn_f32_mfma(const hrt_attn_args& a, int which, hipStream_t s) {
  if (!hrt::grid_fits(cdiv(which == 1 ? a.Sk : a.Sq, 32) * a.B * a.H, 256)) return false;
  const int64_t lim = ((int64_t)1 << 31) / (4 * 130);
  if (a.q_ss >= lim || a.k_ss >= lim || a.v_ss >= lim || (which != 0 && a.do_ss >= lim)) return false;
  // 16-byte accesses: whole 16-byte chunks of d, rows of every operand and output on 16-byte lines
  bool w16 = a.D % 4 == 0 && (a.q | a.k | a.v) % 16 == 0 &&
             (a.q_sb | a.q_sh | a.q_ss | a.k_sb | a.k_sh | a.k_ss | a.v_sb | a.v_sh | a.v_ss) % 4 == 0;
  if (which == 0) w16 = w16 && (a.o | a.o32) % 16 == 0;
  else w16 = w16 && a.dout % 16 == 0 && (a.do_sb | a.do_sh | a.do_ss) % 4 == 0 && (which == 1 ? a.dk | a.dv : a.dq) % 16 == 0;
  if (which == 0) w16 ? queue_d<0, true>(a, s) : queue_d<0, false>(a, s);
  else if (which == 1) w16 ? queue_d<1, true>(a, s) : queue_d<1, false>(a, s);
  else w16 ? queue_d<2, true>(a, s) : queue_d<2, false>(a, s);
  return true;
}

}  // namespace hk
