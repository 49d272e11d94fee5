// fp32 products on the fp32 matrix cores: "mm_f32" wherever an operand tile's offsets fit 31 bits and the reduction is
// not a short one (gemm.hip keeps the rest).  c = alpha * a @ b + beta * bias, fp32 multiplies and fp32 accumulation throughout (v_mfma_f32_32x32x2_f32:
// no rounding of the inputs), as the scalar kernel it replaces and vkrt/shaders/mm.comp.in:90-154.
//
// Bound: the fp32 matrix rate (157 TFLOP/s published; 64 cycles per 32 x 32 x 2 MFMA and SIMD).  A 64 x 64 x 32 step of
// a workgroup is 64 MFMAs over four SIMDs (1024 cycles) against 16 KB of copies and 64 16-byte LDS reads, so neither
// bandwidth is near its limit and small tiles, which balance better over 256 CUs, cost nothing.
//   * K advances in steps of 32 floats through a ring of three LDS buffers filled by buffer -> LDS copies issued two
//     steps ahead; a row of 32 floats is 128 bytes, the geometry and swizzle of the 16-bit kernel's tiles;
//   * an operand contiguous along K is staged [row][k] and read 16 bytes per lane: the lanes of the lower half-wave
//     take k .. k + 3, the upper half k + 4 .. k + 7, and MFMA i multiplies k + i and k + 4 + i (any pairing of k will
//     do as long as A and B agree); an operand contiguous along M or N is staged [k][row] and read 4 bytes per lane;
//   * 16-byte aligned rows are copied 16 bytes per lane; any other strides 4 bytes per lane, each lane with an
//     address of its own, which the long MFMA phase hides as well;
//   * edges: lanes past M, N or K read zeros by the buffer's range check, the partial K step comes first (as
//     gemm_dma_kernel.h).
// Measured: 4096^3 NT 975 us, 141 TFLOP/s; x W^T / g W / g^T x of 1024 tokens, 1024 -> 2048: 141 / 187 / 325 us in the
// scalar kernel (gemm.hip), 39.0 / 46.7 / 40.2 here (the layer 659 -> 136.6); relative L2 error against float64 the same (5.7e-7 at K = 1024).
#include <type_traits>
#include <utility>

#include "../hrt/registry.h"
#include "lds_stage.h"

namespace hk {

bool mm_f32_mfma(const hrt_mm_args& a, hipStream_t s);
bool mm_check_operands(const hrt_mm_args& a, uint64_t elem, hrt::LaunchCtx& ctx);

namespace {

constexpr int FBK = 32;  // K floats per step

// This wavefront's IPW copies of a ROWS x COLS tile of floats at row stride ss, column stride cs (bytes): offsets of
// the elements that exist ([row_lo, row_hi) x [c_lo, c_hi)), kNoRow elsewhere.  W16: 16-byte copies (cs = 4).
template <int COLS, int IPW, bool W16>
__device__ __forceinline__ void f32_lane_offsets(uint32_t (&off)[IPW], uint32_t ss, uint32_t cs, int lane, int j0, int row_lo,
                                                 int row_hi, int c_lo, int c_hi) {
  constexpr int NCH = COLS / 4;
  if constexpr (W16) {
    edge_lane_offsets<NCH, IPW>(off, ss, lane, j0, row_lo, row_hi, c_lo / 4, c_hi / 4);
  } else {
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int d = (j0 + i) * 64 + lane, row = d / COLS, c = (((d % COLS) >> 2) ^ tile_swz<NCH>(row)) * 4 + (d & 3);
      off[i] = row >= row_lo && row < row_hi && c >= c_lo && c < c_hi ? (uint32_t)row * ss + (uint32_t)c * cs : kNoRow;
    }
  }
}
template <bool W16>
__device__ __forceinline__ void f32_copy(__amdgpu_buffer_rsrc_t rs, HK_L uint8_t* tile, int j, uint32_t off) {
  if constexpr (W16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, tile + j * 1024, 16, (int)off, 0, 0, 0);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, tile + j * 256, 4, (int)off, 0, 0, 0);
}

template <int BM, int BN, int WM, int WN, bool ATR, bool BTR, bool W16>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void mm_f32_dma(hrt_mm_args p, int tiles_m, int tiles_n,
                                                                        int64_t kslice) {
  constexpr int WNN = BN / WN, NW = (BM / WM) * WNN, FM = WM / 32, FN = WN / 32;
  constexpr int A_COLS = ATR ? BM : FBK, B_COLS = BTR ? BN : FBK;  // floats per tile row
  constexpr int A_TILE = BM * FBK * 4, B_TILE = BN * FBK * 4, CB = W16 ? 1024 : 256;  // bytes per copy instruction
  constexpr int IPA = A_TILE / CB / NW, IPB = B_TILE / CB / NW;
  static_assert(IPA * NW * CB == A_TILE && IPB * NW * CB == B_TILE && IPA + IPB < 32, "copy split");
  __shared__ __attribute__((aligned(1024))) uint8_t a0[A_TILE], a1[A_TILE], a2[A_TILE], b0[B_TILE], b1[B_TILE], b2[B_TILE];
  auto abuf = [&](auto ic) { constexpr int I = decltype(ic)::value; return (HK_L uint8_t*)(I == 0 ? a0 : I == 1 ? a1 : a2); };
  auto bbuf = [&](auto ic) { constexpr int I = decltype(ic)::value; return (HK_L uint8_t*)(I == 0 ? b0 : I == 1 ? b1 : b2); };

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WNN, wn = wave % WNN, l32 = lane & 31, h = lane >> 5;
  const uint32_t tile = blockIdx.x;
  const uint32_t tn = tile % (uint32_t)tiles_n, tm = (tile / (uint32_t)tiles_n) % (uint32_t)tiles_m;
  const int64_t bz = tile / ((uint32_t)tiles_n * (uint32_t)tiles_m), m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  // this workgroup's K range: all of it, or slice bz of a product split along K
  int64_t k0 = kslice > 0 ? bz * kslice : 0;
  const int K = (int)(kslice > 0 && p.K - k0 > kslice ? kslice : p.K - k0);
  const int nk = (K + FBK - 1) / FBK, kskip = nk * FBK - K;
  k0 -= kskip;
  const HK_G uint8_t* Ab = reinterpret_cast<const HK_G uint8_t*>(gcptr<float>(p.a) + bz * p.a_sb + m0 * p.a_sm + k0 * p.a_sk);
  const HK_G uint8_t* Bb = reinterpret_cast<const HK_G uint8_t*>(gcptr<float>(p.b) + bz * p.b_sb + n0 * p.b_sn + k0 * p.b_sk);
  const int64_t astep = FBK * p.a_sk * 4, bstep = FBK * p.b_sk * 4;
  const int ml = p.M - m0 < BM ? (int)(p.M - m0) : BM, nl = p.N - n0 < BN ? (int)(p.N - n0) : BN;
  const uint32_t ams = (uint32_t)(p.a_sm * 4), aks = (uint32_t)(p.a_sk * 4), bns = (uint32_t)(p.b_sn * 4), bks = (uint32_t)(p.b_sk * 4);
  uint32_t ao[IPA], ao0[IPA], bo[IPB], bo0[IPB];  // whole steps; step 0, whose first kskip elements are zeros
  if constexpr (ATR) {
    f32_lane_offsets<A_COLS, IPA, W16>(ao, aks, ams, lane, wave * IPA, 0, FBK, 0, ml);
    f32_lane_offsets<A_COLS, IPA, W16>(ao0, aks, ams, lane, wave * IPA, kskip, FBK, 0, ml);
  } else {
    f32_lane_offsets<A_COLS, IPA, W16>(ao, ams, aks, lane, wave * IPA, 0, ml, 0, FBK);
    f32_lane_offsets<A_COLS, IPA, W16>(ao0, ams, aks, lane, wave * IPA, 0, ml, kskip, FBK);
  }
  if constexpr (BTR) {
    f32_lane_offsets<B_COLS, IPB, W16>(bo, bks, bns, lane, wave * IPB, 0, FBK, 0, nl);
    f32_lane_offsets<B_COLS, IPB, W16>(bo0, bks, bns, lane, wave * IPB, kskip, FBK, 0, nl);
  } else {
    f32_lane_offsets<B_COLS, IPB, W16>(bo, bns, bks, lane, wave * IPB, 0, nl, 0, FBK);
    f32_lane_offsets<B_COLS, IPB, W16>(bo0, bns, bks, lane, wave * IPB, 0, nl, kskip, FBK);
  }
  auto copy = [&](int ks, HK_L uint8_t* At, HK_L uint8_t* Bt) {
    const __amdgpu_buffer_rsrc_t ar = edge_rsrc(Ab + ks * astep), br = edge_rsrc(Bb + ks * bstep);
#pragma unroll
    for (int c = 0; c < IPA; ++c) f32_copy<W16>(ar, At, wave * IPA + c, ks == 0 ? ao0[c] : ao[c]);
#pragma unroll
    for (int c = 0; c < IPB; ++c) f32_copy<W16>(br, Bt, wave * IPB + c, ks == 0 ? bo0[c] : bo[c]);
  };

  // byte offset of element (k = 8 g + 4 h + i, row r) for fragment reads: [row][k] tiles one 16-byte chunk per g, [k][row]
  // tiles one float per (g, i)
  auto frag = [&](auto tr, auto cols, const HK_L uint8_t* T, int r, int g) -> f32x4 {
    constexpr int COLS = decltype(cols)::value;
    if constexpr (!decltype(tr)::value) {
      return *reinterpret_cast<const HK_L f32x4*>(T + tile_off<FBK / 4>(r, 2 * g + h));
    } else {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 8 * g + 4 * h + i;
        v[i] = *reinterpret_cast<const HK_L float*>(T + tile_off<COLS / 4>(k, r >> 2) + (r & 3) * 4);
      }
      return v;
    }
  };
  using AT = std::integral_constant<bool, ATR>;
  using BT = std::integral_constant<bool, BTR>;
  using AC = std::integral_constant<int, A_COLS>;
  using BC = std::integral_constant<int, B_COLS>;

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = zero16();

  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  copy(0, abuf(I0()), bbuf(I0()));
  issue_order_fence();
  if (nk > 1) copy(1, abuf(I1()), bbuf(I1()));
  if (nk > 1) barrier_keep_vm<IPA + IPB>();
  else barrier_keep_vm<0>();
  // step kt: copies of step kt + 2 into the buffer that step kt - 1 read (its readers passed the last barrier), MFMAs of
  // buffer kt % 3; the closing barrier waits for step kt + 1's copies.  No copy past the last step.
  auto step = [&](auto bc, int kt) {
    constexpr int BUF = decltype(bc)::value, NXT = (BUF + 2) % 3;
    const HK_L uint8_t* At = abuf(bc);
    const HK_L uint8_t* Bt = bbuf(bc);
    const bool more = kt + 2 < nk;
    if (more) copy(kt + 2, abuf(std::integral_constant<int, NXT>()), bbuf(std::integral_constant<int, NXT>()));
    f32x4 af[2][FM], bf[2][FN];
    auto rd = [&](int g) {
#pragma unroll
      for (int i = 0; i < FM; ++i) af[g & 1][i] = frag(AT(), AC(), At, wm * WM + i * 32 + l32, g);
#pragma unroll
      for (int j = 0; j < FN; ++j) bf[g & 1][j] = frag(BT(), BC(), Bt, wn * WN + j * 32 + l32, g);
    };
    rd(0);
#pragma unroll
    for (int g = 0; g < FBK / 8; ++g) {
      __builtin_amdgcn_sched_barrier(0);
      if (g + 1 < FBK / 8) rd(g + 1);
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[g & 1][i][k], bf[g & 1][j][k], acc[i][j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) barrier_keep_vm<IPA + IPB>();
    else barrier_keep_vm<0>();
  };
  int kt = 0;
  for (; kt + 3 <= nk; kt += 3) {
    step(I0(), kt);
    step(I1(), kt + 1);
    step(I2(), kt + 2);
  }
  if (kt < nk) step(I0(), kt);
  if (kt + 1 < nk) step(I1(), kt + 1);

  const bool has_bias = p.has_bias != 0;
  const HK_G float* bias = gcptr<float>(p.bias) + bz * p.bias_sb;
  HK_G float* C = gptr<float>(p.c) + bz * p.c_sb;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int64_t gn = n0 + wn * WN + j * 32 + l32;
    if (gn >= p.N) continue;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int64_t gm0 = m0 + wm * WM + i * 32 + 4 * h;
      float bv[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t gm = gm0 + 8 * (e >> 2) + (e & 3);
        bv[e] = has_bias ? bias[(gm < p.M ? gm : p.M - 1) * p.bias_sm + gn * p.bias_sn] : 0.f;
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t gm = gm0 + 8 * (e >> 2) + (e & 3);
        if (gm < p.M) C[gm * p.c_sm + gn * p.c_sn] = has_bias ? p.alpha * acc[i][j][e] + p.beta * bv[e] : p.alpha * acc[i][j][e];
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, bool W16>
void queue_f32(const hrt_mm_args& a, bool atr, bool btr, int64_t kslice, hipStream_t s) {
  const int tm = (int)cdiv(a.M, BM), tn = (int)cdiv(a.N, BN);
  const dim3 g((uint32_t)((int64_t)tm * tn * a.batch)), blk((BM / WM) * (BN / WN) * 64);
  if (!atr && !btr) hipLaunchKernelGGL((mm_f32_dma<BM, BN, WM, WN, false, false, W16>), g, blk, 0, s, a, tm, tn, kslice);
  else if (!atr && btr) hipLaunchKernelGGL((mm_f32_dma<BM, BN, WM, WN, false, true, W16>), g, blk, 0, s, a, tm, tn, kslice);
  else if (atr && !btr) hipLaunchKernelGGL((mm_f32_dma<BM, BN, WM, WN, true, false, W16>), g, blk, 0, s, a, tm, tn, kslice);
  else hipLaunchKernelGGL((mm_f32_dma<BM, BN, WM, WN, true, true, W16>), g, blk, 0, s, a, tm, tn, kslice);
}

constexpr int FT = 64;  // tile edge: 128 x 128 tiles (eight wavefronts of 64 x 32) were slower everywhere (1024 x 2048 x
                        // 1024 73 against 45 us traced, half the CUs idle; 4096^3 1026 against 975)

// Whether a tile's element offsets fit the copies' 31 bits.
bool f32_fits(const hrt_mm_args& a) {
  const int64_t lim = (int64_t)1 << 31;
  return a.K < lim && a.a_sm < lim / 1024 && a.a_sk < lim / 1024 && a.b_sn < lim / 1024 && a.b_sk < lim / 1024 &&
         cdiv(a.M, FT) * cdiv(a.N, FT) * a.batch < lim;
}

// Staged along the contiguous axis; 16-byte copies where every row (and batch entry) starts on a 16-byte line and holds
// whole chunks.
struct F32Form {
  bool atr, btr, w16;
};
F32Form f32_form(const hrt_mm_args& a) {
  const bool atr = a.a_sm == 1 && a.a_sk != 1, btr = a.b_sn == 1 && a.b_sk != 1;
  const auto chunks = [&](uint64_t p, int64_t sb, bool tr, int64_t s_r, int64_t s_k, int64_t rows) {
    return p % 16 == 0 && (a.batch == 1 || sb % 4 == 0) &&
           (tr ? s_k % 4 == 0 && rows % 4 == 0 : s_k == 1 && s_r % 4 == 0 && a.K % 4 == 0);
  };
  return {atr, btr, chunks(a.a, a.a_sb, atr, a.a_sm, a.a_sk, a.M) && chunks(a.b, a.b_sb, btr, a.b_sn, a.b_sk, a.N)};
}

void queue_mm_f32(const hrt_mm_args& a, int64_t kslice, hipStream_t s) {
  const F32Form f = f32_form(a);
  if (f.w16) queue_f32<64, 64, 32, 32, true>(a, f.atr, f.btr, kslice, s);
  else queue_f32<64, 64, 32, 32, false>(a, f.atr, f.btr, kslice, s);
}

// Short reductions stay on the scalar kernel (gemm.hip): it steps by 16 of K and its small workgroups share a CU, where
// a tile here takes whole 32-float steps and the first loads of a deep ring.  Scalar against here, us: 100 x 100 x 16
// 4.4 / 5.4, x 20 equal; 4-byte copies 101 x 99 x 33 6.6 / 7.0, x 49 8.0 / 7.0.  Many tiles mostly past the edge of a
// narrow output last longer: 100000 x 3 x 16 9.3 / 18.7, 60000 x 16 x 48 0.90 of the time here, x 56 1.03; 4-byte copies
// 100001 x 3 x 65 0.85, x 81 1.1; batches of 16384 3 x 5 x 129 0.93, of 1000 15 x 17 x 129 1.03.
bool f32_scalar(const hrt_mm_args& a) {
  if (a.K > 144 || cdiv(a.M, FT) > 65535) return false;
  const bool narrow = a.M < a.N ? a.M <= 32 : a.N <= 32, many = cdiv(a.M, FT) * cdiv(a.N, FT) * a.batch >= 768;
  if (f32_form(a).w16) return a.K <= (narrow && many ? 48 : 16);
  return a.K <= (!narrow || !many ? 48 : a.M <= 32 && a.N <= 32 ? 144 : 80);
}

// K slices of one product (1: none): where its 64 x 64 tiles leave CUs idle.  A 32-float step of a tile takes 0.45 us of
// a CU's matrix cores, however many workgroups share them; a split adds the partial products' write and read (~5 TB/s)
// and a launch (unsplit 128 x 128 x 4096 77 us, 300 x 512 x 3001 70, on 4 and 40 of the 256 CUs).
int64_t f32_splits(const hrt_mm_args& a) {
  if (a.batch != 1 || !f32_fits(a)) return 1;
  const int64_t tiles = cdiv(a.M, FT) * cdiv(a.N, FT), nk = cdiv(a.K, FBK);
  if (tiles > 512) return 1;
  int64_t best = 1;
  double best_us = 0.0, whole_us = 0.0;
  for (int64_t s = 1; s <= 32 && (s == 1 || nk >= 4 * s); ++s) {
    const int64_t per = cdiv(nk, s), n = cdiv(nk, per);
    double us = (double)cdiv(tiles * n, 256) * (per * 0.45 + 1.0);
    if (n > 1) us += 3.3 + 0.3 * n + 1.1 * (double)n * a.M * a.N * 4 / 5e6;
    if (s == 1) whole_us = us;
    if (s == 1 || us < best_us) best_us = us, best = n;
  }
  return best_us > whole_us - 8.0 ? 1 : best;  // the workspace and the second launch cost the host ~4 us, the estimate is rough
}

// c = alpha * (sum of the slices in order) + beta * bias, four outputs per thread.
__global__ __launch_bounds__(256) void mm_reduce_f32(hrt_mm_args p, const float* __restrict__ ws, int splits) {
  const int64_t total = p.M * p.N, i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i0 >= total) return;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
  if (total % 4 == 0) {
    const f32x4* w = reinterpret_cast<const f32x4*>(ws + i0);
    int k = 0;
    for (; k + 4 <= splits; k += 4) {
      f32x4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = w[(k + u) * (total / 4)];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += v[u][e];
    }
    for (; k < splits; ++k) {
      const f32x4 v = w[k * (total / 4)];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += v[e];
    }
  } else {
    for (int k = 0; k < splits; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i0 + e < total) s[e] += ws[k * total + i0 + e];
  }
  const HK_G float* bias = gcptr<float>(p.bias);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t i = i0 + e;
    if (i >= total) break;
    const int64_t m = i / p.N, n = i - m * p.N;
    float o = p.alpha * s[e];
    if (p.has_bias) o += p.beta * bias[m * p.bias_sm + n * p.bias_sn];
    gptr<float>(p.c)[m * p.c_sm + n * p.c_sn] = o;
  }
}

bool launch_mm_splitk_f32(const void* pp, const uint32_t*, hrt::LaunchCtx& ctx) {
  const auto& x = *static_cast<const hrt_mm_splitk_args*>(pp);
  const hrt_mm_args& a = x.mm;
  if (a.flags != 0) return ctx.fail("mm_splitk takes no flags");
  if (!mm_check_operands(a, 4, ctx)) return false;
  const int64_t splits = f32_splits(a);
  if (splits <= 1) {
    if (!mm_f32_mfma(a, ctx.stream)) return ctx.fail("mm_splitk: offsets above 31 bits");
    return hrt::launch_ok(hipGetLastError(), ctx, "mm_f32_dma");
  }
  if (x.ws_floats < splits * a.M * a.N) return ctx.fail("workspace smaller than hrt_mm_workspace says");
  if (x.ws % 16 != 0) return ctx.fail("ws must be 16-byte aligned");
  if (!ctx.check(x.ws, (uint64_t)x.ws_floats * 4, "ws")) return false;
  hrt_mm_args part = a;
  part.c = x.ws, part.batch = splits, part.c_sb = a.M * a.N, part.c_sm = a.N, part.c_sn = 1;
  part.a_sb = part.b_sb = 0, part.alpha = 1.f, part.has_bias = 0;
  queue_mm_f32(part, cdiv(cdiv(a.K, FBK), splits) * FBK, ctx.stream);
  if (!hrt::launch_ok(hipGetLastError(), ctx, "mm_f32_dma")) return false;
  hipLaunchKernelGGL(mm_reduce_f32, dim3((uint32_t)cdiv(a.M * a.N, 1024)), dim3(256), 0, ctx.stream, a,
                     reinterpret_cast<const float*>(x.ws), (int)splits);
  return hrt::launch_ok(hipGetLastError(), ctx, "mm_reduce_f32");
}

HRT_REGISTER("mm_splitk_f32", hrt_mm_splitk_args, launch_mm_splitk_f32);

}  // namespace

bool mm_f32_scalar(const hrt_mm_args& a) { return f32_scalar(a); }

// Queues the product; false (nothing queued) when a tile's element offsets do not fit 31 bits.
bool mm_f32_mfma(const hrt_mm_args& a, hipStream_t s) {
  if (!f32_fits(a)) return false;
  queue_mm_f32(a, 0, s);
  return true;
}

void mm_f32_plan(const hrt_mm_args& a, bool may_split, hrt_mm_plan* out) {
  if (!f32_fits(a) || f32_scalar(a)) return;
  const bool whole = a.M % FT == 0 && a.N % FT == 0 && a.K % FBK == 0;
  *out = hrt_mm_plan{HRT_MM_DIRECT, FT, FT, whole ? 1 : 0, may_split ? f32_splits(a) : 1};
}

int64_t mm_f32_workspace(const hrt_mm_args& a) {
  const int64_t s = f32_splits(a);
  return s > 1 ? s * a.M * a.N : 0;
}

}  // namespace hk
