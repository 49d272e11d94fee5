"""Every tile, operand layout and split of the direct-to-LDS product in its masked form: sizes that leave part of a tile in M
and N and of a K step, at least five K steps (all buffers of a ring), against float64.  The tile is asked for through the
plan query, so that a changed cost model fails here and gets new sizes instead of silently leaving a form untested.
Operands lie in NaNs; tolerance as test_mm_edges: exact products, fp32 sums, one rounding."""

import ctypes

import pytest
import torch

import torch_vulkan
from torch_vulkan import abi
from test_mm_edges import check, dev, dq8_plan, window

# (m, n, k, A stored [k][m], B stored [n][k], tile, K split)
TILES = [(47, 48, 408, False, False, 64, 64, False), (49, 48, 432, False, True, 64, 64, False),
         (48, 40, 546, True, False, 64, 64, False), (48, 40, 432, True, True, 64, 64, False),
         (54, 40, 2000, False, False, 64, 64, True), (60, 41, 2136, False, True, 64, 64, True),
         (40, 40, 2020, True, False, 64, 64, True), (40, 40, 3368, True, True, 64, 64, True),
         (923, 1352, 328, False, False, 64, 128, False), (577, 2897, 328, False, True, 64, 128, False),
         (2224, 584, 332, True, False, 64, 128, False), (584, 2776, 328, True, True, 64, 128, False),
         (66, 1912, 1912, False, False, 64, 128, True), (65, 2016, 3096, False, True, 64, 128, True),
         (1136, 80, 3153, True, False, 64, 128, True), (2280, 68, 2584, True, True, 64, 128, True),
         (3067, 656, 336, False, False, 128, 128, False), (1255, 2128, 328, False, True, 128, 128, False),
         (2520, 776, 336, True, False, 128, 128, False), (2136, 928, 328, True, True, 128, 128, False),
         (65, 2824, 3464, False, False, 128, 128, True), (70, 3096, 3088, False, True, 128, 128, True),
         (72, 2136, 3173, True, False, 128, 128, True), (2120, 66, 3248, True, True, 128, 128, True),
         (2436, 1559, 328, False, True, 128, 192, False), (3280, 1192, 328, True, True, 128, 192, False),
         (1164, 3256, 336, False, False, 128, 256, False), (2997, 1925, 328, False, True, 128, 256, False),
         (3208, 1168, 339, True, False, 128, 256, False), (2440, 2328, 328, True, True, 128, 256, False),
         (388, 2712, 5072, False, False, 128, 256, True), (2690, 392, 5040, False, True, 128, 256, True),
         (2704, 392, 5016, True, False, 128, 256, True), (2704, 385, 5008, True, True, 128, 256, True),
         (2993, 1296, 336, False, False, 256, 128, False), (2469, 3128, 328, False, True, 256, 128, False),
         (2968, 1288, 337, True, False, 256, 128, False), (3224, 2320, 328, True, True, 256, 128, False),
         (3235, 2456, 456, False, False, 256, 256, False), (2335, 3334, 456, False, True, 256, 256, False),
         (2576, 3120, 450, True, False, 256, 256, False), (2344, 3364, 456, True, True, 256, 256, False)]
# (m, n, k, kernel, tile, K split) of the int8 linear
INT8 = [(17, 328, 448, abi.MM_DIRECT, 64, 64, False), (3, 228, 3200, abi.MM_DIRECT, 64, 64, True), (2344, 1285, 192, abi.MM_DIRECT, 128, 128, False),
        (1414, 3317, 192, abi.MM_DIRECT, 256, 128, False), (2290, 44, 576, abi.MM_DEQUANT, 64, 64, False),
        (2972, 727, 640, abi.MM_DEQUANT, 128, 128, False), (2055, 3624, 256, abi.MM_DEQUANT, 128, 256, False),
        (2953, 2694, 512, abi.MM_DEQUANT, 256, 256, False)]


def plan(m, n, k, ta, tb):
    """For operands as window() lays them out: 16-byte aligned, rows padded to whole chunks and 16 elements more."""
    lib, out = ctypes.CDLL(abi._LIB_PATH), abi.MmPlan()
    pitch = lambda c: (c + 7) // 8 * 8 + 16  # noqa: E731
    p = abi.MmArgs(a=4096, b=8192, c=1 << 20, M=m, N=n, K=k, batch=1, a_sm=1 if ta else pitch(k), a_sk=pitch(m) if ta else 1,
                   b_sk=1 if tb else pitch(n), b_sn=pitch(k) if tb else 1, c_sm=n, c_sn=1, alpha=1.0)
    assert lib.hrt_mm_plan_of(ctypes.byref(p), abi.BF16, 1, ctypes.byref(out)) == 0
    return out


def test_sizes_reach_their_tile():
    for m, n, k, ta, tb, bm, bn, split in TILES:
        p = plan(m, n, k, ta, tb)
        assert (p.kernel, p.tile_m, p.tile_n, p.splits > 1, p.whole) == (abi.MM_DIRECT, bm, bn, split, 0), (m, n, k, ta, tb)
        assert m % bm and n % bn and k % 64 and k > 256
    for m, n, k, kernel, bm, bn, split in INT8:
        p = dq8_plan(m, n, k)
        assert (p.kernel, p.tile_m, p.tile_n, p.splits > 1, p.whole) == (kernel, bm, bn, split, 0), (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k,ta,tb,bm,bn,split", TILES)
def test_masked_tiles(m, n, k, ta, tb, bm, bn, split, dt):
    g = torch.Generator().manual_seed(m + n + k)
    A, a = window(m, k, dt, g, ta)
    B, b = window(k, n, dt, g, tb)
    assert A.stride() == ((1, (m + 7) // 8 * 8 + 16) if ta else ((k + 7) // 8 * 8 + 16, 1)) and A.data_ptr() % 16 == B.data_ptr() % 16 == 0
    bias = torch.randn((n,), generator=g).to(dt)
    check(torch.addmm(bias.to(dev), A, B), a.double() @ b.double() + bias.double(), dt)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k,kernel,bm,bn,split", INT8)
def test_masked_int8_tiles(m, n, k, kernel, bm, bn, split, dt):
    g = torch.Generator().manual_seed(m + n)
    X, x = window(m, k, dt, g, False)
    q = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
    s = (torch.rand((n, k // 64), generator=g) * 0.02 + 1e-4).to(torch.bfloat16)
    bias = torch.randn((n,), generator=g).to(dt)
    w = (q.double() * s.double().repeat_interleave(64, 1)).to(dt).double()
    check(torch_vulkan.dequant_int8_linear(X, q.to(dev), s.to(dev), bias.to(dev)), x.double() @ w.t() + bias.double(), dt)


def test_every_tile_is_reached():
    """All seven tiles, split and unsplit where there is a split form, in every layout they exist in."""
    layouts = {(ta, tb) for ta in (False, True) for tb in (False, True)}
    want = {(bm, bn, False, *lay) for bm, bn in ((64, 64), (64, 128), (128, 128), (128, 256), (256, 128), (256, 256)) for lay in layouts}
    want |= {(bm, bn, True, *lay) for bm, bn in ((64, 64), (64, 128), (128, 128), (128, 256)) for lay in layouts}
    want |= {(128, 192, False, ta, True) for ta in (False, True)}
    assert {(bm, bn, split, ta, tb) for _, _, _, ta, tb, bm, bn, split in TILES} == want
