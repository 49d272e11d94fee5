"""Matrix-core products at the edges of their tiles: sizes that leave part of a tile or of a 64-element K step,
every operand layout, K split over partial products, and the int8 linear at such sizes, against float64.

Every operand is a window of a NaN-filled buffer (rows padded to a multiple of 8 elements, as the direct-to-LDS
kernel needs), so a value read past an edge and not masked turns results into NaN.  Tolerance: the products
of 16-bit values are exact in fp32 and summed in fp32 (relative error of the sum below 2^-24 sqrt(K) of the
terms' size, under 1e-5 here), then rounded once: relative L2 below the output's half unit in the last place,
2^-9 (bf16) or 2^-12 (f16), plus 1e-5."""

import ctypes
import os
import random

import pytest
import torch

import torch_vulkan
from torch_vulkan import abi

dev = torch.device("vk")
gpu = pytest.mark.gpu
REL = {torch.bfloat16: 2.0**-9 + 1e-5, torch.float16: 2.0**-12 + 1e-5}


def window(rows, cols, dt, gen, transposed):
    """A [rows, cols] operand on vk inside NaNs, stored row-major or transposed, and its values."""
    v = torch.randn((rows, cols), generator=gen).to(dt)
    r, c = (cols, rows) if transposed else (rows, cols)
    host = torch.full((r + 3, (c + 7) // 8 * 8 + 16), float("nan"), dtype=dt)
    host[1 : 1 + r, 8 : 8 + c] = v.t() if transposed else v
    d = host.to(dev)[1 : 1 + r, 8 : 8 + c]
    return (d.t() if transposed else d), v


def check(out, ref, dt):
    o = out.detach().cpu().double()
    assert torch.isfinite(o).all()
    assert ((o - ref).norm() / ref.norm()).item() <= REL[dt]


# (M, N, K): one past / one short of the 64-, 128- and 256-wide tiles, K steps with 8 or 56 elements in the partial
# one, K below one step; the last ones are split along K
EDGES = [(65, 72, 72), (127, 136, 120), (129, 264, 64), (257, 248, 136), (200, 1000, 40), (600, 520, 1096), (2000, 1304, 264),
         (4020, 2048, 328), (120, 640, 2936), (24, 72, 4168), (604, 704, 5192)]


@gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("m,n,k", EDGES)
def test_ragged_products(m, n, k, ta, tb, dt):
    if ta:
        m = (m + 7) // 8 * 8  # a whole number of 16-byte chunks along the contiguous axis
    g = torch.Generator().manual_seed(m + n + k)
    A, a = window(m, k, dt, g, ta)
    B, b = window(k, n, dt, g, tb)
    bias = torch.randn((n,), generator=g).to(dt)
    ref = a.double() @ b.double()
    check(torch.mm(A, B), ref, dt)
    out = torch.addmm(bias.to(dev), A, B, alpha=0.5, beta=2.0)
    check(out, 0.5 * ref + 2.0 * bias.double(), dt)
    assert torch.equal(out.cpu(), torch.addmm(bias.to(dev), A, B, alpha=0.5, beta=2.0).cpu())


@gpu
@pytest.mark.parametrize("m,n,k", [(777, 943, 64), (65, 129, 200), (1000, 333, 2048), (33, 17, 4096)])
def test_output_rows_off_16_byte_lines(m, n, k):
    """N is no multiple of 8 (x W^T): rows of C start at any 2-byte offset."""
    dt = torch.bfloat16
    g = torch.Generator().manual_seed(n)
    A, a = window(m, k, dt, g, False)
    B, b = window(k, n, dt, g, True)
    bias = torch.randn((m, n), generator=g).to(dt)
    check(torch.addmm(bias.to(dev), A, B), a.double() @ b.double() + bias.double(), dt)


@gpu
@pytest.mark.parametrize("ta,tb", [(True, False), (True, True), (False, False)])
@pytest.mark.parametrize("k", [1, 77, 1001])
def test_odd_reduction_of_m_and_n_contiguous_operands(k, ta, tb):
    """K need not be a multiple of 8 where both operands are contiguous along M and N (g^T x over any number of
    tokens); the other layouts at odd K take the general kernel."""
    dt = torch.bfloat16
    g = torch.Generator().manual_seed(k)
    A, a = window(264, k, dt, g, ta)
    B, b = window(k, 328, dt, g, tb)
    check(torch.mm(A, B), a.double() @ b.double(), dt)


@gpu
@pytest.mark.parametrize("m,n,k,ld,dispatches", [(1024, 2048, 8192, 8194, 2), (1024, 2048, 6144, 6145, 2), (2048, 1536, 4096, 4097, 2),
                                                 (256, 512, 6144, 6145, 1), (128, 256, 8192, 8200, 1)])
def test_long_reductions_of_unaligned_operands_are_split(m, n, k, ld, dispatches):
    """Rows off 16-byte lines: the general kernel over K slices, then their ordered sum; few blocks stay whole, aligned
    rows (the last) go to mm_splitk, slices and sum in one dispatch."""
    dt = torch.bfloat16
    g = torch.Generator().manual_seed(ld)
    a, b = torch.randn((m, k), generator=g).to(dt), torch.randn((n, k), generator=g).to(dt)
    wide = torch.full((m, ld), float("nan"), dtype=dt)
    wide[:, :k] = a
    A, B = wide.to(dev)[:, :k], b.to(dev).t()
    torch.vk.synchronize()
    n0 = torch_vulkan.stats()["dispatch_n"]
    out = torch.mm(A, B)
    assert torch_vulkan.stats()["dispatch_n"] - n0 == dispatches
    check(out, a.double() @ b.double().t(), dt)


@gpu
@pytest.mark.parametrize("m,n,k", [(130, 136, 72), (257, 264, 136)])
def test_ragged_batches(m, n, k):
    dt = torch.float16
    g = torch.Generator().manual_seed(m)
    a, b = torch.randn((3, m, k), generator=g).to(dt), torch.randn((3, k, n), generator=g).to(dt)
    check(torch.bmm(a.to(dev), b.to(dev)), torch.bmm(a.double(), b.double()), dt)


@gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 200, 320), (17, 72, 2048), (65, 328, 1088), (300, 2000, 512), (1000, 520, 1024),
                                   (2049, 264, 320)])
def test_int8_linear_at_ragged_sizes(m, n, k, dt):
    g = torch.Generator().manual_seed(m + n)
    X, x = window(m, k, dt, g, False)
    q = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8)
    s = (torch.rand((n, k // 64), generator=g) * 0.02 + 1e-4).to(torch.bfloat16)
    bias = torch.randn((n,), generator=g).to(dt)
    w = (q.double() * s.double().repeat_interleave(64, 1)).to(dt).double()
    y = torch_vulkan.dequant_int8_linear(X, q.to(dev), s.to(dev), bias.to(dev))
    check(y, x.double() @ w.t() + bias.double(), dt)


# fp32 (fp32 matrix cores): 16-byte and 4-byte copies (odd sizes, offset views), every layout, split K, batches.
# Tolerance: an fp32 sum of K products, each fused multiply-add rounding to half a unit in the last place of the
# partial sum: relative L2 below 2^-24 sqrt(K) for random signs, doubled.
F32_EDGES = [(64, 64, 32), (65, 63, 33), (1, 1, 1), (130, 200, 31), (72, 136, 100), (127, 65, 257), (300, 512, 3001), (128, 128, 4096),
             (1000, 1000, 64)]


@gpu
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("m,n,k", F32_EDGES)
def test_f32_products(m, n, k, offset, ta, tb):
    g = torch.Generator().manual_seed(m + n + k)

    def make(rows, cols, transposed):
        v = torch.randn((rows, cols), generator=g)
        r, c = (cols, rows) if transposed else (rows, cols)
        host = torch.full((r + 2, (c + 3) // 4 * 4 + 8), float("nan"))
        host[1 : 1 + r, 4 + offset : 4 + offset + c] = v.t() if transposed else v
        d = host.to(dev)[1 : 1 + r, 4 + offset : 4 + offset + c]
        return (d.t() if transposed else d), v

    A, a = make(m, k, ta)
    B, b = make(k, n, tb)
    bias = torch.randn((n,), generator=g)
    ref = a.double() @ b.double()
    tol = 2.0**-23 * k**0.5 + 2.0**-23
    out = torch.mm(A, B).cpu()
    assert ((out - ref).norm() / ref.norm()).item() <= tol
    out = torch.addmm(bias.to(dev), A, B, alpha=0.5, beta=2.0).cpu()
    want = 0.5 * ref + 2.0 * bias.double()
    assert ((out - want).norm() / want.norm()).item() <= 2 * tol


# (m, n, k, batch, scalar): both sides of the lines between the scalar kernel and the matrix cores: 16-byte rows K = 16,
# many narrow tiles 48; 4-byte copies 48, many narrow tiles 80, a batch of mostly empty ones 144
F32_SHORT = [(100, 100, 16, 1, True), (100, 100, 20, 1, False), (64, 64, 1, 1, True), (101, 99, 47, 1, True), (101, 99, 49, 1, False),
             (50000, 16, 48, 1, True), (50000, 16, 52, 1, False), (50001, 3, 79, 1, True), (50001, 3, 81, 1, False),
             (3, 5, 143, 1000, True), (3, 5, 145, 1000, False), (7, 33, 79, 1000, True), (8, 32, 52, 1000, False)]


@pytest.mark.parametrize("m,n,k,batch,scalar", F32_SHORT)
def test_short_f32_reductions_stay_scalar(m, n, k, batch, scalar):
    p = plan_of(m, n, k, dtype=abi.F32, batch=batch)
    assert p.kernel == (abi.MM_GENERAL if scalar else abi.MM_DIRECT) and p.splits == 1


@gpu
@pytest.mark.parametrize("m,n,k,batch,scalar", F32_SHORT)
def test_short_f32_reductions(m, n, k, batch, scalar):
    g = torch.Generator().manual_seed(m + k)
    a, b = torch.randn((batch, m, k), generator=g), torch.randn((batch, n, k), generator=g)
    ref = a.double() @ b.double().transpose(1, 2)
    A, B = a.to(dev), b.to(dev).transpose(1, 2)
    out = (torch.bmm(A, B) if batch > 1 else torch.mm(A[0], B[0])).cpu().view(ref.shape)
    assert ((out - ref).norm() / ref.norm()).item() <= 2.0**-23 * k**0.5 + 2.0**-23


@gpu
def test_f32_strided_batches_and_small_values():
    g = torch.Generator().manual_seed(0)
    a, b = torch.randn((3, 70, 90), generator=g), torch.randn((3, 50, 180), generator=g)
    A, B = a.to(dev), b.to(dev)[:, :, ::2].transpose(1, 2)  # k strided by 2: no contiguous axis
    ref = a.double() @ b.double()[:, :, ::2].transpose(1, 2)
    assert ((torch.bmm(A, B).cpu() - ref).norm() / ref.norm()).item() <= 2.0**-23 * 90**0.5
    x, y = torch.full((64, 64), 1e-30), torch.full((64, 64), 1e-10)  # subnormal products are kept
    z = torch.mm(x.to(dev), y.to(dev)).cpu().double()
    assert torch.allclose(z, torch.full_like(z, 64e-40), rtol=1e-4)
    inf = torch.zeros((64, 64))
    inf[3, 5] = float("inf")
    o = torch.mm(inf.to(dev), torch.ones((64, 64)).to(dev)).cpu()
    assert torch.isinf(o[3]).all() and torch.equal(o[:3], torch.zeros(3, 64)) and torch.isfinite(o[4:]).all()


@gpu
def test_infinities_and_nans_stay_in_their_rows():
    """A ragged product's masked K elements and rows are zeros: an inf or NaN of the operands reaches exactly the
    outputs whose row or column holds it."""
    a, b = torch.randn((70, 72)), torch.randn((72, 136))
    a[3, 71], b[5, 9] = float("inf"), float("nan")
    a, b = a.bfloat16(), b.bfloat16()
    out = torch.mm(a.to(dev), b.to(dev)).cpu()
    ref = (a.double() @ b.double())
    assert torch.equal(torch.isnan(out), torch.isnan(ref)) and torch.equal(torch.isinf(out), torch.isinf(ref))


@gpu
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(130, 136, 72), (256, 256, 128), (70, 72, 1096)])
def test_expanded_operands(m, n, k, dt):
    """Operands repeated along M, N or K by a zero stride, against the same values laid out."""
    g = torch.Generator().manual_seed(m + k)

    def forms(rows, cols):
        full, row, col = (torch.randn(s, generator=g).to(dt).to(dev) for s in ((rows, cols), (1, cols), (rows, 1)))
        return full, row.expand(rows, cols), col.expand(rows, cols), row[:, :1].expand(rows, cols)

    for i, A in enumerate(forms(m, k)):
        for j, B in enumerate(forms(k, n)):
            if i == j == 0:
                continue
            a, b = A.cpu().double(), B.cpu().double()
            out = torch.mm(A, B).cpu().double()
            # roundings of repeated values do not average out: k of them, each of the sum of the sizes of the terms
            bound = (a.abs() @ b.abs()) * (2.0**-23 * k) + (out.abs() * (2.0**-8 if dt == torch.bfloat16 else 2.0**-23))
            assert ((out - a @ b).abs() <= bound + 1e-30).all(), (i, j)


def plan(m, n, k, a_off=0, dtype=abi.BF16, **kw):
    lib = ctypes.CDLL(abi._LIB_PATH)
    lib.hrt_mm_workspace.restype = ctypes.c_int64
    lib.hrt_mm_workspace.argtypes = [ctypes.c_void_p, ctypes.c_int32]
    p = abi.MmArgs(a=4096 + a_off, b=8192, c=1 << 20, M=m, N=n, K=k, batch=1, a_sm=k, a_sk=1, b_sk=1, b_sn=k, c_sm=n, c_sn=1)
    for name, v in kw.items():
        setattr(p, name, v)
    return lib.hrt_mm_workspace(ctypes.byref(p), dtype)


def plan_of(m, n, k, ta=False, tb=True, dtype=abi.BF16, split=True, off=0, batch=1):
    """hrt_mm_plan_of for contiguous operands (ta: A stored [k][m], tb: B stored [n][k])."""
    lib = ctypes.CDLL(abi._LIB_PATH)
    p = abi.MmArgs(a=4096 + off, b=8192, c=1 << 20, M=m, N=n, K=k, batch=batch, a_sm=1 if ta else k, a_sk=m if ta else 1,
                   b_sk=1 if tb else n, b_sn=k if tb else 1, c_sm=n, c_sn=1, alpha=1.0, a_sb=m * k, b_sb=n * k, c_sb=m * n)
    out = abi.MmPlan()
    assert lib.hrt_mm_plan_of(ctypes.byref(p), dtype, int(split), ctypes.byref(out)) == 0
    return out


def test_plan_query_agrees_with_the_workspace():
    rng = random.Random(0)
    for _ in range(300):
        m, n, k = (rng.choice((rng.randint(1, 4000), 64 * rng.randint(1, 64))) for _ in range(3))
        p = plan_of(m, n, k, tb=True)
        w = plan(m, n, k)
        assert (p.kernel == abi.MM_GENERAL) == (w < 0) and max(w, 0) == (p.splits * m * n if p.splits > 1 else 0), (m, n, k)
        assert not p.whole or (m % p.tile_m == 0 and n % p.tile_n == 0 and k % 64 == 0)
        assert p.kernel != abi.MM_NARROW or min(m, n) <= 16 or k <= 32
        assert plan_of(m, n, k, split=False).splits == 1
    assert plan_of(64, 64, 64, off=2).kernel == abi.MM_GENERAL


# (m, n, k, ta, tb) that an earlier cost model put on a tile 12 to 24% slower than one it had (1152 x 1152 x 1024 on 64 x
# 128 10.3 us, on 64 x 64 8.2), and the tiles within 10% of the fastest, all timed unsplit
TILES = [((1152, 1152, 1024, False, False), {(64, 64)}), ((384, 2816, 2816, True, True), {(64, 64)}),
         ((6144, 512, 1024, True, True), {(128, 128)}), ((5632, 512, 1920, True, True), {(128, 128)}),
         ((8064, 384, 640, True, False), {(128, 128)}), ((1024, 2048, 2048, False, True), {(64, 128)}),
         ((512, 3072, 3072, False, True), {(64, 128)}), ((1024, 1152, 1536, True, True), {(64, 64)}),
         ((1472, 960, 320, False, False), {(64, 64)}), ((2176, 512, 2176, False, False), {(64, 64), (64, 128)}),
         ((320, 4864, 1024, True, False), {(64, 64)}), ((1792, 832, 2944, True, False), {(64, 64), (64, 128)})]


@pytest.mark.parametrize("product,tiles", TILES)
def test_plan_takes_a_fast_tile(product, tiles):
    p = plan_of(*product, split=False)
    assert (p.tile_m, p.tile_n) in tiles


def dq8_plan(m, n, k, with_ws=True):
    lib = ctypes.CDLL(abi._LIB_PATH)
    p = abi.MmDq8Args(x=4096, q=8192, scale=4096, y=4096, M=m, N=n, K=k, nblocks=k // 64, x_sm=k, x_sk=1, alpha=1.0)
    out = abi.MmPlan()
    assert lib.hrt_mm_dq8_plan_of(ctypes.byref(p), int(with_ws), ctypes.byref(out)) == 0
    return out


@pytest.mark.parametrize("m,n,k,kernel", [(2048, 1024, 320, abi.MM_DIRECT), (3120, 1024, 320, abi.MM_DIRECT), (7424, 512, 320, abi.MM_DIRECT),
                                          (2048, 8192, 2048, abi.MM_DEQUANT), (3120, 2048, 8192, abi.MM_DEQUANT), (1024, 8192, 2048, abi.MM_DIRECT)])
def test_int8_weights_are_dequantized_first_only_where_it_pays(m, n, k, kernel):
    """A second launch and pass of its own: 2048 x 1024 x 320 8.8 us against 7.1 fused, 2048 x 8192 x 2048 75 against 96."""
    assert dq8_plan(m, n, k).kernel == kernel and dq8_plan(m, n, k, with_ws=False).kernel == abi.MM_DIRECT


def test_split_plan_on_the_host():
    """hrt_mm_workspace: whole numbers of [M, N] slices, none for full grids and products with kernels of their own,
    -1 for operands off 16-byte lines."""
    assert os.path.exists(abi._LIB_PATH)
    for m, n, k in [(604, 704, 5184), (300, 64, 4096), (1024, 2048, 8192), (113, 632, 2936)]:
        w = plan(m, n, k)
        assert w > 0 and w % (m * n) == 0 and w // (m * n) <= k // 64 // 4, (m, n, k, w)
    for m, n, k in [(4096, 4096, 4096), (1024, 8192, 2048), (1024, 1024, 1024), (16, 4096, 4096), (4096, 4096, 32)]:
        assert plan(m, n, k) == 0
    assert plan(604, 704, 5184, a_off=2) == -1 and plan(604, 704, 5184, c_sn=2) == -1
    assert plan(128, 128, 4096, dtype=abi.F32) % (128 * 128) == 0 and plan(128, 128, 4096, dtype=abi.F32) > 0
    assert plan(2048, 2048, 64, dtype=abi.F32) == 0
    assert plan(604, 704, 5184, batch=2, a_sb=604 * 5184, b_sb=704 * 5184) == 0


def test_int8_workspace_is_the_size_of_what_it_holds():
    """Few rows: the fp32 partial products of 2 to 8 K slices, not the dequantized weights, whose 256 MiB at 16384 x
    8192 would be a reservation from the driver and a wait for the GPU on every call (16 rows: 340 us, 138 without)."""
    lib = ctypes.CDLL(abi._LIB_PATH)
    lib.hrt_mm_dq8_workspace.restype = ctypes.c_int64

    def elems(m, n, k):
        p = abi.MmDq8Args(x=4096, q=8192, scale=4096, y=4096, M=m, N=n, K=k, nblocks=k // 64, x_sm=k, x_sk=1, alpha=1.0)
        return lib.hrt_mm_dq8_workspace(ctypes.byref(p))

    for m, n, k in [(1, 16384, 8192), (16, 16384, 8192), (16, 8192, 16384), (16, 8192, 2048), (100, 2048, 8192)]:
        w = elems(m, n, k)
        assert 0 < w <= n * k and w % (2 * m * n) == 0 and 2 <= w // (2 * m * n) <= 8, (m, n, k, w)
    assert elems(4096, 8192, 2048) == 8192 * 2048 and elems(1024, 8192, 2048) == 0
