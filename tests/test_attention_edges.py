"""Fused attention at the edges of its kernels' tiles, against float64: several streamed stages with a partial last
one, head dimensions at and off the tile widths, row strides and alignments, few keys under many queries.

Operands are windows of NaN-filled buffers, so a value read past an edge and not masked shows.  Tolerance (relative L2
of o, dq, dk, dv): f32 the accumulation of D and S products and two exponentials' rounding, 2^-24 (sqrt(D) + sqrt(S) +
16) with a factor 2; bf16 / f16 the bounds that the other attention tests use."""

import math

import pytest
import torch
import torch.nn.functional as F

import torch_vulkan

pytestmark = pytest.mark.gpu
dev = torch.device("vk")
REL16 = {torch.bfloat16: 1e-2, torch.float16: 4e-3}


@pytest.fixture(autouse=True)
def _always_fused():
    torch_vulkan.set_fused_attention("on")
    yield
    torch_vulkan.set_fused_attention("auto")


def operand(B, S, H, D, dt, g, pad, offset):
    """[B, H, S, D] view of token-major memory with NaN rows and columns around it."""
    v = torch.randn((B, S, H, D), generator=g).to(dt)
    host = torch.full((B, S + 1, H, D + pad), float("nan"), dtype=dt)
    host[:, :S, :, offset : offset + D] = v
    return host.to(dev)[:, :S, :, offset : offset + D].transpose(1, 2).detach().requires_grad_(True), v.double().transpose(1, 2)


def check(B, H, Sq, Sk, D, dt, rel, pad=8, offset=0):
    g = torch.Generator().manual_seed(Sq + Sk + D)
    (q, q64), (k, k64), (v, v64) = (operand(B, s, H, D, dt, g, pad, offset) for s in (Sq, Sk, Sk))
    go = torch.randn((B, H, Sq, D), generator=g).to(dt)
    out = F.scaled_dot_product_attention(q, k, v)
    got = (out,) + torch.autograd.grad(out, (q, k, v), go.to(dev))
    leaves = [t.clone().requires_grad_(True) for t in (q64, k64, v64)]
    ref = torch.softmax(leaves[0] @ leaves[1].transpose(-1, -2) / math.sqrt(D), -1) @ leaves[2]
    want = (ref,) + torch.autograd.grad(ref, leaves, go.double())
    for name, a, b in zip(("o", "dq", "dk", "dv"), got, want):
        a = a.detach().cpu().double()
        assert torch.isfinite(a).all(), name
        e = ((a - b).norm() / b.norm()).item()
        assert e <= rel, (name, e)
    again = F.scaled_dot_product_attention(q, k, v)
    rep = (again,) + torch.autograd.grad(again, (q, k, v), go.to(dev))
    assert all(torch.equal(a.detach().cpu(), b.detach().cpu()) for a, b in zip(got, rep))  # same bits twice


def f32_rel(Sk, D):
    return 2 * 2.0**-24 * (math.sqrt(D) + math.sqrt(Sk) + 16)


@pytest.mark.parametrize("D", [8, 30, 32, 40, 64, 68, 96, 112, 128])
@pytest.mark.parametrize("Sq,Sk", [(333, 777), (129, 64), (64, 129), (260, 31)])
def test_f32_stages_and_head_dims(Sq, Sk, D):
    check(2, 3, Sq, Sk, D, torch.float32, f32_rel(max(Sq, Sk), D))


@pytest.mark.parametrize("D,pad,offset", [(64, 4, 4), (64, 3, 1), (128, 5, 2), (33, 4, 0)])
def test_f32_strides_and_alignments(D, pad, offset):
    check(1, 2, 200, 300, D, torch.float32, f32_rel(300, D), pad, offset)


def test_f32_many_workgroups():
    """More workgroups than the chip holds at once, a partial last stage."""
    check(1, 16, 1050, 1050, 64, torch.float32, f32_rel(1050, 64))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [40, 48, 56, 72, 80, 96, 104, 120, 36])
@pytest.mark.parametrize("Sq,Sk", [(333, 333), (64, 300), (129, 77), (520, 130)])
def test_16_bit_head_dims_between_the_tile_widths(Sq, Sk, D, dt):
    """D % 8 == 0: the direct-to-LDS kernels with masked columns; 36: the general kernel."""
    check(1, 3, Sq, Sk, D, dt, REL16[dt])


@pytest.mark.parametrize("D", [40, 64, 80, 128])
@pytest.mark.parametrize("B,H,Sq,Sk", [(1, 4, 1024, 77), (2, 3, 2048, 8), (1, 2, 1000, 200), (1, 1, 700, 64), (1, 2, 1500, 100), (1, 8, 640, 513), (1, 1, 513, 2)])
def test_few_keys_share_out_the_queries(B, H, Sq, Sk, D):
    """dK / dV of few key blocks: the query stages (whole and partial last) go to several workgroups per block.
    (With one key dq and dk are exactly 0 and have no relative error; two keys is the smallest case here.)"""
    check(B, H, Sq, Sk, D, torch.float16, REL16[torch.float16])


@pytest.mark.parametrize("pad,offset", [(8, 8), (4, 4), (5, 3)])
def test_16_bit_alignments(pad, offset):
    check(1, 2, 300, 200, 80, torch.float16, REL16[torch.float16], pad, offset)


@pytest.mark.parametrize("dt,B,H,D", [(torch.float32, 4097, 4096, 1), (torch.float16, 2049, 4096, 40)])
def test_more_workgroups_than_one_launch_holds(dt, B, H, D):
    """More (batch, head) pairs than workgroups of 256 (f32) or 512 threads fit below 2^32 work items: kernels of fewer
    threads take them, and the last pairs are there as well.  One key: o = v, dv = do, dq = dk = 0."""
    q = torch.ones(1, dtype=dt, device=dev).expand(B * H * D).contiguous().view(B, H, 1, D).requires_grad_(True)
    v = torch.full((1,), 3.0, dtype=dt, device=dev).expand(B * H * D).contiguous().view(B, H, 1, D).requires_grad_(True)
    out = F.scaled_dot_product_attention(q, q, v)
    dq, dv = torch.autograd.grad(out, (q, v), v.detach())
    for t, want in ((out, 3.0), (dv, 3.0), (dq, 0.0)):
        for i in (0, 2047, B - 2, B - 1):
            assert torch.equal(t[i].detach().cpu(), torch.full((H, 1, D), want, dtype=dt)), (i, want)


@pytest.mark.parametrize("D,dt", [(40, torch.bfloat16), (56, torch.float16), (80, torch.float16), (96, torch.bfloat16), (120, torch.float16),
                                  (64, torch.float32), (80, torch.float32)])
@pytest.mark.parametrize("Sq,Sk", [(200, 300), (300, 200), (130, 130), (60, 50), (1100, 60)])
def test_infinities_and_nans_reach_their_column(Sq, Sk, D, dt):
    """An infinity or NaN of v (of the output's gradient) reaches its own column of o (of dv) and nothing else, also from
    a row that a partial last stage copies a second time and masks (zero times infinity would be NaN)."""
    g = torch.Generator().manual_seed(Sq + D)
    q, k, v, go = (torch.randn((1, 2, s, D), generator=g).to(dt) for s in (Sq, Sk, Sk, Sq))
    for s, t in ((Sk, v), (Sq, go)):
        t[0, 0, s - 5, 3] = float("inf")
        t[0, 1, s // 2, D - 1] = float("nan")
        if s > 128:
            t[0, 0, (s - 1) // 128 * 128 - 3, 7] = -float("inf")  # in the stage before the last
    leaves = [t.to(dev).requires_grad_(True) for t in (q, k, v)]
    o = F.scaled_dot_product_attention(*leaves)
    dv = torch.autograd.grad(o, leaves, go.to(dev))[2]
    P = torch.softmax(q.double() @ k.double().transpose(-1, -2) / math.sqrt(D), -1)
    for got, want in ((o, P @ v.double()), (dv, P.transpose(-1, -2) @ go.double())):
        got = got.detach().cpu()
        for f in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(f(got), f(want)), f
