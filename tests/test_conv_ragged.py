"""The direct 3x3 convolution at rows and channels off its tiles (32 pixels x 4 rows x 128 channels), called through
the C ABI so that every case runs it, and convolutions through autograd whose forward or input gradient takes it,
against float64.  Inputs end right before NaNs, so an unmasked read shows.  Tolerance: products exact in fp32, fp32
sums, one rounding: relative L2 below half a unit in the last place (2^-9 bf16, 2^-12 f16) plus 1e-5."""

import pytest
import torch
import torch.nn.functional as F

import torch_vulkan
from torch_vulkan import abi

pytestmark = pytest.mark.gpu
dev = torch.device("vk")
REL = {torch.bfloat16: 2.0**-9 + 1e-5, torch.float16: 2.0**-12 + 1e-5}


def wr_elems(O, I):  # hrt_conv3r_wr_bytes / 2
    return abi.conv3_wr_bytes((O + 127) // 128 * 128, I) // 2


def in_nans(t):
    """t on vk, 16-byte aligned, with NaNs in front of and behind its memory."""
    flat = torch.full((t.numel() + 128,), float("nan"), dtype=t.dtype)
    flat[64 : 64 + t.numel()] = t.reshape(-1)
    return flat.to(dev)[64 : 64 + t.numel()].view(t.shape)


# (N, I, O, H, W): one short row, rows of 8 to 40 pixels around a segment, heights around 4, padded channel blocks
CASES = [(1, 16, 32, 1, 8), (2, 32, 160, 5, 24), (1, 64, 128, 4, 32), (1, 48, 192, 7, 40), (2, 80, 320, 3, 96), (1, 128, 96, 9, 72)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("flip", [0, 1])
@pytest.mark.parametrize("N,I,O,H,W", CASES)
def test_ragged_direct_convolution(N, I, O, H, W, flip, dt):
    g = torch.Generator().manual_seed(I + O + W)
    x = torch.randn((N, I, H, W), generator=g).to(dt)
    w = (torch.randn((I, O, 3, 3) if flip else (O, I, 3, 3), generator=g) * 0.1).to(dt)
    bias = torch.randn((O,), generator=g).to(dt)
    if flip:  # the input gradient of conv(., w) with w [I, O, 3, 3] at output gradient x
        ref = torch.nn.grad.conv2d_input((N, O, H, W), w.double(), x.double(), padding=1)
    else:
        ref = F.conv2d(x.double(), w.double(), padding=1)
    name = "bf16" if dt == torch.bfloat16 else "f16"
    rt = abi.Runtime()
    xd, wd, bd = in_nans(x), in_nans(w), bias.to(dev)
    wr = torch.full((wr_elems(O, I),), float("nan"), dtype=dt, device="cpu").to(dev)
    P = abi.Conv3WprepArgs()
    P.w, P.wr, P.O, P.I, P.flip = wd.data_ptr(), wr.data_ptr(), O, I, flip
    rt.dispatch("conv3x3r_wprep_" + name, P)
    for splits in [s for s in (1, 2) if (I // 16) % s == 0]:
        for has_bias in (0, 1):
            y = torch.full((N, O, H, W), float("nan"), dtype=dt).to(dev)
            ws = torch.full((splits * N * O * H * W,), float("nan")).to(dev)
            A = abi.Conv3Args()
            A.x, A.wr, A.y, A.ws, A.bias = xd.data_ptr(), wr.data_ptr(), y.data_ptr(), ws.data_ptr() if splits > 1 else 0, bd.data_ptr()
            A.N, A.I, A.O, A.H, A.W, A.has_bias, A.splits = N, I, O, H, W, has_bias, splits
            rt.dispatch("conv3x3r_" + name, A)
            want = ref + bias.double().view(1, -1, 1, 1) if has_bias else ref
            got = y.cpu().double()
            assert torch.isfinite(got).all()
            assert ((got - want).norm() / want.norm()).item() <= REL[dt], (splits, has_bias)
    bad = abi.Conv3Args.from_buffer_copy(A)
    bad.W = W + 4  # rows off 16-byte lines
    with pytest.raises(RuntimeError):
        rt.dispatch("conv3x3r_" + name, bad)


@pytest.mark.parametrize("N,C,Co,H,W", [(1, 512, 320, 96, 96), (2, 640, 128, 30, 72), (1, 320, 320, 64, 64), (1, 64, 100, 20, 36)])
def test_convolution_through_autograd(N, C, Co, H, W):
    """Forward with bias and every gradient, whichever path each takes (the last: unfolded, bias in the product)."""
    dt = torch.bfloat16
    g = torch.Generator().manual_seed(C)
    x, w, b = torch.randn((N, C, H, W), generator=g).to(dt), (torch.randn((Co, C, 3, 3), generator=g) * 0.02).to(dt), torch.randn((Co,), generator=g).to(dt)
    go = torch.randn((N, Co, H, W), generator=g).to(dt)
    leaves = [t.to(dev).requires_grad_(True) for t in (x, w, b)]
    out = F.conv2d(*leaves, padding=1)
    got = (out,) + torch.autograd.grad(out, leaves, go.to(dev))
    x64, w64, g64 = x.double(), w.double(), go.double()
    want = (F.conv2d(x64, w64, b.double(), padding=1), torch.nn.grad.conv2d_input(x.shape, w64, g64, padding=1),
            torch.nn.grad.conv2d_weight(x64, w.shape, g64, padding=1), g64.sum((0, 2, 3)))
    # unfolded input gradients round the column matrix too, batched weight gradients each image's: 2 more roundings
    for name, a, r in zip(("y", "dx", "dw", "db"), got, want):
        assert ((a.detach().cpu().double() - r).norm() / r.norm()).item() <= 2.5 * REL[dt], name
    assert not [k for k in torch_vulkan.fallback_counts() if "conv" in k]
