"""Operators whose workspace or intermediates are freed before a recorded graph is replayed: every replay gives the
eager result bit for bit, and leaves tensors alone that were allocated after the recording."""

import pytest
import torch
import torch.nn.functional as F

import torch_vulkan
from torch_vulkan import abi

pytestmark = pytest.mark.gpu
dev = torch.device("vk")


def randn(*shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=torch.Generator().manual_seed(sum(shape))).to(dtype).to(dev)


def mm_bf16():
    a, b = randn(604, 5192), randn(5192, 704)
    return lambda: a @ b


def mm_f32():
    a, b = randn(128, 4096, dtype=torch.float32), randn(4096, 128, dtype=torch.float32)
    return lambda: a @ b


def int8_few_rows():
    x, s = randn(16, 2048), randn(8192, 32).abs()
    q = torch.randint(-127, 128, (8192, 2048), generator=torch.Generator().manual_seed(1), dtype=torch.int8).to(dev)
    return lambda: torch_vulkan.dequant_int8_linear(x, q, s)


def dkdv_few_keys():
    q, k, v = (randn(1, 4, s, 128, dtype=torch.float16) for s in (2048, 77, 77))
    go = randn(1, 4, 2048, 128, dtype=torch.float16)
    fwd = torch.ops.aten._scaled_dot_product_fused_attention_overrideable
    bwd = torch.ops.aten._scaled_dot_product_fused_attention_overrideable_backward
    r = fwd(q, k, v)
    z = torch.zeros((), dtype=torch.long)
    return lambda: torch.cat([t.flatten() for t in bwd(go, q, k, v, None, [True, True, True, False], r[0], r[1], r[2], r[3], 2048, 77, 0.0, False, z, z)[:3]])


def conv_ragged():
    x, w = randn(1, 512, 64, 72), randn(128, 512, 3, 3)
    return lambda: F.conv2d(x, w, padding=1)


@pytest.mark.parametrize("make", [mm_bf16, mm_f32, int8_few_rows, dkdv_few_keys, conv_ragged])
def test_replays_and_later_tensors(make):
    rt, out = abi.Runtime(), {}
    run = make()
    eager = run()
    left_out = torch_vulkan.workspaces_left_out()
    want = eager.cpu()
    blocks = torch_vulkan.live_blocks()

    def record():
        out["y"] = run()

    gid = rt.graph(record)
    assert torch_vulkan.workspaces_left_out() == left_out and torch_vulkan.live_blocks() == blocks + 1
    # everything that fits where the recording's memory was
    later = [torch.full((n,), 7, dtype=torch.uint8, device=dev) for n in (1 << 23, 1 << 22, 1 << 20, 1 << 18, 1 << 16, 1 << 12) for _ in range(4)]
    for _ in range(3):
        out["y"].zero_()
        rt.graph_launch(gid)
        assert torch.equal(out["y"].cpu(), want)
        assert torch.equal(run().cpu(), want)  # eager work between the replays
        overwritten = [t.numel() for t in later if not torch.equal(t.cpu(), torch.full((t.numel(),), 7, dtype=torch.uint8))]
        assert not overwritten
    rt.graph_destroy(gid)
