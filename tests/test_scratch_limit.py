"""Operators whose workspace only makes them faster, with device memory for their results but not for the workspace:
they run without it and say so.  The answer differs by the order of fp32 sums and one rounding of the result, so both are within
one unit in the last place of each other in relative L2 (2^-8 bf16, 2^-11 f16; f32: 2^-24 (sqrt(K) + 2))."""

import math

import pytest
import torch
import torch.nn.functional as F

import torch_vulkan

pytestmark = pytest.mark.gpu
dev = torch.device("vk")
MB = 1 << 20


def randn(*shape, dtype):
    return torch.randn(shape, generator=torch.Generator().manual_seed(sum(shape))).to(dtype).to(dev)


def mm_bf16():
    a, b = randn(1024, 8192, dtype=torch.bfloat16), randn(8192, 2048, dtype=torch.bfloat16)
    return lambda: (a @ b,)


def mm_f32():
    a, b = randn(256, 8192, dtype=torch.float32), randn(8192, 512, dtype=torch.float32)
    return lambda: (a @ b,)


def few_keys():
    q, k, v = (randn(1, 4, s, 128, dtype=torch.float16).requires_grad_(True) for s in (2048, 77, 77))
    o, go = F.scaled_dot_product_attention(q, k, v), randn(1, 4, 2048, 128, dtype=torch.float16)
    return lambda: torch.autograd.grad(o, (k, v), go, retain_graph=True)


def int8_few_rows():
    x = randn(16, 2048, dtype=torch.bfloat16)
    q = torch.randint(-127, 128, (8192, 2048), generator=torch.Generator().manual_seed(1), dtype=torch.int8).to(dev)
    s = randn(8192, 32, dtype=torch.bfloat16).abs()
    return lambda: (torch_vulkan.dequant_int8_linear(x, q, s),)


def conv_few_tiles():
    x, w = randn(1, 512, 64, 72, dtype=torch.bfloat16), randn(128, 512, 3, 3, dtype=torch.bfloat16)
    return lambda: (F.conv2d(x, w, padding=1),)


@pytest.mark.parametrize("make,room_mb,rel", [(mm_bf16, 5, 2.0**-8), (mm_f32, 1, 2.0**-24 * (math.sqrt(8192) + 2)),
                                              (few_keys, 3, 2.0**-11), (int8_few_rows, 1, 2.0**-8), (conv_few_tiles, 3, 2.0**-8)])
def test_runs_without_room_for_the_workspace(make, room_mb, rel):
    torch_vulkan.set_fused_attention("on")
    try:
        run = make()
        want = [t.cpu() for t in run()]
        torch.vk.synchronize()
        room = torch.empty(room_mb * MB, dtype=torch.uint8, device=dev)
        torch.vk.set_memory_limit(1)  # no new reservations; the slabs that are there are filled up below
        fill = []
        for size in (16 * MB, MB, MB // 16):
            while True:
                try:
                    fill.append(torch.empty(size, dtype=torch.uint8, device=dev))
                except RuntimeError:
                    break
        del room
        with pytest.raises(RuntimeError):
            torch.empty((room_mb + 1) * MB, dtype=torch.uint8, device=dev)
        left_out, slabs = torch_vulkan.workspaces_left_out(), torch_vulkan.slab_count()
        got = run()
        torch.vk.synchronize()
        assert torch_vulkan.workspaces_left_out() == left_out + 1  # it did run without
        assert torch_vulkan.slab_count() == slabs  # and gave nothing back to the driver for it
    finally:
        torch.vk.set_memory_limit(0)
        torch_vulkan.set_fused_attention("auto")
    for a, b in zip(got, want):
        a, b = a.cpu().double(), b.double()
        assert ((a - b).norm() / b.norm()).item() <= rel
