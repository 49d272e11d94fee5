"""The masked copies of the direct-to-LDS kernels as the compiler builds them: one instruction each.  A buffer resource
that it cannot prove the same for all lanes makes it wrap every copy in a loop over the lanes (four readfirstlane, two
compares and a branch a copy, between the matrix instructions).  Compiles instances that were built so."""

import os
import re
import subprocess
import sys

import pytest

from conftest import PKG

sys.path.insert(0, PKG)
import build  # noqa: E402

SOURCE = """
#include "gemm_dma_kernel.h"
namespace hk {
void instances() {
#define INSTANCE(...) hipLaunchKernelGGL((mm_dma<__VA_ARGS__>), dim3(1), dim3(512), 0, 0, hrt_mm_args{}, 1, 1, 0, 0, 0, 0)
  INSTANCE(BF16, 256, 256, 64, 128, false, true, false, 2, false, true);
  INSTANCE(F16, 64, 128, 32, 64, true, true, false, 3, true, true);
  INSTANCE(BF16, 128, 128, 32, 64, false, false, true, 3, false, true);
}
}
"""


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="needs hipcc")
def test_masked_copies_are_single_instructions(tmp_path):
    src, asm = tmp_path / "edge.hip", tmp_path / "edge.asm"
    src.write_text(SOURCE)
    flags = [f for f in build.HIP_FLAGS if f != "-Wall"]
    subprocess.run([build.HIPCC, *flags, "-I", os.path.join(build.CSRC, "kernels"), "-x", "hip", "--cuda-device-only", "-S", str(src),
                    "-o", str(asm)], check=True, capture_output=True)
    lines = [x.split(";")[0].strip() for x in asm.read_text().splitlines()]
    lines = [x for x in lines if x]
    copies = [i for i, x in enumerate(lines) if re.match(r"buffer_load_dwordx4 .*\blds\b", x)]
    assert len(copies) >= 60
    looped = [i for i in copies if any("s_xor_b64 exec, exec" in x for x in lines[i + 1 : i + 4])]
    assert not looped, f"{len(looped)} of {len(copies)} copies inside a loop over lanes"
