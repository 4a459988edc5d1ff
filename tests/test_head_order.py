"""The order in which a causal grid's heads share an XCD (FwdParams::head_group): the grouped
numbering over heads, blocks and group sizes on the host, and on the GPU the kernels that use
it against the oracle, with equal groups, an uneven last one and a partial last block."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

from tests.parity_util import TOL, as_f32, check_close, inputs, oracle_f32, say

ROOT = Path(__file__).resolve().parent.parent


def test_grouped_numbering_covers_every_block_once(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "head_order_check"
    subprocess.run(
        [gxx, "-O1", "-std=c++17", "-Wall", "-Werror", f"-I{ROOT / 'tiledattention_amd' / 'csrc'}",
         "-o", str(exe), str(ROOT / "tests" / "native" / "head_order_check.cpp")],
        check=True, capture_output=True, text=True,
    )
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout[-2000:]
    assert res.stdout.startswith("ok ")


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype", [
    ((1, 40, 1000, 128), "bfloat16"),  # five heads an XCD
    ((1, 48, 1024, 160), "float16"),   # six
    ((11, 8, 640, 64), "bfloat16"),    # eleven, an odd number of blocks
    ((8, 16, 1025, 256), "float16"),   # sixteen of nine blocks
])
def test_grouped_heads_against_the_oracle(gpu, shape, dtype):
    import torch

    from tiledattention import sdpa
    from tiledattention.kernels import flash_fwd

    t3 = inputs(shape, dtype, 900 + shape[2])
    args = [t.cuda() for t in t3]
    say(f"{flash_fwd.describe_call(*args, causal=True)['kernel']} {shape}")
    out = sdpa(*args, causal=True)
    torch.cuda.synchronize()
    check_close(as_f32(out), oracle_f32(*t3, causal=True), dtype, tol=TOL[dtype], what=f"head order {shape}")
