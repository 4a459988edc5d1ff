"""The order in which a causal grid's heads share an XCD (FwdParams::head_group): the grouped
numbering over heads, blocks and group sizes on the host, and on the GPU every kernel family
that uses it against the oracle, with one group, equal groups, an uneven last one and a partial
last block, each with the group that the library reports."""

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


def _group(args, causal=True, **kw):
    """(kernel, heads an XCD takes at a time) of the call's launch on a device of 256 CUs."""
    import torch

    from tiledattention import _lib, _runtime
    from tiledattention.kernels import flash_fwd

    plan = flash_fwd._plan_for(torch, *args, causal, kw.get("tile"), kw.get("accum"))
    lib = _runtime.get_native_library()
    return _lib.describe(lib, plan.args, plan.chunk).kernel.decode(), _lib.head_group(lib, plan.args, 256)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype,kernel,group", [
    ((1, 40, 1000, 128), "bfloat16", "ta_fwd_pp_bf16_d128", 5),    # five heads an XCD, one group
    ((1, 48, 1024, 160), "float16", "ta_fwd_pp_f16_d160", 6),      # six
    ((11, 8, 640, 64), "bfloat16", "ta_fwd_rows_", 0),             # eleven of five blocks: one by one
    ((8, 16, 1025, 256), "float16", "ta_fwd_pp_f16_d256", 4),      # sixteen of nine blocks, four groups
    ((7, 8, 1100, 256), "bfloat16", "ta_fwd_pp_bf16_d256", 4),     # seven: 4 + 3, a partial last block
    ((16, 8, 512, 64), "bfloat16", "ta_fwd_rows_", 8),             # small workgroups: 8 + 8
    ((9, 8, 1000, 64), "float16", "ta_fwd_rows_", 9),              # nine, one group
    ((15, 8, 500, 96), "bfloat16", "ta_fwd_rows_", 15),            # fifteen, one group
    ((13, 8, 640, 128), "bfloat16", "ta_fwd_rows_", 13),           # thirteen, more blocks than resident
    ((10, 8, 896, 160), "float16", "ta_fwd_rows_", 10),            # ten, one group
])
def test_grouped_heads_against_the_oracle(gpu, shape, dtype, kernel, group):
    import torch

    from tiledattention import sdpa

    t3 = inputs(shape, dtype, 900 + shape[2])
    args = [t.cuda() for t in t3]
    name, heads = _group(args)
    assert name.startswith(kernel) and heads == group, (name, heads)
    say(f"{name} {shape} group {heads}")
    out = sdpa(*args, causal=True)
    torch.cuda.synchronize()
    check_close(as_f32(out), oracle_f32(*t3, causal=True), dtype, tol=TOL[dtype], what=f"head order {shape}")


@pytest.mark.gpu
@pytest.mark.parametrize("shape,tile_n,group", [((16, 8, 512, 64), 64, 8), ((11, 8, 512, 128), 128, 11), ((7, 8, 768, 64), 128, 7)])
def test_grouped_heads_input_dtype(gpu, shape, tile_n, group):
    import torch

    from oracle import oracle as O
    from tiledattention import torch_op  # noqa: F401  (registers the operator)

    t3 = inputs(shape, "float16", 950 + shape[2])
    args = [t.cuda() for t in t3]
    name, heads = _group(args, tile=(128, tile_n), accum="fp16")
    assert name.startswith(f"ta_fwd_rowsl_n{tile_n}_") and heads == group, (name, heads)
    say(f"{name} {shape} group {heads}")
    out = torch.ops.tiledattention.sdpa_fwd(*args, True, None, 128, tile_n, 1)
    torch.cuda.synchronize()
    bits = O.flash_tiled(*(O.to_bits(t) for t in t3), O.FP16, causal=True, tile_m=128, tile_n=tile_n, accum_lowp=True)
    check_close(as_f32(out), O.upcast(bits, O.FP16), "float16", tol=TOL["float16"], what=f"head order {shape}")
