"""Rows behind a ragged tail: q, k and v are the first S rows of longer buffers whose other
rows are NaN.  The last key step reads past row S into the range check; a row that came
through would make the output NaN (P is 0 there, and 0 x NaN is NaN)."""

from __future__ import annotations

import pytest

from tests.parity_util import TOL, as_f32, check_close, inputs, knobs, oracle_f32, say

pytestmark = pytest.mark.gpu


def _head_of_nan_buffers(t3, bshd):
    import torch

    out = []
    for t in t3:
        b, h, s, d = t.shape
        buf = torch.full((b, s + 200, h, d) if bshd else (b, h, s + 200, d), float("nan"), dtype=t.dtype, device="cuda:0")
        view = buf[:, :s].transpose(1, 2) if bshd else buf[:, :, :s]
        view.copy_(t)
        out.append(view)
    return out


@pytest.mark.parametrize("bshd", [False, True])
@pytest.mark.parametrize("shape,causal,dtype,tile,kernel", [
    # the eight-wave kernel at D = 256: part of a chunk row group, of a wave's half, of a block
    ((2, 4, 65, 256), False, "float16", None, "ta_fwd_pp_f16_d256"),
    ((2, 4, 193, 256), True, "bfloat16", None, "ta_fwd_pp_bf16_d256"),
    ((2, 2, 449, 256), False, "bfloat16", None, "ta_fwd_pp_bf16_d256"),
    ((1, 3, 250, 256), True, "float16", None, "ta_fwd_pp_f16_d256"),
    # the four-wave kernel at D = 256
    ((2, 4, 49, 256), False, "bfloat16", None, "ta_fwd_bf16_d256"),
    ((1, 2, 193, 256), True, "float16", (64, 64), "ta_fwd_f16_d256"),
    # the small workgroups: past a tile, past a block, an odd last tile
    ((33, 8, 65, 64), False, "bfloat16", None, "ta_fwd_rows_"),
    ((17, 8, 197, 128), False, "float16", None, "ta_fwd_rows_"),
    ((17, 8, 129, 96), True, "bfloat16", None, "ta_fwd_rows_"),
    ((17, 8, 250, 160), False, "float16", None, "ta_fwd_rows_"),
])
def test_nan_rows_behind_the_tail(gpu, shape, causal, dtype, tile, kernel, bshd):
    import torch

    from tiledattention import sdpa
    from tiledattention.kernels import flash_fwd

    t3 = inputs(shape, dtype, 40 + shape[2])
    ref = oracle_f32(*t3, causal=causal)
    args = _head_of_nan_buffers(t3, bshd)
    with knobs(**({} if tile is None else {"tile_m": tile[0], "tile_n": tile[1]})):
        desc = flash_fwd.describe_call(*args, causal=causal)
        assert desc["kernel"].startswith(kernel), desc
        say(f"NaN rows behind the tail {desc['kernel']} {shape} bshd={bshd}")
        out = sdpa(*args, causal=causal)
    torch.cuda.synchronize()
    check_close(as_f32(out), ref, dtype, tol=TOL[dtype], what=f"tail {shape}")


@pytest.mark.parametrize("shape,causal,tile_n", [((33, 8, 65, 64), False, 64), ((17, 8, 201, 128), True, 128)])
def test_nan_rows_behind_the_tail_input_dtype(gpu, shape, causal, tile_n):
    import torch

    from oracle import oracle as O
    from tiledattention import torch_op  # noqa: F401  (registers the operator)
    from tiledattention.kernels import flash_fwd

    t3 = inputs(shape, "float16", 50 + shape[2])
    bits = O.flash_tiled(*(O.to_bits(t) for t in t3), O.FP16, causal=causal, tile_m=128, tile_n=tile_n, accum_lowp=True)
    args = _head_of_nan_buffers(t3, False)
    desc = flash_fwd.describe_call(*args, causal=causal, tile=(128, tile_n), accum="fp16")
    assert desc["kernel"].startswith(f"ta_fwd_rowsl_n{tile_n}_"), desc
    say(f"NaN rows behind the tail {desc['kernel']} {shape}")
    out = torch.ops.tiledattention.sdpa_fwd(*args, causal, None, 128, tile_n, 1)
    torch.cuda.synchronize()
    check_close(as_f32(out), O.upcast(bits, O.FP16), "float16", tol=TOL["float16"], what=f"tail {shape}")
