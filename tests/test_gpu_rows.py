"""The small-workgroup kernel (ta_fwd_rows_*: short rows on grids of more than one 128-row block
per CU) against the oracle: one row, one key past a tile, one row past a block, whole tiles
and blocks, rows that end inside a wave, head dims padded in place, every layout, outliers
that move the running max between tiles, and non-finite keys."""

from __future__ import annotations

import numpy as np
import pytest

from tests.parity_util import TOL, as_f32, check_close, inputs, knobs, oracle_f32, say

pytestmark = pytest.mark.gpu


def _on_gpu(t3, layout):
    import torch

    dev = torch.device("cuda:0")
    if layout == "packed":  # slices of one [B, S, 3, H, D] projection
        p = torch.stack([t.transpose(1, 2) for t in t3], dim=2).contiguous().to(dev)
        return [p[:, :, i].transpose(1, 2) for i in range(3)]
    if layout == "bshd":
        return [t.transpose(1, 2).contiguous().to(dev).transpose(1, 2) for t in t3]
    return [t.to(dev) for t in t3]


def _run(t3, causal, layout="bhsd"):
    import torch

    from tiledattention import sdpa
    from tiledattention.kernels import flash_fwd

    args = _on_gpu(t3, layout)
    desc = flash_fwd.describe_call(*args, causal=causal)
    assert desc["kernel"].startswith("ta_fwd_rows_"), desc
    say(f"{desc['kernel']} {tuple(args[0].shape)} {layout}")
    out = sdpa(*args, causal=causal)
    torch.cuda.synchronize()
    return as_f32(out)


@pytest.mark.parametrize("shape,causal,dtype,layout", [
    ((33, 8, 1, 64), True, "float16", "bhsd"),
    ((33, 8, 64, 64), False, "bfloat16", "packed"),
    ((33, 8, 65, 96), True, "bfloat16", "bshd"),
    ((33, 8, 128, 160), False, "float16", "bhsd"),   # whole tiles and blocks: no tail masks
    ((17, 8, 129, 128), False, "float16", "packed"),
    ((17, 8, 197, 64), False, "float16", "packed"),
    ((17, 8, 200, 160), True, "bfloat16", "bhsd"),
    ((17, 8, 256, 96), False, "float16", "packed"),
    ((17, 8, 256, 64), True, "bfloat16", "bhsd"),
    ((17, 8, 225, 40), True, "float16", "bhsd"),     # padded in place to 64
    ((17, 8, 193, 72), False, "bfloat16", "bshd"),   # ... to 96
    ((17, 8, 250, 112), True, "bfloat16", "packed"), # ... to 128
    ((17, 8, 161, 136), False, "float16", "bhsd"),   # ... to 160
    ((17, 8, 150, 100), False, "bfloat16", "bhsd"),  # padded on the host
])
def test_rows_against_the_oracle(gpu, shape, causal, dtype, layout):
    t3 = inputs(shape, dtype, 700 + shape[2] + shape[3])
    ref = oracle_f32(*t3, causal=causal)
    check_close(_run(t3, causal, layout), ref, dtype, tol=TOL[dtype], what=f"rows {shape} {layout}")


@pytest.mark.parametrize("d", [64, 128])
def test_rows_rescale_between_tiles(gpu, d):
    """Keys whose size grows tile by tile raise each row's max past the rescale threshold."""
    import torch

    q, k, v = inputs((33, 8, 256, d), "bfloat16", 81 + d)
    k = (k.float() * torch.linspace(0.1, 12.0, 256)[None, None, :, None]).to(k.dtype)
    ref = oracle_f32(q, k, v, causal=False)
    # nearly one-hot rows: P's rounding (u = 2^-8) moves O by up to 3 u max|v|
    tol = 3 * 2.0 ** -8 * float(v.float().abs().max())
    check_close(_run((q, k, v), False), ref, "bfloat16", tol=tol, what=f"rows rescale D={d}")


def _error_against_64_bits(args, causal):
    """(rows kernel, eight-wave kernel): 2-norm of the error over 2-norm of the exact result."""
    import torch

    from tiledattention import sdpa
    from tiledattention.kernels import flash_fwd

    q, k, v = (t.flatten(0, 1).double() for t in args)
    kt = k.transpose(1, 2).contiguous()
    scores = torch.matmul(q * q.shape[-1] ** -0.5, kt)
    if causal:
        scores.masked_fill_(torch.ones_like(scores[0], dtype=torch.bool).triu(1), float("-inf"))
    exact = torch.matmul(torch.softmax(scores, dim=-1), v)
    errors = []
    for sched, family in ((None, "ta_fwd_rows_"), (3, "ta_fwd_pp_")):  # order 3 keeps the eight-wave kernel
        with knobs(sched=sched):
            assert flash_fwd.describe_call(*args, causal=causal)["kernel"].startswith(family)
            out = sdpa(*args, causal=causal).flatten(0, 1).double()
        errors.append(float((out - exact).norm() / exact.norm()))
    return errors


@pytest.mark.parametrize("shape,causal,dtype", [
    ((40, 8, 70, 64), False, "float16"),
    ((40, 8, 96, 128), False, "bfloat16"),
    ((40, 8, 113, 160), False, "float16"),
    ((40, 8, 128, 64), False, "bfloat16"),
    ((40, 8, 131, 96), False, "bfloat16"),
    ((40, 8, 128, 96), True, "float16"),
    ((40, 8, 150, 64), True, "bfloat16"),
    ((40, 8, 192, 128), True, "float16"),
    ((40, 8, 256, 64), False, "float16"),
])
def test_rows_error_no_larger_than_the_eight_wave_kernels(gpu, shape, causal, dtype):
    """Rows of one to four key tiles.  Rounding P dominates the error; over more than 10^6
    outputs the ratio of two such errors scatters by about 10^-3 (1 / sqrt of their number)."""
    args = _on_gpu(inputs(shape, dtype, 1700 + shape[2]), "bhsd")
    say(f"rows error against 64 bits {shape} causal={causal} {dtype}")
    rows, eight = _error_against_64_bits(args, causal)
    print(f"[check] rows {rows:.4e} eight-wave {eight:.4e} ratio {rows / eight:.4f}", flush=True)
    assert rows <= 1.001 * eight


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
def test_rows_falling_maxima(gpu, dtype):
    """Keys that shrink tile by tile: every tile's max lies far below the one before."""
    import torch

    q, k, v = inputs((33, 8, 256, 64), dtype, 83)
    k = (k.float() * torch.tensor([8.0, 2.0, 0.25, 0.0])[torch.arange(256) // 64][None, None, :, None]).to(k.dtype)
    ref = oracle_f32(q, k, v, causal=True)
    # nearly one-hot rows, as above: P's rounding u moves O by up to 3 u max|v|
    u = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -11
    check_close(_run((q, k, v), True), ref, dtype, tol=3 * u * float(v.float().abs().max()), what="rows falling maxima")


@pytest.mark.parametrize("causal", [False, True])
def test_rows_large_values_with_falling_maxima(gpu, causal):
    """Values near the top of bf16's range, and keys whose tiles' maxima fall: what is kept while
    the reference point follows them stays finite."""
    import torch

    q, k, v = inputs((33, 8, 192, 64), "bfloat16", 84)
    step = torch.tensor([4.0, 2.0, 0.0])[torch.arange(192) // 64]
    q = (q.float().abs() * 0.25 + 0.5).to(q.dtype)
    k = (0.25 * k.float() + step[None, None, :, None]).to(k.dtype)
    v = (v.float().clamp(-2.0, 2.0) * 2.0 ** 118).to(v.dtype)
    ref = oracle_f32(q, k, v, causal=causal) * 2.0 ** -118
    assert np.isfinite(ref).all()
    got = _run((q, k, v), causal) * np.float32(2.0 ** -118)
    # P's rounding u = 2^-8, as above
    check_close(got, ref, "bfloat16", tol=3 * 2.0 ** -8 * 2.0, what=f"rows large values causal={causal}")


@pytest.mark.parametrize("value", [float("nan"), float("-inf")])
def test_rows_nonfinite_keys(gpu, value):
    """A NaN key poisons every row of its head; a key whose scores are -inf or +inf by the
    sign of q's column poisons the rows where they are +inf (inf - inf) and no others."""
    q, k, v = inputs((33, 8, 150, 64), "bfloat16", 5)
    k = k.clone()
    k[0, 1, 3, 7] = value
    with np.errstate(invalid="ignore", over="ignore"):
        ref = oracle_f32(q, k, v, causal=False)
    got = _run((q, k, v), False)
    assert (np.isnan(got) == np.isnan(ref)).all() and np.isnan(ref).any()
    fin = np.isfinite(ref)
    assert np.isfinite(got[fin]).all()
    assert float(np.abs(got[fin] - ref[fin]).max()) <= TOL["bfloat16"]


@pytest.mark.parametrize("shape,causal,dtype,tile_n,layout", [
    ((33, 8, 64, 64), False, "float16", 64, "packed"),     # one tile: the second slice empty
    ((33, 8, 65, 128), True, "bfloat16", 64, "bhsd"),
    ((33, 8, 128, 128), False, "float16", 128, "bhsd"),    # whole tiles and blocks
    ((17, 8, 200, 64), True, "bfloat16", 128, "bshd"),
    ((17, 8, 384, 64), False, "bfloat16", 64, "bhsd"),
    ((17, 8, 321, 40), False, "float16", 64, "bhsd"),      # padded in place to 64
    ((17, 8, 250, 112), True, "float16", 128, "packed"),   # ... to 128
])
def test_rows_input_dtype_accumulation(gpu, shape, causal, dtype, tile_n, layout):
    """Against the oracle's restatement of the rounding sequence at the fp32 tolerance, as the
    eight-wave kernel's results are (each tile's rounding is at most half an ulp of a partial
    sum whose weights add up to at most the row's)."""
    import torch

    from oracle import oracle as O
    from tiledattention import torch_op  # noqa: F401  (registers the operator)
    from tiledattention.kernels import flash_fwd

    t3 = inputs(shape, dtype, 900 + shape[2])
    code = O.FP16 if dtype == "float16" else O.BF16
    bits = O.flash_tiled(*(O.to_bits(t) for t in t3), code, causal=causal, tile_m=128, tile_n=tile_n, accum_lowp=True)
    ref = O.upcast(bits, code)
    args = _on_gpu(t3, layout)
    desc = flash_fwd.describe_call(*args, causal=causal, tile=(128, tile_n), accum="fp16")
    assert desc["kernel"].startswith(f"ta_fwd_rowsl_n{tile_n}_"), desc
    say(f"{desc['kernel']} {shape} {layout}")
    out = torch.ops.tiledattention.sdpa_fwd(*args, causal, None, 128, tile_n, 1)
    torch.cuda.synchronize()
    check_close(as_f32(out), ref, dtype, tol=TOL[dtype], what=f"rowsl {shape} {layout}")
