"""Seeded randomised GPU parity: 40 configurations drawn from one fixed generator, each
against the explicit fp32 attention of the CPU oracle.

Draws whose logits spread like N(0, 1) inputs' (standard deviation of scale * q.k up to
6) are held to the oracle tolerance (2e-3 fp16, 1e-2 bf16; the input-dtype
accumulation bound for ``ACCUM_MODE=fp16``), scaled by the input magnitude.  Sharper draws
(inputs x2 with scale 0.3: a nearly one-hot softmax) are dominated by the rounding of P to
the input dtype, which the reference's algorithm performs too: with unit roundoff u
(2^-8 bf16, 2^-11 fp16), each p_j carries a relative error of at most u, so
O = sum p_j v_j / sum p_j moves by at most u * max |v_j - O| <= 2u max|v|, and rounding O
adds u |O| <= u max|v|; accumulating in the input dtype adds u max|v| per key tile.  Those
draws are held to that bound.

Every draw picks B, H, S (ragged included), a head dim (native, narrower multiples of 8 run
in place, others padded on the host), dtype, causal, scale, input magnitude, a memory
layout ([B,H,S,D] or a [B,S,H,D] view), and the knobs: the default tile or one of the four
tiles, fp32 or input-dtype accumulation, and split key ranges off / auto / forced.  Sizes
keep the oracle at a few seconds in total.  Each case names itself before the GPU run."""

from __future__ import annotations

import random

import pytest

import math

import numpy as np

from tests.parity_util import LOWP_TOL, TOL, as_f32, check_close, inputs, knobs, oracle_f32, say

pytestmark = pytest.mark.gpu

_SEED = 20261201
_N = 40


def _draw(rng: random.Random) -> dict:
    d = rng.choice([64, 128, 64, 128, 160, 256, 96, 48, 72, 120, 100, 200, 8])
    s = rng.choice([1, 7, 64, 127, 128, 129, 255, 300, 511, 640, 1000, 1100])
    b, h = rng.choice([(1, 1), (1, 3), (2, 2), (1, 5), (2, 4)])
    tile = rng.choice([None, None, None, (64, 64), (64, 128), (128, 64), (128, 128)])
    if d > 128 and tile is not None and tile[1] != 64:
        tile = (tile[0], 64)  # head dims above 128 need 64-key tiles
    return dict(
        b=b, h=h, s=s, d=d,
        dtype=rng.choice(["float16", "bfloat16"]),
        causal=rng.random() < 0.5,
        scale=rng.choice([None, None, 0.05, 0.3]),
        mag=rng.choice([0.5, 1.0, 2.0]),
        bshd=rng.random() < 0.3,
        tile=tile,
        accum=rng.choice(["fp32", "fp32", "fp16"]),
        split=rng.choice(["off", "auto", "auto", 1, 2]),
        seed=rng.randrange(1 << 30),
    )


_CASES = [_draw(r) for r in [random.Random(_SEED)] for _ in range(_N)]


@pytest.mark.parametrize("case", _CASES, ids=[f"c{i}" for i in range(_N)])
def test_randomized_parity(gpu, case):
    import torch

    from tiledattention import sdpa

    c = case
    q, k, v = inputs((c["b"], c["h"], c["s"], c["d"]), c["dtype"], c["seed"], scale_inputs=c["mag"])
    scale = c["scale"] if c["scale"] is not None else 1.0 / math.sqrt(c["d"])
    spread = scale * c["mag"] ** 2 * math.sqrt(c["d"])  # std of the logits scale * q.k
    ref = oracle_f32(q, k, v, causal=c["causal"], scale=c["scale"])
    env = {"accum_mode": c["accum"]}
    if c["tile"] is not None:
        env["tile_m"], env["tile_n"] = c["tile"]
    eight_wave = (c["tile"] in (None, (128, 64))) and c["accum"] == "fp32" and c["d"] <= 128
    if c["split"] != "auto" and (c["split"] == "off" or eight_wave):
        env["split"] = c["split"]
    say(f"random {c} logit spread {spread:.1f}")
    dev = torch.device("cuda:0")
    if c["bshd"]:
        qd, kd, vd = (t.transpose(1, 2).contiguous().to(dev).transpose(1, 2) for t in (q, k, v))
    else:
        qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    with knobs(**env):
        out = sdpa(qd, kd, vd, causal=c["causal"], scale=c["scale"])
    torch.cuda.synchronize()
    assert out.shape == q.shape and out.dtype == q.dtype
    tol = (LOWP_TOL if c["accum"] == "fp16" else TOL)[c["dtype"]] * max(1.0, c["mag"])
    if spread > 6.0:
        u = 2.0 ** -8 if c["dtype"] == "bfloat16" else 2.0 ** -11
        tiles = math.ceil(c["s"] / 64) if c["accum"] == "fp16" else 0
        vmax = float(np.abs(v.float().numpy()).max())
        tol = max(tol, (3 + tiles) * u * vmax)
    check_close(as_f32(out), ref, c["dtype"], tol=tol, what=f"random (logit spread {spread:.1f})")
