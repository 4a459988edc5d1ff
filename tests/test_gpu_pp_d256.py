"""The eight-wave kernel at D = 256 (64-key steps, 128-row blocks) against the oracle: one key
more than a step, ragged and whole last steps and blocks, causal and not, [B, S, H, D] views,
head dims padded to 256 on the host, and rows below its rule on the four-wave kernel."""

from __future__ import annotations

import pytest

from tests.parity_util import TOL, as_f32, check_close, inputs, oracle_f32, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,causal,dtype,bshd", [
    ((2, 4, 65, 256), True, "float16", False),     # one key into the second step
    ((2, 4, 128, 256), False, "bfloat16", True),   # the whole-step variant, one block
    ((1, 3, 320, 256), True, "bfloat16", False),   # whole steps, half a last block
    ((2, 2, 449, 256), False, "float16", True),    # one key and one row over
    ((1, 2, 640, 256), True, "float16", False),    # five whole blocks
    ((1, 1, 600, 256), False, "bfloat16", False),  # one head, five blocks, the last ragged
    ((1, 4, 193, 200), True, "bfloat16", False),   # padded to 256 on the host
])
def test_eight_wave_d256(gpu, shape, causal, dtype, bshd):
    import torch

    from tiledattention import sdpa
    from tiledattention.kernels import flash_fwd

    q, k, v = inputs(shape, dtype, 256 + shape[2])
    ref = oracle_f32(q, k, v, causal=causal)
    dev = torch.device("cuda:0")
    args = [t.transpose(1, 2).contiguous().to(dev).transpose(1, 2) if bshd else t.to(dev) for t in (q, k, v)]
    say(f"eight-wave D=256 {dtype} {shape} causal={causal} bshd={bshd}")
    desc = flash_fwd.describe_call(*args, causal=causal)
    assert desc["kernel"].startswith("ta_fwd_pp_") and "_d256_" in desc["kernel"], desc
    out = sdpa(*args, causal=causal)
    torch.cuda.synchronize()
    check_close(as_f32(out), ref, dtype, tol=TOL[dtype], what=f"eight-wave D=256 {shape}")


def test_rule_keeps_one_step_and_one_small_head_on_the_four_wave_kernel(gpu):
    import torch

    from tiledattention.kernels import flash_fwd

    for shape in ((2, 4, 64, 256), (1, 1, 512, 256)):
        q, k, v = (t.to("cuda:0") for t in inputs(shape, "float16", 1))
        desc = flash_fwd.describe_call(q, k, v, causal=True)
        assert desc["kernel"] == "ta_fwd_f16_d256_m128_n64_c1_t%d_a0" % (shape[2] % 128 != 0), desc
    torch.cuda.synchronize()
