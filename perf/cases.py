"""The work that callers have the SDPA forward do, as cases for timing and comparison.

Every case is one attention forward through a public entry point: ``tiledattention.sdpa``,
or the operator ``torch.ops.tiledattention.sdpa_fwd`` where a call chooses the accumulation
type.  The path has a forward only, so there is no backward to time.  The ranges the listed
cases stand for, and ``draw`` samples:

* sequence lengths 32 to 16384, multiples of the tiles and ragged ones;
* 1 to 1024 (batch, head) slices: one prompt on a few heads, batches of prompts, large
  batches of short rows;
* head dims 40 to 256: 64 and 128 above all, the chunked dims 96 and 160, 256, and narrower
  multiples of 8 that run in a wider kernel;
* fp16 and bf16, causal and not, fp32 accumulation and, now and then, input-dtype
  accumulation;
* [B, H, S, D] tensors, views of [B, S, H, D] tensors, and slices of one packed
  [B, S, 3, H, D] projection.

Inputs are N(0, 1), times 0.5 where the case says so, with a share of the keys' entries
times 20 where a case asks for outliers.
"""

from __future__ import annotations

import math

import torch

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}


def _case(name, b, h, s, d, dtype, causal, **kw):
    c = {"name": name, "b": b, "h": h, "s": s, "d": d, "dtype": dtype, "causal": causal,
         "layout": "bhsd", "accum": "fp32", "magnitude": 1.0, "outliers": 0.0}
    c.update(kw)
    return c


def listed():
    return [
        # The example workload: one call on next to no data, all launch and host time.
        _case("example_s64", 1, 2, 64, 64, "float16", True),
        # A short prompt on eight heads, the shortest of the causal sequence sweep.
        _case("prompt_s512", 1, 8, 512, 128, "bfloat16", True),
        # One non-causal sequence of ordinary length, fp16 D = 64.
        _case("encoder_s1024", 1, 8, 1024, 64, "float16", False),
        # A batch of short ragged rows, as an image encoder's patch tokens are, read from
        # the packed projection.
        _case("patches_s197", 32, 12, 197, 64, "float16", False, layout="packed"),
        # A batch of text-encoder rows.
        _case("batch_s512", 16, 16, 512, 64, "bfloat16", False, layout="bshd"),
        # A batch of prompts of a ragged length, heads interleaved.
        _case("prompts_s1500", 2, 16, 1500, 128, "bfloat16", True, layout="bshd"),
        # The chunked head dims of the study grid, one each way.
        _case("d96_s4096", 1, 8, 4096, 96, "float16", True),
        _case("d160_s2048", 1, 8, 2048, 160, "bfloat16", False),
        # The widest head dim.
        _case("d256_s4096", 1, 8, 4096, 256, "bfloat16", True, layout="bshd"),
        # The long causal sequence the forward is quoted on.
        _case("causal_s8192", 1, 8, 8192, 128, "bfloat16", True),
        # A batch of long non-causal rows: the largest case, and with input-dtype
        # accumulation as the accumulation option has it.
        _case("batch_s4096", 4, 16, 4096, 128, "float16", False, magnitude=0.5),
        _case("accum16_s4096", 2, 16, 4096, 64, "float16", False, accum="input", magnitude=0.5),
    ]


def draw(rng):
    d = rng.choice([64, 64, 64, 128, 128, 128, 96, 160, 256, rng.choice([40, 72, 80, 112, 192])])
    s = int(round(2.0 ** rng.uniform(5.0, 14.0)))
    if rng.random() < 0.5:
        s = max(32, s // 64 * 64)
    h = rng.choice([1, 2, 4, 8, 12, 16, 32])
    b = int(round(2.0 ** rng.uniform(0.0, 6.0)))
    accum = "input" if rng.random() < 0.1 else "fp32"
    # No dearer than the largest listed case, which runs the fastest kernel.
    cap = 5.0e11 if d <= 160 and accum == "fp32" else 1.2e11
    while b > 1 and (b * h > 1024 or 4.0 * b * h * s * s * d > cap):
        b //= 2
    while h > 1 and 4.0 * b * h * s * s * d > cap:
        h //= 2
    return {"b": b, "h": h, "s": s, "d": d, "dtype": rng.choice(["float16", "bfloat16"]),
            "causal": rng.random() < 0.5, "layout": rng.choice(["bhsd", "bshd", "packed"]),
            "accum": accum, "magnitude": rng.choice([1.0, 1.0, 0.5]),
            "outliers": 0.01 if rng.random() < 0.1 else 0.0}


def _inputs(case, seed):
    b, h, s, d = case["b"], case["h"], case["s"], case["d"]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    x = torch.randn((3, b, h, s, d), generator=g, device="cuda", dtype=torch.float32)
    x *= case["magnitude"]
    if case["outliers"]:
        x[1] *= torch.where(torch.rand((b, h, s, d), generator=g, device="cuda") < case["outliers"], 20.0, 1.0)
    x = x.to(_DTYPES[case["dtype"]])
    if case["layout"] == "packed":  # [B, S, 3, H, D]
        p = x.permute(1, 3, 0, 2, 4).contiguous()
        return tuple(p[:, :, i].transpose(1, 2) for i in range(3))
    if case["layout"] == "bshd":
        return tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in x)
    return tuple(t.clone() for t in x)


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    if case["accum"] == "input":
        import tiledattention.torch_op  # registers the operator
    else:
        from tiledattention import sdpa  # noqa: F401  (as a program's import does)
    return {"q": q, "k": k, "v": v, "causal": case["causal"], "accum": case["accum"]}


def run(state):
    if state["accum"] == "input":
        return torch.ops.tiledattention.sdpa_fwd(state["q"], state["k"], state["v"], state["causal"], None, 0, 0, 1)
    import tiledattention

    return tiledattention.sdpa(state["q"], state["k"], state["v"], causal=state["causal"])


def work(case):
    b, h, s, d = case["b"], case["h"], case["s"], case["d"]
    pairs = s * (s + 1) // 2 if case["causal"] else s * s
    return {"bytes": 4 * b * h * s * d * 2, "flops": 4 * b * h * pairs * d}


def tolerance(case):
    # Four times what the same path shows with its sums in another order (a row's keys in
    # two, four or eight slices), over the listed and 30 drawn cases: 2-norms up to 2.8e-3
    # bf16 and 3.6e-4 fp16, 1.1e-3 with fp16 accumulation (eight times that for bf16's
    # three bits fewer); largest differences 2.4e-2, 3.9e-3 and 8.6e-3.
    if case["accum"] == "input":
        return {"rel": 3.6e-2, "max": 0.28} if case["dtype"] == "bfloat16" else {"rel": 4.5e-3, "max": 0.035}
    return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bfloat16" else {"rel": 1.5e-3, "max": 0.016}


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    b, h, s, d = q.shape
    q, k, v = (t.reshape(b * h, s, d) for t in (q, k, v))
    out = torch.empty((b * h, s, d), dtype=torch.float64, device=q.device)
    rows = min(s, 2048)
    heads = max(1, (1 << 27) // (rows * s))
    scale = 1.0 / math.sqrt(d)
    keys = torch.arange(s, device=q.device)
    for i in range(0, b * h, heads):
        kt = k[i:i + heads].double().transpose(1, 2).contiguous()
        vd = v[i:i + heads].double()
        for r in range(0, s, rows):
            scores = torch.matmul(q[i:i + heads, r:r + rows].double() * scale, kt)
            if case["causal"]:
                scores.masked_fill_(keys > keys[r:r + rows, None], -math.inf)
            out[i:i + heads, r:r + rows] = torch.matmul(torch.softmax(scores, dim=-1), vd)
    return out.reshape(b, h, s, d)
