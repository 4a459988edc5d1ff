"""The library's own description of a launch (``ta_describe_launch_model``), on the CPU.

Every expectation below is written from the dispatch rules as the header states them
(include/tiledattn.h: ``sched``, ``TA_SPLIT_PAIRS``, ``ta_layout``), not from the
library's code: the kernel symbol per configuration, the layout (whole rows, causal pairs,
256-row blocks, split, paired split), its grid and the tail variant.  Every described
kernel must exist in the code object the description names, so the query cannot name a
kernel the launch would not find.  The launch entry points plan through the same function
(``plan_launch`` in csrc/tiledattn.cpp), so these tables pin what they launch too.
"""

from __future__ import annotations

import itertools

import pytest

from tiledattention import _lib
from tiledattention.kernels import flash_fwd as ff

CU = 256  # MI355X


@pytest.fixture(scope="module")
def lib():
    if not _lib.library_path().exists():
        pytest.fail("libtiledattn.so is not built: run __graft_entry__.build() first")
    return _lib.load()


@pytest.fixture(scope="module")
def objects():
    return {p.name: p.read_bytes() for p in _lib.code_object_paths()}


def _d(lib, chunk=0, cu=CU, **kw):
    return _lib.describe(lib, _lib.shape_args(**kw), chunk, compute_units=cu)


def _expected_symbol(*, dt, d, tm, tn, causal, tail, accum):
    """The whole-row kernel symbol for a configuration, from the families the code objects
    hold: eight-wave fp32 (128 rows: D <= 160; 64 rows: D 64/96/128/160), eight-wave
    input-dtype (D 64/128, one kernel per TILE_N), four-wave otherwise."""
    c, t = int(causal), int(tail)
    if accum == _lib.TA_ACC_FP32 and tm == 128 and d <= 160:
        return "attn_fwd_pp.hsaco", f"ta_fwd_pp_{dt}_d{d}_c{c}_t{t}"
    if accum == _lib.TA_ACC_FP32 and tm == 64 and d in (64, 96, 128, 160):
        return "attn_fwd_pp.hsaco", f"ta_fwd_pp64_{dt}_d{d}_c{c}_t{t}"
    if accum == _lib.TA_ACC_INPUT and d in (64, 128):
        fam = "ppl" if tm == 128 else "ppl64"
        return "attn_fwd_pp.hsaco", f"ta_fwd_{fam}_n{tn}_{dt}_d{d}_c{c}_t{t}"
    return f"attn_fwd_m{tm}_n{tn}.hsaco", f"ta_fwd_{dt}_d{d}_m{tm}_n{tn}_c{c}_t{t}_a{int(accum)}"


def _configs():
    for dtype, tiles, accum in itertools.product((_lib.TA_FP16, _lib.TA_BF16), _lib.TILE_SHAPES,
                                                 (_lib.TA_ACC_FP32, _lib.TA_ACC_INPUT)):
        for d in (64, 96, 128, 160, 256):
            if d == 96 and accum != _lib.TA_ACC_FP32:
                continue
            if d > 128 and tiles[1] != 64:
                continue
            yield dtype, tiles, accum, d


def _wide_rule(bh, s, d, cu=CU):
    """The wide kernel's rule for a whole-row 64-row tile with fp32 accumulation: D 64 or
    128, 32-row blocks in one round of the CUs, at most two passes (512 keys at D = 128,
    1024 at D = 64), or at most four on more than half the CUs."""
    grid = bh * -(-s // 32)
    passes = -(-s // (512 if d == 128 else 1024))
    return d in (64, 128) and grid <= cu and (passes <= 2 or (passes <= 4 and 2 * grid > cu))


@pytest.mark.parametrize("dtype,tiles,accum,d", list(_configs()))
def test_whole_row_kernel_per_configuration(lib, objects, dtype, tiles, accum, d):
    """One small head (B1 H1: no pairs, no 256-row blocks) at an aligned and a ragged S;
    the symbol and the tail variant follow the families, and the kernel exists.  64-row
    fp32 tiles at D = 64 / 128 run the wide kernel on such grids."""
    dt = "bf16" if dtype == _lib.TA_BF16 else "f16"
    tm, tn = tiles
    eight = (accum == _lib.TA_ACC_FP32 and ((tm == 128 and d <= 160) or (tm == 64 and d in (64, 96, 128, 160)))) \
        or (accum == _lib.TA_ACC_INPUT and d in (64, 128))
    for causal in (False, True):
        for s, aligned in ((512, 1), (512, 0), (320, 1), (300, 1)):
            step = 128 if eight else 1  # the eight-wave kernels step by 128 keys
            tail = not (aligned and s % tm == 0 and s % tn == 0 and s % step == 0)
            desc = _d(lib, S=s, D=d, dtype=dtype, tile_m=tm, tile_n=tn, accum=accum, causal=causal,
                      aligned=aligned)
            f, sym = _expected_symbol(dt=dt, d=d, tm=tm, tn=tn, causal=causal, tail=tail, accum=accum)
            wide = accum == _lib.TA_ACC_FP32 and tm == 64 and _wide_rule(1, s, d)
            if wide:
                f, sym = "attn_fwd_wide.hsaco", f"ta_fwd_wide_{dt}_d{d}_c{int(causal)}_t{int(tail)}"
            assert (desc.code_object.decode(), desc.kernel.decode()) == (f, sym)
            assert desc.kernel + b"\x00" in objects[f], sym
            assert desc.layout == (_lib.TA_LAYOUT_WIDE if wide else _lib.TA_LAYOUT_WHOLE_ROWS)
            assert desc.tail == int(tail)
            rows = 32 if wide else tm
            assert desc.grid == -(-s // rows) and desc.rows == rows
            assert desc.block == (512 if eight else 2 * tm)
            assert desc.in_place_pad == int(eight)
            assert desc.split_capable == int(accum == _lib.TA_ACC_FP32 and d <= 160 and (tm == 128 or d != 256))
            assert desc.merge_kernel == b"" and desc.workspace_bytes == 0


# Causal pairs: the eight-wave kernel (tiles (128, 64) / (128, 128), fp32) at D <= 128,
# two or more query blocks a head, and sched 3, or sched 1 with two or more workgroups per CU.
@pytest.mark.parametrize("kw,pairs", [
    (dict(), True),                                      # C3 S=8192: 512 blocks on 256 CUs
    (dict(S=4096), False),                               # 256 blocks: one wave
    (dict(S=4096, sched=3), True),                       # forced
    (dict(sched=0), False), (dict(sched=2), False),
    (dict(causal=False), False), (dict(D=160), False),
    (dict(accum=_lib.TA_ACC_INPUT), False), (dict(tile_m=64), False),
    (dict(S=128, sched=3), False),                       # one block a head
    (dict(S=8192, H=4, sched=1), False),                 # 256 blocks
    (dict(tile_n=128), True), (dict(D=64), True), (dict(D=96), True),
])
def test_pairing_rule(lib, objects, kw, pairs):
    args = dict(B=1, H=8, S=8192, D=128, causal=True, tile_m=128, tile_n=64, accum=_lib.TA_ACC_FP32,
                sched=1, dtype=_lib.TA_BF16)
    args.update(kw)
    desc = _d(lib, **args)
    nq = -(-args["S"] // args["tile_m"])
    assert (desc.layout == _lib.TA_LAYOUT_PAIRS) is pairs
    if pairs:
        assert desc.kernel.decode() == f"ta_fwd_pp_pair_bf16_d{args['D']}_c1_t0"
        assert desc.grid == args["B"] * args["H"] * ((nq + 1) // 2)
    elif desc.layout == _lib.TA_LAYOUT_ROWS256:  # non-causal B1 H8 S8192: one round of 256 rows
        assert not args["causal"] and _rounds_rule(args["B"], args["H"], args["S"])
        assert desc.grid == args["B"] * args["H"] * -(-args["S"] // 256)
    else:
        assert desc.grid == args["B"] * args["H"] * nq
    assert desc.kernel + b"\x00" in objects[desc.code_object.decode()]


def test_pairing_follows_the_compute_units(lib):
    """The same grid is two waves on 256 CUs (pairs) and one on 512 (whole rows)."""
    kw = dict(B=1, H=8, S=8192, D=128, causal=True, sched=1)
    assert _d(lib, cu=256, **kw).layout == _lib.TA_LAYOUT_PAIRS
    assert _d(lib, cu=512, **kw).layout == _lib.TA_LAYOUT_WHOLE_ROWS
    assert _d(lib, cu=512, **kw).compute_units == 512


# 256-row blocks: non-causal, fp32, tiles (128, 64) / (128, 128), D 64 or 128, when the
# 256-row grid needs at most half the rounds (one workgroup per CU) of the 128-row grid:
# 2 * ceil(B*H*ceil(S/256) / CUs) <= ceil(B*H*ceil(S/128) / CUs).
def _rounds_rule(b, h, s, cu=CU):
    r256 = -(-(b * h * -(-s // 256)) // cu)
    r128 = -(-(b * h * -(-s // 128)) // cu)
    return 2 * r256 <= r128


@pytest.mark.parametrize("kw,rows256", [
    (dict(), True),                                     # C4: 64 heads x 16 blocks = 1024
    (dict(D=64), True), (dict(tile_n=128), True),
    (dict(causal=True), False), (dict(D=160), False), (dict(D=96), False),
    (dict(H=7), True),                                  # 448 blocks: 2 rounds against 4
    (dict(H=6), False),                                 # 384: 2 rounds against 3
    (dict(H=10), False),                                # 640: 3 rounds against 5
    (dict(B=1, H=8, S=8192), True),                     # 256 blocks: 1 round against 2
    (dict(B=1, H=8, S=4096), False),                    # 128: 1 round against 1
    (dict(B=1, H=7, S=8192), True),                     # 224: 1 round against 2
    (dict(B=4, H=16, S=2100), False),                   # 576: 3 rounds against 5
    (dict(accum=_lib.TA_ACC_INPUT), False), (dict(tile_m=64), False),
])
def test_rows256_rule(lib, objects, kw, rows256):
    args = dict(B=4, H=16, S=4096, D=128, causal=False, tile_m=128, tile_n=64, accum=_lib.TA_ACC_FP32,
                sched=1, dtype=_lib.TA_FP16)
    args.update(kw)
    if args["D"] in (64, 128) and not args["causal"] and args["tile_m"] == 128 and args["accum"] == _lib.TA_ACC_FP32:
        assert _rounds_rule(args["B"], args["H"], args["S"]) is rows256
    desc = _d(lib, **args)
    assert (desc.layout == _lib.TA_LAYOUT_ROWS256) is rows256
    if rows256:
        assert desc.kernel.decode() == f"ta_fwd_pp256_f16_d{args['D']}_c0_t{int(args['S'] % 256 != 0)}"
        assert desc.grid == args["B"] * args["H"] * -(-args["S"] // 256) and desc.rows == 256
    assert desc.kernel + b"\x00" in objects[desc.code_object.decode()]


def test_rows256_rule_follows_the_compute_units(lib):
    """The same grid is one round of 256-row blocks on 256 CUs, half a round on 512."""
    kw = dict(B=1, H=8, S=8192, D=128, causal=False)
    assert _d(lib, cu=256, **kw).layout == _lib.TA_LAYOUT_ROWS256
    assert _d(lib, cu=512, **kw).layout == _lib.TA_LAYOUT_WHOLE_ROWS


def test_rows256_tail_variant_when_s_is_not_a_multiple_of_256(lib):
    desc = _d(lib, B=4, H=15, S=4224, D=128, causal=False)  # 128-aligned, not 256
    assert desc.layout == _lib.TA_LAYOUT_ROWS256
    assert desc.tail == 1 and desc.kernel.decode() == "ta_fwd_pp256_bf16_d128_c0_t1"
    assert desc.grid == 60 * 17


@pytest.mark.parametrize("d", [64, 96, 128, 160])
@pytest.mark.parametrize("causal", [False, True])
def test_split_descriptions(lib, objects, d, causal):
    """Chunks of 2 steps at S=1000 (8 blocks, 8 key steps): split kernel + merge kernel,
    both in the eight-wave object, a workspace, the kernel's tail variant (S ragged)."""
    desc = _d(lib, 2, B=1, H=2, S=1000, D=d, causal=causal)
    assert desc.layout == _lib.TA_LAYOUT_SPLIT and desc.chunk_steps == 2
    assert desc.kernel.decode() == f"ta_fwd_pp_split_bf16_d{d}_c{int(causal)}_t1"
    assert desc.merge_kernel.decode() == f"ta_fwd_merge_bf16_d{d}_c{int(causal)}"
    assert desc.block == 512 and desc.merge_block > 0 and desc.merge_grid > 0
    assert desc.workspace_bytes > 0
    # 8 blocks, chunks of 2: up to 4 chunks a block, 2 x 6 (causal) or 2 x 8 split blocks,
    # far below 3/8 of the CUs: the merge kernel runs
    assert desc.merge_in_kernel == 0
    need = __import__("ctypes").c_int64(0)
    a = _lib.shape_args(B=1, H=2, S=1000, D=d, causal=causal)
    assert lib.ta_split_workspace_size(__import__("ctypes").byref(a), 2, __import__("ctypes").byref(need)) == 0
    assert need.value == desc.workspace_bytes
    for sym in (desc.kernel, desc.merge_kernel):
        assert sym + b"\x00" in objects["attn_fwd_pp.hsaco"], sym


@pytest.mark.parametrize("kw,chunk,mik", [
    # the paired split: two chunks a block
    (dict(B=1, H=8, S=4096, causal=True), _lib.TA_SPLIT_PAIRS, 1),
    (dict(B=1, H=1, S=4096, causal=True), _lib.TA_SPLIT_PAIRS, 1),
    # at most two chunks a block, any grid
    (dict(B=1, H=1, S=2048, causal=True), 8, 1),        # 16 blocks: 8 split in 2
    (dict(B=1, H=2, S=4096, causal=False), 16, 1),      # 32 steps in 2 chunks
    # more chunks: only with 3/8 of the CUs' worth of split blocks (96 of 256)
    (dict(B=1, H=8, S=2048, causal=True), 4, 1),        # 8 x 12 = 96 split blocks, 4 chunks
    (dict(B=1, H=4, S=4096, causal=True), 11, 0),       # 4 x 21 = 84, 3 chunks
    (dict(B=1, H=1, S=4096, causal=True), 5, 0),        # 27, 7 chunks
    (dict(B=1, H=1, S=2048, causal=False), 4, 0),       # 16, 4 chunks
    (dict(B=1, H=8, S=4096, causal=True), 1, 1),        # 8 x 31 = 248 split blocks
    # more partial slots than a counter region (16384) holds: the merge kernel
    (dict(B=4, H=16, S=4096, causal=True), 1, 0),       # 64 heads x 496 slots
])
def test_in_kernel_merge_rule(lib, kw, chunk, mik):
    """The split kernel merges its own blocks (the last workgroup of a block combines its
    partials; a counter per block, its chunk-0 slot) when the counters fit a region and no
    block has more than two chunks or the split blocks number 3/8 of the CUs or more;
    otherwise the merge kernel runs after it."""
    desc = _d(lib, chunk, D=128, **kw)
    assert desc.layout in (_lib.TA_LAYOUT_SPLIT, _lib.TA_LAYOUT_PAIRED_SPLIT)
    assert desc.merge_in_kernel == mik and desc.merge_grid > 0 and desc.merge_kernel != b""


def test_in_kernel_merge_rule_follows_the_compute_units(lib):
    kw = dict(B=1, H=8, S=2048, D=128, causal=True)  # 96 split blocks of up to 4 chunks
    assert _d(lib, 4, cu=256, **kw).merge_in_kernel == 1
    assert _d(lib, 4, cu=512, **kw).merge_in_kernel == 0
    whole = _d(lib, 0, B=1, H=8, S=4096, D=128, causal=True)
    assert whole.merge_in_kernel == 0 and whole.merge_kernel == b""


def test_paired_split_and_chunks_that_split_nothing(lib):
    desc = _d(lib, _lib.TA_SPLIT_PAIRS, B=1, H=8, S=4096, D=128, causal=True)
    assert desc.layout == _lib.TA_LAYOUT_PAIRED_SPLIT and desc.chunk_steps == _lib.TA_SPLIT_PAIRS
    assert desc.kernel.decode() == "ta_fwd_pp_psplit_bf16_d128_c1_t0"
    assert desc.grid == 8 * 32  # the whole-row grid's size
    # a chunk at least as long as every row splits nothing: whole rows, no workspace
    whole = _d(lib, 64, B=1, H=8, S=4096, D=128, causal=True)
    assert whole.layout == _lib.TA_LAYOUT_WHOLE_ROWS and whole.workspace_bytes == 0
    # the paired split of a non-causal call is the whole-row launch
    assert _d(lib, _lib.TA_SPLIT_PAIRS, B=1, H=8, S=4096, D=128).layout == _lib.TA_LAYOUT_WHOLE_ROWS


def test_split_on_a_configuration_without_split_kernels(lib):
    with pytest.raises(ValueError, match="TA_EUNSUPPORTED"):
        _d(lib, 2, S=1000, D=128, tile_m=64, accum=_lib.TA_ACC_INPUT)
    with pytest.raises(ValueError, match="TA_EUNSUPPORTED"):  # the paired split: 128-row tiles
        _d(lib, _lib.TA_SPLIT_PAIRS, S=8192, D=128, tile_m=64, causal=True)
    # ... unless the chunk splits nothing, which runs whole rows on any kernel
    assert _d(lib, 64, S=1000, D=128, tile_m=64, accum=_lib.TA_ACC_INPUT).layout == _lib.TA_LAYOUT_WHOLE_ROWS


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 96, 128, 160])
def test_64_row_split_descriptions(lib, objects, d, causal):
    """Chunks on the 64-row kernel: the 128-row numbering with two 64-row halves per item
    (twice the workgroups of the 128-row split), the same merge kernel and workspace."""
    d128 = _d(lib, 2, B=1, H=2, S=1000, D=d, causal=causal)
    d64 = _d(lib, 2, B=1, H=2, S=1000, D=d, causal=causal, tile_m=64)
    assert d64.layout == _lib.TA_LAYOUT_SPLIT and d64.rows == 64
    assert d64.kernel.decode() == f"ta_fwd_pp64_split_bf16_d{d}_c{int(causal)}_t1"
    assert d64.grid == 2 * d128.grid
    assert (d64.merge_kernel, d64.merge_grid, d64.workspace_bytes) == (
        d128.merge_kernel, d128.merge_grid, d128.workspace_bytes)
    for sym in (d64.kernel, d64.merge_kernel):
        assert sym + b"\x00" in objects["attn_fwd_pp.hsaco"], sym
    # the dispatch model plans the 128-row kernel only: auto leaves 64-row tiles whole
    plan = lib.ta_split_plan_model(1000, 2, int(causal), 256)
    a = _lib.shape_args(B=1, H=2, S=1000, D=d, causal=causal, tile_m=64)
    out = __import__("ctypes").c_int32(-7)
    assert lib.ta_split_plan(__import__("ctypes").byref(a), __import__("ctypes").byref(out)) in (0, 4)
    assert plan >= 0


def test_zero_size_and_invalid_requests(lib):
    desc = _d(lib, S=0)
    assert desc.grid == 0 and desc.kernel == b""
    with pytest.raises(ValueError, match="head_dim"):
        _d(lib, D=80)
    with pytest.raises(ValueError, match="compute_units"):
        _d(lib, cu=0)
    with pytest.raises(ValueError, match="chunk_steps"):
        _d(lib, -5)


def test_policy_defaults_run_the_described_kernels(lib):
    """The host policy's default tiles for the study's configurations, through the library:
    C1 64-row tile on the wide kernel (tail variant: S = 64 is not a whole 128-key step), C2
    (64, 64) non-causal and C3 S = 512 the wide kernel (32-row blocks in one round of the
    CUs), C3 S = 2048 the 64-row kernel (512 blocks of 32 rows would be two rounds), S = 4096
    whole 128-row blocks, S=8192 causal pairs, C4 256-row blocks, C5 causal pairs."""
    cases = [
        ((1, 2, 64, 64), True, "ta_fwd_wide_f16_d64_c1_t1", _lib.TA_LAYOUT_WIDE, _lib.TA_FP16),
        ((1, 8, 1024, 64), False, "ta_fwd_wide_f16_d64_c0_t0", _lib.TA_LAYOUT_WIDE, _lib.TA_FP16),
        ((1, 8, 512, 128), True, "ta_fwd_wide_bf16_d128_c1_t0", _lib.TA_LAYOUT_WIDE, _lib.TA_BF16),
        ((1, 8, 1024, 128), True, "ta_fwd_wide_bf16_d128_c1_t0", _lib.TA_LAYOUT_WIDE, _lib.TA_BF16),
        ((1, 8, 2048, 128), True, "ta_fwd_pp64_bf16_d128_c1_t0", _lib.TA_LAYOUT_WHOLE_ROWS, _lib.TA_BF16),
        ((1, 8, 4096, 128), True, "ta_fwd_pp_bf16_d128_c1_t0", _lib.TA_LAYOUT_WHOLE_ROWS, _lib.TA_BF16),
        ((1, 8, 8192, 128), True, "ta_fwd_pp_pair_bf16_d128_c1_t0", _lib.TA_LAYOUT_PAIRS, _lib.TA_BF16),
        ((4, 16, 4096, 128), False, "ta_fwd_pp256_bf16_d128_c0_t0", _lib.TA_LAYOUT_ROWS256, _lib.TA_BF16),
        ((4, 16, 4096, 64), False, "ta_fwd_pp256_f16_d64_c0_t0", _lib.TA_LAYOUT_ROWS256, _lib.TA_FP16),
        ((1, 8, 16384, 128), True, "ta_fwd_pp_pair_f16_d128_c1_t0", _lib.TA_LAYOUT_PAIRS, _lib.TA_FP16),
    ]
    for (b, h, s, d), causal, kernel, layout, dtype in cases:
        tm, tn = ff._default_tile_config_for_shape_gfx950(seq_len=s, head_dim=d, causal=causal, n_bh=b * h,
                                                          compute_units=CU)
        if (b, h, s, d) == (1, 8, 1024, 64):
            tm, tn = 64, 64  # C2 pins its tile
        n_qblk = -(-s // tm)
        sched = ff._resolve_sched(n_blocks=b * h * n_qblk, causal=causal, tile_m=tm, tile_n=tn,
                                  head_dim=d, compute_units=CU)
        desc = _d(lib, B=b, H=h, S=s, D=d, causal=causal, tile_m=tm, tile_n=tn, sched=sched, dtype=dtype)
        assert (desc.kernel.decode(), desc.layout) == (kernel, layout), (b, h, s, d)


# Small-workgroup kernel: 128-row fp32 tiles, more 128-row blocks than CUs, short rows.
@pytest.mark.parametrize("d,causal,b,s,rows", [
    (64, False, 32, 128, False), (64, False, 33, 128, True),        # 256 / 264 blocks of 256 CUs
    (64, False, 24, 512, True), (64, False, 24, 513, False),        # 768 / 960 blocks
    (64, False, 16, 1024, True), (64, False, 16, 1025, False),      # four blocks a CU
    (96, False, 8, 1024, True), (96, False, 8, 1025, False),
    (128, False, 9, 512, True), (128, False, 9, 513, False),
    (160, False, 8, 768, True), (160, False, 8, 769, False),
    # causal: whole heads on every XCD
    (64, True, 16, 384, True), (64, True, 16, 512, True),
    (64, True, 7, 1024, False), (64, True, 8, 1024, True),          # 448 / 512 blocks
    (64, True, 6, 1280, False), (64, True, 8, 1280, True), (64, True, 8, 1536, True),
    (64, True, 10, 1408, False), (64, True, 16, 1408, True),        # resident at once, odd; past it
    (64, True, 6, 2048, False), (64, True, 8, 2048, True), (64, True, 10, 3073, False),
    (96, True, 7, 896, False), (96, True, 8, 960, True), (96, True, 8, 1024, False),
    (96, True, 8, 1536, True), (96, True, 8, 1920, True), (96, True, 8, 1921, False),
    (128, True, 10, 388, True), (128, True, 12, 512, False), (128, True, 16, 512, False),
    (128, True, 14, 640, True), (128, True, 9, 1024, True), (128, True, 9, 1025, False),
    (160, True, 9, 512, True), (160, True, 8, 640, False), (160, True, 10, 640, True),
    (160, True, 8, 1024, False), (160, True, 9, 1024, True), (160, True, 10, 896, True), (160, True, 8, 1536, True),
    (160, True, 8, 1537, False),
])
def test_small_workgroup_rule(lib, objects, d, causal, b, s, rows):
    for aligned in (0, 1):
        desc = _d(lib, B=b, H=8, S=s, D=d, causal=causal, tile_m=128, sched=1, aligned=aligned)
        assert desc.kernel.decode().startswith("ta_fwd_rows_") is rows, desc.kernel
        assert desc.kernel + b"\x00" in objects[desc.code_object.decode()]
        if rows:
            assert desc.kernel.decode() == f"ta_fwd_rows_bf16_d{d}_c{int(causal)}_t{int(not (aligned and s % 128 == 0))}"
            assert (desc.grid, desc.block, desc.rows) == (8 * b * -(-s // 128), 256, 128)
            assert desc.layout == _lib.TA_LAYOUT_WHOLE_ROWS
    # Forced pairs and 64-row tiles keep the eight-wave kernels (the wide one on small grids, which
    # these are not).
    for kw, prefix in ((dict(sched=3), "ta_fwd_pp"), (dict(tile_m=64), "ta_fwd_pp64_")):
        args = dict(B=b, H=8, S=s, D=d, causal=causal, tile_m=128, sched=1)
        args.update(kw)
        assert _d(lib, **args).kernel.decode().startswith(prefix)
    # Input-dtype accumulation has its own small workgroups, by a rule of its own.
    if d in (64, 128):
        desc = _d(lib, B=b, H=8, S=s, D=d, causal=causal, tile_m=128, sched=1, accum=_lib.TA_ACC_INPUT)
        n = 8 * b * -(-s // 128)
        line = 512 if not causal else 3072 if d == 64 and n >= 6 * CU else 2048 if n >= 3 * CU else 1024
        free = not causal and (d == 64 or s <= 4096)
        near_one = causal and s > 512 and (n * 3 <= 4 * CU if -(-s // 128) == 7 else n * 8 < 9 * CU and -s % 128 < 64)
        fam = "rowsl" if n > CU and (free or (causal and s <= line and not (s <= 1024 and near_one))) else "ppl"
        assert desc.kernel.decode() == f"ta_fwd_{fam}_n64_bf16_d{d}_c{int(causal)}_t{int(s % 128 != 0)}"


# Heads that the XCDs cannot take whole: small workgroups and pairs by the grid's size alone.
@pytest.mark.parametrize("d,h,s,family", [
    (64, 129, 512, "rows"), (64, 63, 1024, "pp"), (64, 65, 1024, "rows"), (64, 129, 1024, "rows"), (64, 129, 1537, "pp_pair"),
    (128, 129, 512, "rows"), (128, 65, 640, "pp"), (128, 129, 640, "rows"), (128, 129, 769, "pp_pair"),
    (160, 65, 640, "rows"), (160, 65, 641, "pp"),
    # whole heads on every XCD: pairs only where they fill the rounds of the CUs
    (128, 32, 2048, "pp_pair"), (128, 40, 2048, "pp"), (128, 41, 2048, "pp_pair"), (128, 40, 3072, "pp_pair"),
    (128, 40, 3200, "pp_pair"), (128, 48, 2688, "pp"),  # eight single blocks left over; sixteen of 24
])
def test_causal_family(lib, objects, d, h, s, family):
    desc = _d(lib, B=1, H=h, S=s, D=d, causal=True, tile_m=128, sched=1)
    assert desc.kernel.decode() == f"ta_fwd_{family}_bf16_d{d}_c1_t{int(s % 128 != 0)}"
    assert desc.kernel + b"\x00" in objects[desc.code_object.decode()]


# The same workgroups with input-dtype accumulation: 128-row tiles, more blocks than CUs.
@pytest.mark.parametrize("d,tn,causal,b,s,rows", [
    (64, 64, False, 32, 128, False), (64, 64, False, 33, 128, True), (64, 128, False, 4, 16384, True),
    (64, 64, True, 8, 1024, True), (64, 64, True, 4, 2048, False), (64, 128, True, 6, 2048, True),
    (64, 64, True, 6, 3072, False), (64, 64, True, 8, 3072, True), (64, 64, True, 16, 3073, False),
    (128, 64, False, 2, 4096, True), (128, 64, False, 2, 4097, False), (128, 64, True, 16, 2048, True),
    (128, 64, True, 16, 2049, False), (128, 128, False, 16, 768, True), (128, 128, False, 16, 769, False),
    (128, 128, True, 16, 512, True), (128, 128, True, 16, 513, False),
])
def test_small_workgroup_rule_input_dtype(lib, objects, d, tn, causal, b, s, rows):
    desc = _d(lib, B=b, H=8, S=s, D=d, causal=causal, tile_m=128, tile_n=tn, sched=1, accum=_lib.TA_ACC_INPUT)
    fam = "rowsl" if rows else "ppl"
    assert desc.kernel.decode() == f"ta_fwd_{fam}_n{tn}_bf16_d{d}_c{int(causal)}_t{int(s % 128 != 0)}"
    assert desc.kernel + b"\x00" in objects[desc.code_object.decode()]
    assert (desc.grid, desc.block, desc.rows) == (8 * b * -(-s // 128), 256 if rows else 512, 128)
    d64 = _d(lib, B=b, H=8, S=s, D=d, causal=causal, tile_m=64, tile_n=tn, sched=1, accum=_lib.TA_ACC_INPUT)
    assert d64.kernel.decode().startswith("ta_fwd_ppl64_")


# Just above one block per CU a causal grid of longer rows keeps the eight-wave kernel.
@pytest.mark.parametrize("d,tn,h,s,rows", [
    (64, 64, 65, 512, True), (64, 64, 56, 533, True), (64, 64, 52, 576, True), (64, 64, 52, 577, False),
    (64, 64, 52, 640, False), (64, 128, 64, 640, True),
    (64, 64, 47, 768, False), (64, 64, 48, 768, True), (64, 128, 40, 896, False), (64, 64, 48, 896, False),
    (64, 64, 49, 896, True), (64, 128, 39, 1024, False), (64, 64, 40, 1024, True), (128, 64, 48, 768, True),
    (128, 64, 65, 512, True), (128, 64, 56, 640, False), (128, 64, 64, 640, True), (128, 64, 53, 768, False),
    (128, 64, 40, 776, False), (128, 64, 40, 834, False), (128, 64, 48, 896, False), (128, 64, 49, 896, True),
    (128, 64, 39, 1024, False), (128, 64, 40, 1024, True),
])
def test_small_workgroup_rule_input_dtype_near_one_block_a_cu(lib, d, tn, h, s, rows):
    desc = _d(lib, B=1, H=h, S=s, D=d, causal=True, tile_m=128, tile_n=tn, sched=1, accum=_lib.TA_ACC_INPUT)
    fam = "rowsl" if rows else "ppl"
    assert desc.kernel.decode() == f"ta_fwd_{fam}_n{tn}_bf16_d{d}_c1_t{int(s % 128 != 0)}"
    free = _d(lib, B=1, H=h, S=s, D=d, causal=False, tile_m=128, tile_n=tn, sched=1, accum=_lib.TA_ACC_INPUT)
    assert free.kernel.decode().startswith(f"ta_fwd_rowsl_n{tn}_")  # not causal: every block is as long


# Where the small workgroups' grid is no multiple of 8 blocks (no XCD order) or just past a round
# of pairs, the eight-wave kernels keep it.
@pytest.mark.parametrize("d,causal,h,s,rows", [
    (64, False, 65, 512, False), (64, False, 66, 512, True), (64, False, 89, 449, False), (64, False, 102, 512, True),
    (64, False, 129, 512, True), (64, False, 179, 256, True), (64, False, 253, 256, False), (64, False, 253, 245, True),
    (64, False, 89, 440, True), (64, False, 121, 512, True), (128, False, 71, 405, False), (128, False, 121, 405, True),
    (128, False, 89, 512, False), (128, False, 121, 512, False), (128, False, 179, 224, False),
    (128, False, 221, 224, True), (64, False, 89, 384, True),
    (128, False, 65, 512, False), (128, False, 102, 512, True), (128, False, 179, 199, False), (128, False, 221, 243, True),
    (128, False, 160, 199, True), (128, False, 179, 192, True), (128, False, 100, 330, True), (128, False, 257, 256, True),
    (64, True, 58, 1152, False), (64, True, 71, 1152, True), (64, True, 58, 1024, False), (96, True, 58, 1152, False),
    (96, True, 57, 1088, True), (96, True, 57, 1089, False), (96, True, 52, 1280, True),
    (64, True, 43, 1536, True), (96, True, 129, 1472, True), (96, True, 86, 1536, True), (96, True, 71, 1152, True),
    (96, True, 53, 1536, True),
    (96, True, 67, 1536, False), (64, True, 67, 1536, True),
    (128, True, 105, 576, True), (128, True, 105, 640, False), (128, True, 105, 609, False), (128, True, 107, 711, True),
    (128, True, 107, 736, True), (128, True, 107, 768, False), (128, True, 127, 768, False),
    (128, True, 278, 768, False), (128, True, 278, 736, True),
    (128, True, 118, 640, True),
    (160, True, 52, 640, False), (160, True, 52, 580, True), (160, True, 54, 640, True), (160, True, 65, 512, True),
])
def test_small_workgroup_rule_without_xcd_order(lib, d, causal, h, s, rows):
    desc = _d(lib, B=1, H=h, S=s, D=d, causal=causal, tile_m=128, sched=1)
    assert desc.kernel.decode().startswith("ta_fwd_rows_") is rows, desc.kernel


@pytest.mark.parametrize("d,accum", [(d, _lib.TA_ACC_FP32) for d in (64, 96, 128, 160, 256)]
                         + [(d, _lib.TA_ACC_INPUT) for d in (64, 128)])
def test_head_groups_are_even_and_bounded(lib, d, accum):
    """Groups of the causal head order: none below two heads, at most twice plus one the heads (two to
    eight) whose K and V fit 4 MiB, and no last group of half the others' heads or fewer."""
    grouped = few = 0
    for heads in range(2, 41):  # a group per XCD
        for s in (256, 384, 512, 640, 896, 1024, 1152, 1280, 1408, 2048, 2500, 4096):
            args = _lib.shape_args(B=heads, H=8, S=s, D=d, causal=True, sched=1, accum=accum)
            g = _lib.head_group(lib, args, CU)
            if not g:
                continue
            grouped += 1
            fit = min(8, max(2, (4 << 20) // (s * d * 4)))
            last = heads % g or g
            assert 2 <= g <= heads and g <= 2 * fit + 1, (heads, s, g, fit)
            # (37 heads: 37 = 4 * 8 + 5 is the first size that leaves more than half)
            assert 2 * last > g or not any(heads % n == 0 or 2 * (heads % n) > n for n in range(g, 2 * fit + 2)), (heads, s, g)
            few += heads <= 20 and 2 * last <= g
    assert grouped > 100 and few == 0
    for kw in (dict(causal=False), dict(sched=0), dict(H=7)):
        args = dict(B=20, H=8, S=1024, D=d, causal=True, sched=1, accum=accum)
        args.update(kw)
        assert _lib.head_group(lib, _lib.shape_args(**args), CU) == 0


@pytest.mark.parametrize("d,heads,s,group", [
    (256, 56, 1408, 4), (256, 104, 1408, 5), (256, 80, 1152, 5), (256, 40, 2048, 3), (256, 64, 2048, 2),
    (128, 40, 1000, 5), (160, 48, 1024, 6), (64, 88, 640, 0),
])
def test_head_group_sizes(lib, d, heads, s, group):
    assert _lib.head_group(lib, _lib.shape_args(B=1, H=heads, S=s, D=d, causal=True, sched=1), CU) == group
