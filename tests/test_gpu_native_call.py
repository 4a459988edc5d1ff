"""The native tail of a Python call (_tiledattn_call.launch): taken where nothing is copied,
left where something is, and equal to the operator's results either way; on a side stream, in
a captured graph, from two threads, and with a failing launch."""

from __future__ import annotations

import threading

import pytest

from tests.parity_util import inputs, knobs, say

pytestmark = pytest.mark.gpu


def _qkv(shape=(1, 2, 200, 64), dtype="float16", seed=3):
    return [t.to("cuda:0") for t in inputs(shape, dtype, seed)]


def _plan(q, k, v, causal):
    import torch

    from tiledattention.kernels import flash_fwd

    return flash_fwd._plan_for(torch, q, k, v, causal, None, None)


def test_taken_and_left(gpu):
    import torch

    from tiledattention import sdpa, torch_op

    q, k, v = _qkv()
    assert _plan(q, k, v, True).launch is not None
    say("native call: plain, misaligned, strided, subclass, sync mode, split, padded on the host")
    want = torch_op.sdpa_fwd(q, k, v, True)
    assert torch.equal(sdpa(q, k, v, causal=True), want)
    buf = torch.empty(q.numel() + 4, dtype=q.dtype, device=q.device)  # 8 bytes off 16
    qm = buf[4:].view(q.shape).copy_(q)
    assert qm.data_ptr() % 16 == 8 and torch.equal(sdpa(qm, k, v, causal=True), want)
    wide = torch.zeros(1, 2, 200, 68, dtype=q.dtype, device=q.device)
    wide[..., :64] = q
    qw = wide[..., :64]
    assert _plan(qw, k, v, True).launch is None and torch.equal(sdpa(qw, k, v, causal=True), want)

    class Sub(torch.Tensor):
        pass

    assert torch.equal(sdpa(q, k.as_subclass(Sub), v, causal=True).as_subclass(torch.Tensor), want)
    with knobs(sync_mode="post"):
        assert _plan(q, k, v, True).launch is None and torch.equal(sdpa(q, k, v, causal=True), want)
    for shape in ((1, 2, 4096, 128), (1, 2, 64, 100)):  # a split workspace; host padding
        a = _qkv(shape)
        assert _plan(*a, True).launch is None
        assert torch.equal(sdpa(*a, causal=True), torch_op.sdpa_fwd(*a, True))
    torch.cuda.synchronize()


def test_streams_capture_and_threads(gpu):
    import torch

    from tiledattention import sdpa, torch_op

    q, k, v = _qkv((1, 8, 300, 64), "bfloat16")
    want = torch_op.sdpa_fwd(q, k, v, False)
    torch.cuda.synchronize()
    say("native call on a side stream, captured and replayed, and from two threads")
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        got = sdpa(q, k, v)
    side.synchronize()
    assert torch.equal(got, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = sdpa(q, k, v)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(sdpa(q, k, v), want)
    bad = []

    def work():
        for _ in range(50):
            if not torch.equal(sdpa(q, k, v), want):
                bad.append(1)

    ts = [threading.Thread(target=work) for _ in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


def test_library_status_is_raised(gpu):
    """A plan whose arguments the library refuses raises its status, as the ctypes path does."""
    from tiledattention import InvalidShapeError, sdpa

    q, k, v = _qkv((1, 2, 77, 64))
    plan = _plan(q, k, v, False)
    plan.args.dtype = 9
    try:
        with pytest.raises(InvalidShapeError, match="dtype 9"):
            sdpa(q, k, v)
    finally:
        plan.args.dtype = 0
    sdpa(q, k, v)


def test_plan_made_by_another_tensor_type(gpu, monkeypatch):
    """The first call of a layout with a Parameter, or a subclass, as q: later plain calls are
    native all the same."""
    import torch

    from tiledattention import sdpa
    from tiledattention.kernels import flash_fwd

    class Sub(torch.Tensor):
        pass

    q, k, v = _qkv((1, 3, 140, 64))
    want = sdpa(q, k, v, causal=True)
    for first in (torch.nn.Parameter(q, requires_grad=False), torch.nn.Parameter(q), q.as_subclass(Sub)):
        monkeypatch.setattr(flash_fwd, "_PLANS", {})
        monkeypatch.setattr(flash_fwd, "_PLANS_BY_LAYOUT", {})
        say(f"plan made by {type(first).__name__}")
        out = sdpa(first, k, v, causal=True)
        assert torch.equal(out.as_subclass(torch.Tensor), want) and not out.requires_grad
        assert _plan(q, k, v, True).launch is not None and torch.equal(sdpa(q, k, v, causal=True), want)


def test_calls_work_without_the_module(gpu, monkeypatch, tmp_path):
    """A library directory without the module: the ctypes path launches the same kernel."""
    import torch

    from tiledattention import _lib, sdpa
    from tiledattention.kernels import flash_fwd

    q, k, v = _qkv((1, 3, 130, 64))
    want = sdpa(q, k, v, causal=True)
    monkeypatch.setattr(_lib, "call_module_path", lambda: tmp_path / "absent.so")
    monkeypatch.setattr(_lib, "_call", None)
    monkeypatch.setattr(flash_fwd, "_PLANS", {})
    monkeypatch.setattr(flash_fwd, "_PLANS_BY_LAYOUT", {})
    say("ctypes call without the native module")
    for _ in range(2):
        assert torch.equal(sdpa(q, k, v, causal=True), want)
    assert _plan(q, k, v, True).launch is None and _lib.loaded_call() is None


_WAITER = r"""
#include <unistd.h>
extern "C" int flag = 0;
extern "C" int wait_for_flag(const void*, void*) {  // a ta_sdpa_fwd that blocks, 3 s at most
  for (int i = 0; i < 3000; ++i) {
    if (__atomic_load_n(&flag, __ATOMIC_ACQUIRE)) return 0;
    usleep(1000);
  }
  return 4;
}
"""


def test_other_threads_run_while_the_library_call_blocks(gpu, tmp_path):
    """The interpreter lock is free during the allocation and the library call, as in the ctypes
    path: here the call returns only once another Python thread has set its flag."""
    import ctypes
    import shutil
    import subprocess
    import time

    import torch

    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "waiter.cpp").write_text(_WAITER)
    so = tmp_path / "waiter.so"
    subprocess.run([gxx, "-O1", "-shared", "-fPIC", "-o", str(so), str(tmp_path / "waiter.cpp")], check=True)
    waiter = ctypes.CDLL(str(so))
    flag = ctypes.c_int.in_dll(waiter, "flag")
    q, k, v = _qkv()
    plan = _plan(q, k, v, False)
    say("native call of a library function that waits for another thread")

    def release():
        time.sleep(0.05)
        flag.value = 1

    t = threading.Thread(target=release)
    t.start()
    out = plan.launch(ctypes.cast(waiter.wait_for_flag, ctypes.c_void_p).value, plan.args_addr, q, k, v, 1.0)
    t.join()
    assert isinstance(out, torch.Tensor), f"status {out}: no other thread ran"
