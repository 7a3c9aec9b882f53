"""The C++ call path of the Python binding (mx230_amd._binding): it takes plain
GPU tensors only, and gives what the Python path (taken with an explicit
stream) gives, bit for bit."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

import mx230_amd as mx


def test_leaves_other_calls_to_python():
    import torch
    q = torch.zeros(1, 1, 4, 64)
    c = mx._calls()
    assert c.attention_fwd(q, q, q, True, 0.0) is NotImplemented  # CPU tensors
    assert c.attention_fwd(q, q, None, True, 0.0) is NotImplemented
    assert c.attention_bwd(q, q, q, q, q, q, True, 0.0) is NotImplemented
    assert c.prefill(q, q, q, q, None, 0, 0, 1, 1, 64, 0.0, False, None) is NotImplemented
    assert c.prefill() is NotImplemented


def test_without_the_module(monkeypatch):
    """Where _binding.so is missing or does not load, the package warns once and
    takes the Python path."""
    import torch
    monkeypatch.setattr(mx, "_native", None)
    monkeypatch.delattr(mx, "_binding", raising=False)
    monkeypatch.setitem(sys.modules, "mx230_amd._binding", None)
    with pytest.warns(RuntimeWarning, match="_binding.so"):
        c = mx._calls()
    assert c.prefill() is NotImplemented and mx._calls() is c
    q = torch.zeros(1, 1, 4, 64)
    with pytest.raises(ValueError, match="device tensor"):  # raised by the Python path
        mx.attention_fwd(q, q, q, True)


@pytest.mark.parametrize("python,built", [(sys.executable, True), ("/bin/false", False)])
def test_make_without_torch(python, built):
    """The C library's build needs no torch and no Python headers: where they are
    missing the extension module is left out."""
    r = subprocess.run(["make", "-n", "-B", "-C", os.path.join(os.path.dirname(mx.LIB_PATH), "csrc"),
                        f"PYTHON={python}"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    assert ("binding.cpp" in r.stdout) == built and "libmxfa.so" in r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 6, 2, 65, 64, "bfloat16"), (1, 4, 4, 33, 128, "bfloat16"),
                                   (0, 3, 1, 20, 64, "float32")])
def test_same_as_python_path(shape):
    import torch
    B, Hq, Hkv, N, d, dt = shape  # B = 0: the 2-D single-head layout
    dt = getattr(torch, dt)
    dims = (lambda h: (B, h, N, d)) if B else (lambda h: (N, d))
    torch.manual_seed(1)
    q, k, v, do = (torch.randn(dims(h), device="cuda").to(dt) for h in (Hq, Hkv, Hkv, Hq))
    s = torch.cuda.current_stream()
    for a, b in zip(mx.attention_fwd(q, k, v, True), mx.attention_fwd(q, k, v, True, stream=s)):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    o, lse = mx.attention_fwd(q, k, v, True)
    for a, b in zip(mx.attention_bwd(q, k, v, o, lse, do, True), mx.attention_bwd(q, k, v, o, lse, do, True, stream=s)):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    with pytest.raises(ValueError):
        mx.attention_fwd(q, k, v.float() if dt == torch.bfloat16 else v.bfloat16(), True)
    if B:
        with pytest.raises(ValueError):
            mx.attention_fwd(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), True)


@pytest.mark.gpu
@pytest.mark.parametrize("n,pos0", [(1, 100), (1, 3000), (33, 2000)])
def test_prefill_same_as_python_path(n, pos0):
    import torch
    Hq, Hkv, d = 8, 2, 64
    torch.manual_seed(2)
    qkv = torch.randn(n, (Hq + 2 * Hkv) * d, device="cuda").bfloat16()
    q, rows = qkv[:, :Hq * d], -(-(pos0 + n) // 16) * 16
    k, v = (torch.randn(rows, Hkv * d, device="cuda").bfloat16() for _ in range(2))
    table = torch.randperm(rows // 16, device="cuda").to(torch.int32)
    ws = torch.empty(max(16, mx.prefill_workspace_bytes(n, pos0, Hq, Hkv, d)), dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream()
    calls = [lambda o, st: mx.run_prefill(q, k, v, o, pos0, Hq, Hkv, d, stream=st),
             lambda o, st: mx.run_prefill_split(q, k, v, o, pos0, Hq, Hkv, d, workspace=ws, stream=st),
             lambda o, st: mx.run_prefill_paged(q, k, v, o, table, 16, pos0, Hq, Hkv, d, stream=st),
             lambda o, st: mx.run_prefill_paged(q, k, v, o, table, 16, pos0, Hq, Hkv, d, stream=st, split=True,
                                                workspace=ws)]
    for f in calls:
        a, b = (torch.empty(n, Hq * d, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        assert (f(a, None) is ws) == (f(b, s) is ws)
        assert torch.equal(a, b)
    with pytest.raises(ValueError):  # too few cache rows
        mx.run_prefill(q, k[:pos0], v[:pos0], a, pos0, Hq, Hkv, d)
    with pytest.raises(mx.MxfaError):  # a head size the kernels do not have
        mx.run_prefill(q, k, v, a, pos0, Hq, Hkv, 32)


@pytest.mark.gpu
def test_current_stream_and_capture():
    """The calls run on torch's current stream: captured into a graph there and
    replayed on new inputs (with eager work between), each replay gives the
    eager result."""
    import torch
    torch.manual_seed(4)
    shape = (1, 2, 100, 64)
    q, k, v = (torch.randn(shape, device="cuda") for _ in range(3))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        mx.attention_fwd(q, k, v, True)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        o, lse = mx.attention_fwd(q, k, v, True)
        grads = mx.attention_bwd(q, k, v, o, lse, o, True)
    for _ in range(3):
        for x in (q, k, v):
            x.copy_(torch.randn(shape, device="cuda"))
        g.replay()
        torch.cuda.synchronize()
        eo, el = mx.attention_fwd(q, k, v, True)
        for a, b in zip((o, lse, *grads), (eo, el, *mx.attention_bwd(q, k, v, eo, el, eo, True))):
            assert torch.equal(a, b)


@pytest.mark.gpu
def test_out_of_memory_keeps_its_type():
    import torch
    if not hasattr(torch, "OutOfMemoryError"):
        pytest.skip("this torch has no OutOfMemoryError")
    q = torch.zeros(1, 1, 128, 64, device="cuda", dtype=torch.bfloat16)
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(1e-6)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            keep = []
            for _ in range(4096):
                keep.append(mx.attention_fwd(q, q, q, False))
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
