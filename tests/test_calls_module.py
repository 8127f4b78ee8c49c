"""The short calls of qlinear.py in native code (csrc/python/calls.cpp): what they refuse, before any device call, and that they use the
caller's outputs, workspaces and stream."""
import types

import numpy as np
import pytest
import torch

from mllm_amd import _lib, qlinear as ql
from gpu_util import announce


class _W:
    wtype, N, K, buf = 0, 64, 64, torch.zeros(1, dtype=torch.uint8)


class _G(_W):
    layout = "gemm"


class _V(_W):
    layout = "gemv"


X = torch.zeros(3, 64)


@pytest.mark.parametrize("call,error", [
    (lambda: ql.linear_q_gemv(_W, X), AssertionError), (lambda: ql.linear_q_gemv(_W, None), TypeError),
    (lambda: ql.linear_q_gemv_multi([], X), AssertionError), (lambda: ql.linear_q_gemv_multi([_W] * 5, X), AssertionError),
    (lambda: ql.linear_q_gemv_multi([_W], X), AssertionError), (lambda: ql.linear_q_gemv_multi(None, X), TypeError),
    (lambda: ql.softmax(X), AssertionError), (lambda: ql.topk(X, 3), AssertionError),
    (lambda: ql.matmul(X, X), AssertionError), (lambda: ql.matmul(X, X.double()), AssertionError), (lambda: ql.matmul(X[0], X[0]), IndexError),
    (lambda: ql.matmul(X.t(), X.t()), AssertionError), (lambda: ql.matmul(X.double(), X.double(), False, True), AssertionError),
    (lambda: ql.matmul(torch.zeros(2, 3, 4), torch.zeros(3, 4, 5)), AssertionError),
    (lambda: ql.w8a8_linear_packed(X, X, 64, X), AssertionError), (lambda: ql.w8a8_linear_packed(X[0], X, 64, X), ValueError),
    (lambda: ql.linear_q_gemm(_G, X), AssertionError), (lambda: ql.linear_q_gemm(_V, X), AssertionError), (lambda: ql.linear_kq_gemm(_G, X, short=True), AssertionError),
    (lambda: ql.linear_q_gemm(_G, None), TypeError), (lambda: ql.linear_kq_gemm(_W, None), TypeError),
    (lambda: ql.w4a16_gemm_packed(X, X, 64), AssertionError), (lambda: ql.w4a16_gemm_packed(X.bfloat16(), X, 64), AssertionError)])
def test_calls_refuse_what_the_kernels_do_not_take(call, error):
    with pytest.raises(error):
        call()


def _moe(call, wtype, size):
    """an MoE FFN call whose workspace is a byte short"""
    E = types.SimpleNamespace(wtype=wtype, E=4, N=256, K=256, ptr=0, layout="gemm")
    need = getattr(_lib.lib(), size)(3, 256, 256, 4, 2)
    return lambda: call(E, E, E, torch.zeros(3, 256), torch.zeros((3, 2), dtype=torch.int32), torch.zeros(3, 2), workspace=torch.empty(need - 1, dtype=torch.uint8))


def _short(size):
    return torch.empty(size - 1, dtype=torch.uint8)


@pytest.mark.parametrize("call", [
    _moe(ql.moe_ffn_q, 0, "mllm_hip_moe_workspace_bytes"), _moe(ql.moe_ffn_q_gemm, 0, "mllm_hip_moe_gemm_workspace_bytes"), _moe(ql.moe_ffn_kq, 2, "mllm_hip_moe_kq_workspace_bytes"),
    lambda: ql.w8a8_linear(X, torch.zeros((64, 64), dtype=torch.int8), X, workspace=_short(_lib.lib().mllm_hip_w8a8_workspace_bytes(3, 64))),
    lambda: ql.w8a8_linear_packed(X, torch.zeros(_lib.lib().mllm_hip_w8a8_packed_bytes(64, 64), dtype=torch.uint8), 64, X,
                                  workspace=_short(_lib.lib().mllm_hip_w8a8_workspace_bytes(3, 64)))])
def test_a_workspace_that_is_too_small_is_refused(call):
    """before any device call; the kernels wrote past it"""
    with pytest.raises(_lib.HipQLinearError, match="needed"):
        call()


@pytest.mark.gpu
def test_a_workspace_that_is_too_small_for_a_linear_is_refused():
    """the calls that look at the device first: a byte short, and one sized under a form that needs no partial results.  One of another type counts in bytes"""
    L, g = _lib.lib(), torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((70, 512), device="cuda", generator=g)
    room = lambda size: torch.empty(size, dtype=torch.uint8, device="cuda")  # noqa: E731
    announce("workspaces that are too small")
    for kq in (False, True):
        make, wtype = (ql.PackedKWeight, ql.Q6_K) if kq else (ql.PackedQWeight, ql.Q4_0)
        gemm, gemv = (make.synthetic(wtype, 256, 512, g, layout=layout) for layout in ("gemm", "gemv"))
        call = ql.linear_kq_gemm if kq else ql.linear_q_gemm
        plain = (L.mllm_hip_linear_kq_gemm_workspace_bytes if kq else L.mllm_hip_linear_q_gemm_workspace_bytes)(70, 512)
        size = L.mllm_hip_linear_kq_gemm_short_workspace_bytes if kq else L.mllm_hip_linear_q_gemm_short_workspace_bytes
        other, need = (ql.linear_kq, L.mllm_hip_kq_workspace_bytes(70, 512)) if kq else (ql.linear_q, L.mllm_hip_linear_q_workspace_bytes(70, 512))
        want = call(gemm, x)
        assert torch.equal(call(gemm, x, workspace=room(plain)), want) and torch.equal(call(gemm, x, workspace=torch.empty((plain + 3) // 4, device="cuda")), want)
        assert torch.equal(other(gemv, x, workspace=torch.empty((need + 3) // 4, device="cuda")), other(gemv, x))
        try:
            assert L.mllm_hip_q_gemm_set_form(3) == 0
            whole = size(70, 256, 512)
            assert L.mllm_hip_q_gemm_set_form(8) == 0 and size(70, 256, 512) >= whole + 4 * 70 * 256 * 4
            bad = [lambda: call(gemm, x, workspace=room(whole), short=True), lambda: call(gemm, x, workspace=room(size(70, 256, 512) - 1), short=True),
                   lambda: call(gemm, x, workspace=room(plain - 1)), lambda: other(gemv, x, workspace=room(need - 1))]
            for one in bad:
                with pytest.raises(_lib.HipQLinearError, match="needed"):
                    one()
        finally:
            assert L.mllm_hip_q_gemm_set_form(0) == 0


def test_missing_module_fails_loudly(monkeypatch):
    monkeypatch.setattr(ql, "_native", None)
    monkeypatch.setattr(_lib, "CALLS_PATH", "/nonexistent/mllm_calls.so")
    with pytest.raises(_lib.HipQLinearError):
        ql.softmax(X)


@pytest.mark.gpu
@pytest.mark.parametrize("short", [False, True])
@pytest.mark.parametrize("kq", [False, True])
def test_many_row_calls_use_the_callers_outputs_workspaces_and_stream(kq, short):
    g = torch.Generator(device="cuda").manual_seed(3)
    make, call = (ql.PackedKWeight, ql.linear_kq_gemm) if kq else (ql.PackedQWeight, ql.linear_q_gemm)
    w, v = (make.synthetic(ql.Q6_K if kq else ql.Q4_0, 256, 512, g, layout=layout) for layout in ("gemm", "gemv"))
    x, bias = torch.randn((70, 512), device="cuda", generator=g), torch.randn(256, device="cuda", generator=g)
    L = _lib.lib()
    size = ((L.mllm_hip_linear_kq_gemm_short_workspace_bytes if kq else L.mllm_hip_linear_q_gemm_short_workspace_bytes)(70, 256, 512) if short else
            (L.mllm_hip_linear_kq_gemm_workspace_bytes if kq else L.mllm_hip_linear_q_gemm_workspace_bytes)(70, 512))
    announce("many-row calls with and without outputs", kq, short)
    y = call(w, x, bias, short=short)
    assert y.shape == (70, 256) and y.dtype == torch.float32
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        torch.cuda._sleep(200_000_000)  # a call on the default stream would not wait for what follows
        out, work = torch.full((70, 256), float("nan"), device="cuda"), torch.empty(size, dtype=torch.uint8, device="cuda")
        assert call(w, x * 1, bias, out=out, workspace=work, short=short) is out
    stream.synchronize()
    assert torch.equal(out, y)
    for bad, error in ((lambda: call(v, x), AssertionError), (lambda: call(w, x[:, :256]), AssertionError), (lambda: call(w, x.half()), TypeError),
                       (lambda: call(w, x[:0]), _lib.HipQLinearError)):
        with pytest.raises(error):
            bad()


@pytest.mark.gpu
def test_calls_use_the_callers_outputs_and_stream():
    g = torch.Generator(device="cuda").manual_seed(2)
    rand = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    w, x, a, b = ql.PackedQWeight.synthetic(ql.Q4_0, 256, 256, g), rand(3, 256), rand(2, 70, 40), rand(2, 40, 50)
    bias, room = rand(256), ql.gemv_workspace(3, 256, 512)
    out = lambda *s: torch.full(s, float("nan"), device="cuda")  # noqa: E731
    announce("calls with and without outputs")
    y, c = ql.linear_q_gemv(w, x, bias), ql.matmul(a, b)
    ys = ql.linear_q_gemv_multi([w, w], x, [bias, None])
    assert torch.equal(y, ys[0]) and torch.equal(y, ys[1] + bias) and y.shape == (3, 256) and c.shape == (2, 70, 50) and c.dtype == torch.float32
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        torch.cuda._sleep(200_000_000)  # a call on the default stream would not wait for what follows
        xs, outs = x * 1, [out(3, 256), out(3, 256)]
        y1, c1 = out(3, 256), out(2, 70, 50)
        assert ql.linear_q_gemv(w, xs, bias, out=y1) is y1 and ql.matmul(a * 1, b, out=c1) is c1
        assert ql.linear_q_gemv_multi([w, w], xs, [bias, None], outs=outs, workspace=room) is outs
        p = ql.softmax(xs)
        values, ids = ql.topk(p, 7)
    stream.synchronize()
    assert torch.equal(y1, y) and torch.equal(c1, c) and float((outs[0] - y).norm() / y.norm()) < 1e-5
    assert torch.equal(ids.long(), p.topk(7).indices) and torch.equal(values, p.topk(7).values)
    with pytest.raises(_lib.HipQLinearError):
        ql.topk(p, 257)
    with pytest.raises(TypeError):
        ql.linear_q_gemv(w, x.half())
    assert torch.equal(ql.topk(p, 7, np.bool_(True), np.bool_(True))[1], ids)
    assert np.isfinite(y.cpu().numpy()).all()
