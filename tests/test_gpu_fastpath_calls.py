"""The C++ fast path's other entry points (velograd_amd/csrc/torch_fastpath.cpp) against the general
Python path to the same kernels: the same bits, types and shapes, the calls they decline, and the
same exceptions."""

import pytest
import torch

from velograd_amd import _lib
from velograd_amd import kernels as vk

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture
def both(monkeypatch):
    """Runs a call through the fast path and through the general path."""
    if _lib.fastpath() is None:
        pytest.skip("the fast path is not built (velograd_amd.build builds it)")

    def run(f):
        fast = f()
        with monkeypatch.context() as m:
            m.setattr(_lib, "fastpath", lambda: None)
            general = f()
        assert len(fast) == len(general)
        for a, b in zip(fast, general):
            if b is None:
                assert a is None
                continue
            assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
        return fast
    return run


def _randn(*shape, dtype=BF):
    return torch.randn(shape, device="cuda").to(dtype)


@pytest.mark.parametrize("dtype,wdt", [(BF, BF), (HF, F32), (F32, F32), (BF, None)])
@pytest.mark.parametrize("shape", [(7, 64), (2, 3, 1024), (1, 1, 96)])
def test_every_call_matches_the_general_path(both, shape, dtype, wdt):
    torch.manual_seed(1)
    d = shape[-1]
    x, r, g, gh = (_randn(*shape, dtype=dtype) for _ in range(4))
    w = _randn(d, dtype=wdt) if wdt is not None else None
    for res in (r, None):
        both(lambda: vk.fused_rmsnorm_residual_forward_fp8(x, res, w, 1e-5))
        for fmt in ("e4m3", "e2m1"):
            both(lambda: vk.fused_rmsnorm_residual_forward_mx(x, res, w, 1e-5, fmt=fmt))
    _, h, inv = vk.fused_rmsnorm_residual_forward(x, r, w, 1e-5)
    for is_h in (True, False):
        for ghv in (None, gh):
            dres = torch.empty_like(x)
            dx, _ = both(lambda: vk.fused_rmsnorm_residual_backward(
                g, h, w, inv, saved_is_h=is_h, grad_h=ghv, dresidual_out=dres))
            assert torch.equal(dx, dres)
    both(lambda: (vk.fused_rope_interleaved(x, 1e4), vk.fused_rope_interleaved(g, 1e4, True)))
    for res in (r, None):
        both(lambda: vk.rmsnorm_rope_forward(x, w, 1e-5, 1e4, res))
    both(lambda: vk.rmsnorm_rope_backward(g, h, w, inv, 1e4))
    q, k = _randn(2, 5, 4, 64, dtype=dtype), _randn(2, 5, 1, 80, dtype=dtype)
    for head_dim in (None, 32):
        both(lambda: vk.fused_rope_forward(q, k, head_dim))
        both(lambda: vk.fused_rope_backward(q, None, head_dim, 5e5))


def test_h_is_x_without_a_residual():
    x = _randn(4, 64)
    assert vk.fused_rmsnorm_residual_forward_fp8(x, None, None)[2] is x
    assert vk.rmsnorm_rope_forward(x, None)[1] is x


def test_declined_calls_take_the_general_path():
    fp = _lib.fastpath()
    if fp is None:
        pytest.skip("the fast path is not built")
    x, g = _randn(8, 64), _randn(8, 64)
    inv = torch.rand(8, 1, device="cuda") + 0.5
    strided = _randn(64, 8).t()
    assert fp.backward(strided, x, None, inv, True, None, None) == []
    assert fp.backward(g, x.float(), None, inv, True, None, None) == []
    assert fp.backward(g, x, None, inv.half(), True, None, None) == []
    assert fp.backward(g, x, None, inv[:4], True, None, None) == []
    assert fp.backward(g, x, _randn(1, 64), inv, True, None, None) == []
    assert fp.backward(g[:0], x[:0], None, inv[:0], True, None, None) == []
    assert fp.forward_quantised(x[:, :48].contiguous(), None, None, 1e-6, 0) == []
    assert fp.rope(x, None, 0, 1e4, False) == []                       # 2-D: split into heads
    assert fp.rope(_randn(2, 3, 4, 7), None, 0, 1e4, False) == []      # odd
    assert fp.rope(_randn(1, 3, 4, 8), _randn(1, 2, 4, 8), 0, 1e4, False) == []
    assert fp.rope_interleaved(_randn(3, 7), 1e4, False) == []
    assert fp.norm_rope(x.cpu(), None, None, 1e-6, 1e4, 0.0) == []
    dx, dw = vk.fused_rmsnorm_residual_backward(strided, x, None, inv, saved_is_h=True)
    assert dx.shape == x.shape and dw is None


def test_errors_are_those_of_the_general_path():
    x, inv = _randn(8, 64), torch.rand(8, 1, device="cuda")
    with pytest.raises(ValueError):
        vk.fused_rope_forward(_randn(1, 3, 2, 8), theta=-1.0)
    with pytest.raises(ValueError):
        vk.rmsnorm_rope_forward(x, None, base=float("inf"))
    with pytest.raises(ValueError):
        vk.fused_rmsnorm_residual_backward(x, x, None, inv, dresidual_out=x)
    with pytest.raises(ValueError):
        vk.fused_rmsnorm_residual_backward(x, x[:4], None, inv)
    with pytest.raises(TypeError):
        vk.fused_rmsnorm_residual_backward(x, x.float(), None, inv)


def test_calls_follow_the_current_stream_and_capture():
    x, w = _randn(64, 256), _randn(256)
    g = _randn(64, 256)
    _, h, inv = vk.fused_rmsnorm_residual_forward(x, x, w, 1e-5)
    want = vk.fused_rmsnorm_residual_backward(g, h, w, inv, saved_is_h=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = vk.fused_rmsnorm_residual_backward(g, h, w, inv, saved_is_h=True)
    torch.cuda.current_stream().wait_stream(s)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = vk.fused_rmsnorm_residual_backward(g, h, w, inv, saved_is_h=True)
    for scale in (1.0, 2.0, 0.5):
        g.copy_(_randn(64, 256) * scale)
        eager = vk.fused_rmsnorm_residual_backward(g, h, w, inv, saved_is_h=True)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], eager[0]) and torch.equal(out[1], eager[1])
