"""bwd_ring_kernel's kRingAny: rows of any length and alignment in chunks whose last one overlaps
the one before it.  Lengths around the element-strided bound, whole waves, one and two chunks a
thread and the layout's end; fewer rows than slots, a row past whole walks; streams that start
anywhere; dx in grad_h's place (which keeps the kernels that store each column once)."""

import numpy as np
import pytest
import torch

from oracle import fused_rmsnorm as ora
from velograd_amd import _lib
from velograd_amd import kernels as vk

from tests import _parity as P

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _rand(rng, rows, d, dtype, off):
    t = P.to_device(P.gaussian(rng, (off + rows * d,)), dtype)
    return t[off:].view(rows, d)


def _inputs(rows, d, dtype, wdtype, gh, off):
    rng = np.random.default_rng(rows * 3 + d)
    g, h = _rand(rng, rows, d, dtype, off), _rand(rng, rows, d, dtype, (2 * off) % 8)
    w = P.to_device(P.weight_vec(rng, d), wdtype) if wdtype is not None else None
    inv = 1.0 / torch.sqrt(h.float().square().mean(-1, keepdim=True) + 1e-5)
    return g, h, w, inv, (_rand(rng, rows, d, dtype, off) if gh else None)


CASES = [
    # rows, dim, dtype, weight, grad_h, offset in elements, saved is h
    (300, 192, BF, BF, False, 0, True), (300, 193, BF, BF, False, 0, True),
    (300, 193, BF, F32, True, 1, True), (5, 201, HF, HF, False, 3, False),
    (2000, 511, BF, BF, True, 0, True), (2000, 513, BF, None, False, 5, True),
    (1, 1001, BF, BF, False, 0, True), (515, 1001, BF, BF, True, 7, True),
    (515, 1024, BF, BF, False, 1, True),     # whole chunks, off a line
    (300, 2047, BF, F32, False, 0, True), (300, 2049, BF, BF, True, 0, False),
    (300, 2561, HF, HF, False, 0, True), (300, 3073, BF, BF, False, 0, True),
    (777, 4095, BF, BF, True, 0, True), (300, 4097, BF, BF, False, 0, True),
    (300, 8191, BF, BF, True, 0, True), (40, 8193, BF, BF, False, 0, True),  # generic
    (300, 511, F32, F32, False, 0, True), (300, 513, F32, F32, False, 0, True),
    (300, 201, F32, F32, True, 1, True), (600, 1023, F32, F32, True, 3, True),
    (300, 4095, F32, F32, False, 0, False), (40, 4097, F32, None, True, 0, True),
]


@pytest.mark.parametrize("rows,d,dtype,wdtype,gh,off,is_h", CASES,
                         ids=[f"{c[0]}x{c[1]}-{str(c[2])[6:]}-{c[5]}" for c in CASES])
def test_matches_oracle(rows, d, dtype, wdtype, gh, off, is_h):
    g, h, w, inv, ghv = _inputs(rows, d, dtype, wdtype, gh, off)
    saved = h if is_h else (h.float() * inv).to(dtype)
    dres = torch.empty_like(g)
    dx, dw = vk.fused_rmsnorm_residual_backward(g, saved, w, inv, saved_is_h=is_h, grad_h=ghv,
                                                dresidual_out=dres)
    g32, s32, inv32 = P.upcast(g), P.upcast(saved), P.upcast(inv)
    w32 = P.upcast(w) if w is not None else None
    if is_h:
        xhat = s32 * inv32
    else:
        xhat = s32
    rdx, rdw = ora.fused_rmsnorm_residual_backward(g32, xhat, w32, inv32)
    gw = g32 * w32 if w is not None else g32
    scale = np.abs(inv32 * gw) + np.abs(inv32 * xhat) * np.mean(np.abs(gw * xhat), -1, keepdims=True)
    if gh:
        rdx = rdx + P.upcast(ghv)
        scale = scale + np.abs(P.upcast(ghv))
    err = np.abs(P.upcast(dx).astype(np.float64) - rdx)
    # half an output ulp and the float32 row sum's error (see _parity's dx tolerance)
    ulp = {BF: 2.0 ** -8, HF: 2.0 ** -11, F32: 0.0}[dtype]
    sums = 1e-5 if dtype == F32 else P.DX_FLOOR
    assert np.all(err <= ulp * np.abs(rdx) + sums * scale + 2.0 ** -25)
    assert torch.equal(dx, dres)
    if w is not None:
        acc = np.einsum("rd,rd->d", g32.astype(np.float64), xhat.astype(np.float64))
        P.assert_dweight(P.upcast(dw), acc, "dweight")
        dx2, dw2 = vk.fused_rmsnorm_residual_backward(g, saved, w, inv, saved_is_h=is_h, grad_h=ghv)
        assert torch.equal(dx, dx2) and torch.equal(dw, dw2)


@pytest.mark.parametrize("rows,d,dtype", [(300, 1001, BF), (300, 4097, BF), (70, 601, F32)])
def test_dx_in_place_of_grad_h(rows, d, dtype):
    g, h, w, inv, gh = _inputs(rows, d, dtype, dtype, True, 0)
    code = _lib.TORCH_DTYPE_CODES[dtype]
    ws_bytes = vk.bwd_workspace_bytes(rows, d, g.device)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=g.device)

    def run(dx):
        dw = torch.empty(d, device=g.device)
        rc = _lib.load().velograd_rmsnorm_residual_bwd(
            g.data_ptr(), h.data_ptr(), 1, w.data_ptr(), inv.data_ptr(), dx_gh.data_ptr(),
            dx.data_ptr(), None, dw.data_ptr(), ws.data_ptr(), ws_bytes, rows, d, d, d, d, d, d,
            code, code, torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "bwd")
        return dx, dw

    dx_gh = gh
    want, want_dw = run(torch.empty_like(g))
    dx_gh = gh.clone()
    got, got_dw = run(dx_gh)
    # the same sums in another order: an output ulp, and float32 sums of `rows` terms
    tol = {BF: 2.0 ** -7, F32: 1e-5}[dtype]
    assert torch.allclose(got.double(), want.double(), rtol=tol, atol=tol)
    P.assert_dweight(P.upcast(got_dw), P.upcast(want_dw), "dweight")


@pytest.mark.parametrize("rows,d,fits", [(1100, 4099, False), (900, 4099, True),
                                         (1100, 4095, True)])
def test_noalloc_keeps_its_limit(rows, d, fits):
    g, h, w, inv, _ = _inputs(rows, d, BF, BF, False, 0)
    dx, dw = torch.empty_like(g), torch.empty(d, device=g.device)
    code = _lib.TORCH_DTYPE_CODES[BF]
    rc = _lib.load().velograd_rmsnorm_residual_bwd_noalloc(
        g.data_ptr(), h.data_ptr(), 1, w.data_ptr(), inv.data_ptr(), None, dx.data_ptr(), None,
        dw.data_ptr(), rows, d, d, d, d, d, d, code, code,
        torch.cuda.current_stream().cuda_stream)
    assert rc == (0 if fits else _lib.ERR_WORKSPACE_TOO_SMALL)
    if fits:
        want_dx, want_dw = vk.fused_rmsnorm_residual_backward(g, h, w, inv, saved_is_h=True)
        assert torch.equal(dx, want_dx) and torch.equal(dw, want_dw)
