"""fwd_vec_kernel's rows of any length and alignment: lengths around a chunk, the element-strided
rows' bound, one and two chunks a thread and the register layout's end; streams that start
anywhere in a 16-byte line, alike or not; every output form, with and without a residual."""

import numpy as np
import pytest
import torch

from oracle import fused_rmsnorm as ora
from velograd_amd import kernels as vk

from tests._parity import assert_within_ulp, gaussian, rel_err, FP32_REL_TOL, to_device, upcast

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


def _strided(rng, rows, dim, ld, off, dtype):
    """A [rows, dim] tensor of row stride ld whose first element is `off` elements into its
    allocation."""
    buf = to_device(gaussian(rng, (off + rows * ld,)), dtype)
    return buf[off:].as_strided((rows, dim), (ld, 1))


def _case(rows, dim, dtype, wdtype, with_res, offsets, ld_extra):
    rng = np.random.default_rng(dim * 7 + rows)
    x = _strided(rng, rows, dim, dim + ld_extra, offsets[0], dtype)
    r = _strided(rng, rows, dim, dim, offsets[1], dtype) if with_res else None
    w = None
    if wdtype is not None:
        w = to_device(gaussian(rng, (offsets[2] + dim,)), wdtype)[offsets[2]:]
    return x, r, w


def _up(t):
    return None if t is None else upcast(t.contiguous())


CASES = [
    # rows, dim, dtype, weight, residual, (x, residual, weight) offsets in elements, extra stride
    (5, 65, torch.bfloat16, torch.bfloat16, True, (0, 0, 0), 0),
    (9, 66, torch.float16, torch.float32, True, (1, 1, 1), 0),
    (7, 71, torch.bfloat16, torch.float32, False, (3, 0, 5), 2),
    (300, 511, torch.bfloat16, torch.bfloat16, True, (0, 0, 0), 0),
    (300, 513, torch.bfloat16, None, True, (2, 5, 0), 1),
    (129, 519, torch.bfloat16, torch.bfloat16, False, (7, 0, 3), 0),
    (64, 520, torch.bfloat16, torch.bfloat16, True, (1, 1, 1), 0),      # whole chunks, off a line
    (33, 3079, torch.float16, torch.float16, True, (0, 0, 0), 0),       # 384 chunks: two a thread
    (33, 3081, torch.bfloat16, torch.bfloat16, True, (0, 4, 1), 0),     # 385: one
    (17, 4095, torch.bfloat16, torch.bfloat16, True, (0, 0, 0), 0),
    (17, 4100, torch.bfloat16, torch.float32, True, (0, 0, 0), 0),
    (9, 8199, torch.bfloat16, torch.bfloat16, True, (0, 0, 0), 0),      # 1024 chunks
    (9, 8207, torch.bfloat16, torch.bfloat16, True, (0, 0, 0), 0),      # 1025: two a thread again
    (5, 16391, torch.bfloat16, torch.bfloat16, True, (0, 0, 0), 0),     # 2048: the last that fit
    (5, 16392, torch.bfloat16, torch.bfloat16, True, (1, 1, 1), 0),     # past them: generic
    (40, 67, torch.float32, torch.float32, True, (1, 0, 2), 0),
    (40, 1001, torch.float32, torch.float32, True, (0, 0, 0), 0),
    (40, 1537, torch.float32, None, False, (3, 0, 0), 1),
    (6, 8195, torch.float32, torch.float32, True, (0, 0, 0), 0),
]


@pytest.mark.parametrize("rows,dim,dtype,wdtype,with_res,offsets,ld_extra", CASES,
                         ids=[f"{c[0]}x{c[1]}-{str(c[2])[6:]}-{c[5]}" for c in CASES])
def test_plain_output(rows, dim, dtype, wdtype, with_res, offsets, ld_extra):
    x, r, w = _case(rows, dim, dtype, wdtype, with_res, offsets, ld_extra)
    y, h, inv = vk.fused_rmsnorm_residual_forward(x, r, w, 1e-6)
    ry, rh, rinv = ora.fused_rmsnorm_residual_forward(_up(x), _up(r), _up(w), 1e-6)
    if dtype == torch.float32:
        assert rel_err(upcast(y), ry) <= FP32_REL_TOL
        assert rel_err(upcast(h), rh) == 0.0
    else:
        assert_within_ulp(y, ry, 1, "y")
        assert_within_ulp(h, rh, 0, "h")
    assert rel_err(upcast(inv), rinv) <= FP32_REL_TOL


@pytest.mark.parametrize("rows,dim,dtype,offsets", [
    (3, 8, torch.bfloat16, (1, 0, 0)), (3, 9, torch.bfloat16, (7, 7, 0)),
    (3, 15, torch.float16, (1, 2, 3)), (70, 255, torch.bfloat16, (0, 0, 0)),
    (70, 513, torch.bfloat16, (0, 0, 1)), (20, 4095, torch.bfloat16, (0, 0, 0)),
    (20, 4100, torch.bfloat16, (0, 0, 0)), (5, 13, torch.float32, (1, 1, 1)),
    (20, 2051, torch.float32, (0, 0, 0)), (3, 7, torch.bfloat16, (0, 0, 0))])
@pytest.mark.parametrize("with_res", [True, False])
def test_fp8_output(rows, dim, dtype, offsets, with_res):
    x, r, w = _case(rows, dim, dtype, dtype, with_res, offsets, 0)
    yq, scale, _, inv = vk.fused_rmsnorm_residual_forward_fp8(x, r, w, 1e-5)
    codes, rscale, _, _ = ora.fused_rmsnorm_residual_forward_fp8(_up(x), _up(r), _up(w), 1e-5,
                                                                 inv_rms=upcast(inv))
    assert np.array_equal(yq.view(torch.uint8).cpu().numpy(), codes)
    assert np.array_equal(upcast(scale), rscale)


@pytest.mark.parametrize("fmt", ["e4m3", "e2m1"])
@pytest.mark.parametrize("rows,dim,dtype", [(9, 32, torch.bfloat16), (9, 1056, torch.bfloat16),
                                            (9, 4128, torch.float16), (9, 96, torch.float32)])
def test_mx_output_off_a_line(fmt, rows, dim, dtype):
    x, r, w = _case(rows, dim, dtype, dtype, True, (1, 2, 3), 0)
    yq, scales, _, inv = vk.fused_rmsnorm_residual_forward_mx(x, r, w, 1e-5, fmt=fmt)
    codes, rscales, _, _ = ora.fused_rmsnorm_residual_forward_mx(
        _up(x), _up(r), _up(w), 1e-5, fmt=fmt, inv_rms=upcast(inv))
    assert np.array_equal(yq.view(torch.uint8).cpu().numpy(), codes)
    assert np.array_equal(scales.view(torch.uint8).cpu().numpy(), rscales)


def test_nan_and_inf_stay_in_their_row():
    x, r, w = _case(6, 1001, torch.bfloat16, torch.bfloat16, True, (1, 1, 0), 0)
    x, r = x.clone(), r.clone()
    x[1, 0] = float("nan")        # the element before the first chunk
    x[3, 1000] = float("inf")     # after the last
    y, h, inv = vk.fused_rmsnorm_residual_forward(x, r, w, 1e-6)
    assert torch.isnan(y[1]).all() and torch.isnan(inv[1]).all()
    assert float(inv[3]) == 0.0 and torch.isnan(y[3, 1000]) and bool((y[3, :1000] == 0).all())
    for row in (0, 2, 4, 5):
        assert torch.isfinite(y[row]).all() and torch.isfinite(h[row]).all()
