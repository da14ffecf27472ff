"""The norm + RoPE forward over sequences shorter than its tiles (decode steps), whose tiles take one
position of consecutive sequences, against the same composition in 64 bits."""

import pytest
import torch

from test_gpu_norm_rope_tiles import HALF_ULP, PAIR_ERR, _exact
from velograd_amd import kernels as vk

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32

CASES = [
    # outer, seq, dim, dtype, weight, residual, base
    (1, 1, 64, BF, BF, False, 1e4), (3, 1, 4096, BF, BF, False, 1e4),
    (1027, 1, 4096, BF, BF, False, 1e4), (1027, 1, 768, HF, F32, True, 1e4),
    (2050, 2, 512, BF, BF, False, 5e5), (515, 2, 4096, BF, BF, False, 0.5),
    (701, 3, 1000, BF, F32, False, 1e4), (401, 3, 3002, BF, BF, False, 1e4),   # ragged
    (1026, 1, 8194, BF, BF, False, 1e4), (517, 1, 8194, HF, HF, True, 1e4),    # two chunks a thread
    (1027, 1, 1024, F32, F32, False, 1e4), (403, 3, 4098, F32, F32, False, 5e5),
    (2050, 2, 6, F32, F32, False, 0.25), (518, 1, 2048, F32, None, True, 1e4),
]


@pytest.mark.parametrize("outer,seq,dim,dtype,wdtype,with_res,base", CASES,
                         ids=[f"{c[0]}x{c[1]}x{c[2]}-{str(c[3])[6:]}" for c in CASES])
def test_short_sequences(outer, seq, dim, dtype, wdtype, with_res, base):
    gen = torch.Generator(device="cuda").manual_seed(outer + dim)

    def rand(*shape, dt=dtype):
        return torch.randn(shape, generator=gen, device="cuda").to(dt)

    x = rand(outer, seq, dim)
    r = rand(outer, seq, dim) if with_res else None
    w = 1 + rand(dim, dt=wdtype) / 8 if wdtype is not None else None
    y, h, inv = vk.rmsnorm_rope_forward(x, w, 1e-6, base, r)
    ry, rh, rinv, pair = _exact(x, r, w, 1e-6, base)
    bound = HALF_ULP[dtype] * ry.abs() + PAIR_ERR * pair + 1e-30
    assert bool(((y.double() - ry).abs() <= bound).all())
    assert bool(((inv.double() / rinv - 1).abs() <= 1e-6).all())
    assert torch.equal(h, rh.to(dtype) if with_res else x)
