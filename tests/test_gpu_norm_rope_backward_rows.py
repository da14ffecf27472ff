"""bwd_rope_ring_kernel over rows that are not whole chunks or waves, one and two chunks a thread,
and walks whose positions neither advance nor return to their first one (they are evaluated
afresh at each sequence's start), against the same composition in 64 bits."""

import pytest
import torch

from velograd_amd import kernels as vk

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32
# half an output ulp of dx; the float32 rotation's drift over 16 rows (about 3 * 2^-24 a step), the
# row sum's and the statistic's error, relative to dx's operands
HALF_ULP = {BF: 2.0 ** -8, HF: 2.0 ** -11, F32: 2.0 ** -24}
OPERANDS = 8e-6

CASES = [
    # outer, seq, dim, dtype, weight, base, offset in elements
    (3, 700, 8, BF, BF, 1e4, 0), (1, 300, 10, BF, BF, 1e4, 0), (2, 515, 74, HF, F32, 1e4, 0),
    (5, 1000, 512, BF, BF, 1e4, 0),       # whole waves; sequences that no walk divides
    (3, 333, 1000, BF, BF, 5e5, 0), (1, 520, 3002, BF, BF, 1e4, 1),
    (1, 300, 4096, BF, BF, 1e4, 3),       # off a line
    (700, 3, 4094, BF, BF, 1e4, 0),       # a new sequence every few rows
    (2, 300, 4098, BF, BF, 1e4, 0),       # 513 chunks: two a thread
    (1, 300, 8190, BF, None, 1e4, 0), (3, 111, 8192, BF, BF, 1e4, 0),
    (1, 40, 8194, BF, BF, 1e4, 0),        # past them
    (2, 300, 6, F32, F32, 1e4, 0), (5, 1000, 258, F32, F32, 0.5, 0),
    (1, 600, 2046, F32, F32, 1e4, 1), (3, 171, 4094, F32, F32, 1e4, 0),
    (1, 40, 4098, F32, F32, 1e4, 0), (1, 9, 2, F32, F32, 1e4, 0),
]


@pytest.mark.parametrize("outer,seq,dim,dtype,wdtype,base,off", CASES,
                         ids=[f"{c[0]}x{c[1]}x{c[2]}-{str(c[3])[6:]}" for c in CASES])
def test_norm_rope_backward(outer, seq, dim, dtype, wdtype, base, off):
    gen = torch.Generator(device="cuda").manual_seed(seq + dim)

    def rand(n, dt):
        return torch.randn(n + off, generator=gen, device="cuda").to(dt)[off:]

    g = rand(outer * seq * dim, dtype).view(outer, seq, dim)
    h = rand(outer * seq * dim, dtype).view(outer, seq, dim)
    w = 1 + rand(dim, wdtype) / 8 if wdtype is not None else None
    inv = 1.0 / torch.sqrt(h.float().square().mean(-1, keepdim=True) + 1e-6)
    dx, dw = vk.rmsnorm_rope_backward(g, h, w, inv, base)

    freq = base ** (-torch.arange(0, dim, 2, dtype=torch.float64, device="cuda") / dim)
    ang = torch.outer(torch.arange(seq, dtype=torch.float64, device="cuda"), freq)
    c, s = ang.cos(), ang.sin()
    a, b = g.double()[..., 0::2], g.double()[..., 1::2]
    gr = torch.stack((a * c + b * s, b * c - a * s), -1).flatten(-2)
    pair = torch.sqrt(a * a + b * b).repeat_interleave(2, -1)
    wd = w.double() if w is not None else torch.ones(dim, dtype=torch.float64, device="cuda")
    xhat, iv = h.double() * inv.double(), inv.double()
    gw = gr * wd
    rdx = iv * (gw - xhat * (gw * xhat).mean(-1, keepdim=True))
    scale = iv * (pair * wd.abs() + xhat.abs() * (pair * wd.abs() * xhat.abs()).mean(-1, keepdim=True))
    bound = HALF_ULP[dtype] * rdx.abs() + OPERANDS * scale + 1e-7
    assert bool(((dx.double() - rdx).abs() <= bound).all())
    if w is None:
        assert dw is None
        return
    terms = gr * xhat
    rdw = terms.flatten(0, -2).sum(0)
    mass = (pair * xhat.abs()).flatten(0, -2).sum(0)
    assert bool(((dw.double() - rdw).abs() <= 1e-5 * mass).all())
    dx2, dw2 = vk.rmsnorm_rope_backward(g, h, w, inv, base)
    assert torch.equal(dx, dx2) and torch.equal(dw, dw2)
