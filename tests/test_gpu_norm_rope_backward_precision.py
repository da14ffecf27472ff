"""The norm + RoPE backward over rows that are not whole chunks keeps the precision of angles formed at
every row: its error against 64 bits is that of the same arithmetic in float32 with each row's cos
and sin rounded from 64 bits, not that of a rotation advanced in float32 (dx 2.8 times, dweight 1.5
times as far off)."""

import pytest
import torch

from velograd_amd import kernels as vk

pytestmark = pytest.mark.gpu

# the kernel's rotation is one more rounding of cos and sin (1 ulp against half), which adds about a
# tenth to the error of the four roundings that follow it
FACTOR = 1.2
SLOTS, WAVES = 512, 16  # row slots of a walk, and waves of dweight's second stage

CASES = [
    # outer, seq, dim, dtype
    (1, 8192, 1002, torch.float32), (2, 4096, 2046, torch.float32), (1, 4096, 4094, torch.float32),
    (1, 8192, 2050, torch.float16), (1, 8192, 4098, torch.bfloat16),
]


def _error(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("outer,seq,dim,dtype", CASES,
                         ids=[f"{c[0]}x{c[1]}x{c[2]}-{str(c[3])[6:]}" for c in CASES])
def test_ragged_rows_hold_their_precision(outer, seq, dim, dtype):
    gen = torch.Generator(device="cuda").manual_seed(dim)
    rows = outer * seq
    g, h = (torch.randn(rows, dim, generator=gen, device="cuda").to(dtype) for _ in range(2))
    w = (1 + torch.randn(dim, generator=gen, device="cuda") / 8).to(dtype)
    inv = 1.0 / torch.sqrt(h.float().square().mean(-1, keepdim=True) + 1e-6)
    freq = 1e4 ** (-torch.arange(0, dim, 2, dtype=torch.float64, device="cuda") / dim)
    ang = torch.outer(torch.arange(seq, dtype=torch.float64, device="cuda"), freq).repeat(outer, 1)

    def in_order(terms):
        acc = torch.zeros_like(terms[0])
        for row in terms:
            acc = acc + row
        return acc

    def backward(t):  # every operation in t, the row mean from 64 bits
        c, s = ang.cos().to(t), ang.sin().to(t)
        a, b = g.to(t)[:, 0::2], g.to(t)[:, 1::2]
        gr = torch.stack((a * c + b * s, b * c - a * s), -1).flatten(-2)
        xhat = h.to(t) * inv.to(t)
        gw = gr * w.to(t)
        mean = (gw.double() * xhat.double()).mean(-1, keepdim=True).to(t)
        # a slot's rows, then the slots of each wave, then the waves
        partial = in_order((gr * xhat).view(rows // SLOTS, SLOTS, dim))
        dw = in_order(in_order(partial.view(SLOTS // WAVES, WAVES, dim)))
        return inv.to(t) * (gw - xhat * mean), dw

    rdx, rdw = backward(torch.float64)
    fdx, fdw = backward(torch.float32)
    dx, dw = vk.rmsnorm_rope_backward(g.view(outer, seq, dim), h.view(outer, seq, dim), w,
                                      inv.view(outer, seq, 1))
    if dtype == torch.float32:
        assert _error(dx.view(rows, dim), rdx) <= FACTOR * _error(fdx, rdx)
    assert _error(dw, rdw) <= FACTOR * _error(fdw, rdw)
