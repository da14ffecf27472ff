"""fwd_rope_tile_kernel: tiles of one, two and four positions against sequences that end inside
them, several short rows a workgroup, one and two chunks a thread, rows whose last chunk overlaps
the one before it, streams off a 16-byte line, and the rows past the registers (generic kernel),
against the same composition in 64 bits."""

import pytest
import torch

from velograd_amd import kernels as vk

pytestmark = pytest.mark.gpu

# half an output ulp, relative; the rotation's and the statistic's float32 error, relative to the
# pair (cos and sin within 2 ulps, three float steps of 3 ulps, inv_rms within 1e-6)
HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}
PAIR_ERR = 3e-6


def _exact(x, r, w, eps, base):
    h = x.double() + (r.double() if r is not None else 0.0)
    mean_sq = h.square().mean(-1, keepdim=True).clamp(min=1e-12)
    inv = 1.0 / torch.sqrt(mean_sq + eps)
    n = h * inv * (w.double() if w is not None else 1.0)
    seq, d = x.shape[-2:]
    freq = base ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    ang = torch.outer(torch.arange(seq, dtype=torch.float64, device=x.device), freq)
    a, b = n[..., 0::2], n[..., 1::2]
    c, s = ang.cos(), ang.sin()
    y = torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)
    pair = torch.sqrt(a * a + b * b).repeat_interleave(2, -1)
    return y, h, inv, pair


CASES = [
    # (bases are float32 numbers, as the entry point takes them: 0.3 is 4e-8 of itself off, which at
    # position 5000 and 3.3 radians a position turns a pair by up to 5e-4)
    # outer, seq, dim, dtype, weight, residual, base, offset in elements
    (1, 1, 8, torch.bfloat16, torch.bfloat16, False, 1e4, 0),
    (3, 1, 64, torch.bfloat16, None, True, 1e4, 0),
    (2, 2, 10, torch.float16, torch.float32, False, 1e4, 0),
    (5, 3, 74, torch.bfloat16, torch.bfloat16, True, 1e4, 2),
    (2, 511, 768, torch.bfloat16, torch.bfloat16, False, 1e4, 0),
    (1, 1023, 768, torch.bfloat16, torch.bfloat16, False, 5e5, 0),     # tiles of two
    (1, 4097, 768, torch.bfloat16, torch.bfloat16, False, 1e4, 0),     # of four
    (3, 1027, 1000, torch.bfloat16, torch.float32, False, 1e4, 0),
    (2, 1030, 520, torch.bfloat16, torch.bfloat16, True, 1e4, 1),      # odd start
    (1, 1030, 3002, torch.bfloat16, torch.bfloat16, False, 1e4, 0),
    (1, 1030, 4100, torch.float16, torch.float16, True, 1e4, 0),
    (1, 70, 8192, torch.bfloat16, torch.bfloat16, False, 1e4, 0),      # 1024 chunks
    (1, 1026, 8194, torch.bfloat16, torch.bfloat16, False, 1e4, 0),    # two a thread
    (1, 514, 16384, torch.bfloat16, torch.bfloat16, True, 1e4, 0),
    (1, 6, 16386, torch.bfloat16, torch.bfloat16, False, 1e4, 0),      # generic
    (4, 300, 256, torch.bfloat16, torch.bfloat16, False, 0.5, 0),      # steps past a radian
    (1, 9, 2, torch.float32, torch.float32, False, 1e4, 0),            # generic: under a chunk
    (2, 2050, 6, torch.float32, torch.float32, False, 1e4, 0),
    (1, 5000, 512, torch.float32, torch.float32, True, 1e4, 0),
    (1, 5000, 512, torch.float32, torch.float32, False, 0.25, 0),
    (2, 1030, 4098, torch.float32, torch.float32, False, 5e5, 3),
    (1, 700, 8192, torch.float32, torch.float32, True, 1e4, 0),
]


@pytest.mark.parametrize("outer,seq,dim,dtype,wdtype,with_res,base,off", CASES,
                         ids=[f"{c[0]}x{c[1]}x{c[2]}-{str(c[3])[6:]}" for c in CASES])
def test_norm_rope_tiles(outer, seq, dim, dtype, wdtype, with_res, base, off):
    gen = torch.Generator(device="cuda").manual_seed(seq * 7 + dim)

    def rand(n, dt):
        return torch.randn(n + off, generator=gen, device="cuda").to(dt)[off:]

    x = rand(outer * seq * dim, dtype).view(outer, seq, dim)
    r = rand(outer * seq * dim, dtype).view(outer, seq, dim) if with_res else None
    w = 1 + rand(dim, wdtype) / 8 if wdtype is not None else None
    y, h, inv = vk.rmsnorm_rope_forward(x, w, 1e-6, base, r)
    ry, rh, rinv, pair = _exact(x, r, w, 1e-6, base)
    bound = HALF_ULP[dtype] * ry.abs() + PAIR_ERR * pair + 1e-30
    assert bool(((y.double() - ry).abs() <= bound).all())
    assert bool(((inv.double() / rinv - 1).abs() <= 1e-6).all())
    assert torch.equal(h, rh.to(dtype) if with_res else x)
