"""The forwards' workgroup-to-row mapping (launch_plan.h: xcd_item) compiled for the CPU with
AddressSanitizer and UBSan (tests/xcd_run_check.cpp), and the forward over row counts around its
spans on the GPU: every row's outputs must be that row's."""

import os
import shutil
import subprocess

import pytest
import torch

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_mapping_is_a_permutation_in_runs(tmp_path):
    exe = tmp_path / "xcd_run_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-I", os.path.join(REPO, "velograd_amd", "csrc"),
                    os.path.join(HERE, "xcd_run_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 255, 256, 257, 1024, 1300])
@pytest.mark.parametrize("dim", [512, 4096, 20000])
def test_forward_rows_around_the_spans(rows, dim):
    from velograd_amd import kernels as vk
    gen = torch.Generator(device="cuda").manual_seed(rows * 31 + dim)
    x = torch.randn(rows, dim, generator=gen, device="cuda")
    r = torch.randn(rows, dim, generator=gen, device="cuda")
    y, h, inv = vk.fused_rmsnorm_residual_forward(x, r, None, 1e-6)
    assert torch.equal(h, x + r)
    want = 1.0 / torch.sqrt(h.double().square().mean(-1, keepdim=True) + 1e-6)
    # fp32 sums of dim squares in another order: a few ulps
    assert torch.allclose(inv.double(), want, rtol=4e-6, atol=0)
    assert torch.equal(y, h * inv)
