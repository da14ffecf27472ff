"""The register-resident forward issues all of a row's loads before it waits for any of them: its
gfx950 assembly (hipcc, no GPU needed) holds no wait on vector memory between the first load and
the last one of a row.  A wait there costs 2-10% of the pass and shows in no result.  (An fp32 weight
beside 2-byte activations, with two or more chunks a thread, is loaded after the wait on purpose.)"""

import os
import re
import shutil
import subprocess

import pytest

from velograd_amd import build

SRC = os.path.join(build.CSRC_DIR, "rmsnorm_residual.hip")
HOST_PART = "// Launch-shape knobs, read once per process"
BF16, F16, F32 = 2, 1, 0
DTYPE, FP8, MXFP8, MXFP4, DTYPE_LATE_H = 0, 1, 2, 3, 5
CHUNKS, ANY_NO_RES = 0, 2

# dtype, weight dtype, chunks a thread, output, rows
KERNELS = [(BF16, BF16, nv, out, CHUNKS) for nv in (1, 2, 3, 4)
           for out in (DTYPE, DTYPE_LATE_H, FP8, MXFP8, MXFP4)]
KERNELS += [(F16, F32, 2, FP8, CHUNKS), (BF16, F32, 2, DTYPE, CHUNKS), (BF16, F32, 1, DTYPE, CHUNKS),
            (F32, F32, 2, DTYPE, CHUNKS)]
KERNELS += [(BF16, BF16, 1, out, ANY_NO_RES) for out in (FP8, MXFP8, MXFP4)]


def _early_waits(body, weight_late):
    """The waits between the first and the last of the loads before the first store or barrier;
    `weight_late`: of the activations' (non-temporal) alone."""
    seq = []
    for line in body:
        line = line.strip()
        if line.startswith(("global_store", "s_barrier")):
            break
        if line.startswith("global_load") or (line.startswith("s_waitcnt") and "vmcnt" in line):
            seq.append(line)
    loads = [i for i, line in enumerate(seq)
             if line.startswith("global_load") and (not weight_late or line.split()[-1] == "nt")]
    assert len(loads) >= 2, seq
    return [line for line in seq[:loads[-1]] if line.startswith("s_waitcnt")]


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not available")
def test_no_wait_between_a_rows_loads(tmp_path):
    with open(SRC) as f:
        device = f.read().split(HOST_PART)[0]
    unit = tmp_path / "forward.hip"
    unit.write_text(device + "".join(
        f"template __global__ void fwd_vec_kernel<{', '.join(map(str, k))}>(FwdArgs);\n"
        for k in KERNELS) + "}  // namespace\n")
    asm = tmp_path / "forward.s"
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-Wall")]
    subprocess.run([build.find_hipcc(), *flags, "-S", "--cuda-device-only", "-I", build.INCLUDE_DIR,
                    "-I", build.CSRC_DIR, str(unit), "-o", str(asm)],
                   check=True, capture_output=True, text=True)
    bodies, name = {}, None
    for line in asm.read_text().splitlines():
        m = re.match(r"_Z\w*14fwd_vec_kernelI((?:Li\d+E){5})E\w*:", line)
        if m:
            name = tuple(int(v) for v in re.findall(r"Li(\d+)E", m.group(1)))
            bodies[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name is not None:
            bodies[name].append(line)
    assert set(KERNELS) <= set(bodies)
    early = {k: _early_waits(bodies[k], k[0] != F32 and k[1] == F32 and k[2] > 1) for k in KERNELS}
    assert not any(early.values()), {k: w for k, w in early.items() if w}
