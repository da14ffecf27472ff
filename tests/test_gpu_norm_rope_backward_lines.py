"""Both sides of the line between the generic kernel and the ring for short ragged rows of the norm +
RoPE backward, against the composition in 64 bits."""

import pytest
import torch

from test_gpu_norm_rope_backward_rows import test_norm_rope_backward as check

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("outer,seq,dim,dtype", [
    (3, 341, 10, BF), (4, 256, 10, BF), (1, 1100, 510, HF), (256, 1, 514, BF), (1, 257, 1002, HF),
    (256, 1, 6, F32), (1, 257, 254, F32), (64, 1, 258, F32), (65, 1, 510, F32),
])
def test_short_ragged_rows(outer, seq, dim, dtype):
    check(outer, seq, dim, dtype, dtype, 1e4, 1)
