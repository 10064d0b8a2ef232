"""The fused dropout + down-projection at few rows, where its K split goes down to three chunks
of 64 per split (waves without a chunk, a last split that is shorter)."""

import pytest
import torch

from test_gpu_layers import test_dropout_down_vs_dropout_kernel_and_fp64 as _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,slots,dtype,p", [
    (1, 384, 1, torch.bfloat16, 0.05),    # two splits of 3 chunks
    (1, 320, 2, torch.float16, 0.3),      # too short to split
    (16, 896, 3, torch.bfloat16, 0.05),   # 14 chunks: 4 + 4 + 4 + 2
    (33, 4928, 4, torch.float16, 0.1),    # 77 chunks over 16 splits
    (1001, 3584, 1, torch.float16, 0.05), # 63 row blocks, 4 splits
    (2048, 896, 3, torch.bfloat16, 0.1),  # 128 row blocks, 2 splits: the chip just full
    (2049, 896, 1, torch.bfloat16, 0.1),  # one block more: no split
])
def test_short_splits(M, K, slots, dtype, p):
    _check(M, K, slots, dtype, p)
