"""The grouped dequantisations on both sides of the output size up to which they keep their
results in the caches: bit-identical to the single-weight entries (exact)."""

import pytest
import torch

from hackathon_amd import nf4, quant

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    [(64, 128)],                            # one weight, one tile
    [(4096, 4096)],                         # 32 MiB
    [(4104, 4096)],                         # one 8-row step more
    [(2048, 4096), (1024, 4096), (1024, 4096)],
    [(2048, 4096), (1024, 4096), (1032, 4096)],
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_group_equals_single(shapes, dtype):
    print(f"nf4 group {shapes} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(len(shapes) + shapes[0][0])
    K = shapes[0][1]
    items = [quant.quantize_nf4(torch.randn(n, k, device="cuda", generator=g) * 0.02, 64)
             for n, k in shapes]
    rows = [n for n, _ in shapes]
    w = torch.empty(sum(rows), K, dtype=dtype, device="cuda")
    wt = torch.empty(K, sum(rows), dtype=dtype, device="cuda")
    nf4._group_call("qlora_nf4_dequant_group", items, list(w.split(rows)), dtype)
    nf4._group_call("qlora_nf4_dequant_t_group", items, list(wt.split(rows, dim=1)), dtype,
                    wt.stride(0))
    for (packed, state), part in zip(items, w.split(rows)):
        one = nf4.dequantize_nf4(packed, state, dtype)
        assert torch.equal(part.view(torch.int16), one.view(torch.int16))
    assert torch.equal(wt.view(torch.int16), w.t().contiguous().view(torch.int16))
