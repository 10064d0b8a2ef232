"""Flash attention where the launch changes form: numbers of work items on both sides of one and
two per compute unit (the order in which workgroups take them changes there), lengths that end
inside a tile. Reference and bounds as in test_gpu_attention (fp32 causal softmax attention;
output rtol = atol = 1e-2 for operands and probabilities rounded to 16 bits, gradients 1e-2
relative), the same for fp16, whose rounding is finer."""

import math

import pytest
import torch

from hackathon_amd import attention
from test_gpu_attention import _ref, _ref_grads, _rel_err

pytestmark = pytest.mark.gpu


# (heads, length): 128-row items 1, 255, 256, 257, 300, 511, 512, 513; the 64-row ones twice as many
@pytest.mark.parametrize("H,S", [(1, 1), (85, 383), (64, 512), (257, 127), (30, 1250), (73, 891),
                                 (64, 1000), (57, 1100)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_item_is_taken_once(H, S, dtype):
    print(f"attention items H={H} S={S} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(H + S)
    q, k, v = (torch.randn(1, S, h, 128, device="cuda", generator=g).to(dtype).transpose(1, 2)
               for h in (H, 1, 1))
    do = torch.randn(1, S, H, 128, device="cuda", generator=g).to(dtype)
    scale = 1.0 / math.sqrt(128)
    o, lse = attention.attn_fwd(q, k, v, scale)
    o_ref, lse_ref = _ref(q, k, v, scale)
    torch.testing.assert_close(o.transpose(1, 2).float(), o_ref, rtol=1e-2, atol=1e-2)
    torch.testing.assert_close(lse, lse_ref, rtol=0, atol=1e-4)
    del o_ref
    for name, got, want in zip(("dq", "dk", "dv"), attention.attn_bwd(q, k, v, o, lse, do, scale),
                               _ref_grads(q, k, v, do, scale)):
        # one key of length 1: dq and dk are exactly zero in the reference
        assert (got.float() - want).norm() <= 1e-2 * want.norm() + 1e-3, name


@pytest.mark.parametrize("row_stride", [(1 << 24) - 8, 1 << 24])
def test_row_strides_around_the_whole_tile_loads(row_stride):
    """Rows 32 MiB apart: whole tiles go out as one piece below 2^24 elements and load by load
    from there on; either way the same bits as with dense rows."""
    S = 70
    buf = torch.empty(S * row_stride, device="cuda", dtype=torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = dense = [torch.randn(1, 1, S, 128, device="cuda", generator=g).to(torch.bfloat16)
                       for _ in range(3)]
    far = [buf.as_strided((1, 1, S, 128), (S * row_stride, 128, row_stride, 1), 128 * i)
           for i in range(3)]
    for a, b in zip(far, dense):
        a.copy_(b)
    do = torch.randn(1, S, 1, 128, device="cuda", generator=g).to(torch.bfloat16)
    scale = 1.0 / math.sqrt(128)
    want = attention.attn_fwd(q, k, v, scale)
    got = attention.attn_fwd(*far, scale)
    want += tuple(attention.attn_bwd(q, k, v, *want, do, scale))
    got += tuple(attention.attn_bwd(*far, *got, do, scale))
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), got, want):
        assert torch.equal(a, b), name


# (heads, length): more than two 64-row workgroups per compute unit with few blocks a head, where
# 128 rows are taken from fewer items than two per unit
@pytest.mark.parametrize("H,S", [(280, 65), (448, 100), (224, 129), (112, 512), (168, 383)])
def test_many_short_heads(H, S):
    test_every_item_is_taken_once(H, S, torch.bfloat16)
