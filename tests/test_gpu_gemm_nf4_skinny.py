"""qlora_gemm_nf4 for a few rows (the decode path, up to 32 rows): the 4-bit linear whose
workgroups hold 16 or 32 weight rows and split K over their waves, against an fp64 product of
the weight qlora_nf4_dequant writes, at the edges of its tiles."""

import pytest
import torch

from hackathon_amd import nf4, quant

pytestmark = pytest.mark.gpu

CASES = [
    # M, N, K, nested, dtype, blocksize, LoRA segment
    (1, 8, 64, True, torch.bfloat16, 64, False),        # one 64-k lane group, one row of x
    (4, 18944, 3584, True, torch.bfloat16, 64, True),   # Qwen2.5-7B gate/up, decoding
    (16, 8200, 320, True, torch.float16, 64, True),     # 32-row workgroups, ragged N and K
    (17, 3584, 18944, True, torch.bfloat16, 256, True),  # second group of x rows, 16-wave K
    (32, 8205, 448, False, torch.float16, 64, False),   # N not a multiple of 4, plain absmax
    (31, 250, 1024, True, torch.bfloat16, 1024, True),  # a block per 1024 weights
]


@pytest.mark.parametrize("M,N,K,nested,dtype,bs,lora", CASES)
def test_few_rows_against_fp64(M, N, K, nested, dtype, bs, lora):
    print(f"gemm_nf4 M={M} N={N} K={K} nested={nested} {dtype} bs={bs} lora={lora}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    packed, st = quant.quantize_nf4(torch.randn(N, K, device="cuda", generator=g) * 0.02, bs,
                                    compress_statistics=nested)
    x = torch.randn(M, K + 8, device="cuda", generator=g).to(dtype)[:, :K]  # row stride K + 8
    bias = (torch.randn(N, device="cuda", generator=g) * 0.1).to(dtype)
    a2 = b2 = None
    if lora:
        a2 = torch.zeros(M, 64, device="cuda", dtype=dtype)
        a2[:, :48] = torch.randn(M, 48, device="cuda", generator=g).to(dtype)
        b2 = torch.zeros(N, 64, device="cuda", dtype=dtype)
        b2[:, :48] = (torch.randn(N, 48, device="cuda", generator=g) * 0.02).to(dtype)
    out = torch.full((M + 1, N + 3), 7.0, device="cuda", dtype=dtype)
    got = nf4.gemm_nf4(x, packed, st, out=out[:M, :N], a2=a2, b2=b2, bias=bias, alpha=0.5)
    torch.cuda.synchronize()
    w = nf4.dequantize_nf4(packed, st, dtype).double()
    ref, mag = x.double() @ w.t(), x.double().abs() @ w.abs().t()
    if lora:
        ref += a2.double() @ b2.double().t()
        mag += a2.double().abs() @ b2.double().abs().t()
    ref = 0.5 * ref + bias.double()
    # fp32 accumulation over K + 64 terms, then one rounding to the 16-bit output
    ulp16 = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = (K + 64) * 2.0 ** -24 * 0.5 * mag + ulp16 * ref.abs() + 1e-6
    assert torch.all((got.double() - ref).abs() <= bound)
    assert (out[M:] == 7).all() and (out[:, N:] == 7).all()  # nothing outside [M, N] written


def test_few_rows_zero_weight_past_k_meets_no_inf():
    """A chunk's lanes past K multiply zeros: an infinity in x's first columns (where those
    lanes' clamped loads point) reaches only the products it belongs to."""
    packed, st = quant.quantize_nf4(torch.zeros(64, 320, device="cuda"), 64)
    x = torch.ones(2, 320, device="cuda", dtype=torch.bfloat16)
    got = nf4.gemm_nf4(x, packed, st)
    w = nf4.dequantize_nf4(packed, st, torch.bfloat16)
    assert torch.isfinite(got).all()
    x[0, 0] = float("inf")
    got = nf4.gemm_nf4(x, packed, st)
    assert torch.equal(got[1], nf4.gemm_nf4(x[1:], packed, st)[0])
    assert torch.equal(got[0].isnan(), (x[:1].double() @ w.double().t())[0].isnan())
