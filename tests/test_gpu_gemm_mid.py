"""The NT GEMM's smaller tiles (gemm_mid.hip: 128 x 128, 64 x 128, 128 x 256), which
qlora_gemm_nt_cat takes where 256 x 256 tiles would leave CUs idle: ragged edges, both K
segments, split K, every epilogue, against an fp64 product."""

import pytest
import torch

from hackathon_amd import gemm

pytestmark = pytest.mark.gpu

CASES = [
    # M, N, K, LoRA segment, dtype: the tile the cost model takes
    (1001, 3584, 3584, 64, torch.float16),    # 128 x 128, the last tile row 105 high
    (2048, 1536, 8960, 0, torch.bfloat16),    # 128 x 128, 140 steps
    (257, 3583, 1024, 128, torch.bfloat16),   # one row in the last tile row, odd N
    (2048, 512, 1536, 64, torch.bfloat16),    # 64 x 128, one workgroup per CU
    (333, 1000, 3584, 64, torch.float16),     # 64 x 128, K split
    (4095, 500, 1536, 0, torch.bfloat16),     # 64 x 128, N not a multiple of 8
    (333, 18944, 3584, 64, torch.bfloat16),   # 128 x 256
    (333, 3584, 18944, 128, torch.bfloat16),  # 128 x 256, K split
    (300, 512, 128, 0, torch.bfloat16),       # two K steps: fewer than the stages
    (600, 512, 64, 64, torch.float16),        # one step of each segment
    (64, 3584, 3584, 64, torch.bfloat16),     # few rows: the 256-row tile's split count
]


def _bound(ref, mag, K, ulp16):
    # fp32 accumulation over the K terms (and the partials), then one rounding
    return (K + 16) * 2.0 ** -24 * mag + ulp16 * ref.abs() + 1e-6


@pytest.mark.parametrize("M,N,K,K2,dtype", CASES)
def test_mid_tiles_against_fp64(M, N, K, K2, dtype):
    print(f"gemm_nt_cat M={M} N={N} K={K} K2={K2} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    b = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(dtype)
    a2 = b2 = None
    ref, mag = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    if K2:
        a2 = torch.randn(M, K2, device="cuda", generator=g).to(dtype)
        b2 = (torch.randn(N, K2, device="cuda", generator=g) * 0.05).to(dtype)
        ref += a2.double() @ b2.double().t()
        mag += a2.double().abs() @ b2.double().abs().t()
    ulp16 = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    pitch = (N + 7) // 8 * 8 + 8
    out = torch.full((M + 1, pitch), 7.0, device="cuda", dtype=dtype)
    bias = torch.randn(N, device="cuda", generator=g).to(dtype)
    got = gemm.gemm_nt_cat(a, b, a2, b2, out[:M, :N], bias=bias, alpha=0.5)
    want = 0.5 * ref + bias.double()
    assert torch.all((got.double() - want).abs() <= _bound(want, 0.5 * mag, K + K2, ulp16))
    assert (out[M:] == 7).all() and (out[:, N:] == 7).all()  # nothing outside [M, N] written
    # fp32 output: no 16-bit rounding
    got32 = torch.empty(M, N, device="cuda", dtype=torch.float32)
    gemm.gemm_nt_cat(a, b, a2, b2, got32)
    assert torch.all((got32.double() - ref).abs() <= _bound(ref, mag, K + K2, 2.0 ** -23))
    # the residual form is the product rounded, then the add rounded, bit for bit
    if N % 8 == 0:
        res = torch.randn(M, N, device="cuda", generator=g).to(dtype)
        plain = gemm.gemm_nt_cat(a, b, a2, b2, torch.empty(M, N, device="cuda", dtype=dtype))
        fused = gemm.gemm_nt_cat(a, b, a2, b2, torch.empty(M, N, device="cuda", dtype=dtype),
                                 residual=res)
        assert torch.equal(fused, res + plain)
