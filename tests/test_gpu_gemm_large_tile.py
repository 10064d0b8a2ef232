"""The NT GEMM's 256-row tile where the planner keeps it: ragged M and N on both tile widths, output
rows that no vector store takes, the residual add and split K, against an fp64 product. Each case
names the tile and split it must run (qlora_gemm_nt_plan)."""

import pytest
import torch

from hackathon_amd import gemm

pytestmark = pytest.mark.gpu

CASES = [
    # M, N, K, K2, dtype, ldc, plan
    (2050, 4604, 64, 64, torch.bfloat16, 4604, (256, 256, 1)),   # one step of each segment
    (3001, 3005, 128, 0, torch.float16, 3005, (256, 256, 1)),    # odd N, odd row length
    (2050, 4612, 128, 128, torch.bfloat16, 4613, (256, 256, 1)),  # unaligned output rows
    (4001, 3584, 128, 64, torch.bfloat16, 3584, (256, 224, 1)),  # 224 wide, ragged M
    (3001, 3584, 64, 0, torch.float16, 3592, (256, 224, 1)),
    (1001, 4604, 8192, 64, torch.bfloat16, 4604, (256, 256, 3)),  # split K, four outputs a thread
    (1500, 3005, 8192, 0, torch.float16, 3005, (256, 256, 3)),   # split K, one output a thread
    (1500, 3584, 8192, 64, torch.bfloat16, 3584, (256, 256, 3)),
]


@pytest.mark.parametrize("M,N,K,K2,dtype,ldc,plan", CASES)
def test_against_fp64(M, N, K, K2, dtype, ldc, plan):
    print(f"large tile M={M} N={N} K={K} K2={K2} {dtype} ldc={ldc}", flush=True)
    assert gemm.nt_plan(M, N, K) == plan
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
    bias = torch.randn(N, device="cuda", generator=g).to(dtype)
    ulp16 = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    buf = torch.full(((M + 1) * ldc,), 7.0, device="cuda", dtype=dtype)
    out = buf.as_strided((M, N), (ldc, 1))
    got = gemm.gemm_nt_cat(a, b, a2, b2, out, bias=bias, alpha=0.5)
    want = 0.5 * ref + bias.double()
    # fp32 accumulation over the K + K2 terms (and the partials), then one rounding
    bound = (K + K2 + 16) * 2.0 ** -24 * 0.5 * mag + ulp16 * want.abs() + 1e-6
    assert torch.all((got.double() - want).abs() <= bound)
    assert (buf[M * ldc:] == 7).all()
    if ldc > N:
        assert (buf[:M * ldc].view(M, ldc)[:, N:] == 7).all()
    got32 = gemm.gemm_nt_cat(a, b, a2, b2, torch.empty(M, N, device="cuda"))
    bound = (K + K2 + 16) * 2.0 ** -24 * mag + 2.0 ** -23 * ref.abs() + 1e-6
    assert torch.all((got32.double() - ref).abs() <= bound)
    del ref, mag, want, bound
    # the residual form is the product rounded, then the add rounded, bit for bit
    ldr = (N + 7) // 8 * 8 + 8
    res = torch.randn(M, ldr, device="cuda", generator=g).to(dtype)[:, :N]
    plain = gemm.gemm_nt_cat(a, b, a2, b2, torch.empty(M, N, device="cuda", dtype=dtype))
    fused = gemm.gemm_nt_cat(a, b, a2, b2, out, residual=res)
    assert torch.equal(fused, res + plain)
    # accumulating: the 256-row tile's own split, whatever the plan
    acc = got32.clone()
    gemm.gemm(a, b, out=acc, beta=2.0, alpha=0.5)
    alone = gemm.gemm(a, b, out_dtype=torch.float32)
    torch.testing.assert_close(acc, 2.0 * got32 + 0.5 * alone, rtol=1e-4, atol=1e-3)
