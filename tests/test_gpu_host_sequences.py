"""The 4-bit LoRA layers whose launches the native host code queues (csrc/host/host.cpp), at the
operand forms a caller may hand in, against an fp64 product."""

import pytest
import torch

from hackathon_amd import _host, _lib, gemm, lora, nf4, quant

pytestmark = pytest.mark.gpu


def _layer(N, K, seed, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    packed, st = quant.quantize_nf4(torch.randn(N, K, device="cuda", generator=g) * 0.02, 64)
    a = torch.randn(16, K, device="cuda", generator=g) / K ** 0.5
    b = torch.randn(N, 16, device="cuda", generator=g) * 0.05
    return g, packed, st, a, b


def _check(y, x, packed, st, a, b, bias, dtype=torch.bfloat16):
    w = nf4.dequantize_nf4(packed, st, dtype).double()
    K = w.shape[1]
    a16, sb = a.to(dtype).double(), (2.0 * b).to(dtype).double()
    u = x.double() @ a16.t()
    ref = x.double() @ w.t() + u @ sb.t() + bias.double()
    mag = x.double().abs() @ w.abs().t() + (x.double().abs() @ a16.abs().t()) @ sb.abs().t()
    # fp32 accumulation over K + 16 terms, u rounded once, then one rounding to the output
    ulp16 = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = ((K + 32) * 2.0 ** -24 * mag + ulp16 * (u.abs() @ sb.abs().t()) + ulp16 * ref.abs()
             + 1e-6)
    assert torch.all((y.double() - ref).abs() <= bound)


@pytest.mark.parametrize("M", [3, 40, 300])
def test_strided_bias(M):
    """A bias that is a column of a wider tensor, already in the compute dtype."""
    print(f"strided bias M={M}", flush=True)
    g, packed, st, a, b = _layer(256, 128, M)
    x = torch.randn(M, 128, device="cuda", generator=g).bfloat16()
    bias = torch.randn(256, 3, device="cuda", generator=g).bfloat16()[:, 1]
    if M <= nf4.LORA_FEW_MAX_ROWS:
        _check(lora.LoraNF4Few.apply(x, a, b, packed, st, bias, 2.0), x, packed, st, a, b, bias)
    y = lora.LoraNF4Linear.apply(x, a, b, packed, st, bias, 2.0, 0.0, 0)
    _check(y, x, packed, st, a, b, bias)


def _step(x, packed, st, a, b, dy):
    a, b, x = (t.detach().clone().requires_grad_() for t in (a, b, x))
    y = lora.LoraNF4Linear.apply(x, a, b, packed, st, None, 2.0, 0.0, 0)
    return [y.detach(), *torch.autograd.grad(y, [x, a, b], dy)]


@pytest.mark.parametrize("M,storage", [(300, torch.int8), (40, torch.int8), (40, torch.bfloat16)])
def test_codes_stored_as_another_type(M, storage):
    """The packed bytes held by a tensor of another type (bitsandbytes' quant_storage): the same
    bits as from uint8, forward and backward. A type wider than a byte is taken up to 256 rows;
    above, the forward refuses a buffer with fewer than half as many elements as weights."""
    print(f"codes stored as {storage} M={M}", flush=True)
    g, packed, st, a, b = _layer(256, 128, M)
    x = torch.randn(M, 128, device="cuda", generator=g).bfloat16()
    dy = torch.randn(M, 256, device="cuda", generator=g).bfloat16()
    want = _step(x, packed, st, a, b, dy)
    got = _step(x, packed.view(-1).view(storage), st, a, b, dy)
    assert all(torch.equal(p, q) for p, q in zip(got, want))


def test_wide_codes_refused_by_the_dense_forward():
    g, packed, st, a, b = _layer(256, 128, 1)
    x = torch.randn(300, 128, device="cuda", generator=g).bfloat16()
    with pytest.raises(ValueError, match="packed buffer is smaller"):
        lora.LoraNF4Linear.apply(x, a, b, packed.view(-1).view(torch.bfloat16), st, None, 2.0,
                                 0.0, 0)


def _offset_codes(packed, nbytes):
    buf = torch.empty(packed.numel() + nbytes, dtype=torch.uint8, device="cuda")
    buf[nbytes:] = packed.reshape(-1)
    return buf[nbytes:]


@pytest.mark.parametrize("kind", ["alike", "nested and plain", "codes off 4 bytes",
                                  "codes off 16 bytes"])
def test_group_and_single_dequantisation_give_the_same_product(kind):
    """The native group calls dequantise up to four weights that fit the group kernels in one
    launch, and others one by one: with the adapters zero, the products of the dequantised weights
    bit for bit."""
    print(f"native dequantisation: {kind}", flush=True)
    M, K, N = 300, 256, 192
    G = 2
    g = torch.Generator(device="cuda").manual_seed(7)
    items = []
    for i in range(G):
        w = torch.randn(N, K, device="cuda", generator=g) * 0.02
        packed, st = quant.quantize_nf4(w, 64, compress_statistics=kind != "nested and plain" or i)
        if kind.startswith("codes off"):
            packed = _offset_codes(packed, 2 if "4" in kind else 4)
        items.append((packed, st))
    x = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    dy = torch.randn(M, G * N, device="cuda", generator=g).bfloat16()
    z = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    host, table, stream = _host.load(), nf4._nf4_table(x.device), _lib.stream_of(x)
    weights = [nf4.weight_args(*it) for it in items]
    w = torch.cat([nf4.dequantize_nf4(p, st, torch.bfloat16) for p, st in items])
    y, _, _ = host.group_forward(x, z(16 * G, K), z(G * N, 64), weights, None, 0.0, [], table,
                                 stream)
    want = gemm.gemm_nt_cat(x, w, z(M, 64), z(G * N, 64), z(M, G * N))
    assert torch.equal(y, want)
    if kind.startswith("codes off"):
        return  # the transposed kernel takes codes aligned to 16 bytes only
    ut = z(16 * G, 304)[:, :M]
    dx, grads = host.group_backward(dy, x, z(K, 64), z(16 * G, G * N), ut, weights, [1.0] * G, True,
                                    [False] * (2 * G), None, None, [], 0.0, None, [], table, stream)
    want = gemm.gemm_nt_cat(dy, w.t().contiguous(), z(M, 64), z(K, 64), z(M, K))
    assert torch.equal(dx, want) and grads == [None] * (2 * G)


def test_codes_off_16_bytes_are_refused_by_the_transposed_dequantisation():
    g, packed, st, a, b = _layer(256, 128, 2)
    x = torch.randn(300, 128, device="cuda", generator=g).bfloat16()
    t = torch.zeros(16, 256, device="cuda", dtype=torch.bfloat16)
    at = torch.zeros(128, 64, device="cuda", dtype=torch.bfloat16)
    dy = torch.randn(300, 256, device="cuda", generator=g).bfloat16()
    with pytest.raises(RuntimeError, match="alignment"):
        _host.load().group_backward(dy, x, at, t, torch.zeros(16, 304, device="cuda",
                                                              dtype=torch.bfloat16)[:, :300],
                                    [nf4.weight_args(_offset_codes(packed, 4), st)], [1.0], True,
                                    [False, False], None, None, [], 0.0, None, [],
                                    nf4._nf4_table(x.device), _lib.stream_of(x))
