"""The few-row paths of the 4-bit LoRA layer (nf4.lora_few, lora.LoraNF4Few, LoraNF4Linear up to 256
rows) refuse operands their kernels would read out of range, before any launch; the launches are
recorded instead of made."""

import pytest
import torch

from hackathon_amd import _lib, lora, nf4, quant

K, N = 128, 64


@pytest.fixture
def launches(monkeypatch):
    calls = []
    monkeypatch.setattr(_lib, "call", lambda *a: calls.append(a))
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    return calls


def _operands():
    packed, qs = quant.quantize_nf4(torch.randn(N, K), 64)
    x = torch.randn(2, K).bfloat16()
    return x, packed, qs, torch.randn(16, K), torch.randn(N, 16)


def test_operands_that_fit_are_launched(launches, monkeypatch):
    from torch._subclasses.fake_tensor import FakeTensorMode

    _, _, qs, _, _ = _operands()
    monkeypatch.setattr(nf4, "_nf4_table", lambda device: torch.zeros(16))
    with FakeTensorMode():  # a GPU's device, no storage
        t = lambda *shape, dtype: torch.empty(*shape, dtype=dtype, device="cuda:0")  # noqa: E731
        monkeypatch.setattr(nf4, "_scale_args", lambda qs: (t(128, dtype=torch.uint8), 0, None,
                                                            None, 0.0, 1))
        monkeypatch.setattr(_lib, "workspace", lambda *a, device: (None, 0))
        monkeypatch.setattr(torch.Tensor, "data_ptr", lambda self: 0)
        for bias in (None, t(N, dtype=torch.bfloat16), t(N, dtype=torch.float32)):
            y = nf4.lora_few(t(2, K, dtype=torch.bfloat16), t(N * K // 2, dtype=torch.uint8), qs,
                             t(16, K, dtype=torch.float32), t(N, 16, dtype=torch.float32), 2.0,
                             bias)
            assert y.shape == (2, N)
    assert [c[0] for c in launches] == ["qlora_nf4_lora_few"] * 3


@pytest.mark.parametrize("what,error", [
    ("wide x", ValueError), ("narrow x", ValueError), ("short A", ValueError),
    ("short B", ValueError), ("rank 8", ValueError), ("fp32 x", TypeError),
    ("bf16 A", TypeError), ("bf16 B", TypeError), ("strided x", ValueError),
    ("strided A", ValueError), ("strided B", ValueError), ("few codes", ValueError)])
def test_operands_that_do_not_fit_raise_before_the_launch(launches, what, error):
    x, packed, qs, a, b = _operands()
    if what == "wide x":
        x = torch.randn(2, 2 * K).bfloat16()
    elif what == "narrow x":
        x = x[:, :64].contiguous()
    elif what == "short A":
        a = a[:, :64].contiguous()
    elif what == "short B":
        b = b[:32]
    elif what == "rank 8":
        a, b = a[:8], b[:, :8].contiguous()
    elif what == "fp32 x":
        x = x.float()
    elif what == "bf16 A":
        a = a.bfloat16()
    elif what == "bf16 B":
        b = b.bfloat16()
    elif what == "strided x":
        x = torch.randn(2, 2 * K).bfloat16()[:, ::2]
    elif what == "strided A":
        a = torch.randn(16, 2 * K)[:, ::2]
    elif what == "strided B":
        b = torch.randn(16, N).t()
    else:
        packed = packed[: packed.shape[0] // 2]
    with pytest.raises(error):
        nf4.lora_few(x, packed, qs, a, b, 2.0)
    assert not launches


def test_operands_off_the_gpu_raise():
    with pytest.raises(ValueError, match="on a GPU device"):
        x, packed, qs, a, b = _operands()
        nf4.lora_few(x, packed, qs, a, b, 2.0)


@pytest.mark.parametrize("width", [2 * K, 64])
def test_layer_of_another_width_raises_without_gradients(launches, width):
    base = quant.Linear4bit.from_weight(torch.randn(N, K).bfloat16(),
                                        compute_dtype=torch.bfloat16)
    layer = lora.LoraLinear4bit(base, compute_dtype=torch.bfloat16)
    x = torch.randn(2, width).bfloat16()
    a, b = layer.lora_A["default"].weight, layer.lora_B["default"].weight
    with torch.no_grad(), pytest.raises(ValueError, match=f"x has {width} columns"):
        assert lora._takes_few(x, a, b, base.weight, base.weight.quant_state)
        lora.LoraNF4Few.apply(x, a, b, base.weight, base.weight.quant_state, None, 2.0)
    assert not launches


@pytest.mark.parametrize("p", [0.0, 0.1])
def test_layer_of_another_width_raises_with_gradients(launches, monkeypatch, p):
    """The path with gradients forms the down-projection before its GEMM compares the widths: a
    wider x must not get as far as reading past A."""
    packed, qs = quant.quantize_nf4(torch.randn(N, K), 64)
    a, b = torch.randn(16, K).requires_grad_(), torch.randn(N, 16).requires_grad_()
    t = torch.zeros(16, K, dtype=torch.bfloat16)
    monkeypatch.setattr(lora.adapter_packs, "pack", lambda *_: (t, t, t, t))
    monkeypatch.setattr(_lib, "require_rows", lambda dtype, **_: None)
    x = torch.randn(2, 2 * K).bfloat16()
    with pytest.raises(ValueError, match=f"x has {2 * K} columns"):
        lora.LoraNF4Linear.apply(x, a, b, packed, qs, None, 2.0, p, 1)
    assert not launches


def test_strided_bias_reaches_the_few_row_launch_dense(launches, monkeypatch):
    x, packed, qs, a, b = _operands()
    bias = torch.randn(N, 2).bfloat16()[:, 0]
    seen = []

    class Host:
        @staticmethod
        def few_rows_operands(x, packed, a, b, bias, n, k):
            seen.append(bias)
            return 0, 0, 0, 0, 0

    monkeypatch.setattr(nf4._host, "load", lambda: Host)
    lora.LoraNF4Few.apply(x, a, b, packed, qs, bias, 2.0)
    assert seen[0].is_contiguous() and torch.equal(seen[0], bias)


def test_bias_of_another_length_raises():
    from torch._subclasses.fake_tensor import FakeTensorMode

    host = lora._host.load()
    with FakeTensorMode():
        t = lambda *shape, dtype=torch.float32: torch.empty(*shape, dtype=dtype,  # noqa: E731
                                                            device="cuda:0")
        with pytest.raises(ValueError, match="bias must be 64"):
            host.few_rows_operands(t(2, K, dtype=torch.bfloat16), t(N * K // 2, dtype=torch.uint8),
                                   t(16, K), t(N, 16), t(32, dtype=torch.bfloat16), N, K)


def test_strided_bias_reaches_the_native_calls_dense(launches, monkeypatch):
    packed, qs = quant.quantize_nf4(torch.randn(N, K), 64)
    a, b = torch.randn(16, K), torch.randn(N, 16)
    t = torch.zeros(16, K, dtype=torch.bfloat16)
    monkeypatch.setattr(lora.adapter_packs, "pack", lambda *_: (t, t, t, t))
    seen = []

    class Host:
        @staticmethod
        def group_forward(x, a16, bs, weights, bias, *rest):
            seen.append(bias)
            return torch.zeros(x.shape[0], N), t, []

    monkeypatch.setattr(lora._host, "load", lambda: Host)
    bias = torch.randn(N, 2).bfloat16()[:, 0]
    lora.LoraNF4Linear.apply(torch.randn(300, K).bfloat16(), a, b, packed, qs, bias, 2.0,
                             0.0, 0)
    assert seen[0].is_contiguous() and torch.equal(seen[0], bias)
