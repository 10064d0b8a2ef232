"""The native host code of the fused layers (csrc/host/host.cpp): bound to entry points that the
C-ABI binding knows, and refusing operands the kernels do not take before any launch."""

import pytest
import torch

from hackathon_amd import _host, _lib, nf4, quant


def test_every_entry_is_a_known_symbol():
    names = _host.load().entry_names()
    assert len(set(names)) == len(names)
    assert set(names) <= set(_lib.exported_symbols())


def _args(dtype=torch.bfloat16, k=128, n=64):
    w = torch.randn(n, k)
    packed, qs = quant.quantize_nf4(w, 64)
    weight = nf4.weight_args(packed, qs)
    x = torch.zeros(300, k, dtype=dtype)
    return x, torch.zeros(16, k, dtype=dtype), torch.zeros(n, 64, dtype=dtype), [weight]


def test_cpu_and_mistyped_operands_raise():
    host = _host.load()
    x, a16, bs, weights = _args()
    table = torch.zeros(16)
    with pytest.raises(ValueError, match="x must be on a GPU device"):
        host.group_forward(x, a16, bs, weights, None, 0.0, [], table, 0)
    with pytest.raises(ValueError, match="g must be on a GPU device"):
        host.group_backward(x, x, a16, a16, a16, weights, [1.0], True, [True, True], None, None,
                            [], 0.0, None, [], table, 0)
    with pytest.raises(TypeError):
        host.group_forward(x, a16, bs, weights, None, 0.0, [], None, 0)


def test_weight_args_hold_a_contiguous_copy_of_strided_codes():
    w = torch.randn(64, 128)
    packed, qs = quant.quantize_nf4(w, 64)
    wide = torch.zeros(packed.shape[0], 2, dtype=torch.uint8)
    wide[:, :1] = packed
    args = nf4.weight_args(wide[:, :1], qs)
    assert args[0].is_contiguous() and torch.equal(args[0], packed)
    assert args[-2:] == (64, 128)
