"""Cross-entropy rows whose exponentials leave fp32's normal range (the sweeps then take the
scaled exponential), with ties, entries far below the rest and a NaN, against the CPU oracle and
torch. Bounds as in test_gpu_ce."""

import pytest
import torch

from hackathon_amd import _lib
from oracle import ops

pytestmark = pytest.mark.gpu


def _rows(z, t, ignore_mode=1, scale=3.0):
    R, V = z.shape
    out = [torch.empty(R, device="cuda"), torch.empty(R, device="cuda"),
           torch.empty(R, dtype=torch.int32, device="cuda"),
           torch.empty(R, dtype=torch.int64, device="cuda")]
    _lib.call("qlora_ce_rows", z.data_ptr(), _lib.tag(z.dtype), V, R, V, t.data_ptr(),
              *[o.data_ptr() for o in out], ignore_mode, 1, scale, _lib.stream_of(z))
    return [o.cpu() for o in out]


@pytest.mark.parametrize("V", [8, 4096, 4104, 40007])
@pytest.mark.parametrize("dtype,spread", [(torch.bfloat16, 60.0), (torch.float32, 60.0),
                                          (torch.float16, 40.0), (torch.float32, 0.0)])
def test_wide_rows_and_ties(V, dtype, spread):
    print(f"ce rows V={V} {dtype} spread={spread}", flush=True)
    g = torch.Generator().manual_seed(V)
    z = (torch.randn(17, V, generator=g) * spread).to(dtype)  # spread 0: every entry a tie
    z[3, V // 2:] = -1e4
    t = torch.randint(0, V // 2, (17,), generator=g)
    t[5] = -100
    zf = z.double()
    lse = torch.logsumexp(zf, 1)
    p = torch.softmax(zf, 1)
    zg, tg = z.cuda(), t.cuda()
    loss, ent, cor, pred = _rows(zg, tg)
    lab = t >= 0
    want = torch.where(lab, lse - zf.gather(1, t.clamp(min=0)[:, None])[:, 0], torch.zeros(17).double())
    torch.testing.assert_close(loss.double(), want, rtol=1e-4, atol=1e-4)
    first = (zf == zf.max(1, keepdim=True).values).int().argmax(1)
    assert torch.equal(pred, first)
    assert torch.equal(cor, ((pred == t) & lab).int())
    p[torch.arange(17), t.clamp(min=0)] -= lab.double()
    dz = p * 3.0 * lab.double()[:, None]
    # fp32: the log-sum-exp of about 250 is held to 2^-17, which scales every probability by as much
    tol = 1e-2 if dtype == torch.bfloat16 else (2e-3 if dtype == torch.float16 else 4e-5)
    torch.testing.assert_close(zg.cpu().double(), dz.to(dtype).double(), rtol=tol, atol=tol)
    # subnormal probabilities are kept, not flushed: down to where fp32 ends
    if dtype == torch.float32 and spread:
        got = zg.cpu().double()
        small = (dz > 2.0**-140) & (dz < 2.0**-127)
        # an argument near -100 carries 2^-18 of absolute error; a subnormal result 2^-149
        assert torch.all((got - dz).abs()[small] <= dz[small] * 2.0**-14 + 2.0**-147)


def test_a_nan_reaches_the_loss_and_its_row_only():
    z = torch.randn(4, 4096, generator=torch.Generator().manual_seed(1))
    t = torch.tensor([1, 2, 3, 4])
    z[2, 800] = float("nan")
    zg = z.cuda()
    loss, _, _, pred = _rows(zg, t.cuda())
    assert torch.isnan(loss[2]) and not torch.isnan(loss[[0, 1, 3]]).any()
    assert torch.equal(pred[[0, 1, 3]], z[[0, 1, 3]].argmax(1))
    ref = ops.ce_rows(z[:2], t[:2], 1, grad_scale=3.0)
    torch.testing.assert_close(loss[:2].double(), ref[0], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("V", [1, 7, 511, 513, 2047, 2049, 2561, 4097])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_element_rows_around_whole_pieces(V, dtype):
    """Rows that go element by element, on both sides of one element and of one piece of four for
    each of the 512 threads."""
    print(f"ce element rows V={V} {dtype}", flush=True)
    g = torch.Generator().manual_seed(V)
    z = torch.randn(5, V, generator=g).to(dtype)
    t = torch.randint(0, V, (5,), generator=g)
    t[2] = -100
    lse = torch.logsumexp(z.double(), 1)
    lab = t >= 0
    at = z.double().gather(1, t.clamp(min=0)[:, None])[:, 0]
    zg = z.cuda()
    loss, ent, cor, pred = _rows(zg, t.cuda())
    torch.testing.assert_close(loss.double(), torch.where(lab, lse - at, 0.0), rtol=1e-4, atol=1e-4)
    p = torch.softmax(z.double(), 1)
    logp = torch.log_softmax(z.double(), 1)
    torch.testing.assert_close(ent.double(), -(p * logp).sum(1), rtol=1e-4, atol=1e-4)
    assert torch.equal(pred, (z.double() == z.double().max(1, keepdim=True).values).int().argmax(1))
    p[torch.arange(5), t.clamp(min=0)] -= lab.double()
    dz = p * 3.0 * lab.double()[:, None]
    tol = 1e-2 if dtype == torch.bfloat16 else 4e-5
    torch.testing.assert_close(zg.cpu().double(), dz.to(dtype).double(), rtol=tol, atol=tol)
