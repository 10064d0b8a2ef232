"""Which tile and split of K the NT GEMM takes (qlora_gemm_nt_plan), on the host."""

import pytest
import torch

from hackathon_amd import _lib, gemm


@pytest.mark.parametrize("M,N,K", [(4096, 1536, 8960), (757, 8192, 8960), (2798, 2048, 8960),
                                   (700, 8192, 8192)])
def test_long_loops_on_part_of_the_chip_keep_the_large_tile(M, N, K):
    """Two splits of the 256-row tile on three quarters of the CUs beat four of 128 x 256."""
    assert gemm.nt_plan(M, N, K) == (256, 256, 2)


@pytest.mark.parametrize("M,N,K,tile", [(4096, 18944, 3584, (256, 256)),
                                        (4096, 3584, 3584, (256, 224)),
                                        (1001, 3584, 3584, (128, 128)),
                                        (512, 3584, 3584, (64, 128)),
                                        (333, 18944, 3584, (128, 256)),
                                        (3205, 1152, 18944, (128, 128))])
def test_unsplit_tiles(M, N, K, tile):
    assert gemm.nt_plan(M, N, K) == (*tile, 1)


def test_sizes_the_kernel_does_not_take_are_refused():
    for sizes in ((0, 64, 64), (64, 0, 64), (64, 64, 0), (64, 64, 96)):
        with pytest.raises(RuntimeError, match="inconsistent sizes"):
            gemm.nt_plan(*sizes)


@pytest.mark.parametrize("M,N,K", [(4096, 512, 3584), (1001, 3584, 3584), (512, 512, 4096)])
def test_plain_products_ask_for_their_own_partials_only(monkeypatch, M, N, K):
    """The accumulating plan's splits (7 of 4096 x 512: 59 MB) are not allocated where beta is 0."""
    plan = gemm.nt_plan(M, N, K)[2]
    asked = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: asked.append(a[-2]))
    monkeypatch.setattr(_lib, "require_device", lambda *t: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    a, b = torch.empty(M, K, dtype=torch.bfloat16), torch.empty(N, K, dtype=torch.bfloat16)
    out = torch.empty(M, N, dtype=torch.bfloat16)
    gemm.gemm(a, b, out=out)
    gemm.gemm(a, b, out=out, beta=1.0)
    assert asked[0] == (plan * M * N * 4 if plan > 1 else 0)
    assert asked[1] == _lib.load().qlora_gemm_workspace_size(0, 0, M, N, K) > 0


def test_the_tile_tests_run_the_tiles_they_name():
    """The planner's choice for the cases of test_gpu_gemm_mid: refitting it must not leave a tile
    untested."""
    from test_gpu_gemm_mid import CASES

    assert [gemm.nt_plan(*c[:3]) for c in CASES] == [
        (128, 128, 1), (128, 128, 1), (64, 128, 1), (64, 128, 1), (64, 128, 5), (64, 128, 1),
        (128, 256, 1), (128, 256, 6), (64, 128, 1), (64, 128, 1), (64, 128, 7)]


def test_the_large_tile_tests_run_the_large_tile():
    from test_gpu_gemm_large_tile import CASES

    assert all(gemm.nt_plan(*c[:3]) == c[6] for c in CASES)
    assert {c[6][1] for c in CASES} == {224, 256} and {c[6][2] for c in CASES} == {1, 3}
