"""Which tile and split of K the NT GEMM takes (qlora_gemm_nt_plan), on the host."""

import pytest

from hackathon_amd import gemm


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
