"""Which kernel and tile a matrix product runs on, from the host-side launch plans (no GPU)."""
import pytest

import cgadimpl_amd as agk


@pytest.mark.parametrize("M,N,shape", [(1024, 1024, {256: 1, 32: 2}), (2048, 2048, {256: 2, 32: 2}),
                                       (512, 512, {256: 0, 128: 0, 32: 1})], ids=str)
def test_f32_tile_follows_the_compute_units(M, N, shape):
    """Fewer compute units (a partitioned device): larger tiles, as the tiles per unit grow."""
    for cus, want in shape.items():
        assert agk.gemm_f32_launch_plan(M, N, cus=cus)["shape"] == want, cus


def test_f32_tile_of_few_rows():
    """An operand whose rows are contiguous needs four of them for the staged tiles."""
    for M, N, ta, tb in ((3, 1 << 20, True, False), (1 << 20, 3, False, False)):
        assert agk.gemm_f32_launch_plan(M, N, trans_a=ta, trans_b=tb, cus=256)["shape"] == 0
