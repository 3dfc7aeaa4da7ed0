"""Which kernel and tile a matrix product runs on, from the host-side launch plans (no GPU)."""
import pytest

import cgadimpl_amd as agk
from test_gemm import PLAN_CASES, SHAPE_IDS


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


MOST_LANES = 2 ** 32 - 1  # along a grid dimension


@pytest.mark.parametrize("M,N,K", [(2 ** 30 + 8, 8, 8), (2 ** 30 + 8, 8, 64), (2 ** 30 + 64, 64, 56),
                                   (300_000, 300_000, 8), (300_000, 300_000, 64),
                                   (8, 2 ** 31 - 512, 64), (2 ** 31 - 512, 8, 8)])
def test_bf16_grids_fit_a_launch(M, N, K):
    p = agk.gemm_bf16_launch_plan(M, N, K, cus=256)
    assert p["grid_x"] * 256 <= MOST_LANES, p
    assert p["grid_x"] >= -(-M // p["tile_m"]) * -(-N // p["tile_n"])
    assert K >= 64 or p["shape"] != 0  # the 256 x 256 kernel starts from a whole k-tile


@pytest.mark.parametrize("M,N,ta", [(8, 2 ** 29 + 32, False), (1, 2 ** 31 - 1, False),
                                    (2, 2 ** 30 + 7, True), (64, 2 ** 30 + 64, False),
                                    (40, 2 ** 30 + 64, True)])
def test_f32_grids_fit_a_launch(M, N, ta):
    p = agk.gemm_f32_launch_plan(M, N, trans_a=ta, cus=256)
    assert p["grid_x"] * 256 <= MOST_LANES and p["grid_y"] <= 65535, p
    assert p["grid_x"] * p["grid_y"] >= -(-M // p["tile_m"]) * -(-N // p["tile_n"])
    assert not (ta and M < 4) or p["shape"] == 0


def test_bf16_cases_reach_every_shape():
    """The GPU tests' sizes take the shapes they stand for, on 256 compute units, and leave none
    out."""
    assert sorted(SHAPE_IDS) == list(range(9))
    for shape, halves, M, N, K in PLAN_CASES:
        p = agk.gemm_bf16_launch_plan(M, N, K, cus=256)
        assert (p["shape"], p["halves"] > 0) == (shape, halves), (M, N, K, p)
        assert M % p["tile_m"] or N % p["tile_n"], (M, N, K, p)  # ragged last tiles
