"""Which GEMM kernel a shape takes (vpq_qmm_plan), where the wrong one costs much.  Times of the kernels in
microseconds, on an idle MI355X with 256 CUs, beside each; no GPU needed: without one the plan is for 256 CUs."""
import pytest

import vpipe_amd


@pytest.mark.parametrize("K,N,M,fmt,gated,want", [
    # 432 large tiles are 1.7 rounds that take no longer than 1.5: 469 us against 604 of 128 x 128 tiles
    (12288, 5120, 4096, (4, 64, 0), 0, -192),
    (5120, 5120, 4096, (4, 64, 0), 0, -192),         # 203 / 254
    (17408, 5120, 3400, (8, 64, 0), 0, -192),        # 665 / 821
    (5120, 19328, 3400, (4, 32, 0), 0, -256),        # 653 / 796
    (5120, 9664, 2048, (4, 64, 1), 0, -192),         # 210 / 239
    # a short K: three rounds of 256 x 128 tiles with a store each, 49, against 36 for the smaller tiles
    (512, 24576, 800, (4, 32, 0), 0, 96),
    # every 128 x 128 tile reads x, 1.1 GB from the shared cache: 235 against 202 on one round of large tiles
    (12288, 2048, 4096, (4, 64, 0), 0, -128),
    # the gated store of a large tile is long, and a K of 512 short: 105 against 70 of the smaller tiles
    (512, 19328, 2048, (4, 64, 0), 1, 64),
    # few rows: 64 rows a workgroup fill the chip
    (4096, 4096, 333, (4, 64, 0), 0, 64),
])
def test_plan(K, N, M, fmt, gated, want):
    assert vpipe_amd.load().vpq_qmm_plan(K, N, M, *fmt, gated, 1) == want


def test_plan_refuses_what_the_entrances_refuse():
    L = vpipe_amd.load()
    for args in [(96, 64, 64, 4, 64, 0, 0, 1), (64, 0, 64, 4, 64, 0, 0, 1), (64, 63, 64, 4, 64, 0, 1, 1), (64, 64, 64, 8, 32, 0, 0, 1),
                 (64, 64, 64, 4, 32, 1, 0, 1), (64, 64, 64, 8, 64, 0, 0, 2), (64, 64, 64, 4, 64, 0, 0, 17)]:
        assert L.vpq_qmm_plan(*args) == -2
