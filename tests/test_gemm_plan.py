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


@pytest.mark.parametrize("K,N,M,fmt,gated,want", [
    # 8 bits: as many 96-row tiles as fill the chip by halves, 183 / 76 / 246 us against 215 / 89 / 267 of 256 x 128 tiles
    (12288, 3072, 1500, (8, 64, 0), 0, 96),
    (5120, 3072, 1500, (8, 64, 0), 0, 96),
    (17408, 3072, 1500, (8, 64, 0), 0, 96),
    (6144, 4608, 798, (8, 64, 0), 0, 96),            # 86 / 110
    # less than a round of large tiles over a short K: 21.2 against 27.4 of 256 x 128 large tiles
    (512, 9664, 1024, (8, 64, 0), 0, -192),
    (1024, 16832, 768, (4, 64, 0), 0, -256),         # 35 / 45
    # two thirds of a round of 256-wide tiles against three and a half of 128-row ones: 156 / 191, 192-wide 86 / 105
    (7168, 2560, 3933, (4, 32, 0), 0, -256),
    (4096, 2240, 3667, (4, 64, 1), 0, -192),
    (4096, 6208, 1350, (4, 64, 1), 0, -192),         # 86 / 103
    # one round and a half of large gated tiles: 207 against 268
    (2560, 28160, 1212, (8, 64, 0), 1, 128),
    (512, 3584, 1637, (8, 64, 0), 1, 128),           # 18 / 24
    # 2.8 rounds of 192-wide tiles, by whose order the busiest XCD has 3.5: 305 against 356
    (4608, 19456, 1663, (4, 64, 0), 0, 128),
])
def test_plan_where_other_kernels_than_the_obvious_one_are_faster(K, N, M, fmt, gated, want):
    assert vpipe_amd.load().vpq_qmm_plan(K, N, M, *fmt, gated, 1) == want


def test_plan_refuses_what_the_entrances_refuse():
    L = vpipe_amd.load()
    for args in [(96, 64, 64, 4, 64, 0, 0, 1), (64, 0, 64, 4, 64, 0, 0, 1), (64, 63, 64, 4, 64, 0, 1, 1), (64, 64, 64, 8, 32, 0, 0, 1),
                 (64, 64, 64, 4, 32, 1, 0, 1), (64, 64, 64, 8, 64, 0, 0, 2), (64, 64, 64, 4, 64, 0, 0, 17)]:
        assert L.vpq_qmm_plan(*args) == -2


# Expert-sorted GEMMs: tokens, top_k, experts, blocks of the map (0: as the sort leaves it), rows of x per workgroup.  Times as
# gate|up + down of 2048 -> 768, 160 rows against 64.
@pytest.mark.parametrize("tokens,top_k,E,used,want", [
    (4, 8, 128, 0, 64), (64, 8, 128, 0, 64), (512, 8, 128, 0, 64),     # 93 + 44 / 86 + 38
    (768, 8, 128, 0, 160), (1024, 8, 128, 0, 160),                     # 112 + 55 / 138 + 66
    (4096, 1, 128, 0, 64), (512, 16, 128, 0, 160),
    (64, 8, 128, 126, 64), (512, 8, 128, 128, 64),                     # the map cut down to the blocks in use
    (1024, 8, 128, 128, 160), (4096, 8, 128, 256, 160),
])
def test_expert_sorted_plan(tokens, top_k, E, used, want):
    L = vpipe_amd.load()
    pairs, B = tokens * top_k, L.vpq_qmm_grouped_block_rows()
    npad = B * (used or -(-pairs // B) + min(E, pairs))
    assert L.vpq_qmm_grouped_plan(1536, npad, E, tokens, 1) == want
    assert L.vpq_qmm_grouped_plan(2048, npad, E, pairs, 0) == want
    assert L.vpq_qmm_grouped_plan(512, npad, 64, tokens, 1) == 160     # within one round


def test_expert_sorted_plan_refuses_what_the_entrances_refuse():
    for args in [(0, 128, 8, 4, 0), (64, 100, 8, 4, 0), (64, 128, 0, 4, 0), (64, 128, 8, 0, 0), (63, 128, 8, 4, 1)]:
        assert vpipe_amd.load().vpq_qmm_grouped_plan(*args) == -2
