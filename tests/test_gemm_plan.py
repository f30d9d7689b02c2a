"""How the GEMM splits its work, over random sizes (the planner runs on the
host and needs no GPU)."""
import math
import random

import pytest

from cppnet_amd import ops


def sizes(n, seed):
    rng = random.Random(seed)
    for _ in range(n):
        M, N, K = (int(round(math.exp(rng.uniform(math.log(33), math.log(12000))))) for _ in range(3))
        yield M, N, K, rng.choice([1, 1, 1, 1, rng.randint(2, 300)]), rng.random() < 0.5, rng.random() < 0.5


def plan(M, N, K, batch=1, ta=False, tb=False, reads_c=False):
    return ops.gemm_plan(ta, tb, M, N, K, K if ta else M, N if tb else K, batch, reads_c)


def check_halves(tile, splits, reads_c):
    # a 256 x 256 tile forms two half sums of opposite sign: one after the
    # other in C, or in an even number of splits
    if tile == (256, 256):
        assert splits % 2 == 0 or (splits == 1 and not reads_c), splits


@pytest.mark.parametrize("M,N,K", [(162, 6975, 9148), (5559, 136, 9583), (143, 3229, 6674), (4096, 4096, 4096), (300, 500, 400)])
@pytest.mark.parametrize("reads_c", [False, True])
def test_large_tiles_run_as_two_half_sums(M, N, K, reads_c):
    m, n, splits, _, _ = plan(M, N, K, reads_c=reads_c)
    check_halves((m, n), splits, reads_c)


def test_plans_cover_the_product():
    for M, N, K, batch, ta, tb in sizes(3000, 5):
        for reads_c in (False, True):
            m, n, splits, kps, scratch = plan(M, N, K, batch, ta, tb, reads_c)
            what = (M, N, K, batch, ta, tb, reads_c, m, n, splits, kps)
            if m == 0:
                continue
            check_halves((m, n), splits, reads_c)
            # every split has work, and all of them together cover K
            assert kps % 32 == 0 and (splits - 1) * kps < K <= splits * kps, what
            assert scratch == (splits * M * N * batch * 4 if splits > 1 else 0), what
            # the partial sums stay within the no-allocation entry points' array
            assert scratch <= 32 << 20, what


# (M, N, K, batch, trans_a, trans_b): measured, microseconds in the 64 x 64
# fp32 tile / the best split-operand tile
@pytest.mark.parametrize("M,N,K,batch,ta,tb", [
    (128, 128, 128, 1, False, True),        # 5.8 / 8.6
    (512, 512, 64, 1, False, False),        # 4.8 / 7.8
    (1001, 515, 785, 1, False, False),      # 21 / 26
    (100, 100, 10000, 1, False, True),      # 18 / 33
    (256, 256, 64, 256, False, False),      # 31 / 46
    (200, 64, 200, 16, False, True),        # 9.6 / 15.5
    (8102, 613, 4079, 1, False, True),      # 427 / 624
    (1024, 1024, 256, 1, False, False),     # 9 / 15.6
])
def test_short_small_and_ragged_products_take_the_fp32_tile(M, N, K, batch, ta, tb):
    assert plan(M, N, K, batch, ta, tb)[:2] == (64, 64)


@pytest.mark.parametrize("M,N,K,tile", [(4096, 4096, 4096, 256),   # 630 us; 64 x 64: 1130
                                        (8192, 512, 2048, 128),    # 96; 142
                                        (2048, 2048, 512, 128),    # 32; 40
                                        (512, 512, 8192, 128)])    # 38; 45
def test_large_whole_products_take_the_split_tiles(M, N, K, tile):
    assert plan(M, N, K)[:2] == (tile, tile)


def test_plans_do_not_depend_on_what_was_planned_before():
    rng = random.Random(9)
    jobs = [s for s in sizes(400, 11)]
    first = [plan(M, N, K, b, ta, tb) for M, N, K, b, ta, tb in jobs]
    order = list(range(len(jobs)))
    rng.shuffle(order)
    for i in order:
        M, N, K, b, ta, tb = jobs[i]
        assert plan(M, N, K, b, ta, tb) == first[i]
        plan(M, N, K, b, ta, tb, reads_c=True)


# What tests/test_gpu_gemm_split.py is to reach: (M, N, K), tile, splits
@pytest.mark.parametrize("size,tile,splits", [((100, 515, 2000), 64, 21), ((1001, 515, 785), 64, 5), ((8192, 512, 512), 128, 1),
                                              ((2050, 1561, 425), 128, 1), ((196, 2287, 3134), 128, 7),
                                              ((2048, 2048, 512), 128, 1), ((4096, 4096, 2048), 256, 1),
                                              ((4090, 4087, 2051), 256, 1), ((6731, 586, 2027), 256, 2),
                                              ((4057, 257, 5017), 256, 8), ((1361, 385, 8687), 256, 16)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_the_gpu_tests_reach_every_tile(size, tile, splits, ta, tb):
    assert plan(*size, 1, ta, tb)[:3] == (tile, tile, splits)
