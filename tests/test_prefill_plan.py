"""How the prefill GEMMs are cut (host code): tiles, K pieces, the workspace the pieces need."""
import itertools
import random

import pytest

from kata_amd import ops

WS_FLOATS = 2 * 256 * 128                       # workspace floats per CU


def _cdiv(a, b):
    return -(-a // b)


@pytest.mark.parametrize("fmt", ["f16", "q8", "i8"])
def test_plans_hold(fmt):
    """Every tile is covered once, pieces are at least a block long and fit the workspace, and
    without the workspace there are none."""
    rng = random.Random(1)
    shapes = list(itertools.product((1, 31, 33, 64, 129, 257, 1000, 7300), (128, 384, 1920, 5120, 17408),
                                    (1, 255, 257, 1024, 5120, 17408), (256, 304, 64)))
    shapes += [(rng.randint(1, 9000), 128 * rng.randint(1, 200), rng.randint(1, 40000), rng.choice((256, 80))) for _ in range(3000)]
    for M, K, N, n_cu in shapes:
        Ns = [N, rng.randint(1, 20000)] if fmt == "f16" and rng.random() < 0.3 else [N]
        p = ops.prefill_plan(fmt, M, K, Ns, n_cu)
        tiles = _cdiv(M, p.tile_rows) * sum(_cdiv(n, p.tile_cols) for n in Ns)
        assert p.whole + p.split == tiles, (M, K, Ns, p)
        assert (1 < p.pieces <= min(16, K // 128)) if p.split else p.pieces == 1, (M, K, Ns, p)
        assert p.split * p.pieces * p.tile_rows * p.tile_cols <= n_cu * WS_FLOATS, (M, K, Ns, p)
        assert ops.prefill_plan(fmt, M, K, Ns, n_cu, workspace=False).split == 0


@pytest.mark.parametrize("M,K,N,shorter", [(25, 1920, 1500, True), (41, 1024, 1024, True), (41, 1920, 5000, True),
                                           (25, 5120, 1024, True), (100, 4096, 4096, False), (100, 5120, 12288, False)])
def test_f16_pieces_follow_time(M, K, N, shorter):
    """Few tiles of short rows are split into pieces below 8 blocks (measured 1.3 to 1.9 times faster
    than without); where that gains little or nothing, 8 blocks are the least."""
    p = ops.prefill_plan("f16", M, K, N)
    assert p.split and (K // 128 / p.pieces < 8) == shorter, p
