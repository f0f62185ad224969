"""How the prefill GEMMs are cut (host code): tiles, K pieces, and the workspace the pieces need."""
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
