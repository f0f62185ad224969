"""The int8 prefill GEMM over the sizes where its kernels, tile shapes and schedules change: rows at
the edges of the 32, 64 and 128 row tiles and around where the 256-row kernel takes over, columns
around the 256 column tiles, odd and even numbers of 128-groups, K splits, a scale row stride
wider than M.  Where a test means a tile height or a split it asks the planner.

Reference: exact int32 group sums (float64 products of integers) folded in float64.  Bar: 1e-6
relative L2: one fp32 rounding per group and output, at most 136 of them."""
import numpy as np
import pytest
import torch

from kata_amd import ops
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 31, 33, 64, 65, 128, 129, 190, 257])
@pytest.mark.parametrize("K,N", [(128, 257), (384, 1000), (2176, 255), (5120, 2048)])
def test_tile_edges(dev, M, K, N):
    W = torch.from_numpy(orc.synth_ptq1(N, K, M + K + N)[0]).to(dev)
    A = torch.from_numpy(orc.synth_x(M, K, M + 2)).to(dev)
    Q, SX = ops.quant_rows(A, ldS=M + 5)
    T8, SW = ops.expand_i8(W, K, N)
    x = (Q.double().view(M, -1, 128) * SX[:, :M].double().t()[:, :, None]).view(M, K)
    w = (T8.double().view(N, -1, 128) * SW.double()[:, :, None]).view(N, K)
    ref = x @ w.t()
    C = ops.gemm_ptq1_i8(Q, SX, W, K, N)
    err = float((C.double() - ref).norm() / ref.norm())
    assert err < 1e-6, err
    assert torch.equal(ops.gemm_ptq1_i8(Q, SX, W, K, N, out_dtype=torch.float16), C.half())


def _plan_is(dev, M, K, N, rows, kind):
    p = ops.prefill_plan("i8", M, K, N, torch.cuda.get_device_properties(dev).multi_processor_count)
    assert p.tile_rows == rows and (p.whole > 0, p.split > 0) == {"whole": (True, False), "split": (False, True), "both": (True, True)}[kind], p


def _check_device(dev, M, K, N, bar):
    g = torch.Generator(device=dev).manual_seed(M + K)
    W = torch.randint(0, 256, (N, K // 128, 28), generator=g, device=dev, dtype=torch.uint8)
    W[:, :, 26:] = (0.02 * torch.randn((N, K // 128, 1), generator=g, device=dev)).abs().half().view(torch.uint8)
    W = W.view(N, -1)
    Q, SX = ops.quant_rows(torch.randn((M, K), generator=g, device=dev).half(), ldS=M + 5)
    T8, SW = ops.expand_i8(W, K, N)
    x = (Q.double().view(M, -1, 128) * SX[:, :M].double().t()[:, :, None]).view(M, K)
    w = (T8.double().view(N, -1, 128) * SW.double()[:, :, None]).view(N, K)
    ref = x @ w.t()
    C = ops.gemm_ptq1_i8(Q, SX, W, K, N)
    err = float((C.double() - ref).norm() / ref.norm())
    assert err < bar, err
    assert torch.equal(ops.gemm_ptq1_i8(Q, SX, W, K, N, out_dtype=torch.float16), C.half())


@pytest.mark.parametrize("rows,kind,M,K,N", [
    (32, "split", 1, 1152, 700), (64, "whole", 1000, 384, 2050), (64, "split", 1000, 1920, 700),
    (64, "split", 41, 5120, 10240), (128, "whole", 257, 384, 17001), (128, "split", 257, 3968, 5120),
    (128, "split", 100, 5120, 12288), (128, "both", 700, 1152, 12001), (256, "whole", 513, 384, 8003),
    (256, "split", 600, 5120, 2050), (256, "both", 1000, 1152, 9000)])
def test_tile_heights(dev, rows, kind, M, K, N):
    """Every tile height with whole tiles, all tiles split and (128, 256) a split rest, ragged rows
    and columns, even and odd numbers of groups."""
    _plan_is(dev, M, K, N, rows, kind)
    _check_device(dev, M, K, N, 1e-6)


def test_rows_beyond_32_bit_offsets(dev):
    """From K = 2^23 the tall kernel takes every size (the short tiles' row offsets are 32-bit).  Bar:
    16 pieces of 4097 group sums, a walk of sqrt(4097 / 2) 2^-24 0.6 = 1.6e-6."""
    K = (1 << 23) + 128
    _plan_is(dev, 2, K, 3, 256, "split")
    _plan_is(dev, 2, K - 128, 3, 32, "split")
    _check_device(dev, 2, K, 3, 7e-6)
    _check_device(dev, 2, K - 128, 3, 7e-6)


@pytest.mark.parametrize("rows,M,K,N", [(32, 1, 1408, 257), (32, 20, 1408, 300), (64, 1000, 1920, 700), (128, 257, 3968, 5120),
                                        (256, 600, 3200, 2050)])
def test_integer_sums_exact(dev, rows, M, K, N):
    """Unit scales: the exact integer sum, whatever the tile height and the split."""
    _plan_is(dev, M, K, N, rows, "split")
    rng = np.random.default_rng(M)
    t = rng.integers(-1, 2, (N, K)).astype(np.int8)
    W = torch.from_numpy(orc.pack(t, np.ones((N, K // 128), np.float16))).to(dev)
    A8 = rng.integers(-127, 128, (M, K)).astype(np.int8)
    C = ops.gemm_ptq1_i8(torch.from_numpy(A8).to(dev), torch.ones((K // 128, M), device=dev), W, K, N)
    assert np.array_equal(C.cpu().numpy().astype(np.float64), A8.astype(np.float64) @ t.astype(np.float64).T)
