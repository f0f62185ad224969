"""The int8 prefill GEMM over the sizes where its kernels, tile shapes and schedules change: rows at
the edges of the 32, 64 and 128 row tiles and around where the 256-row kernel takes over, columns
around the 256 column tiles, odd and even numbers of 128-groups, K splits, a scale row stride
wider than M.

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


@pytest.mark.parametrize("M", [20, 50, 100])
def test_integer_sums_exact(dev, M):
    """Unit scales: the exact integer sum, whatever the split."""
    rng = np.random.default_rng(M)
    K, N = 1408, 300
    t = rng.integers(-1, 2, (N, K)).astype(np.int8)
    W = torch.from_numpy(orc.pack(t, np.ones((N, K // 128), np.float16))).to(dev)
    A8 = rng.integers(-127, 128, (M, K)).astype(np.int8)
    C = ops.gemm_ptq1_i8(torch.from_numpy(A8).to(dev), torch.ones((K // 128, M), device=dev), W, K, N)
    assert np.array_equal(C.cpu().numpy().astype(np.int64), A8.astype(np.int64) @ t.astype(np.int64).T)
