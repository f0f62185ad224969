"""The Q8_0 prefill GEMM over the sizes where its tile shapes and schedules change: rows at the
edges of the 64 row tiles and ragged ones of 128 and 256, columns around the 256 column tiles, one
to many 128-k blocks, K splits, and the last rows of the matrix at the end of an allocation.

Reference: float64 products of the expanded weights.  Bar: 1e-5 relative L2 (fp32 sums of K fp16
products err by about sqrt(K) 2^-24 of their scale)."""
import numpy as np
import pytest
import torch

from kata_amd import ops
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _check(dev, M, K, N):
    W_np, q, d = orc.synth_q8(N, K, M + K + N)
    W = torch.from_numpy(W_np).to(dev)
    A = torch.from_numpy(orc.synth_x(M, K, M + 1)).to(dev)
    C = ops.gemm_q8_f16(A, W, K, N)
    w = (torch.from_numpy(q).to(dev).double().view(N, K // 32, 32) *
         torch.from_numpy(d.astype(np.float64)).to(dev)[:, :, None]).half().double().view(N, K)
    ref = A.double() @ w.t()
    err = float((C.double() - ref).norm() / ref.norm())
    assert err < 1e-5, err
    assert torch.equal(ops.gemm_q8_f16(A, W, K, N, out_dtype=torch.float16), C.half())


@pytest.mark.parametrize("rows,kind,M,K,N", [
    (64, "split", 1, 1152, 257), (64, "whole", 100, 384, 1000), (128, "whole", 200, 384, 17001),
    (128, "split", 600, 2432, 2050), (128, "both", 400, 1408, 17001), (256, "whole", 400, 384, 17001),
    (256, "split", 129, 5120, 12001), (256, "split", 1000, 10240, 5120), (256, "both", 1000, 1152, 17001)])
def test_tile_heights(dev, rows, kind, M, K, N):
    """Every tile height with whole tiles, all tiles split and (128, 256) a split rest."""
    p = ops.prefill_plan("q8", M, K, N, torch.cuda.get_device_properties(dev).multi_processor_count)
    assert p.tile_rows == rows and (p.whole > 0, p.split > 0) == {"whole": (True, False), "split": (False, True), "both": (True, True)}[kind], p
    _check(dev, M, K, N)


@pytest.mark.parametrize("M", [1, 63, 64, 65, 128, 129, 256, 300, 900])
@pytest.mark.parametrize("K,N", [(128, 3), (256, 257), (640, 255), (5120, 1024)])
def test_tile_edges(dev, M, K, N):
    _check(dev, M, K, N)
