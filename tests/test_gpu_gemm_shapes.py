"""The fp16 prefill GEMM over the sizes where its tile shapes and schedules change: rows at
the edges of the 32, 64, 128 and 256 row tiles, columns around the 256 column tiles, odd and
even numbers of 128-k blocks (the packed weights are copied two blocks at a time), K splits of
all tiles and of the last round, scales of 1 and more (another decode form), several matrices in
one launch, rows too far apart for 32-bit offsets, weight rows too long for them.  Where a test
means a tile height or a split it asks the planner, so that a shape that no longer takes it fails.

Reference: float64 products of the expanded weights.  Bar: fp32 sums of K fp16 products err by
about sqrt(K) 2^-24 of their scale, at most 8e-6 at K = 17408 (1e-5 as for the other shapes)."""
import ctypes

import numpy as np
import pytest
import torch

from kata_amd import ops
from kata_amd.capi import check, lib
from kata_amd.engine import Dispatch, dispatch_work_bytes
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _weights(dev, K, N, seed, big):
    rng = np.random.default_rng(seed)
    t = rng.integers(-1, 2, (N, K)).astype(np.int8)
    d = np.abs(rng.normal(0, 0.02, (N, K // 128)))
    if big == "tiny":                           # subnormal fp16 scales, in the fast decode form
        d *= 2e-5
    elif big:                                   # blocks at and above 1, tiny and zero scales
        d[:, ::3] *= 5000.0
        d[1::7] = 1.0
        d[::5, 1::4] = 3e-7
        d[::11] = 0.0
    return torch.from_numpy(orc.pack(t, d.astype(np.float16))).to(dev)


def _check(C, A, W, K, N):
    ref = A.double() @ ops.expand_f16(W, K, N).double().t()
    err = float((C.double() - ref).norm() / ref.norm())
    assert err < 1e-5, err


@pytest.mark.parametrize("big", [False, "tiny", True])
@pytest.mark.parametrize("M", [1, 31, 32, 33, 64, 65, 127, 129, 256, 257, 700])
@pytest.mark.parametrize("K,N", [(128, 257), (384, 1000), (2176, 256), (5120, 255)])
def test_tile_edges(dev, M, K, N, big):
    W = _weights(dev, K, N, M + K + N, big)
    A = torch.from_numpy(orc.synth_x(M, K, M + 5)).to(dev)
    _check(ops.gemm_ptq1_f16(A, W, K, N), A, W, K, N)


def _plan_is(dev, fmt, M, K, N, rows, kind):
    p = ops.prefill_plan(fmt, M, K, N, torch.cuda.get_device_properties(dev).multi_processor_count)
    assert p.tile_rows == rows and (p.whole > 0, p.split > 0) == {"whole": (True, False), "split": (False, True), "both": (True, True)}[kind], p


def _device_weights(dev, K, N, seed, late):
    """Weights made on the GPU; late: in every other 32 columns each third block from block 2 on
    has a scale of 1 and more, so those waves change the decode form inside their piece."""
    g = torch.Generator(device=dev).manual_seed(seed)
    W = torch.randint(0, 256, (N, K // 128, 28), generator=g, device=dev, dtype=torch.uint8)
    d = (0.02 * torch.randn((N, K // 128), generator=g, device=dev)).abs()
    if late:
        d[(torch.arange(N, device=dev) // 32) % 2 == 1, 2::3] *= 5000.0
    W[:, :, 26:] = d.half().view(torch.uint8).view(N, -1, 2)
    return W.view(N, -1)


@pytest.mark.parametrize("late", [False, True])
@pytest.mark.parametrize("rows,kind,M,K,N", [
    (32, "split", 1, 1152, 257), (64, "whole", 1000, 384, 2050), (64, "split", 513, 3968, 257),
    (128, "whole", 513, 384, 8003), (128, "split", 1000, 3968, 2050), (128, "both", 400, 1920, 17001),
    (128, "both", 1000, 5120, 9000), (256, "whole", 700, 384, 12001), (256, "both", 1000, 5120, 17001)])
def test_tile_heights(dev, rows, kind, M, K, N, late):
    """Every tile height with whole tiles, all tiles split or (128, 256) a split rest, ragged rows and columns,
    even and odd numbers of blocks; every column by itself, so small ones count beside large, in
    units of the norm that a column of such products has (a lone sum may come out near zero)."""
    _plan_is(dev, "f16", M, K, N, rows, kind)
    W = _device_weights(dev, K, N, M + K, late)
    A = torch.from_numpy(orc.synth_x(M, K, M + 6)).to(dev)
    C = ops.gemm_ptq1_f16(A, W, K, N)
    w = ops.expand_f16(W, K, N).double()
    err = (C.double() - A.double() @ w.t()).norm(dim=0) / (A.double().norm() * w.norm(dim=1) / K ** 0.5)
    assert float(err.max()) < 1e-5, float(err.max())
    assert torch.equal(ops.gemm_ptq1_f16(A, W, K, N, out_dtype=torch.float16), C.half())


@pytest.mark.parametrize("op", ["f16", "q8"])
def test_rows_far_apart(dev, op):
    """Rows more than 2^24 elements apart go one by one: the bits of each row's own call."""
    M, K, N, lda = 3, 640, 300, (1 << 24) + 8
    A = torch.zeros((M, lda), dtype=torch.float16, device=dev)
    A[:, :K] = torch.from_numpy(orc.synth_x(M, K, 11)).to(dev)
    W = _weights(dev, K, N, 12, True) if op == "f16" else torch.from_numpy(orc.synth_q8(N, K, 12)[0]).to(dev)
    gemm = ops.gemm_ptq1_f16 if op == "f16" else ops.gemm_q8_f16
    C = gemm(A, W, K, N)
    for m in range(M):
        assert torch.equal(C[m:m + 1], gemm(A[m:m + 1, :K].contiguous(), W, K, N)), m


def test_long_weight_rows(dev):
    """Weight rows of 2^24 bytes and more (256 of them span 4 GiB) go 255 columns at a time: the bits
    of those columns' own calls.  Against float64 sums of 7.7e7 products: a single wrong 128-block
    of a row would show as 1.1e-3 = 1 / sqrt(K / 128) and more, the roundings of the 3e5 adds of each
    piece as 1.3e-4; the bar lies between them."""
    K, N = 128 * 599187, 257
    W = _device_weights(dev, K, N, 13, False)
    assert W.shape[1] * 256 > 0xffffffff >= W.shape[1] * 255
    A = torch.randn((1, K), generator=torch.Generator(device=dev).manual_seed(14), device=dev).half()
    C = ops.gemm_ptq1_f16(A, W, K, N)
    for a, b in ((0, 255), (255, 257)):
        assert torch.equal(C[:, a:b], ops.gemm_ptq1_f16(A, W[a:b], K, b - a))
    cols = [0, 7, 254, 255, 256]
    ref = torch.stack([A[0].double() @ ops.expand_f16(W[n:n + 1], K, 1)[0].double() for n in cols])
    err = float((C[0, cols].double() - ref).norm() / ref.norm())
    assert err < 5e-4, err


def test_strided_and_unaligned(dev):
    """lda > K, an odd ldc > N, and a weight base at a 2-byte (not 4-byte) address."""
    M, K, N = 70, 640, 301
    W = _weights(dev, K, N, 9, False)
    buf = torch.zeros(W.numel() + 2, dtype=torch.uint8, device=dev)
    buf[2:] = W.reshape(-1)
    A = torch.from_numpy(orc.synth_x(M, K + 8, 10)).to(dev)
    out = torch.full((M, N + 6), 7.0, device=dev)
    ops.gemm_ptq1_f16(A, buf[2:], K, N, out=out)
    _check(out[:, :N], A[:, :K], W, K, N)
    assert bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("M", [30, 200])
def test_matrices_of_one_launch(dev, M):
    """The dispatcher's prefill form runs the matrices that share an input as one launch: ragged
    widths, each against its own product; an int8 one among them goes its own way."""
    H = 1024
    Ns, names = (300, 1024, 129, 2050), ("qkv", "wq", "wk", "z")
    Ws = [_weights(dev, H, N, 20 + i, False) for i, N in enumerate(Ns)]
    offs = np.cumsum([0] + [W.numel() for W in Ws])
    d = Dispatch(torch.cat([W.reshape(-1) for W in Ws]))
    x = torch.from_numpy(orc.synth_x(M, H, 30)).to(dev).float()
    gs = torch.ones(H, device=dev)
    work = torch.empty(dispatch_work_bytes("prefill", H, M), dtype=torch.uint8, device=dev)
    for i8 in ("none", "wq"):
        d.set_i8(i8)
        outs = d.sub_in("prefill", [(int(offs[i]), Ns[i], names[i]) for i in range(4)], x, None, gs, work=work)
        h = work[:2 * M * H].view(torch.float16).view(M, H)
        for W, N, nm, C in zip(Ws, Ns, names, outs):
            if nm == i8:
                Q, SX = ops.quant_rows(h.contiguous())
                assert torch.equal(C, ops.gemm_ptq1_i8(Q, SX, W, H, N))
            else:
                _check(C, h, W, H, N)


@pytest.mark.parametrize("op,M,K,N", [("f16", 40, 2048, 1024), ("q8", 40, 2048, 1024), ("i8", 41, 5120, 1024), ("i8", 512, 5120, 5120)])
def test_first_call_captured(dev, op, M, K, N):
    """A stream's first GEMM may be captured: without the workspace no tile is split.  Every replay
    gives the bits of the others and, but for the order of its sums, the eager call's result."""
    A = torch.from_numpy(orc.synth_x(M, K, 41)).to(dev)
    if op == "q8":
        W = torch.from_numpy(orc.synth_q8(N, K, 40)[0]).to(dev)
        call = lambda C: ops.gemm_q8_f16(A, W, K, N, out=C)
    else:
        W = _weights(dev, K, N, 40, False)
        Q, SX = ops.quant_rows(A)
        call = (lambda C: ops.gemm_ptq1_i8(Q, SX, W, K, N, out=C)) if op == "i8" else (lambda C: ops.gemm_ptq1_f16(A, W, K, N, out=C))
    C, eager = torch.empty((M, N), device=dev), torch.empty((M, N), device=dev)
    call(eager)
    torch.cuda.synchronize()
    s = torch.cuda.Stream(dev)
    check(lib().kata_release_stream(ctypes.c_void_p(s.cuda_stream)))    # torch reuses streams: no workspace left
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(C)
    first = None
    for _ in range(3):
        C.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        first = C.clone() if first is None else first
        assert torch.equal(C, first)
        err = float((C.double() - eager.double()).norm() / eager.double().norm())
        assert err < 2e-5, err                  # two sums in fp32, each within 1e-5 of the exact one
