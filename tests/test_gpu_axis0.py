"""Axis-0 reduce_max, its mask and its gradients where the split over row
bands can go wrong: bands that do not divide the rows, columns past a
64-column block, strided and unaligned rows, in-place outputs, a scratch
shared between streams, and a graph that the caller records (which takes the
one-pass kernels).  Maxima, indices, masks and one-hot gradients are the
strict fold's bits whatever the split, so every comparison is exact."""
import numpy as np
import pytest

import bwpp
from conftest import assert_bits_equal

pytestmark = pytest.mark.gpu


def _matrix(rows, cols, seed):
    """Few distinct values (ties in every column), a column of -inf, one of
    NaN, one whose maximum is a zero of both signs."""
    rng = np.random.default_rng(seed)
    x = rng.integers(-6, 3, (rows, cols)).astype(np.float32)
    x[rng.random((rows, cols)) < 0.01] = np.nan
    if cols > 3:
        x[:, 0] = -np.inf
        x[:, 1] = np.nan
        x[:, 2] = -np.abs(x[:, 2]) - 1
        x[rows // 2, 2] = -0.0
        x[rows - 1, 2] = 0.0 if rows > 1 else -0.0
    return x


def _padded(x, ld, fill):
    import torch
    t = torch.full((x.shape[0], ld), fill, device="cuda")
    t[:, : x.shape[1]] = torch.from_numpy(x).cuda()
    return t


@pytest.mark.parametrize("rows,cols,pad", [(1, 1, 0), (31, 64, 0), (32, 65, 0), (65, 4, 4), (1000, 63, 3),
                                           (2049, 257, 0), (8200, 128, 4), (20011, 5, 0), (300, 4100, 1)])
def test_axis0(be, oracle, rows, cols, pad):
    import torch
    x = _matrix(rows, cols, rows + cols)
    ld = cols + pad
    p = bwpp.ReduceParams(rows, cols, ld, 0)
    xd = _padded(x, ld, 5.0)
    mv, ix = torch.zeros(cols, device="cuda"), torch.zeros(cols, dtype=torch.int32, device="cuda")
    be.dispatch_reduce_max(xd, mv, ix, p)
    wm, wi = oracle.reduce_max(x, 0)
    assert_bits_equal(mv.cpu().numpy(), wm)
    assert np.array_equal(ix.cpu().numpy(), wi)
    dy = np.random.default_rng(3).standard_normal(cols).astype(np.float32)
    dyd = torch.from_numpy(dy).cuda()
    want_mask = oracle.reduce_max_mask(x, 0)
    want_dx = oracle.reduce_max_grad(dy, x.shape, x=x, axis=0)
    for name, run, want in (
            ("mask", lambda s, d: be.dispatch_reduce_max_mask(s, d, p), want_mask),
            ("grad x", lambda s, d: be.dispatch_reduce_max_grad_argmax(s, None, dyd, d, p), want_dx),
            ("grad argmax", lambda s, d: be.dispatch_reduce_max_grad_argmax(None, ix, dyd, d, p), want_dx)):
        for in_place in (False, True):
            src = xd.clone()
            dst = src if in_place else torch.full_like(src, 9.0)
            run(src, dst)
            got = dst.cpu().numpy()
            assert np.array_equal(got[:, :cols], want), (name, in_place)
            assert np.all(got[:, cols:] == (5.0 if in_place else 9.0)), (name, in_place)


def test_axis0_streams_and_capture(oracle):
    """One handle on two streams in turn (the second's use of the scratch
    waits for the first's), then a graph recorded by the caller: the same
    results, from the kernels that take no scratch, on every replay."""
    import torch
    rows, cols = 4100, 192
    xs = [_matrix(rows, cols, 50 + i) for i in range(2)]
    wants = [oracle.reduce_max_mask(x, 0) for x in xs]
    p = bwpp.ReduceParams(rows, cols, cols, 0)
    h = bwpp.HipBackend(0)
    try:
        xd = [torch.from_numpy(x).cuda() for x in xs]
        out = [torch.zeros_like(t) for t in xd]
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        torch.cuda.synchronize()
        for _ in range(3):
            for s, x, o in zip(streams, xd, out):
                h.set_stream(s)
                h.dispatch_reduce_max_mask(x, o, p)
        torch.cuda.synchronize()
        assert h.last_kernel == "bwpp_col_mask_apply_v4"
        for o, w in zip(out, wants):
            assert np.array_equal(o.cpu().numpy(), w)
        g = torch.cuda.CUDAGraph()
        buf, res = xd[0].clone(), torch.zeros_like(xd[0])
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            h.set_stream(torch.cuda.current_stream())
            h.dispatch_reduce_max_mask(buf, res, p)
        assert h.last_kernel == "bwpp_col_mask"
        h.set_stream(streams[0])
        for i in (1, 0, 1):
            buf.copy_(xd[i])
            res.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(res.cpu().numpy(), wants[i])
            h.dispatch_reduce_max_mask(xd[i], out[i], p)  # eager work between the replays
            torch.cuda.synchronize()
            assert np.array_equal(out[i].cpu().numpy(), wants[i])
    finally:
        torch.cuda.synchronize()
        h.close()


@pytest.mark.parametrize("cols", [(1 << 30) + 4, (1 << 30) + 5])
def test_most_columns(be, cols):
    """More columns than one launch of 64 a block takes (2^32 threads): two
    rows of 2^30 columns, in pieces."""
    import torch
    x = torch.randn(2, cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    mv, ix = torch.full((cols,), 9.0, device="cuda"), torch.full((cols,), 9, device="cuda", dtype=torch.int32)
    p = bwpp.ReduceParams(2, cols, cols, 0)
    be.dispatch_reduce_max(x, mv, ix, p)
    assert torch.equal(mv, torch.maximum(x[0], x[1])) and torch.equal(ix, (x[1] > x[0]).int())
    dx = torch.full_like(x, 9.0)
    be.dispatch_reduce_max_grad_argmax(None, ix, mv, dx, p)
    for r in range(2):
        assert torch.equal(dx[r], torch.where(ix == r, mv, torch.zeros((), device="cuda")))
