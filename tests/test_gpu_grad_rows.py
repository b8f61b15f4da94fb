"""The row-in-register gradient kernels and the axis-0 sum at the edges of
their layouts: the last row length of one layout and the first of the next,
rows at 4-byte addresses, strided rows, a row count that leaves a block's
last rows empty, in-place outputs.  Bars: 1e-5 of the largest result, about
50 times the rounding of an fp32 sum of the longest rows."""
import numpy as np
import pytest

import bwpp
from bwpp import synth
from conftest import rel_max_err

pytestmark = pytest.mark.gpu
TOL = 1e-5
PAD = 5.0

COLS = [(3, 0), (256, 0), (257, 0), (1024, 4), (1025, 0), (2048, 0), (2050, 0), (4096, 1), (4100, 0), (8191, 0),
        (8192, 0), (8196, 0)]


def _dev(x, ld):
    import torch
    t = torch.full((x.shape[0], ld), PAD, device="cuda")
    t[:, : x.shape[1]] = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    return t


def _host(t, cols):
    a = t.cpu().numpy()
    assert np.all(a[:, cols:] == PAD)
    return a[:, :cols]


@pytest.mark.parametrize("rows", [1, 5, 600])
@pytest.mark.parametrize("cols,pad", COLS + [(16384, 0), (16383, 0), (16388, 0)])
def test_softmax_grad_layouts(be, oracle, rows, cols, pad):
    if rows * cols > 5_000_000:
        rows = 37
    y = np.abs(synth.normal((rows, cols), 1, 0))
    y = (y / y.sum(axis=1, keepdims=True)).astype(np.float32)
    dy = synth.normal((rows, cols), 1, 1)
    want = oracle.softmax_grad(y, dy)
    ld = cols + pad
    p = bwpp.SoftmaxParams(rows, cols, ld)
    yd, dyd = _dev(y, ld), _dev(dy, ld)
    out = _dev(np.zeros_like(y), ld)
    be.dispatch_softmax_grad(yd, dyd, out, p)
    assert rel_max_err(_host(out, cols), want) <= TOL
    be.dispatch_softmax_grad(yd, dyd, dyd, p)  # dx in dy's place
    assert np.array_equal(_host(dyd, cols), _host(out, cols))


@pytest.mark.parametrize("rows", [1, 6, 1100])
@pytest.mark.parametrize("cols,pad", COLS)
def test_rmsnorm_grad_layouts(be, oracle, rows, cols, pad):
    import torch
    if rows * cols > 5_000_000:
        rows = 261  # one row more per block for some of the 256 blocks
    x, dy, acc = (synth.normal((rows, cols), 2, i) for i in range(3))
    g = synth.uniform((cols,), 2, 3, 0.5, 1.5)
    want, wg, wb = oracle.rmsnorm_grad(x, g, dy, 1e-5)
    ld = cols + pad
    p = bwpp.RmsnormParams(rows, cols, ld, 1e-5)
    xd, dyd, gd = _dev(x, ld), _dev(dy, ld), torch.from_numpy(g).cuda()
    dx = _dev(np.zeros_like(x), ld)
    parts = cols <= 8192
    dg, db = (torch.full((cols,), 7.0, device="cuda") if parts else None for _ in range(2))
    be.dispatch_rmsnorm_grad(xd, gd, dyd, dx, dg, db, p)
    got = _host(dx, cols)
    assert rel_max_err(got, want) <= TOL
    if parts:
        assert rel_max_err(dg.cpu().numpy(), wg) <= TOL
        assert rel_max_err(db.cpu().numpy(), wb) <= TOL
    accd = _dev(acc, ld)  # the accumulating form, in place: one rounded add
    be.dispatch_rmsnorm_grad_acc(xd, gd, dyd, accd, accd, None, None, p)
    if parts:
        assert np.array_equal(_host(accd, cols), acc + got)
    else:
        assert rel_max_err(_host(accd, cols), acc + want) <= TOL


@pytest.mark.parametrize("rows,cols,pad", [(1, 3, 0), (63, 64, 0), (64, 65, 0), (1000, 130, 2), (40000, 7, 0),
                                           (2050, 4097, 0)])
def test_reduce_sum_axis0_bands(be, rows, cols, pad):
    import torch
    x = synth.normal((rows, cols), 3, 0)
    out = torch.full((cols,), 7.0, device="cuda")
    be.dispatch_reduce_sum(_dev(x, cols + pad), out, bwpp.ReduceParams(rows, cols, cols + pad, 0))
    want = x.astype(np.float64).sum(axis=0)
    # an fp32 sum's error bound, gamma_n of the band and merge sums' depth (< 100 additions)
    bound = 100 * 2.0 ** -24 * np.abs(x.astype(np.float64)).sum(axis=0)
    assert np.all(np.abs(out.cpu().numpy() - want) <= bound)


@pytest.mark.parametrize("rows", [(1 << 26) - 4, (1 << 26) + 5])
def test_softmax_grad_most_rows(be, rows):
    """The last row count that one launch of four rows a block can take, and
    the first beyond it (2^32 threads); one column, dx = y (dy - dy y), three
    roundings."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(1)
    y = torch.rand(rows, device="cuda", generator=gen)
    dy = torch.randn(rows, device="cuda", generator=gen)
    out = torch.full_like(y, 7.0)
    be.dispatch_softmax_grad(y, dy, out, bwpp.SoftmaxParams(rows, 1, 1))
    torch.cuda.synchronize()
    want = y.double() * (dy.double() - dy.double() * y.double())
    assert bool(((out.double() - want).abs() <= 3 * 2.0 ** -24 * dy.double().abs()).all())
