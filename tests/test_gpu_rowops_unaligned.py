"""Row operators on rows that start at any 4-byte address: odd row lengths at
the edges of the register layouts, strides that no vector width divides,
buffers offset by one to three floats, with the words around every row left
alone.  Bars as in the other row-operator tests (1e-4; maxima, indices and
one-hot gradients bit for bit)."""
import numpy as np
import pytest

import bwpp
from bwpp import synth
from conftest import assert_bits_equal, rel_max_err

pytestmark = pytest.mark.gpu
TOL = 1e-4
GUARD = 5.0


def _at(x, ld, off):
    """(buffer, view address) of x in rows of ld floats, off floats in."""
    import torch
    rows, cols = x.shape
    buf = torch.full((rows * ld + 8,), GUARD, device="cuda")
    buf[off:off + rows * ld].view(rows, ld)[:, :cols] = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    return buf, buf.data_ptr() + 4 * off


def _get(buf, rows, cols, ld, off):
    b = buf.cpu().numpy()
    m = b[off:off + rows * ld].reshape(rows, ld)
    assert np.all(b[:off] == GUARD) and np.all(b[off + rows * ld:] == GUARD) and np.all(m[:, cols:] == GUARD)
    return m[:, :cols]


@pytest.mark.parametrize("rows,cols,pad,off", [
    (1, 1, 0, 1), (700, 2, 0, 0), (300, 3, 1, 2), (9, 4, 0, 1), (9, 5, 0, 3), (33, 255, 0, 0), (17, 257, 0, 1), (600, 1023, 0, 2), (31, 1024, 1, 0),
    (13, 1537, 0, 3), (9, 2049, 0, 0), (700, 4096, 3, 1), (11, 4097, 0, 0), (5, 5003, 0, 2), (5, 8191, 0, 0),
    (3, 16383, 0, 1), (3, 32767, 0, 3), (2, 32769, 0, 1)])
def test_unaligned_rows(be, oracle, rows, cols, pad, off):
    import torch
    x = synth.normal((rows, cols), cols, 0)
    x[:, cols // 2] = x[:, 0]  # a tie now and then
    g, bt = synth.uniform((cols,), cols, 1, 0.5, 1.5), synth.normal((cols,), cols, 2, 0.0, 0.1)
    dy = synth.normal((rows,), cols, 3)
    ld = cols + pad
    xb, xp = _at(x, ld, off)
    gb, gp = _at(g[None], cols, (off + 1) % 4)
    bb, bp = _at(bt[None], cols, (off + 2) % 4)
    blank = np.zeros_like(x)
    rp = bwpp.RmsnormParams(rows, cols, ld, 1e-5)
    mp = bwpp.ReduceParams(rows, cols, ld, 1)
    for name, run, want in (
            ("softmax", lambda y: be.dispatch_softmax(xp, y, bwpp.SoftmaxParams(rows, cols, ld)), oracle.softmax(x)),
            ("layernorm", lambda y: be.dispatch_layernorm(xp, gp, bp, y, rp), oracle.layernorm(x, g, bt, 1e-5)),
            ("rmsnorm", lambda y: be.dispatch_rmsnorm(xp, gp, None, y, rp), oracle.rmsnorm(x, g, None, 1e-5))):
        yb, yp = _at(blank, ld, (off + 3) % 4)
        run(yp)
        assert rel_max_err(_get(yb, rows, cols, ld, (off + 3) % 4), want) <= TOL, name
    dyd = torch.from_numpy(dy).cuda()
    for name, run, want in (
            ("mask", lambda y: be.dispatch_reduce_max_mask(xp, y, mp), oracle.reduce_max_mask(x, 1)),
            ("grad", lambda y: be.dispatch_reduce_max_grad_argmax(xp, None, dyd, y, mp),
             oracle.reduce_max_grad(dy, x.shape, x=x, axis=1))):
        yb, yp = _at(blank, ld, off)
        run(yp)
        assert np.array_equal(_get(yb, rows, cols, ld, off), want), name
    mv, ix = torch.zeros(rows, device="cuda"), torch.zeros(rows, dtype=torch.int32, device="cuda")
    be.dispatch_reduce_max(xp, mv, ix, mp)
    wm, wi = oracle.reduce_max(x, 1)
    assert_bits_equal(mv.cpu().numpy(), wm)
    assert np.array_equal(ix.cpu().numpy(), wi)
    _get(xb, rows, cols, ld, off), _get(gb, 1, cols, cols, (off + 1) % 4), _get(bb, 1, cols, cols, (off + 2) % 4)


@pytest.mark.parametrize("cols", [2, 4])
def test_most_rows(be, cols):
    """More rows than one launch takes at four rows a block (2^32 threads, run
    in pieces of 2^25 rows); softmax within 1e-5, the others exact."""
    import torch
    rows = (1 << 26) + 5
    x = torch.randn(rows, cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    y = torch.full_like(x, GUARD)
    be.dispatch_softmax(x, y, bwpp.SoftmaxParams(rows, cols, cols))
    assert bool(((y - torch.softmax(x, dim=1)).abs() <= 1e-5).all())
    mp = bwpp.ReduceParams(rows, cols, cols, 1)
    mv, ix = torch.full((rows,), GUARD, device="cuda"), torch.full((rows,), 7, device="cuda", dtype=torch.int32)
    be.dispatch_reduce_max(x, mv, ix, mp)
    want, arg = x.max(dim=1)
    assert torch.equal(mv, want) and torch.equal(x.gather(1, ix.long()[:, None])[:, 0], want)
    be.dispatch_reduce_max_grad_argmax(x, None, mv, y, mp)
    assert torch.equal(y, torch.zeros_like(x).scatter_(1, ix.long()[:, None], want[:, None]))


@pytest.mark.parametrize("rows,cols", [(4000, 1921), (4000, 4095), (4000, 5003), (2000, 9001)])
def test_softmax_scale_error(be, rows, cols):
    """The rounding of a row's sum (its common factor: the row's outputs add
    up to 1 but for that) where 4 and 8 waves share a row.  Rounded additions
    of the whole sum's size: 1 + 1/2 + 1/4 for eight waves in pairs, about 1/4
    in the lanes, and the reciprocal: 3.0, and sqrt(3.0) 2^-24 / sqrt(3) over
    the mean mantissa (1.25) is 0.80 x 2^-24; eight waves one after another
    make it 4.4, 0.97.  The bar lies between, ten deviations of the estimate
    from the first."""
    import torch
    x = torch.randn(rows, cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    y = torch.empty_like(x)
    be.dispatch_softmax(x, y, bwpp.SoftmaxParams(rows, cols, cols))
    rms = float((y.double().sum(dim=1) - 1).pow(2).mean().sqrt())
    assert rms <= (0.88 if cols > 4096 else 0.83) * 2.0 ** -24
