"""The fp32 GEMM kernels for any M, N and K: every tile, all transposes, with
and without a K split, at the edges of the tiles and of the last K stage, rows
at any 4-byte address with NaN in their padding, and the fused tails (residual
in place, dual output, SiLU gradient) on ragged columns.  Against float64; the
bar is 2^-20 of the sum of magnitudes: chains of at most 128 fp32 additions
inside the MFMA accumulators (2^-24 each, random signs), then as many sums."""
import pytest

import bwpp

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 4), (4, 5, 37), (33, 35, 133), (64, 65, 128), (129, 67, 257), (128, 128, 300), (70, 260, 31)]


def _operand(rows, cols, pad, off, gen):
    import torch
    buf = torch.full((off + rows * (cols + pad) + 8,), float("nan"), device="cuda")
    v = buf[off:off + rows * (cols + pad)].view(rows, cols + pad)
    v[:, :cols] = torch.randn(rows, cols, device="cuda", generator=gen)
    return v


def _check(h, M, N, K, ta, tb, pad, off, epi, fuse):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(M * 7 + N * 3 + K)
    a = _operand(*((K, M) if ta else (M, K)), pad, off, gen)
    b = _operand(*((N, K) if tb else (K, N)), pad, (off + 1) % 4, gen)
    bias = torch.randn(N + 1, device="cuda", generator=gen)[1:]
    aux = torch.randn(M, N + 1, device="cuda", generator=gen)
    c = torch.full((M, N + pad), 7.0, device="cuda")
    c2 = torch.full((M, N + 3), 7.0, device="cuda")
    want = ((a[:, :M].t() if ta else a[:, :K]).double().contiguous() @
            (b[:, :K].t() if tb else b[:, :N]).double().contiguous())
    mag = ((a[:, :M].t() if ta else a[:, :K]).double().abs().contiguous() @
           (b[:, :K].t() if tb else b[:, :N]).double().abs().contiguous()) + 2
    if fuse == 3:
        epi = 0
    if fuse == 2:
        epi &= 1
    prm = bwpp.MatmulParams(M, N, K, a.shape[1], b.shape[1], N + pad, int(bwpp.DType.F32), epi, ta, tb)
    if fuse == 1:  # residual in place
        c[:, :N] = aux[:, :N]
        aux_p, ld_aux = c.data_ptr(), N + pad
    else:
        aux_p, ld_aux = aux.data_ptr(), N + 1
    if fuse:
        h.dispatch_matmul_fused(a.data_ptr(), b.data_ptr(), c.data_ptr(), bias.data_ptr(),
                                aux_p if fuse != 2 else None, c2.data_ptr() if fuse == 2 else None, prm,
                                bwpp.FusionParams(fuse, ld_aux if fuse != 2 else 0, N + 3 if fuse == 2 else 0))
    else:
        h.dispatch_matmul(a.data_ptr(), b.data_ptr(), c.data_ptr(), bias.data_ptr(), prm)
    torch.cuda.synchronize()
    if epi & 1:
        want = want + bias.double()
    if epi & 2:
        want = want * torch.sigmoid(want)
    x = aux[:, :N].double()
    if fuse == 1:
        want = want + x
    if fuse == 3:
        s = torch.sigmoid(x)
        want = want * (s * (1 + x * (1 - s)))
    tag = (M, N, K, ta, tb, pad, off, epi, fuse)
    assert bool(((c[:, :N].double() - want).abs() <= 2.0 ** -20 * 2 * mag).all()), tag
    assert bool((c[:, N:] == 7.0).all()), tag
    if fuse == 2:
        assert bool(((c2[:, :N].double() - want * torch.sigmoid(want)).abs() <= 2.0 ** -20 * 3 * mag).all()), tag
        assert bool((c2[:, N:] == 7.0).all()), tag


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tile", [1, 2, 3])
def test_every_tile(monkeypatch, tile, ta, tb):
    import torch
    for split in (1, 2, 3):
        monkeypatch.setenv("BWPP_GEMM_RING", f"{tile},{split}")
        h = bwpp.HipBackend(0)
        try:
            h.set_stream(torch.cuda.current_stream())
            for i, (M, N, K) in enumerate(SHAPES):
                if (ta and M < 4) or ((not ta or tb) and K < 4):
                    continue
                for fuse in range(4):
                    _check(h, M, N, K, ta, tb, i % 3, i % 4, (i + fuse) % 4, fuse)
                    first = h.recent_kernel(1 if h.last_kernel == "bwpp_gemm_f32_splitk_reduce" else 0)
                    assert first.startswith("bwpp_gemm_f32r"), first
        finally:
            torch.cuda.synchronize()
            h.close()


@pytest.mark.parametrize("M,N,K,ta,tb", [(3, 2, 1000, 0, 0), (2, 300, 3, 0, 1), (1, 1, 1, 1, 0), (256, 256, 256, 0, 0),
                                         (32, 384, 5823, 0, 0), (1, 4096, 129, 0, 1), (600, 3, 70, 0, 1)])
def test_chosen(be, M, N, K, ta, tb):
    """The default choice, with operands below the 16-byte chunks among them
    (the guarded edge kernel)."""
    for fuse in range(4):
        _check(be, M, N, K, ta, tb, 1, 2, 3, fuse)


@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("M,N,K", [(128, 128, 4096), (256, 256, 8192)])
def test_caller_capture(monkeypatch, M, N, K, warm):
    """A full-tile size that splits K through the workspace: a graph that the
    caller records after a warm-up call splits too (the same kernels, the same
    bits); one recorded on a new handle, which may not allocate, takes the
    choice of a handle that never splits."""
    import torch

    def names(h):
        return [h.recent_kernel(i) for i in (0, 1)]

    gen = torch.Generator(device="cuda").manual_seed(1)
    a, b = torch.randn(M, K, device="cuda", generator=gen), torch.randn(K, N, device="cuda", generator=gen)
    e, c = torch.zeros(M, N, device="cuda"), torch.zeros(M, N, device="cuda")
    p = bwpp.MatmulParams(M, N, K, K, N, N, int(bwpp.DType.F32), 0, 0, 0)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    if not warm:
        monkeypatch.setenv("BWPP_GEMM_SPLITK", "0")
    ref = bwpp.HipBackend(0)
    monkeypatch.delenv("BWPP_GEMM_SPLITK", raising=False)
    h = ref if warm else bwpp.HipBackend(0)
    try:
        ref.set_stream(s)
        h.set_stream(s)
        ref.dispatch_matmul(a, b, e, None, p)
        want = names(ref)
        assert (want[0] == "bwpp_gemm_f32_splitk_reduce") == warm
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            h.dispatch_matmul(a, b, c, None, p)
        assert names(h) == want if warm else h.last_kernel == want[0]
        for _ in range(3):
            c.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                g.replay()
            torch.cuda.synchronize()
            assert torch.equal(c, e)
            e.zero_()
            torch.cuda.synchronize()
            ref.dispatch_matmul(a, b, e, None, p)  # eager work between the replays
            torch.cuda.synchronize()
    finally:
        torch.cuda.synchronize()
        ref.close()
        if h is not ref:
            h.close()


def test_most_columns(be):
    """Columns for which 64-wide tiles would be a launch of 2^32 threads."""
    import torch
    N, K, step = 1 << 30, 4, 1 << 27
    gen = torch.Generator(device="cuda").manual_seed(1)
    a, b = torch.randn(1, K, device="cuda", generator=gen), torch.randn(K, N, device="cuda", generator=gen)
    c = torch.full((1, N), 7.0, device="cuda")
    be.dispatch_matmul(a, b, c, None, bwpp.MatmulParams(1, N, K, K, N, N, int(bwpp.DType.F32), 0, 0, 0))
    assert be.last_kernel.startswith("bwpp_gemm_f32r")
    for n in range(0, N, step):
        t = a[0, :, None].double() * b[:, n:n + step].double()
        assert bool(((c[0, n:n + step].double() - t.sum(0)).abs() <= 2.0 ** -21 * t.abs().sum(0)).all())
