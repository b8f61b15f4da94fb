"""The bf16 GEMM kernels for any M, N and K: every tile, through LDS DMA and
through registers, all transposes, with and without a K split, at the edges of
the tiles and of the last K stage, rows at 2-byte addresses, NaN in the padding
of the operands' rows (never multiplied) and C's padding left alone.  Against
float64; the bar is the bf16 rounding of the result (2^-8) and 2^-17 of the sum
of magnitudes for the fp32 accumulation (K <= 700 terms of 2^-24, either
order)."""
import numpy as np
import pytest

import bwpp

pytestmark = pytest.mark.gpu

SHAPES = [(128, 128, 128), (129, 136, 136), (33, 72, 264), (8, 8, 128), (257, 264, 392)]   # 16-byte rows (but M with ta)
ODD = [(1, 9, 129), (65, 131, 133), (9, 257, 255), (130, 8, 641), (256, 512, 160)]


def _operand(rows, cols, pad, off, gen):
    """rows x cols in rows of cols + pad, off elements into a NaN-filled buffer."""
    import torch
    buf = torch.full((off + rows * (cols + pad) + 16,), float("nan"), device="cuda", dtype=torch.bfloat16)
    v = buf[off:off + rows * (cols + pad)].view(rows, cols + pad)
    v[:, :cols] = torch.randn(rows, cols, device="cuda", generator=gen).to(torch.bfloat16)
    return buf, v


def _check(h, M, N, K, ta, tb, pad, off, epi):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(M * 7 + N * 3 + K)
    _, a = _operand(*((K, M) if ta else (M, K)), pad, off, gen)
    _, b = _operand(*((N, K) if tb else (K, N)), pad, off, gen)
    bias = torch.randn(N + 1, device="cuda", generator=gen).to(torch.bfloat16)[1:]
    cbuf = torch.full((off + M * (N + pad) + 16,), 7.0, device="cuda", dtype=torch.bfloat16)
    c = cbuf[off:off + M * (N + pad)].view(M, N + pad)
    h.dispatch_matmul(a.data_ptr(), b.data_ptr(), c.data_ptr(), bias.data_ptr(),
                      bwpp.MatmulParams(M, N, K, a.shape[1], b.shape[1], N + pad, int(bwpp.DType.BF16), epi, ta, tb))
    torch.cuda.synchronize()
    A = (a[:, :M].t() if ta else a[:, :K]).double().contiguous()
    B = (b[:, :K].t() if tb else b[:, :N]).double().contiguous()
    want = A @ B
    mag = A.abs() @ B.abs()
    if epi & 1:
        want = want + bias.double()
    if epi & 2:
        want = want * torch.sigmoid(want)
    err = (c[:, :N].double() - want).abs()
    assert bool((err <= 2.0 ** -8 * want.abs() + 2.0 ** -17 * (mag + 1)).all()), (M, N, K, float(err.max()))
    assert bool((c[:, N:] == 7.0).all()) and bool((cbuf[:off] == 7.0).all()) and bool((cbuf[-16:] == 7.0).all())


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5])
def test_every_tile(monkeypatch, tile, ta, tb):
    import torch
    for split in (1, 2, 3):
        for unaligned in ("", "u"):
            monkeypatch.setenv("BWPP_GEMM_RING", f"{tile},{split}{unaligned}")
            h = bwpp.HipBackend(0)
            try:
                h.set_stream(torch.cuda.current_stream())
                for i, (M, N, K) in enumerate(SHAPES):
                    _check(h, M, N, K, ta, tb, 8 * (i % 2), 0, i % 4)
                    first = h.recent_kernel(1 if h.last_kernel == "bwpp_gemm_bf16_splitk_reduce" else 0)
                    dma = not unaligned and (M if ta else K) % 8 == 0 and (K if tb else N) % 8 == 0
                    assert first.startswith("bwpp_gemm_bf16r") and first.endswith("_u") != dma, first
                for i, (M, N, K) in enumerate(ODD):
                    if (ta and M < 8) or (not tb and N < 8):
                        continue
                    _check(h, M, N, K, ta, tb, i % 3, i % 2, 3 - i % 4)
            finally:
                torch.cuda.synchronize()
                h.close()


@pytest.mark.parametrize("M,N,K,tb", [(16, 1024, 2048, 0), (1, 4096, 512, 1), (300, 77, 4100, 0), (2, 5, 300, 0),
                                      (3, 7, 1000, 1), (1, 64, 64, 0), (300, 264, 8, 1), (2000, 64, 100, 0),
                                      (33, 40, 31, 0), (255, 1000, 127, 1), (9, 13, 7, 0)])
def test_chosen(be, M, N, K, tb):
    """The default choice, and the fewest columns (N < 8, B row-major: the
    guarded edge kernel), and K from the edge kernel's 7 to less than one K
    stage."""
    _check(be, M, N, K, 0, tb, 0, 0, 3)


@pytest.mark.parametrize("M,N,K,ta,tb", [(256, 3000, 33, 1, 0), (512, 264, 63, 0, 1), (1024, 100, 48, 1, 1),
                                         (256, 11008, 8, 0, 0), (256, 520, 31, 1, 0)])
def test_whole_row_tiles_short_k(be, M, N, K, ta, tb):
    """Whole 256-row tiles whose K is short and no multiple of 32 (a gradient
    over a few tokens): no 256-wide kernel runs there."""
    _check(be, M, N, K, ta, tb, 0, 0, 3)
    assert be.last_kernel.startswith("bwpp_gemm_bf16r")


def test_caller_capture(be):
    """A graph the caller records takes no split (it may be replayed beside
    the handle's other work); its replays match the eager result to the
    rounding of another order of the sums."""
    import torch
    M, N, K = 8, 512, 4096
    h = bwpp.HipBackend(0)
    try:
        gen = torch.Generator(device="cuda").manual_seed(1)
        a, b = (torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
        c, e = (torch.zeros(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(2))
        p = bwpp.MatmulParams(M, N, K, K, N, N, int(bwpp.DType.BF16), 0, 0, 0)
        side = torch.cuda.Stream()
        h.set_stream(side)
        torch.cuda.synchronize()
        h.dispatch_matmul(a, b, e, None, p)
        assert h.last_kernel == "bwpp_gemm_bf16_splitk_reduce"
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            h.set_stream(torch.cuda.current_stream())
            h.dispatch_matmul(a, b, c, None, p)
        assert h.last_kernel.startswith("bwpp_gemm_bf16r")
        h.set_stream(side)
        for _ in range(3):
            c.zero_()
            g.replay()
            h.dispatch_matmul(a, b, e, None, p)
            torch.cuda.synchronize()
            assert bool(((c.double() - e.double()).abs() <= 2.0 ** -7 * e.double().abs() + 1e-3).all())
    finally:
        torch.cuda.synchronize()
        h.close()


@pytest.mark.parametrize("M,N,K", [(128, 1024, 4096), (512, 512, 4096)])
def test_caller_capture_tile(monkeypatch, M, N, K):
    """A graph the caller records takes the tile that is best without a
    split, which a handle that never splits chooses, and not the split's."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(1)
    a, b = (torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    c, e = (torch.zeros(M, N, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    p = bwpp.MatmulParams(M, N, K, K, N, N, int(bwpp.DType.BF16), 0, 0, 0)
    h = bwpp.HipBackend(0)
    monkeypatch.setenv("BWPP_GEMM_SPLITK", "0")
    ref = bwpp.HipBackend(0)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        h.set_stream(s)
        ref.set_stream(s)
        h.dispatch_matmul(a, b, c, None, p)
        assert h.last_kernel == "bwpp_gemm_bf16_splitk_reduce"
        ref.dispatch_matmul(a, b, e, None, p)
        assert ref.last_kernel != h.recent_kernel(1)  # the split's tile is another
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            h.dispatch_matmul(a, b, c, None, p)
        assert h.last_kernel == ref.last_kernel
        for _ in range(3):
            c.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                g.replay()
            torch.cuda.synchronize()
            assert torch.equal(c, e)
            ref.dispatch_matmul(a, b, e, None, p)
            torch.cuda.synchronize()
    finally:
        torch.cuda.synchronize()
        h.close()
        ref.close()


def test_first_split_while_another_stream_is_recorded():
    """The scratch's one allocation does not disturb a recording (in the mode
    that forbids allocations to the whole process) on another stream, and the
    call splits."""
    import torch
    M, N, K = 8, 512, 4096
    gen = torch.Generator(device="cuda").manual_seed(1)
    a, b = (torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) for s in ((M, K), (K, N)))
    c, x = torch.zeros(M, N, device="cuda", dtype=torch.bfloat16), torch.zeros(64, device="cuda")
    h = bwpp.HipBackend(0)
    try:
        h.set_stream(torch.cuda.Stream())
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, capture_error_mode="global"):
            x.add_(1.0)
            h.dispatch_matmul(a, b, c, None, bwpp.MatmulParams(M, N, K, K, N, N, int(bwpp.DType.BF16), 0, 0, 0))
        assert h.last_kernel == "bwpp_gemm_bf16_splitk_reduce"
        for i in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert bool((x == i + 1).all())
        want = a.double() @ b.double()
        assert bool(((c.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-3).all())
    finally:
        torch.cuda.synchronize()
        h.close()
