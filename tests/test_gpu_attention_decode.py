"""The bf16 forward for at most 32 queries (a block's waves split the keys,
long caches are split over blocks), where it can go wrong: fewer keys than a
tile or than waves, key counts around the tile and around a split, every query
count with the causal mask, strided rows, infinite and NaN values in V at
masked and visible keys, and a graph the caller records.  The bar is the bf16
rounding of the result (2^-8) with 1e-4 for everything before."""
import numpy as np
import pytest

import bwpp
from bwpp import synth
from conftest import rel_max_err

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -8 + 1e-4


def _bf16(x):
    import torch
    bits = synth.to_bf16_bits(np.ascontiguousarray(x, np.float32))
    return torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16), synth.bf16_bits_to_f32(bits)


def _forward(be, q, k, v, scale, causal, pad=0, out=None):
    import torch
    B, H, M, D = q.shape
    N, ld = k.shape[2], D + pad

    def rows(t):
        r = torch.full(t.shape[:3] + (ld,), 3.0, dtype=torch.bfloat16, device="cuda")
        r[..., :D] = t
        return r

    o = torch.full((B, H, M, ld), 5.0, dtype=torch.bfloat16, device="cuda")
    lse = torch.full((B, H, M), 5.0, device="cuda")
    be.dispatch_attention_lse(rows(q), rows(k), rows(v), o, lse,
                              bwpp.AttentionParams(M=M, N=N, K=D, D=D, ldq=ld, ldk=ld, ldv=ld, ldo=ld, batch=B, heads=H,
                                                   scale=scale, causal=int(causal), dtype=int(bwpp.DType.BF16)))
    torch.cuda.synchronize()
    assert bool((o[..., D:] == 5.0).all())
    return o[..., :D].float().cpu().numpy(), lse.cpu().numpy()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,M,N,pad", [(1, 1, 1, 1, 0), (1, 2, 1, 31, 0), (2, 2, 3, 33, 8), (1, 1, 32, 32, 0),
                                         (1, 2, 32, 100, 0), (2, 1, 17, 9, 0), (1, 3, 2, 1024, 0), (1, 1, 5, 4133, 8),
                                         (3, 2, 1, 3000, 0), (1, 300, 1, 170, 0)])
@pytest.mark.parametrize("causal", [False, True])
def test_decode(be, oracle, D, B, H, M, N, pad, causal):
    (q, qh), (k, kh), (v, vh) = (_bf16(synth.normal((B, H, r, D), M + N, i)) for i, r in enumerate((M, N, N)))
    for scale in (D ** -0.5, 0.5):
        o, lse = _forward(be, q, k, v, scale, causal, pad)
        split = be.last_kernel == "bwpp_attn_dec_combine_bf16"
        assert be.recent_kernel(1 if split else 0) == f"bwpp_attn_bf16_dec_d{D}" + ("_causal" if causal else "")
        assert split == (N >= 1024)  # few slices: long caches are split
        assert rel_max_err(o, oracle.attention_bh(qh, kh, vh, scale, causal)) <= TOL
        want = oracle.attention_lse(qh, kh, scale, causal)
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(lse), fin)
        assert np.all(np.abs(lse[fin] - want[fin]) <= 1e-5 * np.maximum(1.0, np.abs(want[fin])))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("M,N,causal", [(20, 70, True), (8, 2060, True), (4, 45, False)])
def test_non_finite_values(be, D, M, N, causal):
    """An infinity or NaN in V reaches exactly the queries that see its key."""
    H = 3
    (q, _), (k, _), (_, vh) = (_bf16(synth.normal((1, H, r, D), 9, i)) for i, r in enumerate((M, N, N)))
    vh = vh.copy()
    vh[0, 0, N - 1, 5] = np.inf  # the last key: the row that padding re-reads
    vh[0, 1, N - 3, 7] = -np.inf
    vh[0, 1, N - 3, 8] = np.nan
    vh[0, 2, 3, 60] = np.inf     # seen by all
    v, vh = _bf16(vh)
    o, _ = _forward(be, q, k, v, D ** -0.5, causal)
    g, _ = _forward(be, q, k, v, D ** -0.5, causal, 3)  # generic path
    assert np.array_equal(np.isnan(o), np.isnan(g))
    assert np.array_equal(np.isposinf(o), np.isposinf(g)) and np.array_equal(np.isneginf(o), np.isneginf(g))
    fin = np.isfinite(g)
    assert np.all(np.abs(o[fin] - g[fin]) <= 2.0 ** -7 * np.abs(g[fin]) + 1e-4)


def test_caller_capture():
    """A graph the caller records runs unsplit; replays between eager (split)
    calls agree to the rounding of the results."""
    import torch
    h = bwpp.HipBackend(0)
    try:
        gen = torch.Generator(device="cuda").manual_seed(1)
        q, k, v = (torch.randn(1, 2, n, 128, device="cuda", generator=gen).to(torch.bfloat16) for n in (1, 4000, 4000))
        o, e = torch.zeros_like(q), torch.zeros_like(q)
        p = bwpp.AttentionParams(M=1, N=4000, K=128, D=128, batch=1, heads=2, scale=0.09, dtype=int(bwpp.DType.BF16))
        side = torch.cuda.Stream()
        h.set_stream(side)
        torch.cuda.synchronize()
        h.dispatch_attention(q, k, v, e, p)
        assert h.last_kernel == "bwpp_attn_dec_combine_bf16"
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            h.set_stream(torch.cuda.current_stream())
            h.dispatch_attention(q, k, v, o, p)
        assert h.last_kernel == "bwpp_attn_bf16_dec_d128"
        h.set_stream(side)
        for _ in range(3):
            o.zero_()
            g.replay()
            h.dispatch_attention(q, k, v, e, p)
            torch.cuda.synchronize()
            assert bool(((o.float() - e.float()).abs() <= 2.0 ** -7 * e.float().abs() + 1e-5).all())
    finally:
        torch.cuda.synchronize()
        h.close()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,M,N,pad", [(1, 1, 1, 1, 0), (1, 2, 1, 31, 0), (2, 2, 3, 33, 4), (1, 1, 32, 32, 0),
                                         (1, 2, 32, 100, 0), (2, 1, 17, 9, 0), (1, 1, 5, 4133, 4), (1, 300, 1, 70, 0)])
@pytest.mark.parametrize("causal", [False, True])
def test_decode_f32(be, oracle, D, B, H, M, N, pad, causal):
    """The fp32 kernel; bar 1e-5 of the largest result (sums of up to 4133
    terms in a dozen partial sums, 2^-24 each)."""
    import torch
    q, k, v = (synth.normal((B, H, r, D), M + N, i) for i, r in enumerate((M, N, N)))
    ld, scale = D + pad, D ** -0.5

    def rows(t):
        r = torch.full(t.shape[:3] + (ld,), 3.0, device="cuda")
        r[..., :D] = torch.from_numpy(t).cuda()
        return r

    o = torch.full((B, H, M, ld), 5.0, device="cuda")
    lse = torch.full((B, H, M), 5.0, device="cuda")
    prm = bwpp.AttentionParams(M=M, N=N, K=D, D=D, ldq=ld, ldk=ld, ldv=ld, ldo=ld, batch=B, heads=H, scale=scale,
                               causal=int(causal))
    be.dispatch_attention_lse(rows(q), rows(k), rows(v), o, lse, prm)
    torch.cuda.synchronize()
    split = be.last_kernel == "bwpp_attn_dec_combine_f32"
    assert be.recent_kernel(1 if split else 0) == f"bwpp_attn_f32_dec_d{D}" + ("_causal" if causal else "")
    assert split == (N >= 1024)
    assert bool((o[..., D:] == 5.0).all())
    assert rel_max_err(o[..., :D].cpu().numpy(), oracle.attention_bh(q, k, v, scale, causal)) <= 1e-5
    want, got = oracle.attention_lse(q, k, scale, causal), lse.cpu().numpy()
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin)
    assert np.all(np.abs(got[fin] - want[fin]) <= 1e-5 * np.maximum(1.0, np.abs(want[fin])))
    if M == 1:  # an infinity at the last key, whose row the padding re-reads
        vi = v.copy()
        vi[..., N - 1, 3] = np.inf
        be.dispatch_attention(rows(q), rows(k), rows(vi), o, prm)
        torch.cuda.synchronize()
        assert bool(torch.isposinf(o[..., 0, 3]).all()) and bool(torch.isfinite(o[..., 0, 4:D]).all())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("M,N,causal", [(20, 70, True), (8, 2060, True), (4, 45, False), (32, 32, True)])
def test_non_finite_values_f32(be, D, M, N, causal):
    """The same for the fp32 kernel, against the generic path (rows that no
    16-byte load divides); finite results within 1e-5 of the largest."""
    import torch
    H = 3
    q, k, v = (synth.normal((1, H, r, D), 9, i) for i, r in enumerate((M, N, N)))
    v[0, 0, N - 1, 5] = np.inf   # seen by the last query only under the mask
    v[0, 1, N - 3, 7] = -np.inf
    v[0, 1, N - 3, 8] = np.nan
    v[0, 2, 3, 60] = np.inf

    def run(ld):
        def rows(t):
            r = torch.full(t.shape[:3] + (ld,), 3.0, device="cuda")
            r[..., :D] = torch.from_numpy(t).cuda()
            return r

        o = torch.full((1, H, M, ld), 5.0, device="cuda")
        be.dispatch_attention(rows(q), rows(k), rows(v), o,
                              bwpp.AttentionParams(M=M, N=N, K=D, D=D, ldq=ld, ldk=ld, ldv=ld, ldo=ld, batch=1, heads=H,
                                                   scale=D ** -0.5, causal=int(causal)))
        torch.cuda.synchronize()
        return o[..., :D].cpu().numpy()

    o, first = run(D), be.recent_kernel(1 if be.last_kernel == "bwpp_attn_dec_combine_f32" else 0)
    assert first.startswith(f"bwpp_attn_f32_dec_d{D}")
    g = run(D + 1)
    assert be.last_kernel.startswith("bwpp_attn_generic_f32")
    assert np.array_equal(np.isnan(o), np.isnan(g))
    assert np.array_equal(np.isposinf(o), np.isposinf(g)) and np.array_equal(np.isneginf(o), np.isneginf(g))
    fin = np.isfinite(g)
    assert np.all(np.abs(o[fin] - g[fin]) <= 1e-5 * np.abs(g[fin]).max())
