"""The bf16 forward at head dims 32, 64 and 96 (matrix-core kernels with the
probabilities split into two bf16 terms), where it can go wrong: edges of the
128-query and 64-key tiles, more queries than keys, strided rows, and
infinite or NaN values in V.  The bar is the bf16 rounding of the result
(2^-8 of it: 8 significant bits) with 1e-4 for everything before: the fp32 arithmetic of the
generic path, which a row stride that is no multiple of 8 still takes."""
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


def _forward(be, q, k, v, scale, causal, pad=0):
    """O and lse (float32) through rows of D + pad elements."""
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


@pytest.mark.parametrize("D", [32, 64, 96])
@pytest.mark.parametrize("B,H,M,N,pad", [(1, 1, 33, 1, 0), (2, 4, 128, 64, 0), (1, 3, 127, 129, 8), (1, 2, 129, 65, 0),
                                         (2, 1, 33, 1000, 16), (1, 1, 513, 200, 0), (1, 2, 300, 300, 0)])
@pytest.mark.parametrize("causal", [False, True])
def test_small_head_dims(be, oracle, D, B, H, M, N, pad, causal):
    (q, qh), (k, kh), (v, vh) = (_bf16(synth.normal((B, H, r, D), M + N, i)) for i, r in enumerate((M, N, N)))
    for scale in (D ** -0.5, 1.0):
        o, lse = _forward(be, q, k, v, scale, causal, pad)
        assert be.last_kernel == f"bwpp_attn_bf16_d{D}" + ("_causal" if causal else "")
        assert rel_max_err(o, oracle.attention_bh(qh, kh, vh, scale, causal)) <= TOL
        want = oracle.attention_lse(qh, kh, scale, causal)
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(lse), fin)
        assert np.all(np.abs(lse[fin] - want[fin]) <= 1e-5 * np.maximum(1.0, np.abs(want[fin])))
    # against the generic path on the same values: the same bf16 results up to one rounding
    g, _ = _forward(be, q, k, v, 1.0, causal, 3)
    assert be.last_kernel == "bwpp_attn_generic_bf16" + ("_causal" if causal else "")
    assert np.all(np.abs(o - g) <= 2.0 ** -7 * np.abs(g) + 2e-5 * np.abs(vh).max())


@pytest.mark.parametrize("D", [32, 64, 96])
@pytest.mark.parametrize("M,N,causal", [(200, 200, True), (70, 150, True), (40, 100, False)])
def test_non_finite_values(be, D, M, N, causal):
    """An infinity reaches exactly the queries that see its key, a NaN the
    same, wherever the key lies in its tile; other outputs are finite."""
    H = 3
    (q, _), (k, _), (_, vh) = (_bf16(synth.normal((1, H, r, D), 9, i)) for i, r in enumerate((M, N, N)))
    vh = vh.copy()
    vh[0, 0, N - 1, 5] = np.inf     # the last key: the row that padding re-reads
    vh[0, 1, N // 2 + 3, 7] = -np.inf
    vh[0, 1, N // 2 + 3, 8] = np.nan
    v, vh = _bf16(vh)
    o, _ = _forward(be, q, k, v, D ** -0.5, causal)
    g, _ = _forward(be, q, k, v, D ** -0.5, causal, 3)  # generic path
    assert np.array_equal(np.isnan(o), np.isnan(g))
    assert np.array_equal(np.isposinf(o), np.isposinf(g)) and np.array_equal(np.isneginf(o), np.isneginf(g))
    fin = np.isfinite(g)
    assert np.all(np.abs(o[fin] - g[fin]) <= 2.0 ** -7 * np.abs(g[fin]) + 1e-4)


@pytest.mark.parametrize("B,H,M,N,D,causal", [(4, 8, 335, 335, 64, 0), (2, 8, 500, 500, 32, 0), (2, 8, 500, 500, 96, 1),
                                              (8, 8, 16, 513, 64, 1), (4, 8, 1, 1200, 128, 0)])
def test_lse_error(be, B, H, M, N, D, causal):
    """lse is rounded once (with at most 32 queries too): rms 1/sqrt(12) =
    0.29 ulp, and 0.2 ulp for the sums before; 0.57 to 0.62 ulp with a logf of
    the whole sum and plain additions.  Bar 0.45."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(B, H, r, D, device="cuda", generator=gen).to(torch.bfloat16) for r in (M, N, N))
    o, lse = torch.zeros_like(q), torch.zeros(B, H, M, device="cuda")
    be.dispatch_attention_lse(q, k, v, o, lse, bwpp.AttentionParams(M=M, N=N, K=D, D=D, batch=B, heads=H, scale=D ** -0.5,
                                                                    causal=causal, dtype=int(bwpp.DType.BF16)))
    err = []
    for b in range(B):
        for h in range(H):
            s = (q[b, h].double() @ k[b, h].double().t().contiguous()) * D ** -0.5
            if causal:
                m = torch.arange(M, device="cuda")[:, None]
                s.masked_fill_(torch.arange(N, device="cuda")[None] > m + (N - M), -float("inf"))
            want = torch.logsumexp(s, dim=1)
            ulp = 2.0 ** (torch.floor(torch.log2(want.abs().clamp(min=0.5))) - 23)
            err.append((lse[b, h].double() - want) / ulp)
    assert float(torch.cat(err).pow(2).mean().sqrt()) <= 0.45
