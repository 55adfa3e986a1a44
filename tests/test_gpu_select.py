"""The candidate-based top-k and nucleus kernels (GPU) at their edges.

d3d_filter_rows must give the filter of d3d_row_filter (the general
multi-pass selection) bit for bit: both place the cut with the same exact
64-bit masses.  Every row's draw must lie in its bar of the float64 CDF of the
kept entries.  Supports and top-k are checked against a stable CPU sort.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from d3d_amd import _lib
from d3d_amd import draft as dr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
INF = float("inf")


def _rows(kind, N, V, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(N, V, generator=g) * 2.0
    if kind == "ties":       # few distinct values: long runs at every cut
        x = x.round()
    elif kind == "flat":     # one value per row: no candidate list holds it
        x = torch.zeros(N, V)
        x[:, V // 2] = 1.0
    elif kind == "masked":   # most of the vocabulary at -inf
        x[:, ::2] = -INF
        x[N // 2:, 40:] = -INF
    elif kind == "odd":      # NaN, infinities, zeros, denormals, a far outlier
        x[0, ::7] = float("nan")
        x[1, 5] = INF
        x[2, :] = -INF
        x[3, ::3] = 0.0
        x[3, 1::3] = 1e-41
        x[4, V - 1] = 3e38
    elif kind == "sorted":   # the k largest are neighbours: few groups hold them
        x = x.sort(-1, descending=True).values
    return x.to(dtype).to(DEV)


def _general(x, T, k, p):
    N, V = x.shape
    zf = torch.empty(N, device=DEV)
    lim = torch.empty(N, dtype=torch.int32, device=DEV)
    st = _lib.load().d3d_row_filter(x.data_ptr(), _lib.dtype_code(x), N, V, T, k, p, zf.data_ptr(), lim.data_ptr(),
                                    _lib.stream_ptr(DEV))
    _lib.check(st, "d3d_row_filter")
    return zf, lim


def _check_draws(x, T, zf, lim, u, tok, prob):
    """Each row's u lies in the drawn entry's bar of the fp64 CDF of the kept entries, ids in order."""
    x, zf, lim, u, tok, prob = (t.cpu() for t in (x, zf, lim, u, tok, prob))
    z = x.float() / torch.tensor(T)
    ids = torch.arange(x.shape[1])
    for n in range(x.shape[0]):
        kept = (z[n] > zf[n]) | ((z[n] == zf[n]) & (ids <= lim[n]))
        top = z[n][kept].max() if kept.any() else torch.tensor(-INF)
        w = torch.where(kept, (z[n].double() - top.double()).exp(), 0.0).nan_to_num(0.0)
        t = int(tok[n])
        if not torch.isfinite(top):  # no entry has a weight
            assert t == _lib.D3D_TOKEN_EMPTY_DISTRIBUTION and float(prob[n]) == 0
            continue
        q = w / w.sum()
        hi = float(q[:t + 1].sum())
        # z = x / T and z - max round to fp32: 2^-19 of a weight at |z| < 16; the
        # masses' units are 2^-40 and finer
        assert t >= 0 and bool(kept[t])
        assert hi - float(q[t]) - 2e-6 <= float(u[n]) <= hi + 2e-6
        assert abs(float(prob[n]) - float(q[t])) <= 4e-6 * float(q[t])


@pytest.mark.parametrize("kind", ["plain", "ties", "flat", "masked", "odd", "sorted"])
@pytest.mark.parametrize("V,k,p", [(151936, 0, 0.9), (151936, 0, 0.05), (32771, 0, 0.999), (4097, 0, 0.5),
                                   (151936, 1, 1.0), (151936, 64, 0.8), (32771, 257, 0.3), (151936, 1025, 1.0),
                                   (8192, 4096, 0.9), (20000, 300, 1.0), (9, 4, 0.6), (262144, 2000, 0.95)])
@pytest.mark.parametrize("dtype,T", [(torch.bfloat16, 0.7), (torch.float32, 1.3), (torch.float32, 1.0)])
def test_filter_rows_equals_the_general_filter(kind, V, k, p, dtype, T):
    N = 6
    x = _rows(kind, N, V, dtype, V + k)
    u = torch.rand(N, generator=torch.Generator().manual_seed(k)).to(DEV)
    zf, lim = _general(x, T, k, p)
    kk, pp, fused = dr._filter_args(V, k, p)
    assert fused
    got = dr._filters(x, T, kk, pp, fused)
    torch.cuda.synchronize()
    assert torch.equal(got[0], zf) and torch.equal(got[1], lim)
    tok, prob = dr.sample_with_prob(x, T, k, p, uniforms=u)
    _check_draws(x, T, zf, lim, u, tok, prob)


def test_filter_rows_takes_rows_in_batches():
    """More rows than one batch (256), whose scratch the next batch reuses."""
    N, V = 520, 6001
    x = _rows("plain", N, V, torch.bfloat16, 4)
    u = torch.rand(N, device=DEV)
    for k, p in ((0, 0.9), (70, 0.9)):
        zf, lim = _general(x, 0.8, k, p)
        got = dr._filters(x, 0.8, k, p, True)
        tok, _ = dr.sample_with_prob(x, 0.8, k, p, uniforms=u)
        one, _ = dr.sample_with_prob(x[300:301], 0.8, k, p, uniforms=u[300:301])
        torch.cuda.synchronize()
        assert torch.equal(got[0], zf) and torch.equal(got[1], lim) and torch.equal(tok[300:301], one)


def _sorted_ids(x, T, S):
    z = (x.float().cpu() / T).numpy().astype(np.float32)
    out = np.full((z.shape[0], S), -1, np.int64)
    for n, row in enumerate(z):
        ok = np.flatnonzero(~np.isnan(row))  # NaN entries are never selected
        order = ok[np.lexsort((ok, -(row[ok] + np.float32(0))))][:S]
        out[n, :order.size] = order
    return out


@pytest.mark.parametrize("kind", ["plain", "ties", "flat", "masked", "odd", "sorted"])
@pytest.mark.parametrize("V,S", [(151936, 9), (151936, 64), (32771, 256), (32771, 512), (20000, 513), (9000, 4096),
                                 (16, 9), (12, 12)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_support_and_topk_match_a_stable_sort(kind, V, S, dtype):
    N, T = 5 if kind == "odd" else 3, 0.8
    x = _rows(kind, N, V, dtype, V + S)
    u = torch.rand(N, generator=torch.Generator().manual_seed(S)).to(DEV)
    tok, ids, probs = dr.sample_with_sparse_probs(x, T, S, 0.95, uniforms=u)
    ref = _sorted_ids(x, T, S)
    np.testing.assert_array_equal(ids.cpu().numpy(), ref)
    # Rows whose maximum is infinite (of either sign) have no distribution.
    live = torch.isfinite(x.float().nan_to_num(-INF, INF, -INF).amax(-1) / T)
    assert torch.allclose(probs.sum(-1), live.float(), rtol=1e-5)
    assert torch.equal((ids == tok[:, None]).any(-1), live)
    assert bool((tok[~live] == _lib.D3D_TOKEN_EMPTY_DISTRIBUTION).all())
    if S <= 64:
        top, vals = dr.topk_tokens(x, S, with_values=True)
        np.testing.assert_array_equal(top.cpu().numpy(), _sorted_ids(x, 1.0, S))
        assert torch.equal(vals, torch.where(top < 0, -INF, x.float().gather(1, top.clamp(min=0))))


def test_masses_are_as_exact_as_the_exponential_allows():
    """Rows of one 0, n entries of one d and a filtered one, the 0 drawn: its
    probability is 1 / W, W = 1 + n e^d.  In units of 2^-20 of W's value (the
    spacing at [8, 16)), rms: W's rounding 0.289; the quotient's, 2^-27 of p
    against p W^-1 2^-20, 0.289 W^2 / 128, 0.38 over these W; n times e^d's own
    error, 62 / 64 of a unit for each 2^-26 of e^d: 0.29 for the 0.30 of an
    argument-reduced exponential.  Together 0.56, and 0.62 with an e^d of 0.40."""
    N, n, V = 65535, 62, 64
    d = torch.linspace(-2.07, -1.39, N).float()  # e^d in [1/8, 1/4), the sum in [8, 16.5)
    x = d[:, None].repeat(1, V)
    x[:, 0] = 0.0
    x[:, V - 1] = -50.0
    tok, prob = dr.sample_with_prob(x.to(DEV), 1.0, V - 1, uniforms=torch.zeros(N, device=DEV))
    assert bool((tok == 0).all())
    exact = 1.0 / (1.0 + n * d.double().exp())
    err = (prob.cpu().double() / exact - 1) / (exact * 2.0 ** -20)
    assert float(err.square().mean().sqrt()) < 0.59
