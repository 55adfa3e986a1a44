"""Selection on rows with about k entries that are not masked (GPU): by -inf, NaN,
the dtype's lowest value or another value shared by most of the row.

Expected, from a stable sort: the other entries, then the masked ones by
ascending id, and no NaN entry -- slots left over hold -1 (in supports wider
than 64 the first NaN entries, with probability 0).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from d3d_amd import _lib
from d3d_amd import draft as dr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
INF, NAN = float("inf"), float("nan")


def _rows(V, k, dtype):
    """(rows, entries that are not NaN): k + d finite entries and d' at -inf, the rest -inf or NaN."""
    g = torch.Generator().manual_seed(V + k)
    out = []
    for finite, inf, rest in ((0, 0, -INF), (1, 0, -INF), (k - 1, 0, -INF), (k, 0, -INF), (k + 1, 0, -INF),
                              (k // 2, k, NAN), (k // 2, k - k // 2, NAN), (k // 2, 1, NAN), (0, 0, NAN)):
        row = torch.full((V,), rest)
        at = torch.randperm(V, generator=g)
        row[at[:finite]] = (torch.randn(finite, generator=g) * 3).to(dtype).float()
        row[at[finite:finite + inf]] = -INF
        out.append(row)
    return torch.stack(out).to(dtype)


def _shared(V, k, value, dtype):
    """Rows of one value but for k + d larger entries (and, in odd rows, some smaller ones)."""
    g = torch.Generator().manual_seed(V + k)
    out = []
    for n, larger in enumerate((0, 1, k - 1, k, k + 1)):
        row = torch.full((V,), value)
        at = torch.randperm(V, generator=g)
        up = torch.rand(larger, generator=g) * 4 + 0.5
        row[at[:larger]] = value + up if abs(value) < 1e5 else up
        if n % 2:
            row[at[larger:larger + V // 8]] = -INF
        out.append(row)
    return torch.stack(out).to(dtype)


def _sorted_ids(x, k):
    out = np.full((x.shape[0], k), -1, np.int64)
    for n, row in enumerate(x.float().numpy()):
        ok = np.flatnonzero(~np.isnan(row))
        order = ok[np.lexsort((ok, -row[ok]))][:k]
        out[n, :order.size] = order
    return out


@pytest.mark.parametrize("V,k", [(151936, 64), (151936, 9), (9000, 64), (300, 33), (64, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_top_k_and_support(V, k, dtype):
    x = _rows(V, min(k, V - 1), dtype)
    ref = _sorted_ids(x, k)
    ids, vals = dr.topk_tokens(x.to(DEV), k, with_values=True)
    np.testing.assert_array_equal(ids.cpu().numpy(), ref)
    want = torch.where(ids.cpu() < 0, -INF, x.float().gather(1, ids.cpu().clamp(min=0)))
    assert torch.equal(vals.cpu(), want)
    u = torch.rand(x.shape[0], generator=torch.Generator().manual_seed(k)).to(DEV)
    tok, sid, probs = dr.sample_with_sparse_probs(x.to(DEV), 0.8, k, uniforms=u)
    np.testing.assert_array_equal(sid.cpu().numpy(), ref)
    _check_support(x, tok.cpu(), sid.cpu(), probs.cpu())


@pytest.mark.parametrize("value", ["lowest", -1e9, -10000.0, -2.0, 0.0, 3.0])
@pytest.mark.parametrize("V,k", [(151936, 64), (151935, 64), (20000, 400), (20000, 4000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_most_of_the_row_shares_a_value(value, V, k, dtype):
    x = _shared(V, k, torch.finfo(dtype).min if value == "lowest" else value, dtype)
    N, T = x.shape[0], 1.25
    xd = x.to(DEV)
    u = torch.rand(N, generator=torch.Generator().manual_seed(k))
    tok, sid, probs = dr.sample_with_sparse_probs(xd, T, k, uniforms=u.to(DEV))
    z = x.float() / T
    np.testing.assert_array_equal(sid.cpu().numpy(), _sorted_ids(z, k))
    q = z.double().gather(1, sid.cpu()).softmax(-1)
    # fp32 exponentials, an fp64 sum, a division
    assert torch.allclose(probs.cpu().double(), q, rtol=1e-6, atol=1e-37)
    if k <= 64:
        ids, vals = dr.topk_tokens(xd, k, with_values=True)
        np.testing.assert_array_equal(ids.cpu().numpy(), _sorted_ids(x, k))
        assert torch.equal(vals, x.float().to(DEV).gather(1, ids))
    for p in (1.0, 0.8):
        _check_filter(x, T, k, p, u)


def _check_support(x, tok, sid, probs):
    live = x.float().gather(1, sid.clamp(min=0))
    live = (sid >= 0) & (live > -INF)
    assert torch.equal(probs > 0, live)
    for n in range(x.shape[0]):
        if live[n].any():
            assert abs(float(probs[n].sum()) - 1) < 1e-5 and int(tok[n]) in sid[n][live[n]].tolist()
        else:
            assert int(tok[n]) == _lib.D3D_TOKEN_EMPTY_DISTRIBUTION


@pytest.mark.parametrize("V", [151936, 9000])
def test_wide_support(V):
    k = 300
    x = _rows(V, k, torch.bfloat16)
    u = torch.full((x.shape[0],), 0.5, device=DEV)
    tok, sid, probs = dr.sample_with_sparse_probs(x.to(DEV), 0.8, k, uniforms=u)
    ref = _sorted_ids(x, k)
    for n in range(ref.shape[0]):  # the first NaN entries fill the row up
        nan = np.flatnonzero(np.isnan(x[n].float().numpy()))
        gap = ref[n] < 0
        ref[n][gap] = nan[:gap.sum()]
    np.testing.assert_array_equal(sid.cpu().numpy(), ref)
    _check_support(x, tok.cpu(), sid.cpu(), probs.cpu())


@pytest.mark.parametrize("V,k", [(151936, 50), (151936, 1025), (9000, 300), (300, 33)])
@pytest.mark.parametrize("p", [1.0, 0.8])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_filter_and_draw(V, k, p, dtype):
    x = _rows(V, k, dtype)
    _check_filter(x, 0.8, k, p, torch.rand(x.shape[0], generator=torch.Generator().manual_seed(k)))


def _check_filter(x, T, k, p, u):
    """(zfloor, zlimit) against the general filter, the draw against the fp64 sums of the kept entries."""
    N, V = x.shape
    xd = x.to(DEV)
    zf, lim = torch.empty(N, device=DEV), torch.empty(N, dtype=torch.int32, device=DEV)
    st = _lib.load().d3d_row_filter(xd.data_ptr(), _lib.dtype_code(xd), N, V, T, k, p, zf.data_ptr(), lim.data_ptr(),
                                    _lib.stream_ptr(DEV))
    _lib.check(st, "d3d_row_filter")
    got = dr._filters(xd, T, k, p, True)
    assert torch.equal(got[0].view(torch.int32), zf.view(torch.int32)) and torch.equal(got[1], lim)
    tok, prob = (t.cpu() for t in dr.sample_with_prob(xd, T, k, p, uniforms=u.to(DEV)))
    z = (x.float() / T).double()
    ids = torch.arange(V)
    for n in range(N):
        f, l = float(zf[n]), int(lim[n])
        kept = (z[n] > f) | ((z[n] == f) & (ids <= l))
        w = torch.where(kept & (z[n] > -INF), (z[n] - z[n][kept].max() if kept.any() else z[n]).exp(), 0.0)
        if not float(w.sum()) > 0:
            assert int(tok[n]) == _lib.D3D_TOKEN_EMPTY_DISTRIBUTION
            continue
        q = w / w.sum()
        t = int(tok[n])
        hi = float(q[:t + 1].sum())
        # the masses are whole multiples of 2^-40 of the largest weight, the
        # scaled logits' fp32 rounding moves each by some 2^-20
        assert hi - float(q[t]) - 1e-5 <= float(u[n]) <= hi + 1e-5
        assert abs(float(prob[n]) - float(q[t])) <= 2e-5 * float(q[t])


def test_scaling_that_overflows_counts_as_minus_infinity():
    V, k, T = 20000, 12, 0.5
    x = torch.full((1, V), -INF)
    x[0, 100:116] = -3.0e38  # / T: -inf
    x[0, 5000:5004] = torch.tensor([1.0, 4.0, 2.0, 3.0])
    tok, sid, probs = dr.sample_with_sparse_probs(x.to(DEV), T, k, uniforms=torch.zeros(1, device=DEV))
    assert sid[0].tolist() == [5001, 5003, 5002, 5000] + list(range(8))
    assert int(tok[0]) == 5001 and bool((probs[0, 4:] == 0).all())


@pytest.mark.parametrize("unit,T", [(2.0 ** -149, 1.7), (2.0 ** -149, 40.0), (2.0 ** -120, 3e8), (2.0 ** -30, 3.3e38)])
@pytest.mark.parametrize("k", [20, 300])
def test_denormal_quotients_tie(unit, T, k):
    """Small multiples of a unit whose quotients by T are a few denormals (or zeros), so different entries tie."""
    V, N = 20000, 4
    g = torch.Generator().manual_seed(k)
    x = (torch.randint(-400, 401, (N, V), generator=g).double() * unit).float()
    x[1:] = x[1:] * (torch.rand(N - 1, V, generator=g) < 0.05)
    z = (x.double() / float(np.float32(T))).float()  # the double quotient rounds once: denormals have few bits
    u = torch.rand(N, generator=g)
    tok, sid, probs = dr.sample_with_sparse_probs(x.to(DEV), T, k, uniforms=u.to(DEV))
    np.testing.assert_array_equal(sid.cpu().numpy(), _sorted_ids(z, k))
    zf, lim = dr._filters(x.to(DEV), T, k, 1.0, True)
    kth = z.sort(dim=-1, descending=True).values[:, k - 1]
    assert torch.equal(zf.cpu(), kth) and bool((lim.cpu() == 2 ** 31 - 1).all())
    # Every kept entry weighs the same (exp(0)): the draw is the floor(u n)-th kept id.
    tok, prob = (t.cpu() for t in dr.sample_with_prob(x.to(DEV), T, k, uniforms=u.to(DEV)))
    for n in range(N):
        kept = torch.nonzero(z[n] >= kth[n])[:, 0]
        at = int(float(u[n]) * len(kept))
        assert int(tok[n]) == int(kept[at]) and abs(float(prob[n]) * len(kept) - 1) < 1e-6
