"""Rows of more than 2^18 entries, which the candidate selection does not take (GPU)."""
from __future__ import annotations

import pytest
import torch

from d3d_amd import draft as dr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
V = (1 << 18) + 1


def _rows(N, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(N, V, generator=g) * 3).to(dtype)


@pytest.mark.parametrize("S", [8, 9, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_support_of_up_to_64(S, dtype):
    N, T = 3, 0.8
    x = _rows(N, dtype, S)
    u = torch.rand(N, generator=torch.Generator().manual_seed(S))
    tok, ids, probs = dr.sample_with_sparse_probs(x.to(DEV), T, S, uniforms=u.to(DEV))
    order = x.float().sort(dim=-1, descending=True, stable=True)
    assert torch.equal(ids.cpu(), order.indices[:, :S])
    p = (order.values[:, :S].double() / T).softmax(-1)
    # up to 64 fp32 exponentials, their sum and a division: under 2^7 roundings of 2^-24
    assert torch.allclose(probs.cpu().double(), p, rtol=2.0 ** -17, atol=0)
    at = (ids.cpu() == tok.cpu()[:, None]).double()
    assert bool((at.sum(-1) == 1).all())
    hi = (p.cumsum(-1) * at).sum(-1)
    lo = hi - (p * at).sum(-1)
    assert bool(((u >= lo - 1e-5) & (u <= hi + 1e-5)).all())


@pytest.mark.parametrize("k", [5, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_top_k_filter_takes_its_floor_from_the_rounds(k, dtype, monkeypatch):
    N, T = 3, 0.8
    x = _rows(N, dtype, 100 + k)
    rounds = []
    topk = dr.topk_tokens
    monkeypatch.setattr(dr, "topk_tokens", lambda *a, **kw: rounds.append(a[1]) or topk(*a, **kw))
    u = torch.rand(N, generator=torch.Generator().manual_seed(k))
    tok, prob = dr.sample_with_prob(x.to(DEV), T, k, uniforms=u.to(DEV))
    dense = dr.sampling_probs(x.to(DEV), T, k)
    assert rounds == [k, k]
    z = x.double() / T
    floor = x.float().sort(dim=-1, descending=True).values[:, k - 1:k]
    p = z.masked_fill(x.float() < floor, -float("inf")).softmax(-1)
    # as above
    assert torch.allclose(dense.cpu().double(), p, rtol=2.0 ** -17, atol=0)
    assert torch.allclose(prob.cpu().double(), p.gather(-1, tok.cpu()[:, None])[:, 0], rtol=2.0 ** -17, atol=0)


def test_a_wider_top_k_or_a_nucleus_takes_the_general_filter():
    N, T = 2, 0.8
    x = _rows(N, torch.float32, 7)
    for k, p in ((65, 1.0), (64, 0.9), (0, 0.9)):
        probs = dr.sampling_probs(x.to(DEV), T, k, p).cpu()
        order = (x.double() / T).sort(dim=-1, descending=True).values
        if k:
            order = order[:, :k]
        q = order.softmax(-1)
        if p < 1.0:  # entries while the mass before them is at most p
            q = q * (q.cumsum(-1) - q <= p)
        # a cut within an fp32 sum's rounding of p may fall one entry off
        assert bool(((probs > 0).sum(-1) - (q > 0).sum(-1)).abs().max() <= 1)
        assert torch.allclose(probs.sum(-1), torch.ones(N), rtol=1e-4)


@pytest.mark.parametrize("k", [16, 31, 32, 64])  # 65 chunks: 1,040, 2,015, 2,080 and 4,160 candidates in the merge
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_top_k_on_both_sides_of_the_wide_merge(k, dtype):
    x = _rows(2, dtype, k)
    ids, vals = dr.topk_tokens(x.to(DEV), k, with_values=True)
    order = x.float().sort(dim=-1, descending=True, stable=True)
    assert torch.equal(ids.cpu(), order.indices[:, :k]) and torch.equal(vals.cpu(), order.values[:, :k])
