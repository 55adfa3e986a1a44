"""Many short rows, on both sides of every limit of the top-k kernels' rounds (GPU)."""
from __future__ import annotations

import pytest
import torch

from d3d_amd import draft as dr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("N", [256, 257])
@pytest.mark.parametrize("V", [100, 4096, 4097, 8192, 8193])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k", [5, 10, 11, 14, 15, 18, 19, 32, 33])
def test_top_k_support_and_draw(N, V, dtype, k):
    T = 0.8
    g = torch.Generator().manual_seed(V + k)
    x = (torch.randn(N, V, generator=g) * 2).to(dtype)
    u = torch.rand(N, generator=g)
    xd, ud = x.to(DEV), u.to(DEV)
    order = x.float().sort(dim=-1, descending=True, stable=True)
    ids, vals = dr.topk_tokens(xd, k, with_values=True)
    assert torch.equal(ids.cpu(), order.indices[:, :k]) and torch.equal(vals.cpu(), order.values[:, :k])
    tok, sid, probs = (t.cpu() for t in dr.sample_with_sparse_probs(xd, T, k, uniforms=ud))
    q = (order.values[:, :k].double() / T).softmax(-1)
    # fp32 quotients, exponentials and sums of at most 33: under 2^6 roundings of 2^-24
    assert torch.allclose(probs.double(), q, rtol=2.0 ** -18, atol=0)
    z = x.float() / torch.tensor(T)
    if dtype == torch.bfloat16:  # distinct fp32 logits may share a quotient, whose order is then by id
        assert torch.equal(sid, order.indices[:, :k])
    assert torch.equal(z.gather(1, sid), z.gather(1, order.indices[:, :k]))
    _in_bar(q.cumsum(-1), q, (sid == tok[:, None]).double().argmax(-1), u)
    tok, prob = (t.cpu() for t in dr.sample_with_prob(xd, T, k, uniforms=ud))
    p = z.double().masked_fill(x.float() < order.values[:, k - 1:k], -float("inf")).softmax(-1)
    _in_bar(p.cumsum(-1), p, tok, u)
    assert torch.allclose(prob.double(), p.gather(-1, tok[:, None])[:, 0], rtol=2.0 ** -18)
    assert torch.allclose(dr.sampling_probs(xd, T, k).cpu().double(), p, rtol=2.0 ** -18, atol=0)


def _in_bar(cdf, p, at, u):
    hi = cdf.gather(-1, at[:, None])[:, 0]
    lo = hi - p.gather(-1, at[:, None])[:, 0]
    assert bool(((u >= lo - 1e-5) & (u <= hi + 1e-5)).all())
