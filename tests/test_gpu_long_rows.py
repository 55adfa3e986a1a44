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
