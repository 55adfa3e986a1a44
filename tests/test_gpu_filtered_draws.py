"""Draws under a top-k or nucleus filter against the float64 CDF of the kept entries (GPU)."""
from __future__ import annotations

import pytest
import torch

from d3d_amd import draft as dr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _row(V, at, z):
    x = torch.full((1, V), -500.0)
    x[0, at] = z
    return x


@pytest.mark.parametrize("V", [5000, 151936])
@pytest.mark.parametrize("depth", [20.0, 25.0, 30.0])
def test_small_weights_at_the_front_of_the_row(V, depth):
    """k - 1 entries of weight e^-depth before the maximum, drawn at the middle
    of their bars: every bar as wide as its weight, to half a bar over k of them."""
    k = 120
    at = torch.arange(k) * 7
    at[-1] = V - 3
    z = torch.full((k,), -depth)
    z[-1] = 0.0
    w = z.double().exp()
    mid = ((w.cumsum(0) - w / 2) / w.sum())[:-1]
    x = _row(V, at, z).repeat(k - 1, 1)
    tok, prob = (t.cpu() for t in dr.sample_with_prob(x.to(DEV), 1.0, k, uniforms=mid.float().to(DEV)))
    assert torch.equal(tok, at[:-1])
    assert torch.allclose(prob.double(), (w / w.sum())[:-1], rtol=1e-6)


@pytest.mark.parametrize("V", [5000, 151936])
@pytest.mark.parametrize("depth", [26.0, 40.0, 80.0])
def test_every_kept_entry_can_be_drawn(V, depth):
    """u = 0 draws the first kept entry that expf gives a weight."""
    x = _row(V, torch.tensor([4, 11, V - 3]), torch.tensor([-depth - 30.0, -depth, 0.0]))
    tok, prob = dr.sample_with_prob(x.to(DEV), 1.0, 3, uniforms=torch.zeros(1, device=DEV))
    first = 4 if depth + 30 < 103 else 11
    assert int(tok) == first
    want = x[0, first].double().exp()
    assert abs(float(prob) / float(want) - 1) < 1e-6


def _kept(z, k, p):
    """Kept entries [V] bool of fp32 scaled logits: top-k with ties, then the nucleus by value and id."""
    keep = torch.ones_like(z, dtype=torch.bool)
    if k:
        keep = z >= z.sort(descending=True).values[k - 1]
    if p < 1:
        order = z.sort(descending=True, stable=True).indices
        order = order[keep[order]]
        w = (z[order].double() - z[order[0]].double()).exp()
        n = int((w.cumsum(0) <= p * w.sum()).sum()) + 1
        keep = torch.zeros_like(keep)
        keep[order[:n]] = True
    return keep


@pytest.mark.parametrize("dtype,T", [(torch.bfloat16, 0.7), (torch.float32, 1.0)])
@pytest.mark.parametrize("V,k,p", [(151936, 0, 0.9), (151935, 0, 0.5), (4097, 0, 0.95), (151936, 50, 1.0),
                                   (151936, 64, 0.8), (32771, 2000, 1.0), (32771, 2000, 0.95), (9, 4, 0.6)])
def test_draws_lie_in_their_bars(V, k, p, dtype, T):
    """u over the whole range, dense at both ends: each draw's bar holds its u."""
    N = 48
    g = torch.Generator().manual_seed(V + k)
    x = torch.randn(1, V, generator=g) * 2.0
    x[0, torch.randint(0, V, (min(32, V),), generator=g)] += 6.0
    x = x.to(dtype)
    u = torch.cat([torch.zeros(1), 10.0 ** -torch.linspace(7, 1, 15), torch.linspace(0.02, 0.98, 24),
                   1 - 2.0 ** -torch.linspace(5, 24, 8).floor()])[:N].float()
    tok, prob = (t.cpu() for t in dr.sample_with_prob(x.repeat(N, 1).to(DEV), T, k, p, uniforms=u.to(DEV)))
    z = x[0].float() / torch.tensor(T)
    keep = _kept(z, k, p)
    w = torch.where(keep, (z.double() - z.double().max()).exp(), 0.0)
    q = w / w.sum()
    hi = q.cumsum(0)[tok]
    # exp of an fp32 z - max (|z - max| < 2^5: 2^-20 relative), the integer masses
    # (2^-40 each): 2^-19 of the bar's edge, and 2^-23 for all roundings near 1.
    slack = 2.0 ** -19 * torch.minimum(hi, 1 - hi + q[tok]) + 2.0 ** -23
    assert bool(keep[tok].all())
    assert bool((u.double() >= hi - q[tok] - slack).all()) and bool((u.double() <= hi + slack).all())
    assert torch.allclose(prob.double(), q[tok], rtol=2.0 ** -19)
