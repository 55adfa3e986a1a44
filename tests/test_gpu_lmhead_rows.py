"""The row-streaming LM head (H of 2048 and 4096) and the LM head's logits (GPU).

Ids and log-probabilities against the logits of the plain product by the same
kernels' rounding: the fp64 product bounds each bf16 logit, and a row's top-k
is compared where its logits decide it (no other logit within two bf16 steps
of the k-th).
"""
from __future__ import annotations

import pytest
import torch

from d3d_amd import layers as ly
from d3d_amd.lmhead import lmhead_topk

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
BF = torch.bfloat16


def _operands(T, V, H, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(T, H, generator=g, device=DEV).to(BF),
            (torch.randn(V, H, generator=g, device=DEV) * 0.02).to(BF))


@pytest.mark.parametrize("H", [2048, 4096])
@pytest.mark.parametrize("T,V,k", [(1, 129, 1), (16, 5000, 2), (17, 4999, 3), (64, 128, 8), (65, 3001, 5), (128, 40000, 2),
                                   (129, 2000, 4), (200, 1000, 8)])
def test_topk_of_the_row_streaming_head(T, V, k, H):
    h, w = _operands(T, V, H, T + V + H)
    ids, vals = lmhead_topk(h, w, k, with_values=True, log_softmax=True)
    x = (h.double() @ w.double().T)
    ref, order = x.topk(min(k + 1, V), -1)
    step = x.abs().amax() * 2.0 ** -7  # two bf16 steps of the largest logit
    lp = x.log_softmax(-1)
    # a bf16 logit is half a step off its product, the log-sum another fraction
    assert bool(((vals.double() - lp.topk(k, -1).values).abs() <= step).all())
    gaps = (ref[:, :-1] - ref[:, 1:]).amin(-1) if ref.shape[1] > 1 else ref.new_full((T,), 1.0)
    sure = gaps > step
    assert torch.equal(ids[sure], order[sure, :k])
    assert bool((x.gather(-1, ids) >= ref[:, k - 1:k] - step).all())


@pytest.mark.parametrize("M,K", [(1, 2048), (16, 4096), (17, 2048), (32, 4096), (33, 2048), (64, 2048), (64, 4096)])
def test_lm_head_logits(M, K, monkeypatch):
    V = 131072 + 128
    x, w = _operands(M, V, K, M + K)
    library = []
    linear = ly.F.linear
    monkeypatch.setattr(ly.F, "linear", lambda *a: library.append(1) or linear(*a))
    y = ly.lm_head(x.view(1, M, K), w)
    assert y.shape == (1, M, V) and bool(library) == ((M, K) == (64, 4096))
    for at in range(0, V, 16384):
        ww = w[at:at + 16384].double()
        ref = x.double() @ ww.T
        slack = (x.double().abs() @ ww.abs().T) * (2.0 * K * 2.0 ** -24)
        ulp = torch.clamp(ref.abs(), min=2.0 ** -100).log2().floor().exp2() * 2.0 ** -7
        assert bool(((y[0, :, at:at + 16384].double() - ref).abs() <= ulp + slack).all())
