"""Prefill of many tokens (64-token slices) against the same prompts one by one (16-token slices)."""
from __future__ import annotations

import pytest
import torch

from d3d_amd.model import ModelShape, PagedKV, Qwen3PagedModel, Sequence, prefill

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TINY = ModelShape(layers=2, hidden=256, heads=8, kv_heads=2, head_dim=128, mlp=512, vocab=1000)


@pytest.mark.parametrize("lens", [(2049, 1, 64, 65, 1920), (63, 4033)])
def test_wide_slices_equal_narrow_ones(lens):
    assert sum(lens) >= 4096
    model = Qwen3PagedModel(TINY, DEV, draft=False, seed=3, init_std=0.05)
    g = torch.Generator().manual_seed(sum(lens))
    prompts = [torch.randint(0, 1000, (n,), generator=g).tolist() for n in lens]

    def caches(groups):
        kv = PagedKV(TINY, 400, 16, DEV)
        out, kvs = [], []
        for group in groups:
            seqs = [Sequence(i, p) for i, p in enumerate(group)]
            out.append(prefill(model, kv, seqs, "t"))
            for s, p in zip(seqs, group):
                at = torch.tensor(s.pages["t"], device=DEV)
                kvs.append(torch.stack([kv.k[-1][at], kv.v[-1][at]]).flatten(1, 2)[:, :len(p)].clone())
        return torch.cat(out), kvs

    with torch.inference_mode():
        h, kv = caches([prompts])
        h1, kv1 = caches([[p] for p in prompts])
    # The library rounds its products of other row counts in another order:
    # bf16 steps (2^-8) of two layers' sums.
    assert (h.float() - h1.float()).norm() <= 0.02 * h1.float().norm()
    for a, b in zip(kv, kv1):
        assert a.shape == b.shape and (a.float() - b.float()).norm() <= 0.02 * b.float().norm()


@pytest.mark.parametrize("lens,block", [((14,) * 300, 16), ((2049, 2100), 32)])
def test_rows_that_go_through_the_model(lens, block, monkeypatch):
    """Many short prompts keep the default slices, a caller's own block stays as it is."""
    model = Qwen3PagedModel(TINY, DEV, draft=False, seed=3, init_std=0.05)
    shapes = []
    forward = model.forward
    monkeypatch.setattr(model, "forward", lambda ids, *a, **kw: shapes.append(tuple(ids.shape)) or forward(ids, *a, **kw))
    kv = PagedKV(TINY, 400, 16, DEV)
    with torch.inference_mode():
        prefill(model, kv, [Sequence(i, [1] * n) for i, n in enumerate(lens)], "t", block=block)
    assert shapes == [(sum(-(-n // block) for n in lens), block)]
