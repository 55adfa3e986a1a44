"""The embedding lookup fused with the first norm (GPU) against the two steps."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from d3d_amd import layers as ly

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("T,V,H", [(1, 5, 8), (16, 1000, 4096), (33, 997, 2048), (1088, 300, 256), (3, 7, 8192)])
def test_equals_lookup_then_norm(T, V, H):
    g = torch.Generator(device=DEV).manual_seed(T + H)
    table = torch.randn(V, H, generator=g, device=DEV).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(H, generator=g, device=DEV)).to(torch.bfloat16)
    ids = torch.randint(0, V, (T,), generator=g, device=DEV)
    ids[0], ids[-1] = V - 1, 0
    residual, out = ly.embed_rmsnorm(ids, table, w, 1e-6)
    want = F.embedding(ids, table)
    assert torch.equal(residual, want)
    assert torch.equal(out, ly.add_rmsnorm(None, want, w, 1e-6))
