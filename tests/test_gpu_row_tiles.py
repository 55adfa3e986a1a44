"""Row reads at the edges of a vector, a tile and a row (GPU).

Row lengths around 16 bytes, the 4096-entry chunk and odd ones (rows at every
element alignment), against torch in float64.  Every entry of a row counts
towards its softmax sum, so a value read twice, missed or taken from the next
row moves the confidence; the softmax draw's probability bounds it again.
"""
from __future__ import annotations

import pytest
import torch

from d3d_amd import draft as dr

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("V", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 2047, 2049, 4095, 4096, 4097, 4103, 6151, 12289])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1.0, 0.7])
def test_row_sums_at_every_length(V, dtype, T):
    B, Q = 2, 9
    g = torch.Generator().manual_seed(V)
    x = (torch.rand(B, Q, V, generator=g) * 2).to(dtype)  # every entry weighs about the same
    xd = x.to(DEV)
    block = torch.full((B, Q), V, dtype=torch.int64, device=DEV)
    x0, conf = dr.confidence_topk_unmask(xd, block, V, 1, T)
    tok, prob = dr.sample_with_prob(xd, T, uniforms=torch.rand(B, Q, generator=g).to(DEV))
    torch.cuda.synchronize()
    p = (x.double() / T).softmax(-1)
    assert torch.equal(x0.cpu(), x.float().argmax(-1))
    # 16 entries per thread, 8 steps per workgroup and up to 4 chunks in fp32:
    # under 2^6 roundings of 2^-24, and as many of z = x / T before exp
    assert torch.allclose(conf.cpu().double(), p.amax(-1), rtol=8e-6)
    assert torch.allclose(prob.cpu().double(), p.gather(-1, tok.cpu()[..., None])[..., 0], rtol=8e-6)
