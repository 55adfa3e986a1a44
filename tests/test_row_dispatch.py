"""Which blocks take the row-tiled products (no device needed)."""
from __future__ import annotations

import pytest
import torch

from d3d_amd import layers as ly


@pytest.mark.parametrize("M,H,K,fused", [
    (64, 6144, 2048, True), (65, 6144, 2048, True), (192, 6144, 2048, True), (193, 6144, 2048, False),
    (16, 12288, 4096, True), (64, 12288, 4096, True), (65, 12288, 4096, True), (128, 12288, 4096, True),
    (129, 12288, 4096, False), (192, 12288, 4096, False),   # more than a round of tiles
    (64, 4096, 8192, True), (65, 4096, 8192, False), (192, 4096, 8192, False),  # tiles for half of the CUs
    (64, 14336, 4096, True), (65, 14336, 4096, False), (64, 6144, 2560, False)])
def test_gate_up_route(M, H, K, fused):
    assert ly.rows_silu_ok(M, H, K) == fused


def test_project_refuses_operands_that_disagree():
    """Also at sizes the HIP kernel would take, which reads K entries of every weight row."""
    x = torch.zeros(4, 4096, dtype=torch.bfloat16)
    w = torch.zeros(4096, 2048, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="shapes cannot be multiplied"):
        ly.project(x, w)
