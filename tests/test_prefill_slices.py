"""Prefill's slice width: padding decides, not the batch's token total."""
from __future__ import annotations

import pytest

from d3d_amd.model import _slice_tokens


@pytest.mark.parametrize("lens,width", [
    ([2000] * 4, 64), ([4096], 64), ([4095], 16), ([1024] * 4, 64), ([700] * 6, 64), ([2049, 1, 64, 65, 1920], 64),
    ([17] * 256, 16), ([14] * 300, 16), ([8] * 512, 16), ([100] * 41, 16), ([300] * 14, 16), ([1] * 5000, 16),
    ([64] * 64, 64), ([4000] + [1] * 100, 16)])
def test_slices_widen_only_where_padding_stays_small(lens, width):
    assert _slice_tokens(lens, 16) == width


@pytest.mark.parametrize("block", [1, 8, 32, 64])
def test_a_callers_own_block_is_kept(block):
    assert _slice_tokens([2000] * 4, block) == block
