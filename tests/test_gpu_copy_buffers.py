"""d3d_copy_buffers: several small device copies in one launch (GPU)."""
from __future__ import annotations

import ctypes

import pytest
import torch

from d3d_amd import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _copy(src, dst):
    n = len(src)
    arr = ctypes.c_void_p * n
    return _lib.load().d3d_copy_buffers(n, arr(*(t.data_ptr() for t in src)), arr(*(t.data_ptr() for t in dst)),
                                        (ctypes.c_size_t * n)(*(t.numel() * t.element_size() for t in src)),
                                        _lib.stream_ptr(DEV))


@pytest.mark.parametrize("sizes", [(1,), (1, 255, 256, 257, 3), (70000, 0, 5), (17,) * 8])
def test_copies_every_word_and_nothing_else(sizes):
    src = [torch.randint(-2**31, 2**31 - 1, (s,), dtype=torch.int32, device=DEV) for s in sizes]
    room = [torch.full((s + 2,), 7, dtype=torch.int32, device=DEV) for s in sizes]
    assert _copy(src, [r[1:-1] for r in room]) == 0
    for s, r in zip(src, room):
        assert torch.equal(r[1:-1], s) and r[0].item() == 7 and r[-1].item() == 7


def test_refusals():
    a = torch.zeros(16, dtype=torch.uint8, device=DEV)
    assert _copy([a[:3]], [a[8:11]]) == -1       # not a multiple of 4 bytes
    assert _copy([a[1:5]], [a[8:12]]) == -5      # not 4-byte aligned
    assert _copy([a[:4]] * 9, [a[8:12]] * 9) == -1
    assert _lib.load().d3d_copy_buffers(1, None, None, None, _lib.stream_ptr(DEV)) == -4
