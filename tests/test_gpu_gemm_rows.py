"""The weight-streaming GEMM at every row tile (16, 32, 64, 128, 192) and its remainders (GPU).

d3d_gemm_rows192 through layers.project against the fp64 product of the same
bf16 operands.  Bound per entry: one bf16 step of the exact value plus
2 K 2^-24 sum_k |x_k w_k|, twice the classical error bound of an fp32 sum of K
products in any order.  The fused gate-up equals the plain product followed by
silu_mul bit for bit.
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from d3d_amd import _lib
from d3d_amd import layers as ly

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
BF = torch.bfloat16


def _operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=DEV).to(BF)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(BF)
    return x, w


def _check(y, x, w):
    K = x.shape[1]
    ref = x.double() @ w.double().T
    slack = (x.double().abs() @ w.double().abs().T) * (2.0 * K * 2.0 ** -24)
    ulp = torch.clamp(ref.abs(), min=2.0 ** -100).log2().floor().exp2() * 2.0 ** -7
    assert bool(((y.double() - ref).abs() <= ulp + slack).all())


@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 12288), (4096, 2048), (2048, 2048), (2048, 6144)])
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 80, 128, 129, 191, 192])
def test_project_at_every_row_tile(N, K, M):
    x, w = _operands(M, N, K, M + N + K)
    got = ly.project(x, w, ly.ROWS192)
    assert isinstance(got, ly.SplitProduct)  # the HIP kernel, not the library
    _check(got.value(), x, w)


@pytest.mark.parametrize("M", [16, 32, 64, 100, 192])
@pytest.mark.parametrize("K,splits", [(256, 1), (512, 1), (768, 1), (1024, 1), (1536, 1), (2048, 2), (6144, 2), (4096, 1)])
def test_every_step_count(M, K, splits):
    lib = _lib.load()
    N = 192
    x, w = _operands(M, N, K, K + M)
    y = torch.empty(M, N, dtype=BF, device=DEV)
    parts = torch.empty(splits, M, N, device=DEV)
    st = lib.d3d_gemm_rows192(x.data_ptr(), w.data_ptr(), y.data_ptr(), parts.data_ptr(), M, N, K, splits,
                              _lib.stream_ptr(DEV))
    assert st == 0
    _check(y if splits == 1 else ly.SplitProduct(parts, splits).value(), x, w)


@pytest.mark.parametrize("H,K", [(6144, 2048), (12288, 4096), (256, 1024), (8224, 1024), (12000, 1024)])
@pytest.mark.parametrize("M", [16, 20, 64, 65, 128, 129, 192])
def test_fused_gate_up_equals_the_two_kernels(H, K, M):
    lib = _lib.load()
    x, w = _operands(M, 2 * H, K, H + M)
    gu = torch.empty(M, 2 * H, dtype=BF, device=DEV)
    st = _lib.stream_ptr(DEV)
    assert lib.d3d_gemm_rows192(x.data_ptr(), w.data_ptr(), gu.data_ptr(), None, M, 2 * H, K, 1, st) == 0
    want = ly.silu_mul(gu)
    got = torch.zeros(M, H, dtype=BF, device=DEV)
    assert lib.d3d_gemm_rows192_silu_mul(x.data_ptr(), w.data_ptr(), got.data_ptr(), M, H, K, st) == 0
    assert torch.equal(got, want)
    if ly.rows_silu_ok(M, H, K):
        assert torch.equal(ly.gate_up_silu(x, w), want)


def test_larger_blocks_and_other_step_counts_take_the_library():
    x, w = _operands(193, 4096, 4096, 1)
    assert torch.equal(ly.project(x, w, ly.ROWS192), F.linear(x, w))
    lib = _lib.load()
    args = (x.data_ptr(), w.data_ptr(), x.data_ptr(), None)
    st = _lib.stream_ptr(DEV)
    assert lib.d3d_gemm_rows192(*args, 193, 4096, 4096, 1, st) == -1
    assert lib.d3d_gemm_rows192(*args, 65, 64, 640, 1, st) == -5  # five steps, refused before a launch
