"""The few-row products of a generate step (csrc/few.hip) against float64.

Tolerance: exact bf16 products summed in fp32 and rounded to bf16 once or twice
(2^-9 each): 8e-3; fp32 outputs 1e-5.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import bdh_hip_ext as ext  # noqa: E402

BF = torch.bfloat16


def _randn(*shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(BF)


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm().clamp_min(1e-300))


# tokens 1 .. 32 (33 takes the tile kernel), N below, at and across a wave's 32
# and a workgroup's 128 columns, every K
@pytest.mark.parametrize("B,T", [(1, 1), (8, 1), (3, 7), (32, 1), (11, 3)])
@pytest.mark.parametrize("nh,N,K", [(1, 8, 64), (2, 40, 128), (4, 136, 256), (3, 1024, 512)])
def test_relu_and_gated_products(B, T, nh, N, K):
    y, wt = _randn(B, nh, T, K, seed=0), _randn(nh, N, K, seed=1, std=0.1)
    x = torch.relu(_randn(B, T, nh, N + 8, seed=2))[..., :N]
    s = torch.stack([y[:, h].double() @ wt[h].double().t() for h in range(nh)], 2).clamp_min(0)
    assert _rel(ext.relu_gemm(y, wt), s) <= 8e-3
    shared = y[:, :1].expand(B, nh, T, K)  # the heads share one row set
    s0 = torch.stack([y[:, 0].double() @ wt[h].double().t() for h in range(nh)], 2).clamp_min(0)
    assert _rel(ext.relu_gemm(shared, wt), s0) <= 8e-3
    got = ext.gated_gemm(y, wt, x, torch.empty(B, T, nh, N + 8, dtype=BF, device="cuda")[..., :N])
    assert _rel(got, s * x.double()) <= 8e-3


@pytest.mark.parametrize("M", [1, 8, 31, 33, 64, 65])
@pytest.mark.parametrize("K", [128, 640, 32768])
@pytest.mark.parametrize("odt", [torch.float32, BF])
def test_split_decoder_product(M, K, odt):
    a, b = _randn(M, K + 8, seed=0)[:, :K], _randn(K, 256, seed=1)
    got = ext.small_gemm(a, b, odt)
    assert torch.equal(got, ext.small_gemm(a, b, odt))
    assert _rel(got, a.double() @ b.double()) <= (1e-5 if odt == torch.float32 else 4e-3)
