"""Decode with the past cut into 4- to 64-key chunks (csrc/decode.hip
dec_chunk), every kernel and its half-row form, against float64.

Tolerance: fp32 arithmetic over N products and S keys, 1e-5; bf16 outputs round
once more (2^-9 relative), 4e-3.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import bdh_hip_ext as ext  # noqa: E402


# rows (B * H) and S around the chunk sizes; N: the streaming kernels with and
# without the half-row form (8192 / 2048 / 512), and the generic kernel (200)
@pytest.mark.parametrize("qdt,kdt", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                     (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("N", [8192, 2048, 512, 200])
@pytest.mark.parametrize("B,H,S", [(1, 1, 1), (1, 4, 3), (1, 4, 5), (2, 4, 63), (1, 4, 301), (16, 8, 65), (32, 8, 190)])
def test_chunked_past_matches_float64(B, H, S, N, qdt, kdt):
    g = torch.Generator(device="cuda").manual_seed(S * N)
    k = torch.randn(B, H, S + 3, N, generator=g, device="cuda").to(kdt)
    v = torch.randn(B, 1, S + 3, 40, generator=g, device="cuda").to(kdt)
    q = torch.randn(B, H, 1, N, generator=g, device="cuda").to(qdt)
    ks, vs = k.narrow(2, 0, S), v.narrow(2, 0, S)
    got = ext.tril_decode(q, ks, vs)
    want = torch.stack([(q[b].double() @ ks[b].double().transpose(-2, -1).contiguous()) @ vs[b, 0].double()
                        for b in range(B)])
    err = float((got.double() - want).norm() / want.norm())
    assert err <= (1e-5 if qdt == torch.float32 else 4e-3), err
    assert torch.equal(got, ext.tril_decode_noalloc(q, ks, vs))
