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


# a workspace of the 32-key partials alone (sized for a longer past, say): larger chunks, nothing past its end
@pytest.mark.parametrize("S", [5, 301, 1024])
@pytest.mark.parametrize("N,dt", [(8192, torch.bfloat16), (512, torch.float32), (200, torch.float32)])
def test_smallest_workspace(S, N, dt):
    H, Dv = 4, 64
    g = torch.Generator(device="cuda").manual_seed(S)
    k = torch.randn(1, H, S, N, generator=g, device="cuda").to(dt)
    v = torch.randn(1, 1, S, Dv, generator=g, device="cuda").to(dt)
    q = torch.randn(1, H, 1, N, generator=g, device="cuda").to(dt)
    n = (S + 31) // 32 * H * Dv
    ws = torch.full((n + 64,), 7.0, device="cuda")
    out = torch.empty(1, H, 1, Dv, dtype=dt, device="cuda")

    def call(nbytes):
        return ext._lib.bdh_tril_decode(ext._t4(q), ext._t4(k), ext._t4(v), ext._t4(out), ws.data_ptr(), nbytes,
                                        ext._stream(out.device))

    assert call(4 * n) == 0
    want = (q[0].double() @ k[0].double().transpose(-2, -1).contiguous()) @ v[0].double()
    assert float((out[0].double() - want).norm() / want.norm()) <= (1e-5 if dt == torch.float32 else 4e-3)
    assert bool((ws[n:] == 7.0).all())
    assert call(4 * n - 4) != 0
