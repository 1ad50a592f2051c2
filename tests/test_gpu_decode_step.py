"""The native generate step (bdh_decode_step) against the layer-by-layer path
it replaces: same kernels, except the encoder's product (bit-identical to the
library's), so the same cache rows and logits.

Tolerance: two bf16 roundings of a layer's output, 2^-8, through the layers.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import bdh_harness as H  # noqa: E402

BF = torch.bfloat16


@pytest.mark.parametrize("L,D,nh,mult,B,S", [(1, 64, 2, 4, 1, 1), (2, 128, 4, 5, 3, 7), (3, 256, 4, 32, 65, 70),
                                             (2, 512, 8, 16, 2, 300), (2, 64, 2, 24, 256, 33),
                                             (3, 256, 4, 32, 9, 40), (2, 256, 4, 32, 40, 5), (2, 1024, 4, 5, 2, 9)])
def test_native_step_equals_layer_by_layer(L, D, nh, mult, B, S, monkeypatch):
    torch.manual_seed(0)
    m = H.BDH(H.BDHConfig(n_layer=L, n_embd=D, n_head=nh, mlp_internal_dim_multiplier=mult)).cuda()
    idx = torch.randint(0, 256, (B, S + 2), device="cuda")

    def run(native):
        monkeypatch.setattr(H, "_steps_native", H_native if native else (lambda *a: False))
        cache = H.KVCache(m.config, B, S + 2, BF, "cuda")
        cache.kr.zero_()
        cache.v.zero_()
        with torch.no_grad(), torch.autocast("cuda", dtype=BF):
            m(idx[:, :S], cache=cache, impl="hip", last_only=True)
            logits = [m(idx[:, s:s + 1], cache=cache, impl="hip")[0] for s in (S, S + 1)]
        with pytest.raises(ValueError), torch.no_grad():
            m(idx[:, :1], cache=cache, impl="hip")  # the cache is full
        return torch.stack(logits), cache

    H_native = H._steps_native
    got, c = run(True)
    want, w = run(False)
    for a, b in ((got, want), (c.kr, w.kr), (c.v, w.v)):
        assert float((a.double() - b.double()).norm() / b.double().norm()) <= 2.0 ** -8
    assert c.seq_len == S + 2
