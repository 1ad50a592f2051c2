"""The training layer's kernels (csrc/gated_bwd.hip, the ReLU form of the
saved RoPE backward) against float64, and the fused autograd functions.

Tolerance: bf16 operands are exact in float64; each result is rounded to bf16
once (2^-9 relative) from fp32 sums, and relu(s) once more inside dx, so 8e-3
covers two roundings of every element; the compared tensors differ by their
norm, where roundings average to about 3e-3.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import bdh_harness as H  # noqa: E402
import bdh_hip_ext as ext  # noqa: E402
import kernels  # noqa: E402

BF = torch.bfloat16
TOL = 8e-3


def _randn(*shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(BF)


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm().clamp_min(1e-300))


# tokens around the 128-row tile, N around the 128-column tile (a multiple of
# 8), one and several K stages of 32
@pytest.mark.parametrize("B,T,nh,N,K", [(1, 1, 1, 8, 32), (1, 127, 2, 128, 64), (3, 43, 4, 136, 96), (2, 150, 3, 1000, 256),
                                        (1, 257, 2, 264, 512)])
@pytest.mark.parametrize("padded", [False, True])
def test_gated_backward_matches_float64(B, T, nh, N, K, padded):
    y, wt = _randn(B, nh, T, K, seed=0), _randn(nh, N, K, seed=1, std=0.05)
    dec, dout = _randn(nh * N, K, seed=2, std=0.05), _randn(B, T, K, seed=3)
    x = torch.relu(_randn(B, T, nh, N, seed=4))
    s = torch.einsum("bhtk,hnk->bthn", y.double(), wt.double())
    g = torch.einsum("btk,hnk->bthn", dout.double(), dec.double().view(nh, N, K))
    dx, dz = None, None
    if padded:  # padded token rows and head-major rows
        x = H._padded_rows(B, T, nh, N, BF, "cuda").copy_(x)
        dx = H._padded_rows(B, T, nh, N, BF, "cuda")
        dz = torch.empty(nh, B, T, N + 8, dtype=BF, device="cuda")[..., :N].permute(1, 2, 0, 3)
    dx, dz = ext.gated_bwd(y, wt, x, dec, dout, dx=dx, dz=dz)
    sure = s.abs() > 1e-3  # (the sign of a sum near zero is its rounding's)
    assert _rel(dx, g * s.clamp_min(0)) <= TOL
    assert _rel(dz[sure], (g * x.double() * (s > 0))[sure]) <= TOL
    with pytest.raises(RuntimeError):
        ext.gated_bwd(y, wt, x, dec, dout, dx=dx, dz=dx)


@pytest.mark.parametrize("B,T,nh,N", [(1, 1, 1, 8), (2, 33, 3, 2056), (1, 5, 4, 4096)])
def test_relu_backward_add_is_exact(B, T, nh, N):
    a, b = _randn(B, nh, T, N, seed=0).permute(0, 2, 1, 3), _randn(B, T, nh, N, seed=1)
    x = torch.relu(_randn(B, T, nh, N, seed=2))
    x[0, 0, 0, 1] = float("nan")
    want = torch.where(x <= 0, torch.zeros_like(b), a + b)
    assert torch.equal(ext.relu_bwd_add(a, b, x), want)
    assert torch.equal(ext.relu_bwd_add(a, b, x, out=b), want)  # in place


@pytest.mark.parametrize("B,T,nh,N,D", [(2, 100, 2, 256, 64), (1, 300, 4, 512, 256), (2, 512, 1, 256, 128)])
def test_saved_backward_through_the_relu(B, T, nh, N, D):
    """The fused sum and mask equal the separate pass up to its extra rounding."""
    xt = H._padded_rows(B, T, nh, N, BF, "cuda").copy_(torch.relu(_randn(B, T, nh, N, seed=0, std=0.3)))
    x, v, do = xt.permute(0, 2, 1, 3), _randn(B, 1, T, D, seed=1), _randn(B, nh, T, D, seed=2)
    add = _randn(B, T, nh, N, seed=3, std=3.0)
    freqs = kernels.get_freqs(N).cuda()
    _, scores = ext.tril_rope_score_v_save(x, v, freqs, 2)
    assert scores is not None
    dx, dv = ext.tril_rope_score_v_bwd_saved(x, v, do, freqs, 2, scores)
    out = H._padded_rows(B, T, nh, N, BF, "cuda")
    got, dv2 = ext.tril_rope_score_v_bwd_saved(x, v, do, freqs, 2, scores, dx=out.permute(0, 2, 1, 3),
                                               relu_add=add.permute(0, 2, 1, 3))
    assert torch.equal(dv, dv2)
    want = ext.relu_bwd_add(dx.permute(0, 2, 1, 3), add, xt)
    assert not out[xt <= 0].any()
    # the separate pass rounds dx to bf16 before the sum: 2^-9 of dx, as the sum's own rounding
    assert _rel(out, want.double()) <= 4e-3


# the fused functions and, with n_embd = 48 (not a multiple of 32), the plain graph
@pytest.mark.parametrize("D,nh,mult,B,T", [(64, 2, 8, 2, 33), (128, 4, 16, 3, 130), (48, 2, 16, 2, 40)])
@pytest.mark.parametrize("frozen", [(), ("encoder",), ("encoder_v", "decoder")])
def test_training_step_gradients_follow_eager_attention(D, nh, mult, B, T, frozen, monkeypatch):
    """Against the same step on the plain autograd graph (the layer's masks see
    the same bits): gradients within bf16 rounding of each other."""
    torch.manual_seed(0)
    m = H.BDH(H.BDHConfig(n_layer=2, n_embd=D, n_head=nh, mlp_internal_dim_multiplier=mult)).cuda()
    for n in frozen:
        getattr(m, n).requires_grad_(False)
    idx = torch.randint(0, 256, (B, T), device="cuda")

    def grads():
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=BF):
            loss = m(idx, idx.roll(-1, 1), impl="hip")[1]
        loss.backward()
        return loss.detach(), {n: p.grad for n, p in m.named_parameters() if p.requires_grad}

    loss, got = grads()
    monkeypatch.setattr(H, "_trains_fused", lambda *a: False)
    want_loss, want = grads()
    assert abs(float(loss - want_loss)) <= 1e-4 * float(want_loss)
    assert set(got) == set(want)
    for n, g in want.items():
        assert got[n].shape == g.shape and got[n].dtype == g.dtype
        assert _rel(got[n], g.double()) <= 3e-2, n


# rows in one and several 32-row stages and splits; output rows below, at and
# over a 256-row tile; row pitches wider than the row
@pytest.mark.parametrize("nh,K,M,N,splits", [(1, 32, 8, 256, 1), (2, 192, 264, 512, 3), (4, 2048, 256, 1024, 2),
                                             (1, 4096, 64, 256, 8)])
def test_row_contraction_matches_float64(nh, K, M, N, splits):
    """fp32 sums of exact bf16 products: K roundings of 2^-24, in norm below 1e-5."""
    a, b = _randn(nh, K, M + 8, seed=0)[..., :M], _randn(nh, K, N + 128, seed=1)[..., :N]
    got = ext.tn_gemm(a, b, splits)
    want = torch.stack([a[h].double().t() @ b[h].double() for h in range(nh)])
    assert got.dtype == torch.float32 and _rel(got, want) <= 1e-5
    with pytest.raises(RuntimeError):
        ext.tn_gemm(a, b, splits + 4)  # K is not a multiple of 32 (splits + 4)


def _tiny():
    torch.manual_seed(0)
    return H.BDHConfig(n_layer=2, n_embd=64, n_head=2, mlp_internal_dim_multiplier=8)


def _train(m, idx):
    with torch.autocast("cuda", dtype=BF):
        loss = m(idx, idx.roll(-1, 1), impl="hip")[1]
    loss.backward()
    return {n: p.grad.clone() for n, p in m.named_parameters()}


def test_a_replaced_operator_or_attention_is_run(monkeypatch):
    """The fused training layer and the native generate step stand in for the class's own
    attention over the surface's own operators, and for nothing else."""
    calls = []

    class Own(H.BDH):
        def _attention(self, *a):
            calls.append("attention")
            return 0.5 * super()._attention(*a)

    cfg = _tiny()
    m = H.BDH(cfg).cuda()
    own = Own(cfg).cuda()
    own.load_state_dict(m.state_dict())
    idx = torch.randint(0, 256, (2, 33), device="cuda")
    plain = _train(m, idx)
    _train(own, idx)
    assert calls == ["attention"] * cfg.n_layer
    # a generate step after the prompt
    del calls[:]
    own.generate(idx, 1, cache_dtype=BF, amp_dtype=BF, impl="hip")
    assert calls == ["attention"] * (2 * cfg.n_layer)

    rope = kernels.bdh_attn_rope

    def fp32(x, v, freqs, rope_start=0, out_kr=None, impl=None):
        calls.append("rope")
        return rope(x.float(), v.float(), freqs, rope_start, impl=impl).to(x.dtype)

    del calls[:]
    monkeypatch.setattr(kernels, "bdh_attn_rope", fp32)
    m.zero_grad(set_to_none=True)
    assert any(not torch.equal(g, plain[n]) for n, g in _train(m, idx).items())
    assert calls == ["rope"] * cfg.n_layer

    monkeypatch.undo()
    decode = kernels.bdh_attn_decode
    monkeypatch.setattr(kernels, "bdh_attn_decode", lambda *a, **k: calls.append("decode") or decode(*a, **k))
    del calls[:]
    m.generate(idx, 1, cache_dtype=BF, amp_dtype=BF, impl="hip")
    assert calls == ["decode"] * cfg.n_layer


@pytest.mark.parametrize("splits", [1, 2, 4])
def test_row_contraction_holds_only_its_own_storage(splits):
    """A weight gradient becomes a parameter's .grad: no split's partial sums may live on in it."""
    a, b = _randn(2, 512, 64, seed=0), _randn(2, 512, 256, seed=1)
    got = ext.tn_gemm(a, b, splits)
    assert got.is_contiguous() and got.untyped_storage().nbytes() == got.numel() * 4


# weight gradients on the row-contracting kernel (at least 1024 tokens a split), from kept tiles;
# no kept tiles: n_embd over 256, N not a multiple of 256, or switched off
@pytest.mark.parametrize("D,nh,mult,B,T,keep,kernel", [
    (256, 2, 2, 16, 512, "1", "k_dq_sy_tn"), (256, 1, 3, 8, 1056, "1", "k_dq_sy_tn"),
    (512, 2, 2, 2, 150, "1", "k_relu_bwd_add"), (96, 2, 4, 3, 130, "1", "k_relu_bwd_add"),
    (64, 2, 8, 2, 33, "0", "k_relu_bwd_add"), (512, 1, 1, 4, 2048, "1", "k_dq_sy_tn")])
def test_training_step_takes_each_route(D, nh, mult, B, T, keep, kernel, monkeypatch):
    """Gradients of the routes that a small kept-tiles step does not reach, against the plain
    autograd graph, from which single bf16 roundings (2^-9) of the latent's gradients set them
    apart: 3e-3 to 5e-3 measured, 1.2e-2 allowed."""
    torch.manual_seed(0)
    monkeypatch.setenv("BDH_ATTN_SAVE_SCORES", keep)
    m = H.BDH(H.BDHConfig(n_layer=2, n_embd=D, n_head=nh, mlp_internal_dim_multiplier=mult)).cuda()
    idx = torch.randint(0, 256, (B, T), device="cuda")
    ext.profile_enable(True)
    try:
        got = _train(m, idx)
        torch.cuda.synchronize()
        names = {n for n, _ in ext.profile_collect()}
    finally:
        ext.profile_enable(False)
    assert kernel in names and "k_gated_bwd" in names, names
    m.zero_grad(set_to_none=True)
    monkeypatch.setattr(H, "_trains_fused", lambda *a: False)
    want = _train(m, idx)
    assert set(got) == set(want)
    for n, g in want.items():
        e = _rel(got[n], g.double())
        print(f"  {n}: {e:.3e}", flush=True)
        assert got[n].dtype == g.dtype and e <= 1.2e-2, n
