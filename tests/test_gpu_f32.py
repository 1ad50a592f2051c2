"""fp32 attention on the bf16 matrix cores (csrc/f32.hip) at the edges of its
tiles, against the same formula in float64.

The tolerance: operands are represented exactly by three bf16 planes and the
dropped plane products are at most 2^-24 of a product, a rounding, so what
remains is fp32 accumulation, at most about sqrt(K) 2^-24 of a sum for K updates
(3e-6 at the widths here); 5e-6 leaves the rest of a forward or backward its own
rounding.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import bdh_hip_ext as ext  # noqa: E402
import kernels  # noqa: E402

TOL = 5e-6


def _randn(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def _latent(*shape, seed):
    return torch.relu(0.32 * _randn(*shape, seed=seed))


def _rel(got, want):
    got, want = got.double().cpu(), want.double()
    return float((got - want).norm() / want.norm().clamp_min(1e-300))


def _rope64(x, freqs, start):
    T = x.size(-2)
    pos = torch.arange(start, start + T, dtype=torch.float32)
    ph = ((pos[:, None] * freqs.reshape(1, -1)) % 1).double() * (2 * torch.pi)
    c, s = torch.cos(ph)[:, 0::2], torch.sin(ph)[:, 0::2]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * c - x1 * s, x1 * c + x0 * s), dim=-1).flatten(-2)


def _attn64(q, k, v):
    return (q @ k.transpose(-2, -1)).tril(-1) @ v


# T: one 128-row tile, one and two 256-row tiles and an odd third, each at its
# edges; N: below and across a stage of 16, unaligned rows, several splits;
# D: one and two column tiles, odd
SHAPES = [(1, 16, 2, 1), (2, 17, 30, 5), (1, 127, 16, 64), (1, 128, 34, 128), (1, 129, 66, 130), (2, 200, 1024, 32),
          (1, 256, 48, 65), (1, 257, 514, 96), (1, 385, 1040, 129), (1, 513, 80, 40), (1, 700, 256, 256)]


@pytest.mark.parametrize("T,N,D", [s[1:] for s in SHAPES])
@pytest.mark.parametrize("rope", [False, True])
def test_forward_and_backward_at_tile_edges(T, N, D, rope):
    B, H, start = 2, 3, 5
    x = _latent(B, H, T, N, seed=0)
    v, do = _randn(B, 1, T, D, seed=1), _randn(B, H, T, D, seed=2)
    freqs = kernels.get_freqs(N)
    x64, v64 = x.double().requires_grad_(True), v.double().requires_grad_(True)
    r64 = _rope64(x64, freqs, start) if rope else x64
    want = _attn64(r64, r64, v64)
    gx, gv = torch.autograd.grad(want, (x64, v64), do.double())
    xd, vd, dd, fd = x.cuda(), v.cuda(), do.cuda(), freqs.cuda()
    if rope:
        qr = torch.empty_like(xd)
        got = ext.tril_rope_score_v(xd, vd, fd, start, qr_out=qr)
        assert torch.equal(got, ext.tril_rope_score_v(xd, vd, fd, start))  # the copy changes nothing
        assert _rel(qr, r64.detach()) <= TOL
        dx, dv = ext.tril_rope_score_v_bwd(xd, vd, dd, fd, start)
        out, scores = ext.tril_rope_score_v_save(xd, vd, fd, start)
        assert torch.equal(out, got)
        for a, b in zip(ext.tril_rope_score_v_bwd_saved(xd, vd, dd, fd, start, scores), (dx, dv)):
            assert torch.equal(a, b)  # the kept tiles are those the backward would make
    else:
        got = ext.tril_score_v(xd, xd, vd)
        dx, _, dv = ext.tril_score_v_bwd(xd, None, vd, dd)
    assert _rel(got, want.detach()) <= TOL and not got[:, :, 0].any()
    assert _rel(dx, gx) <= TOL and _rel(dv, gv) <= TOL


@pytest.mark.parametrize("T,N,D", [(100, 40, 7), (300, 96, 64), (520, 130, 130)])
def test_distinct_keys_per_head_values_and_offsets(T, N, D):
    """q is not k, V per head, and queries at an offset (past on and off tile edges)."""
    B, H = 1, 3
    q, k = _latent(B, H, T, N, seed=3), _latent(B, H, T, N, seed=4)
    v, do = _randn(B, H, T, D, seed=5), _randn(B, H, T, D, seed=6)
    q64, k64, v64 = (t.double().requires_grad_(True) for t in (q, k, v))
    want = _attn64(q64, k64, v64)
    grads = torch.autograd.grad(want, (q64, k64, v64), do.double())
    got = ext.tril_score_v(q.cuda(), k.cuda(), v.cuda())
    assert _rel(got, want.detach()) <= TOL
    for g, w in zip(ext.tril_score_v_bwd(q.cuda(), k.cuda(), v.cuda(), do.cuda()), grads):
        assert _rel(g, w) <= TOL
    full = _attn64(k.double(), k.double(), v.double())
    for past in (1, T // 2, T - 1):
        kd = k.cuda()
        assert _rel(ext.tril_score_v_past(kd[:, :, past:], kd, v.cuda(), past), full[:, :, past:]) <= TOL


@pytest.mark.parametrize("T", [100, 300, 520])
@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3.4e38])
def test_values_bf16_cannot_hold_take_fp32_products(T, bad):
    """Infinities, NaN and values that round to infinity in bf16 give what fp32 arithmetic gives."""
    N, D, row = 64, 32, T // 2
    x = _latent(1, 2, T, N, seed=7) + 0.01
    v, do = _randn(1, 1, T, D, seed=8), _randn(1, 2, T, D, seed=9)
    x[0, 1, row, 3] = bad
    small = bad == 3.4e38
    if small:  # keep every product finite
        x[0, 1, :, 3] = torch.where(torch.arange(T) == row, x[0, 1, :, 3], x[0, 1, :, 3] * 1e-36)
    got = ext.tril_score_v(x.cuda(), x.cuda(), v.cuda()).cpu()
    dx, _, dv = ext.tril_score_v_bwd(x.cuda(), None, v.cuda(), do.cuda())
    s = (x @ x.transpose(-2, -1)).tril(-1)
    want = s @ v
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    ok = torch.isfinite(want)
    assert _rel(got[ok], want[ok]) <= 1e-5
    wdv = sum(s[:, h].transpose(-2, -1) @ do[:, h] for h in range(2))
    assert torch.equal(torch.isfinite(dv.cpu()[:, 0]), torch.isfinite(wdv))
    g = (do @ v.transpose(-2, -1)).tril(-1)
    wdx = (g + g.transpose(-2, -1)) @ x
    assert torch.equal(torch.isfinite(dx.cpu()), torch.isfinite(wdx))
    okx = torch.isfinite(wdx)
    assert _rel(dx.cpu()[okx], wdx[okx]) <= 1e-5


@pytest.mark.parametrize("T", [100, 300, 520])
def test_products_that_only_their_leading_planes_overflow(T):
    """1.8425e19^2 = 3.39e38 is finite in fp32; its leading bf16 planes are 2^64 each."""
    N, D, big = 64, 32, 1.8425e19
    x = _latent(1, 2, T, N, seed=10) * 1e-3
    x[..., 3] = 0
    x[0, :, [0, T - 1], 3] = big
    v = _randn(1, 1, T, D, seed=11) * 1e-3
    got = ext.tril_score_v(x.cuda(), x.cuda(), v.cuda()).cpu()
    assert torch.isfinite(got).all() and _rel(got, _attn64(x.double(), x.double(), v.double())) <= TOL
    # G = dO V^T of the backward, and M^T dO and G x with both factors large
    do, w = torch.zeros(1, 2, T, D), torch.zeros(1, 1, T, D)
    do[0, :, T - 1, 0] = w[0, 0, 0, 0] = big
    y = _latent(1, 2, T, N, seed=12) * 1e-3
    dx, _, dv = ext.tril_score_v_bwd(y.cuda(), None, w.cuda(), do.cuda())
    y64, w64 = y.double().requires_grad_(True), w.double().requires_grad_(True)
    wdx, wdv = torch.autograd.grad(_attn64(y64, y64, w64), (y64, w64), do.double())
    assert torch.isfinite(dx).all() and _rel(dx, wdx) <= TOL and _rel(dv, wdv) <= TOL


@pytest.mark.parametrize("T", [100, 300, 520])
@pytest.mark.parametrize("e", [112, 120, 126])
def test_small_values_keep_their_bits(T, e):
    """Operands down to fp32's smallest normal: three bf16 planes of the plain value would miss
    its last bits (6e-4 of the result at 2^-124)."""
    N, D, small = 64, 32, 2.0**-e
    x = _latent(1, 2, T, N, seed=13)
    v, do = _randn(1, 1, T, D, seed=14), _randn(1, 2, T, D, seed=15)
    x64, v64 = x.double().requires_grad_(True), v.double().requires_grad_(True)
    want = _attn64(x64, x64, v64)
    wdx, wdv = torch.autograd.grad(want, (x64, v64), do.double())
    got = ext.tril_score_v(x.cuda(), x.cuda(), (v * small).cuda())
    dx, _, dv = ext.tril_score_v_bwd(x.cuda(), None, v.cuda(), (do * small).cuda())
    # (scaled back in 64 bits; a value of v below 2^-126 is its fp32 rounding, 2^-23 of the largest)
    assert _rel(got.double() / small, want.detach()) <= TOL
    assert _rel(dx.double() / small, wdx) <= TOL and _rel(dv.double() / small, wdv) <= TOL
    # score tiles that are that small: both factors, taken back up by V
    got = ext.tril_score_v(x.cuda() * 2.0**(-e // 2), x.cuda() * 2.0**(-e // 2), (v * 2.0**40).cuda())
    assert _rel(got.double() * 2.0**(-40 - 2 * (-e // 2)), want.detach()) <= TOL
