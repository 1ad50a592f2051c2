"""The work that users of this framework have it do, as measurable cases.

Each case is one pass through public entry points: the ``kernels`` operators
that BDH model code calls, and ``bdh_harness.BDH`` for whole calls.  Sizes are
those of the repository's own configurations (C1 to C5 of ``bench.py``), its
tests, or generic.

The ranges (``draw``): batch 1 to 64, heads 2 to 8, n_embd 32 to 512, latent
width N = mult * n_embd / heads with mult 4 to 128 (16 to 32768; 16320 at most
for decode, the entry point's limit), sequence length 1 to 2048 with no alignment, fp32 and bf16, contiguous and permuted
latents, packed and capacity-strided caches.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

_PKG = str(Path.cwd() / "bdh-gpu-fast_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import bdh_harness  # noqa: E402
import kernels  # noqa: E402

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


# ------------------------------------------------------------------- cases
def listed():
    return [
        # A short prompt on a small model, fp32: the smallest call (launches and latency).
        dict(name="attn_small_fp32", kind="attn", B=2, nh=4, T=128, N=64, D=128, dtype="fp32"),
        # The headline: fused RoPE attention of one layer over a 512-token batch, bf16 autocast.
        dict(name="attn_prefill_bf16", kind="attn", B=8, nh=4, T=512, N=8192, D=256, dtype="bf16"),
        # The same layer for users who run without autocast (fp32 operands and results).
        dict(name="attn_prefill_fp32", kind="attn", B=8, nh=4, T=512, N=8192, D=256, dtype="fp32"),
        # bdh.py unchanged on this surface: RoPE, then bdh_attn(QR, QR, V), on the model's
        # permuted latent view and a ragged document length.
        dict(name="attn_route_ragged_bf16", kind="route", B=6, nh=4, T=777, N=8192, D=256, dtype="bf16"),
        # Training at context 1024 under AMP: attention forward and backward of one layer.
        dict(name="attn_train_bf16", kind="train", B=16, nh=4, T=1024, N=8192, D=256, dtype="bf16", rope=False),
        # Training without AMP, ragged length: the fused op's forward and backward in fp32.
        dict(name="attn_train_fp32", kind="train", B=2, nh=4, T=387, N=8192, D=256, dtype="fp32", rope=True),
        # A batched generate step late in the sequence: decode over the bf16 KV cache.
        dict(name="decode_batch_bf16", kind="decode", B=64, nh=4, S=511, cap=512, N=8192, D=256, dtype="bf16"),
        # Interactive generate: one sequence, the reference's default fp32 cache.
        dict(name="decode_single_fp32", kind="decode", B=1, nh=4, S=301, cap=1024, N=8192, D=256, dtype="fp32"),
        # The dense part of a prefill layer: encoder, LayerNorm, gated product, decoder, residual LN.
        dict(name="mlp_prefill_bf16", kind="mlp", B=32, nh=4, T=512, N=8192, D=256),
        # Long context: one layer of the 512-wide, 8-head model over 2048 tokens, to logits.
        dict(name="layer_long_bf16", kind="forward", B=4, nh=8, T=2048, D=512, mult=128, L=1),
        # An AMP training step of the 256-wide model (two of its layers): loss and all gradients.
        dict(name="model_train_amp", kind="step", B=32, nh=4, T=512, D=256, mult=128, L=2),
        # A generate step of the whole 6-layer model for a few sequences: logits of the next token.
        dict(name="model_decode_bf16", kind="token", B=8, nh=4, S=300, D=256, mult=128, L=6),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, then sizes over that kind's range, spread by logarithm."""
    kind = rng.choice(["attn", "attn", "route", "train", "train", "decode", "decode", "mlp", "forward", "step", "token"])
    for _ in range(1000):
        nh = rng.choice([2, 4, 8])
        D = rng.choice([32, 64, 96, 128, 192, 256, 256, 384, 512])
        mult = rng.choice([4, 8, 16, 32, 64, 128, 128])
        c = dict(kind=kind, B=_logint(rng, 1, 64), nh=nh, D=D)
        if kind in ("attn", "route", "train"):
            c.update(T=_logint(rng, 2, 2048), N=mult * D // nh, dtype=rng.choice(["fp32", "bf16"]))
            if kind == "train":
                c["rope"] = rng.choice([True, False])
        elif kind == "decode":
            S = _logint(rng, 1, 2048)
            c.update(S=S, cap=S + rng.randrange(0, 65), N=mult * D // nh, dtype=rng.choice(["fp32", "bf16"]))
        elif kind == "mlp":
            c.update(D=rng.choice([128, 256, 256, 512]), T=_logint(rng, 1, 2048))
            c["N"] = max(16, mult) * c["D"] // nh
        else:
            c.update(D=rng.choice([64, 128, 256, 256, 512]), mult=mult, L=rng.choice([1, 2]))
            if kind == "token":
                c.update(S=_logint(rng, 2, 1024), L=rng.choice([2, 4, 6]))
            else:
                c["T"] = _logint(rng, 16, 1024 if kind == "step" else 2048)
        if kind in ("decode", "token") and c.get("N", mult * c["D"] // nh) > 16320:
            continue
        w = work(c)
        if w["flops"] <= _MOST_FLOPS[kind] and w["bytes"] <= 2.5e9:
            return c
    raise RuntimeError("no case drawn")


_MOST_FLOPS = {"attn": 6e11, "route": 6e11, "train": 1.7e12, "decode": 1e12, "mlp": 9e11, "forward": 1.3e12,
               "step": 4e12, "token": 1e12}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _latent(g, B, nh, T, N, dt, permuted=False):
    """The sparse ReLU latent, about half zeros; ``permuted``: the model's (B, T, nh, N) memory."""
    if permuted:
        return torch.relu(_randn(g, B, T, nh, N, std=0.32)).to(dt).permute(0, 2, 1, 3)
    return torch.relu(_randn(g, B, nh, T, N, std=0.32)).to(dt)


def _model(c, g):
    cfg = bdh_harness.BDHConfig(n_layer=c["L"], n_embd=c["D"], n_head=c["nh"], mlp_internal_dim_multiplier=c["mult"])
    with torch.device("cuda"):
        model = bdh_harness.BDH(cfg)
    with torch.no_grad():
        model.freqs.copy_(kernels.get_freqs(cfg.n_latent))
        for p in model.parameters():
            p.normal_(std=0.02, generator=g)
    return model


def _inputs(c, seed):
    """Inputs of one case, as ``run`` and ``exact`` both take them."""
    g = _gen(seed)
    kind = c["kind"]
    s = {}
    if kind in ("attn", "route", "train"):
        dt = _DTYPES[c["dtype"]]
        B, nh, T, N, D = c["B"], c["nh"], c["T"], c["N"], c["D"]
        s["x"] = _latent(g, B, nh, T, N, dt, permuted=kind == "route")
        s["v"] = _randn(g, B, 1, T, D).to(dt)
        s["freqs"] = kernels.get_freqs(N).to("cuda")
        if kind == "train":
            s["dy"] = _randn(g, B, nh, T, D).to(dt)
        if kind == "route":
            s["cos"], s["sin"] = kernels.rope_cos_sin(T, 0, s["freqs"])
    elif kind == "decode":
        dt = _DTYPES[c["dtype"]]
        B, nh, N, D = c["B"], c["nh"], c["N"], c["D"]
        s["kr"] = _latent(g, B, nh, c["cap"], N, dt)
        s["vc"] = _randn(g, B, 1, c["cap"], D).to(dt)
        s["q"] = _latent(g, B, nh, 1, N, dt)
    elif kind == "mlp":
        B, nh, T, N, D = c["B"], c["nh"], c["T"], c["N"], c["D"]
        s["x"] = F.layer_norm(_randn(g, B, T, D), (D,))
        s["ykv"] = _randn(g, B, nh, T, D).bfloat16()
        s["enc_t"] = _randn(g, nh, N, D, std=0.02).bfloat16()
        s["encv_t"] = _randn(g, nh, N, D, std=0.02).bfloat16()
        s["dec"] = _randn(g, nh * N, D, std=0.02).bfloat16()
    else:
        s["model"] = _model(c, g)
        T = c["S"] + 1 if kind == "token" else c["T"]
        s["idx"] = torch.randint(0, 256, (c["B"], T), generator=g, device="cuda")
        if kind == "step":
            s["targets"] = torch.randint(0, 256, (c["B"], T), generator=g, device="cuda")
    return s


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    s["case"] = dict(c)
    if c["kind"] == "train":
        s["x"].requires_grad_(True)
        s["v"].requires_grad_(True)
    elif c["kind"] == "decode":
        s["past_k"] = s["kr"].narrow(2, 0, c["S"])  # capacity-strided views, as the cache hands them out
        s["past_v"] = s["vc"].narrow(2, 0, c["S"])
    elif c["kind"] == "token":
        m = s["model"]
        s["cache"] = bdh_harness.KVCache(m.config, c["B"], c["S"] + 1, torch.bfloat16, "cuda")
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
            m(s["idx"][:, : c["S"]].contiguous(), cache=s["cache"], impl="hip", last_only=True)
        s["next"] = s["idx"][:, c["S"]:].contiguous()
    return s


# --------------------------------------------------------------------- run
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "attn":
        return kernels.bdh_attn_rope(s["x"], s["v"], s["freqs"], 0, impl="hip")
    if kind == "route":
        qr = kernels.bdh_rope_rotate(s["x"], s["cos"], s["sin"], impl="hip")
        return qr, kernels.bdh_attn(qr, qr, s["v"], impl="hip")
    if kind == "train":
        x, v = s["x"], s["v"]
        if c["rope"]:
            out = kernels.bdh_attn_rope(x, v, s["freqs"], 0, impl="hip")
        else:
            out = kernels.bdh_attn(x, x, v, impl="hip")
        return (out.detach(), *torch.autograd.grad(out, (x, v), s["dy"]))
    if kind == "decode":
        return kernels.bdh_attn_decode(s["q"], s["past_k"], s["past_v"], impl="hip")
    if kind == "mlp":
        B, nh, T, D = c["B"], c["nh"], c["T"], c["D"]
        xb = s["x"].to(torch.bfloat16)
        xs = kernels.relu_gemm(xb.unsqueeze(1).expand(B, nh, T, D), s["enc_t"])
        y = kernels.layer_norm_rows(s["ykv"], out_dtype=torch.bfloat16)
        if D == 256:
            y = kernels.gated_decoder(y, s["encv_t"], xs, s["dec"])
        else:
            y = kernels.gated_gemm(y, s["encv_t"], xs).view(B, T, -1) @ s["dec"]
        return xs, kernels.layer_norm_rows(y, s["x"], out_dtype=torch.float32)
    m = s["model"]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        if kind == "step":
            m.zero_grad(set_to_none=True)
            _, loss = m(s["idx"], s["targets"], impl="hip")
            loss.backward()
            return {"loss": loss.detach(), **{n: p.grad for n, p in m.named_parameters()}}
        with torch.no_grad():
            if kind == "forward":
                return m(s["idx"], impl="hip")[0]
            s["cache"].seq_len = c["S"]  # the same step again: its rows are written anew
            return m(s["next"], cache=s["cache"], impl="hip", last_only=True)[0]


# -------------------------------------------------------------------- work
def work(case):
    c, kind = case, case["kind"]
    B, nh, D = c["B"], c["nh"], c["D"]
    if kind in ("attn", "route", "train"):
        T, N, e = c["T"], c["N"], 2 if c["dtype"] == "bf16" else 4
        fwd = B * nh * (N + D) * T * (T - 1)
        x, v, o = e * B * nh * T * N, e * B * T * D, e * B * nh * T * D
        if kind == "train":
            return {"flops": 3 * fwd, "bytes": 2 * x + 2 * v + 2 * o}
        return {"flops": fwd, "bytes": x + v + o + (x if kind == "route" else 0)}
    if kind == "decode":
        e, S, N = 2 if c["dtype"] == "bf16" else 4, c["S"], c["N"]
        return {"flops": 2 * B * nh * S * (N + D), "bytes": e * (B * nh * S * N + B * S * D + B * nh * (N + D))}
    if kind == "mlp":
        M, N = B * c["T"], c["N"]
        return {"flops": 6 * M * nh * N * D, "bytes": 2 * M * nh * N + M * D * (8 + 2 * nh) + 6 * nh * N * D}
    N, L = c["mult"] * D // nh, c["L"]
    T = 1 if kind == "token" else c["T"]
    S = c.get("S", 0)
    dense = 6 * B * T * nh * N * D
    attn = B * nh * (N + D) * (T * (T - 1) + 2 * T * S)
    head = 2 * B * T * D * 256
    weights = 3 * nh * N * D * L + 512 * D  # the layers share weights, but each layer reads them
    cache = 2 * L * B * S * (nh * N + D)
    if kind == "step":
        # the latent is the one large tensor a layer has to keep for its backward
        lat = 2 * B * T * nh * N * L
        return {"flops": 3 * (L * (dense + attn) + head), "bytes": 2 * lat + 6 * weights + 8 * (3 * nh * N * D + 512 * D)}
    return {"flops": L * (dense + attn) + head, "bytes": 2 * weights + cache + 4 * B * T * 256}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    kind = case["kind"]
    if kind in ("attn", "route", "train", "decode"):
        return {"rel": 1e-5 if case["dtype"] == "fp32" else 1e-2}
    # whole calls: bf16 rounding of one layer travels through the next (measured against exact():
    # logits 0.005 to 0.01, gradients of a step up to 0.053)
    return {"rel": {"mlp": 1e-2, "forward": 2e-2, "token": 4e-2, "step": 2e-1}[kind]}


# ------------------------------------------------------------------- exact
def _rope64(x, freqs, start=0):
    """RoPE with the phase as the model defines it (fp32 position * frequency, mod 1), the rest in 64 bits."""
    T = x.size(-2)
    pos = torch.arange(start, start + T, device=x.device, dtype=torch.float32)
    ph = ((pos[:, None] * freqs.reshape(1, -1)) % 1).double() * (2 * math.pi)
    c, sn = torch.cos(ph)[:, 0::2], torch.sin(ph)[:, 0::2]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack((x0 * c - x1 * sn, x1 * c + x0 * sn), dim=-1).flatten(-2)


def _tril64(q, v):
    """(q q^T).tril(-1) @ v for one (T, N), (T, D) pair."""
    return (q @ q.t()).tril(-1) @ v


def _layer64(x, w_enc, w_v, dec, freqs):
    """One BDH layer of one sequence in 64 bits: x (T, D), weights (nh, D, N) and (nh*N, D)."""
    nh, D, N = w_enc.shape
    ln = lambda t: F.layer_norm(t, (t.size(-1),), eps=1e-5)  # noqa: E731
    y = 0
    for h in range(nh):
        lat = F.relu(x @ w_enc[h])
        q = _rope64(lat, freqs)
        yv = F.relu(ln(_tril64(q, x)) @ w_v[h])
        y = y + (lat * yv) @ dec[h * N:(h + 1) * N]
    return ln(x + ln(y))


def exact(case, seed):
    c, kind = case, case["kind"]
    if work(case)["flops"] > 1e13:
        return None
    s = _inputs(case, seed)
    if kind in ("attn", "route"):
        B, nh, T, D = c["B"], c["nh"], c["T"], c["D"]
        out = torch.empty(B, nh, T, D, dtype=torch.float64, device="cuda")
        qr = torch.empty(B, nh, T, c["N"], dtype=torch.float64, device="cuda") if kind == "route" else None
        for b in range(B):
            for h in range(nh):
                q = _rope64(s["x"][b, h].double(), s["freqs"])
                out[b, h] = _tril64(q, s["v"][b, 0].double())
                if qr is not None:
                    qr[b, h] = q
        return out if qr is None else (qr, out)
    if kind == "train":
        B, nh, T, D = c["B"], c["nh"], c["T"], c["D"]
        out = torch.empty(B, nh, T, D, dtype=torch.float64, device="cuda")
        dx = torch.empty(B, nh, T, c["N"], dtype=torch.float64, device="cuda")
        dv = torch.zeros(B, 1, T, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            for h in range(nh):
                x = s["x"][b, h].double().requires_grad_(True)
                v = s["v"][b, 0].double().requires_grad_(True)
                o = _tril64(_rope64(x, s["freqs"]) if c["rope"] else x, v)
                gx, gv = torch.autograd.grad(o, (x, v), s["dy"][b, h].double())
                out[b, h], dx[b, h] = o.detach(), gx
                dv[b, 0] += gv
        return out, dx, dv
    if kind == "decode":
        B, nh, S = c["B"], c["nh"], c["S"]
        out = torch.empty(B, nh, 1, c["D"], dtype=torch.float64, device="cuda")
        for b in range(B):
            v = s["vc"][b, 0, :S].double()
            for h in range(nh):
                out[b, h] = (s["q"][b, h].double() @ s["kr"][b, h, :S].double().t()) @ v
        return out
    if kind == "mlp":
        B, nh, T, N, D = c["B"], c["nh"], c["T"], c["N"], c["D"]
        ln = lambda t: F.layer_norm(t, (D,), eps=1e-5)  # noqa: E731
        xs = torch.empty(B, T, nh, N, dtype=torch.float64, device="cuda")
        out = torch.empty(B, T, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            x, y = s["x"][b].double(), 0
            for h in range(nh):
                lat = F.relu(x @ s["enc_t"][h].double().t())
                g = F.relu(ln(s["ykv"][b, h].double()) @ s["encv_t"][h].double().t())
                y = y + (lat * g) @ s["dec"][h * N:(h + 1) * N].double()
                xs[b, :, h] = lat
            out[b] = ln(x + ln(y))
        return xs, out
    m = s["model"].double()
    freqs = m.freqs.float()
    grads = kind == "step"
    ps = dict(m.named_parameters())
    logits, loss = [], 0.0
    with torch.set_grad_enabled(grads):
        for b in range(c["B"]):  # one sequence at a time: gradients add up
            x = F.layer_norm(m.embed(s["idx"][b]), (c["D"],), eps=1e-5)
            for _ in range(c["L"]):
                x = _layer64(x, m.encoder, m.encoder_v, m.decoder, freqs)
            z = x @ m.lm_head
            if grads:
                part = F.cross_entropy(z, s["targets"][b]) / c["B"]
                part.backward()
                loss += float(part.detach())
            else:
                logits.append(z[-1:] if kind == "token" else z)
    if grads:
        return {"loss": loss, **{n: p.grad for n, p in ps.items()}}
    return torch.stack(logits)
