"""What the speed of this framework is measured on: the calls that a user of the library makes, from the
single ops that a drop-in binding calls up to the separation of audio, over the range of lengths they are
made with.

A case names the entry point (``kind``) and its sizes: ``frames`` of one chunk (100 frames a second at the
44.1 kHz model's hop of 441), ``bands`` (62: the full model, 29: the small test model), ``batch`` chunks, and
the options.  Every length is odd somewhere: audio has no round length, and a 17 s chunk has 1701 frames.

Weights have the model's shapes and the default initialisation of its layers, with gains and biases moved off
1 and 0; activations are normal with a scale that differs from band to band, as band-split tokens are.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "turbo-roformer_amd"))

DIM, HEADS, HEAD_DIM, INNER, HIDDEN, QKVG = 256, 8, 64, 512, 1024, 1544
DEV = "cuda"

# Frequencies per band, STFT size and hop, hidden size of the mask estimator's MLPs.
MODELS = {
    62: dict(freqs=(2,) * 24 + (4,) * 12 + (12,) * 8 + (24,) * 8 + (48,) * 8 + (128, 129), n_fft=2048, hop=441, mlp=4),
    29: dict(freqs=(4,) * 16 + (8,) * 8 + (16,) * 4 + (65,), n_fft=512, hop=128, mlp=2),
}
DEPTH = 12
DIM_T = 1700  # a chunk is hop * (DIM_T - 1) samples: 17 s


def _dins(bands: int) -> list[int]:
    return [4 * f for f in MODELS[bands]["freqs"]]  # (re, im) of two channels


def _cfg(bands: int, depth: int) -> dict:
    m = MODELS[bands]
    return dict(dim=DIM, depth=depth, stereo=True, num_stems=1, time_transformer_depth=1, freq_transformer_depth=1,
                linear_transformer_depth=0, freqs_per_bands=m["freqs"], dim_head=HEAD_DIM, heads=HEADS,
                dim_freqs_in=m["n_fft"] // 2 + 1, stft_n_fft=m["n_fft"], stft_hop_length=m["hop"],
                stft_win_length=m["n_fft"], stft_normalized=False, mask_estimator_depth=2,
                mlp_expansion_factor=m["mlp"])


# ------------------------------------------------------------------------------------------------ the cases


def listed() -> list[dict]:
    return [
        # One second of audio through the whole stack: the latency of a short call, 24 sub-layers of few blocks.
        dict(name="stack_1s", kind="stack", frames=101, bands=62, batch=1, precision="ff_fp16"),
        # The headline workload: the stack on one 17 s chunk.
        dict(name="stack_17s", kind="stack", frames=1701, bands=62, batch=1, precision="ff_fp16"),
        # A 20.5 s stereo recording from host memory to host memory: two overlapping chunks, STFT to overlap-add.
        dict(name="separate_20s", kind="separate", samples=904_051, bands=62, channels=2, precision="bf16"),
        # Time attention on a ragged 4.9 s clip, as a program that keeps its own layer loop calls it.
        dict(name="attn_time_5s", kind="attn", mode=0, frames=487, bands=62, batch=1),
        # Frequency attention over two 17 s chunks at once (a song runs batched).
        dict(name="attn_freq_34s", kind="attn", mode=1, frames=1701, bands=62, batch=2),
        # The feed-forward block in the most accurate arithmetic (the reference's "fp32" precision), one chunk.
        dict(name="ff_split_17s", kind="ff", frames=1701, bands=62, batch=1, precision="ff_split"),
        # The feed-forward block of a 3 s clip in the default arithmetic.
        dict(name="ff_fp16_3s", kind="ff", frames=303, bands=62, batch=1, precision="ff_fp16"),
        # The mask head after the stack, one chunk, fp32-level arithmetic (the default).
        dict(name="mask_split_17s", kind="mask", frames=1701, bands=62, precision="split"),
        # The mask head of a short clip at the reduced precision.
        dict(name="mask_fp16_1s", kind="mask", frames=101, bands=62, precision="fp16"),
        # The band split before the stack, one chunk.
        dict(name="band_split_17s", kind="split", frames=1701, bands=62),
        # One sub-layer on the op-by-op binding (time attention: norm, QKV, attention, three GEMMs), one chunk.
        dict(name="ops_time_17s", kind="ops", mode=0, frames=1701, bands=62, batch=1),
        # The same over frequency (one fused op for QKV and attention) on a 2.5 s clip.
        dict(name="ops_freq_2s", kind="ops", mode=1, frames=251, bands=62, batch=1),
    ]


def _log_uniform(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("stack", "separate", "attn", "attn", "ff", "mask", "split", "ops"))
    bands = rng.choice((62, 62, 62, 29))
    if kind == "separate":  # from a third of a second up to one whole chunk and its tail
        return dict(kind=kind, samples=_log_uniform(rng, 15_000, 850_000), bands=62, channels=rng.choice((1, 2)),
                    precision=rng.choice(("bf16", "fp32")))
    frames = _log_uniform(rng, 9, 1701)
    batch = rng.randint(1, max(1, min(3, 1701 // frames)))
    if kind == "stack":
        return dict(kind=kind, frames=frames, bands=bands, batch=batch,
                    precision=rng.choice(("ff_fp16", "ff_fp16", "ff_split", "bf16")))
    if kind == "ff":
        return dict(kind=kind, frames=frames, bands=bands, batch=batch,
                    precision=rng.choice(("ff_fp16", "ff_split", "bf16")))
    if kind == "mask":
        return dict(kind=kind, frames=frames * batch, bands=bands, precision=rng.choice(("split", "fp16")))
    if kind == "split":
        return dict(kind=kind, frames=frames * batch, bands=bands)
    return dict(kind=kind, mode=rng.randint(0, 1), frames=frames, bands=bands, batch=batch)


# ------------------------------------------------------------------------------------------------ inputs


def _gen(seed: int, stream: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(1_000_003 * (seed + 1) + stream)


def _uniform(g: torch.Generator, *shape: int) -> torch.Tensor:
    return (torch.rand(*shape, generator=g, device=DEV) * 2 - 1) / math.sqrt(shape[-1])


def _gain(g: torch.Generator, n: int) -> torch.Tensor:
    return 1.0 + 0.25 * torch.randn(n, generator=g, device=DEV)


def _bias(g: torch.Generator, n: int) -> torch.Tensor:
    return 0.05 * torch.randn(n, generator=g, device=DEV)


def _freqs() -> torch.Tensor:
    return 1.0 / (10000.0 ** (torch.arange(0, HEAD_DIM, 2).float() / HEAD_DIM))


def _stack_weights(seed: int, depth: int, modes=(0, 1)) -> dict[str, torch.Tensor]:
    g = _gen(seed, 1)
    sd = {}
    for i in range(depth):
        for m in modes:
            p = f"layers.{i}.{m}.layers.0"
            sd[f"{p}.0.rotary_embed.freqs"] = _freqs()
            sd[f"{p}.0.norm.gamma"] = _gain(g, DIM)
            sd[f"{p}.0.to_qkv.weight"] = _uniform(g, 3 * INNER, DIM)
            sd[f"{p}.0.to_gates.weight"] = _uniform(g, HEADS, DIM)
            sd[f"{p}.0.to_gates.bias"] = _bias(g, HEADS)
            sd[f"{p}.0.to_out.0.weight"] = _uniform(g, DIM, INNER)
            sd[f"{p}.1.net.0.gamma"] = _gain(g, DIM)
            sd[f"{p}.1.net.1.weight"] = _uniform(g, HIDDEN, DIM)
            sd[f"{p}.1.net.1.bias"] = _bias(g, HIDDEN)
            sd[f"{p}.1.net.4.weight"] = _uniform(g, DIM, HIDDEN)
            sd[f"{p}.1.net.4.bias"] = _bias(g, DIM)
    return sd


def _split_weights(seed: int, bands: int) -> dict[str, torch.Tensor]:
    g = _gen(seed, 2)
    sd = {}
    for i, d in enumerate(_dins(bands)):
        sd[f"band_split.to_features.{i}.0.gamma"] = _gain(g, d)
        sd[f"band_split.to_features.{i}.1.weight"] = _uniform(g, DIM, d)
        sd[f"band_split.to_features.{i}.1.bias"] = _bias(g, DIM)
    return sd


def _mask_weights(seed: int, bands: int) -> dict[str, torch.Tensor]:
    g = _gen(seed, 3)
    hidden = DIM * MODELS[bands]["mlp"]
    sd = {"final_norm.gamma": _gain(g, DIM)}
    for i, d in enumerate(_dins(bands)):
        p = f"mask_estimators.0.to_freqs.{i}.0"
        sd[f"{p}.0.weight"] = _uniform(g, hidden, DIM)
        sd[f"{p}.0.bias"] = _bias(g, hidden)
        sd[f"{p}.2.weight"] = _uniform(g, 2 * d, hidden)
        sd[f"{p}.2.bias"] = _bias(g, 2 * d)
    return sd


def _tokens(seed: int, batch: int, frames: int, bands: int) -> torch.Tensor:
    """[batch * frames * bands, 256] fp32, token (chunk, frame, band)."""
    g = _gen(seed, 4)
    scale = torch.exp(0.5 * torch.randn(1, bands, 1, generator=g, device=DEV))
    x = torch.randn(batch * frames, bands, DIM, generator=g, device=DEV) * scale
    return x.reshape(-1, DIM).contiguous()


def _features(seed: int, frames: int, bands: int) -> torch.Tensor:
    """[frames, sum(dins)] fp32: a spectrum that falls off with frequency, as music's does."""
    g = _gen(seed, 5)
    width = sum(_dins(bands))
    fall = 30.0 / torch.sqrt(1.0 + torch.arange(width, device=DEV) / 8.0)
    return torch.randn(frames, width, generator=g, device=DEV) * fall


def _audio(seed: int, channels: int, n: int) -> np.ndarray:
    """(channels, n) float32: a vibrato tone over noise with a 1/f spectrum, louder than full scale at its peak."""
    rng = np.random.default_rng(seed)
    spec = np.fft.rfft(rng.standard_normal((channels, n), dtype=np.float32), axis=1)
    x = np.fft.irfft(spec / np.sqrt(1.0 + np.arange(spec.shape[1])), n, axis=1)
    x = x / x.std()
    t = np.arange(n) / 44100.0
    x = x + np.sin(2 * np.pi * 220.0 * t + 3.0 * np.sin(2 * np.pi * 5.5 * t))
    return (1.1 * x / np.abs(x).max()).astype(np.float32)


def _folded(sd: dict, mode: int) -> dict[str, torch.Tensor]:
    """Plain folded fp32 weights of a sub-layer: 16 * gamma into the next Linear's columns, 1/8 into W_q."""
    p = f"layers.0.{mode}.layers.0"
    ga = 16.0 * sd[f"{p}.0.norm.gamma"][None, :]
    gf = 16.0 * sd[f"{p}.1.net.0.gamma"][None, :]
    wqkv = sd[f"{p}.0.to_qkv.weight"] * ga
    wqkv[:INNER] *= 0.125
    return dict(w_qkvg=torch.cat([wqkv, sd[f"{p}.0.to_gates.weight"] * ga]), b_gate=sd[f"{p}.0.to_gates.bias"],
                w_out=sd[f"{p}.0.to_out.0.weight"], w_ff1=sd[f"{p}.1.net.1.weight"] * gf,
                b_ff1=sd[f"{p}.1.net.1.bias"], w_ff2=sd[f"{p}.1.net.4.weight"], b_ff2=sd[f"{p}.1.net.4.bias"])


# ------------------------------------------------------------------------------------------------ prepare


def prepare(case: dict, seed: int) -> dict:
    from turbo_roformer_amd import _hip
    from turbo_roformer_amd.band_split import HipBandSplit
    from turbo_roformer_amd.mask import HipMaskHead
    from turbo_roformer_amd.separator import Separator
    from turbo_roformer_amd.stack import HipStack, rope_table

    kind, bands = case["kind"], case["bands"]
    s = dict(case)
    if kind == "separate":
        sd = {**_stack_weights(seed, DEPTH), **_split_weights(seed, bands), **_mask_weights(seed, bands)}
        s["separator"] = Separator(sd, _cfg(bands, DEPTH), DIM_T, precision=case["precision"], backend="hip")
        s["mix"] = _audio(seed, case["channels"], case["samples"])
        return s
    if kind == "split":
        s["split"] = HipBandSplit(_split_weights(seed, bands), _cfg(bands, 0))
        s["feats"] = _features(seed, case["frames"], bands)
        return s
    if kind == "mask":
        s["head"] = HipMaskHead(_mask_weights(seed, bands), _cfg(bands, 0), precision=case["precision"])
        s["X"] = _tokens(seed, 1, case["frames"], bands)
        return s
    T, b = case["frames"], case["batch"]
    s["X0"] = _tokens(seed, b, T, bands)
    s["X"] = torch.empty_like(s["X0"])
    if kind != "ops":
        s["stack"] = HipStack(_stack_weights(seed, DEPTH if kind == "stack" else 1), precision=case.get("precision", "ff_fp16"))
        s["stack"].workspace(b, T, bands)
        s["stack"].table(0, T), s["stack"].table(1, bands)
        return s
    mode, bf = case["mode"], torch.bfloat16
    w = _folded(_stack_weights(seed, 1), mode)
    w = {k: v.to(bf) if k.startswith("w_") else v for k, v in w.items()}
    layer = torch.empty(_hip.layer_packed_bytes(), dtype=torch.uint8, device=DEV)
    _hip.pack_layer(*(w[k] for k in ("w_qkvg", "b_gate", "w_out", "w_ff1", "b_ff1", "w_ff2", "b_ff2")), layer)
    L, n = (T if mode == 0 else bands), b * T * bands
    s.update(layer=layer, rope=rope_table(_freqs(), L).to(DEV), L=L, b1=w["b_ff1"], b2=w["b_ff2"])
    s.update(wo=_hip.pack_weight(w["w_out"]), w1=_hip.pack_weight(w["w_ff1"]), w2=_hip.pack_weight(w["w_ff2"]))
    if L > 64:
        s["seq"] = _hip.seq_buffers(mode, b, T, bands)
    s["xn"] = torch.empty(n, DIM, dtype=bf, device=DEV)
    s["O"] = torch.empty(n, INNER, dtype=bf, device=DEV)
    s["H"] = torch.empty(n, HIDDEN, dtype=bf, device=DEV)
    return s


# ------------------------------------------------------------------------------------------------ run


def run(s: dict):
    from turbo_roformer_amd import _hip

    kind, bands = s["kind"], s["bands"]
    if kind == "separate":
        return s["separator"].separate(s["mix"])
    if kind == "split":
        return s["split"](s["feats"])
    if kind == "mask":
        return s["head"](s["X"])
    T, b, X = s["frames"], s["batch"], s["X"]
    X.copy_(s["X0"])  # the layers work in place on the residual stream
    if kind == "stack":
        return s["stack"](X, b, T, bands)
    if kind == "attn":
        return s["stack"].attn_block(X, b, T, bands, s["mode"])
    if kind == "ff":
        return s["stack"].ff_block(X, b, T, bands, 0)
    mode, xn, O, H = s["mode"], s["xn"], s["O"], s["H"]
    _hip.add_rmsnorm(X, None, xn)
    if s["L"] <= 64:
        _hip.qkv_attention_short(xn, s["layer"], s["rope"], mode, b, T, bands, O)
    else:
        _hip.qkv_rope_gemm(xn, s["layer"], s["rope"], mode, b, T, bands, *s["seq"])
        _hip.attention(*s["seq"], O, mode, b, T, bands)
    _hip.gemm_res_norm(O, s["wo"], None, X, xn)
    _hip.gemm_gelu(xn, s["w1"], s["b1"], H)
    _hip.gemm_res_norm(H, s["w2"], s["b2"], X, xn)
    return dict(X=X, xn=xn, O=O, H=H)


# ------------------------------------------------------------------------------------------------ work


def _layer_work(tokens: int, nseq: int, L: int, attn: bool, ff: bool) -> tuple[float, float]:
    """(flops, weight bytes) of a sub-layer's attention and feed-forward halves."""
    fl = by = 0.0
    if attn:
        fl += 2.0 * tokens * DIM * (QKVG + INNER) + 4.0 * nseq * HEADS * L * L * HEAD_DIM
        by += 2.0 * DIM * (QKVG + INNER)
    if ff:
        fl += 4.0 * tokens * DIM * HIDDEN
        by += 4.0 * DIM * HIDDEN
    return fl, by


def _stack_work(b: int, T: int, bands: int, depth: int) -> tuple[float, float]:
    n = b * T * bands
    ft, bt = _layer_work(n, b * bands, T, True, True)
    ff, bf = _layer_work(n, b * T, bands, True, True)
    return depth * (ft + ff), 2.0 * n * DIM * 4 + depth * (bt + bf)


def _split_work(frames: int, bands: int) -> tuple[float, float]:
    w = sum(_dins(bands))
    return 2.0 * frames * w * DIM, 4.0 * (frames * w + frames * bands * DIM + w * DIM)


def _mask_work(frames: int, bands: int, precision: str) -> tuple[float, float]:
    w, hidden = sum(_dins(bands)), DIM * MODELS[bands]["mlp"]
    weights = hidden * (bands * DIM + 2 * w)
    # the weights are held as fp16, in two parts where the products are split
    return 2.0 * frames * weights, 4.0 * frames * (bands * DIM + w) + (2 if precision == "fp16" else 4) * weights


def _chunks(n: int, hop: int) -> tuple[int, list[int]]:
    """(samples of a chunk, its starts): overlap 2, the last chunk ends with the signal."""
    chunk = min(hop * (DIM_T - 1), n)
    step, starts, s = max(1, chunk // 2), [], 0
    while s + chunk < n:
        starts.append(s)
        s += step
    if not starts or starts[-1] != n - chunk:
        starts.append(n - chunk)
    return chunk, starts


def _padded(n: int, hop: int) -> int:
    return n if n >= hop * (DIM_T - 1) else max(-(-n // hop) * hop, 3 * hop)


def work(case: dict) -> dict:
    kind, bands = case["kind"], case["bands"]
    if kind == "separate":
        m = MODELS[bands]
        n = _padded(case["samples"], m["hop"])
        chunk, starts = _chunks(n, m["hop"])
        T, b = chunk // m["hop"] + 1, len(starts)
        fl = _stack_work(b, T, bands, DEPTH)[0] + _split_work(b * T, bands)[0] + _mask_work(b * T, bands, "split")[0]
        fl += 2 * 2 * b * T * 5.0 * m["n_fft"] / 2 * math.log2(m["n_fft"])
        by = 4.0 * case["samples"] * (case["channels"] + 2)
        by += DEPTH * 2 * 2.0 * DIM * (QKVG + INNER + 2 * HIDDEN) + 4.0 * sum(_dins(bands)) * DIM
        by += 4.0 * DIM * m["mlp"] * (bands * DIM + 2 * sum(_dins(bands)))
        return dict(bytes=by, flops=fl)
    if kind == "split":
        fl, by = _split_work(case["frames"], bands)
        return dict(bytes=by, flops=fl)
    if kind == "mask":
        fl, by = _mask_work(case["frames"], bands, case["precision"])
        return dict(bytes=by, flops=fl)
    T, b = case["frames"], case["batch"]
    n = b * T * bands
    if kind == "stack":
        fl, by = _stack_work(b, T, bands, DEPTH)
        return dict(bytes=by, flops=fl)
    mode = case.get("mode", 0)
    nseq, L = (b * bands, T) if mode == 0 else (b * T, bands)
    fl, by = _layer_work(n, nseq, L, kind != "ff", kind != "attn")
    by += 2.0 * n * DIM * 4
    if kind == "ops":  # each op's tensors go through memory once: that is its interface
        by += n * (2.0 * DIM * 2 + 2 * INNER * 2 + 2 * HIDDEN * 2 + 2 * DIM * 4 + 2 * DIM * 2)
        if L > 64:
            by += n * (2.0 * 3 * INNER * 2 + 2 * HEADS * 4)
    return dict(bytes=by, flops=fl)


# ------------------------------------------------------------------------------------------------ tolerance


# About four times the error against 64 bits that each path shows at the sizes above.


def tolerance(case: dict):
    kind, precision = case["kind"], case.get("precision")
    if kind == "split":
        return {"rel": 1e-6}  # fp32 products and sums
    if kind == "mask":
        return {"rel": 5e-6 if precision == "split" else 1.6e-3}
    if kind == "attn":
        return {"rel": 4e-4}  # bf16 operands; the fp32 residual is most of the output
    if kind == "ff":
        return {"rel": {"ff_split": 5e-6, "ff_fp16": 3e-4, "bf16": 2e-3}[precision]}
    if kind == "ops":
        return {"rel": 1.2e-2}  # bf16 in and out of every op
    if kind == "separate":
        return {"rel": 6e-3}
    return {"rel": 1.2e-2 if precision == "bf16" else 4e-3}  # 24 sub-layers in 16 bits


# ------------------------------------------------------------------------------------------------ exact


def _norm64(x: torch.Tensor) -> torch.Tensor:
    return x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)


def _rotate64(x: torch.Tensor) -> torch.Tensor:
    """x [..., L, 64]: interleaved pairs turned by p * freq."""
    L = x.shape[-2]
    # the angles are fp32 inputs of the op (its cos / sin table)
    ang = torch.arange(L, dtype=torch.float32)[:, None] * _freqs()[None, :]
    c, s = ang.cos().double().to(x.device), ang.sin().double().to(x.device)
    out = torch.empty_like(x)
    out[..., 0::2] = x[..., 0::2] * c - x[..., 1::2] * s
    out[..., 1::2] = x[..., 1::2] * c + x[..., 0::2] * s
    return out


def _attn64(X: torch.Tensor, w: dict, mode: int, b: int, T: int, bands: int) -> torch.Tensor:
    """Gated attention output O [tokens, 512] of the folded weights, 64 bits."""
    n = b * T * bands
    wq, bg = w["w_qkvg"].double(), w["b_gate"].double()
    O = torch.empty(b, T, bands, HEADS, HEAD_DIM, dtype=torch.float64, device=X.device)
    xn = _norm64(X).view(b, T, bands, DIM)
    groups = range(0, bands, 4) if mode == 0 else range(0, T, 512)
    for c in range(b):
        for g0 in groups:
            xs = xn[c, :, g0 : g0 + 4].transpose(0, 1) if mode == 0 else xn[c, g0 : g0 + 512]
            xs = xs.contiguous()  # [sequences, L, 256]
            y = xs.reshape(-1, DIM) @ wq.t().contiguous()
            ns, L = xs.shape[:2]
            qkv = y[:, : 3 * INNER].view(ns, L, 3, HEADS, HEAD_DIM).permute(2, 0, 3, 1, 4).contiguous()
            q, k, v = _rotate64(qkv[0]), _rotate64(qkv[1]), qkv[2]
            gate = torch.sigmoid(y[:, 3 * INNER :] + bg).view(ns, L, HEADS, 1)
            o = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()), -1)
            o = torch.matmul(o, v.contiguous()).permute(0, 2, 1, 3) * gate
            if mode == 0:
                O[c, :, g0 : g0 + 4] = o.transpose(0, 1)
            else:
                O[c, g0 : g0 + 512] = o
    return O.view(n, INNER)


def _hidden64(X: torch.Tensor, w: dict) -> torch.Tensor:
    h = _norm64(X) @ w["w_ff1"].double().t().contiguous() + w["b_ff1"].double()
    return 0.5 * h * (1.0 + torch.erf(h / math.sqrt(2.0)))


def _ff64(X: torch.Tensor, w: dict) -> torch.Tensor:
    w2, b2 = w["w_ff2"].double().t().contiguous(), w["b_ff2"].double()
    return torch.cat([x + _hidden64(x, w) @ w2 + b2 for x in X.split(65536)])


def _stack64(X: torch.Tensor, sd: dict, b: int, T: int, bands: int, depth: int) -> torch.Tensor:
    for i in range(depth):
        for mode in (0, 1):
            p, q = f"layers.{i}.{mode}.", f"layers.0.{mode}."
            w = _folded({q + k[len(p):]: v.double() for k, v in sd.items() if k.startswith(p)}, mode)
            X = X + _attn64(X, w, mode, b, T, bands) @ w["w_out"].t().contiguous()
            X = _ff64(X, w)
    return X


def _split64(feats: torch.Tensor, sd: dict, bands: int) -> torch.Tensor:
    out = []
    for i, x in enumerate(feats.double().split(_dins(bands), dim=-1)):
        p = f"band_split.to_features.{i}"
        x = _norm64(x) * math.sqrt(x.shape[-1]) * sd[f"{p}.0.gamma"].double()
        out.append(x @ sd[f"{p}.1.weight"].double().t().contiguous() + sd[f"{p}.1.bias"].double())
    return torch.stack(out, 1).reshape(-1, DIM)


def _mask64(X: torch.Tensor, sd: dict, bands: int) -> torch.Tensor:
    x = (_norm64(X.double()) * 16.0 * sd["final_norm.gamma"].double()).view(-1, bands, DIM)
    out = []
    for i, d in enumerate(_dins(bands)):
        p = f"mask_estimators.0.to_freqs.{i}.0"
        h = torch.tanh(x[:, i] @ sd[f"{p}.0.weight"].double().t().contiguous() + sd[f"{p}.0.bias"].double())
        y = h @ sd[f"{p}.2.weight"].double().t().contiguous() + sd[f"{p}.2.bias"].double()
        out.append(y[:, :d] * torch.sigmoid(y[:, d:]))
    return torch.cat(out, 1)


def _separate64(case: dict, seed: int) -> np.ndarray:
    bands, n0 = case["bands"], case["samples"]
    m = MODELS[bands]
    x = _audio(seed, case["channels"], n0).astype(np.float64)
    if x.shape[0] == 1:
        x = np.repeat(x, 2, 0)
    n = _padded(n0, m["hop"])
    x = np.pad(x, ((0, 0), (0, n - n0)))
    gain = min(1.0, 0.9 / np.abs(x).max())
    x = torch.from_numpy(x * gain).to(DEV)
    chunk, starts = _chunks(n, m["hop"])
    sd = {**_stack_weights(seed, DEPTH), **_split_weights(seed, bands), **_mask_weights(seed, bands)}
    win = torch.hann_window(m["n_fft"], dtype=torch.float64, device=DEV)
    kw = dict(n_fft=m["n_fft"], hop_length=m["hop"], win_length=m["n_fft"], window=win, normalized=False)
    k = torch.arange(chunk, dtype=torch.float64, device=DEV)
    ham = 0.54 - 0.46 * torch.cos(2.0 * math.pi * k / (chunk - 1))
    acc, wsum = torch.zeros_like(x), torch.zeros(n, dtype=torch.float64, device=DEV)
    for s in starts:
        st = torch.stft(x[:, s : s + chunk], return_complex=True, **kw)  # (2, bins, T)
        T = st.shape[-1]
        X = _split64(torch.view_as_real(st).permute(2, 1, 0, 3).reshape(T, -1), sd, bands)
        mask = _mask64(_stack64(X, sd, 1, T, bands, DEPTH), sd, bands)
        mask = torch.view_as_complex(mask.view(T, -1, 2, 2).permute(2, 1, 0, 3).contiguous())
        y = torch.istft(st * mask, **kw)
        L = min(chunk, y.shape[-1])
        acc[:, s : s + L] += y[:, :L] * ham[:L]
        wsum[s : s + L] += ham[:L]
    return (acc / wsum.clamp_min(1e-10) / gain)[:, :n0].cpu().numpy()


def exact(case: dict, seed: int):
    kind, bands = case["kind"], case["bands"]
    if kind == "separate":
        return _separate64(case, seed)
    if kind == "split":
        return _split64(_features(seed, case["frames"], bands), _split_weights(seed, bands), bands)
    if kind == "mask":
        return _mask64(_tokens(seed, 1, case["frames"], bands), _mask_weights(seed, bands), bands)
    T, b = case["frames"], case["batch"]
    X = _tokens(seed, b, T, bands).double()
    sd = _stack_weights(seed, DEPTH if kind == "stack" else 1)
    if kind == "stack":
        return _stack64(X, sd, b, T, bands, DEPTH)
    mode = case.get("mode", 0)
    w = _folded(sd, mode)
    if kind == "ff":
        return _ff64(X, w)
    if kind == "attn":
        return X + _attn64(X, w, mode, b, T, bands) @ w["w_out"].double().t().contiguous()
    # the ops get their weights in bf16
    w = {k: v.to(torch.bfloat16) if k.startswith("w_") else v for k, v in w.items()}
    O = _attn64(X, w, mode, b, T, bands)
    X = X + O @ w["w_out"].double().t().contiguous()
    H = _hidden64(X, w)
    X = X + H @ w["w_ff2"].double().t().contiguous() + w["b_ff2"].double()
    return dict(X=X, xn=_norm64(X), O=O, H=H)
