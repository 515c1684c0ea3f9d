"""The mask head's kernel for few frames (32-frame workgroups whose waves share out the hidden tiles) against
the oracle and against the 128-frame kernel, at both sides of the rule that picks it (256 frames)."""

from __future__ import annotations

import pytest
import torch

from turbo_roformer_amd import weights
from turbo_roformer_amd.mask import HipMaskHead

from .conftest import rand_x, snr_db


@pytest.mark.gpu
@pytest.mark.parametrize("precision,floor", [("split", 100.0), ("fp16", 55.0)])
@pytest.mark.parametrize("hidden", [256, 768])  # 8 hidden tiles, one a wave, and 24
@pytest.mark.parametrize("n_frames", [1, 33, 256, 257])
def test_mask_head_few_frames(hip, precision, floor, hidden, n_frames):
    """Widths of 1, 2, 3 and 4 output pairs (the last cut into two jobs), one of them not a multiple of 32.
    Floors as in the other mask tests: ~2^-22 relative products (split), fp16 operands (fp16)."""
    freqs = (2, 10, 24, 32)
    dims = [4 * f for f in freqs]
    cfg = dict(weights.TINY_CFG, freqs_per_bands=freqs, mlp_expansion_factor=hidden // 256)
    g = torch.Generator().manual_seed(hidden)
    sd = {"final_norm.gamma": 1.0 + 0.2 * torch.randn(256, generator=g)}
    for i, d in enumerate(dims):
        p = f"mask_estimators.0.to_freqs.{i}.0"
        for k, (o, c) in {"0": (hidden, 256), "2": (2 * d, hidden)}.items():
            sd[f"{p}.{k}.weight"] = (torch.rand(o, c, generator=g) * 2 - 1) / c**0.5
            sd[f"{p}.{k}.bias"] = 0.1 * torch.randn(o, generator=g)
    X = rand_x(n_frames * len(dims), 17)
    print(f"mask head {precision} hidden={hidden} n_frames={n_frames}", flush=True)
    got = HipMaskHead(sd, cfg, "cuda", precision)(X.cuda(), n_frames).cpu()
    x = X.double().view(n_frames, len(dims), 256)
    x = x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12) * 16.0 * sd["final_norm.gamma"].double()
    ref = []
    for i, d in enumerate(dims):
        p = f"mask_estimators.0.to_freqs.{i}.0"
        w = {k: sd[f"{p}.{k}"].double() for k in ("0.weight", "0.bias", "2.weight", "2.bias")}
        h = torch.tanh(x[:, i] @ w["0.weight"].t() + w["0.bias"])
        y = h @ w["2.weight"].t() + w["2.bias"]
        ref.append(y[:, :d] * torch.sigmoid(y[:, d:]))
    assert snr_db(torch.cat(ref, 1).numpy(), got.double().numpy()) >= floor
