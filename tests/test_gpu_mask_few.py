"""The mask head's kernel for few frames (32-frame workgroups whose waves share out the hidden tiles and then the
outputs) against the oracle, and bit for bit against the 128-frame kernel that larger launches run on."""

from __future__ import annotations

import pytest
import torch

from turbo_roformer_amd import _hip, weights
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


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["split", "fp16"])
@pytest.mark.parametrize("hidden", [64, 320, 1024])  # 2 hidden tiles (6 waves have none), 10 (two groups), 32
def test_mask_rows_do_not_depend_on_the_launch(hip, precision, hidden):
    """A frame's mask is the same bits in a launch of few frames and in one of 3,200, which the other kernel
    takes (4 bands: 1.7 times the load per CU up to which the kernel for few frames runs).  Widths of 1, 2, 3 and
    9 output pairs: the last is jobs of 3 pairs in one kernel, of 5 and 4 in the other."""
    dims, n = (8, 40, 96, 260), 3200
    g = torch.Generator().manual_seed(hidden)
    bands = [tuple(t.cuda() for t in (torch.randn(hidden, 256, generator=g) / 16, torch.randn(hidden, generator=g) * 0.1,
                                      torch.randn(2 * d, hidden, generator=g) / hidden**0.5,
                                      torch.randn(2 * d, generator=g) * 0.1)) for d in dims]
    packed = torch.empty(_hip.mask_head_packed_bytes(dims, hidden), dtype=torch.uint8, device="cuda")
    _hip.pack_mask_head(bands, dims, hidden, (1.0 + 0.2 * torch.randn(256, generator=g)).cuda(), packed)
    X = rand_x(n * len(dims), 19).cuda()

    def run(k):
        mask = torch.full((k, sum(dims)), float("nan"), device="cuda")
        _hip.mask_head(X[: k * len(dims)], k, dims, hidden, packed, mask, precision)
        return mask

    print(f"mask rows {precision} hidden={hidden}", flush=True)
    whole = run(n)
    assert torch.isfinite(whole).all()
    for k in (1, 31, 33, 257):
        assert torch.equal(run(k), whole[:k]), f"{k} frames"
