"""Packed weights belong to an ABI version: a program may keep them (in a file, in a pool) and hand them to any
library of that version, so their bytes must not change under it.  The digests are of weights that every
library packs alike (small multiples of 1/128, exact in bf16 and fp16); a new order or a new layout fails here
until TRF_ABI_VERSION and the table move with it."""

from __future__ import annotations

import hashlib

import pytest
import torch

from turbo_roformer_amd import _hip

DIMS, HIDDEN = (8, 12, 40), 64  # widths that are and are not multiples of 8 and 32

DIGESTS = {
    8: dict(layer="ddee62a8510e2eb7", weight="dcdd05bc9a30ca15", split="40f5e39aa2d17a34", mask="63f3ccc16cd229a3"),
    9: dict(layer="ba11292b83c04e32", weight="dcdd05bc9a30ca15", split="ad9d6dd26d253ad3", mask="63f3ccc16cd229a3"),
}


def _w(*shape: int, seed: int) -> torch.Tensor:
    n = 1
    for s in shape:
        n *= s
    return (((torch.arange(n, dtype=torch.int64) * (2 * seed + 7) + seed) % 251 - 125).float() / 128).reshape(shape).cuda()


def _bf(*shape: int, seed: int) -> torch.Tensor:
    return _w(*shape, seed=seed).to(torch.bfloat16)


def _digest(blob: torch.Tensor) -> str:
    return hashlib.sha256(blob.cpu().numpy().tobytes()).hexdigest()[:16]


def _blob(n: int) -> torch.Tensor:
    return torch.zeros(n, dtype=torch.uint8, device="cuda")


def packed() -> dict[str, str]:
    layer = _blob(_hip.layer_packed_bytes())
    _hip.pack_layer(_bf(1544, 256, seed=1), _w(8, seed=2), _bf(256, 512, seed=3), _bf(1024, 256, seed=4), _w(1024, seed=5),
                    _bf(256, 1024, seed=6), _w(256, seed=7), layer, _bf(1024, 256, seed=8) / 256, _bf(256, 1024, seed=9) / 256)
    weight = _hip.pack_weight(_bf(96, 48, seed=10), _blob(_hip.weight_packed_bytes(96, 48)))
    split = _blob(_hip.band_split_packed_bytes(DIMS))
    _hip.pack_band_split([(_w(256, d, seed=d), _w(256, seed=d + 1), _w(d, seed=d + 2)) for d in DIMS], DIMS, split)
    mask = _blob(_hip.mask_head_packed_bytes(DIMS, HIDDEN))
    _hip.pack_mask_head([(_w(HIDDEN, 256, seed=d), _w(HIDDEN, seed=d + 1), _w(2 * d, HIDDEN, seed=d + 2), _w(2 * d, seed=d + 3))
                         for d in DIMS], DIMS, HIDDEN, torch.ones(256, device="cuda"), mask)
    return dict(layer=_digest(layer), weight=_digest(weight), split=_digest(split), mask=_digest(mask))


@pytest.mark.gpu
def test_packed_bytes_of_this_abi_version(hip):
    got = packed()
    print(_hip.ABI_VERSION, got)
    assert got == DIGESTS[_hip.ABI_VERSION]
