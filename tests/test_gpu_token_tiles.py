"""The token-tile kernels at the edges of their dispatch and of their tiles: 32-token tiles while one per CU
covers the launch (256 CUs: 8,192 tokens), 64-token tiles beyond, partial last tiles, and for the per-op
GEMMs widths that are not a multiple of a panel, of a k-step group or of the eight waves' tiles.

References are the oracle's emulations of the same arithmetic, as in test_gpu_ops.py and test_gpu_blocks.py.
"""

from __future__ import annotations

import pytest
import torch

from oracle import folded, kernels as ok, reference
from turbo_roformer_amd import _hip, weights
from turbo_roformer_amd.stack import HipStack

from .conftest import assert_bf16_close, rand_x, snr_db

DEV = "cuda"
CFG = dict(weights.TINY_CFG, depth=1)


def _weight(rows, k, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(rows, k, generator=g) / k**0.5).to(torch.bfloat16), torch.randn(rows, generator=g) * 0.1


@pytest.mark.gpu
@pytest.mark.parametrize("n", [33, 8195])
@pytest.mark.parametrize("K", [16, 144, 528, 1040])
def test_gemm_res_norm_widths(hip, n, K):
    W, b = _weight(256, K, K)
    A = (rand_x(n, 60 + K).repeat(1, K // 256 + 1)[:, :K] * 0.5).to(torch.bfloat16).contiguous()
    X = rand_x(n, 61, 2.0)
    Xr, xnr = ok.gemm_res_norm(A, W, b, X)
    Xd, xn = X.to(DEV), torch.empty(n, 256, dtype=torch.bfloat16, device=DEV)
    print(f"gemm_res_norm K={K} n={n}", flush=True)
    _hip.gemm_res_norm(A.to(DEV), _hip.pack_weight(W.to(DEV)), b.to(DEV), Xd, xn)
    torch.cuda.synchronize()
    torch.testing.assert_close(Xd.cpu(), Xr, rtol=1e-5, atol=1e-5)  # fp32 sums of bf16 products
    assert_bf16_close(xnr, xn, "xn", min_snr=55)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [33, 8195])
@pytest.mark.parametrize("n_out", [32, 288, 544])
def test_gemm_gelu_widths(hip, n, n_out):
    W, b = _weight(n_out, 256, n_out)
    xn = (rand_x(n, 70) * 0.5).to(torch.bfloat16)
    Hr = ok.gemm_gelu(xn, W, b)
    H = torch.empty(n, n_out, dtype=torch.bfloat16, device=DEV)
    print(f"gemm_gelu n_out={n_out} n={n}", flush=True)
    _hip.gemm_gelu(xn.to(DEV), _hip.pack_weight(W.to(DEV)), b.to(DEV), H)
    torch.cuda.synchronize()
    assert_bf16_close(Hr, H, "H", min_snr=50)


@pytest.mark.gpu
def test_gemm_gelu_is_as_close_as_erff(hip):
    """Zero weights, so the outputs are the GELU of the biases: 2^20 normal ones, of which 0.5 x (1 + erff(x /
    sqrt 2)) in float32 rounds 2.4e-5 to the wrong bf16 (+- 5e-6: sampling).  A&S 7.1.26 rounds 9.6e-5."""
    n_out = 1 << 18
    xn = torch.zeros(1, 256, dtype=torch.bfloat16, device=DEV)
    Wp = _hip.pack_weight(torch.zeros(n_out, 256, dtype=torch.bfloat16, device=DEV))
    wrong = 0
    for seed in range(4):
        b = torch.randn(n_out, generator=torch.Generator().manual_seed(seed))
        b[:8] = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), 1e30, -1e30, 75.0, -75.0])
        H = torch.empty(1, n_out, dtype=torch.bfloat16, device=DEV)
        print(f"gemm_gelu of biases, seed {seed}", flush=True)
        _hip.gemm_gelu(xn, Wp, b.to(DEV), H)
        x = b.double()
        exact = 0.5 * x * (1 + torch.erf(x / 2**0.5))
        exact[3] = 0.0  # the limit (0.5 inf 0)
        wrong += int((H[0].cpu() != exact.float().to(torch.bfloat16)).sum())
        assert torch.equal(H[0, :8].cpu().float(), exact[:8].to(torch.bfloat16).float())
    assert wrong <= 40, f"{wrong} of 2^20 outputs round to the wrong bf16"


@pytest.mark.gpu
@pytest.mark.parametrize("n_out,n", [(32, 16385), (64, 32773)])
def test_gemm_gelu_narrow(hip, n_out, n):
    """One or two weight tiles and more than 16,384 tokens a tile: the kernel without LDS, the same bits as the
    other one's on a part of the tokens (the last workgroup and the last wave are partial)."""
    W, b = _weight(n_out, 256, 7)
    xn = (rand_x(n, 71) * 0.5).to(torch.bfloat16)
    Wp = _hip.pack_weight(W.to(DEV))
    H = torch.full((n + 1, n_out), 7.0, dtype=torch.bfloat16, device=DEV)
    print(f"gemm_gelu narrow n_out={n_out} n={n}", flush=True)
    _hip.gemm_gelu(xn.to(DEV), Wp, b.to(DEV), H[:n])
    assert bool((H[n] == 7.0).all())
    part = slice(n - 4001, n)
    Hp = torch.empty(4001, n_out, dtype=torch.bfloat16, device=DEV)
    _hip.gemm_gelu(xn[part].contiguous().to(DEV), Wp, b.to(DEV), Hp)
    assert torch.equal(H[part], Hp)
    assert_bf16_close(ok.gemm_gelu(xn[part], W, b), Hp, "H", min_snr=50)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["ff_fp16", "ff_split", "bf16"])
@pytest.mark.parametrize("n", [1, 33, 8192, 8193])
def test_feed_forward_tiles(hip, precision, n):
    """The feed-forward sub-layer at both tile sizes against the float64 one, with a floor for each arithmetic as
    in test_gpu_blocks.py: a kernel that ran another one would be 15 dB and more below (the emulations here: bf16
    50.2, fp16 68.3, split without one of its lo parts 56.2)."""
    sd = weights.init_state_dict(CFG, seed=5, init="normal")
    stack = HipStack(sd, DEV, precision=precision)
    X = rand_x(n, 80 + n)
    Xd = X.to(DEV)
    print(f"feed-forward tiles n={n} {precision}", flush=True)
    stack.ff_block(Xd, 1, n, 1, 0)
    torch.cuda.synchronize()
    ref = reference.feed_forward(X.double(), {k: v.double() for k, v in sd.items()}, "layers.0.0.layers.0.1")
    floor = {"ff_split": 90.0, "ff_fp16": 66.0, "bf16": 48.5}[precision]
    assert snr_db(ref.numpy(), (Xd.cpu() - X).numpy()) >= floor


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["ff_fp16", "ff_split", "bf16"])
@pytest.mark.parametrize("T,F", [(11, 3), (2765, 3)])
def test_fused_block_matches_its_halves(hip, precision, T, F):
    """Out-projection and feed-forward in one kernel (the stack) against the same as two (the attention
    block's out-projection, then the feed-forward block).  They differ by the fp32 order of the residual
    sums, which moves an operand of the feed-forward across a rounding boundary now and then: 60 dB allows
    one half-step of bf16 (2^-9) in 1 of 4 operands."""
    sd = weights.init_state_dict(CFG, seed=6, init="normal")
    stack = HipStack(sd, DEV, precision=precision)
    X = rand_x(T * F, 90).to(DEV)
    print(f"fused block T={T} F={F} {precision}", flush=True)
    got = stack(X.clone(), 1, T, F)
    want = X.clone()
    for layer in range(len(stack.modes)):
        stack.attn_block(want, 1, T, F, layer)
        stack.ff_block(want, 1, T, F, layer)
    torch.cuda.synchronize()
    assert snr_db((want - X).cpu().numpy(), (got - X).cpu().numpy()) >= 60.0


@pytest.mark.gpu
@pytest.mark.parametrize("T,spiked", [(128, False), (129, False), (383, True), (385, False), (640, True), (641, False)])
def test_attention_query_blocks(hip, T, spiked):
    """Time attention at the edges of its 128- and 256-query workgroups; spiked: one key scores 100 above the
    rest for half a query tile, so the workgroup redoes its sweep with the guarded shift.  Floor as in
    test_gpu_ops.py."""
    F, g = 2, torch.Generator().manual_seed(T)
    sd = weights.init_state_dict(CFG, seed=3, init="normal")
    w = ok.bf16_weights(folded.fold(sd, 1)[0])
    xn = ok.l2_rows(torch.randn(T * F, 256, generator=g)).to(torch.bfloat16)
    Q, K, Vt, G = ok.qkv_rope(xn, w["W"], w["b_gate"], w["freqs"], 0, 1, T, F)
    if spiked:
        K[:, :, :, 350, :] = 4.0
        Q[:, :, :, 96:112, :] = 100.0 / (64 * 16.0) * 4.0
    want = ok.attention(Q, K, Vt, G, 0, 1, T, F)
    O = torch.empty(T * F, 512, dtype=torch.bfloat16, device=DEV)
    print(f"attention query blocks T={T} spiked={spiked}", flush=True)
    _hip.attention(Q.to(DEV), K.to(DEV), Vt.to(DEV), G.to(DEV), O, 0, 1, T, F)
    torch.cuda.synchronize()
    assert_bf16_close(want, O, "O", min_snr=48)
