"""tk_small_forward_packed: weights in fragment order give tk_small_forward's results bit for bit."""

from __future__ import annotations

import pytest
import torch

import tkmi
from tkmi import _lib, ops

DEV = "cuda:0"

# split (causal, several row blocks, few sequences) and whole-sequence workgroups; every head dim
SHAPES = [(64, 128, 128, 4, 128, 4, True), (3, 97, 128, 8, 128, 3, True), (2, 64, 128, 2, 128, 2, True),
          (5, 128, 128, 1, 128, 2, True), (300, 33, 128, 4, 128, 2, True), (3, 77, 128, 2, 128, 2, False),
          (2, 128, 128, 1, 128, 1, False), (1, 17, 128, 8, 128, 2, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "b{}s{}h{}l{}{}".format(s[0], s[1], s[3], s[5], "c" if s[6] else ""))
def test_packed_matches_row_major(shape):
    torch.manual_seed(81)
    opt = tkmi.OptimizedTransformer(tkmi.TransformerConfig(*shape)).to(DEV).eval()
    x = torch.randn(*shape[:3], generator=torch.Generator().manual_seed(82)).to(DEV)
    with torch.inference_mode():
        stacked = opt._stacked_weights()
        rows = {k: v for k, v in stacked.items() if k != "packed"}
        lw = opt._weights()[0]
        outs = []
        for w in (stacked, rows, stacked):  # the third: hand-off counts left at zero by the first
            out = torch.full_like(x, float("nan"))
            ops.small_forward(x, out, w, opt._final, lw.n1_eps, lw.n2_eps, opt.num_heads, opt.head_dim_padded, 128,
                              shape[6], opt.attn_scale)
            outs.append(out)
        torch.cuda.synchronize()
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.gpu
def test_pack_layout():
    w = [torch.arange(2 * n * 128, device=DEV).remainder(2039).half().view(2, n, 128) for n in (384, 128, 128, 128)]
    packed = ops.small_pack(dict(zip(("w_qkv", "w_o", "w_1", "w_2"), w))).view(2, 24, 8, 64, 8).cpu()
    rows = torch.cat(w, 1).cpu().view(2, 24, 32, 8, 2, 8)  # layer, block, row, fragment, half, 8 columns
    assert torch.equal(packed, rows.permute(0, 1, 3, 4, 2, 5).reshape(2, 24, 8, 64, 8))


def test_bad_calls_are_refused():
    lib = _lib.load()
    assert lib.tk_small_pack_halves(3) == 3 * 192 * 512 and lib.tk_small_pack_halves(-1) < 0
    assert lib.tk_small_pack(None, 16, 16, 16, 16, 1, None) == _lib.TK_ERR_ARG
    assert lib.tk_small_pack(16, 16, 16, 24, 16, 1, None) == _lib.TK_ERR_ARG
    assert lib.tk_small_pack(16, 16, 16, 16, 16, 0, None) == _lib.TK_ERR_ARG
    args = [16, 16, 1, 32, 4, 32, 1, 1, None] + [16] * 10 + [1e-5, 1e-5, 1e-5, 1.0, None]
    assert lib.tk_small_forward_packed(*args) == _lib.TK_ERR_ARG


@pytest.mark.gpu
def test_layers_share_the_whole_forward_fragments():
    """Width 128 with ffn_dim 128: what the narrow kernels are given of the stacked fragments is the
    fragment order of that layer's own weights (as the ffn_dim-256 model packs them one by one)."""
    torch.manual_seed(83)
    model = tkmi.OptimizedTransformer(tkmi.TransformerConfig(2, 200, 128, 4, 128, 3, True)).to(DEV).eval()
    built, native = model._weights(), model._native_model()
    packed = model._stacked["packed"]
    for i, lw in enumerate(built):
        for name in ("w_qkv", "w_o", "w_1", "w_2"):
            w = getattr(lw, name)
            assert torch.equal(model._stacked[name][i], w)
            at = (getattr(native.layers[i], name + "_packed") - packed.data_ptr()) // 2
            want = w.view(-1, 32, 8, 2, 8).permute(0, 2, 3, 1, 4)  # block, fragment, half, row, 8 columns
            assert torch.equal(packed[at:at + w.numel()], want.flatten())
