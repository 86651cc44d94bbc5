"""16-bit models: the input and output conversions inside the first and last LayerNorm."""

from __future__ import annotations

import ctypes

import pytest
import torch

from conftest import seeded
import tkmi
from tkmi import _lib

DEV = "cuda:0"


# Vector and element-wise LayerNorm rows (width 330: not a multiple of 4), one row, the
# widths of several register counts; the fp32 model of the same (rounded) values is exact here:
# the conversions round where .float() and .to() did.
@pytest.mark.gpu
@pytest.mark.parametrize("padded", [False, True], ids=["dense", "padded"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("shape", [(1, 1, 512, 8, 512, 1), (3, 77, 330, 5, 200, 2), (2, 64, 512, 8, 1024, 1),
                                   (2, 100, 1024, 16, 1024, 2), (1, 33, 2048, 16, 512, 1)],
                         ids=lambda s: "b{}s{}d{}".format(*s[:3]))
def test_same_bits_as_separate_conversions(shape, dtype, padded):
    torch.manual_seed(3)
    cfg = tkmi.TransformerConfig(*shape, True)
    model = tkmi.OptimizedTransformer(cfg).to(DEV).eval().to(dtype)
    b, s, d = shape[:3]
    x = seeded(b, s, d, seed=4).to(DEV).to(dtype)
    keep = x.clone()
    mask = None
    if padded:
        mask = torch.arange(s, device=DEV)[None] < torch.tensor([max(1, s - 20 * i) for i in range(b)], device=DEV)[:, None]
        if b == 1:
            mask = mask & (torch.arange(s, device=DEV) < max(1, s - 5))
    with torch.inference_mode():
        got = model(x, mask)
        want = model(x.float(), mask).to(dtype)
    assert got.dtype == dtype
    assert torch.equal(got, want)
    assert torch.equal(x, keep)


def test_flags_are_checked():
    layers = (_lib.Layer * 1)()
    model = _lib.Model(d_model=256, heads=4, head_dim=64, ffn_dim=512, num_layers=1, layers=layers, nf_w=256, nf_b=256)
    lib = _lib.load()
    ref = ctypes.byref(model)
    size = lib.tk_forward_workspace(ref, 2, 10, 1, 0)
    args = (ref, 256, 256, 2, 10, None, 256, size)
    both = _lib.TK_FWD_IO_F16 | _lib.TK_FWD_IO_BF16
    assert lib.tk_forward(*args, both, 0, 0, None) == _lib.TK_ERR_ARG
    assert lib.tk_forward(*args, 32, 0, 0, None) == _lib.TK_ERR_ARG
    fused = _lib.TK_FWD_IO_F16 | _lib.TK_FWD_FUSED_NORM
    assert lib.tk_forward(*args, fused, 0, 0, None) == _lib.TK_ERR_UNSUPPORTED
