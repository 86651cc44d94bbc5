"""GEMM launches of few tiles, whose K loop is split over groups of a workgroup's waves."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded
from oracle import baseline as ob
import tkmi
from tkmi import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

SHAPES = {
    "one_row": (1, 72, 768),             # 32 x 32 tiles, four groups of three K-tiles
    "t32_most": (250, 1024, 1024),       # 256 of them
    "t32_odd": (33, 328, 1280),
    "wide_first": (257, 1024, 768),      # 32 x 64 tiles, four groups
    "wide_most": (500, 1032, 1024),
    "wide_two_groups": (100, 520, 896),  # K an odd multiple of 128
    "small_first": (513, 1032, 768),     # 64 x 64 tiles, two groups
    "small_most": (1000, 1016, 1152),
    "odd_k": (100, 520, 960),            # K an odd multiple of 64: one group
}


@pytest.mark.parametrize("epi", ["bias", "gelu", "resid", "resid_rows"])
@pytest.mark.parametrize("shape", SHAPES.values(), ids=SHAPES.keys())
def test_split_k_tiles(shape, epi):
    m, n, k = shape
    a = seeded(m, k, seed=61).half()
    w = (seeded(n, k, seed=62) / k ** 0.5).half()
    bias = seeded(n, seed=63) * 0.1
    ref = a.float() @ w.float().T + bias
    guard = 7.0
    if epi in ("bias", "gelu"):
        buf = torch.full((m + 2, n + 16), guard, dtype=torch.float16, device=DEV)
        ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), gelu=epi == "gelu", out=buf[:m, :n])
        want = (ob.gelu_ref(ref) if epi == "gelu" else ref).half().float()
        tol = dict(atol=1e-3, rtol=1e-3)  # one fp16 rounding (4.9e-4 relative)
    else:
        resid = seeded(m, n, seed=64)
        buf = torch.full((m + 2, n + 16), guard, dtype=torch.float32, device=DEV)
        view = buf[:m, :n]
        view.copy_(resid)  # in place: the residual is the output
        valid = None
        want = resid + ref
        if epi == "resid_rows":
            valid = torch.rand(m, generator=torch.Generator().manual_seed(65)) < 0.7
            want = torch.where(valid[:, None], want, resid)
        ops.linear_residual(a.to(DEV), w.to(DEV), bias.to(DEV), view, out=view,
                            row_valid=None if valid is None else valid.to(DEV))
        tol = dict(atol=5e-5, rtol=1e-5)  # fp32 sums in another order
    got = buf.cpu()
    torch.testing.assert_close(got[:m, :n].float(), want, **tol)
    assert bool((got[m:] == guard).all()) and bool((got[:m, n:] == guard).all())


def test_batch_invariant_model():
    """batch_invariant: sequences alone (few tiles, split K) equal themselves in a batch (none)."""
    torch.manual_seed(5)
    cfg = tkmi.TransformerConfig(40, 64, 768, 12, 1536, 1, False)
    settings = tkmi.OptimizerSettings(batch_invariant=True)
    model = tkmi.OptimizedTransformer(cfg, settings).to(DEV).eval()
    x = seeded(40, 64, 768, seed=6).to(DEV)
    with torch.inference_mode():
        whole, alone = model(x), torch.cat([model(x[i:i + 1]) for i in range(40)])
    assert torch.equal(whole, alone)
