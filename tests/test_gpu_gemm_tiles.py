"""Every tile of the GEMM dispatch at ragged sizes, against the fp32 product.

The outputs are views of wider buffers, so a store outside the M x N block
shows as a changed guard value.
"""

from __future__ import annotations

import pytest
import torch

from conftest import seeded
from oracle import baseline as ob
from tkmi import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

SHAPES = {
    "small_one_row": (1, 72, 64),            # 64 x 64 tiles
    "small": (65, 1032, 192),
    "tall_three_stages": (520, 2056, 192),   # 128 x 64, two K-tiles in flight
    "tall_two_stages": (777, 3080, 192),
    "mid_three_stages": (777, 3080, 2048),   # 128 x 128, 8 waves
    "mid_long_k": (1500, 4104, 2048),
    "wide_one_to_a_row": (20993, 256, 2048),  # 128 x 256, last tile row one row
    "wide_two_to_a_row": (14493, 512, 2048),
    "tall_short_k": (1500, 3976, 192),
    "mid": (1500, 4104, 576),
    "two_stage_256": (4000, 2824, 576),      # 256 x 256, K an odd multiple of 64
    "pingpong_one_round": (4001, 3336, 512),  # last tile row 161 rows, last column 8 columns
    "pingpong_smallest": (4353, 3080, 512),  # one row and 8 columns past whole tiles
    "pingpong_persistent": (8200, 3592, 768),
    "pingpong_short_k": (8200, 3592, 256),   # (residual epilogues: 128 x 128)
}


@pytest.mark.parametrize("epi", ["bias", "gelu", "resid", "resid_rows"])
@pytest.mark.parametrize("shape", SHAPES.values(), ids=SHAPES.keys())
def test_gemm_tiles_at_ragged_sizes(shape, epi):
    m, n, k = shape
    a = seeded(m, k, seed=51).half()
    w = (seeded(n, k, seed=52) / k ** 0.5).half()
    bias = seeded(n, seed=53) * 0.1
    ref = a.float() @ w.float().T + bias
    guard = 7.0
    if epi in ("bias", "gelu"):
        buf = torch.full((m + 2, n + 16), guard, dtype=torch.float16, device=DEV)
        ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), gelu=epi == "gelu", out=buf[:m, :n])
        want = (ob.gelu_ref(ref) if epi == "gelu" else ref).half().float()
        tol = dict(atol=1e-3, rtol=1e-3)  # one fp16 rounding (4.9e-4 relative)
    else:
        resid = seeded(m, n, seed=54)
        buf = torch.full((m + 2, n + 16), guard, dtype=torch.float32, device=DEV)
        view = buf[:m, :n]
        view.copy_(resid)  # in place: the residual is the output
        valid = None
        want = resid + ref
        if epi == "resid_rows":
            valid = torch.rand(m, generator=torch.Generator().manual_seed(55)) < 0.7
            want = torch.where(valid[:, None], want, resid)
        ops.linear_residual(a.to(DEV), w.to(DEV), bias.to(DEV), view, out=view,
                            row_valid=None if valid is None else valid.to(DEV))
        tol = dict(atol=5e-5, rtol=1e-5)  # fp32 sums in another order
    got = buf.cpu()
    torch.testing.assert_close(got[:m, :n].float(), want, **tol)
    assert bool((got[m:] == guard).all()) and bool((got[:m, n:] == guard).all())
