"""Non-causal attention through the generated steady-state loops, and key masks whose tail is skipped.

Every launch here is small enough for the default call to split its keys over a
workgroup's waves (tests/test_gpu_attention_keysplit.py); batch_invariant rules
that out, so that these reach the loops and the trimmed tile counts.
"""

from __future__ import annotations

import pytest
import torch

from conftest import or_rule_violations, seeded
from tkmi import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _reference(q, k, v, causal, valid):
    """fp64 softmax of the fp16 operands; rows without a valid key are NaN."""
    s = q.shape[2]
    scores = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * q.shape[3] ** -0.5
    ok = torch.ones(s, s, dtype=torch.bool).tril() if causal else torch.ones(s, s, dtype=torch.bool)
    if valid is not None:
        ok = ok & valid[:, None, None, :]
    p = torch.softmax(scores.masked_fill(~ok, float("-inf")), -1)
    return torch.matmul(p, v.double()).transpose(1, 2).flatten(2)


def _check(q, k, v, causal, valid=None):
    b, h, s, hd = q.shape
    got = ops.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), hd ** -0.5, causal,
                              key_valid=None if valid is None else valid.to(DEV), batch_invariant=True).cpu()
    want = _reference(q, k, v, causal, valid)
    seen = torch.isfinite(want).all(-1)
    bad, err = or_rule_violations(got[seen], want[seen].float())
    assert bad == 0, err
    assert not bool(torch.isfinite(got[~seen]).any())


# key tiles: 2 (no loop step) .. 21, whole and one key off; head_dim 128 loops in groups of 4, 64 of 2
@pytest.mark.parametrize("s", [129, 191, 256, 383, 384, 449, 512, 833, 1344])
@pytest.mark.parametrize("hd", [64, 128])
def test_full_attention_over_tile_counts(s, hd):
    q, k, v = (seeded(2, 2, s, hd, dtype=torch.float16, seed=60 + i) for i in range(3))
    _check(q, k, v, False)
    # scores rising along the keys: every tile moves the running max
    ramp = torch.arange(s, dtype=torch.float32)[:, None] * 0.05
    _check(q, (k.float() + ramp * q.float().mean((0, 1, 2)).sign()).half(), v, False)


@pytest.mark.parametrize("masked", [False, True], ids=["dense", "masked"])
@pytest.mark.parametrize("s", [448, 777, 1344])
def test_full_loop_is_bit_identical(s, masked):
    """head_dim 128: the loop does the compiled epochs' arithmetic in their order, also without the causal
    mask.  K/V rows 4 MiB apart put the copies' span past 32-bit offsets, so the same values take the
    compiled epochs."""
    b, h, hd, rs = 2, 1, 128, 1 << 21
    q, k, v = (seeded(b, h, s, hd, dtype=torch.float16, seed=90 + i).to(DEV) for i in range(3))
    valid = None
    if masked:
        valid = torch.rand(b, s, generator=torch.Generator().manual_seed(5)) > 0.3
        valid[1, s - 100:] = False
        valid = valid.to(DEV)
    wide = torch.zeros(2, b, s, rs, dtype=torch.float16, device=DEV)
    wide[0, :, :, :hd], wide[1, :, :, :hd] = k[:, 0], v[:, 0]
    kw, vw = wide[0, :, None, :, :hd], wide[1, :, None, :, :hd]
    compact = ops.flash_attention(q, k, v, hd ** -0.5, False, key_valid=valid, batch_invariant=True)
    spread = ops.flash_attention(q, kw, vw, hd ** -0.5, False, key_valid=valid, batch_invariant=True)
    assert torch.equal(compact, spread)


@pytest.mark.parametrize("pattern", ["tail", "short", "head", "holes", "one_batch_empty"])
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("hd", [32, 64, 128, 256, 80])
def test_key_masks(hd, causal, pattern):
    b, h, s = 3, 2, 777
    q, k, v = (seeded(b, h, s, hd, dtype=torch.float16, seed=70 + i) for i in range(3))
    valid = torch.ones(b, s, dtype=torch.bool)
    if pattern == "tail":  # one key, a whole number of tiles, one key past it
        valid[0, 1:] = False
        valid[1, 512:] = False
        valid[2, 513:] = False
    elif pattern == "short":  # one tile, a key past it, two tiles and a key
        valid[0, 64:] = False
        valid[1, 65:] = False
        valid[2, 129:] = False
    elif pattern == "head":
        valid[:, :200] = False
    elif pattern == "holes":
        valid = torch.rand(b, s, generator=torch.Generator().manual_seed(5)) > 0.3
    else:
        valid[1] = False
    _check(q, k, v, causal, valid)


def test_eight_byte_value_rows_keep_their_path():
    """head_dim 128, V rows 8-byte but not 16-byte aligned: no DMA copy possible."""
    b, h, s, hd = 2, 2, 400, 128
    q, k, v = (seeded(b, h, s, hd, dtype=torch.float16, seed=80 + i) for i in range(3))
    wide = torch.zeros(b, h, s, hd + 4, dtype=torch.float16, device=DEV)
    wide[..., 4:] = v.to(DEV)
    got = ops.flash_attention(q.to(DEV), k.to(DEV), wide[..., 4:], hd ** -0.5, False, batch_invariant=True).cpu()
    bad, err = or_rule_violations(got, _reference(q, k, v, False, None).float())
    assert bad == 0, err


@pytest.mark.parametrize("hd", [16, 32, 64, 128, 256, 80])
@pytest.mark.parametrize("s", [85, 86, 170, 171, 192, 193, 321])
def test_tail_skipping_around_its_line(s, hd):
    """Key masks at lengths with the scan for the last valid key and their neighbours without it,
    in launches of up to as many workgroups as CUs and of more (the scan's other condition);
    batch_invariant launches take it at every batch, with the same bits."""
    h = 96
    valid = torch.ones(3, s, dtype=torch.bool)
    valid[0, 1:] = False
    valid[1, 200:] = False
    q, k, v = (seeded(3, 1, s, hd, dtype=torch.float16, seed=60 + i).expand(3, h, s, hd).to(DEV) for i in range(3))
    want = _reference(*(t[:, :1].cpu() for t in (q, k, v)), False, valid).float()
    whole = ops.flash_attention(q, k, v, hd ** -0.5, False, key_valid=valid.to(DEV), batch_invariant=True)
    for b in (1, 3):
        got = ops.flash_attention(q[:b], k[:b], v[:b], hd ** -0.5, False, key_valid=valid[:b].to(DEV))
        bad, err = or_rule_violations(got[..., -hd:], want[:b])
        assert bad == 0, (b, err)
        got = ops.flash_attention(q[:b], k[:b], v[:b], hd ** -0.5, False, key_valid=valid[:b].to(DEV),
                                  batch_invariant=True)
        assert torch.equal(got, whole[:b])


@pytest.mark.parametrize("b,s", [(65, 513), (89, 513), (90, 513), (65, 300)])
def test_element_loads_around_one_workgroup_per_cu(b, s):
    """Causal head_dim 100: 325 and 445 workgroups (one per CU), 450 and short sequences (two)."""
    q, k, v = (seeded(b, 1, s, 100, dtype=torch.float16, seed=30 + i) for i in range(3))
    got = ops.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), 0.1, True).cpu()
    bad, err = or_rule_violations(got[-3:], _reference(q[-3:], k[-3:], v[-3:], True, None).float())
    assert bad == 0, err
