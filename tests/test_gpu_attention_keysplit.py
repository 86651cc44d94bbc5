"""Attention launches with few query blocks: the key-split kernel, its edges and its rule."""

from __future__ import annotations

import pytest
import torch

import tkmi
from oracle import baseline as ob
from tkmi import ops

from conftest import or_rule_violations, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _qkv(b, h, s, hd, seed):
    return (seeded(b, s, 3, h, hd, seed=seed).half()).permute(2, 0, 3, 1, 4).unbind(0)


# One key past a tile, fewer tiles than waves, tiles of four and eight waves that end
# unevenly, 512 blocks of 32 rows (the last launch inside the rule at most head dims) and
# more (for head_dim 256 that is the pipelined generic kernel).
@pytest.mark.parametrize("causal", [True, False], ids=["causal", "full"])
@pytest.mark.parametrize("hd", [32, 64, 128, 256])
@pytest.mark.parametrize("b,h,s", [(1, 1, 65), (2, 3, 127), (1, 5, 200), (1, 2, 513), (1, 2, 1057), (2, 1, 1990),
                                   (16, 8, 128), (16, 8, 129), (13, 3, 385), (20, 4, 300)])
def test_edges(b, h, s, hd, causal):
    q, k, v = _qkv(b, h, s, hd, seed=s + hd)
    out = ops.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), hd ** -0.5, causal)
    bad, err = or_rule_violations(out, ob.attention_ref(q, k, v, hd ** -0.5, causal))
    assert bad == 0, err


@pytest.mark.parametrize("causal", [True, False], ids=["causal", "full"])
@pytest.mark.parametrize("hd,s,h", [(32, 300, 2), (64, 1090, 2), (128, 300, 2), (256, 300, 2), (256, 300, 18)],
                         ids=["d32", "d64", "d128", "d256", "d256_past_rule"])
def test_key_mask(hd, s, h, causal):
    """Padded tails, whole tiles without a valid key, holes; rows without any valid key
    come out non-finite, as from the other kernels."""
    b = 3
    q, k, v = _qkv(b, h, s, hd, seed=s)
    valid = torch.ones(b, s, dtype=torch.bool)
    valid[0, s - 90:] = False
    valid[1, :130] = False
    valid[2] = torch.rand(s, generator=torch.Generator().manual_seed(3)) > 0.4
    valid[2, 0] = True
    out = ops.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), hd ** -0.5, causal, key_valid=valid.to(DEV)).cpu()
    scores = torch.matmul(q.float(), k.float().transpose(-2, -1).contiguous()) * hd ** -0.5
    gone = ~valid[:, None, None, :].expand(b, h, s, s).clone()
    if causal:
        gone |= torch.ones(s, s, dtype=torch.bool).triu(1)
    ref = torch.matmul(torch.softmax(scores.masked_fill(gone, float("-inf")), -1), v.float())
    ref = ref.permute(0, 2, 1, 3).reshape(b, s, h * hd)
    none = gone.all(-1)[:, 0]
    assert not torch.isfinite(out[none]).any()
    bad, err = or_rule_violations(out[~none], ref[~none])
    assert bad == 0, err


@pytest.mark.parametrize("hd", [32, 64, 128, 256])
def test_growing_scores(hd):
    """Row maxima that rise from tile to tile by up to 40 in the exponent, and scores past
    fp16's range: every wave's sums are rescaled and merged at different references."""
    b, h, s = 1, 2, 700
    q, k, v = _qkv(b, h, s, hd, seed=9)
    k = (k.float() * torch.linspace(0.1, 12.0, s)[:, None]).half()
    q = (q.float() * 8).half()
    for causal in (True, False):
        out = ops.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), hd ** -0.5, causal)
        bad, err = or_rule_violations(out, ob.attention_ref(q, k, v, hd ** -0.5, causal))
        assert bad == 0, (causal, err)


@pytest.mark.parametrize("hd,s", [(64, 640), (64, 1300), (128, 1025), (128, 1300)])
def test_asm_loops_still_equal_compiled_steps(hd, s):
    """Launches just past the rule keep the hand-ordered loops: K/V rows 4 MiB apart
    take the compiled steps, bit for bit the same (heads share one K and V, stride 0)."""
    h = 520 // ((s + 31) // 32) + 1
    q = seeded(1, h, s, hd, seed=s).half().to(DEV)
    k, v = (seeded(1, 1, s, hd, seed=s + i).half().to(DEV) for i in (1, 2))
    compact = ops.flash_attention(q, k.expand(1, h, s, hd), v.expand(1, h, s, hd), hd ** -0.5, True)
    rs = 1 << 21
    wide_k, wide_v = (torch.zeros(s, rs, dtype=torch.float16, device=DEV) for _ in range(2))
    wide_k[:, :hd], wide_v[:, :hd] = k[0, 0], v[0, 0]
    kw, vw = (t[:, :hd][None, None].expand(1, h, s, hd) for t in (wide_k, wide_v))
    assert kw.stride(2) == rs
    spread = ops.flash_attention(q, kw, vw, hd ** -0.5, True)
    assert torch.equal(compact, spread)


def test_batch_invariant_model():
    """batch_invariant: a sequence alone (which would split its keys) equals itself in a batch."""
    torch.manual_seed(5)
    cfg = tkmi.TransformerConfig(24, 200, 256, 4, 512, 1, True)
    model = tkmi.OptimizedTransformer(cfg, tkmi.OptimizerSettings(batch_invariant=True)).to(DEV).eval()
    x = seeded(24, 200, 256, seed=6).to(DEV)
    with torch.inference_mode():
        whole, alone = model(x), torch.cat([model(x[i:i + 1]) for i in range(24)])
    assert torch.equal(whole, alone)


# Two workgroups per CU: one key tile too few, B*H off the XCD count, and the first inside each line.
@pytest.mark.parametrize("b,s,hd,causal,masked,split", [
    (128, 128, 128, True, False, False), (128, 128, 128, True, True, True), (170, 96, 128, False, True, False),
    (128, 96, 128, False, False, False), (128, 97, 128, False, False, True), (80, 160, 128, True, False, True),
    (72, 192, 256, False, False, False), (64, 256, 256, False, False, True), (43, 320, 256, False, True, False),
    (72, 192, 256, True, False, False), (73, 193, 256, True, False, True),
    (85, 192, 64, False, False, False), (85, 192, 64, False, True, True), (80, 192, 64, False, False, True),
    (52, 256, 64, True, False, True), (19, 512, 64, False, False, True),
    (170, 192, 32, True, False, False), (170, 192, 32, True, True, True), (168, 192, 32, True, False, True),
    (122, 96, 32, False, False, False)])
def test_rule_past_one_workgroup_per_cu(b, s, hd, causal, masked, split):
    q, k, v = (t.to(DEV) for t in _qkv(b, 1, s, hd, seed=s + hd))
    valid = None
    if masked:
        valid = torch.arange(s, device=DEV)[None] < torch.linspace(s - 40, s, b, device=DEV).long()[:, None]
    out = ops.flash_attention(q, k, v, hd ** -0.5, causal, key_valid=valid)
    other = ops.flash_attention(q, k, v, hd ** -0.5, causal, key_valid=valid, batch_invariant=True)
    assert torch.equal(out, other) != split
    few = slice(0, 4)
    qf, kf, vf = (t[few].cpu().float() for t in (q, k, v))
    if not masked:
        ref = ob.attention_ref(qf, kf, vf, hd ** -0.5, causal)
    else:
        gone = ~valid[few].cpu()[:, None, None, :].expand(4, 1, s, s).clone()
        if causal:
            gone |= torch.ones(s, s, dtype=torch.bool).triu(1)
        scores = torch.matmul(qf, kf.transpose(-2, -1).contiguous()) * hd ** -0.5
        ref = torch.matmul(scores.masked_fill(gone, float("-inf")).softmax(-1), vf)[:, 0]
    bad, err = or_rule_violations(out[few], ref)
    assert bad == 0, err
