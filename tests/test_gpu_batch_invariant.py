"""Operators asked for batch invariance: a row's (sequence's) bits are the same alone, where the default
call splits its sums over the waves of a workgroup, and in a batch that fills the chip, where it does not."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded
from tkmi import _lib, ops

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("epi", ["bias", "gelu", "resid", "add_ln"])
def test_rows_of_a_gemm(epi):
    m, n, k = 9000, 512, 1024
    a = seeded(m, k, seed=1).half().to(DEV)
    w = (seeded(n, k, seed=2) / k ** 0.5).half().to(DEV)
    b = seeded(n, seed=3).to(DEV)
    resid = seeded(m, n, seed=4).to(DEV)

    def call(lo, hi, **kw):
        if epi in ("bias", "gelu"):
            return ops.linear(a[lo:hi], w, b, gelu=epi == "gelu", **kw)
        if epi == "resid":
            return ops.linear_residual(a[lo:hi], w, b, resid[lo:hi], **kw)
        s = torch.empty(hi - lo, n, device=DEV)
        h = ops.linear_add_ln(a[lo:hi], w, b, resid[lo:hi], b, b, 1e-5, sum_out=s, **kw)
        return torch.cat([s, h.float()], 1)

    whole = call(0, m, batch_invariant=True)
    assert torch.equal(whole, call(0, m))  # past the split's range
    for lo, hi in ((0, 1), (100, 164), (64, 600)):
        assert torch.equal(call(lo, hi, batch_invariant=True), whole[lo:hi])
    assert not torch.equal(call(100, 164), whole[100:164])  # the default splits K here


@pytest.mark.gpu
@pytest.mark.parametrize("masked", [False, True], ids=["dense", "masked"])
@pytest.mark.parametrize("causal", [True, False], ids=["causal", "full"])
@pytest.mark.parametrize("hd", [32, 64, 128, 256])
def test_sequences_of_an_attention(hd, causal, masked):
    b, h, s = 40, 4, 300
    q, k, v = seeded(b, s, 3, h, hd, seed=hd).half().to(DEV).permute(2, 0, 3, 1, 4).unbind(0)
    valid = None
    if masked:
        valid = torch.rand(b, s, generator=torch.Generator().manual_seed(6)) < 0.8
        valid[:, 0] = True
        valid[3, 70:] = False
        valid = valid.to(DEV)

    def call(lo, hi, **kw):
        return ops.flash_attention(q[lo:hi], k[lo:hi], v[lo:hi], hd ** -0.5, causal,
                                   key_valid=None if valid is None else valid[lo:hi], **kw)

    whole = call(0, b, batch_invariant=True)
    assert torch.equal(whole, call(0, b))  # past the key split's range
    for i in (0, 3, b - 1):
        assert torch.equal(call(i, i + 1, batch_invariant=True)[0], whole[i])
    assert not torch.equal(call(3, 4)[0], whole[3])  # the default splits the keys here


@pytest.mark.gpu
@pytest.mark.parametrize("batch,heads", [(2, 12), (2, 16), (4, 12)])
def test_fused_qkv_attention_is_the_invariant_pair(batch, heads):
    """From d_model 768 on a default tk_gemm may split K, which the fused kernel does not."""
    d = heads * 64
    h = seeded(batch * 64, d, seed=8).half().to(DEV)
    w = (seeded(3 * d, d, seed=9) / d ** 0.5).half().to(DEV)
    b = seeded(3 * d, seed=10).to(DEV)
    qkv = ops.linear(h, w, b, batch_invariant=True).view(batch, 64, 3, heads, 64).permute(2, 0, 3, 1, 4)
    want = ops.flash_attention(*qkv.unbind(0), 0.125, True, batch_invariant=True)
    assert torch.equal(ops.qkv_attention(h, w, b, batch, 64, heads, 64, 0.125, True).view(batch, 64, d), want)


def test_bad_calls_are_refused():
    lib = _lib.load()
    st = _lib.strides3((1, 1, 1))
    assert lib.tk_gemm_invariant(None, 8, None, 8, None, None, 0, None, 8, 1, 8, 8, 0, None, 0, None) == _lib.TK_ERR_ARG
    assert lib.tk_gemm_bias_add_ln_invariant(None, 8, None, 8, None, None, None, None, None, None, 0, 1, 128, 8, 1e-5,
                                             None, 0, None) == _lib.TK_ERR_ARG
    assert lib.tk_flash_attn_fwd_invariant(None, None, None, None, 1, 1, 1, 16, st, st, st, st, 1.0, 0, None, 0,
                                           None) == _lib.TK_ERR_ARG
