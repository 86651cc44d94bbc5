"""The schedule that tk_forward picks, read from its step names: host code only, no launch."""

import ctypes

import pytest

from tkmi import _lib


def _steps(d_model=128, b_1=0x1000, packed=0x1000, layers=2, flags=_lib.TK_FWD_FUSED_NORM):
    """Step names of a forward of a model whose addresses are made up (the schedule reads none)."""
    lib = _lib.load()
    rows = (_lib.Layer * layers)()
    for row in rows:
        for name, ctype in _lib.Layer._fields_:
            if not name.endswith("_eps"):
                setattr(row, name, packed if name.endswith("_packed") else 0x1000)
    rows[-1].b_1 = b_1
    model = _lib.Model(d_model=d_model, heads=4, head_dim=d_model // 4, ffn_dim=d_model, num_layers=layers,
                       layers=rows, nf_w=0x1000, nf_b=0x1000, nf_eps=1e-5, scale=1.0, causal=1)
    ref = ctypes.byref(model)
    n = lib.tk_forward_steps(ref, 3, 100, 1, flags)
    return [lib.tk_forward_step_name(ref, 3, 100, 1, flags, i).decode() for i in range(n)]


def test_width_128_runs_the_narrow_kernels():
    assert _steps() == ["ln_qkv", "flash_attn", "block_tail", "qkv", "flash_attn", "block_tail"]


@pytest.mark.parametrize("kw", [dict(b_1=0x1004), dict(b_1=0x1008), dict(packed=None)])
def test_width_128_that_the_narrow_kernels_do_not_take(kw):
    """A bias off a 16-byte boundary, which tk_narrow_tail refuses, or no packed weights: separate launches."""
    layer = ["qkv", "flash_attn", "out_proj_ln", "ffn_up_gelu", "ffn_down_ln"]
    assert _steps(**kw) == ["ln_in"] + 2 * layer


def _names(batch, flags):
    """Step names at S = 64, d_model 128 in 2 heads of 64, ffn 256, which the whole-forward kernel does not take."""
    lib = _lib.load()
    rows = (_lib.Layer * 2)()
    for row in rows:
        for name, _ in _lib.Layer._fields_:
            if not name.endswith("_eps"):
                setattr(row, name, 0x1000)
    model = _lib.Model(d_model=128, heads=2, head_dim=64, ffn_dim=256, num_layers=2, layers=rows, nf_w=0x1000,
                       nf_b=0x1000, nf_eps=1e-5, scale=1.0, causal=1)
    ref = ctypes.byref(model)
    return [lib.tk_forward_step_name(ref, batch, 64, 1, flags, i)
            for i in range(lib.tk_forward_steps(ref, batch, 64, 1, flags))]


def test_batch_invariant_schedule_is_that_of_every_batch():
    """The fused QKV + attention kernel takes even batches only, and at width 128 the launches that it
    replaces are others than those of the odd ones, with other roundings."""
    flags = _lib.TK_FWD_FUSED_NORM | _lib.TK_FWD_QKV_ATTENTION
    assert _names(1, flags) != _names(2, flags)
    flags |= _lib.TK_FWD_BATCH_INVARIANT
    assert all(_names(b, flags) == _names(1, flags) for b in range(2, 9))
