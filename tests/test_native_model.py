"""The weights' addresses and the settings that a model hands to tk_forward: host code only, no launch."""

import weakref
from dataclasses import replace

import pytest
import torch

import tkmi


def _model(d_model=256, heads=4, ffn=512, layers=2):
    torch.manual_seed(7)
    return tkmi.OptimizedTransformer(tkmi.TransformerConfig(2, 16, d_model, heads, ffn, layers, True)).eval()


def test_changed_settings_reach_the_next_call():
    """The separate launches read the causal flag and the scale at every forward; so does the one call."""
    model = _model()
    native = model._native_model()
    assert model._native_model() is native
    assert (native.causal, native.scale) == (1, 0.125)
    model.config = replace(model.config, causal=False)
    assert model._native_model().causal == 0
    model.attn_scale = 0.5
    assert model._native_model().scale == 0.5


@pytest.mark.parametrize("ffn", [128, 256])
def test_narrow_fragments_are_packed_with_the_weights(ffn):
    """Every form of the weights exists once _weights() has run, whichever path a forward takes: a
    capture of a path that an earlier forward did not take records no packing."""
    model = _model(d_model=128, ffn=ffn)
    built = model._weights()
    n, k = built[0].w_qkv.shape
    want = built[0].w_qkv.view(n // 32, 32, 8, 2, 8).permute(0, 2, 3, 1, 4)  # block, fragment, half, row, 8 columns
    assert torch.equal(built[0].w_qkv_packed.flatten(), want.flatten())
    held = [getattr(lw, name) for lw in built for name in ("w_qkv_packed", "w_o_packed", "w_1_packed", "w_2_packed")]
    native = model._native_model()
    assert all(getattr(lw, name) is t for (lw, name), t in zip(
        [(lw, name) for lw in built for name in ("w_qkv_packed", "w_o_packed", "w_1_packed", "w_2_packed")], held))
    assert native.layers[1].w_2_packed == held[7].data_ptr()
    assert _model()._weights()[0].w_qkv_packed is None  # width 256: no kernel reads them


def test_addresses_outlive_a_repacking_by_another_thread():
    """The table holds the tensors whose addresses it gives away: another thread that packs changed
    weights drops the model's own references, while this one has not launched yet."""
    model = _model(d_model=128)
    native = model._native_model()
    refs = [weakref.ref(t) for lw in model._weights() for t in vars(lw).values() if isinstance(t, torch.Tensor)]
    refs += [weakref.ref(t) for t in model._final[:2]]
    with torch.no_grad():
        for p in model.parameters():
            p.add_(1.0)
    model._weights()
    assert native.layers[0].w_qkv != model._native_model().layers[0].w_qkv
    assert all(r() is not None for r in refs)
    del native
    assert all(r() is None for r in refs)
