"""The weights' addresses and the settings that a model hands to tk_forward: host code only, no launch."""

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
