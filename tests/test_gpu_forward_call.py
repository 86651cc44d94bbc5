"""tk_forward (the layer loop as one call) against the same launches issued one by one."""

from __future__ import annotations

import copy
import ctypes

import pytest
import torch

import tkmi
from tkmi import _lib, ops

DEV = "cuda:0"

# B, S, D, H, F, L, causal: fused and split norms, fused QKV + attention, padded head dims, odd sizes
SHAPES = [
    (3, 77, 256, 4, 512, 2, True),
    (2, 64, 512, 8, 1024, 2, False),
    (2, 130, 384, 12, 200, 3, True),
    (5, 33, 240, 6, 120, 1, False),
    (1, 1, 128, 2, 200, 2, True),
]


def _separate(model, x, mask):
    """The forward of a model as the single operators give it."""
    b, s, d = x.shape
    nh, hd = model.num_heads, model.head_dim_padded
    st = model.settings
    fuse = st.fused_norm and d <= st.fused_norm_max_d and ops.gemm_ln_supported(d)
    fused_qa = mask is None and st.qkv_attention and hd == model.head_dim and ops.qkv_attention_supported(b, s, nh, hd)
    built, fin = model._weights(), model._final
    rows = None if mask is None else mask.reshape(-1)
    resid = x.reshape(b * s, d)
    h = ops.ln_fwd(resid, built[0].n1_w, built[0].n1_b, built[0].n1_eps, torch.float16)
    for i, lw in enumerate(built):
        if fused_qa:
            ctx = ops.qkv_attention(h, lw.w_qkv, lw.b_qkv, b, s, nh, hd, model.attn_scale, model.config.causal)
        else:
            qkv = ops.linear(h, lw.w_qkv, lw.b_qkv).view(b, s, 3, nh, hd).permute(2, 0, 3, 1, 4)
            ctx = ops.flash_attention(*qkv.unbind(0), model.attn_scale, model.config.causal, key_valid=mask)
        ctx = ctx.view(b * s, nh * hd)
        last = i + 1 == len(built)
        nw, nb, ne = fin if last else (built[i + 1].n1_w, built[i + 1].n1_b, built[i + 1].n1_eps)
        dt = torch.float32 if last else torch.float16
        if fuse:
            r2 = torch.empty_like(resid)
            h = ops.linear_add_ln(ctx, lw.w_o, lw.b_o, resid, lw.n2_w, lw.n2_b, lw.n2_eps, sum_out=r2,
                                  row_valid=rows)
            u = ops.linear(h, lw.w_1, lw.b_1, gelu=True)
            mode = ops.TK_ROWS_ZERO_ALL if last else ops.TK_ROWS_ZERO
            r3 = torch.empty_like(resid)
            h = ops.linear_add_ln(u, lw.w_2, lw.b_2, r2, nw, nb, ne, dt, sum_out=r3, row_valid=rows, row_mode=mode)
            resid = r3
        else:
            resid = ops.linear_residual(ctx, lw.w_o, lw.b_o, resid, row_valid=rows)
            h = ops.ln_fwd(resid, lw.n2_w, lw.n2_b, lw.n2_eps, torch.float16)
            u = ops.linear(h, lw.w_1, lw.b_1, gelu=True)
            resid = ops.linear_residual(u, lw.w_2, lw.b_2, resid, row_valid=rows, row_mode=ops.TK_ROWS_ZERO)
            h = ops.ln_fwd(resid, nw, nb, ne, dt, row_valid=rows if last else None)
    return h.view(b, s, d)


def _model_and_input(shape):
    torch.manual_seed(71)
    model = tkmi.OptimizedTransformer(tkmi.TransformerConfig(*shape),
                                      tkmi.OptimizerSettings(small_forward=False)).to(DEV).eval()
    gen = torch.Generator().manual_seed(72)
    x = torch.randn(shape[0], shape[1], shape[2], generator=gen).to(DEV)
    mask = torch.rand(shape[0], shape[1], generator=gen) < 0.7
    mask[:, 0] = True
    return model, x, mask.to(DEV)


@pytest.mark.gpu
@pytest.mark.parametrize("padded", [False, True], ids=["dense", "padded"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "b{}s{}d{}h{}f{}l{}".format(*s[:6]))
def test_one_call_matches_separate_launches(shape, padded):
    model, x, mask = _model_and_input(shape)
    if not padded or bool(mask.all()):
        mask = None
    with torch.inference_mode():
        got = model(x, mask)
        want = _separate(model, x, mask)
        with ops.kernel_timer() as rec:  # the same launches, one call each
            stepped = model(x, mask)
        torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert torch.equal(got, stepped)
    assert rec[0][0] == "ln_in" and rec[-1][0] in ("ln_final", "ffn_down_ln")


# Width 128: ln_qkv and block_tail in the place of the launches above; F = 128 and
# wider, rows one off the 64-row trips, more trips than workgroups.
@pytest.mark.gpu
@pytest.mark.parametrize("padded", [False, True], ids=["dense", "padded"])
@pytest.mark.parametrize("shape", [(1, 1, 128, 4, 128, 1, True), (3, 171, 128, 2, 128, 3, True),
                                   (1, 129, 128, 4, 384, 2, False), (7, 1300, 128, 1, 256, 1, True),
                                   (37, 1000, 128, 8, 128, 2, True)],
                         ids=lambda s: "b{}s{}h{}f{}l{}".format(s[0], s[1], s[3], s[4], s[5]))
def test_narrow_blocks_match_separate_launches(shape, padded):
    """The same arithmetic with other roundings only in the LayerNorm statistics
    (merged means instead of one sum): fp32 reassociation, which moves fp16
    roundings of h by at most one unit, as between the whole-forward kernel and the
    layer path (1e-3, measured 6.3e-4 over up to 4 layers)."""
    model, x, mask = _model_and_input(shape)
    if not padded or bool(mask.all()):
        mask = None
    with torch.inference_mode():
        with ops.kernel_timer() as rec:
            got = model(x, mask)
        want = _separate(model, x, mask)
        again = model(x, mask)
        torch.cuda.synchronize()
    assert [r[0] for r in rec][:3] == ["ln_qkv", "flash_attn", "block_tail"] and len(rec) == 3 * shape[5]
    assert torch.equal(got, again)
    assert (got - want).abs().max().item() <= 1e-3
    if mask is not None:
        assert bool((got[~mask] == 0).all())


@pytest.mark.gpu
def test_workspace_is_not_overrun():
    model, x, _ = _model_and_input(SHAPES[2])
    b, s, _ = x.shape
    lib = _lib.load()
    with torch.inference_mode():
        want = model(x)
        ref = ctypes.byref(model._native_model())
        size = lib.tk_forward_workspace(ref, b, s, 1, 0)
        buf = torch.full((size + 1024,), 0x5A, dtype=torch.uint8, device=DEV)
        ws = buf.data_ptr() + 256
        out = torch.empty_like(x)
        stream = torch.cuda.current_stream().cuda_stream
        args = (ref, x.data_ptr(), out.data_ptr(), b, s, None)
        _lib.call("tk_forward", *args, ws, size, 0, 0, -1, stream)
        assert lib.tk_forward(*args, ws, size - 1, 0, 0, -1, stream) == _lib.TK_ERR_ARG
        torch.cuda.synchronize()
    assert torch.equal(out, want)
    assert bool((buf[:256] == 0x5A).all()) and bool((buf[256 + size:] == 0x5A).all())


@pytest.mark.gpu
def test_copied_model_uses_its_own_weights():
    model, x, _ = _model_and_input(SHAPES[2])
    with torch.inference_mode():
        want = model(x)
    twin = copy.deepcopy(model)
    assert twin._native is None
    with torch.inference_mode():
        got = twin(x)
        assert torch.equal(got, want)
        assert twin._native.layers[0].w_qkv == twin._weights()[0].w_qkv.data_ptr()
        assert twin._native.layers[0].w_qkv != model._native.layers[0].w_qkv


@pytest.mark.gpu
@pytest.mark.parametrize("warm,captured", [(64, 200), (200, 64)], ids=["whole_then_layers", "layers_then_whole"])
def test_capture_after_a_warm_up_of_the_other_path(warm, captured):
    """Width 128: the capture holds launches of the forward only, so an eager call before the
    first replay, and each replay, give what a model of the same weights gives eagerly."""
    torch.manual_seed(73)
    cfg = tkmi.TransformerConfig(2, 200, 128, 4, 128, 2, True)
    model = tkmi.OptimizedTransformer(cfg).to(DEV).eval()
    fresh = copy.deepcopy(model)
    gen = torch.Generator().manual_seed(74)
    x = torch.randn(2, captured, 128, generator=gen).to(DEV)
    with torch.inference_mode():
        want = fresh(x)
        model(torch.randn(2, warm, 128, generator=gen).to(DEV))
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(x)
        assert torch.equal(model(x), want)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            assert torch.equal(model(x), want)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(6, 64, 128, 2, 256, 2, True), (6, 64, 768, 12, 768, 1, False)],
                         ids=["narrow", "wide"])
def test_batch_invariant_bits_at_one_key_tile(shape):
    """S = 64, head_dim 64: batches that the fused QKV + attention kernel takes (even ones) and that it does not."""
    torch.manual_seed(75)
    model = tkmi.OptimizedTransformer(tkmi.TransformerConfig(*shape),
                                      tkmi.OptimizerSettings(batch_invariant=True)).to(DEV).eval()
    x = torch.randn(shape[:3], generator=torch.Generator().manual_seed(76)).to(DEV)
    with torch.inference_mode():
        whole = model(x)
        for n in (1, 2, 3):
            assert torch.equal(whole, torch.cat([model(x[i:i + n]) for i in range(0, 6, n)])), n


def test_bad_calls_are_refused():
    lib = _lib.load()
    assert lib.tk_forward_workspace(None, 1, 1, 1, 0) == _lib.TK_ERR_ARG
    layers = (_lib.Layer * 1)()
    model = _lib.Model(d_model=256, heads=4, head_dim=64, ffn_dim=512, num_layers=1, layers=layers, nf_w=256, nf_b=256)
    ref = ctypes.byref(model)
    size = lib.tk_forward_workspace(ref, 2, 10, 1, 0)
    # resid fp32, h and ctx fp16, max(q|k|v, hidden) fp16, each rounded up to 256 bytes
    assert size == 20 * 256 * 4 + 2 * 20 * 256 * 2 + 20 * 3 * 256 * 2
    assert lib.tk_forward_steps(ref, 2, 10, 1, 0) == 8
    assert lib.tk_forward_steps(ref, 2, 10, 1, _lib.TK_FWD_FUSED_NORM) == 6
    assert lib.tk_forward_steps(ref, 2, 64, 1, _lib.TK_FWD_QKV_ATTENTION) == 7
    assert lib.tk_forward_step_name(ref, 2, 10, 1, 0, 7) == b"ln_final"
    assert lib.tk_forward_step_name(ref, 2, 10, 1, 0, 8) is None
    bad = [
        (None, 256, 256, 2, 10, None, 256, size, 0, 0, -1, None),
        (ref, None, 256, 2, 10, None, 256, size, 0, 0, -1, None),
        (ref, 256, 256, 2, 10, None, 256, size - 1, 0, 0, -1, None),
        (ref, 256, 256, 2, 10, None, 264, size, 0, 0, -1, None),
        (ref, 256, 256, 2, 10, None, 256, size, 0, 0, 9, None),
        (ref, 256, 256, -1, 10, None, 256, size, 0, 0, -1, None),
    ]
    for args in bad:
        assert lib.tk_forward(*args) == _lib.TK_ERR_ARG
        assert lib.tk_last_error_string()
