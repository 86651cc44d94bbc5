"""``OptimizedTransformer``: the reference's drop-in model on MI355X kernels.

Interface (src/optimized.py:85-157,200-232,393-408):
  * ``OptimizedTransformer(config, settings=None)`` subclasses
    ``BaselineTransformer`` so ``state_dict`` keys match the baseline's and the
    harness's strict weight copy works; no parameters or persistent buffers
    are added (packed weights are plain attributes, dropped in ``_apply``).
  * ``forward(x, valid_token_mask=None) -> Tensor`` returns ``[B, S, D]`` in
    ``x.dtype``.
  * ``OptimizerSettings`` / ``configure(**kw)`` / ``active_settings()``: the
    harness constructs the model with no extra arguments, so settings are a
    module-level default.

Per layer the forward launches five kernels (src/optimized.py:488-554 is the
reference schedule it replaces), all of them from one call into the library
(tk_forward; the schedule is written down in csrc/tk_model.hip):

  1. QKV GEMM       h[T,D] . Wqkv[3D,D]^T + b          -> qkv fp16 [T, 3D]
  2. attention      flash forward over strided q/k/v    -> ctx fp16 [B, S, H*hd]
  3. out-proj GEMM  + residual + LayerNorm2 + cast      -> resid fp32, h fp16
  4. FFN-up GEMM    + bias + exact GELU                 -> u fp16 [T, F]
  5. FFN-down GEMM  + residual + LayerNorm(next) + cast -> resid fp32, h fp16
                    (the last layer's applies final_norm and writes fp32 out)

plus one LayerNorm before the first layer.  For one-key-tile sequences (S =
64, head_dim 64; the reference's config 2) steps 1 and 2 run as one kernel
that keeps q, k and v on chip.  Steps 3 and 5 are a residual-epilogue GEMM
followed by the LayerNorm kernel; at width 128 steps 3 to 5 run as one kernel,
as do the first LayerNorm and step 1.  The
residual stream and all statistics stay fp32; only GEMM/attention operands
are fp16 (docs/pass1-decisions.md:41-65 of the reference).
"""

from __future__ import annotations

import weakref
from dataclasses import dataclass, replace
from typing import List, Optional

import torch

from . import _lib, ops
from ._lib import TK_FWD_BATCH_INVARIANT, TK_FWD_FUSED_NORM, TK_FWD_IO_BF16, TK_FWD_IO_F16, TK_FWD_QKV_ATTENTION
from .modules import BaselineTransformer

__all__ = ["OptimizerSettings", "OptimizedTransformer", "configure", "active_settings"]


@dataclass(frozen=True)
class OptimizerSettings:
    """Knobs of the MI355X path (counterpart of src/optimized.py:85-139).

    fused_norm        -- at width 128, run everything after attention as one
                         kernel (tk_narrow_tail); at other widths up to
                         fused_norm_max_d, residual + LayerNorm + cast as one
                         operator after the out-proj / FFN-down GEMM
                         (tk_gemm_bias_add_ln: a residual GEMM and a LayerNorm
                         launch).  Off: the same launches as separate steps.
    fused_norm_max_d  -- widest d_model that takes those.
    assume_dense_mask -- skip the one device->host sync per new mask object
                         that checks the padding mask is all-True.
    small_forward     -- run dense forwards of narrow models (d_model =
                         ffn_dim = 128, S <= 128) as one whole-forward kernel
                         (tk_small_forward) instead of the layer loop.
    qkv_attention     -- for dense one-key-tile sequences (S = 64, head_dim
                         64) run the QKV projection and attention as one
                         kernel (tk_qkv_attention), q/k/v kept on chip.
    batch_invariant   -- only kernels whose order of sums does not depend on the
                         batch size, so that a sequence's output bits are the
                         same in dense batches of every size, and in padded
                         ones (small_forward, for dense batches only, rounds
                         otherwise than the layers); off (default), launches
                         that would leave the chip idle split their sums.
    """

    fused_norm: bool = True
    fused_norm_max_d: int = 256
    assume_dense_mask: bool = False
    small_forward: bool = True
    qkv_attention: bool = True
    batch_invariant: bool = False


_ACTIVE = OptimizerSettings()


def configure(**kwargs) -> OptimizerSettings:
    """Set the settings used by ``OptimizedTransformer(config)`` (src/optimized.py:145-153)."""
    global _ACTIVE
    _ACTIVE = replace(_ACTIVE, **kwargs)
    return _ACTIVE


def active_settings() -> OptimizerSettings:
    return _ACTIVE


@dataclass
class _LayerWeights:
    """One block's weights packed for the kernels.

    GEMM weights fp16 (``[out, in]``, K-contiguous); biases and LayerNorm
    parameters stay fp32 (biases are added to the fp32 accumulator).
    """

    n1_w: torch.Tensor
    n1_b: torch.Tensor
    n1_eps: float
    w_qkv: torch.Tensor  # [3D, D] = cat(Wq, Wk, Wv)
    b_qkv: torch.Tensor  # [3D]
    w_o: torch.Tensor
    b_o: torch.Tensor
    n2_w: torch.Tensor
    n2_b: torch.Tensor
    n2_eps: float
    w_1: torch.Tensor  # [F, D]
    b_1: torch.Tensor
    w_2: torch.Tensor  # [D, F]
    b_2: torch.Tensor
    # The same in the narrow kernels' fragment order (width 128 only, else None; with ffn_dim
    # 128 they are parts of the whole-forward kernel's, OptimizedTransformer._stacked).
    w_qkv_packed: Optional[torch.Tensor] = None
    w_o_packed: Optional[torch.Tensor] = None
    w_1_packed: Optional[torch.Tensor] = None
    w_2_packed: Optional[torch.Tensor] = None


def _fragments(w: torch.Tensor) -> torch.Tensor:
    """A packed weight [N, K] as [K/128][N/32] blocks of MFMA fragments (include/tkmi.h, tk_narrow_tail)."""
    n, k = w.shape
    return w.view(n // 32, 32, k // 128, 8, 2, 8).permute(2, 0, 3, 4, 1, 5).contiguous()


_BLOCK_BYTES = 32 * 128 * 2  # 32 rows by 128 columns of a packed weight

# Input dtypes that tk_forward takes, and returns, as they are.
_IO_FLAGS = {torch.float16: TK_FWD_IO_F16, torch.bfloat16: TK_FWD_IO_BF16}

# Head dims the attention kernel has tiles for (tk_attention_supported).
_KERNEL_HEAD_DIMS = (16, 32, 64, 128, 256)


def _padded_head_dim(hd: int) -> Optional[int]:
    """Smallest kernel head dim >= hd, or None above 256."""
    for k in _KERNEL_HEAD_DIMS:
        if hd <= k:
            return k
    return None


class OptimizedTransformer(BaselineTransformer):
    """Drop-in replacement for the harness's ``UserOptimizedTransformer``."""

    def __init__(self, config, settings: Optional[OptimizerSettings] = None) -> None:
        super().__init__(config)
        self.settings = settings if settings is not None else _ACTIVE
        self.d_model = config.d_model
        self.num_heads = config.num_heads
        self.head_dim = config.d_model // config.num_heads
        self.attn_scale = self.head_dim ** -0.5
        # Head dims the attention kernel has no tile for run zero-padded to the
        # next one it has (the reference's kernel pads its head-dim block to a
        # power of two >= 16, src/kernels.py:268); see _weights().
        self.head_dim_padded = _padded_head_dim(self.head_dim)
        self._weight_cache: Optional[List[_LayerWeights]] = None
        self._weight_cache_key: Optional[tuple] = None
        self._param_list: Optional[list] = None  # walking the module tree costs ~60 us per forward
        self._stacked: Optional[dict] = None
        self._native: Optional[_lib.Model] = None
        self._small_ok: dict = {}  # seq -> tk_small_forward_supported
        self._dense_mask_ref: Optional[weakref.ReferenceType] = None
        self._dense_mask_value = False

    # -- caches ------------------------------------------------------------- #

    def _apply(self, *args, **kwargs):
        result = super()._apply(*args, **kwargs)
        self._native = None
        self._weight_cache = None
        self._weight_cache_key = None
        self._param_list = None
        return result

    def _weights(self) -> List[_LayerWeights]:
        """Packed weights, rebuilt when the device or any parameter changes.

        The key includes every parameter's version counter, so an in-place
        update (``load_state_dict`` after a forward) invalidates the cache.
        The parameter list itself is cached (dropped with the packed weights in
        ``_apply``): replacing a Parameter object by attribute assignment after
        a forward is not seen -- the reference's cache sees neither that nor
        in-place updates (src/optimized.py:265-285).
        """
        params = self._param_list
        if params is None:
            params = self._param_list = list(self.parameters())
        key = (params[0].device, sum(p._version for p in params), len(params))
        if self._weight_cache is not None and self._weight_cache_key == key:
            return self._weight_cache
        f16 = lambda t: t.detach().to(torch.float16).contiguous()  # noqa: E731
        f32 = lambda t: t.detach().to(torch.float32).contiguous()  # noqa: E731
        nh, hd, hp = self.num_heads, self.head_dim, self.head_dim_padded

        def pad_rows(w):  # [H*hd, ...] -> [H*hp, ...], zero rows after each head's hd
            if hp == hd:
                return w
            out = w.new_zeros((nh, hp) + tuple(w.shape[1:]))
            out[:, :hd] = w.reshape((nh, hd) + tuple(w.shape[1:]))
            return out.reshape((nh * hp,) + tuple(w.shape[1:]))

        def pad_cols(w):  # [D, H*hd] -> [D, H*hp]
            return w if hp == hd else pad_rows(w.t()).t()

        built = []
        with torch.no_grad():
            for layer in self.layers:
                at = layer.attention
                built.append(
                    _LayerWeights(
                        n1_w=f32(layer.norm1.weight), n1_b=f32(layer.norm1.bias), n1_eps=layer.norm1.eps,
                        w_qkv=f16(torch.cat([pad_rows(at.q_proj.weight), pad_rows(at.k_proj.weight),
                                             pad_rows(at.v_proj.weight)], 0)),
                        b_qkv=f32(torch.cat([pad_rows(at.q_proj.bias), pad_rows(at.k_proj.bias),
                                             pad_rows(at.v_proj.bias)], 0)),
                        w_o=f16(pad_cols(at.out_proj.weight)), b_o=f32(at.out_proj.bias),
                        n2_w=f32(layer.norm2.weight), n2_b=f32(layer.norm2.bias), n2_eps=layer.norm2.eps,
                        w_1=f16(layer.ffn_in.weight), b_1=f32(layer.ffn_in.bias),
                        w_2=f16(layer.ffn_out.weight), b_2=f32(layer.ffn_out.bias),
                    )
                )
        final = (f32(self.final_norm.weight), f32(self.final_norm.bias), self.final_norm.eps)
        stacked = self._pack_fragments(built)
        self._final, self._stacked, self._native = final, stacked, None
        self._weight_cache = built
        self._weight_cache_key = key
        return built

    def _pack_fragments(self, built: List[_LayerWeights]) -> Optional[dict]:
        """The fragment orders that the kernels of width 128 read, made with the weights and not when
        a path first runs: a capture after a warm-up through another path would record the packing,
        and the weights would hold nothing until its first replay.  Returns _stacked_weights()."""
        dp, f = self.num_heads * (self.head_dim_padded or 0), self.config.ffn_dim
        if not ops.narrow_supported(self.d_model, dp, f):
            return None
        names = ("w_qkv", "w_o", "w_1", "w_2")
        if not (built[0].w_qkv.is_cuda
                and ops.small_forward_supported(1, self.d_model, self.num_heads, self.head_dim_padded, f)):
            for lw in built:
                for n in names:
                    setattr(lw, n + "_packed", _fragments(getattr(lw, n)))
            return None
        # One copy per dtype: all layers' tensors of a name are a slice of it, in layer order.
        stacked = {}
        for group in (names, ("b_qkv", "b_o", "b_1", "b_2", "n1_w", "n1_b", "n2_w", "n2_b")):
            flat = torch.cat([getattr(lw, n).reshape(-1) for n in group for lw in built])
            at = 0
            for n in group:
                t = getattr(built[0], n)
                stacked[n] = flat[at:at + len(built) * t.numel()].view(len(built), *t.shape)
                at += len(built) * t.numel()
        stacked["packed"] = ops.small_pack(stacked)
        return stacked

    def _native_model(self) -> _lib.Model:
        """Addresses of the packed weights as the library's host call takes them, with the
        causal flag and the scale as they are now (both may be assigned between calls).
        The result holds the tensors: it may outlive the model's own references, when
        another thread packs changed weights before this one has launched."""
        built = self._weights()
        now = (bool(self.config.causal), float(self.attn_scale))
        native = self._native
        if native is None or native.made_for != now:
            stacked = self._stacked
            layers = (_lib.Layer * len(built))()
            for i, (dst, lw) in enumerate(zip(layers, built)):
                for name, _ in _lib.Layer._fields_:
                    val = getattr(lw, name)
                    setattr(dst, name, val.data_ptr() if isinstance(val, torch.Tensor) else val)
                if stacked is not None:  # a layer's 12 + 4 + 4 + 4 blocks of 32 rows by 128 columns
                    at = stacked["packed"].data_ptr() + i * 24 * _BLOCK_BYTES
                    dst.w_qkv_packed, dst.w_o_packed = at, at + 12 * _BLOCK_BYTES
                    dst.w_1_packed, dst.w_2_packed = at + 16 * _BLOCK_BYTES, at + 20 * _BLOCK_BYTES
            nf_w, nf_b, nf_eps = self._final
            native = _lib.Model(
                d_model=self.d_model, heads=self.num_heads, head_dim=self.head_dim_padded,
                ffn_dim=self.config.ffn_dim, num_layers=len(built), layers=layers, nf_w=nf_w.data_ptr(),
                nf_b=nf_b.data_ptr(), nf_eps=nf_eps, scale=now[1], causal=int(now[0]))
            native.made_for = now
            native.tensors = (built, stacked, self._final)
            self._native = native
        return native

    def __getstate__(self):
        # The addresses belong to this object's packed weights: a copy makes its own.
        state = self.__dict__.copy()
        state["_native"] = None
        return state

    def _stacked_weights(self) -> dict:
        """The per-layer packed weights stacked over layers (tk_small_forward's layout)."""
        self._weights()
        return self._stacked

    def _small_forward_ok(self, seq: int, built: List[_LayerWeights]) -> bool:
        if not self.settings.small_forward or self.head_dim_padded is None:
            return False
        if len({lw.n1_eps for lw in built}) != 1 or len({lw.n2_eps for lw in built}) != 1:
            return False
        ok = self._small_ok.get(seq)
        if ok is None:
            ok = self._small_ok[seq] = ops.small_forward_supported(
                seq, self.d_model, self.num_heads, self.head_dim_padded, self.config.ffn_dim)
        return ok

    def _mask_is_dense(self, valid_token_mask: Optional[torch.Tensor]) -> bool:
        """True when no token is padded (src/optimized.py:362-389).

        One device->host sync per distinct mask object, memoised by weakref
        identity; the harness passes one mask object for all timed calls.
        """
        if valid_token_mask is None or self.settings.assume_dense_mask:
            return True
        if self._dense_mask_ref is None or self._dense_mask_ref() is not valid_token_mask:
            self._dense_mask_value = bool(valid_token_mask.all())
            self._dense_mask_ref = weakref.ref(valid_token_mask)
        return self._dense_mask_value

    # -- forward ------------------------------------------------------------ #

    def forward(self, x: torch.Tensor, valid_token_mask: Optional[torch.Tensor] = None) -> torch.Tensor:
        if not x.is_cuda:
            raise RuntimeError(
                "OptimizedTransformer runs on the MI355X HIP kernels only; "
                f"input is on {x.device}"
            )
        if x.dim() != 3 or x.shape[-1] != self.d_model:
            raise ValueError(f"expected [B, S, {self.d_model}] input, got {tuple(x.shape)}")
        mask = None
        if not self._mask_is_dense(valid_token_mask):
            if tuple(valid_token_mask.shape) != tuple(x.shape[:2]):
                raise ValueError(f"valid_token_mask must be [B, S] = {tuple(x.shape[:2])}, "
                                 f"got {tuple(valid_token_mask.shape)}")
            mask = valid_token_mask.to(device=x.device, dtype=torch.bool).contiguous()
        if self.head_dim_padded is None:
            raise NotImplementedError(f"head_dim {self.head_dim} > 256 has no attention kernel")
        out = self._run_layers(x, mask)
        return out.to(x.dtype)

    def _run_layers(self, x: torch.Tensor, mask: Optional[torch.Tensor] = None) -> torch.Tensor:
        """The fused schedule; ``mask`` ([B, S] bool, None when dense) follows the
        baseline's padding semantics (src/torch_transformer_benchmark.py:105-121,
        143-144,170-171): padded keys are masked in attention, a padded row's
        attention output is 0 (the residual keeps x), its block output is 0,
        and its final-norm output is 0."""
        bsz, seq, d = x.shape
        t = bsz * seq
        nh, hd = self.num_heads, self.head_dim_padded
        weights = self._weights()
        fn_w, fn_b, fn_eps = self._final
        dev = x.device
        xin = x.reshape(t, d)
        small = mask is None and self._small_forward_ok(seq, weights)
        flags = 0
        if self.settings.fused_norm and d <= self.settings.fused_norm_max_d:
            flags |= TK_FWD_FUSED_NORM
        elif not small and x.dtype in _IO_FLAGS:  # converted in the first and last LayerNorm
            flags |= _IO_FLAGS[x.dtype]
        if xin.dtype != torch.float32 and not flags & (TK_FWD_IO_F16 | TK_FWD_IO_BF16):
            xin = xin.float()
        xin = xin.contiguous()
        if small:
            out = torch.empty((bsz, seq, d), dtype=torch.float32, device=dev)
            ops.small_forward(xin.view(bsz, seq, d), out, self._stacked_weights(), (fn_w, fn_b, fn_eps),
                              weights[0].n1_eps, weights[0].n2_eps, nh, hd, self.config.ffn_dim,
                              self.config.causal, self.attn_scale)
            return out

        out = torch.empty((bsz, seq, d), dtype=xin.dtype, device=dev)
        if self.settings.qkv_attention:
            flags |= TK_FWD_QKV_ATTENTION
        if self.settings.batch_invariant:
            flags |= TK_FWD_BATCH_INVARIANT
        ops.transformer_forward(self._native_model(), xin.view(bsz, seq, d), out, mask, flags)
        return out
