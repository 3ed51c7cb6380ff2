"""EncoderLayer / DecoderLayer: the pre-norm residual blocks of the reference's Transformer
(onmt/models/transformer_layers.py:83-351), composed of this package's fused operators.

    x = x + dropout(attention(LayerNorm(x)))          [decoder: once more with the encoder context]
    x = x + dropout(ffn_scale * FFN(LayerNorm(x)))

with the optional macaron half-step FFN in front (ffn_scale 0.5), stochastic depth (a layer is skipped with
probability `death_rate` during training and its sub-layer outputs are scaled by 1 / (1 - death_rate) when it
runs), and the clamp of inf / nan that fp16 training occasionally produces. Attribute names are the reference's,
so state_dicts interchange. `opt` is the reference's option namespace; the fields read are model_size, inner_size,
n_heads, dropout, attn_dropout, variational_dropout, macaron, rezero, ffn_activation, ffn_glu, fast_self_attention,
fast_xattention, fast_feed_forward and (decoder) ignore_source. Only the fast_* = True forms exist here: they are the
ones that run on the native extensions; the reference's plain-PyTorch attention and feed-forward modules are not part
of this package and asking for them raises.
"""
import torch
from torch import nn
from torch.nn.modules.module import _has_any_global_hook

from .. import _lib as L
from ..native import flash_attn_cuda
from . import feed_forward, flash_core, incremental as incremental_steps
from .encdec_attention import EncdecMultiheadAttn
from .encdec_attention_func import encdec_attn_func
from .feed_forward import PositionWiseFeedForward
from .layer_norm import LayerNorm
from .pre_post_processing import Bottle, PrePostProcessing
from .self_attention import SelfMultiheadAttn
from .self_attention_func import self_attn_func


class Identity(nn.Module):
    def forward(self, x, *args, **kwargs):
        return x


def preprocessing(rezero, *args, **kwargs):
    """ReZero layers carry no pre-normalisation (transformer_layers.py:75-80)."""
    return Identity() if rezero else PrePostProcessing(*args, **kwargs)


def _opt(opt, name, default):
    return getattr(opt, name, default)


def _require_fast(opt, *names):
    for n in names:
        if not _opt(opt, n, True):
            raise NotImplementedError(f"{n}=False selects the reference's plain-PyTorch module, which this package does not carry")


def _clamp_non_finite_(x):
    if torch.isinf(x).any() or torch.isnan(x).any():
        clamp_value = torch.finfo(x.dtype).max - 1000
        x.clamp_(min=-clamp_value, max=clamp_value)
    return x


def _called_as_built(attributes):
    """Whether calling the module of these instance attributes runs its class's forward and nothing else."""
    return not (attributes["_forward_hooks"] or attributes["_forward_pre_hooks"] or attributes["_backward_hooks"]
                or attributes["_backward_pre_hooks"] or "forward" in attributes)


class _Layer(nn.Module):
    def _common(self, opt, death_rate):
        self.variational = _opt(opt, "variational_dropout", False)
        self.death_rate = death_rate
        self.fast_self_attention = _opt(opt, "fast_self_attention", True)
        self.macaron = _opt(opt, "macaron", False)
        self.ffn_scale = 0.5 if self.macaron else 1
        rezero = _opt(opt, "rezero", False)
        if self.macaron:
            self.preprocess_mcr_ffn = preprocessing(rezero, opt.model_size, opt.dropout, sequence="n")
            self.postprocess_mcr_ffn = PrePostProcessing(opt.model_size, opt.dropout, sequence="da", variational=self.variational)
            self.mcr_feedforward = self._ffn(opt)
        self.preprocess_attn = PrePostProcessing(opt.model_size, opt.dropout, sequence="n")
        self.postprocess_attn = PrePostProcessing(opt.model_size, opt.dropout, sequence="da", variational=self.variational)

    def _ffn(self, opt):
        return PositionWiseFeedForward(opt.model_size, opt.inner_size, opt.dropout, variational=self.variational,
                                       activation=_opt(opt, "ffn_activation", "relu"), glu=_opt(opt, "ffn_glu", False))

    def _ffn_blocks(self, opt):
        self.preprocess_ffn = PrePostProcessing(opt.model_size, opt.dropout, sequence="n")
        self.postprocess_ffn = PrePostProcessing(opt.model_size, opt.dropout, sequence="da", variational=self.variational)
        self.feedforward = self._ffn(opt)

    def _alive(self):
        if self.training:
            return torch.rand(1)[0].item() >= self.death_rate
        return True

    def _scaled_ffn_scale(self):
        if self.training and self.death_rate > 0:
            return self.ffn_scale / (1 - self.death_rate)
        return self.ffn_scale

    def _survivor_scale(self, out):
        if self.training and self.death_rate > 0:
            return out / (1 - self.death_rate)
        return out

    def _times(self, out, scale):
        return out if scale == 1 else out * scale

    def _macaron_step(self, input):
        if self.macaron:
            out = self.mcr_feedforward(self.preprocess_mcr_ffn(input))
            input = self.postprocess_mcr_ffn(self._times(out, self._scaled_ffn_scale()), input)
        return input

    def _ffn_step(self, input):
        out = self.feedforward(self.preprocess_ffn(input))
        return self.postprocess_ffn(self._times(out, self._scaled_ffn_scale()), input)


    # -- the layer as one node of the host layer (csrc/host/layers.cpp) -------------------------------------------------
    # Taken by the plain form: 16-bit tensors on the GPU, LayerNorm with affine parameters in front, dropout + add behind,
    # no gate, no variational dropout, no stochastic depth, no macaron block, nothing that listens to or replaces the call of
    # a sub-module at any depth, and either training with a backward to come or evaluation without one. Everything else runs
    # operator by operator below.
    _PRE, _POST = ["n"], ["d", "a"]

    def _sub_parameters(self, pre, mods):
        """The parameters of the sub-modules in the order of the native layer, or None where one is not of the plain form. (An
        entry is None where a sub-module carries a plain tensor in a parameter's place: the native layer then declines.)"""
        if _has_any_global_hook():
            return None
        train, subs, out = self.training, self._modules, []
        for name in mods:
            m = subs.get(name)
            if m is None:
                return None
            kind, d = type(m), m.__dict__            # (instance attributes read from the dict: this runs on every call)
            if d["training"] is not train or not _called_as_built(d):
                return None
            if kind is PrePostProcessing:
                if name in pre:
                    n = d["_modules"]["layer_norm"] if d["steps"] == self._PRE else None
                    if type(n) is not Bottle or not _called_as_built(n.__dict__):
                        return None
                    n = n._modules["function"]
                    if type(n) is not LayerNorm or n.eps != 1e-5 or n.memory_efficient or not _called_as_built(n.__dict__):
                        return None
                    p = n._parameters.get
                    out += (p("weight"), p("bias"))
                else:
                    n = d["_modules"].get("dropout")
                    if d["steps"] != self._POST or d["variational"] or type(n) is not nn.Dropout or n.training is not train \
                            or not n.p == d["dropout_p"] == subs["postprocess_ffn"].dropout_p or not _called_as_built(n.__dict__):
                        return None
            elif kind is SelfMultiheadAttn:
                if d["rotary_pos_enc"] or d["head_dim"] not in (64, 128) or d["attn_func"] is not self_attn_func:
                    return None
                p = d["_parameters"].get
                out += (p("in_proj_weight"), p("in_proj_bias"), p("out_proj_weight"), p("out_proj_bias"))
            elif kind is EncdecMultiheadAttn:
                if d["attn_func"] is not encdec_attn_func:
                    return None
                p = d["_parameters"].get
                out += (p("in_proj_weight_q"), p("in_proj_weight_kv"), p("out_proj_weight"))
            elif kind is PositionWiseFeedForward:
                if d["glu"] or d["variational"] or d["dropout_residual"] or d["fused_function"] is not feed_forward.FUNCTIONS.get(d["activation"]):
                    return None
                p = d["_parameters"].get
                out += (p("in_proj_weight"), p("in_proj_bias"), p("out_proj_weight"), p("out_proj_bias"))
            else:
                return None
        return out

    def _native_mode(self, x, inputs, params):
        if params is None or self.macaron or self.death_rate > 0 or feed_forward.recompute or torch.is_autocast_enabled() \
                or not flash_core.switched_on() or L.tracing():
            return 0
        mode = L.host().layer_mode(x, inputs, params)
        return mode if (mode == 2) is self.training else 0


class EncoderLayer(_Layer):
    """forward(input [T, B, model_size], attn_mask: key-padding mask [B, T], nonzero = padded) -> [T, B, model_size]."""

    def __init__(self, opt, death_rate=0.0, **kwargs):
        super().__init__()
        _require_fast(opt, "fast_self_attention", "fast_feed_forward")
        self._common(opt, death_rate)
        self._ffn_blocks(opt)
        self.multihead = SelfMultiheadAttn(opt.model_size, opt.n_heads, opt.attn_dropout)

    _SUB = ("preprocess_attn", "multihead", "postprocess_attn", "preprocess_ffn", "feedforward", "postprocess_ffn")

    def _native_forward(self, x, attn_mask):
        params = self._sub_parameters(("preprocess_attn", "preprocess_ffn"), self._SUB)
        mode = self._native_mode(x, (), params)
        if mode == 0:
            return None
        host, train = L.host(), self.training
        mh, ff = self._modules["multihead"], self._modules["feedforward"]
        heads = mh.num_heads
        p_attn, p_res, p_ffn = (mh.dropout, self._modules["postprocess_ffn"].dropout_p, ff.dropout) if train else (0.0, 0.0, 0.0)
        x = x.contiguous()
        pad = host.mask_bytes(attn_mask, x, x.shape[1], x.shape[0])
        z, stats, lin, q, k, v = host.layer_begin(x, *params[:4], heads)
        ctx, lse, state = flash_attn_cuda.fwd_batched(q, k, v, pad, p_attn, mh.head_dim ** -0.5, False)
        return host.encoder_end(x, z, stats, lin, ctx, lse, state, pad, params, heads, ff.activation_code, p_attn, p_res, p_ffn, mode == 2)

    def forward(self, input, attn_mask):
        if self._alive():
            if input.is_cuda:
                out = self._native_forward(input, attn_mask)
                if out is not None:
                    return out
            input = self._macaron_step(input)
            query = self.preprocess_attn(input)
            out, _ = self.multihead(query, None, attn_mask, None, return_coverage=False)    # the coverage is dropped here
            input = self.postprocess_attn(self._survivor_scale(out), input)
            input = self._ffn_step(input)
        return _clamp_non_finite_(input)


class DecoderLayer(_Layer):
    """forward(input [Tq, B, E], context [Tk, B, E], mask_tgt: time mask [Tq, Tq], mask_src: key-padding mask
    [B, Tk]) -> (output, coverage, incremental_cache)."""

    def __init__(self, opt, death_rate=0.0):
        super().__init__()
        _require_fast(opt, "fast_self_attention", "fast_feed_forward")
        self.ignore_source = _opt(opt, "ignore_source", False)
        if not self.ignore_source:
            _require_fast(opt, "fast_xattention")
        self._common(opt, death_rate)
        self.multihead_tgt = SelfMultiheadAttn(opt.model_size, opt.n_heads, opt.attn_dropout)
        if not self.ignore_source:
            self.preprocess_src_attn = PrePostProcessing(opt.model_size, opt.dropout, sequence="n")
            self.postprocess_src_attn = PrePostProcessing(opt.model_size, opt.dropout, sequence="da",
                                                          variational=self.variational)
            self.multihead_src = EncdecMultiheadAttn(opt.n_heads, opt.model_size, opt.attn_dropout)
        self._ffn_blocks(opt)

    _SUB = ("preprocess_attn", "multihead_tgt", "postprocess_attn", "preprocess_src_attn", "multihead_src", "postprocess_src_attn",
            "preprocess_ffn", "feedforward", "postprocess_ffn")

    def _native_forward(self, x, context, mask_tgt, mask_src):
        params = self._sub_parameters(("preprocess_attn", "preprocess_src_attn", "preprocess_ffn"), self._SUB)
        mode = self._native_mode(x, (context,), params)
        if mode == 0 or context.dim() != 3 or context.shape[0] > 4096 or context.shape[1:] != x.shape[1:]:
            return None
        host, train = L.host(), self.training
        mh, mc, ff = self._modules["multihead_tgt"], self._modules["multihead_src"], self._modules["feedforward"]
        heads = mh.num_heads
        if mc.num_heads != heads:
            return None
        p_attn, p_cross, p_res, p_ffn = ((mh.dropout, mc.dropout, self._modules["postprocess_ffn"].dropout_p, ff.dropout) if train
                                         else (0.0, 0.0, 0.0, 0.0))
        x = x.contiguous()
        time = None
        if mask_tgt is not None:
            time = host.mask_bytes(mask_tgt if mask_tgt.dtype in (torch.bool, torch.uint8) else mask_tgt.to(torch.bool), x, x.shape[0],
                                   x.shape[0])
        pad = host.mask_bytes(mask_src, x, context.shape[1], context.shape[0])
        z, stats, lin, q, k, v = host.layer_begin(x, *params[:4], heads)
        ctx, lse, state = flash_attn_cuda.fwd_batched(q, k, v, None, p_attn, mh.head_dim ** -0.5, False, time_mask=time)
        return host.decoder_end(x, context, z, stats, lin, ctx, lse, state, time, pad, params, heads, ff.activation_code, p_attn, p_cross,
                                p_res, p_ffn, mode == 2)

    def _native_step(self, x, mask_tgt, mask_src, cache):
        params = self._sub_parameters(("preprocess_attn", "preprocess_src_attn", "preprocess_ffn"), self._SUB)
        if mask_tgt is not None or self._native_mode(x, (), params) != 1:
            return None
        heads = self._modules["multihead_tgt"].num_heads
        if self._modules["multihead_src"].num_heads != heads:
            return None
        return incremental_steps.layer_step(L.host().decoder_step, x, params, heads, self._modules["feedforward"].activation_code, mask_src, cache)

    def forward(self, input, context, mask_tgt, mask_src, incremental=False, incremental_cache=None, reuse_source=True):
        if incremental and incremental_cache is None:
            incremental_cache = dict()
        coverage = None
        if self._alive():
            if input.is_cuda and incremental and not self.ignore_source:
                native = self._native_step(input, mask_tgt, mask_src, incremental_cache)
                if native is not None:
                    return native[0], native[1], incremental_cache
            if input.is_cuda and not incremental and not self.ignore_source and context is not None:
                native = self._native_forward(input, context, mask_tgt, mask_src)
                if native is not None:
                    return native[0], native[1], incremental_cache
            input = self._macaron_step(input)
            query = self.preprocess_attn(input)
            out, _ = self.multihead_tgt(query, None, None, mask_tgt, incremental=incremental,
                                        incremental_cache=incremental_cache, return_coverage=False)   # dropped here
            input = self.postprocess_attn(self._survivor_scale(out), input)
            if not self.ignore_source:
                query = self.preprocess_src_attn(input)
                out, coverage = self.multihead_src(query, context, context, mask_src, incremental=incremental,
                                                   incremental_cache=incremental_cache)
                input = self.postprocess_src_attn(self._survivor_scale(out), input)
            input = self._ffn_step(input)
        return _clamp_non_finite_(input), coverage, incremental_cache
