"""What this library is timed on: the work that a translation or speech model built on it has it do, through the modules,
autograd functions and optimizer that such a program calls.

`listed()` are the representative cases, `draw(rng)` gives more of the same ranges; `prepare(case, seed)` makes what the program
has in hand (module or parameters, inputs, masks), `run(state)` is one pass as the program runs it and returns everything the
pass computes (outputs, gradients, updated state), `work(case)` the bytes and operations a pass cannot do without, and
`tolerance(case)` how far two correct implementations of the same precision may lie apart.

Sizes follow the benchmark (bench.py, nmtgminor_amd/synthetic.py): model dimension 512 with inner dimension 2048 (the base
transformer) and 1024 with 4096 (the large one), heads of 64, sentences up to 512 positions, 1500 encoder frames for speech,
vocabularies up to 250 054. Training draws its dropout masks from the device generator (rate 0.1), as a training program does.
"""
import math
from types import SimpleNamespace

import torch

from nmtgminor_amd.modules.flash_mha import flash_bert_mha
from nmtgminor_amd.modules.feed_forward import PositionWiseFeedForward
from nmtgminor_amd.modules.fused_adam import FusedAdam
from nmtgminor_amd.modules.fused_clip_norm import fused_clip_grad_norm
from nmtgminor_amd.modules.generator_loss import GeneratorLoss
from nmtgminor_amd.modules.layer_norm import LayerNorm
from nmtgminor_amd.modules.self_attention import SelfMultiheadAttn
from nmtgminor_amd.modules.softmax_xentropy import SoftmaxCrossEntropyLoss
from nmtgminor_amd.modules.transformer_layers import DecoderLayer, EncoderLayer

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}
HEAD = 64                      # head dimension of every configuration
P = 0.1                        # dropout rate of every configuration
PAD = 1                        # padding index of the targets
LARGEST_LOGITS = 4096 * 250054


def listed():
    return [
        # A LayerNorm in fp32 training, forward and backward: the benchmark's first configuration. Launches and latency count.
        dict(name="layer_norm_train_f32", kind="layer_norm", rows=4096, hidden=512, dtype="f32"),
        # The base transformer's feed-forward block, forward and backward: the benchmark's second configuration.
        dict(name="ffn_train_f16", kind="ffn", t=128, b=64, e=512, act="gelu", dtype="f16"),
        # Encoder self-attention as a drop-in for the reference's module, which returns the coverage: third configuration.
        dict(name="self_attn_train_coverage", kind="self_attn", t=512, b=32, e=1024, dtype="bf16"),
        # One encoder layer of the large model in training, a full batch of long sentences.
        dict(name="encoder_layer_train_large", kind="encoder_layer", t=512, b=32, e=1024, act="relu", dtype="bf16"),
        # One encoder layer of the base model in training on a small ragged batch (the short sentences of a bucketed corpus).
        dict(name="encoder_layer_train_small", kind="encoder_layer", t=37, b=13, e=512, act="relu", dtype="f16"),
        # One decoder layer of the base model in training, an ordinary batch with odd sentence lengths.
        dict(name="decoder_layer_train_ragged", kind="decoder_layer", tq=61, tk=73, b=48, e=512, act="relu", dtype="bf16"),
        # Speech decoder layer, evaluation of whole target sentences over 1500 encoder frames: fourth configuration.
        dict(name="decoder_layer_eval_speech", kind="decoder_eval", tq=128, tk=1500, b=16, e=1024, act="relu", dtype="bf16"),
        # One step of incremental decoding: a beam of 5 over one sentence and its cache.
        dict(name="decode_step_beam5", kind="decode_step", prev=24, tk=61, b=5, e=512, act="relu", dtype="f16"),
        # Attention over packed sequences (speech encoder without padding), forward and backward.
        dict(name="packed_attn_train", kind="packed_attn", max_len=512, b=32, heads=16, causal=False, dtype="bf16"),
        # Label-smoothed cross-entropy over a large multilingual vocabulary: fifth configuration, a quarter of its rows.
        dict(name="xentropy_train_250k", kind="xentropy", rows=4096, vocab=250054, dtype="bf16"),
        # Output projection and loss together, the large model with a large vocabulary.
        dict(name="generator_loss_train", kind="generator", rows=4096, vocab=250054, e=1024, dtype="bf16"),
        # Gradient clipping and the AdamW step over the base model's parameter list (60 M elements in 193 tensors).
        dict(name="clip_and_adam_step", kind="adam", layers=6, e=512, vocab=32000, dtype="f32"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("layer_norm", "ffn", "self_attn", "encoder_layer", "encoder_layer", "decoder_layer", "decoder_eval",
                       "decode_step", "packed_attn", "xentropy", "generator", "adam"))
    half = rng.choice(("f16", "bf16"))
    e = rng.choice((512, 1024))
    act = rng.choice(("relu", "gelu", "silu"))
    if kind == "layer_norm":
        return dict(kind=kind, rows=_log(rng, 32, 65536), hidden=rng.choice((512, 768, 1024)), dtype=rng.choice(("f32", "f16", "bf16")))
    if kind == "ffn":
        return dict(kind=kind, t=_log(rng, 8, 512), b=_log(rng, 1, 32), e=e, act=act, dtype=half)
    if kind == "self_attn":
        return dict(kind=kind, t=_log(rng, 8, 512), b=_log(rng, 1, 32), e=e, dtype=half)
    if kind == "encoder_layer":
        return dict(kind=kind, t=_log(rng, 8, 512), b=_log(rng, 1, 32), e=e, act=act, dtype=half)
    if kind == "decoder_layer":
        return dict(kind=kind, tq=_log(rng, 8, 256), tk=_log(rng, 8, 512), b=_log(rng, 1, 32), e=e, act=act, dtype=half)
    if kind == "decoder_eval":
        return dict(kind=kind, tq=_log(rng, 2, 256), tk=_log(rng, 50, 1500), b=_log(rng, 1, 32), e=e, act=act, dtype=half)
    if kind == "decode_step":
        return dict(kind=kind, prev=_log(rng, 2, 255), tk=_log(rng, 16, 1500), b=_log(rng, 1, 64), e=e, act=act, dtype=half)
    if kind == "packed_attn":
        return dict(kind=kind, max_len=_log(rng, 32, 1500), b=_log(rng, 1, 32), heads=e // HEAD, causal=rng.random() < 0.3, dtype=half)
    if kind == "xentropy":
        vocab = _log(rng, 8000, 250054)
        return dict(kind=kind, rows=_log(rng, 64, min(16384, LARGEST_LOGITS // vocab)), vocab=vocab, dtype=half)
    if kind == "generator":
        vocab = _log(rng, 8000, 250054)
        return dict(kind=kind, rows=_log(rng, 64, min(16384, LARGEST_LOGITS // vocab)), vocab=vocab, e=e, dtype=half)
    return dict(kind="adam", layers=rng.randint(1, 8), e=e, vocab=_log(rng, 8000, 64000), dtype=rng.choice(("f32", "bf16")))


# ------------------------------------------------------------------------------------------------------------- inputs
def _options(case):
    return SimpleNamespace(model_size=case["e"], inner_size=4 * case["e"], n_heads=case["e"] // HEAD, dropout=P, attn_dropout=P,
                           variational_dropout=False, macaron=False, rezero=False, ffn_activation=case["act"], ffn_glu=False,
                           fast_self_attention=True, fast_xattention=True, fast_feed_forward=True, ignore_source=False)


def _trained(module, dtype, train):
    """The module in the working precision, its biases and affine parameters away from their initial constants."""
    with torch.no_grad():
        for p in module.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    return module.to(dtype).train(train)


def _randn(shape, dtype, scale=1.0):
    return (scale * torch.randn(shape, device=DEVICE)).to(dtype)


def _lengths(b, t):
    """Sentence lengths between half of the padded length and all of it; the longest fills it."""
    n = torch.randint(max(1, t // 2), t + 1, (b,), device=DEVICE)
    n[0] = t
    return n


def _key_padding(b, t):
    return torch.arange(t, device=DEVICE)[None, :] >= _lengths(b, t)[:, None]


def _causal(t):
    return torch.triu(torch.ones(t, t, device=DEVICE), 1).bool()


def _targets(rows, vocab):
    """Ranks of a Zipf-like distribution, one position in ten padded."""
    u = torch.rand(rows, device=DEVICE)
    y = (torch.exp(u * math.log(vocab)) - 1).long().clamp_(0, vocab - 1)
    return torch.where(torch.rand(rows, device=DEVICE) < 0.1, torch.full_like(y, PAD), y)


def _adam_shapes(case):
    e, f = case["e"], 4 * case["e"]
    layer = [(3 * e, e), (3 * e,), (e, e), (e,), (f, e), (f,), (e, f), (e,), (e,), (e,), (e,), (e,)]
    cross = [(e, e), (e,), (2 * e, e), (2 * e,), (e, e), (e,), (e,), (e,)]
    return [(case["vocab"], e)] + layer * case["layers"] + (layer + cross) * case["layers"]


def _cut(flat, shapes):
    out, at = [], 0
    for s in shapes:
        n = math.prod(s)
        out.append(flat[at:at + n].view(s))
        at += n
    return out


def prepare(case, seed):
    torch.manual_seed(seed)                  # the device generator too: weights, inputs and the dropout masks of run()
    with torch.device(DEVICE):
        return _PREPARE[case["kind"]](case, DTYPES[case["dtype"]])


def _prepare_layer_norm(case, dtype):
    m = _trained(LayerNorm((case["hidden"],)), dtype, True)
    x = _randn((case["rows"], case["hidden"]), dtype).requires_grad_()
    return dict(kind="module", module=m, inputs=(x,), args=(), dy=_randn(x.shape, dtype))


def _prepare_ffn(case, dtype):
    m = _trained(PositionWiseFeedForward(case["e"], 4 * case["e"], P, activation=case["act"]), dtype, True)
    x = _randn((case["t"], case["b"], case["e"]), dtype).requires_grad_()
    return dict(kind="module", module=m, inputs=(x,), args=(), dy=_randn(x.shape, dtype))


def _prepare_self_attn(case, dtype):
    m = _trained(SelfMultiheadAttn(case["e"], case["e"] // HEAD, P), dtype, True)
    x = _randn((case["t"], case["b"], case["e"]), dtype).requires_grad_()
    return dict(kind="module", module=m, inputs=(x,), args=(None, _key_padding(case["b"], case["t"])), dy=_randn(x.shape, dtype))


def _prepare_encoder_layer(case, dtype):
    m = _trained(EncoderLayer(_options(case)), dtype, True)
    x = _randn((case["t"], case["b"], case["e"]), dtype).requires_grad_()
    return dict(kind="module", module=m, inputs=(x,), args=(_key_padding(case["b"], case["t"]),), dy=_randn(x.shape, dtype))


def _prepare_decoder_layer(case, dtype):
    m = _trained(DecoderLayer(_options(case)), dtype, True)
    x = _randn((case["tq"], case["b"], case["e"]), dtype).requires_grad_()
    context = _randn((case["tk"], case["b"], case["e"]), dtype).requires_grad_()
    return dict(kind="module", module=m, inputs=(x, context), args=(_causal(case["tq"]), _key_padding(case["b"], case["tk"])),
                dy=_randn(x.shape, dtype))


def _prepare_decoder_eval(case, dtype):
    m = _trained(DecoderLayer(_options(case)), dtype, False)
    return dict(kind="eval", module=m, x=_randn((case["tq"], case["b"], case["e"]), dtype),
                context=_randn((case["tk"], case["b"], case["e"]), dtype), time=_causal(case["tq"]),
                pad=_key_padding(case["b"], case["tk"]))


def _prepare_decode_step(case, dtype):
    """The cache as the steps before this one left it: encoder keys and values projected, `prev` positions decoded."""
    m = _trained(DecoderLayer(_options(case)), dtype, False)
    context = _randn((case["tk"], case["b"], case["e"]), dtype)
    pad = _key_padding(case["b"], case["tk"])
    cache = {}
    with torch.no_grad():
        first = case["prev"] - 1
        m(_randn((first, case["b"], case["e"]), dtype), context, _causal(first), pad, incremental=True, incremental_cache=cache)
        m(_randn((1, case["b"], case["e"]), dtype), context, None, pad, incremental=True, incremental_cache=cache)
    return dict(kind="step", module=m, x=_randn((1, case["b"], case["e"]), dtype), context=context, pad=pad, cache=cache)


def _prepare_packed_attn(case, dtype):
    # the lengths of a packed batch fill its token budget: spread evenly over [n / 2, n], in random order
    lens = torch.linspace(case["max_len"], max(1, case["max_len"] // 2), case["b"]).round().long()[torch.randperm(case["b"])]
    cu = torch.zeros(case["b"] + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(lens, 0)
    qkv = _randn((int(cu[-1]), 3, case["heads"], HEAD), dtype).requires_grad_()
    return dict(kind="packed", qkv=qkv, cu=cu, max_len=case["max_len"], causal=case["causal"], dy=_randn((qkv.shape[0],) + qkv.shape[2:], dtype))


def _prepare_xentropy(case, dtype):
    logits = torch.empty(case["rows"], case["vocab"], dtype=dtype)
    for r in range(0, case["rows"], 1024):
        logits[r:r + 1024] = _randn((min(1024, case["rows"] - r), case["vocab"]), dtype, 2.0)
    return dict(kind="xentropy", logits=logits.requires_grad_(), labels=_targets(case["rows"], case["vocab"]))


def _prepare_generator(case, dtype):
    m = GeneratorLoss(case["e"], case["vocab"], label_smoothing=0.1, padding_idx=PAD).to(dtype).train()
    x = _randn((case["rows"], case["e"]), dtype).requires_grad_()
    return dict(kind="generator", module=m, x=x, labels=_targets(case["rows"], case["vocab"]))


def _prepare_adam(case, dtype):
    """Parameters, gradients and moments in four flat buffers (as a program that reduces gradients in buckets keeps them)."""
    shapes = _adam_shapes(case)
    n = sum(math.prod(s) for s in shapes)
    flat = [_randn(n, dtype, 0.1), _randn(n, dtype, 1e-2), _randn(n, dtype, 1e-3), _randn(n, dtype, 1e-2).square_()]
    params = [torch.nn.Parameter(p) for p in _cut(flat[0], shapes)]
    opt = FusedAdam(params, lr=1e-4, betas=(0.9, 0.98), weight_decay=0.01)
    for p, g, m, v in zip(params, *(_cut(f, shapes) for f in flat[1:])):
        p.grad = g
        opt.state[p] = dict(exp_avg=m, exp_avg_sq=v)
    return dict(kind="adam", params=params, opt=opt, flat=flat)


_PREPARE = dict(layer_norm=_prepare_layer_norm, ffn=_prepare_ffn, self_attn=_prepare_self_attn, encoder_layer=_prepare_encoder_layer,
                decoder_layer=_prepare_decoder_layer, decoder_eval=_prepare_decoder_eval, decode_step=_prepare_decode_step,
                packed_attn=_prepare_packed_attn, xentropy=_prepare_xentropy, generator=_prepare_generator, adam=_prepare_adam)


# --------------------------------------------------------------------------------------------------------------- passes
def run(state):
    return _RUN[state["kind"]](state)


def _run_module(s):
    """A training step of one module: forward, backward, every gradient fresh (the optimizer cleared them)."""
    m = s["module"]
    params = list(m.parameters())
    for p in params:
        p.grad = None
    for x in s["inputs"]:
        x.grad = None
    out = m(*s["inputs"], *s["args"])
    first = out[0] if isinstance(out, tuple) else out
    first.backward(s["dy"])
    extra = [o.detach() for o in out[1:] if torch.is_tensor(o)] if isinstance(out, tuple) else []
    return [first.detach(), *extra, *(x.grad for x in s["inputs"]), *(p.grad for p in params)]


def _run_eval(s):
    with torch.no_grad():
        out, coverage, _ = s["module"](s["x"], s["context"], s["time"], s["pad"])
    return [out, coverage]


def _run_step(s):
    cache = dict(s["cache"])                 # every pass decodes the same next position
    with torch.no_grad():
        out, coverage, cache = s["module"](s["x"], s["context"], None, s["pad"], incremental=True, incremental_cache=cache)
    return [out, coverage, cache["k"], cache["v"]]


def _run_packed(s):
    s["qkv"].grad = None
    out = flash_bert_mha(s["qkv"], s["cu"], s["max_len"], P, None, s["causal"], False)
    out.backward(s["dy"])
    return [out.detach(), s["qkv"].grad]


def _run_xentropy(s):
    s["logits"].grad = None
    losses = SoftmaxCrossEntropyLoss.apply(s["logits"], s["labels"], 0.1, PAD, True)
    losses.sum().backward()
    return [losses.detach(), s["logits"].grad]


def _run_generator(s):
    m = s["module"]
    m.linear.weight.grad = m.linear.bias.grad = s["x"].grad = None
    r = m(s["x"], s["labels"])
    r["loss"].backward()
    return [r["loss"].detach(), r["data"], s["x"].grad, m.linear.weight.grad, m.linear.bias.grad]


def _run_adam(s):
    norm = fused_clip_grad_norm(s["params"], 1.0)
    s["opt"].step()
    return [norm, *s["flat"]]


_RUN = dict(module=_run_module, eval=_run_eval, step=_run_step, packed=_run_packed, xentropy=_run_xentropy, generator=_run_generator,
            adam=_run_adam)


# ----------------------------------------------------------------------------------------------------------- accounting
def _attn_flops(tq, tk, b, e):
    return 4.0 * b * tq * tk * e             # scores and context, all heads


def work(case):
    """Every input read once, every output written once; products at two operations per multiply-add."""
    kind, s = case["kind"], BYTES[case["dtype"]]
    if kind == "layer_norm":
        n = case["rows"] * case["hidden"]
        return dict(bytes=4 * n * s + 4 * case["hidden"] * s, flops=16.0 * n)          # x, dy in; y, dx out; affine and its gradients
    if kind == "ffn":
        n, e = case["t"] * case["b"], case["e"]
        w = 8 * e * e + 5 * e
        return dict(bytes=(4 * n * e + 2 * w) * s, flops=3 * 2.0 * n * 8 * e * e)
    if kind == "self_attn":
        t, b, e = case["t"], case["b"], case["e"]
        w = 4 * e * e + 4 * e
        cover = b * (e // HEAD) * t * t
        return dict(bytes=(4 * t * b * e + 2 * w + cover) * s + t * b, flops=3 * (2.0 * t * b * 4 * e * e + _attn_flops(t, t, b, e)))
    if kind == "encoder_layer":
        t, b, e = case["t"], case["b"], case["e"]
        w = 12 * e * e + 13 * e
        return dict(bytes=(4 * t * b * e + 2 * w) * s + t * b, flops=3 * (2.0 * t * b * 12 * e * e + _attn_flops(t, t, b, e)))
    if kind in ("decoder_layer", "decoder_eval"):
        tq, tk, b, e = case["tq"], case["tk"], case["b"], case["e"]
        w = 16 * e * e + 15 * e
        cover = b * (e // HEAD) * tq * tk
        flops = 2.0 * tq * b * 14 * e * e + 2.0 * tk * b * 2 * e * e + _attn_flops(tq, tq, b, e) + _attn_flops(tq, tk, b, e)
        rows = (2 * tq + tk) * b * e
        if kind == "decoder_eval":
            return dict(bytes=(rows + w + cover) * s + tk * b + tq * tq, flops=flops)
        return dict(bytes=(rows + (2 * tq + tk) * b * e + 2 * w + cover) * s + tk * b + tq * tq, flops=3 * flops)
    if kind == "decode_step":
        t, tk, b, e = case["prev"] + 1, case["tk"], case["b"], case["e"]
        w = 14 * e * e + 15 * e                                                        # the encoder keys / values are cached
        return dict(bytes=(w + 2 * (t + 0.75 * tk) * b * e + 2 * b * e + b * (e // HEAD) * tk) * s + tk * b,
                    flops=2.0 * b * 14 * e * e + _attn_flops(1, t, b, e) + _attn_flops(1, tk, b, e))
    if kind == "packed_attn":
        n, h = case["max_len"], case["heads"]
        tokens, pairs = 0.75 * n * case["b"], case["b"] * n * n * 7.0 / 12             # lengths uniform in [n / 2, n]
        return dict(bytes=8 * tokens * h * HEAD * s, flops=3 * 4.0 * pairs * h * HEAD * (0.5 if case["causal"] else 1.0))
    if kind == "xentropy":
        n = case["rows"] * case["vocab"]
        return dict(bytes=2.0 * n * s + 12 * case["rows"], flops=8.0 * n)
    if kind == "generator":
        n, v, e = case["rows"], case["vocab"], case["e"]
        return dict(bytes=2.0 * (n * e + v * e + v) * s + 8 * n, flops=3 * 2.0 * n * v * e)
    n = sum(math.prod(x) for x in _adam_shapes(case))
    return dict(bytes=8.0 * n * s, flops=16.0 * n)                                     # p, g, m, v in and out (the clipped gradients are kept)


def tolerance(case):
    """32-bit: sums in another order. 16-bit: every stored intermediate of a chain of operators may round the other way, half a
    unit in the last place each (bf16 2^-9, fp16 2^-12), and a relu may gate an element within rounding of zero."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] in ("layer_norm", "xentropy", "adam"):
        return {"rel": 4e-3 if case["dtype"] == "bf16" else 5e-4}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
