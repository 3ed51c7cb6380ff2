"""The layers as one native node (csrc/host/layers.cpp) against the same layer run operator by operator (a forward hook on a
sub-module keeps a layer on that path), and the kernels it adds (LayerNorm over a residual sum and its backward, the guarded
dropout + add) against the separate ones, at the edges of their shapes."""
import math
from types import SimpleNamespace

import pytest
import torch

from nmtgminor_amd import _lib as L
from nmtgminor_amd.modules.softmax_xentropy import SoftmaxCrossEntropyLoss
from nmtgminor_amd.modules.transformer_layers import DecoderLayer, EncoderLayer
from nmtgminor_amd.native import fast_layer_norm_cuda as ln
from util import assert_close, rel_err

pytestmark = pytest.mark.gpu
F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


def options(e, p, act):
    return SimpleNamespace(model_size=e, inner_size=2 * e, n_heads=e // 64, dropout=p, attn_dropout=p, variational_dropout=False,
                           macaron=False, rezero=False, ffn_activation=act, ffn_glu=False, fast_self_attention=True,
                           fast_xattention=True, fast_feed_forward=True, ignore_source=False)


def randomised(layer, dev, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for p in layer.parameters():
            p.add_((0.1 if p.dim() == 1 else 0.02) * torch.randn(p.shape, generator=g))
    return layer.to(dev).to(dtype)


def both_paths(layer, hooked, call, inputs, dy):
    """[outputs and gradients] of the native path and of the operator-by-operator one, with the same dropout masks"""
    res = []
    for by_operator in (False, True):
        handle = hooked.register_forward_hook(lambda m, i, o: None) if by_operator else None
        torch.manual_seed(3)
        torch.cuda.manual_seed(5)
        for t in list(inputs) + list(layer.parameters()):
            t.grad = None
        out = call()
        out = out if isinstance(out, tuple) else (out,)
        if dy is not None:
            out[0].backward(dy)
        res.append([o for o in out if torch.is_tensor(o)] + ([t.grad for t in inputs] + [p.grad for p in layer.parameters()] if dy is not None else []))
        if handle is not None:
            handle.remove()
    return res


def same(pair, dtype):
    """The two paths round at the same points; where their kernels sum in another order a rounding may fall the other way."""
    for a, b in zip(*pair):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(torch.isnan(a), torch.isnan(b))
            assert rel_err(torch.nan_to_num(a), torch.nan_to_num(b)) < (1e-2 if dtype == BF16 else 2e-3)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("t,b,e,p,act,train", [(1, 1, 128, 0.1, "relu", True), (37, 13, 512, 0.1, "gelu", True), (130, 3, 256, 0.0, "silu", True),
                                               (64, 2, 1024, 0.1, "relu", True), (33, 5, 512, 0.1, "relu", False)])
def test_encoder_layer(dev, dtype, t, b, e, p, act, train):
    layer = randomised(EncoderLayer(options(e, p, act)), dev, dtype, 1).train(train)
    x = torch.randn(t, b, e, device=dev).to(dtype).requires_grad_(train)
    pad = torch.arange(t, device=dev)[None] >= torch.randint((t + 1) // 2, t + 1, (b,), device=dev)[:, None]
    dy = torch.randn(t, b, e, device=dev).to(dtype)
    with torch.set_grad_enabled(train):
        same(both_paths(layer, layer.feedforward, lambda: layer(x, pad), [x] if train else [], dy if train else None), dtype)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("tq,tk,b,e,p,train", [(1, 4, 1, 128, 0.1, True), (61, 73, 6, 512, 0.1, True), (129, 64, 3, 256, 0.0, True),
                                               (31, 100, 4, 512, 0.1, False), (5, 61, 2, 128, 0.0, False)])
def test_decoder_layer(dev, dtype, tq, tk, b, e, p, train):
    layer = randomised(DecoderLayer(options(e, p, "gelu")), dev, dtype, 2).train(train)
    x = torch.randn(tq, b, e, device=dev).to(dtype).requires_grad_(train)
    c = torch.randn(tk, b, e, device=dev).to(dtype).requires_grad_(train)
    pad = torch.arange(tk, device=dev)[None] >= torch.randint((tk + 1) // 2, tk + 1, (b,), device=dev)[:, None]
    causal = torch.triu(torch.ones(tq, tq, device=dev), 1).bool()
    dy = torch.randn(tq, b, e, device=dev).to(dtype)
    with torch.set_grad_enabled(train):
        same(both_paths(layer, layer.feedforward, lambda: layer(x, c, causal, pad), [x, c] if train else [], dy if train else None), dtype)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("b,tk,prev,e", [(1, 1, 2, 128), (5, 61, 24, 512), (33, 130, 64, 256), (64, 300, 70, 1024), (3, 1500, 255, 128)])
def test_decoding_step(dev, dtype, b, tk, prev, e):
    """Three steps in a row: the cache grows inside its buffer, into a new buffer, and from entries the caller replaced."""
    layer = randomised(DecoderLayer(options(e, 0.1, "relu")), dev, dtype, 6).eval()
    c = torch.randn(tk, b, e, device=dev).to(dtype)
    pad = torch.arange(tk, device=dev)[None] >= torch.randint((tk + 1) // 2, tk + 1, (b,), device=dev)[:, None]
    steps = torch.randn(3, 1, b, e, device=dev).to(dtype)
    prefix = torch.randn(prev, b, e, device=dev).to(dtype)
    res = []
    for by_operator in (False, True):
        handle = layer.feedforward.register_forward_hook(lambda m, i, o: None) if by_operator else None
        cache, outs = {}, []
        with torch.no_grad():
            layer(prefix, c, torch.triu(torch.ones(prev, prev, device=dev), 1).bool(), pad, incremental=True, incremental_cache=cache)
            for i in range(3):
                if i == 2:
                    order = torch.randperm(b, generator=torch.Generator().manual_seed(1)).to(dev)
                    for name in list(cache):
                        cache[name] = cache[name].index_select(1, order)
                out, coverage, cache = layer(steps[i], c, None, pad, incremental=True, incremental_cache=cache)
                outs += [out, coverage, cache["k"].clone(), cache["v"].clone()]
        res.append(outs)
        if handle is not None:
            handle.remove()
    same(res, dtype)


@pytest.mark.parametrize("tk", [64, 61])                    # the one-kernel inference path; stored scores
@pytest.mark.parametrize("shift", [0, 1, 2, 4])             # bytes the mask starts behind a multiple of eight
@pytest.mark.parametrize("probs", ["1", "0"])
@pytest.mark.parametrize("train", [True, False])
def test_a_mask_at_any_address_and_with_the_inference_kernel_switched_off(dev, monkeypatch, tk, shift, probs, train):
    e, tq, b, dtype = 128, 9, 3, F16
    monkeypatch.setenv("NMTG_ATTN_PROBS", probs)
    # gelu: the paths round the cross-attention at different points, and behind a relu a hidden element within that rounding of
    # zero would pass its whole gradient on one path and none on the other: of 27 x 256 hidden elements half of them live, one
    # is sqrt(1 / 3456) = 1.7e-2 of the gradient in front of it, beyond the 2e-3 that the roundings themselves are held to
    layer = randomised(DecoderLayer(options(e, 0.1, "gelu")), dev, dtype, 7).train(train)
    x = torch.randn(tq, b, e, device=dev).to(dtype).requires_grad_(train)
    c = torch.randn(tk, b, e, device=dev).to(dtype).requires_grad_(train)
    buf = torch.zeros(8 + b * tk, dtype=torch.uint8, device=dev)
    pad = buf[shift:shift + b * tk].view(b, tk)
    pad.copy_(torch.arange(tk, device=dev)[None] >= torch.tensor([tk, tk - 3, tk // 2], device=dev)[:, None])
    assert pad.data_ptr() % 8 == shift
    causal = torch.triu(torch.ones(tq, tq, device=dev), 1).bool()
    dy = torch.randn(tq, b, e, device=dev).to(dtype)
    with torch.set_grad_enabled(train):
        same(both_paths(layer, layer.feedforward, lambda: layer(x, c, causal, pad), [x, c] if train else [], dy if train else None), dtype)


@pytest.mark.parametrize("train", [True, False])
def test_a_forward_mode_tangent_is_refused_and_not_dropped(dev, train):
    import torch.autograd.forward_ad as fwd
    e, t, b = 128, 6, 2
    enc = randomised(EncoderLayer(options(e, 0.1, "gelu")), dev, F16, 8).train(train).requires_grad_(train)
    dec = randomised(DecoderLayer(options(e, 0.1, "gelu")), dev, F16, 8).train(train).requires_grad_(train)
    x = torch.randn(t, b, e, device=dev).half()
    causal, pad = torch.triu(torch.ones(t, t, device=dev), 1).bool(), torch.zeros(b, t, dtype=torch.bool, device=dev)
    cache = {}
    with torch.no_grad():
        dec.eval()(x, x, causal, pad, incremental=True, incremental_cache=cache)
    dec.train(train)
    with fwd.dual_level():
        dual = fwd.make_dual(x, torch.ones_like(x))
        for call in (lambda: enc(dual, pad), lambda: dec(dual, x, causal, pad), lambda: dec(x, dual, causal, pad), lambda: enc.feedforward(dual),
                     lambda: enc.preprocess_ffn(dual), lambda: enc.multihead(dual, None, pad, None)):
            with pytest.raises(RuntimeError, match="jvp"):
                call()
        if not train:
            with torch.no_grad(), pytest.raises(RuntimeError, match="jvp"):
                dec(dual[:1], x, None, pad, incremental=True, incremental_cache=dict(cache))
        for name in ("in_proj_weight", "in_proj_bias", "out_proj_bias"):
            w = getattr(enc.feedforward, name)
            with pytest.raises(RuntimeError, match="jvp"):
                torch.func.functional_call(enc.feedforward, {name: fwd.make_dual(w.detach(), torch.ones_like(w))}, (x,))
            with pytest.raises(RuntimeError, match="jvp"):
                torch.func.functional_call(enc, {"feedforward." + name: fwd.make_dual(w.detach(), torch.ones_like(w))}, (x, pad))


@pytest.mark.parametrize("where", ["preprocess_attn.layer_norm.function.weight", "multihead_tgt.in_proj_bias", "multihead_src.out_proj_weight",
                                   "feedforward.in_proj_weight"])
@pytest.mark.parametrize("train", [True, False])
def test_a_plain_tensor_in_the_place_of_a_parameter(dev, where, train):
    """As a hyper-network or a weight computed from another leaves it: deleted as a parameter, set as a tensor."""
    e, t, b = 128, 6, 2
    layer = randomised(DecoderLayer(options(e, 0.0, "gelu")), dev, F16, 9).train(train)
    x = torch.randn(t, b, e, device=dev).half().requires_grad_(train)
    causal, pad = torch.triu(torch.ones(t, t, device=dev), 1).bool(), torch.zeros(b, t, dtype=torch.bool, device=dev)
    with torch.set_grad_enabled(train):
        want = layer(x, x, causal, pad)[0]
        owner = layer.get_submodule(where.rsplit(".", 1)[0])
        name = where.rsplit(".", 1)[1]
        source = getattr(owner, name)
        delattr(owner, name)
        setattr(owner, name, source * 1.0)
        got = layer(x, x, causal, pad)[0]
        assert rel_err(got, want) < 2e-3
        if train:
            got.backward(torch.ones_like(got))
            assert source.grad is not None and torch.isfinite(source.grad).all() and source.grad.any()


@pytest.mark.parametrize("train", [True, False])
def test_shapes_that_do_not_fit_are_refused_before_a_kernel_sees_them(dev, train):
    e, t, b = 128, 6, 2
    enc = randomised(EncoderLayer(options(e, 0.1, "gelu")), dev, F16, 8).train(train)
    dec = randomised(DecoderLayer(options(e, 0.1, "gelu")), dev, F16, 8).train(train)
    causal, pad = torch.triu(torch.ones(t, t, device=dev), 1).bool(), torch.zeros(b, t, dtype=torch.bool, device=dev)
    x, wide, slim = (torch.randn(t, b, n, device=dev).half() for n in (e, 2 * e, e // 2))
    with torch.set_grad_enabled(train):
        for bad in (wide, slim):
            for call in (lambda: enc(bad, pad), lambda: dec(bad, bad, causal, pad), lambda: dec(x, bad, causal, pad)):
                with pytest.raises(RuntimeError):
                    call()
        if not train:
            cache = {}
            dec(x, x, causal, pad, incremental=True, incremental_cache=cache)
            with pytest.raises(RuntimeError):
                dec(wide[:1], x, None, pad, incremental=True, incremental_cache=dict(cache))
        for layer, call in ((enc, lambda: enc(x, pad)), (dec, lambda: dec(x, x, causal, pad))):
            for name in ("in_proj_weight", "out_proj_weight", "in_proj_bias", "out_proj_bias"):
                w = getattr(layer.feedforward, name)
                setattr(layer.feedforward, name, torch.nn.Parameter(w[:-8].detach().contiguous()))
                with pytest.raises(RuntimeError, match="mlp: (weight|bias) shape"):
                    call()
                setattr(layer.feedforward, name, w)
            call()


def test_a_traced_module_computes_on_its_new_inputs(dev):
    """torch.jit.trace records Python autograd functions and cannot see the host layer: what it cannot see would be a constant.
    (A layer's dropout + add works in place, which a traced program refuses to run.)"""
    e, t, b = 128, 6, 2
    enc = randomised(EncoderLayer(options(e, 0.1, "gelu")), dev, F16, 8).eval().requires_grad_(False)
    pad = torch.zeros(b, t, dtype=torch.bool, device=dev)
    x, new = torch.randn(2, t, b, e, device=dev).half()
    trace = lambda call, y: torch.jit.trace(call, (y,), check_trace=False)
    with torch.no_grad():
        for call in (enc.preprocess_ffn, enc.feedforward, lambda y: enc.multihead(y, None, pad)[0]):
            assert rel_err(trace(call, x)(new), call(new)) < 2e-3
        with pytest.raises(RuntimeError, match="not supported in the JIT"):
            trace(lambda y: enc(y, pad), x)(new)
    rows = torch.randn(2, 40, 100, device=dev).half()
    labels = torch.randint(0, 100, (40,), device=dev)
    loss = lambda z: SoftmaxCrossEntropyLoss.apply(z, labels, 0.1, 1, True)
    assert rel_err(trace(loss, rows[0])(rows[1]), loss(rows[1])) < 1e-5


def test_a_mask_in_host_memory_is_refused(dev):
    """Wherever a layer hands a mask's address to a kernel; on the native path and operator by operator."""
    e, tq, tk, b = 128, 5, 8, 2
    x, c = torch.randn(tq, b, e, device=dev).half(), torch.randn(tk, b, e, device=dev).half()
    causal = torch.triu(torch.ones(tq, tq, device=dev), 1).bool()
    good, bad = torch.zeros(b, tk, dtype=torch.bool, device=dev), torch.zeros(b, tk, dtype=torch.bool)
    dec = randomised(DecoderLayer(options(e, 0.1, "relu")), dev, F16, 5)
    enc = randomised(EncoderLayer(options(e, 0.1, "relu")), dev, F16, 5)
    for by_operator in (False, True):
        handles = [m.feedforward.register_forward_hook(lambda m, i, o: None) for m in (dec, enc) if by_operator]
        for train in (True, False):
            with torch.set_grad_enabled(train):
                for call in (lambda: enc.train(train)(c, bad), lambda: dec.train(train)(x, c, causal, bad),
                             lambda: dec.train(train)(x, c, causal.cpu(), good)):
                    with pytest.raises(RuntimeError, match="expected a tensor|must be contiguous uint8"):
                        call()
        with torch.no_grad():
            dec.eval()
            cache = {}
            dec(x, c, causal, good, incremental=True, incremental_cache=cache)
            for mask in (bad, bad[:, None]):
                with pytest.raises(RuntimeError, match="expected a tensor|key mask of shape"):
                    dec(x[:1], c, None, mask, incremental=True, incremental_cache=dict(cache))
            with pytest.raises(RuntimeError, match="expected a tensor"):
                dec(x[:1], c, None, good, incremental=True, incremental_cache=dict(cache, c_k=cache["c_k"].cpu()))
            assert torch.isfinite(dec(x[:1], c, None, good, incremental=True, incremental_cache=cache)[0]).all()
        for h in handles:
            h.remove()


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
def test_a_stream_that_is_not_finite_is_clamped_and_its_gradient_stops(dev, dtype, bad):
    layer = randomised(EncoderLayer(options(128, 0.1, "relu")), dev, dtype, 4).train()
    x = torch.randn(9, 3, 128, device=dev).to(dtype)
    x[2, 1, 5] = 65000.0 if dtype == F16 else 3e38            # above fp16's bound: clamped with the rest of the tensor
    with torch.no_grad():
        layer.feedforward.out_proj_bias[7] = bad
    x.requires_grad_()
    pad = torch.zeros(3, 9, dtype=torch.bool, device=dev)
    pair = both_paths(layer, layer.feedforward, lambda: layer(x, pad), [x], torch.randn(9, 3, 128, device=dev).to(dtype))
    out = pair[0][0]
    assert torch.equal(torch.nan_to_num(out, nan=0.5), torch.nan_to_num(pair[1][0], nan=0.5))
    if not math.isnan(bad):
        assert torch.isfinite(out).all() and out.abs().max().item() >= 64512
    same([pair[0][1:], pair[1][1:]], dtype)


def add_ln(x, r, gamma, beta, p, seed):
    rows, hidden = x.shape
    h, z = torch.empty_like(x), torch.empty_like(x)
    mask = torch.full((rows, hidden), 9, dtype=torch.uint8, device=x.device)
    mu, rs = torch.empty(rows, device=x.device), torch.empty(rows, device=x.device)
    flag = torch.ones(1, dtype=torch.int32, device=x.device)
    import ctypes
    L.call("nmtg_add_ln_fwd", L.ptr(x), L.ptr(r), L.ptr(h), L.ptr(mask), L.i32(2 if p else 0), L.f32(p), ctypes.c_uint64(seed), ctypes.c_uint64(8),
           L.ptr(flag), L.ptr(gamma), L.ptr(beta), L.ptr(z), L.ptr(mu), L.ptr(rs), L.i64(rows), L.i64(hidden), L.f32(1e-5),
           L.i32(L.dtype_code(x)), L.stream_of(x))
    assert flag.item() == 0
    return h, mask, z, mu, rs


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (5, 7), (3, 520), (67, 512), (9, 2056), (2, 8200)])
@pytest.mark.parametrize("p", [0.0, 0.25])
def test_layer_norm_over_a_residual_sum(dev, dtype, rows, hidden, p):
    import ctypes
    g = torch.Generator().manual_seed(rows * hidden)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    x, r, gamma, beta, dz, dr = mk(rows, hidden), mk(rows, hidden), mk(hidden), mk(hidden), mk(rows, hidden), mk(rows, hidden)
    h, mask, z, mu, rs = add_ln(x, r, gamma, beta, p, 77)
    want_h, want_mask = x.clone(), torch.ones(rows, hidden, dtype=torch.uint8, device=dev)
    L.call("nmtg_dropout_add_fwd", L.ptr(want_h), L.ptr(r), L.ptr(want_mask), L.i64(x.numel()), L.f32(p), L.i32(2 if p else 0), ctypes.c_uint64(77),
           ctypes.c_uint64(8), L.i32(L.dtype_code(x)), L.stream_of(x))
    assert torch.equal(h, want_h)
    if p:
        assert torch.equal(mask, want_mask)
    want_z, want_mu, want_rs = ln.ln_fwd(want_h, gamma, beta, 1e-5)
    for a, b in ((z, want_z), (mu, want_mu), (rs, want_rs)):         # the compiler fuses a multiply-add here or there
        assert rel_err(a, b) < 1e-4
    # backward: the LayerNorm's gradient plus the stream's (not where the guard byte says so), and the dropped branch's
    guard = (torch.rand(rows, hidden, generator=g) < 0.2).to(torch.uint8).mul_(2).to(dev)
    keep = (torch.rand(rows, hidden, generator=g) < 0.7).to(torch.uint8).to(dev)
    plain = ln.ln_bwd(dz, h, mu, rs, gamma, None, False)
    parts = plain[3].shape[0]
    for use_guard in (False, True):
        for drop in (False, True):
            dx, dy, dg, db = torch.empty_like(x), torch.empty_like(x), torch.empty_like(gamma), torch.empty_like(gamma)
            part = torch.empty(2, parts, hidden, device=dev)
            L.call("nmtg_ln_bwd_add", L.ptr(dz), L.ptr(h), L.ptr(mu), L.ptr(rs), L.ptr(gamma), L.ptr(dr), L.ptr(guard if use_guard else None),
                   L.ptr(keep if drop else None), L.f32(0.25), L.ptr(dx), L.ptr(dy if drop else None), L.ptr(dg), L.ptr(db), L.ptr(part[0]),
                   L.ptr(part[1]), L.i64(parts), L.i64(rows), L.i64(hidden), L.i32(L.dtype_code(x)), L.stream_of(x))
            want = plain[0] + (dr.masked_fill(guard != 0, 0.0) if use_guard else dr)
            assert torch.equal(dg, plain[1]) and torch.equal(db, plain[2])
            assert rel_err(dx, want) < 1e-4                            # a fused multiply-add here or there
            assert_close(dx, want.double().cpu(), dtype, "dx", atol=1e-5)
            if drop:
                assert_close(dy, want.double().cpu() * keep.cpu() / 0.75, dtype, "dy", atol=1e-5 if dtype == F32 else None)


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("n", [1, 7, 4096, 70003])
def test_guarded_dropout_add(dev, dtype, n):
    import ctypes
    g = torch.Generator().manual_seed(n)
    x, r = torch.randn(n, generator=g).to(dtype).to(dev), torch.randn(n, generator=g).to(dtype).to(dev)
    for p in (0.0, 0.5):
        for bad in (None, math.inf, math.nan):
            src = r.clone()
            if bad is not None:
                src[n // 2] = bad
                if dtype == F16:
                    src[n - 1] = 65504.0 if n > 1 else bad
            want, mask = x.clone(), torch.ones(n, dtype=torch.uint8, device=dev)
            L.call("nmtg_dropout_add_fwd", L.ptr(want), L.ptr(src), L.ptr(mask), L.i64(n), L.f32(p), L.i32(2 if p else 0), ctypes.c_uint64(5),
                   ctypes.c_uint64(4), L.i32(L.dtype_code(x)), L.stream_of(x))
            ref = want.clone().requires_grad_()
            out = ref * 1.0
            if not bool(torch.isfinite(out).all()):
                out = out.clamp(-(torch.finfo(dtype).max - 1000), torch.finfo(dtype).max - 1000)
            out.backward(torch.ones_like(out))
            got, gm = x.clone(), torch.empty(n, dtype=torch.uint8, device=dev)
            flag = torch.zeros(1, dtype=torch.int32, device=dev)
            L.call("nmtg_dropout_add_guard_fwd", L.ptr(got), L.ptr(src), L.ptr(gm), L.i64(n), L.f32(p), L.i32(2 if p else 0), ctypes.c_uint64(5),
                   ctypes.c_uint64(4), L.ptr(flag), L.i32(L.dtype_code(x)), L.stream_of(x))
            assert torch.equal(torch.nan_to_num(got, nan=0.25), torch.nan_to_num(out.detach(), nan=0.25))
            assert torch.equal(gm & 1, mask) and torch.equal((gm & 2) == 0, ref.grad != 0)
            dx = torch.empty_like(x)
            L.call("nmtg_dropout_add_guard_bwd", L.ptr(r), L.ptr(gm), L.ptr(dx), L.i64(n), L.f32(p), L.i32(L.dtype_code(x)), L.stream_of(x))
            assert_close(dx, r.double().cpu() * (gm == 1).cpu() / (1 - p), dtype, "dx")
