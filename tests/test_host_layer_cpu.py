"""What the native host layer (nmtgminor_amd/_host.so) decides before it touches a GPU: it loads and binds without one."""
from types import SimpleNamespace

import pytest
import torch

from nmtgminor_amd import _lib as L
from nmtgminor_amd.modules.pre_post_processing import PrePostProcessing
from nmtgminor_amd.modules.transformer_layers import DecoderLayer, EncoderLayer


def test_the_host_layer_loads_and_finds_every_entry_point():
    assert L.host().bind is not None                    # L.host() has bound it: a missing symbol raises there


@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.int64])
def test_a_mask_becomes_bytes_on_the_device_of_its_operand(dtype):
    x = torch.empty(3, 2, 8)
    mask = torch.tensor([[0, 1, 1], [0, 0, 1]]).to(dtype)
    got = L.host().mask_bytes(mask.t().contiguous().t(), x, 2, 3)
    assert got.dtype == torch.uint8 and got.is_contiguous() and got.tolist() == [[0, 1, 1], [0, 0, 1]]
    assert L.host().mask_bytes(None, x, 2, 3) is None and L.host().mask_bytes(mask[:0], x, 0, 3) is None
    with pytest.raises(RuntimeError, match="mask must be"):
        L.host().mask_bytes(mask, x, 3, 3)
    with pytest.raises(RuntimeError, match="expected a tensor on meta, got one on cpu"):
        L.host().mask_bytes(mask, x.to("meta"), 2, 3)   # the address of a host mask is nothing for a kernel


def test_operands_of_a_call_share_a_device():
    meta = torch.empty(5, 8, device="meta")
    hidden = torch.empty(5 * 16, dtype=torch.uint8)
    with pytest.raises(RuntimeError, match="expected a tensor"):
        L.host().mlp(meta, torch.empty(16, 8), torch.empty(8, 16), None, None, hidden, 0.1, L.ACT_RELU)
    step = [torch.empty(1, 2, 64, device="meta")] + [torch.empty(4, 2, 64, device="meta")] * 2
    for at in range(5):
        cache = [torch.empty(4, 2, 64, device="cpu" if i == at else "meta") for i in range(4)]
        pad = torch.zeros(2, 4, dtype=torch.uint8, device="cpu" if at == 4 else "meta")
        with pytest.raises(RuntimeError, match="expected a tensor on meta, got one on cpu"):
            L.host().decoder_step(step[0], cache[0], cache[1], 3, cache[2], cache[3], pad, [], 1, L.ACT_RELU)


def _layers():
    opt = SimpleNamespace(model_size=128, inner_size=256, n_heads=2, dropout=0.1, attn_dropout=0.1, ffn_activation="swish")
    yield EncoderLayer(opt), ("preprocess_attn", "preprocess_ffn"), 12
    yield DecoderLayer(opt), ("preprocess_attn", "preprocess_src_attn", "preprocess_ffn"), 17


LISTEN = {"forward_hook": lambda m: m.register_forward_hook(lambda *a: None),
          "forward_pre_hook": lambda m: m.register_forward_pre_hook(lambda *a: None),
          "backward_hook": lambda m: m.register_full_backward_hook(lambda *a: None),
          "backward_pre_hook": lambda m: m.register_full_backward_pre_hook(lambda *a: None)}


@pytest.mark.parametrize("kind", list(LISTEN) + ["forward", "mode"])
def test_what_listens_to_a_sub_module_keeps_the_layer_off_the_native_form(kind):
    """At any depth: the operators call every sub-module, the native form none."""
    for layer, pre, count in _layers():
        def native():
            return layer._sub_parameters(pre, layer._SUB) is not None
        assert native() and len(layer._sub_parameters(pre, layer._SUB)) == count
        inner = [(n, m) for n, m in layer.named_modules() if n]
        assert {type(m).__name__ for _, m in inner} >= {"PrePostProcessing", "Bottle", "LayerNorm", "Dropout", "SelfMultiheadAttn",
                                                        "PositionWiseFeedForward"}
        for name, m in inner:
            if kind == "forward":
                plain = m.forward
                m.forward = lambda *a, **k: plain(*a, **k)
                assert not native(), name
                del m.forward
            elif kind == "mode":
                if type(m).__name__ in ("Bottle", "LayerNorm"):
                    continue                              # no difference between their modes
                m.train(not layer.training)
                assert not native(), name
                layer.train(layer.training)
            else:
                handle = LISTEN[kind](m)
                assert not native(), name
                handle.remove()
            assert native(), name


def test_hooks_on_every_module_and_replaced_functions_keep_the_layer_off_the_native_form():
    from torch.nn.modules import module as mod
    for layer, pre, _ in _layers():
        def native():
            return layer._sub_parameters(pre, layer._SUB) is not None
        for register in (mod.register_module_forward_hook, mod.register_module_forward_pre_hook, mod.register_module_full_backward_hook,
                         mod.register_module_full_backward_pre_hook):
            handle = register(lambda *a: None)
            assert not native()
            handle.remove()
            assert native()
        for name, m in layer.named_modules():
            for function in ("attn_func", "fused_function"):
                if hasattr(m, function):
                    plain = getattr(m, function)
                    setattr(m, function, lambda *a, **k: plain(*a, **k))
                    assert not native(), name
                    setattr(m, function, plain)
        layer.postprocess_attn.dropout.p = 0.3
        assert not native()


class _View(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return (2 * x).view(2, 3, 4)

    @staticmethod
    def backward(ctx, g):
        return 2 * g.view(24)


def test_dropout_and_add_draw_alike_with_and_without_gradients():
    """The forward of a reentrant checkpoint runs without gradients and its recomputation with them: a result that is a view of an
    autograd function's own tensor takes torch's dropout in both."""
    post = PrePostProcessing(4, 0.5, sequence="da").train()
    x, residual = torch.ones(24, requires_grad=True), torch.zeros(2, 3, 4)
    with_gradients = post._fusable(0, _View.apply(x), residual)
    with torch.no_grad():
        assert post._fusable(0, _View.apply(x), residual) is with_gradients is False
        assert post._fusable(0, _View.apply(x).clone(), residual) is post.eval()._fusable(0, _View.apply(x), residual) is True
