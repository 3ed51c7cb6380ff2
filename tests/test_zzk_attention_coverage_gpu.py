"""Attention in training with its coverage on the tiled core (csrc/host/attention.cpp): outputs, probabilities and gradients
against the formula in fp64 under the dropout mask that the extension modules draw for the same generator state."""
import pytest
import torch

from nmtgminor_amd.modules.encdec_attention_func import encdec_attn_func
from nmtgminor_amd.modules.encdec_attention_func_bias import encdec_attn_bias_func
from nmtgminor_amd.modules.self_attention_func import self_attn_func
from nmtgminor_amd.native import encdec_multihead_attn_bias_blaslt, encdec_multihead_attn_cuda, self_multihead_attn_blaslt

pytestmark = pytest.mark.gpu
D = torch.float64
P = 0.2


def core(q, k, v, dead, keep, heads):
    """q [Tq, B, E], k / v [Tk, B, E], dead broadcastable to [B, H, Tq, Tk] -> context, probabilities, dropped ones [B * H, Tq, Tk]"""
    tq, b, e = q.shape
    split = lambda t: t.reshape(t.shape[0], b, heads, e // heads).permute(1, 2, 0, 3)
    s = (split(q) @ split(k).transpose(2, 3)) * (e // heads) ** -0.5
    prob = torch.softmax(s.masked_fill(dead, float("-inf")), -1).nan_to_num(0.0) if dead is not None else torch.softmax(s, -1)
    dropped = prob * keep.view_as(prob).to(D) / (1 - P)
    ctx = (dropped @ split(v)).permute(2, 0, 1, 3).reshape(tq, b, e)
    flat = lambda t: t.reshape(b * heads, tq, -1).detach()
    return ctx, flat(prob), flat(dropped)


def close(got, want, dtype):
    for a, w in zip([x.detach() for x in got], want):
        assert a.shape == w.shape and torch.isfinite(a).all()
        size = max(float(w.norm()), 0.5 * w.numel() ** 0.5)          # few keys: gradients of the scores are next to nothing
        assert float((a.to(D) - w).norm()) / size < (1.2e-2 if dtype == torch.bfloat16 else 2e-3)


def tensors(shapes, dtype, dev, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for i, s in enumerate(shapes):
        scale = 1.0 if len(s) == 3 else s[-1] ** -0.5 if len(s) == 2 else 0.1
        out.append((scale * torch.randn(s, generator=g)).to(dtype).to(dev).requires_grad_())
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("t,b,e,heads,mask", [(1, 2, 64, 1, None), (37, 3, 128, 2, "pad"), (64, 2, 256, 2, "time"), (130, 2, 128, 2, "time"),
                                              (201, 2, 256, 4, "pad"), (512, 1, 128, 2, "pad"), (640, 1, 128, 1, None), (72, 5, 192, 3, "time")])
@pytest.mark.parametrize("bias", [True, False])
def test_self_attention_with_coverage(dev, dtype, t, b, e, heads, mask, bias):
    x, wi, wo, bi, bo = tensors([(t, b, e), (3 * e, e), (e, e), (3 * e,), (e,)], dtype, dev, t)
    if not bias:
        bi = bo = None
    m = dead = None
    if mask == "pad":
        m = torch.arange(t, device=dev)[None] >= torch.randint((t + 1) // 2, t + 1, (b,), device=dev)[:, None]
        m[0, 0] = True                                            # a masked key in front of the live ones
        dead = m[:, None, None, :]
    elif mask == "time":
        m = torch.triu(torch.ones(t, t, device=dev), 1).bool()
        dead = m[None, None]
    dy = torch.randn(t, b, e, device=dev).to(dtype)
    torch.cuda.manual_seed(11)
    drawn = self_multihead_attn_blaslt.forward(mask == "time", True, heads, *(z if z is None else z.detach() for z in (x, wi, wo, bi, bo)), m, P)
    ins = [z for z in (x, wi, wo, bi, bo) if z is not None]
    xd, wid, wod = (z.detach().to(D).requires_grad_() for z in (x, wi, wo))
    bid, bod = (None if z is None else z.detach().to(D).requires_grad_() for z in (bi, bo))
    lin = torch.nn.functional.linear(xd, wid, bid).view(t, b, heads, 3, e // heads)
    ctx, _, dropped = core(*(lin[:, :, :, i].reshape(t, b, e) for i in range(3)), dead, drawn[3], heads)
    out = torch.nn.functional.linear(ctx, wod, bod)
    want = [out.detach(), dropped] + list(torch.autograd.grad(out, [z for z in (xd, wid, wod, bid, bod) if z is not None], dy.to(D)))
    torch.cuda.manual_seed(11)
    y, cov = self_attn_func(mask == "time", True, heads, x, wi, wo, bi, bo, m, P, False, None, False, None, True, True, False)
    assert y.grad_fn.name().find("SelfAttentionNode") >= 0 and not cov.requires_grad
    close([y, cov] + list(torch.autograd.grad(y, ins, dy)), want, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tq,tk,b,e,heads", [(1, 3, 1, 64, 1), (5, 130, 3, 128, 2), (61, 73, 4, 128, 2), (129, 64, 2, 256, 2), (40, 700, 2, 64, 1)])
@pytest.mark.parametrize("bias", [True, False])
def test_encoder_decoder_attention_with_coverage(dev, dtype, tq, tk, b, e, heads, bias):
    ins = tensors([(tq, b, e), (tk, b, e), (e, e), (2 * e, e), (e, e)] + ([(e,), (2 * e,), (e,)] if bias else []), dtype, dev, tk)
    m = torch.arange(tk, device=dev)[None] >= torch.randint((tk + 1) // 2, tk + 1, (b,), device=dev)[:, None]
    dy = torch.randn(tq, b, e, device=dev).to(dtype)
    det = [z.detach() for z in ins]
    torch.cuda.manual_seed(12)
    keep = (encdec_multihead_attn_bias_blaslt.forward(True, heads, *det[:5], *det[5:], m, P) if bias
            else encdec_multihead_attn_cuda.forward(True, heads, *det, m, P))[4]
    ref = [z.detach().to(D).requires_grad_() for z in ins]
    bq, bkv, bo = ref[5:] if bias else (None, None, None)
    kv = torch.nn.functional.linear(ref[1], ref[3], bkv).view(tk, b, heads, 2, e // heads)
    ctx, prob, dropped = core(torch.nn.functional.linear(ref[0], ref[2], bq), kv[:, :, :, 0].reshape(tk, b, e), kv[:, :, :, 1].reshape(tk, b, e),
                              m[:, None, None, :], keep, heads)
    out = torch.nn.functional.linear(ctx, ref[4], bo)
    want = [out.detach(), dropped if bias else prob] + list(torch.autograd.grad(out, ref, dy.to(D)))
    torch.cuda.manual_seed(12)
    if bias:
        y, cov = encdec_attn_bias_func(False, True, heads, *ins, m, P, False, None, False, None, None, True, True)
    else:
        y, cov = encdec_attn_func(False, True, heads, *ins, m, P, False, None, False, None, None, False, True)
    assert y.grad_fn.name().find("CrossAttentionNode") >= 0
    close([y, cov] + list(torch.autograd.grad(y, ins, dy)), want, dtype)
