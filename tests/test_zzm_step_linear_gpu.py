"""nmtg_step_linear: a decoding step's product with the LayerNorm in front of it, and with the activation or the layer's guarded
addition behind it, against fp64 with the rounding points of the separate kernels (h, the normalised row, the product with its
bias, the result)."""
import math

import pytest
import torch

from nmtgminor_amd import _lib as L

pytestmark = pytest.mark.gpu
ACTS = {"none": lambda v: v, "relu": torch.relu, "gelu": lambda v: 0.5 * v * (1 + torch.erf(v / math.sqrt(2))), "silu": lambda v: v * torch.sigmoid(v)}


def step(x, w, bias, dtype, *, residual=None, gamma=None, beta=None, act="none", add=None, y=None, h=None):
    rows, out = x.shape[0], w.shape[0]
    dev = x.device
    y = torch.full((rows, out), 7.0, dtype=dtype, device=dev) if y is None else y
    h = torch.full_like(x, 7.0) if residual is not None and h is None else h
    clear = torch.full((1,), 5, dtype=torch.int32, device=dev) if gamma is not None else None
    guard = torch.zeros(1, dtype=torch.int32, device=dev) if add is not None else None
    L.call("nmtg_step_linear", L.i64(rows), L.i64(out), L.i64(x.shape[1]), L.ptr(x), L.ptr(residual), L.ptr(gamma), L.ptr(beta), L.f32(1e-5),
           L.ptr(h), L.ptr(clear), L.ptr(w), L.ptr(bias), L.i32(L.ACT_CODES[act]), L.ptr(add), L.ptr(guard), L.ptr(y), L.i32(L.dtype_code(x)),
           L.stream_of(x))
    if clear is not None:
        assert clear.tolist() == [0]
    return y, h


def tensors(dev, dtype, rows, out, k, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s, scale=1.0: (scale * torch.randn(*s, generator=g)).to(dtype).to(dev)
    return dict(x=r(rows, k), w=r(out, k, scale=k ** -0.5), bias=r(out, scale=0.1), residual=r(rows, k), gamma=r(k, scale=0.1) + 1, beta=r(k, scale=0.1),
                add=r(rows, out))


def close(got, want, dtype, what):
    """Three roundings on the way, each to half a unit of values whose magnitude the last factor covers; fp32 sums of at most 4096 terms."""
    eps = torch.finfo(dtype).eps
    want = want.cpu()
    err = (got.double().cpu() - want).abs()
    assert bool((err <= 3 * eps * (want.abs() + want.abs().mean() + 0.25)).all()), (what, float(err.max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,out,k", [(1, 64, 64), (5, 100, 512), (31, 96, 520), (33, 64, 1024), (64, 130, 128), (8, 2048, 1016)])
@pytest.mark.parametrize("pre,act", [("none", "none"), ("none", "gelu"), ("norm", "none"), ("add", "none"), ("add", "relu"), ("add", "gelu"), ("add", "silu")])
def test_normalisation_product_activation(dev, dtype, rows, out, k, pre, act):
    t = tensors(dev, dtype, rows, out, k, rows + k)
    y, h = step(t["x"], t["w"], t["bias"], dtype, act=act, residual=t["residual"] if pre == "add" else None, gamma=None if pre == "none" else t["gamma"],
                beta=t["beta"])
    z = t["x"].double()
    if pre == "add":
        z = (z + t["residual"].double()).to(dtype)
        assert torch.equal(h, z)
        z = z.double()
    if pre != "none":
        z = torch.nn.functional.layer_norm(z, (k,), t["gamma"].double(), t["beta"].double(), 1e-5).to(dtype).double()
    v = (z @ t["w"].double().t() + t["bias"].double()).to(dtype).double()
    close(y, ACTS[act](v), dtype, f"{rows} x {out} x {k} {pre} {act}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,out,k", [(2, 64, 64), (5, 512, 2048), (40, 72, 136)])
@pytest.mark.parametrize("spoilt", [False, True])
def test_product_and_guarded_addition(dev, dtype, rows, out, k, spoilt):
    """With an element that is not finite every fp16 element beyond the bound is clamped, in whichever block it lies."""
    t = tensors(dev, dtype, rows, out, k, rows)
    big = torch.finfo(dtype).max
    if spoilt:
        t["add"][0, 0], t["add"][-1, -1], t["add"][-1, 0], t["add"][0, -1] = float("inf"), float("nan"), -big, big
    y, _ = step(t["x"], t["w"], None, dtype, add=t["add"])
    want = t["add"].double() + (t["x"].double() @ t["w"].double().t()).to(dtype).double()
    if spoilt:
        limit = 64512.0 if dtype == torch.float16 else big
        assert torch.isnan(y[-1, -1]) and torch.isfinite(y).sum() == y.numel() - 1
        for at in ((0, 0), (0, -1)):
            assert float(y[at]) == limit
        assert float(y[-1, 0]) == -limit
        keep = torch.ones_like(y, dtype=torch.bool)
        for at in ((0, 0), (-1, -1), (-1, 0), (0, -1)):
            keep[at] = False
        y, want = y[keep], want[keep.to(want.device)]
    close(y, want, dtype, f"{rows} x {out} x {k}")


def test_outputs_over_inputs_are_refused(dev):
    """One block's outputs are other blocks' inputs: such calls are refused whatever their size, whole or in part. y = add stays."""
    dtype = torch.bfloat16
    t = tensors(dev, dtype, 5, 512, 512, 1)
    norm = dict(gamma=t["gamma"], beta=t["beta"])
    both = torch.zeros(8, 512, dtype=dtype, device=dev)                       # two overlapping tensors of five rows
    low, high = both[:5], both[3:]
    for kw in (dict(residual=t["residual"], h=t["residual"], **norm), dict(residual=t["residual"], h=t["x"], **norm),
               dict(residual=t["residual"], y=t["residual"], **norm), dict(residual=t["residual"], y=t["x"], **norm), dict(y=t["x"], **norm), dict(y=t["x"]),
               dict(residual=low, h=high, **norm), dict(residual=t["residual"], y=low, h=high, **norm), dict(add=low, y=high), dict(y=t["w"][:5]),
               dict(residual=t["residual"], h=t["w"][-5:], **norm)):
        with pytest.raises(RuntimeError, match="overlap"):
            step(t["x"], t["w"], t["bias"], dtype, **kw)
    want = t["add"].double() + (t["x"].double() @ t["w"].double().t()).to(dtype).double()
    y, _ = step(t["x"], t["w"], None, dtype, add=t["add"], y=t["add"])
    close(y, want, dtype, "y = add")
