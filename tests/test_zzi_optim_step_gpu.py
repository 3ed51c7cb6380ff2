"""Gradient clipping with the factor on the device, and the optimizer's step through the host layer: list lengths around the
kernels' tables, tensors around the block size, unaligned storage, and what the host layer leaves to the Python side."""
import pytest
import torch

from nmtgminor_amd.modules.fused_adam import FusedAdam
from nmtgminor_amd.modules.fused_clip_norm import fused_clip_grad_norm
from nmtgminor_amd.native import fused_optim
from oracle import fused_optim as ofo
from util import assert_close

pytestmark = pytest.mark.gpu
D = torch.float64


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sizes", [[1], [8191, 8192, 8193, 0, 3 * 8192 + 4], [5] * 160, [65] * 161 + [40000]])
@pytest.mark.parametrize("max_norm", [0.25, 1e9])
def test_clip_factor_on_the_device(dev, dtype, sizes, max_norm):
    g = torch.Generator().manual_seed(len(sizes))
    grads = [torch.randn(n, generator=g).to(dtype) for n in sizes]
    params = [torch.zeros(n, dtype=dtype, device=dev).requires_grad_() for n in sizes]
    for p, x in zip(params, grads):
        store = torch.empty(x.numel() + 1, dtype=dtype, device=dev)                  # every other one starts off a 16-byte boundary
        p.grad = store[1:] if p is params[-1] else store[:x.numel()]
        p.grad.copy_(x)
    norm = fused_clip_grad_norm(params, max_norm)
    want, _ = ofo.l2norm(grads, D)
    assert norm.dim() == 0
    assert_close(norm, want, torch.float32, "norm", rtol=2e-6)
    factor = min(1.0, max_norm / (float(want) + 1e-6))
    for p, x in zip(params, grads):
        if factor == 1.0:
            assert torch.equal(p.grad.cpu(), x)
        else:
            assert_close(p.grad, x.to(D) * factor, dtype, f"clipped gradient of {x.numel()}", atol=1e-6 if dtype == torch.float32 else None)


def test_a_non_finite_norm_spoils_every_gradient(dev):
    params = [torch.zeros(9000, device=dev).requires_grad_() for _ in range(3)]
    for bad in (float("nan"), float("inf")):
        for p in params:
            p.grad = torch.ones_like(p)
        params[1].grad[8500] = bad
        norm = fused_clip_grad_norm(params, 1.0)
        assert not torch.isfinite(norm)
        if bad != bad:
            assert all(torch.isnan(p.grad).all() for p in params)
        else:                                                              # 1 / inf = 0; inf * 0 is NaN
            assert torch.isnan(params[1].grad[8500]) and float(params[0].grad.abs().sum()) == 0.0


@pytest.mark.parametrize("mixed", [False, True])
def test_step_of_the_host_layer_is_that_of_the_lists(dev, mixed):
    shapes = [(33, 7), (8193,), (1,), (0,)] + [(17,)] * 90
    g = torch.Generator().manual_seed(4)
    make = lambda i: torch.randn(shapes[i], generator=g).to(torch.bfloat16 if mixed and i % 3 == 0 else torch.float32)
    values = [[make(i) for i in range(len(shapes))] for _ in range(4)]
    a = [v.to(dev).requires_grad_() for v in values[0]]
    b = [v.to(dev) for v in values[0]]
    m, v = [torch.zeros_like(x) for x in b], [torch.zeros_like(x) for x in b]
    opt = FusedAdam(a, lr=1e-2, betas=(0.9, 0.98), weight_decay=0.01)
    for step in range(1, 4):                                               # the first creates the moments on the Python side
        for x, w in zip(a, values[step]):
            x.grad = w.to(dev)
        opt.step()
        for dtype in (torch.float32, torch.bfloat16):
            at = [i for i in range(len(b)) if b[i].dtype == dtype]
            if at:
                fused_optim.multi_tensor_adam(0, None, [[a[i].grad for i in at], [b[i] for i in at], [m[i] for i in at], [v[i] for i in at]],
                                              1e-2, 0.9, 0.98, 1e-8, step, 1, 1, 0.01)
    for i, x in enumerate(a):
        assert torch.equal(x.detach(), b[i]) and torch.equal(opt.state[x]["exp_avg"], m[i]) and torch.equal(opt.state[x]["exp_avg_sq"], v[i]), i
    a[0].grad = a[0].grad.t().contiguous().t()                             # a layout the host layer refuses: same step
    opt.step()
    assert torch.isfinite(a[0]).all()
