"""Products whose reduction ends inside a 64-element step (token counts, vocabularies), split and unsplit, and the loss
backward with the column sums of its result."""
import pytest
import torch

from nmtgminor_amd.native import linear_gemm, xentropy_cuda
from util import assert_close

pytestmark = pytest.mark.gpu
D = torch.float64


def _pitched(rows, cols, dtype, dev, g, poison):
    """[rows, cols] view of rows padded to 16 bytes; what lies behind a row's end is NaN."""
    pitch = (cols + 7) // 8 * 8
    full = torch.full((rows, pitch), float("nan") if poison else 0.0)
    full[:, :cols] = torch.randn(rows, cols, generator=g)
    return full.to(dtype).to(dev)[:, :cols]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k", [1, 7, 63, 65, 127, 200, 1031, 4097])
@pytest.mark.parametrize("m,n,trans_a", [(72, 128, True), (320, 264, True), (72, 128, False), (300, 520, False), (2048, 512, True)])
def test_reduction_that_ends_inside_a_step(dev, dtype, k, m, n, trans_a):
    g = torch.Generator().manual_seed(k * 1000 + m)
    a = _pitched(k, m, dtype, dev, g, True) if trans_a else _pitched(m, k, dtype, dev, g, True)
    b = _pitched(k, n, dtype, dev, g, True)
    want = (a.t() if trans_a else a).cpu().to(D) @ b.cpu().to(D)
    for split in (True, False):
        got = linear_gemm.gemm(a, b, trans_a=trans_a, split_k=split)
        assert_close(got, want, dtype, f"k {k} split {split}", scale_atol=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", [(1, 5), (7, 2047), (128, 2049), (129, 4104), (300, 10007)])
@pytest.mark.parametrize("one_grad", [False, True])
def test_loss_backward_with_column_sums(dev, dtype, rows, vocab, one_grad):
    g = torch.Generator().manual_seed(rows + vocab)
    pitch = (vocab + 63) // 64 * 64
    full = torch.zeros(rows, pitch, dtype=dtype, device=dev)
    z = full[:, :vocab]
    z.copy_(2 * torch.randn(rows, vocab, generator=g))
    labels = torch.randint(0, vocab, (rows,), generator=g).to(dev)
    labels[::3] = 1
    _, lse = xentropy_cuda.forward(z, labels, 0.1, True, padding_idx=1)
    grad = torch.randn(1 if one_grad else rows, generator=g).to(dev)
    want = xentropy_cuda.backward(grad.expand(rows), z, lse, labels, 0.1, padding_idx=1)
    got, sums = xentropy_cuda.backward_with_colsum(grad, z, lse, labels, 0.1, 1, z)
    assert_close(got, want.cpu().to(D), dtype, "gradient", scale_atol=True)
    assert_close(sums, want.cpu().to(D).sum(0), dtype, "column sums", scale_atol=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(4200, 4100, 192), (4096, 4352, 256), (256 * 300 + 8, 256, 320), (264, 256 * 260 + 24, 1024)])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
def test_more_tiles_than_compute_units(dev, dtype, m, n, k, layout):
    """One block per unit walks several 256 x 256 tiles: whole ones, ragged ends in both directions, uneven shares."""
    g = torch.Generator(device=dev).manual_seed(m + k)
    make = lambda r, c: torch.randn(r, c, generator=g, device=dev).to(dtype)
    a, b = make(k, m) if layout == "tn" else make(m, k), make(n, k) if layout == "nt" else make(k, n)
    bias = make(1, n)[0] if layout == "nt" else None
    pitched = torch.full((m, n + 8), 7.0, dtype=dtype, device=dev)
    got = linear_gemm.gemm(a, b, trans_a=layout == "tn", trans_b=layout == "nt", bias=bias, out=pitched[:, :n], split_k=False)
    want = (a.t() if layout == "tn" else a).float() @ (b.t() if layout == "nt" else b).float() + (0 if bias is None else bias.float())
    bound = (5e-3 if dtype == torch.float16 else 4e-2) * k ** 0.5
    for r in range(0, m, 8192):
        assert float((got[r:r + 8192].float() - want[r:r + 8192]).abs().max()) < bound
    assert bool((pitched[:, n:] == 7.0).all())
