"""What the native host layer (nmtgminor_amd/_host.so) decides before it touches a GPU: it loads and binds without one."""
import pytest
import torch

from nmtgminor_amd import _lib as L


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
