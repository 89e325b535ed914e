"""The bias table's gradient added from workspace slots: the same bits every time, and the same sums as with atomics (what a
caller without the larger workspace gets)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# blocks of 64 and of 128 rows, packed sequences with and without rows in the last block, an empty one, more buckets than a slot holds
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,L,lens,causal,nb", [(2, 4, 300, None, False, 32), (40, 12, 257, None, True, 32), (1, 2, 1, None, False, 32),
                                                  (1, 8, 0, [1, 700, 0, 63, 64, 65], False, 32), (1, 8, 0, [33, 129, 2], True, 64),
                                                  (2, 4, 300, None, False, 128)])
def test_slots_against_atomics(gpu_device, monkeypatch, dtype, B, H, L, lens, causal, nb):
    import turbot5_amd as t5
    from turbot5_amd import ops
    g = torch.Generator().manual_seed(L + H)
    shape = (sum(lens), H, 64) if lens else (B, H, L, 64)
    ins = [(0.5 * torch.randn(*shape, generator=g)).to(dtype).to(gpu_device).requires_grad_() for _ in range(3)]
    table = torch.randn(nb, H, generator=g).to(gpu_device).requires_grad_()
    dout = (0.5 * torch.randn(*shape, generator=g)).to(dtype).to(gpu_device)

    def grads():
        kw = dict(causal=causal, sm_scale=1.0, NUM_BUCKETS=nb)
        if lens:
            cu = torch.tensor([0] + lens, device=gpu_device).cumsum(0).to(torch.int32)
            o = t5.flash_attention_with_fusing_bias_varlen(*ins, table, cu, cu, max(lens), max(lens), **kw)
        else:
            o = t5.flash_attention_with_fusing_bias(*ins, table, **kw)
        return torch.autograd.grad(o, [*ins, table], dout)

    with_slots = grads()
    if nb <= 64:
        assert all(torch.equal(a, b) for a, b in zip(with_slots, grads()))
    monkeypatch.setattr(ops, "_backward_workspace", lambda lib, need, *rest: torch.empty(max(need, 16), device=gpu_device, dtype=torch.uint8))
    without = grads()
    for a, b in zip(with_slots[:3], without[:3]):
        assert torch.equal(a, b)
    # sums of up to some 1e5 terms of size 1 in another order
    scale = without[3].abs().max().clamp(min=1.0)
    assert (with_slots[3] - without[3]).abs().max() <= 1e-5 * scale
