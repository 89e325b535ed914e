"""The attention ops' native autograd nodes: what autograd promises about a node, and the calls that keep the Python function."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(dev, packed=False, dtype=torch.bfloat16, table_dtype=torch.float32, D=64):
    g = torch.Generator().manual_seed(11)
    shape = (200, 4, D) if packed else (2, 4, 100, D)
    ins = [(0.5 * torch.randn(*shape, generator=g)).to(dtype).to(dev).requires_grad_() for _ in range(3)]
    ins.append(torch.randn(32, 4, generator=g).to(table_dtype).to(dev).requires_grad_())
    return ins, (0.5 * torch.randn(*shape, generator=g)).to(dtype).to(dev)


def _call(ins, packed=False, **kw):
    import turbot5_amd as t5
    if not packed:
        return t5.flash_attention_with_fusing_bias(*ins, sm_scale=1.0, **kw)
    cu = torch.tensor([0, 37, 200], device=ins[0].device)          # (int64: converted)
    return t5.flash_attention_with_fusing_bias_varlen(*ins, cu, cu, 163, 163, sm_scale=1.0, **kw)


def _function(monkeypatch):
    """The Python autograd.Function in the node's place."""
    from turbot5_amd import ops
    monkeypatch.setattr(ops, "_takes_node", lambda *a: False)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("dtype,table_dtype", [(torch.bfloat16, torch.float32), (torch.float16, torch.bfloat16), (torch.float32, torch.float64)])
def test_node_against_the_python_function(gpu_device, monkeypatch, packed, dtype, table_dtype):
    ins, dout = _inputs(gpu_device, packed, dtype, table_dtype)
    o, lse = _call(ins, packed, return_lse=True)
    assert o.grad_fn.name() == ("FlashAttentionBiasVarlenBackward" if packed else "FlashAttentionBiasBackward") and not lse.requires_grad
    strided = torch.empty(*dout.shape[:-1], 2 * dout.shape[-1], device=gpu_device, dtype=dtype)[..., ::2].copy_(dout)     # (a copy is made)
    got = torch.autograd.grad(o, ins, strided, retain_graph=True)
    again = torch.autograd.grad(o, ins[:1] + ins[3:], dout)                 # some inputs only, graph freed
    assert torch.equal(got[0], again[0]) and torch.equal(got[3], again[1])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, ins, dout)
    _function(monkeypatch)
    o2 = _call(ins, packed)
    assert torch.equal(o, o2)
    for a, b in zip(got, torch.autograd.grad(o2, ins, dout)):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("packed", [False, True])
def test_saved_tensors(gpu_device, packed):
    from torch.utils.checkpoint import checkpoint
    ins, dout = _inputs(gpu_device, packed)
    want = torch.autograd.grad(_call(ins, packed), ins, dout)
    with torch.autograd.graph.save_on_cpu():
        o = _call(ins, packed)
    assert all(torch.equal(a, b) for a, b in zip(want, torch.autograd.grad(o, ins, dout)))
    o = checkpoint(lambda *a: _call(a, packed), *ins, use_reentrant=False)
    assert all(torch.equal(a, b) for a, b in zip(want, torch.autograd.grad(o, ins, dout)))
    o = _call(ins, packed)
    with torch.no_grad():
        ins[1].mul_(2.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(o, ins, dout)


def test_streams_frozen_inputs_and_changed_results(gpu_device):
    ins, dout = _inputs(gpu_device)
    want = torch.autograd.grad(_call(ins), ins, dout)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        o = _call(ins)
    got = torch.autograd.grad(o, ins, dout)         # (the engine runs the node on the forward's stream)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    table = ins[3].detach().requires_grad_()
    o = _call([t.detach() for t in ins[:3]] + [table])
    assert torch.equal(torch.autograd.grad(o, table, dout)[0], want[3])
    o = _call(ins).mul_(2.0)                        # (not a view, so it may be changed, but the backward needs it)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(o, ins[:1], dout)
    no_table = _call([*ins[:3], None])
    assert len(torch.autograd.grad(no_table, ins[:3], dout)) == 3


def test_refusals_and_switches_at_the_time_of_the_backward(gpu_device, monkeypatch):
    from turbot5_amd import ops
    ins, dout = _inputs(gpu_device, dtype=torch.float32, D=128)
    o = _call(ins)
    with pytest.raises(NotImplementedError, match="head_dim 128"):
        torch.autograd.grad(o, ins, dout)
    ins, dout = _inputs(gpu_device)
    o = _call(ins)
    fast = torch.autograd.grad(o, ins, dout, retain_graph=True)
    monkeypatch.setattr(ops, "BACKWARD_FP32_MATH", True)
    wide = torch.autograd.grad(o, ins, dout)
    assert not torch.equal(fast[0], wide[0])
    o, lse = _call(ins, return_lse=True)
    want = ops._dense_backward(*ins, o.detach(), lse, dout, False, 1.0, 32, 128, None)
    assert all(torch.equal(a, b) for a, b in zip(wide[:3], want))                   # (the table's gradient by atomics there)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("node", [True, False])
def test_second_derivatives_raise(gpu_device, monkeypatch, packed, node):
    """A kept graph gives the same first derivatives; what would lack the terms through the attention is an error."""
    if not node:
        _function(monkeypatch)
    ins, dout = _inputs(gpu_device, packed)
    want = torch.autograd.grad(_call(ins, packed), ins, dout)
    got = torch.autograd.grad(_call(ins, packed), ins, dout, create_graph=True)
    assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(want, got))
    x = ins[0].detach().float().requires_grad_()
    first = torch.autograd.grad(_call([(x * x).bfloat16(), *ins[1:]], packed).float().square().sum(), x, create_graph=True)[0]
    with pytest.raises(RuntimeError, match="second derivative"):
        torch.autograd.grad(first.square().sum(), x)
    frozen = torch.autograd.grad(_call([*ins[:3], ins[3].detach()], packed), ins[0], dout, create_graph=True)
    assert torch.equal(frozen[0], want[0])


def test_a_copy_of_the_package_under_another_name(gpu_device, tmp_path, monkeypatch):
    """Its nodes read its own switch, whatever the other copy's says."""
    import importlib
    import os
    import shutil
    import turbot5_amd as t5
    from turbot5_amd import ops
    shutil.copytree(os.path.dirname(t5.__file__), tmp_path / "vendored_attention", ignore=shutil.ignore_patterns("csrc", "__pycache__"))
    monkeypatch.syspath_prepend(str(tmp_path))
    copy = importlib.import_module("vendored_attention")
    copy_ops = importlib.import_module("vendored_attention.ops")
    ins, dout = _inputs(gpu_device)

    def grads(package):
        return torch.autograd.grad(package.flash_attention_with_fusing_bias(*ins, sm_scale=1.0), ins[:3], dout)

    assert copy_ops._nodes() is not ops._nodes()
    fast = grads(t5)
    assert all(torch.equal(a, b) for a, b in zip(fast, grads(copy)))
    monkeypatch.setattr(copy_ops, "BACKWARD_FP32_MATH", True)
    wide = grads(copy)
    assert all(torch.equal(a, b) for a, b in zip(fast, grads(t5))) and not torch.equal(fast[0], wide[0])


def test_calls_that_keep_the_python_function(gpu_device):
    from turbot5_amd import ops
    ins, _ = _inputs(gpu_device)

    class Sub(torch.Tensor):
        pass

    assert ops._takes_node(*ins)
    assert not ops._takes_node(ins[0].detach().as_subclass(Sub), *ins[1:])
    with torch.autograd.forward_ad.dual_level():
        assert not ops._takes_node(torch.autograd.forward_ad.make_dual(ins[0].detach(), torch.ones_like(ins[0])), *ins[1:])
    seen = []
    torch.vmap(lambda x: (seen.append(ops._takes_node(x, *ins[1:])), x)[1])(ins[0].detach())
    torch.jit.trace(lambda x: (seen.append(ops._takes_node(x, *ins[1:])), x * 1)[1], ins[0].detach(), check_trace=False)
    from torch.utils.flop_counter import FlopCounterMode
    with FlopCounterMode(display=False):
        seen.append(ops._takes_node(*ins))
    assert seen and not any(seen)
