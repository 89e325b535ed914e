"""GPU parity of the fused RMS norm / side-token producer against the CPU oracle (through the C ABI)."""
import pytest
import torch

from oracle import t5_basic as O
from oracle.t5_model import tglobal_side_inputs

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


@pytest.mark.parametrize("xdt,wdt", [("bf16", "bf16"), ("f32", "f32"), ("f32", "bf16"), ("bf16", "f32"), ("f16", "f16")])
@pytest.mark.parametrize("shape", [(2, 100, 768), (3, 7, 512), (1, 16384, 768), (5, 4096), (2, 9, 64), (4, 33, 4096)])
def test_rms_norm_matches_the_oracle(gpu_device, xdt, wdt, shape):
    from turbot5_amd.ops import rms_norm
    g = torch.Generator().manual_seed(sum(shape) + len(xdt) * 7 + len(wdt))
    x = (2.0 * torch.randn(*shape, generator=g)).to(DT[xdt])
    w = (1.0 + 0.2 * torch.randn(shape[-1], generator=g)).to(DT[wdt])
    want = O.rms_norm(x, w, 1e-6)
    got = rms_norm(x.to(gpu_device), w.to(gpu_device), 1e-6)
    assert got.dtype == want.dtype and got.shape == want.shape
    diff = (got.float().cpu() - want.float()).abs()
    if want.dtype == torch.float32:
        assert (diff <= 2e-6 + 1e-5 * want.float().abs()).all()
    else:
        # two roundings (scaled value, then product): a last-bit difference of the fp32 scale can move the
        # result by up to two units in the last place; it almost never does
        ulp = 2.0 ** -7 if want.dtype == torch.bfloat16 else 2.0 ** -10
        assert (diff <= 2 * ulp * want.float().abs() + 1e-6).all()
        assert (diff == 0).float().mean().item() > 0.98


def test_rms_norm_strided_rows_and_closed_form(gpu_device):
    from turbot5_amd.ops import rms_norm
    big = torch.randn(4, 50, 1024, generator=torch.Generator().manual_seed(3))
    x = big[:, :, 256:768]                                           # row stride 1024, 512 columns
    w = torch.ones(512)
    got = rms_norm(x.to(gpu_device)[:, :, :], w.to(gpu_device)).cpu()
    assert torch.allclose(got.pow(2).mean(-1), torch.ones(4, 50), atol=1e-4)   # unit RMS by definition
    assert torch.allclose(got, O.rms_norm(x, w), atol=1e-5, rtol=1e-5)
    const = torch.full((3, 64), 5.0)                                 # constant row -> weight itself
    w2 = torch.linspace(-1, 1, 64)
    assert torch.allclose(rms_norm(const.to(gpu_device), w2.to(gpu_device), 0.0).cpu(), w2.expand(3, 64), atol=1e-6)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("L,gbs", [(512, 16), (100, 16), (37, 8), (16, 16), (15, 16), (2048, 1), (130, 64)])
def test_side_token_producer_matches_the_oracle(gpu_device, dtype, L, gbs):
    """Block sums + norm in one kernel, against the one-hot einsum + norm of the oracle; L % gbs != 0
    exercises the orphan tokens that join the last full block."""
    from turbot5_amd.ops import rms_norm
    B, d = 3, 256
    g = torch.Generator().manual_seed(L * 31 + gbs)
    hidden = torch.randn(B, L, d, generator=g).to(DT[dtype])
    w = (1.0 + 0.1 * torch.randn(d, generator=g)).to(DT[dtype])
    want = tglobal_side_inputs(hidden, gbs, w, 1e-6)
    got = rms_norm(hidden.to(gpu_device), w.to(gpu_device), 1e-6, group=gbs)
    assert got.shape == want.shape == (B, L // gbs, d)
    if want.numel():
        tol = 1e-5 if dtype == "f32" else 2e-2                        # bf16: the einsum's accumulation order is free
        assert (got.float().cpu() - want.float()).abs().max().item() <= tol * max(1.0, want.float().abs().max().item())


def test_layer_norm_module_uses_the_kernel(gpu_device):
    from turbot5_amd.attentions import T5LayerNorm
    torch.manual_seed(0)
    m = T5LayerNorm(768).to(gpu_device).to(torch.bfloat16)
    x = torch.randn(2, 300, 768).to(torch.bfloat16)
    want = O.rms_norm(x, m.weight.detach().cpu(), m.eps)
    got = m(x.to(gpu_device))
    assert got.dtype == torch.bfloat16
    assert (got.float().cpu() - want.float()).abs().max().item() <= 2.0 ** -6


@pytest.mark.parametrize("xdt,wdt", [("bf16", "bf16"), ("f32", "f32"), ("f16", "f16"), ("f32", "bf16")])
@pytest.mark.parametrize("shape", [(2, 100, 768), (1, 4096, 768), (3, 7, 512), (2, 9, 64), (2, 33, 4096), (1, 5, 2048)])
def test_add_then_norm_in_one_kernel(gpu_device, xdt, wdt, shape):
    """x + residual (rounded to x's type, exactly torch's add) and the norm of that sum; covers rows held
    in registers (two and four chunks per lane) and the two-pass form (4096 columns)."""
    from turbot5_amd.ops import rms_norm
    g = torch.Generator().manual_seed(sum(shape) + len(xdt))
    x = (2.0 * torch.randn(*shape, generator=g)).to(DT[xdt])
    r = (1.5 * torch.randn(*shape, generator=g)).to(DT[xdt])
    w = (1.0 + 0.2 * torch.randn(shape[-1], generator=g)).to(DT[wdt])
    total, got = rms_norm(x.to(gpu_device), w.to(gpu_device), 1e-6, residual=r.to(gpu_device))
    assert torch.equal(total.cpu(), x + r)                      # one correctly rounded add: bit-exact
    want = O.rms_norm(x + r, w, 1e-6)
    assert got.dtype == want.dtype and got.shape == want.shape and total.dtype == x.dtype
    plain = rms_norm((x + r).to(gpu_device), w.to(gpu_device), 1e-6)
    assert torch.equal(got, plain)                              # same arithmetic as the norm alone on the sum
    diff = (got.float().cpu() - want.float()).abs()
    ulp = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -6, torch.float16: 2.0 ** -9}[want.dtype]
    assert (diff <= ulp * want.float().abs() + 2e-6).all()


def test_add_norm_rejects_bad_arguments(gpu_device):
    from turbot5_amd.ops import rms_norm
    x = torch.randn(2, 8, 64, device=gpu_device)
    w = torch.ones(64, device=gpu_device)
    with pytest.raises(ValueError):
        rms_norm(x, w, residual=x[:, :4])
    with pytest.raises(ValueError):
        rms_norm(x, w, group=2, residual=x)
    with pytest.raises(ValueError):
        rms_norm(x, w, residual=x.half())


def test_layer_norm_add_norm_and_stack_equivalence(gpu_device):
    """The stack hands each sub-layer's update to the next norm; block.forward adds it itself: same numbers."""
    from turbot5_amd import T5Config, T5EncoderModel
    torch.manual_seed(3)
    cfg = T5Config(vocab_size=100, d_model=128, d_kv=64, d_ff=256, num_layers=2, num_heads=2, dropout_rate=0.0,
                   attention_type="flash")
    m = T5EncoderModel(cfg).eval().to(gpu_device).to(torch.bfloat16)
    ids = torch.randint(0, 100, (2, 70), device=gpu_device)
    with torch.no_grad():
        got = m(ids)
        h = m.shared(ids)
        bias = None
        for blk in m.encoder.block:
            h, _, bias = blk(h, position_bias=bias)
        want = m.encoder.final_layer_norm(h)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("L,gbs,lens", [(512, 16, [512, 300, 17, 0]), (100, 16, [99, 16, 15, 64]), (64, 8, [64, 63, 9, 1])])
def test_side_token_producer_with_sequence_lengths(gpu_device, dtype, L, gbs, lens):
    """Right-padded batch: a sequence of n tokens has n // gbs side tokens (its last tokens join the last
    full block, padding is left out), the remaining output rows are zero -- the oracle's mask path."""
    from turbot5_amd.ops import rms_norm
    B, d = len(lens), 256
    g = torch.Generator().manual_seed(L * 13 + gbs)
    hidden = torch.randn(B, L, d, generator=g).to(DT[dtype])
    w = (1.0 + 0.1 * torch.randn(d, generator=g)).to(DT[dtype])
    mask = (torch.arange(L)[None, :] < torch.tensor(lens)[:, None]).float()
    want = tglobal_side_inputs(hidden, gbs, w, 1e-6, mask)
    got = rms_norm(hidden.to(gpu_device), w.to(gpu_device), 1e-6, group=gbs,
                   seq_lens=torch.tensor(lens, dtype=torch.int32, device=gpu_device))
    assert got.shape == want.shape == (B, L // gbs, d)
    tol = 1e-5 if dtype == "f32" else 2e-2
    assert (got.float().cpu() - want.float()).abs().max().item() <= tol * max(1.0, want.float().abs().max().item())
    for b, n in enumerate(lens):
        assert (got[b, n // gbs:] == 0).all()
    # one side token per token (group 1): every valid row normalised by itself, padding rows zero
    tl = torch.tensor(lens, dtype=torch.int32, device=gpu_device)
    one = rms_norm(hidden.to(gpu_device), w.to(gpu_device), 1e-6, group=1, seq_lens=tl)
    want1 = tglobal_side_inputs(hidden, 1, w, 1e-6, mask)
    assert one.shape == want1.shape == (B, L, d)
    assert (one.float().cpu() - want1.float()).abs().max().item() <= tol * max(1.0, want1.float().abs().max().item())
    with pytest.raises(ValueError):
        rms_norm(hidden.to(gpu_device), w.to(gpu_device), 1e-6, group=1, seq_lens=tl, residual=hidden.to(gpu_device))


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("L,gbs", [(512, 16), (100, 16), (64, 8), (777, 32)])
def test_side_token_producer_with_masks_of_any_shape(gpu_device, dtype, L, gbs):
    """key_bits and group_counts: a side token sums the valid tokens of its block, the last one every valid token
    from its block on, rows past the count are zero -- the oracle's block ids and aggregates for any mask"""
    from turbot5_amd.ops import pack_key_bits, rms_norm, side_token_counts
    B, d = 5, 256
    g = torch.Generator().manual_seed(L * 7 + gbs)
    hidden = torch.randn(B, L, d, generator=g).to(DT[dtype])
    w = (1.0 + 0.1 * torch.randn(d, generator=g)).to(DT[dtype])
    mask = torch.ones(B, L)
    mask[0] = (torch.rand(L, generator=g) > 0.3).float()
    mask[1, : L // 3] = 0
    mask[2, L // 5: L // 2] = 0
    mask[2, -(gbs + 3):] = 0
    mask[3, gbs - 1::gbs] = 0          # no block END is valid: no side token
    want = tglobal_side_inputs(hidden, gbs, w, 1e-6, mask)
    dmask = mask.to(gpu_device)
    counts = side_token_counts(dmask, gbs)
    got = rms_norm(hidden.to(gpu_device), w.to(gpu_device), 1e-6, group=gbs, key_bits=pack_key_bits(dmask, gbs),
                   group_counts=counts)
    assert got.shape == want.shape == (B, L // gbs, d)
    tol = 1e-5 if dtype == "f32" else 2e-2
    assert (got.float().cpu() - want.float()).abs().max().item() <= tol * max(1.0, want.float().abs().max().item())
    assert (got[3] == 0).all() and counts[3].item() == 0
    for b in range(B):
        assert (got[b, counts[b].item():] == 0).all()
    with pytest.raises(ValueError):
        rms_norm(hidden.to(gpu_device), w.to(gpu_device), 1e-6, group=gbs, key_bits=pack_key_bits(dmask, gbs))


def _formula(x, w, eps):
    n = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)
    return w * n


@pytest.mark.parametrize("xdt,wdt", [("f32", "f32"), ("bf16", "bf16"), ("f32", "f16"), ("f16", "f32")])
@pytest.mark.parametrize("rows,d", [(1, 8), (3, 256), (5, 264), (2050, 512), (9000, 768), (130, 1024), (33, 2048)])
@pytest.mark.parametrize("with_residual", [False, True])
def test_norm_gradients_match_the_formula_in_64_bits(gpu_device, xdt, wdt, rows, d, with_residual):
    """Module in training mode: dx (with the residual stream's gradient added) and dweight.  Rows from one wavefront's
    to several per wavefront, columns around the register chunks of 256.  Bounds: fp32 sums of up to 9000 terms, 2e-6
    of the largest times their root; 16-bit weights round n and g (2^-9 each) and the results once more."""
    from turbot5_amd.attentions import T5LayerNorm
    g = torch.Generator().manual_seed(rows * 7 + d)
    x = torch.randn(rows, d, generator=g).to(DT[xdt])
    r = torch.randn(rows, d, generator=g).to(DT[xdt])
    w = (1.0 + 0.2 * torch.randn(d, generator=g)).to(DT[wdt])
    norm = T5LayerNorm(d).to(gpu_device).train()
    norm.weight = torch.nn.Parameter(w.to(gpu_device))
    xg, rg = (t.to(gpu_device).requires_grad_() for t in (x, r))
    total, y = norm.add_norm(xg, rg if with_residual else None)
    with torch.no_grad():     # bit for bit the formula in torch's operations
        tt = xg + rg if with_residual else xg
        n = tt * torch.rsqrt(tt.float().pow(2).mean(-1, keepdim=True) + norm.eps)
        assert torch.equal(total, tt) and torch.equal(y, norm.weight * (n.to(w.dtype) if w.dtype != torch.float32 else n))
    dy, ds = torch.randn(rows, d, generator=g).to(y.dtype), torch.randn(rows, d, generator=g).to(total.dtype)
    outs, grads = ([total, y], [ds, dy]) if with_residual else ([y], [dy])
    torch.autograd.backward(outs, [t.to(gpu_device) for t in grads])
    x64 = ((x + r) if with_residual else x).double().requires_grad_()
    w64 = w.double().requires_grad_()
    (_formula(x64, w64, 1e-6) * dy.double()).sum().backward()
    want = x64.grad + (ds.double() if with_residual else 0)
    tol = 2e-5 if xdt == wdt == "f32" else 2e-2 if "bf16" in (xdt, wdt) else 4e-3
    scale = want.abs().max().item()
    assert (xg.grad.double().cpu() - want).abs().max().item() <= tol * scale
    if with_residual:
        assert torch.equal(xg.grad, rg.grad)
    assert xg.grad.dtype == x.dtype and norm.weight.grad.dtype == w.dtype
    assert (norm.weight.grad.double().cpu() - w64.grad).abs().max().item() <= tol * w64.grad.abs().max().item()


def test_norm_gradients_where_the_kernel_is_passed_by(gpu_device):
    """Differentiating the gradient, function transforms, forward mode, widths past the kernel's and empty batches take the
    formula in torch's operations; a saved-tensor hook sees what is saved."""
    from turbot5_amd.attentions import T5LayerNorm
    norm = T5LayerNorm(64).to(gpu_device).train()
    with torch.no_grad():
        norm.weight.copy_(torch.linspace(0.5, 1.5, 64))
    x = torch.randn(6, 64, generator=torch.Generator().manual_seed(1)).to(gpu_device).requires_grad_()

    def second(f):
        gx, = torch.autograd.grad(f(x).pow(3).sum(), x, create_graph=True)
        return torch.autograd.grad(gx.pow(2).sum(), (x, norm.weight))
    for got, want in zip(second(norm), second(lambda t: _formula(t, norm.weight, 1e-6))):
        assert torch.allclose(got, want, rtol=1e-3, atol=1e-3)
    total, y = norm.add_norm(x, 2 * x)
    gx, = torch.autograd.grad(y.pow(2).sum() + total.sum(), x, create_graph=True)
    assert gx.requires_grad
    t = torch.randn_like(x)
    got = torch.func.jvp(norm, (x.detach(),), (t,))[1]
    want = torch.func.jvp(lambda v: _formula(v, norm.weight, 1e-6), (x.detach(),), (t,))[1]
    assert torch.allclose(got, want, atol=1e-5)
    assert torch.allclose(torch.vmap(norm)(x), norm(x), atol=1e-6)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda s: seen.append(s) or s, lambda s: s):
        norm(x).sum().backward()
    assert seen and x.grad is not None
    wide = T5LayerNorm(4096).to(gpu_device).train()
    wide(torch.randn(2, 4096, device=gpu_device)).sum().backward()
    assert wide.weight.grad is not None
    norm(torch.empty(0, 64, device=gpu_device)).sum().backward()


def test_norm_gradients_in_batches_and_with_tangents(gpu_device):
    """Several gradients at once (batched reverse mode, a vmap around it, a vectorised jacobian) and a gradient that carries
    a tangent: a module in training mode takes them, row for row what they are one at a time."""
    import torch.autograd.forward_ad as fwd
    from turbot5_amd.attentions import T5LayerNorm
    norm = T5LayerNorm(64).to(gpu_device).train()
    with torch.no_grad():
        norm.weight.copy_(torch.linspace(0.5, 1.5, 64))
    g = torch.Generator().manual_seed(2)
    x, r = (torch.randn(3, 64, generator=g).to(gpu_device).requires_grad_() for _ in range(2))
    dy, ds = (torch.randn(5, 3, 64, generator=g).to(gpu_device) for _ in range(2))
    total, y = norm.add_norm(x, r)
    ins = (x, r, norm.weight)
    want = [torch.autograd.grad((total, y), ins, (a, b), retain_graph=True) for a, b in zip(ds, dy)]
    for got in (torch.autograd.grad((total, y), ins, (ds, dy), retain_graph=True, is_grads_batched=True),
                torch.vmap(lambda a, b: torch.autograd.grad((total, y), ins, (a, b), retain_graph=True))(ds, dy),
                torch.autograd.grad((total, y), ins, (ds, dy), retain_graph=True, is_grads_batched=True, create_graph=True)):
        for i in range(3):
            assert torch.allclose(got[i], torch.stack([w[i] for w in want]), rtol=1e-5, atol=1e-5)
    eye = torch.eye(3 * 64, device=gpu_device).view(-1, 3, 64)
    z = norm(x)
    rows = torch.stack([torch.autograd.grad(z, x, e, retain_graph=True)[0] for e in eye]).view(3, 64, 3, 64)
    jac = torch.autograd.functional.jacobian(norm, x.detach(), vectorize=True)
    assert torch.allclose(jac, rows, rtol=1e-5, atol=1e-5)
    with fwd.dual_level():     # the backward is linear in dy: its tangent is the gradient of the tangent
        gx, = torch.autograd.grad(z, x, fwd.make_dual(dy[0], dy[1]), retain_graph=True)
        value, tangent = fwd.unpack_dual(gx)
    assert tangent is not None
    for got, seed in ((value, dy[0]), (tangent, dy[1])):
        assert torch.allclose(got, torch.autograd.grad(z, x, seed, retain_graph=True)[0], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("x_grad,r_grad", [(False, False), (True, False), (False, True)])
def test_residual_stream_carries_a_graph_only_where_it_has_one(gpu_device, x_grad, r_grad):
    """Training the norm's weight alone does not make the residual stream part of the graph."""
    from turbot5_amd.attentions import T5LayerNorm
    norm = T5LayerNorm(64).to(gpu_device).train()
    x, r = torch.randn(3, 64, device=gpu_device, requires_grad=x_grad), torch.randn(3, 64, device=gpu_device, requires_grad=r_grad)
    total, y = norm.add_norm(x, r)
    assert total.requires_grad == (x_grad or r_grad) and y.requires_grad
    y.sum().backward()
    assert norm.weight.grad is not None and (x.grad is not None) == x_grad and (r.grad is not None) == r_grad


@pytest.mark.parametrize("with_residual", [False, True])
def test_norm_of_a_training_step_under_compilation_and_tracing(gpu_device, with_residual):
    """A module in training mode compiles as one graph, traces, and runs under a dispatch mode: all in torch's operations,
    bit for bit what the kernel's forward gives, with gradients that agree."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from turbot5_amd.attentions import T5LayerNorm

    class Count(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.n += 1
            return func(*args, **(kwargs or {}))

    class Step(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.norm = T5LayerNorm(64)

        def forward(self, a, b):
            return self.norm.add_norm(a, b)[1] if with_residual else self.norm(a)
    plain = Step().to(gpu_device).train()
    norm = plain.norm
    x, r = (torch.randn(3, 64, device=gpu_device, requires_grad=True) for _ in range(2))
    compiled = torch.compile(plain, backend="aot_eager", fullgraph=True)
    want = plain(x, r)
    dy = torch.randn_like(want)
    grads = torch.autograd.grad(want, (x, norm.weight), dy)
    with Count():
        moded = plain(x, r)
    assert Count.n > 0
    for got in (compiled(x, r), moded, torch.jit.trace(plain, (x, r), check_trace=False)(x, r)):
        assert torch.allclose(got, want, rtol=1e-6, atol=1e-6)
        for a, b in zip(torch.autograd.grad(got, (x, norm.weight), dy), grads):
            assert torch.allclose(a, b, rtol=1e-5, atol=1e-5)
