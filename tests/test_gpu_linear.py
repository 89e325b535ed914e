"""Linear layers of a training step on the bf16 matrix cores (t5a_gemm_f32): forms, edges, non-finite values, gradients and
the calls that stay with torch.  Oracle: the same products in 64 bits."""
import ctypes as C
import math

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


def _rand(g, *shape, dtype=F32, dev="cuda"):
    return torch.randn(*shape, generator=g, device=dev).to(dtype)


def _bound(a, b, k):
    """Per element: six products per sixteen indices, each sum rounded (or cut) to fp32, three dropped products of at most
    2^-24 each, a few splits."""
    return (6 * math.ceil(k / 16) + 24) * 2.0 ** -23 * (a.abs() @ b.abs().t())


# sizes around a tile (64, 128 rows; 64 columns; 32 indices per step), one step, one split more than the steps fill evenly
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (63, 64, 32), (65, 72, 40), (129, 136, 264), (300, 512, 512), (257, 8, 2048), (72, 200, 4096)])
@pytest.mark.parametrize("form,adt,bdt", [("nn", F32, F32), ("nn", BF16, F32), ("nt", F32, F32), ("nt", BF16, F32),
                                          ("tt", F32, F32), ("tt", BF16, F32), ("tt", F32, BF16)])
def test_products_against_64_bits(gpu_device, M, N, K, form, adt, bdt):
    from turbot5_amd.linear import _gemm
    at, bt = form[0] == "t", form[1] == "t"
    if at and M % 8:
        M += 8 - M % 8
    if at:
        K += 3            # (both transposed: the contraction may have any length)
    g = torch.Generator(device=gpu_device).manual_seed(M * 7 + N * 3 + K)
    a, b = _rand(g, M, K, dtype=adt), _rand(g, N, K, dtype=bdt)
    out = torch.full((M, N), 7.0, device=gpu_device)
    _gemm([a.t().contiguous() if at else a], [b.t().contiguous() if bt else b], [out], a_trans=at, b_trans=bt)
    ad, bd = a.double(), b.double()
    assert ((out.double() - ad @ bd.t()).abs() <= _bound(ad, bd, K)).all()


def test_no_less_accurate_than_fp32_products(gpu_device):
    from turbot5_amd.linear import _gemm
    g = torch.Generator(device=gpu_device).manual_seed(5)
    for M, N, K, spread in [(300, 512, 512, 0.0), (1000, 512, 2048, 0.0), (512, 2048, 1000, 0.0), (300, 512, 512, 3.0)]:
        a, b = _rand(g, M, K), _rand(g, N, K)
        a, b = (t * torch.exp(spread * torch.randn(t.shape, generator=g, device=gpu_device)) for t in (a, b))
        out = torch.empty(M, N, device=gpu_device)
        _gemm([a], [b], [out])
        want = a.double() @ b.double().t()
        mine, theirs = ((t.double() - want).norm() / want.norm() for t in (out, a @ b.t()))
        assert mine <= 1.05 * theirs, (M, N, K, spread, mine.item(), theirs.item())


def test_groups_factor_and_finishes(gpu_device):
    from turbot5_amd.linear import _gemm
    g = torch.Generator(device=gpu_device).manual_seed(9)
    M, N, K = 131, 72, 520
    a = [_rand(g, M, K) for _ in range(3)]
    b = [_rand(g, N, K) for _ in range(3)]
    want = [x.double() @ y.double().t() for x, y in zip(a, b)]
    bound = [_bound(x.double(), y.double(), K) for x, y in zip(a, b)]
    for dtype, ulp in ((F32, 2.0 ** -23), (BF16, 2.0 ** -8), (torch.float16, 2.0 ** -11)):
        out = [torch.empty(M, N, device=gpu_device, dtype=dtype) for _ in range(3)]
        _gemm(a, b, out, alpha=1.5)
        for i, f in enumerate((1.5, 1.0, 1.0)):
            assert ((out[i].double() - f * want[i]).abs() <= f * bound[i] + ulp * (f * want[i]).abs()).all()
    out = torch.empty(M, N, device=gpu_device)
    total = 1.5 * want[0] + want[1] + want[2]
    for n in (3, 2):       # (two groups: splits that end inside the first one)
        _gemm(a[:n], b[:n], [out], sum_groups=True, alpha=1.5)
        ref = total if n == 3 else 1.5 * want[0] + want[1]
        assert ((out.double() - ref).abs() <= 3 * sum(bound)).all()
    _gemm(a[:1], b[:1], [out], relu=True)
    assert ((out.double() - want[0].clamp(min=0)).abs() <= bound[0]).all() and (out >= 0).all()
    pos = _rand(g, M, N)
    pos[3] = 0.0
    _gemm(a[:1], b[:1], [out], positive=pos)
    assert ((out.double() - want[0] * (pos > 0)).abs() <= bound[0]).all() and (out[pos <= 0] == 0).all()


@pytest.mark.parametrize("form", ["nn", "nt", "tt"])
def test_values_that_are_not_finite(gpu_device, form):
    """Infinities, NaN and values that round to infinity in bf16: where fp32 products give infinity, NaN or a finite result."""
    from turbot5_amd.linear import _gemm
    g = torch.Generator(device=gpu_device).manual_seed(2)
    M, N, K = 200, 136, 72
    a, b = _rand(g, M, K), _rand(g, N, K)
    a[5, 3], a[77, 1], a[130, 0] = math.inf, math.nan, 3.4e38
    b[9, 2], b[20], b[30, 1] = -math.inf, 0.0, math.inf
    a[131] = 0.0
    a[132] = 1e30
    b[40] = 1e30          # (sums past the largest fp32 number)
    out = torch.empty(M, N, device=gpu_device)
    _gemm([a.t().contiguous() if form[0] == "t" else a], [b.t().contiguous() if form[1] == "t" else b], [out],
          a_trans=form[0] == "t", b_trans=form[1] == "t")
    want = (a.double() @ b.double().t()).float()
    assert torch.equal(out.isnan(), want.isnan())
    assert torch.equal(out[out.isinf()], want[want.isinf()]) and torch.equal(out.isinf(), want.isinf())
    rest = want.isfinite()
    scale = (a.double().abs() @ b.double().abs().t())[rest]
    assert ((out.double() - a.double() @ b.double().t())[rest].abs() <= (K + 30) * 2.0 ** -23 * scale).all()


@pytest.mark.parametrize("scale", [2.0 ** -90, 2.0 ** -106, 2.0 ** -115, 2.0 ** -124])
def test_small_magnitudes_keep_their_bits(gpu_device, scale):
    """A whole operand of numbers whose bf16 parts would be denormal."""
    from turbot5_amd.linear import _gemm
    g = torch.Generator(device=gpu_device).manual_seed(3)
    a, b = _rand(g, 130, 64), _rand(g, 72, 64)
    out = torch.empty(130, 72, device=gpu_device)
    _gemm([a * scale], [b], [out])
    want = (a.double() * scale) @ b.double().t()
    assert (out.double() - want).norm() <= 1e-6 * want.norm()


# results from 2^-70 to 2^-125; operands with bf16 parts below the smallest such number, the last two denormal themselves
@pytest.mark.parametrize("form", ["nn", "nt", "tt"])
@pytest.mark.parametrize("small,large", [(2.0 ** -112, 2.0 ** 20), (2.0 ** -118, 2.0 ** 48), (2.0 ** -124, 2.0 ** 30), (2.0 ** -124, 2.0 ** 100),
                                         (2.0 ** -134, 2.0 ** 60), (2.0 ** -146, 2.0 ** 21)])
def test_small_operands_against_large_ones(gpu_device, form, small, large):
    """Numbers of which an unscaled bf16 part would lose bits, in products that are no small numbers, on either side."""
    from turbot5_amd.linear import _gemm
    g = torch.Generator(device=gpu_device).manual_seed(12)
    M, N, K = 136, 72, 520
    a, b = _rand(g, M, K) * small, _rand(g, N, K) * large
    a[5], b[9, 3] = 0.0, 0.0
    for x, y in ((a, b), (b, a)):
        out = torch.full((x.shape[0], y.shape[0]), 7.0, device=gpu_device)
        _gemm([x.t().contiguous() if form[0] == "t" else x], [y.t().contiguous() if form[1] == "t" else y], [out],
              a_trans=form[0] == "t", b_trans=form[1] == "t")
        X, Y = x.double(), y.double()
        # (a step of the denormal numbers for each of the sums)
        assert ((out.double() - X @ Y.t()).abs() <= _bound(X, Y, K) + K * 2.0 ** -149).all()


def _layers(g, dev, n, d_in, d_out):
    out = []
    for _ in range(n):
        m = nn.Linear(d_in, d_out, bias=False, device=dev)
        m.weight.data.copy_(_rand(g, d_out, d_in) * d_in ** -0.5)
        out.append(m)
    return out


@pytest.mark.parametrize("xdt,dtype", [(F32, F32), (F32, BF16), (F32, torch.float16), (BF16, F32)])
@pytest.mark.parametrize("rows", [1, 301])
def test_projections_and_their_gradients(gpu_device, xdt, dtype, rows):
    from turbot5_amd import linear
    g = torch.Generator(device=gpu_device).manual_seed(rows)
    layers = _layers(g, gpu_device, 3, 128, 64)
    x = _rand(g, rows, 128, dtype=xdt).requires_grad_()
    assert linear.takes(x, *layers)
    out = linear.project(x, dtype, 1.25, *layers)
    dy = [_rand(g, rows, 64, dtype=dtype) for _ in range(3)]
    got = torch.autograd.grad(out, [x, *(m.weight for m in layers)], dy)
    X, W = x.detach().double().requires_grad_(), [m.weight.detach().double().requires_grad_() for m in layers]
    ref = [X @ w.t() * (1.25 if i == 0 else 1.0) for i, w in enumerate(W)]
    want = torch.autograd.grad(ref, [X, *W], [t.double() for t in dy])
    step = {F32: 1e-6, BF16: 2.0 ** -8, torch.float16: 2.0 ** -11}
    for o, r in zip(out, ref):
        assert o.dtype == dtype and (o.double() - r).norm() <= step[dtype] * r.norm()
    for t, r in zip(got, want):
        assert (t.double() - r).norm() <= step[t.dtype] * r.norm()
    # frozen weights and rows
    layers[0].weight.requires_grad_(False)
    again = torch.autograd.grad(linear.project(x, dtype, 1.25, *layers), [layers[1].weight, layers[2].weight], dy)
    for t, r in zip(again, want[2:]):
        assert (t.double() - r).norm() <= 1e-6 * r.norm()


def test_feed_forward_and_its_gradients(gpu_device):
    from turbot5_amd import T5Config
    from turbot5_amd.modeling import T5DenseActDense
    g = torch.Generator(device=gpu_device).manual_seed(1)
    ff = T5DenseActDense(T5Config(d_model=64, d_ff=256, dropout_rate=0.0)).to(gpu_device)
    x = _rand(g, 2, 150, 64).requires_grad_()
    y = ff(x)
    assert y.grad_fn.next_functions[0][0].name() == "FeedForwardReluBackward"
    dy = _rand(g, 2, 150, 64)
    got = torch.autograd.grad(y, [x, ff.wi.weight, ff.wo.weight], dy)
    X, WI, WO = (t.detach().double().requires_grad_() for t in (x, ff.wi.weight, ff.wo.weight))
    Y = torch.relu(X @ WI.t()) @ WO.t()
    want = torch.autograd.grad(Y, [X, WI, WO], dy.double())
    assert (y.double() - Y).norm() <= 1e-6 * Y.norm()
    for t, r in zip(got, want):
        assert (t.double() - r).norm() <= 2e-6 * r.norm()


def test_second_derivatives_batches_and_checkpoints(gpu_device):
    from torch.utils.checkpoint import checkpoint
    from turbot5_amd import linear
    g = torch.Generator(device=gpu_device).manual_seed(4)
    wi, = _layers(g, gpu_device, 1, 32, 64)
    wo, = _layers(g, gpu_device, 1, 64, 32)
    x = _rand(g, 256, 32).requires_grad_()

    def run(x):
        return linear.feed_forward_relu(linear.project(x, F32, 0.5, wi)[0] @ wo.weight.t(), wi, wo)

    def plain(x):
        return torch.relu((x @ wi.weight.t() * 0.5 @ wo.weight.t()) @ wi.weight.t()) @ wo.weight.t()

    params = [x, wi.weight, wo.weight]
    results = []
    for f in (run, plain):
        y = f(x)
        first = torch.autograd.grad(y.square().sum(), params, create_graph=True)
        results.append([*first, *torch.autograd.grad(sum(t.square().sum() for t in first), params)])
    for a, b in zip(*results):
        assert (a - b).norm() <= 1e-5 * b.norm()
    dy = _rand(g, 3, 256, 32)
    batched = torch.autograd.grad(run(x), params, dy, is_grads_batched=True)
    for i in range(3):
        for t, r in zip(batched, torch.autograd.grad(plain(x), params, dy[i])):
            assert (t[i] - r).norm() <= 1e-5 * r.norm()
    direct = torch.autograd.grad(run(x), params, dy[0])
    kept = torch.autograd.grad(checkpoint(run, x, use_reentrant=False), params, dy[0])
    assert all(torch.equal(a, b) for a, b in zip(direct, kept))
    offloaded = None
    with torch.autograd.graph.save_on_cpu():
        offloaded = run(x)
    assert all(torch.equal(a, b) for a, b in zip(direct, torch.autograd.grad(offloaded, params, dy[0])))


def test_calls_that_stay_with_torch(gpu_device):
    from turbot5_amd import linear
    g = torch.Generator(device=gpu_device).manual_seed(4)
    m, = _layers(g, gpu_device, 1, 32, 64)
    x = _rand(g, 256, 32)
    assert linear.takes(x, m)
    with torch.no_grad():
        assert not linear.takes(x, m)
    assert not linear.takes(x[:0], m) and not linear.takes(x.half(), m) and not linear.takes(x[:, :16], m)
    with torch.autocast("cuda", dtype=BF16):
        assert not linear.takes(x, m)
    torch.set_float32_matmul_precision("high")
    try:
        assert not linear.takes(x, m)
    finally:
        torch.set_float32_matmul_precision("highest")
    with torch.autograd.forward_ad.dual_level():
        assert not linear.takes(x, m)
    handle = m.register_forward_hook(lambda *a: None)
    assert not linear.takes(x, m)
    handle.remove()
    assert linear.takes(x, m)
    for other in (nn.Linear(32, 64, device=gpu_device), nn.Linear(32, 64, bias=False, device=gpu_device, dtype=BF16),
                  nn.utils.parametrizations.weight_norm(nn.Linear(32, 64, bias=False, device=gpu_device)),
                  nn.Linear(32, 60, bias=False, device=gpu_device)):
        assert not linear.takes(x, other)


def test_captured_step_replays(gpu_device):
    """Products in several splits, captured with their workspace: every replay as the eager result."""
    from turbot5_amd.linear import _gemm
    g = torch.Generator(device=gpu_device).manual_seed(8)
    a, b = _rand(g, 300, 2048), _rand(g, 512, 2048)
    out = torch.empty(300, 512, device=gpu_device)
    _gemm([a], [b], [out])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _gemm([a], [b], [out])
    for seed in range(3):
        a.copy_(_rand(g, 300, 2048))
        want = torch.empty_like(out)
        _gemm([a], [b], [want])
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
