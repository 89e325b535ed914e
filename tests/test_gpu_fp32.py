"""fp32 attention at head_dim 64, whose products run on the bf16 matrix cores: both block sizes, edges, and values whose bf16
parts are no numbers.  Oracle: the formulas in 64 bits."""
import math

import pytest
import torch

from oracle import t5_basic as O
from tests.closed_forms import dense_64_bits

pytestmark = pytest.mark.gpu


def _exact(q, k, v, table, causal, scale, dout=None, far=128):
    """o and the gradients of q, k, v and the table."""
    return dense_64_bits(q, k, v, table, causal, scale, far, dout)


# (blocks of 64 rows: up to 256, causal 640; of 128 beyond) x tile edges, one row, rows without keys, more keys than rows
@pytest.mark.parametrize("B,H,M,N,causal", [(1, 2, 1, 1, False), (1, 2, 63, 65, False), (2, 2, 64, 64, True), (1, 3, 33, 300, True),
                                            (1, 2, 200, 90, True), (2, 4, 257, 257, False), (65, 4, 65, 40, False),
                                            (40, 8, 97, 161, True), (33, 8, 130, 31, True)])
def test_forward_and_gradients_against_64_bits(gpu_device, B, H, M, N, causal):
    import turbot5_amd as t5
    g = torch.Generator().manual_seed(B + M + N)
    q, k, v, d = (0.5 * torch.randn(B, n, H, 64, generator=g) for n in (M, N, N, M))
    table = torch.randn(32, H, generator=g)
    ins = [t.to(gpu_device).transpose(1, 2).requires_grad_() for t in (q, k, v)] + [table.to(gpu_device).requires_grad_()]
    dout = d.to(gpu_device).transpose(1, 2)
    o = t5.flash_attention_with_fusing_bias(*ins, causal=causal, sm_scale=1.0)
    got = [o, *torch.autograd.grad(o, ins, dout)]
    want = _exact(*ins, causal, 1.0, dout)
    # four times what the sums' roundings were seen to leave over such shapes (5e-7 forward, 1.7e-6 gradients)
    # (with one key the gradients are differences of equal terms, of norm 1 and more)
    for t, r, tol in zip(got, want, (2e-6, 7e-6, 7e-6, 7e-6, 7e-6)):
        assert (t.double().cpu() - r).norm() <= tol * r.norm().clamp(min=1.0)


@pytest.mark.parametrize("nb,far", [(64, 1000), (64, 1250)])
def test_bucketings_with_and_without_room_for_the_larger_tiles(gpu_device, nb, far):
    """Saturated at 773 and 952, either side of 779: blocks of 64 rows for both passes, and of 128 for dq."""
    import turbot5_amd as t5
    g = torch.Generator().manual_seed(far)
    q, k, v, d = (0.5 * torch.randn(1, 2, 1000, 64, generator=g) for _ in range(4))
    ins = [t.to(gpu_device).requires_grad_() for t in (q, k, v, torch.randn(nb, 2, generator=g))]
    o = t5.flash_attention_with_fusing_bias(*ins, causal=False, sm_scale=1.0, NUM_BUCKETS=nb, MAX_DISTANCE=far)
    got = [o, *torch.autograd.grad(o, ins, d.to(gpu_device))]
    for t, r, tol in zip(got, _exact(*ins, False, 1.0, d, far), (2e-6, 7e-6, 7e-6, 7e-6, 7e-6)):
        assert (t.double().cpu() - r).norm() <= tol * r.norm()


@pytest.mark.parametrize("B", [1, 48])
def test_values_that_have_no_bf16_parts(gpu_device, B):
    """A number that rounds to infinity in bf16 (3.4e38) among small ones: results that fp32 holds are finite; infinite keys: scores of
    minus infinity hide them, the other rows are NaN; a NaN key reaches the rows that see it."""
    import turbot5_amd as t5
    H, L = 8, 96
    g = torch.Generator().manual_seed(3)
    q, k, v, d = (0.5 * torch.randn(B, H, L, 64, generator=g) for _ in range(4))
    table = torch.randn(32, H, generator=g)
    big_q, big_k, big_v = q.clone(), k.clone(), v.clone()
    tiny = 2e-38 * (1.0 + torch.rand(B, H, L, generator=g)) * (1 - 2 * torch.randint(0, 2, (B, H, L), generator=g))
    big_q[..., 0] = tiny           # (products of some 7 to 14)
    big_k[:, :, 5, 0] = 3.4e38
    big_v[:, :, 7, 3] = 3.4e38
    d2 = d.clone()
    d2[..., 3] = tiny.flip(-1)
    ins = [t.to(gpu_device).requires_grad_() for t in (big_q, big_k, big_v, table)]
    o = t5.flash_attention_with_fusing_bias(*ins, causal=False, sm_scale=1.0)
    got = [o, *torch.autograd.grad(o, ins, d2.to(gpu_device))]
    want = _exact(*ins, False, 1.0, d2)
    for t, r in zip(got, want):
        t, fits = t.detach().double().cpu(), r.abs() < 3.39e38
        assert t[fits].isfinite().all() and t[r.abs() > 3.41e38].isinf().all()
        # (a column's scale; columns of sums below the smallest normal number aside.  Products on the fp32 matrix cores are up to
        # 5e-5 from the formulas here: scores reach 25 and one key has most rows' weight)
        assert ((t - r).abs() <= 2e-4 * r.abs().amax(dim=-2, keepdim=True) + 1e-36)[fits].all()
    bad_k = k.clone()
    bad_k[:, :, 40, 0] = math.inf
    for causal in (False, True):
        out = t5.flash_attention_with_fusing_bias(q.to(gpu_device), bad_k.to(gpu_device), v.to(gpu_device), table.to(gpu_device),
                                                  causal=causal, sm_scale=1.0).cpu()
        clean = t5.flash_attention_with_fusing_bias(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), table.to(gpu_device),
                                                    causal=causal, sm_scale=1.0).cpu()
        sees = torch.arange(L)[None, None, :] >= (40 if causal else 0)
        hidden = q[..., 0] < 0          # score of minus infinity
        assert out[(sees & ~hidden).expand(B, H, L)].isnan().all()
        rest = sees & hidden
        assert out[rest.expand(B, H, L)].isfinite().all()
        drop = torch.ones(L, dtype=torch.bool)
        drop[40] = False
        rel = torch.arange(L)[None, :] - torch.arange(L)[:, None]
        s = (q.double() @ k.double().transpose(2, 3)) + table.double()[O.relative_position_bucket(rel, not causal, 32, 128)].permute(2, 0, 1)
        s = s.masked_fill(~drop[None, :] | ((rel > 0) if causal else torch.zeros_like(rel, dtype=torch.bool)), -math.inf)
        without = torch.softmax(s, -1) @ v.double()
        pick = rest.expand(B, H, L)
        assert (out.double()[pick] - without[pick]).norm() <= 2e-6 * without[pick].norm()
        if causal:
            before = (~sees).expand(B, H, L) & (torch.arange(L) < 32)[None, None, :]
            assert (out[before] - clean[before]).norm() <= 2e-6 * clean[before].norm()


# operands of which unscaled bf16 parts would lose bits: all of v (down to denormal ones), of dout, of k or of q, a factor of the scores, and products
# of dout and v that leave no room for a factor
@pytest.mark.parametrize("B,causal", [(1, False), (40, True)])
@pytest.mark.parametrize("small,by", [("v", 2.0 ** -112), ("v", 2.0 ** -124), ("v", 2.0 ** -138), ("d", 2.0 ** -112), ("d", 2.0 ** -124), ("k", 2.0 ** -112),
                                      ("k", 2.0 ** -124), ("q", 2.0 ** -124), ("s", 2.0 ** -100), ("vd", 2.0 ** 50)])
def test_small_operands_keep_their_bits(gpu_device, B, causal, small, by):
    import turbot5_amd as t5
    H, L = 8, 130
    g = torch.Generator().manual_seed(B + len(small))
    q, k, v, d = (0.5 * torch.randn(B, H, L, 64, generator=g) for _ in range(4))
    table = torch.randn(32, H, generator=g)
    scale = 1.0
    if small == "v":
        v *= by
    elif small == "d":
        d *= by
    elif small == "vd":
        v, d = v * by, d * by
    elif small == "k":
        k *= by
    elif small == "q":
        q *= by
    else:
        scale, q, k = by, q * 2.0 ** 60, k * 2.0 ** 40
    ins = [t.to(gpu_device).requires_grad_() for t in (q, k, v, table)]
    o = t5.flash_attention_with_fusing_bias(*ins, causal=causal, sm_scale=scale)
    got = [o, *torch.autograd.grad(o, ins, d.to(gpu_device))]
    # relative as in the test of ordinary sizes (a gradient's terms cancel to a few per cent of their size); half a step of the denormal numbers for each
    # term of a sum, and a result that is rounded to one
    for t, r, tol in zip(got, _exact(*ins, causal, scale, d), (2e-6, 7e-6, 7e-6, 7e-6, 7e-6)):
        assert (t.double().cpu() - r).norm() <= tol * r.norm() + L * 2.0 ** -149 * r.numel() ** 0.5, small


@pytest.mark.parametrize("B", [1, 48])
def test_scores_of_the_smallest_and_the_largest_numbers(gpu_device, B):
    """Scores of some 6 to 13 from numbers of 2e-38 and 3.3e38 (finite in bf16)."""
    import turbot5_amd as t5
    H, L = 8, 96
    g = torch.Generator().manual_seed(7)
    q, k, v, d = (0.5 * torch.randn(B, H, L, 64, generator=g) for _ in range(4))
    table = torch.randn(32, H, generator=g)
    q[..., 0] = 2e-38 * (1.0 + torch.rand(B, H, L, generator=g))
    k[:, :, 5, 0] = 3.3e38
    d *= 0.1                       # (dq holds a tenth of the largest number)
    ins = [t.to(gpu_device).requires_grad_() for t in (q, k, v, table)]
    o = t5.flash_attention_with_fusing_bias(*ins, causal=False, sm_scale=1.0)
    got = [o, *torch.autograd.grad(o, ins, d.to(gpu_device))]
    # (the first column of dq and dk is far from the others.  Scores that reach 15 carry the roundings of their sums into probabilities: 1e-5
    # to 6e-5 of a head's largest value; scores off by 5e-3, as lost bits make them, are above)
    for i, (t, r) in enumerate(zip(got, _exact(*ins, False, 1.0, d))):
        for columns in (slice(0, 1), slice(1, None)) if i in (1, 2) else (slice(None),):
            a, b = t.double().cpu()[..., columns], r[..., columns]
            assert ((a - b).abs() <= 1e-4 * b.abs().amax(dim=(-2, -1), keepdim=True) + L * 2.0 ** -149).all()


@pytest.mark.parametrize("B", [1, 48])
@pytest.mark.parametrize("fp32_math", [False, True])
@pytest.mark.parametrize("what", ["k", "v"])
def test_a_row_that_is_not_finite_stays_within_its_blocks(gpu_device, monkeypatch, B, fp32_math, what):
    """Causal backward, key 70 infinite (or its value NaN): dq of queries before its block of 32 keys and queries is that without it, and
    queries behind it that see it are NaN; queries 64 to 69, in one block with some that see it, may be either."""
    import turbot5_amd as t5
    from turbot5_amd import ops
    monkeypatch.setattr(ops, "BACKWARD_FP32_MATH", fp32_math)
    H, L = 8, 160
    g = torch.Generator().manual_seed(13)
    q, k, v, d = (0.5 * torch.randn(B, H, L, 64, generator=g) for _ in range(4))
    q[..., 0] = q[..., 0].abs() + 0.1         # (a score of plus infinity)
    table = torch.randn(32, H, generator=g)

    def dq(k, v):
        ins = [t.to(gpu_device).requires_grad_() for t in (q, k, v, table)]
        return torch.autograd.grad(t5.flash_attention_with_fusing_bias(*ins, causal=True, sm_scale=1.0), ins[0], d.to(gpu_device))[0]

    clean = dq(k, v)
    if what == "k":
        k[:, :, 70, 0] = math.inf
    else:
        v[:, :, 70, 5] = math.nan
    got = dq(k, v)
    assert got[:, :, 70:].isnan().all()
    assert (got[:, :, :64] - clean[:, :, :64]).norm() <= 7e-6 * clean[:, :, :64].norm()


# (a block of 64 rows and one more; packed sequences with an empty one)
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("causal", [False, True])
def test_products_on_the_fp32_matrix_cores_on_demand(gpu_device, monkeypatch, packed, causal):
    """BACKWARD_FP32_MATH, fp32_math of the C entry points: the kernels of the other head sizes."""
    import turbot5_amd as t5
    from turbot5_amd import ops
    g = torch.Generator().manual_seed(9)
    shape = (195, 4, 64) if packed else (2, 4, 130, 64)
    q, k, v, d = (0.5 * torch.randn(*shape, generator=g) for _ in range(4))
    table = torch.randn(32, 4, generator=g)
    ins = [t.to(gpu_device).requires_grad_() for t in (q, k, v, table)]
    if packed:
        cu = torch.tensor([0, 65, 65, 195], dtype=torch.int32, device=gpu_device)
        o = t5.flash_attention_with_fusing_bias_varlen(*ins, cu, cu, 130, 130, causal=causal, sm_scale=1.0)
        parts = [_exact(*(t[a:b].transpose(0, 1)[None] for t in (q, k, v)), table, causal, 1.0, d[a:b].transpose(0, 1)[None]) for a, b in ((0, 65), (65, 195))]
        want = [torch.cat([p[i][0].transpose(0, 1) for p in parts]) for i in range(1, 4)] + [parts[0][4] + parts[1][4]]
    else:
        o = t5.flash_attention_with_fusing_bias(*ins, causal=causal, sm_scale=1.0)
        want = _exact(q, k, v, table, causal, 1.0, d)[1:]
    dout = d.to(gpu_device)
    split = torch.autograd.grad(o, ins, dout, retain_graph=True)
    monkeypatch.setattr(ops, "BACKWARD_FP32_MATH", True)
    cores = torch.autograd.grad(o, ins, dout)
    assert not any(torch.equal(a, b) for a, b in zip(split[:3], cores))
    for a, b, r in zip(split, cores, want):
        assert all((t.double().cpu() - r).norm() <= 7e-6 * r.norm() for t in (a, b))


def test_lut_of_a_table_is_not_marked_built_by_an_fp32_call(gpu_device):
    """The fp32 kernel reads no distance image: a 16-bit call with the same table builds its own."""
    import turbot5_amd as t5
    g = torch.Generator().manual_seed(6)
    q, k, v = (0.5 * torch.randn(1, 4, 200, 64, generator=g) for _ in range(3))
    table = torch.randn(32, 4, generator=g).to(gpu_device)
    t5.flash_attention_with_fusing_bias(*(t.to(gpu_device) for t in (q, k, v)), table, sm_scale=1.0)
    b = [t.bfloat16() for t in (q, k, v)]
    out = t5.flash_attention_with_fusing_bias(*(t.to(gpu_device) for t in b), table, sm_scale=1.0)
    want = O.dense_attention(*b, table.cpu(), False, 1.0)
    assert (out.float().cpu() - want).abs().max() <= 2e-2
