"""16-bit backward: the block sizes that a launch's size chooses (four, two or one wavefront to 32 rows), against the formulas in
64 bits."""
import pytest
import torch

from tests.closed_forms import dense_64_bits

pytestmark = pytest.mark.gpu


# 64-row blocks: up to 256 (causal 384), with at most 128 rows of the other kind and with more / more blocks, fewer than 512 of 128 rows (head_dim 128: 320, causal: 768) / more still; edges
# of tiles of 64 and 128, one row, rows without keys; bucketings without room for the largest tiles: saturated
# at 773 (head_dim 128, whose limit is 219; 64 has room) and at 952 (64 too, whose limit is 901)
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.float16)])
@pytest.mark.parametrize("B,H,M,N,causal,nb,far", [(1, 2, 1, 129, False, 32, 128), (1, 2, 129, 127, False, 32, 128), (2, 3, 128, 129, False, 32, 128),
                                                   (2, 4, 300, 257, True, 32, 128), (2, 2, 65, 500, True, 32, 128),
                                                   (1, 2, 200, 130, True, 32, 128), (17, 16, 100, 97, False, 32, 128),
                                                   (40, 10, 97, 65, True, 32, 128), (33, 16, 130, 33, False, 32, 128),
                                                   (1, 2, 700, 700, False, 64, 1000), (1, 2, 1000, 1000, False, 64, 1250)])
def test_gradients_against_64_bits(gpu_device, D, dtype, B, H, M, N, causal, nb, far):
    import turbot5_amd as t5
    g = torch.Generator().manual_seed(B + M + N + D)
    q, k, v, d = ((0.5 * torch.randn(B, n, H, D, generator=g)).to(dtype).to(gpu_device).transpose(1, 2) for n in (M, N, N, M))
    ins = [t.requires_grad_() for t in (q, k, v, torch.randn(nb, H, generator=g).to(gpu_device))]
    o = t5.flash_attention_with_fusing_bias(*ins, causal=causal, sm_scale=0.5, NUM_BUCKETS=nb, MAX_DISTANCE=far)
    got = torch.autograd.grad(o, ins, d)
    # bf16's half unit is 2^-9: of o (in delta), of a probability and of dS, and of the result: 4 x 2^-9 at most, 1 % with the sums
    for t, r in zip(got, dense_64_bits(*ins, causal, 0.5, far, d)[1:]):
        assert (t.double().cpu() - r).norm() <= 1e-2 * r.norm()
