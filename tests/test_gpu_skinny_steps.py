"""The few-row bf16 product where a wave's share of K is a part of a batch of k-steps, one batch, or some and a part: whole-number data, whose sums are exact in fp32 whatever their order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('M', [1, 16, 17, 33, 64])
@pytest.mark.parametrize('steps', [1, 2, 3, 5, 6, 7, 8, 11, 13])
def test_every_number_of_k_steps_a_wave(M, steps):
    from callireader_amd import engine as E
    K, N = 256 * steps, 208                                   # eight waves of 32-deep steps; 13 row tiles
    g = torch.Generator().manual_seed(100 * M + steps)
    A, W = torch.randint(-2, 3, (M, K), generator=g).float(), torch.randint(-2, 3, (N, K), generator=g).float()
    a, w = A.bfloat16().cuda(), W.bfloat16().cuda()
    ref = A @ W.t()                                           # |sum| <= 4 K < 2^24
    dl = (1, E.op_decode_swizzle(1, w))
    for layout in (None, dl):
        assert torch.equal(E.op_gemm(6, a, w, out_dtype=torch.float32, kernel=3, decode_layout=layout).cpu(), ref.bfloat16().float())
        parts = E.op_gemm(7, a, w, kernel=3, decode_layout=layout).reshape(8, M, N).cpu()
        assert torch.equal(parts.sum(0), ref)

