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


# (columns, depth, K-slices that the geometry picks, k-steps of a wave): two, three and four row tiles a workgroup, whose batches are 3 or 4 k-steps up to 32 rows and 4, 2 and 2 beyond
TALL = {2: [(2080, 512, 2, 1), (608, 3584, 7, 2), (2080, 1536, 2, 3), (2080, 2560, 2, 5), (4192, 1792, 1, 7)],
        3: [(2064, 512, 2, 1), (624, 3584, 7, 2), (2064, 1536, 2, 3), (2064, 2560, 2, 5), (1776, 7168, 4, 7)],
        4: [(1216, 1792, 7, 1), (1216, 3584, 7, 2), (4160, 1536, 2, 3), (4160, 2560, 2, 5), (4736, 3584, 2, 7)]}


@pytest.mark.parametrize('M', [16, 32, 48, 64])
@pytest.mark.parametrize('N,K,slices,steps', [s for t in TALL.values() for s in t])
def test_slices_of_taller_workgroups(M, N, K, slices, steps):
    from callireader_amd import engine as E
    g = torch.Generator(device='cuda').manual_seed(M + N + K)
    a, w = (torch.randint(-2, 3, (n, K), device='cuda', generator=g).to(torch.bfloat16) for n in (M, N))
    dl = (1, E.op_decode_swizzle(1, w))
    for layout in (None, dl):
        parts = E.op_gemm(7, a, w, kernel=3, decode_layout=layout).reshape(8, M, N)
        assert K == 256 * slices * steps and [bool(p.any()) for p in parts] == [True] * slices + [False] * (8 - slices)
        for s in range(slices):                               # |sum| <= 4 K < 2^24: exact whatever the order
            k = slice(s * K // slices, (s + 1) * K // slices)
            assert torch.equal(parts[s], a[:, k].float() @ w[:, k].float().t())


@pytest.mark.parametrize('M', [16, 32, 48, 64])
@pytest.mark.parametrize('steps', [1, 3, 5, 8])
def test_wide_products_of_four_waves(M, steps):
    from callireader_amd import engine as E
    K, N = 128 * steps, 16400                                 # four row tiles a workgroup, the last one of one
    g = torch.Generator(device='cuda').manual_seed(M + K)
    a, w = (torch.randint(-2, 3, (n, K), device='cuda', generator=g).to(torch.bfloat16) for n in (M, N))
    ref = (a.float() @ w.float().t()).bfloat16().float()
    for layout in (None, (1, E.op_decode_swizzle(1, w))):
        assert torch.equal(E.op_gemm(6, a, w, out_dtype=torch.float32, kernel=3, decode_layout=layout), ref)
