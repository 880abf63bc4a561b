"""The 256x256 kernel's tiles of 192 rows against its tiles of 256: the same bits from every epilogue, rows around a wave's 96 and the tile's 192, N around a wave's 64 columns and a
tile's 256, one and several rounds of tiles, both schedules.  (The 256-row tiles are held against fp32 expressions elsewhere.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu
SHAPES = [(1, 64, 128), (95, 256, 256), (97, 328, 384), (191, 520, 128), (193, 264, 256), (385, 1088, 512), (1920, 8192, 128), (2016, 8256, 256)]


@pytest.mark.parametrize('M,N,K', SHAPES)
def test_the_same_bits_as_256_rows(M, N, K):
    from callireader_amd import engine as E
    g = torch.Generator().manual_seed(M + N)
    dev = torch.device('cuda', 0)
    A, W = torch.randn(M, K, generator=g).bfloat16().to(dev), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(dev)
    bias, scale, res = ((torch.randn(*s, generator=g) * 0.3).bfloat16().to(dev) for s in ((N,), (N,), (M, N)))
    group = next(d for d in (8, 5, 1) if M % d == 0)
    cases = [(0, dict(bias=bias)), (1, dict(bias=bias)), (2, dict(bias=bias, scale=scale, res=res)), (3, dict(res=res)), (5, dict(bias=bias, res=res[:1].repeat(group + 1, 1), group=group)),
             (6, dict(out_dtype=torch.float32)), (12, {})] + [(4, {})] * (N % 16 == 0) + [(8, {})] * (N % 64 == 0 and M > 64)
    for epi, kw in cases:
        a, b, c = (E.op_gemm(epi, A, W, kernel=k, **kw) for k in (5, 7, 8))
        torch.cuda.synchronize()
        if epi == 5:                                         # class rows belong to another launch
            a, b, c = (t.view(M // group, group + 1, N)[:, 1:] for t in (a, b, c))
        if epi == 8:
            a, b, c = (t[:, :N // 64] for t in (a, b, c))
        assert torch.equal(a, b) and torch.equal(a, c), epi
