"""The step of gemm_mid.hip's K loop at its edges: K from one K-tile to more than a round of the buffers and what is asked for beyond it, in each depth of buffers that a tile shape has (one workgroup a
CU, or several), row tiles of every number of fragments, and rows so far apart that a lane's address takes 64 bits.  A row's sum is the same chain of MFMAs whatever the shape: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(M, N, K):
    g = torch.Generator().manual_seed(M + 7 * N + 13 * K)
    return [torch.randn(*s, generator=g).bfloat16().cuda() for s in ((M, K), (N, K), (N,), (M, N))]


# K-tiles: fewer than the buffers, then none, one and two rounds and a rest of each depth (a round of 3 to 12 K-tiles, 14 of seven buffers, and as many again asked for ahead; K = 2304 is two rounds of twelve);
# workgroups: at most one a CU, or several (1500 x 1500: 288 to 8 836 of every shape up to 128 x 64 and 64 x 128)
@pytest.mark.parametrize('K', [64, 192, 320, 448, 704, 960, 1024, 1088, 1216, 1472, 1536, 1792, 2304])
@pytest.mark.parametrize('M,N', [(150, 136), (145, 512), (1111, 1111), (1500, 1500)])
def test_depths_of_buffers(M, N, K):
    from callireader_amd import engine as E
    A, W, bias, res = operands(M, N, K)
    scale = bias.flip(0).contiguous()
    want = (A.double() @ W.double().T + bias.double()).float()
    first = None
    for tile in range(16, 29):
        out = E.op_gemm(0, A, W, bias=bias, kernel=tile)
        if first is None:
            torch.testing.assert_close(out.float(), want, rtol=1e-2, atol=1e-2 * K ** 0.5 / 8)      # one rounding to bf16 (2^-9), sums of K products of unit size in float32
            first, rows = out, E.op_gemm(2, A, W, bias=bias, scale=scale, res=res, kernel=tile)
        assert torch.equal(out, first), tile
        assert torch.equal(E.op_gemm(2, A, W, bias=bias, scale=scale, res=res, kernel=tile), rows), tile
    assert torch.equal(E.op_gemm(0, A, W, bias=bias), first)


@pytest.mark.parametrize('M', [16, 65, 130, 144, 161, 1025])
def test_the_largest_shapes_row_tiles(M):
    """160 x 128: a wave's rows are five fragments or fewer, down to none; every epilogue of it."""
    from callireader_amd import engine as E
    N, K = 208, 640
    A, W, bias, res = operands(M, N, K)
    for epi, kw in ((0, dict(bias=bias)), (1, dict(bias=bias)), (2, dict(bias=bias, scale=bias, res=res)), (3, dict(res=res)), (4, {}), (6, dict(out_dtype=torch.float32)), (12, {}), (7, dict(group=5))):
        assert torch.equal(E.op_gemm(epi, A, W, kernel=28, **kw), E.op_gemm(epi, A, W, kernel=16, **kw)), epi


@pytest.mark.parametrize('far', ['activations', 'weights'])
@pytest.mark.parametrize('ld', [2 ** 31 // 14 * 2 // 8 * 8 - 16, 2 ** 31 // 14 * 2 // 8 * 8 + 8])   # seven rows of bf16 just within 4 GiB (offsets of 32 bits, the last above 2^31), and past it
def test_rows_that_span_4_gib_between_eight(far, ld):
    from callireader_amd import engine as E
    assert (7 * 2 * ld + 128 < 2 ** 32) == (ld < 2 ** 31 // 7)
    M, N, K = (20, 64, 192) if far == 'activations' else (70, 20, 192)
    A, W, bias, _ = operands(M, N, K)
    rows = M if far == 'activations' else N
    wide = torch.empty((rows - 1) * ld + K, device='cuda', dtype=torch.bfloat16).as_strided((rows, K), (ld, 1))
    wide.copy_(A if far == 'activations' else W)
    args = (wide, W) if far == 'activations' else (A, wide)
    for tile in (1, 16, 20, 25, 27, 28):                 # (the dispatcher's choice, and shapes with four to eight rows of both operands to a wave's piece)
        assert torch.equal(E.op_gemm(0, *args, bias=bias, kernel=tile), E.op_gemm(0, A, W, bias=bias, kernel=tile)), tile
