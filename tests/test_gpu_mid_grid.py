"""Workgroup numbers of the tiled product become tiles by multiplications instead of divisions: every tile once, whatever is left over of row tiles, super-groups of eight of them and fragments, and on both sides
of the row count from which on the kernel divides again (1600 row tiles).  Whole numbers, exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


TILES, GRIDS = [(0, 16, 32), (4, 64, 64), (9, 128, 128), (12, 160, 128)], [(1, 1), (7, 3), (8, 1), (9, 5), (15, 7), (17, 11)]


# (as many row tiles as 1600 with the smallest tile alone)
@pytest.mark.parametrize('tile,bm,bn,rows,cols', [(*t, *g) for g in GRIDS for t in TILES] + [(*TILES[0], *g) for g in ((1599, 1), (1601, 2))])
def test_every_tile_once(tile, bm, bn, rows, cols):
    from callireader_amd import engine as E
    g = torch.Generator().manual_seed(rows + cols)
    M, N, K = rows * bm - bm // 2 + 3, cols * bn - 8, 128
    A, W = (torch.randint(-3, 4, s, generator=g).to(torch.bfloat16).cuda() for s in ((M, K), (N, K)))
    out = torch.full((M, N), 7.5, device='cuda', dtype=torch.bfloat16)
    E.op_gemm(0, A, W, kernel=16 + tile, out=out)
    assert torch.equal(out, (A.float() @ W.float().t()).to(torch.bfloat16))
