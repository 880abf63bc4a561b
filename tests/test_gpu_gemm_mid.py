"""The tile shapes of gemm_mid.hip: every epilogue of every shape at the edges of tiles, K pipelines and vector stores, against a plain fp32 expression (outputs are bf16: two ulp, 1.6e-2,
and an absolute floor for cancellation) and, bit for bit, against each other and the 256x256 kernel: a row's sum is the same chain of MFMAs whichever kernel takes it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TILES = range(16, 29)                                   # cr_op_gemm's pins of gemm_mid's shapes
# K-tiles from one to more than any shape keeps in flight; N with and without whole vectors and fragments; rows around fragments and row tiles
SHAPES = [(1, 64, 64), (15, 200, 128), (17, 72, 704), (33, 331, 192), (65, 272, 1344), (129, 512, 256), (300, 1040, 640)]


def rb(t):
    return t.to(torch.bfloat16).float()


@pytest.mark.parametrize('M,N,K', SHAPES)
def test_every_shape_and_epilogue(M, N, K):
    from callireader_amd import engine as E
    g = torch.Generator().manual_seed(M * 1000 + N)
    dev = torch.device('cuda', 0)
    A, W = torch.randn(M, K, generator=g).bfloat16().to(dev), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(dev)
    bias, scale, res = ((torch.randn(*s, generator=g) * 0.3).bfloat16().to(dev) for s in ((N,), (N,), (M + 8, N)))
    acc = A.float() @ W.float().T
    lin = rb(acc + bias.float())
    cases = {'store': (0, dict(bias=bias), lin), 'gelu': (1, dict(bias=bias), rb(torch.nn.functional.gelu(lin))),
             'scaled residual': (2, dict(bias=bias, scale=scale, res=res), rb(res[:M].float() + rb(lin * scale.float()))), 'residual': (3, dict(res=res), rb(res[:M].float() + rb(acc))),
             'fp32': (6, dict(out_dtype=torch.float32), rb(acc)), 'relu2': (12, {}, rb(acc.clamp(min=0).square()))}
    if N % 16 == 0:
        gu = rb(acc).view(M, N // 16, 2, 8)
        cases['swiglu'] = (4, {}, rb(rb(torch.nn.functional.silu(gu[:, :, 0])) * gu[:, :, 1]).reshape(M, N // 2))
    for name, (epi, kw, want) in cases.items():
        first = None
        for tile in list(TILES) + ([2] if K % 128 == 0 else []):
            out = E.op_gemm(epi, A, W, kernel=tile, **kw)
            torch.cuda.synchronize()
            if first is None:
                first = out
                torch.testing.assert_close(out.float(), want, rtol=1.6e-2, atol=2e-2, msg=lambda m: f'{name}: {m}')
            assert torch.equal(out, first), (name, tile)


@pytest.mark.parametrize('tile', [*range(16, 26), 28, 29, 255])
def test_a_shape_that_cannot_take_the_epilogue_is_an_error(tile):
    """First maxima of 64-column blocks need a wave of 64 columns, which 96 x 256 and 128 x 256 alone have (26 and 27); pins past the last shape (28) name none."""
    from callireader_amd import engine as E
    A, W = torch.zeros(70, 128, device='cuda', dtype=torch.bfloat16), torch.zeros(192, 128, device='cuda', dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        E.op_gemm(8, A, W, kernel=tile)


@pytest.mark.parametrize('far', ['activations', 'weights'])
def test_rows_more_than_4_gib_apart(far):
    """The 256x256 kernel, which this shape would take, reaches its rows by 32-bit byte offsets; an operand that spans more goes to the tile shapes here, and a pin is an error."""
    from callireader_amd import engine as E
    g = torch.Generator().manual_seed(7)
    dev = torch.device('cuda', 0)
    M, N, K = 1536, 8192, 512
    A, W = torch.randn(M, K, generator=g).bfloat16().to(dev), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(dev)
    want = E.op_gemm(0, A, W)
    rows = M if far == 'activations' else N
    ld = (2 ** 31 // (rows - 1) + 15) // 8 * 8
    wide = torch.zeros(rows * ld, device=dev, dtype=torch.bfloat16).view(rows, ld)[:, :K]
    wide.copy_(A if far == 'activations' else W)
    args = (wide, W) if far == 'activations' else (A, wide)
    assert torch.equal(E.op_gemm(0, *args), want)
    with pytest.raises(RuntimeError):
        E.op_gemm(0, *args, kernel=2)
    near = (args[0][:-2], W) if far == 'activations' else (A, args[1][:-2])      # the last offset below 4 GiB
    torch.testing.assert_close(E.op_gemm(0, *near, kernel=2), want[:-2] if far == 'activations' else want[:, :-2], rtol=0, atol=0)


def test_rows_of_patches_keys_of_the_table_and_slices():
    """Position rows behind a class row (epi 5), first maxima of 64-column blocks (epi 8), K-slices (epi 7), an output in place of its residual."""
    from callireader_amd import engine as E
    g = torch.Generator().manual_seed(3)
    dev = torch.device('cuda', 0)
    M, N, K, group = 3 * 40, 192, 320, 40
    A, W = torch.randint(-2, 3, (M, K), generator=g).bfloat16().to(dev), torch.randint(-2, 3, (N, K), generator=g).bfloat16().to(dev)
    W[70] = W[66]                                        # equal keys: the first one wins
    pos, acc = torch.randn(group + 1, N, generator=g).bfloat16().to(dev), A.float() @ W.float().T
    for tile in TILES:
        out = E.op_gemm(5, A, W, res=pos, group=group, kernel=tile).view(3, group + 1, N)
        assert torch.equal(out[:, 1:].float(), rb(rb(acc).view(3, group, N) + pos[1:].float())), tile
        x = pos[:1].repeat(M, 1).contiguous()
        E.op_gemm(3, A, W, res=x, out=x, kernel=tile)
        assert torch.equal(x.float(), rb(pos[:1].float() + rb(acc))), tile
        part = E.op_gemm(7, A, W, group=5, kernel=tile).view(8, M, N)
        assert torch.equal(part[:5].sum(0), acc) and float(part[5:].abs().max()) == 0.0, tile
    for tile in (26, 27):
        out = E.op_gemm(8, A, W, kernel=tile)[:, :3].cpu()
        val = ((out >> 32) & 0xFFFFFFFF).to(torch.int32).view(torch.float32)
        mx, at = rb(acc).cpu().view(M, 3, 64).max(-1)
        assert torch.equal(val, mx) and torch.equal(out & 0xFFFFFFFF, at + 64 * torch.arange(3)), tile
