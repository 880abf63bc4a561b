"""More tiles than one chunk of the vision tower holds (255) run as chunks of one size: every tile's features are those it has alone, at both ends of each chunk."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('tiles', [255, 256, 257])
def test_tiles_around_the_largest_chunk(tiles):
    from callireader_amd import synthetic
    from callireader_amd.config import ModelDims
    from callireader_amd.engine import Engine
    dims = ModelDims.reduced(vit_layers=1, rs_depth=1, llm_layers=1, vocab=8192)
    eng = Engine(dims)
    eng.load_state_dict(synthetic.make_state_dict(dims, parts=('vit', 'mlp1'), seed=0))
    eng.load_rope()
    eng.finalize()
    g = torch.Generator(device='cuda').manual_seed(tiles)
    px = torch.randn(tiles, 3, 448, 448, generator=g, device='cuda').to(torch.bfloat16)
    out = eng.extract_feature(px)
    for i in (0, (tiles + 1) // 2 - 1, (tiles + 1) // 2, tiles - 1):
        assert torch.equal(out[i], eng.extract_feature(px[i:i + 1])[0]), i
