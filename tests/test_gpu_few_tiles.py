"""Few tiles through the vision tower: beside the second norm of a layer workgroups read fc2's weights, for up to four tiles.  Reading leaves nothing behind: a tile's rows have the same bits alone, among
four (the last count with reading) and among five (the first without)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('count', [1, 4])
def test_weights_read_beside_the_norm(count):
    from callireader_amd import synthetic
    from callireader_amd.config import ModelDims
    from callireader_amd.modeling_internvl_chat import InternVLChatModel
    dims = ModelDims.reduced(vit_layers=2, rs_depth=0, llm_layers=0)
    m = InternVLChatModel.from_state_dict(synthetic.make_state_dict(dims, seed=3, parts=('vit', 'mlp1')), dims, max_tokens=64)
    px = synthetic.make_pixels(5, seed=4).cuda()
    five = m.extract_feature(px)
    few = m.extract_feature(px[:count].contiguous())
    torch.cuda.synchronize()
    assert torch.isfinite(few).all() and torch.equal(few, five[:count])
