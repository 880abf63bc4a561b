"""Experts with more rows than eight tiles of the 256x256 kernel hold: the order of the tile list goes by groups of eight tiles of one expert.  Against the oracle, at the bar of
test_gpu_linasun.py for bfloat16 (0.03 of the logits' spread), rows on both sides of eight tiles; and the same bits whatever else shares the pass."""
import pytest
import torch

import linasun_cases as LC
from oracle import linasun as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows', [2047, 2048, 2049, 2305])
def test_experts_of_many_tiles(rows):
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = LC.config(256, 120, [(LC.mixer(4, 64, 64, 64, 64, 0.15), LC.moe(2, 2, 128, 1.5)), (LC.mixer(4, 64, 64, 64, 64, 0.15), LC.moe(3, 2, 256, 1.5))])
    w = LC.weights(cfg, 31)
    m = LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.bfloat16, max_tokens=rows, max_seqs=2)
    a, b = LC.tokens(cfg, rows, 3), LC.tokens(cfg, 300, 4)
    want = sorted({0, 255, 256, 1023, 2046, rows - 1})
    z = m.step([('a', a, want)]).cpu()
    m.end('a')
    both = m.step([('a', a, want), ('b', b, [299])]).cpu()
    m.close()
    assert LC.rel(z, O.forward(w, cfg, a)[want]) < 0.03
    assert torch.equal(both[:len(want)], z)
