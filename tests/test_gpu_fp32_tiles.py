"""float32 prompt products with more K-tiles than lie in LDS, and row tiles of few live fragments: 65 to 80 rows of a 12800-column product go to 128-row tiles whose waves hold two and three of four
fragments, 81 and 113 fill more of them.  Against the oracle (2e-5 of the logits' spread, the bar of test_gpu_few_rows.py), and the same bits beside another prompt, where other tiles take the rows."""
import pytest
import torch

import linasun_cases as LIN
import lugasun_cases as LUG
from oracle import linasun as OLIN
from oracle import lugasun as OLUG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows', [65, 80, 81, 113])
@pytest.mark.parametrize('name', ['wide', 'deep', 'experts'])
def test_fp32_prompt_tiles(name, rows):
    from callireader_amd import modeling_decoder as MD
    if name == 'experts':
        cases, oracle, cls, cfg = LIN, OLIN, MD.LinasunForCausalLM, LIN.config(640, 300, [(LIN.mixer(3, 64, 72, 96, 64, 0.15), LIN.moe(3, 2, 704, 1.5))])
    else:
        cases, oracle, cls = LUG, OLUG, MD.LugasunForCausalLM
        cfg = LUG.config(512 if name == 'wide' else 1088, 300, [LUG.layer(LUG.heads(3, 1, 64, 40, 4096), LUG.ret(64, 72, (0.9,)), 12800 if name == 'wide' else 1472)], side=20)
    w = cases.weights(cfg, 47)
    m = cls.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=rows, max_seqs=2)
    t, want = cases.tokens(cfg, rows, seed=6), [0, 15, 16, rows // 2, rows - 17, rows - 1]
    z = m.step([('a', t, want)]).cpu()
    m.end('a')
    both = m.step([('a', t, want), ('b', t[:61], [0])]).cpu()
    m.close()
    assert cases.rel(z, oracle.forward(w, cfg, t)[want]) < 2e-5
    assert torch.equal(both[:len(want)], z)
