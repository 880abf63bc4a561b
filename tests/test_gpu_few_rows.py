"""Decode batches in float32 at the edges of the few-row kernels (16-row operand tiles, 64 rows at most; K-slices and a wave's share of K that do not divide), against the oracles.
float32 differences are rounding of sums (2e-5 of the logits' spread, the bar of test_gpu_lugasun.py and test_gpu_linasun.py)."""
import pytest
import torch

import linasun_cases as LIN
import lugasun_cases as LUG
from oracle import linasun as OLIN
from oracle import lugasun as OLUG

pytestmark = pytest.mark.gpu
CASES = {'lugasun_ragged': (LUG, OLUG, LUG.RAGGED), 'lugasun_huge': (LUG, OLUG, LUG.HUGE), 'linasun_ragged': (LIN, OLIN, LIN.RAGGED), 'linasun_many_heads': (LIN, OLIN, LIN.MANY_HEADS)}


@pytest.mark.parametrize('rows', [1, 15, 16, 17, 33, 64, 65])
@pytest.mark.parametrize('name', CASES)
def test_fp32_decode_rows(name, rows):
    from callireader_amd import modeling_decoder as MD
    cases, oracle, cfg = CASES[name]
    cls = MD.LugasunForCausalLM if cases is LUG else MD.LinasunForCausalLM
    w = cases.weights(cfg, 41)
    m = cls.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=48, max_seqs=rows)
    toks = [cases.tokens(cfg, 3 + 5 * i % 29, seed=i) for i in range(rows)]
    m.step([(i, t[:-1], []) for i, t in enumerate(toks)])
    z = m.step([(i, t[-1:], [0]) for i, t in enumerate(toks)]).cpu()
    m.close()
    for i in sorted({0, rows // 2, min(15, rows - 1), min(16, rows - 1), rows - 1}):
        assert cases.rel(z[i:i + 1], oracle.forward(w, cfg, toks[i])[-1:]) < 2e-5, i


def test_fp32_long_context_decode():
    """More keys than one block of the plain attention holds (1024), and a latent wider than a thread's one column quad."""
    from callireader_amd import modeling_decoder as MD
    cfg = LUG.config(64, 50, [LUG.layer(LUG.heads(2, 1, 64, 40, 4096), LUG.ret(16, 16, (0.9,)), 32)], side=4)
    for cases, oracle, cls, cfg, n in ((LUG, OLUG, MD.LugasunForCausalLM, cfg, 1100), (LIN, OLIN, MD.LinasunForCausalLM, LIN.DEEP_LATENT, 1030)):
        w, t = cases.weights(cfg, 5), cases.tokens(cfg, n)
        m = cls.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=n)
        m.step([('r', t[:-3], [])])
        z = torch.cat([m.step([('r', [x], [0])]) for x in t[-3:]]).cpu()
        m.close()
        assert cases.rel(z, oracle.forward(w, cfg, t)[-3:]) < 1e-4      # (angles of a thousand radians: 6e-5 radians of fp32 rounding)
