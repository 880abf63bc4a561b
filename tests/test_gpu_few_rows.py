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


@pytest.mark.parametrize('rows', [1, 16, 17, 49, 127, 129, 290, 1030])
@pytest.mark.parametrize('name', ['lugasun', 'linasun'])
def test_fp32_prompt_rows(name, rows):
    """Prompts in float32: row counts around the row tiles' fragments (16) and heights, widths that leave columns over in every tile shape, a K of one K-tile, of odd and even numbers of
    them; the last rows and some inside against the oracle, and the same bits whatever else is prefilled with them."""
    from callireader_amd import modeling_decoder as MD
    if name == 'lugasun':
        cases, oracle, cls = LUG, OLUG, MD.LugasunForCausalLM
        cfg = LUG.config(192, 300, [LUG.layer(LUG.heads(3, 1, 64, 40, 4096), LUG.ret(64, 72, (0.9,)), 328)], side=20)
    else:
        cases, oracle, cls, cfg = LIN, OLIN, MD.LinasunForCausalLM, LIN.config(320, 300, [(LIN.mixer(3, 64, 72, 96, 64, 0.15), LIN.moe(3, 2, 200, 1.5))])
    w = cases.weights(cfg, 43)
    m = cls.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=rows, max_seqs=2)
    t, want = cases.tokens(cfg, rows, seed=5), sorted({0, rows // 3, max(rows - 17, 0), rows - 1})
    z = m.step([('a', t, want)]).cpu()
    m.end('a')
    both = m.step([('a', t, want), ('b', t[:min(rows, 70)], [0])]).cpu()
    m.close()
    assert cases.rel(z, oracle.forward(w, cfg, t)[want]) < 2e-5
    assert torch.equal(both[:len(want)], z)


@pytest.mark.parametrize('name', ['lugasun_huge', 'linasun_many_heads'])
def test_fp32_decode_row_alone_and_among_others(name):
    from callireader_amd import modeling_decoder as MD
    cases, _, cfg = CASES[name]
    cls = MD.LugasunForCausalLM if cases is LUG else MD.LinasunForCausalLM
    m = cls.from_state_dict(cases.weights(cfg, 44), cfg, dtype=torch.float32, max_tokens=48, max_seqs=61)
    toks = [cases.tokens(cfg, 3 + 7 * i % 40, seed=i) for i in range(60)]
    m.step([(i, t[:-1], []) for i, t in enumerate(toks)])
    z = m.step([(i, t[-1:], [0]) for i, t in enumerate(toks)]).cpu()
    m.step([('a', toks[7][:-1], [])])
    alone = m.step([('a', toks[7][-1:], [0])]).cpu()
    m.close()
    assert torch.equal(alone[0], z[7])


# sums cut into parts (K of 1024 and 2048 in four, the feed-forward's 1088 in two of 17 blocks, which chains of three do not divide)
WIDE_SUMS = LUG.config(1024, 300, [LUG.layer(LUG.heads(4, 2, 64, 64, 4096), LUG.ret(64, 64, (0.9, 0.99)), 1088)], side=20, loop=(0, 1, 2))


@pytest.mark.parametrize('name', [*CASES, 'lugasun_wide_sums'])
def test_fp32_row_among_64_and_65(name):
    """64 rows are the few-row kernel's, 65 the tile kernel's: a row's bits are the same alone, among 64 and among 65, decoded or asked for in a prompt."""
    from callireader_amd import modeling_decoder as MD
    cases, oracle, cfg = CASES.get(name, (LUG, OLUG, WIDE_SUMS))
    cls = MD.LugasunForCausalLM if cases is LUG else MD.LinasunForCausalLM
    w = cases.weights(cfg, 45)
    m = cls.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=100, max_seqs=65)
    toks = [cases.tokens(cfg, 3 + 7 * i % 40, seed=i) for i in range(65)]

    def decoded(n):
        m.step([(i, t[:-1], []) for i, t in enumerate(toks[:n])])
        z = m.step([(i, t[-1:], [0]) for i, t in enumerate(toks[:n])])
        m.slots.clear()
        return z

    def asked(n):
        z = m.step([('a', t, list(range(90 - n, 90)))])
        m.slots.clear()
        return z

    one, few, many = decoded(1), decoded(64), decoded(65)
    assert torch.equal(few, many[:64]) and torch.equal(one, few[:1])
    assert cases.rel(many[64:].cpu(), oracle.forward(w, cfg, toks[64])[-1:]) < 2e-5
    t = cases.tokens(cfg, 90, seed=3)
    one, few, many = asked(1), asked(64), asked(65)
    assert torch.equal(few, many[1:]) and torch.equal(one, few[-1:])
    assert cases.rel(many.cpu(), oracle.forward(w, cfg, t)[25:]) < 2e-5
    m.close()


# a latent of more column quads than a prompt's workgroup has threads
WIDE_LATENT = LIN.config(128, 90, [(LIN.mixer(2, 90, 100, 40, 1100, 0.1), None)])


@pytest.mark.parametrize('name,n', [('linasun_ragged', 60), ('linasun_many_heads', 90), ('deep_latent', 70), ('deep_latent', 1030), ('wide_latent', 40), ('wide_latent', 1100)])
def test_fp32_row_decoded_and_in_a_prompt(name, n):
    """The last tokens of a sequence as one prompt, as decode steps, and as a prompt of one token beside another request: the same bits.  (Cached rows of 64 to 1152 columns, one and two
    blocks of keys.  Retention's two kernels add the squares of a row in orders of their own.)"""
    from callireader_amd import modeling_decoder as MD
    cfg = {'deep_latent': LIN.DEEP_LATENT, 'wide_latent': WIDE_LATENT}.get(name) or CASES[name][2]
    w, t = LIN.weights(cfg, 46), LIN.tokens(cfg, n, seed=4)
    m = MD.LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=n, max_seqs=2)
    whole = m.step([('a', t, [n - 2, n - 1])])
    m.slots.clear()
    m.step([('a', t[:-2], [])])
    steps = torch.cat([m.step([('a', [x], [0])]) for x in t[-2:]])
    m.slots.clear()
    m.step([('a', t[:-1], [])])
    beside = m.step([('a', t[-1:], [0]), ('b', t[:9], [])])
    m.close()
    assert torch.equal(whole, steps) and torch.equal(whole[1:], beside)
    assert LIN.rel(whole.cpu(), OLIN.forward(w, cfg, t)[-2:]) < (2e-5 if n < 1000 else 1e-4)      # (angles of a thousand radians: 6e-5 radians of fp32 rounding)
