"""Routing of many tokens: the router product through LDS and the fragment-ordered weights, at widths and expert counts that its chunks of 512 columns and blocks of 16 do not divide, and the
assignments' plan in one workgroup (up to 8192) and in parts (above): against the oracle."""
import pytest
import torch

import linasun_cases as LC
from oracle import linasun as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('width,experts,top,groups,keep,n', [(320, 3, 1, 1, 1, 333), (2304, 40, 2, 5, 3, 700), (1024, 96, 6, 8, 4, 683), (4224, 33, 4, 3, 2, 1025), (512, 200, 5, 10, 4, 1400), (320, 33, 8, 3, 3, 1024),
                                                                  (320, 33, 8, 3, 3, 1025), (512, 200, 10, 10, 9, 1300)])
def test_many_tokens(width, experts, top, groups, keep, n):
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = LC.config(width, 120, [(LC.mixer(2, 64, 64, 64, 64, 0.15), LC.moe(experts, top, 64, 2.0, (groups, keep)))])
    w = {k: (6 * v.float()).to(v.dtype) if k.endswith('router') else v for k, v in LC.weights(cfg, 51).items()}      # (choices that rounding does not turn)
    t = LC.tokens(cfg, n, seed=3)
    m = LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.bfloat16, max_tokens=n)
    z = m.step([('r', t, list(range(n)))]).cpu()
    m.close()
    ref = O.forward(w, cfg, t)
    d = z - ref
    err = (d - d.mean(-1, keepdim=True)).pow(2).mean(-1).sqrt() / ref.std()
    assert float(err.median()) < 2e-2 and float((err > 0.1).float().mean()) < 0.02, (float(err.median()), float(err.max()))


@pytest.mark.parametrize('width,experts,top,groups,keep', [(64, 3, 1, 1, 1), (320, 17, 2, 1, 1), (1088, 33, 3, 3, 2), (2048, 64, 4, 8, 4), (1536, 64, 4, 8, 4), (2048, 32, 4, 4, 2)])
def test_decoded_rows(width, experts, top, groups, keep):
    """Decoded rows: update, scores and choice in one launch, at widths that the sixteen K-slices and expert counts that the blocks of 16 do not divide."""
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = LC.config(width, 120, [(LC.mixer(2, 64, 64, 64, 64, 0.15), LC.moe(experts, top, 64, 2.0, (groups, keep)))])
    w = {k: (6 * v.float()).to(v.dtype) if k.endswith('router') else v for k, v in LC.weights(cfg, 53).items()}
    rows, n, new = 7, 12, 6
    t = [LC.tokens(cfg, n + new, seed=20 + r) for r in range(rows)]
    m = LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.bfloat16, max_tokens=64)
    m.step([(r, t[r][:n], []) for r in range(rows)])
    z = torch.stack([m.step([(r, [t[r][n + i]], [0]) for r in range(rows)]).cpu() for i in range(new)], 1)
    m.close()
    ref = torch.stack([O.forward(w, cfg, t[r])[n:] for r in range(rows)])
    d = z - ref
    err = (d - d.mean(-1, keepdim=True)).pow(2).mean(-1).sqrt() / ref.std()
    assert float(err.median()) < 2e-2 and float((err > 0.1).float().mean()) < 0.05, (float(err.median()), float(err.max()))      # (at most two of 42 rows: a turned choice)


@pytest.mark.parametrize('layout', ['1', '0'])
@pytest.mark.parametrize('width,experts,top,groups,keep', [(64, 3, 1, 1, 1), (320, 17, 3, 1, 1), (1088, 33, 3, 3, 2), (1536, 64, 5, 8, 4), (2048, 32, 3, 4, 2)])
def test_joined_choice_has_the_bits_of_the_separate_kernels(width, experts, top, groups, keep, layout, monkeypatch):
    """Update, scores and choice in one launch against the residual update, the sliced router and the routing kernel, bit for bit, with fragment-ordered weights and without.  Experts come in pairs that
    only the rounding of sums tells apart: the second has the first's weights with columns of equal activations exchanged across K-slices, so another order of a sum turns choices."""
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = LC.config(width, 120, [(LC.mixer(2, 64, 64, 64, 64, 0.15), LC.moe(experts, top, 64, 2.0, (groups, keep)))] * 2)
    w = LC.without_attention(LC.weights(cfg, 57))
    c = torch.arange(width // 4 | 1, width, 2)                # odd columns: cosines of the position, close to one in the last three quarters
    half = len(c) // 2
    a, b = c[:half], c[half:2 * half]
    for name in ('embed', *(f'l{i}.norm{j}' for i in range(2) for j in ('1', '1b', '2', '2b'))):
        w[name][..., b] = w[name][..., a]
    for i in range(2):
        r = w[f'l{i}.mlp.router'].mul_(3)
        twin = r[:experts // 2 * 2:2].clone()
        twin[:, a], twin[:, b] = twin[:, b], twin[:, a].clone()
        r[1:experts // 2 * 2:2] = twin
        w[f'l{i}.mlp.correction'].zero_()
    rows, n, new = 64, 3, 6
    t = [LC.tokens(cfg, n + new, seed=100 + r) for r in range(rows)]
    monkeypatch.setenv('CR_DECODE_LAYOUT', layout)
    got = []
    for joined in ('1', '0'):
        monkeypatch.setenv('CR_DECODE_JOINED', joined)
        m = LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.bfloat16, max_tokens=16, max_seqs=rows)
        m.step([(r, t[r][:n], []) for r in range(rows)])
        z = [m.step([(r, [t[r][n + i]], [0]) for r in range(rows)]) for i in range(new)]
        z += [m.step([(0, [5], [0])])]                        # (one row alone: the same routes)
        got.append(torch.cat(z).cpu())
        m.close()
    assert torch.equal(*got), int((got[0] != got[1]).any(-1).sum())
