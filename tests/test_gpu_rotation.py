"""The rotation of a head's entries, where half of it is a multiple of eight (a lane's partners side by side) and where it is not: one arithmetic."""
import pytest
import torch

import lugasun_cases as LC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('entry', range(8))
def test_odd_halves_rotate_as_even_ones_do(entry):
    """Base one turns all pairs alike.  Heads whose only entries are `entry` and its partner then give the same float32 bits with a partner 8 entries on (a rotation of 16) and 9 (of 18): each sum has the
    same two terms.  Prompts and decoded rows, attention and retention."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    got = []
    for half in (8, 9):
        cfg = LC.config(128, 90, [LC.layer(LC.heads(2, 1, 64, 64, 64, rot=(1.0, 2 * half)), LC.ret(64, 64, (0.9, 0.97), rot=(1.0, 2 * half)), None)], side=8)
        w = LC.weights(cfg, 41)
        for name in ('left.q', 'left.k', 'right.q', 'right.k'):
            full = w['l0.mix.' + name].view(-1, 64, 128)
            few = torch.zeros_like(full)
            few[:, [entry, entry + half]] = 6 * full[:, :2]
            w['l0.mix.' + name] = few.flatten(0, 1)
        for name in ('left.q.norm', 'left.k.norm'):
            gain = w['l0.mix.' + name].clone()
            w['l0.mix.' + name][[entry, entry + half]] = gain[:2]
        m = LugasunForCausalLM.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=64, max_seqs=2)
        t = LC.tokens(cfg, 40, seed=7)
        z = [m.step([('r', t[:32], list(range(32)))])] + [m.step([('r', [x], [0])]) for x in t[32:]]
        got.append(torch.cat(z).cpu())
        m.close()
    assert torch.equal(*got), float((got[0] - got[1]).abs().max())
