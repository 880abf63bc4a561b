"""The rotation of a head's entries, where half of it is a multiple of eight (a lane's partners side by side) and where it is not: one arithmetic."""
import pytest
import torch

import lugasun_cases as LC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('entry', range(8))
def test_odd_halves_rotate_as_even_ones_do(entry):
    """Base one turns all pairs alike.  Heads whose only entries are `entry` and its partner then give the same float32 bits with a partner 8 entries on (a rotation of 16), 9 (of 18) and
    12 (of 24, by fours): each sum has the same two terms.  Prompts and decoded rows, attention and retention."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    got = []
    for half in (8, 9, 12):
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
    for z in got[1:]:
        assert torch.equal(z, got[0]), float((z - got[0]).abs().max())


@pytest.mark.parametrize('halves', [(8, 16), (12, 20), (9, 14)])
@pytest.mark.parametrize('heads', [(2, 1, 2), (12, 3, 9), (32, 16, 17)])
def test_a_row_is_the_same_in_workgroups_of_any_width(heads, halves):
    """Rows of prompts alone and in portions long enough for each number of waves a workgroup of the row kernel has (four beside each other; one for every task or every second; four; even shares):
    what the layer keeps of them -- cached keys and values and retention's state, which the same decoded rows then read -- has the same bits.  5, 8 and 14 tasks; halves of a multiple of eight, of four, of neither."""
    from callireader_amd.modeling_decoder import LugasunForCausalLM
    H, G, R = heads
    cfg = LC.config(64, 60, [LC.layer(LC.heads(H, G, 48, 48, 4096, rot=(100.0, 2 * halves[0])), LC.ret(48, 48, (0.9,) * R, rot=(50.0, 2 * halves[1])), None)], side=8)
    m = LugasunForCausalLM.from_state_dict(LC.weights(cfg, 43), cfg, dtype=torch.float32, max_tokens=2100, max_seqs=2)
    t, last = LC.tokens(cfg, 40, seed=9), LC.tokens(cfg, 8, seed=10)
    got = []
    for n in (0, 480, 560, 1100, 1700, 2050):
        others = [('o', LC.tokens(cfg, n, seed=11), [0])] if n else []
        m.step([('r', t, [39])] + others)
        got.append(torch.cat([m.step([('r', [x], [0])]) for x in last]).cpu())
        for s in ['r'] + ['o'] * bool(n):
            m.end(s)
    m.close()
    for z in got[1:]:
        assert torch.equal(z, got[0]), float((z - got[0]).abs().max())
