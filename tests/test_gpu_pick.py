"""The greedy pick over a vocabulary of several parts: equal scores at the parts' edges, with and without a repetition penalty, one and several rows.  Only seven rows of the head are
not zero and they are one vector or its negative, so every step's scores are z, -z and 0 exactly and the pick is a matter of indices."""
import pytest
import torch

import linasun_cases as LC
from oracle import linasun as O

pytestmark = pytest.mark.gpu
PLUS, MINUS = [5, 4095, 4096, 8192, 8999], [17, 4100]


def expected(w, cfg, prompt, n, penalty):
    ids, out = list(prompt), []
    for _ in range(n):
        z = float(O.forward(w, cfg, ids)[-1][PLUS[0]])
        score = torch.zeros(cfg['vocab'], dtype=torch.float64)
        score[PLUS], score[MINUS] = z, -z
        for t in set(out):
            score[t] = score[t] / penalty if score[t] > 0 else score[t] * penalty
        out.append(int(score.argmax()))
        ids.append(out[-1])
    return out


@pytest.mark.parametrize('penalty', [1.0, 1.5])
def test_equal_scores_in_several_parts(penalty):
    from callireader_amd.modeling_decoder import LinasunForCausalLM
    cfg = dict(LC.TINY, vocab=9000)
    w = LC.weights(cfg, 4)
    r = w['head'][0].clone()
    w['head'].zero_()
    for i in PLUS:
        w['head'][i] = r
    for i in MINUS:
        w['head'][i] = -r
    m = LinasunForCausalLM.from_state_dict(w, cfg, dtype=torch.float32, max_tokens=64, max_seqs=3)
    prompts = [LC.tokens(cfg, n, seed=n) for n in (3, 9, 20)]
    want = [expected(w, cfg, p, 12, penalty) for p in prompts]
    for _ in range(2):                                       # a second batch on the same cache object
        assert m.generate(prompts, max_new_tokens=12, repetition_penalty=penalty) == want
    assert m.generate([prompts[2]], max_new_tokens=12, repetition_penalty=penalty) == [want[2]]
    m.close()
    assert any(t > 4096 for t in sum(want, [])) or penalty == 1.0
