"""csrc/lm_upload.hpp by itself, with address and undefined-behaviour checks: what a described decoder's prompt call uploads, word for word, and whether the rows asked for are the
segments' last rows, for calls from a few rows to more than the array's first block (8190 rows: 128 KiB)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = r'''
#include <stdio.h>
#include "lm_upload.hpp"
static int in() { int v; if (scanf("%d", &v) != 1) v = 0; return v; }
int main() {
    std::vector<PromptSeg> segs(in());
    int M = 0, Mk = 0;
    for (size_t i = 0; i < segs.size(); i++) {
        const int S = in(), pos0 = in();
        segs[i] = {M, S, pos0, (int)(segs.size() - 1 - i), Mk};
        M += S; Mk += pos0 + S;
    }
    std::vector<int64_t> tokens(M);
    for (int i = 0; i < M; i++) tokens[i] = 7 * i;
    std::vector<int32_t> want(in());
    for (int32_t& w : want) w = in();
    std::vector<int> chunks(in());
    for (int& c : chunks) c = in();
    const int max_tokens = in(), ret = in();
    const PromptUpload u = prompt_upload(segs, M, tokens.data(), want.data(), (int)want.size(), chunks, max_tokens, ret);
    printf("%d %d %d %zu\n", (int)u.want_is_last, u.snaps, u.longest, u.words.size());
    printf("%zu %zu %zu %zu %zu %zu %zu %zu\n", u.row_seq, u.row_pos, u.seg, u.rseg, u.last, u.snap0, u.want, u.chunks);
    for (const PromptKeys& k : u.keys) printf("%d %d %d %d %zu %zu %zu %zu %zu %zu\n", k.ring, k.n_pieces, k.longest, k.n_pre, k.Mk, k.row_key, k.row_slot, k.pieces, k.pre_key, k.pre_slot);
    for (int32_t w : u.words) printf("%d\n", w);
}
'''


@pytest.fixture(scope='module')
def program(tmp_path_factory):
    if not shutil.which('g++'):
        pytest.skip('no host compiler')
    d = tmp_path_factory.mktemp('upload')
    (d / 'main.cpp').write_text(MAIN)
    subprocess.run(['g++', '-std=c++17', '-g', '-O1', '-fsanitize=address,undefined', '-fno-sanitize-recover=all', '-I' + os.path.join(ROOT, 'callireader_amd', 'csrc'), str(d / 'main.cpp'),
                    '-o', str(d / 'upload')], check=True)

    def run(segs, want, chunks, max_tokens, ret):
        words = [len(segs), *(v for s in segs for v in s), len(want), *want, len(chunks), *chunks, max_tokens, ret]
        r = subprocess.run([str(d / 'upload')], input=' '.join(map(str, words)), capture_output=True, text=True, env=dict(os.environ, ASAN_OPTIONS='verify_asan_link_order=0'))
        assert r.returncode == 0, r.stderr[-2000:]
        return [[int(v) for v in line.split()] for line in r.stdout.splitlines()]
    return run


def expected(segs, want, chunks, max_tokens, ret):
    """(words by name, key plans by name), from the definition"""
    row0 = [sum(s for s, _ in segs[:i]) for i in range(len(segs))]
    seq = [len(segs) - 1 - i for i in range(len(segs))]
    M = sum(s for s, _ in segs)
    rows = [(i, t) for i, (s, _) in enumerate(segs) for t in range(s)]
    parts = dict(tokens=[v for i in range(M) for v in (7 * i, 0)], row_seq=[seq[i] for i, _ in rows], row_pos=[segs[i][1] + t for i, t in rows],
                 seg=[v for i, (s, p) in enumerate(segs) for v in (row0[i], s, p, sum(a + b for a, b in segs[:i]))], rseg=[v for i, (s, p) in enumerate(segs) for v in (row0[i], s, p, seq[i])],
                 last=[row0[i] + s - 1 for i, (s, _) in enumerate(segs)], snap0=[sum(-(-s // ret) for s, _ in segs[:i]) for i in range(len(segs))], want=list(want),
                 chunks=[v for i, (s, _) in enumerate(segs) for t in range(0, s, ret) for v in (row0[i] + t, min(ret, s - t))])
    plans = []
    for c in chunks:
        ring, base, k = min(c, max_tokens), 0, dict(row_key=[], row_slot=[], pieces=[], pre_key=[], pre_slot=[])
        for i, (s, p) in enumerate(segs):
            pre = p % c
            k['pre_key'] += range(base, base + pre)
            k['pre_slot'] += [seq[i] * ring + j for j in range(pre)]
            k['row_key'] += range(base + pre, base + pre + s)
            k['row_slot'] += [seq[i] * ring + q % c if q // c == (p + s - 1) // c else -1 for q in range(p, p + s)]
            for first in sorted({p} | {q for q in range(p, p + s) if q % c == 0}):
                n = min(p + s, first - first % c + c) - first
                k['pieces'] += [row0[i] + first - p, n, first % c, base + pre + first - p - first % c]
            base += pre + s
        plans.append((ring, base, k))
    return parts, plans


@pytest.mark.parametrize('segs', [[(1, 0)], [(100, 0)] * 4, [(3, 5), (1, 36), (90, 37)], [(2048, 0)] * 4, [(2730, 3), (1, 0), (5500, 74)]])
@pytest.mark.parametrize('chunks', [[2**31 - 1], [37, 2**31 - 1], []])
def test_words_and_last_rows(program, segs, chunks):
    M, last = sum(s for s, _ in segs), [sum(s for s, _ in segs[:i + 1]) - 1 for i in range(len(segs))]
    for want in (last, last[::-1], [max(r - 1, 0) for r in last], [], last + [0], list(range(min(M, 70)))):
        head, at, *rest = program(segs, want, chunks, 6000, 256)
        parts, plans = expected(segs, want, chunks, 6000, 256)
        assert head[0] == int(want == last) and head[1] == sum(-(-s // 256) for s, _ in segs) and head[2] == max(s for s, _ in segs)
        words = [r[0] for r in rest[len(chunks):]]
        flat = [v for name in ('tokens', 'row_seq', 'row_pos', 'seg', 'rseg', 'last', 'snap0', 'want', 'chunks') for v in parts[name]]
        for (ring, mk, k), line in zip(plans, rest):
            assert line[0] == ring and line[1] == len(k['pieces']) // 4 and line[2] == max(k['pieces'][1::4]) and line[3] == len(k['pre_key']) and line[4] == mk
            for name, place in zip(('row_key', 'row_slot', 'pieces', 'pre_key', 'pre_slot'), line[5:]):
                assert place == len(flat), name
                flat += k[name]
        assert words == flat and head[3] == len(flat)
        for name, place in zip(('row_seq', 'row_pos', 'seg', 'rseg', 'last', 'snap0', 'want', 'chunks'), at):
            assert words[place:place + len(parts[name])] == parts[name], name
