"""Which bytes the workgroups of csrc/l2_ahead.hpp fetch: its host arithmetic, compiled for this machine and walked as the kernel walks it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason='hipcc not found')

WALK = r'''
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "l2_ahead.hpp"

// units of a weight of N rows and K columns, `tiles` tiles of 16 rows a workgroup of its reader; own workgroups ahead of the fetching ones, `width` of them side by side
int main(int n, char** v) {
    if (n == 3) return printf("%ld\n", (long)l2_ahead_beside_latent(atol(v[1]), atol(v[2]))), 0;
    if (n == 4) return printf("%d\n", (int)l2_ahead_beside_attention(atol(v[1]) * atol(v[2]), atoi(v[3]))), 0;
    if (n == 5) {
        const L2AheadRoom r = l2_ahead_beside_mixer(atoi(v[1]), atol(v[2]), atoi(v[3]), atoi(v[4]));
        return printf("%ld %ld %d\n", (long)(r.most >> 20), (long)(r.least >> 20), r.products), 0;
    }
    if (n == 6) {
        const L2AheadRoom r = l2_ahead_beside_mixer(true, atol(v[1]), atoi(v[2]), 256, atoi(v[3]), atol(v[4]) * atol(v[5]));
        return printf("%ld %ld %d\n", (long)(r.most >> 20), (long)(r.least >> 20), r.products), 0;
    }
    const long N = atol(v[1]), K = atol(v[2]), es = atol(v[3]), tiles = atol(v[4]), own = atol(v[5]), width = atol(v[6]);
    static char base;
    const L2Ahead a = l2_ahead_of(&base, N * K * es, (int)(N / (16 * tiles)));
    if (!a.at) return puts("nothing"), 0;
    const long bytes = N * K * es, piece = a.unit_bytes / a.pieces, groups = (own + l2_ahead_extra((int)own) + width - 1) / width * width;
    std::vector<char> seen(bytes / 16);
    long most = 0;
    for (long linear = own; linear < groups; linear++) {
        const int nth = l2_ahead_nth((int)linear, (int)own);
        if (nth < 0 || nth >= L2_AHEAD_GROUPS) continue;
        if ((nth & 7) != (linear & 7)) return puts("remainder"), 1;
        long took = 0;
        for (int j = nth >> 3; j < (a.units + 7) / 8 * a.pieces; j += L2_AHEAD_GROUPS / 8) {
            const long off = l2_ahead_piece(a, (int)linear, j);
            if (off < 0) break;
            if (off % 16 || piece % 16 || off + piece > bytes) return printf("piece %ld at %ld\n", piece, off), 1;
            if (off / a.unit_bytes % 8 != (linear & 7)) return puts("another XCD"), 1;
            for (long i = off / 16; i < (off + piece) / 16; i++) seen[i]++;
            took += piece;
        }
        most = most > took ? most : took;
    }
    for (long i = 0; i < bytes / 16; i++)
        if (seen[i] != 1) return printf("vector %ld read %d times\n", i, seen[i]), 1;
    printf("pieces %d most %ld\n", a.pieces, most);
}
'''


@pytest.fixture(scope='module')
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp('l2_ahead')
    (d / 'walk.cpp').write_text(WALK)
    subprocess.run([HIPCC, '-x', 'hip', '--offload-arch=gfx950', '--offload-host-only', '-std=c++17', '-O1', '-I', os.path.join(ROOT, 'callireader_amd', 'csrc'), str(d / 'walk.cpp'), '-o',
                    str(d / 'walk')], check=True, capture_output=True, timeout=300)
    return lambda *n: subprocess.run([str(d / 'walk'), *map(str, n)], capture_output=True, text=True, timeout=60)


# widths whose tiles eight pieces, or any power of two of them, do not divide evenly among the fetching workgroups; tiles a workgroup as few-row products have them; own workgroups that eight and the
# grid's width do not divide
@pytest.mark.parametrize('own,width', [(8, 8), (10, 10), (51, 17), (480, 12)])
@pytest.mark.parametrize('N,K,es,tiles', [(640, 640, 2, 1), (640, 640, 4, 1), (768, 1152, 4, 1), (1152, 768, 2, 3), (1280, 2560, 2, 2), (2560, 640, 4, 1), (2560, 5120, 2, 4), (4096, 4096, 2, 1), (4096, 4096, 2, 4),
                                          (4096, 1024, 4, 1), (128, 128, 2, 1), (16, 64, 2, 1), (208, 64, 2, 1)])
def test_every_byte_once_in_16_byte_vectors_on_its_readers_xcd(walk, N, K, es, tiles, own, width):
    r = walk(N, K, es, tiles, own, width)
    assert r.returncode == 0 and r.stdout.startswith('pieces'), r.stdout + r.stderr
    pieces, most = int(r.stdout.split()[1]), int(r.stdout.split()[3])
    assert pieces in (1, 2, 4, 8)
    units = N // (16 * tiles)
    if -(-units // 8) * 8 * pieces <= 256:                              # a piece a workgroup at most
        assert most == N * K * es // units // pieces


def test_what_cannot_be_cut_is_left_alone(walk):
    assert walk(100, 64, 2, 1, 8, 8).stdout == 'nothing\n'             # 6 units, which do not divide 12 800 bytes
    assert walk(8, 64, 2, 1, 8, 8).stdout == 'nothing\n'               # none


def test_beside_attention_until_its_keys_need_the_caches(walk):
    takes = lambda rows, keys: walk(rows, 8 * -(-keys // 256), 256).stdout == '1\n'      # noqa: E731
    assert takes(1, 77) and takes(13, 3164) and takes(64, 2000) and takes(32, 4500)
    assert not takes(64, 3164) and not takes(64, 3900)


def test_beside_latent_attention_as_much_as_the_caches_hold(walk):
    room = lambda own: int(walk(own, 256).stdout)                      # noqa: E731
    assert 4096 * 4096 * 2 <= room(1) == room(128) < 5120 * 8192 * 2   # 64 heads of 128 on 5120 columns: more than all L2 caches together
    assert 2048 * 2048 * 2 <= room(129) == room(512) < 3072 * 3072 * 2


def test_beside_a_mixer_less_where_the_chip_is_full(walk):
    room = lambda *n: tuple(map(int, walk(*n, 256).stdout.split()))    # noqa: E731  (float32, own workgroups, key splits)
    assert room(0, 10, 1) == room(0, 256, 4) == (34, 0, 5)
    assert room(0, 257, 1) == room(0, 320, 2) == (26, 8, 5) and room(0, 321, 2) == (0, 0, 0)
    assert room(1, 128, 1) == (34, 0, 5) and room(1, 129, 1) == room(1, 192, 1) == (16, 0, 1) and room(1, 193, 1) == (0, 0, 0)


def test_beside_a_float32_mixer_until_its_keys_need_the_caches(walk):
    # rows of 2048 wide, 16 heads of 128 and 8 of retention; heads of 64, 768 wide
    wide = lambda rows, keys: walk(24 * rows, -(-keys // 256), 128, 16 * 2 * 128 * 4, rows * keys).stdout      # noqa: E731
    assert wide(1, 40) == wide(1, 1200) == wide(4, 400) == wide(5, 300) == '34 0 5\n'
    assert wide(1, 2000) == wide(4, 520) == wide(5, 400) == '0 0 0\n'
    assert walk(128, 8, 64, 12 * 2 * 64 * 4, 8 * 2000).stdout == '34 0 5\n'
