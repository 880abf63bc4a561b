"""Which kernel and which tile shape a tiled product goes to, by the laws of csrc/gemm_mid.hip, gemm256.hip and gemm.hip for 256 compute units: sizes at which the ways differ by 5 to 27 % (us, measured, beside
each).  The library's own functions, asked by a small program."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'callireader_amd', 'csrc')
HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason='hipcc not found')

ASK = r'''
#include <cstdio>
#include <cstdlib>
#include "common.hpp"
double gemm_mid_cost(int epi, const GemmParams& p, int* tile, int* row_tiles);
int gemm_tiled_rows(int epi, const GemmParams& p);

int main(int, char** v) {
    GemmParams p{};
    p.M = atoi(v[1]); p.N = atoi(v[2]); p.K = atoi(v[3]);
    p.lda = p.ldw = p.K; p.ldc = p.N;
    int tile = 0, row_tiles = 0;
    gemm_mid_cost(EPI_STORE, p, &tile, &row_tiles);
    printf("%d %d\n", gemm_tiled_rows(EPI_STORE, p), tile);
}
'''


@pytest.fixture(scope='module')
def ask(tmp_path_factory):
    import callireader_amd.build as build
    d = tmp_path_factory.mktemp('choice')
    (d / 'ask.cpp').write_text(ASK)
    subprocess.run([HIPCC, '-x', 'hip', '--offload-arch=gfx950', '--offload-host-only', '-std=c++17', '-O1', '-I', CSRC, str(d / 'ask.cpp'), '-x', 'none', build.build(), '-o', str(d / 'ask'),
                    f'-Wl,-rpath,{CSRC}'], check=True, capture_output=True, timeout=600)
    env = {k: x for k, x in os.environ.items() if k != 'CR_CUS'}
    return lambda *n: tuple(map(int, subprocess.run([str(d / 'ask'), *map(str, n)], capture_output=True, text=True, timeout=60, check=True, env=env).stdout.split()))


# tile: one more than a shape's number in gemm_mid.hip
@pytest.mark.parametrize('M,N,K,tile', [
    (3075, 9216, 448, 12),        # 128 x 256 39.9, 160 x 128 48.3
    (6124, 9216, 2240, 12),       # 228, 260
    (13325, 9216, 3008, 12),      # 678, 741
    (1500, 9216, 2240, 12),       # 67.5, 77.1
    (356, 12800, 14336, 11),      # 96 x 256 177, 96 x 128 215
    (1923, 2560, 14336, 11),      # 162, 186
    (2050, 2048, 2048, 13),       # 160 x 128 24.2, 128 x 256 29.4
    (1025, 4096, 1024, 13),       # 14.4, 18.1
    (4100, 2048, 2240, 13),       # 47.3, 56.5
])
def test_tile_shape(ask, M, N, K, tile):
    assert ask(M, N, K)[1] == tile


@pytest.mark.parametrize('M,N,K,rows', [
    (3162, 4096, 4096, 3162),     # whole 80.3, its last 90 rows apart 85.6
    (3112, 4096, 14336, 3112),    # 265, 279
    (6145, 2048, 2048, 6145),     # 43.1, 45.6
    (6234, 4096, 1024, 6234),     # 47.9, 50.9
    (696, 28672, 8192, 696),      # 278, 325
    (4111, 8192, 256, 4111),      # 25.2, 34.0
    (4100, 4096, 4096, 4096),     # 126, 99.7
    (6145, 4096, 4096, 6144),     # 157, 149
    (6145, 6144, 4096, 6144),     # 241, 219
    (98400, 4096, 1024, 98304),   # 640, 627
    (41132, 28672, 4096, 40960),  # 6539, 6354
    (632, 28672, 4096, 512),      # 143, 135
    (12373, 2048, 4096, 12288),   # 157, 152
    (4180, 8192, 1024, 4180),     # 63.8, 69.5
    (800, 16384, 14336, 800),     # 315, 361
    (11275, 4096, 1024, 11275), (1025, 4096, 1024, 0), (77, 4096, 4096, 0)])
def test_rows_apart(ask, M, N, K, rows):
    assert ask(M, N, K)[0] == rows
