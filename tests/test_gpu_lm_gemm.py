"""launch_lm_gemm's float32 prompt products with operands that no model hands over: rows gathered by a list without experts, and rows so far apart that eight of them reach past 2 GiB (32-bit offsets above 2^31)
and past 4 GiB (64 bits a lane), on both sides of the line.  A row's sum has one order whatever kernel takes it: the bits of the same rows side by side, and those within 5 x 2^-24 K of sums in 64 bits (K
additions of unit products, each rounding a sum of some sqrt(K) by 2^-24 of it and sqrt(K) of those at random: 2^-24 K).  Called through a small library that hands the product's arguments over by name."""
import ctypes
import os
import shutil
import subprocess

import pytest
import torch

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'callireader_amd', 'csrc')
HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'

CALL = r'''
#include "lm.hpp"
extern "C" int call_lm_gemm(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, int M, int N, int K, const int32_t* perm, int gather_div, int scatter, void* stream) {
    LmGemmParams p{};
    p.A = A; p.lda = lda; p.W = W; p.ldw = ldw; p.C = C; p.ldc = ldc; p.M = M; p.N = N; p.K = K; p.perm = perm; p.gather_div = gather_div; p.scatter = scatter;
    return launch_lm_gemm(true, LM_STORE, p, (hipStream_t)stream);
}
'''


@pytest.fixture(scope='module')
def product(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip('hipcc is not on this box')
    import callireader_amd._binding as B
    d = tmp_path_factory.mktemp('lm_gemm')
    (d / 'call.cpp').write_text(CALL)
    lib = B.lib._name
    subprocess.run([HIPCC, '-x', 'hip', '--offload-arch=gfx950', '--offload-host-only', '-std=c++17', '-O1', '-fPIC', '-shared', '-I', CSRC, str(d / 'call.cpp'), '-x', 'none', lib, '-o', str(d / 'call.so'),
                    f'-Wl,-rpath,{os.path.dirname(os.path.abspath(lib))}'], check=True, capture_output=True, timeout=300)
    f = ctypes.CDLL(str(d / 'call.so')).call_lm_gemm
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_void_p, ctypes.c_int64] * 3 + [ctypes.c_int] * 3 + [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]

    def call(A, W, perm=None, div=0, scatter=0, rows=None):
        M = rows or A.shape[0]
        C = torch.full((M, W.shape[0]), float('nan'), device='cuda')
        assert f(A.data_ptr(), A.stride(0), W.data_ptr(), W.stride(0), C.data_ptr(), C.stride(0), M, W.shape[0], A.shape[1], perm.data_ptr() if perm is not None else None, div, scatter,
                 torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        return C
    return call


def operands(M, N, K):
    g = torch.Generator().manual_seed(M + 7 * N)
    return [torch.randn(*s, generator=g).cuda() for s in ((M, K), (N, K))]


@pytest.mark.parametrize('scatter', [0, 1])
@pytest.mark.parametrize('div', [0, 1, 3])
@pytest.mark.parametrize('M,N,K', [(5, 40, 64), (70, 200, 192), (201, 1040, 576)])
def test_rows_named_by_a_list_without_experts(product, M, N, K, div, scatter):
    A, W = operands(M, N, K)                             # (M rows, also where the list names a third of them)
    perm = torch.randperm(M, generator=torch.Generator().manual_seed(3))
    rows = A[(perm // div).cuda()] if div else A
    want = product(rows.contiguous(), W)
    torch.testing.assert_close(want, (rows.double() @ W.double().T).float(), rtol=1e-6, atol=5 * 2 ** -24 * K)
    got = product(A, W, perm.int().cuda(), div, scatter)
    assert torch.equal(got[perm.cuda()] if scatter else got, want)


@pytest.mark.parametrize('far', ['activations', 'weights'])
@pytest.mark.parametrize('ld', [2 ** 27 - 4, 2 ** 27])   # the last that is reached by 32 bits, and the first that is not
def test_rows_far_apart(product, far, ld):
    M, N, K = (20, 70, 192) if far == 'activations' else (70, 20, 192)
    A, W = operands(M, N, K)
    want = product(A, W)
    near = A if far == 'activations' else W
    wide = torch.empty((len(near) - 1) * ld + K, device='cuda').as_strided(near.shape, (ld, 1))
    wide.copy_(near)
    assert torch.equal(product(*((wide, W) if far == 'activations' else (A, wide))), want)
