"""gemm_mid.hip's shallow forms, taken where there are more workgroups than compute units, leave a CU room for a second workgroup: eight waves of 128 registers at most each (their LDS is asserted in the source); and no
shape's fragments spill.  Read from the notes of the library's own object file."""
import os
import re
import shutil
import subprocess

import pytest

LLVM = '/opt/rocm/llvm/bin'
pytestmark = pytest.mark.skipif(not os.path.exists(f'{LLVM}/llvm-readelf') or not (shutil.which('hipcc') or os.path.exists('/opt/rocm/bin/hipcc')), reason='ROCm tools not found')


@pytest.fixture(scope='module')
def kernels(tmp_path_factory):
    import callireader_amd.build as build
    build.build()
    obj = os.path.join(build.CSRC, 'build', 'gemm_mid.o')
    if not os.path.exists(obj):
        pytest.skip('the library was not built here')
    d = tmp_path_factory.mktemp('co')
    run = lambda *a: subprocess.run([f'{LLVM}/{a[0]}', *map(str, a[1:])], check=True, capture_output=True, text=True, timeout=60).stdout      # noqa: E731
    run('llvm-objcopy', '--dump-section', f'.hip_fatbin={d}/fat', obj, d / 'rest.o')
    run('clang-offload-bundler', '--unbundle', '--type=o', '--targets=hipv4-amdgcn-amd-amdhsa--gfx950', f'--input={d}/fat', f'--output={d}/code')
    found = {}
    for name, vgpr, spill in re.findall(r'\.name:\s+(\S+).*?\.vgpr_count:\s+(\d+).*?\.vgpr_spill_count: (\d+)', run('llvm-readelf', '--notes', d / 'code'), re.S):
        m = re.search(r'gemm_mid_kernelILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELb0E', name)
        if m:
            found[tuple(map(int, m.groups()))] = (int(vgpr), int(spill))
    return found


@pytest.mark.parametrize('shape', [(2, 4, 2, 1, 4), (2, 4, 3, 1, 3), (2, 4, 4, 1, 3), (2, 4, 2, 2, 3)])       # waves in rows and columns, fragments a wave, K-tiles in LDS
def test_registers_of_the_shallow_forms(kernels, shape):
    vgpr, spill = kernels[shape]
    assert vgpr <= 128 and spill == 0


def test_no_shape_spills(kernels):
    assert len(kernels) >= 13 and not {k: v for k, v in kernels.items() if v[1]}
