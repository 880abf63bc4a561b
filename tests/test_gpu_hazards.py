"""Systematic screen of the hand-placed LDS-DMA waits: a diagnostic build (-DCR_POISON) overwrites every LDS piece
with bf16 NaNs right before it is refilled -- the point from which, by the schedules' own WAR / RAW rules, nobody may read it until the new bytes
have landed.  A read that breaks either rule then returns NaNs, so the integer-exact / bit-exact kernel tests FAIL on such a build instead of passing
whenever the old bytes happen to be still (or the new ones already) there.  This test builds that variant of gemm256.hip
(both schedules, both tile heights, grouped), gemm_mid.hip, lm_gemm_tiles.hip, lm_gemm_rows.hip, lm_ahead.hip, lm_mix.hip, moe.hip (the router) and attention_vit.hip and runs the kernel tests on it in a child process.  What the screen cannot see: a staged piece that always lands
in time whether or not the schedule waits for it; those waits are correct by construction, not by test."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_kernel_tests_pass_on_the_poisoned_build():
    if not (shutil.which('hipcc') or os.path.exists('/opt/rocm/bin/hipcc')):
        pytest.skip('hipcc is not on this box: the diagnostic variant cannot be built')
    env = dict(os.environ, PATH=os.environ.get('PATH', '') + ':/opt/rocm/bin')
    b = subprocess.run([sys.executable, os.path.join(ROOT, 'scripts', 'build_variant.py'), 'poison', 'gemm256.hip,gemm_mid.hip,lm_gemm_tiles.hip,lm_gemm_rows.hip,lm_ahead.hip,lm_mix.hip,moe.hip,attention_vit.hip', '-DCR_POISON=1'],
                       capture_output=True, text=True, env=env, cwd=ROOT, timeout=900)
    assert b.returncode == 0, b.stdout[-2000:] + b.stderr[-2000:]
    lib = os.path.join(ROOT, 'ab', 'libpoison.so')
    assert os.path.exists(lib)
    sel = 'gemm256 or gemm_epilogues or gelu or both_schedules or back_to_back or attention_vit or patch_rows or swiglu or argmax or tail_rows'
    files = {'test_gpu_gemm192.py': 'same_bits', 'test_gpu_gemm_mid.py': 'every_shape or patches', 'test_gpu_few_rows.py': 'fp32_decode_rows or prompt_rows or among_64', 'test_gpu_grouped.py': 'many_tiles',
             'test_gpu_decode_mixer.py': 'one_launch or residual_updates', 'test_gpu_routing.py': 'many_tokens', 'test_gpu_gemm_steps.py': 'depths_of_buffers or largest_shapes',
             'test_gpu_fp32_tiles.py': 'prompt_tiles', 'test_gpu_lm_gemm.py': 'named_by_a_list'}
    sel += ' or ' + ' or '.join(files.values())
    r = subprocess.run([sys.executable, '-m', 'pytest', *(os.path.join(ROOT, 'tests', f) for f in ('test_gpu_ops.py', *files)), '-x', '-q', '-m', 'gpu', '-k', sel],
                       capture_output=True, text=True, env=dict(env, CR_HIP_LIB=lib), cwd=ROOT, timeout=900)
    tail = r.stdout[-1500:]
    assert r.returncode == 0, tail
    assert ' passed' in tail and 'failed' not in tail, tail
