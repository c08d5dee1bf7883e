"""Which problems the persistent gathered GEMM of the mixture of experts takes, asked on the host from the header that its
launcher and its kernel share: lists of tiles stay in LDS, and large problems are taken.  No GPU."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope='module')
def plan(tmp_path_factory):
    compiler = shutil.which('g++') or shutil.which('c++')
    if compiler is None:
        pytest.skip('no host compiler')
    exe = str(tmp_path_factory.mktemp('moe') / 'moe_plan')
    subprocess.run([compiler, '-O2', '-std=c++17', '-Wall', '-Werror', '-I', os.path.join(ROOT, 'sparta_amd', 'csrc'),
                    os.path.join(ROOT, 'tests', 'moe_plan.cpp'), '-o', exe], check=True)

    def run(cases):
        text = ''.join(' '.join(map(str, case)) + '\n' for case in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
        return [tuple(map(int, line.split())) for line in out]
    return run


@pytest.mark.parametrize('case,fits', [
    # tokens, K, N, experts, [E, out, in], CUs: many tiles over all workgroups (16640 are 66 rounds of 256), and over few
    ((131072, 512, 8192, 8, 0, 256), 1), ((131072, 512, 8192, 8, 1, 256), 1), ((131072, 512, 8192, 8, 0, 8), 0), ((1000000, 1024, 65536, 64, 0, 256), 0),
    # k of 64 and more that four stages fit
    ((16384, 256, 4096, 8, 0, 256), 1), ((16384, 192, 4096, 8, 0, 256), 0),
    # 4 GB of tokens
    ((65536, 32704, 1024, 8, 0, 256), 1), ((65536, 32768, 1024, 8, 0, 256), 0)])
def test_which_problems_the_persistent_tiles_take(case, fits, plan):
    assert plan([case])[0][0] == fits
