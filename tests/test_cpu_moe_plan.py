"""Which problems the persistent gathered GEMM of the mixture of experts takes, asked on the host from the header that its
launcher and its kernel share: byte offsets stay in 32 bits, lists of tiles in LDS, and large problems are taken.  No GPU."""
import os
import random
import shutil
import subprocess

import pytest

from conftest import ROOT

LDS_OF_CU = 160 * 1024


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
    # 4 GB of tokens, of 64 rows of k, of 256 rows of columns
    ((65536, 32704, 1024, 8, 0, 256), 1), ((65536, 32768, 1024, 8, 0, 256), 0), ((255, (1 << 23) - 64, 512, 2, 1, 256), 1), ((200, 1 << 23, 512, 2, 1, 256), 0),
    ((200, (1 << 23) + 64, 512, 2, 1, 256), 0), ((200, (1 << 23) + 64, 512, 2, 0, 256), 1)])
def test_which_problems_the_persistent_tiles_take(case, fits, plan):
    assert plan([case])[0][0] == fits


def test_offsets_and_lists_of_all_that_is_taken(plan):
    rng = random.Random(3)
    log = lambda low, high: int(low * (high / low) ** rng.random())
    cases = [(log(1, 4000000), 64 * log(4, 300000), 8 * log(1, 5000000), log(1, 2048), rng.randint(0, 1), rng.choice([32, 64, 256, 304])) for _ in range(60000)]
    taken = [(case, p) for case, p in zip(cases, plan(cases)) if p[0]]
    assert len(taken) > 1000
    for case, (_, _, reach, tokens, weights) in taken:
        assert reach <= LDS_OF_CU and tokens <= 1 << 32 and weights <= 1 << 32, case
