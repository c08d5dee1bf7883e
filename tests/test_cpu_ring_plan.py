"""The division of the LDS-ring kernel's tiles, walked on the host from the header that its launcher and its workgroups
share: the list of a workgroup's tiles lies inside the LDS that the launch asks for on every XCD - their lists of tiles
differ in length - and every tile belongs to exactly one workgroup.  No GPU."""
import os
import random
import re
import shutil
import subprocess
from typing import NamedTuple

import pytest

from conftest import ROOT
from helpers import RESULTS_K_N, RESULTS_THROUGH
from sparta_amd import _lib

LIST_MAX, LDS_OF_CU = 128, 160 * 1024
# (16-bit 32 x 64 blocks of 768 -> 3072, 128-row tiles; fp32 32 x 32; batched products) sizes at which the XCDs lie on the
# two sides of the longest list: elem_bytes, TM, BN, swap, M, K, N, batch
STRADDLING = [(2, 128, 32, 1, 131073, 768, 3072, 1), (2, 128, 32, 1, 131968, 768, 3072, 1), (4, 128, 32, 1, 65537, 1024, 4096, 1),
              (4, 128, 32, 1, 87936, 768, 3072, 1), (2, 128, 32, 1, 6208, 768, 4096, 16), (4, 128, 32, 1, 5504, 3072, 768, 48),
              # what the GPU tests run
              (2, 64, 16, 1, 109100, 64, 1536, 1), (2, 128, 16, 1, 131200, 64, 1536, 1), (2, 64, 16, 1, 4160, 64, 240, 128)]


# (element bytes, width of a tile, groups of wavefronts) that launches of 64-row tiles make
GROUPS = {(2, w, g) for w in (16, 32, 64) for g in (1, 2, 3)} | {(4, 16, g) for g in (1, 2, 3)} | {(4, 32, 1), (4, 64, 1)}


class Walk(NamedTuple):
    slots: int
    smem: int
    fewest: int    # tiles of a workgroup, over the XCDs
    most: int
    reach: int     # end of the list
    covered: int
    side_by_side: int
    counted_on: int
    sub: int             # log2 of the parts of a block-column, 64-row tiles
    parts_covered: int
    alone: int           # each tile has a workgroup to itself
    groups: int
    groups_smem: int
    groups_per_cu: int
    through: int         # results with an activation go through to the last-level cache


@pytest.fixture(scope='module')
def walk(tmp_path_factory):
    compiler = shutil.which('g++') or shutil.which('c++')
    if compiler is None:
        pytest.skip('no host compiler')
    exe = str(tmp_path_factory.mktemp('ring') / 'ring_plan_walk')
    subprocess.run([compiler, '-O2', '-std=c++17', '-Wall', '-Werror', '-I', os.path.join(ROOT, 'sparta_amd', 'csrc'),
                    os.path.join(ROOT, 'tests', 'ring_plan_walk.cpp'), '-o', exe], check=True)

    def run(cases, cover=False):
        text = ''.join(' '.join(map(str, case)) + f' {int(cover)}\n' for case in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
        assert len(out) == len(cases)
        return [Walk(*map(int, line.split())) for line in out]
    return run


def check(cases, walks):
    for case, w in zip(cases, walks):
        assert w.reach <= w.smem <= LDS_OF_CU, (case, w)
        assert w.slots in (0, w.most) and w.slots <= LIST_MAX, (case, w)
        assert w.fewest >= 1 and w.most - w.fewest <= max(1, w.most // 2), (case, w)


def test_lists_of_the_xcds_on_the_two_sides_of_the_longest(walk):
    walks = walk(STRADDLING)
    for case, w in zip(STRADDLING, walks):
        assert w.fewest <= LIST_MAX < w.most and w.slots == 0, (case, w)
    check(STRADDLING, walks)


def test_list_fits_the_lds_of_every_launch(walk):
    rng = random.Random(5)
    cases = []
    for _ in range(60000):
        es, TM, BN, swap = rng.choice([2, 4]), rng.choice([64, 128]), rng.choice([16, 32, 64]), rng.randint(0, 1)
        N = BN * int(2 ** rng.uniform(0, 9))
        batch = int(2 ** rng.uniform(0, 8))
        if rng.random() < 0.5:   # around the longest list: 128 tiles to each of the workgroups that fit
            mtiles = LIST_MAX * 8 * max(1, 32 * rng.randint(1, 5) // batch) // (N // BN) + rng.randint(-9, 9)
        else:
            mtiles = int(2 ** rng.uniform(0, 11))
        cases.append((es, TM, BN, swap, max(1, max(1, mtiles) * TM - rng.randint(0, TM - 1)), 64 * rng.randint(1, 64), N, batch))
    walks = walk(cases)
    check(cases, walks)
    # the sizes reach both sides of every line
    assert any(w.slots == LIST_MAX for w in walks) and any(w.most == LIST_MAX + 1 for w in walks)
    assert sum(w.fewest <= LIST_MAX < w.most for w in walks) > 20 and any(w.most == 1 for w in walks)


def test_every_tile_has_one_workgroup(walk):
    rng = random.Random(6)
    cases = [(es, TM, BN, 1, m, 64 * rng.randint(1, 64), BN * rng.randint(1, 40), rng.choice([1, 1, 2, 7, 40, 200]))
             for es in (2, 4) for TM in (64, 128) for BN in (16, 32, 64)
             for m in (1, 64, 65, 500, 1024, 3000, 4161, 8200, 20000, 70000)]
    for case, w in zip(cases, walk(cases, cover=True)):
        assert w.covered == 1, (case, w)


def test_parts_of_a_block_column_and_groups_of_wavefronts(walk):
    """A block-column is cut only into tiles that there are instances for and that have a workgroup each, each of them once; the
    workgroups with several groups of wavefronts that share a CU fit its LDS."""
    rng = random.Random(7)
    cases = [(es, 64, BN, swap, rng.randint(1, 64) if rng.random() < 0.3 else int(2 ** rng.uniform(6, 13)), 64 * rng.randint(1, 64),
              BN * int(2 ** rng.uniform(0, 7)), rng.choice([1, 1, 1, 2, 7, 40, 300]))
             for es in (2, 4) for BN in (16, 32, 64) for swap in (0, 1) for _ in range(400)]
    walks = walk(cases, cover=True)
    for case, w in zip(cases, walks):
        es, _, BN = case[:3]
        assert w.parts_covered == 1, (case, w)
        assert w.sub == 0 or (w.alone and BN >> w.sub >= (32 if es == 2 else 16)), (case, w)
        assert w.groups_smem <= LDS_OF_CU, (case, w)
        if w.groups > 1:
            piece = 1280   # LDS is given out in pieces
            assert w.groups <= 3 and w.groups_per_cu * (-(-w.groups_smem // piece) * piece) <= LDS_OF_CU, (case, w)
            # the sums that the other groups leave (16 bytes to a lane and 16 columns) fit the rings that carried the operands
            columns, stages = BN >> w.sub, 2 if es == 2 else 3
            assert (w.groups - 1) * 4 * (columns // 16) * 64 * 16 <= w.groups * stages * (64 + columns) * 128, (case, w)
    assert {(c[0], c[2], w.sub) for c, w in zip(cases, walks)} == {(2, 16, 0), (2, 32, 0), (2, 64, 0), (2, 64, 1), (4, 16, 0), (4, 32, 0),
                                                                   (4, 32, 1), (4, 64, 0), (4, 64, 1), (4, 64, 2)}
    assert {(c[0], c[2] >> w.sub, w.groups) for c, w in zip(cases, walks) if w.groups} == GROUPS


def test_the_library_has_the_groups_that_launches_make():
    """... and none that no launch reaches: a width and a number of groups are 24 kernels or more."""
    if shutil.which('nm') is None or not os.path.exists(_lib.LIB_PATH):
        pytest.skip('no nm, or nothing is built')
    names = subprocess.run(['nm', '-D', '--defined-only', _lib.LIB_PATH], capture_output=True, text=True, check=True).stdout
    kernels = re.findall(r'spmm_ring_kernelI(f|DF16_|NS_\w+?)Li(\d+)ELi(\d+)ELi(\d+)E((?:Lb[01]E)+)Li(\d)E', names)
    assert len(kernels) > 100
    assert {(4 if t == 'f' else 2, int(width), int(groups)) for t, _, width, _, _, groups in kernels} == GROUPS


def test_results_with_an_activation_that_are_written_through(walk):
    """Both sides of each line, and the sizes that the GPU test of the stores runs (their values are the same either way)."""
    sizes = [(8192, 768, 3072, 1), (5121, 768, 1536, 1), (5120, 768, 3072, 0), (8192, 768, 1504, 0), (16384, 1024, 1024, 0), (8192, 1024, 2048, 1)]
    for M, K, N, through in sizes:
        assert walk([(2, 64, 32, 1, M, K, N, 1)])[0].through == through, (M, K, N)
    for (TM, M), through in RESULTS_THROUGH.items():
        assert walk([(2, TM, 32, 1, M, *RESULTS_K_N, 1)])[0].through == through, (TM, M)
    assert set(RESULTS_THROUGH.values()) == {0, 1}


@pytest.mark.parametrize('TM', [64, 128])
@pytest.mark.parametrize('BN', [16, 32, 64])
@pytest.mark.parametrize('swap', [0, 1])
def test_rounds_of_a_tile_height_are_those_of_its_launch(TM, BN, swap, walk):
    """The choice between 64-row and 128-row tiles of 16-bit types counts rounds of the workgroups that fit the chip: the
    rounds that the launch takes, where the panels deal out evenly over the XCDs."""
    cases = [(2, TM, BN, swap, TM * mtiles, 768, BN * cols, 1) for mtiles in (64, 128, 192, 320) for cols in range(1, 200, 7)]
    for case, w in zip(cases, walk(cases)):
        tiles = case[4] // TM * (case[6] // BN)
        assert w.most == -(-tiles // w.counted_on), (case, w)
        assert w.side_by_side <= w.counted_on
