"""The LDS-ring kernel (tile configs 11 and 12) against the numpy oracle: all four operand layouts in
both output orientations, rows that end inside a tile, block-columns without, with one and with an odd
number of blocks, several tiles per workgroup, and more block-columns than its table holds."""
import pytest
import torch

from test_gpu_matmul import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('tile_cfg', [11, 12])
@pytest.mark.parametrize('mode,tA,tB', [('dsd', False, True), ('dsd', False, False), ('dsd', True, True), ('dsd', True, False),
                                        ('sdd', False, True), ('sdd', False, False), ('sdd', True, True), ('sdd', True, False)])
@pytest.mark.parametrize('dtype,blocks', [(torch.float32, (32, 32, 32)), (torch.float32, (16, 16, 16)), (torch.float16, (32, 32, 64)),
                                          (torch.bfloat16, (64, 64, 32)), (torch.float32, (64, 64, 16)), (torch.bfloat16, (16, 64, 64)),
                                          (torch.float16, (32, 32, 16))])
def test_ring_layouts(tile_cfg, mode, tA, tB, dtype, blocks, gpu):
    for compressed, rows, sparsity in ((True, 200, 0.7), (False, 328, 0.9)):
        run_case(gpu, mode, tA, tB, True, compressed, dtype, blocks, batch=2, M=rows if mode == 'dsd' else 128, K=320,
                 N=128 if mode == 'dsd' else rows, gran=(16, 16), sparsity=sparsity, seed=51, tile_cfg=tile_cfg)


@pytest.mark.parametrize('tile_cfg', [11, 12])
@pytest.mark.parametrize('dtype,blocks', [(torch.float32, (32, 32, 32)), (torch.float16, (32, 32, 32)), (torch.bfloat16, (32, 64, 64))])
def test_ring_rows_and_rounds(tile_cfg, dtype, blocks, gpu):
    """One row; a whole tile and one row more; many tiles per workgroup (panels that do and do not deal
    out evenly over the XCDs), with and without the fused activation."""
    for M, N in ((1, 192), (64, 192), (65, 192), (129, 192), (2100, 2048), (1500, 1088)):
        run_case(gpu, 'dsd', False, True, True, True, dtype, blocks, batch=1, M=M, K=192, N=N, gran=(blocks[2], blocks[1]),
                 sparsity=0.8, seed=M, tile_cfg=tile_cfg, activation='relu' if M % 2 else None)


def test_ring_more_block_columns_than_the_table(gpu):
    run_case(gpu, 'dsd', False, True, False, True, torch.float16, (32, 32, 16), batch=1, M=520, K=96, N=16 * 1100,
             gran=(16, 32), sparsity=0.6, seed=61, tile_cfg=11)
