"""The LDS-ring kernel (tile configs 11 and 12) against the numpy oracle: all four operand layouts in
both output orientations, rows that end inside a tile, block-columns without, with one and with an odd
number of blocks, several tiles per workgroup, and more block-columns than its table holds."""
import numpy as np
import pytest
import torch

from helpers import RESULTS_K_N, RESULTS_THROUGH, assert_close, chained_sum_error, launched_kernels, template_numbers
from oracle import ops
from sparta_amd.specializer.kernels import SparTASparseMatMulKernel
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


@pytest.mark.parametrize('mode,compressed', [('dsd', True), ('dsd', False), ('sdd', True), ('sdd', False)])
@pytest.mark.parametrize('dtype,wide,rows,columns,tile', [
    # fp32: quarters, halves and whole block-columns as the workgroups allow (four to a CU with 16-wide tiles); one row
    (torch.float32, 64, 1000, 16, 16), (torch.float32, 64, 1000, 17, 32), (torch.float32, 64, 1024, 65, 64),
    (torch.float32, 32, 1000, 32, 16), (torch.float32, 32, 1000, 33, 32), (torch.float32, 64, 8, 3, 16), (torch.float32, 16, 200, 5, 16),
    # 16-bit types: halves of 64-wide block-columns up to 96 tiles
    (torch.float16, 64, 200, 24, 32), (torch.bfloat16, 64, 200, 25, 64), (torch.bfloat16, 64, 8, 96, 32), (torch.float16, 32, 200, 3, 32)])
def test_ring_parts_of_a_block_column(mode, compressed, dtype, wide, rows, columns, tile, gpu):
    """64-row tiles narrower than the blocks: both sides of the sizes from which a block-column is cut, both storages of the
    sparse operand, either way round, with bias."""
    blocks = (32, 64, wide) if mode == 'dsd' else (wide, 64, 32)
    M, N = (rows, wide * columns) if mode == 'dsd' else (wide * columns, rows)
    _, names = launched_kernels(lambda: run_case(gpu, mode, False, mode == 'dsd', True, compressed, dtype, blocks, batch=1, M=M, K=192, N=N,
                                                 gran=(wide, 64), sparsity=0.4, seed=rows + columns, tile_cfg=11))
    assert [n[1] for n in template_numbers(names, 'spmm_ring_kernel')] == [tile]


@pytest.mark.parametrize('mode,transposed,compressed', [('dsd', True, True), ('dsd', False, True), ('dsd', True, False), ('sdd', False, True)])
@pytest.mark.parametrize('dtype,wide,depth,columns,K,sparsity,groups', [
    # eight panels of rows, a tile of every column to an XCD: 32 and 64 of them, and one more
    (torch.float16, 32, 64, 32, 768, 0.6, 3), (torch.bfloat16, 32, 64, 33, 768, 0.6, 2), (torch.float16, 64, 64, 64, 768, 0.6, 2),
    (torch.float16, 32, 64, 65, 768, 0.6, 1), (torch.float32, 16, 32, 32, 512, 0.6, 3), (torch.float32, 16, 64, 64, 512, 0.6, 2),
    (torch.float32, 32, 32, 40, 512, 0.6, 1),     # halves: 80 tiles
    # two blocks to a stage: odd walks, shares of one block, columns with fewer blocks than groups, and with none
    (torch.float16, 32, 32, 20, 480, 0.5, 3), (torch.bfloat16, 32, 32, 50, 320, 0.4, 2), (torch.float32, 16, 16, 24, 240, 0.6, 3),
    (torch.float16, 32, 64, 20, 640, 0.9, 1)])   # a stage or less to a walk: one group
def test_ring_groups(mode, transposed, compressed, dtype, wide, depth, columns, K, sparsity, groups, gpu, rows=504):
    """A walk shared out over groups of wavefronts: both sides of the sizes at which their number changes, with bias and rows
    that end inside a tile."""
    blocks = (32, depth, wide) if mode == 'dsd' else (wide, depth, 32)
    M, N = (rows, wide * columns) if mode == 'dsd' else (wide * columns, rows)
    _, names = launched_kernels(lambda: run_case(gpu, mode, False, transposed, True, compressed, dtype, blocks, batch=1, M=M, K=K, N=N,
                                                 gran=(depth, wide) if mode == 'dsd' and not transposed else (wide, depth), sparsity=sparsity, seed=columns, tile_cfg=11))
    numbers = template_numbers(names, 'spmm_ring_kernel')
    assert len(numbers) == 1
    # (where the blocks are not counted, an eighth of the places: two stages or less here)
    assert numbers[0][-1] == (groups if compressed else 1), numbers


@pytest.mark.parametrize('mode,transposed,compressed', [('dsd', True, True), ('dsd', False, True), ('dsd', True, False), ('dsd', False, False),
                                                        ('sdd', False, True), ('sdd', False, False)])
@pytest.mark.parametrize('dtype,wide,depth,rows,columns,batch,K,tile,groups', [
    # 16-bit block-columns 64 wide cut in halves whose walks are shared: 96 of them, few rows, a tile to a batch entry and XCD
    (torch.float16, 64, 64, 504, 12, 1, 1280, 32, 3), (torch.bfloat16, 64, 32, 8, 44, 1, 3392, 32, 3), (torch.float16, 64, 64, 40, 2, 40, 1280, 32, 2),
    # as many stages as the estimate of uncounted blocks has to reach
    (torch.float16, 32, 32, 504, 20, 1, 1280, 32, 3), (torch.bfloat16, 32, 64, 504, 40, 1, 1280, 32, 2), (torch.float32, 64, 16, 200, 10, 1, 640, 16, 3),
    (torch.float32, 16, 64, 504, 40, 1, 640, 16, 2)])
def test_ring_groups_of_cut_and_of_uncounted_block_columns(mode, transposed, compressed, dtype, wide, depth, rows, columns, batch, K, tile, groups, gpu):
    """Walks shared out over groups of wavefronts where a tile is half of a block-column, and where the sparse operand is a dense
    tensor under a mask, i.e. the groups follow from its places."""
    blocks = (32, depth, wide) if mode == 'dsd' else (wide, depth, 32)
    M, N = (rows, wide * columns) if mode == 'dsd' else (wide * columns, rows)
    _, names = launched_kernels(lambda: run_case(gpu, mode, False, transposed, True, compressed, dtype, blocks, batch=batch, M=M, K=K, N=N,
                                                 gran=(depth, wide) if mode == 'dsd' and not transposed else (wide, depth), sparsity=0.7,
                                                 seed=columns, tile_cfg=11))
    numbers = template_numbers(names, 'spmm_ring_kernel')
    assert [(n[1], n[-1]) for n in numbers] == [(tile, groups)], numbers


@pytest.mark.parametrize('tile_cfg', [11, 12])
@pytest.mark.parametrize('dtype,blocks', [(torch.float16, (32, 32, 32)), (torch.bfloat16, (32, 64, 32))])
def test_ring_results_with_an_activation(tile_cfg, dtype, blocks, gpu):
    """64-byte row pieces that are written through the L2s and that are not, rows that end inside a tile.  Which of the sizes are
    does not show in the values: test_cpu_ring_plan.py asks the rule that the kernel asks."""
    K, N = RESULTS_K_N
    for M in [m for rows, m in RESULTS_THROUGH if rows == (64 if tile_cfg == 11 else 128)]:
        run_case(gpu, 'dsd', False, True, True, M != 2200, dtype, blocks, batch=1, M=M, K=K, N=N, gran=(blocks[2], blocks[1]),
                 sparsity=0.7, seed=M, tile_cfg=tile_cfg, activation='relu')


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('M,N,batch', [(512, 1024, 1), (512, 1056, 1), (480, 512, 2), (480, 544, 2), (2000, 96, 1), (65, 5120, 1), (320, 5152, 1)])
def test_ring_one_tile_to_a_workgroup(M, N, batch, dtype, gpu, K=4096):
    """Both sides of one workgroup to a CU, where the launch order is left out, and of one tile to a workgroup; more
    panels than the L2 of an XCD holds, and block-columns cut in parts."""
    run_case(gpu, 'dsd', False, True, True, True, dtype, (32, 32, 32), batch=batch, M=M, K=K, N=N, gran=(32, 32),
             sparsity=0.97, seed=M + N, tile_cfg=11)


def test_ring_more_block_columns_than_the_table(gpu):
    run_case(gpu, 'dsd', False, True, False, True, torch.float16, (32, 32, 16), batch=1, M=520, K=96, N=16 * 1100,
             gran=(16, 32), sparsity=0.6, seed=61, tile_cfg=11)


@pytest.mark.parametrize('dtype,blocks,M,K,N,sparsity', [
    # split columns: first and last row count, ragged rows, a result wide enough for 512 tiles of 256 rows
    (torch.float32, (16, 16, 16), 257, 784, 512, 0.8), (torch.float32, (16, 16, 16), 520, 832, 2736, 0.95),
    (torch.float32, (16, 16, 16), 1024, 1056, 2048, 0.9),
    # ... more rows: up to 32 and up to 64 block-columns, both sides of the live-block limits
    (torch.float32, (16, 16, 16), 1025, 1056, 512, 0.8), (torch.float32, (16, 16, 16), 1500, 1056, 1024, 0.7),
    (torch.float32, (16, 16, 16), 1025, 800, 512, 0.95), (torch.float32, (16, 16, 16), 1025, 1056, 1040, 0.8),
    # fp32 16 x 16 around the rows and columns that the ring kernel is looked at for (test_dispatch_of_fp32_blocks_of_16 reads the launches)
    (torch.float32, (16, 16, 16), 700, 784, 1040, 0.7), (torch.float32, (16, 16, 16), 699, 784, 1040, 0.7), (torch.float32, (16, 16, 16), 900, 1408, 1552, 0.84),
    (torch.float32, (16, 16, 16), 900, 1408, 1536, 0.7), (torch.float32, (16, 16, 16), 2049, 768, 1536, 0.86), (torch.float32, (16, 16, 16), 6001, 512, 512, 0.9),
    # ring: 1100 tiles of 64 rows in tiles of 64 and of 128, and one column fewer
    (torch.float16, (32, 32, 32), 257, 1024, 7040, 0.95), (torch.float16, (32, 32, 32), 257, 1024, 7008, 0.95),
    # 256-row tiles: a block or less to a block-column, and one side of each limit
    (torch.float16, (32, 32, 64), 4100, 512, 1024, 0.9), (torch.bfloat16, (64, 64, 64), 4096, 256, 2048, 0.8),
    (torch.float16, (32, 32, 64), 4100, 512, 1024, 0.8), (torch.float16, (32, 32, 64), 4095, 512, 1024, 0.9),
    (torch.bfloat16, (32, 32, 32), 1024, 1056, 2208, 0.9), (torch.bfloat16, (32, 32, 32), 1200, 1024, 1888, 0.9)])
def test_dispatch_of_few_rows_and_long_columns(dtype, blocks, M, K, N, sparsity, gpu):
    """The sizes at which the library's own choice changes, compressed (where it knows the number of live
    blocks) and not, with bias and with every other call's activation fused."""
    for compressed in (True, False):
        run_case(gpu, 'dsd', False, True, True, compressed, dtype, blocks, batch=1, M=M, K=K, N=N, gran=(blocks[2], blocks[1]),
                 sparsity=sparsity, seed=71, tile_cfg=0, activation='relu' if compressed else None)


@pytest.mark.parametrize('storage', ['dense', 'capacity', 'counted'])
@pytest.mark.parametrize('M,K,N,live,kernels', [
    # few rows, up to 32 places to a column: up to 256 tiles and more
    (128, 512, 1536, 1, ('direct', 'direct')), (128, 512, 1536, 10, ('direct', 'ring')), (256, 768, 3072, 2, ('ring', 'direct')),
    # ... up to 48 rows and more
    (48, 704, 704, 11, ('direct', 'direct')), (48, 704, 704, 12, ('direct', 'ring')), (49, 704, 704, 6, ('direct', 'ring')),
    # four live blocks to a column and five, up to 256 tiles and more
    (128, 1280, 1024, 4, ('ring', 'ksplit')), (128, 1280, 1024, 5, ('ring', 'ring')), (300, 1280, 1664, 4, ('ring', 'ring')),
    # 39 places, 40, 64 and 65; more than 256 tiles with fewer
    (300, 1248, 1024, 8, ('ksplit', 'ring')), (300, 1280, 1024, 3, ('ring', 'ksplit')), (300, 2048, 1024, 8, ('ring', 'ring')),
    (300, 2080, 1024, 8, ('ksplit', 'ring')), (300, 1088, 2048, 8, ('ring', 'ring')),
    # wide results of 1025 to 1536 rows
    (1500, 1024, 3072, 2, ('ring', 'panel')), (1500, 1024, 3072, 5, ('ring', 'ring'))])
def test_dispatch_of_few_tiles(M, K, N, live, kernels, storage, gpu):
    """16-bit blocks of 32 x 32, few tiles.  A dense operand under a mask and a compressed one at the capacity of its index take the kernel
    that fits the places (first of `kernels`), one that is counted the kernel that fits its live blocks."""
    rng = np.random.default_rng(M + K)
    nb, cols = N // 32, K // 32
    grid = np.zeros(nb * cols, np.uint8)
    grid[rng.permutation(nb * cols)[:live * nb]] = 1
    mask = torch.from_numpy(np.kron(grid.reshape(nb, cols), np.ones((32, 32), np.uint8))).to(gpu)
    kernel = SparTASparseMatMulKernel(mode='dsd', biased=False, transpose_A=False, transpose_B=True, compressed=storage != 'dense')
    kernel.ports['B'].set_mask(mask)
    kernel.ports['B'].at_capacity = storage == 'capacity'
    kernel.set_shape(1, M, K, N)
    kernel.compile({'BLOCK_SIZE_M_VALUE': 32, 'BLOCK_SIZE_K_VALUE': 32, 'BLOCK_SIZE_N_VALUE': 32})
    g = torch.Generator(device=gpu).manual_seed(M)
    A, B = (torch.randn(s, generator=g, device=gpu).half() for s in ((1, M, K), (1, N, K)))
    B = B * mask
    packed = B if storage == 'dense' else kernel.ports['B'].indexes.convert(B, at_capacity=storage == 'capacity')
    C, names = launched_kernels(lambda: kernel(A, packed))
    assert_close(C, torch.matmul(A[0].double(), B[0].double().T).cpu().numpy()[None], torch.float16, f'{M}x{K}x{N} {storage}')
    taken = [k for k in ('direct', 'ksplit', 'ring', 'panel', 'stream') if any(f'spmm_{k}' in n for n in names)]
    assert taken == [kernels[storage == 'counted']], names


@pytest.mark.parametrize('tile_cfg', [0, 11, 12])
@pytest.mark.parametrize('mode,depth', [('dsd', 16), ('sdd', 16), ('dsd', 64)])
def test_ring_sums_of_narrow_fp32_blocks(tile_cfg, mode, depth, gpu, size=1024, sparsity=0.65):
    """fp32 blocks 16 wide: four chains to a sum, as long as where four wavefronts share a block-column (the column-split kernel,
    which some of these sizes went through).  In one chain the error would be twice the expected one."""
    kernel = SparTASparseMatMulKernel(mode=mode, biased=False, transpose_A=False, transpose_B=True, compressed=True)
    port, tile = ('B', (16, depth)) if mode == 'dsd' else ('A', (16, depth))
    mask = torch.from_numpy(ops.block_mask((size, size), tile, sparsity, seed=9)).to(gpu)
    kernel.ports[port].set_mask(mask)
    kernel.set_shape(1, size, size, size)
    kernel.compile({'BLOCK_SIZE_M_VALUE': 16, 'BLOCK_SIZE_K_VALUE': depth, 'BLOCK_SIZE_N_VALUE': 16, 'TILE_CFG': tile_cfg})
    g = torch.Generator(device=gpu).manual_seed(6)
    A, B = (torch.randn((1, size, size), generator=g, device=gpu) for _ in range(2))
    sparse = (B if mode == 'dsd' else A) * mask
    A, B = (A, sparse) if mode == 'dsd' else (sparse, B)
    packed = kernel.ports[port].indexes.convert(sparse)
    got = kernel(A, packed) if mode == 'dsd' else kernel(packed, B)
    want = A[0].double() @ B[0].double().t()
    assert float((got[0].double() - want).norm() / want.norm()) <= 1.3 * chained_sum_error((1 - sparsity) * size / 4)


@pytest.mark.parametrize('M,K,N,live,kernel', [
    # split columns or ring: one round of tiles with 22 blocks to a column and with 32; two rounds, a quarter of the second, and three full ones
    (1024, 1024, 1024, 22 * 64, 'ring'), (1024, 1024, 1024, 32 * 64, 'ksplit'), (1809, 1056, 704, 20 * 44, 'ksplit'), (774, 784, 3584, 12 * 224, 'ring'),
    # first row count, longest columns, and the ones beside them
    (700, 784, 1024, 12 * 64, 'ring'), (699, 784, 1024, 12 * 64, 'ksplit'), (700, 1408, 1024, 12 * 64, 'ring'), (700, 1424, 1024, 12 * 64, 'ksplit'),
    # 256-row tiles or ring: five panels and eight
    (1044, 1328, 3648, 8 * 228, 'ring'), (1848, 1040, 1920, 7 * 120, 'panel'),
    # more rows: nine panels and sixteen, columns of up to 48 k-blocks, two to eight blocks to a column, up to 96 columns, last row count
    (2049, 576, 1024, 2 * 64, 'ring'), (2049, 576, 1024, 2 * 64 - 1, 'panel'), (2199, 512, 1408, 8 * 88, 'ring'), (2199, 512, 1408, 8 * 88 + 1, 'panel'),
    (2049, 576, 1552, 4 * 97, 'panel'), (3995, 512, 960, 2 * 60, 'panel'), (4577, 768, 512, 5 * 32, 'ring'), (4577, 784, 512, 5 * 32, 'panel'),
    (6000, 512, 576, 3 * 36, 'ring'), (6001, 512, 576, 3 * 36, 'panel')])
def test_dispatch_of_fp32_blocks_of_16(M, K, N, live, kernel, gpu):
    """fp32 blocks of 16 x 16 run through the ring kernel, with 64-row tiles, where the estimates say so: both sides of what they turn
    on, and of the sizes that they are asked for."""
    import sparta_amd as sparta
    grid = np.zeros(N // 16 * (K // 16), dtype=np.uint8)
    grid[np.random.default_rng(M + live).permutation(grid.size)[:live]] = 1
    mask_np = np.repeat(np.repeat(grid.reshape(N // 16, K // 16), 16, 0), 16, 1)
    lin = torch.nn.Linear(K, N, bias=True, device=gpu)
    x = torch.randn((M, K), generator=torch.Generator(device=gpu).manual_seed(7), device=gpu)
    op = sparta.nn.SparseLinear(lin, weight_mask=torch.from_numpy(mask_np).to(gpu))
    op.build({'forward:C': {'_impl': 'sparta', 'BLOCK_SIZE_M_VALUE': 32, 'BLOCK_SIZE_K_VALUE': 16, 'BLOCK_SIZE_N_VALUE': 16}}, sample_inputs=[x])
    with torch.no_grad():
        y, names = launched_kernels(lambda: op(x))
    assert [k for k in ('ring', 'ksplit', 'panel') if any(f'spmm_{k}' in n for n in names)] == [kernel], names
    if kernel == 'ring':
        assert [n[0] for n in template_numbers(names, 'spmm_ring_kernel')] == [64], names
    want = x.double().cpu().numpy() @ (lin.weight.detach().double().cpu().numpy() * mask_np).T + lin.bias.detach().double().cpu().numpy()
    assert_close(y, want, torch.float32, f'{M} x {K} -> {N}, {live} blocks')


@pytest.mark.parametrize('M', [110100, 40000])
def test_ring_more_tiles_than_the_list(M, gpu, K=64, N=1536):
    """More than 128 tiles to a workgroup, which then looks every tile up, and 32 of them."""
    import sparta_amd as sparta
    g = torch.Generator(device=gpu).manual_seed(5)
    mask = (torch.rand((N // 16, K // 32), generator=g, device=gpu) < 0.6).to(torch.uint8).repeat_interleave(16, 0).repeat_interleave(32, 1).contiguous()
    lin = torch.nn.Linear(K, N, bias=True, device=gpu, dtype=torch.float16)
    x = torch.randn((M, K), generator=g, device=gpu).half()
    op = sparta.nn.SparseLinear(lin, weight_mask=mask)
    op.build({'forward:C': {'_impl': 'sparta', 'BLOCK_SIZE_M_VALUE': 32, 'BLOCK_SIZE_K_VALUE': 32, 'BLOCK_SIZE_N_VALUE': 16, 'TILE_CFG': 11}},
             sample_inputs=[x])
    weight = (lin.weight.detach() * mask).float().t().contiguous()
    with torch.no_grad():
        y = op(x)
        for r in range(0, M, 16384):
            want = torch.matmul(x[r:r + 16384].float(), weight) + lin.bias.float()
            # result rounded to 11 bits; sums of 64 products in fp32
            assert float((y[r:r + 16384].float() - want).abs().max()) <= 2 ** -11 * float(want.abs().max()) + 1e-5


@pytest.mark.parametrize('tile_cfg,batch,M,N', [
    # 64-row tiles: 128 tiles to a workgroup on some XCDs and 129 on others, in every row of 16-wide block-columns
    (11, 1, 109100, 1536), (11, 1, 109056, 1536),
    # 128-row tiles: 128 and 129, and 128 everywhere
    (12, 1, 131200, 1536), (12, 1, 131072, 1536),
    # a batch that leaves an XCD one workgroup an entry: 120 and 135, and 120 everywhere
    (11, 128, 4160, 240), (11, 128, 4096, 240)])
def test_ring_xcds_on_the_two_sides_of_the_longest_list(tile_cfg, batch, M, N, gpu, K=64):
    mask_np = ops.block_mask((N, K), (16, 32), 0.4, seed=9)
    mask = torch.from_numpy(mask_np).to(gpu)
    g = torch.Generator(device=gpu).manual_seed(6)
    A, B, bias = (torch.randn(shape, generator=g, device=gpu).half() for shape in ((batch, M, K), (batch, N, K), (batch, N)))
    kernel = SparTASparseMatMulKernel(mode='dsd', biased=True, transpose_A=False, transpose_B=True, compressed=True)
    kernel.ports['B'].set_mask(mask)
    kernel.set_shape(batch, M, K, N)
    kernel.compile({'BLOCK_SIZE_M_VALUE': 32, 'BLOCK_SIZE_K_VALUE': 32, 'BLOCK_SIZE_N_VALUE': 16, 'TILE_CFG': tile_cfg})
    B = B * mask.half()
    C = kernel(A, kernel.ports['B'].indexes.convert(B), bias)
    for i in range(batch):
        weight = B[i].float().t().contiguous()
        for r in range(0, M, 32768):
            want = torch.matmul(A[i, r:r + 32768].float(), weight) + bias[i].float()
            # result rounded to 11 bits; sums of 64 products in fp32
            assert float((C[i, r:r + 32768].float() - want).abs().max()) <= 2 ** -11 * float(want.abs().max()) + 1e-5


@pytest.mark.parametrize('dtype,blocks,M,K,N,sparsity', [
    # 64-row tiles in one round and in two, 128-row tiles in one; and both in two
    (torch.float16, (32, 32, 32), 2560, 64, 1024, 0.5), (torch.float16, (32, 32, 32), 2561, 64, 1024, 0.5),
    (torch.bfloat16, (32, 64, 32), 2500, 128, 2048, 0.6), (torch.bfloat16, (64, 64, 64), 4096, 128, 832, 0.6),
    # few rows, long columns: both sides of 700 tiles, and of 512 with few and with many blocks to a column
    (torch.float16, (32, 32, 32), 770, 1024, 1696, 0.7), (torch.float16, (32, 32, 32), 770, 1024, 1728, 0.7),
    # wide results of 2048 to 3072 rows
    (torch.float16, (32, 32, 32), 2049, 1024, 2048, 0.9), (torch.float16, (32, 32, 32), 3073, 1024, 2048, 0.9),
    (torch.bfloat16, (32, 32, 32), 1000, 1056, 1024, 0.9), (torch.bfloat16, (32, 32, 32), 1000, 1056, 1024, 0.6),
    (torch.bfloat16, (32, 32, 32), 1000, 1056, 992, 0.9)])
def test_dispatch_of_rows_to_a_tile(dtype, blocks, M, K, N, sparsity, gpu):
    for compressed in (True, False):
        run_case(gpu, 'dsd', False, True, True, compressed, dtype, blocks, batch=1, M=M, K=K, N=N, gran=(blocks[2], blocks[1]),
                 sparsity=sparsity, seed=81, tile_cfg=0)
