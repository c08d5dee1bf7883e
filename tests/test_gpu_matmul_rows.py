"""The kernel that keeps 64 rows of the dense operand in LDS (matmul_spmm_rows.hpp), through the library's own choice: 16-bit
compressed blocks of 32 x 32 over 2200 rows and more."""
import pytest
import torch

from helpers import launched_kernels
from test_gpu_matmul import run_case

pytestmark = pytest.mark.gpu


def takes_rows(names):
    return any('spmm_rows_kernel' in n for n in names)


@pytest.mark.parametrize('dtype,M,K,N,sparsity,taken', [
    # first row count, the one before, and workgroups that fill less than half of the chip; a tile of one row, of 63
    (torch.float16, 2200, 768, 1600, 0.8, True), (torch.float16, 2199, 768, 1600, 0.8, False), (torch.float16, 2200, 768, 1088, 0.8, False),
    (torch.float16, 2199, 768, 1088, 0.8, False), (torch.bfloat16, 3649, 768, 1088, 0.8, True), (torch.float16, 3647, 768, 1088, 0.8, True),
    # both sides of two blocks to a column, and of four where rows are short
    (torch.float16, 4100, 768, 1024, 0.91, True), (torch.float16, 4100, 768, 1024, 0.93, False), (torch.bfloat16, 4100, 512, 1024, 0.74, True),
    (torch.bfloat16, 4100, 512, 1024, 0.77, False),
    # shares of unequal length, more columns to a share than wavefronts and fewer, one share, two rounds
    (torch.float16, 2624, 832, 2016, 0.7, True), (torch.float16, 4160, 832, 1184, 0.7, True), (torch.float16, 2624, 832, 1184, 0.7, False),
    (torch.float16, 8300, 768, 1024, 0.75, True), (torch.bfloat16, 8200, 576, 1056, 0.7, True), (torch.float16, 16300, 512, 512, 0.6, True),
    # the longest rows that fit, few and many block-columns beside them, and the first that do not
    (torch.float16, 2500, 1152, 2080, 0.7, True), (torch.bfloat16, 8200, 1216, 512, 0.7, True), (torch.float16, 4160, 1216, 1024, 0.8, True),
    (torch.bfloat16, 4100, 1216, 512, 0.7, False), (torch.float16, 4100, 1216, 512, 0.91, False), (torch.float16, 4100, 1280, 512, 0.7, False),
    (torch.float16, 8200, 1280, 512, 0.7, False)])
def test_rows_in_lds(dtype, M, K, N, sparsity, taken, gpu):
    _, names = launched_kernels(lambda: run_case(
        gpu, 'dsd', False, True, M % 2 == 0, True, dtype, (32, 32, 32), batch=1, M=M, K=K, N=N, gran=(32, 32),
        sparsity=sparsity, seed=M + N, tile_cfg=0, activation='relu' if K == 768 else None))
    assert takes_rows(names) == taken, names


@pytest.mark.parametrize('dtype,M,K,N,sparsity', [
    (torch.float16, 2200, 768, 1600, 0.8), (torch.bfloat16, 4160, 1216, 1024, 0.8), (torch.float16, 8200, 576, 1056, 0.7)])
def test_rows_in_lds_give_the_bits_of_256_row_tiles(dtype, M, K, N, sparsity, gpu):
    """Both add up the blocks of a column in index order, 16 k at a time."""
    import sparta_amd as sparta
    g = torch.Generator(device=gpu).manual_seed(8)
    mask = (torch.rand((N // 32, K // 32), generator=g, device=gpu) > sparsity).to(torch.uint8).repeat_interleave(32, 0).repeat_interleave(32, 1).contiguous()
    lin = torch.nn.Linear(K, N, bias=True, device=gpu, dtype=dtype)
    x = torch.randn((M, K), generator=g, device=gpu).to(dtype)
    got = []
    for tile_cfg in (0, 7):
        op = sparta.nn.SparseLinear(lin, weight_mask=mask)
        op.build({'forward:C': {'_impl': 'sparta', 'BLOCK_SIZE_M_VALUE': 32, 'BLOCK_SIZE_K_VALUE': 32, 'BLOCK_SIZE_N_VALUE': 32, 'TILE_CFG': tile_cfg}},
                 sample_inputs=[x])
        with torch.no_grad():
            y, names = launched_kernels(lambda: op(x))
        assert takes_rows(names) == (tile_cfg == 0) and any('spmm_panel_kernel' in n for n in names) == (tile_cfg == 7), names
        got.append(y)
    assert torch.equal(*got)


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
def test_rows_in_lds_shares_without_a_block(dtype, gpu, M=5800, K=768, N=1024):
    """Full block-columns on the left, none on the right: the second share has no block to read.  Infinities next to them
    stay out of the result."""
    import sparta_amd as sparta
    g = torch.Generator(device=gpu).manual_seed(3)
    mask = torch.zeros((N, K), dtype=torch.uint8, device=gpu)
    mask[:256] = 1
    lin = torch.nn.Linear(K, N, bias=True, device=gpu, dtype=dtype)
    x = torch.randn((M, K), generator=g, device=gpu).to(dtype)
    x[5, 7] = float('inf')
    op = sparta.nn.SparseLinear(lin, weight_mask=mask)
    op.build({'forward:C': {'_impl': 'sparta', 'BLOCK_SIZE_M_VALUE': 32, 'BLOCK_SIZE_K_VALUE': 32, 'BLOCK_SIZE_N_VALUE': 32}}, sample_inputs=[x])
    with torch.no_grad():
        y, names = launched_kernels(lambda: op(x))
    assert takes_rows(names), names
    y = y.float()
    bias = lin.bias.detach().float()
    assert torch.equal(y[:, 256:], bias[256:].expand(M, -1))
    rows = torch.arange(M, device=gpu) != 5
    want = torch.matmul(x[rows].double(), lin.weight.detach()[:256].double().t()) + bias[:256].double()
    # result rounded to 11 or 8 bits, sums of 768 products in fp32
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert float((y[rows][:, :256] - want).abs().max()) <= unit * float(want.abs().max()) + 1e-4
    assert not torch.isfinite(y[5, :256]).any()


def test_rows_in_lds_batches(gpu):
    _, names = launched_kernels(lambda: run_case(gpu, 'dsd', False, True, True, True, torch.float16, (32, 32, 32), batch=3, M=2241, K=832, N=544,
                                                 gran=(32, 32), sparsity=0.7, seed=19, tile_cfg=0))
    assert takes_rows(names), names
