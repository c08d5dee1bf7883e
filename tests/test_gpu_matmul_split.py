"""The k-split sparse-output product (spx_matmul_split) against the numpy oracle: every slice count,
depths below one stage, ragged and with slices that stay empty, the four operand layouts, and the
column sums that ride along as the bias gradient of a linear layer."""
import numpy as np
import pytest
import torch

import sparta_amd as sparta
from oracle import bcs, ops
from sparta_amd import _lib
from sparta_amd.tesa import get_bcs_function
from helpers import randn, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('slices', [0, 1, 2, 4, 8])
@pytest.mark.parametrize('K', [16, 80, 784])
@pytest.mark.parametrize('tA,tB', [(True, False), (False, True), (True, True), (False, False)])
@pytest.mark.parametrize('dtype,block', [(torch.float16, (32, 64)), (torch.bfloat16, (16, 16)), (torch.float32, (32, 32)),
                                         (torch.float32, (64, 64)), (torch.float16, (64, 16))])
def test_split_product_and_column_sums(slices, K, tA, tB, dtype, block, gpu, M=192, N=256, batch=2):
    BM, BN = block
    a_np, a = randn((batch, K, M) if tA else (batch, M, K), 1, dtype)
    b_np, b = randn((batch, N, K) if tB else (batch, K, N), 2, dtype)
    mask_np = ops.block_mask((M, N), block, 0.7, seed=3)
    idx = get_bcs_function(BM, BN, True, False).build_indexes(torch.from_numpy(mask_np).to(gpu))
    nnz, lib, code = idx.block_nnz, _lib.load(), _lib.dtype_code(dtype)
    a, b = a.to(gpu), b.to(gpu)
    op_a = a_np.transpose(0, 2, 1) if tA else a_np
    want = op_a @ (b_np.transpose(0, 2, 1) if tB else b_np)
    for compressed in (True, False):
        stride = nnz * BM * BN
        out = torch.full((batch, stride), float('nan'), dtype=dtype, device=gpu) if compressed \
            else torch.zeros((batch, M, N), dtype=dtype, device=gpu)
        sums = torch.full((batch, M), float('nan'), dtype=dtype, device=gpu) if tA else None
        nbytes = lib.spx_matmul_split_workspace_bytes(code, tA, tB, nnz, batch, M, K, N, BM, BN, slices, tA)
        ws = torch.empty((max(nbytes, 16),), dtype=torch.uint8, device=gpu)
        rc = lib.spx_matmul_split(code, tA, tB, compressed, _lib.dev_ptr(a), _lib.dev_ptr(b), _lib.dev_ptr(out), _lib.dev_ptr(sums),
                                  _lib.dev_ptr(idx.row_ptr), _lib.dev_ptr(idx._bcsr_buf), nnz, stride, batch, M, K, N, BM, BN,
                                  slices, _lib.dev_ptr(ws), nbytes, _lib.current_stream(gpu))
        _lib.check(rc, 'spx_matmul_split')
        expect = bcs.convert(want, idx.BCSR_idx.cpu().numpy(), 'bcsr', BM, BN) if compressed else want * idx.get_mask().cpu().numpy()
        assert_close(out, expect, dtype, f'slices={slices} compressed={compressed}')
        if tA:
            assert_close(sums, op_a.sum(2), dtype, 'column sums')


@pytest.mark.parametrize('M', [16, 208, 1040])
@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16, torch.float32])
def test_linear_training_step_with_ragged_token_counts(M, dtype, gpu, K=256, N=192):
    """Gradients of SparseLinear for token counts that are no multiple of a stage, every gradient in the
    shape of its tensor; with the bias frozen, and with only the bias trained."""
    _, x = randn((M, K), 4, dtype)
    _, w = randn((N, K), 5, dtype, scale=0.1)
    _, bias = randn((N,), 6, dtype)
    _, gy = randn((M, N), 7, dtype)
    mask_np = ops.block_mask((N, K), (32, 64), 0.5, seed=8)
    lin = torch.nn.Linear(K, N, device=gpu, dtype=dtype)
    with torch.no_grad():
        lin.weight.copy_((w * torch.from_numpy(mask_np).to(dtype)).to(gpu))
        lin.bias.copy_(bias.to(gpu))
    op = sparta.nn.SparseLinear(lin, weight_mask=torch.from_numpy(mask_np).to(gpu))
    mm = lambda m, k, n: {'_impl': 'sparta', 'BLOCK_SIZE_M_VALUE': m, 'BLOCK_SIZE_K_VALUE': k, 'BLOCK_SIZE_N_VALUE': n}
    op.build({'forward:C': mm(32, 64, 32), 'backward:A': mm(32, 32, 64), 'backward:B': mm(32, 32, 64)}, sample_inputs=[x.to(gpu)])
    xn, wn, gn = x.double().numpy(), (w.double() * torch.from_numpy(mask_np)).numpy(), gy.double().numpy()
    want = {'x': gn @ wn, 'w': (gn.T @ xn) * mask_np, 'b': gn.sum(0)}
    for train_w, train_b in ((True, True), (True, False), (False, True)):
        op.weight.requires_grad_(train_w)
        op.bias.requires_grad_(train_b)
        op.weight.grad = op.bias.grad = None
        xs = x.to(gpu).requires_grad_(True)
        op(xs).backward(gy.to(gpu))
        assert xs.grad.shape == xs.shape
        scale = float(np.sqrt(max(M, N)))   # sums of that many products of N(0, 1) values
        assert_close(xs.grad, want['x'], dtype, 'grad_x', scale=scale)
        assert (op.weight.grad is not None) == train_w and (op.bias.grad is not None) == train_b
        if train_w:
            assert op.weight.grad.shape == op.weight.shape
            assert_close(op.get_sparse_indexes('B').inverse(op.weight.grad), want['w'], dtype, 'grad_w', scale=scale)
        if train_b:
            assert_close(op.bias.grad, want['b'], dtype, 'grad_b', scale=scale)
