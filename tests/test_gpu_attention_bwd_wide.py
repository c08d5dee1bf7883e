"""The backward kernels of attention with 32 queries or keys per wavefront: element masks at every
block shape, and block-level masks from the number of workgroups on at which they take over, through
SparseAttention against float64."""
import numpy as np
import pytest
import torch

from sparta_amd.nn import SparseAttention
from helpers import randn
from test_gpu_attention import train_config

pytestmark = pytest.mark.gpu

# 2-norm error of a gradient: five 16-bit roundings of half an ulp (probabilities, score gradient, scaled
# operands, output, result), 2^-12 and 2^-9 each at most, add up in squares to 6e-4 and 5e-3
REL = {torch.float16: 1.2e-3, torch.bfloat16: 1e-2}


def step(att, leaves, g):
    for t in leaves:
        t.grad = None
    att(*leaves).backward(g)
    return [t.grad.detach().double() for t in leaves]


def exact(leaves, g, mask):
    q, k, v = (t.detach().double().requires_grad_(True) for t in leaves)
    scores = torch.matmul(q, k.transpose(1, 2).contiguous()) / float(np.sqrt(q.shape[-1]))
    probs = torch.softmax(scores.masked_fill(mask == 0, float('-inf')), -1).nan_to_num(0.0)
    torch.matmul(probs, v).backward(g.double())
    return [t.grad for t in (q, k, v)]


def check(got, want, dtype, what):
    for name, a, b in zip(('q', 'k', 'v'), got, want):
        assert torch.isfinite(a).all(), f'{what}: gradient of {name}'
        rel = float((a - b).norm() / b.norm())
        assert rel <= REL[dtype], f'{what}: gradient of {name} off by {rel:.2e}'


def block_mask(Nt, Ns, bh, bw, seed, density=0.4):
    rng = np.random.default_rng(seed)
    grid = rng.random((Nt // bh, Ns // bw)) < density
    grid[0] = False        # a block row without an entry
    grid[:, 1] = False     # a block column without one
    grid[1, 0] = True
    return np.kron(grid, np.ones((bh, bw), np.uint8)).astype(np.uint8)


def build(mask, bh, bw, q, k, v, gpu):
    att = SparseAttention(mask=torch.from_numpy(mask).to(gpu))
    leaves = [t.to(gpu).requires_grad_(True) for t in (q, k, v)]
    att.build(train_config(bh, bw), sample_inputs=[t.detach() for t in leaves])
    return att, leaves


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('bh,bw', [(32, 32), (64, 64), (32, 64), (64, 32)])
def test_element_mask(dtype, bh, bw, gpu, H=9, Nt=256, Ns=512):
    """Partly live blocks, fully masked queries and keys, values of the mask other than one."""
    rng = np.random.default_rng(3)
    mask = block_mask(Nt, Ns, bh, bw, 1) * (rng.random((Nt, Ns)) < 0.7).astype(np.uint8)
    mask[:, 5 * bw // 4:] |= np.tril(block_mask(Nt, Ns, bh, bw, 2))[:, 5 * bw // 4:]
    mask[bh + 3] = 0
    mask[:, 7] = 0
    mask[bh:, 40:60] *= 2
    q, k, v, g = (randn(s, i, dtype)[1] for i, s in enumerate([(H, Nt, 64), (H, Ns, 64), (H, Ns, 64), (H, Nt, 64)]))
    att, leaves = build(mask, bh, bw, q, k, v, gpu)
    att._fused_forward_train = None   # nothing is stored
    m = torch.from_numpy(mask).to(gpu)
    got = step(att, leaves, g.to(gpu))
    check(got, exact(leaves, g.to(gpu), m), dtype, f'{dtype} {bh}x{bw}')
    assert float(got[0][:, bh + 3].abs().max()) == 0.0 and float(got[1][:, 7].abs().max()) == 0.0


def test_element_mask_is_the_one_of_the_forward_pass(gpu, H=8, N=256):
    """The caller's mask tensor may be overwritten, and the operator's mask updated, ahead of the backward pass."""
    mask = np.tril(np.ones((N, N), np.uint8))
    q, k, v, g = (randn((H, N, 64), i, torch.float16)[1] for i in range(4))
    att, leaves = build(mask, 64, 64, q, k, v, gpu)
    out = att(*leaves)
    att.mask.zero_()
    att.update_mask(torch.from_numpy(block_mask(N, N, 64, 64, 5)).to(gpu))
    out.backward(g.to(gpu))
    want = exact(leaves, g.to(gpu), torch.from_numpy(mask).to(gpu))
    check([t.grad.double() for t in leaves], want, torch.float16, 'after an update')


def test_long_rows_of_an_element_mask(gpu, H=2, Nt=1024, Ns=4096 + 64):
    """More than 64 entries to a block row, an int32 and an int64 index."""
    mask = np.ones((Nt, Ns), np.uint8)
    mask[::3, ::5] = 0
    q, k, v, g = (randn((H, n, 64), i, torch.float16)[1] for i, n in enumerate((Nt, Ns, Ns, Nt)))
    for n, (bh, bw) in enumerate([(32, 32), (64, 64)]):
        att, leaves = build(mask, bh, bw, q, k, v, gpu)
        att._fused_forward_train = None
        check(step(att, leaves, g.to(gpu)), exact(leaves, g.to(gpu), torch.from_numpy(mask).to(gpu)), torch.float16, f'{bh}x{bw}')


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('H,N', [(96, 512), (95, 512), (49, 1024)])
@pytest.mark.parametrize('bh,bw', [(64, 64), (64, 32), (32, 64)])
def test_block_level_mask(dtype, H, N, bh, bw, gpu):
    """768 workgroups and the sizes next to it; numbers of heads that are no multiple of eight."""
    mask = block_mask(N, N, bh, bw, 7, density=0.25)
    q, k, v, g = (randn((H, N, 64), i, dtype)[1] for i in range(4))
    att, leaves = build(mask, bh, bw, q, k, v, gpu)
    check(step(att, leaves, g.to(gpu)), exact(leaves, g.to(gpu), torch.from_numpy(mask).to(gpu)), dtype, f'{H} x {N} {bh}x{bw}')


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('bh,bw', [(64, 64), (32, 32)])
def test_element_mask_with_the_wide_forward_kernel(dtype, bh, bw, gpu, H=64, N=1024):
    """65536 queries: the forward pass that records the row statistic is the one with 32 queries per wavefront."""
    mask = np.tril(block_mask(N, N, bh, bw, 9, density=0.3) | np.kron(np.eye(N // bh), np.ones((bh, bw))).astype(np.uint8))
    mask[70] = 0
    q, k, v, g = (randn((H, N, 64), i, dtype)[1] for i in range(4))
    att, leaves = build(mask, bh, bw, q, k, v, gpu)
    m = torch.from_numpy(mask).to(gpu)
    check(step(att, leaves, g.to(gpu)), exact(leaves, g.to(gpu), m), dtype, f'{dtype} {bh}x{bw}')
    with torch.no_grad():
        out = att(*leaves)
    assert float(out[:, 70].abs().max()) == 0.0


@pytest.mark.parametrize('H,N,window', [(1, 8192, 3), (4, 4096, 2)])
def test_element_mask_keeps_no_copy_of_all_of_it(H, N, window, gpu, blk=64):
    """A training step holds the bytes of the live blocks until its backward pass: beside the output and a float per
    query half of what one head's probabilities take, where the whole mask is N x N bytes."""
    i = np.arange(N // blk)
    grid = (i[:, None] >= i) & (i[:, None] - i < window)
    mask = np.tril(np.kron(grid, np.ones((blk, blk), np.uint8)))
    q, k, v, g = (randn((H, N, 64), j, torch.float16)[1] for j in range(4))
    att, leaves = build(mask, blk, blk, q, k, v, gpu)
    att(*leaves).sum().backward()   # the launch objects and what is kept of the index
    del leaves
    leaves = [t.to(gpu).requires_grad_(True) for t in (q, k, v)]
    live = int(grid.sum()) * blk * blk
    def step_bytes():
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        out = att(*leaves)
        held = torch.cuda.memory_allocated() - before
        out.backward(g.to(gpu))
        peak = torch.cuda.max_memory_allocated() - before
        for t in leaves:
            t.grad = None
        return held, peak
    held, peak = step_bytes()
    slack = 4 * 2 << 20   # four allocations, each rounded to 2 MB at most
    assert held <= H * N * 64 * 2 + H * N * 4 + live + slack, f'{held} bytes held'
    att._recompute = False    # the probabilities of the live blocks are stored
    stored, stored_peak = step_bytes()
    assert held <= stored and peak <= stored_peak


@pytest.mark.parametrize('bh,bw', [(32, 32), (64, 32), (32, 64)])
def test_whole_mask_and_its_live_blocks_give_the_same_gradients(bh, bw, gpu, H=3, Nt=256, Ns=2304):
    """The C entry points that read the [Nt, Ns] mask against the ones that read its live blocks, the columns through the
    int64 index and the int32 one, which orders the blocks by column; more than 64 entries to a block row."""
    from sparta_amd import _lib
    rng = np.random.default_rng(11)
    mask_np = (np.kron(rng.random((Nt // bh, Ns // bw)) < 0.95, np.ones((bh, bw))) * (rng.random((Nt, Ns)) < 0.8)).astype(np.uint8)
    q, k, v, g = (randn(s, i, torch.float16)[1] for i, s in enumerate([(H, Nt, 64), (H, Ns, 64), (H, Ns, 64), (H, Nt, 64)]))
    att, (q, k, v) = build(mask_np, bh, bw, q, k, v, gpu)
    q, k, v, g = q.detach(), k.detach(), v.detach(), g.to(gpu)
    indexes, mask = att._sparse_port.indexes, att._element_mask()
    out, lse = att._fused_forward_lse(q, k, v)
    live = att._live_mask()
    assert torch.equal(live, indexes.convert(mask).flatten())
    grad_q, dot = att._recompute_backward_q(g, out, q, k, v, lse, indexes, live)
    grad_k, grad_v = att._recompute_backward_kv(g, q, k, v, lse, dot, indexes, live)
    lib, ptr, stream = _lib.load(), _lib.dev_ptr, _lib.current_stream(gpu)
    code, inv_t = _lib.dtype_code(q.dtype), float(att._inv_temperature)
    sizes = (inv_t, H, Nt, Ns, 64, bh, bw, stream)
    whole_q, whole_dot = torch.empty_like(q), torch.empty_like(dot)
    _lib.check(lib.spx_attention_backward_q_masked(code, ptr(g), ptr(out), ptr(q), ptr(k), ptr(v), ptr(lse), ptr(whole_q), ptr(whole_dot),
                                                   ptr(indexes.row_ptr), ptr(indexes._bcsr_buf), ptr(mask), *sizes), 'masked')
    assert torch.equal(whole_q, grad_q) and torch.equal(whole_dot, dot)
    by_column = indexes.function_context.__class__(bh, bw, False, True).build_indexes(mask)
    for idx, kind, data, call in ((indexes._bcsc_buf, _lib.IDX_BCSC_I64, mask, lib.spx_attention_backward_kv_masked),
                                  (by_column._bcsc_buf, _lib.IDX_BCSC_I32, mask, lib.spx_attention_backward_kv_masked),
                                  (by_column._bcsc_buf, _lib.IDX_BCSC_I32, by_column.convert(mask), lib.spx_attention_backward_kv_live_mask)):
        whole_k, whole_v = torch.empty_like(k), torch.empty_like(v)
        _lib.check(call(code, ptr(g), ptr(q), ptr(k), ptr(v), ptr(lse), ptr(dot), ptr(whole_k), ptr(whole_v), ptr(indexes.col_ptr),
                        ptr(idx), kind, ptr(data), *sizes), 'masked')
        assert torch.equal(whole_k, grad_k) and torch.equal(whole_v, grad_v)


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('H,N,E,blk,elements', [
    (64, 4096, 64, 64, False), (64, 4096, 64, 32, False), (2, 256, 128, 64, False), (9, 512, 128, 32, False),   # 32 queries per wavefront forward
    (24, 2048, 64, 64, False), (2, 256, 64, 32, False),                                                         # and 16
    (64, 1024, 64, 64, True), (63, 1024, 64, 32, True), (12, 512, 64, 64, True), (9, 256, 64, 32, True)])       # under an element mask
def test_recomputed_probabilities_add_up_to_one(dtype, H, N, E, blk, elements, gpu):
    """The row statistic belongs to the scores that the row-side kernel works out again, also where these are large: with a
    column of ones in K, dP = T for every key and D = 0, that column of dQ is the sum of a query's probabilities."""
    mask = np.kron((np.arange(N // blk)[:, None] - np.arange(N // blk)) % (N // blk) < 4, np.ones((blk, blk), np.uint8)).astype(np.uint8)
    if elements:
        mask[:, ::3] = 0
    q, k, v = (randn((H, N, E), i, dtype)[1] for i in range(3))
    q = q * 8                   # scores / T of 8 or so
    k[..., 0] = 1
    att, (q, k, v) = build(mask, blk, blk, q, k, v, gpu)
    q, k, v = q.detach(), k.detach(), torch.zeros_like(v)
    assert att._recompute_supported(q) and (att._element_mask() is not None) == elements
    g = torch.zeros_like(q)
    g[..., 0] = v[..., 0] = 4   # dP / T = 16 / T
    out, lse = att._fused_forward_lse(q, k, v)
    grad_q, dot = att._recompute_backward_q(g, torch.zeros_like(out), q, k, v, lse, att._sparse_port.indexes, att._live_mask())
    assert float(dot.abs().max()) == 0.0
    sums = grad_q[..., 0].double() * (float(np.sqrt(E)) / 16)
    # dO / T, the score gradients and the result are rounded, by half of 2^-10 or 2^-7 at most each; 2^-20 for the fp32 sums
    bound = 3 * 2 ** (-11 if dtype == torch.float16 else -8) + 2 ** -20
    off = float((sums - 1).abs().max())
    assert off <= bound, f'{off:.2e} against {bound:.2e}'


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('H,N,E,bh,bw,elements', [
    (8, 512, 128, 64, 64, False), (9, 256, 128, 32, 32, False), (3, 512, 128, 64, 32, False), (9, 512, 64, 64, 64, True), (8, 256, 64, 32, 64, True)])
def test_gradients_where_scores_are_large(dtype, H, N, E, bh, bw, elements, gpu):
    """Scores of 8 or so, scaled in fp32 on both sides of the step: their size adds nothing to the errors."""
    mask = block_mask(N, N, bh, bw, 13)
    if elements:
        mask[:, ::3] = 0
    q, k, v, g = (randn((H, N, E), i, dtype)[1] for i in range(4))
    att, leaves = build(mask, bh, bw, q * 8, k, v, gpu)
    assert att._recompute_supported(leaves[0])
    check(step(att, leaves, g.to(gpu)), exact(leaves, g.to(gpu), torch.from_numpy(mask).to(gpu)), dtype, f'{dtype} {bh}x{bw} {E}')


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('bh,bw', [(128, 128), (128, 64), (64, 128)])
def test_large_scores_in_blocks_of_128(dtype, bh, bw, gpu, H=3, Nt=512, Ns=384, E=128):
    """Blocks that the library takes and the operator does not; the last ones scale to 16 bits on both sides."""
    from sparta_amd import _lib
    from sparta_amd.tesa import get_bcs_function
    mask = torch.from_numpy(block_mask(Nt, Ns, bh, bw, 17, density=0.7)).to(gpu)
    idx = get_bcs_function(bh, bw, True, True).build_indexes(mask)
    kernel = _lib.native().AttentionKernel(idx.row_ptr, idx._bcsr_buf, idx.col_ptr, idx._bcsc_buf, None, E ** -0.5, Nt, Ns, bh, bw)
    q, k, v, g = (randn(s, i, dtype)[1].to(gpu) for i, s in enumerate([(H, Nt, E), (H, Ns, E), (H, Ns, E), (H, Nt, E)]))
    if bw <= bh:
        q = q * 8
    out, lse = kernel.forward_lse(q, k, v)
    grad_q, dot = kernel.backward_q(g, out, q, k, v, lse)
    got = [t.double() for t in (grad_q, *kernel.backward_kv(g, q, k, v, lse, dot))]
    check(got, exact((q, k, v), g, mask), dtype, f'{dtype} {bh}x{bw}')


def test_element_mask_that_is_not_aligned(gpu, H=16, N=256):
    """The kernels that recompute the probabilities read 16 bytes of the mask at a time: a mask at an odd place stores them."""
    mask = np.tril(np.ones((N, N), np.uint8))
    q, k, v, g = (randn((H, N, 64), i, torch.bfloat16)[1] for i in range(4))
    att, leaves = build(mask, 64, 64, q, k, v, gpu)
    assert att._recompute_supported(leaves[0])
    odd = torch.zeros(N * N + 4, dtype=torch.uint8, device=gpu)[4:].view(N, N)
    odd.copy_(torch.from_numpy(mask))
    att.update_mask(odd)
    assert att._element_mask().data_ptr() % 16 == 4 and not att._recompute_supported(leaves[0])
    check(step(att, leaves, g.to(gpu)), exact(leaves, g.to(gpu), torch.from_numpy(mask).to(gpu)), torch.bfloat16, 'at an odd place')


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('H,Nt,Ns,bh,bw,elements', [
    (9, 256, 512, 32, 32, True), (9, 256, 512, 64, 64, True), (8, 256, 512, 64, 32, True),   # element masks; whole groups of 8 heads and not
    (2, 1024, 2112, 32, 32, True),                                                           # more than 64 entries to a block row
    (75, 512, 256, 64, 64, False), (74, 512, 256, 64, 32, False)])                           # 600 workgroups on the row side, and 592
def test_head_dim_128(dtype, H, Nt, Ns, bh, bw, elements, gpu, E=128):
    """Element masks: row side with 32 queries per wavefront, column side with 16 keys; partly live blocks, queries and keys
    without any, values other than one, large scores.  Block-level masks next to the size from which the row side changes."""
    rng = np.random.default_rng(19)
    mask = block_mask(Nt, Ns, bh, bw, 1, density=0.97 if Ns > 2048 else 0.4)
    if elements:
        mask *= (rng.random((Nt, Ns)) < 0.7).astype(np.uint8)
        mask[:, 5 * bw // 4:] |= np.tril(block_mask(Nt, Ns, bh, bw, 2))[:, 5 * bw // 4:]
        mask[bh + 3] = 0
        mask[:, 7] = 0
        mask[bh:, 40:60] *= 2
    q, k, v, g = (randn(s, i, dtype)[1] for i, s in enumerate([(H, Nt, E), (H, Ns, E), (H, Ns, E), (H, Nt, E)]))
    att, leaves = build(mask, bh, bw, q * 4, k, v, gpu)
    assert att._recompute_supported(leaves[0]) and (att._element_mask() is not None) == elements
    got = step(att, leaves, g.to(gpu))
    check(got, exact(leaves, g.to(gpu), torch.from_numpy(mask).to(gpu)), dtype, f'{dtype} {bh}x{bw}')
    if not elements:
        return
    assert float(got[0][:, bh + 3].abs().max()) == 0.0 and float(got[1][:, 7].abs().max()) == 0.0
    # the mask itself, and an index by column, at the C entry points
    from sparta_amd import _lib
    q, k, v, g = (t.detach() for t in (*leaves, g.to(gpu)))
    indexes, whole = att._sparse_port.indexes, att._element_mask()
    out, lse = att._fused_forward_lse(q, k, v)
    grad_q, dot = torch.empty_like(q), torch.empty_like(lse)
    lib, ptr, code = _lib.load(), _lib.dev_ptr, _lib.dtype_code(dtype)
    sizes = (float(att._inv_temperature), H, Nt, Ns, E, bh, bw, _lib.current_stream(gpu))
    _lib.check(lib.spx_attention_backward_q_masked(code, ptr(g), ptr(out), ptr(q), ptr(k), ptr(v), ptr(lse), ptr(grad_q), ptr(dot),
                                                   ptr(indexes.row_ptr), ptr(indexes._bcsr_buf), ptr(whole), *sizes), 'masked')
    assert torch.equal(grad_q.double(), got[0])
    by_column = indexes.function_context.__class__(bh, bw, False, True).build_indexes(whole)
    for data, call in ((whole, lib.spx_attention_backward_kv_masked), (by_column.convert(whole), lib.spx_attention_backward_kv_live_mask)):
        grad_k, grad_v = torch.empty_like(k), torch.empty_like(v)
        _lib.check(call(code, ptr(g), ptr(q), ptr(k), ptr(v), ptr(lse), ptr(dot), ptr(grad_k), ptr(grad_v), ptr(by_column.col_ptr),
                        ptr(by_column._bcsc_buf), _lib.IDX_BCSC_I32, ptr(data), *sizes), 'masked')
        assert torch.equal(grad_k.double(), got[1]) and torch.equal(grad_v.double(), got[2])
