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
