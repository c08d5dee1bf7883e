"""Sequence-length attention where its work is dealt out longest entry first: entries in groups of 64,
pairs of (entry, head) over eight XCDs, query blocks without a position at the end."""
import numpy as np
import pytest
import torch

from sparta_amd.nn import SeqlenDynamicSparseAttention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('E', [64, 128])
@pytest.mark.parametrize('batch,heads,N,lens', [
    (65, 3, 256, 'mixed'),      # a second group with one entry
    (70, 5, 288, 'mixed'),      # N is no multiple of the 128 queries of a workgroup
    (64, 6, 256, 'none'),       # nothing but zeros
    (64, 6, 256, 'full'),
    (48, 8, 256, 'one'),        # one position each, one entry that is full
    (3, 16, 992, 'mixed'),
    (130, 3, 256, 'clamped'),   # lengths below 0 and above N
])
def test_longest_first(batch, heads, N, lens, E, gpu):
    assert batch * heads * ((N + 127) // 128) >= 384   # the kernel with 32 queries to a wavefront takes it
    check(batch, heads, N, lens, E, gpu)


@pytest.mark.parametrize('E', [64, 128])
@pytest.mark.parametrize('batch,heads,N,lens', [
    (2, 16, 992, 'mixed'), (1, 3, 928, 'full'),   # stages of 128 keys with head dim 64; N no multiple of a stage
    (7, 12, 320, 'edges'), (24, 8, 256, 'edges'), # and of 64; lengths that end in the first or second share of a stage, or leave one out
    (8, 16, 192, 'mixed'), (48, 8, 192, 'edges'),
    (3, 8, 1056, 'clamped'), (33, 5, 288, 'one'),
    (768, 1, 96, 'mixed'), (767, 1, 224, 'mixed'),
    (16, 8, 1024, 'mixed'), (19, 9, 768, 'mixed')])   # 1024 workgroups of 128 queries, and 1026
def test_shared_keys(batch, heads, N, lens, E, gpu):
    """Both sides of the sizes at which two wavefronts share the keys of their queries out."""
    check(batch, heads, N, lens, E, gpu)


def check(batch, heads, N, lens, E, gpu):
    rng = np.random.default_rng(11)
    n = {'mixed': rng.integers(0, N + 1, batch), 'none': np.zeros(batch, int), 'full': np.full(batch, N),
         'one': np.ones(batch, int), 'clamped': rng.integers(-N, 2 * N, batch),
         'edges': np.resize([1, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 160, 192], batch)}[lens]
    if lens == 'one':
        n[5] = N
    g = torch.Generator(device=gpu).manual_seed(3)
    q, k, v = (torch.randn((batch, heads, N, E), generator=g, device=gpu).half() for _ in range(3))
    q = q / E ** 0.5
    got = SeqlenDynamicSparseAttention(global_mode=False)(q, k, v, torch.from_numpy(n.astype(np.int32)).to(gpu)).float()
    for b in range(batch):
        m = int(min(max(n[b], 0), N))
        assert float(got[b, :, m:].abs().max()) == 0.0 if m < N else True
        if m:
            s = torch.matmul(q[b, :, :m].float(), k[b, :, :m].float().transpose(1, 2).contiguous())
            want = torch.matmul(torch.softmax(s, -1), v[b, :, :m].float())
            # probabilities and result rounded to 11 bits, 2^-12 of the value each at most
            rel = float((got[b, :, :m] - want).norm() / want.norm())
            assert rel <= 1e-3, f'entry {b} of length {m}: {rel:.2e}'


@pytest.mark.parametrize('E', [64, 128])
@pytest.mark.parametrize('batch', [8, 11, 32])   # shared keys, stages of 128 (head dim 64) and of 64; not shared
def test_nan_stays_in_its_rows(batch, E, gpu, heads=12, N=320, n=200):
    """A query or key that is NaN makes its own row or all rows of its head NaN; past the length it makes nothing."""
    g = torch.Generator(device=gpu).manual_seed(4)
    q, k, v = (torch.randn((batch, heads, N, E), generator=g, device=gpu).half() for _ in range(3))
    q = q / E ** 0.5
    op = SeqlenDynamicSparseAttention(global_mode=False)
    lens = torch.full((batch,), n, dtype=torch.int32, device=gpu)
    want = op(q, k, v, lens)
    q[0, 1, 7] = q[0, 1, n] = k[1, 2, 150] = k[1, 3, n] = v[1, 4, n + 7] = float('nan')
    got = op(q, k, v, lens)
    bad = torch.zeros((batch, heads, N), dtype=torch.bool, device=gpu)
    bad[0, 1, 7] = True
    bad[1, 2, :n] = True
    assert bool(got[bad].isnan().all())
    # other rows of its wavefront may move their reference point with it: probabilities and result rounded to 11 bits, twice
    assert float((got[~bad].float() - want[~bad].float()).abs().max()) <= 2 ** -9 * float(v.nan_to_num().abs().max())
