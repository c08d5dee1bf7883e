"""GPU parity of the MoE path against the numpy oracle: the token->expert index
bit-exact (stable order), the gathered GEMM within tolerance.  Base case from the
reference's test/unit/test_sparse_moe.py (4096 tokens, 8 experts, 3072 -> 768,
fp16 and fp32, three routings), plus skewed routing, empty experts and ragged
token counts."""
import os

import numpy as np
import pytest
import torch

from oracle import ops
from sparta_amd.nn import DynamicSparseMoE
from helpers import assert_close, launched_kernels, template_numbers

pytestmark = pytest.mark.gpu
GOLD = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), 'golden', 'vectors.npz'))


def make_moe(n_exp, in_dims, out_dims, dtype, gpu, seed=2022, scale=0.05):
    rng = np.random.default_rng(seed)
    w = torch.from_numpy(rng.standard_normal((n_exp, out_dims, in_dims)).astype(np.float32) * scale).to(dtype)
    mods = []
    for e in range(n_exp):
        lin = torch.nn.Linear(in_dims, out_dims, bias=False, dtype=dtype, device=gpu)
        with torch.no_grad():
            lin.weight.copy_(w[e].to(gpu))
        mods.append(lin)
    weights_np = w.to(torch.float64).numpy().transpose(0, 2, 1)  # [E, in, out]
    return DynamicSparseMoE(mods), weights_np


def check_forward(moe, weights_np, n_tok, ids_np, dtype, gpu, seed):
    rng = np.random.default_rng(seed)
    data = torch.from_numpy(rng.random((n_tok, weights_np.shape[1]), dtype=np.float32)).to(dtype)
    out = moe(data.to(gpu), torch.from_numpy(ids_np).to(gpu))
    count, offset, perm = ops.moe_index_reference(ids_np, weights_np.shape[0])
    assert np.array_equal(moe.expert_count.cpu().numpy(), count)
    assert np.array_equal(moe.expert_offset.cpu().numpy(), offset)
    assert np.array_equal(moe.sparse_index[:n_tok].cpu().numpy(), perm)
    want = ops.moe_reference(data.to(torch.float64).numpy(), weights_np, ids_np)
    assert out.dtype == dtype and tuple(out.shape) == want.shape
    assert_close(out, want, dtype, f'moe {dtype} n_tok={n_tok}')


@pytest.mark.parametrize('dtype', [torch.float16, torch.float32, torch.bfloat16])
def test_moe_reference_case(dtype, gpu):
    moe, w = make_moe(8, 3072, 768, dtype, gpu)
    for seed in range(3):  # dynamic routing: a new assignment every call
        ids = np.random.default_rng(seed).integers(0, 8, 4096).astype(np.int32)
        check_forward(moe, w, 4096, ids, dtype, gpu, seed)


def test_moe_zipf_skew_exceeds_reference_capacity(gpu):
    """Zipf(1.2) routing: the busiest expert gets more than the 4096-token capacity
    the reference hard-codes (sparse_moe.py:23)."""
    n_tok, n_exp = 16384, 8
    p = np.arange(1, n_exp + 1, dtype=np.float64) ** -1.2
    ids = np.random.default_rng(2022).choice(n_exp, size=n_tok, p=p / p.sum()).astype(np.int32)
    assert np.bincount(ids).max() > 4096
    moe, w = make_moe(n_exp, 256, 512, torch.float16, gpu)
    check_forward(moe, w, n_tok, ids, torch.float16, gpu, 1)


@pytest.mark.parametrize('n_tok', [1, 100, 1000, 1025, 3000])
def test_moe_ragged_token_counts_and_empty_experts(n_tok, gpu):
    n_exp = 6
    moe, w = make_moe(n_exp, 128, 136, torch.float16, gpu)
    ids = np.random.default_rng(n_tok).choice([0, 2, 5], size=n_tok).astype(np.int32)  # experts 1,3,4 stay empty
    check_forward(moe, w, n_tok, ids, torch.float16, gpu, 2)


def test_moe_single_expert_is_one_gemm(gpu):
    moe, w = make_moe(1, 256, 256, torch.float32, gpu)
    check_forward(moe, w, 512, np.zeros(512, dtype=np.int32), torch.float32, gpu, 3)


def test_moe_many_experts(gpu):
    n_exp = 200
    moe, w = make_moe(n_exp, 64, 64, torch.float16, gpu, scale=0.1)
    ids = np.random.default_rng(7).integers(0, n_exp, 5000).astype(np.int32)
    check_forward(moe, w, 5000, ids, torch.float16, gpu, 4)


def test_moe_golden_vectors(gpu):
    tokens, weights, ids = GOLD['moe_tokens'], GOLD['moe_weights'], GOLD['moe_ids']
    mods = []
    for e in range(weights.shape[0]):
        lin = torch.nn.Linear(64, 48, bias=False, dtype=torch.float16, device=gpu)
        with torch.no_grad():
            lin.weight.copy_(torch.from_numpy(weights[e].T.copy()).to(gpu))
        mods.append(lin)
    moe = DynamicSparseMoE(mods)
    out = moe(torch.from_numpy(tokens).half().to(gpu), torch.from_numpy(ids).to(gpu))
    assert np.array_equal(moe.sparse_index[:96].cpu().numpy(), GOLD['moe_perm'])
    assert np.array_equal(moe.expert_offset.cpu().numpy(), GOLD['moe_offset'])
    assert_close(out, GOLD['moe_out'], torch.float16, 'moe golden')

@pytest.mark.parametrize('n_tok,n_exp', [
    (700, 3),          # 256-token chunks, count table scanned by the placement workgroups
    (16384, 8),        # 64 chunks x 9 counts
    (50000, 8),        # 512-token chunks
    (100000, 8),       # 1024-token chunks, still within the 1024-entry table
    (4096, 200),       # many experts: 1024-token chunks, 4 x 201 counts
    (200000, 8),       # table too large: separate scan launch
    (30000, 200),      # separate scan launch, many experts
    (257, 1),
])
def test_moe_index_launch_paths(n_tok, n_exp, gpu):
    """spx_moe_index through the C ABI on routings that take every chunk size of the
    two-launch path and the three-launch path, ids outside [0, n_exp) included: counts,
    offsets and the stable permutation are bit-exact against the oracle."""
    from sparta_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(n_tok + n_exp)
    p = np.arange(1, n_exp + 1, dtype=np.float64) ** -1.2
    ids_np = rng.choice(n_exp, size=n_tok, p=p / p.sum()).astype(np.int32)
    bad = rng.random(n_tok) < 0.01
    ids_np[bad] = rng.choice([-3, n_exp, n_exp + 7], size=int(bad.sum()))
    ids = torch.from_numpy(ids_np).to(gpu)
    count = torch.full((n_exp,), -1, dtype=torch.int32, device=gpu)
    offset = torch.full((n_exp + 1,), -1, dtype=torch.int32, device=gpu)
    perm = torch.full((n_tok,), -1, dtype=torch.int32, device=gpu)
    ws = torch.empty(max(lib.spx_moe_index_workspace_bytes(n_tok, n_exp), 256), dtype=torch.uint8, device=gpu)
    for _ in range(2):  # the workspace is reused as it was left
        _lib.check(lib.spx_moe_index(_lib.dev_ptr(ids), n_tok, n_exp, _lib.dev_ptr(count), _lib.dev_ptr(offset),
                                     _lib.dev_ptr(perm), _lib.dev_ptr(ws), ws.numel(), _lib.current_stream(gpu)),
                   'spx_moe_index')
    valid = (ids_np >= 0) & (ids_np < n_exp)
    key = np.where(valid, ids_np, n_exp)                  # out-of-range ids sort behind every expert
    want_count = np.bincount(key, minlength=n_exp + 1)[:n_exp].astype(np.int32)
    want_offset = np.zeros(n_exp + 1, dtype=np.int32)
    np.cumsum(want_count, out=want_offset[1:])
    want_perm = np.argsort(key, kind='stable').astype(np.int32)
    c2, o2, p2 = ops.moe_index_reference(ids_np[valid], n_exp)
    assert np.array_equal(want_count, c2) and np.array_equal(want_offset, o2)   # the oracle on the valid ids
    assert np.array_equal(count.cpu().numpy(), want_count)
    assert np.array_equal(offset.cpu().numpy(), want_offset)
    assert np.array_equal(perm.cpu().numpy(), want_perm)
    assert np.array_equal(np.flatnonzero(valid)[p2], want_perm[:int(valid.sum())])


def test_moe_weight_layouts_agree(gpu):
    """The [E, in, out] layout of the reference's stacked weight (what the operator feeds
    the kernels) gives the same result as an [E, out, in] copy of it."""
    from sparta_amd import _lib
    moe, w = make_moe(4, 128, 256, torch.float16, gpu)
    ids = torch.from_numpy(np.random.default_rng(0).integers(0, 4, 700).astype(np.int32)).to(gpu)
    x = torch.rand((700, 128), dtype=torch.float16, device=gpu)
    want = moe(x, ids)
    out = torch.empty_like(want)
    w_nk = moe.weight.detach().transpose(1, 2).contiguous()
    rc = _lib.load().spx_moe_forward(_lib.F16, _lib.dev_ptr(x), _lib.dev_ptr(w_nk), 1,
                                     _lib.dev_ptr(out), _lib.dev_ptr(moe.expert_offset),
                                     _lib.dev_ptr(moe.sparse_index), 700, 128, 256, 4, 0,
                                     _lib.current_stream(gpu))
    _lib.check(rc, 'spx_moe_forward')
    assert torch.equal(out, want)


def test_moe_follows_in_place_weight_updates(gpu):
    """The operator reads its stacked parameter at every call: writes through `.data`
    (which do not advance the version counter), `.half()` and optimizer-style updates
    all show up in the next forward."""
    moe, w = make_moe(3, 128, 136, torch.float32, gpu)
    ids_np = np.random.default_rng(3).integers(0, 3, 300).astype(np.int32)
    check_forward(moe, w, 300, ids_np, torch.float32, gpu, 5)
    with torch.no_grad():
        moe.weight.data.mul_(-0.5)
        moe.weight.data[1].add_(0.25)
    w2 = w * -0.5
    w2[1] += 0.25
    check_forward(moe, w2, 300, ids_np, torch.float32, gpu, 6)
    moe.half()
    w3 = moe.weight.detach().to(torch.float64).cpu().numpy()
    check_forward(moe, w3, 300, ids_np, torch.float16, gpu, 7)


def test_moe_out_of_range_ids_give_zero_rows(gpu):
    """Tokens whose expert id is negative or >= n_exp (the reference indexes out of bounds
    for them) get zero output rows and are listed, ascending, behind the routed tokens."""
    n_exp, n_tok = 4, 1000
    moe, w = make_moe(n_exp, 128, 256, torch.float16, gpu)
    rng = np.random.default_rng(11)
    ids_np = rng.integers(0, n_exp, n_tok).astype(np.int32)
    bad = rng.choice(n_tok, 77, replace=False)
    ids_np[bad[:40]] = -3
    ids_np[bad[40:]] = n_exp + 2
    data = torch.from_numpy(rng.random((n_tok, 128), dtype=np.float32)).half()
    out = torch.full((n_tok, 256), float('nan'), dtype=torch.float16, device=gpu)
    got = moe(data.to(gpu), torch.from_numpy(ids_np).to(gpu))
    valid = (ids_np >= 0) & (ids_np < n_exp)
    want = np.zeros((n_tok, 256))
    want[valid] = ops.moe_reference(data.to(torch.float64).numpy()[valid], w, ids_np[valid])
    assert_close(got, want, torch.float16, 'moe with out-of-range ids')
    assert float(got[torch.from_numpy(~valid).to(gpu)].abs().max()) == 0.0
    offset = moe.expert_offset.cpu().numpy()
    assert offset[n_exp] == valid.sum()
    assert np.array_equal(moe.sparse_index[offset[n_exp]:n_tok].cpu().numpy(), np.sort(bad))


@pytest.mark.parametrize('layout', [0, 1])
@pytest.mark.parametrize('tile_cfg', [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize('dtype,n_tok,in_dims,out_dims', [
    (torch.float16, 3000, 256, 520), (torch.bfloat16, 1500, 128, 256), (torch.float32, 700, 96, 136),
    (torch.float16, 5, 64, 64), (torch.float16, 2500, 192, 776)])
def test_moe_tile_configs(layout, tile_cfg, dtype, n_tok, in_dims, out_dims, gpu):
    """Every gathered-GEMM variant through the C ABI, in both weight layouts, on the same
    routing (one stage, two stages and more; ragged last tiles in both directions; an
    empty expert)."""
    from sparta_amd import _lib
    if dtype == torch.float32 and layout == 0 and tile_cfg != 1:
        pytest.skip('fp32 weights stored [E, in, out] run through tile config 1')
    if dtype == torch.float32 and tile_cfg == 6:
        pytest.skip('the cross-stage pipelined configuration takes 16-bit types')
    n_exp = 5
    moe, w = make_moe(n_exp, in_dims, out_dims, dtype, gpu)
    ids_np = np.random.default_rng(n_tok).choice([0, 1, 2, 4], size=n_tok, p=[0.6, 0.2, 0.15, 0.05]).astype(np.int32)
    x = torch.from_numpy(np.random.default_rng(1).random((n_tok, in_dims), dtype=np.float32)).to(dtype)
    xg = x.to(gpu)
    moe(xg, torch.from_numpy(ids_np).to(gpu))  # builds the index
    weight = moe.weight.detach() if layout == 0 else moe.weight.detach().transpose(1, 2).contiguous()
    out = torch.full((n_tok, out_dims), float('nan'), dtype=dtype, device=gpu)
    rc = _lib.load().spx_moe_forward(_lib.dtype_code(dtype), _lib.dev_ptr(xg), _lib.dev_ptr(weight), layout,
                                     _lib.dev_ptr(out), _lib.dev_ptr(moe.expert_offset),
                                     _lib.dev_ptr(moe.sparse_index), n_tok, in_dims, out_dims, n_exp, tile_cfg,
                                     _lib.current_stream(gpu))
    _lib.check(rc, 'spx_moe_forward')
    want = ops.moe_reference(x.to(torch.float64).numpy(), w, ids_np)
    assert_close(out, want, dtype, f'moe tile config {tile_cfg} layout {layout} {dtype}')


@pytest.mark.parametrize('layout', [0, 1])
@pytest.mark.parametrize('dtype,n_tok,in_dims,out_dims,n_exp', [
    # 256 workgroups.  No whole round: quarters of a tile, halves (15 tiles to an XCD), whole ones; the shortest k (four stages)
    (torch.float16, 300, 256, 264, 3), (torch.bfloat16, 5000, 320, 1032, 5), (torch.float16, 9000, 256, 1288, 3),
    # whole rounds and a rest; more experts than lanes; a strip that is not full
    (torch.bfloat16, 20000, 576, 1544, 4), (torch.float16, 17000, 256, 1032, 70), (torch.float16, 1, 256, 8, 2)])
def test_moe_persistent_tiles(layout, dtype, n_tok, in_dims, out_dims, n_exp, gpu):
    """Tile config 5 through the C ABI: every cut of the last round, experts that end inside a tile and inside a half of one, an
    empty expert, tokens without one, and a token of NaN that reaches no other row.  A single token is finite."""
    from sparta_amd import _lib
    moe, w = make_moe(n_exp, in_dims, out_dims, dtype, gpu)
    rng = np.random.default_rng(n_tok)
    share = np.r_[np.arange(1, n_exp + 1, dtype=np.float64) ** -0.8, 0.05]   # id n_exp: no expert
    share[n_exp // 2] = 0.0
    ids_np = rng.choice(n_exp + 1, size=n_tok, p=share / share.sum()).astype(np.int32)
    x = torch.from_numpy(rng.random((n_tok, in_dims), dtype=np.float32)).to(dtype)
    xg, bad = x.to(gpu), np.arange(n_tok) == (n_tok - 1 if n_tok > 1 else -1)
    ids_np[-1] = 0
    xg[torch.from_numpy(bad).to(gpu)] = float('nan')
    moe(xg, torch.from_numpy(ids_np).to(gpu))  # builds the index
    weight = moe.weight.detach() if layout == 0 else moe.weight.detach().transpose(1, 2).contiguous()
    out = torch.full((n_tok, out_dims), float('nan'), dtype=dtype, device=gpu)
    out[torch.from_numpy(bad).to(gpu)] = 7.0   # (a row that nobody writes is not NaN)

    def call():
        _lib.check(_lib.load().spx_moe_forward(_lib.dtype_code(dtype), _lib.dev_ptr(xg), _lib.dev_ptr(weight), layout, _lib.dev_ptr(out),
                                               _lib.dev_ptr(moe.expert_offset), _lib.dev_ptr(moe.sparse_index), n_tok, in_dims, out_dims,
                                               n_exp, 5, _lib.current_stream(gpu)), 'spx_moe_forward')

    _, names = launched_kernels(call)
    assert any('moe_persist_kernel' in n for n in names), names
    rows = ~bad
    assert bool(torch.isnan(out[torch.from_numpy(bad).to(gpu)]).all())
    want = ops.moe_reference(x.to(torch.float64).numpy(), np.concatenate([w, np.zeros_like(w[:1])]), ids_np)
    assert_close(out[torch.from_numpy(rows).to(gpu)], want[rows], dtype, f'persistent moe {n_tok} x {in_dims} -> {out_dims} over {n_exp}')


def test_moe_persistent_tiles_of_a_large_layer(gpu, n_tok=131072, in_dims=256, out_dims=8192, n_exp=8):
    """16640 tiles and more, 66 to a workgroup, through the library's own choice."""
    moe, w = make_moe(n_exp, in_dims, out_dims, torch.float16, gpu)
    rng = np.random.default_rng(5)
    ids_np = rng.choice(n_exp, size=n_tok, p=np.arange(1, n_exp + 1) / (n_exp * (n_exp + 1) / 2)).astype(np.int32)
    x = torch.from_numpy(rng.random((n_tok, in_dims), dtype=np.float32)).half()
    x_dev, ids = x.to(gpu), torch.from_numpy(ids_np).to(gpu)
    got, names = launched_kernels(lambda: moe(x_dev, ids))
    assert any('moe_persist_kernel' in n for n in names), names
    weight = moe.weight.detach().float()   # [E, in, out]
    for e in range(n_exp):
        rows = torch.nonzero(ids == e).flatten()
        for r in range(0, rows.numel(), 8192):
            some = rows[r:r + 8192]
            want = torch.matmul(x_dev[some].float(), weight[e])
            # result rounded to 11 bits; fp32 sums of 256 products in another order
            assert float((got[some].float() - want).abs().max()) <= 2 ** -11 * float(want.abs().max()) + 1e-4


@pytest.mark.parametrize('n_exp', [1, 2, 7, 8, 63, 64, 900])
@pytest.mark.parametrize('n_tok', [1, 255, 1025, 2049, 4095, 4096, 4097, 20000])
def test_moe_index_orders_tokens(n_tok, n_exp, gpu):
    """Counted by the placement workgroups and by a launch of their own, every number of bits to an expert, with ids that
    are out of range on both sides: what a stable sort by expert gives, to the last token."""
    from sparta_amd import _lib
    lib = _lib.load()
    ids = np.random.default_rng(n_tok + n_exp).integers(-1, n_exp + 2, n_tok).astype(np.int32)
    key = np.where((ids < 0) | (ids >= n_exp), n_exp, ids)
    on = lambda n: torch.full((n,), -1, dtype=torch.int32, device=gpu)
    dev_ids, count, offset, perm = torch.from_numpy(ids).to(gpu), on(n_exp), on(n_exp + 1), on(n_tok)
    nbytes = lib.spx_moe_index_workspace_bytes(n_tok, n_exp)
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device=gpu)
    _lib.check(lib.spx_moe_index(_lib.dev_ptr(dev_ids), n_tok, n_exp, _lib.dev_ptr(count), _lib.dev_ptr(offset), _lib.dev_ptr(perm),
                                 _lib.dev_ptr(ws), nbytes, _lib.current_stream(gpu)), 'spx_moe_index')
    want = np.bincount(key, minlength=n_exp + 1)
    assert np.array_equal(perm.cpu().numpy(), np.argsort(key, kind='stable'))
    assert np.array_equal(count.cpu().numpy(), want[:n_exp])
    assert np.array_equal(offset.cpu().numpy(), np.cumsum(want) - want)


@pytest.mark.parametrize('n_tok,n_exp,single', [(4097, 5, True), (12289, 63, True), (20480, 8, True), (20480, 64, False), (20481, 8, False)])
def test_moe_index_in_one_launch(n_tok, n_exp, single, gpu):
    """Both sides of the lines up to which one launch counts and places the tokens, nearly all of them with one expert (whose
    counters every lane of a wavefront adds to), ids out of range among them: a stable sort, to the last token."""
    from sparta_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(n_tok + n_exp)
    ids = np.where(rng.random(n_tok) < 0.95, n_exp - 1, rng.integers(-2, n_exp + 2, n_tok)).astype(np.int32)
    on = lambda n: torch.full((n,), -1, dtype=torch.int32, device=gpu)
    dev_ids, count, offset, perm = torch.from_numpy(ids).to(gpu), on(n_exp), on(n_exp + 1), on(n_tok)
    nbytes = lib.spx_moe_index_workspace_bytes(n_tok, n_exp)
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device=gpu)
    _, names = launched_kernels(lambda: _lib.check(lib.spx_moe_index(
        _lib.dev_ptr(dev_ids), n_tok, n_exp, _lib.dev_ptr(count), _lib.dev_ptr(offset), _lib.dev_ptr(perm), _lib.dev_ptr(ws),
        nbytes, _lib.current_stream(gpu)), 'spx_moe_index'))
    assert any('moe_index_kernel' in n for n in names) == single, names
    key = np.where((ids < 0) | (ids >= n_exp), n_exp, ids)
    want = np.bincount(key, minlength=n_exp + 1)
    assert np.array_equal(perm.cpu().numpy(), np.argsort(key, kind='stable'))
    assert np.array_equal(count.cpu().numpy(), want[:n_exp])
    assert np.array_equal(offset.cpu().numpy(), np.cumsum(want) - want)


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('n_tok,in_dims,out_dims,n_exp,rows,stages', [
    # behind the 32-row tiles (256 of 128 x 128): 64-row tiles in three stages, up to 288 of 128 x 128; one stage of k, ragged columns
    (1, 64, 4616, 8, 32, 0), (1, 64, 16520, 8, 64, 3), (512, 64, 3000, 8, 64, 3), (512, 64, 3080, 8, 128, 2),
    # ... with more than 128 rows to an expert, up to 224
    (520, 192, 776, 4, 64, 3), (1600, 256, 776, 4, 64, 3), (1600, 256, 1640, 4, 64, 3), (1600, 256, 1672, 4, 128, 2),
    # both sides of 48 rows to an expert and of 1024 of 128 x 128: 64-row tiles in two stages, 128-row tiles
    (767, 128, 4096, 16, 64, 2), (769, 320, 4096, 16, 128, 2), (767, 64, 5888, 16, 64, 2), (767, 64, 5896, 16, 128, 2),
    # 256-row tiles that fit a round, whose unused halves fit one, and do not
    (13000, 64, 768, 8, 256, 2), (4200, 128, 2056, 16, 256, 2), (4200, 128, 2312, 16, 128, 2)])
def test_moe_dispatch(dtype, n_tok, in_dims, out_dims, n_exp, rows, stages, gpu):
    """Tile height and stages at the sizes at which the library's own choice of tiles changes, with an empty expert and a crowded one."""
    moe, w = make_moe(n_exp, in_dims, out_dims, dtype, gpu)
    p = np.ones(n_exp)
    p[0], p[1] = 0.0, 3.0
    ids_np = np.random.default_rng(n_tok).choice(n_exp, size=n_tok, p=p / p.sum()).astype(np.int32)
    x = torch.from_numpy(np.random.default_rng(1).random((n_tok, in_dims), dtype=np.float32)).to(dtype)
    x_dev, ids = x.to(gpu), torch.from_numpy(ids_np).to(gpu)
    got, names = launched_kernels(lambda: moe(x_dev, ids))
    tiles = [(n[0], n[4]) for n in template_numbers(names, 'moe_gemm_direct_kernel')]   # rows, columns, wavefronts, .., stages
    assert tiles == ([] if rows == 32 else [(rows, stages)]) and any('moe_rows_kernel' in n for n in names) == (rows == 32), names
    assert_close(got, ops.moe_reference(x.to(torch.float64).numpy(), w, ids_np), dtype, f'moe {n_tok} x {in_dims} -> {out_dims} over {n_exp}')


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
@pytest.mark.parametrize('n_tok,in_dims,out_dims', [(1, 64, 8), (5, 64, 520), (33, 192, 136), (64, 128, 128), (300, 2048, 264)])
def test_moe_few_rows_kernel(dtype, n_tok, in_dims, out_dims, gpu):
    """Tile config 7 through the C ABI: fewer k-stages than wavefronts and more, rows that end inside a tile,
    several row tiles to an expert, columns that end inside a tile, tokens without an expert, and a
    token of NaN that reaches no other row."""
    from sparta_amd import _lib
    n_exp = 5
    moe, w = make_moe(n_exp, in_dims, out_dims, dtype, gpu)
    rng = np.random.default_rng(n_tok)
    ids_np = rng.choice([0, 1, 2, 4, 7], size=n_tok, p=[0.6, 0.2, 0.1, 0.05, 0.05]).astype(np.int32)
    x = torch.from_numpy(rng.random((n_tok, in_dims), dtype=np.float32)).to(dtype)
    bad = n_tok - 1 if n_tok > 1 else None
    if bad is not None:
        ids_np[bad] = 0
    xg = x.to(gpu)
    if bad is not None:
        xg[bad] = float('nan')
    moe(xg, torch.from_numpy(ids_np).to(gpu))  # builds the index
    out = torch.full((n_tok, out_dims), float('nan'), dtype=dtype, device=gpu)
    rc = _lib.load().spx_moe_forward(_lib.dtype_code(dtype), _lib.dev_ptr(xg), _lib.dev_ptr(moe.weight.detach()), 0,
                                     _lib.dev_ptr(out), _lib.dev_ptr(moe.expert_offset), _lib.dev_ptr(moe.sparse_index),
                                     n_tok, in_dims, out_dims, n_exp, 7, _lib.current_stream(gpu))
    _lib.check(rc, 'spx_moe_forward')
    valid = ids_np < n_exp
    want = np.zeros((n_tok, out_dims))
    if valid.any():
        want[valid] = ops.moe_reference(x.to(torch.float64).numpy()[valid], w, ids_np[valid])
    rows = np.arange(n_tok) != (-1 if bad is None else bad)
    assert_close(out[torch.from_numpy(rows).to(gpu)], want[rows], dtype, f'moe few-row kernel {dtype} {(n_tok, in_dims, out_dims)}')
    if bad is not None:
        assert bool(torch.isnan(out[bad]).all())
    rc = _lib.load().spx_moe_forward(_lib.dtype_code(dtype), _lib.dev_ptr(xg), _lib.dev_ptr(moe.weight.detach()), 1,
                                     _lib.dev_ptr(out), _lib.dev_ptr(moe.expert_offset), _lib.dev_ptr(moe.sparse_index),
                                     n_tok, in_dims, out_dims, n_exp, 7, _lib.current_stream(gpu))
    assert rc != 0   # [E, out, in] weights are refused


@pytest.mark.parametrize('n_tok,n_exp', [(1, 3), (255, 1000), (1024, 8), (1024, 200), (1025, 8)])
def test_moe_index_of_few_tokens(n_tok, n_exp, gpu):
    """Around the token count up to which the placement workgroups count the experts themselves."""
    test_moe_index_launch_paths(n_tok, n_exp, gpu)
