"""Shared helpers of the GPU parity tests: seeded CPU inputs (so the oracle and
the HIP path see identical bits) and tolerance tables."""
import re
from typing import NamedTuple

import numpy as np
import torch

# 1e-2 (rtol and atol) for 16-bit outputs, 1e-4 for fp32
TOL = {torch.float32: dict(rtol=1e-4, atol=1e-4),
       torch.float16: dict(rtol=1e-2, atol=1e-2),
       torch.bfloat16: dict(rtol=1e-2, atol=1e-2)}


def rng(seed):
    return np.random.default_rng(seed)


def randn(shape, seed, dtype=torch.float32, scale=1.0):
    """N(0, scale^2) values rounded to `dtype`; returns (numpy float64 of the rounded
    values, torch tensor on CPU in dtype)."""
    t = torch.from_numpy(rng(seed).standard_normal(shape).astype(np.float32) * scale).to(dtype)
    return t.to(torch.float64).numpy(), t


def rand(shape, seed, dtype=torch.float32):
    t = torch.from_numpy(rng(seed).random(shape, dtype=np.float32)).to(dtype)
    return t.to(torch.float64).numpy(), t


def assert_close(got: torch.Tensor, want: np.ndarray, dtype, what='', scale=1.0):
    tol = TOL[dtype]
    g = got.detach().to(torch.float64).cpu().numpy()
    err = np.abs(g - want)
    bound = tol['atol'] * scale + tol['rtol'] * np.abs(want)
    bad = ~(err <= bound)   # NaN counts as off
    assert not bad.any(), (f'{what}: {bad.sum()} of {bad.size} entries off, max err {err.max():.3e} '
                           f'(bound there {bound.flat[err.argmax()]:.3e})')


def chained_sum_error(additions):
    """Relative error (2-norm) of fp32 sums of products of N(0, 1) values that are added up in chains of so many additions.
    A rounded addition is off by 2^-23 / sqrt(12) of its sum's power of two, 0.41 * 2^-24 of the sum (rms, mantissas evenly
    spread over 1 to 2), and the sums of a chain grow like the root of the additions before them."""
    return 0.41 * 2.0 ** -24 * (additions / 2) ** 0.5


# Ring kernel: (rows of a tile, M) of products K -> N with an activation, and whether their results are written through: more rows
# and fewer, panels in one part, in two and in eight
RESULTS_K_N = (192, 544)
RESULTS_THROUGH = {(64, 1024): 0, (64, 2200): 0, (64, 1090): 0, (64, 65): 0, (64, 5120): 0, (64, 5130): 1, (64, 6100): 1,
                   (128, 1024): 0, (128, 2200): 0, (128, 65): 0, (128, 5130): 0, (128, 5600): 1, (128, 6100): 1}


def launched_kernels(call):
    """(what `call` returns, names of the kernels that it launched; they may be mangled)."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        result = call()
        torch.cuda.synchronize()
    return result, [event.name for event in prof.events()]


def template_numbers(names, kernel):
    """The numbers among the template arguments (truth values as 0 and 1) of every launch of `kernel` in `names`."""
    found = []
    for name in names:
        mangled = re.search(kernel + r'I(.*)', name)
        plain = re.search(kernel + r'<([^>]*)>', name)
        if plain:
            args = plain.group(1).replace('true', '1').replace('false', '0').split(', ')
            found.append(tuple(int(a) for a in args if a.isdigit()))
        elif mangled:
            found.append(tuple(map(int, re.findall(r'L[ib](\d+)E', mangled.group(1)))))
    return found


class SeqlenInstance(NamedTuple):
    head_dim: int
    stage: int     # keys to a stage
    shares: int    # wavefronts that share the keys of 32 queries


def seqlen_instance(names):
    """The instance of the sequence-length kernel with 32 queries to a wavefront among the kernels launched; None: there is none."""
    # head dim, tiles of 32 keys to a stage, wavefronts, element mask, sequence lengths, shares
    found = [SeqlenInstance(n[0], 32 * n[1], n[5]) for n in template_numbers(names, 'attention_wide_kernel') if n[4]]
    assert len(found) <= 1, names
    return found[0] if found else None
