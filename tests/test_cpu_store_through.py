"""The store that writes results through the L2s (csrc/common.hpp), compiled here for gfx950 behind MFMAs: the registers that an
MFMA writes are not ready for some clocks, and nothing but wait states in the code keeps a store from reading them before.
They have to be those that the compiler puts in front of a plain store.  No GPU."""
import re
import subprocess

import pytest

from sparta_amd import build

_SOURCE = '''
#include "common.hpp"
using namespace spx;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
template <bool THROUGH, bool HALF>
__global__ void results_of_mfmas(float* out, const float* a, const f16x8_t* h) {
    const float x = a[threadIdx.x];
    const f16x8_t y = h[threadIdx.x];
    float* const to = out + threadIdx.x * 4;
    f32x4_t acc = *reinterpret_cast<f32x4_t*>(to);   // (so that the address is ready before the MFMAs)
    for (int i = 0; i < 2; ++i) {
        if constexpr (HALF) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(y, y, acc, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x, x, acc, 0, 0, 0);
    }
    if constexpr (THROUGH) store16_through(to, __builtin_bit_cast(vec16, acc));
    else *reinterpret_cast<f32x4_t*>(to) = acc;
}
template __global__ void results_of_mfmas<false, false>(float*, const float*, const f16x8_t*);
template __global__ void results_of_mfmas<false, true>(float*, const float*, const f16x8_t*);
template __global__ void results_of_mfmas<true, false>(float*, const float*, const f16x8_t*);
template __global__ void results_of_mfmas<true, true>(float*, const float*, const f16x8_t*);
'''


@pytest.fixture(scope='module')
def listing(tmp_path_factory):
    tmp = tmp_path_factory.mktemp('through')
    (tmp / 'probe.hip').write_text(_SOURCE)
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, '-I', build.CSRC, '--cuda-device-only', '-S', str(tmp / 'probe.hip'), '-o',
                    str(tmp / 'probe.s')], check=True, capture_output=True)
    return (tmp / 'probe.s').read_text()


def _store_behind_mfma(listing, through, half):
    """(wait states between the last MFMA and the store, the store) of a kernel."""
    name = f'_Z16results_of_mfmasILb{int(through)}ELb{int(half)}EEv'
    body = re.search(rf'^{name}\w*:.*?s_endpgm', listing, re.S | re.M).group(0)
    waited = None
    for line in body.splitlines():
        text = line.split(';')[0].strip()
        if not re.match(r'[a-z]+_', text):
            continue
        if text.startswith('v_mfma'):
            waited = 0
        elif text.startswith('global_store_dwordx4') and waited is not None:
            return waited, text
        elif waited is not None:
            nop = re.match(r's_nop (\d+)', text)
            waited += int(nop.group(1)) + 1 if nop else 1
    raise AssertionError(f'no store behind an MFMA in {name}')


@pytest.mark.parametrize('half', [False, True])
def test_results_of_mfmas_are_ready_for_the_store(listing, half):
    plain, _ = _store_behind_mfma(listing, False, half)
    waited, store = _store_behind_mfma(listing, True, half)
    assert plain >= 3 and waited >= plain, (waited, plain)
    assert re.search(r'\bsc1\b', store) and not re.search(r'\b(sc0|nt)\b', store), store
