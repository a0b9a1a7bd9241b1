"""Device memory of an engine per slot of its main list."""
import ctypes as C

import pytest

from hande_amd import _native as N
from hande_amd import api
from test_gpu_production_lockstep import _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sites,electrons,words,spaces", [(30, 4, 1, 1), (30, 4, 1, 2), (40, 4, 2, 1), (40, 4, 2, 2),
                                                          (60, 20, 2, 1), (60, 20, 2, 2)])
def test_a_slot_takes_no_more_than_without_kept_sort_values(sites, electrons, words, spaces):
    """Two buffers of determinants, populations and K_ii, the post-death
    populations, attempts, their offsets and the flags at eight bytes each, bits
    and block sums: what a slot took when the merge compared determinants.  The
    last two systems' sort values are two words.  (Half a byte a slot is the
    granularity of the allocations at this capacity.)"""
    lib = N.lib()
    hip = C.CDLL("libamdhip64.so.7")  # the engine's own runtime, loaded with it
    system = api.hubbard_k(electrons=electrons, lattice=[[sites]], ms=0, sym=1, U=2.0, t=1.0)
    assert system.view.nwords == words

    def taken(capacity):
        p = _params(5, spaces=spaces, cap=1 << 10)
        p.main_capacity = capacity
        before, after, total, eng = C.c_size_t(), C.c_size_t(), C.c_size_t(), C.c_void_p()
        assert hip.hipMemGetInfo(C.byref(before), C.byref(total)) == 0
        N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
        assert hip.hipMemGetInfo(C.byref(after), C.byref(total)) == 0
        lib.fq_destroy(eng)
        return before.value - after.value

    taken(1 << 10)  # what the first engine alone makes stays out
    slots = 1 << 25
    per_slot = (taken(slots) - taken(1 << 10)) / slots
    without = 2 * (8 * words + 8 * spaces + 8) + 3 * 8 * spaces + 8 + 24 / 64 + 56 / 256
    print(f"{sites} sites, {spaces} spaces: {per_slot:.2f} bytes a slot, {without:.2f} without", flush=True)
    assert 0 < per_slot < without + 0.5
