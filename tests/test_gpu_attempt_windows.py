"""Parent windows of the spawning tiles: every tile's window runs from the
parent of its first attempt to the parent of its last, whatever entries
without attempts lie between or behind them (a list in a bound-sized launch
ends in such entries)."""
import ctypes as C
import itertools

import numpy as np
import pytest

from hande_amd import _native as N
from hande_amd import api
from test_gpu_production_lockstep import _params

pytestmark = pytest.mark.gpu


def _dets(nb, nel, n):
    """The first n determinants in list order."""
    words = np.array([sum(1 << o for o in c) for c in itertools.combinations(range(nb), nel)], dtype=np.uint64)
    return np.sort(words)[:n]


@pytest.mark.parametrize("spaces", [1, 2])
@pytest.mark.parametrize("n,live,per", [(3000, 3000, 9), (5000, 900, 9), (13000, 4096, 5), (13000, 4095, 5),
                                        (38000, 12000, 3), (38000, 100, 3), (38000, 1, 1025)])
def test_windows_are_the_parents_of_the_first_and_last_attempts(n, live, per, spaces):
    """Determinants from `live` on hold no walkers; before it 0 to `per` each."""
    lib = N.lib()
    system = api.hubbard_k(electrons=6, lattice=[[10]], ms=0, sym=1, U=3.0, t=1.0)
    eng = C.c_void_p()
    N.check(lib.fq_create(system.view, C.byref(_params(77, spaces=spaces)), C.byref(eng)), "fq_create")
    try:
        rng = np.random.default_rng(n + live)
        pops = np.zeros((n, spaces), dtype=np.int64)
        pops[:live] = rng.integers(0, per + 1, (live, spaces)) * rng.choice([-1, 1], (live, spaces))
        pops[live - 1] = per
        if np.abs(pops).sum() % 1024 == 0:
            pops[0] += 1
        ptr = lambda a, t: a.ctypes.data_as(C.POINTER(t))
        N.check(lib.fq_load(eng, ptr(_dets(20, 6, n), C.c_uint64), ptr(pops, C.c_int64), ptr(np.zeros(n), C.c_double),
                            n), "fq_load")
        sh, out = (C.c_double * 2)(0.0, 0.0), N.FqCycleOut()
        for tile in (1024, 256):  # the attempts of a loaded list are unknown, then bounded: large and small tiles
            attempts = np.abs(pops).reshape(-1)
            parent = np.repeat(np.arange(len(attempts)), attempts)
            N.check(lib.fq_cycle(eng, sh, sh, 1e-5, C.byref(out)), "fq_cycle")
            assert out.nattempts == len(parent)
            first = np.arange(0, len(parent), tile)
            last = np.minimum(first + tile, len(parent)) - 1
            win = np.zeros((len(first), 2), dtype=np.int64)
            N.check(lib.fqt_tile_windows(eng, ptr(win, C.c_int64), len(first)), "fqt_tile_windows")
            assert np.array_equal(win, np.stack([parent[first], parent[last]], axis=1)), tile
            pops = np.zeros((out.nstates, spaces), dtype=np.int64)
            got = C.c_int64()
            N.check(lib.fq_download(eng, None, ptr(pops, C.c_int64), None, out.nstates, C.byref(got)), "fq_download")
    finally:
        lib.fq_destroy(eng)
