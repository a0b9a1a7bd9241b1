"""The one-block sort of short spawned lists where its words hold few index
bits: a value of 52 to 56 bits leaves 12 to 8 of them, which is the list it
takes; longer lists, and values of 57 bits, go through the passes."""
import ctypes as C

import numpy as np
import pytest

from hande_amd import _native as N
from hande_amd import api
from helpers import download, odownload, oracle
from test_gpu_production_lockstep import _params

pytestmark = pytest.mark.gpu


def _random_words(rng, nb, nel, n, W):
    occ = np.argsort(rng.random((n, nb)), axis=1)[:, :nel]
    words = np.zeros((n, W), dtype=np.uint64)
    for k in range(nel):
        words[np.arange(n), occ[:, k] // 64] |= np.uint64(1) << (occ[:, k] % 64).astype(np.uint64)
    words = np.unique(words[:, ::-1], axis=0)[:, ::-1]  # list order: the last word first
    assert len(words) == n
    return np.ascontiguousarray(words)


@pytest.mark.parametrize("spaces", [1, 2])
@pytest.mark.parametrize("sites,electrons,limit", [(26, 26, 4096), (28, 28, 2048), (27, 26, 1024), (32, 20, 512),
                                                   (33, 20, 256), (34, 20, 128)])
def test_lists_around_the_longest_the_index_bits_hold(sites, electrons, limit, spaces):
    """Integer pairs: the oracle inserts, as the reference does, a determinant
    whose only walkers lie in a space the initiator rule clears, and drops it a
    cycle later; the engine never inserts a determinant without walkers."""
    lib, orc = N.lib(), oracle()
    system = api.hubbard_k(electrons=electrons, lattice=[[sites]], ms=0, sym=1, U=1)
    W = system.view.nwords
    p = _params(3, initiator=True, spaces=spaces, cap=1 << 15)
    ptr = lambda a, t: a.ctypes.data_as(C.POINTER(t))
    for n in (limit - 1, limit, limit + 1):
        rng = np.random.default_rng(n + sites)
        pool = _random_words(rng, 2 * sites, electrons, 1000 + n // 2, W)
        main = np.ascontiguousarray(pool[np.sort(rng.choice(len(pool), 700, replace=False))])
        pops = rng.integers(1, 9, (700, spaces)) * rng.choice([-1, 1], (700, spaces))
        sk = np.ascontiguousarray(pool[rng.integers(0, len(pool), n)])
        sp = np.zeros((n, spaces), dtype=np.int64)
        sp[np.arange(n), rng.integers(0, spaces, n)] = rng.integers(1, 4, n) * rng.choice([-1, 1], n)
        sf = rng.integers(0, 1 << spaces, n)
        eng = C.c_void_p()
        N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
        h = orc.orc_create(system.view, C.byref(p), 1)
        orc.orc_set_stable_order(h, 1)
        try:
            lst = (ptr(main, C.c_uint64), ptr(pops, C.c_int64), ptr(np.zeros(700), C.c_double), 700)
            N.check(lib.fq_load(eng, *lst), "fq_load")
            orc.orc_load(h, *lst)
            o1, o2 = N.FqCycleOut(), N.FqCycleOut()
            spawned = (ptr(sk, C.c_uint64), ptr(sp, C.c_int64), ptr(sf, C.c_int64), n)
            N.check(lib.fq_annihilate(eng, *spawned, C.byref(o1)), "fq_annihilate")
            orc.orc_annihilate(h, *spawned, C.byref(o2))
            want = [x.reshape(o2.nstates, -1) for x in odownload(orc, h, W, spaces)]
            held = want[1].any(axis=1)
            assert o1.nstates == held.sum() > 700 and (spaces == 2 or held.all())
            for x, y in zip(download(lib, eng, W, spaces), want):
                assert np.array_equal(x, y[held].reshape(-1)), n
        finally:
            lib.fq_destroy(eng)
            orc.orc_destroy(h)
