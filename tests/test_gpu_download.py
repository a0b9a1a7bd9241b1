"""fq_download returns the list fq_load took, whatever its length against the
pinned slots it leaves through (1 MiB each, one per thread)."""
import ctypes as C
import threading

import numpy as np
import pytest

from hande_amd import api, _native as N
from helpers import engine_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sites,spaces", [(12, 1), (12, 2), (40, 1), (40, 2)])
@pytest.mark.parametrize("n", [1, 1000, 21845, 43691, 200001])
def test_download_returns_the_loaded_list(sites, spaces, n):
    lib = N.lib()
    system = api.hubbard_k(electrons=2, lattice=[[sites]], ms=0, sym=1, U=1)
    W = system.view.nwords
    p = engine_params(system.view, api.qmc_in({"tau": 0.01}, rng_mode="philox"))
    p.nspaces, p.main_capacity, p.spawn_capacity = spaces, n + 7, 1 << 10
    rng = np.random.default_rng(n + sites)
    states = np.sort(rng.integers(0, 1 << 24, n, dtype=np.uint64)).repeat(W)  # any words: they are only copied
    pops, dat = rng.integers(-9, 9, n * spaces), rng.normal(size=n)
    ptr = lambda a, t: a.ctypes.data_as(C.POINTER(t))
    eng, got = C.c_void_p(), C.c_int64()
    N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
    try:
        N.check(lib.fq_load(eng, ptr(states, C.c_uint64), ptr(pops, C.c_int64), ptr(dat, C.c_double), n), "fq_load")
        a = [np.zeros(n * W, np.uint64), np.zeros(n * spaces, np.int64), np.zeros(n)]
        N.check(lib.fq_download(eng, ptr(a[0], C.c_uint64), ptr(a[1], C.c_int64), ptr(a[2], C.c_double), n,
                                C.byref(got)), "fq_download")
        assert got.value == n
        assert np.array_equal(a[0], states) and np.array_equal(a[1], pops) and np.array_equal(a[2], dat)
        assert lib.fq_download(eng, ptr(a[0], C.c_uint64), ptr(a[1], C.c_int64), ptr(a[2], C.c_double), n - 1,
                               C.byref(got)) == -5  # FQ_ERR_CAPACITY
        b = np.zeros(n * spaces, np.int64)  # arrays that are not asked for
        N.check(lib.fq_download(eng, None, ptr(b, C.c_int64), None, n, C.byref(got)), "fq_download")
        assert np.array_equal(b, pops)
    finally:
        lib.fq_destroy(eng)


@pytest.mark.parametrize("n", [3000, 200001])
def test_threads_download_at_the_same_time(n):
    """Four threads, the first downloads of the engine among them, each take the
    whole list ten times."""
    lib = N.lib()
    system = api.hubbard_k(electrons=2, lattice=[[12]], ms=0, sym=1, U=1)
    p = engine_params(system.view, api.qmc_in({"tau": 0.01}, rng_mode="philox"))
    p.main_capacity, p.spawn_capacity = n, 1 << 10
    rng = np.random.default_rng(n)
    states = np.sort(rng.integers(0, 1 << 24, n, dtype=np.uint64))
    pops, dat = rng.integers(-9, 9, n), rng.normal(size=n)
    ptr = lambda a, t: a.ctypes.data_as(C.POINTER(t))
    eng = C.c_void_p()
    N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
    same = []

    def take():
        for _ in range(10):
            a, got = [np.zeros(n, np.uint64), np.zeros(n, np.int64), np.zeros(n)], C.c_int64()
            rc = lib.fq_download(eng, ptr(a[0], C.c_uint64), ptr(a[1], C.c_int64), ptr(a[2], C.c_double), n, C.byref(got))
            same.append(rc == 0 and got.value == n and all(np.array_equal(x, y) for x, y in zip(a, (states, pops, dat))))

    try:
        N.check(lib.fq_load(eng, ptr(states, C.c_uint64), ptr(pops, C.c_int64), ptr(dat, C.c_double), n), "fq_load")
        threads = [threading.Thread(target=take) for _ in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len(same) == 40 and all(same)
    finally:
        lib.fq_destroy(eng)
