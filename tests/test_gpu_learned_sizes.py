"""Sizes at which the learned proposal's kernels change shape: rows of the
inference (16 or 64 to a block), samples of the training products (chunks of
four slabs), list lengths around the tiles that number the network's rows."""
import contextlib
import ctypes as C
import itertools

import numpy as np
import pytest

from hande_amd import _native as N
from helpers import download
from test_gpu_learned import M, P, _engine, _forward, _orb_info, _random_dets, _random_samples, _set_params, _system

pytestmark = pytest.mark.gpu


def test_inference_rows_do_not_depend_on_the_list(tmp_path):
    """Every list gives the first rows of the longest one, bit for bit; those
    agree with the oracle within the bounds of the inference test."""
    system = _system(tmp_path, 8, 4, 308)
    nb, eps, _ = _orb_info(system)
    lib, eng = _engine(system)
    try:
        params = M.init_params(nb, 17)
        _set_params(lib, eng, params)
        dets, _ = _random_dets(nb, 4, 8257, np.random.default_rng(5))
        full = _forward(lib, eng, dets, nb)
        ref = np.clip(M.forward(params, M.occupations(dets, nb), eps, bf16_inference=True), -M.CLIP, M.CLIP)
        err = np.abs(np.log(full.astype(np.float64)) - ref)
        assert err.max() < 3e-2 and err.mean() < 2e-3
        for n in (1, 15, 16, 17, 63, 64, 65, 8191, 8192, 8193):
            assert np.array_equal(_forward(lib, eng, dets[:n], nb), full[:n]), n
    finally:
        lib.fq_destroy(eng)


@pytest.mark.parametrize("ns", [1, 15, 16, 17, 63, 64, 65, 127, 129, 257, 1030])
def test_gradient_at_sample_counts(tmp_path, ns):
    system = _system(tmp_path, 8, 4, 808)
    nb, eps, orb_sym = _orb_info(system)
    lib, eng = _engine(system)
    try:
        params = M.init_params(nb, 23)
        _set_params(lib, eng, params)
        dets, _occs, exc, w = _random_samples(nb, 4, orb_sym, ns, np.random.default_rng(ns))
        w[0] = 1.0
        flat = np.zeros(ns, dtype=np.int32)
        loss = C.c_double()
        grad = np.zeros(len(params), dtype=np.float32)
        N.check(lib.fq_mlp_loss_grad(eng, np.ascontiguousarray(dets).ctypes.data_as(P(C.c_uint64)),
                                     exc.ctypes.data_as(P(C.c_int32)), w.ctypes.data_as(P(C.c_double)),
                                     flat.ctypes.data_as(P(C.c_int32)), ns, C.byref(loss),
                                     grad.ctypes.data_as(P(C.c_float))), "fq_mlp_loss_grad")
        ref_loss, ref_grad = M.loss_and_grad(params.astype(np.float64), M.occupations(dets, nb), eps, orb_sym,
                                             [tuple(int(x) for x in e) for e in exc], w, flat.astype(bool))
        assert abs(loss.value - ref_loss) < 1e-5 * abs(ref_loss)
        for name, (o, cnt) in M.sizes(nb)[2].items():
            g, r = grad[o:o + cnt].astype(np.float64), ref_grad[o:o + cnt]
            assert np.abs(g - r).max() <= 2e-4 * np.abs(r).max() + 1e-9, name
    finally:
        lib.fq_destroy(eng)


@pytest.mark.parametrize("min_attempts", [0, 1, 4])
@pytest.mark.parametrize("n", [1, 255, 1023, 1024, 1025, 2500])
def test_network_rows_are_the_determinants_with_enough_attempts(tmp_path, n, min_attempts):
    """Integer populations make |N| attempts.  The first cycle of a loaded list
    counts the rows, the second has them bounded by the first one's list."""
    system = _system(tmp_path, 10, 6, 1010)
    nb, _eps, _sym = _orb_info(system)
    lib = N.lib()
    p = N.FqParams()
    p.nspaces, p.excit_gen, p.rng_mode, p.philox_seed = 1, N.FQ_EXCIT_LEARNED, N.FQ_RNG_PHILOX, 7
    p.main_capacity = p.spawn_capacity = 1 << 15
    p.proposal_mix, p.proposal_min_attempts = 0.1, min_attempts
    eng = C.c_void_p()
    N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
    try:
        rng = np.random.default_rng(n)
        dets = np.unique(_random_dets(nb, 6, 2 * n + 8, rng)[0][:, 0])
        dets = np.sort(rng.permutation(dets)[:n])
        pops = rng.choice([-1, 1], n) * rng.integers(1, 7, n)
        N.check(lib.fq_load(eng, dets.ctypes.data_as(P(C.c_uint64)), pops.ctypes.data_as(P(C.c_int64)),
                            np.zeros(n).ctypes.data_as(P(C.c_double)), n), "fq_load")
        for _ in range(3):
            o, pr = N.FqCycleOut(), N.FqProfileOut()
            N.check(lib.fq_cycle(eng, (C.c_double * 2)(0.0, 0.0), (C.c_double * 2)(0.0, 0.0), 0.01, C.byref(o)),
                    "fq_cycle")
            N.check(lib.fq_last_profile(eng, C.byref(pr)), "fq_last_profile")
            assert o.nattempts == np.abs(pops).sum()
            assert pr.proposal_rows == (np.abs(pops) >= min_attempts).sum()
            pops = np.zeros(o.nstates, dtype=np.int64)
            got = C.c_int64()
            N.check(lib.fq_download(eng, None, pops.ctypes.data_as(P(C.c_int64)), None, o.nstates, C.byref(got)),
                    "fq_download")
    finally:
        lib.fq_destroy(eng)


def _many_dets(norb, nel, n):
    """n determinants of nel/2 alpha and nel/2 beta electrons in list order."""
    half = np.array([sum(1 << (2 * o) for o in c) for c in itertools.combinations(range(norb), nel // 2)], dtype=np.uint64)
    beta = half[:-(-n // len(half))] << np.uint64(1)
    return np.sort((half[:, None] | beta[None, :]).reshape(-1))[:n]


@contextlib.contextmanager
def _no_memory_left():
    """The card's memory taken until it has no 128 MB to give."""
    hip, hog = C.CDLL("libamdhip64.so.7"), []  # the engine's own runtime, loaded with it
    try:
        for size in (1 << 33, 128 << 20):
            while hip.hipMalloc(C.byref(block := C.c_void_p()), C.c_size_t(size)) == 0:
                hog.append(block)
            hip.hipGetLastError()
        yield
    finally:
        for block in hog:
            hip.hipFree(block)


def _list_of_1e6(tmp_path, min_attempts):
    """A system, its parameters and 1e6 determinants of one walker, every 500th of five."""
    p = N.FqParams()
    p.nspaces, p.excit_gen, p.rng_mode, p.philox_seed = 1, N.FQ_EXCIT_LEARNED, N.FQ_RNG_PHILOX, 9
    p.main_capacity = p.spawn_capacity = 1 << 22
    p.proposal_mix, p.proposal_min_attempts = 0.1, min_attempts
    pops = np.ones(1000000, dtype=np.int64)
    pops[::500] = 5
    return _system(tmp_path, 20, 8, 2008), p, _many_dets(20, 8, len(pops)), pops


def _load(lib, eng, dets, pops):
    N.check(lib.fq_load(eng, dets.ctypes.data_as(P(C.c_uint64)), pops.ctypes.data_as(P(C.c_int64)),
                        np.zeros(len(pops)).ctypes.data_as(P(C.c_double)), len(pops)), "fq_load")


def test_rows_follow_the_list_where_their_bound_has_no_memory(tmp_path):
    """At a threshold of two the attempts bound the rows by 5e5 (160 MB of
    weights), a few thousand are there.  Where the card has no 128 MB left the
    cycle runs as it does with all of it."""
    lib = N.lib()
    system, p, dets, pops = _list_of_1e6(tmp_path, 2)
    engs, results = [], []
    sh = (C.c_double * 2)(0.0, 0.0)
    try:
        for _ in range(2):
            eng = C.c_void_p()
            N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
            engs.append(eng)
            _load(lib, eng, dets, pops)
            N.check(lib.fq_cycle(eng, sh, sh, 1e-3, C.byref(N.FqCycleOut())), "fq_cycle")
        for eng, memory in ((engs[0], _no_memory_left()), (engs[1], contextlib.nullcontext())):
            out, prof = N.FqCycleOut(), N.FqProfileOut()
            with memory:
                N.check(lib.fq_cycle(eng, sh, sh, 1e-3, C.byref(out)), "fq_cycle")
            N.check(lib.fq_last_profile(eng, C.byref(prof)), "fq_last_profile")
            assert out.nattempts > 8e5 and 1000 < prof.proposal_rows < 65536
            results.append((out.nstates, out.nspawn_events, out.nattempts, out.ndeath, out.nparticles[0],
                            prof.proposal_rows, *[x.tobytes() for x in download(lib, eng, 1, 1)]))
        assert results[0] == results[1]
    finally:
        for eng in engs:
            lib.fq_destroy(eng)


def test_a_cycle_without_memory_leaves_nothing_to_the_next_call(tmp_path):
    """Without a threshold every determinant needs its row: 320 MB are not there.
    The walkers stay, and the annihilation of an empty list after it reports no
    estimators of the cycle that failed."""
    lib = N.lib()
    system, p, dets, pops = _list_of_1e6(tmp_path, 0)
    dets[0], pops[0] = system.view.f0[0], 7  # the reference determinant, the list's first
    assert dets[0] < dets[1]
    eng, out = C.c_void_p(), N.FqCycleOut()
    sh = (C.c_double * 2)(0.0, 0.0)
    N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
    try:
        _load(lib, eng, dets, pops)
        with _no_memory_left():
            assert lib.fq_cycle(eng, sh, sh, 1e-3, C.byref(out)) == -2  # FQ_ERR_NOMEM
        none, empty = np.zeros(1, np.uint64), np.zeros(1, np.int64)
        N.check(lib.fq_annihilate(eng, none.ctypes.data_as(P(C.c_uint64)), empty.ctypes.data_as(P(C.c_int64)),
                                  empty.ctypes.data_as(P(C.c_int64)), 0, C.byref(out)), "fq_annihilate")
        assert (out.proj_energy[0], out.D0_population[0], out.ndeath, out.nattempts) == (0.0, 0.0, 0, 0)
        assert out.nstates == len(dets) and out.nparticles[0] == np.abs(pops).sum()
        got = download(lib, eng, 1, 1)
        assert np.array_equal(got[0], dets) and np.array_equal(got[1], pops)
        N.check(lib.fq_cycle(eng, sh, sh, 1e-3, C.byref(out)), "fq_cycle")
        assert out.D0_population[0] == 7.0 and out.nattempts == np.abs(pops).sum()
    finally:
        lib.fq_destroy(eng)
