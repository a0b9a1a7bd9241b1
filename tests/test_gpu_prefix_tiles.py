"""The prefixes of a cycle's counts: added up by the kernels that need them
while the counts are few, scanned first when they are many.  With the scans
from the first count on, the tests of the annihilation, the production cycles,
the learned rows and the graph cycles pass as they do without; at the lengths
where the scans begin both ways give the same walkers."""
import ctypes as C
import itertools

import numpy as np
import pytest

import test_gpu_annihilate as annihilate
import test_gpu_batch as batch
import test_gpu_learned_sizes as learned
import test_gpu_production_lockstep as lockstep
import test_gpu_semi_stoch as semi_stoch
from hande_amd import _native as N
from hande_amd import api
from helpers import download

pytestmark = pytest.mark.gpu

P = C.POINTER
NEVER = 1 << 40


@pytest.fixture
def scans(monkeypatch):
    """Every engine made scans its counts from the first on."""
    lib, made = N.lib(), []

    def scanning(create):
        def wrapped(*args):
            rc = create(*args)
            if rc == N.FQ_OK:
                N.check(lib.fqt_prefix_tiles(args[-1]._obj, 0, 0, 0), "fqt_prefix_tiles")
                made.append(args[-1]._obj)
            return rc
        return wrapped

    for name in ("fq_create", "fq_create_batch"):
        monkeypatch.setattr(lib, name, scanning(getattr(lib, name)))
    yield
    assert made


@pytest.mark.parametrize("real", [False, True])
def test_annihilation_replay(scans, real):
    hub = api.hubbard_k(electrons=6, lattice=[[3, 0], [0, 3]], ms=0, sym="tot_sym", U=2)
    annihilate.test_annihilate_replay_matches_oracle(hub, True, real, 7)


def test_annihilation_long_lists(scans):
    annihilate.test_annihilate_production_large_lists(600_000, 1_200_000)


def test_annihilation_two_word_values(scans):
    annihilate.test_annihilate_production_two_word_rank_keys()


@pytest.mark.parametrize("kind", ["real", "pair", "renorm", "heat_bath", "two_words", "core"])
def test_production_cycles(scans, tmp_path, kind):
    if kind == "real":
        lockstep.test_hubbard_k(True, True)
    elif kind == "pair":
        lockstep.test_hubbard_k_replica_pair()
    elif kind == "two_words":
        lockstep.test_two_word_determinants(tmp_path)
    elif kind == "core":
        semi_stoch.test_production_semi_stochastic_molecular(tmp_path, 0)
    else:
        lockstep.test_molecular_real_initiator(tmp_path, kind)


@pytest.mark.parametrize("n", [1024, 2500])
def test_learned_rows(scans, tmp_path, n):
    learned.test_network_rows_are_the_determinants_with_enough_attempts(tmp_path, n, 4)


def test_graph_cycles(scans):
    batch.test_graph_cycles_match_ordinary_cycles()


def _ring_list(sites, nalpha, n):
    """n determinants of nalpha electrons of either spin in list order."""
    half = np.array([sum(1 << (2 * o) for o in c) for c in itertools.combinations(range(sites), nalpha)], dtype=np.uint64)
    beta = half[:-(-n // len(half))] << np.uint64(1)
    return np.sort((half[:, None] | beta[None, :]).reshape(-1))[:n]


def _load(lib, eng, dets, pops):
    N.check(lib.fq_load(eng, dets.ctypes.data_as(P(C.c_uint64)), pops.ctypes.data_as(P(C.c_int64)),
                        np.zeros(len(dets)).ctypes.data_as(P(C.c_double)), len(dets)), "fq_load")


def _fields(o):
    return (o.nstates, o.nspawn_events, o.ndeath, o.nattempts, o.nparticles[0], o.proj_energy[0], o.D0_population[0])


# 1024 entries a main tile (2048 of them), 256 a block of attempts (16384)
@pytest.mark.parametrize("n", [2048 * 1024, 2048 * 1024 + 1, 16384 * 256, 16384 * 256 + 1])
def test_cycles_at_the_lengths_where_the_scans_begin(n):
    """Cycles of the engine as it is, with scans throughout and with none; the
    first cycle's list has the length, and enough spawned entries for the run
    tiles (4096) to pass theirs."""
    lib = N.lib()
    system = api.hubbard_k(electrons=18, lattice=[[18]], ms=0, sym=1, U=1.0, t=1.0)
    dets, pops = _ring_list(18, 9, n), np.full(n, 6, dtype=np.int64)
    sh = (C.c_double * 2)(0.0, 0.0)
    results = []
    for limits in (None, (0, 0, 0), (NEVER, NEVER, NEVER)):
        eng, out = C.c_void_p(), N.FqCycleOut()
        N.check(lib.fq_create(system.view, C.byref(lockstep._params(41, cap=1 << 25)), C.byref(eng)), "fq_create")
        try:
            if limits:
                N.check(lib.fqt_prefix_tiles(eng, *limits), "fqt_prefix_tiles")
            _load(lib, eng, dets, pops)
            got = []
            for _ in range(2):
                N.check(lib.fq_cycle(eng, sh, sh, 0.02, C.byref(out)), "fq_cycle")
                got.append(_fields(out))
                print(f"  {n} {limits}: attempts {out.nattempts}, spawned {out.nspawn_events}, {out.nstates} after",
                      flush=True)
                assert out.nspawn_events > 4096 * 1024 and not out.spawn_overflow and not out.main_overflow
            results.append((got, download(lib, eng, 1, 1)))
        finally:
            lib.fq_destroy(eng)
    for got, lst in results[1:]:
        assert got == results[0][0]
        for x, y in zip(lst, results[0][1]):
            assert np.array_equal(x, y)


def test_graph_cycles_with_tiled_scans():
    """2.3e6 determinants make more counts (8192) than one block scans: graph
    cycles whose launches write the scan scratch, replayed after a longer list's
    graphs were captured, against ordinary cycles without scans."""
    lib = N.lib()
    systems = [api.hubbard_k(electrons=18, lattice=[[18]], ms=0, sym=1, U=u, t=1.0) for u in (1.0, 2.0)]
    arr = (N.FqSystem * 2)(*[s.view for s in systems])
    sh, tau, outs = np.zeros(2), np.full(2, 0.002), [(N.FqCycleOut * 2)(), (N.FqCycleOut * 2)()]
    engs = []
    try:
        for graph in (0, 1):
            eng = C.c_void_p()
            N.check(lib.fq_create_batch(arr, 2, C.byref(lockstep._params(43, cap=1 << 24)), C.byref(eng)), "create")
            engs.append(eng)
            limit = 0 if graph else NEVER
            N.check(lib.fqt_prefix_tiles(eng, limit, limit, limit), "fqt_prefix_tiles")
            N.check(lib.fq_batch_graph(eng, graph), "fq_batch_graph")
        for per in (1150000, 1900000, 1150000):
            dets, inst = np.tile(_ring_list(18, 9, per), 2), np.repeat(np.arange(2, dtype=np.int32), per)
            pops = np.ones(2 * per, dtype=np.int64)
            for eng in engs:
                N.check(lib.fq_load_batch(eng, inst.ctypes.data_as(P(C.c_int32)), dets.ctypes.data_as(P(C.c_uint64)),
                                          pops.ctypes.data_as(P(C.c_int64)),
                                          np.zeros(2 * per).ctypes.data_as(P(C.c_double)), 2 * per), "load")
            for cyc in range(6):
                for eng, out in zip(engs, outs):
                    N.check(lib.fq_cycle_batch(eng, sh.ctypes.data_as(P(C.c_double)), sh.ctypes.data_as(P(C.c_double)),
                                               tau.ctypes.data_as(P(C.c_double)), out), "fq_cycle_batch")
                for a, b in zip(*outs):
                    assert _fields(a) == _fields(b), (per, cyc)
            for x, y in zip(download(lib, engs[0], 1, 1), download(lib, engs[1], 1, 1)):
                assert np.array_equal(x, y), per
        info = N.FqScheduleOut()
        N.check(lib.fq_batch_schedule(engs[1], C.byref(info)), "fq_batch_schedule")
        assert info.graph_cycles == 15 and info.eager_cycles == 3
    finally:
        for eng in engs:
            lib.fq_destroy(eng)
