"""Attempts beyond the spawned list's capacity are made in several launches,
whatever the tiles: the chain is the oracle's, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from hande_amd import _native as N
from hande_amd import api
from helpers import download, production_lockstep
from test_gpu_production_lockstep import _mol, _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity", [2047, 2048, 2049, 5000])
@pytest.mark.parametrize("kind", ["hub", "pair", "renorm", "heat_bath"])
def test_attempts_in_several_launches(tmp_path, kind, capacity):
    if kind in ("hub", "pair"):
        system = api.hubbard_k(electrons=6, lattice=[[10]], ms=0, sym=1, U=3.0, t=1.0)
        p = _params(211, spaces=2 if kind == "pair" else 1)
    else:
        system = _mol(tmp_path, 12, 6, 1207)
        p = _params(212, getattr(N, "FQ_EXCIT_" + kind.upper()))
    p.spawn_capacity = capacity
    outs = production_lockstep(system, p, 8, 20000, tau=0.001, label=f"{kind} {capacity}")
    assert outs[-1].nattempts > 3 * capacity


@pytest.mark.parametrize("capacity", [2047, 2048, 2049, 5000])
def test_learned_attempts_in_several_launches(tmp_path, capacity):
    """The learned generator makes its attempts in tiles of 256 where one launch
    holds them and of 1024 in several: the same chain either way."""
    lib, system = N.lib(), _mol(tmp_path, 12, 6, 1207)
    W, sh, chains = system.view.nwords, (C.c_double * 2)(0.0, 0.0), []
    for cap in (capacity, 1 << 18):
        p, eng, out = _params(213, N.FQ_EXCIT_LEARNED), C.c_void_p(), N.FqCycleOut()
        p.spawn_capacity, p.proposal_mix, p.proposal_min_attempts = cap, 0.1, 4
        N.check(lib.fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
        try:
            f0 = np.array([system.view.f0[w] for w in range(W)], dtype=np.uint64)
            N.check(lib.fq_load(eng, f0.ctypes.data_as(C.POINTER(C.c_uint64)),
                                np.array([20000]).ctypes.data_as(C.POINTER(C.c_int64)),
                                np.zeros(1).ctypes.data_as(C.POINTER(C.c_double)), 1), "fq_load")
            chain = []
            for _ in range(8):
                N.check(lib.fq_cycle(eng, sh, sh, 0.001, C.byref(out)), "fq_cycle")
                assert not out.spawn_overflow and out.nattempts > 3 * capacity
                chain.append((out.nstates, out.nspawn_events, out.ndeath, out.nattempts, out.nparticles[0],
                              out.proj_energy[0], *[x.tobytes() for x in download(lib, eng, W, 1)]))
            chains.append(chain)
        finally:
            lib.fq_destroy(eng)
    assert chains[0] == chains[1]
