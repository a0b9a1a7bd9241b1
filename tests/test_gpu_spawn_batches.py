"""Attempts beyond the spawned list's capacity are made in several launches,
whatever the tiles: the chain is the oracle's, bit for bit."""
import pytest

from hande_amd import _native as N
from hande_amd import api
from helpers import production_lockstep
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
