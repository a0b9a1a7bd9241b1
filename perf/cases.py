"""The work that programs have this engine do, as cases that can be timed.

Every case is one call pattern of a real run, through the public entry points
(``hande_amd.api`` or the C-ABI of ``include/fqmc.h``):

* ``cycles``: an engine holding an equilibrated walker list runs a block of
  Monte Carlo cycles with the report loop's shift update and then hands the
  list back (``fq_cycle`` ... ``fq_download``: a block of a long run that ends
  with a restart dump).  The systems, generators and population encodings are
  those of the benchmark and of the regression decks: Hubbard rings with
  integer populations, synthetic molecules with real ones, the renormalised,
  heat-bath and learned generators, replica pairs, a semi-stochastic core.
* ``batch``: many independent rings in one engine (``fq_cycle_batch`` with
  graph launches), then the list.
* ``run``: one whole ``api.fciqmc`` call that continues a stored run and
  returns the report table and the state for the next restart file.
* ``train``: Adam steps of the learned proposal on samples of the walker list.
* ``grad``: loss and gradient of caller-supplied training samples.

A state keeps its chain from pass to pass, as a run does; the populations are
held at their target by the shift, so every pass is the same amount of work.
"""
import ctypes as C
import functools
import math
import os
import random
import tempfile

import numpy as np
import torch

from hande_amd import _native as N
from hande_amd import api, synthetic

REPORT = 5  # cycles between shift updates


# ---- the cases ---------------------------------------------------------------
def _mol(name, norb, nel, seed, walkers, cycles, gen="renorm", **more):
    """An i-FCIQMC case on a synthetic molecule with the benchmark's options."""
    case = dict(name=name, kind="cycles", system="mol", norb=norb, nel=nel, seed=seed, U=0.0, gen=gen, bits=31,
                initiator=True, spaces=1, walkers=walkers, cycles=cycles, tau=1e-3, min_attempts=0, core=0,
                separate=True)
    case.update(more)
    return case


def _ring(name, sites, nel, U, walkers, cycles, **more):
    """A Hubbard ring in momentum space with integer populations; the time step
    keeps the early growth to some percent a cycle, as a run's input does."""
    case = dict(name=name, kind="cycles", system="ring", norb=sites, nel=nel, seed=0, U=U, gen="renorm", bits=0,
                initiator=False, spaces=1, walkers=walkers, cycles=cycles,
                tau=round(min(0.005, 0.1 / (U * sites)), 5), min_attempts=0, core=0, separate=True)
    case.update(more)
    return case


def listed():
    mol26, mol40, mol60 = (synthetic.MOLECULAR_CONFIGS[k] for k in ("mol26", "mol40", "mol60"))
    return [
        # a regression deck's ring with real_64 initiator populations, run from a stored state to the next one
        dict(name="run_ring14_9e4", kind="run", norb=14, nel=10, U=2.0, walkers=90000, reports=30, tau=0.002, bits=31,
             initiator=True),
        # the smallest engines: a short test or the start of any run
        _ring("ring10_1e3", 10, 10, 4.0, 1000, 50),
        # a molecule while its population still grows
        _mol("mol26_1e4", *mol26, 10000, 50),
        # the determinant-rich end of the integer path
        _ring("ring18_3e6", 18, 18, 2.0, 3000000, 50),
        # the benchmark's configuration at its full population
        _mol("mol26_1e7", *mol26, 10000000, 50),
        # the reference's heat-bath generator on the same molecule
        _mol("mol26_heat_3e5", *mol26, 300000, 50, gen="heat_bath"),
        # the learned proposal at the population and threshold of its comparison
        _mol("mol40_learned_1e6", *mol40, 1000000, 50, gen="learned", min_attempts=64),
        # the two-word replica-pair configuration
        _mol("mol60_pair_1e6", *mol60, 1000000, 20, spaces=2),
        # a deterministic core in the main list
        _mol("mol26_core_3e5", *mol26, 300000, 50, core=1000),
        # many small rings in one engine
        dict(name="rings64", kind="batch", instances=64, low=4.0, high=5.5, cycles=50, tau=0.005),
        # training the proposal before and during a run
        dict(name="train_mol40", kind="train", norb=mol40[0], nel=mol40[1], seed=mol40[2], walkers=200000,
             batch=16384, steps=4, min_attempts=64, objective=1),
        # loss and gradient of samples that the caller holds
        dict(name="grad_mol26", kind="grad", norb=mol26[0], nel=mol26[1], seed=mol26[2], batch=4096, objective=0),
    ]


def draw(rng: random.Random):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["ring", "ring", "mol", "mol", "mol", "mol", "batch", "run", "train", "grad"])
    if kind == "ring":
        sites = rng.choice([8, 10, 12, 14, 16, 18])
        nel = sites + (0 if sites < 10 else rng.choice([-2, 0, 0, 2]))
        most = {8: 2000, 10: 30000, 12: 300000}.get(sites, 3000000)
        case = _ring("", sites, nel, round(rng.uniform(1.0, 6.0), 3), logint(500, most), rng.randint(20, 50),
                     gen=rng.choice(["renorm", "renorm", "no_renorm"]), initiator=rng.random() < 0.3,
                     bits=rng.choice([0, 0, 11, 31]), spaces=rng.choice([1, 1, 2]))
    elif kind == "mol":
        gen = rng.choice(["renorm", "renorm", "heat_bath", "learned"])
        norb = rng.randint(16, 40)
        nel = 2 * rng.randint(3, 8)
        case = _mol("", norb, nel, rng.randint(1, 9999), logint(3000, 3000000 if gen == "renorm" else 500000),
                    rng.randint(20, 50), gen=gen, bits=rng.choice([31, 31, 11]), spaces=rng.choice([1, 1, 1, 2]))
        if gen == "learned":
            case["min_attempts"] = rng.choice([0, 4, 64])
        elif gen == "renorm" and rng.random() < 0.3:
            case.update(core=logint(50, 3000), separate=rng.random() < 0.5)
    elif kind == "batch":
        case = dict(kind="batch", instances=rng.randint(2, 96), low=3.0, high=round(rng.uniform(3.5, 5.5), 2),
                    cycles=rng.randint(20, 50), tau=0.005)
    elif kind == "run":
        sites = rng.choice([10, 12, 14, 16])
        bits = rng.choice([0, 11, 31])
        case = dict(kind="run", norb=sites, nel=sites - rng.choice([0, 2, 4]), U=round(rng.uniform(1.0, 2.5), 3),
                    walkers=logint(1000, 90000), reports=rng.randint(10, 40), tau=0.001, bits=bits,
                    initiator=bits != 0 or rng.random() < 0.5)
    else:
        case = dict(kind=kind, norb=rng.randint(12, 40), nel=2 * rng.randint(3, 7), seed=rng.randint(1, 9999),
                    batch=logint(100, 16384), objective=rng.choice([0, 1]))
        if kind == "train":
            case.update(walkers=logint(5000, 200000), steps=rng.randint(1, 6), min_attempts=rng.choice([0, 4, 64]))
    case.pop("name", None)
    return case


# ---- systems and engines -----------------------------------------------------
@functools.lru_cache(maxsize=8)
def _molecule(norb, nel, seed):
    with tempfile.TemporaryDirectory(prefix="fqmc_cases_") as tmp:
        path = synthetic.write_fcidump(os.path.join(tmp, "FCIDUMP"), norb, nel, seed)
        return api.read_in(int_file=path, nel=nel, ms=0)


@functools.lru_cache(maxsize=256)
def _ring_system(sites, nel, U):
    return api.hubbard_k(electrons=nel, lattice=[[sites]], ms=0, sym=1, U=U, t=1.0)


def _system(case):
    if case.get("system", "mol") == "ring" or case["kind"] == "run":
        return _ring_system(case["norb"], case["nel"], case["U"])
    return _molecule(case["norb"], case["nel"], case["seed"])


def _params(cap, seed, gen="renorm", bits=31, initiator=True, spaces=1, min_attempts=0):
    p = N.FqParams()
    p.nspaces = spaces
    p.initiator = int(initiator)
    p.initiator_pop = 3.0
    p.quadrature_initiator = 1
    p.real_amplitudes = int(bits > 0)
    p.pop_bit_shift = bits
    p.spawn_cutoff = int(math.ceil(0.01 * (1 << bits))) if bits else 0
    p.excit_gen = {"renorm": N.FQ_EXCIT_RENORM, "no_renorm": N.FQ_EXCIT_NO_RENORM,
                   "heat_bath": N.FQ_EXCIT_HEAT_BATH, "learned": N.FQ_EXCIT_LEARNED}[gen]
    p.rng_mode = N.FQ_RNG_PHILOX
    p.philox_seed = seed
    p.main_capacity = p.spawn_capacity = cap
    p.device = 0
    p.proposal_mix = 0.1
    p.proposal_min_attempts = min_attempts
    return p


def _ptr(a, t):
    return a.ctypes.data_as(C.POINTER(t))


class Handle:
    """An engine and the host buffers its lists are handed back in."""

    def __init__(self, eng, cap, words, spaces):
        self.lib, self.eng = N.lib(), eng
        self.words, self.spaces, self.room = words, spaces, cap // 2
        self.states = np.zeros(self.room * words, dtype=np.uint64)
        self.pops = np.zeros(self.room * spaces, dtype=np.int64)
        self.dat = np.zeros(self.room)
        self.got = C.c_int64()

    def load(self, states, pops, dat):
        N.check(self.lib.fq_load(self.eng, _ptr(states, C.c_uint64), _ptr(pops, C.c_int64), _ptr(dat, C.c_double),
                                 len(dat)), "fq_load")

    def download(self):
        """The list, at the front of buffers whose size does not follow it."""
        N.check(self.lib.fq_download(self.eng, _ptr(self.states, C.c_uint64), _ptr(self.pops, C.c_int64),
                                     _ptr(self.dat, C.c_double), self.room, C.byref(self.got)), "fq_download")
        return {"states": self.states.view(np.int64), "pops": self.pops, "dat": self.dat, "n": self.got.value}

    def __del__(self):
        if self.eng:
            self.lib.fq_destroy(self.eng)
            self.eng = None


def _engine(system, cap, seed, **options):
    eng = C.c_void_p()
    p = _params(cap, seed, **options)
    N.check(N.lib().fq_create(system.view, C.byref(p), C.byref(eng)), "fq_create")
    return Handle(eng, cap, system.view.nwords, p.nspaces)


class Chain:
    """The report loop's side of a run: every REPORT cycles the shift moves by
    the population's change (and, so that it stays at the target, by its
    distance from it) and the projected energy of the report is kept."""

    def __init__(self, handle, case, tau):
        self.h, self.tau, self.target, self.S = handle, tau, float(case["walkers"]), handle.spaces
        self.shift, self.eold = (C.c_double * 2)(), (C.c_double * 2)()
        self.out = N.FqCycleOut()
        self.old = [0.0, 0.0]
        self.proj, self.d0 = [0.0, 0.0], [0.0, 0.0]
        self.count, self.vary = 0, False
        # a ring's population grows by some percent a cycle: its shift varies at once
        self.hold_from = 0.8 * self.target if case["system"] == "mol" else 0.0

    def cycle(self, damping=0.05):
        o = self.out
        N.check(self.h.lib.fq_cycle(self.h.eng, self.shift, self.eold, self.tau, C.byref(o)), "fq_cycle")
        if o.spawn_overflow or o.main_overflow:
            raise RuntimeError("a walker list is full")
        self.count += 1
        for s in range(self.S):
            self.proj[s] += o.proj_energy[s]
            self.d0[s] += o.D0_population[s]
        if self.count % REPORT == 0:
            for s in range(self.S):
                n, dt = o.nparticles[s], self.tau * REPORT
                if n <= 0:
                    raise RuntimeError("the population died out")
                if self.vary and self.old[s] > 0:
                    self.shift[s] -= (damping * math.log(n / self.old[s]) +
                                      damping ** 2 * math.log(n / self.target)) / dt
                if self.d0[s]:
                    self.eold[s] = self.proj[s] / self.d0[s]
                self.old[s], self.proj[s], self.d0[s] = n, 0.0, 0.0
            self.vary = self.vary or min(self.old[:self.S]) > self.hold_from
        return o

    def grow(self, hold, most):
        """From the reference determinant to the target population."""
        left = hold
        for _ in range(most):
            self.cycle(0.2)
            left -= self.vary and min(self.old[:self.S]) > 0.7 * self.target
            if left <= 0:
                break


def _grown(case, seed):
    """An engine whose list has grown from the reference determinant."""
    system = _system(case)
    cap = max((4 if case["system"] == "mol" else 8) * case["walkers"] * case["spaces"], 1 << 16)
    h = _engine(system, cap, seed, gen=case["gen"], bits=case["bits"], initiator=case["initiator"],
                spaces=case["spaces"], min_attempts=case["min_attempts"])
    pop = max(20, case["walkers"] // (30 if case["system"] == "mol" else 100)) << case["bits"]
    h.load(system.f0(), np.full(case["spaces"], pop, dtype=np.int64), np.zeros(1))
    chain = Chain(h, case, case["tau"])
    chain.grow(60, 1500)
    return h, chain


# ---- prepare, run --------------------------------------------------------------
def prepare(case, seed):
    return {"cycles": _prepare_cycles, "batch": _prepare_batch, "run": _prepare_run, "train": _prepare_train,
            "grad": _prepare_grad}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_cycles(case, seed):
    h, chain = _grown(case, 1000 + seed)
    if case["core"]:
        N.check(h.lib.fq_semi_stoch_init(h.eng, case["core"], int(case["separate"])), "fq_semi_stoch_init")
        for _ in range(2 * REPORT):
            chain.cycle()
    return {"run": _run_cycles, "handle": h, "chain": chain, "cycles": case["cycles"]}


def _row(o, spaces):
    return ([v[s] for s in range(spaces) for v in (o.proj_energy, o.D0_population, o.nparticles)],
            [o.nstates, o.nspawn_events, o.ndeath, o.nattempts])


def _run_cycles(state):
    chain, h = state["chain"], state["handle"]
    rows = [_row(chain.cycle(), h.spaces) for _ in range(state["cycles"])]
    return {"estimators": np.array([r[0] for r in rows]), "counts": np.array([r[1] for r in rows], dtype=np.int64),
            "shift": np.array(list(chain.shift)), **h.download()}


def _rings(case):
    """Rings of 10-18 sites near half filling with U/t in [1, 8] and targets
    spread over the case's decades, as the batched benchmark takes them."""
    rng = np.random.default_rng(2024)
    systems, targets = [], []
    for _ in range(case["instances"]):
        sites = int(rng.choice([10, 12, 14, 16, 18]))
        systems.append(_ring_system(sites, sites + int(rng.choice([-2, 0, 0, 2])), float(rng.uniform(1.0, 8.0))))
        targets.append(float(10 ** rng.uniform(case["low"], case["high"])))
    return systems, np.array(targets)


def _prepare_batch(case, seed):
    systems, targets = _rings(case)
    K, lib = len(systems), N.lib()
    cap = int(6 * targets.sum()) + (1 << 18)
    p = _params(cap, 1000 + seed, bits=0, initiator=False)
    eng = C.c_void_p()
    views = (N.FqSystem * K)(*[s.view for s in systems])
    N.check(lib.fq_create_batch(views, K, C.byref(p), C.byref(eng)), "fq_create_batch")
    h = Handle(eng, cap, 1, 1)
    N.check(lib.fq_batch_graph(eng, 1), "fq_batch_graph")
    inst = np.arange(K, dtype=np.int32)
    f0 = np.array([int(s.f0()[0]) for s in systems], dtype=np.uint64)
    pops = np.maximum(10, targets / 100).astype(np.int64)
    N.check(lib.fq_load_batch(eng, _ptr(inst, C.c_int32), _ptr(f0, C.c_uint64), _ptr(pops, C.c_int64),
                              _ptr(np.zeros(K), C.c_double), K), "fq_load_batch")
    state = {"run": _run_batch, "handle": h, "cycles": case["cycles"], "tau": np.full(K, case["tau"]),
             "targets": targets, "shift": np.zeros(K), "eold": np.zeros(K), "old": np.zeros(K),
             "vary": np.zeros(K, bool), "outs": (N.FqCycleOut * K)(), "count": 0, "proj": np.zeros(K),
             "d0": np.zeros(K)}
    for _ in range(500):
        _batch_cycle(state, 0.2)
    return state


def _batch_cycle(state, damping=0.05):
    h, outs, K = state["handle"], state["outs"], len(state["tau"])
    N.check(h.lib.fq_cycle_batch(h.eng, _ptr(state["shift"], C.c_double), _ptr(state["eold"], C.c_double),
                                 _ptr(state["tau"], C.c_double), outs), "fq_cycle_batch")
    rows = [_row(outs[k], 1) for k in range(K)]
    est, cnt = np.array([r[0] for r in rows]), np.array([r[1] for r in rows], dtype=np.int64)
    state["proj"] += est[:, 0]
    state["d0"] += est[:, 1]
    state["count"] += 1
    if state["count"] % REPORT == 0:
        n, dt = est[:, 2], state["tau"] * REPORT
        upd = state["vary"] & (state["old"] > 0) & (n > 0)
        state["shift"][upd] -= ((damping * np.log(n[upd] / state["old"][upd]) +
                                 damping ** 2 * np.log(n[upd] / state["targets"][upd])) / dt[upd])
        state["vary"] |= n > state["targets"] / 20
        ok = state["d0"] != 0
        state["eold"][ok] = state["proj"][ok] / state["d0"][ok]
        state["old"][:] = n
        state["proj"][:] = state["d0"][:] = 0.0
    return est, cnt


def _run_batch(state):
    rows = [_batch_cycle(state) for _ in range(state["cycles"])]
    return {"estimators": np.array([r[0] for r in rows]), "counts": np.array([r[1] for r in rows]),
            "shift": state["shift"].copy(), **state["handle"].download()}


def _run_options(case, seed, reports):
    cap = max(16 * case["walkers"], 1 << 17)
    return dict(tau=case["tau"], rng_seed=7 + seed, init_pop=max(10, case["walkers"] // 30), mc_cycles=10,
                nreports=reports, target_population=case["walkers"], initiator=case["initiator"],
                real_amplitudes=case["bits"] > 0, real_amplitude_force_32=case["bits"] == 11, spawn_cutoff=0.01,
                state_size=cap, spawned_state_size=cap)


def _prepare_run(case, seed):
    system = _system(case)
    _, start = api.fciqmc(system, _run_options(case, 500 + seed, 80), rng_mode="philox", return_state=True)
    room = _run_options(case, seed, 1)["state_size"]
    return {"run": _run_run, "system": system, "start": start, "qmc": _run_options(case, seed, case["reports"]),
            "states": np.zeros(room, dtype=np.int64), "pops": np.zeros(room, dtype=np.int64), "dat": np.zeros(room)}


def _run_run(state):
    table, end = api.fciqmc(state["system"], state["qmc"], rng_mode="philox", restart=state["start"],
                            return_state=True)
    n = end.nstates  # kept at the front of buffers whose size does not follow it
    state["states"][:n] = end.states.reshape(-1).view(np.int64)
    state["pops"][:n] = end.pops.reshape(-1)
    state["dat"][:n] = end.dat
    return {"table": table, "states": state["states"], "pops": state["pops"], "dat": state["dat"], "n": n}


def _network(handle, seed):
    """Parameters of a partly trained network (all blocks nonzero)."""
    n = C.c_int64()
    N.check(handle.lib.fq_mlp_nparams(handle.eng, C.byref(n)), "fq_mlp_nparams")
    p = np.empty(n.value, dtype=np.float32)
    N.check(handle.lib.fq_mlp_get_params(handle.eng, _ptr(p, C.c_float), n.value), "fq_mlp_get_params")
    return p + np.random.default_rng(seed).normal(0.0, 0.02, n.value).astype(np.float32)


def _prepare_train(case, seed):
    grown = _mol("", case["norb"], case["nel"], case["seed"], case["walkers"], 0, gen="learned",
                 min_attempts=case["min_attempts"])
    h, _ = _grown(grown, 1000 + seed)
    N.check(h.lib.fq_mlp_online(h.eng, 0, 0, 1, 1e-3, case["objective"]), "fq_mlp_online")
    return {"run": _run_train, "handle": h, "p0": _network(h, seed), "batch": case["batch"], "steps": case["steps"],
            "losses": np.zeros(case["steps"]), "seed": 5 + seed}


def _run_train(state):
    h, p0 = state["handle"], state["p0"]
    N.check(h.lib.fq_mlp_set_params(h.eng, _ptr(p0, C.c_float), len(p0)), "fq_mlp_set_params")
    N.check(h.lib.fq_mlp_train(h.eng, state["batch"], state["steps"], 1e-3, state["seed"],
                               _ptr(state["losses"], C.c_double)), "fq_mlp_train")
    p = np.empty_like(p0)
    N.check(h.lib.fq_mlp_get_params(h.eng, _ptr(p, C.c_float), len(p)), "fq_mlp_get_params")
    # the network and its losses are computed in float32
    return {"losses": state["losses"].astype(np.float32), "params": p}


def _samples(case, seed):
    """Doubles i<j -> a<b of random determinants (equal numbers of alpha and
    beta electrons), weights and |H| spread as heat-bath samples' are, a part
    of them on determinants without a network row."""
    rng = np.random.default_rng(seed)
    norb, nel, B = case["norb"], case["nel"], case["batch"]
    nb = 2 * norb
    occ = np.zeros((B, nb), dtype=bool)
    for spin in (0, 1):  # the lower orbitals more likely, as in a correlated ground state
        score = rng.gumbel(size=(B, norb)) - 4.0 * np.arange(norb) / norb
        pick = np.argsort(-score, axis=1)[:, :nel // 2]
        np.put_along_axis(occ[:, spin::2], pick, True, axis=1)
    score = rng.random((B, nb))
    order_o = np.argsort(np.where(occ, score, 2.0), axis=1)
    ij = np.sort(order_o[:, :2], axis=1)
    free = np.argsort(np.where(occ, 2.0, score), axis=1)[:, :nb - nel]
    # a and b with the spins of i and j
    spins = np.stack([ij[:, 0] % 2, ij[:, 1] % 2], axis=1)
    fs = free % 2
    rank = np.cumsum(fs[:, :, None] == np.array([0, 1])[None, None, :], axis=1)  # how many of each spin so far
    need = np.stack([np.ones(B, dtype=int), 1 + (spins[:, 0] == spins[:, 1])], axis=1)
    ab = np.empty((B, 2), dtype=np.int64)
    for k in (0, 1):
        hit = (fs == spins[:, k:k + 1]) & (np.take_along_axis(rank, spins[:, k][:, None, None], axis=2)[:, :, 0]
                                           == need[:, k:k + 1])
        ab[:, k] = free[np.arange(B), np.argmax(hit, axis=1)]
    ab = np.sort(ab, axis=1)
    words = -(-nb // 64)
    dets = np.zeros((B, words), dtype=np.uint64)
    for o in range(nb):
        dets[:, o // 64] |= occ[:, o].astype(np.uint64) << np.uint64(o % 64)
    return {"occ": occ, "dets": dets.reshape(-1), "exc": (np.concatenate([ij, ab], axis=1) + 1).astype(np.int32),
            "w": np.exp(rng.normal(0.0, 1.0, B)), "habs": 0.1 * np.exp(rng.normal(0.0, 0.5, B)),
            "flat": (rng.random(B) < 0.3).astype(np.int32)}


def _prepare_grad(case, seed):
    system = _molecule(case["norb"], case["nel"], case["seed"])
    h = _engine(system, 1 << 16, 11, gen="learned")
    p = _network(h, seed)
    N.check(h.lib.fq_mlp_set_params(h.eng, _ptr(p, C.c_float), len(p)), "fq_mlp_set_params")
    return {"run": _run_grad, "handle": h, "params": p, "samples": _samples(case, seed),
            "objective": case["objective"]}


def _run_grad(state):
    h, x, n = state["handle"], state["samples"], len(state["samples"]["w"])
    loss, grad = C.c_double(), np.empty_like(state["params"])
    lead = (h.eng, _ptr(x["dets"], C.c_uint64), _ptr(x["exc"], C.c_int32), _ptr(x["w"], C.c_double))
    tail = (_ptr(x["flat"], C.c_int32), n, C.byref(loss), _ptr(grad, C.c_float))
    if state["objective"]:
        N.check(h.lib.fq_mlp_variance_grad(*lead, _ptr(x["habs"], C.c_double), *tail), "fq_mlp_variance_grad")
    else:
        N.check(h.lib.fq_mlp_loss_grad(*lead, *tail), "fq_mlp_loss_grad")
    return {"loss": np.float32(loss.value), "grad": grad}  # computed in float32


# ---- exact values --------------------------------------------------------------
def exact(case, seed):
    """grad: the loss and its gradient in 64 bits by autograd.  The others are
    Markov chains, whose whole numbers are compared as they are."""
    if case["kind"] != "grad":
        return None
    state = _prepare_grad(case, seed)
    x, nb, H = state["samples"], 2 * case["norb"], 256
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.tensor(state["params"], dtype=torch.float64, device=dev, requires_grad=True)
    eps = np.array(_molecule(case["norb"], case["nel"], case["seed"]).basis()[2])
    occ = torch.tensor(x["occ"], device=dev)
    feat = torch.cat([occ.double(), occ * torch.tensor(eps, device=dev).float().double()], dim=1)
    sizes = [(2 * nb, H), (H,), (H, H), (H,), (H, 2 * nb), (2 * nb,), (nb, nb)]
    w1, b1, w2, b2, w3, b3, theta = (t.reshape(s) for t, s in zip(p.split([int(np.prod(s)) for s in sizes]), sizes))
    gelu = torch.nn.functional.gelu
    z = gelu(gelu(feat @ w1 + b1) @ w2 + b2) @ w3 + b3
    z = torch.where(torch.tensor(x["flat"], device=dev)[:, None] > 0, torch.zeros_like(z), z)
    e, f = z.clamp(-60, 60).exp().split(nb, dim=1)
    A = theta.clamp(-60, 60).exp()
    i, j, a, b = (torch.tensor(x["exc"][:, k].astype(np.int64) - 1, device=dev) for k in range(4))
    rows, orb = torch.arange(len(i), device=dev), torch.arange(nb, device=dev)
    free = ~occ
    zh = (e * occ).sum(1)
    wi, wj = f * A[i] * free, f * A[j] * free  # f_p A[hole][p] over the unoccupied orbitals

    def partners(first):  # the class that first's partner is drawn from
        odd = (i + j + first) % 2
        return free & (orb[None] % 2 == odd[:, None]) & (orb[None] != first[:, None])

    z1i, z1j = wi.sum(1), wj.sum(1)
    cb, ca = partners(a), partners(b)
    zbi, zbj, zai, zaj = (wi * cb).sum(1), (wj * cb).sum(1), (wi * ca).sum(1), (wj * ca).sum(1)
    ei, ej = e[rows, i], e[rows, j]
    pij, pji = ei / zh * ej / (zh - ei), ej / zh * ei / (zh - ej)
    ia, ib, ja, jb = wi[rows, a], wi[rows, b], wj[rows, a], wj[rows, b]
    q = pij * (ia / z1i * jb / zbj + ib / z1i * ja / zaj) + pji * (ja / z1j * ib / zbi + jb / z1j * ia / zai)
    w = torch.tensor(x["w"], device=dev)
    term = torch.tensor(x["habs"], device=dev) / q if case["objective"] else -q.log()
    loss = (w * term).sum() / w.sum()
    loss.backward()
    return {"loss": loss.item(), "grad": p.grad.cpu().numpy()}


# ---- work ----------------------------------------------------------------------
def work(case):
    """Bytes a pass cannot do without: the cycle's lists (main list read by
    spawning and by annihilation and written once, spawned list written and
    read once) and the list handed back; for training, the samples, the
    parameters and the products of forward and backward."""
    if case["kind"] in ("train", "grad"):
        nb, B, steps = 2 * case["norb"], case["batch"], case.get("steps", 1)
        weights = 4 * nb * 256 + 256 * 256
        params = weights + 512 + 2 * nb + nb * nb
        moved = 4 * params * (6 if case["kind"] == "train" else 2) + B * 56
        return {"bytes": float(steps * moved), "flops": float(steps * 6 * B * weights)}
    if case["kind"] == "batch":
        _, targets = _rings(case)
        dets, spawned, words, spaces = 0.6 * targets.sum(), 0.1 * targets.sum(), 1, 1
        cycles = case["cycles"]
    else:
        mol = case.get("system") == "mol"
        words = -(-2 * case["norb"] // 64)
        spaces = case.get("spaces", 1)
        dets = (0.4 if mol else 0.5) * case["walkers"]
        spawned = (0.35 if mol else 0.1) * case["walkers"] * spaces
        cycles = case["cycles"] if case["kind"] == "cycles" else 10 * case["reports"]
    entry, spawn = 8 * words + 8 * spaces + 8, 8 * words + 8 * spaces + 8
    return {"bytes": float(cycles * (3 * dets * entry + 2 * spawned * spawn) + dets * entry), "flops": 0.0}
