"""Vertices of very many nets, with neighbouring numbers, among ordinary ones:
degrees at the edges of the chunks of nets and in the thousands; and rounds of
more slots than the evaluation's waves have lanes. Bit-exact against the
oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_BAL, SCHED_REF, Engine, schedule
from oracle import oracle as O
from oracle_refine import assert_same_state, refine

pytestmark = pytest.mark.gpu


def _graph(seed, nov=6001, first=700):
    rng = np.random.default_rng(seed)
    hubs = [500, 511, 512, 513, 575, 576, 577, 1000, 2048, 3000, 5500, 5999]
    noe = nov
    base = rng.integers(0, nov, (noe, 3))
    nets = [set(b) | {n} for n, b in enumerate(base)]
    for h, d in enumerate(hubs):
        for n in rng.choice(noe, size=d, replace=False):
            nets[n].add(first + h)
    nets = [np.array(sorted(int(x) for x in n)) for n in nets]
    net_ptr = np.zeros(noe + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum([len(n) for n in nets])
    # a quarter of the nets have a hub as their source, where they hold one
    src = np.array([n[np.searchsorted(n, first)] if i % 4 == 0 and np.searchsorted(n, first) < len(n) else i
                    for i, n in enumerate(nets)], np.int32)
    return H.Hypergraph.from_nets(nov, net_ptr, np.concatenate(nets).astype(np.uint32), src)


@pytest.mark.parametrize("metric", ["TV", "TM", "MSM", "MSV", "MSRV"])
@pytest.mark.parametrize("K", [3, 130, 300, 384, 448, 512, 700])
def test_hubs(metric, K):
    hg = _graph(K)
    rng = np.random.default_rng(K + 1)
    part = rng.integers(0, K, hg.nov).astype(np.int32)
    C, max_pw, min_pw = H.ref_constants(hg.nov, K, 2.0)
    for R in (2500, hg.nov):
        if metric == "TV":
            cap = H.balance_cap(hg.nov, K, 0.5)
            sched = schedule(SCHED_BAL, R, C, cap, 0, cap)
        else:
            sched = schedule(SCHED_REF, R, C, max_pw, min_pw)
        print(f"hubs: {metric} K={K} R={R} pins={hg.pins}", flush=True)
        with Engine(0) as eng:
            eng.upload(hg)
            eng.set_partition(K, part)
            moves = eng.refine(metric, 3, sched).moves
            got = eng.get_state()
        st, want = refine(hg, K, metric, sched, O.build_state(hg, K, part), 3)
        assert want is None or moves == want
        assert_same_state(got, st)


def test_more_slots_than_the_waves_lanes():
    # 7,168 waves of 64 lanes hold 458,752 slots
    hg = H.colnet(520_003, H.DEG_FIXED, 2, seed=2)
    K = 5
    part = np.random.default_rng(3).integers(0, K, hg.nov).astype(np.int32)
    C, max_pw, min_pw = H.ref_constants(hg.nov, K, 0.5)
    cap = H.balance_cap(hg.nov, K, 0.5)
    for metric, sched in (("TV", schedule(SCHED_BAL, hg.nov, C, cap, 0, cap)),
                          ("MSV", schedule(SCHED_REF, hg.nov, C, max_pw, min_pw))):
        print(f"slots: {metric}", flush=True)
        with Engine(0) as eng:
            eng.upload(hg)
            eng.set_partition(K, part)
            eng.refine(metric, 2, sched)
            got = eng.get_state()
        st, _ = refine(hg, K, metric, sched, O.build_state(hg, K, part), 2)
        assert_same_state(got, st)
