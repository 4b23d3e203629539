"""Few nets of many pins, which the TV apply takes one to a wavefront: on both
sides of 64 pins a net on average. Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_BAL, SCHED_REF, Engine, schedule
from oracle import oracle as O
from oracle_refine import assert_same_state, refine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noe,sizes", [(1, (800, 801)), (5, (300, 2_000)), (131, (64, 65)), (131, (65, 66)), (131, (1, 900))])
@pytest.mark.parametrize("K", [6, 200, 600])
def test_few_nets(noe, sizes, K):
    rng = np.random.default_rng(noe + K)
    nov = 2_100
    nets = [rng.choice(nov, size=int(rng.integers(*sizes)), replace=False) for _ in range(noe)]
    net_ptr = np.zeros(noe + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum([len(n) for n in nets])
    hg = H.Hypergraph.from_nets(nov, net_ptr, np.concatenate(nets).astype(np.uint32),
                                np.array([n[0] for n in nets], np.int32))
    part = rng.integers(0, K, nov).astype(np.int32)
    C, cap = 1.5 * nov / K, int(1.3 * nov / K) + 3
    print(f"few nets: nets={noe} K={K} pins={hg.pins}", flush=True)
    with Engine(0) as eng:
        eng.upload(hg)
        for sched in (schedule(SCHED_BAL, 500, C, cap, 0, cap), schedule(SCHED_REF, 700, C, nov, 0)):
            eng.set_partition(K, part)
            eng.refine("TV", 3, sched)
            st, _ = refine(hg, K, "TV", sched, O.build_state(hg, K, part), 3)
            assert_same_state(eng.get_state(), st)
        eng.initial_partition(1, K, 400, C, 0, cap)
        st, _ = O.round_ldg(hg, K, "ldg", C, 0, 400, cap)
        assert_same_state(eng.get_state(), st)
