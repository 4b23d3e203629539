"""The TV apply on both sides of the K up to which its waves keep a part ->
position index of a list in LDS (2,450), and up to the largest K of a
refinement with a schedule (3,200). Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_BAL, SCHED_REF, Engine, schedule
from oracle import oracle as O
from oracle_refine import assert_same_state

pytestmark = pytest.mark.gpu


def _graph(seed, nov=6500):
    rng = np.random.default_rng(seed)
    sizes = [8, 9, 63, 64, 65, 255, 256, 257, 2600, 6000] * 4 + list(rng.integers(1, 13, 2 * nov))
    net_ptr = np.zeros(len(sizes) + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum(sizes)
    nets = [rng.choice(nov, size=s, replace=False) for s in sizes]
    return H.Hypergraph.from_nets(nov, net_ptr, np.concatenate(nets).astype(np.uint32),
                                  np.array([n[0] for n in nets], np.int32))


@pytest.mark.parametrize("K", [2040, 2449, 2450, 2451, 2460, 2493, 2494, 2730, 3200])
def test_apply_around_the_index_limit(K):
    hg = _graph(K)
    part = np.random.default_rng(K + 1).integers(0, K, hg.nov).astype(np.int32)
    C, cap = 1.5 * hg.nov / K, int(1.3 * hg.nov / K) + 3
    print(f"apply: K={K} pins={hg.pins}", flush=True)
    with Engine(0) as eng:
        eng.upload(hg)
        for R in (900, hg.nov):
            eng.set_partition(K, part)
            moves = eng.refine("TV", 2, schedule(SCHED_BAL, R, C, cap, 0, cap)).moves
            st = O.build_state(hg, K, part)
            O.tv_refine_bal(hg, st, C, cap, 0, cap, 2, R)
            assert moves > 0
            assert_same_state(eng.get_state(), st)
        eng.set_partition(K, part)
        moves = eng.refine("TV", 2, schedule(SCHED_REF, 700, C, hg.nov, 0)).moves
        st = O.build_state(hg, K, part)
        st.sizes = st.sizes.astype(np.int32)
        O.tv_refine_par(hg, st, C, hg.nov, 0, 2, 700)
        assert moves > 0
        assert_same_state(eng.get_state(), st)
        eng.initial_partition(1, K, 1000, C, 0, cap)
        st, _ = O.round_ldg(hg, K, "ldg", C, 0, 1000, cap)
        assert_same_state(eng.get_state(), st)
