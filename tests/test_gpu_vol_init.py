"""The volumes of the resident state, from few nets with long lists to many:
nets per wavefront 1, 2 and more, lists on both sides of what one lane takes.
They decide the refinement's moves, which are compared with the oracle's."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_REF, Engine, schedule
from oracle import oracle as O
from oracle_refine import assert_same_state, refine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", ["MSV", "MSRV"])
@pytest.mark.parametrize("noe,sizes", [(1, (900, 901)), (63, (1, 400)), (300, (15, 300)), (4_097, (14, 19)),
                                       (9_000, (1, 18))])
def test_volumes_of_few_and_many_nets(metric, noe, sizes):
    rng = np.random.default_rng(noe)
    nov, K = 2_500, 90
    nets = [rng.choice(nov, size=int(rng.integers(*sizes)), replace=False) for _ in range(noe)]
    net_ptr = np.zeros(noe + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum([len(n) for n in nets])
    hg = H.Hypergraph.from_nets(nov, net_ptr, np.concatenate(nets).astype(np.uint32),
                                np.array([n[0] for n in nets], np.int32))
    part = rng.integers(0, K, nov).astype(np.int32)
    C, max_pw, min_pw = H.ref_constants(nov, K, 2.0)
    sched = schedule(SCHED_REF, 600, C, max_pw, min_pw)
    print(f"volumes: {metric} nets={noe} pins={hg.pins}", flush=True)
    with Engine(0) as eng:
        eng.upload(hg)
        eng.set_partition(K, part)
        moves = eng.refine(metric, 3, sched).moves
        got = eng.get_state()
    st, want = refine(hg, K, metric, sched, O.build_state(hg, K, part), 3)
    assert moves == want
    assert_same_state(got, st)
