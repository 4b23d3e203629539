"""One resident hypergraph refined with a small K first and a larger one after:
what the context keeps between refinements has to fit the larger K too.
Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_REF, Engine, schedule
from oracle import oracle as O
from oracle_refine import assert_same_state, refine

pytestmark = pytest.mark.gpu


def test_message_events_of_a_larger_k():
    # nets of up to 60 pins in random parts: at K = 2 a list has two entries,
    # at K = 300 up to 60, and a source's move has two events for each
    rng = np.random.default_rng(4)
    nov = 2000
    sizes = list(rng.integers(1, 4, nov)) + list(rng.integers(20, 61, 60))
    nets = [rng.choice(nov, size=s, replace=False) for s in sizes]
    net_ptr = np.zeros(len(nets) + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum(sizes)
    hg = H.Hypergraph.from_nets(nov, net_ptr, np.concatenate(nets).astype(np.uint32),
                                np.array([n[0] for n in nets], np.int32))
    with Engine(0) as eng:
        eng.upload(hg)
        for K in (2, 7, 300, 20, 600):
            C, max_pw, min_pw = H.ref_constants(nov, K)
            part = rng.integers(0, K, nov).astype(np.int32)
            sched = schedule(SCHED_REF, 400, C, max_pw, min_pw)
            print(f"message events: K={K}", flush=True)
            eng.set_partition(K, part)
            moves = eng.refine("MSM", 3, sched).moves
            st, want = refine(hg, K, "MSM", sched, O.build_state(hg, K, part), 3)
            assert moves == want
            assert_same_state(eng.get_state(), st)
