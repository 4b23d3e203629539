"""MSV and MSRV through the part masks at the edges of their 64-part words, with
vertices of 62 to 129 nets (the chunks of nets are 63 or 64 long), in both
visiting orders. Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_REF, Engine, schedule
from oracle import oracle as O
from oracle_refine import assert_same_state, refine

pytestmark = pytest.mark.gpu


def _graph(seed, nov=2500, hubs=(62, 63, 64, 65, 126, 127, 128, 129)):
    rng = np.random.default_rng(seed)
    sizes = [63, 64, 65, 128, 257, 900] + list(rng.integers(1, 6, nov))
    nets = [list(rng.choice(np.arange(len(hubs), nov), size=s, replace=False)) for s in sizes]
    for h, d in enumerate(hubs):
        for i in rng.choice(np.arange(6, len(nets)), size=d, replace=False):
            nets[i].append(h)
    net_ptr = np.zeros(len(nets) + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum([len(n) for n in nets])
    return H.Hypergraph.from_nets(nov, net_ptr, np.concatenate([np.array(n) for n in nets]).astype(np.uint32),
                                  np.array([n[rng.integers(len(n))] for n in nets], np.int32))


@pytest.mark.parametrize("metric,permuted", [("MSV", False), ("MSRV", False), ("MSRV", True)])
@pytest.mark.parametrize("K", [63, 64, 65, 128, 129, 192, 193, 256, 257, 320, 321, 384, 385, 448, 449, 512])
def test_volumes_at_word_edges(metric, permuted, K):
    hg = _graph(K)
    rng = np.random.default_rng(K + 1)
    order = rng.permutation(hg.nov).astype(np.int32) if permuted else None
    part = rng.integers(0, K, hg.nov).astype(np.int32)
    part[rng.random(hg.nov) < 0.2] = K - 1  # one part well above the others, in the last word
    C, max_pw, min_pw = H.ref_constants(hg.nov, K, 3.0)
    for R in (300, hg.nov):
        sched = schedule(SCHED_REF, R, C, max_pw, min_pw)
        print(f"mask words: {metric} K={K} R={R} permuted={permuted}", flush=True)
        with Engine(0) as eng:
            eng.upload(hg, ordering=order)
            eng.set_partition(K, part)
            moves = eng.refine(metric, 3, sched).moves
            got = eng.get_state()
        st, want = refine(hg, K, metric, sched, O.build_state(hg, K, part, order), 3, ordering=order)
        assert moves == want and moves > 0
        assert_same_state(got, st)
