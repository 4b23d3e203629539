"""Vertices of few list entries, for K past the part masks: net
sizes at the edge of a row (15 | 16 parts), degrees at the edges of a window,
a group and the limit (4, 16, 32 | 33 rows), isolated vertices, mixed with
long lists. Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_REF, Engine, schedule
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _graph(seed, nov=3000, longs=20):
    rng = np.random.default_rng(seed)
    hubs = [1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 40, 70, 0, 0]
    sizes = list(rng.integers(1, 16, 3 * nov)) + [15, 16, 17] * longs + [64, 65, 300] * (longs // 5)
    nets = [list(rng.choice(np.arange(len(hubs), nov), size=s, replace=False)) for s in sizes]
    for h, d in enumerate(hubs):
        for i in rng.choice(3 * nov, size=d, replace=False):
            if len(nets[i]) < 15:
                nets[i].append(h)
    net_ptr = np.zeros(len(nets) + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum([len(n) for n in nets])
    pins = np.concatenate([np.array(n) for n in nets]).astype(np.uint32)
    return H.Hypergraph.from_nets(nov, net_ptr, pins, np.array([n[0] for n in nets], np.int32))


def _same(got, st):
    for k in ("part", "ep_ends", "ep_parts", "ep_cnt"):
        assert np.array_equal(getattr(got, k), getattr(st, k)), k
    assert np.array_equal(got.sizes, st.sizes.astype(np.int64))


@pytest.mark.parametrize("metric,permuted", [("MSV", False), ("MSRV", False), ("MSRV", True)])
@pytest.mark.parametrize("K", [513, 640, 1024, 1025])
def test_volume_short_lists(metric, permuted, K):
    hg = _graph(K, longs=20 if K != 640 else 0)
    order = np.random.default_rng(K + 1).permutation(hg.nov).astype(np.int32) if permuted else None
    C, max_pw, min_pw = H.ref_constants(hg.nov, K)
    for R in (300, hg.nov):
        st = O.msv_ldg(hg, K, C) if metric == "MSV" else O.msrv_ldg(hg, K, C, ordering=order)
        print(f"short lists: {metric} K={K} R={R} permuted={permuted} pins={hg.pins}", flush=True)
        with Engine(0) as eng:
            eng.upload(hg, ordering=order)
            eng.set_state(K, st.part, st.ep_ends, st.ep_parts, st.ep_cnt)
            moves = eng.refine(metric, 4, schedule(SCHED_REF, R, C, max_pw, min_pw)).moves
            got = eng.get_state()
        if metric == "MSV":
            want = O.msv_refine_par(hg, st, C, 4, R)
        else:
            want = O.msrv_refine_par(hg, st, C, 4, R, ordering=order)
        assert moves == want
        _same(got, st)
