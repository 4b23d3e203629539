"""A server whose budget has no room for the nets' part masks: requests are
evaluated through the lists, with K in the masks' range, and run side by side
where their footprints without masks allow it. Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_BAL, SCHED_REF, Server, schedule
from oracle import oracle as O
from oracle_refine import refine

pytestmark = pytest.mark.gpu


def _graph(seed, nov=3000, hubs=(62, 63, 64, 65, 127, 129, 190)):
    rng = np.random.default_rng(seed)
    sizes = [8, 9, 64, 65, 128, 300, 700] * 3 + list(rng.integers(1, 13, 2 * nov))
    nets = [list(rng.choice(np.arange(len(hubs), nov), size=s, replace=False)) for s in sizes]
    for h, d in enumerate(hubs):
        for i in rng.choice(np.arange(21, len(nets)), size=d, replace=False):
            nets[i].append(h)
    net_ptr = np.zeros(len(nets) + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum([len(n) for n in nets])
    return H.Hypergraph.from_nets(nov, net_ptr, np.concatenate([np.array(n) for n in nets]).astype(np.uint32),
                                  np.array([n[rng.integers(len(n))] for n in nets], np.int32))


def _sched(metric, hg, K, R):
    C, max_pw, min_pw = H.ref_constants(hg.nov, K, 1.0)
    if metric == "CN":
        return None
    if metric == "TV":
        cap = H.balance_cap(hg.nov, K, 0.3)
        return schedule(SCHED_BAL, R, C, cap, 0, cap)
    return schedule(SCHED_REF, R, C, max_pw, min_pw)


def _mask_bytes(hg, K):
    return 16 * ((K + 63) // 64) * (hg.noe + 1)


@pytest.mark.parametrize("metric", ["TV", "TM", "MSM", "MSV", "MSRV"])
@pytest.mark.parametrize("K", [2, 33, 64, 129, 300, 512])
def test_requests_without_room_for_masks(metric, K):
    hg = _graph(K)
    rng = np.random.default_rng(K + 1)
    part = rng.integers(0, K, hg.nov).astype(np.int32)
    sched = _sched(metric, hg, K, hg.nov if metric == "TM" else 700)
    got = []
    budget = 1 << 36
    for _ in range(2):
        with Server(0, hbm_budget=budget, workers=1) as srv:
            srv.add_graph(hg)
            print(f"no masks: {metric} K={K} budget {budget}", flush=True)
            got.append(srv.wait(srv.submit(0, metric, K, part, sched, 3)))
        budget = got[0][0]["footprint"] - 1
    assert got[1][0]["footprint"] == got[0][0]["footprint"] - _mask_bytes(hg, K)
    st, moves = refine(hg, K, metric, sched, O.build_state(hg, K, part), 3)
    for info, out in got:
        assert np.array_equal(out, st.part)
        assert moves is None or info["moves"] == moves


def test_masks_come_and_go_on_one_context():
    # a request with masks, then ones that fit only without the first one's
    hg = _graph(7)
    rng = np.random.default_rng(8)
    reqs = [(m, K, rng.integers(0, K, hg.nov).astype(np.int32), _sched(m, hg, K, 700))
            for m, K in (("TV", 512), ("MSV", 64), ("CN", 64), ("TV", 512), ("MSRV", 512), ("MSM", 40))]

    def run(budget):
        with Server(0, hbm_budget=budget, workers=1) as srv:
            srv.add_graph(hg)
            return [srv.wait(srv.submit(0, m, K, part, sched, 2)) for m, K, part, sched in reqs]

    wide = run(1 << 36)
    # what the first request needs with its masks: the third and the last fit it only by themselves
    tight = run(max(info["footprint"] - _mask_bytes(hg, 512) for info, _ in wide) + _mask_bytes(hg, 64))
    for (m, K, part, sched), (i0, p0), (i1, p1) in zip(reqs, wide, tight):
        st, _ = refine(hg, K, m, sched, O.build_state(hg, K, part), 2)
        assert np.array_equal(p0, st.part) and np.array_equal(p1, st.part), (m, K)
        assert i0["metrics"] == i1["metrics"]


def test_requests_that_fit_without_masks_run_side_by_side():
    hg = H.colnet(60_000, H.DEG_FIXED, 6, seed=4)
    K, passes = 512, 60
    part = H.initial_partition_for("MSRV", hg, K)
    sched = _sched("MSRV", hg, K, 2048)

    def run(budget, workers):
        with Server(0, hbm_budget=budget, workers=workers) as srv:
            ids = [srv.add_graph(hg) for _ in range(workers)]
            rids = [srv.submit(g, "MSRV", K, part, sched, passes) for g in ids]
            return [srv.wait(r) for r in rids], srv.stats()

    (one,), _ = run(1 << 36, 1)
    without = one[0]["footprint"] - _mask_bytes(hg, K)
    both, stats = run(2 * without, 2)
    assert stats["peak_inflight"] == 2 and stats["peak_bytes"] <= 2 * without
    for info, out in both:
        assert np.array_equal(out, one[1]) and info["metrics"] == one[0]["metrics"]
