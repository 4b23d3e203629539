"""What a context holds of the device's memory, and what it says it holds."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import SCHED_BAL, SCHED_REF, Engine, Server, schedule

pytestmark = pytest.mark.gpu


def _refine(eng, hg, metric, K):
    C, max_pw, min_pw = H.ref_constants(hg.nov, K)
    eng.set_partition(K, (np.arange(hg.nov) * K // hg.nov).astype(np.int32))
    eng.refine(metric, 1, schedule(SCHED_REF, 4096, C, max_pw, min_pw))


def test_part_masks_of_a_smaller_k_are_given_back():
    hg = H.colnet(40_000, H.DEG_FIXED, 4, seed=3)
    with Engine(0) as eng:
        eng.upload(hg)
        _refine(eng, hg, "TV", 512)
        direct = eng.device_bytes()
    with Engine(0) as eng:
        eng.upload(hg)
        for K in range(64, 513, 64):
            _refine(eng, hg, "TV", K)
        stepwise = eng.device_bytes()
        state = eng.get_state()
        eng.upload(hg)
        _refine(eng, hg, "TV", 512)
        assert eng.device_bytes() <= stepwise
        again = eng.get_state()
    # 16 bytes a net and 64 parts: all eight arrays together are 23 MB, the last one 5.1 MB
    assert stepwise - direct < 2 * 16 * 8 * hg.noe
    assert np.array_equal(state.part, again.part) and np.array_equal(state.ep_parts, again.ep_parts)


def test_message_events_of_a_smaller_k_are_given_back():
    # half a million pins: an event takes 8 bytes, a source's move has two for
    # each part that its net can touch
    hg = H.colnet(20_000, H.DEG_FIXED, 24, seed=3)
    steps = (2, 5, 8, 11, 14, 17, 20, 23)
    with Engine(0) as eng:
        eng.upload(hg)
        _refine(eng, hg, "MSM", steps[-1])
        direct = eng.device_bytes()
    with Engine(0) as eng:
        eng.upload(hg)
        for K in steps:
            _refine(eng, hg, "MSM", K)
        stepwise = eng.device_bytes()
    # all eight arrays together are 93 MB, the last one 15; a slab or two
    # of the small arrays may be left
    last = 8 * (2 * (hg.pins - hg.noe) + 2 * steps[-1] * hg.noe)
    print(f"message events: direct {direct} stepwise {stepwise} last {last}", flush=True)
    assert stepwise - direct < 2 * last


@pytest.mark.parametrize("nov", [1, 300, 1_000, 20_000])
def test_a_context_says_what_it_holds(nov):
    # its slabs: a few times its arrays, and no more once a refinement's
    # scratch is cut from what they have left
    hg = H.colnet(nov, H.DEG_FIXED, min(4, nov - 1), seed=3)
    arrays = 22 * (hg.pins + hg.noe) + 16 * hg.nov
    with Engine(0) as eng:
        eng.upload(hg)
        held = eng.device_bytes()
        assert arrays <= held <= 4 * arrays + (64 << 10)
        if nov > 1:
            _refine(eng, hg, "TV", 16)
            eng.metrics()
            assert eng.device_bytes() == held


@pytest.mark.parametrize("metric,K", [("TV", 3_000), ("CN", 2_000), ("TM", 3_200), ("MSM", 3_200), ("MSV", 3_200),
                                      ("MSRV", 3_200), ("TM", 300), ("MSRV", 100)])
def test_a_requests_footprint_covers_what_its_calls_allocate(metric, K):
    # an engine of its own does the request's calls: of what it allocates, no
    # more than the last two slabs can be unused
    hg = H.colnet(4_200, H.DEG_FIXED, 1, seed=3)
    C, max_pw, min_pw = H.ref_constants(hg.nov, K)
    cap = H.balance_cap(hg.nov, K, 0.05)
    sched = {"CN": None, "TV": schedule(SCHED_BAL, hg.nov, C, cap, 0, cap)}.get(
        metric, schedule(SCHED_REF, hg.nov, C, max_pw, min_pw))
    part = (np.arange(hg.nov) * K // hg.nov).astype(np.int32)
    with Engine(0) as eng:
        eng.upload(hg)
        slab = eng.device_bytes()
        eng.set_partition(K, part)
        eng.refine(metric, 1, sched)
        eng.metrics()
        used = eng.device_bytes() - 2 * slab
    with Server(0, hbm_budget=1 << 36, workers=1) as srv:
        srv.add_graph(hg)
        info, _ = srv.wait(srv.submit(0, metric, K, part, sched, 1))
    print(f"footprint: {metric} K={K} slab {slab} used {used} footprint {info['footprint']}", flush=True)
    assert used <= info["footprint"]
