"""The device's streaming partition on nets of more than 64 pins, whose pins of
a round come 64 at a time: sizes at the edges of a window and of the windows
loaded together, few parts (many pins to a part) and many (most pins bring one),
K past the part masks, placement in a permuted order. Bit-exact against the
oracle's buffered round stream, list order included."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import Engine
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _graph(seed, nov=2500):
    rng = np.random.default_rng(seed)
    sizes = [64, 65, 66, 127, 128, 129, 255, 256, 257, 320, 511, 513, 1000, nov - 1, nov]
    sizes += list(rng.integers(1, 9, nov))
    net_ptr = np.zeros(len(sizes) + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum(sizes)
    pins = np.concatenate([rng.choice(nov, size=s, replace=False) for s in sizes]).astype(np.uint32)
    return H.Hypergraph.from_nets(nov, net_ptr, pins, None)


@pytest.mark.parametrize("mode,code", [("ldg_bands", 0), ("ldg", 1), ("cn_ldg", 2)])
@pytest.mark.parametrize("permuted", [False, True])
@pytest.mark.parametrize("K", [1, 3, 64, 511, 900])
def test_stream_of_large_nets(mode, code, permuted, K):
    hg = _graph(K)
    order = np.random.default_rng(K + 1).permutation(hg.nov).astype(np.int32) if permuted else None
    C, max_pw, _ = H.ref_constants(hg.nov, K, 0.05)
    cap = H.balance_cap(hg.nov, K, 0.05)
    for R in (1, 700, hg.nov):
        print(f"stream: {mode} K={K} R={R} permuted={permuted} pins={hg.pins}", flush=True)
        with Engine(0) as eng:
            eng.upload(hg, ordering=order)
            eng.initial_partition(code, K, R, C, max_pw, cap)
            got = eng.get_state()
        want, _ = O.round_ldg(hg, K, mode, C, max_pw, R, cap, ordering=order)
        for k in ("part", "ep_ends", "ep_parts", "ep_cnt"):
            assert np.array_equal(getattr(got, k), getattr(want, k)), k
        assert np.array_equal(got.sizes, want.sizes)
