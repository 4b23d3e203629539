"""The lists built from a part vector: nets that fill, overflow and leave gaps
in a window of 64 pins (0, 1, 2, 31 .. 65, 128 pins, thousands), chunks of nets
cut short, few and many parts. Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import Engine
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("permuted", [False, True])
@pytest.mark.parametrize("K", [1, 2, 5, 64, 300, 2000, 4096])
def test_lists_from_a_partition(K, permuted):
    rng = np.random.default_rng(K)
    nov = 6000
    edge = [0, 1, 2, 31, 32, 33, 62, 63, 64, 65, 127, 128, 129, 511, 513, 3000]
    for nets in (1, 63, 20000):
        sizes = rng.permutation(edge + list(rng.integers(0, 9, nets)))[:nets]
        net_ptr = np.zeros(nets + 1, dtype=np.uint32)
        net_ptr[1:] = np.cumsum(sizes)
        pins = np.concatenate([rng.choice(nov, size=s, replace=False) for s in sizes] + [[]]).astype(np.uint32)
        hg = H.Hypergraph.from_nets(nov, net_ptr, pins, None)
        order = rng.permutation(nov).astype(np.int32) if permuted else None
        part = rng.integers(0, K, nov).astype(np.int32)
        print(f"build: K={K} nets={nets} pins={hg.pins} permuted={permuted}", flush=True)
        with Engine(0) as eng:
            eng.upload(hg, order)
            for _ in range(2):  # over the segments of an earlier state too
                eng.set_partition(K, part)
                got, st = eng.get_state(), O.build_state(hg, K, part, order)
                for k in ("part", "ep_ends", "ep_parts", "ep_cnt"):
                    assert np.array_equal(getattr(got, k), getattr(st, k)), k
                part = np.minimum(part, K // 2).astype(np.int32)
