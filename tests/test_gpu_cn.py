"""Cut-net evaluation over packed windows: nets of two parts of every size
around a window (2 .. 64 | 65 pins and thousands), few nets per wave, and the
pushes of nets with more ops than a wavefront. Bit-exact against the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import Engine
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nets", [70, 9000, 40000])
@pytest.mark.parametrize("K", [2, 3, 40])
def test_cut_nets_of_two_parts(K, nets):
    rng = np.random.default_rng(K + nets)
    nov = 5000
    # neighbouring vertices share a part, so that nets over a run of vertices have one or two
    part = (np.arange(nov) // 25 % K).astype(np.int32)
    edge = [1, 2, 31, 32, 33, 62, 63, 64, 65, 66, 127, 128, 129, 300, 2000]
    sizes = rng.permutation(edge * 4 + list(rng.integers(1, 8, nets)))[:nets]
    pins = []
    for s in sizes:
        if s <= 40:
            pins.append((rng.integers(0, nov) + rng.choice(max(int(s), 40), size=s, replace=False)) % nov)
        else:  # two parts only
            two = np.flatnonzero((part == 0) | (part == 1))
            pins.append(rng.choice(two, size=min(int(s), len(two)), replace=False))
    net_ptr = np.zeros(nets + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum([len(p) for p in pins])
    hg = H.Hypergraph.from_nets(nov, net_ptr, np.concatenate(pins).astype(np.uint32),
                                np.array([p[0] for p in pins], np.int32))
    print(f"cut nets: K={K} nets={nets} pins={hg.pins}", flush=True)
    with Engine(0) as eng:
        eng.upload(hg)
        eng.set_partition(K, part)
        eng.refine("CN", 3)
        got = eng.get_state()
    st = O.build_state(hg, K, part)
    st.sizes = st.sizes.astype(np.int32)
    O.cn_refine(hg, st, 3, serial=False)
    for k in ("part", "ep_ends", "ep_parts", "ep_cnt"):
        assert np.array_equal(getattr(got, k), getattr(st, k)), k
    assert np.array_equal(got.sizes, st.sizes.astype(np.int64))
