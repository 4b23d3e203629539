"""The streaming initial partition's sub-rounds on either side of the sizes from
which their touched nets go to the apply as a list (262,144 nets, 32 nets a
slot): rounds just below and above, hub vertices of more than 64 nets, K
through the masks, past them, and past the apply's index. Bit-exact against
the oracle."""
import numpy as np
import pytest

from fastpartitioner_amd import hypergraph as H
from fastpartitioner_amd.engine import Engine
from oracle import oracle as O
from oracle_refine import assert_same_state

pytestmark = pytest.mark.gpu


def _graph(noe, nov, seed):
    """noe nets of 1 to 4 pins, some of 9, 70 and 300; vertices 0 to 3 in 64, 65, 128 and 700 of them."""
    rng = np.random.default_rng(seed)
    sizes = rng.integers(1, 5, noe)
    sizes[rng.choice(noe, 60, replace=False)] = np.repeat([9, 70, 300], 20)
    n = np.repeat(np.arange(noe), sizes)
    v = rng.integers(4, nov, n.size)
    for h, d in enumerate((64, 65, 128, 700)):
        n = np.concatenate([n, rng.choice(noe, d, replace=False)])
        v = np.concatenate([v, np.full(d, h)])
    key = np.unique(n.astype(np.int64) * nov + v)
    n, v = key // nov, key % nov
    net_ptr = np.zeros(noe + 1, dtype=np.uint32)
    net_ptr[1:] = np.cumsum(np.bincount(n, minlength=noe))
    src = v[net_ptr[:-1].astype(np.int64)].astype(np.int32)
    return H.Hypergraph.from_nets(nov, net_ptr, v.astype(np.uint32), src)


@pytest.mark.parametrize("noe", [262_143, 262_144, 262_209])
def test_stream_around_the_list_rule(noe):
    hg = _graph(noe, 40_000, noe % 7)
    for K, mode, R in ((5, 0, 8_192), (5, 0, 8_193), (300, 1, 5_000), (40, 2, 6_000), (700, 1, 8_000), (2_440, 1, 8_192)):
        name = ("ldg_bands", "ldg", "cn_ldg")[mode]
        C, max_pw, cap = 1.2 * hg.nov / K, int(1.4 * hg.nov / K) + 1, int(1.2 * hg.nov / K) + 8
        print(f"stream: nets={noe} K={K} {name} R={R} pins={hg.pins}", flush=True)
        with Engine(0) as eng:
            eng.upload(hg)
            eng.initial_partition(mode, K, R, C, max_pw, cap)
            got = eng.get_state()
        st, _ = O.round_ldg(hg, K, name, C, max_pw, R, cap)
        assert_same_state(got, st)
