"""The prefix table of the state index on both sides of the size at which its
entries share their searches (2^20 entries: about 262 144 states): every listed
state has its place and no other state has one."""
import numpy as np
import pytest

import lsamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 1000, 262144, 262145, 600000])
def test_index_of_listed_and_other_states(engine, count):
    bits = 40
    rng = np.random.default_rng(count)
    drawn = rng.integers(0, 1 << bits, size=2 * count + 64, dtype=np.uint64)
    clustered = np.arange(2 * count + 64, dtype=np.uint64) + (np.uint64(3) << np.uint64(bits - 3))
    for xs in (drawn, clustered):
        xs = rng.permutation(np.unique(xs))
        listed, other = np.sort(xs[:count]), xs[count:]
        basis = lsamd.DeviceBasis(bits)
        basis.set_states(listed)
        print(count, listed.size, flush=True)
        assert np.array_equal(basis.index(listed), np.arange(listed.size))
        assert np.all(basis.index(other) == -1)
