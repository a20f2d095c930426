"""The row-pair search (tori with rows of at most 6 sites) and the run search
(chains) against the oracle's element-by-element state_info, bit for bit:
representatives, characters and norms, over lattice shapes at the edges of the
searches' ranges, both spin-inversion characters, sectors with characters -1,
and states with large stabilisers."""
import numpy as np
import pytest

import lsamd
from lsamd import models
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def torus(lx, ly, point="full"):
    """Translations of the lx x ly torus (site r * lx + c), with its reflections
    ("full": and the rotation where lx = ly), both combined ("c2"), the
    rotation alone ("c4"), or none."""
    site = lambda r, c: (r % ly) * lx + c % lx  # noqa: E731
    table = lambda f: np.array([f(r, c) for r in range(ly) for c in range(lx)], dtype=np.int32)  # noqa: E731
    gens = [table(lambda r, c: site(r, c + 1)), table(lambda r, c: site(r + 1, c))]
    if point == "full":
        gens += [table(lambda r, c: site(r, -1 - c)), table(lambda r, c: site(-1 - r, c))]
    if point == "c2":
        gens += [table(lambda r, c: site(-1 - r, -1 - c))]
    if point == "mirror":
        gens += [table(lambda r, c: site(r, -1 - c))]
    if point in ("full", "c4") and lx == ly:
        gens += [table(lambda r, c: site(c, -1 - r))]
    return gens


def chain(n, parity=True):
    return [models.chain_translation(n)] + ([models.chain_parity(n)] if parity else [])


CASES = []
for shape in [(2, 2), (3, 3), (4, 4), (5, 5), (6, 6), (6, 2), (2, 6), (3, 6), (6, 4), (4, 8), (5, 3), (6, 5), (6, 8),
              (7, 4), (8, 3), (2, 9)]:
    CASES.append((f"torus{shape[0]}x{shape[1]}", torus(*shape), None))
for point in ("c2", "c4", "mirror", "none"):
    CASES.append((f"torus4x4-{point}", torus(4, 4, point), None))
    CASES.append((f"torus6x6-{point}", torus(6, 6, point), None))
CASES.append(("torus4x4-pi", torus(4, 4), [2, 2, 0, 0, 0]))
CASES.append(("torus4x4-b1", torus(4, 4), [0, 0, 1, 1, 0]))
CASES.append(("torus6x6-pi-b2", torus(6, 6), [3, 3, 1, 1, 2]))
for n in (2, 3, 5, 8, 9, 16, 17, 31, 32, 33, 40, 63, 64):
    CASES.append((f"chain{n}", chain(n), None))
    CASES.append((f"chain{n}-t", chain(n, False), None))
CASES.append(("chain32-pi", chain(32), [16, 1]))
CASES.append(("chain12-p-", chain(12), [0, 1]))


def states_of(n, rng):
    full = (1 << n) - 1
    special = [0, full, 1, full >> 1, full ^ 1]
    for period in range(1, n):
        if n % period == 0:
            for word in range(min(1 << period, 64)):
                special.append(sum(word << (period * k) for k in range(n // period)))
    special += [1 << k for k in range(n)] + [((1 << k) - 1) for k in range(n)]
    drawn = [int(x) & int(y) if k % 3 == 0 else int(x)
             for k, (x, y) in enumerate(rng.integers(0, full, size=(4000, 2), endpoint=True, dtype=np.uint64))]
    return np.unique(np.array([x & full for x in special + drawn], dtype=np.uint64))


@pytest.mark.parametrize("name,gens,sectors", CASES, ids=[c[0] for c in CASES])
def test_search_equals_the_element_by_element_reduction(engine, name, gens, sectors):
    n = len(gens[0])
    S = lsamd.Symmetries([lsamd.Symmetry(g, s) for g, s in zip(gens, sectors or [0] * len(gens))])
    xs = states_of(n, np.random.default_rng(n))
    for si in (None, 1, -1):
        og = O.Group(n, S.elements(), S.characters.real, S.characters.imag, si or 0)
        basis = lsamd.DeviceBasis(n, None if si is None else n // 2, si, S)
        print(name, si, xs.size, flush=True)
        got = basis.state_info(xs)
        reps, chars, norms = og.state_info(xs)
        assert np.array_equal(got[0], reps)
        assert np.array_equal(got[1], chars)
        assert np.array_equal(got[2], norms)
