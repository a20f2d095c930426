"""The split enumeration of tori (upper and lower rows listed apart) against
the element-by-element filter, over shapes, fillings, sectors and ranges."""
import numpy as np
import pytest

import lsamd
from test_gpu_orbit_search import torus

pytestmark = pytest.mark.gpu

# lx, ly, weight, spin inversion, point group, sectors of its generators
CASES = [
    (5, 5, 12, None, "full", None),
    (5, 5, 11, None, "c4", None),
    (5, 5, 13, None, "full", [0, 0, 1, 1, 2]),
    (4, 7, 14, 1, "full", None),
    (4, 7, 14, -1, "c2", None),
    (4, 7, 9, None, "none", None),
    (6, 5, 15, 1, "full", [3, 0, 0, 0]),
    (6, 5, 8, None, "mirror", [3, 0, 1]),
    (5, 6, 15, -1, "full", None),
    (3, 8, 12, 1, "full", None),
    (4, 8, 8, None, "full", None),
    (6, 6, 7, None, "full", [3, 3, 1, 1, 2]),
    (6, 6, 6, None, "c4", None),
    (2, 8, 8, 1, "full", None),
    (2, 2, 2, 1, "full", None),
    (3, 3, 1, None, "full", None),
    (4, 4, 0, None, "full", None),
    (4, 4, 16, None, "c4", None),
    (6, 2, 6, -1, "full", None),
    (6, 6, 1, None, "full", None),
    (6, 6, 35, None, "none", None),
]


def states(case, filtered, bounds=None):
    lx, ly, weight, inversion, point, sectors = case
    gens = torus(lx, ly, point)
    S = lsamd.Symmetries([lsamd.Symmetry(g, s) for g, s in zip(gens, sectors or [0] * len(gens))])
    basis = lsamd.DeviceBasis(lx * ly, weight, inversion, S)
    lsamd.load().ls_amd_set_factored_enumeration(0 if filtered else 1)
    try:
        basis.build(*(bounds or ()))
    finally:
        lsamd.load().ls_amd_set_factored_enumeration(1)
    return basis.states


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[:5])))
def test_split_lists_the_same_states(engine, case):
    print(case, flush=True)
    want = states(case, True)
    assert np.array_equal(states(case, False), want)


def test_split_keeps_to_a_range(engine):
    case = (5, 6, 15, 1, "full", None)
    every = states(case, True)
    low, high = int(every[every.size // 7]), int(every[-every.size // 5])
    want = every[(every >= low) & (every <= high)]
    assert np.array_equal(states(case, False, (low, high)), want)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[:5])))
def test_small_sectors_by_either_enumeration(engine, case):
    """Sectors too small for the split to pay take the filter; forced onto the
    split they list the same states."""
    print(case, flush=True)
    want = states(case, True)
    lib = lsamd.load()
    for mode in (1, 2):
        lib.ls_amd_set_factored_enumeration(mode)
        try:
            lx, ly, weight, inversion, point, sectors = case
            gens = torus(lx, ly, point)
            S = lsamd.Symmetries([lsamd.Symmetry(g, s) for g, s in zip(gens, sectors or [0] * len(gens))])
            basis = lsamd.DeviceBasis(lx * ly, weight, inversion, S)
            basis.build()
        finally:
            lib.ls_amd_set_factored_enumeration(1)
        assert np.array_equal(basis.states, want)
