"""The table search of spinful fermion groups against the oracle's
element-by-element state_info (bit for bit), its enumeration against the
element-by-element filter, and its matrices against the element-by-element
fill: lattices of 1 to 16 sites, sectors with characters -1, fillings from
empty to full, and a group that has to keep the general path."""
import numpy as np
import pytest

import lsamd
from lsamd import models
from oracle import oracle as O
from test_gpu_orbit_search import chain, torus

pytestmark = pytest.mark.gpu

CASES = [
    ("chain2", chain(2), None),
    ("chain3", chain(3), None),
    ("chain5-t", chain(5, False), None),
    ("chain8", chain(8), [4, 1]),
    ("chain16", chain(16), None),
    ("chain16-pi", chain(16), [8, 0]),
    ("torus2x2", torus(2, 2), None),
    ("torus3x3", torus(3, 3), [0, 0, 1, 1, 0]),
    ("torus3x4", torus(3, 4), None),
    ("torus4x4", torus(4, 4), None),
    ("torus4x4-pi", torus(4, 4), [2, 2, 1, 1, 2]),
    ("torus4x4-c4", torus(4, 4, "c4"), [0, 0, 2]),
    ("chain6-complex", chain(6, False), [1]),
]


def spinful(gens, n):
    return [np.concatenate([g, g + n]).astype(np.int32) for g in gens]


def oracle_group(n, S):
    og = O.Group(2 * n, S.elements(), S.characters.real, S.characters.imag, 0)
    O.lib().ora_group_set_fermionic.argtypes = [O.C.c_void_p, O.C.c_int]
    assert O.lib().ora_group_set_fermionic(og.h, 2) == 0
    return og


def fillings(n):
    return sorted({(0, 0), (n // 2, n // 2), (1, n - 1), (n, 1), (n // 2, max(n // 2 - 1, 0))})


@pytest.mark.parametrize("name,gens,sectors", CASES, ids=[c[0] for c in CASES])
def test_species_search(engine, name, gens, sectors):
    n = len(gens[0])
    S = lsamd.Symmetries([lsamd.Symmetry(g, s) for g, s in zip(spinful(gens, n), sectors or [0] * len(gens))])
    og = oracle_group(n, S)
    rng = np.random.default_rng(n)
    xs = rng.integers(0, 1 << (2 * n), size=4000, dtype=np.uint64)
    periodic = np.array([sum(w << (p * k) for k in range(n // p)) for p in range(1, n + 1) if n % p == 0
                         for w in range(min(1 << p, 32))], dtype=np.uint64)
    xs = np.unique(np.concatenate([xs, (periodic[:, None] << np.uint64(n) | periodic[None, :]).ravel()]))
    print(name, xs.size, flush=True)
    basis = lsamd.DeviceBasis.fermions(n, n // 2, n // 2, S)
    got, want = basis.state_info(xs), og.state_info(xs)
    for g, w in zip(got, want):
        assert np.array_equal(g, w, equal_nan=g.dtype.kind != "u")


@pytest.mark.parametrize("name,gens,sectors", CASES, ids=[c[0] for c in CASES])
def test_species_basis_and_matrix(engine, name, gens, sectors):
    n = len(gens[0])
    S = lsamd.Symmetries([lsamd.Symmetry(g, s) for g, s in zip(spinful(gens, n), sectors or [0] * len(gens))])
    lib = lsamd.load()
    hops = [(i, (i + 1) % n) for i in range(n)] if name.startswith("chain") else \
        sorted({tuple(sorted((i, int(g[i])))) for g in gens[:2] for i in range(n)})
    expr = models.hubbard(n, [b for b in hops if b[0] != b[1]], t=1.0, U=4.0)
    for up, down in fillings(n):
        print(name, up, down, flush=True)
        bases = []
        for on in (1, 0):
            lib.ls_amd_set_factored_enumeration(on)
            b = lsamd.DeviceBasis.fermions(n, up, down, S)
            if name.endswith("complex"):
                b.set_norm_tolerance(1e-9)
            b.build()
            bases.append(b)
        lib.ls_amd_set_factored_enumeration(1)
        assert np.array_equal(bases[0].states, bases[1].states)
        size = bases[0].number_states
        if size == 0 or size > 200000:
            continue
        fast, slow = lsamd.DeviceOperator(bases[0], expr), lsamd.DeviceOperator(bases[0], expr)
        slow.set_factored(False)
        for op in (fast, slow):
            op.set_csr_packing(False)
            op.build_csr(128)
        for a, b in zip(fast.csr_arrays(), slow.csr_arrays()):
            assert np.array_equal(a, b)


def test_species_basis_takes_little_scratch(engine):
    """A trivial group on 16 sites lists every product: 23 M states, whose
    scratch has to stay far below their own 8 bytes each."""
    n = 16
    S = lsamd.Symmetries([lsamd.Symmetry(np.arange(2 * n, dtype=np.int32), 0)])
    basis = lsamd.DeviceBasis.fermions(n, 4, 8, S)
    lsamd.device_trim()
    basis.build()
    assert lsamd.device_trim() <= basis.number_states
    states = basis.states
    assert basis.number_states == 1820 * 12870
    assert np.all(np.diff(states.view(np.int64)) > 0)
    low = np.uint64((1 << n) - 1)
    for species, weight in ((states & low, 4), (states >> np.uint64(n), 8)):
        assert np.all(np.unpackbits(species.view(np.uint8).reshape(-1, 8), axis=1).sum(axis=1) == weight)
