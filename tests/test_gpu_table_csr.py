"""The value-table CSR build (targets counted and placed by the fill pass)
against the general build: the same rows, columns, values and products, at
the edges of its formats -- 256 and 257 distinct values, rows of one entry to
more than the register sort takes, a target row too long for its place bits,
and rows of a wave that end inside it."""
import numpy as np
import pytest

import lsamd
from lsamd import models
from lsamd.expr import Expr, Term, sigma_minus, sigma_plus, sum_exprs

pytestmark = pytest.mark.gpu


def basis(n, weight=None, group=False, inversion=None):
    S = None
    if group:
        S = lsamd.Symmetries([lsamd.Symmetry(models.chain_translation(n), 0), lsamd.Symmetry(models.chain_parity(n), 0)])
    b = lsamd.DeviceBasis(n, weight, inversion, S)
    b.build()
    return b


def fields(n, couplings):
    return sum_exprs((sigma_plus(i) + sigma_minus(i)) * c for i, c in zip(range(n), couplings))


def collective(n):
    """Every state of one flipped spin goes to |0...01>: row 0 gets them all."""
    return sum_exprs(sigma_minus(i) * sigma_plus(0) * (1.0 + (i % 3)) for i in range(1, n))


CASES = {
    "chain16": lambda: (basis(16, 8, True, 1), models.j1j2_chain(16)),
    "chain13": lambda: (basis(13, 5, True), models.j1j2_chain(13)),
    "chain9-all": lambda: (basis(9), models.heisenberg_chain(9)),
    "field12": lambda: (basis(12), fields(12, [0.5 + i for i in range(12)])),
    "two-states": lambda: (basis(2, 1), models.heisenberg_chain(2)),
    "values256": lambda: (basis(24, 2), pair_hops(24, 128)),
    "values257": lambda: (basis(24, 2), pair_hops(24, 129)),
    "collective60": lambda: (basis(60, 1), collective(60)),
    "flips300": lambda: (basis(10), all_flips(10, 300)),
    "flips1023": lambda: (basis(10), all_flips(10, 1023)),
    "flips4500": lambda: (basis(13), all_flips(13, 4500)),
}


def pair_hops(n, count):
    """`count` hops with couplings of their own, both directions: 2 x count values at most."""
    pairs = [(i, j) for i in range(n) for j in range(i + 1, n)][:count]
    return sum_exprs(sigma_plus(i) * sigma_minus(j) * (1.0 + 0.25 * k) + sigma_plus(j) * sigma_minus(i) * (-1.0 - 0.25 * k)
                     for k, (i, j) in enumerate(pairs))


def all_flips(n, count):
    """Flips of `count` subsets of the sites: rows of `count` entries."""
    out = {}
    for mask in range(1, count + 1):
        t = Term(0.5 + mask % 7, 0, 0, 0, mask, 0)
        out[(t.m, t.l, t.r, t.x, t.s)] = t.v
    return Expr(out)


@pytest.mark.parametrize("name", CASES)
def test_table_build_equals_the_general_build(engine, name):
    b, expr = CASES[name]()
    print(name, b.number_states, flush=True)
    table, plain = lsamd.DeviceOperator(b, expr), lsamd.DeviceOperator(b, expr)
    plain.set_csr_packing(False)
    assert table.build_csr(96) == plain.build_csr(96)
    for got, want in zip(table.csr_arrays(), plain.csr_arrays()):
        assert np.array_equal(got, want)
    x = np.random.default_rng(1).standard_normal(b.number_states)
    assert np.array_equal(table.matvec(x, "csr"), plain.matvec(x, "csr"))
    # the fused product adds a row's L entries in another order: each of the L
    # sums rounds by at most eps times the sum of L products
    longest = 1 + np.diff(plain.csr_arrays()[0]).max(initial=0)
    scale = max(np.abs(a).max(initial=0) for a in plain.csr_arrays()[2:]) * np.abs(x).max()
    bound = np.finfo(float).eps * longest ** 2 * scale
    assert np.abs(table.matvec(x, "otf") - plain.matvec(x, "csr")).max() <= bound


def projected_flips(count):
    """`count` distinct values: term k flips bits above the low six where these
    hold k mod 64, so a row has count / 64 entries."""
    out = {}
    for k in range(count):
        low = k % 64
        x = (k // 64 + 1) << 6
        out[(63, low, low, x, 0)] = 1.0 + k / 4096.0
    return Expr(out)


def conditional_hops(n):
    """Hops i -> j that ask for a third site up or down, each with a coupling of its own."""
    out = {}
    for i in range(n):
        for j in range(n):
            if i == j:
                continue
            k = next(q % n for q in range(max(i, j) + 1, max(i, j) + 4) if q % n not in (i, j))
            for up in (0, 1):
                m, r = 1 << i | 1 << j | 1 << k, 1 << i | up << k
                out[(m, r ^ 1 << i ^ 1 << j, r, 1 << i | 1 << j, 0)] = 1.0 + len(out) / 4096.0
    return Expr(out)


# More workgroups than fit the chip at once, so that some start before and some
# after the value hash is found full: without a group on both sides of its
# limit, and with the row-pair search staged beside the terms (576 elements;
# 2520 couplings times at least two norm ratios).
FULL_HASH = {
    "values4096": (lambda: (basis(16), projected_flips(4096)), 4096),
    "values4097": (lambda: (basis(16), projected_flips(4097)), None),
    "torus6x6": (lambda: (torus_basis(6, 7), conditional_hops(36)), None),
}


def torus_basis(side, weight):
    S = lsamd.Symmetries([lsamd.Symmetry(g, 0) for g in models.square_generators(side)])
    b = lsamd.DeviceBasis(side * side, weight, None, S)
    b.build()
    return b


@pytest.mark.parametrize("name", FULL_HASH)
def test_a_full_value_hash_leaves_the_general_build(engine, name):
    make, distinct = FULL_HASH[name]
    b, expr = make()
    print(name, b.number_states, flush=True)
    plain = lsamd.DeviceOperator(b, expr)
    plain.set_csr_packing(False)
    nnz = plain.build_csr(64)
    want = plain.csr_arrays()
    for _ in range(3):
        op = lsamd.DeviceOperator(b, expr)
        assert op.build_csr(64) == nnz
        info = op.csr_info
        assert not info["packed"]
        assert (info["wide"], info["table_size"]) == ((True, distinct) if distinct else (False, 0))
        for got, ref in zip(op.csr_arrays(), want):
            assert np.array_equal(got, ref)
    if distinct is None:
        assert np.unique(want[2]).size > 4096


def test_a_full_value_hash_still_reports_states_outside_the_basis(engine):
    b = basis(16, 8)
    op = lsamd.DeviceOperator(b, projected_flips(4097))
    for _ in range(2):
        with pytest.raises(lsamd.EngineError, match="invalid index"):
            op.build_csr(64)
    good = lsamd.DeviceOperator(b, models.heisenberg_chain(16))
    assert good.build_csr(64) > 0


def test_a_long_row_of_few_values_is_still_packed(engine):
    """The table pass gives up on a row too long for its tags; the general
    build then packs the few values."""
    b, expr = CASES["flips4500"]()
    op = lsamd.DeviceOperator(b, expr)
    op.build_csr(64)
    info = op.csr_info
    assert info["packed"] and info["table_size"] == len(set(expr.terms.values()))


def same_target_hops(count, seed):
    """`count` terms, all of which take the one-particle orbit of the 4x4
    lattice to itself: hops from site 0 with other sites asked to be empty."""
    values = np.random.default_rng(seed).permutation(count) / 1024.0 + 1.0
    out = {}
    for q in range(count):
        j, sub = 1 + q % 15, q // 15
        rest = [s for s in range(1, 16) if s != j]
        m = 1 | 1 << j | sum((sub >> p & 1) << s for p, s in enumerate(rest))
        out[(m, 1 << j, 1, 1 | 1 << j, 0)] = float(values[q])
    return Expr(out)


@pytest.mark.parametrize("count", [2, 63, 64, 65, 66, 300, 1024, 1025, 3000])
def test_many_entries_of_one_column_in_ascending_value(engine, count):
    """Both builds list a column's entries in ascending value, whatever sort a
    run of them takes (one row of `count` entries)."""
    b = torus_basis(4, 1)
    expr = same_target_hops(count, count)
    for packing in (True, False):
        op = lsamd.DeviceOperator(b, expr)
        op.set_csr_packing(packing)
        assert op.build_csr(64) == count
        rows, cols, vals, _ = op.csr_arrays()
        assert list(rows) == [0, count] and not cols.any()
        assert np.array_equal(vals, np.sort(np.array(list(expr.terms.values())).real))


@pytest.mark.parametrize("count", [1, 2, 4, 5, 63, 64, 65, 300])
def test_values_met_by_all_waves_at_once_are_counted_once(engine, count):
    """`count` values over 1024 terms: up to kGroups (4) values of a wave are
    inserted by one lane each, further ones by every lane that holds them."""
    b = basis(16)
    values = [1.0 + (k % count) / 512.0 for k in range(1024)]
    expr = Expr(dict(zip(projected_flips(1024).terms, values)))
    plain = lsamd.DeviceOperator(b, expr)
    plain.set_csr_packing(False)
    nnz = plain.build_csr(64)
    for _ in range(3):
        op = lsamd.DeviceOperator(b, expr)
        assert op.build_csr(64) == nnz
        assert op.csr_info["table_size"] == count
        for got, want in zip(op.csr_arrays(), plain.csr_arrays()):
            assert np.array_equal(got, want)
