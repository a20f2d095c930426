"""The engine's work as measured cases: what a program that diagonalises
lattice models asks of it, through the Python layer's public entry points.

A case is one call (or the few calls that belong together) on one model:

  basis       DeviceBasis.build: enumerate the representatives of a sector
  setup       a new operator's CSR and its first product
  onthefly    a product without a stored matrix (real, or complex fermions)
  product     a product with the stored CSR: FP64 vector, FP32 or FP64 block
  sectors     one product over every (momentum, spin inversion) sector
  host        the reference's entry point: host x in, host y out
  stateinfo   the reference's batched state_info on host arrays
  ground      the ground-state energy by the block eigensolver

Models: the Heisenberg chain (J2 > 0: J1-J2) with translations and parity,
the J1-J2 square lattice with translations and point group, both with spin
inversion where half filling allows it, and the Hubbard model on the square
lattice.  "random" couplings give every bond its own J, so the stored matrix
has many distinct values.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "lattice-symmetries_amd"))

import lsamd  # noqa: E402
from lsamd import models, sectors  # noqa: E402
from lsamd.expr import heisenberg_bond, sum_exprs  # noqa: E402

HOPPING, REPULSION = 1.0, 4.0


# --- models -----------------------------------------------------------------

def _spin(kind, lattice, size, weight=None, j2=0.5, couplings="uniform", **more):
    sites = size if lattice == "chain" else size * size
    w = sites // 2 if weight is None else weight
    return {"kind": kind, "lattice": lattice, "size": size, "weight": w,
            "inversion": 2 * w == sites and sites % 2 == 0, "j2": j2, "couplings": couplings, **more}


def _hubbard(kind, size, up, down, **more):
    return {"kind": kind, "lattice": "hubbard", "size": size, "up": up, "down": down, **more}


def _sites(case):
    return case["size"] if case["lattice"] == "chain" else case["size"] ** 2


def _bits(case):
    return 2 * _sites(case) if case["lattice"] == "hubbard" else _sites(case)


def _generators(case):
    n = case["size"]
    if case["lattice"] == "chain":
        return [models.chain_translation(n), models.chain_parity(n)]
    gens = models.square_generators(n)
    if case["lattice"] == "hubbard":
        gens = [np.concatenate([g, g + n * n]).astype(np.int32) for g in gens]
    return gens


def _bonds(case):
    """(i, j, J) of every bond."""
    n = case["size"]
    if case["lattice"] == "chain":
        near = [(i, (i + 1) % n) for i in range(n)]
        far = [(i, (i + 2) % n) for i in range(n)]
    else:
        at = lambda r, c: (r % n) * n + c % n  # noqa: E731
        near = [b for r in range(n) for c in range(n) for b in ((at(r, c), at(r, c + 1)), (at(r, c), at(r + 1, c)))]
        far = [b for r in range(n) for c in range(n)
               for b in ((at(r, c), at(r + 1, c + 1)), (at(r, c), at(r + 1, c - 1)))]
    bonds = [(i, j, 1.0) for i, j in near]
    if case["lattice"] != "hubbard" and case["j2"] != 0.0:
        bonds += [(i, j, case["j2"]) for i, j in far]
    if case.get("couplings") == "random":
        u = np.random.default_rng(7).random(len(bonds)) - 0.5
        bonds = [(i, j, J * (1.0 + 0.5 * u[k])) for k, (i, j, J) in enumerate(bonds)]
    return bonds


def _expression(case):
    bonds = _bonds(case)
    if case["lattice"] == "hubbard":
        return models.hubbard(_sites(case), [(i, j) for i, j, _ in bonds], t=HOPPING, U=REPULSION)
    return sum_exprs([heisenberg_bond(i, j, J) for i, j, J in bonds])


def _sectors_of(case, seed):
    """One of the lattice's real sectors: the phase of every generator, and the
    spin-inversion eigenvalue (None without)."""
    n = case["size"]

    def choose(options):
        nonlocal seed
        seed, at = divmod(seed, len(options))
        return options[at]

    reflection = choose([0, 1])
    translation = choose([0, n // 2]) if n % 2 == 0 else 0
    inversion = choose([1, -1]) if case.get("inversion") else None
    rotation = choose([0, 2])
    if case["lattice"] == "chain":
        return [translation, reflection], inversion
    return [translation, translation, reflection, reflection, rotation], inversion


def _symmetric_sector(case):
    return [0] * len(_generators(case)), 1 if case.get("inversion") else None


def _symmetries(case, phases):
    return lsamd.Symmetries([lsamd.Symmetry(g, p) for g, p in zip(_generators(case), phases)])


def _device_basis(case, symmetries, inversion):
    if case["lattice"] == "hubbard":
        return lsamd.DeviceBasis.fermions(_sites(case), case["up"], case["down"], symmetries)
    return lsamd.DeviceBasis(_sites(case), case["weight"], inversion, symmetries)


# --- the cases ---------------------------------------------------------------

def listed():
    return [
        # a scan over sectors starts with the basis: the flagship 6x6 lattice
        # (4.5 G candidates, 15.8 M representatives), and a fermionic sector
        # whose group carries signs (131 M candidates)
        {"name": "basis-square6", **_spin("basis", "square", 6)},
        {"name": "basis-hubbard4", **_hubbard("basis", 4, 7, 7)},
        # the largest: a new Hamiltonian on a built basis, up to its first
        # product (every change of a coupling pays this)
        {"name": "setup-square6", **_spin("setup", "square", 6)},
        # products where no matrix is stored: a long chain, and the complex
        # product of a fermionic sector
        {"name": "onthefly-chain32", **_spin("onthefly", "chain", 32, j2=0.0)},
        {"name": "onthefly-hubbard4", **_hubbard("onthefly", 4, 7, 7)},
        # the smallest call of a Krylov loop: 257 states, latency only
        {"name": "product-chain16", **_spin("product", "chain", 16, j2=0.0, columns=1, bits=64)},
        # the product of a Krylov loop at full size, one FP64 vector and the
        # FP32 block of the mixed-precision eigensolver
        {"name": "product-square6", **_spin("product", "square", 6, columns=1, bits=64)},
        {"name": "product-square6-f32x8", **_spin("product", "square", 6, columns=8, bits=32)},
        # all momenta and spin-inversion sectors of a chain in one product
        {"name": "sectors-chain26", **_spin("sectors", "chain", 26, columns=8, bits=32)},
        # the drop-in entry points on host memory: a product as scipy's eigsh
        # drives it, and state_info on the reference's batch of 10 240 states
        {"name": "host-square6", **_spin("host", "square", 6)},
        {"name": "stateinfo-square6", **_spin("stateinfo", "square", 6, batch=10240)},
        # the whole calculation, mixed precision, on a stored matrix
        {"name": "ground-square6", **_spin("ground", "square", 6)},
    ]


def _drawn_model(rng, kind, shortest, longest, random_couplings=True, **more):
    """A chain (its length spreads the work over a logarithmic scale) or a
    square lattice, odd sizes and fillings off one half among them."""
    couplings = rng.choice(["uniform", "uniform", "random"]) if random_couplings else "uniform"
    if rng.random() < 0.35:
        size = rng.choice([4, 5, 6] if longest >= 28 else [4, 5])
        weight = rng.choice([18, 18, 13, 11, 9] if size == 6 else [None, None, size * size // 2 - 1])
        return _spin(kind, "square", size, weight=weight, couplings=couplings, **more)
    size = rng.randint(shortest, longest)
    return _spin(kind, "chain", size, weight=rng.choice([None, None, size // 2 - 1, size // 3]),
                 j2=rng.choice([0.0, 0.5, 0.2411]), couplings=couplings, **more)


def draw(rng):
    kind = rng.choice(["basis", "setup", "onthefly", "product", "product", "sectors", "host", "stateinfo", "ground"])
    if kind in ("basis", "onthefly") and rng.random() < 0.25:
        size = rng.choice([3, 4])
        return _hubbard(kind, size, rng.randint(2, size * size // 2), rng.randint(2, size * size // 2))
    if kind == "product":
        columns, bits = rng.choice([(1, 64), (1, 64), (8, 32), (4, 32), (2, 32), (1, 32), (2, 64), (4, 64), (8, 64)])
        return _drawn_model(rng, kind, 10, 30, columns=columns, bits=bits)
    if kind == "sectors":
        return _spin(kind, "chain", 2 * rng.randint(4, 12), j2=rng.choice([0.0, 0.5]),
                     columns=rng.choice([1, 2, 4, 8, 8]), bits=rng.choice([32, 32, 64]))
    if kind == "stateinfo":
        return _drawn_model(rng, kind, 8, 32, batch=int(round(2 ** rng.uniform(0, 18))))
    if kind == "ground":
        return _drawn_model(rng, kind, 16, 28, random_couplings=False)
    return _drawn_model(rng, kind, 10, 32 if kind == "basis" else 30)


# --- inputs -------------------------------------------------------------------

class _Buffer:
    """A device tensor as the engine's entry points take it."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()


class _States:
    """The device list of a built basis; keeps the basis alive."""

    def __init__(self, basis):
        self.basis = basis
        self.__cuda_array_interface__ = {
            "shape": (basis.number_states,), "typestr": "<i8", "version": 3, "strides": None,
            "data": (lsamd.load().ls_amd_basis_states_device(basis.handle), False)}


def _room(case):
    """Places for the list of any of the case's sectors."""
    return int(1.05 * _shape(case)[0]) + 4096


def _keep(room, states):
    """A sector's list in its row of a scan's table, filled up with -1."""
    count = 0 if states is None else states.numel()
    if count:
        room[:count].copy_(states)
    room[count:].fill_(-1)
    return room


def _normal(shape, bits, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32 if bits == 32 else torch.float64)


def _sector_input(n, case, seed):
    return _normal((n, 2, case["columns"]), case["bits"], seed)  # [state][re | im][column]


def _random_states(case, seed):
    """States of the sector's weight, in any order: what H makes of a batch of
    representatives."""
    rng = np.random.default_rng(seed)
    n, w, count = _sites(case), case["weight"], case["batch"]
    order = np.argsort(rng.random((count, n)), axis=1)[:, :w]
    return np.bitwise_or.reduce(np.uint64(1) << order.astype(np.uint64), axis=1)


def _ground_case(case, seed):
    """A point of a scan over the second-neighbour coupling."""
    return {**case, "j2": 0.45 + 0.1 * float(np.random.default_rng(seed).random())}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sectors":
        batch = sectors.chain_sector_batch(case["size"], case["weight"], _expression(case))
        batch.autotune(case["columns"])
        x = _sector_input(batch.number_states, case, seed)
        return {"kind": kind, "batch": batch, "columns": case["columns"], "bits": case["bits"],
                "x": _Buffer(x), "y": _Buffer(torch.zeros_like(x))}
    phases, inversion = _sectors_of(case, seed) if kind == "basis" else _symmetric_sector(case)
    symmetries = _symmetries(case, phases)
    if kind == "basis":
        room = torch.empty(_room(case), dtype=torch.int64, device="cuda")
        return {"kind": kind, "case": dict(case), "symmetries": symmetries, "inversion": inversion, "room": room}
    if kind in ("host", "stateinfo"):
        basis = lsamd.SpinBasis(_sites(case), case["weight"], inversion, symmetries)
        if kind == "stateinfo":
            return {"kind": kind, "basis": basis, "states": _random_states(case, seed)}
        basis.build()
        operator = lsamd.Operator(basis, _expression(case))
        x = np.random.default_rng(seed).standard_normal(basis.number_states)
        y = np.zeros_like(x)
        operator.matvec(x, out=y)  # the program's first product builds the cached operator
        return {"kind": kind, "operator": operator, "x": x, "y": y}
    basis = _device_basis(case, symmetries, inversion)
    n = basis.build()
    if kind == "ground":
        case = _ground_case(case, seed)
    expression = _expression(case)
    if kind == "setup":
        x = _normal((n,), 64, seed)
        return {"kind": kind, "basis": basis, "expression": expression, "x": _Buffer(x), "y": _Buffer(torch.zeros_like(x))}
    operator = lsamd.DeviceOperator(basis, expression)
    if kind == "onthefly":
        complex_values = case["lattice"] == "hubbard"
        x = _normal((n, 2) if complex_values else (n,), 64, seed)
        return {"kind": kind, "operator": operator, "complex": complex_values,
                "x": _Buffer(x), "y": _Buffer(torch.zeros_like(x))}
    operator.build_csr(96)
    if kind == "ground":
        return {"kind": kind, "operator": operator, "seed": int(seed) % (1 << 31)}
    x = _normal((n,) if case["columns"] == 1 else (n, case["columns"]), case["bits"], seed)
    return {"kind": kind, "operator": operator, "columns": case["columns"], "bits": case["bits"],
            "x": _Buffer(x), "y": _Buffer(torch.zeros_like(x))}


def run(state):
    kind = state["kind"]
    if kind == "basis":
        basis = _device_basis(state["case"], state["symmetries"], state["inversion"])
        return _keep(state["room"], torch.as_tensor(_States(basis), device="cuda") if basis.build() else None)
    if kind == "setup":
        operator = lsamd.DeviceOperator(state["basis"], state["expression"])
        nonzeros = operator.build_csr(96)
        operator.csr_matvec(state["x"], state["y"])
        return {"nonzeros": nonzeros, "y": state["y"].tensor}
    if kind == "onthefly":
        if state["complex"]:
            state["operator"].matvec_complex(state["x"], state["y"])
        else:
            state["operator"].matvec_otf(state["x"], state["y"])
        return state["y"].tensor
    if kind == "product":
        if state["bits"] == 32:
            state["operator"].csr_matvec_f32(state["columns"], state["x"], state["y"])
        elif state["columns"] == 1:
            state["operator"].csr_matvec(state["x"], state["y"])
        else:
            state["operator"].csr_matvec_f64_block(state["columns"], state["x"], state["y"])
        return state["y"].tensor
    if kind == "sectors":
        state["batch"].matvec_device(state["columns"], state["x"], state["y"], state["bits"])
        return state["y"].tensor
    if kind == "host":
        return state["operator"].matvec(state["x"], out=state["y"])
    if kind == "stateinfo":
        return list(state["basis"].state_info(state["states"]))
    result = state["operator"].block_eigensolve(mode="fp32", block_size=2, nev=1, max_blocks=16, keep_blocks=4,
                                                tol=1e-8, switch_tol=1e-5, seed=state["seed"])
    return {"eigenvalues": result["eigenvalues"], "converged": result["converged"]}


# --- work ---------------------------------------------------------------------

def _choose(n, k):
    out = 1
    for i in range(k):
        out = out * (n - i) // (i + 1)
    return out


def _shape(case):
    """(states, off-diagonal entries) expected of a sector (over all sectors
    for "sectors"): free orbits, and the mean number of bonds that act."""
    n, bonds = _sites(case), len(_bonds(case))
    if case["lattice"] == "hubbard":
        up, down = case["up"], case["down"]
        dim = _choose(n, up) * _choose(n, down) / (8 * n)
        return dim, dim * bonds * sum(2 * k * (n - k) / (n * (n - 1)) for k in (up, down))
    w = case["weight"]
    group = 1 if case["kind"] == "sectors" else (2 if case["lattice"] == "chain" else 8) * n
    dim = _choose(n, w) / (group * (2 if case["inversion"] and case["kind"] != "sectors" else 1))
    return max(dim, 1.0), max(dim, 1.0) * bonds * 2 * w * (n - w) / (n * (n - 1))


def work(case):
    """The path's own inputs and outputs once: representatives (8 B each),
    vectors, and for a stored matrix its columns and values (one 32-bit word
    per entry where few values occur, 12 B of column and value otherwise)."""
    kind = case["kind"]
    dim, nnz = _shape(case)
    entry = 4.0 if case.get("couplings") == "uniform" else 12.0
    if kind == "basis":
        return {"bytes": 8 * dim, "flops": 0.0}
    if kind == "stateinfo":
        return {"bytes": 40.0 * case["batch"], "flops": 0.0}
    if kind == "setup":
        return {"bytes": 24 * dim + 2 * entry * nnz, "flops": 2 * nnz}
    if kind == "onthefly":
        width = 2 if case["lattice"] == "hubbard" else 1
        return {"bytes": (8 + 16 * width) * dim, "flops": 2 * nnz * width}
    if kind == "sectors":
        size = case["bits"] // 8
        return {"bytes": nnz * (4 + 2 * size) + dim * (8 + size + 4 * size * case["columns"]),
                "flops": 8 * nnz * case["columns"]}
    if kind == "product":
        size = case["bits"] // 8
        return {"bytes": nnz * entry + dim * (8 + size + 2 * size * case["columns"]), "flops": 2 * nnz * case["columns"]}
    if kind == "host":
        return {"bytes": nnz * entry + dim * 32, "flops": 2 * nnz}
    products = 60  # of two columns, until the residual is below the tolerance
    return {"bytes": products * (nnz * entry + dim * 32), "flops": products * 4 * nnz}


# --- the same in plain 64-bit torch ------------------------------------------

CHUNK = 12


class _Group:
    """Images of states under every element: tables over CHUNK bits at a time
    (fermion species: one table each, with the sign of its reordering)."""

    def __init__(self, n, perms, device, species=1):
        self.species = species
        self.size = len(perms)
        self.device = device
        per = n // species
        widths = [per] * species if species > 1 else [min(CHUNK, n - c) for c in range(0, n, CHUNK)]
        self.parts = []
        first = 0
        for width in widths:
            values = torch.arange(1 << width, device=device)
            images = torch.zeros(self.size, 1 << width, dtype=torch.int64, device=device)
            signs = torch.ones(self.size, 1 << width, dtype=torch.int64, device=device) if species > 1 else None
            for e, p in enumerate(perms):
                to = {int(b): i for i, b in enumerate(p)}  # bit b of x becomes bit to[b]
                for b in range(width):
                    images[e] |= ((values >> b) & 1) << to[first + b]
                if species > 1:
                    for a in range(width):
                        for b in range(a + 1, width):
                            if to[first + a] > to[first + b]:
                                signs[e] *= 1 - 2 * (((values >> a) & (values >> b)) & 1)
            self.parts.append((first, (1 << width) - 1, images, signs))
            first += width

    def image(self, e, x):
        y, s = None, None
        for first, mask, images, signs in self.parts:
            c = (x >> first) & mask
            y = images[e][c] if y is None else y | images[e][c]
            if signs is not None:
                s = signs[e][c] if s is None else s * signs[e][c]
        return y, None if s is None else s.to(torch.float64)

    def least(self, x, flip=0, flip_character=0, characters=None):
        """(orbit minimum, character of an element reaching it, stabiliser sum)."""
        best = x.clone()
        chi = None
        if characters is not None or self.species > 1 or flip_character < 0:
            chi = torch.ones(x.shape, dtype=torch.complex128, device=self.device)
        stab = torch.zeros(x.shape, dtype=torch.float64, device=self.device)
        for e in range(self.size):
            y, s = self.image(e, x)
            c = 1.0 if characters is None else complex(characters[e])
            for f in ((0, 1) if flip_character else (0,)):
                z = y ^ flip if f else y
                factor = c * (flip_character if f else 1)
                here = complex(factor).real if s is None else s * complex(factor).real
                stab += (z == x).to(torch.float64) * here
                if chi is None:
                    best = torch.minimum(best, z)
                    continue
                less = z < best
                best = torch.where(less, z, best)
                chi = torch.where(less, torch.full_like(chi, factor) if s is None else s.to(chi.dtype) * factor, chi)
        return best, chi, stab

    def is_least(self, x, flip=0):
        """x as a mask-free subset: the states no element maps below themselves."""
        for e in range(self.size):
            y, _ = self.image(e, x)
            keep = y >= x
            if flip:
                keep &= (y ^ flip) >= x
            x = x[keep]
            if x.numel() == 0:
                break
        return x


def _closure(gens, phases):
    """Every element of the group and its character."""
    def order(g):
        p, k = list(g), 1
        while p != list(range(len(g))):
            p, k = [p[int(i)] for i in g], k + 1
        return k

    factors = [np.exp(-2j * np.pi * s / order(g)) for g, s in zip(gens, phases)]
    found = {tuple(range(len(gens[0]))): 1.0 + 0j}
    new = list(found)
    while new:
        made = []
        for p in new:
            for g, f in zip(gens, factors):
                q = tuple(p[int(i)] for i in g)
                if q not in found:
                    found[q] = found[p] * f
                    made.append(q)
        new = made
    return list(found), [c.real if abs(c.imag) < 1e-9 else c for c in found.values()]


def _weight_states(n, w, device, pieces):
    """All n-bit states of weight w, ascending, in pieces."""
    low = min(16, n)
    values = torch.arange(1 << low, device=device)
    count = sum((values >> b) & 1 for b in range(low))
    lists = [values[count == k] for k in range(low + 1)]
    high = torch.arange(1 << (n - low), device=device)
    weight = sum(((high >> b) & 1 for b in range(n - low)), torch.zeros_like(high))
    gathered, total = [], 0
    for h, k in zip(high.tolist(), (w - weight).tolist()):
        if 0 <= k <= low and lists[k].numel():
            gathered.append(lists[k] | (h << low))
            total += lists[k].numel()
            if total > pieces:
                yield torch.cat(gathered)
                gathered, total = [], 0
    if gathered:
        yield torch.cat(gathered)


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _sector(case, group, device, characters, inversion):
    """(representatives, norms, mask and character of the inversion) of a sector."""
    n = _bits(case)
    flip, sign = 0, inversion or 0
    if case["lattice"] != "hubbard":
        flip = (1 << n) - 1
        found = [group.is_least(x, flip if sign else 0) for x in _weight_states(n, case["weight"], device, 1 << 23)]
        reps = torch.cat(found)
    else:
        half = _sites(case)
        ups = torch.cat(list(_weight_states(half, case["up"], device, 1 << 23)))
        downs = torch.cat(list(_weight_states(half, case["down"], device, 1 << 23)))
        step = max(1, (1 << 23) // ups.numel())
        reps = torch.cat([group.is_least(((d << half)[:, None] | ups[None, :]).reshape(-1)) for d in downs.split(step)])
    stab = torch.cat([group.least(x, flip, sign, characters)[2] for x in reps.split(1 << 22)])
    keep = stab > 1e-9
    size = group.size * (2 if sign else 1)
    return reps[keep], torch.sqrt(stab[keep] / size), flip, sign


def _moves(case, states):
    """(which states, images, coefficients) of every off-diagonal move."""
    n = _sites(case)
    for i, j, J in _bonds(case):
        if case["lattice"] != "hubbard":
            on = torch.nonzero(((states >> i) ^ (states >> j)) & 1).reshape(-1)
            yield on, states[on] ^ ((1 << i) | (1 << j)), 2.0 * J
            continue
        for shift in (0, n):
            a, b = sorted((i + shift, j + shift))
            on = torch.nonzero(((states >> a) ^ (states >> b)) & 1).reshape(-1)
            x = states[on]
            parity = torch.zeros_like(x)
            for bit in range(a + 1, b):
                parity ^= (x >> bit) & 1
            yield on, x ^ ((1 << a) | (1 << b)), -HOPPING * (1.0 - 2.0 * parity.to(torch.float64))


def _diagonal(case, states):
    n = _sites(case)
    out = torch.zeros(states.shape, dtype=torch.float64, device=states.device)
    if case["lattice"] == "hubbard":
        for i in range(n):
            out += REPULSION * ((states >> i) & (states >> (i + n)) & 1).to(torch.float64)
        return out
    for i, j, J in _bonds(case):
        out += J * (1.0 - 2.0 * (((states >> i) ^ (states >> j)) & 1).to(torch.float64))
    return out


def _apply(case, group, reps, norms, flip, sign, characters, x):
    """M x for the sector's matrix, x of shape (states, columns)."""
    y = _diagonal(case, reps)[:, None] * x

    def add(gathered):
        o, z, k = (torch.cat(parts) for parts in zip(*gathered))
        rep, chi, _ = group.least(z, flip, sign, characters)
        at = torch.searchsorted(reps, rep).clamp(max=reps.numel() - 1)
        value = (reps[at] == rep) * k * norms[at] / norms[o]
        if chi is not None:
            value = value * (chi if x.is_complex() else chi.real)
        for part in range(0, o.numel(), 1 << 21):
            s = slice(part, part + (1 << 21))
            y.index_add_(0, at[s], value[s].to(x.dtype)[:, None] * x[o[s]])

    gathered, total = [], 0
    for on, images, c in _moves(case, reps):
        c = c if isinstance(c, torch.Tensor) else torch.full(on.shape, c, dtype=torch.float64, device=on.device)
        gathered.append((on, images, c))
        total += on.numel()
        if total > 1 << 23:
            add(gathered)
            gathered, total = [], 0
    if gathered:
        add(gathered)
    return y


def _operations(case):
    """About how many image computations `exact` does."""
    dim, nnz = _shape(case)
    n = _sites(case)
    group = (8 * n if case["lattice"] != "chain" else 2 * n) if case["kind"] != "sectors" else n
    candidates = _choose(n, case["up"]) * _choose(n, case["down"]) if case["lattice"] == "hubbard" \
        else _choose(n, case["weight"])
    if case["kind"] in ("basis", "setup", "product", "onthefly", "host", "ground"):
        return group * nnz + 4 * candidates
    if case["kind"] == "sectors":
        return 2 * group * nnz + 8 * n * candidates
    return group * case["batch"]


def exact(case, seed):
    kind = case["kind"]
    if _operations(case) > 2e10:
        return None
    device = _device()
    if kind == "sectors":
        return _exact_sectors(case, seed, device)
    phases, inversion = _sectors_of(case, seed) if kind == "basis" else _symmetric_sector(case)
    perms, characters = _closure(_generators(case), phases)
    group = _Group(_bits(case), perms, device, 2 if case["lattice"] == "hubbard" else 1)
    characters = characters if any(c != 1.0 for c in characters) else None
    if kind == "stateinfo":
        states = torch.from_numpy(_random_states(case, seed).astype(np.int64)).to(device)
        n = _sites(case)
        rep, _, stab = group.least(states, (1 << n) - 1, inversion or 0)
        norms = torch.sqrt(stab / (group.size * (2 if case["inversion"] else 1)))
        return [rep, np.ones(case["batch"], dtype=np.complex128), norms]
    reps, norms, flip, sign = _sector(case, group, device, characters, inversion)
    if kind == "basis":
        return _keep(torch.empty(_room(case), dtype=torch.int64, device=device), reps)
    if kind == "ground":
        if reps.numel() > 3000:
            return None
        case = _ground_case(case, seed)
        eye = torch.eye(reps.numel(), dtype=torch.float64, device=device)
        values = torch.linalg.eigvalsh(_apply(case, group, reps, norms, flip, sign, None, eye).cpu())
        return {"eigenvalues": values[:1].numpy(), "converged": None}
    if kind == "host":
        x = torch.from_numpy(np.random.default_rng(seed).standard_normal(reps.numel())).to(device)[:, None]
        return _apply(case, group, reps, norms, flip, sign, None, x)[:, 0]
    if kind == "onthefly" and case["lattice"] == "hubbard":
        x = torch.view_as_complex(_normal((reps.numel(), 2), 64, seed))[:, None]
        return torch.view_as_real(_apply(case, group, reps, norms, flip, sign, None, x)[:, 0])
    columns = case["columns"] if kind == "product" else 1
    bits = case["bits"] if kind == "product" else 64
    x = _normal((reps.numel(),) if columns == 1 else (reps.numel(), columns), bits, seed).to(torch.float64)
    y = _apply(case, group, reps, norms, flip, sign, None, x.reshape(-1, columns)).reshape(x.shape)
    return {"nonzeros": None, "y": y} if kind == "setup" else y


def _exact_sectors(case, seed, device):
    n = case["size"]
    translation = models.chain_translation(n)
    perms = [tuple(range(n))]
    while len(perms) < n:
        perms.append(tuple(perms[-1][int(i)] for i in translation))
    group = _Group(n, perms, device)
    parts = []
    for k, inversion in sectors.chain_sectors(n):
        characters = [np.exp(-2j * np.pi * ((k * m) % n) / n) for m in range(n)]
        parts.append((characters, *_sector(case, group, device, characters, inversion)))
    x = _sector_input(sum(p[1].numel() for p in parts), case, seed).to(torch.float64)
    x = torch.complex(x[:, 0], x[:, 1])
    out, at = [], 0
    for characters, reps, norms, flip, sign in parts:
        out.append(_apply(case, group, reps, norms, flip, sign, characters, x[at:at + reps.numel()]))
        at += reps.numel()
    y = torch.cat(out)
    return torch.stack([y.real, y.imag], dim=1)
