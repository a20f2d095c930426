"""Python host layer of the MI355X lattice-symmetries engine.

Mirrors the reference's Python API for the hot path
(python/lattice_symmetries/__init__.py: Symmetry :68-120, Symmetries,
SpinBasis :123-330, Operator :591-752) on top of liblsamd.so.  Objects are
the reference's C structs (ls_hs_basis, ls_hs_operator, ...) built the way
the reference's Haskell layer builds them (Basis.hs:788-810,
Operator.hs:150-169), and every call goes through the reference-named C
entry points, so this layer exercises exactly the drop-in boundary.

The DeviceBasis / DeviceOperator classes use the additive ls_amd_* entry
points, which keep states and vectors in device memory.

There is no CPU fallback: every computation runs on the GPU through
liblsamd.so, and a missing library or device raises EngineError.
"""
from __future__ import annotations

import ctypes as C
from typing import Optional, Sequence

import numpy as np

from . import _abi
from ._abi import EngineError, check, load
from .expr import Expr, Term

__all__ = [
    "EngineError",
    "Symmetry",
    "Symmetries",
    "SpinBasis",
    "Operator",
    "DeviceArray",
    "DeviceBasis",
    "DeviceOperator",
    "DeviceSectorBatch",
    "Expr",
    "Model",
    "Term",
    "device_available",
    "device_trim",
]


def device_available() -> bool:
    return load().ls_amd_device_available() == 0


def device_trim() -> int:
    """Gives the device memory that the engine keeps for reuse back to the
    driver (for torch or another allocator); returns the bytes."""
    return int(load().ls_amd_device_trim())


def _u64ptr(a: np.ndarray):
    return a.ctypes.data_as(C.POINTER(C.c_uint64))


def _f64ptr(a: np.ndarray):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def _as_u64(x) -> np.ndarray:
    return np.ascontiguousarray(np.asarray(x, dtype=np.uint64))


# ---------------------------------------------------------------------------
# Symmetries
# ---------------------------------------------------------------------------


class Symmetry:
    """A permutation of sites with a momentum sector (Group.hs:58-85):
    bit i of g(x) is bit permutation[i] of x; the phase is sector / period."""

    def __init__(self, permutation: Sequence[int], sector: int):
        self.permutation = np.asarray(permutation, dtype=np.int32)
        self.sector = int(sector)

    @property
    def number_sites(self) -> int:
        return int(self.permutation.size)


class Symmetries:
    """The group generated by a list of Symmetry (Group.hs:106-132), with
    Benes networks and characters as ls_hs_permutation_group."""

    def __init__(self, generators: Sequence[Symmetry]):
        lib = load()
        self.generators = list(generators)
        if not self.generators:
            raise ValueError("at least one generator is required")
        n = self.generators[0].number_sites
        if any(g.number_sites != n for g in self.generators):
            raise ValueError("symmetries have different number of sites")
        perms = np.ascontiguousarray(np.stack([g.permutation for g in self.generators]).astype(np.int32))
        sectors = np.asarray([g.sector for g in self.generators], dtype=np.int32)
        ptr = lib.ls_amd_permutation_group_create(
            n, len(self.generators), perms.ctypes.data_as(C.POINTER(C.c_int32)),
            sectors.ctypes.data_as(C.POINTER(C.c_int32)))
        if not ptr:
            raise ValueError(_abi.last_error())
        self._ptr = ptr
        self.number_sites = n

    def __del__(self):
        if getattr(self, "_ptr", None) and _abi._lib is not None:
            _abi._lib.ls_amd_permutation_group_destroy(self._ptr)
            self._ptr = None

    @property
    def pointer(self):
        return self._ptr

    def __len__(self) -> int:
        return int(self._ptr.contents.number_masks)

    @property
    def depth(self) -> int:
        return int(self._ptr.contents.number_shifts)

    @property
    def masks(self) -> np.ndarray:
        g = self._ptr.contents
        return np.ctypeslib.as_array(g.masks, shape=(g.number_shifts, g.number_masks)).copy()

    @property
    def shifts(self) -> np.ndarray:
        g = self._ptr.contents
        return np.ctypeslib.as_array(g.shifts, shape=(g.number_shifts,)).copy()

    @property
    def characters(self) -> np.ndarray:
        g = self._ptr.contents
        re = np.ctypeslib.as_array(g.eigvals_re, shape=(g.number_masks,))
        im = np.ctypeslib.as_array(g.eigvals_im, shape=(g.number_masks,))
        return re + 1j * im

    def elements(self) -> np.ndarray:
        out = np.zeros((len(self), self.number_sites), dtype=np.int32)
        load().ls_amd_permutation_group_elements(self._ptr, out.ctypes.data_as(C.POINTER(C.c_int32)))
        return out


# ---------------------------------------------------------------------------
# Basis through the reference ABI
# ---------------------------------------------------------------------------

_chpl_initialised = False


def _ensure_chpl():
    global _chpl_initialised
    lib = load()
    if not device_available():
        raise EngineError("no usable gfx950 device: " + _abi.last_error())
    if not _chpl_initialised:
        lib.ls_chpl_init()
        _chpl_initialised = True
    return lib


class SpinBasis:
    """Spin-1/2 basis (python/lattice_symmetries/__init__.py:123-330)."""

    def __init__(self, number_spins: int, hamming_weight: Optional[int] = None,
                 spin_inversion: Optional[int] = None, symmetries: Optional[Symmetries] = None):
        lib = _ensure_chpl()
        if spin_inversion is not None and hamming_weight is None:
            hamming_weight = number_spins // 2  # the reference infers n/2
        if spin_inversion not in (None, 1, -1):
            raise ValueError("spin_inversion must be None, 1 or -1")
        if symmetries is not None and symmetries.number_sites != number_spins:
            raise ValueError("symmetries act on a different number of sites")
        self.number_spins = number_spins
        self.hamming_weight = hamming_weight
        self.spin_inversion = spin_inversion or 0
        self.symmetries = symmetries
        has_perms = symmetries is not None and len(symmetries) > 0
        self._kernels = _abi.ls_hs_basis_kernels()
        if has_perms or self.spin_inversion != 0:
            if has_perms:
                data = lib.ls_internal_create_halide_kernel_data(symmetries.pointer, self.spin_inversion)
                check("ls_internal_create_halide_kernel_data")
                if not data:
                    raise EngineError(_abi.last_error())
                self._kernels.state_info_kernel = C.cast(lib.ls_hs_state_info_halide_kernel, C.c_void_p)
                self._kernels.state_info_data = data
                self._kernels.is_representative_kernel = C.cast(lib.ls_hs_is_representative_halide_kernel, C.c_void_p)
                self._kernels.is_representative_data = data
        self._basis = _abi.ls_hs_basis()
        b = self._basis
        b.refcount = 1
        b.number_sites = number_spins
        b.number_particles = number_spins
        b.number_up = -1 if hamming_weight is None else hamming_weight
        b.particle_type = _abi.LS_HS_SPIN
        b.spin_inversion = self.spin_inversion
        b.state_index_is_identity = (hamming_weight is None and self.spin_inversion == 0 and not has_perms)
        b.requires_projection = has_perms or self.spin_inversion != 0
        b.kernels = C.pointer(self._kernels)
        self._states = None

    def __del__(self):
        lib = _abi._lib
        if lib is None:
            return
        k = getattr(self, "_kernels", None)
        if k is not None:
            if k.state_index_data:
                lib.ls_hs_destroy_state_index_binary_search_kernel_data(k.state_index_data)
                k.state_index_data = None
            if k.state_info_data:
                lib.ls_internal_destroy_halide_kernel_data(k.state_info_data)
                k.state_info_data = None
        b = getattr(self, "_basis", None)
        if b is not None and b.representatives.num_elts > 0:
            lib.ls_hs_internal_destroy_external_array(C.byref(b.representatives))
            b.representatives.num_elts = 0

    @property
    def pointer(self):
        return C.pointer(self._basis)

    @property
    def number_bits(self) -> int:
        return self.number_spins

    @property
    def requires_projection(self) -> bool:
        return bool(self._basis.requires_projection)

    @property
    def has_permutation_symmetries(self) -> bool:
        return self.symmetries is not None and len(self.symmetries) > 0

    # Basis.hs:734-774
    @property
    def min_state_estimate(self) -> int:
        h = self.hamming_weight
        return 0 if h is None else (1 << h) - 1

    @property
    def max_state_estimate(self) -> int:
        n, h = self.number_spins, self.hamming_weight
        if h is None:
            return (1 << n) - 1
        ones = (1 << h) - 1
        return ones << (n - h) if self.spin_inversion == 0 else ones << (n - h - 1)

    def build(self) -> None:
        """ls_hs_basis_build: enumerate representatives on the GPU."""
        lib = load()
        if self._basis.representatives.num_elts == 0:
            lib.ls_hs_build_representatives(self.pointer, self.min_state_estimate, self.max_state_estimate)
            check("build")
        self._states = None

    @property
    def is_built(self) -> bool:
        return self._basis.kernels.contents.state_index_kernel is not None and \
            bool(self._basis.kernels.contents.state_index_data)

    @property
    def number_states(self) -> int:
        if not self.is_built:
            raise ValueError("basis states have not been built yet")
        return int(self._basis.representatives.num_elts)

    @property
    def states(self) -> np.ndarray:
        n = self.number_states
        if n == 0:
            return np.zeros(0, dtype=np.uint64)
        p = C.cast(self._basis.representatives.elts, C.POINTER(C.c_uint64))
        return np.ctypeslib.as_array(p, shape=(n,))

    def index(self, x):
        """Index of each state, -1 when absent (ls_hs_state_index)."""
        scalar = np.ndim(x) == 0
        xs = _as_u64(np.atleast_1d(x))
        out = np.zeros(xs.size, dtype=np.int64)
        if xs.size:
            load().ls_hs_state_index(self.pointer, xs.size, _u64ptr(xs), 1,
                                     out.ctypes.data_as(C.POINTER(C.c_ssize_t)), 1)
            check("index")
        return int(out[0]) if scalar else out

    def state_info(self, x):
        """(representatives, characters, norms) (ls_hs_state_info)."""
        scalar = np.ndim(x) == 0
        xs = _as_u64(np.atleast_1d(x))
        n = xs.size
        if self.has_permutation_symmetries:
            betas = np.zeros(n, dtype=np.uint64)
            chars = np.zeros(n, dtype=np.complex128)
            norms = np.zeros(n, dtype=np.float64)
            if n:
                load().ls_hs_state_info(self.pointer, n, _u64ptr(xs), 1, _u64ptr(betas), 1,
                                        chars.ctypes.data_as(C.POINTER(_abi.ls_hs_scalar)), _f64ptr(norms))
                check("state_info")
        elif self.spin_inversion != 0:  # python/lattice_symmetries/__init__.py:280-287
            mask = np.uint64((1 << self.number_bits) - 1)
            flipped = np.bitwise_xor(xs, mask)
            when = flipped < xs
            betas = np.where(when, flipped, xs)
            chars = np.where(when, float(self.spin_inversion), 1.0).astype(np.complex128)
            norms = np.ones(n)
        else:
            betas, chars, norms = xs.copy(), np.ones(n, dtype=np.complex128), np.ones(n)
        if scalar:
            return int(betas[0]), complex(chars[0]), float(norms[0])
        return betas, chars, norms

    def is_representative(self, x):
        """(flags, norms) (ls_hs_is_representative)."""
        xs = _as_u64(np.atleast_1d(x))
        flags = np.zeros(xs.size, dtype=np.uint8)
        norms = np.zeros(xs.size, dtype=np.float64)
        if xs.size:
            load().ls_hs_is_representative(self.pointer, xs.size, _u64ptr(xs), 1,
                                           flags.ctypes.data_as(C.POINTER(C.c_uint8)), _f64ptr(norms))
            check("is_representative")
        return flags, norms


# ---------------------------------------------------------------------------
# Operator through the reference ABI
# ---------------------------------------------------------------------------


class _TermArrays:
    """ls_hs_nonbranching_terms with owned numpy storage (Operator.hs:109-135)."""

    def __init__(self, terms: Sequence[Term], number_bits: int):
        n = len(terms)
        self.v = np.zeros(2 * max(n, 1), dtype=np.float64)
        self.m = np.zeros(max(n, 1), dtype=np.uint64)
        self.l = np.zeros(max(n, 1), dtype=np.uint64)
        self.r = np.zeros(max(n, 1), dtype=np.uint64)
        self.x = np.zeros(max(n, 1), dtype=np.uint64)
        self.s = np.zeros(max(n, 1), dtype=np.uint64)
        mask = (1 << 64) - 1
        for i, t in enumerate(terms):
            self.v[2 * i] = complex(t.v).real
            self.v[2 * i + 1] = complex(t.v).imag
            self.m[i], self.l[i], self.r[i] = t.m & mask, t.l & mask, t.r & mask
            self.x[i], self.s[i] = t.x & mask, t.s & mask
        self.struct = _abi.ls_hs_nonbranching_terms(
            n, number_bits, self.v.ctypes.data_as(C.POINTER(_abi.ls_hs_scalar)),
            _u64ptr(self.m), _u64ptr(self.l), _u64ptr(self.r), _u64ptr(self.x), _u64ptr(self.s))
        self.count = n

    def pointer(self):
        return C.pointer(self.struct) if self.count > 0 else None


class Operator:
    """Operator over a built basis (python/lattice_symmetries/__init__.py:591-752)."""

    def __init__(self, basis: SpinBasis, expr: Expr):
        self.basis = basis
        self.expression = expr
        diag, off = expr.split()
        self._diag = _TermArrays(diag, basis.number_bits)
        self._off = _TermArrays(off, basis.number_bits)
        self._op = _abi.ls_hs_operator()
        self._op.refcount = 1
        self._op.basis = basis.pointer
        if self._off.count:
            self._op.off_diag_terms = C.pointer(self._off.struct)
        if self._diag.count:
            self._op.diag_terms = C.pointer(self._diag.struct)

    def __del__(self):
        if getattr(self, "_op", None) is not None and _abi._lib is not None:
            _abi._lib.ls_amd_forget_operator(C.pointer(self._op))

    @property
    def pointer(self):
        return C.pointer(self._op)

    @property
    def number_off_diag_terms(self) -> int:
        return self._off.count

    @property
    def number_diag_terms(self) -> int:
        return self._diag.count

    def matvec(self, x: np.ndarray, out: Optional[np.ndarray] = None) -> np.ndarray:
        """y = H x for a real vector (ls_chpl_matrix_vector_product)."""
        x = np.ascontiguousarray(np.asarray(x, dtype=np.float64))
        n = self.basis.number_states
        if x.shape != (n,):
            raise ValueError(f"expected a vector of shape ({n},), got {x.shape}")
        if out is None:
            y = np.zeros(n)
        else:
            if not (isinstance(out, np.ndarray) and out.dtype == np.float64 and out.shape == (n,)
                    and out.flags.c_contiguous and out.flags.writeable):
                raise ValueError(f"out must be a writeable contiguous float64 array of shape ({n},)")
            y = out
        load().ls_chpl_matrix_vector_product(self.pointer, 1, _f64ptr(x), _f64ptr(y))
        check("matvec")
        return y

    def __matmul__(self, x):
        return self.matvec(x)

    def apply_diag(self, alphas, xs=None) -> np.ndarray:
        """ls_internal_operator_apply_diag_x1."""
        a = _as_u64(alphas)
        ys = np.zeros(a.size)
        xp = None
        if xs is not None:
            xs = np.ascontiguousarray(xs, dtype=np.float64)
            xp = _f64ptr(xs)
        load().ls_internal_operator_apply_diag_x1(self.pointer, a.size, _u64ptr(a), _f64ptr(ys), xp)
        check("apply_diag")
        return ys

    def apply_off_diag(self, alphas, xs=None):
        """ls_internal_operator_apply_off_diag_x1: (betas, coeffs, offsets)."""
        a = _as_u64(alphas)
        cap = max(a.size * self._off.count, 1)
        betas = np.zeros(cap, dtype=np.uint64)
        coeffs = np.zeros(cap, dtype=np.complex128)
        offsets = np.zeros(a.size + 1, dtype=np.int64)
        xp = None
        if xs is not None:
            xs = np.ascontiguousarray(xs, dtype=np.float64)
            xp = _f64ptr(xs)
        load().ls_internal_operator_apply_off_diag_x1(
            self.pointer, a.size, _u64ptr(a), _u64ptr(betas),
            coeffs.ctypes.data_as(C.POINTER(_abi.ls_hs_scalar)),
            offsets.ctypes.data_as(C.POINTER(C.c_ssize_t)), xp)
        check("apply_off_diag")
        k = int(offsets[-1])
        return betas[:k], coeffs[:k], offsets


# ---------------------------------------------------------------------------
# Device-resident API (ls_amd_*)
# ---------------------------------------------------------------------------


class DeviceArray:
    """A device allocation owned by the engine."""

    def __init__(self, nbytes: int):
        lib = load()
        self.nbytes = int(nbytes)
        self.ptr = lib.ls_amd_device_malloc(max(self.nbytes, 1))
        if not self.ptr:
            raise EngineError("device allocation failed: " + _abi.last_error())

    @staticmethod
    def from_numpy(a: np.ndarray) -> "DeviceArray":
        a = np.ascontiguousarray(a)
        d = DeviceArray(a.nbytes)
        if a.nbytes and load().ls_amd_memcpy_h2d(d.ptr, a.ctypes.data, a.nbytes) != 0:
            raise EngineError("host to device copy failed")
        return d

    def to_numpy(self, dtype, shape) -> np.ndarray:
        out = np.empty(shape, dtype=dtype)
        if out.nbytes > self.nbytes:
            raise ValueError("requested more bytes than allocated")
        if out.nbytes and load().ls_amd_memcpy_d2h(out.ctypes.data, self.ptr, out.nbytes) != 0:
            raise EngineError("device to host copy failed")
        return out

    def upload(self, a: np.ndarray) -> None:
        a = np.ascontiguousarray(a)
        if a.nbytes > self.nbytes:
            raise ValueError("array larger than the allocation")
        if a.nbytes and load().ls_amd_memcpy_h2d(self.ptr, a.ctypes.data, a.nbytes) != 0:
            raise EngineError("host to device copy failed")

    def __del__(self):
        if getattr(self, "ptr", None) and _abi._lib is not None:
            _abi._lib.ls_amd_device_free(self.ptr)
            self.ptr = None


class DeviceBasis:
    """Basis whose representatives stay in device memory (ls_amd_basis_*)."""

    def __init__(self, number_spins: int, hamming_weight: Optional[int] = None,
                 spin_inversion: Optional[int] = None, symmetries: Optional[Symmetries] = None):
        lib = load()
        if not device_available():
            raise EngineError("no usable gfx950 device: " + _abi.last_error())
        if spin_inversion is not None and hamming_weight is None:
            hamming_weight = number_spins // 2
        self.number_spins = number_spins
        self.hamming_weight = hamming_weight
        self.spin_inversion = spin_inversion or 0
        self.symmetries = symmetries
        gp = symmetries.pointer if symmetries is not None else None
        self._h = lib.ls_amd_basis_create(number_spins, -1 if hamming_weight is None else hamming_weight,
                                          self.spin_inversion, gp)
        if not self._h:
            raise EngineError(_abi.last_error())

    @classmethod
    def fermions(cls, number_sites: int, number_up: int, number_down: Optional[int] = None,
                 symmetries: Optional[Symmetries] = None) -> "DeviceBasis":
        """Fermion basis (ls_amd_fermion_basis_create): spinful when number_down
        is given (up species in the low bits); symmetries act on all bits."""
        lib = load()
        if not device_available():
            raise EngineError("no usable gfx950 device: " + _abi.last_error())
        self = cls.__new__(cls)
        self.number_spins = number_sites
        self.number_sites = number_sites
        self.hamming_weight = None
        self.spin_inversion = 0
        self.symmetries = symmetries
        self._bits = 2 * number_sites if number_down is not None else number_sites
        gp = symmetries.pointer if symmetries is not None else None
        self._h = lib.ls_amd_fermion_basis_create(number_sites, number_up,
                                                  -1 if number_down is None else number_down, gp)
        if not self._h:
            raise EngineError(_abi.last_error())
        return self

    @classmethod
    def _adopt(cls, handle, model) -> "DeviceBasis":
        """Wraps a basis created by the model front-end."""
        self = cls.__new__(cls)
        self.number_spins = model.number_sites
        self.number_sites = model.number_sites
        self.hamming_weight = model.hamming_weight
        self.spin_inversion = model.spin_inversion or 0
        self.symmetries = None
        self._bits = 2 * model.number_sites if model.particle == "spinful-fermion" else model.number_sites
        self._h = handle
        return self

    def __del__(self):
        if getattr(self, "_h", None) and _abi._lib is not None:
            _abi._lib.ls_amd_basis_destroy(self._h)
            self._h = None

    @property
    def handle(self):
        return self._h

    @property
    def number_bits(self) -> int:
        return getattr(self, "_bits", self.number_spins)

    @property
    def min_state_estimate(self) -> int:
        return int(load().ls_amd_basis_min_state(self._h))

    @property
    def max_state_estimate(self) -> int:
        return int(load().ls_amd_basis_max_state(self._h))

    def set_norm_tolerance(self, eps: float) -> None:
        """Count stabiliser sums <= eps as zero (ls_amd_basis_set_norm_tolerance)."""
        if load().ls_amd_basis_set_norm_tolerance(self._h, eps) != 0:
            raise EngineError(_abi.last_error())

    def build(self, lower: Optional[int] = None, upper: Optional[int] = None) -> int:
        lo = self.min_state_estimate if lower is None else lower
        hi = self.max_state_estimate if upper is None else upper
        n = load().ls_amd_basis_build(self._h, lo, hi)
        if n < 0:
            raise EngineError(_abi.last_error())
        return int(n)

    def set_states(self, states: np.ndarray) -> None:
        s = _as_u64(states)
        if load().ls_amd_basis_set_states(self._h, _u64ptr(s), s.size) != 0:
            raise EngineError(_abi.last_error())

    @property
    def number_states(self) -> int:
        return int(load().ls_amd_basis_number_states(self._h))

    @property
    def number_candidates(self) -> int:
        return int(load().ls_amd_basis_number_candidates(self._h))

    @property
    def states(self) -> np.ndarray:
        out = np.zeros(self.number_states, dtype=np.uint64)
        if out.size and load().ls_amd_basis_copy_states(self._h, _u64ptr(out)) != 0:
            raise EngineError(_abi.last_error())
        return out

    def _device_call(self, fn, xs, outs):
        lib = load()
        x = DeviceArray.from_numpy(_as_u64(xs))
        douts = [DeviceArray(max(int(np.prod(s)) * np.dtype(d).itemsize, 1)) for d, s in outs]
        if fn(self._h, len(xs), x.ptr, *[d.ptr for d in douts]) != 0:
            raise EngineError(_abi.last_error())
        return [d.to_numpy(dt, s) for d, (dt, s) in zip(douts, outs)]

    def state_info(self, xs):
        n = len(xs)
        reps, chars, norms = self._device_call(load().ls_amd_basis_state_info_device, xs,
                                               [(np.uint64, (n,)), (np.float64, (n, 2)), (np.float64, (n,))])
        return reps, chars[:, 0] + 1j * chars[:, 1], norms

    def is_representative(self, xs):
        n = len(xs)
        return tuple(self._device_call(load().ls_amd_basis_is_representative_device, xs,
                                       [(np.uint8, (n,)), (np.float64, (n,))]))

    def index(self, xs):
        n = len(xs)
        (out,) = self._device_call(load().ls_amd_basis_index_device, xs, [(np.int64, (n,))])
        return out


def _lanczos_dict(res) -> dict:
    return {
        "steps": res.steps,
        "refine_steps": res.refine_steps,
        "eigenvalues": [res.eigenvalues[i] for i in range(res.number_eigenvalues)],
        "rayleigh": res.rayleigh,
        "residual_norm": res.residual_norm,
        "matvec_seconds": res.matvec_seconds,
        "matvec_calls": res.matvec_calls,
        "total_seconds": res.total_seconds,
    }


class DeviceOperator:
    """Operator over a DeviceBasis with device-resident vectors."""

    def __init__(self, basis: DeviceBasis, expr: Expr):
        lib = load()
        self.basis = basis
        diag, off = expr.split()
        self._diag = _TermArrays(diag, basis.number_bits)
        self._off = _TermArrays(off, basis.number_bits)
        self._h = lib.ls_amd_operator_create(basis.handle, self._diag.pointer(), self._off.pointer())
        if not self._h:
            raise EngineError(_abi.last_error())
        self.csr_nnz = None

    @classmethod
    def _adopt(cls, handle, basis) -> "DeviceOperator":
        """Wraps an operator created by the model front-end."""
        self = cls.__new__(cls)
        self.basis = basis
        self._diag = self._off = None
        self._h = handle
        self.csr_nnz = None
        return self

    def __del__(self):
        if getattr(self, "_h", None) and _abi._lib is not None:
            _abi._lib.ls_amd_operator_destroy(self._h)
            self._h = None

    @property
    def handle(self):
        return self._h

    def _ok(self, rc):
        if rc != 0:
            raise EngineError(_abi.last_error())

    def matvec_otf(self, dx: DeviceArray, dy: DeviceArray, accumulate: bool = False):
        self._ok(load().ls_amd_matvec_f64(self._h, dx.ptr, dy.ptr, int(accumulate)))

    def matvec_complex(self, dx: DeviceArray, dy: DeviceArray):
        self._ok(load().ls_amd_matvec_c128(self._h, dx.ptr, dy.ptr))

    def build_csr(self, precision: int = 96) -> int:
        nnz = load().ls_amd_operator_build_csr(self._h, precision)
        if nnz < 0:
            raise EngineError(_abi.last_error())
        self.csr_nnz = int(nnz)
        return self.csr_nnz

    def set_factored(self, enable: bool) -> None:
        """Translation-factorised orbit search in the fused kernels (default on
        where the group allows it; the stored CSR is the same either way)."""
        self._ok(load().ls_amd_operator_set_factored(self._h, 1 if enable else 0))

    @property
    def uses_factored(self) -> bool:
        return load().ls_amd_operator_uses_factored(self._h) == 1

    def is_hermitian(self, mode: int = 2) -> bool:
        """<u, M v> = <M u, v> for the product of a mode (0 FP64 CSR, 1 FP32
        CSR, 2 on-the-fly, 3 on-the-fly complex) on seeded vectors."""
        rc = load().ls_amd_operator_is_hermitian(self._h, mode)
        if rc < 0:
            raise EngineError(_abi.last_error())
        return rc == 1

    def autotune(self) -> int:
        return int(load().ls_amd_operator_autotune(self._h))

    def set_csr_packing(self, enable: bool) -> None:
        """Allow the value-table CSR (default); call before build_csr."""
        self._ok(load().ls_amd_operator_set_csr_packing(self._h, int(enable)))

    @property
    def csr_info(self) -> dict:
        out = (C.c_int64 * 4)()
        self._ok(load().ls_amd_operator_csr_info(self._h, out))
        return {"nnz": out[0], "packed": out[1] == 1, "wide": out[1] == 2, "table_size": out[2],
                "complex": bool(out[3])}

    @property
    def schedule(self) -> dict:
        out = (C.c_int * 5)()
        self._ok(load().ls_amd_operator_schedule(self._h, out))
        return {"lanes_f64": out[0], "flags_f64": out[1], "lanes_f32": out[2], "flags_f32": out[3],
                "persistent_blocks": out[4]}

    def set_schedule(self, lanes_f64: int, flags_f64: int, lanes_f32: int, flags_f32: int):
        self._ok(load().ls_amd_operator_set_schedule(self._h, lanes_f64, flags_f64, lanes_f32, flags_f32))

    def csr_matvec(self, dx: DeviceArray, dy: DeviceArray):
        self._ok(load().ls_amd_csr_matvec_f64(self._h, dx.ptr, dy.ptr))

    def csr_matvec_f32(self, k: int, dx: DeviceArray, dy: DeviceArray):
        self._ok(load().ls_amd_csr_matvec_f32(self._h, k, dx.ptr, dy.ptr))

    def csr_matvec_f64_block(self, k: int, dx: DeviceArray, dy: DeviceArray):
        self._ok(load().ls_amd_csr_matvec_f64_block(self._h, k, dx.ptr, dy.ptr))

    def csr_arrays(self):
        n = self.basis.number_states
        nnz = int(load().ls_amd_operator_csr_nnz(self._h))
        cplx = self.csr_info["complex"]
        rp = np.zeros(n + 1, dtype=np.int64)
        cols = np.zeros(max(nnz, 1), dtype=np.uint32)
        vals = np.zeros((2 if cplx else 1) * max(nnz, 1), dtype=np.float64)
        diag = np.zeros(max(n, 1), dtype=np.float64)
        self._ok(load().ls_amd_operator_copy_csr(
            self._h, rp.ctypes.data_as(C.POINTER(C.c_int64)), cols.ctypes.data_as(C.POINTER(C.c_uint32)),
            _f64ptr(vals), _f64ptr(diag)))
        if cplx:
            return rp, cols[:nnz], vals[0:2 * nnz:2] + 1j * vals[1:2 * nnz:2], diag[:n]
        return rp, cols[:nnz], vals[:nnz], diag[:n]

    def lanczos(self, mode: str = "fp64", max_steps: int = 200, k: int = 1, tol: float = 1e-12,
                seed: int = 42, refine_steps: int = 0, ritz: Optional[DeviceArray] = None) -> dict:
        """Lowest eigenvalues by Lanczos (ls_amd_lanczos); mode fp64 | fp32 | otf |
        otf_complex (complex vectors: each eigenvalue of the complex matrix once)."""
        m = {"fp64": 0, "fp32": 1, "otf": 2, "otf_complex": 3}[mode]
        res = _abi.ls_amd_lanczos_result()
        rc = load().ls_amd_lanczos(self._h, m, max_steps, k, tol, seed, refine_steps,
                                   ritz.ptr if ritz is not None else None, C.byref(res))
        self._ok(rc)
        return _lanczos_dict(res)

    def block_lanczos(self, mode: str = "fp32", block_size: int = 8, max_blocks: int = 40, k: int = 1,
                      tol: float = 1e-10, seed: int = 42, refine_steps: int = 0,
                      ritz: Optional[DeviceArray] = None) -> dict:
        """Lowest eigenvalues by block Lanczos (ls_amd_block_lanczos); mode fp64 | fp32."""
        m = {"fp64": 0, "fp32": 1}[mode]
        res = _abi.ls_amd_lanczos_result()
        rc = load().ls_amd_block_lanczos(self._h, m, block_size, max_blocks, k, tol, seed, refine_steps,
                                         ritz.ptr if ritz is not None else None, C.byref(res))
        self._ok(rc)
        return _lanczos_dict(res)

    def block_eigensolve(self, mode: str = "fp32", block_size: int = 8, nev: int = 1, max_blocks: int = 12,
                         keep_blocks: int = 2, max_cycles: int = 40, tol: float = 1e-7, switch_tol: float = 1e-5,
                         seed: int = 1, ritz: Optional[DeviceArray] = None,
                         eigenvectors: Optional[DeviceArray] = None) -> dict:
        """Thick-restart block Lanczos (ls_amd_block_eigensolve); mode fp64 | fp32 (then fp64).
        ritz receives the lowest Ritz vector; eigenvectors (ls_amd_block_eigenvectors)
        all nev of them, as nev rows of number_states values."""
        m = {"fp64": 0, "fp32": 1}[mode]
        ev = np.zeros(nev)
        rs = np.zeros(nev)
        info = _abi.ls_amd_eig_info()
        if eigenvectors is not None:
            if ritz is not None:
                raise ValueError("pass ritz or eigenvectors, not both")
            rc = load().ls_amd_block_eigenvectors(self._h, m, block_size, nev, max_blocks, keep_blocks, max_cycles,
                                                  tol, switch_tol, seed, _f64ptr(ev), _f64ptr(rs), eigenvectors.ptr,
                                                  C.byref(info))
        else:
            rc = load().ls_amd_block_eigensolve(self._h, m, block_size, nev, max_blocks, keep_blocks, max_cycles,
                                                tol, switch_tol, seed, _f64ptr(ev), _f64ptr(rs),
                                                ritz.ptr if ritz is not None else None, C.byref(info))
        self._ok(rc)
        return {"eigenvalues": ev, "residuals": rs, "cycles": info.cycles, "fp64_cycles": info.fp64_cycles,
                "blocks": info.blocks, "converged": bool(info.converged), "products": info.products,
                "product_seconds": info.product_seconds, "total_seconds": info.total_seconds,
                "max_residual": info.max_residual}

    # numpy conveniences
    def matvec(self, x: np.ndarray, mode: str = "otf") -> np.ndarray:
        x = np.ascontiguousarray(x, dtype=np.float64)
        dx = DeviceArray.from_numpy(x)
        dy = DeviceArray(x.nbytes)
        if mode == "otf":
            self.matvec_otf(dx, dy)
        elif mode == "csr":
            self.csr_matvec(dx, dy)
        else:
            raise ValueError(mode)
        return dy.to_numpy(np.float64, x.shape)

    def matvec_c(self, x: np.ndarray) -> np.ndarray:
        x = np.ascontiguousarray(x, dtype=np.complex128)
        dx = DeviceArray.from_numpy(x)
        dy = DeviceArray(x.nbytes)
        self.matvec_complex(dx, dy)
        return dy.to_numpy(np.complex128, x.shape)

    def matvec_block(self, X: np.ndarray, precision: int = 32) -> np.ndarray:
        n, k = X.shape
        dt = np.float32 if precision == 32 else np.float64
        Xc = np.ascontiguousarray(X, dtype=dt)
        dx = DeviceArray.from_numpy(Xc)
        dy = DeviceArray(Xc.nbytes)
        if precision == 32:
            self.csr_matvec_f32(k, dx, dy)
        else:
            self.csr_matvec_f64_block(k, dx, dy)
        return dy.to_numpy(dt, (n, k))


class DeviceSectorBatch:
    """Several symmetry sectors as one block-diagonal complex operator
    (ls_amd_sector_batch_*).  Every operator must have its complex CSR built
    (``build_csr(128)``).  Vectors are numpy complex arrays of shape
    (number_states, k) over all sectors in order."""

    def __init__(self, operators):
        lib = load()
        operators = list(operators)  # the batch copies their matrices
        arr = (C.c_void_p * len(operators))(*[op.handle for op in operators])
        self._h = lib.ls_amd_sector_batch_create(arr, len(operators))
        if not self._h:
            raise EngineError(_abi.last_error())
        self.count = len(operators)
        self.sectors = None
        self.number_states = int(lib.ls_amd_sector_batch_number_states(self._h))
        self.nnz = int(lib.ls_amd_sector_batch_nnz(self._h))
        off = np.zeros(self.count + 1, dtype=np.int64)
        self._ok(lib.ls_amd_sector_batch_offsets(self._h, off.ctypes.data_as(C.POINTER(C.c_int64))))
        self.offsets = off

    def __del__(self):
        if getattr(self, "_h", None) and _abi._lib is not None:
            _abi._lib.ls_amd_sector_batch_destroy(self._h)
            self._h = None

    def _ok(self, rc):
        if rc != 0:
            raise EngineError(_abi.last_error())

    @property
    def handle(self):
        return self._h

    def autotune(self, k: int = 8) -> dict:
        self._ok(load().ls_amd_sector_batch_autotune(self._h, k))
        return self.schedule

    @property
    def schedule(self) -> dict:
        lanes, blocks, die = C.c_int(), C.c_int(), C.c_int()
        self._ok(load().ls_amd_sector_batch_get_schedule(self._h, C.byref(lanes), C.byref(blocks), C.byref(die)))
        return {"lanes": lanes.value, "blocks": blocks.value, "die_aware": die.value}

    def set_schedule(self, lanes: int, blocks: int, die_aware: bool = True):
        self._ok(load().ls_amd_sector_batch_set_schedule(self._h, lanes, blocks, int(die_aware)))

    def matvec_device(self, k: int, dx: DeviceArray, dy: DeviceArray, precision: int = 32):
        if precision == 32:
            self._ok(load().ls_amd_sector_batch_matvec_f32(self._h, k, dx.ptr, dy.ptr))
        else:
            self._ok(load().ls_amd_sector_batch_matvec_f64(self._h, k, dx.ptr, dy.ptr))

    @staticmethod
    def to_embedded(X: np.ndarray, dtype) -> np.ndarray:
        """(n, k) complex -> [state][re | im][k] real layout."""
        n, k = X.shape
        out = np.empty((n, 2, k), dtype=dtype)
        out[:, 0, :] = X.real
        out[:, 1, :] = X.imag
        return out

    @staticmethod
    def from_embedded(Y: np.ndarray) -> np.ndarray:
        return Y[:, 0, :].astype(np.float64) + 1j * Y[:, 1, :].astype(np.float64)

    def matvec(self, X: np.ndarray, precision: int = 64) -> np.ndarray:
        """Y = M X for complex X of shape (number_states, k), k in {1, 2, 4, 8}."""
        X = np.asarray(X)
        if X.ndim == 1:
            X = X[:, None]
        n, k = X.shape
        dt = np.float32 if precision == 32 else np.float64
        E = self.to_embedded(X, dt)
        dx = DeviceArray.from_numpy(E)
        dy = DeviceArray(E.nbytes)
        self.matvec_device(k, dx, dy, precision)
        return self.from_embedded(dy.to_numpy(dt, E.shape))

    def eigensolve(self, nev: int = 4, block_size: int = 4, max_blocks: int = 16, keep_blocks: int = 4,
                   max_cycles: int = 40, tol: float = 1e-7, switch_tol: float = 1e-5, seed: int = 1) -> dict:
        """Lowest nev eigenvalues of every sector (ls_amd_sector_batch_eigensolve);
        block_size complex columns per Krylov block (nev <= block_size <= 4)."""
        ev = np.zeros(self.count * nev)
        rs = np.zeros(self.count * nev)
        info = _abi.ls_amd_eig_info()
        rc = load().ls_amd_sector_batch_eigensolve(self._h, block_size, nev, max_blocks, keep_blocks, max_cycles,
                                                   tol, switch_tol, seed, _f64ptr(ev), _f64ptr(rs), C.byref(info))
        self._ok(rc)
        return {
            "eigenvalues": ev.reshape(self.count, nev),
            "residuals": rs.reshape(self.count, nev),
            "cycles": info.cycles,
            "fp64_cycles": info.fp64_cycles,
            "blocks": info.blocks,
            "converged": bool(info.converged),
            "products": info.products,
            "product_seconds": info.product_seconds,
            "total_seconds": info.total_seconds,
            "max_residual": info.max_residual,
        }


from .model import Model  # noqa: E402  (needs the classes above)
