// orbit_device.hpp -- device functions for group orbits on gfx950.
//
// A state is a machine word W (uint32_t when the Benes network spans at most
// 32 bits, else uint64_t).  One lane owns one state and walks the group
// elements in their stored (ascending) order; element indices are
// wave-uniform, so masks and characters are read through scalar loads.
//
// The reductions reproduce the order of the reference's Halide kernels
// (kernels/generator.cpp) literally, so representatives, selected characters
// and the floating-point norms agree bit for bit with a sequential
// restatement of those kernels.
#pragma once

#include "lsamd_internal.hpp"

namespace lsamd {

// Shift of stage k in a Benes network of depth D built for N = 2^L bits:
// 1, 2, ..., N/2, N/4, ..., 1 (Benes.hs:295-323).
template <int D> __host__ __device__ constexpr int benes_shift(int k) {
  return k < (D + 1) / 2 ? (1 << k) : (1 << (D - 1 - k));
}

// One delta swap (generator.cpp:5-8): exchange bits i and i+d for every i
// set in m.
template <typename W>
__device__ __forceinline__ W delta_swap(W x, W m, int d) {
  W const y = ((x >> d) ^ x) & m;
  return (x ^ y) ^ (y << d);
}

// Apply the Benes network of group element e.  D > 0: compile-time
// canonical shifts; D == 0: depth and shifts read from the view.
template <typename W, int D>
__device__ __forceinline__ W group_apply(GroupView const &g, int e, W x) {
  if constexpr (D > 0) {
    uint64_t const *m = g.masks + static_cast<size_t>(e) * D;
#pragma unroll
    for (int k = 0; k < D; ++k) x = delta_swap<W>(x, static_cast<W>(m[k]), benes_shift<D>(k));
    return x;
  } else {
    int const depth = g.depth;
    uint64_t const *m = g.masks + static_cast<size_t>(e) * depth;
    for (int k = 0; k < depth; ++k)
      x = delta_swap<W>(x, static_cast<W>(m[k]), static_cast<int>(g.shifts[k]));
    return x;
  }
}

// Same, with the masks of element e given as a pointer (e.g. into LDS).
template <typename W, int D>
__device__ __forceinline__ W benes_apply_ptr(W const *m, W x,
                                             uint64_t const *shifts, int depth) {
  if constexpr (D > 0) {
#pragma unroll
    for (int k = 0; k < D; ++k) x = delta_swap<W>(x, m[k], benes_shift<D>(k));
    return x;
  } else {
    for (int k = 0; k < depth; ++k)
      x = delta_swap<W>(x, m[k], static_cast<int>(shifts[k]));
    return x;
  }
}

// ---------------------------------------------------------------------------
// state_info (generator.cpp:10-166)
// ---------------------------------------------------------------------------
//
// Eight accumulators (the Halide chunk 2 * natural_vector_size(uint64) of the
// avx2 target) each see elements e = 8c + j in order; each keeps the smallest
// image and the first element reaching it, and sums Re(chi) over elements
// fixing x.  Accumulators are merged left to right (earlier lane wins ties),
// then the remaining |G| mod 8 elements are folded in one by one.
// The selected element is kept as an index (2e + flip) and its character is
// read at the end; sel == -1 means no image is smaller than x (chi = 1).

constexpr int kStateInfoLanes = 8;
constexpr int kIsRepresentativeLanes = 4;

// SI selects the symmetry flavour of the orbit kernels: 0 no spin
// inversion, +-1 spin inversion with that character, 2 fermionic signs (no
// inversion).
constexpr int kFermionic = 2;

// Sign of group element e on state x for fermions: the state is the ordered
// product of creation operators (bit order, the Jordan-Wigner order of the
// sign masks); e relabels orbital b as image[b], and the sign is the parity
// of the inversions among the relabelled occupied orbitals.
__device__ __forceinline__ double fermion_sign(GroupView const &g, int e, uint64_t x) {
  uint8_t const *img = g.image + static_cast<size_t>(e) * g.nbits;
  uint64_t seen = 0;
  int parity = 0;
  while (x != 0) {
    int const b = __builtin_ctzll(x);
    x &= x - 1;
    int const i = img[b];
    parity ^= __popcll(seen >> i) & 1; // earlier orbitals now placed above i
    seen |= uint64_t{1} << i;
  }
  return parity ? -1.0 : 1.0;
}

template <typename W>
__device__ __forceinline__ void si_update(W &r, int &sel, double &n, W x, W y,
                                          int code, double re) {
  if (y < r) {
    r = y;
    sel = code;
  }
  if (y == x) n = n + re;
}

struct StateInfo {
  uint64_t rep;
  double c_re, c_im;
  double norm;
};

template <typename W, int D, int SI>
__device__ __forceinline__ StateInfo state_info_one(GroupView const &g,
                                                    uint64_t x64) {
  constexpr int L = kStateInfoLanes;
  W const x = static_cast<W>(x64);
  W const flip = static_cast<W>(g.flip);
  W r[L];
  int sel[L];
  double n[L];
#pragma unroll
  for (int j = 0; j < L; ++j) {
    r[j] = x;
    sel[j] = -1;
    n[j] = 0.0;
  }
  int const G = g.size;
  int const nch = G / L;
  constexpr bool kFermi = SI == kFermionic;
  for (int c = 0; c < nch; ++c) {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      int const e = c * L + j;
      W const y = group_apply<W, D>(g, e, x);
      double re = g.eig_re[e];
      if constexpr (kFermi) {
        if (y == x) re = re * fermion_sign(g, e, x64);
        si_update<W>(r[j], sel[j], n[j], x, y, 2 * e, re);
      } else {
        si_update<W>(r[j], sel[j], n[j], x, y, 2 * e, re);
        if constexpr (SI != 0)
          si_update<W>(r[j], sel[j], n[j], x, static_cast<W>(y ^ flip), 2 * e + 1,
                       SI == 1 ? re : -re);
      }
    }
  }
  W rr = r[0];
  int ss = sel[0];
  double nn = n[0];
#pragma unroll
  for (int j = 1; j < L; ++j) {
    if (r[j] < rr) {
      rr = r[j];
      ss = sel[j];
    }
    nn = nn + n[j];
  }
  for (int e = nch * L; e < G; ++e) {
    W const y = group_apply<W, D>(g, e, x);
    double re = g.eig_re[e];
    if constexpr (kFermi) {
      if (y == x) re = re * fermion_sign(g, e, x64);
      si_update<W>(rr, ss, nn, x, y, 2 * e, re);
    } else {
      si_update<W>(rr, ss, nn, x, y, 2 * e, re);
      if constexpr (SI != 0)
        si_update<W>(rr, ss, nn, x, static_cast<W>(y ^ flip), 2 * e + 1,
                     SI == 1 ? re : -re);
    }
  }
  StateInfo out;
  out.rep = static_cast<uint64_t>(rr);
  if (ss < 0) {
    out.c_re = 1.0;
    out.c_im = 0.0;
  } else {
    int const e = ss >> 1;
    double cre = g.eig_re[e], cim = g.eig_im[e];
    if (SI == -1 && (ss & 1)) {
      cre = -cre;
      cim = -cim;
    }
    if constexpr (kFermi) {
      double const sg = fermion_sign(g, e, x64);
      cre = cre * sg;
      cim = cim * sg;
    }
    out.c_re = cre;
    out.c_im = cim;
  }
  double const denom = (SI == 0 || kFermi) ? static_cast<double>(G) : static_cast<double>(2 * G);
  out.norm = (g.norm_eps > 0.0 && !(nn > g.norm_eps)) ? 0.0 : sqrt(nn / denom);
  return out;
}

// state_info through the translation factorisation of the group (fact_nq >
// 0, real parts of the characters +-1, no fermionic signs): for every point
// element q, y = q(x) by its Benes network, then the translations t_{a,b}(y)
// of the torus by column and row rotations (a few word operations each
// instead of a network per element).  The orbit minimum does not depend on
// the visiting order, and the stabiliser sum of +-1 terms is exact in any
// order.  The character is that of the minimiser state_info_one selects:
// fact_key ranks each element (and its spin-flipped copy, key + 1) by the
// order in which the eight-lane reduction reaches it -- lane e mod 8 first,
// then position within the lane, the |G| mod 8 tail elements last -- and
// among equal images the lowest rank wins, as the strict comparisons of
// that reduction decide.  rep, character and norm equal state_info_one's
// bit for bit.
//
// With row tables (rows of at most kRowTableBits sites), the translations of
// q(x) are not all formed: the least image has the least top row, and the
// top row of t_(a, b)(y) is row (b - 1) mod ly of y rotated by a, so the
// least rotation of each row (a table lookup) gives the least top row and
// the few (a, b) that reach it; only those images are formed and compared
// (none when that row exceeds the top row of the current minimum).  Images
// equal to x need a row in the rotation class of x's top row, found the
// same way.  Every image equal to the minimum, or to x, is still visited,
// so the result is the same.
constexpr int kRowTableBits = 8;

struct RowTables {
  uint8_t minrot[1 << kRowTableBits]; // least rotation of a row value
  uint8_t amin[1 << kRowTableBits];   // rotations a that reach it (bit a)
  uint64_t lo[kRowTableBits], hi[kRowTableBits];
};

__device__ __forceinline__ bool row_tables_apply(GroupView const &g) {
  return g.fact_nq > 0 && g.fact_lx >= 1 && g.fact_lx <= kRowTableBits && g.fact_ly <= kRowTableBits;
}

// Fills the tables (every thread of the workgroup must call it).
__device__ inline void row_tables_init(GroupView const &g, RowTables &t) {
  if (row_tables_apply(g)) {
    int const lx = g.fact_lx;
    uint32_t const rm = (1u << lx) - 1;
    for (uint32_t v = threadIdx.x; v <= rm; v += blockDim.x) {
      uint32_t best = 0xFFu, mask = 0;
      for (int a = 0; a < lx; ++a) {
        uint32_t const r = ((v >> a) | (v << (lx - a))) & rm; // rotation by a
        if (r < best) {
          best = r;
          mask = 1u << a;
        } else if (r == best) {
          mask |= 1u << a;
        }
      }
      t.minrot[v] = static_cast<uint8_t>(best);
      t.amin[v] = static_cast<uint8_t>(mask);
    }
    if (static_cast<int>(threadIdx.x) < lx) {
      int const a = static_cast<int>(threadIdx.x);
      uint64_t lo = 0, hi = 0;
      for (int r = 0; r < g.fact_ly; ++r)
        for (int c = 0; c < lx; ++c) (c < lx - a ? lo : hi) |= uint64_t{1} << (r * lx + c);
      t.lo[a] = lo;
      t.hi[a] = hi;
    }
  }
  __syncthreads();
}

template <typename W, int D, int SI>
__device__ __forceinline__ StateInfo state_info_factored(GroupView const &g, uint64_t x64,
                                                        RowTables const *rt = nullptr) {
  W const x = static_cast<W>(x64);
  W const flip = static_cast<W>(g.flip);
  W const m1 = static_cast<W>(g.fact_m1), m2 = static_cast<W>(g.fact_m2);
  int const lx = g.fact_lx, ly = g.fact_ly, nq = g.fact_nq;
  int const up = g.nbits - lx; // row rotation: the bottom row moves to the top
  // The candidate (q, s, b, a) has position k = (q * ly + b) * lx + a in the
  // tables and code 2 k + s; the minimiser is kept as a code (-1: x itself)
  // and the tables are read only on the rare ties and stabiliser hits, which
  // the branches skip when no lane of the wave has one.
  W best = x;
  int best_code = -1;
  double nn = 0.0;
  if (rt != nullptr && row_tables_apply(g)) {
    uint32_t const rm = (1u << lx) - 1;
    int const top = (ly - 1) * lx;
    uint32_t const xt = static_cast<uint32_t>(x >> top) & rm;
    uint32_t const xcls = rt->minrot[xt];
    // t_(0, b)(y): bit i is bit (i + b lx) mod n of y; t_(a, 0): bit (r, c) is
    // bit (r, (c + a) mod lx)
    auto rows_by = [&](W y, int b) -> W {
      return b == 0 ? y : static_cast<W>((y >> (b * lx)) | ((y << (g.nbits - b * lx)) & flip));
    };
    auto columns_by = [&](W y, int a) -> W {
      return static_cast<W>(((y >> a) & static_cast<W>(rt->lo[a])) | ((y << (lx - a)) & static_cast<W>(rt->hi[a])));
    };
    for (int q = 0; q < nq; ++q) {
      W const y = group_apply<W, D>(g, g.fact_q[q], x);
#pragma unroll
      for (int s = 0; s < (SI != 0 ? 2 : 1); ++s) {
        W const ys = s == 1 ? static_cast<W>(y ^ flip) : y;
        // least rotation of every row; rows reaching the least one (cmask)
        // and rows in the rotation class of x's top row (smask)
        uint32_t mr[kRowTableBits];
        uint32_t m = 0xFFu, smask = 0, cmask = 0;
#pragma unroll
        for (int j = 0; j < kRowTableBits; ++j) {
          mr[j] = j < ly ? rt->minrot[static_cast<uint32_t>(ys >> (j * lx)) & rm] : 0xFFu;
          m = mr[j] < m ? mr[j] : m;
          smask |= (j < ly && mr[j] == xcls ? 1u : 0u) << j;
        }
#pragma unroll
        for (int j = 0; j < kRowTableBits; ++j) cmask |= (j < ly && mr[j] == m ? 1u : 0u) << j;
        if (m > (static_cast<uint32_t>(best >> top) & rm)) cmask = 0;
        for (; cmask != 0; cmask &= cmask - 1) {
          int const j = __ffs(cmask) - 1;
          uint32_t const vj = static_cast<uint32_t>(ys >> (j * lx)) & rm;
          int const b = j + 1 == ly ? 0 : j + 1;
          W const yb = rows_by(ys, b);
          for (uint32_t am = rt->amin[vj]; am != 0; am &= am - 1) {
            int const a = __ffs(am) - 1;
            W const w = columns_by(yb, a);
            int const k = (q * ly + b) * lx + a;
            int const code = 2 * k + s;
            if (w < best) {
              best = w;
              best_code = code;
            } else if (w == best && best_code >= 0 && w != x) {
              int const rank_new = g.fact_key[k] + s;
              int const rank_old = g.fact_key[best_code >> 1] + (best_code & 1);
              if (rank_new < rank_old) best_code = code;
            }
          }
        }
        for (; smask != 0; smask &= smask - 1) {
          int const j = __ffs(smask) - 1;
          uint32_t const vj = static_cast<uint32_t>(ys >> (j * lx)) & rm;
          int const b = j + 1 == ly ? 0 : j + 1;
          W const yb = rows_by(ys, b);
          for (int a = 0; a < lx; ++a) {
            if ((((vj >> a) | (vj << (lx - a))) & rm) != xt) continue;
            if (columns_by(yb, a) == x) {
              double const re = g.eig_re[g.fact_elem[(q * ly + b) * lx + a]];
              nn = nn + ((s == 1 && SI == -1) ? -re : re);
            }
          }
        }
      }
    }
  } else {
  for (int q = 0; q < nq; ++q) {
    W const y = group_apply<W, D>(g, g.fact_q[q], x);
#pragma unroll
    for (int s = 0; s < (SI != 0 ? 2 : 1); ++s) {
      W row = s == 1 ? static_cast<W>(y ^ flip) : y;
      for (int b = 0; b < ly; ++b) {
        W w = row;
        int const k0 = (q * ly + b) * lx;
        for (int a = 0; a < lx; ++a) {
          int const code = 2 * (k0 + a) + s;
          if (w < best) {
            best = w;
            best_code = code;
          } else if (w == best && best_code >= 0 && w != x) {
            // tie below x: the lower rank in the reference's reduction wins
            int const rank_new = g.fact_key[k0 + a] + s;
            int const rank_old = g.fact_key[best_code >> 1] + (best_code & 1);
            if (rank_new < rank_old) best_code = code;
          }
          if (w == x) {
            double const re = g.eig_re[g.fact_elem[k0 + a]];
            nn = nn + ((s == 1 && SI == -1) ? -re : re);
          }
          w = static_cast<W>(((w >> 1) & m1) | ((w << (lx - 1)) & m2));
        }
        if (ly > 1) row = static_cast<W>((row >> lx) | ((row << up) & flip));
      }
    }
  }
  }
  StateInfo out;
  out.rep = static_cast<uint64_t>(best);
  if (best_code < 0) {
    out.c_re = 1.0;
    out.c_im = 0.0;
  } else {
    int const e = g.fact_elem[best_code >> 1];
    double const cre = g.eig_re[e], cim = g.eig_im[e];
    bool const neg = SI == -1 && (best_code & 1);
    out.c_re = neg ? -cre : cre;
    out.c_im = neg ? -cim : cim;
  }
  int const G = g.size;
  double const denom = SI == 0 ? static_cast<double>(G) : static_cast<double>(2 * G);
  out.norm = (g.norm_eps > 0.0 && !(nn > g.norm_eps)) ? 0.0 : sqrt(nn / denom);
  return out;
}

// ---------------------------------------------------------------------------
// Least image and stabiliser sum from the elements that reach the minimum
// ---------------------------------------------------------------------------
//
// The searches below visit every element that can reach the orbit minimum and
// no others.  The elements reaching it form a coset of the stabiliser of x,
// so with characters +-1 their signed count is +-(sum of chi over the
// stabiliser), and 0 exactly when that sum is 0.  The character is that of
// the lowest-ranked element of the coset (state_info_factored), or 1 when x
// itself is the minimum.  A symmetric sector (fact_uniform) reads no tables.
template <typename W, int SI> struct OrbitMinimum {
  W best = ~W{0};
  int code = -1; // 2 k + s of the lowest-ranked element reaching best
  int sum = 0;   // signed number of them
  __device__ __forceinline__ void visit(GroupView const &g, W w, int k, int s) {
    if (w > best) return;
    if (w < best) {
      best = w;
      sum = 0;
      code = -1;
    }
    int sign = (SI == -1 && s == 1) ? -1 : 1;
    int const now = 2 * k + s;
    if (!g.fact_uniform) {
      sign = g.eig_re[g.fact_elem[k]] < 0.0 ? -sign : sign;
      if (code >= 0 && g.fact_key[code >> 1] + (code & 1) < g.fact_key[k] + s) {
        sum += sign;
        return;
      }
    }
    code = now;
    sum += sign;
  }
  // norm_1: sqrt(1 / denom), the norm of a state without a stabiliser
  __device__ __forceinline__ StateInfo info(GroupView const &g, W x, double norm_1) const {
    StateInfo out;
    out.rep = static_cast<uint64_t>(best);
    if (best == x) {
      out.c_re = 1.0;
      out.c_im = 0.0;
    } else {
      int const e = g.fact_uniform ? 0 : g.fact_elem[code >> 1];
      double const cre = g.eig_re[e], cim = g.eig_im[e];
      bool const neg = SI == -1 && (code & 1);
      out.c_re = neg ? -cre : cre;
      out.c_im = neg ? -cim : cim;
    }
    int const count = sum < 0 ? -sum : sum;
    if (count == 1 && g.norm_eps <= 0.0) {
      out.norm = norm_1;
    } else {
      double const nn = static_cast<double>(count);
      double const denom = static_cast<double>(SI == 0 ? g.size : 2 * g.size);
      out.norm = (g.norm_eps > 0.0 && !(nn > g.norm_eps)) ? 0.0 : sqrt(nn / denom);
    }
    return out;
  }
};

template <int SI> __device__ __forceinline__ double free_orbit_norm(GroupView const &g) {
  return sqrt(1.0 / static_cast<double>(SI == 0 ? g.size : 2 * g.size));
}

// Row-pair search (GroupView::line_*; rows of at most 6 sites).  The least
// image has the least two top rows, and those are a pair of neighbouring
// rows of base(x) for a class base, possibly mirrored, upside down, rotated
// and flipped: one table lookup per pair gives the least value all of those
// can give.  The minimum over the 2 ly pairs (6x6: 12 lookups) leaves, most
// often, the one image that is the orbit minimum, and only the images that
// reach it are formed, row by row.
//
// On the 6x6 lattice (576 elements) this replaces 8 networks of 11 stages,
// 96 row lookups and the divergent loops that formed every image with the
// least top row, and the images in x's own class for the stabiliser sum:
// state_info of the 15.8 M representatives takes 0.50 ms against 1.87 ms
// (state_info_factored); the CSR fill's 1.17 G searches, index lookups and
// counting atomics take 43 ms, the pairs dealt to lanes (181 ms with
// state_info_factored, one lane to a row and no atomics).  Bound by VALU and LDS lookups in the first part, by divergence over the
// images that are formed in the second.
template <typename W, int SI> struct LineSearch {
  W *base, *kept;       // LDS: images of rows under the class bases; one base image per lane and class
  uint16_t const *key;  // LDS
  uint8_t const *rot;   // LDS
  double norm_1;

  static __host__ __device__ size_t lds_bytes(int classes, int lx, int ly, int threads) {
    size_t const nv = size_t{1} << lx;
    return sizeof(W) * (static_cast<size_t>(classes - 1) * (ly * nv + threads)) + 2 * (nv << lx) +
           (2 * lx * nv + 7) / 8 * 8;
  }

  // Every thread of the workgroup must call it; a barrier follows.
  __device__ __forceinline__ void stage(GroupView const &g, void *smem) {
    int const lx = g.fact_lx, nv = 1 << lx, nb = (g.line_classes - 1) * g.fact_ly * nv, pairs = nv << lx;
    base = static_cast<W *>(smem);
    kept = base + nb;
    auto *k = reinterpret_cast<uint16_t *>(kept + static_cast<size_t>(g.line_classes - 1) * blockDim.x);
    auto *r = reinterpret_cast<uint8_t *>(k + pairs);
    for (int i = threadIdx.x; i < nb; i += blockDim.x) base[i] = static_cast<W>(g.line_base[i]);
    for (int i = threadIdx.x; i < pairs / 2; i += blockDim.x)
      reinterpret_cast<uint32_t *>(k)[i] = reinterpret_cast<uint32_t const *>(g.line_key)[i];
    for (int i = threadIdx.x; i < 2 * lx * nv; i += blockDim.x) r[i] = g.line_rot[i];
    key = k;
    rot = r;
    norm_1 = free_orbit_norm<SI>(g);
  }

  __device__ __forceinline__ uint32_t pair(W y, int j, int lx, int top, uint32_t rm, uint32_t pm) const {
    if (j * lx == top) return ((static_cast<uint32_t>(y) & rm) << lx) | (static_cast<uint32_t>(y >> top) & rm);
    return static_cast<uint32_t>(y >> (j * lx)) & pm;
  }

  __device__ __forceinline__ OrbitMinimum<W, SI> minimum(GroupView const &g, W x) const {
    int const lx = g.fact_lx, ly = g.fact_ly, top = (ly - 1) * lx;
    uint32_t const rm = (1u << lx) - 1, pm = (1u << (2 * lx)) - 1;
    W const all = static_cast<W>(g.flip);
    uint32_t least = ~0u, hits = 0; // bit c * ly + j: pair j of class c reaches it
    for (int c = 0; c < g.line_classes; ++c) {
      W y = x;
      if (c > 0) {
        W const *b = base + static_cast<size_t>(c - 1) * (ly << lx);
        y = 0;
#pragma unroll
        for (int r = 0; r < kMaxLineRows; ++r)
          if (r < ly) y |= b[(r << lx) + static_cast<int>(static_cast<uint32_t>(x >> (r * lx)) & rm)];
        kept[static_cast<size_t>(c - 1) * blockDim.x + threadIdx.x] = y;
      }
#pragma unroll
      for (int j = 0; j < kMaxLineRows; ++j)
        if (j < ly) {
          uint32_t const k = key[pair(y, j, lx, top, rm, pm)];
          hits = k < least ? 0u : hits;
          least = k < least ? k : least;
          hits |= (k == least ? 1u : 0u) << (c * ly + j);
        }
    }
    OrbitMinimum<W, SI> out;
    uint64_t mask = 0;
    W y = x;
    int c = 0, j = 0;
    while ((hits | static_cast<uint32_t>(mask) | static_cast<uint32_t>(mask >> 32)) != 0) {
      if (mask == 0) {
        int const h = __ffs(hits) - 1;
        hits &= hits - 1;
        c = h / ly;
        j = h - c * ly;
        y = c == 0 ? x : kept[static_cast<size_t>(c - 1) * blockDim.x + threadIdx.x];
        mask = g.line_mask[pair(y, j, lx, top, rm, pm)];
      }
      int const bit = __ffsll(static_cast<unsigned long long>(mask)) - 1;
      mask &= mask - 1;
      int const a = bit & 7, s = (bit >> 3) & 1, v = bit >> 4; // v: mirrored + 2 * upside down
      bool const up = (v & 2) != 0;
      int const row = up ? j : (j + 1 == ly ? 0 : j + 1); // of y, the image's top row
      int const at = up && row != 0 ? ly - row : row;     // its place in the point element's image
      uint8_t const *rt = rot + (((v & 1) * lx + a) << lx);
      // y flipped and turned so that its rows run from the image's top row
      // down (or up, upside down): the rows below it first
      W z = s ? static_cast<W>(y ^ all) : y;
      int const turn = (up ? row : (row + 1 == ly ? 0 : row + 1)) * lx;
      z = turn == 0 ? z : static_cast<W>(((z & all) >> turn) | ((z << (g.nbits - turn)) & all));
      W w = 0;
#pragma unroll
      for (int i = 0; i < kMaxLineRows; ++i)
        if (i < ly) w = static_cast<W>(w << lx) | rt[static_cast<uint32_t>(z >> (up ? i * lx : top - i * lx)) & rm];
      int const k = g.fact_uniform ? 0 : (g.line_q[4 * c + v] * ly + (at + 1 == ly ? 0 : at + 1)) * lx + a;
      out.visit(g, w, k, s);
    }
    return out;
  }

  __device__ __forceinline__ StateInfo info(GroupView const &g, uint64_t x) const {
    return minimum(g, static_cast<W>(x)).info(g, static_cast<W>(x), norm_1);
  }
};

// Run search (chains: one row of n sites).  The least rotation of a word
// starts, at its top, with its longest run of zeros, so of the n rotations of
// every q(x) and its flipped copy only those that bring a longest run to the
// top are formed.  rotl(z, L) & rotl(z, L - 1) & .. & z leaves one bit at the
// top end of every run of at least L + 1 zeros.  On the 32-site chain (64
// elements with parity, flipped copies too) about 5 such steps and 2 images
// per word replace 32 rotations: the on-the-fly product takes 1.75 ms against
// 5.76 ms with all rotations formed (one lane to a row; 1.92 ms so with this
// search).  Bound by VALU work; a word per point
// element and flip is kept in LDS, so at most kMaxRunPoints of them.
template <typename W, int D, int SI> struct RunSearch {
  static constexpr int kFlips = SI != 0 ? 2 : 1;
  W *kept; // LDS: [2 kMaxRunPoints][2][threads]: word, run ends
  double norm_1;
  static __host__ __device__ size_t lds_bytes(int threads) {
    return sizeof(W) * 2 * (kFlips * kMaxRunPoints) * static_cast<size_t>(threads);
  }
  __device__ __forceinline__ void stage(GroupView const &g, void *smem) {
    kept = static_cast<W *>(smem);
    norm_1 = free_orbit_norm<SI>(g);
  }
  __device__ __forceinline__ OrbitMinimum<W, SI> minimum(GroupView const &g, W x) const {
    int const n = g.nbits;
    W const all = static_cast<W>(g.flip);
    int longest = -1;
    uint32_t hits = 0;
#pragma unroll
    for (int q = 0; q < kMaxRunPoints; ++q) {
      if (q >= g.run_points) continue;
      W const y = group_apply<W, D>(g, g.fact_q[q], x);
#pragma unroll
      for (int s = 0; s < kFlips; ++s) {
        int const c = q * kFlips + s;
        W const ys = s == 1 ? static_cast<W>(y ^ all) : y;
        W ends = all, z = static_cast<W>(~ys & all);
        int run = 0;
        while (run < n && (ends & z) != 0) {
          ends &= z;
          z = static_cast<W>(((z << 1) | (z >> (n - 1))) & all);
          ++run;
        }
        hits = run > longest ? 0u : hits;
        longest = run > longest ? run : longest;
        hits |= (run == longest ? 1u : 0u) << c;
        kept[(2 * c) * blockDim.x + threadIdx.x] = ys;
        kept[(2 * c + 1) * blockDim.x + threadIdx.x] = ends;
      }
    }
    OrbitMinimum<W, SI> out;
    W ends = 0, ys = 0;
    int c = 0;
    while (hits != 0 || ends != 0) {
      if (ends == 0) {
        c = __ffs(hits) - 1;
        hits &= hits - 1;
        ys = kept[(2 * c) * blockDim.x + threadIdx.x];
        ends = kept[(2 * c + 1) * blockDim.x + threadIdx.x];
      }
      int const p = __ffsll(static_cast<unsigned long long>(ends)) - 1;
      ends &= ends - 1;
      int const a = p + 1 == n ? 0 : p + 1; // the rotation that takes bit p to the top
      W const w = a == 0 ? ys : static_cast<W>(((ys >> a) | (ys << (n - a))) & all);
      out.visit(g, w, (c / kFlips) * n + a, c % kFlips);
    }
    return out;
  }
  __device__ __forceinline__ StateInfo info(GroupView const &g, uint64_t x) const {
    return minimum(g, static_cast<W>(x)).info(g, static_cast<W>(x), norm_1);
  }
};

// Spinful search (GroupView::species_*).  Every element acts alike on the two
// species, and the down species holds the high bits, so the least image has
// the least image of the down state, reached by a few elements (one, unless
// the down state has a stabiliser) that a table lists; only their images of
// the up state are formed.  Signs come from a bit table per species: the
// species do not pass each other.  On the 4x4 Hubbard sector (128 elements)
// this replaces 128 networks of 9 stages per state: the complex on-the-fly
// product takes 1.68 ms against 13.6 ms (11.8 ms element by element with the
// pairs dealt to lanes), now bound by its atomics (42 G/s), and the norms 0.02 ms.
template <typename W, int D> struct SpeciesSearch {
  W *masks; // LDS: the networks, element-major
  double norm_1;

  // Every thread of the workgroup must call it; a barrier follows.
  __device__ __forceinline__ void stage(GroupView const &g, void *smem) {
    masks = static_cast<W *>(smem);
    int const count = g.size * g.depth;
    for (int i = threadIdx.x; i < count; i += blockDim.x) masks[i] = static_cast<W>(g.masks[i]);
    norm_1 = sqrt(1.0 / static_cast<double>(g.size));
  }

  __device__ __forceinline__ bool odd(GroupView const &g, int e, uint32_t s, int words) const {
    return (g.species_sign[static_cast<size_t>(e) * words + (s >> 5)] >> (s & 31) & 1u) != 0;
  }

  __device__ __forceinline__ W up_image(GroupView const &g, int e, W up) const {
    return benes_apply_ptr<W, D>(masks + static_cast<size_t>(e) * g.depth, up, g.shifts, g.depth);
  }

  __device__ __forceinline__ StateInfo info(GroupView const &g, uint64_t x) const {
    int const sites = g.nbits / 2, words = ((1 << sites) + 31) / 32;
    uint32_t const mask = (1u << sites) - 1;
    uint32_t const up = static_cast<uint32_t>(x) & mask, down = static_cast<uint32_t>(x >> sites) & mask;
    uint64_t const entry = g.species_entry[down];
    int const count = static_cast<int>(entry >> 16 & 0xffffu);
    uint16_t const *list = g.species_list + (entry >> 32);
    W best = ~W{0};
    int element = 0, sum = 0;
    double sign = 1.0;
    for (int i = 0; i < count; ++i) {
      int const e = list[i];
      W const y = up_image(g, e, static_cast<W>(up));
      if (y > best) continue;
      bool const minus = odd(g, e, up, words) != odd(g, e, down, words);
      int const term = (g.eig_re[e] < 0.0) != minus ? -1 : 1;
      if (y < best || g.species_rank[e] < g.species_rank[element]) { // of equal images the lowest rank
        element = e;
        sign = minus ? -1.0 : 1.0;
      }
      sum = y < best ? term : sum + term;
      best = y;
    }
    StateInfo out;
    out.rep = (entry & 0xffffu) << sites | static_cast<uint64_t>(best);
    if (out.rep == x) {
      out.c_re = 1.0;
      out.c_im = 0.0;
    } else {
      out.c_re = g.eig_re[element] * sign;
      out.c_im = g.eig_im[element] * sign;
    }
    int const n = sum < 0 ? -sum : sum;
    if (n == 1 && g.norm_eps <= 0.0) {
      out.norm = norm_1;
    } else {
      double const nn = static_cast<double>(n);
      out.norm = (g.norm_eps > 0.0 && !(nn > g.norm_eps)) ? 0.0 : sqrt(nn / static_cast<double>(g.size));
    }
    return out;
  }
};

// state_info of one kernel kind, with its tables staged in LDS: static shared
// memory for kFactored, dynamic at `smem` (search_lds_bytes) for the others.
template <typename W, int D, int SI, int KIND> struct OrbitSearch {
  __device__ __forceinline__ void stage(GroupView const &, void *) {}
  __device__ __forceinline__ StateInfo info(GroupView const &g, uint64_t x) const { return state_info_one<W, D, SI>(g, x); }
};
template <typename W, int D, int SI> struct OrbitSearch<W, D, SI, kFactored> {
  RowTables const *rt;
  __device__ __forceinline__ void stage(GroupView const &g, void *) {
    __shared__ RowTables tables;
    row_tables_init(g, tables);
    rt = &tables;
  }
  __device__ __forceinline__ StateInfo info(GroupView const &g, uint64_t x) const {
    return state_info_factored<W, D, SI>(g, x, rt);
  }
};
template <typename W, int D, int SI> struct OrbitSearch<W, D, SI, kLines> : LineSearch<W, SI> {
  __device__ __forceinline__ void stage(GroupView const &g, void *smem) {
    LineSearch<W, SI>::stage(g, smem);
    __syncthreads();
  }
};
template <typename W, int D, int SI> struct OrbitSearch<W, D, SI, kRuns> : RunSearch<W, D, SI> {};
template <typename W, int D, int SI> struct OrbitSearch<W, D, SI, kSpecies> : SpeciesSearch<W, D> {
  __device__ __forceinline__ void stage(GroupView const &g, void *smem) {
    SpeciesSearch<W, D>::stage(g, smem);
    __syncthreads();
  }
};

template <typename W, int D, int SI, int KIND> size_t search_lds_bytes(GroupData const *g, int threads) {
  if constexpr (KIND == kLines) return LineSearch<W, SI>::lds_bytes(g->line_classes, g->fact_lx, g->fact_ly, threads);
  if constexpr (KIND == kRuns) return RunSearch<W, D, SI>::lds_bytes(threads);
  if constexpr (KIND == kSpecies) return species_lds_bytes(*g);
  return 0;
}

// ---------------------------------------------------------------------------
// is_representative (generator.cpp:168-272)
// ---------------------------------------------------------------------------
//
// Chunks of four elements (natural_vector_size(uint64) on avx2): within a
// chunk the terms (y == x) * Re(chi) are summed from 0 in order and the chunk
// sum is added to the total; the flag is the AND of y >= x (and y^flip >= x).
// Chunks stop after the first one that clears the flag; the remaining
// |G| mod 4 elements are always folded in.  is_rep = norm > 0 ? flag : 0.

template <typename W, int D, int SI>
__device__ __forceinline__ void is_rep_term(GroupView const &g, int e, W x,
                                            double &t, bool &f) {
  W const y = group_apply<W, D>(g, e, x);
  double re = g.eig_re[e];
  if constexpr (SI == kFermionic) {
    if (y == x) re = re * fermion_sign(g, e, static_cast<uint64_t>(x));
    t = static_cast<double>(y == x) * re;
    f = y >= x;
  } else if constexpr (SI == 0) {
    t = static_cast<double>(y == x) * re;
    f = y >= x;
  } else {
    W const yf = static_cast<W>(y ^ static_cast<W>(g.flip));
    double const a = static_cast<double>(y == x);
    double const b = static_cast<double>(yf == x);
    t = (SI == 1 ? (a + b) : (a - b)) * re;
    f = (y >= x) && (yf >= x);
  }
}

template <typename W, int D, int SI>
__device__ __forceinline__ void is_representative_one(GroupView const &g,
                                                      uint64_t x64,
                                                      uint8_t &flag_out,
                                                      double &norm_out) {
  constexpr int L = kIsRepresentativeLanes;
  W const x = static_cast<W>(x64);
  int const G = g.size;
  int const nch = G / L;
  double total = 0.0;
  bool flag = true;
  for (int c = 0; c < nch; ++c) {
    if (!flag) break;
    double lane = 0.0;
    bool lf = true;
#pragma unroll
    for (int j = 0; j < L; ++j) {
      double t;
      bool f;
      is_rep_term<W, D, SI>(g, c * L + j, x, t, f);
      lane = lane + t;
      lf = lf && f;
    }
    total = total + lane;
    flag = flag && lf;
  }
  for (int e = nch * L; e < G; ++e) {
    double t;
    bool f;
    is_rep_term<W, D, SI>(g, e, x, t, f);
    total = total + t;
    flag = flag && f;
  }
  norm_out = total;
  flag_out = (total > g.norm_eps) ? static_cast<uint8_t>(flag) : static_cast<uint8_t>(0);
}

// ---------------------------------------------------------------------------
// State index lookup over the prefix table (indexing.c:273-325 semantics)
// ---------------------------------------------------------------------------
__device__ __forceinline__ int64_t index_lookup(IndexView const &idx, uint64_t x) {
  uint64_t const b = x >> idx.shift;
  if (b >= (uint64_t{1} << idx.prefix_bits)) return -1;
  int64_t lo = idx.offsets[b];
  int64_t n = static_cast<int64_t>(idx.offsets[b + 1]) - lo;
  // branch-free lower bound in [lo, lo + n)
  while (n > 0) {
    int64_t const half = n >> 1;
    uint64_t const v = idx.reps[lo + half];
    bool const less = v < x;
    lo = less ? lo + half + 1 : lo;
    n = less ? n - half - 1 : half;
  }
  uint64_t const hi_bucket_end = idx.offsets[b + 1];
  return (static_cast<uint64_t>(lo) < hi_bucket_end && idx.reps[lo] == x) ? lo : -1;
}

// ---------------------------------------------------------------------------
// Dispatch on (word type, Benes depth, spin inversion)
// ---------------------------------------------------------------------------
//
// f is a generic callable invoked as f.template operator()<W, D, SI>().
// Canonical networks of depth 7 and 9 (9..32 sites) run on 32-bit words,
// depth 11 (33..64 sites) on 64-bit words; anything else uses the runtime
// depth path.
template <typename F> bool dispatch_group(GroupData const &g, F &&f) {
  auto by_si = [&]<typename W, int D>() -> bool {
    if (g.fermion_species != 0) return f.template operator()<W, D, kFermionic>();
    switch (g.spin_inversion) {
    case 0: return f.template operator()<W, D, 0>();
    case 1: return f.template operator()<W, D, 1>();
    case -1: return f.template operator()<W, D, -1>();
    default: return fail("invalid spin_inversion");
    }
  };
  if (g.canonical_shifts) {
    switch (g.depth) {
    case 7: return by_si.template operator()<uint32_t, 7>();
    case 9: return by_si.template operator()<uint32_t, 9>();
    case 11: return by_si.template operator()<uint64_t, 11>();
    default: break;
    }
  }
  return by_si.template operator()<uint64_t, 0>();
}

// Dispatch on (W, D, SI, KIND) of the orbit search of a group: the row-pair,
// run or spinful search where the group has one and its tables fit LDS beside the `lds`
// bytes the kernel needs for itself, else the factorised search where it
// factors (`factored` allowed), else element by element.  The row-pair search
// applies no networks, so its kernels do not depend on the depth.
constexpr size_t kSearchLds = 64 << 10;

template <typename F> bool dispatch_search(GroupData const &g, bool factored, size_t lds, F &&f) {
  return dispatch_group(g, [&]<typename W, int D, int SI>() -> bool {
    if constexpr (SI != kFermionic) {
      if (factored && g.lines() && lds + search_lds_bytes<W, 0, SI, kLines>(&g, 256) <= kSearchLds)
        return f.template operator()<W, 0, SI, kLines>();
      if (factored && g.runs() && lds + search_lds_bytes<W, D, SI, kRuns>(&g, 256) <= kSearchLds)
        return f.template operator()<W, D, SI, kRuns>();
      if (factored && g.factored()) return f.template operator()<W, D, SI, kFactored>();
    } else {
      if (factored && g.species() && lds + species_lds_bytes(g) <= kSearchLds)
        return f.template operator()<W, D, SI, kSpecies>();
    }
    return f.template operator()<W, D, SI, kPermutations>();
  });
}

inline int grid_for(int64_t n, int block) {
  int64_t const b = (n + block - 1) / block;
  return static_cast<int>(b < 1 ? 1 : b);
}

} // namespace lsamd
