// operator.hip -- term application, fused product and the CSR cache's build.
//
// The reference applies H in push form: every representative alpha_i emits
// (beta, c) pairs, c is rescaled by chi_beta n_beta / n_alpha after
// state_info, and y[index(rep beta)] += Re(c) x_i with relaxed atomics
// (chapel/src/BatchedOperator.chpl:207-253,
// chapel/src/DistributedMatrixVector.chpl:91-143).  The engine computes the
// same matrix M, M[index(rep beta), i] = C, for every operator, Hermitian or
// not:
// - the fused on-the-fly product is push form too: one lane per (alpha_i,
//   term) pair, the diagonal pass first, then atomic adds of Re(c) (or c x_i
//   for complex vectors) into y;
// - the CSR build emits the pairs of every alpha_i and turns them into target
//   rows on the device: with a value table the fill pass counts and places the
//   targets and one scatter writes the final words; otherwise the entries are
//   counted, scattered and sorted by key.  Row j of the cached matrix holds
//   every (i, C) with target j, in ascending i.  Products then gather x along
//   a row and write y once, without atomics, and every build stores the same
//   bits.
#include <algorithm>
#include <cstring>

#include "operator_internal.hpp"
#include "orbit_device.hpp"

namespace lsamd {

// ---------------------------------------------------------------------------
// Terms
// ---------------------------------------------------------------------------

bool Terms::load(ls_hs_nonbranching_terms const *t) {
  count = 0;
  h_v.clear();
  h_m.clear();
  h_r.clear();
  h_x.clear();
  h_s.clear();
  if (t == nullptr || t->number_terms == 0) return true;
  if (t->number_bits > 64) return fail("bases with more than 64 bits are not yet implemented");
  count = t->number_terms;
  h_v.resize(2 * static_cast<size_t>(count));
  std::memcpy(h_v.data(), t->v, sizeof(double) * 2 * count);
  h_m.assign(t->m, t->m + count);
  h_r.assign(t->r, t->r + count);
  h_x.assign(t->x, t->x + count);
  h_s.assign(t->s, t->s + count);
  std::vector<uint64_t> actions(4 * static_cast<size_t>(count));
  for (int k = 0; k < count; ++k) {
    actions[4 * k] = h_x[k];
    actions[4 * k + 1] = h_s[k];
    std::memcpy(&actions[4 * k + 2], &h_v[2 * k], 16);
  }
  return d_actions.upload(actions.data(), actions.size()) && d_v.upload(h_v.data(), h_v.size()) && d_m.upload(h_m.data(), count) &&
         d_r.upload(h_r.data(), count) && d_x.upload(h_x.data(), count) &&
         d_s.upload(h_s.data(), count);
}

uint64_t Terms::fingerprint() const {
  uint64_t h = 1469598103934665603ull ^ static_cast<uint64_t>(count);
  auto mix = [&](uint64_t v) {
    h ^= v;
    h *= 1099511628211ull;
  };
  for (int i = 0; i < count; ++i) {
    uint64_t vb[2];
    std::memcpy(vb, &h_v[2 * i], 16);
    mix(vb[0]);
    mix(vb[1]);
    mix(h_m[i]);
    mix(h_r[i]);
    mix(h_x[i]);
    mix(h_s[i]);
  }
  return h;
}

// ---------------------------------------------------------------------------
// reference.c:67-134 on device arrays
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void apply_diag_kernel(TermsView t, int64_t count,
                                                         uint64_t const *__restrict__ alphas,
                                                         double *__restrict__ ys,
                                                         double const *__restrict__ xs) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint64_t const a = alphas[i];
  double acc = 0;
  for (int k = 0; k < t.count; ++k) {
    int const delta = (a & t.m[k]) == t.r[k];
    if (delta) {
      int const sign = 1 - 2 * (__popcll(a & t.s[k]) % 2);
      double const factor =
          xs != nullptr ? static_cast<double>(delta * sign) * xs[i] : static_cast<double>(delta * sign);
      acc += t.v[2 * k] * factor;
    }
  }
  ys[i] = acc;
}

__global__ __launch_bounds__(256) void count_applicable_kernel(TermsView t, int64_t count,
                                                               uint64_t const *__restrict__ alphas,
                                                               uint32_t *__restrict__ counts) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint64_t const a = alphas[i];
  uint32_t c = 0;
  for (int k = 0; k < t.count; ++k) c += (a & t.m[k]) == t.r[k];
  counts[i] = c;
}

__global__ __launch_bounds__(256) void apply_off_diag_kernel(TermsView t, int64_t count,
                                                             uint64_t const *__restrict__ alphas,
                                                             double const *__restrict__ xs,
                                                             int64_t const *__restrict__ offsets,
                                                             uint64_t *__restrict__ betas,
                                                             double *__restrict__ coeffs) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint64_t const a = alphas[i];
  int64_t o = offsets[i];
  for (int k = 0; k < t.count; ++k) {
    int const delta = (a & t.m[k]) == t.r[k];
    if (delta) {
      int const sign = 1 - 2 * (__popcll(a & t.s[k]) % 2);
      double const factor =
          xs != nullptr ? static_cast<double>(delta * sign) * xs[i] : static_cast<double>(delta * sign);
      coeffs[2 * o] = t.v[2 * k] * factor;
      coeffs[2 * o + 1] = t.v[2 * k + 1] * factor;
      betas[o] = a ^ t.x[k];
      ++o;
    }
  }
}

bool apply_diag_device(Terms const &t, int64_t count, uint64_t const *d_alphas, double *d_ys,
                       double const *d_xs) {
  if (count <= 0) return true;
  if (t.count == 0) {
    LSAMD_HIP(hipMemsetAsync(d_ys, 0, sizeof(double) * count, stream()));
    return true;
  }
  apply_diag_kernel<<<grid_for(count, 256), 256, 0, stream()>>>(t.view(), count, d_alphas, d_ys, d_xs);
  LSAMD_HIP(hipGetLastError());
  return true;
}

bool apply_off_diag_device(Terms const &t, int64_t count, uint64_t const *d_alphas,
                           double const *d_xs, DeviceArray<uint64_t> &betas,
                           DeviceArray<double> &coeffs, DeviceArray<int64_t> &offsets,
                           int64_t &total) {
  total = 0;
  if (!offsets.allocate(static_cast<size_t>(count + 1))) return false;
  if (t.count == 0 || count == 0) {
    LSAMD_HIP(hipMemsetAsync(offsets.ptr, 0, sizeof(int64_t) * (count + 1), stream()));
    betas.reset();
    coeffs.reset();
    return true;
  }
  DeviceArray<uint32_t> counts;
  if (!counts.allocate(static_cast<size_t>(count))) return false;
  count_applicable_kernel<<<grid_for(count, 256), 256, 0, stream()>>>(t.view(), count, d_alphas,
                                                                     counts.ptr);
  LSAMD_HIP(hipGetLastError());
  uint64_t tot = 0;
  if (!exclusive_scan(counts.ptr, count, reinterpret_cast<uint64_t *>(offsets.ptr), tot)) return false;
  int64_t const tot_i = static_cast<int64_t>(tot);
  LSAMD_HIP(hipMemcpyAsync(offsets.ptr + count, &tot_i, sizeof(int64_t), hipMemcpyHostToDevice, stream()));
  if (!betas.allocate(static_cast<size_t>(tot > 0 ? tot : 1))) return false;
  if (!coeffs.allocate(static_cast<size_t>(2 * (tot > 0 ? tot : 1)))) return false;
  apply_off_diag_kernel<<<grid_for(count, 256), 256, 0, stream()>>>(t.view(), count, d_alphas, d_xs,
                                                                   offsets.ptr, betas.ptr, coeffs.ptr);
  LSAMD_HIP(hipGetLastError());
  LSAMD_HIP(hipStreamSynchronize(stream()));
  total = tot_i;
  return true;
}

// ---------------------------------------------------------------------------
// Fused product
// ---------------------------------------------------------------------------

struct OpView {
  TermsView diag;
  TermsView off;
  IndexView idx;
  double const *norms;
  int64_t n;
  uint64_t flip;
  int identity_index;
};

OpView make_view(OperatorCore const &op) {
  return OpView{op.diag.view(), op.off.view(), op.index, op.d_norms, op.number_states,
                op.number_bits >= 64 ? ~uint64_t{0} : ((uint64_t{1} << op.number_bits) - 1),
                op.identity_index ? 1 : 0};
}

__device__ __forceinline__ int64_t target_index(OpView const &op, uint64_t beta) {
  return op.identity_index ? static_cast<int64_t>(beta) : index_lookup(op.idx, beta);
}

// Off-diagonal terms: the masks that every row is tested against staged in
// LDS, what an applicable term does read from memory (it is a few KB, and the
// LDS it does not take makes room for more workgroups).
struct TermsLds {
  uint64_t *m, *r;
  ulonglong2 const *__restrict__ actions;
};

__device__ __forceinline__ TermsLds stage_terms(TermsView const &t, uint64_t *smem) {
  int const T = t.count;
  TermsLds l{smem, smem + T, reinterpret_cast<ulonglong2 const *>(t.actions)};
  for (int k = threadIdx.x; k < T; k += blockDim.x) {
    l.m[k] = t.m[k];
    l.r[k] = t.r[k];
  }
  __syncthreads();
  return l;
}

inline size_t terms_lds_bytes(int T) { return static_cast<size_t>(T) * 16; }

// The (row, term) pairs of the source rows, one wave at a time.  A wave owns
// `rows` consecutive rows (a power of two, at most 64) and tests 64 / rows
// terms of all of them per step, lane t * rows + r the term k + t of row r.
// The applicable pairs join a queue in LDS, and whenever it holds 64 of them
// every lane takes one.  No lane idles while a neighbour finishes a longer
// row (about 20 % on 6x6 with one lane to a row), and a wave's 64 pairs are
// one or two terms on neighbouring rows: their targets lie close together, so
// the index lookups and the atomics share cache lines.  Listing a row's pairs
// together instead spreads every wave over the whole basis: 57 against 43 ms
// for the CSR fill on 6x6.  One lane to a row: 81 ms there without the counting
// atomics, and 1.92 against 1.75 ms for the 32-site chain's on-the-fly product.
// The 6x6 fill issues 1.7e10 VALU instructions (28 of its 43 ms) and misses L2
// 1.77 G times under lookups and counting atomics (41 G/s; random atomics alone
// reach the basis at 42 G/s), so it is bound by both.
constexpr int kPairThreads = 256;
constexpr int kWaveRows = 64;
constexpr int kPairTermBits = 13; // of a term and of a pair's rank in its row
constexpr int kMaxPairTerms = 1 << kPairTermBits;

struct WaveRows {
  uint64_t alpha[kWaveRows];
  double norm[kWaveRows];  // state_info norm of alpha
  uint32_t queue[2 * 64];  // row << 26 | term << 13 | rank among the row's applicable terms
};
constexpr size_t kPairLds = sizeof(WaveRows) * (kPairThreads / 64);

// Rows of a wave: enough waves for the chip first; more rows share more cache
// lines, fewer leave less to the last waves.  Where the line lies depends on the
// cost of a pair.  On-the-fly product, ms at 4, 8, 16, 32, 64 rows:
//   107 k rows (6x6, weight 8)   0.59 0.54 0.60 1.00 1.90   (16 taken)
//   330 k rows (6x6, weight 9)   1.34 1.20 1.17 1.22 1.84   (64)
//   718 k rows (28-site chain)   0.65 0.58 0.54 0.55 0.55   (64)
//   4.4 M rows (6x6, weight 12)  12.7 11.2 10.5 10.2 10.2   (64)
// Doubling at 49 152 rows a step instead would win 6x6 with weight 9 (1.20 ms)
// and lose without an orbit search (185 k states of 20 sites, all pairs: 0.28 ->
// 0.37 ms, its CSR build 0.89 -> 1.06).
inline int wave_rows(int64_t n) {
  int rows = 4;
  while (rows < kWaveRows && n >= int64_t{8192} * rows) rows *= 2;
  return rows;
}
inline int pair_grid(int64_t n, int rows) { return grid_for(n, rows * (kPairThreads / 64)); }

// Loads the wave's rows [i0, i0 + count); no barrier follows (a wave reads
// only what it wrote).
template <bool NORMS>
__device__ __forceinline__ void load_rows(WaveRows &w, OpView const &op, int64_t i0, int count) {
  int const lane = static_cast<int>(threadIdx.x) & 63;
  if (lane < count) {
    w.alpha[lane] = op.idx.reps[i0 + lane];
    w.norm[lane] = NORMS ? op.norms[i0 + lane] : 1.0;
  }
  __builtin_amdgcn_wave_barrier();
}

// Calls take(row, term, rank, lane_of_step, pairs_before) on every pair; lanes
// without one sit out of the last step.
template <typename Take>
__device__ __forceinline__ void for_each_pair(WaveRows &w, TermsLds const &l, int T, int rows, int count, Take &&take) {
  int const lane = static_cast<int>(threadIdx.x) & 63;
  int const r = lane & (rows - 1), t = lane / rows, step = 64 / rows;
  uint64_t const a = r < count ? w.alpha[r] : 0;
  uint64_t row_lanes = 0; // the lanes that test this lane's row
  for (int q = 0; q < step; ++q) row_lanes |= uint64_t{1} << (q * rows + r);
  uint64_t const below = (uint64_t{1} << lane) - 1;
  uint32_t queued = 0, rank = 0;
  int64_t before = 0;
  auto drain = [&](uint32_t n) {
    __builtin_amdgcn_wave_barrier();
    if (static_cast<uint32_t>(lane) < n) {
      uint32_t const pair = w.queue[lane];
      take(static_cast<int>(pair >> 26), static_cast<int>(pair >> kPairTermBits & (kMaxPairTerms - 1)),
           static_cast<int>(pair & (kMaxPairTerms - 1)), before + lane);
    }
    before += n;
    __builtin_amdgcn_wave_barrier();
  };
  for (int k0 = 0; k0 < T; k0 += step) {
    int const k = k0 + t;
    bool const on = r < count && k < T && (a & l.m[k]) == l.r[k];
    uint64_t const mask = __ballot(on);
    if (mask == 0) continue;
    if (on)
      w.queue[queued + __popcll(mask & below)] = static_cast<uint32_t>(r) << 26 |
                                                 static_cast<uint32_t>(k) << kPairTermBits |
                                                 (rank + __popcll(mask & row_lanes & below));
    rank += static_cast<uint32_t>(__popcll(mask & row_lanes));
    queued += static_cast<uint32_t>(__popcll(mask));
    if (queued >= 64) {
      drain(64);
      queued -= 64;
      if (static_cast<uint32_t>(lane) < queued) w.queue[lane] = w.queue[64 + lane];
    }
  }
  if (queued > 0) drain(queued);
}

// Coefficient of term k for alpha with the factor `scale` (x_alpha, or 1):
// returns the representative of beta in `beta` and
// c = chi_beta v (-1)^popcount(alpha & s) scale n_beta / n_alpha in
// (c_re, c_im), with the reference's order of operations
// (reference.c:97-134 multiplies v by sign * x; BatchedOperator.chpl:241-247
// scales by n_beta / n_alpha and then multiplies by chi).
template <typename W, int D, int SI, int KIND>
__device__ __forceinline__ void off_diag_entry(GroupView const &g, OpView const &op,
                                               TermsLds const &l, int k, uint64_t alpha,
                                               double n_alpha, double scale, uint64_t &beta,
                                               double &c_re, double &c_im,
                                               OrbitSearch<W, D, SI, KIND> const &search) {
  ulonglong2 const xs = l.actions[2 * k], v = l.actions[2 * k + 1];
  double const factor = ((__popcll(alpha & xs.y) & 1) ? -1.0 : 1.0) * scale;
  double re = __longlong_as_double(static_cast<long long>(v.x)) * factor;
  double im = __longlong_as_double(static_cast<long long>(v.y)) * factor;
  beta = alpha ^ xs.x;
  if constexpr (KIND == kInversionOnly) {
    uint64_t const inv = beta ^ op.flip; // BatchedOperator.chpl:192-199
    if (inv < beta) {
      beta = inv;
      re *= static_cast<double>(SI);
      im *= static_cast<double>(SI);
    }
  } else if constexpr (projects_orbits(KIND)) {
    // BatchedOperator.chpl:232-247
    StateInfo const s = search.info(g, beta);
    double const t_re = (re * s.norm) / n_alpha;
    // a real term skips the division unless it would give NaN (a listed state of norm 0)
    double const t_im = im != 0.0 || !(n_alpha > 0.0) ? (im * s.norm) / n_alpha : im;
    re = s.c_re * t_re - s.c_im * t_im;
    im = s.c_re * t_im + s.c_im * t_re;
    beta = s.rep;
  }
  c_re = re;
  c_im = im;
}

__device__ __forceinline__ void record_error(int *err, uint64_t *err_state, uint64_t beta) {
  if (atomicCAS(err, 0, 1) == 0) *err_state = beta;
}

// Diagonal pass of the fused product (DistributedMatrixVector.chpl:34-71):
// y_i = sum_k Re(v_k) (-1)^.. x_i in the term order of reference.c:67-95;
// without diagonal terms y is zeroed, or left as it is when accumulating.
template <bool CPLX>
__global__ __launch_bounds__(256) void otf_diag_kernel(OpView op, double const *__restrict__ x,
                                                       double *__restrict__ y, int accumulate) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= op.n) return;
  if (op.diag.count == 0) {
    if (!accumulate) {
      if constexpr (CPLX) {
        y[2 * i] = 0.0;
        y[2 * i + 1] = 0.0;
      } else {
        y[i] = 0.0;
      }
    }
    return;
  }
  uint64_t const alpha = op.idx.reps[i];
  double const xr = CPLX ? x[2 * i] : x[i];
  double const xi = CPLX ? x[2 * i + 1] : 0.0;
  double base_re = 0, base_im = 0;
  for (int k = 0; k < op.diag.count; ++k) {
    if ((alpha & op.diag.m[k]) != op.diag.r[k]) continue;
    double const sign = (__popcll(alpha & op.diag.s[k]) & 1) ? -1.0 : 1.0;
    base_re += op.diag.v[2 * k] * (sign * xr);
    if constexpr (CPLX) base_im += op.diag.v[2 * k] * (sign * xi);
  }
  if constexpr (CPLX) {
    y[2 * i] = base_re;
    y[2 * i + 1] = base_im;
  } else {
    y[i] = base_re;
  }
}

// Off-diagonal pass, push form (DistributedMatrixVector.chpl:91-143): a lane
// takes one pair (alpha_i, term) at a time and adds it into y at index(rep
// beta).  Real vectors follow the reference exactly: c includes x_i, and a
// pair whose real part is 0 is skipped before the index lookup.  Complex
// vectors add c x_i for every nonzero c.
template <typename W, int D, int SI, int KIND, bool CPLX>
__global__ __launch_bounds__(kPairThreads) void otf_push_kernel(GroupView g, OpView op, int rows,
                                                                double const *__restrict__ x, double *__restrict__ y,
                                                                int *err, uint64_t *err_state) {
  extern __shared__ uint64_t smem[];
  __shared__ WaveRows waves[kPairThreads / 64];
  int const T = op.off.count;
  TermsLds const l = stage_terms(op.off, smem);
  OrbitSearch<W, D, SI, KIND> search;
  search.stage(g, smem + 2 * static_cast<size_t>(T));
  int const wave = static_cast<int>(threadIdx.x) >> 6;
  int64_t const i0 = (static_cast<int64_t>(blockIdx.x) * (kPairThreads / 64) + wave) * rows;
  if (i0 >= op.n) return;
  int const count = static_cast<int>(min(static_cast<int64_t>(rows), op.n - i0));
  WaveRows &w = waves[wave];
  load_rows<projects_orbits(KIND)>(w, op, i0, count);
  for_each_pair(w, l, T, rows, count, [&](int r, int k, int, int64_t) {
    double const xr = CPLX ? x[2 * (i0 + r)] : x[i0 + r];
    double const xi = CPLX ? x[2 * (i0 + r) + 1] : 0.0;
    uint64_t beta;
    double c_re, c_im;
    off_diag_entry<W, D, SI, KIND>(g, op, l, k, w.alpha[r], w.norm[r], CPLX ? 1.0 : xr, beta, c_re, c_im, search);
    if (!(CPLX ? (c_re != 0 || c_im != 0) : (c_re != 0))) return;
    int64_t const j = target_index(op, beta);
    if (j < 0 || j >= op.n) {
      record_error(err, err_state, beta);
    } else if constexpr (CPLX) {
      unsafeAtomicAdd(&y[2 * j], c_re * xr - c_im * xi);
      unsafeAtomicAdd(&y[2 * j + 1], c_re * xi + c_im * xr);
    } else {
      unsafeAtomicAdd(&y[j], c_re);
    }
  });
}

// LDS of the fused kernels without their search tables.
inline size_t fused_lds_bytes(int T) { return terms_lds_bytes(T) + kPairLds; }

// Dispatch over (W, D, SI, KIND): permutation kernels follow the group,
// the others run on 64-bit words with the spin inversion as SI.
template <typename F> bool dispatch_op(OperatorCore const &op, F &&f) {
  if (op.off.count > kMaxPairTerms) return fail("too many off-diagonal terms: at most " + std::to_string(kMaxPairTerms));
  if (op.kind == kPermutations)
    return dispatch_search(*op.group, op.allow_factored, fused_lds_bytes(op.off.count), f);
  if (op.kind == kInversionOnly) {
    if (op.spin_inversion == 1) return f.template operator()<uint64_t, 0, 1, kInversionOnly>();
    return f.template operator()<uint64_t, 0, -1, kInversionOnly>();
  }
  return f.template operator()<uint64_t, 0, 0, kNoProjection>();
}

GroupView group_view_or_empty(OperatorCore const &op) {
  if (op.group != nullptr) return op.group->view();
  return GroupView{nullptr, nullptr, nullptr, nullptr, 0, 0, 0};
}

bool check_error(OperatorCore &op) {
  int err = 0;
  uint64_t state = 0;
  LSAMD_HIP(hipMemcpyAsync(&err, op.d_err.ptr, sizeof(int), hipMemcpyDeviceToHost, stream()));
  LSAMD_HIP(hipMemcpyAsync(&state, op.d_err_state.ptr, sizeof(uint64_t), hipMemcpyDeviceToHost, stream()));
  LSAMD_HIP(hipStreamSynchronize(stream()));
  if (err != 0) {
    LSAMD_HIP(hipMemsetAsync(op.d_err.ptr, 0, sizeof(int), stream()));
    // DistributedMatrixVector.chpl:133-135
    return fail("invalid index: -1 for state " + std::to_string(state) +
                " (the operator does not respect the basis symmetries)");
  }
  return true;
}

bool ensure_err(OperatorCore &op) {
  if (op.d_err.ptr == nullptr) {
    if (!op.d_err.allocate(1) || !op.d_err_state.allocate(1)) return false;
    LSAMD_HIP(hipMemsetAsync(op.d_err.ptr, 0, sizeof(int), stream()));
  }
  return true;
}

// state_info norm of every representative (n_alpha of BatchedOperator.chpl:244).
bool operator_prepare_norms(OperatorCore &op) {
  if (op.kind != kPermutations || op.d_norms != nullptr) return true;
  int64_t const n = op.number_states;
  DeviceArray<uint64_t> reps_out;
  DeviceArray<double> chars;
  if (!op.owned_norms.allocate(static_cast<size_t>(n > 0 ? n : 1))) return false;
  if (!reps_out.allocate(static_cast<size_t>(n > 0 ? n : 1))) return false;
  if (!chars.allocate(static_cast<size_t>(2 * (n > 0 ? n : 1)))) return false;
  if (!launch_state_info(*op.group, n, op.index.reps, 1, reps_out.ptr, 1, chars.ptr, op.owned_norms.ptr))
    return false;
  LSAMD_HIP(hipStreamSynchronize(stream()));
  op.d_norms = op.owned_norms.ptr;
  return true;
}

bool operator_matvec_otf(OperatorCore &op, double const *d_x, double *d_y, bool accumulate,
                         bool complex_values) {
  if (!ensure_err(op) || !operator_prepare_norms(op)) return false;
  int64_t const n = op.number_states;
  if (n == 0) return true;
  OpView const v = make_view(op);
  GroupView const g = group_view_or_empty(op);
  timer_begin(kTimerOtfF64);
  if (complex_values)
    otf_diag_kernel<true><<<grid_for(n, 256), 256, 0, stream()>>>(v, d_x, d_y, accumulate ? 1 : 0);
  else
    otf_diag_kernel<false><<<grid_for(n, 256), 256, 0, stream()>>>(v, d_x, d_y, accumulate ? 1 : 0);
  LSAMD_HIP(hipGetLastError());
  bool ok = op.off.count == 0 || dispatch_op(op, [&]<typename W, int D, int SI, int KIND>() -> bool {
    size_t const smem = terms_lds_bytes(op.off.count) + search_lds_bytes<W, D, SI, KIND>(op.group, kPairThreads);
    int const rows = wave_rows(n), grid = pair_grid(n, rows);
    if (complex_values)
      otf_push_kernel<W, D, SI, KIND, true><<<grid, kPairThreads, smem, stream()>>>(
          g, v, rows, d_x, d_y, op.d_err.ptr, op.d_err_state.ptr);
    else
      otf_push_kernel<W, D, SI, KIND, false><<<grid, kPairThreads, smem, stream()>>>(
          g, v, rows, d_x, d_y, op.d_err.ptr, op.d_err_state.ptr);
    LSAMD_HIP(hipGetLastError());
    return true;
  });
  timer_end(kTimerOtfF64);
  if (!ok) return false;
  return check_error(op);
}

// ---------------------------------------------------------------------------
// CSR cache
// ---------------------------------------------------------------------------

constexpr uint32_t kDropped = 0xffffffffu;

// What the fill kernel stores per pair.
enum FillOutput {
  kFillReal = 0,    // column, Re(C) as a double, at the pair's place in its source row
  kFillComplex = 1, // column, C as two doubles, likewise
  // Column and a tag, in the order in which the wave meets its rows' pairs:
  // kTagRow bits of row within the wave, kTagPlace bits of place in the
  // target row, and the slot of Re(C) in a hash table of values.
  kFillTable = 2
};
constexpr int kTagRowBits = 6, kTagPlaceBits = 12;

// Hash table of the distinct values (bit patterns) met by a kFillTable pass.
constexpr uint64_t kEmptySlot = ~uint64_t{0}; // a NaN pattern, never a stored value
constexpr int kValueSlots = 4 * kWideTableSize; // slots fit the 14 bits a tag has for them
constexpr int kMaxProbes = 128;

struct ValueHash {
  unsigned long long *slots; // [kValueSlots]
  int *distinct;             // values inserted
  int *overflow;             // kManyValues, kLongRow
};
// Why a kFillTable pass stops: more than kWideTableSize values, or a target row
// too long for a tag's place bits.
constexpr int kManyValues = 1, kLongRow = 2;

__device__ __forceinline__ uint32_t slot_hash(uint64_t k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  return static_cast<uint32_t>(k);
}

__device__ __forceinline__ uint64_t lane_value(uint64_t v, int lane) {
  return static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), lane))) << 32 |
         static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), lane));
}

// Slot of a value, inserted when new.  A plain load that finds the value or a
// stale empty slot is enough: the exchange decides.  When a pass starts every
// lane meets the same few new values at once, so the lanes of a wave that hold
// one value make one exchange (the first kGroups values; lanes with others one
// each): without, 16 to 20 sites without a group (one value) built in 0.64 to
// 1.19 ms instead of 0.41 to 0.52.
constexpr int kGroups = 4;

__device__ __forceinline__ uint32_t value_slot(ValueHash const &h, double v) {
  unsigned long long const key = static_cast<unsigned long long>(__double_as_longlong(v));
  uint32_t slot = slot_hash(key) & (kValueSlots - 1);
  int const lane = static_cast<int>(threadIdx.x) & 63;
  for (int probe = 0; probe < kMaxProbes; ++probe) {
    unsigned long long cur = h.slots[slot];
    if (cur == kEmptySlot) {
      int leader = lane;
      uint64_t pending = __ballot(true);
      for (int g = 0; g < kGroups && pending != 0; ++g) {
        int const l = __ffsll(static_cast<unsigned long long>(pending)) - 1;
        bool const same = key == lane_value(key, l) && slot == static_cast<uint32_t>(lane_value(slot, l));
        leader = same ? l : leader;
        pending &= ~__ballot(same);
      }
      if (leader == lane) {
        cur = atomicCAS(&h.slots[slot], static_cast<unsigned long long>(kEmptySlot), key);
        if (cur == kEmptySlot && atomicAdd(h.distinct, 1) >= kWideTableSize) atomicOr(h.overflow, kManyValues);
      }
      cur = __shfl(cur, leader, 64);
      if (cur == kEmptySlot) return slot;
    }
    if (cur == key) return slot;
    slot = (slot + 1) & (kValueSlots - 1);
  }
  atomicOr(h.overflow, kLongRow); // a crowded stretch of a table with room: the values may still be few
  return 0;
}

// The pairs of every source row with their targets.  kept[i] counts row i's
// entries (kFillReal, kFillComplex); kFillTable counts the entries of every
// target row into `targets` instead, and the count an entry finds there is its
// place in that row.
template <typename W, int D, int SI, int KIND, int OUT>
__global__ __launch_bounds__(kPairThreads) void csr_fill_kernel(GroupView g, OpView op, int rows,
                                                                int64_t const *__restrict__ row_ptr,
                                                                uint32_t *__restrict__ cols,
                                                                double *__restrict__ vals,
                                                                uint32_t *__restrict__ kept,
                                                                uint32_t *__restrict__ tags,
                                                                uint32_t *__restrict__ targets, ValueHash hash,
                                                                int *err, uint64_t *err_state) {
  extern __shared__ uint64_t smem[];
  __shared__ WaveRows waves[kPairThreads / 64];
  __shared__ uint32_t s_kept[OUT == kFillTable ? 1 : kPairThreads];
  if constexpr (OUT == kFillTable) {
    // The pass is repeated without the table.  Other workgroups raise the flag
    // at any time, so one thread reads it for all: the staging below needs
    // every thread of a workgroup that goes on.
    __shared__ int s_stop;
    if (threadIdx.x == 0) s_stop = *static_cast<int volatile *>(hash.overflow);
    __syncthreads();
    if (s_stop != 0) return;
  }
  int const T = op.off.count;
  TermsLds const l = stage_terms(op.off, smem);
  OrbitSearch<W, D, SI, KIND> search;
  search.stage(g, smem + 2 * static_cast<size_t>(T));
  int const wave = static_cast<int>(threadIdx.x) >> 6, lane = static_cast<int>(threadIdx.x) & 63;
  int64_t const i0 = (static_cast<int64_t>(blockIdx.x) * (kPairThreads / 64) + wave) * rows;
  if (i0 >= op.n) return;
  int const count = static_cast<int>(min(static_cast<int64_t>(rows), op.n - i0));
  WaveRows &w = waves[wave];
  uint32_t *const my_kept = s_kept + (OUT == kFillTable ? 0 : 64 * wave);
  load_rows<projects_orbits(KIND)>(w, op, i0, count);
  if constexpr (OUT != kFillTable) my_kept[lane] = 0;
  int64_t const base = row_ptr[i0];
  for_each_pair(w, l, T, rows, count, [&](int r, int k, int rank, int64_t at) {
    uint64_t beta;
    double c_re, c_im;
    off_diag_entry<W, D, SI, KIND>(g, op, l, k, w.alpha[r], w.norm[r], 1.0, beta, c_re, c_im, search);
    uint32_t col = kDropped;
    if (OUT == kFillComplex ? (c_re != 0 || c_im != 0) : (c_re != 0)) {
      int64_t const j = target_index(op, beta);
      if (j < 0 || j >= op.n) record_error(err, err_state, beta);
      else col = static_cast<uint32_t>(j);
    }
    if constexpr (OUT == kFillTable) {
      int64_t const o = base + at;
      cols[o] = col;
      if (col != kDropped) {
        uint32_t const place = atomicAdd(&targets[col], 1u);
        if (place >> kTagPlaceBits != 0) atomicOr(hash.overflow, kLongRow);
        tags[o] = (value_slot(hash, c_re) << kTagPlaceBits | (place & ((1u << kTagPlaceBits) - 1))) << kTagRowBits |
                  static_cast<uint32_t>(r);
      }
    } else {
      int64_t const o = row_ptr[i0 + r] + rank;
      bool const dropped = col == kDropped;
      cols[o] = col;
      if constexpr (OUT == kFillComplex) {
        vals[2 * o] = dropped ? 0.0 : c_re;
        vals[2 * o + 1] = dropped ? 0.0 : c_im;
      } else {
        vals[o] = dropped ? 0.0 : c_re;
      }
      if (!dropped) atomicAdd(&my_kept[r], 1u);
    }
  });
  __builtin_amdgcn_wave_barrier();
  if constexpr (OUT != kFillTable)
    if (lane < count) kept[i0 + lane] = my_kept[lane];
}

// diag[i] = sum of the diagonal terms' real parts, in term order.
__global__ __launch_bounds__(256) void csr_diag_kernel(OpView op, double *__restrict__ diag) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= op.n) return;
  uint64_t const alpha = op.idx.reps[i];
  double d = 0;
  for (int k = 0; k < op.diag.count; ++k) {
    if ((alpha & op.diag.m[k]) != op.diag.r[k]) continue;
    double const sign = (__popcll(alpha & op.diag.s[k]) & 1) ? -1.0 : 1.0;
    d += op.diag.v[2 * k] * sign;
  }
  diag[i] = d;
}

__global__ __launch_bounds__(256) void csr_compact_kernel(int64_t n, int64_t const *__restrict__ old_ptr,
                                                          uint32_t const *__restrict__ old_cols,
                                                          double const *__restrict__ old_vals,
                                                          uint64_t const *__restrict__ new_ptr,
                                                          uint32_t *__restrict__ cols,
                                                          double *__restrict__ vals, int width) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t o = new_ptr[i];
  for (int64_t k = old_ptr[i]; k < old_ptr[i + 1]; ++k) {
    if (old_cols[k] == kDropped) continue;
    cols[o] = old_cols[k];
    for (int q = 0; q < width; ++q) vals[o * width + q] = old_vals[k * width + q];
    ++o;
  }
}

// ---------------------------------------------------------------------------
// Source rows -> target rows.  Entry t of source row i (column j, value C)
// becomes an entry of row j with column i.  Keys i << 24 | t are scattered
// into the target rows through atomic cursors, each target row's keys are
// sorted, and the sorted keys give the final columns and values: row j then
// lists its sources in ascending i, whatever order the atomics took (within
// one i in ascending value; complex entries in term order).
// ---------------------------------------------------------------------------

constexpr int kKeyLocalBits = 24; // entries per source row < 2^24 (one per term at most)
constexpr int kSortCap = 1024;    // longest row sorted in LDS; longer rows are heap-sorted in place

// The count and scatter passes give kPushLanes lanes to a source row: lane l
// takes its entries b + l, b + l + kPushLanes, ..., so a wave reads the
// column stream coalesced and has a row's atomics in flight together.  Slot
// order within a target row follows the atomics, and the sort that comes
// next fixes it.
constexpr int kPushLanes = 16;

__global__ __launch_bounds__(256) void push_count_kernel(int64_t n, int64_t const *__restrict__ rp,
                                                         uint32_t const *__restrict__ cols,
                                                         uint32_t *__restrict__ counts) {
  int64_t const i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kPushLanes;
  int const l = static_cast<int>(threadIdx.x) % kPushLanes;
  if (i >= n) return;
  int64_t const e = rp[i + 1];
  for (int64_t p = rp[i] + l; p < e; p += kPushLanes) atomicAdd(&counts[cols[p]], 1u);
}

// Sort keys of the transpose: the source row in the high bits (the column of
// M, the order within a target row) and, below it, the entry's global
// position when every position fits 32 bits (wide keys), else its position
// within the source row (kKeyLocalBits).  Both sort a row the same way.
__global__ __launch_bounds__(256) void push_scatter_kernel(int64_t n, int64_t const *__restrict__ rp,
                                                           uint32_t const *__restrict__ cols,
                                                           int64_t const *__restrict__ target_ptr,
                                                           uint32_t *__restrict__ cursor,
                                                           uint64_t *__restrict__ keys, int wide_keys) {
  int64_t const i = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kPushLanes;
  int const l = static_cast<int>(threadIdx.x) % kPushLanes;
  if (i >= n) return;
  int64_t const b = rp[i], e = rp[i + 1];
  for (int64_t p = b + l; p < e; p += kPushLanes) {
    uint32_t const j = cols[p];
    uint32_t const slot = atomicAdd(&cursor[j], 1u);
    keys[target_ptr[j] + slot] = wide_keys ? (static_cast<uint64_t>(i) << 32) | static_cast<uint64_t>(p)
                                           : (static_cast<uint64_t>(i) << kKeyLocalBits) | static_cast<uint64_t>(p - b);
  }
}

template <typename Key, typename Less> __device__ void heap_sort(Key *a, int64_t n, Less const &less) {
  auto sift = [a, &less](int64_t root, int64_t end) {
    while (true) {
      int64_t child = 2 * root + 1;
      if (child >= end) return;
      if (child + 1 < end && less(a[child], a[child + 1])) ++child;
      if (!less(a[root], a[child])) return;
      Key const t = a[root];
      a[root] = a[child];
      a[child] = t;
      root = child;
    }
  };
  for (int64_t r = n / 2 - 1; r >= 0; --r) sift(r, n);
  for (int64_t end = n - 1; end > 0; --end) {
    Key const t = a[0];
    a[0] = a[end];
    a[end] = t;
    sift(0, end);
  }
}

// Largest entry of counts[0, n) into *out (which starts at zero).
__global__ __launch_bounds__(256) void max_count_kernel(uint32_t const *__restrict__ counts, int64_t n,
                                                        uint32_t *__restrict__ out) {
  uint32_t m = 0;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    m = max(m, counts[i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), off, 64)));
  if ((threadIdx.x & 63) == 0) atomicMax(out, m);
}

// One wave per row: bitonic sort of the row's keys in LDS (dynamic, `cap`
// keys: the longest row's power of two, at most kSortCap, so that more
// workgroups fit a CU), padded to a power of two with all-ones keys.  Longer
// rows are heap-sorted in place.  The row index is uniform over the
// workgroup, so every barrier is reached by all its threads.
//
// With `vals` (the entries' real values by global position; wide keys or
// `src_ptr` give it), entries of one column are put in ascending value: the
// order in which the value-table build lists them.
__device__ __forceinline__ double key_value(uint64_t key, int64_t const *src_ptr, double const *vals) {
  if (src_ptr == nullptr) return vals[key & 0xffffffffull];
  return vals[src_ptr[key >> kKeyLocalBits] + static_cast<int64_t>(key & ((uint64_t{1} << kKeyLocalBits) - 1))];
}

// One lane orders a run: by insertion while that is short (a run is as many
// terms as take one state to the same other one; a 1-state basis with 2000 of
// them took 160 ms so, 64-entry runs about as long either way).
constexpr int kInsertionRun = 64;

__device__ __forceinline__ void order_ties(uint64_t *a, int64_t len, int64_t const *src_ptr, double const *vals) {
  int const shift = src_ptr == nullptr ? 32 : kKeyLocalBits;
  for (int64_t q = threadIdx.x; q + 1 < len; q += 64) {
    uint64_t const i = a[q] >> shift;
    if ((q > 0 && (a[q - 1] >> shift) == i) || (a[q + 1] >> shift) != i) continue; // not the start of a run
    int64_t end = q + 2;
    while (end < len && (a[end] >> shift) == i) ++end;
    if (end - q > kInsertionRun) {
      heap_sort(a + q, end - q,
                [&](uint64_t x, uint64_t y) { return key_value(x, src_ptr, vals) < key_value(y, src_ptr, vals); });
      continue;
    }
    for (int64_t t = q + 1; t < end; ++t) {
      uint64_t const key = a[t];
      double const v = key_value(key, src_ptr, vals);
      int64_t u = t;
      while (u > q && key_value(a[u - 1], src_ptr, vals) > v) {
        a[u] = a[u - 1];
        --u;
      }
      a[u] = key;
    }
  }
}

// 32-bit keys are those of the packed value table (column << 8 | value index):
// they are stored as its words, column | value index << 24.
__device__ __forceinline__ uint64_t stored_key(uint64_t key) { return key; }
__device__ __forceinline__ uint32_t stored_key(uint32_t key) { return key >> 8 | key << 24; }

// Rows of more than min_len entries.
template <typename Key>
__global__ __launch_bounds__(64) void sort_rows_kernel(int64_t n, int64_t const *__restrict__ rp,
                                                       Key *__restrict__ keys, int cap, int min_len,
                                                       int64_t const *__restrict__ src_ptr,
                                                       double const *__restrict__ vals) {
  extern __shared__ uint64_t sort_lds[];
  Key *const s = reinterpret_cast<Key *>(sort_lds);
  for (int64_t row = blockIdx.x; row < n; row += gridDim.x) {
    int64_t const b = rp[row];
    int64_t const len = rp[row + 1] - b;
    if (len <= min_len) continue;
    if (len > cap) {
      if (threadIdx.x == 0) heap_sort(keys + b, len, [](Key x, Key y) { return x < y; });
      __syncthreads();
      if constexpr (sizeof(Key) == 8) {
        if (vals != nullptr) order_ties(keys + b, len, src_ptr, vals);
      } else {
        for (int64_t q = threadIdx.x; q < len; q += 64) keys[b + q] = stored_key(keys[b + q]);
      }
      __syncthreads();
      continue;
    }
    int P = 2;
    while (P < len) P <<= 1;
    for (int q = threadIdx.x; q < P; q += 64) s[q] = q < len ? keys[b + q] : static_cast<Key>(~Key{0});
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int q = threadIdx.x; q < P / 2; q += 64) {
          int const lo = 2 * stride * (q / stride) + (q % stride);
          int const hi = lo + stride;
          bool const ascending = (lo & size) == 0;
          Key const a = s[lo], c = s[hi];
          if ((a > c) == ascending) {
            s[lo] = c;
            s[hi] = a;
          }
        }
        __syncthreads();
      }
    }
    if constexpr (sizeof(Key) == 8) {
      if (vals != nullptr) {
        order_ties(s, len, src_ptr, vals);
        __syncthreads();
      }
    }
    for (int q = threadIdx.x; q < len; q += 64) keys[b + q] = stored_key(s[q]);
    __syncthreads();
  }
}

// Rows of at most kShortRow entries, one wave per row, in registers: entry
// 64 e + lane of the padded row in v[e], a bitonic network over swizzles for
// distances below 64 and within the lane above; which lanes keep the smaller
// key is a constant of the step.  VALU-bound: 6.0 ms for the 15.8 M rows of
// 6x6 (74 entries each), against 24 ms with 64-bit keys in LDS (barriers and
// LDS round trips in every step).
constexpr int kShortRow = 256;

// The value of lane ^ kMask: a swizzle within 32 lanes needs no addresses.
template <int kMask> __device__ __forceinline__ uint32_t exchange(uint32_t v) {
  if constexpr (kMask < 32)
    return static_cast<uint32_t>(__builtin_amdgcn_ds_swizzle(static_cast<int>(v), 0x1f | kMask << 10));
  else
    return __shfl_xor(v, kMask, 64);
}
template <int kMask> __device__ __forceinline__ uint64_t exchange(uint64_t v) {
  return static_cast<uint64_t>(exchange<kMask>(static_cast<uint32_t>(v >> 32))) << 32 |
         exchange<kMask>(static_cast<uint32_t>(v));
}

// Lanes that keep the smaller key in a step: bit l set when lane l is the
// lower of its pair and the run of `size` entries is ascending, or neither.
// `first` is the entry of lane 0.
constexpr uint64_t keep_smaller(int first, int size, int stride) {
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l)
    if (((l & stride) == 0) == (((first + l) & size) == 0)) m |= uint64_t{1} << l;
  return m;
}

template <int E, int kSize, int kStride, typename Key> __device__ __forceinline__ void sort_step(Key (&v)[E]) {
  if constexpr (kStride >= 64) {
    constexpr int d = kStride / 64;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if ((e & d) == 0) {
        bool const ascending = ((64 * e) & kSize) == 0;
        Key const a = v[e], c = v[e + d], lo = a < c ? a : c, hi = a < c ? c : a;
        v[e] = ascending ? lo : hi;
        v[e + d] = ascending ? hi : lo;
      }
  } else {
    auto pair = [&]<int e>() {
      constexpr uint64_t keep = keep_smaller(64 * e, kSize, kStride);
      Key const other = exchange<kStride>(v[e]);
      Key const lo = other < v[e] ? other : v[e], hi = other < v[e] ? v[e] : other;
      v[e] = __builtin_amdgcn_inverse_ballot_w64(keep) ? lo : hi;
    };
    pair.template operator()<0>();
    if constexpr (E > 1) pair.template operator()<1>();
    if constexpr (E > 2) {
      pair.template operator()<2>();
      pair.template operator()<3>();
    }
  }
}

template <int E, int kSize, int kStride, typename Key> __device__ __forceinline__ void sort_steps(Key (&v)[E]) {
  sort_step<E, kSize, kStride>(v);
  if constexpr (kStride > 1) sort_steps<E, kSize, kStride / 2>(v);
  else if constexpr (kSize < 64 * E) sort_steps<E, 2 * kSize, kSize>(v);
}

template <int E, typename Key> __device__ __forceinline__ void sort_row_registers(Key *__restrict__ row, int len) {
  int const lane = static_cast<int>(threadIdx.x) & 63;
  Key v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = 64 * e + lane < len ? row[64 * e + lane] : static_cast<Key>(~Key{0});
  sort_steps<E, 2, 1>(v);
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (64 * e + lane < len) row[64 * e + lane] = stored_key(v[e]);
}

template <typename Key>
__global__ __launch_bounds__(256) void sort_short_rows_kernel(int64_t n, int64_t const *__restrict__ rp,
                                                              Key *__restrict__ keys) {
  int64_t const row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= n) return;
  int64_t const b = rp[row];
  int64_t const length = rp[row + 1] - b;
  if (length == 0 || length > kShortRow) return;
  int const len = static_cast<int>(length);
  if (len <= 64) sort_row_registers<1>(keys + b, len);
  else if (len <= 128) sort_row_registers<2>(keys + b, len);
  else sort_row_registers<4>(keys + b, len);
}

// Sorts every row of `keys` (and turns 32-bit keys into table words).
template <typename Key>
bool sort_table_rows(int64_t n, int64_t const *rp, Key *keys, uint32_t max_len) {
  sort_short_rows_kernel<Key><<<grid_for(n, 4), 256, 0, stream()>>>(n, rp, keys);
  LSAMD_HIP(hipGetLastError());
  if (max_len > kShortRow) {
    int const cap = max_len > 512 ? kSortCap : 512;
    sort_rows_kernel<Key><<<static_cast<int>(std::min<int64_t>(n, 1 << 16)), 64, sizeof(Key) * cap, stream()>>>(
        n, rp, keys, cap, kShortRow, nullptr, nullptr);
    LSAMD_HIP(hipGetLastError());
  }
  return true;
}

__global__ __launch_bounds__(256) void push_finalize_kernel(int64_t nnz, uint64_t const *__restrict__ keys,
                                                            int64_t const *__restrict__ src_ptr,
                                                            double const *__restrict__ src_vals, int width,
                                                            uint32_t *__restrict__ cols,
                                                            double *__restrict__ vals, int wide_keys) {
  int64_t const q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= nnz) return;
  uint64_t const key = keys[q];
  int64_t i, p;
  if (wide_keys) {
    i = static_cast<int64_t>(key >> 32);
    p = static_cast<int64_t>(key & 0xffffffffull);
  } else {
    i = static_cast<int64_t>(key >> kKeyLocalBits);
    p = src_ptr[i] + static_cast<int64_t>(key & ((uint64_t{1} << kKeyLocalBits) - 1));
  }
  cols[q] = static_cast<uint32_t>(i);
  for (int w = 0; w < width; ++w) vals[q * width + w] = src_vals[p * width + w];
}

// The largest of n row lengths.
bool longest_row(uint32_t const *counts, int64_t n, uint32_t &max_len) {
  DeviceArray<uint32_t> longest;
  if (!longest.allocate(1)) return false;
  LSAMD_HIP(hipMemsetAsync(longest.ptr, 0, sizeof(uint32_t), stream()));
  max_count_kernel<<<static_cast<int>(std::min<int64_t>(grid_for(n, 256), 1024)), 256, 0, stream()>>>(counts, n,
                                                                                                  longest.ptr);
  LSAMD_HIP(hipGetLastError());
  LSAMD_HIP(hipMemcpyAsync(&max_len, longest.ptr, sizeof(uint32_t), hipMemcpyDeviceToHost, stream()));
  LSAMD_HIP(hipStreamSynchronize(stream()));
  return true;
}

// Replaces the source-row CSR (row_ptr, cols, vals of `width` doubles per
// entry, nnz entries over n rows) by its target-row form.
bool transpose_to_targets(int64_t n, int64_t nnz, int width, DeviceArray<int64_t> &row_ptr,
                          DeviceArray<uint32_t> &cols, DeviceArray<double> &vals) {
  if (n == 0 || nnz == 0) return true;
  DeviceArray<uint32_t> counts;
  DeviceArray<int64_t> target_ptr;
  DeviceArray<uint64_t> keys;
  if (!counts.allocate(static_cast<size_t>(n)) || !target_ptr.allocate(static_cast<size_t>(n + 1)) ||
      !keys.allocate(static_cast<size_t>(nnz)))
    return false;
  LSAMD_HIP(hipMemsetAsync(counts.ptr, 0, sizeof(uint32_t) * n, stream()));
  push_count_kernel<<<grid_for(n * kPushLanes, 256), 256, 0, stream()>>>(n, row_ptr.ptr, cols.ptr, counts.ptr);
  LSAMD_HIP(hipGetLastError());
  // the longest target row sizes the sort's LDS
  uint32_t max_len = 0;
  if (!longest_row(counts.ptr, n, max_len)) return false;
  int sort_cap = 2;
  while (sort_cap < kSortCap && sort_cap < static_cast<int>(std::min<uint32_t>(max_len, kSortCap))) sort_cap <<= 1;
  uint64_t total = 0;
  if (!exclusive_scan(counts.ptr, n, reinterpret_cast<uint64_t *>(target_ptr.ptr), total)) return false;
  if (static_cast<int64_t>(total) != nnz) return fail("CSR transpose: entry count mismatch");
  int64_t const last = nnz;
  LSAMD_HIP(hipMemcpyAsync(target_ptr.ptr + n, &last, sizeof(int64_t), hipMemcpyHostToDevice, stream()));
  LSAMD_HIP(hipMemsetAsync(counts.ptr, 0, sizeof(uint32_t) * n, stream()));
  int const wide_keys = nnz <= int64_t{0xffffffff} ? 1 : 0;
  push_scatter_kernel<<<grid_for(n * kPushLanes, 256), 256, 0, stream()>>>(n, row_ptr.ptr, cols.ptr,
                                                                           target_ptr.ptr, counts.ptr, keys.ptr,
                                                                           wide_keys);
  LSAMD_HIP(hipGetLastError());
  int const sort_grid = static_cast<int>(std::min<int64_t>(n, 1 << 16));
  sort_rows_kernel<uint64_t><<<sort_grid, 64, sizeof(uint64_t) * sort_cap, stream()>>>(
      n, target_ptr.ptr, keys.ptr, sort_cap, 1, wide_keys ? nullptr : row_ptr.ptr, width == 1 ? vals.ptr : nullptr);
  LSAMD_HIP(hipGetLastError());
  LSAMD_HIP(hipStreamSynchronize(stream()));
  counts.reset();
  cols.reset();
  DeviceArray<uint32_t> cols2;
  DeviceArray<double> vals2;
  if (!cols2.allocate(static_cast<size_t>(nnz)) || !vals2.allocate(static_cast<size_t>(nnz) * width)) return false;
  push_finalize_kernel<<<grid_for(nnz, 256), 256, 0, stream()>>>(nnz, keys.ptr, row_ptr.ptr, vals.ptr, width,
                                                                 cols2.ptr, vals2.ptr, wide_keys);
  LSAMD_HIP(hipGetLastError());
  LSAMD_HIP(hipStreamSynchronize(stream()));
  row_ptr = std::move(target_ptr);
  cols = std::move(cols2);
  vals = std::move(vals2);
  return true;
}

__global__ __launch_bounds__(256) void to_f32_kernel(int64_t n, double const *__restrict__ in,
                                                     float *__restrict__ out) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = static_cast<float>(in[i]);
}

// ---------------------------------------------------------------------------
// Value table: distinct off-diagonal values (bit patterns) through a per-block
// LDS hash merged into a global hash, then column | index << 24 packing.
// ---------------------------------------------------------------------------

constexpr int kLocalSlots = 2 * kWideTableSize; // per-block LDS hash (64 KB)

__global__ __launch_bounds__(256) void distinct_values_kernel(double const *__restrict__ vals, int64_t nnz,
                                                              unsigned long long *__restrict__ table,
                                                              int *__restrict__ overflow) {
  __shared__ unsigned long long local[kLocalSlots];
  __shared__ int local_overflow;
  for (int i = threadIdx.x; i < kLocalSlots; i += blockDim.x) local[i] = kEmptySlot;
  if (threadIdx.x == 0) local_overflow = 0;
  __syncthreads();
  for (int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; k < nnz;
       k += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    unsigned long long const key = static_cast<unsigned long long>(__double_as_longlong(vals[k]));
    uint32_t slot = slot_hash(key) & (kLocalSlots - 1);
    int probes = 0;
    while (true) {
      unsigned long long const prev = atomicCAS(&local[slot], static_cast<unsigned long long>(kEmptySlot), key);
      if (prev == kEmptySlot || prev == key) break;
      slot = (slot + 1) & (kLocalSlots - 1);
      if (++probes >= kLocalSlots) {
        local_overflow = 1;
        break;
      }
    }
    if (local_overflow) break;
  }
  __syncthreads();
  if (local_overflow) {
    if (threadIdx.x == 0) atomicExch(overflow, 1);
    return;
  }
  for (int i = threadIdx.x; i < kLocalSlots; i += blockDim.x) {
    unsigned long long const key = local[i];
    if (key == kEmptySlot) continue;
    uint32_t slot = slot_hash(key) & (kValueSlots - 1);
    int probes = 0;
    while (true) {
      unsigned long long const prev = atomicCAS(&table[slot], static_cast<unsigned long long>(kEmptySlot), key);
      if (prev == kEmptySlot || prev == key) break;
      slot = (slot + 1) & (kValueSlots - 1);
      if (++probes >= kValueSlots) {
        atomicExch(overflow, 1);
        break;
      }
    }
  }
}

// cols[k] |= index of vals[k] in the sorted table << 24
__global__ __launch_bounds__(256) void pack_columns_kernel(double const *__restrict__ vals, int64_t nnz,
                                                           double const *__restrict__ table, int size,
                                                           uint32_t *__restrict__ cols) {
  __shared__ double t[kValueTableSize];
  for (int i = threadIdx.x; i < size; i += blockDim.x) t[i] = table[i];
  __syncthreads();
  int64_t const k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  double const v = vals[k];
  int lo = 0, hi = size - 1;
  while (lo < hi) {
    int const mid = (lo + hi) >> 1;
    if (t[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  cols[k] = (cols[k] & kPackedColumnMask) | (static_cast<uint32_t>(lo) << 24);
}

// vidx[k] = index of vals[k] in the sorted table (wide value table)
__global__ __launch_bounds__(256) void pack_wide_kernel(double const *__restrict__ vals, int64_t nnz,
                                                        double const *__restrict__ table, int size,
                                                        uint16_t *__restrict__ vidx) {
  __shared__ double t[kWideTableSize];
  for (int i = threadIdx.x; i < size; i += blockDim.x) t[i] = table[i];
  __syncthreads();
  int64_t const k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  double const v = vals[k];
  int lo = 0, hi = size - 1;
  while (lo < hi) {
    int const mid = (lo + hi) >> 1;
    if (t[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  vidx[k] = static_cast<uint16_t>(lo);
}

// For matrices that build_table_csr leaves to the general build although
// their values are few (a target row of more than 4096 entries).
// Replaces the value arrays of a real CSR by a value table: packed into the
// column words when it has at most 256 distinct values and fewer than 2^24
// rows, else a wide table with 16-bit indices when it has at most
// kWideTableSize.  vals is the FP64 value array (kept by the caller until
// this returns).
bool try_pack_values(Csr &c, double const *vals) {
  if (c.nnz == 0) return true;
  DeviceArray<unsigned long long> table;
  DeviceArray<int> overflow;
  if (!table.allocate(kValueSlots) || !overflow.allocate(1)) return false;
  LSAMD_HIP(hipMemsetAsync(table.ptr, 0xFF, sizeof(unsigned long long) * kValueSlots, stream()));
  LSAMD_HIP(hipMemsetAsync(overflow.ptr, 0, sizeof(int), stream()));
  distinct_values_kernel<<<2048, 256, 0, stream()>>>(vals, c.nnz, table.ptr, overflow.ptr);
  LSAMD_HIP(hipGetLastError());
  std::vector<unsigned long long> h(kValueSlots);
  int ovf = 0;
  LSAMD_HIP(hipMemcpyAsync(h.data(), table.ptr, sizeof(unsigned long long) * kValueSlots, hipMemcpyDeviceToHost,
                           stream()));
  LSAMD_HIP(hipMemcpyAsync(&ovf, overflow.ptr, sizeof(int), hipMemcpyDeviceToHost, stream()));
  LSAMD_HIP(hipStreamSynchronize(stream()));
  if (ovf) return true;
  std::vector<double> values;
  for (unsigned long long k : h)
    if (k != kEmptySlot) {
      double v;
      std::memcpy(&v, &k, sizeof(v));
      values.push_back(v);
    }
  bool const fits_word = values.size() <= static_cast<size_t>(kValueTableSize) && c.rows < (int64_t{1} << 24);
  if (values.empty() || (!fits_word && values.size() > static_cast<size_t>(kWideTableSize))) return true;
  std::sort(values.begin(), values.end());
  std::vector<float> values32(values.size());
  for (size_t i = 0; i < values.size(); ++i) values32[i] = static_cast<float>(values[i]);
  if (!c.table64.upload(values.data(), values.size()) || !c.table32.upload(values32.data(), values32.size()))
    return false;
  int const size = static_cast<int>(values.size());
  if (fits_word) {
    pack_columns_kernel<<<grid_for(c.nnz, 256), 256, 0, stream()>>>(vals, c.nnz, c.table64.ptr, size, c.cols.ptr);
  } else {
    if (!c.vidx.allocate(static_cast<size_t>(c.nnz))) return false;
    pack_wide_kernel<<<grid_for(c.nnz, 256), 256, 0, stream()>>>(vals, c.nnz, c.table64.ptr, size, c.vidx.ptr);
  }
  LSAMD_HIP(hipGetLastError());
  LSAMD_HIP(hipStreamSynchronize(stream()));
  c.packed = fits_word;
  c.wide = !fits_word;
  c.table_size = size;
  return true;
}

// Launches the fill pass (FillOutput).
struct FillTargets {
  uint32_t *cols = nullptr;
  double *vals = nullptr;
  uint32_t *kept = nullptr, *tags = nullptr, *targets = nullptr;
  ValueHash hash{nullptr, nullptr, nullptr};
};

template <int OUT> bool launch_fill(OperatorCore &op, int64_t const *row_ptr, FillTargets const &t) {
  int64_t const n = op.number_states;
  OpView const v = make_view(op);
  GroupView const g = group_view_or_empty(op);
  return dispatch_op(op, [&]<typename W, int D, int SI, int KIND>() -> bool {
    size_t const smem = terms_lds_bytes(op.off.count) + search_lds_bytes<W, D, SI, KIND>(op.group, kPairThreads);
    int const rows = wave_rows(n);
    csr_fill_kernel<W, D, SI, KIND, OUT><<<pair_grid(n, rows), kPairThreads, smem, stream()>>>(
        g, v, rows, row_ptr, t.cols, t.vals, t.kept, t.tags, t.targets, t.hash,
        op.d_err.ptr, op.d_err_state.ptr);
    LSAMD_HIP(hipGetLastError());
    return true;
  });
}

// Entries of a kFillTable pass into their target rows, one workgroup to the
// rows of one of its waves.  An entry's place within the row came from the
// fill pass, so no atomics are needed.  Key: the source row over the rank of
// the entry's value in the sorted table.
template <typename Key, int kRankBits, typename Ptr>
__global__ __launch_bounds__(256) void table_scatter_kernel(int64_t n, int rows, int64_t const *__restrict__ rp,
                                                            uint32_t const *__restrict__ cols,
                                                            uint32_t const *__restrict__ tags,
                                                            uint16_t const *__restrict__ rank,
                                                            Ptr const *__restrict__ target_ptr,
                                                            Key *__restrict__ keys) {
  int64_t const i0 = static_cast<int64_t>(blockIdx.x) * rows;
  int64_t const e = rp[min(i0 + rows, n)];
  for (int64_t p = rp[i0] + threadIdx.x; p < e; p += 256) {
    uint32_t const j = cols[p];
    if (j == kDropped) continue;
    uint32_t const tag = tags[p];
    uint32_t const place = tag >> kTagRowBits & ((1u << kTagPlaceBits) - 1);
    keys[target_ptr[j] + place] = static_cast<Key>(i0 + (tag & ((1u << kTagRowBits) - 1))) << kRankBits |
                                  rank[tag >> (kTagRowBits + kTagPlaceBits)];
  }
}

__global__ __launch_bounds__(256) void narrow_kernel(int64_t n, int64_t const *__restrict__ in,
                                                     uint32_t *__restrict__ out) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = static_cast<uint32_t>(in[i]);
}

template <typename Key, int kRankBits>
bool scatter_to_targets(int64_t n, int64_t const *rp, uint32_t const *cols, uint32_t const *tags,
                        uint16_t const *rank, int64_t const *target_ptr, int64_t nnz, DeviceArray<uint32_t> &targets,
                        Key *keys) {
  int const rows = wave_rows(n), grid = grid_for(n, rows);
  if (nnz <= int64_t{0xffffffff}) { // 4-byte row starts: half the gathered bytes; `targets` is free by now
    narrow_kernel<<<grid_for(n, 256), 256, 0, stream()>>>(n, target_ptr, targets.ptr);
    table_scatter_kernel<Key, kRankBits><<<grid, 256, 0, stream()>>>(n, rows, rp, cols, tags, rank,
                                                                     static_cast<uint32_t const *>(targets.ptr), keys);
  } else {
    table_scatter_kernel<Key, kRankBits><<<grid, 256, 0, stream()>>>(n, rows, rp, cols, tags, rank, target_ptr, keys);
  }
  LSAMD_HIP(hipGetLastError());
  return true;
}

__global__ __launch_bounds__(256) void split_wide_keys_kernel(int64_t nnz, uint64_t const *__restrict__ keys,
                                                              uint32_t *__restrict__ cols, uint16_t *__restrict__ vidx) {
  int64_t const q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= nnz) return;
  uint64_t const key = keys[q];
  cols[q] = static_cast<uint32_t>(key >> 16);
  vidx[q] = static_cast<uint16_t>(key);
}

// Real CSR with a value table, straight from the fill pass.  The pass records
// for every pair its target row, its place in that row and its value's slot in
// a hash table, so the values themselves are never stored per entry, the
// target rows need no counting pass of their own, and the scatter writes the
// final words (or 48-bit keys of the wide table) with no atomics.
// On 6x6 (1.17 G entries) a scatter of 25 ms, bound by its random 4-byte
// writes, and a sort of 6 ms replace a counting pass (28 ms), a scatter of
// 8-byte keys through atomic cursors (42 ms), their LDS sort (24 ms), a gather
// of the values in target order (23 ms), the distinct-value pass and the
// packing (9 ms), and the temporaries shrink from 28 to 14 GB.  `done` stays
// false when the matrix has too many values (`many`), a target row of more than
// 4096 entries, or no entries: then the general build runs.
bool build_table_csr(OperatorCore &op, int64_t up, int64_t const *row_ptr, bool &done, bool &many) {
  done = many = false;
  int64_t const n = op.number_states;
  Csr &c = op.csr;
  DeviceArray<uint32_t> cols, tags, targets;
  DeviceArray<unsigned long long> slots;
  DeviceArray<int> flags; // distinct values, overflow
  DeviceArray<int64_t> target_ptr;
  if (!cols.allocate(static_cast<size_t>(up)) || !tags.allocate(static_cast<size_t>(up)) ||
      !targets.allocate(static_cast<size_t>(n)) || !slots.allocate(kValueSlots) || !flags.allocate(2) ||
      !target_ptr.allocate(static_cast<size_t>(n + 1)))
    return false;
  LSAMD_HIP(hipMemsetAsync(targets.ptr, 0, sizeof(uint32_t) * n, stream()));
  LSAMD_HIP(hipMemsetAsync(slots.ptr, 0xFF, sizeof(unsigned long long) * kValueSlots, stream()));
  LSAMD_HIP(hipMemsetAsync(flags.ptr, 0, 2 * sizeof(int), stream()));
  FillTargets t;
  t.cols = cols.ptr;
  t.tags = tags.ptr;
  t.targets = targets.ptr;
  t.hash = ValueHash{slots.ptr, flags.ptr, flags.ptr + 1};
  if (!launch_fill<kFillTable>(op, row_ptr, t)) return false;
  std::vector<unsigned long long> h(kValueSlots);
  int h_flags[2] = {0, 0};
  LSAMD_HIP(hipMemcpyAsync(h.data(), slots.ptr, sizeof(unsigned long long) * kValueSlots, hipMemcpyDeviceToHost,
                           stream()));
  LSAMD_HIP(hipMemcpyAsync(h_flags, flags.ptr, sizeof(h_flags), hipMemcpyDeviceToHost, stream()));
  // Waits for the copies.  A pass that stopped early reports what it met, too:
  // the general build would find the same.
  if (!check_error(op)) return false;
  many = (h_flags[1] & kManyValues) != 0;
  if (h_flags[1] != 0 || h_flags[0] == 0) return true;
  std::vector<std::pair<double, int>> values;
  for (int q = 0; q < kValueSlots; ++q)
    if (h[q] != kEmptySlot) {
      double v;
      std::memcpy(&v, &h[q], sizeof(v));
      values.emplace_back(v, q);
    }
  std::sort(values.begin(), values.end());
  std::vector<uint16_t> rank(kValueSlots, 0);
  std::vector<double> table64(values.size());
  std::vector<float> table32(values.size());
  for (size_t r = 0; r < values.size(); ++r) {
    rank[values[r].second] = static_cast<uint16_t>(r);
    table64[r] = values[r].first;
    table32[r] = static_cast<float>(values[r].first);
  }
  DeviceArray<uint16_t> d_rank;
  uint64_t total = 0;
  uint32_t max_len = 0;
  if (!d_rank.upload(rank.data(), rank.size()) || !c.table64.upload(table64.data(), table64.size()) ||
      !c.table32.upload(table32.data(), table32.size()) || !longest_row(targets.ptr, n, max_len) ||
      !exclusive_scan(targets.ptr, n, reinterpret_cast<uint64_t *>(target_ptr.ptr), total))
    return false;
  int64_t const nnz = static_cast<int64_t>(total);
  LSAMD_HIP(hipMemcpyAsync(target_ptr.ptr + n, &nnz, sizeof(int64_t), hipMemcpyHostToDevice, stream()));
  bool const fits_word = values.size() <= static_cast<size_t>(kValueTableSize) && n < (int64_t{1} << 24);
  if (fits_word) {
    DeviceArray<uint32_t> words;
    if (!words.allocate(static_cast<size_t>(nnz))) return false;
    if (!scatter_to_targets<uint32_t, 8>(n, row_ptr, cols.ptr, tags.ptr, d_rank.ptr, target_ptr.ptr, nnz, targets,
                                         words.ptr))
      return false;
    if (!sort_table_rows(n, target_ptr.ptr, words.ptr, max_len)) return false;
    c.cols = std::move(words);
  } else {
    DeviceArray<uint64_t> keys;
    if (!keys.allocate(static_cast<size_t>(nnz))) return false;
    if (!scatter_to_targets<uint64_t, 16>(n, row_ptr, cols.ptr, tags.ptr, d_rank.ptr, target_ptr.ptr, nnz, targets,
                                          keys.ptr))
      return false;
    if (!sort_table_rows(n, target_ptr.ptr, keys.ptr, max_len)) return false;
    LSAMD_HIP(hipStreamSynchronize(stream()));
    if (!c.vidx.allocate(static_cast<size_t>(nnz))) return false;
    if (cols.count < static_cast<size_t>(nnz)) return fail("CSR build: entry count mismatch");
    split_wide_keys_kernel<<<grid_for(nnz, 256), 256, 0, stream()>>>(nnz, keys.ptr, cols.ptr, c.vidx.ptr);
    LSAMD_HIP(hipGetLastError());
    c.cols = std::move(cols);
  }
  LSAMD_HIP(hipStreamSynchronize(stream()));
  c.row_ptr = std::move(target_ptr);
  c.nnz = nnz;
  c.packed = fits_word;
  c.wide = !fits_word;
  c.table_size = static_cast<int>(values.size());
  done = true;
  return true;
}

// The product schedule when neither the caller nor the autotuner chose one:
// lanes per row so that each lane sums about four entries of a mean row, and
// for a million rows or more the die-aware mapping with one workgroup per
// tile, the autotuner's choice on 6x6 (16 lanes and that mapping).  Plain against
// die-aware grid, ms: FP32 block of 8 at 0.36 M rows 0.062 / 0.062, 0.72 M
// 0.123 / 0.112, 0.89 M (59 entries a row) 0.376 / 0.342, 1.3 M 0.244 / 0.223,
// 4.7 M 0.893 / 0.870, 15.8 M (6x6) 10.2 / 9.2.  The FP64 vector gains only where
// x outgrows the caches: 1.3 M 0.114 / 0.129, 4.4 M 1.59 / 1.67.
void default_schedule(OperatorCore &op) {
  Csr const &c = op.csr;
  double const mean = c.rows > 0 ? static_cast<double>(c.nnz) / static_cast<double>(c.rows) : 0.0;
  int lanes = 2;
  while (lanes < 64 && 8.0 * lanes <= mean) lanes *= 2;
  op.lanes_f64 = lanes;
  op.flags_f64 = c.rows >= (int64_t{1} << 20) ? 6 : 0;
  op.lanes_f32 = lanes;
  op.flags_f32 = op.flags_f64;
}

// Values and diagonal of a real CSR in the precisions asked for; `vals` holds
// its values when it has no table.
bool finish_real_csr(OperatorCore &op, int precision, DeviceArray<double> &vals) {
  Csr &c = op.csr;
  int64_t const n = c.rows;
  if (precision == 32 || precision == 96) {
    if (!c.diag32.allocate(static_cast<size_t>(n > 0 ? n : 1))) return false;
    if (!c.has_table()) {
      if (!c.vals32.allocate(static_cast<size_t>(c.nnz > 0 ? c.nnz : 1))) return false;
      if (c.nnz > 0) to_f32_kernel<<<grid_for(c.nnz, 256), 256, 0, stream()>>>(c.nnz, vals.ptr, c.vals32.ptr);
    }
    if (n > 0) to_f32_kernel<<<grid_for(n, 256), 256, 0, stream()>>>(n, c.diag64.ptr, c.diag32.ptr);
    LSAMD_HIP(hipGetLastError());
    c.has32 = true;
  }
  if (precision == 64 || precision == 96) {
    if (!c.has_table()) c.vals64 = std::move(vals);
    c.has64 = true;
  } else {
    c.diag64.reset();
  }
  if (!op.schedule_set) default_schedule(op);
  LSAMD_HIP(hipStreamSynchronize(stream()));
  return true;
}

bool operator_build_csr(OperatorCore &op, int precision) {
  if (precision != 32 && precision != 64 && precision != 96 && precision != 128)
    return fail("precision must be 32, 64, 96 (real) or 128 (complex)");
  bool const cplx = precision == 128;
  int const width = cplx ? 2 : 1;
  if (op.number_states >= (int64_t{1} << 32) - 1) return fail("CSR columns are 32-bit: too many states");
  if (op.off.count >= (1 << kKeyLocalBits)) return fail("CSR build: too many off-diagonal terms");
  if (!ensure_err(op) || !operator_prepare_norms(op)) return false;
  int64_t const n = op.number_states;
  Csr &c = op.csr;
  c = Csr{};
  c.rows = n;
  DeviceArray<uint32_t> counts;
  DeviceArray<int64_t> row_ptr;
  if (!counts.allocate(static_cast<size_t>(n > 0 ? n : 1))) return false;
  if (!row_ptr.allocate(static_cast<size_t>(n + 1))) return false;
  if (!c.diag64.allocate(static_cast<size_t>(n > 0 ? n : 1))) return false;
  uint64_t upper = 0;
  if (n > 0) {
    if (op.off.count > 0) {
      count_applicable_kernel<<<grid_for(n, 256), 256, 0, stream()>>>(op.off.view(), n, op.index.reps,
                                                                     counts.ptr);
      LSAMD_HIP(hipGetLastError());
    } else {
      LSAMD_HIP(hipMemsetAsync(counts.ptr, 0, sizeof(uint32_t) * n, stream()));
    }
    if (!exclusive_scan(counts.ptr, n, reinterpret_cast<uint64_t *>(row_ptr.ptr), upper)) return false;
  }
  int64_t const up = static_cast<int64_t>(upper);
  LSAMD_HIP(hipMemcpyAsync(row_ptr.ptr + n, &up, sizeof(int64_t), hipMemcpyHostToDevice, stream()));
  timer_begin(kTimerCsrBuild);
  if (n > 0) {
    csr_diag_kernel<<<grid_for(n, 256), 256, 0, stream()>>>(make_view(op), c.diag64.ptr);
    LSAMD_HIP(hipGetLastError());
  }
  DeviceArray<uint32_t> cols;
  DeviceArray<double> vals;
  bool table = false, many = false;
  if (!cplx && op.allow_packing && up > 0 && !build_table_csr(op, up, row_ptr.ptr, table, many)) return false;
  if (table) {
    timer_end(kTimerCsrBuild);
    return finish_real_csr(op, precision, vals);
  }
  if (!cols.allocate(static_cast<size_t>(up > 0 ? up : 1))) return false;
  if (!vals.allocate(static_cast<size_t>(width * (up > 0 ? up : 1)))) return false;
  if (n > 0) {
    FillTargets t;
    t.cols = cols.ptr;
    t.vals = vals.ptr;
    t.kept = counts.ptr;
    if (!(cplx ? launch_fill<kFillComplex>(op, row_ptr.ptr, t) : launch_fill<kFillReal>(op, row_ptr.ptr, t)))
      return false;
  }
  timer_end(kTimerCsrBuild);
  if (!check_error(op)) return false;
  // Drop zero coefficients (the reference skips c == 0,
  // DistributedMatrixVector.chpl:127).
  uint64_t kept = 0;
  DeviceArray<uint64_t> new_ptr;
  if (!new_ptr.allocate(static_cast<size_t>(n + 1))) return false;
  if (n > 0 && !exclusive_scan(counts.ptr, n, new_ptr.ptr, kept)) return false;
  if (static_cast<int64_t>(kept) != up) {
    DeviceArray<uint32_t> cols2;
    DeviceArray<double> vals2;
    if (!cols2.allocate(static_cast<size_t>(kept > 0 ? kept : 1))) return false;
    if (!vals2.allocate(static_cast<size_t>(width * (kept > 0 ? kept : 1)))) return false;
    csr_compact_kernel<<<grid_for(n, 256), 256, 0, stream()>>>(n, row_ptr.ptr, cols.ptr, vals.ptr,
                                                               new_ptr.ptr, cols2.ptr, vals2.ptr, width);
    LSAMD_HIP(hipGetLastError());
    int64_t const kk = static_cast<int64_t>(kept);
    LSAMD_HIP(hipMemcpyAsync(new_ptr.ptr + n, &kk, sizeof(int64_t), hipMemcpyHostToDevice, stream()));
    LSAMD_HIP(hipStreamSynchronize(stream()));
    DeviceArray<int64_t> rp2;
    rp2.ptr = reinterpret_cast<int64_t *>(new_ptr.ptr);
    rp2.count = new_ptr.count;
    new_ptr.ptr = nullptr;
    new_ptr.count = 0;
    row_ptr = std::move(rp2);
    cols = std::move(cols2);
    vals = std::move(vals2);
  }
  c.nnz = static_cast<int64_t>(kept);
  // Source rows (the pairs each alpha_i emits) -> rows of M.
  if (!transpose_to_targets(n, c.nnz, width, row_ptr, cols, vals)) return false;
  c.row_ptr = std::move(row_ptr);
  c.cols = std::move(cols);
  if (cplx) {
    // complex values (re, im) in FP64 and FP32 for the embedded products
    int64_t const m = 2 * c.nnz;
    if (!c.vals32.allocate(static_cast<size_t>(m > 0 ? m : 1))) return false;
    if (!c.diag32.allocate(static_cast<size_t>(n > 0 ? n : 1))) return false;
    if (m > 0) to_f32_kernel<<<grid_for(m, 256), 256, 0, stream()>>>(m, vals.ptr, c.vals32.ptr);
    if (n > 0) to_f32_kernel<<<grid_for(n, 256), 256, 0, stream()>>>(n, c.diag64.ptr, c.diag32.ptr);
    LSAMD_HIP(hipGetLastError());
    c.vals64 = std::move(vals);
    c.has32 = c.has64 = true;
    c.is_complex = true;
    LSAMD_HIP(hipStreamSynchronize(stream()));
    return true;
  }
  if (op.allow_packing && !many && !try_pack_values(c, vals.ptr)) return false;
  return finish_real_csr(op, precision, vals);
}

} // namespace lsamd
