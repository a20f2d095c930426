// species.hip -- tables of spinful fermion groups, and the bases that use them.
//
// A spinful state is (down << sites) | up and every group element permutes the
// sites of both species alike, so an image is (e(down), e(up)) and the least
// one has the least image of `down`.  For at most 16 sites the least image of
// every species state, the elements that reach it and the sign of every
// element on every species state fit tables of about 2 MB, which take 0.16 ms
// of kernels to make.  With them the 4x4 basis of 7 + 7 fermions (131 M products, 1.02 M
// representatives) lists the down states that are their own least image and
// tests 1.3 M products: 3.3 -> 0.54 ms with the making of group and tables, 0.4 ms
// where those are there, most of it launches and copies of a few KB.
#include <algorithm>

#include "orbit_device.hpp"

namespace lsamd {

size_t species_lds_bytes(GroupData const &g) {
  bool const narrow = g.canonical_shifts && (g.depth == 7 || g.depth == 9); // the words dispatch_group picks
  return (static_cast<size_t>(g.size) * g.depth * (narrow ? 4 : 8) + 7) / 8 * 8;
}

// Least image of every species state and how many elements reach it.
template <typename W, int D>
__global__ __launch_bounds__(256) void species_least_kernel(GroupView g, int states, uint64_t *__restrict__ entry,
                                                            uint32_t *__restrict__ counts) {
  int const s = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (s >= states) return;
  W least = ~W{0};
  uint32_t count = 0;
  for (int e = 0; e < g.size; ++e) {
    W const y = group_apply<W, D>(g, e, static_cast<W>(s));
    count = y < least ? 1u : count + (y == least ? 1u : 0u);
    least = y < least ? y : least;
  }
  entry[s] = static_cast<uint64_t>(least) | static_cast<uint64_t>(count) << 16;
  counts[s] = count;
}

template <typename W, int D>
__global__ __launch_bounds__(256) void species_list_kernel(GroupView g, int states,
                                                           uint64_t const *__restrict__ places,
                                                           uint64_t *__restrict__ entry, uint16_t *__restrict__ list) {
  int const s = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (s >= states) return;
  uint64_t const at = places[s], mine = entry[s];
  uint64_t o = at;
  for (int e = 0; e < g.size; ++e)
    if (group_apply<W, D>(g, e, static_cast<W>(s)) == static_cast<W>(mine & 0xffffu)) list[o++] = static_cast<uint16_t>(e);
  entry[s] = mine | at << 32;
}

// sign[e][s / 32], bit s % 32: element e reorders the operators of s by an odd
// permutation.  fermion_sign reads orbital images of the whole state; a
// species state is its low half.
__global__ __launch_bounds__(256) void species_sign_kernel(GroupView g, int states, int words,
                                                           uint32_t *__restrict__ sign) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<int64_t>(g.size) * words) return;
  int const e = static_cast<int>(i / words), w = static_cast<int>(i % words);
  uint32_t bits = 0;
  for (int q = 0; q < 32; ++q) {
    int const s = 32 * w + q;
    if (s < states && fermion_sign(g, e, static_cast<uint64_t>(s)) < 0.0) bits |= 1u << q;
  }
  sign[i] = bits;
}

bool group_plan_species(GroupData &g) {
  int const sites = g.number_bits / 2, G = g.size;
  if (sites < 1 || sites > kMaxSpeciesSites || G < 1 || G > 0xffff || species_lds_bytes(g) > kMaxSpeciesLds) return true;
  for (int e = 0; e < G; ++e)
    if (g.h_eig_re[e] != 1.0 && g.h_eig_re[e] != -1.0) return true;
  int const states = 1 << sites, words = (states + 31) / 32;
  // rank of element e in the eight-lane state_info reduction: lane e mod 8,
  // then position within the lane, the G mod 8 tail elements last
  int const lanes = kStateInfoLanes, chunks = G / lanes;
  std::vector<int32_t> rank(static_cast<size_t>(G));
  for (int e = 0; e < G; ++e) rank[e] = e < chunks * lanes ? (e % lanes) * chunks + e / lanes : e;
  DeviceArray<uint64_t> entry, places;
  DeviceArray<uint32_t> counts, sign;
  DeviceArray<uint16_t> list;
  if (!entry.allocate(static_cast<size_t>(states)) || !places.allocate(static_cast<size_t>(states)) ||
      !counts.allocate(static_cast<size_t>(states)) || !sign.allocate(static_cast<size_t>(G) * words) ||
      !g.d_species_rank.upload(rank.data(), rank.size()))
    return false;
  GroupView const v = g.view();
  uint64_t total = 0;
  bool const ok = dispatch_group(g, [&]<typename W, int D, int SI>() -> bool {
    if constexpr (SI == kFermionic) {
      species_least_kernel<W, D><<<grid_for(states, 256), 256, 0, stream()>>>(v, states, entry.ptr, counts.ptr);
      LSAMD_HIP(hipGetLastError());
      if (!exclusive_scan(counts.ptr, states, places.ptr, total) || !list.allocate(static_cast<size_t>(total)))
        return false;
      species_list_kernel<W, D><<<grid_for(states, 256), 256, 0, stream()>>>(v, states, places.ptr, entry.ptr, list.ptr);
      LSAMD_HIP(hipGetLastError());
      return true;
    }
    return fail("species tables need a fermionic group");
  });
  if (!ok) return false;
  species_sign_kernel<<<grid_for(static_cast<int64_t>(G) * words, 256), 256, 0, stream()>>>(v, states, words, sign.ptr);
  LSAMD_HIP(hipGetLastError());
  LSAMD_HIP(hipStreamSynchronize(stream()));
  g.d_species_entry = std::move(entry);
  g.d_species_list = std::move(list);
  g.d_species_sign = std::move(sign);
  return true;
}

// ---------------------------------------------------------------------------
// Enumeration: the down state of a representative is its own least image, and
// no element that keeps it may take the up state below itself; the signed sum
// over those that keep both is the squared norm.
// ---------------------------------------------------------------------------

// Flags of the species states of one weight in [lower, upper], with `least`
// only those that are their own least image.
__global__ __launch_bounds__(256) void species_flags_kernel(uint64_t const *__restrict__ entry, int states, int weight,
                                                            uint32_t lower, uint32_t upper, int least,
                                                            uint32_t *__restrict__ flags) {
  int const s = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (s >= states) return;
  uint32_t const u = static_cast<uint32_t>(s);
  flags[s] = __popc(u) == weight && u >= lower && u <= upper && (!least || (entry[s] & 0xffffu) == u) ? 1u : 0u;
}

__global__ __launch_bounds__(256) void species_compact_kernel(uint32_t const *__restrict__ flags,
                                                              uint64_t const *__restrict__ places, int states,
                                                              uint32_t *__restrict__ out) {
  int const s = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (s < states && flags[s] != 0) out[places[s]] = static_cast<uint32_t>(s);
}

// Acceptance bits of the products (one word a wave) and how many a workgroup
// accepts: a fifth of a byte of scratch per product.
template <typename W, int D>
__global__ __launch_bounds__(256) void species_count_kernel(GroupView g, uint32_t const *__restrict__ downs,
                                                            uint32_t const *__restrict__ ups, int64_t nup,
                                                            int64_t total, uint64_t *__restrict__ bits,
                                                            uint32_t *__restrict__ counts) {
  extern __shared__ uint64_t search_lds[];
  SpeciesSearch<W, D> search;
  search.stage(g, search_lds);
  __syncthreads();
  int64_t const c = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  bool ok = c < total;
  if (ok) {
    uint32_t const down = downs[c / nup], up = ups[c % nup];
    int const words = ((1 << (g.nbits / 2)) + 31) / 32;
    uint64_t const entry = g.species_entry[down];
    int const count = static_cast<int>(entry >> 16 & 0xffffu);
    uint16_t const *list = g.species_list + (entry >> 32);
    int sum = 0;
    for (int i = 0; i < count && ok; ++i) {
      int const e = list[i];
      W const y = search.up_image(g, e, static_cast<W>(up));
      ok = y >= static_cast<W>(up);
      if (y == static_cast<W>(up)) {
        bool const minus = search.odd(g, e, up, words) != search.odd(g, e, down, words);
        sum += (g.eig_re[e] < 0.0) != minus ? -1 : 1;
      }
    }
    ok = ok && static_cast<double>(sum) > g.norm_eps;
  }
  uint64_t const mask = __ballot(ok);
  if ((threadIdx.x & 63) == 0) bits[c >> 6] = mask;
  int const accepted = __syncthreads_count(ok);
  if (threadIdx.x == 0) counts[blockIdx.x] = static_cast<uint32_t>(accepted);
}

__global__ __launch_bounds__(256) void species_write_kernel(uint32_t const *__restrict__ downs,
                                                            uint32_t const *__restrict__ ups, int64_t nup,
                                                            int sites, uint64_t const *__restrict__ bits,
                                                            uint64_t const *__restrict__ offsets,
                                                            uint64_t *__restrict__ out) {
  int64_t const c = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  uint64_t const word = bits[c >> 6];
  if ((word >> (c & 63) & 1u) == 0) return;
  uint64_t o = offsets[blockIdx.x] + static_cast<uint64_t>(__popcll(word & ((uint64_t{1} << (c & 63)) - 1)));
  for (int64_t w = static_cast<int64_t>(blockIdx.x) * 4; w < c >> 6; ++w) o += static_cast<uint64_t>(__popcll(bits[w]));
  out[o] = static_cast<uint64_t>(downs[c / nup]) << sites | ups[c % nup];
}

bool enumerate_species(GroupData const &g, uint64_t min_up, uint64_t max_up, uint64_t min_down, uint64_t max_down,
                       DeviceArray<uint64_t> &out, uint64_t &kept) {
  GroupView const v = g.view();
  int const sites = g.number_bits / 2, states = 1 << sites, grid = grid_for(states, 256);
  DeviceArray<uint32_t> flags, list[2];
  DeviceArray<uint64_t> places;
  if (!flags.allocate(static_cast<size_t>(states)) || !places.allocate(static_cast<size_t>(states))) return false;
  int64_t size[2] = {0, 0};
  kept = 0;
  for (int down = 0; down < 2; ++down) {
    uint64_t const lower = down ? min_down : min_up, upper = down ? max_down : max_up;
    uint64_t count = 0;
    species_flags_kernel<<<grid, 256, 0, stream()>>>(g.d_species_entry.ptr, states, __builtin_popcountll(lower),
                                                     static_cast<uint32_t>(lower), static_cast<uint32_t>(upper), down,
                                                     flags.ptr);
    LSAMD_HIP(hipGetLastError());
    if (!exclusive_scan(flags.ptr, states, places.ptr, count)) return false;
    if (count == 0) {
      out.reset();
      return true;
    }
    if (!list[down].allocate(static_cast<size_t>(count))) return false;
    species_compact_kernel<<<grid, 256, 0, stream()>>>(flags.ptr, places.ptr, states, list[down].ptr);
    LSAMD_HIP(hipGetLastError());
    size[down] = static_cast<int64_t>(count);
  }
  int64_t const total = size[0] * size[1];
  int const groups = grid_for(total, 256);
  DeviceArray<uint32_t> counts;
  DeviceArray<uint64_t> bits, offsets;
  if (!bits.allocate(4 * static_cast<size_t>(groups)) || !counts.allocate(static_cast<size_t>(groups)) ||
      !offsets.allocate(static_cast<size_t>(groups)))
    return false;
  bool const ok = dispatch_group(g, [&]<typename W, int D, int SI>() -> bool {
    if constexpr (SI == kFermionic) {
      species_count_kernel<W, D><<<groups, 256, species_lds_bytes(g), stream()>>>(
          v, list[1].ptr, list[0].ptr, size[0], total, bits.ptr, counts.ptr);
      LSAMD_HIP(hipGetLastError());
      return true;
    }
    return fail("species tables need a fermionic group");
  });
  if (!ok || !exclusive_scan(counts.ptr, groups, offsets.ptr, kept) || !out.allocate(static_cast<size_t>(kept)))
    return false;
  if (kept > 0) {
    species_write_kernel<<<groups, 256, 0, stream()>>>(list[1].ptr, list[0].ptr, size[0], sites, bits.ptr, offsets.ptr,
                                                       out.ptr);
    LSAMD_HIP(hipGetLastError());
  }
  LSAMD_HIP(hipStreamSynchronize(stream()));
  return true;
}

} // namespace lsamd
