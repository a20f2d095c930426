// products.hip -- products with the cached CSR: FP64 vectors, FP64 and FP32
// blocks of right-hand sides, and the choice of their schedules.
#include <algorithm>

#include "operator_internal.hpp"
#include "orbit_device.hpp"

namespace lsamd {

// ---------------------------------------------------------------------------
// SpMV kernels: LPR lanes share one row
// ---------------------------------------------------------------------------

template <typename F> bool dispatch_lpr(int lpr, F &&f) {
  switch (lpr) {
  case 1: return f.template operator()<1>();
  case 2: return f.template operator()<2>();
  case 4: return f.template operator()<4>();
  case 8: return f.template operator()<8>();
  case 16: return f.template operator()<16>();
  case 32: return f.template operator()<32>();
  case 64: return f.template operator()<64>();
  default: return fail("lanes per row must be a power of two <= 64");
  }
}

// flags: bit 0 non-temporal stream loads, bit 1 die-aware persistent grid
template <typename F> bool dispatch_flags(int flags, F &&f) {
  switch (flags & 3) {
  case 0: return f.template operator()<false, false>();
  case 1: return f.template operator()<true, false>();
  case 2: return f.template operator()<false, true>();
  default: return f.template operator()<true, true>();
  }
}

// Grid of a product launch: one workgroup per tile; with the die-aware
// mapping (flags bit 1) either the persistent grid or, with bit 2, one
// workgroup per tile rounded up to a multiple of 8, where each workgroup
// takes one tile of its die's contiguous range.
int product_grid(OperatorCore const &op, int64_t n, int lpr, int flags) {
  int const tiles = grid_for(n * lpr, 256);
  if (flags & 2) return (flags & 4) ? (tiles + 7) / 8 * 8 : op.persistent_blocks;
  return tiles;
}

template <typename F> bool dispatch_k(int k, F &&f) {
  switch (k) {
  case 1: return f.template operator()<1>();
  case 2: return f.template operator()<2>();
  case 4: return f.template operator()<4>();
  case 8: return f.template operator()<8>();
  case 16: return f.template operator()<16>();
  default: return fail("block size must be 1, 2, 4, 8 or 16");
  }
}

// The schedule of a block product, by the bytes of x it gathers per stored
// entry: up to 16 B (FP32 blocks of 1, 2, 4; FP64 blocks of 1, 2) the one
// tuned on the FP64 vector (8 B), above that the one tuned on the FP32 block
// of 8 (32 B).  On 6x6 both are fastest with 16 lanes on the die-aware full
// grid (the FP32 block of 2 5.6 against 6.8 ms on the plain grid, the block of
// 8 9.2 against 10.2 ms); where x stays on chip the widths may differ.
struct Schedule {
  int lanes, flags;
};
Schedule block_schedule(OperatorCore const &op, size_t row_bytes) {
  return row_bytes <= 16 ? Schedule{op.lanes_f64, op.flags_f64} : Schedule{op.lanes_f32, op.flags_f32};
}

// The FP64 CSR product over `n` rows starting at row_ptr `rp` and output
// `y` (offsets of the whole arrays; x and the columns stay global).
bool launch_csr_f64(OperatorCore &op, int64_t const *rp, int64_t n, double const *d_x, double *d_y, int accumulate,
                    int has_diag) {
  Csr const &c = op.csr;
  int const grid = product_grid(op, n, op.lanes_f64, op.flags_f64);
  return dispatch_lpr(op.lanes_f64, [&]<int LPR>() -> bool {
    return dispatch_flags(op.flags_f64, [&]<bool NT, bool DIE>() -> bool {
      if (c.wide)
        csr_f64_wide_kernel<LPR, NT, DIE><<<grid, 256, sizeof(double) * c.table_size, stream()>>>(
            n, rp, c.cols.ptr, c.vidx.ptr, c.table64.ptr, c.table_size, c.diag64.ptr, d_x, d_y, accumulate, has_diag);
      else if (c.packed)
        csr_f64_kernel<LPR, NT, DIE, true><<<grid, 256, 0, stream()>>>(
            n, rp, c.cols.ptr, nullptr, c.table64.ptr, c.table_size, c.diag64.ptr, d_x, d_y, accumulate, has_diag);
      else
        csr_f64_kernel<LPR, NT, DIE, false><<<grid, 256, 0, stream()>>>(
            n, rp, c.cols.ptr, c.vals64.ptr, nullptr, 0, c.diag64.ptr, d_x, d_y, accumulate, has_diag);
      LSAMD_HIP(hipGetLastError());
      return true;
    });
  });
}

bool operator_csr_f64(OperatorCore &op, double const *d_x, double *d_y, bool accumulate) {
  Csr const &c = op.csr;
  if (c.is_complex) return fail("the CSR holds complex values: use a sector batch for its products");
  if (!c.has64) return fail("FP64 CSR has not been built");
  int64_t const n = c.rows;
  if (n == 0) return true;
  timer_begin(kTimerCsrF64);
  bool const ok = launch_csr_f64(op, c.row_ptr.ptr, n, d_x, d_y, accumulate ? 1 : 0, op.diag.count > 0 ? 1 : 0);
  timer_end(kTimerCsrF64);
  return ok;
}

__global__ __launch_bounds__(256) void diag_times_kernel(int64_t n, double const *__restrict__ diag,
                                                         double const *__restrict__ x, double *__restrict__ y) {
  int64_t const i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) y[i] = diag[i] * x[i];
}

bool operator_csr_f64_diag(OperatorCore &op, double const *d_x, double *d_y) {
  Csr const &c = op.csr;
  if (c.is_complex || !c.has64) return fail("FP64 CSR has not been built");
  if (c.rows == 0) return true;
  diag_times_kernel<<<grid_for(c.rows, 256), 256, 0, stream()>>>(c.rows, c.diag64.ptr, d_x, d_y);
  LSAMD_HIP(hipGetLastError());
  return true;
}

bool operator_csr_f64_rows(OperatorCore &op, double const *d_x, double *d_y, int64_t r0, int64_t r1) {
  Csr const &c = op.csr;
  if (c.is_complex || !c.has64) return fail("FP64 CSR has not been built");
  if (r0 < 0 || r1 > c.rows || r0 > r1) return fail("row range outside the CSR");
  if (r1 == r0) return true;
  return launch_csr_f64(op, c.row_ptr.ptr + r0, r1 - r0, d_x, d_y + r0, 1, 0);
}

bool operator_csr_f32_block(OperatorCore &op, int k, float const *d_x, float *d_y) {
  Csr const &c = op.csr;
  if (c.is_complex) return fail("the CSR holds complex values: use a sector batch for its products");
  if (!c.has32) return fail("FP32 CSR has not been built");
  int64_t const n = c.rows;
  if (n == 0) return true;
  Schedule const s = block_schedule(op, sizeof(float) * static_cast<size_t>(k));
  timer_begin(kTimerCsrF32);
  bool ok = dispatch_k(k, [&]<int K>() -> bool {
    return dispatch_lpr(s.lanes, [&]<int LPR>() -> bool {
      int const grid = product_grid(op, n, LPR, s.flags);
      return dispatch_flags(s.flags, [&]<bool NT, bool DIE>() -> bool {
        if (c.wide)
          csr_block_wide_kernel<K, LPR, float, float, NT, DIE><<<grid, 256, sizeof(float) * c.table_size, stream()>>>(
              n, c.row_ptr.ptr, c.cols.ptr, c.vidx.ptr, c.table32.ptr, c.table_size, c.diag32.ptr, d_x, d_y);
        else if (c.packed)
          csr_block_kernel<K, LPR, float, float, NT, DIE, true><<<grid, 256, 0, stream()>>>(
              n, c.row_ptr.ptr, c.cols.ptr, nullptr, c.table32.ptr, c.table_size, c.diag32.ptr, d_x, d_y);
        else
          csr_block_kernel<K, LPR, float, float, NT, DIE, false><<<grid, 256, 0, stream()>>>(
              n, c.row_ptr.ptr, c.cols.ptr, c.vals32.ptr, nullptr, 0, c.diag32.ptr, d_x, d_y);
        LSAMD_HIP(hipGetLastError());
        return true;
      });
    });
  });
  timer_end(kTimerCsrF32);
  return ok;
}

bool operator_csr_f64_block(OperatorCore &op, int k, double const *d_x, double *d_y) {
  Csr const &c = op.csr;
  if (c.is_complex) return fail("the CSR holds complex values: use a sector batch for its products");
  if (!c.has64) return fail("FP64 CSR has not been built");
  int64_t const n = c.rows;
  if (n == 0) return true;
  Schedule const s = block_schedule(op, sizeof(double) * static_cast<size_t>(k));
  timer_begin(kTimerCsrF64Block);
  bool ok = dispatch_k(k, [&]<int K>() -> bool {
    return dispatch_lpr(s.lanes, [&]<int LPR>() -> bool {
      int const grid = product_grid(op, n, LPR, s.flags);
      return dispatch_flags(s.flags, [&]<bool NT, bool DIE>() -> bool {
        if (c.wide)
          csr_block_wide_kernel<K, LPR, double, double, NT, DIE><<<grid, 256, sizeof(double) * c.table_size,
                                                                   stream()>>>(
              n, c.row_ptr.ptr, c.cols.ptr, c.vidx.ptr, c.table64.ptr, c.table_size, c.diag64.ptr, d_x, d_y);
        else if (c.packed)
          csr_block_kernel<K, LPR, double, double, NT, DIE, true><<<grid, 256, 0, stream()>>>(
              n, c.row_ptr.ptr, c.cols.ptr, nullptr, c.table64.ptr, c.table_size, c.diag64.ptr, d_x, d_y);
        else
          csr_block_kernel<K, LPR, double, double, NT, DIE, false><<<grid, 256, 0, stream()>>>(
              n, c.row_ptr.ptr, c.cols.ptr, c.vals64.ptr, nullptr, 0, c.diag64.ptr, d_x, d_y);
        LSAMD_HIP(hipGetLastError());
        return true;
      });
    });
  });
  timer_end(kTimerCsrF64Block);
  return ok;
}

// Times every product schedule (lanes per row x stream-load kind x grid
// mapping) on the cached matrix and keeps the fastest, separately for the
// FP64 kernel and the FP32 block-of-8 kernel: the schedules of the narrow
// and the wide gathers (block_schedule).
// plain, non-temporal, die-aware persistent (with / without non-temporal),
// die-aware over the full grid (with / without non-temporal)
constexpr int kScheduleFlags[] = {0, 1, 2, 3, 6, 7};

int operator_autotune(OperatorCore &op) {
  Csr const &c = op.csr;
  int64_t const n = c.rows;
  if (n == 0 || c.is_complex) return op.lanes_f64;
  op.schedule_set = true;
  hipDeviceProp_t prop;
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) {
    // four workgroups per CU; with the wide table as many as fit beside their
    // LDS copies of it (up to eight), so each CU stages the table a few times
    int per_cu = 4;
    if (c.wide)
      per_cu = static_cast<int>(std::min<size_t>(
          8, std::max<size_t>(1, (160u << 10) / (sizeof(double) * static_cast<size_t>(c.table_size)))));
    op.persistent_blocks = std::max(8, (prop.multiProcessorCount * per_cu / 8) * 8);
  }
  int const cand[] = {2, 4, 8, 16, 32, 64};
  hipEvent_t e0, e1;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  auto time_it = [&](auto &&launch) -> float {
    launch();
    (void)hipEventRecord(e0, stream());
    for (int r = 0; r < 3; ++r) launch();
    (void)hipEventRecord(e1, stream());
    (void)hipEventSynchronize(e1);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, e0, e1);
    return ms;
  };
  if (c.has64) {
    DeviceArray<double> x, y;
    if (x.allocate(n) && y.allocate(n)) {
      (void)hipMemsetAsync(x.ptr, 0, sizeof(double) * n, stream());
      float best = 1e30f;
      int best_l = op.lanes_f64, best_f = op.flags_f64;
      for (int f : kScheduleFlags)
        for (int l : cand) {
          op.lanes_f64 = l;
          op.flags_f64 = f;
          float const ms = time_it([&] { (void)operator_csr_f64(op, x.ptr, y.ptr, false); });
          if (ms < best) {
            best = ms;
            best_l = l;
            best_f = f;
          }
        }
      op.lanes_f64 = best_l;
      op.flags_f64 = best_f;
    }
  }
  if (c.has32) {
    DeviceArray<float> x, y;
    if (x.allocate(static_cast<size_t>(n) * 8) && y.allocate(static_cast<size_t>(n) * 8)) {
      (void)hipMemsetAsync(x.ptr, 0, sizeof(float) * n * 8, stream());
      float best = 1e30f;
      int best_l = op.lanes_f32, best_f = op.flags_f32;
      for (int f : kScheduleFlags)
        for (int l : cand) {
          op.lanes_f32 = l;
          op.flags_f32 = f;
          float const ms = time_it([&] { (void)operator_csr_f32_block(op, 8, x.ptr, y.ptr); });
          if (ms < best) {
            best = ms;
            best_l = l;
            best_f = f;
          }
        }
      op.lanes_f32 = best_l;
      op.flags_f32 = best_f;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipStreamSynchronize(stream());
  return op.lanes_f64;
}

} // namespace lsamd
