// trid_adjoint.hip -- adjoint of the strided-batch solves
// (tridXmtsvStridedBatchAdjoint of include/trid_adjoint.h).
//
// One kernel solves the transposed systems and forms the coefficient
// gradients from the solution in registers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>

#include "../../include/trid_adjoint.h"
#include "../../include/trid_hip_ext.h"
#include "trid_launch.hpp"
#include "trid_runtime.hpp"

namespace tridhip {

// Adjoint of a strided batch in one pass: lambda = A^{-T} g and, from the
// same registers, grad_a_i = -lambda_i x_{i-1}, grad_b_i = -lambda_i x_i,
// grad_c_i = -lambda_i x_{i+1}, grad_d = lambda.  Every array has the layout
// of SysDesc array 0.  The partitioned solve and its lane mappings are those
// of part_block; the transposed rows are the c of the row above and the a of
// the row below.
//   ORDER 1 (VEC 0): systems in consecutive lanes, rows read and written as
//            coalesced runs across systems.
//   ORDER 0, VEC 4: each wave's chunks cover one contiguous span of every
//            array, moved in 16-byte pieces through the wave's LDS buffer
//            (gspan_load / gspan_store); the rows just outside the span are
//            read one by one.
//   ORDER 0, VEC 0: per-lane rows, for layouts the staging does not take.
// Every a, b, c and g row a work-group reads is read before its first store,
// so grad_a .. grad_d may overwrite them.
// HBM-bound: 9 words per unknown (a, b, c, x, g in, four gradients out), of
// which the separate solve and elementwise gradient kernel it replaces moved
// 12.  FP32 1000 x 4000, solvedim 0: 160 us (per-lane rows) + 24 us before,
// 33 us now (4.3 TB/s); FP64 [100, 300, 80], solvedim 1: 49 us + 151 us (the
// gradient kernel's threads ran along the strided rows) before, 50 us (3.5 TB/s)
// now.
template <typename T, int ORDER, int R, int VEC, typename I, int CP>
__global__ void __launch_bounds__((VEC == 4 || (R >= 16 && sizeof(T) == 8)) ? 512 : 1024)
    k_adj(const T *__restrict__ A, const T *__restrict__ B, const T *__restrict__ C,
          const T *__restrict__ X, const T *__restrict__ G, T *__restrict__ GA,
          T *__restrict__ GB, T *__restrict__ GC, T *__restrict__ GD, SysDesc D, int chunks,
          int spb_log2, int xcd) {
  constexpr bool GSTAGE = VEC == 4;
  constexpr int SW = kWave * R + (GSTAGE ? Vec16<T>::n : 0);  // a wave's staging buffer
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *sm = reinterpret_cast<T *>(smem_raw);
  long long block = blockIdx.x;
  if (xcd) {
    const unsigned nb8 = gridDim.x & ~7u;
    if (blockIdx.x < nb8) block = (long long)(blockIdx.x & 7u) * (nb8 >> 3) + (blockIdx.x >> 3);
  }
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int cps_log2 = chunks;  // (ORDER 0; ORDER 1: the count, any number)
  const int cps = ORDER == 0 ? 1 << chunks : chunks, spb = 1 << spb_log2;
  const int k = ORDER == 0 ? tid & (cps - 1) : tid >> spb_log2;
  const int slot = ORDER == 0 ? tid >> cps_log2 : tid & (spb - 1);
  const long long q = block * spb + slot;
  const bool active = q < D.nsys;
  const int N = D.N, row0 = k * R;
  I offs[5] = {0, 0, 0, 0, 0};
  if (active) sys_offsets<I>(D, q, offs);
  const I off = offs[0], s = (I)D.sstr[0];

  // the wave's span (VEC 4): wave_len elements from wave_off; the lane's
  // chunk starts at span element g_idx
  T *stage = sm + (tid >> 6) * SW;
  bool wave_active = active;
  int wave_len = 0, g_idx = 0;
  I wave_off = 0;
  if constexpr (GSTAGE) {
    const long long q0 = ((long long)__builtin_amdgcn_readfirstlane((int)(q >> 32)) << 32) |
                         (unsigned)__builtin_amdgcn_readfirstlane((int)(q & 0xffffffffLL));
    const int row0w = __builtin_amdgcn_readfirstlane(row0);
    wave_active = q0 < D.nsys && row0w < N;
    if (cps <= kWave) {
      const long long nact = D.nsys - q0 < (kWave >> cps_log2) ? D.nsys - q0 : (kWave >> cps_log2);
      wave_len = (int)(nact * N);
      g_idx = (int)(q - q0) * N + row0;
    } else {
      wave_len = N - row0w < kWave * R ? N - row0w : kWave * R;
      g_idx = row0 - row0w;
    }
    const I o = off + (I)row0;
    if constexpr (sizeof(I) == 4) {
      wave_off = (I)__builtin_amdgcn_readfirstlane((int)o);
    } else {
      const int lo = __builtin_amdgcn_readfirstlane((int)(o & 0xffffffffLL));
      const int hi = __builtin_amdgcn_readfirstlane((int)(o >> 32));
      wave_off = (I)(((long long)hi << 32) | (unsigned)lo);
    }
  }
  // v[r] = element of row row0 + r + SH (SH in -1..1), `fill` off the system
  auto rows = [&](auto shift, const T *__restrict__ p, T (&v)[R], T fill) {
    constexpr int SH = decltype(shift)::value;
    if constexpr (GSTAGE) {
      if (!wave_active) return;
      const int sh = gspan_load<T, R, I, CP>(p, wave_off, wave_len, stage, lane);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int row = row0 + r + SH, j = g_idx + r + SH;
        const bool ok = active && row >= 0 && row < N;
        // the first / last row of a wave may have its neighbour in another wave
        const bool edge = (SH < 0 && r == 0 && j < 0) || (SH > 0 && r == R - 1 && j >= wave_len);
        T t = fill;
        if (ok && !edge) t = stage[sh + j];
        if (SH != 0 && ok && edge) t = *at(p, off + (I)row);
        v[r] = t;
      }
      __builtin_amdgcn_wave_barrier();
    } else {
#pragma unroll
      for (int r = 0; r < R; r++) {
        const int row = row0 + r + SH;
        v[r] = active && row >= 0 && row < N ? ld_stream<CP>(at(p, off + (I)row * s)) : fill;
      }
    }
  };
  auto put = [&](T *__restrict__ p, const T (&v)[R]) {
    if constexpr (GSTAGE) {
      if (!wave_active) return;
      const int sh = (int)(wave_off & (I)(Vec16<T>::n - 1));
#pragma unroll
      for (int r = 0; r < R; r++)
        if (active && row0 + r < N) stage[sh + g_idx + r] = v[r];
      __builtin_amdgcn_wave_barrier();
      gspan_store<T, R, I, CP>(p, wave_off, wave_len, stage, lane, false);
    } else {
#pragma unroll
      for (int r = 0; r < R; r++)
        if (active && row0 + r < N) st_stream<CP>(at(p, off + (I)(row0 + r) * s), v[r]);
    }
  };
  using Prev = std::integral_constant<int, -1>;
  using Same = std::integral_constant<int, 0>;
  using Next = std::integral_constant<int, 1>;

  T a[R], b[R], c[R], d[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    a[r] = T(0);
    b[r] = T(1);
    c[r] = T(0);
    d[r] = T(0);
  }
  rows(Prev(), C, a, T(0));
  rows(Same(), B, b, T(1));
  rows(Next(), A, c, T(0));
  rows(Same(), G, d, T(0));
  // rows past the system's end are identity rows; the row below the last is
  // off the system, so its a is zero already
#pragma unroll
  for (int r = 1; r < R; r++)
    if (row0 + r >= N) a[r] = T(0);
  if (row0 >= N) a[0] = T(0);
  Row<T> f, l;
  chunk_reduce<T, R>(a, b, c, d, f, l);
  T xf, xl;
  if (ORDER == 0 && cps <= kWave)
    reduced_wave<T>(f, l, k, cps, lane, xf, xl);
  else if (GSTAGE)
    reduced_multi<T>(f, l, k, cps, slot, sm + (size_t)(blockDim.x >> 6) * SW, xf, xl);
  else if (cps <= kWave)
    reduced_lds_w<T>(f, l, k, cps, slot, spb, sm, xf, xl);
  else
    reduced_lds<T>(f, l, k, cps, slot, spb, sm, xf, xl);
  T y[R];
  chunk_expand<T, R>(a, c, d, xf, xl, y);

  put(GD, y);
  T x[R], t[R];
  rows(Same(), X, x, T(0));
  // x of the rows around the chunk: ORDER 0 has the neighbour chunks in the
  // neighbour lanes, except across waves
  T xp = T(0), xn = T(0);
  bool lp = active && row0 > 0 && row0 <= N, ln = active && row0 + R < N;
  if constexpr (ORDER == 0) {
    xp = lane_read(x[R - 1], lane > 0 ? lane - 1 : 0);
    xn = lane_read(x[0], lane < kWave - 1 ? lane + 1 : lane);
    lp = lp && lane == 0;
    ln = ln && lane == kWave - 1;
  }
  if (lp) xp = *at(X, off + (I)(row0 - 1) * s);
  if (ln) xn = *at(X, off + (I)(row0 + R) * s);
#pragma unroll
  for (int r = 0; r < R; r++) t[r] = -y[r] * x[r];
  put(GB, t);
#pragma unroll
  for (int r = 0; r < R; r++) t[r] = row0 + r > 0 ? -y[r] * (r > 0 ? x[r > 0 ? r - 1 : 0] : xp) : T(0);
  put(GA, t);
#pragma unroll
  for (int r = 0; r < R; r++)
    t[r] = row0 + r + 1 < N ? -y[r] * (r + 1 < R ? x[r + 1 < R ? r + 1 : 0] : xn) : T(0);
  put(GC, t);
}

template <typename T, int ORDER, int R, int VEC>
hipError_t launch_adj_t(const PartCfg &cfg, const T *a, const T *b, const T *c, const T *x,
                        const T *g, T *ga, T *gb, T *gc, T *gd, const SysDesc &D,
                        hipStream_t st) {
  const int cps = chunk_count(cfg), spb = 1 << cfg.spb_log2, threads = cps * spb;
  const unsigned blocks = (unsigned)((D.nsys + spb - 1) / spb);
  size_t lds = 0;
  if (ORDER == 1 || cps > kWave) lds = 2 * 3 * (size_t)cps * (spb + 1) * sizeof(T);
  if (VEC == 4)
    lds = (size_t)(threads / kWave) * (kWave * R + 16 / sizeof(T) + (cps > kWave ? 12 : 0)) *
          sizeof(T);
#define TRID_ADJ(II, CC)                                                                     \
  hipLaunchKernelGGL((k_adj<T, ORDER, R, VEC, II, CC>), dim3(blocks), dim3(threads), lds, st, a, \
                     b, c, x, g, ga, gb, gc, gd, D, chunk_arg(cfg), cfg.spb_log2, cfg.xcd)
  if (!cfg.idx32) TRID_ADJ(long long, kStream);
  else if (cfg.cp == kCached) TRID_ADJ(uint32_t, kCached);
  else TRID_ADJ(uint32_t, kStream);
#undef TRID_ADJ
  return hipGetLastError();
}

template <typename T>
hipError_t launch_adj(const PartCfg &cfg, const T *a, const T *b, const T *c, const T *x,
                      const T *g, T *ga, T *gb, T *gc, T *gd, const SysDesc &D,
                      hipStream_t st) {
#define TRID_CASE(ORD, RR, VV)                                 \
  if (cfg.order == ORD && cfg.R == RR && cfg.vec == VV)        \
    return launch_adj_t<T, ORD, RR, VV>(cfg, a, b, c, x, g, ga, gb, gc, gd, D, st);
  TRID_CASE(0, 8, 4)
  TRID_CASE(0, 12, 4)
  TRID_CASE(0, 16, 4)
  TRID_CASE(0, 8, 0)
  TRID_CASE(0, 16, 0)
  TRID_CASE(1, 8, 0)
  TRID_CASE(1, 16, 0)
#undef TRID_CASE
  return hipErrorInvalidValue;
}

}  // namespace tridhip

using namespace tridhip;

namespace {

// Chunk layout of a contiguous (solvedim 0) adjoint: general staging with the
// chunk length that pads the system to the fewest rows (16 rows only past
// the 6144 that 512 chunks of 12 hold).  The lengths are within 5 % of each
// other where more than one fits (FP64 1000 x 4000: 8, 12 and 16 rows 172,
// 173 and 178 us for forward and backward through autograd).  kind 0 where
// the staging does not apply: arrays not 16-byte aligned, or padded systems
// that share a wave.
// Batches of at most one wave of 8-row chunks per SIMD (65536 lanes) wait on
// each chunk's serial rows, not on bandwidth: the shortest chunks, in one-wave
// work-groups (FP64, N x systems, against the fewest rows in 256 threads: 20 x
// 1000 10.7 -> 7.9 us, 40 x 40 9.9 -> 7.9, 1000 x 10 11.4 -> 10.2, 90 x 4000
// 13.5 -> 11.6; above the line 600 x 800 14.7 -> 15.7, 150 x 8000 17.8 -> 20.3).
// Past 256 chunks per system the reduced solve costs more than the rows save
// (3000 x 5, 512 chunks of 8 rows 14.6 us, 256 of 12 13.4).
PartCfg adj_rows(int N, long long nsys, bool aligned, bool dense) {
  PartCfg best;
  best.kind = 0;
  const PartCfg small = make_cfg(0, 8, N, 0, kWave);
  if (N <= 2048 && gstage_ok(small, aligned, dense) && nsys << small.cps_log2 <= 65536) {
    best = small;
    best.vec = 4;
    return best;
  }
  for (int R : {8, 12, 16}) {
    PartCfg c = make_cfg(0, R, N, 0, 256);
    if (!gstage_ok(c, aligned, dense)) continue;
    if (best.kind == 1 && ((long long)R << c.cps_log2) >= ((long long)best.R << best.cps_log2))
      continue;
    best = c;
    best.vec = 4;
  }
  return best;
}

template <typename T>
tridStatus_t strided_adjoint(const T *a, const T *b, const T *c, const T *x, const T *g,
                             T *ga, T *gb, T *gc, T *gd, int ndim, int solvedim,
                             const int *dims, const int *pads, int sync) {
  clear_error();
  if (!dims) return fail(TRID_STATUS_INVALID_VALUE, "dims is NULL");
  if (ndim < 1 || ndim > MAXDIM) return fail(TRID_STATUS_INVALID_VALUE, "ndim must be in [1, 8]");
  if (solvedim < 0 || solvedim >= ndim)
    return fail(TRID_STATUS_INVALID_VALUE, "solvedim must be in [0, ndim)");
  if (!pads) pads = dims;
  SysDesc D;
  memset(&D, 0, sizeof D);
  D.N = dims[solvedim];
  D.nsys = 1;
  long long cum = 1, ext = 1;
  for (int k = 0; k < ndim; k++) {
    if (dims[k] < 0 || pads[k] < dims[k])
      return fail(TRID_STATUS_INVALID_VALUE, "bad dims/pads");
    if (k == solvedim) {
      for (int t = 0; t < 5; t++) D.sstr[t] = cum;
    } else {
      D.osize[D.nother] = dims[k];
      for (int t = 0; t < 5; t++) D.ostr[t][D.nother] = cum;
      D.nother++;
      D.nsys *= dims[k];
    }
    ext += (long long)(dims[k] - 1) * cum;
    cum *= pads[k];
  }
  if (D.N == 0 || D.nsys == 0) return TRID_STATUS_SUCCESS;
  if (!a || !b || !c || !x || !g || !ga || !gb || !gc || !gd)
    return fail(TRID_STATUS_INVALID_VALUE, "NULL array");
  D.small_index = D.nsys < (1LL << 31) && !wide_index();
  hipStream_t st = current_stream();
  const int order = solvedim == 0 ? 0 : 1;
  PartCfg cfg = heuristic(order, D.N, 0, sizeof(T));
  if (cfg.kind != 1) return fail(TRID_STATUS_INVALID_VALUE, "system too long for the adjoint kernel");
  cfg.vec = 0;
  bool dense = true, aligned = true;
  for (int k = 0; k < ndim; k++) dense &= pads[k] == dims[k];
  const void *ptrs[9] = {a, b, c, x, g, ga, gb, gc, gd};
  for (const void *p : ptrs) aligned &= aligned16(p);
  if (order == 1) {
    // the strided batches' layout (most systems per work-group)
    const PartCfg s = strided_default(D.N, sizeof(T));
    if (s.kind == 1) cfg = s;
    RowRuns rr;
    rr.inc = true;  // (as many values per row in flight)
    const PartCfg w = strided_wide(D.N, D.nsys, sizeof(T), rr);
    if (w.kind == 1) cfg = w;
  } else {
    const PartCfg s = adj_rows(D.N, D.nsys, aligned, dense);
    if (s.kind == 1) cfg = s;
  }
  const size_t bytes = (size_t)ext * sizeof(T);
  cfg.idx32 = bytes < (1ULL << 32) && !wide_index();
  // nine arrays; there is no mixed form
  cfg.cp = cfg.idx32 && cache_policy(9 * bytes) == kCached ? kCached : kStream;
  tridStatus_t s = check_hip(launch_adj<T>(cfg, a, b, c, x, g, ga, gb, gc, gd, D, st),
                             "adjoint launch");
  if (s) return s;
  if (sync) return check_hip(hipStreamSynchronize(st), "hipStreamSynchronize");
  return TRID_STATUS_SUCCESS;
}

}  // namespace

EXTERN_C tridStatus_t tridDmtsvStridedBatchAdjoint(
    const double *a, const double *b, const double *c, const double *x,
    const double *g, double *grad_a, double *grad_b, double *grad_c,
    double *grad_d, int ndim, int solvedim, int *dims, int *pads, int sync) {
  return strided_adjoint<double>(a, b, c, x, g, grad_a, grad_b, grad_c, grad_d, ndim,
                                 solvedim, dims, pads, sync);
}

EXTERN_C tridStatus_t tridSmtsvStridedBatchAdjoint(
    const float *a, const float *b, const float *c, const float *x,
    const float *g, float *grad_a, float *grad_b, float *grad_c, float *grad_d,
    int ndim, int solvedim, int *dims, int *pads, int sync) {
  return strided_adjoint<float>(a, b, c, x, g, grad_a, grad_b, grad_c, grad_d, ndim,
                                solvedim, dims, pads, sync);
}
