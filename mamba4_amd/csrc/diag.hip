// Spectral and finiteness probes of the final selective precision: restates
// selective_diagnostics (lm/kernels/mamba4.py:358-376).
//
// diag_eigen_kernel: one 256-thread block per (batch, head) state, float64
// throughout (exact for the float32 inputs).  The symmetrised precision
// (E + E^T) / 2 + diag(floor) is brought to tridiagonal form by Householder
// reflections, and the two extreme eigenvalues are found by multisection on
// the Sturm counts of the tridiagonal (Barth, Martin and Wilkinson,
// Numerische Mathematik 9 (1967) 386-393): 64 shifts a round, one per lane,
// so a round narrows the interval 65 times and ten reach float64.  Both steps
// are backward stable, as eigvalsh's own; the extremes are then rounded to
// float32.  Rows and columns are taken in descending order of the diagonal's
// magnitude, so a coordinate far above the others (a large floor) is split off
// before it can mix with them, and no tolerance is relative to the largest
// entry: the small eigenvalues of such a precision keep their own precision.
//
// Thread (r, w) holds columns 16w..16w+15 of row r of that order in registers.  A
// reflection takes a product of the matrix with the vector (16 multiply-adds
// a thread, the four waves' parts meeting in LDS) and a rank-two update (32),
// two barriers in all.  Bound by that chain of 62 reflections.  A cyclic
// Jacobi iteration, every eigenvalue by up to forty sweeps of 63 rounds of
// four barriers on one wave, took 4,557 us for 192 states of 64; this takes
// 124.
// The same pass takes the state's finiteness and the cross statistics'
// largest magnitude.
//
// diag_summary_kernel: one block reduces the per-state values and the floor.
#include "common.hpp"

namespace m4 {

__device__ __forceinline__ float wave_min(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fminf(x, __shfl_xor(x, o));
  return x;
}
__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
  return x;
}
// x at the lane of this lane's 16-lane row that the DPP pattern selects.
template <int CTRL>
__device__ __forceinline__ double dpp64(double x) {
  const uint2 u = __builtin_bit_cast(uint2, x);
  return __builtin_bit_cast(
      double, uint2{(unsigned)__builtin_amdgcn_update_dpp(0, (int)u.x, CTRL, 0xf, 0xf, true),
                    (unsigned)__builtin_amdgcn_update_dpp(0, (int)u.y, CTRL, 0xf, 0xf, true)});
}

// Sum over the wave's 64 lanes, the same total in every lane.
__device__ __forceinline__ double wave_sum(double x) {
  x += dpp64<0xB1>(x);   // quad_perm [1,0,3,2]
  x += dpp64<0x4E>(x);   // quad_perm [2,3,0,1]
  x += dpp64<0x141>(x);  // row_half_mirror
  x += dpp64<0x140>(x);  // row_mirror
  uint2 u = __builtin_bit_cast(uint2, x);
  auto lo = __builtin_amdgcn_permlane16_swap(u.x, u.x, false, false);
  auto hi = __builtin_amdgcn_permlane16_swap(u.y, u.y, false, false);
  x = __builtin_bit_cast(double, uint2{lo[0], hi[0]}) +
      __builtin_bit_cast(double, uint2{lo[1], hi[1]});
  u = __builtin_bit_cast(uint2, x);
  lo = __builtin_amdgcn_permlane32_swap(u.x, u.x, false, false);
  hi = __builtin_amdgcn_permlane32_swap(u.y, u.y, false, false);
  return __builtin_bit_cast(double, uint2{lo[0], hi[0]}) +
         __builtin_bit_cast(double, uint2{lo[1], hi[1]});
}

// x at lane `lane` (the same for the whole wave).
__device__ __forceinline__ double lane_double(double x, int lane) {
  const uint2 u = __builtin_bit_cast(uint2, x);
  return __builtin_bit_cast(double, uint2{(unsigned)__builtin_amdgcn_readlane((int)u.x, lane),
                                          (unsigned)__builtin_amdgcn_readlane((int)u.y, lane)});
}

// 1 / q to float64 rounding or so: the hardware's estimate and two Newton
// steps (q neither zero nor subnormal).
__device__ __forceinline__ double reciprocal(double q) {
  double r = __builtin_amdgcn_rcp(q);
  r = __builtin_fma(__builtin_fma(-q, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-q, r, 1.0), r, r);
}

// Eigenvalues below x of the tridiagonal with diagonal d and squared
// off-diagonal e2 (e2[i] between i and i + 1), n rows: the negative pivots of
// T - x (a pivot under kTiny counts as -kTiny: below any float32, and float32's
// squares over it are finite).
constexpr double kTiny = 0x1p-700;
__device__ __forceinline__ int sturm_count(const double* d, const double* e2, int n, double x) {
  int count = 0;
  double q = d[0] - x;
  for (int i = 0;; ++i) {
    if (fabs(q) < kTiny) q = -kTiny;
    count += q < 0.0;
    if (i + 1 == n) return count;
    q = (d[i + 1] - x) - e2[i] * reciprocal(q);
  }
}

// per_state[4 bh + 0..3] = min eigenvalue, max eigenvalue (both NaN when the
// precision has a non-finite entry, as eigvalsh gives), 1 if every entry of
// the state (evidence and cross) is finite else 0, max |cross| (NaN if a
// cross entry is NaN, as jnp.max gives).
__global__ __launch_bounds__(256) void diag_eigen_kernel(const float* __restrict__ evidence,
                                                         const float* __restrict__ cross,
                                                         const float* __restrict__ floor, int H,
                                                         int D, int P,
                                                         float* __restrict__ per_state) {
  __shared__ double column[2][64];  // the next column to reduce (double buffered)
  __shared__ double part[4][64];
  __shared__ double diagonal[64], off2[64];
  __shared__ int order[64];
  __shared__ float extreme[2], wave_max_cross[4];
  const int bh = blockIdx.x, h = bh % H, r = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float* E = evidence + (long)bh * D * D;
  bool finite = true, prec_finite = true, cross_nan = false;
  // order[i]: the row with the i-th largest diagonal magnitude (as ordered bits,
  // ties by row; rows past D last).
  const float fl = r < D ? floor[h * D + r] : 0.f;
  const unsigned key = r < D ? __float_as_uint(fabsf(E[r * D + r] + fl)) : 0u;
  int rank = 0;
#pragma unroll
  for (int j = 0; j < 64; ++j) {
    const unsigned other = (unsigned)__builtin_amdgcn_readlane((int)key, j);
    rank += other > key || (other == key && j < r);
  }
  if (w == 0) order[rank] = r;
  __syncthreads();
  const int pr = order[r];  // below D for r < D
  const float fr = __shfl(fl, pr);
  double a[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int c = 16 * w + j, pc = order[c];
    a[j] = 0.0;
    if (r < D && c < D) {
      const float x = E[pr * D + pc], y = E[pc * D + pr];
      finite = finite && isfinite(x);
      a[j] = 0.5 * ((double)x + (double)y);
      if (c == r) {
        prec_finite = isfinite(fr);
        a[j] += (double)fr;
      }
    }
  }
  prec_finite = prec_finite && finite;
  float cmax = 0.f;
  const float* C = cross + (long)bh * P * D;
  for (long i = threadIdx.x; i < (long)P * D; i += 256) {
    const float v = C[i];
    finite = finite && isfinite(v);
    cross_nan = cross_nan || isnan(v);
    cmax = fmaxf(cmax, fabsf(v));
  }
  cmax = wave_max(cmax);
  if (r == 0) wave_max_cross[w] = cmax;
  if (w == 0) column[0][r] = a[0];
  // Uniform over the block from here on.
  const bool any_bad_precision = __syncthreads_or(!prec_finite);
  const bool any_bad = __syncthreads_or(!finite);
  const bool any_cross_nan = __syncthreads_or(cross_nan);

  // Column k at step k is final up to row k; its entries below are reflected
  // onto row k + 1.  Rows and columns up to k hold stale values afterwards
  // that nothing reads.
  if (!any_bad_precision) {
    // A column of norm below 2^-300 (nothing beside any float32) under its first
    // entry is reduced already: what is left of a rank-deficient matrix
    // would otherwise shrink by 2^-53 a step until its squares underflow.
    constexpr double negligible = 0x1p-600;
    for (int k = 0; k < D; ++k) {
      const double x = column[k & 1][r];
      if (w == 0 && r == k) diagonal[k] = x;
      if (k + 1 == D) break;
      const double below = r > k + 1 && r < D ? x : 0.0;
      const double tail = wave_sum(below * below), head = lane_double(x, k + 1);
      double off = head;
      if (tail > negligible) {  // the same in every thread: uniform
        const double norm = sqrt(head * head + tail);
        off = head > 0.0 ? -norm : norm;
        const double v = r == k + 1 ? head - off : below;
        // 2 / v^T v = 1 / (norm (norm + |head|)).
        const double beta = 1.0 / (norm * (norm + fabs(head)));
        double p = 0.0;
#pragma unroll
        for (int j = 0; j < 16; ++j) p = __builtin_fma(a[j], lane_double(v, 16 * w + j), p);
        part[w][r] = p;
        __syncthreads();
        p = r > k && r < D ? beta * (part[0][r] + part[1][r] + part[2][r] + part[3][r]) : 0.0;
        const double u = p - 0.5 * beta * wave_sum(p * v) * v;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          a[j] = __builtin_fma(-v, lane_double(u, 16 * w + j), a[j]);
          a[j] = __builtin_fma(-u, lane_double(v, 16 * w + j), a[j]);
        }
      }
      if (w == 0 && r == 0) off2[k] = off * off;
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (16 * w + j == k + 1) column[(k + 1) & 1][r] = a[j];
      __syncthreads();
    }
    __syncthreads();

    // Wave 0 finds the smallest eigenvalue (the least x with a count of 1),
    // wave 1 the largest (with a count of D), between Gershgorin's bounds.
    if (w < 2) {
      const double d = r < D ? diagonal[r] : 0.0;
      const double left = r > 0 && r < D ? sqrt(off2[r - 1]) : 0.0;
      const double right = r + 1 < D ? sqrt(off2[r]) : 0.0;
      double lo = r < D ? d - left - right : INFINITY, hi = r < D ? d + left + right : -INFINITY;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, o));
        hi = fmax(hi, __shfl_xor(hi, o));
      }
      lo -= fabs(lo) * 0x1p-48 + kTiny;
      hi += fabs(hi) * 0x1p-48 + kTiny;
      const int want = w == 0 ? 1 : D;
      // Ten rounds where the extremes are within some orders of magnitude; the
      // bound covers float32's whole range (an interval below 2^-170 rounds to
      // zero).
      for (int round = 0; round < 60; ++round) {
        if (hi - lo <= fmax(0x1p-52 * fmax(fabs(lo), fabs(hi)), 0x1p-170)) break;  // uniform
        const double step = (hi - lo) * (1.0 / 65.0), x = lo + step * (r + 1);
        const unsigned long long at = __ballot(sturm_count(diagonal, off2, D, x) >= want);
        // The counts grow with the shift (up to rounding): the first lane
        // that reaches the count bounds the eigenvalue from above.
        const int first = at ? __builtin_ctzll(at) : 64;
        hi = first < 64 ? lane_double(x, first) : hi;
        lo = first > 0 ? lane_double(x, first - 1) : lo;
      }
      if (r == 0) extreme[w] = (float)(0.5 * lo + 0.5 * hi);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    per_state[4 * bh + 0] = any_bad_precision ? NAN : extreme[0];
    per_state[4 * bh + 1] = any_bad_precision ? NAN : extreme[1];
    per_state[4 * bh + 2] = any_bad ? 0.f : 1.f;
    per_state[4 * bh + 3] =
        any_cross_nan ? NAN
                      : fmaxf(fmaxf(wave_max_cross[0], wave_max_cross[1]),
                              fmaxf(wave_max_cross[2], wave_max_cross[3]));
  }
}

// summary[0..6] = min eigenvalue, max eigenvalue, max condition (per state,
// max / max(min, 1e-30)), all finite (1 / 0), max |cross|, min floor, max
// floor (lm/kernels/mamba4.py:368-376).  One block of sixteen waves: a chain of
// loads per thread (16 us with four waves at 192 states of 64, 5.8 with sixteen).
constexpr int kSummaryThreads = 1024;
__global__ __launch_bounds__(kSummaryThreads) void diag_summary_kernel(const float* __restrict__ per_state,
                                                           int states, const float* __restrict__ floor,
                                                           int floors, float* __restrict__ summary) {
  __shared__ float part[7][kSummaryThreads / 64];
  float lo = INFINITY, hi = -INFINITY, cond = -INFINITY, fin = 1.f, cm = 0.f;
  float flo = INFINITY, fhi = -INFINITY;
  bool nan_ev = false, nan_cross = false, nan_floor = false;
  for (int i = threadIdx.x; i < states; i += kSummaryThreads) {
    const float a = per_state[4 * i], b = per_state[4 * i + 1];
    nan_ev = nan_ev || isnan(a) || isnan(b);
    nan_cross = nan_cross || isnan(per_state[4 * i + 3]);
    lo = fminf(lo, a);
    hi = fmaxf(hi, b);
    cond = fmaxf(cond, b / fmaxf(a, 1e-30f));
    fin = fminf(fin, per_state[4 * i + 2]);
    cm = fmaxf(cm, per_state[4 * i + 3]);
  }
  #pragma unroll 4
  for (int i = threadIdx.x; i < floors; i += kSummaryThreads) {
    const float f = floor[i];
    nan_floor = nan_floor || isnan(f);
    flo = fminf(flo, f);
    fhi = fmaxf(fhi, f);
  }
  const float vals[7] = {lo, hi, cond, fin, cm, flo, fhi};
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const bool is_min = k == 0 || k == 3 || k == 5;
    const float v = is_min ? wave_min(vals[k]) : wave_max(vals[k]);
    if (l == 0) part[k][w] = v;
  }
  const bool any_ev = __syncthreads_or(nan_ev), any_cross = __syncthreads_or(nan_cross);
  const bool any_floor = __syncthreads_or(nan_floor);
  if (threadIdx.x < 7) {
    const int k = threadIdx.x;
    const bool is_min = k == 0 || k == 3 || k == 5;
    float v = part[k][0];
    for (int j = 1; j < kSummaryThreads / 64; ++j) v = is_min ? fminf(v, part[k][j]) : fmaxf(v, part[k][j]);
    // The reference's jnp.min / jnp.max propagate NaN; fminf / fmaxf drop
    // it, so it is put back where the reference would have it.
    if ((k <= 2 && any_ev) || (k == 4 && any_cross) || (k >= 5 && any_floor)) v = NAN;
    summary[k] = v;
  }
}

}  // namespace m4
