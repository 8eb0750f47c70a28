// Batched SPD solves wider than 64 (spd_solve, lm/kernels/mamba4.py:188-217,
// whose _factor_and_solve :164-187 takes any width).  Widths up to 64 take
// the four-systems-per-wave kernels of factor.hip; these take one block per
// system.
//
// Up to kBlockMaxDim (208): a blocked right-looking Cholesky in LDS
// (spd_block_kernel).  Above, a column at a time in the caller's factor
// buffer (spd_wide_kernel):
//
//   - the system's lower triangle is copied into it (upper triangle zeroed);
//   - one column per step: the reciprocal pivot 1/L_jj = rsq(M_jj)
//     (v_rsq_f32, as the 64-wide path and the reference's lax.rsqrt pivot),
//     the column scaled below the diagonal and copied into an LDS vector,
//     then the rank-one update of the trailing lower triangle, rows split
//     over eight groups of 32 lanes, columns over the group's lanes, so a
//     row's update is one contiguous run; M_jj ends holding 1/L_jj;
//   - forward substitution L w = b by columns (every step scales the final
//     w_j and updates the entries below it in parallel) and backward
//     substitution L^T y = w by rows of L (contiguous), one barrier per
//     step.
//
// A non-positive pivot gives NaN, which propagates to the solution, as the
// reference's does.  Stored factor (dense, [dim][dim] row-major): L below the
// diagonal, 1/L_ii on it, zero above.
#include "common.hpp"

namespace m4 {

// M: the system's lower triangle (row stride ld); col: dim floats of LDS.
__device__ void wide_factor(float* M, int ld, int dim, float* col) {
  const int tid = threadIdx.x, grp = tid >> 5, c = tid & 31;
  for (int j = 0; j < dim; ++j) {
    const float rs = __builtin_amdgcn_rsqf(M[j * ld + j]);
    for (int i = j + 1 + tid; i < dim; i += kWideThreads) {
      const float l = M[i * ld + j] * rs;
      M[i * ld + j] = l;
      col[i] = l;
    }
    __syncthreads();  // column j is final and in col
    for (int i = j + 1 + grp; i < dim; i += kWideThreads / 32) {
      const float lij = col[i];
      for (int k = j + 1 + c; k <= i; k += 32) M[i * ld + k] -= lij * col[k];
    }
    // Every thread read M_jj before the barrier above; no step after this
    // one reads or writes it.
    if (tid == 0) M[j * ld + j] = rs;
    __syncthreads();  // the trailing update is done before the next pivot
  }
}

// L w = b then L^T y = w with M holding the factor as wide_factor leaves it.
// w: dim floats of LDS holding b on entry (overwritten); t: dim floats of
// LDS, y on return.
__device__ void wide_solve(const float* M, int ld, int dim, float* w, float* t) {
  const int tid = threadIdx.x;
  for (int j = 0; j < dim; ++j) {
    // w_j is final: every column before j has updated it (barrier below).
    const float wj = w[j] * M[j * ld + j];
    for (int i = j + 1 + tid; i < dim; i += kWideThreads) w[i] -= M[i * ld + j] * wj;
    if (tid == 0) t[j] = wj;
    __syncthreads();
  }
  for (int i = tid; i < dim; i += kWideThreads) w[i] = t[i];
  __syncthreads();
  for (int j = dim - 1; j >= 0; --j) {
    const float yj = w[j] * M[j * ld + j];
    for (int i = tid; i < j; i += kWideThreads) w[i] -= M[j * ld + i] * yj;
    if (tid == 0) t[j] = yj;
    __syncthreads();
  }
}

// precision [N,dim,dim] (only k <= i read), rhs [N,dim] -> solution [N,dim]
// and the dense factor [N,dim,dim], in which the factorization runs.
__global__ __launch_bounds__(kWideThreads) void spd_wide_kernel(
    const float* __restrict__ precision, const float* __restrict__ rhs, int dim,
    float* __restrict__ solution, float* __restrict__ factors) {
  extern __shared__ float sm[];
  const long n = blockIdx.x, dd = (long)dim * dim;
  const int tid = threadIdx.x;
  float* const col = sm;
  float* const w = col + dim;
  float* const t = w + dim;
  float* const M = factors + n * dd;
  const float* const A = precision + n * dd;
  for (long e = tid; e < dd; e += kWideThreads) {
    const int i = (int)(e / dim), k = (int)(e - (long)i * dim);
    M[e] = k <= i ? A[e] : 0.f;
  }
  for (int i = tid; i < dim; i += kWideThreads) w[i] = rhs[n * dim + i];
  __syncthreads();
  wide_factor(M, dim, dim, col);
  wide_solve(M, dim, dim, w, t);
  for (int i = tid; i < dim; i += kWideThreads) solution[n * dim + i] = t[i];
}

// VJP (lm/kernels/mamba4.py:204-215): z = A^-1 g from the stored dense
// factor, d_rhs = z, d_precision = -(z y^T + y z^T) / 2 (exactly symmetric).
__global__ __launch_bounds__(kWideThreads) void spd_wide_backward_kernel(
    const float* __restrict__ factors, const float* __restrict__ solution,
    const float* __restrict__ d_solution, int dim, float* __restrict__ d_precision,
    float* __restrict__ d_rhs) {
  extern __shared__ float sm[];
  const long n = blockIdx.x, dd = (long)dim * dim;
  const int tid = threadIdx.x;
  float* const y = sm;
  float* const w = y + dim;
  float* const t = w + dim;
  const float* const M = factors + n * dd;
  for (int i = tid; i < dim; i += kWideThreads) {
    w[i] = d_solution[n * dim + i];
    y[i] = solution[n * dim + i];
  }
  __syncthreads();
  wide_solve(M, dim, dim, w, t);
  for (int i = tid; i < dim; i += kWideThreads) d_rhs[n * dim + i] = t[i];
  for (long e = tid; e < dd; e += kWideThreads) {
    // Both products rounded on their own, so d_precision is exactly
    // symmetric.
#pragma clang fp contract(off)
    const int i = (int)(e / dim), k = (int)(e - (long)i * dim);
    d_precision[n * dd + e] = -0.5f * (t[i] * y[k] + y[i] * t[k]);
  }
}

// ---------------------------------------------------------------------------
// Widths 65 .. kBlockMaxDim: 16-column panels, the system in LDS as the
// 16x16 tiles of its lower triangle (row stride 17), padded with an identity
// block to a multiple of 16.  Per panel:
//
//   - every row from the panel down is one lane's: its sixteen values in
//     registers, eliminated column by column with the panel's own rows' values
//     read from their lanes into scalar registers.  Each of the NW waves holds
//     the panel's 16 rows itself (lanes 0..15) and 48 rows below, so the
//     elimination crosses no wave: NW = 2 up to width 112, 3 to 160, 4 to 208.
//     The forward substitution runs along (as in factor.hip);
//   - the panel's rank-16 update of the trailing tiles on fp32 MFMA, the
//     tiles dealt over the waves.
//
// Two barriers a panel where a column at a time took two a column and the
// whole trailing triangle through LDS each: 2,048 systems of 96 took 334 us
// and take 89 (the backward, whose two substitutions run on one wave, 111 and
// 46), bound by the panels' elimination chain.

__device__ __forceinline__ int tile_at(int I, int K) { return (I * (I + 1) / 2 + K) * kBlockTile; }
__device__ __forceinline__ int tile_element(int i, int k) {
  return tile_at(i >> 4, k >> 4) + (i & 15) * 17 + (k & 15);
}
__device__ __forceinline__ float lane_at(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// The lower triangle of a dense [dim][dim] matrix into tiles, padded with an
// identity block and with zeros above the diagonal of its diagonal tiles.
// Sixteen rows' loads go out together (row by row, each waiting for its own,
// the loads of 2,048 systems of 96 took most of 125 us).
template <int NW>
__device__ __forceinline__ void load_tiles(float* tiles, const float* A, int dim, int nb, int wave,
                                           int l) {
  for (int I = wave; I < nb; I += NW)
    for (int k0 = 0; k0 < 16 * (I + 1); k0 += 64) {
      const int k = k0 + l;
      float v[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 16 * I + r;
        v[r] = A[(long)min(i, dim - 1) * dim + min(k, dim - 1)];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 16 * I + r;
        if (k < 16 * (I + 1))
          tiles[tile_element(i, k)] = i < dim ? (k <= i ? v[r] : 0.f) : i == k ? 1.f : 0.f;
      }
    }
}

// L^T y = w for the factor in `tiles`, by one wave: w [dp] in LDS on entry, y
// on return.  Block rows from the last up: sixteen steps inside the block
// (lane k holds column k of the diagonal tile), then every earlier entry takes
// the block's solution.
__device__ __forceinline__ void block_backward(const float* tiles, int nb, float* w) {
  const int l = threadIdx.x & 63, r = l & 15;
  for (int P = nb - 1; P >= 0; --P) {
    const float* diag = tiles + tile_at(P, P);
    float c[16], x = w[16 * P + r], y = 0.f, ys[16];
#pragma unroll
    for (int J = 0; J < 16; ++J) c[J] = diag[J * 17 + r];
    const float inv = diag[r * 17 + r];
#pragma unroll
    for (int J = 15; J >= 0; --J) {
      ys[J] = lane_at(x * inv, J);
      y = r == J ? ys[J] : y;
      x -= c[J] * ys[J];  // only the lanes below J are used again
    }
    if (l < 16) w[16 * P + r] = y;
    for (int k = l; k < 16 * P; k += 64) {
      const float* row = tiles + tile_at(P, k >> 4) + (k & 15);
      float acc = w[k];
#pragma unroll
      for (int J = 0; J < 16; ++J) acc -= row[J * 17] * ys[J];
      w[k] = acc;
    }
  }
}

// The padding's entries, which the forward substitution leaves at 0 times the
// system's own (not a number where one of those is infinite): none of it may
// reach the backward substitution.  One wave.
__device__ __forceinline__ void clear_padding(float* w, int dim, int nb) {
  const int l = threadIdx.x & 63;
  if (dim + l < 16 * nb) w[dim + l] = 0.f;
}

// L w = b likewise (b in `w` on entry), block rows from the first down.
__device__ __forceinline__ void block_forward(const float* tiles, int nb, float* w) {
  const int l = threadIdx.x & 63, r = l & 15;
  for (int P = 0; P < nb; ++P) {
    const float* diag = tiles + tile_at(P, P);
    float c[16], x = w[16 * P + r], y = 0.f, ws[16];
#pragma unroll
    for (int J = 0; J < 16; ++J) c[J] = diag[r * 17 + J];
    const float inv = diag[r * 17 + r];
#pragma unroll
    for (int J = 0; J < 16; ++J) {
      ws[J] = lane_at(x * inv, J);
      y = r == J ? ws[J] : y;
      x -= c[J] * ws[J];  // only the lanes above J are used again
    }
    if (l < 16) w[16 * P + r] = y;
    for (int i = 16 * (P + 1) + l; i < 16 * nb; i += 64) {
      const float* row = tiles + tile_at(i >> 4, P) + (i & 15) * 17;
      float acc = w[i];
#pragma unroll
      for (int J = 0; J < 16; ++J) acc -= row[J] * ws[J];
      w[i] = acc;
    }
  }
}

template <int NW>
__global__ __launch_bounds__(64 * NW) void spd_block_kernel(const float* __restrict__ precision,
                                                            const float* __restrict__ rhs, int dim,
                                                            float* __restrict__ solution,
                                                            float* __restrict__ factors) {
  extern __shared__ float sm[];
  const int nb = (dim + 15) / 16, dp = 16 * nb;
  float* const panel = sm;  // [dp][20]: the panel's rows below its diagonal tile
  float* const w = panel + dp * 20;
  float* const tiles = w + dp;
  const long n = blockIdx.x;
  const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float* A = precision + n * dim * dim;
  load_tiles<NW>(tiles, A, dim, nb, wave, l);
  for (int i = threadIdx.x; i < dp; i += 64 * NW) w[i] = i < dim ? rhs[n * dim + i] : 0.f;
  __syncthreads();
  for (int P = 0; P < nb; ++P) {
    const int j0 = 16 * P, row = l < 16 ? j0 + l : j0 + 48 * wave + l;
    const bool valid = row < dp, mine = valid && (l >= 16 || wave == 0);
    float* at = tiles + tile_element(valid ? row : j0, j0);
    float a[16], x = w[valid ? row : j0], solved = 0.f, inv = 0.f;
#pragma unroll
    for (int J = 0; J < 16; ++J) a[J] = at[J];
#pragma unroll
    for (int J = 0; J < 16; ++J) {
      const float rs = __builtin_amdgcn_rsqf(lane_at(a[J], J));
      const float wj = lane_at(x, J) * rs;
      a[J] *= rs;
      // Rows of the panel above J hold scratch here that nothing reads.
      x -= a[J] * wj;
      solved = l == J ? wj : solved;
      inv = l == J ? rs : inv;
#pragma unroll
      for (int K = J + 1; K < 16; ++K) a[K] -= a[J] * lane_at(a[J], K);
    }
    __syncthreads();  // every wave has read the panel's rows and w
    if (mine) {
      w[row] = l < 16 ? solved : x;
#pragma unroll
      for (int J = 0; J < 16; ++J) at[J] = l >= 16 || J < l ? a[J] : J == l ? inv : 0.f;
      if (l >= 16)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<f4*>(panel + row * 20 + 4 * q) =
              f4{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
    }
    __syncthreads();
    // Tile (I, K) -= L_I L_K^T: lane (g, r) gives rows 16 I + r and 16 K + r at
    // k = 4g + e in step e, and holds rows 16 I + 4g + q of column 16 K + r.
    int t = 0;
    for (int I = P + 1; I < nb; ++I) {
      const f4 li = *reinterpret_cast<const f4*>(panel + (16 * I + r) * 20 + 4 * g);
      for (int K = P + 1; K <= I; ++K, ++t) {
        if (t % NW != wave) continue;  // uniform over the wave
        const f4 lk = *reinterpret_cast<const f4*>(panel + (16 * K + r) * 20 + 4 * g);
        float* c = tiles + tile_at(I, K) + 4 * g * 17 + r;
        f4 acc = f4{c[0], c[17], c[34], c[51]};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-li[e], lk[e], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) c[17 * q] = acc[q];
      }
    }
    __syncthreads();
  }
  if (wave == 0) {
    clear_padding(w, dim, nb);
    block_backward(tiles, nb, w);
    for (int i = l; i < dim; i += 64) solution[n * dim + i] = w[i];
  }
  // The factor goes out on the other waves meanwhile.
  if (factors && wave > 0)
    for (int i = wave - 1; i < dim; i += NW - 1)
      for (int k = l; k < dim; k += 64)
        factors[(n * dim + i) * dim + k] = k <= i ? tiles[tile_element(i, k)] : 0.f;
}

template <int NW>
__global__ __launch_bounds__(64 * NW) void spd_block_backward_kernel(
    const float* __restrict__ factors, const float* __restrict__ solution,
    const float* __restrict__ d_solution, int dim, float* __restrict__ d_precision,
    float* __restrict__ d_rhs) {
  extern __shared__ float sm[];
  const int nb = (dim + 15) / 16, dp = 16 * nb;
  float* const z = sm;
  float* const y = z + dp;
  float* const tiles = y + dp;
  const long n = blockIdx.x;
  const int l = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  load_tiles<NW>(tiles, factors + n * dim * dim, dim, nb, wave, l);
  for (int i = threadIdx.x; i < dp; i += 64 * NW) {
    z[i] = i < dim ? d_solution[n * dim + i] : 0.f;
    y[i] = i < dim ? solution[n * dim + i] : 0.f;
  }
  __syncthreads();
  if (wave == 0) {
    block_forward(tiles, nb, z);
    clear_padding(z, dim, nb);
    block_backward(tiles, nb, z);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < dim; i += 64 * NW) d_rhs[n * dim + i] = z[i];
  for (int i = wave; i < dim; i += NW) {
    const float zi = z[i], yi = y[i];
    for (int k = l; k < dim; k += 64) {
      // Both products rounded on their own, so d_precision is exactly
      // symmetric.
#pragma clang fp contract(off)
      d_precision[(n * dim + i) * dim + k] = -0.5f * (zi * y[k] + yi * z[k]);
    }
  }
}

#define M4_SPD_BLOCK(NW)                                                                      \
  template __global__ void spd_block_kernel<NW>(const float*, const float*, int, float*,      \
                                                float*);                                      \
  template __global__ void spd_block_backward_kernel<NW>(const float*, const float*,          \
                                                         const float*, int, float*, float*);
M4_SPD_BLOCK(2)
M4_SPD_BLOCK(3)
M4_SPD_BLOCK(4)
#undef M4_SPD_BLOCK

}  // namespace m4
