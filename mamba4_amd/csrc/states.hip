// Chunk-boundary states: chunk statistics on MFMA plus an elementwise scan.
//
// Forward (lm/kernels/mamba4_fused.py:411-425 with chunk_carry,
// lm/kernels/prefix.py:27-44).  fwd_stats_kernel computes, for every chunk
// in parallel, the statistics K^T diag(tail) K of each sub-chunk and
// V^T diag(tail) K of the chunk, tail_s = beta_s exp(P_last - P_s), and
// writes them into the start-state buffers.  fwd_scan_kernel then turns them
// into start states in place, walking chunks in order per matrix element:
//   start[u] = running;  running = exp(sum of log decays in u) running + stat[u]
// and writes the final state.
//
// Value-dependent states (cross statistics and their cotangents) are NV
// stacked 64x64 tiles per state; each tile is one more product, and the scans
// treat the NV * 4096 elements of a cross state alike.
//
// Either pair gives the same bits as states_kernel's walk below: the same
// weights and decays from one scan of a chunk's log decays, a chunk's product
// summed from zero in the same order, and one multiply-add per state and step.
//
// Backward: the transpose of that carry.  bwd_local_kernel computes each
// chunk's start-state cotangents U = -(M + M^T)/2, M = Z^T diag(e^P) Y, and
// V = dOut^T diag(e^P) Y; bwd_scan_kernel walks chunks in reverse,
//   end[n] = running;  running = U_n + exp(sum of log decays in n) running,
// leaving each chunk's end-state cotangent and the initial-state gradient.
// The evidence end-state cotangents G are stored as G + G^T: every use the
// chunk gradients make of G is through its symmetric part ((G + G^T) k,
// k^T G k, <G, S> with S symmetric), and a symmetric G + G^T takes one
// product where G itself takes two.
#include "common.hpp"

namespace m4 {

__device__ __forceinline__ float* mat(float* base, long index) { return base + index * 4096; }

// a x + b, one rounding each.
__device__ __forceinline__ f4 fma4(float a, const f4& x, const f4& b) {
  f4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = __builtin_fmaf(a, x[e], b[e]);
  return r;
}

// acc += (A diag(wt))^T B over k in [k0, k0 + 16) for rows 16 w.. of the result
// and its columns 4r + jb: A(i, k) = A[k][16w + i] wt[k], B(k, c) = B[k][c]
// (tile_mma's QUAD convention, the weights applied as the operand leaves LDS).
__device__ __forceinline__ void weighted_strip(f4 acc[4], const float* A, const float* B,
                                               const float* wt, int k0, int w) {
  const int l = lane_id(), r = l & 15, kk = k0 + 4 * (l >> 4);
  const f4 t = *reinterpret_cast<const f4*>(wt + kk);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = A[(kk + e) * LDT + 16 * w + r] * t[e];
    const f4 bv = *reinterpret_cast<const f4*>(B + (kk + e) * LDT + 4 * r);
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
      acc[jb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bv[jb], acc[jb], 0, 0, 0);
  }
}

// One block per chunk of a sequence.  Every tile is loaded at once and staged
// behind one barrier, and each product weighs its tokens as it reads them: a
// weighted copy of the keys and values in LDS (an exponential per element,
// two barriers per product) had a B1 T2000 H12 P128 launch at 23.8 us, now 13.9 (and bwd_local
// at B8 T1737 H8 P64 44.9, now 35.1).
//
// MIX: the keys come from the mixer's raw projections, shifted and normalised
// as they are staged, and the gates from theirs (`gates`), written out for the
// later kernels (as states_kernel's evidence walks do).
template <typename In, bool MIX>
__global__ __launch_bounds__(256) void fwd_stats_kernel(
    Dims d, const In* __restrict__ keys, const In* __restrict__ values,
    const float* __restrict__ beta, const float* __restrict__ log_decay,
    float* __restrict__ start_s, float* __restrict__ start_c, MixerIn mix, MixerGates gates) {
  extern __shared__ float smem[];
  float* K = smem;
  float* V = K + TILE;  // NV tiles
  __shared__ ChunkScalars cs;
  __shared__ alignas(16) float wt[3][MAXC];  // the sub-chunks' weights, then the chunk's
  const long seq = blockIdx.x;
  const int n = (int)(seq % d.NC), bh = (int)(seq / d.NC), b = bh / d.H, h = bh % d.H;
  const int len = chunk_len(d, n), w = threadIdx.x >> 6, c4 = 4 * (lane_id() & 15);
  const long row = token_head(d, b, n * d.chunk, h);
  RowTile<In> rk, rv0, rv1;
  if constexpr (MIX)
    rk.fetch_mix_keys(len, mix, d, b, h, n * d.chunk);
  else
    rk.fetch_tokens(len, keys + row * 64, (unsigned)(d.H * 64));
  rv0.fetch_tokens(len, values + row * d.P, (unsigned)(d.H * d.P));
  rv1.fetch_tokens(d.NV > 1 ? len : 0, values + row * d.P + (d.NV > 1 ? 64 : 0),
                   (unsigned)(d.H * d.P));
  if constexpr (MIX) {
    if (threadIdx.x < 64) {
      const int s = threadIdx.x;
      const long th = row + (long)(s < len ? s : 0) * d.H;
      const float dt = gates.dt_raw[th], bt = gates.beta_raw[th];
      const float g = s < len ? mix_log_decay(gates, dt, h) : 0.f;
      const float be = s < len ? mix_beta(gates, bt, h) : 0.f;
      if (s < len) {
        gates.log_decay[th] = g;
        gates.beta[th] = be;
      }
      finish_chunk_scalars(cs, g, be);
      if (n == 0 && b == 0)
        gates.floor[h * 64 + s] = gates.floor_min + mix_softplus(gates.floor_raw[h * 64 + s]);
    }
    if (n == 0 && gates.shifted && threadIdx.x < 16)
      *reinterpret_cast<f4*>(gates.shifted + (long)bh * 64 + 4 * threadIdx.x) =
          *reinterpret_cast<const f4*>(mix.key + token_head(d, b, d.T - 1, h) * 64 +
                                       4 * threadIdx.x);
  } else {
    load_chunk_scalars(cs, d, beta, log_decay, b, h, n);
  }
  if (threadIdx.x < 64) {
    // The sub-chunks' weights, and the chunk's, as states_kernel stages them.
    const int s = threadIdx.x, cut = d.rsub == 2 ? min(d.sub, len) : len;
    const float p = cs.prefix[s], bt = cs.beta[s];  // this wave's own writes
    const float mid = read_lane(p, cut - 1), last = read_lane(p, 63);
    wt[0][s] = s < cut ? bt * expf(mid - p) : 0.f;
    wt[1][s] = s >= cut ? bt * expf(last - p) : 0.f;
    wt[2][s] = s < len ? bt * expf(read_lane(p, len - 1) - p) : 0.f;
  }
  if constexpr (MIX)
    rk.store_unit(K, mix.key_shift && !mix.previous && n == 0);
  else
    rk.store(K);
  rv0.store(V);
  if (d.NV > 1) rv1.store(V + TILE);
  __syncthreads();
  for (int u = 0; u < d.rsub; ++u) {
    const int first = sub_first(d, u), cnt = sub_len(d, n, u), end = cnt > 0 ? first + cnt : 0;
    f4 acc[4];
    zero4(acc);
    for (int k0 = first & ~15; k0 < end; k0 += 16) weighted_strip(acc, K, K, wt[u], k0, w);
    float* out = mat(start_s, (long)bh * d.NS + (long)n * d.rsub + u);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f4*>(out + acc_row(w, q) * 64 + c4) = quad_row(acc, q);
  }
  for (int v = 0; v < d.NV; ++v) {
    f4 acc[4];
    zero4(acc);
    for (int k0 = 0; k0 < len; k0 += 16) weighted_strip(acc, V + v * TILE, K, wt[2], k0, w);
    float* out = mat(start_c, ((long)bh * d.NC + n) * d.NV + v);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f4*>(out + acc_row(w, q) * 64 + c4) = quad_row(acc, q);
  }
}

// The decays of the scan's steps first .. first + count - 1 (count <= 64), the
// two sub-chunks of each chunk (parts = 2) or chunks (parts = 1), from the
// chunk's log-decay prefix as states_kernel takes them.  A 256-thread block: a
// wave per chunk and a token per lane, every load at once, then a thread per
// exponential (a wave per exponential had fwd_scan at 30 us, now 25, where B1
// T4096 H8 P64 gives it two times 64 steps).
struct StepSums {
  float mid[64], last[64];  // the prefix at the first sub-chunk's end and the chunk's
};
__device__ __forceinline__ void step_decays(float* decay, StepSums& sums, const Dims& d,
                                            const float* log_decay, int b, int h, int first,
                                            int count, int parts) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id();
  const int halves = parts - 1, n0 = first >> halves, chunks = count >> halves;
  const int tokens = min(chunks * d.chunk, d.T - n0 * d.chunk);
  // Tokens past the sequence and lanes past the chunk read zero.
  const BufRsrc rows = buf_rsrc(log_decay + token_head(d, b, n0 * d.chunk, h),
                                (unsigned)(tokens - 1) * d.H * 4 + 4);
  const unsigned step = (unsigned)d.chunk * d.H * 4;
  const unsigned token = l < d.chunk ? (unsigned)l * d.H * 4 : kNoRow;
  float g[16], mid = 0.f, last = 0.f;  // lane j: of the wave's chunk j
#pragma unroll
  for (int j = 0; j < 16; ++j) g[j] = buf_load1(rows, token + (w + 4 * j) * step);
#pragma unroll
  for (int j0 = 0; j0 < 16; j0 += 4) {
    if (4 * j0 >= chunks) break;
#pragma unroll
    for (int j = j0; j < j0 + 4; ++j) {
      const float p = wave_inclusive_sum(g[j]);
      const int cut = max(min(d.sub, chunk_len(d, n0 + w + 4 * j)), 1);
      float at_cut = read_lane(p, cut - 1), at_end = read_lane(p, 63);
      // Read here, so that the choices below stay selects (no branch per chunk).
      asm volatile("" : "+s"(at_cut), "+s"(at_end));
      mid = l == j ? at_cut : mid;
      last = l == j ? at_end : last;
    }
  }
  if (l < 16) {
    sums.mid[w + 4 * l] = mid;
    sums.last[w + 4 * l] = last;
  }
  __syncthreads();
  const int i = threadIdx.x, k = i >> halves;
  if (i < count)
    decay[i] = expf(parts == 1 ? sums.last[k] : i & 1 ? sums.last[k] - sums.mid[k] : sums.mid[k]);
}

// Steps of a scan whose loads are issued together.
constexpr int SCAN_BATCH = 8;

// Grid (B*H, 4 + 4 NV): y in 0..3 scans evidence elements [1024y, 1024y+1024)
// over the NS sub-chunks, y >= 4 the cross-statistic elements
// [1024(y-4), 1024(y-3)) of the NV * 4096 per state over NC chunks.
__global__ __launch_bounds__(256) void fwd_scan_kernel(
    Dims d, const float* __restrict__ log_decay, const float* __restrict__ init_s,
    const float* __restrict__ init_c, float* __restrict__ start_s, float* __restrict__ start_c,
    float* __restrict__ final_s, float* __restrict__ final_c) {
  const int bh = blockIdx.x, b = bh / d.H, h = bh % d.H;
  const bool cross = blockIdx.y >= 4;
  const int elem = 1024 * (cross ? blockIdx.y - 4 : blockIdx.y) + 4 * threadIdx.x;
  const int steps = cross ? d.NC : d.NS;
  const long size = cross ? 4096L * d.NV : 4096L;  // floats per state
  float* buf = (cross ? start_c : start_s) + (long)bh * steps * size;
  const float* init = cross ? init_c : init_s;
  __shared__ float decay[64];
  __shared__ StepSums sums;
  f4 running = f4{0.f, 0.f, 0.f, 0.f};
  if (init) running = *reinterpret_cast<const f4*>(init + (long)bh * size + elem);
  for (int base = 0; base < steps; base += 64) {
    const int count = min(64, steps - base);
    f4 stat[SCAN_BATCH];
    // Steps past the last read it again: no branch around a load.
    auto load = [&](int i0) {
#pragma unroll
      for (int j = 0; j < SCAN_BATCH; ++j)
        stat[j] = *reinterpret_cast<const f4*>(buf + (long)min(base + i0 + j, steps - 1) * size +
                                               elem);
    };
    load(0);
    __syncthreads();  // the previous steps' decays are read
    step_decays(decay, sums, d, log_decay, b, h, base, count, cross ? 1 : d.rsub);
    __syncthreads();
    for (int i0 = 0; i0 < count; i0 += SCAN_BATCH) {
      f4 cur[SCAN_BATCH];
#pragma unroll
      for (int j = 0; j < SCAN_BATCH; ++j) cur[j] = stat[j];
      if (i0 + SCAN_BATCH < count) load(i0 + SCAN_BATCH);
#pragma unroll
      for (int j = 0; j < SCAN_BATCH; ++j)
        if (i0 + j < count) {
          *reinterpret_cast<f4*>(buf + (long)(base + i0 + j) * size + elem) = running;
          running = fma4(decay[i0 + j], running, cur[j]);
        }
    }
  }
  float* fin = cross ? final_c : final_s;
  *reinterpret_cast<f4*>(fin + (long)bh * size + elem) = running;
}

// One block per chunk, loads and weights as in fwd_stats_kernel.  GATE: d_output
// is the gated output's cotangent, each token's weighed by its read gate.
template <bool GATE>
__global__ __launch_bounds__(256) void bwd_local_kernel(
    Dims d, const float* __restrict__ beta, const float* __restrict__ log_decay,
    const float* __restrict__ solved, const float* __restrict__ z,
    const float* __restrict__ d_output, float* __restrict__ end_s, float* __restrict__ end_c,
    const float* __restrict__ variance, const float* __restrict__ confidence_scale) {
  extern __shared__ float smem[];
  float* Y = smem;
  float* Z = Y + TILE;
  float* D = Z + TILE;
  float* M = D + TILE;
  __shared__ ChunkScalars cs;
  __shared__ alignas(16) float wt[MAXC], wt_cross[MAXC];
  const long seq = blockIdx.x;
  const int n = (int)(seq % d.NC), bh = (int)(seq / d.NC), b = bh / d.H, h = bh % d.H;
  const int len = chunk_len(d, n), w = threadIdx.x >> 6, c4 = 4 * (lane_id() & 15);
  const long row = token_head(d, b, n * d.chunk, h);
  RowTile<float> ry, rz, rd0, rd1;
  ry.fetch_tokens(len, solved + row * 64, (unsigned)(d.H * 64));
  rz.fetch_tokens(len, z + row * 64, (unsigned)(d.H * 64));
  rd0.fetch_tokens(len, d_output + row * d.P, (unsigned)(d.H * d.P));
  rd1.fetch_tokens(d.NV > 1 ? len : 0, d_output + row * d.P + (d.NV > 1 ? 64 : 0),
                   (unsigned)(d.H * d.P));
  load_chunk_scalars(cs, d, beta, log_decay, b, h, n);
  if (threadIdx.x < 64) {
    const int s = threadIdx.x;
    const float e = s < len ? expf(cs.prefix[s]) : 0.f;
    wt[s] = e;
    wt_cross[s] = e;
    if (GATE && s < len)
      wt_cross[s] = read_gate(confidence_scale[h], variance[row + (long)s * d.H]) * e;
  }
  ry.store(Y);
  rz.store(Z);
  rd0.store(D);
  __syncthreads();
  auto store_cross = [&](const f4 (&acc)[4], int v) {
    float* uc = mat(end_c, ((long)bh * d.NC + n) * d.NV + v);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f4*>(uc + acc_row(w, q) * 64 + c4) = quad_row(acc, q);
  };
  f4 acc[4], cross[4];
  zero4(acc);
  for (int k0 = 0; k0 < len; k0 += 16) weighted_strip(acc, Z, Y, wt, k0, w);  // sum_t e^P z_t y_t^T
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<f4*>(M + acc_row(w, q) * LDT + c4) = quad_row(acc, q);
  zero4(cross);
  for (int k0 = 0; k0 < len; k0 += 16) weighted_strip(cross, D, Y, wt_cross, k0, w);  // e^P dout y^T
  store_cross(cross, 0);
  __syncthreads();  // M is whole, and Z and D are read
  if (d.NV > 1) rd1.store(Z);
  float* us = mat(end_s, (long)bh * d.NC + n);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = acc_row(w, q);
    f4 v;
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) v[jb] = -(acc[jb][q] + M[(c4 + jb) * LDT + i]);
    *reinterpret_cast<f4*>(us + i * 64 + c4) = v;
  }
  if (d.NV > 1) {
    __syncthreads();
    zero4(cross);
    for (int k0 = 0; k0 < len; k0 += 16) weighted_strip(cross, Z, Y, wt_cross, k0, w);
    store_cross(cross, 1);
  }
}

// Grid (B*H, 4 + 4 NV) as fwd_scan_kernel, walking chunks in reverse.
__global__ __launch_bounds__(256) void bwd_scan_kernel(
    Dims d, const float* __restrict__ log_decay, const float* __restrict__ d_final_s,
    const float* __restrict__ d_final_c, float* __restrict__ end_s, float* __restrict__ end_c,
    float* __restrict__ d_init_s, float* __restrict__ d_init_c) {
  const int bh = blockIdx.x, b = bh / d.H, h = bh % d.H;
  const bool cross = blockIdx.y >= 4;
  const int elem = 1024 * (cross ? blockIdx.y - 4 : blockIdx.y) + 4 * threadIdx.x;
  const long size = cross ? 4096L * d.NV : 4096L;  // floats per state
  float* buf = (cross ? end_c : end_s) + (long)bh * d.NC * size;
  const float* fin = cross ? d_final_c : d_final_s;
  __shared__ float decay[64];
  __shared__ StepSums sums;
  // Evidence: the scan carries G + G^T (it starts from D + D^T and adds the
  // local terms 2U = -(M + M^T), as bwd_local_kernel stores them), so every
  // stored end-state cotangent is symmetric; the initial-state gradient is
  // the full one, half the carried sum plus the decayed antisymmetric part
  // of D.  Cross states carry their cotangent as is.
  f4 running = f4{0.f, 0.f, 0.f, 0.f}, anti = f4{0.f, 0.f, 0.f, 0.f};
  float total = 1.f;  // the product of every chunk's decay
  if (fin) {
    running = *reinterpret_cast<const f4*>(fin + (long)bh * size + elem);
    if (!cross) {
      const int i = elem >> 6, j = elem & 63;
      f4 tr;
#pragma unroll
      for (int e = 0; e < 4; ++e) tr[e] = fin[(long)bh * size + (j + e) * 64 + i];
      anti = 0.5f * (running - tr);
      running += tr;
    }
  }
  for (int top = d.NC; top > 0; top -= 64) {
    const int count = min(64, top), low = top - count;  // chunks low .. top - 1
    f4 local[SCAN_BATCH];
    auto load = [&](int i0) {
#pragma unroll
      for (int j = 0; j < SCAN_BATCH; ++j)
        local[j] = *reinterpret_cast<const f4*>(buf + (long)(low + max(i0 - j, 0)) * size + elem);
    };
    load(count - 1);
    __syncthreads();  // the previous steps' decays are read
    step_decays(decay, sums, d, log_decay, b, h, low, count, 1);
    __syncthreads();
    for (int i0 = count - 1; i0 >= 0; i0 -= SCAN_BATCH) {
      f4 cur[SCAN_BATCH];
#pragma unroll
      for (int j = 0; j < SCAN_BATCH; ++j) cur[j] = local[j];
      if (i0 - SCAN_BATCH >= 0) load(i0 - SCAN_BATCH);
#pragma unroll
      for (int j = 0; j < SCAN_BATCH; ++j)
        if (i0 - j >= 0) {
          *reinterpret_cast<f4*>(buf + (long)(low + i0 - j) * size + elem) = running;
          running = fma4(decay[i0 - j], running, cur[j]);
          total *= decay[i0 - j];
        }
    }
  }
  float* dinit = cross ? d_init_c : d_init_s;
  if (!cross) running = fma4(total, anti, 0.5f * running);
  *reinterpret_cast<f4*>(dinit + (long)bh * size + elem) = running;
}

// ---------------------------------------------------------------------------
// Fused statistics and carry, for batches with enough (b, h) sequences to
// fill the chip.  One 512-thread block walks one state sequence of one (b, h)
// chunk by chunk, keeping the carried state in its MFMA accumulators:
// blockIdx.y 0 is the evidence, y = 1 + v cross tile v.  Each chunk (each
// sub-chunk, for the forward evidence) stores the state it starts from, then
// takes state = decay * state + sum_t wt_t a_t b_t^T over its tokens; the
// statistics never go through HBM.
//   forward:  a = key (evidence) or value tile, b = key,
//             wt = beta_t exp(P_last - P_t);  states ascend from init.
//   backward: evidence a, b = (z, y) with wt = -exp(P_t), the product added
//             with its transpose; cross a = d_output tile, b = y with wt =
//             exp(P_t) (MIX: the read gate g_t exp(P_t), d_output being the
//             cotangent of the mixer's gated output g_t read_t + skip
//             value_t);  states descend from the final-state cotangent (the
//             transpose of the forward carry, as bwd_local_kernel +
//             bwd_scan_kernel).
// A step's product is summed from zero and added to the decayed state by one
// multiply-add, as the scans of the chunk-parallel pair add it.
// A step's rows load into registers two steps before it multiplies.  NBUF =
// 2: LDS holds two step buffers and each step takes one barrier (the next
// step staged while this one multiplies).  NBUF = 1: one buffer, staged
// between two barriers, half the LDS, so three blocks fit a CU instead of
// two; the launch takes it when the walks would not fit the chip at two per
// CU (the extra resident blocks beat the exposed staging there).
// Wave w computes rows 16 (w % 4) .. +15 and column quads' halves w / 4 of
// the 64x64 state tile.

constexpr int STATES_THREADS = 512;

// One chunk step in LDS: per part (the forward evidence's sub-chunks, else
// the whole chunk) the token weights, zero outside the part, the decay over
// the part and its token range [lo, hi).
struct alignas(16) StepBuffer {  // wt is read as float4
  float wt[2][MAXC];
  float decay[2];
  int lo[2], hi[2];
};

// acc += (A diag(wt))^T-by-B over k in [k0, k0 + 16) for rows 16 s.. of the
// result and its columns 4r + 2hf + j (j = 0, 1): A(i, k) = A[k][16s + i]
// wt[k], B(k, c) = B[k][c] (the tile_mma_half QUAD convention).  FIRST: from
// zero, whatever acc holds.
template <bool FIRST>
__device__ __forceinline__ void weighted_block(f4 acc[2], const float* A, const float* B,
                                               const float* wt, int k0, int s, int hf) {
  const int l = lane_id(), r = l & 15, kk = k0 + 4 * (l >> 4);
  const f4 t = *reinterpret_cast<const f4*>(wt + kk);
  f4 a;
#pragma unroll
  for (int e = 0; e < 4; ++e) a[e] = A[(kk + e) * LDT + 16 * s + r] * t[e];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float2 b = *reinterpret_cast<const float2*>(B + (kk + e) * LDT + 4 * r + 2 * hf);
    const bool zero = FIRST && e == 0;
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b.x, zero ? f4{} : acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b.y, zero ? f4{} : acc[1], 0, 0, 0);
  }
}

// In: element type of the forward's key and value rows (the backward's rows
// are float32).
// The one-buffer backward walk is held to six waves per SIMD (three blocks
// per CU, as its LDS allows), a budget of 80 VGPRs at which the compiler
// may spill to per-lane scratch (it fits today); the two-buffer walks have
// room to spare.
template <bool BWD, typename In, bool MIX, int NBUF>
__global__ __launch_bounds__(STATES_THREADS)
__attribute__((amdgpu_waves_per_eu(NBUF == 1 && BWD ? 6 : 1))) void states_kernel(Dims d,
                                                                                  StateArgs g) {
  // MIX: the forward's keys come from the mixer's raw projections; the
  // backward's cross weights take the mixer's read gate.
  constexpr bool MIX_KEYS = MIX && !BWD, GATED = MIX && BWD;
  const In* rows_a = static_cast<const In*>(g.rows_a);
  const In* rows_ac = static_cast<const In*>(g.rows_ac);
  const In* rows_b = static_cast<const In*>(g.rows_b);
  extern __shared__ float smem[];  // buffer u: b tile at 2u TILE, a tile at (2u + 1) TILE
  __shared__ StepBuffer sb[2];
  const int bh = blockIdx.x, b = bh / d.H, h = bh % d.H;
  const bool cross = blockIdx.y > 0;
  const int v = cross ? (int)blockIdx.y - 1 : 0;
  // The forward evidence stores a state per sub-chunk: its chunk steps have
  // rsub parts.
  const int parts = !BWD && !cross ? d.rsub : 1;
  const int steps = d.NC;
  // Evidence a rows: the keys themselves (forward) or z (backward).
  const bool own_a = cross || BWD;
  const int w = threadIdx.x >> 6, s = w & 3, hf = w >> 2, l = lane_id();
  const int elem = (16 * s + 4 * (l >> 4)) * 64 + 4 * (l & 15) + 2 * hf;  // + 64 q + j

  // The state stored before part `part` of chunk n.
  auto state_index = [&](int n, int part) {
    return cross ? ((long)bh * d.NC + n) * d.NV + v : ((long)bh * d.NC + n) * parts + part;
  };
  const long edge = cross ? (long)bh * d.NV + v : bh;

  // MIX forward: the head's gate parameters, loaded once (the gates are
  // computed per step on the walk's critical path).
  // The backward's gated cross walk: the head's confidence scale.
  float rate = 0.f, dt_bias = 0.f, beta_bias = 0.f, cscale = 0.f;
  if constexpr (GATED) cscale = g.confidence_scale[h];
  if constexpr (MIX_KEYS) {
    rate = expf(g.gates.a_log[h]);
    dt_bias = g.gates.dt_bias[h];
    beta_bias = g.gates.beta_bias[h];
    // The evidence walks of batch row 0 write their head's floor; each
    // evidence walk its (b, h)'s shifted key.
    if (!cross && b == 0 && threadIdx.x < 64)
      g.gates.floor[h * 64 + threadIdx.x] =
          g.gates.floor_min + mix_softplus(g.gates.floor_raw[h * 64 + threadIdx.x]);
    if (!cross && g.gates.shifted && threadIdx.x < 16)
      *reinterpret_cast<f4*>(g.gates.shifted + ((long)b * d.H + h) * 64 + 4 * threadIdx.x) =
          *reinterpret_cast<const f4*>(g.mix.key + token_head(d, b, d.T - 1, h) * 64 +
                                       4 * threadIdx.x);
  }
  f4 acc[2];
  zero2(acc);
  if (const float* first = cross ? g.first_c : g.first_s) {
    const float* src = first + edge * 4096 + elem;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float2 x = *reinterpret_cast<const float2*>(src + 64 * q);
      acc[0][q] = x.x;
      acc[1][q] = x.y;
    }
  }
  // The backward evidence walk carries G + G^T: it starts from D + D^T, D the
  // final-state cotangent (which need not be symmetric), and adds each step's
  // product with its transpose, which comes back through an LDS tile.  Every
  // chunk end state is then exactly symmetric, and the chunk gradients use
  // nothing else of it; the initial-state gradient is half the last one plus
  // the decayed antisymmetric part of D (dscale the decay), D read again at
  // the end.  A step's product goes to the tile before the barrier that ends
  // the reads of its step buffer and is added after it (add_own; one tile per
  // step buffer).  Both step buffer counts do this, so a batch's rows give the
  // same bits whichever variant the batch size selects.  The one-buffer walk
  // is held to 80 VGPRs for three blocks per CU.
  const bool sym = BWD && !cross;
  const int r0 = 16 * s + 4 * (l >> 4), c0 = 4 * (l & 15) + 2 * hf;  // elem's row and column
  float dscale = 1.f;
  const float* const d_final = sym && g.first_s ? g.first_s + edge * 4096 : nullptr;
  if (d_final)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[j] += *reinterpret_cast<const f4*>(d_final + (c0 + j) * 64 + r0);
  float* const tr = smem + 2 * NBUF * TILE;  // the transpose tiles (backward only)
  f4 own[2];        // the part's product,
  float own_decay;  // and its decay
  auto add_own = [&](int u) {
    if (!sym) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      own[j] += *reinterpret_cast<const f4*>(tr + u * TILE + (c0 + j) * LDT + r0);
      acc[j] = fma4(own_decay, acc[j], own[j]);
    }
    dscale *= own_decay;
  };
  // The state this lane holds (rows r0 + q, columns c0 + j), for dst
  // (+ 64 q + j).
  auto state_now = [&](float2 (&out)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) out[q] = float2{acc[0][q], acc[1][q]};
  };
  auto store_state = [&](const float2 (&v)[4], float* dst) {
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<float2*>(dst + 64 * q) = v[q];
  };
  // The state after the last step (the backward evidence's initial-state
  // gradient).
  auto put_state = [&](float* dst) {
    if (sym) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f4 anti = f4{0.f, 0.f, 0.f, 0.f};
        if (d_final) {
#pragma unroll
          for (int q = 0; q < 4; ++q) anti[q] = d_final[elem + 64 * q + j];
          anti = 0.5f * (anti - *reinterpret_cast<const f4*>(d_final + (c0 + j) * 64 + r0));
        }
        acc[j] = fma4(dscale, anti, 0.5f * acc[j]);
      }
    }
    float2 v[4];
    state_now(v);
    store_state(v, dst);
  };
  // A step's start states (one per part), taken before its products and
  // stored after its staging: the staging's waits for the loads issued a step
  // earlier then come before these stores in issue order, so they never
  // wait for a store (the wait counter retires loads and stores in order).
  // (parts <= 2: the forward evidence's two sub-chunks, else one; the two
  // sets are named, not indexed, so they stay in registers.)
  float2 held0[4], held1[4];
  int held_i = 0;  // the step the held states start
  auto store_held = [&]() {
    float* base = cross ? g.steps_c : g.steps_s;
    store_state(held0, base + state_index(held_i, 0) * 4096 + elem);
    if (parts == 2) store_state(held1, base + state_index(held_i, 1) * 4096 + elem);
  };

  // Rows and scalars of one step on their way from HBM to LDS.  Two sets
  // rotate, so a step's loads are issued two steps before it multiplies.
  struct StepRegs {
    RowTile<In, STATES_THREADS> ra, rb;
    float pg, pb;
  };
  // MIX (forward): the b rows are the keys from the mixer's raw projections
  // (shifted; position 0's zero row reads its query row and is zeroed at
  // staging), normalised at staging.
  const MixerIn& mix = g.mix;
  // Every step issues the same loads: a step past the walk's end (i outside
  // 0 .. steps - 1) loads with no rows in range (zeros, no memory access), so
  // the compiler can count the memory operations in flight and each wait
  // retires only what it needs.
  auto fetch = [&](StepRegs& R, int i) {
    const bool valid = i >= 0 && i < steps;
    const int ic = valid ? i : 0;
    const int first = ic * d.chunk, cnt = valid ? chunk_len(d, ic) : 0;
    if constexpr (MIX_KEYS) {
      R.rb.fetch_mix_keys(cnt, mix, d, b, h, first);
    } else {
      R.rb.fetch_tokens(cnt, rows_b + token_head(d, b, first, h) * 64, (unsigned)d.H * 64);
    }
    {
      // (The forward evidence walk has no a rows: no rows in range.)
      const int width = cross ? d.P : 64, offset = cross ? 64 * v : 0;
      R.ra.fetch_tokens(own_a ? cnt : 0,
                        (cross ? rows_ac : rows_a) + token_head(d, b, first, h) * width + offset,
                        (unsigned)(d.H * width));
    }
    // Wave 0's lane l: token l's log decay and beta (zero past the chunk; the
    // other waves read out of range).  MIX forward: their raw projections
    // dt_raw and beta_raw; the backward's gated cross walk: the variance in
    // place of beta.
    const long th = token_head(d, b, first, h);
    const unsigned bytes = cnt > 0 ? (unsigned)(cnt - 1) * d.H * 4 + 4 : 0;
    const unsigned off = w == 0 ? (unsigned)l * d.H * 4 : kNoRow;
    R.pg = buf_load1(buf_rsrc((MIX_KEYS ? g.gates.dt_raw : g.log_decay) + th, bytes), off);
    const float* pb_src = BWD ? g.variance : MIX_KEYS ? g.gates.beta_raw : g.beta;
    R.pb = BWD && !(GATED && cross) ? 0.f : buf_load1(buf_rsrc(pb_src + th, bytes), off);
  };
  auto stage = [&](const StepRegs& R, int u, int i) {
    if constexpr (MIX_KEYS)
      R.rb.store_unit(smem + 2 * u * TILE, mix.key_shift && !mix.previous && i == 0);
    else
      R.rb.store(smem + 2 * u * TILE);
    if (own_a) R.ra.store(smem + (2 * u + 1) * TILE);
    if (w == 0) {
      const int cnt = chunk_len(d, i), cut = parts == 2 ? min(d.sub, cnt) : cnt;
      float pg = R.pg, pb = R.pb;
      if constexpr (MIX_KEYS) {
        // The gates from their raw projections (zero past the chunk); the
        // evidence walk writes them out for the factor and read kernels.
        const bool in = l < cnt;
        // mix_log_decay and mix_beta with the head's parameters preloaded.
        pg = in ? -rate * mix_softplus(R.pg + dt_bias) : 0.f;
        pb = in ? g.gates.beta_max * mix_sigmoid(R.pb + beta_bias) : 0.f;
        if (!cross && in) {
          const long th = token_head(d, b, i * d.chunk + l, h);
          g.gates.log_decay[th] = pg;
          g.gates.beta[th] = pb;
        }
      }
      // Inclusive log-decay prefix over the chunk; part 0 ends at token
      // `cut` - 1 (the sub-chunk boundary, or the chunk end).
      const float p = wave_inclusive_sum(pg), last = read_lane(p, 63);
      const float mid = cut > 0 ? read_lane(p, cut - 1) : 0.f;  // cut is uniform
      if (BWD) {
        float c = cross ? 1.f : -1.f;
        if (GATED && cross) c = read_gate(cscale, pb);
        sb[u].wt[0][l] = c * expf(p);
      } else {
        sb[u].wt[0][l] = l < cut ? pb * expf(mid - p) : 0.f;
        sb[u].wt[1][l] = l >= cut ? pb * expf(last - p) : 0.f;
      }
      if (l == 0) {
        sb[u].decay[0] = expf(parts == 2 ? mid : last);
        sb[u].decay[1] = expf(last - mid);
        sb[u].lo[0] = 0;
        sb[u].hi[0] = cut;
        sb[u].lo[1] = cut;
        sb[u].hi[1] = cnt;
      }
    }
  };

  const int i0 = BWD ? steps - 1 : 0, stride = BWD ? -1 : 1;
  // Step k's products on LDS buffer u.
  auto multiply = [&](int k, int u) {
    const int i = i0 + k * stride;
    const float* tb = smem + 2 * u * TILE;
    const float* ta = own_a ? smem + (2 * u + 1) * TILE : tb;
    held_i = i;
    // 16-token blocks that hold a part's tokens; the weights are zero outside
    // the part (an empty part takes one block of zeros).
    auto product = [&](int part, f4 (&sum)[2]) {
      const int lo = sb[u].lo[part], hi = lo < sb[u].hi[part] ? sb[u].hi[part] : 0;
      const float* wt = sb[u].wt[part];
      int k0 = lo & ~15;
      weighted_block<true>(sum, ta, tb, wt, k0, s, hf);
      for (k0 += 16; k0 < hi; k0 += 16) weighted_block<false>(sum, ta, tb, wt, k0, s, hf);
    };
    auto one_part = [&](int part, float2 (&held)[4]) {
      state_now(held);
      product(part, own);
      own_decay = sb[u].decay[part];
      if (sym) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float2*>(tr + u * TILE + (r0 + q) * LDT + c0) =
              float2{own[0][q], own[1][q]};
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = fma4(own_decay, acc[j], own[j]);
      }
    };
    one_part(0, held0);
    if (parts == 2) one_part(1, held1);
  };
  if constexpr (NBUF == 1 && BWD) {
    // One register set, loaded one step ahead (the backward walk's 16 fewer
    // VGPRs keep three blocks per CU; the other blocks cover the shorter
    // lead).
    StepRegs R;
    fetch(R, i0);
    stage(R, 0, i0);
    __syncthreads();
    fetch(R, i0 + stride);
    for (int k = 0; k < steps; ++k) {
      multiply(k, 0);
      __syncthreads();  // every wave is done with the buffer
      add_own(0);
      if (k + 1 < steps) stage(R, 0, i0 + (k + 1) * stride);
      store_held();
      fetch(R, i0 + (k + 2) * stride);
      __syncthreads();
    }
  } else {
    StepRegs R0, R1;
    fetch(R0, i0);
    fetch(R1, i0 + stride);
    stage(R0, 0, i0);
    __syncthreads();
    // Step k multiplies LDS buffer k & 1 (NBUF = 2); `next` holds step k + 1
    // (staged at the end), `spare` (step k, already staged) receives step
    // k + 2.
    auto step = [&](int k, const StepRegs& next, StepRegs& spare) {
      const int i = i0 + k * stride, u = NBUF == 2 ? k & 1 : 0;
      fetch(spare, i + 2 * stride);
      if (BWD && k > 0) add_own(u ^ 1);
      multiply(k, u);
      if constexpr (NBUF == 2) {
        if (k + 1 < steps) stage(next, u ^ 1, i + stride);
      } else {
        __syncthreads();  // every wave is done with the buffer
        if (k + 1 < steps) stage(next, 0, i + stride);
      }
      store_held();
      __syncthreads();
    };
    // Two steps per iteration (the register sets alternate).  The first
    // iteration is peeled and an odd last step follows the loop, so the loop
    // is entered with the loads and stores in flight that each iteration
    // leaves and its body has no conditional loads: the compiler's count of
    // what is in flight at each wait stays exact.
    if (steps >= 2) {
      step(0, R1, R0);
      step(1, R0, R1);
      int k = 2;
      for (; k + 1 < steps; k += 2) {
        step(k, R1, R0);
        step(k + 1, R0, R1);
      }
      if (k < steps) step(k, R1, R0);
    } else {
      step(0, R1, R0);
    }
    if (BWD) add_own((steps - 1) & 1);
  }
  put_state((cross ? g.last_c : g.last_s) + edge * 4096 + elem);
}

#define M4_STATES(BWD, IN, MIX)                                          \
  template __global__ void states_kernel<BWD, IN, MIX, 1>(Dims, StateArgs); \
  template __global__ void states_kernel<BWD, IN, MIX, 2>(Dims, StateArgs);
M4_STATES(false, float, false)
M4_STATES(false, bf16_t, false)
M4_STATES(true, float, false)
M4_STATES(false, float, true)
M4_STATES(true, float, true)
#undef M4_STATES
#define M4_STATS_KERNEL(In, MIX)                                                              \
  template __global__ void fwd_stats_kernel<In, MIX>(Dims, const In*, const In*, const float*, \
                                                     const float*, float*, float*, MixerIn,    \
                                                     MixerGates);
M4_STATS_KERNEL(float, false)
M4_STATS_KERNEL(bf16_t, false)
M4_STATS_KERNEL(float, true)
template __global__ void bwd_local_kernel<false>(Dims, const float*, const float*, const float*,
                                                 const float*, const float*, float*, float*,
                                                 const float*, const float*);
template __global__ void bwd_local_kernel<true>(Dims, const float*, const float*, const float*,
                                                const float*, const float*, float*, float*,
                                                const float*, const float*);

}  // namespace m4
