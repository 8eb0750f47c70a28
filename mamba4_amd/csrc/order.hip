// The order head's gated vector scan (lm/models/mamba4.py:46-95, called at
// :274-289): per batch row, head and channel,
//   h_t = lam_t h_(t-1) + (1 - lam_t) v_t,   lam_t = exp(log_decay_t),
// with the inflow 1 - lam_t taken as -expm1(log_decay_t) as the reference's
// chunked form does, from h_(-1) = initial (zero when absent).
//
// Layout: values and output [B,T,H,W], log_decay [B,T,H], initial and the
// initial-state gradient [B,H,W].  One thread per channel; a block covers
// every channel of one (b, h) and one chunk of 64 tokens, two runs of 32, so
// a wave's access to a token is one contiguous row of up to 64 floats.  Three
// passes each way:
//   forward:  order_local  - each run's scan from zero: its end state and
//                            its decay;
//             order_carry  - the state every run starts from, run by run per
//                            (b, h, channel), in place;
//             order_apply  - each run's scan from its start state.
//   backward: the same three over the reverse recurrence of the cotangent
//             g_t = dout_t + lam_(t+1) g_(t+1): d v_t = (1 - lam_t) g_t,
//             d log_decay_t = lam_t sum_c g_t,c (h_(t-1),c - v_t,c) (summed
//             over channels in a fixed order), d initial = lam_0 g_0.
// Where enough (b, h) fill the chip, or the sequence is short, one kernel each
// way does the whole scan instead (order_walk, order_bwd_walk below).  Both
// forms take the same runs, multiply-adds and sums in the same order (which
// product of a step is rounded is spelled out), so a batch row has the same
// bits whichever form its batch size selects.
#include "common.hpp"

namespace m4 {

__device__ __forceinline__ long order_row(const OrderDims& d, int b, int t, int h) {
  return ((long)b * d.T + t) * d.H + h;
}

// Block (b, h, n) of a grid over B*H*NC chunks.
struct OrderBlock {
  int b, h, n, bh, t0, len;
};

__device__ __forceinline__ OrderBlock order_block(const OrderDims& d) {
  OrderBlock o;
  o.n = blockIdx.x % d.NC;
  o.bh = blockIdx.x / d.NC;
  o.b = o.bh / d.H;
  o.h = o.bh % d.H;
  o.t0 = o.n * MAXC;
  o.len = min(MAXC, d.T - o.t0);
  return o;
}

// The per-chunk kernels walk their chunk in groups of ORDER_GROUP tokens, a
// group's loads issued before the previous group is used, every load
// unconditional (tokens past the chunk's length re-read its last row and are
// then masked to value 0).  A token's decay and inflow are the same for every
// channel: lane l computes them for the chunk's token l once (zero log decay
// past the chunk's end, which leaves the scan as it is), and each step reads
// them from that lane.
// The grids hold about one wave per chunk, a few per SIMD: the kernels are
// built for two waves per SIMD, so the scheduler keeps the group loads
// ahead of their use instead of minimising registers.
constexpr int ORDER_GROUP = 16;
constexpr int ORDER_GROUPS = MAXC / ORDER_GROUP;
constexpr int ORDER_RUN = MAXC / 2;
constexpr int ORDER_RUN_GROUPS = ORDER_RUN / ORDER_GROUP;

struct RowGroup {
  float x[ORDER_GROUP];
};

// Loads group `g` of channel c from `rows` (W-float rows): the chunk's row t
// is at first[t * stride] with first = &rows[chunk's first row][c] and
// stride = H W; tokens past the chunk re-read its last row.
__device__ __forceinline__ void load_group(RowGroup& r, const OrderBlock& o, int g,
                                           const float* first, long stride) {
#pragma unroll
  for (int i = 0; i < ORDER_GROUP; ++i)
    r.x[i] = first[min(g * ORDER_GROUP + i, o.len - 1) * stride];
  // Keep the group's loads here, ahead of the previous group's use (the
  // scheduler would otherwise sink each load next to its use).
  __builtin_amdgcn_sched_barrier(0);
}

// Per-token gate of the chunk held by lane l = token l: the log decay (0
// past the chunk), lam = exp and the inflow 1 - lam = -expm1.
struct TokenGates {
  float lg, lam, inflow;

  __device__ __forceinline__ TokenGates(const OrderDims& d, const OrderBlock& o,
                                        const float* log_decay) {
    const int l = lane_id();
    lg = l < o.len ? log_decay[order_row(d, o.b, o.t0 + min(l, o.len - 1), o.h)] : 0.f;
    lam = expf(lg);
    inflow = -expm1f(lg);
  }
  // The decay over the chunk's run k (every lane receives it).
  __device__ __forceinline__ float total(int k) const {
    return expf(group4_sum(row16_sum(lane_id() / ORDER_RUN == k ? lg : 0.f)));
  }
};

__device__ __forceinline__ float lane_value(float x, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// One step of the scan.
__device__ __forceinline__ float order_step(float lam, float s, float inflow, float v) {
  return __builtin_fmaf(lam, s, inflow * v);
}

// Forward pass 1: ends[bh][run][c] = the run's scan from zero at its last
// token; totals[bh][run] = its decay.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void order_local_kernel(OrderDims d, const float* values,
                                                          const float* log_decay, float* ends,
                                                          float* totals) {
  const OrderBlock o = order_block(d);
  const int c = threadIdx.x, cc = min(c, d.W - 1);
  const TokenGates gate(d, o, log_decay);
  const float decay[2] = {gate.total(0), gate.total(1)};
  const long stride = (long)d.H * d.W;
  const float* first = values + order_row(d, o.b, o.t0, o.h) * d.W + cc;
  RowGroup r[2];
  load_group(r[0], o, 0, first, stride);
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < ORDER_GROUPS; ++k) {
    if (k + 1 < ORDER_GROUPS) load_group(r[(k + 1) & 1], o, k + 1, first, stride);
#pragma unroll
    for (int i = 0; i < ORDER_GROUP; ++i) {
      const int t = k * ORDER_GROUP + i;
      s = order_step(lane_value(gate.lam, t), s, lane_value(gate.inflow, t), r[k & 1].x[i]);
    }
    if ((k + 1) % ORDER_RUN_GROUPS == 0) {  // a run is done
      const int half = k / ORDER_RUN_GROUPS, run = 2 * o.n + half;
      const long slot = (long)o.bh * d.NR + run;
      if (run < d.NR) {
        if (c < d.W) ends[slot * d.W + c] = s;
        if (c == 0) totals[slot] = decay[half];
      }
      s = 0.f;
    }
  }
}

// Runs of a carry whose loads are issued together.
constexpr int ORDER_CARRY_BATCH = 16;

// The n-th run a carry comes to: from the first one, or from the last.
template <bool REVERSE>
__device__ __forceinline__ int carry_run(const OrderDims& d, int n) {
  return REVERSE ? d.NR - 1 - n : n;
}

// A batch of runs' own states of one coordinate and decays (past the last
// run: that run's again).
template <bool REVERSE>
struct CarryBatch {
  float local[ORDER_CARRY_BATCH], decay[ORDER_CARRY_BATCH];
  __device__ __forceinline__ void load(const OrderDims& d, const float* states,
                                       const float* totals, int n0) {
#pragma unroll
    for (int j = 0; j < ORDER_CARRY_BATCH; ++j) {
      const int run = carry_run<REVERSE>(d, min(n0 + j, d.NR - 1));
      local[j] = states[(long)run * d.W];
      decay[j] = totals[run];
    }
  }
  // Replaces the states of `count` runs from n0 by the carried ones.
  __device__ __forceinline__ float apply(const OrderDims& d, float* states, int n0, int count,
                                         float s) const {
#pragma unroll
    for (int j = 0; j < ORDER_CARRY_BATCH; ++j)
      if (j < count) {
        states[(long)carry_run<REVERSE>(d, n0 + j) * d.W] = s;
        s = __builtin_fmaf(decay[j], s, local[j]);
      }
    return s;
  }
};

// Carries one coordinate's state through a sequence's runs, in place.  Bound
// by the latency of its loads (few blocks, one dependent fma per run), so a
// batch is loaded while the one before it is carried; the last, which may be
// short, leaves the loop, so that no wait in it has to allow for fewer stores.
template <bool REVERSE>
__device__ __forceinline__ float carry_runs(const OrderDims& d, float* states,
                                            const float* totals, float s) {
  constexpr int N = ORDER_CARRY_BATCH;
  CarryBatch<REVERSE> a, b;
  a.load(d, states, totals, 0);
  for (int n0 = 0;; n0 += 2 * N) {
    b.load(d, states, totals, n0 + N);
    if (n0 + N > d.NR) return a.apply(d, states, n0, d.NR - n0, s);
    s = a.apply(d, states, n0, N, s);
    a.load(d, states, totals, n0 + 2 * N);
    if (n0 + 2 * N > d.NR) return b.apply(d, states, n0 + N, d.NR - n0 - N, s);
    s = b.apply(d, states, n0 + N, N, s);
  }
}

// Forward pass 2, grid B*H: turns ends into the state each run starts from
// (in place), starting from `initial`.
__global__ __launch_bounds__(256) void order_carry_kernel(OrderDims d, const float* initial,
                                                          float* ends, const float* totals) {
  const long bh = blockIdx.x;
  const int c = threadIdx.x;
  if (c >= d.W) return;
  carry_runs<false>(d, ends + bh * d.NR * d.W + c, totals + bh * d.NR,
                    initial ? initial[bh * d.W + c] : 0.f);
}

// Forward pass 3: each run's scan from its start state.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void order_apply_kernel(OrderDims d, const float* values,
                                                          const float* log_decay,
                                                          const float* starts, float* output) {
  const OrderBlock o = order_block(d);
  const int c = threadIdx.x, cc = min(c, d.W - 1);
  const TokenGates gate(d, o, log_decay);
  const long stride = (long)d.H * d.W;
  const float* first = values + order_row(d, o.b, o.t0, o.h) * d.W + cc;
  RowGroup r[2];
  load_group(r[0], o, 0, first, stride);
  const float* start = starts + (long)o.bh * d.NR * d.W + cc;
  const float next = start[(long)min(2 * o.n + 1, d.NR - 1) * d.W];
  float s = start[2L * o.n * d.W];
  float* out = output + order_row(d, o.b, o.t0, o.h) * d.W + c;
#pragma unroll
  for (int k = 0; k < ORDER_GROUPS; ++k) {
    if (k + 1 < ORDER_GROUPS) load_group(r[(k + 1) & 1], o, k + 1, first, stride);
    if (k == ORDER_RUN_GROUPS) s = next;
#pragma unroll
    for (int i = 0; i < ORDER_GROUP; ++i) {
      const int t = k * ORDER_GROUP + i;
      s = order_step(lane_value(gate.lam, t), s, lane_value(gate.inflow, t), r[k & 1].x[i]);
      if (t < o.len && c < d.W) out[t * stride] = s;
    }
  }
}

// Backward pass 1: each run's reverse scan of the cotangent from zero;
// heads[bh][run][c] = lam_first g_first (what reaches the previous run),
// totals[bh][run] = the run's decay.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void order_bwd_local_kernel(OrderDims d, const float* d_output,
                                                              const float* log_decay,
                                                              float* heads, float* totals) {
  const OrderBlock o = order_block(d);
  const int c = threadIdx.x, cc = min(c, d.W - 1);
  const TokenGates gate(d, o, log_decay);
  const float decay[2] = {gate.total(0), gate.total(1)};
  const long stride = (long)d.H * d.W;
  const float* first = d_output + order_row(d, o.b, o.t0, o.h) * d.W + cc;
  RowGroup r[2];
  load_group(r[1], o, ORDER_GROUPS - 1, first, stride);
  float g = 0.f, up = 1.f;  // g_(t+1) and its decay lam_(t+1)
#pragma unroll
  for (int k = ORDER_GROUPS - 1; k >= 0; --k) {
    if (k > 0) load_group(r[(k - 1) & 1], o, k - 1, first, stride);
#pragma unroll
    for (int i = ORDER_GROUP - 1; i >= 0; --i) {
      const int t = k * ORDER_GROUP + i;
      g = __builtin_fmaf(up, g, t < o.len ? r[k & 1].x[i] : 0.f);
      up = lane_value(gate.lam, t);
    }
    if (k % ORDER_RUN_GROUPS == 0) {  // a run is done
      const int half = k / ORDER_RUN_GROUPS, run = 2 * o.n + half;
      const long slot = (long)o.bh * d.NR + run;
      if (run < d.NR) {
        if (c < d.W) heads[slot * d.W + c] = up * g;
        if (c == 0) totals[slot] = decay[half];
      }
      g = 0.f;
      up = 1.f;
    }
  }
}

// Backward pass 2, grid B*H: heads become the cotangent reaching each run's
// last token from later runs (in place); what reaches the initial state is
// its gradient.
__global__ __launch_bounds__(256) void order_bwd_carry_kernel(OrderDims d, float* heads,
                                                              const float* totals,
                                                              float* d_initial) {
  const long bh = blockIdx.x;
  const int c = threadIdx.x;
  if (c >= d.W) return;
  const float s = carry_runs<true>(d, heads + bh * d.NR * d.W + c, totals + bh * d.NR, 0.f);
  if (d_initial) d_initial[bh * d.W + c] = s;
}

constexpr int ORDER_MAX_WAVES = 4;  // W <= 256

template <int CTRL>
__device__ __forceinline__ float order_dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}

// x[i] + x[i + half] exchanged with the lane whose bit `bit` differs, via a
// DPP pattern pairing exactly those lanes within a row: the lane with the
// bit set keeps (and sums) the upper element.
template <int CTRL, int BIT, int HALF>
__device__ __forceinline__ void dpp_stage(float (&x)[ORDER_RUN], int l) {
  const bool hi = (l >> BIT) & 1;
#pragma unroll
  for (int i = 0; i < HALF; ++i) {
    const float send = hi ? x[i] : x[i + HALF];
    const float keep = hi ? x[i + HALF] : x[i];
    x[i] = keep + order_dpp<CTRL>(send);
  }
}

// Sum over a wave's 64 lanes of x[0..31]: afterwards every lane holds the
// total of element l >> 1 (lane l).  A butterfly: each exchange halves the
// elements a lane keeps, selected by one lane bit.  Bits 5 and 4 exchange by
// v_permlane32_swap / v_permlane16_swap (the two results are the own and the
// partner's element of the kept half), bits 3..0 by DPP row_mirror (lane
// 15 - i), row_half_mirror (7 - i) and quad permutations, each pairing lanes
// that differ in that bit and agree in the bits above it.
__device__ __forceinline__ float wave_sums32(float (&x)[ORDER_RUN]) {
  const int l = lane_id();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[i]),
                                                    __float_as_uint(x[i + 16]), false, false);
    x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[i]),
                                                    __float_as_uint(x[i + 8]), false, false);
    x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  dpp_stage<0x140, 3, 4>(x, l);  // row_mirror
  dpp_stage<0x141, 2, 2>(x, l);  // row_half_mirror
  dpp_stage<0x4E, 1, 1>(x, l);   // quad_perm [2,3,0,1]
  return x[0] + order_dpp<0xB1>(x[0]);  // quad_perm [1,0,3,2]
}

// Backward pass 3: each run's reverse scan from the carried cotangent,
// d values, and d log_decay summed over channels (within each wave by the
// butterfly above, then over the waves in order).  h_(t-1) is rebuilt from the
// values and the one stored output before the run, as the one-pass kernel
// rebuilds it, and needs no pass over the outputs (B2 T4096 H16 W128: 43 us,
// 53 with one).  Both runs' rows load at once, the second run's first.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void order_bwd_apply_kernel(
    OrderDims d, const float* values, const float* log_decay, const float* initial,
    const float* output, const float* d_output, const float* carried, float* d_values,
    float* d_log_decay) {
  __shared__ float part[ORDER_MAX_WAVES][MAXC];
  const OrderBlock o = order_block(d);
  const int c = threadIdx.x, wave = c >> 6, l = lane_id();
  const bool on = c < d.W;
  const int cc = min(c, d.W - 1);
  const TokenGates gate(d, o, log_decay);
  struct Run {
    float dy[ORDER_RUN], v[ORDER_RUN], h, g;
  };
  Run r[2];
#pragma unroll
  for (int k = 1; k >= 0; --k) {
    const int t0 = o.t0 + ORDER_RUN * k;
    r[k].g = carried[((long)o.bh * d.NR + min(2 * o.n + k, d.NR - 1)) * d.W + cc];
    // The state before the run: the previous token's output, or the initial
    // state (zero when absent) before the first token.
    r[k].h = t0 > 0   ? output[order_row(d, o.b, min(t0, d.T) - 1, o.h) * d.W + cc]
             : initial ? initial[(long)o.bh * d.W + cc]
                       : 0.f;
#pragma unroll
    for (int i = 0; i < ORDER_RUN; ++i) {
      const long at = order_row(d, o.b, o.t0 + min(ORDER_RUN * k + i, o.len - 1), o.h) * d.W + cc;
      r[k].dy[i] = d_output[at];
      r[k].v[i] = values[at];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int k = 1; k >= 0; --k) {
    // v becomes h_(t-1) - v_t.
    float h = r[k].h, g = r[k].g, up = 1.f, term[ORDER_RUN];
#pragma unroll
    for (int i = 0; i < ORDER_RUN; ++i) {
      const int t = ORDER_RUN * k + i;
      const float v = r[k].v[i];
      r[k].v[i] = h - v;
      h = order_step(lane_value(gate.lam, t), h, lane_value(gate.inflow, t), v);
    }
#pragma unroll
    for (int i = ORDER_RUN - 1; i >= 0; --i) {
      const int t = ORDER_RUN * k + i;
      const bool in = t < o.len && on;
      g = __builtin_fmaf(up, g, t < o.len ? r[k].dy[i] : 0.f);
      if (in) d_values[order_row(d, o.b, o.t0 + t, o.h) * d.W + c] = lane_value(gate.inflow, t) * g;
      term[i] = in ? g * r[k].v[i] : 0.f;
      up = lane_value(gate.lam, t);
    }
    const float sum = wave_sums32(term);
    if ((l & 1) == 0) part[wave][ORDER_RUN * k + (l >> 1)] = sum;
  }
  __syncthreads();
  const int waves = (int)(blockDim.x >> 6);
  if (c < o.len) {  // wave 0: lane c holds token c's gate
    float sum = 0.f;
    for (int w = 0; w < waves; ++w) sum += part[w][c];
    d_log_decay[order_row(d, o.b, o.t0 + c, o.h)] = gate.lam * sum;
  }
}

// ---------------------------------------------------------------------
// The same scan with each value read once: one block per (b, h) holds
// WALK_TOKENS tokens of every channel in registers per wave, its waves
// covering consecutive runs of tokens (`groups` of them) times 64-channel
// columns.  Each step, every wave scans its run from zero, the runs' ends and
// total decays meet in LDS, and every wave takes its start state from them
// and scans its registers again, writing the results.  The backward also
// rebuilds h_(t-1) from the values and the one stored output before its run.
//
// Bound by HBM: 2 + 3 passes over the values' size instead of the three-pass
// kernels' 3 + 4 (B16 T1000 H12 W128: 40 us forward and 71 backward, 4.9 and
// 4.1 TB/s, against 61 and 95).  It needs a (b, h) per compute unit or so to
// fill the chip, the three-pass kernels a chunk (order_walks in the host code
// chooses).  The decays and the row offsets are scalars; some 60 of them
// overflow into lanes of vector registers.  (Stepping from row to row, so that
// none did, had the forward at 41 us instead of 39 on one card.)  Runs of 32
// tokens: the backward's two values per token fill the 128 vector registers
// that sixteen waves leave each lane, without scratch memory as long as its
// stores step from row to row (by offsets, 12 bytes a lane spilled).
constexpr int WALK_TOKENS = 32;
constexpr int WALK_MAX_WAVES = 16;

struct WalkWave {
  int bh, b, h, tg, groups, c, cc, l;
  bool on;

  __device__ __forceinline__ explicit WalkWave(const OrderDims& d) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), columns = (d.W + 63) >> 6;
    l = lane_id();
    bh = blockIdx.x;
    b = bh / d.H;
    h = bh % d.H;
    tg = wave / columns;
    groups = (int)(blockDim.x >> 6) / columns;
    c = (wave % columns) * 64 + l;
    on = c < d.W;
    cc = min(c, d.W - 1);
  }
};

// A run's gates: lane l < WALK_TOKENS holds token l (no decay and no inflow
// past the run's end, which leaves a scan as it is).
struct WalkGates {
  float lg, lam, inflow;

  __device__ __forceinline__ WalkGates(const OrderDims& d, const WalkWave& w, int t0, int len,
                                       const float* log_decay) {
    lg = w.l < len ? log_decay[order_row(d, w.b, t0 + w.l, w.h)] : 0.f;
    lam = expf(lg);
    inflow = -expm1f(lg);
  }
  // The run's decay (every lane receives it).
  __device__ __forceinline__ float total() const { return expf(group4_sum(row16_sum(lg))); }
};

__device__ __forceinline__ int run_len(const OrderDims& d, int t0) {
  return max(min(WALK_TOKENS, d.T - t0), 0);
}

// Rows t0.. of `rows` at this lane's channel, zeros past the run.
__device__ __forceinline__ void load_run(float (&x)[WALK_TOKENS], const OrderDims& d,
                                         const WalkWave& w, int t0, int len, const float* rows) {
  if (len == WALK_TOKENS) {
    const float* first = rows + order_row(d, w.b, t0, w.h) * d.W + w.cc;
    const long stride = (long)d.H * d.W;
#pragma unroll
    for (int i = 0; i < WALK_TOKENS; ++i) x[i] = first[i * stride];
  } else {
    const long last = max(min(t0 + len, d.T) - 1, 0);
#pragma unroll
    for (int i = 0; i < WALK_TOKENS; ++i) {
      const float v = rows[order_row(d, w.b, (int)min((long)t0 + i, last), w.h) * d.W + w.cc];
      x[i] = i < len ? v : 0.f;
    }
  }
}

__global__ __launch_bounds__(64 * WALK_MAX_WAVES) void order_walk_kernel(
    OrderDims d, const float* values, const float* log_decay, const float* initial,
    float* output) {
  __shared__ float ends[2][WALK_MAX_WAVES][64];
  __shared__ float decays[2][WALK_MAX_WAVES];
  const WalkWave w(d);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int columns = (d.W + 63) >> 6, column = wave % columns;
  const long stride = (long)d.H * d.W;
  float carry = initial ? initial[(long)w.bh * d.W + w.cc] : 0.f;
  int buf = 0;
  for (int base = 0; base < d.T; base += w.groups * WALK_TOKENS, buf ^= 1) {
    const int t0 = base + w.tg * WALK_TOKENS, len = run_len(d, t0);
    float x[WALK_TOKENS];
    load_run(x, d, w, t0, len, values);
    const WalkGates gate(d, w, t0, len, log_decay);
    float lam[WALK_TOKENS], s = 0.f;
#pragma unroll
    for (int i = 0; i < WALK_TOKENS; ++i) {
      lam[i] = lane_value(gate.lam, i);
      x[i] *= lane_value(gate.inflow, i);
      s = __builtin_fmaf(lam[i], s, x[i]);
    }
    ends[buf][wave][w.l] = s;
    decays[buf][wave] = gate.total();  // by every lane: its sum crosses lanes
    __syncthreads();
    s = carry;
    for (int j = 0; j < w.groups; ++j) {
      if (j == w.tg) s = carry;
      carry = __builtin_fmaf(decays[buf][j * columns], carry, ends[buf][j * columns + column][w.l]);
    }
    float* out = output + order_row(d, w.b, t0, w.h) * d.W + w.c;
    if (len == WALK_TOKENS && w.on) {
#pragma unroll
      for (int i = 0; i < WALK_TOKENS; ++i) {
        s = __builtin_fmaf(lam[i], s, x[i]);
        out[i * stride] = s;
      }
    } else {
#pragma unroll
      for (int i = 0; i < WALK_TOKENS; ++i) {
        s = __builtin_fmaf(lam[i], s, x[i]);
        if (i < len && w.on) out[i * stride] = s;
      }
    }
  }
}

__global__ __launch_bounds__(64 * WALK_MAX_WAVES) void order_bwd_walk_kernel(
    OrderDims d, const float* values, const float* log_decay, const float* initial,
    const float* output, const float* d_output, float* d_values, float* d_log_decay,
    float* d_initial) {
  static_assert(WALK_TOKENS == ORDER_RUN, "a run is one butterfly");
  __shared__ float heads[2][WALK_MAX_WAVES][64];
  __shared__ float decays[2][WALK_MAX_WAVES];
  __shared__ float part[2][WALK_MAX_WAVES][WALK_TOKENS];
  const WalkWave w(d);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int columns = (d.W + 63) >> 6, column = wave % columns;
  const long stride = (long)d.H * d.W;
  float carry = 0.f;  // the cotangent reaching the step's last token from later ones
  int buf = 0;
  const int span = w.groups * WALK_TOKENS;
  for (int base = (d.T - 1) / span * span; base >= 0; base -= span, buf ^= 1) {
    const int t0 = base + w.tg * WALK_TOKENS, len = run_len(d, t0);
    float dy[WALK_TOKENS], v[WALK_TOKENS];
    load_run(dy, d, w, t0, len, d_output);
    load_run(v, d, w, t0, len, values);
    float h = t0 > 0 ? output[order_row(d, w.b, min(t0, d.T) - 1, w.h) * d.W + w.cc]
              : initial ? initial[(long)w.bh * d.W + w.cc]
                        : 0.f;
    const WalkGates gate(d, w, t0, len, log_decay);
    float g = 0.f, up = 1.f;  // g_(t+1) and its decay lam_(t+1)
#pragma unroll
    for (int i = WALK_TOKENS - 1; i >= 0; --i) {
      g = __builtin_fmaf(up, g, dy[i]);
      up = lane_value(gate.lam, i);
    }
    heads[buf][wave][w.l] = up * g;
    decays[buf][wave] = gate.total();  // by every lane: its sum crosses lanes
    // v becomes h_(t-1) - v_t.
#pragma unroll
    for (int i = 0; i < WALK_TOKENS; ++i) {
      const float x = v[i];
      v[i] = h - x;
      h = order_step(lane_value(gate.lam, i), h, lane_value(gate.inflow, i), x);
    }
    __syncthreads();
    g = carry;
    for (int j = w.groups - 1; j >= 0; --j) {
      if (j == w.tg) g = carry;
      carry = __builtin_fmaf(decays[buf][j * columns], carry, heads[buf][j * columns + column][w.l]);
    }
    up = 1.f;
    float* dv = d_values + order_row(d, w.b, t0, w.h) * d.W + (WALK_TOKENS - 1) * stride;
    if (len == WALK_TOKENS && w.on) {
#pragma unroll
      for (int i = WALK_TOKENS - 1; i >= 0; --i, dv -= stride) {
        g = __builtin_fmaf(up, g, dy[i]);
        dv[w.c] = lane_value(gate.inflow, i) * g;
        v[i] *= g;
        up = lane_value(gate.lam, i);
      }
    } else {
#pragma unroll
      for (int i = WALK_TOKENS - 1; i >= 0; --i, dv -= stride) {
        const bool in = i < len && w.on;
        g = __builtin_fmaf(up, g, dy[i]);
        if (in) dv[w.c] = lane_value(gate.inflow, i) * g;
        v[i] = in ? g * v[i] : 0.f;
        up = lane_value(gate.lam, i);
      }
    }
    const float sum = wave_sums32(v);
    if (columns == 1) {
      const float mine = __shfl(sum, 2 * (w.l & 31));  // lane l < 32: token l
      if (w.l < len) d_log_decay[order_row(d, w.b, t0 + w.l, w.h)] = gate.lam * mine;
    } else {
      if ((w.l & 1) == 0) part[buf][wave][w.l >> 1] = sum;
      __syncthreads();
      if (column == 0 && w.l < len) {
        float all = 0.f;
        for (int j = 0; j < columns; ++j) all += part[buf][wave + j][w.l];
        d_log_decay[order_row(d, w.b, t0 + w.l, w.h)] = gate.lam * all;
      }
    }
  }
  if (d_initial && w.tg == 0 && w.on) d_initial[(long)w.bh * d.W + w.c] = carry;
}

}  // namespace m4
