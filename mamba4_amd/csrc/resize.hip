// Matrices copied between widths, several arrays in one launch: the memory
// read's 64-wide (64 or 128 for values) arrays from and to the caller's
// narrower ones.
//
// Bound by the launch at the sizes of a short call: padding six inputs one by
// one (a fill and a strided copy each) and narrowing their gradients took 22
// launches, 80 us of device time and more of the host's, at B2 T251 H3 D48
// P100; two launches of about 4 us do it here.  A thread copies four
// consecutive columns of the destination, stored together where the width
// allows, for one index division: B38 T469 H7 D42 50 us both ways (about 4.2
// TB/s), where one element a thread left the call 5% slower than separate
// fills and copies (78 us) had it.
#include "common.hpp"

namespace m4 {

template <typename E>
__device__ __forceinline__ void resize_four(const ResizeJob& job, long quad) {
  typedef E four __attribute__((ext_vector_type(4)));
  const unsigned quads = (unsigned)(job.dst_cols + 3) / 4;  // per row
  const long row = quad < (1L << 32) ? (long)((unsigned)quad / quads) : quad / quads;
  const int c = 4 * (int)(quad - row * quads);
  long from_row = row;
  bool in = true;
  if (job.dst_rows != 1 || job.src_rows != 1) {
    const long o = row / job.dst_rows, r = row - o * job.dst_rows;
    in = r < job.src_rows;
    from_row = o * job.src_rows + r;
  }
  const E* src = static_cast<const E*>(job.src) + (in ? from_row : 0) * job.src_cols;
  E v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const bool here = in && c + k < job.src_cols;
    v[k] = (E)job.fill;
    if (here) v[k] = src[c + k];
  }
  E* dst = static_cast<E*>(job.dst) + row * job.dst_cols + c;
  if (job.aligned) {
    *reinterpret_cast<four*>(dst) = four{v[0], v[1], v[2], v[3]};
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c + k < job.dst_cols) dst[k] = v[k];
  }
}

__global__ __launch_bounds__(256) void resize_kernel(ResizeJobs jobs) {
  long e = (long)blockIdx.x * 256 + threadIdx.x;
  // Every job's arguments are read by a constant index; the quads of the jobs
  // before this thread's are counted off.
#pragma unroll
  for (int j = 0; j < kResizeJobs; ++j) {
    if (j >= jobs.count) return;
    const ResizeJob& job = jobs.job[j];
    if (e < job.quads) {
      if (job.bytes == 4)
        resize_four<unsigned>(job, e);
      else
        resize_four<unsigned short>(job, e);
      return;
    }
    e -= job.quads;
  }
}

}  // namespace m4
