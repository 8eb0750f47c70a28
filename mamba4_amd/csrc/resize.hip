// Matrices copied between widths, several arrays in one launch: the memory
// read's 64-wide (64 or 128 for values) arrays from and to the caller's
// narrower ones.
//
// Bound by the launch at the sizes of a short call: padding six inputs one by
// one (a fill and a strided copy each) and narrowing their gradients took 22
// launches, 80 us of device time and more of the host's, at B2 T251 H3 D48
// P100; two or three launches of about 4 us do it here.  A thread copies one
// element of the destination, so the writes are contiguous for every width
// and no alignment is assumed.
#include "common.hpp"

namespace m4 {

__global__ __launch_bounds__(256) void resize_kernel(ResizeJobs jobs) {
  long e = (long)blockIdx.x * 256 + threadIdx.x;
  // Every job's arguments are read by a constant index; the elements of the
  // jobs before this thread's are counted off.
#pragma unroll
  for (int j = 0; j < kResizeJobs; ++j) {
    if (j >= jobs.count) return;
    const ResizeJob& job = jobs.job[j];
    if (e >= 0 && e < job.elements) {
      const unsigned matrix = (unsigned)job.dst_rows * job.dst_cols;
      const long o = e / matrix;
      const unsigned in = (unsigned)(e - o * matrix), r = in / job.dst_cols,
                     c = in - r * job.dst_cols;
      const bool inside = (int)r < job.src_rows && (int)c < job.src_cols;
      const long from = (o * job.src_rows + r) * job.src_cols + c;
      if (job.bytes == 4)
        static_cast<unsigned*>(job.dst)[e] =
            inside ? static_cast<const unsigned*>(job.src)[from] : job.fill;
      else
        static_cast<unsigned short*>(job.dst)[e] =
            inside ? static_cast<const unsigned short*>(job.src)[from] : (unsigned short)job.fill;
      return;
    }
    e -= job.elements;
  }
}

}  // namespace m4
