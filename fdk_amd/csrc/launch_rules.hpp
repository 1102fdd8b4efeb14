// Rules of the launches that need no device: which form of a kernel a call's sizes
// take.  Host code without HIP, so that tests check them by themselves.
#pragma once
#include <cstdint>

namespace fdk {
namespace rules {

// Forms of the row filter: the in-place kernel, filter_wide_kernel with 32-bit offsets
// in a view, and with every point outside its row left out before the store.
enum FilterForm { kFilterInPlace = 0, kFilterWide = 1, kFilterWideFar = 2 };

// filter_wide_kernel (N = 2^7 .. 2^14) stores a thread's point u of a transposed FP32
// view at byte 4 (u nrows + row) mod 2^32 and lets the view's resource drop the points
// outside the row, u = 1 - N/16 .. -1 and nu .. nu + N/16 - 2.  They fall outside the
// view up to (nu + N/16) nrows = 2^30; past that (views much shorter than N of a million
// rows) some would wrap into it.  The resource itself spans less than 2 GiB.  Row-major
// stores have a resource a row, 16-bit stores 64-bit addresses, so they have no such limit.
inline FilterForm filter_form(int nu, int nrows, int nviews, int log_n, bool transposed_f32) {
  if (log_n < 7 || log_n > 14) return kFilterInPlace;
  if ((int64_t)(nrows + 64) * nviews >= (int64_t)1 << 29) return kFilterInPlace;  // the kernel's ints
  if (transposed_f32 && ((int64_t)nu * nrows * 4 >= (int64_t)1 << 31 ||
                         (int64_t)(nu + (1 << log_n) / 16) * nrows * 4 > (int64_t)1 << 32))
    return kFilterWideFar;
  return kFilterWide;
}

}  // namespace rules
}  // namespace fdk
