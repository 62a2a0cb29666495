// Rules of the host code that need no device: tested on the CPU.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace idft {

// Optional workspace: all of bufs[0 .. n-1] with `count` elements, or none of them.
// Returns false, with every one of them released, where an allocation fails (the
// caller goes on without); Failure is what a failed allocation throws.
template <typename Failure, typename Buf>
bool resize_all_or_none(Buf* bufs, int n, size_t count) {
  try {
    for (int i = 0; i < n; ++i) bufs[i].resize(count);
    return true;
  } catch (const Failure&) {
    for (int i = 0; i < n; ++i) bufs[i].release();
    return false;
  }
}

// Columns per pass over a block of b columns where the cell kernel takes at most
// `cols` and the 32-bit index of the cell scratch `fit`: b if it fits, otherwise even
// (the gather stores two columns at a time where a row starts at an even column), or 1.
inline int quad_slice(int b, int cols, int64_t fit) {
  const int w = (int)std::min<int64_t>(std::min(b, cols), std::max<int64_t>(fit, 1));
  return w < b && w > 1 ? w - w % 2 : w;
}

}  // namespace idft
