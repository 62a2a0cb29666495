// Rules of the host code that need no device: tested on the CPU.
#pragma once
#include <cstddef>

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

}  // namespace idft
