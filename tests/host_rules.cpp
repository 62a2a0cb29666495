// Prints what the host rules of invdft_amd/csrc/host_rules.h do, for test_host_rules.py.
#include <cstdio>
#include <stdexcept>

#include "host_rules.h"

struct Full : std::runtime_error {
  Full() : std::runtime_error("full") {}
};
static int left;  // allocations until one fails
struct Buf {
  size_t n = 0;
  void release() { n = 0; }
  void resize(size_t count) {
    if (count <= n) return;
    release();
    if (left-- == 0) throw Full();
    n = count;
  }
};

int main() {
  // five buffers, one of them large enough already, with room for `room` allocations
  for (int room = 0; room <= 5; ++room) {
    Buf b[5];
    b[3].n = 70;
    left = room;
    const bool ok = idft::resize_all_or_none<Full>(b, 5, 64);
    std::printf("alloc %d %d", room, (int)ok);
    for (const Buf& x : b) std::printf(" %zu", x.n);
    std::printf("\n");
  }
  for (int b = 1; b <= 80; ++b)
    for (int fit : {0, 1, 2, 3, 7, 16, 33, 79, 80, 1000})
      std::printf("slice %d %d %d\n", b, fit, idft::quad_slice(b, 80, fit));
  return 0;
}
