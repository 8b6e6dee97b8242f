// A buffer that is replaced by a larger one when a request exceeds it and otherwise kept.
#pragma once

#include <cstddef>

namespace fw {

struct GrowBuffer {
  void* p = nullptr;
  size_t bytes = 0;
};

inline size_t round_bytes(size_t b) { return (b + 255) & ~size_t(255); }

// `b` with room for `need` bytes, or nullptr. A larger buffer takes the place of the old one, which is
// released first: twice the need, so that slowly growing requests do not replace it each time, or the
// need alone where twice that is not to be had. alloc(bytes) gives nullptr on failure; `b` is then
// empty, so that no later request is answered with the buffer already released.
template <typename Alloc, typename Release>
void* grow(GrowBuffer& b, size_t need, Alloc&& alloc, Release&& release) {
  if (b.bytes >= need) return b.p;
  if (b.p) release(b.p);
  b = GrowBuffer{};
  for (const size_t want : {round_bytes(2 * need), round_bytes(need)})
    if (void* p = alloc(want)) {
      b = GrowBuffer{p, want};
      return p;
    }
  return nullptr;
}

}  // namespace fw
