// A buffer kept from call to call: its growth, apart from where the memory comes from.
#pragma once
#include <cstddef>
#include <initializer_list>

namespace efh {

struct KeptBuffer {
  void* p = nullptr;
  size_t bytes = 0;
};

constexpr size_t kKeptLeast = size_t(1) << 20;

// k's memory with at least `bytes` bytes.  A smaller buffer is given back first; the new one is `bytes`
// rounded up to a power of two (so that slowly growing calls do not each replace it), or exactly `bytes`
// where that much cannot be had.  Null, with nothing kept, when neither can.  alloc(n) returns memory or
// null, release(p) takes it back.
template <class Alloc, class Release>
void* kept_at_least(KeptBuffer& k, size_t bytes, Alloc&& alloc, Release&& release) {
  if (k.p != nullptr && k.bytes >= bytes) return k.p;
  if (k.p != nullptr) {
    void* old = k.p;
    k = KeptBuffer{};
    release(old);
  }
  size_t want = kKeptLeast;
  while (want < bytes) want *= 2;
  for (const size_t n : {want, bytes}) {
    if (void* p = alloc(n)) {
      k.p = p;
      k.bytes = n;
      return p;
    }
    if (n == bytes) break;
  }
  return nullptr;
}

}  // namespace efh
