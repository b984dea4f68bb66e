// kept_at_least over an allocator with a limit: prints one line per call, "allocations -> kept bytes".
#include <cstdio>
#include <cstdlib>
#include <map>

#include "kept.h"

int main() {
  std::map<void*, size_t> live;
  size_t in_use = 0, limit = 0;
  efh::KeptBuffer k;
  auto call = [&](size_t bytes) {
    auto alloc = [&](size_t n) -> void* {
      std::printf("ask %zu ", n);
      if (in_use + n > limit) return nullptr;
      void* p = std::malloc(1);
      live[p] = n;
      in_use += n;
      return p;
    };
    auto release = [&](void* p) {
      std::printf("free %zu ", live.at(p));
      in_use -= live.at(p);
      live.erase(p);
      std::free(p);
    };
    void* p = efh::kept_at_least(k, bytes, alloc, release);
    if (p != k.p || live.size() != (p ? 1u : 0u)) return false;
    if (p != nullptr && (live.at(p) != k.bytes || k.bytes < bytes)) return false;
    std::printf("-> %zu\n", k.bytes);
    return true;
  };
  const size_t mb = size_t(1) << 20;
  limit = 100 * mb;
  bool ok = call(5) && call(mb) && call(mb + 1) && call(3) && call(40 * mb);  // growth by doubling, reuse
  limit = 90 * mb;
  ok = ok && call(70 * mb);  // 128 MB refused, 70 fit
  ok = ok && call(70 * mb) && call(64 * mb);
  ok = ok && call(91 * mb);  // neither: nothing kept, nothing leaked
  ok = ok && call(64 * mb);  // a power of two: asked for once
  limit = 60 * mb;
  ok = ok && call(128 * mb) && call(60 * mb);
  for (auto& e : live) std::free(e.first);
  return ok ? 0 : 1;
}
