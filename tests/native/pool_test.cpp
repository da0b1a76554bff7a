// Test-only: the context's memory pool (csrc/internal.hpp: DevPool, DevBuf) under
// two threads, with the stand-in of the HIP runtime.
#include <atomic>
#include <thread>

#include "../../thrml-rs_amd/csrc/internal.hpp"

namespace thrml {
int fail(int code, const std::string &) { return code; }
int hip_fail(hipError_t, const char *) { return THRML_EHIP; }
}  // namespace thrml

// A buffer taken before the stream changes is let go of while it changes, n
// times over: how often the pool kept it, for the next object on the new stream.
extern "C" uint64_t pool_kept_across_stream_change(uint64_t n) {
  thrml::DevPool pool;
  thrml::DevBuf buf;
  std::atomic<uint64_t> go{0}, done{0};
  std::thread other([&] {
    for (uint64_t i = 1; i <= n; ++i) {
      while (go.load() < i) {}
      for (volatile uint64_t spin = 0; spin < i % 64u; ++spin) {}
      buf.release();
      done.store(i);
    }
  });
  uint64_t kept = 0;
  for (uint64_t i = 1; i <= n; ++i) {
    if (buf.alloc(4096, &pool)) return ~0ull;
    go.store(i);
    for (volatile uint64_t spin = 0; spin < 8u; ++spin) {}
    pool.new_stream();
    while (done.load() < i) {}
    size_t cap;
    uint64_t era;
    if (void *p = pool.take(4096, &cap, &era)) {
      ++kept;
      (void)hipFree(p);
    }
  }
  other.join();
  return kept;
}
