// CPU test of StagingRing::download (orcaml_amd/csrc/runtime_host.cpp) against the HIP API
// stand-in: sizes around its parts and the ring's capacity, destinations at odd addresses, reads
// after uploads still in flight and from two contexts at once.  Built under the address and
// undefined-behaviour sanitizers, and under the thread sanitizer, by tests/test_native_download.py.
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "runtime.hpp"

using namespace orca_hip;

#define CHECK(cond)                                                          \
  do {                                                                       \
    if (!(cond)) {                                                           \
      std::fprintf(stderr, "CHECK failed at line %d: %s\n", __LINE__, #cond); \
      std::abort();                                                          \
    }                                                                        \
  } while (0)

static void reads(unsigned seed) {
  orca_hip_ctx ctx;
  const size_t M = size_t(1) << 20, sizes[] = {1, 4, M - 1, M, M / 2, M / 2 + 3, 8 * M - 1, 8 * M, 8 * M + 5,
                                               16 * M, 16 * M + 1, 18 * M, 41 * M + 12345};
  std::vector<unsigned char> device(42 * M);
  for (size_t i = 0; i < device.size(); ++i) device[i] = (unsigned char)((i * 2654435761u + seed) >> 13);
  std::vector<unsigned char> up(2 * M, 1), host;
  for (size_t n : sizes) {
    for (size_t shift : {size_t(0), size_t(3)}) {
      host.assign(n + shift + 16, 0xAB);
      // an upload in flight holds part of the ring
      ctx.staging.upload(&ctx, device.data() + 41 * M + 20000, up.data(), 1000, nullptr);
      const auto waits = ctx.host_syncs.load();
      ctx.staging.download(&ctx, host.data() + shift, device.data() + shift, n, nullptr);
      CHECK(ctx.host_syncs.load() > waits);
      CHECK(std::memcmp(host.data() + shift, device.data() + shift, n) == 0);
      for (size_t i = 0; i < shift; ++i) CHECK(host[i] == 0xAB);
      for (size_t i = 0; i < 16; ++i) CHECK(host[shift + n + i] == 0xAB);
      ctx.staging.upload(&ctx, up.data() + M, up.data(), M, nullptr);  // the ring is whole again
    }
  }
  ctx.staging.download(&ctx, nullptr, nullptr, 0, nullptr);
}

int main() {
  hip_stub::event_delay() = 1;
  reads(1);
#ifndef __SANITIZE_THREAD__  // the stand-in's own counters are plain globals
  std::thread a([] { reads(2); }), b([] { reads(3); });  // one context each
  a.join();
  b.join();
#endif
  std::puts("all checks passed");
}
