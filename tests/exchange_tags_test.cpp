// Host program behind tests/test_exchange_tags.py: the rule of csrc/exchange_tags.h that keeps launches apart.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <thread>
#include <utility>
#include <vector>

#include "exchange_tags.h"

using namespace relax_amd;

#define REQUIRE(x) \
  if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), 1

int main() {
  // many threads on one ring: no two launches share a tag, and they are enqueued in the order of their tags
  RingTags ring;
  std::vector<std::pair<unsigned, unsigned>> enqueued;  // (base, laps), in the order of the enqueues
  std::vector<std::thread> threads;
  for (int t = 0; t < 8; ++t)
    threads.emplace_back([&, t] {
      for (int i = 0; i < 2000; ++i) {
        const unsigned laps = 1 + (t + i) % 3;
        std::lock_guard<std::mutex> hold(ring.lock);
        unsigned base = 0;
        ring.take(laps, base);
        enqueued.emplace_back(base, laps);
      }
    });
  for (auto& t : threads) t.join();
  unsigned next = 1;
  for (auto [base, laps] : enqueued) {
    REQUIRE(base == next);
    next += laps;
  }
  // the ring is cleared before a tag comes round again; tag 0 (a cleared word) and the last one are never handed out
  unsigned base = 0;
  ring.used = 0xffffffffu - 3;
  REQUIRE(!ring.take(2, base) && base == 0xffffffffu - 2 && ring.used == 0xffffffffu - 1);
  REQUIRE(ring.take(1, base) && base == 1);
  REQUIRE(!ring.take(65536, base) && base == 2);
  ring.used = 0xffffffffu - 65536;
  REQUIRE(ring.take(65536, base) && base == 1 && ring.used == 65536);
  // a ring per stream for the first kOwnedRings, asked by several threads at once; one ring for all others
  RingOwners owners;
  int streams[kOwnedRings + 3];
  std::vector<std::thread> askers;
  int got[4][kOwnedRings + 3];
  for (int t = 0; t < 4; ++t)
    askers.emplace_back([&, t] {
      for (int i = 0; i < kOwnedRings; ++i) got[t][i] = owners.of(&streams[(i + t) % kOwnedRings]);
    });
  for (auto& t : askers) t.join();
  bool seen[kOwnedRings] = {};
  for (int i = 0; i < kOwnedRings; ++i) {
    const int r = owners.of(&streams[i]);
    REQUIRE(r >= 0 && r < kOwnedRings && !seen[r]);
    seen[r] = true;
    for (int t = 0; t < 4; ++t) REQUIRE(got[t][(i - t + 2 * kOwnedRings) % kOwnedRings] == r);
  }
  for (int i = kOwnedRings; i < kOwnedRings + 3; ++i) REQUIRE(owners.of(&streams[i]) == kSharedRing);
  REQUIRE(kCaptureRing != kSharedRing && kCaptureRing < kExchangeRings);
  std::puts("ok");
  return 0;
}
