// Which exchange ring a launch of the one-shot steps uses and under which tags: the host's share of row_exchange.h, in
// plain C++ (no HIP types), so that it can be run and tested without a GPU.
//
// The rule that keeps launches apart: no two launches that use the same ring have a tag in common (until the ring is
// cleared, which is ordered behind the one and before the other).  A workgroup therefore never takes a word of another
// launch for its neighbours', whichever threads and streams the launches come from and however their enqueues interleave.
#pragma once

#include <mutex>

namespace relax_amd {

constexpr int kOwnedRings = 4;                   // rings that belong to a stream each
constexpr int kSharedRing = kOwnedRings;         // the ring of all other streams, whose launches wait for each other
constexpr int kCaptureRing = kOwnedRings + 1;    // the ring of launches recorded into graphs
constexpr int kExchangeRings = kOwnedRings + 2;
constexpr unsigned kCapturedLaunches = 4096;     // launches a process may record per GPU

// The tags of one ring.  `lock` is held from take() until the launch is enqueued: the launches of a ring's stream are then
// enqueued in the order of their tags, and a clearing lies between the tags before and those after it.
struct RingTags {
  std::mutex lock;
  unsigned used = 0;  // tags 1 .. used have been handed out since the ring was cleared (0 is a cleared word)

  // base .. base + laps - 1: tags of the launch that follows.  True when the ring has to be cleared in front of it.
  bool take(unsigned laps, unsigned& base) {
    const bool clear = laps >= 0xffffffffu - used;  // the last tag stays free: the waits' test offset is added to a tag
    if (clear) used = 0;
    base = used + 1;
    used += laps;
    return clear;
  }
};

// The streams that own a ring: the first kOwnedRings a GPU's launches come from.  A stream runs its launches one after
// another, so they may share a ring's slots.
class RingOwners {
 public:
  // the ring of the stream, or kSharedRing
  int of(const void* stream) {
    std::lock_guard<std::mutex> hold(lock_);
    for (int i = 0; i < used_; ++i)
      if (streams_[i] == stream) return i;
    if (used_ == kOwnedRings) return kSharedRing;
    streams_[used_] = stream;
    return used_++;
  }

 private:
  std::mutex lock_;
  const void* streams_[kOwnedRings] = {};
  int used_ = 0;
};

}  // namespace relax_amd
