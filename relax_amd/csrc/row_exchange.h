// Exchange of per-wave partial results between the one-shot workgroups that share a row (actor_step_split.hip,
// actor_step_split_any.hip, reverse_kl_split.hip).
//
// A ring of slots in device memory, one per (row mod kRing); a slot holds, for each of the row's waves, a few eight-byte
// words, each a float and a 32-bit tag, written and read with relaxed device-scope atomics.  The tag names the launch and
// the lap of the ring, and a reader tells a stale word from the one it waits for without any fence.  The workgroups of a
// row have consecutive indices; a workgroup only waits for those, which are resident or next in dispatch order whatever
// else the chip runs, so every wait ends.  It is bounded all the same: the first wait of a launch that gives up raises a
// flag that ends the launch's other waits at their next look at it, and counts itself.
//
// Whose ring, and which tags (exchange_tags.h).  The host gives every launch tags of its own and hands them over as a
// kernel argument, so two launches never take each other's words for their own, whichever threads enqueue them.  Slots
// are kept apart too: each of the first kOwnedRings streams of a GPU has a ring, whose launches follow each other; all other
// streams share one, where a launch waits (an event) for the one before it.  A launch that is being captured cannot be
// given tags by the host, since each replay needs new ones: a one-workgroup kernel recorded in front of it takes them from a
// counter on the device and leaves them in a word that belongs to that recorded launch alone.  Captured launches share a
// ring; replays of two of them that overlap can overwrite each other's slots, and because their tags differ this ends as
// waits that give up, never as a wrong number taken for right.
// (With one counter on the device for all launches, advanced by a launch in front of each step, two threads that enqueued
// on one stream could interleave as advance, advance, step, step and give both steps the same tags.)
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <mutex>

#include "device_utils.h"
#include "exchange_tags.h"
#include "relax_amd.h"

namespace relax_amd {

constexpr unsigned kRing = 4096;           // rows whose slots exist at a time
constexpr unsigned kWaitPolls = 1u << 17;  // looks at a neighbour's word before a wait gives up (a few suffice; each takes microseconds)
// behind a ring's slots: 32-bit words [0] the tag counter of captured launches, [1] the count of waits that gave up, [2]
// the first tag of the last launch one of whose waits gave up
constexpr int kRingTailWords = 32;

// relax_amd_set_exchange_wait(): the bound of a wait and an offset added to the tag it waits for
unsigned exchange_max_polls();
unsigned exchange_wait_tag_offset();

// Forgets every word of a ring, and of `extra` (a second array of tagged words that shares the ring's tags, or null), by
// one workgroup.
template <size_t RING_WORDS>
__device__ __forceinline__ void exchange_clear(unsigned long long* ring, unsigned long long* extra, size_t extra_words) {
  for (size_t i = threadIdx.x; i < RING_WORDS; i += 256) ring[i] = 0ull;
  if (extra)
    for (size_t i = threadIdx.x; i < extra_words; i += 256) extra[i] = 0ull;
  if (threadIdx.x == 0) reinterpret_cast<unsigned*>(ring + RING_WORDS)[2] = 0u;
}

// in front of the launch that would need a 33rd bit of tag
template <size_t RING_WORDS>
__global__ __launch_bounds__(256) void exchange_ring_clear_kernel(unsigned long long* ring, unsigned long long* extra,
                                                                  size_t extra_words) {
  exchange_clear<RING_WORDS>(ring, extra, extra_words);
}

// In front of a captured launch: `laps` tags from the device's counter, the first of them into *word.
template <size_t RING_WORDS>
__global__ __launch_bounds__(256) void exchange_capture_tags_kernel(unsigned long long* ring, unsigned laps,
                                                                    unsigned* word, unsigned long long* extra,
                                                                    size_t extra_words) {
  unsigned* counter = reinterpret_cast<unsigned*>(ring + RING_WORDS);
  const unsigned last = 0xffffffffu - laps - 1u;
  __shared__ unsigned used;
  if (threadIdx.x == 0) used = atomicAdd(counter, laps);
  __syncthreads();
  if (used > last) {
    exchange_clear<RING_WORDS>(ring, extra, extra_words);
    __syncthreads();
    if (threadIdx.x == 0)
      for (int i = 0; i < 3 && used > last; ++i) used = atomicAdd(counter, laps);  // once or twice past the wrap
  }
  if (threadIdx.x == 0) *word = used + 1u;
}

// the first tag of this launch
__device__ __forceinline__ unsigned exchange_first_tag(unsigned base, const unsigned* word) { return word ? *word : base; }

__device__ __forceinline__ void exchange_store(unsigned long long* word, unsigned tag, float val) {
  __hip_atomic_store(word, (static_cast<unsigned long long>(tag) << 32) | __float_as_uint(val), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// Waits, boundedly, for `word` to carry `tag`; false when the wait gave up (its own bound, or another wait of the launch
// did).
__device__ __forceinline__ bool exchange_wait(const unsigned long long* word, unsigned tag, unsigned max_polls,
                                              unsigned* status, unsigned first_tag, float& out) {
  unsigned polls = 0;
  while (true) {
    const unsigned long long w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (unsigned(w >> 32) == tag) {
      out = __uint_as_float(unsigned(w));
      return true;
    }
    ++polls;
    if (polls > max_polls ||
        ((polls & 63u) == 0u && __hip_atomic_load(status + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == first_tag))
      return false;
    __builtin_amdgcn_s_sleep(1);
  }
}

// one lane of a wave whose wait gave up: counts it and ends the launch's other waits
__device__ __forceinline__ void exchange_report_give_up(unsigned* status, unsigned first_tag) {
  atomicAdd(status + 1, 1u);
  __hip_atomic_store(status + 2, first_tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Words of a family's file-scope __device__ array: its rings, then the captured launches' words.
template <size_t RING_WORDS>
constexpr size_t exchange_array_words() {
  return kExchangeRings * (RING_WORDS + kRingTailWords) + kCapturedLaunches / 2;
}

// What the host knows about a kernel family's rings on one GPU, and on all of them.
struct ExchangeDevice {
  std::mutex lock;  // of the look-up
  unsigned long long* rings = nullptr;
  unsigned long long* extra = nullptr;
  RingOwners owners;
  RingTags tags[kOwnedRings + 1];
  hipEvent_t shared_done = nullptr;  // behind the last launch on the shared ring (guarded by that ring's tags)
  bool shared_broken = false;        // that launch could not be marked: nothing may follow it on the ring
  std::atomic<unsigned> captured{0};
};
struct ExchangeFamily {
  static constexpr int kMaxDevices = 64;
  const char* who;
  ExchangeDevice devices[kMaxDevices];
};

// relax_amd_advance_exchange_tags() for one family on the current device, which is idle: no ring goes back.
template <size_t RING_WORDS>
int exchange_advance_tags(ExchangeFamily& family, const void* ring_symbol, unsigned used) {
  int index = -1;
  void* rings = nullptr;
  hipError_t e = hipGetDevice(&index);
  if (e == hipSuccess && (index < 0 || index >= ExchangeFamily::kMaxDevices)) e = hipErrorInvalidDevice;
  if (e == hipSuccess) e = hipGetSymbolAddress(&rings, ring_symbol);
  unsigned counter = 0;
  if (e == hipSuccess) {
    unsigned* on_device = reinterpret_cast<unsigned*>(static_cast<unsigned long long*>(rings) +
                                                      kCaptureRing * (RING_WORDS + kRingTailWords) + RING_WORDS);
    e = hipMemcpy(&counter, on_device, sizeof(counter), hipMemcpyDeviceToHost);
    if (e == hipSuccess && counter < used) e = hipMemcpy(on_device, &used, sizeof(used), hipMemcpyHostToDevice);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
    set_error("%s: exchange tags: %s", family.who, hipGetErrorString(e));
    return RELAX_AMD_ELAUNCH;
  }
  for (RingTags& t : family.devices[index].tags) {
    std::lock_guard<std::mutex> hold(t.lock);
    if (t.used < used) t.used = used;
  }
  return RELAX_AMD_OK;
}

// The ring and the tags of one launch, held while it is enqueued.
class ExchangeLaunch {
 public:
  unsigned long long* ring = nullptr;
  unsigned long long* extra = nullptr;
  unsigned base = 0;               // first tag
  const unsigned* word = nullptr;  // where a captured launch finds it

  // `own_ring_only`: RELAX_AMD_EUNSUPPORTED (before anything is enqueued) for a stream without a ring of its own and for
  // a captured launch.
  template <size_t RING_WORDS>
  int open(ExchangeFamily& family, const void* ring_symbol, const void* extra_symbol, size_t extra_words,
           hipStream_t stream, unsigned laps, bool own_ring_only) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess) {
      (void)hipGetLastError();
      return RELAX_AMD_EUNSUPPORTED;
    }
    const bool captured = capture != hipStreamCaptureStatusNone;
    if (captured && own_ring_only) return RELAX_AMD_EUNSUPPORTED;
    int index = 0;
    hipError_t e = hipGetDevice(&index);
    if (e != hipSuccess || index < 0 || index >= ExchangeFamily::kMaxDevices) {
      set_error("%s: no usable current device (%s)", family.who,
                e == hipSuccess ? "index out of range" : hipGetErrorString(e));
      return RELAX_AMD_EINVAL;
    }
    ExchangeDevice& dev = family.devices[index];
    {
      std::lock_guard<std::mutex> hold(dev.lock);
      if (int rc = look_up(family, index, ring_symbol, dev.rings)) return rc;
      if (extra_symbol)
        if (int rc = look_up(family, index, extra_symbol, dev.extra)) return rc;
    }
    constexpr size_t kStride = RING_WORDS + kRingTailWords;
    auto take_ring = [&](int i) {
      ring = dev.rings + size_t(i) * kStride;
      extra = dev.extra ? dev.extra + size_t(i) * extra_words : nullptr;
    };
    if (captured) {
      const unsigned n = dev.captured.fetch_add(1, std::memory_order_relaxed);
      if (n >= kCapturedLaunches) {
        dev.captured.store(kCapturedLaunches, std::memory_order_relaxed);
        return RELAX_AMD_EUNSUPPORTED;
      }
      take_ring(kCaptureRing);
      unsigned* mine = reinterpret_cast<unsigned*>(dev.rings + kExchangeRings * kStride) + n;
      word = mine;
      hipLaunchKernelGGL(exchange_capture_tags_kernel<RING_WORDS>, dim3(1), dim3(256), 0, stream, ring, laps, mine,
                         extra, extra_words);
      return RELAX_AMD_OK;
    }
    // a per-thread default stream is another stream in every thread under one handle: it cannot own a ring
    const int i = stream == hipStreamPerThread ? kSharedRing : dev.owners.of(stream);
    if (i == kSharedRing && own_ring_only) return RELAX_AMD_EUNSUPPORTED;
    hold_ = std::unique_lock<std::mutex>(dev.tags[i].lock);
    if (i == kSharedRing) {
      if (dev.shared_broken) return RELAX_AMD_EUNSUPPORTED;
      if (dev.shared_done) {
        e = hipStreamWaitEvent(stream, dev.shared_done, 0);
      } else {
        e = hipEventCreateWithFlags(&dev.shared_done, hipEventDisableTiming);
        if (e != hipSuccess) dev.shared_done = nullptr;
      }
      if (e != hipSuccess) {
        (void)hipGetLastError();
        return RELAX_AMD_EUNSUPPORTED;
      }
      shared_ = &dev;
      stream_ = stream;
    }
    take_ring(i);
    if (dev.tags[i].take(laps, base))
      hipLaunchKernelGGL(exchange_ring_clear_kernel<RING_WORDS>, dim3(1), dim3(256), 0, stream, ring, extra, extra_words);
    return RELAX_AMD_OK;
  }

  ~ExchangeLaunch() {
    if (shared_ && hipEventRecord(shared_->shared_done, stream_) != hipSuccess) {
      (void)hipGetLastError();
      shared_->shared_broken = true;
    }
  }

 private:
  // the current device's copy of a file-scope __device__ array: looked up once per device, with that device current
  static int look_up(const ExchangeFamily& family, int device, const void* symbol, unsigned long long*& ptr) {
    if (ptr) return RELAX_AMD_OK;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, symbol);
    if (e != hipSuccess || !p) {
      set_error("%s: hipGetSymbolAddress failed on device %d: %s", family.who, device, hipGetErrorString(e));
      return RELAX_AMD_ELAUNCH;
    }
    ptr = static_cast<unsigned long long*>(p);
    return RELAX_AMD_OK;
  }

  std::unique_lock<std::mutex> hold_;  // destroyed after the destructor has marked the shared ring's launch
  ExchangeDevice* shared_ = nullptr;
  hipStream_t stream_ = nullptr;
};

}  // namespace relax_amd
