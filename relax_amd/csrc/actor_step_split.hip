// Fused actor step with every row shared between eight one-shot workgroups: the same computation and the same bits
// as actor_step_resident_kernel (log-prob + entropy forward, per-token policy-loss coefficients, dlogits backward, each
// logit read once and each gradient written once), in the launch shape this memory system streams fastest: many small
// workgroups that touch their memory once and retire, dispatched in address order (a mixed read / write stream of
// this shape moves 6.1 - 6.6 TB/s on the box where 256 persistent row-sized streams move 5.6; this kernel on the
// 65536 x 151936 bf16 step: 5.64 - 5.74 ms compiled for three waves per SIMD, 5.74 - 5.89 for four, where the
// persistent kernel takes 6.44 - 6.58; 6.0 ms with 256-thread and 6.3 ms with 64-thread workgroups).
//
// A row is scanned by 1024 "virtual threads" exactly as scan_row() lays it out for a 1024-thread workgroup (virtual
// thread t takes the 16-byte vectors t, t + 1024, ...; four at a time while it has four to go, then single ones).  A
// workgroup here is 128 of those virtual threads (two waves: virtual waves 2q and 2q + 1 of the row), holds its
// share of the row in registers (19 vectors per thread at V = 151936 bf16), reduces each wave to its (max, sum exp,
// sum exp * x) triple by the same butterfly, publishes the two triples, fetches the row's sixteen, merges them in
// wave order as scan_block_merge() does, and turns its registers into the gradient.  Log-probs, entropy and gradients
// are therefore bit-identical to the forward-only kernel's and the other fused kernels'.
//
// Exchange: the tagged ring of row_exchange.h, a slot of 16 x 3 words per row; a workgroup that gives up its wait
// writes NaN log-probs instead of hanging.
//
// Rows whose share does not fit the registers of three waves per SIMD (16-bit rows of more than 20 vectors per thread,
// fp32 rows of more than 16: vocabularies of 100352 .. 163840 entries as fp32, 200 k .. 262 k entries as 16-bit,
// 248320 as either) keep twelve to nineteen vectors of every thread's share in LDS, put there by global -> LDS loads
// without a register in between (LDS_VECS).  An fp32 row of 151936 entries is thereby read once as it is (5.85 -
// 5.95 ms per 32768 rows whether its values are widened bf16 or genuinely fp32).
//
// Replaces, like the other fused kernels, _VocabParallelLogProbEntropy.forward + .backward
// (relax/utils/training/ppo_utils.py:481-629) and the per-token part of policy_loss_function
// (relax/backends/megatron/loss.py:961-1100) for one micro-batch.
//
// As in actor_step_resident.hip the row sits at the edge of the register file:
// hipcc-flags: -mllvm -amdgpu-use-amdgpu-trackers=1
#include <atomic>

#include "actor_step_resident.h"
#include "actor_step_split.h"

namespace relax_amd {

// The exchange rings (1.5 MB each) and, of the same tags, those of the logits at a token's top-K ids (8 MB each).  The
// logits are gathered once per row: each workgroup of a row fetches its share of the K scattered entries and publishes
// them (one tagged word per entry), every workgroup's first wave collects all K.  Gathered by each of the eight workgroups
// for itself, the K scattered lines crossed the fabric eight times per row (3.4 GB on 65536 x 151936 rows with K = 64, a
// tenth of the step's traffic).
static __device__ __align__(256) unsigned long long split_rings[exchange_array_words<kRingWords>()];
static __device__ __align__(256) unsigned long long split_topk_rings[kExchangeRings * kTopkRingWords];

namespace {
ExchangeFamily split_family{"actor_step_split", {}};
// relax_amd_set_exchange_wait: the bound of a workgroup's wait and an offset added to the tag it waits for
std::atomic<unsigned> g_max_polls{kWaitPolls}, g_wait_tag_offset{0u};
}  // namespace

unsigned exchange_max_polls() { return g_max_polls.load(std::memory_order_relaxed); }
unsigned exchange_wait_tag_offset() { return g_wait_tag_offset.load(std::memory_order_relaxed); }

int kl_advance_exchange_tags(unsigned used);  // reverse_kl_split.hip

int open_split_exchange(ExchangeLaunch& x, hipStream_t stream, int64_t n_rows, bool own_ring_only) {
  return x.open<kRingWords>(split_family, reinterpret_cast<const void*>(&split_rings),
                            reinterpret_cast<const void*>(&split_topk_rings), kTopkRingWords, stream,
                            unsigned((n_rows + kRing - 1) / kRing), own_ring_only);
}

// Waves per SIMD the kernel is compiled for.  Long 16-bit rows without the top-K term run fastest with three (six
// workgroups per CU, up to 168 registers a lane: 5.64 - 5.66 ms on the 65536 x 151936 step where four give 5.74 and
// two 6.03; rows of 15 and more vectors per thread all gain 1 - 2.5 %), the top-K instantiations and rows of up to 13
// vectors per thread with four or more (their thread 0 works longer per row, or they need few registers anyway).
template <int NV, bool TOPK, int VN>
constexpr int split_waves_min() {
  return (!TOPK && VN == 8 && NV >= 15) ? 3 : 4;
}
template <int NV, bool TOPK, int VN>
constexpr int split_waves_max() {
  return (!TOPK && VN == 8 && NV >= 15) ? 3 : 8;
}
#define RELAX_AMD_SPLIT_KERNEL(WIDTH, NVF, PARTIAL, TOPK)                                                             \
  actor_step_split_kernel<T, NVF, PARTIAL, TOPK, WIDTH, split_waves_min<NVF + (PARTIAL ? 1 : 0), TOPK, VN>(),         \
                          split_waves_max<NVF + (PARTIAL ? 1 : 0), TOPK, VN>()>
#define RELAX_AMD_SPLIT_ROW(WIDTH, NVF, PARTIAL)                                                                      \
  if (width == WIDTH && full == NVF && partial == PARTIAL) {                                                          \
    if (a.topk_ids)                                                                                                   \
      hipLaunchKernelGGL((RELAX_AMD_SPLIT_KERNEL(WIDTH, NVF, PARTIAL, true)), grid, block, 0, stream, logits,        \
                         row_stride, vocab, n_rows, token_of_row, sample_ids, targets, inv_t * kLog2e, inv_t, a,     \
                         grad_scale, log_prob, entropy, lse, spx, dlogits, d_stride, x.ring, x.extra,                 \
                         x.base, x.word, max_polls, tag_offset);                                                      \
    else                                                                                                              \
      hipLaunchKernelGGL((RELAX_AMD_SPLIT_KERNEL(WIDTH, NVF, PARTIAL, false)), grid, block, 0, stream, logits,       \
                         row_stride, vocab, n_rows, token_of_row, sample_ids, targets, inv_t * kLog2e, inv_t, a,     \
                         grad_scale, log_prob, entropy, lse, spx, dlogits, d_stride, x.ring, x.extra,                 \
                         x.base, x.word, max_polls, tag_offset);                                                      \
    return check_launch("actor_step_split");                                                                          \
  }
#define RELAX_AMD_SPLIT(NVF, PARTIAL) RELAX_AMD_SPLIT_ROW(1024, NVF, PARTIAL)
// Rows of more vectors per thread than the register file holds at three waves per SIMD (16-bit rows of more than 20,
// fp32 rows of more than 16): part of every thread's share sits in LDS.  16-bit: twelve or thirteen vectors (24 - 26 KB
// of the 26.7 a workgroup can have when six share a CU), three waves per SIMD.  fp32 rows of up to 40 vectors per
// thread (100352 .. 163840 entries): thirteen in LDS, three waves; of 61 (248320 entries): nineteen in LDS (38 KB), two
// waves.  With the top-K term (4 KB of LDS more, a longer serial stretch): sixteen in LDS and two waves per SIMD.
template <int NV, bool TOPK, int VN>
constexpr int split_lds_vecs() {
  return TOPK ? 16 : (VN == 4 && NV > 40) ? 19 : (VN == 8 && NV <= 25) ? 12 : 13;
}
template <int NV, bool TOPK, int VN>
constexpr int split_lds_waves() {
  return (TOPK || (VN == 4 && NV > 40)) ? 2 : 3;
}
#define RELAX_AMD_SPLIT_LDS_KERNEL(NVF, PARTIAL, TOPK)                                                                \
  actor_step_split_kernel<T, NVF, PARTIAL, TOPK, 1024, split_lds_waves<NVF + (PARTIAL ? 1 : 0), TOPK, VN>(),          \
                          split_lds_waves<NVF + (PARTIAL ? 1 : 0), TOPK, VN>(),                                       \
                          split_lds_vecs<NVF + (PARTIAL ? 1 : 0), TOPK, VN>()>
#define RELAX_AMD_SPLIT_LDS(NVF, PARTIAL, WITH_TOPK)                                                                  \
  if (width == 1024 && full == NVF && partial == PARTIAL) {                                                           \
    if (a.topk_ids) {                                                                                                 \
      if constexpr (WITH_TOPK)                                                                                        \
        hipLaunchKernelGGL((RELAX_AMD_SPLIT_LDS_KERNEL(NVF, PARTIAL, true)), grid, block, 0, stream, logits,         \
                           row_stride, vocab, n_rows, token_of_row, sample_ids, targets, inv_t * kLog2e, inv_t, a,   \
                           grad_scale, log_prob, entropy, lse, spx, dlogits, d_stride, x.ring, x.extra,               \
                           x.base, x.word, max_polls, tag_offset);                                                    \
    } else {                                                                                                          \
      hipLaunchKernelGGL((RELAX_AMD_SPLIT_LDS_KERNEL(NVF, PARTIAL, false)), grid, block, 0, stream, logits,          \
                         row_stride, vocab, n_rows, token_of_row, sample_ids, targets, inv_t * kLog2e, inv_t, a,     \
                         grad_scale, log_prob, entropy, lse, spx, dlogits, d_stride, x.ring, x.extra,                 \
                         x.base, x.word, max_polls, tag_offset);                                                      \
    }                                                                                                                 \
    return check_launch("actor_step_split");                                                                          \
  }

template <typename T>
int launch_actor_step_split(const T* logits, int64_t row_stride, int64_t vocab, int64_t n_rows,
                            const int32_t* token_of_row, const int32_t* sample_ids, const int64_t* targets,
                            float inv_t, const relax_amd_policy_loss_args& a, float grad_scale, float* log_prob,
                            float* entropy, float* lse, float* spx, T* dlogits, int64_t d_stride,
                            hipStream_t stream) {
  constexpr int VN = Row<T>::kPerVec;
  const int width = scan_threads(vocab, VN);  // the virtual threads of a row: the forward-only kernel's workgroup
  if (vocab % VN != 0 || width < 512 || n_rows * kSplit > 2147483647LL) return RELAX_AMD_EUNSUPPORTED;
  const int64_t nvec = vocab / VN;
  const int full = int(nvec / width);
  const bool partial = nvec % width != 0;
  // the row shapes launch_actor_step_resident is built for, and 16-bit rows of 3585 .. 4096 and 6145 .. 6656 vectors
  // (32000 / 32768 and 50304 entries) scanned by 512 virtual threads
  if (width == 512) {
    if (sizeof(T) != 2 || !((full == 7 && partial) || (full == 8 && !partial) || (full == 12 && partial)))
      return RELAX_AMD_EUNSUPPORTED;
  } else if constexpr (sizeof(T) == 2) {
    const bool lds_row = (full == 24 && partial) || (full == 30 && partial) || (full == 31 && partial) ||
                         (full == 32 && !partial);
    if (!(lds_row || (full == 20 && !partial) || (full == 19 && partial) || (full == 18 && partial) ||
          (full == 15 && partial) || (full == 16 && !partial) || (full == 12 && partial) || (full == 8 && !partial) ||
          (full == 7 && partial)))
      return RELAX_AMD_EUNSUPPORTED;
  } else {
    // fp32: 100352 / 102400 (25088 / 25600 vectors), 128256 / 129280 (32064 / 32320), 131072 (32768), 151936 / 152064 /
    // 154880 (37984 / 38016 / 38720), 163840 (40960), 248320 (62080; the top-K term is left to the two-walk kernel)
    const bool lds_row = (full == 24 && partial) || (full == 25 && !partial) || (full == 31 && partial) ||
                         (full == 32 && !partial) || (full == 37 && partial) || (full == 40 && !partial) ||
                         (full == 60 && partial);
    if (full == 60 && a.topk_ids) return RELAX_AMD_EUNSUPPORTED;
    if (!(lds_row || (full == 7 && partial) || (full == 8 && !partial) || (full == 12 && partial) ||
          (full == 15 && partial) || (full == 16 && !partial)))
      return RELAX_AMD_EUNSUPPORTED;
  }
  ExchangeLaunch x;
  if (int rc = open_split_exchange(x, stream, n_rows, false)) return rc;
  const unsigned max_polls = exchange_max_polls();
  const unsigned tag_offset = exchange_wait_tag_offset();
  const dim3 grid(static_cast<unsigned>(n_rows * (width / kSplitThreads))), block(kSplitThreads);
  if constexpr (sizeof(T) == 2) {
    RELAX_AMD_SPLIT_ROW(512, 7, true)
    RELAX_AMD_SPLIT_ROW(512, 8, false)
    RELAX_AMD_SPLIT_ROW(512, 12, true)
    // 200064 / 201088 / 202048 (25008 / 25136 / 25256 vectors), 250880 (31360), 256000 (32000), 262144 (32768) entries
    RELAX_AMD_SPLIT_LDS(24, true, true)
    RELAX_AMD_SPLIT_LDS(30, true, true)
    RELAX_AMD_SPLIT_LDS(31, true, true)
    RELAX_AMD_SPLIT_LDS(32, false, true)
    RELAX_AMD_SPLIT(20, false)
    RELAX_AMD_SPLIT(19, true)
    RELAX_AMD_SPLIT(18, true)
    RELAX_AMD_SPLIT(15, true)
    RELAX_AMD_SPLIT(16, false)
    RELAX_AMD_SPLIT(12, true)
    RELAX_AMD_SPLIT(8, false)
    RELAX_AMD_SPLIT(7, true)
  } else {
    RELAX_AMD_SPLIT_LDS(37, true, true)
    RELAX_AMD_SPLIT_LDS(31, true, true)
    RELAX_AMD_SPLIT_LDS(32, false, true)
    RELAX_AMD_SPLIT_LDS(40, false, true)
    RELAX_AMD_SPLIT_LDS(24, true, true)
    RELAX_AMD_SPLIT_LDS(25, false, true)
    RELAX_AMD_SPLIT_LDS(60, true, false)
    RELAX_AMD_SPLIT(7, true)
    RELAX_AMD_SPLIT(8, false)
    RELAX_AMD_SPLIT(12, true)
    RELAX_AMD_SPLIT(15, true)
    RELAX_AMD_SPLIT(16, false)
  }
  return RELAX_AMD_EUNSUPPORTED;
}
#undef RELAX_AMD_SPLIT_LDS
#undef RELAX_AMD_SPLIT_LDS_KERNEL
#undef RELAX_AMD_SPLIT
#undef RELAX_AMD_SPLIT_ROW
#undef RELAX_AMD_SPLIT_KERNEL


template int launch_actor_step_split<float>(const float*, int64_t, int64_t, int64_t, const int32_t*, const int32_t*,
                                            const int64_t*, float, const relax_amd_policy_loss_args&, float, float*,
                                            float*, float*, float*, float*, int64_t, hipStream_t);
template int launch_actor_step_split<bf16_t>(const bf16_t*, int64_t, int64_t, int64_t, const int32_t*, const int32_t*,
                                             const int64_t*, float, const relax_amd_policy_loss_args&, float, float*,
                                             float*, float*, float*, bf16_t*, int64_t, hipStream_t);
template int launch_actor_step_split<f16_t>(const f16_t*, int64_t, int64_t, int64_t, const int32_t*, const int32_t*,
                                            const int64_t*, float, const relax_amd_policy_loss_args&, float, float*,
                                            float*, float*, float*, f16_t*, int64_t, hipStream_t);

}  // namespace relax_amd


extern "C" int relax_amd_set_exchange_wait(int max_polls, int wait_tag_offset) {
  if (max_polls < 0 || wait_tag_offset < 0) {
    relax_amd::set_error("set_exchange_wait: negative argument");
    return RELAX_AMD_EINVAL;
  }
  relax_amd::g_max_polls.store(max_polls == 0 ? relax_amd::kWaitPolls : unsigned(max_polls), std::memory_order_relaxed);
  relax_amd::g_wait_tag_offset.store(unsigned(wait_tag_offset), std::memory_order_relaxed);
  return RELAX_AMD_OK;
}

extern "C" int relax_amd_advance_exchange_tags(uint32_t used) {
  using namespace relax_amd;
  if (int rc = exchange_advance_tags<kRingWords>(split_family, reinterpret_cast<const void*>(&split_rings), used))
    return rc;
  return kl_advance_exchange_tags(used);
}
