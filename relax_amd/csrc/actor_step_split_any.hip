// The one-shot actor step (actor_step_split.hip) for rows of any length that begin at any element: vocabularies extended
// by a few tokens, odd row strides, lengths that no model of the built list has.  Same bits as the two-walk kernel, which
// these rows took before: it reads a row twice (the second time out of cache) and keeps one workgroup per row.
//
// What bounds it: the memory system's rate for accesses that straddle its lines (reads + writes of 2 GiB at odd
// 2-byte offsets 5.2 TB/s, 6.2 aligned).  Kernel time, two-walk -> this, 1.2 GB of bf16 logits with 20 % of the tokens
// masked: rows of 17001 entries 602 -> 491 us, 32003 516 -> 461, 50261 513 -> 465, 75003 527 -> 425, 110003 558 -> 436,
// 155001 578 -> 438; aligned rows of 40000 387 -> 356.  fp32 rows at 4-byte offsets gain nothing (32001 entries 387 ->
// 401, 65001 415 -> 408) and keep the two-walk kernel.
// hipcc-flags: -mllvm -amdgpu-use-amdgpu-trackers=1
#include "actor_step_resident.h"
#include "actor_step_split.h"

namespace relax_amd {

template <int NVF>
constexpr int any_waves_min() {
  return NVF + 2 >= 15 ? 3 : 4;  // as split_waves_min()
}
template <int NVF>
constexpr int any_waves_max() {
  return NVF + 2 >= 15 ? 3 : 8;
}

// One instantiation serves two row widths' worth of lengths (NVF .. NVF + 2 vectors per virtual thread).
#define RELAX_AMD_SPLIT_ANY(WIDTH, NVF)                                                                               \
  if (width == WIDTH && nvec >= int64_t(NVF) * WIDTH && nvec <= int64_t(NVF + 2) * WIDTH) {                           \
    hipLaunchKernelGGL((actor_step_split_kernel<T, NVF, false, false, WIDTH, any_waves_min<NVF>(),                    \
                                                any_waves_max<NVF>(), 0, true>),                                      \
                       dim3(static_cast<unsigned>(n_rows * (width / kSplitThreads))), dim3(kSplitThreads), 0, stream, \
                       logits, row_stride, vocab, n_rows, token_of_row, sample_ids, targets, inv_t * kLog2e, inv_t,   \
                       a, grad_scale, log_prob, entropy, lse, spx, dlogits, d_stride, x.ring, nullptr, x.base,       \
                       nullptr, exchange_max_polls(), exchange_wait_tag_offset());                                    \
    return check_launch("actor_step_split");                                                                          \
  }

template <typename T>
int launch_actor_step_split_any(const T* logits, int64_t row_stride, int64_t vocab, int64_t n_rows,
                                const int32_t* token_of_row, const int32_t* sample_ids, const int64_t* targets,
                                float inv_t, const relax_amd_policy_loss_args& a, float grad_scale, float* log_prob,
                                float* entropy, float* lse, float* spx, T* dlogits, int64_t d_stride,
                                hipStream_t stream) {
  constexpr int VN = Row<T>::kPerVec;
  static_assert(VN == 8, "16-bit rows");
  const int width = scan_threads(vocab, VN);
  const int64_t nvec = vocab / VN;
  // 16-bit rows of up to the 20 vectors per thread that the register file holds; the top-K term is left to the two-walk
  // kernel
  if (nvec < 4 * 512 || nvec > 20 * 1024 || a.topk_ids || n_rows * kSplit > 2147483647LL) return RELAX_AMD_EUNSUPPORTED;
  // streams without an exchange ring of their own and captured launches are left to the two-walk kernel
  ExchangeLaunch x;
  if (int rc = open_split_exchange(x, stream, n_rows, true)) return rc;
  RELAX_AMD_SPLIT_ANY(512, 4)
  RELAX_AMD_SPLIT_ANY(512, 6)
  RELAX_AMD_SPLIT_ANY(512, 8)
  RELAX_AMD_SPLIT_ANY(512, 10)
  RELAX_AMD_SPLIT_ANY(512, 12)
  RELAX_AMD_SPLIT_ANY(1024, 7)
  RELAX_AMD_SPLIT_ANY(1024, 9)
  RELAX_AMD_SPLIT_ANY(1024, 11)
  RELAX_AMD_SPLIT_ANY(1024, 13)
  RELAX_AMD_SPLIT_ANY(1024, 15)
  RELAX_AMD_SPLIT_ANY(1024, 17)
  RELAX_AMD_SPLIT_ANY(1024, 18)
  return RELAX_AMD_EUNSUPPORTED;
}
#undef RELAX_AMD_SPLIT_ANY

template int launch_actor_step_split_any<bf16_t>(const bf16_t*, int64_t, int64_t, int64_t, const int32_t*,
                                                 const int32_t*, const int64_t*, float,
                                                 const relax_amd_policy_loss_args&, float, float*, float*, float*,
                                                 float*, bf16_t*, int64_t, hipStream_t);
template int launch_actor_step_split_any<f16_t>(const f16_t*, int64_t, int64_t, int64_t, const int32_t*,
                                                const int32_t*, const int64_t*, float,
                                                const relax_amd_policy_loss_args&, float, float*, float*, float*,
                                                float*, f16_t*, int64_t, hipStream_t);

}  // namespace relax_amd
