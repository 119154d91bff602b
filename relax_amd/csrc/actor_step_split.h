// Kernel of the one-shot actor step (actor_step_split.hip: layout, exchange and figures there), shared with the
// instantiations for rows of any length and alignment (actor_step_split_any.hip).
#pragma once

#include <type_traits>

#include "device_utils.h"
#include "loss_math.h"
#include "opd_topk_math.h"
#include "row_exchange.h"
#include "row_scan.h"

namespace relax_amd {

constexpr int kRowWaves = 16;             // waves of the 1024 virtual threads of a row
constexpr int kSlotWords = kRowWaves * 3;
constexpr int kSplitThreads = 128;        // virtual threads per workgroup
constexpr int kSplit = 1024 / kSplitThreads;
constexpr size_t kRingWords = size_t(kRing) * kSlotWords;
constexpr size_t kTopkRingWords = size_t(kRing) * RELAX_AMD_FUSED_TOPK_MAX;

// the ring and the tags of an actor step about to be enqueued (actor_step_split.hip)
int open_split_exchange(ExchangeLaunch& x, hipStream_t stream, int64_t n_rows, bool own_ring_only);

// scan_absorb() over the values of kScanUnroll raw vectors (as in actor_step_resident.hip: same arithmetic, same
// order)
// KEEP: whether the second walk may use the values the first one unpacked (32 registers for 16-bit rows); without, the
// raw vectors are marked as changed in between, so that the compiler unpacks them again
template <typename T, bool KEEP = true>
__device__ __forceinline__ void split_absorb_raw_group(u32x4* raw, float c, SoftmaxAcc& st) {
  constexpr int VN = Row<T>::kPerVec;
  float vmax = 0.f;
#pragma unroll
  for (int u = 0; u < kScanUnroll; ++u) {
    float v[VN];
    Row<T>::unpack(raw[u], v);
#pragma unroll
    for (int k = 0; k < VN; ++k) vmax = (u == 0 && k == 0) ? v[0] : fmaxf(vmax, v[k]);
    __builtin_amdgcn_sched_barrier(0);
  }
  const float mc = __fmul_rn(vmax, c);
  if (mc > st.m) {
    const float sc = fast_exp2(fmaf(-vmax, c, st.m));  // one rounding, spelled out (see scan_finish)
    st.s = __fmul_rn(st.s, sc);
    st.t = __fmul_rn(st.t, sc);
    st.m = mc;
  }
#pragma unroll
  for (int u = 0; u < kScanUnroll; ++u) {
    if constexpr (!KEEP) asm volatile("" : "+v"(raw[u].x), "+v"(raw[u].y), "+v"(raw[u].z), "+v"(raw[u].w));
    float v[VN];
    Row<T>::unpack(raw[u], v);  // the compiler keeps the first walk's values: with wave 0's share parked in LDS
                                // during thread 0's arithmetic there is room for them next to the row
#pragma unroll
    for (int k = 0; k < VN; ++k) {
      const float e = fast_exp2(fmaf(v[k], c, -st.m));
      st.s = __fadd_rn(st.s, e);
      st.t = fmaf(e, v[k], st.t);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Lane 0's triple of this wave (the butterfly's merge is not symmetric in its last bits: scan_block_merge() takes lane
// 0's) into the row's slot, as three tagged words written by lanes 0..2.
__device__ __forceinline__ void split_publish(unsigned long long* slot, unsigned tag, int vt, const SoftmaxAcc& st) {
  const float m0 = lane_value(st.m), s0 = lane_value(st.s), t0 = lane_value(st.t);
  const int lane = vt & (kWave - 1), vwave = vt / kWave;
  if (lane < 3) {
    const float val = lane == 0 ? m0 : (lane == 1 ? s0 : t0);
    exchange_store(slot + vwave * 3 + lane, tag, val);
  }
}

// Wave 0 of a workgroup: lanes 0 .. 3 * ROW_WAVES - 1 fetch one word of the row's triples each (waiting, boundedly,
// for the tag of this launch and lap), then every lane merges the ROW_WAVES triples in wave order, as thread 0 of a
// workgroup of that many waves does in scan_block_merge().
template <int ROW_WAVES = kRowWaves>
__device__ __forceinline__ SoftmaxAcc split_collect(const unsigned long long* slot, unsigned tag, int tid,
                                                    unsigned max_polls, unsigned* status, unsigned first_tag,
                                                    bool& any_gave_up) {
  float word = 0.f;
  bool gave_up = false;
  if (tid < ROW_WAVES * 3) gave_up = !exchange_wait(slot + tid, tag, max_polls, status, first_tag, word);
  any_gave_up = __any(gave_up);
  if (any_gave_up && tid == 0) exchange_report_give_up(status, first_tag);
  auto of_lane = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(word), l)); };
  SoftmaxAcc whole{of_lane(0), of_lane(1), of_lane(2)};
#pragma unroll
  for (int i = 1; i < ROW_WAVES; ++i) scan_merge(whole, of_lane(3 * i), of_lane(3 * i + 1), of_lane(3 * i + 2));
  return whole;
}

// this workgroup's LDS_VECS x 128 vectors of the row that live in LDS (only instantiated, and only allocated, for
// LDS_VECS > 0)
template <int LDS_VECS>
__device__ __forceinline__ u32x4* split_lds_rows() {
  __shared__ u32x4 rows[LDS_VECS * kSplitThreads];
  return rows;
}

// where wave 0's share waits during thread 0's serial stretch (only instantiated, and only allocated, for PARK > 0)
template <int PARK>
__device__ __forceinline__ u32x4 (*split_parked())[kWave] {
  __shared__ u32x4 parked[PARK][kWave];
  return parked;
}

// ROW_THREADS: the virtual threads that scan a row, i.e. the width scan_threads() gives the forward-only kernel for this
// row length (1024, or 512 for rows of 2048 .. 7167 vectors); ROW_THREADS / 128 workgroups share a row.
// WAVES_MIN / WAVES_MAX: the waves per SIMD the register allocation aims for (see split_waves_min()).
// LDS_VECS: rows longer than the register file holds at three waves per SIMD (16-bit vocabularies above 163840 entries)
// keep the first LDS_VECS vectors of every thread's share in LDS, where global -> LDS loads put them without a
// register in between; wave 0 then has registers to spare for thread 0's serial stretch and parks nothing.
// ANY: the row may begin at any element and end anywhere: NVF is the least number of full vector positions and a thread
// has up to NVF + 2 vectors, as the row's length says; the vocab % VN elements behind the last whole vector go to virtual
// threads 0, 1, ..., one each, after their vectors (scan_row()'s order).
template <typename T, int NVF, bool PARTIAL, bool TOPK, int ROW_THREADS, int WAVES_MIN, int WAVES_MAX, int LDS_VECS = 0,
          bool ANY = false>
__global__ __launch_bounds__(kSplitThreads) __attribute__((amdgpu_waves_per_eu(WAVES_MIN, WAVES_MAX)))
void actor_step_split_kernel(
    const T* __restrict__ logits, int64_t row_stride, int64_t vocab, int64_t n_rows,
    const int32_t* __restrict__ token_of_row, const int32_t* __restrict__ sample_ids,
    const int64_t* __restrict__ targets, float c, float inv_t, relax_amd_policy_loss_args a, float grad_scale,
    float* __restrict__ log_prob, float* __restrict__ entropy, float* __restrict__ lse_out,
    float* __restrict__ spx_out, T* __restrict__ dlogits, int64_t d_stride, unsigned long long* __restrict__ ring,
    unsigned long long* __restrict__ topk_ring, unsigned tag_base, const unsigned* __restrict__ tag_word,
    unsigned max_polls, unsigned wait_tag_offset) {
  constexpr int kU = kScanUnroll, kParts = ROW_THREADS / kSplitThreads;
  constexpr int VN = Row<T>::kPerVec;
  constexpr int NV = NVF + (ANY ? 2 : PARTIAL ? 1 : 0);
  constexpr int kGroups = (NV + kU - 1) / kU;
  __shared__ float bc[5];
  __shared__ int64_t bc_target;
  __shared__ float topk_stage[TOPK ? kTopkStageFloats : 1];
  // vectors of wave 0's share that wait in LDS during thread 0's serial stretch (see there): all of them, or as many
  // as leave room for eight workgroups per CU next to the top-K term's staging area
  constexpr int kPark = LDS_VECS > 0 ? 0 : (NV < (TOPK ? 15 : 19) ? NV : (TOPK ? 15 : 19));
  u32x4(*parked)[kWave] = nullptr;
  if constexpr (kPark > 0) parked = split_parked<kPark>();
  constexpr int NR = NV - LDS_VECS;  // vectors of the share in registers
  static_assert(LDS_VECS <= NVF && NR >= kU, "only full vector positions go to LDS");
  const int tid = threadIdx.x;
  const bool wave0 = __builtin_amdgcn_readfirstlane(tid) < kWave;
  const unsigned part = blockIdx.x % kParts;
  const int64_t row = blockIdx.x / kParts;
  const int vt = int(part) * kSplitThreads + tid;  // virtual thread of the row
  const int rem = int(vocab / VN) - NVF * ROW_THREADS;
  auto has = [&](int j) -> bool {
    if constexpr (ANY) return j < NVF || vt + (j - NVF) * ROW_THREADS < rem;
    return j < NVF || (PARTIAL && j == NVF && vt < rem);
  };
  using Vec = std::conditional_t<ANY, any_vec, u32x4>;
  Vec* dv = reinterpret_cast<Vec*>(dlogits + row * d_stride);
  // this thread's element behind the last whole vector, or -1
  [[maybe_unused]] const int64_t tail_at = ANY && vt < int(vocab % VN) ? vocab / VN * VN + vt : -1;

  // token of the row, or -1 when the row scores nothing or both of its masks are zero (uniform over the workgroup)
  int64_t tok = token_of_row ? int64_t(token_of_row[row]) : row;
  const int64_t t0 = tok;
  if (tok >= 0) {
    const float m = a.loss_mask[tok];
    const float mp = a.pg_loss_mask ? a.pg_loss_mask[tok] : m;
    if (m == 0.f && mp == 0.f && !a.read_masked_rows) tok = -1;
  }
  if (tok < 0) {  // a zero row: no read, no exchange
    if (t0 >= 0 && part == 0 && tid == 0) {
      log_prob[t0] = 0.f;
      entropy[t0] = 0.f;
      lse_out[t0] = 0.f;
      spx_out[t0] = 0.f;
      a.coef_log_prob[t0] = 0.f;
      if (a.coef_entropy) a.coef_entropy[t0] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (has(j)) store_stream(dv + vt + j * ROW_THREADS, u32x4{0u, 0u, 0u, 0u});
    if constexpr (ANY)
      if (tail_at >= 0) Row<T>::store1(dlogits + row * d_stride + tail_at, 0.f);
    return;
  }

  const Vec* xv = reinterpret_cast<const Vec*>(logits + row * row_stride);
  // this workgroup's share of the row's K gathered logits: entries part * chunk .. + chunk, one per lane of the second
  // wave; the id is requested ahead of the row, the logit behind it
  int my_k = -1;
  int64_t my_id = -1;
  if constexpr (TOPK) {
    const int kmax = a.topk_k, chunk = (kmax + kParts - 1) / kParts, t1 = tid - kWave;
    if (t1 >= 0 && t1 < chunk && int(part) * chunk + t1 < kmax) {
      my_k = int(part) * chunk + t1;
      my_id = a.topk_ids[tok * kmax + my_k];
    }
  }
  u32x4 reg[NR];
  if constexpr (LDS_VECS > 0) {
    u32x4* rows = split_lds_rows<LDS_VECS>();
    const int wave_base = __builtin_amdgcn_readfirstlane(tid / kWave) * kWave;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if (j < LDS_VECS)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(xv + vt + j * ROW_THREADS),
                                         (__attribute__((address_space(3))) void*)(rows + j * kSplitThreads + wave_base),
                                         16, 0, 0);
      else if (has(j))
        reg[j - LDS_VECS] = load_stream(xv + vt + j * ROW_THREADS);
    }
  } else {
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (has(j)) reg[j] = load_stream(xv + vt + j * ROW_THREADS);
  }
  float tail_x = 0.f;
  if constexpr (ANY)
    if (tail_at >= 0) tail_x = Row<T>::load1(logits + row * row_stride + tail_at);
  // vector j of this thread's share
  auto vec = [&](int j) -> u32x4 {
    if constexpr (LDS_VECS > 0) {
      if (j < LDS_VECS) return split_lds_rows<LDS_VECS>()[(j < LDS_VECS ? j : 0) * kSplitThreads + tid];
    }
    return reg[j < LDS_VECS ? 0 : j - LDS_VECS];
  };
  const unsigned first_tag = exchange_first_tag(tag_base, tag_word), tag = first_tag + unsigned(row / kRing);
  float my_gathered = 0.f;
  if constexpr (TOPK) {
    if (my_k >= 0) my_gathered = topk_gather_one<T>(a, logits + row * row_stride, vocab, my_id);
  }

  // the scan, group by group as the vectors arrive, in scan_row()'s order
  SoftmaxAcc st{kNegHuge, 0.f, 0.f};
  bool grouped = true;
#pragma unroll
  for (int g = 0; g < kGroups; ++g) {
    if (grouped && kU * g + kU - 1 < NV && has(kU * g + kU - 1)) {
      if constexpr (LDS_VECS > 0) {
        u32x4 grp[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) grp[u] = vec((kU * g < NV - kU ? kU * g : NV - kU) + u);
        split_absorb_raw_group<T, false>(grp, c, st);
      } else {
        split_absorb_raw_group<T>(&reg[kU * g < NV - kU ? kU * g : NV - kU], c, st);
      }
    } else {
      grouped = false;
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (kU * g + u < NV && has(kU * g + u)) {
          float v[VN];
          Row<T>::unpack(vec(kU * g + u < NV ? kU * g + u : NV - 1), v);
          scan_absorb(v, c, st);
        }
    }
    asm volatile("" : "+v"(st.m), "+v"(st.s), "+v"(st.t));
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (ANY)
    if (tail_at >= 0) {
      float v[1] = {tail_x};
      scan_absorb(v, c, st);
    }
  // each wave to its triple (scan_block_merge()'s first half), published by its lanes 0..2
  wave_butterfly([&](auto o) {
    constexpr int O = decltype(o)::value;
    scan_merge(st, lane_xor<O>(st.m), lane_xor<O>(st.s), lane_xor<O>(st.t));
  });
  unsigned long long* slot = ring + size_t(row % kRing) * kSlotWords;
  split_publish(slot, tag, vt, st);
  unsigned long long* topk_slot = nullptr;
  if constexpr (TOPK) {
    topk_slot = topk_ring + size_t(row % kRing) * RELAX_AMD_FUSED_TOPK_MAX;
    if (my_k >= 0) exchange_store(topk_slot + my_k, tag, my_gathered);
  }

  if (wave0) {
    // thread 0 runs a serial stretch from here to the barrier while the other waves of the workgroup wait
    __builtin_amdgcn_s_setprio(3);
    // wave 0's share of the row waits in LDS meanwhile: thread 0's loss arithmetic needs some thirty registers of its
    // own, which every wave of the kernel would otherwise have to set aside next to the row
#pragma unroll
    for (int j = 0; j < kPark; ++j) parked[j][tid] = reg[j];
    // thread 0's view of the token, fetched while the triples travel
    TokenInputs tin{};
    float x_target = 0.f, den = 1.f, pg_den = 1.f;
    int64_t tg = -1;
    if (tid == 0) {
      tin = load_token_inputs(a, tok);
      tg = targets[tok];
      if (tg >= 0 && tg < vocab) x_target = Row<T>::load1(logits + row * row_stride + tg);
      const int32_t sid = sample_ids ? sample_ids[tok] : 0;
      den = a.sample_denom ? a.sample_denom[sid] : 1.0f;
      pg_den = a.pg_sample_denom ? a.pg_sample_denom[sid] : den;
    }
    TopkGather gathered{};
    TopkRowShape topk_shape{};
    if constexpr (TOPK) {
      int lane = tid;
      asm volatile("" : "+v"(lane));
      gathered = topk_gather_meta(a, tok, lane);
      topk_shape = topk_row_shape(a, tok);
    }
    bool any_gave_up = false;
    const SoftmaxAcc whole = split_collect<ROW_THREADS / kWave>(slot, tag + wait_tag_offset, tid, max_polls,
                                                                reinterpret_cast<unsigned*>(ring + kRingWords),
                                                                first_tag, any_gave_up);
    if constexpr (TOPK) {
      // the row's gathered logits, entry lane + 64 i from the workgroup that fetched it
      unsigned* status = reinterpret_cast<unsigned*>(ring + kRingWords);
      bool gave_up = any_gave_up;
#pragma unroll
      for (int i = 0; i < kTopkPerLane; ++i) {
        const int k = tid + i * kWave;
        if (k < a.topk_k && !gave_up)
          gave_up = !exchange_wait(topk_slot + k, tag + wait_tag_offset, max_polls, status, first_tag, gathered.x[i]);
      }
      const bool any_topk_gave_up = __any(gave_up);
      if (any_topk_gave_up && !any_gave_up && tid == 0) exchange_report_give_up(status, first_tag);
      any_gave_up = any_topk_gave_up;
    }
    float lse = 0.f, spx = 0.f, ent = 0.f, lp = 0.f;
    if (tid == 0) {
      scan_finish(whole, x_target, tg >= 0 && tg < vocab, inv_t, lse, spx, ent, lp);
      if (any_gave_up) lp = lse = __builtin_nanf("");
      if (part == 0) {
        log_prob[tok] = lp;
        entropy[tok] = ent;
        lse_out[tok] = lse;
        spx_out[tok] = spx;
      }
    }
    float g_topk = 0.f;
    if constexpr (TOPK) {
      int lane = tid;
      asm volatile("" : "+v"(lane));
      g_topk = topk_distill_row(a, gathered, topk_shape, tok, lane_value(lse), inv_t, lane_value(lp),
                                lane_value(tin.has_old ? tin.old_lp : lp), lane_value(tin.extra_lp), lane, topk_stage,
                                part == 0);
    }
    if (tid == 0) {
      relax_amd_policy_loss_args al = a;
      asm volatile("" : "+s"(al.eps_clip), "+s"(al.eps_clip_high), "+s"(al.eps_clip_c), "+s"(al.entropy_coef),
                   "+s"(al.kl_coef), "+s"(al.tis_lo), "+s"(al.tis_hi), "+s"(al.tau_pos), "+s"(al.tau_neg));
      const TokenResult tr = token_terms(al, tin, lp, ent, false, 0.f, den, pg_den);
      if (part == 0) {
        a.coef_log_prob[tok] = tr.coef_lp;
        if (a.coef_entropy) a.coef_entropy[tok] = tr.coef_ent;
      }
      const float glp = tr.coef_lp * grad_scale, gh = tr.coef_ent * grad_scale;
      const float gsm = TOPK ? glp + g_topk * grad_scale : glp;
      const float b = gh * inv_t;
      bc[0] = -lse * kLog2e;           // k0: p = exp2(x*c + k0)
      bc[1] = -gsm * inv_t + b * spx;  // a0
      bc[2] = -b * inv_t;              // a1: d = p * (a0 + a1*x)
      bc[3] = glp * inv_t;             // added at the target
      bc[4] = (gsm == 0.f && glp == 0.f && gh == 0.f) ? 1.f : 0.f;
      bc_target = tg;
    }
#pragma unroll
    for (int j = 0; j < kPark; ++j) reg[j] = parked[j][tid];
    __builtin_amdgcn_s_setprio(0);
  }
  __syncthreads();
  const float k0 = bc[0], a0 = bc[1], a1 = bc[2], hot = bc[3];
  const int64_t tgt = bc_target;
  const bool emit_zero = bc[4] != 0.f;
  const int tvec = (tgt >= 0 && tgt < vocab) ? int(tgt / VN) : -1;
  const int tsub = int(tgt % VN);
  if (emit_zero) {  // uniform over the workgroup: both gradient coefficients vanish, a zero row whatever the logits hold
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (has(j)) store_stream(dv + vt + j * ROW_THREADS, u32x4{0u, 0u, 0u, 0u});
    if constexpr (ANY)
      if (tail_at >= 0) Row<T>::store1(dlogits + row * d_stride + tail_at, 0.f);
    return;
  }
  if constexpr (ANY)
    if (tail_at >= 0) {
      float g = fast_exp2(fmaf(tail_x, c, k0)) * fmaf(tail_x, a1, a0);
      if (tail_at == tgt) g += hot;
      Row<T>::store1(dlogits + row * d_stride + tail_at, g);
    }
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    int lane_id = vt;
    asm volatile("" : "+v"(lane_id));
    const int idx = lane_id + j * ROW_THREADS;
    float v[VN];
    Row<T>::unpack(vec(j), v);
#pragma unroll
    for (int k = 0; k < VN; ++k) {
      v[k] = fast_exp2(fmaf(v[k], c, k0)) * fmaf(v[k], a1, a0);
      if (k == VN / 2 - 1) __builtin_amdgcn_sched_barrier(0);
    }
    u32x4 out = Row<T>::pack(v);
    // The element at the target gets `hot` added before it is rounded.  One wave in 300 holds it: that wave takes a
    // jump (the ballot is wave-uniform) and packs the vector again; as a per-lane select on every vector the same
    // update costs two vector instructions per element, an eighth of the kernel's arithmetic.
    if (__builtin_amdgcn_ballot_w64(idx == tvec) != 0ull) {
#pragma unroll
      for (int k = 0; k < VN; ++k)
        if (idx == tvec && k == tsub) v[k] += hot;
      out = Row<T>::pack(v);
    }
    if (has(j)) store_stream(dv + idx, out);
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace relax_amd
