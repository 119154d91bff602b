// Fused LM-head projection + log-prob / entropy: logits = hidden @ weight^T are produced tile by tile on the bf16
// matrix cores (v_mfma_f32_32x32x16_bf16) and consumed in registers, so the [N, V] logits never reach HBM.
//
// Replaces the deferred-LM-head path of relax/backends/megatron/loss.py:391-419 (per 1024-row sub-chunk:
// F.linear -> .float() -> /T -> calculate_log_probs_and_entropy), and adds the entropy the reference leaves out.
//
// Tiling.  A workgroup (256 threads = 4 wave64) owns 256 tokens and walks a range of 256-wide vocabulary tiles; the
// K loop over the hidden size runs in 64-wide slices through a two-stage LDS ring (2 x (256 + 256) rows x 128 B).
// Slices are copied global -> LDS directly (global_load_lds_dwordx4, no staging registers): every lane fetches one
// 16-byte vector and the wave's 64 vectors land contiguously, i.e. 8 rows x 128 B per instruction.  The LDS has 64
// four-byte banks and serves 16 lanes of a 16-byte read per clock, so the fragment reads of 16 consecutive rows (same
// k offset) must hit 16 distinct bank quads: with 128-byte rows the bank quad is (row parity, slot), hence lane
// (row r, slot v) fetches global vector v ^ ((r >> 1) & 7) and fragment reads apply the same XOR (no padding).
// The 16 copies of slice k+1 (or of the next vocabulary tile's first slice) are slotted between the 64 MFMAs of slice
// k, one per two MFMAs, and awaited at the slice boundary; fragments for the next 16-wide k-step are fetched from LDS
// while the current 16 MFMAs issue.
//
// The MFMA "A" operand is the WEIGHT tile and "B" the HIDDEN tile, so in the 32x32 accumulator layout a lane's column
// is a TOKEN and its 16 registers are 16 vocabulary entries: the online softmax over the vocabulary is then a
// per-lane reduction over 64 accumulator values per token (4 tokens per lane, 12 state registers), with one cross-lane
// and one cross-wave merge at the very end.  Each wave computes 128 vocab x 128 tokens = 4x4 MFMA tiles (256 fp32
// accumulators per lane, held in AGPRs).  Vocabulary ranges are split over workgroups (flash-decoding style) and
// merged by a small combine kernel; the target logit comes from a gather-dot kernel (one wave per token).
// The same pipeline drives the backward's recompute kernel, whose epilogue turns each accumulator block into the
// gradient w.r.t. the logits and stores it transposed in bf16, and the forward variant that keeps the bf16 logits.
//
// Workgroup -> (row block, vocab split): LmTaskGrid (lmhead_pipeline.h); the 32 workgroups resident on one XCD are up to
// 8 row blocks x 4 or more vocab splits, so that hidden and weight tiles are shared inside that XCD's L2.
//
// The split count.  A chip-wide round is 256 workgroups and the kernel lasts as many vocabulary tiles as the longest
// chain of workgroups on one CU walks, so lm_plan_splits() takes the split count that makes (rounds) x (tiles per split)
// smallest.  With powers of two up to 32 (what 32 workgroups per XCD divide into without strips) 26 row blocks of a
// 151936-entry vocabulary took two rounds of 38 tiles where one of 66 does it, and one row block left 224 of the 256
// CUs idle.  Forward at V = 151936, H = 4096: 250 response tokens 1726 -> 431 us, 4200 7350 -> 4077, 6640 7390 -> 6395.
#include <algorithm>
#include <mutex>

#include "device_utils.h"
#include "lmhead_pipeline.h"
#include "relax_amd.h"

namespace relax_amd {

// STORE: also writes the logits, rounded to bf16, into l_t [vocab, l_stride] (token contiguous), and takes the softmax
// statistics from the rounded values (what the reference's bf16 F.linear hands to its fp32 log-softmax), so that a
// backward pass reading l_t sees exactly the distribution the forward pass normalised.
template <bool STORE, bool PAIRS>
__global__ __launch_bounds__(kLmThreads, 1) void lmhead_fwd_kernel(const uint16_t* __restrict__ hidden,
                                                                   const uint16_t* __restrict__ weight, LmGeom g,
                                                                   float c, float* __restrict__ partial,
                                                                   uint16_t* __restrict__ l_t, int64_t l_stride,
                                                                   const LmLivePlan* __restrict__ live) {
  __shared__ __attribute__((aligned(1024))) unsigned char w0[kLmOperandBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char h0[kLmOperandBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char w1[kLmOperandBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char h1[kLmOperandBytes];
  unsigned char* smem = w0;
  lm_take_live(g, live);
  int rb, split;
  if (!lm_block_coords(g, rb, split)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wv = wave >> 1, wt = wave & 1;
  const int64_t tok0 = int64_t(rb) * kLmTile;
  float m[4], s[4], t[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    m[j] = kNegHuge;
    s[j] = 0.f;
    t[j] = 0.f;
  }
  const int vt_begin = split * g.tiles_per_split;
  const int vt_end = min(g.n_tiles, vt_begin + g.tiles_per_split);
  LmSlabWriter writer;
  if (STORE) writer.init(l_t, l_stride, g.vocab, g.n_tokens, tok0, wv, wt, lane);
  lm_pipeline<STORE>(LmLds{w0, h0, w1, h1}, hidden, weight, g, tok0, vt_begin, vt_end, [&](floatx16 (&acc)[4][4], int64_t v0) {
    const int limit = int(min<int64_t>(g.vocab - v0, kLmTile));
    if (STORE) writer.set_tile(v0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // one 16-value block at a time: without the barrier all 256 accumulators are copied out of the AGPRs first
        floatx16 blk = acc[i][j];
        if (STORE) {
          float x[16];
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            x[r] = blk[r];
            x[r + 1] = blk[r + 1];
            const uint32_t pk = pack_bf16(x[r], x[r + 1]);
            blk[r] = bf16_lo(pk);
            blk[r + 1] = bf16_hi(pk);
          }
          writer.template store<PAIRS>(x, i, j);
        }
        if (limit < kLmTile)  // ragged last tile: entries past the vocabulary are masked out
          lm_absorb_block<true>(blk, wv * 128 + i * 32 + 4 * (lane >> 5), limit, c, m[j], s[j], t[j]);
        else
          lm_absorb_block<false>(blk, 0, 0, c, m[j], s[j], t[j]);
        __builtin_amdgcn_sched_barrier(0);
      }
  });
  // merge the two lane halves (same tokens, different vocab rows), then the two waves sharing the tokens
  float* red = reinterpret_cast<float*>(smem);  // [2 (wv)][256 tokens][3]
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float m2 = lane_xor<32>(m[j]), s2 = lane_xor<32>(s[j]), t2 = lane_xor<32>(t[j]);
    const float mn = fmaxf(m[j], m2);
    const float fa = fast_exp2(m[j] - mn), fb = fast_exp2(m2 - mn);
    s[j] = s[j] * fa + s2 * fb;
    t[j] = t[j] * fa + t2 * fb;
    m[j] = mn;
    if (lane < 32) {
      float* o = red + (wv * kLmTile + wt * 128 + j * 32 + lane) * 3;
      o[0] = m[j];
      o[1] = s[j];
      o[2] = t[j];
    }
  }
  __syncthreads();
  const int64_t tok = tok0 + threadIdx.x;
  if (tok < g.n_tokens) {
    const float* a = red + threadIdx.x * 3;
    const float* b = red + (kLmTile + threadIdx.x) * 3;
    const float mn = fmaxf(a[0], b[0]);
    const float fa = fast_exp2(a[0] - mn), fb = fast_exp2(b[0] - mn);
    float* o = partial + (int64_t(split) * g.n_tokens + tok) * 3;
    o[0] = mn;
    o[1] = a[1] * fa + b[1] * fb;
    o[2] = a[2] * fa + b[2] * fb;
  }
}

// logits[target] per token: one wave per token, fp32 accumulation of bf16 products.
__global__ __launch_bounds__(256) void lmhead_target_logit_kernel(const uint16_t* __restrict__ hidden,
                                                                  const uint16_t* __restrict__ weight, LmGeom g,
                                                                  const int64_t* __restrict__ targets,
                                                                  float* __restrict__ x_target) {
  const int lane = threadIdx.x & 63;
  const int64_t tok = blockIdx.x * 4LL + (threadIdx.x >> 6);
  if (tok >= g.n_tokens) return;
  const int64_t tg = targets[tok];
  if (tg < 0 || tg >= g.vocab) {
    if (lane == 0) x_target[tok] = __builtin_nanf("");
    return;
  }
  const u32x4* h = reinterpret_cast<const u32x4*>(hidden + tok * g.h_stride);
  const u32x4* w = reinterpret_cast<const u32x4*>(weight + tg * g.w_stride);
  float acc = 0.f;
  for (int64_t i = lane; i < g.hidden / 8; i += kWave) {
    float a[8], b[8];
    Row<bf16_t>::unpack(h[i], a);
    Row<bf16_t>::unpack(w[i], b);
#pragma unroll
    for (int k = 0; k < 8; ++k) acc = fmaf(a[k], b[k], acc);
  }
  acc = wave_sum(acc);
  if (lane == 0) x_target[tok] = acc;
}

// The per-split softmax partials of a token into its log-prob: one wave per token, a lane per split (a short input has
// hundreds of splits: one thread per token walked 198 of them in 58 us at 250 tokens, under 12 us this way).
__global__ __launch_bounds__(256) void lmhead_combine_kernel(const float* __restrict__ partial,
                                                             const float* __restrict__ x_target, int64_t n_tokens,
                                                             int splits, float inv_t, float* __restrict__ log_prob,
                                                             float* __restrict__ entropy, float* __restrict__ lse_out,
                                                             float* __restrict__ spx_out,
                                                             const LmLivePlan* __restrict__ live,
                                                             const int32_t* __restrict__ token_map) {
  if (live) n_tokens = live->n_tokens, splits = live->splits;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t tok = blockIdx.x * 4LL + threadIdx.x / kWave;
  if (tok >= n_tokens) return;
  float m = kNegHuge, s = 0.f, t = 0.f;
  auto merge = [&](float m2, float s2, float t2) {
    const float mn = fmaxf(m, m2);
    const float fa = fast_exp2(m - mn), fb = fast_exp2(m2 - mn);
    s = s * fa + s2 * fb;
    t = t * fa + t2 * fb;
    m = mn;
  };
  for (int k = lane; k < splits; k += kWave) {
    const float* p = partial + (int64_t(k) * n_tokens + tok) * 3;
    merge(p[0], p[1], p[2]);
  }
  wave_butterfly([&](auto o) {
    constexpr int O = decltype(o)::value;
    merge(lane_xor<O>(m), lane_xor<O>(s), lane_xor<O>(t));
  });
  if (lane != 0) return;
  const float lse = m * kLn2 + logf(s);
  const float spx = (t / s) * inv_t;
  log_prob[token_map ? token_map[tok] : tok] = x_target[tok] * inv_t - lse;
  if (entropy) entropy[tok] = lse - spx;
  if (lse_out) lse_out[tok] = lse;
  if (spx_out) spx_out[tok] = spx;
}

// Target logit read back from the stored bf16 logits (so log_prob uses the very value the statistics saw).
__global__ __launch_bounds__(256) void lmhead_target_from_logits_kernel(const uint16_t* __restrict__ l_t,
                                                                        int64_t l_stride, int64_t n_tokens,
                                                                        int64_t vocab,
                                                                        const int64_t* __restrict__ targets,
                                                                        float* __restrict__ x_target,
                                                                        const LmLivePlan* __restrict__ live) {
  if (live) n_tokens = live->n_tokens;
  const int64_t tok = blockIdx.x * 256LL + threadIdx.x;
  if (tok >= n_tokens) return;
  const int64_t tg = targets[tok];
  x_target[tok] = (tg < 0 || tg >= vocab) ? __builtin_nanf("") : bf16_lo(l_t[tg * l_stride + tok]);
}

// Backward from stored logits: overwrites l_t [vocab, stride] (bf16 logits, token contiguous) with the gradient
// dT[v, n] = inv_T * ( g_lp*(onehot - p) + g_H * p * (spx - x) ),  p = exp(x - lse)  -- the same expression the
// recomputing kernel evaluates on its accumulators.  A thread owns eight neighbouring tokens (one 16-byte access per
// vocabulary row) and keeps their per-token coefficients in registers while it walks `rows_per_block` rows.  Columns
// n_tokens .. ceil8(n_tokens) - 1 (the rest of the last 16-byte vector) are written as zeros, later ones not at all; with a
// live plan zeros go on to ceil128(n_tokens), where the backward products stop reading: nobody else knows that place.
constexpr int kLmInplaceThreads = 256;
__global__ __launch_bounds__(kLmInplaceThreads) void lmhead_dlogits_inplace_kernel(
    uint16_t* __restrict__ l_t, int64_t stride, int64_t n_tokens, int64_t vocab, int rows_per_block, float c,
    float inv_t, const int64_t* __restrict__ targets, const float* __restrict__ lse, const float* __restrict__ spx,
    const float* __restrict__ g_lp, const float* __restrict__ g_ent, const float* __restrict__ grad_scale_dev,
    const LmLivePlan* __restrict__ live) {
  if (live) n_tokens = live->n_tokens;
  const int64_t tok8 = (int64_t(blockIdx.x) * kLmInplaceThreads + threadIdx.x) * 8;
  if (tok8 >= (live ? (n_tokens + 127) / 128 * 128 : n_tokens)) return;
  const float gs = grad_scale_dev ? *grad_scale_dev : 1.0f;
  float k0[8], a0[8], a1[8], hot[8];
  int64_t tg[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int64_t tk = tok8 + k < n_tokens ? tok8 + k : n_tokens - 1;
    const float glp = g_lp[tk] * gs, gh = g_ent ? g_ent[tk] * gs : 0.f;
    const float b = gh * inv_t;
    k0[k] = -lse[tk] * kLog2e;
    a0[k] = -glp * inv_t + (g_ent ? b * spx[tk] : 0.f);
    a1[k] = -b * inv_t;
    hot[k] = glp * inv_t;
    tg[k] = tok8 + k < n_tokens ? targets[tk] : -1;
  }
  const int64_t v_begin = int64_t(blockIdx.y) * rows_per_block;
  const int64_t v_end = min<int64_t>(vocab, v_begin + rows_per_block);
  // four rows in flight per thread: the loads of a group are issued before its first store (in place, so the compiler
  // must not be asked to reorder them itself)
  for (int64_t v = v_begin; v < v_end; v += 4) {
    u32x4 raw[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (v + u < v_end) raw[u] = *reinterpret_cast<const u32x4*>(l_t + (v + u) * stride + tok8);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (v + u >= v_end) break;
      float x[8], d[8];
      Row<bf16_t>::unpack(raw[u], x);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        d[k] = fast_exp2(fmaf(x[k], c, k0[k])) * fmaf(x[k], a1[k], a0[k]);
        if (v + u == tg[k]) d[k] += hot[k];
        if (tok8 + k >= n_tokens) d[k] = 0.f;  // the vector's tail past the last token: padding, kept at zero
      }
      u32x4 o;
      o.x = pack_bf16(d[0], d[1]);
      o.y = pack_bf16(d[2], d[3]);
      o.z = pack_bf16(d[4], d[5]);
      o.w = pack_bf16(d[6], d[7]);
      *reinterpret_cast<u32x4*>(l_t + (v + u) * stride + tok8) = o;
    }
  }
}

// Which tokens of a micro-batch take part in a loss that is a weighted sum of log-probs, and how their projection is cut.
// A weight of zero (prompt remainder, tool output, truncation) leaves nothing of a token in the loss or in any gradient,
// so the projection, its backward products and the [V, N] slab carry the others only: a sixth to a third of a packed
// micro-batch's matrix work.  The count stays on the device (reading it back would stop the host until the GPU has
// caught up): this one-workgroup kernel numbers the live tokens in order and finds the split counts each slab's launches
// take; 8 us at 8192 tokens.
constexpr int kLmPlanThreads = 1024;
__global__ __launch_bounds__(kLmPlanThreads) void lmhead_live_plan_kernel(
    const float* __restrict__ token_weight, int64_t n, int64_t slab_tokens, int n_slabs, int n_tiles, int dh_cols,
    int dh_steps, int32_t* __restrict__ token_map, LmLivePlan* __restrict__ plans) {
  constexpr int kWaves = kLmPlanThreads / kWave;
  __shared__ int wave_count[kWaves];
  __shared__ unsigned long long best_fwd, best_dh;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  int64_t base = 0;
  for (int64_t i0 = 0; i0 < n; i0 += kLmPlanThreads) {
    const int64_t i = i0 + tid;
    const bool live = i < n && token_weight[i] != 0.f;
    const unsigned long long vote = __ballot(live);
    if (lane == 0) wave_count[wave] = __popcll(vote);
    __syncthreads();
    int64_t at = base;
    for (int w = 0; w < kWaves; ++w) {
      if (w < wave) at += wave_count[w];
      base += wave_count[w];
    }
    if (live) token_map[at + __popcll(vote & ((1ull << lane) - 1ull))] = int32_t(i);
    __syncthreads();
  }
  for (int slab = 0; slab < n_slabs; ++slab) {
    const int64_t left = base - slab * slab_tokens;
    const int64_t cnt = left < 0 ? 0 : (left < slab_tokens ? left : slab_tokens);
    const int64_t rows = (cnt + kLmTile - 1) / kLmTile;
    if (tid == 0) best_fwd = best_dh = ~0ull;
    __syncthreads();
    const int64_t s = tid + 1;
    if (rows > 0) {
      if (s <= lm_max_splits(rows) && s <= n_tiles)
        atomicMin(&best_fwd, (static_cast<unsigned long long>(lm_split_cost(rows, n_tiles, s)) << 16) | unsigned(s));
      if (s <= gemm_max_splits(rows) && s <= dh_steps)
        atomicMin(&best_dh, (static_cast<unsigned long long>(gemm_split_cost(rows * dh_cols, dh_steps, s)) << 16) | unsigned(s));
    }
    __syncthreads();
    if (tid == 0) {
      LmLivePlan p{};
      p.n_tokens = int(cnt);
      p.row_blocks = int(rows);
      p.splits = p.tiles_per_split = p.strip = p.dh_splits = p.dh_per_split = 1;
      if (rows > 0) {
        const int sf = int(best_fwd & 0xffffu), sd = int(best_dh & 0xffffu);
        p.tiles_per_split = (n_tiles + sf - 1) / sf;
        p.splits = (n_tiles + p.tiles_per_split - 1) / p.tiles_per_split;
        p.strip = lm_strip_height(rows);
        p.dh_per_split = (dh_steps + sd - 1) / sd;
        p.dh_splits = (dh_steps + p.dh_per_split - 1) / p.dh_per_split;
      }
      plans[slab] = p;
    }
    __syncthreads();
  }
}

// Rows, targets and d loss / d log-prob of the live tokens, side by side: one workgroup per place.
__global__ __launch_bounds__(256) void lmhead_live_gather_kernel(
    const uint16_t* __restrict__ rows, int64_t row_stride, int64_t hidden, const int32_t* __restrict__ row_ids,
    const int64_t* __restrict__ targets, const float* __restrict__ token_weight, float weight_scale,
    int64_t slab_tokens, const int32_t* __restrict__ token_map, const LmLivePlan* __restrict__ plans,
    uint16_t* __restrict__ picked, int64_t* __restrict__ picked_targets, float* __restrict__ g_lp,
    int32_t* __restrict__ row_map) {
  const int64_t i = blockIdx.x, slab = i / slab_tokens;
  if (i - slab * slab_tokens >= plans[slab].n_tokens) return;
  const int32_t tok = token_map[i], row = row_ids[tok];
  const any_vec* from = reinterpret_cast<const any_vec*>(rows + row * row_stride);
  u32x4* to = reinterpret_cast<u32x4*>(picked + i * hidden);
  for (int64_t k = threadIdx.x; k < hidden / 8; k += 256) to[k] = from[k];
  if (threadIdx.x == 0) {
    picked_targets[i] = targets[tok];
    g_lp[i] = token_weight[tok] * weight_scale;
    row_map[i] = row;
  }
}

// Backward helper: recompute one [chunk, V] slab of logits on the matrix cores and emit, transposed, the bf16
// gradient w.r.t. the logits  dT[v, n] = inv_T * ( g_lp*(onehot - p) + g_H * p * (spx - x) ),  p = exp(x - lse).
// dT is [vocab, chunk] (token-contiguous) so a lane's 32 neighbours write one 64-byte segment.
template <bool PAIRS>
__global__ __launch_bounds__(kLmThreads, 1) void lmhead_dlogits_kernel(
    const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ weight, LmGeom g, float c, float inv_t,
    const int64_t* __restrict__ targets, const float* __restrict__ lse, const float* __restrict__ spx,
    const float* __restrict__ g_lp, const float* __restrict__ g_ent, const float* __restrict__ grad_scale_dev,
    uint16_t* __restrict__ d_t, int64_t d_stride) {
  __shared__ __attribute__((aligned(1024))) unsigned char w0[kLmOperandBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char h0[kLmOperandBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char w1[kLmOperandBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char h1[kLmOperandBytes];
  int rb, split;
  if (!lm_block_coords(g, rb, split)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wv = wave >> 1, wt = wave & 1;
  const int64_t tok0 = int64_t(rb) * kLmTile;
  const float gs = grad_scale_dev ? *grad_scale_dev : 1.0f;
  float k0[4], a0[4], a1[4], hot[4];
  int64_t tg[4], tokj[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    tokj[j] = tok0 + wt * 128 + j * 32 + (lane & 31);
    const int64_t tk = tokj[j] < g.n_tokens ? tokj[j] : g.n_tokens - 1;
    const float glp = g_lp[tk] * gs, gh = g_ent ? g_ent[tk] * gs : 0.f;
    const float b = gh * inv_t;
    k0[j] = -lse[tk] * kLog2e;
    a0[j] = -glp * inv_t + (g_ent ? b * spx[tk] : 0.f);
    a1[j] = -b * inv_t;
    hot[j] = glp * inv_t;
    tg[j] = targets[tk];
  }
  const int vt_begin = split * g.tiles_per_split;
  const int vt_end = min(g.n_tiles, vt_begin + g.tiles_per_split);
  LmSlabWriter writer;
  writer.init(d_t, d_stride, g.vocab, g.n_tokens, tok0, wv, wt, lane);
  lm_pipeline<true>(LmLds{w0, h0, w1, h1}, hidden, weight, g, tok0, vt_begin, vt_end, [&](floatx16 (&acc)[4][4], int64_t v0) {
    writer.set_tile(v0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t vb = v0 + wv * 128 + i * 32 + 4 * (lane >> 5);
        const floatx16 blk = acc[i][j];
        float d[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float x = blk[r];
          d[r] = fast_exp2(fmaf(x, c, k0[j])) * fmaf(x, a1[j], a0[j]);
          if (vb + 8 * (r >> 2) + (r & 3) == tg[j]) d[r] += hot[j];
        }
        writer.template store<PAIRS>(d, i, j);
        __builtin_amdgcn_sched_barrier(0);
      }
  });
}

}  // namespace relax_amd

using namespace relax_amd;

static void lm_plan_splits(int64_t row_blocks, LmGeom& g);

static int lm_geometry(const char* what, int dtype, int64_t n, int64_t hidden, int64_t vocab, int64_t h_stride,
                       int64_t w_stride, const void* h, const void* w, LmGeom& g) {
  if (dtype != RELAX_AMD_BF16) {
    set_error("%s: hidden states and weight must be bf16", what);
    return RELAX_AMD_EUNSUPPORTED;
  }
  if (n <= 0 || hidden <= 0 || vocab <= 0 || h_stride < hidden || w_stride < hidden || n > (1LL << 30)) {
    set_error("%s: bad shape n_tokens=%lld hidden=%lld vocab=%lld", what, (long long)n, (long long)hidden,
              (long long)vocab);
    return RELAX_AMD_EINVAL;
  }
  if (hidden % (2 * kLmBK) != 0 || h_stride % 8 != 0 || w_stride % 8 != 0 || !aligned16(h) || !aligned16(w) ||
      int64_t(kLmTile) * h_stride >= (1LL << 31) || int64_t(kLmTile) * w_stride >= (1LL << 31)) {
    set_error("%s: hidden size must be a multiple of %d and rows 16-byte aligned (hidden=%lld)", what, 2 * kLmBK,
              (long long)hidden);
    return RELAX_AMD_EUNSUPPORTED;
  }
  g.n_tokens = n;
  g.hidden = hidden;
  g.vocab = vocab;
  g.h_stride = h_stride;
  g.w_stride = w_stride;
  const int64_t row_blocks = (n + kLmTile - 1) / kLmTile;
  g.n_tiles = int((vocab + kLmTile - 1) / kLmTile);
  lm_plan_splits(row_blocks, g);
  return RELAX_AMD_OK;
}

static void lm_plan_splits(int64_t row_blocks, LmGeom& g) {
  const int64_t most = std::min<int64_t>(lm_max_splits(row_blocks), g.n_tiles);
  int64_t best = 1, best_cost = INT64_MAX;
  for (int64_t s = 1; s <= most; ++s) {
    const int64_t cost = lm_split_cost(row_blocks, g.n_tiles, s);
    if (cost < best_cost) best = s, best_cost = cost;
  }
  g.tiles_per_split = int((g.n_tiles + best - 1) / best);
  g.tasks.rows = int(row_blocks);
  g.tasks.cols = (g.n_tiles + g.tiles_per_split - 1) / g.tiles_per_split;
  g.tasks.strip = lm_strip_height(row_blocks);
}

// Floats of per-split softmax partials in the workspace (three per token and split): room for whatever split count
// lm_plan_splits() takes for this many tokens or fewer.  (Sized for the count alone it was 787 k floats at 256 tokens and
// 769 k at 1000: a caller with one buffer for its largest chunk would have been written past by a shorter one.)
static int64_t lm_partial_floats(int64_t n_tokens) {
  return std::max(kLmMaxTasks, (n_tokens + kLmTile - 1) / kLmTile) * kLmTile * 3;
}

static unsigned lm_grid(const LmGeom& g) { return lm_task_blocks(int64_t(g.tasks.rows) * g.tasks.cols); }

extern "C" int64_t relax_amd_lmhead_workspace_bytes(int64_t n_tokens) {
  if (n_tokens <= 0) return 0;
  return (lm_partial_floats(n_tokens) + n_tokens) * int64_t(sizeof(float));
}

// 4-byte paired stores need an even row stride and a 4-byte aligned base
static bool lm_pairs_ok(const void* p, int64_t stride) {
  return stride % 2 == 0 && reinterpret_cast<uintptr_t>(p) % 4 == 0;
}
// the slab writer keeps byte offsets inside a 256-row tile in 32 bits
static int lm_slab_stride_ok(const char* what, int64_t stride) {
  if (int64_t(kLmTile + 1) * stride * 2 >= (1LL << 31)) {
    set_error("%s: slab row stride %lld too large", what, (long long)stride);
    return RELAX_AMD_EUNSUPPORTED;
  }
  return RELAX_AMD_OK;
}

static int lm_forward(const char* what, const void* hidden, const void* weight, int dtype, int64_t n_tokens,
                      int64_t hidden_size, int64_t vocab, int64_t h_stride, int64_t w_stride, const int64_t* targets,
                      float inv_temperature, void* workspace, float* log_prob, float* entropy, float* lse, float* spx,
                      uint16_t* l_t, int64_t l_stride, void* stream) {
  LmGeom g;
  if (int rc = lm_geometry(what, dtype, n_tokens, hidden_size, vocab, h_stride, w_stride, hidden, weight, g)) return rc;
  if (!targets || !workspace || !log_prob || !(inv_temperature > 0.f)) {
    set_error("%s: NULL argument or non-positive inv_temperature", what);
    return RELAX_AMD_EINVAL;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* partial = static_cast<float*>(workspace);
  float* x_target = partial + lm_partial_floats(n_tokens);
  const uint16_t* h = static_cast<const uint16_t*>(hidden);
  const uint16_t* w = static_cast<const uint16_t*>(weight);
  const float c = inv_temperature * kLog2e;
  const dim3 grid(lm_grid(g)), block(kLmThreads);
  if (!l_t) {
    hipLaunchKernelGGL(lmhead_target_logit_kernel, dim3(unsigned((n_tokens + 3) / 4)), dim3(256), 0, s, h, w, g,
                       targets, x_target);
    if (int rc = check_launch("lmhead_target_logit")) return rc;
    hipLaunchKernelGGL((lmhead_fwd_kernel<false, false>), grid, block, 0, s, h, w, g, c, partial, nullptr, int64_t(0),
                       nullptr);
  } else if (lm_pairs_ok(l_t, l_stride)) {
    hipLaunchKernelGGL((lmhead_fwd_kernel<true, true>), grid, block, 0, s, h, w, g, c, partial, l_t, l_stride, nullptr);
  } else {
    hipLaunchKernelGGL((lmhead_fwd_kernel<true, false>), grid, block, 0, s, h, w, g, c, partial, l_t, l_stride, nullptr);
  }
  if (int rc = check_launch("lmhead_fwd")) return rc;
  if (l_t) {
    hipLaunchKernelGGL(lmhead_target_from_logits_kernel, dim3(unsigned((n_tokens + 255) / 256)), dim3(256), 0, s, l_t,
                       l_stride, n_tokens, vocab, targets, x_target, nullptr);
    if (int rc = check_launch("lmhead_target_from_logits")) return rc;
  }
  hipLaunchKernelGGL(lmhead_combine_kernel, dim3(unsigned((n_tokens + 3) / 4)), dim3(256), 0, s, partial, x_target,
                     n_tokens, g.tasks.cols, inv_temperature, log_prob, entropy, lse, spx, nullptr, nullptr);
  return check_launch("lmhead_combine");
}

extern "C" int relax_amd_lmhead_logprob_fwd(const void* hidden, const void* weight, int dtype, int64_t n_tokens,
                                            int64_t hidden_size, int64_t vocab, int64_t h_stride, int64_t w_stride,
                                            const int64_t* targets, float inv_temperature, void* workspace,
                                            float* log_prob, float* entropy, float* lse, float* spx, void* stream) {
  if (n_tokens == 0) return RELAX_AMD_OK;
  return lm_forward("lmhead_logprob_fwd", hidden, weight, dtype, n_tokens, hidden_size, vocab, h_stride, w_stride,
                    targets, inv_temperature, workspace, log_prob, entropy, lse, spx, nullptr, 0, stream);
}

// Scratch of the allocation-free entry point: the per-split softmax partials and the target logits of up to
// RELAX_AMD_LMHEAD_STATIC_MAX_TOKENS tokens.  One copy per GPU, held until the process ends.  The name is a host-side
// stand-in, not a device address: host code only ever uses the pointer hipGetSymbolAddress returns for the current
// device.
static __device__ __align__(256) float lm_static_scratch[RELAX_AMD_LMHEAD_STATIC_SCRATCH_BYTES / sizeof(float)];

namespace {
constexpr int kLmMaxDevices = 64;
std::mutex lm_static_mutex;
void* lm_static_ptr[kLmMaxDevices] = {};
}  // namespace

// The current device's copy of lm_static_scratch (looked up once per device, with that device current).
static int lm_static_workspace(const char* what, void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kLmMaxDevices) {
    set_error("%s: no usable current device (%s)", what, e == hipSuccess ? "index out of range" : hipGetErrorString(e));
    return RELAX_AMD_EINVAL;
  }
  std::lock_guard<std::mutex> lock(lm_static_mutex);
  if (!lm_static_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(lm_static_scratch));
    if (e != hipSuccess || !p) {
      set_error("%s: hipGetSymbolAddress failed on device %d: %s", what, dev, hipGetErrorString(e));
      return RELAX_AMD_ELAUNCH;
    }
    lm_static_ptr[dev] = p;
  }
  *out = lm_static_ptr[dev];
  return RELAX_AMD_OK;
}

extern "C" int relax_amd_lmhead_logprob_fwd_static(const void* hidden, const void* weight, int dtype,
                                                   int64_t n_tokens, int64_t hidden_size, int64_t vocab,
                                                   int64_t h_stride, int64_t w_stride, const int64_t* targets,
                                                   float inv_temperature, float* log_prob, float* entropy, float* lse,
                                                   float* spx, void* stream) {
  if (n_tokens == 0) return RELAX_AMD_OK;
  if (n_tokens < 0 || n_tokens > RELAX_AMD_LMHEAD_STATIC_MAX_TOKENS ||
      relax_amd_lmhead_workspace_bytes(n_tokens) > int64_t(RELAX_AMD_LMHEAD_STATIC_SCRATCH_BYTES)) {
    set_error("lmhead_logprob_fwd_static: n_tokens=%lld is outside 0..%d, the size the built-in scratch holds; use "
              "relax_amd_lmhead_logprob_fwd with a caller workspace", (long long)n_tokens,
              RELAX_AMD_LMHEAD_STATIC_MAX_TOKENS);
    return RELAX_AMD_EUNSUPPORTED;
  }
  void* workspace = nullptr;
  if (int rc = lm_static_workspace("lmhead_logprob_fwd_static", &workspace)) return rc;
  // every partial and target logit the combine kernel reads is written by this call's own launches first, so the
  // contents a previous call left behind need no clearing
  return lm_forward("lmhead_logprob_fwd_static", hidden, weight, dtype, n_tokens, hidden_size, vocab, h_stride,
                    w_stride, targets, inv_temperature, workspace, log_prob, entropy, lse, spx, nullptr, 0, stream);
}

extern "C" int relax_amd_lmhead_logprob_fwd_keep(const void* hidden, const void* weight, int dtype, int64_t n_tokens,
                                                 int64_t hidden_size, int64_t vocab, int64_t h_stride,
                                                 int64_t w_stride, const int64_t* targets, float inv_temperature,
                                                 void* workspace, float* log_prob, float* entropy, float* lse,
                                                 float* spx, void* logits_t, int64_t l_stride, void* stream) {
  if (n_tokens == 0) return RELAX_AMD_OK;
  if (!logits_t || l_stride < n_tokens) {
    set_error("lmhead_logprob_fwd_keep: NULL logits_t or l_stride < n_tokens");
    return RELAX_AMD_EINVAL;
  }
  if (int rc = lm_slab_stride_ok("lmhead_logprob_fwd_keep", l_stride)) return rc;
  return lm_forward("lmhead_logprob_fwd_keep", hidden, weight, dtype, n_tokens, hidden_size, vocab, h_stride,
                    w_stride, targets, inv_temperature, workspace, log_prob, entropy, lse, spx,
                    static_cast<uint16_t*>(logits_t), l_stride, stream);
}

extern "C" int relax_amd_lmhead_dlogits_from_logits_t(void* logits_t, int64_t n_tokens, int64_t vocab,
                                                      int64_t l_stride, const int64_t* targets, const float* lse,
                                                      const float* spx, const float* g_lp, const float* g_ent,
                                                      const float* grad_scale_dev, float inv_temperature,
                                                      void* stream) {
  if (n_tokens == 0 || vocab == 0) return RELAX_AMD_OK;
  if (n_tokens < 0 || vocab < 0 || !logits_t || !targets || !lse || !g_lp || (g_ent && !spx) ||
      !(inv_temperature > 0.f)) {
    set_error("lmhead_dlogits_from_logits_t: NULL argument, negative size or non-positive inv_temperature");
    return RELAX_AMD_EINVAL;
  }
  if (l_stride % 8 != 0 || l_stride < n_tokens || !aligned16(logits_t)) {
    set_error("lmhead_dlogits_from_logits_t: l_stride must be a multiple of 8 and >= n_tokens, base 16-byte aligned");
    return RELAX_AMD_EUNSUPPORTED;
  }
  constexpr int kRows = 64;
  const int64_t col_blocks = (n_tokens + 8LL * kLmInplaceThreads - 1) / (8LL * kLmInplaceThreads);
  const int64_t row_blocks = (vocab + kRows - 1) / kRows;
  if (row_blocks > 65535 || col_blocks > 2147483647LL) {
    set_error("lmhead_dlogits_from_logits_t: vocab=%lld too large", (long long)vocab);
    return RELAX_AMD_EUNSUPPORTED;
  }
  hipLaunchKernelGGL(lmhead_dlogits_inplace_kernel, dim3(unsigned(col_blocks), unsigned(row_blocks)),
                     dim3(kLmInplaceThreads), 0, static_cast<hipStream_t>(stream), static_cast<uint16_t*>(logits_t),
                     l_stride, n_tokens, vocab, kRows, inv_temperature * kLog2e, inv_temperature, targets, lse, spx,
                     g_lp, g_ent, grad_scale_dev, nullptr);
  return check_launch("lmhead_dlogits_inplace");
}

extern "C" int relax_amd_lmhead_dlogits_t(const void* hidden, const void* weight, int dtype, int64_t n_tokens,
                                          int64_t hidden_size, int64_t vocab, int64_t h_stride, int64_t w_stride,
                                          const int64_t* targets, const float* lse, const float* spx,
                                          const float* g_lp, const float* g_ent, const float* grad_scale_dev,
                                          float inv_temperature, void* d_t, int64_t d_stride, void* stream) {
  if (n_tokens == 0) return RELAX_AMD_OK;
  LmGeom g;
  if (int rc = lm_geometry("lmhead_dlogits_t", dtype, n_tokens, hidden_size, vocab, h_stride, w_stride, hidden,
                           weight, g))
    return rc;
  if (!targets || !lse || !g_lp || !d_t || (g_ent && !spx) || d_stride < n_tokens || !(inv_temperature > 0.f)) {
    set_error("lmhead_dlogits_t: NULL argument, short d_stride or non-positive inv_temperature");
    return RELAX_AMD_EINVAL;
  }
  if (int rc = lm_slab_stride_ok("lmhead_dlogits_t", d_stride)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (lm_pairs_ok(d_t, d_stride))
    hipLaunchKernelGGL(lmhead_dlogits_kernel<true>, dim3(lm_grid(g)), dim3(kLmThreads), 0, s,
                       static_cast<const uint16_t*>(hidden), static_cast<const uint16_t*>(weight), g,
                       inv_temperature * kLog2e, inv_temperature, targets, lse, spx, g_lp, g_ent, grad_scale_dev,
                       static_cast<uint16_t*>(d_t), d_stride);
  else
    hipLaunchKernelGGL(lmhead_dlogits_kernel<false>, dim3(lm_grid(g)), dim3(kLmThreads), 0, s,
                       static_cast<const uint16_t*>(hidden), static_cast<const uint16_t*>(weight), g,
                       inv_temperature * kLog2e, inv_temperature, targets, lse, spx, g_lp, g_ent, grad_scale_dev,
                       static_cast<uint16_t*>(d_t), d_stride);
  return check_launch("lmhead_dlogits");
}

extern "C" int64_t relax_amd_lmhead_live_plan_bytes(int64_t n_tokens, int64_t slab_tokens) {
  if (n_tokens <= 0 || slab_tokens <= 0) return 0;
  return (n_tokens + slab_tokens - 1) / slab_tokens * int64_t(sizeof(LmLivePlan));
}

extern "C" int relax_amd_lmhead_live_rows(const void* rows, int64_t row_stride, int64_t hidden_size, int64_t vocab,
                                          const int32_t* row_ids, const int64_t* targets, const float* token_weight,
                                          float weight_scale, int64_t n_tokens, int64_t slab_tokens, void* plans,
                                          int32_t* token_map, void* picked, int64_t* picked_targets, float* g_lp,
                                          int32_t* row_map, void* stream) {
  if (n_tokens == 0) return RELAX_AMD_OK;
  if (!rows || !row_ids || !targets || !token_weight || !plans || !token_map || !picked || !picked_targets || !g_lp ||
      !row_map || n_tokens < 0 || n_tokens > (1LL << 30) || slab_tokens <= 0 || slab_tokens % 128 != 0 ||
      hidden_size <= 0 || vocab <= 0 || row_stride < hidden_size) {
    set_error("lmhead_live_rows: NULL argument or bad shape n_tokens=%lld slab=%lld", (long long)n_tokens,
              (long long)slab_tokens);
    return RELAX_AMD_EINVAL;
  }
  if (hidden_size % (2 * kLmBK) != 0 || !aligned16(picked) || n_tokens / slab_tokens >= 65536) {
    set_error("lmhead_live_rows: hidden size must be a multiple of %d, picked 16-byte aligned", 2 * kLmBK);
    return RELAX_AMD_EUNSUPPORTED;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t slabs = (n_tokens + slab_tokens - 1) / slab_tokens;
  hipLaunchKernelGGL(lmhead_live_plan_kernel, dim3(1), dim3(kLmPlanThreads), 0, s, token_weight, n_tokens, slab_tokens,
                     int(slabs), int((vocab + kLmTile - 1) / kLmTile), int((hidden_size + kLmTile - 1) / kLmTile),
                     int((vocab + 127) / 128), token_map, static_cast<LmLivePlan*>(plans));
  if (int rc = check_launch("lmhead_live_plan")) return rc;
  hipLaunchKernelGGL(lmhead_live_gather_kernel, dim3(unsigned(n_tokens)), dim3(256), 0, s,
                     static_cast<const uint16_t*>(rows), row_stride, hidden_size, row_ids, targets, token_weight,
                     weight_scale, slab_tokens, token_map, static_cast<const LmLivePlan*>(plans),
                     static_cast<uint16_t*>(picked), picked_targets, g_lp, row_map);
  return check_launch("lmhead_live_gather");
}

static int64_t lm_round4(int64_t x) { return (x + 3) / 4 * 4; }

static int64_t lm_live_workspace_bytes(int64_t max_tokens, int64_t hidden_size, int64_t vocab) {
  if (max_tokens <= 0 || hidden_size <= 0) return 0;
  return (lm_partial_floats(max_tokens) + 2 * lm_round4(max_tokens) +
          lm_live_dhidden_floats(max_tokens, hidden_size, vocab)) * int64_t(sizeof(float));
}

extern "C" int64_t relax_amd_lmhead_live_workspace_bytes(int64_t max_tokens, int64_t hidden_size) {
  return lm_live_workspace_bytes(max_tokens, hidden_size, 0);
}

extern "C" int64_t relax_amd_lmhead_live_step_workspace_bytes(int64_t max_tokens, int64_t hidden_size, int64_t vocab) {
  return vocab <= 0 ? 0 : lm_live_workspace_bytes(max_tokens, hidden_size, vocab);
}

extern "C" int relax_amd_lmhead_live_step(const void* plan, const void* picked, const void* weight, int64_t w_stride,
                                          int64_t max_tokens, int64_t hidden_size, int64_t vocab,
                                          const int64_t* picked_targets, const float* g_lp, const int32_t* token_map,
                                          const int32_t* row_map, float inv_temperature, void* slab,
                                          int64_t slab_rows, int64_t slab_stride, void* workspace,
                                          int64_t workspace_bytes, float* log_prob, void* d_rows, int64_t dr_stride,
                                          void* d_weight, int64_t dw_stride, int dw_out_mode, void* stream) {
  if (max_tokens == 0) return RELAX_AMD_OK;
  const char* what = "lmhead_live_step";
  LmGeom g;
  if (int rc = lm_geometry(what, RELAX_AMD_BF16, max_tokens, hidden_size, vocab, hidden_size, w_stride, picked, weight,
                           g))
    return rc;
  if (!plan || !picked_targets || !g_lp || !token_map || !row_map || !slab || !workspace || !log_prob ||
      !(inv_temperature > 0.f) || !aligned16(workspace) ||
      workspace_bytes < lm_live_workspace_bytes(max_tokens, hidden_size, vocab)) {
    set_error("%s: NULL argument, non-positive inv_temperature or short workspace", what);
    return RELAX_AMD_EINVAL;
  }
  if (slab_rows < (vocab + 127) / 128 * 128) {
    set_error("%s: the slab must hold ceil128(vocab) rows, got %lld", what, (long long)slab_rows);
    return RELAX_AMD_EUNSUPPORTED;
  }
  if (int rc = lm_slab_stride_ok(what, slab_stride)) return rc;
  if (d_rows)
    if (int rc = gemm_check(what, slab, slab_stride, weight, w_stride, max_tokens, hidden_size, vocab, d_rows,
                            dr_stride, RELAX_AMD_GEMM_OUT_BF16))
      return rc;
  if (d_weight)
    if (int rc = gemm_check(what, slab, slab_stride, picked, hidden_size, max_tokens, hidden_size, vocab, d_weight,
                            dw_stride, dw_out_mode))
      return rc;
  if (slab_stride < (max_tokens + 127) / 128 * 128 || slab_stride % 8 != 0 || !aligned16(slab)) {
    set_error("%s: the slab needs 16-byte aligned rows of at least ceil128(max_tokens) elements", what);
    return RELAX_AMD_EUNSUPPORTED;
  }
  constexpr int kRows = 64;
  const int64_t col_blocks = (max_tokens + 8LL * kLmInplaceThreads - 1) / (8LL * kLmInplaceThreads);
  const int64_t row_groups = (vocab + kRows - 1) / kRows;
  if (row_groups > 65535) {
    set_error("%s: vocab=%lld too large", what, (long long)vocab);
    return RELAX_AMD_EUNSUPPORTED;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const LmLivePlan* live = static_cast<const LmLivePlan*>(plan);
  float* partial = static_cast<float*>(workspace);
  float* x_target = partial + lm_partial_floats(max_tokens);
  float* lse = x_target + lm_round4(max_tokens);
  float* dh_part = lse + lm_round4(max_tokens);
  uint16_t* l_t = static_cast<uint16_t*>(slab);
  const float c = inv_temperature * kLog2e;
  // the device's row blocks times splits is at most this
  const dim3 grid(lm_task_blocks(std::max<int64_t>(kLmMaxTasks, g.tasks.rows))), block(kLmThreads);
  const dim3 per_token(unsigned((max_tokens + 255) / 256));
  hipLaunchKernelGGL((lmhead_fwd_kernel<true, true>), grid, block, 0, s, static_cast<const uint16_t*>(picked),
                     static_cast<const uint16_t*>(weight), g, c, partial, l_t, slab_stride, live);
  if (int rc = check_launch("lmhead_fwd")) return rc;
  hipLaunchKernelGGL(lmhead_target_from_logits_kernel, per_token, dim3(256), 0, s, l_t, slab_stride, max_tokens, vocab,
                     picked_targets, x_target, live);
  hipLaunchKernelGGL(lmhead_combine_kernel, dim3(unsigned((max_tokens + 3) / 4)), dim3(256), 0, s, partial, x_target, max_tokens, 1,
                     inv_temperature, log_prob, nullptr, lse, nullptr, live, token_map);
  hipLaunchKernelGGL(lmhead_dlogits_inplace_kernel, dim3(unsigned(col_blocks), unsigned(row_groups)),
                     dim3(kLmInplaceThreads), 0, s, l_t, slab_stride, max_tokens, vocab, kRows, c, inv_temperature,
                     picked_targets, lse, nullptr, g_lp, nullptr, nullptr, live);
  if (int rc = check_launch("lmhead_dlogits_inplace")) return rc;
  if (d_rows)
    if (int rc = lm_live_dhidden(slab, slab_stride, weight, w_stride, max_tokens, hidden_size, vocab, live, dh_part,
                                 row_map, d_rows, dr_stride, s))
      return rc;
  if (d_weight)
    return lm_live_dweight(slab, slab_stride, picked, hidden_size, max_tokens, hidden_size, vocab, live, d_weight,
                           dw_stride, dw_out_mode, s);
  return RELAX_AMD_OK;
}
