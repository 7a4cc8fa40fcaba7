// tokpath_logprob.hip -- selective log-softmax gather + softmax entropy (gfx950).
//
// One workgroup of 256 threads streams one row, or one of the slices a row is
// cut into when there are few rows, once (tokpath_stream.h: double-buffered
// 16-byte loads, 8 vectors per thread per step, non-temporal because nothing
// re-reads the row).  Each thread keeps an online (m, s, t) state in base-2
// units:
//   d_i = (x_i - m) * log2(e),  s = sum 2^{d_i},  t = sum 2^{d_i} * d_i
// so logprob = x_target - m - ln s and entropy = ln s - ln2 * t / s.
// The row is never written back (no [N, V] log-softmax), so the kernel is
// bounded by one HBM read of the logits and by the VALU work per element.
//
// Replaces sequence_log_probs_from_logits (src/graspo/core/graspo_loss.py:19-21)
// and the logsumexp / logaddexp chunk loop of _selected_token_log_probs_from_hidden
// (src/graspo/backends/graspoflow/tensor_utils.py:180-186).
#include <chrono>
#include <thread>

#include "tokpath_stream.h"

namespace gtp {

int64_t device_cus();  // compute units of the current device

constexpr int kLpBlock = 256;
constexpr int kLpVecs = 8;  // 16-byte vectors per thread per step

// Scalar fold of one logit (a row's ends).
__device__ __forceinline__ void lse_fold_one(Lse3& st, float x) {
  if (x > st.m) {
    if (st.s > 0.0f) {
      const float dl = (st.m - x) * kLog2e;
      const float f = __builtin_amdgcn_exp2f(dl);
      st.t = f * __builtin_fmaf(dl, st.s, st.t);
      st.s *= f;
    }
    st.m = x;
  }
  if (x != x) st.s = __builtin_nanf("");
  const float d = (x - (st.m == kNegInf ? 0.0f : st.m)) * kLog2e;
  const float e = __builtin_amdgcn_exp2f(d);
  st.s += e;
  st.t = __builtin_fmaf(e, fmaxf(d, -256.0f), st.t);
}

// Elements of a row [0, V) before its first 16-byte boundary, taken one by
// one so that the rest streams as aligned vectors.  An odd vocabulary starts
// its contiguous rows at every alignment: three of four fp32 rows and seven
// of eight bf16 rows.  Reading and writing such rows by elements took 121 us
// forward and 125 us backward at fp32 [999, 50257]; a whole policy step of
// that size went from 401 to 262 us with the vectors.  (A row not aligned to its own elements has no vectors.)
template <typename T>
__device__ __forceinline__ int64_t row_head(const T* row, int64_t V) {
  const uint32_t up = (0u - (uint32_t)reinterpret_cast<uintptr_t>(row)) & 15u;
  return up % sizeof(T) ? V : min((int64_t)(up / sizeof(T)), V);
}

// Calls f(i) for this thread's share of the elements outside
// [head, head + body).
template <typename F>
__device__ __forceinline__ void for_edges(int64_t V, int64_t head, int64_t body, F&& f) {
  for (int64_t j = threadIdx.x; j < V - body; j += kLpBlock) f(j < head ? j : j + body);
}

// Elements [e0, e1) of a row that one workgroup takes: slice k of `slices`,
// cut at whole vectors of the row's aligned body, the first slice with the
// row's head and the last one with its end.
struct Slice {
  int64_t v0, v1;  // vectors of the aligned body
  bool first, last;
};
template <int E>
__device__ __forceinline__ Slice slice_of(int64_t nvec, int k, int slices) {
  // whole groups of 64 vectors, so that a wave's 1 KB loads never straddle two slices
  const int64_t per = ((nvec + slices - 1) / slices + 63) / 64 * 64;
  const int64_t v0 = min((int64_t)k * per, nvec);
  return {v0, min(v0 + per, nvec), k == 0, k == slices - 1};
}

// Whole vectors of the fold: the entropy's moment is summed as e * d, which
// is NaN where d = -inf (a logit of -inf, or the padding of the last step).
// A wave clamps d only from the first block on whose moment came out NaN
// (`clamp`, which it keeps; that block is summed again) and in a `padded`
// one.  Clamping every element took one VALU instruction in nine of the fold:
// bf16 [8192, 151936] 401 us, without it 392.  Summing every block twice that
// holds -inf took more than that: [4096, 151936] with 92% of the logits at
// -inf 248 us, this way 198 (dense rows 204; [1000, 50257] 48 -> 42).
template <bool kEntropy, int NG, int E>
__device__ __forceinline__ void lp_fold_block(Lse3& st, const float (&x)[NG][E], bool& clamp,
                                              bool padded) {
  if constexpr (!kEntropy) {
    lse_fold_block<false, NG, E>(st, x);
  } else {
    if (!(clamp || padded)) {
      Lse3 nt = st;
      lse_fold_block_max<true, NG, E, false>(nt, x, block_max_raw<NG, E>(x));
      clamp = __ballot(nt.t != nt.t) != 0ull;
      if (!clamp) {
        st = nt;
        return;
      }
    }
    lse_fold_block<true, NG, E>(st, x);
  }
}

// A row's sum is cut in chunks of whole steps of the stream, `per` steps each
// and at most kMaxChunks of them, by its vocabulary alone: a chunk's state is
// the merge of its four waves' and a row's is the merge of its chunks',
// whichever workgroups take them.  So a row has the same bits scored alone, in
// a small batch (where its chunks go to several workgroups) and in a large
// one.
constexpr int kMaxChunks = 32;
constexpr int kLpStep = kLpBlock * kLpVecs;  // vectors
struct Chunks {
  int n, per;
};
template <typename T>
Chunks chunks_of(int64_t V) {
  const int64_t steps = max((int64_t)1, (V / Vec<T>::kE + kLpStep - 1) / kLpStep);
  const int64_t per = (steps + kMaxChunks - 1) / kMaxChunks;
  return {(int)((steps + per - 1) / per), (int)per};
}

// The four waves' states of a chunk, as wave_lse3_max merges lanes.
__device__ __forceinline__ Lse3 merge_waves(const float (*red)[kMaxChunks][3], int c) {
  constexpr int kW = kLpBlock / kWave;
  float m = red[0][c][0];
#pragma unroll
  for (int w = 1; w < kW; ++w) m = fmaxf(m, red[w][c][0]);
  float s = 0.0f, t = 0.0f;
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    const float wm = red[w][c][0], ws = red[w][c][1];
    const float dl = wm == m ? 0.0f : fmaxf((wm - m) * kLog2e, -256.0f);
    const float f = __builtin_amdgcn_exp2f(dl);
    s += ws * f;
    t += f * __builtin_fmaf(dl, ws, red[w][c][2]);
  }
  return {m, s, t};
}

// Chunks [c0, c1) of a row [0, V): lane l of wave 0 gets chunk c0 + l's state
// (the lanes past them an empty one).  Every thread calls; `red` is the
// workgroup's.  A wave reduces its chunk as soon as it has folded it, on DPP:
// a call of bf16 [8192, 151936], ten chunks a row, 381 us with one reduction
// per row, 384 with ten (375 with the shorter prefetch past the stream's end).
// A workgroup alone on a CU waits some 0.14 us for each (logprob_entropy of
// fp32 [1, 248320], 31 chunks, 21.4 -> 25.8 us); rows in slices do not.
template <typename T, bool kEntropy>
__device__ __forceinline__ Lse3 chunk_states(const T* __restrict__ row, int64_t V, Chunks ch,
                                             int c0, int c1, float (*red)[kMaxChunks][3]) {
  constexpr int E = Vec<T>::kE;
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const int64_t head = row_head(row, V);
  const int64_t nvec = (V - head) / E;
  const int64_t v0 = min((int64_t)c0 * ch.per * kLpStep, nvec);
  const int64_t v1 = min((int64_t)c1 * ch.per * kLpStep, nvec);
  const bool partial = (v1 - v0) % kLpStep != 0;
  const Lse3 empty{kNegInf, 0.0f, 0.0f};
  Lse3 st = empty, held = empty;
  int c = 0, left = ch.per;
  bool clamp = false;
  auto close = [&]() __attribute__((always_inline)) {
    if constexpr (kEntropy)
      st = wave_lse3_max(st);
    else
      wave_lse2(st.m, st.s);
    if (lane == c) held = st;
    st = empty;
    left = ch.per;
    ++c;
  };
  stream_vectors<T, kLpBlock, kLpVecs, true>(
      row + head, v0, v1, [&](float(&x)[kLpVecs][E], int64_t vbase, bool last) {
        if (left == 0) close();
        --left;
        if (last) mask_tail<kLpVecs, E, kLpBlock>(x, vbase, v1);
        lp_fold_block<kEntropy, kLpVecs, E>(st, x, clamp, last && partial);
      });
  // the row's ends go to its last chunk
  if (c1 == ch.n) {
    if (c < ch.n - 1 - c0) close();
    for_edges(V, head, nvec * E, [&](int64_t i) { lse_fold_one(st, Elem<T>::get(row, i)); });
  }
  close();
  if (lane < c1 - c0) {
    red[wid][lane][0] = held.m;
    red[wid][lane][1] = held.s;
    red[wid][lane][2] = held.t;
  }
  __syncthreads();
  return lane < c1 - c0 ? merge_waves(red, lane) : empty;
}

__device__ __forceinline__ int64_t load_target(const void* targets, int t64, int64_t n) {
  return t64 ? reinterpret_cast<const int64_t*>(targets)[n]
             : (int64_t)reinterpret_cast<const int32_t*>(targets)[n];
}

// B x S rows of logits and their targets, each [B, S] with strides of its
// own (a shifted view of [B, S + 1, V] logits is read in place).
struct TokenRows {
  const void* logits;
  const void* targets;
  int64_t V, S, bstride, rstride, tbstride, trstride, ignore;
  int B, t64, has_ignore;
  __device__ __forceinline__ int64_t rows() const { return (int64_t)B * S; }
  // (sequence, position) of row n; one sequence needs no division
  __device__ __forceinline__ void at(int64_t n, int64_t& b, int64_t& s) const {
    b = B > 1 ? (uint32_t)n / (uint32_t)S : 0;
    s = n - b * S;
  }
  template <typename T>
  __device__ __forceinline__ const T* row(int64_t b, int64_t s) const {
    return reinterpret_cast<const T*>(logits) + b * bstride + s * rstride;
  }
  __device__ __forceinline__ int64_t target(int64_t b, int64_t s) const {
    return load_target(targets, t64, b * tbstride + s * trstride);
  }
};

// Workgroup of a grid that goes on in y: a launch holds fewer than 2^32 work
// items in one dimension, 2^24 workgroups of 256.
constexpr int64_t kGridX = 1 << 23;
__device__ __forceinline__ int64_t flat_workgroup() {
  return blockIdx.x + (int64_t)blockIdx.y * gridDim.x;
}
inline dim3 flat_grid(int64_t n) {
  return n <= kGridX ? dim3((unsigned)n) : dim3((unsigned)kGridX, (unsigned)((n + kGridX - 1) / kGridX));
}

// What a row's state gives: logprob, entropy and status.
struct TokenOut {
  float* lp;
  float* H;
  int32_t* status;
  __device__ __forceinline__ void put(int64_t n, const Lse3& st, float xt, bool ok) const {
    const float ln_s = __builtin_amdgcn_logf(st.s) * kLn2;
    lp[n] = ok ? raw_logprob(xt, st.m, ln_s) : __builtin_nanf("");
    if (H) H[n] = ln_s - kLn2 * st.t / st.s;
    if (status) status[n] = ok ? GTP_ROW_OK : GTP_ROW_BAD_TARGET;
  }
};

// Target of a row; an ignored one reads as token 0, which is never bad.
__device__ __forceinline__ int64_t row_target(const TokenRows& a, int64_t b, int64_t s) {
  const int64_t t = a.target(b, s);
  return a.has_ignore && t == a.ignore ? 0 : t;
}

// Ahead of the rows: clears their arrival counters (n_ctr of them) and tells
// the host, through one word of its own per workgroup (pinned host memory),
// whether some target lies outside [0, V).  The host raises on a bad target
// as soon as this kernel has run (2 us for 61 targets, 5 for 8192), while
// the rows are still streaming; a reduction of per-row statuses after the
// rows and its copy to the host held it for the whole kernel and 20 us more
// (a scoring call of 61 rows 41.6 -> 18.2 us, of 8192 402 -> 382).
constexpr int kVerdictBlock = 1024;
__global__ __launch_bounds__(kVerdictBlock) void token_targets_kernel(
    TokenRows a, int64_t N, uint32_t* __restrict__ ctr, int n_ctr, const uint32_t* flag_a,
    const uint32_t* flag_b, uint32_t* __restrict__ verdict) {
  const int64_t first = (int64_t)blockIdx.x * kVerdictBlock + threadIdx.x;
  const int64_t step = (int64_t)gridDim.x * kVerdictBlock;
  for (int64_t n = first; n < n_ctr; n += step) ctr[n] = 0;
  if (!verdict) return;
  bool bad = false;
  for (int64_t n = first; n < N; n += step) {
    int64_t b, s;
    a.at(n, b, s);
    const int64_t t = row_target(a, b, s);
    bad |= t < 0 || t >= a.V;
  }
  const int any = __syncthreads_or(bad ? 1 : 0);
  if (threadIdx.x != 0) return;
  uint32_t w = GTP_VERDICT_GOOD | (any ? GTP_VERDICT_BAD : 0u);
  if ((flag_a && *flag_a) || (flag_b && *flag_b)) w |= GTP_VERDICT_FLAGGED;
  __hip_atomic_store(verdict + blockIdx.x, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// slices == 1: one workgroup per row.  Otherwise workgroup (row, slice) takes
// its share of the row's chunks and publishes their (m, s, t), and the last of
// the row's workgroups to arrive merges them.  A second launch for the merge
// took 4 us after the 12 of 61 rows.
template <typename T, bool kEntropy>
__global__ __launch_bounds__(kLpBlock) void token_logprob_kernel(TokenRows a, TokenOut out,
                                                                 Chunks ch, int slices,
                                                                 uint32_t* __restrict__ ctr,
                                                                 float* __restrict__ partial) {
  __shared__ float red[kLpBlock / kWave][kMaxChunks][3];
  // (rows in slices are few: one dimension)
  const int64_t n = slices > 1 ? blockIdx.x / (uint32_t)slices : flat_workgroup();
  if (n >= a.rows()) return;
  const int k = slices > 1 ? (int)(blockIdx.x - n * slices) : 0;
  int64_t b, s;
  a.at(n, b, s);
  const T* row = a.row<T>(b, s);
  const int64_t tgt = row_target(a, b, s);
  const bool ok = tgt >= 0 && tgt < a.V;
  float xt = 0.0f;
  if (threadIdx.x == 0 && ok) xt = Elem<T>::get(row, tgt);
  const int c0 = k * ch.n / slices, c1 = (k + 1) * ch.n / slices;
  Lse3 st = chunk_states<T, kEntropy>(row, a.V, ch, c0, c1, red);
  if (threadIdx.x >= kWave) return;
  const int lane = threadIdx.x;
  if (slices > 1) {
    // No release operation: gfx950's agent-scope stores write through to
    // where the other XCDs' agent-scope loads see them, and vmcnt(0) waits
    // for their completion before the arrival (a release fence would write
    // the whole L2 back).
    float* p = partial + n * ch.n * 3;  // [3][chunks]
    if (lane < c1 - c0) {
      __hip_atomic_store(p + c0 + lane, st.m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(p + ch.n + c0 + lane, st.s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(p + 2 * ch.n + c0 + lane, st.t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t arrived = 0;
    if (lane == 0)
      arrived = __hip_atomic_fetch_add(ctr + n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane((int)arrived) != slices - 1) return;
    asm volatile("" ::: "memory");
    p += min(lane, ch.n - 1);
    const float m = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const float sm = __hip_atomic_load(p + ch.n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const float t = __hip_atomic_load(p + 2 * ch.n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    st = lane < ch.n ? Lse3{m, sm, t} : Lse3{kNegInf, 0.0f, 0.0f};
  }
  if (ch.n > 1) st = wave_lse3_max(st);
  if (threadIdx.x == 0) out.put(n, st, xt, ok);
}

// Chunk state layout: [N][4] = (m, s, t_nat, x_target), t_nat = ln2 * t.
template <typename T>
__global__ __launch_bounds__(kLpBlock) void lse_partial_kernel(
    const T* __restrict__ logits, int64_t Vc, int64_t row_stride, int64_t col_offset,
    const void* __restrict__ targets, int t64, float* __restrict__ state, int accumulate,
    Chunks ch) {
  __shared__ float red[kLpBlock / kWave][kMaxChunks][3];
  const int64_t n = blockIdx.x;
  const T* row = logits + n * row_stride;
  const int64_t tgt = targets ? load_target(targets, t64, n) - col_offset : -1;
  Lse3 st = chunk_states<T, true>(row, Vc, ch, 0, ch.n, red);
  if (threadIdx.x >= kWave) return;
  if (ch.n > 1) st = wave_lse3_max(st);
  if (threadIdx.x == 0) {
    float* sp = state + n * 4;
    float xt = __builtin_nanf("");
    if (accumulate) {
      const Lse3 old{sp[0], sp[1], sp[2] * kLog2e};
      st = lse3_merge(old, st);
      xt = sp[3];
    }
    if (tgt >= 0 && tgt < Vc) xt = Elem<T>::get(row, tgt);
    sp[0] = st.m;
    sp[1] = st.s;
    sp[2] = st.t * kLn2;
    sp[3] = xt;
  }
}

__global__ void lse_finalize_kernel(const float* __restrict__ state, int64_t N,
                                    float* __restrict__ out_lp, float* __restrict__ out_H) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  const float m = state[n * 4 + 0], s = state[n * 4 + 1], t = state[n * 4 + 2], xt = state[n * 4 + 3];
  const float ln_s = __builtin_amdgcn_logf(s) * kLn2;
  if (out_lp) out_lp[n] = raw_logprob(xt, m, ln_s);
  if (out_H) out_H[n] = ln_s - t / s;
}

// ---------------------------------------------------------------- backward
//
// d logprob / d x_i = [i == target] - p_i with p_i = exp(x_i - lse), so the
// gradient of a loss with dL/dlogprob = g per row is g * ([i == t] - p_i):
// one read of the row and one write of the gradient in the logits' dtype.
// A row with g == 0 (an ignored SFT position) is written as zeros without
// reading it.

// fp32 -> bf16 bit pattern, round to nearest even (NaN stays NaN)
__device__ __forceinline__ uint32_t bf16_rne(float f) {
  const uint32_t u = f2u(f);
  const uint32_t r = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
  return (u & 0x7FFFFFFFu) > 0x7F800000u ? 0x7FC0u : r;
}

template <typename T>
struct GradOut;
template <>
struct GradOut<uint16_t> {
  // 8 gradients -> one 16-byte vector of bf16
  __device__ static __forceinline__ u32x4 pack(const float (&g)[8]) {
    u32x4 v;
    v.x = bf16_rne(g[0]) | (bf16_rne(g[1]) << 16);
    v.y = bf16_rne(g[2]) | (bf16_rne(g[3]) << 16);
    v.z = bf16_rne(g[4]) | (bf16_rne(g[5]) << 16);
    v.w = bf16_rne(g[6]) | (bf16_rne(g[7]) << 16);
    return v;
  }
  __device__ static __forceinline__ void put(uint16_t* p, int64_t i, float g) {
    p[i] = (uint16_t)bf16_rne(g);
  }
};
template <>
struct GradOut<_Float16> {
  __device__ static __forceinline__ u32x4 pack(const float (&g)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const _Float16 lo = (_Float16)g[2 * k], hi = (_Float16)g[2 * k + 1];
      w[k] = (uint32_t)__builtin_bit_cast(uint16_t, lo) |
             ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
    }
    u32x4 v;
    v.x = w[0];
    v.y = w[1];
    v.z = w[2];
    v.w = w[3];
    return v;
  }
  __device__ static __forceinline__ void put(_Float16* p, int64_t i, float g) {
    p[i] = (_Float16)g;
  }
};
template <>
struct GradOut<float> {
  __device__ static __forceinline__ u32x4 pack(const float (&g)[4]) {
    u32x4 v;
    v.x = f2u(g[0]);
    v.y = f2u(g[1]);
    v.z = f2u(g[2]);
    v.w = f2u(g[3]);
    return v;
  }
  __device__ static __forceinline__ void put(float* p, int64_t i, float g) { p[i] = g; }
};

// One slice of a row of g * ([i == t] - p_i), p_i = 2^((x_i - lse) log2 e):
// its whole vectors (of the nvec from element `head` on) go to
// emit_vec(vector index, gradients); the last slice also takes the elements
// before and after the vectors (every element when nvec == 0), one by one to
// emit_one(i, gradient).
template <typename T, typename EmitVec, typename EmitOne>
__device__ __forceinline__ void logprob_backward_row(const T* __restrict__ row, int64_t V,
                                                     int64_t head, int64_t nvec, const Slice& sl,
                                                     int64_t tgt, float g, float lse,
                                                     EmitVec&& emit_vec, EmitOne&& emit_one) {
  constexpr int E = Vec<T>::kE;
  const float ng = -g;
  stream_vectors<T, kLpBlock, kLpVecs, true>(
      row + head, sl.v0, sl.v1, [&](float(&x)[kLpVecs][E], int64_t vbase, bool last) {
#pragma unroll
        for (int k = 0; k < kLpVecs; ++k) {
          const int64_t vi = vbase + (int64_t)k * kLpBlock;
          if (last && vi >= sl.v1) continue;
          float gr[E];
#pragma unroll
          for (int j = 0; j < E; ++j)
            gr[j] = ng * __builtin_amdgcn_exp2f((x[k][j] - lse) * kLog2e);
          const int64_t d = tgt - head - vi * E;
          if (d >= 0 && d < E) {
            // g (1 - p_t) as -g expm1(x_t - lse): no cancellation when p_t ~ 1
#pragma unroll
            for (int j = 0; j < E; ++j)
              if (j == (int)d) gr[j] = -g * expm1f(x[k][j] - lse);
          }
          emit_vec(vi, gr);
        }
      });
  if (!sl.last) return;
  for_edges(V, head, nvec * E, [&](int64_t i) {
    const float xi = Elem<T>::get(row, i);
    emit_one(i, i == tgt ? -g * expm1f(xi - lse)
                         : ng * __builtin_amdgcn_exp2f((xi - lse) * kLog2e));
  });
}

// Slice k of one row's gradient in the logits' dtype; zeros, without reading
// the row, where g == 0.
template <typename T>
__device__ __forceinline__ void logprob_backward_slice(const T* __restrict__ row, int64_t V,
                                                       int64_t tgt, float g, float lse,
                                                       T* __restrict__ grow, int k, int slices) {
  constexpr int E = Vec<T>::kE;
  // a gradient row at the logits row's own alignment (always, when both are
  // contiguous) has its 16-byte boundaries at the same elements
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(row) ^ reinterpret_cast<uintptr_t>(grow)) & 15u) == 0;
  const int64_t head = row_head(row, V);
  const int64_t nvec = vec_ok ? (V - head) / E : 0;
  const Slice sl = slice_of<E>(nvec, k, slices);
  u32x4* gv = reinterpret_cast<u32x4*>(grow + head);
  if (g == 0.0f) {
    const u32x4 z = {0u, 0u, 0u, 0u};
    for (int64_t vi = sl.v0 + threadIdx.x; vi < sl.v1; vi += kLpBlock)
      __builtin_nontemporal_store(z, gv + vi);
    if (sl.last)
      for_edges(V, head, nvec * E, [&](int64_t i) { GradOut<T>::put(grow, i, 0.0f); });
    return;
  }
  logprob_backward_row<T>(
      row, V, head, nvec, sl, tgt, g, lse,
      [&](int64_t vi, const float(&gr)[E]) {
        __builtin_nontemporal_store(GradOut<T>::pack(gr), gv + vi);
      },
      [&](int64_t i, float gi) { GradOut<T>::put(grow, i, gi); });
}

template <typename T>
__global__ __launch_bounds__(kLpBlock) void logprob_backward_kernel(
    const T* __restrict__ logits, int64_t V, int64_t row_stride, int64_t col_offset,
    const void* __restrict__ targets, int t64, const float* __restrict__ grad_lp,
    const float* __restrict__ lse_in, T* __restrict__ grad, int64_t grad_stride, int slices) {
  const int64_t n = slices > 1 ? blockIdx.x / (uint32_t)slices : blockIdx.x;
  const int64_t tgt = load_target(targets, t64, n) - col_offset;  // outside [0, V): no one-hot term
  logprob_backward_slice<T>(logits + n * row_stride, V, tgt, grad_lp[n], lse_in[n],
                            grad + n * grad_stride, (int)(blockIdx.x - n * slices), slices);
}

// The gradient of the logprobs of token_logprob_kernel: each row's lse is
// x_t - logprob, from one load of its target's logit.  Rows past the first
// St positions of a sequence, and ignored ones, get zeros.  g is grad_lp per
// row, or (count given) the gradient of the mean -sum(lp) / count of one
// scalar.
template <typename T>
__global__ __launch_bounds__(kLpBlock) void token_logprob_backward_kernel(
    TokenRows a, int64_t St, const float* __restrict__ lp, const float* __restrict__ grad_lp,
    const int64_t* __restrict__ count, T* __restrict__ grad, int64_t gbstride, int64_t grstride,
    int slices) {
  const int64_t n = slices > 1 ? blockIdx.x / (uint32_t)slices : flat_workgroup();
  if (n >= a.rows()) return;
  int64_t b, s;
  a.at(n, b, s);
  const T* row = a.row<T>(b, s);
  float g = 0.0f, lse = 0.0f;
  int64_t tgt = 0;
  if (s < St) {
    tgt = a.target(b, s);
    if (!(a.has_ignore && tgt == a.ignore)) {
      const int64_t m = b * St + s;
      g = count ? -grad_lp[0] / (float)count[0] : grad_lp[m];
      // a target outside the row has a NaN logprob
      lse = (tgt >= 0 && tgt < a.V ? Elem<T>::get(row, tgt) : 0.0f) - lp[m];
    }
  }
  logprob_backward_slice<T>(row, a.V, tgt, g, lse, grad + b * gbstride + s * grstride,
                            slices > 1 ? (int)(blockIdx.x - n * slices) : 0, slices);
}

// loss = -sum lp_n / count over the count rows that are not ignored:
// F.cross_entropy's mean, which no value of an ignored row reaches (its
// logprob, token 0's, may be NaN or -inf).  One workgroup: at most some ten
// thousand rows, 4 bytes of logprob and one target each.
__global__ __launch_bounds__(1024) void token_mean_kernel(TokenRows a, int64_t N,
                                                          const float* __restrict__ lp,
                                                          float* __restrict__ loss,
                                                          int64_t* __restrict__ count) {
  __shared__ double rs[1024 / kWave];
  __shared__ int64_t rc[1024 / kWave];
  double sum = 0.0;
  int64_t c = 0;
  for (int64_t n = threadIdx.x; n < N; n += 1024) {
    int64_t b, s;
    a.at(n, b, s);
    if (a.has_ignore && a.target(b, s) == a.ignore) continue;
    sum += (double)lp[n];
    ++c;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    sum += __shfl_xor(sum, o, kWave);
    c += __shfl_xor(c, o, kWave);
  }
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  if (lane == 0) {
    rs[wid] = sum;
    rc[wid] = c;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
#pragma unroll
  for (int w = 1; w < 1024 / kWave; ++w) {
    sum += rs[w];
    c += rc[w];
  }
  loss[0] = (float)(-sum / (double)c);
  count[0] = c;
}

// The same gradient of fp32 logits written as two bf16 arrays, hi = the
// gradient rounded to bf16 and lo = the remainder rounded to bf16, so that
// |grad - hi - lo| <= 2^-16 |grad| (each bf16 rounding is within 2^-8): bf16
// matrix-core GEMMs of both parts carry about 16 significant bits.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split_bf16(float v, uint32_t& hi, uint32_t& lo) {
  hi = bf16_rne(v);
  lo = (hi & 0x7F80u) == 0x7F80u ? 0u : bf16_rne(v - u2f(hi << 16));  // inf / NaN: no remainder
}
__global__ __launch_bounds__(kLpBlock) void logprob_backward_split_kernel(
    const float* __restrict__ logits, int64_t V, int64_t row_stride, int64_t col_offset,
    const void* __restrict__ targets, int t64, const float* __restrict__ grad_lp,
    const float* __restrict__ lse_in, uint16_t* __restrict__ ghi, uint16_t* __restrict__ glo,
    int64_t grad_stride) {
  const int64_t n = blockIdx.x;
  const float* row = logits + n * row_stride;
  uint16_t* hrow = ghi + n * grad_stride;
  uint16_t* lrow = glo + n * grad_stride;
  const float g = grad_lp[n];
  const int64_t tgt = load_target(targets, t64, n) - col_offset;
  const int64_t head = row_head(row, V);
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(hrow + head) |
                        reinterpret_cast<uintptr_t>(lrow + head)) & 7u) == 0;
  const int64_t nvec = vec_ok ? (V - head) / 4 : 0;
  u32x2* hv = reinterpret_cast<u32x2*>(hrow + head);
  u32x2* lv = reinterpret_cast<u32x2*>(lrow + head);
  if (g == 0.0f) {
    const u32x2 z = {0u, 0u};
    for (int64_t vi = threadIdx.x; vi < nvec; vi += kLpBlock) {
      __builtin_nontemporal_store(z, hv + vi);
      __builtin_nontemporal_store(z, lv + vi);
    }
    for_edges(V, head, nvec * 4, [&](int64_t i) { hrow[i] = lrow[i] = 0; });
    return;
  }
  logprob_backward_row<float>(
      row, V, head, nvec, Slice{0, nvec, true, true}, tgt, g, lse_in[n],
      [&](int64_t vi, const float(&gr)[4]) {
        uint32_t h[4], l[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) split_bf16(gr[j], h[j], l[j]);
        const u32x2 ho = {h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
        const u32x2 lo = {l[0] | (l[1] << 16), l[2] | (l[3] << 16)};
        __builtin_nontemporal_store(ho, hv + vi);
        __builtin_nontemporal_store(lo, lv + vi);
      },
      [&](int64_t i, float gi) {
        uint32_t h, l;
        split_bf16(gi, h, l);
        hrow[i] = (uint16_t)h;
        lrow[i] = (uint16_t)l;
      });
}

}  // namespace gtp

using namespace gtp;

namespace {
// Chunks of a row's sum, and the slices of the gradient.
Chunks row_chunks(int dtype, int64_t V) {
  return dtype == GTP_DTYPE_F32 ? chunks_of<float>(V) : chunks_of<uint16_t>(V);
}

// Workgroups per row: eight resident workgroups on every CU when there are
// fewer rows than that, each with a chunk or more (mostly one full step of
// its stream, 32 KB); one per row otherwise.  bf16 [61, 151936] takes 10.5 us
// in ten slices and 16.4 us in one workgroup per row; from 8 x 256 rows on the
// chip is full without them ([8192, 248320] runs at 6.8 TB/s of the 7.0 that a
// read-only pass reaches).
int row_slices(int dtype, int64_t N, int64_t V) {
  const int64_t want = (8 * device_cus() + N - 1) / N;
  return (int)max((int64_t)1, min(want, (int64_t)row_chunks(dtype, V).n));
}

// Workspace: the rows' arrival counters, then 3 floats per chunk.
size_t row_slices_bytes(int64_t N, int slices, int chunks) {
  return slices > 1 ? (size_t)N * 4 + (size_t)(N * chunks) * 12 : 0;
}

// The look at the targets: a few thousand per workgroup; the words of
// workgroups that are not launched are good.
void targets_launch(const TokenRows& a, int64_t N, uint32_t* ctr, int n_ctr, const uint32_t* flag_a,
                    const uint32_t* flag_b, uint32_t* verdict, hipStream_t s) {
  const int blocks = (int)max((int64_t)1, min((int64_t)GTP_VERDICT_WORDS, (N + 4095) / 4096));
  for (int i = blocks; verdict && i < GTP_VERDICT_WORDS; ++i) verdict[i] = GTP_VERDICT_GOOD;
  hipLaunchKernelGGL(token_targets_kernel, dim3((unsigned)blocks), dim3(kVerdictBlock), 0, s, a, N,
                     ctr, n_ctr, flag_a, flag_b, verdict);
}

template <typename T>
void token_logprob_launch(const TokenRows& a, const TokenOut& out, int64_t N, int slices,
                          uint32_t* ctr, hipStream_t s) {
  const Chunks ch = chunks_of<T>(a.V);
  const dim3 grid = flat_grid(N * slices), block(kLpBlock);
  float* partial = reinterpret_cast<float*>(ctr + (slices > 1 ? N : 0));
  if (out.H)
    launch_timed(token_logprob_kernel<T, true>, grid, block, s, a, out, ch, slices, ctr, partial);
  else
    launch_timed(token_logprob_kernel<T, false>, grid, block, s, a, out, ch, slices, ctr, partial);
}

// GTP_OK and the device form of `r`, with sequences that follow one another
// at the rows' own stride joined into one.
int token_rows(const gtp_token_rows* r, TokenRows& a, bool need_targets = true) {
  if (!r || r->B < 0 || r->S < 0 || r->V <= 0 || (r->S > 1 && r->row_stride < r->V) ||
      r->batch_stride < 0 || r->row_stride < 0 || r->target_batch_stride < 0 ||
      r->target_row_stride < 0 || r->dtype < GTP_DTYPE_F32 || r->dtype > GTP_DTYPE_F16)
    return GTP_ERR_INVALID_ARGUMENT;
  if (r->B > 0x7FFFFFFFll || r->S > 0x7FFFFFFFll || (r->B > 0 && r->S > 0x7FFFFFFFll / r->B) ||
      r->V > 0x7FFFFFFFll)
    return GTP_ERR_UNSUPPORTED;
  if (r->B > 0 && r->S > 0 && (!r->logits || (need_targets && !r->targets)))
    return GTP_ERR_INVALID_ARGUMENT;
  a = TokenRows{r->logits, r->targets, r->V, r->S, r->batch_stride, r->row_stride,
                r->target_batch_stride, r->target_row_stride, r->ignore_index, (int)r->B,
                r->targets_int64 ? 1 : 0, r->has_ignore ? 1 : 0};
  return GTP_OK;
}

// One sequence of B * S rows where both strides allow it (St: positions with
// a target; the outputs must be indexed alike).
void join_rows(TokenRows& a, int64_t St) {
  if (a.B > 1 && St == a.S && a.bstride == a.S * a.rstride && a.tbstride == a.S * a.trstride) {
    a.S *= a.B;
    a.B = 1;
  }
}
}  // namespace

extern "C" size_t gtp_token_logprob_workspace_bytes(int dtype, int64_t N, int64_t V) {
  if (N <= 0 || V <= 0 || N > 0x3FFFFFFll) return 0;
  return row_slices_bytes(N, row_slices(dtype, N, V), row_chunks(dtype, V).n);
}

extern "C" int gtp_token_logprob_rows(const gtp_token_rows* rows, float* out_logprob,
                                      float* out_entropy, int32_t* out_status, uint32_t* verdict,
                                      void* workspace, size_t workspace_bytes, void* stream) {
  TokenRows a;
  const int rc = token_rows(rows, a);
  if (rc != GTP_OK) return rc;
  const int64_t N = (int64_t)a.B * a.S;
  if (N > 0 && !out_logprob) return GTP_ERR_INVALID_ARGUMENT;
  if (N == 0) {
    for (int i = 0; verdict && i < GTP_VERDICT_WORDS; ++i) verdict[i] = GTP_VERDICT_GOOD;
    return GTP_OK;
  }
  join_rows(a, a.S);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  int slices = row_slices(rows->dtype, N, a.V);
  if (!workspace ||
      workspace_bytes < row_slices_bytes(N, slices, row_chunks(rows->dtype, a.V).n))
    slices = 1;
  uint32_t* ctr = reinterpret_cast<uint32_t*>(workspace);
  if (slices > 1 || verdict)
    targets_launch(a, N, ctr, slices > 1 ? (int)N : 0, nullptr, nullptr, verdict, s);
  const TokenOut out{out_logprob, out_entropy, out_status};
  switch (rows->dtype) {
    case GTP_DTYPE_BF16:
      token_logprob_launch<uint16_t>(a, out, N, slices, ctr, s);
      break;
    case GTP_DTYPE_F16:
      token_logprob_launch<_Float16>(a, out, N, slices, ctr, s);
      break;
    default:
      token_logprob_launch<float>(a, out, N, slices, ctr, s);
  }
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

extern "C" int gtp_stream_capturing(void* stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(reinterpret_cast<hipStream_t>(stream), &st) == hipSuccess &&
         st != hipStreamCaptureStatusNone;
}

extern "C" int gtp_verdict_wait(const uint32_t* verdict, int* found, void* stream) {
  if (!verdict || !found) return GTP_ERR_INVALID_ARGUMENT;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto pending = [&] {
    for (int i = 0; i < GTP_VERDICT_WORDS; ++i)
      if (__atomic_load_n(verdict + i, __ATOMIC_RELAXED) == GTP_VERDICT_PENDING) return true;
    return false;
  };
  // The word lands about a microsecond after its kernel; waiting for the
  // stream instead would wait for the rows too.  The stream's state is
  // looked at now and then, so that failed work ends the wait.
  bool done = !pending();
  for (int round = 0; !done; ++round) {
    for (int i = 0; i < 2000 && !done; ++i) {
      __builtin_ia32_pause();
      done = !pending();
    }
    if (done) break;
    const hipError_t e = hipStreamQuery(s);
    if (e != hipErrorNotReady) {
      if (e != hipSuccess || pending()) return GTP_ERR_LAUNCH;
      break;
    }
    // after a few hundred microseconds the stream has other work to do first
    if (round > 16) std::this_thread::sleep_for(std::chrono::microseconds(20));
  }
  uint32_t all = 0;
  for (int i = 0; i < GTP_VERDICT_WORDS; ++i) all |= __atomic_load_n(verdict + i, __ATOMIC_RELAXED);
  *found = (int)(all >> 1);  // without GTP_VERDICT_GOOD
  return GTP_OK;
}

extern "C" int gtp_targets_verdict(const void* targets, int targets_int64, int64_t N,
                                   int64_t target_stride, int64_t V, const uint32_t* flag_a,
                                   const uint32_t* flag_b, uint32_t* verdict, void* stream) {
  if (N < 0 || V <= 0 || target_stride < 0 || (N > 0 && !targets) || !verdict)
    return GTP_ERR_INVALID_ARGUMENT;
  if (N > 0x7FFFFFFFll) return GTP_ERR_UNSUPPORTED;
  const TokenRows a{nullptr, targets, V, N, 0, 0, 0, target_stride, 0, 1, targets_int64 ? 1 : 0, 0};
  // at least one workgroup, which looks at the flags
  targets_launch(a, N, nullptr, 0, flag_a, flag_b, verdict, reinterpret_cast<hipStream_t>(stream));
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}


extern "C" int gtp_token_mean_loss(const gtp_token_rows* rows, const float* logprob, float* loss,
                                   int64_t* count, void* stream) {
  TokenRows a;
  const int rc = token_rows(rows, a);
  if (rc != GTP_OK) return rc;
  const int64_t N = (int64_t)a.B * a.S;
  if (!loss || !count || (N > 0 && !logprob)) return GTP_ERR_INVALID_ARGUMENT;
  join_rows(a, a.S);
  hipLaunchKernelGGL(token_mean_kernel, dim3(1), dim3(1024), 0,
                     reinterpret_cast<hipStream_t>(stream), a, N, logprob, loss, count);
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

extern "C" int gtp_token_logprob_backward(const gtp_token_rows* rows, int64_t positions,
                                          const float* logprob, const float* grad,
                                          const int64_t* mean_count, void* grad_logits,
                                          int64_t grad_batch_stride, int64_t grad_row_stride,
                                          void* stream) {
  TokenRows a;
  const int rc = token_rows(rows, a, positions != 0);
  if (rc != GTP_OK) return rc;
  const int64_t N = (int64_t)a.B * a.S;
  if (positions < 0 || positions > a.S || grad_batch_stride < 0 ||
      (a.S > 1 && grad_row_stride < a.V))
    return GTP_ERR_INVALID_ARGUMENT;
  if (N == 0) return GTP_OK;
  if (!grad || !grad_logits || (positions > 0 && !logprob)) return GTP_ERR_INVALID_ARGUMENT;
  if (grad_batch_stride == a.S * grad_row_stride) join_rows(a, positions);
  if (a.B == 1) positions = positions == rows->S ? a.S : positions;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int slices = row_slices(rows->dtype, N, a.V);
  const dim3 grid = flat_grid(N * slices), block(kLpBlock);
  switch (rows->dtype) {
    case GTP_DTYPE_BF16:
      launch_timed(token_logprob_backward_kernel<uint16_t>, grid, block, s, a, positions, logprob,
                   grad, mean_count, reinterpret_cast<uint16_t*>(grad_logits), grad_batch_stride,
                   grad_row_stride, slices);
      break;
    case GTP_DTYPE_F16:
      launch_timed(token_logprob_backward_kernel<_Float16>, grid, block, s, a, positions, logprob,
                   grad, mean_count, reinterpret_cast<_Float16*>(grad_logits), grad_batch_stride,
                   grad_row_stride, slices);
      break;
    default:
      launch_timed(token_logprob_backward_kernel<float>, grid, block, s, a, positions, logprob,
                   grad, mean_count, reinterpret_cast<float*>(grad_logits), grad_batch_stride,
                   grad_row_stride, slices);
  }
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

extern "C" int gtp_logprob_entropy_rows(const void* logits, int dtype, int64_t N, int64_t V,
                                        int64_t row_stride, const void* targets, int targets_int64,
                                        float* out_logprob, float* out_entropy, int32_t* out_status,
                                        void* stream) {
  if (N < 0 || V <= 0 || row_stride < V || (N > 0 && (!logits || !targets || !out_logprob)))
    return GTP_ERR_INVALID_ARGUMENT;
  if (N > 0x7FFFFFFFll) return GTP_ERR_UNSUPPORTED;
  if (N == 0) return GTP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const TokenRows a{logits, targets, V, N, 0, row_stride, 0, 1, 0, 1, targets_int64 ? 1 : 0, 0};
  const TokenOut out{out_logprob, out_entropy, out_status};
  switch (dtype) {
    case GTP_DTYPE_BF16:
      token_logprob_launch<uint16_t>(a, out, N, 1, nullptr, s);
      break;
    case GTP_DTYPE_F16:
      token_logprob_launch<_Float16>(a, out, N, 1, nullptr, s);
      break;
    case GTP_DTYPE_F32:
      token_logprob_launch<float>(a, out, N, 1, nullptr, s);
      break;
    default:
      return GTP_ERR_INVALID_ARGUMENT;
  }
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

namespace gtp {
thread_local LaunchEvents g_next_launch_events{nullptr, nullptr};
}

extern "C" int gtp_time_next_launch(void* start_event, void* stop_event) {
  if (!start_event || !stop_event) return GTP_ERR_INVALID_ARGUMENT;
  g_next_launch_events = LaunchEvents{reinterpret_cast<hipEvent_t>(start_event),
                                      reinterpret_cast<hipEvent_t>(stop_event)};
  return GTP_OK;
}

namespace gtp {
// Read-only streaming floor: one workgroup of 1024 threads per row reads the
// row's 16-byte vectors once (non-temporal, 8 per lane in flight, the
// samplers' access pattern) and XORs them; a row whose XOR equals a fixed
// pattern writes it, so the loads cannot be dropped.
__global__ __launch_bounds__(1024) void stream_read_kernel(const unsigned char* __restrict__ data,
                                                           int64_t row_bytes, int64_t stride,
                                                           uint32_t* __restrict__ out) {
  typedef uint32_t v4 __attribute__((ext_vector_type(4)));
  const v4* row = reinterpret_cast<const v4*>(data + (int64_t)blockIdx.x * stride);
  const int64_t nvec = row_bytes / 16;
  constexpr int G = 8;
  v4 acc = {0u, 0u, 0u, 0u};
  for (int64_t v0 = threadIdx.x; v0 < nvec; v0 += (int64_t)1024 * G) {
    v4 q[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int64_t v = v0 + (int64_t)g * 1024;
      q[g] = v < nvec ? __builtin_nontemporal_load(row + v) : v4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int g = 0; g < G; ++g) acc ^= q[g];
  }
  const uint32_t x = acc.x ^ acc.y ^ acc.z ^ acc.w;
  if (x == 0x9E3779B9u) out[blockIdx.x] = x;
}
}  // namespace gtp

extern "C" int gtp_stream_read_rows(const void* data, int64_t rows, int64_t row_bytes,
                                    int64_t row_stride_bytes, uint32_t* out, void* stream) {
  if (rows < 0 || row_bytes < 0 || row_stride_bytes < row_bytes || (rows > 0 && (!data || !out)))
    return GTP_ERR_INVALID_ARGUMENT;
  if ((reinterpret_cast<uintptr_t>(data) & 15u) || (row_bytes & 15) || (row_stride_bytes & 15))
    return GTP_ERR_UNSUPPORTED;
  if (rows > 0x7FFFFFFFll) return GTP_ERR_UNSUPPORTED;
  if (rows == 0 || row_bytes == 0) return GTP_OK;
  launch_timed(stream_read_kernel, dim3((unsigned)rows), dim3(1024),
               reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const unsigned char*>(data),
               row_bytes, row_stride_bytes, out);
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

extern "C" int gtp_lse_partial_rows(const void* logits, int dtype, int64_t N, int64_t Vc,
                                    int64_t row_stride, int64_t col_offset, const void* targets,
                                    int targets_int64, float* state, int accumulate, void* stream) {
  if (N < 0 || Vc <= 0 || row_stride < Vc || col_offset < 0 || (N > 0 && (!logits || !state)))
    return GTP_ERR_INVALID_ARGUMENT;
  if (N > 0x7FFFFFFFll) return GTP_ERR_UNSUPPORTED;
  if (N == 0) return GTP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)N), block(kLpBlock);
  switch (dtype) {
    case GTP_DTYPE_BF16:
      hipLaunchKernelGGL(lse_partial_kernel<uint16_t>, grid, block, 0, s,
                         reinterpret_cast<const uint16_t*>(logits), Vc, row_stride, col_offset,
                         targets, targets_int64, state, accumulate, chunks_of<uint16_t>(Vc));
      break;
    case GTP_DTYPE_F16:
      hipLaunchKernelGGL(lse_partial_kernel<_Float16>, grid, block, 0, s,
                         reinterpret_cast<const _Float16*>(logits), Vc, row_stride, col_offset,
                         targets, targets_int64, state, accumulate, chunks_of<_Float16>(Vc));
      break;
    case GTP_DTYPE_F32:
      hipLaunchKernelGGL(lse_partial_kernel<float>, grid, block, 0, s,
                         reinterpret_cast<const float*>(logits), Vc, row_stride, col_offset,
                         targets, targets_int64, state, accumulate, chunks_of<float>(Vc));
      break;
    default:
      return GTP_ERR_INVALID_ARGUMENT;
  }
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

extern "C" int gtp_lse_finalize_rows(const float* state, int64_t N, float* out_logprob,
                                     float* out_entropy, void* stream) {
  if (N < 0 || (N > 0 && !state)) return GTP_ERR_INVALID_ARGUMENT;
  if (N > 0x7FFFFFFFll) return GTP_ERR_UNSUPPORTED;
  if (N == 0) return GTP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)((N + 255) / 256);
  hipLaunchKernelGGL(lse_finalize_kernel, dim3(blocks), dim3(256), 0, s, state, N, out_logprob,
                     out_entropy);
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

extern "C" const char* gtp_version(void) { return "graspo_tokpath 0.2 gfx950"; }

extern "C" int gtp_logprob_backward_split_rows(const float* logits, int64_t N, int64_t V,
                                               int64_t row_stride, int64_t col_offset,
                                               const void* targets, int targets_int64,
                                               const float* grad_logprob, const float* lse,
                                               uint16_t* grad_hi, uint16_t* grad_lo,
                                               int64_t grad_stride, void* stream) {
  if (N < 0 || V <= 0 || row_stride < V || grad_stride < V ||
      (N > 0 && (!logits || !targets || !grad_logprob || !lse || !grad_hi || !grad_lo)))
    return GTP_ERR_INVALID_ARGUMENT;
  if (N > 0x7FFFFFFFll) return GTP_ERR_UNSUPPORTED;
  if (N == 0) return GTP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(logprob_backward_split_kernel, dim3((unsigned)N), dim3(kLpBlock), 0, s,
                     logits, V, row_stride, col_offset, targets, targets_int64, grad_logprob,
                     lse, grad_hi, grad_lo, grad_stride);
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

// bf16(-g_n p) of vocabulary-major fp32 logits, p = exp(x_t[v, n] - lse_n):
// the softmax part of g_n ([v == t_n] - p) without the one-hot term, which
// the caller adds in fp32 (it is the one term of a token's gradient near g
// in size; here every element is g p, rounded once to bf16, within 2^-8 of
// it).  A workgroup takes 1024 consecutive tokens (4 per thread, their g and
// lse held in registers) of kSgRows vocabulary rows; a token with g == 0
// gets zeros.
constexpr int kSgRows = 16;
typedef float f32x4v __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void softmax_grad_bf16_cols_kernel(
    const float* __restrict__ logits_t, int64_t V, int64_t N, int64_t ld,
    const float* __restrict__ grad_lp, const float* __restrict__ lse_in,
    uint16_t* __restrict__ grad_t, int64_t gld, int vec) {
  const int64_t n0 = (int64_t)blockIdx.x * 1024 + threadIdx.x * 4;
  if (n0 >= N) return;
  const int64_t v0 = (int64_t)blockIdx.y * kSgRows;
  const int cnt = (int)min((int64_t)4, N - n0);
  float ng[4], c[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float g = j < cnt ? grad_lp[n0 + j] : 0.0f;
    ng[j] = -g;
    // a token with g == 0 gets exactly zero
    c[j] = g == 0.0f ? kNegInf : (j < cnt ? lse_in[n0 + j] : 0.0f);
  }
  // x - lse first: exact for x near lse at any magnitude
  auto grad_of = [&](float x, int j) {
    return c[j] == kNegInf ? 0.0f : ng[j] * __builtin_amdgcn_exp2f((x - c[j]) * kLog2e);
  };
  if (vec && cnt == 4) {
#pragma unroll 4
    for (int r = 0; r < kSgRows; ++r) {
      const int64_t v = v0 + r;
      if (v >= V) break;
      const f32x4v x = __builtin_nontemporal_load(reinterpret_cast<const f32x4v*>(logits_t + v * ld + n0));
      const u32x2 o = {bf16_rne(grad_of(x.x, 0)) | (bf16_rne(grad_of(x.y, 1)) << 16),
                       bf16_rne(grad_of(x.z, 2)) | (bf16_rne(grad_of(x.w, 3)) << 16)};
      __builtin_nontemporal_store(o, reinterpret_cast<u32x2*>(grad_t + v * gld + n0));
    }
    return;
  }
  for (int r = 0; r < kSgRows; ++r) {
    const int64_t v = v0 + r;
    if (v >= V) break;
    for (int j = 0; j < cnt; ++j)
      grad_t[v * gld + n0 + j] = (uint16_t)bf16_rne(grad_of(logits_t[v * ld + n0 + j], j));
  }
}

// The same values written token-major as well, grad_n[n, v] (and, unless
// grad_t is null, vocabulary-major as above), from one read of the logits: a
// workgroup takes 256 tokens x 64 vocabulary rows.  Each thread computes 4
// consecutive tokens of 16 rows (16-byte loads along the tokens, 8-byte
// vocabulary-major stores) and puts them in an LDS tile [64][256 + 2]; then
// each group of 8 lanes writes one token's 64 values, a whole 128-byte line,
// 16 bytes a lane.  The tile's row pitch of 129 words puts the 8 rows a group
// reads at once on distinct banks.
constexpr int kDgTok = 256, kDgRows = 64, kDgPitch = kDgTok + 2;
__global__ __launch_bounds__(256) void softmax_grad_bf16_dual_kernel(
    const float* __restrict__ logits_t, int64_t V, int64_t N, int64_t ld,
    const float* __restrict__ grad_lp, const float* __restrict__ lse_in,
    uint16_t* __restrict__ grad_t, int64_t gld, uint16_t* __restrict__ grad_n, int64_t nld,
    int vec) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[kDgRows * kDgPitch];
  const int t = threadIdx.x;
  const int64_t nb = (int64_t)blockIdx.x * kDgTok, vb = (int64_t)blockIdx.y * kDgRows;
  const int nl = (t & 63) * 4;  // the thread's first token in the tile
  const int64_t n0 = nb + nl;
  const int cnt = (int)max((int64_t)0, min((int64_t)4, N - n0));
  float ng[4], c[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float g = j < cnt ? grad_lp[n0 + j] : 0.0f;
    ng[j] = -g;
    c[j] = g == 0.0f ? kNegInf : (j < cnt ? lse_in[n0 + j] : 0.0f);
  }
  auto grad_of = [&](float x, int j) {
    return c[j] == kNegInf ? 0.0f : ng[j] * __builtin_amdgcn_exp2f((x - c[j]) * kLog2e);
  };
#pragma unroll 4
  for (int i = 0; i < kDgRows / 4; ++i) {
    const int r = (t >> 6) + 4 * i;
    const int64_t v = vb + r;
    uint32_t o[4] = {0u, 0u, 0u, 0u};
    if (v < V) {
      if (vec && cnt == 4) {
        const f32x4v x = __builtin_nontemporal_load(reinterpret_cast<const f32x4v*>(logits_t + v * ld + n0));
        o[0] = bf16_rne(grad_of(x.x, 0));
        o[1] = bf16_rne(grad_of(x.y, 1));
        o[2] = bf16_rne(grad_of(x.z, 2));
        o[3] = bf16_rne(grad_of(x.w, 3));
        if (grad_t) {
          const u32x2 w = {o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
          __builtin_nontemporal_store(w, reinterpret_cast<u32x2*>(grad_t + v * gld + n0));
        }
      } else {
        for (int j = 0; j < cnt; ++j) {
          o[j] = bf16_rne(grad_of(logits_t[v * ld + n0 + j], j));
          if (grad_t) grad_t[v * gld + n0 + j] = (uint16_t)o[j];
        }
      }
    }
    uint32_t* dst = reinterpret_cast<uint32_t*>(tile + r * kDgPitch + nl);
    dst[0] = o[0] | (o[1] << 16);
    dst[1] = o[2] | (o[3] << 16);
  }
  __syncthreads();
  // token-major: 8 lanes per token, lane c8 of the group the values of rows
  // 8 c8 .. 8 c8 + 7, 32 tokens per pass
  const int c8 = t & 7;
  const int64_t nv = min((int64_t)kDgRows, V - vb);
#pragma unroll 2
  for (int p = 0; p < kDgTok / 32; ++p) {
    const int tl = p * 32 + (t >> 3);
    const int64_t n = nb + tl;
    if (n >= N) break;
    uint16_t* row = grad_n + n * nld + vb;
    if (vec && nv == kDgRows) {
      uint32_t h[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) h[k] = tile[(8 * c8 + k) * kDgPitch + tl];
      const u32x4 w = {h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                       h[6] | (h[7] << 16)};
      *reinterpret_cast<u32x4*>(row + 8 * c8) = w;
    } else {
      for (int k = 0; k < 8; ++k)
        if (8 * c8 + k < nv) row[8 * c8 + k] = tile[(8 * c8 + k) * kDgPitch + tl];
    }
  }
}

extern "C" int gtp_softmax_grad_bf16_cols(const float* logits_t, int64_t V, int64_t N,
                                          int64_t logits_stride, const float* grad_logprob,
                                          const float* lse, uint16_t* grad_t, int64_t grad_stride,
                                          uint16_t* grad_n, int64_t grad_n_stride,
                                          void* stream) {
  if (N < 0 || V <= 0 || logits_stride < N || (grad_t && grad_stride < N) ||
      (grad_n && grad_n_stride < V) ||
      (N > 0 && (!logits_t || !grad_logprob || !lse || (!grad_t && !grad_n))))
    return GTP_ERR_INVALID_ARGUMENT;
  if (N > 0x7FFFFFFFll || V > ((int64_t)65535 * kSgRows) ||
      logits_stride > ((int64_t)1 << 40) / V || (grad_t && grad_stride > ((int64_t)1 << 40) / V) ||
      (grad_n && (N > 0 && grad_n_stride > ((int64_t)1 << 40) / N)))
    return GTP_ERR_UNSUPPORTED;
  if (N == 0) return GTP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool in_vec = (reinterpret_cast<uintptr_t>(logits_t) & 15u) == 0 && (logits_stride & 3) == 0;
  const bool t_vec = !grad_t || ((reinterpret_cast<uintptr_t>(grad_t) & 7u) == 0 && (grad_stride & 3) == 0);
  if (grad_n) {
    const int vec = in_vec && t_vec && (reinterpret_cast<uintptr_t>(grad_n) & 15u) == 0 &&
                            (grad_n_stride & 7) == 0
                        ? 1
                        : 0;
    const dim3 grid((unsigned)((N + kDgTok - 1) / kDgTok), (unsigned)((V + kDgRows - 1) / kDgRows));
    launch_timed(softmax_grad_bf16_dual_kernel, grid, dim3(256), s, logits_t, V, N, logits_stride,
                 grad_logprob, lse, grad_t, grad_stride, grad_n, grad_n_stride, vec);
  } else {
    const int vec = in_vec && t_vec ? 1 : 0;
    const dim3 grid((unsigned)((N + 1023) / 1024), (unsigned)((V + kSgRows - 1) / kSgRows));
    launch_timed(softmax_grad_bf16_cols_kernel, grid, dim3(256), s, logits_t, V, N, logits_stride,
                 grad_logprob, lse, grad_t, grad_stride, vec);
  }
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

extern "C" int gtp_logprob_backward_rows(const void* logits, int dtype, int64_t N, int64_t V,
                                         int64_t row_stride, int64_t col_offset,
                                         const void* targets, int targets_int64,
                                         const float* grad_logprob, const float* lse, void* grad,
                                         int64_t grad_stride, void* stream) {
  if (N < 0 || V <= 0 || row_stride < V || grad_stride < V ||
      (N > 0 && (!logits || !targets || !grad_logprob || !lse || !grad)))
    return GTP_ERR_INVALID_ARGUMENT;
  if (N > 0x7FFFFFFFll) return GTP_ERR_UNSUPPORTED;
  if (N == 0) return GTP_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int slices = N <= 0x3FFFFFF ? row_slices(dtype, N, V) : 1;
  const dim3 grid((unsigned)(N * slices)), block(kLpBlock);
  switch (dtype) {
    case GTP_DTYPE_BF16:
      launch_timed(logprob_backward_kernel<uint16_t>, grid, block, s,
                         reinterpret_cast<const uint16_t*>(logits), V, row_stride, col_offset,
                         targets, targets_int64, grad_logprob, lse,
                         reinterpret_cast<uint16_t*>(grad), grad_stride, slices);
      break;
    case GTP_DTYPE_F16:
      launch_timed(logprob_backward_kernel<_Float16>, grid, block, s,
                         reinterpret_cast<const _Float16*>(logits), V, row_stride, col_offset,
                         targets, targets_int64, grad_logprob, lse,
                         reinterpret_cast<_Float16*>(grad), grad_stride, slices);
      break;
    case GTP_DTYPE_F32:
      launch_timed(logprob_backward_kernel<float>, grid, block, s,
                         reinterpret_cast<const float*>(logits), V, row_stride, col_offset,
                         targets, targets_int64, grad_logprob, lse,
                         reinterpret_cast<float*>(grad), grad_stride, slices);
      break;
    default:
      return GTP_ERR_INVALID_ARGUMENT;
  }
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}
