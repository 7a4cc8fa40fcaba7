// tokpath_sampler_greedy.h -- greedy rows in one read (gfx950).
//
// Greedy decoding is an argmax of the allowed tokens' penalised logits and
// the raw row's log-sum-exp (the logprob output), the reference's
// logits.argmax(dim=-1) (src/graspo/backends/graspoflow/tensor_utils.py:658).
// It needs none of the candidate machinery of sampler_split_kernel (a pilot,
// a threshold, a pool, a ranking), whose serial steps were most of a small
// call.  Each row is cut into S slices; every thread folds its tokens into
// (m, s) and its best (y, id), and the last of the row's workgroups to arrive
// merges the slices.  Rows may start at any element.  The slices and their
// threads' shares are the split kernel's, so in 16-bit types a slice within
// that kernel's pilot (four vectors per thread, three in fp16) gives the same
// log-sum-exp to the bit: the logprob of a row that is nearly one-hot, ln(1 +
// a little), magnifies a unit of the sum.  (Past its pilot the split kernel's
// waves share a slice out as they go, and its sum varies from call to call;
// this kernel's never does.)
//
// Bound by the latency of a launch, one trip to memory and the arrival on
// small batches, by the stream on large ones.  bf16 [1, 151936], the split
// kernel before: 15.5 -> 7.0 us; [64, 151936] 20.6 -> 9.2; [256, 151936] 18.5
// -> 16.7; fp32 [256, 248320] 71.9 -> 42.7; unaligned bf16 [16, 50257] (the
// row-wise kernel before) 30.4 -> 7.8.
#pragma once

namespace gtp {
namespace greedy {

using spread::put;
using spread::Range;
using spread::take;

constexpr int kT = 1024;   // threads of a workgroup

// One slice's results (the arrival counters lie elsewhere).
struct Part {
  unsigned long long key;  // rank_key of the best token, 0: none
  float m, s;
  uint32_t bad, pad[3];
};

// The row's outputs; all lanes of one wave, with the merged results.
template <typename T>
__device__ __forceinline__ void finish(const SamplerArgs& a, int64_t b, uint32_t* pen,
                                       unsigned long long key, float m, float s, bool bad) {
  const bool raw_nonfinite = s != s || m == kPosInf;
  const float lse_ln = __builtin_amdgcn_logf(s) * kLn2;
  const float y = rank_key_y(key);
  if (!bad && (raw_nonfinite || key == 0ull || y == kPosInf)) {
    greedy_argmax_rescan<T>(a, b, pen, true, raw_nonfinite, m, lse_ln);
    return;
  }
  if ((threadIdx.x & (kWave - 1)) != 0) return;
  const bool fin = a.finished && a.finished[b];
  if (bad) {
    write_row_f(a, b, fin, GTP_ROW_BAD_HISTORY, -1, 0.f, 0.f, 0, 0.f, -1);
    return;
  }
  const int32_t id = rank_key_id(key);
  const T* row = reinterpret_cast<const T*>(a.logits) + b * a.row_stride;
  write_row_f(a, b, fin, GTP_ROW_OK, id, raw_logprob(Elem<T>::get(row, id), m, lse_ln), 0.0f, 1, y,
              id);
}

// kExtra: an allow mask or a penalty.
// per: groups of 8 tokens per slice, a multiple of 4.
template <typename T, bool kExtra>
__global__ __launch_bounds__(kT) void sampler_greedy_kernel(SamplerArgs a, uint32_t per,
                                                            uint32_t* ctr, Part* parts) {
  __shared__ uint32_t pen_bits[GTP_SAMPLER_MAX_V / 32];
  __shared__ unsigned long long red_k[kT / kWave];
  __shared__ float red[kT / kWave][2];
  const int k = blockIdx.x, S = gridDim.x;
  const int64_t b = blockIdx.y;
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const T* row = reinterpret_cast<const T*>(a.logits) + b * a.row_stride;
  const uint32_t* mrow = a.mask ? a.mask + b * a.mask_stride : nullptr;
  const uint32_t ng = (uint32_t)(a.V / 8), g0 = min((uint32_t)k * per, ng);
  const Range r{g0, min(g0 + per, ng), k == S - 1};
  const bool use_pen = kExtra && a.hist_len > 0 && a.rho != 1.0f;
  bool bad = false;
  if (a.hist_len > 0 && (use_pen || k == 0)) bad = spread::slice_pen(a, b, r, use_pen, pen_bits, kT);
  Lse3 st{kNegInf, 0.0f, 0.0f};
  float by = kNegInf;
  uint32_t bid = 0u;
  spread::for_groups<T, kT, kExtra>(
      row, mrow, use_pen ? reinterpret_cast<const uint8_t*>(pen_bits) : nullptr, a.V, r,
      [&](const float(&x)[8], uint32_t id, uint32_t al, uint32_t pb, int n) {
        float y[8];
        float g;
        if (n == 8) {
          g = vec_max<8>(x);
          float z[1][8];
#pragma unroll
          for (int j = 0; j < 8; ++j) z[0][j] = x[j];
          lse_fold_block_max<false, 1, 8>(st, z, g);
          if (kExtra) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              y[j] = (al >> j) & 1u ? spread::penalise(x[j], (pb >> j) & 1u, a.rho) : kNegInf;
            g = vec_max<8>(y);
          }
        } else {
          const float z[1][4] = {{x[0], kNegInf, kNegInf, kNegInf}};
          lse_fold_block_max<false, 1, 4>(st, z, x[0]);
          g = y[0] = al ? spread::penalise(x[0], pb, a.rho) : kNegInf;
        }
        if (g > by) {  // ids ascend: the first of equals stays
          by = g;
          uint32_t j = 0u;
          if (n == 8) {
#pragma unroll
            for (int i = 7; i >= 0; --i) j = (kExtra ? y[i] : x[i]) == g ? (uint32_t)i : j;
          }
          bid = id + j;
        }
      });
  unsigned long long key = by > kNegInf ? rank_key(by + 0.0f, (int32_t)bid) : 0ull;
  key = wave_max_u64(key);
  float m = st.m, s = st.s;
  wave_lse2(m, s);
  if (lane == 0) {
    red_k[wid] = key;
    red[wid][0] = m;
    red[wid][1] = s;
  }
  __syncthreads();
  if (wid != 0) return;
  const bool in = lane < kT / kWave;
  key = wave_max_u64(in ? red_k[lane] : 0ull);
  m = in ? red[lane][0] : kNegInf;
  s = in ? red[lane][1] : 0.0f;
  wave_lse2(m, s);
  if (S > 1) {
    // published and counted as in the other split kernels: agent-scope stores
    // write through, and vmcnt(0) waits for them before the arrival
    Part* p = parts + b * S;
    uint32_t arrived = 0;
    if (lane == 0) {
      put(&p[k].key, key);
      put(&p[k].m, m);
      put(&p[k].s, s);
      put(&p[k].bad, bad ? 1u : 0u);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane == 0)
      arrived = __hip_atomic_fetch_add(ctr + b, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane((int)arrived) != S - 1) return;
    asm volatile("" ::: "memory");
    // every workgroup of the row has arrived: back to zero for the next call
    if (lane == 0) put(ctr + b, 0u);
    const bool mine = lane < S;
    p += mine ? lane : 0;
    const unsigned long long pk = take(&p->key);
    const float pm = take(&p->m), ps = take(&p->s);
    const uint32_t pbad = take(&p->bad);
    key = wave_max_u64(mine ? pk : 0ull);
    m = mine ? pm : kNegInf;
    s = mine ? ps : 0.0f;
    wave_lse2(m, s);
    bad = __ballot(mine && pbad != 0u) != 0ull;
  }
  finish<T>(a, b, pen_bits, key, m, s, bad);
}

template <typename T, bool kExtra>
void launch_as(const SamplerArgs& a, int64_t B, int S, uint32_t per, uint32_t* ctr, Part* parts,
               hipStream_t s) {
  launch_timed(sampler_greedy_kernel<T, kExtra>, dim3((unsigned)S, (unsigned)B), dim3(kT), s, a, per,
               ctr, parts);
}

template <typename T>
void launch(const SamplerArgs& a, int64_t B, int S, uint32_t per, uint32_t* ctr, Part* parts,
            hipStream_t s) {
  if (a.mask || (a.hist_len > 0 && a.rho != 1.0f))
    launch_as<T, true>(a, B, S, per, ctr, parts, s);
  else
    launch_as<T, false>(a, B, S, per, ctr, parts, s);
}

}  // namespace greedy

int launch_greedy(const SamplerArgs& a, int dtype, int64_t B, int S, int64_t per, void* counters,
                  void* parts, hipStream_t s) {
  uint32_t* ctr = reinterpret_cast<uint32_t*>(counters);
  greedy::Part* p = reinterpret_cast<greedy::Part*>(parts);
  if (dtype == GTP_DTYPE_BF16)
    greedy::launch<uint16_t>(a, B, S, (uint32_t)per, ctr, p, s);
  else if (dtype == GTP_DTYPE_F16)
    greedy::launch<_Float16>(a, B, S, (uint32_t)per, ctr, p, s);
  else
    greedy::launch<float>(a, B, S, (uint32_t)per, ctr, p, s);
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

}  // namespace gtp
