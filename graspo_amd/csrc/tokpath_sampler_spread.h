// tokpath_sampler_spread.h -- sampling rows without top-k spread over the
// chip (gfx950): three launches, each over every row's S slices.
//
// Serves small batches of plain or top-p sampling (no top-k) in any dtype,
// alignment and vocabulary, with the repetition penalty and the allow mask of
// the contract in include/graspo_tokpath.h, bit for bit: the reference's
// decode step (src/graspo/backends/graspoflow/tensor_utils.py:649-683) on one
// prompt group.  The kernels that give each row one workgroup leave most of
// the chip idle on such a batch, and their serial tail (weights, cut, draw
// and a second read by one CU) is most of their time.  The steps need the
// row's maximum before the weights and the weights' sum before the cut, so
// the row is read three times, each time by S workgroups at once and, after
// the first, from the caches; a launch boundary between the steps costs about
// 2 us and needs no workgroup to wait for another.
//
// 1. spread_max: per slice the largest allowed x' (m = that / T exactly:
//    division by T is monotone), the raw (m, s) of the log-softmax, and
//    whether the row is one that the contract's status rules catch.
// 2. spread_weights: per slice every token's fixed-point weight
//    DETEXP_FIX(y - m), their sum, and counts and weights in 512 bins of
//    width 1/16 in m - y.  Equal y share a bin, so a bin is an interval of
//    the rank order.
// 3. spread_pick: every workgroup merges its row's bins (48 KB for 8 slices,
//    from the L2), finds the bin of the cut floor(P W) and the bins that can
//    hold the draw floor(u W') (W' lies between the cut bin's edges), and
//    appends its slice's tokens of these bins to the row's two lists; the
//    last slice to arrive cuts each list into 256 parts by y, ranks the one
//    that holds the cut (the draw) by (y desc, id asc) and writes the outputs.
//    (Merging the bins once, in the last workgroup of step 2 to arrive, took
//    8 us there against 2 here.)
// A row outside these bounds (a status, a non-finite or huge m, bins beyond
// the lists' capacity, the cut or the draw below the bins) runs the row-wise
// path in step 3, in one workgroup, so every row gets the contract's answer.
#pragma once

namespace gtp {
namespace spread {

typedef unsigned long long u64;

constexpr int kT = 512;               // threads of steps 1 and 2
constexpr int kW = kT / kWave;
constexpr int kB3 = 1024;             // threads of step 3 (the row-wise path's)
constexpr int kMaxS = 16;             // slices per row
constexpr int kNB = 512;              // bins
constexpr float kScale = 16.0f;       // bins per unit of y
constexpr int kList = 8192;           // tokens of a row's two lists together
constexpr int kSlice = 4096;          // tokens of a list from one slice
constexpr int kSub = 256;             // parts of a list's bins
constexpr int kSel = 2048;            // tokens of the part that is ranked
constexpr int kRows = 4096;           // rows of one pass; more take several
constexpr float kMMax = 32768.0f;     // |m| below this: step 3's pre-test margin
constexpr int kG = 4;                 // groups of 8 tokens per thread and trip

// Per-row words, cleared by step 1: arrivals in step 3, list lengths.
struct RowCtr {
  uint32_t pick, len[2], pad;
};
// Step 1's and step 2's results per slice.
struct MaxPart {
  float mx, m, s;
  uint32_t bad;
};
struct SumPart {
  u64 W, low_key;
  uint32_t valid, pad[3];
};
struct Ws {
  RowCtr* ctr;
  MaxPart* mx;
  SumPart* sum;
  u64* wbin;       // [B][S][kNB]
  uint32_t* cbin;  // [B][S][kNB]
  u64* list;       // [B][cap] rank keys: the cut's list, then the draw's
  int cap;
};

// Tokens of a row's two lists together.
inline int list_cap(int64_t V) { return (int)(2 * V < kList ? 2 * V : kList); }

// The workspace grows with the rows of a pass and not with the call's: at
// most 300 MB (6 KB of bins per slice and up to 64 KB of lists per row), where
// one pass over any batch took 9 GB at 65535 rows whatever V.  Passes of 1024
// rows took 5 to 9% longer at 4096 rows and more (fp16 [4096, 151936] 1748 us
// in one pass, 1913 in four).
__host__ __device__ inline size_t align256(size_t n) { return (n + 255) / 256 * 256; }
inline size_t ws_bytes(int64_t B, int S, int64_t V) {
  const size_t r = (size_t)B, rs = r * (size_t)S;
  return align256(r * sizeof(RowCtr)) + align256(rs * sizeof(MaxPart)) +
         align256(rs * sizeof(SumPart)) + rs * kNB * 12 + align256(r * list_cap(V) * 8);
}
// Rows of a pass: as many passes as needed, of equal size.
inline int64_t pass_rows(int64_t B) {
  const int64_t passes = (B + kRows - 1) / kRows;
  return (B + passes - 1) / passes;
}
inline Ws ws_of(void* p, int64_t B, int S, int64_t V) {
  unsigned char* q = reinterpret_cast<unsigned char*>(p);
  const size_t r = (size_t)B, rs = r * (size_t)S;
  auto take = [&](size_t n) {
    unsigned char* at = q;
    q += align256(n);
    return at;
  };
  Ws w;
  w.ctr = reinterpret_cast<RowCtr*>(take(r * sizeof(RowCtr)));
  w.mx = reinterpret_cast<MaxPart*>(take(rs * sizeof(MaxPart)));
  w.sum = reinterpret_cast<SumPart*>(take(rs * sizeof(SumPart)));
  w.wbin = reinterpret_cast<u64*>(take(rs * kNB * 8));
  w.cbin = reinterpret_cast<uint32_t*>(take(rs * kNB * 4));
  w.cap = list_cap(V);
  w.list = reinterpret_cast<u64*>(take(r * w.cap * 8));
  return w;
}

// ------------------------------------------------------------ token access

// 8 tokens from a row that may start at any element: 16-byte loads at the
// elements' own alignment (gfx950 takes them unaligned; an odd vocabulary's
// rows start anywhere).
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
template <typename T>
struct Raw8;
template <>
struct Raw8<uint16_t> {
  u32x4 v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const u32x4_a2*>(p); }
  __device__ __forceinline__ void get(float (&x)[8]) const { Vec<uint16_t>::cvt(v, x); }
};
template <>
struct Raw8<_Float16> {
  u32x4 v;
  __device__ __forceinline__ void load(const _Float16* p) { v = *reinterpret_cast<const u32x4_a2*>(p); }
  __device__ __forceinline__ void get(float (&x)[8]) const { Vec<_Float16>::cvt(v, x); }
};
template <>
struct Raw8<float> {
  u32x4 v, w;
  __device__ __forceinline__ void load(const float* p) {
    v = *reinterpret_cast<const u32x4_a4*>(p);
    w = *reinterpret_cast<const u32x4_a4*>(p + 4);
  }
  __device__ __forceinline__ void get(float (&x)[8]) const {
    x[0] = u2f(v.x); x[1] = u2f(v.y); x[2] = u2f(v.z); x[3] = u2f(v.w);
    x[4] = u2f(w.x); x[5] = u2f(w.y); x[6] = u2f(w.z); x[7] = u2f(w.w);
  }
};

// Groups [g0, g1) of 8 tokens of slice k (whole mask words: multiples of 4
// groups); the row's last V mod 8 tokens go with the last slice.
struct Range {
  uint32_t g0, g1;
  bool tail;
};
__device__ __forceinline__ Range range_of(int64_t V, int k, int S) {
  const uint32_t ng = (uint32_t)(V / 8);
  const uint32_t per = ((ng + (uint32_t)S - 1) / (uint32_t)S + 3u) / 4u * 4u;
  const uint32_t g0 = min((uint32_t)k * per, ng);
  return {g0, min(g0 + per, ng), k == S - 1};
}

// Calls f(x, first id, allow bits, penalty bits, count) for this thread's
// groups of a slice, count 8, and for the row's last V mod 8 tokens, one at
// a time (count 1).  `pen`: the slice's penalty bits by byte (null: none).
// Without kExtra there is neither mask nor penalty.
template <typename T, int NT, bool kExtra, typename F>
__device__ __forceinline__ void for_groups(const T* __restrict__ row, const uint32_t* __restrict__ mrow,
                                           const uint8_t* pen, int64_t V, const Range& r, F&& f) {
  const uint32_t tid = threadIdx.x;
  for (uint32_t g = r.g0 + tid; g < r.g1; g += NT * kG) {
    Raw8<T> q[kG];
    uint32_t mw[kG];
#pragma unroll
    for (int i = 0; i < kG; ++i) {
      const uint32_t gi = min(g + (uint32_t)i * NT, r.g1 - 1u);
      q[i].load(row + (int64_t)gi * 8);
      mw[i] = kExtra && mrow ? mrow[gi >> 2] >> ((gi & 3u) * 8u) : 0xFFu;
    }
#pragma unroll
    for (int i = 0; i < kG; ++i) {
      const uint32_t gi = g + (uint32_t)i * NT;
      if (gi < r.g1) {
        float x[8];
        q[i].get(x);
        f(x, gi * 8u, mw[i] & 0xFFu, kExtra && pen ? (uint32_t)pen[gi - r.g0] : 0u, 8);
      }
    }
  }
  const uint32_t id = (uint32_t)(V / 8) * 8u + tid;
  if (r.tail && id < (uint32_t)V) {
    float x[8];
    x[0] = Elem<T>::get(row, id);
    const uint32_t al = kExtra && mrow ? (mrow[id >> 5] >> (id & 31u)) & 1u : 1u;
    const uint32_t pb = kExtra && pen ? ((uint32_t)pen[(id >> 3) - r.g0] >> (id & 7u)) & 1u : 0u;
    f(x, id, al, pb, 1);
  }
}

// The slice's penalty bitmap (bit id - 8 g0) from the row's history; true
// when an id lies beyond the vocabulary.  Call with every thread; syncs.
__device__ __forceinline__ bool slice_pen(const SamplerArgs& a, int64_t b, const Range& r, bool use,
                                          uint32_t* bits, int nt) {
  const int32_t* h = a.hist + b * a.hist_stride;
  const uint32_t id0 = r.g0 * 8u, id1 = r.tail ? (uint32_t)a.V : r.g1 * 8u;
  for (uint32_t i = threadIdx.x; use && i < (id1 - id0 + 31u) / 32u; i += (uint32_t)nt) bits[i] = 0u;
  __syncthreads();
  bool bad = false;
  for (int64_t j = threadIdx.x; j < a.hist_len; j += nt) {
    const int32_t id = h[j];
    bad |= id >= a.V;
    if (use && id >= 0 && (uint32_t)id >= id0 && (uint32_t)id < id1)
      atomicOr(&bits[((uint32_t)id - id0) >> 5], 1u << (((uint32_t)id - id0) & 31u));
  }
  return __syncthreads_or(bad ? 1 : 0) != 0;
}

__device__ __forceinline__ float penalise(float x, bool pen, float rho) {
  if (pen) return x < 0.0f ? x * rho : x / rho;
  return x;
}

// Publishing to the row's other workgroups and counting one's arrival.  No
// release operation: gfx950's agent-scope stores write through to where the
// other XCDs' agent-scope loads see them, each wave waits for its own
// (vmcnt(0)) and the barrier joins the waves (a release fence would write
// the whole L2 back).  True in every thread of the last workgroup.
template <typename U>
__device__ __forceinline__ void put(U* p, U v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ __forceinline__ U take(const U* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool arrive_last(uint32_t* ctr, int S) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int last = 0;
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           (uint32_t)S - 1u;
  return __syncthreads_or(last) != 0;
}

// ------------------------------------------------------------- step 1

template <typename T, bool kExtra>
__global__ __launch_bounds__(kT) void spread_max_kernel(SamplerArgs a, Ws ws, int S) {
  __shared__ uint32_t pen_bits[GTP_SAMPLER_MAX_V / 32];
  __shared__ float red[kW][3];
  const int k = blockIdx.x;
  const int64_t b = blockIdx.y;
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const T* row = reinterpret_cast<const T*>(a.logits) + b * a.row_stride;
  const uint32_t* mrow = a.mask ? a.mask + b * a.mask_stride : nullptr;
  const Range r = range_of(a.V, k, S);
  const bool use_pen = kExtra && a.hist_len > 0 && a.rho != 1.0f;
  bool bad = false;
  if (a.hist_len > 0) bad = slice_pen(a, b, r, use_pen, pen_bits, kT);
  if (k == 0 && threadIdx.x < 4) reinterpret_cast<uint32_t*>(ws.ctr + b)[threadIdx.x] = 0u;
  float mx = kNegInf;
  Lse3 st{kNegInf, 0.0f, 0.0f};
  for_groups<T, kT, kExtra>(row, mrow, use_pen ? reinterpret_cast<const uint8_t*>(pen_bits) : nullptr, a.V,
                    r, [&](const float(&x)[8], uint32_t, uint32_t al, uint32_t pb, int n) {
                      if (n == 8) {
                        float z[1][8];
#pragma unroll
                        for (int j = 0; j < 8; ++j) z[0][j] = x[j];
                        lse_fold_block_max<false, 1, 8>(st, z, vec_max<8>(x));
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                          const float xp = kExtra ? penalise(x[j], (pb >> j) & 1u, a.rho) : x[j];
                          mx = !kExtra || ((al >> j) & 1u) ? fmaxf(mx, xp) : mx;
                        }
                      } else {
                        const float z[1][4] = {{x[0], kNegInf, kNegInf, kNegInf}};
                        lse_fold_block_max<false, 1, 4>(st, z, x[0]);
                        if (al) mx = fmaxf(mx, penalise(x[0], pb, a.rho));
                      }
                    });
  mx = wave_max_f(mx);
  wave_lse2(st.m, st.s);
  if (lane == 0) {
    red[wid][0] = mx;
    red[wid][1] = st.m;
    red[wid][2] = st.s;
  }
  __syncthreads();
  if (wid != 0) return;
  mx = wave_max_f(lane < kW ? red[lane][0] : kNegInf);
  float m = lane < kW ? red[lane][1] : kNegInf, s = lane < kW ? red[lane][2] : 0.0f;
  wave_lse2(m, s);
  // a NaN or +inf logit leaves s NaN
  if (lane == 0) ws.mx[b * S + k] = MaxPart{mx, m, s, (bad || s != s) ? 1u : 0u};
}

// Step 1's results of a row, merged by every wave; false for a row that the
// row-wise path takes (the same in every workgroup).
struct RowMax {
  float m, lse_m, lse_s;
};
__device__ __forceinline__ bool row_max(const SamplerArgs& a, const Ws& ws, int64_t b, int S,
                                        RowMax& r) {
  const int lane = threadIdx.x & (kWave - 1);
  MaxPart p{kNegInf, kNegInf, 0.0f, 0u};
  if (lane < S) p = ws.mx[b * S + lane];
  const float mx = wave_max_f(p.mx);
  wave_lse2(p.m, p.s);
  const float Tc = a.T > 1e-6f ? a.T : 1e-6f;
  const float u = a.uniforms[b];
  r = RowMax{mx / Tc + 0.0f, p.m, p.s};
  return __ballot(p.bad != 0u) == 0ull && fabsf(r.m) < kMMax && u >= 0.0f && u < 1.0f;
}

// ------------------------------------------------------------- step 2

struct Smem2 {
  uint32_t pen_bits[GTP_SAMPLER_MAX_V / 32];
  u64 w[kNB];
  uint32_t c[kNB];
  u64 red_w[kW], red_k[kW];
  uint32_t red_c[kW];
};

template <typename T, bool kExtra>
__global__ __launch_bounds__(kT) void spread_weights_kernel(SamplerArgs a, Ws ws, int S) {
  __shared__ Smem2 sm;
  const int k = blockIdx.x;
  const int64_t b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
  RowMax rm;
  if (!row_max(a, ws, b, S, rm)) return;
  const float m = rm.m;
  const float Tc = a.T > 1e-6f ? a.T : 1e-6f;
  const T* row = reinterpret_cast<const T*>(a.logits) + b * a.row_stride;
  const uint32_t* mrow = a.mask ? a.mask + b * a.mask_stride : nullptr;
  const Range r = range_of(a.V, k, S);
  const bool use_pen = kExtra && a.hist_len > 0 && a.rho != 1.0f;
  for (int i = tid; i < kNB; i += kT) {
    sm.w[i] = 0ull;
    sm.c[i] = 0u;
  }
  if (use_pen) slice_pen(a, b, r, true, sm.pen_bits, kT);
  __syncthreads();
  const bool top_p = a.P > 0.0f && a.P < 1.0f;
  const float rT = 1.0f / Tc, bh = div_by_t_bound(Tc);
  u64 wsum = 0ull;
  uint32_t valid = 0u;
  float ylow = kPosInf;
  uint32_t idlow = 0u;
  auto tok = [&](float x, uint32_t id, bool al, bool pn) __attribute__((always_inline)) {
    const float y = div_by_t(kExtra ? penalise(x, pn, a.rho) : x, Tc, rT, bh) + 0.0f;
    const bool in = (!kExtra || al) && y > kNegInf;
    const float q = (m - y) * kScale;
    if (!top_p && in && y <= ylow) {  // ascending ids: the last of equals
      ylow = y;
      idlow = id;
    }
    valid += in ? 1u : 0u;
    if (in && q < (float)kNB) {  // (below the bins every weight is zero)
      const u64 w = detexp_fix(y - m);
      wsum += w;
      atomicAdd(&sm.c[(int)q], 1u);
      atomicAdd(&sm.w[(int)q], w);
    }
  };
  for_groups<T, kT, kExtra>(row, mrow, use_pen ? reinterpret_cast<const uint8_t*>(sm.pen_bits) : nullptr,
                    a.V, r, [&](const float(&x)[8], uint32_t id, uint32_t al, uint32_t pb, int n) {
                      if (n == 8) {
#pragma unroll
                        for (int j = 0; j < 8; ++j) tok(x[j], id + j, (al >> j) & 1u, (pb >> j) & 1u);
                      } else {
                        tok(x[0], id, al, pb);
                      }
                    });
  {
    const u64 sw = lane63_u64(wave_scan_u64(wsum));
    const uint32_t sc = wave_total_u32(valid);
    // the smallest key: the smallest y, of equals the largest id
    const u64 key = wave_max_u64(valid && !top_p ? ~rank_key(ylow, (int32_t)idlow) : 0ull);
    if (lane == 0) {
      sm.red_w[wid] = sw;
      sm.red_c[wid] = sc;
      sm.red_k[wid] = key;
    }
  }
  __syncthreads();
  const int64_t sl = b * S + k;
  for (int i = tid; i < kNB; i += kT) {
    ws.wbin[sl * kNB + i] = sm.w[i];
    ws.cbin[sl * kNB + i] = sm.c[i];
  }
  if (tid != 0) return;
  SumPart p{};
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    p.W += sm.red_w[i];
    p.valid += sm.red_c[i];
    p.low_key = sm.red_k[i] > p.low_key ? sm.red_k[i] : p.low_key;
  }
  ws.sum[sl] = p;
}

// ------------------------------------------------------------- step 3

struct Smem3 {
  uint32_t pen_bits[GTP_SAMPLER_MAX_V / 32];
  union {
    u64 slice[2][kSlice];  // the slice's tokens of each list, as rank keys
    u64 key[kList];        // then, in the last workgroup, both lists
  };
  u64 sel_w[kSel];         // the ranked part's weights
  uint16_t sel[kSel];      // ... and places in the list
  union {
    struct {
      u64 pre_w[kNB + 1];  // weight and tokens before each bin
      uint32_t pre_c[kNB + 1];
    };
    struct {
      u64 sub_w[kSub];
      uint32_t sub_c[kSub];
    };
  };
  u64 red_w[kNB / kWave];
  uint32_t red_c[kNB / kWave];
  int32_t bin[3];          // the cut's bin, the draw's first and last
  uint32_t n[2], at[2];
  uint32_t part, part_before, sel_n;
  u64 part_base;
  // the token found in a list: rank, weight before it, weight, key
  uint32_t found_r;
  u64 found_s, found_w, found_key;
};

// What the merged bins say of a row: its total weight and, per list (0: the
// cut, 1: the draw), its bins [lo, hi] (lo > hi: none), the tokens in them
// and the weight and tokens before them.
struct Plan {
  u64 W, low_key, base[2];
  uint32_t valid, before[2], n[2];
  int lo[2], hi[2];
};

// False (in every thread) when the row must run the row-wise path.
__device__ __forceinline__ bool plan_row(const SamplerArgs& a, const Ws& ws, int64_t b, int S,
                                         Smem3& sm, Plan& p) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
  // the first 8 waves merge the bins, one per thread (every instruction of
  // all 16 waves would be paid for)
  const int v = tid;
  const bool mine = tid < kNB;
  u64 w = 0ull, iw = 0ull;
  uint32_t c = 0u, ic = 0u;
  SumPart part{};
  if (lane < S) part = ws.sum[b * S + lane];
  if (mine) {
#pragma unroll
    for (int j = 0; j < kMaxS; ++j) {
      const int64_t at = (b * S + min(j, S - 1)) * kNB + v;
      const u64 wj = ws.wbin[at];
      const uint32_t cj = ws.cbin[at];
      w += j < S ? wj : 0ull;
      c += j < S ? cj : 0u;
    }
    iw = wave_scan_u64(w);
    ic = wave_scan_u32(c);
    if (lane == kWave - 1) {
      sm.red_w[wid] = iw;
      sm.red_c[wid] = ic;
    }
    if (tid < 3) sm.bin[tid] = -1;
  }
  p.W = lane63_u64(wave_scan_u64(part.W));
  p.valid = wave_total_u32(part.valid);
  p.low_key = ~wave_max_u64(part.low_key);
  __syncthreads();
  u64 end = iw, in_bins = 0ull;
  uint32_t ec = ic;
#pragma unroll
  for (int i = 0; i < kNB / kWave; ++i) {
    if (i < wid) {
      end += sm.red_w[i];
      ec += sm.red_c[i];
    }
    in_bins += sm.red_w[i];
  }
  if (mine) {
    sm.pre_w[v] = end - w;
    sm.pre_c[v] = ec - c;
    if (v == kNB - 1) {
      sm.pre_w[kNB] = end;
      sm.pre_c[kNB] = ec;
    }
  }
  const bool top_p = a.P > 0.0f && a.P < 1.0f;
  const u64 X = top_p ? floor_mul(a.P, p.W) : 0ull;
  if (X >= in_bins) return false;
  // the bin whose weight interval holds X: one bin at most
  if (mine && top_p && end - w <= X && X < end) sm.bin[0] = v;
  __syncthreads();
  p.lo[0] = p.hi[0] = sm.bin[0];
  u64 wlo = p.W, whi = p.W;  // bounds of the kept weight W'
  if (top_p) {
    wlo = X + 1ull;  // the last kept token's interval holds X
    const u64 e = sm.pre_w[sm.bin[0] + 1];
    whi = ((u64)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(e >> 32)) << 32) |
          (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)e);
  } else {
    p.lo[0] = 0;
  }
  const float u = a.uniforms[b];
  const u64 ulo = floor_mul(u, wlo), uhi = floor_mul(u, whi);
  if (uhi >= in_bins) return false;
  if (mine && end - w <= ulo && ulo < end) sm.bin[1] = v;
  if (mine && end - w <= uhi && uhi < end) sm.bin[2] = v;
  __syncthreads();
  p.lo[1] = sm.bin[1];
  p.hi[1] = sm.bin[2];
#pragma unroll
  for (int l = 0; l < 2; ++l) {
    const bool some = p.lo[l] <= p.hi[l];
    p.base[l] = some ? sm.pre_w[p.lo[l]] : 0ull;
    p.before[l] = some ? sm.pre_c[p.lo[l]] : 0u;
    p.n[l] = some ? sm.pre_c[p.hi[l] + 1] - p.before[l] : 0u;
  }
  return p.n[0] + p.n[1] <= (uint32_t)ws.cap;
}

// The token of the list at sm.key[at0] (n tokens of bins [lo, hi], `base`
// weight and `before` tokens ahead of them) whose weight interval holds X;
// false (in every thread) when there is none, or too many share its part.  The list is cut into kSub parts of equal width
// in y (equal y share a part), their exact weights name the part, and its
// few tokens are ranked by comparing all pairs, 2^q threads to a token.
__device__ __forceinline__ bool resolve(Smem3& sm, int at0, int n, int lo, int hi, float m,
                                        u64 base, uint32_t before, u64 X) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const u64* key = sm.key + at0;
  if (tid < kSub) {
    sm.sub_w[tid] = 0ull;
    sm.sub_c[tid] = 0u;
  }
  if (tid == 0) {
    sm.found_w = 0ull;
    sm.part = kSub;
    sm.sel_n = 0u;
  }
  __syncthreads();
  const float per = (float)kSub / (float)(hi - lo + 1);
  auto part_of = [&](float y) {
    const float f = ((m - y) * kScale - (float)lo) * per;  // every step monotone in y
    return (int)fminf(fmaxf(f, 0.0f), (float)(kSub - 1));
  };
  for (int i = tid; i < n; i += kB3) {
    const float y = rank_key_y(key[i]);
    const int q = part_of(y);
    atomicAdd(&sm.sub_w[q], (u64)detexp_fix(y - m));
    atomicAdd(&sm.sub_c[q], 1u);
  }
  __syncthreads();
  if (tid < kWave) {
    u64 w[kSub / kWave], sum = 0ull;
    uint32_t c[kSub / kWave], cs = 0u;
#pragma unroll
    for (int q = 0; q < kSub / kWave; ++q) {
      w[q] = sm.sub_w[lane * (kSub / kWave) + q];
      c[q] = sm.sub_c[lane * (kSub / kWave) + q];
      sum += w[q];
      cs += c[q];
    }
    u64 at = base + wave_scan_u64(sum) - sum;
    uint32_t ahead = before + wave_scan_u32(cs) - cs;
#pragma unroll
    for (int q = 0; q < kSub / kWave; ++q) {
      if (at <= X && X < at + w[q]) {
        sm.part = (uint32_t)(lane * (kSub / kWave) + q);
        sm.part_base = at;
        sm.part_before = ahead;
      }
      at += w[q];
      ahead += c[q];
    }
  }
  __syncthreads();
  const uint32_t part = sm.part;
  for (int i = tid; i < n; i += kB3) {
    const float y = rank_key_y(key[i]);
    if ((uint32_t)part_of(y) == part) {
      const uint32_t at = atomicAdd(&sm.sel_n, 1u);
      if (at < (uint32_t)kSel) {
        sm.sel[at] = (uint16_t)i;
        sm.sel_w[at] = detexp_fix(y - m);
      }
    }
  }
  __syncthreads();
  const int ns = (int)sm.sel_n;
  if (ns > kSel) return false;
  const u64 pbase = sm.part_base;
  const int parts = ns <= kB3 / 8 ? 8 : ns <= kB3 / 4 ? 4 : ns <= kB3 / 2 ? 2 : 1;
  const int mine = tid & (parts - 1);
  for (int i0 = 0; i0 < ns; i0 += kB3 / parts) {
    const int i = i0 + tid / parts;
    const bool in = i < ns;
    const u64 ki = in ? key[sm.sel[i]] : ~0ull;
    u64 s = 0ull;
    uint32_t r = 0u;
    for (int j = mine; in && j < ns; j += parts) {
      const bool ahead = key[sm.sel[j]] > ki;
      s += ahead ? sm.sel_w[j] : 0ull;
      r += ahead ? 1u : 0u;
    }
    for (int o = 1; o < parts; o <<= 1) {
      s += shfl_xor_u64(s, o);
      r += (uint32_t)__shfl_xor((int)r, o, kWave);
    }
    if (in && mine == 0 && pbase + s <= X && X < pbase + s + sm.sel_w[i]) {
      sm.found_r = sm.part_before + r;
      sm.found_s = pbase + s;
      sm.found_w = sm.sel_w[i];
      sm.found_key = ki;
    }
  }
  __syncthreads();
  return sm.found_w != 0ull;
}

// False (in every thread) when this workgroup must run the row-wise path for
// the row.
template <typename T>
__device__ __forceinline__ bool pick_row(const SamplerArgs& a, const Ws& ws, int64_t b, int k,
                                         int S, int S12, Smem3& sm) {
  const int tid = threadIdx.x;
  RowMax rm;
  Plan p;
  // a row handed over: its first workgroup takes it
  if (!row_max(a, ws, b, S12, rm) || !plan_row(a, ws, b, S12, sm, p)) return k != 0;
  const float m = rm.m;
  const T* row = reinterpret_cast<const T*>(a.logits) + b * a.row_stride;
  const uint32_t* mrow = a.mask ? a.mask + b * a.mask_stride : nullptr;
  const Range r = range_of(a.V, k, S);
  const bool use_pen = a.hist_len > 0 && a.rho != 1.0f;
  if (tid < 2) sm.n[tid] = 0u;
  if (use_pen) slice_pen(a, b, r, true, sm.pen_bits, kB3);
  __syncthreads();
  const float Tc = a.T > 1e-6f ? a.T : 1e-6f;
  const float rT = 1.0f / Tc;
  // a token of bin v has (m - x' rT) kScale within e of [v, v + 1]
  const float e = kScale * 4e-7f * (fabsf(m) + 33.0f) + 1e-3f;
  const float lo0 = (float)p.lo[0] - e, hi0 = (float)(p.hi[0] + 1) + e;
  const float lo1 = (float)p.lo[1] - e, hi1 = (float)(p.hi[1] + 1) + e;
  const bool cut = p.hi[0] >= p.lo[0];
  auto tok = [&](float x, uint32_t id, bool al, bool pn) __attribute__((always_inline)) {
    const float xp = penalise(x, pn, a.rho);
    const float q = (m - xp * rT) * kScale;
    if (al && ((cut && q >= lo0 && q <= hi0) || (q >= lo1 && q <= hi1))) {
      const float y = xp / Tc + 0.0f;
      const int v = (int)fminf((m - y) * kScale, (float)kNB);
#pragma unroll
      for (int l = 0; l < 2; ++l)
        if (v >= p.lo[l] && v <= p.hi[l]) {
          const uint32_t at = atomicAdd(&sm.n[l], 1u);
          if (at < (uint32_t)kSlice) sm.slice[l][at] = rank_key(y, (int32_t)id);
        }
    }
  };
  for_groups<T, kB3, true>(row, mrow, use_pen ? reinterpret_cast<const uint8_t*>(sm.pen_bits) : nullptr,
                     a.V, r, [&](const float(&x)[8], uint32_t id, uint32_t al, uint32_t pb, int n) {
                       if (n == 8) {
#pragma unroll
                         for (int j = 0; j < 8; ++j)
                           tok(x[j], id + j, (al >> j) & 1u, (pb >> j) & 1u);
                       } else {
                         tok(x[0], id, al, pb);
                       }
                     });
  __syncthreads();
  // append the slice's tokens to the row's lists; a slice with more than it
  // can hold leaves a length that no plan has
  if (tid < 2) {
    const uint32_t n = sm.n[tid];
    sm.at[tid] = n ? __hip_atomic_fetch_add(&ws.ctr[b].len[tid], n > (uint32_t)kSlice ? 1u << 30 : n,
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                   : 0u;
  }
  __syncthreads();
  u64* list = ws.list + b * ws.cap;
#pragma unroll
  for (int l = 0; l < 2; ++l)
    for (uint32_t i = tid; i < min(sm.n[l], (uint32_t)kSlice) && sm.at[l] + i < p.n[l]; i += kB3)
      put(list + (l ? p.n[0] : 0u) + sm.at[l] + i, sm.slice[l][i]);
  if (!arrive_last(&ws.ctr[b].pick, S)) return true;
  bool whole = true;
#pragma unroll
  for (int l = 0; l < 2; ++l) whole = whole && take(&ws.ctr[b].len[l]) == p.n[l];
  if (!whole) return false;
  for (uint32_t i = tid; i < p.n[0] + p.n[1]; i += kB3) sm.key[i] = take(list + i);
  __syncthreads();
  // the cut, then the draw
  u64 Wk = p.W;
  uint32_t kept = p.valid;
  u64 last = p.low_key;
  if (cut) {
    if (!resolve(sm, 0, (int)p.n[0], p.lo[0], p.hi[0], m, p.base[0], p.before[0],
                 floor_mul(a.P, p.W)))
      return false;
    Wk = sm.found_s + sm.found_w;
    kept = sm.found_r + 1u;
    last = sm.found_key;
    __syncthreads();
  }
  if (!resolve(sm, (int)p.n[0], (int)p.n[1], p.lo[1], p.hi[1], m, p.base[1], p.before[1],
               floor_mul(a.uniforms[b], Wk)))
    return false;
  if (tid == 0) {
    const int32_t id = rank_key_id(sm.found_key);
    const float slp = __builtin_amdgcn_logf((float)((double)sm.found_w / (double)Wk)) * kLn2;
    const float lse_ln = __builtin_amdgcn_logf(rm.lse_s) * kLn2;
    write_row_f(a, b, a.finished && a.finished[b], GTP_ROW_OK, id,
                raw_logprob(Elem<T>::get(row, id), rm.lse_m, lse_ln), slp, (int32_t)kept,
                rank_key_y(last), rank_key_id(last));
  }
  return true;
}

template <typename T>
__global__ __launch_bounds__(kB3) void spread_pick_kernel(SamplerArgs a, Ws ws, int S, int S12) {
  __shared__ union {
    Smem3 t;
    SamplerSmem g;
  } smu;
  const int64_t b = blockIdx.y;
  if (!pick_row<T>(a, ws, b, blockIdx.x, S, S12, smu.t)) {
    __syncthreads();
    rowwise_row<T>(a, b, smu.g);
  }
}

// Slices per row of steps 1 and 2: two workgroups of 512 threads per CU.
inline int slices(int64_t B) {
  const int64_t want = (2 * device_cus() + B - 1) / B;
  return (int)(want < 1 ? 1 : want > kMaxS ? kMaxS : want);
}
// ... and of step 3: one of 1024 per CU (the row-wise path's LDS), no more
// workgroups than CUs.
inline int pick_slices(int64_t B) {
  const int64_t want = device_cus() / B;
  return (int)(want < 1 ? 1 : want > kMaxS ? kMaxS : want);
}

// The call's rows from b0 on.
template <typename T>
SamplerArgs rows_from(SamplerArgs a, int64_t b0) {
  a.logits = reinterpret_cast<const T*>(a.logits) + b0 * a.row_stride;
  if (a.hist) a.hist += b0 * a.hist_stride;
  if (a.mask) a.mask += b0 * a.mask_stride;
  a.uniforms += b0;
  if (a.finished) a.finished += b0;
  a.out_ids += b0;
  if (a.out_lp) a.out_lp += b0;
  if (a.out_slp) a.out_slp += b0;
  if (a.out_kept) a.out_kept += b0;
  if (a.out_tv) a.out_tv += b0;
  if (a.out_tid) a.out_tid += b0;
  if (a.out_status) a.out_status += b0;
  return a;
}

// Passes of pass_rows(B) rows over one workspace, each three launches.  They
// follow one another on the stream, and each clears its own counters.
template <typename T, bool kExtra>
int launch_as(const SamplerArgs& call, int64_t B, void* workspace, hipStream_t s) {
  const int64_t R = pass_rows(B);
  const int S = slices(R), S3 = pick_slices(R);
  const Ws ws = ws_of(workspace, R, S, call.V);
  // the timing hook spans all launches
  const LaunchEvents e = g_next_launch_events;
  const bool timed = e.start && e.stop;
  g_next_launch_events = LaunchEvents{nullptr, nullptr};
  for (int64_t b0 = 0; b0 < B; b0 += R) {
    const SamplerArgs a = rows_from<T>(call, b0);
    const unsigned rows = (unsigned)(B - b0 < R ? B - b0 : R);
    const dim3 grid((unsigned)S, rows), grid3((unsigned)S3, rows);
    if (timed && b0 == 0)
      hipExtLaunchKernelGGL((spread_max_kernel<T, kExtra>), grid, dim3(kT), 0, s, e.start, nullptr, 0, a, ws, S);
    else
      hipLaunchKernelGGL((spread_max_kernel<T, kExtra>), grid, dim3(kT), 0, s, a, ws, S);
    hipLaunchKernelGGL((spread_weights_kernel<T, kExtra>), grid, dim3(kT), 0, s, a, ws, S);
    if (timed && b0 + R >= B)
      hipExtLaunchKernelGGL(spread_pick_kernel<T>, grid3, dim3(kB3), 0, s, nullptr, e.stop, 0, a, ws, S3, S);
    else
      hipLaunchKernelGGL(spread_pick_kernel<T>, grid3, dim3(kB3), 0, s, a, ws, S3, S);
  }
  return hipGetLastError() == hipSuccess ? GTP_OK : GTP_ERR_LAUNCH;
}

template <typename T>
int launch(const SamplerArgs& a, int64_t B, void* workspace, hipStream_t s) {
  const bool pen = a.hist_len > 0 && a.rho != 1.0f;
  return a.mask || pen ? launch_as<T, true>(a, B, workspace, s)
                       : launch_as<T, false>(a, B, workspace, s);
}

}  // namespace spread
}  // namespace gtp
