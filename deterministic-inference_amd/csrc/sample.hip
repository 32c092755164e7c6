// Greedy token selection: per-row argmax over the fp32 logits with torch's
// semantics (first index among equal maxima; NaN counts as the maximum, the
// first NaN wins). The (value, index) order used below is total, so the
// result does not depend on the reduction tree.
#include "common.h"

#include <algorithm>

namespace sid {
namespace {

__device__ __forceinline__ bool better(float v, int64_t i, float bv, int64_t bi) {
  const bool vn = v != v;
  const bool bn = bv != bv;
  if (vn || bn) {
    if (vn && bn) return i < bi;
    return vn;
  }
  return v > bv || (v == bv && i < bi);
}

// ---- stochastic sampling (temperature / top-k / top-p / seeded Gumbel-max) ---------------
//
// The reference's sample() (sid/engine/sampler.py:32-69) with its truncation made exact:
//   temperature <= 0: the greedy argmax (first index, NaN wins), as argmax_kernel.
//   otherwise p = softmax(logits / T) (max, then the sum of exp(x - max) in a fixed order,
//   p = exp(x - max) / sum); tokens are ranked by (p descending, index ascending); rank r is
//   kept iff r < top_k (top_k <= 0: no limit) and the probability mass of the ranks before
//   it is <= top_p (top_p >= 1: no limit); rank 0 is always kept. The draw is
//   argmax over kept tokens of log(p + 1e-10) + gumbel(seed, position, token), with the
//   reference's int64 hash (sid/engine/sampler.py:22-29) and first-index ties.
// The mass before a rank is accumulated in 64-bit fixed point (units of 2^-48, each p
// rounded down), so it is an exact integer sum: the cut does not depend on any summation
// order. (The reference sums a float cumsum in sorted order; the two differ only when the
// mass lands within rounding of top_p.) The cut is found without sorting: p >= 0, so the
// bits of p order like p, and a 4-level 8-bit radix select over those bits, with LDS
// histograms of (count, fixed-point mass), descends to the key of the last kept rank; the
// tie position among equal keys follows from the index order.
//
// Two forms with the same bits. Few long rows take four launches: the first three spread a row
// over kParts workgroups, one per wave of the 1024-thread column layout for_each_col defines:
// sample_max_kernel takes the maximum, sample_sum_kernel the sum of exp(x - max) (each of the
// 1024 layout threads' chains in its own order, so the bits are those of one 1024-thread
// workgroup) with the number and mass of the columns above a few thresholds,
// sample_list_kernel lists the columns above the first threshold that should hold the cut, or
// draws part by part from a row without limits. sample_select_kernel<false>, one workgroup
// per row, finds the cut and draws over the list in LDS: tens to thousands of keys instead of
// the vocabulary. Rows whose cut is not provably among kListCap columns (flat distributions,
// non-finite sums) take the passes over all columns there. Top-k / top-p mixes over peaked
// rows of 151936 columns: 1 row 31 us, 64 rows 69 (max 6 / 11, sum 12 / 30, list 6 / 12, select
// 9 / 20); nine passes over all columns by one workgroup per row took 205 and 366. Listing in
// the sum pass at fixed thresholds (three launches): 27 and 173, as rows with top-k alone
// reach far below the maximum.
//
// Many rows, or short ones, take sample_select_kernel<true> alone, a workgroup per row for
// everything: the chip is full without the parts, and greedy and unlimited rows don't pay for
// launches and early exits they don't need. See one_workgroup_per_row for both sides' times.
constexpr int kSampleThreads = 1024;
constexpr int kSampleWaves = kSampleThreads / 64;
constexpr double kMassUnit = 281474976710656.0;  // 2^48
constexpr int kHistCopies = 16;

// floor(p * 2^48) for the bits of a p in [0, 1] (0 for a NaN): its 24-bit significand shifted.
__device__ __forceinline__ uint64_t mass_of(uint32_t key) {
  const int e = static_cast<int>(key >> 23);
  const uint64_t m = e == 0 ? key & 0x7fffffu : (key & 0x7fffffu) | 0x800000u;
  const int sh = (e == 0 ? 1 : e) - 102;  // p = m 2^(e - 150)
  if (e >= 255) return 0;
  return sh >= 0 ? m << min(sh, 39) : sh > -64 ? m >> -sh : 0;
}

// Calls f(value, column) for every column of a row: 16-byte loads, UNROLL of them in flight
// per thread, when the row is 16-byte aligned (else one element per load). Which thread sees
// which column is fixed by the row's alignment and length alone.
template <int UNROLL, typename F>
__device__ __forceinline__ void for_each_col(const float* __restrict__ row, int cols, F&& f) {
  const int tid = threadIdx.x;
  int vec = 0;
  if ((reinterpret_cast<uintptr_t>(row) & 15) == 0) {
    const float4* row4 = reinterpret_cast<const float4*>(row);
    const int n4 = cols >> 2;
    constexpr int kStep = kSampleThreads * UNROLL;
    int base = 0;
    for (; base + kStep <= n4; base += kStep) {
      float4 v[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) v[u] = row4[base + u * kSampleThreads + tid];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int c = 4 * (base + u * kSampleThreads + tid);
        f(v[u].x, c);
        f(v[u].y, c + 1);
        f(v[u].z, c + 2);
        f(v[u].w, c + 3);
      }
    }
    // The rest (fewer than kStep vectors) in one more pass with every load issued first; a
    // thread visits the same columns in the same order as a loop over them would.
    if (base < n4) {
      float4 v[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int i = base + u * kSampleThreads + tid;
        if (i < n4) v[u] = row4[i];
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int i = base + u * kSampleThreads + tid;
        if (i < n4) {
          f(v[u].x, 4 * i);
          f(v[u].y, 4 * i + 1);
          f(v[u].z, 4 * i + 2);
          f(v[u].w, 4 * i + 3);
        }
      }
    }
    vec = 4 * n4;
  }
  for (uint32_t c = vec + tid; c < static_cast<uint32_t>(cols); c += kSampleThreads)
    f(row[c], static_cast<int>(c));
}

// Best (value, index) of the block under better(); every thread gets the result.
__device__ __forceinline__ void block_best(float& bv, int64_t& bi, float* s_v, int64_t* s_i) {
  for (int mask = 1; mask < 64; mask <<= 1) {
    const float ov = lane_xor(bv, mask);
    const int lo = __builtin_amdgcn_ds_bpermute((__lane_id() ^ mask) << 2, static_cast<int>(bi));
    const int hi = __builtin_amdgcn_ds_bpermute((__lane_id() ^ mask) << 2, static_cast<int>(bi >> 32));
    const int64_t oi = (static_cast<int64_t>(hi) << 32) | static_cast<uint32_t>(lo);
    if (better(ov, oi, bv, bi)) {
      bv = ov;
      bi = oi;
    }
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    s_v[threadIdx.x >> 6] = bv;
    s_i[threadIdx.x >> 6] = bi;
  }
  __syncthreads();
  bv = s_v[0];
  bi = s_i[0];
  for (int w = 1; w < kSampleWaves; ++w) {
    if (better(s_v[w], s_i[w], bv, bi)) {
      bv = s_v[w];
      bi = s_i[w];
    }
  }
}

// Every thread's x folded by f: over each wave's lanes, then over the waves in order; every
// thread gets the result.
template <typename F>
__device__ __forceinline__ float block_fold(float x, float* s_v, F&& f) {
  for (int mask = 1; mask < 64; mask <<= 1) x = f(x, lane_xor(x, mask));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_v[threadIdx.x >> 6] = x;
  __syncthreads();
  x = s_v[0];
  for (int w = 1; w < kSampleWaves; ++w) x = f(x, s_v[w]);
  return x;
}

// Greedy argmax of one row per workgroup.
__global__ void __launch_bounds__(kSampleThreads) argmax_kernel(const float* __restrict__ logits,
                                                                int64_t ld, int64_t* __restrict__ out,
                                                                int64_t cols) {
  __shared__ float s_bv[kSampleWaves];
  __shared__ int64_t s_bi[kSampleWaves];
  const float* row = logits + static_cast<int64_t>(blockIdx.x) * ld;
  float bv = -INFINITY;
  int64_t bi = cols;  // sentinel larger than any index
  for_each_col<8>(row, static_cast<int>(cols), [&](float v, int c) {
    if (better(v, c, bv, bi)) {
      bv = v;
      bi = c;
    }
  });
  block_best(bv, bi, s_bv, s_bi);
  if (threadIdx.x == 0) out[blockIdx.x] = bi < cols ? bi : 0;
}

// ---- a row over kParts workgroups ----------------------------------------------------------

constexpr int kParts = kSampleWaves;   // one workgroup per wave of for_each_col's layout
constexpr int kPartThreads = 256;
constexpr int kPartSteps = 40;         // layout steps staged in LDS at a time
// Thresholds of e = exp(x - max): the sum pass counts the row's columns and their mass at or
// above each, the list pass lists the columns above the first one that should hold the cut.
constexpr int kCuts = 6;
__device__ constexpr float kCutMin[kCuts] = {0x1p-6f, 0x1p-9f, 0x1p-12f, 0x1p-15f, 0x1p-18f, 0x1p-21f};
constexpr int kListCap = 16384;  // listed columns handled in LDS

// Per (row, part) results of the first three launches.
struct PartStats {
  float* best;       // maximum logit (greedy rows: under better(), with its column)
  int32_t* best_at;
  float* sum;
  int32_t* count;    // [kCuts][row, part]: columns with e >= kCutMin[j]
  float* mass;       // [kCuts][row, part]: their sum of e (a guide: any rounding)
  int64_t stride;    // between thresholds
  int32_t* cut_at;   // the row's threshold of the list (part 0; kCuts: no list)
};
constexpr int kPartWords = 4 + 2 * kCuts;

// Where part q's columns are: layout thread vt = 64 q + lane visits element vectors vt, vt +
// 1024, ... below `vecs` (16-byte vectors when the row is aligned, else single columns), then
// column 4 vecs + vt of an aligned row's remainder.
struct PartCols {
  bool vec;
  uint32_t vecs; // vectors (or columns) in the strided part
  int steps;     // steps that any lane of the part takes
  int list0;     // first entry of the part's list in the row's buffer
  int first;     // the part's first vector
  // The lane's vector of a step (past 2^31 where the last step of such a row is not full).
  __device__ __forceinline__ uint32_t at(int lane, int step) const {
    return static_cast<uint32_t>(first + lane) + static_cast<uint32_t>(kSampleThreads) * step;
  }
};

__device__ __forceinline__ PartCols part_cols(const float* row, int cols, int q) {
  PartCols p;
  p.vec = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  const int vecs = p.vec ? cols >> 2 : cols;
  p.vecs = vecs;
  p.first = 64 * q;
  p.steps = vecs > p.first ? (vecs - p.first - 1) / kSampleThreads + 1 : 0;
  const int full = vecs / kSampleThreads, rem = vecs % kSampleThreads;
  const int before = 64 * full * q + min(rem, 64 * q);  // vectors of the parts before
  p.list0 = p.vec ? 4 * before + (q > 0 ? cols & 3 : 0) : before;
  return p;
}

__global__ void __launch_bounds__(kPartThreads) sample_max_kernel(
    const float* __restrict__ logits, int64_t ld, const float* __restrict__ temps, int cols,
    PartStats st) {
  __shared__ float s_v[kPartThreads / 64];
  __shared__ int s_i[kPartThreads / 64];
  const int64_t r = blockIdx.x / kParts;
  const int q = blockIdx.x % kParts;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float* row = logits + r * ld;
  const bool greedy = !(temps[r] > 0.0f);
  const PartCols pc = part_cols(row, cols, q);
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  auto take = [&](float v, int c) {
    if (greedy) {
      if (better(v, c, bv, bi)) {
        bv = v;
        bi = c;
      }
    } else {
      bv = fmaxf(bv, v);
    }
  };
  // Wave w takes every fourth step; kPartSteps / 4 loads in flight per thread.
  constexpr int U = kPartSteps / 4;
  for (int m0 = 0; m0 < pc.steps; m0 += kPartSteps) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = pc.at(lane, m0 + wave + 4 * u);
      if (i < pc.vecs) {
        if (pc.vec) {
          v[u] = reinterpret_cast<const float4*>(row)[i];
        } else {
          v[u].x = row[i];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = pc.at(lane, m0 + wave + 4 * u);
      if (i < pc.vecs) {
        if (pc.vec) {
          take(v[u].x, 4 * i);
          take(v[u].y, 4 * i + 1);
          take(v[u].z, 4 * i + 2);
          take(v[u].w, 4 * i + 3);
        } else {
          take(v[u].x, i);
        }
      }
    }
  }
  if (pc.vec && q == 0 && wave == 0 && 4 * pc.vecs + lane < static_cast<uint32_t>(cols))
    take(row[4 * pc.vecs + lane], 4 * pc.vecs + lane);
  for (int mask = 1; mask < 64; mask <<= 1) {
    const float ov = lane_xor(bv, mask);
    const int oi = __builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, bi);
    if (greedy ? better(ov, oi, bv, bi) : ov > bv) {
      bv = ov;
      bi = oi;
    }
  }
  if (lane == 0) {
    s_v[wave] = bv;
    s_i[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kPartThreads / 64; ++w) {
      if (greedy ? better(s_v[w], s_i[w], bv, bi) : s_v[w] > bv) {
        bv = s_v[w];
        bi = s_i[w];
      }
    }
    st.best[blockIdx.x] = bv;
    st.best_at[blockIdx.x] = bi;
  }
}

// x / t for one divisor t: y = 1 / t rounded, q = x y, then one correction (Markstein: the
// quotient correctly rounded), 5 operations instead of a division's 12. An infinite or NaN q
// stays. Outside kQuotMin .. kQuotMax, where y or a product could leave the normal range, the
// plain division.
constexpr float kQuotMin = 1e-18f, kQuotMax = 1e18f;
struct Quot {
  float t, y;
  bool plain;
};
__device__ __forceinline__ Quot quot_of(float t) {
  return Quot{t, 1.0f / t, !(t > kQuotMin && t < kQuotMax)};
}
__device__ __forceinline__ float quot(float x, const Quot& d) {
  if (d.plain) return x / d.t;  // uniform
  const float q = x * d.y;
  const float c = fmaf(fmaf(-q, d.t, x), d.y, q);
  return fabsf(q) < INFINITY ? c : q;
}

// max(x / T) over the row = max(x) / T (division by T > 0 is monotone).
__device__ __forceinline__ float row_max(const PartStats& st, int64_t r, float t) {
  float mx = -INFINITY;
  for (int q = 0; q < kParts; ++q) mx = fmaxf(mx, st.best[r * kParts + q]);
  return mx / t;
}

__device__ __forceinline__ float row_sum(const PartStats& st, int64_t r) {
  float sum = st.sum[r * kParts];
  for (int q = 1; q < kParts; ++q) sum += st.sum[r * kParts + q];
  return sum;
}

// A row's limits: ranks and fixed-point mass before a kept rank.
struct Limits {
  uint64_t k, mass;
  bool truncate;
};
__device__ __forceinline__ Limits limits_of(int64_t k, float tp, int64_t cols) {
  Limits l;
  l.k = (k > 0 && k < cols) ? static_cast<uint64_t>(k) : static_cast<uint64_t>(cols);
  l.mass = tp < 1.0f ? (tp > 0.0f ? static_cast<uint64_t>(static_cast<double>(tp) * kMassUnit) : 0ull)
                     : ~0ull;
  l.truncate = tp < 1.0f || l.k < static_cast<uint64_t>(cols);
  return l;
}

// The first threshold that should hold the row's cut, by its count, or by its mass with a
// margin (one that does not is found out by the select); kCuts: none, or more columns than a
// list takes, or sums that are not finite.
__device__ __forceinline__ int list_cut(const int* cnt, const float* mass, const Limits& lim,
                                        float top_p, float sum, int cols) {
  int j = 0;
  while (j < kCuts && !(static_cast<uint64_t>(cnt[j]) >= lim.k ||
                        mass[j] > (top_p + 1e-3f) * sum || cnt[j] == cols))
    ++j;
  return j < kCuts && cnt[j] <= kListCap && sum < INFINITY ? j : kCuts;
}

// A little below the smallest logit with exp(x / t - mx) >= floor.
__device__ __forceinline__ float list_min(float floor, float t, float mx) {
  const float ln = logf(floor) - 1e-3f;
  return t * (mx + ln) - 1e-5f * (fabsf(t * mx) - t * ln);
}

__global__ void __launch_bounds__(kPartThreads) sample_sum_kernel(
    const float* __restrict__ logits, int64_t ld, const float* __restrict__ temps,
    const int64_t* __restrict__ top_ks, const float* __restrict__ top_ps, int cols, PartStats st) {
  __shared__ __align__(16) float4 s_e[kPartSteps][64];
  __shared__ int s_count[kPartThreads / 64][kCuts];
  __shared__ float s_mass[kPartThreads / 64][kCuts];
  const int64_t r = blockIdx.x / kParts;
  const int q = blockIdx.x % kParts;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float* row = logits + r * ld;
  const float t = temps[r];
  if (!(t > 0.0f)) return;  // greedy row
  const bool cuts = limits_of(top_ks[r], top_ps[r], cols).truncate;
  const PartCols pc = part_cols(row, cols, q);
  const float mx = row_max(st, r, t);
  const Quot div = quot_of(t);
  int n_cut[kCuts] = {};  // this wave's (uniform)
  float m_cut[kCuts] = {};
  auto exp_of = [&](float v, bool valid) {
    const float e = expf(quot(v, div) - mx);
    const bool hit = cuts && valid && e >= kCutMin[kCuts - 1];
    if (__builtin_amdgcn_ballot_w64(hit) != 0) {
#pragma unroll
      for (int j = 0; j < kCuts; ++j) {
        const bool in = hit && e >= kCutMin[j];
        n_cut[j] += __popcll(__builtin_amdgcn_ballot_w64(in));
        m_cut[j] += in ? e : 0.0f;
      }
    }
    return e;
  };
  constexpr int U = kPartSteps / 4;
  float part = 0.0f;  // wave 0: this layout thread's chain
  for (int m0 = 0; m0 < pc.steps; m0 += kPartSteps) {
    // Every load of the block first, then the exponentials.
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = pc.at(lane, m0 + wave + 4 * u);
      v[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (i < pc.vecs) {
        if (pc.vec) {
          v[u] = reinterpret_cast<const float4*>(row)[i];
        } else {
          v[u].x = row[i];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int m = m0 + wave + 4 * u;
      if (m < pc.steps) {  // uniform
        const uint32_t i = pc.at(lane, m);
        const bool ok = i < pc.vecs;
        float4 e = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        e.x = exp_of(v[u].x, ok);
        if (pc.vec) {
          e.y = exp_of(v[u].y, ok);
          e.z = exp_of(v[u].z, ok);
          e.w = exp_of(v[u].w, ok);
        }
        s_e[m - m0][lane] = e;
      }
    }
    __syncthreads();
    if (wave == 0) {
      const int n = min(kPartSteps, pc.steps - m0);
      for (int m1 = 0; m1 < n; m1 += 8) {
        float4 e[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) e[m] = s_e[min(m1 + m, n - 1)][lane];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
          if (m1 + m < n && pc.at(lane, m0 + m1 + m) < pc.vecs) {
            part += e[m].x;
            if (pc.vec) {
              part += e[m].y;
              part += e[m].z;
              part += e[m].w;
            }
          }
        }
      }
    }
    __syncthreads();
  }
  if (wave == 0 && pc.vec && q == 0 && (cols & 3) != 0) {
    const uint32_t c = 4 * pc.vecs + lane;
    const bool ok = c < static_cast<uint32_t>(cols);
    const float e = exp_of(ok ? row[c] : 0.0f, ok);
    if (ok) part += e;
  }
  for (int mask = 1; mask < 64; mask <<= 1) {
    part += lane_xor(part, mask);
#pragma unroll
    for (int j = 0; j < kCuts; ++j) m_cut[j] += lane_xor(m_cut[j], mask);
  }
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < kCuts; ++j) {
      s_count[wave][j] = n_cut[j];
      s_mass[wave][j] = m_cut[j];
    }
  }
  __syncthreads();
  if (cuts && threadIdx.x < kCuts) {
    int n = 0;
    float m = 0.0f;
    for (int w = 0; w < kPartThreads / 64; ++w) {
      n += s_count[w][threadIdx.x];
      m += s_mass[w][threadIdx.x];
    }
    st.count[st.stride * threadIdx.x + blockIdx.x] = n;
    st.mass[st.stride * threadIdx.x + blockIdx.x] = m;
  }
  if (threadIdx.x == 0) st.sum[blockIdx.x] = part;
}

// A row without limits: the best draw over the part's columns. e / sum as quot: exact to the
// bit wherever it reaches 2^-59, and below that p + 1e-10 is 1e-10 either way. (1 row 38 us in
// all, against 104 by one workgroup per row.)
__device__ __forceinline__ void draw_all(const float* __restrict__ row, int cols, int q, float t,
                                         float mx, float sum, uint32_t row_hash, float* best,
                                         int32_t* best_at) {
  __shared__ float s_v[kPartThreads / 64];
  __shared__ int s_i[kPartThreads / 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const PartCols pc = part_cols(row, cols, q);
  const Quot div = quot_of(t), inv = quot_of(sum);
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  auto take = [&](float v, int c) {
    const float p = quot(expf(quot(v, div) - mx), inv);
    const float s = logf(p + kSampleEps) + seeded_gumbel(row_hash, c);
    if (better(s, c, bv, bi)) {
      bv = s;
      bi = c;
    }
  };
  constexpr int U = kPartSteps / 4;
  for (int m0 = 0; m0 < pc.steps; m0 += kPartSteps) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = pc.at(lane, m0 + wave + 4 * u);
      v[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (i < pc.vecs) {
        if (pc.vec) {
          v[u] = reinterpret_cast<const float4*>(row)[i];
        } else {
          v[u].x = row[i];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = pc.at(lane, m0 + wave + 4 * u);
      if (i < pc.vecs) {
        if (pc.vec) {
          take(v[u].x, 4 * i);
          take(v[u].y, 4 * i + 1);
          take(v[u].z, 4 * i + 2);
          take(v[u].w, 4 * i + 3);
        } else {
          take(v[u].x, i);
        }
      }
    }
  }
  if (pc.vec && q == 0 && wave == 0 && 4 * pc.vecs + lane < static_cast<uint32_t>(cols))
    take(row[4 * pc.vecs + lane], 4 * pc.vecs + lane);
  for (int mask = 1; mask < 64; mask <<= 1) {
    const float ov = lane_xor(bv, mask);
    const int oi = __builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, bi);
    if (better(ov, oi, bv, bi)) {
      bv = ov;
      bi = oi;
    }
  }
  if (lane == 0) {
    s_v[wave] = bv;
    s_i[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kPartThreads / 64; ++w) {
      if (better(s_v[w], s_i[w], bv, bi)) {
        bv = s_v[w];
        bi = s_i[w];
      }
    }
    *best = bv;
    *best_at = bi;
  }
}

// (bound: one read of the logits from L2 / the last-level cache and the launch; sum: also ~45
// VALU operations an element, 30 us at 64 rows.)
// The columns of the part with e >= kCutMin[j], j = list_cut. Candidates are picked by the
// logit itself, a little below the threshold; only those take an exponential.
__global__ void __launch_bounds__(kPartThreads) sample_list_kernel(
    const float* __restrict__ logits, int64_t ld, const float* __restrict__ temps,
    const int64_t* __restrict__ top_ks, const float* __restrict__ top_ps,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ positions, int cols,
    PartStats st, uint32_t* __restrict__ lists) {
  __shared__ int s_cnt[kCuts];
  __shared__ float s_mass[kCuts];
  __shared__ int s_n;
  const int64_t r = blockIdx.x / kParts;
  const int q = blockIdx.x % kParts;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float t = temps[r];
  if (!(t > 0.0f)) return;  // greedy row
  const float tp = top_ps[r];
  const Limits lim = limits_of(top_ks[r], tp, cols);
  const float* row = logits + r * ld;
  if (!lim.truncate) {
    draw_all(row, cols, q, t, row_max(st, r, t), row_sum(st, r),
             gumbel_row(seeds[r], positions[r]), st.mass + blockIdx.x, st.count + blockIdx.x);
    return;
  }
  // (threshold, part) totals: kParts = 16 lanes per threshold
  static_assert(kParts == 16 && kCuts * kParts <= kPartThreads, "one thread per total");
  if (threadIdx.x < kCuts * kParts) {
    const int64_t at = st.stride * (threadIdx.x / kParts) + r * kParts + threadIdx.x % kParts;
    int c = st.count[at];
    float m = st.mass[at];
    for (int mask = 1; mask < kParts; mask <<= 1) {
      c += __shfl_xor(c, mask);
      m += __shfl_xor(m, mask);
    }
    s_cnt[threadIdx.x / kParts] = c;
    s_mass[threadIdx.x / kParts] = m;
  }
  if (threadIdx.x == 0) s_n = 0;
  const float mx = row_max(st, r, t);
  const float sum = row_sum(st, r);
  __syncthreads();
  const int j = list_cut(s_cnt, s_mass, lim, tp, sum, cols);
  if (q == 0 && threadIdx.x == 0) st.cut_at[r * kParts] = j;
  if (j == kCuts) return;
  const PartCols pc = part_cols(row, cols, q);
  uint32_t* list = lists + r * cols + pc.list0;
  const float floor = kCutMin[j];
  const float v_min = list_min(floor, t, mx);
  const Quot div = quot_of(t);
  auto take = [&](float v, int c, bool valid) {
    if (__builtin_amdgcn_ballot_w64(valid && v >= v_min) == 0) return;
    const bool in = valid && expf(quot(v, div) - mx) >= floor;
    const uint64_t hits = __builtin_amdgcn_ballot_w64(in);
    int at = 0;
    if (lane == 0) at = atomicAdd(&s_n, __popcll(hits));
    at = __builtin_amdgcn_readfirstlane(at) + __popcll(hits & ((1ull << lane) - 1));
    if (in) list[at] = c;
  };
  constexpr int U = kPartSteps / 4;
  for (int m0 = 0; m0 < pc.steps; m0 += kPartSteps) {
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = pc.at(lane, m0 + wave + 4 * u);
      v[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (i < pc.vecs) {
        if (pc.vec) {
          v[u] = reinterpret_cast<const float4*>(row)[i];
        } else {
          v[u].x = row[i];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int m = m0 + wave + 4 * u;
      if (m < pc.steps) {  // uniform
        const uint32_t i = pc.at(lane, m);
        const bool ok = i < pc.vecs;
        if (pc.vec) {
          take(v[u].x, 4 * i, ok);
          take(v[u].y, 4 * i + 1, ok);
          take(v[u].z, 4 * i + 2, ok);
          take(v[u].w, 4 * i + 3, ok);
        } else {
          take(v[u].x, i, ok);
        }
      }
    }
  }
  if (wave == 0 && pc.vec && q == 0 && (cols & 3) != 0) {
    const uint32_t c = 4 * pc.vecs + lane;
    const bool ok = c < static_cast<uint32_t>(cols);
    take(ok ? row[c] : 0.0f, c, ok);
  }
}

// ---- the cut and the draw, one workgroup per row ------------------------------------------

constexpr int kFewKeys = 64;    // keys around the cut that one wave ranks directly
constexpr int kListCopies = 4;  // histogram copies for the list (the passes over all columns: 16)

// Radix histograms, one copy per few lanes (so few lanes of a wave instruction hit one
// address); rows padded to 257 entries so equal bins of different copies fall in different
// LDS banks.
struct Hist {
  uint64_t* mass;  // [copies][257]
  uint32_t* cnt;
  int copies;
};

struct Cut {
  uint32_t key;                    // of the last kept rank (its leading bits, if stopped early)
  uint64_t cnt_above, mass_above;  // ranks with larger keys
  uint64_t cnt;                    // ranks with this key
};

// The radix select: each(f) calls f(key) for the caller's share of the n keys. Stops once at
// most `enough` keys share the cut's leading bits (pmask). Every thread returns the same cut.
template <typename Each>
__device__ __forceinline__ Cut select_cut(const Hist& h, uint64_t* s_sel, uint64_t k_lim,
                                          uint64_t mass_lim, uint64_t n, uint64_t enough,
                                          uint32_t& pmask, Each&& each) {
  const int tid = threadIdx.x;
  const int copy = tid & (h.copies - 1);
  Cut cut{0, 0, 0, n};
  pmask = 0;
  for (int level = 0; level < 4 && cut.cnt > enough; ++level) {
    const int shift = 24 - 8 * level;
    for (int i = tid; i < h.copies * 257; i += kSampleThreads) {
      h.cnt[i] = 0;
      h.mass[i] = 0;
    }
    __syncthreads();
    each([&](uint32_t key) {
      if ((key & pmask) == cut.key) {
        const int b = copy * 257 + ((key >> shift) & 255);
        atomicAdd(&h.cnt[b], 1u);
        atomicAdd(reinterpret_cast<unsigned long long*>(&h.mass[b]),
                  static_cast<unsigned long long>(mass_of(key)));
      }
    });
    __syncthreads();
    if (tid < 256) {  // integer totals: exact in any order
      uint32_t cn = 0;
      uint64_t ms = 0;
      for (int w = 0; w < h.copies; ++w) {
        cn += h.cnt[w * 257 + tid];
        ms += h.mass[w * 257 + tid];
      }
      h.cnt[tid] = cn;
      h.mass[tid] = ms;
    }
    __syncthreads();
    if (tid < 64) {
      // Lane l holds bins 255 - 4l .. 252 - 4l. The bin of the last kept rank is the lowest
      // non-empty one whose first rank is kept, i.e. with fewer than k_lim ranks and at most
      // mass_lim of mass above it (both only grow downwards).
      uint32_t cn[4];
      uint64_t ms[4];
      uint64_t c = 0, m = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        cn[k] = h.cnt[255 - 4 * tid - k];
        ms[k] = h.mass[255 - 4 * tid - k];
        c += cn[k];
        m += ms[k];
      }
      uint64_t ci = c, mi = m;  // inclusive sums over the lanes above
      for (int off = 1; off < 64; off <<= 1) {
        const uint64_t oc = __shfl_up(ci, off), om = __shfl_up(mi, off);
        if (tid >= off) {
          ci += oc;
          mi += om;
        }
      }
      uint64_t before_c = cut.cnt_above + ci - c, before_m = cut.mass_above + mi - m;
      int chosen = -1;
      uint64_t at_c = 0, at_m = 0, at_n = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (cn[k] != 0 && before_c < k_lim && before_m <= mass_lim) {
          chosen = 255 - 4 * tid - k;
          at_c = before_c;
          at_m = before_m;
          at_n = cn[k];
        }
        before_c += cn[k];
        before_m += ms[k];
      }
      const uint64_t have = __builtin_amdgcn_ballot_w64(chosen >= 0);
      // (rank 0 is always kept: with no such bin, the highest non-empty one)
      if (have != 0 && tid == 63 - __clzll(have)) {
        s_sel[0] = cut.key | (static_cast<uint32_t>(chosen) << shift);
        s_sel[1] = at_c;
        s_sel[2] = at_m;
        s_sel[3] = at_n;
      }
    }
    __syncthreads();
    cut = Cut{static_cast<uint32_t>(s_sel[0]), s_sel[1], s_sel[2], s_sel[3]};
    pmask |= 0xffu << shift;
  }
  return cut;
}

// How many of the cut's equal keys are kept (>= 1).
__device__ __forceinline__ uint64_t ties_kept(const Cut& c, uint64_t k_lim, uint64_t mass_lim) {
  uint64_t n = c.cnt;
  if (k_lim - c.cnt_above < n) n = k_lim - c.cnt_above;
  const uint64_t q = mass_of(c.key);
  if (mass_lim != ~0ull && q > 0) {
    const uint64_t by_mass = (mass_lim - c.mass_above) / q + 1;
    if (by_mass < n) n = by_mass;
  }
  return n;
}

constexpr int kSelectLds = kListCap * 8;                          // keys and columns of the list
static_assert(kHistCopies * 257 * 12 <= kSelectLds, "the full passes' histograms fit there");
constexpr int kListHistLds = kListCopies * 257 * 12 + 8;

// WHOLE: the one launch of a call; the row's maximum, sum and list are made here, with the
// bits and in the order of the launches above, and rows of any kind are finished.
template <bool WHOLE>
__global__ void __launch_bounds__(kSampleThreads) sample_select_kernel(
    const float* __restrict__ logits, int64_t ld, const float* __restrict__ temps,
    const int64_t* __restrict__ top_ks, const float* __restrict__ top_ps,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ positions, int64_t cols,
    PartStats st, uint32_t* __restrict__ keys_ws, int64_t* __restrict__ out) {
  extern __shared__ __align__(16) char s_mem[];
  __shared__ float s_bv[kSampleWaves];
  __shared__ int64_t s_bi[kSampleWaves];
  __shared__ int64_t s_scan[kSampleThreads];
  __shared__ uint64_t s_sel[4];
  __shared__ int64_t s_cut;
  __shared__ int s_ties, s_listed;
  __shared__ int s_cnt[kSampleWaves][kCuts];
  __shared__ float s_mass[kSampleWaves][kCuts];
  __shared__ uint32_t s_few_key[kFewKeys], s_few_col[kFewKeys];

  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int ncols = static_cast<int>(cols);
  const float* row = logits + r * ld;
  const float t = temps[r];

  float bv = -INFINITY;
  int64_t bi = cols;
  const Limits lim = limits_of(top_ks[r], top_ps[r], cols);
  if (!WHOLE && (!(t > 0.0f) || !lim.truncate)) {  // the parts' best logits or draws
    if (tid == 0) {
      const float* v = t > 0.0f ? st.mass : st.best;
      const int32_t* i = t > 0.0f ? st.count : st.best_at;
      for (int q = 0; q < kParts; ++q) {
        const int at = i[r * kParts + q];
        if (at < ncols && better(v[r * kParts + q], at, bv, bi)) {
          bv = v[r * kParts + q];
          bi = at;
        }
      }
      out[r] = bi < cols ? bi : 0;
    }
    return;
  }
  uint32_t* ws = keys_ws + r * cols;
  const uint64_t k_lim = lim.k, mass_lim = lim.mass;
  const uint32_t row_hash = gumbel_row(seeds[r], positions[r]);
  const Quot by_t = quot_of(t);
  auto take = [&](float s, int c) {
    if (better(s, c, bv, bi)) {
      bv = s;
      bi = c;
    }
  };
  auto draw = [&](uint32_t key, int c) {
    take(logf(__uint_as_float(key) + kSampleEps) + seeded_gumbel(row_hash, c), c);
  };
  auto finish = [&]() {
    block_best(bv, bi, s_bv, s_bi);
    if (tid == 0) out[r] = bi < cols ? bi : 0;
  };

  float mx, sum;
  int cut_at;
  if constexpr (WHOLE) {
    if (!(t > 0.0f)) {  // greedy row
      for_each_col<8>(row, ncols, take);
      finish();
      return;
    }
    float m = -INFINITY;
    for_each_col<8>(row, ncols, [&](float v, int) { m = fmaxf(m, v); });
    mx = block_fold(m, s_bv, [](float x, float y) { return fmaxf(x, y); }) / t;
    float part = 0.0f;
    int n_cut[kCuts] = {};
    float m_cut[kCuts] = {};
    for_each_col<4>(row, ncols, [&](float v, int) {
      const float e = expf(quot(v, by_t) - mx);
      part += e;
      if (lim.truncate && __builtin_amdgcn_ballot_w64(e >= kCutMin[kCuts - 1]) != 0) {
#pragma unroll
        for (int j = 0; j < kCuts; ++j) {
          n_cut[j] += e >= kCutMin[j];
          m_cut[j] += e >= kCutMin[j] ? e : 0.0f;
        }
      }
    });
    sum = block_fold(part, s_bv, [](float x, float y) { return x + y; });
    if (!lim.truncate) {  // (e / sum as quot: see draw_all)
      const Quot inv = quot_of(sum);
      for_each_col<4>(row, ncols, [&](float v, int c) {
        draw(__float_as_uint(quot(expf(quot(v, by_t) - mx), inv)), c);
      });
      finish();
      return;
    }
    for (int j = 0; j < kCuts; ++j) {
      for (int mask = 1; mask < 64; mask <<= 1) {
        n_cut[j] += __shfl_xor(n_cut[j], mask);
        m_cut[j] += lane_xor(m_cut[j], mask);
      }
      if ((tid & 63) == 0) {
        s_cnt[tid >> 6][j] = n_cut[j];
        s_mass[tid >> 6][j] = m_cut[j];
      }
    }
    __syncthreads();
    if (tid < kCuts) {
      for (int w = 1; w < kSampleWaves; ++w) {
        s_cnt[0][tid] += s_cnt[w][tid];
        s_mass[0][tid] += s_mass[w][tid];
      }
    }
    if (tid == 0) s_listed = 0;
    __syncthreads();
    cut_at = list_cut(s_cnt[0], s_mass[0], lim, top_ps[r], sum, ncols);
  } else {
    mx = row_max(st, r, t);
    sum = row_sum(st, r);
    cut_at = st.cut_at[r * kParts];
  }

  // The list: every column with e >= kCutMin[cut_at]. A column outside has p at most
  // fl(kCutMin[cut_at] / sum), so a cut key above that lies, with all its ties and everything
  // kept, inside, provided that the list does not end before the limits are reached.
  if (cut_at < kCuts) {
    uint32_t* l_key = reinterpret_cast<uint32_t*>(s_mem);
    uint32_t* l_col = l_key + kListCap;
    uint64_t* lh_mass = reinterpret_cast<uint64_t*>(s_mem + kSelectLds);
    const Hist lh{lh_mass, reinterpret_cast<uint32_t*>(lh_mass + kListCopies * 257), kListCopies};
    int n = 0;
    if constexpr (WHOLE) {
      n = s_cnt[0][cut_at];
      const float floor = kCutMin[cut_at];
      const float v_min = list_min(floor, t, mx);
      for_each_col<8>(row, ncols, [&](float v, int c) {
        if (v < v_min) return;
        const float e = expf(quot(v, by_t) - mx);
        if (e >= floor) {
          const int at = atomicAdd(&s_listed, 1);
          l_col[min(at, kListCap - 1)] = c;
          l_key[min(at, kListCap - 1)] = __float_as_uint(e / sum);
        }
      });
    } else {
      // Wave w reads part w's list.
      const int32_t* counts = st.count + st.stride * cut_at + r * kParts;
      const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
      int first = 0;
      for (int q = 0; q < kParts; ++q) {
        if (q == wave) first = n;
        n += counts[q];
      }
      const uint32_t* list = ws + part_cols(row, ncols, wave).list0;
#pragma unroll 4
      for (int i = tid & 63; i < counts[wave]; i += 64) {
        const uint32_t c = min(list[i], static_cast<uint32_t>(ncols - 1));
        l_col[first + i] = c;
        l_key[first + i] = __float_as_uint(expf(quot(row[c], by_t) - mx) / sum);
      }
    }
    if (tid == 0) s_ties = 0;
    __syncthreads();
    // The select narrows the cut to at most kFewKeys keys; one wave ranks those directly (by
    // key, then column: ties need no separate step). More equal keys than that: the passes
    // over all columns.
    uint32_t pmask;
    const Cut cut = select_cut(lh, s_sel, k_lim, mass_lim, n, kFewKeys, pmask, [&](auto&& f) {
      for (int i = tid; i < n; i += kSampleThreads) f(l_key[i]);
    });
    if (cut.cnt <= kFewKeys) {
      for (int i = tid; i < n; i += kSampleThreads) {
        if ((l_key[i] & pmask) == cut.key) {
          const int at = atomicAdd(&s_ties, 1);
          s_few_key[at] = l_key[i];
          s_few_col[at] = l_col[i];
        }
      }
      __syncthreads();
      const int few = static_cast<int>(cut.cnt);
      if (tid < few) {
        const uint32_t key = s_few_key[tid], col = s_few_col[tid];
        uint64_t rank = cut.cnt_above, mass = cut.mass_above;
        for (int i = 0; i < few; ++i) {
          const uint32_t ok = s_few_key[i];
          if (ok > key || (ok == key && s_few_col[i] < col)) {
            ++rank;
            mass += mass_of(ok);
          }
        }
        // Kept ranks are a prefix: the last kept one is the one with the highest rank.
        const bool kept = rank == 0 || (rank < k_lim && mass <= mass_lim);
        const uint64_t all = __builtin_amdgcn_ballot_w64(kept);
        if (kept && rank == cut.cnt_above + __popcll(all) - 1) {
          s_sel[0] = key;
          // whether the next rank, listed or not, is known to be dropped
          s_sel[1] = rank + 1 < static_cast<uint64_t>(n) || rank + 1 == k_lim ||
                     mass + mass_of(key) > mass_lim;
          s_cut = col;
        }
      }
      __syncthreads();
      const uint32_t key_cut = static_cast<uint32_t>(s_sel[0]);
      const int idx_cut = static_cast<int>(s_cut);
      if (n == ncols || (s_sel[1] != 0 && key_cut > __float_as_uint(kCutMin[cut_at] / sum))) {
        for (int i = tid; i < n; i += kSampleThreads) {
          const int c = static_cast<int>(l_col[i]);
          if (l_key[i] > key_cut || (l_key[i] == key_cut && c <= idx_cut)) draw(l_key[i], c);
        }
        finish();
        return;
      }
    }
    __syncthreads();  // the list's LDS and workspace are free
  }

  // Over all columns: keys = bits of p (p >= 0, so they order like p), written once, read by
  // every level.
  uint32_t* keys = ws;
  for_each_col<4>(row, ncols, [&](float v, int c) {
    keys[c] = __float_as_uint(expf(v / t - mx) / sum);
  });
  __syncthreads();  // keys visible to the block
  uint64_t* h_mass = reinterpret_cast<uint64_t*>(s_mem);
  const Hist h{h_mass, reinterpret_cast<uint32_t*>(h_mass + kHistCopies * 257), kHistCopies};
  uint32_t pmask;
  const Cut cut = select_cut(h, s_sel, k_lim, mass_lim, cols, 0, pmask, [&](auto&& f) {
    for_each_col<8>(reinterpret_cast<const float*>(keys), ncols,
                    [&](float kv, int) { f(__float_as_uint(kv)); });
  });
  const uint64_t keep = ties_kept(cut, k_lim, mass_lim);
  int64_t idx_cut = cols;  // among keys == cut.key, indices <= idx_cut are kept
  if (keep < cut.cnt) {
    // Index of the keep-th tie in index order: contiguous chunks, block scan.
    const int64_t chunk = (cols + kSampleThreads - 1) / kSampleThreads;
    const int64_t c0 = min(cols, chunk * tid);
    const int64_t c1 = min(cols, c0 + chunk);
    int64_t mine = 0;
    for (int64_t c = c0; c < c1; ++c) mine += keys[c] == cut.key;
    s_scan[tid] = mine;
    __syncthreads();
    for (int off = 1; off < kSampleThreads; off <<= 1) {  // inclusive scan
      const int64_t add = tid >= off ? s_scan[tid - off] : 0;
      __syncthreads();
      s_scan[tid] += add;
      __syncthreads();
    }
    const int64_t before = s_scan[tid] - mine;
    const int64_t want = static_cast<int64_t>(keep) - 1;  // 0-based tie position
    if (want >= before && want < before + mine) {
      int64_t seen = before;
      for (int64_t c = c0; c < c1; ++c) {
        if (keys[c] == cut.key) {
          if (seen == want) {
            s_cut = c;
            break;
          }
          ++seen;
        }
      }
    }
    __syncthreads();
    idx_cut = s_cut;
  }
  for_each_col<4>(reinterpret_cast<const float*>(keys), ncols, [&](float kv, int c) {
    const uint32_t key = __float_as_uint(kv);
    if (key > cut.key || (key == cut.key && c <= idx_cut)) draw(key, c);
  });
  finish();
}

// A launch holds fewer than 2^32 work-items (beyond that rows are silently left out).
constexpr int64_t kRowsPerLaunch = 1 << 19;
static_assert(kRowsPerLaunch * kParts * kPartThreads < (1ll << 32) &&
                  kRowsPerLaunch * kSampleThreads < (1ll << 32),
              "a launch's work-items");

// The rule between the forms (see the top of the file): from 144 rows, 9 / 16 of the CUs, and
// from fewer where rows are short, as three launches' cost does not shrink with them. One
// launch vs four, us; greedy rows / rows without limits / top-p 0.9 over peaked rows:
//   151936 columns:  64 rows  29 vs  23   112 vs  67    70 vs  58
//                   128       30 vs  35   116 vs 112    76 vs  94
//                   256       34 vs  55   129 vs 190    85 vs 152
//   65536 columns:   64       15 vs  15    49 vs  34    36 vs  34
//                   128       16 vs  21    51 vs  55    37 vs  52
//   32000 columns:   64       10 vs  13    29 vs  27    27 vs  30
//                   128       10 vs  16    30 vs  38    26 vs  39
//   16000 columns:    1        7 vs  11    18 vs  17    16 vs  19
//    4096 columns:    1        5 vs  11     9 vs  16    13 vs  18
//                  1024       19 vs  63    36 vs 155    59 vs 169
bool one_workgroup_per_row(int64_t rows, int64_t cols) {
  return (144 - rows) * cols <= 144ll * 16000;
}

}  // namespace
}  // namespace sid

using namespace sid;

extern "C" int sid_argmax_rows(const float* logits, int64_t ld, int64_t* out, int64_t rows,
                               int64_t cols, void* stream) {
  SID_REQUIRE(rows >= 0 && cols >= 0, "argmax_rows: negative size");
  if (rows == 0) return SID_OK;
  SID_REQUIRE(logits && out, "argmax_rows: null pointer");
  SID_REQUIRE(cols > 0 && ld >= cols, "argmax_rows: bad row stride %lld for %lld columns",
              (long long)ld, (long long)cols);
  SID_REQUIRE(rows < (1ll << 31) && cols < (1ll << 31), "argmax_rows: too large");
  for (int64_t r0 = 0; r0 < rows; r0 += kRowsPerLaunch) {
    hipLaunchKernelGGL(argmax_kernel, dim3((unsigned)std::min(kRowsPerLaunch, rows - r0)),
                       dim3(kSampleThreads), 0, static_cast<hipStream_t>(stream), logits + r0 * ld,
                       ld, out + r0, cols);
    const int rc = check_launch("argmax_rows");
    if (rc != SID_OK) return rc;
  }
  return SID_OK;
}

// Per row: one word per column (the listed columns, or every column's key), then the parts'
// statistics.
extern "C" int64_t sid_sample_workspace_bytes(int64_t rows, int64_t cols) {
  if (rows <= 0 || cols <= 0) return 0;
  return rows * (cols + kPartWords * kParts) * static_cast<int64_t>(sizeof(uint32_t));
}

extern "C" int sid_sample_rows(const float* logits, int64_t ld, const float* temperatures,
                               const int64_t* top_ks, const float* top_ps, const int64_t* seeds,
                               const int64_t* positions, int64_t rows, int64_t cols,
                               void* workspace, int64_t workspace_bytes, int64_t* out,
                               void* stream) {
  SID_REQUIRE(rows >= 0 && cols >= 0, "sample_rows: negative size");
  if (rows == 0) return SID_OK;
  SID_REQUIRE(logits && temperatures && top_ks && top_ps && seeds && positions && out,
              "sample_rows: null pointer");
  SID_REQUIRE(cols > 0 && ld >= cols, "sample_rows: bad row stride %lld for %lld columns",
              (long long)ld, (long long)cols);
  SID_REQUIRE(rows < (1ll << 31) && cols < (1ll << 31), "sample_rows: too large");
  const int64_t need = sid_sample_workspace_bytes(rows, cols);
  SID_REQUIRE(workspace != nullptr && workspace_bytes >= need,
              "sample_rows: workspace %lld bytes, need %lld", (long long)workspace_bytes,
              (long long)need);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  uint32_t* lists = static_cast<uint32_t*>(workspace);
  float* stats = reinterpret_cast<float*>(lists + rows * cols);
  const int64_t parts = rows * kParts;
  const bool whole = one_workgroup_per_row(rows, cols);
  auto select = whole ? &sample_select_kernel<true> : &sample_select_kernel<false>;
  hipFuncSetAttribute(reinterpret_cast<const void*>(select),
                      hipFuncAttributeMaxDynamicSharedMemorySize, kSelectLds + kListHistLds);
  for (int64_t r0 = 0; r0 < rows; r0 += kRowsPerLaunch) {
    const int64_t n = std::min(kRowsPerLaunch, rows - r0);
    const float* lg = logits + r0 * ld;
    float* s0 = stats + r0 * kParts;
    const PartStats st{s0, reinterpret_cast<int32_t*>(s0 + parts), s0 + 2 * parts,
                       reinterpret_cast<int32_t*>(s0 + 3 * parts), s0 + (3 + kCuts) * parts, parts,
                       reinterpret_cast<int32_t*>(s0 + (3 + 2 * kCuts) * parts)};
    int rc = SID_OK;
    if (!whole) {
      const dim3 grid((unsigned)(n * kParts));
      hipLaunchKernelGGL(sample_max_kernel, grid, dim3(kPartThreads), 0, s, lg, ld,
                         temperatures + r0, (int)cols, st);
      rc = check_launch("sample_rows max");
      if (rc != SID_OK) return rc;
      hipLaunchKernelGGL(sample_sum_kernel, grid, dim3(kPartThreads), 0, s, lg, ld,
                         temperatures + r0, top_ks + r0, top_ps + r0, (int)cols, st);
      rc = check_launch("sample_rows sum");
      if (rc != SID_OK) return rc;
      hipLaunchKernelGGL(sample_list_kernel, grid, dim3(kPartThreads), 0, s, lg, ld,
                         temperatures + r0, top_ks + r0, top_ps + r0, seeds + r0, positions + r0,
                         (int)cols, st, lists + r0 * cols);
      rc = check_launch("sample_rows list");
      if (rc != SID_OK) return rc;
    }
    hipLaunchKernelGGL(select, dim3((unsigned)n), dim3(kSampleThreads), kSelectLds + kListHistLds, s,
                       lg, ld, temperatures + r0, top_ks + r0, top_ps + r0, seeds + r0,
                       positions + r0, cols, st, lists + r0 * cols, out + r0);
    rc = check_launch("sample_rows");
    if (rc != SID_OK) return rc;
  }
  return SID_OK;
}
