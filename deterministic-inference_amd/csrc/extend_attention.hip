// Varlen causal "extend" attention over the paged KV pool, gfx950 MFMA.
//
// Used for prefill and for the DVR verify pass (sid/kernels/extend_attention.py
// :1-22 states the contract). All keys, prefix and freshly written window, are
// read from the pool through kv_indices, and causality is by absolute position:
// query j of request b is at position prefix_b + j and sees keys <= that.
//
// Reduction order (what makes results bitwise invariant to the window offset
// and to co-batched requests): keys are cut into splits of KSPLIT = 256
// positions anchored at absolute position 0, each split into 64-key tiles.
// Inside a split a query row runs an online softmax from a fresh state over the
// split's tiles in order; the split states are then folded into the row's
// running state in increasing split order by fold(). Tiles and splits beyond a
// row's position are exact no-ops for it (rescale 2^0 = 1, p = 0, fold
// weight 2^(-1e30 - m) = 0). States keep their maximum m in log2 units
// (scores times sm_scale * log2(e)). So a row's bits depend only on its q, its
// absolute position and its sequence's keys. A launch either walks a query
// tile's splits sequentially in one workgroup, or (when a workspace is given
// and the grid would be small, e.g. the 4 x 32 verify pass) gives every split
// its own workgroup and folds the saved split states afterwards with the same
// fold() in the same order: identical bits, many more workgroups.
//
// Workgroup = (request, kv head, 32-query tile[, split]) with 4 waves; the two
// query heads of the GQA pair share every K/V tile (wave w: head w / 2, query
// rows 16 * (w % 2) .. +15). Per 64-key tile:
//   S^T = K Q^T   : 4 key blocks x 4 k-steps of v_mfma_f32_16x16x32_bf16, with
//                   A = K rows from LDS and B = q held in registers. Key rows are
//                   assigned to MFMA rows so that each lane ends up holding 8
//                   consecutive keys for its query, which is exactly the B
//                   operand layout of the PV product (no shuffles needed);
//   softmax       : online, per query row, with a lazy reference maximum (moved
//                   only when a tile's maximum exceeds it by 2^8); reductions
//                   over the 4 lanes of a row by xor 16 / xor 32 (max is
//                   order-free, sums commute);
//   O^T += V^T P^T: 8 dim blocks x 2 k-steps, A = V^T from a transposed LDS
//                   copy of the V tile, B = bf16(P) (P is rounded to bf16
//                   before the PV product, as sid/kernels/extend_attention.py:106).
#include "common.h"

#include <type_traits>

namespace sid {
namespace {

constexpr int D = 128;
constexpr int BN = 64;          // keys per tile
constexpr int BQ = 32;          // query positions per workgroup (x 2 heads = 64 rows)
constexpr int KSPLIT = 256;     // keys per split (4 tiles), anchored at position 0
// LDS row strides (bf16) of the K and V tiles: 304 bytes each. Layout only (bit-identical);
// of 136-152 x 136-160 this measured best on the verify fan-out (~4% over 272 / 288 bytes)
// and equal on prefill.
constexpr int KS_STRIDE = D + 24;
constexpr int VS_STRIDE = D + 24;
constexpr float NEG_BIG = -1e30f;
constexpr float LOG2E = 1.4426950408889634f;
// Slack of the lazy softmax maximum, in log2 units: scores up to 2^LAZY_T above the row's
// reference maximum are taken without moving it.
constexpr float LAZY_T = 8.0f;

// 2^x by the hardware instruction (v_exp_f32): the argument is at most LAZY_T, and results
// that would be denormal may flush to zero.
__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Reductions over lanes l and l ^ 16 (l ^ 32): v_permlane16/32_swap hand each lane the
// values of both lanes of its pair as (lower lane's, upper lane's), so both lanes compute
// the same expression on the same operands (identical bits) without an LDS round trip.
__device__ __forceinline__ float pair16_max(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
__device__ __forceinline__ float pair32_max(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
__device__ __forceinline__ float pair16_sum(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
__device__ __forceinline__ float pair32_sum(float v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

typedef short s16x4_v __attribute__((ext_vector_type(4)));
typedef short s16x8_v __attribute__((ext_vector_type(8)));

typedef __attribute__((address_space(3))) char* lds_char_t;

// 4 bf16 of a V^T fragment through the LDS transpose read: within each 16-lane group,
// lane L receives element L % 4 of the 8-byte values addressed by lanes L / 4 + 4j
// (j = 0..3) of its group.
__device__ __forceinline__ s16x4_v ld_tr16(const bf16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_v*)(p));
}

// acc / l (l > 0), shared by every path that divides: y = 1 / l rounded, q = acc y, then one
// correction (Markstein: the quotient correctly rounded), 5 operations for each of a row's
// dims instead of a division's 12. An infinite or NaN q stays.
__device__ __forceinline__ float div_row(float acc, float l, float y) {
  const float q = acc * y;
  const float c = __builtin_fmaf(__builtin_fmaf(-q, l, acc), y, q);
  return __builtin_fabsf(q) < INFINITY ? c : q;
}

// Per-lane softmax state of one query row (the lane's 32 output dims).
struct RowState {
  float m;
  float l;
  f32x4_v acc[8];
};

__device__ __forceinline__ void fresh(RowState& s) {
  s.m = NEG_BIG;
  s.l = 0.0f;
#pragma unroll
  for (int db = 0; db < 8; ++db) s.acc[db] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
}

// run <- fold(run, part): the one merge used by every path.
// The fold's per-row scalars and its elementwise step, shared by every path that folds.
struct FoldScale {
  float mn, alpha, beta;
};
__device__ __forceinline__ FoldScale fold_scale(float run_m, float m) {
  const float mn = fmaxf(run_m, m);
  return {mn, exp2_fast(run_m - mn), exp2_fast(m - mn)};
}
// Written as one explicit fma over a separately rounded product, so the compiler has no
// contraction choice to make differently in different kernels.
__device__ __forceinline__ float fold_elem(float run, float part, const FoldScale& f) {
  return __builtin_fmaf(run, f.alpha, part * f.beta);
}

__device__ __forceinline__ void fold(RowState& run, float m, float l, const f32x4_v (&a)[8]) {
  const FoldScale f = fold_scale(run.m, m);
  run.l = fold_elem(run.l, l, f);
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i) run.acc[db][i] = fold_elem(run.acc[db][i], a[db][i], f);
  run.m = f.mn;
}

// The row's output: acc / l rounded to bf16 (this lane: dims 16 db + 4 g .. +3).
__device__ __forceinline__ void store_row(bf16_t* op, const RowState& run, int g) {
  const float y = 1.0f / run.l;
#pragma unroll
  for (int db = 0; db < 8; ++db) {
    const f32x4_v a = run.acc[db];
    uint2 u;
    u.x = pack_bf16x2(div_row(a[0], run.l, y), div_row(a[1], run.l, y));
    u.y = pack_bf16x2(div_row(a[2], run.l, y), div_row(a[3], run.l, y));
    *reinterpret_cast<uint2*>(op + 16 * db + 4 * g) = u;
  }
}

struct Ctx {
  const bf16_t* k_cache;
  const bf16_t* v_cache;
  const int32_t* idx;
  int64_t row_stride;
  int64_t num_slots;
  int kv_len;
  int h_kv;
  int q_abs;
  int q_min;
  int q_max;
  bool row_ok;
  int r, g, wave, lane, tid;
};

// Global -> register staging of one 64-key tile (K row-major, V for the transposed copy).
// Loaded one tile ahead of the math, so the next tile's HBM round trip overlaps the
// current tile's MFMAs; 8 x 16 bytes per thread.
struct TileRegs {
  u32x4_v k[4];
  u32x4_v v[4];
};

// Pool slots of the split's keys, staged in LDS once per split (s_idx[j] = slot of key
// split_start + j; 0 past the sequence or out of range), so a tile's K/V loads wait on
// LDS rather than on a global index load.
__device__ __forceinline__ void stage_slots(int32_t* s_idx, const Ctx& c, int split_start) {
  const int pos = split_start + c.tid;
  int32_t slot = pos < c.kv_len ? c.idx[pos] : 0;
  if (slot < 0 || slot >= c.num_slots) slot = 0;
  s_idx[c.tid] = slot;
}

__device__ __forceinline__ void load_tile(TileRegs& r, const Ctx& c, const int32_t* s_idx,
                                          int k0) {
  // K: vector v = tid + 256*i -> key v/16, 16-byte chunk v%16 (k0: tile offset in split).
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int v = c.tid + 256 * i;
    const int64_t slot = s_idx[k0 + (v >> 4)];
    r.k[i] = reinterpret_cast<const u32x4_v*>(c.k_cache + slot * c.row_stride + c.h_kv * D)[v & 15];
  }
  // V: the same key / chunk assignment (rows stored as they are; transposed on read).
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int v = c.tid + 256 * i;
    const int64_t slot = s_idx[k0 + (v >> 4)];
    r.v[i] = reinterpret_cast<const u32x4_v*>(c.v_cache + slot * c.row_stride + c.h_kv * D)[v & 15];
  }
}

__device__ __forceinline__ void store_tile(const TileRegs& r, const Ctx& c, bf16_t* sK,
                                           bf16_t* sV) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int v = c.tid + 256 * i;
    *reinterpret_cast<u32x4_v*>(&sK[(v >> 4) * KS_STRIDE + (v & 15) * 8]) = r.k[i];
    *reinterpret_cast<u32x4_v*>(&sV[(v >> 4) * VS_STRIDE + (v & 15) * 8]) = r.v[i];
  }
}

// Softmax of one tile's scores s (in place: s becomes p), in the exp2 domain:
// p = 2^(s * sc2 - m) with sc2 = sm_scale * log2(e) and m the row's reference maximum in
// the same units. The reference maximum is lazy: it moves to the tile's maximum only when
// that exceeds it by more than LAZY_T, so p <= 2^LAZY_T and most tiles leave it (and the
// accumulator) alone. Every decision is per row (per lane group), so a row's bits depend
// on its own scores only. MASK: apply causality and row validity (keys beyond the row's
// position give p = 0). Returns the accumulator's rescale factor (exactly 1 when the
// reference maximum stays).
template <bool MASK>
__device__ __forceinline__ float softmax_tile(float (&s)[16], RowState& st, const Ctx& c, int t0,
                                              float sc2) {
  bool vis[16];
  float tmax = NEG_BIG;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if constexpr (MASK) {
      const int key = t0 + 32 * (i >> 3) + 8 * c.g + (i & 7);
      vis[i] = (key <= c.q_abs) & c.row_ok;
      tmax = fmaxf(tmax, vis[i] ? s[i] : NEG_BIG);
    } else {
      tmax = fmaxf(tmax, s[i]);
    }
  }
  tmax = pair16_max(tmax);
  tmax = pair32_max(tmax);
  const float mc = tmax * sc2;
  const float m_used = mc > st.m + LAZY_T ? mc : st.m;
  const float rescale = exp2_fast(st.m - m_used);
  float psum = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float p = exp2_fast(__builtin_fmaf(s[i], sc2, -m_used));
    if constexpr (MASK) s[i] = vis[i] ? p : 0.0f;
    else s[i] = p;
    psum += s[i];
  }
  psum = pair16_sum(psum);
  psum = pair32_sum(psum);
  st.l = __builtin_fmaf(st.l, rescale, psum);
  st.m = m_used;
  return rescale;
}

// p of a tile as the PV product's B operand (p is finite: exp of a finite difference, or 0).
__device__ __forceinline__ void pack_p(bf16x8_v (&pf)[2], const float (&s)[16]) {
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    uint4 u;
    u.x = pack_bf16x2(s[8 * kb + 0], s[8 * kb + 1]);
    u.y = pack_bf16x2(s[8 * kb + 2], s[8 * kb + 3]);
    u.z = pack_bf16x2(s[8 * kb + 4], s[8 * kb + 5]);
    u.w = pack_bf16x2(s[8 * kb + 6], s[8 * kb + 7]);
    pf[kb] = __builtin_bit_cast(bf16x8_v, u);
  }
}

// x * 1 == x: the rescale is skipped (same bits) unless some row of the wave moved its
// reference maximum.
__device__ __forceinline__ void apply_rescale(RowState& st, float rescale) {
  if (__builtin_amdgcn_ballot_w64(rescale != 1.0f) != 0) {
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      st.acc[db][0] *= rescale;
      st.acc[db][1] *= rescale;
      st.acc[db][2] *= rescale;
      st.acc[db][3] *= rescale;
    }
  }
}

// The 64-key tile starting at absolute key t0, already in LDS, folded into `st` (online
// softmax).
__device__ __forceinline__ void tile_math(RowState& st, const Ctx& c, int t0,
                                          const bf16x8_v (&qf)[4], float sc2,
                                          const bf16_t* sK, const bf16_t* sV) {
  // S^T blocks: lane holds logits of its query for keys 8g..8g+7 (s[0..7]) and
  // 32+8g..32+8g+7 (s[8..15]). MFMA row m of key block j holds key
  // 32*(j/2) + 8*(m/4) + 4*(j%2) + m%4.
  const int key_a0 = 8 * (c.r >> 2) + (c.r & 3);
  float s[16];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int key = 32 * (j >> 1) + 4 * (j & 1) + key_a0;
    f32x4_v st4 = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const bf16x8_v kf = *reinterpret_cast<const bf16x8_v*>(&sK[key * KS_STRIDE + 32 * ks + 8 * c.g]);
      st4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[ks], st4, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) s[4 * j + i] = st4[i];
  }

  // `full` (wave-uniform): every row of the wave sees every key of the tile, so no mask.
  const float rescale = t0 + BN - 1 <= c.q_min ? softmax_tile<false>(s, st, c, t0, sc2)
                                              : softmax_tile<true>(s, st, c, t0, sc2);

  bf16x8_v pf[2];
  pack_p(pf, s);
  apply_rescale(st, rescale);
#pragma unroll
  for (int db = 0; db < 8; ++db) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      // A = V^T rows 16 db + r (dims), columns 32 kb + 8 g .. +7 (keys): lane s of a group
      // addresses key 32 kb + 8 g + s / 4 (+ 4), dims 16 db + 4 (s % 4) .. +3.
      const bf16_t* vb = &sV[(32 * kb + 8 * c.g + (c.r >> 2)) * VS_STRIDE + 16 * db + 4 * (c.r & 3)];
      const s16x4_v lo = ld_tr16(vb);
      const s16x4_v hi = ld_tr16(vb + 4 * VS_STRIDE);
      const bf16x8_v vf = __builtin_bit_cast(
          bf16x8_v, static_cast<s16x8_v>(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
      st.acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[kb], st.acc[db], 0, 0, 0);
    }
  }
}

// Keys [t_begin, t_end) of one split (t_begin = split start, at most KSPLIT keys) folded
// into `st` tile by tile, with the next tile's loads in flight during each tile's math.
// (Issuing all of the split's tile loads up front measured slower on the verify fan-out:
// 20.0 -> 21.6 us per layer.)
__device__ __forceinline__ void run_tiles(RowState& st, const Ctx& c, int t_begin, int t_end,
                                          const bf16x8_v (&qf)[4], float sc2, bf16_t* sK,
                                          bf16_t* sV, int32_t* s_idx) {
  if (t_begin >= t_end) return;
  __syncthreads();  // previous split's tiles done with s_idx
  stage_slots(s_idx, c, t_begin);
  __syncthreads();
  TileRegs r;
  load_tile(r, c, s_idx, 0);
  int t0 = t_begin;
  for (; t0 + BN < t_end; t0 += BN) {
    __syncthreads();  // previous tile's math done with the LDS tiles
    store_tile(r, c, sK, sV);
    __syncthreads();
    load_tile(r, c, s_idx, t0 + BN - t_begin);
    tile_math(st, c, t0, qf, sc2, sK, sV);
  }
  __syncthreads();
  store_tile(r, c, sK, sV);
  __syncthreads();
  // The last tile may lie past the wave's last row. It is then left out, as in the prefill
  // kernel: it would add p = 0 times its values, which is NaN where a hidden value is not
  // finite. (A test on every tile instead: 17.7 -> 18.0 us a verify layer's attention.)
  if (t0 <= c.q_max) tile_math(st, c, t0, qf, sc2, sK, sV);
}

// part_* layout: [split][total_q][HQ]; part_a holds the unnormalised accumulator
// (128 dims), part_ml = (m, l). Lane holds dims 16*db + 4*g .. +3 of its row.
__global__ void __launch_bounds__(256) extend_fanout_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ qo_indptr,
    const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_indices,
    int num_q_heads, int num_kv_heads, int64_t num_slots, float sm_scale, int mtiles,
    int64_t total_q, float* __restrict__ part_a,
    float* __restrict__ part_ml, int32_t* __restrict__ part_n) {
  __shared__ __align__(16) bf16_t sK[BN * KS_STRIDE];
  __shared__ __align__(16) bf16_t sV[BN * VS_STRIDE];
  __shared__ int32_t s_idx[KSPLIT];

  const int b = blockIdx.x;
  const int h_kv = blockIdx.y;
  const int mtile = static_cast<int>(blockIdx.z) % mtiles;
  const int split = static_cast<int>(blockIdx.z) / mtiles;

  Ctx c;
  c.tid = threadIdx.x;
  c.wave = c.tid >> 6;
  c.lane = c.tid & 63;
  c.r = c.lane & 15;
  c.g = c.lane >> 4;

  const int q_start = qo_indptr[b];
  const int extend_len = qo_indptr[b + 1] - q_start;
  if (mtile * BQ >= extend_len) return;
  const int kv_start = kv_indptr[b];
  const int kv_len = kv_indptr[b + 1] - kv_start;
  const int prefix = kv_len - extend_len;
  if (prefix < 0) return;  // malformed batch: the kv range must cover the extend tokens

  const int hq = h_kv * 2 + (c.wave >> 1);
  const int qr = mtile * BQ + 16 * (c.wave & 1) + c.r;  // extend-local query row of this lane
  c.row_ok = qr < extend_len;
  c.q_abs = prefix + qr;
  const int w_row = mtile * BQ + 16 * (c.wave & 1);
  c.q_min = prefix + w_row;  // the wave's first row, and its last one (-1: no rows)
  c.q_max = __builtin_amdgcn_readfirstlane(
      w_row < extend_len ? prefix + min(extend_len, w_row + 16) - 1 : -1);
  const float sc2 = sm_scale * LOG2E;
  c.k_cache = k_cache;
  c.v_cache = v_cache;
  c.idx = kv_indices + kv_start;
  c.row_stride = static_cast<int64_t>(num_kv_heads) * D;
  c.num_slots = num_slots;
  c.kv_len = kv_len;
  c.h_kv = h_kv;

  const int last_row = min(extend_len, (mtile + 1) * BQ) - 1;
  const int visible_end = min(kv_len, prefix + last_row + 1);
  const int nsplits = ceil_div(visible_end, KSPLIT);
  if (split >= nsplits) return;  // the merge never reads this split

  // q fragments (B operand of S^T = K Q^T): row qr, dims 32*ks + 8*g .. +7.
  bf16x8_v qf[4];
  {
    const bf16_t* qp = q + (static_cast<int64_t>(q_start + (c.row_ok ? qr : 0)) * num_q_heads + hq) * D;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      qf[ks] = *reinterpret_cast<const bf16x8_v*>(qp + 32 * ks + 8 * c.g);
      if (!c.row_ok) qf[ks] = bf16x8_v{};
    }
  }

  const int64_t prow = static_cast<int64_t>(q_start + (c.row_ok ? qr : 0)) * num_q_heads + hq;
  RowState st;
  fresh(st);
  run_tiles(st, c, split * KSPLIT, min(visible_end, (split + 1) * KSPLIT), qf, sc2, sK,
            sV, s_idx);
  if (!c.row_ok) return;
  const int64_t pr = static_cast<int64_t>(split) * total_q * num_q_heads + prow;
  float* pa = part_a + pr * D;
#pragma unroll
  for (int db = 0; db < 8; ++db)
    *reinterpret_cast<f32x4_v*>(pa + 16 * db + 4 * c.g) = st.acc[db];
  if (c.g == 0) {
    part_ml[2 * pr] = st.m;
    part_ml[2 * pr + 1] = st.l;
    if (split == 0) part_n[prow] = nsplits;
  }
}

// ---- one workgroup per query tile: prefill, large decode-through-extend batches -----------
//
// Workgroup = (request, kv head, 8 NW query positions), NW waves; wave w: head w / (NW / 2),
// one block of 16 query rows. The splits are walked in order with the tile math of the kernel
// above (the same operations on the same values, so the same bits).
//
// What bounds it is instruction issue: a tile costs a wave 32 MFMAs (8 issue cycles each of
// their 16) and 16 scores per lane through fma, exp, sum and pack, and everything else it
// does per tile comes on top. So K and V are DMAed into two LDS buffers (no staging
// registers, no LDS writes by the waves), the next tile in flight during a tile's math, with
// one barrier per tile; the swizzled rows need no padding and little addressing; and a row's
// 128 divisions share one reciprocal. 4 x 2048 tokens 162 -> 136 us (NW = 4) / 129 (NW = 8),
// 1 x 2048 55 -> 50, 8420 ragged tokens 174 -> 154 / 138, 200 decode rows 168 -> 153.
// Measured and not taken: softmax interleaved with the next tile's S MFMAs over four-deep
// rings (141), two row blocks per wave (122, but 90 for 1 x 2048), six waves (173).
//
// LDS tiles are 64 rows of 256 bytes; 16-byte piece p of key's row sits at p ^ swz(key): over
// the 16 keys of a fragment or transpose read swz takes 16 values.
__device__ __forceinline__ int swz(int key) { return (key & 3) | (((key >> 3) & 3) << 2); }

// Lane l's 16 bytes at its address -> LDS byte lds + 16 l.
__device__ __forceinline__ void dma16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds)
               : "memory", "m0");
}
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off),
               "s"(base), "s"(lds)
               : "memory", "m0");
}

constexpr int kTileBytes = BN * D * 2;  // one K or V tile

// OFF32: the pool is smaller than 4 GiB, so 32-bit offsets address it.
template <int NW, bool OFF32>
__global__ void __launch_bounds__(NW * 64, NW / 2) extend_prefill_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ qo_indptr,
    const int32_t* __restrict__ kv_indptr, const int32_t* __restrict__ kv_indices,
    int batch, int num_q_heads, int num_kv_heads, int64_t num_slots, float sm_scale, int mtiles,
    bf16_t* __restrict__ o) {
  extern __shared__ __align__(1024) char lds[];  // [2][K tile, V tile]
  constexpr int ROWS = 8 * NW;  // query positions of the workgroup
  // (The grid's padding returns with the empty tiles: a branch of its own before the loads of
  // the indices cost every workgroup their latency, 512 x 16 tokens 35.1 -> 35.7 us.)
  const int b = min(static_cast<int>(blockIdx.x), batch - 1);
  const int h_kv = blockIdx.y;
  // Late query tiles walk the most keys: dispatch them first.
  const int mtile = mtiles - 1 - static_cast<int>(blockIdx.z);
  const int q_start = qo_indptr[b];
  const int extend_len = qo_indptr[b + 1] - q_start;
  if (mtile * ROWS >= extend_len || static_cast<int>(blockIdx.x) >= batch) return;
  const int kv_start = kv_indptr[b];
  const int kv_len = kv_indptr[b + 1] - kv_start;
  const int prefix = kv_len - extend_len;
  if (prefix < 0) return;  // malformed batch: the kv range must cover the extend tokens

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int hq = h_kv * 2 + wave / (NW / 2);
  const int w_row = mtile * ROWS + 16 * (wave % (NW / 2));  // the wave's first query row
  const int qr = w_row + (lane & 15);
  const bool row_ok = qr < extend_len;
  const int64_t prow = static_cast<int64_t>(q_start + (row_ok ? qr : 0)) * num_q_heads + hq;
  bf16x8_v qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    qf[ks] = *reinterpret_cast<const bf16x8_v*>(q + prow * D + 32 * ks + 8 * (lane >> 4));
    if (!row_ok) qf[ks] = bf16x8_v{};
  }
  const float sc2 = sm_scale * LOG2E;
  const int last_row = min(extend_len, (mtile + 1) * ROWS) - 1;
  const int ntiles = ceil_div(min(kv_len, prefix + last_row + 1), BN);
  const int w_first = prefix + w_row;  // the wave's first and last positions
  const int w_last = prefix + min(extend_len, w_row + 16) - 1;

  // A wave loads KP pieces (4 keys, 1 KB) of the K tile and of the V tile, lane l key l / 16 of
  // the piece; K and V rows share their offsets. A tile's slots are read one tile ahead.
  constexpr int KP = 16 / NW;
  const int32_t* idx = kv_indices + kv_start;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char_t)lds));
  const uint32_t max_slots = static_cast<uint32_t>(min<int64_t>(num_slots, 0x7fffffff));
  const int row_bytes = num_kv_heads * D * 2;
  const char* kbase = reinterpret_cast<const char*>(k_cache + h_kv * D);
  const char* vbase = reinterpret_cast<const char*>(v_cache + h_kv * D);
  struct Slots {
    uint32_t s[KP];
  };
  auto load_slots = [&](int tile) {
    Slots v;
    const int key0 = tile * BN + 4 * wave + (lane >> 4);
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int key = key0 + 4 * NW * i;
      v.s[i] = key < kv_len ? idx[key] : 0;
    }
    return v;
  };
  auto load_tile_dma = [&](const Slots& v, int buf) {
    int l = lane;  // opaque: per-lane constants are not kept in registers between tiles
    asm volatile("" : "+v"(l));
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int key = 4 * (wave + NW * i) + (l >> 4);
      const uint32_t slot = v.s[i] < max_slots ? v.s[i] : 0u;
      const uint32_t piece = 16 * ((l & 15) ^ swz(key));
      const uint32_t dst = lds0 + buf * 2 * kTileBytes + 1024u * (wave + NW * i);
      if constexpr (OFF32) {  // fewer than 2^24 slots: rows are at least 256 bytes
        const uint32_t off = __umul24(slot, row_bytes) + piece;
        dma16(kbase, off, dst);
        dma16(vbase, off, dst + kTileBytes);
      } else {
        const int64_t off = static_cast<int64_t>(slot) * row_bytes + piece;
        dma16(kbase + off, dst);
        dma16(vbase + off, dst + kTileBytes);
      }
    }
  };

  RowState run, st;
  fresh(run);
  fresh(st);
  // One tile's math out of LDS buffer `buf`. MASK: some key is hidden from some row.
  auto tile = [&](auto mask, int t0, int buf) {
    int l = lane;
    asm volatile("" : "+v"(l));
    const int r = l & 15, g = l >> 4;
    const int key_a0 = 8 * (r >> 2) + (r & 3);
    const uint32_t ka = lds0 + buf * 2 * kTileBytes + key_a0 * 256 + 16 * (g ^ swz(key_a0));
    f32x4_v s4[4];
#pragma unroll
    for (int i = 0; i < 16; ++i) {  // key block j, k-step ks
      const int j = i & 3, ks = i >> 2;
      const bf16x8_v kf = *(__attribute__((address_space(3))) const bf16x8_v*)(
          (ka ^ (64u * ks)) + 256 * (32 * (j >> 1) + 4 * (j & 1)));
      s4[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          kf, qf[ks], ks == 0 ? f32x4_v{0.0f, 0.0f, 0.0f, 0.0f} : s4[j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    Ctx c;
    c.g = g;
    c.q_abs = w_first + r;
    c.row_ok = row_ok;
    float s[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = s4[i >> 2][i & 3];
    const float rescale = softmax_tile<decltype(mask)::value>(s, st, c, t0, sc2);
    bf16x8_v pf[2];
    pack_p(pf, s);
    __builtin_amdgcn_sched_barrier(0);
    apply_rescale(st, rescale);
    const int key_v = 8 * g + (r >> 2);
    const uint32_t va = lds0 + (buf * 2 + 1) * kTileBytes + key_v * 256 +
                        16 * (((r & 3) >> 1) ^ swz(key_v)) + 8 * (r & 1);
#pragma unroll
    for (int i = 0; i < 16; ++i) {  // dim block db, key half kb
      const int db = i & 7, kb = i >> 3;
      typedef __attribute__((address_space(3))) s16x4_v* tr_ptr_t;
      const uint32_t p = (va ^ (32u * db)) + 8192 * kb;
      const s16x4_v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)p);
      const s16x4_v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(p + 1024));
      const bf16x8_v vf = __builtin_bit_cast(
          bf16x8_v, static_cast<s16x8_v>(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
      st.acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[kb], st.acc[db], 0, 0, 0);
    }
  };

  load_tile_dma(load_slots(0), 0);
  Slots slots = load_slots(1);
  for (int t = 0; t < ntiles; ++t) {
    // Tile t has landed and every wave is done with the other buffer.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 < ntiles) {
      load_tile_dma(slots, (t + 1) & 1);
      slots = load_slots(t + 2);
    }
    const int t0 = t * BN;
    if (t0 + BN - 1 <= w_first && w_row < extend_len) {
      tile(std::false_type{}, t0, t & 1);
    } else if (t0 <= w_last && w_row < extend_len) {
      tile(std::true_type{}, t0, t & 1);
    }
    if ((t & 3) == 3 || t + 1 == ntiles) {  // the split's end
      fold(run, st.m, st.l, st.acc);
      fresh(st);
    }
  }
  if (row_ok) store_row(o + prow * D, run, lane >> 4);
}

// Fold the fanned-out split states of every (query row, head) item in split order: one
// wave per item (global item = row * HQ + head), lane l owning dims 2l and 2l + 1. fold()
// is elementwise with per-row scalars, so any assignment of dims to lanes computes the
// same bits as the attention kernel's own layout. The item's split count (written by the
// attention kernel's split-0 workgroup) is loaded first, then up to MERGE_CHUNK of its
// splits' states together, then folded.
constexpr int MERGE_CHUNK = 16;

__global__ void __launch_bounds__(256) extend_merge_kernel(
    int64_t items, int splits, const float* __restrict__ part_a,
    const float* __restrict__ part_ml, const int32_t* __restrict__ part_n,
    bf16_t* __restrict__ o) {
  const int lane = threadIdx.x & 63;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (item >= items) return;  // whole waves: no barrier below
  // Only the item's own splits are loaded: the grid's split count follows the pass's
  // key-length bucket (up to twice the longest sequence), and the splits past the item's
  // own hold nothing it reads (measured: verify pass, 4 x 32 rows over 2k keys, 22.1 ->
  // 20.5 us per layer with the fan-out).
  const int nsplits = min(part_n[item], splits);
  float m = NEG_BIG, l = 0.0f;
  float2 acc = make_float2(0.0f, 0.0f);
  for (int c0 = 0; c0 < nsplits; c0 += MERGE_CHUNK) {
    const int n = min(MERGE_CHUNK, nsplits - c0);
    float2 a[MERGE_CHUNK];
    float sm[MERGE_CHUNK], sl[MERGE_CHUNK];
#pragma unroll
    for (int sp = 0; sp < MERGE_CHUNK; ++sp) {
      if (sp < n) {
        const int64_t pr = static_cast<int64_t>(c0 + sp) * items + item;
        a[sp] = reinterpret_cast<const float2*>(part_a + pr * D)[lane];
        sm[sp] = part_ml[2 * pr];
        sl[sp] = part_ml[2 * pr + 1];
      }
    }
#pragma unroll
    for (int sp = 0; sp < MERGE_CHUNK; ++sp) {
      if (sp < n) {  // fold() on two dims
        const FoldScale f = fold_scale(m, sm[sp]);
        l = fold_elem(l, sl[sp], f);
        acc.x = fold_elem(acc.x, a[sp].x, f);
        acc.y = fold_elem(acc.y, a[sp].y, f);
        m = f.mn;
      }
    }
  }
  const float y = 1.0f / l;
  reinterpret_cast<uint32_t*>(o + item * D)[lane] = pack_bf16x2(div_row(acc.x, l, y), div_row(acc.y, l, y));
}

// Fan the splits out when the grid would leave most CUs idle.
constexpr int kFanoutBelowWg = 512;
// Query positions of a prefill workgroup. The 64-row ones (8 waves) load each key tile half as
// often, but a causal grid ends on its longest ones, and a short request leaves some of their
// waves idle. They win once the rows that exist (total_q, not batch x longest) fill 2.6 of
// them per CU of 256 and at least half of the batch x longest rows exist. 32- vs 64-row, us:
// 1 x 4096 131 vs 152, 2 x 2304 78 vs 85, 1 x 5120 173 vs 180, 3 x 1800 77 vs 70, 2 x 3000
// 127 vs 113, 4 x 2048 122 vs 116, 1 x 8192 416 vs 380; 12 x 512 36 vs 39, 16 x 512 47 vs 49,
// 6 x 1024 54 vs 53; 3000 + 40 x 33 80 vs 120, 2048 + 15 x 16 54 vs 80, 1024 + 60 x 120 39 vs
// 45, 5000 + 3000 229 vs 204.
constexpr int64_t kWideWg = 672;
constexpr int kWideMinLen = 1024;
int prefill_rows(int batch, int64_t total_q, int num_kv_heads, int max_extend_len) {
  const bool uniform = 2 * total_q >= static_cast<int64_t>(batch) * max_extend_len;
  return max_extend_len >= kWideMinLen && uniform &&
                 num_kv_heads * ((total_q + 63) / 64) >= kWideWg
             ? 64
             : 32;
}

}  // namespace
}  // namespace sid

using namespace sid;

extern "C" int sid_extend_attention_query_rows(int batch, int64_t total_q, int num_kv_heads,
                                               int max_extend_len) {
  return prefill_rows(batch, total_q, num_kv_heads, max_extend_len);
}

extern "C" int64_t sid_extend_attention_workspace_bytes(int batch, int64_t total_q,
                                                        int num_q_heads, int num_kv_heads,
                                                        int max_extend_len, int max_kv_len) {
  if (batch <= 0 || total_q <= 0 || max_extend_len <= 0 || max_kv_len <= 0) return 0;
  const int64_t mtiles = ceil_div(max_extend_len, BQ);
  if (static_cast<int64_t>(batch) * num_kv_heads * mtiles >= kFanoutBelowWg) return 0;
  const int64_t splits = ceil_div(max_kv_len, KSPLIT);
  // per (split, row, head): 128 accumulator floats + (m, l); per (row, head): split count
  return (splits * (D + 2) + 1) * total_q * num_q_heads * static_cast<int64_t>(sizeof(float));
}

extern "C" int sid_extend_attention_fwd(const void* q, const void* k_cache, const void* v_cache,
                                        const int32_t* qo_indptr, const int32_t* kv_indptr,
                                        const int32_t* kv_indices, int batch, int64_t total_q,
                                        int num_q_heads, int num_kv_heads, int head_dim,
                                        int64_t num_slots, int max_extend_len, int max_kv_len,
                                        float sm_scale, void* workspace, int64_t workspace_bytes,
                                        void* o, void* stream) {
  SID_REQUIRE(batch >= 0 && total_q >= 0, "extend_attention: negative size");
  if (batch == 0 || total_q == 0 || max_extend_len <= 0) return SID_OK;
  SID_REQUIRE(q && k_cache && v_cache && qo_indptr && kv_indptr && kv_indices && o,
              "extend_attention: null pointer");
  SID_REQUIRE(head_dim == D, "extend_attention: head_dim must be %d, got %d", D, head_dim);
  SID_REQUIRE(num_kv_heads > 0 && num_q_heads == 2 * num_kv_heads,
              "extend_attention: expected 2 q heads per kv head (got %d q, %d kv)", num_q_heads,
              num_kv_heads);
  SID_REQUIRE(num_slots > 0, "extend_attention: empty KV pool");
  SID_REQUIRE(batch <= 65535 && num_kv_heads <= 65535, "extend_attention: grid too large");
  const int mtiles = ceil_div(max_extend_len, BQ);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t need = sid_extend_attention_workspace_bytes(batch, total_q, num_q_heads,
                                                           num_kv_heads, max_extend_len,
                                                           max_kv_len);
  const bool fanout = need > 0 && workspace != nullptr && workspace_bytes >= need;
  if (fanout) {
    const int splits = ceil_div(max_kv_len, KSPLIT);
    SID_REQUIRE(static_cast<int64_t>(mtiles) * splits <= 65535, "extend_attention: grid too large");
    const int64_t items = total_q * num_q_heads;
    float* pa = static_cast<float*>(workspace);
    float* pml = pa + static_cast<int64_t>(splits) * items * D;
    int32_t* pn = reinterpret_cast<int32_t*>(pml + static_cast<int64_t>(splits) * items * 2);
    hipLaunchKernelGGL(extend_fanout_kernel, dim3(batch, num_kv_heads, mtiles * splits),
                       dim3(256), 0, s, (const bf16_t*)q, (const bf16_t*)k_cache,
                       (const bf16_t*)v_cache, qo_indptr, kv_indptr, kv_indices, num_q_heads,
                       num_kv_heads, num_slots, sm_scale, mtiles, total_q, pa, pml, pn);
    int rc = check_launch("extend_attention");
    if (rc != SID_OK) return rc;
    const int64_t groups = (items + 3) / 4;
    SID_REQUIRE(groups < (1ll << 31), "extend_attention: too many rows for the merge");
    hipLaunchKernelGGL(extend_merge_kernel, dim3((unsigned)groups), dim3(256), 0, s, items,
                       splits, pa, pml, pn, (bf16_t*)o);
    return check_launch("extend_attention merge");
  }
  SID_REQUIRE(mtiles <= 65535, "extend_attention: grid too large");
  // Request b's workgroups are `batch` ids apart. Where only some requests reach the late tiles
  // an even distance puts a long request's on few XCDs and CUs, so the grid then has an odd
  // one (2048 + 15 x 16 445 -> 54 us, 31 x 1 + 4000 3160 -> 126, 5000 + 3000 268 -> 209; full
  // batches keep theirs: 12 x 512 36 vs 38 padded, 8 x 1024 69 vs 72).
  const bool ragged = 8 * total_q < 7 * static_cast<int64_t>(batch) * max_extend_len;
  auto prefill = [&](auto kern, int nw) {
    const int mt = ceil_div(max_extend_len, 8 * nw);
    hipLaunchKernelGGL(kern, dim3(ragged ? batch | 1 : batch, num_kv_heads, mt), dim3(nw * 64),
                       4 * kTileBytes, s, (const bf16_t*)q, (const bf16_t*)k_cache,
                       (const bf16_t*)v_cache, qo_indptr, kv_indptr, kv_indices, batch, num_q_heads,
                       num_kv_heads, num_slots, sm_scale, mt, (bf16_t*)o);
  };
  const bool off32 = num_slots * num_kv_heads * D * 2 < (1ll << 32);
  if (prefill_rows(batch, total_q, num_kv_heads, max_extend_len) == 64) {
    off32 ? prefill(extend_prefill_kernel<8, true>, 8) : prefill(extend_prefill_kernel<8, false>, 8);
  } else {
    off32 ? prefill(extend_prefill_kernel<4, true>, 4) : prefill(extend_prefill_kernel<4, false>, 4);
  }
  return check_launch("extend_attention");
}
