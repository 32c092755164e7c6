// Decode-step GEMMs y = x @ w^T on gfx950 bf16 MFMA (v_mfma_f32_16x16x32_bf16).
//
// Reduction order (the determinism contract of sid_linear): K is cut into
// 256-wide chunks; chunk c is accumulated from zero by 8 MFMA k-steps of 32
// in increasing k, and the output is the left fold c0 + c1 + c2 + ... in
// increasing chunk order, then + bias, then one rounding to bf16. That order
// depends only on K, never on M, on the tile a row lands in, or on which
// kernel folds the chunks, so a row's bits are identical whether it is
// computed alone or inside any batch (the batch-invariance property that
// sid/kernels/matmul_persistent.py:1-9 buys with a separate slow kernel is
// here true of the one fast kernel).
//
// Kernels (all with that order):
//   * linear_chunk_kernel: split-K partials for decode-sized M (sid_linear_partials): one
//     256-wide chunk of 64 columns per 4-wave workgroup, x chunk staged in LDS, weights
//     streamed straight into MFMA B operands; writes partials[c][m][n], which the consumer
//     kernel folds in chunk order (norm_rope.hip). No cross-workgroup synchronisation.
//   * linear_tile_kernel: direct y (prefill, and decode / verify rows past the split-K cuts),
//     persistent tiles of four shapes; also gate_up with the SwiGLU epilogue and the lm_head
//     of more than 64 rows with the argmax or sampler epilogue;
//   * linear_kernel: direct y (or greedy argmax) for rows past the tile kernel's 32-bit offsets;
//   * linear_stream_kernel: lm_head-shaped N (persistent grid, x staged once per CU), with
//     an optional fused greedy argmax.
#include "common.h"

#include <algorithm>

namespace sid {
namespace {

constexpr int KC = 256;      // chunk width of the canonical reduction order
constexpr int KSTEP = 32;    // MFMA 16x16x32 k-step
constexpr int NSTEP = KC / KSTEP;
constexpr int MROWS = 64;    // rows per row group (4 MFMA row blocks)
constexpr int NTILE_MIN = 64;  // column granularity (4 waves x 16); N must be a multiple
constexpr int XS = KC + 8;   // LDS row stride of the staged x chunk (bf16 elements)

__device__ __forceinline__ bf16x8_v ld_frag(const bf16_t* p) {
  return *reinterpret_cast<const bf16x8_v*>(p);
}

// x chunk in registers: thread t holds 16-byte vector t%32 of rows t/32 + 2*NW*i. The
// row-count test is written per pass (i < rows16 / (2*NW), uniform over the workgroup
// because rows16 is a multiple of 16 and 2*NW divides 16 or is 32), which keeps the 8 vectors in registers: a per-lane test
// here, or HIP's struct-wrapped uint4 as the element type, made the compiler demote them
// to scratch and serialise every load (native vector types stay in registers).
template <int NW>
__device__ __forceinline__ void load_x(bf16x8_v (&xv)[8], const bf16_t* __restrict__ x, int64_t ldx,
                                       int64_t m0, int64_t M, int rows16, int64_t k0) {
  constexpr int RPP = NW * 2;  // rows per pass: 32 threads per row
  const int tid = threadIdx.x;
  const int vec = tid & 31;
  const int passes = rows16 / RPP;
#pragma unroll
  for (int i = 0; i < 64 / RPP; ++i) {
    if (i < passes) {
      const int row = (tid >> 5) + RPP * i;
      const int64_t gr = min<int64_t>(m0 + row, M - 1);  // rows >= M are clamped and discarded
      xv[i] = ld_frag(x + gr * ldx + k0 + vec * 8);
    }
  }
}

template <int NW>
__device__ __forceinline__ void store_x(bf16_t* sx, const bf16x8_v (&xv)[8], int rows16) {
  constexpr int RPP = NW * 2;
  const int tid = threadIdx.x;
  const int vec = tid & 31;
  const int passes = rows16 / RPP;
#pragma unroll
  for (int i = 0; i < 64 / RPP; ++i) {
    if (i < passes) {
      const int row = (tid >> 5) + RPP * i;
      *reinterpret_cast<bf16x8_v*>(&sx[row * XS + vec * 8]) = xv[i];
    }
  }
}

__device__ __forceinline__ void load_w(bf16x8_v (&wf)[NSTEP], const bf16_t* wrow, int64_t k0) {
#pragma unroll
  for (int s = 0; s < NSTEP; ++s) wf[s] = ld_frag(wrow + k0 + KSTEP * s);
}

// One chunk of one wave's 16 columns: acc[mb] = sum over the chunk, from zero.
__device__ __forceinline__ void chunk_mfma(f32x4_v (&acc)[4], const bf16x8_v (&wf)[NSTEP],
                                           const bf16_t* sx, int mbs, int r, int g) {
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) acc[mb] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < NSTEP; ++s) {
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      if (mb < mbs) {
        const bf16x8_v af =
            *reinterpret_cast<const bf16x8_v*>(&sx[(16 * mb + r) * XS + KSTEP * s + 8 * g]);
        acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf[s], acc[mb], 0, 0, 0);
      }
    }
  }
}

// Greedy argmax order over (value, column), torch's: larger value, then smaller index; NaN
// above everything, first NaN wins. A total order, so a maximum over any split of the
// columns into candidates, reduced in any order, is the same (value, column).
__device__ __forceinline__ bool argmax_better(float v, int i, float bv, int bi) {
  const bool vn = v != v;
  const bool bn = bv != bv;
  if (vn || bn) {
    if (vn && bn) return i < bi;
    return vn;
  }
  return v > bv || (v == bv && i < bi);
}

// Direct y = x w^T (+ bias) for one 64-row group and 16*NW columns: every chunk in order,
// the next chunk's weights and x prefetched into registers during the current chunk's
// MFMAs. NW waves share one staged x chunk. (Only for sizes that tiles_fit refuses.)
// AM: also each row's best (bf16-rounded logit, column) of the wave's 16 columns, to
// best_val / best_idx [wave of the grid][M]; y may then be null.
template <int NW, bool AM>
__global__ void __launch_bounds__(NW * 64) linear_kernel(
    const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w,
    const bf16_t* __restrict__ bias, void* __restrict__ y, int64_t M, int64_t N, int64_t K,
    int out_fp32, float* __restrict__ best_val, int* __restrict__ best_idx) {
  __shared__ __align__(16) bf16_t sx[MROWS * XS];

  const int nchunks = static_cast<int>(K / KC);
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * (16 * NW);
  const int64_t m0 = static_cast<int64_t>(blockIdx.z) * MROWS;
  const int mrows = static_cast<int>(min<int64_t>(MROWS, M - m0));
  const int mbs = (mrows + 15) >> 4;
  const int rows16 = mbs * 16;
  const bf16_t* wrow = w + (n0 + 16 * wave + r) * K + 8 * g;
  const int col = 16 * wave + r;

  const int c_begin = 0;
  const int c_end = nchunks;

  bf16x8_v wf[NSTEP];
  bf16x8_v xr[8];
  load_w(wf, wrow, static_cast<int64_t>(c_begin) * KC);
  load_x<NW>(xr, x, ldx, m0, M, rows16, static_cast<int64_t>(c_begin) * KC);

  f32x4_v total[4];
  for (int c = c_begin; c < c_end; ++c) {
    if (c != c_begin) __syncthreads();  // previous chunk's x fully consumed
    store_x<NW>(sx, xr, rows16);
    __syncthreads();
    bf16x8_v wcur[NSTEP];
#pragma unroll
    for (int s = 0; s < NSTEP; ++s) wcur[s] = wf[s];
    if (c + 1 < c_end) {  // prefetch the next chunk while this one computes
      load_w(wf, wrow, static_cast<int64_t>(c + 1) * KC);
      load_x<NW>(xr, x, ldx, m0, M, rows16, static_cast<int64_t>(c + 1) * KC);
    }
    f32x4_v acc[4];
    chunk_mfma(acc, wcur, sx, mbs, r, g);
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      if (c == c_begin) {
        total[mb] = acc[mb];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) total[mb][i] += acc[mb][i];
      }
    }
  }

  // Lane holds rows 16*mb + 4*g + i of column `col`.
  const float bv = bias != nullptr ? bf16_to_f32(bias[n0 + col]) : 0.0f;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    if (mb < mbs) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * mb + 4 * g + i;
        if (row < mrows) {
          float v = total[mb][i];
          if (bias != nullptr) v += bv;
          const int64_t off = (m0 + row) * N + n0 + col;
          if constexpr (AM) {  // (the 16 lanes of a row are active together)
            v = round_bf16(v);
            if (y != nullptr) static_cast<float*>(y)[off] = v;
            int ix = static_cast<int>(n0) + col;
#pragma unroll
            for (int mask = 1; mask < 16; mask <<= 1) {
              const float ov = lane_xor(v, mask);
              const int oi = __builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, ix);
              if (argmax_better(ov, oi, v, ix)) {
                v = ov;
                ix = oi;
              }
            }
            if (r == 0) {
              const int64_t o = (static_cast<int64_t>(blockIdx.x) * NW + wave) * M + m0 + row;
              best_val[o] = v;
              best_idx[o] = ix;
            }
          } else if (out_fp32) {
            static_cast<float*>(y)[off] = round_bf16(v);
          } else {
            static_cast<bf16_t*>(y)[off] = f32_to_bf16(v);
          }
        }
      }
    }
  }
}

// Partial mode: one 256-wide chunk per workgroup (blockIdx.y), fp32 tile written to
// partials[chunk][row][col]. MBS (16-row blocks in the row group) is a compile-time
// constant so the 8 x MBS MFMAs and their LDS reads are straight-line code; the chunk's
// MFMA sequence is chunk_mfma's, so the partials are the bits linear_kernel folds.
template <int NW, int MBS>
__global__ void __launch_bounds__(NW * 64) linear_chunk_kernel(
    const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, int64_t M, int64_t N,
    int64_t K, float* __restrict__ partials) {
  __shared__ __align__(16) bf16_t sx[MBS * 16 * XS];
  constexpr int RPP = NW * 2;  // x rows per pass: 32 threads per row
  constexpr int PASSES = (MBS * 16 + RPP - 1) / RPP;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * (16 * NW);
  const int c = blockIdx.y;
  const int64_t m0 = static_cast<int64_t>(blockIdx.z) * MROWS;
  const int mrows = static_cast<int>(min<int64_t>(MROWS, M - m0));
  const int64_t k0 = static_cast<int64_t>(c) * KC;

  bf16x8_v wf[NSTEP];
  load_w(wf, w + (n0 + 16 * wave + r) * K + 8 * g, k0);
  bf16x8_v xv[PASSES];
  const int vec = threadIdx.x & 31;
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int row = (threadIdx.x >> 5) + RPP * i;
    const int64_t gr = min<int64_t>(m0 + min(row, MBS * 16 - 1), M - 1);  // clamped, discarded
    xv[i] = ld_frag(x + gr * ldx + k0 + vec * 8);
  }
#pragma unroll
  for (int i = 0; i < PASSES; ++i) {
    const int row = (threadIdx.x >> 5) + RPP * i;
    if (row < MBS * 16) *reinterpret_cast<bf16x8_v*>(&sx[row * XS + vec * 8]) = xv[i];
  }
  __syncthreads();
  f32x4_v acc[MBS];
#pragma unroll
  for (int mb = 0; mb < MBS; ++mb) acc[mb] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < NSTEP; ++s) {
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) {
      const bf16x8_v af =
          *reinterpret_cast<const bf16x8_v*>(&sx[(16 * mb + r) * XS + KSTEP * s + 8 * g]);
      acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf[s], acc[mb], 0, 0, 0);
    }
  }
  float* dst = partials + (static_cast<int64_t>(c) * M + m0) * N + n0 + 16 * wave + r;
  if (mrows == MBS * 16) {  // full row group (uniform): unguarded stores
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[static_cast<int64_t>(16 * mb + 4 * g + i) * N] = acc[mb][i];
    }
    return;
  }
#pragma unroll
  for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * mb + 4 * g + i;
      if (row < mrows) dst[static_cast<int64_t>(row) * N] = acc[mb][i];
    }
  }
}

struct SampleStats {
  float* mx;
  float* sm;
  float* a1v;
  float* a1x;
  float* a2v;
  int* a1i;
};

__device__ __forceinline__ void softmax_merge(float& m, float& s, float om, float os) {
  const float nm = fmaxf(m, om);
  const float a = m == -INFINITY ? 0.0f : s * expf(m - nm);
  const float b = om == -INFINITY ? 0.0f : os * expf(om - nm);
  m = nm;
  s = a + b;
}

// One lane's sampler statistics over the columns it has seen (see linear_sample_kernel):
// greedy rows keep only (v1, i1) = the best (logit, column) under argmax_better.
struct SState {
  float m, s, v1, x1, v2;
  int i1;
};

__device__ __forceinline__ SState sstate_empty() {
  return SState{-INFINITY, 0.0f, -INFINITY, -INFINITY, -INFINITY, 0x7fffffff};
}

// Column `col` with bf16-rounded logit vr, for a row with temperature t and noise row hash h.
__device__ __forceinline__ void sstate_add(SState& a, float vr, int col, float t, uint32_t h) {
  if (!(t > 0.0f)) {
    if (argmax_better(vr, col, a.v1, a.i1)) {
      a.v1 = vr;
      a.i1 = col;
    }
    return;
  }
  const float xv = vr / t;
  if (xv > a.m) {
    a.s = a.s * expf(a.m - xv) + 1.0f;
    a.m = xv;
  } else {
    a.s += expf(xv - a.m);
  }
  const float xg = xv + seeded_gumbel(h, col);
  if (xg > a.v1 || (xg == a.v1 && col < a.i1)) {
    a.v2 = a.v1;
    a.v1 = xg;
    a.x1 = xv;
    a.i1 = col;
  } else {
    a.v2 = fmaxf(a.v2, xg);
  }
}

// sstate_add to the empty state (the same values without its exponential).
__device__ __forceinline__ SState sstate_first(float vr, int col, float t, uint32_t h) {
  SState a = sstate_empty();
  if (!(t > 0.0f)) {
    a.v1 = vr;
    a.i1 = col;
    return a;
  }
  const float xv = vr / t;
  const bool some = xv > -INFINITY;
  a.m = some ? xv : -INFINITY;
  a.s = some ? 1.0f : xv - xv;  // (-inf and NaN: NaN)
  const float xg = xv + seeded_gumbel(h, col);
  if (xg >= -INFINITY) {
    a.v1 = xg;
    a.x1 = xv;
    a.i1 = col;
  }
  return a;
}

// a <- a merged with b (a fixed function of the two states).
__device__ __forceinline__ void sstate_merge(SState& a, const SState& b, bool greedy) {
  if (greedy) {
    if (argmax_better(b.v1, b.i1, a.v1, a.i1)) {
      a.v1 = b.v1;
      a.i1 = b.i1;
    }
    return;
  }
  softmax_merge(a.m, a.s, b.m, b.s);
  if (b.v1 > a.v1 || (b.v1 == a.v1 && b.i1 < a.i1)) {
    a.v2 = fmaxf(a.v1, b.v2);
    a.v1 = b.v1;
    a.x1 = b.x1;
    a.i1 = b.i1;
  } else {
    a.v2 = fmaxf(a.v2, fmaxf(b.v1, b.v2));
  }
}

// Merge over the lanes that differ in the bits LO .. HI / 2 (xor butterfly; each of them ends
// with the same state).
template <int LO, int HI>
__device__ __forceinline__ void sstate_merge_xor(SState& a, bool greedy) {
  const int lane = __lane_id();
#pragma unroll
  for (int mask = LO; mask < HI; mask <<= 1) {
    SState b;
    b.m = lane_xor(a.m, mask);
    b.s = lane_xor(a.s, mask);
    b.v1 = lane_xor(a.v1, mask);
    b.x1 = lane_xor(a.x1, mask);
    b.v2 = lane_xor(a.v2, mask);
    b.i1 = __builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, a.i1);
    sstate_merge(a, b, greedy);
  }
}

__device__ __forceinline__ void sstate_store(const SampleStats& st, int64_t o, const SState& a) {
  st.mx[o] = a.m;
  st.sm[o] = a.s;
  st.a1v[o] = a.v1;
  st.a1x[o] = a.x1;
  st.a2v[o] = a.v2;
  st.a1i[o] = a.i1;
}

inline SampleStats sample_stats_at(const SampleStats& st, int64_t row) {
  return {st.mx + row, st.sm + row, st.a1v + row, st.a1x + row, st.a2v + row, st.a1i + row};
}

// Per-row inputs of a fused sampler epilogue; statistics go to st at [group][cand_rows].
struct SampleIn {
  const float* temps;
  const int64_t* seeds;
  const int64_t* positions;
  SampleStats st;
  int64_t cand_rows;
};

// ---- pipelined tile GEMM (direct projections of any M, verify passes, wide heads) ----------
//
// Persistent workgroups of WM x WN waves; wave (wm, wn) owns MB x NB MFMA blocks
// (16 MB x 16 NB outputs) of a TM x TN tile. K streams in 64-deep sub-tiles through a ring of
// ST LDS stages that buffer_load ... lds fills ST - 1 sub-tiles ahead, across tile boundaries
// too, so a tile's first loads are in flight while the previous tile is stored. One barrier
// per sub-tile: a wave that passes it has finished reading the stage about to be refilled, and
// its wait count leaves the ST - 2 later sub-tiles in flight. Between two barriers the
// fragment reads of one 32-deep k-step run beside the MFMAs of the k-step before it
// (scheduling barriers keep that order), so neither LDS nor memory latency is exposed.
//
// LDS: a stage's rows are 128 bytes (64 bf16) without padding, 16-byte piece p of row q at
// p ^ ((q >> 1) & 7): the DMA writes whole 1 KB runs (the permutation is on the global side,
// inside one 128-byte line) and the fragment reads are conflict-free (SQ_LDS_BANK_CONFLICT 512
// a 256 x 128 tile at any K, from the store staging alone). Rows past M or N are dropped by the buffer range check (zeros); their outputs are not
// stored. Weights are the MFMA's A operand, so a lane holds four consecutive columns of one
// row and a tile is stored through LDS as whole 128-byte lines.
//
// Every output element keeps the canonical order: each 256-wide chunk accumulated from zero
// by 8 MFMA k-steps in increasing k, the chunk sums left-folded in order, then + bias and one
// rounding; products commute, so the bits are linear_kernel's for any M and any tile.
//
// Bound: MFMA issue and its power (random operands run ~20% below zeros); above that the
// LDS fills, 47 bytes per clock and CU at the MFMA peak with 256 x 128 tiles. Two accumulator
// sets (the chunk's and the fold's) limit a wave to 64 x 64 outputs. Measured against the
// register-staged 128 x 128 tiles this replaced (us): 8192 x 4096 x 1024 96.4 -> 75.2,
// 8192 x 6144 x 1024 129.5 -> 95.2, 8192 x 1024 x 3072 68.3 -> 46.0 (1.12 PFLOP/s),
// 2048 x 1024 x 2048 17.9 -> 12.7, 777 x 1024 x 3072 21.4 -> 11.6; the vendor BLAS (not
// batch-invariant) takes 57.6, 98.6 and 52.5 on the first three.
//
// EPI selects the epilogue: bf16 / fp32 y (+ bias); SwiGLU; the greedy or the seeded
// sampler's statistics of the lm_head.
constexpr int BK = 64;
constexpr int SUBS = KC / BK;
constexpr int EPI_Y = 0, EPI_SWIGLU = 1, EPI_ARGMAX = 2, EPI_SAMPLE = 3;

typedef uint32_t u32x2_v __attribute__((ext_vector_type(2)));

// Lane l's 16 bytes at srd base + voff + soff (range-checked) -> LDS byte lds + 16 l.
__device__ __forceinline__ void dma16(uint32_t voff, u32x4_v srd, uint32_t soff, uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff),
      "s"(srd), "s"(soff), "s"(lds)
      : "memory", "m0");
}

// All but this wave's N newest loads have landed, its LDS reads are done, and every wave of
// the workgroup got here.
template <int N>
__device__ __forceinline__ void wait_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ u32x4_v raw_srd(const void* p, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uintptr_t>(p);
  return u32x4_v{static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32) & 0xffffu, bytes,
                 0x00020000u};
}
__device__ __forceinline__ u32x4_v pick(bool c, const u32x4_v& a, const u32x4_v& b) {
  return u32x4_v{c ? a[0] : b[0], c ? a[1] : b[1], c ? a[2] : b[2], c ? a[3] : b[3]};
}

// Output side of a launch. wide: y (and N) allow 16-byte stores. inter (SwiGLU): y is
// [M][inter] and w holds inter gate rows, then inter up rows (N = 2 inter).
struct TileOut {
  void* y;
  const bf16_t* bias;
  int out_fp32;
  int wide;
  float* best_val;
  int* best_idx;
  SampleIn sp;
};

template <int WM, int WN, int MB, int NB, int ST>
struct TileShape {
  static constexpr int NW = WM * WN;
  static constexpr int TM = WM * MB * 16;
  static constexpr int TN = WN * NB * 16;
  static constexpr int STAGE = (TM + TN) * BK * 2;
  static constexpr int SCRATCH = NW * 2048;  // epilogue: 2 KB per wave
  static constexpr int LDS = ST * STAGE + SCRATCH;
};

template <int WM, int WN, int MB, int NB, int ST, int OCC, int EPI>
__global__ void __launch_bounds__(WM * WN * 64, OCC) linear_tile_kernel(
    const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, int M, int N, int K,
    int mt, int nt, TileOut out) {
  using S = TileShape<WM, WN, MB, NB, ST>;
  constexpr int NW = S::NW, TM = S::TM, TN = S::TN, STAGE = S::STAGE;
  constexpr int PA = TM / 8 / NW, PB = TN / 8 / NW;  // 1 KB pieces a wave loads per sub-tile
  constexpr int PER = PA + PB;
  static_assert(PA * 8 * NW == TM && PB * 8 * NW == TN && NB % 2 == 0, "tile");
  static_assert(EPI != EPI_SWIGLU || (NW / 2) % NB == 0, "a wave's w pieces are all gate or all up");
  extern __shared__ __align__(1024) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int wm = wave / WN;
  const int wn = wave % WN;
  const int tiles = mt * nt;
  const int nsub = K / BK;  // a multiple of 4, at least ST - 1 (the host's choice of shape)
  const int nch = K / KC;
  const uint32_t lds0 = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));

  // Tile order: bands of 4 row tiles, rows fastest, so the tiles in flight share x and w
  // rows; XCD k (workgroups k mod 8) takes a contiguous eighth of each round of the grid.
  auto tile_mn = [&](int t, int& tm, int& tn) {
    constexpr int BAND = 4;
    const int band = t / (BAND * nt);
    const int rem = t - band * BAND * nt;
    const int rows = min(BAND, mt - band * BAND);
    tn = rem / rows;
    tm = band * BAND + rem - tn * rows;
  };
  const int grid = gridDim.x;
  int t = blockIdx.x;
  if (grid % 8 == 0) t = (blockIdx.x % 8) * (grid / 8) + blockIdx.x / 8;

  // Loads: piece p = wave + NW i is rows 8p .. 8p+7 of the stage's x (w) part, lane l row
  // l / 8, global 16-byte piece (l % 8) ^ swizzle. SwiGLU: LDS row j of the w part is, in
  // wave column block order, a gate row (first NB / 2 blocks) or the up row of the same
  // output column; a piece lies in one block, so the wave loads only gate or only up rows.
  uint32_t voa[PA], vob[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int row = 8 * (wave + NW * i) + (lane >> 3);
    voa[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(2 * ldx) +
             16u * ((lane & 7) ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int row = 8 * (wave + NW * i) + (lane >> 3);
    int src = row;
    if constexpr (EPI == EPI_SWIGLU) {
      const int block = row / 16;
      src = (block / NB) * (NB / 2) * 16 + (block % NB % (NB / 2)) * 16 + row % 16;
    }
    vob[i] = static_cast<uint32_t>(src) * static_cast<uint32_t>(2 * K) +
             16u * ((lane & 7) ^ ((row >> 1) & 7));
  }
  u32x4_v sa, sb, na, nb;  // this tile's and the next one's buffers
  auto tile_srd = [&](int tt, u32x4_v& a, u32x4_v& b) {
    int tm, tn;
    const bool ok = tt < tiles;  // no next tile: every load is out of range
    tile_mn(ok ? tt : 0, tm, tn);
    const int m0 = tm * TM;
    a = raw_srd(x + static_cast<int64_t>(m0) * ldx,
                ok ? static_cast<uint32_t>(min(TM, M - m0) - 1) * static_cast<uint32_t>(2 * ldx) +
                         2u * K
                   : 0u);
    int n0 = tn * TN, rows = min(TN, N - n0);
    if constexpr (EPI == EPI_SWIGLU) {
      const int inter = N / 2;
      n0 = tn * (TN / 2);
      rows = min(TN / 2, inter - n0);
      if ((wave / 2) % NB >= NB / 2) n0 += inter;
    }
    b = raw_srd(w + static_cast<int64_t>(n0) * K,
                ok ? static_cast<uint32_t>(rows) * static_cast<uint32_t>(2 * K) : 0u);
  };
  uint32_t lbuf = 0;  // the stage that the next loads fill
  uint32_t cbuf = 0;  // the stage being multiplied
  auto next_stage = [&](uint32_t b) { return b + STAGE == ST * STAGE ? 0u : b + STAGE; };
  auto load_piece = [&](int i, const u32x4_v& a, const u32x4_v& b, uint32_t koff) {
    const uint32_t dst = lds0 + lbuf + 1024u * wave;
    if (i < PA) {
      dma16(voa[i], a, koff, dst + 1024u * NW * i);
    } else {
      dma16(vob[i - PA], b, koff, dst + TM * 128u + 1024u * NW * (i - PA));
    }
  };
  tile_srd(t, sa, sb);
#pragma unroll
  for (int s = 0; s < ST - 1; ++s) {
#pragma unroll
    for (int i = 0; i < PER; ++i) load_piece(i, sa, sb, 128u * s);
    lbuf = next_stage(lbuf);
  }

  const uint32_t abase = (wm * MB * 16 + r) * 128 + 16 * (g ^ ((r >> 1) & 7));
  const uint32_t bbase = TM * 128 + (wn * NB * 16 + r) * 128 + 16 * (g ^ ((r >> 1) & 7));
  bf16x8_v fa[2][MB], fb[2][NB];
  f32x4_v acc[MB][NB], tot[MB][NB];
  auto read_frag = [&](int s, int i) {
    if (i < NB) {
      fb[s][i] = *reinterpret_cast<const bf16x8_v*>(lds + cbuf + (bbase ^ (64u * s)) + 2048 * i);
    } else {
      fa[s][i - NB] =
          *reinterpret_cast<const bf16x8_v*>(lds + cbuf + (abase ^ (64u * s)) + 2048 * (i - NB));
    }
  };
  // Half a sub-tile: the fragments of its k-step s are read while the k-step before is
  // multiplied (mul), two MFMAs per read, the next stage's loads (load) among them. zero:
  // the products start a chunk. fold: first fold the block's finished chunk sum into tot
  // (keep = -0 for a tile's first chunk: tot is +0 then, and -0 * 0 + acc is acc bit for bit).
  constexpr int NR = MB + NB, NM = MB * NB;
  auto half = [&](int s, bool mul, bool zero, bool fold, float keep, bool load, const u32x4_v& a,
                  const u32x4_v& b, uint32_t koff) {
    int reads = 0, loads = 0;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int want = ((k + 2) * NR * 4 + 3 * NM - 1) / (3 * NM);  // all in 3/4 of the MFMAs
        if (reads < NR && reads < want) read_frag(s, reads++);
      }
      if (load && loads < PER) {
        load_piece(loads, a, b, koff);
        ++loads;
      }
      if (mul) {
        const int i = k / NB, j = k % NB;
        if (fold) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            tot[i][j][e] = __builtin_fmaf(tot[i][j][e], keep, acc[i][j][e]);
        }
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            fb[1 - s][j], fa[1 - s][i], zero ? f32x4_v{0.0f, 0.0f, 0.0f, 0.0f} : acc[i][j], 0, 0,
            0);
        if (k % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (; reads < NR; ++reads) read_frag(s, reads);
    if (load) {
#pragma unroll
      for (; loads < PER; ++loads) load_piece(loads, a, b, koff);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  while (t < tiles) {
    const int t_next = t + grid;
    tile_srd(t_next, na, nb);
    for (int c = 0; c < nch; ++c) {
      const float keep = c == 1 ? -0.0f : 1.0f;
#pragma unroll
      for (int j = 0; j < SUBS; ++j) {
        wait_barrier<PER * (ST - 2)>();
        // Load sub-tile q + ST - 1 of the stream into the stage read last before the barrier.
        const int sub = SUBS * c + j + ST - 1;
        const bool next = sub >= nsub;
        const u32x4_v a = pick(next, na, sa);
        const u32x4_v b = pick(next, nb, sb);
        const uint32_t koff = 128u * (next ? sub - nsub : sub);
        if (j == 0 && c == 0) {
          half(0, false, false, false, 1.0f, true, a, b, koff);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int q = 0; q < NB; ++q) tot[mb][q] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
          half(1, true, true, false, 1.0f, false, a, b, 0);
        } else {
          half(0, true, false, false, 1.0f, true, a, b, koff);
          half(1, true, j == 0, j == 0, keep, false, a, b, 0);
        }
        lbuf = next_stage(lbuf);
        cbuf = next_stage(cbuf);
      }
    }
    // The last k-step's products and the last fold.
    const float keep = nch == 1 ? -0.0f : 1.0f;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[1][j], fa[1][i], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          tot[i][j][e] = __builtin_fmaf(tot[i][j][e], keep, acc[i][j][e]);
      }
    }
    // Lane: row 16 i + r of the wave's rows, columns 16 j + 4 g .. +3. (el is the lane,
    // opaque to the compiler: addresses derived from it are not kept through the main loop.)
    int el = lane;
    asm volatile("" : "+v"(el));
    const int er = el & 15, eg = el >> 4;
    int tm, tn;
    tile_mn(t, tm, tn);
    const int row0 = tm * TM + wm * MB * 16;
    char* scratch = lds + ST * STAGE;
    if constexpr (EPI == EPI_Y || EPI == EPI_SWIGLU) {
      // One row block (IB of them where a store covers more than 16 rows) at a time. bf16
      // goes through the wave's 2 KB of scratch, so that a store covers whole 32 CB-byte row
      // segments (direct 8-byte stores: 8192 x 6144 104.9 -> 95.2 us).
      constexpr int CB = EPI == EPI_SWIGLU ? NB / 2 : NB;  // column blocks written per wave
      constexpr int PPR = 2 * CB;                          // 16-byte pieces per staged row
      constexpr int RPS = 64 / PPR;                        // rows per store
      constexpr int IB = RPS > 16 ? RPS / 16 : 1;
      static_assert(MB % IB == 0 && 16 * IB * 16 * PPR <= 2048, "store staging");
      const int ncols = EPI == EPI_SWIGLU ? N / 2 : N;
      const int col0 = (tn * WN + wn) * CB * 16;
      char* st = scratch + wave * 2048;
#pragma unroll
      for (int i0 = 0; i0 < MB; i0 += IB) {
#pragma unroll
        for (int i = i0; i < i0 + IB; ++i) {
          const int64_t row = row0 + 16 * i + er;
#pragma unroll
          for (int j = 0; j < CB; ++j) {
            const int col = col0 + 16 * j + 4 * eg;
            f32x4_v v = tot[i][j];
            if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                v[e] = silu_mul1(round_bf16(v[e]), round_bf16(tot[i][j + NB / 2][e]));
            } else if (out.bias != nullptr && col < N) {
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] += bf16_to_f32(out.bias[col + e]);
            }
            const u32x2_v u = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            if (out.wide && !out.out_fp32) {
              *reinterpret_cast<u32x2_v*>(st + (16 * (i - i0) + er) * (16 * PPR) +
                                          16 * ((2 * j + (eg >> 1)) ^ (er & (PPR - 1))) +
                                          8 * (eg & 1)) = u;
            } else if (row < M && col < ncols) {
              if (out.out_fp32) {
                float* y = static_cast<float*>(out.y) + row * ncols + col;
                const f32x4_v q = {bf16_lo(u[0]), bf16_hi(u[0]), bf16_lo(u[1]), bf16_hi(u[1])};
                if (out.wide) {
                  *reinterpret_cast<f32x4_v*>(y) = q;
                } else {
#pragma unroll
                  for (int e = 0; e < 4; ++e) y[e] = q[e];
                }
              } else {
                bf16_t* y = static_cast<bf16_t*>(out.y) + row * ncols + col;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  y[e] = static_cast<bf16_t>(u[e / 2] >> (16 * (e % 2)));
              }
            }
          }
        }
        if (out.wide && !out.out_fp32) {
          bf16_t* y = static_cast<bf16_t*>(out.y);
          const int pp = el % PPR;
#pragma unroll
          for (int q = 0; q < 16 * IB / RPS; ++q) {
            const int lr = RPS * q + el / PPR;
            const u32x4_v u = *reinterpret_cast<const u32x4_v*>(
                st + lr * (16 * PPR) + 16 * (pp ^ (lr & (PPR - 1))));
            const int64_t row = row0 + 16 * i0 + lr;
            const int col = col0 + 8 * pp;
            if (row < M && col < ncols) *reinterpret_cast<u32x4_v*>(y + row * ncols + col) = u;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // lm_head epilogues: each lane's best (EPI_ARGMAX) of a row over its 4 NB columns, or its
      // sampler state (EPI_SAMPLE; logits written as fp32 when y is given), merged over the 4
      // lanes of the row, then over the WN waves of the row band in wave order through LDS: one
      // record per (column tile, row).
      float* s_f = reinterpret_cast<float*>(scratch);
      static_assert(6 * WN * TM * 4 <= S::SCRATCH, "statistics exceed the scratch");
      int* s_i = reinterpret_cast<int*>(s_f + 5 * WN * TM);
      const int col0 = (tn * WN + wn) * NB * 16;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int lr = wm * MB * 16 + 16 * i + er;
        const int64_t row = static_cast<int64_t>(tm) * TM + lr;
        const bool row_ok = row < M;
        float temp = 0.0f;
        uint32_t h = 0;
        if constexpr (EPI == EPI_SAMPLE) {
          const int64_t rc = row_ok ? row : M - 1;
          temp = out.sp.temps[rc];
          h = gumbel_row(out.sp.seeds[rc], out.sp.positions[rc]);
        }
        // Sampler state of each column residue mod 16 (four a lane), in the order that is part of
        // a row's softmax sum: a residue's columns, then residues r and r ^ 1, ^ 2, ^ 4, ^ 8.
        SState a = sstate_empty(), c[4] = {a, a, a, a};
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int col = col0 + 16 * j + 4 * eg;
          if (col >= N || !row_ok) continue;
          f32x4_v q;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = tot[i][j][e];
            if (EPI == EPI_ARGMAX && out.bias != nullptr) v += bf16_to_f32(out.bias[col + e]);
            q[e] = round_bf16(v);
            if constexpr (EPI == EPI_SAMPLE) {
              if (j == 0) {
                c[e] = sstate_first(q[e], col + e, temp, h);
              } else {
                sstate_add(c[e], q[e], col + e, temp, h);
              }
            } else if (argmax_better(q[e], col + e, a.v1, a.i1)) {
              a.v1 = q[e];
              a.i1 = col + e;
            }
          }
          if (out.y != nullptr) {
            float* y = static_cast<float*>(out.y) + row * N + col;
            if (out.wide) {
              *reinterpret_cast<f32x4_v*>(y) = q;
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) y[e] = q[e];
            }
          }
        }
        if constexpr (EPI == EPI_SAMPLE) {
          const bool greedy = !(temp > 0.0f);
          sstate_merge(c[0], c[1], greedy);
          sstate_merge(c[2], c[3], greedy);
          sstate_merge(c[0], c[2], greedy);
          a = c[0];
        }
        sstate_merge_xor<16, 64>(a, EPI == EPI_ARGMAX || !(temp > 0.0f));
        if (eg == 0) {
          const int o = wn * TM + lr;
          s_f[2 * WN * TM + o] = a.v1;
          s_i[o] = a.i1;
          if constexpr (EPI == EPI_SAMPLE) {
            s_f[o] = a.m;
            s_f[WN * TM + o] = a.s;
            s_f[3 * WN * TM + o] = a.x1;
            s_f[4 * WN * TM + o] = a.v2;
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      for (int lr = threadIdx.x; lr < TM; lr += NW * 64) {
        const int64_t row = static_cast<int64_t>(tm) * TM + lr;
        if (row >= M) continue;
        SState a = sstate_empty();
        const bool greedy = EPI == EPI_ARGMAX || !(out.sp.temps[row] > 0.0f);
#pragma unroll
        for (int q = 0; q < WN; ++q) {
          const int o = q * TM + lr;
          SState b = sstate_empty();
          b.v1 = s_f[2 * WN * TM + o];
          b.i1 = s_i[o];
          if constexpr (EPI == EPI_SAMPLE) {
            b.m = s_f[o];
            b.s = s_f[WN * TM + o];
            b.x1 = s_f[3 * WN * TM + o];
            b.v2 = s_f[4 * WN * TM + o];
          }
          if (q == 0) {
            a = b;
          } else {
            sstate_merge(a, b, greedy);
          }
        }
        if constexpr (EPI == EPI_SAMPLE) {
          sstate_store(out.sp.st, static_cast<int64_t>(tn) * out.sp.cand_rows + row, a);
        } else {
          out.best_val[static_cast<int64_t>(tn) * out.sp.cand_rows + row] = a.v1;
          out.best_idx[static_cast<int64_t>(tn) * out.sp.cand_rows + row] = a.i1;
        }
      }
    }
    t = t_next;
    sa = na;
    sb = nb;
  }
  // Loads issued past the last sub-tile (out of range) still write LDS: they must land
  // before the workgroup's LDS is given back.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Compute units of the current device.
int cu_count() {
  static int count[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (count[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    count[dev] = n;
  }
  return count[dev];
}

template <int WM, int WN, int MB, int NB, int ST, int OCC, int PER_CU, int EPI>
void launch_tile(const void* x, int64_t ldx, const void* w, int64_t m, int64_t n, int64_t k,
                 const TileOut& out, hipStream_t s) {
  using S = TileShape<WM, WN, MB, NB, ST>;
  static_assert(S::LDS * PER_CU <= 160 * 1024, "LDS");
  auto kern = linear_tile_kernel<WM, WN, MB, NB, ST, OCC, EPI>;
  static bool attr_set = false;
  if (!attr_set) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                        hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
    attr_set = true;
  }
  const int mt = static_cast<int>((m + S::TM - 1) / S::TM);
  const int nt = static_cast<int>((n + S::TN - 1) / S::TN);
  const int grid = static_cast<int>(
      std::min<int64_t>(static_cast<int64_t>(mt) * nt, static_cast<int64_t>(cu_count()) * PER_CU));
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(S::NW * 64), S::LDS, s, (const bf16_t*)x, ldx,
                     (const bf16_t*)w, (int)m, (int)n, (int)k, mt, nt, out);
}
// The tile shapes, and the one a problem takes: the cheapest by a model of the main loop, the
// grid's rounds times a round's time per 64-deep sub-tile (ns; identical bits, so this is
// only speed). Measured with K = 1024-3072, M = 100-8420: 256 x 128 970 and 128 x 128 500 (all
// CUs busy), 128 x 64 330, 64 x 64 210 while every CU has at most one tile and 380 with two.
// Large problems are at the MFMA / power bound with the first two, small ones at the memory
// round trips of few workgroups, which smaller tiles spread over more CUs: 777 x 1024 x 3072
// 20.7 (128 x 128) vs 11.6 us (64 x 64), 2048 x 1024 x 2048 15.1 (128 x 128) vs 12.7 (128 x
// 64), 8420 x 1024 x 2048 50.5 (256 x 128, a second round for 8 tiles) vs 43.7 (128 x 128).
int tile_shape(int64_t m, int64_t n) {
  const int64_t cus = cu_count();
  auto tiles = [&](int tm, int tn) { return ((m + tm - 1) / tm) * ((n + tn - 1) / tn); };
  auto rounds = [&](int64_t t, int64_t slots) { return (t + slots - 1) / slots; };
  const int64_t t64 = tiles(64, 64);
  const int64_t cost[4] = {970 * rounds(tiles(256, 128), cus), 500 * rounds(tiles(128, 128), cus),
                           330 * rounds(tiles(128, 64), cus),
                           t64 <= cus ? 210 : 380 * rounds(t64, 2 * cus)};
  int best = 0;
  for (int i = 1; i < 4; ++i)
    if (cost[i] < cost[best]) best = i;
  return best;
}

template <int EPI>
void launch_tiles(const void* x, int64_t ldx, const void* w, int64_t m, int64_t n, int64_t k,
                  const TileOut& out, hipStream_t s) {
  if constexpr (EPI == EPI_ARGMAX || EPI == EPI_SAMPLE) {
    // 128-column tiles: the candidate grouping of the lm_head epilogues
    launch_tile<4, 2, 2, 4, 4, 2, 1, EPI>(x, ldx, w, m, n, k, out, s);
  } else {
    switch (tile_shape(m, n)) {
      case 0: launch_tile<4, 2, 4, 4, 3, 2, 1, EPI>(x, ldx, w, m, n, k, out, s); break;
      case 1: launch_tile<4, 2, 2, 4, 4, 2, 1, EPI>(x, ldx, w, m, n, k, out, s); break;
      case 2: launch_tile<4, 2, 2, 2, 5, 2, 1, EPI>(x, ldx, w, m, n, k, out, s); break;
      default: launch_tile<2, 2, 2, 2, 4, 1, 2, EPI>(x, ldx, w, m, n, k, out, s); break;
    }
  }
}

// Sizes whose tile offsets fit the kernel's 32-bit buffer ranges and indices (256 rows of x).
bool tiles_fit(int64_t ldx, int64_t m, int64_t n, int64_t k) {
  return ldx < (1ll << 23) && k < (1ll << 23) && m < (1ll << 31) && n < (1ll << 30);
}

TileOut tile_out(void* y, const void* bias = nullptr, int out_fp32 = 0) {
  TileOut o{};
  o.y = y;
  o.bias = static_cast<const bf16_t*>(bias);
  o.out_fp32 = out_fp32;
  o.wide = (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  return o;
}

// sid_linear_silu_mul takes the tile kernel above this many rows. Up to two 16-row blocks the
// streaming kernel's eight-column workgroups put more weight loads in flight (I = 3072,
// weights from HBM, streaming vs tiles, us: 16 rows 5.6 vs 7.3, 32 rows 6.6 vs 7.4; 48 rows
// 7.8 vs 7.6, 64 rows 8.9 vs 7.9, 95 rows 12.6 vs 7.5; I = 9728: 32 rows 14.5 vs 12.3,
// 64 rows 20.1 vs 13.8).
constexpr int64_t kLinearSiluStreamMaxM = 32;

// The lm_head epilogues' launch: 128-row tiles in slices of as many rows as the 32-bit
// buffer offsets hold (one slice but for row strides of 16M elements and more).
template <int EPI>
void launch_head_tiles(const void* x, int64_t ldx, const void* w, int64_t m, int64_t n, int64_t k,
                       const TileOut& out, hipStream_t s) {
  const int64_t step = ldx < (1ll << 24) ? m : std::max<int64_t>(1, 0xffffffffll / (2 * ldx));
  for (int64_t r0 = 0; r0 < m; r0 += step) {
    TileOut o = out;
    if (o.y != nullptr) o.y = static_cast<float*>(o.y) + r0 * n;
    if constexpr (EPI == EPI_ARGMAX) {
      o.best_val += r0;
      o.best_idx += r0;
    } else {
      SampleIn& p = o.sp;
      p.temps += r0;
      p.seeds += r0;
      p.positions += r0;
      p.st = sample_stats_at(p.st, r0);
    }
    launch_tiles<EPI>(static_cast<const bf16_t*>(x) + r0 * ldx, ldx, w, std::min(step, m - r0), n,
                      k, o, s);
  }
}

// K of the streaming kernel below, its chunk count and LDS row stride of staged x.
constexpr int WIDE_K = 1024;
constexpr int WIDE_NCH = WIDE_K / KC;
constexpr int WXS = WIDE_K + 8;

// Streaming wide-N GEMM for K = 1024, M <= 64 (lm_head at decode), optionally with the
// greedy argmax fused into its epilogue.
//
// A persistent grid of one 8-wave workgroup per CU stages the x row group in LDS once;
// every wave then owns every (number of waves)-th 16-column wave tile and streams its weights
// chunk by chunk (16 columns x 256 k = 8 KiB per chunk) through a ring of three register
// buffers, so two chunks are always in flight while the MFMAs of the third run. Each
// chunk's MFMA sequence and the left fold of the four chunks are those of linear_kernel,
// so the logits have the same bits. With ARGMAX, each lane keeps the best (value, column)
// of the rows it holds over its wave's columns (the values compared are the bf16-rounded
// logits the unfused path writes); the workgroup's best per row goes to a workspace
// [workgroups][M] that argmax_finalize_kernel reduces. The (value, index) order is total
// (torch's: larger value, then smaller index; NaN above everything, first NaN wins), so
// the result does not depend on how the columns are split.
constexpr int STREAM_WAVES = 8;

template <int MBS, bool ARGMAX, bool LEAN = false>
__global__ void __launch_bounds__(STREAM_WAVES * 64) linear_stream_kernel(
    const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w,
    const bf16_t* __restrict__ bias, void* __restrict__ y, int M, int N, int out_fp32,
    float* __restrict__ best_val, int* __restrict__ best_idx, int cand_rows, int row0) {
  extern __shared__ __align__(16) bf16_t lx[];  // [MBS*16][WXS]
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int gw = blockIdx.x * STREAM_WAVES + wave;
  const int num_waves = gridDim.x * STREAM_WAVES;
  const int tiles = N / 16;
  // Wave gw owns tiles gw, gw + num_waves, ...: at any moment the chip's waves read
  // neighbouring tiles (measured against contiguous runs per wave: M = 1 67.8 -> 65.4 us,
  // M = 64 82.2 -> 81.0). The argmax order is total, so the assignment does not matter.
  const int t_begin = gw, t_step = num_waves;
  const int units = (gw < tiles ? (tiles - gw + num_waves - 1) / num_waves : 0) * WIDE_NCH;

  // Unit u = (tile t_begin + (u/4) * t_step, chunk u%4); loads past the end are clamped to
  // the last unit (redundant, never consumed) so every issue point is unconditional.
  auto unit_ptr = [&](int u) {
    u = min(u, max(units - 1, 0));
    const int64_t col = static_cast<int64_t>(t_begin + (u >> 2) * t_step) * 16 + r;
    return w + col * WIDE_K + (u & 3) * KC + 8 * g;
  };
  bf16x8_v b0[NSTEP], b1[NSTEP], b2[NSTEP];
  if (units > 0) {
    load_w(b0, unit_ptr(0), 0);
    load_w(b1, unit_ptr(1), 0);
  }

  // Stage x (rows >= M clamped to row M-1; their outputs are discarded).
  constexpr int ROWS = MBS * 16;
  constexpr int VPR = WIDE_K / 8;  // 16-byte vectors per row
  constexpr int VPT = ROWS * VPR / (STREAM_WAVES * 64);
  {
    bf16x8_v xv[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * STREAM_WAVES * 64;
      const int row = v / VPR;
      xv[i] = ld_frag(x + static_cast<int64_t>(min(row, M - 1)) * ldx + (v % VPR) * 8);
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * STREAM_WAVES * 64;
      *reinterpret_cast<bf16x8_v*>(&lx[(v / VPR) * WXS + (v % VPR) * 8]) = xv[i];
    }
  }
  __syncthreads();
  // A wave without columns (N/16 < waves) still writes its (-inf, none) candidates.
  if (!ARGMAX && units == 0) return;

  f32x4_v total[MBS];
  float bv[MBS][4];
  int bi[MBS][4];
  if constexpr (ARGMAX) {
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bv[mb][i] = -INFINITY;
        bi[mb][i] = 0x7fffffff;
      }
    }
  }

  auto consume = [&](const bf16x8_v (&wf)[NSTEP], int u) {
    const int c = u & 3;
    f32x4_v acc[MBS];
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) acc[mb] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < NSTEP; ++s) {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb) {
        const bf16x8_v af = *reinterpret_cast<const bf16x8_v*>(
            &lx[(16 * mb + r) * WXS + c * KC + KSTEP * s + 8 * g]);
        acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf[s], acc[mb], 0, 0, 0);
      }
    }
    if (c == 0) {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb) total[mb] = acc[mb];
    } else {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) total[mb][i] += acc[mb][i];
      }
    }
    if (c != 3) return;
    const int col = (t_begin + (u >> 2) * t_step) * 16 + r;
    // LEAN: no bias and no logits written (the greedy-only call), so the epilogue holds no
    // load and no store that the weight stream's waits would have to account for.
    const bool has_bias = !LEAN && bias != nullptr;
    const bool has_y = !LEAN && y != nullptr;
    const float bias_v = has_bias ? bf16_to_f32(bias[col]) : 0.0f;
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * mb + 4 * g + i;
        float v = total[mb][i];
        if (has_bias) v += bias_v;
        const float vr = round_bf16(v);
        if (has_y && row < M) {
          const int64_t off = static_cast<int64_t>(row) * N + col;
          if (out_fp32) {
            static_cast<float*>(y)[off] = vr;
          } else {
            static_cast<bf16_t*>(y)[off] = f32_to_bf16(v);
          }
        }
        if constexpr (ARGMAX) {
          if (argmax_better(vr, col, bv[mb][i], bi[mb][i])) {
            bv[mb][i] = vr;
            bi[mb][i] = col;
          }
        }
      }
    }
  };

  for (int u = 0; u < units; u += 3) {
    load_w(b2, unit_ptr(u + 2), 0);
    consume(b0, u);
    load_w(b0, unit_ptr(u + 3), 0);
    if (u + 1 < units) consume(b1, u + 1);
    load_w(b1, unit_ptr(u + 4), 0);
    if (u + 2 < units) consume(b2, u + 2);
  }

  if constexpr (ARGMAX) {
    // Best over the 16 column lanes of each row (lanes r = 0..15 of a row group g).
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = bv[mb][i];
        int ix = bi[mb][i];
#pragma unroll
        for (int mask = 1; mask < 16; mask <<= 1) {
          const float ov = lane_xor(v, mask);
          const int oi = __builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, ix);
          if (argmax_better(ov, oi, v, ix)) {
            v = ov;
            ix = oi;
          }
        }
        bv[mb][i] = v;
        bi[mb][i] = ix;
      }
    }
    // Then over the workgroup's waves (x is no longer read, its LDS is reused): one candidate
    // per row and workgroup for the finalize to gather from lines that hold all rows (a
    // candidate per wave: 64 rows x 2048 candidates took the finalize 7.3 us, 256 take 4.8;
    // 64 x 151936 greedy 75.7 -> 71.9 us in all).
    __syncthreads();
    float* s_v = reinterpret_cast<float*>(lx);
    int* s_i = reinterpret_cast<int*>(s_v + STREAM_WAVES * ROWS);
    if (r == 0) {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s_v[wave * ROWS + 16 * mb + 4 * g + i] = bv[mb][i];
          s_i[wave * ROWS + 16 * mb + 4 * g + i] = bi[mb][i];
        }
      }
    }
    __syncthreads();
    const int row = threadIdx.x;
    if (row < M && row < ROWS) {
      float v = s_v[row];
      int ix = s_i[row];
#pragma unroll
      for (int q = 1; q < STREAM_WAVES; ++q) {
        const float ov = s_v[q * ROWS + row];
        const int oi = s_i[q * ROWS + row];
        if (argmax_better(ov, oi, v, ix)) {
          v = ov;
          ix = oi;
        }
      }
      best_val[static_cast<int64_t>(blockIdx.x) * cand_rows + row0 + row] = v;
      best_idx[static_cast<int64_t>(blockIdx.x) * cand_rows + row0 + row] = ix;
    }
  }
}

// Per row: the best of the candidates (any order gives the same answer).
__global__ void __launch_bounds__(256) argmax_finalize_kernel(const float* __restrict__ best_val,
                                                              const int* __restrict__ best_idx,
                                                              int num_cands, int M,
                                                              int64_t* __restrict__ out) {
  const int row = blockIdx.x;
  float v = -INFINITY;
  int ix = 0x7fffffff;
  // Eight candidates per thread loaded at once (one round trip for up to 2048 of the tiled
  // path instead of eight); the order is total, so the visiting order is free.
  constexpr int U = 8;
  for (int base = threadIdx.x; base < num_cands; base += 256 * U) {
    float cv[U];
    int ci[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int wv = base + 256 * u;
      const bool in = wv < num_cands;
      const int64_t off = static_cast<int64_t>(wv) * M + row;
      cv[u] = -INFINITY;
      ci[u] = 0x7fffffff;
      if (in) {
        cv[u] = best_val[off];
        ci[u] = best_idx[off];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (argmax_better(cv[u], ci[u], v, ix)) {
        v = cv[u];
        ix = ci[u];
      }
    }
  }
  for (int mask = 1; mask < 64; mask <<= 1) {
    const float ov = lane_xor(v, mask);
    const int oi = __builtin_amdgcn_ds_bpermute((__lane_id() ^ mask) << 2, ix);
    if (argmax_better(ov, oi, v, ix)) {
      v = ov;
      ix = oi;
    }
  }
  __shared__ float s_v[4];
  __shared__ int s_i[4];
  if ((threadIdx.x & 63) == 0) {
    s_v[threadIdx.x >> 6] = v;
    s_i[threadIdx.x >> 6] = ix;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; ++k) {
      if (argmax_better(s_v[k], s_i[k], v, ix)) {
        v = s_v[k];
        ix = s_i[k];
      }
    }
    out[row] = ix == 0x7fffffff ? 0 : ix;
  }
}

// ---- lm_head with the stochastic sampler fused into its epilogue ---------------------------
//
// The draw of sid/engine/sampler.py:32-69 without truncation (top_k <= 0, top_p >= 1):
// token = argmax_c log(p_c + eps) + g_c with p = softmax(l / T) and g the seeded Gumbel
// noise; greedy rows (T <= 0) take the argmax of the logits. Nothing of the logits is
// written. linear_sample_kernel is linear_stream_kernel (same grid, same per-column MFMA
// sequence and chunk fold, so the same logit bits l_c) with this epilogue: for every row it
// holds, each lane keeps over its wave's columns
//   mx, sm   online softmax state of x = l / T (sm = sum of exp(x - mx), rescaled when mx
//            grows),
//   a1       the column with the largest x + g (value a1v, its x a1x, index a1i; ties to the
//            lower index), a2v the second largest x + g;
// the 16 lanes of a row are merged in a fixed butterfly and written per (wave, row).
// sample_finalize_kernel takes one row: M = max mx, S = sum of sm exp(mx - M) in wave order,
// then the exact score log(exp(x - M) / S + eps) + g of every wave's a1 (the formula of the
// unfused sampler). Any other column c of a wave scores
//   log(exp(x_c + g_c - M) / S + eps exp(g_c)) <= log(exp(a2v - M) / S + eps exp(G)),
// increasing in x_c + g_c and in g_c (G: the largest value the noise takes, at u = 1 - 2^-24),
// so a wave whose bound stays below the best candidate
// (by a margin far above float rounding) cannot hold the winner. A wave that fails the test
// (a near-tie, or non-finite statistics: then every wave) has its logits recomputed for the
// row with the same MFMA sequence (identical bits) and every column scored exactly.
template <int MBS>
__global__ void __launch_bounds__(STREAM_WAVES * 64) linear_sample_kernel(
    const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, int M, int N,
    const float* __restrict__ temps, const int64_t* __restrict__ seeds,
    const int64_t* __restrict__ positions, SampleStats st, int cand_rows, int row0) {
  extern __shared__ __align__(16) bf16_t lx[];  // [MBS*16][WXS]
  __shared__ float s_t[64];
  __shared__ uint32_t s_h[64];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int gw = blockIdx.x * STREAM_WAVES + wave;
  const int num_waves = gridDim.x * STREAM_WAVES;
  const int tiles = N / 16;
  const int t_begin = static_cast<int>(static_cast<int64_t>(gw) * tiles / num_waves);
  const int t_end = static_cast<int>(static_cast<int64_t>(gw + 1) * tiles / num_waves);
  const int units = (t_end - t_begin) * WIDE_NCH;

  auto unit_ptr = [&](int u) {
    u = min(u, max(units - 1, 0));
    const int64_t col = static_cast<int64_t>(t_begin + (u >> 2)) * 16 + r;
    return w + col * WIDE_K + (u & 3) * KC + 8 * g;
  };
  bf16x8_v b0[NSTEP], b1[NSTEP], b2[NSTEP];
  if (units > 0) {
    load_w(b0, unit_ptr(0), 0);
    load_w(b1, unit_ptr(1), 0);
  }
  constexpr int ROWS = MBS * 16;
  constexpr int VPR = WIDE_K / 8;
  constexpr int VPT = ROWS * VPR / (STREAM_WAVES * 64);
  {
    bf16x8_v xv[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * STREAM_WAVES * 64;
      const int row = v / VPR;
      xv[i] = ld_frag(x + static_cast<int64_t>(min(row, M - 1)) * ldx + (v % VPR) * 8);
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int v = threadIdx.x + i * STREAM_WAVES * 64;
      *reinterpret_cast<bf16x8_v*>(&lx[(v / VPR) * WXS + (v % VPR) * 8]) = xv[i];
    }
  }
  if (threadIdx.x < 64) {
    const int row = min(static_cast<int>(threadIdx.x), M - 1) + row0;
    s_t[threadIdx.x] = temps[row];
    s_h[threadIdx.x] = gumbel_row(seeds[row], positions[row]);
  }
  __syncthreads();

  f32x4_v total[MBS];
  float mx[MBS][4], sm[MBS][4], a1v[MBS][4], a1x[MBS][4], a2v[MBS][4];
  int a1i[MBS][4];
#pragma unroll
  for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      mx[mb][i] = -INFINITY;
      sm[mb][i] = 0.0f;
      a1v[mb][i] = -INFINITY;
      a1x[mb][i] = -INFINITY;
      a2v[mb][i] = -INFINITY;
      a1i[mb][i] = 0x7fffffff;
    }
  }

  auto consume = [&](const bf16x8_v (&wf)[NSTEP], int u) {
    const int c = u & 3;
    f32x4_v acc[MBS];
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) acc[mb] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < NSTEP; ++s) {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb) {
        const bf16x8_v af = *reinterpret_cast<const bf16x8_v*>(
            &lx[(16 * mb + r) * WXS + c * KC + KSTEP * s + 8 * g]);
        acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf[s], acc[mb], 0, 0, 0);
      }
    }
    if (c == 0) {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb) total[mb] = acc[mb];
    } else {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) total[mb][i] += acc[mb][i];
      }
    }
    if (c != 3) return;
    const int col = (t_begin + (u >> 2)) * 16 + r;
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * mb + 4 * g + i;
        const float vr = round_bf16(total[mb][i]);
        const float t = s_t[row];
        if (!(t > 0.0f)) {  // greedy row: the logit itself
          if (argmax_better(vr, col, a1v[mb][i], a1i[mb][i])) {
            a1v[mb][i] = vr;
            a1i[mb][i] = col;
          }
          continue;
        }
        const float xv = vr / t;
        if (xv > mx[mb][i]) {
          sm[mb][i] = sm[mb][i] * expf(mx[mb][i] - xv) + 1.0f;
          mx[mb][i] = xv;
        } else {
          sm[mb][i] += expf(xv - mx[mb][i]);
        }
        const float gn = seeded_gumbel(s_h[row], col);
        const float xg = xv + gn;
        if (xg > a1v[mb][i] || (xg == a1v[mb][i] && col < a1i[mb][i])) {
          a2v[mb][i] = a1v[mb][i];
          a1v[mb][i] = xg;
          a1x[mb][i] = xv;
          a1i[mb][i] = col;
        } else {
          a2v[mb][i] = fmaxf(a2v[mb][i], xg);
        }
      }
    }
  };

  for (int u = 0; u < units; u += 3) {
    load_w(b2, unit_ptr(u + 2), 0);
    consume(b0, u);
    load_w(b0, unit_ptr(u + 3), 0);
    if (u + 1 < units) consume(b1, u + 1);
    load_w(b1, unit_ptr(u + 4), 0);
    if (u + 2 < units) consume(b2, u + 2);
  }

  // Merge the 16 column lanes of each row (fixed butterfly), lane r = 0 writes.
#pragma unroll
  for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * mb + 4 * g + i;
      const bool greedy = !(s_t[row] > 0.0f);
      float m = mx[mb][i], sv = sm[mb][i], v1 = a1v[mb][i], x1 = a1x[mb][i], v2 = a2v[mb][i];
      int i1 = a1i[mb][i];
#pragma unroll
      for (int mask = 1; mask < 16; mask <<= 1) {
        const int src = (lane ^ mask) << 2;
        const float om = lane_xor(m, mask);
        const float os = lane_xor(sv, mask);
        const float ov1 = lane_xor(v1, mask);
        const float ox1 = lane_xor(x1, mask);
        const float ov2 = lane_xor(v2, mask);
        const int oi1 = __builtin_amdgcn_ds_bpermute(src, i1);
        if (greedy) {
          if (argmax_better(ov1, oi1, v1, i1)) {
            v1 = ov1;
            i1 = oi1;
          }
          continue;
        }
        softmax_merge(m, sv, om, os);
        if (ov1 > v1 || (ov1 == v1 && oi1 < i1)) {
          v2 = fmaxf(v1, ov2);
          v1 = ov1;
          x1 = ox1;
          i1 = oi1;
        } else {
          v2 = fmaxf(v2, fmaxf(ov1, ov2));
        }
      }
      if (r == 0 && row < M) {
        const int64_t o = static_cast<int64_t>(gw) * cand_rows + row0 + row;
        st.mx[o] = m;
        st.sm[o] = sv;
        st.a1v[o] = v1;
        st.a1x[o] = x1;
        st.a2v[o] = v2;
        st.a1i[o] = i1;
      }
    }
  }
}

__device__ __forceinline__ bool score_better(float v, int i, float bv, int bi) {
  return argmax_better(v, i, bv, bi);
}

// Best (value, index) over the block under argmax_better; every thread gets the result.
__device__ __forceinline__ void block_best_i32(float& bv, int& bi, float* s_v, int* s_i) {
  for (int mask = 1; mask < 64; mask <<= 1) {
    const float ov = lane_xor(bv, mask);
    const int oi = __builtin_amdgcn_ds_bpermute((__lane_id() ^ mask) << 2, bi);
    if (argmax_better(ov, oi, bv, bi)) {
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
  for (int k = 1; k < static_cast<int>(blockDim.x >> 6); ++k) {
    if (argmax_better(s_v[k], s_i[k], bv, bi)) {
      bv = s_v[k];
      bi = s_i[k];
    }
  }
  __syncthreads();
}

constexpr int kFinThreads = 256;
constexpr float kCertMargin = 1e-3f;  // the certificate's slack over float rounding

__global__ void __launch_bounds__(kFinThreads) sample_finalize_kernel(
    const bf16_t* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, int N,
    SampleStats st, int num_waves, int M, const float* __restrict__ temps,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ positions,
    int* __restrict__ redo, int64_t* __restrict__ out, int recompute_all, int group_tiles) {
  __shared__ float s_v[kFinThreads / 64];
  __shared__ int s_i[kFinThreads / 64];
  __shared__ float s_red[kFinThreads / 64];
  __shared__ int s_nredo;
  __shared__ __align__(16) bf16_t s_x[WIDE_K];
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const float t = temps[row];
  auto at = [&](int wv) { return static_cast<int64_t>(wv) * M + row; };

  float bv = -INFINITY;
  int bi = 0x7fffffff;
  if (!(t > 0.0f)) {  // greedy row
    for (int wv = tid; wv < num_waves; wv += kFinThreads) {
      if (argmax_better(st.a1v[at(wv)], st.a1i[at(wv)], bv, bi)) {
        bv = st.a1v[at(wv)];
        bi = st.a1i[at(wv)];
      }
    }
    block_best_i32(bv, bi, s_v, s_i);
    if (tid == 0) out[row] = bi == 0x7fffffff ? 0 : bi;
    return;
  }
  // M and S (fixed order: each thread's waves in order, then the butterfly, then waves)
  float m = -INFINITY;
  for (int wv = tid; wv < num_waves; wv += kFinThreads) m = fmaxf(m, st.mx[at(wv)]);
  for (int mask = 1; mask < 64; mask <<= 1) m = fmaxf(m, lane_xor(m, mask));
  if ((tid & 63) == 0) s_red[tid >> 6] = m;
  __syncthreads();
  m = s_red[0];
  for (int k = 1; k < kFinThreads / 64; ++k) m = fmaxf(m, s_red[k]);
  __syncthreads();
  float part = 0.0f;
  for (int wv = tid; wv < num_waves; wv += kFinThreads) {
    const float mw = st.mx[at(wv)];
    if (mw != -INFINITY) part += st.sm[at(wv)] * expf(mw - m);
  }
  for (int mask = 1; mask < 64; mask <<= 1) part += lane_xor(part, mask);
  if ((tid & 63) == 0) s_red[tid >> 6] = part;
  __syncthreads();
  float sum = s_red[0];
  for (int k = 1; k < kFinThreads / 64; ++k) sum += s_red[k];
  const bool full = recompute_all || !isfinite(m) || !isfinite(sum) || !(sum > 0.0f);
  // eps * exp(G), G = the largest noise value (u = 1 - 2^-24), rounded up a little
  const float g_max = -logf(-logf(16777215.0f / 16777216.0f + kSampleEps) + kSampleEps);
  const float eps_g = kSampleEps * expf(g_max) * 1.0001f;
  const uint32_t h = gumbel_row(seeds[row], positions[row]);
  auto score = [&](float xv, int col) {
    return logf(expf(xv - m) / sum + kSampleEps) + seeded_gumbel(h, col);
  };
  // Every wave's candidate, scored exactly.
  if (!full) {
    for (int wv = tid; wv < num_waves; wv += kFinThreads) {
      const int c = st.a1i[at(wv)];
      if (c == 0x7fffffff) continue;
      const float sc = score(st.a1x[at(wv)], c);
      if (argmax_better(sc, c, bv, bi)) {
        bv = sc;
        bi = c;
      }
    }
  }
  block_best_i32(bv, bi, s_v, s_i);
  // Waves whose other columns might beat the best candidate.
  if (tid == 0) s_nredo = 0;
  __syncthreads();
  int* list = redo + static_cast<int64_t>(row) * num_waves;
  for (int wv = tid; wv < num_waves; wv += kFinThreads) {
    bool need = full;
    if (!need && st.a1i[at(wv)] != 0x7fffffff) {
      const float bound = logf(expf(st.a2v[at(wv)] - m) / sum + eps_g);
      need = !(bound + kCertMargin < bv);
    }
    if (need) list[atomicAdd(&s_nredo, 1)] = wv;
  }
  __syncthreads();
  const int nredo = s_nredo;
  if (nredo > 0) {
    for (int i = tid; i < WIDE_K / 8; i += kFinThreads)
      *reinterpret_cast<bf16x8_v*>(&s_x[8 * i]) =
          *reinterpret_cast<const bf16x8_v*>(x + static_cast<int64_t>(row) * ldx + 8 * i);
    __syncthreads();
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int r = lane & 15;
    const int g = lane >> 4;
    const int tiles = N / 16;
    // Recompute the listed waves' logits (the streaming kernel's MFMA sequence and chunk fold
    // with this row in all 16 A rows, so every lane's result is the row's logit of its
    // column) and score every column.
    for (int k = wave; k < nredo; k += kFinThreads / 64) {
      const int wv = list[k];
      // The group's 16-column tiles: a streaming wave's run, or a fixed-width column tile.
      const int tb = group_tiles > 0 ? wv * group_tiles
                                     : static_cast<int>(static_cast<int64_t>(wv) * tiles / num_waves);
      const int te = group_tiles > 0 ? min(tiles, (wv + 1) * group_tiles)
                                     : static_cast<int>(static_cast<int64_t>(wv + 1) * tiles / num_waves);
      for (int tile = tb; tile < te; ++tile) {
        const int col = tile * 16 + r;
        const bf16_t* wrow = w + static_cast<int64_t>(col) * WIDE_K + 8 * g;
        f32x4_v tot = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < WIDE_NCH; ++c) {
          bf16x8_v wf[NSTEP];
          load_w(wf, wrow, c * KC);
          f32x4_v acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int s = 0; s < NSTEP; ++s) {
            const bf16x8_v af = *reinterpret_cast<const bf16x8_v*>(&s_x[c * KC + KSTEP * s + 8 * g]);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf[s], acc, 0, 0, 0);
          }
          if (c == 0) {
            tot = acc;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) tot[i] += acc[i];
          }
        }
        if (g == 0) {
          const float vr = round_bf16(tot[0]);
          const float sc = score(vr / t, col);
          if (argmax_better(sc, col, bv, bi)) {
            bv = sc;
            bi = col;
          }
        }
      }
    }
    block_best_i32(bv, bi, s_v, s_i);
  }
  if (tid == 0) out[row] = bi == 0x7fffffff ? 0 : bi;
}

int check_shapes(const void* x, int64_t ldx, const void* w, int64_t m, int64_t n, int64_t k,
                 const char* name) {
  SID_REQUIRE(x && w, "%s: null pointer", name);
  SID_REQUIRE(k > 0 && k % KC == 0, "%s: K=%lld must be a positive multiple of %d", name,
              (long long)k, KC);
  SID_REQUIRE(n % NTILE_MIN == 0, "%s: N=%lld must be a multiple of %d", name, (long long)n,
              NTILE_MIN);
  SID_REQUIRE(ldx >= k && ldx % 8 == 0,
              "%s: row stride %lld of x must be >= K and a multiple of 8", name, (long long)ldx);
  SID_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
              "%s: x and w must be 16-byte aligned", name);
  SID_REQUIRE((m + MROWS - 1) / MROWS <= 65535 && n / NTILE_MIN < (1ll << 31),
              "%s: problem too large", name);
  return SID_OK;
}

// The streaming kernel serves sid_linear from this many columns up (lm_head-sized N).
constexpr int64_t kStreamMinN = 32768;

// Row groups of up to 64 rows are streamed one after the other (the weights are re-read
// per group); up to this many rows that still beats the tiled kernel on lm_head shapes.
constexpr int64_t kStreamMaxM = 256;

bool stream_shape_ok(int64_t m, int64_t n, int64_t k) {
  return m >= 1 && m <= kStreamMaxM && k == WIDE_K && n % 16 == 0 && n < (1ll << 31);
}

template <int MBS, bool AM, bool LEAN>
void launch_stream_form(const bf16_t* x, int64_t ldx, const void* w, const void* bias, void* y,
                        int m, int n, int out_fp32, float* bv, int* bi, int cand_rows, int row0,
                        hipStream_t s) {
  const size_t lds = static_cast<size_t>(MBS * 16) * WXS * sizeof(bf16_t);
  static bool attr_set = false;
  if (!attr_set) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&linear_stream_kernel<MBS, AM, LEAN>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    attr_set = true;
  }
  hipLaunchKernelGGL((linear_stream_kernel<MBS, AM, LEAN>), dim3(cu_count()),
                     dim3(STREAM_WAVES * 64), lds, s, x, ldx, (const bf16_t*)w,
                     (const bf16_t*)bias, y, m, n, out_fp32, bv, bi, cand_rows, row0);
}

template <int MBS, bool AM>
void launch_stream_mbs(const bf16_t* x, int64_t ldx, const void* w, const void* bias, void* y,
                       int m, int n, int out_fp32, float* bv, int* bi, int cand_rows, int row0,
                       hipStream_t s) {
  if constexpr (AM) {
    if (bias == nullptr && y == nullptr) {
      launch_stream_form<MBS, AM, true>(x, ldx, w, bias, y, m, n, out_fp32, bv, bi, cand_rows,
                                        row0, s);
      return;
    }
  }
  launch_stream_form<MBS, AM, false>(x, ldx, w, bias, y, m, n, out_fp32, bv, bi, cand_rows, row0,
                                     s);
}

// One launch per 64-row group; group g reads x rows 64g.., writes y rows 64g.. and the
// candidate rows 64g.. of the [workgroups][m] workspace.
template <bool AM>
void launch_stream(const void* x, int64_t ldx, const void* w, const void* bias, void* y, int m,
                   int n, int out_fp32, float* bv, int* bi, hipStream_t s) {
  for (int r0 = 0; r0 < m; r0 += MROWS) {
    const int mg = min(MROWS, m - r0);
    const bf16_t* xg = static_cast<const bf16_t*>(x) + static_cast<int64_t>(r0) * ldx;
    void* yg = nullptr;
    if (y != nullptr) {
      const int64_t off = static_cast<int64_t>(r0) * n;
      yg = out_fp32 ? static_cast<void*>(static_cast<float*>(y) + off)
                    : static_cast<void*>(static_cast<bf16_t*>(y) + off);
    }
    switch ((mg + 15) / 16) {
      case 1: launch_stream_mbs<1, AM>(xg, ldx, w, bias, yg, mg, n, out_fp32, bv, bi, m, r0, s); break;
      case 2: launch_stream_mbs<2, AM>(xg, ldx, w, bias, yg, mg, n, out_fp32, bv, bi, m, r0, s); break;
      case 3: launch_stream_mbs<3, AM>(xg, ldx, w, bias, yg, mg, n, out_fp32, bv, bi, m, r0, s); break;
      default: launch_stream_mbs<4, AM>(xg, ldx, w, bias, yg, mg, n, out_fp32, bv, bi, m, r0, s); break;
    }
  }
}

// ---- gate_up projection with the SwiGLU epilogue (decode-sized M) -----------------------
//
// out[m, j] = bf16(bf16(silu(g)) * u), g = bf16(x w[j]^T), u = bf16(x w[I + j]^T), each a
// canonical chunk fold: the same bits as sid_linear_partials + sid_silu_mul_partials, with
// neither the fp32 partials' round trip through memory nor the second launch. A workgroup
// has one wave per 256-wide chunk (NCH waves, K = 256 NCH) and owns 8 NB output columns of
// a 64-row group; in MFMA column block nb, lanes 0-7 are gate rows j0+8nb.. and lanes 8-15
// the matching up rows I+j0+8nb.. of w. Wave c accumulates chunk c from zero with x and w
// fragments loaded straight from global memory (each wave reads a different chunk, so
// nothing is shared through LDS; the NB column blocks share the wave's x fragments); the
// chunk sums meet in LDS and are folded c0 + c1 + ... in order.
template <int NCH, int MBS, int NB>
__global__ void __launch_bounds__(NCH * 64) linear_silu_kernel(const bf16_t* __restrict__ x,
                                                               const bf16_t* __restrict__ w,
                                                               int64_t M, int64_t inter,
                                                               bf16_t* __restrict__ out) {
  constexpr int64_t K = static_cast<int64_t>(NCH) * KC;
  constexpr int SS = 16 * NB + 1;  // LDS row stride of a chunk sum tile (floats)
  __shared__ float sacc[NCH][MROWS * SS];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int64_t j0 = static_cast<int64_t>(blockIdx.x) * (8 * NB);
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * MROWS;
  const int mrows = static_cast<int>(min<int64_t>(MROWS, M - m0));
  const int64_t k0 = static_cast<int64_t>(wave) * KC;

  bf16x8_v wf[NB][NSTEP];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int64_t wr = r < 8 ? j0 + 8 * nb + r : inter + j0 + 8 * nb + (r - 8);
    load_w(wf[nb], w + wr * K + 8 * g, k0);
  }
  bf16x8_v xf[MBS][NSTEP];
#pragma unroll
  for (int mb = 0; mb < MBS; ++mb) {
    const int64_t row = min<int64_t>(m0 + 16 * mb + r, M - 1);  // clamped rows are dropped
#pragma unroll
    for (int s = 0; s < NSTEP; ++s) xf[mb][s] = ld_frag(x + row * K + k0 + KSTEP * s + 8 * g);
  }
  // Every load is issued before the first MFMA (one memory latency per workgroup; left to
  // itself the compiler interleaves loads and MFMAs and waits on each group).
  __builtin_amdgcn_sched_barrier(0);
  f32x4_v acc[NB][MBS];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) acc[nb][mb] = f32x4_v{0.0f, 0.0f, 0.0f, 0.0f};
  }
#pragma unroll
  for (int s = 0; s < NSTEP; ++s) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
      for (int mb = 0; mb < MBS; ++mb)
        acc[nb][mb] =
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[mb][s], wf[nb][s], acc[nb][mb], 0, 0, 0);
    }
  }
  // Lane holds rows 16 mb + 4 g + i of column block nb, column r.
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
    for (int mb = 0; mb < MBS; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sacc[wave][(16 * mb + 4 * g + i) * SS + 16 * nb + r] = acc[nb][mb][i];
    }
  }
  __syncthreads();
  // 64 rows x 8 NB outputs, two adjacent outputs per thread per pass.
  for (int o = threadIdx.x; o < MBS * 16 * 4 * NB; o += NCH * 64) {
    const int row = o / (4 * NB);
    const int q = o % (4 * NB);
    const int nb = q >> 2;
    const int col = 2 * (q & 3);  // within the block's 8 gate columns
    if (row >= mrows) continue;
    const int base = row * SS + 16 * nb + col;
    float y[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      float gs = sacc[0][base + e];
      float us = sacc[0][base + 8 + e];
#pragma unroll
      for (int c = 1; c < NCH; ++c) {
        gs += sacc[c][base + e];
        us += sacc[c][base + 8 + e];
      }
      y[e] = silu_mul1(round_bf16(gs), round_bf16(us));
    }
    *reinterpret_cast<uint32_t*>(out + (m0 + row) * inter + j0 + 8 * nb + col) =
        pack_bf16x2(y[0], y[1]);
  }
}

}  // namespace
}  // namespace sid

using namespace sid;

extern "C" int sid_linear_tile(int64_t m, int64_t n) {
  constexpr int shape[4] = {256 << 16 | 128, 128 << 16 | 128, 128 << 16 | 64, 64 << 16 | 64};
  return m > 0 && n > 0 ? shape[tile_shape(m, n)] : 0;
}

extern "C" int sid_linear(const void* x, int64_t ldx, const void* w, const void* bias, void* y,
                          int64_t m, int64_t n, int64_t k, int out_fp32, void* stream) {
  SID_REQUIRE(m >= 0 && n >= 0 && k >= 0, "linear: negative size");
  if (m == 0 || n == 0) return SID_OK;
  SID_REQUIRE(y != nullptr, "linear: null output");
  int rc = check_shapes(x, ldx, w, m, n, k, "linear");
  if (rc != SID_OK) return rc;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  // The streaming kernel reads the weights once per 64-row group; past one group the tile
  // kernel is faster (M = 128, 151936 x 1024 fp32 logits 165 vs 90 us, identical bits), and
  // below kStreamMinN columns at any M: its loads run up to four sub-tiles ahead where the
  // row-group kernel waits for each chunk. Weights from HBM, row group vs tiles, us:
  // 1 x 1024 x 2048 15.4 vs 7.9, 32 x 1024 x 3072 29.9 vs 10.8, 16 x 4096 x 1024 10.6 vs 6.7,
  // 63 x 12288 x 4096 59.7 vs 24.2, 1 x 64 x 512 5.8 vs 3.5.
  if (m <= MROWS && stream_shape_ok(m, n, k) && n >= kStreamMinN) {
    launch_stream<false>(x, ldx, w, bias, y, static_cast<int>(m), static_cast<int>(n), out_fp32,
                         nullptr, nullptr, s);
  } else if (tiles_fit(ldx, m, n, k)) {
    launch_tiles<EPI_Y>(x, ldx, w, m, n, k, tile_out(y, bias, out_fp32), s);
  } else {
    const dim3 grid((unsigned)(n / 64), 1u, (unsigned)((m + MROWS - 1) / MROWS));
    hipLaunchKernelGGL((linear_kernel<4, false>), grid, dim3(256), 0, s, (const bf16_t*)x, ldx,
                       (const bf16_t*)w, (const bf16_t*)bias, y, m, n, k, out_fp32, nullptr,
                       nullptr);
  }
  return check_launch("linear");
}

extern "C" int sid_linear_partials(const void* x, int64_t ldx, const void* w, float* partials,
                                   int64_t m, int64_t n, int64_t k, void* stream) {
  SID_REQUIRE(m >= 0 && n >= 0 && k >= 0, "linear_partials: negative size");
  if (m == 0 || n == 0) return SID_OK;
  SID_REQUIRE(partials != nullptr, "linear_partials: null output");
  int rc = check_shapes(x, ldx, w, m, n, k, "linear_partials");
  if (rc != SID_OK) return rc;
  SID_REQUIRE(k / KC <= 65535, "linear_partials: too many chunks");
  // Row groups of 64; a single group smaller than 64 rows gets the matching MBS.
  const int mbs = m >= MROWS ? 4 : static_cast<int>((m + 15) / 16);
  const dim3 grid((unsigned)(n / 64), (unsigned)(k / KC), (unsigned)((m + MROWS - 1) / MROWS));
  const hipStream_t s = static_cast<hipStream_t>(stream);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, (const bf16_t*)x, ldx, (const bf16_t*)w, m, n, k,
                       partials);
  };
  switch (mbs) {
    case 1: go(linear_chunk_kernel<4, 1>); break;
    case 2: go(linear_chunk_kernel<4, 2>); break;
    case 3: go(linear_chunk_kernel<4, 3>); break;
    default: go(linear_chunk_kernel<4, 4>); break;
  }
  return check_launch("linear_partials");
}

// sid_linear_argmax: up to one 64-row group streams the weights once (linear_stream_kernel,
// one candidate per workgroup); more rows take the tiled GEMM with the argmax epilogue (one
// candidate per 128-column tile, no logits needed: verify pass, 128 rows x 151936,
// 85 us; with logits 90 + argmax_rows 32). Both reduce with argmax_finalize_kernel. The
// workspace holds cu_count() * STREAM_WAVES candidates per row, which bounds the tiled
// path's column tiles.
static bool argmax_streams(int64_t m, int64_t n, int64_t k) {
  return m <= MROWS && stream_shape_ok(m, n, k);
}

static int64_t argmax_candidates() { return static_cast<int64_t>(cu_count()) * STREAM_WAVES; }

extern "C" int64_t sid_linear_argmax_workspace_bytes(int64_t m) {
  if (m < 1 || (m + MROWS - 1) / MROWS > 65535) return 0;
  return argmax_candidates() * m * static_cast<int64_t>(sizeof(float) + sizeof(int));
}

extern "C" int sid_linear_argmax(const void* x, int64_t ldx, const void* w, const void* bias,
                                 float* logits, int64_t m, int64_t n, int64_t k, void* workspace,
                                 int64_t workspace_bytes, int64_t* out_idx, void* stream) {
  SID_REQUIRE(m >= 0 && n >= 0 && k >= 0, "linear_argmax: negative size");
  if (m == 0) return SID_OK;
  SID_REQUIRE(n > 0, "linear_argmax: no columns");
  SID_REQUIRE(out_idx != nullptr && workspace != nullptr, "linear_argmax: null pointer");
  int rc = check_shapes(x, ldx, w, m, n, k, "linear_argmax");
  if (rc != SID_OK) return rc;
  const int64_t need = sid_linear_argmax_workspace_bytes(m);
  SID_REQUIRE(need > 0 && workspace_bytes >= need, "linear_argmax: workspace %lld bytes, need %lld",
              (long long)workspace_bytes, (long long)need);
  SID_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
              "linear_argmax: workspace must be 16-byte aligned");
  const int64_t cands = argmax_candidates();
  float* bv = static_cast<float*>(workspace);
  int* bi = reinterpret_cast<int*>(bv + cands * m);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  int used;
  if (argmax_streams(m, n, k)) {
    launch_stream<true>(x, ldx, w, bias, logits, static_cast<int>(m), static_cast<int>(n), 1, bv,
                        bi, s);
    used = cu_count();
  } else if (k >= (1ll << 23)) {
    // Weight rows past the tile kernel's 32-bit offsets; one candidate per 16 columns.
    SID_REQUIRE(n / 16 <= cands, "linear_argmax: N=%lld has more than %lld column blocks",
                (long long)n, (long long)cands);
    const dim3 grid((unsigned)(n / 64), 1u, (unsigned)((m + MROWS - 1) / MROWS));
    hipLaunchKernelGGL((linear_kernel<4, true>), grid, dim3(256), 0, s, (const bf16_t*)x, ldx,
                       (const bf16_t*)w, (const bf16_t*)bias, logits, m, n, k, 1, bv, bi);
    used = static_cast<int>(n / 16);
  } else {
    const int64_t tiles = (n + 127) / 128;
    SID_REQUIRE(tiles <= cands, "linear_argmax: N=%lld has more than %lld column tiles",
                (long long)n, (long long)cands);
    SID_REQUIRE((m + 127) / 128 <= 65535, "linear_argmax: too many rows");
    TileOut out = tile_out(logits, bias, 1);
    out.best_val = bv;
    out.best_idx = bi;
    out.sp.cand_rows = m;
    launch_head_tiles<EPI_ARGMAX>(x, ldx, w, m, n, k, out, s);
    used = static_cast<int>(tiles);
  }
  rc = check_launch("linear_argmax");
  if (rc != SID_OK) return rc;
  hipLaunchKernelGGL(argmax_finalize_kernel, dim3((unsigned)m), dim3(256), 0, s, bv, bi, used,
                     static_cast<int>(m), out_idx);
  return check_launch("linear_argmax finalize");
}

// Workspace of sid_linear_sample: 6 per-(wave, row) statistics + the finalize's lists.
static int64_t sample_ws_bytes(int64_t m) {
  const int64_t waves = static_cast<int64_t>(cu_count()) * STREAM_WAVES;
  return waves * m * 4 * 7;
}

// Rows one sid_linear_sample call takes: the streaming grouping up to kStreamMaxM, the
// 128-column tiles up to this many (prefill / verify passes of large batches).
constexpr int64_t kTiledSampleMaxM = 4096;

extern "C" int64_t sid_linear_sample_workspace_bytes(int64_t m) {
  if (m < 1 || m > kTiledSampleMaxM) return 0;
  return sample_ws_bytes(m);
}

template <int MBS>
static void launch_sample_mbs(const bf16_t* x, int64_t ldx, const void* w, int m, int n,
                              const float* temps, const int64_t* seeds, const int64_t* pos,
                              SampleStats st, int cand_rows, int row0, hipStream_t s) {
  const size_t lds = static_cast<size_t>(MBS * 16) * WXS * sizeof(bf16_t);
  static bool attr_set = false;
  if (!attr_set) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(&linear_sample_kernel<MBS>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    attr_set = true;
  }
  hipLaunchKernelGGL((linear_sample_kernel<MBS>), dim3(cu_count()), dim3(STREAM_WAVES * 64),
                     lds, s, x, ldx, (const bf16_t*)w, m, n, temps, seeds, pos, st, cand_rows,
                     row0);
}

// The streaming sampler reads the weights once per 64-row group; above this many rows (or
// when asked) the tiled GEMM with the sampler epilogue reads them once per 128-row tile
// (candidate groups: 128-column tiles instead of streaming waves). Measured at T = 0.7,
// 151936 x 1024, graph-timed (streaming vs tiled, us): 1 row 75 vs 97, 64 rows 112 vs
// 128, 96 rows 183 vs 144, 128 rows 199 vs 147, 200 rows 354 vs 234, 256 rows 378 vs 250.
constexpr int64_t kStreamSampleMaxM = 64;

extern "C" int sid_linear_sample(const void* x, int64_t ldx, const void* w, int64_t m, int64_t n,
                                 int64_t k, const float* temperatures, const int64_t* seeds,
                                 const int64_t* positions, void* workspace,
                                 int64_t workspace_bytes, int64_t* out_idx, float* logits,
                                 int flags, void* stream) {
  SID_REQUIRE(m >= 0 && n >= 0 && k >= 0, "linear_sample: negative size");
  SID_REQUIRE((flags & ~7) == 0 && (flags & 6) != 6, "linear_sample: bad flags %d", flags);
  if (m == 0) return SID_OK;
  SID_REQUIRE(n > 0, "linear_sample: no columns");
  SID_REQUIRE(out_idx && workspace && temperatures && seeds && positions,
              "linear_sample: null pointer");
  int rc = check_shapes(x, ldx, w, m, n, k, "linear_sample");
  if (rc != SID_OK) return rc;
  const bool tiled =
      (flags & 2) != 0 || ((flags & 4) == 0 && (m > kStreamSampleMaxM || logits != nullptr));
  SID_REQUIRE(stream_shape_ok(tiled ? 1 : m, n, k) && m <= kTiledSampleMaxM,
              "linear_sample: needs K == %d and 1 <= M <= %d (%d with the 128-column tiles); "
              "got M=%lld, K=%lld",
              WIDE_K, (int)kStreamMaxM, (int)kTiledSampleMaxM, (long long)m, (long long)k);
  const int64_t need = sample_ws_bytes(m);
  SID_REQUIRE(workspace_bytes >= need, "linear_sample: workspace %lld bytes, need %lld",
              (long long)workspace_bytes, (long long)need);
  SID_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
              "linear_sample: workspace must be 16-byte aligned");
  SID_REQUIRE(!(flags & 4) || logits == nullptr,
              "linear_sample: the streaming grouping writes no logits");
  const int stream_groups = cu_count() * STREAM_WAVES;
  const int groups = tiled ? static_cast<int>((n + 127) / 128) : stream_groups;
  SID_REQUIRE(groups <= stream_groups, "linear_sample: N=%lld has more than %d column tiles",
              (long long)n, stream_groups);
  const int64_t plane = static_cast<int64_t>(stream_groups) * m;
  float* base = static_cast<float*>(workspace);
  SampleStats st{base, base + plane, base + 2 * plane, base + 3 * plane, base + 4 * plane,
                 reinterpret_cast<int*>(base + 5 * plane)};
  int* redo = reinterpret_cast<int*>(base + 6 * plane);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int mi = static_cast<int>(m);
  if (tiled) {
    SID_REQUIRE((m + 127) / 128 <= 65535, "linear_sample: too many rows");
    TileOut out = tile_out(logits, nullptr, 1);
    out.sp = SampleIn{temperatures, seeds, positions, st, m};
    launch_head_tiles<EPI_SAMPLE>(x, ldx, w, m, n, k, out, s);
    rc = check_launch("linear_sample");
    if (rc != SID_OK) return rc;
  } else {
    for (int r0 = 0; r0 < mi; r0 += MROWS) {
      const int mg = min(MROWS, mi - r0);
      const bf16_t* xg = static_cast<const bf16_t*>(x) + static_cast<int64_t>(r0) * ldx;
      switch ((mg + 15) / 16) {
        case 1: launch_sample_mbs<1>(xg, ldx, w, mg, (int)n, temperatures, seeds, positions, st, mi, r0, s); break;
        case 2: launch_sample_mbs<2>(xg, ldx, w, mg, (int)n, temperatures, seeds, positions, st, mi, r0, s); break;
        case 3: launch_sample_mbs<3>(xg, ldx, w, mg, (int)n, temperatures, seeds, positions, st, mi, r0, s); break;
        default: launch_sample_mbs<4>(xg, ldx, w, mg, (int)n, temperatures, seeds, positions, st, mi, r0, s); break;
      }
      rc = check_launch("linear_sample");
      if (rc != SID_OK) return rc;
    }
  }
  hipLaunchKernelGGL(sample_finalize_kernel, dim3((unsigned)m), dim3(kFinThreads), 0, s,
                     (const bf16_t*)x, ldx, (const bf16_t*)w, (int)n, st, groups, mi,
                     temperatures, seeds, positions, redo, out_idx, flags & 1,
                     tiled ? 8 : 0);
  return check_launch("linear_sample finalize");
}

extern "C" int sid_linear_silu_mul(const void* x, const void* w, void* out, int64_t m, int64_t k,
                                   int64_t inter, void* stream) {
  SID_REQUIRE(m >= 0 && k >= 0 && inter >= 0, "linear_silu_mul: negative size");
  if (m == 0 || inter == 0) return SID_OK;
  SID_REQUIRE(x && w && out, "linear_silu_mul: null pointer");
  SID_REQUIRE(k == 4 * KC, "linear_silu_mul: K must be %d, got %lld", 4 * KC, (long long)k);
  SID_REQUIRE(inter % 8 == 0, "linear_silu_mul: intermediate size %lld not a multiple of 8",
              (long long)inter);
  SID_REQUIRE(inter / 8 <= 0x7fffffff && (m + MROWS - 1) / MROWS <= 65535,
              "linear_silu_mul: too large");
  SID_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(out) % 4 == 0,
              "linear_silu_mul: misaligned operand");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (m > kLinearSiluStreamMaxM && inter % 64 == 0 && tiles_fit(k, m, 2 * inter, k)) {
    // The tile kernel with the SwiGLU epilogue (grid over the 2 * inter projection columns;
    // the [M, 2 * inter] projection is never written). Same bits as the kernel below and as
    // sid_linear + sid_silu_mul.
    launch_tiles<EPI_SWIGLU>(x, k, w, m, 2 * inter, k, tile_out(out), s);
    return check_launch("linear_silu_mul");
  }
  const int mbs = m >= MROWS ? 4 : static_cast<int>((m + 15) / 16);
  // Two column blocks per wave halve the x read per output (M = 64, I = 3072, weights from
  // HBM: 12.3 -> 9.3 us); an I that is not a multiple of 16 takes one block per wave.
  const int nb = inter % 16 == 0 ? 2 : 1;
  const dim3 grid((unsigned)(inter / (8 * nb)), (unsigned)((m + MROWS - 1) / MROWS));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(4 * 64), 0, s, (const bf16_t*)x, (const bf16_t*)w, m,
                       inter, (bf16_t*)out);
  };
  if (nb == 2) {
    switch (mbs) {
      case 1: go(linear_silu_kernel<4, 1, 2>); break;
      case 2: go(linear_silu_kernel<4, 2, 2>); break;
      case 3: go(linear_silu_kernel<4, 3, 2>); break;
      default: go(linear_silu_kernel<4, 4, 2>); break;
    }
  } else {
    switch (mbs) {
      case 1: go(linear_silu_kernel<4, 1, 1>); break;
      case 2: go(linear_silu_kernel<4, 2, 1>); break;
      case 3: go(linear_silu_kernel<4, 3, 1>); break;
      default: go(linear_silu_kernel<4, 4, 1>); break;
    }
  }
  return check_launch("linear_silu_mul");
}
