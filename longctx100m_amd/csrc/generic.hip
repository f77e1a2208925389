// fp32-math attention kernels for any head_dim <= 256 and fp32 or bf16
// inputs, on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: full fp32 products
// and sums).  They carry the reference's exact arithmetic (fp32 scores, fp32
// probabilities, fp32 accumulation; bf16 inputs are upcast on load, the
// Python twin's rule at src/longctx100m/ring_attention.py:17,28) and serve the
// fp32 path, LC_FLAG_PRECISE, and head dims the bf16 kernels do not take.
//   forward: online softmax exactly as online_update
//            (rust/longctx100m-model/src/ring_attention.rs:15-55).
//   dQ     : rs:433-454 (pass 2 of the reference backward).
//   dK/dV  : rs:383-409 (pass 1), summed over the GQA group in the workgroup.
//
// Work split.  A wave owns 16 * NB stationary rows (queries in the forward and
// dQ, 16 keys in dK/dV) and streams 16-row tiles of the other operand straight
// from global memory into registers: at fp32 a 16 x 16 tile of one product is
// DP / 4 MFMAs of 32 cycles, so a tile's 8 KB per operand (head_dim 128) come
// from L1/L2 well within its MFMA time and LDS staging with its barriers would
// only add latency.  The streamed range is interleaved over several waves of
// the workgroup when the stationary rows alone do not fill the chip; their
// partial results meet in LDS.
//
// Operand layouts (lane l: c = l % 16, g = l / 16; MFMA k-slot = g):
//   row fragment r[j]    = X[c][16 j + 4 g .. + 3]: A or B operand whose k
//                          index is the head dim, element t used by MFMA (j, t);
//   column fragment x[i][db] = X[4 g + i][NJ c + db]: A operand X^T whose k
//                          index is the tile row 4 g + i, M index c = dim NJ c + db;
//   score element i      = S[tile row 4 g + i][stationary row c], which is the
//                          B operand of the product with the column fragments;
//   accumulator acc[db][i] = element (dim NJ (4 g + i) + db) of stationary row c.
// (NJ = DP / 16; DP is head_dim rounded up to 16, 32, 64, 96, 128 or 256; dims
// past head_dim are zeros.)
//
// Bound by the fp32 matrix cores (157 TFLOP/s; a library fp32 GEMM reaches
// 152).  Measured, causal, 4,096 tokens x 16 heads of 128: forward 22.0 ms
// with per-lane dot products on the VALU -> 1.30 ms here (53 TFLOP/s), dQ
// 18.0 -> 1.25 ms (82), dK/dV 39.2 -> 1.54 ms (89).  Small problems are bound
// by latency: two ranks of 512 tokens, 9/3 heads of 64, forward of both and
// one backward 6.28 -> 0.17 ms.
#include "common.h"
#include "kernels.h"

#include <type_traits>

namespace lc {
namespace {

struct GenArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* dout;
  const float* lse2;
  const float* delta;
  float* o;
  float* m;
  float* l;
  float* dq;
  float* dk;
  float* dv;
  int B, Nq, Nk, Hq, Hkv, D, group, n_tiles;
  int64_t q_pos0, k_pos0, valid;
  int causal;
  int accumulate;  // forward: merge into the running (o, m, l) instead of writing them
  int vec;         // rows can be loaded in vectors of up to four elements
  int split;       // waves of a workgroup that share its stationary rows (forward, dQ)
  float scale;
  int init;                      // backward: replace the accumulators' contents
  uint16_t *out, *dk16, *dv16;   // set: o (dQ), dK, dV go here as bf16 instead
};

__device__ __forceinline__ f32x4 mfma16x16x4(float a, float b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// W consecutive elements (W = 1, 2 or 4; p aligned to them) as fp32, in one
// load; the other elements of the result are zeros.
template <typename T, int W>
__device__ __forceinline__ f32x4 load_vec(const T* p) {
  f32x4 r = {0.f, 0.f, 0.f, 0.f};
  if constexpr (W == 1) {
    r[0] = load_f32(p);
  } else if constexpr (sizeof(T) == 4) {
    typedef float vt __attribute__((ext_vector_type(W)));
    const vt x = *reinterpret_cast<const vt*>(p);
#pragma unroll
    for (int e = 0; e < W; ++e) r[e] = x[e];
  } else {
    uint2 u = {0u, 0u};
    if constexpr (W == 2) u.x = *reinterpret_cast<const uint32_t*>(p);
    else u = *reinterpret_cast<const uint2*>(p);
    r = f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u),
              __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u)};
  }
  return r;
}

// The same of dims d0 .. d0 + W - 1 of a row whose dims at or past D are zeros
// and are not read; in single elements unless vec (which implies D % 4 == 0).
template <typename T, int W>
__device__ __forceinline__ f32x4 load_w(const T* row, int d0, int D, bool vec) {
  f32x4 r = {0.f, 0.f, 0.f, 0.f};
  if (vec) {
    if (d0 < D) r = load_vec<T, W>(row + d0);
  } else {
#pragma unroll
    for (int e = 0; e < W; ++e)
      if (d0 + e < D) r[e] = load_f32(row + d0 + e);
  }
  return r;
}

// Row fragments of the 16 rows from row0 (rows at or past nrows are zeros).
template <typename T, int NJ>
__device__ __forceinline__ void load_rows(f32x4 (&r)[NJ], const T* base, int64_t stride, int row0,
                                          int nrows, int D, bool vec, int c, int g) {
  const int row = row0 + c;
  if (vec && D == 16 * NJ && row0 + 16 <= nrows) {  // uniform: a whole tile, no checks per load
    const T* p = base + (int64_t)row * stride + 4 * g;
#pragma unroll
    for (int j = 0; j < NJ; ++j) r[j] = load_vec<T, 4>(p + 16 * j);
  } else {
    const bool ok = row < nrows;
    const T* p = base + (int64_t)(ok ? row : 0) * stride;
#pragma unroll
    for (int j = 0; j < NJ; ++j) r[j] = load_w<T, 4>(p, ok ? 16 * j + 4 * g : D, D, vec);
  }
}

// Column fragments of the 16 rows from row0 (rows at or past nrows are zeros).
template <typename T, int NJ>
__device__ __forceinline__ void load_cols(float (&x)[4][NJ], const T* base, int64_t stride,
                                          int row0, int nrows, int D, bool vec, int c, int g) {
  constexpr int W = NJ % 4 == 0 ? 4 : (NJ % 2 == 0 ? 2 : 1);
  const bool whole = vec && D == 16 * NJ && row0 + 16 <= nrows;
  if (whole) {
    const T* p = base + (int64_t)(row0 + 4 * g) * stride + NJ * c;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < NJ / W; ++e) {
        const f32x4 r = load_vec<T, W>(p + i * stride + W * e);
#pragma unroll
        for (int k = 0; k < W; ++k) x[i][W * e + k] = r[k];
      }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = row0 + 4 * g + i;
      const bool ok = row < nrows;
      const T* p = base + (int64_t)(ok ? row : 0) * stride;
#pragma unroll
      for (int e = 0; e < NJ / W; ++e) {
        const f32x4 r = load_w<T, W>(p, ok ? NJ * c + W * e : D, D, vec);
#pragma unroll
        for (int k = 0; k < W; ++k) x[i][W * e + k] = r[k];
      }
    }
  }
}

// Keeps the loads of a phase from moving into an earlier one: each operand's
// registers are reloaded one phase after their last use, which is as far
// ahead as the register file allows at head_dim 128.
__device__ __forceinline__ void phase() { __builtin_amdgcn_sched_barrier(0); }

// S (or dP) of one 16 x 16 tile: rows of a against the stationary rows b.
// Two accumulators halve the dependent chain; PARTS restarts keep the sums as
// short as four-lane dot products have them (two: the output of 1,000 causal
// tokens, 32/8 heads of 128, is 2.8e-7 from float64, with one 3.1e-7).
template <int NJ, int PARTS, typename Frag>
__device__ __forceinline__ f32x4 score_tile(const f32x4 (&a)[NJ], const Frag& b) {
  constexpr int kPer = NJ >= PARTS ? NJ / PARTS : NJ;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j0 = 0; j0 < NJ; j0 += kPer) {
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int j = j0; j < j0 + kPer; ++j) {
      const f32x4 bj = b[j];
      s0 = mfma16x16x4(a[j][0], bj[0], s0);
      s1 = mfma16x16x4(a[j][1], bj[1], s1);
      s0 = mfma16x16x4(a[j][2], bj[2], s0);
      s1 = mfma16x16x4(a[j][3], bj[3], s1);
    }
    sum = j0 == 0 ? s0 + s1 : sum + (s0 + s1);
    if (j0 + kPer < NJ) phase();  // one part's registers at a time
  }
  return sum;
}

// Stationary row fragments: in registers, or (kLds) in LDS, one copy for the
// workgroup, each lane at its own 16 bytes of fragment j.
template <int NJ, bool kLds>
struct RowFrags {
  f32x4 r[NJ];
  __device__ __forceinline__ const f32x4& operator[](int j) const { return r[j]; }
};
template <int NJ>
struct RowFrags<NJ, true> {
  const f32x4* p;  // fragment j of lane l at p[64 j] (p already at the lane)
  __device__ __forceinline__ f32x4 operator[](int j) const { return p[64 * j]; }
};

template <int NJ>
__device__ __forceinline__ void accumulate_tile(f32x4 (&acc)[NJ], const float (&x)[4][NJ],
                                                const f32x4& p) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int db = 0; db < NJ; ++db) acc[db] = mfma16x16x4(x[i][db], p[i], acc[db]);
}

// Number of leading keys of the shard that the query at index row sees.
__device__ __forceinline__ int visible_keys(const GenArgs& a, int row) {
  int64_t n = min((int64_t)a.Nk, a.valid - a.k_pos0);
  if (a.causal) n = min(n, a.q_pos0 + row - a.k_pos0 + 1);
  return n < 0 ? 0 : (int)n;
}

// Waves per workgroup at most: eight, four at head_dim 256 (LDS and registers).
__host__ __device__ constexpr int max_waves(int nj) { return nj <= 8 ? 8 : 4; }

// Row pitch (floats) of a wave's partial accumulators in LDS: 16 rows of DP.
__host__ __device__ constexpr int part_pitch(int dp) { return dp + 4; }

template <int NJ>
__device__ __forceinline__ void store_part(float* part, const f32x4 (&acc)[NJ], int c, int g) {
  float* row = part + c * part_pitch(16 * NJ) + 4 * NJ * g;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int db = 0; db < NJ; ++db) row[NJ * i + db] = acc[db][i];
}

// ----------------------------------------------------------------- forward --

// Wave w of the workgroup: query block w / split, key tiles w % split, + split, ...
template <typename T, int NJ, int NB>
__global__ __launch_bounds__(64 * max_waves(NJ)) void fwd_generic_kernel(GenArgs a) {
  constexpr int DP = 16 * NJ;
  constexpr int kPart = 16 * part_pitch(DP);
  __shared__ __attribute__((aligned(16))) float smem[max_waves(NJ) * kPart];  // partial accumulators
  __shared__ float msm[max_waves(NJ) * 16], lsm[max_waves(NJ) * 16], mtop[max_waves(NJ) * 16];
  const int nw = blockDim.x >> 6;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;
  const int qsub = wave / a.split;
  const int ksub = wave - qsub * a.split;
  const int rows_wg = nw / a.split * 16 * NB;

  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int qt = a.n_tiles - 1 - L % a.n_tiles;  // long query tiles first
  const int bh = L / a.n_tiles;
  const int h = bh % a.Hq;
  const int b = bh / a.Hq;
  const int hk = h / a.group;
  const int D = a.D;
  const bool vec = a.vec != 0;

  const int64_t qs = (int64_t)a.Hq * D, ks = (int64_t)a.Hkv * D;
  const T* qb = static_cast<const T*>(a.q) + (int64_t)b * a.Nq * qs + (int64_t)h * D;
  const T* kb = static_cast<const T*>(a.k) + (int64_t)b * a.Nk * ks + (int64_t)hk * D;
  const T* vb = static_cast<const T*>(a.v) + (int64_t)b * a.Nk * ks + (int64_t)hk * D;

  const int q0 = qt * rows_wg + qsub * 16 * NB;  // the wave's first query
  f32x4 qr[NB][NJ], o[NB][NJ];
  float m[NB], l[NB];
  int klim[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    load_rows<T, NJ>(qr[n], qb, qs, q0 + 16 * n, a.Nq, D, vec, c, g);
#pragma unroll
    for (int j = 0; j < NJ; ++j) o[n][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[n] = -INFINITY;
    l[n] = 0.f;
    klim[n] = visible_keys(a, min(q0 + 16 * n + c, a.Nq - 1));
  }
  const int kend = q0 < a.Nq ? visible_keys(a, min(q0 + 16 * NB, a.Nq) - 1) : 0;
  const int ntiles = (kend + 15) / 16;

  f32x4 kr[NJ];
  float vc[4][NJ];
  if (ksub < ntiles) {
    load_rows<T, NJ>(kr, kb, ks, 16 * ksub, a.Nk, D, vec, c, g);
    load_cols<T, NJ>(vc, vb, ks, 16 * ksub, a.Nk, D, vec, c, g);
  }
  for (int t = ksub; t < ntiles; t += a.split) {
    f32x4 s[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      s[n] = score_tile<NJ, 2>(kr, qr[n]);
      phase();
    }
    const bool more = t + a.split < ntiles;
    phase();
    if (more) load_rows<T, NJ>(kr, kb, ks, 16 * (t + a.split), a.Nk, D, vec, c, g);
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      float bm = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = s[n][i] * a.scale;
        s[n][i] = 16 * t + 4 * g + i >= klim[n] ? -INFINITY : x;
        bm = fmaxf(bm, s[n][i]);
      }
      const float mnew = fmaxf(m[n], group4_max(bm));
      if (__any(mnew > m[n])) {  // elsewhere the factor is 1
        const float alpha = mnew > m[n] ? expf(m[n] - mnew) : 1.f;  // m = -inf: 0
        l[n] *= alpha;
#pragma unroll
        for (int j = 0; j < NJ; ++j) o[n][j] *= alpha;
        m[n] = mnew;
      }
      const float muse = mnew == -INFINITY ? 0.f : mnew;  // no key yet: p = 0
#pragma unroll
      for (int i = 0; i < 4; ++i) s[n][i] = expf(s[n][i] - muse);
      l[n] += (s[n][0] + s[n][1]) + (s[n][2] + s[n][3]);
    }
#pragma unroll
    for (int n = 0; n < NB; ++n) accumulate_tile<NJ>(o[n], vc, s[n]);
    phase();
    if (more) load_cols<T, NJ>(vc, vb, ks, 16 * (t + a.split), a.Nk, D, vec, c, g);
  }

  // The key splits of each query merge by log-sum-exp: every wave brings its
  // partial to the maximum of its query's splits, then takes every split-th
  // row of its query block and sums along the dims.  accumulate: the result
  // then merges into the running state of the row, with the arithmetic of
  // lc_attn_merge on the normalised partial.
  const int p0 = qsub * a.split;  // the query block's first wave
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const float ln = group4_sum(l[n]);
    float M = m[n];
    if (a.split > 1) {
      if (n > 0) __syncthreads();
      if (g == 0) msm[wave * 16 + c] = M;
      __syncthreads();
#pragma unroll
      for (int s = 0; s < max_waves(NJ); ++s)
        M = fmaxf(M, msm[(p0 + min(s, a.split - 1)) * 16 + c]);
    }
    const float f = m[n] == -INFINITY ? 0.f : expf(m[n] - M);  // 1 without splits
#pragma unroll
    for (int j = 0; j < NJ; ++j) o[n][j] *= f;
    if (n > 0) __syncthreads();
    store_part<NJ>(smem + wave * kPart, o[n], c, g);
    if (g == 0) {
      lsm[wave * 16 + c] = ln * f;
      if (ksub == 0) mtop[qsub * 16 + c] = M;
    }
    __syncthreads();
    for (int r = ksub; r < 16; r += a.split) {
      const int row = q0 + 16 * n + r;
      if (row >= a.Nq) break;
      M = mtop[qsub * 16 + r];
      float lt = 0.f;
#pragma unroll
      for (int s = 0; s < max_waves(NJ); ++s) {
        const float x = lsm[(p0 + min(s, a.split - 1)) * 16 + r];
        lt += s < a.split ? x : 0.f;
      }
      const float den = lt > kFltMin ? lt : kFltMin;
      const int64_t oi = (((int64_t)b * a.Nq + row) * a.Hq + h) * D;
      const int64_t si = ((int64_t)b * a.Hq + h) * a.Nq + row;
      MergeW w{};
      if (a.accumulate) w = merge_weights(a.m[si], a.l[si], M, lt);
      for (int d = lane; d < D; d += 64) {
        float acc = 0.f;
#pragma unroll
        for (int s = 0; s < max_waves(NJ); ++s) {
          const float x = smem[(p0 + min(s, a.split - 1)) * kPart + r * part_pitch(DP) + d];
          acc += s < a.split ? x : 0.f;
        }
        const float r = a.accumulate ? a.o[oi + d] * w.wa + (acc / den) * w.wb : acc / den;
        if (a.out != nullptr) a.out[oi + d] = f32_to_bf16(r);
        else a.o[oi + d] = r;
      }
      if (lane == 0) {
        a.m[si] = a.accumulate ? w.m : M;
        a.l[si] = a.accumulate ? w.l : lt;
      }
    }
  }
}

// ---------------------------------------------------------------------- dQ --

template <typename T, int NJ>
__global__ __launch_bounds__(64 * max_waves(NJ)) void dq_generic_kernel(GenArgs a) {
  constexpr int DP = 16 * NJ;
  constexpr int kPart = 16 * part_pitch(DP);
  __shared__ __attribute__((aligned(16))) float smem[max_waves(NJ) * kPart];  // partial accumulators
  const int nw = blockDim.x >> 6;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;
  const int qsub = wave / a.split;
  const int ksub = wave - qsub * a.split;
  const int rows_wg = nw / a.split * 16;

  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int qt = a.n_tiles - 1 - L % a.n_tiles;
  const int bh = L / a.n_tiles;
  const int h = bh % a.Hq;
  const int b = bh / a.Hq;
  const int hk = h / a.group;
  const int D = a.D;
  const bool vec = a.vec != 0;
  const float sl2 = a.scale * kLog2e;

  const int64_t qs = (int64_t)a.Hq * D, ks = (int64_t)a.Hkv * D;
  const T* qb = static_cast<const T*>(a.q) + (int64_t)b * a.Nq * qs + (int64_t)h * D;
  const T* ob = static_cast<const T*>(a.dout) + (int64_t)b * a.Nq * qs + (int64_t)h * D;
  const T* kb = static_cast<const T*>(a.k) + (int64_t)b * a.Nk * ks + (int64_t)hk * D;
  const T* vb = static_cast<const T*>(a.v) + (int64_t)b * a.Nk * ks + (int64_t)hk * D;

  const int q0 = qt * rows_wg + qsub * 16;
  const int kend_wg = visible_keys(a, min(qt * rows_wg + rows_wg, a.Nq) - 1);
  if (kend_wg == 0 && !a.init && a.out == nullptr) return;  // nothing visible: no contribution
  f32x4 qr[NJ], dor[NJ], acc[NJ];
  load_rows<T, NJ>(qr, qb, qs, q0, a.Nq, D, vec, c, g);
  load_rows<T, NJ>(dor, ob, qs, q0, a.Nq, D, vec, c, g);
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool ok = q0 + c < a.Nq;
  const int64_t si = ((int64_t)b * a.Hq + h) * a.Nq + q0 + c;
  const float lse = ok ? a.lse2[si] : INFINITY;
  const float dl = ok ? a.delta[si] : 0.f;
  const int klim = visible_keys(a, min(q0 + c, a.Nq - 1));
  const int kend = q0 < a.Nq ? visible_keys(a, min(q0 + 16, a.Nq) - 1) : 0;
  const int ntiles = (kend + 15) / 16;

  f32x4 kr[NJ], vr[NJ];
  if (ksub < ntiles) {
    load_rows<T, NJ>(kr, kb, ks, 16 * ksub, a.Nk, D, vec, c, g);
    load_rows<T, NJ>(vr, vb, ks, 16 * ksub, a.Nk, D, vec, c, g);
  }
  for (int t = ksub; t < ntiles; t += a.split) {
    const bool more = t + a.split < ntiles;
    const f32x4 s = score_tile<NJ, 2>(kr, qr);
    phase();
    float kc[4][NJ];
    load_cols<T, NJ>(kc, kb, ks, 16 * t, a.Nk, D, vec, c, g);
    const f32x4 dp = score_tile<NJ, 2>(vr, dor);
    phase();
    if (more) load_rows<T, NJ>(kr, kb, ks, 16 * (t + a.split), a.Nk, D, vec, c, g);
    f32x4 ds;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = 16 * t + 4 * g + i >= klim ? 0.f : fast_exp2(s[i] * sl2 - lse);
      ds[i] = p * (dp[i] - dl);
    }
    accumulate_tile<NJ>(acc, kc, ds);
    phase();
    if (more) load_rows<T, NJ>(vr, vb, ks, 16 * (t + a.split), a.Nk, D, vec, c, g);
  }

  store_part<NJ>(smem + wave * kPart, acc, c, g);
  __syncthreads();
  for (int r = ksub; r < 16; r += a.split) {
    const int row = q0 + r;
    if (row >= a.Nq) break;
    const int64_t qi = (((int64_t)b * a.Nq + row) * a.Hq + h) * D;
    for (int d = lane; d < D; d += 64) {
      float sum = 0.f;
#pragma unroll
      for (int s = 0; s < max_waves(NJ); ++s) {
        const float x = smem[(qsub * a.split + min(s, a.split - 1)) * kPart + r * part_pitch(DP) + d];
        sum += s < a.split ? x : 0.f;
      }
      grad1(a.dq, a.out, a.init, qi + d, sum * a.scale);
    }
  }
}

// ------------------------------------------------------------------- dK/dV --

constexpr int64_t kGridRow = int64_t(1) << 22;

// Workgroup = 16 keys of one KV head; its waves take the steps (query head of
// the group, 16-query tile) in turn.
template <typename T, int NJ>
__global__ __launch_bounds__(64 * max_waves(NJ)) void dkdv_generic_kernel(GenArgs a) {
  constexpr int DP = 16 * NJ;
  constexpr int kPart = 16 * part_pitch(DP);
  __shared__ __attribute__((aligned(16))) float smem[max_waves(NJ) * kPart];  // dK's partials, then dV's
  // From head_dim 97 on K and V stay in LDS during the walk (in the space of
  // the partials): with dK and dV they would take all the registers of two
  // waves per SIMD.
  constexpr bool kKvLds = NJ >= 8;
  f32x4* kvsm = reinterpret_cast<f32x4*>(smem);  // K fragments, then V fragments
  static_assert(2 * 64 * NJ * 4 <= max_waves(NJ) * kPart, "K and V fit in the partials' space");
  const int nw = blockDim.x >> 6;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;

  // Grid rows of kGridRow workgroups: 16-key tiles of a large problem exceed
  // the 2^32 threads of one grid dimension.
  const int64_t L = (int64_t)blockIdx.y * kGridRow + xcd_remap(blockIdx.x, gridDim.x);
  const int64_t bh = L / a.n_tiles;
  if (bh >= (int64_t)a.B * a.Hkv) return;
  const int kt = (int)(L - bh * a.n_tiles);  // early keys see the most queries: dispatched first
  const int hk = (int)(bh % a.Hkv);
  const int b = (int)(bh / a.Hkv);
  const int D = a.D;
  const bool vec = a.vec != 0;
  const float sl2 = a.scale * kLog2e;
  const int k0 = 16 * kt;

  const int64_t qs = (int64_t)a.Hq * D, ks = (int64_t)a.Hkv * D;
  const T* kb = static_cast<const T*>(a.k) + (int64_t)b * a.Nk * ks + (int64_t)hk * D;
  const T* vb = static_cast<const T*>(a.v) + (int64_t)b * a.Nk * ks + (int64_t)hk * D;

  // Queries that see any key of the tile.
  const int64_t kp_first = a.k_pos0 + k0;
  int qstart = 0;
  if (a.causal) {
    const int64_t first = kp_first - a.q_pos0;
    qstart = first <= 0 ? 0 : (first >= a.Nq ? a.Nq : (int)first);
  }
  qstart = qstart / 16 * 16;
  const int ntq = kp_first < a.valid ? (a.Nq - qstart + 15) / 16 : 0;
  if (ntq <= 0 && !a.init && a.dk16 == nullptr) return;  // no visible pair: no contribution
  const int nsteps = ntq * a.group;
  // First query that sees the lane's key.
  int rmin = 0;
  if (k0 + c >= a.Nk || kp_first + c >= a.valid) {
    rmin = a.Nq;
  } else if (a.causal) {
    const int64_t first = kp_first + c - a.q_pos0;
    rmin = first <= 0 ? 0 : (first >= a.Nq ? a.Nq : (int)first);
  }

  RowFrags<NJ, kKvLds> kr, vr;
  if constexpr (kKvLds) {
    if (wave < 2) {  // the workgroup's K (wave 0) and V (wave 1)
      f32x4 x[NJ];
      load_rows<T, NJ>(x, wave == 0 ? kb : vb, ks, k0, a.Nk, D, vec, c, g);
#pragma unroll
      for (int j = 0; j < NJ; ++j) kvsm[64 * (NJ * wave + j) + lane] = x[j];
    }
    kr.p = kvsm + lane;
    vr.p = kvsm + 64 * NJ + lane;
    __syncthreads();
  } else {
    load_rows<T, NJ>(kr.r, kb, ks, k0, a.Nk, D, vec, c, g);
    load_rows<T, NJ>(vr.r, vb, ks, k0, a.Nk, D, vec, c, g);
  }
  f32x4 dk[NJ], dv[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) dk[j] = dv[j] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 qr[NJ], dor[NJ];
  auto qbase = [&](int step) {
    return static_cast<const T*>(a.q) + (int64_t)b * a.Nq * qs + (int64_t)(hk * a.group + step / ntq) * D;
  };
  auto obase = [&](int step) {
    return static_cast<const T*>(a.dout) + (int64_t)b * a.Nq * qs + (int64_t)(hk * a.group + step / ntq) * D;
  };
  auto qrow = [&](int step) { return qstart + 16 * (step % ntq); };
  if (wave < nsteps) {
    load_rows<T, NJ>(qr, qbase(wave), qs, qrow(wave), a.Nq, D, vec, c, g);
    load_rows<T, NJ>(dor, obase(wave), qs, qrow(wave), a.Nq, D, vec, c, g);
  }
  for (int step = wave; step < nsteps; step += nw) {
    const int next = step + nw;
    const int qrow0 = qrow(step);
    float lse[4], dl[4];
    const int64_t si = ((int64_t)b * a.Hq + hk * a.group + step / ntq) * a.Nq;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = qrow0 + 4 * g + i;
      const bool ok = row < a.Nq;
      lse[i] = ok ? a.lse2[si + row] : INFINITY;
      dl[i] = ok ? a.delta[si + row] : 0.f;
    }
    const f32x4 s = score_tile<NJ, 2>(qr, kr);
    phase();
    float oc[4][NJ], qc[4][NJ];
    load_cols<T, NJ>(oc, obase(step), qs, qrow0, a.Nq, D, vec, c, g);
    const f32x4 dp = score_tile<NJ, NJ <= 4 ? 2 : 1>(dor, vr);
    phase();
    load_cols<T, NJ>(qc, qbase(step), qs, qrow0, a.Nq, D, vec, c, g);
    f32x4 p, ds;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = qrow0 + 4 * g + i < rmin ? 0.f : fast_exp2(s[i] * sl2 - lse[i]);
      ds[i] = p[i] * (dp[i] - dl[i]);
    }
    accumulate_tile<NJ>(dv, oc, p);
    phase();
    if (next < nsteps) load_rows<T, NJ>(qr, qbase(next), qs, qrow(next), a.Nq, D, vec, c, g);
    accumulate_tile<NJ>(dk, qc, ds);
    phase();
    if (next < nsteps) load_rows<T, NJ>(dor, obase(next), qs, qrow(next), a.Nq, D, vec, c, g);
  }

  // Sum of the waves' partials; thread (row, dims) of the workgroup.
  auto reduce = [&](const f32x4 (&acc)[NJ], float* dst, uint16_t* out, float scale) {
    store_part<NJ>(smem + wave * kPart, acc, c, g);
    __syncthreads();
    for (int r = wave; r < 16 && k0 + r < a.Nk; r += nw) {
      const int64_t ki = (((int64_t)b * a.Nk + k0 + r) * a.Hkv + hk) * D;
      for (int d = lane; d < D; d += 64) {
        const float old = a.init ? 0.f : dst[ki + d];  // on its way during the sum
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < max_waves(NJ); ++w) {
          const float x = smem[min(w, nw - 1) * kPart + r * part_pitch(DP) + d];
          sum += w < nw ? x : 0.f;
        }
        const float x = old + sum * scale;
        if (out != nullptr) out[ki + d] = f32_to_bf16(x);
        else dst[ki + d] = x;
      }
    }
  };
  if constexpr (kKvLds) __syncthreads();  // every wave is done with K and V
  reduce(dk, a.dk, a.dk16, a.scale);
  __syncthreads();
  reduce(dv, a.dv, a.dv16, 1.f);
}

// Waves the chip holds at two per SIMD, the occupancy of these kernels.
constexpr int64_t kWaveSlots = 2048;

// How many waves share each block of stationary rows: enough, up to the
// largest workgroup, to fill the chip, but none without two tiles to stream
// (512 queries x 9 heads over 512 keys of 64 dims: forward 40 us with one
// wave per block, 19-20 us with four or eight; dQ 50 us against 22-27).
int split_for(int64_t blocks, int64_t tiles, int most) {
  int s = 1;
  while (s < most && blocks * s < kWaveSlots && tiles >= 4 * s) s *= 2;
  return s;
}

GenArgs make_args(const Problem& p, const void* q, const void* k, const void* v,
                  const void* dout) {
  GenArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.dout = dout;
  a.B = p.B;
  a.Nq = p.Nq;
  a.Nk = p.Nk;
  a.Hq = p.Hq;
  a.Hkv = p.Hkv;
  a.D = p.D;
  a.group = p.Hq / p.Hkv;
  a.q_pos0 = p.q_pos0;
  a.k_pos0 = p.k_pos0;
  a.valid = p.valid;
  a.causal = p.causal ? 1 : 0;
  a.accumulate = p.accumulate ? 1 : 0;
  a.scale = p.scale;
  a.split = 1;
  // Vectors of four elements: every row of every operand starts aligned to them.
  const uintptr_t all = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                        reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(dout);
  a.vec = p.D % 4 == 0 && (all & (p.dtype == 1 ? 7u : 15u)) == 0;
  return a;
}

// Calls f with integral constants <bf16 inputs, head_dim blocks of 16>.
template <typename F>
void dispatch(const Problem& p, const F& f) {
  auto by_dim = [&](auto tag) {
    using T = decltype(tag);
    if (p.D <= 16) f(T{}, std::integral_constant<int, 1>{});
    else if (p.D <= 32) f(T{}, std::integral_constant<int, 2>{});
    else if (p.D <= 64) f(T{}, std::integral_constant<int, 4>{});
    else if (p.D <= 96) f(T{}, std::integral_constant<int, 6>{});
    else if (p.D <= 128) f(T{}, std::integral_constant<int, 8>{});
    else f(T{}, std::integral_constant<int, 16>{});
  };
  if (p.dtype == 1) by_dim(uint16_t{});
  else by_dim(float{});
}

}  // namespace

hipError_t launch_fwd_generic(const Problem& p, const void* q, const void* k, const void* v,
                              float* o, float* m, float* l, hipStream_t s, uint16_t* out) {
  if (p.D > 256) return hipErrorInvalidValue;
  GenArgs a = make_args(p, q, k, v, nullptr);
  a.out = out;
  a.o = o;
  a.m = m;
  a.l = l;
  dispatch(p, [&](auto tag, auto nj) {
    using T = decltype(tag);
    constexpr int NJ = decltype(nj)::value;
    const int64_t heads = (int64_t)p.B * p.Hq, blocks = heads * ((p.Nq + 15) / 16);
    // Two 16-query blocks per wave (each key tile loaded once for both) once
    // the waves fill the chip anyway.
    const bool two = NJ <= 8 && blocks >= 2 * kWaveSlots;
    a.split = two ? 1 : split_for(blocks, (p.Nk + 15) / 16, max_waves(NJ));
    const int nw = a.split > 4 ? a.split : 4;
    const int rows = nw / a.split * (two ? 32 : 16);
    a.n_tiles = (p.Nq + rows - 1) / rows;
    const dim3 grid((unsigned)(a.n_tiles * heads)), block(64 * nw);
    if (two)
      hipLaunchKernelGGL((fwd_generic_kernel<T, NJ, NJ <= 8 ? 2 : 1>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((fwd_generic_kernel<T, NJ, 1>), grid, block, 0, s, a);
  });
  return hipGetLastError();
}

hipError_t launch_bwd_dq_generic(const Problem& p, const void* q, const void* k, const void* v,
                                 const void* dout, const float* lse2, const float* delta,
                                 float* dq, hipStream_t s, const Sink& to) {
  if (p.D > 256) return hipErrorInvalidValue;
  GenArgs a = make_args(p, q, k, v, dout);
  a.init = to.init;
  a.out = to.out;
  a.lse2 = lse2;
  a.delta = delta;
  a.dq = dq;
  dispatch(p, [&](auto tag, auto nj) {
    using T = decltype(tag);
    constexpr int NJ = decltype(nj)::value;
    const int64_t heads = (int64_t)p.B * p.Hq;
    a.split = split_for(heads * ((p.Nq + 15) / 16), (p.Nk + 15) / 16, max_waves(NJ));
    const int nw = a.split > 4 ? a.split : 4;
    const int rows = nw / a.split * 16;
    a.n_tiles = (p.Nq + rows - 1) / rows;
    hipLaunchKernelGGL((dq_generic_kernel<T, NJ>), dim3((unsigned)(a.n_tiles * heads)),
                       dim3(64 * nw), 0, s, a);
  });
  return hipGetLastError();
}

hipError_t launch_bwd_dkdv_generic(const Problem& p, const void* q, const void* k, const void* v,
                                   const void* dout, const float* lse2, const float* delta,
                                   float* dk, float* dv, hipStream_t s, const Sink& to) {
  if (p.D > 256) return hipErrorInvalidValue;
  GenArgs a = make_args(p, q, k, v, dout);
  a.init = to.init;
  a.dk16 = to.out;
  a.dv16 = to.out2;
  a.lse2 = lse2;
  a.delta = delta;
  a.dk = dk;
  a.dv = dv;
  dispatch(p, [&](auto tag, auto nj) {
    using T = decltype(tag);
    constexpr int NJ = decltype(nj)::value;
    a.n_tiles = (p.Nk + 15) / 16;
    const int64_t blocks = (int64_t)a.n_tiles * p.Hkv * p.B;
    const int nw = blocks * 4 < kWaveSlots ? max_waves(NJ) : 4;
    const dim3 grid((unsigned)(blocks < kGridRow ? blocks : kGridRow),
                    (unsigned)((blocks + kGridRow - 1) / kGridRow));
    hipLaunchKernelGGL((dkdv_generic_kernel<T, NJ>), grid, dim3(64 * nw), 0, s, a);
  });
  return hipGetLastError();
}

}  // namespace lc
