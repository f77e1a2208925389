// One ring hop for head_dim 64 on bf16 MFMA (gfx950 v_mfma_f32_32x32x16_bf16,
// fp32 accumulation): forward, dQ and dK/dV.
//
// Semantics: the reference's tiled online-softmax update over one KV shard and
// its finalize (rust/longctx100m-model/src/ring_attention.rs:15-106, :195-219,
// :227), and its recomputing backward (rs:383-409, :433-454):
//   P  = 2^(s*scale*log2e - lse2), dS = P * (dO V^T - delta),
//   dQ += dS K * scale,  dK += dS^T Q * scale,  dV += P^T dO
// Deterministic: every output element has one owner per launch, no atomics.
//
// Work split.  At head_dim 64 a tile is small (32 rows are 4 KB) and its
// softmax costs as much as its MFMAs, so every wave works alone: it owns 32
// stationary rows (64 in the large forward and dQ, so that each LDS read
// feeds two MFMAs) and streams 32-row tiles of the other side through its own
// double-buffered LDS by LDS DMA, with no barrier in the walk.  The streamed
// range (in dK/dV the query heads of the GQA group times their tiles) is
// interleaved over `split` waves of the workgroup when the stationary rows
// alone do not fill the chip; their partials meet in LDS at the end.
//
// LDS tiles: 32 rows of 128 bytes; row r's eight 16-byte chunks stored at
// chunk ^ ((r >> 1) & 7).  With gfx950's LDS service rules (tile128.h) both
// reads are free of bank conflicts: ds_read_b128 of one chunk of 32 rows (its
// 16 rows per cycle hold, per parity, eight distinct r >> 1 modulo 8), and
// transposed reads of rows {a, a+1, a+8, a+9} x 64 bytes (rows eight apart
// differ in chunk bit 2).
//
// Operand layouts (lane l, c = l % 32, hh = l / 32; MFMA layouts in common.h):
//   row operand, k-step t    X[c][16t + 8hh .. +7]
//   score element v          S[8(v/4) + 4hh + v%4][c]: tile row x stationary row
//   as a B operand, k-step u (tile rows 16u ..) slot 4p + t takes element
//   8u + 2p + t%2 + 4(t/2), and the transposed A operand reads the same rows.
//
// Bound by instruction issue: per wave and 32 x 32 tile the MFMAs (256 cycles
// in the forward, 384 in dQ, 512 in dK/dV) and the softmax's VALU work (about
// 450) hardly overlap; waits for the DMA are 2-8% of the walk.  Measured,
// causal, against workgroups of four 32-row waves sharing register-staged
// tiles, 16x16x32 MFMA (GPU time of a call): 2 x 2,047 tokens, 9/3 heads, forward
// 66 -> 36 us, dQ 105 -> 39, dK/dV 421 -> 42; 4,096 tokens, 32/8 heads 167 -> 120,
// 365 -> 141, 1130 -> 191; 16,384 tokens, 16 heads 0.89 -> 0.72 ms (770 TFLOP/s),
// 2.60 -> 0.90 (917), 4.65 -> 1.30 (848).
#include "common.h"
#include "kernels.h"
#include "tile128.h"

#include <algorithm>

namespace lc {
namespace {

constexpr int D = 64;
constexpr int kRows = 32;                 // rows per tile and per stationary block
constexpr int kTile = kRows * 2 * D;      // bytes
constexpr int kPitch = D + 4;             // floats per row of a wave's partial
constexpr int kPart = kRows * kPitch;     // floats of a partial block
// A wave's LDS: two buffers of two tiles, later its partial(s).
constexpr int kWaveLds = 4 * kTile > 2 * kPart * 4 ? 4 * kTile : 2 * kPart * 4;

struct Args64 {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* dout;
  const float* lse2;
  const float* delta;
  float* o;
  float* m;
  float* l;
  float* dq;
  float* dk;
  float* dv;
  int Nq, Nk, Hq, Hkv, group, n_tiles, split;
  int64_t q_pos0, k_pos0, valid;
  int causal;
  int accumulate;  // forward: merge into the running (o, m, l) instead of writing them
  float sl2;       // scale * log2(e)
  float scale;
  int init;                      // backward: replace the accumulators' contents
  uint16_t *out, *dk16, *dv16;   // set: o (dQ), dK, dV go here as bf16 instead
};

__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

// LDS DMA of a 32-row tile: 8 rows per wave instruction.  Rows at or past
// nrows re-read the last row (finite data; callers mask them).
struct Loader {
  uint32_t off[4];
  __device__ __forceinline__ void init(int64_t stride, int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + (lane >> 3);
      off[i] = (uint32_t)(r * stride * 2 + 16 * ((lane & 7) ^ swz(r)));
    }
  }
  __device__ __forceinline__ void load(const uint16_t* base, int64_t stride, int row0, int nrows,
                                       uint32_t lds, int lane) const {
    const uint8_t* tb = reinterpret_cast<const uint8_t*>(base + (int64_t)row0 * stride);
    if (row0 + kRows <= nrows) {
#pragma unroll
      for (int i = 0; i < 4; ++i) t128::dma_b128(tb, off[i], lds + 1024 * i);
    } else {
      const int last = nrows - 1 - row0, ln = opaque(lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (ln >> 3);
        t128::dma_b128(tb, (uint32_t)(min(r, last) * (int)stride * 2 + 16 * ((ln & 7) ^ swz(r))),
                       lds + 1024 * i);
      }
    }
  }
};

// Per-lane offsets of the operand reads: k-step t of the row operand is
// row ^ (32 t); dim block d and k-step u of the transposed operand are
// (tr[p] ^ (64 d)) + u * 16 rows.
struct Offsets {
  int row, tr[2];
  __device__ __forceinline__ void init(int lane) {
    const int c = lane & 31, hh = lane >> 5;
    row = c * 2 * D + 16 * (hh ^ swz(c));
    const int G = lane >> 4, i = lane & 15, t = i >> 2, col = 16 * (G & 1) + 4 * (i & 3);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int r = 4 * (G >> 1) + 2 * p + (t & 1) + 8 * (t >> 1);
      tr[p] = r * 2 * D + 16 * ((col >> 3) ^ swz(r)) + 2 * (col & 7);
    }
  }
  __device__ __forceinline__ bf16x8 rows(const uint8_t* tile, int t) const {
    return *reinterpret_cast<const bf16x8*>(tile + (row ^ (32 * t)));
  }
  __device__ __forceinline__ bf16x8 cols(const uint8_t* tile, int u, int d) const {
    return concat_bf16x4(t128::ds_read_tr(tile + (tr[0] ^ (64 * d)) + u * 32 * D),
                         t128::ds_read_tr(tile + (tr[1] ^ (64 * d)) + u * 32 * D));
  }
};

// Keeps the operand reads of a product from moving ahead of the one before it
// (all of a tile's reads in flight at once exceed two waves' registers).
__device__ __forceinline__ void phase() { __builtin_amdgcn_sched_barrier(0); }

// Elements 8u .. 8u+7 of a score block as the B operand of k-step u.
__device__ __forceinline__ bf16x8 pack_scores(const f32x16& s, int u) {
  return pack_bf16x8(f32x4{s[8 * u], s[8 * u + 1], s[8 * u + 4], s[8 * u + 5]},
                     f32x4{s[8 * u + 2], s[8 * u + 3], s[8 * u + 6], s[8 * u + 7]});
}

// Scores of keys at or past lim (relative to the lane's first key) to -inf.
__device__ __forceinline__ void mask_keys(f32x16& s, int lim) {
#pragma unroll
  for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + (v & 3) >= lim ? -INFINITY : s[v];
}

// The stationary rows row0 + c as B operands (rows past the end re-read the last).
__device__ __forceinline__ void load_stationary(bf16x8 (&r)[4], const uint16_t* base, int64_t stride,
                                                int row0, int nrows, int lane) {
  const int row = min(row0 + (lane & 31), nrows - 1);
  const uint16_t* p = base + (int64_t)row * stride + 8 * (lane >> 5);
#pragma unroll
  for (int t = 0; t < 4; ++t) r[t] = *reinterpret_cast<const bf16x8*>(p + 16 * t);
}

// A wave's transposed accumulators (dim 32 d + 8(v/4) + 4hh + v%4 of row c) to
// its partial, row-major.
__device__ __forceinline__ void store_part(float* part, const f32x16 (&acc)[2], float f, int lane) {
  float* row = part + (lane & 31) * kPitch + 4 * (lane >> 5);
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int w = 0; w < 4; ++w)
      *reinterpret_cast<f32x4*>(row + 32 * d + 8 * w) =
          f32x4{acc[d][4 * w], acc[d][4 * w + 1], acc[d][4 * w + 2], acc[d][4 * w + 3]} * f;
}

// Number of leading keys of the shard that the query at index row sees.
__device__ __forceinline__ int visible_keys(const Args64& a, int row) {
  int64_t n = min((int64_t)a.Nk, a.valid - a.k_pos0);
  if (a.causal) n = min(n, a.q_pos0 + row - a.k_pos0 + 1);
  return n < 0 ? 0 : (int)n;
}

// Sum over the splits of four dims of one partial row.
template <int W>
__device__ __forceinline__ f32x4 sum_parts(const uint8_t* smem, int wave0, int split, int off) {
  f32x4 x[W];
#pragma unroll
  for (int s = 0; s < W; ++s)
    x[s] = *reinterpret_cast<const f32x4*>(smem + (wave0 + min(s, split - 1)) * kWaveLds + 4 * off);
  f32x4 acc = x[0];
#pragma unroll
  for (int s = 1; s < W; ++s)
    if (s < split) acc += x[s];
  return acc;
}

// What an accumulator holds before a contribution (init: nothing).
__device__ __forceinline__ f32x4 grad_old(const float* acc, int init, int64_t i) {
  f32x4 r = {0.f, 0.f, 0.f, 0.f};
  if (!init) r = *reinterpret_cast<const f32x4*>(acc + i);
  return r;
}

// ----------------------------------------------------------------- forward --

// Wave w of the workgroup: query block w / split (NQ x 32 queries), key tiles
// w % split, + split, ...
template <int NQ, int W>
__global__ __launch_bounds__(64 * W, 2) void fwd64_kernel(Args64 a) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W * kWaveLds];
  __shared__ float msm[W][kRows], lsm[W][kRows], mtop[W][kRows];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int qsub = wave / a.split, ksub = wave - qsub * a.split;
  const int rows_wg = W / a.split * kRows * NQ;

  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int qt = a.n_tiles - 1 - L % a.n_tiles;  // long query tiles first
  const int bh = L / a.n_tiles;
  const int h = bh % a.Hq;
  const int b = bh / a.Hq;
  const int hk = h / a.group;
  const int64_t qs = (int64_t)a.Hq * D, ks = (int64_t)a.Hkv * D;
  const uint16_t* qb = a.q + (int64_t)b * a.Nq * qs + (int64_t)h * D;
  const uint16_t* kb = a.k + (int64_t)b * a.Nk * ks + (int64_t)hk * D;
  const uint16_t* vb = a.v + (int64_t)b * a.Nk * ks + (int64_t)hk * D;

  const int q0 = qt * rows_wg + qsub * kRows * NQ;
  const int kend = q0 < a.Nq ? visible_keys(a, min(q0 + kRows * NQ, a.Nq) - 1) : 0;
  const int kall = q0 < a.Nq ? visible_keys(a, q0) : 0;  // keys every query of the wave sees
  const int ntiles = (kend + kRows - 1) / kRows;

  const uint32_t lds = t128::lds_addr(smem) + wave * kWaveLds;
  uint8_t* mem = smem + wave * kWaveLds;
  Loader ld;
  ld.init(ks, lane);
  auto issue = [&](int t, int buf) {
    ld.load(kb, ks, t * kRows, a.Nk, lds + buf * 2 * kTile, lane);
    ld.load(vb, ks, t * kRows, a.Nk, lds + buf * 2 * kTile + kTile, lane);
  };
  if (ksub < ntiles) issue(ksub, 0);

  bf16x8 qr[NQ][4];
  f32x16 o[NQ][2];
  float mrun[NQ], lsum[NQ];  // running maximum (log2 units), partial sum
  int klim[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    load_stationary(qr[n], qb, qs, q0 + kRows * n, a.Nq, lane);
    o[n][0] = o[n][1] = f32x16{};
    mrun[n] = -INFINITY;
    lsum[n] = 0.f;
    klim[n] = visible_keys(a, min(q0 + kRows * n + c, a.Nq - 1));
  }
  Offsets of;
  of.init(lane);

  auto tile = [&](const uint8_t* kt, const uint8_t* vt, int key0) {
    const bool masked = key0 + kRows > kall;  // uniform
    f32x16 s[NQ];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bf16x8 A = of.rows(kt, t);
#pragma unroll
      for (int n = 0; n < NQ; ++n) s[n] = mfma32x32x16(A, qr[n][t], t == 0 ? f32x16{} : s[n]);
    }
    phase();
    bf16x8 pb[NQ][2];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      if (masked) mask_keys(s[n], klim[n] - key0 - 4 * hh);
      float mx = s[n][0];
#pragma unroll
      for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[n][v]);
      mx = xor32_max(mx) * a.sl2;
      if (__any(mx > mrun[n])) {
        const float mnew = fmaxf(mrun[n], mx);
        const float alpha = mx > mrun[n] ? fast_exp2(mrun[n] - mnew) : 1.f;  // mrun = -inf: 0
        mrun[n] = mnew;
        lsum[n] *= alpha;
        o[n][0] *= alpha;
        o[n][1] *= alpha;
      }
      const float muse = mrun[n] == -INFINITY ? 0.f : mrun[n];  // no key yet: p = 0
      float ts = 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float p = fast_exp2(fmaf(s[n][v], a.sl2, -muse));
        ts += p;
        s[n][v] = p;
      }
      lsum[n] += ts;
      pb[n][0] = pack_scores(s[n], 0);
      pb[n][1] = pack_scores(s[n], 1);
      phase();
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const bf16x8 A = of.cols(vt, u, d);
#pragma unroll
        for (int n = 0; n < NQ; ++n) o[n][d] = mfma32x32x16(A, pb[n][u], o[n][d]);
      }
  };
  int buf = 0;
  for (int t = ksub; t < ntiles; t += a.split, buf ^= 1) {
    t128::wait_vmem();
    if (t + a.split < ntiles) issue(t + a.split, buf ^ 1);
    const uint8_t* kt = mem + buf * 2 * kTile;
    tile(kt, kt + kTile, t * kRows);
  }

  // The key splits of each query merge by log-sum-exp; accumulate: then into
  // the running state of the row with lc_attn_merge's weights.
  const int p0 = qsub * a.split;
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const float ln = xor32_sum(lsum[n]);
    float M = mrun[n];
    if (n > 0) __syncthreads();
    if (a.split > 1) {
      if (hh == 0) msm[wave][c] = M;
      __syncthreads();
#pragma unroll
      for (int s = 0; s < W; ++s) M = fmaxf(M, msm[p0 + min(s, a.split - 1)][c]);
    }
    const float f = mrun[n] == -INFINITY ? 0.f : fast_exp2(mrun[n] - M);  // 1 without splits
    store_part(reinterpret_cast<float*>(mem), o[n], f, lane);
    if (hh == 0) {
      lsm[wave][c] = ln * f;
      mtop[wave][c] = M;
    }
    __syncthreads();
    // 16 threads per row; the waves of the query block take its rows in turn.
    const int d = 4 * (lane & 15), r0 = 4 * ksub + (lane >> 4), step = 4 * a.split;
    const int rows = min(kRows, a.Nq - (q0 + kRows * n));  // of the block, may be negative
    auto stat_at = [&](int r) { return ((int64_t)b * a.Hq + h) * a.Nq + q0 + kRows * n + r; };
    auto out_at = [&](int r) {
      return (((int64_t)b * a.Nq + q0 + kRows * n + r) * a.Hq + h) * D + d;
    };
    // Row r of the block; accumulate: old, om and ol are its running state.
    auto finish = [&](int r, const f32x4& old, float om, float ol) {
      const f32x4 acc = sum_parts<W>(smem, p0, a.split, r * kPitch + d);
      float lt = 0.f;
#pragma unroll
      for (int s = 0; s < W; ++s) {
        const float x = lsm[p0 + min(s, a.split - 1)][r];
        lt += s < a.split ? x : 0.f;
      }
      const float top = mtop[p0][r];
      const float inv = lt > 0.f ? 1.f / lt : 0.f;
      MergeW w{0.f, 1.f, top == -INFINITY ? -INFINITY : top * kLn2, lt};
      f32x4 x = acc * inv;
      if (a.accumulate) {
        w = merge_weights(om, ol, w.m, lt);
        x = old * w.wa + acc * (w.wb * inv);
      }
      const int64_t oi = out_at(r);
      store4(a.o + oi, a.out != nullptr ? a.out + oi : nullptr, x);
      if (d == 0) {  // every thread of the row has read the old statistics: they are in one wave
        a.m[stat_at(r)] = w.m;
        a.l[stat_at(r)] = w.l;
      }
    };
    if (!a.accumulate) {
      for (int r = r0; r < rows; r += step) finish(r, f32x4{0.f, 0.f, 0.f, 0.f}, 0.f, 0.f);
    } else {
      // Four rows at a time, whose old state is read together: one memory
      // latency instead of four (1,000 queries over 512 keys, 8 x 16 heads,
      // 49 us with one row at a time).
      for (int r = r0; r < rows; r += 4 * step) {
        f32x4 old[4];
        float om[4], ol[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int rj = min(r + j * step, rows - 1);
          old[j] = *reinterpret_cast<const f32x4*>(a.o + out_at(rj));
          om[j] = a.m[stat_at(rj)];
          ol[j] = a.l[stat_at(rj)];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (r + j * step < rows) finish(r + j * step, old[j], om[j], ol[j]);
      }
    }
  }
}

// ---------------------------------------------------------------------- dQ --

template <int NQ, int W>
__global__ __launch_bounds__(64 * W, 2) void dq64_kernel(Args64 a) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W * kWaveLds];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int qsub = wave / a.split, ksub = wave - qsub * a.split;
  const int rows_wg = W / a.split * kRows * NQ;

  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int qt = a.n_tiles - 1 - L % a.n_tiles;
  const int bh = L / a.n_tiles;
  const int h = bh % a.Hq;
  const int b = bh / a.Hq;
  const int hk = h / a.group;
  const int64_t qs = (int64_t)a.Hq * D, ks = (int64_t)a.Hkv * D;
  const uint16_t* qb = a.q + (int64_t)b * a.Nq * qs + (int64_t)h * D;
  const uint16_t* ob = a.dout + (int64_t)b * a.Nq * qs + (int64_t)h * D;
  const uint16_t* kb = a.k + (int64_t)b * a.Nk * ks + (int64_t)hk * D;
  const uint16_t* vb = a.v + (int64_t)b * a.Nk * ks + (int64_t)hk * D;

  if (visible_keys(a, min(qt * rows_wg + rows_wg, a.Nq) - 1) == 0 && !a.init && a.out == nullptr)
    return;  // no contribution
  const int q0 = qt * rows_wg + qsub * kRows * NQ;
  const int kend = q0 < a.Nq ? visible_keys(a, min(q0 + kRows * NQ, a.Nq) - 1) : 0;
  const int kall = q0 < a.Nq ? visible_keys(a, q0) : 0;
  const int ntiles = (kend + kRows - 1) / kRows;

  const uint32_t lds = t128::lds_addr(smem) + wave * kWaveLds;
  uint8_t* mem = smem + wave * kWaveLds;
  Loader ld;
  ld.init(ks, lane);
  auto issue = [&](int t, int buf) {
    ld.load(kb, ks, t * kRows, a.Nk, lds + buf * 2 * kTile, lane);
    ld.load(vb, ks, t * kRows, a.Nk, lds + buf * 2 * kTile + kTile, lane);
  };
  if (ksub < ntiles) issue(ksub, 0);

  bf16x8 qr[NQ][4], dor[NQ][4];
  f32x16 acc[NQ][2];
  float lse[NQ], dl[NQ];
  int klim[NQ];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    load_stationary(qr[n], qb, qs, q0 + kRows * n, a.Nq, lane);
    load_stationary(dor[n], ob, qs, q0 + kRows * n, a.Nq, lane);
    acc[n][0] = acc[n][1] = f32x16{};
    const int row = min(q0 + kRows * n + c, a.Nq - 1);
    const int64_t si = ((int64_t)b * a.Hq + h) * a.Nq + row;
    lse[n] = a.lse2[si];
    dl[n] = a.delta[si];
    klim[n] = visible_keys(a, row);
  }
  Offsets of;
  of.init(lane);

  auto tile = [&](const uint8_t* kt, const uint8_t* vt, int key0) {
    const bool masked = key0 + kRows > kall;  // uniform
    f32x16 s[NQ], dp[NQ];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bf16x8 A = of.rows(kt, t);
#pragma unroll
      for (int n = 0; n < NQ; ++n) s[n] = mfma32x32x16(A, qr[n][t], t == 0 ? f32x16{} : s[n]);
    }
    phase();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bf16x8 A = of.rows(vt, t);
#pragma unroll
      for (int n = 0; n < NQ; ++n) dp[n] = mfma32x32x16(A, dor[n][t], t == 0 ? f32x16{} : dp[n]);
    }
    phase();
    bf16x8 db[NQ][2];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      if (masked) mask_keys(s[n], klim[n] - key0 - 4 * hh);
#pragma unroll
      for (int v = 0; v < 16; ++v)
        s[n][v] = fast_exp2(fmaf(s[n][v], a.sl2, -lse[n])) * (dp[n][v] - dl[n]);
      db[n][0] = pack_scores(s[n], 0);
      db[n][1] = pack_scores(s[n], 1);
      phase();
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const bf16x8 A = of.cols(kt, u, d);
#pragma unroll
        for (int n = 0; n < NQ; ++n) acc[n][d] = mfma32x32x16(A, db[n][u], acc[n][d]);
      }
  };
  int buf = 0;
  for (int t = ksub; t < ntiles; t += a.split, buf ^= 1) {
    t128::wait_vmem();
    if (t + a.split < ntiles) issue(t + a.split, buf ^ 1);
    const uint8_t* kt = mem + buf * 2 * kTile;
    tile(kt, kt + kTile, t * kRows);
  }

#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    if (n > 0) __syncthreads();
    store_part(reinterpret_cast<float*>(mem), acc[n], a.scale, lane);
    __syncthreads();
    for (int r = 4 * ksub + (lane >> 4); r < kRows; r += 4 * a.split) {
      const int row = q0 + kRows * n + r;
      if (row >= a.Nq) break;
      const int d = 4 * (lane & 15);
      const int64_t i = (((int64_t)b * a.Nq + row) * a.Hq + h) * D + d;
      const f32x4 old = grad_old(a.dq, a.init, i);  // on its way during the sum
      store4(a.dq + i, a.out != nullptr ? a.out + i : nullptr,
             old + sum_parts<W>(smem, qsub * a.split, a.split, r * kPitch + d));
    }
  }
}

// ------------------------------------------------------------------- dK/dV --

// Wave w of the workgroup: key block w / split (32 keys of one KV head), steps
// (query head of the group, query tile) w % split, + split, ...
template <int W>
__global__ __launch_bounds__(64 * W, 2) void dkdv64_kernel(Args64 a) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W * kWaveLds];
  __shared__ __attribute__((aligned(16))) float stat[W][2][64];  // [buffer]: lse2, then delta
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int ksub = wave / a.split, qsub = wave - ksub * a.split;
  const int keys_wg = W / a.split * kRows;

  const int L = xcd_remap(blockIdx.x, gridDim.x);
  const int kt = L % a.n_tiles;  // early keys see the most queries: dispatched first
  const int bh = L / a.n_tiles;
  const int hk = bh % a.Hkv;
  const int b = bh / a.Hkv;
  const int64_t qs = (int64_t)a.Hq * D, ks = (int64_t)a.Hkv * D;
  const uint16_t* kb = a.k + (int64_t)b * a.Nk * ks + (int64_t)hk * D;
  const uint16_t* vb = a.v + (int64_t)b * a.Nk * ks + (int64_t)hk * D;

  // First query that sees key index key (Nq: none).
  auto first_query = [&](int key) {
    if (key >= a.Nk || a.k_pos0 + key >= a.valid) return a.Nq;
    if (!a.causal) return 0;
    const int64_t first = a.k_pos0 + key - a.q_pos0;
    return first <= 0 ? 0 : (first >= a.Nq ? a.Nq : (int)first);
  };
  if (first_query(kt * keys_wg) >= a.Nq && !a.init && a.dk16 == nullptr)
    return;  // no visible pair: no contribution
  const int k0 = kt * keys_wg + ksub * kRows;
  const int qstart = first_query(k0) / kRows * kRows;
  const int qall = first_query(k0 + kRows - 1);  // queries from here on see all the wave's keys
  const int rmin = first_query(k0 + c);
  const int ntq = first_query(k0) < a.Nq ? (a.Nq - qstart + kRows - 1) / kRows : 0;
  const int nsteps = ntq * a.group;

  const uint32_t lds = t128::lds_addr(smem) + wave * kWaveLds;
  const uint32_t stat_lds = t128::lds_addr(stat) + wave * 512;
  uint8_t* mem = smem + wave * kWaveLds;
  Loader ld;
  ld.init(qs, lane);
  auto issue = [&](int hq, int qrow0, int buf) {
    const int64_t base = (int64_t)b * a.Nq * qs + (int64_t)hq * D;
    ld.load(a.q + base, qs, qrow0, a.Nq, lds + buf * 2 * kTile, lane);
    ld.load(a.dout + base, qs, qrow0, a.Nq, lds + buf * 2 * kTile + kTile, lane);
    const int64_t si = ((int64_t)b * a.Hq + hq) * a.Nq + min(qrow0 + c, a.Nq - 1);
    t128::dma_b32((hh == 0 ? a.lse2 : a.delta) + si, stat_lds + buf * 256);
  };
  // The wave's steps in order: (head, tile) advanced by split without divisions.
  int nh = 0, nt = qsub;
  auto wrap = [&]() {
    while (nt >= ntq && nh < a.group) {
      nt -= ntq;
      ++nh;
    }
  };
  if (nsteps > 0) wrap();
  const bool any = nsteps > 0 && nh < a.group;
  if (any) issue(hk * a.group + nh, qstart + nt * kRows, 0);

  bf16x8 kr[4], vr[4];
  load_stationary(kr, kb, ks, k0, a.Nk, lane);
  load_stationary(vr, vb, ks, k0, a.Nk, lane);
  // dP = dO V^T runs with -V from delta to delta - dP: dS = -(P (delta - dP)).
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    vr[t] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, vr[t]) ^ 0x80008000u);
  }
  f32x16 dk[2], dv[2];
  dk[0] = dk[1] = dv[0] = dv[1] = f32x16{};
  Offsets of;
  of.init(lane);

  auto tile = [&](const uint8_t* qt, const uint8_t* ot, const float* st, int qrow0) {
    f32x16 s, e;
#pragma unroll
    for (int t = 0; t < 4; ++t) s = mfma32x32x16(of.rows(qt, t), kr[t], t == 0 ? f32x16{} : s);
    phase();
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(st + 32 + 8 * w + 4 * hh);
#pragma unroll
      for (int r = 0; r < 4; ++r) e[4 * w + r] = d4[r];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) e = mfma32x32x16(of.rows(ot, t), vr[t], e);
    phase();
    if (qrow0 < qall || qrow0 + kRows > a.Nq) {  // uniform
      const int lo = rmin - qrow0 - 4 * hh, hi = a.Nq - qrow0 - 4 * hh;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int q = 8 * (v >> 2) + (v & 3);
        s[v] = q < lo || q >= hi ? -INFINITY : s[v];
      }
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(st + 8 * w + 4 * hh);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int v = 4 * w + r;
        const float p = fast_exp2(fmaf(s[v], a.sl2, -l4[r]));
        s[v] = p;
        e[v] = -(p * e[v]);
      }
    }
    phase();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bf16x8 pb = pack_scores(s, u), db = pack_scores(e, u);
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        dv[d] = mfma32x32x16(of.cols(ot, u, d), pb, dv[d]);
        dk[d] = mfma32x32x16(of.cols(qt, u, d), db, dk[d]);
      }
    }
  };
  int buf = 0;
  bool have = any;
  while (have) {
    const int qrow0 = qstart + nt * kRows;
    nt += a.split;
    wrap();
    have = nh < a.group;
    t128::wait_vmem();
    if (have) issue(hk * a.group + nh, qstart + nt * kRows, buf ^ 1);
    const uint8_t* qt = mem + buf * 2 * kTile;
    tile(qt, qt + kTile, stat[wave][buf], qrow0);
    buf ^= 1;
  }

  store_part(reinterpret_cast<float*>(mem), dk, a.scale, lane);
  store_part(reinterpret_cast<float*>(mem) + kPart, dv, 1.f, lane);
  __syncthreads();
  for (int r = 4 * qsub + (lane >> 4); r < kRows; r += 4 * a.split) {
    if (k0 + r >= a.Nk) break;
    const int d = 4 * (lane & 15);
    const int64_t i = (((int64_t)b * a.Nk + k0 + r) * a.Hkv + hk) * D + d;
    const f32x4 oldk = grad_old(a.dk, a.init, i), oldv = grad_old(a.dv, a.init, i);
    store4(a.dk + i, a.dk16 != nullptr ? a.dk16 + i : nullptr,
           oldk + sum_parts<W>(smem, ksub * a.split, a.split, r * kPitch + d));
    store4(a.dv + i, a.dv16 != nullptr ? a.dv16 + i : nullptr,
           oldv + sum_parts<W>(smem, ksub * a.split, a.split, kPart + r * kPitch + d));
  }
}

Args64 make_args(const Problem& p, const void* q, const void* k, const void* v, const void* dout) {
  Args64 a{};
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.dout = static_cast<const uint16_t*>(dout);
  a.Nq = p.Nq;
  a.Nk = p.Nk;
  a.Hq = p.Hq;
  a.Hkv = p.Hkv;
  a.group = p.Hq / p.Hkv;
  a.split = 1;
  a.q_pos0 = p.q_pos0;
  a.k_pos0 = p.k_pos0;
  a.valid = p.valid;
  a.causal = p.causal ? 1 : 0;
  a.accumulate = p.accumulate ? 1 : 0;
  a.sl2 = p.scale * kLog2e;
  a.scale = p.scale;
  return a;
}

constexpr int64_t kWaveSlots = 2048;  // waves the chip holds (two per SIMD)

// Waves that share a block of stationary rows in dQ and dK/dV: enough to fill
// the chip `over` times, with at least two streamed tiles each, and up to four
// times while they keep 32 tiles.  Twice over evens out the causal walks'
// lengths (dK/dV, 4,096 tokens x 32/8 heads: 195 us against 250 at once over,
// 2,048 tokens 54 against 65); four times with 64-row waves, whose walks differ
// more (dQ 153 us against 163 and 217 at twice and once over), and over long
// walks (8,192 tokens x 9/3 heads, dQ 179 against 204).
int split_for(int64_t blocks, int64_t tiles, int over) {
  int s = 1;
  while (s < 8 && tiles >= 4 * s &&
         blocks * s < (tiles >= 64 * s ? 4 : over) * kWaveSlots)
    s *= 2;
  return s;
}

// The same for the forward (where long walks gain alike: 4,096 tokens x 32/8 heads
// 130 us at four times over against 141 and 187 at twice and once, 8,192 x 9/3
// heads 162 against 186), whose short walks pay more for a further split (the
// merge in LDS, a second round of workgroups) than they gain: within the waves
// the chip holds while there are tiles for them (200 queries over 512 keys, 8 x
// 16 heads: 14.3 us with two, 22.7 with eight; 100 queries over 64 keys, 8
// heads: 7.1 us with one, 4.7 with four), past them while each wave keeps
// `keep` / 2 tiles (1,000 tokens, 32/8 heads 18.8 us with four, 20.4 with two).
int fwd_split(int64_t blocks, int64_t tiles, int over, int keep) {
  int s = 1;
  while (s < 8 && tiles >= s &&
         (2 * s * blocks <= kWaveSlots ||
          (tiles >= std::max(32, keep * s) &&
           blocks * s < (tiles >= 64 * s ? 4 : over) * kWaveSlots)))
    s *= 2;
  return s;
}

// Blocks of 64 stationary rows per wave once those fill the chip, given rows
// for the second half.
bool two_blocks(int64_t blocks, int rows) { return blocks >= 2 * kWaveSlots && rows > kRows; }

// Splits for which a workgroup's four waves all have rows: a head with one or
// two row blocks has the others take keys (16 queries over 500 keys, 128 x 32/8
// heads: 109 us with three waves idle, 52 with all four on the keys).
int least_split(int rows, int per_wave) {
  return rows <= per_wave ? 4 : rows <= 2 * per_wave ? 2 : 1;
}

}  // namespace

bool mfma_supported(const Problem& p) {
  return p.dtype == 1 && !p.precise && (p.D == 64 || p.D == 128);
}

hipError_t launch_fwd64(const Problem& p, const void* q, const void* k, const void* v, float* o,
                        float* m, float* l, hipStream_t s, uint16_t* out) {
  if (p.D != D) return hipErrorInvalidValue;
  Args64 a = make_args(p, q, k, v, nullptr);
  a.out = out;
  a.o = o;
  a.m = m;
  a.l = l;
  const int64_t heads = (int64_t)p.B * p.Hq, blocks = heads * ((p.Nq + kRows - 1) / kRows);
  const bool two = two_blocks(blocks, p.Nq);
  const int64_t tiles = (p.Nk + kRows - 1) / kRows;
  a.split = two ? std::min(4, fwd_split(blocks / 2, tiles, 4, 32)) : fwd_split(blocks, tiles, 2, 16);
  a.split = std::max(a.split, least_split(p.Nq, two ? 2 * kRows : kRows));
  const int nw = a.split == 8 ? 8 : 4, rows = nw / a.split * kRows * (two ? 2 : 1);
  a.n_tiles = (p.Nq + rows - 1) / rows;
  const dim3 grid((unsigned)(a.n_tiles * heads));
  if (two) hipLaunchKernelGGL((fwd64_kernel<2, 4>), grid, dim3(256), 0, s, a);
  else if (nw == 4) hipLaunchKernelGGL((fwd64_kernel<1, 4>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((fwd64_kernel<1, 8>), grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_dq64(const Problem& p, const void* q, const void* k, const void* v,
                       const void* dout, const float* lse2, const float* delta, float* dq,
                       hipStream_t s, const Sink& to) {
  if (p.D != D) return hipErrorInvalidValue;
  Args64 a = make_args(p, q, k, v, dout);
  a.init = to.init;
  a.out = to.out;
  a.lse2 = lse2;
  a.delta = delta;
  a.dq = dq;
  const int64_t heads = (int64_t)p.B * p.Hq, blocks = heads * ((p.Nq + kRows - 1) / kRows);
  const bool two = two_blocks(blocks, p.Nq);
  const int64_t tiles = (p.Nk + kRows - 1) / kRows;
  a.split = two ? std::min(4, split_for(blocks / 2, tiles, 4)) : split_for(blocks, tiles, 2);
  a.split = std::max(a.split, least_split(p.Nq, two ? 2 * kRows : kRows));
  const int nw = a.split == 8 ? 8 : 4, rows = nw / a.split * kRows * (two ? 2 : 1);
  a.n_tiles = (p.Nq + rows - 1) / rows;
  const dim3 grid((unsigned)(a.n_tiles * heads));
  if (two) hipLaunchKernelGGL((dq64_kernel<2, 4>), grid, dim3(256), 0, s, a);
  else if (nw == 4) hipLaunchKernelGGL((dq64_kernel<1, 4>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((dq64_kernel<1, 8>), grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_dkdv64(const Problem& p, const void* q, const void* k, const void* v,
                         const void* dout, const float* lse2, const float* delta, float* dk,
                         float* dv, hipStream_t s, const Sink& to) {
  if (p.D != D) return hipErrorInvalidValue;
  Args64 a = make_args(p, q, k, v, dout);
  a.init = to.init;
  a.dk16 = to.out;
  a.dv16 = to.out2;
  a.lse2 = lse2;
  a.delta = delta;
  a.dk = dk;
  a.dv = dv;
  const int64_t heads = (int64_t)p.B * p.Hkv, blocks = heads * ((p.Nk + kRows - 1) / kRows);
  a.split = split_for(blocks, (int64_t)a.group * ((p.Nq + kRows - 1) / kRows), 2);
  const int nw = a.split == 8 ? 8 : 4, keys = nw / a.split * kRows;
  a.n_tiles = (p.Nk + keys - 1) / keys;
  const dim3 grid((unsigned)(a.n_tiles * heads));
  if (nw == 4) hipLaunchKernelGGL((dkdv64_kernel<4>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((dkdv64_kernel<8>), grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

}  // namespace lc
