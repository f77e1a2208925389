// Split-KV decode attention for head_dim 64 and 128 on bf16 MFMA (gfx950): a
// few new query tokens against a long KV cache.
//
// Same semantics and outputs as the blockwise forward of one ring hop
// (rust/longctx100m-model/src/ring_attention.rs:15-106 and the finalize of
// :227): normalised o [B, Nq, Hq, D] fp32 and the row statistics m, l.  The
// work split is the decode one: each (batch, KV head) has R = Nq * group
// query rows (group = Hq / Hkv), taken in blocks of 16 or 32 (MFMA columns),
// and the key range is split over the waves of S workgroups, each wave streaming
// its own tiles.  The waves of a workgroup meet in LDS; with S > 1
// each workgroup leaves a partial (acc, m, l) in the workspace and
// decode_merge_kernel combines them, with S = 1 (short caches, or enough
// sequences to fill the chip) the workgroup writes the result itself.
//
// Per wave: Q^T of the rows in VGPRs (B operand, rows past R are zero); tiles
// of 8 KB: K straight into VGPRs (the A operand of S^T = K Q^T wants each
// lane's 8 dims of one key, which a 16-byte global load gives), V
// double-buffered in LDS by direct global->LDS loads, both one tile ahead;
// S^T = K Q^T, exact online softmax per row in the log2 domain, O^T += V^T P^T
// with V^T from transposed LDS reads.
//
// Bound by the cache read once it is long (262,144 keys x 8 KV heads of 128:
// 153-157 us + 5 us of merge, 6.8-7.0 TB/s) and by latency when it is short: a
// tile takes 2 us to arrive, a workgroup 1 us to start.  Measured against the
// blockwise forward that head_dim 64 and more than 16 rows took before (GPU
// time of a call, caches cold): 4 sequences x 3,001 keys, 9/3 heads of 64
// 70.9 -> 10.0 us; 8 tokens x 32/8 heads of 128 over 16,001 keys 272 -> 23.4 us;
// 16 sequences x 60,000 keys of the same 1309 -> 726 us.  Against one-wave
// workgroups with a merge for every shape: 8,001 keys x 32/8 heads
// 15.2 -> 12.9 us, 16 x 4,000 66.7 -> 53 us.
#include "common.h"
#include "kernels.h"
#include "tile128.h"

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <type_traits>

namespace lc {

// Workspace of lc_attn_decode_static: split partials of the decode kernel,
// read back by the merge kernel.  Every partial is written before it is read,
// so nothing here needs clearing between calls.  Each device holds its own
// copy from the library's load until the process ends, and every call on a
// device shares it (calls that overlap on one device race).  Host code never
// passes `scratch` itself to a kernel: its host-side name is not a device
// address; decode_static_scratch() returns the device address.
static __device__ __align__(256) uint8_t scratch[kDecodeStaticScratchBytes];

namespace {

// V tiles in LDS per wave: the one in use and one in flight.  With K staged in
// LDS as well, one layer of 262,144 keys x 8 KV heads of 128 read the cache at
// 4.72-5.24 TB/s (2-5 stages); K in VGPRs (the LDS round trip costs SIMD
// cycles per byte) and eight waves per CU (the register limit of two waves per
// SIMD) read it at 5.68 TB/s, non-temporal loads at 6.58.
constexpr int kStages = 2;
constexpr int kWaves = 4;          // waves per workgroup (kStreamWaves for long single streams)
constexpr int kStreamWaves = 1;
constexpr int64_t kWaveSlots = 256 * 8;  // waves the chip holds
constexpr int kTileBytes = 8192;   // K (or V) bytes per tile

template <int D>
struct DecodeTile {
  static constexpr int TK = kTileBytes / (2 * D);  // keys per tile
  static constexpr int MB = TK / 16;               // 16-key blocks
  static constexpr int KS = D / 32;                // MFMA k-steps over head_dim
  static constexpr int DB = D / 16;                // 16-dim blocks
};

struct DecodeArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  float* o;
  float* m;
  float* l;
  float* o_part;  // [S][B*Nq*Hq][D] (unnormalised, relative to m_part)
  float* m_part;  // [S][B*Nq*Hq] (log2 units)
  float* l_part;
  int Nq, Nk, Hq, Hkv, group, rows, row_blocks, S, chunk;  // chunk: keys per workgroup
  int64_t prows;  // B * Nq * Hq: rows of one split's partial
  int64_t q_pos0, k_pos0, valid;
  int causal;
  float sl2;  // scale * log2(e)
};

// V tile in LDS.  head_dim 128: tile128.h's layout.  head_dim 64: rows of 128
// bytes, the eight 16-byte chunks of row r stored at chunk ^ swz64(r).  A
// transposed read serves lanes 0-31 and 32-63 in separate cycles, i.e. eight
// consecutive rows x one chunk pair; rows of equal parity share a half of the
// 256 bytes of banks, and swz64 gives the four of them distinct chunk pairs,
// so the reads are free of bank conflicts.
__device__ __forceinline__ int swz64(int r) { return r & 6; }

template <int D>
struct VTile;
template <>
struct VTile<128> {
  t128::RowLoader<DecodeTile<128>::TK, 1> ld;
  __device__ __forceinline__ void init(int64_t stride, int lane) { ld.init(stride, 0, lane); }
  __device__ __forceinline__ void load(const uint16_t* base, int64_t stride, int row0, int nrows,
                                       uint32_t lds, int lane) const {
    ld.load<false, true>(base, stride, row0, nrows, lds, 0, lane);
  }
  static __device__ __forceinline__ int tr_off(int col0, int lane) { return t128::tr_off(0, col0, lane); }
};
template <>
struct VTile<64> {
  static constexpr int kInst = kTileBytes / 1024;  // 8 rows per wave instruction
  uint32_t off[kInst];
  __device__ __forceinline__ void init(int64_t stride, int lane) {
#pragma unroll
    for (int i = 0; i < kInst; ++i) {
      const int r = 8 * i + (lane >> 3);
      off[i] = (uint32_t)(r * stride * 2 + 16 * ((lane & 7) ^ swz64(r)));
    }
  }
  // Rows at or past nrows re-read the last row (callers mask them).
  __device__ __forceinline__ void load(const uint16_t* base, int64_t stride, int row0, int nrows,
                                       uint32_t lds, int lane) const {
    if (row0 + 8 * kInst <= nrows) {
      const uint8_t* tb = reinterpret_cast<const uint8_t*>(base + (int64_t)row0 * stride);
#pragma unroll
      for (int i = 0; i < kInst; ++i) t128::dma_b128_nt(tb, off[i], lds + 1024 * i);
    } else {
#pragma unroll
      for (int i = 0; i < kInst; ++i) {
        const int r = 8 * i + (lane >> 3);
        const int row = min(row0 + r, nrows - 1);
        t128::dma_b128_nt(base + (int64_t)row * stride + 8 * ((lane & 7) ^ swz64(r)), lds + 1024 * i);
      }
    }
  }
  // Lane 4t + q of group g addresses row 4g + t, columns col0 + 4q .. +3.
  static __device__ __forceinline__ int tr_off(int col0, int lane) {
    const int i = lane & 15, r = 4 * (lane >> 4) + (i >> 2), col = col0 + 4 * (i & 3);
    return r * 128 + 16 * ((col >> 3) ^ swz64(r)) + 2 * (col & 7);
  }
};

template <int D, int NB, int W>
__global__ __launch_bounds__(64 * W, NB * W == 1 ? 1 : 2) void decode_kernel(DecodeArgs a) {
  using C = DecodeTile<D>;
  constexpr int TK = C::TK, MB = C::MB, KS = C::KS, DB = C::DB;
  constexpr int kRows = 16 * NB;
  // head_dim 128, one row block: the probabilities that are rounded to bf16
  // are relative to their own tile's maximum, and the tile's product joins the
  // fp32 state with an fp32 weight.  Each tile's largest probability is then
  // exact; relative to a maximum that runs over the four tiles of a wave the
  // outputs were further from 64 bits (500 keys x 32/8 heads: 1.3e-3 against
  // 1.1e-3 here).  The kernel waits for memory: the 64 multiplications more per
  // tile leave that call at 14.4 us.  Long single streams (W = 1) keep the
  // running maximum: 1.4e-3 either way.
  constexpr bool kTileRef = TK == 32 && NB == 1 && W > 1;
  constexpr int kPitch = D + 4;  // floats per row of a wave's partial
  constexpr int kVBytes = W * kStages * kTileBytes;
  constexpr int kPartBytes = W * kRows * kPitch * 4;
  // The V tiles, then (after the walk) the waves' partials.
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kVBytes > kPartBytes ? kVBytes : kPartBytes];
  __shared__ float msm[W][kRows], lsm[W][kRows], mtop[kRows];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;
  const int s = blockIdx.x % a.S;
  const int rest = blockIdx.x / a.S;
  int rb = 0, bh = rest;
  if (a.row_blocks > 1) {
    rb = rest % a.row_blocks;
    bh = rest / a.row_blocks;
  }
  const int hk = bh % a.Hkv;
  const int b = bh / a.Hkv;

  const int64_t ks = (int64_t)a.Hkv * D;
  const uint16_t* kbase = a.k + (int64_t)b * a.Nk * ks + (int64_t)hk * D;
  const uint16_t* vbase = a.v + (int64_t)b * a.Nk * ks + (int64_t)hk * D;

  // Keys any row can see, then the workgroup's share of them, whose tiles its
  // waves take in turn (they then stream one region of the cache together).
  int64_t kend = a.Nk;
  if (a.causal) kend = min(kend, a.q_pos0 + a.Nq - a.k_pos0);
  kend = min(kend, a.valid - a.k_pos0);
  const int64_t kb0 = (int64_t)s * a.chunk + wave * TK;
  const int64_t kb1 = min((int64_t)(s + 1) * a.chunk, kend);
  const int ntiles = kb1 > kb0 ? (int)((kb1 - kb0 + W * TK - 1) / (W * TK)) : 0;

  VTile<D> ld;
  ld.init(ks, lane);
  const uint32_t vlds = t128::lds_addr(smem) + wave * kStages * kTileBytes;
  const uint8_t* vmem = smem + wave * kStages * kTileBytes;
  auto issue = [&](int j) {  // V tile j into stage j % kStages
    ld.load(vbase, ks, (int)(kb0 + (int64_t)j * (W * TK)), a.Nk, vlds + (j % kStages) * kTileBytes, lane);
  };
  // K tile j straight into VGPRs: lane (c, g) holds key 16 mb + c of the
  // tile, dims 32 kk + 8 g.  The cache is read once per step: non-temporal.
  auto kload = [&](int j, bf16x8 (&kr)[MB][KS]) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      int64_t row = kb0 + (int64_t)j * (W * TK) + 16 * mb + c;
      row = row < a.Nk ? row : a.Nk - 1;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        kr[mb][kk] = __builtin_nontemporal_load(
            reinterpret_cast<const bf16x8*>(kbase + row * ks + 32 * kk + 8 * g));
    }
  };

  bf16x8 kra[MB][KS], krb[MB][KS];
  if (ntiles > 0) {
    issue(0);
    kload(0, kra);
  }

  // Row r of this (batch, KV head): query head hk*group + r / Nq, query r % Nq.
  bf16x8 qreg[NB][KS];
  int klim[NB];  // leading keys of the shard the row sees (0: no such row)
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int r = rb * kRows + 16 * nb + c;
    const bool ok = r < a.rows;
    const int qi = ok ? r % a.Nq : 0;
    const int qh = hk * a.group + (ok ? r / a.Nq : 0);
    const uint16_t* qrow = a.q + (((int64_t)b * a.Nq + qi) * a.Hq + qh) * D;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      qreg[nb][kk] = *reinterpret_cast<const bf16x8*>(qrow + 32 * kk + 8 * g);
      if (!ok) qreg[nb][kk] = bf16x8{};
    }
    int64_t n = kend;
    if (a.causal) n = min(n, a.q_pos0 + qi + 1 - a.k_pos0);
    klim[nb] = ok && n > 0 ? (int)n : 0;
  }

  // Q is in VGPRs from here on (the compiler, which cannot count the tile
  // loads below, would otherwise wait for every load before each use of Q).
  t128::wait_vmem();

  int voff[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) voff[db] = VTile<D>::tr_off(16 * db, lane);

  f32x4 o[NB][DB];
  float mrow[NB], lsum[NB];  // running max (log2 units), lane-partial sum of p
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
    for (int db = 0; db < DB; ++db) o[nb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
    mrow[nb] = -INFINITY;
    lsum[nb] = 0.f;
  }

  // Tile j: wait for V(j) in LDS and K(j) in VGPRs (both issued at tile j - 1),
  // issue V(j + 1) into the other stage (read by tile j - 1, done) and
  // K(j + 1) into the other register set, then compute tile j.
  auto tile = [&](int j, bf16x8 (&kc)[MB][KS], bf16x8 (&kn)[MB][KS]) {
    t128::wait_vmem();
    if (j + 1 < ntiles) {
      issue(j + 1);
      kload(j + 1, kn);
    }
    const uint8_t* vt = vmem + (j % kStages) * kTileBytes;
    const int key0 = (int)(kb0 + (int64_t)j * (W * TK));
    const int kmax = (int)min((int64_t)TK, kb1 - key0);  // keys of this tile inside the workgroup's share

    float alpha = 1.f, beta = 1.f;  // kTileRef: weights of the state and of the tile
    f32x4 sc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) sc[nb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) sc[nb][mb] = mfma16x16x32(kc[mb][kk], qreg[nb][kk], sc[nb][mb]);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      // Mask: past the workgroup's share, valid_length, causal (per row).
      const int lim = min(kmax, klim[nb] - key0);
      float mx = -INFINITY;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[nb][mb][i] = 16 * mb + 4 * g + i >= lim ? -INFINITY : sc[nb][mb][i] * a.sl2;
          mx = fmaxf(mx, sc[nb][mb][i]);
        }
      mx = group4_max(mx);
      if constexpr (kTileRef) {
        const float mnew = fmaxf(mrow[nb], mx);
        alpha = mrow[nb] == -INFINITY ? 0.f : fast_exp2(mrow[nb] - mnew);
        beta = mx == -INFINITY ? 0.f : fast_exp2(mx - mnew);
        mrow[nb] = mnew;
      } else if (mx > mrow[nb]) {
        const float up = fast_exp2(mrow[nb] - mx);  // mrow = -inf: 0
        lsum[nb] *= up;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[nb][db] *= up;
        mrow[nb] = mx;
      }
      const float ref = kTileRef ? mx : mrow[nb];
      const float muse = ref == -INFINITY ? 0.f : ref;  // no key yet: p = 0
      float tsum = 0.f;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = fast_exp2(sc[nb][mb][i] - muse);
          if constexpr (kTileRef) tsum += p;
          else lsum[nb] += p;
          sc[nb][mb][i] = p;
        }
      if constexpr (kTileRef) lsum[nb] = lsum[nb] * alpha + tsum * beta;
    }
#pragma unroll
    for (int k2 = 0; k2 < TK / 32; ++k2) {
      bf16x8 pb[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) pb[nb] = pack_bf16x8(sc[nb][2 * k2], sc[nb][2 * k2 + 1]);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const uint8_t* p = vt + voff[db] + 32 * k2 * 2 * D;
        const bf16x8 va = concat_bf16x4(t128::ds_read_tr(p), t128::ds_read_tr(p + 16 * 2 * D));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          if constexpr (kTileRef)
            o[nb][db] = o[nb][db] * alpha + mfma16x16x32(va, pb[nb], f32x4{0.f, 0.f, 0.f, 0.f}) * beta;
          else
            o[nb][db] = mfma16x16x32(va, pb[nb], o[nb][db]);
        }
      }
    }
  };
  for (int j = 0; j < ntiles; j += 2) {
    tile(j, kra, krb);
    if (j + 1 < ntiles) tile(j + 1, krb, kra);
  }

  // Four dims from d of row r (unnormalised acc with sum L, relative to M).
  auto emit = [&](int r, int d, const f32x4& acc, float L, float M) {
    const int qi = r % a.Nq, qh = hk * a.group + r / a.Nq;
    const int64_t row = ((int64_t)b * a.Nq + qi) * a.Hq + qh;
    if (a.S == 1) {
      *reinterpret_cast<f32x4*>(a.o + row * D + d) = acc * (L > 0.f ? 1.f / L : 0.f);
      if (d == 0) {
        const int64_t si = ((int64_t)b * a.Hq + qh) * a.Nq + qi;
        a.m[si] = L > 0.f ? M * kLn2 : -INFINITY;
        a.l[si] = L;
      }
    } else {
      const int64_t prow = (int64_t)s * a.prows + row;
      *reinterpret_cast<f32x4*>(a.o_part + prow * D + d) = acc;
      if (d == 0) {
        a.m_part[prow] = M;
        a.l_part[prow] = L;
      }
    }
  };
  if constexpr (W == 1) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const float L = group4_sum(lsum[nb]);
      const int r = rb * kRows + 16 * nb + c;
      if (r < a.rows)
#pragma unroll
        for (int db = 0; db < DB; ++db) emit(r, 16 * db + 4 * g, o[nb][db], L, mrow[nb]);
    }
    return;
  }

  // The waves' partials, brought to each row's maximum, meet in LDS.
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
    if (g == 0) msm[wave][16 * nb + c] = mrow[nb];
  __syncthreads();  // also: every wave is done with its V tiles
  float* part = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) M = fmaxf(M, msm[w][16 * nb + c]);
    const float f = mrow[nb] == -INFINITY ? 0.f : fast_exp2(mrow[nb] - M);
    const float lt = group4_sum(lsum[nb]) * f;
    if (g == 0) {
      lsm[wave][16 * nb + c] = lt;
      if (wave == 0) mtop[16 * nb + c] = M;
    }
#pragma unroll
    for (int db = 0; db < DB; ++db)
      *reinterpret_cast<f32x4*>(part + (wave * kRows + 16 * nb + c) * kPitch + 16 * db + 4 * g) = o[nb][db] * f;
  }
  __syncthreads();
  constexpr int kPer = D / 4;  // threads per row
  for (int it = threadIdx.x; it < kRows * kPer; it += 64 * W) {
    const int rr = it / kPer, d = 4 * (it % kPer);
    const int r = rb * kRows + rr;
    if (r >= a.rows) break;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      acc += *reinterpret_cast<const f32x4*>(part + (w * kRows + rr) * kPitch + d);
      L += lsm[w][rr];
    }
    emit(r, d, acc, L, mtop[rr]);
  }
}

// Log-sum-exp merge of the S workgroup partials of each row (b, i, h) =
// ((b * Nq) + i) * Hq + h of o, PARTS workgroups of NT threads per row, each
// over D / PARTS dims: thread t holds the statistics of split t (S <= NT), wave
// shuffles and one LDS exchange give the maximum and the weights, then thread
// (d, g) sums four dims over the splits g, g + groups, ..., and the groups'
// sums meet by shuffles and in LDS.  The first partials are loaded before the
// statistics are reduced, so the row costs little more than one memory
// latency.  A decode step has few rows, so many splits (long single streams)
// take the 1024 x 4 form, whose chains are the shorter.
constexpr int kMaxSplits = 1024;

template <int D, int NT, int PARTS>
__global__ __launch_bounds__(NT) void decode_merge_kernel(
    int64_t nrows, int S, int Nq, int Hq, const float* o_part, const float* m_part,
    const float* l_part, float* o, float* m, float* l) {
  constexpr int kLanes = D / 4 / PARTS;  // threads across the workgroup's dims
  constexpr int kGroups = NT / kLanes;   // splits in flight
  // Partials loaded up front: all of 256 splits (with four, half of the loads
  // re-read the last split: 262,144 keys 160.5 us a call against 159.4 before
  // this form, 160.8 against 160.4 with two), or of the 32 of a small grid.
  constexpr int kFirst = NT == 1024 ? 2 : 4;
  constexpr int kNW = NT / 64;
  __shared__ float w[NT];
  __shared__ float wmax[kNW], wsum[kNW];
  __shared__ f32x4 part[kNW][kLanes];
  const int t = threadIdx.x;
  const int64_t row = blockIdx.x / PARTS;
  const int d = 4 * (t % kLanes + (int)(blockIdx.x % PARTS) * kLanes);
  const int g = t / kLanes;
  const float* op = o_part + row * D + d;
  const int64_t stride = nrows * D;
  f32x4 first[kFirst];
#pragma unroll
  for (int i = 0; i < kFirst; ++i) {
    const int sp = min(g + i * kGroups, S - 1);
    first[i] = *reinterpret_cast<const f32x4*>(op + sp * stride);
  }
  const float ms = t < S ? m_part[t * nrows + row] : -INFINITY;
  const float ls = t < S ? l_part[t * nrows + row] : 0.f;
  float M = ms;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
  if ((t & 63) == 0) wmax[t >> 6] = M;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kNW; ++i) M = fmaxf(M, wmax[i]);
  const float f = ms == -INFINITY ? 0.f : fast_exp2(ms - M);
  w[t] = f;
  float L = ls * f;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off, 64);
  if ((t & 63) == 0) wsum[t >> 6] = L;
  __syncthreads();
  L = 0.f;
#pragma unroll
  for (int i = 0; i < kNW; ++i) L += wsum[i];
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < kFirst; ++i) {
    const int sp = g + i * kGroups;
    if (sp < S) acc += first[i] * w[sp];
  }
#pragma unroll 4
  for (int sp = g + kFirst * kGroups; sp < S; sp += kGroups)
    acc += *reinterpret_cast<const f32x4*>(op + sp * stride) * w[sp];
#pragma unroll
  for (int off = kLanes; off < 64; off <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
  if ((t & 63) < kLanes) part[t >> 6][t & 63] = acc;
  __syncthreads();
  if (t >= kLanes) return;
#pragma unroll
  for (int i = 1; i < kNW; ++i) acc += part[i][t];
  *reinterpret_cast<f32x4*>(o + row * D + d) = acc * (L > 0.f ? 1.f / L : 0.f);
  if (d == 0) {
    const int h = (int)(row % Hq);
    const int64_t bi = row / Hq;
    const int64_t si = (bi / Nq * Hq + h) * Nq + bi % Nq;
    m[si] = L > 0.f ? M * kLn2 : -INFINITY;
    l[si] = L;
  }
}

// Query rows per workgroup: 32 once a (batch, KV head) has more than 16.
int row_block(const Problem& p) { return (int64_t)p.Nq * (p.Hq / p.Hkv) <= 16 ? 16 : 32; }

int64_t row_blocks(const Problem& p) {
  const int64_t rows = (int64_t)p.Nq * (p.Hq / p.Hkv);
  return (rows + row_block(p) - 1) / row_block(p);
}

// Waves per workgroup.  Four waves that share a region of the cache and merge
// in LDS (fewer partials, often none) are the faster for most shapes: 16,001
// keys x 8 KV heads and 32 rows 22.4 us against 28.4 with one-wave workgroups
// and 30.0 with eight; 8,001 keys and 4 rows 12.7 / 16.9 / 16.0; 16 sequences
// of 4,000 keys 52.7 / 55.9 / 82.4.  A long single stream is the exception:
// one-wave workgroups put the same keys of up to eight KV heads, adjacent in
// memory, on one CU, which reads 262,144 keys x 8 heads at 6.4 against 5.5
// TB/s (1,000,000 x 16 at 6.2 against 5.7; 60,000 x 8 in 45 us against 46).
int waves_for(const Problem& p) {
  const int64_t units = (int64_t)p.B * p.Hkv * row_blocks(p);
  const int64_t tiles = (int64_t)p.Nk * p.D * 2 / kTileBytes;
  return units <= 16 && tiles * units >= 6 * kWaveSlots ? kStreamWaves : kWaves;
}

// Workgroups per (batch, KV head, row block).  A workgroup saturates its CU's
// share of the memory, so their number should be just below a multiple of the
// 256 CUs: the S for up to four per CU that takes the fewest tile steps, a
// start counting as one (8 KV heads: 8,000 keys 13.0 us with 32 splits against
// 14.8 with 48 and 16.4 with 16, 24,000 keys 23.8 / 26.4 / 26.6; 14 KV heads x
// 20,000 keys 30.8 us with 224 workgroups against 41.2 with 266).  Once every
// wave would walk twelve tiles eight per CU even out the CUs' rates (64 KV
// heads x 50,000 keys of 64 135 us against 150 with four, 256 heads x 60,000
// 1.22 ms against 1.33); short caches take a tile per wave (4,000 keys 9.8 us
// against 11.6 at two).  Up to four tiles a wave one workgroup saves the merge's
// launch: on the GPU it is as fast to 300 keys of 128 and slower from there (512
// keys, 8 KV heads 12.2 us against 8.6, one CU reading what four could), but a
// call from Python takes 14.7 us against 17.6, and a decoder layer, bound by
// the GPU, 88.8 against 87.1 at 500 keys and 86.0 against 87.5 at 300.
int choose_splits(const Problem& p) {
  const int64_t units = (int64_t)p.B * p.Hkv * row_blocks(p);
  const int tk = kTileBytes / (2 * p.D);
  const int64_t tiles = ((int64_t)p.Nk + tk - 1) / tk, waves = waves_for(p);
  const int64_t most = std::min<int64_t>((tiles + waves - 1) / waves, kMaxSplits);
  if (tiles <= 4 * waves) return 1;
  if (waves == kStreamWaves) return (int)std::min((kWaveSlots + units - 1) / units, most);
  int64_t best = 1, best_steps = INT64_MAX;
  for (int64_t k = 1; k <= 4; ++k) {
    const int64_t s = std::min(std::max<int64_t>(1, 256 * k / units), most);
    const int64_t steps = ((units * s + 255) / 256) * ((tiles + s * waves - 1) / (s * waves) + 1);
    if (steps < best_steps) {
      best = s;
      best_steps = steps;
    }
  }
  if (tiles >= 12 * waves * best) best = std::min(std::max(best, kWaveSlots / units), most);
  return (int)best;
}

size_t partial_bytes(const Problem& p, int64_t S) {
  const int64_t rows = (int64_t)p.B * p.Nq * p.Hq;
  return (size_t)(S * rows * p.D * 4 + 2 * S * rows * 4);
}

// The shapes whose workspace size is part of the ABI since its first version:
// callers size buffers by it and a smaller workspace is an error.
bool fixed_workspace(const Problem& p) { return p.D == 128 && row_block(p) == 16; }

// Splits that size takes: one per wave of eight waves per CU, at least two
// 32-key tiles per split.
int64_t fixed_splits(const Problem& p) {
  const int64_t tiles = ((int64_t)p.Nk + 31) / 32;
  const int64_t want = (2048 + (int64_t)p.B * p.Hkv - 1) / ((int64_t)p.B * p.Hkv);
  const int64_t most = std::max<int64_t>(1, tiles / 2);
  return std::min<int64_t>(std::min<int64_t>(std::max<int64_t>(1, want), most), 4096);
}

// Where the blockwise forward (one walk of the cache per query head, up to 128
// query rows at once) is not the better choice; the shapes with a required
// workspace run here in any case.  Times are this kernel's over the forward's.
bool splits_pay(const Problem& p) {
  const int64_t rb = row_blocks(p), units = (int64_t)p.B * p.Hkv * rb, group = p.Hq / p.Hkv;
  const int64_t tk = kTileBytes / (2 * p.D), tiles = ((int64_t)p.Nk + tk - 1) / tk;
  // A full chip of heads that share KV heads: the forward walks each cache
  // `group` times (64 sequences, 32/8 heads, 8 tokens: 0.4-0.9).
  if (group >= 4 * rb && (int64_t)p.B * p.Hq > 256) return true;
  // Otherwise long caches of few sequences.  head_dim 128: the forward is as
  // fast on the first few hundred keys (1.0-1.2) and, reading the cache once
  // for all rows, on grids of 256 and more (64 rows: 1.3-2.4, 17 rows over
  // 2,000 keys and more 1.0-1.3).
  if (p.D == 128) return units < 256 && tiles > 6 * (rb + 1);
  // head_dim 64: the forward splits keys over its waves too, which is as good
  // as one workgroup per unit (up to 1,024 keys 1.0-1.4, and 0.7-0.9 from 2,000
  // on); with two row blocks it takes more keys per sequence (8 KV heads: 1.9
  // at 1,000 keys, 0.9 at 2,000; 32: 1.0 at 4,000; 128 and more: 1.3-2.1).
  if (rb == 1) return units < 512 && tiles > 16;
  return units < 256 && tiles > std::max<int64_t>(24, units);
}

}  // namespace

int decode_splits(const Problem& p) {
  const int s = choose_splits(p);
  return fixed_workspace(p) ? (int)std::min<int64_t>(s, fixed_splits(p)) : s;
}

bool decode_supported(const Problem& p) {
  return p.dtype == 1 && !p.precise && (p.D == 64 || p.D == 128) && p.Nq > 0 &&
         (int64_t)p.Nq * (p.Hq / p.Hkv) <= kDecodeMaxRows && (fixed_workspace(p) || splits_pay(p));
}

bool decode_workspace_required(const Problem& p) { return fixed_workspace(p); }

size_t decode_workspace_bytes(const Problem& p) {
  if (fixed_workspace(p)) return partial_bytes(p, fixed_splits(p));
  const int s = decode_splits(p);
  return s > 1 ? partial_bytes(p, s) : 0;
}

hipError_t decode_static_scratch(hipStream_t st, void** ptr) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  // The kernels run on the stream's device, so the array must be that
  // device's copy: a null stream means the current device.
  int cur = 0;
  hipError_t e = hipGetDevice(&cur);
  if (e != hipSuccess) return e;
  int dev = cur;
  if (st != nullptr) {
    hipDevice_t sd = 0;
    e = hipStreamGetDevice(st, &sd);
    if (e != hipSuccess) return e;
    dev = (int)sd;
  }
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (addr[dev] == nullptr) {
    // hipGetSymbolAddress resolves the symbol on the current device: make
    // the stream's device current for the lookup, then restore the caller's.
    if (dev != cur && (e = hipSetDevice(dev)) != hipSuccess) return e;
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (dev != cur) {
      const hipError_t r = hipSetDevice(cur);
      if (e == hipSuccess) e = r;
    }
    if (e != hipSuccess) return e;
    addr[dev] = p;
  }
  *ptr = addr[dev];
  return hipSuccess;
}

hipError_t launch_decode(const Problem& p, const void* q, const void* k, const void* v, float* o,
                         float* m, float* l, void* ws, hipStream_t st) {
  if (!decode_supported(p)) return hipErrorInvalidValue;
  const int S = decode_splits(p);
  const int64_t rows = (int64_t)p.B * p.Nq * p.Hq;
  DecodeArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.o = o;
  a.m = m;
  a.l = l;
  a.o_part = static_cast<float*>(ws);
  a.m_part = a.o_part + (int64_t)S * rows * p.D;
  a.l_part = a.m_part + (int64_t)S * rows;
  a.Nq = p.Nq;
  a.Nk = p.Nk;
  a.Hq = p.Hq;
  a.Hkv = p.Hkv;
  a.group = p.Hq / p.Hkv;
  a.rows = p.Nq * a.group;
  a.row_blocks = (int)row_blocks(p);
  a.S = S;
  a.prows = rows;
  const int tk = kTileBytes / (2 * p.D);
  const int64_t tiles = ((int64_t)p.Nk + tk - 1) / tk;
  a.chunk = (int)((tiles + S - 1) / S * tk);
  a.q_pos0 = p.q_pos0;
  a.k_pos0 = p.k_pos0;
  a.valid = p.valid;
  a.causal = p.causal ? 1 : 0;
  a.sl2 = p.scale * kLog2e;
  const int64_t wgs = (int64_t)S * a.row_blocks * p.Hkv * p.B;
  auto split = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(64 * waves), 0, st, a);
  };
  auto rows_of = [&](auto d, auto w) {
    constexpr int kD = decltype(d)::value, kW = decltype(w)::value;
    if (row_block(p) == 32) split(decode_kernel<kD, 2, kW>, kW);
    else split(decode_kernel<kD, 1, kW>, kW);
  };
  auto waves_of = [&](auto d) {
    if (waves_for(p) == kWaves) rows_of(d, std::integral_constant<int, kWaves>{});
    else rows_of(d, std::integral_constant<int, kStreamWaves>{});
  };
  if (p.D == 128) waves_of(std::integral_constant<int, 128>{});
  else waves_of(std::integral_constant<int, 64>{});
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || S == 1) return e;
  auto merge = [&](auto kernel, int threads, int parts) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(rows * parts)), dim3(threads), 0, st, rows, S, p.Nq,
                       p.Hq, a.o_part, a.m_part, a.l_part, o, m, l);
  };
  if (p.D == 128 && S > 64) merge(decode_merge_kernel<128, 1024, 4>, 1024, 4);
  else if (p.D == 128) merge(decode_merge_kernel<128, 256, 1>, 256, 1);
  else if (S > 64) merge(decode_merge_kernel<64, 1024, 4>, 1024, 4);
  else merge(decode_merge_kernel<64, 256, 1>, 256, 1);
  return hipGetLastError();
}

}  // namespace lc
