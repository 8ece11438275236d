// k_attn16.hip -- causal attention at head width 64 on bf16 operands held in
// HBM as bf16: forward, dQ and dK / dV over the tiled family's stats-row
// contract (instruction.h:174-190, 234-259), for the models that train in
// bf16 activations (BASELINE configs[2] bf16, [3], [4]).
//
// Staging.  Every tile that enters a product is a 64-row block of one
// (b, h) slice -- 64 rows x 64 dims of bf16 -- copied from HBM straight into
// LDS by buffer_load ... lds (no registers, no conversion).  A tile is two
// halves (dims 0-31, 32-63) of 64-byte rows; chunk c (16 bytes) of row r
// sits at physical chunk (c + r / 4) mod 4, which keeps the MFMA fragment
// reads free of bank conflicts (the W8A8 kernel's measured rotation).  Rows
// past the sequence end read as zeros through the buffer range check.
//
// Products.  v_mfma_f32_32x32x16_bf16 with the scores formed transposed
// (S^T = K Q^T): the accumulator layout -- lane (g = lane / 32, c = lane %
// 32) holding rows 8q + 4g + e of column c -- is then the B operand of the
// next product, so probabilities never leave registers.  Operands whose
// reduction index runs down a tile's rows (V^T in O^T = V^T P^T, K^T in
// dQ^T = K^T dS^T, Q^T and dO^T in dK^T / dV^T) are read with gfx950's
// ds_read_b64_tr_b16, which hands each lane one column of a 4 x 16 block
// gathered from its 16-lane group: no transposed copies.
//
// Every output element has one writer; no atomics; the reductions run in a
// fixed order, so results repeat bit for bit.
#include "attn_tile.h"

namespace seeai {
namespace {

// ---------------------------------------------------------------------------
// Forward.  A workgroup of kFwdWaves waves owns kFwdWaves * 32 queries of one
// (b, h), 32 per wave.  Keys stream in 64-row blocks through two stage
// buffers.  The scores arrive as q.k; x = q.k * log2(e)/sqrt(d) - m_use (one
// FMA) is the base-2 exponent of the weight.
//
// Lazy offset.  Lane (g, c) holds 16 of query c's scores per tile, lane
// (1 - g, c) the other 16, and both must weigh against the same m_use.  Each
// half tracks its own maximum; m_use moves only when some half's tile
// maximum passes it by more than 2^8, or on the first tile a half sees --
// rare events, in which the pair first agrees on its maximum by one lane
// swap.  The common tile therefore has no cross-lane traffic: l and the true
// maximum are per half until the end.  The stats row (m, 1/l) is stated
// against the true maximum; l sums the bf16-rounded weights that enter P V.
//
// Every tile runs one body; on the diagonal (and at document starts) a
// uniform branch masks the exponents, so the accumulators keep their
// registers across the branch.
// ---------------------------------------------------------------------------
constexpr float kLazy = 8.0f;

template <int kFwdWaves, int kStages, int kMinBlocks>
__global__ void __launch_bounds__(kFwdWaves * kWave, kMinBlocks)
Attn16Fwd(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
          const uint16_t* __restrict__ v, float* __restrict__ o, float* __restrict__ stats, int S,
          int H, const int32_t* __restrict__ starts, Bf16Sink sink) {
  constexpr int kFwdRows = kFwdWaves * 32;
  SEEAI_STAGE_RING(kStages);
  __shared__ int wave_lo[kFwdWaves];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 32, c = lane % 32;
  const int nq = (S + kFwdRows - 1) / kFwdRows;
  int bh, rank;
  UnitOf(nq, bh, rank);
  const int qblk = nq - 1 - rank;
  const int b = bh / H, h = bh % H;
  const int ld = H * kD;
  const size_t base = static_cast<size_t>(b) * S * ld + static_cast<size_t>(h) * kD;
  const int qw = qblk * kFwdRows + wave * 32;  // this wave's first query
  const int i = qw + c;
  const int ic = min(i, S - 1);
  int jstart = 0;
  if (starts) {
    const int v0 = starts[static_cast<size_t>(b) * S + ic];
    jstart = v0 <= 0 ? 0 : min(v0, ic);
  }
  const int w_hi_start = WaveMaxI(jstart);
  if (lane == 0) wave_lo[wave] = WaveMinI(jstart);
  __syncthreads();
  int lo = wave_lo[0];
#pragma unroll
  for (int w = 1; w < kFwdWaves; ++w) lo = min(lo, wave_lo[w]);
  const int blk_lo = Uniform(lo) / kBlkRows;
  const int q_hi = min(qblk * kFwdRows + kFwdRows - 1, S - 1);
  const int nblk = q_hi / kBlkRows + 1 - blk_lo;

  bf16x8 qf[4];
  {
    const uint16_t* row = q + base + static_cast<size_t>(ic) * ld;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = OwnedFrag(row, s, lane);
  }
  const float scl = kLog2e * 0.125f;  // log2(e) / sqrt(64)

  // Loads: per stage 16 wave-loads (K then V, 2 halves x 4 row groups); wave
  // w takes u = kFwdWaves j + w.
  constexpr int kLoadsPerWave = 16 / kFwdWaves;
  static_assert(kLoadsPerWave * kFwdWaves == 16, "16 wave-loads per block");
  int voff[kLoadsPerWave];
#pragma unroll
  for (int j = 0; j < kLoadsPerWave; ++j)
    voff[j] = TileLoadOffset((kFwdWaves * j + wave) % 8, lane, ld);
  auto issue = [&](int jb, uint8_t* st) {
    const int j0 = (blk_lo + jb) * kBlkRows;
    const __amdgpu_buffer_rsrc_t rk = SliceRsrc(k + base, ld, S, j0);
    const __amdgpu_buffer_rsrc_t rv = SliceRsrc(v + base, ld, S, j0);
#pragma unroll
    for (int j = 0; j < kLoadsPerWave; ++j) {
      const int u = kFwdWaves * j + wave;
      if (u < 8)
        TileLoad(rk, st, u, voff[j]);
      else
        TileLoad(rv, st + kTile, u - 8, voff[j]);
    }
  };

  const FragOffsets fo = MakeFragOffsets(lane);
  v16f oacc[2] = {};  // [dt]
  float m_use = 0.0f, m_half = -INFINITY, l_half = 0.0f;
  float thr = -INFINITY;  // a half's tile maximum above this moves m_use: -inf until it sees a score

  const bf16x2 ones = {static_cast<__bf16>(1.0f), static_cast<__bf16>(1.0f)};

  // A 32-key tile kt of a staged block: S^T = K Q^T (four MFMAs) ...
  auto scores = [&](const uint8_t* kt_tile, int kt) {
    v16f sc = {};
#pragma unroll
    for (int s = 0; s < 4; ++s) sc = Mfma(RowFrag(kt_tile, fo, 32 * kt, s), qf[s], sc);
    return sc;
  };
  // ... the softmax weights (VALU) and O^T += V^T P^T (four MFMAs).
  auto weigh = [&](const v16f& sc, bool masked, const uint8_t* vt_tile, int kt, int jt) {
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = __builtin_fmaf(sc[r], scl, -m_use);
    if (masked) {  // keep key jt + row in [jstart, i]
      const int hi_rel = i - jt - 4 * g, lo_rel = jstart - jt - 4 * g;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        x[r] = OrNegInf(x[r], Outside(hi_rel - RowConst(r), RowConst(r) - lo_rel));
    }
    float hmax = x[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) hmax = fmaxf(hmax, x[r]);  // relative to m_use
    const float m_prev = m_half;
    m_half = fmaxf(m_half, m_use + hmax);
    if (__any(hmax > thr)) {
      const float bmax = SwapMax(hmax);
      const bool first = SwapMax(m_prev) == -INFINITY;
      const bool need = first ? bmax != -INFINITY : bmax > kLazy;
      const float shift = need ? bmax : 0.0f;
      const float alpha = first ? 0.0f : Exp2(-shift);
      m_use += shift;
      l_half *= alpha;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) oacc[dt] *= alpha;
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] -= shift;
      thr = m_half == -INFINITY ? -INFINITY : kLazy;
    }
    float p[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = Exp2(x[r]);
    bf16x8 pb[2];
    PackTile(p, pb);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        l_half = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{pb[hh][2 * e], pb[hh][2 * e + 1]}, ones,
                                                 l_half, false);
    // O^T += V^T P^T over the tile's 32 keys (two 16-key steps).
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
        oacc[dt] = Mfma(ColFrag(vt_tile, fo, dt, 32 * kt + 16 * hh), pb[hh], oacc[dt]);
  };

  const int qmin = qw, qmax = qw + 31;
  auto step = [&](int jb, const uint8_t* cur) {
    const int j0 = (blk_lo + jb) * kBlkRows;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const int jt = j0 + 32 * kt;
      if (jt > qmax) continue;  // keys wholly after this wave's queries
      weigh(scores(cur, kt), !(jt + 31 <= qmin && jt >= w_hi_start), cur + kTile, kt, jt);
    }
  };
  RunRing<kStages, kLoadsPerWave>(nblk, issue, step, stage);

  const float l = SwapSum(l_half);
  const float m_true = SwapMax(m_half);
  if (i >= S) return;
  const float inv = 1.0f / l;
  const size_t orow0 = base + static_cast<size_t>(i) * ld;
  float* orow = o + orow0;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      const float4 ov = make_float4(oacc[dt][4 * qq] * inv, oacc[dt][4 * qq + 1] * inv,
                                    oacc[dt][4 * qq + 2] * inv, oacc[dt][4 * qq + 3] * inv);
      const int col = dt * 32 + 8 * qq + 4 * g;
      if (sink.store_f32) *reinterpret_cast<float4*>(orow + col) = ov;
      if (sink.out) SinkStore4(sink, orow0 + col, ov);  // the next product's bf16 A'
    }
  if (g == 0) {
    float* sr = stats + (static_cast<size_t>(bh) * S + i) * 4;
    sr[0] = m_true * kLn2;
    sr[1] = inv * Exp2(m_true - m_use);
    sr[2] = 0.0f;
    sr[3] = static_cast<float>(jstart);
  }
}

// Row offset of the base-2 exponent: p = 2^(s c - mm) with c = log2(e)/8
// and mm = m log2(e) + log2(l), from the stats row (m, 1/l).
__device__ __forceinline__ float RowOffset(float m, float inv) { return m * kLog2e - log2f(inv); }

// Stats start column: the document start stored as a float (instruction.h:
// 246-250), clamped to the row.
__device__ __forceinline__ int StatsStart(float stored, int i) {
  if (!(stored > 0.0f)) return 0;
  const float cap = static_cast<float>(i);
  return stored >= cap ? i : static_cast<int>(stored);
}

// ---------------------------------------------------------------------------
// dQ and the stats row's delta = sum_j p dP, in one walk over K / V: with
// dS = p (dP - delta) linear in delta,
//   dQ^T = K^T (p dP)^T - delta K^T p^T,
// and delta accumulates beside the two products (four per tile -- S^T,
// dP^T and the two accumulations -- one exponential per score).  Four waves
// of 32 queries; K and V blocks staged as in the forward, K^T read by
// transpose reads.  dQ is scaled by 1/sqrt(d) once, at the end.
// ---------------------------------------------------------------------------
constexpr int kBwdWaves = 4;
constexpr int kBwdRows = kBwdWaves * 32;

template <int kStages, int kMinBlocks>
__global__ void __launch_bounds__(kBwdWaves * kWave, kMinBlocks)
Attn16DQ(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
         const uint16_t* __restrict__ v, const uint16_t* __restrict__ dout,
         float* __restrict__ stats, float* __restrict__ dq, int S, int H) {
  SEEAI_STAGE_RING(kStages);
  __shared__ int wave_lo[kBwdWaves];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 32;
  const int nq = (S + kBwdRows - 1) / kBwdRows;
  int bh, rank;
  UnitOf(nq, bh, rank);
  const int qblk = nq - 1 - rank;
  const int b = bh / H, h = bh % H;
  const int ld = H * kD;
  const size_t base = static_cast<size_t>(b) * S * ld + static_cast<size_t>(h) * kD;
  const int qw = qblk * kBwdRows + wave * 32;
  const int i = qw + lane % 32;
  const int ic = min(i, S - 1);
  float* st = stats + (static_cast<size_t>(bh) * S + ic) * 4;
  const float4 st4 = *reinterpret_cast<const float4*>(st);
  const float mm = RowOffset(st4.x, st4.y);
  const int jstart = StatsStart(st4.w, ic);
  const int w_hi_start = WaveMaxI(jstart);
  if (lane == 0) wave_lo[wave] = WaveMinI(jstart);
  __syncthreads();
  int lo = wave_lo[0];
#pragma unroll
  for (int w = 1; w < kBwdWaves; ++w) lo = min(lo, wave_lo[w]);
  const int blk_lo = Uniform(lo) / kBlkRows;
  const int q_hi = min(qblk * kBwdRows + kBwdRows - 1, S - 1);
  const int nblk = q_hi / kBlkRows + 1 - blk_lo;
  const float scl = kLog2e * 0.125f;

  bf16x8 qf[4], df[4];
  {
    const uint16_t* qrow = q + base + static_cast<size_t>(ic) * ld;
    const uint16_t* drow = dout + base + static_cast<size_t>(ic) * ld;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = OwnedFrag(qrow, s, lane), df[s] = OwnedFrag(drow, s, lane);
  }
  int voff[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) voff[j] = TileLoadOffset((4 * j + wave) % 8, lane, ld);
  auto issue = [&](int jb, uint8_t* sb) {
    const int j0 = (blk_lo + jb) * kBlkRows;
    const __amdgpu_buffer_rsrc_t rk = SliceRsrc(k + base, ld, S, j0);
    const __amdgpu_buffer_rsrc_t rv = SliceRsrc(v + base, ld, S, j0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int u = 4 * j + wave;
      if (u < 8)
        TileLoad(rk, sb, u, voff[j]);
      else
        TileLoad(rv, sb + kTile, u - 8, voff[j]);
    }
  };
  const FragOffsets fo = MakeFragOffsets(lane);
  v16f acc[2] = {}, acc_p[2] = {};  // [dt]
  float delta = 0.0f;

  // A 32-key tile kt: S^T = K Q^T and dP^T = V dO^T (eight MFMAs) ...
  auto front = [&](const uint8_t* ktile, const uint8_t* vtile, int kt, v16f& sc, v16f& dp) {
    sc = v16f{};
    dp = v16f{};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      sc = Mfma(RowFrag(ktile, fo, 32 * kt, s), qf[s], sc);
      dp = Mfma(RowFrag(vtile, fo, 32 * kt, s), df[s], dp);
    }
  };
  // ... the weights (VALU) and the two accumulations (eight MFMAs).
  auto back = [&](const v16f& sc, const v16f& dp, bool masked, const uint8_t* ktile, int kt,
                  int jt) {
    float w[16], p[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = Exp2(__builtin_fmaf(sc[r], scl, -mm));
    if (masked) {  // keep key jt + row in [jstart, i]
      const int hi_rel = i - jt - 4 * g, lo_rel = jstart - jt - 4 * g;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        p[r] = OrZero(p[r], Outside(hi_rel - RowConst(r), RowConst(r) - lo_rel));
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      delta = __builtin_fmaf(dp[r], p[r], delta);
      w[r] = p[r] * dp[r];
    }
    bf16x8 wb[2], pb[2];
    PackTile(w, wb);
    PackTile(p, pb);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        const bf16x8 kf = ColFrag(ktile, fo, dt, 32 * kt + 16 * hh);
        acc[dt] = Mfma(kf, wb[hh], acc[dt]);
        acc_p[dt] = Mfma(kf, pb[hh], acc_p[dt]);
      }
  };

  const int qmin = qw, qmax = qw + 31;
  auto step = [&](int jb, const uint8_t* cur) {
    const int j0 = (blk_lo + jb) * kBlkRows;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const int jt = j0 + 32 * kt;
      if (jt > qmax) continue;
      v16f sc, dp;
      front(cur, cur + kTile, kt, sc, dp);
      back(sc, dp, !(jt + 31 <= qmin && jt >= w_hi_start), cur, kt, jt);
    }
  };
  RunRing<kStages, 4>(nblk, issue, step, stage);
  delta = SwapSum(delta);
  if (i >= S) return;
  const float isd = 0.125f;
  float* drow = dq + base + static_cast<size_t>(i) * ld;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) {
    const v16f r = acc[dt] - delta * acc_p[dt];
#pragma unroll
    for (int qq = 0; qq < 4; ++qq)
      *reinterpret_cast<float4*>(drow + dt * 32 + 8 * qq + 4 * g) =
          make_float4(r[4 * qq] * isd, r[4 * qq + 1] * isd, r[4 * qq + 2] * isd,
                      r[4 * qq + 3] * isd);
  }
  if (g == 0) st[2] = delta;
}

// ---------------------------------------------------------------------------
// dK and dV: four waves of 32 keys walking the query blocks from the
// diagonal.  S = Q K^T and dP = dO V^T are formed query-major (Q and dO
// tiles as the row operand, K and V held in registers), so the score
// accumulator's layout is the k operand of dV^T = dO^T P and
// dK^T = Q^T dS, whose dO^T and Q^T come by transpose reads.  Per query
// row the exponent offset -mm and -delta come from a row-terms array
// staged beside the tiles; four products per tile, one exponential per
// score.  dK is scaled by 1/sqrt(d) once, at the end.
// ---------------------------------------------------------------------------
template <int kStages, int kMinBlocks>
__global__ void __launch_bounds__(kBwdWaves * kWave, kMinBlocks)
Attn16DKDV(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
           const uint16_t* __restrict__ v, const uint16_t* __restrict__ dout,
           const float* __restrict__ stats, float* __restrict__ out_k,
           float* __restrict__ out_v, int S, int H, Bf16Sink sink_v) {
  SEEAI_STAGE_RING(kStages);
  // Per streamed query row: -mm, -delta and the document start.  Rows are
  // contiguous, so a lane's 16 rows of a tile (8q + 4g + e) are four 16-byte
  // reads in accumulator order.
  __shared__ __attribute__((aligned(16))) float Smm[2][kBlkRows];
  __shared__ __attribute__((aligned(16))) float Sdl[2][kBlkRows];
  __shared__ int Sst[2][kBlkRows];
  __shared__ int Smax[2];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int g = lane / 32;
  const int nk = (S + kBwdRows - 1) / kBwdRows;
  int bh, kblk;
  UnitOf(nk, bh, kblk);  // rank 0 = the first keys, the longest columns
  const int b = bh / H, h = bh % H;
  const int ld = H * kD;
  const size_t base = static_cast<size_t>(b) * S * ld + static_cast<size_t>(h) * kD;
  const int jw = kblk * kBwdRows + wave * 32;
  const int j = jw + lane % 32;
  const int jc = min(j, S - 1);
  const float scl = kLog2e * 0.125f;
  const float4* st_bh = reinterpret_cast<const float4*>(stats) + static_cast<size_t>(bh) * S;

  bf16x8 kf[4], vf[4];
  {
    const uint16_t* krow = k + base + static_cast<size_t>(jc) * ld;
    const uint16_t* vrow = v + base + static_cast<size_t>(jc) * ld;
#pragma unroll
    for (int s = 0; s < 4; ++s) kf[s] = OwnedFrag(krow, s, lane), vf[s] = OwnedFrag(vrow, s, lane);
  }
  const int blk_first = (kblk * kBwdRows) / kBlkRows;
  int nblk = (S + kBlkRows - 1) / kBlkRows - blk_first;
  __shared__ LiveBlocks live;
  const int nlive = ListLiveBlocks<kBwdWaves * kWave>(
      live, S, blk_first, nblk, kblk * kBwdRows + kBwdRows - 1,
      [&](int row) { return StatsStart(st_bh[row].w, row); });
  if (nlive >= 0) nblk = nlive;
  // Blocks ib, ib + 1 and ib + 2 of the walk (past its end, the last), one looked
  // up a block: looking up each where it is used, four times a block, took dK /
  // dV without documents from 34.2 to 34.6 us at B4 H3 S1159.
  const auto block = [&](int ib) {
    const int n = min(ib, nblk - 1);
    return blk_first + (nlive >= 0 ? Uniform(live.idx[n]) : n);
  };
  int blk0 = block(0), blk1 = block(1), blk2 = block(2);
  int voff[4];
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) voff[jj] = TileLoadOffset((4 * jj + wave) % 8, lane, ld);
  static_assert(kStages == 2, "a block's loads go out while the one before is computed");
  auto issue_block = [&](int blk, uint8_t* sb) {
    const int r0 = blk * kBlkRows;
    const __amdgpu_buffer_rsrc_t rq = SliceRsrc(q + base, ld, S, r0);
    const __amdgpu_buffer_rsrc_t rd = SliceRsrc(dout + base, ld, S, r0);
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int u = 4 * jj + wave;
      if (u < 8)
        TileLoad(rq, sb, u, voff[jj]);
      else
        TileLoad(rd, sb + kTile, u - 8, voff[jj]);
    }
  };
  // The row terms of block ib, by wave 0 (64 queries): fetched from HBM one
  // block ahead of their store into LDS, so the load's latency hides behind
  // a block's products.
  float4 pend = {};
  auto fetch = [&](int blk) {
    const int iq = blk * kBlkRows + lane;
    if (iq < S) pend = st_bh[iq];
  };
  auto put = [&](int blk, int buf) {
    const int iq = blk * kBlkRows + lane;
    int start = 0;
    if (iq < S) {
      Smm[buf][lane] = -RowOffset(pend.x, pend.y);
      Sdl[buf][lane] = -pend.z;
      start = StatsStart(pend.w, iq);
    } else {
      Smm[buf][lane] = -INFINITY;  // weight 0 past the sequence end
      Sdl[buf][lane] = 0.0f;
    }
    Sst[buf][lane] = start;
    const int mx = WaveMaxI(start);
    if (lane == 0) Smax[buf] = mx;
  };
  // This lane's 16 per-row values of tile qt (rows 8q + 4g + e).
  // A lane's 16 values of one row-term array for tile qt, in accumulator
  // order.
  auto rows16 = [&](const float* terms, int qt) {
    v16f r;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const float4 a = *reinterpret_cast<const float4*>(terms + qt * 32 + 8 * q4 + 4 * g);
      r[4 * q4] = a.x, r[4 * q4 + 1] = a.y, r[4 * q4 + 2] = a.z, r[4 * q4 + 3] = a.w;
    }
    return r;
  };
  const FragOffsets fo = MakeFragOffsets(lane);
  v16f acc_k[2] = {}, acc_v[2] = {};  // [dt]

  // A 32-query tile qt: S = Q K^T and dP = dO V^T (eight MFMAs) ...
  // dP starts at -delta, so the product arrives as dP - delta.
  auto front = [&](const uint8_t* qtile, const uint8_t* dtile, int buf, int qt, v16f& sc,
                   v16f& dp) {
    sc = v16f{};
    dp = rows16(Sdl[buf], qt);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      sc = Mfma(RowFrag(qtile, fo, 32 * qt, s), kf[s], sc);
      dp = Mfma(RowFrag(dtile, fo, 32 * qt, s), vf[s], dp);
    }
  };
  // ... the weights (VALU) and dK^T += Q^T dS, dV^T += dO^T P (eight MFMAs).
  auto back = [&](const v16f& sc, const v16f& dp, bool masked, const uint8_t* qtile,
                  const uint8_t* dtile, int buf, int qt, int r0) {
    const v16f mmv = rows16(Smm[buf], qt);
    float w[16], p[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = Exp2(__builtin_fmaf(sc[r], scl, mmv[r]));
    if (masked) {  // keep query row >= j and its start <= j
      const int lo_rel = r0 + 32 * qt + 4 * g - j;  // query row minus this lane's key
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int il = qt * 32 + RowConst(r) + 4 * g;
        p[r] = OrZero(p[r], Outside(lo_rel + RowConst(r), j - Sst[buf][il]));
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) w[r] = p[r] * dp[r];
    bf16x8 wb[2], pb[2];
    PackTile(w, wb);
    PackTile(p, pb);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        acc_k[dt] = Mfma(ColFrag(qtile, fo, dt, 32 * qt + 16 * hh), wb[hh], acc_k[dt]);
        acc_v[dt] = Mfma(ColFrag(dtile, fo, dt, 32 * qt + 16 * hh), pb[hh], acc_v[dt]);
      }
  };

  // Row terms run one block ahead of the tiles (two LDS buffers, by
  // parity): block ib's are stored during block ib - 1, from a load issued
  // during block ib - 2.
  if (wave == 0) {
    fetch(blk0);
    put(blk0, 0);
    if (1 < nblk) fetch(blk1);
  }
  auto step = [&](int ib, const uint8_t* cur) {
    const int buf = ib & 1;
    if (wave == 0 && ib + 1 < nblk) {
      put(blk1, buf ^ 1);
      if (ib + 2 < nblk) fetch(blk2);
    }
    const int r0 = blk0 * kBlkRows;
    blk0 = blk1, blk1 = blk2, blk2 = block(ib + 3);
    const int smax = Uniform(Smax[buf]);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int rt = r0 + 32 * qt;
      if (rt + 31 < jw) continue;  // queries wholly before this wave's keys
      v16f sc, dp;
      front(cur, cur + kTile, buf, qt, sc, dp);
      back(sc, dp, !(rt >= jw + 31 && rt + 32 <= S && smax <= jw), cur, cur + kTile, buf, qt, r0);
    }
  };
  auto issue = [&](int ib, uint8_t* sb) { issue_block(ib == 0 ? blk0 : blk1, sb); };
  RunRing<kStages, 4>(nblk, issue, step, stage);
  if (j >= S) return;
  const float isd = 0.125f;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      const size_t at = base + static_cast<size_t>(j) * ld + dt * 32 + 8 * qq + 4 * g;
      if (out_k)
        *reinterpret_cast<float4*>(out_k + at) =
            make_float4(acc_k[dt][4 * qq] * isd, acc_k[dt][4 * qq + 1] * isd,
                        acc_k[dt][4 * qq + 2] * isd, acc_k[dt][4 * qq + 3] * isd);
      if (out_v) {
        const float4 v4 = make_float4(acc_v[dt][4 * qq], acc_v[dt][4 * qq + 1],
                                      acc_v[dt][4 * qq + 2], acc_v[dt][4 * qq + 3]);
        *reinterpret_cast<float4*>(out_v + at) = v4;
        if (sink_v.out) SinkStore4(sink_v, at, v4);  // a later product's copy of dV
      }
    }
}

}  // namespace

bool Attn16Fits(size_t B, size_t S, size_t H, size_t d) {
  return d == kD && S > 0 && (S - 1) * H * kD * 2 + kD * 2 < (size_t{1} << 31) &&
         (S + 127) / 128 * B * H < (size_t{1} << 31);
}

hipError_t LaunchAttn16Fwd(const uint16_t* q, const uint16_t* k, const uint16_t* v, float* o,
                           float* stats, size_t B, size_t S, size_t H, const int32_t* starts,
                           hipStream_t s, const Bf16Sink& sink) {
  if (B * H * S == 0) return hipSuccess;
  // Four waves, two stages, four workgroups per CU (measured against 3-4
  // stages and 8-wave workgroups at B16 H16 S2048).
  const dim3 grid(static_cast<unsigned>((S + 127) / 128 * B * H));
  hipLaunchKernelGGL((Attn16Fwd<4, 2, 4>), grid, dim3(256), 0, s, q, k, v, o, stats,
                     static_cast<int>(S), static_cast<int>(H), starts, sink);
  return hipGetLastError();
}

hipError_t LaunchAttn16DQ(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                          const uint16_t* dout, float* stats, float* dq, size_t B, size_t S,
                          size_t H, hipStream_t s) {
  if (B * H * S == 0) return hipSuccess;
  const dim3 grid(static_cast<unsigned>((S + kBwdRows - 1) / kBwdRows * B * H));
  // Three stages, three workgroups per CU (160 VGPRs, 48 KiB of LDS each).
  hipLaunchKernelGGL((Attn16DQ<3, 3>), grid, dim3(kBwdWaves * kWave), 0, s, q, k, v, dout, stats,
                     dq, static_cast<int>(S), static_cast<int>(H));
  return hipGetLastError();
}

hipError_t LaunchAttn16DKDV(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                            const uint16_t* dout, const float* stats, float* dk, float* dv,
                            size_t B, size_t S, size_t H, hipStream_t s, const Bf16Sink& sink_v) {
  if (B * H * S == 0) return hipSuccess;
  if (!dk && !dv) return hipErrorInvalidValue;
  if (sink_v.out && (!dv || !sink_v.store_f32)) return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>((S + kBwdRows - 1) / kBwdRows * B * H));
  // Two stages, two workgroups per CU (about 200 VGPRs).
  hipLaunchKernelGGL((Attn16DKDV<2, 2>), grid, dim3(kBwdWaves * kWave), 0, s, q, k, v, dout,
                     stats, dk, dv, static_cast<int>(S), static_cast<int>(H), sink_v);
  return hipGetLastError();
}

}  // namespace seeai
