// k_attn3.hip -- the exact family of causal attention (kAttnFwdTiled,
// kAttnDQTiled, kAttnDKTiled, kAttnDVTiled; source/plan/instruction.h:
// 158-259) at head width 64: f32 products formed on bf16 MFMA.  The
// reference's expressions per score (attention.cc:405-590): s = (q . k) /
// sqrt(d), p = exp(s - m) * (1/l), delta = sum_j p dP (in double), dS =
// p (dP - delta), dQ += (dS / sqrt(d)) k, dK += (dS / sqrt(d)) q, dV += p dO.
//
// Products.  Every f32 operand is split three ways, x = h + m + l, each part
// the bf16 nearest to what is left: 8 + 8 + 8 significant bits, so the parts
// hold x (to the last bit or so; below 2^-109 to 2^-134, where bf16 ends).  A
// product sums six of the nine part products -- hh in the accumulator, hm, mh,
// mm, hl, lh in one of their own that joins it at the end; the three left out are
// below 2^-26 of the operands' product -- each exact in the MFMA, summed in f32.
// Against float64 the results are as close as sums of v_mfma_f32_16x16x4f32 (a
// chain of rounded f32 terms) or closer: fewer roundings at the accumulator's
// magnitude.  Six bf16 products take 3/8 of the f32 MFMA's time, which bounded these kernels
// (v_mfma_f32_16x16x4f32 at 55-60 % of its rate).  us, f32 MFMA / here:
//
//   B8 H12 S1024     forward 175 / 114   dQ 414 / 240    dK + dV 350 / 258
//   B16 H16 S2048            1517 / 894     3626 / 2129          3229 / 2232
//   B1 H8 S328                 43 / 28        95 / 42              66 / 47
//
// 2-norm error against float64 at H4 S2048, f32 MFMA / here: unit normals O
// 4.0e-7 / 1.7e-7, dQ 4.6e-7 / 2.1e-7, dK 1.1e-6 / 4.3e-7, dV 1.1e-6 / 4.4e-7;
// scores of standard deviation 8, dQ 1.9e-6 / 7.9e-7; means of 3 in K and V, dQ
// 8.7e-6 / 7.3e-6.  What bounds them now is a wave's own chain (products, exps,
// splits) at 1.4 waves a SIMD (0.9 for dQ and dK / dV): MFMA busy 32 / 31 / 28 %,
// VALU 49 / 41 / 34 % of the forward, dQ, dK / dV at B8 H12 S1024.
//
// Geometry.  A workgroup of four waves owns 128 rows of one (b, h) -- queries
// for the forward and dQ, keys for dK / dV -- each wave 32 of them, their parts
// held as MFMA fragments.  The other side streams in 64-row blocks, split once
// as it is staged into three bf16 tiles in LDS; one buffer (48 KiB for the
// pair) and the next block in flight in registers, so two of the forward's
// workgroups share a CU and one multiplies while the other stages.  Tiles,
// fragments and the transposed score layout are k_attn16.hip's.
//
// An infinity, a NaN, or a float past the largest bf16 (3.3895e38) has no such
// parts: its last one is NaN, and with it every sum it joins.  A wave whose sums
// come out NaN forms its rows again in plain f32 (PlainFwd, PlainDQ, PlainDKDV),
// so they hold what f32 arithmetic gives and only where it does.
//
// Every output element has one writer and every sum a fixed order; dK and dV
// are one template, so the fused pass has the separate passes' bits.
#include "attn_tile.h"

namespace seeai {
namespace {

constexpr float kLog2eLo =  // log2(e) - kLog2e
    static_cast<float>(1.4426950408889634074 - static_cast<double>(kLog2e));

constexpr int kWaves = 4, kThreads = kWaves * kWave, kRowsWG = kWaves * 32;
constexpr float kIsd = 0.125f;  // 1 / sqrt(64)

// instruction.h:240-247: a stored start clamped into [0, i], NaN to 0.
__device__ __forceinline__ int StartOf(float stored, int i) {
  if (!(stored > 0.0f)) return 0;
  const float cap = static_cast<float>(i);
  return stored >= cap ? i : static_cast<int>(stored);
}

// Workgroup w -> (b, h) and its row block's rank, the longest first over all
// (b, h); with B H a multiple of 8 every block of a slice lands on one XCD (the
// hardware deals workgroups to XCDs round-robin).
__device__ __forceinline__ void UnitOf3(int nb, int& bh, int& rank) {
  const int units = gridDim.x / nb;
  bh = blockIdx.x % units;
  rank = blockIdx.x / units;
}

struct Parts {
  bf16x8 p[3];  // h, m, l
};
// Eight floats in their parts.
__device__ __forceinline__ Parts Split(const float (&x)[8]) {
  Parts r;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    r.p[0][i] = static_cast<__bf16>(x[i]);
    const float rest = x[i] - static_cast<float>(r.p[0][i]);
    r.p[1][i] = static_cast<__bf16>(rest);
    r.p[2][i] = static_cast<__bf16>(rest - static_cast<float>(r.p[1][i]));
  }
  return r;
}

// hi += hh, lo += the five smaller part products, in an order that kSwap turns
// with the operands' sides.
template <bool kSwap = false>
__device__ __forceinline__ void Mfma3(const Parts& a, const Parts& b, v16f& hi, v16f& lo) {
  constexpr int kA = kSwap ? 2 : 0;
  lo = Mfma(a.p[kA], b.p[2 - kA], lo);
  lo = Mfma(a.p[2 - kA], b.p[kA], lo);
  lo = Mfma(a.p[1], b.p[1], lo);
  lo = Mfma(a.p[kA / 2], b.p[1 - kA / 2], lo);
  lo = Mfma(a.p[1 - kA / 2], b.p[kA / 2], lo);
  hi = Mfma(a.p[0], b.p[0], hi);
}

// One staged 64-row block: its floats in flight, then its three tiles.
struct Tile3 {
  uint8_t part[3][kTile];
};
struct Block3 {
  float4 r[4];  // two chunks of eight dims: rows tid / 8 and 32 + tid / 8, chunk tid % 8

  __device__ __forceinline__ void Load(const float* __restrict__ base, size_t ld, int row0, int S) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int row = row0 + e * 32 + static_cast<int>(threadIdx.x) / 8;
      const float* p = base + static_cast<size_t>(min(row, S - 1)) * ld + threadIdx.x % 8 * 8;
      r[2 * e] = *reinterpret_cast<const float4*>(p);
      r[2 * e + 1] = *reinterpret_cast<const float4*>(p + 4);
    }
  }
  // Rows past the sequence are left as its last row: their scores are masked.
  __device__ __forceinline__ void Store(Tile3& t) const {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int row = e * 32 + threadIdx.x / 8, ch = threadIdx.x % 8;
      const float x[8] = {r[2 * e].x,     r[2 * e].y,     r[2 * e].z,     r[2 * e].w,
                          r[2 * e + 1].x, r[2 * e + 1].y, r[2 * e + 1].z, r[2 * e + 1].w};
      const Parts s = Split(x);
      const int at = ch / 4 * kHalf + row * 64 + Phys(row, ch % 4) * 16;
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(t.part[p] + at) = s.p[p];
    }
  }
};

// This lane's fragments of one own row: dims 16 s + 8 g .. + 8, s < 4.
__device__ __forceinline__ void OwnParts(const float* __restrict__ row, int lane, Parts (&f)[4]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const float* p = row + 16 * s + 8 * (lane / 32);
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    f[s] = Split(x);
  }
}
__device__ __forceinline__ Parts RowParts(const Tile3& t, const FragOffsets& fo, int row0, int s) {
  return Parts{{RowFrag(t.part[0], fo, row0, s), RowFrag(t.part[1], fo, row0, s),
                RowFrag(t.part[2], fo, row0, s)}};
}
__device__ __forceinline__ Parts ColParts(const Tile3& t, const FragOffsets& fo, int dt, int k0) {
  return Parts{{ColFrag(t.part[0], fo, dt, k0), ColFrag(t.part[1], fo, dt, k0),
                ColFrag(t.part[2], fo, dt, k0)}};
}
// Staged rows row0 .. + 32 against the own rows, over the 64 dims: lane (g, c)
// gets rows 8q + 4g + e against own row c.  kOwnKeys: the own rows are keys or
// values (dK / dV), else the staged ones are; either way a query's and a key's
// dot has the same bits, so dP - delta is 0 for a query that sees one key.
template <bool kOwnKeys = false>
__device__ __forceinline__ v16f Dot3(const Tile3& t, const FragOffsets& fo, int row0,
                                     const Parts (&own)[4]) {
  v16f hi = {}, lo = {};
#pragma unroll
  for (int s = 0; s < 4; ++s) Mfma3<kOwnKeys>(RowParts(t, fo, row0, s), own[s], hi, lo);
  return hi + lo;
}
// acc[dt] += (the tile's columns 32 dt ..)^T over rows row0 .. + 32 times w,
// the rows' values in score order.
__device__ __forceinline__ void Accum3(const Tile3& t, const FragOffsets& fo, int row0,
                                       const float (&w)[16], v16f (&acc)[2]) {
  Parts b[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float x[8] = {w[8 * h],     w[8 * h + 1], w[8 * h + 2], w[8 * h + 3],
                        w[8 * h + 4], w[8 * h + 5], w[8 * h + 6], w[8 * h + 7]};
    b[h] = Split(x);
  }
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) {
    v16f lo = {};
#pragma unroll
    for (int h = 0; h < 2; ++h) Mfma3(ColParts(t, fo, dt, row0 + 16 * h), b[h], acc[dt], lo);
    acc[dt] += lo;
  }
}

// exp(y) for y <= 0 as 2^n 2^f, n the integer nearest to y log2(e) and f the
// rest of it in two fused steps, so that it errs like expf (y = -75 .. 0: 3.5e-8
// of itself in the mean square); 2^t of t = y log2(e) rounded errs by |y| 2^-24.
// n is held at -200: -inf and all that is far below f32 give 0; NaN stays.  us,
// forward / dQ / dK and dV at B8 H12 S1024: 107 / 231 / 243 here, 114 / 242 / 258
// with expf and its range checks, 98 / 221 / 232 with 2^t.
__device__ __forceinline__ float ExpOf(float y) {
  const float n = fmaxf(__builtin_rintf(y * kLog2e), -200.0f);
  const float f = __builtin_fmaf(y, kLog2eLo, __builtin_fmaf(y, kLog2e, -n));
  return __builtin_amdgcn_ldexpf(Exp2(f), static_cast<int>(n));
}

// In pairs: the sums of weights have few roundings, so that p's add up to 1 as
// closely as they can (what is left over scales a component that all keys share).
__device__ __forceinline__ float Sum16(const float (&x)[16]) {
  float s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = x[2 * i] + x[2 * i + 1];
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

__device__ __forceinline__ void StoreRow(float* row, int g, const v16f (&acc)[2], float scale) {
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<float4*>(row + 32 * dt + 8 * q + 4 * g) =
          make_float4(acc[dt][4 * q] * scale, acc[dt][4 * q + 1] * scale,
                      acc[dt][4 * q + 2] * scale, acc[dt][4 * q + 3] * scale);
}

// The key range of a workgroup's queries: from the earliest start to the last
// query, in blocks.
__device__ __forceinline__ void KeyBlocks(int start, int i0, int S, int& first, int& count) {
  __shared__ int lo[kWaves];
  const int l = WaveMinI(start);
  if (threadIdx.x % kWave == 0) lo[threadIdx.x / kWave] = l;
  __syncthreads();
  first = min(min(lo[0], lo[1]), min(lo[2], lo[3])) / kBlkRows;
  count = min(i0 + kRowsWG - 1, S - 1) / kBlkRows - first + 1;
}

// ---------------------------------------------------------------------------
// The same rows in plain f32, a multiply-add at a time, each over the rows it
// sees and no other: for the waves whose sums came out NaN.  Two lanes a row
// (lane % 32), 32 of the 64 dims each; slow and rare.
// ---------------------------------------------------------------------------
struct Half {  // a lane's 32 dims of a row, StoreRow's
  v16f x[2] = {};
  Half() = default;
  __device__ __forceinline__ Half(const float* row, int g) {
#pragma unroll
    for (int e = 0; e < 32; e += 4) {
      const float4 v = *reinterpret_cast<const float4*>(row + 2 * e + 4 * g);
      x[e / 16][e % 16] = v.x, x[e / 16][e % 16 + 1] = v.y;
      x[e / 16][e % 16 + 2] = v.z, x[e / 16][e % 16 + 3] = v.w;
    }
  }
  // this += w r
  __device__ __forceinline__ void Add(float w, const Half& r) {
#pragma unroll
    for (int e = 0; e < 32; ++e)
      x[e / 16][e % 16] = __builtin_fmaf(w, r.x[e / 16][e % 16], x[e / 16][e % 16]);
  }
};
// The rows' dot over both lanes, the same in both.
__device__ __forceinline__ float Dot(const Half& a, const Half& b) {
  float s = 0.0f;
#pragma unroll
  for (int e = 0; e < 32; ++e) s = __builtin_fmaf(a.x[e / 16][e % 16], b.x[e / 16][e % 16], s);
  return SwapSum(s);
}

// Whether any of the wave's sums is NaN (wave-uniform).
__device__ __forceinline__ bool AnyNaN(const v16f (&acc)[2], bool nan = false) {
#pragma unroll
  for (int r = 0; r < 16; ++r) nan |= __builtin_isunordered(acc[0][r], acc[1][r]);
  return __ballot(nan) != 0;
}

// Query i's keys start .. i; every lane walks the wave's range first .. last.
__device__ __forceinline__ void PlainFwd(const float* q_row, const float* k, const float* v,
                                         size_t ld, int i, int start, int first, int last, int g,
                                         Half& acc, float& m, float& l) {
  const Half q(q_row, g);
  m = -INFINITY, l = 0.0f;
#pragma unroll 1
  for (int j = first; j <= last; ++j) {
    const float s = Dot(Half(k + static_cast<size_t>(j) * ld, g), q) * kIsd;
    if (j < start || j > i) continue;
    const float mn = fmaxf(m, s), alpha = m == -INFINITY ? 0.0f : expf(m - mn);
    const float p = s == -INFINITY ? 0.0f : expf(s - mn);
    l = l * alpha + p;
    m = mn;
    acc.x[0] *= alpha;
    acc.x[1] *= alpha;
    acc.Add(p, Half(v + static_cast<size_t>(j) * ld, g));
  }
}

__device__ __forceinline__ void PlainDQ(const float* q_row, const float* d_row, const float* k,
                                        const float* v, size_t ld, float m, float inv, int i,
                                        int start, int first, int last, int g, Half& acc,
                                        float& delta) {
  const Half q(q_row, g), d(d_row, g);
  double sum = 0.0;
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    delta = static_cast<float>(sum);
#pragma unroll 1
    for (int j = first; j <= last; ++j) {
      const Half kj(k + static_cast<size_t>(j) * ld, g);
      const float s = Dot(kj, q), dp = Dot(Half(v + static_cast<size_t>(j) * ld, g), d);
      if (j < start || j > i) continue;
      const float p = expf(s * kIsd - m) * inv;
      if (pass == 0)
        sum += static_cast<double>(dp) * p;
      else
        acc.Add((p * (dp - delta)) * kIsd, kj);
    }
  }
}

// Key j's queries first .. S - 1 that see it.
template <bool kDK, bool kDV>
__device__ __forceinline__ void PlainDKDV(const float* k_row, const float* v_row, const float* q,
                                          const float* dout, size_t ld, const float4* st, int j,
                                          int first, int S, int g, Half& dk, Half& dv) {
  const Half k(k_row, g), v(kDK ? v_row : k_row, g);
#pragma unroll 1
  for (int i = first; i < S; ++i) {
    const float4 t = st[i];
    const Half qi(q + static_cast<size_t>(i) * ld, g), di(dout + static_cast<size_t>(i) * ld, g);
    const float s = Dot(qi, k), dp = kDK ? Dot(di, v) : 0.0f;
    if (j > i || j < StartOf(t.w, i)) continue;
    const float p = expf(s * kIsd - t.x) * t.y;
    if (kDV) dv.Add(p, di);
    if (kDK) dk.Add((p * (dp - t.z)) * kIsd, qi);
  }
}

// ---------------------------------------------------------------------------
// Forward (attention.cc:448-493): online softmax over 64-key blocks; the stats
// row gets the row max, 1/l, 0 and the clamped start.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kThreads, 2)
Attn3Fwd(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
         float* __restrict__ o, float* __restrict__ stats, int S, int H,
         const int32_t* __restrict__ starts) {
  __shared__ __attribute__((aligned(1024))) Tile3 kt, vt;
  const int lane = threadIdx.x % kWave, g = lane / 32;
  const int wave = Uniform(threadIdx.x / kWave);
  const int nb = (S + kRowsWG - 1) / kRowsWG;
  int bh, rank;
  UnitOf3(nb, bh, rank);
  const int b = bh / H, h = bh % H;
  const size_t ld = static_cast<size_t>(H) * kD;
  const size_t base = static_cast<size_t>(b) * S * ld + static_cast<size_t>(h) * kD;
  const int i0 = (nb - 1 - rank) * kRowsWG, iw = i0 + wave * 32, i = iw + lane % 32;
  const int ic = min(i, S - 1);
  int start = 0;
  if (starts) {
    const int s0 = starts[static_cast<size_t>(b) * S + ic];
    start = s0 <= 0 ? 0 : (s0 < ic ? s0 : ic);
  }
  int jb0, nblk;
  KeyBlocks(start, i0, S, jb0, nblk);
  const int wave_last = min(iw + 31, S - 1), wave_start = WaveMaxI(start);
  Parts qf[4];
  OwnParts(q + base + static_cast<size_t>(ic) * ld, lane, qf);

  const FragOffsets fo = MakeFragOffsets(lane);
  v16f acc[2] = {};
  float m = -INFINITY, l = 0.0f;  // l: this half's share
  Block3 nk, nv;
  nk.Load(k + base, ld, jb0 * kBlkRows, S);
  nv.Load(v + base, ld, jb0 * kBlkRows, S);
  for (int n = 0; n < nblk; ++n) {
    const int j0 = (jb0 + n) * kBlkRows;
    if (n > 0) __syncthreads();  // the last block's reads are done
    nk.Store(kt);
    nv.Store(vt);
    __syncthreads();
    if (n + 1 < nblk) {
      nk.Load(k + base, ld, j0 + kBlkRows, S);
      nv.Load(v + base, ld, j0 + kBlkRows, S);
    }
    if (j0 > wave_last) continue;
    float p[2][16];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int jt = j0 + 32 * t;
      if (jt > wave_last) {  // wave-uniform: wholly above the diagonal
#pragma unroll
        for (int r = 0; r < 16; ++r) p[t][r] = -INFINITY;
        continue;
      }
      const v16f sc = Dot3(kt, fo, 32 * t, qf);
#pragma unroll
      for (int r = 0; r < 16; ++r) p[t][r] = sc[r] * kIsd;
      if (!(jt + 31 <= iw && jt >= wave_start && iw + 31 < S)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = jt + RowConst(r) + 4 * g;
          p[t][r] = j <= i && j >= start && i < S ? p[t][r] : -INFINITY;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, p[t][r]);
    }
    const float mn = fmaxf(m, SwapMax(mx));
    const float ref = mn == -INFINITY ? 0.0f : mn;
    const float alpha = m == -INFINITY ? 0.0f : ExpOf(m - ref);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) p[t][r] = ExpOf(p[t][r] - ref);
    l = l * alpha + (Sum16(p[0]) + Sum16(p[1]));
    m = mn;
    acc[0] *= alpha;
    acc[1] *= alpha;
#pragma unroll
    for (int t = 0; t < 2; ++t)
      if (j0 + 32 * t <= wave_last) Accum3(vt, fo, 32 * t, p[t], acc);
  }
  l = SwapSum(l);
  const size_t at = base + static_cast<size_t>(ic) * ld;
  const auto store = [&](const v16f (&row)[2], float row_m, float row_l) {
    if (i >= S) return;
    const float inv = 1.0f / row_l;
    StoreRow(o + at, g, row, inv);
    if (g == 0)
      *reinterpret_cast<float4*>(stats + (static_cast<size_t>(bh) * S + i) * 4) =
          make_float4(row_m, inv, 0.0f, static_cast<float>(start));
  };
  const bool plain = AnyNaN(acc, l != l);
  store(acc, m, l);
  if (plain) {  // over the same addresses, lane by lane
    Half row;
    float row_m, row_l;
    PlainFwd(q + at, k + base, v + base, ld, ic, start, WaveMinI(start), wave_last, g, row, row_m,
             row_l);
    store(row.x, row_m, row_l);
  }
}

// ---------------------------------------------------------------------------
// dQ (attention.cc:495-535) in one walk over the keys: dS = p (dP - delta) is
// linear in delta, so dQ = (sum p (dP - ref) k - (delta - ref) sum p k) / sqrt(d)
// for any ref, with delta = sum p dP (in double) from the same walk -- four
// products and one exponential a score where a walk for delta and one for dQ
// take five and two (395 us at B8 H12 S1024, two walks, 224 us here).  ref is
// the mean of the dP met so far, weighted as delta weights them, and the sums
// move with it, so what they hold is as small as dP - delta even where all keys
// or values share a component (emulated, ref = 0 errs up to seven times as far as
// two walks there, the first block's mean up to six, the running mean as far).
// A query that sees one key has ref = delta = dP and dQ exactly 0.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kThreads, 1)
Attn3DQ(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
        const float* __restrict__ dout, float* __restrict__ stats, float* __restrict__ dq, int S,
        int H) {
  __shared__ __attribute__((aligned(1024))) Tile3 kt, vt;
  const int lane = threadIdx.x % kWave, g = lane / 32;
  const int wave = Uniform(threadIdx.x / kWave);
  const int nb = (S + kRowsWG - 1) / kRowsWG;
  int bh, rank;
  UnitOf3(nb, bh, rank);
  const int b = bh / H, h = bh % H;
  const size_t ld = static_cast<size_t>(H) * kD;
  const size_t base = static_cast<size_t>(b) * S * ld + static_cast<size_t>(h) * kD;
  const int i0 = (nb - 1 - rank) * kRowsWG, iw = i0 + wave * 32, i = iw + lane % 32;
  const int ic = min(i, S - 1);
  const float4 st = *reinterpret_cast<const float4*>(stats + (static_cast<size_t>(bh) * S + ic) * 4);
  const int start = StartOf(st.w, ic);
  int jb0, nblk;
  KeyBlocks(start, i0, S, jb0, nblk);
  const int wave_last = min(iw + 31, S - 1), wave_start = WaveMaxI(start);
  Parts qf[4], df[4];
  OwnParts(q + base + static_cast<size_t>(ic) * ld, lane, qf);
  OwnParts(dout + base + static_cast<size_t>(ic) * ld, lane, df);

  const FragOffsets fo = MakeFragOffsets(lane);
  v16f acc_d[2] = {}, acc_p[2] = {};  // sums of p (dP - ref) k and of p k
  double dsum = 0.0;                  // this half's sum of p dP
  float psum = 0.0f, ref = 0.0f;
  Block3 nk, nv;
  nk.Load(k + base, ld, jb0 * kBlkRows, S);
  nv.Load(v + base, ld, jb0 * kBlkRows, S);
  for (int n = 0; n < nblk; ++n) {
    const int j0 = (jb0 + n) * kBlkRows;
    if (n > 0) __syncthreads();
    nk.Store(kt);
    nv.Store(vt);
    __syncthreads();
    if (n + 1 < nblk) {
      nk.Load(k + base, ld, j0 + kBlkRows, S);
      nv.Load(v + base, ld, j0 + kBlkRows, S);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int jt = j0 + 32 * t;
      if (jt > wave_last) continue;  // wave-uniform
      const v16f sc = Dot3(kt, fo, 32 * t, qf), dp = Dot3(vt, fo, 32 * t, df);
      float p[16], w[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] = ExpOf(sc[r] * kIsd - st.x) * st.y;
      if (!(jt + 31 <= iw && jt >= wave_start && iw + 31 < S)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = jt + RowConst(r) + 4 * g;
          p[r] = j <= i && j >= start && i < S ? p[r] : 0.0f;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) dsum += static_cast<double>(dp[r]) * p[r];
      psum += Sum16(p);
      // The weighted mean of the keys' dP so far; what is summed moves to it.
      const float weight = SwapSum(psum), sum = SwapSum(static_cast<float>(dsum));
      const float mean = weight > 0.0f ? sum / weight : ref;
      const float move = mean - ref;
      ref = mean;
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) acc_d[dt] -= move * acc_p[dt];
#pragma unroll
      for (int r = 0; r < 16; ++r) w[r] = p[r] * (dp[r] - ref);
      Accum3(kt, fo, 32 * t, w, acc_d);
      Accum3(kt, fo, 32 * t, p, acc_p);
    }
  }
  dsum += __shfl_xor(dsum, 32, kWave);
  float delta = static_cast<float>(dsum);
  const float rest = static_cast<float>(dsum - static_cast<double>(ref));
  v16f acc[2];
#pragma unroll
  for (int dt = 0; dt < 2; ++dt) acc[dt] = (acc_d[dt] - rest * acc_p[dt]) * kIsd;
  const size_t at = base + static_cast<size_t>(ic) * ld;
  const auto store = [&](const v16f (&row)[2], float row_delta) {
    if (i >= S) return;
    StoreRow(dq + at, g, row, 1.0f);
    if (g == 0) stats[(static_cast<size_t>(bh) * S + i) * 4 + 2] = row_delta;
  };
  const bool plain = AnyNaN(acc, delta != delta);
  store(acc, delta);
  if (plain) {
    Half row;
    PlainDQ(q + at, dout + at, k + base, v + base, ld, st.x, st.y, ic, start, WaveMinI(start),
            wave_last, g, row, delta);
    store(row.x, delta);
  }
}

// ---------------------------------------------------------------------------
// dK and dV (attention.cc:537-590): each wave's 32 keys against 64-query
// blocks from the diagonal down.  kDK / kDV pick the outputs; each output's
// arithmetic is the same whichever else is formed.
// ---------------------------------------------------------------------------
template <bool kDK, bool kDV>
__global__ void __launch_bounds__(kThreads, kDK ? 1 : 2)
Attn3DKDV(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
          const float* __restrict__ dout, const float* __restrict__ stats, float* __restrict__ dk,
          float* __restrict__ dv, int S, int H) {
  __shared__ __attribute__((aligned(1024))) Tile3 qt, dt;
  // Per staged query: m, 1/l, delta, and its first key.
  __shared__ __attribute__((aligned(16))) float sm[kBlkRows], si[kBlkRows], sd[kBlkRows];
  __shared__ __attribute__((aligned(16))) int ss[kBlkRows];
  __shared__ int smax;
  __shared__ LiveBlocks live;
  const int lane = threadIdx.x % kWave, g = lane / 32;
  const int wave = Uniform(threadIdx.x / kWave);
  const int nb = (S + kRowsWG - 1) / kRowsWG;
  int bh, rank;
  UnitOf3(nb, bh, rank);  // rank 0: the first keys, the longest columns
  const int b = bh / H, h = bh % H;
  const size_t ld = static_cast<size_t>(H) * kD;
  const size_t base = static_cast<size_t>(b) * S * ld + static_cast<size_t>(h) * kD;
  const int jw = rank * kRowsWG + wave * 32, j = jw + lane % 32, jc = min(j, S - 1);
  const float4* st = reinterpret_cast<const float4*>(stats) + static_cast<size_t>(bh) * S;
  const int qb0 = rank * kRowsWG / kBlkRows;
  int nblk = (S - 1) / kBlkRows - qb0 + 1;
  const int nlive = ListLiveBlocks<kThreads>(live, S, qb0, nblk, rank * kRowsWG + kRowsWG - 1,
                                             [&](int row) { return StartOf(st[row].w, row); });
  if (nlive >= 0) nblk = nlive;
  const auto block = [&](int n) { return qb0 + (nlive >= 0 ? Uniform(live.idx[n]) : n); };

  Parts kf[4], vf[kDK ? 4 : 1];
  OwnParts(k + base + static_cast<size_t>(jc) * ld, lane, kf);
  if constexpr (kDK) OwnParts(v + base + static_cast<size_t>(jc) * ld, lane, vf);
  const FragOffsets fo = MakeFragOffsets(lane);
  v16f acc_k[2] = {}, acc_v[2] = {};
  Block3 nq, nd;
  float4 ns = make_float4(0.f, 0.f, 0.f, 0.f);
  auto load = [&](int qb) {
    nq.Load(q + base, ld, qb * kBlkRows, S);
    nd.Load(dout + base, ld, qb * kBlkRows, S);
    if (threadIdx.x < kBlkRows) ns = st[min(qb * kBlkRows + static_cast<int>(threadIdx.x), S - 1)];
  };
  const auto rows = [&](const auto* terms, int t, int r) { return terms[32 * t + RowConst(r) + 4 * g]; };
  load(block(0));
  for (int n = 0; n < nblk; ++n) {
    const int i0 = block(n) * kBlkRows;
    if (n > 0) __syncthreads();
    nq.Store(qt);
    nd.Store(dt);
    if (wave == 0) {
      const int start = StartOf(ns.w, min(i0 + lane, S - 1));
      sm[lane] = ns.x, si[lane] = ns.y, sd[lane] = ns.z, ss[lane] = start;
      const int mx = WaveMaxI(start);
      if (lane == 0) smax = mx;
    }
    __syncthreads();
    if (n + 1 < nblk) load(block(n + 1));
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int it = i0 + 32 * t;
      if (it >= S || it + 31 < jw) continue;  // wave-uniform: no query sees a key
      const v16f sc = Dot3<true>(qt, fo, 32 * t, kf);
      float p[16];
#pragma unroll
      for (int r = 0; r < 16; ++r)
        p[r] = ExpOf(sc[r] * kIsd - rows(sm, t, r)) * rows(si, t, r);
      if (!(it >= jw + 31 && it + 31 < S && Uniform(smax) <= jw)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = it + RowConst(r) + 4 * g;
          p[r] = i < S && j <= i && j >= rows(ss, t, r) ? p[r] : 0.0f;
        }
      }
      if constexpr (kDV) Accum3(dt, fo, 32 * t, p, acc_v);
      if constexpr (kDK) {
        const v16f dp = Dot3<true>(dt, fo, 32 * t, vf);
        float w[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
          w[r] = (p[r] * (dp[r] - rows(sd, t, r))) * kIsd;
        Accum3(qt, fo, 32 * t, w, acc_k);
      }
    }
  }
  const size_t at = base + static_cast<size_t>(jc) * ld;
  const bool plain_k = kDK && AnyNaN(acc_k), plain_v = kDV && AnyNaN(acc_v);
  if (j < S) {
    if constexpr (kDK) StoreRow(dk + at, g, acc_k, 1.0f);
    if constexpr (kDV) StoreRow(dv + at, g, acc_v, 1.0f);
  }
  if (plain_k || plain_v) {
    Half row_k, row_v;
    PlainDKDV<kDK, kDV>(k + at, v + (kDK ? at : 0), q + base, dout + base, ld, st, jc, jw, S, g,
                        row_k, row_v);
    if (plain_k && j < S) StoreRow(dk + at, g, row_k.x, 1.0f);
    if (plain_v && j < S) StoreRow(dv + at, g, row_v.x, 1.0f);
  }
}

dim3 GridOf(size_t B, size_t S, size_t H) {
  return dim3(static_cast<unsigned>((S + kRowsWG - 1) / kRowsWG * B * H));
}

}  // namespace

hipError_t LaunchAttn3Fwd(const float* q, const float* k, const float* v, float* o, float* stats,
                          size_t B, size_t S, size_t H, const int32_t* starts, hipStream_t s) {
  hipLaunchKernelGGL(Attn3Fwd, GridOf(B, S, H), dim3(kThreads), 0, s, q, k, v, o, stats,
                     static_cast<int>(S), static_cast<int>(H), starts);
  return hipGetLastError();
}

hipError_t LaunchAttn3DQ(const float* q, const float* k, const float* v, const float* dout,
                         float* stats, float* dq, size_t B, size_t S, size_t H, hipStream_t s) {
  hipLaunchKernelGGL(Attn3DQ, GridOf(B, S, H), dim3(kThreads), 0, s, q, k, v, dout, stats, dq,
                     static_cast<int>(S), static_cast<int>(H));
  return hipGetLastError();
}

hipError_t LaunchAttn3DKDV(const float* q, const float* k, const float* v, const float* dout,
                           const float* stats, float* dk, float* dv, size_t B, size_t S, size_t H,
                           hipStream_t s) {
  const int Si = static_cast<int>(S), Hi = static_cast<int>(H);
#define SEEAI_DKDV(K, V)                                                                         \
  hipLaunchKernelGGL((Attn3DKDV<K, V>), GridOf(B, S, H), dim3(kThreads), 0, s, q, k, v, dout, stats, \
                     dk, dv, Si, Hi)
  if (dk && dv) SEEAI_DKDV(true, true);
  else if (dk) SEEAI_DKDV(true, false);
  else SEEAI_DKDV(false, true);
#undef SEEAI_DKDV
  return hipGetLastError();
}

}  // namespace seeai
