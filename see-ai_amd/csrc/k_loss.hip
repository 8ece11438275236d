// k_loss.hip -- softmax cross-entropy forward / backward (and the masked
// pair) on gfx950 (runtime/executor/loss.cc:21-126).
//
// Forward: rows of up to 32768 columns in one pass with the row in registers
// (XEntRowKernel), longer ones in three (the row max, the exp-sum, the
// probabilities); either way the exp-sum has the reference's own association,
// a serial f32 chain per row -- at a 32k vocabulary a tree sum differs from it
// by more than the 1e-5 parity bar -- and each row leaves its -log p[label] as
// a double, which a one-workgroup kernel sums in a fixed tree into the f32
// mean: deterministic, no float atomics.
// Backward: scale = seed / N (or / T) divided on the device exactly as the
// reference divides it, then one coalesced pass.
#include "common.h"

namespace seeai {
namespace {

// --- long rows, pass 1: row max (order-free: fmax ignores NaN as std::fmax does) ------
constexpr int kMaxThreads = 256;

// Rows of 16-byte multiples move as float4 with two running maxima per lane.
__host__ __device__ __forceinline__ bool Vec4Rows(const void* p, size_t C) {
  return C % 4 == 0 && (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

__global__ void __launch_bounds__(kMaxThreads)
XEntRowMaxKernel(const float* __restrict__ logits, float* __restrict__ row_max, size_t C) {
  __shared__ float red[kMaxThreads / kWave];
  const float* x = logits + static_cast<size_t>(blockIdx.x) * C;
  float mx = NAN, mx2 = NAN;  // the identity of fmax
  if (Vec4Rows(logits, C)) {
    // Four 16-byte loads in flight per lane (a 32k-column row is 31 per
    // lane), each into its own running maximum.
    const float4* x4 = reinterpret_cast<const float4*>(x);
    const size_t n4 = C / 4;
    float m4[4] = {NAN, NAN, NAN, NAN};
    size_t c = threadIdx.x;
    for (; c + 3 * kMaxThreads < n4; c += 4 * kMaxThreads) {
      float4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = x4[c + u * kMaxThreads];
#pragma unroll
      for (int u = 0; u < 4; ++u) m4[u] = fmaxf(m4[u], fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w)));
    }
    for (; c < n4; c += kMaxThreads) {
      const float4 v = x4[c];
      mx = fmaxf(mx, fmaxf(v.x, v.y));
      mx2 = fmaxf(mx2, fmaxf(v.z, v.w));
    }
    mx = fmaxf(mx, fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3])));
  } else {
    for (size_t c = threadIdx.x; c < C; c += kMaxThreads) mx = fmaxf(mx, x[c]);
  }
  mx = BlockMaxF<kMaxThreads>(fmaxf(mx, mx2), red);
  if (threadIdx.x == 0) row_max[blockIdx.x] = mx;
}

// The row max from the partial maxima the producing GEMM's epilogue left
// ([rows, parts], fmax over each group of 64 columns): fmax is exact and
// order-free, so this is pass 1's value without a pass over the logits.
__global__ void __launch_bounds__(kMaxThreads)
XEntRowMaxPartsKernel(const float* __restrict__ parts, size_t P, float* __restrict__ row_max) {
  __shared__ float red[kMaxThreads / kWave];
  const float* p = parts + static_cast<size_t>(blockIdx.x) * P;
  float mx = NAN;
  for (size_t c = threadIdx.x; c < P; c += kMaxThreads) mx = fmaxf(mx, p[c]);
  mx = BlockMaxF<kMaxThreads>(mx, red);
  if (threadIdx.x == 0) row_max[blockIdx.x] = mx;
}

// --- long rows, pass 2: the exp-sum in the reference's order ------------------------------
// loss.cc:24-29 sums exp(x - max) in f32, column by column, one chain per
// row.  That association is reproduced exactly, with the chain apart from
// the exps: a workgroup takes 32 rows; waves 1-7 evaluate exp over 32-row x
// 224-column tiles into LDS (16-byte loads, double-buffered) while lane r
// of wave 0 adds row r's previous tile in column order, sixteen LDS values
// read ahead of its adds.  The chain wave does nothing else, so a tile
// costs the longer of its 224 dependent adds and the producers' exps.

// The exps that feed the long rows' chain: 2^(x log2 e) on the hardware's exp2
// (two instructions where the libm expf takes about fifteen; 4096 x 40000 641
// us against 732).  The rounding of x log2 e moves a term by at most |x| 1e-7
// of itself (below 2e-6 down to x = -30, where a term is 1e-13 of the row's
// largest one), so the chain's sum stays within 1e-6 of expf's.
__device__ __forceinline__ float SumExp(float x) {
  return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}

// --- the exp-sum chain in parallel ------------------------------------------------
//
// A serial f32 sum of nonnegative terms, bit for bit, without walking it term
// by term.  While the running sum S stays in one binade [2^k, 2^(k+1)) every
// addition rounds to the grid u = 2^(k-23), of which S is a multiple: the sum
// moves by the term rounded to that grid, whatever S is -- unless the term
// lies halfway between two grid points, where S's parity decides.  Grid
// multiples below 2^(k+1) add exactly in any order, so a run of terms without
// a tie or a crossing adds its rounded terms as a tree; a tie or the term that
// leaves the binade is added by itself.

// The biased exponent of a nonnegative float.
__device__ __forceinline__ int ExponentOf(float s) {
  return static_cast<int>(__float_as_uint(s) >> 23);
}

template <int kCtrl, int kRows>
__device__ __forceinline__ float DppAdd(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, kRows, 0xf, false));
}
// Inclusive sum over the wave's lanes in order.
__device__ __forceinline__ float WaveScan(float v) {
  v = DppAdd<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8 within rows of 16
  v = DppAdd<0x112, 0xf>(v);
  v = DppAdd<0x114, 0xf>(v);
  v = DppAdd<0x118, 0xf>(v);
  v = DppAdd<0x142, 0xa>(v);  // lane 15 of a row to the next row
  return DppAdd<0x143, 0xc>(v);  // lane 31 to the upper half
}
// The lane before's value, 0 in lane 0 (wave_shr 1).
__device__ __forceinline__ float WaveShift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float ReadLane(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Each of n = 1 .. 16 (a power of two) values summed over the wave: lane l
// gets the sum of value SumIndex<n>(l), the wave halving the values it still
// carries at each exchange.
template <int n, int bit = kWave / 2>
__device__ __forceinline__ float WaveSums(const float (&in)[n], int lane) {
  if constexpr (n > 1) {
    float out[n / 2];
    const bool up = lane & bit;
#pragma unroll
    for (int i = 0; i < n / 2; ++i) {
      const float keep = up ? in[n / 2 + i] : in[i], send = up ? in[i] : in[n / 2 + i];
      out[i] = keep + __shfl_xor(send, bit, kWave);
    }
    return WaveSums<n / 2, bit / 2>(out, lane);
  } else {
    float v = in[0];
#pragma unroll
    for (int x = bit; x > 0; x /= 2) v += __shfl_xor(v, x, kWave);
    return v;
  }
}
template <int n>
__device__ __forceinline__ int SumIndex(int lane) {
  return lane / (kWave / n);
}

constexpr int kSumThreads = 512;
constexpr int kSumRows = 32;
constexpr int kTileCols = 224;                      // 56 float4 per row
constexpr int kTileLd = kTileCols + 4;
constexpr int kProducers = kSumThreads - kWave;     // waves 1-7

__global__ void __launch_bounds__(kSumThreads)
XEntSerialSumKernel(const float* __restrict__ logits, const float* __restrict__ row_max,
                    float* __restrict__ row_sum, size_t N, size_t C) {
  __shared__ __attribute__((aligned(16))) float tile[2][kSumRows][kTileLd];
  const size_t r0 = static_cast<size_t>(blockIdx.x) * kSumRows;
  const int t = threadIdx.x;
  const size_t ntiles = (C + kTileCols - 1) / kTileCols;
  const bool vec = Vec4Rows(logits, C);
  // Producer p fills float4 slots p + 448 i (i < 4): row = slot / 56,
  // column quad = slot % 56 (consecutive lanes read consecutive quads); the
  // four loads are issued before any exp.
  constexpr int kSlots = kSumRows * (kTileCols / 4) / kProducers;
  static_assert(kSlots * kProducers == kSumRows * (kTileCols / 4), "whole slots per producer");
  auto fill = [&](size_t k, int buf) {
    const int p = t - kWave;
    float4 v[kSlots];
    float mx[kSlots];
    bool full[kSlots];
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int f = p + i * kProducers, r = f / (kTileCols / 4), c4 = f % (kTileCols / 4);
      const size_t row = r0 + r, c = k * kTileCols + 4 * c4;
      full[i] = vec && row < N && c + 4 <= C;
      mx[i] = row < N ? row_max[row] : 0.0f;
      v[i] = full[i] ? *reinterpret_cast<const float4*>(logits + row * C + c)
                     : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int f = p + i * kProducers, r = f / (kTileCols / 4), c4 = f % (kTileCols / 4);
      const size_t row = r0 + r, c = k * kTileCols + 4 * c4;
      float e[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (full[i]) {
        e[0] = SumExp(v[i].x - mx[i]), e[1] = SumExp(v[i].y - mx[i]);
        e[2] = SumExp(v[i].z - mx[i]), e[3] = SumExp(v[i].w - mx[i]);
      } else if (row < N) {
        for (int u = 0; u < 4; ++u)
          if (c + u < C) e[u] = SumExp(logits[row * C + c + u] - mx[i]);
      }
      *reinterpret_cast<float4*>(&tile[buf][r][4 * c4]) = make_float4(e[0], e[1], e[2], e[3]);
    }
  };
  if (t >= kWave) fill(0, 0);
  __syncthreads();
  float sum = 0.0f;
  for (size_t k = 0; k < ntiles; ++k) {
    if (t >= kWave) {
      if (k + 1 < ntiles) fill(k + 1, (k + 1) & 1);
    } else if (t < kSumRows) {
      const float* row = tile[k & 1][t];
      const size_t w = k + 1 < ntiles ? kTileCols : C - k * kTileCols;
      if (w == kTileCols) {
#pragma unroll 2
        for (int j0 = 0; j0 < kTileCols; j0 += 16) {
          float4 v[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const float4*>(row + j0 + 4 * q);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            sum += v[q].x;
            sum += v[q].y;
            sum += v[q].z;
            sum += v[q].w;
          }
        }
      } else {
        for (size_t j = 0; j < w; ++j) sum += row[j];
      }
    }
    __syncthreads();
  }
  if (t < kSumRows && r0 + t < N) row_sum[r0 + t] = sum;
}

// --- long rows, pass 3: probabilities and the label term ----------------------------------
constexpr int kProbThreads = 256;

// With kBwd (the backward fused behind the forward, every row 16-byte
// aligned): each probability also becomes its gradient, scale * p minus
// scale at the label (zero on a masked row) -- XEntBwdKernel's expression on
// the same f32 p -- stored with the sink; probs is stored only where given.
template <bool kBwd>
__global__ void __launch_bounds__(kProbThreads)
XEntProbsKernel(const float* __restrict__ logits, const int32_t* __restrict__ labels,
                const float* __restrict__ row_max, const float* __restrict__ row_sum,
                float* __restrict__ probs, double* __restrict__ row_loss, size_t C, int masked,
                const float* __restrict__ scale_p, float* __restrict__ dl, Bf16Sink sink) {
  const size_t r = blockIdx.x;
  const float* x = logits + r * C;
  float* p = probs + r * C;
  const float mx = row_max[r];
  const float inv_sum = 1.0f / row_sum[r];  // loss.cc:30
  if constexpr (kBwd) {
    const float scale = *scale_p;
    const int32_t lab = labels[r];
    const bool zero = masked && lab < 0;
    const size_t lc = static_cast<size_t>(lab);
    const float4* x4 = reinterpret_cast<const float4*>(x);
    float4* d4 = reinterpret_cast<float4*>(dl + r * C);
    for (size_t c = threadIdx.x; c < C / 4; c += kProbThreads) {
      const float4 v = x4[c];
      const float4 q = make_float4(expf(v.x - mx) * inv_sum, expf(v.y - mx) * inv_sum,
                                   expf(v.z - mx) * inv_sum, expf(v.w - mx) * inv_sum);
      if (probs) reinterpret_cast<float4*>(p)[c] = q;
      float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
      if (!zero) {
        g = make_float4(scale * q.x, scale * q.y, scale * q.z, scale * q.w);
        if (lc / 4 == c) {
          const size_t l = lc % 4;
          if (l == 0) g.x -= scale;
          else if (l == 1) g.y -= scale;
          else if (l == 2) g.z -= scale;
          else g.w -= scale;
        }
      }
      if (sink.store_f32) d4[c] = g;
      if (sink.out) SinkStore4(sink, r * C + 4 * c, g);
    }
  } else if (Vec4Rows(logits, C) && Vec4Rows(probs, C)) {
    const float4* x4 = reinterpret_cast<const float4*>(x);
    float4* p4 = reinterpret_cast<float4*>(p);
    for (size_t c = threadIdx.x; c < C / 4; c += kProbThreads) {
      const float4 v = x4[c];
      p4[c] = make_float4(expf(v.x - mx) * inv_sum, expf(v.y - mx) * inv_sum,
                          expf(v.z - mx) * inv_sum, expf(v.w - mx) * inv_sum);
    }
  } else {
    for (size_t c = threadIdx.x; c < C; c += kProbThreads) p[c] = expf(x[c] - mx) * inv_sum;
  }
  if (threadIdx.x == 0) {
    const int32_t lab = labels[r];
    double term = 0.0;
    if (!(masked && lab < 0)) {
      // The label's probability exactly as stored; NaN propagates, the
      // clamp only rescues underflow (loss.cc:45-51).
      const float pl = expf(x[static_cast<size_t>(lab)] - mx) * inv_sum;
      const double safe = pl != pl ? static_cast<double>(pl) : static_cast<double>(fmaxf(pl, 1e-12f));
      term = -log(safe);
    }
    row_loss[r] = term;
  }
}

// --- the whole row in registers -----------------------------------------------------
//
// A workgroup per row of up to kT * 4 * kV columns: one read of the logits
// serves the row max, the exp-sum chain, the probabilities and (kBwd, the
// backward fused behind the forward) the gradient, so the pass is bound by one
// read and the writes -- the three kernels above read the logits three times.
// Lane t holds float4 e T + t, e < kV, so (e, wave) is a segment of 256
// consecutive columns and segments in order are the row.  The chain:
//   1. every segment's plain sum, and their running sum P (one wave).  After n
//      terms the serial sum is within n 2^-24 of the exact one, and P, a tree,
//      within 20 2^-24; (n + 256) 2^-24 around P, n to the segment's end, bounds
//      the binades a segment runs through.
//   2. One binade and no tie: its terms rounded to that grid are summed.  Else
//      the terms go to an LDS slot, and with one or two binades the running
//      sums over the lanes on both grids and the lanes that hold a tie.
//   3. One wave walks the segments with a slot, ten or so a row; those between
//      two of them lie in one binade, so their rounded sums add in any order.
//      In a walked segment S moves by the running sum of its binade up to the
//      next lane that crosses or ties, and by that lane's four terms one by
//      one.  A segment of more binades (the row's first), or of many ties,
//      goes term by term.  Without a free slot a segment's terms are formed
//      from the logits again.
// The sum is bit for bit the serial one of the terms expf(x - max).
constexpr int kSegTerms = 4 * kWave;

struct RowSlot {
  float term[kSegTerms];
  float lower[kWave], upper[kWave];  // inclusive, over the lanes
  unsigned long long tie[2];         // the lanes with a tie, per grid
};

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // rows of any C: dword-aligned

template <int kT, int kV, bool kBwd, int kOcc>
__global__ void __launch_bounds__(kT, kOcc)
XEntRowKernel(const float* __restrict__ logits, const int32_t* __restrict__ labels,
              float* __restrict__ probs, double* __restrict__ row_loss, int C, int masked,
              const float* __restrict__ scale_p, float* __restrict__ dl, Bf16Sink sink) {
  constexpr int kWaves = kT / kWave, kSegs = kV * kWaves;
  static_assert(kSegs <= 2 * kWave, "two segments a lane in the walk");
  constexpr int kRowSlots = kSegs < 12 ? kSegs : 12;
  __shared__ float sred[kWaves];
  __shared__ float ssum[kSegs];     // 1: plain sums; 2: rounded sums
  __shared__ int sinfo[kSegs];      // 1: binade, kTwo + lower binade or kMany; 2: with the slot
  __shared__ __attribute__((aligned(16))) RowSlot slots[kRowSlots + 1];  // the last: no free slot
  __shared__ int nslots;
  __shared__ float sinv;
  // Per-segment codes: kOne + binade, kTwo + (lower) binade, kMany (binades
  // fit 8 bits, biased); step 2 adds the slot's index in the bits above 16 and
  // makes a kOne with a tie a kTwo.
  constexpr int kOne = 0, kTwo = 1 << 8, kMany = 2 << 8, kKind = 3 << 8;
  const int tid = threadIdx.x, lane = tid % kWave, wave = Uniform(tid / kWave);
  const size_t r = blockIdx.x;
  const float* x = logits + r * C;
  const float kNegInf = -INFINITY;

  // Four terms at lane offset 4 i of the columns from c0 (wave-uniform; c0 +
  // span is past the last lane's).
  const auto load = [&](int c0, int i, int span) {
    const float* p = x + c0;
    if (c0 + span <= C) return *reinterpret_cast<const f4u*>(p + 4 * i);
    const int left = C - c0 - 4 * i;
    if (left >= 4) return *reinterpret_cast<const f4u*>(p + 4 * i);
    return f4u{left > 0 ? p[4 * i] : kNegInf, left > 1 ? p[4 * i + 1] : kNegInf,
               left > 2 ? p[4 * i + 2] : kNegInf, kNegInf};
  };

  f4u v[kV];
  float mx = NAN;  // the identity of fmax
#pragma unroll
  for (int e = 0; e < kV; ++e) v[e] = load(e * 4 * kT, tid, 4 * kT);
#pragma unroll
  for (int e = 0; e < kV; ++e)
    mx = fmaxf(mx, fmaxf(fmaxf(v[e].x, v[e].y), fmaxf(v[e].z, v[e].w)));
  mx = WaveMaxF(mx);
  if (lane == 0) sred[wave] = mx;
  if (tid == 0) nslots = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, sred[w]);
  const auto terms = [&](int seg) {  // a segment's four terms of this lane
    const f4u t = load(seg * kSegTerms, lane, kSegTerms);
    return f4u{expf(t.x - mx), expf(t.y - mx), expf(t.z - mx), expf(t.w - mx)};
  };

  // The row's exps in its registers (columns past the row: exp(-inf) = 0).
  // 1. plain sums
  float part[kV];
#pragma unroll
  for (int e = 0; e < kV; ++e) {
    v[e] = f4u{expf(v[e].x - mx), expf(v[e].y - mx), expf(v[e].z - mx), expf(v[e].w - mx)};
    part[e] = (v[e].x + v[e].y) + (v[e].z + v[e].w);
    __builtin_amdgcn_sched_barrier(0);  // one float4's temporaries at a time
  }
  {
    const float t = WaveSums<kV>(part, lane);
    if (lane % (kWave / kV) == 0) ssum[SumIndex<kV>(lane) * kWaves + wave] = t;
  }
  __syncthreads();
  if (wave == 0) {
    const int s0 = 2 * lane;
    const float a0 = s0 < kSegs ? ssum[s0] : 0.0f, a1 = s0 + 1 < kSegs ? ssum[s0 + 1] : 0.0f;
    // The sum before each segment: the lanes' before, not this lane's less its
    // own, which would err by the size of what comes next.
    const float p0 = WaveShift(WaveScan(a0 + a1)), p1 = p0 + a0;
    const auto info = [&](int s, float p, float a) {
      const float margin = static_cast<float>(s + 2) * 0x1p-16f;
      const float lo = p * (1.0f - margin), hi = (p + a) * (1.0f + margin);
      const int k0 = ExponentOf(lo), k1 = ExponentOf(hi);
      return !(lo >= 0x1p-90f) || k1 > k0 + 1 ? kMany : (k1 == k0 ? kOne : kTwo) + k0;
    };
    if (s0 < kSegs) sinfo[s0] = info(s0, p0, a0);
    if (s0 + 1 < kSegs) sinfo[s0 + 1] = info(s0 + 1, p1, a1);
  }
  __syncthreads();
  // 2. rounded sums; the segments that need a slot get it from a loop of its
  // own, on terms formed from the logits again (one or two a wave: unrolled
  // over the registers its code would not fit the instruction cache).
  const auto grid = [](const f4u& t, uint32_t bits, bool& tie) {  // of binade 2^k, as bits
    const float b = __uint_as_float(bits), half = __uint_as_float(bits - (24u << 23));
    const float g0 = (t.x + b) - b, g1 = (t.y + b) - b, g2 = (t.z + b) - b, g3 = (t.w + b) - b;
    // No term is further than half a step from the grid: a tie is the largest.
    tie = fmaxf(fmaxf(fabsf(t.x - g0), fabsf(t.y - g1)), fmaxf(fabsf(t.z - g2), fabsf(t.w - g3))) ==
          half;
    return (g0 + g1) + (g2 + g3);
  };
  const int codes = lane < kV ? sinfo[lane * kWaves + wave] : 0;  // this wave's segments
  uint32_t slotted = 0;                                           // wave-uniform
#pragma unroll
  for (int e = 0; e < kV; ++e) {
    const int code = __builtin_amdgcn_readlane(codes, e);
    bool tie;
    const float sum = grid(v[e], static_cast<uint32_t>(code & 0xff) << 23, tie);
    const bool slot = static_cast<int>((code & kKind) != kOne) | static_cast<int>(__ballot(tie) != 0);
    slotted |= slot ? 1u << e : 0u;
    part[e] = slot ? 0.0f : sum;
    __builtin_amdgcn_sched_barrier(0);
  }
  {
    const float t = WaveSums<kV>(part, lane);
    if (lane % (kWave / kV) == 0) ssum[SumIndex<kV>(lane) * kWaves + wave] = t;
  }
  for (; slotted; slotted &= slotted - 1) {
    const int seg = (__ffs(slotted) - 1) * kWaves + wave;
    int code = __builtin_amdgcn_readlane(codes, __ffs(slotted) - 1), at = 0;
    if (lane == 0) at = min(atomicAdd(&nslots, 1), kRowSlots);
    at = Uniform(at);
    if (at < kRowSlots) {
      RowSlot& s = slots[at];
      const f4u t = terms(seg);
      *reinterpret_cast<float4*>(&s.term[4 * lane]) = make_float4(t.x, t.y, t.z, t.w);
      if ((code & kKind) != kMany) {
        const uint32_t bits = static_cast<uint32_t>(code & 0xff) << 23;
        bool tie, tie_up;
        s.lower[lane] = WaveScan(grid(t, bits, tie));
        s.upper[lane] = WaveScan(grid(t, bits + (1u << 23), tie_up));
        const unsigned long long tl = __ballot(tie), tu = __ballot(tie_up);
        if (lane == 0) s.tie[0] = tl, s.tie[1] = tu;
        code = (__popcll(tl | tu) > 12 ? kMany : kTwo) | (code & 0xff);
      }
    } else {
      code = kMany;
    }
    if (lane == 0) sinfo[seg] = code + (at << 16);
  }
  __syncthreads();
  // 3. the walk
  if (wave == 0) {
    __builtin_amdgcn_s_setprio(3);
    float S = 0.0f;
    for (int half = 0; half < (kSegs + kWave - 1) / kWave; ++half) {
      const int mine = half * kWave + lane;
      const float rs = mine < kSegs ? ssum[mine] : 0.0f;
      const int st = mine < kSegs ? sinfo[mine] : kOne;
      unsigned long long walk = __ballot((st & kKind) != kOne);
      int from = 0;
      while (true) {
        const int i = walk ? __ffsll(walk) - 1 : kWave;
        S += ReadLane(WaveScan(lane >= from && lane < i ? rs : 0.0f), kWave - 1);
        if (i == kWave) break;
        from = i + 1;
        walk &= walk - 1;
        const int code = __builtin_amdgcn_readlane(st, i);
        RowSlot& s = slots[code >> 16];
        if ((code & kKind) == kTwo) {
          const float lower = s.lower[lane], upper = s.upper[lane];
          const float4 t = *reinterpret_cast<const float4*>(&s.term[4 * lane]);
          const unsigned long long tie_lower = s.tie[0], tie_upper = s.tie[1];
          const float top = __uint_as_float(static_cast<uint32_t>((code & 0xff) + 1) << 23);
          for (int p = 0; p < kWave;) {  // lanes before p are added
            const bool low = !(S >= top);
            const float inc = low ? lower : upper;
            const float after = S + (inc - (p > 0 ? ReadLane(inc, p - 1) : 0.0f));
            const unsigned long long stop =
                (__ballot(low && after >= top) | (low ? tie_lower : tie_upper)) & (~0ull << p);
            const int f = stop ? __ffsll(stop) - 1 : kWave;
            if (f > p) S = ReadLane(after, f - 1);  // exact: below the crossing
            if (f < kWave) {
              S += ReadLane(t.x, f);
              S += ReadLane(t.y, f);
              S += ReadLane(t.z, f);
              S += ReadLane(t.w, f);
            }
            p = f + 1;
          }
        } else {
          if (code >> 16 == kRowSlots) {
            const f4u t = terms(half * kWave + i);
            *reinterpret_cast<float4*>(&s.term[4 * lane]) = make_float4(t.x, t.y, t.z, t.w);
          }
          const auto read = [&](int j, float4 (&t)[4]) {
#pragma unroll
            for (int q = 0; q < 4; ++q) t[q] = *reinterpret_cast<const float4*>(&s.term[j + 4 * q]);
          };
          float4 now[4], next[4];
          read(0, now);
          for (int j = 0; j < kSegTerms; j += 16) {  // the next terms' reads ahead of the adds
            read(min(j + 16, kSegTerms - 16), next);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              S += now[q].x;
              S += now[q].y;
              S += now[q].z;
              S += now[q].w;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) now[q] = next[q];
          }
        }
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if (lane == 0) sinv = 1.0f / S;  // loss.cc:30
  }
  __syncthreads();
  const float inv_sum = sinv;

  const int32_t lab = labels[r];
  const bool zero = masked && lab < 0;
  const size_t lc = static_cast<size_t>(lab);
  const float scale = kBwd ? *scale_p : 0.0f;
  float* const pr = probs + r * C;
#pragma unroll
  for (int e = 0; e < kV; ++e) {
    const int c0 = e * 4 * kT, left = C - c0 - 4 * tid;
    const f4u q = v[e] * inv_sum;
    if (c0 + 4 * kT <= C || left >= 4) {  // the first wave-uniform
      if (probs) *reinterpret_cast<f4u*>(pr + c0 + 4 * tid) = q;
      if constexpr (kBwd) {
        float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!zero) {
          g = make_float4(scale * q.x, scale * q.y, scale * q.z, scale * q.w);
          if (lc / 4 == static_cast<size_t>(c0 / 4 + tid)) {
            const size_t l = lc % 4;
            if (l == 0) g.x -= scale;
            else if (l == 1) g.y -= scale;
            else if (l == 2) g.z -= scale;
            else g.w -= scale;
          }
        }
        if (sink.store_f32) *reinterpret_cast<float4*>(dl + r * C + c0 + 4 * tid) = g;
        if (sink.out) SinkStore4(sink, r * C + c0 + 4 * tid, g);
      }
    } else if (probs) {  // kBwd: C % 4 == 0, no partial group
      if (left > 0) pr[c0 + 4 * tid] = q.x;
      if (left > 1) pr[c0 + 4 * tid + 1] = q.y;
      if (left > 2) pr[c0 + 4 * tid + 2] = q.z;
    }
  }
  if (tid == 0) {
    double term = 0.0;
    if (!zero) {
      // The label's probability exactly as stored; NaN propagates, the
      // clamp only rescues underflow (loss.cc:45-51).
      const float pl = expf(x[lc] - mx) * inv_sum;
      const double safe = pl != pl ? static_cast<double>(pl) : static_cast<double>(fmaxf(pl, 1e-12f));
      term = -log(safe);
    }
    row_loss[r] = term;
  }
}

// Fixed-order mean of the per-row terms (and, masked, the target count).
__global__ void __launch_bounds__(1024)
XEntFinishKernel(const double* __restrict__ row_loss, const int32_t* __restrict__ labels,
                 float* __restrict__ loss, size_t N, int masked) {
  __shared__ double red[1024 / kWave];
  double total = 0.0, targets = 0.0;
  for (size_t r = threadIdx.x; r < N; r += 1024) {
    total += row_loss[r];
    if (!masked || labels[r] >= 0) targets += 1.0;
  }
  total = BlockSumD<1024>(total, red);
  targets = BlockSumD<1024>(targets, red);
  if (threadIdx.x == 0) {
    if (masked)
      *loss = targets > 0.0 ? static_cast<float>(total / targets) : 0.0f;
    else
      *loss = static_cast<float>(total / static_cast<double>(N));
  }
}

// The backward scale: seed / N, or seed / T over the target rows (masked).
__global__ void __launch_bounds__(1024)
XEntScaleKernel(const int32_t* __restrict__ labels, const float* __restrict__ seed,
                float* __restrict__ scale, size_t N, int masked) {
  __shared__ double red[1024 / kWave];
  double t = 0.0;
  if (masked)
    for (size_t r = threadIdx.x; r < N; r += 1024) t += labels[r] >= 0 ? 1.0 : 0.0;
  t = BlockSumD<1024>(t, red);
  if (threadIdx.x == 0) {
    if (masked) {
      const uint64_t T = static_cast<uint64_t>(t);
      *scale = T ? *seed / static_cast<float>(T) : 0.0f;
    } else {
      *scale = *seed / static_cast<float>(N);
    }
  }
}

// One workgroup per row (grid-stride over rows): the label is read once,
// the row moves as float4 where it can.
__global__ void __launch_bounds__(256)
XEntBwdKernel(const float* __restrict__ probs, const int32_t* __restrict__ labels,
              const float* __restrict__ scale_p, float* __restrict__ dl, size_t N, size_t C,
              int masked, Bf16Sink sink) {
  const float scale = *scale_p;
  const bool vec = Vec4Rows(probs, C) && Vec4Rows(dl, C);  // always, with a sink
  for (size_t r = blockIdx.x; r < N; r += gridDim.x) {
    const int32_t lab = labels[r];
    const float* pr = probs + r * C;
    float* dr = dl + r * C;
    const bool zero = masked && lab < 0;
    const size_t lc = static_cast<size_t>(lab);
    if (vec) {
      const float4* p4 = reinterpret_cast<const float4*>(pr);
      float4* d4 = reinterpret_cast<float4*>(dr);
      for (size_t c = threadIdx.x; c < C / 4; c += 256) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!zero) {
          const float4 q = p4[c];
          v = make_float4(scale * q.x, scale * q.y, scale * q.z, scale * q.w);
          if (lc / 4 == c) {  // the label's element, by component
            const size_t l = lc % 4;
            if (l == 0) v.x -= scale;
            else if (l == 1) v.y -= scale;
            else if (l == 2) v.z -= scale;
            else v.w -= scale;
          }
        }
        if (sink.store_f32) d4[c] = v;
        if (sink.out) SinkStore4(sink, r * C + 4 * c, v);
      }
    } else {
      for (size_t c = threadIdx.x; c < C; c += 256) {
        float v = 0.0f;
        if (!zero) {
          v = scale * pr[c];
          if (lc == c) v -= scale;
        }
        dr[c] = v;
      }
    }
  }
}

// The whole loss turn for a few rows (N <= 1024, N x C <= kSmallFloats, rows
// 16-byte aligned) in one workgroup: the seed's fill, the row max, the
// exps into LDS, the exp-sum chain of each row in column order, the
// probabilities and their gradient, the loss -- every value the
// multi-kernel path's expression in its association (the chain's
// sum += e, the probability e * (1 / sum), XEntFinishKernel's tree over the
// row terms), so the bits are the same.  Small plans run the turn in one
// dispatch instead of six.
constexpr int kSmallThreads = 1024;
constexpr size_t kSmallFloats = 16384;
__global__ void __launch_bounds__(kSmallThreads)
XEntSmallKernel(const float* __restrict__ logits, const int32_t* __restrict__ labels,
                float* __restrict__ loss, float* __restrict__ probs, float* fill_dst,
                uint64_t fill_n, float fill_v, const float* seed, float* __restrict__ dl,
                size_t N, size_t C, int masked, Bf16Sink sink) {
  // Rows four floats apart from their length: the chains' 16-byte reads, a
  // row per lane, then fall on different banks.
  __shared__ __attribute__((aligned(16))) float e[kSmallFloats + 4 * kSmallThreads];
  const size_t ld = C + 4;
  __shared__ float smax[kSmallThreads], sinv[kSmallThreads];
  __shared__ double rloss[kSmallThreads];
  __shared__ double red[kSmallThreads / kWave];
  __shared__ float sscale;
  constexpr int kWaves = kSmallThreads / kWave;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  for (uint64_t i = tid; i < fill_n; i += kSmallThreads) fill_dst[i] = fill_v;
  for (size_t r = wave; r < N; r += kWaves) {  // row max, a wave per row
    const float4* x4 = reinterpret_cast<const float4*>(logits + r * C);
    float mx = NAN, mx2 = NAN;
    for (size_t c = lane; c < C / 4; c += kWave) {
      const float4 v = x4[c];
      mx = fmaxf(mx, fmaxf(v.x, v.y));
      mx2 = fmaxf(mx2, fmaxf(v.z, v.w));
    }
    mx = WaveMaxF(fmaxf(mx, mx2));
    if (lane == 0) smax[r] = mx;
  }
  __syncthreads();
  for (size_t i = tid; i < N * C / 4; i += kSmallThreads) {  // the exps
    const float4 v = reinterpret_cast<const float4*>(logits)[i];
    const float mx = smax[4 * i / C];
    *reinterpret_cast<float4*>(e + 4 * i / C * ld + 4 * i % C) =
        make_float4(expf(v.x - mx), expf(v.y - mx), expf(v.z - mx), expf(v.w - mx));
  }
  __syncthreads();
  if (static_cast<size_t>(tid) < N) {  // each row's chain in column order, reads ahead of its adds
    const float4* er = reinterpret_cast<const float4*>(e + tid * ld);
    float sum = 0.0f;
    float4 now = er[0];
    for (size_t c = 0; c < C / 4; ++c) {
      const float4 next = er[c + 1];  // past the row: its padding
      sum += now.x;
      sum += now.y;
      sum += now.z;
      sum += now.w;
      now = next;
    }
    sinv[tid] = 1.0f / sum;  // loss.cc:30
  }
  double t = 0.0;
  if (masked)
    for (size_t r = tid; r < N; r += kSmallThreads) t += labels[r] >= 0 ? 1.0 : 0.0;
  t = BlockSumD<kSmallThreads>(t, red);  // also orders the fill and the chains before what follows
  if (tid == 0) {
    if (masked) {
      const uint64_t T = static_cast<uint64_t>(t);
      sscale = T ? *seed / static_cast<float>(T) : 0.0f;
    } else {
      sscale = *seed / static_cast<float>(N);
    }
  }
  __syncthreads();
  const float scale = sscale;
  for (size_t r = wave; r < N; r += kWaves) {  // probabilities, gradient, the row's term
    const float inv_sum = sinv[r];
    const int32_t lab = labels[r];
    const bool zero = masked && lab < 0;
    const size_t lc = static_cast<size_t>(lab);
    const float4* e4 = reinterpret_cast<const float4*>(e + r * ld);
    for (size_t c = lane; c < C / 4; c += kWave) {
      const float4 v = e4[c];
      const float4 q = make_float4(v.x * inv_sum, v.y * inv_sum, v.z * inv_sum, v.w * inv_sum);
      if (probs) reinterpret_cast<float4*>(probs + r * C)[c] = q;
      float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
      if (!zero) {
        g = make_float4(scale * q.x, scale * q.y, scale * q.z, scale * q.w);
        if (lc / 4 == c) {
          const size_t l = lc % 4;
          if (l == 0) g.x -= scale;
          else if (l == 1) g.y -= scale;
          else if (l == 2) g.z -= scale;
          else g.w -= scale;
        }
      }
      if (sink.store_f32) reinterpret_cast<float4*>(dl + r * C)[c] = g;
      if (sink.out) SinkStore4(sink, r * C + 4 * c, g);
    }
    if (lane == 0) {
      double term = 0.0;
      if (!zero) {
        const float pl = e[r * ld + lc] * inv_sum;
        const double safe = pl != pl ? static_cast<double>(pl) : static_cast<double>(fmaxf(pl, 1e-12f));
        term = -log(safe);
      }
      rloss[r] = term;
    }
  }
  __syncthreads();
  double total = 0.0, targets = 0.0;
  for (size_t r = tid; r < N; r += kSmallThreads) {
    total += rloss[r];
    if (!masked || labels[r] >= 0) targets += 1.0;
  }
  total = BlockSumD<kSmallThreads>(total, red);
  targets = BlockSumD<kSmallThreads>(targets, red);
  if (tid == 0) {
    if (masked)
      *loss = targets > 0.0 ? static_cast<float>(total / targets) : 0.0f;
    else
      *loss = static_cast<float>(total / static_cast<double>(N));
  }
}

// Rows the row kernel holds: up to 32768 columns, as few waves a row as the
// registers allow so that more rows are in flight (the walk leaves a row's
// other waves waiting).  Forward, us, the three kernels / here: 8192 rows of
// 1000 columns 34.8 / 32.7, 4000 92 / 69, 8000 206 / 125, 16000 420 / 237,
// 32000 837 / 500 (the copy rate: 419); 1000 x 7629 (rows off 16 bytes) 146 /
// 27, 32 x 32000 163 / 28.
constexpr size_t kRowMostCols = 512 * 4 * 16;

template <bool kBwd>
void LaunchRow(const float* logits, const int32_t* labels, float* probs, double* row_loss, size_t N,
               size_t C, int masked, const float* scale, float* dl, const Bf16Sink& sink,
               hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(N));
  const int c = static_cast<int>(C);
#define SEEAI_ROW(T, V, O)                                                                          \
  hipLaunchKernelGGL((XEntRowKernel<T, V, kBwd, O>), grid, dim3(T), 0, s, logits, labels, probs,     \
                     row_loss, c, masked, scale, dl, sink)
  if (C <= 128 * 4 * 2) SEEAI_ROW(128, 2, 8);
  else if (C <= 256 * 4 * 4) SEEAI_ROW(256, 4, 8);
  else if (C <= 256 * 4 * 8) SEEAI_ROW(256, 8, 6);
  else if (C <= 512 * 4 * 8) SEEAI_ROW(512, 8, 6);
  else SEEAI_ROW(512, 16, 4);
#undef SEEAI_ROW
}

}  // namespace

size_t XEntFwdScratchBytes(size_t N) { return N * (8 + 4 + 4) + 256; }

hipError_t LaunchXEntFwd(const float* logits, const int32_t* labels, float* loss, float* probs,
                         size_t N, size_t C, int masked, void* ws, hipStream_t s) {
  if (N == 0) return hipSuccess;
  double* row_loss = static_cast<double*>(ws);
  float* row_max = reinterpret_cast<float*>(row_loss + N);
  float* row_sum = row_max + N;
  const unsigned rows = static_cast<unsigned>(N);
  if (C > 0 && XEntRowResident(C)) {
    LaunchRow<false>(logits, labels, probs, row_loss, N, C, masked, nullptr, nullptr, Bf16Sink{}, s);
    hipLaunchKernelGGL(XEntFinishKernel, dim3(1), dim3(1024), 0, s, row_loss, labels, loss, N, masked);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(XEntRowMaxKernel, dim3(rows), dim3(kMaxThreads), 0, s, logits, row_max, C);
  hipLaunchKernelGGL(XEntSerialSumKernel, dim3(static_cast<unsigned>((N + kSumRows - 1) / kSumRows)),
                     dim3(kSumThreads), 0, s, logits, row_max, row_sum, N, C);
  hipLaunchKernelGGL((XEntProbsKernel<false>), dim3(rows), dim3(kProbThreads), 0, s, logits, labels,
                     row_max, row_sum, probs, row_loss, C, masked, nullptr, nullptr, Bf16Sink{});
  hipLaunchKernelGGL(XEntFinishKernel, dim3(1), dim3(1024), 0, s, row_loss, labels, loss, N, masked);
  return hipGetLastError();
}

bool XEntRowResident(size_t C) { return C <= kRowMostCols; }

bool XEntOneWorkgroup(size_t N, size_t C) {
  return N <= static_cast<size_t>(kSmallThreads) && N * C <= kSmallFloats;
}

bool XEntFusedFits(const float* logits, const float* probs, const float* dlogits, size_t C) {
  return C > 0 && Vec4Rows(logits, C) && (!probs || Vec4Rows(probs, C)) && Vec4Rows(dlogits, C);
}

hipError_t LaunchXEntFwdBwd(const float* logits, const int32_t* labels, float* loss, float* probs,
                            float* fill_dst, uint64_t fill_n, float fill_v, const float* seed,
                            float* dlogits, size_t N, size_t C, int masked, void* ws,
                            hipStream_t s, const Bf16Sink& sink, const float* max_parts) {
  if (N == 0) return hipSuccess;
  if (!XEntFusedFits(logits, probs, dlogits, C)) return hipErrorInvalidValue;
  if (XEntOneWorkgroup(N, C)) {
    hipLaunchKernelGGL(XEntSmallKernel, dim3(1), dim3(kSmallThreads), 0, s, logits, labels, loss,
                       probs, fill_dst, fill_n, fill_v, seed, dlogits, N, C, masked, sink);
    return hipGetLastError();
  }
  if (hipError_t e = LaunchFill(fill_dst, fill_v, fill_n, s); e != hipSuccess) return e;
  double* row_loss = static_cast<double*>(ws);
  float* row_max = reinterpret_cast<float*>(row_loss + N);
  float* row_sum = row_max + N;
  float* scale = row_sum + N;  // in the scratch's spare tail
  const unsigned rows = static_cast<unsigned>(N);
  hipLaunchKernelGGL(XEntScaleKernel, dim3(1), dim3(1024), 0, s, labels, seed, scale, N, masked);
  if (XEntRowResident(C)) {
    LaunchRow<true>(logits, labels, probs, row_loss, N, C, masked, scale, dlogits, sink, s);
    hipLaunchKernelGGL(XEntFinishKernel, dim3(1), dim3(1024), 0, s, row_loss, labels, loss, N, masked);
    return hipGetLastError();
  }
  if (max_parts)
    hipLaunchKernelGGL(XEntRowMaxPartsKernel, dim3(rows), dim3(kMaxThreads), 0, s, max_parts,
                       (C + 63) / 64, row_max);
  else
    hipLaunchKernelGGL(XEntRowMaxKernel, dim3(rows), dim3(kMaxThreads), 0, s, logits, row_max, C);
  hipLaunchKernelGGL(XEntSerialSumKernel, dim3(static_cast<unsigned>((N + kSumRows - 1) / kSumRows)),
                     dim3(kSumThreads), 0, s, logits, row_max, row_sum, N, C);
  hipLaunchKernelGGL((XEntProbsKernel<true>), dim3(rows), dim3(kProbThreads), 0, s, logits, labels,
                     row_max, row_sum, probs, row_loss, C, masked, scale, dlogits, sink);
  hipLaunchKernelGGL(XEntFinishKernel, dim3(1), dim3(1024), 0, s, row_loss, labels, loss, N, masked);
  return hipGetLastError();
}

bool XEntBwdSinkFits(const float* probs, const float* dlogits, size_t C) {
  return C > 0 && Vec4Rows(probs, C) && Vec4Rows(dlogits, C);
}

hipError_t LaunchXEntBwd(const float* probs, const int32_t* labels, const float* seed,
                         float* dlogits, size_t N, size_t C, int masked, void* ws,
                         hipStream_t s, const Bf16Sink& sink) {
  if (N == 0) return hipSuccess;
  if ((sink.out || !sink.store_f32) && !XEntBwdSinkFits(probs, dlogits, C)) return hipErrorInvalidValue;
  float* scale = static_cast<float*>(ws);
  hipLaunchKernelGGL(XEntScaleKernel, dim3(1), dim3(1024), 0, s, labels, seed, scale, N, masked);
  hipLaunchKernelGGL(XEntBwdKernel, dim3(static_cast<unsigned>(N < 65536 ? N : 65536)), dim3(256), 0,
                     s, probs, labels, scale, dlogits, N, C, masked, sink);
  return hipGetLastError();
}

}  // namespace seeai
