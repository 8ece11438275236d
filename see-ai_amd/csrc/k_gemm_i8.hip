// k_gemm_i8.hip -- the W8A8 GEMM on CDNA4 int8 MFMA: per-row symmetric
// int8 activations x per-output-channel symmetric int8 weights, int32
// accumulation, f32 dequant C[m,n] = (f32(acc) * sa[m]) * sw[n].
//
// The reference has no such kernel (its q8 GEMM widens int8 weights into f32
// arithmetic); the quantizer follows the reference's int8 weight packer
// (compiler/backend/allocation/arena_binder.cc:129-177): scale = max|x|/127,
// an all-zero vector takes 1, a subnormal quotient FLT_MIN, levels
// clamp(round(x / scale), -127, 127) by a true division, ties away from zero.
// int8 x int8 products summed in int32 are exact (|sum| <= 127^2 K < 2^31 for
// K <= 133,144), so every accumulation order gives the same bits.
//
// Layout: activations QA [M, K] row-major, weights packed once into
// QWt [N, K] (K contiguous: both MFMA operands then read 16 contiguous
// bytes per lane).
//
// K a multiple of 16 (and the operands 16-byte aligned): GemmI8DmaKernel, K
// staged 64 bytes at a time through LDS buffers filled by direct-to-LDS buffer
// loads, several stages in flight, on v_mfma_i32_32x32x32_i8.  Its tile goes
// from 256 x 256 (eight waves, a prefill batch) down to 32 x 32 with K split
// over four wave groups of the workgroup (decode, M <= 64): PickTile has the
// rule.  Other K or alignments: GemmI8TileKernel with unaligned loads, staged
// through registers into two padded LDS buffers.
#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstdlib>

#include "common.h"

namespace seeai {
namespace {

// --- quantizers --------------------------------------------------------------

__device__ __forceinline__ float QuantScale(float max_abs) {
  if (max_abs == 0.0f) return 1.0f;
  const float s = __fdiv_rn(max_abs, 127.0f);
  return s > FLT_MIN ? s : FLT_MIN;
}
__device__ __forceinline__ int8_t QuantLevel(float x, float scale) {
  float r = roundf(__fdiv_rn(x, scale));
  r = fminf(fmaxf(r, -127.0f), 127.0f);
  return static_cast<int8_t>(r);
}

constexpr int kQThreads = 256;

// One workgroup per row.  Rows up to kQThreads * 4 * kQRegs floats stay in
// registers between the max pass and the level pass, so X is read from HBM
// once; longer (or unaligned) rows are read twice.
constexpr int kQRegs = 8;

__device__ __forceinline__ uint32_t PackLevels(float4 v, float s) {
  return static_cast<uint32_t>(static_cast<uint8_t>(QuantLevel(v.x, s))) |
         (static_cast<uint32_t>(static_cast<uint8_t>(QuantLevel(v.y, s))) << 8) |
         (static_cast<uint32_t>(static_cast<uint8_t>(QuantLevel(v.z, s))) << 16) |
         (static_cast<uint32_t>(static_cast<uint8_t>(QuantLevel(v.w, s))) << 24);
}

__global__ void __launch_bounds__(kQThreads)
QuantizeRowsKernel(const float* __restrict__ X, int8_t* __restrict__ Q, float* __restrict__ scale,
                   size_t cols) {
  __shared__ float red[kQThreads / kWave];
  const size_t r = blockIdx.x;
  const float* x = X + r * cols;
  int8_t* q = Q + r * cols;
  const bool vec = (cols % 4 == 0) && ((reinterpret_cast<uintptr_t>(x) & 15) == 0) &&
                   ((reinterpret_cast<uintptr_t>(q) & 3) == 0);
  const bool resident = vec && cols <= static_cast<size_t>(kQThreads) * 4 * kQRegs;
  float mx = 0.0f;
  float4 keep[kQRegs];
  if (resident) {
#pragma unroll
    for (int i = 0; i < kQRegs; ++i) {
      const size_t c = (threadIdx.x + static_cast<size_t>(i) * kQThreads) * 4;
      keep[i] = c < cols ? *reinterpret_cast<const float4*>(x + c) : make_float4(0.f, 0.f, 0.f, 0.f);
      mx = fmaxf(mx, fmaxf(fmaxf(fabsf(keep[i].x), fabsf(keep[i].y)),
                           fmaxf(fabsf(keep[i].z), fabsf(keep[i].w))));
    }
  } else if (vec) {
    for (size_t c = threadIdx.x * 4; c < cols; c += kQThreads * 4) {
      const float4 v = *reinterpret_cast<const float4*>(x + c);
      mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
  } else {
    for (size_t c = threadIdx.x; c < cols; c += kQThreads) mx = fmaxf(mx, fabsf(x[c]));
  }
  mx = BlockMaxF<kQThreads>(mx, red);
  const float s = QuantScale(mx);
  if (threadIdx.x == 0) scale[r] = s;
  if (resident) {
#pragma unroll
    for (int i = 0; i < kQRegs; ++i) {
      const size_t c = (threadIdx.x + static_cast<size_t>(i) * kQThreads) * 4;
      if (c < cols) *reinterpret_cast<uint32_t*>(q + c) = PackLevels(keep[i], s);
    }
  } else if (vec) {
    for (size_t c = threadIdx.x * 4; c < cols; c += kQThreads * 4)
      *reinterpret_cast<uint32_t*>(q + c) = PackLevels(*reinterpret_cast<const float4*>(x + c), s);
  } else {
    for (size_t c = threadIdx.x; c < cols; c += kQThreads) q[c] = QuantLevel(x[c], s);
  }
}

// The level of x at scale s from the reciprocal: a = fl(x * fl(1/s)) is
// within 2^-24 + 2^-24 (relative) of x / s, so for |x / s| <= 128 it lies
// within 2^-15 of the correctly rounded quotient fl(x / s).  Round-half-away
// and the clamp can then only disagree when a is within 2^-15 of a half
// integer; a group of four with any element inside 2^-12 of one is redone by
// the true division (QuantLevel).  So the levels are bitwise QuantLevel(x, s)
// for every |x| <= 128 s, which the row's own max guarantees (NaN and
// infinities give what the division gives: inf * 0 and inf / inf are both
// NaN, clamped alike).
__device__ __forceinline__ uint32_t LevelByteFast(float x, float inv, bool& near) {
  const float a = x * inv;
  near = near || fabsf(fabsf(a - truncf(a)) - 0.5f) < 0x1p-12f;
  const float l = fminf(fmaxf(roundf(a), -127.0f), 127.0f);
  return static_cast<uint32_t>(static_cast<uint8_t>(static_cast<int8_t>(l)));
}

__device__ __forceinline__ uint32_t PackLevelsInv(float4 v, float s, float inv) {
  bool near = false;
  const uint32_t w = LevelByteFast(v.x, inv, near) | (LevelByteFast(v.y, inv, near) << 8) |
                     (LevelByteFast(v.z, inv, near) << 16) | (LevelByteFast(v.w, inv, near) << 24);
  return near ? PackLevels(v, s) : w;
}

// Rows of at most 256 * kR floats (16-byte aligned, a multiple of 4): each
// wave walks rows g, g + W, g + 2W, ... (W waves in the grid) with the next
// row's loads in flight while it quantizes the current one.  Lane l holds
// float4 chunks l, l + 64, ... of a row, read by buffer loads over a range of
// exactly that row: chunks past the row end, and the whole of a row past the
// matrix end (the last prefetch), read as zeros without touching memory, so
// every load is issued unconditionally.  The max is a butterfly inside the
// wave (no LDS, no barrier).
template <int kR>
__device__ __forceinline__ void LoadRowChunks(const float* X, size_t row, size_t rows, size_t cols,
                                              int lane, float4 (&v)[kR]) {
  const size_t r = row < rows ? row : rows;
  const bool live = r < rows;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(X) + (live ? r * cols : 0), 0,
      live ? static_cast<int>(cols * 4) : 0, 0x00020000);
#pragma unroll
  for (int i = 0; i < kR; ++i) {
    const auto q = __builtin_amdgcn_raw_buffer_load_b128(rs, (lane + i * kWave) * 16, 0, 0);
    v[i] = *reinterpret_cast<const float4*>(&q);
  }
}

template <int kR>
__device__ __forceinline__ void QuantizeRowChunks(const float4 (&v)[kR], int8_t* q, float* scale,
                                                  size_t cols, int lane) {
  float mx = 0.0f;
#pragma unroll
  for (int i = 0; i < kR; ++i) {
    mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
  }
  mx = WaveMaxF(mx);
  const float s = QuantScale(mx);
  const float inv = 1.0f / s;
  if (lane == 0) *scale = s;
  // The level bytes leave through a buffer range of exactly this row: the
  // stores of chunks past its end are dropped by the range check.
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc(q, 0, static_cast<int>(cols), 0x00020000);
#pragma unroll
  for (int i = 0; i < kR; ++i)
    __builtin_amdgcn_raw_buffer_store_b32(PackLevelsInv(v[i], s, inv), rs, (lane + i * kWave) * 4,
                                          0, 0);
}

template <int kR>
__global__ void __launch_bounds__(kQThreads)
QuantizeRowsWaveKernel(const float* __restrict__ X, int8_t* __restrict__ Q,
                       float* __restrict__ scale, size_t rows, size_t cols) {
  const int lane = threadIdx.x % kWave;
  const size_t W = static_cast<size_t>(gridDim.x) * (kQThreads / kWave);
  // The row index is wave-uniform: kept in scalar registers, so the buffer
  // ranges built from it need no per-lane resolution.
  size_t r = static_cast<size_t>(
      Uniform(static_cast<int>(blockIdx.x * (kQThreads / kWave) + threadIdx.x / kWave)));
  if (r >= rows) return;
  float4 a[kR], b[kR];
  LoadRowChunks<kR>(X, r, rows, cols, lane, a);
  for (;;) {
    LoadRowChunks<kR>(X, r + W, rows, cols, lane, b);
    QuantizeRowChunks<kR>(a, Q + r * cols, scale + r, cols, lane);
    r += W;
    if (r >= rows) break;
    LoadRowChunks<kR>(X, r + W, rows, cols, lane, a);
    QuantizeRowChunks<kR>(b, Q + r * cols, scale + r, cols, lane);
    r += W;
    if (r >= rows) break;
  }
}

// Rows of 1024 kR floats or fewer (16-byte aligned, a multiple of 4): a
// workgroup of four waves per row.  Lane t of the workgroup holds float4
// chunks t, t + 256, ... of the row, read by buffer loads over exactly the
// row (chunks past its end read as zeros and their stores are dropped); the
// row max is a butterfly in each wave, then the four waves' maxima through
// LDS.  Spreading a row over four waves puts more rows' loads in flight per
// CU than the wave-per-row kernel and lets each row's stores start sooner:
// 4096 x 4096 on MI355X 14.3 us against 17.9 us (two waves per row 15.8,
// eight 14.6).  Max-abs is exact in any order and the levels are
// PackLevelsInv's, so the bytes are the wave kernel's.
template <int kR>
__global__ void __launch_bounds__(kQThreads)
QuantizeRowsBlockKernel(const float* __restrict__ X, int8_t* __restrict__ Q,
                        float* __restrict__ scale, size_t cols) {
  constexpr int kWaves = kQThreads / kWave;
  __shared__ float red[kWaves];
  const size_t r = blockIdx.x;
  const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(X) + r * cols, 0, static_cast<int>(cols * 4), 0x00020000);
  float4 v[kR];
#pragma unroll
  for (int i = 0; i < kR; ++i) {
    const auto q = __builtin_amdgcn_raw_buffer_load_b128(rs, (t + i * kQThreads) * 16, 0, 0);
    v[i] = *reinterpret_cast<const float4*>(&q);
  }
  float mx = 0.0f;
#pragma unroll
  for (int i = 0; i < kR; ++i)
    mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
  mx = WaveMaxF(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = red[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, red[w]);
  const float s = QuantScale(mx);
  const float inv = 1.0f / s;
  if (t == 0) scale[r] = s;
  const __amdgpu_buffer_rsrc_t ws = __builtin_amdgcn_make_buffer_rsrc(
      Q + r * cols, 0, static_cast<int>(cols), 0x00020000);
#pragma unroll
  for (int i = 0; i < kR; ++i)
    __builtin_amdgcn_raw_buffer_store_b32(PackLevelsInv(v[i], s, inv), ws, (t + i * kQThreads) * 4,
                                          0, 0);
}

// Column max-abs of W [K, N]: one lane per column, coalesced across lanes.
__global__ void __launch_bounds__(kQThreads)
ColumnScaleKernel(const float* __restrict__ W, float* __restrict__ scale, size_t K, size_t N) {
  const size_t n = static_cast<size_t>(blockIdx.x) * kQThreads + threadIdx.x;
  if (n >= N) return;
  float mx = 0.0f;
  for (size_t k = 0; k < K; ++k) mx = fmaxf(mx, fabsf(W[k * N + n]));
  scale[n] = QuantScale(mx);
}

// Quantize and transpose W [K, N] -> Qt [N, K] through a 32 x 32 LDS tile.
__global__ void __launch_bounds__(kQThreads)
PackTransposeKernel(const float* __restrict__ W, const float* __restrict__ scale,
                    int8_t* __restrict__ Qt, size_t K, size_t N) {
  __shared__ int8_t tile[32][33];
  const size_t k0 = static_cast<size_t>(blockIdx.y) * 32, n0 = static_cast<size_t>(blockIdx.x) * 32;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;  // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    const size_t k = k0 + r, n = n0 + tx;
    tile[r][tx] = (k < K && n < N) ? QuantLevel(W[k * N + n], scale[n]) : 0;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const size_t n = n0 + r, k = k0 + tx;
    if (n < N && k < K) Qt[n * K + k] = tile[tx][r];
  }
}

// --- the large-M GEMM ----------------------------------------------------------

constexpr int kThreads = 256;

// Tile -> workgroup order.  The hardware deals workgroups round-robin over
// the 8 XCDs (workgroup b runs on XCD b % 8), each with its own L2.  When
// the tile count divides by 8, the tiles are renumbered so each XCD owns a
// contiguous run, and the run walks column-major within bands of kGroupM
// row tiles: an XCD's 32 concurrent tiles at 4096^2 share 4 row panels of A
// and 8 column panels of W, so each k-slice of A and W leaves HBM once per
// XCD instead of once per tile row or column.
constexpr int kGroupM = 4;

__device__ __forceinline__ void TileOf(int b, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int ntiles = tiles_m * tiles_n;
  int t = b;
  if (ntiles % 8 == 0) t = (b % 8) * (ntiles / 8) + b / 8;
  const int per_group = kGroupM * tiles_n;
  const int g = t / per_group;
  const int first_m = g * kGroupM;
  const int rows = min(tiles_m - first_m, kGroupM);
  const int off = t % per_group;
  tm = first_m + off % rows;
  tn = off / rows;
}

// 16 bytes of a row: rows of 16-byte multiples are read aligned (kAl), others
// with loads marked unaligned.
template <bool kAl>
__device__ __forceinline__ v4i LoadChunk(const int8_t* p) {
  if constexpr (kAl) {
    return *reinterpret_cast<const v4i*>(p);
  } else {
    typedef int v4iu __attribute__((ext_vector_type(4), aligned(1)));
    return *reinterpret_cast<const v4iu*>(p);
  }
}

// 16 bytes of a row from its byte k, bytes at K and past it zero.
__device__ __forceinline__ v4i LoadTail(const int8_t* row, int64_t k, int64_t K) {
  if (k + 16 <= K) return LoadChunk<false>(row + k);
  v4i v = {0, 0, 0, 0};
  for (int e = 0; e < 16 && k + e < K; ++e)
    v[e / 4] |= static_cast<int>(static_cast<uint32_t>(static_cast<uint8_t>(row[k + e])) << (8 * (e % 4)));
  return v;
}

// BM x BN tile per workgroup of WGM x WGN waves, each wave a (BM/WGM) x
// (BN/WGN) block of 32 x 32 x 32 int8 MFMAs.  K advances BK bytes per step
// through two LDS buffers (rows padded by 16 bytes): the next step's global
// loads are issued before the current step's MFMAs and land in the other
// buffer after them, so one barrier per step orders both hazards.  Without
// kAl, rows of any length and alignment: unaligned loads, the last step's
// bytes past K masked to zero.
template <int BM, int BN, int BK, int WGM, int WGN, bool kAl>
__global__ void __launch_bounds__(WGM * WGN * kWave)
GemmI8TileKernel(const int8_t* __restrict__ QA, const float* __restrict__ sa,
                 const int8_t* __restrict__ QW, const float* __restrict__ sw,
                 float* __restrict__ C, int32_t* __restrict__ acc_out, int M, int N, int64_t K,
                 size_t ldc) {
  constexpr int kT = WGM * WGN * kWave;        // lanes per workgroup
  constexpr int LDK = BK + 16;                 // padded LDS row stride (bytes)
  constexpr int WM = BM / WGM, WN = BN / WGN;  // per-wave block
  constexpr int TM = WM / 32, TN = WN / 32;    // 32 x 32 MFMA tiles per wave
  constexpr int kChunksRow = BK / 16;          // 16-byte chunks per tile row
  constexpr int NA = BM * kChunksRow / kT;
  constexpr int NB = BN * kChunksRow / kT;
  static_assert(NA * kT == BM * kChunksRow && NB * kT == BN * kChunksRow, "tile / lanes");
  // One LDS block: two A buffers then two B buffers (rows padded by 16 B);
  // the epilogue reuses all of it as per-wave staging.
  __shared__ __attribute__((aligned(16))) int8_t smem[2 * (BM + BN) * LDK];
  auto As = [&](int buf) { return smem + buf * (BM * LDK); };
  auto Bs = [&](int buf) { return smem + 2 * BM * LDK + buf * (BN * LDK); };

  const int tid = threadIdx.x;
  const int wave = tid / kWave, lane = tid % kWave;
  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  int tm, tn;
  TileOf(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  v16i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  v4i ra[NA], rb[NB];
  auto load = [&](int64_t k0) {
    const bool whole = k0 + BK <= K;  // wave-uniform
#pragma unroll
    for (int e = 0; e < NA; ++e) {
      const int c = tid + e * kT;
      const int m = m0 + c / kChunksRow;
      const int64_t k = k0 + c % kChunksRow * 16;
      const int8_t* row = QA + static_cast<size_t>(m) * K;
      ra[e] = !(m < M) || k >= K ? v4i{0, 0, 0, 0}
              : kAl || whole      ? LoadChunk<kAl>(row + k)
                                  : LoadTail(row, k, K);
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int c = tid + e * kT;
      const int n = n0 + c / kChunksRow;
      const int64_t k = k0 + c % kChunksRow * 16;
      const int8_t* row = QW + static_cast<size_t>(n) * K;
      rb[e] = !(n < N) || k >= K ? v4i{0, 0, 0, 0}
              : kAl || whole      ? LoadChunk<kAl>(row + k)
                                  : LoadTail(row, k, K);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int e = 0; e < NA; ++e) {
      const int c = tid + e * kT;
      *reinterpret_cast<v4i*>(As(buf) + (c / kChunksRow) * LDK + (c % kChunksRow) * 16) = ra[e];
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
      const int c = tid + e * kT;
      *reinterpret_cast<v4i*>(Bs(buf) + (c / kChunksRow) * LDK + (c % kChunksRow) * 16) = rb[e];
    }
  };

  const int nsteps = static_cast<int>((K + BK - 1) / BK);
  constexpr int KS = BK / 32;  // 32-byte k-steps per LDS buffer
  v4i af[2][TM], bf[2][TN];
  auto read_frags = [&](int buf, int ks, int slot) {
    const int koff = ks * 32 + (lane / 32) * 16;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      af[slot][i] = *reinterpret_cast<const v4i*>(As(buf) + (wm + i * 32 + lane % 32) * LDK + koff);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      bf[slot][j] = *reinterpret_cast<const v4i*>(Bs(buf) + (wn + j * 32 + lane % 32) * LDK + koff);
  };
  load(0);
  store(0);
  __syncthreads();
  for (int it = 0; it < nsteps; ++it) {
    const int buf = it & 1;
    if (it + 1 < nsteps) load(static_cast<int64_t>(it + 1) * BK);
    // Fragments double-buffered in registers: the next k-step's LDS reads
    // are in flight while the current k-step's MFMAs issue.
    read_frags(buf, 0, 0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 1 < KS) read_frags(buf, ks + 1, (ks + 1) & 1);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[ks & 1][i], bf[ks & 1][j],
                                                            acc[i][j], 0, 0, 0);
    }
    if (it + 1 < nsteps) store(buf ^ 1);
    __syncthreads();
  }

  // Epilogue.  Lane holds column (lane % 32) and rows 8*(r/4) + 4*(lane/32)
  // + r%4 of each 32 x 32 tile.  The dequantized tile goes through this
  // wave's slice of LDS (free now: the loop ended on a barrier) so C leaves
  // in row-contiguous 16-byte stores; the row scales are read once per
  // 4-row group as float4.
  if (acc_out) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + wm + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + (r % 4);
          const int n = n0 + wn + j * 32 + lane % 32;
          if (m < M && n < N) acc_out[static_cast<size_t>(m) * ldc + n] = acc[i][j][r];
        }
  }
  constexpr int SLD = WN + 4;  // staging row stride (floats)
  static_assert(WGM * WGN * 32 * SLD * 4 <= 2 * (BM + BN) * LDK, "staging fits in LDS");
  float* stage = reinterpret_cast<float*>(smem) + wave * 32 * SLD;
  const bool vec_out = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  float swv[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 32 + lane % 32;
    swv[j] = n < N ? sw[n] : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int mb = m0 + wm + i * 32;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m4 = mb + 8 * q + 4 * (lane / 32);
      float sav[4];
      if (kAl && m4 + 3 < M && (M % 4) == 0) {
        const float4 v = *reinterpret_cast<const float4*>(sa + m4);
        sav[0] = v.x, sav[1] = v.y, sav[2] = v.z, sav[3] = v.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) sav[e] = m4 + e < M ? sa[m4 + e] : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = 8 * q + 4 * (lane / 32) + e;
          stage[row * SLD + j * 32 + lane % 32] =
              (static_cast<float>(acc[i][j][4 * q + e]) * sav[e]) * swv[j];
        }
    }
    __builtin_amdgcn_wave_barrier();
    constexpr int kVecRow = WN / 4;  // float4 per staged row
#pragma unroll
    for (int t = 0; t < 32 * kVecRow / kWave; ++t) {
      const int idx = lane + t * kWave;
      const int row = idx / kVecRow, c4 = idx % kVecRow;
      const int m = mb + row, n = n0 + wn + c4 * 4;
      const float4 v = *reinterpret_cast<const float4*>(stage + row * SLD + c4 * 4);
      if (m >= M) continue;
      float* dst = C + static_cast<size_t>(m) * ldc + n;
      if (vec_out && n + 3 < N) {
        *reinterpret_cast<float4*>(dst) = v;
      } else {
        if (n < N) dst[0] = v.x;
        if (n + 1 < N) dst[1] = v.y;
        if (n + 2 < N) dst[2] = v.z;
        if (n + 3 < N) dst[3] = v.w;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// --- the GEMM staged by direct-to-LDS loads ---------------------------------------
//
// BM x BN tile per workgroup of KG k-groups of WGM x WGN waves, each wave a
// (BM/WGM) x (BN/WGN) block of v_mfma_i32_32x32x32_i8 accumulators over its
// group's K / KG.  K moves 64 bytes per stage through each group's kStages LDS
// buffers (BM A rows + BN W rows of 64 bytes) filled by buffer_load ... lds,
// which writes a wave's 64 x 16 bytes to consecutive LDS addresses from M0
// without passing through registers; kStages - 1 stages are in flight while
// one is multiplied.  One barrier per stage: every wave's loads of the
// stage it is about to read have landed (vmcnt), and every wave has
// finished reading the buffer the next load overwrites.
//
// The 256 x 256 tile runs eight waves (two per SIMD, 2 x 4, blocks of 128 x
// 64: 128 int32 accumulators per lane), measured 6-7 % faster than four waves
// of 128 x 128 (one per SIMD, 256 accumulators) at 4096^3 and 8192^3: the
// second wave on each SIMD issues MFMAs while the first waits on LDS or the
// barrier.  Small tiles are bound by the latency of their stages' loads, which
// is why K splits over groups there: four groups walk a quarter of the stages
// each with four times the loads in flight, and their int32 partials add
// through LDS (exact in any order).  32 x 4096 x 4096: 9.2 us on fragments
// straight from global memory (16 rows of 64 bytes an instruction), 7.0 us
// here; 256 x 4096 x 4096: 31.5 us on register-staged 128 x 128 tiles, 13.2
// us on 64 x 64 with two groups.
//
// LDS rows are 64 bytes, four 16-byte chunks; chunk c of row r sits at
// physical chunk (c + r/4) mod 4.  The fragment reads (lane l: row l % 32,
// chunk 2ks + l / 32) are then free of bank conflicts -- measured with
// SQ_LDS_BANK_CONFLICT on gfx950 for ds_read_b128, which also counts
// conflicts for rotations that bring in r/8 or r/16.  Loads pick the global
// chunk that belongs at each physical slot.  Rows past M (or N) and chunks
// past K read as zeros (buffer range check); K must be a multiple of 16.
constexpr int kDmaBK = 64;
constexpr int kDmaChunks = kDmaBK / 16;

typedef __attribute__((address_space(3))) void* LdsPtr;

__device__ __forceinline__ int DmaPhys(int row, int c) { return (c + row / 4) & 3; }

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding:
// vmcnt[3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8]).
template <int n>
__device__ __forceinline__ void WaitVm() {
  static_assert(n >= 0 && n < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14));
}

template <int BM, int BN, int kStages, int WGM, int WGN, int KG, bool kTail = true,
          bool kHeld = false>
__global__ void __launch_bounds__(KG * WGM * WGN * kWave)
GemmI8DmaKernel(const int8_t* __restrict__ QA, const float* __restrict__ sa,
                const int8_t* __restrict__ QW, const float* __restrict__ sw,
                float* __restrict__ C, int32_t* __restrict__ acc_out, int M, int N, int K) {
  constexpr int kWaves = WGM * WGN;                 // waves of one k-group
  constexpr int WM = BM / WGM, WN = BN / WGN;       // per-wave block
  constexpr int TM = WM / 32, TN = WN / 32;         // 32 x 32 accumulators per wave
  constexpr int kRowsPerLoad = kWave / kDmaChunks;  // rows one wave-load fills (16)
  constexpr int kLoadsA = BM / kRowsPerLoad / kWaves;  // wave-loads per stage and wave
  constexpr int kLoadsB = BN / kRowsPerLoad / kWaves;
  static_assert(kTail || KG == 1, "one group");
  static_assert(kLoadsA * kRowsPerLoad * kWaves == BM && kLoadsB * kRowsPerLoad * kWaves == BN,
                "loads cover the tile");
  constexpr int kStageA = BM * kDmaBK;               // bytes
  constexpr int kStage = (BM + BN) * kDmaBK;
  constexpr int kPerStage = kLoadsA + kLoadsB;       // vmcnt units per stage
  __shared__ __attribute__((aligned(1024))) int8_t smem_all[KG * kStages * kStage];

  const int tid = threadIdx.x;
  const int wave_wg = tid / kWave, lane = tid % kWave;
  const int wave = wave_wg % kWaves, kg = KG > 1 ? Uniform(wave_wg / kWaves) : 0;
  int8_t* const smem = smem_all + kg * (kStages * kStage);
  int tm, tn;
  TileOf(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  // Operand ranges start at this tile's first row: offsets stay below
  // BM * K, and rows past the operand's end fall outside num_records.
  const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(QA) + static_cast<size_t>(m0) * K, 0,
      Uniform((M - m0) * K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_b = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(QW) + static_cast<size_t>(n0) * K, 0,
      Uniform((N - n0) * K), 0x00020000);
  // This lane's slot in each wave-load: row rbase + lane / 4, physical chunk
  // lane % 4, which holds logical chunk (p - r/4) mod 4 (the same for all of
  // its rows: they differ by multiples of 16).
  // (Fixed capacity: an array sized by a template-dependent constant and
  // captured by the lambdas below loses the kernel's host-side stub.)
  static_assert(kLoadsA <= 4 && kLoadsB <= 4, "voff capacity");
  constexpr int kLoads = kLoadsA > kLoadsB ? kLoadsA : kLoadsB;
  int voff[4];
  const int chunk = ((lane % kDmaChunks - (lane / kDmaChunks) / 4) & 3) * 16;
#pragma unroll
  for (int j = 0; j < kLoads; ++j)
    voff[j] = ((j * kWaves + wave) * kRowsPerLoad + lane / kDmaChunks) * K + chunk;
  // This k-group's stages: [kg T, kg T + T) of the K / 64 (rounded up); a
  // chunk at K or past it is read from outside the operand's range, which
  // leaves zeros in LDS.  Without kTail (K % 64 == 0, one group) every stage
  // is whole and its offset stays scalar: the per-lane select costs the 256 x
  // 256 tile 0.7 % at 4096^3.
  const int nsteps_all = (K + kDmaBK - 1) / kDmaBK;
  const int nsteps = (nsteps_all + KG - 1) / KG;
  const int kbase = kg * nsteps * kDmaBK;
  auto issue = [&](int st, int buf) {
    int8_t* sA = smem + buf * kStage;
    int8_t* sB = sA + kStageA;
    const int k0 = kbase + st * kDmaBK;
    const int kadd = !kTail ? 0 : k0 + chunk < K ? k0 : INT32_MIN;
    const int soff = kTail ? 0 : k0;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int rbase = Uniform((j * kWaves + wave) * kRowsPerLoad);
      if (j < kLoadsA)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (LdsPtr)(sA + rbase * kDmaBK), 16,
                                                 voff[j] + kadd, soff, 0, 0);
      if (j < kLoadsB)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_b, (LdsPtr)(sB + rbase * kDmaBK), 16,
                                                 voff[j] + kadd, soff, 0, 0);
    }
  };

  v16i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
  const int lr = lane % 32, h = lane / 32;
  // Fragment offsets within a buffer for k-steps 0 and 1 (logical chunks h
  // and 2 + h of row lr; the tile rows wm + 32 i add multiples of 32 rows,
  // which leave the swizzle unchanged).
  const int frag0 = lr * kDmaBK + DmaPhys(lr, h) * 16;
  const int frag1 = lr * kDmaBK + DmaPhys(lr, 2 + h) * 16;

  // Software pipeline, one k-step (32 bytes of K) ahead in registers: while
  // the MFMAs of one k-step issue, the fragments of the next are read from
  // LDS (spread over the MFMAs).  The barrier sits between a stage's two
  // k-steps: after it, stage it + 1 has landed, and every wave has consumed
  // its reads of stage it - 1 (their MFMAs were issued before the barrier),
  // whose buffer then takes the loads of stage it + kStages - 1.
  v4i fa[2][TM], fb[2][TN];
  auto read = [&](int buf, int fo, int slot) {
    const int8_t* sA = smem + buf * kStage;
    const int8_t* sB = sA + kStageA;
#pragma unroll
    for (int i = 0; i < TM; ++i)
      fa[slot][i] = *reinterpret_cast<const v4i*>(sA + (wm + i * 32) * kDmaBK + fo);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      fb[slot][j] = *reinterpret_cast<const v4i*>(sB + (wn + j * 32) * kDmaBK + fo);
  };
  auto mfmas = [&](int slot) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[slot][j], fa[slot][i], acc[i][j],
                                                          0, 0, 0);
  };
  // The next k-step's TM + TN LDS reads spread over a k-step's TM x TN MFMAs
  // from its start; after the barrier, the stage's loads take the last MFMA
  // slots.
  constexpr int kMfmas = TM * TN, kReads = TM + TN;
  constexpr int kPerSlot = (kReads + kMfmas - 1) / kMfmas;
  auto interleave = [&](bool loads) {
#pragma unroll
    for (int g = 0; g < kMfmas; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (g * kPerSlot < kReads) __builtin_amdgcn_sched_group_barrier(0x100, kPerSlot, 0);
      if (loads && kMfmas >= kPerStage && g >= kMfmas - kPerStage)
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
  };

  // A K that the buffers hold whole (kHeld): every stage at once and one wait,
  // 1 x 2048 x 512 3.4 -> 3.0 us.  Else every iteration loads one stage: past the
  // last stage the loads repeat it (in bounds, into a buffer no later stage
  // uses), so the number of stages in flight at each barrier is always kStages - 3.
  const int last = nsteps - 1;
  if constexpr (kHeld) {  // last < kStages
#pragma unroll
    for (int s = 0; s < kStages; ++s)
      if (s <= last) issue(s, s);
    WaitVm<0>();
    __builtin_amdgcn_s_barrier();
    for (int s = 0; s <= last; ++s) {
      read(s, frag0, 0);
      read(s, frag1, 1);
      mfmas(0);
      mfmas(1);
    }
  } else {
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s) issue(min(s, last), s);
    WaitVm<(kStages - 2) * kPerStage>();
    __builtin_amdgcn_s_barrier();
    read(0, frag0, 0);
    for (int it = 0; it < last; ++it) {
      const int buf = it % kStages;
      read(buf, frag1, 1);
      mfmas(0);
      interleave(false);
      WaitVm<(kStages - 3) * kPerStage>();
      __builtin_amdgcn_s_barrier();
      issue(min(it + kStages - 1, last), (it + kStages - 1) % kStages);
      read((it + 1) % kStages, frag0, 0);
      mfmas(1);
      interleave(true);
    }
    read(last % kStages, frag1, 1);
    mfmas(0);
    interleave(false);
    mfmas(1);
    WaitVm<0>();  // the repeated loads have landed before the workgroup ends
  }

  // The products are C^T tiles (W fragments as the A operand): lane (h, lr)
  // holds columns n = 32 j + 8 q + 4 h + e, e < 4, of row m = 32 i + lr --
  // four consecutive floats of one C row, stored as 16 bytes straight from
  // registers.  Rows off 16 bytes go through LDS (the stages are done with) and
  // leave a row's consecutive floats a wave: four-byte stores of a lane's own
  // quad touch 32 rows each and took 98 us at 3500 x 5630 x 64, 45 here; 1004
  // x 2902 x 304 20.0 and 12.5.
  const bool vec_out = (N % 4) == 0 && ((reinterpret_cast<uintptr_t>(C) |
                                         reinterpret_cast<uintptr_t>(sw) |
                                         reinterpret_cast<uintptr_t>(acc_out)) & 15) == 0;
  auto store = [&](int m, int n, float s_a, int a0, int a1, int a2, int a3) {
    const size_t at = static_cast<size_t>(m) * N + n;
    if (n >= N) return;  // N % 4 == 0: whole quads
    const float4 s4 = *reinterpret_cast<const float4*>(sw + n);
    *reinterpret_cast<float4*>(C + at) =
        make_float4((static_cast<float>(a0) * s_a) * s4.x, (static_cast<float>(a1) * s_a) * s4.y,
                    (static_cast<float>(a2) * s_a) * s4.z, (static_cast<float>(a3) * s_a) * s4.w);
    if (acc_out) *reinterpret_cast<int4*>(acc_out + at) = make_int4(a0, a1, a2, a3);
  };
  // The same quad into a staged row (and, rarely asked for, its accumulators).
  auto stage_quad = [&](float* row, int m, int n, float s_a, int a0, int a1, int a2, int a3) {
    const int a[4] = {a0, a1, a2, a3};
    float c[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] = (static_cast<float>(a[e]) * s_a) * sw[min(n + e, N - 1)];
    *reinterpret_cast<float4*>(row) = make_float4(c[0], c[1], c[2], c[3]);
    if (acc_out && m < M)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) acc_out[static_cast<size_t>(m) * N + n + e] = a[e];
  };
  if constexpr (KG == 1) {
    if (!vec_out) {  // a wave's 32 rows at a time, through its own slice
      constexpr int kLd = WN + 4;
      static_assert(kWaves * 32 * kLd * 4 <= kStages * kStage, "rows fit");
      __syncthreads();
      float* rows = reinterpret_cast<float*>(smem) + wave * 32 * kLd;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int mb = m0 + wm + i * 32;
        const float s_a = sa[min(mb + lr, M - 1)];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            stage_quad(rows + lr * kLd + j * 32 + 8 * q + 4 * h, mb + lr,
                       n0 + wn + j * 32 + 8 * q + 4 * h, s_a, acc[i][j][4 * q],
                       acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
        __builtin_amdgcn_wave_barrier();
#pragma unroll 4
        for (int x = lane; x < 32 * WN; x += kWave) {
          const int m = mb + x / WN, n = n0 + wn + x % WN;
          if (m < M && n < N) C[static_cast<size_t>(m) * N + n] = rows[x / WN * kLd + x % WN];
        }
        __builtin_amdgcn_wave_barrier();
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + wm + i * 32 + lr;
      if (m >= M) continue;
      const float s_a = sa[m];
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          store(m, n0 + wn + j * 32 + 8 * q + 4 * h, s_a, acc[i][j][4 * q], acc[i][j][4 * q + 1],
                acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
    }
  } else {
    // The k-groups' partials meet in LDS (the stages are done with): every
    // wave leaves its quads, then sums and stores one KG-th of its block's.
    constexpr int kQuads = TM * TN * 4;
    static_assert(KG * kWaves * kQuads * kWave * 16 <= KG * kStages * kStage, "partials fit");
    static_assert(kQuads % KG == 0, "whole quads per group");
    constexpr int kParts = KG * kWaves * kQuads * kWave * 16, kLd = BN + 4;
    static_assert(kParts + BM * kLd * 4 <= KG * kStages * kStage, "rows fit");
    float* const rows = reinterpret_cast<float*>(smem_all + kParts);
    __syncthreads();
    v4i* part = reinterpret_cast<v4i*>(smem_all);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          part[((kg * kWaves + wave) * kQuads + (i * TN + j) * 4 + q) * kWave + lane] =
              v4i{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kQuads / KG; ++e) {
      const int x = kg * (kQuads / KG) + e, q = x % 4, j = x / 4 % TN, i = x / 4 / TN;
      v4i sum = part[(wave * kQuads + x) * kWave + lane];
#pragma unroll
      for (int w = 1; w < KG; ++w) sum += part[((w * kWaves + wave) * kQuads + x) * kWave + lane];
      const int mr = wm + i * 32 + lr, m = m0 + mr, nr = wn + j * 32 + 8 * q + 4 * h;
      if (!vec_out)
        stage_quad(rows + mr * kLd + nr, m, n0 + nr, sa[min(m, M - 1)], sum[0], sum[1], sum[2], sum[3]);
      else if (m < M)
        store(m, n0 + nr, sa[m], sum[0], sum[1], sum[2], sum[3]);
    }
    if (vec_out) return;
    __syncthreads();
    for (int x = tid; x < BM * BN; x += KG * kWaves * kWave) {
      const int m = m0 + x / BN, n = n0 + x % BN;
      if (m < M && n < N) C[static_cast<size_t>(m) * N + n] = rows[x / BN * kLd + x % BN];
    }
  }
}

inline bool Aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

}  // namespace

int DeviceCUs() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    n = 256;
  cached[dev].store(n, std::memory_order_relaxed);
  return n;
}

namespace {

enum class Tile { k32, k64Split, k64, k128, k256x128, k256, kStaged128 };

// The tile for an M x N output: the direct-to-LDS one whose measured time at
// its number of tiles per CU (x) is least.  A tile's time grows with K much
// alike for all of them, so K stays out but for the largest.  Measured at K =
// 4096, us, MI355X:
//
//   tile (k-groups)    x <= 1               past that
//   32 x 32 (4)        7.2                  11.2 at 2, 21.6 at 4
//   64 x 64 (2)        10.9 at 1/2, 13.2    22.6 at 2, 40.7 at 4
//   64 x 64 (1)        14.5 at 1/2, 15.9    19.3 at 2, 43 at 4, 81 at 8
//   128 x 128          22 at 1/2, 28        50.7 at 2, 71 at 3, 93 at 4
//   256 x 128          33 at 1/2, 45        74 at 1.5, 86.6 at 2
//   256 x 256          47 at 1/4, 50 at 1/2, 59.6 at 3/4, 73 at 1
//
// The two largest run one workgroup per CU, so they pay by whole rounds of
// the CUs.  Over a short K a second round of 256 x 256 is mostly its C stores
// with nothing beside them, and the register-staged 128 x 128 tiles are faster:
// 3500 x 5632 (x = 1.2), K = 64 / 256 / 512 / 1024, 27.9 / 32.6 / 38.2 / 48.5 us
// against 25.5 / 27.2 / 34.4 / 47.0.  Register-staged tiles of 128 x 128 ran all of these
// before: 30-36 us for M from 65 to 1024 at 4096 x 4096, now 11-28.
Tile PickTile(size_t M, size_t N, size_t K) {
  const double cus = DeviceCUs();
  const auto x = [&](size_t bm, size_t bn) {
    return static_cast<double>((M + bm - 1) / bm) * static_cast<double>((N + bn - 1) / bn) / cus;
  };
  const auto rounds = [](double v, double whole, double first, double slope) {
    const double full = std::floor(v), part = v - full;
    return whole * full + (part > 0 ? first + slope * part : 0.0);
  };
  const double x32 = x(32, 32), x64 = x(64, 64), x128 = x(128, 128);
  const double t[] = {std::max(7.2, 6.0 * x32),
                      std::max(9.5 + 3.7 * x64, 11.0 * x64),
                      std::max(14.0 + 2.7 * x64, 10.2 * x64),
                      std::max(17.0 + 11.0 * x128, 23.5 * x128),
                      rounds(x(256, 128), 43.0, 20.0, 25.0),
                      rounds(x(256, 256), 73.0, 25.0, 48.0)};
  const Tile best = static_cast<Tile>(std::min_element(t, t + 6) - t);
  const double x256 = x(256, 256);
  if (best == Tile::k256 && K <= 1024 && x256 > 1.0 && x256 != std::floor(x256))
    return Tile::kStaged128;
  return best;
}

}  // namespace

hipError_t LaunchQuantizeRows(const float* X, int8_t* Q, float* scale, size_t rows, size_t cols,
                              int waves_per_cu, hipStream_t s) {
  if (rows == 0) return hipSuccess;
  const bool vec = cols > 0 && cols % 4 == 0 && Aligned(X, 16) && Aligned(Q, 4);
  if (vec && cols > 1024 && cols <= 8 * 1024 && rows < (size_t{1} << 31)) {
    // Long rows: a workgroup of four waves per row.
    const dim3 grid(static_cast<unsigned>(rows));
    if (cols <= 2 * 1024)
      hipLaunchKernelGGL(QuantizeRowsBlockKernel<2>, grid, dim3(kQThreads), 0, s, X, Q, scale, cols);
    else if (cols <= 4 * 1024)
      hipLaunchKernelGGL(QuantizeRowsBlockKernel<4>, grid, dim3(kQThreads), 0, s, X, Q, scale, cols);
    else
      hipLaunchKernelGGL(QuantizeRowsBlockKernel<8>, grid, dim3(kQThreads), 0, s, X, Q, scale, cols);
    return hipGetLastError();
  }
  if (vec && cols <= 16 * 256 && rows < (size_t{1} << 31)) {
    // waves_per_cu waves per compute unit walk the rows (at least one row each).
    const int cus = DeviceCUs();
    const size_t waves = std::min(rows, static_cast<size_t>(cus) * static_cast<size_t>(waves_per_cu > 0 ? waves_per_cu : 32));
    const size_t per_wg = kQThreads / kWave;
    const dim3 grid(static_cast<unsigned>((waves + per_wg - 1) / per_wg));
    if (cols <= 4 * 256)
      hipLaunchKernelGGL(QuantizeRowsWaveKernel<4>, grid, dim3(kQThreads), 0, s, X, Q, scale,
                         rows, cols);
    else if (cols <= 8 * 256)
      hipLaunchKernelGGL(QuantizeRowsWaveKernel<8>, grid, dim3(kQThreads), 0, s, X, Q, scale,
                         rows, cols);
    else
      hipLaunchKernelGGL(QuantizeRowsWaveKernel<16>, grid, dim3(kQThreads), 0, s, X, Q, scale,
                         rows, cols);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(QuantizeRowsKernel, dim3(static_cast<unsigned>(rows)), dim3(kQThreads), 0, s,
                     X, Q, scale, cols);
  return hipGetLastError();
}

hipError_t LaunchPackWeightsI8(const float* W, int8_t* Qt, float* scale, size_t K, size_t N,
                               hipStream_t s) {
  if (N == 0) return hipSuccess;
  hipLaunchKernelGGL(ColumnScaleKernel, dim3(GridFor(N, kQThreads)), dim3(kQThreads), 0, s, W,
                     scale, K, N);
  if (K == 0) return hipGetLastError();
  hipLaunchKernelGGL(PackTransposeKernel,
                     dim3(static_cast<unsigned>((N + 31) / 32), static_cast<unsigned>((K + 31) / 32)),
                     dim3(kQThreads), 0, s, W, scale, Qt, K, N);
  return hipGetLastError();
}

hipError_t LaunchGemmW8A8(const int8_t* QA, const float* sa, const int8_t* QWt, const float* sw,
                          float* C, int32_t* acc, size_t M, size_t N, size_t K,
                          const TilePolicy& policy, hipStream_t s) {
  if (M == 0 || N == 0) return hipSuccess;
  const bool dma = K > 0 && K % 16 == 0 && Aligned(QA, 16) && Aligned(QWt, 16) &&
                   M < (1u << 30) && N < (1u << 30) && K * 256 < (1ull << 31) &&
                   M * K < (1ull << 31) && N * K < (1ull << 31);
  if (!dma) {
    // Any K and alignment, in blocks whose indices fit 32 bits.  64 x 64 tiles
    // up to three per CU, 128 x 128 of eight waves past that: 1024 x 4096 x
    // 4095 68 / 56 us, 512 x 4096 x 4095 39 / 48 us, 1000 x 3000 x 999 18.2 /
    // 18.5 us (one lane per output, as before: 11.5 ms).
    constexpr size_t kMost = size_t{1} << 30;
    for (size_t m0 = 0; m0 < M; m0 += kMost)
      for (size_t n0 = 0; n0 < N; n0 += kMost) {
        const size_t m = std::min(M - m0, kMost), n = std::min(N - n0, kMost);
        const auto tiles = [&](size_t b) { return (m + b - 1) / b * ((n + b - 1) / b); };
        const bool large = tiles(64) > 3 * static_cast<size_t>(DeviceCUs());
        if (tiles(large ? 128 : 64) >= (size_t{1} << 31)) return hipErrorInvalidValue;
        const size_t at = m0 * N + n0;
        if (large)
          hipLaunchKernelGGL((GemmI8TileKernel<128, 128, 128, 2, 4, false>),
                             dim3(static_cast<unsigned>(tiles(128))), dim3(512), 0, s, QA + m0 * K,
                             sa + m0, QWt + n0 * K, sw + n0, C + at, acc ? acc + at : nullptr,
                             static_cast<int>(m), static_cast<int>(n), static_cast<int64_t>(K), N);
        else
          hipLaunchKernelGGL((GemmI8TileKernel<64, 64, 128, 2, 2, false>),
                             dim3(static_cast<unsigned>(tiles(64))), dim3(256), 0, s, QA + m0 * K,
                             sa + m0, QWt + n0 * K, sw + n0, C + at, acc ? acc + at : nullptr,
                             static_cast<int>(m), static_cast<int>(n), static_cast<int64_t>(K), N);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
      }
    return hipSuccess;
  }
  const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
  const auto tiles = [&](size_t bm, size_t bn) {
    return dim3(static_cast<unsigned>(((M + bm - 1) / bm) * ((N + bn - 1) / bn)));
  };
  // Tile geometry (TilePolicy): from M, N >= w8a8_large_min the policy's
  // large kernel -- by default the direct-to-LDS 256 x 256.
  const bool big = M >= policy.w8a8_large_min && N >= policy.w8a8_large_min;
  if (big && policy.w8a8_large_kernel == 2)
    hipLaunchKernelGGL((GemmI8TileKernel<256, 256, 128, 4, 4, true>), tiles(256, 256), dim3(1024), 0,
                       s, QA, sa, QWt, sw, C, acc, m, n, static_cast<int64_t>(k), N);
  else if (big && policy.w8a8_large_kernel >= 3)
    hipLaunchKernelGGL((GemmI8TileKernel<128, 128, 128, 2, 2, true>), tiles(128, 128), dim3(256), 0,
                       s, QA, sa, QWt, sw, C, acc, m, n, static_cast<int64_t>(k), N);
  else
    switch (big ? Tile::k256 : PickTile(M, N, K)) {
      case Tile::k32:
        if (K <= 4 * 6 * kDmaBK)
          hipLaunchKernelGGL((GemmI8DmaKernel<32, 32, 6, 1, 1, 4, true, true>), tiles(32, 32),
                             dim3(256), 0, s, QA, sa, QWt, sw, C, acc, m, n, k);
        else
          hipLaunchKernelGGL((GemmI8DmaKernel<32, 32, 6, 1, 1, 4>), tiles(32, 32), dim3(256), 0, s,
                             QA, sa, QWt, sw, C, acc, m, n, k);
        break;
      case Tile::k64Split:
        if (K <= 2 * 4 * kDmaBK)
          hipLaunchKernelGGL((GemmI8DmaKernel<64, 64, 4, 2, 2, 2, true, true>), tiles(64, 64),
                             dim3(512), 0, s, QA, sa, QWt, sw, C, acc, m, n, k);
        else
          hipLaunchKernelGGL((GemmI8DmaKernel<64, 64, 4, 2, 2, 2>), tiles(64, 64), dim3(512), 0, s,
                             QA, sa, QWt, sw, C, acc, m, n, k);
        break;
      case Tile::k64:
        hipLaunchKernelGGL((GemmI8DmaKernel<64, 64, 4, 2, 2, 1>), tiles(64, 64), dim3(256), 0, s, QA,
                           sa, QWt, sw, C, acc, m, n, k);
        break;
      case Tile::k128:
        hipLaunchKernelGGL((GemmI8DmaKernel<128, 128, 4, 2, 2, 1>), tiles(128, 128), dim3(256), 0, s,
                           QA, sa, QWt, sw, C, acc, m, n, k);
        break;
      case Tile::k256x128:
        hipLaunchKernelGGL((GemmI8DmaKernel<256, 128, 4, 4, 2, 1>), tiles(256, 128), dim3(512), 0, s,
                           QA, sa, QWt, sw, C, acc, m, n, k);
        break;
      case Tile::k256:
        if (K % kDmaBK == 0)
          hipLaunchKernelGGL((GemmI8DmaKernel<256, 256, 4, 2, 4, 1, false>), tiles(256, 256),
                             dim3(512), 0, s, QA, sa, QWt, sw, C, acc, m, n, k);
        else
          hipLaunchKernelGGL((GemmI8DmaKernel<256, 256, 4, 2, 4, 1>), tiles(256, 256), dim3(512), 0,
                             s, QA, sa, QWt, sw, C, acc, m, n, k);
        break;
      case Tile::kStaged128:
        hipLaunchKernelGGL((GemmI8TileKernel<128, 128, 128, 2, 2, true>), tiles(128, 128), dim3(256),
                           0, s, QA, sa, QWt, sw, C, acc, m, n, static_cast<int64_t>(k), N);
        break;
    }
  return hipGetLastError();
}

}  // namespace seeai
