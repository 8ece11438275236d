// attn_tile.h -- the staged bf16 tile of the head-width-64 attention kernels
// (k_attn16.hip, k_attn3.hip) and its MFMA fragments.
#ifndef SEEAI_ATTN_TILE_H_
#define SEEAI_ATTN_TILE_H_

#include "common.h"

namespace seeai {
namespace {

constexpr int kD = 64;          // head width
constexpr int kBlkRows = 64;    // rows of a staged tile
constexpr int kTile = kBlkRows * kD * 2;  // bytes of one staged tile (8 KiB)
constexpr int kHalf = kTile / 2;          // one 64-byte-row half
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int kRsrcWord3 = 0x00020000;   // raw buffer, 32-bit format, range-checked

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* LdsPtr;
typedef __attribute__((address_space(3))) bf16x4* LdsBf16x4;

__device__ __forceinline__ float Exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ v16f Mfma(const bf16x8& a, const bf16x8& b, const v16f& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ int Phys(int row, int chunk) { return (chunk + row / 4) & 3; }

// s_waitcnt vmcnt(n), the other counters left alone.
template <int n>
__device__ __forceinline__ void WaitVm() {
  static_assert(n >= 0 && n < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14));
}

// f(integral_constant<I>) for I = 0 .. N-1, unrolled.
template <int I, int N>
struct Unroll {
  template <class F>
  __device__ __forceinline__ static void Run(F&& f) {
    if constexpr (I < N) {
      f(std::integral_constant<int, I>{});
      Unroll<I + 1, N>::Run(f);
    }
  }
};

// The stage ring of a kernel: kStages buffers of one K-and-V (or Q-and-dO)
// block, each a separate LDS object named at compile time (stage ids are
// template constants after unrolling), so the compiler can tell a fragment
// read of one stage from the DMA into another and does not make the read
// wait for that DMA.
#define SEEAI_STAGE_RING(kStages)                                                          \
  static_assert(kStages >= 2 && kStages <= 4, "2 to 4 stages");                            \
  __shared__ __attribute__((aligned(1024))) uint8_t stage_0[2 * kTile];                    \
  __shared__ __attribute__((aligned(1024))) uint8_t stage_1[2 * kTile];                    \
  __shared__ __attribute__((aligned(1024))) uint8_t stage_2[kStages > 2 ? 2 * kTile : 1];  \
  __shared__ __attribute__((aligned(1024))) uint8_t stage_3[kStages > 3 ? 2 * kTile : 1];  \
  auto stage = [&](auto id) -> uint8_t* {                                                  \
    constexpr int kId = decltype(id)::value % kStages;                                     \
    if constexpr (kId == 0) return stage_0;                                                \
    else if constexpr (kId == 1) return stage_1;                                           \
    else if constexpr (kId == 2) return stage_2;                                           \
    else return stage_3;                                                                   \
  }

// Runs blocks 0 .. nblk-1 through the ring: block jb computes from stage
// jb % kStages while blocks jb + 1 .. jb + kStages - 1 land in the others.
// issue(jb, stage) starts block jb's loads (kLoads per wave); step(jb, stage)
// computes it.  Past the last block the last is loaded again into a stage
// no later block reads, so every wait counts the same number of loads.
template <int kStages, int kLoads, class Issue, class Step, class Stage>
__device__ __forceinline__ void RunRing(int nblk, Issue&& issue, Step&& step, Stage&& stage) {
  const int last = nblk - 1;
  Unroll<0, kStages - 1>::Run([&](auto id) { issue(min(decltype(id)::value, last), stage(id)); });
  for (int jb0 = 0; jb0 < nblk; jb0 += kStages) {
    Unroll<0, kStages>::Run([&](auto id) {
      constexpr int kId = decltype(id)::value;
      const int jb = jb0 + kId;
      if (jb >= nblk) return;
      WaitVm<(kStages - 2) * kLoads>();  // block jb's loads have landed
      __syncthreads();  // ... in every wave, and block jb - 1's stage is free
      issue(min(jb + kStages - 1, last), stage(std::integral_constant<int, kId + kStages - 1>{}));
      step(jb, static_cast<const uint8_t*>(stage(id)));
    });
  }
  WaitVm<0>();  // no load into LDS outlives the workgroup
}

// The (b, h) slice of a [B*S, H*64] bf16 tensor as a buffer resource whose
// first record is row `row0`; rows at or past S are out of range (zeros).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t SliceRsrc(const uint16_t* slice, int ld, int S,
                                                            int row0) {
  const int rows = S - row0;
  const int bytes = rows > 0 ? ((rows - 1) * ld + kD) * 2 : 0;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(slice) +
                                               static_cast<size_t>(row0) * ld,
                                           0, Uniform(bytes), kRsrcWord3);
}

// One wave-load of a tile: 16 rows x 64 bytes of one half, lane l filling
// row r0 + l / 4, physical chunk l % 4.  `u` = half * 4 + row group.
__device__ __forceinline__ int TileLoadOffset(int u, int lane, int ld) {
  const int half = u / 4, row = (u % 4) * 16 + lane / 4;
  const int c = (lane % 4 - row / 4) & 3;
  return row * ld * 2 + half * 64 + c * 16;
}
__device__ __forceinline__ void TileLoad(__amdgpu_buffer_rsrc_t rs, uint8_t* tile, int u,
                                         int voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (LdsPtr)(tile + (u / 4) * kHalf + (u % 4) * 1024),
                                           16, voff, 0, 0, 0);
}

// Per-lane byte offsets of the two fragment kinds within a tile.  The
// swizzle's phase repeats every 16 rows, so a fragment 16 k rows further
// down (or 32 rows, for the row kind) is the same offset plus a constant:
// the offsets are computed once and the rest folds into the read's
// immediate.
struct FragOffsets {
  int row[2];  // row kind, k-step parity 0 / 1
  int col[2];  // column kind, lo / hi quads
};
__device__ __forceinline__ FragOffsets MakeFragOffsets(int lane) {
  FragOffsets f;
  const int r = lane % 32, g = lane / 32;
#pragma unroll
  for (int p = 0; p < 2; ++p) f.row[p] = r * 64 + Phys(r, 2 * p + g) * 16;
  const int grp = lane / 16, j = lane % 16;
  const int row = 4 * (grp / 2) + j / 4;
  const int byte = 32 * (grp % 2) + 8 * (j % 4);  // within the 64-byte half row
  const int chunk = byte / 16, in = byte % 16;
  f.col[0] = row * 64 + Phys(row, chunk) * 16 + in;
  f.col[1] = (row + 8) * 64 + Phys(row + 8, chunk) * 16 + in;
  return f;
}

// A fragment with the reduction along the tile's columns: lane (g, c) gets
// row `row0 + c` dims 16 s + 8 g .. + 8 (k-step s of the 64 dims); row0 a
// multiple of 32.
__device__ __forceinline__ bf16x8 RowFrag(const uint8_t* tile, const FragOffsets& f, int row0,
                                          int s) {
  return *reinterpret_cast<const bf16x8*>(tile + (s / 2) * kHalf + row0 * 64 + f.row[s % 2]);
}

// A fragment with the reduction down the tile's rows: lane (g, c) gets
// column `32 dt + c` at rows k0 + 4 g + {0..3} (elements 0-3) and
// k0 + 8 + 4 g + {0..3} (elements 4-7) -- the k order PackTile gives the
// register operand it meets; k0 a multiple of 16.  Two transpose reads of
// 4 rows x 16 columns per 16-lane group: lane 16 G + j points at row
// k0 + 4 (G / 2) + j / 4, columns 32 dt + 16 (G % 2) + 4 (j % 4) .. + 4, and
// receives column 32 dt + 16 (G % 2) + j of the group's four rows.
__device__ __forceinline__ bf16x8 ColFrag(const uint8_t* tile, const FragOffsets& f, int dt,
                                          int k0) {
  const uint8_t* base = tile + dt * kHalf + k0 * 64;
  const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((LdsBf16x4)(base + f.col[0]));
  const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((LdsBf16x4)(base + f.col[1]));
  return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// A 32 x 32 score tile's 16 values in this lane (rows 8q + 4g + e in
// w[4q + e]) as the two B operands of a 16-row-step product over those rows:
// out[h] holds rows 16h + 4g + {0..3} and 16h + 8 + 4g + {0..3}.
__device__ __forceinline__ void PackTile(const float* w, bf16x8* out) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
    out[h] = bf16x8{static_cast<__bf16>(w[8 * h + 0]), static_cast<__bf16>(w[8 * h + 1]),
                    static_cast<__bf16>(w[8 * h + 2]), static_cast<__bf16>(w[8 * h + 3]),
                    static_cast<__bf16>(w[8 * h + 4]), static_cast<__bf16>(w[8 * h + 5]),
                    static_cast<__bf16>(w[8 * h + 6]), static_cast<__bf16>(w[8 * h + 7])};
}

// Lane (g, c)'s 8 dims 16 s + 8 g .. + 8 of one bf16 row, from HBM.
__device__ __forceinline__ bf16x8 OwnedFrag(const uint16_t* row, int s, int lane) {
  return *reinterpret_cast<const bf16x8*>(row + 16 * s + 8 * (lane / 32));
}

// Lanes c and c + 32 combined by v_permlane32_swap (no LDS round trip): the
// swap of v with itself leaves lanes c's value in .x and lane c + 32's in .y
// of both lanes, so the sum is formed in the same order in both.
__device__ __forceinline__ float SwapMax(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float SwapSum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ int WaveMaxI(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, kWave));
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int WaveMinI(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, kWave));
  return __builtin_amdgcn_readfirstlane(v);
}
// all ones when a < 0 or b < 0
__device__ __forceinline__ int Outside(int a, int b) { return (a | b) >> 31; }
__device__ __forceinline__ float OrNegInf(float x, int bad) {
  return __int_as_float((__float_as_int(x) & ~bad) | (static_cast<int>(0xff800000u) & bad));
}
__device__ __forceinline__ float OrZero(float x, int bad) { return __int_as_float(__float_as_int(x) & ~bad); }
// Row r (0..15) of a lane's accumulator within its 32-row tile, less 4 g.
__device__ __forceinline__ constexpr int RowConst(int r) { return 8 * (r / 4) + (r % 4); }

// Work unit: (bh, rank), rank 0 the heaviest of the nb row blocks of one
// (b, h); consecutive workgroup ids go to the 8 XCDs in turn, so ids are
// regrouped to give each XCD whole (b, h) slices, heavy blocks first.
__device__ __forceinline__ void UnitOf(int nb, int& bh, int& rank) {
  const int w = blockIdx.x, total = gridDim.x;
  const int t = total % 8 == 0 ? (w % 8) * (total / 8) + w / 8 : w;
  bh = t / nb;
  rank = t % nb;
}

}  // namespace
}  // namespace seeai

#endif  // SEEAI_ATTN_TILE_H_
