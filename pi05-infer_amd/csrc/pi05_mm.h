// bf16 matrix products of the prefill and the vision tower on gfx950 MFMA, with their epilogues fused.
//
//   C[M, N] = A[M, K] (row-major activations) . W[N, K]^T (nn.Linear layout), fp32 accumulation,
//
// K a multiple of 64.  Both operands are copied into LDS by direct-to-LDS loads in k-tiles of 64:
// a row's 64 values are one 128-byte line, eight lines a copy (copies of 64-byte half lines, as a
// 16 x 32 fragment read straight from a row-major operand would make them, reach 25-37 GB/s a CU
// against 95-110).  Chunk c (16 bytes) of row r is stored at slot c ^ (r % 8) -- the lanes of a copy
// pick their source chunk so -- which spreads the fragment reads over the banks.  The products are
// formed as W . A^T, so a lane ends with four consecutive columns of one row.
//
// The fragment reads are inline assembly, whole and with their wait in one statement: the compiler
// cannot tell the copies in flight from the slots that are read, and would wait for all of them.
//
// Two kernels:
//
// mm_pp (tiles of 256 x 256, 256 x 192 and 192 x 256): 8 waves, each over its own part of the tile; the two waves
//   of a SIMD belong to different groups, and while one reads its fragments and issues copies
//   (M), the other multiplies (C), one barrier between.  With operands resident this runs at 97 % of the matrix
//   cores' issue rate (2112 of 2048 clocks a k-tile); the copies must not sit between the MFMAs (2590
//   clocks: a copy that has to wait for its place in the address queue holds the wave's MFMAs back),
//   so M issues them all.  The W ring is three deep because W comes from HBM (one k-tile in
//   flight: 3100 clocks of latency and transfer; three: 2250).  On real values the clock falls to
//   1.7-1.9 GHz, so energy counts too; that is no floor: on the same normal operands the library's product takes 275 us
//   where this kernel takes 306 with its GeGLU (M = 2848, N = 32768, K = 2048), and 101 against 107 at M = 968.
// mm_pw (tiles of 64 x 64 to 128 x 128): 8 multiplying waves and two copying ones.  The multiplying
//   waves form two groups that take alternate k-tiles, each over the whole tile (the largest wave
//   tiles, so the fewest LDS reads), and one k-tile passes per barrier; the groups' sums are exchanged
//   through LDS at the end.  What binds it is the copies (about 45 bytes a clock and CU): issued by
//   the multiplying waves they delayed the fragment reads behind them (128 x 128: 1200 clocks a
//   k-tile against 750).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>
#include <vector>

#include "pi05_blocks.h"

namespace pi05 {

// kMmBf16: bf16(sum + bias); kMmGelu: bf16(gelu_tanh(bf16(sum + bias))); kMmF32: the fp32 sums of each
// K split; kMmGeglu: W's rows alternate 16 gate rows and 16 up rows, C = bf16(gelu_tanh(bf16(gate)) bf16(up))
// [M, N / 2]
enum MmEpi { kMmBf16 = 0, kMmGelu = 1, kMmF32 = 2, kMmGeglu = 3 };

struct MmArgs {
  const u16 *A, *W;
  void* C;
  const float* bias;  // fp32 [N] or NULL (kMmBf16, kMmGelu)
  int M, N, K;
  int lda, ldw, ldc;  // row lengths in elements (split s of kMmF32 at C + s M ldc)
  int split;          // K splits (kMmF32), each a run of whole k-tiles
  int cold;           // 1: W comes from HBM (mm_cold)
};

typedef __amdgpu_buffer_rsrc_t mm_rsrc;
typedef __attribute__((address_space(3))) u16 mm_lds;

// Both operands' fragments of one k-tile and wave: a[ks][m] and w[ks][n], rows 16 i + lane % 16, chunks
// 4 ks + lane / 16; a0 / a1 (w0 / w1): the LDS byte addresses of fragment 0 at ks 0 / 1.
template <int FM, int FN>
struct MmFrags;
#define MM_RD(d, a, o) "ds_read_b128 %" #d ", %" #a " offset:" #o "\n\t"
template <>
struct MmFrags<8, 4> {
  bf16x8 a[2][8], w[2][4];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 26, 0) MM_RD(1, 24, 0) MM_RD(2, 24, 2048) MM_RD(3, 24, 4096) MM_RD(4, 24, 6144) MM_RD(5, 24, 8192) MM_RD(6, 24, 10240)
        MM_RD(7, 24, 12288) MM_RD(8, 24, 14336) MM_RD(9, 26, 2048) MM_RD(10, 26, 4096) MM_RD(11, 26, 6144) MM_RD(12, 27, 0) MM_RD(13, 25, 0)
        MM_RD(14, 25, 2048) MM_RD(15, 25, 4096) MM_RD(16, 25, 6144) MM_RD(17, 25, 8192) MM_RD(18, 25, 10240) MM_RD(19, 25, 12288)
        MM_RD(20, 25, 14336) MM_RD(21, 27, 2048) MM_RD(22, 27, 4096) MM_RD(23, 27, 6144)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(a[0][4]), "=&v"(a[0][5]), "=&v"(a[0][6]),
          "=&v"(a[0][7]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[0][3]), "=&v"(w[1][0]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[1][2]),
          "=&v"(a[1][3]), "=&v"(a[1][4]), "=&v"(a[1][5]), "=&v"(a[1][6]), "=&v"(a[1][7]), "=&v"(w[1][1]), "=&v"(w[1][2]), "=&v"(w[1][3])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
template <>
struct MmFrags<8, 3> {
  bf16x8 a[2][8], w[2][3];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 24, 0) MM_RD(1, 22, 0) MM_RD(2, 22, 2048) MM_RD(3, 22, 4096) MM_RD(4, 22, 6144) MM_RD(5, 22, 8192) MM_RD(6, 22, 10240)
        MM_RD(7, 22, 12288) MM_RD(8, 22, 14336) MM_RD(9, 24, 2048) MM_RD(10, 24, 4096) MM_RD(11, 25, 0) MM_RD(12, 23, 0) MM_RD(13, 23, 2048)
        MM_RD(14, 23, 4096) MM_RD(15, 23, 6144) MM_RD(16, 23, 8192) MM_RD(17, 23, 10240) MM_RD(18, 23, 12288) MM_RD(19, 23, 14336)
        MM_RD(20, 25, 2048) MM_RD(21, 25, 4096)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(a[0][4]), "=&v"(a[0][5]), "=&v"(a[0][6]),
          "=&v"(a[0][7]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[1][0]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[1][2]), "=&v"(a[1][3]),
          "=&v"(a[1][4]), "=&v"(a[1][5]), "=&v"(a[1][6]), "=&v"(a[1][7]), "=&v"(w[1][1]), "=&v"(w[1][2])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
template <>
struct MmFrags<6, 4> {
  bf16x8 a[2][6], w[2][4];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 22, 0) MM_RD(1, 20, 0) MM_RD(2, 20, 2048) MM_RD(3, 20, 4096) MM_RD(4, 20, 6144) MM_RD(5, 20, 8192) MM_RD(6, 20, 10240)
        MM_RD(7, 22, 2048) MM_RD(8, 22, 4096) MM_RD(9, 22, 6144) MM_RD(10, 23, 0) MM_RD(11, 21, 0) MM_RD(12, 21, 2048) MM_RD(13, 21, 4096)
        MM_RD(14, 21, 6144) MM_RD(15, 21, 8192) MM_RD(16, 21, 10240) MM_RD(17, 23, 2048) MM_RD(18, 23, 4096) MM_RD(19, 23, 6144)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(a[0][4]), "=&v"(a[0][5]), "=&v"(w[0][1]),
          "=&v"(w[0][2]), "=&v"(w[0][3]), "=&v"(w[1][0]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[1][2]), "=&v"(a[1][3]), "=&v"(a[1][4]),
          "=&v"(a[1][5]), "=&v"(w[1][1]), "=&v"(w[1][2]), "=&v"(w[1][3])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
template <>
struct MmFrags<4, 4> {
  bf16x8 a[2][4], w[2][4];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 18, 0) MM_RD(1, 16, 0) MM_RD(2, 16, 2048) MM_RD(3, 16, 4096) MM_RD(4, 16, 6144) MM_RD(5, 18, 2048) MM_RD(6, 18, 4096)
        MM_RD(7, 18, 6144) MM_RD(8, 19, 0) MM_RD(9, 17, 0) MM_RD(10, 17, 2048) MM_RD(11, 17, 4096) MM_RD(12, 17, 6144) MM_RD(13, 19, 2048)
        MM_RD(14, 19, 4096) MM_RD(15, 19, 6144)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[0][3]),
          "=&v"(w[1][0]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[1][2]), "=&v"(a[1][3]), "=&v"(w[1][1]), "=&v"(w[1][2]), "=&v"(w[1][3])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
template <>
struct MmFrags<4, 3> {
  bf16x8 a[2][4], w[2][3];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 16, 0) MM_RD(1, 14, 0) MM_RD(2, 14, 2048) MM_RD(3, 14, 4096) MM_RD(4, 14, 6144) MM_RD(5, 16, 2048) MM_RD(6, 16, 4096)
        MM_RD(7, 17, 0) MM_RD(8, 15, 0) MM_RD(9, 15, 2048) MM_RD(10, 15, 4096) MM_RD(11, 15, 6144) MM_RD(12, 17, 2048) MM_RD(13, 17, 4096)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[1][0]),
          "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[1][2]), "=&v"(a[1][3]), "=&v"(w[1][1]), "=&v"(w[1][2])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
template <>
struct MmFrags<4, 2> {
  bf16x8 a[2][4], w[2][2];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 14, 0) MM_RD(1, 12, 0) MM_RD(2, 12, 2048) MM_RD(3, 12, 4096) MM_RD(4, 12, 6144) MM_RD(5, 14, 2048) MM_RD(6, 15, 0) MM_RD(7, 13, 0)
        MM_RD(8, 13, 2048) MM_RD(9, 13, 4096) MM_RD(10, 13, 6144) MM_RD(11, 15, 2048)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[0][2]), "=&v"(a[0][3]), "=&v"(w[0][1]), "=&v"(w[1][0]), "=&v"(a[1][0]),
          "=&v"(a[1][1]), "=&v"(a[1][2]), "=&v"(a[1][3]), "=&v"(w[1][1])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
template <>
struct MmFrags<2, 3> {
  bf16x8 a[2][2], w[2][3];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 12, 0) MM_RD(1, 10, 0) MM_RD(2, 10, 2048) MM_RD(3, 12, 2048) MM_RD(4, 12, 4096) MM_RD(5, 13, 0) MM_RD(6, 11, 0) MM_RD(7, 11, 2048)
        MM_RD(8, 13, 2048) MM_RD(9, 13, 4096)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(w[0][1]), "=&v"(w[0][2]), "=&v"(w[1][0]), "=&v"(a[1][0]), "=&v"(a[1][1]),
          "=&v"(w[1][1]), "=&v"(w[1][2])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
template <>
struct MmFrags<2, 2> {
  bf16x8 a[2][2], w[2][2];
  __device__ __forceinline__ void load(uint32_t a0, uint32_t a1, uint32_t w0, uint32_t w1) {
    asm volatile(
        MM_RD(0, 10, 0) MM_RD(1, 8, 0) MM_RD(2, 8, 2048) MM_RD(3, 10, 2048) MM_RD(4, 11, 0) MM_RD(5, 9, 0) MM_RD(6, 9, 2048) MM_RD(7, 11, 2048)
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0][0]), "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(w[0][1]), "=&v"(w[1][0]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(w[1][1])
        : "v"(a0), "v"(a1), "v"(w0), "v"(w1)
        : "memory");
  }
};
#undef MM_RD

template <int N>
__device__ __forceinline__ void mm_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// s_barrier alone: what it must order (fragments read, copies landed) was waited for before it
__device__ __forceinline__ void mm_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
template <int V>
struct MmInt {
  static constexpr int v = V;
};

// Tiles are numbered in bands of up to kMmBand m-tiles, m fastest, one K split after the other, and XCD x takes
// one contiguous run of them (workgroups are dealt round-robin over the 8 XCDs): the 32 tiles an XCD works on
// at a time share few rows of A and of W in its L2.  Workgroup w of the g
// on XCD x takes the run's tiles w, w + g, ...: with one workgroup per tile exactly one, as a run of n tiles
// has n workgroups then.
constexpr int kMmBand = 6;
__device__ __forceinline__ int mm_tiles(const MmArgs& a, int bm, int bn) { return ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn) * a.split; }
__device__ __forceinline__ int mm_last(int tiles) {
  const int x = blockIdx.x & 7, r = tiles & 7;
  return (x + 1) * (tiles >> 3) + (x + 1 < r ? x + 1 : r);
}
__device__ __forceinline__ int mm_first(int tiles) {
  const int x = blockIdx.x & 7, r = tiles & 7;
  return x * (tiles >> 3) + (x < r ? x : r) + (blockIdx.x >> 3);
}
__device__ __forceinline__ void mm_tile(const MmArgs& a, int bm, int bn, int id, int& mt, int& nt, int& sp) {
  const int tm = (a.M + bm - 1) / bm, tn = (a.N + bn - 1) / bn;
  sp = id / (tm * tn);
  id -= sp * tm * tn;
  const int band = id / (kMmBand * tn), h = tm - band * kMmBand < kMmBand ? tm - band * kMmBand : kMmBand;
  id -= band * kMmBand * tn;
  mt = band * kMmBand + id % h;
  nt = id / h;
}

// gelu_tanh(x) = x (1 + tanh(u)) / 2 = x / (1 + exp(-2 u)), u = sqrt(2 / pi) (x + 0.044715 x^3): one hardware exp2 and
// reciprocal and five other operations.  The epilogues evaluate it 64 times a lane with the matrix cores
// idle (gelu_tanh's fourteen operations: 6 us of a 256 x 256 tile's 55).
__device__ __forceinline__ float mm_gelu(float x) {
  const float k = -2.0f * 0.7978845608028654f * 1.4426950408889634f;  // exp(-2 u) = exp2(k (x + 0.044715 x^3))
  const float e = __builtin_amdgcn_exp2f(x * __builtin_fmaf(x * x, k * 0.044715f, k));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// The epilogue of four columns col .. col + 3 of one row.
template <int EPI>
__device__ __forceinline__ void mm_store(const MmArgs& a, int sp, int row, int col, f32x4 v) {
  if constexpr (EPI == kMmF32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(a.C) + ((size_t)sp * a.M + row) * a.ldc + col) = v;
  } else {
    if (a.bias) {
      const float4 b = *reinterpret_cast<const float4*>(a.bias + col);
      v[0] = fadd(v[0], b.x), v[1] = fadd(v[1], b.y), v[2] = fadd(v[2], b.z), v[3] = fadd(v[3], b.w);
    }
    u16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = EPI == kMmGelu ? f2bf(mm_gelu(round_bf(v[i]))) : f2bf(v[i]);
    *reinterpret_cast<u16x4*>(static_cast<u16*>(a.C) + (size_t)row * a.ldc + col) = o;
  }
}
__device__ __forceinline__ void mm_store_geglu(const MmArgs& a, int row, int col, f32x4 g, f32x4 u) {
  u16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = f2bf(fmul(mm_gelu(round_bf(g[i])), round_bf(u[i])));
  *reinterpret_cast<u16x4*>(static_cast<u16*>(a.C) + (size_t)row * a.ldc + col) = o;
}

// Lane l of a copy fetches chunk (l % 8) ^ (l / 8) of row l / 8; rows past the operand's last one fetch it
// again (their products are not stored).
__device__ __forceinline__ int mm_src(int row, int last, int ld, int lane) {
  return (row < last ? row : last) * ld * 2 + ((lane & 7) ^ (lane >> 3)) * 16;
}
__device__ __forceinline__ mm_rsrc mm_make_rsrc(const u16* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(p), (short)0, 0x7fffffff, 0x00020000);
}

// Tile 32 FM x 64 FN: group wave / 4 owns one M half, wave % 4 one N quarter.  M(t) copies A(t + AS - 1) (this
// group's half) and W(t + WS - 1) into the ring slots that tile t - 1 left, and reads the fragments of tile t;
// C(t) multiplies.  Group 0 runs M(t) in slot 2 t and C(t) in slot 2 t + 1, group 1 one slot later.
template <int FM, int FN, int AS, int WS, int EPI>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void mm_pp_kernel(MmArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = FM * 32, BN = FN * 64;
  constexpr int PA = BM / 64, PW = BN / 64, PT = PA + PW;  // 1 KiB copies of one wave and k-tile
  constexpr int kA = BM * 128, kW = BN * 128;
  static_assert(BM % 64 == 0 && AS * kA + WS * kW <= 160 * 1024 && AS >= 2 && WS >= 2, "tile");
  static_assert(EPI != kMmGeglu || FN % 2 == 0, "gate and up tiles in pairs");
  __shared__ __align__(1024) uint8_t lds[AS * kA + WS * kW];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wave >> 2, wn = wave & 3;
  mm_lds* ldsb = (mm_lds*)lds;
  const uint32_t base = (uint32_t)(uintptr_t)ldsb;
  const int fr = lane & 15, fg = lane >> 4;
  const uint32_t ao = base + (grp * (BM / 2) + fr) * 128, wo = base + AS * kA + (wn * (BN / 4) + fr) * 128;
  const uint32_t x0 = (fg ^ (fr & 7)) * 16, x1 = ((4 + fg) ^ (fr & 7)) * 16;
  constexpr int kMax = AS > WS ? AS : WS;
  // copies that may still be in flight when a slot ends (a wave's loads complete in order): after the
  // group's own A(t + 1), after W(t + 1), after both
  constexpr int wa = PW + (AS - 2) * PT, wb = (WS - 2) * PT, wab = wa < wb ? wa : wb;
  // the tile being multiplied; its operands' copies
  int m0, n0, sp, T;
  mm_rsrc ra, rw;
  int va[PA], vw[PW];
  auto cp_a = [&](int kt, int st) {
#pragma unroll
    for (int i = 0; i < PA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, ldsb + st * (kA / 2) + grp * (BM * 32) + (i * 4 + wn) * 512, 16, va[i], kt * 128, 0, 0);
  };
  auto cp_w = [&](int kt, int st) {
#pragma unroll
    for (int i = 0; i < PW; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, ldsb + AS * (kA / 2) + st * (kW / 2) + (i * 8 + wave) * 512, 16, vw[i], kt * 128, 0, 0);
  };
  // sets out on tile id: its first copies, M(1 - kMax) .. M(-1)
  auto begin = [&](int id) {
    int m_t, n_t;
    mm_tile(a, BM, BN, id, m_t, n_t, sp);
    m0 = m_t * BM, n0 = n_t * BN;
    const int t0 = sp * (a.K / 64) / a.split;
    T = (sp + 1) * (a.K / 64) / a.split - t0;
    ra = mm_make_rsrc(a.A + (size_t)m0 * a.lda + t0 * 64), rw = mm_make_rsrc(a.W + (size_t)n0 * a.ldw + t0 * 64);
#pragma unroll
    for (int i = 0; i < PA; ++i) va[i] = mm_src(grp * (BM / 2) + (i * 4 + wn) * 8 + (lane >> 3), a.M - 1 - m0, a.lda, lane);
#pragma unroll
    for (int i = 0; i < PW; ++i) vw[i] = mm_src((i * 8 + wave) * 8 + (lane >> 3), a.N - 1 - n0, a.ldw, lane);
#pragma unroll
    for (int s = 1 - kMax; s < 0; ++s) {
      if (s + AS - 1 >= 0 && s + AS - 1 < T) cp_a(s + AS - 1, s + AS - 1);
      if (s + WS - 1 >= 0 && s + WS - 1 < T) cp_w(s + WS - 1, s + WS - 1);
    }
  };
  const int tiles = mm_tiles(a, BM, BN);
  int id = mm_first(tiles);
  const int stride = ((int)gridDim.x + 7 - (int)(blockIdx.x & 7)) >> 3, last = mm_last(tiles);  // stride: this XCD's workgroups, at least one
  begin(id);
  mm_wait_vm<wab>();
  for (;;) {
    f32x4 acc[FN][FM];
#pragma unroll
    for (int n = 0; n < FN; ++n)
#pragma unroll
      for (int m = 0; m < FM; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    MmFrags<FM, FN> f;
    int as = 0, ws = 0, al = AS - 1, wl = WS - 1;  // ring slots of the tile being read, of the next copies
    int t = 0;
    if (T < kMax) mm_wait_vm<0>();
    mm_barrier();
    // kin: every copy of the step exists; w0 / w1 / w2 may stay in flight (group 0's C, group 1's M and C)
    auto step = [&](auto kin, auto w0, auto w1, auto w2) {
      if (decltype(kin)::v || t + AS - 1 < T) cp_a(t + AS - 1, al);
      if (decltype(kin)::v || t + WS - 1 < T) cp_w(t + WS - 1, wl);
      const uint32_t sa = as * kA, sw = ws * kW;
      f.load(ao + x0 + sa, ao + x1 + sa, wo + x0 + sw, wo + x1 + sw);
      if (grp) mm_wait_vm<decltype(w1)::v>();
      mm_barrier();
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int n = 0; n < FN; ++n)
#pragma unroll
          for (int m = 0; m < FM; ++m) acc[n][m] = mfma16x16x32(f.w[ks][n], f.a[ks][m], acc[n][m]);
      __builtin_amdgcn_s_setprio(0);
      if (grp) mm_wait_vm<decltype(w2)::v>();
      else mm_wait_vm<decltype(w0)::v>();
      mm_barrier();
      as = as + 1 == AS ? 0 : as + 1, al = al + 1 == AS ? 0 : al + 1;
      ws = ws + 1 == WS ? 0 : ws + 1, wl = wl + 1 == WS ? 0 : wl + 1;
    };
    if (grp) mm_barrier();
    for (; t < T - kMax + 1; ++t) step(MmInt<1>{}, MmInt<wab>{}, MmInt<wb>{}, MmInt<wa>{});
    for (; t < T; ++t) step(MmInt<0>{}, MmInt<0>{}, MmInt<0>{}, MmInt<0>{});
    if (!grp) mm_barrier();
    // every fragment has been read: the next tile's first copies land while this one is stored
    const int em0 = m0, en0 = n0, esp = sp;
    const bool more = id + stride < last;
    if (more) {
      id += stride;
      begin(id);
    }
    // lane l: columns 16 n + 4 (l / 16) .. + 3 of row l % 16
#pragma unroll
    for (int m = 0; m < FM; ++m) {
      const int row = em0 + grp * (BM / 2) + m * 16 + fr, col = en0 + wn * (BN / 4);
      if (row >= a.M) continue;
      if constexpr (EPI == kMmGeglu) {
#pragma unroll
        for (int n = 0; n < FN; n += 2)
          if (col + n * 16 < a.N) mm_store_geglu(a, row, (col + n * 16) / 2 + fg * 4, acc[n][m], acc[n + 1][m]);
      } else {
#pragma unroll
        for (int n = 0; n < FN; ++n)
          if (col + n * 16 < a.N) mm_store<EPI>(a, esp, row, col + n * 16 + fg * 4, acc[n][m]);
      }
    }
    if (!more) return;
    mm_wait_vm<0>();  // copies and stores (which complete in no order with the copies)
  }
#endif
}

// Tile 32 FM x 32 FN: group t % 2 (of 2 x 2 waves) reads tile t's fragments in slot t while the other group
// multiplies tile t - 1; the NP copying waves keep S - 1 tiles in flight.
template <int FM, int FN, int S, int NP, int EPI>
__global__ __launch_bounds__(512 + NP * 64) void mm_pw_kernel(MmArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = FM * 32, BN = FN * 32;
  constexpr int PA = BM / 8 / NP, PW = BN / 8 / NP, PT = PA + PW;  // copies of one copying wave and k-tile
  constexpr int kStage = (BM + BN) * 128, kRed = BM * BN * 4;
  static_assert(S * kStage <= 160 * 1024 && kRed <= S * kStage && (S - 2) * PT < 64 && FM % 2 == 0, "tile");
  static_assert(BM % (8 * NP) == 0 && BN % (8 * NP) == 0, "copies");
  static_assert(EPI != kMmGeglu || FN % 2 == 0, "gate and up tiles in pairs");
  __shared__ __align__(1024) uint8_t lds[S * kStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int m_t, n_t, sp;
  mm_tile(a, BM, BN, mm_first(mm_tiles(a, BM, BN)), m_t, n_t, sp);
  const int m0 = m_t * BM, n0 = n_t * BN;
  const int t0 = sp * (a.K / 64) / a.split, T = (sp + 1) * (a.K / 64) / a.split - t0;
  mm_lds* ldsb = (mm_lds*)lds;
  if (wave >= 8) {
    const int p = wave - 8;  // rows 8 (i NP + p) .. + 7 of both operands
    const mm_rsrc ra = mm_make_rsrc(a.A + (size_t)m0 * a.lda + t0 * 64), rw = mm_make_rsrc(a.W + (size_t)n0 * a.ldw + t0 * 64);
    int va[PA], vw[PW];
#pragma unroll
    for (int i = 0; i < PA; ++i) va[i] = mm_src((i * NP + p) * 8 + (lane >> 3), a.M - 1 - m0, a.lda, lane);
#pragma unroll
    for (int i = 0; i < PW; ++i) vw[i] = mm_src((i * NP + p) * 8 + (lane >> 3), a.N - 1 - n0, a.ldw, lane);
    auto copy = [&](int kt, int st) {
      mm_lds* d = ldsb + st * (kStage / 2);
#pragma unroll
      for (int i = 0; i < PA; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, d + (i * NP + p) * 512, 16, va[i], kt * 128, 0, 0);
#pragma unroll
      for (int i = 0; i < PW; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, d + BM * 64 + (i * NP + p) * 512, 16, vw[i], kt * 128, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
      if (s < T) copy(s, s);
    if (T >= S - 1) mm_wait_vm<(S - 2) * PT>();
    else mm_wait_vm<0>();
    mm_barrier();
    int sl = S - 1;
    for (int t = 0; t < T; ++t) {  // slot t: copies tile t + S - 1 into tile t - 1's place, waits for tile t + 1
      if (t + S - 1 < T) {
        copy(t + S - 1, sl);
        mm_wait_vm<(S - 2) * PT>();
      } else {
        mm_wait_vm<0>();
      }
      mm_barrier();
      sl = sl + 1 == S ? 0 : sl + 1;
    }
    mm_barrier();
    __syncthreads();
    return;
  }
  const int grp = wave >> 2, wq = wave & 3, wm = wq >> 1, wn = wq & 1;
  const uint32_t base = (uint32_t)(uintptr_t)ldsb;
  const int fr = lane & 15, fg = lane >> 4;
  const uint32_t ao = base + (wm * (BM / 2) + fr) * 128, wo = base + BM * 128 + (wn * (BN / 2) + fr) * 128;
  const uint32_t x0 = (fg ^ (fr & 7)) * 16, x1 = ((4 + fg) ^ (fr & 7)) * 16;
  f32x4 acc[FN][FM];
#pragma unroll
  for (int n = 0; n < FN; ++n)
#pragma unroll
    for (int m = 0; m < FM; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  MmFrags<FM, FN> f;
  // Where W comes from HBM: its k-tiles behind the ring's first ones into this XCD's L2, one 128-byte line a
  // load, shared between the m-tiles of a whole band.  The multiplying waves have nothing to do yet, and where all of
  // them are there (M = 768: 6 of 128) the copies after the first few find their lines near instead of waiting for HBM
  // with only the ring in flight (27 layers: 12 % of the tower).  A tile fetches 2048 lines at most, so a long K run over
  // few m-tiles is covered in part; and a shorter last band fetches its tiles' shares only: with all of a band's lines
  // shared between the tiles that it has, the second band of 968 rows (2 of 8 m-tiles) made q|k|v 19.4 us instead of 18.2
  // in the pass and o_proj 16.4 instead of 15.9.  Weights that stay in the 256 MB cache behind the L2s gain nothing and
  // pay for the loads (6 layers: 2 %).  The values are not used.
  constexpr int kPf = 4;
  uint32_t pf[kPf];
  {
    const int tm = (a.M + BM - 1) / BM, share = tm < kMmBand ? tm : kMmBand, lines = BN * (T - (S - 1));
    const u16* wp = a.W + (size_t)n0 * a.ldw + (size_t)(t0 + S - 1) * 64;
#pragma unroll
    for (int j = 0; j < kPf; ++j) {
      const int i = m_t % share + share * (tid + j * 512), kt = i / BN, row = i % BN < a.N - 1 - n0 ? i % BN : a.N - 1 - n0;
      pf[j] = 0;
      if (a.cold && i < lines) pf[j] = *reinterpret_cast<const uint32_t*>(wp + (size_t)row * a.ldw + kt * 64);
    }
  }
  mm_barrier();
  int st = grp;
  if (grp) mm_barrier();
  for (int t = grp; t < T; t += 2) {
    const uint32_t so = st * kStage;
    f.load(ao + x0 + so, ao + x1 + so, wo + x0 + so, wo + x1 + so);
    mm_barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int n = 0; n < FN; ++n)
#pragma unroll
        for (int m = 0; m < FM; ++m) acc[n][m] = mfma16x16x32(f.w[ks][n], f.a[ks][m], acc[n][m]);
    __builtin_amdgcn_s_setprio(0);
    mm_barrier();
    st = st + 2 >= S ? st + 2 - S : st + 2;
  }
  if ((T & 1) == grp) mm_barrier();  // T + 1 slots for either group
#pragma unroll
  for (int j = 0; j < kPf; ++j) asm volatile("" ::"v"(pf[j]));
  // group 0 finishes the m-tiles below FM / 2 of each wave tile, group 1 the others: sum = group 0's + group 1's
  constexpr int HM = FM / 2;
  float* red = reinterpret_cast<float*>(lds) + (size_t)wq * (FM * FN * 256) + lane * 4;
  if (grp) {
#pragma unroll
    for (int n = 0; n < FN; ++n)
#pragma unroll
      for (int m = 0; m < HM; ++m) *reinterpret_cast<f32x4*>(red + (n * FM + m) * 256) = acc[n][m];
  } else {
#pragma unroll
    for (int n = 0; n < FN; ++n)
#pragma unroll
      for (int m = HM; m < FM; ++m) *reinterpret_cast<f32x4*>(red + (n * FM + m) * 256) = acc[n][m];
  }
  __syncthreads();
#pragma unroll
  for (int mm = 0; mm < HM; ++mm) {
    const int m = grp ? HM + mm : mm, row = m0 + wm * (BM / 2) + m * 16 + fr;
    if (row >= a.M) continue;
    f32x4 v[FN];
#pragma unroll
    for (int n = 0; n < FN; ++n) {
      const f32x4 o = *reinterpret_cast<const f32x4*>(red + (n * FM + m) * 256);
      v[n] = grp ? o + acc[n][HM + mm] : acc[n][mm] + o;
    }
    const int col = n0 + wn * (BN / 2);
    if constexpr (EPI == kMmGeglu) {
#pragma unroll
      for (int n = 0; n < FN; n += 2)
        if (col + n * 16 < a.N) mm_store_geglu(a, row, (col + n * 16) / 2 + fg * 4, v[n], v[n + 1]);
    } else {
#pragma unroll
      for (int n = 0; n < FN; ++n)
        if (col + n * 16 < a.N) mm_store<EPI>(a, sp, row, col + n * 16 + fg * 4, v[n]);
    }
  }
#endif
}

// ---------------------------------------------------------------------------------------------
// host: the tiles there are, launches and the choice among them
// ---------------------------------------------------------------------------------------------
constexpr unsigned kMmCus = 256;
enum MmCfg { kMm256x256 = 0, kMm256x192, kMm192x256, kMm128x128, kMm128x96, kMm128x64, kMm64x96, kMm64x64, kMmCfgs };
constexpr int kMmBm[kMmCfgs] = {256, 256, 192, 128, 128, 128, 64, 64}, kMmBn[kMmCfgs] = {256, 192, 256, 128, 96, 64, 96, 64};

inline bool mm_cfg_has(int cfg, int epi) { return epi != kMmGeglu || (cfg != kMm256x192 && cfg != kMm128x96 && cfg != kMm64x96); }

template <int EPI>
inline bool mm_launch_epi(int cfg, const MmArgs& a, hipStream_t st) {
  const unsigned grid = (unsigned)((a.M + kMmBm[cfg] - 1) / kMmBm[cfg]) * (unsigned)((a.N + kMmBn[cfg] - 1) / kMmBn[cfg]) * (unsigned)a.split;
  const unsigned pp = grid < kMmCus ? grid : kMmCus;  // mm_pp: one workgroup per CU, which takes tile after tile
  switch (cfg) {
    case kMm256x256: mm_pp_kernel<8, 4, 2, 3, EPI><<<pp, 512, 0, st>>>(a); break;
    case kMm192x256: mm_pp_kernel<6, 4, 2, 3, EPI><<<pp, 512, 0, st>>>(a); break;
    case kMm128x128: mm_pw_kernel<4, 4, 4, 2, EPI><<<grid, 640, 0, st>>>(a); break;
    case kMm128x64: mm_pw_kernel<4, 2, 6, 2, EPI><<<grid, 640, 0, st>>>(a); break;
    case kMm64x64: mm_pw_kernel<2, 2, 5, 2, EPI><<<grid, 640, 0, st>>>(a); break;
    default:
      if constexpr (EPI != kMmGeglu) {
        if (cfg == kMm256x192) mm_pp_kernel<8, 3, 2, 3, EPI><<<pp, 512, 0, st>>>(a);
        else if (cfg == kMm128x96) mm_pw_kernel<4, 3, 5, 2, EPI><<<grid, 640, 0, st>>>(a);
        else if (cfg == kMm64x96) mm_pw_kernel<2, 3, 6, 2, EPI><<<grid, 640, 0, st>>>(a);
        else return false;
        break;
      }
      return false;
  }
  return hipGetLastError() == hipSuccess;
}

// What the kernels assume of a product: whole k-tiles, at least one per split, 16-byte rows and chunks,
// and tile-relative byte offsets that fit 31 bits.
inline bool mm_fits(int cfg, int epi, const MmArgs& a) {
  auto al16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  return cfg >= 0 && cfg < kMmCfgs && mm_cfg_has(cfg, epi) && a.M > 0 && a.N > 0 && a.N % (epi == kMmGeglu ? 32 : 16) == 0 && a.K > 0 &&
         a.K % 64 == 0 && a.split >= 1 && a.split <= a.K / 64 && (epi == kMmF32 || a.split == 1) && a.lda % 8 == 0 && a.ldw % 8 == 0 &&
         a.ldc % 4 == 0 && a.lda >= a.K && a.ldw >= a.K && a.ldc >= (epi == kMmGeglu ? a.N / 2 : a.N) && (int64_t)a.lda * 512 + a.K * 2 < (1ll << 31) &&
         (int64_t)a.ldw * 512 + a.K * 2 < (1ll << 31) && al16(a.A) && al16(a.W) && al16(a.C) && al16(a.bias);
}

inline bool mm_launch(int cfg, int epi, const MmArgs& a, hipStream_t st) {
  if (!mm_fits(cfg, epi, a)) return false;
  switch (epi) {
    case kMmBf16: return mm_launch_epi<kMmBf16>(cfg, a, st);
    case kMmGelu: return mm_launch_epi<kMmGelu>(cfg, a, st);
    case kMmF32: return mm_launch_epi<kMmF32>(cfg, a, st);
    case kMmGeglu: return mm_launch_epi<kMmGeglu>(cfg, a, st);
    default: return false;
  }
}

// Whether layers' weights of this many bytes in all come from HBM on every pass: more than the memory-side cache keeps.
// A context knows its own weights only: a small model's count as cached also where a larger one runs between its
// passes and flushes them (a 6-layer tower before a 4 GB prefill); it then goes without the lines fetched ahead.
inline int mm_cold(size_t weight_bytes) { return weight_bytes > (256ull << 20) ? 1 : 0; }

// Holds the stream for `ticks` of the 100 MHz counter (or the bounded number of polls).
static __global__ void mm_hold_kernel(unsigned ticks) {
#ifdef __HIP_DEVICE_COMPILE__
  const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
  for (int i = 0; i < 1 << 16 && __builtin_amdgcn_s_memrealtime() - t0 < ticks; ++i) __builtin_amdgcn_s_sleep(2);
#endif
}

// Time of one of `reps` runs in a row (launch(r) enqueues run r), the same for every candidate of a product.  The
// stream is held while the host enqueues them: a 6 us product is otherwise timed at the rate the host launches it,
// where all candidates look alike (a 256-row layer's picks then changed from context to context).
constexpr int kMmFinalists = 6, kMmRounds = 4, kMmRuns = 20;  // the fastest again, in interleaved rounds of so many runs
template <class F>
inline bool mm_time(F&& launch, int reps, hipEvent_t e0, hipEvent_t e1, hipStream_t st, float* ms) {
  if (!launch(reps - 1)) return false;
  mm_hold_kernel<<<1, 1, 0, st>>>(1500u * (unsigned)reps);  // 15 us a run
  bool ok = hipEventRecord(e0, st) == hipSuccess;
  for (int r = 0; r < reps && ok; ++r) ok = launch(r);
  ok = hipEventRecord(e1, st) == hipSuccess && ok;
  ok = hipEventSynchronize(e1) == hipSuccess && ok && hipEventElapsedTime(ms, e0, e1) == hipSuccess;
  *ms /= (float)reps;
  return ok;
}

// The tile and the K split of one product, and whether W comes from HBM (MmArgs::cold): a product is launched as
// it was timed.
struct MmPlan {
  int cfg = -1, split = 1, cold = 0;
  float ms = 1e30f;  // time of the product alone
};

// Operands for timing: normal values, as activations and weights are.  Zeros will not do: they switch little in the
// matrix cores, so a large tile keeps a clock that it does not have in use (gate|up and its GeGLU, M = 1024: 87 us
// on zeros, 102 on values of four exponents, 105 on normal ones; tiles up to 128 x 128: the same).  On zeros
// down_proj at 968 rows took 192 x 256 (62 us on random values) in place of 256 x 192 (59).
static __global__ __launch_bounds__(256) void mm_random_kernel(u16* p, size_t n, float std) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    uint64_t h = (i + 1) * 0x9e3779b97f4a7c15ull;
    h = (h ^ (h >> 32)) * 0xd6e8feb86659fd93ull;
    h ^= h >> 32;
    const float u = ((float)(h & 0xffffff) + 0.5f) * 0x1p-24f, v = (float)((h >> 24) & 0xffffff) * 0x1p-24f;
    p[i] = f2bf(std * sqrtf(-2.0f * __logf(u)) * __cosf(6.2831853f * v));
  }
}
inline bool mm_random(u16* p, size_t n, float std, hipStream_t st) {
  mm_random_kernel<<<4096, 256, 0, st>>>(p, n, std);
  return hipGetLastError() == hipSuccess;
}

// The fastest tile and K split for a product: every tile with every split in [smin, smax] that leaves a split
// at least 4 k-tiles, timed on the caller's buffers (random values: see mm_random_kernel) as the layer loop runs
// them (run r reads the weights at a.W + (r mod w_count) * w_stride bytes, so from beyond the L2s), the fastest
// again.  Timed rather than computed from the sizes because two effects of equal size decide: how evenly the tiles fill 256 CUs (M = 768, N =
// 4304: 128 x 128 12.6 us, 128 x 96 19.6 us) and the copies per MFMA (M = 968, N = 32768: 256 x 256 115 us,
// 128 x 128 166 us).  split_ms: what the reader of the partial sums pays per split.
inline bool mm_tune(MmArgs a, int epi, int smin, int smax, float split_ms, size_t w_stride, int w_count, hipStream_t st, MmPlan* out) {
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return false;
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return false;
  }
  const u16* w = a.W;
  auto time = [&](const MmPlan& c, int reps, float* ms) {
    a.split = c.split;
    auto launch = [&](int r) {
      a.W = w + (size_t)(r % w_count) * (w_stride / 2);
      return mm_launch(c.cfg, epi, a, st);
    };
    return mm_time(launch, reps, e0, e1, st, ms);
  };
  std::vector<std::pair<float, MmPlan>> c;
  bool ok = true;
  MmPlan warm;
  warm.cfg = kMm128x128, warm.split = smin;
  float ms0 = 0.f;
  ok = time(warm, 40, &ms0);  // the clock ramps up here
  for (int cfg = 0; cfg < kMmCfgs && ok; ++cfg)
    for (int s = smin; s <= smax && ok; ++s) {
      MmPlan p;
      p.cfg = cfg, p.split = a.split = s, p.cold = a.cold;
      a.W = w;
      if (!mm_fits(cfg, epi, a) || (s > 1 && a.K / 64 / s < 4)) continue;
      ok = time(p, 6, &p.ms);
      c.emplace_back(p.ms + split_ms * (float)s, p);
    }
  std::sort(c.begin(), c.end(), [](const auto& x, const auto& y) { return x.first < y.first; });
  const size_t n = std::min<size_t>(c.size(), kMmFinalists);
  for (size_t i = 0; i < n; ++i) c[i].second.ms = 1e30f;
  for (int round = 0; round < kMmRounds && ok; ++round)
    for (size_t i = 0; i < n && ok; ++i) {
      float ms = 0.f;
      ok = time(c[i].second, kMmRuns, &ms);
      c[i].second.ms = std::min(c[i].second.ms, ms);
    }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *out = MmPlan{};
  float best = 1e30f;
  for (size_t i = 0; i < n; ++i)
    if (c[i].second.ms + split_ms * (float)c[i].second.split < best) best = c[i].second.ms + split_ms * (float)c[i].second.split, *out = c[i].second;
  return ok && n > 0;
}

}  // namespace pi05
