// The pi0.5 vision tower on gfx950: SigLIP So400m/14 + PaliGemma's projector (get_image_features,
// gemma_pytorch.py:106-107; the tower itself is transformers' SiglipVisionModel).  Per image:
//   h = bf16(conv + bpatch + pos)              patch_embed_kernel (fp32 MFMA straight from the pixels)
//   27 x [ n = LN1(h); q|k|v = n.W^T + b      product (bias epilogue)
//          attention, 16 heads of 72          vision_attn_kernel (MFMA, K/V staged in LDS)
//          h = bf16(h + o.Wo^T + bo); n = LN2 product (split-K when faster) + layernorm_kernel
//          a = gelu_tanh(n.W1^T + b1)          product (bias and GELU epilogue)
//          h = bf16(h + a.W2^T + b2) ]         product (split-K when faster) + layernorm_kernel
//                                              (the next LN1 / post_layernorm)
//   out = (n.Wproj^T + bproj) * out_scale     product (+ scale_kernel)
// The bf16 products run on pi05_mm.h; above kVLibRows rows q|k|v, out_proj, fc2 and the projector on
// hipBLASLt where it measured faster when the context was created.
#include <hip/hip_runtime.h>
#include <hipblaslt/hipblaslt.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "pi05_blocks.h"
#include "pi05_gemm.h"
#include "pi05_mm.h"
#include "pi05_siglip.h"

namespace pi05 {
namespace {

constexpr int kVW = 1152, kVH = 16, kVD = 72, kVI = 4304, kVPatch = 14, kVImg = 224, kVC = 3, kVProj = 2048;
// the MLP's hidden dim padded to 4352 = 64 x 68 in the fc1 output and the fc2 weight rows (the pad
// columns stay zero: gelu(0) = 0 and zero products add exactly nothing), so fc2 splits into 4 or 8
// K slices of 16-byte-aligned width
constexpr int kVIp = 4352;
constexpr int kVGrid = kVImg / kVPatch, kVS = kVGrid * kVGrid;  // 16 x 16 = 256 patches
constexpr int kVPD = kVC * kVPatch * kVPatch;                   // 588 values per patch
constexpr int kVQkvN = 3 * kVW;                                 // 3456 fused q|k|v columns
constexpr int kVDt = 5;  // d-tiles of 16 of P.V, the last one half used
// per-layer packed bf16 weights: [Wq; Wk; Wv] | Wo | W1 | W2; fp32 parameters: bqkv | bo | b1 | b2 |
// ln1w | ln1b | ln2w | ln2b
constexpr size_t kVOffQkv = 0, kVOffO = kVOffQkv + (size_t)kVQkvN * kVW, kVOff1 = kVOffO + (size_t)kVW * kVW,
                 kVOff2 = kVOff1 + (size_t)kVI * kVW, kVLayerElems = kVOff2 + (size_t)kVW * kVIp;
constexpr size_t kVPOffBqkv = 0, kVPOffBo = kVQkvN, kVPOffB1 = kVPOffBo + kVW, kVPOffB2 = kVPOffB1 + kVI,
                 kVPOffLn1w = kVPOffB2 + kVW, kVPOffLn1b = kVPOffLn1w + kVW, kVPOffLn2w = kVPOffLn1b + kVW,
                 kVPOffLn2b = kVPOffLn2w + kVW, kVLayerParams = kVPOffLn2b + kVW;
constexpr size_t kVWorkspace = 32ull << 20;  // hipBLASLt's, where it is a candidate
constexpr int kVMaxSplits = 8;  // K splits of out_proj and fc2 at most
// Rows up to which the products run on pi05_mm.h alone, without a hipBLASLt candidate: a layer's products are faster
// here in sum (us, here / library: 256 rows q|k|v 7.5 / 7.9, out_proj 5.5 / 6.7, fc2 8.7 / 14.0; 768 rows 11.8 / 11.4, 7.3 / 7.8,
// 14.2 / 17.0; 1024 rows 14.5 / 13.2, 8.5 / 9.1, 17.6 / 21.5; the projector within 6 %), and a context is there in 0.15 s
// instead of 0.6.  Above, the library gains (1280 rows: q|k|v 23 / 16; 6144 rows: 59 / 55 and out_proj 28 / 21).
constexpr int kVLibRows = 1024;

thread_local std::string g_vision_err;

// Attention operands in LDS, per (image, head), rows as they come from the q|k|v product: V rows of 72 head
// dims, then K rows of 72 dims, 8 zeros (what the third d-step of Q.K^T reads past dim 71) and 8 of padding.
// Pitches of 144 and 176 bytes spread the 16 rows of a fragment read evenly over the banks, and the whole is 80 KiB:
// two workgroups a CU.
constexpr int kVVPitch = kVD, kVKPitch = 88, kVAttnLds = kVS * (kVVPitch + kVKPitch);  // in bf16 elements

// h = bf16(conv + patch bias + position embedding) (SiglipVisionEmbeddings, fp32 until here), the 14 x 14 patch
// convolution as an fp32 MFMA product straight from the pixels: h[(n, 16 py + px)][o] sums pixels[n][c][14 py +
// ky][14 px + kx] W[o][c 196 + ky 14 + kx], W packed by pack_patch_kernel (1 KiB a wave load: 64-byte pieces of W's
// own rows took four times as long to load).  Workgroup = 64 output channels, one 16-channel tile a wave, for every
// stride-th patch row of 16 patches: its weights stay in registers, and a patch row's pixels (14 whole image rows a
// channel, contiguous) go to LDS as they are, the next patch row's while this one is multiplied.  Lane l holds
// four consecutive k of channel l % 16, so the four MFMAs of a 16-wide step take k = 16 S + 4 (l / 16) + j; s_off
// gives the LDS offset of each k within a patch.  Bound by the fp32 matrix rate (157 TFLOP/s: 2.2 us an image).
// Against im2col, a library product and an embedding pass (us): 1 image 21 -> 13, 3 images 28 -> 20, 24 images 104 -> 98.
constexpr int kVSteps = (kVPD + 15) / 16, kVRowPix = kVPatch * kVImg;  // 37 steps; 3136 pixels of a patch row and channel

// wp[o / 16][k / 16][lane][4]: lane l holds k = 16 s + 4 (l / 16) .. + 3 of channel l % 16, zeros from k = 588
__global__ __launch_bounds__(256) void pack_patch_kernel(const float* w, float* wp) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kVW / 16 * kVSteps * 256) return;
  const int j = i & 3, l = (i >> 2) & 63, s = (i >> 8) % kVSteps, ot = (i >> 8) / kVSteps, k = s * 16 + (l >> 4) * 4 + j;
  wp[i] = k < kVPD ? w[(size_t)(ot * 16 + (l & 15)) * kVPD + k] : 0.f;
}

__global__ __launch_bounds__(256) void patch_embed_kernel(const float* px, const float* w, const float* pb, const float* pos, u16* h,
                                                          int rows, int stride) {
#ifdef __HIP_DEVICE_COMPILE__
  // two arrays, not one of two: the compiler then knows that a copy into the one leaves the other alone
  __shared__ __align__(16) float s_pa[kVC * kVRowPix], s_pb[kVC * kVRowPix];
  __shared__ __align__(16) uint16_t s_off[kVSteps * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
  constexpr int kNt = kVW / 64;
  const int o0 = ((int)blockIdx.x % kNt) * 64 + wave * 16;
  const bool vec = reinterpret_cast<uintptr_t>(px) % 16 == 0;  // a patch row's pixels are 12544 bytes: aligned as px is
  auto stage = [&](int row, float* buf) {  // patch row `row` (16 an image)
    const float* src = px + ((size_t)(row / kVGrid) * kVC * kVImg + (row % kVGrid) * kVPatch) * kVImg;
    if (vec) {
#pragma unroll
      for (int c = 0; c < kVC; ++c)
#pragma unroll
        for (int i = 0; i < (kVRowPix + 1023) / 1024; ++i) {
          const int at = i * 1024 + wave * 256;
          if (at + lane * 4 < kVRowPix)
            __builtin_amdgcn_global_load_lds(const_cast<float*>(src) + (size_t)c * kVImg * kVImg + at + lane * 4,
                                             (__attribute__((address_space(3))) float*)buf + c * kVRowPix + at, 16, 0, 0);
        }
    } else {
      for (int c = 0; c < kVC; ++c)
        for (int i = tid; i < kVRowPix; i += 256) buf[c * kVRowPix + i] = src[(size_t)c * kVImg * kVImg + i];
    }
  };
  int row = (int)blockIdx.x / kNt;
  stage(row, s_pa);
  f32x4 wf[kVSteps];
  const float* wr = w + (size_t)(o0 / 16) * kVSteps * 256 + lane * 4;
#pragma unroll
  for (int s = 0; s < kVSteps; ++s) wf[s] = *reinterpret_cast<const f32x4*>(wr + s * 256);
  for (int k = tid; k < kVSteps * 16; k += 256) {
    const int c = k / (kVPatch * kVPatch), ky = k / kVPatch % kVPatch;
    s_off[k] = (uint16_t)(k < kVPD ? c * kVRowPix + ky * kVImg + k % kVPatch : 0);
  }
  const int o = o0 + g * 4;
  const f32x4 bias = *reinterpret_cast<const f32x4*>(pb + o);
  auto patch_row = [&](float* cur, float* other) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies of the patch row
    __syncthreads();                                  // every wave's; and the other buffer is no longer read
    if (row + stride < rows) stage(row + stride, other);
    const float* pr = cur + r * kVPatch;
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int s = 0; s < kVSteps; ++s) {
      const u16x4 off = *reinterpret_cast<const u16x4*>(s_off + s * 16 + g * 4);
#pragma unroll
      for (int p = 0; p < 2; ++p) {  // an even k and the next one are neighbours in a patch's row (14 is even)
        float2 v = *reinterpret_cast<const float2*>(pr + off[2 * p]);
        if (s * 16 + 16 > kVPD && s * 16 + g * 4 >= kVPD) v = float2{0.f, 0.f};
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[s][2 * p], v.x, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[s][2 * p + 1], v.y, acc[1], 0, 0, 0);
      }
    }
    // lane l: channels o0 + 4 (l / 16) .. + 3 of patch l % 16
    const int t = row * kVGrid + r;
    const f32x4 ps = *reinterpret_cast<const f32x4*>(pos + (size_t)(t % kVS) * kVW + o);
    u16x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = f2bf(fadd(fadd(fadd(acc[0][i], acc[1][i]), bias[i]), ps[i]));
    *reinterpret_cast<u16x4*>(h + (size_t)t * kVW + o) = v;
    row += stride;
  };
  while (row < rows) {
    patch_row(s_pa, s_pb);
    if (row < rows) patch_row(s_pb, s_pa);
  }
#endif
}

// h = bf16(x + y), n = bf16((h - mean) / sqrt(var + eps) * w + b) with fp32 statistics
// (nn.LayerNorm after the residual add).  y is the bf16 Linear output, or (ys != null) the Linear
// as nsplit fp32 split-K partials reduced here: y = bf16(sum + ybias); neither: h = x.  One wave
// per 1152-wide row (9 pairs of bf16 per lane), 4 rows per workgroup.
__global__ __launch_bounds__(256) void layernorm_kernel(const u16* x, const u16* y, const float* ys, int nsplit, size_t split_stride,
                                                       const float* ybias, const float* w, const float* b, u16* h_out, u16* n_out,
                                                       float eps, int rows) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= rows) return;
  const size_t ro = (size_t)row * kVW;
  // every load of the row is issued before the first use, the norm's weight and bias included
  float2 wv[9], bv[9];
#pragma unroll
  for (int j = 0; j < 9; ++j) {
    wv[j] = *reinterpret_cast<const float2*>(w + 2 * (lane + 64 * j));
    bv[j] = *reinterpret_cast<const float2*>(b + 2 * (lane + 64 * j));
  }
  uint32_t xv[9];
#pragma unroll
  for (int j = 0; j < 9; ++j) xv[j] = *reinterpret_cast<const uint32_t*>(x + ro + 2 * (lane + 64 * j));
  float h[18];
#pragma unroll
  for (int j = 0; j < 9; ++j) h[2 * j] = bf2f((u16)(xv[j] & 0xffff)), h[2 * j + 1] = bf2f((u16)(xv[j] >> 16));
  if (ys) {
    // every split's partial row is loaded before the first sum (the splits are summed in order, as
    // before): a loop that waited for each split's loads in turn paid one memory round trip per split
    float2 acc[9], a[kVMaxSplits - 1][9], yb[9];
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      acc[j] = *reinterpret_cast<const float2*>(ys + ro + 2 * (lane + 64 * j));
      yb[j] = *reinterpret_cast<const float2*>(ybias + 2 * (lane + 64 * j));
    }
#pragma unroll
    for (int sp = 1; sp < kVMaxSplits; ++sp)
      if (sp < nsplit)
#pragma unroll
        for (int j = 0; j < 9; ++j) a[sp - 1][j] = *reinterpret_cast<const float2*>(ys + (size_t)sp * split_stride + ro + 2 * (lane + 64 * j));
#pragma unroll
    for (int sp = 1; sp < kVMaxSplits; ++sp)
      if (sp < nsplit)
#pragma unroll
        for (int j = 0; j < 9; ++j) acc[j].x += a[sp - 1][j].x, acc[j].y += a[sp - 1][j].y;
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      h[2 * j] = round_bf(fadd(h[2 * j], round_bf(fadd(acc[j].x, yb[j].x))));
      h[2 * j + 1] = round_bf(fadd(h[2 * j + 1], round_bf(fadd(acc[j].y, yb[j].y))));
    }
  } else if (y) {
    uint32_t yv[9];
#pragma unroll
    for (int j = 0; j < 9; ++j) yv[j] = *reinterpret_cast<const uint32_t*>(y + ro + 2 * (lane + 64 * j));
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      h[2 * j] = round_bf(fadd(h[2 * j], bf2f((u16)(yv[j] & 0xffff))));
      h[2 * j + 1] = round_bf(fadd(h[2 * j + 1], bf2f((u16)(yv[j] >> 16))));
    }
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 18; ++i) s += h[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  const float mean = s * (1.0f / kVW);
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < 18; ++i) q += (h[i] - mean) * (h[i] - mean);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o);
  const float rstd = 1.0f / sqrtf(q * (1.0f / kVW) + eps);
  const bool write_h = (y || ys) && h_out;
#pragma unroll
  for (int j = 0; j < 9; ++j) {
    const int e = 2 * (lane + 64 * j);
    const u16 n0 = f2bf(fadd(fmul(fmul(fsub(h[2 * j], mean), rstd), wv[j].x), bv[j].x));
    const u16 n1 = f2bf(fadd(fmul(fmul(fsub(h[2 * j + 1], mean), rstd), wv[j].y), bv[j].y));
    *reinterpret_cast<uint32_t*>(n_out + ro + e) = (uint32_t)n0 | ((uint32_t)n1 << 16);
    if (write_h) *reinterpret_cast<uint32_t*>(h_out + ro + e) = (uint32_t)f2bf(h[2 * j]) | ((uint32_t)f2bf(h[2 * j + 1]) << 16);
  }
}

// MHA over one image's 256 patches, straight from the fused q|k|v product [M, 3456]: workgroup =
// (image, head, half of the queries), wave w = query m-tile 8 half + w over all 256 keys.  Scores are fp32
// (no bf16 rounding of the scores: the reference runs SDPA's flash kernel); all of a query's 256 scores fit
// the wave's registers, so the softmax is one pass (one maximum, one sum, no rescaling of O), and P is rounded
// to bf16 for P.V.  S^T = K Q^T leaves a lane the keys 4 (l / 16) .. + 3 of a key tile, which is the P^T operand's
// order once V's fragments take the same keys: ds_read_b64_tr_b16 reads them transposed from V's rows (lane i of
// 16 points at 4 dims of key i / 4 and gets dim i of the 4 keys).
// Bound by latency (a chain of load, LDS, MFMA, exp): two workgroups a CU hide it where there are enough.
// 1 image 9.9 -> 7.7 us, 24 images 38 -> 25.8 us against the online softmax over V fragments scattered by 2-byte stores.
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 4))) void vision_attn_kernel(const u16* qkv, u16* out) {
#ifdef __HIP_DEVICE_COMPILE__
  __shared__ __align__(16) u16 s_kv[kVAttnLds];
  u16 *s_v = s_kv, *s_k = s_kv + kVS * kVVPitch;
  const int half = blockIdx.x & 1, head = (blockIdx.x >> 1) % kVH, n = (blockIdx.x >> 1) / kVH;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, mt = half * 8 + wave, r = lane & 15, g = lane >> 4;
  const u16* base = qkv + (size_t)n * kVS * kVQkvN + head * kVD;  // row i of the image: q | k | v at +0 | +W | +2W
  constexpr int kChunks = kVS * (kVD / 8), kPass = (kChunks + 511) / 512;  // 16-byte chunks of K (of V)
  u16x8 kc[kPass], vc[kPass];
#pragma unroll
  for (int t = 0; t < kPass; ++t) {
    const int i = t * 512 + tid;
    if (i < kChunks) {
      const u16* src = base + (size_t)(i / 9) * kVQkvN + (i % 9) * 8;
      kc[t] = *reinterpret_cast<const u16x8*>(src + kVW);
      vc[t] = *reinterpret_cast<const u16x8*>(src + 2 * kVW);
    }
  }
  // B operand of S^T: query r, dims 32 ds + 8 g .. + 7 (zero from 72)
  const u16* qrow = base + (size_t)(mt * 16 + r) * kVQkvN;
  const bf16x8 q0 = load_frag(qrow + g * 8), q1 = load_frag(qrow + 32 + g * 8);
  const bf16x8 q2 = g == 0 ? load_frag(qrow + 64) : zero_frag();
#pragma unroll
  for (int t = 0; t < kPass; ++t) {
    const int i = t * 512 + tid;
    if (i < kChunks) {
      *reinterpret_cast<u16x8*>(s_k + (i / 9) * kVKPitch + (i % 9) * 8) = kc[t];
      *reinterpret_cast<u16x8*>(s_v + i * 8) = vc[t];
    }
  }
  if (tid < kVS) *reinterpret_cast<u16x8*>(s_k + tid * kVKPitch + kVD) = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
  __syncthreads();
  f32x4 s[kVS / 16];
#pragma unroll
  for (int kt = 0; kt < kVS / 16; ++kt) {
    const u16* k = s_k + (kt * 16 + r) * kVKPitch;
    f32x4 acc = mfma16x16x32(load_frag(k + g * 8), q0, f32x4{0.f, 0.f, 0.f, 0.f});
    acc = mfma16x16x32(load_frag(k + 32 + g * 8), q1, acc);
    s[kt] = mfma16x16x32(load_frag(k + (g == 0 ? 64 : kVD)), q2, acc);  // every group past the row's end: its zeros
  }
  float m = s[0][0];
#pragma unroll
  for (int kt = 0; kt < kVS / 16; ++kt)
#pragma unroll
    for (int i = 0; i < 4; ++i) m = fmaxf(m, s[kt][i]);
  m = lane_max_xor32(lane_max_xor16(m));
  // exp((s - m) 72^-0.5) as exp2
  const float c = 0.11785113019775793f * 1.4426950408889634f;
  float l = 0.f;
  bf16x8 p[kVS / 32];
#pragma unroll
  for (int kb = 0; kb < kVS / 32; ++kb) {
    u16x8 pf;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = __builtin_amdgcn_exp2f((s[2 * kb + j / 4][j % 4] - m) * c);
      l += e;
      pf[j] = f2bf(e);
    }
    p[kb] = as_bf16x8(pf);
  }
  l = lane_sum_xor32(lane_sum_xor16(l));
  const float inv = 1.0f / l;
  // A operand of O^T = V^T P^T: keys 4 g .. + 3 and 16 + 4 g .. + 3 of block kb, dim 16 dt + r (dims past 71 read
  // what follows the row; their rows of O^T are not stored)
  const u16* vl = s_v + (4 * g + (r >> 2)) * kVVPitch + (r & 3) * 4;
  f32x4 o[kVDt];
#pragma unroll
  for (int dt = 0; dt < kVDt; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < kVS / 32; ++kb)
#pragma unroll
    for (int dt = 0; dt < kVDt; ++dt) {
      const u16* v = vl + kb * 32 * kVVPitch + dt * 16;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)v);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(v + 16 * kVVPitch));
      u16x8 f;
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = (u16)lo[j], f[4 + j] = (u16)hi[j];
      o[dt] = mfma16x16x32(as_bf16x8(f), p[kb], o[dt]);
    }
  u16* orow = out + ((size_t)n * kVS + mt * 16 + r) * kVW + head * kVD + g * 4;
#pragma unroll
  for (int dt = 0; dt < kVDt; ++dt)
    if (dt * 16 + g * 4 < kVD)
      *reinterpret_cast<u16x4*>(orow + dt * 16) = u16x4{f2bf(o[dt][0] * inv), f2bf(o[dt][1] * inv), f2bf(o[dt][2] * inv), f2bf(o[dt][3] * inv)};
#endif
}

__global__ __launch_bounds__(256) void scale_kernel(u16* x, size_t total, float s) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) x[i] = f2bf(bf2f(x[i]) * s);
}

__global__ __launch_bounds__(256) void bf16_to_f32_kernel(const u16* src, float* dst, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = bf2f(src[i]);
}

struct VLayerBind {
  const void* p[16] = {};  // wq bq wk bk wv bv wo bo w1 b1 w2 b2 ln1w ln1b ln2w ln2b
};

struct VisionPlan {
  int L = 0, N = 0, M = 0, cold = 0;
  size_t w, par, head, h, qkv, act, part, ws;
  size_t total() const { return w + par + head + 4 * h + qkv + act + part + ws + 16 * 256; }
};

size_t vrup(size_t x) { return (x + 255) / 256 * 256; }

VisionPlan vplan_of(const pi05_vision_dims& d) {
  VisionPlan p;
  p.L = d.depth, p.N = d.n_images, p.M = d.n_images * kVS;
  const size_t M = p.M;
  p.w = vrup((size_t)p.L * kVLayerElems * 2);
  p.cold = mm_cold(p.w);
  p.par = vrup((size_t)p.L * kVLayerParams * 4);
  // heads: packed patch_w + patch_b + pos [256, W] + post w/b (fp32), proj_w bf16, proj_b fp32
  p.head = vrup(((size_t)kVW * kVSteps * 16 + kVW + (size_t)kVS * kVW + 2 * kVW + kVProj) * 4 + (size_t)kVProj * kVW * 2);
  p.h = vrup(M * kVW * 2);
  p.qkv = vrup(M * kVQkvN * 2);
  p.part = vrup((size_t)kVMaxSplits * M * kVW * 4);
  p.act = vrup(M * kVIp * 2);
  p.ws = p.M > kVLibRows ? kVWorkspace : 0;
  return p;
}

bool check_vision_dims(const pi05_vision_dims* d, std::string* m) {
  if (!d) {
    *m = "dims is NULL";
    return false;
  }
  if (d->width != kVW || d->num_heads != kVH || d->mlp_dim != kVI || d->patch != kVPatch || d->image != kVImg || d->channels != kVC ||
      d->proj_dim != kVProj) {
    *m = "vision geometry must be width 1152, 16 heads, mlp_dim 4304, patch 14, image 224, 3 channels, proj_dim 2048";
    return false;
  }
  if (d->depth < 1 || d->depth > 64 || d->n_images < 1 || d->n_images > 64) {
    *m = "depth must be in [1, 64] and n_images in [1, 64]";
    return false;
  }
  if (!(d->ln_eps > 0.f) || !(d->out_scale > 0.f)) {
    *m = "ln_eps and out_scale must be > 0";
    return false;
  }
  return true;
}

unsigned grid_for(size_t total) {
  const size_t g = (total + 255) / 256;
  return (unsigned)(g < 8192 ? g : 8192);
}

}  // namespace
}  // namespace pi05

using namespace pi05;

struct pi05_vision_ctx {
  pi05_vision_dims d{};
  VisionPlan plan;
  std::string err;
  std::vector<VLayerBind> binds;
  const float *b_patch_w = nullptr, *b_patch_b = nullptr, *b_pos = nullptr;
  const void *b_post_w = nullptr, *b_post_b = nullptr, *b_proj_w = nullptr, *b_proj_b = nullptr;
  bool refreshed = false;
  char* base = nullptr;
  u16 *w = nullptr, *h = nullptr, *n = nullptr, *y = nullptr, *attn = nullptr, *qkv = nullptr, *act = nullptr, *proj_w = nullptr;
  float *par = nullptr, *patch_w = nullptr, *patch_b = nullptr, *pos = nullptr, *post_w = nullptr, *post_b = nullptr, *proj_b = nullptr,
        *part = nullptr;
  void* ws = nullptr;
  hipblasLtHandle_t lt = nullptr;
  // the bf16 products: on pi05_mm.h, or (above kVLibRows rows, where it measured faster) on hipBLASLt
  GemmPlan g_qkv, g_o, g_fc2, g_proj;
  MmPlan m_qkv, m_o, m_fc1, m_fc2, m_proj;
  bool lib_qkv = false, lib_o = false, lib_fc2 = false, lib_proj = false;
};

namespace {

int vfail(pi05_vision_ctx* c, int code, const std::string& m) {
  if (c) c->err = m;
  else g_vision_err = m;
  return code;
}

int vgemm(pi05_vision_ctx* c, const GemmPlan& p, const void* W, const void* A, void* C, const float* bias, hipStream_t st) {
  const hipblasStatus_t s = run_plan(c->lt, p, p.algo, p.ws, W, A, C, bias, c->ws, st);
  if (!lt_ok(s)) return vfail(c, PI05_E_HIP, "hipblasLtMatmul failed (status " + std::to_string((int)s) + ")");
  return PI05_OK;
}

int vmm(pi05_vision_ctx* c, const MmPlan& p, int epi, MmArgs a, hipStream_t st) {
  a.split = p.split;
  a.cold = p.cold;
  if (!mm_launch(p.cfg, epi, a, st)) return vfail(c, PI05_E_HIP, "product launch failed");
  return PI05_OK;
}

}  // namespace

extern "C" {

void pi05_vision_default_dims(pi05_vision_dims* d) {
  if (!d) return;
  *d = pi05_vision_dims{kVW, 27, kVH, kVI, kVPatch, kVImg, kVC, kVProj, 3, 1e-6f, 1.0f};
}

int pi05_vision_check_dims(const pi05_vision_dims* dims) {
  std::string m;
  if (!check_vision_dims(dims, &m)) return vfail(nullptr, PI05_E_INVALID, m);
  return PI05_OK;
}

size_t pi05_vision_device_bytes(const pi05_vision_dims* dims) {
  std::string m;
  if (!check_vision_dims(dims, &m)) return 0;
  return vplan_of(*dims).total();
}

const char* pi05_vision_last_error(const pi05_vision_ctx* ctx) { return ctx ? ctx->err.c_str() : g_vision_err.c_str(); }

int pi05_vision_create(const pi05_vision_dims* dims, pi05_vision_ctx** out) {
  if (!out) return vfail(nullptr, PI05_E_INVALID, "out is NULL");
  *out = nullptr;
  std::string m;
  if (!check_vision_dims(dims, &m)) return vfail(nullptr, PI05_E_INVALID, m);
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return vfail(nullptr, PI05_E_NODEVICE, std::string("no HIP device: ") + hipGetErrorString(e));
  hipDeviceProp_t prop;
  e = hipGetDeviceProperties(&prop, dev);
  if (e != hipSuccess || strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return vfail(nullptr, PI05_E_NODEVICE, std::string("device is not gfx950 (MI355X): ") + (e == hipSuccess ? prop.gcnArchName : hipGetErrorString(e)));
  pi05_vision_ctx* c = new pi05_vision_ctx();
  c->d = *dims;
  c->plan = vplan_of(*dims);
  c->binds.resize(dims->depth);
  const VisionPlan& p = c->plan;
  e = hipMalloc(&c->base, p.total());
  if (e != hipSuccess) {
    delete c;
    return vfail(nullptr, PI05_E_NOMEM, std::string("vision context allocation failed: ") + hipGetErrorString(e));
  }
  char* q = c->base;
  auto take = [&](size_t bytes) {
    char* r = q;
    q += bytes;
    return r;
  };
  c->w = reinterpret_cast<u16*>(take(p.w));
  c->par = reinterpret_cast<float*>(take(p.par));
  char* hd = take(p.head);
  c->patch_w = reinterpret_cast<float*>(hd);
  c->patch_b = c->patch_w + (size_t)kVW * kVSteps * 16;
  c->pos = c->patch_b + kVW;
  c->post_w = c->pos + (size_t)kVS * kVW;
  c->post_b = c->post_w + kVW;
  c->proj_b = c->post_b + kVW;
  c->proj_w = reinterpret_cast<u16*>(c->proj_b + kVProj);
  c->h = reinterpret_cast<u16*>(take(p.h));
  c->n = reinterpret_cast<u16*>(take(p.h));
  c->y = reinterpret_cast<u16*>(take(p.h));
  c->attn = reinterpret_cast<u16*>(take(p.h));
  c->qkv = reinterpret_cast<u16*>(take(p.qkv));
  c->act = reinterpret_cast<u16*>(take(p.act));
  c->part = reinterpret_cast<float*>(take(p.part));
  c->ws = p.ws ? take(p.ws) : nullptr;
  // defined values wherever the tuning below reads (zero biases)
  e = hipMemset(c->base, 0, p.total());
  if (e != hipSuccess) {
    hipFree(c->base);
    delete c;
    return vfail(nullptr, PI05_E_HIP, std::string("vision context initialisation failed: ") + hipGetErrorString(e));
  }
  std::string perr;
  const int M = p.M;
  GemmOpts bias;
  bias.bias = true;
  GemmOpts fc2o = bias;
  fc2o.ld_k = kVIp;
  const bool lib = p.ws != 0;
  bool ok = !lib || (lt_ok(hipblasLtCreate(&c->lt)) && make_plan(c->lt, M, kVQkvN, kVW, kVWorkspace, &c->g_qkv, &perr, bias) &&
                     make_plan(c->lt, M, kVW, kVW, kVWorkspace, &c->g_o, &perr, bias) && make_plan(c->lt, M, kVW, kVIp, kVWorkspace, &c->g_fc2, &perr, fc2o) &&
                     make_plan(c->lt, M, kVProj, kVW, kVWorkspace, &c->g_proj, &perr, bias));
  if (ok) {
    const float* bz = c->par;  // any fp32 vector long enough (zeros) stands in for the biases while timing
    // (weights rotate over the layers' blocks while timing, as the layer loop streams them; the projector's too:
    // the tower's weights have passed through the caches since its own were read)
    static_assert((size_t)kVProj * kVW <= kVLayerElems, "the projector is timed on the layers' blocks");
    const size_t ls = kVLayerElems * 2;
    const int nl = p.L;
    // what a reader of fp32 partials pays per split: 4 bytes per output element at ~4 TB/s, less the
    // bf16 output it would read and the product write otherwise
    const float part_ms = (float)(4.0 * M * kVW / 4e12 * 1e3), bf_ms = (float)(2.0 * M * kVW / 4e12 * 1e3);
    ok = mm_random(c->w, (size_t)nl * kVLayerElems, 0.02f, nullptr) && mm_random(c->n, M * (size_t)kVW, 1.f, nullptr) &&
         mm_random(c->attn, M * (size_t)kVW, 1.f, nullptr) && mm_random(c->act, M * (size_t)kVIp, 1.f, nullptr) &&
         mm_tune({c->n, c->w, c->qkv, bz, M, kVQkvN, kVW, kVW, kVW, kVQkvN, 1, p.cold}, kMmBf16, 1, 1, 0.f, ls, nl, nullptr, &c->m_qkv) &&
         mm_tune({c->n, c->w, c->act, bz, M, kVI, kVW, kVW, kVW, kVIp, 1, p.cold}, kMmGelu, 1, 1, 0.f, ls, nl, nullptr, &c->m_fc1) &&
         mm_tune({c->n, c->w, c->act, bz, M, kVProj, kVW, kVW, kVW, kVProj, 1, p.cold}, kMmBf16, 1, 1, 0.f, ls, nl, nullptr, &c->m_proj);
    // out_proj and fc2: one product with its bias, or fp32 K splits that the LayerNorm adds
    auto tune_n = [&](const u16* A, int K, MmPlan* out) {
      MmPlan one, sp;
      if (!mm_tune({A, c->w, c->y, bz, M, kVW, K, K, K, kVW, 1, p.cold}, kMmBf16, 1, 1, 0.f, ls, nl, nullptr, &one) ||
          !mm_tune({A, c->w, c->part, nullptr, M, kVW, K, K, K, kVW, 1, p.cold}, kMmF32, 2, kVMaxSplits, part_ms, ls, nl, nullptr, &sp))
        return false;
      *out = sp.ms + part_ms * (float)sp.split - bf_ms < one.ms ? sp : one;
      return true;
    };
    ok = ok && tune_n(c->attn, kVW, &c->m_o) && tune_n(c->act, kVIp, &c->m_fc2);
    if (ok && lib) {
      ok = tune_plan(c->lt, &c->g_qkv, c->w, c->n, c->qkv, c->ws, nullptr, bz, ls, nl) &&
           tune_plan(c->lt, &c->g_o, c->w, c->attn, c->y, c->ws, nullptr, bz, ls, nl) &&
           tune_plan(c->lt, &c->g_fc2, c->w, c->act, c->y, c->ws, nullptr, bz, ls, nl) &&
           tune_plan(c->lt, &c->g_proj, c->w, c->n, c->act, c->ws, nullptr, bz, ls, nl);
      auto cost = [&](const MmPlan& m) { return m.split > 1 ? m.ms + part_ms * (float)m.split - bf_ms : m.ms; };
      c->lib_qkv = c->g_qkv.ms < c->m_qkv.ms;
      c->lib_o = c->g_o.ms < cost(c->m_o);
      c->lib_fc2 = c->g_fc2.ms < cost(c->m_fc2);
      c->lib_proj = c->g_proj.ms < c->m_proj.ms;
    }
    if (!ok && perr.empty()) perr = "GEMM tuning failed";
  }
  if (!ok) {
    if (perr.empty()) perr = "hipblasLtCreate failed";
    pi05_vision_destroy(c);
    return vfail(nullptr, PI05_E_HIP, perr);
  }
  // the columns past 4304 of fc2's operands are read and never written: zero from here on
  e = hipMemset(c->base, 0, p.total());
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    pi05_vision_destroy(c);
    return vfail(nullptr, PI05_E_HIP, std::string("vision context initialisation failed: ") + hipGetErrorString(e));
  }
  *out = c;
  return PI05_OK;
}

int pi05_vision_product(pi05_vision_ctx* c, int which, int32_t* choice, float* us) {
  if (!c) return vfail(nullptr, PI05_E_INVALID, "ctx is NULL");
  if (which < 0 || which > 4 || !choice || !us) return vfail(c, PI05_E_INVALID, "which must be in [0, 4], choice and us non-NULL");
  const MmPlan* const m[5] = {&c->m_qkv, &c->m_o, &c->m_fc1, &c->m_fc2, &c->m_proj};
  const GemmPlan* const g[5] = {&c->g_qkv, &c->g_o, nullptr, &c->g_fc2, &c->g_proj};
  const bool lib[5] = {c->lib_qkv, c->lib_o, false, c->lib_fc2, c->lib_proj};
  choice[0] = m[which]->cfg, choice[1] = m[which]->split, choice[2] = m[which]->cold, choice[3] = lib[which];
  us[0] = m[which]->ms * 1e3f, us[1] = g[which] ? g[which]->ms * 1e3f : 0.f;
  return PI05_OK;
}

int pi05_vision_destroy(pi05_vision_ctx* c) {
  if (!c) return PI05_OK;
  for (GemmPlan* g : {&c->g_qkv, &c->g_o, &c->g_fc2, &c->g_proj})
    free_plan(g);
  if (c->lt) hipblasLtDestroy(c->lt);
  if (c->base) hipFree(c->base);
  delete c;
  return PI05_OK;
}

int pi05_vision_bind_layer(pi05_vision_ctx* c, int layer, const void* wq, const void* bq, const void* wk, const void* bk, const void* wv,
                           const void* bv, const void* wo, const void* bo, const void* w1, const void* b1, const void* w2, const void* b2,
                           const void* ln1_w, const void* ln1_b, const void* ln2_w, const void* ln2_b) {
  if (!c) return vfail(nullptr, PI05_E_INVALID, "ctx is NULL");
  if (layer < 0 || layer >= c->d.depth) return vfail(c, PI05_E_INVALID, "layer out of range");
  const void* ps[16] = {wq, bq, wk, bk, wv, bv, wo, bo, w1, b1, w2, b2, ln1_w, ln1_b, ln2_w, ln2_b};
  VLayerBind b;
  for (int i = 0; i < 16; ++i) {
    if (!ps[i]) return vfail(c, PI05_E_INVALID, "a weight pointer is NULL");
    if (reinterpret_cast<uintptr_t>(ps[i]) % 16) return vfail(c, PI05_E_INVALID, "weight pointers must be 16-byte aligned");
    b.p[i] = ps[i];
  }
  c->binds[layer] = b;
  c->refreshed = false;
  return PI05_OK;
}

int pi05_vision_bind_heads(pi05_vision_ctx* c, const float* patch_w, const float* patch_b, const float* pos, const void* post_w,
                           const void* post_b, const void* proj_w, const void* proj_b) {
  if (!c) return vfail(nullptr, PI05_E_INVALID, "ctx is NULL");
  const void* ps[7] = {patch_w, patch_b, pos, post_w, post_b, proj_w, proj_b};
  for (const void* x : ps) {
    if (!x) return vfail(c, PI05_E_INVALID, "a weight pointer is NULL");
    if (reinterpret_cast<uintptr_t>(x) % 16) return vfail(c, PI05_E_INVALID, "weight pointers must be 16-byte aligned");
  }
  c->b_patch_w = patch_w, c->b_patch_b = patch_b, c->b_pos = pos;
  c->b_post_w = post_w, c->b_post_b = post_b, c->b_proj_w = proj_w, c->b_proj_b = proj_b;
  c->refreshed = false;
  return PI05_OK;
}

int pi05_vision_refresh_weights(pi05_vision_ctx* c, void* stream) {
  if (!c) return vfail(nullptr, PI05_E_INVALID, "ctx is NULL");
  if (!c->b_patch_w) return vfail(c, PI05_E_STATE, "heads are not bound");
  for (int l = 0; l < c->d.depth; ++l)
    if (!c->binds[l].p[0]) return vfail(c, PI05_E_STATE, "layer " + std::to_string(l) + " is not bound");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const hipMemcpyKind k = hipMemcpyDeviceToDevice;
  hipError_t e = hipSuccess;
  auto to_f32 = [&](const void* src, float* dst, size_t n) {
    bf16_to_f32_kernel<<<grid_for(n), 256, 0, st>>>(static_cast<const u16*>(src), dst, n);
  };
  for (int l = 0; l < c->d.depth && e == hipSuccess; ++l) {
    const VLayerBind& b = c->binds[l];
    u16* w = c->w + (size_t)l * kVLayerElems;
    float* pr = c->par + (size_t)l * kVLayerParams;
    const size_t ww = (size_t)kVW * kVW * 2;
    e = hipMemcpyAsync(w + kVOffQkv, b.p[0], ww, k, st);
    if (e == hipSuccess) e = hipMemcpyAsync(w + kVOffQkv + (size_t)kVW * kVW, b.p[2], ww, k, st);
    if (e == hipSuccess) e = hipMemcpyAsync(w + kVOffQkv + (size_t)2 * kVW * kVW, b.p[4], ww, k, st);
    if (e == hipSuccess) e = hipMemcpyAsync(w + kVOffO, b.p[6], ww, k, st);
    if (e == hipSuccess) e = hipMemcpyAsync(w + kVOff1, b.p[8], (size_t)kVI * kVW * 2, k, st);
    if (e == hipSuccess) e = hipMemcpy2DAsync(w + kVOff2, (size_t)kVIp * 2, b.p[10], (size_t)kVI * 2, (size_t)kVI * 2, kVW, k, st);
    to_f32(b.p[1], pr + kVPOffBqkv, kVW);
    to_f32(b.p[3], pr + kVPOffBqkv + kVW, kVW);
    to_f32(b.p[5], pr + kVPOffBqkv + 2 * kVW, kVW);
    to_f32(b.p[7], pr + kVPOffBo, kVW);
    to_f32(b.p[9], pr + kVPOffB1, kVI);
    to_f32(b.p[11], pr + kVPOffB2, kVW);
    to_f32(b.p[12], pr + kVPOffLn1w, kVW);
    to_f32(b.p[13], pr + kVPOffLn1b, kVW);
    to_f32(b.p[14], pr + kVPOffLn2w, kVW);
    to_f32(b.p[15], pr + kVPOffLn2b, kVW);
  }
  if (e == hipSuccess) pack_patch_kernel<<<kVW / 16 * kVSteps, 256, 0, st>>>(c->b_patch_w, c->patch_w);
  if (e == hipSuccess) e = hipMemcpyAsync(c->patch_b, c->b_patch_b, kVW * 4, k, st);
  if (e == hipSuccess) e = hipMemcpyAsync(c->pos, c->b_pos, (size_t)kVS * kVW * 4, k, st);
  if (e == hipSuccess) e = hipMemcpyAsync(c->proj_w, c->b_proj_w, (size_t)kVProj * kVW * 2, k, st);
  if (e == hipSuccess) {
    to_f32(c->b_post_w, c->post_w, kVW);
    to_f32(c->b_post_b, c->post_b, kVW);
    to_f32(c->b_proj_b, c->proj_b, kVProj);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return vfail(c, PI05_E_HIP, std::string("weight packing: ") + hipGetErrorString(e));
  c->refreshed = true;
  return PI05_OK;
}

int pi05_vision_forward(pi05_vision_ctx* c, const float* pixels, void* out, void* stream) {
  if (!c) return vfail(nullptr, PI05_E_INVALID, "ctx is NULL");
  if (!pixels || !out) return vfail(c, PI05_E_INVALID, "pixels and out must be non-NULL");
  if (reinterpret_cast<uintptr_t>(out) % 16) return vfail(c, PI05_E_INVALID, "out must be 16-byte aligned");
  if (!c->refreshed) return vfail(c, PI05_E_STATE, "weights are not bound and refreshed");
  const VisionPlan& p = c->plan;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const float eps = c->d.ln_eps;
  const size_t M = p.M;
  int rc;
  // two workgroups a CU (their LDS): 28 x 18, the patch rows dealt out evenly
  const int rows = p.N * kVGrid, each = (rows + 27) / 28, stride = (rows + each - 1) / each;
  patch_embed_kernel<<<(unsigned)(stride * (kVW / 64)), 256, 0, st>>>(pixels, c->patch_w, c->patch_b, c->pos, c->h, rows, stride);
  const float* pr0 = c->par;
  const unsigned ln_grid = (unsigned)((M + 3) / 4);
  const size_t pstride = M * kVW;
  layernorm_kernel<<<ln_grid, 256, 0, st>>>(c->h, nullptr, nullptr, 0, 0, nullptr, pr0 + kVPOffLn1w, pr0 + kVPOffLn1b, nullptr, c->n, eps, (int)M);
  const int iM = (int)M;
  // h += A . W^T + bias, n = LayerNorm(h)
  auto residual = [&](bool lib, const GemmPlan& g, const MmPlan& m, const u16* A, int K, const u16* W, const float* bias, const float* nw,
                      const float* nb) {
    const bool parts = !lib && m.split > 1;
    const int e = lib ? vgemm(c, g, W, A, c->y, bias, st)
                      : parts ? vmm(c, m, kMmF32, {A, W, c->part, nullptr, iM, kVW, K, K, K, kVW, 1}, st)
                              : vmm(c, m, kMmBf16, {A, W, c->y, bias, iM, kVW, K, K, K, kVW, 1}, st);
    if (e != PI05_OK) return e;
    layernorm_kernel<<<ln_grid, 256, 0, st>>>(c->h, parts ? nullptr : c->y, parts ? c->part : nullptr, parts ? m.split : 0, pstride,
                                              parts ? bias : nullptr, nw, nb, c->h, c->n, eps, iM);
    return (int)PI05_OK;
  };
  for (int l = 0; l < p.L; ++l) {
    const u16* w = c->w + (size_t)l * kVLayerElems;
    const float* pr = c->par + (size_t)l * kVLayerParams;
    rc = c->lib_qkv ? vgemm(c, c->g_qkv, w + kVOffQkv, c->n, c->qkv, pr + kVPOffBqkv, st)
                    : vmm(c, c->m_qkv, kMmBf16, {c->n, w + kVOffQkv, c->qkv, pr + kVPOffBqkv, iM, kVQkvN, kVW, kVW, kVW, kVQkvN, 1}, st);
    if (rc != PI05_OK) return rc;
    vision_attn_kernel<<<(unsigned)(p.N * kVH * 2), 512, 0, st>>>(c->qkv, c->attn);
    if ((rc = residual(c->lib_o, c->g_o, c->m_o, c->attn, kVW, w + kVOffO, pr + kVPOffBo, pr + kVPOffLn2w, pr + kVPOffLn2b)) != PI05_OK) return rc;
    if ((rc = vmm(c, c->m_fc1, kMmGelu, {c->n, w + kVOff1, c->act, pr + kVPOffB1, iM, kVI, kVW, kVW, kVW, kVIp, 1}, st)) != PI05_OK) return rc;
    const bool last = l + 1 == p.L;
    const float* nw = last ? c->post_w : c->par + (size_t)(l + 1) * kVLayerParams + kVPOffLn1w;
    const float* nb = last ? c->post_b : c->par + (size_t)(l + 1) * kVLayerParams + kVPOffLn1b;
    if ((rc = residual(c->lib_fc2, c->g_fc2, c->m_fc2, c->act, kVIp, w + kVOff2, pr + kVPOffB2, nw, nb)) != PI05_OK) return rc;
  }
  rc = c->lib_proj ? vgemm(c, c->g_proj, c->proj_w, c->n, out, c->proj_b, st)
                   : vmm(c, c->m_proj, kMmBf16, {c->n, c->proj_w, out, c->proj_b, iM, kVProj, kVW, kVW, kVW, kVProj, 1}, st);
  if (rc != PI05_OK) return rc;
  if (c->d.out_scale != 1.0f) scale_kernel<<<grid_for(M * kVProj), 256, 0, st>>>(static_cast<u16*>(out), M * kVProj, c->d.out_scale);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return vfail(c, PI05_E_HIP, std::string("vision launch: ") + hipGetErrorString(e));
  return PI05_OK;
}

}  // extern "C"
