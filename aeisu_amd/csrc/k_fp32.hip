// FP32 policy: the controller and the reconstruction head in FP32 arithmetic, one kernel per stage
// (the reference's PyTorch path, aeisu/model.py:473-496 and aeisu/reconstruction.py:15-83, which
// users of aeisu/runtime.py run).  Activations stay FP32 in device memory (NHWC):
//   skip  [B][Hq][Wq][32]   project output (analysis features -> project 1x1 -> LeakyReLU)
//   low   [B][Hl][Wl][64]   compress and the four grouped 3x3 layers (ping-pong)
//   work  [B][Hq][Wq][32]   pixel_shuffle(expand) + skip
//   meta  [B][Hq][Wq][64]   refine 3x3 + LeakyReLU -> tail 1x1 (the packed coefficients)
// and the head writes the clipped 2x frame.
//
// The project runs as FP32 MFMAs, every other product as hi / lo FP16 splits on the FP16 MFMA (below);
// all sums are FP32, in a fixed order that differs from the reference's convolution order only by FP32
// rounding.
#include <algorithm>

#include "common.hpp"
#include "features.hpp"
#include "kernels.hpp"

namespace aeisu {

constexpr int kF32Threads = 256;
typedef float f2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ float to_f32(T v) { return (float)v; }

// ---- analysis features + project 1x1 + LeakyReLU ----------------------------------------------------
// One wave per block takes 64 packed pixels: each lane computes one pixel's 32 features, hands them over
// through LDS, and the wave runs the product as FP32 MFMAs (FP32 operands: the project weights reach 31 with
// heavy cancellation, and split operands would double the layer's error).  K step j takes feature j of the four
// phases (input channels 4j .. 4j + 3); features lie in LDS by phase, so that a lane's operands are 32
// contiguous bytes.  With the product as 1,024 FMAs per
// thread each wave waited for 1,024 weights from the scalar cache and stored 128 bytes per lane: 46 us at
// 1080p, 11 to 15 us for 256 x 256.
constexpr int kF32FeatRow = 36;                              // floats of a pixel's features in LDS (32 + 4 pad)
template <typename Tin>
__global__ __launch_bounds__(64) void f32_project_kernel(const Tin* __restrict__ src, const float* __restrict__ wimg,
                                                         float* __restrict__ skip, int H, int W, int Hq, int Wq, int py,
                                                         int px, long pixels) {
  __shared__ __attribute__((aligned(16))) float feat[64 * kF32FeatRow];
  const int lane = threadIdx.x, n = lane & 15, g = lane >> 4;
  const long first = (long)blockIdx.x * 64, idx = min(first + lane, pixels - 1);
  const int b = (int)(idx / ((long)Hq * Wq));
  const int rem = (int)(idx - (long)b * Hq * Wq);
  const int qy = rem / Wq, qx = rem - qy * Wq;
  const size_t plane = (size_t)H * W;
  const Tin* s = src + (size_t)b * 3 * plane;
  // 4x4 LR window on the padded grid (one halo pixel each side), replicate-clamped into the source
  float w[3][4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int sy = min(max(2 * qy - 1 + a - py, 0), H - 1);
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) {
      const int sx = min(max(2 * qx - 1 + c4 - px, 0), W - 1);
      const size_t o = (size_t)sy * W + sx;
#pragma unroll
      for (int c = 0; c < 3; ++c) w[c][a][c4] = to_f32(s[c * plane + o]);
    }
  }
  float A[2][8];
  f4 bs[2];
#pragma unroll
  for (int T = 0; T < 2; ++T) {
    bs[T] = *reinterpret_cast<const f4*>(wimg + kF32Project + 1024 + 16 * T + 4 * g);
#pragma unroll
    for (int j = 0; j < 8; ++j) A[T][j] = wimg[kF32Project + (4 * j + g) * 32 + 16 * T + n];
  }
  const Analysis an = analysis_from(wimg + kF32Analysis);
  float f[8][4];
  window_features(w, an, f);
#pragma unroll
  for (int q = 0; q < 8; ++q)                                // phase q >> 1, features 4 (q & 1) .. + 3
    *reinterpret_cast<float4*>(feat + lane * kF32FeatRow + 4 * q) =
        make_float4(f[4 * (q & 1)][q >> 1], f[4 * (q & 1) + 1][q >> 1], f[4 * (q & 1) + 2][q >> 1], f[4 * (q & 1) + 3][q >> 1]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // one wave: its LDS stores are done
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float* row = feat + (16 * p + n) * kF32FeatRow + 8 * g;
    const f4 lo = *reinterpret_cast<const f4*>(row), hi = *reinterpret_cast<const f4*>(row + 4);
    f4 acc[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int T = 0; T < 2; ++T)
        acc[T] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[T][j], j < 4 ? lo[j] : hi[j - 4], acc[T], 0, 0, 0);
    const long o = first + 16 * p + n;
    if (o < pixels) {
#pragma unroll
      for (int T = 0; T < 2; ++T) {
        f4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = leaky(acc[T][i] + bs[T][i], 0.1f);
        *reinterpret_cast<f4*>(skip + o * 32 + 16 * T + 4 * g) = r;
      }
    }
  }
}

// ---- split products on the FP16 MFMA ----------------------------------------------------------------
// An FP32 operand x is scaled by a power of two and written as hi + lo, hi = fp16(x), lo = fp16(x - hi),
// and a product is hi hi' + (hi lo' + lo hi'): three FP16 MFMAs in place of the FP32 FMAs, at 5 times the
// rate of the FP32 MFMA and 10 times that of the unpacked FMA.  hi + lo carries 22 to 23 bits, and the
// MFMA rounds its FP32 accumulator once per 8 products where the FMA chain rounds at every one, so the
// result is nearer to the exact sum than the chain's (64 x 96 frames of three kinds, both checkpoints,
// against 64 bits: coefficients 0.72 to 0.98 of the chain's error).  The cross terms go to an accumulator
// of their own: added to the main sum they would be rounded at its magnitude.
//
// The scale keeps FP32's range: the largest magnitude that shares it goes to [2^14, 2^15), so nothing overflows
// FP16, and the lo halves end at 2^-39 of that.  The 1x1 layers take a scale per pixel.  The 3x3 layers
// take the tile's largest (finite) pixel, and pixels below 2^-14 of it in a pass of their own with their own
// scale (bands): a pixel's values are thus held to 2^-22 of themselves or 2^-25 of its largest, whatever lies
// beside it.  Weights are scaled by output (row): 2^e with the row's largest in [2^14, 2^15).  A sum is brought back
// by 2^(-x - kF32Unscale) for an operand scale 2^x and then by the row's 2^(kF32Unscale - e), which no sum of FP32 operands
// (weights below 2^118) leaves FP32's range between.
__device__ __forceinline__ float residual_lo(float v, unsigned w) {   // v - (low half of w), exact
  float r;
  asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(v));
  return r;
}
__device__ __forceinline__ float residual_hi(float v, unsigned w) {
  float r;
  asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(v));
  return r;
}
// Four values -> their hi halves (two dwords) and lo halves.
__device__ __forceinline__ void split4(float a, float b, float c, float d, u2& hi, u2& lo) {
  const unsigned h0 = pack_h2(a, b), h1 = pack_h2(c, d);
  hi = u2{h0, h1};
  lo = u2{pack_h2(residual_lo(a, h0), residual_hi(b, h0)), pack_h2(residual_lo(c, h1), residual_hi(d, h1))};
}
__device__ __forceinline__ float pow2f(int e) { return __builtin_bit_cast(float, (unsigned)(e + 127) << 23); }
// Exponent e with m 2^e in [2^14, 2^15), for a finite m >= 0 (clamped for tiny m).
__device__ __forceinline__ int scale_exponent(float m) {
  return min(14 + 127 - (int)(__builtin_bit_cast(unsigned, m) >> 23), 100);
}
__device__ __forceinline__ float finite_abs(float v) {
  const float a = fabsf(v);
  return a < __builtin_inff() ? a : 0.f;
}
__device__ __forceinline__ float inverse_scale(int e) { return pow2f(-e - kF32Unscale); }   // e in [-113, 100]
template <int CTRL>
__device__ __forceinline__ unsigned dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppRor8 = 0x128;
// Magnitudes are compared as the bits of non-negative floats.
__device__ __forceinline__ unsigned max_of_8(unsigned m) {   // over 8 neighbouring lanes
  m = max(m, dpp<kDppXor1>(m));
  m = max(m, dpp<kDppXor2>(m));
  return max(m, dpp<kDppHalfMirror>(m));
}
__device__ __forceinline__ unsigned max_of_rows(unsigned m) {   // over the lanes n, n + 16, n + 32, n + 48
  unsigned a = m, b = m;
  permlane16_swap_u(a, b);
  a = b = max(a, b);
  permlane32_swap_u(a, b);
  return max(a, b);
}
__device__ __forceinline__ unsigned max_of_wave(unsigned m) {
  m = max_of_8(m);
  return max_of_rows(max(m, dpp<kDppRor8>(m)));
}
__device__ __forceinline__ float as_float(unsigned v) { return __builtin_bit_cast(float, v); }
__device__ __forceinline__ unsigned as_bits(float v) { return __builtin_bit_cast(unsigned, v); }

// ---- 3x3 layers: persistent blocks of four waves over tiles of 16 x TH pixels -----------------------
// A wave serves 32 output channels (two MFMA row tiles) of some of the tile's pixel rows and keeps their 36
// weight fragments (9 taps x 2 tiles x hi, lo: 144 VGPRs) for the launch: from LDS or L2 the fragments would be read once per pixel row and more often than the activations.  The tile's
// input halo is staged in LDS as hi and lo halves, split once per value.  Two blocks per CU (two waves per
// SIMD at 256 VGPRs): one block's staging and barriers overlap the other's products.
constexpr int kConvTW = 16, kConvPW = kConvTW + 2;
constexpr int kConvPix = 144;                        // LDS bytes per halo pixel: 32 channels hi, lo, pad
constexpr int kConvThreads = 256;

__device__ __forceinline__ void conv_weights(h8 (&A)[9][2][2], const h8* __restrict__ frag, int role, int lane) {
#pragma unroll
  for (int T = 0; T < 2; ++T)
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
      for (int part = 0; part < 2; ++part) A[tap][T][part] = frag[(((2 * role + T) * 9 + tap) * 2 + part) * 64 + lane];
}

// R neighbouring rows of 16 pixels: acc[r][T] = sum over the 9 taps of the wave's two row tiles.  p: the lane's
// operand of the first row's top left tap.  The rows share the operands of the input rows between them: R = 2
// reads 24 operands from LDS instead of 36 (1080p: refine + tail 80 -> 78 us, a grouped layer 27 -> 25).
template <int R>
__device__ __forceinline__ void conv_rows(const unsigned char* p, const h8 (&A)[9][2][2], f4 (&acc)[R][2]) {
  f4 small[R][2];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int T = 0; T < 2; ++T) acc[r][T] = small[r][T] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int iy = 0; iy < R + 2; ++iy)
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) {
      const unsigned char* q = p + (iy * kConvPW + dx) * kConvPix;
      const h8 bh = *reinterpret_cast<const h8*>(q), bl = *reinterpret_cast<const h8*>(q + 64);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (iy - r < 0 || iy - r > 2) continue;
        const int tap = 3 * (iy - r) + dx;
#pragma unroll
        for (int T = 0; T < 2; ++T) acc[r][T] = mfma_f16(A[tap][T][0], bh, acc[r][T]);
#pragma unroll
        for (int T = 0; T < 2; ++T) small[r][T] = mfma_f16(A[tap][T][0], bl, small[r][T]);
#pragma unroll
        for (int T = 0; T < 2; ++T) small[r][T] = mfma_f16(A[tap][T][1], bh, small[r][T]);
      }
    }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int T = 0; T < 2; ++T) acc[r][T] += small[r][T];
}

template <int TH>
struct ConvLayout {
  static constexpr int Rows = TH + 2, Chunks = Rows * kConvPW * 8;   // float4 chunks of the halo
  static constexpr int Per = (Chunks + kConvThreads - 1) / kConvThreads;
  static constexpr int SizeHalo = Rows * kConvPW * kConvPix;
  static constexpr int RPix = 272;                   // refine outputs: 64 channels hi, 64 lo, two inverse scales, pad
  static constexpr int LdsRefine = SizeHalo + TH * kConvTW * RPix;
};
struct F32ConvTiles {
  int H, W, tiles_x, tiles_y, num;
};
// The tile's halo, 32 of the CH channels of a pixel (in: the first of them), zero outside the grid.
template <int PER, int CH>
__device__ __forceinline__ void conv_fetch(float4 (&v)[PER], const float* __restrict__ in, const F32ConvTiles& G, int tidx,
                                           int th, int chunks, int tid) {
  const int per = G.tiles_x * G.tiles_y, b = tidx / per, rem = tidx - b * per;
  const int ty = rem / G.tiles_x, y0 = ty * th - 1, x0 = (rem - ty * G.tiles_x) * kConvTW - 1;
  const float* f = in + (size_t)b * G.H * G.W * CH;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + k * kConvThreads, pix = i >> 3, c = i & 7;
    const int py = pix / kConvPW, y = y0 + py, x = x0 + pix - py * kConvPW;
    const bool in_grid = (unsigned)y < (unsigned)G.H && (unsigned)x < (unsigned)G.W && i < chunks;
    v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (in_grid) v[k] = *reinterpret_cast<const float4*>(f + ((size_t)y * G.W + x) * CH + 4 * c);
  }
}
__device__ __forceinline__ float abs_max(float4 v) {
  return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}
__device__ __forceinline__ float finite_max(float4 v) {
  return fmaxf(fmaxf(finite_abs(v.x), finite_abs(v.y)), fmaxf(finite_abs(v.z), finite_abs(v.w)));
}
template <int PER>
__device__ __forceinline__ float chunk_max(const float4 (&v)[PER]) {
  float m = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) m = fmaxf(m, abs_max(v[k]));
  if (!(m < __builtin_inff())) {                     // an infinity somewhere: the largest finite value
    m = 0.f;
#pragma unroll
    for (int k = 0; k < PER; ++k) m = fmaxf(m, finite_max(v[k]));
  }
  return m;
}
// Largest magnitude of a set of pixels and smallest that is not zero (infinite if there is none).
struct PixelRange {
  float top, bottom;
};
// Over the block (uniform); through `red`, 8 words.  Holds a block barrier, before which every wave has left the LDS
// data of the tile or band before.  bottom: bits - 1, so that zeros count as the largest.
__device__ __forceinline__ PixelRange block_range(unsigned top, unsigned bottom, unsigned* red, int wave, int lane) {
  top = max_of_wave(top);
  bottom = ~max_of_wave(~bottom);
  if (lane == 0) {
    red[wave] = top;
    red[4 + wave] = bottom;
  }
  lds_barrier();
  const u4 t = *reinterpret_cast<const u4*>(red), b = *reinterpret_cast<const u4*>(red + 4);
  top = __builtin_amdgcn_readfirstlane(max(max(t[0], t[1]), max(t[2], t[3])));
  bottom = __builtin_amdgcn_readfirstlane(min(min(b[0], b[1]), min(b[2], b[3])));
  return {as_float(top), bottom == 0xffffffffu ? __builtin_inff() : as_float(bottom + 1u)};
}
// A tile's pixels are staged in bands, magnitudes from a band's largest down to kBand of it: a band's pixels share a
// scale, the others are staged as zeros, and each band's products are added to the sums.  A pixel's magnitude is
// its largest finite value (8 lanes hold a pixel); it is zero for zeros, infinities and NaN alone.
constexpr float kBand = 0x1p-14f;
template <int PER>
__device__ __forceinline__ PixelRange range_below(const float4 (&v)[PER], float cap, unsigned* red, int wave, int lane) {
  unsigned top = 0u, bottom = 0xffffffffu;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const unsigned p = max_of_8(as_bits(finite_max(v[k])));
    if (as_float(p) < cap) {
      top = max(top, p);
      bottom = min(bottom, p - 1u);
    }
  }
  return block_range(top, bottom, red, wave, lane);
}
template <int PER>
__device__ __forceinline__ void keep_band(float4 (&v)[PER], float low, float cap) {
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const float p = as_float(max_of_8(as_bits(finite_max(v[k]))));
    if (p > 0.f && (p < low || p >= cap)) v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}
// The whole tile's range; of its chunks of four channels where they all lie in one band, as nearly always, since that
// takes no exchange between the lanes of a pixel.  red: 16 words.
template <int PER>
__device__ __forceinline__ PixelRange tile_range(const float4 (&v)[PER], unsigned* red, int wave, int lane) {
  unsigned top = 0u, bottom = 0xffffffffu;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const unsigned m = as_bits(abs_max(v[k]));
    top = max(top, m);
    bottom = min(bottom, m - 1u);
  }
  const PixelRange r = block_range(top, bottom, red, wave, lane);
  if (r.top < __builtin_inff() && r.bottom >= r.top * kBand) return r;
  return range_below<PER>(v, __builtin_inff(), red + 8, wave, lane);
}

// Splits the staged chunks into LDS: hi halves of a pixel's 32 channels first, lo halves after.
template <int PER>
__device__ __forceinline__ void conv_stage(const float4 (&v)[PER], unsigned char* lds, float s, int chunks, int tid) {
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + k * kConvThreads, pix = i >> 3, c = i & 7;
    if (i < chunks) {
      u2 hi, lo;
      split4(v[k].x * s, v[k].y * s, v[k].z * s, v[k].w * s, hi, lo);
      unsigned char* d = lds + pix * kConvPix + 8 * c;
      *reinterpret_cast<u2*>(d) = hi;
      *reinterpret_cast<u2*>(d + 64) = lo;
    }
  }
}

// A grouped 3x3 layer (2 groups of 32 -> 32, zero padding) + LeakyReLU: blockIdx.y is the conv group, so the
// block's waves share its weights and split the tile's rows.  One thread per pixel and group with FP32 FMAs:
// 147 us at 1080p, 50 us for 256 x 256, now 29 and 5.7 (28 and 5.6 with one scale per tile and per layer).
template <int TH>
__global__ __launch_bounds__(kConvThreads, 2) void f32_grouped_kernel(const float* __restrict__ in, const h8* __restrict__ frag,
                                                                      const float* __restrict__ bias, float* __restrict__ out,
                                                                      F32ConvTiles G) {
  typedef ConvLayout<TH> LY;
  __shared__ __attribute__((aligned(16))) unsigned char smem[LY::SizeHalo];
  __shared__ __attribute__((aligned(16))) unsigned red[16];
  __shared__ __attribute__((aligned(16))) float rows[32];
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, grp = blockIdx.y;
  const float row = bias[kF32Rows + 32 * grp + (tid & 31)];   // stored once the loads below are under way
  const int n = lane & 15, g = lane >> 4;
  float4 v[LY::Per];
  int tidx = tile_of(0, G.num);
  if (tidx < G.num) conv_fetch<LY::Per, 64>(v, in + 32 * grp, G, tidx, TH, LY::Chunks, tid);
  h8 A[9][2][2];
  conv_weights(A, frag, grp, lane);
  f4 bs[2];
#pragma unroll
  for (int T = 0; T < 2; ++T) bs[T] = *reinterpret_cast<const f4*>(bias + 32 * grp + 16 * T + 4 * g);
  if (tid < 32) rows[tid] = row;                     // the loop's barriers are before the reads
  const int iters = tile_iters(G.num);
  for (int it = 0; it < iters; ++it) {
    if (tidx >= G.num) break;                        // block-uniform
    const int per = G.tiles_x * G.tiles_y, b = tidx / per, rem = tidx - b * per;
    const int ty = rem / G.tiles_x, y0 = ty * TH, x0 = (rem - ty * G.tiles_x) * kConvTW;
    const int next = tile_of(it + 1, G.num);
    PixelRange rg = tile_range(v, red, wave, lane);
    for (float cap = __builtin_inff();;) {           // over the tile's bands: one but for tiles with outliers
      const float low = rg.top * kBand;
      const bool first = cap == __builtin_inff(), last = rg.bottom >= low;
      const int ex = scale_exponent(rg.top);
      if (!(first && last)) keep_band<LY::Per>(v, low, cap);
      conv_stage<LY::Per>(v, smem, pow2f(ex), LY::Chunks, fresh(tid));
      if (last && it + 1 < iters && next < G.num) conv_fetch<LY::Per, 64>(v, in + 32 * grp, G, next, TH, LY::Chunks, fresh(tid));
      lds_barrier();
      const float inv = inverse_scale(ex);
      constexpr int R = TH / 4;                      // rows R wave .. R wave + R - 1
      f4 acc[R][2];
      conv_rows<R>(smem + (R * wave * kConvPW + n) * kConvPix + 16 * g, A, acc);
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int y = y0 + R * wave + j, x = x0 + n;
        if (y < G.H && x < G.W) {
          float* d = out + (((size_t)b * G.H + y) * G.W + x) * 64 + 32 * grp + 4 * g;
#pragma unroll
          for (int T = 0; T < 2; ++T) {
            const f4 sc = *reinterpret_cast<const f4*>(rows + 16 * T + 4 * g);
            f4 r = bs[T];
            if (!first) r = *reinterpret_cast<const f4*>(d + 16 * T);   // the sum so far
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              r[i] = fmaf(acc[j][T][i] * inv, sc[i], r[i]);
              if (last) r[i] = leaky(r[i], 0.1f);
            }
            *reinterpret_cast<f4*>(d + 16 * T) = r;
          }
        }
      }
      if (last) break;
      cap = low;
      conv_fetch<LY::Per, 64>(v, in + 32 * grp, G, tidx, TH, LY::Chunks, fresh(tid));
      rg = range_below<LY::Per>(v, cap, red + 8, wave, lane);
    }
    tidx = next;
  }
}

// refine 3x3 (32 -> 64) + LeakyReLU + tail 1x1 (64 -> 64).  One thread per pixel with FP32 FMAs was bound by
// their issue (22,528 per pixel): 511 us at 1080p, 98 us for 256 x 256, now 88 and 10 (81 and 9
// with one scale per tile and per layer, 94 with a scale per pixel for the tail of every tile).  Its 210 MB take 41 us
// of HBM time at 1080p and its MFMAs 34; the rest is the splitting and the LDS reads (320 KB per tile), which
// two waves per SIMD do not hide.  The refine outputs go to LDS as hi and lo halves
// (scaled by their bound from the tile's largest input and the weights; where a tile has several bands, a scale for
// each pixel's 32 channels of a wave, kept beside them) and wave w computes tail channels 16 w .. + 15 from them; refine: channels 32 (w & 1) .. + 31 of the rows of half w >> 1.
template <int TH>
__global__ __launch_bounds__(kConvThreads, 2) void f32_refine_tail_kernel(const float* __restrict__ work,
                                                                          const h8* __restrict__ rfrag,
                                                                          const h8* __restrict__ tfrag,
                                                                          const float* __restrict__ rbias,
                                                                          const float* __restrict__ tbias,
                                                                          float* __restrict__ meta, F32ConvTiles G,
                                                                          F32Bound bound) {
  typedef ConvLayout<TH> LY;
  __shared__ __attribute__((aligned(16))) unsigned char smem[LY::LdsRefine];
  __shared__ __attribute__((aligned(16))) unsigned red[16];
  __shared__ __attribute__((aligned(16))) float rb[128], tb[128];   // biases and row scales: in registers the kernel spills
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, role = wave & 1, half = wave >> 1;
  float4 v[LY::Per];
  const float row = (tid < 128 ? rbias : tbias)[(tid & 63) + (tid & 64 ? kF32Rows : 0)];
  int tidx = tile_of(0, G.num);
  if (tidx < G.num) conv_fetch<LY::Per, 32>(v, work, G, tidx, TH, LY::Chunks, tid);
  h8 A[9][2][2];
  conv_weights(A, rfrag, role, lane);
  (tid < 128 ? rb : tb)[tid & 127] = row;            // the loop's barriers are before the reads
  const int iters = tile_iters(G.num);
  for (int it = 0; it < iters; ++it) {
    if (tidx >= G.num) break;                        // block-uniform
    const int per = G.tiles_x * G.tiles_y, b = tidx / per, rem = tidx - b * per;
    const int ty = rem / G.tiles_x, y0 = ty * TH, x0 = (rem - ty * G.tiles_x) * kConvTW;
    const int next = tile_of(it + 1, G.num);
    PixelRange rg = tile_range(v, red, wave, lane);
    // a tile of one band scales its refine outputs by their bound
    const bool single = rg.bottom >= rg.top * kBand;
    const int eb = scale_exponent(fminf(fmaf(bound.gain, rg.top, bound.offset), 0x1p126f));
    for (float cap = __builtin_inff();;) {           // over the tile's bands
      const float low = rg.top * kBand;
      const bool first = cap == __builtin_inff(), last = rg.bottom >= low;
      const int ex = scale_exponent(rg.top);
      if (!(first && last)) keep_band<LY::Per>(v, low, cap);
      conv_stage<LY::Per>(v, smem, pow2f(ex), LY::Chunks, fresh(tid));
      if (last && it + 1 < iters && next < G.num) conv_fetch<LY::Per, 32>(v, work, G, next, TH, LY::Chunks, fresh(tid));
      lds_barrier();
      const float inv = inverse_scale(ex);
      constexpr int R = TH >= 4 ? 2 : 1;
      for (int row = half * (TH / 2); row < (half + 1) * (TH / 2); row += R) {
        const int ln = fresh(lane), n = ln & 15, g = ln >> 4;
        f4 acc[R][2];
        conv_rows<R>(smem + (row * kConvPW + n) * kConvPix + 16 * g, A, acc);
        f4 b0[2], sc[2];
#pragma unroll
        for (int T = 0; T < 2; ++T) {
          b0[T] = *reinterpret_cast<const f4*>(rb + 32 * role + 16 * T + 4 * g);
          sc[T] = *reinterpret_cast<const f4*>(rb + 64 + 32 * role + 16 * T + 4 * g);
        }
#pragma unroll
        for (int j = 0; j < R; ++j) {
          unsigned char* pix = smem + LY::SizeHalo + ((row + j) * kConvTW + n) * LY::RPix;
          unsigned char* d = pix + 64 * role + 8 * g;
          f4 r[2];
#pragma unroll
          for (int T = 0; T < 2; ++T) {
            r[T] = b0[T];
            if (!first) {                            // the sum so far
              const f2 a = *reinterpret_cast<const f2*>(d + 32 * T), c = *reinterpret_cast<const f2*>(d + 32 * T + 128);
              r[T] = f4{a[0], a[1], c[0], c[1]};
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              r[T][i] = fmaf(acc[j][T][i] * inv, sc[T][i], r[T][i]);
              if (last) r[T][i] = leaky(r[T][i], 0.1f);
            }
          }
          if (last) {
            float s = pow2f(eb);
            if (!single) {                           // by the pixel's 32 channels in this wave
              const float m = fmaxf(abs_max(make_float4(r[0][0], r[0][1], r[0][2], r[0][3])),
                                    abs_max(make_float4(r[1][0], r[1][1], r[1][2], r[1][3])));
              const int er = scale_exponent(as_float(max_of_rows(as_bits(m))));
              s = pow2f(er);
              if (g == 0) *reinterpret_cast<float*>(pix + 256 + 4 * role) = inverse_scale(er);
            }
#pragma unroll
            for (int T = 0; T < 2; ++T) {
              u2 hi, lo;
              split4(r[T][0] * s, r[T][1] * s, r[T][2] * s, r[T][3] * s, hi, lo);
              *reinterpret_cast<u2*>(d + 32 * T) = hi;
              *reinterpret_cast<u2*>(d + 32 * T + 128) = lo;
            }
          } else {
#pragma unroll
            for (int T = 0; T < 2; ++T) {
              *reinterpret_cast<f2*>(d + 32 * T) = f2{r[T][0], r[T][1]};
              *reinterpret_cast<f2*>(d + 32 * T + 128) = f2{r[T][2], r[T][3]};
            }
          }
        }
      }
      if (last) break;
      cap = low;
      conv_fetch<LY::Per, 32>(v, work, G, tidx, TH, LY::Chunks, fresh(tid));
      rg = range_below<LY::Per>(v, cap, red + 8, wave, lane);
    }
    // the tail fragments are read for every tile: kept, they do not fit the 256 VGPRs
    h8 At[2][2];
    const h8* tf = tfrag + wave * 4 * 64 + fresh(lane);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int part = 0; part < 2; ++part) At[k][part] = tf[(k * 2 + part) * 64];
    lds_barrier();
    const int ln = fresh(lane), n = ln & 15, g = ln >> 4;
    const f4 bias = *reinterpret_cast<const f4*>(tb + 16 * wave + 4 * g), sc = *reinterpret_cast<const f4*>(tb + 64 + 16 * wave + 4 * g);
#pragma unroll 2
    for (int row = 0; row < TH; ++row) {
      const unsigned char* pix = smem + LY::SizeHalo + (row * kConvTW + n) * LY::RPix;
      f4 acc[2];                                     // K chunk k: channels 32 k .. + 31, which share a scale
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const h8 bh = *reinterpret_cast<const h8*>(pix + 16 * g + 64 * k), bl = *reinterpret_cast<const h8*>(pix + 16 * g + 64 * k + 128);
        f4 small = mfma_f16(At[k][0], bl, f4{0.f, 0.f, 0.f, 0.f});
        acc[k] = mfma_f16(At[k][0], bh, f4{0.f, 0.f, 0.f, 0.f});
        acc[k] += mfma_f16(At[k][1], bh, small);
      }
      float2 inv = make_float2(inverse_scale(eb), inverse_scale(eb));
      if (!single) inv = *reinterpret_cast<const float2*>(pix + 256);
      const int qy = y0 + row, qx = x0 + n;
      if (qy < G.H && qx < G.W) {
        f4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = fmaf(fmaf(acc[0][i], inv.x, acc[1][i] * inv.y), sc[i], bias[i]);
        *reinterpret_cast<f4*>(meta + (((size_t)b * G.H + qy) * G.W + qx) * 64 + 16 * wave + 4 * g) = o;
      }
    }
    tidx = next;
  }
}

// ---- 1x1 layers of the low grid ---------------------------------------------------------------------
// A wave takes 16 low pixels at a time: a lane reads the 8 channels of its MFMA K slots straight from memory
// (32 contiguous bytes), splits them in registers, and the pixel's scale comes from the four lanes that hold
// its channels.  All 32 weight fragments stay in registers (128 VGPRs).  The next group's loads are in flight
// during the products.
__device__ __forceinline__ void split8(float4 a, float4 b, float s, h8& hi, h8& lo) {
  u2 h0, l0, h1, l1;
  split4(a.x * s, a.y * s, a.z * s, a.w * s, h0, l0);
  split4(b.x * s, b.y * s, b.z * s, b.w * s, h1, l1);
  hi = __builtin_bit_cast(h8, u4{h0[0], h0[1], h1[0], h1[1]});
  lo = __builtin_bit_cast(h8, u4{l0[0], l0[1], l1[0], l1[1]});
}
struct LowPixel {
  int b, y, x;
};
__device__ __forceinline__ LowPixel low_pixel(int idx, int Hl, int Wl) {
  const int per = Hl * Wl, b = idx / per, rem = idx - b * per, y = rem / Wl;
  return {b, y, rem - y * Wl};
}

// pixel_unshuffle + compress 1x1 (128 -> 64) + LeakyReLU: K chunk k is phase k's 32 skip channels.  At 1080p
// 103 us with one thread per pixel and FP32 FMAs.
__global__ __launch_bounds__(kF32Threads, 2) void f32_compress_kernel(const float* __restrict__ skip,
                                                                      const h8* __restrict__ frag,
                                                                      const float* __restrict__ bias,
                                                                      float* __restrict__ low, int Hl, int Wl, int pixels) {
  const int lane = lane_id(), n = lane & 15, g = lane >> 4, waves = gridDim.x * (kF32Threads / 64);
  const int groups = (pixels + 15) >> 4;
  int grp = blockIdx.x * (kF32Threads / 64) + (threadIdx.x >> 6);
  auto fetch = [&](int gi, float4 (&v)[8]) {
    const LowPixel p = low_pixel(min(gi * 16 + n, pixels - 1), Hl, Wl);
    const float* s = skip + (((size_t)p.b * 2 * Hl + 2 * p.y) * 2 * Wl + 2 * p.x) * 32 + 8 * g;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float* q = s + (size_t)(k >> 1) * 2 * Wl * 32 + (k & 1) * 32;
      v[2 * k] = *reinterpret_cast<const float4*>(q);
      v[2 * k + 1] = *reinterpret_cast<const float4*>(q + 4);
    }
  };
  __shared__ __attribute__((aligned(16))) float rows[64];
  const float row = bias[kF32Rows + (threadIdx.x & 63)];
  float4 v[8];
  if (grp < groups) fetch(grp, v);
  h8 A[4][4][2];
  f4 bs[4];
#pragma unroll
  for (int T = 0; T < 4; ++T) {
    bs[T] = *reinterpret_cast<const f4*>(bias + 16 * T + 4 * g);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int part = 0; part < 2; ++part) A[T][k][part] = frag[((T * 4 + k) * 2 + part) * 64 + lane];
  }
  if (threadIdx.x < 64) rows[threadIdx.x] = row;
  lds_barrier();
  for (; grp < groups; grp += waves) {
    const int ex = scale_exponent(as_float(max_of_rows(as_bits(chunk_max(v)))));
    const float s = pow2f(ex), inv = inverse_scale(ex);
    h8 bh[4], bl[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) split8(v[2 * k], v[2 * k + 1], s, bh[k], bl[k]);
    if (grp + waves < groups) fetch(grp + waves, v);
    const int idx = grp * 16 + n;
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      f4 acc = {0.f, 0.f, 0.f, 0.f}, small = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        acc = mfma_f16(A[T][k][0], bh[k], acc);
        small = mfma_f16(A[T][k][0], bl[k], small);
        small = mfma_f16(A[T][k][1], bh[k], small);
      }
      const f4 sc = *reinterpret_cast<const f4*>(rows + 16 * T + 4 * g);
      f4 r;
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = leaky(fmaf((acc[i] + small[i]) * inv, sc[i], bs[T][i]), 0.1f);
      if (idx < pixels) *reinterpret_cast<f4*>(low + (size_t)idx * 64 + 16 * T + 4 * g) = r;
    }
  }
}

// expand 1x1 (64 -> 128) + LeakyReLU, pixel_shuffle, + skip: row tile T holds channels 16 (T >> 2) .. + 15 of
// phase T & 3 (expand output channel c * 4 + 2i + j goes to channel c of packed pixel (2ly + i, 2lx + j)).  At
// 1080p 118 us with one thread per pixel and FP32 FMAs.
__global__ __launch_bounds__(kF32Threads, 2) void f32_expand_kernel(const float* __restrict__ low,
                                                                    const float* __restrict__ skip,
                                                                    const h8* __restrict__ frag,
                                                                    const float* __restrict__ bias,
                                                                    float* __restrict__ work, int Hl, int Wl, int pixels) {
  const int lane = lane_id(), n = lane & 15, g = lane >> 4, waves = gridDim.x * (kF32Threads / 64);
  const int groups = (pixels + 15) >> 4;
  int grp = blockIdx.x * (kF32Threads / 64) + (threadIdx.x >> 6);
  auto fetch = [&](int gi, float4 (&v)[4]) {
    const float* s = low + (size_t)min(gi * 16 + n, pixels - 1) * 64 + 8 * g;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      v[2 * k] = *reinterpret_cast<const float4*>(s + 32 * k);
      v[2 * k + 1] = *reinterpret_cast<const float4*>(s + 32 * k + 4);
    }
  };
  __shared__ __attribute__((aligned(16))) float sb[256];   // bias, then row scale, by row tile and row
  const int rt = threadIdx.x >> 4 & 7;
  const float row = bias[(threadIdx.x < 128 ? 0 : kF32Rows) + (16 * (rt >> 2) + (threadIdx.x & 15)) * 4 + (rt & 3)];
  float4 v[4];
  if (grp < groups) fetch(grp, v);
  h8 A[8][2][2];
#pragma unroll
  for (int T = 0; T < 8; ++T)
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int part = 0; part < 2; ++part) A[T][k][part] = frag[((T * 2 + k) * 2 + part) * 64 + lane];
  sb[threadIdx.x] = row;
  lds_barrier();
  for (; grp < groups; grp += waves) {
    const int idx = grp * 16 + n;
    const LowPixel p = low_pixel(min(idx, pixels - 1), Hl, Wl);
    const size_t o = (((size_t)p.b * 2 * Hl + 2 * p.y) * 2 * Wl + 2 * p.x) * 32 + 4 * g;
    auto at = [&](int T) { return o + (size_t)((T & 3) >> 1) * 2 * Wl * 32 + (T & 1) * 32 + 16 * (T >> 2); };
    f4 sk[8];
#pragma unroll
    for (int T = 0; T < 8; ++T) sk[T] = *reinterpret_cast<const f4*>(skip + at(T));
    const int ex = scale_exponent(as_float(max_of_rows(as_bits(chunk_max(v)))));
    const float s = pow2f(ex), inv = inverse_scale(ex);
    h8 bh[2], bl[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) split8(v[2 * k], v[2 * k + 1], s, bh[k], bl[k]);
    if (grp + waves < groups) fetch(grp + waves, v);
#pragma unroll
    for (int T = 0; T < 8; ++T) {
      f4 acc = {0.f, 0.f, 0.f, 0.f}, small = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        acc = mfma_f16(A[T][k][0], bh[k], acc);
        small = mfma_f16(A[T][k][0], bl[k], small);
        small = mfma_f16(A[T][k][1], bh[k], small);
      }
      const f4 bs = *reinterpret_cast<const f4*>(sb + 16 * T + 4 * g), sc = *reinterpret_cast<const f4*>(sb + 128 + 16 * T + 4 * g);
      f4 r;
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = leaky(fmaf((acc[i] + small[i]) * inv, sc[i], bs[i]), 0.1f) + sk[T][i];
      if (idx < pixels) *reinterpret_cast<f4*>(work + at(T)) = r;
    }
  }
}

// ---- head: clamp, polyphase filter synthesis, 5x5 application, clip ----------------------------------
// coefficient_clamp (aeisu/reconstruction.py:15-17) in FP32 with the reference's separate multiply
// and add: sign(a) min(|a|, 2 + 0.05 (|a| - 2), 2.5), since the line lies above |a| up to 2 and below it
// after.  gfx950's v_minimum3_f32 propagates NaN: a NaN coefficient stays NaN (so does the output, which raises
// the non-finite flag).
__device__ __forceinline__ float clamp_coef(float a) {
#pragma clang fp contract(off)
  const float v = 2.f + 0.05f * (fabsf(a) - 2.f);
  float c;
  asm("v_minimum3_f32 %0, |%1|, %2, %3" : "=v"(c) : "v"(a), "v"(v), "s"(2.5f));
  return __builtin_copysignf(c, a);
}

// Persistent blocks over tiles of 64 x 4 LR pixels, one row per wave, in two chunks of 32 pixels.  The filter
// weights of a chunk's even and odd pixels are two MFMA products of 16 columns, as in k_head.hip: row 4g + i of
// row tile t is (phase g, tap 4t + i), so accumulator lane (n, g) holds all 25 taps of phase g of pixels 2n and
// 2n + 1, with bank and coefficients in three FP16 parts each (exact to 2^-25),
// [K_3 | K_hi] . [c_hi ; c_3] + [K_lo | K_hi] . [c_lo ; c_lo] + [K_lo | K_hi] . [c_hi ; c_hi], small terms
// first, since the MFMA cuts off the bits of all terms below the largest of a pass; the FP32 base is added to
// the sum, not taken as its first addend.  Cutting off lowers every sum, by 1e-9 on average, and the 25 taps add
// that up: bank and base of odd taps are negated and their weights applied with the other sign, so that neighbouring
// taps take it from each other (mean error of the output -1.3e-8 without, 4e-9 (area) and 4e-10 (DIV2K) with it).  Against 64
// bits (frames of 33 x 65 to 1080p) the output's error is 1.08e-7 (area) and 1.17e-7 (DIV2K); one FP32 FMA chain
// per weight gave 1.17e-7 and 1.26e-7, all sums of one sign 1.21e-7 and 1.20e-7, FP32 MFMAs 1.15e-7 and 1.23e-7 and
// 113 us instead of 88 at 1080p.  Bank and base are scaled by a power of two, the RGB tile by its inverse.
// The lane applies them with FP32 FMAs in tap order.  Two neighbouring pixels share 20 of their 25 window
// positions: 30 LDS reads of 16 bytes instead of 50, which would take 46 us of LDS time at 1080p; the tile
// holds even and odd columns apart, so that the lanes' reads are contiguous.  One thread per pixel took 168 us
// at 1080p (1,600 FMAs of synthesis and strided coefficient reads).
constexpr int kF32HW = 64, kF32HH = 4;                       // LR pixels of a tile
constexpr int kF32HLW = kF32HW + 4, kF32HLH = kF32HH + 4;    // with the 2-pixel halo
constexpr int kF32HPos = kF32HLW * kF32HLH, kF32HPer = (kF32HPos + kF32Threads - 1) / kF32Threads;
constexpr int kF32HPlane = kF32HPos / 2;
struct F32HeadGeom {
  int H, W, Hq, Wq, py, px, tiles_x, tiles_y, num;
  float unscale;                                             // of the bank's power of two
};
struct F32HeadTile {
  int b, y0, x0;
};
__device__ __forceinline__ F32HeadTile f32_head_tile(int tidx, const F32HeadGeom& G) {
  const int per = G.tiles_x * G.tiles_y, b = tidx / per, rem = tidx - b * per, ty = rem / G.tiles_x;
  return {b, ty * kF32HH, (rem - ty * G.tiles_x) * kF32HW};
}
template <typename Tin>
__device__ __forceinline__ void f32_head_rgb(Tin (&v)[kF32HPer][3], const Tin* __restrict__ src, F32HeadTile t,
                                             const F32HeadGeom& G, int tid) {
  const size_t plane = (size_t)G.H * G.W;
  const Tin* s = src + (size_t)t.b * 3 * plane;
#pragma unroll
  for (int k = 0; k < kF32HPer; ++k) {
    const int q = min(tid + kF32Threads * k, kF32HPos - 1), ly = q / kF32HLW, lx = q - ly * kF32HLW;
    const size_t o = (size_t)min(max(t.y0 + ly - 2, 0), G.H - 1) * G.W + min(max(t.x0 + lx - 2, 0), G.W - 1);
#pragma unroll
    for (int c = 0; c < 3; ++c) v[k][c] = s[c * plane + o];
  }
}
// The lane's eight coefficients of pixels 2n and 2n + 1 of chunk j of the wave's row.  Pixels past the frame edge
// take the edge's (inside the tensor) and are not stored.
__device__ __forceinline__ void f32_head_coef(float4 (&c)[2][2], const float* __restrict__ meta, F32HeadTile t,
                                              const F32HeadGeom& G, int j, int wave, int lane) {
  const int n = lane & 15, Y = min(t.y0 + wave, G.H - 1) + G.py;
  const float* row = meta + ((size_t)t.b * G.Hq + (Y >> 1)) * G.Wq * 64 + 32 * (Y & 1) + 8 * ((lane >> 4) & 1);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int X = min(t.x0 + 32 * j + 2 * n + p, G.W - 1) + G.px;
    const float* q = row + (size_t)(X >> 1) * 64 + 16 * (X & 1);
    c[p][0] = *reinterpret_cast<const float4*>(q);
    c[p][1] = *reinterpret_cast<const float4*>(q + 4);
  }
}
// The output is written once and not read here: the non-temporal hint keeps it from displacing the coefficients
// (16 frames in turn: 1080p 411 -> 408 us a call, 540p 141.4 -> 138; 256 x 256 unchanged).
// Output columns 4n .. 4n + 3 of a chunk row and channel: pixels 2n and 2n + 1, left and right.
__device__ __forceinline__ void store_quad(float* p, float a, float b, float c, float d, bool second) {
  if (second) __builtin_nontemporal_store(f4{a, b, c, d}, reinterpret_cast<f4*>(p));
  else *reinterpret_cast<float2*>(p) = make_float2(a, b);
}
__device__ __forceinline__ void store_quad(_Float16* p, float a, float b, float c, float d, bool second) {
  if (second) __builtin_nontemporal_store(u2{pack_h2(a, b), pack_h2(c, d)}, reinterpret_cast<u2*>(p));
  else *reinterpret_cast<unsigned*>(p) = pack_h2(a, b);
}

template <typename Tin, typename Tout>
__global__ __launch_bounds__(kF32Threads, 3) void f32_head_kernel(const Tin* __restrict__ src, const float* __restrict__ meta,
                                                                  const h8* __restrict__ bank, Tout* __restrict__ out,
                                                                  F32HeadGeom G, unsigned* __restrict__ nonfinite) {
  __shared__ float4 tiles[2][2][kF32HPlane];                 // [buffer][column parity]
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, n = lane & 15, g = lane >> 4;
  __shared__ h8 bank3[7 * 64];                               // the third parts' fragments and the base: kept in
  __shared__ f4 base[4 * 7];                                 // registers they cost the third wave per SIMD
  h8 A[7];
#pragma unroll
  for (int t = 0; t < 7; ++t) A[t] = bank[t * 64 + lane];
  for (int i = tid; i < 7 * 64; i += kF32Threads) bank3[i] = bank[7 * 64 + i];
  if (tid < 28) base[tid] = reinterpret_cast<const f4*>(bank + 14 * 64)[tid];
  const size_t oplane = (size_t)4 * G.H * G.W;
  float chk = 0.f;                                           // NaN once an output was not finite
  const int iters = tile_iters(G.num);
  int tidx = tile_of(0, G.num);
  // in flight: the next tile's RGB and the next chunk's coefficients (read as soon as the last ones are used)
  Tin rgb[kF32HPer][3];
  float4 coef[2][2];                                         // [pixel parity][half of the lane's eight]
  if (tidx < G.num) {
    const F32HeadTile t = f32_head_tile(tidx, G);
    f32_head_rgb(rgb, src, t, G, tid);
    f32_head_coef(coef, meta, t, G, 0, wave, lane);
  }
  for (int it = 0; it < iters; ++it) {
    if (tidx >= G.num) break;                                // block-uniform
    const F32HeadTile t = f32_head_tile(tidx, G);
    float4(*buf)[kF32HPlane] = tiles[it & 1];
#pragma unroll
    for (int k = 0; k < kF32HPer; ++k) {
      const int q = tid + kF32Threads * k;                   // positions of a row alternate between the planes
      if (q < kF32HPos) buf[q & 1][q >> 1] = make_float4((float)rgb[k][0] * G.unscale, (float)rgb[k][1] * G.unscale, (float)rgb[k][2] * G.unscale, 0.f);
    }
    const int next = tile_of(it + 1, G.num);
    const bool more = it + 1 < iters && next < G.num;
    tidx = more ? next : G.num;
    const F32HeadTile tn = f32_head_tile(more ? next : 0, G);
    if (more) f32_head_rgb(rgb, src, tn, G, fresh(tid));
    lds_barrier();                                           // buf complete; the other buffer is free again
    const int y = t.y0 + wave;
    if (y >= G.H) {                                          // wave-uniform; the barriers are above
      if (more) f32_head_coef(coef, meta, tn, G, 0, wave, fresh(lane));
      continue;
    }
    for (int j = 0; j < 2; ++j) {
      const int lane_j = fresh(lane);
      f4 w[2][7];
      h8 bh[2], bl[2], bt[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const float4 c0 = coef[p][0], c1 = coef[p][1];
        const float c[8] = {clamp_coef(c0.x), clamp_coef(c0.y), clamp_coef(c0.z), clamp_coef(c0.w),
                            clamp_coef(c1.x), clamp_coef(c1.y), clamp_coef(c1.z), clamp_coef(c1.w)};
        u4 hi, lo, third;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          hi[e] = pack_h2(c[2 * e], c[2 * e + 1]);
          const float r0 = residual_lo(c[2 * e], hi[e]), r1 = residual_hi(c[2 * e + 1], hi[e]);
          lo[e] = pack_h2(r0, r1);
          const unsigned t3 = pack_h2(residual_lo(r0, lo[e]), residual_hi(r1, lo[e]));
          third[e] = (lane_j >> 4) < 2 ? hi[e] : t3;
        }
        bh[p] = __builtin_bit_cast(h8, hi);
        bl[p] = __builtin_bit_cast(h8, lo);
        bt[p] = __builtin_bit_cast(h8, third);
      }
#pragma unroll
      for (int q = 0; q < 7; ++q) {
        const h8 a3 = bank3[q * 64 + lane_j];
        const f4 bs = base[(lane_j >> 4) * 7 + q];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          w[p][q] = mfma_f16(a3, bt[p], f4{0.f, 0.f, 0.f, 0.f});
          w[p][q] = mfma_f16(A[q], bl[p], w[p][q]);
          w[p][q] = mfma_f16(A[q], bh[p], w[p][q]);
          w[p][q] += bs;
        }
      }
      if (j == 0) f32_head_coef(coef, meta, t, G, 1, wave, lane_j);
      else if (more) f32_head_coef(coef, meta, tn, G, 0, wave, lane_j);
      float u[2][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
#pragma unroll
      for (int dy = 0; dy < 5; ++dy)
#pragma unroll
        for (int dx = 0; dx < 6; ++dx) {
          const float4 L = buf[dx & 1][(wave + dy) * (kF32HLW / 2) + 16 * j + n + (dx >> 1)];
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            if (dx - p < 0 || dx - p > 4) continue;
            const int tap = dy * 5 + dx - p;
            const float wt = tap & 1 ? -w[p][tap >> 2][tap & 3] : w[p][tap >> 2][tap & 3];
            u[p][0] = fmaf(wt, L.x, u[p][0]);
            u[p][1] = fmaf(wt, L.y, u[p][1]);
            u[p][2] = fmaf(wt, L.z, u[p][2]);
          }
        }
      // pair phases (TL, TR) in lane groups 0 and 1 and (BL, BR) in 2 and 3: even groups then store channel 0
      // and channel 2, odd groups channel 1
      const int x = t.x0 + 32 * j + 2 * n;
      float left[2][3], right[2][3];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const bool inside = x + p < G.W;
        chk = fmaf(inside ? u[p][0] + u[p][1] + u[p][2] : 0.f, 0.f, chk);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          left[p][c] = __builtin_amdgcn_fmed3f(u[p][c], 0.f, 1.f);
          right[p][c] = left[p][c];
          permlane16_swap(left[p][c], right[p][c]);
        }
      }
      if (x < G.W) {
        const bool second = x + 1 < G.W, odd = g & 1;
        Tout* o = out + (size_t)t.b * 3 * oplane + (size_t)(2 * y + (g >> 1)) * (2 * G.W) + 2 * x;
        store_quad(o + (odd ? oplane : 0), odd ? left[0][1] : left[0][0], odd ? right[0][1] : right[0][0],
                   odd ? left[1][1] : left[1][0], odd ? right[1][1] : right[1][0], second);
        if (!odd) store_quad(o + 2 * oplane, left[0][2], right[0][2], left[1][2], right[1][2], second);
      }
    }
  }
  if (nonfinite && __ballot(chk != chk) != 0ull && lane == 0) atomicOr(nonfinite, 1u);
}

// ---- launchers ---------------------------------------------------------------------------------------
static F32ConvTiles conv_tiles(int H, int W, int th, int batch) {
  F32ConvTiles G{H, W, (W + kConvTW - 1) / kConvTW, (H + th - 1) / th, 0};
  G.num = batch * G.tiles_x * G.tiles_y;
  return G;
}
template <int TH>
static hipError_t launch_grouped_t(const float* in, const F32Weights& W, int l, float* out, int Hl, int Wl, int batch, int cus,
                                   hipStream_t stream) {
  const F32ConvTiles G = conv_tiles(Hl, Wl, TH, batch);
  hipLaunchKernelGGL(f32_grouped_kernel<TH>, dim3(persistent_grid(G.num, cus), 2), dim3(kConvThreads), 0, stream, in,
                     (const h8*)W.grouped[l], W.image + kF32BiasGrouped + 64 * l, out, G);
  return hipGetLastError();
}
static hipError_t launch_f32_grouped(const float* in, const F32Weights& W, int l, float* out, int Hl, int Wl, int batch,
                                     int cus, hipStream_t stream) {
  // tiles of 8 or of 4 rows (one per wave), whichever takes less: rounds of the resident blocks (cus per conv group)
  // times a tile's rows and about four for its halo, staging and barriers.  360 x 640: 143 tiles of 8 rows in one
  // round where tiles of 4 rows take two, frame 87.9 -> 83.3 us; 256 x 256 keeps 90 tiles of 4 rows, 540p 8 rows.
  auto cost = [&](int th) { return ((long)conv_tiles(Hl, Wl, th, batch).num + cus - 1) / cus * (th + 4); };
  return cost(8) <= cost(4)
             ? launch_grouped_t<8>(in, W, l, out, Hl, Wl, batch, cus, stream)
             : launch_grouped_t<4>(in, W, l, out, Hl, Wl, batch, cus, stream);
}
template <int TH>
static hipError_t launch_refine_t(const float* work, const F32Weights& W, float* meta, int Hq, int Wq, int batch, int cus,
                                  hipStream_t stream) {
  const F32ConvTiles G = conv_tiles(Hq, Wq, TH, batch);
  hipLaunchKernelGGL(f32_refine_tail_kernel<TH>, dim3(persistent_grid(G.num, 2 * cus)), dim3(kConvThreads), 0, stream, work,
                     (const h8*)W.refine, (const h8*)W.tail, W.image + kF32BiasRefine, W.image + kF32BiasTail, meta, G, W.refine_bound);
  return hipGetLastError();
}
static hipError_t launch_f32_refine_tail(const float* work, const F32Weights& W, float* meta, int Hq, int Wq, int batch,
                                         int cus, hipStream_t stream) {
  // tiles of 8 rows where they fill the 2 x cus resident blocks, else of 2 rows (more blocks, less work each).  The
  // line is not a measured one: just below it (270 x 480 has 320 tiles of 8 rows, one round) 2 rows take three rounds.
  return conv_tiles(Hq, Wq, 8, batch).num >= 2 * cus ? launch_refine_t<8>(work, W, meta, Hq, Wq, batch, cus, stream)
                                                     : launch_refine_t<2>(work, W, meta, Hq, Wq, batch, cus, stream);
}

hipError_t launch_f32_controller(int in_fp32, const void* src, const F32Weights& wts, float* skip, float* low0, float* low1,
                                 float* const* lows, float* work, float* meta, int H, int W, int Hq, int Wq, int py, int px,
                                 int batch, int cus, hipStream_t stream, hipEvent_t* ev) {
  const int Hl = Hq / 2, Wl = Wq / 2;
  const float* wimg = wts.image;
  const long packed = (long)batch * Hq * Wq, lowpx = (long)batch * Hl * Wl;
  if (in_fp32)
    hipLaunchKernelGGL(f32_project_kernel<float>, dim3((unsigned)((packed + 63) / 64)), dim3(64), 0, stream,
                       (const float*)src, wimg, skip, H, W, Hq, Wq, py, px, packed);
  else
    hipLaunchKernelGGL(f32_project_kernel<_Float16>, dim3((unsigned)((packed + 63) / 64)), dim3(64), 0, stream,
                       (const _Float16*)src, wimg, skip, H, W, Hq, Wq, py, px, packed);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (ev && (e = hipEventRecord(ev[1], stream)) != hipSuccess) return e;
  // layer outputs: lows[i] when every layer is kept, else ping-pong between low0 and low1
  float* dst[5];
  for (int i = 0; i < 5; ++i) dst[i] = lows ? lows[i] : (i % 2 ? low1 : low0);
  const int low_blocks = (int)std::min((lowpx + 63) / 64, 2L * cus);     // four groups of 16 pixels a block, persistent
  hipLaunchKernelGGL(f32_compress_kernel, dim3(low_blocks), dim3(kF32Threads), 0, stream, (const float*)skip,
                     (const h8*)wts.compress, wimg + kF32BiasCompress, dst[0], Hl, Wl, (int)lowpx);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (ev && (e = hipEventRecord(ev[2], stream)) != hipSuccess) return e;
  for (int l = 0; l < 4; ++l)
    if ((e = launch_f32_grouped(dst[l], wts, l, dst[l + 1], Hl, Wl, batch, cus, stream)) != hipSuccess) return e;
  if (ev && (e = hipEventRecord(ev[3], stream)) != hipSuccess) return e;
  hipLaunchKernelGGL(f32_expand_kernel, dim3(low_blocks), dim3(kF32Threads), 0, stream, (const float*)dst[4],
                     (const float*)skip, (const h8*)wts.expand, wimg + kF32BiasExpand, work, Hl, Wl, (int)lowpx);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (ev && (e = hipEventRecord(ev[4], stream)) != hipSuccess) return e;
  if ((e = launch_f32_refine_tail(work, wts, meta, Hq, Wq, batch, cus, stream)) != hipSuccess) return e;
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (ev && (e = hipEventRecord(ev[5], stream)) != hipSuccess) return e;
  return hipSuccess;
}

hipError_t launch_f32_head(int in_fp32, int out_fp32, const void* src, const float* meta, const F32Weights& wts, void* out,
                           int H, int W, int Hq, int Wq, int py, int px, int batch, int cus, unsigned* nonfinite,
                           hipStream_t stream) {
  F32HeadGeom G{H, W, Hq, Wq, py, px, (W + kF32HW - 1) / kF32HW, (H + kF32HH - 1) / kF32HH, 0, wts.head_unscale};
  G.num = batch * G.tiles_x * G.tiles_y;
  const int grid = persistent_grid(G.num, 3 * cus);
#define AEISU_F32_HEAD(TI, TO)                                                                                        \
  hipLaunchKernelGGL((f32_head_kernel<TI, TO>), dim3(grid), dim3(kF32Threads), 0, stream, (const TI*)src, meta,       \
                     (const h8*)wts.head, (TO*)out, G, nonfinite)
  if (in_fp32 && out_fp32) AEISU_F32_HEAD(float, float);
  else if (in_fp32) AEISU_F32_HEAD(float, _Float16);
  else if (out_fp32) AEISU_F32_HEAD(_Float16, float);
  else AEISU_F32_HEAD(_Float16, _Float16);
#undef AEISU_F32_HEAD
  return hipGetLastError();
}

}  // namespace aeisu
