// Refine 3x3 (32 -> 64) + LeakyReLU + linear 1x1 tail (64 -> 64) at packed
// (half) resolution, producing the FP16 parity-major coefficient tensor.
//
// Reference: aeisu/model.py:489-490 (refine_540, metadata_head); native
// fused_native_fp16_refine_tail_conv_kernel,
// optimized/native/src/neural/srcpyr/SrcPyrNativeFp16Refine.cuh:334-557
// (FP16 operands, FP32 accumulation, FP32 refine bias, FP16-rounded tail bias).
//
// gfx950 mapping: persistent blocks of 8 waves, two per CU (four waves per SIMD, 128 VGPRs), over tiles of 32 x 8
// packed pixels.  All weight fragments (45 KB) and the zero-padded 34 x 10 x 32 FP16 input patch (80-byte pixel
// stride) sit in LDS; a wave runs one row, two 16-pixel MFMA column groups that share each fragment read, and the
// next tile's patch is in flight in registers meanwhile.  The refine accumulators are converted to FP16 and used
// directly as the tail's B operand (the tail's K order is permuted on the host to match the accumulator layout),
// so the 64-channel refine activation never leaves registers.  With the fragments in registers (208 VGPRs, one
// wave per SIMD, no prefetch) nothing hid the latency of loads, LDS and MFMA chains: 32.6 us at 720p, now
// 18.6; its 48 MB take 9.4 us, its MFMAs 4.9.
#include "common.hpp"
#include "kernels.hpp"

namespace aeisu {

constexpr int kRTW = 32, kRTH = 8, kRThreads = 64 * kRTH;
constexpr int kRPW = kRTW + 2, kRPH = kRTH + 2;
constexpr int kRPix = 40;                     // halves per LDS pixel (32 + 8 pad)
constexpr int kRefineFrag = 4 * 9 * 64;       // h8 fragments
constexpr int kTailFrag = 4 * 2 * 64;
constexpr int kROffBias = (kRefineFrag + kTailFrag) * 16, kROffPatch = kROffBias + 512;
constexpr int kRLds = kROffPatch + kRPH * kRPW * kRPix * 2;
constexpr int kRChunks = kRPH * kRPW * 4, kRPer = (kRChunks + kRThreads - 1) / kRThreads;   // 16-byte patch chunks
static_assert(2 * kRLds <= 160 * 1024, "two blocks per CU");

struct RefineTile {
  int b, y0, x0;
};
__device__ __forceinline__ RefineTile refine_tile(int tidx, int tiles_x, int tiles_y) {
  const int b = tidx / (tiles_x * tiles_y), rem = tidx - b * tiles_x * tiles_y, ty = rem / tiles_x;
  return {b, ty * kRTH, (rem - ty * tiles_x) * kRTW};
}
__device__ __forceinline__ void refine_fetch(u4 (&v)[kRPer], const _Float16* __restrict__ work, RefineTile t, int Hq, int Wq,
                                             int tid) {
  const _Float16* in = work + (size_t)t.b * Hq * Wq * 32;
#pragma unroll
  for (int k = 0; k < kRPer; ++k) {
    const int q = tid + kRThreads * k, pix = q >> 2, ch = (q & 3) * 8, ly = pix / kRPW;
    const int gy = t.y0 + ly - 1, gx = t.x0 + pix - ly * kRPW - 1;
    v[k] = u4{0u, 0u, 0u, 0u};
    if (q < kRChunks && (unsigned)gy < (unsigned)Hq && (unsigned)gx < (unsigned)Wq)
      v[k] = *reinterpret_cast<const u4*>(in + ((size_t)gy * Wq + gx) * 32 + ch);
  }
}

__global__ __launch_bounds__(kRThreads, 4) void refine_tail_kernel(
    const _Float16* __restrict__ work, const h8* __restrict__ wfrag, const float* __restrict__ rbias,
    const float* __restrict__ tbias, _Float16* __restrict__ meta, int Hq, int Wq, int batch) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const int n = lane & 15, g = lane >> 4;
  const int tiles_x = (Wq + kRTW - 1) / kRTW, tiles_y = (Hq + kRTH - 1) / kRTH;
  const int num_tiles = batch * tiles_x * tiles_y;
  const int iters = tile_iters(num_tiles);
  int tidx = tile_of(0, num_tiles);
  u4 v[kRPer];
  if (tidx < num_tiles) refine_fetch(v, work, refine_tile(tidx, tiles_x, tiles_y), Hq, Wq, tid);
  {
    const u4* srcw = reinterpret_cast<const u4*>(wfrag);
    u4* dst = reinterpret_cast<u4*>(smem);
    for (int i = tid; i < kRefineFrag + kTailFrag; i += kRThreads) dst[i] = srcw[i];
    float* bias = reinterpret_cast<float*>(smem + kROffBias);
    if (tid < 64) bias[tid] = rbias[tid];
    else if (tid < 128) bias[tid] = tbias[tid - 64];
  }
  const h8* wf = reinterpret_cast<const h8*>(smem) + lane;
  const f4* bias = reinterpret_cast<const f4*>(smem + kROffBias) + g;
  unsigned char* patch = smem + kROffPatch;
  for (int it = 0; it < iters; ++it) {
    if (tidx >= num_tiles) break;                    // block-uniform
    const RefineTile t = refine_tile(tidx, tiles_x, tiles_y);
    if (it) lds_barrier();                           // the last tile's patch reads are done
#pragma unroll
    for (int k = 0; k < kRPer; ++k) {
      const int q = tid + kRThreads * k;
      if (q < kRChunks) *reinterpret_cast<u4*>(patch + ((q >> 2) * kRPix + (q & 3) * 8) * 2) = v[k];
    }
    tidx = tile_of(it + 1, num_tiles);
    if (it + 1 < iters && tidx < num_tiles) refine_fetch(v, work, refine_tile(tidx, tiles_x, tiles_y), Hq, Wq, fresh(tid));
    lds_barrier();                                   // patch (and weights) visible
    const unsigned char* base = patch + ((wave * kRPW + n) * kRPix + 8 * g) * 2;
    f4 acc[4][2];
#pragma unroll
    for (int T = 0; T < 4; ++T) acc[T][0] = acc[T][1] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      h8 bop[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        bop[j] = *reinterpret_cast<const h8*>(base + (((k / 3) * kRPW + k % 3 + 16 * j) * kRPix) * 2);
#pragma unroll
      for (int T = 0; T < 4; ++T) {
        const h8 a = wf[(T * 9 + k) * 64];
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[T][j] = mfma_f16(a, bop[j], acc[T][j]);
      }
    }
    h8 bt[2][2];
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      const f4 rb = bias[4 * T];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) bt[j][T >> 1][(T & 1) * 4 + r] = (_Float16)leaky(acc[T][j][r] + rb[r], 0.1f);
    }
    u2 o[4][2];
#pragma unroll
    for (int T = 0; T < 4; ++T) {
      const h8 t0 = wf[kRefineFrag + (T * 2) * 64], t1 = wf[kRefineFrag + (T * 2 + 1) * 64];
      const f4 tb = bias[16 + 4 * T];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f4 c = mfma_f16(t0, bt[j][0], f4{0.f, 0.f, 0.f, 0.f});
        c = mfma_f16(t1, bt[j][1], c);
        o[T][j] = u2{pack_h2(c[0] + tb[0], c[1] + tb[1]), pack_h2(c[2] + tb[2], c[3] + tb[3])};
      }
    }
#pragma unroll
    for (int k = 0; k < kRPer; ++k) asm volatile("" : "+v"(v[k]));   // the prefetch is waited for before the stores
    const int yq = t.y0 + wave;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int xq = t.x0 + 16 * j + n;
      _Float16* dst = meta + (((size_t)t.b * Hq + yq) * Wq + xq) * 64 + 16 * (g & 1) + 8 * (g >> 1);
#pragma unroll
      for (int T = 0; T < 4; T += 2) {
        // one swap per register pairs tiles T and T + 1 between lane groups 2k and 2k + 1: eight neighbouring
        // channels per lane, one 16-byte store
        unsigned x0 = o[T][j][0], x1 = o[T][j][1], y0 = o[T + 1][j][0], y1 = o[T + 1][j][1];
        permlane16_swap_u(x0, y0);
        permlane16_swap_u(x1, y1);
        if (yq < Hq && xq < Wq) *reinterpret_cast<u4*>(dst + 16 * T) = u4{x0, x1, y0, y1};
      }
    }
  }
}

int refine_num_tiles(int batch, int Hq, int Wq) {
  return batch * ((Hq + kRTH - 1) / kRTH) * ((Wq + kRTW - 1) / kRTW);
}

hipError_t launch_refine_tail(const void* work, const void* wfrag, const float* rbias, const float* tbias,
                              void* meta, int Hq, int Wq, int batch, int grid, hipStream_t stream) {
  hipLaunchKernelGGL(refine_tail_kernel, dim3(grid), dim3(kRThreads), kRLds, stream, (const _Float16*)work,
                     (const h8*)wfrag, rbias, tbias, (_Float16*)meta, Hq, Wq, batch);
  return hipGetLastError();
}

// Allows the kernel's dynamic LDS above the default limit; called once per device.
hipError_t refine_prepare() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&refine_tail_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                             kRLds);
}

int refine_blocks_per_cu() {
  int n = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, refine_tail_kernel, kRThreads, kRLds);
  return e == hipSuccess && n > 0 ? n : 1;
}

}  // namespace aeisu
