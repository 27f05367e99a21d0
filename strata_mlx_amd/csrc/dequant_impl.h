// Dequant to float16 of the dense types (Q4_K, Q5_K, Q6_K, Q8_0): what a long chunk's library product reads
// (strata_mlx/dense.py:234-241). A thread takes a run pair (64 weights) with the matvecs' field loads, its codes become
// float32 byte by byte (one conversion instruction each) and give each weight, the exact float32 value that
// strata_unpack32 gives (the products fit 24 bits; Q4_K's and Q5_K's fma is the one rounding there too), rounded once to
// float16. dequant_kernel, a byte load a code, took 47 us for 12288 x 4096 of Q6_K (41 MB in, 101 MB out: 28 us at a
// large copy's rate; its stores, 16 bytes a lane at 64-byte steps, made contiguous through LDS here) and 40 us for as much
// of Q4_K; this 24 and 21.
#pragma once
#include "direct_impl.h"

namespace strata_mv {

template <int KIND>
constexpr bool kFastDequant = KIND == K_Q4_K || KIND == K_Q5_K || KIND == K_Q6_K || KIND == K_Q8_0;

// Four codes (bytes of c) as weights, two float16 pairs: code * a + b in one fma, or (SIGNED) (code + b) * a, whose zero
// code keeps the sign of a. v_cvt_f16_f32 keeps subnormals, and written out it is not
// fused into packed conversions that do not.
template <bool SIGNED>
__device__ __forceinline__ void codes_to_half(uint32_t c, float a, float b, uint32_t* w) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float c0 = (float)((c >> (16 * i)) & 255u), c1 = (float)((c >> (16 * i + 8)) & 255u);
    const float lo = SIGNED ? (c0 + b) * a : __builtin_fmaf(c0, a, b);
    const float hi = SIGNED ? (c1 + b) * a : __builtin_fmaf(c1, a, b);
    uint32_t l, h;
    asm("v_cvt_f16_f32 %0, %1" : "=v"(l) : "v"(lo));
    asm("v_cvt_f16_f32 %0, %1" : "=v"(h) : "v"(hi));
    w[i] = (l & 0xffffu) | (h << 16);
  }
}

template <int KIND>
__global__ __launch_bounds__(256) void dequant_half_kernel(const uint8_t* blocks, int64_t pairs_total, uint32_t per_row,
                                                           int row_bytes, f16* out) {
  __shared__ u32x4 turn[4][512];  // a wave's 64 run pairs: their results' 16-byte pieces in order, turned within eights
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t u0 = (int64_t)blockIdx.x * 256 + 64 * wave;
  const int64_t u = min(u0 + lane, pairs_total - 1);  // past the last: the last again, written nowhere
  const int64_t row = u / per_row;
  const int j = (int)(u - row * per_row);
  RunPair<KIND> f;
  load_fields<KIND>(blocks + row * row_bytes, 0u, lane_offsets<KIND>(j), f);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    uint32_t w[16];
    if constexpr (KIND == K_Q8_0) {
      const float d = half_bits(h ? f.d[1] : f.d[0]);
#pragma unroll
      for (int i = 0; i < 8; ++i) codes_to_half<true>(f.q[2 * h + i / 4][i % 4] ^ 0x80808080u, d, -128.0f, w + 2 * i);
    } else if constexpr (KIND == K_Q6_K) {
      const int r2 = 2 * ((j & 1) + 2 * h);
      const uint32_t sc = h ? f.sc[1] : f.sc[0];
      const float d = half_bits(f.d), s0 = d * (float)(int8_t)(sc & 255), s1 = d * (float)(int8_t)(sc >> 8);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t lo = (f.ql[i / 4][i % 4] >> (4 * h)) & 0x0F0F0F0Fu;
        const uint32_t hb = (f.qh[i / 4][i % 4] >> r2) & 0x03030303u;
        const float s = i < 4 ? s0 : s1;
        codes_to_half<true>(lo | (hb << 4), s, -32.0f, w + 2 * i);
      }
    } else {
      const int sb = 2 * (j & 3) + h, tb = 8 * (sb & 3);
      const uint32_t b0 = (f.sm[0] >> tb) & 255, b1 = (f.sm[1] >> tb) & 255, b2 = (f.sm[2] >> tb) & 255;
      const uint32_t sc = sb >= 4 ? ((b2 & 15) | ((b0 >> 6) << 4)) : (b0 & 63);
      const uint32_t mn = sb >= 4 ? ((b2 >> 4) | ((b1 >> 6) << 4)) : (b1 & 63);
      const float scale = half_bits(f.dd & 0xffff) * (float)sc, bias = -(half_bits(f.dd >> 16) * (float)mn);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        uint32_t c = (f.qs[i / 4][i % 4] >> (4 * h)) & 0x0F0F0F0Fu;
        if constexpr (KIND == K_Q5_K) c |= ((f.qh[i / 4][i % 4] >> sb) & 0x01010101u) << 4;
        codes_to_half<false>(c, scale, bias, w + 2 * i);
      }
    }
    const int run = run_of<KIND>(lane, h);  // among the wave's (a row is whole blocks: four lanes a block)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c = 4 * run + v;
      turn[wave][c ^ ((c >> 3) & 7)] = u32x4{w[4 * v], w[4 * v + 1], w[4 * v + 2], w[4 * v + 3]};
    }
  }
  __builtin_amdgcn_wave_barrier();  // the wave's own pieces: its LDS operations are in order
  u32x4* o = reinterpret_cast<u32x4*>(out) + u0 * 8;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = 64 * i + lane;
    if (u0 * 8 + c < pairs_total * 8) o[c] = turn[wave][c ^ ((c >> 3) & 7)];
  }
}

// Whole run pairs a row, results at a 16-byte boundary.
template <int KIND>
int launch_dequant_any(const uint8_t* blocks, int64_t runs_total, int runs_per_row, int row_bytes, void* out,
                       int out_dtype, hipStream_t s) {
  if constexpr (kFastDequant<KIND>) {
    const int64_t groups = (runs_total / 2 + 255) / 256;
    if (out_dtype == DT_F16 && runs_per_row % 2 == 0 && ((uintptr_t)out & 15) == 0 && groups <= INT32_MAX) {
      hipLaunchKernelGGL((dequant_half_kernel<KIND>), dim3((unsigned)groups), dim3(256), 0, s, blocks, runs_total / 2,
                         (uint32_t)(runs_per_row / 2), row_bytes, (f16*)out);
      STRATA_CHECK_LAUNCH();
      return STRATA_OK;
    }
  }
  return launch_dequant_kind<KIND>(blocks, runs_total, runs_per_row, row_bytes, out, out_dtype, s);
}

}  // namespace strata_mv
