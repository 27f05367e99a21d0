// A dense layer's product with a chunk of tokens (17 to a few hundred) on MFMA, straight from the blocks: every type,
// float16 or bfloat16 tokens (strata_mlx/dense.py:234-242, which unpacks the weights and multiplies floats).
//
// out[t, r] = W[r, :] . x[t, :]. A workgroup takes 32 rows and up to four tiles of 16 tokens, its waves the K steps of
// 256 columns in turn: at these sizes the layer is a few megabytes and the launch a few microseconds, so what counts is
// that every CU has rows of its own and every wave loads at once. (Rows dequantized for a library product, as longer
// chunks go, take five launches and write and read the float16 layer: 4096 x 4096 Q4_K at 77 tokens 59 us.) A wave
// decodes its step's rows once for all the tiles, in registers, as prompt_impl.h does, and the waves' partial sums meet
// in LDS at the end.
//
// The tokens come packed by chunk_pack_kernel in the order of the MFMA operands, 1 KB a (tile, step, MFMA), so that a
// wave's loads of them are contiguous: read from the rows as they lie, each load touched 64 cache lines. The same pass
// scales bfloat16 tokens, and those of types with mins, into float16's upper range by a power of two each and adds the
// runs' sums of the types with mins (window_impl.h: each lane its own two runs).
#pragma once
#include "window_impl.h"

namespace strata_chunk {

using strata_mv::DirectTables;
using strata_mv::LaneOffsets;
using strata_mv::RunPair;
using strata_prompt::f16x8;
using strata_prompt::f32x4;
using strata_prompt::kHasMin;
using strata_prompt::kMayPart;
using strata_prompt::kStep;
using strata_prompt::kStepBytes;

constexpr int kMaxWaves = 8;
constexpr int kAhead = 3;      // MFMAs that the packed tokens are loaded ahead of their use
constexpr int kMaxTiles = 4;   // tiles of 16 tokens a workgroup at most

struct ChunkParams {
  const uint8_t* blocks;
  const u32x4* a;         // packed tokens: [tile][step][MFMA][lane]
  const u32x2* sums;      // the types with mins: [tile][step][lane], a word a run
  const uint32_t* a_max;  // scaled tokens: each one's largest magnitude, or null
  void* out;
  int rows, cols, row_bytes, tokens, nsteps;
};

struct PackParams {
  const void* x;
  u32x4* a;
  uint32_t* sums;
  uint32_t* a_max;
  int cols, nsteps;
  int scaled, q6;  // scale the rows; Q6_K's order of runs
};

constexpr int kPackThreads = 256;

// One workgroup a token: its largest magnitude, then its 16-byte pieces (8 columns) scaled into their places; pieces
// past the row (a partial last step) zeros. MIN: the runs' sums, four pieces a run.
template <typename XT, bool MIN>
__global__ __launch_bounds__(kPackThreads) void chunk_pack_kernel(PackParams p) {
  __shared__ uint32_t wmax[kPackThreads / 64];
  const int64_t t = blockIdx.x;
  const u32x4* src = reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(p.x) + t * p.cols);
  const int pieces = p.cols / 8, all = p.nsteps * (kStep / 8);
  int ex = 0;
  if (p.scaled) {
    strata_window::us2 m = strata_window::us2{0, 0};
    for (int c = threadIdx.x; c < pieces; c += kPackThreads) {
      const u32x4 v = src[c];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        m = __builtin_elementwise_max(m, __builtin_bit_cast(strata_window::us2, v[i] & 0x7fff7fffu));
    }
    uint32_t u = max((uint32_t)m[0], (uint32_t)m[1]);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) u = max(u, (uint32_t)__shfl_xor((int)u, d));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = u;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kPackThreads / 64; ++w) u = max(u, wmax[w]);
    u = __float_as_uint(to_f32(__builtin_bit_cast(XT, (uint16_t)u)));
    ex = row_exponent(u);
    if (threadIdx.x == 0) p.a_max[t] = u;
  }
  const int tile = (int)(t >> 4), n = (int)(t & 15);
  for (int c = threadIdx.x; c < all; c += kPackThreads) {  // `all` is a multiple of 32: a run's four threads together
    u32x4 v = c < pieces ? src[c] : u32x4{0u, 0u, 0u, 0u};
    if (p.scaled) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float lo = to_f32(__builtin_bit_cast(XT, (uint16_t)(v[i] & 0xffffu)));
        const float hi = to_f32(__builtin_bit_cast(XT, (uint16_t)(v[i] >> 16)));
        v[i] = strata_window::half_of(__builtin_ldexpf(lo, -ex)) | (strata_window::half_of(__builtin_ldexpf(hi, -ex)) << 16);
      }
    }
    const int step = c / 32, r = (c % 32) / 4, q = c % 4;
    const int g = p.q6 ? 2 * (r >> 2) + (r & 1) : r >> 1, h = p.q6 ? (r >> 1) & 1 : r & 1;
    const int64_t at = (int64_t)tile * p.nsteps + step;
    p.a[(at * 8 + 4 * h + q) * 64 + 16 * g + n] = v;
    if constexpr (MIN) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t w = v[i];  // (a bit cast of a vector's element itself takes the vector's first)
        s = __builtin_amdgcn_fdot2(__builtin_bit_cast(strata_mv::h2_t, w),
                                   __builtin_bit_cast(strata_mv::h2_t, 0x3C003C00u), s, false);
      }
      s += strata_mv::lanes_apart(s, 1);
      s += strata_mv::lanes_apart(s, 2);
      if (q == 0) p.sums[(at * 64 + 16 * g + n) * 2 + h] = strata_window::split_sum(s);
    }
  }
}

// RG groups of 16 rows and NT tiles of 16 tokens a workgroup. STAGED (the dword types, prompt_impl.h): a wave's rows of
// a step come into its LDS slots by direct loads, the next step's once this step's fields are in registers.
template <int KIND, typename OT, int RG, int NT, bool STAGED>
__global__ __launch_bounds__(64 * kMaxWaves, 2) void chunk_kernel(ChunkParams p) {
  __shared__ DirectTables<KIND> tab;
  __shared__ f32x4 red[kMaxWaves][RG * NT][64];
  constexpr int kGL = STAGED ? strata_prompt::kGroupLoads<KIND> : 1;
  constexpr int kGB = 256 * kGL;  // a group's slots
  __shared__ __attribute__((aligned(16))) uint8_t slots[STAGED ? kMaxWaves * RG * kGB : 16];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int row_blocks = (p.rows + 16 * RG - 1) / (16 * RG), tile0 = blockIdx.y * NT;
  const int last_tile = (p.tokens + 15) / 16 - 1;

  const int last_pairs = kMayPart<KIND> ? (p.cols - (p.nsteps - 1) * kStep) / 64 : 4;
  const uint32_t back = (uint32_t)max(0, g - (last_pairs - 1)) * (kStepBytes<KIND> / 4);  // in a partial last step
  const LaneOffsets<KIND> o = strata_mv::lane_offsets<KIND>(g);
  // row block rb's first row as a base; rows past the last block's are the matrix's last row
  auto block_at = [&](int rb) { return p.blocks + (int64_t)rb * (16 * RG) * p.row_bytes; };
  auto load = [&](int rb, int k, RunPair<KIND>(&f)[RG]) {
    const uint32_t at = (uint32_t)k * kStepBytes<KIND> - (kMayPart<KIND> && k == p.nsteps - 1 ? back : 0u);
#pragma unroll
    for (int i = 0; i < RG; ++i) {
      const int row = min(16 * i + n, p.rows - 1 - rb * (16 * RG));
      strata_mv::load_fields<KIND>(block_at(rb), (uint32_t)row * (uint32_t)p.row_bytes + at, o, f[i]);
    }
  };
  uint32_t voff[RG][kGL];
  const uint32_t slot0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)slots + (uint32_t)(wave * RG * kGB));
  if constexpr (STAGED) {
    constexpr int kPitchDw = strata_prompt::kSlotPitch<KIND>;
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int l = 0; l < kGL; ++l) {
        const int c = 64 * l + lane, q = min(c / kPitchDw, 15), d = min(c % kPitchDw, strata_prompt::kSlotDwords<KIND> - 1);
        voff[r][l] = (uint32_t)(16 * r + q) * (uint32_t)p.row_bytes + 4u * (uint32_t)d;
      }
  }
  auto stage = [&](int rb, int k) {
    const uint8_t* base = block_at(rb) + strata_prompt::dword_first<KIND>(k, p.row_bytes);
    const int last = p.rows - 1 - rb * (16 * RG);  // the block's last row
    if (last < 16 * RG - 1) {
#pragma unroll
      for (int r = 0; r < RG; ++r)
#pragma unroll
        for (int l = 0; l < kGL; ++l) {
          const int q = 16 * r + min((64 * l + lane) / strata_prompt::kSlotPitch<KIND>, 15);
          strata_prompt::dma_dword(base, voff[r][l] - (uint32_t)max(0, q - last) * (uint32_t)p.row_bytes,
                                   slot0 + (uint32_t)(r * kGB + 256 * l));
        }
    } else {
#pragma unroll
      for (int r = 0; r < RG; ++r)
#pragma unroll
        for (int l = 0; l < kGL; ++l) strata_prompt::dma_dword(base, voff[r][l], slot0 + (uint32_t)(r * kGB + 256 * l));
    }
  };
  const u32x4* at[NT];  // tile i's operands of step 0 (past the last tile: the last again, written nowhere)
  const u32x2* sat[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int64_t t = min(tile0 + i, last_tile);
    at[i] = p.a + t * p.nsteps * (8 * 64) + lane;
    sat[i] = p.sums + t * p.nsteps * 64 + lane;
  }
  u32x4 a[kAhead + 1][NT];
  auto load_a = [&](int k, int m, u32x4(&dst)[NT]) {
#pragma unroll
    for (int i = 0; i < NT; ++i) dst[i] = at[i][(k * 8 + m) * 64];
  };
  int k = wave, rb = blockIdx.x;
  RunPair<KIND> f[RG];
  if constexpr (STAGED)
    stage(rb, k);
  else
    load(rb, k, f);
#pragma unroll
  for (int m = 0; m < kAhead; ++m) load_a(k, m, a[m]);
  for (int i = tid; i < 256; i += blockDim.x) {  // the tables
    strata_mv::TableFetch<KIND> tf;
    strata_mv::fetch_tables<KIND>(tf, i);
    strata_mv::store_tables<KIND>(tab, tf, i);
  }
  auto write = [&](int b) {
    for (int c = wave; c < RG * NT; c += waves) {  // one (row group, tile) a wave: lane (n, g) row n, tokens 4 g + j
      f32x4 t = red[0][c][lane];
#pragma unroll
      for (int w = 1; w < kMaxWaves; ++w) {
        if (w < waves) {
          const f32x4 v = red[w][c][lane];
#pragma unroll
          for (int j = 0; j < 4; ++j) t[j] += v[j];
        }
      }
      const int row = b * (16 * RG) + 16 * (c / NT) + n;
      if (row >= p.rows) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int token = (tile0 + c % NT) * 16 + 4 * g + j;
        if (token >= p.tokens) continue;
        const float v = p.a_max != nullptr ? __builtin_ldexpf(t[j], row_exponent(p.a_max[token])) : t[j];
        reinterpret_cast<OT*>(p.out)[(int64_t)token * p.rows + row] = from_f32<OT>(v);
      }
    }
  };
  f32x4 acc[RG][NT];
#pragma unroll
  for (int r = 0; r < RG; ++r)
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  strata_prompt::lds_barrier();  // the tables are written; the loads stay in flight

  for (;;) {
    // the wave's next step: of this row block, or the first of the workgroup's next one
    const bool done = k + waves >= p.nsteps;
    const int next = done ? wave : k + waves, nrb = done ? rb + gridDim.x : rb;
    const bool more = nrb < row_blocks;
    RunPair<KIND> fn[STAGED ? 1 : RG];
    if constexpr (STAGED) {
      strata_prompt::wait_loads();
      const uint32_t off = (uint32_t)(k * kStepBytes<KIND>) - strata_prompt::dword_first<KIND>(k, p.row_bytes);
      const int gl = kMayPart<KIND> && k == p.nsteps - 1 ? min(g, last_pairs - 1) : g;
#pragma unroll
      for (int r = 0; r < RG; ++r)
        strata_prompt::dword_fields<KIND>(slots + (wave * RG + r) * kGB + 4 * strata_prompt::kSlotPitch<KIND> * n, off,
                                          gl, f[r]);
      if (more) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        stage(nrb, next);
      }
    } else {
      load(more ? nrb : rb, next, fn);
    }
    f32x4 part[RG][NT];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int i = 0; i < NT; ++i) part[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x2 sm[NT];
    if constexpr (kHasMin<KIND>) {
#pragma unroll
      for (int i = 0; i < NT; ++i) sm[i] = sat[i][k * 64];
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {  // MFMA m: run m / 4's weights 8 (m % 4) ..
      load_a(m + kAhead < 8 ? k : next, (m + kAhead) % 8, a[(m + kAhead) % (kAhead + 1)]);
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        uint32_t w[4];
        strata_prompt::decode_folded4<KIND>(f[r], m >> 2, g, m & 3, w, tab);
        const f16x8 b = __builtin_bit_cast(f16x8, u32x4{w[0], w[1], w[2], w[3]});
#pragma unroll
        for (int i = 0; i < NT; ++i)
          part[r][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[m % (kAhead + 1)][i]), b, part[r][i], 0,
                                                              0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      const float d = strata_prompt::step_scale<KIND>(f[r]);
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[r][i][j] = __builtin_fmaf(d, part[r][i][j], acc[r][i][j]);
      if constexpr (kHasMin<KIND>) {
        const f16x8 b = strata_window::own_mins<KIND>(f[r], g);
        const float dm = strata_prompt::kSumScale * strata_mv::half_bits(f[r].dd >> 16);
        const f32x4 z = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const f32x4 mm = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(f16x8, u32x4{sm[i][0], sm[i][1], 0u, 0u}), b, z, 0, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[r][i][j] = __builtin_fmaf(-dm, mm[j], acc[r][i][j]);
        }
      }
    }
    if constexpr (!STAGED) {
#pragma unroll
      for (int r = 0; r < RG; ++r) f[r] = fn[r];
    }
    if (done) {  // the row block's sums: the waves' parts meet in LDS
      if (rb != (int)blockIdx.x) strata_prompt::lds_barrier();  // the last block's parts have been read
#pragma unroll
      for (int r = 0; r < RG; ++r)
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          red[wave][r * NT + i][lane] = acc[r][i];
          acc[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      strata_prompt::lds_barrier();
      write(rb);
      if (!more) break;
    }
    k = next;
    rb = nrb;
  }
}

// Bytes of workspace: the packed tokens, the sums, the tokens' largest magnitudes.
inline int64_t chunk_workspace(int64_t tokens, int64_t cols) {
  const int64_t tiles = (tokens + 15) / 16, nsteps = (cols + kStep - 1) / kStep;
  return tiles * nsteps * (8 * 64 * 16 + 64 * 8) + tokens * 4;
}

template <int KIND, typename OT>
int launch_chunk(ChunkParams& p, const void* x, void* workspace, hipStream_t s) {
  const int tiles = (p.tokens + 15) / 16;
  PackParams q = {};
  q.x = x;
  q.a = reinterpret_cast<u32x4*>(workspace);
  q.sums = reinterpret_cast<uint32_t*>(q.a + (int64_t)tiles * p.nsteps * (8 * 64));
  q.a_max = q.sums + (int64_t)tiles * p.nsteps * (64 * 2);
  q.cols = p.cols;
  q.nsteps = p.nsteps;
  q.scaled = std::is_same<OT, bf16_t>::value || kHasMin<KIND>;
  q.q6 = KIND == K_Q6_K;
  p.a = q.a;
  p.sums = reinterpret_cast<const u32x2*>(q.sums);
  p.a_max = q.scaled ? q.a_max : nullptr;
  hipLaunchKernelGGL((chunk_pack_kernel<OT, kHasMin<KIND>>), dim3((unsigned)p.tokens), dim3(kPackThreads), 0, s, q);
  STRATA_CHECK_LAUNCH();
  const int rounds = (p.nsteps + kMaxWaves - 1) / kMaxWaves, waves = (p.nsteps + rounds - 1) / rounds;
  const int blocks = (tiles + kMaxTiles - 1) / kMaxTiles, nt = (tiles + blocks - 1) / blocks;
  const int token_blocks = (tiles + nt - 1) / nt;
  if (token_blocks > 65535) return STRATA_ERR_SHAPE;
  const dim3 block(64 * waves);
  // staged rows: whole dwords, rows of a slot or more
  const bool staged = p.row_bytes % 4 == 0 && ((uintptr_t)p.blocks & 3) == 0 &&
                      p.row_bytes >= 4 * strata_prompt::kSlotDwords<KIND>;
  auto go = [&](auto rg, auto ntc) {
    constexpr int RG = decltype(rg)::value, NT = decltype(ntc)::value;
    // one workgroup a CU, which goes on to its next row block: its rows are asked for before the last one's sums meet
    const int blocks_x = (p.rows + 16 * RG - 1) / (16 * RG);
    const dim3 grid((unsigned)min(blocks_x, max(1, strata_mv::device_cus() / token_blocks)), (unsigned)token_blocks);
    if constexpr (strata_prompt::kDwordRows<KIND>) {
      if (staged) {
        hipLaunchKernelGGL((chunk_kernel<KIND, OT, RG, NT, true>), grid, block, 0, s, p);
        return;
      }
    }
    hipLaunchKernelGGL((chunk_kernel<KIND, OT, RG, NT, false>), grid, block, 0, s, p);
  };
  auto by_nt = [&](auto rg) {
    switch (nt) {
      case 1:
      case 2: go(rg, std::integral_constant<int, 2>()); break;
      case 3: go(rg, std::integral_constant<int, 3>()); break;
      default: go(rg, std::integral_constant<int, 4>()); break;
    }
  };
  // 16 rows a workgroup where 32 would leave CUs without one
  if ((int64_t)((p.rows + 31) / 32) * token_blocks < strata_mv::device_cus())
    by_nt(std::integral_constant<int, 1>());
  else
    by_nt(std::integral_constant<int, 2>());
  STRATA_CHECK_LAUNCH();
  return STRATA_OK;
}

}  // namespace strata_chunk
