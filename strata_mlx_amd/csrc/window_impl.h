// A dense layer's product with a window of up to 16 tokens on MFMA: every block type, float16 or bfloat16 tokens, rows
// of at most 4096 inputs (strata_mlx/blocks.py:383-394, dense.py:205-242).
//
// out[t, r] = W[r, :] . x[t, :]. The rows are read and decoded once for all tokens: bound by HBM, where the matvecs
// decode a row again for each token (an lm_head of 151936 x 4096 Q6_K at five tokens 301 -> 114 us; 93-101 is its 510 MB
// at a large copy's rate; Q4_K 319 -> 81, Q8_0 410 -> 118; Q6_K 4096 x 4096 15.4 -> 9.6 us).
//
// The K steps (256 columns) are split over a workgroup's waves, up to eight of them, SPW = 1 or 2 steps each: a wave
// keeps its steps' activations of all 16 slots in registers, as MFMA operands, for the whole launch (32 registers a
// step), and streams its part of every row group (16 rows) of the workgroup: lane (n, g) holds the fields of one run
// pair of row n a step, as in prompt_impl.h, loaded a row group ahead. A group's partial sums (16 rows x 16 slots a
// wave) meet in LDS, one barrier a group and one wave adding them, the waves in turn; two buffers, so that the others
// go on with the next group meanwhile.
//
// Staged rows (Q4_K, Q6_K, Q8_0, Q4_0, Q5_0 and IQ4_NL rows of a multiple of 16 bytes; kStagedRows). Read straight into registers, a wave's
// field loads touch the cache lines of 16 rows each and one row group is in flight: the texture units, not HBM, set
// the pace (lm_head 183 us; staged, and with inexact weights, 111). Staged, a wave's part of a row group comes by contiguous 16-byte direct loads
// (global_load_lds_dwordx4) into one of its two slabs, and the fields are read from there into registers, after which
// the slab takes the group after next: two groups in flight all along. A slab's row pitch is an odd number of 16-byte
// pieces, so that the 16 rows' reads spread over the banks.
//
// The weights are exact: the types whose folded weights need more than 11 bits (kInexact) multiply them in two float16
// parts, the second what rounding the first left, at two MFMAs for one (the matrix cores have the time).
//
// bfloat16 tokens, and the tokens of types with mins, are scaled by a power of two each into float16's upper range
// (as strata_rows_to_f16 scales them) once, in the registers: a token's largest magnitude over its lanes and waves.
// The mins' product takes, as its K order, each lane's own two runs: their sums' high and low parts against the runs'
// mins, one MFMA a step.
#pragma once
#include "prompt_impl.h"

namespace strata_window {

using strata_mv::DirectTables;
using strata_mv::LaneOffsets;
using strata_mv::RunPair;
using strata_prompt::f16x8;
using strata_prompt::f32x4;
using strata_prompt::h2v;
using strata_prompt::kHasMin;
using strata_prompt::kMayPart;
using strata_prompt::kStep;
using strata_prompt::kStepBytes;

typedef unsigned short us2 __attribute__((ext_vector_type(2)));

constexpr int kSlots = 16;         // tokens at most
constexpr int kMaxWaves = 8;       // waves a workgroup at most
constexpr int kMaxCols = 4096;     // two steps a wave

struct WindowParams {
  const uint8_t* blocks;  // src_rows x row_bytes
  const void* x;          // tokens x cols
  void* out;              // tokens x rows
  const uint32_t* ids;    // the rows to compute (an id past the matrix reads row 0 and writes NaN), or null: all
  int rows, src_rows, cols, row_bytes, tokens;
};

// float32 -> float16 to nearest even, subnormals included: the one conversion instruction, which the compiler cannot
// fuse into a packed one that flushes them.
__device__ __forceinline__ uint32_t half_of(float v) {
  uint32_t r;
  asm("v_cvt_f16_f32 %0, %1" : "=v"(r) : "v"(v));
  return r & 0xffffu;
}

// A lane's run sum as the min product takes it: its high part and what that leaves, over kSumScale.
__device__ __forceinline__ uint32_t split_sum(float s) {
  const float v = s * (1.0f / strata_prompt::kSumScale);
  const uint32_t hi = half_of(v);
  return hi | (half_of(v - half_bits_to_f32(hi)) << 16);
}

// The mins' side of a step's min product: lane (n, g)'s two runs' mins of row n, against their sums' two parts each.
template <int KIND>
__device__ __forceinline__ f16x8 own_mins(const RunPair<KIND>& f, int g) {
  uint32_t mn[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int sb = 2 * g + h, tb = 8 * (sb & 3);
    const uint32_t b1 = (f.sm[1] >> tb) & 255, b2 = (f.sm[2] >> tb) & 255;
    const uint32_t v = sb >= 4 ? ((b2 >> 4) | ((b1 >> 6) << 4)) : (b1 & 63);
    mn[h] = __builtin_bit_cast(uint32_t, strata_prompt::both((int)v));
  }
  return __builtin_bit_cast(f16x8, u32x4{mn[0], mn[1], 0u, 0u});
}

// The tokens of a workgroup's slots into float16's upper range, each by a power of two (exact down to 2^-31 of its
// largest), in the registers of the waves that hold them: a slot's largest magnitude over its lanes and waves (peak).
// ex_out: the exponents of the slots that the lane writes; sums: the lane's run sums (the types with mins).
template <int KIND, typename XT, int SPW>
__device__ __forceinline__ void scale_tokens(u32x4 (&a)[SPW][2][4], uint32_t (&sums)[SPW][2], int (&ex_out)[4],
                                             uint32_t (*peak)[kSlots], int wave, int waves, int n, int g) {
  us2 m = us2{0, 0};  // magnitudes compare as their bits do
#pragma unroll
  for (int s = 0; s < SPW; ++s)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          m = __builtin_elementwise_max(m, __builtin_bit_cast(us2, a[s][h][q][c] & 0x7fff7fffu));
  uint32_t u = max((uint32_t)m[0], (uint32_t)m[1]);
  u = max(u, (uint32_t)__shfl_xor((int)u, 16));
  u = max(u, (uint32_t)__shfl_xor((int)u, 32));
  if (g == 0) peak[wave][n] = u;
  __syncthreads();
  auto exponent = [&](int slot) {
    uint32_t v = 0;
#pragma unroll
    for (int w = 0; w < kMaxWaves; ++w) v = max(v, w < waves ? peak[w][slot] : 0u);
    return row_exponent(__float_as_uint(to_f32(__builtin_bit_cast(XT, (uint16_t)v))));
  };
  const int ex = exponent(n);
#pragma unroll
  for (int j = 0; j < 4; ++j) ex_out[j] = exponent(4 * g + j);
  // float16 tokens by three powers of two (2^38 at most together, 2^15 each), each product exact
  const int e1 = min(-ex, 15), e2 = min(-ex - e1, 15), e3 = -ex - e1 - e2;
  const f16 b1 = (f16)__builtin_ldexpf(1.0f, e1), b2 = (f16)__builtin_ldexpf(1.0f, e2), b3 = (f16)__builtin_ldexpf(1.0f, e3);
#pragma unroll
  for (int s = 0; s < SPW; ++s) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float sum = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t v = a[s][h][q][c];
          uint32_t w;
          if constexpr (std::is_same<XT, bf16_t>::value) {  // exact down to 2^-31 of the token's largest
            w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(
                                                 __builtin_ldexpf(__uint_as_float(v << 16), -ex),
                                                 __builtin_ldexpf(__uint_as_float(v & 0xffff0000u), -ex)));
          } else {
            w = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2v, v) * h2v{b1, b1} * h2v{b2, b2} * h2v{b3, b3});
          }
          a[s][h][q][c] = w;
          if constexpr (kHasMin<KIND>)
            sum = __builtin_amdgcn_fdot2(__builtin_bit_cast(strata_mv::h2_t, w),
                                         __builtin_bit_cast(strata_mv::h2_t, 0x3C003C00u), sum, false);
        }
      if constexpr (kHasMin<KIND>) sums[s][h] = split_sum(sum);
    }
  }
}

// One K step's products added to acc: the step's fields against the lane's operands of it.
template <int KIND>
__device__ __forceinline__ void add_step(const RunPair<KIND>& f, const u32x4 (&a)[2][4], const uint32_t (&sums)[2], int g,
                                         const DirectTables<KIND>& tab, f32x4& acc) {
  f32x4 part = f32x4{0.f, 0.f, 0.f, 0.f};
  auto run = [&](auto hc) {  // run h a constant from the start: the fields' pairs indexed by it stay in registers
    constexpr int h = decltype(hc)::value;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t w[4], lo[4];
      if constexpr (strata_prompt::kInexact<KIND>)
        strata_prompt::decode_linear4<KIND, true>(f, h, g, q, w, lo, tab);
      else
        strata_prompt::decode_folded4<KIND>(f, h, g, q, w, tab);
      part = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[h][q]),
                                                    __builtin_bit_cast(f16x8, u32x4{w[0], w[1], w[2], w[3]}), part, 0, 0, 0);
      if constexpr (strata_prompt::kInexact<KIND>)
        part = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[h][q]),
                                                      __builtin_bit_cast(f16x8, u32x4{lo[0], lo[1], lo[2], lo[3]}), part,
                                                      0, 0, 0);
    }
  };
  run(std::integral_constant<int, 0>());
  run(std::integral_constant<int, 1>());
  const float d = strata_prompt::step_scale<KIND>(f);
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = __builtin_fmaf(d, part[j], acc[j]);
  if constexpr (kHasMin<KIND>) {
    const f32x4 z = f32x4{0.f, 0.f, 0.f, 0.f};
    const f32x4 mm = __builtin_amdgcn_mfma_f32_16x16x32_f16(
        __builtin_bit_cast(f16x8, u32x4{sums[0], sums[1], 0u, 0u}), own_mins<KIND>(f, g), z, 0, 0, 0);
    const float dm = strata_prompt::kSumScale * strata_mv::half_bits(f.dd >> 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = __builtin_fmaf(-dm, mm[j], acc[j]);
  }
}

template <int KIND>
constexpr bool kStagedRows = KIND == K_Q4_K || KIND == K_Q6_K || KIND == K_Q8_0 || KIND == K_IQ4_NL || KIND == K_Q4_0 ||
                             KIND == K_Q5_0;
// 16-byte pieces of a wave's part of a row, from the aligned one that holds its first byte (an even one), and the pitch
template <int KIND, int SPW>
constexpr int kPieces = (SPW * kStepBytes<KIND>) % 16 == 0 ? SPW * kStepBytes<KIND> / 16
                                                           : (14 + SPW * kStepBytes<KIND> + 15) / 16;
template <int KIND, int SPW>
constexpr int kPitch = kPieces<KIND, SPW> | 1;
template <int KIND, int SPW>
constexpr int kSlabLoads = (16 * kPitch<KIND, SPW> + 63) / 64;

// lane l's 16 bytes at base + voff into LDS at lds + 16 l (M0 as in dma_dword); NT: the non-temporal cache policy
template <bool NT>
__device__ __forceinline__ void dma_x4(const uint8_t* base, uint32_t voff, uint32_t lds) {
  uint32_t saved;
  if constexpr (NT)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3 nt\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "s"(lds), "v"(voff), "s"(base)
                 : "memory");
  else
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "s"(lds), "v"(voff), "s"(base)
                 : "memory");
}

// run pair g's fields of a step that starts at byte `off` of LDS (the types of 16-byte steps: a multiple of 16)
template <int KIND>
__device__ __forceinline__ void staged_fields(const uint8_t* lds, uint32_t off, int g, RunPair<KIND>& f) {
  typedef strata_prompt::u32x4a16 u32x4a;
  if constexpr (KIND == K_Q4_K) {
    const u32x4a h = strata_prompt::lds_at<u32x4a>(lds, off);
    f.dd = h[0];
    f.sm = u32x4{h[1], h[2], h[3], 0u};
#pragma unroll
    for (int i = 0; i < 2; ++i) f.qs[i] = strata_prompt::lds_at<u32x4a>(lds, off + 16 + 32 * g + 16 * i);
  } else {
    strata_prompt::dword_fields<KIND>(lds, off, g, f);
  }
}

template <int KIND, typename XT, int SPW, bool STAGED, bool NT>
__global__ __launch_bounds__(64 * kMaxWaves, 2) void window_kernel(WindowParams p) {
  constexpr bool kScaled = std::is_same<XT, bf16_t>::value || kHasMin<KIND>;
  __shared__ DirectTables<KIND> tab;
  __shared__ f32x4 red[2][kMaxWaves][64];
  __shared__ uint32_t peak[kMaxWaves][kSlots];
  constexpr int kSlab = STAGED ? 16 * 16 * kPitch<KIND, SPW> : 16;  // bytes
  __shared__ __attribute__((aligned(16))) uint8_t slabs[STAGED ? kMaxWaves * 2 * kSlab : 16];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  {
    strata_mv::TableFetch<KIND> tf;
    const int t = min(tid, 255);
    if (blockDim.x >= 256) {
      strata_mv::fetch_tables<KIND>(tf, t);
      if (tid < 256) strata_mv::store_tables<KIND>(tab, tf, t);
    } else {  // fewer threads than the tables' entries of a pass
      for (int i = tid; i < 256; i += blockDim.x) {
        strata_mv::fetch_tables<KIND>(tf, i);
        strata_mv::store_tables<KIND>(tab, tf, i);
      }
    }
  }

  // the wave's steps; past the row's last step, the last again with zero activations
  const int nsteps = (p.cols + kStep - 1) / kStep;
  const int last_pairs = kMayPart<KIND> ? (p.cols - (nsteps - 1) * kStep) / 64 : 4;
  const LaneOffsets<KIND> o = strata_mv::lane_offsets<KIND>(g);
  uint32_t at[SPW];  // the lane's byte offset in a row

  // STAGED: the lane's piece of each load of a slab (row, piece) as an offset from the row group, and its loads
  const uint32_t part0 = (uint32_t)(wave * SPW) * kStepBytes<KIND>;  // the wave's part of a row
  const int groups = (p.rows + 15) / 16;
  constexpr int kLoads = STAGED ? kSlabLoads<KIND, SPW> : 1;
  uint32_t voff[kLoads];
  const uint32_t slab0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)slabs + (uint32_t)(wave * 2 * kSlab));
  auto stage = [&](int i, int which) {
    if constexpr (STAGED) {
      if (i >= groups) return;  // nothing to ask for past the last group
      const uint8_t* base = p.blocks + (int64_t)i * 16 * p.row_bytes;
      if (16 * i + 16 > p.rows) {  // the last group, cut short: rows past the matrix read its last
#pragma unroll
        for (int l = 0; l < kLoads; ++l) {
          const int c = 64 * l + lane, r = c / kPitch<KIND, SPW>;
          const uint32_t past = (uint32_t)max(0, r - (p.rows - 1 - 16 * i)) * (uint32_t)p.row_bytes;
          if (c < 16 * kPitch<KIND, SPW>) dma_x4<NT>(base, voff[l] - past, slab0 + (uint32_t)(which * kSlab + 1024 * l));
        }
      } else {
#pragma unroll
        for (int l = 0; l < kLoads; ++l)
          if (64 * l + lane < 16 * kPitch<KIND, SPW>)
            dma_x4<NT>(base, voff[l], slab0 + (uint32_t)(which * kSlab + 1024 * l));
      }
    }
  };
  if constexpr (STAGED) {
    const uint32_t first = part0 & ~15u;
    const int pieces = (int)min((uint32_t)kPieces<KIND, SPW>, ((uint32_t)p.row_bytes - first) / 16);
#pragma unroll
    for (int l = 0; l < kLoads; ++l) {
      const int c = 64 * l + lane;
      voff[l] = (uint32_t)(c / kPitch<KIND, SPW>) * (uint32_t)p.row_bytes + first +
                16u * (uint32_t)min(c % kPitch<KIND, SPW>, pieces - 1);
    }
    stage(blockIdx.x, 0);
  }
  u32x4 a[SPW][2][4];
#pragma unroll
  for (int s = 0; s < SPW; ++s) {
    const int k = wave * SPW + s, kc = min(k, nsteps - 1);
    const int gl = kc == nsteps - 1 ? min(g, last_pairs - 1) : g;  // a run pair past the row's: its last
    at[s] = (uint32_t)kc * kStepBytes<KIND> - (uint32_t)(g - gl) * (kStepBytes<KIND> / 4);
    if constexpr (STAGED) at[s] = (uint32_t)kc * kStepBytes<KIND> - (part0 & ~15u);  // the step's place in a slot
    const bool live = k == kc && gl == g && n < p.tokens;
    const uint16_t* row = reinterpret_cast<const uint16_t*>(p.x) + (int64_t)min(n, p.tokens - 1) * p.cols + kc * kStep;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(row + strata_prompt::a_col<KIND>(gl, h, q));
        a[s][h][q] = live ? v : u32x4{0u, 0u, 0u, 0u};
      }
  }

  // row group i's fields of the wave's steps
  RunPair<KIND> f[SPW];
  auto load = [&](int i, RunPair<KIND>(&dst)[SPW]) {
    const uint8_t* base = p.blocks;
    uint32_t row = 0;
    if (p.ids == nullptr) {
      base += (int64_t)i * 16 * p.row_bytes;
      row = (uint32_t)min(n, p.rows - 1 - 16 * i) * (uint32_t)p.row_bytes;
    } else {
      const uint32_t id = p.ids[min(16 * i + n, p.rows - 1)];
      row = (id < (uint32_t)p.src_rows ? id : 0u) * (uint32_t)p.row_bytes;
    }
#pragma unroll
    for (int s = 0; s < SPW; ++s) strata_mv::load_fields<KIND>(base, row + at[s], o, dst[s]);
  };
  int i = blockIdx.x;
  if constexpr (STAGED)
    stage(i + gridDim.x, 1);
  else
    load(i, f);

  // the tokens into float16's upper range, and the types with mins' sums
  uint32_t sums[SPW][2];
  int ex_out[4] = {0, 0, 0, 0};  // the exponents of the slots the lane writes
  if constexpr (kScaled) {
    scale_tokens<KIND, XT, SPW>(a, sums, ex_out, peak, wave, waves, n, g);
  }
  __syncthreads();  // the tables

  for (int it = 0; i < groups; ++it) {
    const int next = i + gridDim.x;
    RunPair<KIND> fn[STAGED ? 1 : SPW];
    if constexpr (STAGED) {  // this group's loads are in (the next one's may be in flight); its fields, then the slab
      constexpr int kNext = kLoads;
      if (next < groups)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kNext) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const uint8_t* slot = slabs + (wave * 2 + (it & 1)) * kSlab + 16 * kPitch<KIND, SPW> * n;
#pragma unroll
      for (int s = 0; s < SPW; ++s) staged_fields<KIND>(slot, at[s], g, f[s]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      stage(i + 2 * gridDim.x, it & 1);
    } else {
      load(next < groups ? next : i, fn);
    }
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < SPW; ++s) add_step<KIND>(f[s], a[s], sums[s], g, tab, acc);
    f32x4(*buf)[64] = red[it & 1];
    buf[wave][lane] = acc;
    strata_prompt::lds_barrier();  // waits for LDS only: the next group's fields stay in flight
    if (wave == it % waves) {      // lane (n, g): row n, slots 4 g + j
      f32x4 t = buf[0][lane];
#pragma unroll
      for (int w = 1; w < kMaxWaves; ++w) {
        if (w < waves) {
          const f32x4 v = buf[w][lane];
#pragma unroll
          for (int j = 0; j < 4; ++j) t[j] += v[j];
        }
      }
      const int r = 16 * i + n;
      if (r < p.rows) {
        const bool past = p.ids != nullptr && p.ids[r] >= (uint32_t)p.src_rows;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int slot = 4 * g + j;
          if (slot >= p.tokens) continue;
          const float v = kScaled ? __builtin_ldexpf(t[j], ex_out[j]) : t[j];
          reinterpret_cast<XT*>(p.out)[(int64_t)slot * p.rows + r] = from_f32<XT>(past ? __builtin_nanf("") : v);
        }
      }
    }
    if constexpr (!STAGED) {
#pragma unroll
      for (int s = 0; s < SPW; ++s) f[s] = fn[s];
    }
    i = next;
  }
}

constexpr int kMinRows = 512;  // (float16) rows below which the matvecs keep a window

// Whether window_kernel takes a dense product: up to 16 tokens whose rows lie at 16-byte boundaries, rows of whole
// run pairs (whole steps in the types with blocks of 256) and at most 4096 inputs; listed rows where the matrix's
// byte offsets fit 32 bits.
// A float16 layer of fewer than 512 rows, at most 32 row groups, stays on the matvecs, which spread it over more CUs (two
// tokens of Q8_0 64 x 2048 5.8 against 6.0 us) and give a token the bits it has alone.
inline bool window_takes(int kind, const WindowParams& p, bool f16_tokens) {
  return (!f16_tokens || p.src_rows >= kMinRows) && strata_prompt::tiles_take(kind, p.cols) && p.cols <= kMaxCols && p.tokens >= 1 && p.tokens <= kSlots &&
         ((uintptr_t)p.x & 15) == 0 &&
         (p.ids == nullptr || (int64_t)p.src_rows * p.row_bytes < ((int64_t)1 << 32));
}

constexpr int kPastCaches = 65536;  // rows from which the rows' loads take the non-temporal policy (stream_impl.h)

template <int KIND, typename XT>
int launch_window(const WindowParams& p, hipStream_t s) {
  const int nsteps = (p.cols + kStep - 1) / kStep;
  const int spw = nsteps > kMaxWaves ? 2 : 1, waves = (nsteps + spw - 1) / spw;
  const int groups = (p.rows + 15) / 16;
  const int per_cu = max(1, kMaxWaves / waves);
  const dim3 grid((unsigned)min(groups, strata_mv::device_cus() * per_cu)), block(64 * waves);
  auto go = [&](auto spwc, auto staged, auto nt) {
    hipLaunchKernelGGL((window_kernel<KIND, XT, decltype(spwc)::value, decltype(staged)::value, decltype(nt)::value>),
                       grid, block, 0, s, p);
  };
  auto by_spw = [&](auto staged, auto nt) {
    if (spw == 2)
      go(std::integral_constant<int, 2>(), staged, nt);
    else
      go(std::integral_constant<int, 1>(), staged, nt);
  };
  bool done = false;
  if constexpr (kStagedRows<KIND>) {
    // rows at 16-byte boundaries, every wave's steps within the row and whole
    if (p.ids == nullptr && p.row_bytes % 16 == 0 && ((uintptr_t)p.blocks & 15) == 0 && nsteps == spw * waves &&
        p.cols % kStep == 0) {
      if (p.rows >= kPastCaches)
        by_spw(std::true_type(), std::true_type());
      else
        by_spw(std::true_type(), std::false_type());
      done = true;
    }
  }
  if (!done) by_spw(std::false_type(), std::false_type());
  STRATA_CHECK_LAUNCH();
  return STRATA_OK;
}

}  // namespace strata_window
