// Routed matvecs of a few tokens on MFMA: gate and up with the SwiGLU, or one matrix, for up to 128 pairs, every block
// type, float16 or bfloat16 tokens, rows of at most 4096 inputs (strata_mlx/blocks.py:196-259, 939-986).
//
// out[p, r] = W[idx[p], r, :] . x[p / share, :]. A distinct expert's rows are read and decoded once for all the pairs
// naming it, 16 of them an item (window_impl.h's window of 16 slots); the matvecs read them once a pair, or decode them
// once a pair. A workgroup lists the items from the pairs' ids by ballots, and takes a contiguous range of the units
// (item, 16 rows; with gate and up: 16 rows of each), so that it changes item seldom. The K steps are split over its
// waves, one or two steps each; a wave keeps the item's tokens of its steps in registers as MFMA operands, scaled into
// float16's upper range where the type or bfloat16 asks for it (window_impl.h), and its part of a unit's rows comes
// by direct loads into LDS, the next unit's as soon as this one's fields are in registers. The waves' partial sums meet
// in LDS, one barrier a unit, and one wave in turn adds and writes them. Weights are exact (two float16 parts where a
// type needs them, kInexact).
#pragma once
#include "window_impl.h"

namespace strata_rwin {

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

constexpr int kMaxWaves = 8;
constexpr int kMaxCols = 4096;
constexpr int kMaxPairs = 128;  // two ballots
constexpr int kSlots = 16;

struct RwinParams {
  const uint8_t* blocks[2];  // gate and up, or one stack
  const uint32_t* idx;
  const void* x;             // pairs / share rows
  void* out[2];              // gate . x and up . x (may be null with h), or the product
  void* h;                   // silu(gate . x) * (up . x) as mlx-lm rounds it, or null
  int64_t mat_bytes;
  uint32_t experts;
  int rows, cols, row_bytes, pairs, share;
};

// A step's fields from a staged slot: lds_fields' types by the step's parity, the dword types by their window.
template <int KIND>
__device__ __forceinline__ void slot_fields(const uint8_t* slot, int k, int row_bytes, int g, RunPair<KIND>& f) {
  if constexpr (strata_prompt::kDwordRows<KIND>) {
    strata_prompt::dword_fields<KIND>(slot, (uint32_t)(k * kStepBytes<KIND>) - strata_prompt::dword_first<KIND>(k, row_bytes),
                                      g, f);
  } else {
    if (k & 1)
      strata_prompt::lds_fields<KIND, 2>(slot, g, f);
    else
      strata_prompt::lds_fields<KIND, 0>(slot, g, f);
  }
}

template <int KIND, typename XT, int MATS, int SPW, bool STAGED>
__global__ __launch_bounds__(64 * kMaxWaves, 2) void rwin_kernel(RwinParams p) {
  constexpr bool kScaled = std::is_same<XT, bf16_t>::value || kHasMin<KIND>;
  constexpr int kGL = STAGED ? strata_prompt::kGroupLoads<KIND> : 1, kGB = 256 * kGL;
  __shared__ DirectTables<KIND> tab;
  __shared__ f32x4 red[2][kMaxWaves][MATS][64];
  __shared__ uint32_t peak[2][kMaxWaves][kSlots];
  __shared__ int slot_pair[kMaxWaves][kSlots];
  __shared__ int2 item_pair[kMaxPairs];  // an item's leading pair and its expert
  __shared__ __attribute__((aligned(16))) uint8_t slots[STAGED ? kMaxWaves * MATS * SPW * kGB : 16];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  for (int i = tid; i < 256; i += blockDim.x) {
    strata_mv::TableFetch<KIND> tf;
    strata_mv::fetch_tables<KIND>(tf, i);
    strata_mv::store_tables<KIND>(tab, tf, i);
  }

  // pairs lane and lane + 64: their experts, each one's rank among the pairs naming its expert, and the items: a pair
  // whose rank is a multiple of 16 leads one, of the up to 16 pairs from its rank on
  uint32_t e[2];
  bool valid[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int q = 64 * c + lane;
    e[c] = q < p.pairs ? p.idx[q] : 0xffffffffu;
    valid[c] = e[c] < p.experts;
  }
  uint64_t same[2][2];  // [of pair c][among pairs d]
#pragma unroll
  for (int d = 0; d < 2; ++d) same[0][d] = same[1][d] = __ballot(valid[d]);
  for (uint32_t b = 0; (p.experts - 1) >> b != 0; ++b) {
    const uint64_t m[2] = {__ballot((e[0] >> b) & 1), __ballot((e[1] >> b) & 1)};
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int d = 0; d < 2; ++d) same[c][d] &= (e[c] >> b) & 1 ? m[d] : ~m[d];
  }
  const uint64_t below = (1ull << lane) - 1;
  const int rank[2] = {(int)__popcll(same[0][0] & below),
                       (int)(__popcll(same[1][0]) + __popcll(same[1][1] & below))};
  const uint64_t lead0 = __ballot(valid[0] && rank[0] % kSlots == 0), lead1 = __ballot(valid[1] && rank[1] % kSlots == 0);
  const int items = (int)(__popcll(lead0) + __popcll(lead1));
  if (wave == 0) {
    if ((lead0 >> lane) & 1) item_pair[__popcll(lead0 & below)] = make_int2(lane, (int)e[0]);
    if ((lead1 >> lane) & 1) item_pair[__popcll(lead0) + __popcll(lead1 & below)] = make_int2(64 + lane, (int)e[1]);
  }
  __syncthreads();  // the tables and the items

  // rows of NaN for the pairs naming no expert, a pair a workgroup in turn
  for (int q = blockIdx.x; q < p.pairs; q += gridDim.x) {
    if (p.idx[q] < p.experts) continue;
    const XT nan = from_f32<XT>(__builtin_nanf(""));
    for (int r = tid; r < p.rows; r += blockDim.x) {
      const int64_t o = (int64_t)q * p.rows + r;
#pragma unroll
      for (int m = 0; m < MATS; ++m)
        if (p.out[m] != nullptr) reinterpret_cast<XT*>(p.out[m])[o] = nan;
      if (MATS == 2 && p.h != nullptr) reinterpret_cast<XT*>(p.h)[o] = nan;
    }
  }

  const int groups = (p.rows + 15) / 16;
  const int units = items * groups, each = (units + gridDim.x - 1) / gridDim.x;
  const int u0 = blockIdx.x * each, u1 = min(u0 + each, units);
  if (u0 >= u1) return;

  // the wave's steps; past the row's last step, the last again with zero activations
  const int nsteps = (p.cols + kStep - 1) / kStep;
  const int last_pairs = kMayPart<KIND> ? (p.cols - (nsteps - 1) * kStep) / 64 : 4;
  const LaneOffsets<KIND> lo = strata_mv::lane_offsets<KIND>(g);
  int ks[SPW], gl[SPW];
#pragma unroll
  for (int s = 0; s < SPW; ++s) {
    ks[s] = min(wave * SPW + s, nsteps - 1);
    gl[s] = ks[s] == nsteps - 1 ? min(g, last_pairs - 1) : g;  // a run pair past the row's: its last
  }

  uint32_t voff[kGL];
  const uint32_t slot0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)slots + (uint32_t)(wave * MATS * SPW * kGB));
  if constexpr (STAGED) {
    constexpr int kPitchDw = strata_prompt::kSlotPitch<KIND>;
#pragma unroll
    for (int l = 0; l < kGL; ++l) {
      const int c = 64 * l + lane, q = min(c / kPitchDw, 15), d = min(c % kPitchDw, strata_prompt::kSlotDwords<KIND> - 1);
      voff[l] = (uint32_t)q * (uint32_t)p.row_bytes + 4u * (uint32_t)d;
    }
  }
  RunPair<KIND> f[MATS][SPW], fn[STAGED ? 1 : MATS][SPW];
  // unit u's rows of the wave's steps: into the wave's slots, or (not staged) into registers
  auto fetch = [&](int u, RunPair<KIND>(*dst)[SPW]) {
    const int item = u / groups, r0 = (u - item * groups) * 16;
    const uint32_t expert = (uint32_t)__builtin_amdgcn_readfirstlane(item_pair[item].y);
    const int last = p.rows - 1 - r0;
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
      const uint8_t* mat = p.blocks[m] + (int64_t)expert * p.mat_bytes + (int64_t)r0 * p.row_bytes;
#pragma unroll
      for (int s = 0; s < SPW; ++s) {
        if constexpr (STAGED) {
          const uint32_t first = strata_prompt::kDwordRows<KIND> ? strata_prompt::dword_first<KIND>(ks[s], p.row_bytes)
                                                                 : (uint32_t)(ks[s] * kStepBytes<KIND>) & ~3u;
          const uint8_t* base = mat + first;
          const uint32_t at = slot0 + (uint32_t)((m * SPW + s) * kGB);
          if (last < 15) {
#pragma unroll
            for (int l = 0; l < kGL; ++l) {
              const int q = min((64 * l + lane) / strata_prompt::kSlotPitch<KIND>, 15);
              strata_prompt::dma_dword(base, voff[l] - (uint32_t)max(0, q - last) * (uint32_t)p.row_bytes, at + 256u * l);
            }
          } else {
#pragma unroll
            for (int l = 0; l < kGL; ++l) strata_prompt::dma_dword(base, voff[l], at + 256u * l);
          }
        } else {
          strata_mv::load_fields<KIND>(mat, (uint32_t)min(n, last) * (uint32_t)p.row_bytes +
                                                (uint32_t)ks[s] * kStepBytes<KIND> - (uint32_t)(g - gl[s]) * (kStepBytes<KIND> / 4),
                                       lo, dst[m][s]);
        }
      }
    }
  };
  if constexpr (STAGED)
    fetch(u0, nullptr);
  else
    fetch(u0, f);

  u32x4 a[SPW][2][4];
  uint32_t sums[SPW][2];
  int ex_out[4] = {0, 0, 0, 0};
  int count = 0, cur = -1;
  for (int u = u0, it = 0; u < u1; ++u, ++it) {
    const int item = u / groups, r0 = (u - item * groups) * 16;
    if (item != cur) {  // the item's pairs, and their tokens into registers
      cur = item;
      const int lp = __builtin_amdgcn_readfirstlane(item_pair[item].x), c = lp >> 6;
      const uint32_t le = (uint32_t)__builtin_amdgcn_readfirstlane(item_pair[item].y);
      const int first = c ? __builtin_amdgcn_readlane(rank[1], lp & 63) : __builtin_amdgcn_readlane(rank[0], lp & 63);
      const bool in0 = valid[0] && e[0] == le && rank[0] >= first && rank[0] < first + kSlots;
      const bool in1 = valid[1] && e[1] == le && rank[1] >= first && rank[1] < first + kSlots;
      if (in0) slot_pair[wave][rank[0] - first] = lane;
      if (in1) slot_pair[wave][rank[1] - first] = 64 + lane;
      count = (int)(__popcll(__ballot(in0)) + __popcll(__ballot(in1)));
      __builtin_amdgcn_wave_barrier();  // the wave's slots are written
      const int pr = slot_pair[wave][min(n, count - 1)];
      const uint16_t* row = reinterpret_cast<const uint16_t*>(p.x) + (int64_t)(pr / p.share) * p.cols;
#pragma unroll
      for (int s = 0; s < SPW; ++s) {
        const bool live = wave * SPW + s < nsteps && gl[s] == g && n < count;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            u32x4 v = u32x4{0u, 0u, 0u, 0u};
            if (live) v = *reinterpret_cast<const u32x4*>(row + ks[s] * kStep + strata_prompt::a_col<KIND>(g, h, q));
            a[s][h][q] = v;
          }
      }
      if constexpr (kScaled) strata_window::scale_tokens<KIND, XT, SPW>(a, sums, ex_out, peak[it & 1], wave, waves, n, g);
    }

    if constexpr (STAGED) {  // the unit's rows are in; their fields, then the slots take the next unit's
      strata_prompt::wait_loads();
#pragma unroll
      for (int m = 0; m < MATS; ++m)
#pragma unroll
        for (int s = 0; s < SPW; ++s)
          slot_fields<KIND>(slots + ((wave * MATS + m) * SPW + s) * kGB + 4 * strata_prompt::kSlotPitch<KIND> * n, ks[s],
                            p.row_bytes, gl[s], f[m][s]);
      if (u + 1 < u1) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        fetch(u + 1, nullptr);
      }
    } else {
      fetch(min(u + 1, u1 - 1), fn);
    }
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < SPW; ++s)
        strata_window::add_step<KIND>(f[m][s], a[s], sums[s], g, tab, acc);
      red[it & 1][wave][m][lane] = acc;
    }
    strata_prompt::lds_barrier();
    if (wave == it % waves) {  // lane (n, g): row n, slots 4 g + j
      f32x4 t[MATS];
#pragma unroll
      for (int m = 0; m < MATS; ++m) {
        t[m] = red[it & 1][0][m][lane];
#pragma unroll
        for (int w = 1; w < kMaxWaves; ++w) {
          if (w < waves) {
            const f32x4 v = red[it & 1][w][m][lane];
#pragma unroll
            for (int j = 0; j < 4; ++j) t[m][j] += v[j];
          }
        }
      }
      const int r = r0 + n;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int slot = 4 * g + j;
        if (slot >= count || r >= p.rows) continue;
        const int64_t o = (int64_t)slot_pair[wave][slot] * p.rows + r;
        XT v[MATS];
#pragma unroll
        for (int m = 0; m < MATS; ++m) {
          v[m] = from_f32<XT>(kScaled ? __builtin_ldexpf(t[m][j], ex_out[j]) : t[m][j]);
          if (p.out[m] != nullptr) reinterpret_cast<XT*>(p.out[m])[o] = v[m];
        }
        if constexpr (MATS == 2) {
          if (p.h != nullptr)
            reinterpret_cast<XT*>(p.h)[o] = from_f32<XT>(strata_mv::swiglu_rounded<XT>(v[0], v[1]));
        }
      }
    }
    if constexpr (!STAGED) {
#pragma unroll
      for (int m = 0; m < MATS; ++m)
#pragma unroll
        for (int s = 0; s < SPW; ++s) f[m][s] = fn[m][s];
    }
  }
}

// Whether the waves' slots fit in LDS beside the sums (not for two Q8_0 matrices at two steps a wave).
template <int KIND, int MATS, int SPW>
constexpr bool slots_fit() {
  return kMaxWaves * MATS * SPW * 256 * strata_prompt::kGroupLoads<KIND> <= 120 * 1024;
}

// Whether rwin_kernel takes a routed product: 16-bit tokens in rows at 16-byte boundaries, up to 128 pairs, rows of
// whole run pairs (whole steps in the types with blocks of 256) and at most 4096 inputs, a matrix below 4 GiB.
inline bool rwin_takes(int kind, const RwinParams& p) {
  return strata_prompt::tiles_take(kind, p.cols) && p.cols <= kMaxCols && p.pairs <= kMaxPairs &&
         ((uintptr_t)p.x & 15) == 0 && p.mat_bytes < ((int64_t)1 << 32);
}

template <int KIND, typename XT, int MATS>
int launch_rwin(const RwinParams& p, hipStream_t s) {
  const int nsteps = (p.cols + kStep - 1) / kStep;
  const int spw = nsteps > kMaxWaves ? 2 : 1, waves = (nsteps + spw - 1) / spw;
  const int64_t most = (int64_t)((p.rows + 15) / 16) * p.pairs;
  if (most > INT32_MAX) return STRATA_ERR_SHAPE;
  const int per_cu = MATS == 2 || waves > 6 ? 1 : max(1, 12 / waves);  // one round of resident workgroups
  const dim3 grid((unsigned)min(most, (int64_t)strata_mv::device_cus() * per_cu)), block(64 * waves);
  const bool staged = ((uintptr_t)p.blocks[0] & 3) == 0 && ((uintptr_t)p.blocks[1] & 3) == 0 && p.row_bytes % 4 == 0 &&
                      p.row_bytes >= 4 * strata_prompt::kSlotDwords<KIND> &&
                      (strata_prompt::kDwordRows<KIND> || p.cols % kStep == 0);
  auto go = [&](auto spwc, auto st) {
    constexpr int SPW = decltype(spwc)::value;
    constexpr bool kStaged = decltype(st)::value && slots_fit<KIND, MATS, SPW>();
    hipLaunchKernelGGL((rwin_kernel<KIND, XT, MATS, SPW, kStaged>), grid, block, 0, s, p);
  };
  auto by_spw = [&](auto st) {
    if (spw == 2)
      go(std::integral_constant<int, 2>(), st);
    else
      go(std::integral_constant<int, 1>(), st);
  };
  if constexpr (strata_prompt::kStagedKind<KIND>) {
    if (staged) {
      by_spw(std::true_type());
      STRATA_CHECK_LAUNCH();
      return STRATA_OK;
    }
  }
  by_spw(std::false_type());
  STRATA_CHECK_LAUNCH();
  return STRATA_OK;
}

}  // namespace strata_rwin
