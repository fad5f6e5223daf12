// GEMM kernel for a few rows on gfx950: no K loop to speak of.
//
//   C[M,N] = epilogue(A[M,K] * B[N,K]^T)   (both operands K-contiguous and 16-byte aligned, K a multiple of 128 bytes)
//
// With up to some dozen rows a product is neither bound by bytes nor by the matrix pipes but by waits in a row: launch,
// first operands, then one LDS stage after the other with a barrier each (10 x 3072 x 768 fp16 on the 32 x 64 ring tile:
// 0.3 + 0.7 + twelve steps of 0.18 + 0.4 us, and 1.4 between two launches).  Here a workgroup owns 16 columns and 16 or 32
// rows, its sixteen wavefronts divide K among themselves, and each requests its share into a part of LDS of its own: one
// wait instead of twelve, and no barrier before the partial tiles meet in LDS.  They are summed in a fixed order by the
// threads that store them; what those need besides (bias, residual, scales, destination) is requested in front.
// (Straight from memory to registers is slower: the 64 bytes of K that a matrix instruction takes of a row are half a
// cache line, and a CU then fetches 43 GB/s instead of 115.)
// Narrow tiles spread the weights over many CUs; every row tile reads them again.
//
// LayerNorm in front (NormRows): every workgroup normalises the rows of its tile itself, a row per wavefront, while its first
// weights are on their way, and keeps them in LDS for the whole of K.  The rows are a few KB that L2 serves, so the repeated
// work hides under the wait for the weights; a launch of its own and the gap in front of the next one are gone.
// Six decoder layers, fp16, 8 x 1 tokens, 41 keys: 67 launches and 343 us a step before, 49 and 264 after.
#pragma once

#include "gemm_split.h"

namespace ttmi {

template <typename T>
__device__ __forceinline__ void flat_mma(const Chunk& a, const Chunk& b, typename RingMma<T>::Acc& c) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (std::is_same<T, f16>::value) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  } else if constexpr (std::is_same<T, bf16>::value) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else if constexpr (std::is_same<T, int8_t>::value) {
    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(intx4, a), __builtin_bit_cast(intx4, b), c, 0, 0, 0);
  } else {
#pragma unroll
    for (int part = 0; part < 4; ++part) {
      const uint32_t x = a.w[part], y = b.w[part];
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y), c, 0, 0, 0);
    }
  }
#endif
}

// What becomes of the rows of A on their way in.
struct PlainRows {};
template <typename T>
struct NormRows {  // beta + gamma * (x - mean) / sqrt(var + eps), rounded to T as a tensor of its own would be
  const T *gamma, *beta;
  float eps;
};

constexpr int kFlatWaves = 16;
constexpr int kFlatPitch = 20;  // words of a row of a partial tile: 16-byte aligned, four rows apart on other banks
template <int MB>
constexpr int flat_stage_bytes() { return (MB + 1) * 16 * kRowBytes; }
template <int MB>
constexpr int flat_partial_bytes() { return kFlatWaves * MB * 16 * kFlatPitch * 4; }

// MB: blocks of 16 rows.  D: LDS stages per wavefront (steps of 128 bytes of K; one suffices for a share of one step).
// LDS: (normalised rows: a block of MB * 16 rows x 128 bytes per step of K, then) the stages of the wavefronts that have a
// share; afterwards one partial tile per wavefront.
template <typename T, int MB, int D, typename Epi, typename Rows = PlainRows>
__global__ __launch_bounds__(kFlatWaves * kWave) void gemm_flat_kernel(const GemmArgs g, const Epi epi, const Rows rows) {
  constexpr bool NORM = !std::is_same<Rows, PlainRows>::value;
  constexpr int NW = kFlatWaves, PITCH = kFlatPitch, STAGE = NORM ? flat_stage_bytes<0>() : flat_stage_bytes<MB>();
  constexpr int A_LOADS = NORM ? 0 : 2 * MB, LOADS = A_LOADS + 2;  // 1 KB loads of a step: eight rows each
  using Acc = typename RingMma<T>::Acc;
  using AccScalar = typename Epi::Acc;
  extern __shared__ __align__(16) char smem[];
  AccScalar* const part = reinterpret_cast<AccScalar*>(smem);  // [NW][MB * 16][PITCH]

  const int tiles = g.tiles_m * g.tiles_n, total = tiles * g.slices;
  const bool remap = total >= kXcdRemapMinTiles;
  const int per_xcd = (total + kNumXcd - 1) / kNumXcd;
  int logical = remap ? (int)(blockIdx.x % kNumXcd) * per_xcd + (int)(blockIdx.x / kNumXcd) : (int)blockIdx.x;
  if (logical >= total) {
    if constexpr (Dequantises<Epi>::value)
      if (epi.absmax_slots() != nullptr && threadIdx.x == 0) epi.absmax_slots()[blockIdx.x] = 0.f;
    return;
  }
  int slice = 0;
  if (g.slices > 1) {
    slice = logical / tiles;
    logical -= slice * tiles;
  }
  // the row tiles of a column tile are neighbours: an XCD reads its weights once
  const int tile_n = logical / g.tiles_m, tile_m = logical - tile_n * g.tiles_m;
  const int m0 = tile_m * (MB * 16), n0 = tile_n * 16;
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int lrow = lane & 15, lgrp = lane >> 4;

  int kdim = g.k, z_epi = 0;
  uint32_t k_lo = 0;  // bytes
  if (g.k_chunk > 0) {
    const int lo = slice * g.k_chunk;
    kdim = min(g.k_chunk, g.k - lo);
    k_lo = (uint32_t)lo * (uint32_t)sizeof(T);
    z_epi = slice;
  }
  const int steps = kdim * (int)sizeof(T) / kRowBytes;
  const int share = (steps + NW - 1) / NW;
  const int s_lo = wave * share, s_hi = min(s_lo + share, steps);
  const bool busy = s_lo < s_hi;  // uniform per wavefront

  // ---- loads: as in the ring kernel, with the XOR swizzle on the global side; steps past the share return at once
  uint32_t voff[LOADS];
  {
    const uint32_t lda_bytes = (uint32_t)(g.lda * (int64_t)sizeof(T)), ldb_bytes = (uint32_t)(g.ldb * (int64_t)sizeof(T));
    const int sub = lane >> 3, c = lane & 7;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int row = i * 8 + sub;  // of the stage: (MB * 16 rows of A,) 16 of B
      const uint32_t at = i < A_LOADS ? (uint32_t)min(m0 + row, g.m - 1) * lda_bytes : (uint32_t)min(n0 + row - A_LOADS * 8, g.n - 1) * ldb_bytes;
      voff[i] = at + ((c ^ ((row >> 1) & 7)) << 4);
    }
  }
  const int stage0 = (NORM ? steps * (MB * 16 * kRowBytes) : 0) + wave * (D * STAGE);
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) char lds_char;
  lds_char* lds0 = reinterpret_cast<lds_char*>(reinterpret_cast<uintptr_t>(smem));
  const int a_size = (int)((int64_t)g.m * g.lda * (int64_t)sizeof(T)), b_size = (int)((int64_t)g.n * g.ldb * (int64_t)sizeof(T));
  auto load = [&](int s, int stage) __attribute__((always_inline)) {
    const bool live = s < s_hi;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(g.a), 0, live ? a_size : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(g.b), 0, live ? b_size : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < A_LOADS ? ra : rb, lds0 + stage0 + stage * STAGE + i * 1024, 16, voff[i], k_lo + s * kRowBytes, 0, 0);
  };
#else
  auto load = [&](int, int) {};
#endif

  // ---- rows to normalise: a wavefront takes every sixteenth, 16 bytes per lane and turn (K is at most 16 * D steps)
  constexpr int KPC = 16 / (int)sizeof(T), TURNS = NORM ? 2 * D : 1, ROWS = NORM ? MB : 1;
  Vec<T, KPC> xr[ROWS][TURNS], gm[TURNS], bt[TURNS];
  if constexpr (NORM) {
#pragma unroll
    for (int t = 0; t < TURNS; ++t) {
      const int col = (t * kWave + lane) * KPC;
      if (col < kdim) {
#pragma unroll
        for (int i = 0; i < ROWS; ++i)
          xr[i][t] = load_vec<T, KPC>(reinterpret_cast<const T*>(g.a) + min(m0 + wave + i * NW, g.m - 1) * g.lda + col);
        gm[t] = load_vec<T, KPC>(rows.gamma + col);
        bt[t] = load_vec<T, KPC>(rows.beta + col);
      }
    }
  }

  // ---- the thread's piece of the output: eight columns of one row
  const bool stores = tid < MB * 32;
  const int m = m0 + (tid >> 1), n = n0 + (tid & 1) * 8;
  bool row_piece = stores && m < g.m && n < g.n;
  bool column_piece = false;
  if constexpr (HasColumnPass<Epi>::value) {
    if (epi.column_pass()) {
      row_piece = row_piece && n < epi.first_column_of_pass();
      column_piece = stores && n0 + (tid & 15) >= epi.first_column_of_pass() && n0 + (tid & 15) < g.n && m0 + (tid >> 4) * 8 < g.m;
    }
  }
  // (in front of the loads to LDS: loads return in order)
  float wide[8], scale[8], res[8];
  float act_scale = 0.f, column_bias = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) wide[e] = 0.f, scale[e] = 0.f, res[e] = 0.f;
  typename RingDest<Epi>::Elem* dest = nullptr;
  const auto* bias = epi.bias_ptr();
  if (row_piece) {
    if (bias != nullptr) load_row8(bias + n, wide);
    if constexpr (Dequantises<Epi>::value) {
      act_scale = epi.act_scale[0];
      load_row8<float>(epi.w_scale + n, scale);
    }
    if constexpr (AddsResidual<Epi>::value) load_row8(epi.residual + (int64_t)m * epi.ldc + n, res);
    dest = RingDest<Epi>::column(epi, z_epi, n) + RingDest<Epi>::row(epi, m);
  }
  if (column_piece && bias != nullptr) column_bias = to_float(bias[n0 + (tid & 15)]);

  Acc acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[i][e] = 0;
  if (busy) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(s_lo + d, d);
  }
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      float x[TURNS][KPC], sum = 0.f, sumsq = 0.f;
#pragma unroll
      for (int t = 0; t < TURNS; ++t)
        if ((t * kWave + lane) * KPC < kdim)
#pragma unroll
          for (int j = 0; j < KPC; ++j) {
            x[t][j] = to_float(xr[i][t].v[j]);
            sum += x[t][j];
            sumsq += x[t][j] * x[t][j];
          }
      sum = group_sum<kWave>(sum);
      sumsq = group_sum<kWave>(sumsq);
      const float mean = sum / (float)kdim;
      const float var = fmaxf(sumsq / (float)kdim - mean * mean, 0.f);  // as in layer_norm_rows
      const float rstd = 1.0f / sqrtf(var + rows.eps);
      const int row = wave + i * NW;
#pragma unroll
      for (int t = 0; t < TURNS; ++t) {
        const int piece = t * kWave + lane;  // of the row: step piece / 8, chunk piece % 8, at the swizzled place
        if (piece * KPC < kdim) {
          Vec<T, KPC> o;
#pragma unroll
          for (int j = 0; j < KPC; ++j) o.v[j] = from_float<T>(to_float(bt[t].v[j]) + to_float(gm[t].v[j]) * rstd * (x[t][j] - mean));
          store_vec<T, KPC>(reinterpret_cast<T*>(smem + (piece >> 3) * (MB * 16 * kRowBytes) + row * kRowBytes + (((piece & 7) ^ ((row >> 1) & 7)) << 4)), o);
        }
      }
    }
    __syncthreads();
  }
  if (busy) {
    const uint32_t lds_rows = (uint32_t)reinterpret_cast<uintptr_t>(smem), lds_base = lds_rows + stage0;
    const int swz = (lrow >> 1) & 7;
    int stage = 0;
#pragma unroll 1
    for (int s = s_lo; s < s_hi; ++s) {
      // fragment reads as instructions, as in the ring kernel: the compiler would wait for every load in flight
      Chunk fa[2][MB], fb[2];
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * LOADS) : "memory");
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t in_row = lrow * kRowBytes + (((h * 4 + lgrp) ^ swz) << 4);
        const uint32_t at = lds_base + stage * STAGE + in_row, at_a = NORM ? lds_rows + s * (MB * 16 * kRowBytes) + in_row : at;
#pragma unroll
        for (int i = 0; i < MB; ++i)
          asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(reinterpret_cast<Quad&>(fa[h][i])) : "v"(at_a), "n"(i * 16 * kRowBytes) : "memory");
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(reinterpret_cast<Quad&>(fb[h])) : "v"(at), "n"(A_LOADS * 8 * kRowBytes) : "memory");
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < MB; ++i) asm volatile("" : "+v"(reinterpret_cast<Quad&>(fa[h][i])));
        asm volatile("" : "+v"(reinterpret_cast<Quad&>(fb[h])));
      }
      if (D > 1) load(s + D, stage);
      stage = stage + 1 == D ? 0 : stage + 1;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < MB; ++i) flat_mma<T>(fa[h][i], fb[h], acc[i]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the share have returned before LDS is reused
  }
  __syncthreads();  // (a partial tile may lie in another wavefront's stages)

  // ---- acc[i][e] = C[16i + 4*lgrp + e][lrow]
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[(wave * MB * 16 + i * 16 + lgrp * 4 + e) * PITCH + lrow] = acc[i][e];
  __syncthreads();
  float amax = 0.f;
  if (row_piece) {
    AccScalar v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const AccScalar* from = part + (w * MB * 16 + (tid >> 1)) * PITCH + (tid & 1) * 8;
      const Vec<AccScalar, 4> lo = load_vec<AccScalar, 4>(from), hi = load_vec<AccScalar, 4>(from + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += lo.v[e], v[4 + e] += hi.v[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (Dequantises<Epi>::value) {
        const float r = epi.activate(dequantise(v[e], act_scale, scale[e], wide[e], epi.has_bias()));
        amax = fmaxf(amax, fabsf(r));
        v[e] = __builtin_bit_cast(AccScalar, r);
      } else {
        v[e] += (AccScalar)wide[e];
      }
    }
    if constexpr (std::is_same<Epi, EpiInt32>::value) {
      epi.store8(z_epi, m, n, v, 8);
    } else {
      float fin[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) fin[e] = RingDest<Epi>::finish(epi, v[e]) + res[e];
      store_row8(dest, fin);
    }
  }
  if constexpr (HasColumnPass<Epi>::value) {
    if (column_piece) {
      const int r0 = (tid >> 4) * 8, c = tid & 15;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[e] = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v[e] += part[(w * MB * 16 + r0 + e) * PITCH + c];
        v[e] += column_bias;
      }
      epi.store_col8(m0 + r0, g.m, n0 + c, v);
    }
  }
  publish_absmax(epi, amax, reinterpret_cast<float*>(smem), NW * kWave);
}

template <typename T, int MB, int D, typename Epi, typename Rows = PlainRows>
inline int launch_flat_tile(GemmArgs g, const Epi& epi, int slices, hipStream_t s, const Rows& rows = Rows{}) {
  if (describe_only("dma", kFlatWaves, MB * 16, 16, slices)) return 0;
  g.tiles_m = (g.m + MB * 16 - 1) / (MB * 16);
  g.tiles_n = (g.n + 15) / 16;
  g.slices = slices;
  const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n * slices;
  TTMI_REQUIRE(tiles < (1ll << 30), "GEMM grid too large");
  const unsigned grid_x = tiles >= kXcdRemapMinTiles ? (unsigned)(ceil_div(tiles, kNumXcd) * kNumXcd) : (unsigned)tiles;
  if (!absmax_grid_ok(epi, grid_x, 1)) return launch_flat_tile<T, MB, D>(g, without_absmax(epi), slices, s, rows);
  const int64_t steps = (g.k_chunk > 0 ? g.k_chunk : g.k) * (int64_t)sizeof(T) / kRowBytes;
  const int64_t share = ceil_div(steps, kFlatWaves);
  constexpr bool norm = !std::is_same<Rows, PlainRows>::value;
  if (norm) TTMI_REQUIRE(g.k_chunk == 0 && steps <= kFlatWaves * D, "rows to normalise come whole");
  const int64_t stages = norm ? steps * MB * 16 * kRowBytes + ceil_div(steps, share) * D * flat_stage_bytes<0>()
                              : ceil_div(steps, share) * D * flat_stage_bytes<MB>();
  const int lds = (int)std::max<int64_t>(stages, flat_partial_bytes<MB>());
  auto kern = gemm_flat_kernel<T, MB, D, Epi, Rows>;
  static_assert(kFlatWaves * 2 * flat_stage_bytes<1>() <= kLdsPerCu, "stages exceed the LDS");
  TTMI_REQUIRE(lds <= kLdsPerCu, "stages exceed the LDS");
  if (lds > 64 * 1024) {
    const int rc = allow_large_lds(reinterpret_cast<const void*>(kern), kLdsPerCu);
    if (rc != 0) return rc;
  }
  hipLaunchKernelGGL(kern, dim3(grid_x), dim3(kFlatWaves * kWave), lds, s, g, epi, rows);
  return launch_status("gemm_flat_kernel");
}

// Steps of the longest K (slice) that a tile of MB blocks takes: its stages fit the LDS.
template <int MB>
inline bool flat_fits(int64_t steps) {
  const int64_t share = ceil_div(steps, kFlatWaves);
  return ceil_div(steps, share) * std::min<int64_t>(share, 2) * flat_stage_bytes<MB>() <= kLdsPerCu;
}

// The form for few rows wins while every workgroup has a CU of its own and K is short enough that reading A once per 16
// columns does not count.  us, ring tile / this (weights not in L2): fp16 10 x 3072 x 768 4.7 / 3.9, 32 x 3072 x 768 4.9 /
// 4.0, 64 x 2304 x 768 (288 workgroups) 4.8 / 4.7, 10 x 768 x 3072 3.8 and a reduction of 4 / 5.4; fp32 10 x 3072 x 768
// 9.4 / 5.7, 96 x 768 x 768 9.2 / 5.8, 40 x 2304 x 768 (432 workgroups) 9.4 / 9.7.
template <typename T>
inline bool flat_wins(const GemmArgs& g, int64_t most_steps) {
  const int64_t steps = g.k * (int64_t)sizeof(T) / kRowBytes;
  const int64_t rows = g.m <= 16 || !flat_fits<2>(steps) ? 16 : 32;
  return steps <= most_steps && ceil_div(g.m, rows) * ceil_div(g.n, 16) <= compute_units();
}

template <typename T, typename Epi>
inline int launch_flat(const GemmArgs& g, const Epi& epi, int slices, hipStream_t s) {
  const int64_t steps = (g.k_chunk > 0 ? g.k_chunk : g.k) * (int64_t)sizeof(T) / kRowBytes;
  const bool one = steps <= kFlatWaves;
  if (g.m <= 16 || !flat_fits<2>(steps)) return one ? launch_flat_tile<T, 1, 1>(g, epi, slices, s) : launch_flat_tile<T, 1, 2>(g, epi, slices, s);
  return one ? launch_flat_tile<T, 2, 1>(g, epi, slices, s) : launch_flat_tile<T, 2, 2>(g, epi, slices, s);
}

// The same with LayerNorm in front, for rows of at most two steps per wavefront (2048 16-bit or 1024 fp32 values).
// The line is that of the product alone: one workgroup per CU, so that nobody normalises a row twice.  (A LayerNorm launch
// of 8 x 768 is 2.9 us on the GPU and 3.5 on the host.)
template <typename T, int MB>
inline bool flat_norm_fits(int64_t steps) {
  const int64_t share = ceil_div(steps, kFlatWaves);
  return share <= 2 && steps * MB * 16 * kRowBytes + ceil_div(steps, share) * share * flat_stage_bytes<0>() <= kLdsPerCu;
}
template <typename T>
inline bool flat_norm_wins(const GemmArgs& g) {
  const int64_t steps = g.k * (int64_t)sizeof(T) / kRowBytes;
  const int64_t rows = g.m <= 16 || !flat_norm_fits<T, 2>(steps) ? 16 : 32;
  return flat_norm_fits<T, 1>(steps) && ceil_div(g.m, rows) * ceil_div(g.n, 16) <= compute_units();
}
template <typename T, typename Epi>
inline int launch_flat_norm(const GemmArgs& g, const Epi& epi, const NormRows<T>& rows, hipStream_t s) {
  const int64_t steps = g.k * (int64_t)sizeof(T) / kRowBytes;
  const bool one = steps <= kFlatWaves;
  if (g.m <= 16 || !flat_norm_fits<T, 2>(steps)) return one ? launch_flat_tile<T, 1, 1>(g, epi, 1, s, rows) : launch_flat_tile<T, 1, 2>(g, epi, 1, s, rows);
  return one ? launch_flat_tile<T, 2, 1>(g, epi, 1, s, rows) : launch_flat_tile<T, 2, 2>(g, epi, 1, s, rows);
}

}  // namespace ttmi
