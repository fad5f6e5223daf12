// Mid-size GEMM kernel for gfx950: small tiles in an LDS ring of three or four K steps, whose loads are spread evenly
// between the matrix instructions.
//
//   C[M,N] = epilogue(A[M,K] * B[N,K]^T)   (both operands K-contiguous and 16-byte aligned, K a multiple of 128 bytes)
//
// What bounds a product of some hundred to a few thousand rows is neither memory nor the matrix pipe.  A CU fetches
// 115 GB/s from L2 (one 1 KB `global -> LDS` load per 18 cycles), and the older kernels of gemm_impl.h issue the loads of
// a K step in one burst behind its barrier: a wavefront that waits at the full load queue issues no matrix instruction, so
// the two times add up (a 128 x 128 step: 580 + 510 cycles).  Here a load goes out every few matrix instructions over the
// whole step, half of them behind the step's barrier and half in front of the next one's, and the two overlap: a step of
// 128 x 64 takes 0.25 us instead of 0.35, of 128 x 192 0.44 against a matrix time of 0.35.
// The other half of such a launch is what a workgroup spends outside its K loop, so everything there is short: eight
// wavefronts where the tile has room for them (a lone wavefront per SIMD issues dependent instructions every eight cycles),
// destinations as column part + row part, 16-byte stores straight from the accumulator layout (epilogue of a 128 x 192 tile
// 4.7 -> 1.3 us).  Steps past the last one are requested from a buffer of size 0: they return at once, the loop needs no
// tail and its wait counters stay constants.
// Measured, fp16, us per launch before / after: 2000 x 2304 x 768 16.7 / 12.5, 2000 x 768 x 768 8.3 / 6.2, 2000 x 3072 x 768
// 16.5 / 12.5, 2000 x 768 x 3072 24.4 (four K slices) / 14.0, 387 x 2304 x 768 8.9 / 5.7; fp32: 87 / 63, 33 / 23, 100 / 74,
// 93 / 77.
#pragma once

#include "gemm_impl.h"
#include "gemm_w4.h"

namespace ttmi {

// One 16 x 16 block of the output per 64 bytes of K, accumulator pinned to the AGPR half (see MmaBlock in gemm_w4.h).
// PARTS instructions per 16-byte chunk: the fp32 instruction takes one of the chunk's four values at a time.
template <typename T>
struct RingMma;
template <>
struct RingMma<f16> {
  using Acc = floatx4;
  static constexpr int PARTS = 1;
  static __device__ __forceinline__ void run(const Chunk& a, const Chunk& b, Acc& c, int) { MmaBlock<f16, 16>::run(a, b, c); }
};
template <>
struct RingMma<bf16> {
  using Acc = floatx4;
  static constexpr int PARTS = 1;
  static __device__ __forceinline__ void run(const Chunk& a, const Chunk& b, Acc& c, int) { MmaBlock<bf16, 16>::run(a, b, c); }
};
template <>
struct RingMma<int8_t> {
  using Acc = intx4;
  static constexpr int PARTS = 1;
  static __device__ __forceinline__ void run(const Chunk& a, const Chunk& b, Acc& c, int) {
    asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(c) : "v"(__builtin_bit_cast(intx4, a)), "v"(__builtin_bit_cast(intx4, b)));
  }
};
template <>
struct RingMma<float> {
  using Acc = floatx4;
  static constexpr int PARTS = 4;
  static __device__ __forceinline__ void run(const Chunk& a, const Chunk& b, Acc& c, int part) {
    asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+a"(c) : "v"(a.w[part]), "v"(b.w[part]));
  }
};

// Where an epilogue's output goes, as column part + row part, and what finishes a value.
template <typename Epi>
struct RingDest;
template <typename Epi>
struct AddsResidual : std::false_type {};
template <typename T, int ACT, bool HAS_ACT>
struct AddsResidual<EpiBias<T, ACT, HAS_ACT, true>> : std::true_type {};
template <typename T, int ACT, bool HAS_ACT, bool HAS_RES>
struct RingDest<EpiBias<T, ACT, HAS_ACT, HAS_RES>> {
  using Epi = EpiBias<T, ACT, HAS_ACT, HAS_RES>;
  using Elem = T;
  static __device__ __forceinline__ T* column(const Epi& e, int, int n) { return e.c + n; }
  static __device__ __forceinline__ int64_t row(const Epi& e, int m) { return (int64_t)m * e.ldc; }
  static __device__ __forceinline__ float finish(const Epi& e, float x) { return e.finish(x); }
};
template <typename T>
struct RingDest<EpiF32<T>> {
  using Elem = float;
  static __device__ __forceinline__ float* column(const EpiF32<T>& e, int, int n) { return e.c + n; }
  static __device__ __forceinline__ int64_t row(const EpiF32<T>& e, int m) { return (int64_t)m * e.ldc; }
  static __device__ __forceinline__ float finish(const EpiF32<T>&, float x) { return x; }
};
template <>
struct RingDest<EpiPartial> {
  using Elem = float;
  static __device__ __forceinline__ float* column(const EpiPartial& e, int z, int n) { return e.ws + (int64_t)z * e.mn + n; }
  static __device__ __forceinline__ int64_t row(const EpiPartial& e, int m) { return (int64_t)m * e.ldn; }
  static __device__ __forceinline__ float finish(const EpiPartial&, float x) { return x; }
};
template <typename T, bool PAD>
struct RingDest<EpiQkvSplit<T, PAD>> {
  using Elem = T;
  static __device__ __forceinline__ T* column(const EpiQkvSplit<T, PAD>& e, int, int n) { return e.col_part((uint32_t)n); }
  static __device__ __forceinline__ int64_t row(const EpiQkvSplit<T, PAD>& e, int m) { return e.row_part(m); }
  static __device__ __forceinline__ float finish(const EpiQkvSplit<T, PAD>&, float x) { return x; }
};

template <>
struct RingDest<EpiInt32> {
  using Elem = int32_t;
  static __device__ __forceinline__ int32_t* column(const EpiInt32& e, int, int n) { return e.c + n; }
  static __device__ __forceinline__ int64_t row(const EpiInt32& e, int m) { return (int64_t)m * e.ldc; }
};
template <>
struct RingDest<EpiDequant> {
  using Elem = float;
  static __device__ __forceinline__ float* column(const EpiDequant& e, int, int n) { return e.c + n; }
  static __device__ __forceinline__ int64_t row(const EpiDequant& e, int m) { return (int64_t)m * e.ldc; }
  static __device__ __forceinline__ float finish(const EpiDequant&, int x) { return __builtin_bit_cast(float, x); }
};
template <>
struct RingDest<EpiDequantQkvSplit> {
  using Elem = float;
  static __device__ __forceinline__ float* column(const EpiDequantQkvSplit& e, int, int n) { return e.split.col_part((uint32_t)n); }
  static __device__ __forceinline__ int64_t row(const EpiDequantQkvSplit& e, int m) { return e.split.row_part(m); }
  static __device__ __forceinline__ float finish(const EpiDequantQkvSplit&, int x) { return __builtin_bit_cast(float, x); }
};

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(const F& f, std::integer_sequence<int, I...>) {
  (f(template_int<I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(const F& f) {  // f(0), ..., f(N - 1) with compile-time arguments
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Rows of 32-bit results (operands swapped: of block (i, j) a lane owns four columns of a row): 16 bytes a store straight from the
// accumulators, the four lanes of a row side by side.  (Eight columns a lane, as 16-bit results are stored, are two stores that
// each touch every other 16 bytes of a row: BERT base, us a pass, so / here: int8 20 x 128 tokens 1341 / 1314, fp32 20 x 100 1756 / 1722.)
// What a lane needs of its columns, requested before the K loop.
template <typename BT, int CB, bool SCALE>
struct ColumnQuads {
  Vec<BT, 4> bias[CB];
  float4 scale[SCALE ? CB : 1];
  bool present;
  // `fallback`: as in BiasVec
  __device__ __forceinline__ void load(const BT* b, const float* w_scale, int n_first, int n, int lgrp, const void* fallback) {
    present = b != nullptr;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const int col = min(n_first + j * 16 + lgrp * 4, n - 4);
      bias[j] = load_vec<BT, 4>(present ? b + col : static_cast<const BT*>(fallback));
      if constexpr (SCALE) scale[j] = *reinterpret_cast<const float4*>(w_scale + col);
    }
  }
};
// read(i, j, e): element e of the lane's part of block (i, j).  through: see writes_through().
template <int RB, int CB, typename Epi, typename Quads, typename Read>
__device__ __forceinline__ void store_rows32(const GemmArgs& g, const Epi& epi, const Quads& quads, int z_epi, int m_first, int n_first, int lrow, int lgrp,
                                             float& amax, bool through, const Read& read) {
  using Dest = RingDest<Epi>;
  using Elem = typename Dest::Elem;
  float act_scale = 0.f;
  if constexpr (Dequantises<Epi>::value) act_scale = epi.act_scale[0];
  int64_t row_at[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) row_at[i] = Dest::row(epi, min(m_first + i * 16 + lrow, g.m - 1));
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int n = n_first + j * 16 + lgrp * 4;  // (N is a multiple of eight: the four columns are all inside, or none)
    Elem* const col = Dest::column(epi, z_epi, min(n, g.n - 4));
    float wide[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) wide[e] = quads.present ? to_float(quads.bias[j].v[e]) : 0.f;
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      Vec<Elem, 4> out;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (Dequantises<Epi>::value) {
          const float scale[4] = {quads.scale[j].x, quads.scale[j].y, quads.scale[j].z, quads.scale[j].w};
          out.v[e] = epi.activate(dequantise(read(i, j, e), act_scale, scale[e], wide[e], quads.present));
          amax = fmaxf(amax, fabsf(out.v[e]));
        } else if constexpr (std::is_same<Elem, int32_t>::value) {
          out.v[e] = read(i, j, e);
        } else {
          out.v[e] = Dest::finish(epi, read(i, j, e) + wide[e]);
        }
      }
      if (m_first + i * 16 + lrow < g.m && n < g.n) {
        if constexpr (AddsResidual<Epi>::value) {
          const Vec<Elem, 4> res = load_vec<Elem, 4>(epi.residual + (col - epi.c) + row_at[i]);
#pragma unroll
          for (int e = 0; e < 4; ++e) out.v[e] += res.v[e];
        }
        if (through) store_through(col + row_at[i], out);
        else store_vec<Elem, 4>(col + row_at[i], out);
      }
    }
  }
}

// Tiles of 32 rows are for launches that store little: they are compiled without the question.  So are those of int8, which come in
// two forms: its products are short (4 x 128 tokens, the head split in 128 x 64 tiles 7.5 us with the question, 7.2 without).
enum class Stores { kAsk, kStay, kThrough };
template <typename Epi>
constexpr Stores default_stores(int tile_rows) { return tile_rows > 32 && !Dequantises<Epi>::value ? Stores::kAsk : Stores::kStay; }
// The stores of a launch of whole output tiles: written through where they are many.  The head split of int8, whose
// tiles leave in pieces of a head's 256 bytes, only from 12 MiB on.  us a forward of int8, its stores staying / through, the other products' as
// they are: base 4 x 128 tokens (4.5 MiB) 770 / 779, 5 x 128 (5.6) 785 / 790, 8 x 128 (9) 900 / 907, 10 x 128 (11.3)
// 933 / 936, 12 x 128 (13.5) 1005 / 1000, 20 x 128 (22.5) 1223 / 1219; large 3 x 128 (4.5) 1725 / 1738, 6 x 128 (9) 2064 / 2067, 8 x 128 (12) 2163 /
// 2152; 512 wide 6 x 128 (4.5) 1925 / 1957, 8 x 128 (6) 1986 / 2000, 12 x 128 (9) 2266 / 2269, 16 x 128 (12) 2366 / 2359.  Its other products from
// 2 MiB on, as everywhere: base 4 x 128 (up to 6 MiB) 770 / 762, 6 x 128 848 / 831, 16 x 128 1126 / 1092, 20 x 100 1136 / 1102; large 4 x 128
// 1838 / 1808; only 512 wide 4 x 128 (4 MiB) 1815 / 1819.
template <typename Epi>
inline bool stores_through(const GemmArgs& g) {
  const int64_t bytes = (int64_t)g.m * g.n * g.slices * (int64_t)sizeof(typename RingDest<Epi>::Elem);
  // The products of many rounds of tiles stay: 24576 x 1024 x 4096 in bf16, 101 MB of fp32, 196 us / 206 through
  constexpr int64_t kMostThrough = 90ll << 20, kInt8HeadsThrough = 12ll << 20;
  return bytes <= kMostThrough && (std::is_same<Epi, EpiDequantQkvSplit>::value ? bytes >= kInt8HeadsThrough : writes_through(bytes));
}

template <int BM, int BN, int NS>
constexpr int ring_lds_bytes() { return NS * (BM + BN) * kRowBytes; }

// A workgroup of WM x WN wavefronts owns one BM x BN tile (and, with g.k_chunk, one K slice of it).  LDS: NS stages of
// [A rows | B rows], 128 bytes of K per row, XOR-swizzled as in gemm_w4.h.
// K step s: multiply its first half while its second half is read and the rest of step s - 1 + NS is requested; wait until
// step s + 1 has landed (the NS - 2 younger steps stay in flight) and everyone has read step s; multiply the second half
// while the first half of step s + 1 is read and the first loads of step s + NS go into the stage just freed.
template <typename T, int BM, int BN, int WM, int WN, int NS, typename Epi, Stores STORES>
__global__ __launch_bounds__(WM * WN * kWave, 1) void gemm_ring_kernel(const GemmArgs g, const Epi epi) {
  constexpr int NW = WM * WN;
  constexpr int RB = BM / WM / 16, CB = BN / WN / 16;  // 16 x 16 blocks per wavefront
  constexpr int A_BYTES = BM * kRowBytes, B_BYTES = BN * kRowBytes, STAGE = A_BYTES + B_BYTES;
  constexpr int A_LOADS = BM / 8 / NW, B_LOADS = BN / 8 / NW, LOADS = A_LOADS + B_LOADS;
  constexpr int L1 = LOADS / 2, L0 = LOADS - L1;  // loads issued behind the barrier of a step / in the next step's first half
  constexpr int YOUNGER = (NS - 2) * LOADS;       // loads that may be in flight at a step's barrier
  static_assert(BM / 8 % NW == 0 && BN / 8 % NW == 0, "tile rows must split evenly over the wavefronts");
  static_assert(CB % 2 == 0, "blocks are stored in pairs");
  static_assert(NS >= 2 && YOUNGER < 64, "vmcnt is a six-bit counter");
  using MB = RingMma<T>;
  using Acc = typename MB::Acc;

  extern __shared__ __align__(16) char smem[];

  // One index over slices and tiles, so that the padding to whole XCDs is at most seven workgroups: with a padded row of
  // tiles per slice, 252 workgroups became 264, an XCD got 33 for its 32 CUs and one CU two of them (fp32 896 x 768 x 3072
  // in three slices: 63 us instead of 36).
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
  int tile_m, tile_n;
  tile_coords(logical, g.tiles_m, g.tiles_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm0 = (wave / WN) * (BM / WM), wn0 = (wave % WN) * (BN / WN);
  const int lrow = lane & 15, lgrp = lane >> 4;
  const int a_row0 = (wm0 + lrow) * kRowBytes, b_row0 = A_BYTES + (wn0 + lrow) * kRowBytes;
  const int swz = (lrow >> 1) & 7;
  int kdim = g.k, z_epi = 0;
  uint32_t k_lo = 0;  // bytes
  if (g.k_chunk > 0) {
    const int lo = slice * g.k_chunk;
    kdim = min(g.k_chunk, g.k - lo);
    k_lo = (uint32_t)lo * (uint32_t)sizeof(T);
    z_epi = slice;
  }
  const int ksteps = kdim / (kRowBytes / (int)sizeof(T));

  // ---- load cursor: per-lane offsets of this wavefront's rows (rows past the edge repeat the last one)
  const uint32_t lda_bytes = (uint32_t)(g.lda * (int64_t)sizeof(T)), ldb_bytes = (uint32_t)(g.ldb * (int64_t)sizeof(T));
  uint32_t voff[LOADS];
  {
    const int sub = lane >> 3, p = lane & 7;
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int row = (wave * A_LOADS + i) * 8 + sub;
      voff[i] = (uint32_t)min(m0 + row, g.m - 1) * lda_bytes + ((p ^ ((row >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
      const int row = (wave * B_LOADS + i) * 8 + sub;
      voff[A_LOADS + i] = (uint32_t)min(n0 + row, g.n - 1) * ldb_bytes + ((p ^ ((row >> 1) & 7)) << 4);
    }
  }
  int dma_step = 0, dma_stage = 0;
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) char lds_char;
  lds_char* lds0 = reinterpret_cast<lds_char*>(reinterpret_cast<uintptr_t>(smem));
  const int a_size = (int)((int64_t)g.m * lda_bytes), b_size = (int)((int64_t)g.n * ldb_bytes);
  auto issue_one = [&](int i) __attribute__((always_inline)) {
    const bool live = dma_step < ksteps;
    if (i < A_LOADS) {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(g.a), 0, live ? a_size : 0, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds0 + dma_stage + (wave * A_LOADS + i) * 1024, 16, voff[i], k_lo + dma_step * kRowBytes, 0, 0);
    } else {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(g.b), 0, live ? b_size : 0, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds0 + dma_stage + A_BYTES + (wave * B_LOADS + i - A_LOADS) * 1024, 16, voff[i], k_lo + dma_step * kRowBytes, 0, 0);
    }
  };
#else
  auto issue_one = [&](int) {};
#endif
  auto advance = [&]() __attribute__((always_inline)) {
    ++dma_step;
    dma_stage = dma_stage == (NS - 1) * STAGE ? 0 : dma_stage + STAGE;
  };

  Chunk fa[2][RB], fb[2][CB];
  Acc acc[RB][CB];
  constexpr int READS = RB + CB, BLOCKS = RB * CB, MMAS = BLOCKS * MB::PARTS;
  constexpr int RPM = (READS + MMAS - 1) / MMAS;  // reads per matrix instruction
  // Fragment reads are written as instructions: in front of an LDS read that it knows of, the compiler waits for EVERY
  // global -> LDS load in flight (vmcnt(0) in each half step), which empties the ring.  They are ordered by hand: behind a
  // barrier that their stage has passed, and landed() before the first use names every register they wrote.
  auto read_a = [&](Chunk& dst, uint32_t at, auto i) __attribute__((always_inline)) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(reinterpret_cast<Quad&>(dst)) : "v"(at), "n"(decltype(i)::value * 16 * kRowBytes) : "memory");
  };
  const uint32_t lds_base = (uint32_t)reinterpret_cast<uintptr_t>(smem);  // low half of a generic LDS address = LDS offset
  auto landed = [&](Chunk (&a)[RB], Chunk (&b)[CB]) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < RB; ++i) asm volatile("" : "+v"(reinterpret_cast<Quad&>(a[i])));
#pragma unroll
    for (int j = 0; j < CB; ++j) asm volatile("" : "+v"(reinterpret_cast<Quad&>(b[j])));
  };
  // LO, NL: the loads of the cursor's step issued here, evenly spread over the matrix instructions
  auto substep = [&](auto swap_tag, auto cur_tag, auto sub_tag, auto lo_tag, auto nl_tag, int rd) __attribute__((always_inline)) {
    constexpr bool SWAP = decltype(swap_tag)::value;
    constexpr int CUR = decltype(cur_tag)::value, SUB = decltype(sub_tag)::value, LO = decltype(lo_tag)::value, NL = decltype(nl_tag)::value;
    const uint32_t off = (uint32_t)(((SUB * 4 + lgrp) ^ swz) << 4) + (uint32_t)rd + lds_base;
    const uint32_t a_at = a_row0 + off, b_at = b_row0 + off;
    static_for<MMAS>([&](auto m_tag) __attribute__((always_inline)) {
      constexpr int m = decltype(m_tag)::value;
      constexpr int part = m / BLOCKS, blk = m % BLOCKS, i = blk / CB, j = blk % CB;  // (a block's parts apart: they form a chain)
      if constexpr (SWAP) MB::run(fb[CUR][j], fa[CUR][i], acc[i][j], part);
      else MB::run(fa[CUR][i], fb[CUR][j], acc[i][j], part);
      // the fragments of the next half step, read as early as one per instruction allows
      static_for<RPM>([&](auto r_tag) __attribute__((always_inline)) {
        constexpr int r = m * RPM + decltype(r_tag)::value;
        if constexpr (r < RB) read_a(fa[CUR ^ 1][r], a_at, template_int<r>{});
        else if constexpr (r < READS) read_a(fb[CUR ^ 1][r - RB], b_at, template_int<r - RB>{});
      });
#pragma unroll
      for (int l = m * NL / MMAS; l < (m + 1) * NL / MMAS; ++l) issue_one(LO + l);
      __builtin_amdgcn_sched_barrier(0);
    });
    landed(fa[CUR ^ 1], fb[CUR ^ 1]);
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- prologue: NS - 1 steps and the first part of one more are requested, the first step has landed
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) issue_one(i);
    advance();
  }
#pragma unroll
  for (int i = 0; i < L1; ++i) issue_one(i);

  const auto* bias = epi.bias_ptr();
  using BiasT = typename std::remove_cv<typename std::remove_pointer<decltype(bias)>::type>::type;
  BiasVec<BiasT> bv[CB / 2];
  auto unit_chunk = [&](int p) __attribute__((always_inline)) { return 2 * (2 * p + (lgrp & 1)) + (lgrp >> 1); };

#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0;
      asm volatile("" : "+a"(acc[i][j]));
    }
  asm volatile("s_nop 7");  // (the matrix instructions are inline asm: no hazard is seen between them and the zeroing)
  dma_landed_barrier_but<(NS - 2) * LOADS + L1>();
  {
    const uint32_t off = (uint32_t)((lgrp ^ swz) << 4) + lds_base;
    static_for<RB>([&](auto i) __attribute__((always_inline)) { read_a(fa[0][decltype(i)::value], a_row0 + off, i); });
    static_for<CB>([&](auto j) __attribute__((always_inline)) { read_a(fb[0][decltype(j)::value], b_row0 + off, j); });
    landed(fa[0], fb[0]);
  }
  auto k_loop = [&](auto swap_tag) __attribute__((always_inline)) {
    int rd = 0;
#pragma unroll 1
    for (int s = 0; s < ksteps; ++s) {
      substep(swap_tag, template_int<0>{}, template_int<1>{}, template_int<L1>{}, template_int<L0>{}, rd);
      advance();
      __builtin_amdgcn_sched_barrier(0);
      dma_landed_barrier_but<YOUNGER>();
      __builtin_amdgcn_sched_barrier(0);
      rd = rd == (NS - 1) * STAGE ? 0 : rd + STAGE;
      substep(swap_tag, template_int<1>{}, template_int<0>{}, template_int<0>{}, template_int<L1>{}, rd);
    }
    asm volatile("s_nop 15\n\ts_nop 15");
  };

  float amax = 0.f;
  const bool through = STORES == Stores::kThrough || (STORES == Stores::kAsk && g.write_through);
  bool swap = true;
  if constexpr (HasColumnPass<Epi>::value) swap = !(epi.column_pass() && n0 + wn0 >= epi.first_column_of_pass());
  using Dest = RingDest<Epi>;
  if (swap) {
    if constexpr (sizeof(typename Dest::Elem) == 4) {
      ColumnQuads<BiasT, CB, Dequantises<Epi>::value> quads;
      const float* w_scale = nullptr;
      if constexpr (Dequantises<Epi>::value) w_scale = epi.w_scale;
      quads.load(bias, w_scale, n0 + wn0, g.n, lgrp, g.b);
      k_loop(std::true_type{});
      store_rows32<RB, CB>(g, epi, quads, z_epi, m0 + wm0, n0 + wn0, lrow, lgrp, amax, through,
                           [&](int i, int j, int e) __attribute__((always_inline)) { return acc_read(acc[i][j][e]); });
    } else {
#pragma unroll
      for (int p = 0; p < CB / 2; ++p) bv[p].load(bias, min(n0 + wn0 + unit_chunk(p) * 8, g.n - 8), g.b);
      k_loop(std::true_type{});
      // Destination of a unit = a part that depends on its columns + a part that depends on its row, each found once.
      typename Dest::Elem* col_at[CB / 2];
      int64_t row_at[RB];
#pragma unroll
      for (int p = 0; p < CB / 2; ++p) col_at[p] = Dest::column(epi, z_epi, min(n0 + wn0 + unit_chunk(p) * 8, g.n - 8));
#pragma unroll
      for (int i = 0; i < RB; ++i) row_at[i] = Dest::row(epi, min(m0 + wm0 + i * 16 + lrow, g.m - 1));
#pragma unroll
      for (int p = 0; p < CB / 2; ++p) {
        const int n = n0 + wn0 + unit_chunk(p) * 8;
        float wide[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) wide[e] = 0.f;
        if (bias != nullptr) bv[p].widen(wide);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          float out[8];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            auto a = acc_read(acc[i][2 * p][e]), b = acc_read(acc[i][2 * p + 1][e]);
            pair_swap<16>(a, b);
            out[e] = a;
            out[4 + e] = b;
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) out[e] += wide[e];
          const int m = m0 + wm0 + i * 16 + lrow;
          if (m < g.m && n < g.n) {
            float fin[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) fin[e] = Dest::finish(epi, out[e]);
            if constexpr (AddsResidual<Epi>::value) {
              float res[8];
              load_row8(epi.residual + (col_at[p] - epi.c) + row_at[i], res);
#pragma unroll
              for (int e = 0; e < 8; ++e) fin[e] += res[e];
            }
            Vec<typename Dest::Elem, 8> rounded;
#pragma unroll
            for (int e = 0; e < 8; ++e) rounded.v[e] = from_float<typename Dest::Elem>(fin[e]);
            if (through) store_through(col_at[p] + row_at[i], rounded);
            else store_vec(col_at[p] + row_at[i], rounded);
          }
        }
      }
    }
  } else {
    if constexpr (HasColumnPass<Epi>::value) {
      float bj[CB];
      load_bias_columns_stride<CB, 16>(epi, n0 + wn0 + lrow, g.n, bj);
      k_loop(std::false_type{});
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const int n = n0 + wn0 + j * 16 + lrow;
        if constexpr (RB % 2 == 0) {
#pragma unroll
          for (int p = 0; p < RB / 2; ++p) {
            float out[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float a = acc_read(acc[2 * p][j][e]), b = acc_read(acc[2 * p + 1][j][e]);
              pair_swap<16>(a, b);
              out[e] = a + bj[j];
              out[4 + e] = b + bj[j];
            }
            const int m = m0 + wm0 + unit_chunk(p) * 8;
            if (m < g.m && n < g.n) epi.store_col8(m, g.m, n, out);
          }
        } else {
#pragma unroll
          for (int i = 0; i < RB; ++i) {
            float out[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = acc_read(acc[i][j][e]) + bj[j];
            const int m = m0 + wm0 + i * 16 + lgrp * 4;
            if (m < g.m && n < g.n) epi.store_col4(m, g.m, n, out);
          }
        }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the loads past the last step have returned before the LDS is given back
  publish_absmax(epi, amax, reinterpret_cast<float*>(smem), NW * kWave);
}

template <typename T, int BM, int BN, int WM, int WN, int NS, typename Epi>
inline int launch_ring(GemmArgs g, const Epi& epi, int slices, hipStream_t s) {
  constexpr int LDS = ring_lds_bytes<BM, BN, NS>();
  static_assert(LDS <= kLdsPerCu, "tile does not fit in LDS");
  if (describe_only("dma", WM * WN, BM, BN, slices)) return 0;
  g.tiles_m = (g.m + BM - 1) / BM;
  g.tiles_n = (g.n + BN - 1) / BN;
  g.slices = slices;
  const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n * slices;
  TTMI_REQUIRE(tiles < (1ll << 30), "GEMM grid too large");
  const unsigned grid_x = tiles >= kXcdRemapMinTiles ? (unsigned)(ceil_div(tiles, kNumXcd) * kNumXcd) : (unsigned)tiles;
  if (!absmax_grid_ok(epi, grid_x, 1)) return launch_ring<T, BM, BN, WM, WN, NS>(g, without_absmax(epi), slices, s);
  g.write_through = stores_through<Epi>(g);
  auto launch = [&](auto kern) -> int {
    if (LDS > 64 * 1024) {
      const int rc = allow_large_lds(reinterpret_cast<const void*>(kern), LDS);
      if (rc != 0) return rc;
    }
    hipLaunchKernelGGL(kern, dim3(grid_x), dim3(WM * WN * kWave), LDS, s, g, epi);
    return launch_status("gemm_ring_kernel");
  };
  if constexpr (Dequantises<Epi>::value)
    if (g.write_through) return launch(gemm_ring_kernel<T, BM, BN, WM, WN, NS, Epi, Stores::kThrough>);
  return launch(gemm_ring_kernel<T, BM, BN, WM, WN, NS, Epi, default_stores<Epi>(BM)>);
}

// ------------------------------------------------------------------------ selection -----
// Tiles and the time model that picks one, in microseconds.  With q = workgroups per CU (rounded up) and R = how many of
// them are resident there at once,
//   time = first + again * (q - 1) + K steps * max(lone * ceil(q / R), shared * q):
// `first` and `again` are what a workgroup costs beyond its K loop (launch, first operands, epilogue), `lone` a K step of
// a workgroup that waits for its own latencies, `shared` one on a CU whose matrix pipe or operand path is full.  The
// numbers are least-squares fits to launches of M = 72 ... 16384 rows by the four encoder products of hidden 768 and
// 1024 (fp16, fp32, int8); over those the tile the model picks is 0.3 % (fp32: 2.5 %) slower than the best one.
// Tiles of 160 rows or columns (16-bit) stand between those that powers of two give: where 128 x 192 are just too many for a round or
// leave a quarter of the CUs idle.  us, the best tile without / with them: 6275 x 3072 x 768 40.8 / 35.1 (256 x 160), 6275 x 768 x 3072 29.9 /
// 27.9, 3200 x 3072 x 768 23.0 / 20.5, 2560 x 4096 x 1024 27.4 / 24.7 (160 x 128), 800 x 3072 x 768 8.5 / 7.7 (160 x 64); a forward: base
// fp16 49 x 128 tokens 1704 / 1612, 20 packed requests 1786 / 1704, 25 x 128 1005 / 993, 3 x 300 637 / 625, large bf16 20 x 128 2594 / 2520, 8 x 100 1478 / 1444.
// (96 x 192, 160 x 192, 192 x 128, 192 x 192, 96 x 128, 192 x 96 and 128 x 160 as well: 0.1 % more over those launches.)
struct RingTile {
  int bm, bn, wave_cols, resident;
  float first, again, lone, shared;
  bool lone_block;  // a wavefront's 16-row blocks do not pair up: a column of V leaves by the four rows, not by eight
};
// X(BM, BN, WM, WN, stages, resident, first, again, lone, shared)
#define TTMI_RING_TILES_16(X)                                \
  X(32, 64, 2, 2, 4, 3, 2.90f, 0.27f, 0.152f, 0.128f)        \
  X(64, 64, 4, 2, 4, 2, 3.10f, 0.65f, 0.177f, 0.177f)        \
  X(64, 96, 4, 1, 4, 2, 3.27f, 1.15f, 0.188f, 0.212f)        \
  X(128, 64, 2, 2, 4, 1, 3.19f, 2.17f, 0.252f, 0.252f)       \
  X(160, 64, 2, 2, 4, 1, 3.40f, 2.60f, 0.305f, 0.305f)       \
  X(128, 96, 4, 1, 3, 1, 3.58f, 2.66f, 0.325f, 0.326f)       \
  X(128, 128, 4, 2, 3, 1, 3.74f, 4.03f, 0.374f, 0.373f)      \
  X(160, 128, 2, 2, 3, 1, 4.65f, 5.20f, 0.411f, 0.411f)      \
  X(128, 192, 4, 2, 3, 1, 4.88f, 6.69f, 0.464f, 0.461f)      \
  X(256, 128, 4, 2, 3, 1, 5.36f, 8.33f, 0.576f, 0.571f)      \
  X(256, 160, 4, 1, 3, 1, 7.10f, 9.60f, 0.661f, 0.661f)
#define TTMI_RING_TILES_32(X)                                \
  X(32, 64, 2, 2, 4, 3, 3.40f, 0.11f, 0.215f, 0.263f)        \
  X(64, 64, 2, 2, 3, 3, 3.83f, 0.22f, 0.332f, 0.499f)        \
  X(64, 64, 4, 2, 4, 2, 4.58f, 0.82f, 0.126f, 0.480f)        \
  X(64, 96, 4, 1, 3, 2, 4.90f, 1.32f, 0.680f, 0.671f)        \
  X(64, 128, 4, 2, 3, 2, 5.03f, 0.97f, 0.272f, 0.907f)       \
  X(64, 192, 4, 2, 3, 1, 4.43f, 7.73f, 1.399f, 1.392f)       \
  X(128, 192, 4, 2, 3, 1, 6.53f, 10.7f, 2.684f, 2.683f)
#define TTMI_RING_TILES_8(X)                                 \
  X(32, 64, 2, 2, 4, 3, 3.55f, 0.74f, 0.141f, 0.120f)        \
  X(64, 64, 4, 2, 4, 2, 4.06f, 1.59f, 0.173f, 0.173f)        \
  X(64, 96, 4, 1, 4, 2, 5.47f, 2.29f, 0.203f, 0.214f)        \
  X(128, 64, 2, 2, 4, 1, 5.08f, 4.03f, 0.258f, 0.258f)       \
  X(64, 192, 4, 2, 3, 1, 6.02f, 5.34f, 0.379f, 0.377f)       \
  X(128, 128, 4, 2, 3, 1, 6.55f, 6.98f, 0.376f, 0.376f)      \
  X(128, 192, 4, 2, 3, 1, 8.73f, 10.6f, 0.465f, 0.465f)      \
  X(256, 128, 4, 2, 3, 1, 11.0f, 10.9f, 0.594f, 0.594f)

// X(BM, BN, WM, WN, K groups, A steps in registers, B stages, resident, first, again, lone, shared): fp32 with packed weights
// (gemm_split.h).  Fits of the same kind (M = 40 ... 10240, K = 256 ... 3072; the tile the model picks is 0.1 % slower than the best one).
// 96 x 192 in twelve wavefronts is for a head split just short of a round of 128 x 192, whose stores the smaller tile takes better: 2000 x 2304 x 768
// at 100 tokens 27.1 / 22.8 us, a forward of base fp32 20 x 100 1540 / 1512, 20 x 200 2717 / 2590.  (The other products gain in a loop, 1600 x 3072 x
// 768 24.6 / 21.6, and lose in a forward, where the chip is at its power limit: 15 x 100 1420 / 1425, 12 x 128 1410 / 1414.  Four or six wavefronts 5 %
// more; 96 x 128, 160 x 64, 160 x 128 and 128 x 160 win nowhere.)
#define TTMI_SPLIT_TILES(X)                                        \
  X(32, 32, 2, 1, 4, 4, 5, 1, 4.80f, 3.23f, 0.100f, 0.100f)        \
  X(32, 64, 2, 2, 1, 4, 6, 2, 3.02f, 1.19f, 0.260f, 0.161f)        \
  X(32, 64, 2, 2, 3, 2, 4, 1, 4.55f, 3.18f, 0.154f, 0.154f)        \
  X(64, 64, 4, 2, 1, 4, 6, 2, 3.97f, 1.59f, 0.298f, 0.246f)        \
  X(64, 64, 2, 2, 2, 2, 4, 1, 4.69f, 3.90f, 0.233f, 0.234f)        \
  X(64, 128, 2, 4, 1, 4, 6, 1, 4.47f, 4.90f, 0.390f, 0.389f)       \
  X(64, 192, 4, 2, 1, 2, 4, 1, 4.96f, 7.32f, 0.508f, 0.509f)       \
  X(64, 256, 2, 4, 1, 2, 4, 1, 5.62f, 9.16f, 0.603f, 0.603f)       \
  X(128, 128, 4, 2, 1, 2, 4, 1, 5.71f, 9.31f, 0.573f, 0.573f)      \
  X(96, 192, 6, 2, 1, 2, 4, 1, 6.60f, 7.50f, 0.620f, 0.620f)       \
  X(128, 192, 4, 2, 1, 2, 4, 1, 7.29f, 13.8f, 0.738f, 0.738f)

#define TTMI_RING_ROW(BM, BN, WM, WN, NS, R, F, A, L, S) RingTile{BM, BN, BN / WN, R, F, A, L, S, BM / WM / 16 > 1 && BM / WM / 16 % 2 != 0},
#define TTMI_SPLIT_ROW(BM, BN, WM, WN, KG, DA, SB, R, F, A, L, S) RingTile{BM, BN, BN / WN, R, F, A, L, S, BM / WM / 16 > 1 && BM / WM / 16 % 2 != 0},
template <size_t ELEM>
struct RingTiles;
template <>
struct RingTiles<2> {
  static constexpr RingTile k[] = {TTMI_RING_TILES_16(TTMI_RING_ROW)};
};
template <>
struct RingTiles<4> {
  static constexpr RingTile k[] = {TTMI_RING_TILES_32(TTMI_RING_ROW)};
};
template <>
struct RingTiles<1> {
  static constexpr RingTile k[] = {TTMI_RING_TILES_8(TTMI_RING_ROW)};
};
struct SplitTiles {
  static constexpr RingTile k[] = {TTMI_SPLIT_TILES(TTMI_SPLIT_ROW)};
};
#undef TTMI_RING_ROW
#undef TTMI_SPLIT_ROW

enum class RingUse { kWhole, kSliced, kCut, kLayerNorm };  // never cut along K / cut where it pays / always cut / slices summed by the LayerNorm
struct RingPlan {
  int tile = -1, slices = 1;
  int64_t rounds = 0;  // workgroups per CU, rounded up
  int tile_values = 0;
  double us = 1e300;
};

// column_limit > 0: a wavefront's columns must not straddle it (the start of a transposed V), and its rows come in pairs of blocks (a
// forward of fp16 base, without / with tiles of 160 rows there, 16 x 128 tokens 718 / 724 us, 20 x 100 733 / 736)
// head_split: tiles of kHeadSplitRows rows are for it alone (above) and for up to kHeadSplitRounds workgroups a CU, and it has registers for kRingWidestSplit
// columns of a wavefront.  Beyond, the launch is long enough that the chip runs at its power limit, which the model does not know: us per forward of base fp32,
// without / with such tiles, 18 x 464 tokens 6019 / 6134, 20 x 440 6145 / 6259, 20 x 480 6445 / 6542, 24 x 500 8025 / 8088, 32 x 500 9872 / 10214; up to three
// rounds 19 x 100 1529 / 1495, 20 x 200 2746 / 2628, 12 x 460 4229 / 4036, 12 x 500 4334 / 4199.
constexpr int kHeadSplitRows = 96, kHeadSplitRounds = 3, kRingWidestSplit = 128;
template <typename Epi>
constexpr bool ring_takes(int rows, int wave_cols) { return HasColumnPass<Epi>::value ? wave_cols <= kRingWidestSplit : rows != kHeadSplitRows; }
constexpr int kRingColumns = 32;  // the narrowest wavefront's: a limit that is no multiple of it suits no tile
template <typename Tiles>
constexpr bool ring_columns_ok() {
  bool narrowest = false;
  for (const RingTile& t : Tiles::k) {
    if (t.wave_cols % kRingColumns != 0) return false;
    narrowest = narrowest || t.wave_cols == kRingColumns;
  }
  return narrowest;
}

// All tiles and slices are compared in front of every launch, so the loop over the slices has no divisions and ends where no
// number of slices can win any more (the partial products so far, and K shared evenly by all CUs, already take longer).
// Host time, ns, with a plain loop / so: fp32 128 x 768 x 3072 2070 / 260, fp16 8 x 768 x 3072 2310 / 190, 2000 x 768 x 3072
// 730 / 110, whole 145 / 80.
template <typename Tiles>
inline RingPlan pick_tile_of(int64_t m, int64_t n, int64_t ksteps, RingUse use, int64_t column_limit, bool head_split) {
  static_assert(ring_columns_ok<Tiles>(), "kRingColumns");
  constexpr uint32_t kMostSlices = 16;
  constexpr uint64_t kMostTiles = 1u << 27;  // (launch_ring refuses such grids: 32-bit arithmetic suffices)
  const uint32_t cus = (uint32_t)compute_units(), rows = (uint32_t)m, cols = (uint32_t)n, steps = (uint32_t)ksteps;
  const bool norm = use == RingUse::kLayerNorm;
  const double per_slice = m * n * 4 / 4e6;  // us: a partial product is written and read once more
  uint32_t most = use == RingUse::kWhole ? 1 : std::min(kMostSlices, std::max(1u, steps / 4));
  while (most > 1 && most * m * n * 4 > (32ll << 20)) --most;
  uint32_t share[kMostSlices + 1];
  for (uint32_t s = 1; s <= most; ++s) share[s] = (steps + s - 1) / s;
  RingPlan best;
  int index = 0;
  for (const RingTile& t : Tiles::k) {
    const int i = index++;
    if (head_split ? t.wave_cols > kRingWidestSplit : t.bm == kHeadSplitRows) continue;
    if (column_limit > 0 && (column_limit % t.wave_cols != 0 || t.lone_block)) continue;
    const uint32_t tiles = (uint32_t)std::min<uint64_t>((uint64_t)((rows + t.bm - 1) / t.bm) * ((cols + t.bn - 1) / t.bn), kMostTiles);
    if (t.bm == kHeadSplitRows && tiles > kHeadSplitRounds * cus) continue;
    const double least = t.first + steps * t.shared * (double)tiles / cus;
    uint32_t room = 0, q = 0;  // room: q workgroups on every CU
    for (uint32_t s = 1; s <= most; ++s) {
      // partial products, and a launch of their own where no LayerNorm follows
      const double extra = (s > 1 || norm ? s * per_slice : 0) + (s > 1 && !norm ? 4.0 : 0);
      if (least + extra > best.us) break;
      if (tiles * s > room) {
        q = s == 1 || tiles > cus ? (tiles * s + cus - 1) / cus : q + 1;
        room = q * cus;
      }
      if (use == RingUse::kCut && s == 1 && most > 1) continue;
      const double us = t.first + t.again * (q - 1.0) + share[s] * std::max<double>(t.lone * (q <= (uint32_t)t.resident ? 1 : (q + t.resident - 1) / t.resident), t.shared * q) + extra;
      if (us < best.us) best = RingPlan{i, (int)s, q, t.bm * t.bn, us};
    }
  }
  return best;
}
template <typename T>
inline RingPlan pick_ring(const GemmArgs& g, RingUse use, int64_t column_limit = 0, bool head_split = false) {
  const int64_t ksteps = g.k / (kRowBytes / (int)sizeof(T));
  if constexpr (sizeof(T) == 4)
    if (g.b_split != nullptr) return pick_tile_of<SplitTiles>(g.m, g.n, ksteps, use, column_limit, head_split);
  return pick_tile_of<RingTiles<sizeof(T)>>(g.m, g.n, ksteps, use, column_limit, head_split);
}

template <typename T>
inline bool ring_operands_ok(const GemmArgs& g) {  // 32-bit buffer offsets, columns in groups of eight
  const int64_t limit = (int64_t)1 << 31;
  return g.n % 8 == 0 && (int64_t)g.m * g.lda * (int64_t)sizeof(T) < limit && (int64_t)g.n * g.ldb * (int64_t)sizeof(T) < limit;
}

template <int BM, int BN, int WM, int WN, int KG, int DA, int SB, typename Epi>
int launch_split(GemmArgs g, const Epi& epi, int slices, hipStream_t s);  // gemm_split.h

template <typename T, typename Epi>
inline int launch_ring_tile(int tile, const GemmArgs& g, const Epi& epi, int slices, hipStream_t s) {
  int index = 0;
  if constexpr (sizeof(T) == 4) {
    if (g.b_split != nullptr) {
#define TTMI_SPLIT_TRY(BM, BN, WM, WN, KG, DA, SB, R, F, A, L, S) \
  if constexpr (ring_takes<Epi>(BM, BN / WN))                     \
    if (tile == index) return launch_split<BM, BN, WM, WN, KG, DA, SB>(g, epi, slices, s); \
  ++index;
      TTMI_SPLIT_TILES(TTMI_SPLIT_TRY)
#undef TTMI_SPLIT_TRY
      return fail(TTMI_EINVAL, "no such tile");
    }
  }
#define TTMI_RING_TRY(BM, BN, WM, WN, NS, R, F, A, L, S) \
  if constexpr (ring_takes<Epi>(BM, BN / WN))            \
    if (tile == index) return launch_ring<T, BM, BN, WM, WN, NS>(g, epi, slices, s); \
  ++index;
  if constexpr (sizeof(T) == 2) { TTMI_RING_TILES_16(TTMI_RING_TRY) }
  if constexpr (sizeof(T) == 4) { TTMI_RING_TILES_32(TTMI_RING_TRY) }
  if constexpr (sizeof(T) == 1) { TTMI_RING_TILES_8(TTMI_RING_TRY) }
#undef TTMI_RING_TRY
  return fail(TTMI_EINVAL, "no such tile");
}

// The product in `plan.slices` K slices: fp32 partial products in the split-K workspace, summed by `reduce(ws, slices, vec, stream)`.
template <typename T, typename Reduce>
inline int launch_ring_slices(GemmArgs g, const RingPlan& plan, hipStream_t s, const Reduce& reduce) {
  constexpr int BK = kRowBytes / (int)sizeof(T);
  g.k_chunk = (int)ceil_div(g.k / BK, plan.slices) * BK;
  const int used = (int)ceil_div(g.k, g.k_chunk);
  float* ws = nullptr;
  if (tl_describe == nullptr) {
    const int rc = splitk_workspace((size_t)used * g.m * g.n * sizeof(float), s, &ws);
    if (rc != 0) return rc;
  }
  const EpiPartial part{ws, (int64_t)g.m * g.n, g.n, true};
  const int rc = launch_ring_tile<T>(plan.tile, g, part, used, s);
  if (rc != 0 || tl_describe != nullptr) return rc;
  reduce(ws, used, true, s);
  return launch_status("gemm_ring_slices");
}

}  // namespace ttmi
