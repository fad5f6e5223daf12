// GEMM kernel for fp32 operands on gfx950 whose weights are packed (ttmi_split_weights): three products on the 16-bit matrix
// instruction in place of one on the fp32 instruction (split_f32.h).
//
//   C[M,N] = epilogue(A[M,K] * B[N,K]^T)   (both operands K-contiguous and 16-byte aligned, K a multiple of 128 bytes)
//
// What bounds it: up to some hundred rows the instructions of a step (below), then the matrix pipe: 128 x 192 tiles take 0.77 us a step
// against 0.55 of matrix time, and 10240 x 3072 x 768 runs at 0.98 PFLOP/s of 16-bit products, where fp16 tiles run.
// us per launch, fp32 ring tiles / here: 2000 x 2304 x 768 56 / 27, 2000 x 768 x 768 22.4 / 14.4, 2000 x 3072 x 768 (GELU) 73 / 31,
// 264 x 3072 x 768 16.5 / 10.9, 128 x 2304 x 768 9.9 / 8.0, 10240 x 768 x 3072 335 / 141.
#pragma once

#include "gemm_ring.h"
#include "split_f32.h"

namespace ttmi {

// The swizzle of an LDS row's 16-byte chunks: that of the ring tiles, and odd rows the other half of the row.  An 8-byte store
// instruction writes half a row of hi (or lo) per eight lanes, 128 bytes a cycle: two neighbouring rows must take different banks.
__device__ __forceinline__ int split_swizzle(int row) { return ((row >> 1) & 7) ^ ((row & 1) << 2); }

constexpr int kSplitStagesA = 3;
template <int BM, int BN, int SB>
constexpr int split_lds_bytes() { return (kSplitStagesA * BM + SB * BN) * kRowBytes; }

// A workgroup of WM x WN wavefronts owns one BM x BN tile (and, with g.k_chunk, one K slice of it).  LDS: three stages of A rows and
// SB of B rows, 32 values of K per row as 64 bytes of hi and 64 of lo.
// K step s: multiply, of one operand out of registers, of the other with a block read just ahead; meanwhile the fragments of
// step s + 1 are read, A's step s + 2, which has arrived in registers, is split and written (once per workgroup, not once per
// wavefront that multiplies it), its step s + 2 + DA is requested into the registers just read, and the halves of B's steps up to
// s + SB - 1 are on their way into LDS without passing a register.  All of it goes out between the matrix instructions: a wavefront
// issues an instruction every eight cycles, so what a step costs besides its matrix time is the number of its instructions
// (B split on the way in as well, 2000 x 3072 x 768: 35.7 us; fragments split by each wavefront behind LDS would be more still).
// KG > 1: as many such groups of wavefronts share a tile, each with its part of the K steps and stages of its own, and meet in LDS at
// the end.  Where the tiles are fewer than the CUs a step is a chain of waits, whose number this
// divides (us, one group / here: 128 x 768 x 3072 27 / 13.6, 128 x 768 x 768 8.5 / 7.0, 128 x 2304 x 768 9.0 / 8.0, 264 x 3072 x 768 12.0 / 10.9).
template <int BM, int BN, int WM, int WN, int KG, int DA, int SB, typename Epi>
__global__ __launch_bounds__(KG * WM * WN * kWave, 1) void gemm_split_kernel(const GemmArgs g, const Epi epi) {
  constexpr int NW = WM * WN, NT = NW * kWave, ROWS = NT / 8;  // of a group; a thread loads 16 bytes of A, eight threads a row
  constexpr int PASSES = BM / ROWS, B_LOADS = BN / 8 / NW;
  constexpr int RB = BM / WM / 16, CB = BN / WN / 16;    // 16 x 16 blocks per wavefront
  constexpr int A_STAGE = BM * kRowBytes, B_STAGE = BN * kRowBytes, B_BASE = kSplitStagesA * A_STAGE;
  constexpr int BK = kRowBytes / (int)sizeof(float);
  static_assert(BM % ROWS == 0 && BN / 8 % NW == 0 && ROWS % 16 == 0, "rows must split evenly over threads and wavefronts");
  static_assert(CB % 2 == 0, "blocks are stored in pairs");
  static_assert((DA == 2 || DA == 4) && SB >= 4 && (SB - 3) * (PASSES + B_LOADS) + 2 * PASSES + DA * PASSES < 64, "vmcnt is a six-bit counter");
  using Acc = floatx4;

  extern __shared__ __align__(16) char lds[];

  const int tiles = g.tiles_m * g.tiles_n, total = tiles * g.slices;  // (as in gemm_ring_kernel)
  const bool remap = total >= kXcdRemapMinTiles;
  const int per_xcd = (total + kNumXcd - 1) / kNumXcd;
  int logical = remap ? (int)(blockIdx.x % kNumXcd) * per_xcd + (int)(blockIdx.x / kNumXcd) : (int)blockIdx.x;
  if (logical >= total) return;
  int slice = 0;
  if (g.slices > 1) {
    slice = logical / tiles;
    logical -= slice * tiles;
  }
  int tile_m, tile_n;
  tile_coords(logical, g.tiles_m, g.tiles_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int group = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
  char* const smem = lds + group * split_lds_bytes<BM, BN, SB>();
  const int tid = threadIdx.x - group * NT, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm0 = (wave / WN) * (BM / WM), wn0 = (wave % WN) * (BN / WN);
  const int lrow = lane & 15, lgrp = lane >> 4;
  int kdim = g.k, z_epi = 0;
  uint32_t k_lo = 0;  // bytes
  if (g.k_chunk > 0) {
    const int lo = slice * g.k_chunk;
    kdim = min(g.k_chunk, g.k - lo);
    k_lo = (uint32_t)lo * (uint32_t)sizeof(float);
    z_epi = slice;
  }
  // a group's share: `ksteps` steps of K, of which the last group's may be short (a step past its `valid` ones reads zeros)
  const int ksteps = (kdim / BK + KG - 1) / KG, valid = KG > 1 ? max(min(kdim / BK - group * ksteps, ksteps), 0) : ksteps;
  if constexpr (KG > 1) k_lo += (uint32_t)(group * ksteps) * kRowBytes;

  // ---- loads (rows past the edge repeat the last one; steps past the last read zeros)
  const int sub = tid >> 3, kq = tid & 7;
  const uint32_t lda_bytes = (uint32_t)(g.lda * (int64_t)sizeof(float)), ldb_bytes = (uint32_t)(g.ldb * (int64_t)sizeof(float));
  uint32_t voff_a[PASSES], voff_b[B_LOADS];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) voff_a[p] = (uint32_t)min(m0 + p * ROWS + sub, g.m - 1) * lda_bytes + kq * 16;
#pragma unroll
  for (int i = 0; i < B_LOADS; ++i) {
    const int row = (wave * B_LOADS + i) * 8 + (lane >> 3);
    voff_b[i] = (uint32_t)min(n0 + row, g.n - 1) * ldb_bytes + (((lane & 7) ^ split_swizzle(row)) << 4);
  }
  floatx4 raw[DA][PASSES];
  float largest[PASSES];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) largest[p] = 0.f;
  static_assert(BN <= NT && KG * NW * (int)sizeof(int) <= 256, "a column per thread, an answer per wavefront");
  const int column_flag_here = tid < BN ? g.b_flags[min(n0 + tid, g.n - 1)] : 0;
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) char lds_char;
  lds_char* lds0 = reinterpret_cast<lds_char*>(reinterpret_cast<uintptr_t>(smem));
  const int a_size = (int)((int64_t)g.m * lda_bytes), b_size = (int)((int64_t)g.n * ldb_bytes);
  auto request_a = [&](int p, int step, floatx4& dst) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(g.a), 0, step < valid ? a_size : 0, 0x00020000);
    dst = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff_a[p], k_lo + step * kRowBytes, 0));
  };
  auto request_b = [&](int i, int step, int at) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(g.b_split), 0, step < valid ? b_size : 0, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds0 + at + (wave * B_LOADS + i) * 1024, 16, voff_b[i], k_lo + step * kRowBytes, 0, 0);
  };
#else
  auto request_a = [&](int, int, floatx4&) {};
  auto request_b = [&](int, int, int) {};
#endif

  // LDS is read and written by instructions: in front of an access that it knows of, the compiler waits for every load that is
  // on its way into LDS.  They are ordered by hand, by counted waits and the barrier of a step.
  const uint32_t lds_base = (uint32_t)reinterpret_cast<uintptr_t>(smem);  // low half of a generic LDS address = LDS offset
  auto lds_read = [&](Chunk& dst, uint32_t at, auto offset) __attribute__((always_inline)) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(reinterpret_cast<Quad&>(dst)) : "v"(at), "n"(decltype(offset)::value) : "memory");
  };
  auto lds_write = [&](uint32_t at, const uint32_t (&v)[2], auto offset) __attribute__((always_inline)) {
    asm volatile("ds_write_b64 %0, %1 offset:%2" : : "v"(at), "v"((uint64_t)v[0] | (uint64_t)v[1] << 32), "n"(decltype(offset)::value) : "memory");
  };
  auto landed = [&](Chunk& c) __attribute__((always_inline)) { asm volatile("" : "+v"(reinterpret_cast<Quad&>(c))); };

  // ---- the split of 16 bytes of A, in four parts (the matrix instructions go between them)
  const uint32_t put = lds_base + (uint32_t)(sub * kRowBytes + (((kq >> 1) ^ split_swizzle(sub)) << 4) + (kq & 1) * 8);
  uint32_t hi[2], lo[2];
  auto split_part = [&](auto part_tag, auto p_tag, floatx4& x, int wr, int next) __attribute__((always_inline)) {
    constexpr int PART = decltype(part_tag)::value, P = decltype(p_tag)::value;
    if constexpr (PART == 0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        hi[h] = split_hi(x[2 * h], x[2 * h + 1]);
        split_max(largest[P], x[2 * h], x[2 * h + 1]);
      }
    } else if constexpr (PART < 3) {
      lo[PART - 1] = split_lo(hi[PART - 1], x[2 * PART - 2], x[2 * PART - 1]);
    } else {
      lds_write(put + wr, hi, template_int<P * ROWS * kRowBytes>{});
      lds_write((put ^ 64) + wr, lo, template_int<P * ROWS * kRowBytes>{});
      request_a(P, next, x);
    }
  };

  // Of the operand with fewer blocks a step's fragments are held (two sets: the next step's are read meanwhile), those of the
  // other pass by, read one block ahead.
  constexpr bool HOLD_A = RB <= CB;
  constexpr int HELD = HOLD_A ? RB : CB, PASSING = HOLD_A ? CB : RB, GROUP = HELD * 3, MMAS = GROUP * PASSING, PARTS = PASSES * 4;
  Acc acc[RB][CB], cross[RB][CB];
  Chunk held[2][HELD][2], passing[2][2];
  const uint32_t get = lds_base + (uint32_t)(lrow * kRowBytes + ((lgrp ^ split_swizzle(lrow)) << 4));
  const uint32_t get_a = wm0 * kRowBytes + get, get_b = B_BASE + wn0 * kRowBytes + get;
  // (get's bits 4 to 6 come from the swizzle alone: every other part is a multiple of 128)
  const uint32_t get_held = HOLD_A ? get_a : get_b, get_passing = HOLD_A ? get_b : get_a;
  auto read_held = [&](auto par_tag, auto q_tag, uint32_t stage) __attribute__((always_inline)) {
    constexpr int PAR = decltype(par_tag)::value, Q = decltype(q_tag)::value;
    lds_read(held[PAR][Q / 2][Q % 2], (get_held ^ (Q % 2 * 64)) + stage, template_int<Q / 2 * 16 * kRowBytes>{});
  };
  auto read_passing = [&](auto buf_tag, auto blk_tag, uint32_t stage) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_tag)::value, BLK = decltype(blk_tag)::value;
    lds_read(passing[BUF][0], get_passing + stage, template_int<BLK * 16 * kRowBytes>{});
    lds_read(passing[BUF][1], (get_passing ^ 64) + stage, template_int<BLK * 16 * kRowBytes>{});
  };
  // LDS stages of a step: A's own, the next step's, the one written; B's own, the next step's, the one requested
  struct Stages {
    int a0, a1, a2, b0, b1, b_new;
  };
  auto k_step = [&](auto swap_tag, auto turn_tag, int s, const Stages& st) __attribute__((always_inline)) {
    constexpr bool SWAP = decltype(swap_tag)::value;
    constexpr int PAR = decltype(turn_tag)::value % 2, SLOT = (decltype(turn_tag)::value + 2) % DA;
    const uint32_t held_next = HOLD_A ? st.a1 : st.b1, passing_now = HOLD_A ? st.b0 : st.a0, passing_next = HOLD_A ? st.b1 : st.a1;
    static_for<MMAS>([&](auto m_tag) __attribute__((always_inline)) {
      constexpr int m = decltype(m_tag)::value;
      constexpr int p = m / GROUP, part = m % GROUP / HELD, h = m % HELD, buf = (PAR * PASSING + p) & 1;
      if constexpr (m % GROUP == 0) {
        if constexpr (p > 0) {  // the block read in the previous group, in front of `behind` other LDS instructions, has landed
          constexpr int behind = [] {
            int count = 0;
            for (int q = 0; q < 2 * HELD; ++q) count += q * MMAS / (2 * HELD) / GROUP == p - 1;
            for (int q = 3; q < PARTS; q += 4) count += 2 * (q * MMAS / PARTS / GROUP == p - 1);
            return count < 15 ? count : 15;
          }();
          asm volatile("s_waitcnt lgkmcnt(%0)" : : "n"(behind) : "memory");
          landed(passing[buf][0]);
          landed(passing[buf][1]);
        }
        if constexpr (p + 1 < PASSING) read_passing(template_int<buf ^ 1>{}, template_int<p + 1>{}, passing_now);
        else read_passing(template_int<buf ^ 1>{}, template_int<0>{}, passing_next);
      }
      const Chunk &x = held[PAR][h][part == 2], &y = passing[buf][part == 1];  // (the two products of `cross` apart: they form a chain)
      constexpr int i = HOLD_A ? h : p, j = HOLD_A ? p : h;
      Acc& c = part == 0 ? acc[i][j] : cross[i][j];
      if constexpr (SWAP == HOLD_A) MmaBlock<f16, 16>::run(y, x, c);
      else MmaBlock<f16, 16>::run(x, y, c);
      static_for<2 * HELD>([&](auto q_tag) __attribute__((always_inline)) {
        if constexpr (decltype(q_tag)::value * MMAS / (2 * HELD) == m) read_held(template_int<PAR ^ 1>{}, q_tag, held_next);
      });
      static_for<PARTS>([&](auto q_tag) __attribute__((always_inline)) {
        constexpr int q = decltype(q_tag)::value;
        if constexpr (q * MMAS / PARTS == m) split_part(template_int<q % 4>{}, template_int<q / 4>{}, raw[SLOT][q / 4], st.a2, s + 2 + DA);
      });
#pragma unroll
      for (int l = m * B_LOADS / MMAS; l < (m + 1) * B_LOADS / MMAS; ++l) request_b(l, s + SB - 1, B_BASE + st.b_new);
      __builtin_amdgcn_sched_barrier(0);
    });
    // B's step s + 2 has landed: requested SB - 3 steps ago, or in front of the loop, where DA of A's steps followed it at least
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((SB - 3) * B_LOADS + (SB - 3 < DA ? SB - 3 : DA) * PASSES) : "memory");
#pragma unroll
    for (int q = 0; q < 2 * HELD; ++q) landed(held[PAR ^ 1][q / 2][q % 2]);
    landed(passing[(PAR * PASSING + PASSING) & 1][0]);
    landed(passing[(PAR * PASSING + PASSING) & 1][1]);
    __builtin_amdgcn_sched_barrier(0);
  };

  static_for<SB - 1>([&](auto step_tag) __attribute__((always_inline)) {  // the two steps that are multiplied first in front
    constexpr int step = decltype(step_tag)::value;
    if constexpr (step < DA)
#pragma unroll
      for (int p = 0; p < PASSES; ++p) request_a(p, step, raw[step][p]);
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) request_b(i, step, B_BASE + step * B_STAGE);
  });

  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.f, cross[i][j][e] = 0.f;
        asm volatile("" : "+a"(acc[i][j]), "+a"(cross[i][j]));
      }
    asm volatile("s_nop 7");  // (the matrix instructions are inline asm: no hazard is seen between them and the zeroing)
  };
  floatx4 value[RB][CB];  // what the tile's (and group's) K steps add up to
  auto sum = [&](int i, int j, int e) __attribute__((always_inline)) {
    return __builtin_fmaf(acc_read(cross[i][j][e]), 1.f / kSplitScale, acc_read(acc[i][j][e]));
  };
  // What the main loop leaves to do where a row or a column of the tile is outside the window (split_f32.h): columns are scaled back, and
  // rows of A, like columns with an infinity, are formed again with the fp32 instruction, from operands in fp32: the 16 x 16 blocks that
  // one crosses, of which its elements are taken.  Every other element keeps its bits, whatever shares its tile.  Each wavefront for
  // itself, straight from global memory: seldom, and in few registers.  us per launch, nothing / one row / every 32nd row of A / every
  // 32nd column outside, and all of it on the fp32 tiles: 128 x 2304 x 768 8 / 19 / 19 / 8, 9.6; 2000 x 3072 x 768 31 / 64 / 103 / 32, 72;
  // 10240 x 768 x 3072 144 / 242 / 554 / 147, 332.
  constexpr int TOPS = 256, FLAGS = TOPS + KG * BM * 4, EXACT = FLAGS + BN * 4;  // behind the wavefronts' answers
  static_assert(EXACT + KG * BM * BN * 4 <= KG * split_lds_bytes<BM, BN, SB>(), "a tile in fp32 beside what is known about its rows");
  float* const tops = reinterpret_cast<float*>(lds + TOPS);             // the largest value of each row in each group's part of K
  int* const column_flags = reinterpret_cast<int*>(lds + FLAGS);       // of the columns: split_f32.h
  auto fp32_blocks = [&](auto swap_tag) __attribute__((always_inline)) {
    constexpr bool SWAP = decltype(swap_tag)::value;
    constexpr int PER_ROW = SWAP ? 1 : 4, PER_COL = SWAP ? 4 : 1;  // a lane holds a row's four columns of a block, or the other way round
    static_assert(RB * PER_ROW <= 32, "a bit per row of a lane");
    floatx4* const exact_at = reinterpret_cast<floatx4*>(lds + EXACT) + (group * NW + wave) * (RB * CB * kWave) + lane;
    auto row_outside = [&](int i, int e) __attribute__((always_inline)) {
      const int row = wm0 + i * 16 + (SWAP ? lrow : lgrp * 4 + e);
      float top = tops[row];
#pragma unroll
      for (int o = 1; o < KG; ++o) top = fmaxf(top, tops[o * BM + row]);
      return split_outside(top);
    };
    auto column_flag = [&](int j, int e) __attribute__((always_inline)) { return column_flags[wn0 + j * 16 + (SWAP ? lgrp * 4 + e : lrow)]; };
    uint32_t row_bits = 0, row_blocks = 0, col_blocks = 0;  // of this lane; of the wavefront's blocks
#pragma unroll
    for (int q = 0; q < RB * PER_ROW; ++q) {
      const bool out = row_outside(q / PER_ROW, q % PER_ROW);
      row_bits |= (uint32_t)out << q;
      row_blocks |= (uint32_t)(__ballot(out) != 0) << (q / PER_ROW);
    }
#pragma unroll
    for (int q = 0; q < CB * PER_COL; ++q) {
      const bool out = column_flag(q / PER_COL, q % PER_COL) == kSplitOutside;
      col_blocks |= (uint32_t)(__ballot(out) != 0) << (q / PER_COL);
    }
#pragma unroll 1
    for (int i = 0; i < RB; ++i) {
      const uint32_t blocks = (row_blocks >> i & 1) != 0 ? ~0u : col_blocks;
      if (blocks == 0) continue;
      floatx4 exact[CB];
#pragma unroll
      for (int j = 0; j < CB; ++j) exact[j] = floatx4{0.f, 0.f, 0.f, 0.f};
      const char* const a = g.a + k_lo + (size_t)min(m0 + wm0 + i * 16 + lrow, g.m - 1) * lda_bytes + lgrp * 16;
      const char* const b = g.b + k_lo + lgrp * 16;
#pragma unroll 1
      for (int at = 0; at < valid * kRowBytes; at += 64) {  // a lane's four values of K of sixteen
        const floatx4 fa = *reinterpret_cast<const floatx4*>(a + at);
        floatx4 fb[CB];
#pragma unroll
        for (int j = 0; j < CB; ++j) fb[j] = *reinterpret_cast<const floatx4*>(b + (uint32_t)min(n0 + wn0 + j * 16 + lrow, g.n - 1) * ldb_bytes + at);
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          if ((blocks >> j & 1) == 0) continue;
#pragma unroll
          for (int part = 0; part < 4; ++part)
            exact[j] = SWAP ? __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][part], fa[part], exact[j], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f32_16x16x4f32(fa[part], fb[j][part], exact[j], 0, 0, 0);
        }
      }
#pragma unroll
      for (int j = 0; j < CB; ++j) exact_at[(i * CB + j) * kWave] = exact[j];
    }
#pragma unroll
    for (int i = 0; i < RB; ++i) {
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const floatx4 exact = exact_at[(i * CB + j) * kWave];  // (its lane's own: nothing is waited for; unspecified where no element is taken)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int flag = column_flag(j, SWAP ? e : 0);
          const bool out = ((row_bits >> (SWAP ? i : i * 4 + e) & 1) != 0) | (flag == kSplitOutside);
          value[i][j][e] = out ? exact[e] : __builtin_ldexpf(value[i][j][e], -flag);
        }
      }
    }
  };
  auto k_loop = [&](auto swap_tag) __attribute__((always_inline)) {
    clear();
    static_for<2>([&](auto step_tag) __attribute__((always_inline)) {  // the first two steps
      constexpr int step = decltype(step_tag)::value;
      static_for<PARTS>([&](auto q_tag) __attribute__((always_inline)) {
        constexpr int q = decltype(q_tag)::value;
        split_part(template_int<q % 4>{}, template_int<q / 4>{}, raw[step][q / 4], step * A_STAGE, step + DA);
      });
    });
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(DA * PASSES + (SB - 3) * B_LOADS) : "memory");
    static_for<2 * HELD>([&](auto q_tag) __attribute__((always_inline)) { read_held(template_int<0>{}, q_tag, 0); });
    read_passing(template_int<0>{}, template_int<0>{}, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#pragma unroll
    for (int q = 0; q < 2 * HELD; ++q) landed(held[0][q / 2][q % 2]);
    landed(passing[0][0]);
    landed(passing[0][1]);
    Stages st{0, A_STAGE, 2 * A_STAGE, 0, B_STAGE, (SB - 1) * B_STAGE};
    auto turn = [&](auto turn_tag, int s) __attribute__((always_inline)) {
      k_step(swap_tag, turn_tag, s, st);
      const int after = st.b1 == (SB - 1) * B_STAGE ? 0 : st.b1 + B_STAGE;
      st = Stages{st.a1, st.a2, st.a0, st.b1, after, st.b0};
      return s + 1 < ksteps;
    };
    if constexpr (DA == 2) {
#pragma unroll 1
      for (int s = 0; turn(template_int<0>{}, s) && turn(template_int<1>{}, s + 1); s += 2) {}
    } else {
#pragma unroll 1
      for (int s = 0; turn(template_int<0>{}, s) && turn(template_int<1>{}, s + 1) && turn(template_int<2>{}, s + 2) && turn(template_int<3>{}, s + 3); s += 4) {}
    }
    asm volatile("s_nop 15\n\ts_nop 15");
    bool outside = column_flag_here != 0;
    // (every stage has been read, and the loads past the last step are waited for: the front of LDS holds the wavefronts' answers
    // and what they are about)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const float top = group_max<8>(largest[p]);
      outside = outside || split_outside(top);
      if (kq == 0) tops[group * BM + p * ROWS + sub] = top;
    }
    if (group == 0 && tid < BN) column_flags[tid] = column_flag_here;
    int* const answers = reinterpret_cast<int*>(lds);
    const bool any = __ballot(outside) != 0;
    if (lane == 0) answers[group * NW + wave] = any;
    __syncthreads();
    int again = 0;
#pragma unroll
    for (int w = 0; w < KG * NW; ++w) again |= answers[w];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j) value[i][j] = floatx4{sum(i, j, 0), sum(i, j, 1), sum(i, j, 2), sum(i, j, 3)};
    if (__builtin_amdgcn_readfirstlane(again) != 0) fp32_blocks(swap_tag);
  };

  // the groups' sums meet: those of the others pass through LDS, lane by lane
  floatx4 other[KG > 1 ? RB : 1][KG > 1 ? CB : 1];
  auto read = [&](int i, int j, int e) __attribute__((always_inline)) {
    if constexpr (KG > 1) return value[i][j][e] + other[i][j][e];
    else return value[i][j][e];
  };
  auto meet = [&]() __attribute__((always_inline)) {
    if constexpr (KG > 1) {
      floatx4* const at = reinterpret_cast<floatx4*>(lds) + wave * (RB * CB * kWave) + lane;
      constexpr int PER_GROUP = NW * RB * CB * kWave;
      __syncthreads();  // (the wavefronts' answers have been read)
      if (group != 0) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int j = 0; j < CB; ++j) at[(group - 1) * PER_GROUP + (i * CB + j) * kWave] = value[i][j];
      }
      __syncthreads();
      if (group != 0) return false;
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          other[i][j] = at[(i * CB + j) * kWave];
#pragma unroll
          for (int o = 1; o < KG - 1; ++o) other[i][j] += at[o * PER_GROUP + (i * CB + j) * kWave];
        }
    }
    return true;
  };
  auto unit_chunk = [&](int p) __attribute__((always_inline)) { return 2 * (2 * p + (lgrp & 1)) + (lgrp >> 1); };
  bool swap = true;
  if constexpr (HasColumnPass<Epi>::value) swap = !(epi.column_pass() && n0 + wn0 >= epi.first_column_of_pass());
  if (swap) {
    float amax = 0.f;
    ColumnQuads<float, CB, false> quads;
    quads.load(epi.bias_ptr(), nullptr, n0 + wn0, g.n, lgrp, g.b);
    k_loop(std::true_type{});
    if (!meet()) return;
    store_rows32<RB, CB>(g, epi, quads, z_epi, m0 + wm0, n0 + wn0, lrow, lgrp, amax, default_stores<Epi>(BM) == Stores::kAsk && g.write_through, read);
  } else {
    if constexpr (HasColumnPass<Epi>::value) {
      float bj[CB];
      load_bias_columns_stride<CB, 16>(epi, n0 + wn0 + lrow, g.n, bj);
      k_loop(std::false_type{});
      if (!meet()) return;
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const int n = n0 + wn0 + j * 16 + lrow;
        if constexpr (RB % 2 == 0) {
#pragma unroll
          for (int p = 0; p < RB / 2; ++p) {
            float out[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float a = read(2 * p, j, e), b = read(2 * p + 1, j, e);
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
            for (int e = 0; e < 4; ++e) out[e] = read(i, j, e) + bj[j];
            const int m = m0 + wm0 + i * 16 + lgrp * 4;
            if (m < g.m && n < g.n) epi.store_col4(m, g.m, n, out);
          }
        }
      }
    }
  }
}

template <int BM, int BN, int WM, int WN, int KG, int DA, int SB, typename Epi>
int launch_split(GemmArgs g, const Epi& epi, int slices, hipStream_t s) {
  constexpr int LDS = KG * split_lds_bytes<BM, BN, SB>();
  static_assert(LDS <= kLdsPerCu, "tile does not fit in LDS");
  if (describe_only("dma", KG * WM * WN, BM, BN, slices)) return 0;
  g.tiles_m = (g.m + BM - 1) / BM;
  g.tiles_n = (g.n + BN - 1) / BN;
  g.slices = slices;
  const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n * slices;
  TTMI_REQUIRE(tiles < (1ll << 30), "GEMM grid too large");
  const unsigned grid_x = tiles >= kXcdRemapMinTiles ? (unsigned)(ceil_div(tiles, kNumXcd) * kNumXcd) : (unsigned)tiles;
  auto kern = gemm_split_kernel<BM, BN, WM, WN, KG, DA, SB, Epi>;
  if (LDS > 64 * 1024) {
    const int rc = allow_large_lds(reinterpret_cast<const void*>(kern), LDS);
    if (rc != 0) return rc;
  }
  g.write_through = stores_through<Epi>(g);
  hipLaunchKernelGGL(kern, dim3(grid_x), dim3(KG * WM * WN * kWave), LDS, s, g, epi);
  return launch_status("gemm_split_kernel");
}

}  // namespace ttmi
