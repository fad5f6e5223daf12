// A stack of encoder layers over up to 16 rows as ONE launch (16-bit types).
//
// With a handful of rows a layer is six dependent launches of 3.7 to 5.3 us each, of which nothing but the change from one to the next
// is long: launch, first operands, drain.  Here workgroups of sixteen wavefronts stay, and what one step of the chain leaves for the next goes
// through memory (chain.h).  The weights and parameters of an item are requested in front of its rows and arrive while it waits for them.
//
// Steps of a layer, and items (16 or 32 columns each) of a step:
//   0  LayerNorm of the previous layer's rows, QKV product                     3H/32 items
//   1  attention of all heads (a wavefront each), output projection, residual  H/16
//   2  LayerNorm, FFN1, GELU                                                   F/32
//   3  FFN2, residual                                                          H/16
// and the last LayerNorm.  Rows in front of a LayerNorm travel in fp32; each item normalises all of them for itself (the attention is
// likewise computed by every item of step 1): a few hundred cycles instead of one more exchange.
//
// us per forward, layer by layer / as one launch: fp16 base 1 x 1 token 280 / 156, 1 x 8 291 / 175, 1 x 10 297 / 188, 4 x 4 308 / 198; bf16 large 1 x 8
// 661 / 420, 1 x 16 675 / 485 (the exchange memory filled by a launch of its own in front: 3 to 5 more; every wavefront asking for rows and parameters,
// also those that have no row: large 461 and 511, base level).  What bounds a step of 3.2 to 4 us: the exchange 1.0 to 1.5 (a store to memory, and a load
// that finds it), the LayerNorm of 16 rows on every CU 0.5 to 1.2 (vector instructions: 16 rows are four a SIMD), the product and the sum over the
// wavefronts 0.6.
// Measured and no better: 16 columns an item (240 workgroups instead of 144) level; Q, K, V and the intermediate rows row by row instead
// of in the order of the registers 10 rows 218 / 183, 16 251 / 194 (the launch alone).
//
// Progress does not depend on how many of the workgroups are resident.  Items are pure functions of the step before, and who executes an
// item a second time writes the same bits.  A workgroup that has waited `patience` polls in vain (others hold the CUs, or the
// grid is smaller than the items) executes the steps that it misses by itself, from the last one whose inputs it has seen, and
// goes on; workgroups that start late find everything written.  That ends whatever an item waits for (chain_walk.h): where nobody writes it, in an error.
// Beside a busy stream that is worth more than it costs: one launch gets its CUs once where 76 get them each time anew.  us per forward of base, 1 x 10
// tokens, layer by layer / as one launch, median beside torch's fp16 products on another stream of 1024^3: 330 / 220, 2048^3: 477 / 232, 4096^3: 5640 / 234,
// 8192^3: 10200 / 1405 (one in thirty there takes 16.9 ms: it computes alone); a decoder step of 8 sequences, 40 keys 288 / 212, 390 / 255, 4880 / 1965, 10060 / 9890.
#include <mutex>
#include <set>

#include "chain.h"

namespace ttmi {
namespace {

constexpr int kWaves = kChainWaves, kThreads = kChainThreads, kRows = kChainRows, kColumns = kChainColumns, kPitch = kChainPitch;
constexpr int kMostLayers = 24;
constexpr int kLdsMost = 80 * 1024;

struct ChainLayer {
  const void *qkv_w, *qkv_b, *out_w, *out_b, *gamma1, *beta1, *ffn1_w, *ffn1_b, *ffn2_w, *ffn2_b, *gamma2, *beta2;
};
// Where a layer's results lie in its part of the exchange memory.
struct Places {
  uint32_t qk, vt, x0, sum1, mid, x1, sum2, end;
};
struct ChainArgs {
  ChainLayer layer[kMostLayers];
  const void* input;     // [rows, hidden]
  const float* input32;  // the same unrounded, or null
  const float* mask;     // [rows], additive, or null
  void* out;
  float* out32;
  char *exchange, *other;  // the part of this launch, the part to fill (recorded: the first of the two)
  uint32_t layer_bytes;  // of the exchange memory
  Places at;
  int layers, rows, seq, heads, hidden, ffn, patience;
  float eps, scale_log2e, inv_scale;
  int* error;
  uint32_t* count;  // of recorded launches; last, so that eps stays in the line of 64 bytes that every workgroup has read by then (10 rows 188.2 / 190.4 us)
};

inline uint32_t up256(uint32_t n) { return (n + 255u) & ~255u; }
inline Places places(int rows, int hidden, int ffn, int residual_size) {
  Places p;
  const uint32_t r = (uint32_t)rows, h = (uint32_t)hidden;
  p.qk = 0;                                                  // Q, then K: [H / 8, kRows, 8]
  p.vt = p.qk + 2 * h * kRows * 2;                           // V: [H, kRows]
  p.x0 = p.vt + h * kRows * 2;                               // [H / 16, rows, 16] of the residual's type
  p.sum1 = p.x0 + up256(r * h * (uint32_t)residual_size);    // [rows, H] fp32
  p.mid = p.sum1 + up256(r * h * 4);                         // [F / 64, 2, 4, kRows, 8], see fragment_offset
  p.x1 = p.mid + (uint32_t)ffn * kRows * 2;
  p.sum2 = p.x1 + up256(r * h * (uint32_t)residual_size);
  p.end = p.sum2 + up256(r * h * 4);
  return p;
}

// Q, K and V lie as the wavefronts that read them hold them in registers (as fragment_offset does).  In bytes, of an even column (a pair of rows of V):
__device__ __forceinline__ uint32_t q_offset(int row, int col) { return (uint32_t)(((col >> 3) * kRows + row) * 8 + (col & 7)) * 2; }
__device__ __forceinline__ uint32_t v_offset(int row, int col) { return (uint32_t)(col * kRows + row) * 2; }

// Whether one of the values is an infinity or a NaN.
template <typename T, typename Words>
__device__ __forceinline__ bool unbounded(const Words& x) {
  constexpr uint32_t exponent = std::is_same<T, f16>::value ? 0x7c00u : 0x7f80u;
  bool any = false;
#pragma unroll
  for (uint32_t w = 0; w < sizeof(Words) / 4; ++w) any = any | ((x[w] & exponent) == exponent) | ((x[w] >> 16 & exponent) == exponent);
  return any;
}
// A pair of values of V, zero where its keys are not in [from, to).
__device__ __forceinline__ uint32_t keys_within(uint32_t pair, int key, int from, int to) {
  return (key >= from && key < to ? pair & 0xffffu : 0u) | (key + 1 >= from && key + 1 < to ? pair & 0xffff0000u : 0u);
}

// LDS: rows of the A operand (or, in step 1, the heads' contexts), then the partial tiles.
constexpr int kContextPitch = (kD + 8) * 2;
__host__ __device__ inline int rows_bytes(int hidden) {
  const int rows = kRows * chain_row_pitch(hidden), contexts = kWaves * kRows * kContextPitch;
  return rows > contexts ? rows : contexts;
}
__host__ __device__ inline int lds_bytes(int hidden) { return rows_bytes(hidden) + kWaves * kRows * kPitch * 4; }

// TURNS: turns of 256 columns that a row of the hidden state takes at most; PIECES: 128-byte pieces of a row of FFN2's weight
// that a wavefront takes at most (of the other weights it is one).  RECORDED: the launch finds its part of the exchange memory by itself.
template <typename T, int TURNS, int PIECES, bool RECORDED>
__global__ __launch_bounds__(kThreads) void encoder_chain_kernel(const ChainArgs) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr bool WIDE = std::is_same<T, bf16>::value;  // the residual stays in fp32
  constexpr int RS = WIDE ? 4 : 2;
  extern __shared__ __align__(16) char smem[];
  __shared__ int missing;
  __shared__ ChainLayer layers[kMostLayers];  // (where the arguments lie a first read takes as long as an exchange)
  // The arguments are read, and what depends on the lane is computed, where an item needs it: kept over the loop they are a hundred registers.
  typedef const __attribute__((address_space(4))) ChainArgs Arguments;
  auto arguments = []() __attribute__((always_inline)) {
    uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return reinterpret_cast<Arguments*>(p);
  };
  const int G = gridDim.x, me = blockIdx.x;
  auto items = [&](int step) __attribute__((always_inline)) {
    const Arguments& a = *arguments();
    return step == 4 * a.layers ? 1 : (step & 3) == 0 ? 3 * a.hidden / (16 * kColumns) : (step & 3) == 2 ? a.ffn / (16 * kColumns) : a.hidden / 16;
  };
  // The first item of a step for this workgroup.  Steps 1 and 3 are the last workgroups': others than those of steps 0 and 2 where the
  // grid has as many, so that each has a step's time for its weights to arrive.
  auto first_item = [&](int step) __attribute__((always_inline)) {
    const int first = (step & 1) == 1 ? max(G - arguments()->hidden / 16, 0) : 0;
    return me >= first ? me - first : me - first + G;
  };
  const int last_step = 4 * arguments()->layers;

  __shared__ uint32_t launches;  // recorded: so far
  uint32_t shift = 0;
  if constexpr (!RECORDED) fill_unwritten(arguments()->other, (uint32_t)arguments()->layers * arguments()->layer_bytes, me, G);
  auto leave = [&]() __attribute__((always_inline)) {
    if constexpr (RECORDED) {
      const Arguments& a = *arguments();
      const uint32_t part = (uint32_t)a.layers * a.layer_bytes;
      const int fillers = min(G, items(0));  // (they know the part)
      if (me < fillers) fill_unwritten(a.exchange + (part - shift), part, me, fillers);
      count_launch(a.count, me, G);
    }
  };
  ChainWalk walk;
  walk.item = first_item(0) - G;
  walk.forward(G, last_step + 1, items, first_item);
  if (walk.step > last_step) {
    leave();
    return;
  }
  int seen = 0;  // the last step whose inputs the workgroup has seen
  if (threadIdx.x == 0) {
    missing = 0;
    if (RECORDED) launches = launches_so_far(arguments()->count);
  }
  constexpr int WORDS = sizeof(ChainLayer) / 8;
  if ((int)threadIdx.x < arguments()->layers * WORDS)
    reinterpret_cast<uint64_t*>(layers)[threadIdx.x] = reinterpret_cast<const __attribute__((address_space(4))) uint64_t*>(&arguments()->layer)[threadIdx.x];
  __syncthreads();
  if constexpr (RECORDED) shift = part_offset(__builtin_amdgcn_readfirstlane(launches), (uint32_t)arguments()->layers * arguments()->layer_bytes);
  auto uniform = [](const void* const& p) __attribute__((always_inline)) -> const void* {
    const uint64_t x = reinterpret_cast<const uint64_t&>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x), hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));  // (they return int)
    return reinterpret_cast<const void*>((uint64_t)hi << 32 | lo);
  };

  for (;;) {
    const Arguments& a = *arguments();
    const int step = walk.step, item = walk.item;
    const auto& at = a.at;
    const int H = a.hidden, F = a.ffn, rows = a.rows, patience = a.patience;
    const int pitch = chain_row_pitch(H);
    float* const part = reinterpret_cast<float*>(smem + rows_bytes(H));
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lrow = lane & 15, lgrp = lane >> 4;
    const int l = step >> 2, ph = step & 3;
    const uint32_t base = (uint32_t)l * a.layer_bytes + shift;
    const __amdgpu_buffer_rsrc_t mem = __builtin_amdgcn_make_buffer_rsrc(a.exchange, 0, (RECORDED ? 2 : 1) * a.layers * a.layer_bytes, 0x00020000);
    auto load4 = [&](uint32_t offset) __attribute__((always_inline)) { return (u32x4)__builtin_amdgcn_raw_buffer_load_b128(mem, offset, 0, kThroughMemory); };
    auto load2 = [&](uint32_t offset) __attribute__((always_inline)) { return (u32x2)__builtin_amdgcn_raw_buffer_load_b64(mem, offset, 0, kThroughMemory); };
    auto load1 = [&](uint32_t offset) __attribute__((always_inline)) { return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(mem, offset, 0, kThroughMemory); };
    auto store1 = [&](uint32_t offset, uint32_t x) __attribute__((always_inline)) { __builtin_amdgcn_raw_buffer_store_b32(storable(x), mem, offset, 0, kThroughMemory); };
    // Asks again until there is no unwritten word; `ask` returns the largest of those it has loaded.
    bool late = false;
    auto await = [&](auto&& ask) __attribute__((always_inline)) {
      for (int polls = 0;; ++polls) {
        asm volatile("" ::: "memory");
        if (__builtin_amdgcn_ballot_w64(ask() == kUnwritten) == 0) break;
        if (polls >= patience) {
          late = true;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    };

    // What the item needs besides its rows is requested in front of them: it arrives while the item waits.
    const ChainLayer& y = layers[min(l, a.layers - 1)];
    const int K = ph == 3 ? F : H, N = ph == 0 ? 3 * H : ph == 2 ? F : H;
    const __amdgpu_buffer_rsrc_t weights =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(uniform(ph == 0 ? y.qkv_w : ph == 1 ? y.out_w : ph == 2 ? y.ffn1_w : y.ffn2_w)), 0, step == last_step ? 0 : N * K * 2, 0x00020000);
    const int n0 = item * (ph & 1 ? 16 : 16 * kColumns);
    const uint32_t w_row = (uint32_t)((n0 + lrow) * K + lgrp * 16) * 2;
    // The thread's part of the output: two columns of a row, or two rows of a column of V; 128 threads for 16 x 16 values.
    const int block = tid >> 7, at_tid = tid & 127;
    const bool stores = step != last_step && block < (ph & 1 ? 1 : kColumns), transposed = ph == 0 && n0 >= 2 * H;
    uint32_t bias = 0;
    if (stores) {
      const void* b = uniform(ph == 0 ? y.qkv_b : ph == 1 ? y.out_b : ph == 2 ? y.ffn1_b : y.ffn2_b);
      if (transposed) bias = static_cast<const uint16_t*>(b)[n0 + block * 16 + lrow];
      else bias = *reinterpret_cast<const uint32_t*>(static_cast<const T*>(b) + n0 + block * 16 + 2 * (tid & 7));
    }
    floatx4 acc[kColumns];
#pragma unroll
    for (int c = 0; c < kColumns; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
    float res0 = 0.f, res1 = 0.f;  // the residual of the thread's two columns (steps 1 and 3)
    const bool pairs_here = stores && (at_tid >> 3) < rows;

    if ((ph & 1) == 0) {  // (the last step among them)
      u32x4 wf[kColumns][2];
      // Beyond 768 columns (nearly) all wavefronts have a share: a branch instead of a choice of addresses, large 1 x 8 445 / 420, 1 x 16 509 / 485; with twelve
      // of sixteen base 1 x 10 187.9 / 189.5.
      constexpr bool BRANCH = TURNS > 3;
      if (!BRANCH || wave < H / 64) {
        const uint32_t piece = BRANCH || wave < H / 64 ? w_row + wave * 128 : kOutside;
#pragma unroll
        for (int c = 0; c < kColumns; ++c)
#pragma unroll
          for (int s = 0; s < 2; ++s)
            wf[c][s] = (u32x4)__builtin_amdgcn_raw_buffer_load_b128(weights, BRANCH || wave < H / 64 ? piece + (uint32_t)(c * 16 * H * 2 + s * 16) : kOutside, 0, 0);
      }
      if (step == 0) {
        if (wave < rows)
#pragma unroll
          for (int t = 0; t < TURNS; ++t) {
            const int col = t * 256 + lane * 4;
            if (col < H) *reinterpret_cast<u32x2*>(smem + wave * pitch + col * 2) = *reinterpret_cast<const u32x2*>(static_cast<const T*>(a.input) + wave * H + col);
          }
      } else if (wave < rows) {
        u32x2 gm[TURNS], bt[TURNS];
        {
          const void* gamma = uniform(ph == 2 ? y.gamma1 : layers[l - 1].gamma2);
          const void* beta = uniform(ph == 2 ? y.beta1 : layers[l - 1].beta2);
          const __amdgpu_buffer_rsrc_t g = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(gamma), 0, H * 2, 0x00020000);
          const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(beta), 0, H * 2, 0x00020000);
#pragma unroll
          for (int t = 0; t < TURNS; ++t) {
            gm[t] = (u32x2)__builtin_amdgcn_raw_buffer_load_b64(g, t * 512 + lane * 8, 0, 0);
            bt[t] = (u32x2)__builtin_amdgcn_raw_buffer_load_b64(b, t * 512 + lane * 8, 0, 0);
          }
        }
        // columns that do not exist are zeros
        const uint32_t from = ph == 2 ? base + at.sum1 : base - a.layer_bytes + at.sum2;
        const uint32_t keep = ph == 2 ? base + at.x1 : base + at.x0;
        u32x4 raw[TURNS];
        await([&]() __attribute__((always_inline)) {
          uint32_t m = 0;
#pragma unroll
          for (int t = 0; t < TURNS; ++t) {
            const int col = t * 256 + lane * 4;
            raw[t] = load4(col < H ? from + (uint32_t)(wave * H + col) * 4 : kOutside);
          }
#pragma unroll
          for (int t = 0; t < TURNS; ++t) m = largest(m, raw[t]);
          return m;
        });
        if (late) {
          missing = 1;
        } else {
          float x[TURNS][4], normed[TURNS][4];
#pragma unroll
          for (int t = 0; t < TURNS; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) x[t][e] = __builtin_bit_cast(float, (uint32_t)raw[t][e]);
          normalise_row<T, TURNS>(x, gm, bt, H, a.eps, normed);
#pragma unroll
          for (int t = 0; t < TURNS; ++t) {
            const int col = t * 256 + lane * 4;
            const float (&v)[4] = normed[t];
            const u32x2 r = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
            if (col >= H) continue;
            if (step == last_step) {
              *reinterpret_cast<u32x2*>(static_cast<T*>(a.out) + wave * H + col) = r;
              if (WIDE && a.out32 != nullptr) *reinterpret_cast<floatx4*>(a.out32 + wave * H + col) = floatx4{v[0], v[1], v[2], v[3]};
              continue;
            }
            *reinterpret_cast<u32x2*>(smem + wave * pitch + col * 2) = r;
            if (col / (16 * kColumns) == item) {
              const uint32_t to = keep + (uint32_t)(((col >> 4) * rows + wave) * 16 + (col & 15)) * RS;
              if constexpr (WIDE) {
#pragma unroll
                for (int e = 0; e < 4; ++e) store1(to + 4 * e, __builtin_bit_cast(uint32_t, v[e]));
              } else {
                store1(to, r[0]);
                store1(to + 4, r[1]);
              }
            }
          }
        }
      }
      __syncthreads();
      if (wave < H / 64) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const u32x4 x = *reinterpret_cast<const u32x4*>(smem + lrow * pitch + wave * 128 + lgrp * 32 + s * 16);
#pragma unroll
          for (int c = 0; c < kColumns; ++c) acc[c] = mma16<T>(x, wf[c][s], acc[c]);
        }
      }
    } else {
      // The residual, written a step before what the item waits for (the first layer's is the input).
      const bool from_input = step == 1;
      const int res_index = (tid >> 3) * H + item * 16 + 2 * (tid & 7);
      const uint32_t res_at = pairs_here && !from_input ? (ph == 1 ? base + at.x0 : base + at.x1) + (uint32_t)(item * rows * 16 + 2 * tid) * RS : kOutside;
      u32x2 res = {0u, 0u};
      auto ask_residual = [&]() __attribute__((always_inline)) {
        if constexpr (WIDE) res = load2(res_at);
        else res[0] = load1(res_at);
        return res;
      };
      if (ph == 1) {
        const bool has = wave < a.heads;
        u32x4 wf[2];
        const uint32_t piece = has ? w_row + wave * 128 : kOutside;
#pragma unroll
        for (int s = 0; s < 2; ++s) wf[s] = (u32x4)__builtin_amdgcn_raw_buffer_load_b128(weights, piece + s * 16, 0, 0);
        char* const ctx = smem + wave * (kRows * kContextPitch);
        // Scores transposed: lane = query, four keys a register quad, which is how the second product takes them if V^T comes in the same
        // order (its other four keys of eight are zeros).  A query sees the keys of its own sequence.
        u32x4 qf[2], kf[2];
        u32x2 vf[4];
        const uint32_t mask_bits = a.mask != nullptr ? load_mask(a.mask + min(lrow, rows - 1)) : 0u;
        const int first = lrow / a.seq * a.seq, last = first + a.seq;
        const bool has_row = has && lrow < rows;  // (the others are zeros)
        const uint32_t q_at = base + at.qk + q_offset(lrow, wave * kD + lgrp * 8), k_at = q_at + (uint32_t)H * 32;
        const uint32_t v_at = base + at.vt + v_offset(4 * lgrp, wave * kD + lrow);
        await([&]() __attribute__((always_inline)) {
          const u32x2 r = ask_residual();
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            qf[s] = load4(has_row ? q_at + s * 1024 : kOutside);
            kf[s] = load4(has_row ? k_at + s * 1024 : kOutside);
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) vf[t] = load2(has ? v_at + t * 512 : kOutside);
          uint32_t m = largest(0u, r);
#pragma unroll
          for (int s = 0; s < 2; ++s) m = largest(largest(m, qf[s]), kf[s]);
#pragma unroll
          for (int t = 0; t < 4; ++t) m = largest(m, vf[t]);
          return m;
        });
        if (has) {
          floatx4 st = {0.f, 0.f, 0.f, 0.f};
          const float mk = lrow < rows ? mask_in_scores(mask_bits, a.inv_scale) : -__builtin_inff();
          st = __builtin_amdgcn_mfma_f32_16x16x4f32(lgrp == 0 ? mk : 0.f, 1.f, st, 0, 0, 0);
#pragma unroll
          for (int s = 0; s < 2; ++s) st = mma16<T>(kf[s], qf[s], st);
#pragma unroll
          for (int e = 0; e < 4; ++e) st[e] = 4 * lgrp + e >= first && 4 * lgrp + e < last ? st[e] : -__builtin_inff();
          float mx = fmaxf(fmaxf(st[0], st[1]), fmaxf(st[2], st[3]));
          const LanePair rows2 = swap_rows(mx);
          mx = fmaxf(rows2.a, rows2.b);
          const LanePair halves = swap_halves(mx);
          const float m_run = fmaxf(-kFarthestScore, fmaxf(halves.a, halves.b));
          const float neg_m = relative_scores<4>(st, m_run, a.scale_log2e);
          u32x4 pf = {0u, 0u, 0u, 0u};
          float sum = 0.f;
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            pf[w] = pack2<T>(__builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * w], a.scale_log2e, neg_m)),
                             __builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * w + 1], a.scale_log2e, neg_m)));
            sum = add_pair<T>(pf[w], sum);
          }
          const LanePair sum2 = swap_rows(sum);
          sum = sum2.a + sum2.b;
          const LanePair sum4 = swap_halves(sum);
          const float inv = 1.0f / (sum4.a + sum4.b);
          // (0 * infinity: where V is not finite, one sequence at a time)
          const bool apart = a.seq < rows && __builtin_amdgcn_ballot_w64(unbounded<T>(vf[0]) | unbounded<T>(vf[1]) | unbounded<T>(vf[2]) | unbounded<T>(vf[3])) != 0;
#pragma unroll 1
          for (int from = 0; from < (apart ? rows : 1); from += a.seq) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              u32x2 v = vf[t];
              if (apart)
#pragma unroll
                for (int w = 0; w < 2; ++w) v[w] = keys_within(v[w], 4 * lgrp + 2 * w, from, from + a.seq);
              const floatx4 ot = mma16<T>(u32x4{v[0], v[1], 0u, 0u}, pf, floatx4{0.f, 0.f, 0.f, 0.f});
              if (!apart || first == from)
                *reinterpret_cast<u32x2*>(ctx + lrow * kContextPitch + (t * 16 + 4 * lgrp) * 2) =
                    u32x2{pack2<T>(ot[0] * inv, ot[1] * inv), pack2<T>(ot[2] * inv, ot[3] * inv)};
            }
          }
#pragma unroll
          for (int s = 0; s < 2; ++s) acc[0] = mma16<T>(*reinterpret_cast<const u32x4*>(ctx + lrow * kContextPitch + lgrp * 32 + s * 16), wf[s], acc[0]);
        }
      } else {
        const int share = (F / 64 + kWaves - 1) / kWaves, first = wave * share, mine = min(F / 64 - first, share);
        const int there = lrow < rows ? mine : 0;
        const uint32_t row_at = base + at.mid + fragment_offset<T>(lrow, first * 64 + lgrp * 16);
        u32x4 wf[2 * PIECES], af[2 * PIECES];
#pragma unroll
        for (int p = 0; p < 2 * PIECES; ++p)
          wf[p] = (u32x4)__builtin_amdgcn_raw_buffer_load_b128(weights, p / 2 < mine ? w_row + (first + p / 2) * 128 + (p & 1) * 16 : kOutside, 0, 0);
        await([&]() __attribute__((always_inline)) {
          const u32x2 r = ask_residual();
#pragma unroll
          for (int p = 0; p < 2 * PIECES; ++p) af[p] = load4(p / 2 < there ? row_at + p * (kRows * 64) : kOutside);
          uint32_t m = largest(0u, r);
#pragma unroll
          for (int p = 0; p < 2 * PIECES; ++p) m = largest(m, af[p]);
          return m;
        });
#pragma unroll
        for (int p = 0; p < 2 * PIECES; ++p) acc[0] = mma16<T>(af[p], wf[p], acc[0]);
      }
      if (late) missing = 1;
      if (from_input && pairs_here) {
        if (WIDE && a.input32 != nullptr) res = *reinterpret_cast<const u32x2*>(a.input32 + res_index);
        else res[0] = *reinterpret_cast<const uint32_t*>(static_cast<const T*>(a.input) + res_index);
      }
      if (WIDE && (!from_input || a.input32 != nullptr)) {
        res0 = __builtin_bit_cast(float, (uint32_t)res[0]);
        res1 = __builtin_bit_cast(float, (uint32_t)res[1]);
      } else {
        res0 = low<T>(res[0]);
        res1 = high<T>(res[0]);
      }
    }

#pragma unroll
    for (int c = 0; c < kColumns; ++c)
      if (c == 0 || (ph & 1) == 0)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[(wave * kRows + lgrp * 4 + e) * kPitch + c * 16 + lrow] = acc[c][e];
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(missing) != 0) {  // set in front of the barrier: the same for all
      __syncthreads();
      if (tid == 0) missing = 0;
      if (!walk.late(seen)) {  // (not reached while every item's inputs are some item's outputs)
        if (tid == 0 && a.error != nullptr) *a.error = kRowsNeverCame;
        leave();
        return;
      }
      __syncthreads();
      continue;
    }

    if (stores) {
      if (transposed) {  // V: two rows of a column
        const int r = 2 * (at_tid >> 4);
        const floatx2 v = sum_parts(part, r, block * 16 + lrow, kPitch);
        const float b = low<T>(bias);
        const float v0 = r < rows ? v[0] + b : 0.f, v1 = r + 1 < rows ? v[1] + b : 0.f;
        store1(base + at.vt + v_offset(r, n0 - 2 * H + block * 16 + lrow), pack2<T>(v0, v1));
      } else if (pairs_here) {
        const int r = at_tid >> 3, c = block * 16 + 2 * (tid & 7);
        const floatx2 v = sum_parts(part, r, c, 1);
        const float v0 = v[0] + low<T>(bias), v1 = v[1] + high<T>(bias);
        if (ph == 0) {
          store1(base + at.qk + q_offset(r, n0 + c), pack2<T>(v0, v1));
        } else if (ph == 2) {
          store1(base + at.mid + fragment_offset<T>(r, n0 + c), pack2<T>(gelu_tanh(v0), gelu_tanh(v1)));
        } else {
          const uint32_t to = base + (ph == 1 ? at.sum1 : at.sum2) + (uint32_t)(r * H + n0 + c) * 4;
          store1(to, __builtin_bit_cast(uint32_t, v0 + res0));
          store1(to + 4, __builtin_bit_cast(uint32_t, v1 + res1));
        }
      }
    }
    if (!walk.solo()) seen = step;
    walk.executed(G, last_step + 1, items, first_item);
    if (walk.step > last_step) {
      leave();
      return;
    }
    __syncthreads();  // the rows and partial tiles have been read
  }
#endif
}

int64_t workspace_bytes(int64_t layers, int64_t rows, int64_t heads, int64_t hidden, int64_t ffn, int dtype) {
  // ffn >= hidden: the items of step 2 are those that write x1, each the columns of its own number, which has to reach all of them.
  const bool takes = (dtype == TTMI_F16 || dtype == TTMI_BF16) && layers >= 1 && layers <= kMostLayers && rows >= 1 && rows <= kRows && heads >= 4 &&
                     heads <= kWaves && hidden == heads * kD && ffn >= hidden && ffn % 64 == 0 && ffn <= kWaves * 4 * 64;
  if (!takes) return 0;
  return exchange_bytes(layers * (int64_t)places(kRows, (int)hidden, (int)ffn, dtype == TTMI_BF16 ? 4 : 2).end);  // (of all rows: calls of any number of them take turns)
}

}  // namespace
}  // namespace ttmi

using namespace ttmi;

extern "C" {

int ttmi_encoder_chain_workspace(int64_t layers, int64_t rows, int64_t heads, int64_t hidden, int64_t ffn, int dtype, int64_t* bytes) {
  TTMI_REQUIRE(bytes != nullptr, "null result");
  *bytes = workspace_bytes(layers, rows, heads, hidden, ffn, dtype);
  return 0;
}

int ttmi_encoder_chain(const void* const* weights, const void* input, const float* input32, const float* mask, void* out, float* out32,
                       void* exchange, int turn, int64_t layers, int64_t batch, int64_t seq, int64_t heads, int64_t hidden, int64_t ffn, float eps, int dtype,
                       int workgroups, int patience, void* stream) {
  TTMI_REQUIRE(weights && input && out && exchange, "null tensor");
  TTMI_REQUIRE(batch > 0 && seq > 0 && batch <= kRows && seq <= kRows && workgroups >= 0 && workgroups <= kChainMostWorkgroups && patience >= 0, "bad shape");
  const int64_t rows = batch * seq, bytes = workspace_bytes(layers, rows, heads, hidden, ffn, dtype);
  TTMI_REQUIRE(bytes > 0, "this stack of layers is not run as one launch");
  ChainArgs a{};
  uintptr_t bits = reinterpret_cast<uintptr_t>(input) | reinterpret_cast<uintptr_t>(input32) | reinterpret_cast<uintptr_t>(out) |
                   reinterpret_cast<uintptr_t>(out32) | reinterpret_cast<uintptr_t>(exchange);
  for (int64_t l = 0; l < layers; ++l) {
    const void* const* w = weights + l * 12;
    for (int i = 0; i < 12; ++i) {
      TTMI_REQUIRE(w[i] != nullptr, "null weight");
      bits |= reinterpret_cast<uintptr_t>(w[i]);
    }
    a.layer[l] = {w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], w[9], w[10], w[11]};
  }
  TTMI_REQUIRE((bits & 15) == 0, "tensors must be 16-byte aligned");
  const int64_t values = rows * hidden;
  TTMI_REQUIRE(results_apart({{out, values * 2}, {out32, values * 4}}, {{input, values * 2}, {input32, values * 4}, {mask, rows * 4}}),
               "out and out32 must share no memory with input, input32, mask or each other");
  const int cus = compute_units();
  a.input = input, a.input32 = input32, a.mask = mask, a.out = out, a.out32 = out32;
  a.layer_bytes = (uint32_t)(part_of_exchange(bytes) / layers);
  a.at = places(kRows, (int)hidden, (int)ffn, dtype == TTMI_BF16 ? 4 : 2);
  a.layers = (int)layers, a.rows = (int)rows, a.seq = (int)seq, a.heads = (int)heads, a.hidden = (int)hidden, a.ffn = (int)ffn;
  a.patience = patience > 0 ? patience : kChainPatience;
  a.eps = eps, a.scale_log2e = 0.125f * 1.4426950408889634f, a.inv_scale = 8.0f, a.error = async_error_flag();
  hipStream_t s = (hipStream_t)stream;
  Turn t;
  const int rc = take_turn(exchange, part_of_exchange(bytes), turn, &t);
  if (rc != 0) return rc;
  a.exchange = t.mine, a.other = t.other, a.count = t.count;
  const int64_t widest = std::max(3 * hidden, ffn) / (16 * kColumns) + hidden / 16;
  const unsigned grid = workgroups > 0 ? (unsigned)workgroups : (unsigned)std::min<int64_t>(widest, cus);
  const int lds = lds_bytes((int)hidden);
  // more than 64 KB of dynamic LDS: the limit is raised once per kernel and device
  auto launch = [&](auto kernel) -> int {
    static std::mutex mu;
    static std::set<int> done;
    int dev = 0;
    TTMI_HIP(hipGetDevice(&dev));
    {
      std::lock_guard<std::mutex> lock(mu);
      if (done.count(dev) == 0) {
        TTMI_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMost));
        done.insert(dev);
      }
    }
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), lds, s, a);
    return launch_status("encoder_chain_kernel");
  };
  auto sized = [&](auto turns, auto pieces) -> int {
    constexpr int TURNS = decltype(turns)::value, PIECES = decltype(pieces)::value;
    if (t.count != nullptr) return dtype == TTMI_F16 ? launch(encoder_chain_kernel<f16, TURNS, PIECES, true>) : launch(encoder_chain_kernel<bf16, TURNS, PIECES, true>);
    return dtype == TTMI_F16 ? launch(encoder_chain_kernel<f16, TURNS, PIECES, false>) : launch(encoder_chain_kernel<bf16, TURNS, PIECES, false>);
  };
  if (hidden <= 3 * 256 && ffn <= kWaves * 3 * 64) return sized(std::integral_constant<int, 3>{}, std::integral_constant<int, 3>{});
  return sized(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
}

}  // extern "C"
