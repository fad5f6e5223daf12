// One decoder layer's attention (self attention over a growing cache, or attention over an encoder memory) or its feed-forward block as
// ONE launch: a token each of up to 16 sequences.
//
//   attention     0  LayerNorm, projection of Q (and K, V)                     N/32 items
//                 1  attention, a query each: W wavefronts a head              batch * heads * W / 16
//                 2  output projection, bias, residual                         H/16
//   feed-forward  0  LayerNorm, W1, ReLU                                       F/32
//                 1  W2, bias, residual                                        H/16
//
// Such a call was three launches (two), of 4.3 to 5.8 us each on the GPU and 3 on the host, of which nothing but the change from one to the next is
// long.  The exchange between the steps is that of chain.h, with as many workgroups as there are items, so that every one has requested its
// weights, or its keys and values, before it waits.  Progress does not depend on how many of them are resident, as in encoder_chain.hip: a workgroup that
// has waited in vain executes all items of the steps in front of its own.
//
// us a step of six layers of base (48 launches before, 18 now), by sequences and keys of the two attentions:
//              1 x 6, 20    4 x 201, 30    8 x 41, 100    16 x 41, 100    16 x 251, 256
//   fp16       255 / 151    250 / 169      240 / 179      250 / 213       308 / 262
//   fp32       286 / 229    357 / 257      328 / 278      356 / 317       454 / 395
// What is left of a launch of 8 to 12 in fp16: its start 0.5, arguments and first operands 1.5 to 2.5, LayerNorm and product 1, an exchange 0.7 to 1.3 each,
// attention 1 (3.5 with 64 keys a wavefront), its parts' sum and the last product 1.5.  A load of 16 bytes a lane takes the CU 16 cycles whatever it reads: what
// is asked for, in which order, and by how many wavefronts decides.  The weights first, the rows and parameters of the LayerNorm after them and
// together, nothing by wavefronts without a share: 8 sequences 188 / 178, 4 180 / 169, 1 159 / 151, 16 218 / 214; fp32 level to 1%.
// fp32 multiplies in fp32 (four instructions where 16 bits take one, the weights as they are, not their halves) and reads and exchanges twice the bytes.  Its
// error against 64 bits, rms after six layers, was 3.64 to 4.44e-7 with the split products and is 3.61 to 4.41e-7, that of the probabilities 11% less.
// Rows of 4096 products would not fit its registers: the feed-forward block goes to 3072 there (128 of them, no scratch).  Where it pays stands at
// FeedForwardRunsAsOneLaunch.
// Measured and no better: a wavefront normalises the columns that it multiplies, of all rows (parameters read once a CU, no rows in LDS, but 12 loads more
// a wavefront): fp32 8 sequences 274 / 302, fp16 8 188 / 196, 16 x 251 262 / 258; rows and parameters requested in front of the weights: fp32 274 / 281 to
// 286, 1 x 6 226 / 242 to 245.
// Measured and no better: the arguments held in registers (60 of the scalar ones spill) 11.4 / 12.5 a launch.
#include <mutex>
#include <set>

#include "chain.h"

namespace ttmi {
namespace {

constexpr int kWaves = kChainWaves, kThreads = kChainThreads, kRows = kChainRows, kColumns = kChainColumns, kPitch = kChainPitch;
constexpr int kMostHidden = 1024, kMostInner = 4096, kMostKeys = 512;
constexpr int kMostInner32 = 3072;  // fp32
constexpr int kTurns = kMostHidden / 256;
constexpr int kLdsMost = 112 * 1024;

enum Block { kFeedForward, kSelfAttention, kMemoryAttention };

struct DecoderArgs {
  const void *x, *gamma, *beta, *w_in, *b_in, *w_out, *b_out;  // x [rows, H]
  const void *k_past, *v_past;                                 // [rows, heads, past, 64]
  void *k_out, *v_out;                                         // [rows, heads, keys, 64], or null
  const float* mask;                                           // [rows, keys], or null
  void *probs, *out;                                           // [rows, heads, keys]; [rows, H]
  char *exchange, *other;                                      // the part of this launch, the part to fill (recorded: the first of the two)
  uint32_t* count;                                             // of recorded launches
  uint32_t bytes;                                              // of a part
  int rows, heads, hidden, width, inner;                       // width: of step 0's product; inner: of the last one's rows
  int past, keys, waves, patience;                             // waves: of a head
  float eps, scale;
  int* error;
};

// Exchange memory: step 0's rows ([rows, width]; in front of a product in fragment order), then the attention's in fragment order.
__host__ __device__ inline uint32_t context_at(int width, int element) { return (uint32_t)(kRows * width * element); }

// Eight columns of a row, and column e of them.
template <typename T>
struct Eight {
  u32x4 q[sizeof(T) / 2];
  __device__ __forceinline__ float at(int e) const {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, (uint32_t)q[e >> 2][e & 3]);
    else return e & 1 ? high<T>(q[0][e >> 1]) : low<T>(q[0][e >> 1]);
  }
};
template <typename T>
__device__ __forceinline__ float dot8(const Eight<T>& a, const Eight<T>& b) {
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) sum = __builtin_fmaf(a.at(e), b.at(e), sum);
  return sum;
}
// Lanes that differ by 1, 2 and 4, and by 8, 16 and 32.
template <typename Op>
__device__ __forceinline__ float over_pieces(float v, Op op) {
  v = op(v, dpp_move<0xB1>(v));
  v = op(v, dpp_move<0x4E>(v));
  return op(v, dpp_move<0x141>(v));  // (row_half_mirror: the quads agree)
}
template <typename Op>
__device__ __forceinline__ float over_keys(float v, Op op) {
  v = op(v, dpp_move<0x128>(v));  // row_ror:8
  const LanePair rows = swap_rows(v);
  v = op(rows.a, rows.b);
  const LanePair halves = swap_halves(v);
  return op(halves.a, halves.b);
}

// LOADS: keys of a lane of the attention; pieces of a wavefront of the feed-forward block's last product.  RECORDED: the launch finds its part of the
// exchange memory by itself.
template <typename T, Block BLOCK, int LOADS, bool RECORDED>
__global__ __launch_bounds__(kThreads) void decoder_chain_kernel(const DecoderArgs) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int STEPS = BLOCK == kFeedForward ? 2 : 3;
  constexpr int E = sizeof(T), PIECE = 128 / E;                                     // a piece: 128 bytes of a row
  constexpr int PIECES = kMostHidden / PIECE / kWaves;                              // of a row of H, that a wavefront takes at most
  constexpr int OUT_PIECES = BLOCK != kFeedForward ? PIECES : LOADS;          // of a row in front of the last product
  constexpr float kLog2e = 1.4426950408889634f;
  extern __shared__ __align__(16) char smem[];
  __shared__ int missing;
  __shared__ float stat[2][kWaves];
  // (as in encoder_chain.hip: what depends on the lane or the arguments is not kept over the loop)
  typedef const __attribute__((address_space(4))) DecoderArgs Arguments;
  auto arguments = []() __attribute__((always_inline)) {
    uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return reinterpret_cast<Arguments*>(p);
  };
  const int G = gridDim.x, me = blockIdx.x;
  auto items = [&](int step) __attribute__((always_inline)) {
    const Arguments& a = *arguments();
    if (step == 0) return a.width / (16 * kColumns);
    if (step == STEPS - 1) return a.hidden / 16;
    return (a.rows * a.heads * a.waves + kWaves - 1) / kWaves;
  };
  // The steps' items one after the other over the workgroups.
  auto first_item = [&](int step) __attribute__((always_inline)) {
    int before = 0;
    for (int s = 0; s < step; ++s) before += items(s);
    before %= G;
    return me >= before ? me - before : me - before + G;
  };
  // All of the arguments are requested at once: where they lie a first read takes as long as an exchange.
  {
    const __attribute__((address_space(4))) uint32_t* words = reinterpret_cast<const __attribute__((address_space(4))) uint32_t*>(arguments());
    uint32_t first[sizeof(DecoderArgs) / 64 + 1];
#pragma unroll
    for (uint32_t i = 0; i < sizeof(first) / 4; ++i) first[i] = words[min(i * 16, (uint32_t)sizeof(DecoderArgs) / 4 - 1)];
#pragma unroll
    for (uint32_t i = 0; i < sizeof(first) / 4; ++i) asm volatile("" : : "s"(first[i]));
  }
  __shared__ uint32_t launches;  // recorded: so far
  auto shift = [&]() __attribute__((always_inline)) { return RECORDED ? part_offset(__builtin_amdgcn_readfirstlane(launches), arguments()->bytes) : 0u; };
  // The workgroups that are done first fill the other part of the exchange memory.
  auto leave = [&]() __attribute__((always_inline)) {
    const Arguments& a = *arguments();
    const int fillers = min(G, items(0));
    if (me < fillers) fill_unwritten(RECORDED ? a.exchange + (a.bytes - shift()) : a.other, a.bytes, me, fillers);
    if constexpr (RECORDED) count_launch(a.count, me, G);
  };

  ChainWalk walk;
  walk.item = first_item(0) - G;
  walk.forward(G, STEPS, items, first_item);
  if (walk.step >= STEPS) {
    leave();
    return;
  }
  if (threadIdx.x == 0) {
    missing = 0;
    if (RECORDED && walk.step != 0) launches = launches_so_far(arguments()->count);
  }
  __syncthreads();

  for (;;) {
    const Arguments& a = *arguments();
    const int step = walk.step, item = walk.item;
    const int H = a.hidden, rows = a.rows, heads = a.heads, patience = a.patience;
    float* const part = reinterpret_cast<float*>(smem + kRows * chain_row_pitch(H, E));
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lrow = lane & 15, lgrp = lane >> 4;
    const __amdgpu_buffer_rsrc_t mem = __builtin_amdgcn_make_buffer_rsrc(a.exchange, 0, RECORDED ? 2 * a.bytes : a.bytes, 0x00020000);
    auto load4 = [&](uint32_t offset) __attribute__((always_inline)) { return (u32x4)__builtin_amdgcn_raw_buffer_load_b128(mem, offset, 0, kThroughMemory); };
    auto store1 = [&](uint32_t offset, uint32_t x) __attribute__((always_inline)) { __builtin_amdgcn_raw_buffer_store_b32(storable(x), mem, offset, 0, kThroughMemory); };
    auto store_pair = [&](uint32_t offset, float v0, float v1) __attribute__((always_inline)) {
      if constexpr (E == 4) {
        store1(offset, __builtin_bit_cast(uint32_t, v0));
        store1(offset + 4, __builtin_bit_cast(uint32_t, v1));
      } else {
        store1(offset, pack2<T>(v0, v1));
      }
    };
    // two values of a row
    typedef typename std::conditional<E == 4, u32x2, uint32_t>::type Two;
    auto first_of = [](const Two& x) __attribute__((always_inline)) {
      if constexpr (E == 4) return __builtin_bit_cast(float, (uint32_t)x[0]);
      else return low<T>(x);
    };
    auto second_of = [](const Two& x) __attribute__((always_inline)) {
      if constexpr (E == 4) return __builtin_bit_cast(float, (uint32_t)x[1]);
      else return high<T>(x);
    };
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
    const bool product = step == 0 || step == STEPS - 1;
    const int block = tid >> 7, at_tid = tid & 127, row = at_tid >> 3;
    const int n0 = step == 0 ? item * 16 * kColumns : item * 16;
    const bool stores = product && block < (step == 0 ? kColumns : 1) && row < rows;
    const int column = n0 + block * 16 + 2 * (tid & 7);
    Two bias = {}, residual = {};
    if (stores) {
      bias = *reinterpret_cast<const Two*>(static_cast<const T*>(step == 0 ? a.b_in : a.b_out) + column);
      if (step != 0) residual = *reinterpret_cast<const Two*>(static_cast<const T*>(a.x) + row * H + column);
    }
    floatx4 acc[kColumns];
#pragma unroll
    for (int c = 0; c < kColumns; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};

    if (step == 0) {
      const int pieces = H / PIECE, share = (pieces + kWaves - 1) / kWaves, mine = min(pieces - wave * share, share);
      const __amdgpu_buffer_rsrc_t weights = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.w_in), 0, a.width * H * E, 0x00020000);
      const uint32_t w_row = (uint32_t)((n0 + lrow) * H * E + wave * share * 128 + lgrp * 32);
      const int pitch = chain_row_pitch(H, E);
      u32x4 wf[PIECES][kColumns][2];
      const __amdgpu_buffer_rsrc_t x = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, rows * H * E, 0x00020000);
      const __amdgpu_buffer_rsrc_t g = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.gamma), 0, H * E, 0x00020000);
      const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.beta), 0, H * E, 0x00020000);
      auto four = [&](const __amdgpu_buffer_rsrc_t& from, uint32_t at) __attribute__((always_inline)) {
        if constexpr (E == 4) return (u32x4)__builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0);
        else return (u32x2)__builtin_amdgcn_raw_buffer_load_b64(from, at, 0, 0);
      };
#pragma unroll
      for (int p = 0; p < PIECES; ++p)
#pragma unroll
        for (int c = 0; c < kColumns; ++c)
#pragma unroll
          for (int s = 0; s < 2; ++s)
            wf[p][c][s] = (u32x4)__builtin_amdgcn_raw_buffer_load_b128(weights, p < mine ? w_row + (uint32_t)(c * 16 * H * E + p * 128 + s * 16) : kOutside, 0, 0);
      // Requested in this order and here, not where they are used: the weights come from the furthest.
      asm volatile("" ::: "memory");
      uint32_t so_far = 0;
      if (RECORDED && tid == 0) so_far = launches_so_far(a.count);
      if (wave < rows) {
        Four<T> raw[kTurns], gm[kTurns], bt[kTurns];
#pragma unroll
        for (int t = 0; t < kTurns; ++t) {  // columns that do not exist are zeros
          const int col = t * 256 + lane * 4;
          raw[t] = four(x, col < H ? (uint32_t)((wave * H + col) * E) : kOutside);
          gm[t] = four(g, (uint32_t)(col * E));
          bt[t] = four(b, (uint32_t)(col * E));
        }
        asm volatile("" ::: "memory");
        float v[kTurns][4], normed[kTurns][4];
#pragma unroll
        for (int t = 0; t < kTurns; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[t][e] = of_four<T>(raw[t], e);
        normalise_row<T, kTurns>(v, gm, bt, H, a.eps, normed);
#pragma unroll
        for (int t = 0; t < kTurns; ++t) {
          const int col = t * 256 + lane * 4;
          if (col < H) *reinterpret_cast<Four<T>*>(smem + wave * pitch + col * E) = to_four<T>(normed[t]);
        }
      }
      if (RECORDED && tid == 0) launches = so_far;
      __syncthreads();
#pragma unroll
      for (int p = 0; p < PIECES; ++p)
        if (p < mine)
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const u32x4 rows_here = *reinterpret_cast<const u32x4*>(smem + lrow * pitch + (wave * share + p) * 128 + lgrp * 32 + s * 16);
#pragma unroll
            for (int c = 0; c < kColumns; ++c) acc[c] = mma16<T>(rows_here, wf[p][c][s], acc[c]);
          }
    } else if (step == STEPS - 1) {
      const int K = a.inner, share = (K / PIECE + kWaves - 1) / kWaves, first = wave * share, mine = min(K / PIECE - first, share), there = lrow < rows ? mine : 0;
      const __amdgpu_buffer_rsrc_t weights = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.w_out), 0, H * K * E, 0x00020000);
      const uint32_t w_row = (uint32_t)((n0 + lrow) * K * E + first * 128 + lgrp * 32);
      u32x4 wf[2 * OUT_PIECES], af[2 * OUT_PIECES];
      if (BLOCK == kFeedForward || mine > 0) {  // (the same for the wavefront; all of them have a share of the many rows of W2)
#pragma unroll
        for (int p = 0; p < 2 * OUT_PIECES; ++p) wf[p] = (u32x4)__builtin_amdgcn_raw_buffer_load_b128(weights, p / 2 < mine ? w_row + (p / 2) * 128 + (p & 1) * 16 : kOutside, 0, 0);
        const uint32_t row_at = shift() + (BLOCK == kFeedForward ? 0u : context_at(a.width, E)) + fragment_offset<T>(lrow, first * PIECE + lgrp * (PIECE / 4));
        await([&]() __attribute__((always_inline)) {
#pragma unroll
          for (int p = 0; p < 2 * OUT_PIECES; ++p) af[p] = load4(p / 2 < there ? row_at + p * (kRows * 64) : kOutside);
          uint32_t m = 0;
#pragma unroll
          for (int p = 0; p < 2 * OUT_PIECES; ++p) m = largest(m, af[p]);
          return m;
        });
        if (late) missing = 1;
#pragma unroll
        for (int p = 0; p < 2 * OUT_PIECES; ++p) acc[0] = mma16<T>(af[p], wf[p], acc[0]);
      }
    } else if constexpr (BLOCK != kFeedForward) {
      // A wavefront takes 8 * LOADS keys of a head: a lane eight columns of every eighth key.
      const int pair = item * (kWaves / a.waves) + wave / a.waves, share = wave % a.waves, key0 = share * (8 * LOADS) + (lane >> 3), piece = lane & 7;
      const bool has = pair < rows * heads;
      const int b = has ? pair / heads : 0, head = has ? pair - b * heads : 0, keys = a.keys, past = a.past;
      const __amdgpu_buffer_rsrc_t kp = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.k_past), 0, rows * heads * past * kD * E, 0x00020000);
      const __amdgpu_buffer_rsrc_t vp = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.v_past), 0, rows * heads * past * kD * E, 0x00020000);
      Eight<T> kf[LOADS], vf[LOADS];
      float mk[LOADS];
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int key = key0 + i * 8;
        const uint32_t at = (uint32_t)((pair * past + key) * (kD * E) + piece * (8 * E));
#pragma unroll
        for (int h = 0; h < E / 2; ++h) {
          kf[i].q[h] = (u32x4)__builtin_amdgcn_raw_buffer_load_b128(kp, has && key < past ? at + h * 16 : kOutside, 0, 0);
          vf[i].q[h] = (u32x4)__builtin_amdgcn_raw_buffer_load_b128(vp, has && key < past ? at + h * 16 : kOutside, 0, 0);
        }
        mk[i] = a.mask != nullptr ? a.mask[b * keys + min(key, keys - 1)] : 0.f;
      }
      Eight<T> qf, kn, vn;
      const uint32_t at = shift() + (uint32_t)((b * a.width + head * kD + piece * 8) * E), row_bytes = (uint32_t)(H * E);
      await([&]() __attribute__((always_inline)) {
        uint32_t m = 0;
#pragma unroll
        for (int h = 0; h < E / 2; ++h) {
          qf.q[h] = load4(has ? at + h * 16 : kOutside);
          if constexpr (BLOCK == kSelfAttention) {
            kn.q[h] = load4(has ? at + row_bytes + h * 16 : kOutside);
            vn.q[h] = load4(has ? at + 2 * row_bytes + h * 16 : kOutside);
          }
        }
#pragma unroll
        for (int h = 0; h < E / 2; ++h) {
          m = largest(m, qf.q[h]);
          if constexpr (BLOCK == kSelfAttention) m = largest(largest(m, kn.q[h]), vn.q[h]);
        }
        return m;
      });
      if (late) missing = 1;
      float s[LOADS], mx = -__builtin_inff();
      auto larger = [](float x, float y) { return fmaxf(x, y); };
      auto add = [](float x, float y) { return x + y; };
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int key = key0 + i * 8;
        if constexpr (BLOCK == kSelfAttention) {
          if (key == past) kf[i] = kn, vf[i] = vn;
          if (!late && has && key < keys) {
            const int64_t to = ((int64_t)pair * keys + key) * kD + piece * 8;
#pragma unroll
            for (int h = 0; h < E / 2; ++h) {
              *reinterpret_cast<u32x4*>(static_cast<T*>(a.k_out) + to + h * (16 / E)) = kf[i].q[h];
              *reinterpret_cast<u32x4*>(static_cast<T*>(a.v_out) + to + h * (16 / E)) = vf[i].q[h];
            }
          }
        }
        s[i] = __builtin_fmaf(over_pieces(dot8<T>(kf[i], qf), add), a.scale, mk[i]);
        if (key < keys) mx = fmaxf(mx, s[i]);
      }
      mx = over_keys(mx, larger);
      if (lane == 0) stat[0][wave] = mx;
      __syncthreads();
      const int lead = wave - share;
      for (int w = 0; w < a.waves; ++w) mx = fmaxf(mx, stat[0][lead + w]);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        s[i] = key0 + i * 8 < keys ? __builtin_amdgcn_exp2f((s[i] - mx) * kLog2e) : 0.f;
        sum += s[i];
      }
      sum = over_keys(sum, add);
      if (lane == 0) stat[1][wave] = sum;
      __syncthreads();
      sum = 0.f;
      for (int w = 0; w < a.waves; ++w) sum += stat[1][lead + w];
      const float inv = 1.0f / sum;
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = 0.f;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int key = key0 + i * 8;
        const T p = from_float<T>(s[i] * inv);
        if (!late && has && key < keys && piece == 0) static_cast<T*>(a.probs)[(int64_t)pair * keys + key] = p;
        const float weight = to_float(p);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = __builtin_fmaf(weight, vf[i].at(e), o[e]);  // (keys past the last are zeros)
      }
      // eight groups of lanes have a part each: two of a row of 16 lanes meet here, the rest in LDS
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] += dpp_move<0x128>(o[e]);
      if ((lane & 8) == 0)
#pragma unroll
        for (int e = 0; e < 8; e += 4)
          *reinterpret_cast<floatx4*>(part + (wave * 4 + lgrp) * kD + piece * 8 + e) = floatx4{o[e], o[e + 1], o[e + 2], o[e + 3]};
    }

    if (product) {
#pragma unroll
      for (int c = 0; c < kColumns; ++c)
        if (c == 0 || step == 0)
#pragma unroll
          for (int e = 0; e < 4; ++e) part[(wave * kRows + lgrp * 4 + e) * kPitch + c * 16 + lrow] = acc[c][e];
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(missing) != 0) {  // set in front of the barrier: the same for all
      __syncthreads();
      if (tid == 0) missing = 0;
      if (!walk.late(0)) {  // (not reached while every item's inputs are some item's outputs)
        if (tid == 0 && a.error != nullptr) *a.error = kRowsNeverCame;
        leave();
        return;
      }
      __syncthreads();
      continue;
    }
    if (stores) {
      const floatx2 v = sum_parts(part, row, column - n0, 1);
      const float v0 = v[0] + first_of(bias), v1 = v[1] + second_of(bias);
      if (step == STEPS - 1) {
        Vec<T, 2> r;
        r.v[0] = from_float<T>(v0 + first_of(residual));
        r.v[1] = from_float<T>(v1 + second_of(residual));
        store_vec<T, 2>(static_cast<T*>(a.out) + row * H + column, r);
      } else if constexpr (BLOCK == kFeedForward) {
        store_pair(shift() + fragment_offset<T>(row, column), fmaxf(v0, 0.f), fmaxf(v1, 0.f));
      } else {
        store_pair(shift() + (uint32_t)((row * a.width + column) * E), v0, v1);
      }
    } else if (!product) {
      // the context of the workgroup's heads, two columns a thread
      const int mine = tid / (kD / 2), pair = item * (kWaves / a.waves) + mine, col = 2 * (tid % (kD / 2));
      if (mine < kWaves / a.waves && pair < rows * heads) {
        float v0 = 0.f, v1 = 0.f;
#pragma unroll 4
        for (int w = 0; w < 4 * a.waves; ++w) {
          const floatx2 p = *reinterpret_cast<const floatx2*>(part + (mine * 4 * a.waves + w) * kD + col);
          v0 += p[0];
          v1 += p[1];
        }
        const int b = pair / heads;
        store_pair(shift() + context_at(a.width, E) + fragment_offset<T>(b, (pair - b * heads) * kD + col), v0, v1);
      }
    }
    walk.executed(G, STEPS, items, first_item);
    if (walk.step >= STEPS) {
      leave();
      return;
    }
    __syncthreads();  // the rows and partial tiles have been read
  }
#endif
}

int64_t part_bytes(Block block, int64_t hidden, int64_t width, int64_t element) { return kRows * element * (width + (block == kFeedForward ? 0 : hidden)); }

template <typename T, Block BLOCK, int LOADS, bool RECORDED>
int launch_sized(DecoderArgs a, int workgroups, hipStream_t s) {
  a.waves = 1;
  while (BLOCK != kFeedForward && a.waves * 8 * LOADS < a.keys) a.waves *= 2;
  const int64_t middle = BLOCK == kFeedForward ? 0 : ceil_div((int64_t)a.rows * a.heads * a.waves, kWaves);
  const int64_t all = a.width / (16 * kColumns) + middle + a.hidden / 16;
  const unsigned grid = workgroups > 0 ? (unsigned)workgroups : (unsigned)std::min<int64_t>(all, compute_units());
  const int lds = kRows * chain_row_pitch(a.hidden, sizeof(T)) + kWaves * kRows * kPitch * 4;
  auto kernel = decoder_chain_kernel<T, BLOCK, LOADS, RECORDED>;
  // more than 64 KB of dynamic LDS: the limit is raised once per kernel and device
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
  return launch_status("decoder_chain_kernel");
}

template <typename T, Block BLOCK, bool RECORDED>
int launch_for(const DecoderArgs& a, int workgroups, hipStream_t s) {
  // Few keys a wavefront: the sixteen of a workgroup share four SIMDs, and what the attention of 64 keys takes there is more than an exchange.
  if constexpr (BLOCK != kFeedForward)
    if (a.keys > 16 * kWaves) return launch_sized<T, BLOCK, sizeof(T) == 4 ? 4 : 8, RECORDED>(a, workgroups, s);  // (fp32: 64 keys do not fit the registers)
  if constexpr (BLOCK == kFeedForward) {
    constexpr int kPieces = 3072 * (int)sizeof(T) / 128 / kWaves;
    if (a.inner > 3072) return launch_sized<T, BLOCK, sizeof(T) == 4 ? kPieces : 4, RECORDED>(a, workgroups, s);  // (fp32: refused)
    return launch_sized<T, BLOCK, kPieces, RECORDED>(a, workgroups, s);
  } else {
    return launch_sized<T, BLOCK, 2, RECORDED>(a, workgroups, s);
  }
}

template <typename T, Block BLOCK>
int launch(DecoderArgs a, void* exchange, int turn, int workgroups, hipStream_t s) {
  Turn t;
  const int rc = take_turn(exchange, a.bytes, turn, &t);
  if (rc != 0) return rc;
  a.exchange = t.mine, a.other = t.other, a.count = t.count;
  return t.count != nullptr ? launch_for<T, BLOCK, true>(a, workgroups, s) : launch_for<T, BLOCK, false>(a, workgroups, s);
}

bool takes(int64_t rows, int64_t hidden, int dtype) {
  return (dtype == TTMI_F32 || dtype == TTMI_F16 || dtype == TTMI_BF16) && rows >= 1 && rows <= kRows && hidden >= 64 && hidden % 64 == 0 && hidden <= kMostHidden;
}

}  // namespace
}  // namespace ttmi

using namespace ttmi;

extern "C" {

int ttmi_decoder_chain_workspace(int64_t rows, int64_t heads, int64_t hidden, int64_t inner, int64_t keys, int dtype, int64_t* bytes) {
  TTMI_REQUIRE(bytes != nullptr, "null result");
  *bytes = 0;
  if (!takes(rows, hidden, dtype)) return 0;
  if (heads > 0) {
    if (hidden == heads * kD && keys >= 1 && keys <= kMostKeys && (inner == hidden || inner == 3 * hidden)) *bytes = exchange_bytes(part_bytes(kSelfAttention, hidden, inner, (int64_t)dtype_size(dtype)));
  } else if (inner >= 64 && inner % 64 == 0 && inner <= (dtype == TTMI_F32 ? kMostInner32 : kMostInner)) {
    *bytes = exchange_bytes(part_bytes(kFeedForward, hidden, inner, (int64_t)dtype_size(dtype)));
  }
  return 0;
}

int ttmi_chain_prepare(void* exchange, int64_t bytes, void* stream) {
  TTMI_REQUIRE(exchange && bytes > kCountBytes && bytes % 16 == 0 && (reinterpret_cast<uintptr_t>(exchange) & 15) == 0,
               "exchange memory comes in whole, aligned 16 bytes");
  return launch_prepare_exchange(exchange, bytes, (hipStream_t)stream);
}

int ttmi_decoder_feed_forward(const void* x, const void* gamma, const void* beta, float eps, const void* w1, const void* b1, const void* w2, const void* b2,
                              void* out, void* exchange, int turn, int64_t rows, int64_t hidden, int64_t inner, int dtype, int workgroups, int patience,
                              void* stream) {
  TTMI_REQUIRE(x && gamma && beta && w1 && b1 && w2 && b2 && out && exchange, "null tensor");
  int64_t bytes = 0;
  const int rc = ttmi_decoder_chain_workspace(rows, 0, hidden, inner, 0, dtype, &bytes);
  if (rc != 0) return rc;
  TTMI_REQUIRE(bytes > 0 && workgroups >= 0 && workgroups <= kChainMostWorkgroups && patience >= 0, "this block is not run as one launch");
  uintptr_t bits = 0;
  for (const void* p : {x, gamma, beta, w1, b1, w2, b2, (const void*)out, (const void*)exchange}) bits |= reinterpret_cast<uintptr_t>(p);
  TTMI_REQUIRE((bits & 15) == 0, "tensors must be 16-byte aligned");
  const int64_t e = (int64_t)dtype_size(dtype);
  TTMI_REQUIRE(results_apart({{out, rows * hidden * e}}, {{x, rows * hidden * e}}), "out must share no memory with x");
  DecoderArgs a{};
  a.x = x, a.gamma = gamma, a.beta = beta, a.w_in = w1, a.b_in = b1, a.w_out = w2, a.b_out = b2, a.out = out;
  a.rows = (int)rows, a.hidden = (int)hidden, a.width = (int)inner, a.inner = (int)inner, a.eps = eps, a.heads = 1;
  a.patience = patience > 0 ? patience : kChainPatience, a.error = async_error_flag();
  a.bytes = (uint32_t)part_of_exchange(bytes);
  TTMI_DISPATCH_FLOAT(dtype, T, return (launch<T, kFeedForward>(a, exchange, turn, workgroups, (hipStream_t)stream)));
  return 0;
}

int ttmi_decoder_attention(const void* x, const void* gamma, const void* beta, float eps, const void* w_in, const void* b_in, const void* w_out,
                           const void* b_out, const void* k_past, const void* v_past, void* k_out, void* v_out, const float* mask, void* probs, void* out,
                           void* exchange, int turn, int64_t rows, int64_t heads, int64_t hidden, int64_t keys, float scale, int dtype, int workgroups,
                           int patience, void* stream) {
  TTMI_REQUIRE(x && gamma && beta && w_in && b_in && w_out && b_out && k_past && v_past && probs && out && exchange, "null tensor");
  TTMI_REQUIRE((k_out == nullptr) == (v_out == nullptr), "the grown cache is both tensors or none");
  const bool grows = k_out != nullptr;
  const int64_t width = grows ? 3 * hidden : hidden, past = grows ? keys - 1 : keys;
  int64_t bytes = 0;
  const int rc = ttmi_decoder_chain_workspace(rows, heads, hidden, width, keys, dtype, &bytes);
  if (rc != 0) return rc;
  TTMI_REQUIRE(heads > 0 && bytes > 0 && past > 0 && workgroups >= 0 && workgroups <= kChainMostWorkgroups && patience >= 0, "this attention is not run as one launch");
  uintptr_t bits = 0;
  for (const void* p : {x, gamma, beta, w_in, b_in, w_out, b_out, k_past, v_past, (const void*)k_out, (const void*)v_out, (const void*)out, (const void*)exchange})
    bits |= reinterpret_cast<uintptr_t>(p);
  TTMI_REQUIRE((bits & 15) == 0, "tensors must be 16-byte aligned");
  const int64_t e = (int64_t)dtype_size(dtype), values = rows * hidden * e;
  TTMI_REQUIRE(results_apart({{out, values}, {probs, rows * heads * keys * e}, {k_out, values * keys}, {v_out, values * keys}},
                             {{x, values}, {k_past, values * past}, {v_past, values * past}, {mask, rows * keys * 4}}),
               "the results must share no memory with x, the cache, the mask or each other");
  DecoderArgs a{};
  a.x = x, a.gamma = gamma, a.beta = beta, a.w_in = w_in, a.b_in = b_in, a.w_out = w_out, a.b_out = b_out, a.out = out;
  a.k_past = k_past, a.v_past = v_past, a.k_out = k_out, a.v_out = v_out, a.mask = mask, a.probs = probs;
  a.rows = (int)rows, a.heads = (int)heads, a.hidden = (int)hidden, a.width = (int)width, a.inner = (int)hidden, a.eps = eps, a.scale = scale;
  a.past = (int)past, a.keys = (int)keys;
  a.patience = patience > 0 ? patience : kChainPatience, a.error = async_error_flag();
  a.bytes = (uint32_t)part_of_exchange(bytes);
  if (grows) {
    TTMI_DISPATCH_FLOAT(dtype, T, return (launch<T, kSelfAttention>(a, exchange, turn, workgroups, (hipStream_t)stream)));
  } else {
    TTMI_DISPATCH_FLOAT(dtype, T, return (launch<T, kMemoryAttention>(a, exchange, turn, workgroups, (hipStream_t)stream)));
  }
  return 0;
}

}  // extern "C"
