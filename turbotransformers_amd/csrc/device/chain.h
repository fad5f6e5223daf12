// What the kernels share that run several dependent steps of a few rows as one launch (encoder_chain.hip, decoder_chain.hip).
//
// What one step leaves for the next goes through memory, past the L2s.  The exchange memory is filled with a word that no result has
// (kUnwritten: a NaN that every store here replaces by another one), and a reader asks again until it has words of another value.
// The exchange memory is kept by the caller in parts that take turns: a launch fills the part that the one before it has used.  Where launches are
// recorded and replayed, in an order that nobody knows, the host cannot tell whose turn it is: they have two parts of their own and count themselves behind
// those (count_launch).  us per recorded step of six decoder layers of base, three launches a layer each filling its part by a launch in front / so, and the 48
// launches that they replace: fp16 1 x 6 keys 183 / 168, 220; 8 x 41 214 / 198, 231; 16 x 41 248 / 232, 236; 16 x 201 273 / 255, 262; fp32 8 x 41 306 / 286, 308;
// 16 x 41 345 / 319, 331; an encoder layer of base by itself, 10 rows, 27.5 / 23.7, 27.
// An exchange between 256 workgroups that each read all of it takes 1.3 to 1.6 us for 16 to 32 KB, measured by itself (in the chains, where fewer take
// part or read a share, 0.7 to 1.5); a launch of its own with the same reads and writes 2.9, a
// barrier over the grid with counters 4 to 5.
#pragma once

#include <initializer_list>

#include "attention_common.h"
#include "chain_walk.h"

namespace ttmi {

constexpr int kChainWaves = 16, kChainThreads = kChainWaves * kWave;
constexpr int kChainRows = TTMI_CHAIN_MAX_ROWS;    // of a block of the matrix instruction: as many as a call may have
static_assert(kChainRows == 16 && kChainRows == kChainWaves, "a block of rows, and a row for each wavefront to normalise");
constexpr int kChainColumns = 2;                   // blocks of 16 columns of an item of a step with LayerNorm in front
constexpr int kChainPitch = kChainColumns * 16 + 4;  // words of a row of a partial tile
constexpr uint32_t kUnwritten = 0xffffffffu, kOtherNaN = 0xfffefffeu;
constexpr int kThroughMemory = 17;                 // cache policy sc0 | sc1: not from, and not into, the L2 of the XCD
constexpr uint32_t kOutside = 0xffffff00u;         // an offset past every buffer: a load from there is zero
constexpr int kChainPatience = 512;                // polls, of about a microsecond

__device__ __forceinline__ uint32_t storable(uint32_t word) { return word == kUnwritten ? kOtherNaN : word; }
// The largest word so far: kUnwritten if one of them is.
__device__ __forceinline__ uint32_t largest(uint32_t m, const u32x4& x) { return max(max(max(m, x[0]), max(x[1], x[2])), x[3]); }
__device__ __forceinline__ uint32_t largest(uint32_t m, const u32x2& x) { return max(max(m, x[0]), x[1]); }

// 16 bytes of a row of either operand: eight 16-bit values, or four of fp32 with an instruction for each.
template <typename T>
__device__ __forceinline__ floatx4 mma16(const u32x4& a, const u32x4& b, floatx4 c) {
  if constexpr (std::is_same<T, float>::value) {
    const floatx4 x = __builtin_bit_cast(floatx4, a), y = __builtin_bit_cast(floatx4, b);
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], y[j], c, 0, 0, 0);
    return c;
  } else if constexpr (std::is_same<T, f16>::value) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <typename T>
__device__ __forceinline__ float low(uint32_t pair) { return (float)__builtin_bit_cast(T, (uint16_t)(pair & 0xffffu)); }
template <typename T>
__device__ __forceinline__ float high(uint32_t pair) { return (float)__builtin_bit_cast(T, (uint16_t)(pair >> 16)); }

// Four values of a row.
template <typename T>
using Four = typename std::conditional<sizeof(T) == 4, u32x4, u32x2>::type;
template <typename T>
__device__ __forceinline__ float of_four(const Four<T>& x, int e) {
  if constexpr (sizeof(T) == 4) return __builtin_bit_cast(float, (uint32_t)x[e]);
  else return e & 1 ? high<T>(x[e >> 1]) : low<T>(x[e >> 1]);
}
template <typename T>
__device__ __forceinline__ Four<T> to_four(const float (&v)[4]) {
  if constexpr (sizeof(T) == 4) return __builtin_bit_cast(u32x4, floatx4{v[0], v[1], v[2], v[3]});
  else return u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
}

// Rows that the next step multiplies as they are lie as its wavefronts hold them in registers, a load of one 64 consecutive pieces: what
// goes past the L2 is paid by the line and the load.  [K / 64, 2, 4, kChainRows, 8], of fp32 [K / 32, 2, 4, kChainRows, 4];
// in bytes, of an even column:
template <typename T>
__device__ __forceinline__ uint32_t fragment_offset(int row, int col) {
  if constexpr (sizeof(T) == 4) return (uint32_t)(((((col >> 5) * 2 + ((col >> 2) & 1)) * 4 + ((col >> 3) & 3)) * kChainRows + row) * 4 + (col & 3)) * 4;
  return (uint32_t)(((((col >> 6) * 2 + ((col >> 3) & 1)) * 4 + ((col >> 4) & 3)) * kChainRows + row) * 8 + (col & 7)) * 2;
}

__host__ __device__ inline int chain_row_pitch(int hidden, int element = 2) { return hidden * element + 16; }  // bytes of an LDS row of the A operand; four banks further per row

// A row in front of a product: x, four values of every 256 columns per lane (zeros past the row), becomes v = beta + gamma * (x - mean) / sqrt(var + eps).
template <typename T, int TURNS>
__device__ __forceinline__ void normalise_row(const float (&x)[TURNS][4], const Four<T> (&gamma)[TURNS], const Four<T> (&beta)[TURNS], int width, float eps,
                                              float (&v)[TURNS][4]) {
  float sum = 0.f, sumsq = 0.f;
#pragma unroll
  for (int t = 0; t < TURNS; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sum += x[t][e];
      sumsq += x[t][e] * x[t][e];
    }
  sum = group_sum<kWave>(sum);
  sumsq = group_sum<kWave>(sumsq);
  const float mean = sum / (float)width;
  const float var = fmaxf(sumsq / (float)width - mean * mean, 0.f);  // as in layer_norm_rows
  const float rstd = 1.0f / sqrtf(var + eps);
#pragma unroll
  for (int t = 0; t < TURNS; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[t][e] = of_four<T>(beta[t], e) + of_four<T>(gamma[t], e) * rstd * (x[t][e] - mean);
      asm volatile("" : "+v"(v[t][e]));  // rounded once, from fp32
    }
}

// Two values of a tile that the wavefronts hold in parts: (row, column) and the one `step` words further.
__device__ __forceinline__ floatx2 sum_parts(const float* part, int row, int column, int step) {
  floatx2 v = {0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kChainWaves; ++w) {
    const float* p = part + (w * kChainRows + row) * kChainPitch + column;
    v[0] += p[0];
    v[1] += p[step];
  }
  return v;
}

constexpr int kCountBytes = 256;  // behind the parts: the recorded launches so far, and nothing else in its line
inline int64_t exchange_bytes(int64_t part) { return 4 * part + kCountBytes; }
inline int64_t part_of_exchange(int64_t bytes) { return (bytes - kCountBytes) / 4; }

static __global__ void prepare_exchange_kernel(u32x4* p, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t word = i < n - kCountBytes / 16 ? kUnwritten : 0u;
    p[i] = u32x4{word, word, word, word};
  }
}
inline int launch_prepare_exchange(void* p, int64_t bytes, hipStream_t s) {
  hipLaunchKernelGGL(prepare_exchange_kernel, dim3((unsigned)std::min<int64_t>(ceil_div(bytes / 16, 256), 2 * compute_units())), dim3(256), 0, s,
                     static_cast<u32x4*>(p), bytes / 16);
  return launch_status("prepare_exchange_kernel");
}
// A result of a chain, or what it reads while results are written.
struct Extent {
  const void* at;
  int64_t bytes;
};
// A workgroup that starts late reads late: whether no result shares a byte with what is read, or with another result.
inline bool results_apart(std::initializer_list<Extent> results, std::initializer_list<Extent> reads) {
  auto share = [](const Extent& a, const Extent& b) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a.at), y = reinterpret_cast<uintptr_t>(b.at);
    return x != 0 && y != 0 && x < y + (uintptr_t)b.bytes && y < x + (uintptr_t)a.bytes;
  };
  for (const Extent& r : results) {
    for (const Extent& o : results)
      if (&o != &r && share(r, o)) return false;
    for (const Extent& o : reads)
      if (share(r, o)) return false;
  }
  return true;
}
// The part of a launch, the one that it fills for the next (null: it works out both by itself), and where recorded launches are counted.
struct Turn {
  char *mine, *other;
  uint32_t* count;
};
inline int take_turn(void* exchange, int64_t part, int turn, Turn* to) {
  TTMI_REQUIRE(turn >= 0 && turn <= 2, "turn is 0, 1 or 2");
  char* const at = static_cast<char*>(exchange);
  *to = turn == 2 ? Turn{at + 2 * part, nullptr, reinterpret_cast<uint32_t*>(at + 4 * part)} : Turn{at + turn * part, at + (1 - turn) * part, nullptr};
  return 0;
}

// Recorded launches are counted (chain_walk.h).  Of the count the whole units are the same for all workgroups of a launch: every other launch has the second
// part.  One thread of a workgroup asks, in a first step behind the weights: all wavefronts at one address are a queue (a recorded step of hidden 1024, inner 3072,
// 16 sequences of 200 keys: one thread 264 us, each wavefront once 269, for each of its items 367).
__device__ __forceinline__ uint32_t launches_so_far(const uint32_t* count) { return __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ uint32_t part_offset(uint32_t launches, uint32_t part) { return (0u - (launches / kLaunchUnit & 1u)) & part; }
// At a workgroup's end; a thread of it that has asked has its answer by then.
__device__ __forceinline__ void count_launch(uint32_t* count, int rank, int workgroups) {
  if (threadIdx.x == 0) (void)__hip_atomic_fetch_add(count, launch_share((uint32_t)rank, (uint32_t)workgroups), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Workgroup `rank` of `count` fills its share.
__device__ __forceinline__ void fill_unwritten(char* p, uint32_t bytes, int rank, int count) {
  for (uint32_t at = (uint32_t)(rank * kChainThreads + (int)threadIdx.x) * 16; at < bytes; at += (uint32_t)(count * kChainThreads) * 16)
    *reinterpret_cast<u32x4*>(p + at) = u32x4{kUnwritten, kUnwritten, kUnwritten, kUnwritten};
}

}  // namespace ttmi
