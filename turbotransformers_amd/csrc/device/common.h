// Shared device-side helpers for the gfx950 kernels: element types, 16-byte vector
// access, wave64 reductions and the error plumbing of the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdio>
#include <string>

#include "ttmi.h"

namespace ttmi {

constexpr int kWave = 64;  // CDNA wavefront width

using f16 = _Float16;
using bf16 = __bf16;

// ---- error plumbing -------------------------------------------------------------------
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);
int check_hip(hipError_t e, const char* what);

#define TTMI_HIP(expr)                                   \
  do {                                                   \
    int _rc = ::ttmi::check_hip((expr), #expr);          \
    if (_rc != 0) return _rc;                            \
  } while (0)

#define TTMI_REQUIRE(cond, msg)                                            \
  do {                                                                     \
    if (!(cond)) return ::ttmi::fail(TTMI_EINVAL, std::string(msg) + " [" #cond "]"); \
  } while (0)

inline int launch_status(const char* what) { return check_hip(hipGetLastError(), what); }

int* async_error_flag();  // device-visible pinned int, 0 = ok, 1 = an embedding id out of range, or:
constexpr int kRowsNeverCame = 2;

// ---- kernel-selection switches ----------------------------------------------------------
// Overrides of the launchers' own choices, for A/B timing and for tests of small and ragged shapes.  Each starts
// from an environment variable read ONCE (first use; a launch never scans the environment) and can be changed
// afterwards through ttmi_set_kernel_switch.  kSwitchUnset = the launcher decides.
constexpr int kSwitchUnset = -1;
enum KernelSwitch { kSwitchLargeTile = 0, kSwitchWaveKernel = 1, kSwitchAttentionWaves = 2, kSwitchStaticScratchLimit = 3, kSwitchW4AStages = 4, kSwitchW4SplitK = 5, kNumKernelSwitches = 6 };
int kernel_switch(KernelSwitch which);

// ---- scalar conversion ----------------------------------------------------------------
template <typename T>
__device__ __forceinline__ float to_float(T v) { return static_cast<float>(v); }
template <typename T>
__device__ __forceinline__ T from_float(float v) { return static_cast<T>(v); }

// ---- 16-byte vectors of N elements -----------------------------------------------------
template <typename T, int N>
struct alignas(sizeof(T) * N) Vec {
  T v[N];
};

template <typename T, int N>
__device__ __forceinline__ Vec<T, N> load_vec(const T* p) {
  return *reinterpret_cast<const Vec<T, N>*>(p);
}
template <typename T, int N>
__device__ __forceinline__ void store_vec(T* p, const Vec<T, N>& x) {
  *reinterpret_cast<Vec<T, N>*>(p) = x;
}
// The same store to an address that is only aligned to the element: global memory takes vector stores at any
// alignment (the target's unaligned access mode, which the compiler relies on as well), so this is still one
// instruction; a store that straddles a cache line costs a second request, nothing more.
template <typename T, int N>
struct __attribute__((packed, aligned(alignof(T)))) UnalignedVec {
  Vec<T, N> x;
};
template <typename T, int N>
__device__ __forceinline__ void store_vec_unaligned(T* p, const Vec<T, N>& x) {
  reinterpret_cast<UnalignedVec<T, N>*>(p)->x = x;
}

// ---- stores that do not wait in L2 ---------------------------------------------------------
// What a launch has stored lies in the L2s (4 MB each) until it ends, and the next launch starts when all of it has been written
// back: behind a product that stores 12 MB 3.5 us after its last wavefront, 2.2 if the stores went through L2 at once, while other
// wavefronts still computed.  A store that goes through takes longer (the stores of a 128 x 192 tile 2.0 -> 2.4 us, of a 64 x 96 one
// 1.1 -> 1.8), so few bytes stay: us a forward of base, never / from 0.5, 1.5, 4.5 MB of a launch on: fp16 1 x 387 tokens 477 / 471, 479, 482;
// 8 x 128 600 / 583, 585, 590; 8 x 256 829 / 783, 783, 791; fp32 1 x 128 555 / 547, 549, 560; 3 x 128 802 / 778, 780, 784; decoder prefix 8 x 33
// fp32 667 / 670, 663, 665.  20 x 100 fp16 853 / 814 from 1.5 MB on, 16 x 512 2429 / 2320, 20 packed requests 1875 / 1793.
// Upper lines: kMostThrough of the ring tiles (gemm_ring.h) and of the large ones (gemm_w4.h, whose fp32 outputs stay whatever their size),
// kMostRowsThrough of the quantising passes (quant.hip).  LayerNorms and attention have none.  Two begin later than at 2 MiB: the head split of
// int8 (gemm_ring.h) and LayerNorms in fp32 (rowwise.hip).
// Rows of a transposed V stay, which at most lengths are no whole cache lines: 40 x 100 tokens 1384 / 1465 with them.
constexpr int64_t kWriteThroughBytes = 2ll << 20;
inline bool writes_through(int64_t bytes) { return bytes >= kWriteThroughBytes; }
// A store of 4, 8 or 16 bytes, aligned to the element.  The compiler does not count it, which makes its waits longer than they need to
// be, never shorter.  (The no-op: it does not know either that the next instruction must not overwrite the stored registers.)
template <typename V>
__device__ __forceinline__ void store_through(void* p, const V& x) {
  static_assert(sizeof(V) == 16 || sizeof(V) == 8 || sizeof(V) == 4, "one store");
#if defined(__HIP_DEVICE_COMPILE__)
  typedef uint32_t Quad __attribute__((ext_vector_type(4)));
  typedef uint32_t Pair __attribute__((ext_vector_type(2)));
  if constexpr (sizeof(V) == 16) asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(__builtin_bit_cast(Quad, x)) : "memory");
  else if constexpr (sizeof(V) == 8) asm volatile("global_store_dwordx2 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(__builtin_bit_cast(Pair, x)) : "memory");
  else asm volatile("global_store_dword %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(__builtin_bit_cast(uint32_t, x)) : "memory");
#endif
}

// ---- wave64 reductions over groups of G lanes (G power of two, 4 <= G <= 64) ------------
// Partners come through data-parallel-primitive moves and the row swaps, a few cycles each, where a __shfl_xor is a trip
// through the LDS unit (~100 cycles, six in a chain: the larger part of a LayerNorm over a few rows).  The order is that
// of the butterfly over G/2, ..., 2, 1: once lanes that differ by 16 and 8 agree, rotating a row of 16 by 4, 2 or 1 meets
// the same values as the exclusive or.  (The quantised layers round what follows to 8 bits, so a sum in another order
// would move their results by whole steps.)
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// A value of both half-wavefronts (both halves of every pair of 16-lane rows) in every lane.  The elements of the result are
// copied before the bit cast: the compiler takes element 0 where it casts an element of a vector in place.
struct LanePair {
  float a, b;
};
__device__ __forceinline__ LanePair swap_halves(float v) {
  const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  const unsigned a = sw[0], b = sw[1];
  return {__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)};
}
__device__ __forceinline__ LanePair swap_rows(float v) {
  const auto sw = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  const unsigned a = sw[0], b = sw[1];
  return {__builtin_bit_cast(float, a), __builtin_bit_cast(float, b)};
}
template <int G, typename Op>
__device__ __forceinline__ float group_reduce(float v, Op op) {
  static_assert(G == 4 || G == 8 || G == 16 || G == 32 || G == 64, "group of 4 to 64 lanes");
  if constexpr (G >= 64) {
    const LanePair p = swap_halves(v);
    v = op(p.a, p.b);
  }
  if constexpr (G >= 32) {
    const LanePair p = swap_rows(v);
    v = op(p.a, p.b);
  }
  if constexpr (G >= 16) v = op(v, dpp_move<0x128>(v));  // row_ror:8
  if constexpr (G >= 16) v = op(v, dpp_move<0x124>(v));  // row_ror:4
  else if constexpr (G >= 8) v = op(v, __shfl_xor(v, 4, kWave));
  v = op(v, dpp_move<0x4E>(v));  // quad_perm [2,3,0,1]
  v = op(v, dpp_move<0xB1>(v));  // quad_perm [1,0,3,2]
  return v;
}
template <int G>
__device__ __forceinline__ float group_sum(float v) {
  return group_reduce<G>(v, [](float a, float b) { return a + b; });
}
template <int G>
__device__ __forceinline__ float group_max(float v) {
  return group_reduce<G>(v, [](float a, float b) { return fmaxf(a, b); });
}

// Packed batches of more workgroups than CUs start their long sequences first.  Workgroups start in the order of their index
// and those of a batch of ordinary size are all resident at once, so what a CU gets besides its first workgroup is given by
// that order: with the lengths in the caller's order some get two long ones, others none.  us per attention launch, 12 heads,
// as given / longest first: 20 requests of 5 to 500 tokens fp16 23.8 / 20.4, fp32 146 / 105; 32 of 20 to 512 fp16 32.6 / 26.1;
// 32 of 5 to 200 fp16 11.2 / 9.5.  Where every workgroup has a CU of its own, or none has more than
// two tiles of keys, there is nothing to gain and 0.35 us to lose (fp16, 30 requests of 5 to 60 tokens).
constexpr unsigned kOrderMinWorkgroups = 256;
constexpr int kOrderMinLength = 128;
// The sequence of a packed batch that comes `rank`-th when they are ordered by length, longest first (ties: by index).  Lane i
// holds the length of sequence i; the length of that rank is found bit by bit, which takes a ballot per bit of `longest` (an
// upper bound of the lengths).  Batches of more than 64 sequences are ordered 64 at a time.  `rank` is uniform.
__device__ __forceinline__ int longest_first(const int32_t* __restrict__ cu, int batch, int rank, int longest) {
  const int base = rank & ~(kWave - 1), lane = (int)(threadIdx.x % kWave);
  rank -= base;
  int len = -1;
  if (base + lane < batch) len = cu[base + lane + 1] - cu[base + lane];
  int found = 0;  // the largest length that more than `rank` sequences reach
  for (int bit = 31 - __builtin_clz(longest | 1); bit >= 0; --bit) {
    const int candidate = found | (1 << bit);
    if (__popcll(__ballot(len >= candidate)) > rank) found = candidate;
  }
  uint64_t same = __ballot(len == found);
  for (int skip = rank - __popcll(__ballot(len > found)); skip > 0; --skip) same &= same - 1;
  return base + (same != 0 ? __ffsll((unsigned long long)same) - 1 : rank);  // (lengths past the bound: any sequence of the batch)
}

// tanh-form GELU exactly as the reference states it, written through the logistic identity
// 0.5*(1+tanh(u)) == 1/(1+exp(-2u)), u = sqrt(2/pi)*(x + 0.044715 x^3).  With the constants folded
// into one polynomial in x it is 5 VALU operations plus one v_exp_f32 and one v_rcp_f32 (both
// accurate to 1 ulp; a correctly rounded division would cost ten more instructions).
__device__ __forceinline__ float gelu_tanh(float x) {
  constexpr float c1 = -2.0f * 1.4426950408889634f * 0.7978845608028654f;  // exp(-2u) = exp2(x*(c1 + c3 x^2))
  constexpr float c3 = c1 * 0.044715f;
  const float e = __builtin_amdgcn_exp2f(x * __builtin_fmaf(x * x, c3, c1));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float fast_tanh(float x) {
  // tanh(x) = 1 - 2/(exp(2x)+1); saturates cleanly at +-1 when exp overflows/underflows
  const float e = __builtin_amdgcn_exp2f(x * (2.0f * 1.4426950408889634f));
  return __builtin_fmaf(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f);
}

template <int ACT>
__device__ __forceinline__ float apply_act(float x) {
  if (ACT == TTMI_ACT_GELU) return gelu_tanh(x);
  if (ACT == TTMI_ACT_TANH) return fast_tanh(x);
  return fmaxf(x, 0.0f);
}

inline int compute_units() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    return n;
  }();
  return cus;
}
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

inline size_t dtype_size(int dtype) {
  switch (dtype) {
    case TTMI_F32: return 4;
    case TTMI_F16: return 2;
    case TTMI_BF16: return 2;
    case TTMI_I8: return 1;
    case TTMI_I32: return 4;
    case TTMI_I64: return 8;
    default: return 0;
  }
}

// Dispatch a generic lambda on the floating storage type.
#define TTMI_DISPATCH_FLOAT(dtype, T, ...)                                  \
  switch (dtype) {                                                          \
    case TTMI_F32: { using T = float; __VA_ARGS__; break; }                 \
    case TTMI_F16: { using T = ::ttmi::f16; __VA_ARGS__; break; }           \
    case TTMI_BF16: { using T = ::ttmi::bf16; __VA_ARGS__; break; }         \
    default: return ::ttmi::fail(TTMI_EINVAL, "unsupported dtype");         \
  }

}  // namespace ttmi
