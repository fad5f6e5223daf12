// What the one-kernel attention forms share: vector types, the matrix instruction over a 16-byte piece of both operands, pairs
// of 16-bit probabilities, and masks and scores far from zero.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace ttmi {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4), may_alias));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4), may_alias));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2), may_alias));

constexpr int kD = 64;  // head dim

// Weights that the following products read, brought from HBM into the last-level cache (256 MB, in front of the memory) by
// workgroups of their own behind the `rows` grid rows that compute: attention over few sequences leaves most of the chip and nearly
// all of the memory's bandwidth idle, and a product over few rows cannot hide the latency of HBM (128 x 2304 x 768 in fp32 halves 10.4
// us with cold weights, 8.2 with weights in that cache).
struct Ahead {
  const char* data[TTMI_MAX_AHEAD];
  int64_t bytes[TTMI_MAX_AHEAD];
  int ranges, rows;
};
inline int ahead_ranges(const void* const* data, const int64_t* bytes, int64_t count, Ahead* out) {
  TTMI_REQUIRE(count >= 0 && count <= TTMI_MAX_AHEAD && (count == 0 || (data && bytes)), "bad list of ranges to read ahead");
  for (int64_t i = 0; i < count; ++i) {
    TTMI_REQUIRE(bytes[i] >= 0 && (bytes[i] == 0 || data[i] != nullptr), "bad range to read ahead");
    TTMI_REQUIRE((reinterpret_cast<uintptr_t>(data[i]) & 3) == 0 && (bytes[i] & 3) == 0, "a range to read ahead is whole words");
    out->data[i] = static_cast<const char*>(data[i]);
    out->bytes[i] = bytes[i];
  }
  out->ranges = (int)count;
  return 0;
}
// One word of every 64 bytes, eight of them on the way per thread: 208 workgroups of 256 threads take 3.3 us for 9.4 MB, launch
// included (whole lines 3.4, a word per 128 bytes 3.9).
__device__ __forceinline__ void touch_ahead(const Ahead& ahead, int workgroup, int workgroups) {
  constexpr int kLine = 64, kFlying = 8;
  const int64_t first = ((int64_t)workgroup * blockDim.x + threadIdx.x) * kLine, stride = (int64_t)workgroups * blockDim.x * kLine;
#pragma unroll 1
  for (int r = 0; r < TTMI_MAX_AHEAD; ++r) {
    const char* const data = ahead.data[r];
    const int64_t bytes = ahead.bytes[r];
#pragma unroll 1
    for (int64_t at = first; at < bytes; at += kFlying * stride) {
      uint32_t word[kFlying];
#pragma unroll
      for (int j = 0; j < kFlying; ++j) word[j] = *reinterpret_cast<const uint32_t*>(data + (at + j * stride < bytes ? at + j * stride : at));
#pragma unroll
      for (int j = 0; j < kFlying; ++j) asm volatile("" : : "v"(word[j]));
    }
  }
}
// Grid rows for reading ahead behind `workgroups` of them in rows of `width`, of which `slots` fit the chip at a time: a workgroup
// per idle CU, and half as many as CUs at least (reading ahead is waiting for memory, it shares a CU well).  None where the
// attention takes several rounds.
inline unsigned ahead_rows(const Ahead* ahead, int64_t workgroups, int64_t width, int64_t slots) {
  const int64_t cus = compute_units();
  if (ahead == nullptr || ahead->ranges == 0 || workgroups > slots) return 0;
  return (unsigned)ceil_div(std::max(cus - workgroups, cus / 2), width);
}

// A launch that reads nothing ahead is compiled without the list, whose arrival its workgroups would wait for at their start: us per
// launch with / without, 12 heads, fp16, 1 x 10 tokens 3.84 / 3.72, 8 x 128 5.17 / 5.02, 8 x 256 7.54 / 7.44, 20 x 100 5.67 / 5.53.
struct NothingAhead {};
// The grid rows that compute; whether this workgroup is not one of them, and has read its share.
__device__ __forceinline__ int computing_rows(const Ahead& ahead) { return ahead.rows; }
__device__ __forceinline__ int computing_rows(const NothingAhead&) { return (int)gridDim.y; }
__device__ __forceinline__ bool has_read_ahead(const Ahead& ahead) {
  if ((int)blockIdx.y < ahead.rows) return false;
  const int width = (int)(gridDim.x * gridDim.z);
  touch_ahead(ahead, (int)(blockIdx.y - ahead.rows) * width + (int)(blockIdx.z * gridDim.x + blockIdx.x), (int)(gridDim.y - ahead.rows) * width);
  return true;
}
__device__ __forceinline__ bool has_read_ahead(const NothingAhead&) { return false; }

// D = A B + C over one 16-byte piece of both operands: eight K indices per half-wavefront in one instruction (16-bit types), or
// four, one per instruction (fp32)
template <typename T, typename Piece>
__device__ __forceinline__ floatx16 mma32(const Piece& a, const Piece& b, floatx16 c) {
  static_assert(sizeof(Piece) == 16, "a 16-byte piece");
  if constexpr (std::is_same<T, f16>::value) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  } else if constexpr (std::is_same<T, bf16>::value) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    const floatx4 x = __builtin_bit_cast(floatx4, a), y = __builtin_bit_cast(floatx4, b);
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_32x32x2f32(x[j], y[j], c, 0, 0, 0);
    return c;
  }
}

// Two floats -> one packed register (round to nearest even): v_cvt_pk_{f16,bf16}_f32.
template <typename T>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (std::is_same<T, f16>::value) return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{lo, hi}, halfx2));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{lo, hi}, bf16x2));
}
// acc + lo + hi of a packed pair (v_dot2c_f32_*): the softmax denominator is summed from the ROUNDED probabilities, the same
// values the second product consumes.
template <typename T>
__device__ __forceinline__ float add_pair(uint32_t p, float acc) {
  if constexpr (std::is_same<T, f16>::value)
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(halfx2, p), halfx2{(_Float16)1.0f, (_Float16)1.0f}, acc, false);
  else return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, p), bf16x2{(__bf16)1.0f, (__bf16)1.0f}, acc, false);
}

// Scores are kept in raw units: q . k + mask / scale, and a probability is 2^(s * c - m * c) with c = scale * log2(e), one
// multiply-add, m the running maximum.  A wholly masked row is the mean of V, as a softmax over mask + score gives it, so
// the mask of a valid key stays finite however low it is (the lowest float over the scale would be -inf, every probability
// of such a row 0 and the row 0 / 0), and keys past the end carry -inf, below any mask.  A mask of -inf stays -inf.
constexpr float kFarthestScore = 0x1p127f;  // the running maximum starts at its negative
// The mask is loaded as bits: a NaN has to stay one, but attention.hip is compiled as if there were none.  It is converted where it
// is used, not where it is requested: the conversion waits for its load, and with it for the older ones of the tile.  us per launch,
// 12 heads, converted at the request / where used: fp16 4 x 400 tokens 12.2 / 10.9, 8 x 256 7.6 / 7.4, fp32 4 x 400 40.6 / 37.8.
__device__ __forceinline__ float mask_in_scores(uint32_t mask, float inv_scale) {
  const float x = fminf(fmaxf(__builtin_bit_cast(float, mask) * inv_scale, -kFarthestScore), kFarthestScore);
  return __builtin_bit_cast(float, (mask & 0x7f800000u) != 0x7f800000u ? __builtin_bit_cast(uint32_t, x) : mask);
}
__device__ __forceinline__ uint32_t load_mask(const float* mask) { return *reinterpret_cast<const __attribute__((may_alias)) uint32_t*>(mask); }

// m * c is rounded.  The error is the same for all keys of a row and cancels in the division by the row's sum, but from
// |m * c| = 2^30 on it is 64 and more: the probabilities of a row masked with -1e10 would be 0 or infinite.  Beyond 2^12
// (error 2^-13; no row with an unmasked key comes near) the maximum is subtracted from the scores first, exactly.
// The test is three instructions per 32 keys, 1 to 2 % of a launch: fp16 1 x 400 tokens 6.6 / 6.8, 32 packed requests 23.8 / 24.0,
// fp32 16 x 512 146.1 / 146.6.  (Joined to the test for a maximum that moves it costs registers: 8 x 256 7.8 against 7.6.)
template <int N = 16, typename Scores>
__device__ __forceinline__ float relative_scores(Scores& st, float m_run, float scale_log2e) {
  const float neg_m = -m_run * scale_log2e;
  const bool far = fabsf(neg_m) > 0x1p12f;
  if (__builtin_expect(!__any(far), 1)) return neg_m;
  const float shift = far ? m_run : 0.f;
#pragma unroll
  for (int e = 0; e < N; ++e) st[e] -= shift;
  return far ? 0.f : neg_m;
}

}  // namespace ttmi
