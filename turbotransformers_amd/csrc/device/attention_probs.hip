// Attention that also returns its probabilities, head_dim 64: the attention of a decoder, over a growing key/value cache or
// over an encoder memory, and of an encoder whose caller asked for the attention matrix.
//
//     P = softmax(scale * Q K^T + mask),  out = P V,   K = [k_past | k], V = [v_past | v], both also copied to the grown cache
//
// One launch in place of two concatenations, two cache copies, two batched products and a softmax
// (layers/multi_headed_attention.cpp:205-229, :323-354): for a few hypotheses each of those is a launch of a few KB, and
// the step is bound by their number (8 hypotheses, 41 keys: 7 launches of 2 to 7 us).  The scores stay in registers.
//
// A workgroup owns 32 queries of one head; its NW wavefronts take blocks of 32 keys (wavefront w: blocks w, w + NW).  The
// scores are computed transposed (lane = query, registers = keys) as in attention.hip, the maximum and the sum of a row
// meet in LDS, the probabilities are normalised in fp32, rounded to T, stored, and used as rounded in the second product,
// as a chain through memory would; the NW partial outputs are summed in LDS.  All of K, V and the mask that a wavefront
// needs is requested before the first product.  V is row-major (a cache grows along the sequence): fp32 fragments are read
// one float per lane, 16-bit rows go through LDS, where a lane picks its column.
// Keys past 32 * NW * NB do not fit: the launcher takes the form for up to 128, 256 and 512 keys.
#include "attention_common.h"

namespace ttmi {
namespace {

constexpr int kQ = 32, kKeys = 32;  // queries per workgroup, keys per block
constexpr int kPitch = kD + 4;      // floats of a row of a partial output in LDS

struct ProbsArgs {
  const void *q, *k_past, *v_past, *k, *v;
  void *k_out, *v_out, *probs, *out;
  const float* mask;
  int heads, queries, past, keys;  // keys = past + new
  int mask_per_query;
  float scale;
};

template <typename T, int NW, int NB>
__global__ __launch_bounds__(NW * 64) void attention_probs_kernel(const ProbsArgs p) {
  constexpr int KPC = 16 / (int)sizeof(T);         // elements per 16-byte piece
  constexpr int PIECES = kD / KPC / 2;             // pieces of a row per lane
  constexpr int VPIECES = 4 * (int)sizeof(T) / 2;  // pieces of V per lane and block of keys
  constexpr float kLog2e = 1.4426950408889634f;
  // partial outputs; before them, 16-bit: the V rows of the wavefront's block
  __shared__ __align__(16) float part[NW][kQ][kPitch];
  __shared__ float stat[2][NW][kQ];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int bh = blockIdx.y, b = bh / p.heads, head = bh - b * p.heads;
  const int q0 = blockIdx.x * kQ;
  const int fresh = p.keys - p.past;
  const int blocks = (p.keys + kKeys - 1) / kKeys;
  const T* kp = (const T*)p.k_past + (int64_t)bh * p.past * kD;
  const T* vp = (const T*)p.v_past + (int64_t)bh * p.past * kD;
  const T* kn = (const T*)p.k + (int64_t)bh * fresh * kD;
  const T* vn = (const T*)p.v + (int64_t)bh * fresh * kD;
  T* ko = (T*)p.k_out + (int64_t)bh * p.keys * kD;
  T* vo = (T*)p.v_out + (int64_t)bh * p.keys * kD;
  const bool grow = p.k_out != nullptr && blockIdx.x == 0;
  const int query = min(q0 + lrow, p.queries - 1);  // lanes past the last query repeat it and store nothing
  const float* mrow = p.mask == nullptr ? nullptr
                                        : p.mask + (p.mask_per_query ? ((int64_t)b * p.queries + query) * p.keys : (int64_t)b * p.keys);
  auto key_row = [&](const T* past_rows, const T* new_rows, int key) __attribute__((always_inline)) {
    return key < p.past ? past_rows + (int64_t)key * kD : new_rows + (int64_t)(key - p.past) * kD;
  };

  u32x4 qf[PIECES];
  {
    const T* row = (const T*)p.q + ((int64_t)bh * p.queries + query) * kD + lhalf * KPC;
#pragma unroll
    for (int kk = 0; kk < PIECES; ++kk) qf[kk] = *reinterpret_cast<const u32x4*>(row + 2 * kk * KPC);
  }

  u32x4 kf[NB][PIECES], vf[NB][VPIECES];
  float mk[NB][16];
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int key0 = (wave + n * NW) * kKeys;
    if (key0 >= p.keys) continue;
    const T* row = key_row(kp, kn, min(key0 + lrow, p.keys - 1)) + lhalf * KPC;
#pragma unroll
    for (int kk = 0; kk < PIECES; ++kk) kf[n][kk] = *reinterpret_cast<const u32x4*>(row + 2 * kk * KPC);
    if constexpr (sizeof(T) == 2) {  // row key0 + 8*i + lane / 8, piece lane % 8
#pragma unroll
      for (int i = 0; i < 4; ++i)
        vf[n][i] = *reinterpret_cast<const u32x4*>(key_row(vp, vn, min(key0 + 8 * i + (lane >> 3), p.keys - 1)) + (lane & 7) * 8);
    } else {  // piece 4t+g, word i: V[key0 + 8g + 4*lhalf + i][32t + lrow]
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const T* vr = key_row(vp, vn, min(key0 + 8 * g + 4 * lhalf + i, p.keys - 1)) + lrow;
#pragma unroll
          for (int t = 0; t < 2; ++t) vf[n][4 * t + g][i] = reinterpret_cast<const uint32_t*>(vr)[t * 32];
        }
    }
    if (mrow != nullptr) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) mk[n][4 * g + i] = mrow[min(key0 + 8 * g + 4 * lhalf + i, p.keys - 1)];
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) mk[n][e] = 0.f;
    }
  }

  // ---- scores, the maximum of every query
  floatx16 st[NB];
  float mx = -__builtin_inff();
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int key0 = (wave + n * NW) * kKeys;
    if (key0 >= p.keys) continue;
#pragma unroll
    for (int e = 0; e < 16; ++e) st[n][e] = 0.f;
#pragma unroll
    for (int kk = 0; kk < PIECES; ++kk) st[n] = mma32<T>(kf[n][kk], qf[kk], st[n]);
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float s = __builtin_fmaf(st[n][4 * g + i], p.scale, mk[n][4 * g + i]);
        st[n][4 * g + i] = s;
        if (key0 + 8 * g + 4 * lhalf + i < p.keys) mx = fmaxf(mx, s);
      }
  }
  {
    const LanePair h = swap_halves(mx);
    mx = fmaxf(h.a, h.b);
  }
  if (lhalf == 0) stat[0][wave][lrow] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) mx = fmaxf(mx, stat[0][w][lrow]);

  // ---- the cache rows of the block (their loads are older than every wait above)
  if (grow) {
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const int key0 = (wave + n * NW) * kKeys;
      if (key0 >= p.keys) continue;
      if (key0 + lrow < p.keys) {
#pragma unroll
        for (int kk = 0; kk < PIECES; ++kk)
          *reinterpret_cast<u32x4*>(ko + (int64_t)(key0 + lrow) * kD + (2 * kk + lhalf) * KPC) = kf[n][kk];
      }
      if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + 8 * i + (lane >> 3);
          if (key < p.keys) *reinterpret_cast<u32x4*>(vo + (int64_t)key * kD + (lane & 7) * 8) = vf[n][i];
        }
      } else {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = key0 + 8 * g + 4 * lhalf + i;
            if (key < p.keys) {
#pragma unroll
              for (int t = 0; t < 2; ++t) reinterpret_cast<uint32_t*>(vo + (int64_t)key * kD + lrow)[t * 32] = vf[n][4 * t + g][i];
            }
          }
      }
    }
  }

  // ---- exponentials and their sum
  float sum = 0.f;
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int key0 = (wave + n * NW) * kKeys;
    if (key0 >= p.keys) continue;
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = key0 + 8 * g + 4 * lhalf + i < p.keys ? __builtin_amdgcn_exp2f((st[n][4 * g + i] - mx) * kLog2e) : 0.f;
        st[n][4 * g + i] = e;
        sum += e;
      }
  }
  {
    const LanePair h = swap_halves(sum);
    sum = h.a + h.b;
  }
  if (lhalf == 0) stat[1][wave][lrow] = sum;
  __syncthreads();
  sum = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) sum += stat[1][w][lrow];
  const float inv = 1.0f / sum;

  // ---- probabilities, second product
  floatx16 ot[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) ot[t][e] = 0.f;
  T* prow = (T*)p.probs + ((int64_t)bh * p.queries + query) * p.keys;
  const bool store_p = q0 + lrow < p.queries;
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int key0 = (wave + n * NW) * kKeys;
    if (key0 >= p.keys) continue;
#pragma unroll
    for (int e = 0; e < 16; ++e) st[n][e] *= inv;
    if (store_p) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int key = key0 + 8 * g + 4 * lhalf;
        Vec<T, 4> r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r.v[i] = from_float<T>((float)st[n][4 * g + i]);
        if (key + 4 <= p.keys) {
          store_vec_unaligned<T, 4>(prow + key, r);
        } else {
#pragma unroll
          for (int i = 0; i < 3; ++i)
            if (key + i < p.keys) prow[key + i] = r.v[i];
        }
      }
    }
    if constexpr (sizeof(T) == 2) {
      // the wavefront's V rows through its own part of LDS (its own reads and writes: in order, no barrier)
      T* rows = reinterpret_cast<T*>(&part[wave][0][0]);
      constexpr int VP = kD + 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        u32x4 x = vf[n][i];
        *reinterpret_cast<u32x4*>(rows + (8 * i + (lane >> 3)) * VP + (lane & 7) * 8) = x;
      }
      u32x4 pf[2];
#pragma unroll
      for (int w = 0; w < 8; ++w) pf[w >> 2][w & 3] = pack2<T>(st[n][2 * w], st[n][2 * w + 1]);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          u32x4 a;  // V^T[32t + lrow][16kk + 4*lhalf + {0..3, 8..11}]
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const uint16_t* e = reinterpret_cast<const uint16_t*>(rows) + (16 * kk + 4 * lhalf + 8 * (w >> 1) + 2 * (w & 1)) * VP + t * 32 + lrow;
            a[w] = (uint32_t)e[0] | (uint32_t)e[VP] << 16;
          }
          ot[t] = mma32<T>(a, pf[kk], ot[t]);
        }
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u32x4 pf;
#pragma unroll
        for (int i = 0; i < 4; ++i) pf[i] = __builtin_bit_cast(uint32_t, (float)st[n][4 * g + i]);
#pragma unroll
        for (int t = 0; t < 2; ++t) ot[t] = mma32<T>(vf[n][4 * t + g], pf, ot[t]);
      }
    }
  }

  // ---- sum of the wavefronts' outputs: ot[t][4g+i] = O[query lrow][d = 32t + 8g + 4*lhalf + i]
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<floatx4*>(&part[wave][lrow][t * 32 + 8 * g + 4 * lhalf]) =
          floatx4{ot[t][4 * g], ot[t][4 * g + 1], ot[t][4 * g + 2], ot[t][4 * g + 3]};
  __syncthreads();
  constexpr int EPT = kQ * kD / (NW * 64);  // 8 or 4
  const int qi = tid / (kD / EPT), d0 = (tid % (kD / EPT)) * EPT;
  if (q0 + qi < p.queries) {
    T* dst = (T*)p.out + ((int64_t)b * p.queries + q0 + qi) * (p.heads * kD) + head * kD + d0;
#pragma unroll
    for (int e = 0; e < EPT; e += 4) {
      floatx4 o{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) o += *reinterpret_cast<const floatx4*>(&part[w][qi][d0 + e]);
      Vec<T, 4> r;
#pragma unroll
      for (int j = 0; j < 4; ++j) r.v[j] = from_float<T>((float)o[j]);
      store_vec<T, 4>(dst + e, r);
    }
  }
}

template <typename T>
int launch_attention_probs(const ProbsArgs& p, int64_t batch, hipStream_t s) {
  const dim3 grid((unsigned)ceil_div(p.queries, kQ), (unsigned)(batch * p.heads));
  if (p.keys <= 128) hipLaunchKernelGGL((attention_probs_kernel<T, 4, 1>), grid, dim3(256), 0, s, p);
  else if (p.keys <= 256) hipLaunchKernelGGL((attention_probs_kernel<T, 8, 1>), grid, dim3(512), 0, s, p);
  else hipLaunchKernelGGL((attention_probs_kernel<T, 8, 2>), grid, dim3(512), 0, s, p);
  return launch_status("attention_probs_kernel");
}

}  // namespace
}  // namespace ttmi

using namespace ttmi;

extern "C" {

int ttmi_attention_with_probs(const void* q, const void* k_past, const void* v_past, int64_t past, const void* k, const void* v,
                              void* k_out, void* v_out, const float* mask, int mask_per_query, void* probs, void* out,
                              int64_t batch, int64_t heads, int64_t queries, int64_t keys, int64_t head_dim, float scale,
                              int dtype, void* stream) {
  TTMI_REQUIRE(q && k && v && probs && out, "null tensor");
  TTMI_REQUIRE(head_dim == kD, "built for head_dim 64");
  TTMI_REQUIRE(batch > 0 && heads > 0 && queries > 0 && batch * heads < 65536 && queries < (1 << 24), "bad shape");
  TTMI_REQUIRE(keys > 0 && keys <= TTMI_PROBS_MAX_KEYS, "1 to TTMI_PROBS_MAX_KEYS keys");
  TTMI_REQUIRE(past >= 0 && past < keys && (past == 0 || (k_past && v_past)), "past keys need their tensors and at least one new key");
  TTMI_REQUIRE((k_out == nullptr) == (v_out == nullptr), "the grown cache is both tensors or none");
  uintptr_t bits = 0;
  for (const void* x : {q, k_past, v_past, k, v, (const void*)k_out, (const void*)v_out, (const void*)out}) bits |= reinterpret_cast<uintptr_t>(x);
  TTMI_REQUIRE((bits & 15) == 0, "tensors must be 16-byte aligned");
  const ProbsArgs p{q, k_past, v_past, k, v, k_out, v_out, probs, out, mask, (int)heads, (int)queries, (int)past, (int)keys, mask_per_query, scale};
  TTMI_DISPATCH_FLOAT(dtype, T, return launch_attention_probs<T>(p, batch, (hipStream_t)stream));
  return 0;
}

}  // extern "C"
