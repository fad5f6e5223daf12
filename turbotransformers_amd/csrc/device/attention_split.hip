// Fused self-attention for head_dim 64 where there are few sequences: the keys of a head are split over the wavefronts of a
// workgroup.  Same formulas and matrix instructions as attention.hip (fp16 / bf16) and attention_f32.hip, which describe
// them; what differs is the split of the work.
//
// Those kernels give a wavefront 32 queries and ALL keys of the head, staged through LDS and shared by the four or eight
// wavefronts of the workgroup: the fewest bytes per query, but one sequence of 128 tokens is then 12 workgroups on 256 CUs,
// each a serial chain of key tiles (fp32: 13.7 us, of which the matrix pipes need 0.4).  Here a workgroup owns 32 queries,
// its NW wavefronts take every NW-th block of 32 keys, and each keeps its own running maximum, sum and output block; K and
// V fragments come straight from global memory in the layout of the matrix instruction (a 16-byte piece of a K row or of a
// V^T row per lane), the next block's while this one is multiplied, so the K loop has neither LDS nor barriers.  At the end the NW partial results meet in LDS and are combined
// with the weights 2^(m_w - max m).
// One sequence, 12 heads, us per launch before / after: fp16 387 tokens 10.6 / 7.0, fp32 128 tokens 12.7 / 6.3 (1.5 of each
// is the launch, 1 the first loads; fp32 then runs 64 matrix instructions of 64 cycles in a chain per block of keys).
//
// With the output projection (PROJECT): up to some dozens of rows that product is a launch of its own for a few microseconds of
// waiting.  A workgroup here has the context of 32 queries of one head in its hands, and its wavefronts multiply it by the head's 64
// columns of w, whose loads were sent in front of the attention: an fp32 slice per head, added up by the kernel that
// normalises.  128 columns a workgroup (NW = 4; blockIdx.z), each computing the attention again: 72 workgroups for 10 rows of 12 heads
// are 5.2 us, the two launches they replace 4.3 and 4.0.
#include "attention_common.h"

namespace ttmi {
namespace {

constexpr int kQ = 32, kKeys = 32;  // queries per workgroup, keys per block

// The output projection behind the core (PROJECT): the rows of w (and columns of the product) that the workgroups of one blockIdx.z take.
template <typename T>
struct Projection {
  const T* w;        // [n, n], n = heads * 64
  float* partial;    // [heads, batch * seq, n]
};

// V is [B,h,d,v_pitch]; READS: Ahead or NothingAhead
template <typename T, int NW, bool PROJECT, typename READS>
__global__ __launch_bounds__(NW * 64) void split_attention_kernel(const T* __restrict__ q, const T* __restrict__ k,
                                                                  const T* __restrict__ v, const float* __restrict__ mask,
                                                                  T* __restrict__ out, int heads, int seq, int v_pitch, float scale_log2e, float inv_scale,
                                                                  float* __restrict__ absmax, const READS ahead, const Projection<T> proj) {
  constexpr int KPC = 16 / (int)sizeof(T);   // elements per 16-byte piece
  constexpr int PIECES = kD / KPC / 2;       // pieces of a row per lane: 4 (16-bit), 8 (fp32)
  constexpr int VPIECES = 4 * (int)sizeof(T) / 2;  // pieces of V per lane and block: two halves of d, 32 keys
  constexpr int PITCH = kD + 4;
  __shared__ __align__(16) float part[NW][kQ][PITCH];
  __shared__ float stat[2][NW][kQ];  // m and l of every wavefront's share
  __shared__ float red[NW];
  __shared__ __align__(16) T ctx[PROJECT ? kQ : 1][kD + 8];

  if (has_read_ahead(ahead)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int bh = blockIdx.y, b = bh / heads, head = bh - b * heads;
  const int q0 = blockIdx.x * kQ;
  const T* qb = q + (int64_t)bh * seq * kD;
  const T* kb = k + (int64_t)bh * seq * kD;
  const T* vb = v + (int64_t)bh * kD * v_pitch;
  const float* mb = mask != nullptr ? mask + (int64_t)b * seq : nullptr;

  // the wavefront's 32 columns of the projection; its weights arrive during the attention
  const int hidden = heads * kD, col0 = PROJECT ? (blockIdx.z * NW + wave) * 32 : 0;
  u32x4 wf[PROJECT ? 4 : 1];
  if constexpr (PROJECT) {
    const T* row = proj.w + (int64_t)min(col0 + lrow, hidden - 1) * hidden + head * kD + lhalf * 8;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) wf[kk] = *reinterpret_cast<const u32x4*>(row + kk * 16);
  }

  u32x4 qf[PIECES];
  {
    const T* row = qb + (int64_t)min(q0 + lrow, seq - 1) * kD + lhalf * KPC;  // rows past the end repeat the last one
#pragma unroll
    for (int kk = 0; kk < PIECES; ++kk) qf[kk] = *reinterpret_cast<const u32x4*>(row + 2 * kk * KPC);
  }

  struct Block {
    u32x4 kf[PIECES];
    u32x4 vf[VPIECES];
    uint32_t mk;  // of key lrow
  };
  const int blocks = (seq + kKeys - 1) / kKeys;
  // Keys past the end repeat valid ones; they carry a mask of -inf, so their probability is 0.
  auto load = [&](int blk, Block& x) __attribute__((always_inline)) {
    const int key0 = blk * kKeys;
    const T* row = kb + (int64_t)min(key0 + lrow, seq - 1) * kD + lhalf * KPC;
#pragma unroll
    for (int kk = 0; kk < PIECES; ++kk) x.kf[kk] = *reinterpret_cast<const u32x4*>(row + 2 * kk * KPC);
    x.mk = mb != nullptr ? load_mask(mb + min(key0 + lrow, seq - 1)) : 0u;
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const T* vr = vb + (int64_t)(t * 32 + lrow) * v_pitch;
          const int c = key0 + 16 * kk + 4 * lhalf;
          const u32x2 lo = *reinterpret_cast<const u32x2*>(vr + min(c, v_pitch - 4)), hi = *reinterpret_cast<const u32x2*>(vr + min(c + 8, v_pitch - 4));
          x.vf[2 * t + kk] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          x.vf[4 * t + g] = *reinterpret_cast<const u32x4*>(vb + (int64_t)(t * 32 + lrow) * v_pitch + min(key0 + 8 * g + 4 * lhalf, v_pitch - 4));
    }
  };

  floatx16 ot[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) ot[t][e] = 0.f;
  float m_run = -kFarthestScore, l_run = 0.f;

  auto compute = [&](int blk, Block& x) __attribute__((always_inline)) {
    const int key0 = blk * kKeys;
    const bool ragged = key0 + kKeys > seq;  // uniform
    // scores start from mask / scale of their key: [mask | 0] . [1 | 1], exact in fp32
    floatx16 st;
#pragma unroll
    for (int e = 0; e < 16; ++e) st[e] = 0.f;
    {
      const float mk = key0 + lrow < seq ? mask_in_scores(x.mk, inv_scale) : -__builtin_inff();
      st = __builtin_amdgcn_mfma_f32_32x32x2f32(lhalf == 0 ? mk : 0.f, 1.f, st, 0, 0, 0);
    }
#pragma unroll
    for (int kk = 0; kk < PIECES; ++kk) st = mma32<T>(x.kf[kk], qf[kk], st);
    float mx = st[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, st[e]);
    {
      const LanePair sw = swap_halves(mx);
      mx = fmaxf(sw.a, sw.b);
    }
    const float m_new = fmaxf(m_run, mx);
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2e);
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) ot[t][e] *= alpha;
    const float neg_m = relative_scores(st, m_run, scale_log2e);
    // V^T past the last key may hold anything: 0 * NaN would reach the output.  (Here and not in front of the first product, which
    // would then wait for V.)
    if (ragged) {
#pragma unroll
      for (int p = 0; p < VPIECES; ++p)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if constexpr (sizeof(T) == 2) {
            const int key = key0 + 16 * (p & 1) + 8 * (w >> 1) + 4 * lhalf + 2 * (w & 1);
            if (key >= seq) x.vf[p][w] = 0u;
            else if (key + 1 >= seq) x.vf[p][w] &= 0xffffu;
          } else {
            if (key0 + 8 * (p & 3) + 4 * lhalf + w >= seq) x.vf[p][w] = 0u;
          }
        }
    }
    float psum = 0.f;
    if constexpr (sizeof(T) == 2) {
      u32x4 pf[2];
#pragma unroll
      for (int w = 0; w < 8; ++w) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * w], scale_log2e, neg_m));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[2 * w + 1], scale_log2e, neg_m));
        const uint32_t pair = pack2<T>(p0, p1);
        pf[w >> 2][w & 3] = pair;
        psum = add_pair<T>(pair, psum);
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int t = 0; t < 2; ++t) ot[t] = mma32<T>(x.vf[2 * t + kk], pf[kk], ot[t]);
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        st[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[e], scale_log2e, neg_m));
        psum += st[e];
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u32x4 pf;
#pragma unroll
        for (int i = 0; i < 4; ++i) pf[i] = __builtin_bit_cast(uint32_t, (float)st[4 * g + i]);
#pragma unroll
        for (int t = 0; t < 2; ++t) ot[t] = mma32<T>(x.vf[4 * t + g], pf, ot[t]);
      }
    }
    l_run = l_run * alpha + psum;
  };

  {
    Block x, y;
    int blk = wave;
    if (blk < blocks) load(blk, x);
    while (blk < blocks) {
      if (blk + NW < blocks) load(blk + NW, y);
      compute(blk, x);
      blk += NW;
      if (blk >= blocks) break;
      if (blk + NW < blocks) load(blk + NW, x);
      compute(blk, y);
      blk += NW;
    }
  }

  // ---- the wavefronts' shares meet: ot[t][4g+i] = O[query lrow][d = 32t + 8g + 4*lhalf + i]
  l_run += __shfl_xor(l_run, 32, kWave);
  if (lhalf == 0) {
    stat[0][wave][lrow] = m_run;
    stat[1][wave][lrow] = l_run;
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<floatx4*>(&part[wave][lrow][t * 32 + 8 * g + 4 * lhalf]) =
          floatx4{ot[t][4 * g], ot[t][4 * g + 1], ot[t][4 * g + 2], ot[t][4 * g + 3]};
  __syncthreads();
  constexpr int EPT = kQ * kD / (NW * 64);  // output elements per thread: 8 or 4
  const int qi = tid / (kD / EPT), d0 = (tid % (kD / EPT)) * EPT;
  float m = -kFarthestScore;
#pragma unroll
  for (int w = 0; w < NW; ++w) m = fmaxf(m, stat[0][w][qi]);
  float l = 0.f, o[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) o[e] = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float f = __builtin_amdgcn_exp2f((stat[0][w][qi] - m) * scale_log2e);  // a share without keys has no sum
    l += f * stat[1][w][qi];
#pragma unroll
    for (int e = 0; e < EPT; e += 4) {
      const floatx4 p = *reinterpret_cast<const floatx4*>(&part[w][qi][d0 + e]);
#pragma unroll
      for (int j = 0; j < 4; ++j) o[e + j] += f * p[j];
    }
  }
  const float inv = 1.0f / l;
  if constexpr (PROJECT) {
    // the head's context, rounded as it is where it is stored, times its 64 columns of w: lane = query, four columns a register quad
    Vec<T, EPT> r;
#pragma unroll
    for (int e = 0; e < EPT; ++e) r.v[e] = from_float<T>(o[e] * inv);
    store_vec<T, EPT>(&ctx[qi][d0], r);
    __syncthreads();
    floatx16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) acc = mma32<T>(wf[kk], *reinterpret_cast<const u32x4*>(&ctx[lrow][kk * 16 + lhalf * 8]), acc);
    if (q0 + lrow < seq && col0 < hidden) {
      const int64_t tokens = (int64_t)(computing_rows(ahead) / heads) * seq;  // (the rows: batch * heads)
      float* dst = proj.partial + (head * tokens + (int64_t)b * seq + q0 + lrow) * hidden + col0 + 4 * lhalf;
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<floatx4*>(dst + 8 * g) = floatx4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    }
    return;
  }
  float amax = 0.f;
  if (q0 + qi < seq) {
    T* dst = out + ((int64_t)b * seq + q0 + qi) * (heads * kD) + head * kD + d0;
    Vec<T, EPT> r;
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const float x = o[e] * inv;
      r.v[e] = from_float<T>(x);
      amax = fmaxf(amax, fabsf(x));
    }
    if constexpr (sizeof(Vec<T, EPT>) <= 16) {
      store_vec<T, EPT>(dst, r);
    } else {
#pragma unroll
      for (int e = 0; e < EPT; e += 4) *reinterpret_cast<floatx4*>(dst + e) = floatx4{(float)r.v[e], (float)r.v[e + 1], (float)r.v[e + 2], (float)r.v[e + 3]};
    }
  }
  // Optional (dense fp32 batches): max|out| of this workgroup to its slot, as in attention_f32.hip.
  if (absmax != nullptr) {
    amax = group_max<kWave>(amax);
    if (lane == 0) red[wave] = amax;
    __syncthreads();
    const int wg = (int)(blockIdx.y * gridDim.x + blockIdx.x), wgs = (int)gridDim.x * computing_rows(ahead);
    if (tid == 0) {
      float mx = red[0];
#pragma unroll
      for (int w = 1; w < NW; ++w) mx = fmaxf(mx, red[w]);
      absmax[wg] = mx;
    }
    if (wg == 0)
      for (int i = wgs + tid; i < TTMI_ABSMAX_SLOTS; i += NW * 64) absmax[i] = 0.f;
  }
}

template <typename T>
int launch(const void* q, const void* k, const void* v, const float* mask, void* out, int64_t batch, int64_t heads,
           int64_t seq, int64_t v_pitch, float scale, float* absmax, const Ahead* ahead, hipStream_t s) {
  const unsigned width = (unsigned)ceil_div(seq, kQ), rows = (unsigned)(batch * heads);
  const unsigned more = ahead_rows(ahead, (int64_t)width * rows, width, 2 * compute_units());
  const float sl2 = scale * 1.4426950408889634f, inv_scale = 1.0f / scale;
  auto launch_reading = [&](auto waves, const auto& reads) {
    constexpr int NW = decltype(waves)::value;
    hipLaunchKernelGGL((split_attention_kernel<T, NW, false, std::decay_t<decltype(reads)>>), dim3(width, rows + more), dim3(NW * 64), 0, s, (const T*)q,
                       (const T*)k, (const T*)v, mask, (T*)out, (int)heads, (int)seq, (int)v_pitch, sl2, inv_scale, absmax, reads, Projection<T>{});
  };
  auto launch = [&](auto waves) {
    if (more == 0) return launch_reading(waves, NothingAhead{});
    Ahead read_ahead = *ahead;
    read_ahead.rows = (int)rows;
    launch_reading(waves, read_ahead);
  };
  // eight wavefronts where four would each have more than two blocks of keys
  if (seq > 4 * 2 * kKeys) launch(std::integral_constant<int, 8>{});
  else launch(std::integral_constant<int, 4>{});
  return launch_status("split_attention_kernel");
}

template <typename T>
int launch_projection(const void* q, const void* k, const void* v, const float* mask, const void* w, float* partial, int64_t batch,
                      int64_t heads, int64_t seq, int64_t v_pitch, float scale, const Ahead& ahead, hipStream_t s) {
  const float sl2 = scale * 1.4426950408889634f, inv_scale = 1.0f / scale;
  auto launch = [&](auto waves) {
    constexpr int NW = decltype(waves)::value;
    const unsigned width = (unsigned)ceil_div(seq, kQ), rows = (unsigned)(batch * heads), groups = (unsigned)ceil_div(heads * kD, NW * 32);
    const unsigned more = ahead_rows(&ahead, (int64_t)width * groups * rows, (int64_t)width * groups, 2 * compute_units());
    auto launch_reading = [&](const auto& reads) {
      hipLaunchKernelGGL((split_attention_kernel<T, NW, true, std::decay_t<decltype(reads)>>), dim3(width, rows + more, groups), dim3(NW * 64), 0, s,
                         (const T*)q, (const T*)k, (const T*)v, mask, (T*)nullptr, (int)heads, (int)seq, (int)v_pitch, sl2, inv_scale,
                         (float*)nullptr, reads, Projection<T>{(const T*)w, partial});
    };
    if (more == 0) return launch_reading(NothingAhead{});
    Ahead read_ahead = ahead;
    read_ahead.rows = (int)rows;
    launch_reading(read_ahead);
  };
  if (seq > 4 * 2 * kKeys) launch(std::integral_constant<int, 8>{});
  else launch(std::integral_constant<int, 4>{});
  return launch_status("attention_projection_kernel");
}

}  // namespace

// Arguments were checked by ttmi_fused_attention; absmax (fp32) needs seq / 32 * batch * heads workgroups to fit the slots.
int split_attention(const void* q, const void* k, const void* v, const float* mask, void* out, int64_t batch, int64_t heads,
                    int64_t seq, int64_t v_pitch, float scale, int dtype, float* absmax, const Ahead* ahead, hipStream_t s) {
  if (dtype == TTMI_F16) return launch<f16>(q, k, v, mask, out, batch, heads, seq, v_pitch, scale, nullptr, ahead, s);
  if (dtype == TTMI_BF16) return launch<bf16>(q, k, v, mask, out, batch, heads, seq, v_pitch, scale, nullptr, ahead, s);
  return launch<float>(q, k, v, mask, out, batch, heads, seq, v_pitch, scale, absmax, ahead, s);
}

}  // namespace ttmi

using namespace ttmi;

extern "C" {

int ttmi_attention_projection(const void* q, const void* k, const void* v, const float* mask, const void* w, float* partial,
                              int64_t batch, int64_t heads, int64_t seq, int64_t head_dim, int64_t v_seq_pitch, float scale, int dtype,
                              const void* const* ahead, const int64_t* ahead_bytes, int64_t count, void* stream) {
  TTMI_REQUIRE(q && k && v && w && partial, "null tensor");
  TTMI_REQUIRE(head_dim == kD, "the attention projection is built for head_dim 64");
  TTMI_REQUIRE(dtype == TTMI_F16 || dtype == TTMI_BF16, "the attention projection is built for fp16 / bf16");
  TTMI_REQUIRE(batch > 0 && heads > 0 && seq > 0 && batch * heads < 65536 && heads < 65536 && seq < (1 << 24), "bad shape");
  TTMI_REQUIRE(v_seq_pitch >= seq && v_seq_pitch % 8 == 0 && v_seq_pitch < (1 << 24), "v_seq_pitch must be a multiple of 8 that is >= seq");
  TTMI_REQUIRE(scale > 0.f, "scale must be positive");
  const uintptr_t bits = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                         reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(partial);
  TTMI_REQUIRE((bits & 15) == 0, "tensors must be 16-byte aligned");
  Ahead ranges{};
  const int rc = ahead_ranges(ahead, ahead_bytes, count, &ranges);
  if (rc != 0) return rc;
  if (dtype == TTMI_F16) return launch_projection<f16>(q, k, v, mask, w, partial, batch, heads, seq, v_seq_pitch, scale, ranges, (hipStream_t)stream);
  return launch_projection<bf16>(q, k, v, mask, w, partial, batch, heads, seq, v_seq_pitch, scale, ranges, (hipStream_t)stream);
}

}  // extern "C"
