// Fused self-attention for head_dim 64 in fp32:  out = softmax(scale * Q K^T + mask) V  in one kernel, the fp32
// counterpart of attention.hip (which serves fp16 / bf16).  It replaces the batch_gemm3 -> ApplyMaskAndSoftmax ->
// batch_gemm4 -> TransposeForScore chain of layers/multi_headed_attention.cpp:323-354 when the caller does not ask for
// the probabilities: the [B,h,S,S] scores, written and read twice by that chain, never reach HBM.
//
// Same formulation as the 16-bit kernel.  Scores are computed TRANSPOSED,
//     St[key, query] = K_tile[key, :] . Q[query, :]      (A = K from LDS, B = Q from registers)
// so a lane holds one query column and 16 key rows of a 32-key sub-tile; the online-softmax statistics are lane-local
// plus one exchange between the half-wavefronts, and the probabilities, still in the accumulator registers, are the B operand of
//     Ot[d, query] += Vt[d, keys] . Pt[keys, query]      (A = V^T from LDS, B = P from registers)
// with the keys that a lane holds given to it in V^T as well.  exp is exp2 with scale*log2(e) folded into the argument, the
// additive mask (divided by the scale) seeds the score accumulators.
// Both products run on v_mfma_f32_32x32x16_f16, three instructions for one, with Q, K, V and the probabilities split in fp16 halves
// (split_f32.h): K and V once per workgroup on their way into LDS, the others in registers.  A sub-tile is 24 instructions of 32
// cycles where the fp32 instruction needs 64 of 64, and what bounds the kernel is then the arithmetic around them.  Scores
// have an absolute error, so Q and K only need an upper limit, which depends on the scale (score_limit); a column of V has the window
// of split_f32.h.  A workgroup that meets a value outside starts again on v_mfma_f32_32x32x2_f32: there an instruction takes K index 0 from lanes 0-31 and K index 1
// from lanes 32-63, and accumulator register 4g+i of a lane in half h is key 8g + 4h + i, so keys (8g+i, 8g+4+i) are paired in
// instruction (g, i), A is the 16-byte chunk (2g+h) of a V^T row, and the head dimension is paired the same way.
// us per launch, 12 heads, fp32 instruction / halves: 20 x 100 tokens 13.6 / 10.0, 8 x 256 23.4 / 16.9, 20 x 300 74 / 43, 20 x 512 148 / 72;
// packed, 20 requests of 5 to 500 tokens 100 / 47.
//
// V may be given transposed ([B,h,d,pitch], as the QKV epilogue writes it with v_seq_pitch: its tiles are then copied)
// or row-major ([B,h,S,d]: a thread scatters its four values of a key into four V^T rows).  With cu_seqlens q,k,v are
// the padded tensors of a packed batch (S = longest sequence): keys and queries past a sequence's length are never
// read and the output is packed [sum(len), h*64].
#include <cstdlib>
#include <mutex>
#include <set>

#include "attention_common.h"
#include "split_f32.h"

namespace ttmi {

namespace {

constexpr int kBKV = 64;         // keys per LDS tile
constexpr int kRow = 256;        // bytes of a K row (64 floats) and of a V^T row (64 keys)

// 16-byte chunk `chunk` of row `row` of a tile with 256-byte rows.  The 16 lanes that the LDS serves together read one chunk
// column of 16 rows (0-3, 12-15, 20-27 of 32, or the others), and the scatter of a row-major V writes to every fourth row:
// for both the chunk index is XORed with 16 different values.
__device__ __forceinline__ int tile_off(int row, int chunk) { return row * kRow + ((chunk ^ (((row >> 2) ^ (row << 2)) & 15)) << 4); }
// Where the halves of keys 4 c ... 4 c + 3 lie in a V^T row: the keys that a lane multiplies at once (registers 8 kk ... 8 kk + 7 of
// its scores: keys 4 h + i and 8 + 4 h + i of 16) are one 16-byte chunk.
__device__ __forceinline__ int vt_chunk(int c) { return 2 * (c >> 2) + (c & 1); }
__device__ __forceinline__ int vt_half(int c) { return (c >> 1) & 1; }

// Up to this many keys the fp32 instruction it is: sums of so few products are hardly rounded, and what the halves leave of the operands is
// more.  Error against 64 bits, relative to the result (2-norms), scores of size 0.1, fp32 instruction / halves: 1 key 0 / 4.4e-8, 4 keys 6.6e-8 /
// 8.4e-8, 16 keys 9.5e-8 / 9.7e-8, 32 keys 1.2e-7 / 1.1e-7; scores of size 1, 1 key 0.9e-8 / 4.5e-8, 4 keys 1.1e-7 / 1.1e-7, 32 keys 2.4e-7 / 1.6e-7.
// It is no slower there: us per launch, 12 heads, halves / fp32 instruction on one sub-tile: 20 sequences of 10 tokens 6.3 / 5.8, of 30 6.7 /
// 6.2, 32 of 5 to 30 9.4 / 6.5.  (A form of its own for them: 31 of 20 and one of 300 tokens 18.9 here, 20.2 so.)
constexpr int kFewKeys = 32;

// The absolute values of Q and K have to stay below this for the halves to hold the scores.  What the halves leave of a product is
// 3 * 2^-22 max(|q|, 2^-14) max(|k|, 2^-14) at most (split_f32.h): besides 3 * 2^-22 of the sum of |q k|, which the fp32 instruction leaves
// as well, that is 64 * 3 * 2^-36 of the largest |q| or |k|, times the scale in an exponent: 2^-20 below this limit.  Of scales above 2^22 even
// values below 2^-14 would leave more.
inline float score_limit(float scale) { return scale <= 0x1p22f ? std::min(kSplitLargest, 256.f / scale) : 0.f; }

template <int NW>
constexpr int lds_bytes() {
  constexpr int tiles = 4 * kBKV * kRow + 2 * kBKV * 4, outb = NW * 32 * (kD + 4) * 4;
  return tiles > outb ? tiles : outb;
}

// The scores and the weighted sum of one wavefront's 32 queries (ot: not yet divided by the row sums, of which l_run holds this
// half-wavefront's share).  SPLIT: on the 16-bit matrix instructions, everything in halves (split_f32.h); the answer is whether
// a value does not fit them, the same for the whole workgroup.  Otherwise on the fp32 instruction.
template <int NW, bool VT, bool SPLIT>
__device__ __forceinline__ bool attend(char* const smem, const float* __restrict__ qb, const float* __restrict__ kb, const float* __restrict__ vb,
                                       const float* __restrict__ mask, int q0, int kv_len, int v_pitch, float scale_log2e, float inv_scale,
                                       float qk_limit, floatx16 (&ot)[2], float& l_run) {
  constexpr int kPieces = 1024 / (NW * 64);  // 16-byte pieces of a K (V^T) tile per thread: 64 rows of 16
  constexpr int kTile = kBKV * kRow;         // 16 KB
  const int tid = threadIdx.x, lane = tid & 63;
  const int lrow = lane & 31, lhalf = lane >> 5;
  const int q_len = kv_len;  // self attention: as many queries as keys

  // Q fragments: B operand of the first product.  fp32: chunk 2kk+lhalf of the lane's query row; halves: eight values of the
  // head dimension, hi and lo.
  u32x4 qf[8];
  float largest = 0.f;  // of Q and K
  {
    const int qi = q0 + lrow;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      floatx4 x[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int c = SPLIT ? 4 * kk + 2 * lhalf + j : 4 * kk + 2 * j + lhalf;
        if (qi < q_len) x[j] = *reinterpret_cast<const floatx4*>(qb + (int64_t)qi * kD + c * 4);
        else x[j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
      if constexpr (SPLIT) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float a = x[w >> 1][2 * (w & 1)], b = x[w >> 1][2 * (w & 1) + 1];
          qf[2 * kk][w] = split_hi(a, b);
          qf[2 * kk + 1][w] = split_lo(qf[2 * kk][w], a, b);
          split_max(largest, a, b);
        }
      } else {
        qf[2 * kk] = __builtin_bit_cast(u32x4, x[0]);
        qf[2 * kk + 1] = __builtin_bit_cast(u32x4, x[1]);
      }
    }
  }

  floatx16 oc[2];  // SPLIT: the products of a hi and a lo, 2^16 times too large
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) ot[t][e] = 0.f, oc[t][e] = 0.f;
  float m_run = -kFarthestScore;
  l_run = 0.f;

  // tile staging: thread -> chunk ch of rows r0 + 64*NW/16*p; global -> registers one tile ahead -> LDS.  (Of a row-major V a
  // thread takes neighbouring keys, whose halves are written together.)
  constexpr int kRowsPerPass = NW * 64 / 16;
  const int ch = tid & 15, r0 = tid >> 4;
  auto v_key = [&](int p) __attribute__((always_inline)) { return SPLIT ? (p >> 1) * (2 * kRowsPerPass) + 2 * r0 + (p & 1) : r0 + p * kRowsPerPass; };
  floatx4 kreg[kPieces], vreg[kPieces];
  float v_largest[VT ? kPieces : 4];  // of a V^T row
#pragma unroll
  for (int i = 0; i < (VT ? kPieces : 4); ++i) v_largest[i] = 0.f;
  uint32_t mreg = 0;

  auto load_tile = [&](int tile) __attribute__((always_inline)) {
    const int key0 = tile * kBKV;
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
      const int r = r0 + p * kRowsPerPass;
      kreg[p] = *reinterpret_cast<const floatx4*>(kb + (int64_t)min(key0 + r, kv_len - 1) * kD + ch * 4);
      if constexpr (VT)  // row r of V^T, keys 4ch.. of the tile
        vreg[p] = *reinterpret_cast<const floatx4*>(vb + (int64_t)r * v_pitch + min(key0 + ch * 4, v_pitch - 4));
      else  // a key of the tile, head dimensions 4ch..
        vreg[p] = *reinterpret_cast<const floatx4*>(vb + (int64_t)min(key0 + v_key(p), kv_len - 1) * kD + ch * 4);
    }
    if (tid < kBKV && mask != nullptr) mreg = load_mask(mask + min(key0 + tid, kv_len - 1));
  };
  auto store_tile = [&](int tile, int stage) __attribute__((always_inline)) {
    char* const kt = smem + stage * kTile;
    char* const vt = smem + 2 * kTile + stage * kTile;
    const int nv = kv_len - (tile * kBKV + ch * 4);  // valid keys in this thread's V^T chunk
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
      const int r = r0 + p * kRowsPerPass;
      const floatx4 kx = kreg[p];
      floatx4 x = vreg[p];
      if constexpr (VT) {
        if (nv < 4) {  // only in the last tile: keys past the end may hold anything, zero them
#pragma unroll
          for (int w = 0; w < 4; ++w)
            if (w >= nv) x[w] = 0.f;
        }
      } else if (tile * kBKV + v_key(p) >= kv_len) {
        x = floatx4{0.f, 0.f, 0.f, 0.f};
      }
      if constexpr (SPLIT) {
        const uint2 kh = make_uint2(split_hi(kx[0], kx[1]), split_hi(kx[2], kx[3]));
        char* const at = kt + tile_off(r, ch >> 1) + (ch & 1) * 8;
        *reinterpret_cast<uint2*>(at) = kh;
        *reinterpret_cast<uint2*>(kt + (tile_off(r, (ch >> 1) ^ 8) + (ch & 1) * 8)) = make_uint2(split_lo(kh.x, kx[0], kx[1]), split_lo(kh.y, kx[2], kx[3]));
        split_max(largest, kx[0], kx[1]);
        split_max(largest, kx[2], kx[3]);
        if constexpr (VT) {
          const uint2 vh = make_uint2(split_hi(x[0], x[1]), split_hi(x[2], x[3]));
          *reinterpret_cast<uint2*>(vt + tile_off(r, vt_chunk(ch)) + vt_half(ch) * 8) = vh;
          *reinterpret_cast<uint2*>(vt + tile_off(r, vt_chunk(ch) ^ 8) + vt_half(ch) * 8) = make_uint2(split_lo(vh.x, x[0], x[1]), split_lo(vh.y, x[2], x[3]));
          split_max(v_largest[p], x[0], x[1]);
          split_max(v_largest[p], x[2], x[3]);
        } else if (p % 2 == 1) {  // V^T[d = 4ch + w][two keys]
          floatx4 y = vreg[p - 1];
          if (tile * kBKV + v_key(p - 1) >= kv_len) y = floatx4{0.f, 0.f, 0.f, 0.f};
          const int key = v_key(p - 1), c = key >> 2;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const uint32_t h = split_hi(y[w], x[w]);
            char* const row = vt + vt_half(c) * 8 + (key & 2) * 2;
            *reinterpret_cast<uint32_t*>(row + tile_off(ch * 4 + w, vt_chunk(c))) = h;
            *reinterpret_cast<uint32_t*>(row + tile_off(ch * 4 + w, vt_chunk(c) ^ 8)) = split_lo(h, y[w], x[w]);
            split_max(v_largest[w], y[w], x[w]);
          }
        }
      } else {
        *reinterpret_cast<floatx4*>(kt + tile_off(r, ch)) = kx;
        if constexpr (VT) {
          *reinterpret_cast<floatx4*>(vt + tile_off(r, ch)) = x;
        } else {  // V^T[d = 4ch + w][key r]: float r % 4 of chunk r / 4 of row d
#pragma unroll
          for (int w = 0; w < 4; ++w) *reinterpret_cast<float*>(vt + tile_off(ch * 4 + w, r >> 2) + (r & 3) * 4) = x[w];
        }
      }
    }
    if (tid < kBKV)
      reinterpret_cast<float*>(smem + 4 * kTile)[stage * kBKV + tid] =
          tile * kBKV + tid < kv_len ? mask_in_scores(mreg, inv_scale) : -__builtin_inff();
  };

  // One 64-key tile from LDS stage STAGE.  m_run is kept in raw score units; p = exp2(s*c - m*c), c = scale*log2(e).
  auto compute_tile = [&](auto stage_c) {
    constexpr int STAGE = decltype(stage_c)::value;
    const char* kt = smem + STAGE * kTile;
    const char* vt = smem + 2 * kTile + STAGE * kTile;
    const float* mk = reinterpret_cast<const float*>(smem + 4 * kTile) + STAGE * kBKV;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {  // two 32-key sub-tiles
      if (!SPLIT && sub == 1 && kv_len <= kFewKeys) break;
      const int sk = sub * 32;
      // st[4g+i] = score of (key sk + 8g + 4*lhalf + i, query lrow), seeded with mask/scale
      floatx16 st;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 mv = *reinterpret_cast<const float4*>(mk + sk + 8 * g + 4 * lhalf);
        st[4 * g] = mv.x, st[4 * g + 1] = mv.y, st[4 * g + 2] = mv.z, st[4 * g + 3] = mv.w;
      }
      if constexpr (SPLIT) {
        floatx16 sc;
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[e] = 0.f;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const u32x4 kh = *reinterpret_cast<const u32x4*>(kt + tile_off(sk + lrow, 2 * kk + lhalf));
          const u32x4 kl = *reinterpret_cast<const u32x4*>(kt + tile_off(sk + lrow, (2 * kk + lhalf) ^ 8));
          sc = mma32<f16>(kh, qf[2 * kk + 1], sc);
          st = mma32<f16>(kh, qf[2 * kk], st);
          sc = mma32<f16>(kl, qf[2 * kk], sc);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) st[e] = __builtin_fmaf(sc[e], 1.f / kSplitScale, st[e]);
      } else {
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
          const floatx4 kf = *reinterpret_cast<const floatx4*>(kt + tile_off(sk + lrow, 2 * kk + lhalf));
          st = mma32<float>(kf, __builtin_bit_cast(floatx4, qf[kk]), st);
        }
      }
      float mx = st[0];
#pragma unroll
      for (int e = 1; e < 16; ++e) mx = fmaxf(mx, st[e]);
      {
        // the other half-wavefront holds the remaining 16 keys of this query
        const LanePair sw = swap_halves(mx);
        // fp32: any reference point near the maximum does, since the sums are rounded relative to their own size.  The half that holds
        // the first keys gives it unless the other one's exponentials would leave the fp32 range (2^64 leaves 2^63 to sum).
        // Halves: the maximum itself, so that no probability exceeds 1.
        if constexpr (SPLIT) mx = fmaxf(sw.a, sw.b);
        else mx = (sw.b - sw.a) * scale_log2e > 64.f ? sw.b : sw.a;
      }
      if (__any(mx > m_run)) {
        const float m_new = fmaxf(m_run, mx);
        const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * scale_log2e);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            ot[t][e] *= alpha;
            if constexpr (SPLIT) oc[t][e] *= alpha;
          }
      }
      const float neg_m = relative_scores(st, m_run, scale_log2e);
      float psum = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        st[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[e], scale_log2e, neg_m));
        psum += st[e];
      }
      l_run += psum;
      if constexpr (SPLIT) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          u32x4 ph, pl;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const float a = st[8 * kk + 2 * w], b = st[8 * kk + 2 * w + 1];
            ph[w] = split_hi(a, b);
            pl[w] = split_lo(ph[w], a, b);
          }
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int c = 2 * (sk / 16 + kk) + lhalf;
            const u32x4 vh = *reinterpret_cast<const u32x4*>(vt + tile_off(t * 32 + lrow, c));
            const u32x4 vl = *reinterpret_cast<const u32x4*>(vt + tile_off(t * 32 + lrow, c ^ 8));
            oc[t] = mma32<f16>(vh, pl, oc[t]);
            ot[t] = mma32<f16>(vh, ph, ot[t]);
            oc[t] = mma32<f16>(vl, ph, oc[t]);
          }
        }
      } else {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const floatx4 pf{st[4 * g], st[4 * g + 1], st[4 * g + 2], st[4 * g + 3]};
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const floatx4 vf = *reinterpret_cast<const floatx4*>(vt + tile_off(t * 32 + lrow, sk / 4 + 2 * g + lhalf));
            ot[t] = mma32<float>(vf, pf, ot[t]);
          }
        }
      }
    }
  };

  const int tiles = (kv_len + kBKV - 1) / kBKV;
  const bool wave_active = q0 < q_len;
  load_tile(0);
  store_tile(0, 0);
  __syncthreads();
  for (int tile = 0; tile < tiles; tile += 2) {
    if (tile + 1 < tiles) load_tile(tile + 1);
    if (wave_active) compute_tile(std::integral_constant<int, 0>{});
    if (tile + 1 < tiles) store_tile(tile + 1, 1);
    __syncthreads();
    if (tile + 1 >= tiles) break;
    if (tile + 2 < tiles) load_tile(tile + 2);
    if (wave_active) compute_tile(std::integral_constant<int, 1>{});
    if (tile + 2 < tiles) store_tile(tile + 2, 0);
    __syncthreads();
  }
  if constexpr (SPLIT) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) ot[t][e] = __builtin_fmaf(oc[t][e], 1.f / kSplitScale, ot[t][e]);
    bool outside = largest >= qk_limit;
    if constexpr (VT) {
#pragma unroll
      for (int p = 0; p < kPieces; ++p) outside = outside || split_outside(group_max<16>(v_largest[p]));
    } else {  // (the tiles have been read: the front of LDS holds the maxima of every four keys' share)
      float* const part = reinterpret_cast<float*>(smem);
#pragma unroll
      for (int w = 0; w < 4; ++w) part[r0 * kD + ch * 4 + w] = v_largest[w];
      __syncthreads();
      if (tid < kD) {
        float top = 0.f;
        for (int r = 0; r < kRowsPerPass; ++r) top = fmaxf(top, part[r * kD + tid]);
        outside = outside || split_outside(top);
      }
    }
    return __syncthreads_or(outside) != 0;
  }
  return false;
}

template <int NW, bool VT, bool PACKED, bool SPLIT>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2))) void fused_attention_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ mask,
    float* __restrict__ out, const int32_t* __restrict__ cu, int heads, int seq, int v_pitch, float scale_log2e,
    float inv_scale, float qk_limit, bool through, float* __restrict__ absmax) {
  static_assert(NW == 4 || NW == 8, "four or eight wavefronts");
  constexpr int kBQ = NW * 32;  // queries per workgroup
  // dynamic LDS (lds_bytes<NW>(), more than the 64 KB a kernel gets without asking):
  // [2 x K tile | 2 x V^T tile | 2 x mask]; the front is reused for the output tile
  extern __shared__ __align__(16) char smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 31, lhalf = lane >> 5;
  // A packed batch: sequence by sequence (y) and there block by block, all heads of a block side by side (x; the workgroups of
  // an XCD are then a mixture of first and last blocks).  See longest_first().
  const int major = (PACKED ? blockIdx.x : blockIdx.y) / heads, head = (PACKED ? blockIdx.x : blockIdx.y) - major * heads;
  const int block = PACKED ? major : blockIdx.x;
  int b = PACKED ? blockIdx.y : major;
  if (PACKED && seq > kOrderMinLength && gridDim.x * gridDim.y > kOrderMinWorkgroups) b = __builtin_amdgcn_readfirstlane(longest_first(cu, gridDim.y, b, seq));
  const int bh = b * heads + head;
  const int q0 = block * kBQ + wave * 32;
  int kv_len = seq, out_row0 = b * seq;
  if (PACKED) {
    kv_len = cu[b + 1] - cu[b];
    out_row0 = cu[b];
    if (block * kBQ >= kv_len) return;  // whole workgroup is padding
  }
  const int q_len = kv_len;  // self attention: as many queries as keys

  const float* qb = q + (int64_t)bh * seq * kD;
  const float* kb = k + (int64_t)bh * seq * kD;
  const float* vb = v + (int64_t)bh * kD * (VT ? v_pitch : seq);
  const float* mb = mask != nullptr ? mask + (int64_t)b * seq : nullptr;
  floatx16 ot[2];
  float l_run;
  bool again = true;
  if constexpr (SPLIT)
    if (kv_len > kFewKeys) again = attend<NW, VT, true>(smem, qb, kb, vb, mb, q0, kv_len, v_pitch, scale_log2e, inv_scale, qk_limit, ot, l_run);
  if (again) attend<NW, VT, false>(smem, qb, kb, vb, mb, q0, kv_len, v_pitch, scale_log2e, inv_scale, qk_limit, ot, l_run);

  // normalise and write: ot[t][4g+i] = O[query lrow][d = 32t + 8g + 4*lhalf + i]
  const float l_tot = l_run + __shfl_xor(l_run, 32, kWave);
  const float inv = 1.0f / l_tot;
  // stage the wavefront's 32 x 64 tile in LDS (every wavefront is past the last tile barrier) to store 256-byte rows
  float* stage_o = reinterpret_cast<float*>(smem) + wave * (32 * (kD + 4));
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const floatx4 c{ot[t][4 * g] * inv, ot[t][4 * g + 1] * inv, ot[t][4 * g + 2] * inv, ot[t][4 * g + 3] * inv};
      *reinterpret_cast<floatx4*>(stage_o + lrow * (kD + 4) + t * 32 + 8 * g + 4 * lhalf) = c;
    }
  const int hd = heads * kD;
  float amax = 0.f;
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const int r = p * 4 + (lane >> 4), cchunk = lane & 15;
    const int qi = q0 + r;
    if (qi < q_len) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(stage_o + r * (kD + 4) + cchunk * 4);
      float* const to = out + ((int64_t)out_row0 + qi) * hd + head * kD + cchunk * 4;
      if (through) store_through(to, x);
      else *reinterpret_cast<floatx4*>(to) = x;
      amax = fmaxf(fmaxf(amax, fmaxf(fabsf(x[0]), fabsf(x[1]))), fmaxf(fabsf(x[2]), fabsf(x[3])));
    }
  }
  // Optional (dense batches): max|out| of this workgroup to its slot, for the int8 Linear that quantises `out` next;
  // workgroup 0 zeroes the slots no workgroup owns, so every slot is written by every launch.
  if (absmax != nullptr) {
    amax = group_max<kWave>(amax);
    __syncthreads();  // every wavefront is done with its share of the output stage
    float* red = reinterpret_cast<float*>(smem);
    if (lane == 0) red[wave] = amax;
    __syncthreads();
    const int wg = (int)(blockIdx.y * gridDim.x + blockIdx.x), wgs = (int)(gridDim.x * gridDim.y);
    if (tid == 0) {
      float m = red[0];
#pragma unroll
      for (int w = 1; w < NW; ++w) m = fmaxf(m, red[w]);
      absmax[wg] = m;
    }
    if (wg == 0)
      for (int i = wgs + tid; i < TTMI_ABSMAX_SLOTS; i += NW * 64) absmax[i] = 0.f;
  }
}

}  // namespace

// Launch; arguments were checked by ttmi_fused_attention.
int fused_attention_f32(const float* q, const float* k, const float* v, const float* mask, float* out, const int32_t* cu,
                        int64_t batch, int64_t heads, int64_t seq, int64_t v_seq_pitch, float scale, int nw, bool through,
                        float* absmax, hipStream_t s) {
  dim3 grid((unsigned)ceil_div(seq, nw * 32), (unsigned)(batch * heads));
  if (cu != nullptr) {  // blocks and heads in one row, see the kernel
    TTMI_REQUIRE((int64_t)grid.x * grid.y < (1ll << 31), "attention grid too large");
    grid = dim3((unsigned)(grid.x * heads), (unsigned)batch);
  }
  const float sl2 = scale * 1.4426950408889634f, inv_scale = 1.0f / scale, qk_limit = score_limit(scale);
  // more than 64 KB of dynamic LDS: the limit is raised once per kernel and device
  auto launch = [&](auto kern, int threads, int lds) -> int {
    static std::mutex mu;
    static std::set<std::pair<const void*, int>> done;
    int dev = 0;
    TTMI_HIP(hipGetDevice(&dev));
    {
      std::lock_guard<std::mutex> lock(mu);
      const void* fn = reinterpret_cast<const void*>(kern);
      if (done.count({fn, dev}) == 0) {
        TTMI_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        done.insert({fn, dev});
      }
    }
    hipLaunchKernelGGL(kern, grid, dim3(threads), lds, s, q, k, v, mask, out, cu, (int)heads, (int)seq, (int)v_seq_pitch, sl2,
                       inv_scale, qk_limit, through, absmax);
    return 0;
  };
  const bool vt = v_seq_pitch > 0, packed = cu != nullptr;
  int rc = 0;
#define TTMI_FA32_CASE(NW, VT, PACKED, SPLIT) rc = launch(&fused_attention_f32_kernel<NW, VT, PACKED, SPLIT>, NW * 64, lds_bytes<NW>())
#define TTMI_FA32_WAVES(VT, PACKED, SPLIT)          \
  do {                                              \
    if (nw == 8) TTMI_FA32_CASE(8, VT, PACKED, SPLIT); \
    else TTMI_FA32_CASE(4, VT, PACKED, SPLIT);         \
  } while (0)
  // A dense batch with V row-major is what the quantised layers pass: they round the result to 8 bits, which turns a difference in
  // the last bit into a whole step, so it keeps the fp32 instruction.
  if (vt && packed) TTMI_FA32_WAVES(true, true, true);
  else if (vt) TTMI_FA32_WAVES(true, false, true);
  else if (packed) TTMI_FA32_WAVES(false, true, true);
  else TTMI_FA32_WAVES(false, false, false);
#undef TTMI_FA32_WAVES
#undef TTMI_FA32_CASE
  if (rc != 0) return rc;
  return launch_status("fused_attention_f32_kernel");
}

}  // namespace ttmi
