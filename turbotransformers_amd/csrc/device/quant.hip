// Small kernels around the int8 GEMM (dynamic per-tensor activation quantisation and the
// fp32 dequant+bias epilogue) and the per-token row map of a packed (smart) batch.
#include "common.h"

namespace ttmi {

// max|x| in two steps without atomics or a cleared cell: every workgroup of absmax_kernel writes the
// maximum of its share to partial[blockIdx.x]; every workgroup of quantize_kernel then reduces those (at
// most kMaxPartials) values itself before it quantises its share.  Results do not depend on scheduling.
constexpr int kMaxPartials = 512;

__device__ __forceinline__ float block_max_256(float mx, float* red) {
  mx = group_max<kWave>(mx);
  if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = mx;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__global__ __launch_bounds__(256) void absmax_kernel(const float* __restrict__ x, int64_t n, float* __restrict__ partial) {
  __shared__ float red[4];
  float mx = 0.f;
  int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * 256;
  if ((reinterpret_cast<uintptr_t>(x) & 15) == 0) {  // 16-byte loads over the aligned body
    const int64_t n4 = n / 4;
    for (int64_t j = i; j < n4; j += stride) {
      const float4 v = reinterpret_cast<const float4*>(x)[j];
      mx = fmaxf(fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
    }
    i += n4 * 4;
  }
  for (; i < n; i += stride) mx = fmaxf(mx, fabsf(x[i]));
  mx = block_max_256(mx, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = mx;
}

// rint(x / scale) by the reciprocal that all elements share: q = RN(x y), then RN(q + (x - scale q) y), the correction step of
// Markstein's division; three instructions where the compiler's division of two fp32 numbers takes a dozen, which made the
// kernel as long as its traffic.  The remainder is exact while it stays out of the subnormal numbers, so what is rounded is
// x / scale but for some 2^-24 of an ulp, and the integer can differ from that of the division only next to a half-integer.  There
// both were compared for every mantissa of the scale (127 half-integers, the nine floats around each): none differs, at scales
// down to 2^-100; at 2^-104 two of 9.6e9 do, at 2^-119 one in 80000.
// inv_scale = 0: the scale is out of the range in which that holds, and the division is spelled out.
__device__ __forceinline__ float shared_inverse(float scale) { return scale > 0x1p-96f && scale < 0x1p120f ? 1.0f / scale : 0.f; }
__device__ __forceinline__ int quantize_one(float x, float scale, float inv_scale) {
  float r;
  if (inv_scale != 0.f) {
    const float q = x * inv_scale;
    r = rintf(__builtin_fmaf(__builtin_fmaf(-scale, q, x), inv_scale, q));  // round half to even
  } else {
    r = rintf(x / scale);
  }
  r = fminf(fmaxf(r, -127.f), 127.f);
  return (int)r;
}

// partial: `partials` per-workgroup maxima of |x|, written by absmax_kernel (then scale_dev + 2) or by the kernel
// that produced x.
// A workgroup quantises VECS * 1024 elements.  Bound by the traffic of x, and for a few MB by its waits: the elements are
// requested before the maxima are reduced (2560 x 768: 4.1 -> 3.4 us).  Four 16-byte loads per lane from 2 MiB of values on
// (2560 x 3072: 8.4 us with one, 7.2), two from 512 Ki to there, where four leave a second round of workgroups half empty, one
// below that, where the lane's own chain counts.  us a forward of base, passes of 512 Ki to 2 Mi values with four / one / two: 1 x 200 tokens
// 824 / 815 / 814, 4 x 128 774 / 777 / 773, 10 x 100 889 / 874 / 873, 16 x 100 1002 / 1001 / 986, 13 x 160 1291 / 1306 / 1289, 20 x 128 1159 / 1181 /
// 1154; two for the passes of 2 MiB and more as well: 20 x 128 1179.
template <int VECS, bool THROUGH = false>
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ x, int8_t* __restrict__ q,
                                                       float* __restrict__ scale_dev, const float* __restrict__ partial,
                                                       int partials, int64_t n) {
  __shared__ float red[4];
  const bool vec = ((reinterpret_cast<uintptr_t>(x) & 15) | (reinterpret_cast<uintptr_t>(q) & 3)) == 0;
  const int64_t n4 = vec ? n / 4 : 0;
  const int64_t first = blockIdx.x * (int64_t)(256 * VECS) + threadIdx.x;
  float4 v[VECS];
#pragma unroll
  for (int u = 0; u < VECS; ++u) {
    v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (first + u * 256 < n4) v[u] = reinterpret_cast<const float4*>(x)[first + u * 256];
  }
  float mx = 0.f;
  for (int p = threadIdx.x; p < partials; p += 256) mx = fmaxf(mx, partial[p]);
  mx = block_max_256(mx, red);
  const float scale = mx > 0.f ? mx / 127.0f : 1.0f;
  const float inv_scale = shared_inverse(scale);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    scale_dev[0] = scale;
    scale_dev[1] = mx;
  }
#pragma unroll
  for (int u = 0; u < VECS; ++u)
    if (first + u * 256 < n4) {
      const uint32_t four =
          (uint32_t)(quantize_one(v[u].x, scale, inv_scale) & 255) | ((uint32_t)(quantize_one(v[u].y, scale, inv_scale) & 255) << 8) |
          ((uint32_t)(quantize_one(v[u].z, scale, inv_scale) & 255) << 16) | ((uint32_t)(quantize_one(v[u].w, scale, inv_scale) & 255) << 24);
      uint32_t* at = reinterpret_cast<uint32_t*>(q) + first + u * 256;
      if constexpr (THROUGH) store_through(at, four);
      else *at = four;
    }
  // unaligned tensors, and the last n % 4 elements
  for (int64_t i = n4 * 4 + blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    q[i] = (int8_t)quantize_one(x[i], scale, inv_scale);
}
// rows: tokens.  What is written through is the passes of up to 12288 tokens: us a forward, all passes staying / those of the intermediate
// values through / all through: base 20 x 128 tokens (8 MB of them) 1167 / 1157 / 1157, 8 x 300 1578 / 1568 / 1568, 24 x 200 2641 / 2634 / 2634, 32 x 300 (29 MB)
// 4624 / 4605 / 4606, 16 x 512 level, large 16 x 256 4678 / 4651 / 4651, 16 x 512 (34 MB) 11233 / 11211 / 11207; 32 x 512, inputs of 13 MB and
// intermediate values of 50, 7732 all staying, 7767 the inputs through, 7790 all; 48 x 512 (19 and 75 MB) 11963, 12050, 12036; large 32 x 512
// 21077, 21115, 21125.
constexpr int64_t kMostRowsThrough = 12288;
static int launch_quantize(const float* x, int8_t* q, float* scale_dev, const float* partial, int partials, int64_t rows, int64_t n, hipStream_t s) {
  TTMI_REQUIRE(n < (1ll << 42), "too many elements");
  auto launch = [&](auto kern, int vecs) {
    hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(n, vecs * 1024)), dim3(256), 0, s, x, q, scale_dev, partial, partials, n);
  };
  if (writes_through(n) && rows <= kMostRowsThrough) launch(quantize_kernel<4, true>, 4);
  else if (writes_through(n)) launch(quantize_kernel<4>, 4);
  else if (ceil_div(n, 1024) <= 512) launch(quantize_kernel<1>, 1);
  else launch(quantize_kernel<2>, 2);
  return launch_status("quantize_kernel");
}

__global__ __launch_bounds__(256) void dequant_bias_kernel(const int32_t* __restrict__ acc,
                                                           const float* __restrict__ act_scale,
                                                           const float* __restrict__ w_scale,
                                                           const float* __restrict__ bias,
                                                           float* __restrict__ out, int64_t total, int n) {
  const float sx = act_scale[0];
  int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (; i < total; i += stride) {
#pragma clang fp contract(off)  // each product and the sum rounded, as the int8 GEMM's own dequantising store does
    const int c = (int)(i % n);
    float v = (float)acc[i] * sx * w_scale[c];
    if (bias) v = v + bias[c];
    out[i] = v;
  }
}

// Per-output-channel symmetric weight quantisation: one wavefront per row of w[N,K].
__global__ __launch_bounds__(256) void quantize_weight_rows_kernel(const float* __restrict__ w, int8_t* __restrict__ q,
                                                                   float* __restrict__ scales, int64_t n, int64_t k) {
  const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
  if (row >= n) return;
  const int lane = threadIdx.x % kWave;
  const float* wr = w + row * k;
  float mx = 0.f;
  for (int64_t c = lane; c < k; c += kWave) mx = fmaxf(mx, fabsf(wr[c]));
  mx = group_max<kWave>(mx);
  const float scale = mx > 0.f ? mx / 127.0f : 1.0f;
  if (lane == 0) scales[row] = scale;
  for (int64_t c = lane; c < k; c += kWave) {
    float r = rintf(wr[c] / scale);
    r = fminf(fmaxf(r, -127.f), 127.f);
    q[row * k + c] = (int8_t)r;
  }
}

__global__ void token_rows_kernel(const int32_t* __restrict__ cu, int batch, int max_seq, int total,
                                  int32_t* __restrict__ rows) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  int lo = 0, hi = batch;  // find b with cu[b] <= t < cu[b+1]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu[mid] <= t) lo = mid; else hi = mid;
  }
  rows[t] = lo * max_seq + (t - cu[lo]);
}

static unsigned flat_grid(int64_t n) { return (unsigned)std::min<int64_t>(ceil_div(n, 256), 256 * 16); }

}  // namespace ttmi

using namespace ttmi;

extern "C" {

int ttmi_quantize_rows_i8(const float* x, int8_t* q, float* scale_dev, int64_t m, int64_t k, void* stream) {
  TTMI_REQUIRE(x && q && scale_dev, "null tensor");
  const int64_t n = m * k;
  if (n <= 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const int partials = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 256 * 16), kMaxPartials));
  static_assert(kMaxPartials + 2 == TTMI_QUANT_SCALE_FLOATS, "scale_dev holds the scale, the maximum and the partial maxima");
  hipLaunchKernelGGL(absmax_kernel, dim3((unsigned)partials), dim3(256), 0, s, x, n, scale_dev + 2);
  return launch_quantize(x, q, scale_dev, scale_dev + 2, partials, m, n, s);
}

int ttmi_quantize_rows_i8_from_absmax(const float* x, int8_t* q, float* scale_dev, const float* absmax_slots, int64_t m,
                                      int64_t k, void* stream) {
  TTMI_REQUIRE(x && q && scale_dev && absmax_slots, "null tensor");
  const int64_t n = m * k;
  if (n <= 0) return 0;
  return launch_quantize(x, q, scale_dev, absmax_slots, TTMI_ABSMAX_SLOTS, m, n, (hipStream_t)stream);
}

int ttmi_quantize_weight_rows_i8(const float* w, int8_t* q, float* scales, int64_t n, int64_t k, void* stream) {
  TTMI_REQUIRE(w && q && scales, "null tensor");
  if (n * k <= 0) return 0;
  hipLaunchKernelGGL(quantize_weight_rows_kernel, dim3((unsigned)ceil_div(n, 4)), dim3(256), 0, (hipStream_t)stream, w, q,
                     scales, n, k);
  return launch_status("quantize_weight_rows_i8");
}

int ttmi_dequant_bias(const int32_t* acc, const float* act_scale_dev, const float* w_scale, const float* bias,
                      float* out, int64_t m, int64_t n, void* stream) {
  TTMI_REQUIRE(acc && act_scale_dev && w_scale && out, "null tensor");
  TTMI_REQUIRE(n < (1ll << 31), "N too large");
  if (m * n <= 0) return 0;
  hipLaunchKernelGGL(dequant_bias_kernel, dim3(flat_grid(m * n)), dim3(256), 0, (hipStream_t)stream, acc,
                     act_scale_dev, w_scale, bias, out, m * n, (int)n);
  return launch_status("dequant_bias");
}

int ttmi_build_token_rows(const int32_t* cu_seqlens, int64_t batch, int64_t max_seq, int64_t total,
                          int32_t* token_rows, void* stream) {
  TTMI_REQUIRE(cu_seqlens && token_rows, "null tensor");
  TTMI_REQUIRE(batch > 0 && batch * max_seq < (1ll << 31) && total < (1ll << 31), "bad shape");
  if (total <= 0) return 0;
  hipLaunchKernelGGL(token_rows_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, (hipStream_t)stream,
                     cu_seqlens, (int)batch, (int)max_seq, (int)total, token_rows);
  return launch_status("build_token_rows");
}

}  // extern "C"
