// C ABI of the MFMA GEMM family: argument checks, epilogue selection and the static scratch buffer.
// The kernels, epilogues and launch heuristics live in gemm_impl.h.
#include <cstring>

#include "gemm_impl.h"
#include "split_f32.h"

namespace ttmi {

// gemm_typed.h, instantiated per element type in gemm_<type>.hip
template <typename T>
int gemm_alpha_beta(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t ldc,
                    int inner, int64_t a_outer, int64_t a_inner, int64_t b_outer, int64_t b_inner, int64_t c_outer,
                    int64_t c_inner, int64_t batch, int trans_b, float alpha, float beta, hipStream_t s);
template <typename T>
int gemm_fused_typed(const GemmArgs& g, void* c, int64_t ldc, int epilogue, const ttmi_epilogue_args* args, hipStream_t s,
                     const NormRows<T>* norm);
template <typename T>
int gemm_norm_fused_typed(const GemmArgs& g, const void* gamma, const void* beta, float eps, void* c, int64_t ldc, int epilogue,
                          const ttmi_epilogue_args* args, hipStream_t s);
template <typename T>
int add_slices_layer_norm_typed(const float* slices, int64_t count, void* out, const void* residual, const float* residual_f32,
                                const void* bias, const void* gamma, const void* beta, float* out_f32, int64_t m, int64_t n, float eps,
                                hipStream_t s);
template <typename T>
int gemm_bias_layer_norm_typed(const void* a, const void* w, bool packed, void* out, const void* residual, const float* residual_f32,
                               const void* bias, const void* gamma, const void* beta, float* out_f32, int64_t m, int64_t n,
                               int64_t k, float eps, int dtype, hipStream_t s);

// ------------------------------------------------------------ static scratch buffer -----
// Partial tiles of ttmi_gemm_bias_layer_norm_static: device memory that exists from module load to
// process end on every GPU the library runs on, so that entry point never allocates.  In host code
// the array's name is only a handle: the device address is asked for once per device, with that
// device current, and kept; kernels and fills get that pointer.
constexpr size_t kStaticScratchBytes = TTMI_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

static int static_scratch(float** out) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static float* ptrs[kMaxDevices] = {};
  int dev = 0;
  TTMI_HIP(hipGetDevice(&dev));
  TTMI_REQUIRE(dev >= 0 && dev < kMaxDevices, "device ordinal out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (ptrs[dev] == nullptr) {
    void* p = nullptr;
    TTMI_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    TTMI_REQUIRE(p != nullptr, "the static scratch buffer has no device address");
    ptrs[dev] = static_cast<float*>(p);
  }
  *out = ptrs[dev];
  return 0;
}

// TTMI_F32_PACKED: fp32 with packed weights.
static int packed_operand(int* dtype, int64_t k, int64_t ldb, bool* packed) {
  *packed = *dtype == TTMI_F32_PACKED;
  if (*packed) {
    TTMI_REQUIRE(k % TTMI_PACKED_WEIGHT_K == 0 && ldb == k, "packed weights are contiguous rows of whole groups of K");
    *dtype = TTMI_F32;
  }
  return 0;
}

// The halves of packed weights (split_f32.h) behind their fp32 rows, and a flag per row: the power of two that its halves were scaled by,
// 0 for rows in the window, kSplitOutside for rows with an infinity.  Once per weight: one workgroup per row, 16 bytes of it per
// thread and turn.
static __global__ __launch_bounds__(256) void split_weights_kernel(float* __restrict__ packed, int n, int k) {
  __shared__ float part[256 / kWave];
  const int row = blockIdx.x;
  const float* src = packed + (int64_t)row * k;
  char* dst = reinterpret_cast<char*>(packed + (int64_t)n * k + (int64_t)row * k);
  float largest = 0.f;
  for (int col = threadIdx.x * 4; col < k; col += 1024) {
    const float4 x = *reinterpret_cast<const float4*>(src + col);
    split_max(largest, x.x, x.y);
    split_max(largest, x.z, x.w);
  }
  largest = group_max<kWave>(largest);
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = largest;
  __syncthreads();
  largest = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  const int flag = !split_outside(largest) ? 0 : largest == __builtin_inff() ? kSplitOutside : 1 - __builtin_amdgcn_frexp_expf(largest);
  const int scale = flag == kSplitOutside ? 0 : flag;  // (the row's largest value comes to between 1 and 2)
  for (int col = threadIdx.x * 4; col < k; col += 1024) {
    float4 x = *reinterpret_cast<const float4*>(src + col);
    x = make_float4(__builtin_ldexpf(x.x, scale), __builtin_ldexpf(x.y, scale), __builtin_ldexpf(x.z, scale), __builtin_ldexpf(x.w, scale));
    const uint2 hi = make_uint2(split_hi(x.x, x.y), split_hi(x.z, x.w));
    char* group = dst + (col / TTMI_PACKED_WEIGHT_K) * (TTMI_PACKED_WEIGHT_K * 4) + (col % TTMI_PACKED_WEIGHT_K) * 2;
    *reinterpret_cast<uint2*>(group) = hi;
    *reinterpret_cast<uint2*>(group + TTMI_PACKED_WEIGHT_K * 2) = make_uint2(split_lo(hi.x, x.x, x.y), split_lo(hi.y, x.z, x.w));
  }
  if (threadIdx.x == 0) reinterpret_cast<int*>(packed + 2 * (int64_t)n * k)[row] = flag;
}

static int gemm_bias_layer_norm_impl(const void* a, const void* w, void* out, const void* residual, const float* residual_f32,
                              const void* bias, const void* gamma, const void* beta, float* out_f32, int64_t m, int64_t n,
                              int64_t k, float eps, int dtype, void* stream) {
  TTMI_REQUIRE(a && w && out && bias && gamma && beta, "null tensor");
  TTMI_REQUIRE((residual_f32 != nullptr) == (out_f32 != nullptr), "residual_f32 and out_f32 go together");
  TTMI_REQUIRE(residual != nullptr || residual_f32 != nullptr, "a residual is required");
  // Large problems write the bare product to `out` before the residual is read.
  TTMI_REQUIRE(out != residual && out != a, "out must not alias residual or a");
  TTMI_REQUIRE(m >= 0 && n >= 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 31), "dimension out of range");
  if (m == 0 || n == 0) return 0;
  TTMI_REQUIRE(k > 0, "K must be positive");
  bool packed = false;
  const int rc = packed_operand(&dtype, k, k, &packed);
  if (rc != 0) return rc;
  TTMI_DISPATCH_FLOAT(dtype, T, return gemm_bias_layer_norm_typed<T>(a, w, packed, out, residual, residual_f32, bias, gamma, beta, out_f32, m,
                                                                     n, k, eps, dtype, (hipStream_t)stream));
  return 0;
}

}  // namespace ttmi

using namespace ttmi;

// The name of what `launch`, a call that launches one product, would run.
template <typename Launch>
static int describe(char* out, size_t capacity, const Launch& launch) {
  TTMI_REQUIRE(out != nullptr && capacity > 0, "no room for the answer");
  std::string name;
  struct Install {
    explicit Install(std::string* p) { tl_describe = p; }
    ~Install() { tl_describe = nullptr; }
  } install(&name);
  // operands that pass every alignment test; nothing dereferences them in a dry run
  const int rc = launch(reinterpret_cast<void*>((uintptr_t)1 << 20));
  if (rc != 0) return rc;
  TTMI_REQUIRE(name.size() < capacity, "the answer does not fit");
  std::memcpy(out, name.c_str(), name.size() + 1);
  return 0;
}

extern "C" {

int ttmi_gemm(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb,
              int64_t ldc, int trans_b, float alpha, float beta, int dtype, void* stream) {
  TTMI_REQUIRE(a && b && c, "null matrix");
  TTMI_REQUIRE(lda >= k && ldc >= n && ldb >= (trans_b ? k : n), "leading dimension too small");
  TTMI_DISPATCH_FLOAT(dtype, T, return gemm_alpha_beta<T>(a, b, c, m, n, k, lda, ldb, ldc, 1, 0, 0, 0, 0, 0, 0, 1,
                                                          trans_b, alpha, beta, (hipStream_t)stream));
  return 0;
}

int ttmi_gemm_strided_batched(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda,
                              int64_t ldb, int64_t ldc, int64_t stride_a, int64_t stride_b, int64_t stride_c,
                              int64_t batch_count, int trans_b, float alpha, float beta, int dtype, void* stream) {
  TTMI_REQUIRE(a && b && c, "null matrix");
  TTMI_REQUIRE(lda >= k && ldc >= n && ldb >= (trans_b ? k : n), "leading dimension too small");
  TTMI_REQUIRE(batch_count >= 0 && batch_count < 65536, "batch_count out of range");
  TTMI_DISPATCH_FLOAT(dtype, T, return gemm_alpha_beta<T>(a, b, c, m, n, k, lda, ldb, ldc, 1, stride_a, 0, stride_b,
                                                          0, stride_c, 0, batch_count, trans_b, alpha, beta,
                                                          (hipStream_t)stream));
  return 0;
}

int ttmi_gemm_batched_heads(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda,
                            int64_t ldb, int64_t ldc, int64_t heads, int64_t a_batch, int64_t a_head,
                            int64_t b_batch, int64_t b_head, int64_t c_batch, int64_t c_head, int64_t batch,
                            int trans_b, float alpha, float beta, int dtype, void* stream) {
  TTMI_REQUIRE(a && b && c, "null matrix");
  TTMI_REQUIRE(heads > 0 && batch >= 0 && batch * heads < 65536, "batch*heads out of range");
  TTMI_DISPATCH_FLOAT(dtype, T, return gemm_alpha_beta<T>(a, b, c, m, n, k, lda, ldb, ldc, (int)heads, a_batch,
                                                          a_head, b_batch, b_head, c_batch, c_head, batch * heads,
                                                          trans_b, alpha, beta, (hipStream_t)stream));
  return 0;
}

static int gemm_fused_impl(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda,
                           int64_t ldb, int64_t ldc, int epilogue, const ttmi_epilogue_args* args, int dtype, bool any_form,
                           void* stream) {
  TTMI_REQUIRE(a && b && args, "null argument");
  TTMI_REQUIRE(m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 31), "dimension too large");
  TTMI_REQUIRE(lda >= k && ldb >= k, "leading dimension too small");
  bool packed = false;
  const int rc = packed_operand(&dtype, k, ldb, &packed);
  if (rc != 0) return rc;
  GemmArgs g{};
  g.a = (const char*)a;
  g.b = (const char*)b;
  g.m = (int)m; g.n = (int)n; g.k = (int)k;
  g.lda = lda; g.ldb = ldb;
  g.inner = 1;
  g.any_form = any_form;
  if (packed) use_packed_weights(g);
  TTMI_DISPATCH_FLOAT(dtype, T, return gemm_fused_typed<T>(g, c, ldc, epilogue, args, (hipStream_t)stream, nullptr));
  return 0;
}

int ttmi_gemm_fused(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda,
                    int64_t ldb, int64_t ldc, int epilogue, const ttmi_epilogue_args* args, int dtype,
                    void* stream) {
  return gemm_fused_impl(a, b, c, m, n, k, lda, ldb, ldc, epilogue, args, dtype, false, stream);
}

int ttmi_gemm_bias_act(const void* a, const void* w, const void* bias, void* c, int64_t m, int64_t n, int64_t k, int act, int dtype,
                       void* stream) {
  ttmi_epilogue_args args{};
  args.bias = bias;
  args.act = act;
  return gemm_fused_impl(a, w, c, m, n, k, k, k, n, TTMI_EPI_BIAS_ACT, &args, dtype, true, stream);
}

int ttmi_layer_norm_gemm_fused(const void* x, const void* gamma, const void* beta, float eps, void* normed, const void* w, void* c,
                               int64_t m, int64_t n, int64_t k, int64_t ldc, int epilogue, const ttmi_epilogue_args* args, int dtype,
                               void* stream) {
  TTMI_REQUIRE(x && gamma && beta && normed && w && args && normed != x, "null tensor, or in place");
  TTMI_REQUIRE(m >= 0 && n >= 0 && k >= 0 && m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 31), "dimension out of range");
  GemmArgs g{};
  g.a = (const char*)x;
  g.b = (const char*)w;
  g.m = (int)m; g.n = (int)n; g.k = (int)k;
  g.lda = k; g.ldb = k;
  g.inner = 1;
  bool packed = false;
  int base = dtype, rc = packed_operand(&base, k, k, &packed);
  if (rc != 0) return rc;
  rc = kNormNotTaken;
  TTMI_DISPATCH_FLOAT(base, T, rc = gemm_norm_fused_typed<T>(g, gamma, beta, eps, c, ldc, epilogue, args, (hipStream_t)stream));
  if (rc != kNormNotTaken) return rc;
  rc = ttmi_layer_norm_from(normed, x, gamma, beta, m, k, eps, base, stream);
  if (rc != 0) return rc;
  return ttmi_gemm_fused(normed, w, c, m, n, k, k, k, ldc, epilogue, args, dtype, stream);
}

int ttmi_split_weights(void* packed, int64_t n, int64_t k, void* stream) {
  TTMI_REQUIRE(packed != nullptr && aligned16(packed), "packed weights must be 16-byte aligned");
  TTMI_REQUIRE(n >= 0 && k >= 0 && n < (1ll << 31) && k < (1ll << 31) && k % TTMI_PACKED_WEIGHT_K == 0, "weight size");
  if (n == 0 || k == 0) return 0;
  hipLaunchKernelGGL(split_weights_kernel, dim3((unsigned)n), dim3(256), 0, (hipStream_t)stream, (float*)packed, (int)n, (int)k);
  return launch_status("split_weights_kernel");
}

int ttmi_gemm_describe(int64_t m, int64_t n, int64_t k, int epilogue, const ttmi_epilogue_args* args, int dtype, char* out,
                       size_t capacity) {
  return describe(out, capacity, [&](void* fake) {
    ttmi_epilogue_args filled{};
    if (args != nullptr) filled = *args;
    filled.bias = fake;
    filled.residual = fake;
    filled.q = filled.k = filled.v = fake;
    if (epilogue == TTMI_EPI_QKV_SPLIT_PAD) filled.token_rows = static_cast<const int32_t*>(fake);
    return epilogue == TTMI_EPI_NONE ? ttmi_gemm(fake, fake, fake, m, n, k, k, k, n, 1, 1.f, 0.f, dtype, nullptr)
                                     : ttmi_gemm_fused(fake, fake, fake, m, n, k, k, k, n, epilogue, &filled, dtype, nullptr);
  });
}

int ttmi_gemm_bias_act_describe(int64_t m, int64_t n, int64_t k, int act, int dtype, char* out, size_t capacity) {
  return describe(out, capacity, [&](void* fake) { return ttmi_gemm_bias_act(fake, fake, fake, fake, m, n, k, act, dtype, nullptr); });
}

int ttmi_gemm_bias_layer_norm(const void* a, const void* w, void* out, const void* residual, const float* residual_f32,
                              const void* bias, const void* gamma, const void* beta, float* out_f32, int64_t m, int64_t n,
                              int64_t k, float eps, int dtype, void* stream) {
  return gemm_bias_layer_norm_impl(a, w, out, residual, residual_f32, bias, gamma, beta, out_f32, m, n, k, eps, dtype, stream);
}

int ttmi_add_slices_layer_norm(const float* slices, int64_t count, void* out, const void* residual, const float* residual_f32,
                               const void* bias, const void* gamma, const void* beta, float* out_f32, int64_t m, int64_t n,
                               float eps, int dtype, void* stream) {
  TTMI_REQUIRE(slices && out && bias && gamma && beta, "null tensor");
  TTMI_REQUIRE((residual_f32 != nullptr) == (out_f32 != nullptr), "residual_f32 and out_f32 go together");
  TTMI_REQUIRE(residual != nullptr || residual_f32 != nullptr, "a residual is required");
  TTMI_REQUIRE(count > 0 && count < (1 << 16) && m >= 0 && m < (1ll << 31) && n >= 0 && n <= 4096 && n % 4 == 0, "dimension out of range");
  if (m == 0 || n == 0) return 0;
  TTMI_DISPATCH_FLOAT(dtype, T, return add_slices_layer_norm_typed<T>(slices, count, out, residual, residual_f32, bias, gamma, beta, out_f32,
                                                                      m, n, eps, (hipStream_t)stream));
  return 0;
}

int ttmi_gemm_bias_layer_norm_static(const void* a, const void* w, void* out, const void* residual,
                                     const float* residual_f32, const void* bias, const void* gamma, const void* beta,
                                     float* out_f32, int64_t m, int64_t n, int64_t k, float eps, int dtype, void* stream) {
  float* ws = nullptr;
  {
    const int rc = static_scratch(&ws);
    if (rc != 0) return rc;
  }
  // Every split-K launch below this call takes its partial tiles from the static buffer, or is refused.  (The
  // switch lowers the size that is admitted, so that tests reach the refusal with problems of ordinary size.)
  size_t capacity = kStaticScratchBytes;
  const int limit = kernel_switch(kSwitchStaticScratchLimit);
  if (limit >= 0) capacity = std::min(capacity, (size_t)limit);
  struct Install {
    Install(float* p, size_t bytes) { tl_fixed_workspace = FixedWorkspace{p, bytes}; }
    ~Install() { tl_fixed_workspace = FixedWorkspace{}; }
  } install(ws, capacity);
  return gemm_bias_layer_norm_impl(a, w, out, residual, residual_f32, bias, gamma, beta, out_f32, m, n, k, eps, dtype, stream);
}

}  // extern "C"
