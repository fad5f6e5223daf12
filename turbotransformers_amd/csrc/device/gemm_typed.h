// The entry points of the GEMM family for one element type.  gemm_<type>.hip instantiates them, so that the element
// types compile side by side; gemm.hip holds the C ABI.
#pragma once

#include "gemm_select.h"

namespace ttmi {

template <typename T>
int gemm_alpha_beta(const void* a, const void* b, void* c, int64_t m, int64_t n, int64_t k, int64_t lda,
                           int64_t ldb, int64_t ldc, int inner, int64_t a_outer, int64_t a_inner,
                           int64_t b_outer, int64_t b_inner, int64_t c_outer, int64_t c_inner, int64_t batch,
                           int trans_b, float alpha, float beta, hipStream_t s) {
  TTMI_REQUIRE(m < (1ll << 31) && n < (1ll << 31) && k < (1ll << 31), "dimension too large");
  GemmArgs g{};
  g.a = (const char*)a;
  g.b = (const char*)b;
  g.m = (int)m; g.n = (int)n; g.k = (int)k;
  g.lda = lda; g.ldb = ldb;
  g.inner = inner;
  g.a_outer = a_outer; g.a_inner = a_inner; g.b_outer = b_outer; g.b_inner = b_inner;
  constexpr int KPC = 16 / sizeof(T);
  const bool c_vec = aligned16(c) && ldc % KPC == 0 && c_outer % KPC == 0 && c_inner % KPC == 0;
  EpiAlphaBeta<T> epi{(T*)c, ldc, c_outer, c_inner, inner, alpha, beta, c_vec};
  auto mult = [](int64_t v) { return v % KPC == 0; };
  bool aligned = aligned16(a) && aligned16(b) && mult(lda) && mult(ldb) && mult(a_outer) && mult(a_inner) &&
                 mult(b_outer) && mult(b_inner);
  if (trans_b) {
    aligned = aligned && mult(k);
    return launch_gemm<T, false>(g, epi, (int)batch, aligned, s);
  }
  aligned = aligned && mult(k) && mult(n);
  return launch_gemm<T, true>(g, epi, (int)batch, aligned, s);
}


template <typename T, bool PAD>
inline EpiQkvSplit<T, PAD> qkv_epilogue(const ttmi_epilogue_args* args) {
  const int hidden = (int)(args->heads * args->head_dim);
  const bool vec = aligned16(args->q) && aligned16(args->k) && aligned16(args->v) && aligned16(args->bias) && args->head_dim % 8 == 0;
  return {(T*)args->q, (T*)args->k, (T*)args->v, (const T*)args->bias, PAD ? args->token_rows : nullptr, (int)args->seq,
          (int)args->heads, (int)args->head_dim, hidden, FastDiv((uint32_t)args->seq), FastDiv((uint32_t)hidden),
          FastDiv((uint32_t)args->head_dim), vec, (int)args->v_seq_pitch};
}

// `norm`: A's rows are to be normalised on their way in (gemm_norm_fused_typed has checked that they can be).
template <typename T>
int gemm_fused_typed(const GemmArgs& g, void* c, int64_t ldc, int epilogue, const ttmi_epilogue_args* args, hipStream_t s, const NormRows<T>* norm) {
  const int64_t m = g.m, n = g.n, k = g.k, lda = g.lda, ldb = g.ldb;
  const void *a = g.a, *b = g.b;
  constexpr int KPC = 16 / sizeof(T);
  const bool aligned = aligned16(a) && aligned16(b) && lda % KPC == 0 && ldb % KPC == 0 && k % KPC == 0;
  const bool c_vec = aligned16(c) && ldc % KPC == 0 && aligned16(args->bias) && aligned16(args->residual);
  switch (epilogue) {
    case TTMI_EPI_BIAS: {
      TTMI_REQUIRE(c && args->bias && ldc >= n, "BIAS epilogue needs c and bias");
      EpiBias<T, 0, false, false> epi{(T*)c, (const T*)args->bias, nullptr, ldc, c_vec};
      return (launch_gemm<T, false>(g, epi, 1, aligned, s));
    }
    case TTMI_EPI_BIAS_ACT: {
      TTMI_REQUIRE(c && args->bias && ldc >= n, "BIAS_ACT epilogue needs c and bias");
      if (args->act == TTMI_ACT_GELU) {
        EpiBias<T, TTMI_ACT_GELU, true, false> epi{(T*)c, (const T*)args->bias, nullptr, ldc, c_vec};
        return (launch_gemm<T, false>(g, epi, 1, aligned, s));
      } else if (args->act == TTMI_ACT_TANH) {
        EpiBias<T, TTMI_ACT_TANH, true, false> epi{(T*)c, (const T*)args->bias, nullptr, ldc, c_vec};
        return (launch_gemm<T, false>(g, epi, 1, aligned, s));
      } else if (args->act == TTMI_ACT_RELU) {
        EpiBias<T, TTMI_ACT_RELU, true, false> epi{(T*)c, (const T*)args->bias, nullptr, ldc, c_vec};
        if (norm != nullptr && c_vec) return launch_flat_norm<T>(g, epi, *norm, s);
        if (norm != nullptr) return kNormNotTaken;
        return (launch_gemm<T, false>(g, epi, 1, aligned, s));
      }
      return fail(TTMI_EINVAL, "unknown activation");
    }
    case TTMI_EPI_F32_OUT: {
      TTMI_REQUIRE(c && ldc >= n, "F32_OUT epilogue needs c");
      EpiF32<T> epi{(float*)c, (const T*)args->bias, ldc, aligned16(c) && ldc % 4 == 0 && aligned16(args->bias)};
      return (launch_gemm<T, false>(g, epi, 1, aligned, s));
    }
    case TTMI_EPI_BIAS_RESIDUAL: {
      TTMI_REQUIRE(c && args->bias && args->residual && ldc >= n, "BIAS_RESIDUAL epilogue needs c, bias, residual");
      EpiBias<T, 0, false, true> epi{(T*)c, (const T*)args->bias, (const T*)args->residual, ldc, c_vec};
      return (launch_gemm<T, false>(g, epi, 1, aligned, s));
    }
    case TTMI_EPI_QKV_SPLIT:
    case TTMI_EPI_QKV_SPLIT_PAD: {
      const bool pad = epilogue == TTMI_EPI_QKV_SPLIT_PAD;
      TTMI_REQUIRE(args->seq > 0 && args->heads > 0 && args->head_dim > 0, "QKV epilogue needs seq/heads/head_dim");
      const bool single = n == args->heads * args->head_dim;  // one projection: only q is written
      const bool pair = n == 2 * args->heads * args->head_dim;  // two projections: q and k are written
      TTMI_REQUIRE(single || pair || n == 3 * args->heads * args->head_dim, "N must be one, two or three times heads*head_dim");
      TTMI_REQUIRE(args->q && args->bias && (single || args->k) && (single || pair || args->v), "QKV epilogue needs q, k, v, bias");
      TTMI_REQUIRE(!(single || pair) || args->v_seq_pitch == 0, "v_seq_pitch needs the three-way split");
      if (pad) TTMI_REQUIRE(args->token_rows != nullptr && args->batch > 0, "padded QKV epilogue needs token_rows and batch");
      else TTMI_REQUIRE(m % args->seq == 0, "M must be a multiple of seq");
      const int hidden = (int)(args->heads * args->head_dim);
      const int64_t vp = args->v_seq_pitch;
      TTMI_REQUIRE(vp == 0 || (vp >= args->seq && vp % 8 == 0 && vp < (1ll << 31) && hidden % 8 == 0),
                   "v_seq_pitch must be 0 or a multiple of 8 that is >= seq (hidden a multiple of 8)");
      if (pad) {
        return (launch_gemm<T, false>(g, qkv_epilogue<T, true>(args), 1, aligned, s));
      }
      const EpiQkvSplit<T, false> epi = qkv_epilogue<T, false>(args);
      if (norm != nullptr && epi.vec) return launch_flat_norm<T>(g, epi, *norm, s);
      if (norm != nullptr) return kNormNotTaken;
      return (launch_gemm<T, false>(g, epi, 1, aligned, s));
    }
    default:
      return fail(TTMI_EINVAL, "unknown epilogue");
  }
}

// LayerNorm(x) in front of a product with an epilogue.  One launch where the form for few rows takes the product and its
// epilogue (the bias and ReLU of a feed-forward layer, the head split): two are a wait more each and 3 to 4 us of host time.
// 0: done.  kNormNotTaken: the two launches it is.
template <typename T>
int gemm_norm_fused_typed(const GemmArgs& g, const void* gamma, const void* beta, float eps, void* c, int64_t ldc, int epilogue,
                          const ttmi_epilogue_args* args, hipStream_t s) {
  const bool known = epilogue == TTMI_EPI_QKV_SPLIT || (epilogue == TTMI_EPI_BIAS_ACT && args->act == TTMI_ACT_RELU);
  if (!known || g.m == 0 || g.n == 0 || g.k * (int)sizeof(T) % kRowBytes != 0 || g.k == 0 || !aligned16(g.a) || !aligned16(g.b) ||
      g.lda * (int64_t)sizeof(T) % 16 != 0 || g.ldb * (int64_t)sizeof(T) % 16 != 0 || !aligned16(gamma) || !aligned16(beta) ||
      !ring_operands_ok<T>(g) || !flat_norm_wins<T>(g))
    return kNormNotTaken;
  const NormRows<T> rows{(const T*)gamma, (const T*)beta, eps};
  return gemm_fused_typed<T>(g, c, ldc, epilogue, args, s, &rows);
}

// Where the product in front of a LayerNorm is held in fp32 although nothing else asks for it (RingUse::kLayerNorm: whole or
// in K slices, summed by the kernel that normalises).  Elsewhere a 16-bit product is rounded on its way through `out`.
// Few rows make the extra bytes free, and a long sum loses most to the rounding.
inline bool fp32_product_pays(int64_t m, int64_t n, int64_t k) { return m <= 384 || (k >= 2 * n && m * n * 4 <= (20ll << 20)); }
// ... and where the tiles leave so many CUs idle over so long a K that such products have always been cut along K, which
// holds them: rounded, they would lose precision that callers had.  It costs an fp32 copy of the product; us, fp16, rounded /
// held: 512 x 512 x 512 7.6 / 7.3, 1024 x 1024 x 1024 10.3 / 12.1, 2048 x 1024 x 1024 13.2 / 17.2, 8192 x 768 x 3072 44.9 /
// 50.6, 10752 x 768 x 3072 55.1 / 62.0, 8192 x 1024 x 4096 66.5 / 74.5 (cut, as they were: 7.9, 16.5, 22.5, 53.4, 67.2, 76.9).
inline bool fp32_product_expected(int64_t m, int64_t n, int64_t k) {
  auto tiles = [&](int edge) { return ceil_div(m, edge) * ceil_div(n, edge); };
  const int64_t cus = compute_units();
  return (k >= 512 && tiles(64) <= cus / 4) || (k >= 1024 && tiles(128) <= cus / 2) || (k >= 2048 && tiles(256) <= cus / 2);
}

template <typename T>
void launch_reduce_layer_norm(const float* ws, int slices, int64_t m, int64_t n, const void* bias, const void* residual,
                              const float* residual_f32, const void* gamma, const void* beta, void* out, float* out_f32, float eps,
                              hipStream_t s) {
  auto launch = [&](auto iters, auto at_once) {
    hipLaunchKernelGGL((splitk_reduce_layer_norm_kernel<T, decltype(iters)::value, decltype(at_once)::value>), dim3((unsigned)m), dim3(256), 0, s, ws, slices,
                       (int)m, (int)n, (const T*)bias, (const T*)residual, residual_f32, (const T*)gamma, (const T*)beta, (T*)out,
                       out_f32, eps, writes_through(m * n * (int64_t)(sizeof(T) + (out_f32 != nullptr ? sizeof(float) : 0))));
  };
  // Both outputs count and go through: large bf16, which has the fp32 one, staying / through 3 x 128 tokens 1140 / 1132 us a forward, 8 x 128
  // 1526 / 1516, 12 x 128 1990 / 1974, 32 x 128 3667 / 3655; fp16 base 12 x 128 689 / 686, fp32 base 8 x 128 1177 / 1174, otherwise level.
  // How many slices are on their way at a time: a chain of waits again, but registers that more rows would miss.  Up to 64 rows, where
  // the attention leaves a slice per head, us for both launches with four / eight / twelve / sixteen at a time, 32 tokens: 6 slices 7.7 / 7.8 / 7.8 /
  // 7.8, 8 7.6 / 7.4 / 7.7 / 7.7, 11 8.6 / 8.4 / 8.7 / 8.7, 12 8.2 / 8.1 / 7.9 / 8.3, 15 9.7 / 9.7 / 9.5 / 9.8, 16 8.8 / 8.4 / 8.7 / 8.5; 24 and 32 slices
  // alone 3.0 / 2.8 / 2.9 / 3.3 and 3.3 / 3.1 / 3.3 / 3.3.  384 rows, 8 slices 2.6 / 2.8 / 2.8 / 2.8; 20 x 100 tokens, two slices of 2000 rows, a
  // forward 1 % slower with twelve.
  constexpr std::integral_constant<int, 4> four{};
  constexpr std::integral_constant<int, 1> row{};
  const bool twelve = slices >= 12 && (slices < 16 || m > 64);
  if (n <= 1024 && twelve) launch(row, std::integral_constant<int, 12>{});
  else if (n <= 1024 && slices >= 8 && m <= 64) launch(row, std::integral_constant<int, 8>{});
  else if (n <= 1024) launch(row, four);
  else if (n <= 2048) launch(std::integral_constant<int, 2>{}, four);
  else launch(std::integral_constant<int, 4>{}, four);
}

// The slices of a product + AddBiasLayerNorm; the rows were checked by the caller.
template <typename T>
int add_slices_layer_norm_typed(const float* slices, int64_t count, void* out, const void* residual, const float* residual_f32,
                                const void* bias, const void* gamma, const void* beta, float* out_f32, int64_t m, int64_t n, float eps,
                                hipStream_t s) {
  const uintptr_t rows = reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(gamma) |
                         reinterpret_cast<uintptr_t>(beta) | reinterpret_cast<uintptr_t>(residual);
  TTMI_REQUIRE(rows % (4 * sizeof(T)) == 0 && aligned16(slices) && aligned16(residual_f32) && aligned16(out_f32), "rows must be aligned to four elements");
  launch_reduce_layer_norm<T>(slices, (int)count, m, n, bias, residual, residual_f32, gamma, beta, out, out_f32, eps, s);
  return launch_status("add_slices_layer_norm");
}

// Product + AddBiasLayerNorm.
template <typename T>
int gemm_bias_layer_norm_typed(const void* a, const void* w, bool packed, void* out, const void* residual, const float* residual_f32,
                               const void* bias, const void* gamma, const void* beta, float* out_f32, int64_t m, int64_t n,
                               int64_t k, float eps, int dtype, hipStream_t s) {
  constexpr int KPC = 16 / sizeof(T), BK = kRowBytes / sizeof(T);
  const bool aligned = aligned16(a) && aligned16(w) && k % KPC == 0;
  auto aligned_rows = [&](const void* p, size_t elem) { return (reinterpret_cast<uintptr_t>(p) % (4 * elem)) == 0; };
  const bool rows_ok = n % 4 == 0 && n <= 4096 && aligned_rows(out, sizeof(T)) && aligned_rows(bias, sizeof(T)) &&
                       aligned_rows(gamma, sizeof(T)) && aligned_rows(beta, sizeof(T)) &&
                       (residual_f32 != nullptr ? aligned16(residual_f32) && aligned16(out_f32) : aligned_rows(residual, sizeof(T)));
  GemmArgs g{};
  g.a = (const char*)a;
  g.b = (const char*)w;
  g.m = (int)m; g.n = (int)n; g.k = (int)k;
  g.lda = k; g.ldb = k;
  g.inner = 1;
  if (packed) use_packed_weights(g);
  auto reduce = [&](const float* ws, int slices, bool, hipStream_t st) {
    launch_reduce_layer_norm<T>(ws, slices, m, n, bias, residual, residual_f32, gamma, beta, out, out_f32, eps, st);
  };
  if constexpr (sizeof(T) == 2) {
    int slices = rows_ok ? w4_splitk_slices<T>(g, aligned) : 0;
    // (an optimisation of a product that also runs whole: where the caller has fixed the workspace and the partial
    // products do not fit it, nothing is refused)
    if (slices > 1 && tl_fixed_workspace.ptr != nullptr &&
        (size_t)slices * (size_t)m * (size_t)n * sizeof(float) > tl_fixed_workspace.bytes)
      slices = 0;
    if (slices > 1) return launch_w4_splitk<T>(g, slices, s, reduce);
  }
  const bool ring = aligned && k % BK == 0 && ring_operands_ok<T>(g);
  if (!ring && rows_ok) {  // widths that are no multiple of eight
    const SplitPlan plan = plan_split<T>(m, n, k, 1, aligned);
    if (plan.kind == SplitKind::kDmaTiles) return launch_fast_splitk<T>(g, plan.splits, k / BK, BK, s, reduce);
    if (plan.kind == SplitKind::kSmallTiles) return launch_splitk<T>(g, plan.splits, k / BK, BK, s, reduce);
  }
  // with an fp32 residual stream and room for it the product stays in fp32 without a workspace
  const bool product_in_out32 = sizeof(T) == 2 && residual_f32 != nullptr && out_f32 != residual_f32;
  const bool pays = fp32_product_pays(m, n, k);
  if (ring && rows_ok && (pays || (sizeof(T) == 2 && !product_in_out32 && fp32_product_expected(m, n, k)))) {
    // Few rows: one slice; more of K is cheaper cut (10 x 768 x 3072 in twelve slices 3.8 us, whole 5.4), and so is fp32
    // (128 x 768 x 768 in five slices 5.7 us, whole 6.6).
    const bool flat = sizeof(T) == 2 && flat_wins<T>(g, 32);
    const RingPlan plan = flat ? RingPlan{} : pick_ring<T>(g, RingUse::kLayerNorm);
    const size_t bytes = (size_t)plan.slices * (size_t)m * (size_t)n * sizeof(float);
    // (where the caller has fixed the workspace and the copy does not fit it, the product is rounded and not refused)
    if (pays || tl_fixed_workspace.ptr == nullptr || bytes <= tl_fixed_workspace.bytes) {
      if (!flat) return launch_ring_slices<T>(g, plan, s, reduce);
      float* ws = nullptr;
      if (tl_describe == nullptr) {
        const int rc = splitk_workspace(bytes, s, &ws);
        if (rc != 0) return rc;
      }
      const int rc = launch_flat<T>(g, EpiPartial{ws, m * n, n, true}, 1, s);
      if (rc != 0 || tl_describe != nullptr) return rc;
      reduce(ws, 1, true, s);
      return launch_status("gemm_flat_layer_norm");
    }
  }
  if (product_in_out32) {  // the GEMM stores its accumulators to out_f32 and the LayerNorm pass reads them there
    EpiF32<T> epi{out_f32, nullptr, n, aligned16(out_f32) && n % 4 == 0};
    const int rc = launch_gemm<T, false>(g, epi, 1, aligned, s);
    if (rc != 0) return rc;
    return ttmi_add_bias_layer_norm_product32(out, residual_f32, bias, gamma, beta, out_f32, m, n, eps, dtype, s);
  }
  // (EpiBias without a bias: the plain product, through the selection of the fused ones)
  EpiBias<T, 0, false, false> epi{(T*)out, nullptr, nullptr, n, aligned16(out) && n % KPC == 0};
  const int rc = launch_gemm<T, false>(g, epi, 1, aligned, s);
  if (rc != 0) return rc;
  if (residual_f32 != nullptr)
    return ttmi_add_bias_layer_norm_residual32(out, residual_f32, bias, gamma, beta, out_f32, m, n, eps, dtype, s);
  return ttmi_add_bias_layer_norm(out, residual, bias, gamma, beta, m, n, eps, dtype, s);
}

#define TTMI_INSTANTIATE_GEMM(T)                                                                                            \
  template int gemm_alpha_beta<T>(const void*, const void*, void*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, \
                                  int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, float, float,           \
                                  hipStream_t);                                                                               \
  template int gemm_fused_typed<T>(const GemmArgs&, void*, int64_t, int, const ttmi_epilogue_args*, hipStream_t,              \
                                   const NormRows<T>*);                                                                       \
  template int gemm_norm_fused_typed<T>(const GemmArgs&, const void*, const void*, float, void*, int64_t, int,                \
                                        const ttmi_epilogue_args*, hipStream_t);                                              \
  template int gemm_bias_layer_norm_typed<T>(const void*, const void*, bool, void*, const void*, const float*, const void*,         \
                                             const void*, const void*, float*, int64_t, int64_t, int64_t, float, int,         \
                                             hipStream_t);                                                                    \
  template int add_slices_layer_norm_typed<T>(const float*, int64_t, void*, const void*, const float*, const void*, const void*, \
                                              const void*, float*, int64_t, int64_t, float, hipStream_t);

}  // namespace ttmi
