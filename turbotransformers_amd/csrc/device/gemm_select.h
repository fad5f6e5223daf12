// Selection for the products with an epilogue: few rows (gemm_flat.h), mid-size (gemm_ring.h), fp32 with packed weights
// (gemm_split.h), or for large problems the
// persistent tiles of gemm_w4.h (16-bit types) and of gemm_fast_kernel (int8).
#pragma once

#include "gemm_flat.h"

namespace ttmi {

template <typename Epi>
inline bool epilogue_vec(const Epi& epi) {
  if constexpr (std::is_same<Epi, EpiDequantQkvSplit>::value) return epi.split.vec && aligned16(epi.w_scale) && aligned16(epi.split.bias);
  else if constexpr (std::is_same<Epi, EpiDequant>::value) return epi.vec && aligned16(epi.w_scale) && aligned16(epi.bias);
  else return epi.vec;
}
template <typename Epi>
struct IsGelu : std::false_type {};
template <typename T>
struct IsGelu<EpiBias<T, TTMI_ACT_GELU, true, false>> : std::true_type {};

// The large problems' persistent tiles run their epilogues under the next tile's first loads.
template <typename T, typename Epi>
struct RingKernel {
  static int64_t column_limit(const Epi& epi) {
    if constexpr (HasColumnPass<Epi>::value) return epi.v_pitch > 0 ? 2 * (int64_t)epi.hidden : 0;
    else return 0;
  }
  // 65 to 128 rows with GELU of a width and K for which ttmi_gemm_describe has always named one form: fp32 cut along K (eight
  // steps or more, up to 128 tiles of 64 x 64), 16-bit whole on the wavefront kernel (short of sixteen steps, more than 64
  // tiles).  Neither is the fastest since the ring tiles.  us, kept / ring: fp32 128 x 3072 x 768 14.8 / 9.5, 128 x 4096 x
  // 1024 16.7 / 11.9, 128 x 2048 x 512 9.5 / 7.2; fp16 128 x 3072 x 768 8.4 / 5.0, 72 x 3072 x 768 8.3 / 5.1.  Outside these
  // lines they would cost up to four times the ring's time (fp16 128 x 16384 x 4096 114 / 30, fp32 128 x 8192 x 512 18.1 / 11.4).
  // ttmi_gemm_bias_act, which the layers call, has no such form: us a forward of fp16 base, as ttmi_gemm_fused / so: 1 x 70 tokens 416 / 369, 1 x 128 424 / 378.
  static bool keeps_named_form(const GemmArgs& g) {
    const int64_t ksteps = g.k / (kRowBytes / (int)sizeof(T)), tiles = ceil_div(g.m, 64) * ceil_div(g.n, 64);
    return !g.any_form && g.m > 64 && g.m <= 128 && (sizeof(T) == 4 ? ksteps >= 8 && tiles <= 128 : ksteps < 16 && tiles > 64);
  }
  static RingPlan plan(const GemmArgs& g, const Epi& epi) {
    // a cut needs an epilogue that the reduction kernel can apply to rows of eight columns
    constexpr bool cut = std::is_same<typename Epi::Acc, float>::value;
    RingUse use = cut && column_limit(epi) == 0 ? RingUse::kSliced : RingUse::kWhole;
    if constexpr (IsGelu<Epi>::value && sizeof(T) == 4)
      if (g.b_split == nullptr && keeps_named_form(g)) use = RingUse::kCut;
    return pick_ring<T>(g, use, column_limit(epi), HasColumnPass<Epi>::value);
  }
  static bool ok(const GemmArgs& g, const Epi& epi, int batch) {
    return batch == 1 && g.k_chunk == 0 && ring_operands_ok<T>(g) && epilogue_vec(epi) && column_limit(epi) % kRingColumns == 0;
  }
  static int launch(const GemmArgs& g, const Epi& epi, hipStream_t s) {
    constexpr int BK = kRowBytes / (int)sizeof(T);
    if constexpr (IsGelu<Epi>::value && sizeof(T) == 2)
      if (keeps_named_form(g) && wave_kernel_ok<T>(g, 1, true)) return launch_wave<T>(g, epi, s);
    if (flat_wins<T>(g, 96)) return launch_flat<T>(g, epi, 1, s);
    const RingPlan p = plan(g, epi);
    if constexpr (sizeof(T) == 2) {
      const int force = kernel_switch(kSwitchLargeTile);
      // More than one workgroup per CU: long enough a launch that the chip runs at its power limit, under which the small
      // tiles' extra LDS and L2 traffic costs clock (16384 x 1024 x 4096: 123 us against 106 although the unthrottled
      // model has it 20 % ahead).  Less so the largest of them, 256 x 160 in 16 bits alone, while there are two rounds: 6275 x 3072 x 768 (GELU) in a forward of 20 packed
      // requests 44 us on the large tiles, 37 in 256 x 160.
      const double margin = p.rounds > 1 ? (p.rounds == 2 && p.tile_values >= 256 * 160 ? 1.1 : 1.3) : 1.0;
      if (force != 0 && LargeTileKernel<T, Epi>::eligible(g, epi) && (force == 1 || LargeTileKernel<T, Epi>::us(g, epi) < margin * p.us))
        return LargeTileKernel<T, Epi>::launch(g, epi, s);
    }
    if constexpr (sizeof(T) == 1) {
      auto us = [&](int bn, double first, double again, double step) {
        return first + ceil_div(ceil_div(g.m, 256) * ceil_div(g.n, bn), compute_units()) * (again + g.k / BK * step);
      };
      const double us192 = us(192, 2.8, 11.3, 1.224), us256 = us(256, 2.6, 6.8, 2.761);
      if (std::min(us192, us256) < p.us)
        return us192 < us256 ? launch_fast<T, 256, 192, 4, 2, Epi>(g, epi, 1, s) : launch_fast<T, 256, 256, 2, 4, Epi>(g, epi, 1, s);
    }
    if constexpr (std::is_same<typename Epi::Acc, float>::value)
      if (p.slices > 1) return launch_ring_slices<T>(g, p, s, ReduceWithEpilogue<Epi>{epi, g.m, g.n});
    return launch_ring_tile<T>(p.tile, g, epi, 1, s);
  }
};

}  // namespace ttmi
