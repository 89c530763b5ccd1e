// The deep-ring kernel (mxfp4_gemm_deep.h) on MXFP4 operands.
#include "mxfp4_gemm_deep.h"

namespace wave_mxfp4 {

namespace {

// A stream of B that reaches the workgroups from HBM, with hardly an A beside it: from 17 K tiles on eight K tiles of
// 64x64 on their way are up to 10 % faster than four (2 x 13152 x 12800 preshuffled 24.4 -> 22.4 us; the time of eight over
// that of four, mean: up to 16 rows 0.96 preshuffled and 1.00 row-major, 17 .. 32 preshuffled 0.95, more rows 1.02 - 1.04).
typedef DeepCfg<64, 64, 2, 2, 8> DeepStream;

// Staged row-major scales of 128x128 tiles: a ring of three K tiles leaves room for 31 of them instead of 15 (1792 x 2048 x
// 2304 9.4 us with either).
template <class Cfg>
using DeepRowsCfg = typename std::conditional<Cfg::BM == 128 && Cfg::BN == 128, DeepCfg<128, 128, 2, 4, 3>, Cfg>::type;

template <class Cfg>
hipError_t launch_deep_scales(const GemmParams &p, hipStream_t stream) {
  const bool native = p.a_scale_layout == WAVE_MXFP4_SCALE_MFMA32 && p.b_scale_layout == WAVE_MXFP4_SCALE_MFMA32;
  const bool shuffled = p.a_scale_layout == WAVE_MXFP4_SCALE_E8M0_SHUFFLE && p.b_scale_layout == WAVE_MXFP4_SCALE_E8M0_SHUFFLE;
  if constexpr (Cfg::BM == 64 && Cfg::BN == 64)
    if ((native || shuffled) && p.m <= (p.b_preshuffled ? 32 : 16) && p.tiles_per_split > 16)
      return native ? launch_deep_cfg<DeepStream, kDeepNative>(p, stream) : launch_deep_cfg<DeepStream, kDeepShuffled>(p, stream);
  if (native) return launch_deep_cfg<Cfg, kDeepNative>(p, stream);
  if (shuffled) return launch_deep_cfg<Cfg, kDeepShuffled>(p, stream);
  if (p.tiles_per_split > rows_max_k_tiles<DeepRowsCfg<Cfg>>(8)) return hipErrorInvalidValue;
  return launch_deep_cfg<DeepRowsCfg<Cfg>, kDeepRows>(p, stream);
}

}  // namespace

hipError_t launch_deep_gemm(const GemmParams &p, int shape, hipStream_t stream) {
  return with_deep_shape(shape, hipErrorInvalidValue, [&](auto cfg) { return launch_deep_scales<decltype(cfg)>(p, stream); });
}

int deep_rows_max(int shape, bool fp8) {
  if (fp8) return with_deep8_shape(shape, 0, [](auto cfg) { return rows_max_k_tiles<decltype(cfg)>(4); });
  return with_deep_shape(shape, 0, [](auto cfg) { return rows_max_k_tiles<DeepRowsCfg<decltype(cfg)>>(8); });
}

}  // namespace wave_mxfp4
