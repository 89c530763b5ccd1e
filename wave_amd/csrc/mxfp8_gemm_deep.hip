// The deep-ring kernel (mxfp4_gemm_deep.h) on MXFP8 operands, and on 8-bit against 4-bit ones.
#include "mxfp4_gemm_deep.h"

namespace wave_mxfp4 {

namespace {

// The ring of the small tile is 8 K tiles deep behind a launch that re-lays the scales (a long K:
// 0.97 of the time with four, mean of 8 calls) and 4 where the workgroups stage them (5.6 us against 6.5 at 1024 x 1024 x 1024, 0.94
// of the time over 430 random calls); 128x128 with three K tiles instead of four loses 1 - 3 %.
template <class Cfg, int FMT_A, int FMT_B>
hipError_t launch_deep8_scales(const GemmParams &p, hipStream_t stream) {
  if constexpr (Cfg::BM == 64)
    if (p.a_scale_layout == WAVE_MXFP4_SCALE_MFMA32) return launch_deep_cfg<DeepCfg<64, 64, 2, 2, 8>, kDeepNative, FMT_A, FMT_B>(p, stream);
  if constexpr (Cfg::BM != 64)
    if (p.a_scale_layout == WAVE_MXFP4_SCALE_MFMA32) return launch_deep_cfg<Cfg, kDeepNative, FMT_A, FMT_B>(p, stream);
  if (p.tiles_per_split > rows_max_k_tiles<Cfg>(4)) return hipErrorInvalidValue;
  return launch_deep_cfg<Cfg, kDeepRows, FMT_A, FMT_B>(p, stream);
}

// a_fmt, b_fmt: 0 = e4m3, 1 = e5m2, 2 = e2m1 (one operand at most)
template <class Cfg>
hipError_t launch_deep8_formats(const GemmParams &p, int a_fmt, int b_fmt, hipStream_t stream) {
  switch (a_fmt * 3 + b_fmt) {
    case 0: return launch_deep8_scales<Cfg, 0, 0>(p, stream);
    case 1: return launch_deep8_scales<Cfg, 0, 1>(p, stream);
    case 2: return launch_deep8_scales<Cfg, 0, 4>(p, stream);
    case 3: return launch_deep8_scales<Cfg, 1, 0>(p, stream);
    case 4: return launch_deep8_scales<Cfg, 1, 1>(p, stream);
    case 5: return launch_deep8_scales<Cfg, 1, 4>(p, stream);
    case 6: return launch_deep8_scales<Cfg, 4, 0>(p, stream);
    case 7: return launch_deep8_scales<Cfg, 4, 1>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_deep_gemm_fp8(const GemmParams &p, int shape, int a_fmt, int b_fmt, hipStream_t stream) {
  return with_deep8_shape(shape, hipErrorInvalidValue,
                          [&](auto cfg) { return launch_deep8_formats<decltype(cfg)>(p, a_fmt, b_fmt, stream); });
}

}  // namespace wave_mxfp4
