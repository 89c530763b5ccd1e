// The deep-ring kernel (mxfp4_gemm_deep.h) on MXFP4 operands.
#include "mxfp4_gemm_deep.h"

namespace wave_mxfp4 {

namespace {

template <class Cfg>
hipError_t launch_deep_scales(const GemmParams &p, hipStream_t stream) {
  if (p.a_scale_layout == WAVE_MXFP4_SCALE_MFMA32 && p.b_scale_layout == WAVE_MXFP4_SCALE_MFMA32)
    return launch_deep_cfg<Cfg, kDeepNative>(p, stream);
  if (p.a_scale_layout == WAVE_MXFP4_SCALE_E8M0_SHUFFLE && p.b_scale_layout == WAVE_MXFP4_SCALE_E8M0_SHUFFLE)
    return launch_deep_cfg<Cfg, kDeepShuffled>(p, stream);
  if (p.tiles_per_split > rows_max_k_tiles<Cfg>(8)) return hipErrorInvalidValue;
  return launch_deep_cfg<Cfg, kDeepRows>(p, stream);
}

}  // namespace

hipError_t launch_deep_gemm(const GemmParams &p, int shape, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_deep_scales<DeepCfg<64, 64, 2, 2, 8>>(p, stream);
    case 1: return launch_deep_scales<DeepCfg<64, 128, 2, 2, 6>>(p, stream);
    case 2: return launch_deep_scales<DeepCfg<128, 128, 2, 4, 4>>(p, stream);
    case 3: return launch_deep_scales<DeepCfg<128, 256, 2, 4, 3>>(p, stream);
    case 4: return launch_deep_scales<DeepCfg<256, 128, 4, 2, 3>>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace wave_mxfp4
