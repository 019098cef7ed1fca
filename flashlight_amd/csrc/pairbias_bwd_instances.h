// Launchers of the shared-bias backward (pairbias_bwd_kernel.h): head dims 32 and 64, up to 512 positions.
#pragma once
#include <hip/hip_runtime.h>

#include "pairbias_bwd_kernel.h"

namespace fl {
struct SBShape {
  int nb, waves, lds_bytes;  // 32-row blocks per wave, waves
};
// Eight waves fill a compute unit's registers.  Up to 256 positions of head dim 32 two workgroups of four waves share it
// (two resident entries each, 79 KB); head dim 64 takes one workgroup of up to eight; longer sequences two blocks per wave.
// Two entries stay resident where they fit.
constexpr SBShape pairbias_bwd_shape(int d, int s) {
  const int blocks = (s + 31) / 32;
  SBShape x{};
  x.nb = blocks <= 4 ? 1 : blocks <= 8 ? (d == 32 ? 2 : 1) : 2;
  x.waves = (blocks + x.nb - 1) / x.nb;
  const int slot = x.waves * (x.nb * 128 * d + 512) + 128 * d + 512;
  x.lds_bytes = (2 * slot <= 160 * 1024 ? 2 : 1) * slot;
  return x;
}
hipError_t launch_pairbias_bwd_bf16(int d, const SBShape& shape, bool ahead, const SBParams& p, hipStream_t stream);
hipError_t launch_pairbias_bwd_f16(int d, const SBShape& shape, bool ahead, const SBParams& p, hipStream_t stream);
hipError_t launch_pairbias_bwd_prep_bf16(int d, bool gate, const SBPrepParams& p, hipStream_t stream);
hipError_t launch_pairbias_bwd_prep_f16(int d, bool gate, const SBPrepParams& p, hipStream_t stream);
// bias_f32: the bias gradient's type, fp32 or the element type
hipError_t launch_pairbias_bwd_reduce_bf16(bool bias_f32, const SBParams& p, void* dbias, hipStream_t stream);
hipError_t launch_pairbias_bwd_reduce_f16(bool bias_f32, const SBParams& p, void* dbias, hipStream_t stream);
}  // namespace fl
