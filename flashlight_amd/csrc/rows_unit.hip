// The few-rows forward (rows_kernel.h), every compiled shape for one element type.
// -DFL_INST_F16=1 compiles the fp16 set instead of the bf16 one.
#include "rows_instances.h"

namespace fl {
namespace {
template <int D, int QT, uint32_t MOD, class E>
hipError_t launch_one(const RParams& p, int grid, int waves, hipStream_t stream) {
  using T = RowsTraits<D, QT, MOD, E>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&rows_kernel<T>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, rows_lds_bytes(D, QT, 8));
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((rows_kernel<T>), dim3(grid), dim3(64 * waves), rows_lds_bytes(D, QT, waves), stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.chunks == 1) return e;
  hipLaunchKernelGGL((rows_merge_kernel<D, T::RB, E>), dim3(p.units * p.rows), dim3(256), 0, stream, p);
  return hipGetLastError();
}
template <int D, int QT, class E>
hipError_t launch_mod(uint32_t mod, const RParams& p, int grid, int waves, hipStream_t stream) {
  if (mod == 0) return launch_one<D, QT, 0, E>(p, grid, waves, stream);
  if (mod == F_BIAS) return launch_one<D, QT, F_BIAS, E>(p, grid, waves, stream);
  return launch_one<D, QT, F_ALIBI | F_SOFTCAP, E>(p, grid, waves, stream);
}
template <class E>
hipError_t launch_any(int d, int qt, uint32_t mod, const RParams& p, int grid, int waves, hipStream_t stream) {
  if (d == 64) return qt == 1 ? launch_mod<64, 1, E>(mod, p, grid, waves, stream) : launch_mod<64, 2, E>(mod, p, grid, waves, stream);
  if (d == 128 && qt == 1) return launch_mod<128, 1, E>(mod, p, grid, waves, stream);
  return hipErrorInvalidValue;
}
}  // namespace

#if defined(FL_INST_F16) && FL_INST_F16
hipError_t launch_rows_f16(int d, int qt, uint32_t mod, const RParams& p, int grid, int waves, hipStream_t stream) {
  return launch_any<f16_t>(d, qt, mod, p, grid, waves, stream);
}
#else
hipError_t launch_rows_bf16(int d, int qt, uint32_t mod, const RParams& p, int grid, int waves, hipStream_t stream) {
  return launch_any<bf16_t>(d, qt, mod, p, grid, waves, stream);
}
#endif
}  // namespace fl
