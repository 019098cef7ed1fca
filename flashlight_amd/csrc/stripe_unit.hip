// The shared-bias stripe forward (stripe_kernel.h), every compiled shape for one element type.
// -DFL_INST_F16=1 compiles the fp16 set instead of the bf16 one.
#include "stripe_instances.h"

namespace fl {
namespace {
template <int D, int QB, int NW, bool ROW, class E, bool NEIGHBOURS>
hipError_t launch_one(const StripeParams& p, hipStream_t stream) {
  using T = StripeTraits<D, QB, 2, NW, ROW, E, NEIGHBOURS>;
  static_assert(T::LDS_BYTES == stripe_shape(D, 64 * NW, ROW).lds_bytes && T::PER_CU == stripe_shape(D, 64 * NW, ROW).per_cu, "one rule");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&stripe_kernel<T>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS_BYTES);
  if (attr != hipSuccess) return attr;
  const int64_t units = (int64_t)p.groups * p.chunks * p.H;
  hipLaunchKernelGGL((stripe_kernel<T>), dim3((unsigned)((units + 7) / 8 * 8 * p.tiles)), dim3(64 * NW), T::LDS_BYTES, stream, p);
  return hipGetLastError();
}
template <int D, int QB, bool ROW, class E, int NW = 8>
hipError_t launch_waves(int waves, bool neighbours, const StripeParams& p, hipStream_t stream) {
  if constexpr (NW > 0) {
    if (waves == NW) return neighbours ? launch_one<D, QB, NW, ROW, E, true>(p, stream) : launch_one<D, QB, NW, ROW, E, false>(p, stream);
    return launch_waves<D, QB, ROW, E, NW - 1>(waves, neighbours, p, stream);
  }
  return hipErrorInvalidValue;
}
template <class E>
hipError_t launch_any(int d, int waves, bool neighbours, const StripeParams& p, hipStream_t stream) {
  if (d == 32) return p.row ? launch_waves<32, 2, true, E>(waves, neighbours, p, stream) : launch_waves<32, 2, false, E>(waves, neighbours, p, stream);
  if (d == 64) return p.row ? launch_waves<64, 1, true, E>(waves, neighbours, p, stream) : launch_waves<64, 1, false, E>(waves, neighbours, p, stream);
  return hipErrorInvalidValue;
}
}  // namespace

#if defined(FL_INST_F16) && FL_INST_F16
hipError_t launch_stripe_f16(int d, int waves, bool neighbours, const StripeParams& p, hipStream_t stream) {
  return launch_any<f16_t>(d, waves, neighbours, p, stream);
}
#else
hipError_t launch_stripe_bf16(int d, int waves, bool neighbours, const StripeParams& p, hipStream_t stream) {
  return launch_any<bf16_t>(d, waves, neighbours, p, stream);
}
#endif
}  // namespace fl
