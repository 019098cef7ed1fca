// The shared-bias backward (pairbias_bwd_kernel.h), every compiled shape for one element type.
// -DFL_INST_F16=1 compiles the fp16 set instead of the bf16 one.
#include "pairbias_bwd_instances.h"

namespace fl {
namespace {
template <int D, int NB, int NW, bool ROWB, class E, bool AHEAD>
hipError_t launch_one(const SBParams& p, hipStream_t stream) {
  using TQ = SBTraits<D, 0, NB, NW, ROWB, E, AHEAD>;
  using TKV = SBTraits<D, 1, NB, NW, ROWB, E, AHEAD>;
  static_assert(TQ::SLOTS * TQ::SLOT_BYTES == pairbias_bwd_shape(D, 32 * NB * NW).lds_bytes, "one rule");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&pairbias_bwd_kernel<TQ, TKV>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, TQ::LDS_BYTES);
  if (attr != hipSuccess) return attr;
  const int64_t units = (int64_t)p.groups * p.chunks * p.H;
  const int64_t grid = 2 * ((units + 7) / 8 * 8 * p.tiles);
  hipLaunchKernelGGL((pairbias_bwd_kernel<TQ, TKV>), dim3((unsigned)grid), dim3(64 * NW), TQ::LDS_BYTES, stream, p);
  return hipGetLastError();
}
// the shapes that pairbias_bwd_shape names
template <int D, bool ROWB, class E, int BLOCKS = 16>
hipError_t launch_shape(const SBShape& shape, bool ahead, const SBParams& p, hipStream_t stream) {
  if constexpr (BLOCKS > 0) {
    constexpr SBShape x = pairbias_bwd_shape(D, 32 * BLOCKS);
    if (shape.nb == x.nb && shape.waves == x.waves)
      return ahead ? launch_one<D, x.nb, x.waves, ROWB, E, true>(p, stream) : launch_one<D, x.nb, x.waves, ROWB, E, false>(p, stream);
    return launch_shape<D, ROWB, E, BLOCKS - 1>(shape, ahead, p, stream);
  }
  return hipErrorInvalidValue;
}
template <class E>
hipError_t launch_any(int d, const SBShape& shape, bool ahead, const SBParams& p, hipStream_t stream) {
  if (d == 32) return p.rowb ? launch_shape<32, true, E>(shape, ahead, p, stream) : launch_shape<32, false, E>(shape, ahead, p, stream);
  if (d == 64) return p.rowb ? launch_shape<64, true, E>(shape, ahead, p, stream) : launch_shape<64, false, E>(shape, ahead, p, stream);
  return hipErrorInvalidValue;
}
template <int D, bool GATE, class E>
hipError_t launch_prep_one(const SBPrepParams& p, hipStream_t stream) {
  const int64_t rows = (int64_t)p.B * p.S * p.H, per_block = 256 / (D / 8);
  hipLaunchKernelGGL((pairbias_bwd_prep_kernel<D, GATE, E>), dim3((unsigned)((rows + per_block - 1) / per_block)), dim3(256), 0, stream, p);
  return hipGetLastError();
}
template <class E>
hipError_t launch_prep(int d, bool gate, const SBPrepParams& p, hipStream_t stream) {
  if (d == 32) return gate ? launch_prep_one<32, true, E>(p, stream) : launch_prep_one<32, false, E>(p, stream);
  if (d == 64) return gate ? launch_prep_one<64, true, E>(p, stream) : launch_prep_one<64, false, E>(p, stream);
  return hipErrorInvalidValue;
}
template <class OUT>
hipError_t launch_reduce_one(const SBParams& p, void* dbias, hipStream_t stream) {
  const int64_t rows = (int64_t)p.H * p.S, total4 = p.groups * rows * (p.s_pad / 4);
  hipLaunchKernelGGL((pairbias_bwd_reduce_kernel<OUT>), dim3((unsigned)((total4 + 255) / 256)), dim3(256), 0, stream, p.dbias_part,
                     static_cast<OUT*>(dbias), p.chunks, rows, p.S, p.s_pad, total4);
  return hipGetLastError();
}
}  // namespace

#if defined(FL_INST_F16) && FL_INST_F16
#define FL_SB_NAME(x) x##_f16
typedef f16_t sb_elem;
#else
#define FL_SB_NAME(x) x##_bf16
typedef bf16_t sb_elem;
#endif
hipError_t FL_SB_NAME(launch_pairbias_bwd)(int d, const SBShape& shape, bool ahead, const SBParams& p, hipStream_t stream) {
  return launch_any<sb_elem>(d, shape, ahead, p, stream);
}
hipError_t FL_SB_NAME(launch_pairbias_bwd_prep)(int d, bool gate, const SBPrepParams& p, hipStream_t stream) {
  return launch_prep<sb_elem>(d, gate, p, stream);
}
hipError_t FL_SB_NAME(launch_pairbias_bwd_reduce)(bool bias_f32, const SBParams& p, void* dbias, hipStream_t stream) {
  return bias_f32 ? launch_reduce_one<float>(p, dbias, stream) : launch_reduce_one<sb_elem>(p, dbias, stream);
}
}  // namespace fl
