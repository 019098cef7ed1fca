// Launchers of the backward kernels: one translation unit per (head dim, feature set), both roles in it.
#pragma once
#include <hip/hip_runtime.h>

#include "bwd_kernel.h"
#include "instances.h"

namespace fl {

struct BwdInstance {
  int d;
  uint32_t feat;
  int dtype;  // element type of q, k, v, o, dout and the gradients: FL_BF16 (0) or FL_F16 (2)
  hipError_t (*launch_dq)(const BParams&, hipStream_t);
  hipError_t (*launch_dkv)(const BParams&, hipStream_t);
  hipError_t (*launch_both)(const BParams&, hipStream_t);
  hipError_t (*launch_delta)(const BParams&, hipStream_t);
};

extern const BwdInstance kBwdInstances[];
extern const int kNumBwdInstances;

template <class K>
hipError_t allow_lds(K kernel) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLdsBytes);
}

template <class T>
hipError_t launch_bwd_role(const BParams& bp, int64_t tiles, hipStream_t stream) {
  static const hipError_t attr = allow_lds(&bwd_kernel<T>);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(bwd_kernel<T>, dim3((unsigned)tiles), dim3(T::NT), T::LDS_BYTES, stream, bp);
  return hipGetLastError();
}

inline int64_t bwd_q_tiles(const BParams& bp) { return (int64_t)bp.B * bp.Hq * ((bp.Lq + 127) / 128); }
inline int64_t bwd_k_tiles(const BParams& bp) { return (int64_t)bp.B * bp.Hkv * ((bp.Lk + 127) / 128); }

// dQ, dK and dV in one launch, and the sums of the tiles that were split.
template <int D, uint32_t FEAT, class E>
hipError_t launch_bwd_both(const BParams& bp, hipStream_t stream) {
  using TQ = BwdTraits<D, ROLE_DQ, FEAT, E, true>;
  using TKV = BwdTraits<D, ROLE_DKV, FEAT, E, true>;
  constexpr int lds = TQ::LDS_BYTES > TKV::LDS_BYTES ? TQ::LDS_BYTES : TKV::LDS_BYTES;
  static const hipError_t attr = allow_lds(&bwd_both_kernel<TQ, TKV>);
  if (attr != hipSuccess) return attr;
  const int64_t q_tiles = bwd_q_tiles(bp), k_tiles = bwd_k_tiles(bp);
  hipLaunchKernelGGL((bwd_both_kernel<TQ, TKV>), dim3((unsigned)(q_tiles * bp.splits_dq + k_tiles * bp.splits)), dim3(TQ::NT), lds, stream, bp);
  const hipError_t e = hipGetLastError();
  const int64_t blocks = (bp.splits > 1 ? 8 * k_tiles : 0) + (bp.splits_dq > 1 ? 4 * q_tiles : 0);
  if (e != hipSuccess || blocks == 0) return e;
  hipLaunchKernelGGL((bwd_split_sum_kernel<TQ, TKV>), dim3((unsigned)blocks), dim3(256), 0, stream, bp);
  return hipGetLastError();
}

template <int DV, class E>
hipError_t launch_delta(const BParams& bp, hipStream_t stream) {
  const int rows_per_block = 256 / (DV / 8), blocks = (bp.Lq + rows_per_block - 1) / rows_per_block;
  BParams p = bp;
  p.by_delta_blocks = Div::by(blocks);
  hipLaunchKernelGGL((bwd_delta_kernel<DV, E>), dim3((unsigned)((int64_t)bp.B * bp.Hq * blocks)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace fl

// (D, FEAT) pairs with compiled backward kernels.  FEAT 3 = ALiBi and/or soft-cap (either may be off at run time; at head dims 64 and 128
// a soft-cap, with or without ALiBi), 1 = ALiBi alone (64 and 128),
// 4 = bias operands, 8 = document ids in the element predicate, 11 = document ids with ALiBi and/or a soft-cap,
// 7, 12, 15 = bias operands with ALiBi / soft-cap, with document ids, with both,
// 128 + any of these = the same with dropout (head dims 64 and 128).
#define FL_BWD_LIST(X) X(32, 0) X(32, 3) X(32, 4) X(32, 7) X(32, 8) X(32, 11) X(32, 12) X(32, 15) X(64, 0) X(64, 1) X(64, 3) X(64, 4) X(64, 7) X(64, 8) X(64, 11) X(64, 12) X(64, 15) X(64, 128) X(64, 131) X(64, 132) X(64, 135) X(64, 136) X(64, 139) X(64, 140) X(64, 143) X(128, 0) X(128, 1) X(128, 3) X(128, 4) X(128, 7) X(128, 8) X(128, 11) X(128, 12) X(128, 15) X(128, 128) X(128, 131) X(128, 132) X(128, 135) X(128, 136) X(128, 139) X(128, 140) X(128, 143)

// Every (D, FEAT) pair is compiled for bf16 and for fp16 elements (suffix _bf16 / _f16).
#define FL_BWD_DECL_(D, FEAT, SFX)                                            \
  namespace fl {                                                              \
  hipError_t launch_bwd_dq_##D##_##FEAT##SFX(const BParams&, hipStream_t);    \
  hipError_t launch_bwd_dkv_##D##_##FEAT##SFX(const BParams&, hipStream_t);   \
  hipError_t launch_bwd_both_##D##_##FEAT##SFX(const BParams&, hipStream_t);  \
  hipError_t launch_bwd_delta_##D##_##FEAT##SFX(const BParams&, hipStream_t); \
  }
#define FL_BWD_DECL(D, FEAT) FL_BWD_DECL_(D, FEAT, _bf16) FL_BWD_DECL_(D, FEAT, _f16)
#define FL_BWD_DEF(D, FEAT, SFX, ELEM)                                                                              \
  namespace fl {                                                                                                    \
  hipError_t launch_bwd_dq_##D##_##FEAT##SFX(const BParams& bp, hipStream_t s) {                                    \
    return launch_bwd_role<BwdTraits<D, ROLE_DQ, FEAT, ELEM>>(bp, bwd_q_tiles(bp), s);                              \
  }                                                                                                                 \
  hipError_t launch_bwd_dkv_##D##_##FEAT##SFX(const BParams& bp, hipStream_t s) {                                   \
    if constexpr (D == 128 && FEAT == 0) {                                                                          \
      if (bp.dkv_own == 256) return launch_bwd_role<BwdTraits<D, ROLE_DKV, FEAT, ELEM, false, true>>(bp, (int64_t)bp.B * bp.Hkv * ((bp.Lk + 255) / 256), s); \
    }                                                                                                               \
    return launch_bwd_role<BwdTraits<D, ROLE_DKV, FEAT, ELEM>>(bp, bwd_k_tiles(bp), s);                             \
  }                                                                                                                 \
  hipError_t launch_bwd_both_##D##_##FEAT##SFX(const BParams& bp, hipStream_t s) { return launch_bwd_both<D, FEAT, ELEM>(bp, s); } \
  hipError_t launch_bwd_delta_##D##_##FEAT##SFX(const BParams& bp, hipStream_t s) { return launch_delta<D, ELEM>(bp, s); } \
  }
#define FL_BWD_ROW_(D, FEAT, SFX, DT) \
  {D, FEAT, DT, &fl::launch_bwd_dq_##D##_##FEAT##SFX, &fl::launch_bwd_dkv_##D##_##FEAT##SFX, \
   &fl::launch_bwd_both_##D##_##FEAT##SFX, &fl::launch_bwd_delta_##D##_##FEAT##SFX},
#define FL_BWD_ROW(D, FEAT) FL_BWD_ROW_(D, FEAT, _bf16, 0) FL_BWD_ROW_(D, FEAT, _f16, 2)
