// Kernel instance registry: one launcher per compiled (head dims, tile shape, feature set).
#pragma once
#include <hip/hip_runtime.h>

#include "fwd_kernel.h"

namespace fl {

struct Instance {
  const char* name;
  int dtype;  // element type of q, k, v, o: FL_BF16 (0) or FL_F16 (2)
  int dqk, dv;
  int rw, bn, nw, ns;  // rows per wave, keys per tile, waves per workgroup, K/V tiles resident in LDS
  uint32_t feat;
  int lds_fixed_bytes;  // LDS without the tile list (4 more bytes per key tile)
  int max_groups;  // groups of nw waves a workgroup can be launched with (1, 2 or 4), each with lds_fixed_bytes
  int branches_lds_bytes;  // differential attention: LDS with a group of waves per softmax branch
  hipError_t (*launch)(const KParams&, int groups, int grid, int lds_bytes, hipStream_t);
};

// Defined by instances_table.cpp from the per-file launchers.
extern const Instance kInstances[];
extern const int kNumInstances;

constexpr int kMaxLdsBytes = 160 * 1024;  // per workgroup on gfx950

// Whether a set of features has a kernel with NearCap's polynomial beside that with the exponential (near_cap_pays in api.hip).  With bias operands, whose
// reads and additions are what the loop waits for, it is behind: 2 x 8 x 1024, dense bias and gate, head dim 128, 43.1 us -> 50.0 with the scores in its range
// throughout, 45.9 where they leave it; head dim 64 37.1 -> 36.0 and 38.8.
constexpr bool has_near(uint32_t feat) { return (feat & F_SOFTCAP) && !(feat & (F_DROPOUT | F_BIAS)); }

template <class T, bool NEAR = false>
hipError_t launch_fwd(const KParams& kp, int grid, int lds_bytes, hipStream_t stream) {
  if constexpr (!NEAR && has_near(T::FEAT))
    if (kp.near_cap.last > 0.f) return launch_fwd<T, true>(kp, grid, lds_bytes, stream);
  static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_kernel<T, NEAR>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLdsBytes);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((fwd_kernel<T, NEAR>), dim3(grid), dim3(T::KG * T::NT), lds_bytes, stream, kp);
  return hipGetLastError();
}

template <int DQK, int DV, int RW, int BN, int NW, uint32_t FEAT, int NS>
constexpr int branches_lds_bytes() {
  if constexpr ((FEAT & F_DIFF) != 0) return FwdTraits<DQK, DV, RW, BN, NW, FEAT, NS, bf16_t, 2>::LDS_FIXED_BYTES;
  return 0;
}

// Differential attention with the branches one after the other: 32-key tiles (both results and two tiles of 64 keys have no room in the
// registers), 128 rows; the dump of attended pairs has no other form.
constexpr bool diff_sequential(int bn, int nw) { return bn == 32 && nw == 4; }

// Groups of waves the shape can be launched with (plan_few in api.hip): every instance compiled for them is that many kernels, so
// only the default tiles have them.  Eight waves are two per SIMD, all the registers hold (four groups of four spill).  Differential
// attention (plan_diff): a group per branch, at head dim 128 in 64-key tiles only.
constexpr int max_groups(int dqk, int dv, int rw, int bn, int nw, int ns, uint32_t feat) {
  if (feat & F_DIFF) return feat & F_DUMP || (dqk == 128 && diff_sequential(bn, nw)) ? 1 : 2;
  if (dqk != dv || (dqk != 64 && dqk != 128) || rw != 32 || ns != 2 || (feat & ~(F_ALIBI | F_SOFTCAP | F_DOC))) return 1;
  if (nw == 2) return dqk == 64 ? 4 : 2;
  return nw == 4 && bn == (dqk == 128 && (feat & F_DOC) ? 32 : 64) ? 2 : 1;
}

template <int DQK, int DV, int RW, int BN, int NW, int NS, uint32_t FEAT, class E>
hipError_t launch_fwd_groups(const KParams& kp, int groups, int grid, int lds_bytes, hipStream_t stream) {
  if constexpr ((FEAT & F_DIFF) != 0) {
    if constexpr (max_groups(DQK, DV, RW, BN, NW, NS, FEAT) == 2)
      if (groups == 2) return launch_fwd<FwdTraits<DQK, DV, RW, BN, NW, FEAT, NS, E, 2>>(kp, grid, lds_bytes, stream);
    if constexpr (diff_sequential(BN, NW))
      if (groups == 1) return launch_fwd<FwdTraits<DQK, DV, RW, BN, NW, FEAT, NS, E>>(kp, grid, lds_bytes, stream);
    return hipErrorInvalidValue;
  } else {
  constexpr int MAX = max_groups(DQK, DV, RW, BN, NW, NS, FEAT);
  if constexpr (MAX >= 4)
    if (groups == 4) return launch_fwd<FwdTraits<DQK, DV, RW, BN, NW, FEAT, NS, E, 4>>(kp, grid, lds_bytes, stream);
  if constexpr (MAX >= 2)
    if (groups == 2) return launch_fwd<FwdTraits<DQK, DV, RW, BN, NW, FEAT, NS, E, 2>>(kp, grid, lds_bytes, stream);
  return groups == 1 ? launch_fwd<FwdTraits<DQK, DV, RW, BN, NW, FEAT, NS, E>>(kp, grid, lds_bytes, stream) : hipErrorInvalidValue;
  }
}

}  // namespace fl

// Declares (FL_INSTANCE_DECL) or defines (FL_INSTANCE_DEF) the launcher of one instance for one element type
// (SFX = _bf16 / _f16, ELEM = fl::bf16_t / fl::f16_t), and its row of the table (DT = FL_BF16 / FL_F16).
#define FL_INSTANCE_DECL_(NAME, SFX) \
  namespace fl { hipError_t launch_##NAME##SFX(const KParams&, int, int, int, hipStream_t); }
#define FL_INSTANCE_DECL(NAME, DQK, DV, RW, BN, NW, NS, FEAT) \
  FL_INSTANCE_DECL_(NAME, _bf16) FL_INSTANCE_DECL_(NAME, _f16)
#define FL_INSTANCE_DEF_(NAME, SFX, ELEM, DQK, DV, RW, BN, NW, NS, FEAT)                          \
  namespace fl {                                                                                  \
  hipError_t launch_##NAME##SFX(const KParams& kp, int groups, int grid, int lds, hipStream_t s) { \
    return launch_fwd_groups<DQK, DV, RW, BN, NW, NS, (FEAT), ELEM>(kp, groups, grid, lds, s);     \
  }                                                                                               \
  }
#define FL_INSTANCE_DEF(NAME, SFX, ELEM, ...) FL_INSTANCE_DEF_(NAME, SFX, ELEM, __VA_ARGS__)
#define FL_INSTANCE_ROW_(NAME, SFX, DT, DQK, DV, RW, BN, NW, NS, FEAT) \
  {#NAME, DT, DQK, DV, RW, BN, NW, NS, (FEAT), fl::FwdTraits<DQK, DV, RW, BN, NW, (FEAT), NS>::LDS_FIXED_BYTES, \
   fl::max_groups(DQK, DV, RW, BN, NW, NS, (FEAT)), fl::branches_lds_bytes<DQK, DV, RW, BN, NW, (FEAT), NS>(), &fl::launch_##NAME##SFX},
#define FL_INSTANCE_ROW(NAME, ...) \
  FL_INSTANCE_ROW_(NAME, _bf16, 0, __VA_ARGS__) FL_INSTANCE_ROW_(NAME, _f16, 2, __VA_ARGS__)
