// Launchers of the shared-bias stripe forward (stripe_kernel.h): head dims 32 and 64, up to 512 queries and keys, bf16 or fp16.
#pragma once
#include <hip/hip_runtime.h>

#include "stripe_kernel.h"

namespace fl {
struct StripeShape {
  int qb, waves, lds_bytes, per_cu;  // 32-row blocks of queries per stripe; workgroups that a compute unit holds
};
// Two blocks of 32 keys per wave; two of queries at head dim 32, one at 64 (registers).
constexpr StripeShape stripe_shape(int d, int lk, bool row) {
  StripeShape x{d == 32 ? 2 : 1, (lk + 63) / 64, 0, 0};
  const int slot = x.waves * 256 * d + x.qb * 64 * d, rest = x.waves * ((row ? 512 : 0) + x.qb * 256);
  x.lds_bytes = (2 * slot + rest <= 160 * 1024 ? 2 : 1) * slot + rest;
  x.per_cu = 8 / x.waves < 160 * 1024 / x.lds_bytes ? 8 / x.waves : 160 * 1024 / x.lds_bytes;
  return x;
}
hipError_t launch_stripe_bf16(int d, int waves, bool neighbours, const StripeParams& p, hipStream_t stream);
hipError_t launch_stripe_f16(int d, int waves, bool neighbours, const StripeParams& p, hipStream_t stream);
}  // namespace fl
