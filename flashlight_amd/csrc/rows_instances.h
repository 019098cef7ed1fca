// Launchers of the few-rows forward (rows_kernel.h): head dim 64 with one or two 16-row blocks per wave, head dim 128 with
// one (two need 340 bytes of scratch per lane); plain, ALiBi / soft-cap, row biases.
#pragma once
#include "rows_kernel.h"

namespace fl {
inline bool rows_has_shape(int d) { return d == 64 || d == 128; }
inline int rows_lds_bytes(int d, int qt, int waves) { return waves * 16 * qt * (d + 4 + 2) * 4; }
// qt: 16-row blocks per wave
hipError_t launch_rows_bf16(int d, int qt, uint32_t mod, const RParams& p, int grid, int waves, hipStream_t stream);
hipError_t launch_rows_f16(int d, int qt, uint32_t mod, const RParams& p, int grid, int waves, hipStream_t stream);
}  // namespace fl
