// What the kernels that keep tiles of [rows][D] elements in LDS in TileLayout's two-way image share: the operand reads of the matrix
// instructions (bwd_kernel.h and the shared-bias kernels), and for the shared-bias kernels (pairbias_bwd_kernel.h, stripe_kernel.h),
// whose workgroups walk over batch entries, the place of a workgroup, the rows a transfer brings and where partial sums are parked.
#pragma once
#include "fwd_kernel.h"

namespace fl {

// Operand fragments of v_mfma_f32_32x32x16 for lane (r, h) = (lane % 32, lane / 32)
template <int D, class E>
struct TileOperands {
  typedef E ex8 __attribute__((ext_vector_type(8)));
  typedef E ex4 __attribute__((ext_vector_type(4)));
  using L = TileLayout<D>;
  // row-wise: elements [row][16 ks + 8 h, +8)
  __device__ static __forceinline__ ex8 rows(const unsigned char* tile, int row, int ks, int h) {
    return *reinterpret_cast<const ex8*>(tile + row * (D * 2) + L::swz_kv(row, 2 * ks + h) * 16);
  }
  // transposing: column 32 db + r of the 16 rows of chunk c; slot j is row 16 c + 8 (j / 4) + 4 h + j % 4, the order in which the
  // weights are packed
  __device__ static __forceinline__ ex8 columns(const unsigned char* tile, int c, int db, int lane, int h) {
    ex8 f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i16 = lane % 16, g = (lane / 16) % 2;
      const int row = 16 * c + 8 * j + 4 * h + i16 / 4, col = db * 32 + g * 16 + 4 * (i16 % 4);
      const unsigned char* ap = tile + row * (D * 2) + L::swz_kv(row, col / 8) * 16 + (col % 8) * 2;
      typedef s16x4 __attribute__((address_space(3))) * lds_s16x4_ptr;
      const ex4 b4 = __builtin_bit_cast(ex4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(ap)));
#pragma unroll
      for (int e = 0; e < 4; ++e) f[4 * j + e] = b4[e];
    }
    return f;
  }
  // byte offset of this lane's 16 bytes of the 1 KiB transfer `it` of rows row0 .., rows past the end repeating the last one
  __device__ static __forceinline__ unsigned transfer_offset(int row0, int len, int it, int64_t stride, int lane) {
    constexpr int RPT = 512 / D;  // rows per transfer
    const int row = it * RPT + lane / L::CPR;
    return (uint32_t)min(row0 + row, len - 1) * ((uint32_t)stride * 2u) + (uint32_t)(L::swz_kv(row, lane % L::CPR) * 16);
  }
  // partial sums of one set: [row][D] floats, 16-byte chunks XOR-swizzled with the row
  __device__ static __forceinline__ int park_at(int row, int c) { return row * (D * 4) + ((c ^ row) & (D / 4 - 1)) * 16; }
};

// Brings the cache line at each lane's address into the L2, and four bytes of it into 256 bytes of LDS that nothing reads.
__device__ __forceinline__ void touch(uint64_t lane_address, unsigned lds_base) {
  const unsigned lds_base_uniform = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(lane_address), "s"(lds_base_uniform) : "m0");
}

// Workgroup -> (group of batch entries that share the bias, chunk of them, head, stripe): the stripes of one (chunk, head) read the
// same tensors and stay on one XCD.  unit: (group, chunk, head) as one number; `none`: a workgroup past the last of them.  neighbours: an XCD takes
// an eighth of the units that follow each other, otherwise every eighth unit (forward_neighbours and gradient_neighbours in api.hip).
struct StripePlace {
  int tile, unit;
  template <class P, class Block>
  __device__ __forceinline__ StripePlace(const P& p, const Block block, const bool neighbours) {
    const int x = block % 8, i = block / 8, each = (p.groups * p.chunks * p.H + 7) / 8, of_x = i / p.tiles;
    tile = i % p.tiles;
    unit = !neighbours ? of_x * 8 + x : of_x < each ? x * each + of_x : 8 * each;
  }
  template <class P>
  __device__ __forceinline__ bool none(const P& p) const { return unit >= p.groups * p.chunks * p.H; }
};

}  // namespace fl
