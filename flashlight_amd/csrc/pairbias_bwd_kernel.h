// Backward of attention with one dense bias shared by several consecutive batch entries (the Evoformer's row attention:
// a pair bias over all rows of an alignment), with an optional bias row per batch entry and an optional sigmoid gate.
//
// What bounded it in the general backward (bwd_kernel.h, F_BIAS) were the bias's two ends: a 2-byte global load per score
// in both roles, and the bias gradient as a dense fp32 array of every batch entry's score gradients (4 bytes per score
// cleared, written, and read back by a reduction; 268 MB each for 128 x 8 x 256 x 256).  Here a workgroup stays with one
// 32-row stripe of one head's score matrix and walks over the batch entries: the bias of the stripe is read once into
// registers, and in the role that produces dQ the score gradients of all its entries add up in registers too, so that
// the bias gradient leaves as one fp32 tile per workgroup, summed over the few workgroups that share a stripe by
// pairbias_bwd_reduce_kernel in a fixed order (no atomics).
//
// Two roles, as in the general backward, every product with the streamed tile as the MFMA A operand:
//   ROLE_DQ   owns 32 queries, streams all keys:     S^T = K.Q^T, dP^T = V.dO^T, dQ^T += K^T.dS^T, dBias += dS^T
//   ROLE_DKV  owns 32 keys, streams all queries:     S = Q.K^T,   dP = dO.V^T,   dK^T += Q^T.dS,   dV^T += dO^T.P
// The waves of a workgroup split the streamed rows (NB blocks of 32 each), fetch their own rows into their own part of LDS
// (no barrier for them), and add up their partial dQ / dK, dV through LDS once per batch entry.  The next entry's rows are
// on their way while one is worked on.  The sequence has at most 512 positions.
//
// Measured, 128 x 8 x 256 x 256, head dim 32, mask row and gate, bf16, whole step: 852 -> 168 us (ROLE_DQ 325 -> 46, ROLE_DKV
// 232 -> 56, row sums and gate 150 -> 16, clearing and summing the bias gradient 97 -> 4), then both roles in one launch, wave counts
// compiled in (the sums over a run-time count were loops) and waits that leave the stores outstanding: 103 -> 83; 2 x 230 x 4 x 192 x
// 192: 139 -> 107; 65 x 4 x 384 x 384, head dim 64: 244 -> 119; 256 x 8 x 384 x 384: 811 -> 545.  Per score ten vector
// instructions are left (seven make the weight and its gradient, the rest operands and the sums over the waves), and no global
// load, conversion or store; what bounds the roles is the chain an entry goes through (tiles, two products, weights, products, sums
// over the waves) with two waves per SIMD to cover it.  Two blocks per wave in four waves beat one in eight (67 and 93 us for the two
// roles against 46 and 56: the sums over the waves cost more than the occupancy gains).
#pragma once
#include "tile_operands.h"

namespace fl {

struct SBParams {
  const bf16_t *q, *k, *v, *dout;  // dout: already multiplied by the gate
  const float *lse, *delta;        // [B, H, S]; delta: minus rowsum(dO o O)
  const float* rowb;               // [B, S] in units of the unscaled product, or null
  bf16_t *dq, *dk, *dv;
  int64_t qs[3], ks[3], vs[3], dos[3], dqs[3], dks[3], dvs[3];  // element strides: batch, head, seq
  const void* bias;
  int64_t bs[3];                   // group, head, query (key stride 1)
  int32_t bias_f32;
  int32_t bias_vec;                // rows of the bias may be read four keys at a time
  int32_t B, H, S;
  int32_t div, groups, chunks, chunk_len;  // batch entries per bias; groups = B / div; entries are cut into chunks of chunk_len
  int32_t tiles;                   // 32-row stripes
  int32_t neighbours;              // see StripePlace
  int32_t s_pad;                   // row length of the partial bias gradient (S rounded up to 4)
  float scale, scale_log2;
  float* dbias_part;               // [groups][chunks][H][S][s_pad], or null: no gradient of the bias wanted
};

// rows of an operand that are not in the sequence repeat the last one; their weights are 0 (their bias is -inf)
// AHEAD: rows are touched two entries ahead of their use
template <int D_, int ROLE_, int NB_, int NW_, bool ROWB_, class Elem_, bool AHEAD_ = false>
struct SBTraits {
  using Elem = Elem_;
  static constexpr int D = D_, ROLE = ROLE_, NB = NB_, NW = NW_;
  static constexpr bool ROWB = ROWB_, DQ = ROLE_ == 0;
  static constexpr int KS = D / 16, DB = D / 32;
  static constexpr int T_BYTES = NB * 32 * D * 2;        // one streamed operand of one wave
  static constexpr int O_BYTES = 32 * D * 2;             // one owned operand
  static constexpr int PARK = 32 * D * 4;                // partial sums of one accumulator set of one wave
  // per wave and slot: both streamed operands, and the fp32 values per streamed row (LSE and Delta in ROLE_DKV, the bias
  // row in ROLE_DQ): two areas of 64 floats
  static constexpr int W_BYTES = 2 * T_BYTES + 2 * 256;
  static constexpr int S_OWN = 2 * O_BYTES + 2 * 256;    // per slot: owned operands and their values per row
  static constexpr int TPW = T_BYTES / 1024;             // 1 KiB transfers per streamed operand
  static constexpr int SLOT_BYTES = NW * W_BYTES + S_OWN;  // one batch entry
  // tiles of batch entries resident in LDS
  static constexpr int SLOTS = 2 * SLOT_BYTES <= 160 * 1024 ? 2 : 1;
  static constexpr bool AHEAD = AHEAD_;
  static constexpr int LDS_BYTES = SLOTS * SLOT_BYTES + (AHEAD ? 256 : 0);  // (and where touch() puts what nothing reads)
  // the partial sums go where the consumed tiles were: both sets at once when a wave's two tiles have room for them
  static constexpr bool ONE_PASS = DQ || 2 * T_BYTES >= 2 * PARK;
};

// a store that the waits count; the idle cycles keep it five wait states behind a vector instruction that wrote the address (see dma16)
__device__ __forceinline__ void sb_store8(uint64_t sbase, unsigned voff, u32x2 data) {
  asm volatile("s_nop 4\n\tglobal_store_dwordx2 %0, %1, %2" ::"v"(voff), "v"(data), "s"(sbase) : "memory");
}

// One workgroup's share of a role: workgroup `block` of the role's.
template <class T>
__device__ __forceinline__ void pairbias_bwd_stripe(const SBParams& p, const int block) {
  constexpr int D = T::D, NB = T::NB, KS = T::KS, DB = T::DB, NW = T::NW;
  constexpr bool kDQ = T::DQ, kRowB = T::ROWB;
  constexpr float kLog2e = 1.4426950408889634f;
  using E = typename T::Elem;
  typedef E ex8 __attribute__((ext_vector_type(8)));
  typedef E ex4 __attribute__((ext_vector_type(4)));
  using Ops = TileOperands<D, E>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int r = lane % 32, h = lane / 32;

  const StripePlace place(p, block, p.neighbours != 0);
  if (place.none(p)) return;  // (before any barrier)
  const int tile = place.tile, head = place.unit % p.H, gc = place.unit / p.H, chunk = gc % p.chunks, group = gc / p.chunks;
  const int n0 = group * p.div + chunk * p.chunk_len, n1 = min(group * p.div + p.div, n0 + p.chunk_len);
  const int o0 = tile * 32, S = p.S;
  const int own = o0 + r;                 // this lane's query (ROLE_DQ) or key
  const int w0 = wave * NB * 32;          // first streamed row of this wave

  // ---- the stripe's bias in log2 units, -inf outside the score matrix: register (b, i) is streamed row
  // w0 + 32 b + 8 (i / 4) + 4 h + i % 4 against this lane's owned row
  float bias[NB][16];
  {
    const int64_t base = (int64_t)group * p.bs[0] + (int64_t)head * p.bs[1];
    // (one loop per element type, and the loads before anything looks at them: 16 NB loads in flight together)
    auto fetch = [&](auto* src) FL_INLINE {
      using X = std::remove_const_t<std::remove_pointer_t<decltype(src)>>;
      typedef X x4 __attribute__((ext_vector_type(4)));
      X x[NB][16];
      if (kDQ && p.bias_vec) {  // four consecutive keys of the lane's query in one load (5 -> 1 us for NB = 2)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const x4 v = *reinterpret_cast<const x4*>(src + base + (int64_t)min(own, S - 1) * p.bs[2] + min(w0 + 32 * b + 8 * g + 4 * h, S - 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) x[b][4 * g + e] = v[e];
          }
      } else {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int st = w0 + 32 * b + 8 * (i / 4) + 4 * h + i % 4;
            x[b][i] = src[base + (int64_t)min(kDQ ? own : st, S - 1) * p.bs[2] + min(kDQ ? st : own, S - 1)];
          }
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int st = w0 + 32 * b + 8 * (i / 4) + 4 * h + i % 4;
          bias[b][i] = (st < S && own < S) ? (float)x[b][i] * kLog2e : -INFINITY;
        }
    };
    if (p.bias_f32) fetch(static_cast<const float*>(p.bias));
    else fetch(static_cast<const E*>(p.bias));
  }
  float db[kDQ ? NB : 1][16];
  if constexpr (kDQ) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) db[b][i] = 0.f;
  }

  // ---- transfers of a batch entry into ring slot `slot`.  The per-lane offsets do not change from entry to entry and the
  // scalar base addresses advance by one batch stride: per entry a transfer costs its issue and nothing else.
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem);
  constexpr unsigned w_bytes = T::W_BYTES * NW, slot_bytes = T::SLOT_BYTES;
  struct Operand {
    uint64_t at;   // address of the next entry's [S][D] rows of this head
    uint64_t step;
  };
  auto operand = [&](const void* base, const int64_t (&st)[3]) FL_INLINE -> Operand {
    return {uniform_ptr(static_cast<const bf16_t*>(base) + (int64_t)n0 * st[0] + (int64_t)head * st[1]), (uint64_t)uniform_i64(st[0] * 2)};
  };
  Operand st1 = operand(kDQ ? p.k : p.q, kDQ ? p.ks : p.qs), st2 = operand(kDQ ? p.v : p.dout, kDQ ? p.vs : p.dos);
  Operand ow1 = operand(kDQ ? p.q : p.k, kDQ ? p.qs : p.ks), ow2 = operand(kDQ ? p.dout : p.v, kDQ ? p.dos : p.vs);
  unsigned off1[T::TPW], off2[T::TPW];
#pragma unroll
  for (int it = 0; it < T::TPW; ++it) {
    off1[it] = Ops::transfer_offset(w0, S, it, kDQ ? p.ks[2] : p.qs[2], lane);
    off2[it] = Ops::transfer_offset(w0, S, it, kDQ ? p.vs[2] : p.dos[2], lane);
  }
  // the owned rows: 2 OT transfers shared out over the waves (one wave takes several where there are fewer waves)
  constexpr int OT = T::O_BYTES / 1024, OPW = (2 * OT + NW - 1) / NW;
  unsigned ooff[OPW];
#pragma unroll
  for (int j = 0; j < OPW; ++j) {
    const int x = j * NW + wave;
    ooff[j] = x < OT ? Ops::transfer_offset(o0, S, x, kDQ ? p.qs[2] : p.ks[2], lane) : Ops::transfer_offset(o0, S, x - OT, kDQ ? p.dos[2] : p.vs[2], lane);
  }
  // per-row fp32 values: LSE and Delta rows of this head, the bias row of the entry
  uint64_t lse_at = uniform_ptr(p.lse + ((int64_t)n0 * p.H + head) * S), del_at = uniform_ptr(p.delta + ((int64_t)n0 * p.H + head) * S);
  uint64_t row_at = kRowB ? uniform_ptr(p.rowb + (int64_t)n0 * S) : 0;
  const uint64_t stat_step = (uint64_t)p.H * S * 4u, row_step = (uint64_t)S * 4u;
  const unsigned st_row = (uint32_t)min(w0 + lane, S - 1) * 4u, ow_row = (uint32_t)min(o0 + lane, S - 1) * 4u;
  auto load_entry = [&](int slot) FL_INLINE {
    const unsigned s0 = lds0 + slot * slot_bytes, mine = s0 + wave * T::W_BYTES, own_at = s0 + w_bytes;
#pragma unroll
    for (int it = 0; it < T::TPW; ++it) {
      dma16<3>(st1.at, off1[it], mine + it * 1024);
      dma16<3>(st2.at, off2[it], mine + T::T_BYTES + it * 1024);
    }
    if constexpr (kDQ) {
      if constexpr (kRowB) dma4<3>(row_at, st_row, mine + 2 * T::T_BYTES);
    } else {
      dma4<3>(lse_at, st_row, mine + 2 * T::T_BYTES);
      dma4<3>(del_at, st_row, mine + 2 * T::T_BYTES + 256);
    }
#pragma unroll
    for (int j = 0; j < OPW; ++j) {
      const int x = j * NW + wave;
      if ((j + 1) * NW <= 2 * OT || x < 2 * OT) dma16<3>(x < OT ? ow1.at : ow2.at, ooff[j], own_at + x * 1024);
    }
    if (wave == NW - 1) {
      if constexpr (kDQ) {
        dma4<3>(lse_at, ow_row, own_at + 2 * T::O_BYTES);
        dma4<3>(del_at, ow_row, own_at + 2 * T::O_BYTES + 256);
      } else if constexpr (kRowB) {
        dma4<3>(row_at, ow_row, own_at + 2 * T::O_BYTES);
      }
    }
    st1.at += st1.step;
    st2.at += st2.step;
    ow1.at += ow1.step;
    ow2.at += ow2.step;
    lse_at += stat_step;
    del_at += stat_step;
    if constexpr (kRowB) row_at += row_step;
  };

  constexpr int PC = D / 4;  // 16-byte chunks per row of partial sums
  // where this entry's sums go; pieces of 64 lanes with 4 columns each, which the waves take in turn
  const int rows = min(32, S - o0);
  uint64_t out1 = uniform_ptr((kDQ ? p.dq : p.dk) + (int64_t)n0 * (kDQ ? p.dqs[0] : p.dks[0]) + (int64_t)head * (kDQ ? p.dqs[1] : p.dks[1]));
  uint64_t out2 = kDQ ? 0 : uniform_ptr(p.dv + (int64_t)n0 * p.dvs[0] + (int64_t)head * p.dvs[1]);
  const uint64_t step1 = (uint64_t)uniform_i64((kDQ ? p.dqs[0] : p.dks[0]) * 2), step2 = (uint64_t)uniform_i64(p.dvs[0] * 2);
  constexpr int RPP = 256 / D, PIECES = 32 / RPP, PPW = (PIECES + NW - 1) / NW;
  const int pieces = (rows + RPP - 1) / RPP, my_pieces = (pieces - wave + NW - 1) / NW;

  // The rows of the stripe's own places in both streamed operands, touched two entries ahead: the stripes of a head touch between them all rows
  // that they will all ask for, a cache line per lane.  The stripes ask for the same rows at the same time, so that little is on its way
  // from memory although every wave has an entry in flight: us, forward and gradients, 256 x 8 x 256 x 256, 274 -> 258; 512 entries 562 -> 502;
  // 150 x 8 x 333 x 333, head dim 64, 799 -> 723.
  // (A kernel of its own: the addresses alone were 2 to 4 % of a call of 30 us.)
  const int ahead_end = T::AHEAD && wave == 0 ? n1 : 0;
  uint64_t ahead_at = 0, ahead_step = 0;
  if constexpr (T::AHEAD) {
    const bool second = lane >= 32;
    const bf16_t* base = kDQ ? (second ? p.v : p.k) : (second ? p.dout : p.q);
    const int64_t b = kDQ ? (second ? p.vs[0] : p.ks[0]) : (second ? p.dos[0] : p.qs[0]);
    const int64_t hd = kDQ ? (second ? p.vs[1] : p.ks[1]) : (second ? p.dos[1] : p.qs[1]);
    const int64_t sq = kDQ ? (second ? p.vs[2] : p.ks[2]) : (second ? p.dos[2] : p.qs[2]);
    ahead_at = (uint64_t)(base + (int64_t)(n0 + 1) * b + (int64_t)head * hd + (int64_t)min(own, S - 1) * sq);
    ahead_step = (uint64_t)(b * 2);
  }
  // n: n0 + 1, n0 + 2, ... in this order.  (Only where entry n exists: the wait at the top of the walk's next entry, or of that after it, covers it.)
  auto touch_entry = [&](int n) FL_INLINE {
    if (T::AHEAD && n < ahead_end) {
      touch(ahead_at, lds0 + T::SLOTS * slot_bytes);
      ahead_at += ahead_step;
    }
  };
  if (n0 < n1) load_entry(0);
  touch_entry(n0 + 1);
  for (int n = n0; n < n1; ++n) {
    const int slot = T::SLOTS == 2 ? (n - n0) & 1 : 0;
    // everything this wave has asked for has landed, except the stores that were issued since
    if (T::SLOTS == 1 || n == n0 || my_pieces < PPW) dma_wait<0>();
    else dma_wait<(kDQ ? 1 : 2) * PPW>();
    __syncthreads();  // the owned rows are visible; everyone is done with the other slot
    if (T::SLOTS == 2 && n + 1 < n1) load_entry(slot ^ 1);
    touch_entry(n + 2);

    unsigned char* s0 = smem + slot * slot_bytes;
    unsigned char* mine = s0 + wave * T::W_BYTES;
    const unsigned char* own_at = s0 + w_bytes;
    ex8 o1[KS], o2[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      o1[ks] = Ops::rows(own_at, r, ks, h);
      o2[ks] = Ops::rows(own_at + T::O_BYTES, r, ks, h);
    }
    const float* own_f = reinterpret_cast<const float*>(own_at + 2 * T::O_BYTES);
    const float* st_f = reinterpret_cast<const float*>(mine + 2 * T::T_BYTES);
    const float own_a = kDQ ? own_f[r] : (kRowB ? own_f[r] * p.scale_log2 : 0.f);  // LSE of the query, or the bias row at the key
    f32x16 x2_init;
    if constexpr (kDQ) {
      const float nd = own_f[64 + r];
#pragma unroll
      for (int i = 0; i < 16; ++i) x2_init[i] = nd;
    }
    f32x16 acc1[DB], acc2[kDQ ? 1 : DB];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        acc1[d][i] = 0.f;
        if constexpr (!kDQ) acc2[d][i] = 0.f;
      }
    // The scores and dP of a block; with the row bias the queries' scores start from it.  st_a: the LSE of the streamed queries (ROLE_DKV)
    f32x16 x1[NB], x2[NB];
    float st_a[NB][16];
    ex8 t1[2][DB], t2[2][DB];  // transposed operands of a block's accumulating products
    auto per_row = [&](int b, int at) FL_INLINE -> f32x16 {
      f32x16 x;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(st_f + at + 32 * b + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * g + e] = a[e];
      }
      return x;
    };
    auto scores = [&](int b) FL_INLINE {
      ex8 a1[KS], a2[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        a1[ks] = Ops::rows(mine, 32 * b + r, ks, h);
        a2[ks] = Ops::rows(mine + T::T_BYTES, 32 * b + r, ks, h);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) x1[b][i] = 0.f;
      if constexpr (kDQ) {
        if constexpr (kRowB) x1[b] = per_row(b, 0);
        x2[b] = x2_init;
      } else {
        const f32x16 lse = per_row(b, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) st_a[b][i] = lse[i];
        x2[b] = per_row(b, 64);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        x1[b] = mfma32(a1[ks], o1[ks], x1[b]);
        x2[b] = mfma32(a2[ks], o2[ks], x2[b]);
      }
    };
    auto columns = [&](int b) FL_INLINE {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          t1[c][d] = Ops::columns(mine, 2 * b + c, d, lane, h);
          if constexpr (!kDQ) t2[c][d] = Ops::columns(mine + T::T_BYTES, 2 * b + c, d, lane, h);
        }
    };
    ex8 pf[2], dsf[2];
    auto weights = [&](int b) FL_INLINE {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        // logit in log2 units minus the row's LSE
        float c = bias[b][i];
        if constexpr (kDQ) {
          c -= own_a;
        } else {
          c -= st_a[b][i];
          if constexpr (kRowB) c += own_a;
        }
        const float w = fast_exp2(__builtin_fmaf(x1[b][i], p.scale_log2, c));
        const float ds = w * x2[b][i];
        if constexpr (kDQ) db[b][i] += ds;
        else pf[i / 8][i % 8] = (E)w;
        dsf[i / 8][i % 8] = (E)ds;
      }
    };
    auto accumulate = [&]() FL_INLINE {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          acc1[d] = mfma32(t1[c][d], dsf[c], acc1[d]);
          if constexpr (!kDQ) acc2[d] = mfma32(t2[c][d], pf[c], acc2[d]);
        }
    };
    // The order is kept by the fences: both blocks' scores ahead of the first weights where the registers allow (head dim 32), every LDS
    // read a phase ahead of its product.  Left to the compiler the products of a block stood behind its weights and each behind the
    // wait for its own reads, and the sums over the waves were a wait per wave.  us for a forward and its gradients: 2 x 64 entries of 300, 8 heads,
    // 290 -> 274; 100 of 490 with a mask and the gate 460 -> 437; 64 of 384 with the gate 184 -> 179; head dim 64, 64 of 256, 152 -> 146; 128 of 256
    // with both 140.0 -> 139.1.
    if constexpr (NB == 2 && D == 32) {
      scores(0);
      scores(1);
      columns(0);
      __builtin_amdgcn_sched_barrier(0);
      weights(0);
      __builtin_amdgcn_sched_barrier(0);
      accumulate();
      columns(1);
      __builtin_amdgcn_sched_barrier(0);
      weights(1);
      __builtin_amdgcn_sched_barrier(0);
      accumulate();
    } else {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        scores(b);
        columns(b);
        __builtin_amdgcn_sched_barrier(0);
        weights(b);
        __builtin_amdgcn_sched_barrier(0);
        accumulate();
      }
    }

    // ---- the waves add up: accumulator register i of block d is column 32 d + 8 (i / 4) + 4 h + i % 4 of owned row r
    auto park = [&](const f32x16 (&acc)[DB], unsigned char* at) FL_INLINE {
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f32x4*>(at + Ops::park_at(r, 8 * d + 2 * g + h)) = f32x4{acc[d][4 * g], acc[d][4 * g + 1], acc[d][4 * g + 2], acc[d][4 * g + 3]};
    };
    auto gather = [&](unsigned offset, uint64_t out, int64_t row_stride, float scale) FL_INLINE {
#pragma unroll
      for (int j = 0; j < PPW; ++j) {
        const int piece = j * NW + wave;
        if (piece >= pieces) break;
        // (rows past the end repeat the last one: every wave's stores are counted)
        const int row = min(piece * RPP + lane / PC, rows - 1), c = lane % PC;
        const unsigned char* at = s0 + offset + Ops::park_at(row, c);
        // (all of them in flight together: one after the other they were a wait per wave)
        f32x4 part[NW], sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) part[w] = *reinterpret_cast<const f32x4*>(at + w * T::W_BYTES);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += part[w];
        ex4 o4;
#pragma unroll
        for (int e = 0; e < 4; ++e) o4[e] = (E)(sum[e] * scale);
        // (32-bit offsets inside one (batch entry, head): S rows of at most 2^20 elements)
        sb_store8(out, (uint32_t)((o0 + row) * (int)row_stride + 4 * c) * 2u, __builtin_bit_cast(u32x2, o4));
      }
    };
    // (a wave parks over its own tiles only, which it alone has read)
    park(acc1, mine);
    if constexpr (!kDQ && T::ONE_PASS) park(acc2, mine + T::PARK);
    __syncthreads();
    gather(0, out1, kDQ ? p.dqs[2] : p.dks[2], p.scale);
    if constexpr (!kDQ && T::ONE_PASS) gather(T::PARK, out2, p.dvs[2], 1.0f);
    if constexpr (!kDQ && !T::ONE_PASS) {
      __syncthreads();
      park(acc2, mine);
      __syncthreads();
      gather(0, out2, p.dvs[2], 1.0f);
    }
    out1 += step1;
    out2 += step2;
    if (T::SLOTS == 1 && n + 1 < n1) {
      __syncthreads();  // the sums have been read
      load_entry(0);
    }
  }

  if constexpr (kDQ) {
    if (p.dbias_part != nullptr && own < S) {
      float* out = p.dbias_part + ((((int64_t)group * p.chunks + chunk) * p.H + head) * S + own) * p.s_pad;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int st = w0 + 32 * b + 8 * g + 4 * h;
          if (st < p.s_pad) *reinterpret_cast<f32x4*>(out + st) = f32x4{db[b][4 * g], db[b][4 * g + 1], db[b][4 * g + 2], db[b][4 * g + 3]};
        }
    }
  }
}

// Both roles in one launch, the longer one first: neither needs the other, and the start of a workgroup (the stripe's bias) and the end
// of a launch are latency that the other workgroup of the compute unit covers.
template <class TQ, class TKV>
__global__ __launch_bounds__(64 * TQ::NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
void pairbias_bwd_kernel(const SBParams p) {
  static_assert(TQ::NW == TKV::NW && TQ::LDS_BYTES == TKV::LDS_BYTES, "one workgroup shape");
  const int half = gridDim.x / 2;
  if ((int)blockIdx.x < half) pairbias_bwd_stripe<TKV>(p, blockIdx.x);
  else pairbias_bwd_stripe<TQ>(p, blockIdx.x - half);
}

// Sums the chunks' partial bias gradients (in chunk order) into [groups, H, S, S] of the bias's type.
template <class OUT>
__global__ __launch_bounds__(256) void pairbias_bwd_reduce_kernel(const float* part, OUT* out, int chunks, int64_t rows_per_group,
                                                                  int S, int s_pad, int64_t total4) {
  const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (x >= total4) return;
  const int q4 = s_pad / 4;
  const int64_t row = x / q4, grp = row / rows_per_group, in_grp = row % rows_per_group;  // row: [group][head][query]
  const int c = (int)(x % q4) * 4;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int ch = 0; ch < chunks; ++ch)
    s += *reinterpret_cast<const f32x4*>(part + ((grp * chunks + ch) * rows_per_group + in_grp) * s_pad + c);
  OUT* o = out + row * S + c;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (c + e < S) o[e] = (OUT)s[e];
}

struct SBPrepParams {
  const bf16_t *out, *dout, *gate;
  bf16_t *dgated, *dgate;  // dout * sigmoid(gate); gradient of the gate's logits
  float* delta;            // [B, H, S], minus the row sums
  const void* row;         // bias row per batch entry (or null), and where it goes times row_factor: [B, S]
  float* rowb;
  float row_factor;        // 1 / scale: the products' accumulators start from it
  int64_t row_batch;
  int32_t row_key, row_div, row_f32;
  int32_t ungated;         // `out` is the result before the gate
  int64_t os[3], dos[3], gs[3], dgds[3], dgs[3];
  int32_t B, H, S;
};

// What the two roles need per row, in one pass over dO and the result.  With the gate's weights sg and the result before
// the gate O: the output gradient of the attention dA = dO o sg, as rounded for the roles' products; Delta = rowsum(dA o O);
// and the gradient of the logits dO o O o sg (1 - sg).  A caller that kept only the gated result out = sg o O gets
// Delta = rowsum(dO o out) and dO o out (1 - sg): another rounding than dA's in Delta, and nothing of O where a nearly
// closed gate leaves a 16-bit out few bits (fp16, logits around -12: 1e-2 instead of 3e-4 in the logits' gradient).
template <int D, bool GATE, class E>
__global__ __launch_bounds__(256) void pairbias_bwd_prep_kernel(const SBPrepParams p) {
  typedef E ex8 __attribute__((ext_vector_type(8)));
  constexpr int LPR = D / 8;
  const int64_t rows = (int64_t)p.B * p.S * p.H, x = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  const int c = threadIdx.x % LPR * 8;
  // rows in (batch, position, head) order: the Evoformer's memory order
  const int64_t row = x < rows ? x : rows - 1;
  const int hd = (int)(row % p.H), s = (int)(row / p.H % p.S), b = (int)(row / ((int64_t)p.H * p.S));
  const ex8 d8 = *reinterpret_cast<const ex8*>(p.dout + b * p.dos[0] + hd * p.dos[1] + s * p.dos[2] + c);
  const ex8 o8 = *reinterpret_cast<const ex8*>(p.out + b * p.os[0] + hd * p.os[1] + s * p.os[2] + c);
  ex8 s8 = d8;  // what Delta sums against the result
  if constexpr (GATE) {
    const ex8 g8 = *reinterpret_cast<const ex8*>(p.gate + b * p.gs[0] + hd * p.gs[1] + s * p.gs[2] + c);
    ex8 a8, b8;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sg = fast_rcp(1.0f + fast_exp2(-1.4426950408889634f * (float)g8[e]));
      const float da = (float)d8[e] * sg;
      a8[e] = (E)da;
      b8[e] = (E)((p.ungated ? da : (float)d8[e]) * (float)o8[e] * (1.0f - sg));
    }
    if (p.ungated) s8 = a8;
    if (x < rows) {
      *reinterpret_cast<ex8*>(p.dgated + b * p.dgds[0] + hd * p.dgds[1] + s * p.dgds[2] + c) = a8;
      *reinterpret_cast<ex8*>(p.dgate + b * p.dgs[0] + hd * p.dgs[1] + s * p.dgs[2] + c) = b8;
    }
  }
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) sum += (float)s8[e] * (float)o8[e];
#pragma unroll
  for (int d = 1; d < LPR; d *= 2) sum += __shfl_xor(sum, d);
  if (x < rows && c == 0) {
    p.delta[((int64_t)b * p.H + hd) * p.S + s] = -sum;
    if (p.row != nullptr && hd == 0) {
      const int64_t off = (int64_t)(b / p.row_div) * p.row_batch + (int64_t)s * p.row_key;
      p.rowb[(int64_t)b * p.S + s] =
          p.row_factor * (p.row_f32 ? static_cast<const float*>(p.row)[off] : (float)static_cast<const E*>(p.row)[off]);
    }
  }
}

}  // namespace fl
