// Forward of attention with one dense bias shared by several consecutive batch entries (the Evoformer's row attention; reference
// attention_variants/evoformer.py:8-36): head dims 32 and 64, any lengths up to 512, optionally a bias row per batch entry, a
// sigmoid gate, row statistics and the result before the gate for the gradients.
//
// A workgroup stays with one stripe of 32 QB query rows of one head and walks over the batch entries that share the bias, as the
// gradients do (pairbias_bwd_kernel.h): the stripe's bias against all keys is read once, into fp32 registers, whatever its
// type and alignment, and is the addend of the multiply-add that scales a score.  The waves of the workgroup split the keys (NB
// blocks of 32 each), fetch their own rows of K and V into their own part of LDS, and add up their partial results through
// LDS once per batch entry:
//   S^T = K . Q^T (accumulators start from the bias row),  P = exp2(S^T scale log2(e) + bias),  O^T += V^T . P^T
// No row maximum: the weights are formed against 0, and the row sums, which every wave sees after they have been exchanged,
// tell whether that was safe; if not, the entry is done again with its maxima (as in the general kernel, fwd_kernel.h).
//
// What bounds the general kernel on such calls is the bias: a 2-byte load per score where its rows are not 16-byte addressable,
// a second tile beside every K/V tile where they are, and workgroups that live for a few tiles.  Here a score costs a
// multiply-add, an exponential, half a conversion and half a row sum, and what is left is the chain of an entry (queries, two
// products, exponentials, sums over the waves, stores: about 600 instructions per wave, 350 of them for its four blocks of
// 32 x 32) with two waves per SIMD to cover it.  Two blocks of queries per wave share the K and V operands, and halve what is
// exchanged per score against one (128 x 8 x 256 x 256, head dim 32, gate and row: 61 us with one; head dim 64 has no registers
// for two).  Head dim 32 is at the limit of the 256 registers that two waves per SIMD leave: with a bias row and up to three waves 12 to 72 bytes
// of a lane go to scratch, without one and up to four waves 12 to 36 (one and two waves that take neighbours: 68 and 100); the other shapes
// fit.  Wave counts are compiled in: sums over a run-time count wait for one LDS read after the other (55 us against 39).
// bf16, general kernel -> here: 128 x 8 x 256 x 256, head dim 32, gate, row and statistics: 48 -> 39 us; 2 x 207 x 4 x 494 x 494, head
// dim 32: 806 -> 201; 2 x 17 x 4 x 235 x 235, head dim 64, gate and row: 43 -> 17; 28 x 4 x 106 x 106, head dim 32, gate: 14 -> 6.
#pragma once
#include "tile_operands.h"

namespace fl {

struct StripeParams {
  const bf16_t *q, *k, *v;
  bf16_t* o;
  int64_t qs[3], ks[3], vs[3], os[3];  // element strides: batch, head, seq
  const void* bias;
  int64_t bs[3];                       // group, head, query (key stride 1)
  int32_t bias_f32;
  const void* row;                     // optional: one row of keys per row_div batch entries
  int64_t row_batch;
  int32_t row_key, row_div, row_f32;
  const bf16_t* gate;                  // optional
  int64_t gs[3];
  bf16_t* ungated;                     // optional: the result before the gate, addressed like o
  float* lse;                          // optional [B, H, Lq]
  int32_t B, H, Lq, Lk;
  int32_t div, groups, chunks, chunk_len;  // batch entries per bias; groups = B / div; entries are cut into chunks of chunk_len
  int32_t tiles;                       // stripes of 32 QB rows
  int32_t by_maximum;                  // weights are formed against the row's maximum from the start
  float scale, scale_log2;
};

// NEIGHBOURS: see StripePlace (compiled in: its arithmetic was 0.1 us of a call of 8)
template <int D_, int QB_, int NB_, int NW_, bool ROW_, class Elem_, bool NEIGHBOURS_ = false>
struct StripeTraits {
  using Elem = Elem_;
  static constexpr int D = D_, QB = QB_, NB = NB_, NW = NW_;
  static constexpr bool ROW = ROW_, NEIGHBOURS = NEIGHBOURS_;
  static constexpr int KS = D / 16, DB = D / 32;
  static constexpr int T_BYTES = NB * 32 * D * 2;  // K or V rows of one wave
  static constexpr int W_BYTES = 2 * T_BYTES;
  static constexpr int Q_BYTES = QB * 32 * D * 2;
  static constexpr int TPW = T_BYTES / 1024, QT = Q_BYTES / 1024;  // 1 KiB transfers
  // a wave's partial results go where its consumed tiles were
  static_assert(QB * 32 * D * 4 <= W_BYTES, "room for the partial results");
  static constexpr int RPP = 512 / D;              // result rows that a wave stores at once, 16 bytes per lane
  static constexpr int ROW_BYTES = ROW ? 2 * NB * 32 * 4 : 0;  // per wave: the bias row of this entry and of the next
  static constexpr int SUM_BYTES = QB * 32 * 4;    // per wave: row sums (and, on the rare path, maxima)
  static constexpr int SLOT_BYTES = NW * W_BYTES + Q_BYTES;  // one batch entry
  // tiles of batch entries resident in LDS
  static constexpr int SLOTS = 2 * SLOT_BYTES + NW * (ROW_BYTES + 2 * SUM_BYTES) <= 160 * 1024 ? 2 : 1;
  static constexpr int LDS_BYTES = SLOTS * SLOT_BYTES + NW * (ROW_BYTES + 2 * SUM_BYTES);
  // workgroups that a compute unit holds: two waves per SIMD, and what the LDS has room for
  static constexpr int PER_CU = 8 / NW < 160 * 1024 / LDS_BYTES ? 8 / NW : 160 * 1024 / LDS_BYTES;
};

// stores that the waits count.  As asm they bring the distances that the compiler keeps for its own: five wait states behind a vector
// instruction that wrote the scalar address (see dma16), and two behind a store of more than 8 bytes, which still reads its data
__device__ __forceinline__ void stripe_store16(uint64_t sbase, unsigned voff, u32x4 data) {
  asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2\n\ts_nop 1" ::"v"(voff), "v"(data), "s"(sbase) : "memory");
}
__device__ __forceinline__ void stripe_store4(uint64_t sbase, unsigned voff, float data) {
  asm volatile("s_nop 4\n\tglobal_store_dword %0, %1, %2" ::"v"(voff), "v"(data), "s"(sbase) : "memory");
}

template <class T>
__global__ __launch_bounds__(64 * T::NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
void stripe_kernel(const StripeParams p) {
  constexpr int D = T::D, QB = T::QB, NB = T::NB, NW = T::NW, KS = T::KS, DB = T::DB;
  constexpr bool kRow = T::ROW;
  constexpr float kLog2e = 1.4426950408889634f;
  using E = typename T::Elem;
  typedef E ex8 __attribute__((ext_vector_type(8)));
  typedef E ex2 __attribute__((ext_vector_type(2)));
  using L = TileLayout<D>;
  using Ops = TileOperands<D, E>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int r = lane % 32, h = lane / 32;

  const StripePlace place(p, blockIdx.x, T::NEIGHBOURS);
  if (place.none(p)) return;  // (before any barrier)
  const int tile = place.tile, head = place.unit % p.H, gc = place.unit / p.H, chunk = gc % p.chunks, group = gc / p.chunks;
  const int n0 = group * p.div + chunk * p.chunk_len, n1 = min(group * p.div + p.div, n0 + p.chunk_len);
  const int o0 = tile * QB * 32, Lk = p.Lk;
  const int rows = min(QB * 32, p.Lq - o0);  // of this stripe
  const int w0 = wave * NB * 32;             // first key of this wave

  // ---- addresses.  Per-lane offsets do not change from entry to entry; the scalar bases advance by one batch stride.
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem);
  constexpr unsigned w_bytes = T::W_BYTES * NW, slot_bytes = T::SLOT_BYTES;
  unsigned koff[T::TPW], voff[T::TPW];
#pragma unroll
  for (int it = 0; it < T::TPW; ++it) {
    koff[it] = Ops::transfer_offset(w0, Lk, it, p.ks[2], lane);
    voff[it] = Ops::transfer_offset(w0, Lk, it, p.vs[2], lane);
  }
  uint64_t ka = uniform_ptr(p.k + (int64_t)n0 * p.ks[0] + (int64_t)head * p.ks[1]);  // of the entry to be fetched next
  uint64_t va = uniform_ptr(p.v + (int64_t)n0 * p.vs[0] + (int64_t)head * p.vs[1]);
  uint64_t qa = uniform_ptr(p.q + (int64_t)n0 * p.qs[0] + (int64_t)head * p.qs[1]);
  const uint64_t kstep = (uint64_t)uniform_i64(p.ks[0] * 2), vstep = (uint64_t)uniform_i64(p.vs[0] * 2), qstep = (uint64_t)uniform_i64(p.qs[0] * 2);
  auto load_keys = [&](uint64_t ka, uint64_t va, int slot) FL_INLINE {
    const unsigned mine = lds0 + slot * slot_bytes + wave * T::W_BYTES;
#pragma unroll
    for (int it = 0; it < T::TPW; ++it) dma16<3>(ka, koff[it], mine + it * 1024);
#pragma unroll
    for (int it = 0; it < T::TPW; ++it) dma16<3>(va, voff[it], mine + T::T_BYTES + it * 1024);
  };
  constexpr int QPW = (T::QT + NW - 1) / NW;  // of the stripe's queries, shared out over the waves
  unsigned qoff[QPW];
#pragma unroll
  for (int j = 0; j < QPW; ++j) qoff[j] = Ops::transfer_offset(o0, p.Lq, j * NW + wave, p.qs[2], lane);
  auto load_entry = [&](int slot) FL_INLINE {
    const unsigned q_at = lds0 + slot * slot_bytes + w_bytes;
#pragma unroll
    for (int j = 0; j < QPW; ++j)
      if ((j + 1) * NW <= T::QT || j * NW + wave < T::QT) dma16<3>(qa, qoff[j], q_at + (j * NW + wave) * 1024);
    load_keys(ka, va, slot);
    qa += qstep;
    ka += kstep;
    va += vstep;
  };
  // the bias row of entry n at this lane's key, in units of the unscaled product
  const float row_factor = 1.0f / p.scale;
  auto row_value = [&](int n) FL_INLINE -> float {
    const int64_t at = (int64_t)(n / p.row_div) * p.row_batch + (int64_t)min(w0 + lane % (NB * 32), Lk - 1) * p.row_key;
    return p.row_f32 ? static_cast<const float*>(p.row)[at] : (float)static_cast<const E*>(p.row)[at];
  };
  float* const row_st = reinterpret_cast<float*>(smem + T::SLOTS * slot_bytes + wave * T::ROW_BYTES);
  float* const sums = reinterpret_cast<float*>(smem + T::SLOTS * slot_bytes + NW * T::ROW_BYTES);  // [wave][row]
  float* const maxima = sums + NW * QB * 32;

  if (n0 < n1) load_entry(0);
  if constexpr (kRow) {
    if (n0 < n1) {
      const float x = row_value(n0) * row_factor;
      if (lane < NB * 32) row_st[lane] = x;
    }
  }

  // ---- the stripe's bias in log2 units, -inf past the last key: register (qb, b, i) is key w0 + 32 b + 8 (i / 4) + 4 h + i % 4
  // against query o0 + 32 qb + r
  float bias[QB][NB][16];
  {
    const int64_t base = (int64_t)group * p.bs[0] + (int64_t)head * p.bs[1];
    // four consecutive keys in one load at any alignment (the loads before anything looks at them: all in flight together); a
    // group that the row's end cuts is read four back from the end
    auto fetch = [&](auto* src) FL_INLINE {
      using X = std::remove_const_t<std::remove_pointer_t<decltype(src)>>;
      struct __attribute__((packed, aligned(sizeof(X)))) X4 {
        X x[4];
      };
      X4 x[QB][NB][4];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const X* at = src + base + (int64_t)min(o0 + 32 * qb + r, p.Lq - 1) * p.bs[2];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            x[qb][b][g] = *reinterpret_cast<const X4*>(at + min(w0 + 32 * b + 8 * g + 4 * h, Lk - 4));
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int st = w0 + 32 * b + 8 * g + 4 * h, back = max(0, st - (Lk - 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const X(&v)[4] = x[qb][b][g].x;
              X y = v[e];
#pragma unroll
              for (int d = 1; d < 4; ++d)
                if (e + d < 4) y = back == d ? v[e + d < 4 ? e + d : 3] : y;
              bias[qb][b][4 * g + e] = st + e < Lk ? (float)y * kLog2e : -INFINITY;
            }
          }
    };
    if (p.bias_f32) fetch(static_cast<const float*>(p.bias));
    else fetch(static_cast<const E*>(p.bias));
  }

  uint64_t oa = uniform_ptr(p.o + (int64_t)n0 * p.os[0] + (int64_t)head * p.os[1]);
  uint64_t ua = uniform_ptr(p.ungated + (int64_t)n0 * p.os[0] + (int64_t)head * p.os[1]);
  uint64_t la = uniform_ptr(p.lse + ((int64_t)n0 * p.H + head) * p.Lq);
  const uint64_t ostep = (uint64_t)uniform_i64(p.os[0] * 2), lstep = (uint64_t)p.H * p.Lq * 4u;
  const int pieces = (rows + T::RPP - 1) / T::RPP;  // of RPP rows: the waves store them in turn
  const int my_pieces = (pieces - wave + NW - 1) / NW;
  const int prow = lane / L::CPR, pcol = lane % L::CPR;  // this lane's row of a piece, and its 8 columns

  for (int n = n0; n < n1; ++n) {
    const int cur = (n - n0) & 1, slot = T::SLOTS == 2 ? cur : 0;
    // everything this wave has asked for has landed, except the stores that were issued since
    constexpr int kMost = (QB * D / 16 + NW - 1) / NW;  // pieces that this wave may have stored
    if (T::SLOTS == 1 || n == n0 || my_pieces < kMost) dma_wait<0>();
    else if (p.ungated) dma_wait<2 * kMost>();
    else dma_wait<kMost>();
    __syncthreads();  // the queries are visible; everyone is done with the other slot
    if (T::SLOTS == 2 && n + 1 < n1) load_entry(slot ^ 1);
    float row_next = 0.f;
    if constexpr (kRow) {
      if (n + 1 < n1) row_next = row_value(n + 1);
    }
    ex8 gate_first;  // the logits of this wave's first piece (in most shapes its only one)
    auto gate_at = [&](int piece) FL_INLINE -> ex8 {
      const int row = min(piece * T::RPP + prow, rows - 1);
      return *reinterpret_cast<const ex8*>(p.gate + (int64_t)n * p.gs[0] + (int64_t)head * p.gs[1] + (int64_t)(o0 + row) * p.gs[2] + 8 * pcol);
    };
    if (p.gate && wave < pieces) gate_first = gate_at(wave);

    unsigned char* const s0 = smem + slot * slot_bytes;
    unsigned char* const mine = s0 + wave * T::W_BYTES;
    ex8 qf[QB][KS];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[qb][ks] = Ops::rows(s0 + w_bytes, 32 * qb + r, ks, h);

    f32x16 acc[QB][DB];
    float l[QB];
    auto scores = [&](int b, f32x16 (&x)[QB]) FL_INLINE {
      f32x16 init;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
        if constexpr (kRow) a = *reinterpret_cast<const f32x4*>(row_st + cur * NB * 32 + 32 * b + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) init[4 * g + e] = a[e];
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) x[qb] = init;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const ex8 kf = Ops::rows(mine, 32 * b + r, ks, h);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) x[qb] = mfma32(kf, qf[qb][ks], x[qb]);
      }
    };
    auto clear = [&]() FL_INLINE {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        l[qb] = 0.f;
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[qb][d][i] = 0.f;
      }
    };
    // the row sums (of the rounded weights, the numbers the second product uses) and the second product of block b
    auto accumulate = [&](int b, const ex8 (&pf)[QB][2]) FL_INLINE {
      const ex2 ones = {(E)1.0f, (E)1.0f};
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int i = 0; i < 16; i += 2) l[qb] = dot2acc(ex2{pf[qb][i / 8][i % 8], pf[qb][i / 8][i % 8 + 1]}, ones, l[qb]);
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int d = 0; d < DB; ++d) {
          const ex8 vf = Ops::columns(mine + T::T_BYTES, 2 * b + c, d, lane, h);
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) acc[qb][d] = mfma32(vf, pf[qb][c], acc[qb][d]);
        }
    };
    float ref[QB];  // what the weights are formed against, log2 units
    auto attend_to_zero = [&]() FL_INLINE {
      clear();
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) ref[qb] = 0.f;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        f32x16 x[QB];
        scores(b, x);
        ex8 pf[QB][2];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int i = 0; i < 16; ++i) pf[qb][i / 8][i % 8] = (E)fast_exp2(__builtin_fmaf(x[qb][i], p.scale_log2, bias[qb][b][i]));
        accumulate(b, pf);
      }
    };
    auto attend_to_maximum = [&]() FL_INLINE {
      f32x16 x[NB][QB];
      float m[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) m[qb] = -INFINITY;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        scores(b, x[b]);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            x[b][qb][i] = __builtin_fmaf(x[b][qb][i], p.scale_log2, bias[qb][b][i]);
            m[qb] = __builtin_fmaxf(m[qb], x[b][qb][i]);
          }
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        m[qb] = xhalf_max(m[qb]);
        if (h == 0) maxima[(wave * QB + qb) * 32 + r] = m[qb];
      }
      __syncthreads();
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        // (not below -2^15: scores further down are masks written as finite numbers, whose weights are 0; see fwd_kernel.h)
        ref[qb] = -32768.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) ref[qb] = __builtin_fmaxf(ref[qb], maxima[(w * QB + qb) * 32 + r]);
      }
      clear();
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        ex8 pf[QB][2];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int i = 0; i < 16; ++i) pf[qb][i / 8][i % 8] = (E)fast_exp2(x[b][qb][i] - ref[qb]);
        accumulate(b, pf);
      }
    };
    // leaves this wave's partial results and row sums where the others find them (over its own tiles, which it alone has read)
    auto park = [&]() FL_INLINE {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(mine + Ops::park_at(32 * qb + r, 8 * d + 2 * g + h)) =
                f32x4{acc[qb][d][4 * g], acc[qb][d][4 * g + 1], acc[qb][d][4 * g + 2], acc[qb][d][4 * g + 3]};
        l[qb] = xhalf_sum(l[qb]);
        if (h == 0) sums[(wave * QB + qb) * 32 + r] = l[qb];
      }
    };
    // A weight has overflowed, or a row's weights may have lost their bits to underflow (a bf16 weight keeps them down to 2^-126, an
    // fp16 weight is subnormal below 2^-14): the entry is done again against its maxima.  Every wave reads the same sums and takes
    // the same branch.
    constexpr float kBig = 0x1p24f, kTiny = std::is_same<E, f16_t>::value ? 0x1p-4f : 0x1p-24f;
    float total[QB];
    for (bool by_maximum = p.by_maximum;; by_maximum = true) {
      if (by_maximum) attend_to_maximum();
      else attend_to_zero();
      park();
      __syncthreads();
      bool bad = false;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) t += sums[(w * QB + qb) * 32 + r];
        total[qb] = t;
        bad = bad | !(t <= kBig) | (t < kTiny);
      }
      if (by_maximum || __builtin_amdgcn_ballot_w64(bad) == 0) break;
      // (the next entry's rows have been asked for where there is room for them)
      const int ahead = T::SLOTS == 2 && n + 1 < n1 ? 2 : 1;
      load_keys((uint64_t)uniform_i64((int64_t)(ka - ahead * kstep)), (uint64_t)uniform_i64((int64_t)(va - ahead * vstep)), slot);  // (the partial results lie over this wave's tiles, and nobody has read them)
      dma_wait<0>();
    }

    if constexpr (kRow) {  // (ahead of the stores: the wait for the value would wait for them)
      if (lane < NB * 32) row_st[(cur ^ 1) * NB * 32 + lane] = row_next * row_factor;
    }

    // ---- the waves' partial results added up, normalised, gated and stored, 8 columns per lane
    auto store_piece = [&](int piece, ex8 g8) FL_INLINE {
      const int row = min(piece * T::RPP + prow, rows - 1);  // (rows past the end repeat the last one: every wave's stores are counted)
      const int qb = piece * T::RPP / 32;
      float t = total[0], rf = ref[0];
      if (QB > 1 && qb > 0) {
        t = total[QB - 1];
        rf = ref[QB - 1];
      }
      t = __shfl(t, row % 32);
      f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
      const unsigned char* at0 = s0 + Ops::park_at(row, 2 * pcol);
      const unsigned char* at1 = s0 + Ops::park_at(row, 2 * pcol + 1);
      auto add = [&](int w) FL_INLINE {
        a += *reinterpret_cast<const f32x4*>(at0 + w * T::W_BYTES);
        b += *reinterpret_cast<const f32x4*>(at1 + w * T::W_BYTES);
      };
#pragma unroll
      for (int w = 0; w < NW; ++w) add(w);
      const float inv = t > 0.f ? 1.0f / t : 0.f;  // a row that attends nothing yields zeros
      const unsigned off = (uint32_t)((o0 + row) * (int)p.os[2] + 8 * pcol) * 2u;
      ex8 out;
      if (p.ungated) {
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = (E)((e < 4 ? a[e % 4] : b[e % 4]) * inv);
        stripe_store16(ua, off, __builtin_bit_cast(u32x4, out));
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float x = (e < 4 ? a[e % 4] : b[e % 4]) * inv;
        if (p.gate) x *= fast_rcp(1.0f + fast_exp2(-kLog2e * (float)g8[e]));
        out[e] = (E)x;
      }
      stripe_store16(oa, off, __builtin_bit_cast(u32x4, out));
      if (p.lse) {
        rf = __shfl(rf, row % 32);
        stripe_store4(la, (uint32_t)(o0 + row) * 4u, t > 0.f ? rf + __builtin_amdgcn_logf(t) : INFINITY);
      }
    };
    if (wave < pieces) store_piece(wave, gate_first);
    for (int piece = wave + NW; piece < pieces; piece += NW) {
      ex8 g8;
      if (p.gate) g8 = gate_at(piece);
      store_piece(piece, g8);
    }
    oa += ostep;
    ua += ostep;
    la += lstep;
    if (T::SLOTS == 1 && n + 1 < n1) {
      __syncthreads();  // the partial results have been read
      load_entry(0);
    }
  }
}

}  // namespace fl
