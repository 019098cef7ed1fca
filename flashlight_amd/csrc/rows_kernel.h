// Attention forward for few query rows per key / value head: decoding steps and short prefills.
//
// What bounds such calls is the reading of K and V (a decoding step reads every key once for a handful of rows) and how
// soon it starts: the tile kernel (fwd_kernel.h) spends a 128-row workgroup, an LDS ring and two barriers per key tile on
// 1 .. 16 live rows.  Here a wave owns 16 rows and streams key tiles of its own, straight from memory into the registers
// of the matrix instructions: no LDS, no barrier and no other wave's pace until the end.  The waves of a workgroup take
// every NW-th tile of the workgroup's share of the keys, the shares (`chunks`) of one row tile go to different
// workgroups, and the partial results (fp32, with their maxima and sums) are added up through LDS inside a workgroup and
// by rows_merge_kernel across workgroups.  Every wave keeps the next tile (32 keys: 16 KiB at head dim 128) in flight
// while it works on the current one: eight waves on a compute unit have 128 KiB outstanding.
// Measured (MI355X, bf16, operands larger than the memory-side cache; before: the tile kernel over key chunks made by the
// front end): 32 query heads over 8, one row, 32768 keys, head dim 128: 42.2 -> 31.2 us (27.4 for this kernel = 4.9 TB/s,
// launch included, 4.5 for the merge, now 4); 8 sequences of 3001 keys in longer buffers: 51.6 -> 21.9 us; 32 x 2048 keys 5.5 TB/s;
// causal prefill 2 x 8 heads x 512, head dim 64: 10.9 -> 9.2 us.
// What such a call spends beside its reads is a chain: with the sums over the waves unrolled (a run-time count was one LDS wait after the
// other), no division where one head has all rows, and the merge's loads in flight together, 9.20 -> 8.86, decoding 31.2 -> 30.1, 22.1 ->
// 21.7 and, 2 x 8 heads of 282 rows, 7.8 -> 7.5.  With nothing ahead of the first load that goes through LDS (the tile's bounds) and no
// division at all (Div), 8.87 -> 8.19, decoding 30.0 -> 29.3 and 21.6 -> 20.6; with the parameters' lines asked for together
// (fetch_params) 7.97, 28.5 and 20.1.
//
// Rows are packed: row x of key / value head n is position x % Lq of query head n * G + x / Lq, so the G query heads that
// share a key / value head are rows of one tile and the keys are read once for all of them.
//
// Operand layouts (v_mfma_f32_16x16x32: A and B hold 8 consecutive k per lane, lane = (index % 16, k group g = lane / 16)):
//   S^T[key, q] = K . Q^T      A = K rows as they lie in memory, two 16-key blocks; lane (q, g) ends up with the scores of
//                              keys 16 t + 4 g + i (t = 0, 1; i = 0 .. 3) of row q: eight keys, which are the eight k
//                              slots of that lane's B operand in the second product, packed to 16 bits in place
//   O^T[dv, q] += V^T . P^T    A = V^T: lane (n, g) loads W = DV / 16 consecutive columns of its eight keys and takes
//                              column W n + j of them in product j, a transposition inside the lane (byte permutes);
//                              16 lanes cover whole rows of V, so the loads are contiguous
#pragma once
#include "fwd_kernel.h"

namespace fl {

struct RParams {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  bf16_t* o;
  float* lse;                                // optional, as in KParams
  int64_t qs[3], ks[3], vs[3], os[3];        // element strides: batch, head, seq
  int32_t B, Hq, Hkv, Lq, Lk, group;
  int32_t rows;                              // group * Lq: packed rows per key / value head
  int32_t row_tiles, chunks, units, waves;   // units = B * Hkv; waves per workgroup
  Div by_rows, by_row_tiles, by_chunks, by_Hkv, by_Lq;
  int32_t by_xcd;                            // row tiles of one (unit, chunk) on one XCD (units * chunks >= 8)
  float scale_log2, cap_k1, cap_c;           // as in fwd_kernel; cap_c = 0: no soft-cap
  int32_t dmin, dmax, pfx;                   // attend iff key < Lk && ((dmin <= key - q <= dmax) || key < pfx)
  int32_t alibi_heads;
  // row biases (one value per key and batch entry: padding masks), log2 units are applied here
  const void* bias[2];
  int64_t bias_batch[2];
  int32_t bias_key[2], bias_div[2], bias_f32[2];
  // chunks > 1: unnormalised partial results [unit][row tile][chunk][rows per tile][D] and their (maximum, sum) pairs
  float* part;
  float* part_ml;
};

typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// max / sum over the four lanes that share lane % 16
__device__ __forceinline__ float groups_max(float x) {
  x = __builtin_fmaxf(x, __shfl_xor(x, 16, 64));
  return __builtin_fmaxf(x, __shfl_xor(x, 32, 64));
}
__device__ __forceinline__ float groups_sum(float x) {
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}
// MOD: 0 plain, F_ALIBI | F_SOFTCAP (either may be off at run time), F_BIAS (row biases, and the soft-cap at run time)
// QT: 16-row blocks per wave (1 or 2)
template <int D_, int QT_, uint32_t MOD_, class Elem_>
struct RowsTraits {
  using Elem = Elem_;
  static constexpr int D = D_, QT = QT_, RB = 16 * QT_;
  // both K and V of the next tile in flight during the current one, where the registers allow; otherwise K alone, and V
  // arrives under its own tile's first product
  static constexpr bool V_AHEAD = D_ * QT_ <= 128 && !(D_ == 128 && (MOD_ & F_BIAS));
  static constexpr uint32_t MOD = MOD_;
  static constexpr int KS = D / 32;   // k-steps of the first product
  static constexpr int W = D / 16;    // value columns per lane
  static constexpr int ROW_F = D + 4; // floats per row of the LDS exchange (the pad spreads rows over the banks)
};

template <class T>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
void rows_kernel(const RParams p) {
  constexpr int D = T::D, KS = T::KS, W = T::W, QT = T::QT, RB = T::RB;
  constexpr bool kAlibiCap = T::MOD & F_ALIBI, kBias = T::MOD & F_BIAS;
  constexpr float kLog2e = 1.4426950408889634f;
  using E = typename T::Elem;
  typedef E ex8 __attribute__((ext_vector_type(8)));
  typedef E ex2 __attribute__((ext_vector_type(2)));
  typedef uint32_t vreg __attribute__((ext_vector_type(W / 2)));  // W elements of 16 bits

  fetch_params<RParams>();
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int NW = p.waves;
  const int n16 = lane % 16, g = lane / 16;

  // ---- workgroup -> (unit, chunk, row tile); the row tiles of one (unit, chunk) read the same keys
  int rt, uc;
  if (p.by_xcd) {
    const int x = blockIdx.x % 8, i = blockIdx.x / 8, o = p.by_row_tiles.of(i);
    rt = i - o * p.row_tiles;
    uc = o * 8 + x;
    if (uc >= p.units * p.chunks) return;
  } else {
    uc = p.by_row_tiles.of(blockIdx.x);
    rt = blockIdx.x - uc * p.row_tiles;
  }
  rt = p.row_tiles - 1 - rt;  // under a causal mask the last rows have the most keys: dealt first
  const int unit = p.by_chunks.of(uc), chunk = uc - unit * p.chunks;
  const int batch = p.by_Hkv.of(unit), kvh = unit - batch * p.Hkv;

  // ---- this lane's rows (rows past the end repeat the last one and are not stored) and the interval of keys each attends
  int qpos[QT], head[QT], khi[QT], klo[QT];
  auto first_key = [&](int q) FL_INLINE { return max(0, q + p.dmin); };
  auto last_key = [&](int q) FL_INLINE { return min(p.Lk - 1, max(p.dmax + q, p.pfx - 1)); };
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const int crow = min(rt * RB + u * 16 + n16, p.rows - 1), gh = p.by_Lq.of(crow);
    qpos[u] = crow - gh * p.Lq;
    head[u] = gh;
    khi[u] = last_key(qpos[u]);
    klo[u] = first_key(qpos[u]);
  }
  // Keys that some row and that every row of the tile attends: both bounds grow with the position, so the smallest and the largest one
  // say it, which are the first and the last row's, or 0 and Lq - 1 where the rows run on into another head.  (Taken over the wave
  // by exchanges through LDS this was 24 of them ahead of the first load.)
  const bool one_head = __builtin_amdgcn_readlane(head[0], 0) == __builtin_amdgcn_readlane(head[QT - 1], 15);
  const int q_min = one_head ? __builtin_amdgcn_readlane(qpos[0], 0) : 0;
  const int q_max = one_head ? __builtin_amdgcn_readlane(qpos[QT - 1], 15) : p.Lq - 1;
  const int any_lo = first_key(q_min), any_hi = last_key(q_max), all_lo = first_key(q_max), all_hi = last_key(q_min);
#pragma unroll
  for (int u = 0; u < QT; ++u) head[u] += kvh * p.group;
  int t_end, t;
  {
    const int t0 = any_lo / 32, n = any_hi >= any_lo ? any_hi / 32 + 1 - t0 : 0;
    // chunk c takes n / chunks tiles, the first n % chunks of them one more
    int first = 0, share = n;
    if (p.chunks > 1) {
      share = p.by_chunks.of(n);
      const int more = n - share * p.chunks;
      first = share * chunk + min(chunk, more);
      share += chunk < more ? 1 : 0;
    }
    t = t0 + first + wave;
    t_end = t0 + first + share;
  }

  ex8 qf[QT][KS];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const bf16_t* qp = p.q + (int64_t)batch * p.qs[0] + (int64_t)head[u] * p.qs[1] + (int64_t)qpos[u] * p.qs[2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[u][ks] = *reinterpret_cast<const ex8*>(qp + ks * 32 + g * 8);
  }
  const uint64_t kbase = uniform_ptr(p.k + (int64_t)batch * p.ks[0] + (int64_t)kvh * p.ks[1]);
  const uint64_t vbase = uniform_ptr(p.v + (int64_t)batch * p.vs[0] + (int64_t)kvh * p.vs[1]);
  const uint32_t k_row = (uint32_t)p.ks[2] * 2u, v_row = (uint32_t)p.vs[2] * 2u;  // bytes; below 2^24 (host)

  float slope_l2[QT];
  if constexpr (kAlibiCap) {
#pragma unroll
    for (int u = 0; u < QT; ++u)
      slope_l2[u] = p.alibi_heads > 0 ? exp2f(-8.0f * (float)(head[u] + 1) / (float)p.alibi_heads) * kLog2e : 0.f;
  }

  f32x4 oacc[QT][W];
  float m_run[QT], l_run[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
#pragma unroll
    for (int j = 0; j < W; ++j) oacc[u][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[u] = -INFINITY;
    l_run[u] = 0.f;
  }

  struct KTile {
    ex8 x[2][KS];
  };
  struct VTile {
    vreg x[8];
  };
  // keys past the end repeat the last one (they are masked); row offsets are relative to the tile's first key
  auto load_k = [&](KTile& b, int tt) FL_INLINE {
    const int last = p.Lk - 1 - tt * 32;
    const unsigned char* kb = reinterpret_cast<const unsigned char*>(kbase + (uint64_t)tt * ((uint64_t)k_row * 32));
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t off = __umul24((uint32_t)min(s * 16 + n16, last), k_row) + (uint32_t)(g * 16);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) b.x[s][ks] = *reinterpret_cast<const ex8*>(kb + off + ks * 64);
    }
  };
  auto load_v = [&](VTile& b, int tt) FL_INLINE {
    const int last = p.Lk - 1 - tt * 32;
    const unsigned char* vb = reinterpret_cast<const unsigned char*>(vbase + (uint64_t)tt * ((uint64_t)v_row * 32));
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t off = __umul24((uint32_t)min((e / 4) * 16 + g * 4 + e % 4, last), v_row) + (uint32_t)(n16 * W * 2);
      b.x[e] = *reinterpret_cast<const vreg*>(vb + off);
    }
  };
  // the weights of one tile, packed as the second product's B operand, and the running maximum and sum
  auto weights = [&](const KTile& b, ex8 (&pf)[QT], int tt) FL_INLINE {
    const int k0 = tt * 32 + g * 4;  // key of score (s, i): k0 + 16 s + i
    const bool masked = tt * 32 + 31 > all_hi || tt * 32 < all_lo;  // (wave-uniform)
    float bv[8];
    if constexpr (kBias) {
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const int key = min(k0 + 16 * (x / 4) + x % 4, p.Lk - 1);
        bv[x] = 0.f;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          if (p.bias[nb] == nullptr) continue;
          const int64_t off = (int64_t)(batch / p.bias_div[nb]) * p.bias_batch[nb] + (int64_t)key * p.bias_key[nb];
          bv[x] += p.bias_f32[nb] ? static_cast<const float*>(p.bias[nb])[off] : (float)static_cast<const E*>(p.bias[nb])[off];
        }
      }
    }
    f32x4 sc[QT][2];
#pragma unroll
    for (int u = 0; u < QT; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        sc[u][s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) sc[u][s] = mfma16(b.x[s][ks], qf[u][ks], sc[u][s]);
      }
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      f32x4(&s)[2] = sc[u];
      const float alibi0 = kAlibiCap ? slope_l2[u] * (float)(k0 - qpos[u]) : 0.f;
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        float y = s[x / 4][x % 4];
        if ((kAlibiCap || kBias) && p.cap_c > 0.f) {
          const float rc = fast_rcp(fast_exp2(y * p.cap_k1) + 1.0f);
          y = __builtin_fmaf(rc, -2.0f * p.cap_c, p.cap_c);
        } else {
          y *= p.scale_log2;
        }
        if constexpr (kAlibiCap) y += __builtin_fmaf(slope_l2[u], (float)(16 * (x / 4) + x % 4), alibi0);
        if constexpr (kBias) y = __builtin_fmaf(bv[x], kLog2e, y);
        s[x / 4][x % 4] = y;
      }
      if (masked) {
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          const int key = k0 + 16 * (x / 4) + x % 4;
          s[x / 4][x % 4] = (key <= khi[u] && key >= klo[u]) ? s[x / 4][x % 4] : -INFINITY;
        }
      }
      float mx = s[0][0];
#pragma unroll
      for (int x = 1; x < 8; ++x) mx = __builtin_fmaxf(mx, s[x / 4][x % 4]);
      mx = groups_max(mx);
      // the accumulators are rescaled only when some row's maximum grew by more than 8 (log2 units): weights stay below
      // 2^8 and any reference gives the same quotient.  Finite stand-ins for -inf in additive masks (-1e9, the type's most
      // negative number) never become the reference: below -2^15 everything is a zero against any real score.
      if (__builtin_amdgcn_ballot_w64(mx > m_run[u] + 8.0f) != 0) {  // (m_run = -inf before the first key)
        const float m_new = __builtin_fmaxf(__builtin_fmaxf(m_run[u], mx), kBias ? -32768.0f : -INFINITY);
        const float alpha = m_new == -INFINITY ? 1.0f : fast_exp2(m_run[u] - m_new);
        m_run[u] = m_new;
        l_run[u] *= alpha;
#pragma unroll
        for (int j = 0; j < W; ++j) oacc[u][j] *= alpha;
      }
      const float ref = m_run[u] == -INFINITY ? 0.f : m_run[u];
#pragma unroll
      for (int x = 0; x < 8; ++x) pf[u][x] = (E)fast_exp2(s[x / 4][x % 4] - ref);
      // the sum takes the rounded weights, the very numbers the second product uses
      const ex2 ones = {(E)1.0f, (E)1.0f};
#pragma unroll
      for (int x = 0; x < 8; x += 2) l_run[u] = dot2acc(ex2{pf[u][x], pf[u][x + 1]}, ones, l_run[u]);
    }
  };
  auto second_product = [&](const VTile& b, const ex8 (&pf)[QT]) FL_INLINE {
#pragma unroll
    for (int j = 0; j < W; ++j) {
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e)  // elements j of keys 2 e and 2 e + 1
        w[e] = __builtin_amdgcn_perm(b.x[2 * e + 1][j / 2], b.x[2 * e][j / 2], j % 2 ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int u = 0; u < QT; ++u) oacc[u][j] = mfma16(__builtin_bit_cast(ex8, w), pf[u], oacc[u][j]);
    }
  };

  // two register buffers; every path is a straight line of "loads of the next tile, work on this one", so that the waits
  // before the work count the loads behind it exactly
  if (t < t_end) {
    KTile ka, kb;
    VTile va, vb;
    auto step = [&](KTile& k, VTile& v, KTile& k_next, VTile& v_next, int tt, auto more) FL_INLINE {
      if constexpr (!T::V_AHEAD) load_v(v, tt);
      if constexpr (decltype(more)::value) {
        load_k(k_next, tt + NW);
        if constexpr (T::V_AHEAD) load_v(v_next, tt + NW);
      }
      ex8 pf[QT];
      weights(k, pf, tt);
      second_product(v, pf);
    };
    load_k(ka, t);
    if constexpr (T::V_AHEAD) load_v(va, t);
    VTile& v2 = pick<T::V_AHEAD>(vb, va);
    for (;;) {
      if (t + NW >= t_end) {
        step(ka, va, kb, v2, t, std::false_type{});
        break;
      }
      step(ka, va, kb, v2, t, std::true_type{});
      t += NW;
      if (t + NW >= t_end) {
        step(kb, v2, ka, va, t, std::false_type{});
        break;
      }
      step(kb, v2, ka, va, t, std::true_type{});
      t += NW;
    }
  }

  // ---- the waves of the workgroup add up: O^T register i of product j is column W (4 g + i) + j of row n16
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* xo = reinterpret_cast<float*>(smem);                      // [NW][RB][ROW_F]
  float* xml = xo + (size_t)NW * RB * T::ROW_F;                    // [NW][RB][2]
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const int r = wave * RB + u * 16 + n16;
    const float l = groups_sum(l_run[u]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < W; j += 4) {
        const f32x4 w = {oacc[u][j][i], oacc[u][j + 1][i], oacc[u][j + 2][i], oacc[u][j + 3][i]};
        *reinterpret_cast<f32x4*>(xo + r * T::ROW_F + W * (4 * g + i) + j) = w;
      }
    if (g == 0) {
      xml[r * 2] = m_run[u];
      xml[r * 2 + 1] = l;
    }
  }
  __syncthreads();
  const int n_valid = min(RB, p.rows - rt * RB);
  // (the wave count as a constant: all reads of the exchange in flight together instead of one wait after the other)
  auto add_up = [&](auto nw_tag) FL_INLINE {
    constexpr int N = decltype(nw_tag)::value;
    for (int x = threadIdx.x; x < n_valid * (D / 4); x += N * 64) {
      const int r = x / (D / 4), c = x % (D / 4) * 4;
      f32x2 ml[N];
      f32x4 ow[N];
#pragma unroll
      for (int w = 0; w < N; ++w) {
        ml[w] = *reinterpret_cast<const f32x2*>(xml + (w * RB + r) * 2);
        ow[w] = *reinterpret_cast<const f32x4*>(xo + (w * RB + r) * T::ROW_F + c);
      }
      float M = -INFINITY;
#pragma unroll
      for (int w = 0; w < N; ++w) M = __builtin_fmaxf(M, ml[w][0]);
      const float ref = M == -INFINITY ? 0.f : M;
      float L = 0.f;
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < N; ++w) {
        const float a = fast_exp2(ml[w][0] - ref);
        L += a * ml[w][1];
        o += a * ow[w];
      }
      if (p.chunks == 1) {
        const int pr = rt * RB + r, hd = p.by_Lq.of(pr), pos = pr - hd * p.Lq, oh = kvh * p.group + hd;
        const float inv = L > 0.f ? 1.0f / L : 0.f;  // a row that attends nothing yields zeros
        typedef E ex4 __attribute__((ext_vector_type(4)));
        ex4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = (E)(o[e] * inv);
        *reinterpret_cast<ex4*>(p.o + (int64_t)batch * p.os[0] + (int64_t)oh * p.os[1] + (int64_t)pos * p.os[2] + c) = w;
        if (p.lse != nullptr && c == 0)
          p.lse[((int64_t)batch * p.Hq + oh) * p.Lq + pos] = L > 0.f ? ref + __builtin_log2f(L) : INFINITY;
      } else {
        const int64_t slot = (((int64_t)unit * p.row_tiles + rt) * p.chunks + chunk) * RB + r;
        *reinterpret_cast<f32x4*>(p.part + slot * D + c) = o;
        if (c == 0) *reinterpret_cast<f32x2*>(p.part_ml + slot * 2) = f32x2{M, L};
      }
    }
  };
  if (NW == 8) add_up(std::integral_constant<int, 8>{});
  else if (NW == 4) add_up(std::integral_constant<int, 4>{});
  else add_up(std::integral_constant<int, 2>{});
}

// Adds up the chunks of a row: one workgroup of 256 threads per (unit, row); D / 4 threads take four columns each, and
// the 1024 / D groups of them take every (1024 / D)-th chunk, so that a row's loads are in flight together.
template <int D, int RB, class E>
__global__ __launch_bounds__(256) void rows_merge_kernel(const RParams p) {
  fetch_params<RParams>();
  constexpr int TPR = D / 4, NG = 256 / TPR;
  const int unit = p.by_rows.of(blockIdx.x), row = blockIdx.x - unit * p.rows;
  const int c = threadIdx.x % TPR * 4, grp = threadIdx.x / TPR;
  const int64_t slot0 = (((int64_t)unit * p.row_tiles + row / RB) * p.chunks) * RB + row % RB;
  __shared__ float xo[NG][D];
  __shared__ float xml[NG][2];
  float M = -INFINITY, L = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  // four chunks at a time, pairs and results asked for together (the pairs first and then the results, one after the other, was five
  // trips to memory for 32 chunks: 4.5 us of a decoding step's 31).  The buffers end with the row's last chunk: what lies past it reads as
  // zeros (the last chunk once more, with a weight of 0, is NaN where a value was infinite).  As selects behind the loads that was 0.1 us,
  // as branches around them 0.2; fetching instructions counts in a kernel of 4 us.  (at most 512 chunks of 32 rows: 8 MiB)
  constexpr int kRaw = 0x00027000;  // untyped, range-checked by the byte
  const int last = (p.chunks - 1) * RB;
  const __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc(p.part + slot0 * D, 0, (last + 1) * D * 4, kRaw);
  const __amdgpu_buffer_rsrc_t pairs = __builtin_amdgcn_make_buffer_rsrc(p.part_ml + slot0 * 2, 0, (last + 1) * 8, kRaw);
  for (int base = grp; base < p.chunks; base += 4 * NG) {
    f32x2 ml[4];
    f32x4 part[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = (base + j * NG) * RB;
      ml[j] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(pairs, s * 8, 0, 0));
      part[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(parts, (s * D + c) * 4, 0, 0));
    }
    float M_new = M;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ml[j][0] = base + j * NG < p.chunks ? ml[j][0] : -INFINITY;
      M_new = __builtin_fmaxf(M_new, ml[j][0]);
    }
    const float ref = M_new == -INFINITY ? 0.f : M_new;
    const float keep = fast_exp2(M - ref);  // (0 before the first chunk with a key)
    M = M_new;
    L *= keep;
    o *= keep;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = fast_exp2(ml[j][0] - ref);
      L += a * ml[j][1];
      o += a * part[j];
    }
  }
  *reinterpret_cast<f32x4*>(&xo[grp][c]) = o;
  if (c == 0) {
    xml[grp][0] = M;
    xml[grp][1] = L;
  }
  __syncthreads();
  if (grp != 0) return;
  float Mt = -INFINITY;
#pragma unroll
  for (int w = 0; w < NG; ++w) Mt = __builtin_fmaxf(Mt, xml[w][0]);
  const float reft = Mt == -INFINITY ? 0.f : Mt;
  float Lt = 0.f;
  f32x4 ot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < NG; ++w) {
    const float a = fast_exp2(xml[w][0] - reft);
    Lt += a * xml[w][1];
    ot += a * *reinterpret_cast<const f32x4*>(&xo[w][c]);
  }
  const int batch = p.by_Hkv.of(unit), kvh = unit - batch * p.Hkv, hd = p.by_Lq.of(row), pos = row - hd * p.Lq, oh = kvh * p.group + hd;
  const float inv = Lt > 0.f ? 1.0f / Lt : 0.f;
  typedef E ex4 __attribute__((ext_vector_type(4)));
  ex4 w;
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = (E)(ot[e] * inv);
  *reinterpret_cast<ex4*>(p.o + (int64_t)batch * p.os[0] + (int64_t)oh * p.os[1] + (int64_t)pos * p.os[2] + c) = w;
  if (p.lse != nullptr && c == 0)
    p.lse[((int64_t)batch * p.Hq + oh) * p.Lq + pos] = Lt > 0.f ? reft + __builtin_log2f(Lt) : INFINITY;
}

}  // namespace fl
