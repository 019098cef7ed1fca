// Backward of the fused attention forward for gfx950: dQ, dK, dV from dO, the forward's inputs and its row statistics.
//
// The reference is forward-only (its FLOP helper models a backward, benchmarks/_utils.py:16-21, but no kernel exists);
// the arithmetic is the textbook one for softmax attention with recomputation:
//   P = exp2(S2 - LSE2),  dP = dO V^T,  dS = P o (dP - Delta) * d(score)/d(qk),  dQ = dS K,  dK = dS^T Q,  dV = P^T dO
// with S2 the modified logits in log2 units, LSE2 the forward's log2-sum-exp2 per row and Delta = rowsum(dO o O).
//
// One kernel template, two roles, no atomics:
//   ROLE_DQ   a workgroup owns 128 query rows of one head and streams the key tiles they attend;
//   ROLE_DKV  a workgroup owns 128 keys of one key/value head (256 in the wide form, BwdTraits) and streams the query tiles (of every
//             query head of the group) that attend them.
// In both roles a lane owns one *owner* position (the column of every accumulator it holds) and its registers run over
// the streamed positions, because every product is issued with the streamed tile as the A operand:
//   X1 = T1 . O1^T   (ROLE_DQ: K.Q^T = S^T;   ROLE_DKV: Q.K^T = S)       v_mfma_f32_32x32x16_bf16
//   X2 = T2 . O2^T   (ROLE_DQ: V.dO^T = dP^T; ROLE_DKV: dO.V^T = dP)
//   acc1 += T1^T . dS  (ROLE_DQ: dQ^T;  ROLE_DKV: dK^T),  ROLE_DKV also acc2 += T2^T . P  (dV^T)
// so the fp32 layout of X1/X2 is the bf16 B-operand layout of the accumulating products (as in the forward kernel) and
// P, dS never leave registers.  T1/T2 are staged in LDS by global_load_lds transfers, two slots, one barrier per tile;
// T^T operands come from the same tiles through the transposing LDS read.
#pragma once
#include "tile_operands.h"

namespace fl {

enum : int { ROLE_DQ = 0, ROLE_DKV = 1 };

struct BParams {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  const bf16_t* o;
  const bf16_t* dout;
  const float* lse;    // [B, Hq, Lq], log2 units; +inf for a row that attends nothing
  float* delta;        // [B, Hq, Lq] scratch: minus rowsum(dO o O)
  bf16_t* dq;
  bf16_t* dk;
  bf16_t* dv;
  int64_t qs[3], ks[3], vs[3], os[3], dos[3], dqs[3], dks[3], dvs[3];  // element strides: batch, head, seq
  int32_t B, Hq, Hkv, Lq, Lk, group;
  float scale, scale_log2;
  int32_t mask_kind, window, prefix;
  int32_t dmin, dmax, pfx;  // attend iff key < Lk && ((dmin <= key - q <= dmax) || key < pfx)
  const int64_t* doc_ids;
  int64_t doc_stride;
  const int64_t* doc_table;  // [B][ceil(L / kDocBlock)][2] = (min, max), as in the forward
  int32_t doc_blocks;
  int32_t alibi_heads;
  float softcap;
  uint32_t drop_thr;      // as in KParams: 0 = no dropout
  uint32_t drop_seed[2];
  float drop_rescale;
  // Bias operands (F_BIAS), addressed as in the forward: element (batch / bdiv, head, query, key) through bbs, 16-bit
  // elements of the call's type or fp32.  They are read from global memory where they are used.
  const void* bias[2];
  int64_t bbs[2][4];
  int32_t bdiv[2];
  int32_t bias_f32[2];
  float* dscores;  // optional [B, Hq, Lq, Lk]: d(loss) / d(score), written by the dQ kernel for the tiles it visits
  // Workgroups per owner tile, each with its share of the streamed steps.  With more than one they leave their
  // fp32 sums in `part`, which bwd_split_sum_kernel adds up:
  // [split][owner tile][wave block of 32 positions][dQ, or dK then dV][register / 4][lane][4]
  float* part;
  int32_t splits;
  // bwd_both_kernel: `part` and `splits` are the dK/dV role's, these the dQ role's
  float* part_dq;
  int32_t splits_dq;
  int32_t dkv_own;  // owner positions per workgroup of the dK/dV launch
  // Divisors, per role (0: dQ, 1: dK/dV).  (batch, head) pairs are dealt head_group at a time
  int32_t head_group;
  Div by_head_group, by_group, by_Hq, by_delta_blocks;
  struct {
    Div by_heads, by_rest, by_oh, by_splits, by_tiles;  // head_group * owner tiles; pairs an XCD leaves over; owner heads; splits; tiles
  } role[2];
};

// dot product of eight 16-bit pairs, the same bits wherever it stands (left to itself the compiler forms two-element dot products of fp16
// in one kernel and not in the other)
template <class E8>
__device__ __forceinline__ float dot8(const E8& a, const E8& b) {
  float s = 0.f;
  if constexpr (std::is_same<E8, f16x8>::value) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) s = dot2acc(f16x2{a[e], a[e + 1]}, f16x2{b[e], b[e + 1]}, s);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) s = __builtin_fmaf((float)a[e], (float)b[e], s);
  }
  return s;
}

// delta[b, h, q] = -sum_d dO[b, h, q, d] * O[b, h, q, d]; one row per group of DV / 8 lanes, delta_blocks workgroups per (batch, head):
// bound by reading both (6.4 TB/s at 4 x 16 x 4096, head dim 128).  For calls whose two roles share a launch; with a launch each, dQ's
// workgroups, which hold dO's rows in any case, form the sums (row_sum in bwd_tile, the same bits).
template <int DV, class E>
__global__ __launch_bounds__(256) void bwd_delta_kernel(const BParams p) {
  fetch_params<BParams>();
  typedef E ex8 __attribute__((ext_vector_type(8)));
  constexpr int LPR = DV / 8, RPB = 256 / LPR;  // lanes per row, 16 bytes each; rows per workgroup
  const int bh = p.by_delta_blocks.of(blockIdx.x), first = (blockIdx.x - bh * ((p.Lq + RPB - 1) / RPB)) * RPB;
  const int b = p.by_Hq.of(bh), h = bh - b * p.Hq, q = first + threadIdx.x / LPR, c = threadIdx.x % LPR;
  float s = 0.f;
  if (q < p.Lq) {
    const ex8 a = *reinterpret_cast<const ex8*>(p.dout + b * p.dos[0] + h * p.dos[1] + q * p.dos[2] + 8 * c);
    const ex8 o = *reinterpret_cast<const ex8*>(p.o + b * p.os[0] + h * p.os[1] + q * p.os[2] + 8 * c);
    s = dot8(a, o);
  }
#pragma unroll
  for (int d = 1; d < LPR; d *= 2) s += __shfl_xor(s, d);
  if (q < p.Lq && c == 0) p.delta[(int64_t)bh * p.Lq + q] = -s;  // stored negated: the consumers add it (or start dP's accumulators from it)
}

// LDS image of a [rows][D] tile that is read both ways: blocks of 16 rows x 64 bytes (1 KiB, a wave's transfer), block after block
// along the row, then down the rows; a row's four 16-byte chunks are exchanged by XOR with row / 4 % 4.  Row-wise reads (16 rows at one
// chunk) and transposing ones (4 rows x 64 bytes) touch every bank once, as with rows kept whole and swizzled over their 16 chunks, but the
// chunk index reaches only two bits into the swizzle: all reads of a kind are at two addresses plus constants (six registers instead of 24 at
// head dim 128).
template <int D>
struct QuadLayout {
  static constexpr int BPR = D / 32;  // blocks along a row
  // byte of 16-byte chunk `chunk` of row `row`
  __host__ __device__ static constexpr unsigned at(int row, int chunk) {
    return (unsigned)((row / 16 * BPR + chunk / 4) * 1024 + row % 16 * 64 + ((chunk % 4) ^ (row / 4 % 4)) * 16);
  }
  // the row and the chunk that 16-byte piece `id` of the image holds
  __host__ __device__ static constexpr int row_of(int id) { return id / 64 / BPR * 16 + id % 64 / 4; }
  __host__ __device__ static constexpr int chunk_of(int id) { return id / 64 % BPR * 4 + ((id % 4) ^ (id % 64 / 16)); }
};
static_assert([]() constexpr {
  for (int id = 0; id < 1024; ++id)
    if (QuadLayout<128>::at(QuadLayout<128>::row_of(id), QuadLayout<128>::chunk_of(id)) != 16u * id || QuadLayout<64>::at(QuadLayout<64>::row_of(id), QuadLayout<64>::chunk_of(id)) != 16u * id ||
        QuadLayout<32>::at(QuadLayout<32>::row_of(id), QuadLayout<32>::chunk_of(id)) != 16u * id) return false;
  return true;
}(), "one place per chunk");

// The image with rows kept whole (TileLayout's two-way swizzle), read through TileOperands: T::WHOLE_ROWS
template <int D>
struct RowLayout {
  static constexpr int CPR = D / 8;
  __device__ static __forceinline__ int row_of(int id) { return id / CPR; }
  __device__ static __forceinline__ int chunk_of(int id) { return TileLayout<D>::swz_kv(id / CPR, id % CPR); }
};

// SHARED_: the role as part of bwd_both_kernel, whose two roles have workgroups of one size.  WIDE_: 256 owner positions per workgroup
// (ROLE_DKV at head dim 128, wide_dkv in api.hip): eight waves own 32 keys each, so that a streamed tile comes in once for twice as many
// keys, K stays in registers and nothing is added up at the end.
template <int D_, int ROLE_, uint32_t FEAT_, class Elem_ = bf16_t, bool SHARED_ = false, bool WIDE_ = false>
struct BwdTraits {
  using Elem = Elem_;  // element type of q, k, v, o, dout and the gradients: bf16_t or f16_t
  static constexpr int D = D_, ROLE = ROLE_;
  static constexpr bool SHARED = SHARED_, WIDE = WIDE_;
  static constexpr uint32_t FEAT = FEAT_;
  static constexpr int OWN = WIDE ? 256 : 128;             // owner positions per workgroup
  static constexpr int OB = OWN / 32;                      // blocks of 32 of them, a wave each (two with QH == 2)
  // ROLE_DKV at D = 128 holds 128 accumulator registers per lane; to still run two waves per SIMD its workgroup has
  // 8 waves, two per owner block, which take the two halves of every streamed tile and add up their partial sums
  // through LDS at the end (one workgroup per CU, 128 KB of LDS).
  static constexpr int QH = ((ROLE == ROLE_DKV || SHARED_) && D_ > 64 && !WIDE) ? 2 : 1;   // waves per owner block
  static constexpr int NW = OB * QH, NT = 64 * NW;
  static constexpr int TB = (D_ <= 64) ? 2 : 1;  // 32-position blocks per wave and step (register budget)
  static constexpr int BT = 32 * TB * QH;                  // streamed positions per step
  static constexpr int KS = D / 16, DB = D / 32;
  static constexpr int TBYTES = BT * D * 2;                // one streamed tile
  static constexpr int T_PER_T = TBYTES / (NT * 16);       // 16-byte transfers per thread per tile
  static_assert(TBYTES % (NT * 16) == 0, "streamed tile must divide evenly over the threads");
  // The order of a step's LDS reads, products and vector work is written out (run_ordered).  Left to the compiler, also with
  // sched_group_barrier, most products stood right behind the wait for their own LDS read, and exponentials in a row.  us, gradients, the
  // compiler's order -> this: head dim 64, 4 x 16 x 4096 causal 502 -> 477, 3 x 16 over 4 of 1000 with a prefix 65.2 -> 58.9, 32 over 10 x 8 of 1139
  // 431 -> 393, documents of 32 over 2 x 8 x 8037 1023 -> 1004, ALiBi and soft-cap 239 -> 230; head dim 128, 4 x 16 x 4096 causal 935 -> 922,
  // documents, 16 over 4 x 4 of 3000, 273 -> 252, ALiBi and soft-cap, 32 over 2 x 4 of 2000, 366 -> 355.  How far the reads run ahead hardly
  // matters (2 to 5 products); documents with ALiBi and a soft-cap spill.
  static constexpr bool ORDERED = ((FEAT_ & ~F_DOC) == 0 || (FEAT_ & ~(F_ALIBI | F_SOFTCAP)) == 0) && D_ >= 64;
  static constexpr int AHEAD = 3;
  // Bias operands without documents: rows kept whole.  The compiler orders those steps, and does it worse with all reads at two addresses.
  // us, blocks of 16 rows -> this: head dim 64, a bias row, 2 x 16 of 300 37.7 -> 36.4, dense 47.4 -> 46.4, dense, 3 x 7 of 1200 266 -> 262, 4 x 16 of
  // 2048 1427 -> 1415; with ALiBi 484 -> 470, with dropout 942 -> 927; head dim 128, dense, 2 x 16 over 4 of 1000 243 -> 239, a row, 4 x 16 of 2048
  // 954 -> 933, with dropout 1158 -> 1134; head dim 32, 43.3 -> 42.7.  Beside ALiBi or the soft-cap the addresses spill at head dim 128 (3 x 7 of
  // 1200: 169 against 183; head dim 32, 2048: 431 against 440), and documents lose (a row, 2 x 16 over 4 of 1000: head dim 64 134 against
  // 142, 128 165 against 175).
  static constexpr bool WHOLE_ROWS = (FEAT_ & F_BIAS) && !(FEAT_ & F_DOC) && (D_ == 64 || !(FEAT_ & (F_ALIBI | F_SOFTCAP)));
  // ROLE_DKV: the owner's K and V rows as operands in registers, where there is room, instead of in LDS
  static constexpr bool K_REGS = ROLE == ROLE_DKV && ORDERED && (WIDE || D <= 64), V_REGS = ROLE == ROLE_DQ || (K_REGS && D <= 64);
  static constexpr int OBYTES = (ROLE == ROLE_DKV) ? OWN * D * 2 : 0;  // owner tile kept in LDS (ROLE_DKV: K and V)
  static constexpr int O_PER_T = OBYTES / (NT * 16);
  static_assert(OBYTES % (NT * 16) == 0, "owner tile must divide evenly over the threads");
  // ROLE_DKV also stages the streamed rows' statistics (LSE and Delta, fp32) with every tile: 1 KiB each per slot
  static constexpr int SBYTES = (ROLE == ROLE_DKV) ? 1024 : 0;
  static constexpr int T1_OFF = 0, T2_OFF = 2 * TBYTES, O1_OFF = 4 * TBYTES, O2_OFF = O1_OFF + (K_REGS ? 0 : OBYTES),
                       S1_OFF = O2_OFF + (V_REGS ? 0 : OBYTES), S2_OFF = S1_OFF + 2 * SBYTES;
  // Document masks: the list of live tiles (up to LIST of them at a time, with one count per wave behind it) and, per slot, the ids
  // of the streamed positions
  static constexpr bool DOC = FEAT_ & F_DOC;
  static constexpr int LIST = 1024, LIST_OFF = S2_OFF + 2 * SBYTES, IDS_OFF = LIST_OFF + (DOC ? LIST * 4 + 64 : 0);
  static constexpr int LDS_BYTES = IDS_OFF + (DOC ? 2 * BT * 8 : 0);
  static_assert(QH == 1 || LDS_BYTES >= 4 * 64 * 64 * 4, "the partial sums of one accumulator set must fit in LDS");
  // ROLE_DQ: dP's accumulators start from a tile of -Delta that stays in registers, where there is room for it
  static constexpr bool DELTA_TILE = ROLE_ == ROLE_DQ && (ORDERED || (D_ <= 64 && !(FEAT_ & (F_BIAS | F_DROPOUT))));
  // two steps per turn of the loop, see there (without addresses in registers the dK/dV kernel is 1 to 4 % slower with it; bias
  // operands have no registers for it)
  static constexpr bool UNROLL2 = (ROLE == ROLE_DQ || ORDERED) && !(FEAT_ & F_BIAS);
  static constexpr int WAVES_PER_EU = 2;
  static constexpr bool WIDE_X2 = D_ > 64;                      // dP's fp32 tile declared next to S's
  static constexpr bool EARLY_X2 = ROLE == ROLE_DQ && WIDE_X2;  // and its MFMAs issued right after those of S
};

// The order of a step (run_ordered): products X1 of every block of 32 streamed positions, X2 of every block, dV's (unless DQ), dS's, of TB
// blocks with KS products each and DB columns of 32.  Behind product m the first weights(m) pairs of weights and gradients(m) pairs of score
// gradients have been formed, eight pairs per block.
template <bool DQ, int TB, int KS, int DB>
struct OrderedStep {
  static constexpr int X2 = TB * KS, VP = 2 * X2, KP = VP + (DQ ? 0 : 2 * TB * DB), M = KP + 2 * TB * DB;  // first of each kind, and their number
  static constexpr int weights(int m) {
    if (DQ && TB == 2) return m < 5 ? 0 : m < 9 ? 2 * (m - 4) : m < 16 ? m : 16;
    return m < KS ? 0 : m < KS + 8 * TB ? m - KS : 8 * TB;
  }
  static constexpr int gradients(int m) {
    if (DQ && TB == 2) return m < 13 ? 0 : m < 15 ? 3 * (m - 12) : m < 17 ? 8 : m < 20 ? 8 + 2 * (m - 16) : 16;
    if (DQ) return m < VP - 1 ? 0 : m < VP + 3 ? m - VP + 5 : 8;
    if (TB == 2) return m < VP + 5 ? 0 : m < VP + 12 ? 2 * (m - VP - 4) : 16;
    return m < VP ? 0 : m < VP + 8 ? m - VP : 8;
  }
  // (unless DQ) which four rows' LSE are read in front of product m, into one of two places, or -1
  static constexpr int lse_quad(int m) {
    const int g = m - KS + 1;
    return !DQ && g >= 0 && g % 2 == 0 && g / 2 < 4 * TB ? g / 2 : -1;
  }
  // Every weight behind its block's X1, with its LSE in place; every gradient behind its weight and its block's X2; every product of 16 positions
  // behind their eight pairs; nothing left out.
  static constexpr bool holds() {
    if (TB == 1 ? KS != 8 || DB != 4 : TB != 2 || KS != 4 || DB != 2) return false;  // (the shapes that the places are written for)
    if (weights(-1) != 0 || gradients(-1) != 0 || weights(M - 1) != 8 * TB || gradients(M - 1) != 8 * TB) return false;
    int lse[2] = {-1, -1};
    for (int m = 0; m < M; ++m) {
      if (m >= KP ? gradients(m - 1) < 4 * ((m - KP) / DB) + 4 : m >= VP && weights(m - 1) < 4 * ((m - VP) / DB) + 4) return false;
      if (lse_quad(m) >= 0) lse[lse_quad(m) % 2] = lse_quad(m);
      // (by fours: under the soft-cap the mask follows each four pairs of weights)
      if (weights(m) < weights(m - 1) || gradients(m) < gradients(m - 1) || gradients(m) > weights(m) / 4 * 4) return false;
      for (int w = weights(m - 1); w < weights(m); ++w)
        if (m < (w / 8 + 1) * KS - 1 || (!DQ && lse[w / 2 % 2] != w / 2)) return false;
      for (int w = gradients(m - 1); w < gradients(m); ++w)
        if (m < X2 + (w / 8 + 1) * KS - 1) return false;
    }
    return true;
  }
};

// One workgroup's share of the work of a role: workgroup `block` of tiles * splits.  SPLIT: several workgroups per owner tile
// (one at run time is fine), compiled apart: with the second epilogue in it the dK/dV kernel at head dim 128 is 4 %
// slower (another register allocation throughout).
template <class T, bool SPLIT>
__device__ __forceinline__ void bwd_tile(const BParams& p, const int block, const int splits, float* const part_sums) {
  constexpr int D = T::D, ROLE = T::ROLE, TB = T::TB, BT = T::BT, KS = T::KS, DB = T::DB, NT = T::NT;
  constexpr uint32_t FEAT = T::FEAT;
  constexpr bool kAlibi = FEAT & F_ALIBI, kSoftcap = FEAT & F_SOFTCAP, kDoc = FEAT & F_DOC, kBias = FEAT & F_BIAS;
  constexpr bool kDQ = ROLE == ROLE_DQ;
  using E = typename T::Elem;  // pointers in BParams are typed bf16_t whatever E is: 16 opaque bits
  typedef E ex8 __attribute__((ext_vector_type(8)));
  typedef E ex4 __attribute__((ext_vector_type(4)));
  constexpr bool kDrop = FEAT & F_DROPOUT;
  constexpr float kLog2e = 1.4426950408889634f;
  using L = typename std::conditional<T::WHOLE_ROWS, RowLayout<D>, QuadLayout<D>>::type;
  using Quad = QuadLayout<D>;
  using Ops = TileOperands<D, E>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
  const int r = lane % 32, h = lane / 32;
  const int ow = wave % T::OB;   // owner block of this wave
  const int qh = wave / T::OB;   // which part of every streamed tile this wave takes (0 unless QH == 2)

  // workgroup -> (batch, owner head, owner tile).  All owner tiles of one head stream the same tensors, so they should
  // run at the same time on one XCD (its L2 then serves all but the first read): consecutive workgroup ids land on
  // different XCDs, hence ids are regrouped to give every XCD a contiguous run of (batch, head) pairs, head by head.
  // Under causal-like masks the work of a tile grows with the query position (ROLE_DQ) or shrinks with the key position
  // (ROLE_DKV): heads are taken four at a time and their tiles dealt longest first, so the grid drains on short ones.
  const auto& divs = p.role[kDQ ? 0 : 1];
  const int n_own = kDQ ? (p.Lq + T::OWN - 1) / T::OWN : (p.Lk + T::OWN - 1) / T::OWN;
  const int oh = kDQ ? p.Hq : p.Hkv;
  // The splits of a tile are dealt next to each other.
  const int nbh = p.B * oh;
  int ot, bh, split = 0;
  {
    int i = block, run = nbh, base = 0;
    if (nbh % 8 == 0) {
      run = nbh / 8;
      base = (i % 8) * run;
      i /= 8;
    }
    if constexpr (SPLIT) {
      const int tile = divs.by_splits.of(i);
      split = i - tile * splits;
      i = tile;
    }
    const int G = p.head_group;
    const int g = divs.by_heads.of(i), rem = i - g * (G * n_own);
    const int gg = min(G, run - G * g);
    const int rank = (gg == G ? p.by_head_group : divs.by_rest).of(rem);  // 0 = longest under a causal-like mask
    bh = base + G * g + rem - rank * gg;
    ot = kDQ ? n_own - 1 - rank : rank;
  }
  const int batch = divs.by_oh.of(bh), ohead = bh - batch * oh;
  const int o0 = ot * T::OWN;               // first owner position of the workgroup
  const int o1 = min(o0 + T::OWN, kDQ ? p.Lq : p.Lk);
  const int opos = o0 + ow * 32 + r;        // this lane's owner position (a query row or a key)
  const int olen = kDQ ? p.Lq : p.Lk;
  const int slen = kDQ ? p.Lk : p.Lq;       // streamed sequence length
  const int kvh = kDQ ? (int)p.by_group.of(ohead) : ohead;

  // ---- streamed tile range [t_lo, t_hi] for the workgroup's owner range [o0, o1) under the positional mask ----------
  int t_lo = 0, t_hi = (slen + BT - 1) / BT - 1;
  {
    const bool causal_like = p.mask_kind == MASK_CAUSAL || p.mask_kind == MASK_SLIDING || p.mask_kind == MASK_DOC_CAUSAL;
    if (kDQ) {  // keys attended by queries [o0, o1)
      if (causal_like) t_hi = min(t_hi, (o1 - 1) / BT);
      if (p.mask_kind == MASK_PREFIX) t_hi = min(t_hi, (max(o1, p.prefix) - 1) / BT);
      if (p.mask_kind == MASK_SLIDING) t_lo = max(0, o0 - p.window) / BT;
    } else {    // queries that attend keys [o0, o1)
      if (causal_like) t_lo = o0 / BT;
      if (p.mask_kind == MASK_PREFIX && o0 >= p.prefix) t_lo = o0 / BT;
      if (p.mask_kind == MASK_SLIDING) t_hi = min(t_hi, (int)min((int64_t)o1 - 1 + p.window, (int64_t)slen - 1) / BT);
    }
  }
  const int n_tiles = t_hi >= t_lo ? t_hi - t_lo + 1 : 0;
  const int n_heads = kDQ ? 1 : p.group;   // ROLE_DKV walks the query heads of its group
  const int all_steps = n_tiles * n_heads;
  // first step of a split: all * split / splits, rounded down
  auto split_start = [&](int all, int split) FL_INLINE -> int {
    const int whole = divs.by_splits.of(all);
    return whole * split + divs.by_splits.of((all - whole * splits) * split);
  };
  const int s_first = SPLIT ? split_start(all_steps, split) : 0;
  const int n_steps = SPLIT ? split_start(all_steps, split + 1) : all_steps;  // this workgroup's steps: [s_first, n_steps)

  // ---- per-lane constants ---------------------------------------------------------------------------------------------
  float cap_k1 = 0.f, cap_c = 0.f;
  bool cap_on = false;  // kernels compiled with the soft-cap also serve calls without one
  if constexpr (kSoftcap) {
    cap_on = p.softcap > 0.f;
    cap_k1 = cap_on ? p.scale / p.softcap * 2.0f * kLog2e : 0.f;
    cap_c = p.softcap * kLog2e;
  }
  int64_t odoc = 0;
  if constexpr (kDoc) odoc = p.doc_ids[(int64_t)batch * p.doc_stride + min(opos, olen - 1)];
  int64_t own_mn = 0, own_mx = 0;
  if constexpr (kDoc) doc_range(p.doc_table + (int64_t)batch * p.doc_blocks * 2, o0, o1, own_mn, own_mx);

  // ---- owner operands ---------------------------------------------------------------------------------------------------
  // ROLE_DQ: Q and dO fragments of this lane's query row live in registers (B operands), with its LSE and Delta.
  // ROLE_DKV: so do this lane's K and V rows where the registers have room for them (T::K_REGS, T::V_REGS); otherwise the workgroup's are staged
  // in LDS once and read as B operands where they are used.
  ex8 o1f[kDQ || T::K_REGS ? KS : 1], o2f[T::V_REGS ? KS : 1];
  float lse_o = 0.f, delta_o = 0.f;  // delta_o: minus this row's rowsum(dO o O)
  const bf16_t* kptr = p.k + (int64_t)batch * p.ks[0] + (int64_t)kvh * p.ks[1];
  const bf16_t* vptr = p.v + (int64_t)batch * p.vs[0] + (int64_t)kvh * p.vs[1];
  if constexpr (kDQ) {
    const int qr = min(opos, p.Lq - 1);
    const bf16_t* qp = p.q + (int64_t)batch * p.qs[0] + (int64_t)ohead * p.qs[1] + (int64_t)qr * p.qs[2];
    const bf16_t* dp = p.dout + (int64_t)batch * p.dos[0] + (int64_t)ohead * p.dos[1] + (int64_t)qr * p.dos[2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      o1f[ks] = *reinterpret_cast<const ex8*>(qp + ks * 16 + 8 * h);
      o2f[ks] = *reinterpret_cast<const ex8*>(dp + ks * 16 + 8 * h);
    }
    const int64_t row = ((int64_t)batch * p.Hq + ohead) * p.Lq + qr;
    lse_o = p.lse[row];
    if constexpr (T::SHARED) {
      delta_o = p.delta[row];
    } else {
      // minus rowsum(dO o O), in the order of bwd_delta_kernel, left for the dK/dV launch that follows
      const bf16_t* op = p.o + (int64_t)batch * p.os[0] + (int64_t)ohead * p.os[1] + (int64_t)qr * p.os[2];
      float sum[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const ex8 o = *reinterpret_cast<const ex8*>(op + ks * 16 + 8 * h);
        sum[ks] = xhalf_sum(dot8(o2f[ks], o));
      }
#pragma unroll
      for (int d = 1; d < KS; d *= 2)
#pragma unroll
        for (int ks = 0; ks < KS; ks += 2 * d) sum[ks] += sum[ks + d];
      delta_o = -sum[0];
      if (h == 0 && opos < p.Lq) p.delta[row] = delta_o;
    }
  }

  if constexpr (T::K_REGS) {
    const bf16_t* kp = kptr + (int64_t)min(opos, p.Lk - 1) * p.ks[2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) o1f[ks] = *reinterpret_cast<const ex8*>(kp + ks * 16 + 8 * h);
  }
  if constexpr (!kDQ && T::V_REGS) {
    const bf16_t* vp = vptr + (int64_t)min(opos, p.Lk - 1) * p.vs[2];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) o2f[ks] = *reinterpret_cast<const ex8*>(vp + ks * 16 + 8 * h);
  }

  // ---- global -> LDS transfers of a [rows][D] tile into its image (QuadLayout or RowLayout) -----------------------------------------
  // lane l of a 1 KiB transfer writes LDS bytes [16 l, 16 l + 16); it fetches the chunk that the layout has there.  Rows past `valid` repeat
  // the last valid row (their contributions are masked).
  auto load_tile = [&](uint64_t base, int64_t stride, int valid, unsigned lds_off, int n_per_t) FL_INLINE {
    const unsigned lds0 = (unsigned)(uintptr_t)smem + lds_off + wave * 1024;
    for (int it = 0; it < n_per_t; ++it) {
      const int id = it * NT + tid;
      const unsigned off = (unsigned)(min(L::row_of(id), valid - 1) * (int)stride + L::chunk_of(id) * 8) * 2u;
      dma16(base, off, lds0 + it * NT * 16);
    }
  };
  // The streamed operands: whole tiles are fetched at one per-lane offset that does not change from tile to tile (the rows of a
  // thread's transfers lie a multiple of the swizzle's period apart), from scalar addresses that advance by a tile per step; the last,
  // ragged one works its offsets out.  (Worked out at every transfer, with a step's head and tile as quotient and rest of its number, this was
  // a third of the instructions of the shared launch's loops; us for a training step: 4 x 16 x 4096 causal, head dim 128, 1260 -> 1237, 64, 677 ->
  // 668; 16 over 3 x 4 of 1000 with a prefix 86.8 -> 84.9; 32 over 7 x 8 of 306, head dim 128, 104.9 -> 100.8.)  ROLE_DKV: the statistics of the streamed rows (LSE, Delta) ride the tile transfers into LDS, 4 bytes
  // per lane, so that the loop holds no ordinary global load: the wait such a load needs would also wait for the tile transfers that are
  // in flight for the next step.
  constexpr int ROWS_PER_T = NT / (D / 8);
  static_assert(NT % (D / 8) == 0 && ROWS_PER_T % 16 == 0, "one offset for all transfers of a thread");
  struct Operand {
    uint64_t base;       // of the batch entry's (or, ROLE_DQ, of the head's) first row
    int64_t head_bytes;  // ROLE_DKV: from one query head to the next
    uint32_t tile_bytes, row_bytes;
    unsigned off;
  };
  auto operand = [&](const bf16_t* ptr, const int64_t (&st)[3]) FL_INLINE -> Operand {
    const uint32_t row_bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)st[2] * 2u));
    return {uniform_ptr(ptr), uniform_i64(st[1] * 2), row_bytes * BT, row_bytes,
            (unsigned)L::row_of(tid) * row_bytes + L::chunk_of(tid) * 16u};
  };
  const Operand s1 = operand(kDQ ? kptr : p.q + (int64_t)batch * p.qs[0], kDQ ? p.ks : p.qs);
  const Operand s2 = operand(kDQ ? vptr : p.dout + (int64_t)batch * p.dos[0], kDQ ? p.vs : p.dos);
  const uint64_t lse_at = uniform_ptr(p.lse), delta_at = uniform_ptr(p.delta);
  auto load_tiles = [&](int tile, int hd, int slot) FL_INLINE {
    const int valid = slen - tile * BT;
    auto at = [&](const Operand& s) FL_INLINE -> uint64_t {
      uint64_t a = s.base + (uint64_t)(uint32_t)tile * s.tile_bytes;
      if constexpr (!kDQ) a += (uint64_t)(s.head_bytes * hd);
      return a;
    };
    const uint64_t a1 = at(s1), a2 = at(s2);
    if (valid >= BT) {
      const unsigned lds0 = (unsigned)(uintptr_t)smem + slot * T::TBYTES + wave * 1024;
#pragma unroll
      for (int it = 0; it < T::T_PER_T; ++it) dma16(a1 + (uint64_t)(it * ROWS_PER_T * s1.row_bytes), s1.off, lds0 + T::T1_OFF + it * NT * 16);
#pragma unroll
      for (int it = 0; it < T::T_PER_T; ++it) dma16(a2 + (uint64_t)(it * ROWS_PER_T * s2.row_bytes), s2.off, lds0 + T::T2_OFF + it * NT * 16);
    } else {
      load_tile(a1, kDQ ? p.ks[2] : p.qs[2], valid, T::T1_OFF + slot * T::TBYTES, T::T_PER_T);
      load_tile(a2, kDQ ? p.vs[2] : p.dos[2], valid, T::T2_OFF + slot * T::TBYTES, T::T_PER_T);
    }
    if constexpr (!kDQ) {
      if (wave == 0) {
        // one wave brings both arrays (every wave waits for all of its own transfers before the barrier, so the counts
        // need not match).  Lane l fetches row t0 + l; lanes past the end of the tile or of the sequence repeat the last
        // valid row (those rows are masked).
        static_assert(BT <= 64, "one lane per streamed row");
        const uint64_t row0 = (uint64_t)(((int64_t)batch * p.Hq + hd) * p.Lq + tile * BT) * 4u;
        const unsigned off = (unsigned)min(lane, min(BT, valid) - 1) * 4u;
        dma4(lse_at + row0, off, (unsigned)(uintptr_t)smem + T::S1_OFF + slot * T::SBYTES);
        dma4(delta_at + row0, off, (unsigned)(uintptr_t)smem + T::S2_OFF + slot * T::SBYTES);
      }
    }
  };
  // the ids of the streamed positions, for a step that compares them (positions past the end repeat the last one)
  auto load_ids = [&](int tile, int slot) FL_INLINE {
    const int t0 = tile * BT;
    if (wave != T::NW - 1) return;
#pragma unroll
    for (int j = 0; j < BT / 32; ++j) {
      const int word = 64 * j + lane;  // of the tile's ids, two words each
      const unsigned off = (unsigned)(min(word / 2, slen - 1 - t0) * 8 + word % 2 * 4);
      dma4(uniform_ptr(p.doc_ids + (int64_t)batch * p.doc_stride + t0), off, (unsigned)(uintptr_t)smem + T::IDS_OFF + slot * BT * 8 + j * 256);
    }
  };

  // ---- LDS operand reads --------------------------------------------------------------------------------------------------
  // QuadLayout: two addresses per kind of read, held in registers (the empty asm keeps the compiler from working them out again at every
  // read); everything else is a constant of the instruction.
  unsigned a_row[2], a_own[2], a_tr[2];
  if constexpr (!T::WHOLE_ROWS) {
    const unsigned lds0 = (unsigned)(uintptr_t)smem;
    const int i16 = lane % 16;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      a_row[j] = lds0 + Quad::at(qh * TB * 32 + r, 2 * j + h);
      asm volatile("" : "+v"(a_row[j]));
      if constexpr (!kDQ) {
        a_own[j] = lds0 + T::O1_OFF + Quad::at(ow * 32 + r, 2 * j + h);
        asm volatile("" : "+v"(a_own[j]));
      }
      a_tr[j] = lds0 + Quad::at(qh * TB * 32 + 8 * j + 4 * h + i16 / 4, (lane / 16) % 2 * 2 + i16 % 4 / 2) + i16 % 2 * 8;
      asm volatile("" : "+v"(a_tr[j]));
    }
  }
  typedef __attribute__((address_space(3))) const ex8* lds_ex8_ptr;
  typedef s16x4 __attribute__((address_space(3))) * lds_s16x4_ptr;
  // row-wise: 8 consecutive elements [row][16 ks + 8 h, +8), row = 32 (qh TB + sb) + r of a streamed tile (A operand of X1/X2) or this
  // lane's row of an owner tile (B operand)
  auto frag_row = [&](unsigned tile_off, int sb, int ks) FL_INLINE -> ex8 {
    if constexpr (T::WHOLE_ROWS) return Ops::rows(smem + tile_off, (qh * TB + sb) * 32 + r, ks, h);
    return *(lds_ex8_ptr)(a_row[ks % 2] + tile_off + Quad::at(32 * sb, 4 * (ks / 2)));
  };
  auto frag_own = [&](unsigned tile_off, int ks) FL_INLINE -> ex8 {
    if constexpr (T::WHOLE_ROWS) return Ops::rows(smem + tile_off, ow * 32 + r, ks, h);
    return *(lds_ex8_ptr)(a_own[ks % 2] + (tile_off - T::O1_OFF) + Quad::at(0, 4 * (ks / 2)));
  };
  // transposing: A operand of the accumulating products for 16-position chunk c (of this wave's) and column block db
  auto frag_tr = [&](unsigned tile_off, int c, int db) FL_INLINE -> ex8 {
    if constexpr (T::WHOLE_ROWS) return Ops::columns(smem + tile_off, 2 * TB * qh + c, db, lane, h);
    ex8 f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const ex4 b4 = __builtin_bit_cast(ex4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(a_tr[j] + tile_off + Quad::at(16 * c, 4 * db))));
#pragma unroll
      for (int e = 0; e < 4; ++e) f[4 * j + e] = b4[e];
    }
    return f;
  };

  // -Delta of this lane's row, as the tile that dP's accumulators start from (the asm keeps it in registers: copied into the
  // accumulators on every step it would cost what it saves)
  f32x16 delta_tile;
  if constexpr (T::DELTA_TILE) {
#pragma unroll
    for (int i = 0; i < 16; ++i) delta_tile[i] = delta_o;
    asm volatile("" : "+v"(delta_tile));
  }
  f32x16 acc1[DB], acc2[kDQ ? 1 : DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc1[db][i] = 0.f;
  if constexpr (!kDQ) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc2[db][i] = 0.f;
  }

  if (kDoc ? n_tiles > 0 : n_steps > s_first) {
    if constexpr (!kDQ) {
      const int valid = o1 - o0;
      if constexpr (!T::K_REGS) load_tile(uniform_ptr(kptr + (int64_t)o0 * p.ks[2]), p.ks[2], valid, T::O1_OFF, T::O_PER_T);
      if constexpr (!T::V_REGS) load_tile(uniform_ptr(vptr + (int64_t)o0 * p.vs[2]), p.vs[2], valid, T::O2_OFF, T::O_PER_T);
    }
  }

  // Workgroup-level class of a streamed tile: nothing of it is attended by the workgroup's owner range (returns true: document
  // ranges apart; positional emptiness inside [t_lo, t_hi] only occurs for a prefix-LM mask), everything is (`full`),
  // or every position of the tile and of the owner range carries one and the same document id (`doc_uniform`).
  auto classify_tile = [&](int tile, bool& full, bool& doc_uniform) FL_INLINE -> bool {
    const int t0 = tile * BT;
    const int s1 = min(t0 + BT, slen);
    const int w0 = T::WIDE ? o0 + 32 * ow : o0, w1 = T::WIDE ? min(w0 + 32, olen) : o1;  // (WIDE: this wave's own positions)
    if (T::WIDE && w0 >= olen) return true;
    const int qa = kDQ ? w0 : t0, qb_ = kDQ ? w1 : s1, ka = kDQ ? t0 : w0, kb_ = kDQ ? s1 : w1;
    const int cls = classify_positional(p.mask_kind, qa, qb_, ka, kb_, p.window, p.prefix);
    bool skip = cls == TILE_EMPTY;
    // every pair of the step attended: the positional mask holds everywhere and both ranges lie inside the sequences
    full = cls == TILE_FULL && t0 + BT <= slen && w0 + (T::WIDE ? 32 : T::OWN) <= olen;
    doc_uniform = false;
    if constexpr (kDoc) {
      int64_t mn, mx;
      doc_range(p.doc_table + (int64_t)batch * p.doc_blocks * 2, t0, s1, mn, mx);
      skip = skip || mx < own_mn || mn > own_mx;
      doc_uniform = mn == mx && own_mn == own_mx && mn == own_mn;
      full = full && doc_uniform;
    }
    return skip;
  };
  // Sum of the bias operands at (query, key) of head `hd` (positions inside the sequences)
  auto bias_at = [&](int qpos, int kpos, int hd) FL_INLINE -> float {
    float b = 0.f;
    if constexpr (kBias) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        if (p.bias[nb] == nullptr) continue;
        const int64_t off = (int64_t)(batch / p.bdiv[nb]) * p.bbs[nb][0] + (int64_t)hd * p.bbs[nb][1] +
                            (int64_t)qpos * p.bbs[nb][2] + (int64_t)kpos * p.bbs[nb][3];
        b += p.bias_f32[nb] ? static_cast<const float*>(p.bias[nb])[off] : (float)static_cast<const E*>(p.bias[nb])[off];
      }
    }
    return b;
  };
  // element predicate as an interval of the register offset `off` (8 (i / 4) + i % 4): lo <= off <= hi
  auto bounds = [&](int sbase, int& lo, int& hi) FL_INLINE {
    if constexpr (kDQ) {
      // streamed = key, owner = query: key < Lk && (dmin <= key - q <= dmax || key < pfx)
      const int rel = sbase - opos;
      hi = min(p.Lk - sbase - 1, max(p.dmax - rel, p.pfx - sbase - 1));
      lo = p.dmin - rel;
    } else {
      // streamed = query, owner = key: q < Lq && (dmin <= key - q <= dmax || key < pfx), key = opos
      const int rel = opos - sbase;  // key - q at off = 0; key - q = rel - off
      hi = min(p.Lq - sbase - 1, opos < p.pfx ? (1 << 29) : rel - p.dmin);
      lo = opos < p.pfx ? -(1 << 29) : rel - p.dmax;
      if (opos >= p.Lk) hi = -(1 << 29);
    }
  };
  auto attended = [&](int t0, int sbase, int slot, int off, int lo, int hi, bool doc_uniform) FL_INLINE -> bool {
    bool ok = (off <= hi) & (off >= lo);
    if constexpr (kDoc) {
      if (!doc_uniform) ok = ok & (*reinterpret_cast<const int64_t*>(smem + T::IDS_OFF + slot * BT * 8 + (sbase - t0 + off) * 8) == odoc);
    }
    return ok;
  };
  // ALiBi slope of the streamed head in log2 units, worked out where the head changes
  int slope_head = -1;
  float slope_l2 = 0.f;
  // The blocks of 32 streamed positions of a step with their instructions in a prescribed order (T::ORDERED, see there).  Products: X1 of
  // every block, X2 of every block, (ROLE_DKV) dV's, dS's (OrderedStep).  In front of product m stand the LDS reads of product m + AHEAD,
  // behind it its share of the vector work.
  auto run_ordered = [&](auto tile, const int shead, const int slot, bool full, bool doc_uniform) FL_INLINE {  // (compiled only where it is called)
    const int t0 = tile * BT;
    const unsigned t1 = T::T1_OFF + slot * T::TBYTES, t2 = T::T2_OFF + slot * T::TBYTES;
    using Step = OrderedStep<kDQ, TB, KS, DB>;
    constexpr int X2 = Step::X2, VP = Step::VP, KP = Step::KP, M = Step::M;
    constexpr int AHEAD = T::AHEAD, RING = AHEAD + 1;
    static_assert(Step::holds(), "everything formed behind its products and ahead of those that take it");
    f32x16 x1[TB], x2[TB];
    ex8 fa[RING], fb[T::V_REGS ? 1 : RING];  // operands in flight
    f32x4 lse4[2];
    ex8 pf[2 * TB], dsf[2 * TB];
#pragma unroll
    for (int sb = 0; sb < TB; ++sb)
#pragma unroll
      for (int i = 0; i < 16; ++i) x1[sb][i] = 0.f;
    // 4 consecutive streamed rows' values of a staged per-row fp32 array
    auto rows4 = [&](unsigned staged_off, int sb, int g) FL_INLINE -> f32x4 {
      return *reinterpret_cast<const f32x4*>(smem + staged_off + slot * T::SBYTES + (32 * (qh * TB + sb) + 4 * h + 8 * g) * 4);
    };
    auto read = [&](auto mt) FL_INLINE {
      constexpr int m = decltype(mt)::value;
      if constexpr (m < X2) {
        fa[m % RING] = frag_row(t1, m / KS, m % KS);
        if constexpr (!kDQ && !T::K_REGS) fb[m % RING] = frag_own(T::O1_OFF, m % KS);
      } else if constexpr (m < VP) {
        constexpr int sb = (m - X2) / KS, ks = (m - X2) % KS;
        if constexpr (!kDQ && ks == 0) {  // dP starts from minus Delta
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 nd = rows4(T::S2_OFF, sb, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) x2[sb][4 * g + e] = nd[e];
          }
        }
        fa[m % RING] = frag_row(t2, sb, ks);
        if constexpr (!kDQ && !T::V_REGS) fb[m % RING] = frag_own(T::O2_OFF, ks);
      } else if constexpr (m < KP) {
        fa[m % RING] = frag_tr(t2, (m - VP) / DB, (m - VP) % DB);
      } else if constexpr (m < M) {
        fa[m % RING] = frag_tr(t1, (m - KP) / DB, (m - KP) % DB);
      }
    };
    if constexpr (kAlibi) {
      if (shead != slope_head) {
        slope_head = shead;
        slope_l2 = p.alibi_heads > 0 ? exp2f(-8.0f * (float)(shead + 1) / (float)p.alibi_heads) * kLog2e : 0.f;
      }
    }
    int lo[TB], hi[TB];     // the element mask's bounds, where it is asked
    float alibi0[TB];       // the ALiBi term at register offset 0
    unsigned out[TB];       // positions outside it
    static_while<0, AHEAD>([&](auto m) FL_INLINE { read(m); return true; });
    static_while<0, M>([&](auto mt) FL_INLINE {
      constexpr int m = decltype(mt)::value;
      read(std::integral_constant<int, m + AHEAD>{});
      if constexpr (!kDQ) {  // the LSE of four rows, two products ahead of their weights (the place is free: of the last but one)
        constexpr int q = Step::lse_quad(m);
        if constexpr (q >= 0) lse4[q % 2] = rows4(T::S1_OFF, q / 4, q % 4);
      }
      if constexpr (m < X2) {
        if constexpr (kDQ || T::K_REGS) x1[m / KS] = mfma32(fa[m % RING], o1f[m % KS], x1[m / KS]);
        else x1[m / KS] = mfma32(fa[m % RING], fb[m % RING], x1[m / KS]);
      } else if constexpr (m < VP) {
        constexpr int sb = (m - X2) / KS, ks = (m - X2) % KS;
        if constexpr (kDQ && ks == 0) x2[sb] = mfma32(fa[m % RING], o2f[0], delta_tile);
        else if constexpr (kDQ || T::V_REGS) x2[sb] = mfma32(fa[m % RING], o2f[ks], x2[sb]);
        else x2[sb] = mfma32(fa[m % RING], fb[m % RING], x2[sb]);
      } else if constexpr (m < KP) {
        acc2[(m - VP) % DB] = mfma32(fa[m % RING], pf[(m - VP) / DB], acc2[(m - VP) % DB]);
      } else {
        acc1[(m - KP) % DB] = mfma32(fa[m % RING], dsf[(m - KP) / DB], acc1[(m - KP) % DB]);
      }
#pragma unroll
      for (int w = Step::weights(m - 1); w < Step::weights(m); ++w) {
        const int sb = w / 8, sbase = t0 + 32 * (qh * TB + sb) + 4 * h;  // streamed position of register 0
        if (w % 8 == 0) {
          if constexpr (kAlibi) alibi0[sb] = slope_l2 * (float)(kDQ ? sbase - opos : opos - sbase);
          if (!full) {  // uniform over the workgroup or the wave; the asm keeps it a branch
            bounds(sbase, lo[sb], hi[sb]);
            asm volatile("" : "+v"(lo[sb]), "+v"(hi[sb]));
            out[sb] = outside_word(lo[sb], hi[sb]);
            // the ids of a tile with more than one, as bits besides.  (As a comparison, a branch and a choice at every score: us, forward and gradients,
            // causal documents, 4 x 16 x 2048, head dim 64, 181 -> 149; 16 over 4 x 8000 409 -> 339; 2 x 16 x 4096, head dim 128, 380 -> 335.)
            if constexpr (kDoc) {
              if (!doc_uniform) {
                const unsigned char* ids = smem + T::IDS_OFF + slot * BT * 8 + (sbase - t0) * 8;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
#pragma unroll
                  for (int off = 8 * g; off < 8 * g + 4; ++off) out[sb] |= *reinterpret_cast<const int64_t*>(ids + off * 8) == odoc ? 0u : 1u << off;
                  // (a branch, and four ids at a time, which leaves scratch of 8 bytes a lane where head dim 64 has both roles in one launch and of 20 in
                  // dK and dV at 128.  Two leave none at 64 and the same 20 at 128, but gradients of documents take longer: 4 x 16 x 2048, head dim 64,
                  // 112 -> 114, 16 over 4 x 8000 163 -> 169, 2 x 16 x 4096, head dim 128, 261 -> 268; in a loop 36 bytes; sixteen at once spill.)
                  asm volatile("" : "+v"(out[sb]));
                }
              }
            }
            if constexpr (!kSoftcap) minus_inf_outside(x1[sb], out[sb]);
          }
        }
#pragma unroll
        for (int e = w % 8 * 2; e < w % 8 * 2 + 2; ++e) {
          const float x = x1[sb][e], lse = kDQ ? lse_o : lse4[w / 2 % 2][e % 4], c0 = kAlibi ? alibi0[sb] - lse : -lse;
          const int off = 8 * (e / 4) + e % 4;
          float s2, dfac = 1.0f;  // logit in log2 units minus the LSE; d(score) / d(qk * scale)
          if constexpr (kSoftcap) {
            const float th = __builtin_fmaf(fast_rcp(fast_exp2(x * cap_k1) + 1.0f), -2.0f, 1.0f);  // tanh(x * scale / cap)
            s2 = __builtin_fmaf(th, cap_c, c0);
            dfac = __builtin_fmaf(-th, th, 1.0f);
          } else {
            s2 = __builtin_fmaf(x, p.scale_log2, c0);
          }
          if constexpr (kAlibi) s2 = __builtin_fmaf(kDQ ? slope_l2 : -slope_l2, (float)off, s2);
          float pv = fast_exp2(s2);
          if constexpr (!kDQ) pf[2 * sb + e / 8][e % 8] = (E)pv;
          x1[sb][e] = kSoftcap ? pv * dfac : pv;
        }
        // Under the soft-cap -inf would not do as a score: what is masked is taken out again, eight positions at a time.  (Asked at every score, and
        // with the calls without a cap in the same kernel, a step was 64 branches with two or three vector instructions between them.  us, forward
        // and gradients, causal, ALiBi and a soft-cap, with the branches -> this: 4 x 16 x 2048, head dim 128, 447 -> 426, scores far out 457 -> 436; over 4
        // heads, head dim 64, 293 -> 277, 299 -> 286; 3 x 16 over 4 of 1000, fp16, 117 -> 101.  ALiBi alone, which has kernels without the cap
        // now, 436 -> 364 and 276 -> 208.)
        if constexpr (kSoftcap) {
          if (w % 4 == 3 && !full) {
            const int half = w % 8 / 4;
            int lost[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const int i = 8 * half + e;
              lost[e] = __builtin_amdgcn_sbfe((int)out[sb], 8 * (i / 4) + i % 4, 1);
              x1[sb][i] = __uint_as_float(~(uint32_t)lost[e] & __float_as_uint(x1[sb][i]));
            }
            if constexpr (!kDQ) {
              u32x4 two = __builtin_bit_cast(u32x4, pf[2 * sb + half]);
#pragma unroll
              for (int e = 0; e < 4; ++e) two[e] &= ~(((uint32_t)lost[2 * e] & 0xFFFFu) | ((uint32_t)lost[2 * e + 1] << 16));
              pf[2 * sb + half] = __builtin_bit_cast(ex8, two);
            }
            asm volatile("" : "+v"(x1[sb][8 * half]));  // (a branch)
          }
        }
      }
#pragma unroll
      for (int w = Step::gradients(m - 1); w < Step::gradients(m); ++w)
#pragma unroll
        for (int e = w % 8 * 2; e < w % 8 * 2 + 2; ++e) dsf[w / 8 * 2 + e / 8][e % 8] = (E)(x1[w / 8][e] * x2[w / 8][e]);
      __builtin_amdgcn_sched_barrier(0);
      return true;
    });
  };
  // One step: the tile in ring slot `slot` against the owner operands.
  auto run_tile = [&](int tile, const int shead, int slot, bool full, bool doc_uniform) FL_INLINE {
    if constexpr (T::ORDERED) return run_ordered(tile, shead, slot, full, doc_uniform);
    const int t0 = tile * BT;
    {
      const unsigned t1 = T::T1_OFF + slot * T::TBYTES, t2 = T::T2_OFF + slot * T::TBYTES;
      // ---- X1 = T1 . O1^T, then the weights; X2 = T2 . O2^T, then dS (one after the other: the two fp32 tiles are
      // never live together, which is what lets 128 accumulator registers fit) ----------------------------------------------
      // register i of block sb is streamed position t0 + 32 (qh TB + sb) + 8 (i / 4) + 4 h + i % 4
      if constexpr (kAlibi) {
        if (shead != slope_head) {
          slope_head = shead;
          slope_l2 = p.alibi_heads > 0 ? exp2f(-8.0f * (float)(shead + 1) / (float)p.alibi_heads) * kLog2e : 0.f;
        }
      }
      // 4 consecutive streamed rows of a staged per-row fp32 array
      auto rows4 = [&](unsigned staged_off, int q4) FL_INLINE -> f32x4 {
        return *reinterpret_cast<const f32x4*>(smem + staged_off + slot * T::SBYTES + (q4 - t0) * 4);
      };
      // (document ids beside bias operands: the mask goes with each weight, sixteen ids in flight do not fit in the registers)
      constexpr bool kMaskApart = !(kDoc && kBias);
      constexpr bool kMaskScores = FEAT == 0 || FEAT == F_DOC;
      // X2 = T2 . O2^T (dP).  At D = 128 its fp32 tile is declared out here, next to X1's, and (ROLE_DQ) its MFMAs are issued
      // right after X1's, before the weights' vector work; at D = 64 it lives in the block that consumes it.  Both choices
      // are measured: the first is 15 % faster at D = 128 and 1-2 % slower at D = 64.
      f32x16 x2_wide[TB];
      // dP's accumulators start from zero, or (without dropout) from the -Delta of their rows, staged or (ROLE_DQ) this lane's, which
      // saves the subtraction per score later
      constexpr bool kDeltaInit = !kDrop && (!kDQ || T::DELTA_TILE);
      auto init_x2 = [&](f32x16 (&x2)[TB]) FL_INLINE {
#pragma unroll
        for (int sb = 0; sb < TB; ++sb) {
          if constexpr (T::DELTA_TILE) {
            x2[sb] = delta_tile;
            continue;
          }
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4 nd = {0.f, 0.f, 0.f, 0.f};
            if constexpr (kDeltaInit) nd = rows4(T::S2_OFF, t0 + 32 * (qh * TB + sb) + 4 * h + 8 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) x2[sb][4 * g + e] = nd[e];
          }
        }
      };
      auto second_product = [&](f32x16 (&x2)[TB]) FL_INLINE {
        init_x2(x2);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          ex8 b2;
          if constexpr (kDQ) b2 = o2f[ks]; else b2 = frag_own(T::O2_OFF, ks);
#pragma unroll
          for (int sb = 0; sb < TB; ++sb)
            x2[sb] = mfma32(frag_row(t2, sb, ks), b2, x2[sb]);
        }
      };
      ex8 pf[2 * TB], dsf[2 * TB];
      float pd[TB][16];  // weight times d(score) / d(qk * scale); with dropout its sign bit marks a dropped weight
      // dropout: the owner position's share of the hash argument (see drop_pair_hash); the streamed head changes from step
      // to step in ROLE_DKV
      uint32_t drop_o = 0;
      if constexpr (kDrop) {
        const uint32_t s0 = drop_head_seed(p.drop_seed[0], p.drop_seed[1], (uint32_t)(batch * p.Hq + shead));
        drop_o = s0 + (kDQ ? (uint32_t)opos * kDropQ : (uint32_t)(opos >> 1) * kDropK);
      }
      float pv[TB][16];
      {
        f32x16 x1[TB];
#pragma unroll
        for (int sb = 0; sb < TB; ++sb)
#pragma unroll
          for (int i = 0; i < 16; ++i) x1[sb][i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          ex8 b1;
          if constexpr (kDQ) b1 = o1f[ks]; else b1 = frag_own(T::O1_OFF, ks);
#pragma unroll
          for (int sb = 0; sb < TB; ++sb)
            x1[sb] = mfma32(frag_row(t1, sb, ks), b1, x1[sb]);
        }
        if constexpr (kMaskScores) {
          if (!full) {  // workgroup-uniform; here, so that everything from the weights on is one block to be ordered
#pragma unroll
            for (int sb = 0; sb < TB; ++sb) {
              const int sbase = t0 + 32 * (qh * TB + sb) + 4 * h;
              int lo, hi;
              bounds(sbase, lo, hi);
              asm volatile("" : "+v"(lo), "+v"(hi));
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                if (!attended(t0, sbase, slot, 8 * (i / 4) + i % 4, lo, hi, doc_uniform)) x1[sb][i] = -INFINITY;
              }
            }
          }
        }
        // where the registers allow and it pays (measured), dP's MFMAs are issued before the weights' vector work
        if constexpr (T::EARLY_X2) second_product(x2_wide);
#pragma unroll
        for (int sb = 0; sb < TB; ++sb) {
          const int sbase = t0 + 32 * (qh * TB + sb) + 4 * h;  // streamed position of register 0
          // what does not depend on the register goes into one addend: minus the row's LSE, and the ALiBi term at
          // off = 0 (key - q = rel0 + off in ROLE_DQ, rel0 - off in ROLE_DKV), which leaves slope * off as one
          // multiply-add with a literal per score
          int lo = 0, hi = 0;
          if constexpr (!kMaskApart) bounds(sbase, lo, hi);
          const float alibi0 = kAlibi ? slope_l2 * (float)(kDQ ? sbase - opos : opos - sbase) : 0.f;
          const float slope_off = kDQ ? slope_l2 : -slope_l2;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4 lse4;
            if constexpr (!kDQ) lse4 = rows4(T::S1_OFF, sbase + 8 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int i = 4 * g + e, off = 8 * g + e;
              const float x = x1[sb][i];
              const float lse = kDQ ? lse_o : lse4[e];
              const float c0 = kAlibi ? alibi0 - lse : -lse;  // (0 - lse would be an instruction of its own)
              float s2, dfac = 1.0f;  // logit in log2 units minus the LSE; d(score) / d(qk * scale)
              if constexpr (kSoftcap) {
                const float ex = fast_exp2(x * cap_k1);
                const float rc = fast_rcp(ex + 1.0f);
                const float th = __builtin_fmaf(rc, -2.0f, 1.0f);  // tanh(x * scale / cap)
                s2 = cap_on ? __builtin_fmaf(th, cap_c, c0) : __builtin_fmaf(x, p.scale_log2, c0);
                dfac = cap_on ? __builtin_fmaf(-th, th, 1.0f) : 1.0f;
              } else {
                s2 = __builtin_fmaf(x, p.scale_log2, c0);
              }
              if constexpr (kAlibi) s2 = __builtin_fmaf(slope_off, (float)off, s2);
              if constexpr (kBias) {
                const int sp = min(sbase + off, slen - 1), op = min(opos, olen - 1);
                s2 = __builtin_fmaf(bias_at(kDQ ? op : sp, kDQ ? sp : op, shead), kLog2e, s2);
              }
              pv[sb][i] = fast_exp2(s2);
              if (!kMaskApart && !full && !attended(t0, sbase, slot, off, lo, hi, doc_uniform)) pv[sb][i] = 0.f;
              pd[sb][i] = kSoftcap ? dfac : 1.0f;
            }
          }
        }
      }
      if constexpr (T::WIDE_X2 && !T::EARLY_X2) second_product(x2_wide);
      {
#pragma unroll
        for (int sb = 0; sb < TB; ++sb) {
          const int sbase = t0 + 32 * (qh * TB + sb) + 4 * h;
          if (kMaskApart && !kMaskScores && !full) {  // workgroup-uniform
            // (where -inf would not do as a score: under the soft-cap.  The asm keeps this a branch: as selects it was three vector and two scalar instructions per score on every step,
            // full ones included, beside the four that make a weight and its gradient.  It stands behind the products that
            // do not need it, which the compiler can then interleave.  Gradients of 4 x 16 x 4096, this and the unrolled
            // dQ loop: head dim 128 unmasked 2.00 -> 1.85 ms, causal 1.10 -> 1.01; head dim 64 1.135 -> 0.985, 0.62 -> 0.545)
            int lo, hi;
            bounds(sbase, lo, hi);
            asm volatile("" : "+v"(lo), "+v"(hi));
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              if (!attended(t0, sbase, slot, 8 * (i / 4) + i % 4, lo, hi, doc_uniform)) pv[sb][i] = 0.f;
            }
          }
#pragma unroll
          for (int i = 0; i < 16; ++i) pd[sb][i] = kSoftcap ? pv[sb][i] * pd[sb][i] : pv[sb][i];
          if constexpr (kDrop) {
            // ROLE_DQ: registers (i, i + 1), i even, are the key pair (sbase + off) / 2 of this lane's query: one hash.
            // ROLE_DKV: register i is query sbase + off against this lane's key: its own hash, the key's half of it.
#pragma unroll
            for (int i = 0; i < 16; i += kDQ ? 2 : 1) {
              const int off = 8 * (i / 4) + i % 4;
              if constexpr (kDQ) {
                const uint32_t x = drop_pair_hash(drop_o + (uint32_t)((sbase + off) >> 1) * kDropK);
                const bool keep0 = (x & 0xFFFFu) >= p.drop_thr, keep1 = (x >> 16) >= p.drop_thr;
                pv[sb][i] = keep0 ? pv[sb][i] : 0.f;
                pv[sb][i + 1] = keep1 ? pv[sb][i + 1] : 0.f;
                pd[sb][i] = keep0 ? pd[sb][i] : -pd[sb][i];
                pd[sb][i + 1] = keep1 ? pd[sb][i + 1] : -pd[sb][i + 1];
              } else {
                const uint32_t x = drop_pair_hash(drop_o + (uint32_t)(sbase + off) * kDropQ);
                const bool keep = ((x >> (16 * (opos & 1))) & 0xFFFFu) >= p.drop_thr;
                pv[sb][i] = keep ? pv[sb][i] : 0.f;
                pd[sb][i] = keep ? pd[sb][i] : -pd[sb][i];
              }
            }
          }
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) pf[2 * sb + j][e] = (E)pv[sb][8 * j + e];
        }
      }
      {
        f32x16 x2_here[TB];
        f32x16 (&x2)[TB] = pick<T::WIDE_X2>(x2_wide, x2_here);
        if constexpr (!T::WIDE_X2) {
          init_x2(x2);
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            ex8 b2;
            if constexpr (kDQ) b2 = o2f[ks]; else b2 = frag_own(T::O2_OFF, ks);
#pragma unroll
            for (int sb = 0; sb < TB; ++sb)
              x2[sb] = mfma32(frag_row(t2, sb, ks), b2, x2[sb]);
          }
        }
#pragma unroll
        for (int sb = 0; sb < TB; ++sb) {
          const int sbase = t0 + 32 * (qh * TB + sb) + 4 * h;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4 dl4 = {0.f, 0.f, 0.f, 0.f};  // minus Delta of the four rows, unless dP already started from it
            if constexpr (!kDQ && !kDeltaInit) dl4 = rows4(T::S2_OFF, sbase + 8 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int i = 4 * g + e;
              float ds;
              if constexpr (kDrop) {
                // d(loss) / d(weight) is dP / (1 - p) where the weight was kept and 0 where it was dropped
                const bool kept = __builtin_bit_cast(int, pd[sb][i]) >= 0;
                ds = __builtin_fabsf(pd[sb][i]) * ((kept ? x2[sb][i] * p.drop_rescale : 0.f) + (kDQ ? delta_o : dl4[e]));
              } else {
                ds = kDeltaInit ? pd[sb][i] * x2[sb][i] : pd[sb][i] * (x2[sb][i] + (kDQ ? delta_o : dl4[e]));
              }
              dsf[2 * sb + i / 8][i % 8] = (E)ds;
              if constexpr (kBias && kDQ) {
                // the gradient with respect to the score; with the soft-cap switched on ds carries d(cap) / d(qk * scale)
                // besides, which is not part of it: the host refuses dscores then
                const int key = sbase + 8 * g + e;
                if (p.dscores != nullptr && opos < p.Lq && key < p.Lk)
                  p.dscores[(((int64_t)batch * p.Hq + ohead) * p.Lq + opos) * p.Lk + key] = ds;
              }
            }
          }
        }
      }
      // ---- acc1 += T1^T . dS,  acc2 += T2^T . P -------------------------------------------------------------------------------
      if constexpr (!kDQ && kMaskScores) {  // (dV first: its products cover the vector work that forms dS)
#pragma unroll
        for (int c = 0; c < 2 * TB; ++c)
#pragma unroll
          for (int db = 0; db < DB; ++db) acc2[db] = mfma32(frag_tr(t2, c, db), pf[c], acc2[db]);
      }
#pragma unroll
      for (int c = 0; c < 2 * TB; ++c)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          acc1[db] = mfma32(frag_tr(t1, c, db), dsf[c], acc1[db]);
          if constexpr (!kDQ && !kMaskScores) acc2[db] = mfma32(frag_tr(t2, c, db), pf[c], acc2[db]);
        }
    }
  };
  if constexpr (kDoc) {
    // Most tiles of the range are dead: documents apart.  The live ones are listed first, a wave per LIST / NW tiles with their
    // table reads in flight together; every head of the group then walks the list, and splits share out what is on it.  (Read one after
    // the other as the loop got there, with two dependent table reads each, the dead tiles were most of the time: 2 x 32 over 8
    // heads of 8037 positions in documents of up to 4000, head dim 64: 672 and 1503 us for the two roles, now 495 and 992.)
    uint32_t* const list = reinterpret_cast<uint32_t*>(smem + T::LIST_OFF);
    int* const counts = reinterpret_cast<int*>(smem + T::LIST_OFF + T::LIST * 4);
    for (int w0 = t_lo; w0 <= t_hi; w0 += T::LIST) {
      constexpr int PER = T::LIST / T::NW / 64;  // tiles per lane
      const int mine = w0 + wave * (T::LIST / T::NW);
      uint32_t entry[PER];
      uint64_t live[PER];
      int count = 0;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int tile = mine + 64 * j + lane;
        bool full = false, doc_uniform = false;
        const bool skip = tile > t_hi || classify_tile(min(tile, t_hi), full, doc_uniform);
        entry[j] = (uint32_t)tile << 2 | (full ? 1u : 0u) | (doc_uniform ? 2u : 0u);
        live[j] = __builtin_amdgcn_ballot_w64(!skip);
        count += __builtin_popcountll(live[j]);
      }
      __syncthreads();  // (the previous list has been walked)
      if (lane == 0) counts[wave] = count;
      __syncthreads();
      int n_live = 0, at = 0;
#pragma unroll
      for (int w = 0; w < T::NW; ++w) {
        const int c = __builtin_amdgcn_readfirstlane(counts[w]);
        at += w < wave ? c : 0;
        n_live += c;
      }
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        if ((live[j] >> lane) & 1) list[at + __builtin_popcountll(live[j] & ((1ull << lane) - 1))] = entry[j];
        at += __builtin_popcountll(live[j]);
      }
      __syncthreads();
      const int all_live = n_live * n_heads;
      const int s_first = SPLIT ? split_start(all_live, split) : 0;
      const int n_steps = SPLIT ? split_start(all_live, split + 1) : all_live;
      if (s_first >= n_steps) continue;
      int head = kDQ ? ohead : kvh * p.group + s_first / n_live, i = s_first % n_live;
      auto at_list = [&](int i) FL_INLINE { return (uint32_t)__builtin_amdgcn_readfirstlane((int)list[i]); };
      uint32_t e = at_list(i);
      load_tiles((int)(e >> 2), head, 0);
      if (!(e & 2)) load_ids((int)(e >> 2), 0);
      dma_wait<0>();
      for (int s = s_first, slot = 0; s < n_steps; ++s, slot ^= 1) {
        __syncthreads();  // publishes slot `slot` (every wave waited for its own transfers) and frees the other slot
        const uint32_t now = e;
        const int head_now = head;
        if (s + 1 < n_steps) {
          if (++i == n_live) {
            i = 0;
            ++head;
          }
          e = at_list(i);
          load_tiles((int)(e >> 2), head, slot ^ 1);
          if (!(e & 2)) load_ids((int)(e >> 2), slot ^ 1);
        }
        run_tile((int)(now >> 2), head_now, slot, now & 1, now & 2);
        dma_wait<0>();
      }
    }
    dma_wait<0>();  // (a workgroup that found nothing to do has asked for its owner rows all the same)
  } else {
    // positional masks: every step of [t_lo, t_hi] is visited (a dead one only occurs under a prefix-LM mask); ROLE_DKV walks them for
    // every query head of the group.  The step to be fetched next is (tile, head); its place goes from step to step (worked out from
    // the step's number it was two divisions per step).
    int tile = t_lo + s_first, head = kDQ ? ohead : kvh * p.group;
    if (!kDQ && SPLIT && s_first >= n_tiles && n_tiles > 0) {
      const int skipped = s_first / n_tiles;
      head += skipped;
      tile -= skipped * n_tiles;
    }
    int tile_now = tile, head_now = head;
    auto fetch_next = [&](int slot) FL_INLINE {
      load_tiles(tile, head, slot);
      ++tile;
      if (!kDQ && tile > t_hi) {
        tile = t_lo;
        ++head;
      }
    };
    auto step_at = [&](int s, const int slot) FL_INLINE {
      __syncthreads();  // publishes slot `slot` (every wave waited for its own transfers) and frees the other slot
      const int t = tile_now, hd = head_now;
      tile_now = tile;
      head_now = head;
      if (s + 1 < n_steps) fetch_next(slot ^ 1);
      bool full, doc_uniform;
      if (!classify_tile(t, full, doc_uniform)) run_tile(t, hd, slot, full, doc_uniform);
      dma_wait<0>();
    };
    if constexpr (T::UNROLL2) {
      // (two steps per turn of the loop: the ring slot is then a constant, part of the LDS instructions' offsets instead of 20
      // address additions per step)
      if (n_steps > s_first) fetch_next(0);
      dma_wait<0>();
      int s = s_first;
      for (; s + 1 < n_steps; s += 2) {
        step_at(s, 0);
        step_at(s + 1, 1);
      }
      if (s < n_steps) step_at(s, 0);
    } else {
      if (n_steps > s_first) fetch_next(0);
      dma_wait<0>();
      for (int s = s_first; s < n_steps; ++s) step_at(s, (s - s_first) & 1);
    }
  }

  // ---- the waves of one owner block add up their partial sums: the second wave parks its accumulators in LDS (element
  // (register, lane) of owner block ow at float ((ow * 64 + register) * 64 + lane): consecutive lanes, no conflicts) ----
  if constexpr (T::QH == 2) {
    float* park = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int set = 0; set < (kDQ ? 1 : 2); ++set) {
      __syncthreads();  // the tiles (set 0) or the previous set's sums (set 1) have been read
      if (qh == 1) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) park[((ow * 64 + db * 16 + i) * 64) + lane] = set == 0 ? acc1[db][i] : acc2[kDQ ? 0 : db][i];
      }
      __syncthreads();
      if (qh == 0) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float x = park[((ow * 64 + db * 16 + i) * 64) + lane];
            if (set == 0) acc1[db][i] += x; else acc2[kDQ ? 0 : db][i] += x;
          }
      }
    }
  }

  if (SPLIT && splits > 1) {
    if (qh == 0) {
      constexpr int SETS = kDQ ? 1 : 2;
      float* to = part_sums + ((((int64_t)split * nbh * n_own + (int64_t)bh * n_own + ot) * 4 + ow) * SETS * DB * 16 * 64) + lane * 4;
#pragma unroll
      for (int set = 0; set < SETS; ++set)
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            f32x4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = set == 0 ? acc1[db][4 * g + e] : acc2[kDQ ? 0 : db][4 * g + e];
            *reinterpret_cast<f32x4*>(to + (set * DB * 4 + db * 4 + g) * 256) = x;
          }
    }
    return;
  }

  // ---- epilogue: register i of block db is column 32 db + 8 (i / 4) + 4 h + i % 4 of this lane's owner row ---------------
  if (opos < olen && qh == 0) {
    bf16_t* out1 = kDQ ? p.dq + (int64_t)batch * p.dqs[0] + (int64_t)ohead * p.dqs[1] + (int64_t)opos * p.dqs[2]
                       : p.dk + (int64_t)batch * p.dks[0] + (int64_t)ohead * p.dks[1] + (int64_t)opos * p.dks[2];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        ex4 o4;
#pragma unroll
        for (int e = 0; e < 4; ++e) o4[e] = (E)(acc1[db][4 * g + e] * p.scale);
        *reinterpret_cast<ex4*>(out1 + 32 * db + 8 * g + 4 * h) = o4;
      }
    if constexpr (!kDQ) {
      bf16_t* out2 = p.dv + (int64_t)batch * p.dvs[0] + (int64_t)ohead * p.dvs[1] + (int64_t)opos * p.dvs[2];
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          ex4 o4;
#pragma unroll
          for (int e = 0; e < 4; ++e) o4[e] = (E)(kDrop ? acc2[db][4 * g + e] * p.drop_rescale : acc2[db][4 * g + e]);
          *reinterpret_cast<ex4*>(out2 + 32 * db + 8 * g + 4 * h) = o4;
        }
    }
  }
}

template <class T>
__global__ __launch_bounds__(T::NT) __attribute__((amdgpu_waves_per_eu(T::WAVES_PER_EU, T::WAVES_PER_EU)))
void bwd_kernel(const BParams p) {
  fetch_params<BParams>();
  bwd_tile<T, false>(p, blockIdx.x, 1, nullptr);
}

// Both roles in one launch, dK/dV first: neither needs the other, and a small call's tails and gaps cost as much as its work.
template <class TQ, class TKV>
__global__ __launch_bounds__(TQ::NT) __attribute__((amdgpu_waves_per_eu(TQ::WAVES_PER_EU, TQ::WAVES_PER_EU)))
void bwd_both_kernel(const BParams p) {
  static_assert(TQ::NT == TKV::NT, "one workgroup size");
  // (documents with bias operands at head dim 64: the parameters then spill, us, 2 x 16 x 2048 157 against 170, unmasked documents 285 / 312)
  if constexpr (!(TQ::D == 64 && TQ::FEAT == (F_DOC | F_BIAS))) fetch_params<BParams>();
  const int n_kv = p.B * p.Hkv * ((p.Lk + TKV::OWN - 1) / TKV::OWN) * p.splits;
  if ((int)blockIdx.x < n_kv) bwd_tile<TKV, true>(p, blockIdx.x, p.splits, p.part);
  else bwd_tile<TQ, true>(p, blockIdx.x - n_kv, p.splits_dq, p.part_dq);
}

// Adds up the splits of one owner tile's block of 32 positions and writes its rows of dQ, of dK (set 0) or of dV (set 1).
// Reads in the order the sums were left (1 KiB per wave and load); a workgroup's stores fill whole rows.
template <class T>
__device__ __forceinline__ void bwd_sum_block(const BParams& p, const int block, const int set, const int splits, const float* const part) {
  constexpr int DB = T::DB, SETS = T::ROLE == ROLE_DQ ? 1 : 2;
  constexpr bool kDQ = T::ROLE == ROLE_DQ;
  using E = typename T::Elem;
  typedef E ex4 __attribute__((ext_vector_type(4)));
  const int olen = kDQ ? p.Lq : p.Lk, oh = kDQ ? p.Hq : p.Hkv, n_own = (olen + T::OWN - 1) / T::OWN;
  const auto& divs = p.role[kDQ ? 0 : 1];
  const int tile = block / 4, bh = divs.by_tiles.of(tile), batch = divs.by_oh.of(bh), head = bh - batch * oh;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int pos = (tile - bh * n_own) * T::OWN + block % 4 * 32 + lane % 32;
  if (pos >= olen) return;
  const int64_t split_stride = (int64_t)p.B * oh * n_own * 4 * SETS * DB * 16 * 64;
  const float* from = part + ((int64_t)block * SETS + set) * DB * 16 * 64 + lane * 4;
  const float factor = set == 0 ? p.scale : (T::FEAT & F_DROPOUT) ? p.drop_rescale : 1.0f;
  bf16_t* out = kDQ ? p.dq + (int64_t)batch * p.dqs[0] + (int64_t)head * p.dqs[1] + (int64_t)pos * p.dqs[2]
                : set == 0 ? p.dk + (int64_t)batch * p.dks[0] + (int64_t)head * p.dks[1] + (int64_t)pos * p.dks[2]
                           : p.dv + (int64_t)batch * p.dvs[0] + (int64_t)head * p.dvs[1] + (int64_t)pos * p.dvs[2];
  f32x4 x[DB];  // wave w takes the register groups w, w + 4, ...: DB of the block's 4 DB
#pragma unroll
  for (int j = 0; j < DB; ++j) x[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < splits; ++s)
#pragma unroll
    for (int j = 0; j < DB; ++j) x[j] += *reinterpret_cast<const f32x4*>(from + s * split_stride + (4 * j + wave) * 256);
#pragma unroll
  for (int j = 0; j < DB; ++j) {  // register group 4 j + w: columns 32 j + 8 w + 4 h ...
    ex4 o4;
#pragma unroll
    for (int e = 0; e < 4; ++e) o4[e] = (E)(x[j][e] * factor);
    *reinterpret_cast<ex4*>(out + 32 * j + 8 * wave + 4 * (lane / 32)) = o4;
  }
}

// Workgroups [0, 8 tiles) dK and dV of every block of 32 keys when that role was split, the others dQ.
template <class TQ, class TKV>
__global__ __launch_bounds__(256) void bwd_split_sum_kernel(const BParams p) {
  fetch_params<BParams>();
  int block = blockIdx.x;
  if (p.splits > 1) {
    const int n_kv = p.B * p.Hkv * ((p.Lk + TKV::OWN - 1) / TKV::OWN) * 8;
    if (block < n_kv) return bwd_sum_block<TKV>(p, block / 2, block % 2, p.splits, p.part);
    block -= n_kv;
  }
  bwd_sum_block<TQ>(p, block, 0, p.splits_dq, p.part_dq);
}

}  // namespace fl
