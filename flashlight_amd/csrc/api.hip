// C ABI of libflashlight_amd.so: argument validation (host only), instance selection, launch.
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "flashlight_amd.h"
#include "bwd_instances.h"
#include "instances.h"
#include "pairbias_bwd_instances.h"
#include "pairbias_instances.h"
#include "rows_instances.h"
#include "stripe_instances.h"

namespace fl {
// Builds (min, max) of the document ids of every block of kDocBlock positions.
static __global__ void doc_table_kernel(const int64_t* ids, int64_t ids_stride, int L, int nblocks, int total, int64_t* table) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  int b = i / nblocks, blk = i % nblocks;
  const int64_t* p = ids + (int64_t)b * ids_stride;
  int p0 = blk * kDocBlock, p1 = min(L, p0 + kDocBlock);
  // (the loads are independent of one another: unrolled, they are all in flight together instead of one round trip
  // to memory each; positions past the end repeat the last one)
  int64_t x[kDocBlock];
#pragma unroll
  for (int j = 0; j < kDocBlock; ++j) x[j] = p[min(p0 + j, p1 - 1)];
  int64_t mn = x[0], mx = x[0];
#pragma unroll
  for (int j = 1; j < kDocBlock; ++j) {
    mn = x[j] < mn ? x[j] : mn;
    mx = x[j] > mx ? x[j] : mx;
  }
  table[2 * (int64_t)i] = mn;
  table[2 * (int64_t)i + 1] = mx;
}

// Forward pre-pass for document masks, one workgroup of 1024 threads per (batch, query tile of `bm` rows), straight from
// the ids: lists the key tiles (of `bn` keys) that some row of the query tile attends, with the class of each for every
// wave of the forward (`rw` rows per wave): EMPTY when the id ranges of the tile's keys and the wave's rows do not meet,
// FULL when both are the same single id and the positional part of the mask agrees, ONE_DOC when they are and it does not, PARTIAL otherwise.  Valid for
// arbitrary (unsorted, negative) ids.  The lists are the same for every head.  Output per workgroup: word 0 = number of
// entries, then the entries in key order (bits 0-15 tile index, two class bits per wave from bit 16 on).
// A wave per key tile reads its ids with one coalesced load and leaves their (min, max) in LDS (every load of a wave is in flight before
// the first is looked at: the kernel is a chain of round trips to memory with little to do in between); the place of this query tile
// in the order is found; a thread per key tile classifies it for every wave; the non-empty entries are compacted.
//
// The order: the query tiles of a batch row by falling length of their tile lists (ties by falling index), so that the workgroups still running
// when the grid drains are short ones whatever the document layout.  ORDERS: every workgroup works out the lengths of all query tiles, by a
// binary search each where the ids are sorted and pair by pair where they are not, and writes its own place: a second launch for it was 5 of
// the 15 us of the pre-pass (16384 ids, 16 heads, us for the forward with its pre-pass: 139.9 -> 136.3).  The lengths count the key tiles whose
// range meets the whole query tile's; any order gives the same results.  Without ORDERS doc_order_kernel follows.
//
// ORDERS pays while all workgroups run at once (doc_orders): a compute unit holds one, and every one of them reads the ids of all key tiles, not
// only those up to its diagonal, and looks at all pairs of tiles where the ids are unsorted.  us, two launches -> one, documents of 64 to 512 unless
// said, head dim 64: 1 x 16 x 8192 64.3 -> 63.0, 1 x 16 x 16384 (to 2048) 108 -> 103, 1 x 8 x 32768 83.0 -> 76.3, unmasked 101 -> 94, ids
// unsorted 770 -> 778; head dim 128, 1 x 8 x 32768 113 -> 106, unsorted 1034 -> 1055.  Beyond: 40000 (313 workgroups) 104 -> 116, 65536 119 -> 130,
// unsorted 1538 -> 1657, 262144 656 -> 1063; 6 x 8 x 8192 97 -> 101.  Few query tiles per row, whose order is soon found: 8 x 16 x 2048, head dim
// 128, 85.0 -> 86.6.
constexpr int kDocWaves = 4;  // waves of the forward that a query tile is classified for, at most
template <bool ORDERS>
static __global__ __launch_bounds__(1024) void doc_lists_kernel(const int64_t* ids, int64_t ids_stride, int L, int mask_kind,
                                                                int bm, int rw, int bn, int n_qtiles, int nk, int list_stride,
                                                                uint32_t* lists, int32_t* order) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  int64_t* krange = reinterpret_cast<int64_t*>(lds_raw);                // [nk][2] = (min, max) id of a key tile
  uint32_t* tl = reinterpret_cast<uint32_t*>(lds_raw + (size_t)nk * 16);  // [nk] counts per query tile, then uncompacted entries
  __shared__ int64_t qrange[2 * kDocWaves];  // (min, max) id of the rows of each wave of the forward
  __shared__ uint32_t few[2];                // [0] ids are unsorted, [1] this tile's place
  __shared__ uint16_t kept[16];              // entries per wave (104 bytes of static LDS: the longest call, 8185 key tiles, leaves 128)
  constexpr int kWaves = 16, kBatch = 16;
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int b = blockIdx.x / n_qtiles, qt = blockIdx.x % n_qtiles;
  const int nw = bm / rw, q0 = qt * bm;
  const int64_t* idb = ids + (int64_t)b * ids_stride;
  const bool causal = mask_kind == MASK_DOC_CAUSAL;
  // rows past L repeat the last row (a wave without valid rows is EMPTY for every tile whatever its range)
  const int64_t qid = idb[min(q0 + min(wave, nw - 1) * rw + lane % rw, L - 1)];
  // key tiles some row may attend under the positional part of the mask: all of them, or those up to the diagonal
  const int t_end = causal ? min(nk, (min(q0 + bm, L) - 1) / bn + 1) : nk;
  const int nj = (bn + 63) / 64;  // loads per lane that cover one tile's ids
  if (tid < 2) few[tid] = 0;
  const int turn = ORDERS ? blockIdx.x / 8 : 0;  // (where a workgroup begins: all of an XCD's would ask for the same lines at the same time)
  const int n_read = ORDERS ? nk : t_end;
  for (int t0 = wave; t0 < n_read || t0 == wave; t0 += kWaves * kBatch) {
    int64_t lo[kBatch], hi[kBatch];
    auto tile = [&](int u) FL_INLINE { return t0 + kWaves * ((u + turn) % kBatch); };
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int k0 = min(tile(u), n_read - 1) * bn;
      lo[u] = hi[u] = idb[min(k0 + lane % bn, L - 1)];
      for (int j = 1; j < nj; ++j) {
        const int64_t x = idb[min(k0 + j * 64 + lane, L - 1)];
        lo[u] = x < lo[u] ? x : lo[u];
        hi[u] = x > hi[u] ? x : hi[u];
      }
    }
    if (t0 == wave) {  // (every wave passes here exactly once)
      int64_t mn, mx;
      wave_id_range(qid, mn, mx);
      if (lane == 0 && wave < nw) {
        qrange[2 * wave] = mn;
        qrange[2 * wave + 1] = mx;
      }
    }
    if constexpr (ORDERS) {
      // lane u keeps tile u's range: the first id where all are the same, the others are reduced one by one (reduced as they come, the
      // sixteen were 3 us)
      uint32_t mixed = 0;
      int64_t mn = 0, mx = 0;
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int64_t first = uniform_i64(lo[u]);
        if (__builtin_amdgcn_ballot_w64(lo[u] != first || hi[u] != first) != 0 && tile(u) < n_read) mixed |= 1u << u;
        mn = lane == u ? first : mn;
      }
      mx = mn;
#pragma unroll 1
      for (; mixed != 0; mixed &= mixed - 1) {
        const int which = (int)__builtin_ctz(mixed);
        int64_t x = lo[0], y = hi[0];
#pragma unroll
        for (int u = 1; u < kBatch; ++u) {
          x = which == u ? lo[u] : x;
          y = which == u ? hi[u] : y;
        }
        int64_t least, most, unused;
        wave_id_range(x, least, most);
        if (nj > 1) wave_id_range(y, unused, most);
        mn = lane == which ? least : mn;
        mx = lane == which ? most : mx;
      }
      if (lane < kBatch && tile(lane) < n_read) {
        krange[2 * tile(lane)] = mn;
        krange[2 * tile(lane) + 1] = mx;
      }
    } else {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        if (tile(u) >= n_read) break;
        int64_t mn, mx, unused;
        wave_id_range(lo[u], mn, mx);
        if (nj > 1) wave_id_range(hi[u], unused, mx);
        if (lane == 0) {
          krange[2 * tile(u)] = mn;
          krange[2 * tile(u) + 1] = mx;
        }
      }
    }
  }
  __syncthreads();
  // ---- this query tile's place
  if constexpr (ORDERS) {
    {
      bool falls = false;
      for (int t = tid; t + 1 < nk; t += 1024) falls = falls || krange[2 * t + 1] > krange[2 * t + 2];
      if (__builtin_amdgcn_ballot_w64(falls) != 0 && lane == 0) few[0] = 1;
      for (int j = tid; j < n_qtiles; j += 1024) tl[j] = 0;
    }
    __syncthreads();
    const bool sorted = few[0] == 0;
    auto first_tile = [&](int j) FL_INLINE { return min(j * bm / bn, nk - 1); };  // key tiles that hold the rows of query tile j
    auto last_tile = [&](int j) FL_INLINE { return min((min((j + 1) * bm, L) - 1) / bn, nk - 1); };
    if (!sorted) {
      for (int j0 = 0; j0 < n_qtiles; j0 += 64) {
        const int j = min(j0 + lane, n_qtiles - 1), last = last_tile(j);
        int64_t mn = krange[2 * first_tile(j)], mx = krange[2 * first_tile(j) + 1];
        for (int t = first_tile(j) + 1; t <= last; ++t) {
          mn = krange[2 * t] < mn ? krange[2 * t] : mn;
          mx = krange[2 * t + 1] > mx ? krange[2 * t + 1] : mx;
        }
        uint32_t count = 0;
        for (int t = wave; t < nk; t += kWaves) count += krange[2 * t + 1] >= mn && krange[2 * t] <= mx && (!causal || t <= last);
        if (j0 + lane < n_qtiles) atomicAdd(&tl[j], count);
      }
      __syncthreads();
    }
    auto length = [&](int j) FL_INLINE -> int {
      if (!sorted) return (int)tl[j];
      // first tile whose range reaches the query tile's smallest id; last one whose range begins at or below its largest
      const int64_t mn = krange[2 * first_tile(j)], mx = krange[2 * last_tile(j) + 1];
      int lo = 0, hi = first_tile(j);
      while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (krange[2 * mid + 1] >= mn) hi = mid; else lo = mid + 1;
      }
      int last = last_tile(j);
      if (!causal) {
        int end = nk - 1;
        while (last < end) {
          const int mid = (last + end + 1) / 2;
          if (krange[2 * mid] <= mx) last = mid; else end = mid - 1;
        }
      }
      return last - lo + 1;
    };
    // (the last waves first: the first ones have the entries)
    for (int j0 = (kWaves - 1 - wave) * 64; j0 < n_qtiles; j0 += 1024) {
      const int mine = length(qt), j = j0 + lane, len = length(min(j, n_qtiles - 1));
      const uint64_t before = __builtin_amdgcn_ballot_w64(j < n_qtiles && (len > mine || (len == mine && j > qt)));
      if (lane == 0 && before != 0) atomicAdd(&few[1], (uint32_t)__builtin_popcountll(before));
    }
  }
  // ---- the list
  auto entry_of = [&](int t) FL_INLINE -> uint32_t {
    const int k0 = t * bn, k1 = min(k0 + bn, L);
    const int64_t kmn = krange[2 * t], kmx = krange[2 * t + 1];
    unsigned c = 0;
    for (int w = 0; w < nw; ++w) {
      const int a = q0 + w * rw, e = min(a + rw, L);
      const int64_t qmn = qrange[2 * w], qmx = qrange[2 * w + 1];
      int cw = TILE_EMPTY;
      if (a < e) {
        cw = kmx < qmn || kmn > qmx ? TILE_EMPTY
                                    : classify_document(mask_kind, a, e, k0, k1, kmn == kmx && qmn == qmx && kmn == qmn, k0 + bn > L);
      }
      c |= (unsigned)cw << (2 * w);
    }
    return (c << 16) | (unsigned)t;
  };
  uint32_t* out = lists + (int64_t)blockIdx.x * list_stride;
  if (ORDERS || t_end <= 1024) {  // an entry per thread
    const uint32_t e = tid < t_end ? entry_of(tid) : 0u;
    const bool keep = (e >> 16) != 0;
    const uint64_t m = __builtin_amdgcn_ballot_w64(keep);
    if (lane == 0) kept[wave] = (uint16_t)__builtin_popcountll(m);
    __syncthreads();
    if (ORDERS && tid == 0) order[(int64_t)b * n_qtiles + few[1]] = qt;
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t n = kept[w];
      before += w < wave ? n : 0;
      all += n;
    }
    if (keep) out[1 + before + __builtin_popcountll(m & ((1ull << lane) - 1))] = e;
    if (tid == 0) out[0] = all;
    return;
  }
  for (int t = tid; t < t_end; t += 1024) tl[t] = entry_of(t);
  __syncthreads();
  if (wave == 0) {
    int count = 0;
    for (int base = 0; base < t_end; base += 64) {
      const int t = base + lane;
      const uint32_t e = t < t_end ? tl[t] : 0u;
      const bool keep = (e >> 16) != 0;
      const uint64_t m = __builtin_amdgcn_ballot_w64(keep);
      const int pos = count + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
      if (keep) out[1 + pos] = e;
      count += __builtin_popcountll(m);
    }
    if (lane == 0) out[0] = (uint32_t)count;
  }
}

// Whether the lists' launch finds the order too (see above).  It has a thread per entry, and room for a count per key tile.
static bool doc_orders(int64_t B, int64_t n_qtiles, int64_t nk) { return n_qtiles >= 64 && B * n_qtiles <= 256 && nk <= 1024 && n_qtiles <= nk; }

// The same order from the lengths of the lists, a workgroup per batch row: counts for every query tile how many come before it.
static __global__ __launch_bounds__(1024) void doc_order_kernel(const uint32_t* lists, int list_stride, int n_qtiles, int32_t* order) {
  extern __shared__ uint32_t lengths[];  // n_qtiles words
  const uint32_t* of_row = lists + (int64_t)blockIdx.x * n_qtiles * list_stride;
  for (int i = threadIdx.x; i < n_qtiles; i += 1024) lengths[i] = of_row[(int64_t)i * list_stride];
  __syncthreads();
  for (int i = threadIdx.x; i < n_qtiles; i += 1024) {
    const uint32_t mine = lengths[i];
    int place = 0;
    for (int j = 0; j < n_qtiles; ++j) place += lengths[j] > mine || (lengths[j] == mine && j > i);
    order[(int64_t)blockIdx.x * n_qtiles + place] = i;
  }
}

}  // namespace fl

// Scratch of the entry point that allocates nothing (fl_attn_bwd_static): one copy per GPU the library runs on, held
// until the process ends.  In host code this name is only a handle for hipGetSymbolAddress; kernels and memory calls
// take the device address that call returns (static_scratch_ptr below).
constexpr size_t kStaticScratchBytes = (size_t)FL_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

extern "C" uint64_t fl_bwd_workspace_bytes(const fl_attn_params* p);

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

// Device address of `scratch` on the current device, looked up once per device.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};
int static_scratch_ptr(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail((int)e, "hipGetDevice failed: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(FL_ERR_UNSUPPORTED, "device ordinal %d is beyond the %d this library tracks", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) return fail((int)(e != hipSuccess ? e : hipErrorInvalidSymbol), "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

// Guard of the static scratch: one event per device, recorded behind every eager fl_attn_bwd_static call.  A call on
// another stream while that event has not completed would share the array with kernels still running: it is refused
// instead.  Calls on the stream of the previous call are ordered behind it and pass; calls under stream capture are
// neither checked nor recorded (a graph's replays are the caller's to order).
struct ScratchGuard {
  hipEvent_t done = nullptr;
  hipStream_t last = nullptr;
  bool armed = false;
};
ScratchGuard g_scratch_guard[kMaxDevices];

bool stream_is_capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return st == hipStreamCaptureStatusActive;
}

// 0 when the scratch of the current device may be used by a call on `s`.
int static_scratch_acquire(hipStream_t s, int* dev_out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(FL_ERR_UNSUPPORTED, "no current device the library tracks");
  *dev_out = dev;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  ScratchGuard& g = g_scratch_guard[dev];
  if (!g.done) {
    e = hipEventCreateWithFlags(&g.done, hipEventDisableTiming);
    if (e != hipSuccess) return fail((int)e, "hipEventCreateWithFlags failed: %s", hipGetErrorString(e));
  }
  if (g.armed && g.last != s) {
    e = hipEventQuery(g.done);
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();
      return fail(FL_ERR_WORKSPACE,
                  "fl_attn_bwd_static: the static scratch of this GPU is still in use by a call on another stream; queue "
                  "such calls on one stream, wait for the earlier one, or use fl_attn_bwd with buffers of your own");
    }
    if (e != hipSuccess) return fail((int)e, "hipEventQuery failed: %s", hipGetErrorString(e));
  }
  return 0;
}

void static_scratch_release(hipStream_t s, int dev) {
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  ScratchGuard& g = g_scratch_guard[dev];
  if (g.done && hipEventRecord(g.done, s) == hipSuccess) {
    g.last = s;
    g.armed = true;
  } else {
    (void)hipGetLastError();
  }
}

// Bounds of the element predicate every positional mask reduces to: key < Lk && ((dmin <= key - q <= dmax) || key < pfx)
void position_bounds(const fl_attn_params* p, int32_t* dmin, int32_t* dmax, int32_t* pfx) {
  const int kFar = 1 << 29;
  const bool causal_like = p->mask_kind == FL_MASK_CAUSAL || p->mask_kind == FL_MASK_SLIDING ||
                           p->mask_kind == FL_MASK_PREFIX_LM || p->mask_kind == FL_MASK_DOCUMENT_CAUSAL;
  *dmax = causal_like ? 0 : kFar;
  *dmin = p->mask_kind == FL_MASK_SLIDING ? -(p->window < kFar ? p->window : kFar) : -kFar;
  *pfx = p->mask_kind == FL_MASK_PREFIX_LM ? (p->prefix < 0 ? 0 : p->prefix) : 0;
}

bool is_doc(int kind) { return kind == FL_MASK_DOCUMENT || kind == FL_MASK_DOCUMENT_CAUSAL; }

uint32_t wanted_features(const fl_attn_params* p) {
  uint32_t f = 0;
  if (p->alibi_heads > 0) f |= fl::F_ALIBI;
  if (p->softcap > 0.f) f |= fl::F_SOFTCAP;
  if (p->score_fn != FL_SCORE_NONE) f |= fl::F_SCOREFN;
  if (p->bias[0] || p->bias[1]) f |= fl::F_BIAS;
  if (is_doc(p->mask_kind)) f |= fl::F_DOC;
  if (p->diff) f |= fl::F_DIFF;
  if (p->gate) f |= fl::F_GATE;
  if (p->attended_dump) f |= fl::F_DUMP;
  if (p->dropout_threshold) f |= fl::F_DROPOUT;
  return f;
}

// Features a kernel may be compiled with yet leave unused at run time (null pointer / zero slope).
constexpr uint32_t kOptionalFeatures = fl::F_ALIBI | fl::F_BIAS | fl::F_GATE;

// Calls of few workgroups: a workgroup of 128 rows walks its key tiles one after the other, 0.8 us each with one wave per
// SIMD, and ends when the longest walk does.  Smaller workgroups (64 rows: `waves` = 2) and groups of waves that share the rows and
// take a part of the tiles each (fwd_kernel.h) fill what idles.  Tiles of 128 rows up to one per compute unit: always; up to two under
// masks of growing length, whose longest walk is twice the average, while they belong to few heads (many short heads end together).
// us, 128 rows -> this rule, bf16: head dim 64, causal: 2 x 8 heads of 2048 29.3 -> 19.8, 8 of 4096 52.6 -> 33.6, 16 of 3000 (384 tiles)
// 40.1 -> 31.4, 4 of 4096 in four groups 52.0 -> 26.2 (in two 30.9); ALiBi and soft-cap, 16 of 2048: 41.9 -> 27.4; head dim 128, causal:
// 8 of 4096 69.5 -> 58.3, 16 of 3000 with 128 rows in two groups 58.0 -> 48.5; unmasked, 8 of 4096: 53.5 -> 43.9; documents: 8 heads of 6000,
// head dim 128, 119 -> 85.  Beyond, the second group's prologue and the adding up cost more: causal, 5 x 16 of 1184 (800 tiles) 33.9 -> 36.0,
// 8 x 16 of 512 15.9 -> 17.4, 2 x 32 of 700 under a prefix of 600 16.1 -> 18.7.
struct FewPlan {
  int waves = 0;   // preferred waves per group (0: no preference)
  int groups = 1;  // preferred groups
};
FewPlan plan_few(const fl_attn_params* p, uint32_t want) {
  FewPlan x;
  if (p->Dqk != p->Dv || (p->Dqk != 64 && p->Dqk != 128) || (want & ~(fl::F_ALIBI | fl::F_SOFTCAP | fl::F_DOC | fl::F_DUMP))) return x;
  const int64_t heads = (int64_t)p->B * p->Hq, tiles = heads * ((p->Lq + 127) / 128);
  // Walks of few tiles: the second group's prologue and the adding up cost more than the tiles it takes.  us: head dim 64, causal, 5 x 16
  // of 320 8.8 -> 9.4, 2 x 16 of 400 9.9 -> 8.4; unmasked, 4 x 8 of 512 10.7 -> 11.0, of 800 15.6 -> 14.6; documents, 6 x 16 of 64
  // 12.9 -> 13.8, of 200 18.6 -> 16.9; head dim 128, causal, 2 x 16 of 192 8.4 -> 8.7, of 256 10.6 -> 9.7; unmasked, 4 x 8 of 640 16.7 -> 17.4.
  const int64_t walk = p->mask_kind == FL_MASK_SLIDING ? std::min<int64_t>(p->Lk, (int64_t)p->window + 128) : p->Lk;
  const bool narrow = p->Dqk == 64;
  if (walk < ((want & fl::F_DOC) ? 192 : p->mask_kind == FL_MASK_NONE ? (narrow ? 640 : 1024) : narrow ? 384 : 256)) return x;
  // One head by itself keeps the order of sums it has inside a large call: slices of operands beyond 2^31 elements are compared with it bit
  // by bit.  That costs such a call (us, as is / by the lines below): unmasked, 8192 rows, head dim 128, 131 / 102; 16384 rows, 257 / 199,
  // head dim 64, 194 / 95; up to 8192 rows at head dim 64 the few-rows kernel has them.
  if (heads == 1) return x;
  if (p->mask_kind == FL_MASK_CAUSAL || p->mask_kind == FL_MASK_PREFIX_LM) {
    if (narrow ? tiles > 256 && (tiles > 512 || heads > 48) : tiles > 512 || heads > 48) return x;
    x.waves = narrow || tiles <= 256 ? 2 : 4;
    x.groups = narrow && tiles <= 128 && p->Lk >= 1024 ? 4 : 2;
  } else if (tiles <= 256) {
    x.groups = 2;
    // (walks of one length, half as many tiles as compute units: 64 rows as well, head dim 64 in four groups: 8 of 2048 24.4 -> 17.2, with
    // ALiBi and soft-cap 35.9 -> 23.7, 2 of 8192 77.5 -> 49.2; head dim 128, 8 of 2048 33.8 -> 30.8 and 43.2 -> 34.6)
    if (!(want & fl::F_DOC) && tiles <= 128 && walk >= 1024) {
      x.waves = 2;
      x.groups = narrow ? 4 : 2;
    }
  } else if (want & fl::F_DOC) {
    // (the walks are as long as the documents, which only the device knows: 1 x 16 x 4768, documents of 512 to 2384: 77 -> 55, but
    // 1 x 16 x 4096 in documents of 512 each: 23.5 -> 28.9; from 32 heads on it is even or loses whatever the documents)
    x.groups = tiles <= 1024 && heads <= 16 && p->Lk >= 4000 ? 2 : 1;
  }
  return x;
}

// Differential attention.  A group of waves per softmax branch: each holds one result, which leaves the registers room for 64-key tiles,
// both walk the same V tiles, and a call of few workgroups takes half as long.  One after the other in the same waves, the branches
// need 32-key tiles.  us, one after the other -> this rule: head dim 64, causal: 2 x 16 heads of 4096 238 -> 225, 8 of 16384 853 -> 798,
// 4 x 16 of 512 29.1 -> 17.4, 8 of 1024 47.1 -> 20.5, 4 x 8 of 2048 90.8 -> 62.1; head dim 128, 4 x 8 of 1024 114 -> 67, 2 x 16 of 4096 589 -> 554.
struct DiffPlan {
  int waves = 0;   // preferred waves per branch (0: no preference)
  int keys = 0;    // preferred keys per tile
  int groups = 1;  // 1: the branches one after the other
};
DiffPlan plan_diff(const fl_attn_params* p) {
  DiffPlan x;
  if (!p->diff || p->attended_dump) return x;
  const bool narrow = p->Dqk == 64, window = p->mask_kind == FL_MASK_SLIDING, growing = p->mask_kind == FL_MASK_CAUSAL || p->mask_kind == FL_MASK_PREFIX_LM;
  const int64_t tiles = (int64_t)p->B * p->Hq * ((p->Lq + 127) / 128);
  const int64_t visited = window ? std::min<int64_t>(p->Lk, (int64_t)p->window + 128) : p->Lk;
  x.waves = 4;
  x.keys = 32;
  // Short walks of calls that fill the compute units: one start and one store for both branches, and two workgroups of 128 rows per compute
  // unit.  us, one after the other / a group each.
  // Head dim 64 takes 64 rows with groups, which loses where the last 128 rows have none to save: unmasked, 16 x 16 of 160 14.7 / 17.2, of
  // 450 61.0 / 65.7, of 512 65.0 / 65.7, 896 tiles of 200 1 : 1.13, but 16 x 16 of 300 39.1 / 34.4, 640 tiles of 256 1 : 0.86, of 512 1 : 0.79; full
  // rounds of 600 and 850 1 : 1.02 to 1.04, of 1000 1 : 0.92 to 1.0; heads that do not divide by the 8 XCDs, whose two halves of 128 rows then read the keys on two of them, 651
  // of 200 1 : 1.19, 325 of 512 1 : 1.19, 261 of 600 1 : 1.07, 101 of 1000 1 : 0.90; masks of growing length, 1 : 0.7 to 0.95 from 200 on.
  // Head dim 128, of 200 1 : 1.06 to 1.3 under any mask, of 256 1 : 1.0 to 1.2; unmasked, of 384 1 : 1.07 to 1.16, of 600 1 : 1.04 to 1.12, of
  // 850 1 : 1.02 to 1.05, but a start into a second round of two (512 to 768 tiles) 1 : 0.85 to 1.0, into a third, of 700, 1 : 0.93; causal, of 300
  // 1 : 1.0 to 1.11, of 384 1 : 0.8 to 1.04, of 512 1 : 0.8 to 1.0; heads that do not divide by 8, of 450 1 : 0.97 to 1.15, 187 to 429 of 850
  // 1 : 1.06 to 1.15.
  // Windows, 4 x 16 of 4096, head dim 128: of 256 150 / 171, of 1100 336 / 325 (at head dim 64 with 64 rows: of 256 123 / 96, of 1500 322 / 283).
  const int64_t last = tiles % 512;  // of the last round of two per compute unit
  const bool odd = (int64_t)p->B * p->Hq % 8 != 0, full = last == 0 || last > 384, no_rows_saved = p->Lq % 128 == 0 || p->Lq % 128 > 64;
  bool sequential = false;
  if (window) sequential = !narrow && visited <= 1024;
  else if (tiles <= 256) sequential = false;
  else if (narrow && !growing)
    sequential = (full && visited <= (no_rows_saved ? 900 : 512)) ||
                 (no_rows_saved && ((visited <= 256 && last > 256) || (odd && visited <= 640 && !(visited > 512 && last > 0 && last <= 136 && tiles <= 768))));
  else if (!narrow && growing)
    sequential = visited <= 256 || (visited <= 300 && tiles > 300) || (odd && ((visited > 384 && visited <= 450) || (visited > 768 && visited <= 896 && tiles >= 1300)));
  else if (!narrow)
    sequential = visited <= 256 || (visited <= 900 && !(last > 0 && last <= 256 && (tiles <= 768 || visited > 640)));
  if (sequential) return x;
  x.groups = 2;
  // Up to 16 tiles of 128 rows keep the 128 rows and 32 keys that the dump of attended pairs is compared in at every edge, though not for
  // speed (2 heads of 256, us: the branches one after the other 18.3, a group each 13.9, with 64 rows and keys 8.5).
  if (narrow && tiles <= 16) return x;
  x.keys = 64;
  // 64 rows per workgroup, two of which share a compute unit, where 128 would leave a round far from full or the walks are short (head
  // dim 128 spills so).  us, head dim 64, 128 rows -> 64: causal, 8 heads of 1024 27.7 -> 20.5, 3 x 8 of 2048 52.0 -> 49.8, 6 x 8 of 2048 110 -> 100,
  // 8 x 32 of 300 36.4 -> 27.0, of 1024 152 -> 140; unmasked, 6 of 8192 362 -> 329; causal, 4 x 8 of 2048 62.1 -> 64.1, 2 x 16 of 4096 220 ->
  // 223, 8 of 16384 798 -> 818; unmasked, 8 of 8192 393 -> 414.
  if (narrow && (tiles <= 448 || visited < 2048 || (growing && tiles > 512 && tiles < 1024))) x.waves = 2;
  return x;
}

const fl::Instance* select_instance(const fl_attn_params* p) {
  const uint32_t want = wanted_features(p);
  const fl::Instance* best = nullptr;
  int best_extra = 1 << 30;
  // Tuning knob: FL_TILE=<rows per wave>x<keys per tile>x<waves>x<ring depth>, e.g. 32x32x4x4, restricts the choice
  // to instances of that shape (the default is the first listed instance that fits).
  // The environment is read once, when the first launch is planned.
  struct TileKnob {
    int rw = 0, bn = 0, nw = 0, ns = 0;
    TileKnob() {
      if (const char* e = std::getenv("FL_TILE")) std::sscanf(e, "%dx%dx%dx%d", &rw, &bn, &nw, &ns);
    }
  };
  static const TileKnob knob;
  const int want_rw = knob.rw, want_bn = knob.bn, want_nw = knob.nw, want_ns = knob.ns;
  // Keys one workgroup of 128 query rows visits: the window plus its own rows for a sliding window, else up to Lk.  Where they are few,
  // workgroups of 64 rows: less of each tile lies outside the mask, and more independent workgroups overlap their first loads.
  // Head dim 64, us, 128 rows -> 64: window, 4 x 16 heads of 4096: 64 keys 38.6 -> 34.2, 256 50.7 -> 45.0, 700 78.2 -> 75.5, 1200 105.6 ->
  // 107.2; causal, 20 x 32 of 138 19.3 -> 15.2, 30 x 16 of 700 69.7 -> 62.5, 16 x 16 of 1000 61.6 -> 60.0, 4 x 32 of 1500 even; a prefix
  // of 200 in 700 48.9 -> 44.5, of 600 57.8 -> 60.3; two key tiles at most (16 x 16 of 128 under a window of 64): 7.3 -> 8.1,
  // and whole short walks while 128-row workgroups all run at once: causal, 15 x 8 of 151 7.2 -> 8.0, 6 x 16 of 300 9.3 -> 10.1, of 370 even.
  // Head dim 128, whose tile then has 32 keys: from a window of 256 on the 4-wave tile ties or wins on warm operands and wins by 4 % on
  // cold ones; ALiBi and soft-cap under a window of 100, 4 x 32 of 2000: 69.0 -> 59.0.
  const int64_t visited = p->mask_kind == FL_MASK_SLIDING ? std::min<int64_t>(p->Lk, (int64_t)p->window + 128) : p->Lk;
  const bool thin = p->mask_kind == FL_MASK_SLIDING ||
                    (p->Dqk == 64 && (p->mask_kind == FL_MASK_CAUSAL || (p->mask_kind == FL_MASK_PREFIX_LM && p->prefix <= p->Lk / 2)));
  const bool many = (int64_t)p->B * p->Hq * ((p->Lq + 127) / 128) > 512;
  const bool short_loop = thin && (p->Dqk == 64 ? visited >= (many || visited < p->Lk ? 129 : 384) && visited < 1024 : visited < 384);
  // Unmasked calls at head dim 128 whose grid still fills the part twice over with 256-row workgroups take the
  // 8-wave tile: one workgroup per compute unit brings every K/V tile in once for 256 rows instead of twice, which on
  // ordinary data is worth more than the second workgroup's independence (2.4 % on N(0,1) operands; at head dim 64,
  // under masks and on all-zero operands it is not).
  const bool wide_group = p->mask_kind == FL_MASK_NONE && want == 0 && p->Dqk == 128 && p->Dv == 128 &&
                          (int64_t)p->B * p->Hq * ((p->Lq + 255) / 256) >= 512;
  const FewPlan few = plan_few(p, want);
  const DiffPlan diff = plan_diff(p);
  const int preferred_nw = diff.waves ? diff.waves : few.waves ? few.waves : short_loop ? 2 : (wide_group ? 8 : 4);
  for (int i = 0; i < fl::kNumInstances; ++i) {
    const fl::Instance& in = fl::kInstances[i];
    if (in.dqk != p->Dqk || in.dv != p->Dv || in.dtype != p->dtype) continue;
    if ((in.feat & want) != want) continue;
    const uint32_t extra = in.feat & ~want;
    if (extra & ~kOptionalFeatures) continue;
    if (want_rw && (in.rw != want_rw || in.bn != want_bn || in.nw != want_nw || (want_ns && in.ns != want_ns))) continue;
    // fewer unused features first; among equals the preferred workgroup size, the preferred tile, then the listed order
    const int n = 4 * __builtin_popcount(extra) + (in.nw == preferred_nw ? 0 : 2) + (!diff.keys || in.bn == diff.keys ? 0 : 1);
    if (n < best_extra) {
      best = &in;
      best_extra = n;
    }
  }
  return best;
}

// Device scratch of a document-mask call, in this order (every part a multiple of 16 bytes):
//   table   [B][ceil(L / 32)][2] int64   (min, max) id per 32 positions (backward)
//   lists   [B][query tiles][stride] u32 the key tiles each query tile visits (forward; bm / bn = query rows per
//                                        workgroup and keys per tile of the forward instance)
//   order   [B][query tiles] i32          the query tiles by falling list length (forward), rounded up to 16 bytes
struct DocScratch {
  int64_t blocks, n_qtiles, nk, list_stride;
  uint64_t table_bytes, lists_bytes, order_bytes;
};
DocScratch doc_scratch(int64_t B, int64_t L, int64_t bm, int64_t bn) {
  DocScratch d;
  d.blocks = (L + fl::kDocBlock - 1) / fl::kDocBlock;
  d.n_qtiles = (L + bm - 1) / bm;
  d.nk = (L + bn - 1) / bn;
  d.list_stride = (d.nk + 1 + 3) / 4 * 4;
  d.table_bytes = (uint64_t)B * d.blocks * 2 * sizeof(int64_t);
  d.lists_bytes = (uint64_t)B * d.n_qtiles * d.list_stride * sizeof(uint32_t);
  d.order_bytes = ((uint64_t)B * d.n_qtiles * sizeof(int32_t) + 15) / 16 * 16;
  return d;
}

// LDS bytes of a launch: the instance's fixed part plus, under a document mask, the tile list in whole 1 KiB wave
// transfers.
int64_t lds_bytes_for(const fl::Instance* in, const fl_attn_params* p) {
  if (!(in->feat & fl::F_DOC)) return in->lds_fixed_bytes;
  const DocScratch d = doc_scratch(p->B, p->Lk, (int64_t)in->rw * in->nw, in->bn);
  return in->lds_fixed_bytes + (d.list_stride * 4 + 1023) / 1024 * 1024;
}
// Dynamic LDS bytes of the document-mask pre-pass (doc_lists_kernel): 20 per key tile; it has up to 128 static bytes besides
int64_t prepass_lds_bytes(int64_t n_ktiles) { return n_ktiles * 20; }
// Groups of waves a call is launched with, and the LDS of all of them
int groups_for(const fl::Instance* in, const fl_attn_params* p) {
  // (a tile that has no form with the branches one after the other takes a group for each, whatever the plan prefers: FL_TILE may force it)
  if (p->diff) return fl::diff_sequential(in->bn, in->nw) ? std::min(plan_diff(p).groups, in->max_groups) : in->max_groups;
  const int groups = std::min(plan_few(p, wanted_features(p)).groups, in->max_groups);
  return lds_bytes_for(in, p) + (int64_t)(groups - 1) * in->lds_fixed_bytes <= fl::kMaxLdsBytes ? groups : 1;
}
// Whether a call with a soft-cap runs the kernel that takes NearCap's polynomial where the scores allow.  That kernel saves up to 15 % where they
// stay within five sixths of a quarter of the cap, costs 0 to 1 % (at most 3: 2 x 16 x 2048 with ALiBi at head dim 64, 4 x 16 x 2048 at 32) where they do not, and half a microsecond, whatever the call, where they
// leave that range on the way: a second loop to be fetched, and a tile's scores formed twice where they jump past the range itself.  Short calls
// therefore keep the exponential.  us, exponential -> polynomial, scores N(0,1) and a quarter of the cap at 9 / 4 / 2 of them.  Below the line: 4 x 16 x 300,
// head dim 64, causal, 8.6 -> 8.2 / 9.2 / 8.6; 2 x 8 x 700 14.2 -> 13.1 / 15.0 / 14.3; 8 x 8 x 512 12.3 -> 11.6 / 13.0 / 12.4; head dim 32, 3 x 16 x 600, ALiBi,
// 14.4 -> 12.7 / 15.3 / 14.7; 2 x 32 x 512, head dim 128, 16.8 -> 16.1 / 17.7 / 17.1.  Above: 8 x 2048, head dim 64, ALiBi, causal, 22.2 -> 20.2 / 22.7 / 22.5; 8 x 16 x 512
// 20.2 -> 18.3 / 20.4 / 20.3; 4 x 16 x 700, head dim 128, 26.4 -> 24.5 / 26.7 / 26.8; 4 x 16 x 1024 42.9 -> 38.5 / 43.3 / 43.3; under a window of 256, 4 x 16 x 4096,
// head dim 64, 55.2 -> 51.4 / 55.9 / 55.9; 4 x 16 over 4 x 2048, causal, 75.1 -> 63.6 / 75.5 / 74.8.
bool near_cap_pays(const fl_attn_params* p, const fl::Instance* in, int groups, int64_t grid) {
  if (!fl::has_near(in->feat)) return false;
  // keys of a wave's longest walk, times the waves (of which two per SIMD run at once, and one alone takes as long as half a pair)
  const int64_t walk = p->mask_kind == FL_MASK_SLIDING ? std::min<int64_t>(p->Lk, (int64_t)p->window + in->rw * in->nw) : p->Lk;
  return walk / groups * std::max<int64_t>(1024, grid * in->nw * groups) >= (int64_t)1024 * 1024;
}
int64_t max_keys_for(const fl::Instance* in) {
  int64_t tiles = fl::kMaxKeyTiles;
  if (in->feat & fl::F_DOC) {
    tiles = std::min<int64_t>(tiles, (fl::kMaxLdsBytes - in->lds_fixed_bytes) / 1024 * 256 - 4);
    tiles = std::min<int64_t>(tiles, (fl::kMaxLdsBytes - 128) / 20);  // the pre-pass: 20 bytes of LDS per key tile
  }
  return tiles * in->bn;
}

int check_strides(const char* what, const int64_t* s, int align) {
  if (s[3] != 1) return fail(FL_ERR_STRIDE, "%s: the last (dim) stride must be 1, got %lld", what, (long long)s[3]);
  for (int i = 0; i < 3; ++i) {
    if (s[i] < 0) return fail(FL_ERR_STRIDE, "%s: negative stride %lld", what, (long long)s[i]);
    if (s[i] % align != 0)
      return fail(FL_ERR_ALIGN, "%s: stride[%d]=%lld must be a multiple of %d elements", what, i, (long long)s[i], align);
  }
  return 0;
}

int check_ptr(const char* what, const void* ptr, int align) {
  if (!ptr) return fail(FL_ERR_NULL, "%s pointer is null", what);
  if (reinterpret_cast<uintptr_t>(ptr) % align != 0)
    return fail(FL_ERR_ALIGN, "%s pointer must be %d-byte aligned", what, align);
  return 0;
}

int validate(const fl_attn_params* p, const fl::Instance** out, bool for_bwd = false, uint32_t flags = FL_FLAG_DOC_PREPARED | FL_FLAG_SCRATCH | FL_FLAG_F32_RESULT) {
  if (!p) return fail(FL_ERR_NULL, "params is null");
  int rc;
  if ((rc = check_ptr("q", p->q, 16)) || (rc = check_ptr("k", p->k, 16)) || (rc = check_ptr("v", p->v, 16)) ||
      (rc = check_ptr("o", p->o, 8)))
    return rc;
  if (p->dtype != FL_BF16 && p->dtype != FL_F16)
    return fail(FL_ERR_UNSUPPORTED, "dtype %d is not supported (FL_BF16 or FL_F16)", p->dtype);
  if (p->B <= 0 || p->Hq <= 0 || p->Hkv <= 0 || p->Lq <= 0 || p->Lk <= 0 || p->Dqk <= 0 || p->Dv <= 0)
    return fail(FL_ERR_SHAPE, "sizes must be positive: B=%d Hq=%d Hkv=%d Lq=%d Lk=%d Dqk=%d Dv=%d", p->B, p->Hq, p->Hkv,
                p->Lq, p->Lk, p->Dqk, p->Dv);
  if (p->Hq % p->Hkv != 0)
    return fail(FL_ERR_SHAPE, "query heads (%d) must be a multiple of key/value heads (%d)", p->Hq, p->Hkv);
  if ((int64_t)p->B * p->Hq > (int64_t)1 << 30) return fail(FL_ERR_SHAPE, "B*Hq too large");
  if (!(p->scale > 0.f) || !std::isfinite(p->scale)) return fail(FL_ERR_ARG, "scale must be finite and > 0, got %g", p->scale);
  if ((rc = check_strides("q", p->q_strides, 8)) || (rc = check_strides("k", p->k_strides, 8)) ||
      (rc = check_strides("v", p->v_strides, 8)) || (rc = check_strides("o", p->o_strides, 4)))
    return rc;
  if (p->flags & ~flags) return fail(FL_ERR_ARG, "unknown bits in flags: 0x%x", p->flags);
  if (p->flags & FL_FLAG_F32_RESULT) {
    if (for_bwd || p->gate || p->diff) return fail(FL_ERR_UNSUPPORTED, "a result in fp32 goes with forward calls without gate and differential attention");
    if (reinterpret_cast<uintptr_t>(p->o) % 16) return fail(FL_ERR_ALIGN, "o pointer must be 16-byte aligned");
  }
  if ((p->flags & FL_FLAG_DOC_PREPARED) && !is_doc(p->mask_kind))
    return fail(FL_ERR_ARG, "FL_FLAG_DOC_PREPARED goes with a document mask only");
  if (p->dropout_threshold) {
    if (p->dropout_threshold > 65535u)
      return fail(FL_ERR_ARG, "dropout_threshold must be at most 65535 (rate 65535/65536), got %u", p->dropout_threshold);
    if (p->diff || p->attended_dump)
      return fail(FL_ERR_UNSUPPORTED, "dropout is not built for differential attention and the dump hook");
  }
  if (p->lse) {
    if (reinterpret_cast<uintptr_t>(p->lse) % 4) return fail(FL_ERR_ALIGN, "lse must be 4-byte aligned");
    if (p->diff) return fail(FL_ERR_UNSUPPORTED, "lse is not produced for differential attention");
  }

  switch (p->mask_kind) {
    case FL_MASK_NONE:
    case FL_MASK_CAUSAL: break;
    case FL_MASK_SLIDING:
      if (p->window < 0) return fail(FL_ERR_ARG, "window must be >= 0, got %d", p->window);
      if (p->Lq != p->Lk) return fail(FL_ERR_SHAPE, "sliding window needs Lq == Lk (got %d, %d)", p->Lq, p->Lk);
      break;
    case FL_MASK_PREFIX_LM:
      if (p->Lq != p->Lk) return fail(FL_ERR_SHAPE, "prefix-LM needs Lq == Lk (got %d, %d)", p->Lq, p->Lk);
      break;
    case FL_MASK_DOCUMENT:
    case FL_MASK_DOCUMENT_CAUSAL:
      if (!p->doc_ids) return fail(FL_ERR_NULL, "doc_ids pointer is null");
      if (reinterpret_cast<uintptr_t>(p->doc_ids) % 8) return fail(FL_ERR_ALIGN, "doc_ids must be 8-byte aligned");
      if (p->Lq != p->Lk) return fail(FL_ERR_SHAPE, "document mask needs Lq == Lk (got %d, %d)", p->Lq, p->Lk);
      if (p->doc_stride < 0) return fail(FL_ERR_STRIDE, "doc_stride must be >= 0");
      break;
    default: return fail(FL_ERR_ARG, "unknown mask_kind %d", p->mask_kind);
  }
  if (p->alibi_heads < 0) return fail(FL_ERR_ARG, "alibi_heads must be >= 0");
  if (!(p->softcap >= 0.f) || !std::isfinite(p->softcap)) return fail(FL_ERR_ARG, "softcap must be finite and >= 0");
  if (p->score_fn != FL_SCORE_NONE) {
    if (p->score_fn < FL_SCORE_SIGMOID || p->score_fn > FL_SCORE_POLY) return fail(FL_ERR_ARG, "unknown score_fn %d", p->score_fn);
    const float* c = p->score_fn_params;
    // clamp bounds may be infinite (a one-sided clamp); every other constant is an ordinary number
    const int n_finite = p->score_fn == FL_SCORE_CLAMP ? 2 : 4;
    for (int i = 0; i < n_finite; ++i)
      if (!std::isfinite(c[i])) return fail(FL_ERR_ARG, "score_fn_params[%d] must be finite", i);
    if (p->score_fn == FL_SCORE_CLAMP && !(c[2] <= c[3])) return fail(FL_ERR_ARG, "score_fn clamp: lower bound above upper bound");
    if (p->softcap > 0.f || p->alibi_heads > 0 || is_doc(p->mask_kind) || p->gate || p->diff || p->dropout_threshold)
      return fail(FL_ERR_UNSUPPORTED, "score_fn goes with positional masks and bias operands only (no soft-cap, ALiBi, "
                                      "document mask, gate, differential attention or dropout)");
  }
  for (int nb = 0; nb < 2; ++nb) {
    if (!p->bias[nb]) continue;
    if (p->bias_dtype[nb] != p->dtype && p->bias_dtype[nb] != FL_F32)
      return fail(FL_ERR_UNSUPPORTED, "bias_dtype[%d]=%d is not supported (fp32, or the element type of q)", nb, p->bias_dtype[nb]);
    const int esz = p->bias_dtype[nb] == FL_F32 ? 4 : 2;
    if (reinterpret_cast<uintptr_t>(p->bias[nb]) % esz)
      return fail(FL_ERR_ALIGN, "bias[%d] must be %d-byte aligned", nb, esz);
    if (p->bias_batch_div[nb] <= 0) return fail(FL_ERR_ARG, "bias_batch_div[%d] must be >= 1", nb);
    for (int i = 0; i < 4; ++i)
      if (p->bias_strides[nb][i] < 0) return fail(FL_ERR_STRIDE, "bias[%d]: negative stride", nb);
    if (p->bias_strides[nb][3] > 1) return fail(FL_ERR_STRIDE, "bias[%d]: the key stride must be 0 or 1", nb);
  }
  if (p->gate) {
    if ((rc = check_ptr("gate", p->gate, 8)) || (rc = check_strides("gate", p->gate_strides, 4))) return rc;
  }
  if (p->diff) {
    if (!std::isfinite(p->lambda)) return fail(FL_ERR_ARG, "lambda must be finite");
  }
  const fl::Instance* in = select_instance(p);
  if (!in)
    return fail(FL_ERR_UNSUPPORTED,
                "no kernel instance for Dqk=%d Dv=%d features=0x%x (alibi=1 softcap=2 bias=4 doc=8 diff=16 gate=32 dump=64 "
                "dropout=128 score_fn=256)",
                p->Dqk, p->Dv, wanted_features(p));
  const int64_t nkt = ((int64_t)p->Lk + in->bn - 1) / in->bn;
  if (nkt > fl::kMaxKeyTiles || lds_bytes_for(in, p) > fl::kMaxLdsBytes)
    return fail(FL_ERR_SHAPE, "Lk=%d exceeds the supported maximum of %lld keys for this kernel", p->Lk,
                (long long)max_keys_for(in));
  // per-lane byte offsets inside one key tile are 32-bit
  if (((int64_t)in->bn * p->k_strides[2] + p->Dqk) * 2 >= ((int64_t)1 << 31) ||
      ((int64_t)in->bn * p->v_strides[2] + p->Dv) * 2 >= ((int64_t)1 << 31))
    return fail(FL_ERR_STRIDE, "key/value sequence stride too large (%lld, %lld elements)", (long long)p->k_strides[2],
                (long long)p->v_strides[2]);
  const int64_t bm = (int64_t)in->rw * in->nw;
  const int64_t grid = (int64_t)p->B * p->Hq * (((int64_t)p->Lq + bm - 1) / bm);
  if (grid > 0x7fffffff) return fail(FL_ERR_SHAPE, "too many workgroups (%lld)", (long long)grid);
  if (is_doc(p->mask_kind)) {
    // the forward's pre-pass keeps 20 bytes per key tile (and 128 more) in LDS
    if (!for_bwd && prepass_lds_bytes(nkt) + 128 > fl::kMaxLdsBytes)
      return fail(FL_ERR_SHAPE, "Lk=%d exceeds the supported maximum of %lld keys for a document mask with this kernel", p->Lk,
                  (long long)max_keys_for(in));
    // (a backward call needs the table of id ranges only, not the forward's lists)
    const uint64_t need = for_bwd ? fl_bwd_workspace_bytes(p) : fl_workspace_bytes(p);
    if (!p->workspace || p->workspace_bytes < need)
      return fail(FL_ERR_WORKSPACE, "document mask needs a %llu-byte workspace (got %llu)", (unsigned long long)need,
                  (unsigned long long)(p->workspace ? p->workspace_bytes : 0));
    if (reinterpret_cast<uintptr_t>(p->workspace) % 16) return fail(FL_ERR_ALIGN, "workspace must be 16-byte aligned");
  }
  if (out) *out = in;
  g_err[0] = 0;
  return 0;
}

// Whether *p (already validated) is a call the shared-bias streaming forward covers: head dim 32, no mask or other
// score modification, one dense 16-bit bias operand that several consecutive batch entries share (and optionally one
// row of keys per batch entry), a key count the kernel is compiled for (pairbias_has_shape).  Fills the kernel's
// parameters and launch shape.
bool plan_pairbias(const fl_attn_params* p, fl::PParams* out, int* grid) {
  static const bool disabled = std::getenv("FL_NO_PAIRBIAS") != nullptr;  // A/B knob: the general kernel instead
  if (disabled) return false;
  if (p->Dqk != p->Dv || p->mask_kind != FL_MASK_NONE || p->alibi_heads > 0 || p->softcap > 0.f ||
      p->diff || p->attended_dump || p->dropout_threshold || p->lse || p->score_fn != FL_SCORE_NONE || (p->flags & FL_FLAG_F32_RESULT))
    return false;
  // one operand that several consecutive batch entries share (dense over heads, queries and keys), and optionally one
  // that is a row of keys per batch entry, the same for every head and query; in either order
  int pi = -1, ri = -1;
  for (int i = 0; i < 2; ++i) {
    if (!p->bias[i]) continue;
    const int64_t* st = p->bias_strides[i];
    if (p->bias_dtype[i] != p->dtype || st[3] != 1) return false;
    if (p->bias_batch_div[i] >= 2 && (st[1] != 0 || p->Hq == 1) && st[2] != 0 && pi < 0) pi = i;  // (one head: no head stride)
    else if (p->bias_batch_div[i] == 1 && st[1] == 0 && st[2] == 0 && ri < 0) ri = i;
    else return false;
  }
  if (pi < 0) return false;
  const int64_t* bst = p->bias_strides[pi];
  const int div = p->bias_batch_div[pi];
  if (p->B % div != 0) return false;
  if (p->Lk % 32 != 0 || !fl::pairbias_has_shape(p->Dqk, p->Lk / 32, p->gate != nullptr, ri >= 0)) return false;
  if (reinterpret_cast<uintptr_t>(p->bias[pi]) % 16 != 0 || bst[0] % 8 || bst[1] % 8 || bst[2] % 8) return false;
  if (ri >= 0 && (reinterpret_cast<uintptr_t>(p->bias[ri]) % 16 != 0 || p->bias_strides[ri][0] % 8)) return false;
  // (results leave in 16-byte stores, gate logits arrive in 16-byte loads)
  if (reinterpret_cast<uintptr_t>(p->o) % 16 != 0 || p->o_strides[0] % 8 || p->o_strides[1] % 8 || p->o_strides[2] % 8) return false;
  if (p->gate && (reinterpret_cast<uintptr_t>(p->gate) % 16 != 0 || p->gate_strides[0] % 8 || p->gate_strides[1] % 8 ||
                  p->gate_strides[2] % 8))
    return false;
  // per-lane byte offsets inside one (batch entry, head) slice are 32-bit
  const int64_t worst = std::max(std::max(p->q_strides[2], p->o_strides[2]), p->gate ? p->gate_strides[2] : 0);
  if (((int64_t)p->Lq * worst + 64) * 2 >= ((int64_t)1 << 31)) return false;
  // ... and so are those inside one key tile of 64 rows
  if ((64 * std::max(p->k_strides[2], p->v_strides[2]) + p->Dqk) * 2 >= ((int64_t)1 << 31)) return false;
  // the selector weight 1 / scale must be an ordinary number in the element type (bf16 shares fp32's range; fp16 ends at
  // 65504 and loses precision below 2^-14)
  {
    const float w = 1.0f / p->scale;
    const float w_max = p->dtype == FL_F16 ? 32768.0f : 0x1p100f, w_min = p->dtype == FL_F16 ? 0x1p-10f : 0x1p-100f;
    if (!(w <= w_max) || !(w >= w_min)) return false;
  }
  fl::PParams k;
  std::memset(&k, 0, sizeof(k));
  k.q = static_cast<const fl::bf16_t*>(p->q);
  k.k = static_cast<const fl::bf16_t*>(p->k);
  k.v = static_cast<const fl::bf16_t*>(p->v);
  k.o = static_cast<fl::bf16_t*>(p->o);
  for (int i = 0; i < 3; ++i) {
    k.qs[i] = p->q_strides[i];
    k.ks[i] = p->k_strides[i];
    k.vs[i] = p->v_strides[i];
    k.os[i] = p->o_strides[i];
    k.gs[i] = p->gate_strides[i];
    k.bs[i] = bst[i];
  }
  k.B = p->B;
  k.H = p->Hq;
  if (p->Hq != p->Hkv) return false;
  k.Lq = p->Lq;
  k.Lk = p->Lk;
  k.scale = p->scale;
  k.bias = static_cast<const fl::bf16_t*>(p->bias[pi]);
  k.bdiv = div;
  if (ri >= 0) {
    k.rowb = static_cast<const fl::bf16_t*>(p->bias[ri]);
    k.rbs = p->bias_strides[ri][0];
  }
  k.gate = static_cast<const fl::bf16_t*>(p->gate);
  k.n_qtiles = (p->Lq + 127) / 128;
  // Launch shape: every workgroup should be resident at once (two per compute unit, 32 compute units per XCD), and a
  // unit = (chunk of batch entries, pair of heads) with all its query tiles stays on one XCD.  The batch entries of a
  // bias group are cut into as many chunks as that allows; more chunks than entries make no sense, fewer than one
  // means several rounds of workgroups.
  const int64_t groups = p->B / div;
  k.hgroup = p->Hq % 2 == 0 ? 2 : 1;
  const int64_t per_unit = (int64_t)k.hgroup * k.n_qtiles;
  const int64_t units_per_xcd = std::max<int64_t>(1, 64 / per_unit);
  const int64_t head_groups = p->Hq / k.hgroup;
  int64_t chunks = (8 * units_per_xcd) / (groups * head_groups);
  chunks = std::max<int64_t>(1, std::min<int64_t>(chunks, div));
  k.chunk_len = (int)((div + chunks - 1) / chunks);
  k.chunks = (div + k.chunk_len - 1) / k.chunk_len;
  const int64_t n_units = groups * k.chunks * head_groups;
  const int64_t g = (n_units + 7) / 8 * 8 * per_unit;
  if (n_units > 0x7fffffff || g > 0x7fffffff) return false;
  k.n_units = (int)n_units;
  *grid = (int)g;
  *out = k;
  return true;
}

// Whether bias operand `nb` can travel through LDS with the general forward's K/V tiles: rows addressable in 16-byte pieces, and
// per-lane byte offsets inside one (batch, head) slice in 32 bits.
bool bias_stageable(const fl_attn_params* p, int nb) {
  const int64_t* st = p->bias_strides[nb];
  return p->bias[nb] && st[3] == 1 && reinterpret_cast<uintptr_t>(p->bias[nb]) % 16 == 0 && p->Lk % 8 == 0 && st[0] % 8 == 0 &&
         st[1] % 8 == 0 && st[2] % 8 == 0 && ((int64_t)p->Lq * st[2] + p->Lk) * 4 < ((int64_t)1 << 31);
}

// Into how many chunks the `div` batch entries that share a bias are cut.  A chunk of one head and one group of entries is `tiles`
// workgroups, which stay on one of the 8 XCDs; `per_cu` of them run at once on each of its 32 compute units.  Taken is the number with
// the fewest rounds times what a round takes: the entries of a chunk, and a start worth two and a half of them.  (Gradients, both
// roles, us: 128 x 8 x 256 x 256, head dim 32: 4 chunks in one round 83, 8 in two 92; 65 x 4 x 384 x 384, 64: 2 chunks in one round
// 125, 5 in three 156, 10 in four 125; 256 x 8 x 384 x 384, 32: 1 chunk 707, 2 chunks 670, 5 chunks 550.)
int64_t chunks_of_entries(int64_t heads_and_groups, int64_t tiles, int per_cu, int64_t div) {
  int64_t best = 1;
  double least = 0;
  for (int64_t c = 1; c <= div && (c == 1 || c * heads_and_groups * tiles <= 4 * 256 * per_cu); ++c) {
    const int64_t rounds = ((heads_and_groups * c + 7) / 8 * tiles + 32 * per_cu - 1) / (32 * per_cu);
    const double t = (double)rounds * ((double)((div + c - 1) / c) + 2.5);
    if (c == 1 || t < least) {
      least = t;
      best = c;
    }
  }
  return best;
}

// Whether a bias row may be what the accumulators of a product start from (the shared-bias stripe forward and gradients): times 1 / scale it
// has to stay an ordinary number.  (A scale that has not been set yet is no reason against it.)
bool row_starts_products(const fl_attn_params* p) { return !(p->scale > 0.f) || (p->scale >= 0x1p-100f && p->scale <= 0x1p100f); }

// Whether neighbours among the (chunk of entries, head) pairs share an XCD in the shared-bias kernels that walk over entries (StripePlace), and are not
// dealt round the XCDs.  With operands as the Evoformer has them a head's row is half of a cache line at head dim 32, and dealt round every line comes into
// two L2s (forward and gradients, 128 x 8 x 256 x 256: 134 MB read by each, 67 by neighbours: four pairs to an XCD there, half of a chunk's heads).  What
// it costs is a bias read by more XCDs.  us, dealt round -> neighbours.
// Forward, from chunks of 5 entries on: 400 x 4 x 100 (chunks of 5) 23.7 -> 23.3; 50 x 4 x 333, head dim 64 (5), 41.5 -> 40.7; 150 x 8 x 250 (10) 44.4 ->
// 44.0; 512 x 8 x 160 105.6 -> 102.6; 150 x 8 x 333, head dim 64, 288 -> 244; even: 96 x 8 x 256 (6).  Chunks of 4: 64 x 8 x 256 20.5 -> 20.8.  Nor from 320 keys on at head
// dim 32: 256 x 8 x 384, 100 x 8 x 400, 64 x 8 x 512 even, 96 x 8 x 450 113.0 -> 114.5, with a bias row 135.3 -> 137.4.
bool forward_neighbours(const fl::StripeParams& k, int d) { return k.chunk_len >= 5 && (d != 32 || k.Lk <= 320); }
// Gradients, where q, k, v and dout are more than 24 MB: 96 x 7 x 160 (28 MB) 49.9 -> 48.1; 40 x 8 x 384 (31) 101 -> 91.7; 80 x 8 x 200 (33) 60.0 -> 58.0; 400 x 4 x
// 100 (41) 52.2 -> 49.0; 72 x 8 x 190, head dim 64 (56), 94.8 -> 87.3; 128 x 8 x 256 (67) 101.4 -> 99.3; 256 x 8 x 130 (68) 108 -> 102; but 64 x 8 x 256 (34) 56.8 -> 57.7.
// Below it the L2s hold both copies: 20 x 8 x 300 (12) 42.6 -> 43.3, 32 x 8 x 256 (17) 32.1 -> 33.9, 128 x 4 x 128 (17) 22.4 -> 22.8, 100 x 8 x 100 (20) 28.8 -> 29.3.
int64_t streamed_bytes(const fl_attn_params* p) { return (int64_t)p->B * p->Hq * p->Lq * p->Dqk * 8; }
bool gradient_neighbours(const fl_attn_params* p) { return streamed_bytes(p) > (int64_t)24 << 20; }
// Whether the gradients touch rows two entries ahead (pairbias_bwd_kernel.h): operands that stay in the 256 MB of cache behind the L2s from the kernels
// before arrive soon enough without (67 MB, 128 x 4 x 256 x 256 of head dim 64, 128 -> 130 us), and up to four stripes of a head have few rows to share out (400 x 8
// x 128 100.2 -> 102.4, 1000 x 8 x 64 109 -> 115).  256 x 8 x 256 181 -> 164, 512 x 8 x 160 208 -> 195, 96 x 8 x 450 301 -> 241, 128 x 8 x 320 202 -> 202; head dim 64,
// 64 x 8 x 512 376 -> 265, 100 x 8 x 256 156 -> 147.
bool gradient_ahead(const fl_attn_params* p) { return streamed_bytes(p) > (int64_t)80 << 20 && p->Lk > 128; }

// Whether *p (already validated) is a call the shared-bias stripe forward (stripe_kernel.h) takes.  Fills the kernel's parameters,
// its wave count, and the number of workgroups and their LDS bytes.
bool plan_stripe(const fl_attn_params* p, void* ungated, fl::StripeParams* out, int* waves, int64_t (&launch)[2]) {
  if (p->Dqk != p->Dv || (p->Dqk != 32 && p->Dqk != 64) || p->Hq != p->Hkv || p->Lq > 512 || p->Lk > 512 || p->Lk < 4 ||
      p->mask_kind != FL_MASK_NONE || p->alibi_heads > 0 || p->softcap > 0.f || p->diff || p->attended_dump || p->dropout_threshold ||
      p->score_fn != FL_SCORE_NONE || (p->flags & FL_FLAG_F32_RESULT))
    return false;
  // one operand that several consecutive batch entries share, dense over heads and queries, and optionally one that is a row of keys
  // per batch entry, the same for every head and query; in either order
  int pi = -1, ri = -1;
  for (int i = 0; i < 2; ++i) {
    if (!p->bias[i]) continue;
    const int64_t* st = p->bias_strides[i];
    if (p->bias_batch_div[i] >= 2 && (st[1] != 0 || p->Hq == 1) && (st[2] != 0 || p->Lq == 1) && (st[3] == 1 || p->Lk == 1) && pi < 0) pi = i;
    else if (st[1] == 0 && st[2] == 0 && st[3] <= 0x7fffffff && ri < 0) ri = i;
    else return false;
  }
  if (pi < 0 || (ri >= 0 && !row_starts_products(p))) return false;
  if (p->B % p->bias_batch_div[pi] != 0) return false;  // (workgroups walk whole groups of entries; the general kernel divides per entry)
  // Where the general kernel has to read the bias two bytes at a time (odd lengths, fp32), this one is three to five times sooner
  // (bf16, us: 414 x 4 x 494 x 494, head dim 32: 806 -> 201; 34 x 4 x 235 x 235, head dim 64: 43 -> 17; 28 x 4 x 106 x 106: 14 -> 6).  Where
  // that kernel can stage the bias beside its tiles, this one is ahead at head dim 32 with three or four waves, which fill the
  // compute unit twice over (128 x 8 x 160 / 192 / 256 keys: 39.8 -> 34.7, 38.2 -> 34.4, 44 -> 37) and behind at other lengths (128
  // keys: 18.6 against 21.4; 320: 73 against 87; 512 a tie) and at head dim 64 (256 keys: 60 against 99: one block of queries per
  // workgroup).
  if (p->bias_dtype[pi] != FL_F32 && bias_stageable(p, pi) && !(p->Dqk == 32 && p->Lk > 128 && p->Lk <= 256)) return false;
  // per-lane byte offsets inside one (batch entry, head) are 32-bit; results leave and gate logits arrive 16 bytes at a time
  for (const int64_t* st : {p->q_strides, p->k_strides, p->v_strides, p->o_strides})
    if (st[2] >= (1 << 20)) return false;
  if (reinterpret_cast<uintptr_t>(p->o) % 16 || p->o_strides[0] % 8 || p->o_strides[1] % 8 || p->o_strides[2] % 8) return false;
  if (p->gate && (reinterpret_cast<uintptr_t>(p->gate) % 16 || p->gate_strides[0] % 8 || p->gate_strides[1] % 8 || p->gate_strides[2] % 8))
    return false;
  fl::StripeParams k;
  std::memset(&k, 0, sizeof(k));
  k.q = static_cast<const fl::bf16_t*>(p->q);
  k.k = static_cast<const fl::bf16_t*>(p->k);
  k.v = static_cast<const fl::bf16_t*>(p->v);
  k.o = static_cast<fl::bf16_t*>(p->o);
  for (int i = 0; i < 3; ++i) {
    k.qs[i] = p->q_strides[i];
    k.ks[i] = p->k_strides[i];
    k.vs[i] = p->v_strides[i];
    k.os[i] = p->o_strides[i];
    k.gs[i] = p->gate_strides[i];
    k.bs[i] = p->bias_strides[pi][i];
  }
  k.bias = p->bias[pi];
  k.bias_f32 = p->bias_dtype[pi] == FL_F32;
  k.row_div = 1;
  if (ri >= 0) {
    k.row = p->bias[ri];
    k.row_batch = p->bias_strides[ri][0];
    k.row_key = (int)p->bias_strides[ri][3];
    k.row_div = p->bias_batch_div[ri];
    k.row_f32 = p->bias_dtype[ri] == FL_F32;
  }
  k.gate = static_cast<const fl::bf16_t*>(p->gate);
  k.ungated = static_cast<fl::bf16_t*>(ungated);
  k.lse = p->lse;
  k.B = p->B;
  k.H = p->Hq;
  k.Lq = p->Lq;
  k.Lk = p->Lk;
  k.div = p->bias_batch_div[pi];
  k.groups = p->B / k.div;
  k.scale = p->scale;
  k.scale_log2 = p->scale * 1.4426950408889634f;
  const fl::StripeShape shape = fl::stripe_shape(p->Dqk, p->Lk, ri >= 0);
  // (the general kernel forms the weights of a last tile of fewer than 64 keys against its maximum, which makes the largest
  // weight exact; here the whole row's maximum, at 6 to 20 % of the time)
  k.by_maximum = p->Lk % 64 != 0;
  k.tiles = (p->Lq + 32 * shape.qb - 1) / (32 * shape.qb);
  const int64_t units = (int64_t)k.groups * k.H * k.tiles, most = chunks_of_entries((int64_t)k.groups * k.H, k.tiles, shape.per_cu, k.div);
  k.chunk_len = (int)((k.div + most - 1) / most);
  k.chunks = (k.div + k.chunk_len - 1) / k.chunk_len;
  if (units * k.chunks > (1 << 28)) return false;
  *out = k;
  *waves = shape.waves;
  launch[0] = ((int64_t)k.groups * k.chunks * k.H + 7) / 8 * 8 * k.tiles;
  launch[1] = shape.lds_bytes;
  return true;
}

// Whether *p (already validated) is a call the few-rows forward (rows_kernel.h) takes.  Fills the kernel's parameters and
// launch shape.  `scratch`: bytes of p->workspace it would use to cut the keys into chunks; with less, or without the caller's
// word that the workspace is scratch, the keys of a row tile stay in one workgroup.
bool plan_rows(const fl_attn_params* p, fl::RParams* out, int* grid, int* waves, int* blocks, uint64_t* scratch) {
  if (p->Dqk != p->Dv || !fl::rows_has_shape(p->Dqk) || is_doc(p->mask_kind) || p->diff || p->gate || p->attended_dump ||
      p->dropout_threshold || p->score_fn != FL_SCORE_NONE || (p->flags & FL_FLAG_F32_RESULT))
    return false;
  const bool has_bias = p->bias[0] || p->bias[1];
  if (has_bias && p->alibi_heads > 0) return false;
  for (int i = 0; i < 2; ++i)
    if (p->bias[i] && (p->bias_strides[i][1] != 0 || p->bias_strides[i][2] != 0)) return false;
  // row offsets inside a tile of 32 keys are 24-bit products
  if (p->k_strides[2] >= (1 << 22) || p->v_strides[2] >= (1 << 22)) return false;
  const int64_t units = (int64_t)p->B * p->Hkv, group = p->Hq / p->Hkv, rows = group * p->Lq, tiles = (p->Lk + 31) / 32;
  if (rows > (1 << 28) || units * rows > (1 << 30)) return false;
  const int64_t base16 = units * ((rows + 15) / 16), base32 = units * ((rows + 31) / 32);
  // Decoding (rows <= 32: every key is read once, or twice) belongs here at any size but the shortest: up to 128 keys the
  // tile kernel's one or two steps are 0.5 us sooner until its padded 128-row workgroups fill the part.
  // Longer row counts re-read K and V for every 16 rows (32 at head dim 64), from L2: that pays while one workgroup per
  // compute unit holds all of them, where the tile kernel leaves most of the part idle (head dim 64, 8 heads of 1024
  // causal rows: 16.8 -> 12.2 us; head dim 128, 4 heads: 21.5 -> 14.5 us), and loses beyond (twice as many rows: 17 -> 18
  // and 23 -> 30 us).  Up to 64 keys the tile kernel has a single step.  Against a long cache the front end has the tile
  // kernel over chunks of the keys besides, and takes it where that is sooner (chunks_beat_rows_kernel in host.cpp); a
  // single launch of the tile kernel is the slower one at any length (8 heads, 40 queries of 5000 keys: 81 us, here 17).
  int qt = 1;
  if (rows <= 32) {
    if (p->Lk <= 128 && (int64_t)p->B * p->Hq * ((p->Lq + 127) / 128) <= 256) return false;
    if (rows > 16 && p->Dqk == 64 && p->Lk >= 4096) qt = 2;
  } else if (p->Lk <= 64) {
    return false;
  } else if (base16 > 256) {
    if (p->Dqk != 64 || base32 > 256 || p->Lk <= 256) return false;
    qt = 2;
  }
  const int64_t row_tiles = (rows + 16 * qt - 1) / (16 * qt), base = units * row_tiles;
  // Waves per workgroup and chunks of the keys.  Eight waves fill a compute unit's registers, so 256 workgroups of eight
  // or 512 of four are one round.  Enough row tiles: no chunks, and shorter workgroups the more of them there are.  Few:
  // a chunk has two key tiles per wave at least, and the merge launch behind the chunks costs 4 us, about what reading 512
  // keys in one workgroup costs (1024 where more than two row tiles read them): up to there they stay together.  Eight waves
  // add up inside the workgroup what four would send through memory: worth it once a wave has two tiles.  (8 heads, head dim
  // 128, rows of one workgroup each -> chunks: 128 queries of 2048 keys 23.6 -> 14.8 us, 48 of 3000 keys 31.6 -> 15.3.)
  int nw = 8;
  int64_t chunks = 1;
  if (base >= 1024) {
    nw = tiles < 16 ? 2 : 4;
  } else if (base >= 512) {
    nw = 4;
  } else if (rows > 32 && (p->mask_kind != FL_MASK_NONE || tiles <= 32)) {
    nw = tiles > 8 ? 8 : 4;
  } else if (base < 256 && tiles > 16 && p->mask_kind == FL_MASK_NONE) {
    if (tiles * base >= 16 * 256) {
      chunks = 256 / base;
    } else {
      nw = 4;
      chunks = std::max<int64_t>(1, std::min<int64_t>(512 / base, tiles / 8));
    }
    // the row tiles of one (unit, chunk) stay on one XCD (by_xcd below): no XCD gets more of them than it runs at once (2 heads,
    // 48 queries, 32768 keys: 42 chunks 28.9 us, 40 chunks 18.8)
    if (row_tiles > 2 && units * chunks >= 8)
      chunks = std::max<int64_t>(1, std::min<int64_t>(chunks, 8 * ((nw == 8 ? 32 : 64) / row_tiles) / units));
  }
  fl::RParams k;
  std::memset(&k, 0, sizeof(k));
  *scratch = 0;
  if (chunks > 1) {
    const uint64_t n = (uint64_t)base * chunks * 16 * qt;
    *scratch = n * (p->Dv + 2) * sizeof(float);
    if (!(p->flags & FL_FLAG_SCRATCH) || !p->workspace || p->workspace_bytes < *scratch || reinterpret_cast<uintptr_t>(p->workspace) % 16) {
      chunks = 1;
    } else {
      k.part = static_cast<float*>(p->workspace);
      k.part_ml = k.part + n * p->Dv;
    }
  }
  k.q = static_cast<const fl::bf16_t*>(p->q);
  k.k = static_cast<const fl::bf16_t*>(p->k);
  k.v = static_cast<const fl::bf16_t*>(p->v);
  k.o = static_cast<fl::bf16_t*>(p->o);
  k.lse = p->lse;
  for (int i = 0; i < 3; ++i) {
    k.qs[i] = p->q_strides[i];
    k.ks[i] = p->k_strides[i];
    k.vs[i] = p->v_strides[i];
    k.os[i] = p->o_strides[i];
  }
  k.B = p->B;
  k.Hq = p->Hq;
  k.Hkv = p->Hkv;
  k.Lq = p->Lq;
  k.Lk = p->Lk;
  k.group = (int)group;
  k.rows = (int)rows;
  k.row_tiles = (int)row_tiles;
  k.chunks = (int)chunks;
  k.units = (int)units;
  k.waves = nw;
  k.by_rows = fl::Div::by((uint32_t)rows);
  k.by_row_tiles = fl::Div::by((uint32_t)row_tiles);
  k.by_chunks = fl::Div::by((uint32_t)chunks);
  k.by_Hkv = fl::Div::by((uint32_t)p->Hkv);
  k.by_Lq = fl::Div::by((uint32_t)p->Lq);
  const float l2e = 1.4426950408889634f;
  k.scale_log2 = p->scale * l2e;
  if (p->softcap > 0.f) {
    k.cap_k1 = p->scale / p->softcap * 2.0f * l2e;
    k.cap_c = p->softcap * l2e;
  }
  position_bounds(p, &k.dmin, &k.dmax, &k.pfx);
  k.alibi_heads = p->alibi_heads;
  for (int i = 0; i < 2; ++i) {
    k.bias[i] = p->bias[i];
    k.bias_batch[i] = p->bias_strides[i][0];
    k.bias_key[i] = (int)p->bias_strides[i][3];
    k.bias_div[i] = p->bias[i] ? p->bias_batch_div[i] : 1;
    k.bias_f32[i] = p->bias_dtype[i] == FL_F32;
  }
  k.by_xcd = units * chunks >= 8 && row_tiles > 1;
  *grid = (int)(k.by_xcd ? (units * chunks + 7) / 8 * 8 * row_tiles : units * chunks * row_tiles);
  *waves = nw;
  *blocks = qt;
  *out = k;
  return true;
}


// Layout of the shared-bias backward's scratch, in bytes from its start (parts aligned to 256).
struct SBScratch {
  int dense = -1, row = -1;  // which operand is the shared one, which the row per batch entry
  int chunks = 1, chunk_len = 1;
  uint64_t delta = 0, rowb = 0, dgated = 0, part = 0, total = 0;
};
// Whether the forward call *p is one whose gradients the shared-bias backward computes.
bool plan_shared_bias_bwd(const fl_attn_params* p, SBScratch* out) {
  if (p->Dqk != p->Dv || (p->Dqk != 32 && p->Dqk != 64) || p->Hq != p->Hkv || p->Lq != p->Lk || p->Lk > 512 || p->Lk <= 0 || p->B <= 0 ||
      p->Hq <= 0 || p->mask_kind != FL_MASK_NONE || p->alibi_heads > 0 || p->softcap > 0.f || p->diff || p->attended_dump ||
      p->dropout_threshold || p->score_fn != FL_SCORE_NONE)
    return false;
  SBScratch x;
  for (int i = 0; i < 2; ++i) {
    if (!p->bias[i]) continue;
    const int64_t* st = p->bias_strides[i];
    if (p->bias_batch_div[i] <= 0 || p->B % p->bias_batch_div[i]) return false;
    if (st[1] == 0 && st[2] == 0 && x.row < 0 && (p->Hq > 1 || p->Lq > 1)) x.row = i;
    else if ((st[1] != 0 || p->Hq == 1) && (st[2] != 0 || p->Lq == 1) && (st[3] == 1 || p->Lk == 1) && x.dense < 0) x.dense = i;
    else return false;
  }
  if (x.dense < 0 || (x.row >= 0 && !row_starts_products(p))) return false;
  // per-lane byte offsets inside one (batch entry, head) are 32-bit
  for (const int64_t* st : {p->q_strides, p->k_strides, p->v_strides, p->o_strides})
    if (st[2] < 0 || st[2] >= (1 << 20)) return false;
  if ((int64_t)p->Hq * p->Dv >= (1 << 20)) return false;  // (of a result, and of the gated output gradient, in sequence-major order)
  const int64_t S = p->Lk, H = p->Hq, div = p->bias_batch_div[x.dense], groups = p->B / div, tiles = (S + 31) / 32;
  // (both roles run in one launch)
  const int per_cu = fl::pairbias_bwd_shape(p->Dqk, (int)S).lds_bytes <= 80 * 1024 ? 2 : 1;
  int64_t chunks = chunks_of_entries(groups * H, 2 * tiles, per_cu, div);
  const int64_t len = (div + chunks - 1) / chunks;
  chunks = (div + len - 1) / len;
  if (groups * chunks * H * tiles > (1 << 28)) return false;
  x.chunks = (int)chunks;
  x.chunk_len = (int)len;
  auto add = [&](uint64_t bytes) {
    const uint64_t at = x.total;
    x.total += (bytes + 255) / 256 * 256;
    return at;
  };
  x.delta = add((uint64_t)p->B * H * S * 4);
  x.rowb = add(x.row >= 0 ? (uint64_t)p->B * S * 4 : 0);
  x.dgated = add(p->gate ? (uint64_t)p->B * H * S * p->Dv * 2 : 0);
  x.part = add((uint64_t)groups * chunks * H * S * ((S + 3) / 4 * 4) * 4);
  *out = x;
  return true;
}

}  // namespace

extern "C" {

int fl_version(void) { return FL_ABI_VERSION; }

const char* fl_last_error(void) { return g_err; }

uint64_t fl_params_sizeof(void) { return sizeof(fl_attn_params); }

uint64_t fl_workspace_bytes(const fl_attn_params* p) {
  if (!p || !is_doc(p->mask_kind) || p->B <= 0 || p->Lk <= 0) return 0;
  // tile shape of the instance the forward would run (the largest lists any compiled shape needs, if the call names no
  // valid one)
  const fl::Instance* in = select_instance(p);
  const DocScratch d = doc_scratch(p->B, p->Lk, in ? (int64_t)in->rw * in->nw : 64, in ? in->bn : 32);
  return d.table_bytes + d.lists_bytes + d.order_bytes;
}

uint64_t fl_bwd_workspace_bytes(const fl_attn_params* p) {
  if (!p || !is_doc(p->mask_kind) || p->B <= 0 || p->Lk <= 0) return 0;
  return doc_scratch(p->B, p->Lk, 128, 64).table_bytes;
}

int fl_attn_validate(const fl_attn_params* p) { return validate(p, nullptr); }

int fl_attn_plan(const fl_attn_params* p, int64_t out[8]) {
  const fl::Instance* in = nullptr;
  int rc = validate(p, &in);
  if (rc) return rc;
  if (!out) return fail(FL_ERR_NULL, "out is null");
  const int64_t bm = (int64_t)in->rw * in->nw;
  out[0] = bm;
  out[1] = in->bn;
  out[2] = in->nw * 64;
  out[3] = (int64_t)p->B * p->Hq * ((p->Lq + bm - 1) / bm);
  out[5] = in->feat;
  out[6] = 0;
  out[7] = groups_for(in, p);
  out[4] = p->diff && out[7] == 2 ? in->branches_lds_bytes : lds_bytes_for(in, p);
  {
    // calls the shared-bias streaming forward takes: its fixed shape, and out[6] = 1
    fl::PParams pb;
    int pb_grid = 0;
    if (plan_pairbias(p, &pb, &pb_grid)) {
      out[0] = 128;
      out[1] = 64;
      out[2] = 256;
      out[3] = pb_grid;
      out[4] = 2 * (p->Dqk == 32 ? 6 : 4) * 64 * p->Dqk * 2 + (pb.rowb ? 4 * 2 * 1024 : 0);
      out[6] = 1;
      out[7] = 1;
      return 0;
    }
    fl::StripeParams sp;
    int waves = 0;
    int64_t launch[2];
    if (plan_stripe(p, nullptr, &sp, &waves, launch)) {
      out[0] = p->Dqk == 32 ? 64 : 32;
      out[1] = 64 * waves;
      out[2] = 64 * waves;
      out[3] = launch[0];
      out[4] = launch[1];
      out[6] = 2;
      out[7] = 1;
    }
  }
  return 0;
}

int fl_attn_rows_plan(const fl_attn_params* p, uint64_t* scratch_bytes) {
  // (asked before fl_attn_fwd has checked the call)
  if (!p || !scratch_bytes || p->B <= 0 || p->Hkv <= 0 || p->Hq < p->Hkv || p->Hq % p->Hkv || p->Lq <= 0 || p->Lk <= 0) return 0;
  fl::RParams rp;
  int grid = 0, waves = 0, blocks = 0;
  *scratch_bytes = 0;
  return plan_rows(p, &rp, &grid, &waves, &blocks, scratch_bytes) ? 1 : 0;
}

static int launch_forward(const fl_attn_params* p, void* ungated, void* stream_) {
  const fl::Instance* in = nullptr;
  int rc = validate(p, &in);
  if (rc) return rc;
  hipStream_t stream = static_cast<hipStream_t>(stream_);

  if (!ungated) {
    fl::PParams pb;
    int pb_grid = 0;
    if (plan_pairbias(p, &pb, &pb_grid)) {
      const hipError_t e = (p->dtype == FL_F16 ? fl::launch_pairbias_f16 : fl::launch_pairbias_bf16)(
          p->Dqk, p->Lk / 32, p->gate != nullptr, pb.rowb != nullptr, pb, pb_grid, stream);
      if (e != hipSuccess) return fail((int)e, "launch of the shared-bias forward failed: %s", hipGetErrorString(e));
      return 0;
    }
  }
  {
    fl::StripeParams sp;
    int waves = 0;
    int64_t plan[2];
    if (plan_stripe(p, ungated, &sp, &waves, plan)) {
      const hipError_t e = (p->dtype == FL_F16 ? fl::launch_stripe_f16 : fl::launch_stripe_bf16)(p->Dqk, waves, forward_neighbours(sp, p->Dqk), sp, stream);
      if (e != hipSuccess) return fail((int)e, "launch of the shared-bias stripe forward failed: %s", hipGetErrorString(e));
      return 0;
    }
  }
  {
    fl::RParams rp;
    int rows_grid = 0, rows_waves = 0, rows_blocks = 0;
    uint64_t scratch = 0;
    if (plan_rows(p, &rp, &rows_grid, &rows_waves, &rows_blocks, &scratch)) {
      const uint32_t mod = p->bias[0] || p->bias[1] ? fl::F_BIAS : p->alibi_heads > 0 || p->softcap > 0.f ? fl::F_ALIBI | fl::F_SOFTCAP : 0u;
      const hipError_t e = (p->dtype == FL_F16 ? fl::launch_rows_f16 : fl::launch_rows_bf16)(p->Dqk, rows_blocks, mod, rp, rows_grid, rows_waves, stream);
      if (e != hipSuccess) return fail((int)e, "launch of the few-rows forward failed: %s", hipGetErrorString(e));
      return 0;
    }
  }

  fl::KParams kp;
  std::memset(&kp, 0, sizeof(kp));
  kp.q = static_cast<const fl::bf16_t*>(p->q);
  kp.k = static_cast<const fl::bf16_t*>(p->k);
  kp.v = static_cast<const fl::bf16_t*>(p->v);
  kp.o = static_cast<fl::bf16_t*>(p->o);
  for (int i = 0; i < 3; ++i) {
    kp.qs[i] = p->q_strides[i];
    kp.ks[i] = p->k_strides[i];
    kp.vs[i] = p->v_strides[i];
    kp.os[i] = p->o_strides[i];
    kp.gs[i] = p->gate_strides[i];
  }
  kp.B = p->B;
  kp.Hq = p->Hq;
  kp.Hkv = p->Hkv;
  kp.Lq = p->Lq;
  kp.Lk = p->Lk;
  kp.group = p->Hq / p->Hkv;
  kp.scale = p->scale;
  kp.scale_log2 = p->scale * 1.4426950408889634f;
  kp.mask_kind = p->mask_kind;
  kp.window = p->window;
  kp.prefix = p->prefix;
  position_bounds(p, &kp.dmin, &kp.dmax, &kp.pfx);
  kp.doc_ids = p->doc_ids;
  kp.doc_stride = p->doc_stride;
  kp.alibi_heads = p->alibi_heads;
  kp.softcap = p->softcap;
  if (p->score_fn != FL_SCORE_NONE) {
    // scale and log2(e) folded into the constants (in double): the kernel works on the raw q.k and in log2 units
    const double l2e = 1.4426950408889634, sc = p->scale;
    const float* c = p->score_fn_params;
    kp.score_fn = p->score_fn;
    if (p->score_fn == FL_SCORE_SIGMOID) {
      kp.score_k[0] = (float)(-(double)c[0] * sc * l2e);
      kp.score_k[1] = (float)(-(double)c[1] * l2e);
      kp.score_k[2] = (float)((double)c[2] * l2e);
      kp.score_k[3] = (float)((double)c[3] * l2e);
    } else if (p->score_fn == FL_SCORE_CLAMP) {
      kp.score_k[0] = (float)((double)c[0] * sc * l2e);
      kp.score_k[1] = (float)((double)c[1] * l2e);
      kp.score_k[2] = (float)((double)c[2] * l2e);
      kp.score_k[3] = (float)((double)c[3] * l2e);
    } else {
      kp.score_k[0] = (float)((double)c[0] * l2e);
      kp.score_k[1] = (float)((double)c[1] * sc * l2e);
      kp.score_k[2] = (float)((double)c[2] * sc * sc * l2e);
      kp.score_k[3] = (float)((double)c[3] * sc * sc * sc * l2e);
    }
  }
  for (int nb = 0; nb < 2; ++nb) {
    kp.bias[nb] = static_cast<const fl::bf16_t*>(p->bias[nb]);
    kp.bdiv[nb] = p->bias[nb] ? p->bias_batch_div[nb] : 1;
    kp.bias_f32[nb] = p->bias[nb] && p->bias_dtype[nb] == FL_F32;
    // four consecutive keys of a row in one load: 8 bytes of bf16 or 16 bytes of fp32
    bool vec = p->bias[nb] && p->bias_strides[nb][3] == 1 &&
               reinterpret_cast<uintptr_t>(p->bias[nb]) % (kp.bias_f32[nb] ? 16 : 8) == 0;
    for (int i = 0; i < 4; ++i) {
      kp.bs[nb][i] = p->bias_strides[nb][i];
      if (i < 3 && p->bias_strides[nb][i] % 4 != 0) vec = false;
    }
    kp.bias_vec[nb] = vec ? 1 : 0;
  }
  // Bias operands travel through LDS with the K/V tiles when their rows are addressable in 16-byte pieces: one
  // row-broadcast operand (query stride 0) as single rows, one more as [rows][keys] tiles; any other takes the direct
  // path.
  kp.bias_lds = -1;
  kp.bias_row = -1;
  for (int nb = 0; nb < 2; ++nb) {
    if (!bias_stageable(p, nb)) continue;
    // fp32: staged only as the row-broadcast operand (the [rows][keys] tiles hold 16-bit elements, so a second fp32 row
    // operand takes the direct path)
    if (kp.bias_f32[nb] && (p->bias_strides[nb][2] != 0 || kp.bias_row >= 0)) continue;
    if (p->bias_strides[nb][2] == 0 && kp.bias_row < 0) kp.bias_row = nb;
    else if (kp.bias_lds < 0) kp.bias_lds = nb;
  }
  kp.gate = static_cast<const fl::bf16_t*>(p->gate);
  kp.ungated = static_cast<fl::bf16_t*>(ungated);
  kp.lambda = p->lambda;
  if (p->diff) {
    // heads [0, H) are branch 0, heads [H, 2H) branch 1 (query: H = Hq, key: H = Hkv)
    kp.q_branch_stride = (int64_t)p->Hq * p->q_strides[1];
    kp.k_branch_stride = (int64_t)p->Hkv * p->k_strides[1];
  }
  kp.dump = p->attended_dump;
  kp.lse = p->lse;
  kp.drop_thr = p->dropout_threshold;
  kp.drop_seed[0] = p->dropout_seed[0];
  kp.drop_seed[1] = p->dropout_seed[1];
  kp.drop_rescale = 65536.0f / (65536.0f - (float)p->dropout_threshold);
  const int bm = in->rw * in->nw;
  kp.n_qtiles = (p->Lq + bm - 1) / bm;
  kp.n_ktiles = (p->Lk + in->bn - 1) / in->bn;
  {
    // Masks whose work grows with the query position: (batch, head) pairs are taken four at a time (measured: one at a
    // time costs the document-mask configuration 20 %, whose two heads per XCD then drain one after the other; two, eight
    // or sixteen instead of four change the causal launch by 1-4 %)
    const bool growing = p->mask_kind == FL_MASK_CAUSAL || p->mask_kind == FL_MASK_PREFIX_LM || is_doc(p->mask_kind);
    static const int knob = std::getenv("FL_HEAD_GROUP") ? std::atoi(std::getenv("FL_HEAD_GROUP")) : 0;  // tuning knob
    kp.head_group = !growing ? 1 : (knob > 0 ? knob : 4);
    const uint32_t pairs = (uint32_t)p->B * p->Hq, per_xcd = pairs % 8 ? pairs : pairs / 8, rest = per_xcd % kp.head_group;
    kp.by_heads = fl::Div::by((uint32_t)kp.head_group * kp.n_qtiles);
    kp.by_head_group = fl::Div::by(kp.head_group);
    kp.by_rest = fl::Div::by(rest ? rest : 1);
    kp.by_Hq = fl::Div::by(p->Hq);
    kp.by_group = fl::Div::by(kp.group);
  }
  kp.o_wide = reinterpret_cast<uintptr_t>(p->o) % 16 == 0 && p->o_strides[0] % 8 == 0 && p->o_strides[1] % 8 == 0 &&
              p->o_strides[2] % 8 == 0;
  if (p->flags & FL_FLAG_F32_RESULT) kp.o_wide = 2;
  const int grid = p->B * p->Hq * kp.n_qtiles;

  const int groups = groups_for(in, p);
  if (p->softcap > 0.f && near_cap_pays(p, in, groups, grid)) kp.near_cap = fl::NearCap::of(p->scale, p->softcap);
  int lds = p->diff && groups == 2 ? in->branches_lds_bytes : (int)lds_bytes_for(in, p) + (groups - 1) * in->lds_fixed_bytes;

  if (is_doc(p->mask_kind)) {
    const DocScratch d = doc_scratch(p->B, p->Lk, bm, in->bn);
    uint32_t* lists = reinterpret_cast<uint32_t*>(static_cast<unsigned char*>(p->workspace) + d.table_bytes);
    int32_t* order = reinterpret_cast<int32_t*>(static_cast<unsigned char*>(p->workspace) + d.table_bytes + d.lists_bytes);
    // Few key tiles and workgroups: each workgroup lists its own tiles (fwd_kernel.h) and the pre-pass is not launched.  Up to two rounds:
    // beyond, every workgroup's own list and the order that is missing cost more than the launches (us, launches -> own: 4 x 32 heads
    // of 837 ids, head dim 64, 896 workgroups 39.3 -> 37.3; 2 x 32 of 2500, 1280: 59.8 -> 60.9; 16 x 16 of 1500, 3072: 86 -> 92).
    const bool own = !(p->flags & FL_FLAG_DOC_PREPARED) && kp.n_ktiles <= fl::kOwnListTiles && grid <= 1024 &&
                     lds + fl::kOwnListBytes <= fl::kMaxLdsBytes;
    if (own) {
      kp.doc_own = 1;
      lds += fl::kOwnListBytes;
    } else if (!(p->flags & FL_FLAG_DOC_PREPARED)) {
      if (in->nw > fl::kDocWaves) return fail(FL_ERR_UNSUPPORTED, "%s: more waves than the document lists have classes for", in->name);
      const bool orders = fl::doc_orders(p->B, kp.n_qtiles, kp.n_ktiles);
      const auto make_lists = orders ? &fl::doc_lists_kernel<true> : &fl::doc_lists_kernel<false>;
      static const hipError_t attrs[2] = {
          hipFuncSetAttribute(reinterpret_cast<const void*>(&fl::doc_lists_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, fl::kMaxLdsBytes - 128),
          hipFuncSetAttribute(reinterpret_cast<const void*>(&fl::doc_lists_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, fl::kMaxLdsBytes - 128)};
      if (attrs[orders] != hipSuccess) return fail((int)attrs[orders], "doc_lists_kernel: %s", hipGetErrorString(attrs[orders]));
      hipLaunchKernelGGL(make_lists, dim3(p->B * kp.n_qtiles), dim3(1024), (size_t)prepass_lds_bytes(kp.n_ktiles), stream,
                         p->doc_ids, p->doc_stride, p->Lk, p->mask_kind, bm, in->rw, in->bn, kp.n_qtiles, kp.n_ktiles,
                         (int)d.list_stride, lists, order);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return fail((int)e, "doc_lists_kernel launch failed: %s", hipGetErrorString(e));
      if (!orders) {
        hipLaunchKernelGGL(fl::doc_order_kernel, dim3(p->B), dim3(1024), (size_t)kp.n_qtiles * 4, stream, lists, (int)d.list_stride, kp.n_qtiles, order);
        e = hipGetLastError();
        if (e != hipSuccess) return fail((int)e, "doc_order_kernel launch failed: %s", hipGetErrorString(e));
      }
    }
    kp.doc_lists = lists;
    kp.doc_list_stride = (int)d.list_stride;
    kp.doc_order = order;
  }
  hipError_t e = in->launch(kp, groups, grid, lds, stream);
  if (e != hipSuccess) return fail((int)e, "launch of %s failed: %s", in->name, hipGetErrorString(e));
  return 0;
}

int fl_attn_fwd(const fl_attn_params* p, void* stream) { return launch_forward(p, nullptr, stream); }

int fl_attn_fwd_ungated(const fl_attn_params* p, void* ungated, void* stream) {
  if (!p) return fail(FL_ERR_NULL, "params is null");
  if (!p->gate) return fail(FL_ERR_ARG, "a result before the gate needs a gate");
  const int rc = check_ptr("ungated", ungated, 16);
  return rc ? rc : launch_forward(p, ungated, stream);
}

uint64_t fl_static_scratch_bytes(void) { return kStaticScratchBytes; }

uint64_t fl_bwd_params_sizeof(void) { return sizeof(fl_attn_bwd_params); }

static int validate_bwd(const fl_attn_bwd_params* b, const fl::BwdInstance** out) {
  if (!b) return fail(FL_ERR_NULL, "params is null");
  const fl_attn_params* p = &b->fwd;
  int rc = validate(p, nullptr, true);
  if (rc) return rc;
  if (p->gate || p->diff || p->attended_dump)
    return fail(FL_ERR_UNSUPPORTED, "backward: gate, differential attention and the dump hook are not supported");
  if (p->score_fn != FL_SCORE_NONE) return fail(FL_ERR_UNSUPPORTED, "backward: score_fn is forward-only");
  const bool has_bias = p->bias[0] || p->bias[1];
  if (b->dscores && p->softcap > 0.f)
    return fail(FL_ERR_UNSUPPORTED, "backward: dscores is not produced under a soft-cap (gradients of bias operands added after the cap)");
  if (b->dscores && !has_bias) return fail(FL_ERR_ARG, "backward: dscores is only written for calls with bias operands");
  if (b->dscores && reinterpret_cast<uintptr_t>(b->dscores) % 16) return fail(FL_ERR_ALIGN, "backward: dscores must be 16-byte aligned");
  if (p->Dqk != p->Dv) return fail(FL_ERR_UNSUPPORTED, "backward needs Dqk == Dv (got %d, %d)", p->Dqk, p->Dv);
  if ((rc = check_ptr("dout", b->dout, 16)) || (rc = check_ptr("dq", b->dq, 8)) || (rc = check_ptr("dk", b->dk, 8)) ||
      (rc = check_ptr("dv", b->dv, 8)) || (rc = check_ptr("delta", b->delta, 16)) ||
      (rc = check_ptr("fwd.lse", p->lse, 16)))
    return rc;
  if ((rc = check_strides("dout", b->dout_strides, 8)) || (rc = check_strides("dq", b->dq_strides, 4)) ||
      (rc = check_strides("dk", b->dk_strides, 4)) || (rc = check_strides("dv", b->dv_strides, 4)) ||
      (rc = check_strides("o", p->o_strides, 8)))
    return rc;
  if (reinterpret_cast<uintptr_t>(p->o) % 16) return fail(FL_ERR_ALIGN, "backward: o must be 16-byte aligned");
  for (int i = 0; i < 6; ++i)
    if (b->reserved[i] != 0) return fail(FL_ERR_ARG, "reserved[%d] must be 0", i);
  // per-lane byte offsets inside one staged tile (up to 128 rows) are 32-bit
  const int64_t worst = std::max(std::max(p->q_strides[2], p->k_strides[2]), std::max(p->v_strides[2], b->dout_strides[2]));
  if ((128 * worst + p->Dqk) * 2 >= ((int64_t)1 << 31))
    return fail(FL_ERR_STRIDE, "backward: sequence stride too large (%lld elements)", (long long)worst);
  if ((int64_t)p->B * p->Hq * ((p->Lq + 127) / 128) > 0x7fffffff || (int64_t)p->B * p->Hkv * ((p->Lk + 127) / 128) > 0x7fffffff)
    return fail(FL_ERR_SHAPE, "backward: too many workgroups");
  uint32_t want = 0;
  if (p->alibi_heads > 0 || p->softcap > 0.f) want = fl::F_ALIBI | fl::F_SOFTCAP;
  // ALiBi alone: a kernel without the soft-cap where there is one (T::ORDERED, whose kernels with it take it as given)
  if (want != 0 && !(p->softcap > 0.f) && p->Dqk >= 64 && !is_doc(p->mask_kind) && !has_bias && !p->dropout_threshold) want = fl::F_ALIBI;
  if (is_doc(p->mask_kind)) want |= fl::F_DOC;
  if (has_bias) want |= fl::F_BIAS;
  if (p->dropout_threshold) want |= fl::F_DROPOUT;  // (head dims 64 and 128)
  const fl::BwdInstance* in = nullptr;
  for (int i = 0; i < fl::kNumBwdInstances; ++i)
    if (fl::kBwdInstances[i].d == p->Dqk && fl::kBwdInstances[i].feat == want && fl::kBwdInstances[i].dtype == p->dtype)
      in = &fl::kBwdInstances[i];
  if (!in)
    return fail(FL_ERR_UNSUPPORTED, "backward: no kernel for head dim %d with features 0x%x (compiled: 32, 64 and 128; dropout at 64 "
                "and 128)", p->Dqk, want);
  if (out) *out = in;
  g_err[0] = 0;
  return 0;
}

int fl_attn_bwd_validate(const fl_attn_bwd_params* b) { return validate_bwd(b, nullptr); }

// How the gradient kernels are launched.  A tile of 128 query rows or keys is one workgroup, and a launch that leaves compute
// units idle, or one wave per SIMD, is a chain of latencies: 1.9 us per step of the dK/dV kernel at head dim 64 with one
// wave per SIMD, next to nothing more with two.  So while the tiles of one role alone do not fill the part about twice
// (512 workgroups of four waves, 256 of eight at head dim 128), both roles run in one launch, and tiles whose walk over the
// streamed steps is longer than an even share of all steps (half of them under masks of growing length) are cut into
// splits of about that share.  A split costs the writing and reading of its partial sums and its own prologue, and the
// sums a launch of 5 to 9 us: no split has fewer than eight steps, and a tile of up to one and a half shares stays whole.
// Beyond, a launch per role is the better one (dQ alone has room for more workgroups: 4 x 16 x 4096, head dim 64, causal: 533 us
// against 565; 2 x 16 x 2048, head dim 128, unmasked: 271 against 300), unless the dK/dV launch ends on a second round that is
// far from full (up to 896 tiles at head dim 64) or on the tiles of long documents (up to 2048): dQ's workgroups then fill what the
// two launches leave idle.  Two launches -> one, us, head dim 64: 32 over 10 x 8 heads of 1139, unmasked 497 -> 457, window 300 238 -> 214;
// 16 over 10 x 4 of 2000 with a prefix 505 -> 424; documents: 32 over 2 x 8 of 8037 1475 -> 1063, 16 of 16384 742 -> 647.  Full
// rounds lose (1024 tiles, unmasked: 262 -> 270), and so does head dim 128 (7 x 16 of 1000: 298 -> 302; 6 x 32 over 8 of 2000: 1389 -> 1417).
// A whole dK/dV tile is also too long a walk where it is near a share itself: the compute units that have two of them run late.
// Measured at 0.9 shares and two dozen steps, with a step of this role at five quarters of one of dQ's (head dim 64; us, whole ->
// cut in two): 8 over 12 heads of 3000 (288 tiles of 376 steps) 963 -> 853, over 14: 987 -> 974, over 16: 1088 -> 1095; 32 over 5 x 4 of 1139
// 311 -> 246; head dim 128, 8 over 11 of 1000: 247 -> 199.  For the same reason not a few more splits than compute units at head dim 64
// (8 over 3 of 3730, 90 tiles: 270 splits 423, 360 splits 359).  Under documents the steps that count are fewer than the
// positions tell, and at head dim 128, with one workgroup per compute unit, the longest tile is what the others wait for: three
// quarters of a share there (8 over 2 x 2 of 6000: 553 -> 312, 8 over 5 of 3266 with four draws of documents 345, 263, 363, 254 -> 307, 268, 334, 261).
// Gradients, bf16, a launch per role with whole tiles -> this rule (both with the mask as selects, see bwd_kernel.h), now in
// brackets: 3 x 16 heads over 4 x 1000 prefix rows, head dim 64: 157 -> 77 us (72); 8 x 512 causal, 64: 36 -> 25 (20); 8 over
// 1 x 8192 causal, 64: 1980 -> 342 (284); 8 x 512 causal, 128: 47 -> 29 (27); 8 over 1 x 2048 causal, 128: 568 -> 73 (72);
// 32 over 4 x 4096 causal, 128: 1214 -> 611 (565); 2 x 16 x 2048 causal, 64: 131 -> 107 (94).
namespace {
struct BwdPlan {
  bool both = false;    // one launch
  int dq = 1, dkv = 1;  // splits per tile
  uint64_t dq_bytes = 0, bytes = 0;  // scratch: dQ's partial sums, then dK's and dV's
};
BwdPlan plan_bwd(const fl_attn_params* p) {
  BwdPlan x;
  const int64_t D = p->Dqk, q_tiles = (int64_t)p->B * p->Hq * ((p->Lq + 127) / 128), k_tiles = (int64_t)p->B * p->Hkv * ((p->Lk + 127) / 128);
  const int64_t least = std::min(q_tiles, k_tiles);
  const bool small = D <= 64, doc = is_doc(p->mask_kind);
  x.both = small ? least <= 512 : least < 512;
  if (!x.both) {
    x.both = small && k_tiles <= (doc ? 2048 : 896);
    return x;
  }
  int64_t q_steps = (p->Lk + 63) / 64, k_steps = (p->Lq + 63) / 64;
  if (p->mask_kind == FL_MASK_SLIDING) {
    const int64_t band = ((int64_t)p->window + 128) / 64 + 1;
    q_steps = std::min(q_steps, band);
    k_steps = std::min(k_steps, band);
  }
  k_steps *= p->Hq / p->Hkv;
  const bool growing = p->mask_kind != FL_MASK_NONE && p->mask_kind != FL_MASK_SLIDING;
  const int64_t dq_work = q_tiles * q_steps / (growing ? 2 : 1), dkv_work = k_tiles * k_steps / (growing ? 2 : 1);
  const int64_t slots = small ? 512 : 256;
  const int64_t share = std::max<int64_t>(8, (dq_work + dkv_work) / slots);
  const int64_t dkv_share = small ? (4 * dq_work + 5 * dkv_work) / (5 * slots) : share;
  const auto splits = [](int64_t steps, int64_t share) { return (int)((steps + share - 1) / share); };
  if (2 * q_steps > 3 * share) x.dq = splits(q_steps, share);
  if (2 * k_steps > 3 * share || 10 * k_steps > 9 * dkv_share + 240) {
    x.dkv = std::max(2, splits(k_steps, doc && !small ? std::max<int64_t>(8, share * 3 / 4) : share));
    if (small && k_tiles * x.dkv > 256 && k_tiles * x.dkv <= 320 && k_steps >= 16 * x.dkv) ++x.dkv;
  }
  x.dq_bytes = x.dq > 1 ? (uint64_t)x.dq * q_tiles * 128 * D * sizeof(float) : 0;
  x.bytes = x.dq_bytes + (x.dkv > 1 ? (uint64_t)x.dkv * k_tiles * 128 * D * 2 * sizeof(float) : 0);
  return x;
}

// dK and dV, a launch of their own at head dim 128 without score modifications: 256 keys per workgroup instead of 128, one workgroup of
// eight waves per compute unit either way, so a round takes twice as long and there are half as many.  us, both roles, 128 -> 256 keys:
// A last round that is far from full costs more of them: no mask, 16 heads of 4096 (256 tiles of 256 keys) 428 -> 411, 24 (384) 648 -> 679 (below
// 256 tiles both roles share a launch, of 128 keys); from 1024 tiles on there are rounds enough, 128 heads of 2048 890 -> 850, 129 968 -> 965, 96
// of 3000 (1152) 1398 -> 1381, but 43 of 6000 (1032) 2400 -> 2530.  Windows of 100, 8 x 16 of 4096, 515 -> 487; of 256, 129 of 2048 320 -> 303; of
// more than half the keys, 32 of 4096 424 -> 440, of all of them 492 -> 549, 129 of 2048 833 -> 859, 121 of 1000 240 -> 217.  Few of the keys'
// places may be empty.
// Masks of growing length, whose longest walk is twice the average, want more rounds.  Where the heads divide by the 8 XCDs, causal, 16 of 4096
// 259 -> 303, 32 (512) 464 -> 443, 64 901 -> 863, 104 of 3000 897 -> 906, a prefix, 8 x 16 of 1500, 352 -> 325; with one tile per head full rounds
// only, 1024 of 256 225 -> 213, 1088 233 -> 236.  Where they do not, and tiles go round the XCDs, causal, 121 of 1000 (484) 220 -> 199, but 81
// of 1536 (486) 254 -> 261, 63 of 3000 (756) 620 -> 643; from 1000 tiles on 0.92 to 1.0 of the time at 1100 to 7000 keys (0.93 to 1.02 under a
// prefix), but for tiles per head that are a multiple of 8: 129 of 2048 628 -> 735, 65 of 4096 1053 -> 1079, 43 of 6000 1386 -> 1468.
bool wide_dkv(const fl_attn_params* p) {
  const int64_t narrow = (p->Lk + 127) / 128, wide = (p->Lk + 255) / 256, heads = (int64_t)p->B * p->Hkv, tiles = heads * wide, last = tiles % 256;
  if (p->Dqk != 128 || p->alibi_heads > 0 || p->softcap > 0.f || p->bias[0] || p->bias[1] || is_doc(p->mask_kind) || p->dropout_threshold) return false;
  if (2 * wide > narrow && narrow < 16) return false;
  const bool full = last == 0 || last > 224, window = p->mask_kind == FL_MASK_SLIDING;
  if (p->mask_kind == FL_MASK_CAUSAL || p->mask_kind == FL_MASK_PREFIX_LM) {
    if (heads % 8) return (tiles >= 1000 ? wide % 8 != 0 : p->Lk <= 1024) && (tiles >= 1024 || (tiles > 480 && full));
    return (tiles >= 1024 && wide > 1) || (tiles > 480 && full);
  }
  if (window && 2 * (int64_t)p->window > p->Lk && p->Lk > 1536) return false;
  if (tiles >= 1024) return window || p->Lk <= 4096 || full || last > 64;
  return tiles > (window ? 480 : 0) && full;
}
}  // namespace

uint64_t fl_attn_bwd_split_bytes(const fl_attn_params* p) {
  if (!p || p->B <= 0 || p->Hkv <= 0 || p->Hq < p->Hkv || p->Lq <= 0 || p->Lk <= 0 || p->Dqk <= 0) return 0;
  return plan_bwd(p).bytes;
}

int fl_attn_bwd_plan(const fl_attn_params* p, int64_t out[4]) {
  if (!p || !out) return fail(FL_ERR_NULL, "%s is null", p ? "out" : "params");
  if (p->B <= 0 || p->Hkv <= 0 || p->Hq < p->Hkv || p->Hq % p->Hkv || p->Lq <= 0 || p->Lk <= 0 || p->Dqk <= 0)
    return fail(FL_ERR_SHAPE, "sizes must be positive, query heads a multiple of key/value heads");
  const BwdPlan x = plan_bwd(p);
  out[0] = x.both ? 1 : 2;
  out[1] = x.dq;
  out[2] = x.dkv;
  out[3] = !x.both && wide_dkv(p) ? 256 : 128;
  return 0;
}

// `planned`: sums may be taken in another order than one workgroup per tile and role takes them in, whatever else the call holds
static int launch_gradients(const fl_attn_bwd_params* b, bool planned, void* scratch, uint64_t scratch_bytes, void* stream_) {
  const fl::BwdInstance* in = nullptr;
  int rc = validate_bwd(b, &in);
  if (rc) return rc;
  if (scratch && reinterpret_cast<uintptr_t>(scratch) % 16) return fail(FL_ERR_ALIGN, "scratch must be 16-byte aligned");
  const fl_attn_params* p = &b->fwd;
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  fl::BParams bp;
  std::memset(&bp, 0, sizeof(bp));
  bp.q = static_cast<const fl::bf16_t*>(p->q);
  bp.k = static_cast<const fl::bf16_t*>(p->k);
  bp.v = static_cast<const fl::bf16_t*>(p->v);
  bp.o = static_cast<const fl::bf16_t*>(p->o);
  bp.dout = static_cast<const fl::bf16_t*>(b->dout);
  bp.lse = p->lse;
  bp.delta = b->delta;
  bp.dq = static_cast<fl::bf16_t*>(b->dq);
  bp.dk = static_cast<fl::bf16_t*>(b->dk);
  bp.dv = static_cast<fl::bf16_t*>(b->dv);
  for (int i = 0; i < 3; ++i) {
    bp.qs[i] = p->q_strides[i];
    bp.ks[i] = p->k_strides[i];
    bp.vs[i] = p->v_strides[i];
    bp.os[i] = p->o_strides[i];
    bp.dos[i] = b->dout_strides[i];
    bp.dqs[i] = b->dq_strides[i];
    bp.dks[i] = b->dk_strides[i];
    bp.dvs[i] = b->dv_strides[i];
  }
  bp.B = p->B;
  bp.Hq = p->Hq;
  bp.Hkv = p->Hkv;
  bp.Lq = p->Lq;
  bp.Lk = p->Lk;
  bp.group = p->Hq / p->Hkv;
  bp.scale = p->scale;
  bp.scale_log2 = p->scale * 1.4426950408889634f;
  bp.mask_kind = p->mask_kind;
  bp.window = p->window;
  bp.prefix = p->prefix;
  position_bounds(p, &bp.dmin, &bp.dmax, &bp.pfx);
  bp.doc_ids = p->doc_ids;
  bp.doc_stride = p->doc_stride;
  bp.alibi_heads = p->alibi_heads;
  bp.softcap = p->softcap;
  bp.drop_thr = p->dropout_threshold;
  bp.drop_seed[0] = p->dropout_seed[0];
  bp.drop_seed[1] = p->dropout_seed[1];
  bp.drop_rescale = 65536.0f / (65536.0f - (float)p->dropout_threshold);
  for (int nb = 0; nb < 2; ++nb) {
    bp.bias[nb] = p->bias[nb];
    for (int i = 0; i < 4; ++i) bp.bbs[nb][i] = p->bias_strides[nb][i];
    bp.bdiv[nb] = p->bias_batch_div[nb] > 0 ? p->bias_batch_div[nb] : 1;
    bp.bias_f32[nb] = p->bias_dtype[nb] == FL_F32;
  }
  bp.dscores = b->dscores;
  if (is_doc(p->mask_kind)) {
    const int blocks = (p->Lk + fl::kDocBlock - 1) / fl::kDocBlock;
    const int total = p->B * blocks;
    int64_t* table = static_cast<int64_t*>(p->workspace);
    hipLaunchKernelGGL(fl::doc_table_kernel, dim3((total + 255) / 256), dim3(256), 0, stream, p->doc_ids, p->doc_stride,
                       p->Lk, blocks, total, table);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail((int)e, "doc_table_kernel launch failed: %s", hipGetErrorString(e));
    bp.doc_table = table;
    bp.doc_blocks = blocks;
  }
  BwdPlan plan = plan_bwd(p);
  if (plan.bytes && (!scratch || plan.bytes > scratch_bytes)) planned = false;
  if (!planned) {
    plan.dq = plan.dkv = 1;
    plan.both = plan.both && p->Dqk <= 64;  // (at head dim 128 the shared launch halves every dQ step between two waves)
  }
  bp.part_dq = static_cast<float*>(scratch);
  if (plan.dkv > 1) bp.part = bp.part_dq + plan.dq_bytes / sizeof(float);
  bp.splits_dq = plan.dq;
  bp.splits = plan.dkv;
  bp.dkv_own = planned && !plan.both && wide_dkv(p) ? 256 : 128;
  bp.head_group = p->mask_kind == FL_MASK_CAUSAL || p->mask_kind == FL_MASK_PREFIX_LM || p->mask_kind == FL_MASK_DOCUMENT_CAUSAL ? 4 : 1;
  bp.by_head_group = fl::Div::by(bp.head_group);
  bp.by_group = fl::Div::by(bp.group);
  bp.by_Hq = fl::Div::by(p->Hq);
  for (int r = 0; r < 2; ++r) {
    const uint32_t heads = r ? p->Hkv : p->Hq, own = r ? bp.dkv_own : 128, tiles = ((r ? p->Lk : p->Lq) + own - 1) / own, pairs = p->B * heads;
    const uint32_t rest = (pairs % 8 ? pairs : pairs / 8) % bp.head_group;
    bp.role[r].by_heads = fl::Div::by(bp.head_group * tiles);
    bp.role[r].by_rest = fl::Div::by(rest ? rest : 1);
    bp.role[r].by_oh = fl::Div::by(heads);
    bp.role[r].by_splits = fl::Div::by(r ? plan.dkv : plan.dq);
    bp.role[r].by_tiles = fl::Div::by(tiles);
  }
  hipError_t e;
  if (plan.both) {
    e = in->launch_delta(bp, stream);
    if (e != hipSuccess) return fail((int)e, "backward: launch of the row-sum kernel failed: %s", hipGetErrorString(e));
    e = in->launch_both(bp, stream);
    if (e != hipSuccess) return fail((int)e, "backward: launch of the gradient kernel failed: %s", hipGetErrorString(e));
    return 0;
  }
  e = in->launch_dq(bp, stream);
  if (e != hipSuccess) return fail((int)e, "backward: launch of the dQ kernel failed: %s", hipGetErrorString(e));
  e = in->launch_dkv(bp, stream);
  if (e != hipSuccess) return fail((int)e, "backward: launch of the dK/dV kernel failed: %s", hipGetErrorString(e));
  return 0;
}

int fl_attn_bwd(const fl_attn_bwd_params* b, void* stream) { return launch_gradients(b, false, nullptr, 0, stream); }

int fl_attn_bwd_split(const fl_attn_bwd_params* b, void* scratch, uint64_t scratch_bytes, void* stream) {
  return launch_gradients(b, true, scratch, scratch_bytes, stream);
}

uint64_t fl_attn_shared_bias_bwd_bytes(const fl_attn_params* p) {
  SBScratch x;
  return p && plan_shared_bias_bwd(p, &x) ? x.total : 0;
}

int fl_attn_shared_bias_bwd(const fl_attn_shared_bias_bwd_params* b, void* stream_) {
  if (!b) return fail(FL_ERR_NULL, "params is null");
  const fl_attn_params* p = &b->fwd;
  int rc = validate(p, nullptr, false, FL_FLAG_UNGATED | FL_FLAG_SCRATCH);
  if (rc) return rc;
  SBScratch x;
  if (!plan_shared_bias_bwd(p, &x)) return fail(FL_ERR_UNSUPPORTED, "fl_attn_shared_bias_bwd does not take this call");
  if ((rc = check_ptr("dout", b->dout, 16)) || (rc = check_ptr("dq", b->dq, 8)) || (rc = check_ptr("dk", b->dk, 8)) ||
      (rc = check_ptr("dv", b->dv, 8)) || (rc = check_ptr("fwd.lse", p->lse, 4)) || (rc = check_ptr("fwd.o", p->o, 16)) ||
      (rc = check_strides("o", p->o_strides, 8)) || (rc = check_strides("dout", b->dout_strides, 8)) ||
      (rc = check_strides("dq", b->dq_strides, 4)) || (rc = check_strides("dk", b->dk_strides, 4)) ||
      (rc = check_strides("dv", b->dv_strides, 4)))
    return rc;
  for (const int64_t* st : {b->dout_strides, b->dq_strides, b->dk_strides, b->dv_strides})
    if (st[2] >= (1 << 20)) return fail(FL_ERR_STRIDE, "sequence stride of a gradient too large (%lld elements)", (long long)st[2]);
  if (p->gate && ((rc = check_ptr("gate", p->gate, 16)) || (rc = check_strides("gate", p->gate_strides, 8)) ||
                  (rc = check_ptr("dgate", b->dgate, 16)) || (rc = check_strides("dgate", b->dgate_strides, 8))))
    return rc;
  if ((rc = check_ptr("workspace", b->workspace, 256))) return rc;
  if (b->workspace_bytes < x.total)
    return fail(FL_ERR_WORKSPACE, "workspace of %llu bytes needed, got %llu", (unsigned long long)x.total, (unsigned long long)b->workspace_bytes);
  const bool f32 = p->bias_dtype[x.dense] == FL_F32;
  if (b->dbias && reinterpret_cast<uintptr_t>(b->dbias) % (f32 ? 4 : 2)) return fail(FL_ERR_ALIGN, "dbias is not aligned");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  unsigned char* ws = static_cast<unsigned char*>(b->workspace);
  const bool f16 = p->dtype == FL_F16, gate = p->gate != nullptr;

  fl::SBPrepParams pp;
  std::memset(&pp, 0, sizeof(pp));
  pp.out = static_cast<const fl::bf16_t*>(p->o);
  pp.dout = static_cast<const fl::bf16_t*>(b->dout);
  pp.gate = static_cast<const fl::bf16_t*>(p->gate);
  pp.ungated = (p->flags & FL_FLAG_UNGATED) != 0;
  pp.dgated = reinterpret_cast<fl::bf16_t*>(ws + x.dgated);
  pp.dgate = static_cast<fl::bf16_t*>(b->dgate);
  pp.delta = reinterpret_cast<float*>(ws + x.delta);
  pp.row_div = 1;
  if (x.row >= 0) {
    pp.row = p->bias[x.row];
    pp.rowb = reinterpret_cast<float*>(ws + x.rowb);
    pp.row_factor = 1.0f / p->scale;
    pp.row_batch = p->bias_strides[x.row][0];
    pp.row_key = (int)p->bias_strides[x.row][3];
    pp.row_div = p->bias_batch_div[x.row];
    pp.row_f32 = p->bias_dtype[x.row] == FL_F32;
  }
  pp.B = p->B;
  pp.H = p->Hq;
  pp.S = p->Lq;
  const int64_t row = (int64_t)p->Hq * p->Dv, dgs[3] = {row * p->Lq, p->Dv, row};  // gated dO: [batch][position][head][dim]
  for (int i = 0; i < 3; ++i) {
    pp.os[i] = p->o_strides[i];
    pp.dos[i] = b->dout_strides[i];
    pp.gs[i] = p->gate_strides[i];
    pp.dgs[i] = b->dgate_strides[i];
    pp.dgds[i] = dgs[i];
  }
  hipError_t e = (f16 ? fl::launch_pairbias_bwd_prep_f16 : fl::launch_pairbias_bwd_prep_bf16)(p->Dqk, gate, pp, stream);
  if (e != hipSuccess) return fail((int)e, "shared-bias backward: launch of the row-sum kernel failed: %s", hipGetErrorString(e));

  fl::SBParams sp;
  std::memset(&sp, 0, sizeof(sp));
  sp.q = static_cast<const fl::bf16_t*>(p->q);
  sp.k = static_cast<const fl::bf16_t*>(p->k);
  sp.v = static_cast<const fl::bf16_t*>(p->v);
  sp.dout = gate ? pp.dgated : pp.dout;
  sp.lse = p->lse;
  sp.delta = pp.delta;
  sp.rowb = pp.rowb;
  sp.dq = static_cast<fl::bf16_t*>(b->dq);
  sp.dk = static_cast<fl::bf16_t*>(b->dk);
  sp.dv = static_cast<fl::bf16_t*>(b->dv);
  for (int i = 0; i < 3; ++i) {
    sp.qs[i] = p->q_strides[i];
    sp.ks[i] = p->k_strides[i];
    sp.vs[i] = p->v_strides[i];
    sp.dos[i] = gate ? dgs[i] : b->dout_strides[i];
    sp.dqs[i] = b->dq_strides[i];
    sp.dks[i] = b->dk_strides[i];
    sp.dvs[i] = b->dv_strides[i];
    sp.bs[i] = p->bias_strides[x.dense][i];
  }
  sp.bias = p->bias[x.dense];
  sp.bias_f32 = f32;
  sp.bias_vec = p->Lk % 4 == 0 && sp.bs[0] % 4 == 0 && sp.bs[1] % 4 == 0 && sp.bs[2] % 4 == 0 &&
                reinterpret_cast<uintptr_t>(sp.bias) % (f32 ? 16 : 8) == 0;
  sp.B = p->B;
  sp.H = p->Hq;
  sp.S = p->Lk;
  sp.div = p->bias_batch_div[x.dense];
  sp.groups = sp.B / sp.div;
  sp.chunks = x.chunks;
  sp.chunk_len = x.chunk_len;
  sp.tiles = (sp.S + 31) / 32;
  sp.neighbours = gradient_neighbours(p);
  sp.s_pad = (sp.S + 3) / 4 * 4;
  sp.scale = p->scale;
  sp.scale_log2 = p->scale * 1.4426950408889634f;
  sp.dbias_part = b->dbias ? reinterpret_cast<float*>(ws + x.part) : nullptr;
  const fl::SBShape shape = fl::pairbias_bwd_shape(p->Dqk, sp.S);
  e = (f16 ? fl::launch_pairbias_bwd_f16 : fl::launch_pairbias_bwd_bf16)(p->Dqk, shape, gradient_ahead(p), sp, stream);
  if (e != hipSuccess) return fail((int)e, "shared-bias backward: launch failed: %s", hipGetErrorString(e));
  if (b->dbias) {
    e = (f16 ? fl::launch_pairbias_bwd_reduce_f16 : fl::launch_pairbias_bwd_reduce_bf16)(f32, sp, b->dbias, stream);
    if (e != hipSuccess) return fail((int)e, "shared-bias backward: launch of the reduction failed: %s", hipGetErrorString(e));
  }
  g_err[0] = 0;
  return 0;
}

int fl_attn_bwd_static(const fl_attn_bwd_params* b, void* stream) {
  if (!b) return fail(FL_ERR_NULL, "params is null");
  fl_attn_bwd_params c = *b;
  const fl_attn_params* p = &b->fwd;
  if (p->B <= 0 || p->Hq <= 0 || p->Lq <= 0) return fail(FL_ERR_SHAPE, "sizes must be positive");
  // layout of the static scratch: the row sums (B * Hq * Lq floats, rounded up to 256 bytes), then the document table
  const uint64_t delta_bytes = ((uint64_t)p->B * p->Hq * p->Lq * sizeof(float) + 255) / 256 * 256;
  const uint64_t table_bytes = fl_bwd_workspace_bytes(p);
  if (delta_bytes + table_bytes > kStaticScratchBytes)
    return fail(FL_ERR_WORKSPACE,
                "fl_attn_bwd_static: this call needs %llu bytes of scratch (4 per query row of every head, plus 16 per 32 "
                "positions of every batch row under a document mask), the library's static scratch holds %llu; use "
                "fl_attn_bwd with caller-provided delta and workspace",
                (unsigned long long)(delta_bytes + table_bytes), (unsigned long long)kStaticScratchBytes);
  void* ptr = nullptr;
  int rc = static_scratch_ptr(&ptr);
  if (rc) return rc;
  c.delta = static_cast<float*>(ptr);
  c.fwd.workspace = table_bytes ? static_cast<unsigned char*>(ptr) + delta_bytes : nullptr;
  c.fwd.workspace_bytes = table_bytes;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool capturing = stream_is_capturing(s);
  int dev = -1;
  if (!capturing) {
    rc = static_scratch_acquire(s, &dev);
    if (rc) return rc;
  }
  rc = fl_attn_bwd(&c, stream);
  if (!capturing && dev >= 0) static_scratch_release(s, dev);
  return rc;
}

}  // extern "C"
