// engine.hip -- MI355X (gfx950) engine for uSAP's partition hot path.
//
// Device state per graph: CSR/CSC (int64 offsets, int32 ids), labels int32[N],
// block degrees int32[B], and the interblock edge-count matrix M as one "block
// row" per block a holding both orientations: the slot of key b carries
// o = M[a][b] (edges a -> b) and i = M[b][a] (edges b -> a), so every M[a][b]
// is stored twice (as o in row a and as i in row b) and one probe of row a
// answers both the row and the column lookup of a block pair.  Rows live in
// one slab pool:
//   row a occupies slots [off[a], off[a]+cap[a]);
//   cap[a] == B  -> direct-mapped row (slot = key), used when a hashed row
//                   would need >= B slots (dense regime, small B);
//   cap[a] <  B  -> open-addressing hash (power of two, linear probing);
//                   keys (-1 = empty) and counts (o, i) are arrays of their
//                   own, so eight keys of a chain are two loads, and one 64-bit
//                   atomic updates both counts.
// Keys are never deleted inside a sweep (counts may drop to 0).  Rows too long
// to read whole keep kNBK bucket sums (sum of o + i per key range) for the
// two-level inverse-CDF pick over the combined weights M[a][b] + M[b][a].  An
// increment that finds no free slot near its key during nodal batches is
// parked in an overflow buffer; between two batches k_grow takes the rows that
// have parked increments, and every few batches those marked as past 1/slack of
// their slab, compacts them in place or moves them to a larger slab at the
// pool's tail, and replays the parked increments.
// The host rebuilds M from the labels only when the pool runs out.
//
// Kernels (one wavefront of 64 lanes per proposal item):
//   k_hist / k_hist_sum : M build from labels (graph_parallel.hpp:703-759) for
//        few blocks, by LDS histograms
//   k_degrees / k_caps / k_fill / k_insert_pairs / k_node_lists / k_build_* /
//        k_bucket_sums : for more, by sorted block pairs or row by row
//   k_merge_rows / k_merge_list / k_merge : K merge proposals per block + best per block
//        (graph_parallel.hpp:349-368, :761-988), one wavefront per block, or
//        one workgroup with a wavefront per proposal
//   k_carry_* : the greedy carry-out (graph_parallel.hpp:1225-1279)
//   k_begin / k_draw / k_finish : a sweep's state, random words and result
//   k_nodal   : one nodal proposal per node against the frozen M
//        (graph_parallel.hpp:990-1222), one wavefront per node
//   k_apply   : accepted moves -> M, degrees (atomics) and labels; equals
//        the reference's full rebuild (graph_parallel.hpp:438-443); its
//        block 0 runs the sweep's update step and convergence test
//        (graph_parallel.hpp:433-458) from k_nodal's per-workgroup shares,
//        so a whole sweep runs without the host
//   k_grow    : row growth / compaction and overflow replay between batches;
//        acts on the batch's error and rebuild flags
//   k_entropy : data_S over all non-zeros (graph_parallel.hpp:1281-1319)
//
// The nodal and apply kernels are latency bound (a few hundred bytes per node
// at random rows of M); each wavefront keeps all loads of one step in flight
// at once -- list ids, then labels, then rows, then the first probes of every
// lookup -- instead of paying one memory latency per lookup.
//
// dS uses the factorised form of the reference's term sums: terms whose count
// and degrees do not change cancel exactly in integer arithmetic, so a nodal
// proposal costs O(distinct neighbour blocks) lookups and a merge proposal
// O(min row length) lookups, instead of the reference's O(B) scans.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <numeric>
#include <rocprim/rocprim.hpp>
#include <string>
#include <thread>
#include <vector>

#include "engine_internal.hpp"
#include "usap.h"
#include "usap_common.hpp"

using usap::i128;
using usap::u128;

namespace {

constexpr int kWave = 64;
constexpr int kNodalWaves = 4;           // wavefronts per workgroup in k_nodal / k_apply
constexpr int kMergeWaves = 4;           // wavefronts per workgroup in k_merge
constexpr int kNBK = 512;                // bucket sums per block row
constexpr int kLookupRatio = 8;          // a hashed slab this many times a bucket is looked up per key
constexpr int kScr = 1024;               // per-wavefront LDS scratch (ints) for one bucket
constexpr int kMergeMany = 16;           // and for at most kMergeFew blocks
constexpr int32_t kMergeFew = 512;
constexpr int32_t kMergeGrid = 8192;     // workgroups of k_merge over a list
constexpr int kDegLds = 1024;            // k_degrees privatises its counters for B <= this
constexpr int kHistB = 256;              // M is built by histograms in LDS up to here
constexpr int kEntropyBlocks = 4096;  // k_entropy grid at most
// Partials of the allocation-free MDL (usap_entropy_noalloc): 2 words per
// k_entropy workgroup, 64 KiB per GPU.
static __device__ __align__(256) long scratch[2 * kEntropyBlocks];
constexpr int kNumSnap = 4;

enum : int32_t {
  kFlagFull = 2,      // an insertion found no free slot (increment lost)
  kFlagMissing = 4,   // a decrement did not find its key (bug)
  kFlagNegative = 8,  // a negative count reached an entropy term (bug)
};

struct Status {
  int32_t flags;  // kFlag* raised by the running batch
  int32_t pad[3];
};

// Device state of one nodal sweep (the reference's `update` task,
// graph_parallel.hpp:433-458, run by block 0 of each batch's k_apply).
struct Sweep {
  unsigned long long cum_lo, cum_hi;  // exact cumulative dS of the sweep (int128)
  unsigned long long stream0;         // random stream of the sweep's first batch (pre-drawn: node 0's draw)
  double S;                           // running S: S += dS_sum after every batch
  double mean;                        // moving average of earlier sweeps' dS
  double thr;                         // delta_entropy_threshold1 or 2
  double dS_last;                     // dS_sum after the last batch (itr_delta_entropy[itr])
  unsigned long long moves;
  unsigned long long nodal_bytes, apply_bytes;
  int32_t cum_inf;  // an accepted dS was -inf
  int32_t check;    // itr >= window - 1: the convergence test is active
  int32_t stop;     // 0 run, 1 converged, 2 M needs a rebuild, 3 inconsistent M
  int32_t done;     // batches executed
  int32_t flags;    // OR of the batches' flags
  int32_t stop_n;   // stop as the running batch's k_nodal saw it (0: the batch runs)
};

// A word in the host's memory that a call's last kernel sets once its results
// are there (p null: none).
struct HostWord {
  int32_t* p;
  int32_t value;
};
__device__ __forceinline__ void host_done(const HostWord& w) {
  if (w.p) {
    __threadfence_system();
    __hip_atomic_store(w.p, w.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

struct GraphView {
  int32_t N;
  const int64_t* out_ptr;
  const int32_t* out_idx;
  const int32_t* out_w;
  const int64_t* in_ptr;
  const int32_t* in_idx;
  const int32_t* in_w;
};

// The two counts of a block pair (a, b): o = M[a][b], i = M[b][a]; 8-byte
// aligned, one 64-bit atomic adds to both.
struct __align__(8) Cnt {
  int32_t o, i;
};

// M as block rows, as seen by kernels.
struct MView {
  const int64_t* off;
  const int32_t* cap;
  int32_t* gmark;  // [B]: > 0: k_grow looks at the row (kMarked, room_mark)
  int32_t* key;    // row slabs: keys (-1 empty; unused in a direct row) ...
  Cnt* cnt;        // ... and the counts of each slot
  int32_t* bs;     // [B][kNBK]: sum of the row's o + i per key bucket (rows with row_sums)
  int32_t* gpend;  // [B]: increments of the row waiting in the overflow buffer
  int32_t* ovf;    // [4][ovf_cap]: (row, key, do, di) increments that found no free slot
  int32_t ovf_cap;
  struct GrowState* gst;
  int32_t B;
  int32_t bshift;  // bucket of key k = k >> bshift
  int32_t stride;  // slots from a row to the next while all are direct (direct_stride)
  int32_t slack;   // slab_slack: a hashed row grows past 1/slack load
};

// Rows to grow between two batches; slabs for grown rows come from the free
// tail of the pool.
constexpr int kGrowBlocks = 768;  // k_grow's grid: three workgroups of 52 KB of LDS per CU

// A k_grow workgroup's piece of the free tail: slots [pos, end), their counts 0;
// and what the workgroup did since the engine was created.
struct GrowChunk {
  long long pos, end;
  unsigned long long grows;        // rows grown or compacted
  unsigned long long compactions;  // of them in place
};

struct GrowState {
  int32_t nospace;            // the pool ran out: the host rebuilds M
  int32_t ovf_n;              // entries in the overflow buffer
  unsigned long long used;    // pool slots in use
  unsigned long long full;    // insertions that found no free slot
  unsigned long long nospace_events;
  GrowChunk chunk[kGrowBlocks];
};

__device__ __forceinline__ uint32_t hash32(int32_t b) {
  uint32_t x = (uint32_t)b * 0x9E3779B1u;
  return x ^ (x >> 15);
}

__device__ __forceinline__ int32_t ld_relaxed(int32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Slab of one row: offset and capacity.
struct Row {
  int64_t o;
  int32_t c;
};

// kD: every row of M is direct (the host knows it from the rebuild), so row a
// is the first B of the a-th `stride` slots of the pool: no row header to load
// before a lookup, no key, no probing.
template <bool kD = false>
__device__ __forceinline__ Row m_row(const MView& m, int32_t a) {
  return kD ? Row{(int64_t)a * m.stride, m.B} : Row{m.off[a], m.cap[a]};
}

// A lookup's first probe: the slot with the key and counts found there.  The
// callers issue several probes before resolving any, so a wavefront has all
// of its lookups in flight at once instead of one memory latency per lookup.
struct Probe {
  uint32_t h;  // slot within the row
  int32_t k;
  Cnt c;
};

template <bool kD = false>
__device__ __forceinline__ uint32_t m_home(const MView& m, Row R, int32_t b) {
  return kD || R.c == m.B ? (uint32_t)b : hash32(b) & (uint32_t)(R.c - 1);
}

template <bool kD = false>
__device__ __forceinline__ Probe m_probe(const MView& m, Row R, int32_t b) {
  Probe p;
  p.h = m_home<kD>(m, R, b);
  p.k = kD || R.c == m.B ? b : m.key[R.o + p.h];
  p.c = m.cnt[R.o + p.h];
  return p;
}

// Linear probing on from slot `slot` of a hashed row after a collision there.
__device__ __forceinline__ Cnt m_value_more(const MView& m, Row R, int32_t b, uint32_t h) {
  const uint32_t mask = (uint32_t)R.c - 1;
  for (int32_t probe = 1; probe < R.c; ++probe) {
    h = (h + 1) & mask;
    const int32_t k = m.key[R.o + h];
    if (k == b) return m.cnt[R.o + h];
    if (k < 0) return Cnt{0, 0};
  }
  return Cnt{0, 0};
}

// (M[a][b], M[b][a]) from the first probe p of key b in row R of a.
template <bool kD = false>
__device__ __forceinline__ Cnt m_value(const MView& m, Row R, int32_t b, const Probe& p) {
  if (kD || p.k == b) return p.c;
  if (p.k < 0) return Cnt{0, 0};
  return m_value_more(m, R, b, p.h);
}

// (M[a][b], M[b][a])
__device__ __forceinline__ Cnt m_get(const MView& m, int32_t a, int32_t b) {
  const Row R = m_row(m, a);
  return m_value(m, R, b, m_probe(m, R, b));
}

// o += dout, i += din with one 64-bit atomic.  Exact as long as neither count
// leaves [0, 2^31) at any point, which holds for every caller: a decrement
// only removes edges the count held when the kernel started.
__device__ __forceinline__ void cnt_add(Cnt* q, int32_t dout, int32_t din) {
  const long long d = (long long)din * 4294967296LL + (long long)dout;
  atomicAdd(reinterpret_cast<unsigned long long*>(q), (unsigned long long)d);
}

constexpr uint32_t kMaxWalk = 32;  // probes before a nodal-batch increment is parked
constexpr uint32_t kMarkWalk = 4;  // slots from home at which a new key marks its row for k_grow
// MView::gmark: k_grow looks at rows where it is positive.  A small hashed row's
// is 0 or kMarked; one of more than kScanRow slots (whose long chains would
// mark it in nearly every batch, and whose slab takes a workgroup to count)
// counts new keys up from minus the keys that fit 1/slack load (room_mark).
constexpr int32_t kMarked = 1 << 30;
constexpr int32_t kScanRow = 512;  // slots up to which a hashed slab is read whole
__device__ __forceinline__ int32_t room_mark(int32_t keys, int32_t c, int32_t slack) {
  return c > kScanRow ? min(0, keys - c / slack) : 0;
}

// Whether a row of capacity c keeps bucket sums.  The pick reads a direct row
// of at most kNBK keys and a hashed slab of at most kScanRow slots whole (in
// one round of loads, as the sums would be), so those rows' counts cost
// k_apply one atomic less per update and a rebuild 2 KB less per row.
__device__ __forceinline__ bool row_sums(const MView& m, int32_t c) {
  return c == m.B ? m.B > kNBK : c > kScanRow;
}

// The keys of kWin slots of hashed row R from slot h on are read at once (two
// 16-byte loads; one memory latency for most probe chains); returns the first
// that holds b or is empty, with its slot in h, or, if none does, the
// window's last.  The window ends at the slab's end at the latest.  Keys only
// go from empty to set, so a plain load is as good as a relaxed atomic one.
constexpr int kWin = 8;
typedef int32_t Key4 __attribute__((ext_vector_type(4), aligned(4)));  // 4-byte aligned
__device__ __forceinline__ int32_t m_window(const MView& m, Row R, int32_t b, uint32_t& h) {
  const uint32_t w0 = min(h, (uint32_t)R.c - kWin);  // hashed rows hold >= 32 slots
  const Key4* w = reinterpret_cast<const Key4*>(m.key + R.o + w0);
  const Key4 lo = w[0], hi = w[1];
  const int32_t k[kWin] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  int32_t kk = k[kWin - 1];
  uint32_t pos = w0 + kWin - 1;
#pragma unroll
  for (int q = kWin - 2; q >= 0; --q) {  // the first slot from h on that ends the chain
    if (w0 + q >= h && (k[q] == b || k[q] < 0)) {
      kk = k[q];
      pos = w0 + q;
    }
  }
  h = pos;
  return kk;
}

// A window of row R for key b in flight (direct: only h).
struct Window {
  Key4 lo, hi;
  uint32_t w0, home;
};

__device__ __forceinline__ Window win_issue(const MView& m, Row R, int32_t b, bool direct) {
  Window w;
  if (direct) {
    w.w0 = w.home = (uint32_t)b;
    w.lo = w.hi = Key4{b, b, b, b};
    return w;
  }
  w.home = hash32(b) & ((uint32_t)R.c - 1);
  w.w0 = min(w.home, (uint32_t)R.c - kWin);
  const Key4* k = reinterpret_cast<const Key4*>(m.key + R.o + w.w0);
  w.lo = k[0];
  w.hi = k[1];
  return w;
}

// The slot within the row that ends key b's probe chain (found: it holds b), or
// the window's last one, whose other key k is then returned >= 0.
__device__ __forceinline__ uint32_t win_end(const Window& w, int32_t b, bool direct, int32_t& k) {
  if (direct) {
    k = b;
    return w.home;
  }
  const int32_t kk[kWin] = {w.lo[0], w.lo[1], w.lo[2], w.lo[3], w.hi[0], w.hi[1], w.hi[2], w.hi[3]};
  k = kk[kWin - 1];
  uint32_t pos = w.w0 + kWin - 1;
#pragma unroll
  for (int q = kWin - 2; q >= 0; --q)
    if (w.w0 + q >= w.home && (kk[q] == b || kk[q] < 0)) {
      k = kk[q];
      pos = w.w0 + q;
    }
  return pos;
}

// Where m_add_at starts for key b in row R: the end of its probe chain, or as
// far along it as one window reaches.
template <bool kD = false>
__device__ __forceinline__ int32_t m_first_key(const MView& m, Row R, int32_t b, int64_t& slot) {
  if (kD || R.c == m.B) {
    slot = R.o + b;
    return b;
  }
  uint32_t h = hash32(b) & ((uint32_t)R.c - 1);
  const int32_t k = m_window(m, R, b, h);
  slot = R.o + h;
  return k;
}

// M[a][b] += dout and M[b][a] += din in row R of a (negative only for a key
// that exists), given the key k read at the first probed slot `slot`.  Keys
// only go from empty to set, so an earlier read is a valid first read: a
// stale "empty" makes the claim fail and return the key that is there.
// kBatch (k_apply) also updates the row's bucket sum, and leaves a crowded row
// to k_grow (by a mark, or a parked increment) instead of flagging a rebuild.
template <bool kBatch, bool kD = false>
__device__ __forceinline__ void m_add_at(const MView& m, int32_t a, Row R, int32_t b, int32_t dout,
                                         int32_t din, int64_t slot, int32_t k, int32_t* flags) {
  if (kBatch && dout + din != 0 && row_sums(m, R.c))
    atomicAdd(&m.bs[(int64_t)a * kNBK + (b >> m.bshift)], dout + din);
  if (kD || R.c == m.B || k == b) {
    cnt_add(&m.cnt[slot], dout, din);
    return;
  }
  const bool dec = dout < 0 || din < 0;
  const int64_t o = R.o;
  const int32_t c = R.c;
  const uint32_t mask = (uint32_t)c - 1, home = hash32(b) & mask;
  uint32_t h = (uint32_t)(slot - o);
  // an increment whose key is still absent after kMaxWalk slots is parked
  // (k_grow grows the row) rather than walking a crowded row
  const uint32_t most = kBatch && !dec ? min(kMaxWalk, (uint32_t)c) : (uint32_t)c;
  for (;;) {
    if (k < 0) {
      if (dec) {
        atomicOr(flags, kFlagMissing);
        return;
      }
      k = atomicCAS(&m.key[o + h], -1, b);
      if (k == -1) {
        cnt_add(&m.cnt[o + h], dout, din);
        // a new key kMarkWalk slots or more from home: the row is (or will
        // soon be) past 1/slack load; a large row's new keys are counted
        if (kBatch && c > kScanRow)
          atomicAdd(&m.gmark[a], 1);
        else if (kBatch && ((h - home) & mask) >= kMarkWalk)
          m.gmark[a] = kMarked;
        return;
      }
    }
    if (k == b) {
      cnt_add(&m.cnt[o + h], dout, din);
      return;
    }
    const uint32_t walked = ((h - home) & mask) + 1;  // slots found taken
    if (walked >= most) break;
    h = (h + 1) & mask;
    k = m_window(m, R, b, h);
    if (((h - home) & mask) < walked) break;  // past the whole slab
  }
  if (kBatch && !dec) {  // no free slot near: park the increment until k_grow has grown the row
    const int32_t i = atomicAdd(&m.gst->ovf_n, 1);
    if (i < m.ovf_cap) {
      m.ovf[i] = a;
      m.ovf[m.ovf_cap + i] = b;
      m.ovf[2 * m.ovf_cap + i] = dout;
      m.ovf[3 * m.ovf_cap + i] = din;
      atomicAdd(&m.gpend[a], 1);  // k_grow grows every row with parked increments
      m.gmark[a] = kMarked;
      return;
    }
  }
  atomicOr(flags, dec ? kFlagMissing : kFlagFull);
}

// M[a][b] += dout, M[b][a] += din in row a (M builds)
__device__ __forceinline__ void m_add(const MView& m, int32_t a, int32_t b, int32_t dout,
                                      int32_t din, int32_t* flags) {
  const Row R = m_row(m, a);
  int64_t slot;
  const int32_t k = m_first_key(m, R, b, slot);
  m_add_at<false>(m, a, R, b, dout, din, slot, k, flags);
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// Draw d of a pre-drawn uniform stream: its four words, slot order as the
// Philox outputs they replace.
__device__ __forceinline__ void predrawn(const uint64_t* uni, uint64_t d, uint64_t x[4]) {
  const ulonglong2* q = reinterpret_cast<const ulonglong2*>(uni + 4 * d);
  const ulonglong2 a = q[0], b = q[1];
  x[0] = a.x;
  x[1] = a.y;
  x[2] = b.x;
  x[3] = b.y;
}

// Orders this wavefront's earlier table writes before its later reads.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// v of lane l (l the same in every lane)
__device__ __forceinline__ long read_lane(long v, int l) {
  const unsigned long long u = (unsigned long long)v;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
  return (long)(((unsigned long long)hi << 32) | lo);
}

// v moved across lanes by one DPP step (a register move: no LDS round trip as
// a shuffle makes); lanes of rows outside kRows, or with no source, get 0.
template <int kCtrl, int kRows = 0xf>
__device__ __forceinline__ long dpp_move(long v) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(unsigned long)v, kCtrl, kRows, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), kCtrl, kRows, 0xf, true);
  return (long)(((unsigned long)(uint32_t)hi << 32) | (uint32_t)lo);
}

constexpr int kDppShr1 = 0x111, kDppShr2 = 0x112, kDppShr4 = 0x114, kDppShr8 = 0x118;
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E;                // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int kDppHalfMirror = 0x141, kDppMirror = 0x140;      // within 8, within 16 lanes
constexpr int kDppBcast15 = 0x142, kDppBcast31 = 0x143;        // last lane of the row(s) below

// Sum over the wavefront's 64 lanes, all of them active (the callers' flow is
// uniform): row sums by mirrors, then row to row; lane 63 holds the total.
__device__ __forceinline__ long wave_sum(long v) {
  v += dpp_move<kDppXor1>(v);
  v += dpp_move<kDppXor2>(v);
  v += dpp_move<kDppHalfMirror>(v);
  v += dpp_move<kDppMirror>(v);
  v += dpp_move<kDppBcast15, 0xa>(v);
  v += dpp_move<kDppBcast31, 0xc>(v);
  return read_lane(v, kWave - 1);
}

__device__ __forceinline__ i128 wave_sum128(i128 v) {
  unsigned long lo = (unsigned long)(u128)v;
  long hi = (long)(v >> 64);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const unsigned long lo2 = __shfl_xor(lo, off);
    const long hi2 = __shfl_xor(hi, off);
    const unsigned long s = lo + lo2;
    hi = hi + hi2 + (s < lo ? 1 : 0);
    lo = s;
  }
  return (i128)(((u128)(unsigned long)hi << 64) | (u128)lo);
}

// Inclusive scan over the wavefront's 64 lanes, all of them active.
__device__ __forceinline__ long wave_incl_scan(long v) {
  v += dpp_move<kDppShr1>(v);
  v += dpp_move<kDppShr2>(v);
  v += dpp_move<kDppShr4>(v);
  v += dpp_move<kDppShr8>(v);
  v += dpp_move<kDppBcast15, 0xa>(v);
  v += dpp_move<kDppBcast31, 0xc>(v);
  return v;
}

template <int kCtrl, int kRows = 0xf>
__device__ __forceinline__ uint32_t dpp_move32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, kRows, 0xf, true);
}

__device__ __forceinline__ uint32_t wave_incl_scan32(uint32_t v) {
  v += dpp_move32<kDppShr1>(v);
  v += dpp_move32<kDppShr2>(v);
  v += dpp_move32<kDppShr4>(v);
  v += dpp_move32<kDppShr8>(v);
  v += dpp_move32<kDppBcast15, 0xa>(v);
  v += dpp_move32<kDppBcast31, 0xc>(v);
  return v;
}

__device__ __forceinline__ uint32_t read_lane32(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}

__device__ __forceinline__ uint32_t wave_sum32(uint32_t v) {
  return read_lane32(wave_incl_scan32(v), kWave - 1);
}

// floor(x * W / 2^64) for W < 2^32, as usap::idx_of
__device__ __forceinline__ uint32_t idx32(uint64_t x, uint32_t W) {
  const uint64_t hi = (x >> 32) * W, lo = (x & 0xffffffffull) * W;
  return (uint32_t)((hi + (lo >> 32)) >> 32);
}

// A sum of terms m * L, |m| < 2^31 (a count, degree or sum of them), L a lambda
// or lambda(m) - lambda(x) - lambda(y), |L| < 2^54: each L is split at bit 24 and
// the two products are summed apart, value = h * 2^24 + l, so a term is two 32-bit
// multiply-adds (an int128 product of 64-bit operands is about ten, at a quarter
// of the ALU's rate).  Exact, with W < 2^31 the total weight and lambda <= A =
// ln(2^31) * 2^48 < 2^52.43: out-edges of two blocks weigh at most W together, and
// so do their in-edges.  With C in the corner of the two, a dS has on each side,
// before and after, at most 2 (W - C) in its rows' other counts at A each, C in the
// corner at up to 2 A each, and 2 (W - C) in degree terms at A each (a merge: the
// same, its counts in the overlap).  That is below 4 W A a side, 8 W A in all, and
// an MDL's three sums are below 3 W A: |h| < 2^62.5, and |l| < 8 W 2^24 = 2^58.  With the
// wavefront sums by DPP and a dS's 16 uniform terms spread over 16 lanes it took
// k_nodal from 126 to 90 VGPRs, a resumed chain at N = 50000 from 2.60 to 2.19 ms
// and the N = 20000 partition from 25.5 to 22.5 ms.
constexpr int kAccSplit = 24;
struct Acc {
  long h, l;
};

__device__ __forceinline__ void acc_add(Acc& a, int32_t m, int64_t L) {
  a.h += (long)m * (long)(int32_t)(L >> kAccSplit);
  a.l += (long)m * (long)((int32_t)L & ((1 << kAccSplit) - 1));
}

__device__ __forceinline__ i128 acc_value(const Acc& a) {
  return (i128)(((u128)(i128)a.h << kAccSplit) + (u128)(i128)a.l);
}

// The terms read the lambda table unconditionally (lambda of m <= 0 reads
// lam[0] = 0) and select the result, so the table loads of a whole dS are
// issued together: a load under `if (m > 0)` would sit in its own branch and
// wait for every earlier term's loads first.
__device__ __forceinline__ int64_t lam_of(const int64_t* lam, int32_t m) {
  return lam[max(m, 0)];
}

// - m * lambda(m): one L term (0 for m <= 0)
__device__ __forceinline__ void sub_L(Acc& a, const int64_t* lam, int32_t m) {
  acc_add(a, -max(m, 0), lam_of(lam, m));
}

// sign * m * lambda(d): one degree-factor term; inf when m > 0 and d == 0
__device__ __forceinline__ void add_P(Acc& a, const int64_t* lam, int sign, int32_t m, int32_t d,
                                      bool& inf) {
  inf = inf || (m > 0 && d <= 0);
  acc_add(a, sign * max(m, 0), lam_of(lam, d));
}

// sign * T(m, x, y) = m*(lambda(m)-lambda(x)-lambda(y)); inf when m > 0 and x*y == 0
__device__ __forceinline__ void add_T(Acc& a, const int64_t* lam, int sign, int32_t m, int32_t x,
                                      int32_t y, bool& inf) {
  const int64_t Lm = lam_of(lam, m), Lx = lam_of(lam, x), Ly = lam_of(lam, y);
  const bool bad = x <= 0 || y <= 0;
  inf = inf || (m > 0 && bad);
  acc_add(a, bad ? 0 : sign * max(m, 0), Lm - Lx - Ly);
}

// per-lane part of sum_{lo <= key <= x, key != excl} M[a][key] + M[key][a]
// over row (o, c) of a
__device__ __forceinline__ long count_range_lane(const MView& m, int64_t o, int32_t c, int32_t lo,
                                                 int32_t x, int32_t excl) {
  const int lane = lane_id();
  long acc = 0;
  if (c == m.B) {
    for (int32_t i = lo + lane; i <= x; i += kWave)
      if (i != excl) acc += (long)m.cnt[o + i].o + m.cnt[o + i].i;
  } else {
    for (int32_t j = lane; j < c; j += kWave) {
      const int32_t k = m.key[o + j];
      const Cnt q = m.cnt[o + j];
      if (k >= lo && k <= x && k != excl) acc += (long)q.o + q.i;
    }
  }
  return acc;
}

// scr[k - lo] += M[a][k] + M[k][a] for lo <= k < hi, from row R of a: a
// direct row is read at keys [lo, hi), a hashed row's slab is scanned eight
// slots per lane at a time (all loads of a pass in flight before the LDS adds).
__device__ __forceinline__ void gather_row(const MView& m, Row R, int32_t lo, int32_t hi,
                                           int32_t* scr, long& bytes) {
  const int lane = lane_id();
  if (R.c == m.B) {
    for (int32_t i = lane; i < hi - lo; i += kWave) {
      const Cnt q = m.cnt[R.o + lo + i];
      atomicAdd(&scr[i], q.o + q.i);
    }
    bytes += 8 * (long)(hi - lo);
    return;
  }
  for (int32_t base = 0; base < R.c; base += 8 * kWave) {
    int32_t k[8], v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int32_t j = base + q * kWave + lane;
      k[q] = -1;
      v[q] = 0;
      if (j < R.c) {
        const Cnt x = m.cnt[R.o + j];
        k[q] = m.key[R.o + j];
        v[q] = x.o + x.i;
      }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (k[q] >= lo && k[q] < hi && v[q] != 0) atomicAdd(&scr[k[q] - lo], v[q]);
  }
  bytes += 12 * (long)R.c;
}

// scr[k - lo] = M[a][k] + M[k][a] for lo <= k < hi from hashed row R of a, by
// looking each key up: four keys per lane at a time, every pending walk of
// the wavefront advancing one slot per step with all its loads in flight.  A
// walk ends at its key or at an empty slot, and after R.c slots at the latest
// (a full slab).  For a slab much larger than the bucket this reads a few
// slots per key instead of the whole slab.
__device__ __forceinline__ void lookup_bucket(const MView& m, Row R, int32_t lo, int32_t hi,
                                              int32_t* scr, long& bytes) {
  const int lane = lane_id();
  const uint32_t mask = (uint32_t)R.c - 1;
  for (int32_t base = lo; base < hi; base += 4 * kWave) {
    uint32_t h[4];
    int32_t wv[4];
    uint32_t pend = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int32_t key = base + q * kWave + lane;
      h[q] = hash32(key) & mask;
      wv[q] = 0;
      if (key < hi) pend |= 1u << q;
    }
    for (int32_t step = 0; step < R.c && __ballot(pend != 0); ++step) {
      int32_t k[4];
      Cnt x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if ((pend >> q) & 1) {
          k[q] = m.key[R.o + h[q]];
          x[q] = m.cnt[R.o + h[q]];
        }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bytes += 16 * (long)__popcll(__ballot((pend >> q) & 1));
        if (!((pend >> q) & 1)) continue;
        const int32_t key = base + q * kWave + lane;
        if (k[q] == key) {
          wv[q] = x[q].o + x[q].i;
          pend &= ~(1u << q);
        } else if (k[q] < 0) {
          pend &= ~(1u << q);
        } else {
          h[q] = (h[q] + 1) & mask;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int32_t key = base + q * kWave + lane;
      if (key < hi) scr[key - lo] = wv[q];
    }
  }
}

// A row's weight per key bucket, `per` consecutive buckets per lane (buckets
// past the last key are 0).
constexpr int kBkLane = kNBK / kWave;
struct Sums {
  int per;
  uint32_t w[kBkLane];
};

// Of a row that keeps bucket sums (row_sums), or a direct row of at most kNBK
// keys (a bucket is one key: its counts).
__device__ __forceinline__ Sums load_sums(const MView& M, int32_t u, Row R) {
  static_assert(kBkLane == 8, "two 16-byte loads per lane");
  const int lane = lane_id();
  if (M.B <= kNBK) {
    Sums S{(M.B + kWave - 1) / kWave, {0, 0, 0, 0, 0, 0, 0, 0}};
#pragma unroll
    for (int q = 0; q < kBkLane; ++q)
      if (q < S.per && lane * S.per + q < M.B) {
        const Cnt x = M.cnt[R.o + lane * S.per + q];
        S.w[q] = (uint32_t)x.o + (uint32_t)x.i;
      }
    return S;
  }
  const uint4* p = reinterpret_cast<const uint4*>(M.bs + (int64_t)u * kNBK) + 2 * lane;
  const uint4 a = p[0], b = p[1];
  return Sums{kBkLane, {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
}

// The bucket holding unit t; t becomes the unit within it.
__device__ __forceinline__ int32_t pick_bucket(const Sums& S, uint32_t& t) {
  const int lane = lane_id();
  uint32_t own = 0;
#pragma unroll
  for (int q = 0; q < kBkLane; ++q) own += S.w[q];
  const uint32_t inc = wave_incl_scan32(own);
  const unsigned long long past = __ballot(inc > t);
  const int f = past ? __ffsll(past) - 1 : kWave - 1;
  int j = 0;
  const uint32_t rest = t - (inc - own);  // in lane f: the unit within its buckets
  uint32_t before = 0;
#pragma unroll
  for (int q = 0; q < kBkLane - 1; ++q) {
    before += S.w[q];
    if (rest >= before) j = q + 1;
  }
  before = 0;
#pragma unroll
  for (int q = 0; q < kBkLane - 1; ++q)
    if (q < j) before += S.w[q];
  t = read_lane32(rest - before, f);
  return (int32_t)read_lane32((uint32_t)(lane * S.per + j), f);
}

// The t-th unit among `width` weights, weight(i) for 0 <= i < width in lane i
// % 64, 512 of them in flight at a time; width - 1 if there is none.
template <typename F>
__device__ __forceinline__ int32_t pick_scan(int32_t width, uint32_t t, F weight) {
  const int lane = lane_id();
  for (int32_t base = 0; base < width; base += 8 * kWave) {
    uint32_t v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int32_t i = base + q * kWave + lane;
      v[q] = i < width ? weight(i) : 0;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (base + q * kWave >= width) break;
      const uint32_t c = wave_incl_scan32(v[q]);
      const unsigned long long hit = __ballot(c > t);
      if (hit) return base + q * kWave + __ffsll(hit) - 1;
      t -= read_lane32(c, kWave - 1);
    }
  }
  return width - 1;
}

// Inverse-CDF pick over the combined weights M[u][i] + M[i][u] (block row
// u: o + i), ascending i, skipping i == excl: the first i whose running sum
// exceeds t (graph_parallel.hpp:849-850 / :1061-1062 with exact integer
// weights; a row's weights sum to less than 2^32).  The caller guarantees t <
// total weight.  Two levels: the weight per key bucket locates the bucket [lo,
// hi), then the bucket's keys are searched.  `pre`: the row's sums, loaded
// ahead (a direct row's), or null.
//   direct row: sums as load_sums; one load per key of the bucket.
//   hashed, at most kScanRow slots: the slab is read once, eight slots a lane,
//     and histogrammed over the buckets in the wavefront's LDS scratch `scr`
//     (scr_cap >= kNBK ints), then the bucket's entries gathered there.
//   larger hashed: its bucket sums; then the bucket's weights gathered into scr
//     by a scan of the slab, or, when it holds kLookupRatio times the bucket's
//     keys or more, by looking each key up (a whole-slab scan of a 16384-slot
//     row took one wavefront ~120 us).
template <bool kD>
__device__ __forceinline__ int32_t select_combined(const MView& M, int32_t u, uint32_t t,
                                                   int32_t excl, const Sums* pre, int32_t* scr,
                                                   int32_t scr_cap, long& bytes) {
  const int lane = lane_id();
  const int32_t B = M.B;
  const int sh = M.bshift;
  const int32_t nbk = ((B - 1) >> sh) + 1;
  const Row RM = m_row<kD>(M, u);
  const bool direct = kD || RM.c == B;
  const bool small = !direct && !row_sums(M, RM.c);
  Sums S;
  if (small) {
    constexpr int kQ = kScanRow / kWave;
    for (int32_t i = lane; i < kNBK; i += kWave) scr[i] = 0;
    int32_t key[kQ];
    uint32_t wt[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int32_t j = q * kWave + lane;
      key[q] = -1;
      wt[q] = 0;
      if (j < RM.c) {
        key[q] = M.key[RM.o + j];
        const Cnt x = M.cnt[RM.o + j];
        wt[q] = (uint32_t)x.o + (uint32_t)x.i;
      }
    }
    wave_fence();
#pragma unroll
    for (int q = 0; q < kQ; ++q)
      if (key[q] >= 0 && key[q] != excl && wt[q]) atomicAdd(&scr[key[q] >> sh], (int32_t)wt[q]);
    wave_fence();
    S.per = kBkLane;
#pragma unroll
    for (int q = 0; q < kBkLane; ++q) S.w[q] = (uint32_t)scr[lane * kBkLane + q];
    bytes += 12 + 12 * (long)RM.c;
  } else {
    S = pre ? *pre : load_sums(M, u, RM);
    bytes += 12 + 4 * (long)nbk;
    if (excl >= 0) {
      const Cnt x = m_value<kD>(M, RM, excl, m_probe<kD>(M, RM, excl));
      bytes += 12;
#pragma unroll
      for (int q = 0; q < kBkLane; ++q)
        if (lane * S.per + q == excl >> sh && q < S.per) S.w[q] -= (uint32_t)x.o + (uint32_t)x.i;
    }
  }
  const int32_t jb = min(pick_bucket(S, t), nbk - 1);
  const int32_t lo = jb << sh;
  const int32_t hi = min(B, lo + (1 << sh));
  const int32_t width = hi - lo;
  // a bucket of one key (every bucket when B <= kNBK): the bucket's sum is
  // that key's weight, so the bucket is the pick (the scans below would
  // return lo too, also for the excluded key's emptied bucket)
  if (width == 1) return lo;
  if (direct) {
    bytes += 8 * (long)width;
    return lo + pick_scan(width, t, [&](int32_t i) -> uint32_t {
             if (lo + i == excl) return 0;
             const Cnt x = M.cnt[RM.o + lo + i];
             return (uint32_t)x.o + (uint32_t)x.i;
           });
  }
  if (width > scr_cap) {  // wider than the scratch: bisection inside the bucket
    int32_t a = lo, b = hi - 1;
    while (a < b) {
      const int32_t mid = a + (b - a) / 2;
      const long c = wave_sum(count_range_lane(M, RM.o, RM.c, lo, mid, excl));
      if (c > (long)t)
        b = mid;
      else
        a = mid + 1;
    }
    return a;
  }
  wave_fence();  // the reads of the histogram are done
  if (!small && RM.c >= kLookupRatio * width) {
    lookup_bucket(M, RM, lo, hi, scr, bytes);
  } else {
    for (int32_t i = lane; i < width; i += kWave) scr[i] = 0;
    wave_fence();
    gather_row(M, RM, lo, hi, scr, bytes);
  }
  wave_fence();
  return lo + pick_scan(width, t, [&](int32_t i) -> uint32_t {
           return lo + i == excl ? 0u : (uint32_t)scr[i];
         });
}

// t-th unit of the node's neighbour list (out-neighbours then in-neighbours,
// weight w), graph_parallel.hpp:1010-1027.
__device__ int32_t pick_neighbor(const GraphView& g, int64_t o0, int64_t kco, int64_t i0,
                                 int64_t kci, int64_t t) {
  if (!g.out_w) return t < kco ? g.out_idx[o0 + t] : g.in_idx[i0 + (t - kco)];
  const int lane = lane_id();
  const int64_t kc = kco + kci;
  long acc = 0;
  for (int64_t base = 0; base < kc; base += kWave) {
    const int64_t j = base + lane;
    long w = 0;
    if (j < kco)
      w = g.out_w[o0 + j];
    else if (j < kc)
      w = g.in_w[i0 + (j - kco)];
    const long inc = wave_incl_scan(w);
    const long tot = __shfl(inc, kWave - 1);
    if (acc + tot > t) {
      const unsigned long long hit = __ballot(acc + inc > t);
      const int64_t jj = base + (__ffsll((unsigned long long)hit) - 1);
      return jj < kco ? g.out_idx[o0 + jj] : g.in_idx[i0 + (jj - kco)];
    }
    acc += tot;
  }
  return -1;
}

// ---------------------------------------------------------------------------
// M build
// ---------------------------------------------------------------------------

// A workgroup's nodes by block: slot of block a in the LDS hash `key` of kSlots
// slots (-1: empty) with room for every node of the workgroup.
template <int kSlots>
__device__ __forceinline__ uint32_t block_slot(int32_t* key, int32_t a) {
  uint32_t h = hash32(a) & (kSlots - 1);
  for (;;) {
    const int32_t old = atomicCAS(&key[h], -1, a);
    if (old == -1 || old == a) return h;
    h = (h + 1) & (kSlots - 1);
  }
}

// Block degrees, list entries (weighted graphs; else they are the degrees) and
// node counts from the labels, `per` nodes to a workgroup, summed in LDS first:
// for B <= kDegLds by block, above in a hash of the workgroup's blocks.  A block
// that absorbed 7000 nodes in one merge phase (B = 100000) would take as many
// atomics on one address, ~30 ns each: 363 -> 24 us.  kW: 16 lanes sum a node's
// weights (one lane a node waited for each weight in turn: N = 3000 with hubs
// of 1000 edges 86 -> 13 us).
constexpr int kNodesWg = 1024;
constexpr int kNodesWgW = 256;
constexpr int kWSum = 16;  // lanes per weighted node
template <bool kW, bool kHash>
__global__ __launch_bounds__(256) void k_degrees(GraphView g, const int32_t* __restrict__ labels,
                                                 int32_t B, int32_t per, int32_t* d_out,
                                                 int32_t* d_in, int32_t* ecnt_out,
                                                 int32_t* ecnt_in, int32_t* bsize) {
  constexpr int kC = kW ? 5 : 3;  // counters
  constexpr int kSlots = kHash ? 2 * (kW ? kNodesWgW : kNodesWg) : kDegLds;
  __shared__ int32_t s_c[kC][kSlots];
  __shared__ int32_t s_key[kHash ? kSlots : 1];
  for (int i = threadIdx.x; i < kC * kSlots; i += 256) (&s_c[0][0])[i] = 0;
  if (kHash)
    for (int i = threadIdx.x; i < kSlots; i += 256) s_key[i] = -1;
  __syncthreads();
  const int64_t beg = (int64_t)blockIdx.x * per, end = min<int64_t>(beg + per, g.N);
  constexpr int kL = kW ? kWSum : 1;
  for (int64_t x = beg + threadIdx.x / kL; x < end; x += 256 / kL) {
    const int32_t a = labels[x];
    const int64_t o0 = g.out_ptr[x], o1 = g.out_ptr[x + 1];
    const int64_t i0 = g.in_ptr[x], i1 = g.in_ptr[x + 1];
    int32_t v[5] = {(int32_t)(o1 - o0), (int32_t)(i1 - i0), 1, (int32_t)(o1 - o0),
                    (int32_t)(i1 - i0)};
    if (kW) {
      const int sub = threadIdx.x % kL;
      v[0] = v[1] = 0;
      for (int64_t e = o0 + sub; e < o1; e += kL) v[0] += g.out_w[e];
      for (int64_t e = i0 + sub; e < i1; e += kL) v[1] += g.in_w[e];
#pragma unroll
      for (int d = kL / 2; d > 0; d >>= 1) {  // a node's lanes loop alike
        v[0] += __shfl_xor(v[0], d);
        v[1] += __shfl_xor(v[1], d);
      }
      if (sub != 0) continue;
    }
    const uint32_t h = kHash ? block_slot<kSlots>(s_key, a) : (uint32_t)a;
#pragma unroll
    for (int k = 0; k < kC; ++k)
      if (v[k]) atomicAdd(&s_c[k][h], v[k]);
  }
  __syncthreads();
  int32_t* dst[5] = {d_out, d_in, bsize, ecnt_out, ecnt_in};
  const int32_t n = kHash ? kSlots : B;
  for (int32_t i = threadIdx.x; i < n; i += 256) {
    const int32_t a = kHash ? s_key[i] : i;
    if (a < 0) continue;
#pragma unroll
    for (int k = 0; k < kC; ++k) {
      const int32_t v = s_c[k][i];
      if (v) atomicAdd(&dst[k][a], v);
    }
  }
}

// Slab capacity of a row with ecnt edges: a power of two >= slack*min(B, ecnt)+16
// (so keys inserted by later moves fit without a rebuild), or a direct row of
// B slots once that would reach B/8 (bounds a hashed row's scan; direct rows
// total at most 8*slack*E slots).
__device__ __forceinline__ int32_t cap_for(int32_t B, int32_t ecnt, int32_t slack) {
  const int64_t bound = ecnt < B ? ecnt : B;
  int64_t c = 32;
  while (c < slack * bound + 16) c <<= 1;
  return 8 * c >= B ? B : (int32_t)c;
}

// Block row a holds the keys of its out-edges and of its in-edges: its slab
// is sized for ecnt_out[a] + ecnt_in[a] keys.
// items (if not null): the pieces of the rows k_build_big builds, kBigNodes
// nodes each.
constexpr int kBigNodes = 64;
__device__ __forceinline__ int32_t big_pieces(int32_t nodes) {
  return max(1, (nodes + kBigNodes - 1) / kBigNodes);
}
constexpr int kRowTab = 1024;
__device__ __forceinline__ bool lds_row(int32_t cap, int32_t B) { return cap < B && cap <= kRowTab; }

__global__ void k_caps(int32_t B, int32_t slack, const int32_t* ecnt_out, const int32_t* ecnt_in,
                       const int32_t* bsize, int32_t* cap, int64_t* tmp, int2* items,
                       int32_t* n_items) {
  const int32_t a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a > B) return;
  if (a == B) {
    tmp[B] = 0;
    return;
  }
  const int64_t ec = (int64_t)ecnt_out[a] + ecnt_in[a];
  const int32_t c = cap_for(B, (int32_t)min<int64_t>(ec, (int64_t)B), slack);
  cap[a] = c;
  tmp[a] = c;
  if (items && !lds_row(c, B)) {
    const int32_t k = big_pieces(bsize[a]);
    const int32_t p = atomicAdd(n_items, k);
    for (int32_t i = 0; i < k; ++i) items[p + i] = make_int2(a, i);
  }
}

// key null: every row is direct, no key is read.
__global__ void k_fill(int32_t* key, Cnt* cnt, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    if (key) key[i] = -1;
    cnt[i] = Cnt{0, 0};
  }
}

// Nodes grouped by block (for the per-row build): node x goes to
// nodes[off[labels[x]] + k], k an arrival order in its block, counted by
// workgroup in LDS first (as k_degrees: 292 -> 11 us).
__global__ __launch_bounds__(256) void k_node_lists(int32_t N, const int32_t* __restrict__ labels,
                                                    const int32_t* __restrict__ off, int32_t* cur,
                                                    int32_t* nodes) {
  __shared__ int32_t s_key[2 * kNodesWg], s_n[2 * kNodesWg];
  for (int i = threadIdx.x; i < 2 * kNodesWg; i += 256) {
    s_key[i] = -1;
    s_n[i] = 0;
  }
  __syncthreads();
  constexpr int kQ = kNodesWg / 256;
  uint32_t h[kQ];
  int32_t rank[kQ];
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    const int64_t x = (int64_t)blockIdx.x * kNodesWg + q * 256 + threadIdx.x;
    rank[q] = -1;
    if (x < N) {
      h[q] = block_slot<2 * kNodesWg>(s_key, labels[x]);
      rank[q] = atomicAdd(&s_n[h[q]], 1);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = threadIdx.x; i < 2 * kNodesWg; i += 256) {
    const int32_t a = s_key[i];
    if (a >= 0) s_n[i] = off[a] + atomicAdd(&cur[a], s_n[i]);
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kQ; ++q)
    if (rank[q] >= 0)
      nodes[s_n[h[q]] + rank[q]] =
          (int32_t)((int64_t)blockIdx.x * kNodesWg + q * 256 + threadIdx.x);
}

// M build for large B: each hashed row of more than kMin and at most kSlots
// slots by one wavefront, from the lists of the row's own nodes alone -- an out-edge
// x -> v adds to M[a][label v] (o), an in-edge u -> x to M[label u][a] (i) --
// laid out in LDS and written out whole (a slab that size holds at most
// (kRowTab - 16) / slack list entries, so no wavefront has a long row).  Sending
// every edge to two rows' slabs at random instead took three times as long.
// Two launches, up to 256 slots and above: the LDS of 1024 a row would leave
// a CU 12 wavefronts, and each is one chain of loads (B = 200000: 393 -> 174 + 35 us).
template <int kSlots, int kMin>
__global__ __launch_bounds__(kWave* kNodalWaves) void k_build_rows(
    GraphView g, const int32_t* __restrict__ labels, const int32_t* __restrict__ bl_off,
    const int32_t* __restrict__ bl_nodes, MView M, int32_t* flags) {
  __shared__ int32_t s_k[kNodalWaves][kSlots];
  __shared__ int32_t s_o[kNodalWaves][kSlots];
  __shared__ int32_t s_i[kNodalWaves][kSlots];
  __shared__ int32_t s_pre[kNodalWaves][kWave + 1];
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  const int32_t a = blockIdx.x * kNodalWaves + w;
  if (a >= M.B) return;  // no workgroup barrier below
  const int64_t o = M.off[a];
  const int32_t c = M.cap[a];
  if (!lds_row(c, M.B) || c <= kMin || c > kSlots) return;
  int32_t* tk = s_k[w];
  int32_t* to = s_o[w];
  int32_t* ti = s_i[w];
  int32_t* pre = s_pre[w];
  for (int32_t j = lane; j < c; j += kWave) {
    tk[j] = -1;
    to[j] = 0;
    ti[j] = 0;
  }
  const uint32_t mask = (uint32_t)c - 1;
  const int32_t n0 = bl_off[a], n1 = a + 1 < M.B ? bl_off[a + 1] : g.N;
  bool full = false;
  for (int32_t base = n0; base < n1; base += kWave) {  // 64 nodes at a time
    const int32_t j = base + lane;
    int64_t o0 = 0, i0 = 0;
    long ko = 0, kn = 0;
    if (j < n1) {
      const int32_t x = bl_nodes[j];
      o0 = g.out_ptr[x];
      i0 = g.in_ptr[x];
      ko = g.out_ptr[x + 1] - o0;
      kn = ko + (g.in_ptr[x + 1] - i0);
    }
    const long inc = wave_incl_scan(kn);
    const long tot = __shfl(inc, kWave - 1);
    wave_fence();  // the previous chunk's reads of pre are done
    pre[lane + 1] = (int32_t)inc;
    if (lane == 0) pre[0] = 0;
    wave_fence();
    for (long e0 = 0; e0 < tot; e0 += kWave) {
      const int32_t ei = (int32_t)(e0 + lane);
      int lo = 0, hi = kWave - 1;  // the node k of entry ei: pre[k] <= ei < pre[k + 1]
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= ei)
          lo = mid;
        else
          hi = mid - 1;
      }
      const int64_t xo = __shfl(o0, lo), xi = __shfl(i0, lo);
      const long xko = __shfl(ko, lo);
      if (ei >= tot) continue;
      const long r = ei - pre[lo];
      const bool out = r < xko;
      int32_t v, wt = 1;
      if (out) {
        v = g.out_idx[xo + r];
        if (g.out_w) wt = g.out_w[xo + r];
      } else {
        v = g.in_idx[xi + (r - xko)];
        if (g.in_w) wt = g.in_w[xi + (r - xko)];
      }
      const int32_t b = labels[v];
      uint32_t h = hash32(b) & mask;
      bool done = false;
      for (int32_t probe = 0; probe < c && !done; ++probe) {
        int32_t k = __hip_atomic_load(&tk[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        if (k < 0) {
          k = atomicCAS(&tk[h], -1, b);
          if (k == -1) k = b;
        }
        if (k == b) {
          atomicAdd(out ? &to[h] : &ti[h], wt);
          done = true;
        }
        h = (h + 1) & mask;
      }
      full |= !done;
    }
  }
  wave_fence();
  for (int32_t j = lane; j < c; j += kWave) {
    M.key[o + j] = tk[j];
    M.cnt[o + j] = Cnt{to[j], ti[j]};
  }
  if (__ballot(full)) {
    if (lane == 0) atomicOr(flags, kFlagFull);
  }
}

// Fills the slabs of the rows of `items`, an item's share by gridDim.y
// workgroups: empty keys (null: no row has any), zero counts.
__global__ __launch_bounds__(256) void k_fill_big(MView M, int32_t* key, const int32_t* bsize,
                                                  const int2* items, const int32_t* n_items) {
  const int32_t n = *n_items;
  for (int32_t it = blockIdx.x; it < n; it += gridDim.x) {
    const int2 q = items[it];
    const Row R = m_row(M, q.x);
    const int64_t shares = (int64_t)big_pieces(bsize[q.x]) * gridDim.y;
    const int64_t at = (int64_t)q.y * gridDim.y + blockIdx.y;
    const int32_t j1 = (int32_t)(R.c * (at + 1) / shares);
    for (int32_t j = (int32_t)(R.c * at / shares) + threadIdx.x; j < j1; j += 256) {
      if (key) key[R.o + j] = -1;
      M.cnt[R.o + j] = Cnt{0, 0};
    }
  }
}

// The other rows, kBigNodes nodes of a block (an item of k_caps) to a workgroup,
// an item of many list entries to up to gridDim.y of them: the entries are
// summed per neighbour block in LDS, then each sum goes to M with one atomic.
// (An atomic per edge end piled onto a large block's own count: B = 100000
// with a block of 7000 nodes 526 -> 191 us.)  Keys beyond what the table holds near
// their home are added to M directly.  kHuge: nodes of more than kBigPart entries
// are left out of the items and come kHugePart entries a workgroup (`items`: node
// and part, n_huge of them), where one node in its item's kBigParts workgroups set
// the length of the build (set_labels at N = 100000, B = 20000 with one node of
// 2 M entries 4179 us, now 356, of 200000 648 and 261, of 9000 241 and 233; by parts
// of 2048 entries 376, 273 and 246).  Their rows are always among these: they have
// more than kBigPart entries, or are direct.
constexpr int kBigTab = 4096;
constexpr int kBigWalk = 8;
constexpr int32_t kBigPart = 8192;  // list entries from which an item is split
constexpr int kBigParts = 4;
constexpr int32_t kHugePart = 1024;  // list entries of a huge node to a workgroup
constexpr unsigned kBigGrid = 768;  // three workgroups of 51 KB of LDS per CU
template <bool kHuge>
__global__ __launch_bounds__(256) void k_build_big(GraphView g, const int32_t* __restrict__ labels,
                                                   const int32_t* __restrict__ bl_off,
                                                   const int32_t* __restrict__ bl_nodes, MView M,
                                                   const int2* items, const int32_t* n_items,
                                                   int32_t n_huge, int32_t* flags) {
  __shared__ int32_t s_k[kBigTab], s_o[kBigTab], s_i[kBigTab];
  __shared__ int64_t s_o0[kBigNodes], s_i0[kBigNodes];
  __shared__ long s_ko[kBigNodes], s_pre[kBigNodes + 1];
  const int lane = lane_id();
  const int32_t n = kHuge ? n_huge : *n_items;
  for (int32_t it = blockIdx.x; it < n; it += gridDim.x) {
    const int2 q = items[it];
    const int32_t a = kHuge ? labels[q.x] : q.x;
    const int32_t n0 = kHuge ? 0 : bl_off[a] + q.y * kBigNodes;
    const int32_t n1 = kHuge ? 1 : min(n0 + kBigNodes, a + 1 < M.B ? bl_off[a + 1] : g.N);
    __syncthreads();  // the previous item's table is written out
    if (threadIdx.x < kWave) {
      const int32_t j = n0 + lane;
      int64_t o0 = 0, i0 = 0;
      long ko = 0, kn = 0;
      if (j < n1) {
        const int32_t x = kHuge ? q.x : bl_nodes[j];
        o0 = g.out_ptr[x];
        i0 = g.in_ptr[x];
        ko = g.out_ptr[x + 1] - o0;
        kn = ko + (g.in_ptr[x + 1] - i0);
        if (!kHuge && kn > kBigPart) kn = 0;
      }
      const long inc = wave_incl_scan(kn);
      if (lane < kBigNodes) {
        s_o0[lane] = o0;
        s_i0[lane] = i0;
        s_ko[lane] = ko;
        s_pre[lane + 1] = inc;
        if (lane == 0) s_pre[0] = 0;
      }
    }
    __syncthreads();
    const long tot = s_pre[kBigNodes];
    const long parts = tot > kBigPart ? (long)gridDim.y : 1;
    if (!kHuge && (long)blockIdx.y >= parts) continue;  // the same for every thread
    const long e0 = kHuge ? (long)q.y * kHugePart : tot * (long)blockIdx.y / parts;
    const long e1 = kHuge ? min(tot, e0 + kHugePart) : tot * ((long)blockIdx.y + 1) / parts;
    int32_t tab = 256;  // a power of two >= twice the entries, at most kBigTab
    while (tab < kBigTab && tab < 2 * (e1 - e0)) tab <<= 1;
    for (int i = threadIdx.x; i < tab; i += 256) {
      s_k[i] = -1;
      s_o[i] = 0;
      s_i[i] = 0;
    }
    __syncthreads();
    for (long ei = e0 + threadIdx.x; ei < e1; ei += 256) {
      int lo = 0, hi = kBigNodes - 1;  // the node of entry ei
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_pre[mid] <= ei)
          lo = mid;
        else
          hi = mid - 1;
      }
      const long r = ei - s_pre[lo], ko = s_ko[lo];
      const bool out = r < ko;
      int32_t v, wt = 1;
      if (out) {
        v = g.out_idx[s_o0[lo] + r];
        if (g.out_w) wt = g.out_w[s_o0[lo] + r];
      } else {
        v = g.in_idx[s_i0[lo] + (r - ko)];
        if (g.in_w) wt = g.in_w[s_i0[lo] + (r - ko)];
      }
      const int32_t b = labels[v];
      uint32_t h = hash32(b) & (uint32_t)(tab - 1);
      bool done = false;
      for (int p = 0; p < kBigWalk && !done; ++p) {
        const int32_t old = atomicCAS(&s_k[h], -1, b);
        if (old == -1 || old == b) {
          atomicAdd(out ? &s_o[h] : &s_i[h], wt);
          done = true;
        }
        h = (h + 1) & (uint32_t)(tab - 1);
      }
      if (!done) m_add(M, a, b, out ? wt : 0, out ? 0 : wt, flags);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < tab; i += 256)
      if (s_k[i] >= 0) m_add(M, a, s_k[i], s_o[i], s_i[i], flags);
  }
}

// M build for B <= kHistB (every row is direct there: 8 times the smallest
// hashed slab reaches B): workgroup (g, half) counts the block pairs of its
// share of the edges, of the rows of its half, in LDS, and the degrees and
// sizes with them, and writes its counts out whole; k_hist_sum adds them up.
// No counter is cleared or added to in memory, no row header is needed
// first, and the host waits for nothing.  (Every workgroup's counts by atomics
// on M, and before B = 128 a sort of the edges' pairs: E = 1 M at B = 76 46 us
// in the insert alone, E = 4 M at B = 132 ~250 us.)
constexpr int kHistThreads = 1024;
constexpr int kHistOne = 200;  // B up to which one workgroup's LDS holds every row
struct HistArgs {
  GraphView g;
  const int32_t* src;  // edge sources
  const int32_t* labels;
  int64_t E;
  int32_t B, G, rows;  // rows per workgroup
  int32_t* part;       // [G][B * B] counts
  int32_t* part_d;     // [G * halves][3][kHistB] d_out, d_in, sizes
};

template <int kCells>
__global__ __launch_bounds__(kHistThreads) void k_hist(HistArgs a) {
  __shared__ int32_t s_h[kCells];
  __shared__ int32_t s_size[kHistB];
  const int32_t B = a.B, t = threadIdx.x;
  const int32_t g = blockIdx.x, half = blockIdx.y;
  const int32_t r0 = half * a.rows, nr = min(a.rows, B - r0), cells = nr * B;
  for (int32_t i = t; i < cells; i += kHistThreads) s_h[i] = 0;
  if (t < kHistB) s_size[t] = 0;
  __syncthreads();
  const int64_t e0 = a.E * g / a.G, e1 = a.E * (g + 1) / a.G;
  constexpr int kQ = 4;  // edges in flight per thread
  for (int64_t e = e0 + t; e < e1; e += kQ * kHistThreads) {
    int32_t u[kQ], v[kQ], w[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int64_t j = e + q * kHistThreads;
      u[q] = v[q] = -1;
      w[q] = 1;
      if (j < e1) {
        u[q] = a.src[j];
        v[q] = a.g.out_idx[j];
        if (a.g.out_w) w[q] = a.g.out_w[j];
      }
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q)
      if (u[q] >= 0) {
        u[q] = a.labels[u[q]] - r0;
        v[q] = a.labels[v[q]];
      }
#pragma unroll
    for (int q = 0; q < kQ; ++q)
      if (u[q] >= 0 && u[q] < nr) atomicAdd(&s_h[u[q] * B + v[q]], w[q]);
  }
  const int64_t n0 = (int64_t)a.g.N * g / a.G, n1 = (int64_t)a.g.N * (g + 1) / a.G;
  if (half == 0)
    for (int64_t n = n0 + t; n < n1; n += kHistThreads) atomicAdd(&s_size[a.labels[n]], 1);
  __syncthreads();
  int32_t* out = a.part + (int64_t)g * B * B + (int64_t)r0 * B;
  for (int32_t i = t; i < cells; i += kHistThreads) out[i] = s_h[i];
  int32_t* d = a.part_d + ((int64_t)half * a.G + g) * 3 * kHistB;
  if (t < kHistB) {  // row sums (each row from a column of its own: no bank conflicts)
    int32_t sum = 0;
    if (t >= r0 && t < r0 + nr)
      for (int32_t j = 0, c = t % B; j < B; ++j, c = c + 1 == B ? 0 : c + 1)
        sum += s_h[(t - r0) * B + c];
    d[t] = sum;
  } else if (t < 2 * kHistB) {  // column sums
    int32_t sum = 0;
    if (t - kHistB < B)
      for (int32_t j = 0; j < nr; ++j) sum += s_h[j * B + (t - kHistB)];
    d[t] = sum;
  } else if (t < 3 * kHistB) {
    d[t] = s_size[t - 2 * kHistB];
  }
}

// M, the row headers, degrees and sizes from k_hist's counts: block row a by
// workgroup a, d_out, d_in and sizes by the last three, each by four groups of
// threads with eight parts in flight (one group, and one workgroup with a part
// at a time for the degrees: G = 256, B = 132 66 -> 6.5 us).
struct HistSum {
  MView M;
  int64_t* off;
  int32_t* cap;
  int32_t *d_out, *d_in, *bsize;
  const int32_t* part;
  const int32_t* part_d;
  int32_t G, parts_d;
};

constexpr int kSumGroups = 4;
__global__ __launch_bounds__(kHistB* kSumGroups) void k_hist_sum(HistSum a) {
  __shared__ int32_t s_v[kSumGroups][kHistB];
  const int32_t B = a.M.B, stride = a.M.stride;
  const int32_t t = threadIdx.x % kHistB, w = threadIdx.x / kHistB, r = blockIdx.x;
  const bool row = r < B;
  const int32_t k = r - B;  // which of d_out, d_in, sizes
  const int64_t n = row ? (int64_t)B * B : 3 * kHistB;
  const int32_t* p = row ? a.part + (int64_t)r * B + t : a.part_d + k * kHistB + t;
  const int32_t G = row ? a.G : a.parts_d;
  constexpr int kQ = 8;
  int32_t v = 0;
  if (t < B)
    for (int32_t g = w * kQ; g < G; g += kSumGroups * kQ) {
      int32_t x[kQ];
#pragma unroll
      for (int q = 0; q < kQ; ++q) x[q] = g + q < G ? p[(g + q) * n] : 0;
#pragma unroll
      for (int q = 0; q < kQ; ++q) v += x[q];
    }
  s_v[w][t] = v;
  __syncthreads();
  if (w == 0 && t < B) {
#pragma unroll
    for (int q = 1; q < kSumGroups; ++q) v += s_v[q][t];
    if (row) {
      a.M.cnt[(int64_t)r * stride + t].o = v;
      a.M.cnt[(int64_t)t * stride + r].i = v;
    } else {
      (k == 0 ? a.d_out : k == 1 ? a.d_in : a.bsize)[t] = v;
    }
  }
  if (row)
    for (int32_t i = B + threadIdx.x; i < stride; i += kHistB * kSumGroups)
      a.M.cnt[(int64_t)r * stride + i] = Cnt{0, 0};
  if (row) {
    if (threadIdx.x == 0) {
      a.off[r] = (int64_t)r * stride;
      a.cap[r] = B;
    }
  } else if (k == 0) {
    for (int i = threadIdx.x; i < kGrowBlocks; i += kHistB * kSumGroups)
      a.M.gst->chunk[i].pos = a.M.gst->chunk[i].end = 0;
    if (threadIdx.x == 0) {
      a.off[B] = (int64_t)B * stride;
      a.M.gst->nospace = 0;
      a.M.gst->ovf_n = 0;
      a.M.gst->used = (unsigned long long)B * (unsigned long long)stride;
    }
  }
}

// M build for kHistB < B <= kPairSortB, B < N (rows mostly direct, few distinct
// block pairs, so per-edge atomics would pile onto the same counts): the
// edges' block pairs a*B + b are sorted and summed per pair, then each pair
// is added once.  Above, rows are mostly hashed and the build goes by rows
// (k_build_rows), as it does for B = N, a search's start from one block per node:
// its pairs are as many as its edges, and sorting them takes longer (set_labels at
// B = N = 500 128 us by pairs and 107 by rows, 2000 164 and 123, 4096 177 and 120).
constexpr int32_t kPairSortB = 4096;

__global__ void k_pair_keys(int64_t E, const int32_t* __restrict__ src,
                            const int32_t* __restrict__ dst, const int32_t* __restrict__ w,
                            const int32_t* __restrict__ labels, int32_t B, uint32_t* key,
                            int32_t* val) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
       e += (int64_t)gridDim.x * blockDim.x) {
    key[e] = (uint32_t)labels[src[e]] * (uint32_t)B + (uint32_t)labels[dst[e]];
    val[e] = w ? w[e] : 1;
  }
}

__global__ void k_insert_pairs(int64_t E, const uint32_t* __restrict__ key,
                               const int32_t* __restrict__ val, const int32_t* count, MView M,
                               int32_t* flags) {
  const int64_t n = min<int64_t>(*count, E);
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int32_t a = (int32_t)(key[e] / (uint32_t)M.B), b = (int32_t)(key[e] % (uint32_t)M.B);
    const int32_t w = val[e];
    if (a == b) {
      m_add(M, a, a, w, w, flags);
    } else {
      m_add(M, a, b, w, 0, flags);
      m_add(M, b, a, 0, w, flags);
    }
  }
}

// Bucket sums (o + i) of the block rows that keep them: up to kSumRows rows to a
// workgroup (fewer while that leaves the GPU short of workgroups), which handles
// those of them one by one, eight slots a thread in flight.  Most rows that keep
// sums have up to a few thousand slots: workgroups of 4 wavefronts take 6.1 us at
// B = 513, 12.3 at 2000, 26 at 4000 and 38 at 5000, of 16 11.8, 31, 62 and 75.  Above
// B = 16384 few rows keep sums and one may be longer than 4 wavefronts take in a
// few rounds: a direct row of 100000 slots costs 33 us more with 4, blocks of
// thousands of nodes at B = 20000 take 93 with 4 and 96 with 16; fewer rows a
// workgroup do not help there (two launches at B = 200000 and 100000 89 us with up
// to 64 and 49 rows, 103 with 49 and 25).  Sets the hashed ones' marks too
// (room_mark).
constexpr int kSumRows = 64;
constexpr int32_t kSumLongB = 16384;
__global__ __launch_bounds__(1024) void k_bucket_sums(MView m, int32_t rows) {
  __shared__ int32_t s_b[kNBK];
  __shared__ int32_t s_keys;
  const int lane = lane_id();
  const int64_t a0 = (int64_t)blockIdx.x * rows;
  const int32_t cl = lane < rows && a0 + lane < m.B ? m.cap[a0 + lane] : 0;
  unsigned long long todo = __ballot(cl > 0 && row_sums(m, cl));  // the same in every wavefront
  while (todo) {
    const int l = __ffsll(todo) - 1;
    todo &= todo - 1ull;
    const int64_t a = a0 + l;
    const int32_t c = __shfl(cl, l);
    for (int i = threadIdx.x; i < kNBK; i += blockDim.x) s_b[i] = 0;
    if (threadIdx.x == 0) s_keys = 0;
    __syncthreads();
    int32_t keys = 0;
    const int64_t o = m.off[a];
    const bool direct = c == m.B;
    constexpr int kQ = 8;
    for (int32_t j0 = threadIdx.x; j0 < c; j0 += kQ * blockDim.x) {
      int32_t k[kQ];
      Cnt x[kQ];
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        const int32_t j = j0 + q * (int32_t)blockDim.x;
        k[q] = -1;
        x[q] = Cnt{0, 0};
        if (j < c) {
          k[q] = direct ? j : m.key[o + j];
          x[q] = m.cnt[o + j];
        }
      }
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        const int32_t v = x[q].o + x[q].i;
        keys += k[q] >= 0;
        if (k[q] >= 0 && v != 0) atomicAdd(&s_b[k[q] >> m.bshift], v);
      }
    }
    atomicAdd(&s_keys, keys);
    __syncthreads();
    for (int i = threadIdx.x; i < kNBK; i += blockDim.x) m.bs[a * kNBK + i] = s_b[i];
    if (threadIdx.x == 0 && !direct) m.gmark[a] = room_mark(s_keys, c, m.slack);
    __syncthreads();
  }
}

// The per-block counters and flags a rebuild starts from, zeroed in one
// launch (degrees, edge counts, sizes, growth marks, parked
// counts: B entries each; build_flags[0..2]).
constexpr int kClearArrays = 8;
struct ClearArgs {
  int32_t* p[kClearArrays];
  int32_t n;
  int32_t* flags;
};

__global__ void k_clear_build(ClearArgs c) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int a = 0; a < kClearArrays; ++a)
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < c.n; i += stride)
      c.p[a][i] = 0;
  if (blockIdx.x == 0 && threadIdx.x < 3) c.flags[threadIdx.x] = 0;
}

// Workgroup stamps of profiled batch launches (100 MHz wall clock; 0 = the
// workgroup did not run).  Each workgroup of a profiled k_nodal, k_apply or
// k_grow writes its start at t[b] and its end at t[stride + b] with plain
// stores: one atomic per workgroup on a shared word costs more than the
// kernel's own tail.  Per batch slot: k_nodal's starts and ends (G each),
// k_apply's (G + 1 each), k_grow's (kGrowBlocks each).
__global__ void k_stamp_init(unsigned long long* t, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    t[i] = 0ull;
}

// Per batch slot and kernel (block slot*3 + kernel): the first workgroup start
// and the last workgroup end, to out[6*slot + 2*kernel + {0, 1}].
__global__ __launch_bounds__(256) void k_stamp_reduce(const unsigned long long* t, int32_t G,
                                                     int32_t grow_blocks, unsigned long long* out) {
  __shared__ unsigned long long s_lo[256], s_hi[256];
  const int32_t slot = blockIdx.x / 3, k = blockIdx.x % 3;
  const int64_t base = (int64_t)slot * (4 * (int64_t)G + 2 + 2 * grow_blocks) +
                       (k == 0 ? 0 : k == 1 ? 2 * (int64_t)G : 4 * (int64_t)G + 2);
  const int32_t n = k == 0 ? G : k == 1 ? G + 1 : grow_blocks;
  unsigned long long lo = ~0ull, hi = 0ull;
  for (int32_t i = threadIdx.x; i < n; i += blockDim.x) {
    const unsigned long long a = t[base + i], b = t[base + n + i];
    if (a != 0ull) lo = min(lo, a);
    hi = max(hi, b);
  }
  s_lo[threadIdx.x] = lo;
  s_hi[threadIdx.x] = hi;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      s_lo[threadIdx.x] = min(s_lo[threadIdx.x], s_lo[threadIdx.x + h]);
      s_hi[threadIdx.x] = max(s_hi[threadIdx.x], s_hi[threadIdx.x + h]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[6 * (int64_t)slot + 2 * k] = s_lo[0];
    out[6 * (int64_t)slot + 2 * k + 1] = s_hi[0];
  }
}

// Growth state after a rebuild: nothing parked, the pool used up to
// the new slabs' end (the event counters are kept).
__global__ void k_reset_grow(GrowState* g, unsigned long long used) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kGrowBlocks) g->chunk[i].pos = g->chunk[i].end = 0;
  if (i == 0) {
    g->nospace = 0;
    g->ovf_n = 0;
    g->used = used;
  }
}

// short_of: the carry-out ran out of candidates, the labels stay.
__global__ void k_relabel(int32_t N, int32_t* labels, const int32_t* __restrict__ map,
                          const int32_t* short_of) {
  const int32_t x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x < N && *short_of == 0) labels[x] = map[labels[x]];
}

// ---------------------------------------------------------------------------
// Graph ingest on the device: CSR (out-lists) and CSC (in-lists) extended by
// an increment of edges.  Lists keep the reference's neighbour order -- a
// node's neighbours in the order their edges were delivered
// (graph_parallel.hpp:290-294) -- so node x's new list is its old list, then
// its new edges in delivery order.  With cnt[x] new edges at x, the new
// offsets are new_ptr[x] = old_ptr[x] + sum_{y<x} cnt[y]; old edge j of x
// moves by that shift, and the j-th edge of the increment stably sorted by
// x lands at old_ptr[x+1] + j.
// ---------------------------------------------------------------------------

__global__ void k_count_keys(int64_t n, const int32_t* __restrict__ key, int32_t* cnt) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    atomicAdd(&cnt[key[i]], 1);
}

// deg[x] = old list length + new edges of x, deg[N] = 0 (exclusive-scan input).
__global__ void k_new_deg(int32_t N, const int64_t* __restrict__ old_ptr,
                          const int32_t* __restrict__ cnt, int64_t* deg) {
  const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x < N) deg[x] = old_ptr[x + 1] - old_ptr[x] + cnt[x];
  if (x == N) deg[x] = 0;
}

// Old lists to their new places, one wavefront per node; owner (nullable)
// records the node of each new slot (the CSR's edge sources).
__global__ __launch_bounds__(256) void k_move_lists(int32_t N, const int64_t* __restrict__ old_ptr,
                                                    const int64_t* __restrict__ new_ptr,
                                                    const int32_t* __restrict__ old_idx,
                                                    const int32_t* __restrict__ old_w,
                                                    int32_t* new_idx, int32_t* new_w, int32_t* owner) {
  const int64_t x = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (x >= N) return;
  const int64_t o0 = old_ptr[x], o1 = old_ptr[x + 1], shift = new_ptr[x] - o0;
  for (int64_t j = o0 + lane_id(); j < o1; j += kWave) {
    new_idx[j + shift] = old_idx[j];
    if (new_w) new_w[j + shift] = old_w[j];
    if (owner) owner[j + shift] = (int32_t)x;
  }
}

// The increment's edges (sorted stably by their node key) to their places:
// sorted edge j of node x = key[j] goes to old_ptr[x + 1] + j.  other[] is
// the edge's other end (the target for CSR, the source for CSC).
__global__ void k_place_new(int64_t n, const int32_t* __restrict__ skey,
                            const int32_t* __restrict__ sidx, const int64_t* __restrict__ old_ptr,
                            const int32_t* __restrict__ other, const int32_t* __restrict__ w,
                            int32_t* new_idx, int32_t* new_w, int32_t* owner) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n;
       j += (int64_t)gridDim.x * blockDim.x) {
    const int32_t x = skey[j], i = sidx[j];
    const int64_t pos = old_ptr[x + 1] + j;
    new_idx[pos] = other[i];
    if (new_w) new_w[pos] = w ? w[i] : 1;
    if (owner) owner[pos] = x;
  }
}

__global__ void k_iota(int64_t n, int32_t* v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    v[i] = (int32_t)i;
}

// ---------------------------------------------------------------------------
// Entropy, graph_parallel.hpp:1281-1319:
// data_S = -(sum_ab L(M_ab) - sum_a L(d_out[a]) - sum_b L(d_in[b]))
// ---------------------------------------------------------------------------

// Sum over the workgroup's threads (every thread calls); thread 0 returns it.
__device__ __forceinline__ i128 block_sum(Acc v) {
  __shared__ long s_h[16], s_l[16];
  v.h = wave_sum(v.h);
  v.l = wave_sum(v.l);
  const int w = threadIdx.x / kWave;
  if (lane_id() == 0) {
    s_h[w] = v.h;
    s_l[w] = v.l;
  }
  __syncthreads();
  Acc t{0, 0};
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)(blockDim.x / kWave); ++i) {
      t.h += s_h[i];
      t.l += s_l[i];
    }
  return acc_value(t);
}

__device__ void block_store(Acc v, long* out) {
  const i128 x = block_sum(v);
  if (threadIdx.x == 0) {
    out[0] = (long)(x >> 64);
    out[1] = (long)(unsigned long)(u128)x;
  }
}

// The same for int128 partials.
__device__ __forceinline__ i128 block_sum128(i128 t) {
  __shared__ long s_hi[16];
  __shared__ unsigned long s_lo[16];
  t = wave_sum128(t);
  const int w = threadIdx.x / kWave;
  if (lane_id() == 0) {
    s_hi[w] = (long)(t >> 64);
    s_lo[w] = (unsigned long)(u128)t;
  }
  __syncthreads();
  i128 tot = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)(blockDim.x / kWave); ++i)
      tot += (i128)(((u128)(unsigned long)s_hi[i] << 64) | (u128)s_lo[i]);
  return tot;
}

// minus data_S of a state, for one workgroup: from k_entropy's nparts
// partials, or, M all direct with at most kEntropyOne slots, from M itself
// (one launch and one pass over the partials less).
constexpr int32_t kEntropyOne = 16384;
struct EntropyIn {
  const long* part;
  int32_t nparts;  // 0: from M
  const Cnt* cnt;
  int64_t slots;
  const int32_t *d_out, *d_in;
  int32_t B;
  const int64_t* lam;
};

__device__ __forceinline__ i128 block_entropy(const EntropyIn& a) {
  if (a.nparts > 0) {
    i128 t = 0;
    for (int32_t i = threadIdx.x; i < a.nparts; i += blockDim.x)
      t += (i128)(((u128)(unsigned long)a.part[2 * i] << 64) | (u128)(unsigned long)a.part[2 * i + 1]);
    return block_sum128(t);
  }
  Acc acc{0, 0};
  const int32_t n = (int32_t)a.slots;
  constexpr int kQ = 8;
  for (int32_t i0 = threadIdx.x; i0 < n; i0 += kQ * blockDim.x) {
    int32_t v[kQ];
    int64_t L[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int32_t i = i0 + q * (int32_t)blockDim.x;
      v[q] = i < n ? max(a.cnt[i].o, 0) : 0;
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) L[q] = a.lam[v[q]];
#pragma unroll
    for (int q = 0; q < kQ; ++q) acc_add(acc, v[q], L[q]);
  }
  for (int32_t b = threadIdx.x; b < a.B; b += blockDim.x) {
    sub_L(acc, a.lam, a.d_out[b]);
    sub_L(acc, a.lam, a.d_in[b]);
  }
  return block_sum(acc);
}

// One pass over the pool in use, eight slots per thread in flight and lambda
// from LDS while the counts are small: bound by memory (N = 500000, 1.6 GB of
// slabs 400 -> 338 us; a slot at a time each waited for its own lambda).
constexpr int kLamEnt = 512;
__global__ __launch_bounds__(256) void k_entropy(const Cnt* __restrict__ cnt,
                                                 const GrowState* gst,
                                                 const int32_t* __restrict__ d_out,
                                                 const int32_t* __restrict__ d_in, int32_t B,
                                                 const int64_t* __restrict__ lam, int32_t lam_last,
                                                 int64_t P, long* part) {
  __shared__ int64_t s_lam[kLamEnt];
  const int64_t used = (int64_t)gst->used;  // every live slab lies below
  const int64_t nslots = used < P ? used : P;
  for (int i = threadIdx.x; i < kLamEnt; i += 256) s_lam[i] = lam[min(i, lam_last)];
  __syncthreads();
  Acc acc{0, 0};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int4* pair = reinterpret_cast<const int4*>(cnt);  // (o, i) of two slots
  const int64_t npairs = nslots / 2;
  constexpr int kQ = 4;
  for (int64_t i = t; i < npairs; i += kQ * stride) {
    int32_t v[2 * kQ], top = 0;  // each M[a][b] once, as o of row a
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int64_t j = i + q * stride;
      const int4 x = j < npairs ? pair[j] : make_int4(0, 0, 0, 0);
      v[2 * q] = max(x.x, 0);
      v[2 * q + 1] = max(x.z, 0);
    }
#pragma unroll
    for (int q = 0; q < 2 * kQ; ++q) top = max(top, v[q]);
    if (__ballot(top > 0) == 0) continue;
    const bool small = __ballot(top >= kLamEnt) == 0;
#pragma unroll
    for (int q = 0; q < 2 * kQ; ++q)
      if (v[q] > 0) acc_add(acc, v[q], small ? s_lam[v[q]] : lam[v[q]]);
  }
  if (t == 0 && (nslots & 1)) {
    const int32_t v = cnt[nslots - 1].o;
    if (v > 0) acc_add(acc, v, lam[v]);
  }
  for (int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; b < B; b += stride) {
    sub_L(acc, lam, d_out[b]);
    sub_L(acc, lam, d_in[b]);
  }
  block_store(acc, part + 2 * blockIdx.x);
}

// Carry-out order (graph_parallel.hpp:1230) on the device: blocks sorted by
// (dS, block id), dS an int128 ordered as (signed hi, unsigned lo), by two
// stable radix passes -- lo first, then hi with its sign bit flipped.
__global__ void k_sort_init(int32_t B, const unsigned long* __restrict__ lo,
                            unsigned long long* key, int32_t* idx) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < B) {
    key[i] = lo[i];
    idx[i] = i;
  }
}

__global__ void k_sort_hi(int32_t B, const long* __restrict__ hi, const int32_t* __restrict__ perm,
                          unsigned long long* key) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < B) key[i] = (unsigned long long)hi[perm[i]] ^ (1ull << 63);
}

// Carry-out (graph_parallel.hpp:1225-1279) on the device.  The reference goes
// through the blocks in order and links block i to the current block of its
// target best[i], unless that is i itself, until B_to_merge links are made.
// Only i's own turn links i, so a link fails exactly when it would close a
// cycle of i -> best[i]: each component of that functional graph has one cycle,
// and its member that comes last in the order stays.  So:
//   f^(2^K) maps every block onto a cycle (2^K >= B), and onto all of them;
//   the largest order among i, f(i), ..., by the same doubling, is i's own on
//   a cycle exactly at its last member;
//   the links made are the first B_to_merge successes in the order (a scan);
//   the roots by pointer jumping over them, then the surviving labels ranked
//   ascending.
// The host's loop with its copies took 4 ms at B = 200000 and 60 us and a host
// wait more at B = 50.
struct CarryArgs {
  int32_t B, B_to_merge;
  const int32_t* best;
  const long* hi;            // dS words (k_carry_one up to kCarryRank blocks)
  const unsigned long* lo;
  const int32_t* order;      // blocks by (dS, id), above that
  const int32_t* bsize;
  int32_t* map;
  int32_t* short_of;         // 1: fewer than B_to_merge links can be made
  int32_t* host_short;       // the same, in the host's memory
  HostWord done;             // told after it
};

constexpr int kCarryThreads = 1024;
// Blocks ranked by comparing all pairs, above that by the two sorts: a
// carry-out with its build takes 49 us so and 58 sorted at B = 300, 60 and 58 at
// 400, 71 and 58 at 512, 355 and 294 at 1024.
constexpr int kCarryRank = 384;
constexpr int kCarryOne = 8192;   // blocks one workgroup carries out in its LDS

// Inclusive scan over the workgroup of each thread's own value; the total in
// *total for every thread.
__device__ __forceinline__ int32_t block_scan(int32_t v, int32_t* s_w, int32_t* total) {
  const int w = threadIdx.x / kWave, nw = blockDim.x / kWave;
  const int32_t inc = (int32_t)wave_incl_scan32((uint32_t)v);
  __syncthreads();
  if (lane_id() == kWave - 1) s_w[w] = inc;
  __syncthreads();
  int32_t before = 0, all = 0;
  for (int i = 0; i < nw; ++i) {
    if (i < w) before += s_w[i];
    all += s_w[i];
  }
  *total = all;
  return before + inc;
}

template <int kMax>
__global__ __launch_bounds__(kCarryThreads) void k_carry_one(CarryArgs a) {
  // blocks per thread: t + k * kCarryThreads
  constexpr int kI = (kMax + kCarryThreads - 1) / kCarryThreads;
  __shared__ int32_t s_p[kMax], s_m[kMax], s_a[kMax];
  __shared__ int32_t s_w[kCarryThreads / kWave];
  const int32_t B = a.B, t = threadIdx.x;
  int32_t rank[kI], f[kI], p[kI], m[kI];
  if (kMax <= kCarryRank) {
    __shared__ long s_hi[kCarryRank];
    __shared__ unsigned long s_lo[kCarryRank];
    if (t < B) {
      s_hi[t] = a.hi[t];
      s_lo[t] = a.lo[t];
    }
    __syncthreads();
    rank[0] = 0;
    if (t < B) {
      const long h = s_hi[t];
      const unsigned long l = s_lo[t];
      for (int32_t j = 0; j < B; ++j) {
        const bool before = s_hi[j] < h || (s_hi[j] == h && (s_lo[j] < l || (s_lo[j] == l && j < t)));
        rank[0] += before;
      }
    }
  } else {
    for (int32_t j = t; j < B; j += kCarryThreads) s_a[a.order[j]] = j;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kI; ++k)
      rank[k] = t + k * kCarryThreads < B ? s_a[t + k * kCarryThreads] : 0;
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int32_t i = t + k * kCarryThreads;
    if (i < B) {
      f[k] = p[k] = s_p[i] = a.best[i];
      m[k] = s_m[i] = rank[k];
      s_a[i] = 0;
    }
  }
  for (int32_t w = 1; w < B; w <<= 1) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kI; ++k)
      if (t + k * kCarryThreads < B) {
        m[k] = max(m[k], s_m[p[k]]);
        p[k] = s_p[p[k]];
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kI; ++k)
      if (t + k * kCarryThreads < B) {
        s_p[t + k * kCarryThreads] = p[k];
        s_m[t + k * kCarryThreads] = m[k];
      }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kI; ++k)
    if (t + k * kCarryThreads < B) s_a[p[k]] = 1;
  __syncthreads();
  bool link[kI];
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int32_t i = t + k * kCarryThreads;
    link[k] = false;
    if (i < B) {
      link[k] = !(s_a[i] && m[k] == rank[k]);
      s_p[rank[k]] = link[k];
    }
  }
  __syncthreads();
  // successes up to each rank: thread t scans ranks [t * kI, (t + 1) * kI)
  int32_t mine = 0, total;
#pragma unroll
  for (int k = 0; k < kI; ++k)
    if (t * kI + k < B) mine += s_p[t * kI + k];
  int32_t run = block_scan(mine, s_w, &total) - mine;
#pragma unroll
  for (int k = 0; k < kI; ++k)
    if (t * kI + k < B) {
      run += s_p[t * kI + k];
      s_m[t * kI + k] = run;
    }
  __syncthreads();
  const bool fails = total < a.B_to_merge;
  if (t == 0) {
    *a.short_of = fails;
    *a.host_short = fails;
    host_done(a.done);
  }
  if (fails) return;  // the same for every thread
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int32_t i = t + k * kCarryThreads;
    if (i < B) {
      s_p[i] = link[k] && s_m[rank[k]] <= a.B_to_merge ? f[k] : i;
      s_a[i] = 0;
    }
  }
  for (int32_t w = 1; w < B; w <<= 1) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kI; ++k)  // in place: what is read is an ancestor at least as far
      if (t + k * kCarryThreads < B)
        s_p[t + k * kCarryThreads] = s_p[s_p[t + k * kCarryThreads]];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int32_t i = t + k * kCarryThreads;
    if (i < B && a.bsize[i] > 0) s_a[s_p[i]] = 1;
  }
  __syncthreads();
  mine = 0;
#pragma unroll
  for (int k = 0; k < kI; ++k)
    if (t * kI + k < B) mine += s_a[t * kI + k];
  run = block_scan(mine, s_w, &total) - mine;
#pragma unroll
  for (int k = 0; k < kI; ++k)
    if (t * kI + k < B) {
      s_m[t * kI + k] = run;
      run += s_a[t * kI + k];
    }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int32_t i = t + k * kCarryThreads;
    if (i < B) a.map[i] = s_a[s_p[i]] ? s_m[s_p[i]] : 0;
  }
}

// The same steps over the whole GPU (more than kCarryOne blocks).
__global__ void k_carry_init(int32_t B, const int32_t* __restrict__ order,
                             const int32_t* __restrict__ best, int32_t* rank, int2* pm,
                             int32_t* cyc) {
  const int32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= B) return;
  const int32_t i = order[j];
  rank[i] = j;
  pm[i] = make_int2(best[i], j);
  cyc[i] = 0;
}

// kCarryHops of in's windows joined to one: its end and the last rank in it.
// Two a launch (doubling) took 18 launches at B = 100000, each little more than
// its own launch and gap (6.5 us); eight a launch take 6 of 6 us.
constexpr int kCarryHops = 8;
__global__ void k_carry_jump(int32_t B, const int2* __restrict__ in, int2* __restrict__ out) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B) return;
  int2 x = in[i];
#pragma unroll
  for (int q = 1; q < kCarryHops; ++q) {
    const int2 y = in[x.x];
    x = make_int2(y.x, max(x.y, y.y));
  }
  out[i] = x;
}

__global__ void k_carry_cycle(int32_t B, const int2* __restrict__ pm, int32_t* cyc) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < B) cyc[pm[i].x] = 1;
}

__global__ void k_carry_success(int32_t B, const int2* __restrict__ pm,
                                const int32_t* __restrict__ cyc, const int32_t* __restrict__ rank,
                                int32_t* succ) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < B) succ[rank[i]] = !(cyc[i] && pm[i].y == rank[i]);
}

__global__ void k_carry_link(int32_t B, int32_t B_to_merge, const int32_t* __restrict__ best,
                             const int32_t* __restrict__ rank, const int32_t* __restrict__ succ,
                             const int32_t* __restrict__ scan, int32_t* par, int32_t* alive,
                             int32_t* short_of, int32_t* host_short, HostWord done) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B) return;
  const int32_t r = rank[i];
  par[i] = succ[r] && scan[r] <= B_to_merge ? best[i] : i;
  alive[i] = 0;
  if (i == 0) {
    const int32_t fails = scan[B - 1] < B_to_merge;
    *short_of = fails;
    *host_short = fails;
    host_done(done);
  }
}

// par[i] to the ancestor kRootHops links of par up, or the root: in place, as
// another thread's new value is an ancestor too and at least as far.  So the
// reach is multiplied by kRootHops a launch, whatever the chains (doubling: 18
// launches, now 4).
constexpr int kRootHops = 32;
__global__ void k_carry_root(int32_t B, int32_t* par) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B) return;
  const int32_t first = par[i];
  int32_t x = first;
  for (int q = 1; q < kRootHops; ++q) {
    const int32_t y = par[x];
    if (y == x) break;
    x = y;
  }
  if (x != first) par[i] = x;
}

__global__ void k_carry_alive(int32_t B, const int32_t* __restrict__ bsize,
                              const int32_t* __restrict__ par, int32_t* alive) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < B && bsize[i] > 0) alive[par[i]] = 1;
}

__global__ void k_carry_map(int32_t B, const int32_t* __restrict__ par,
                            const int32_t* __restrict__ alive, const int32_t* __restrict__ before,
                            int32_t* map) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < B) map[i] = alive[par[i]] ? before[par[i]] : 0;
}

// ---------------------------------------------------------------------------
// Block merge, graph_parallel.hpp:761-988 (+ :349-368)
// ---------------------------------------------------------------------------

struct MergeArgs {
  MView M;
  const int32_t* d_out;
  const int32_t* d_in;
  const int64_t* lam;
  int32_t lam_last;  // its last entry, at most kLamMerge - 1
  int32_t B;
  int32_t K;
  uint64_t seed, stream;  // pre-drawn mode: stream = the round's first draw
  const uint64_t* uni;    // pre-drawn stream (4 words per draw), else null
  int32_t* best_s;
  long* best_hi;
  unsigned long* best_lo;
};

// L(m1) + L(m2) - L(m1 + m2) over the two counts of a key in two rows, where
// both are non-zero (no branch per pair: a wavefront's pairs are rarely all
// zero).  lambda from LDS while the counts are small.
constexpr int kLamMerge = 512;
__device__ __forceinline__ void overlap_pair(Acc& acc, const int64_t* lam, const int64_t* s_lam,
                                             Cnt x, Cnt y) {
  const bool bo = x.o > 0 && y.o > 0, bi = x.i > 0 && y.i > 0;
  if (!__ballot(bo || bi)) return;
  const int32_t a = bo ? x.o : 0, b = bo ? y.o : 0, c = bi ? x.i : 0, d = bi ? y.i : 0;
  int64_t L[6];
  if (__ballot(max(a + b, c + d) >= kLamMerge)) {
    L[0] = lam[a];
    L[1] = lam[b];
    L[2] = lam[a + b];
    L[3] = lam[c];
    L[4] = lam[d];
    L[5] = lam[c + d];
  } else {
    L[0] = s_lam[a];
    L[1] = s_lam[b];
    L[2] = s_lam[a + b];
    L[3] = s_lam[c];
    L[4] = s_lam[d];
    L[5] = s_lam[c + d];
  }
  acc_add(acc, a, L[0]);
  acc_add(acc, b, L[1]);
  acc_add(acc, -(a + b), L[2]);
  acc_add(acc, c, L[3]);
  acc_add(acc, d, L[4]);
  acc_add(acc, -(c + d), L[5]);
}

// per-lane part of sum_{i not in {r,s}} [L(m1) + L(m2) - L(m1+m2)] over the
// keys where rows r and s of M are both non-zero, and the same over the
// columns (the only terms that survive the factorised merge dS): one pass
// over the shorter block row, four of its slots per lane at a time, probing
// the other for each of its keys.
__device__ Acc merge_overlap_lane(const MView& m, const int64_t* lam, const int64_t* s_lam,
                                  int32_t r, int32_t s) {
  const int lane = lane_id();
  const bool r_short = m.cap[r] <= m.cap[s];
  const int32_t a1 = r_short ? r : s, a2 = r_short ? s : r;
  const Row R1 = m_row(m, a1), R2 = m_row(m, a2);
  const bool direct = R1.c == m.B;  // then so is the longer row: key j sits at slot j of both
  Acc acc{0, 0};
  constexpr int kOvl = 2;
  for (int32_t base = 0; base < R1.c; base += kOvl * kWave) {
    int32_t k[kOvl];
    Cnt x[kOvl], y[kOvl];
#pragma unroll
    for (int u = 0; u < kOvl; ++u) {
      const int32_t j = base + u * kWave + lane;
      k[u] = -1;
      x[u] = y[u] = Cnt{0, 0};
      if (j < R1.c) {
        k[u] = direct ? j : m.key[R1.o + j];
        x[u] = m.cnt[R1.o + j];
        if (direct) y[u] = m.cnt[R2.o + j];
      }
    }
    if (!direct) {
      Probe p[kOvl];
#pragma unroll
      for (int u = 0; u < kOvl; ++u) {
        if (x[u].o <= 0 && x[u].i <= 0) k[u] = -1;
        if (k[u] >= 0) p[u] = m_probe(m, R2, k[u]);
      }
#pragma unroll
      for (int u = 0; u < kOvl; ++u)
        if (k[u] >= 0) y[u] = m_value(m, R2, k[u], p[u]);
    }
#pragma unroll
    for (int u = 0; u < kOvl; ++u) {
      if (k[u] == r || k[u] == s) x[u] = Cnt{0, 0};
      overlap_pair(acc, lam, s_lam, x[u], y[u]);
    }
  }
  return acc;
}

// A block's row in LDS, shared by its K proposals: its non-zero keys in
// ascending order with both counts and the running sum of o + i (n = -1: the
// row has too many of them and the proposals read it from M).  512 of at most 4096
// slots where K exceeds the workgroup's kMergeWaves: a direct row of 2500 slots
// with 360 of them non-zero is then read once, not scanned beside row s for each
// proposal (B = 2500, K = 10 283 -> 229 us a round, with 256 of 2048 slots).  With
// fewer proposals, all of which run at once, ordering more than 256 keys costs
// more than it saves (B = 500, all non-zero: K = 1 45 us without and 113 with, K = 4
// 45 and 65, K = 5 66 and 67).
constexpr int kRowLds = 512, kRowLdsFew = 256;
constexpr int kRowSlotsPerKey = 8;  // slots of a row looked through for them, per key
struct RowLds {
  const int32_t* k;
  const int32_t* o;
  const int32_t* i;
  const uint32_t* cum;
  int32_t n;
};

// Position of the first entry whose running sum exceeds t (t < the row's
// total).
__device__ __forceinline__ int32_t rowlds_pick(const RowLds& L, uint32_t t) {
  int32_t lo = 0, hi = L.n - 1;
  while (lo < hi) {
    const int32_t mid = (lo + hi) >> 1;
    if (L.cum[mid] > t)
      hi = mid;
    else
      lo = mid + 1;
  }
  return lo;
}

// The counts of key b in the row.
__device__ __forceinline__ Cnt rowlds_find(const RowLds& L, int32_t b) {
  int32_t lo = 0, hi = L.n;
  while (lo < hi) {
    const int32_t mid = (lo + hi) >> 1;
    if (L.k[mid] < b)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo < L.n && L.k[lo] == b ? Cnt{L.o[lo], L.i[lo]} : Cnt{0, 0};
}

// merge_overlap_lane with row r from LDS: r's entries look themselves up in
// row s.
__device__ Acc merge_overlap_lds(const MView& m, const int64_t* lam, const int64_t* s_lam,
                                 int32_t r, int32_t s, Row RS, const RowLds& L) {
  const int lane = lane_id();
  const bool direct = RS.c == m.B;
  Acc acc{0, 0};
  for (int32_t e0 = 0; e0 < L.n; e0 += kWave) {
    const int32_t e = min(e0 + lane, L.n - 1);
    const int32_t b = L.k[e];
    int32_t kk;
    const Window w = win_issue(m, RS, b, direct);
    const uint32_t h = win_end(w, b, direct, kk);
    const bool in = e0 + lane < L.n && b != r && b != s;
    Cnt x{0, 0}, y{0, 0};
    if (in && kk == b)
      y = m.cnt[RS.o + h];
    else if (in && kk >= 0)
      y = m_value_more(m, RS, b, h);
    if (in) x = Cnt{L.o[e], L.i[e]};
    overlap_pair(acc, lam, s_lam, x, y);
  }
  return acc;
}

// The terms of merging r into s outside the overlap: corner and degrees.
__device__ __forceinline__ void merge_terms(Acc& acc, const int64_t* lam, int32_t dor, int32_t dir,
                                            int32_t dos, int32_t dis, int32_t Mrr, int32_t Mrs,
                                            int32_t Msr, int32_t Mss) {
  const int32_t dos2 = dos + dor, dis2 = dis + dir;
  bool inf = false;
  add_T(acc, lam, 1, Mrr, dir, dor, inf);
  add_T(acc, lam, 1, Mrs, dis, dor, inf);
  add_T(acc, lam, 1, Msr, dir, dos, inf);
  add_T(acc, lam, 1, Mss, dis, dos, inf);
  add_T(acc, lam, -1, Mrr + Mrs + Msr + Mss, dis2, dos2, inf);
  const int32_t Xr = dor - Mrr - Mrs, Xs = dos - Msr - Mss;
  const int32_t Yr = dir - Mrr - Msr, Ys = dis - Mrs - Mss;
  add_P(acc, lam, -1, Xr, dor, inf);
  add_P(acc, lam, -1, Xs, dos, inf);
  add_P(acc, lam, 1, Xr + Xs, dos2, inf);
  add_P(acc, lam, -1, Yr, dir, inf);
  add_P(acc, lam, -1, Ys, dis, inf);
  add_P(acc, lam, 1, Yr + Ys, dis2, inf);
}

__device__ __forceinline__ void merge_draw(const MergeArgs& a, int32_t r, int32_t idx,
                                           uint64_t x[4]) {
  if (a.uni)
    predrawn(a.uni, a.stream + (uint64_t)r * (uint64_t)a.K + (uint64_t)idx, x);
  else
    usap::philox4x64((uint64_t)r, (uint64_t)idx, a.stream, usap::kTagMerge, a.seed, 0, x);
}

// One proposal by one wavefront (kD: every row is direct).
template <bool kD>
__device__ void merge_one(const MergeArgs& a, int32_t r, int32_t idx, int32_t* scr,
                          const RowLds& L, const int64_t* s_lam, int32_t& s_out, i128& dS_out) {
  const int32_t B = a.B;
  const int32_t dor = a.d_out[r], dir = a.d_in[r];
  const uint32_t k = (uint32_t)dor + (uint32_t)dir;
  uint64_t x[4];
  merge_draw(a, r, idx, x);
  int32_t s;
  if (k == 0) {
    s = (int32_t)usap::idx_of(x[2], B);
  } else {
    long bytes = 0;
    const uint32_t t0 = idx32(x[0], k);
    const int32_t u = L.n >= 0 ? L.k[rowlds_pick(L, t0)]
                               : select_combined<kD>(a.M, r, t0, -1, nullptr, scr, kScr, bytes);
    const uint32_t da = (uint32_t)a.d_out[u] + (uint32_t)a.d_in[u];
    if (usap::uniform_branch(x[1], da, B)) {
      s = usap::uniform_not_r(x[2], r, B);
    } else {
      const Cnt ur = L.n >= 0 ? rowlds_find(L, u) : m_get(a.M, r, u);  // M[r][u], M[u][r]
      const uint32_t W2 = da - (uint32_t)ur.o - (uint32_t)ur.i;
      s = W2 == 0 ? usap::uniform_not_r(x[2], r, B)
                  : select_combined<kD>(a.M, u, idx32(x[3], W2), r, nullptr, scr, kScr, bytes);
    }
  }
  s_out = s;
  if (s == r) {
    dS_out = 0;
    return;
  }
  const Row RS = m_row(a.M, s);
  const Cnt crs = L.n >= 0 ? rowlds_find(L, s) : m_get(a.M, r, s);  // M[r][s], M[s][r]
  const int32_t Mrr = L.n >= 0 ? rowlds_find(L, r).o : m_get(a.M, r, r).o;
  const int32_t Mss = m_value(a.M, RS, s, m_probe(a.M, RS, s)).o;
  const int32_t dos = a.d_out[s], dis = a.d_in[s];
  const Acc ov = L.n >= 0 ? merge_overlap_lds(a.M, a.lam, s_lam, r, s, RS, L)
                          : merge_overlap_lane(a.M, a.lam, s_lam, r, s);
  Acc acc{wave_sum(ov.h), wave_sum(ov.l)};
  merge_terms(acc, a.lam, dor, dir, dos, dis, Mrr, crs.o, crs.i, Mss);
  dS_out = acc_value(acc);
}

// Blocks: the long rows from r[0] on, n[0] of them, the others from r[B - 1]
// down, n[1] of them (r null: every block).
struct MergeList {
  int32_t* r;
  int32_t* n;
};

// The K proposals of a block by one workgroup, a wavefront each in turn: every
// block, or those k_merge_rows left to it.  kWaves: 4, or, where the blocks are
// too few to fill the GPU, up to 16, so that all of a block's proposals run at
// once (K = 10, us a round with 4 and 16: B = 20 19 and 14, 100 24 and 17, 300 41 and
// 41, 500 54 and 53, 800 58 and 77, 1000 68 and 97).
// kKeys: kRowLds or kRowLdsFew.  The list's long rows come first: one of 20000 slots
// is the length of the launch, and started last it adds to it.  A workgroup
// takes every gridDim.x-th item; kMergeGrid of them are handed out as others end,
// where one per place on the GPU left some with 7 rows and most with 6 (B =
// 8000, K = 10, nearly all rows direct: 1280 workgroups 2270 us, 8192 1705; a list
// of few rows loses nothing to the rest, B = 200000 1345 either way).
template <int kWaves, bool kD, int kKeys>
__global__ __launch_bounds__(kWave* kWaves, 4) void k_merge(MergeArgs a, MergeList list) {
  __shared__ long s_hi[kWaves];
  __shared__ unsigned long s_lo[kWaves];
  __shared__ int32_t s_idx[kWaves];
  __shared__ int32_t s_s[kWaves];
  __shared__ __align__(16) int32_t s_scr[kWaves][kD ? 4 : kScr];  // direct rows need none
  __shared__ int32_t s_uk[kKeys], s_uo[kKeys], s_ui[kKeys];  // as found
  __shared__ int32_t s_rk[kKeys], s_ro[kKeys], s_ri[kKeys];  // by key
  __shared__ uint32_t s_cum[kKeys];
  __shared__ int64_t s_lam[kLamMerge];
  __shared__ int32_t s_rn;
  const int w = threadIdx.x / kWave, lane = lane_id();
  const int nw = blockDim.x / kWave;
  for (int i = threadIdx.x; i < kLamMerge; i += blockDim.x) s_lam[i] = a.lam[min(i, a.lam_last)];
  const int32_t nlong = list.r ? list.n[0] : 0;
  const int32_t count = list.r ? nlong + list.n[1] : a.B;
  for (int32_t item = blockIdx.x; item < count; item += gridDim.x) {
    const int32_t r =
        !list.r ? item : item < nlong ? list.r[item] : list.r[a.B - 1 - (item - nlong)];
    // row r's non-zero keys into LDS once for the K proposals (unordered), then
    // ordered by key (ranks: keys are distinct), then the running sums
    const Row R = m_row(a.M, r);
    const bool fits = R.c <= kRowSlotsPerKey * kKeys;  // the same for every thread
    __syncthreads();
    if (threadIdx.x == 0) s_rn = 0;
    __syncthreads();
    if (fits) {
      const bool direct = R.c == a.B;
      for (int32_t j = threadIdx.x; j < R.c; j += blockDim.x) {
        const Cnt q = a.M.cnt[R.o + j];
        const int32_t key = direct ? j : a.M.key[R.o + j];
        if (key >= 0 && (q.o > 0 || q.i > 0)) {
          const int32_t p = atomicAdd(&s_rn, 1);
          if (p < kKeys) {
            s_uk[p] = key;
            s_uo[p] = q.o;
            s_ui[p] = q.i;
          }
        }
      }
    }
    __syncthreads();
    const int32_t rn = fits ? s_rn : INT32_MAX;
    RowLds L{s_rk, s_ro, s_ri, s_cum, rn <= kKeys ? rn : -1};
    if (L.n > 0) {
      for (int32_t e = threadIdx.x; e < L.n; e += blockDim.x) {
        const int32_t key = s_uk[e];
        int32_t rank = 0;
#pragma unroll 4
        for (int32_t j = 0; j < L.n; ++j) rank += s_uk[j] < key;
        s_rk[rank] = key;
        s_ro[rank] = s_uo[e];
        s_ri[rank] = s_ui[e];
      }
      __syncthreads();
      if (w == 0) {
        constexpr int kPer = kKeys / kWave;
        uint32_t own = 0;
        for (int q = 0; q < kPer; ++q) {
          const int32_t e = lane * kPer + q;
          own += e < L.n ? (uint32_t)s_ro[e] + (uint32_t)s_ri[e] : 0u;
        }
        uint32_t run = wave_incl_scan32(own) - own;
        for (int q = 0; q < kPer; ++q) {
          const int32_t e = lane * kPer + q;
          if (e >= L.n) break;
          run += (uint32_t)s_ro[e] + (uint32_t)s_ri[e];
          s_cum[e] = run;
        }
      }
      __syncthreads();
    }
    int32_t bidx = -1, bs = -1;
    i128 bd = 0;
    for (int32_t idx = w; idx < a.K; idx += nw) {
      int32_t s;
      i128 d;
      merge_one<kD>(a, r, idx, s_scr[w], L, s_lam, s, d);
      if (bidx < 0 || d < bd) {  // strict less: the earliest proposal wins ties
        bidx = idx;
        bs = s;
        bd = d;
      }
    }
    if (lane == 0) {
      s_hi[w] = (long)(bd >> 64);
      s_lo[w] = (unsigned long)(u128)bd;
      s_idx[w] = bidx;
      s_s[w] = bs;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int best = -1;
      i128 bv = 0;
      for (int i = 0; i < nw; ++i) {
        if (s_idx[i] < 0) continue;
        const i128 v = (i128)(((u128)(unsigned long)s_hi[i] << 64) | (u128)s_lo[i]);
        if (best < 0 || v < bv || (v == bv && s_idx[i] < s_idx[best])) {
          best = i;
          bv = v;
        }
      }
      a.best_s[r] = s_s[best];
      a.best_hi[r] = s_hi[best];
      a.best_lo[r] = s_lo[best];
    }
  }
}

// The K proposals of a block by one wavefront, for hashed rows of at most
// kRowSlots slots with at most kRowWave non-zero keys (the others are marked in
// best_s for k_merge).  Proposal j's draws, picks, decision, corner and degree terms
// are lane j's; only a multinomial pick and the overlap are the whole
// wavefront's, proposal by proposal, the overlap two proposals at a time: r's
// entries look themselves up in row s, whose eight-key windows nearly always
// answer in one round of loads, mostly that there is nothing (s is a uniform
// draw most often).  A workgroup per block with a wavefront per proposal spent
// its time in the same chain K times over, three proposals one after another
// per wavefront, Philox and terms in every lane: B = 200000 4890 -> 1150 us a
// round.
constexpr int kRowSlots = 1024;
constexpr int kRowWave = 256;
enum : int32_t { kLeft = -1, kLeftLong = -2 };  // in best_s: a block left to k_merge
__global__ __launch_bounds__(kWave* kMergeWaves, 4) void k_merge_rows(MergeArgs a,
                                                                    MergeList list) {
  __shared__ __align__(16) int32_t s_k[kMergeWaves][kRowWave], s_o[kMergeWaves][kRowWave],
      s_i[kMergeWaves][kRowWave];
  __shared__ uint32_t s_cum[kMergeWaves][kRowWave];
  __shared__ __align__(16) int32_t s_scr[kMergeWaves][kScr];
  __shared__ int64_t s_lam[kLamMerge];
  const int w = threadIdx.x / kWave, lane = lane_id();
  for (int i = threadIdx.x; i < kLamMerge; i += blockDim.x) s_lam[i] = a.lam[min(i, a.lam_last)];
  if (blockIdx.x == 0 && threadIdx.x < 2) list.n[threadIdx.x] = 0;  // for k_merge_list
  const int32_t B = a.B;
  const int32_t r = blockIdx.x * kMergeWaves + w;
  const bool in = r < B;
  const Row R = m_row(a.M, in ? r : 0);
  const int32_t dor = in ? a.d_out[r] : 0, dir = in ? a.d_in[r] : 0;
  __syncthreads();
  if (!in) return;
  if (R.c == B || R.c > kRowSlots) {
    if (lane == 0) a.best_s[r] = R.c > kRowSlotsPerKey * kRowLds ? kLeftLong : kLeft;
    return;
  }
  // the row's non-zero entries, unordered
  int32_t n = 0;
  constexpr int kQ = 4;
  for (int32_t base = 0; base < R.c; base += kQ * kWave) {
    int32_t key[kQ];
    Cnt x[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int32_t j = base + q * kWave + lane;
      key[q] = -1;
      x[q] = Cnt{0, 0};
      if (j < R.c) {
        key[q] = a.M.key[R.o + j];
        x[q] = a.M.cnt[R.o + j];
      }
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const bool live = key[q] >= 0 && (x[q].o > 0 || x[q].i > 0);
      const unsigned long long m = __ballot(live);
      const int32_t p = n + __popcll(m & ((1ull << lane) - 1ull));
      if (live && p < kRowWave) {
        s_k[w][p] = key[q];
        s_o[w][p] = x[q].o;
        s_i[w][p] = x[q].i;
      }
      n += __popcll(m);
    }
    if (n > kRowWave) break;
  }
  if (n > kRowWave) {
    if (lane == 0) a.best_s[r] = kLeft;
    return;
  }
  wave_fence();
  // ordered by key
  constexpr int kPer = kRowWave / kWave;
  {
    int32_t mk[kPer], mo[kPer], mi[kPer], rank[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int32_t e = lane + q * kWave;
      rank[q] = 0;
      mk[q] = e < n ? s_k[w][e] : 0;
      mo[q] = e < n ? s_o[w][e] : 0;
      mi[q] = e < n ? s_i[w][e] : 0;
    }
    for (int32_t j = 0; j < n; ++j) {
      const int32_t k = s_k[w][j];
#pragma unroll
      for (int q = 0; q < kPer; ++q) rank[q] += k < mk[q];
    }
    wave_fence();
#pragma unroll
    for (int q = 0; q < kPer; ++q)
      if (lane + q * kWave < n) {
        s_k[w][rank[q]] = mk[q];
        s_o[w][rank[q]] = mo[q];
        s_i[w][rank[q]] = mi[q];
      }
    wave_fence();
    uint32_t v[kPer], own = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int32_t e = lane * kPer + q;
      own += e < n ? (uint32_t)s_o[w][e] + (uint32_t)s_i[w][e] : 0u;
      v[q] = own;
    }
    const uint32_t before = wave_incl_scan32(own) - own;
#pragma unroll
    for (int q = 0; q < kPer; ++q)
      if (lane * kPer + q < n) s_cum[w][lane * kPer + q] = before + v[q];
    wave_fence();
  }
  const RowLds L{s_k[w], s_o[w], s_i[w], s_cum[w], n};
  const int32_t Mrr = rowlds_find(L, r).o;
  const uint32_t k = (uint32_t)dor + (uint32_t)dir;
  int32_t bidx = -1, bs = -1;  // the best so far, in every lane
  i128 bd = 0;
  for (int32_t j0 = 0; j0 < a.K; j0 += kWave) {
    const int32_t m = min(a.K - j0, kWave);
    const bool act = lane < m;
    uint64_t x[4];
    merge_draw(a, r, j0 + (act ? lane : 0), x);
    int32_t s, u = 0;
    uint32_t t = 0;
    bool pend = false;
    if (k == 0) {
      s = (int32_t)usap::idx_of(x[2], B);
    } else {
      const int32_t e = rowlds_pick(L, idx32(x[0], k));
      u = L.k[e];
      const uint32_t da = (uint32_t)a.d_out[u] + (uint32_t)a.d_in[u];
      s = usap::uniform_not_r(x[2], r, B);
      if (!usap::uniform_branch(x[1], da, B)) {
        const uint32_t W2 = da - (uint32_t)L.o[e] - (uint32_t)L.i[e];
        pend = W2 != 0;
        t = pend ? idx32(x[3], W2) : 0;
      }
    }
    for (unsigned long long todo = __ballot(act && pend); todo; todo &= todo - 1ull) {
      const int l = __ffsll(todo) - 1;
      long bytes = 0;
      const int32_t sel = select_combined<false>(a.M, __builtin_amdgcn_readlane(u, l),
                                                 read_lane32(t, l), r, nullptr, s_scr[w], kScr,
                                                 bytes);
      if (lane == l) s = sel;
    }
    const bool move = act && s != r;
    const Row RS = m_row(a.M, move ? s : r);
    const int32_t dos = a.d_out[move ? s : r], dis = a.d_in[move ? s : r];
    const bool sdir = RS.c == B;
    int32_t Mss = 0;
    if (move) {
      int32_t kk;
      const Window win = win_issue(a.M, RS, s, sdir);
      const uint32_t h = win_end(win, s, sdir, kk);
      if (kk == s)
        Mss = a.M.cnt[RS.o + h].o;
      else if (kk >= 0)
        Mss = m_value_more(a.M, RS, s, h).o;
    }
    const Cnt crs = rowlds_find(L, s);  // M[r][s], M[s][r]
    Acc acc{0, 0};
    if (move) merge_terms(acc, a.lam, dor, dir, dos, dis, Mrr, crs.o, crs.i, Mss);
    // overlaps, two proposals at a time
    unsigned long long todo = __ballot(move);
    while (todo) {
      int l[2];
      l[0] = __ffsll(todo) - 1;
      todo &= todo - 1ull;
      l[1] = todo ? __ffsll(todo) - 1 : -1;
      todo &= todo - 1ull;
      int32_t ss[2];
      Row S[2];
      bool dirct[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int from = l[i] < 0 ? l[0] : l[i];
        ss[i] = __builtin_amdgcn_readlane(s, from);
        S[i] = Row{read_lane((long)RS.o, from), __builtin_amdgcn_readlane(RS.c, from)};
        dirct[i] = S[i].c == B;
      }
      Acc ov[2] = {{0, 0}, {0, 0}};
      bool any[2] = {false, false};
      for (int32_t e0 = 0; e0 < n; e0 += kWave) {
        const int32_t e = min(e0 + lane, n - 1);
        const int32_t b = L.k[e];
        Window win[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) win[i] = win_issue(a.M, S[i], b, dirct[i]);
        Cnt y[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          int32_t kk;
          const uint32_t h = win_end(win[i], b, dirct[i], kk);
          const bool ok = l[i] >= 0 && e0 + lane < n && b != r && b != ss[i];
          y[i] = Cnt{0, 0};
          if (ok && kk == b)
            y[i] = a.M.cnt[S[i].o + h];
          else if (ok && kk >= 0)
            y[i] = m_value_more(a.M, S[i], b, h);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (!__ballot(y[i].o != 0 || y[i].i != 0)) continue;
          any[i] = true;
          overlap_pair(ov[i], a.lam, s_lam, Cnt{L.o[e], L.i[e]}, y[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (!any[i]) continue;
        const long h = wave_sum(ov[i].h), lo = wave_sum(ov[i].l);
        if (lane == l[i]) {
          acc.h += h;
          acc.l += lo;
        }
      }
    }
    // the least dS; the earliest proposal wins ties
    i128 d = act ? acc_value(acc) : (i128)0;
    int32_t idx = act ? j0 + lane : -1, sv = s;
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      const long h2 = __shfl_xor((long)(d >> 64), off);
      const unsigned long l2 = __shfl_xor((unsigned long)(u128)d, off);
      const int32_t i2 = __shfl_xor(idx, off), s2 = __shfl_xor(sv, off);
      const i128 d2 = (i128)(((u128)(unsigned long)h2 << 64) | (u128)l2);
      if (i2 >= 0 && (idx < 0 || d2 < d || (d2 == d && i2 < idx))) {
        d = d2;
        idx = i2;
        sv = s2;
      }
    }
    if (bidx < 0 || d < bd) {
      bidx = idx;
      bs = sv;
      bd = d;
    }
  }
  if (lane == 0) {
    a.best_s[r] = bs;
    a.best_hi[r] = (long)(bd >> 64);
    a.best_lo[r] = (unsigned long)(u128)bd;
  }
}

// The blocks k_merge_rows left.  Two atomics a workgroup: one a block, on one
// counter, took 1.1 ms of the round where 15000 rows were left (~70 ns each, one
// after another).
constexpr int kMergeListThreads = 1024;
__global__ __launch_bounds__(kMergeListThreads) void k_merge_list(
    int32_t B, const int32_t* __restrict__ best_s, MergeList list) {
  __shared__ int32_t s_w[kMergeListThreads / kWave];
  __shared__ int32_t s_base[2];
  const int32_t r = blockIdx.x * kMergeListThreads + threadIdx.x;
  const int32_t left = r < B ? best_s[r] : 0;
  // both ranks in one scan: long rows in the high half (a workgroup has 1024)
  int32_t total;
  const int32_t at =
      block_scan(left == kLeftLong ? 1 << 16 : left == kLeft ? 1 : 0, s_w, &total);
  if (total == 0) return;
  if (threadIdx.x < 2)
    s_base[threadIdx.x] =
        atomicAdd(&list.n[threadIdx.x], threadIdx.x == 0 ? total >> 16 : total & 0xffff);
  __syncthreads();
  if (left == kLeftLong) list.r[s_base[0] + (at >> 16) - 1] = r;
  if (left == kLeft) list.r[B - 1 - (s_base[1] + (at & 0xffff) - 1)] = r;
}

// Ends a call whose last kernel tells the host nothing.
__global__ void k_word(HostWord done) { host_done(done); }

// ---------------------------------------------------------------------------
// Nodal proposal, graph_parallel.hpp:990-1222
// ---------------------------------------------------------------------------


// Workgroups are dispatched to the GPU's 8 XCDs (each with its own L2) in
// turn: workgroup b runs on XCD b % 8.  Block b of a batch kernel takes item
// block xcd_block(b, G) instead of b, so the workgroups of one XCD cover
// consecutive nodes, and the cache lines holding those nodes' CSR/CSC offsets,
// lists and proposal outputs are fetched into one L2 instead of up to eight.
// A bijection of [0, G).
constexpr int kXcds = 8;
__device__ __forceinline__ int32_t xcd_block(int32_t b, int32_t G) {
  const int32_t per = G / kXcds, extra = G % kXcds;
  const int32_t x = b % kXcds, j = b / kXcds;
  return (x < extra ? x * (per + 1) : extra * (per + 1) + (x - extra) * per) + j;
}

// One workgroup's share of a batch, written by k_nodal and summed by block 0
// of k_apply (no same-address atomics per node).
struct BlockPart {
  long sum_hi;  // sum of the accepted finite dS of the block's nodes (int128)
  unsigned long sum_lo;
  unsigned long long nodal_bytes;  // algorithmic bytes of k_nodal
  unsigned long long apply_bytes;  // algorithmic bytes of k_apply
  int32_t moves;
  int32_t ninf;
};

// Algorithmic bytes of one accepted move of a node with kc list entries: the
// list (id, label, weight), per entry up to 4 slots of 12 bytes, the rows
// and degrees of r and s, the label.
__device__ __forceinline__ long apply_tally(int64_t kc) { return 52 + 60 * kc + 32 + 32 + 4; }

// One proposal as k_apply and the callers read it.
struct __align__(16) Prop {
  int32_t s, r;      // proposed block, old block
  int32_t acc, inf;  // accepted; -1: dS is -inf
};

// Its exact dS.
struct __align__(16) PropDs {
  long hi;
  unsigned long lo;
};

struct NodalArgs {
  GraphView g;
  MView M;
  const int32_t* labels;
  const int32_t* d_out;
  const int32_t* d_in;
  const int64_t* lam;
  int32_t lam_last;  // its last entry, at most kLamLds - 1
  int32_t B;
  int32_t beg, end;
  int32_t exact;
  const uint64_t* draws;  // four words per draw: node n's at n, or, predrawn,
  int32_t predrawn;       // at sweep->stream0 + n
  const int64_t* big_off;
  int32_t* big_tab;
  Prop* prop;
  PropDs* prop_ds;
  int32_t* prop_u;  // profiling: block of the drawn neighbour (-1: none), else null
  BlockPart* part;
  Status* status;
  Sweep* sweep;  // read, and stop_n written by block 0
  // kernel timers on (profiling): [0] earliest workgroup start, [1] latest
  // workgroup end of this launch, 100 MHz clock; else null
  unsigned long long* tstamp;  // workgroup stamps (start [b], end [tstride + b]) or null
  int32_t tstride;
};

// List entry j of node n (out-edges then in-edges): neighbour id (-1 past the
// end) and weight.
__device__ __forceinline__ void list_entry(const GraphView& g, int64_t o0, int64_t kco,
                                           int64_t i0, int64_t kc, int64_t j, int32_t& v,
                                           int32_t& w) {
  v = -1;
  w = 1;
  if (j < kco) {
    v = g.out_idx[o0 + j];
    if (g.out_w) w = g.out_w[o0 + j];
  } else if (j < kc) {
    v = g.in_idx[i0 + (j - kco)];
    if (g.in_w) w = g.in_w[i0 + (j - kco)];
  }
}

// Orders this wavefront's LDS writes and atomics before its later LDS reads:
// the LDS runs one wavefront's operations in order, so only the compiler has
// to keep it (no wait for loads in flight).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// What moving node n from r to s changes outside the neighbour blocks: the
// counts of the corner, the degrees of r and s, n's weights into r and s.
struct Corner {
  int32_t rr, rs, sr, ss;      // M[r][r], M[r][s], M[s][r], M[s][s]
  int32_t dor, dir, dos, dis;  // degrees of r and s
  int32_t k_out, k_in;         // n's out- and in-weight
  int32_t wor, wir, wos, wis;  // n's weights into (out) and from (in) r and s
  int32_t wself;               // n's self-loops
};

// lambda(m) from the first kLamLds entries in LDS, or, big, from the table.
constexpr int kLamLds = 256;
__device__ __forceinline__ int64_t lam_at(const int64_t* lam, const int64_t* s_lam, bool big,
                                          int32_t m) {
  return big ? lam[max(m, 0)] : s_lam[max(m, 0)];
}

// Adds the move's 16 corner and degree terms to acc, one per lane (in every
// lane they were a quarter of the kernel's arithmetic); inf: the moved state
// has an infinite term.  Lane bits: col (0: column r, 1: s), row (0: row r, 1:
// s), now (0: before the move, 1: after), deg.
//   deg = 0: T(M[row][col], d_in[col], d_out[row])
//   deg = 1: the row's other out-edges X (col = 0) or the column's other
//            in-edges Y (col = 1) of block `row`, m * lambda(degree)
// each + before and - after, the degree terms the other way round.
// s_lam: LDS copy of lambda's first kLamLds entries, or null.
__device__ __forceinline__ void corner_terms(const NodalArgs& a, const Corner& c,
                                             const int64_t* s_lam, Acc& acc, bool& inf) {
  const int lane = lane_id();
  int32_t rr2, rs2, sr2, ss2;
  if (!a.exact) {  // graph_parallel.hpp:1117-1145: only out-edges update the rows
    rr2 = c.rr - c.wor;
    rs2 = c.rs - c.wos;
    sr2 = c.sr + c.wor;
    ss2 = c.ss + c.wos;
  } else {  // graph.cu:1414-1426, with a self-loop moving (r,r) -> (s,s)
    const int32_t wor_ = c.wor - c.wself, wir_ = c.wir - c.wself;
    rr2 = c.rr - wor_ - c.wself - wir_;
    rs2 = c.rs - c.wos + wir_;
    sr2 = c.sr + wor_ - c.wis;
    ss2 = c.ss + c.wos + c.wis + c.wself;
  }
  const int32_t Wo = c.k_out - c.wor - c.wos, Wi = c.k_in - c.wir - c.wis;
  const int32_t Xr = c.dor - c.rr - c.rs, Xs = c.dos - c.sr - c.ss;
  const int32_t Yr = c.dir - c.rr - c.sr, Ys = c.dis - c.rs - c.ss;
  if (rr2 < 0 || rs2 < 0 || sr2 < 0 || ss2 < 0 || Xr - Wo < 0 || Yr - Wi < 0)
    atomicOr(&a.status->flags, kFlagNegative);
  const bool col = lane & 1, row = lane & 2, now = lane & 4, deg = lane & 8;
  const bool in2 = deg ? row : col;  // whose d_in
  const int32_t dout = (row ? c.dos : c.dor) + (now ? (row ? c.k_out : -c.k_out) : 0);
  const int32_t din = (in2 ? c.dis : c.dir) + (now ? (in2 ? c.k_in : -c.k_in) : 0);
  const int32_t mt = now ? (row ? (col ? ss2 : sr2) : (col ? rs2 : rr2))
                         : (row ? (col ? c.ss : c.sr) : (col ? c.rs : c.rr));
  const int32_t dW = now ? (col ? Wi : Wo) : 0;
  const int32_t mp = (col ? (row ? Ys : Yr) : (row ? Xs : Xr)) + (row ? dW : -dW);
  const int32_t m = deg ? mp : mt;
  // lambda(0) = 0 stands for what a degree term lacks (the table may end there)
  const int32_t d1 = deg && !col ? dout : din, d2 = deg ? 0 : dout;
  const bool bad = d1 <= 0 || (!deg && d2 <= 0);
  int64_t L;
  if (!s_lam || __ballot(lane < 16 && max(max(deg ? 0 : m, d1), d2) >= kLamLds))
    L = lam_of(a.lam, deg ? 0 : m) - lam_of(a.lam, d1) - lam_of(a.lam, d2);
  else  // lanes past 15 read in range too
    L = s_lam[min(max(deg ? 0 : m, 0), kLamLds - 1)] - s_lam[min(max(d1, 0), kLamLds - 1)] -
        s_lam[min(max(d2, 0), kLamLds - 1)];
  if (lane < 16) {
    const int32_t mm = bad ? 0 : max(m, 0);
    acc_add(acc, now ? -mm : mm, L);
  }
  inf = __ballot(lane < 16 && now && bad && m > 0) != 0;
}

// The result of one proposal.
struct Nodal {
  int32_t s, u, acc;
  bool inf;
  i128 dS;
  long bytes;  // algorithmic bytes (profiling)
};

// Adds unit (b, w, in) of a node moving r -> s to acc: its edges to (in: from)
// block b, given block row r's and row s's counts of b.  Branch-free: w = 0
// with zero counts adds nothing.
__device__ __forceinline__ void unit_terms(Acc& acc, const int64_t L[4], int32_t mr, int32_t ms,
                                           int32_t w) {
  acc_add(acc, max(mr, 0), L[0]);
  acc_add(acc, max(ms, 0), L[1]);
  acc_add(acc, -max(mr - w, 0), L[2]);
  acc_add(acc, -max(ms + w, 0), L[3]);
}

constexpr int kLdsWave = 1024;     // LDS ints per wavefront: a unit table, or one key bucket
constexpr int kRegUnits = 4;       // list entries per lane of a node one wavefront handles
constexpr uint32_t kNoUnit = ~0u;  // empty unit-table slot

__device__ __forceinline__ uint32_t unit_key(int32_t b, bool in) {
  return 2u * (uint32_t)b + (in ? 1u : 0u);
}

// One nodal proposal (graph_parallel.hpp:990-1222) by one wavefront, for a
// node of at most 64 U list entries.  A lane holds U entries; those that share
// a block and a direction are summed into one of them, the unit's owner, by
// a hash table in LDS that only decides ownership and sums weights: the unit
// itself, its lookups and its terms stay in the owner's registers.
//
// The kernel is bound by its chain of dependent loads, so each step's are in
// flight together: the list, with r's row header and degrees and those of the
// uniform draw's block; the entries' labels (the drawn neighbour's among
// them); then
//   M dense: row r's counts of every entry's block, the drawn block's degrees
//     and its row's weights (it decides the proposal most often); then s's
//     counts and degrees;
//   M hashed (B is then at least 16 times a row's degree, so the uniform draw
//     is nearly always the proposal): 8-key windows of row r and of the uniform
//     block's row for every entry's block -- the keys alone of a block that
//     most often has none of them, and one round of loads for nearly every
//     probe chain, where slot by slot the longest of 64 lanes' chains took
//     three or four; then the counts found there;
// then the lambda table (hashed rows' counts are small: its first entries are
// in LDS).  Launch averages against one path through an LDS table with row
// headers always read (90 VGPRs, 40 KB of LDS a workgroup, Philox in every
// lane): N = 1000 12.1 -> 5.8 us, N = 20000 (5000-node batches) 28.8 -> 9.8, N =
// 50000 (12500-node batches) 42.5 -> 15.8, 4096-node batches at B = 100000 28.8
// -> 17.5 and at B = 250000 29.2 -> 21.9 (20.1 and 27.3 with single slots and
// the whole lambda table).  Registers: dense 96 VGPRs, none spilled but one with
// hub code; hashed all 128 that four wavefronts a SIMD leave, where U = 4 with its
// windows spills 2 with hub code, 19 weighted and 24 both (60 bytes a lane; hub
// code also spills 99 to 145 scalar registers to vector ones).  A weighted sweep
// on hashed rows takes 4-7% longer than an unweighted one all the same (N = 50000,
// B = 25000, 4096-node batches 623 and 596 us).
template <bool kD, bool kW, int U>
__device__ __forceinline__ void nodal_regs(const NodalArgs& a, int32_t n, int32_t r, int64_t o0,
                                           int64_t i0, int32_t kco, int32_t kc,
                                           const uint64_t x[4], int32_t* lds,
                                           const int64_t* s_lam, Nodal& out) {
  const int lane = lane_id();
  const GraphView& g = a.g;
  const MView& M = a.M;
  const int32_t B = a.B;
  const Row rM = m_row<kD>(M, r);
  const int32_t dor = a.d_out[r], dir = a.d_in[r];
  const int32_t s_pre = (int32_t)idx32(x[2], (uint32_t)B);
  const Row pM = m_row<kD>(M, s_pre);
  const int32_t dos_pre = a.d_out[s_pre], dis_pre = a.d_in[s_pre];
  int32_t v[U], w[U];
#pragma unroll
  for (int q = 0; q < U; ++q) {
    const int32_t j = q * kWave + lane;
    v[q] = -1;
    w[q] = kW ? 0 : 1;
    if (j < kco) {
      v[q] = g.out_idx[o0 + j];
      if (kW) w[q] = g.out_w[o0 + j];
    } else if (j < kc) {
      v[q] = g.in_idx[i0 + (j - kco)];
      if (kW) w[q] = g.in_w[i0 + (j - kco)];
    }
  }
  constexpr int kCap = 128 * U;  // at least twice the units
  static_assert(2 * kCap <= kLdsWave, "unit table exceeds the wavefront's LDS");
  uint32_t* tk = reinterpret_cast<uint32_t*>(lds);
  int32_t* tw = lds + kCap;
  for (int j = 4 * lane; j < 2 * kCap; j += 4 * kWave) {
    const int32_t z = j < kCap ? -1 : 0;
    *reinterpret_cast<int4*>(lds + j) = make_int4(z, z, z, z);
  }
  lds_order();
  // n's weights, and unit t of its list (graph_parallel.hpp:1010-1027)
  int32_t k_out = kco, k_in = kc - kco;
  if (kW) {
    uint32_t so = 0, si = 0;
#pragma unroll
    for (int q = 0; q < U; ++q) (q * kWave + lane < kco ? so : si) += (uint32_t)w[q];
    k_out = (int32_t)wave_sum32(so);
    k_in = (int32_t)wave_sum32(si);
  }
  const uint32_t k = (uint32_t)k_out + (uint32_t)k_in;
  int pq = 0, pl = 0;
  if (k > 0) {
    const uint32_t t = idx32(x[0], k);
    if (!kW) {
      pq = (int)(t / kWave);
      pl = (int)(t % kWave);
    } else {
      uint32_t sum = 0;
      bool found = false;
#pragma unroll
      for (int q = 0; q < U; ++q) {
        const uint32_t inc = wave_incl_scan32((uint32_t)w[q]);
        const unsigned long long hit = __ballot(sum + inc > t);
        if (!found && hit) {
          found = true;
          pq = q;
          pl = __ffsll(hit) - 1;
        }
        sum += read_lane32(inc, kWave - 1);
      }
    }
  }
  int32_t lb[U];
#pragma unroll
  for (int q = 0; q < U; ++q) lb[q] = v[q] >= 0 ? a.labels[v[q]] : -1;
  int32_t lv = lb[0];
#pragma unroll
  for (int q = 1; q < U; ++q) lv = pq == q ? lb[q] : lv;
  const int32_t u = k > 0 ? __builtin_amdgcn_readlane(lv, pl) : r;
  const uint32_t da = (uint32_t)a.d_out[u] + (uint32_t)a.d_in[u];
  Sums bk;
  if (kD) bk = load_sums(M, u, m_row<kD>(M, u));
  // row r's and row s's counts of the unit's block, in its direction: o, or i
  // for an in-edge
  int32_t m0[U], m1[U];
  auto count = [&](Row R, int32_t h, int q) {
    return reinterpret_cast<const int32_t*>(M.cnt + R.o + h)[q * kWave + lane >= kco];
  };
#pragma unroll
  for (int q = 0; q < U; ++q) m0[q] = m1[q] = 0;
  Cnt cRR{0, 0}, cRS{0, 0}, cSS{0, 0};
  // hashed: the windows of kG units a lane at a time, and, with the first
  // ones, the corner's in lanes 0 (row r, key r), 1 (r, s), 2 (s, s)
  constexpr int kG = U == 2 ? 2 : 1;
  const bool rdir = kD || __builtin_amdgcn_readfirstlane(rM.c) == B;
  Window wr[kG], ws[kG], wc;
  auto corner_row = [&](Row sM) { return lane < 2 ? rM : sM; };
  auto corner_key = [&](int32_t s) { return lane == 0 ? r : s; };
  auto issue = [&](int q0, Row sM, bool sdir, bool with_r) {
#pragma unroll
    for (int i = 0; i < kG; ++i) {
      const int32_t b = max(lb[q0 + i], 0);  // an absent entry reads block 0's
      if (with_r) wr[i] = win_issue(M, rM, b, rdir);
      ws[i] = win_issue(M, sM, b, sdir);
    }
  };
  if (kD) {
#pragma unroll
    for (int q = 0; q < U; ++q)
      if (v[q] >= 0) m0[q] = count(rM, lb[q], q);
    cRR = M.cnt[rM.o + r];
  }
  const bool pdir = kD || __builtin_amdgcn_readfirstlane(pM.c) == B;
  if (!kD) {
    issue(0, pM, pdir, true);
    const Row cM = corner_row(pM);
    wc = win_issue(M, cM, corner_key(s_pre), cM.c == B);
  }
  // units: the owner of each (block, direction), its summed weight; every
  // entry's first claim before any is resolved
  uint32_t hs[U], old[U];
  bool own[U];
#pragma unroll
  for (int q = 0; q < U; ++q) {
    const uint32_t key = unit_key(lb[q], q * kWave + lane >= kco);
    hs[q] = hash32((int32_t)key) & (kCap - 1);
    old[q] = key;
    if (v[q] >= 0) old[q] = atomicCAS(&tk[hs[q]], kNoUnit, key);
  }
#pragma unroll
  for (int q = 0; q < U; ++q) {
    own[q] = false;
    if (v[q] >= 0) {
      const uint32_t key = unit_key(lb[q], q * kWave + lane >= kco);
      own[q] = old[q] == kNoUnit;
      while (!own[q] && old[q] != key) {
        hs[q] = (hs[q] + 1) & (kCap - 1);
        old[q] = atomicCAS(&tk[hs[q]], kNoUnit, key);
        own[q] = old[q] == kNoUnit;
      }
      atomicAdd(&tw[hs[q]], w[q]);
    }
  }
  lds_order();
  int32_t wself = 0;
  if (a.exact) {
    uint32_t sum = 0;
#pragma unroll
    for (int q = 0; q < U; ++q)
      if (q * kWave + lane < kco && v[q] == n) sum += (uint32_t)w[q];
    if (__ballot(sum != 0)) wself = (int32_t)wave_sum32(sum);  // self-loops are rare
  }
#pragma unroll
  for (int q = 0; q < U; ++q) w[q] = own[q] ? tw[hs[q]] : 0;
  lds_order();  // the table's LDS may hold a key bucket next
  // list offsets, own label, outputs (s, dS, inf, accept, r) (+ weights)
  long bytes = 32 + 4 + 32 + (kW ? 4 * (long)kc : 0);
  int32_t s = s_pre;
  if (k > 0) {
    bytes += 16;  // drawn neighbour id, its label, d_out[u], d_in[u]
    if (!usap::uniform_branch(x[1], da, B))
      s = select_combined<kD>(M, u, idx32(x[3], da), -1, kD ? &bk : nullptr, lds, kLdsWave, bytes);
  }
  out.s = s;
  out.u = k > 0 ? u : -1;
  out.acc = 0;
  out.inf = false;
  out.dS = 0;
  if (s == r) {
    out.bytes = bytes;
    return;
  }
  const bool pre = s == s_pre;
  const Row sM = pre ? pM : m_row<kD>(M, s);
  const int32_t dos = pre ? dos_pre : a.d_out[s], dis = pre ? dis_pre : a.d_in[s];
  const bool sdir = kD || __builtin_amdgcn_readfirstlane(sM.c) == B;
  // blocks r and s own one unit each per direction at most
  int32_t wor = 0, wir = 0, wos = 0, wis = 0, units = 0;
#pragma unroll
  for (int q = 0; q < U; ++q) {
    const bool in = q * kWave + lane >= kco;
    const bool isr = own[q] && lb[q] == r, iss = own[q] && lb[q] == s;
    if (__ballot(isr)) {
      const unsigned long long o = __ballot(isr && !in), i = __ballot(isr && in);
      if (o) wor = __builtin_amdgcn_readlane(w[q], __ffsll(o) - 1);
      if (i) wir = __builtin_amdgcn_readlane(w[q], __ffsll(i) - 1);
    }
    if (__ballot(iss)) {
      const unsigned long long o = __ballot(iss && !in), i = __ballot(iss && in);
      if (o) wos = __builtin_amdgcn_readlane(w[q], __ffsll(o) - 1);
      if (i) wis = __builtin_amdgcn_readlane(w[q], __ffsll(i) - 1);
    }
    own[q] = own[q] && !isr && !iss;
    units += __popcll(__ballot(own[q]));
  }
  if (kD) {
#pragma unroll
    for (int q = 0; q < U; ++q) {
      if (own[q])
        m1[q] = count(sM, lb[q], q);
      else
        m0[q] = 0;
    }
    cRS = M.cnt[rM.o + s];
    cSS = M.cnt[sM.o + s];
  } else {
    if (!pre) {
      issue(0, sM, sdir, false);
      const Row cM = corner_row(sM);
      wc = win_issue(M, cM, corner_key(s), cM.c == B);
    }
#pragma unroll
    for (int q0 = 0; q0 < U; q0 += kG) {
      if (q0 > 0) issue(q0, sM, sdir, true);
      uint32_t hr[kG], hq[kG];
      int32_t kr[kG], kq[kG];
#pragma unroll
      for (int i = 0; i < kG; ++i) {
        const int32_t b = max(lb[q0 + i], 0);
        hr[i] = win_end(wr[i], b, rdir, kr[i]);
        hq[i] = win_end(ws[i], b, sdir, kq[i]);
        if (!own[q0 + i]) kr[i] = kq[i] = -1;
        if (own[q0 + i] && kr[i] == b) m0[q0 + i] = count(rM, (int32_t)hr[i], q0 + i);
        if (own[q0 + i] && kq[i] == b) m1[q0 + i] = count(sM, (int32_t)hq[i], q0 + i);
      }
      if (q0 == 0) {  // the corner
        const Row cM = corner_row(sM);
        const int32_t ck = corner_key(s);
        int32_t kk;
        const uint32_t h = win_end(wc, ck, cM.c == B, kk);
        Cnt c{0, 0};
        if (lane < 3) {
          if (kk == ck)
            c = M.cnt[cM.o + h];
          else if (kk >= 0)
            c = m_value_more(M, cM, ck, h);
        }
        cRR = Cnt{__builtin_amdgcn_readlane(c.o, 0), __builtin_amdgcn_readlane(c.i, 0)};
        cRS = Cnt{__builtin_amdgcn_readlane(c.o, 1), __builtin_amdgcn_readlane(c.i, 1)};
        cSS = Cnt{__builtin_amdgcn_readlane(c.o, 2), __builtin_amdgcn_readlane(c.i, 2)};
      }
#pragma unroll
      for (int i = 0; i < kG; ++i) {  // chains past a window
        const int32_t b = lb[q0 + i];
        const bool in = (q0 + i) * kWave + lane >= kco;
        if (kr[i] >= 0 && kr[i] != b) {
          const Cnt y = m_value_more(M, rM, b, hr[i]);
          m0[q0 + i] = in ? y.i : y.o;
        }
        if (kq[i] >= 0 && kq[i] != b) {
          const Cnt y = m_value_more(M, sM, b, hq[i]);
          m1[q0 + i] = in ? y.i : y.o;
        }
      }
    }
  }
  // ids + labels (+ weights); rows (offset + capacity) and degrees of r and s;
  // 2 block-row lookups (key + two counts) per unit and 3 corner lookups
  bytes += (kW ? 12 : 8) * (long)kc + 24 + 16 + 12 * (long)(2 * units + 3);
  out.bytes = bytes;
  Acc acc{0, 0};
  int64_t L[U][4];
  bool neg = false, big = kD;
#pragma unroll
  for (int q = 0; q < U; ++q) {
    if (!own[q]) w[q] = 0;
    neg |= m0[q] < w[q];
    big |= max(m0[q], m1[q] + w[q]) >= kLamLds;
  }
  if (!kD) big = __ballot(big) != 0;
#pragma unroll
  for (int q = 0; q < U; ++q) {
    L[q][0] = lam_at(a.lam, s_lam, big, m0[q]);
    L[q][1] = lam_at(a.lam, s_lam, big, m1[q]);
    L[q][2] = lam_at(a.lam, s_lam, big, m0[q] - w[q]);
    L[q][3] = lam_at(a.lam, s_lam, big, m1[q] + w[q]);
  }
  const Corner c{cRR.o, cRS.o, cRS.i, cSS.o, dor, dir, dos, dis,
                 k_out, k_in, wor, wir, wos, wis, wself};
  corner_terms(a, c, kD ? nullptr : s_lam, acc, out.inf);
#pragma unroll
  for (int q = 0; q < U; ++q) unit_terms(acc, L[q], m0[q], m1[q], w[q]);
  if (neg) atomicOr(&a.status->flags, kFlagNegative);
  acc.h = wave_sum(acc.h);
  acc.l = wave_sum(acc.l);
  out.dS = acc_value(acc);
  out.acc = (out.inf || out.dS < 0) ? 1 : 0;
}

// Workgroup scratch of nodal_hub.
struct HubShared {
  long h[kNodalWaves], l[kNodalWaves];
  uint32_t sum[2];
  int32_t s, u, units, wself;
  int32_t w[4];  // weights into r (out, in) and s (out, in)
  long bytes;
};

// The unit table of a node a whole workgroup handles: in LDS, or, when its
// units may exceed that, in the node's global table.  Slots are read by
// relaxed atomic loads (the table may sit in global memory, where the atomics
// that build it bypass the CU's cache).
constexpr int kHubCap = kNodalWaves * kLdsWave / 2;  // slots of the LDS table
constexpr int kHubUnits = kHubCap * 3 / 4;

template <bool kD, bool kW, bool kBig>
__device__ __forceinline__ void hub_terms(const NodalArgs& a, int32_t n, int32_t r, int32_t s,
                                          int64_t o0, int64_t i0, int32_t kco, int32_t kc,
                                          int32_t* lds, HubShared& hub, Row rM, Row sM, Acc& acc) {
  const GraphView& g = a.g;
  const MView& M = a.M;
  int32_t cap = kHubCap;
  uint32_t* tk = reinterpret_cast<uint32_t*>(lds);
  int32_t* tw = lds + kHubCap;
  if (kBig) {
    cap = 1;
    while (cap < 2 * kc) cap <<= 1;
    tk = reinterpret_cast<uint32_t*>(a.big_tab + a.big_off[n]);
    tw = a.big_tab + a.big_off[n] + cap;
  }
  const uint32_t mask = (uint32_t)cap - 1;
  for (int32_t i = threadIdx.x; i < cap; i += blockDim.x) {
    tk[i] = kNoUnit;
    tw[i] = 0;
  }
  __syncthreads();
  uint32_t ws = 0;
  constexpr int kQ = 2;  // entries and slots in flight per thread
#pragma unroll 1
  for (int32_t base = threadIdx.x; base < kc; base += kQ * blockDim.x) {
    int32_t v[kQ], w[kQ], lb[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q)
      list_entry(g, o0, kco, i0, kc, base + q * (int32_t)blockDim.x, v[q], w[q]);
#pragma unroll
    for (int q = 0; q < kQ; ++q) lb[q] = v[q] >= 0 ? a.labels[v[q]] : -1;
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      if (v[q] < 0) continue;
      const bool in = base + q * (int32_t)blockDim.x >= kco;
      if (!in && v[q] == n) ws += (uint32_t)w[q];
      const uint32_t key = unit_key(lb[q], in);
      uint32_t h = hash32((int32_t)key) & mask;
      for (;;) {
        const uint32_t old = atomicCAS(&tk[h], kNoUnit, key);
        if (old == kNoUnit || old == key) break;
        h = (h + 1) & mask;
      }
      atomicAdd(&tw[h], w[q]);
    }
  }
  if (ws) atomicAdd(reinterpret_cast<uint32_t*>(&hub.wself), ws);
  __syncthreads();
  bool neg = false;
#pragma unroll 1
  for (int32_t base = threadIdx.x; base < cap; base += kQ * (int32_t)blockDim.x) {
    uint32_t key[kQ];
    int32_t w[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int32_t i = base + q * (int32_t)blockDim.x;
      key[q] = kNoUnit;
      w[q] = 0;
      if (i < cap) {
        key[q] = __hip_atomic_load(&tk[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        w[q] = __hip_atomic_load(&tw[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    Probe p0[kQ], p1[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int32_t b = (int32_t)(key[q] >> 1);
      if (key[q] == kNoUnit) continue;
      if (b == r || b == s) {
        hub.w[2 * (b == s) + (int)(key[q] & 1u)] = w[q];
        key[q] = kNoUnit;
        continue;
      }
      p0[q] = m_probe<kD>(M, rM, b);
      p1[q] = m_probe<kD>(M, sM, b);
    }
    int32_t m0[kQ], m1[kQ];
    int64_t L[kQ][4];
    int32_t live = 0;
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      m0[q] = m1[q] = 0;
      if (key[q] != kNoUnit) {
        const int32_t b = (int32_t)(key[q] >> 1);
        const Cnt cr = m_value<kD>(M, rM, b, p0[q]), cs = m_value<kD>(M, sM, b, p1[q]);
        const bool in = key[q] & 1u;
        m0[q] = in ? cr.i : cr.o;
        m1[q] = in ? cs.i : cs.o;
        ++live;
      } else {
        w[q] = 0;
      }
      neg |= m0[q] < w[q];
      L[q][0] = lam_of(a.lam, m0[q]);
      L[q][1] = lam_of(a.lam, m1[q]);
      L[q][2] = lam_of(a.lam, m0[q] - w[q]);
      L[q][3] = lam_of(a.lam, m1[q] + w[q]);
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) unit_terms(acc, L[q], m0[q], m1[q], w[q]);
    if (a.tstamp && live) atomicAdd(&hub.units, live);
  }
  if (neg) atomicOr(&a.status->flags, kFlagNegative);
}

// One nodal proposal by the whole workgroup, for a node with more list entries
// than a wavefront's registers take (one wavefront alone set the length of the
// launch: N = 3001 with four 1200-entry hubs 50.6 -> 13.9 us a launch).
// The first wavefront draws; the result is in thread 0's out.
template <bool kD, bool kW>
__device__ __forceinline__ void nodal_hub(const NodalArgs& a, int32_t n, int32_t* lds,
                                          HubShared& hub, Nodal& out) {
  const int lane = lane_id(), w = threadIdx.x / kWave;
  const GraphView& g = a.g;
  const MView& M = a.M;
  const int32_t B = a.B;
  const int32_t r = a.labels[n];
  const int64_t o0 = g.out_ptr[n], i0 = g.in_ptr[n];
  const int32_t kco = (int32_t)(g.out_ptr[n + 1] - o0);
  const int32_t kc = kco + (int32_t)(g.in_ptr[n + 1] - i0);
  uint64_t x[4];
  predrawn(a.draws, (a.predrawn ? a.sweep->stream0 : 0) + (uint64_t)n, x);
  if (threadIdx.x == 0) {
    hub.sum[0] = hub.sum[1] = 0;
    hub.units = hub.wself = 0;
    hub.w[0] = hub.w[1] = hub.w[2] = hub.w[3] = 0;
  }
  __syncthreads();
  int32_t k_out = kco, k_in = kc - kco;
  if (kW) {
    uint32_t so = 0, si = 0;
    for (int32_t j = threadIdx.x; j < kc; j += blockDim.x) {
      if (j < kco)
        so += (uint32_t)g.out_w[o0 + j];
      else
        si += (uint32_t)g.in_w[i0 + (j - kco)];
    }
    so = wave_sum32(so);
    si = wave_sum32(si);
    if (lane == 0) {
      atomicAdd(&hub.sum[0], so);
      atomicAdd(&hub.sum[1], si);
    }
    __syncthreads();
    k_out = (int32_t)hub.sum[0];
    k_in = (int32_t)hub.sum[1];
  }
  const uint32_t k = (uint32_t)k_out + (uint32_t)k_in;
  if (w == 0) {
    long bytes = 32 + 4 + 32 + (kW ? 4 * (long)kc : 0);
    int32_t u = -1, s = (int32_t)idx32(x[2], (uint32_t)B);
    if (k > 0) {
      u = a.labels[pick_neighbor(g, o0, kco, i0, kc - kco, (int64_t)idx32(x[0], k))];
      const uint32_t da = (uint32_t)a.d_out[u] + (uint32_t)a.d_in[u];
      bytes += 16;
      if (!usap::uniform_branch(x[1], da, B))
        s = select_combined<kD>(M, u, idx32(x[3], da), -1, nullptr, lds, kLdsWave, bytes);
    }
    if (lane == 0) {
      hub.s = s;
      hub.u = u;
      hub.bytes = bytes;
    }
  }
  __syncthreads();
  const int32_t s = hub.s;
  out.s = s;
  out.u = hub.u;
  out.acc = 0;
  out.inf = false;
  out.dS = 0;
  out.bytes = hub.bytes;
  if (s == r) return;  // the same for every thread
  const Row rM = m_row<kD>(M, r), sM = m_row<kD>(M, s);
  Acc acc{0, 0};
  const int64_t most = min((int64_t)kc, 2 * (int64_t)B);  // units
  if (most <= kHubUnits)
    hub_terms<kD, kW, false>(a, n, r, s, o0, i0, kco, kc, lds, hub, rM, sM, acc);
  else
    hub_terms<kD, kW, true>(a, n, r, s, o0, i0, kco, kc, lds, hub, rM, sM, acc);
  acc.h = wave_sum(acc.h);
  acc.l = wave_sum(acc.l);
  if (lane == 0) {
    hub.h[w] = acc.h;
    hub.l[w] = acc.l;
  }
  __syncthreads();
  if (w == 0) {
    const Cnt crs = m_value<kD>(M, rM, s, m_probe<kD>(M, rM, s));
    const Corner c{m_value<kD>(M, rM, r, m_probe<kD>(M, rM, r)).o, crs.o, crs.i,
                   m_value<kD>(M, sM, s, m_probe<kD>(M, sM, s)).o,
                   a.d_out[r], a.d_in[r], a.d_out[s], a.d_in[s], k_out, k_in,
                   hub.w[0], hub.w[1], hub.w[2], hub.w[3], hub.wself};
    Acc t{0, 0};
    corner_terms(a, c, nullptr, t, out.inf);
    t.h = wave_sum(t.h);
    t.l = wave_sum(t.l);
    for (int i = 0; i < kNodalWaves; ++i) {
      t.h += hub.h[i];
      t.l += hub.l[i];
    }
    out.dS = acc_value(t);
    out.acc = (out.inf || out.dS < 0) ? 1 : 0;
    out.bytes += (kW ? 12 : 8) * (long)kc + 24 + 16 + 12 * (long)(2 * hub.units + 3);
  }
}

// Batch nodes [beg, end), four to a workgroup, one wavefront each; nodes too
// large for a wavefront are left to the whole workgroup afterwards (kHub: the
// graph has such nodes; their code costs registers).
template <bool kD, bool kW, bool kHub>
__global__ __launch_bounds__(kWave* kNodalWaves, kD ? 5 : 4) void k_nodal(NodalArgs a) {
  __shared__ __align__(16) int32_t s_lds[kNodalWaves][kLdsWave];
  __shared__ unsigned long long s_p[kNodalWaves][6];
  __shared__ int32_t s_large[kNodalWaves];
  __shared__ int64_t s_lam[kD ? 1 : kLamLds];
  const int w = threadIdx.x / kWave;
  if (a.tstamp && threadIdx.x == 0) a.tstamp[blockIdx.x] = wall_clock64();
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.M.gst->ovf_n = 0;  // the previous k_grow replayed the parked increments
    // k_apply decides by this copy whether the batch runs: its block 0
    // updates stop meanwhile
    a.sweep->stop_n = a.sweep->stop;
  }
  const int64_t item0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * kNodalWaves;
  const int64_t item = item0 + w;
  const int64_t n64 = (int64_t)a.beg + item;
  // this node's proposal to memory, and its share of the batch sums: accepted
  // moves, the exact sum of their finite dS, the -inf ones, byte tallies
  auto store = [&](int64_t it, int wv, int32_t r, int32_t kc, const Nodal& p) {
    a.prop[it] = Prop{p.s, r, p.acc, p.inf ? -1 : 0};
    a.prop_ds[it] = PropDs{(long)(p.dS >> 64), (unsigned long)(u128)p.dS};
    if (a.prop_u) a.prop_u[it] = p.u;
    const u128 d = (p.acc && !p.inf) ? (u128)p.dS : (u128)0;
    s_p[wv][0] = (unsigned long long)p.bytes;
    s_p[wv][1] = p.acc ? (unsigned long long)apply_tally(kc) : 0ull;
    s_p[wv][2] = (unsigned long long)d;
    s_p[wv][3] = (unsigned long long)(d >> 64);
    s_p[wv][4] = (unsigned long long)p.acc;
    s_p[wv][5] = (unsigned long long)(p.acc && p.inf);
  };
  bool large = false;
  if (lane_id() == 0)
    for (int i = 0; i < 6; ++i) s_p[w][i] = 0;
  // the sweep's stop flag and lambda's first entries are read together with the
  // node's first loads
  static_assert(kLamLds == kWave * kNodalWaves, "one entry per thread");
  int64_t lam = 0;
  if (!kD) lam = a.lam[min((int32_t)threadIdx.x, a.lam_last)];
  const bool in = n64 < a.end;
  const int32_t n = in ? (int32_t)n64 : a.beg;
  const int32_t stop = a.sweep->stop;
  uint64_t x[4];
  predrawn(a.draws, (a.predrawn ? a.sweep->stream0 : 0) + (uint64_t)n, x);
  const int32_t r = a.labels[n];
  const int64_t o0 = a.g.out_ptr[n], i0 = a.g.in_ptr[n];
  const int64_t kco = a.g.out_ptr[n + 1] - o0, kc = kco + (a.g.in_ptr[n + 1] - i0);
  if (!kD) {
    s_lam[threadIdx.x] = lam;
    __syncthreads();
  }
  if (in && !stop) {
    large = kHub && kc > kRegUnits * kWave;
    if (!large) {
      Nodal p;
      const int32_t ko = (int32_t)kco, kk = (int32_t)kc;
      if (kk <= kWave)
        nodal_regs<kD, kW, 1>(a, n, r, o0, i0, ko, kk, x, s_lds[w], s_lam, p);
      else if (kk <= 2 * kWave)
        nodal_regs<kD, kW, 2>(a, n, r, o0, i0, ko, kk, x, s_lds[w], s_lam, p);
      else
        nodal_regs<kD, kW, kRegUnits>(a, n, r, o0, i0, ko, kk, x, s_lds[w], s_lam, p);
      if (lane_id() == 0) store(item, w, r, kk, p);
    }
  }
  if (kHub && lane_id() == 0) s_large[w] = large;
  __syncthreads();  // every wavefront is done with its LDS
  if (kHub) {
    __shared__ HubShared s_hub;
    for (int i = 0; i < kNodalWaves; ++i) {
      if (!s_large[i]) continue;
      const int32_t n = (int32_t)((int64_t)a.beg + item0 + i);
      Nodal p;
      nodal_hub<kD, kW>(a, n, &s_lds[0][0], s_hub, p);
      if (threadIdx.x == 0)
        store(item0 + i, i, a.labels[n],
              (int32_t)((a.g.out_ptr[n + 1] - a.g.out_ptr[n]) + (a.g.in_ptr[n + 1] - a.g.in_ptr[n])),
              p);
      __syncthreads();
    }
  }
  if (threadIdx.x == 0) {
    unsigned long long nb = 0, ab = 0;
    u128 sum = 0;
    int32_t moves = 0, ninf = 0;
    for (int i = 0; i < kNodalWaves; ++i) {
      nb += s_p[i][0];
      ab += s_p[i][1];
      sum += ((u128)s_p[i][3] << 64) | (u128)s_p[i][2];
      moves += (int32_t)s_p[i][4];
      ninf += (int32_t)s_p[i][5];
    }
    BlockPart& P = a.part[blockIdx.x];
    P.sum_lo = (unsigned long)sum;
    P.sum_hi = (long)(sum >> 64);
    P.nodal_bytes = nb;
    P.apply_bytes = ab;
    P.moves = moves;
    P.ninf = ninf;
    if (a.tstamp) a.tstamp[a.tstride + blockIdx.x] = wall_clock64();
  }
}

// Profiling only: the compulsory bytes of the reference's algorithm for one
// nodal batch, from the batch's own proposals.  graph_parallel.hpp:990-1222
// reads, per node n, its list offsets (16), label (4), neighbour ids and
// labels (8 k_n, + 4 k_n weights) and writes s and dS (12); per distinct
// block b among the batch's old blocks r_n, proposed blocks s_n and drawn
// neighbours' blocks u_n, row and column b of M whole (16 + 8 nnzR(b) +
// 8 nnzC(b)) and its degrees (12); per accepted move, the label (4) and two
// 8-byte read-modify-writes per list entry (16 k_n).  A block counts once per
// batch: the first wavefront to raise its mark to the batch's stamp counts
// the non-zeros of its block row (o > 0: row b, i > 0: column b).  One
// wavefront per batch node; each workgroup adds its per-node bytes to
// acc[2 j] and its block bytes to acc[2 j + 1], j = workgroup % kAqSlots
// (spread over slots: one address would serialise the whole grid's adds).
constexpr int kAqSlots = 64;
struct AqArgs {
  GraphView g;
  MView M;
  int32_t beg, end;
  const Prop* prop;
  const int32_t* prop_u;
  int32_t* mark;
  int32_t stamp;
  const Sweep* sweep;
  unsigned long long* acc;
};

__global__ __launch_bounds__(kWave* kNodalWaves) void k_aq(AqArgs a) {
  const int lane = lane_id();
  const int64_t item = (int64_t)blockIdx.x * kNodalWaves + threadIdx.x / kWave;
  const int64_t n64 = (int64_t)a.beg + item;
  const bool live = n64 < a.end && a.sweep->stop_n == 0;  // uniform per wavefront
  const int32_t n = live ? (int32_t)n64 : a.beg;
  const int64_t kc =
      live ? (a.g.out_ptr[n + 1] - a.g.out_ptr[n]) + (a.g.in_ptr[n + 1] - a.g.in_ptr[n]) : 0;
  int32_t b = -1;
  if (live && lane == 0) b = a.prop[item].r;
  if (live && lane == 1) b = a.prop[item].s;
  if (live && lane == 2) b = a.prop_u[item];
  const bool first = b >= 0 && atomicMax(&a.mark[b], a.stamp) < a.stamp;
  unsigned long long rows = __ballot(first);
  unsigned long long blk = 0;
  while (rows) {
    const int l = __ffsll(rows) - 1;
    rows &= rows - 1ull;
    const int32_t bb = __shfl(b, l);
    const int64_t o = a.M.off[bb];
    const int32_t c = a.M.cap[bb];
    long nz = 0;
    for (int32_t j = lane; j < c; j += kWave) {
      const Cnt q = a.M.cnt[o + j];
      nz += (q.o > 0 ? 1 : 0) + (q.i > 0 ? 1 : 0);
    }
    blk += 16 + 8 * (unsigned long long)wave_sum(nz) + 12;
  }
  __shared__ unsigned long long s_node[kNodalWaves], s_blk[kNodalWaves];
  const int w = threadIdx.x / kWave;
  if (lane == 0) {
    unsigned long long node = 0;
    if (live) {
      node = 16 + 4 + 8 * (unsigned long long)kc + 12;
      if (a.g.out_w) node += 4 * (unsigned long long)kc;
      if (a.prop[item].acc) node += 4 + 16 * (unsigned long long)kc;
    }
    s_node[w] = node;
    s_blk[w] = blk;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long node = 0, bsum = 0;
    for (int i = 0; i < kNodalWaves; ++i) {
      node += s_node[i];
      bsum += s_blk[i];
    }
    const int j = (int)(blockIdx.x % kAqSlots);
    atomicAdd(&a.acc[2 * j], node);
    if (bsum) atomicAdd(&a.acc[2 * j + 1], bsum);
  }
}

// Profiling only: 16 bytes per non-zero of M (its entry read from the row
// and from the column structure of graph_parallel.hpp:761-988), spread over
// acc[0 .. kAqSlots).
__global__ __launch_bounds__(256) void k_nnz_bytes(const Cnt* __restrict__ cnt, int64_t P,
                                                   unsigned long long* acc) {
  long c = 0;
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < P;
       j += (int64_t)gridDim.x * blockDim.x)
    c += cnt[j].o > 0 ? 1 : 0;
  c = wave_sum(c);
  if (lane_id() == 0 && c)
    atomicAdd(&acc[(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) % kAqSlots],
              16ull * (unsigned long long)c);
}

// ---------------------------------------------------------------------------
// Apply accepted moves: block rows of M, degrees, block sizes, batch sum
// (graph_parallel.hpp:433-443; equal to the rebuild from the new labels)
// ---------------------------------------------------------------------------

struct ApplyArgs {
  GraphView g;
  MView M;
  int32_t* labels;
  int32_t* d_out;
  int32_t* d_in;
  int32_t* bsize;
  int32_t beg, end;
  const Prop* prop;
  const BlockPart* part;  // k_nodal's per-workgroup shares of the batch
  uint32_t nparts;
  Status* status;
  Sweep* sweep;
  Sweep* host;    // set: this launch is the sweep's last and ends it
  HostWord done;
  unsigned long long* tstamp;  // as NodalArgs::tstamp, for this kernel
  int32_t tstride;
};

__device__ double fx_to_double_dev(i128 v) {
  const bool neg = v < 0;
  const u128 m = neg ? (u128)0 - (u128)v : (u128)v;
  const unsigned long long hi = (unsigned long long)(m >> 64), lo = (unsigned long long)m;
  const double d = ldexp((double)hi, 64 - usap::kLambdaFrac) + ldexp((double)lo, -usap::kLambdaFrac);
  return neg ? -d : d;
}

// A sweep's beginning.  Workgroup 0 stores its state: `init`, and in S, when
// from_state is set, the MDL of the current state, model + data in the same
// IEEE double operations as usap_entropy on the host.  The others make the
// Philox words of nodes [beg, end), 4 per node, batch i = [beg + i * batch, ...)
// from stream init.stream0 + i: one thread per node, where every lane of a
// node's k_nodal wavefront would compute the same 80 multiplies.
constexpr int kBeginThreads = 1024;
struct BeginArgs {
  Sweep init;
  Sweep* sweep;
  int32_t from_state;
  double model;
  EntropyIn ent;
  int32_t beg, end, batch;
  uint64_t seed;
  uint64_t* draws;
};

__device__ __forceinline__ void draw_node(int64_t n, uint64_t stream, uint64_t seed,
                                          uint64_t* draws) {
  uint64_t x[4];
  usap::philox4x64((uint64_t)n, 0, stream, usap::kTagNodal, seed, 0, x);
  ulonglong2* q = reinterpret_cast<ulonglong2*>(draws + 4 * n);
  q[0] = make_ulonglong2(x[0], x[1]);
  q[1] = make_ulonglong2(x[2], x[3]);
}

__global__ __launch_bounds__(kBeginThreads) void k_begin(BeginArgs a) {
  if (blockIdx.x == 0) {
    double S = a.init.S;
    if (a.from_state) S = a.model + fx_to_double_dev(-block_entropy(a.ent));
    if (threadIdx.x == 0) {
      *a.sweep = a.init;
      a.sweep->S = S;
    }
    return;
  }
  const int64_t i = (int64_t)(blockIdx.x - 1) * kBeginThreads + threadIdx.x;
  if (a.beg + i < a.end)
    draw_node(a.beg + i, a.init.stream0 + (uint64_t)(i / a.batch), a.seed, a.draws);
}

// The words alone, from the state's stream (captured sweeps).
__global__ void k_draw(int32_t beg, int32_t end, int32_t batch, uint64_t seed, const Sweep* sweep,
                       uint64_t* __restrict__ draws) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (beg + i < end) draw_node(beg + i, sweep->stream0 + (uint64_t)(i / batch), seed, draws);
}

// The batches' error and rebuild flags folded into the sweep's state: errors
// override convergence, which overrides a rebuild request, as the decision
// comes after the batch.
__device__ __forceinline__ void fold_flags(Status* status, Sweep* sweep, int32_t f) {
  if (f) {
    atomicOr(&sweep->flags, f);
    if (f & (kFlagMissing | kFlagNegative))
      atomicExch(&sweep->stop, 3);
    else if (f & kFlagFull)
      atomicCAS(&sweep->stop, 0, 2);
    status->flags = 0;
  }
}

// The batches' flags folded into the sweep's state, and the state copied to the
// host's pinned memory (a copy would be a launch of the runtime's own kernel),
// by one workgroup.
__device__ __forceinline__ void finish_sweep(Status* status, Sweep* sweep, Sweep* host,
                                             const HostWord& done) {
  if (threadIdx.x == 0) {
    fold_flags(status, sweep, status->flags);
    __threadfence();
  }
  __syncthreads();
  static_assert(sizeof(Sweep) % 8 == 0 && sizeof(Sweep) / 8 <= kWave, "one word per thread");
  if (threadIdx.x < sizeof(Sweep) / 8) {
    unsigned long long* w = reinterpret_cast<unsigned long long*>(sweep) + threadIdx.x;
    reinterpret_cast<unsigned long long*>(host)[threadIdx.x] =
        __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (threadIdx.x == 0) host_done(done);  // the stores above are this wavefront's
}

// After a sweep, or after a chunk of its batches, where the last k_apply did not.
__global__ __launch_bounds__(kWave) void k_finish(Status* status, Sweep* sweep, Sweep* host,
                                                  HostWord done) {
  finish_sweep(status, sweep, host, done);
}

// graph_parallel.hpp:433-458 after the moves of one batch (sum: exact sum of
// the batch's accepted finite dS, ninf: accepted -inf ones): cumulative dS of
// the sweep, S += dS_sum, the moving-average convergence test.  Same IEEE
// double operations as the host driver.  The batch's error and rebuild flags
// are k_grow's to act on (they may still be raised while this runs).
__device__ void sweep_tail(Sweep* sw, u128 sum, int32_t ninf, int32_t moves,
                           unsigned long long nbytes, unsigned long long abytes) {
  sw->nodal_bytes += nbytes;
  sw->apply_bytes += abytes;
  const u128 cum = (((u128)sw->cum_hi << 64) | sw->cum_lo) + sum;
  sw->cum_lo = (unsigned long long)cum;
  sw->cum_hi = (unsigned long long)(cum >> 64);
  if (ninf > 0) sw->cum_inf = 1;
  const double dS_sum = sw->cum_inf ? -INFINITY : fx_to_double_dev((i128)cum);
  sw->dS_last = dS_sum;
  sw->S += dS_sum;
  sw->done += 1;
  sw->moves += (unsigned long long)moves;
  if (sw->check && -sw->mean < sw->thr * sw->S) atomicExch(&sw->stop, 1);
}

// One record of an accepted move r -> s: n's edges to (wo) and from (wi) the
// neighbours of block x, or, for a neighbour that moves in the same batch, its
// edge n -> neighbour (wo) whose other end goes from block x to y (else y = x).
// Block row r at key x loses (wo, wi), row s at y gains them, row x at r loses
// (wi, wo) and row y at s gains them: four 64-bit atomics on (o, i).  M all
// direct, nothing is read for them; else the four rows' headers, then the four
// key windows, are read together before the adds.
template <bool kD>
__device__ __forceinline__ void apply_record(const ApplyArgs& a, int32_t r, int32_t s, int32_t x,
                                             int32_t y, int32_t wo, int32_t wi) {
  const MView& M = a.M;
  int32_t* flags = &a.status->flags;
  const Row rM = m_row<kD>(M, r), sM = m_row<kD>(M, s);
  const Row xM = m_row<kD>(M, x), yM = m_row<kD>(M, y);
  int64_t sl[4];
  int32_t k[4];
  k[0] = m_first_key<kD>(M, rM, x, sl[0]);
  k[1] = m_first_key<kD>(M, sM, y, sl[1]);
  k[2] = m_first_key<kD>(M, xM, r, sl[2]);
  k[3] = m_first_key<kD>(M, yM, s, sl[3]);
  m_add_at<true, kD>(M, r, rM, x, -wo, -wi, sl[0], k[0], flags);
  m_add_at<true, kD>(M, s, sM, y, wo, wi, sl[1], k[1], flags);
  m_add_at<true, kD>(M, x, xM, r, -wi, -wo, sl[2], k[2], flags);
  m_add_at<true, kD>(M, y, yM, s, wi, wo, sl[3], k[3], flags);
}

// Node n's label and the degrees and sizes of r and s, by lanes 0..5 of one
// wavefront.
__device__ __forceinline__ void move_node(const ApplyArgs& a, int32_t n, int32_t r, int32_t s,
                                          int32_t wo, int32_t wi) {
  const int lane = lane_id();
  if (lane < 6) {
    int32_t* p = lane < 2 ? a.d_out : lane < 4 ? a.d_in : a.bsize;
    const int32_t w = lane < 2 ? wo : lane < 4 ? wi : 1;
    if (w) atomicAdd(&p[lane & 1 ? s : r], lane & 1 ? w : -w);
  }
  if (lane == 0) a.labels[n] = s;
}

// The block v's edges leave (x) and, if v moved in this batch, go to (y; else
// y = x).  Nodes of the batch are read from their proposals: their labels are
// being written.
__device__ __forceinline__ void ends_of(const ApplyArgs& a, int32_t v, int32_t& x, int32_t& y,
                                        bool& moved) {
  if (v >= a.beg && v < a.end) {
    const Prop p = a.prop[v - a.beg];
    x = p.r;
    moved = p.acc != 0;
    y = moved ? p.s : p.r;
  } else {
    x = y = a.labels[v];
    moved = false;
  }
}

constexpr int kMaxRec = kRegUnits * kWave;  // records of a node one wavefront handles
constexpr int kApplyLds = 6 * kMaxRec;      // LDS ints per wavefront

// The records of accepted node n (at most 64 U list entries), by one
// wavefront: its entries to neighbours that stay put, summed per block (so each
// changed pair of counts gets one atomic per node; in registers, an LDS hash
// deciding which entry owns a block), and one per out-edge to a neighbour that
// moves too (the edge's other end leaves it to this one).  They are left in
// the wavefront's LDS as x, y, wo, wi, kMaxRec each; returns their number.
template <bool kW, int U>
__device__ __forceinline__ int32_t apply_records(const ApplyArgs& a, int32_t n, int32_t r,
                                                 int32_t s, int64_t o0, int64_t i0, int32_t kco,
                                                 int32_t kc, int32_t* lds) {
  const int lane = lane_id();
  const GraphView& g = a.g;
  int32_t v[U], w[U];
#pragma unroll
  for (int q = 0; q < U; ++q) {
    const int32_t j = q * kWave + lane;
    v[q] = -1;
    w[q] = kW ? 0 : 1;
    if (j < kco) {
      v[q] = g.out_idx[o0 + j];
      if (kW) w[q] = g.out_w[o0 + j];
    } else if (j < kc) {
      v[q] = g.in_idx[i0 + (j - kco)];
      if (kW) w[q] = g.in_w[i0 + (j - kco)];
    }
  }
  constexpr int kCap = 128 * U;  // at least twice the blocks
  static_assert(3 * kCap <= kApplyLds && 4 * kMaxRec <= kApplyLds, "LDS per wavefront");
  int32_t *tk = lds, *two = lds + kCap, *twi = lds + 2 * kCap;
  for (int j = 4 * lane; j < 3 * kCap; j += 4 * kWave) {
    const int32_t z = j < kCap ? -1 : 0;
    *reinterpret_cast<int4*>(lds + j) = make_int4(z, z, z, z);
  }
  lds_order();
  int32_t wo_sum = kco, wi_sum = kc - kco;
  if (kW) {
    uint32_t so = 0, si = 0;
#pragma unroll
    for (int q = 0; q < U; ++q) (q * kWave + lane < kco ? so : si) += (uint32_t)w[q];
    wo_sum = (int32_t)wave_sum32(so);
    wi_sum = (int32_t)wave_sum32(si);
  }
  int32_t x[U], y[U];
  bool moved[U];
#pragma unroll
  for (int q = 0; q < U; ++q) {
    x[q] = y[q] = -1;
    moved[q] = false;
    if (v[q] >= 0) ends_of(a, v[q], x[q], y[q], moved[q]);
  }
  uint32_t hs[U];
  bool own[U];
#pragma unroll
  for (int q = 0; q < U; ++q) {
    const bool in = q * kWave + lane >= kco;
    own[q] = false;
    hs[q] = 0;
    if (v[q] >= 0 && !moved[q]) {
      uint32_t h = hash32(x[q]) & (kCap - 1);
      for (;;) {
        const int32_t old = atomicCAS(&tk[h], -1, x[q]);
        own[q] = old == -1;
        if (own[q] || old == x[q]) break;
        h = (h + 1) & (kCap - 1);
      }
      hs[q] = h;
      atomicAdd(in ? &twi[h] : &two[h], w[q]);
    }
  }
  lds_order();
  int32_t wo[U], wi[U];
#pragma unroll
  for (int q = 0; q < U; ++q) {
    wo[q] = own[q] ? two[hs[q]] : w[q];
    wi[q] = own[q] ? twi[hs[q]] : 0;
  }
  lds_order();  // the records take the table's place
  int32_t nrec = 0;
#pragma unroll
  for (int q = 0; q < U; ++q) {
    const bool emit = own[q] || (moved[q] && q * kWave + lane < kco);
    const unsigned long long m = __ballot(emit);
    if (emit) {
      const int32_t j = nrec + __popcll(m & ((1ull << lane) - 1ull));
      lds[j] = x[q];
      lds[kMaxRec + j] = y[q];
      lds[2 * kMaxRec + j] = wo[q];
      lds[3 * kMaxRec + j] = wi[q];
    }
    nrec += __popcll(m);
  }
  move_node(a, n, r, s, wo_sum, wi_sum);
  return nrec;
}

// An accepted node with more list entries than a wavefront's registers take, by
// the whole workgroup: edges to neighbours that stay put are summed per block
// in LDS where the blocks are few, else each list entry is a record.
constexpr int kHubBlocks = kNodalWaves * kApplyLds / 2;  // blocks whose two sums fit in LDS

template <bool kD, bool kW>
__device__ __forceinline__ void apply_hub(const ApplyArgs& a, int32_t n, int32_t r, int32_t s,
                                          int32_t* lds, int32_t* sums) {
  const GraphView& g = a.g;
  const int32_t B = a.M.B;
  const int64_t o0 = g.out_ptr[n], i0 = g.in_ptr[n];
  const int64_t kco = g.out_ptr[n + 1] - o0, kc = kco + (g.in_ptr[n + 1] - i0);
  const bool few = B <= kHubBlocks;
  if (few)
    for (int32_t b = threadIdx.x; b < 2 * B; b += blockDim.x) lds[b] = 0;
  if (threadIdx.x == 0) sums[0] = sums[1] = 0;
  __syncthreads();
  int32_t so = 0, si = 0;
  for (int64_t j = threadIdx.x; j < kc; j += blockDim.x) {
    int32_t v, w, x, y;
    bool moved;
    list_entry(g, o0, kco, i0, kc, j, v, w);
    const bool in = j >= kco;
    (in ? si : so) += w;
    ends_of(a, v, x, y, moved);
    if (moved) {
      if (!in) apply_record<kD>(a, r, s, x, y, w, 0);
    } else if (few) {
      atomicAdd(&lds[2 * x + in], w);
    } else {
      apply_record<kD>(a, r, s, x, x, in ? 0 : w, in ? w : 0);
    }
  }
  atomicAdd(&sums[0], so);
  atomicAdd(&sums[1], si);
  __syncthreads();
  if (few)
    for (int32_t b = threadIdx.x; b < B; b += blockDim.x) {
      const int32_t wo = lds[2 * b], wi = lds[2 * b + 1];
      if (wo != 0 || wi != 0) apply_record<kD>(a, r, s, b, b, wo, wi);
    }
  if (threadIdx.x < kWave) move_node(a, n, r, s, sums[0], sums[1]);
  __syncthreads();
}

// The batch's sums over all workgroups' shares (nparts of them), by one
// block, then the sweep step.
__device__ __forceinline__ void batch_tail(const BlockPart* part, uint32_t nparts, Sweep* sw) {
  __shared__ unsigned long s_lo[kNodalWaves];
  __shared__ long s_hi[kNodalWaves];
  __shared__ unsigned long long s_nb[kNodalWaves], s_ab[kNodalWaves];
  __shared__ long s_mv[kNodalWaves], s_ni[kNodalWaves];
  const int w = threadIdx.x / kWave;
  i128 sum = 0;
  long nb = 0, ab = 0, mv = 0, ni = 0;
  for (uint32_t i = threadIdx.x; i < nparts; i += blockDim.x) {
    const BlockPart P = part[i];
    sum += (i128)(((u128)(unsigned long)P.sum_hi << 64) | (u128)P.sum_lo);
    nb += (long)P.nodal_bytes;
    ab += (long)P.apply_bytes;
    mv += P.moves;
    ni += P.ninf;
  }
  sum = wave_sum128(sum);
  nb = wave_sum(nb);
  ab = wave_sum(ab);
  mv = wave_sum(mv);
  ni = wave_sum(ni);
  if (lane_id() == 0) {
    s_lo[w] = (unsigned long)(u128)sum;
    s_hi[w] = (long)(sum >> 64);
    s_nb[w] = (unsigned long long)nb;
    s_ab[w] = (unsigned long long)ab;
    s_mv[w] = mv;
    s_ni[w] = ni;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    u128 tot = 0;
    unsigned long long tnb = 0, tab = 0;
    long tmv = 0, tni = 0;
    for (int i = 0; i < (int)(blockDim.x / kWave); ++i) {
      tot += ((u128)(unsigned long)s_hi[i] << 64) | (u128)s_lo[i];
      tnb += s_nb[i];
      tab += s_ab[i];
      tmv += s_mv[i];
      tni += s_ni[i];
    }
    sweep_tail(sw, tot, (int32_t)tni, (int32_t)tmv, tnb, tab);
  }
  __syncthreads();
}

// Block 0 runs the batch's update step and, where it is the sweep's last and
// every row is direct, ends the sweep: on direct rows the applying blocks raise
// no flags, so there is nothing to wait for (k_finish is one launch more, 6 us
// of a sweep of 4 batches).  Every other block applies the moves
// of its four batch nodes: each moving node's wavefront writes its records,
// then all the block's records are spread over all its threads (a block holds
// 0-4 moving nodes, most often 0 or 1, so a node's records do not wait for its
// own 64 lanes only).  kHub: the graph has nodes larger than kMaxRec entries.
// Its time is one mover's chain of loads, and with 2000 movers of 45 edges a
// batch (B = 100000, after a merge) its atomics: four on counts per record,
// and a claim per new key (key counts and a bucket sum per update doubled
// them).  62.0 -> 42.6 us a launch there; N = 50000 dense 11.2 -> 7.4.
template <bool kD, bool kW, bool kHub>
__global__ __launch_bounds__(kWave* kNodalWaves, 4) void k_apply(ApplyArgs a) {
  __shared__ __align__(16) int32_t s_lds[kNodalWaves][kApplyLds];
  __shared__ int32_t s_n[kNodalWaves], s_r[kNodalWaves], s_s[kNodalWaves];
  if (blockIdx.x == 0) {
    if (a.tstamp && threadIdx.x == 0) a.tstamp[0] = wall_clock64();
    if (a.sweep->stop_n == 0) batch_tail(a.part, a.nparts, a.sweep);
    if (kD && a.host) finish_sweep(a.status, a.sweep, a.host, a.done);
    if (a.tstamp) {
      __syncthreads();
      if (threadIdx.x == 0) a.tstamp[a.tstride] = wall_clock64();
    }
    return;
  }
  const int w = threadIdx.x / kWave;
  const int64_t item0 = (int64_t)xcd_block(blockIdx.x - 1, gridDim.x - 1) * kNodalWaves;
  const int64_t n64 = (int64_t)a.beg + item0 + w;
  const bool in = n64 < a.end;
  const int32_t n = in ? (int32_t)n64 : a.beg;
  // whether the batch runs, the proposal and the node's list bounds in one
  // round of loads
  const int32_t stop = a.sweep->stop_n;  // the same for every block of this launch
  const Prop p = in ? a.prop[item0 + w] : Prop{0, 0, 0, 0};
  const int64_t o0 = a.g.out_ptr[n], i0 = a.g.in_ptr[n];
  const int64_t kco = a.g.out_ptr[n + 1] - o0, kc = kco + (a.g.in_ptr[n + 1] - i0);
  if (stop) return;
  if (a.tstamp && threadIdx.x == 0) a.tstamp[blockIdx.x] = wall_clock64();
  int32_t nrec = 0;
  if (in && p.acc) {
    const int32_t ko = (int32_t)kco, kk = (int32_t)kc;
    if (kHub && kc > kMaxRec)
      nrec = -1;
    else if (kk <= kWave)
      nrec = apply_records<kW, 1>(a, n, p.r, p.s, o0, i0, ko, kk, s_lds[w]);
    else if (kk <= 2 * kWave)
      nrec = apply_records<kW, 2>(a, n, p.r, p.s, o0, i0, ko, kk, s_lds[w]);
    else
      nrec = apply_records<kW, kRegUnits>(a, n, p.r, p.s, o0, i0, ko, kk, s_lds[w]);
  }
  if (lane_id() == 0) {
    s_n[w] = nrec;
    s_r[w] = p.r;
    s_s[w] = p.s;
  }
  __syncthreads();
  int32_t off[kNodalWaves + 1];
  off[0] = 0;
#pragma unroll
  for (int i = 0; i < kNodalWaves; ++i) off[i + 1] = off[i] + max(s_n[i], 0);
  for (int32_t e = threadIdx.x; e < off[kNodalWaves]; e += blockDim.x) {
    int wv = 0;
#pragma unroll
    for (int i = 1; i < kNodalWaves; ++i) wv += e >= off[i];
    const int32_t* rec = s_lds[wv] + (e - off[wv]);
    const int32_t wo = rec[2 * kMaxRec], wi = rec[3 * kMaxRec];
    if (wo != 0 || wi != 0)
      apply_record<kD>(a, s_r[wv], s_s[wv], rec[0], rec[kMaxRec], wo, wi);
  }
  if (kHub) {
    __shared__ int32_t s_sum[2];
    for (int i = 0; i < kNodalWaves; ++i) {
      if (s_n[i] >= 0) continue;
      __syncthreads();  // the records above are read
      apply_hub<kD, kW>(a, (int32_t)((int64_t)a.beg + item0 + i), s_r[i], s_s[i], &s_lds[0][0],
                        s_sum);
    }
  }
  if (a.tstamp) {
    __syncthreads();
    if (threadIdx.x == 0) a.tstamp[a.tstride + blockIdx.x] = wall_clock64();
  }
}

// k_grow: the rows marked by k_apply (a new key far from home, a large row past
// 1/slack load, parked increments), handled between two batches.  A row whose keys are not past
// 1/slack of its slab and that has nothing parked is only unmarked.  Else its
// dead keys (both counts 0) are dropped: a row whose live keys and parked
// increments fit 1/(2 slack) of its slab is rewritten in place, any other
// moves to a slab >= 2*slack*live+16 (direct once that reaches B/8) at the
// free tail of the pool, and its parked increments go in with the rest; the
// old slab's counts are left as zeros.  A slab that is the row's first to keep
// bucket sums gets them here.  Block 0 also acts on the batch's flags.
//
// Right after a merge phase a batch marks thousands of rows (2000 movers of 45
// edges at B = 100000), nearly all of them slabs of 128 to 512 slots: such a
// row is one wavefront's, read once into registers, laid out in LDS and
// written out whole.  The others are the workgroup's, one after another.
// 72.6 -> 20.0 us a launch there (every row by a workgroup, one counter for
// every slab, bucket sums and key counts kept for every row before).
constexpr int kWaveRow = 512;     // slots of a row one wavefront handles (8 per lane)
constexpr int kWaveSlab = 1024;   // and of its new slab
constexpr int kCompact = 4096;    // slots up to which the workgroup compacts in place
constexpr int kGrowLds = 2048;    // entries staged, and slots laid out, in LDS by the workgroup
constexpr int kGrowScan = 512;    // rows a k_grow workgroup checks per round (2 per thread)
constexpr int32_t kOvfCap = 1 << 22;  // parked increments
// Parked increments are handled after their batch.  A mark alone (the row is
// past 1/slack load) can wait: k_grow looks at marks after a call's first batch
// and every kGrowEvery-th from there, and else ends after its flags, 5.0 us
// instead of 9.6 (its launch and first loads), for chains no longer than the
// walk before parking (E = 11 M, N = 500000, 13600 such batches: 1010 -> 916 ms
// in all; every 4th batch 934).
constexpr int kGrowEvery = 8;
static_assert(kNodalWaves * 3 * kWaveSlab == 6 * kGrowLds, "one LDS pool for both paths");

struct GrowSide {
  int64_t* off;
  int32_t* cap;
  int32_t* gmark;
  int32_t* key;
  Cnt* cnt;
  int32_t* bs;
  int32_t* gpend;
  const int32_t* ovf;
  int32_t ovf_cap;
  GrowState* gst;
  int64_t P;
  int32_t slack;
  int32_t chunk;  // slots a workgroup takes from the free tail at a time (0: each row its own)
};

// Slots of the pool for grown rows.  One counter gives out the free tail, and
// an atomic on it costs ~30 ns, one after another: 1500 rows growing after one
// batch (B = 100000, right after a merge) waited 40 us on it.  So a workgroup
// takes `chunk` slots at a time and keeps what is left for later batches.
struct GrowAlloc {
  long long pos, end;    // the workgroup's chunk
  long long last;        // end of what was taken from it
  int32_t grows, compactions;
};

__device__ __forceinline__ long long grow_alloc(const GrowSide& g, GrowAlloc& al, int32_t n) {
  const long long p = (long long)atomicAdd(reinterpret_cast<unsigned long long*>(&al.pos),
                                           (unsigned long long)n);
  if (p + n <= al.end) {
    atomicMax(reinterpret_cast<unsigned long long*>(&al.last), (unsigned long long)(p + n));
    return p;
  }
  const long long q = (long long)atomicAdd(&g.gst->used, (unsigned long long)n);
  if (q + n <= g.P) return q;
  atomicAdd(&g.gst->used, (unsigned long long)(-(long long)n));  // give the slots back
  return -1;
}

struct GrowArgs {
  GrowSide side;
  MView M;
  int32_t B;
  Sweep* sweep;
  Status* status;
  unsigned long long* tstamp;  // as NodalArgs::tstamp, for this kernel
  int32_t tstride;
};

// Slots of the new slab of a row of c slots with `need` keys to hold.
__device__ __forceinline__ int64_t grown_cap(int64_t need, int32_t c, int32_t slack, int32_t B) {
  int64_t nc = 32;
  while (nc < 2 * slack * need + 16) nc <<= 1;
  if (nc < 2 * (int64_t)c) nc = 2 * (int64_t)c;
  return 8 * nc >= B ? B : nc;
}

// The pool ran out: the host rebuilds M from the labels (parked increments
// and all).
__device__ __forceinline__ void grow_nospace(const GrowSide& g, Sweep* sw) {
  g.gst->nospace = 1;
  atomicAdd(&g.gst->nospace_events, 1ull);
  atomicOr(&sw->flags, kFlagFull);
  atomicCAS(&sw->stop, 0, 2);
}

// (key, do, di) into an LDS slab, direct or hashed (never full: it is sized for
// the row's live keys and parked increments).
__device__ __forceinline__ void lds_slab_add(int32_t* tk, int32_t* to, int32_t* ti, uint32_t mask,
                                             bool direct, int32_t k, int32_t dout, int32_t din) {
  uint32_t h = (uint32_t)k;
  if (!direct) {
    h = hash32(k) & mask;
    for (;;) {
      const int32_t old = atomicCAS(&tk[h], -1, k);
      if (old == -1 || old == k) break;
      h = (h + 1) & mask;
    }
  }
  if (dout) atomicAdd(&to[h], dout);
  if (din) atomicAdd(&ti[h], din);
}

// Row a by one wavefront, with 3 * kWaveSlab ints of LDS; false: the row is
// the workgroup's.
__device__ __forceinline__ bool grow_wave(const GrowArgs& ga, int32_t a, int32_t* lds,
                                          GrowAlloc& al) {
  const GrowSide& g = ga.side;
  const int lane = lane_id();
  const int32_t B = ga.B;
  const int64_t o = g.off[a];
  const int32_t c = g.cap[a];
  const int32_t pend = g.gpend[a];  // parked increments (at most one new key each)
  if (c == B || c > kWaveRow) return false;
  constexpr int kQ = kWaveRow / kWave;
  int32_t k[kQ];
  Cnt x[kQ];
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    const int32_t j = q * kWave + lane;
    k[q] = -1;
    x[q] = Cnt{0, 0};
    if (j < c) {
      k[q] = g.key[o + j];
      x[q] = g.cnt[o + j];
    }
  }
  int32_t keys = 0, live = 0;
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    keys += __popcll(__ballot(k[q] >= 0));
    if (x[q].o == 0 && x[q].i == 0) k[q] = -1;
    live += __popcll(__ballot(k[q] >= 0));
  }
  if (pend == 0 && (int64_t)g.slack * keys <= c) {  // not past 1/slack load yet
    if (lane == 0) g.gmark[a] = 0;
    return true;
  }
  const bool inplace = 2 * (int64_t)g.slack * (live + pend) <= c;
  const int64_t nc64 = inplace ? c : grown_cap((int64_t)live + pend, c, g.slack, B);
  if (nc64 > kWaveSlab || nc64 == B) return false;
  const int32_t nc = (int32_t)nc64;
  long long base = 0;  // the slots are taken while the slab is laid out
  if (!inplace && lane == 0) base = grow_alloc(g, al, nc);
  int32_t *tk = lds, *to = lds + kWaveSlab, *ti = lds + 2 * kWaveSlab;
  for (int32_t j = lane; j < nc; j += kWave) {
    tk[j] = -1;
    to[j] = 0;
    ti[j] = 0;
  }
  lds_order();
  const uint32_t mask = (uint32_t)nc - 1;
#pragma unroll
  for (int q = 0; q < kQ; ++q)
    if (k[q] >= 0) lds_slab_add(tk, to, ti, mask, false, k[q], x[q].o, x[q].i);
  if (pend > 0) {
    const int32_t no = min(g.gst->ovf_n, g.ovf_cap);
    constexpr int kP = 8;  // entries in flight per lane: a batch may park thousands
    for (int32_t i0 = lane; i0 < no; i0 += kP * kWave) {
      int32_t row[kP];
#pragma unroll
      for (int q = 0; q < kP; ++q) row[q] = i0 + q * kWave < no ? g.ovf[i0 + q * kWave] : -1;
#pragma unroll
      for (int q = 0; q < kP; ++q) {
        if (row[q] != a) continue;
        const int32_t* e = g.ovf + i0 + q * kWave;
        lds_slab_add(tk, to, ti, mask, false, e[g.ovf_cap], e[2 * (int64_t)g.ovf_cap],
                     e[3 * (int64_t)g.ovf_cap]);
      }
    }
  }
  lds_order();
  int64_t nb = o;
  bool ok = true;
  if (!inplace) {
    nb = read_lane((long)base, 0);
    ok = nb >= 0;
    if (!ok && lane == 0) grow_nospace(g, ga.sweep);
  }
  if (ok) {
    for (int32_t j = lane; j < nc; j += kWave) {
      g.key[nb + j] = tk[j];
      g.cnt[nb + j] = Cnt{to[j], ti[j]};
    }
    if (!inplace)
      for (int32_t j = lane; j < c; j += kWave) g.cnt[o + j] = Cnt{0, 0};
    if (row_sums(ga.M, nc) && !row_sums(ga.M, c)) {  // the row's first bucket sums
      constexpr int kS = kWaveSlab / kWave;
      int32_t sk[kS], sv[kS];
#pragma unroll
      for (int q = 0; q < kS; ++q) {
        const int32_t j = q * kWave + lane;
        sk[q] = j < nc ? tk[j] : -1;
        sv[q] = j < nc ? to[j] + ti[j] : 0;
      }
      lds_order();
      for (int32_t j = lane; j < kNBK; j += kWave) tk[j] = 0;
      lds_order();
#pragma unroll
      for (int q = 0; q < kS; ++q)
        if (sk[q] >= 0 && sv[q] != 0) atomicAdd(&tk[sk[q] >> ga.M.bshift], sv[q]);
      lds_order();
      for (int32_t j = lane; j < kNBK; j += kWave) g.bs[(int64_t)a * kNBK + j] = tk[j];
    }
  }
  if (lane == 0) {
    if (ok) {
      if (!inplace) {
        g.off[a] = nb;
        g.cap[a] = nc;
      } else {
        atomicAdd(&al.compactions, 1);
      }
      atomicAdd(&al.grows, 1);
    }
    g.gpend[a] = 0;
    g.gmark[a] = ok ? room_mark(live + pend, nc, g.slack) : 0;
  }
  lds_order();  // the next row's slab takes this one's LDS
  return true;
}

// Parked increments of row a into its slab (o, c) in the pool (the only block
// touching row a in this launch); an increment that finds no slot asks the
// host for a rebuild.  sums: the row's bucket sums lack them too.
__device__ void replay_row(const GrowArgs& ga, int32_t a, int64_t o, int32_t c, bool sums) {
  const GrowSide& g = ga.side;
  const int32_t no = min(g.gst->ovf_n, g.ovf_cap);
  for (int32_t i = threadIdx.x; i < no; i += blockDim.x) {
    if (g.ovf[i] != a) continue;
    const int32_t b = g.ovf[g.ovf_cap + i];
    const int32_t dout = g.ovf[2 * g.ovf_cap + i], din = g.ovf[3 * g.ovf_cap + i];
    if (sums) atomicAdd(&g.bs[(int64_t)a * kNBK + (b >> ga.M.bshift)], dout + din);
    if (c == ga.B) {
      cnt_add(&g.cnt[o + b], dout, din);
      continue;
    }
    const uint32_t mask = (uint32_t)c - 1;
    uint32_t h = hash32(b) & mask;
    bool done = false;
    for (int32_t probe = 0; probe < c && !done; ++probe) {
      int32_t k = ld_relaxed(&g.key[o + h]);
      if (k < 0) {
        k = atomicCAS(&g.key[o + h], -1, b);
        if (k == -1) k = b;
      }
      if (k == b) {
        cnt_add(&g.cnt[o + h], dout, din);
        done = true;
      }
      h = (h + 1) & mask;
    }
    if (!done) {  // no room (the pool ran out): rebuild M
      atomicOr(&ga.sweep->flags, kFlagFull);
      atomicCAS(&ga.sweep->stop, 0, 2);
    }
  }
}

// The live entries s_k/s_o/s_i[0, live) laid out as a slab of nc slots in
// LDS t_k/t_o/t_i (hashed, or by key when direct), for one coalesced
// write-out: no per-entry CAS round trip to the new slab.
__device__ void lds_slab(const int32_t* s_k, const int32_t* s_o, const int32_t* s_i,
                         int32_t live, int32_t* t_k, int32_t* t_o, int32_t* t_i, int32_t nc,
                         bool direct) {
  for (int32_t j = threadIdx.x; j < nc; j += blockDim.x) {
    t_k[j] = -1;
    t_o[j] = 0;
    t_i[j] = 0;
  }
  __syncthreads();
  for (int32_t i = threadIdx.x; i < live; i += blockDim.x)
    lds_slab_add(t_k, t_o, t_i, (uint32_t)nc - 1, direct, s_k[i], s_o[i], s_i[i]);
  __syncthreads();
}

// Row a by the whole workgroup.
__device__ void grow_block(const GrowArgs& ga, int32_t a, int32_t* pool, GrowAlloc& al) {
  __shared__ long long s_base;
  __shared__ int32_t s_cap, s_live, s_keys;
  int32_t *s_k = pool, *s_o = pool + kGrowLds, *s_i = pool + 2 * kGrowLds;  // live entries
  int32_t *t_k = pool + 3 * kGrowLds, *t_o = t_k + kGrowLds, *t_i = t_o + kGrowLds;  // new slab
  const GrowSide& g = ga.side;
  const int32_t B = ga.B;
  const int64_t o = g.off[a];
  const int32_t c = g.cap[a];
  const int32_t pend = g.gpend[a];
  const bool dold = c == B;  // a direct row never moves
  if (threadIdx.x == 0) s_live = s_keys = 0;
  __syncthreads();
  constexpr int kQ = 4;
  int32_t keys = 0;
  for (int32_t j0 = threadIdx.x; j0 < c && !dold; j0 += kQ * blockDim.x) {
    int32_t k[kQ];
    Cnt x[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const int32_t j = j0 + q * (int32_t)blockDim.x;
      k[q] = j < c ? g.key[o + j] : -1;
      x[q] = j < c ? g.cnt[o + j] : Cnt{0, 0};
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      keys += k[q] >= 0;
      if (k[q] >= 0 && (x[q].o != 0 || x[q].i != 0)) {
        const int32_t i = atomicAdd(&s_live, 1);
        if (i < kGrowLds) {
          s_k[i] = k[q];
          s_o[i] = x[q].o;
          s_i[i] = x[q].i;
        }
      }
    }
  }
  if (keys) atomicAdd(&s_keys, keys);
  __syncthreads();
  const int32_t live = s_live;
  const bool staged = live <= kGrowLds;
  bool fresh = false;  // bucket sums just computed, without the parked increments
  bool moved = false;  // dead keys dropped
  int64_t o2 = o;      // the row's slab after this step
  int32_t c2 = c;
  if (dold || (pend == 0 && (int64_t)g.slack * s_keys <= c)) {
    // nothing to move
  } else if (staged && c <= kCompact && 2 * (int64_t)g.slack * (live + pend) <= c) {
    // in place: the slab rewritten with the live entries only
    moved = true;
    if (c <= kGrowLds) {
      lds_slab(s_k, s_o, s_i, live, t_k, t_o, t_i, c, false);
      for (int32_t j = threadIdx.x; j < c; j += blockDim.x) {
        g.key[o + j] = t_k[j];
        g.cnt[o + j] = Cnt{t_o[j], t_i[j]};
      }
    } else {
      for (int32_t j = threadIdx.x; j < c; j += blockDim.x) {
        g.key[o + j] = -1;
        g.cnt[o + j] = Cnt{0, 0};
      }
      __threadfence_block();
      __syncthreads();
      const uint32_t mask = (uint32_t)c - 1;
      for (int32_t i = threadIdx.x; i < live; i += blockDim.x) {
        uint32_t h = hash32(s_k[i]) & mask;
        while (atomicCAS(&g.key[o + h], -1, s_k[i]) != -1) h = (h + 1) & mask;
        g.cnt[o + h] = Cnt{s_o[i], s_i[i]};
      }
    }
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x == 0) {
      atomicAdd(&al.grows, 1);
      atomicAdd(&al.compactions, 1);
    }
  } else {
    const int64_t nc = grown_cap((int64_t)live + pend, c, g.slack, B);
    // the slots are taken while the new slab is laid out in LDS
    long long base = 0;
    if (threadIdx.x == 0) base = grow_alloc(g, al, (int32_t)nc);
    const bool inlds = staged && nc <= kGrowLds;
    if (inlds) lds_slab(s_k, s_o, s_i, live, t_k, t_o, t_i, (int32_t)nc, nc == B);
    if (threadIdx.x == 0) {
      s_cap = 0;
      if (base < 0) {
        grow_nospace(g, ga.sweep);
      } else {
        s_cap = (int32_t)nc;
        s_base = base;
      }
    }
    __syncthreads();
    const int32_t ncap = s_cap;
    if (ncap > 0) {
      const int64_t nb = s_base;
      if (inlds) {
        for (int32_t j = threadIdx.x; j < ncap; j += blockDim.x) {
          g.key[nb + j] = t_k[j];
          g.cnt[nb + j] = Cnt{t_o[j], t_i[j]};
        }
        // the old slab's counts stay in the pool as zeros until a rebuild
        for (int32_t j = threadIdx.x; j < c; j += blockDim.x) g.cnt[o + j] = Cnt{0, 0};
      } else {
        for (int32_t i = threadIdx.x; i < ncap; i += blockDim.x) {
          g.key[nb + i] = -1;
          g.cnt[nb + i] = Cnt{0, 0};
        }
        __threadfence_block();
        __syncthreads();
        const bool dnew = ncap == B;
        const uint32_t mask = (uint32_t)ncap - 1;
        for (int32_t j0 = threadIdx.x; j0 < c; j0 += kQ * blockDim.x) {
          int32_t k[kQ];
          Cnt x[kQ];
#pragma unroll
          for (int q = 0; q < kQ; ++q) {
            const int32_t j = j0 + q * (int32_t)blockDim.x;
            k[q] = j < c ? g.key[o + j] : -1;
            x[q] = j < c ? g.cnt[o + j] : Cnt{0, 0};
          }
#pragma unroll
          for (int q = 0; q < kQ; ++q) {
            if (k[q] < 0 || (x[q].o == 0 && x[q].i == 0)) continue;
            g.cnt[o + j0 + q * (int32_t)blockDim.x] = Cnt{0, 0};
            if (dnew) {
              g.cnt[nb + k[q]] = x[q];
              continue;
            }
            uint32_t h = hash32(k[q]) & mask;
            while (atomicCAS(&g.key[nb + h], -1, k[q]) != -1) h = (h + 1) & mask;
            g.cnt[nb + h] = x[q];
          }
        }
      }
      __threadfence_block();
      __syncthreads();
      // the new slab's bucket sums, if it is the first to keep them (parked
      // increments added theirs only to a slab that kept them)
      if (row_sums(ga.M, ncap) && !row_sums(ga.M, c)) {
        for (int32_t j = threadIdx.x; j < kNBK; j += blockDim.x) s_k[j] = 0;
        __syncthreads();
        for (int32_t j = threadIdx.x; j < ncap; j += blockDim.x) {
          const int32_t k = ncap == B ? j : ld_relaxed(&g.key[nb + j]);
          const Cnt x = g.cnt[nb + j];
          if (k >= 0 && (x.o != 0 || x.i != 0)) atomicAdd(&s_k[k >> ga.M.bshift], x.o + x.i);
        }
        __syncthreads();
        for (int32_t j = threadIdx.x; j < kNBK; j += blockDim.x)
          g.bs[(int64_t)a * kNBK + j] = s_k[j];
        __threadfence_block();
        __syncthreads();
        fresh = true;
      }
      if (threadIdx.x == 0) {
        g.off[a] = nb;
        g.cap[a] = ncap;
        atomicAdd(&al.grows, 1);
      }
      moved = true;
      o2 = nb;
      c2 = ncap;
    }
  }
  if (pend > 0) replay_row(ga, a, o2, c2, fresh);
  __syncthreads();
  if (threadIdx.x == 0) {
    g.gpend[a] = 0;
    g.gmark[a] = dold ? 0 : room_mark(moved ? live + pend : s_keys, c2, g.slack);
  }
  __syncthreads();
}

__global__ __launch_bounds__(256) void k_grow(GrowArgs ga) {
  __shared__ __align__(16) int32_t s_pool[6 * kGrowLds];
  __shared__ int32_t s_q[kGrowScan];    // marked rows of the scanned chunk
  __shared__ int32_t s_big[kGrowScan];  // those left to the workgroup
  __shared__ int32_t s_nq, s_nbig;
  __shared__ GrowAlloc s_al;
  __shared__ bool s_taken;  // a chunk was taken in this round
  const int32_t B = ga.B;
  const GrowSide& g = ga.side;
  const int w = threadIdx.x / kWave;
  bool any = false;  // thread 0: s_al is loaded
  if (ga.tstamp && threadIdx.x == 0) ga.tstamp[blockIdx.x] = wall_clock64();
  // the batch's flags (raised by its k_nodal and k_apply, both complete)
  const int32_t flags = ga.status->flags, parked = g.gst->ovf_n, done = ga.sweep->done;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    fold_flags(ga.status, ga.sweep, flags);
    if (parked) g.gst->full += (unsigned long long)parked;
  }
  const bool look = parked != 0 || done % kGrowEvery == 1;
  const int32_t per = (B + (int32_t)gridDim.x - 1) / (int32_t)gridDim.x;
  const int32_t lo = (int32_t)blockIdx.x * per, hi = look ? min(B, lo + per) : lo;
  for (int32_t base = lo; base < hi; base += kGrowScan) {
    if (threadIdx.x == 0) s_nq = s_nbig = 0;
    __syncthreads();
    int32_t mq[kGrowScan / 256];
#pragma unroll
    for (int q = 0; q < kGrowScan / 256; ++q) {
      const int32_t r = base + q * 256 + (int32_t)threadIdx.x;
      mq[q] = r < hi ? g.gmark[r] : 0;
    }
#pragma unroll
    for (int q = 0; q < kGrowScan / 256; ++q)
      if (mq[q] > 0) s_q[atomicAdd(&s_nq, 1)] = base + q * 256 + (int32_t)threadIdx.x;
    __syncthreads();
    const int32_t nq = s_nq;
    if (nq == 0) continue;  // the same for every thread; s_nq is next written by thread 0
    if (threadIdx.x == 0) {
      s_taken = false;
      if (!any) {
        const GrowChunk c = g.gst->chunk[blockIdx.x];
        s_al = GrowAlloc{c.pos, c.end, c.pos, 0, 0};
        any = true;
      }
      if (g.chunk > 0 && s_al.end - s_al.last < kWaveSlab) {
        const long long p = (long long)atomicAdd(&g.gst->used, (unsigned long long)g.chunk);
        if (p + g.chunk <= g.P) {
          s_al.pos = s_al.last = p;
          s_al.end = p + g.chunk;
          s_taken = true;
        } else {
          atomicAdd(&g.gst->used, (unsigned long long)(-(long long)g.chunk));
        }
      }
    }
    __syncthreads();
    for (int32_t i = w; i < nq; i += kNodalWaves) {
      const int32_t a = s_q[i];
      if (!grow_wave(ga, a, s_pool + w * 3 * kWaveSlab, s_al) && lane_id() == 0)
        s_big[atomicAdd(&s_nbig, 1)] = a;
    }
    __syncthreads();
    for (int32_t i = 0; i < s_nbig; ++i) grow_block(ga, s_big[i], s_pool, s_al);
    __syncthreads();
    if (s_taken)  // the MDL scan reads the whole used pool
      for (long long j = s_al.last + threadIdx.x; j < s_al.end; j += blockDim.x)
        g.cnt[j] = Cnt{0, 0};
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x == 0) s_al.pos = s_al.last;  // a request that did not fit took nothing
  }
  if (threadIdx.x == 0 && any) {
    GrowChunk& c = g.gst->chunk[blockIdx.x];
    c.pos = s_al.last;
    c.end = s_al.end;
    c.grows += (unsigned long long)s_al.grows;
    c.compactions += (unsigned long long)s_al.compactions;
  }
  if (ga.tstamp) {
    __syncthreads();
    if (threadIdx.x == 0) ga.tstamp[ga.tstride + blockIdx.x] = wall_clock64();
  }
}

}  // namespace

// ===========================================================================
// Host side
// ===========================================================================

struct DevSpM {
  int64_t* off = nullptr;
  int32_t* cap = nullptr;
  int32_t* gmark = nullptr;  // [N]
  int32_t* key = nullptr;  // row slabs [P]: keys
  Cnt* cnt = nullptr;      // and counts
  int32_t* bs = nullptr;  // [bs_rows][kNBK]
  int32_t bs_rows = 0;
  int32_t* gpend = nullptr;  // [N]
  int32_t* ovf = nullptr;    // [4][ovf_cap]
  int32_t ovf_cap = 0;       // parked increments that fit
  GrowState* gst = nullptr;
  int64_t P = 0;      // allocated slots
  int64_t total = 0;  // slots in use after the last rebuild
  int32_t stride = 0;  // MView::stride
  int32_t slack = 2;  // usap_params.slab_slack
};

struct usap_engine {
  usap_params p{};
  hipStream_t stream = nullptr;
  bool own_stream = true;      // false: a worker context's stream, kept at destroy
  hipMemPool_t pool = nullptr;  // a worker context's pool, else the device's default pool
  std::string err;
  // host copy of the graph
  int32_t N = 0;
  int64_t E = 0;
  bool weighted = false;
  std::vector<int64_t> h_out_ptr, h_in_ptr;
  std::vector<int32_t> h_out_idx, h_in_idx, h_out_w, h_in_w;
  usap_graph hg{};
  bool host_stale = false;  // lists appended on the device since the host copy was made
  int64_t Wtot = 0;
  int64_t lam_cap = 0;  // entries of the device lambda table
  // device graph
  int64_t *out_ptr = nullptr, *in_ptr = nullptr;
  int32_t *out_idx = nullptr, *in_idx = nullptr, *out_w = nullptr, *in_w = nullptr;
  int32_t* out_src = nullptr;
  int64_t* lam = nullptr;
  // partition state
  int32_t B = 0;
  bool has_labels = false;
  int32_t* labels = nullptr;
  int32_t *d_out = nullptr, *d_in = nullptr, *ecnt_out = nullptr, *ecnt_in = nullptr,
          *bsize = nullptr;
  // nodes grouped by block for the per-row build: offsets, arrival cursors, nodes
  int32_t *bl_off = nullptr, *bl_cur = nullptr, *bl_nodes = nullptr;
  int2* big_items = nullptr;
  DevSpM M;  // block rows (both orientations of M)
  int64_t* tmpM = nullptr;
  void* scan_tmp = nullptr;
  size_t scan_tmp_bytes = 0;
  // merge
  int32_t* best_s = nullptr;
  long* best_hi = nullptr;
  unsigned long* best_lo = nullptr;
  int32_t merge_B = -1;  // B of the last merge_propose (-1: none)
  int32_t* map = nullptr;
  unsigned long long *sort_key[2] = {nullptr, nullptr};  // carry-out sort buffers [N]
  int32_t* sort_idx[2] = {nullptr, nullptr};
  void* sort_tmp = nullptr;
  size_t sort_tmp_bytes = 0;
  // nodal
  Prop* prop = nullptr;
  PropDs* prop_ds = nullptr;
  uint64_t* draws = nullptr;  // the sweep's (or batch's) Philox words, 4 per node
  int32_t last_beg = 0, last_end = 0;
  // pre-drawn uniform stream (usap_set_uniforms): 4 words per draw, or null
  uint64_t* uni = nullptr;
  int64_t uni_n = 0;    // draws held
  int64_t uni_pos = 0;  // draws consumed
  Status* status = nullptr;   // the running batch
  BlockPart* part = nullptr;  // per-workgroup shares of the running batch
  Sweep* sweep = nullptr;     // device sweep state
  Sweep* h_sweep = nullptr;   // pinned host copy
  Sweep* h_chunk[2] = {nullptr, nullptr};  // sweep state after alternate launch chunks
  Sweep* d_hsweep = nullptr;               // device addresses of the two
  Sweep* d_hchunk[2] = {nullptr, nullptr};
  hipEvent_t chunk_ev[2] = {nullptr, nullptr};
  // reference-algorithm byte counts (profiling): drawn neighbour's block per
  // batch node, per-block batch stamps, device totals [nodal per-node,
  // nodal per-block, merge non-zeros]
  int32_t* prop_u = nullptr;
  int32_t* aq_mark = nullptr;
  unsigned long long* aq_acc = nullptr;
  int32_t aq_stamp = 0;
  unsigned long long* tstamp = nullptr;  // profiled batch launches: workgroup stamps
  size_t tstamp_n = 0;                   // its length
  int32_t tstamp_G = 0;                  // k_nodal / k_apply workgroups per slot this round
  // captured sweep (usap_params.graphs): replayed while its key matches
  hipGraphExec_t gexec = nullptr;
  int32_t g_B = -1, g_batch = -1, g_nb = -1;
  bool g_direct = false;  // all_direct at its capture
  uint64_t g_epoch = 0;
  uint64_t epoch = 0;  // bumped by every device allocation (pointers may change)
  int64_t graph_captures = 0;
  int32_t* build_flags = nullptr;  // [0] build overflow flags; [1] pieces of large rows (a build's),
                                   // [2] distinct block pairs (a build's); both: rows left to
                                   // k_merge (MergeList::n); [3] carry-out out of candidates
  int32_t* h_short = nullptr;      // the last in pinned host memory, and its device address
  int32_t* d_short = nullptr;
  int32_t word_want[3] = {0, 0, 0};
  int32_t word_seq = 0;  // the last value given to a host word (h_short[4 + slot])
  int32_t* hist = nullptr;  // counts of the build by histograms
  int64_t hist_cap = 0;
  uint32_t* pair_key[2] = {nullptr, nullptr};  // block-pair builds [E]
  int32_t* pair_val[2] = {nullptr, nullptr};
  int64_t pair_cap = 0;  // edges the pair buffers hold
  void* pair_tmp = nullptr;
  size_t pair_tmp_bytes = 0;
  int64_t* big_off = nullptr;
  int32_t* big_tab = nullptr;
  int2* huge_parts = nullptr;  // (node, part of kHugePart list entries) of nodes of more than kBigPart
  int32_t n_huge = 0;
  int64_t max_list = 0;  // list entries of the largest node
  // entropy
  long* ent_part = nullptr;
  int64_t* h_fx = nullptr;  // usap_entropy's result in pinned host memory, and its device address
  int64_t* d_fx = nullptr;
  // snapshots
  int32_t* snap_labels[kNumSnap] = {};
  int32_t snap_B[kNumSnap] = {};
  double snap_S[kNumSnap] = {};
  int32_t rebuilds = 0;
  // profiling (HIP events on the engine's stream)
  bool prof = false;
  hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
  bool all_direct = false;  // every row of M direct-mapped (set by each rebuild)
  usap_kernel_prof kp[USAP_NKERNELS] = {};
  std::vector<usap_phase> phase_log;
};

namespace {

int set_err(usap_engine* e, int code, const std::string& msg) {
  if (e) e->err = msg;
  return code;
}

#define HIPCHK(expr)                                                                    \
  do {                                                                                  \
    hipError_t _st = (expr);                                                            \
    if (_st != hipSuccess)                                                              \
      return set_err(e, USAP_EHIP, std::string(#expr) + ": " + hipGetErrorString(_st)); \
  } while (0)

// The runtime's resource calls (stream-ordered allocations and frees, pools,
// streams, events, pinned host buffers, graph instantiation) are made under
// one process-wide lock.  Engines on several host threads (batched and served
// graphs) make these calls concurrently; test processes running several
// engines on host threads have ended in crashes inside native threads with
// no GPU fault and no cause found in this library, so the calls that create,
// grow or release runtime state are kept from overlapping.  They are short
// and few per graph; kernel launches and copies are not locked.
std::mutex g_hip_mu;

// Device memory is stream-ordered (hipMallocAsync / hipFreeAsync on the
// engine's stream): creating and destroying engines never synchronises the
// device, so many engines can come and go while others run (batched and
// served graphs).  The default pool keeps freed memory for reuse.
void prepare_pool(int device) {
  static std::once_flag once;
  std::call_once(once, [device]() {
    hipMemPool_t pool;
    if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess) {
      uint64_t keep = UINT64_MAX;
      (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
    }
  });
}

template <typename T>
int dalloc(usap_engine* e, T** p, size_t n) {
  *p = nullptr;
  if (n == 0) n = 1;
  e->epoch++;
  std::unique_lock<std::mutex> lk(g_hip_mu);
  hipError_t st = e->pool ? hipMallocFromPoolAsync((void**)p, n * sizeof(T), e->pool, e->stream)
                          : hipMallocAsync((void**)p, n * sizeof(T), e->stream);
  lk.unlock();
  if (st != hipSuccess) {
    *p = nullptr;
    return set_err(e, USAP_ENOMEM, std::string("hipMallocAsync: ") + hipGetErrorString(st));
  }
  return USAP_OK;
}

// dalloc for untyped scratch (rocPRIM temporary storage).
int dalloc_raw(usap_engine* e, void** p, size_t bytes) {
  *p = nullptr;
  e->epoch++;
  std::unique_lock<std::mutex> lk(g_hip_mu);
  hipError_t st = e->pool ? hipMallocFromPoolAsync(p, bytes ? bytes : 1, e->pool, e->stream)
                          : hipMallocAsync(p, bytes ? bytes : 1, e->stream);
  lk.unlock();
  if (st != hipSuccess) {
    *p = nullptr;
    return set_err(e, USAP_ENOMEM, std::string("hipMallocAsync: ") + hipGetErrorString(st));
  }
  return USAP_OK;
}

template <typename T>
void dfree(usap_engine* e, T*& p) {
  if (p) {
    std::lock_guard<std::mutex> lk(g_hip_mu);
    (void)hipFreeAsync((void*)p, e->stream);
  }
  p = nullptr;
}

// Pinned host buffers are recycled through a process-wide free list instead
// of being freed (hipHostFree may wait for the device).
std::mutex g_pin_mu;
std::vector<std::pair<size_t, void*>> g_pin_free;

void* pin_get(size_t bytes) {
  {
    std::lock_guard<std::mutex> lk(g_pin_mu);
    for (size_t i = 0; i < g_pin_free.size(); ++i)
      if (g_pin_free[i].first == bytes) {
        void* q = g_pin_free[i].second;
        g_pin_free.erase(g_pin_free.begin() + (long)i);
        return q;
      }
  }
  void* q = nullptr;
  std::lock_guard<std::mutex> lk(g_hip_mu);
  if (hipHostMalloc(&q, bytes) != hipSuccess) return nullptr;
  return q;
}

void pin_put(void* q, size_t bytes) {
  if (!q) return;
  std::lock_guard<std::mutex> lk(g_pin_mu);
  g_pin_free.emplace_back(bytes, q);
}

inline unsigned blocks_for(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

int32_t bucket_shift(int32_t B) {
  int32_t sh = 0;
  while (((B - 1) >> sh) >= kNBK) ++sh;
  return sh;
}

// Slots from a row to the next after a histogram build: for few blocks each row
// begins a 256-byte piece of its own, as k_apply's atomics from all XCDs on a few
// neighbouring lines hold each other up.  N = 100000, 25000-node batches from random
// labels (10000 moves), k_apply packed and so: B = 4 603 and 383 us, 7 696 and 324, 10
// 468 and 270, 20 268 and 200, 30 192 and 185, 50 142 and 140.
int32_t direct_stride(int32_t B) { return B <= 64 ? (B + 31) / 32 * 32 : B; }

MView view(const DevSpM& m, int32_t B) {
  MView v;
  v.off = m.off;
  v.cap = m.cap;
  v.gmark = m.gmark;
  v.key = m.key;
  v.cnt = m.cnt;
  v.bs = m.bs;
  v.gpend = m.gpend;
  v.ovf = m.ovf;
  v.ovf_cap = m.ovf_cap;
  v.gst = m.gst;
  v.B = B;
  v.bshift = bucket_shift(B);
  v.stride = m.stride;
  v.slack = m.slack;
  return v;
}

GraphView gview(const usap_engine* e) {
  GraphView g;
  g.N = e->N;
  g.out_ptr = e->out_ptr;
  g.out_idx = e->out_idx;
  g.out_w = e->out_w;
  g.in_ptr = e->in_ptr;
  g.in_idx = e->in_idx;
  g.in_w = e->in_w;
  return g;
}

double fx_to_double(i128 v) {
  const bool neg = v < 0;
  const u128 m = neg ? (u128)0 - (u128)v : (u128)v;
  const uint64_t hi = (uint64_t)(m >> 64), lo = (uint64_t)m;
  const double d = std::ldexp((double)hi, 64 - usap::kLambdaFrac) +
                   std::ldexp((double)lo, -usap::kLambdaFrac);
  return neg ? -d : d;
}

i128 mk128(long hi, unsigned long lo) { return (i128)(((u128)(unsigned long)hi << 64) | (u128)lo); }

// elapsed ms between two recorded events (0 when profiling is off)
float ev_ms(usap_engine* e, int a, int b) {
  float ms = 0.f;
  if (e->prof && hipEventElapsedTime(&ms, e->ev[a], e->ev[b]) != hipSuccess) ms = 0.f;
  return ms;
}

void ev_rec(usap_engine* e, int i) {
  if (e->prof) (void)hipEventRecord(e->ev[i], e->stream);
}

void prof_add(usap_engine* e, int k, double ms, int64_t launches, double bytes) {
  if (!e->prof) return;
  e->kp[k].ms += ms;
  e->kp[k].launches += launches;
  e->kp[k].bytes += bytes;
}

// The block-pair build (k_pair_keys, sort, sum per pair, k_insert_pairs).
int build_by_pairs(usap_engine* e) {
  const int32_t B = e->B;
  const int64_t E = e->E;
  hipStream_t st = e->stream;
  if (e->pair_cap < E) {  // first use, or the graph grew (usap_set_graph)
    for (int i = 0; i < 2; ++i) {
      dfree(e, e->pair_key[i]);
      dfree(e, e->pair_val[i]);
      if (int rc = dalloc(e, &e->pair_key[i], (size_t)E)) return rc;
      if (int rc = dalloc(e, &e->pair_val[i], (size_t)E)) return rc;
    }
    e->pair_cap = E;
  }
  int bits = 1;
  while (((uint64_t)1 << bits) < (uint64_t)B * (uint64_t)B) ++bits;
  size_t b1 = 0, b2 = 0;
  HIPCHK(rocprim::radix_sort_pairs(nullptr, b1, e->pair_key[0], e->pair_key[1], e->pair_val[0],
                                   e->pair_val[1], (size_t)E, 0, bits, st));
  HIPCHK(rocprim::reduce_by_key(nullptr, b2, e->pair_key[1], e->pair_val[1], (size_t)E,
                                e->pair_key[0], e->pair_val[0], e->build_flags + 2,
                                rocprim::plus<int32_t>(), rocprim::equal_to<uint32_t>(), st));
  const size_t need = std::max(b1, b2);
  if (need > e->pair_tmp_bytes) {
    dfree(e, e->pair_tmp);
    if (int rc = dalloc_raw(e, &e->pair_tmp, need)) return rc;
    e->pair_tmp_bytes = need;
  }
  const unsigned g = std::min<int64_t>(blocks_for(E, 256), 16384);
  k_pair_keys<<<g, 256, 0, st>>>(E, e->out_src, e->out_idx, e->out_w, e->labels, B, e->pair_key[0],
                                 e->pair_val[0]);
  HIPCHK(hipGetLastError());
  size_t bytes = e->pair_tmp_bytes;
  HIPCHK(rocprim::radix_sort_pairs(e->pair_tmp, bytes, e->pair_key[0], e->pair_key[1], e->pair_val[0],
                                   e->pair_val[1], (size_t)E, 0, bits, st));
  bytes = e->pair_tmp_bytes;
  HIPCHK(rocprim::reduce_by_key(e->pair_tmp, bytes, e->pair_key[1], e->pair_val[1], (size_t)E,
                                e->pair_key[0], e->pair_val[0], e->build_flags + 2,
                                rocprim::plus<int32_t>(), rocprim::equal_to<uint32_t>(), st));
  k_insert_pairs<<<g, 256, 0, st>>>(E, e->pair_key[0], e->pair_val[0], e->build_flags + 2,
                                    view(e->M, B), e->build_flags);
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

// The M build by rows: nodes grouped by block (offsets by an exclusive scan of
// the block sizes, then a scatter), k_build_rows for the rows it lays out in LDS,
// k_fill_big and k_build_big for the others.
int build_rows(usap_engine* e) {
  const int32_t B = e->B;
  hipStream_t st = e->stream;
  size_t bytes = 0;
  HIPCHK(rocprim::exclusive_scan(nullptr, bytes, e->bsize, e->bl_off, (int32_t)0, (size_t)B,
                                 rocprim::plus<int32_t>(), st));
  if (bytes > e->scan_tmp_bytes) {
    dfree(e, e->scan_tmp);
    if (int rc = dalloc_raw(e, &e->scan_tmp, bytes)) return rc;
    e->scan_tmp_bytes = bytes;
  }
  bytes = e->scan_tmp_bytes;
  HIPCHK(rocprim::exclusive_scan(e->scan_tmp, bytes, e->bsize, e->bl_off, (int32_t)0, (size_t)B,
                                 rocprim::plus<int32_t>(), st));
  k_node_lists<<<blocks_for(e->N, kNodesWg), 256, 0, st>>>(e->N, e->labels, e->bl_off, e->bl_cur,
                                                           e->bl_nodes);
  const MView M = view(e->M, B);
  const int32_t* n_items = e->build_flags + 1;
  k_fill_big<<<dim3(kBigGrid, kBigParts), 256, 0, st>>>(M, e->all_direct ? nullptr : e->M.key,
                                                        e->bsize, e->big_items, n_items);
  k_build_rows<256, 0><<<blocks_for(B, kNodalWaves), kWave * kNodalWaves, 0, st>>>(
      gview(e), e->labels, e->bl_off, e->bl_nodes, M, e->build_flags);
  k_build_rows<kRowTab, 256><<<blocks_for(B, kNodalWaves), kWave * kNodalWaves, 0, st>>>(
      gview(e), e->labels, e->bl_off, e->bl_nodes, M, e->build_flags);
  k_build_big<false><<<dim3(kBigGrid, kBigParts), 256, 0, st>>>(
      gview(e), e->labels, e->bl_off, e->bl_nodes, M, e->big_items, n_items, 0, e->build_flags);
  if (e->n_huge > 0)
    k_build_big<true><<<std::min<unsigned>((unsigned)e->n_huge, kBigGrid * kBigParts), 256, 0, st>>>(
        gview(e), e->labels, e->bl_off, e->bl_nodes, M, e->huge_parts, nullptr, e->n_huge,
        e->build_flags);
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

// Slots for a rebuild that needs `total`: two thirds of the pool is headroom for
// rows that grow.
int reserve_pool(usap_engine* e, int64_t total) {
  DevSpM& m = e->M;
  m.total = total;
  m.slack = e->p.slab_slack;
  if (3 * total <= m.P) return USAP_OK;
  dfree(e, m.key);
  dfree(e, m.cnt);
  const int64_t P = 3 * total + (int64_t)4 * e->B + 4096;
  m.P = 0;
  if (int rc = dalloc(e, &m.key, (size_t)P)) return rc;
  if (int rc = dalloc(e, &m.cnt, (size_t)P)) return rc;
  m.P = P;
  return USAP_OK;
}

// The build for B <= kHistB.  About 4096 edges a workgroup at least: fewer make
// the counts' way through memory longer than the edges'.
int build_hist(usap_engine* e) {
  const int32_t B = e->B;
  hipStream_t st = e->stream;
  const bool one = B <= kHistOne;
  const int32_t halves = one ? 1 : 2;
  const int32_t G = (int32_t)std::max<int64_t>(1, std::min<int64_t>(e->E / 4096, 256 / halves));
  e->M.stride = direct_stride(B);
  const int64_t need = (int64_t)G * B * B + (int64_t)G * halves * 3 * kHistB;
  if (need > e->hist_cap) {
    dfree(e, e->hist);
    e->hist_cap = 0;
    if (int rc = dalloc(e, &e->hist, (size_t)need)) return rc;
    e->hist_cap = need;
  }
  if (int rc = reserve_pool(e, (int64_t)B * e->M.stride)) return rc;
  e->all_direct = true;
  HistArgs a;
  a.g = gview(e);
  a.src = e->out_src;
  a.labels = e->labels;
  a.E = e->E;
  a.B = B;
  a.G = G;
  a.rows = one ? B : (B + 1) / 2;
  a.part = e->hist;
  a.part_d = e->hist + (int64_t)G * B * B;
  const dim3 grid((unsigned)G, (unsigned)halves);
  // LDS for 128 blocks leaves room for two workgroups a CU, for all 200 for one
  // (B = 128, E = 4 M 26 and 28 us)
  if (B * a.rows <= 16384)
    k_hist<16384><<<grid, kHistThreads, 0, st>>>(a);
  else
    k_hist<kHistOne * kHistOne><<<grid, kHistThreads, 0, st>>>(a);
  HistSum b;
  b.M = view(e->M, B);
  b.off = e->M.off;
  b.cap = e->M.cap;
  b.d_out = e->d_out;
  b.d_in = e->d_in;
  b.bsize = e->bsize;
  b.part = a.part;
  b.part_d = a.part_d;
  b.G = G;
  b.parts_d = G * halves;
  k_hist_sum<<<(unsigned)B + 3, kHistB * kSumGroups, 0, st>>>(b);
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

// Full M build from the labels (graph_parallel.hpp:703-759).
int rebuild_M(usap_engine* e) {
  const int32_t B = e->B;
  hipStream_t st = e->stream;
  ev_rec(e, 0);
  if (B <= kHistB) {
    if (int rc = build_hist(e)) return rc;
    ev_rec(e, 1);
    if (e->prof) {
      HIPCHK(hipStreamSynchronize(st));
      prof_add(e, USAP_K_BUILD, ev_ms(e, 0, 1), 1, 0.0);
    }
    e->rebuilds++;
    return USAP_OK;
  }
  {
    ClearArgs c;
    int32_t* arr[kClearArrays] = {e->d_out, e->d_in, e->ecnt_out, e->ecnt_in,
                                  e->bsize, e->M.gmark, e->M.gpend, e->bl_cur};
    for (int i = 0; i < kClearArrays; ++i) c.p[i] = arr[i];
    c.n = B;
    c.flags = e->build_flags;
    k_clear_build<<<std::max(1u, std::min(blocks_for(B, 256), 1024u)), 256, 0, st>>>(c);
  }
  if (e->N > 0) {
    const auto k = e->out_w ? (B <= kDegLds ? k_degrees<true, false> : k_degrees<true, true>)
                            : (B <= kDegLds ? k_degrees<false, false> : k_degrees<false, true>);
    // fewer nodes a workgroup while full ones would leave CUs without any (N =
    // 20000, B = 1000: 256 nodes 4.1 us and 1024 5.6, weighted 64 16 and 256 26), more
    // where the workgroups' sums meet on the blocks' counters (N = 500000, B = 1000:
    // 256 47 and 1024 17, weighted 64 126 and 256 120)
    const int32_t per = e->out_w ? (e->N < 65536 ? 64 : kNodesWgW) : (e->N < 65536 ? 256 : kNodesWg);
    k<<<blocks_for(e->N, per), 256, 0, st>>>(gview(e), e->labels, B, per, e->d_out, e->d_in,
                                             e->ecnt_out, e->ecnt_in, e->bsize);
  }
  const bool by_rows = B > kPairSortB || B == e->N;
  int2* items = by_rows ? e->big_items : nullptr;
  int32_t* n_items = e->build_flags + 1;
  k_caps<<<blocks_for((int64_t)B + 1, 256), 256, 0, st>>>(
      B, e->p.slab_slack, e->out_w ? e->ecnt_out : e->d_out, e->out_w ? e->ecnt_in : e->d_in,
      e->bsize, e->M.cap, e->tmpM, items, n_items);
  HIPCHK(hipGetLastError());
  size_t bytes = 0;
  HIPCHK(rocprim::exclusive_scan(nullptr, bytes, e->tmpM, e->M.off, (int64_t)0, (size_t)B + 1,
                                 rocprim::plus<int64_t>(), st));
  if (bytes > e->scan_tmp_bytes) {
    dfree(e, e->scan_tmp);
    if (int rc = dalloc_raw(e, &e->scan_tmp, bytes)) return rc;
    e->scan_tmp_bytes = bytes;
  }
  bytes = e->scan_tmp_bytes;
  HIPCHK(rocprim::exclusive_scan(e->scan_tmp, bytes, e->tmpM, e->M.off, (int64_t)0, (size_t)B + 1,
                                 rocprim::plus<int64_t>(), st));
  int64_t tot = 0;
  HIPCHK(hipMemcpyAsync(&tot, e->M.off + B, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  DevSpM& m = e->M;
  if (int rc = reserve_pool(e, tot)) return rc;
  // every row direct-mapped (cap B each; a hashed row's cap is below B/8):
  // no insert probes, so no row ever needs growth or an increment parked until
  // the next rebuild, and k_grow only has the batch's error flags to fold
  e->all_direct = tot == (int64_t)B * B;
  m.stride = B;
  if (m.total > 0 && !by_rows) k_fill<<<std::min<int64_t>(blocks_for(m.total, 256), 8192), 256, 0, st>>>(
      e->all_direct ? nullptr : m.key, m.cnt, m.total);
  k_reset_grow<<<blocks_for(kGrowBlocks, 256), 256, 0, st>>>(m.gst, (unsigned long long)m.total);
  if (B > kNBK && m.bs_rows < B) {
    dfree(e, m.bs);
    if (int rc = dalloc(e, &m.bs, (size_t)B * kNBK)) return rc;
    m.bs_rows = B;
  }
  if (by_rows) {
    if (int rc = build_rows(e)) return rc;
  } else if (e->E > 0) {
    if (int rc = build_by_pairs(e)) return rc;
  }
  if (B > kNBK) {
    const bool lng = B > kSumLongB;
    const int32_t rows = std::min(kSumRows, 1 + B / (lng ? 2048 : 4096));
    k_bucket_sums<<<blocks_for(B, rows), lng ? 1024 : 256, 0, st>>>(view(e->M, B), rows);
  }
  HIPCHK(hipGetLastError());
  ev_rec(e, 1);
  int32_t flags = 0;
  HIPCHK(hipMemcpyAsync(&flags, e->build_flags, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  prof_add(e, USAP_K_BUILD, ev_ms(e, 0, 1), 1, 0.0);
  if (flags & (kFlagFull | kFlagMissing))
    return set_err(e, USAP_ESTATE, "M build overflowed a row slab");
  e->rebuilds++;
  return USAP_OK;
}

int check_engine(usap_engine* e) {
  if (!e) return USAP_EINVAL;
  if (!e->has_labels) return set_err(e, USAP_ESTATE, "labels not set");
  return USAP_OK;
}

}  // namespace

namespace {
int refresh_host_graph(usap_engine* e);
}  // namespace

namespace usap {
namespace {
std::mutex g_err_mu;
std::string g_err;
thread_local std::string t_err;
}  // namespace

void set_detached_error(const std::string& msg) {
  std::lock_guard<std::mutex> lk(g_err_mu);
  if (g_err.empty()) g_err = msg;  // the first failure is the informative one
}

void clear_detached_error() {
  std::lock_guard<std::mutex> lk(g_err_mu);
  g_err.clear();
}

const char* detached_error() {
  std::lock_guard<std::mutex> lk(g_err_mu);
  t_err = g_err.empty() ? "no error recorded" : g_err;
  return t_err.c_str();
}

std::vector<usap_phase>& engine_phase_log(usap_engine* e) { return e->phase_log; }
const usap_graph* engine_host_graph(usap_engine* e) {
  if (refresh_host_graph(e) != USAP_OK) return nullptr;
  return &e->hg;
}
const usap_params* engine_params(const usap_engine* e) { return &e->p; }
int32_t engine_rebuilds(const usap_engine* e) { return e->rebuilds; }
// Growth counters, read on the engine's own stream (never the legacy null
// stream, which other engines' threads must not see).
static bool read_grow_state(usap_engine* e, GrowState* g, long long* grows, long long* compactions) {
  if (hipMemcpyAsync(g, e->M.gst, sizeof(GrowState), hipMemcpyDeviceToHost, e->stream) !=
      hipSuccess)
    return false;
  if (hipStreamSynchronize(e->stream) != hipSuccess) return false;
  *grows = *compactions = 0;
  for (const GrowChunk& c : g->chunk) {
    *grows += (long long)c.grows;
    *compactions += (long long)c.compactions;
  }
  return true;
}
void engine_grow_debug(usap_engine* e, long long out[4]) {
  out[0] = out[1] = out[2] = out[3] = 0;
  GrowState g{};
  if (!read_grow_state(e, &g, &out[0], &out[1])) return;
  out[2] = (long long)g.full;
  out[3] = (long long)g.nospace_events;
}
int64_t engine_grows(usap_engine* e) {
  GrowState g{};
  long long n = 0, c = 0;
  return read_grow_state(e, &g, &n, &c) ? (int64_t)n : 0;
}
void engine_set_error(usap_engine* e, const char* msg) { e->err = msg; }
}  // namespace usap

extern "C" {

void usap_default_params(usap_params* p) {
  p->K = 10;
  p->reduction_rate = 0.5;
  p->max_nodal_itr = 100;
  p->num_batch_nodal_update = 4;
  p->nodal_batch = 0;
  p->thr1 = 5e-4;
  p->thr2 = 1e-4;
  p->avg_window = 3;
  p->dfs_depth = 20;
  p->init = USAP_INIT_SCC;
  p->ds_mode = USAP_DS_REF;
  p->seed = 0;
  p->device = 0;
  p->verbose = 0;
  p->slab_slack = 2;
  p->graphs = 0;
}

const char* usap_last_error(const usap_engine* e) {
  if (e) return e->err.c_str();
  return usap::detached_error();
}

int usap_destroy(usap_engine* e) {
  if (!e) return USAP_OK;
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  dfree(e, e->out_ptr);
  dfree(e, e->in_ptr);
  dfree(e, e->out_idx);
  dfree(e, e->in_idx);
  dfree(e, e->out_w);
  dfree(e, e->in_w);
  dfree(e, e->out_src);
  for (int i = 0; i < 2; ++i) {
    dfree(e, e->pair_key[i]);
    dfree(e, e->pair_val[i]);
  }
  dfree(e, e->pair_tmp);
  dfree(e, e->hist);
  dfree(e, e->lam);
  dfree(e, e->labels);
  dfree(e, e->d_out);
  dfree(e, e->d_in);
  dfree(e, e->ecnt_out);
  dfree(e, e->ecnt_in);
  dfree(e, e->bsize);
  dfree(e, e->bl_off);
  dfree(e, e->bl_cur);
  dfree(e, e->bl_nodes);
  dfree(e, e->big_items);
  for (DevSpM* m : {&e->M}) {
    dfree(e, m->off);
    dfree(e, m->cap);
    dfree(e, m->gmark);
    dfree(e, m->key);
    dfree(e, m->cnt);
    dfree(e, m->bs);
    dfree(e, m->gpend);
    dfree(e, m->ovf);
    dfree(e, m->gst);
  }
  dfree(e, e->tmpM);
  dfree(e, e->scan_tmp);
  dfree(e, e->best_s);
  dfree(e, e->best_hi);
  dfree(e, e->best_lo);
  dfree(e, e->map);
  for (int i = 0; i < 2; ++i) {
    dfree(e, e->sort_key[i]);
    dfree(e, e->sort_idx[i]);
  }
  dfree(e, e->sort_tmp);
  dfree(e, e->prop);
  dfree(e, e->prop_ds);
  dfree(e, e->draws);
  dfree(e, e->part);
  dfree(e, e->status);
  dfree(e, e->sweep);
  dfree(e, e->prop_u);
  dfree(e, e->aq_mark);
  dfree(e, e->aq_acc);
  dfree(e, e->build_flags);
  dfree(e, e->uni);
  if (e->gexec) {
    std::lock_guard<std::mutex> lk(g_hip_mu);
    (void)hipGraphExecDestroy(e->gexec);
  }
  dfree(e, e->tstamp);
  pin_put(e->h_sweep, sizeof(Sweep));
  for (int i = 0; i < 2; ++i) pin_put(e->h_chunk[i], sizeof(Sweep));
  pin_put(e->h_short, 64);
  dfree(e, e->big_off);
  dfree(e, e->big_tab);
  dfree(e, e->huge_parts);
  dfree(e, e->ent_part);
  pin_put(e->h_fx, 64);
  for (int i = 0; i < kNumSnap; ++i) dfree(e, e->snap_labels[i]);
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  {
    std::lock_guard<std::mutex> lk(g_hip_mu);
    for (hipEvent_t& ev : e->ev)
      if (ev) (void)hipEventDestroy(ev);
    for (hipEvent_t& ev : e->chunk_ev)
      if (ev) (void)hipEventDestroy(ev);
    if (e->stream && e->own_stream) (void)hipStreamDestroy(e->stream);
  }
  delete e;
  return USAP_OK;
}

}  // extern "C"

namespace {

// Checks a graph (CSR/CSC consistent, ids in range, weights >= 0, total
// weight < 2^31 since M counts and degrees are int32); *wtot = total weight.
int check_graph(const usap_graph* g, int64_t* wtot) {
  if (!g) return USAP_EINVAL;
  if (g->N < 1 || g->E < 0 || !g->out_ptr || !g->in_ptr || (g->E > 0 && (!g->out_idx || !g->in_idx)))
    return USAP_EINVAL;
  if ((g->out_w == nullptr) != (g->in_w == nullptr)) return USAP_EINVAL;
  const int32_t N = g->N;
  const int64_t E = g->E;
  if (g->out_ptr[0] != 0 || g->out_ptr[N] != E || g->in_ptr[0] != 0 || g->in_ptr[N] != E)
    return USAP_EINVAL;
  int64_t w = E;
  if (g->out_w) {
    w = 0;
    for (int64_t i = 0; i < E; ++i) {
      if (g->out_w[i] < 0) return USAP_EINVAL;
      w += g->out_w[i];
    }
  }
  for (int64_t i = 0; i < E; ++i)
    if (g->out_idx[i] < 0 || g->out_idx[i] >= N || g->in_idx[i] < 0 || g->in_idx[i] >= N)
      return USAP_EINVAL;
  if (w >= (int64_t)1 << 31) return USAP_EINVAL;
  *wtot = w;
  return USAP_OK;
}

// lambda[0..maxv] from one table shared by the process's engines (computed
// again only when a graph needs more entries: batches of graphs would
// otherwise spend most of their host time in log()).
void lambda_range(int64_t lo, int64_t hi, int64_t* out) {
  static std::mutex mu;
  static std::vector<int64_t> tab;
  std::lock_guard<std::mutex> lk(mu);
  if ((int64_t)tab.size() <= hi) {
    tab.assign((size_t)hi + 1, 0);
    usap_lambda_table(hi, tab.data());
  }
  std::memcpy(out, tab.data() + lo, sizeof(int64_t) * (size_t)(hi - lo + 1));
}

void lambda_prefix(int64_t maxv, int64_t* out) { lambda_range(0, maxv, out); }

#define TRY(x)          \
  do {                  \
    int _rc = (x);      \
    if (_rc) return _rc; \
  } while (0)

// Global-memory unit tables of the nodes that may have more units than the
// workgroup's LDS table holds (hub_terms<.., true>), the parts of the nodes that
// builds split (k_build_big<true>), and the largest list, from the host copy of
// the offsets.
int build_big_tables(usap_engine* e) {
  const int32_t N = e->N;
  std::vector<int64_t> big((size_t)N, -1);
  std::vector<int2> huge;
  int64_t big_total = 0;
  e->max_list = 0;
  for (int32_t x = 0; x < N; ++x) {
    const int64_t k = (e->h_out_ptr[x + 1] - e->h_out_ptr[x]) + (e->h_in_ptr[x + 1] - e->h_in_ptr[x]);
    e->max_list = std::max(e->max_list, k);
    if (k > kHubUnits) {
      int64_t cap = 1;
      while (cap < 2 * k) cap <<= 1;
      big[x] = big_total;
      big_total += 2 * cap;
    }
    if (k > kBigPart)
      for (int64_t i = 0; i * kHugePart < k; ++i) huge.push_back(make_int2(x, (int32_t)i));
  }
  dfree(e, e->big_off);
  dfree(e, e->big_tab);
  dfree(e, e->huge_parts);
  e->n_huge = 0;
  TRY(dalloc(e, &e->big_off, N));
  TRY(dalloc(e, &e->big_tab, big_total));
  TRY(dalloc(e, &e->huge_parts, huge.size()));
  HIPCHK(hipMemcpyAsync(e->big_off, big.data(), sizeof(int64_t) * N, hipMemcpyHostToDevice, e->stream));
  if (!huge.empty())
    HIPCHK(hipMemcpyAsync(e->huge_parts, huge.data(), sizeof(int2) * huge.size(),
                          hipMemcpyHostToDevice, e->stream));
  e->n_huge = (int32_t)huge.size();
  HIPCHK(hipStreamSynchronize(e->stream));  // the vectors are released on return
  return USAP_OK;
}

// The graph's edges on the device: host copy, CSR/CSC, edge sources, the
// lambda table over [0, wtot] and the tables of large nodes.  Frees
// the previous graph's arrays first (same N).
int load_graph(usap_engine* e, const usap_graph* g, int64_t wtot) {
  const int32_t N = g->N;
  const int64_t E = g->E;
  e->N = N;
  e->E = E;
  e->weighted = g->out_w != nullptr;
  e->h_out_ptr.assign(g->out_ptr, g->out_ptr + N + 1);
  e->h_in_ptr.assign(g->in_ptr, g->in_ptr + N + 1);
  e->h_out_idx.assign(g->out_idx, g->out_idx + E);
  e->h_in_idx.assign(g->in_idx, g->in_idx + E);
  e->h_out_w.clear();
  e->h_in_w.clear();
  if (e->weighted) {
    e->h_out_w.assign(g->out_w, g->out_w + E);
    e->h_in_w.assign(g->in_w, g->in_w + E);
  }
  e->Wtot = wtot;
  e->hg.N = N;
  e->hg.E = E;
  e->hg.out_ptr = e->h_out_ptr.data();
  e->hg.in_ptr = e->h_in_ptr.data();
  e->hg.out_idx = e->h_out_idx.data();
  e->hg.in_idx = e->h_in_idx.data();
  e->hg.out_w = e->weighted ? e->h_out_w.data() : nullptr;
  e->hg.in_w = e->weighted ? e->h_in_w.data() : nullptr;
  for (int32_t** q : {&e->out_idx, &e->in_idx, &e->out_src, &e->out_w, &e->in_w}) dfree(e, *q);
  for (int64_t** q : {&e->out_ptr, &e->in_ptr, &e->lam}) dfree(e, *q);
  TRY(dalloc(e, &e->out_ptr, N + 1));
  TRY(dalloc(e, &e->in_ptr, N + 1));
  TRY(dalloc(e, &e->out_idx, E));
  TRY(dalloc(e, &e->in_idx, E));
  TRY(dalloc(e, &e->out_src, E));
  if (e->weighted) {
    TRY(dalloc(e, &e->out_w, E));
    TRY(dalloc(e, &e->in_w, E));
  }
  TRY(dalloc(e, &e->lam, wtot + 1));
  e->lam_cap = wtot + 1;
  e->host_stale = false;
  std::vector<int64_t> lam((size_t)wtot + 1);
  lambda_prefix(wtot, lam.data());
  std::vector<int32_t> src((size_t)E);
  for (int32_t x = 0; x < N; ++x)
    for (int64_t j = g->out_ptr[x]; j < g->out_ptr[x + 1]; ++j) src[j] = x;
  hipStream_t st = e->stream;
  HIPCHK(hipMemcpyAsync(e->out_ptr, g->out_ptr, sizeof(int64_t) * (N + 1), hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(e->in_ptr, g->in_ptr, sizeof(int64_t) * (N + 1), hipMemcpyHostToDevice, st));
  if (E > 0) {
    HIPCHK(hipMemcpyAsync(e->out_idx, g->out_idx, sizeof(int32_t) * E, hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(e->in_idx, g->in_idx, sizeof(int32_t) * E, hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(e->out_src, src.data(), sizeof(int32_t) * E, hipMemcpyHostToDevice, st));
    if (e->weighted) {
      HIPCHK(hipMemcpyAsync(e->out_w, g->out_w, sizeof(int32_t) * E, hipMemcpyHostToDevice, st));
      HIPCHK(hipMemcpyAsync(e->in_w, g->in_w, sizeof(int32_t) * E, hipMemcpyHostToDevice, st));
    }
  }
  HIPCHK(hipMemcpyAsync(e->lam, lam.data(), sizeof(int64_t) * (wtot + 1), hipMemcpyHostToDevice, st));
  TRY(build_big_tables(e));
  // the host vectors above are released when this returns: wait for the copies
  HIPCHK(hipStreamSynchronize(st));
  return USAP_OK;
}

// One side (CSR or CSC) of an append: the lists at ptr/idx/w grow by the n
// edges whose node is key[i] and other end other[i] (device arrays).
// owner (nullable): also rebuild the per-slot node array (the CSR's edge
// sources).
int append_side(usap_engine* e, int64_t n, const int32_t* key, const int32_t* other,
                const int32_t* w, int64_t*& ptr, int32_t*& idx, int32_t*& wv, int32_t** owner) {
  const int32_t N = e->N;
  const int64_t E1 = e->E + n;
  hipStream_t st = e->stream;
  int32_t *cnt = nullptr, *kin = nullptr, *kout = nullptr, *vin = nullptr, *vout = nullptr;
  int64_t *deg = nullptr, *nptr = nullptr;
  int32_t *nidx = nullptr, *nw = nullptr, *nown = nullptr;
  void* tmp = nullptr;
  int rc = USAP_OK;
  auto release = [&]() {
    dfree(e, cnt);
    dfree(e, kin);
    dfree(e, kout);
    dfree(e, vin);
    dfree(e, vout);
    dfree(e, deg);
    dfree(e, tmp);
  };
  if ((rc = dalloc(e, &cnt, N)) || (rc = dalloc(e, &deg, (size_t)N + 1)) ||
      (rc = dalloc(e, &nptr, (size_t)N + 1)) || (rc = dalloc(e, &kin, n)) ||
      (rc = dalloc(e, &kout, n)) || (rc = dalloc(e, &vin, n)) || (rc = dalloc(e, &vout, n)) ||
      (rc = dalloc(e, &nidx, E1)) || (e->weighted && (rc = dalloc(e, &nw, E1))) ||
      (owner && (rc = dalloc(e, &nown, E1)))) {
    release();
    dfree(e, nptr);
    dfree(e, nidx);
    dfree(e, nw);
    dfree(e, nown);
    return rc;
  }
  int bits = 1;
  while (((int64_t)1 << bits) < (int64_t)N) ++bits;
  size_t b1 = 0, b2 = 0;
  hipError_t he = rocprim::exclusive_scan(nullptr, b1, deg, nptr, (int64_t)0, (size_t)N + 1,
                                          rocprim::plus<int64_t>(), st);
  if (he == hipSuccess)
    he = rocprim::radix_sort_pairs(nullptr, b2, kin, kout, vin, vout, (size_t)n, 0, bits, st);
  if (he == hipSuccess && !(rc = dalloc_raw(e, &tmp, std::max(b1, b2)))) {
    const unsigned g = (unsigned)std::max<int64_t>(1, std::min<int64_t>(blocks_for(n, 256), 16384));
    if ((he = hipMemsetAsync(cnt, 0, sizeof(int32_t) * N, st)) == hipSuccess) {
      k_count_keys<<<g, 256, 0, st>>>(n, key, cnt);
      k_new_deg<<<blocks_for((int64_t)N + 1, 256), 256, 0, st>>>(N, ptr, cnt, deg);
      size_t b = std::max(b1, b2);
      he = rocprim::exclusive_scan(tmp, b, deg, nptr, (int64_t)0, (size_t)N + 1,
                                   rocprim::plus<int64_t>(), st);
    }
    if (he == hipSuccess) he = hipMemcpyAsync(kin, key, sizeof(int32_t) * n, hipMemcpyDeviceToDevice, st);
    if (he == hipSuccess) {
      k_iota<<<g, 256, 0, st>>>(n, vin);
      size_t b = std::max(b1, b2);
      he = rocprim::radix_sort_pairs(tmp, b, kin, kout, vin, vout, (size_t)n, 0, bits, st);
    }
    if (he == hipSuccess) {
      k_move_lists<<<blocks_for(N, 256 / kWave), 256, 0, st>>>(N, ptr, nptr, idx, wv, nidx, nw, nown);
      k_place_new<<<g, 256, 0, st>>>(n, kout, vout, ptr, other, w, nidx, nw, nown);
      he = hipGetLastError();
    }
  }
  release();
  if (rc == USAP_OK && he != hipSuccess)
    rc = set_err(e, USAP_EHIP, std::string("edge append: ") + hipGetErrorString(he));
  if (rc != USAP_OK) {
    dfree(e, nptr);
    dfree(e, nidx);
    dfree(e, nw);
    dfree(e, nown);
    return rc;
  }
  dfree(e, ptr);
  dfree(e, idx);
  dfree(e, wv);
  ptr = nptr;
  idx = nidx;
  wv = nw;
  if (owner) {
    dfree(e, *owner);
    *owner = nown;
  }
  return USAP_OK;
}

// The host copy of the graph from the device lists (after appends).
int refresh_host_graph(usap_engine* e) {
  if (!e->host_stale) return USAP_OK;
  const int64_t E = e->E;
  hipStream_t st = e->stream;
  e->h_out_idx.resize((size_t)E);
  e->h_in_idx.resize((size_t)E);
  e->h_out_w.resize(e->weighted ? (size_t)E : 0);
  e->h_in_w.resize(e->weighted ? (size_t)E : 0);
  if (E > 0) {
    HIPCHK(hipMemcpyAsync(e->h_out_idx.data(), e->out_idx, sizeof(int32_t) * E, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(e->h_in_idx.data(), e->in_idx, sizeof(int32_t) * E, hipMemcpyDeviceToHost, st));
    if (e->weighted) {
      HIPCHK(hipMemcpyAsync(e->h_out_w.data(), e->out_w, sizeof(int32_t) * E, hipMemcpyDeviceToHost, st));
      HIPCHK(hipMemcpyAsync(e->h_in_w.data(), e->in_w, sizeof(int32_t) * E, hipMemcpyDeviceToHost, st));
    }
  }
  HIPCHK(hipStreamSynchronize(st));
  e->hg.E = E;
  e->hg.out_ptr = e->h_out_ptr.data();
  e->hg.in_ptr = e->h_in_ptr.data();
  e->hg.out_idx = e->h_out_idx.data();
  e->hg.in_idx = e->h_in_idx.data();
  e->hg.out_w = e->weighted ? e->h_out_w.data() : nullptr;
  e->hg.in_w = e->weighted ? e->h_in_w.data() : nullptr;
  e->host_stale = false;
  return USAP_OK;
}

// Appends n edges (host arrays, already checked) on the device.
int append_edges(usap_engine* e, int64_t n, const int32_t* src, const int32_t* dst,
                 const int32_t* w, int64_t wsum) {
  hipStream_t st = e->stream;
  const int64_t W1 = e->Wtot + wsum;
  int32_t *ds = nullptr, *dd = nullptr, *dw = nullptr;
  auto release = [&]() {
    dfree(e, ds);
    dfree(e, dd);
    dfree(e, dw);
  };
  TRY(dalloc(e, &ds, n));
  TRY(dalloc(e, &dd, n));
  if (w) TRY(dalloc(e, &dw, n));
  HIPCHK(hipMemcpyAsync(ds, src, sizeof(int32_t) * n, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(dd, dst, sizeof(int32_t) * n, hipMemcpyHostToDevice, st));
  if (w) HIPCHK(hipMemcpyAsync(dw, w, sizeof(int32_t) * n, hipMemcpyHostToDevice, st));
  int rc = append_side(e, n, ds, dd, dw, e->out_ptr, e->out_idx, e->out_w, &e->out_src);
  if (rc == USAP_OK) rc = append_side(e, n, dd, ds, dw, e->in_ptr, e->in_idx, e->in_w, nullptr);
  // the host arrays are the caller's: the copies above must finish first
  const hipError_t he = hipStreamSynchronize(st);
  release();
  if (rc != USAP_OK) return rc;
  if (he != hipSuccess) return set_err(e, USAP_EHIP, std::string("edge append: ") + hipGetErrorString(he));
  e->E += n;
  e->hg.E = e->E;
  // lambda over [0, W1]: the new range only, the table grown geometrically
  if (W1 + 1 > e->lam_cap) {
    const int64_t cap = std::min<int64_t>((int64_t)1 << 31, std::max<int64_t>(W1 + 1, 2 * e->lam_cap));
    int64_t* nl = nullptr;
    TRY(dalloc(e, &nl, cap));
    HIPCHK(hipMemcpyAsync(nl, e->lam, sizeof(int64_t) * (e->Wtot + 1), hipMemcpyDeviceToDevice, st));
    std::vector<int64_t> add((size_t)(cap - 1 - e->Wtot));
    lambda_range(e->Wtot + 1, cap - 1, add.data());
    HIPCHK(hipMemcpyAsync(nl + e->Wtot + 1, add.data(), sizeof(int64_t) * add.size(),
                          hipMemcpyHostToDevice, st));
    HIPCHK(hipStreamSynchronize(st));
    dfree(e, e->lam);
    e->lam = nl;
    e->lam_cap = cap;
  }
  e->Wtot = W1;
  // host offsets (big tables, driver) now; lists on demand
  e->h_out_ptr.resize((size_t)e->N + 1);
  e->h_in_ptr.resize((size_t)e->N + 1);
  HIPCHK(hipMemcpyAsync(e->h_out_ptr.data(), e->out_ptr, sizeof(int64_t) * (e->N + 1), hipMemcpyDeviceToHost, st));
  HIPCHK(hipMemcpyAsync(e->h_in_ptr.data(), e->in_ptr, sizeof(int64_t) * (e->N + 1), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  e->hg.out_ptr = e->h_out_ptr.data();
  e->hg.in_ptr = e->h_in_ptr.data();
  e->host_stale = true;
  TRY(build_big_tables(e));
  const int64_t ocap = std::min<int64_t>(kOvfCap, 2 * e->E + 4096);
  if (ocap > e->M.ovf_cap) {  // the overflow buffer follows the edge count
    dfree(e, e->M.ovf);
    e->M.ovf_cap = (int32_t)ocap;
    TRY(dalloc(e, &e->M.ovf, (size_t)4 * e->M.ovf_cap));
  }
  return USAP_OK;
}

constexpr size_t kShortBytes = 64;  // usap_engine::h_short, h_fx

// Device arrays sized by N only (labels, degrees, row tables, batch buffers).
int alloc_state(usap_engine* e) {
  const int32_t N = e->N;
  TRY(dalloc(e, &e->labels, N));
  TRY(dalloc(e, &e->d_out, N));
  TRY(dalloc(e, &e->d_in, N));
  TRY(dalloc(e, &e->ecnt_out, N));
  TRY(dalloc(e, &e->ecnt_in, N));
  TRY(dalloc(e, &e->bsize, N));
  TRY(dalloc(e, &e->bl_off, N));
  TRY(dalloc(e, &e->bl_cur, N));
  TRY(dalloc(e, &e->bl_nodes, N));
  TRY(dalloc(e, &e->big_items, (size_t)N + N / kBigNodes + 1));
  for (DevSpM* m : {&e->M}) {
    TRY(dalloc(e, &m->off, (size_t)N + 1));
    TRY(dalloc(e, &m->cap, N));
    TRY(dalloc(e, &m->gmark, N));
    TRY(dalloc(e, &m->gpend, N));
    m->ovf_cap = (int32_t)std::min<int64_t>(kOvfCap, 2 * e->E + 4096);
    TRY(dalloc(e, &m->ovf, (size_t)4 * m->ovf_cap));
    TRY(dalloc(e, &m->gst, 1));
  }
  TRY(dalloc(e, &e->tmpM, (size_t)N + 1));
  TRY(dalloc(e, &e->best_s, N));
  TRY(dalloc(e, &e->best_hi, N));
  TRY(dalloc(e, &e->best_lo, N));
  TRY(dalloc(e, &e->map, N));
  TRY(dalloc(e, &e->prop, N));
  TRY(dalloc(e, &e->prop_ds, N));
  TRY(dalloc(e, &e->draws, (size_t)4 * N));
  TRY(dalloc(e, &e->status, 1));
  TRY(dalloc(e, &e->part, blocks_for(N, kNodalWaves)));
  TRY(dalloc(e, &e->sweep, 1));
  TRY(dalloc(e, &e->build_flags, 4));
  TRY(dalloc(e, &e->ent_part, 2 * kEntropyBlocks));
  e->h_sweep = (Sweep*)pin_get(sizeof(Sweep));
  e->h_fx = (int64_t*)pin_get(kShortBytes);
  for (int i = 0; i < 2; ++i) e->h_chunk[i] = (Sweep*)pin_get(sizeof(Sweep));
  e->h_short = (int32_t*)pin_get(kShortBytes);
  if (!e->h_sweep || !e->h_fx || !e->h_chunk[0] || !e->h_chunk[1] || !e->h_short)
    return set_err(e, USAP_ENOMEM, "hipHostMalloc");
  std::memset(e->h_short, 0, kShortBytes);  // a pooled buffer holds another engine's words
  HIPCHK(hipHostGetDevicePointer((void**)&e->d_short, e->h_short, 0));
  HIPCHK(hipHostGetDevicePointer((void**)&e->d_fx, e->h_fx, 0));
  HIPCHK(hipHostGetDevicePointer((void**)&e->d_hsweep, e->h_sweep, 0));
  for (int i = 0; i < 2; ++i)
    HIPCHK(hipHostGetDevicePointer((void**)&e->d_hchunk[i], e->h_chunk[i], 0));
  hipStream_t st = e->stream;
  HIPCHK(hipMemsetAsync(e->status, 0, sizeof(Status), st));
  HIPCHK(hipMemsetAsync(e->sweep, 0, sizeof(Sweep), st));
  HIPCHK(hipMemsetAsync(e->M.gst, 0, sizeof(GrowState), st));
  std::memset(e->h_sweep, 0, sizeof(Sweep));
  {
    std::lock_guard<std::mutex> lk(g_hip_mu);
    for (hipEvent_t& ev : e->ev) HIPCHK(hipEventCreate(&ev));
    for (hipEvent_t& ev : e->chunk_ev) HIPCHK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  }
  return USAP_OK;
}

#undef TRY

}  // namespace

extern "C" {

int usap_create(const usap_graph* g, const usap_params* p, usap_engine** out) {
  return usap::create_in(nullptr, g, p, out);
}

}  // extern "C"

namespace usap {

// A host worker's device context (see engine_internal.hpp).
struct WorkerCtx {
  int32_t device = 0;
  hipStream_t stream = nullptr;
  hipMemPool_t pool = nullptr;
};

// Worker contexts are kept for the life of the process: a released one goes
// back to a free list (its stream synchronised, its pool trimmed to what is
// in use) and the next worker on that device takes it, so repeated batches
// (the autotuner's trials, one batch after another) create no further
// streams or pools and never destroy one while other workers run.
std::mutex g_ctx_mu;
std::vector<WorkerCtx*> g_ctx_free;

int worker_ctx_create(int32_t device, WorkerCtx** out) {
  if (!out) return USAP_EINVAL;
  *out = nullptr;
  if (hipSetDevice(device) != hipSuccess) return USAP_EHIP;
  {
    std::lock_guard<std::mutex> lk(g_ctx_mu);
    for (size_t i = 0; i < g_ctx_free.size(); ++i)
      if (g_ctx_free[i]->device == device) {
        *out = g_ctx_free[i];
        g_ctx_free.erase(g_ctx_free.begin() + (long)i);
        return USAP_OK;
      }
  }
  WorkerCtx* w = new (std::nothrow) WorkerCtx();
  if (!w) return USAP_ENOMEM;
  w->device = device;
  std::lock_guard<std::mutex> lk(g_hip_mu);
  if (hipStreamCreateWithFlags(&w->stream, hipStreamNonBlocking) != hipSuccess) {
    delete w;
    return USAP_EHIP;
  }
  hipMemPoolProps props{};
  props.allocType = hipMemAllocationTypePinned;
  props.location.type = hipMemLocationTypeDevice;
  props.location.id = device;
  if (hipMemPoolCreate(&w->pool, &props) != hipSuccess) {
    (void)hipStreamDestroy(w->stream);
    delete w;
    return USAP_EHIP;
  }
  uint64_t keep = UINT64_MAX;  // freed blocks stay in the pool for the next graph
  (void)hipMemPoolSetAttribute(w->pool, hipMemPoolAttrReleaseThreshold, &keep);
  *out = w;
  return USAP_OK;
}

void worker_ctx_destroy(WorkerCtx* w) {
  if (!w) return;
  (void)hipSetDevice(w->device);
  (void)hipStreamSynchronize(w->stream);
  {
    std::lock_guard<std::mutex> lk(g_hip_mu);
    (void)hipMemPoolTrimTo(w->pool, 0);  // the blocks its engines freed go back to the device
  }
  std::lock_guard<std::mutex> lk(g_ctx_mu);
  g_ctx_free.push_back(w);
}

int create_in(WorkerCtx* ctx, const usap_graph* g, const usap_params* p, usap_engine** out) {
  if (!g || !out) return USAP_EINVAL;
  *out = nullptr;
  int64_t wtot = 0;
  if (int rc = check_graph(g, &wtot)) return rc;
  usap_engine* e = new (std::nothrow) usap_engine();
  if (!e) return USAP_ENOMEM;
  if (p)
    e->p = *p;
  else
    usap_default_params(&e->p);
  if (e->p.K < 1 || e->p.reduction_rate <= 0 || e->p.reduction_rate >= 1 || e->p.avg_window < 2 ||
      e->p.max_nodal_itr < 1 || e->p.slab_slack < 1 || e->p.slab_slack > 16) {
    delete e;
    return USAP_EINVAL;
  }
  e->N = g->N;
  e->E = g->E;
  hipError_t hst = hipSetDevice(e->p.device);
  if (hst != hipSuccess) {
    const int rc = set_err(e, USAP_EHIP, std::string("hipSetDevice: ") + hipGetErrorString(hst));
    usap_destroy(e);
    return rc;
  }
  if (ctx) {
    if (ctx->device != e->p.device) {
      delete e;
      return USAP_EINVAL;
    }
    e->stream = ctx->stream;
    e->pool = ctx->pool;
    e->own_stream = false;
  } else {
    prepare_pool(e->p.device);
    {
      std::lock_guard<std::mutex> lk(g_hip_mu);
      hst = hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking);
    }
    if (hst != hipSuccess) {
      e->stream = nullptr;
      usap_destroy(e);
      return USAP_EHIP;
    }
  }
  int rc = alloc_state(e);
  if (rc == USAP_OK) rc = load_graph(e, g, wtot);
  if (rc != USAP_OK) {
    usap_destroy(e);
    return rc;
  }
  *out = e;
  return USAP_OK;
}

}  // namespace usap

extern "C" {

int usap_set_graph(usap_engine* e, const usap_graph* g) {
  if (!e) return USAP_EINVAL;
  int64_t wtot = 0;
  if (int rc = check_graph(g, &wtot)) return rc;
  if (g->N != e->N) return set_err(e, USAP_EINVAL, "usap_set_graph: node count differs");
  HIPCHK(hipSetDevice(e->p.device));
  HIPCHK(hipStreamSynchronize(e->stream));
  const int64_t cap = std::min<int64_t>(kOvfCap, 2 * g->E + 4096);
  if (cap > e->M.ovf_cap) {  // the overflow buffer follows the edge count
    dfree(e, e->M.ovf);
    e->M.ovf_cap = (int32_t)cap;
    if (int rc = dalloc(e, &e->M.ovf, (size_t)4 * e->M.ovf_cap)) return rc;
  }
  if (int rc = load_graph(e, g, wtot)) return rc;
  e->merge_B = -1;
  return e->has_labels ? rebuild_M(e) : USAP_OK;
}

int usap_append_edges(usap_engine* e, int64_t n, const int32_t* src, const int32_t* dst,
                      const int32_t* w) {
  if (!e || n < 0 || (n > 0 && (!src || !dst))) return USAP_EINVAL;
  if (w != nullptr && !e->weighted)
    return set_err(e, USAP_EINVAL, "usap_append_edges: weights for an unweighted graph");
  if (n == 0) return USAP_OK;
  int64_t wsum = 0;
  for (int64_t i = 0; i < n; ++i) {
    if (src[i] < 0 || src[i] >= e->N || dst[i] < 0 || dst[i] >= e->N)
      return set_err(e, USAP_EINVAL, "usap_append_edges: node id out of range");
    const int64_t wi = w ? w[i] : 1;
    if (wi < 0) return set_err(e, USAP_EINVAL, "usap_append_edges: negative weight");
    wsum += wi;
  }
  if (e->Wtot + wsum >= (int64_t)1 << 31)
    return set_err(e, USAP_EINVAL, "usap_append_edges: total weight reaches 2^31");
  HIPCHK(hipSetDevice(e->p.device));
  if (int rc = append_edges(e, n, src, dst, w, wsum)) return rc;
  e->merge_B = -1;
  return e->has_labels ? rebuild_M(e) : USAP_OK;
}

int usap_create_from_edges(int32_t N, int64_t E, const int32_t* src, const int32_t* dst,
                           const int32_t* w, const usap_params* p, usap_engine** out) {
  if (!out || N < 1 || E < 0 || (E > 0 && (!src || !dst))) return USAP_EINVAL;
  *out = nullptr;
  std::vector<int64_t> zero((size_t)N + 1, 0);
  const int32_t dummy_w = 1;
  usap_graph g{};
  g.N = N;
  g.E = 0;
  g.out_ptr = zero.data();
  g.in_ptr = zero.data();
  g.out_w = w ? &dummy_w : nullptr;  // weighted iff weights are given
  g.in_w = g.out_w;
  usap_engine* e = nullptr;
  if (int rc = usap_create(&g, p, &e)) return rc;
  if (int rc = usap_append_edges(e, E, src, dst, w)) {
    usap::set_detached_error(std::string("usap_create_from_edges: ") + e->err);
    usap_destroy(e);
    return rc;
  }
  *out = e;
  return USAP_OK;
}

int usap_set_labels(usap_engine* e, const int32_t* labels, int32_t B) {
  if (!e || !labels || B < 1 || B > e->N) return USAP_EINVAL;
  for (int32_t x = 0; x < e->N; ++x)
    if (labels[x] < 0 || labels[x] >= B) return set_err(e, USAP_EINVAL, "label out of range");
  HIPCHK(hipMemcpyAsync(e->labels, labels, sizeof(int32_t) * e->N, hipMemcpyHostToDevice, e->stream));
  e->B = B;
  e->has_labels = true;
  e->merge_B = -1;
  if (int rc = rebuild_M(e)) return rc;
  HIPCHK(hipStreamSynchronize(e->stream));  // the labels are the caller's
  return USAP_OK;
}

int usap_get_labels(usap_engine* e, int32_t* out) {
  if (int rc = check_engine(e)) return rc;
  if (!out) return USAP_EINVAL;
  HIPCHK(hipMemcpyAsync(out, e->labels, sizeof(int32_t) * e->N, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  return USAP_OK;
}

int usap_num_blocks(usap_engine* e, int32_t* B) {
  if (int rc = check_engine(e)) return rc;
  if (!B) return USAP_EINVAL;
  *B = e->B;
  return USAP_OK;
}

int usap_get_degrees(usap_engine* e, int32_t* d_out, int32_t* d_in) {
  if (int rc = check_engine(e)) return rc;
  if (d_out)
    HIPCHK(hipMemcpyAsync(d_out, e->d_out, sizeof(int32_t) * e->B, hipMemcpyDeviceToHost, e->stream));
  if (d_in)
    HIPCHK(hipMemcpyAsync(d_in, e->d_in, sizeof(int32_t) * e->B, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  return USAP_OK;
}

int usap_get_M_coo(usap_engine* e, int64_t cap, int32_t* rows, int32_t* cols, int32_t* vals,
                   int64_t* nnz) {
  if (int rc = check_engine(e)) return rc;
  if (!nnz) return USAP_EINVAL;
  const int32_t B = e->B;
  hipStream_t st = e->stream;
  GrowState gs{};
  HIPCHK(hipMemcpyAsync(&gs, e->M.gst, sizeof(GrowState), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  const int64_t used = std::min<int64_t>((int64_t)gs.used, e->M.P);
  std::vector<int64_t> off((size_t)B + 1);
  std::vector<int32_t> capv((size_t)B);
  std::vector<int32_t> key((size_t)used);
  std::vector<Cnt> cnt((size_t)used);
  HIPCHK(hipMemcpyAsync(off.data(), e->M.off, sizeof(int64_t) * (B + 1), hipMemcpyDeviceToHost, st));
  HIPCHK(hipMemcpyAsync(capv.data(), e->M.cap, sizeof(int32_t) * B, hipMemcpyDeviceToHost, st));
  if (used > 0) {
    HIPCHK(hipMemcpyAsync(key.data(), e->M.key, sizeof(int32_t) * used, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(cnt.data(), e->M.cnt, sizeof(Cnt) * used, hipMemcpyDeviceToHost, st));
  }
  HIPCHK(hipStreamSynchronize(st));
  std::vector<std::pair<int32_t, int32_t>> row;
  int64_t k = 0;
  for (int32_t a = 0; a < B; ++a) {
    row.clear();
    for (int64_t j = 0; j < capv[a]; ++j) {
      const int32_t c = capv[a] == B ? (int32_t)j : key[off[a] + j];
      const int32_t v = cnt[off[a] + j].o;  // M[a][c]
      if (c >= 0 && v != 0) row.emplace_back(c, v);
    }
    std::sort(row.begin(), row.end());
    for (auto& cv : row) {
      if (k < cap && rows && cols && vals) {
        rows[k] = a;
        cols[k] = cv.first;
        vals[k] = cv.second;
      }
      ++k;
    }
  }
  *nnz = k;
  return USAP_OK;
}

}  // extern "C"

namespace {
// The host's wait for a word its last launch sets (kWord*): a few microseconds
// after the kernel's store, where a stream synchronisation queues a marker and
// sleeps on its interrupt (N = 20000, 106 sweeps: 21.6 us from a sweep's last
// kernel to the next one's first, now 15).  It yields between reads, so that with
// more workers than CPUs the others run meanwhile (32 graphs of N = 4000, 8 workers
// on 2 CPUs: 127 graphs/s synchronised, 221 without and 334 with the yield; on 16
// CPUs, and for one engine, the same with it as without).  A sweep that takes
// longer than kSpinUs, or an error, is left to the synchronisation.  Profiled
// calls read events and always synchronise.
enum { kWordShort = 0, kWordSweep = 1, kWordFx = 2 };
constexpr int kSpinUs = 1000;

HostWord host_word(usap_engine* e, int slot) {
  e->word_seq = e->word_seq == INT32_MAX ? 1 : e->word_seq + 1;
  e->word_want[slot] = e->word_seq;
  return HostWord{e->d_short + 4 + slot, e->word_seq};
}

int wait_word(usap_engine* e, int slot) {
  if (!e->prof) {
    const int32_t* p = e->h_short + 4 + slot;
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0;; ++i) {
      if (__atomic_load_n(p, __ATOMIC_ACQUIRE) == e->word_want[slot]) return USAP_OK;
      __builtin_ia32_pause();
      if (i % 64 == 63) {
        if (std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(kSpinUs)) break;
        std::this_thread::yield();
      }
    }
  }
  HIPCHK(hipStreamSynchronize(e->stream));
  return USAP_OK;
}

// k_entropy over the pool in use: about four slots per thread, at most
// kEntropyBlocks workgroups (a scan of 1 GB pools at B = 250k is bound by the
// loads in flight).
// No launch when one workgroup takes M itself (k_begin, k_entropy_out).
EntropyIn launch_entropy(usap_engine* e, long* part) {
  EntropyIn in{part, 0, e->M.cnt, e->M.total, e->d_out, e->d_in, e->B, e->lam};
  if (e->all_direct && in.slots <= kEntropyOne) return in;
  const int64_t work = std::max<int64_t>(e->M.P, e->B);
  const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(kEntropyBlocks, blocks_for(work, 1024)));
  k_entropy<<<grid, 256, 0, e->stream>>>(e->M.cnt, e->M.gst, e->d_out, e->d_in, e->B, e->lam,
                                         (int32_t)std::min<int64_t>(e->Wtot, kLamEnt - 1), e->M.P, part);
  in.nparts = grid;
  return in;
}

// ---- allocation-free MDL -----------------------------------------------------
// usap_entropy_noalloc keeps k_entropy's per-workgroup partials in this
// file-scope array instead of the engine's buffer: kEntropyBlocks partials of
// 16 bytes (64 KiB), one copy per GPU the library runs on, held until the
// process ends.  Host code never passes the symbol itself: each device's copy
// is reached through the address hipGetSymbolAddress returns for it on that
// device.
constexpr int kScratchParts = kEntropyBlocks;
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
long* g_scratch_ptr[kMaxDevices] = {};

// The MDL into the caller's device memory (S: model + data term; fx: the data
// term's int128 words, hi then lo): the same integer sum and IEEE operations as
// usap_entropy on the host.
__global__ __launch_bounds__(kBeginThreads) void k_entropy_out(EntropyIn in, double model, double* S,
                                                               int64_t* fx, HostWord done) {
  const i128 data = -block_entropy(in);
  if (threadIdx.x == 0) {
    if (S) *S = model + fx_to_double_dev(data);
    if (fx) {
      fx[0] = (int64_t)(data >> 64);
      fx[1] = (int64_t)(uint64_t)(u128)data;
    }
    host_done(done);
  }
}

// This device's copy of `scratch`: looked up once per device, with the
// device current, on the first allocation-free call there.
int scratch_on(usap_engine* e, long** out) {
  const int dev = e->p.device;
  if (dev < 0 || dev >= kMaxDevices)
    return set_err(e, USAP_EINVAL, "usap_entropy_noalloc: device ordinal beyond 63");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    int cur = -1;
    HIPCHK(hipGetDevice(&cur));
    if (cur != dev) HIPCHK(hipSetDevice(dev));
    void* p = nullptr;
    const hipError_t st = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    if (st != hipSuccess || !p)
      return set_err(e, USAP_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(st));
    g_scratch_ptr[dev] = static_cast<long*>(p);
  }
  *out = g_scratch_ptr[dev];
  return USAP_OK;
}
}  // namespace

extern "C" {

int usap_entropy(usap_engine* e, double* S, int64_t* hi, uint64_t* lo) {
  if (int rc = check_engine(e)) return rc;
  hipStream_t st = e->stream;
  ev_rec(e, 0);
  const EntropyIn in = launch_entropy(e, e->ent_part);
  ev_rec(e, 1);
  k_entropy_out<<<1, kBeginThreads, 0, st>>>(in, 0.0, nullptr, e->d_fx, host_word(e, kWordFx));
  HIPCHK(hipGetLastError());
  if (int rc = wait_word(e, kWordFx)) return rc;
  prof_add(e, USAP_K_ENTROPY, ev_ms(e, 0, 1), 1, 8.0 * e->B + 16.0 * in.nparts);
  const i128 data = mk128((long)e->h_fx[0], (unsigned long)e->h_fx[1]);
  if (hi) *hi = (int64_t)(data >> 64);
  if (lo) *lo = (uint64_t)(u128)data;
  if (S) *S = usap_model_S(e->N, e->E, e->B) + fx_to_double(data);
  return USAP_OK;
}

int usap_entropy_noalloc(usap_engine* e, double* S_dev, int64_t* fx_dev) {
  if (int rc = check_engine(e)) return rc;
  if (!S_dev && !fx_dev) return USAP_EINVAL;
  long* part = nullptr;
  if (int rc = scratch_on(e, &part)) return rc;
  // k_entropy is grid-strided over the pool with at most kScratchParts
  // workgroups, so every engine state fits the scratch
  const int64_t need = std::min<int64_t>(kEntropyBlocks, blocks_for(std::max<int64_t>(e->M.P, e->B), 1024));
  if (need > kScratchParts)
    return set_err(e, USAP_EINVAL, "usap_entropy_noalloc: more partials than the 64 KiB scratch holds");
  const EntropyIn in = launch_entropy(e, part);
  k_entropy_out<<<1, kBeginThreads, 0, e->stream>>>(in, usap_model_S(e->N, e->E, e->B), S_dev, fx_dev,
                                                    HostWord{nullptr, 0});
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

int usap_merge_propose(usap_engine* e, int32_t K, uint64_t stream, int32_t* best_s,
                       double* best_dS) {
  if (int rc = check_engine(e)) return rc;
  if (K < 1) return USAP_EINVAL;
  const int32_t B = e->B;
  MergeArgs a;
  a.M = view(e->M, B);
  a.d_out = e->d_out;
  a.d_in = e->d_in;
  a.lam = e->lam;
  a.lam_last = (int32_t)std::min<int64_t>(e->Wtot, kLamMerge - 1);
  a.B = B;
  a.K = K;
  a.seed = e->p.seed;
  a.stream = stream;
  a.uni = e->uni;
  if (e->uni) {  // the round takes draws uni_pos + r*K + idx
    const int64_t need = (int64_t)B * K;
    if (need > e->uni_n - e->uni_pos)
      return set_err(e, USAP_ESTATE, "pre-drawn uniform stream exhausted: a merge round needs " +
                                         std::to_string(need) + " draws, " +
                                         std::to_string(e->uni_n - e->uni_pos) + " left");
    a.stream = (uint64_t)e->uni_pos;
  }
  a.best_s = e->best_s;
  a.best_hi = e->best_hi;
  a.best_lo = e->best_lo;
  ev_rec(e, 0);
  if (!e->all_direct) {
    // hashed rows by wavefronts; what they leave (direct or large rows) by
    // workgroups (the rebuild's arrays are scratch)
    const MergeList list{e->ecnt_out, e->build_flags + 1};
    k_merge_rows<<<blocks_for(B, kMergeWaves), kMergeWaves * kWave, 0, e->stream>>>(a, list);
    k_merge_list<<<blocks_for(B, kMergeListThreads), kMergeListThreads, 0, e->stream>>>(B, a.best_s,
                                                                                     list);
    const auto k = K > kMergeWaves ? k_merge<kMergeWaves, false, kRowLds>
                                   : k_merge<kMergeWaves, false, kRowLdsFew>;
    k<<<(unsigned)std::min<int32_t>(B, kMergeGrid), std::min(K, kMergeWaves) * kWave, 0, e->stream>>>(a,
                                                                                                   list);
  } else if (K <= kMergeWaves) {
    k_merge<kMergeWaves, true, kRowLdsFew><<<B, K * kWave, 0, e->stream>>>(a, MergeList{});
  } else if (B <= kMergeFew) {
    k_merge<kMergeMany, true, kRowLds><<<B, std::min(K, kMergeMany) * kWave, 0, e->stream>>>(a,
                                                                                            MergeList{});
  } else {
    k_merge<kMergeWaves, true, kRowLds><<<B, kMergeWaves * kWave, 0, e->stream>>>(a, MergeList{});
  }
  HIPCHK(hipGetLastError());
  if (e->uni) e->uni_pos += (int64_t)B * K;
  ev_rec(e, 1);
  if (e->prof) {  // the reference algorithm's bytes: 2 (4 (B+1) + 8 nnz(M)) + 24 B
    k_nnz_bytes<<<(unsigned)std::min<int64_t>(4096, std::max<int64_t>(1, blocks_for(e->M.P, 256))),
                  256, 0, e->stream>>>(e->M.cnt, e->M.P, e->aq_acc + 2 * kAqSlots);
    HIPCHK(hipGetLastError());
    e->kp[USAP_K_MERGE].model_bytes += 8.0 * ((double)B + 1.0) + 24.0 * (double)B;
  }
  e->merge_B = B;
  if (best_s || best_dS) {
    std::vector<long> h((size_t)B);
    std::vector<unsigned long> l((size_t)B);
    if (best_s)
      HIPCHK(hipMemcpyAsync(best_s, e->best_s, sizeof(int32_t) * B, hipMemcpyDeviceToHost, e->stream));
    if (best_dS) {
      HIPCHK(hipMemcpyAsync(h.data(), e->best_hi, sizeof(long) * B, hipMemcpyDeviceToHost, e->stream));
      HIPCHK(hipMemcpyAsync(l.data(), e->best_lo, sizeof(long) * B, hipMemcpyDeviceToHost, e->stream));
    }
    HIPCHK(hipStreamSynchronize(e->stream));
    if (best_dS)
      for (int32_t r = 0; r < B; ++r) best_dS[r] = fx_to_double(mk128(h[r], l[r]));
  } else if (e->prof) {  // the kernel time is read below; else the caller's next step waits
    HIPCHK(hipStreamSynchronize(e->stream));
  }
  prof_add(e, USAP_K_MERGE, ev_ms(e, 0, 1), 1, 0.0);
  return USAP_OK;
}

int usap_merge_result_fx(usap_engine* e, int32_t* best_s, int64_t* hi, uint64_t* lo) {
  if (int rc = check_engine(e)) return rc;
  if (e->merge_B != e->B) return set_err(e, USAP_ESTATE, "no merge proposals for this state");
  const int32_t B = e->B;
  if (best_s) HIPCHK(hipMemcpyAsync(best_s, e->best_s, sizeof(int32_t) * B, hipMemcpyDeviceToHost, e->stream));
  if (hi) HIPCHK(hipMemcpyAsync(hi, e->best_hi, sizeof(int64_t) * B, hipMemcpyDeviceToHost, e->stream));
  if (lo) HIPCHK(hipMemcpyAsync(lo, e->best_lo, sizeof(uint64_t) * B, hipMemcpyDeviceToHost, e->stream));
  if (!best_s && !hi && !lo) {  // only the wait
    k_word<<<1, 1, 0, e->stream>>>(host_word(e, kWordShort));
    HIPCHK(hipGetLastError());
    return wait_word(e, kWordShort);
  }
  HIPCHK(hipStreamSynchronize(e->stream));
  return USAP_OK;
}

}  // extern "C"

namespace {

// e->map and build_flags[3] (and *h_short) for B_to_merge merges of the last
// proposal round.  The arrays of the next rebuild serve as scratch.
int carry_out(usap_engine* e, int32_t B_to_merge) {
  const int32_t B = e->B;
  hipStream_t st = e->stream;
  CarryArgs a;
  a.B = B;
  a.B_to_merge = B_to_merge;
  a.best = e->best_s;
  a.hi = e->best_hi;
  a.lo = e->best_lo;
  a.order = nullptr;
  a.bsize = e->bsize;
  a.map = e->map;
  a.short_of = e->build_flags + 3;
  a.host_short = e->d_short;
  a.done = host_word(e, kWordShort);
  if (B <= kCarryRank) {
    k_carry_one<kCarryRank><<<1, kCarryThreads, 0, st>>>(a);
    HIPCHK(hipGetLastError());
    return USAP_OK;
  }
  // order by (dS, block id): the reference sorts by dS with an unstable sort
  // (graph_parallel.hpp:1230)
  if (!e->sort_idx[0]) {
    for (int i = 0; i < 2; ++i) {
      if (int rc = dalloc(e, &e->sort_key[i], e->N)) return rc;
      if (int rc = dalloc(e, &e->sort_idx[i], e->N)) return rc;
    }
  }
  size_t bytes = 0, scan_bytes = 0;
  HIPCHK(rocprim::radix_sort_pairs(nullptr, bytes, e->sort_key[0], e->sort_key[1], e->sort_idx[0],
                                   e->sort_idx[1], (size_t)B, 0, 64, st));
  int32_t *cyc = e->ecnt_out, *succ = e->ecnt_in, *scan = e->bl_off, *alive = e->bl_cur,
          *par = e->bl_nodes;
  HIPCHK(rocprim::inclusive_scan(nullptr, scan_bytes, succ, scan, (size_t)B,
                                 rocprim::plus<int32_t>(), st));
  bytes = std::max(bytes, scan_bytes);
  HIPCHK(rocprim::exclusive_scan(nullptr, scan_bytes, alive, scan, (int32_t)0, (size_t)B,
                                 rocprim::plus<int32_t>(), st));
  bytes = std::max(bytes, scan_bytes);
  if (bytes > e->sort_tmp_bytes) {
    dfree(e, e->sort_tmp);
    if (int rc = dalloc_raw(e, &e->sort_tmp, bytes)) return rc;
    e->sort_tmp_bytes = bytes;
  }
  const unsigned g = blocks_for(B, 256);
  k_sort_init<<<g, 256, 0, st>>>(B, e->best_lo, e->sort_key[0], e->sort_idx[0]);
  bytes = e->sort_tmp_bytes;
  HIPCHK(rocprim::radix_sort_pairs(e->sort_tmp, bytes, e->sort_key[0], e->sort_key[1],
                                   e->sort_idx[0], e->sort_idx[1], (size_t)B, 0, 64, st));
  k_sort_hi<<<g, 256, 0, st>>>(B, e->best_hi, e->sort_idx[1], e->sort_key[0]);
  bytes = e->sort_tmp_bytes;
  HIPCHK(rocprim::radix_sort_pairs(e->sort_tmp, bytes, e->sort_key[0], e->sort_key[1],
                                   e->sort_idx[1], e->sort_idx[0], (size_t)B, 0, 64, st));
  a.order = e->sort_idx[0];
  if (B <= kCarryOne) {
    k_carry_one<kCarryOne><<<1, kCarryThreads, 0, st>>>(a);
    HIPCHK(hipGetLastError());
    return USAP_OK;
  }
  int32_t* rank = e->sort_idx[1];
  int2* pm[2] = {reinterpret_cast<int2*>(e->sort_key[0]), reinterpret_cast<int2*>(e->sort_key[1])};
  k_carry_init<<<g, 256, 0, st>>>(B, a.order, a.best, rank, pm[0], cyc);
  int cur = 0;
  for (int64_t w = 1; w < B; w *= kCarryHops, cur ^= 1)
    k_carry_jump<<<g, 256, 0, st>>>(B, pm[cur], pm[cur ^ 1]);
  k_carry_cycle<<<g, 256, 0, st>>>(B, pm[cur], cyc);
  k_carry_success<<<g, 256, 0, st>>>(B, pm[cur], cyc, rank, succ);
  bytes = e->sort_tmp_bytes;
  HIPCHK(rocprim::inclusive_scan(e->sort_tmp, bytes, succ, scan, (size_t)B,
                                 rocprim::plus<int32_t>(), st));
  k_carry_link<<<g, 256, 0, st>>>(B, B_to_merge, a.best, rank, succ, scan, par, alive, a.short_of,
                                  a.host_short, a.done);
  for (int64_t w = 1; w < B; w *= kRootHops) k_carry_root<<<g, 256, 0, st>>>(B, par);
  k_carry_alive<<<g, 256, 0, st>>>(B, a.bsize, par, alive);
  bytes = e->sort_tmp_bytes;
  HIPCHK(rocprim::exclusive_scan(e->sort_tmp, bytes, alive, scan, (int32_t)0, (size_t)B,
                                 rocprim::plus<int32_t>(), st));
  k_carry_map<<<g, 256, 0, st>>>(B, par, alive, scan, a.map);
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

}  // namespace

extern "C" {

int usap_merge_apply(usap_engine* e, int32_t B_to_merge, int32_t* B_new) {
  if (int rc = check_engine(e)) return rc;
  const int32_t B = e->B;
  if (e->merge_B != B) return set_err(e, USAP_ESTATE, "merge_apply without merge_propose");
  if (B_to_merge < 0 || B_to_merge >= B) return set_err(e, USAP_EINVAL, "B_to_merge out of range");
  hipStream_t st = e->stream;
  if (int rc = carry_out(e, B_to_merge)) return rc;
  k_relabel<<<blocks_for(e->N, 256), 256, 0, st>>>(e->N, e->labels, e->map, e->build_flags + 3);
  HIPCHK(hipGetLastError());
  if (int rc = wait_word(e, kWordShort)) return rc;
  if (*e->h_short) return set_err(e, USAP_EINFEASIBLE, "carry-out ran out of candidate merges");
  e->B = B - B_to_merge;
  e->merge_B = -1;
  if (B_new) *B_new = e->B;
  return rebuild_M(e);
}

}  // extern "C"

namespace {

// Profiling of a round of batch launches (slot i = the round's batch i, of
// at most `batch` nodes): every workgroup of k_nodal, k_apply and k_grow
// stamps its start and end, and each kernel's time is its first workgroup
// start to its last workgroup end, the kernel's own execution.  Events on
// these launches would add cache flushes between the kernels and slow them.
int prof_begin(usap_engine* e, size_t nslots, int32_t batch) {
  const int32_t G = (int32_t)blocks_for(batch, kNodalWaves);
  const size_t n = nslots * (4 * (size_t)G + 2 + 2 * kGrowBlocks) + 6 * nslots;
  if (e->tstamp_n < n) {
    dfree(e, e->tstamp);
    if (int rc = dalloc(e, &e->tstamp, n)) return rc;
    e->tstamp_n = n;
  }
  e->tstamp_G = G;
  k_stamp_init<<<std::min<unsigned>(blocks_for((int64_t)n, 256), 4096u), 256, 0, e->stream>>>(
      e->tstamp, (int64_t)n);
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

// Adds the kernel times of the round's first `executed` batch slots to the
// profile (after the round's launches).
int prof_end(usap_engine* e, size_t executed) {
  if (executed == 0) return USAP_OK;
  const int32_t G = e->tstamp_G;
  unsigned long long* out = e->tstamp + e->tstamp_n - 6 * executed;  // past every slot's stamps
  k_stamp_reduce<<<(unsigned)(3 * executed), 256, 0, e->stream>>>(e->tstamp, G, kGrowBlocks, out);
  HIPCHK(hipGetLastError());
  std::vector<unsigned long long> t(6 * executed);
  HIPCHK(hipMemcpyAsync(t.data(), out, sizeof(unsigned long long) * 6 * executed,
                        hipMemcpyDeviceToHost, e->stream));
  HIPCHK(hipStreamSynchronize(e->stream));
  const int kid[3] = {USAP_K_NODAL, USAP_K_APPLY, USAP_K_GROW};
  for (size_t i = 0; i < executed; ++i) {
    for (int k = 0; k < 3; ++k) {
      const unsigned long long t0 = t[6 * i + 2 * k], t1 = t[6 * i + 2 * k + 1];
      if (t1 > t0) e->kp[kid[k]].ms += 1e-5 * (double)(t1 - t0);  // 100 MHz clock
      e->kp[kid[k]].launches += 1;
    }
  }
  return USAP_OK;
}

// k_nodal for M all direct or not, a weighted graph or not, with nodes beyond a
// wavefront's registers or without.
typedef void (*NodalKernel)(NodalArgs);
NodalKernel nodal_kernel(bool dense, bool weighted, bool hubs) {
  static const NodalKernel k[8] = {
      k_nodal<false, false, false>, k_nodal<false, false, true>, k_nodal<false, true, false>,
      k_nodal<false, true, true>,   k_nodal<true, false, false>, k_nodal<true, false, true>,
      k_nodal<true, true, false>,   k_nodal<true, true, true>};
  return k[4 * dense + 2 * weighted + hubs];
}

typedef void (*ApplyKernel)(ApplyArgs);
ApplyKernel apply_kernel(bool dense, bool weighted, bool hubs) {
  static const ApplyKernel k[8] = {
      k_apply<false, false, false>, k_apply<false, false, true>, k_apply<false, true, false>,
      k_apply<false, true, true>,   k_apply<true, false, false>, k_apply<true, false, true>,
      k_apply<true, true, false>,   k_apply<true, true, true>};
  return k[4 * dense + 2 * weighted + hubs];
}

// The device state *h_sweep, and the Philox words of nodes [beg, end) in batches
// of `batch` (pre-drawn mode has its own, a captured sweep makes them in the
// graph).  from_state: the starting S is the MDL of the current state, computed
// on the device (no host wait for it).
int launch_begin(usap_engine* e, int32_t beg, int32_t end, int32_t batch, bool from_state,
                 bool draws) {
  BeginArgs a;
  a.init = *e->h_sweep;
  a.sweep = e->sweep;
  a.from_state = from_state;
  a.model = from_state ? usap_model_S(e->N, e->E, e->B) : 0.0;
  a.ent = EntropyIn{};
  if (from_state) a.ent = launch_entropy(e, e->ent_part);
  a.beg = beg;
  a.end = end;
  a.batch = batch;
  a.seed = e->p.seed;
  a.draws = e->draws;
  const unsigned n = draws && !e->uni ? blocks_for((int64_t)end - beg, kBeginThreads) : 0;
  k_begin<<<1 + n, kBeginThreads, 0, e->stream>>>(a);
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

int launch_finish(usap_engine* e, Sweep* host) {
  k_finish<<<1, kWave, 0, e->stream>>>(e->status, e->sweep, host, host_word(e, kWordSweep));
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

// Launches k_nodal + k_apply + k_grow for nodes [beg, end).
int launch_batch(usap_engine* e, int32_t beg, int32_t end, size_t ev_slot, bool grow = true,
                 bool finish = false) {
  const int32_t B = e->B;
  hipStream_t st = e->stream;
  NodalArgs a;
  a.g = gview(e);
  a.M = view(e->M, B);
  a.labels = e->labels;
  a.d_out = e->d_out;
  a.d_in = e->d_in;
  a.lam = e->lam;
  a.lam_last = (int32_t)std::min<int64_t>(e->Wtot, kLamLds - 1);
  a.B = B;
  a.beg = beg;
  a.end = end;
  a.exact = e->p.ds_mode == USAP_DS_EXACT;
  // profiled: this slot's workgroup stamps (k_nodal: G starts + G ends;
  // k_apply: G + 1 each; k_grow: kGrowBlocks each)
  const int32_t G = e->tstamp_G;
  unsigned long long* ts =
      e->prof ? e->tstamp + ev_slot * (4 * (size_t)G + 2 + 2 * kGrowBlocks) : nullptr;
  a.tstamp = ts;
  a.tstride = G;
  a.big_off = e->big_off;
  a.big_tab = e->big_tab;
  a.prop = e->prop;
  a.prop_ds = e->prop_ds;
  a.prop_u = e->prof ? e->prop_u : nullptr;
  a.draws = e->uni ? e->uni : e->draws;
  a.predrawn = e->uni != nullptr;
  a.part = e->part;
  a.status = e->status;
  a.sweep = e->sweep;
  ApplyArgs b;
  b.g = a.g;
  b.M = a.M;
  b.labels = e->labels;
  b.d_out = e->d_out;
  b.d_in = e->d_in;
  b.bsize = e->bsize;
  b.beg = beg;
  b.end = end;
  b.prop = e->prop;
  const unsigned grid = blocks_for((int64_t)end - beg, kNodalWaves);
  b.part = e->part;
  b.nparts = grid;
  b.status = e->status;
  b.sweep = e->sweep;
  b.host = finish ? e->d_hsweep : nullptr;
  b.done = finish ? host_word(e, kWordSweep) : HostWord{nullptr, 0};
  b.tstamp = ts ? ts + 2 * (size_t)G : nullptr;
  b.tstride = G + 1;
  GrowArgs ga;
  {
    const DevSpM& m = e->M;
    GrowSide& gs = ga.side;
    gs.off = m.off;
    gs.cap = m.cap;
    gs.gmark = m.gmark;
    // an eighth of the tail left by the rebuild, over the workgroups
    const int64_t share = (m.P - m.total) / (8 * kGrowBlocks) / 32 * 32;
    gs.chunk = share < kWaveSlab ? 0 : (int32_t)std::min<int64_t>(share, 8192);
    gs.bs = m.bs;
    gs.key = m.key;
    gs.cnt = m.cnt;
    gs.gpend = m.gpend;
    gs.ovf = m.ovf;
    gs.ovf_cap = m.ovf_cap;
    gs.gst = m.gst;
    gs.P = m.P;
    gs.slack = m.slack;
  }
  ga.M = a.M;
  ga.B = e->all_direct ? 0 : B;  // no row grows while all are direct: only the flags
  ga.sweep = e->sweep;
  ga.status = e->status;
  ga.tstamp = ts ? ts + 4 * (size_t)G + 2 : nullptr;
  ga.tstride = kGrowBlocks;
  if (e->prof && (int64_t)grid > G)
    return set_err(e, USAP_ESTATE, "profiled batch larger than its stamp slot");
  nodal_kernel(e->all_direct, e->weighted, e->max_list > kRegUnits * kWave)<<<
      grid, kWave * kNodalWaves, 0, st>>>(a);
  if (e->prof) {  // the reference algorithm's bytes for this batch (M not yet changed)
    AqArgs q;
    q.g = a.g;
    q.M = a.M;
    q.beg = beg;
    q.end = end;
    q.prop = e->prop;
    q.prop_u = e->prop_u;
    q.mark = e->aq_mark;
    q.stamp = e->aq_stamp++;
    q.sweep = e->sweep;
    q.acc = e->aq_acc;
    k_aq<<<grid, kWave * kNodalWaves, 0, st>>>(q);
  }
  apply_kernel(e->all_direct, e->weighted, e->max_list > kRegUnits * kWave)<<<
      grid + 1, kWave * kNodalWaves, 0, st>>>(b);  // block 0: the update step
  if (grow) k_grow<<<e->all_direct ? 1 : kGrowBlocks, 256, 0, st>>>(ga);
  HIPCHK(hipGetLastError());
  return USAP_OK;
}

// The batches [0, nb) of a sweep as one HIP graph, captured on first use
// and replayed while B, the batch size, every device pointer the batch
// kernels take (epoch) and whether every row of M is direct stay the same; the
// sweep's state (random stream, convergence inputs) lives in device memory, so
// the kernels' arguments do not change between sweeps.  all_direct picks the
// kernels and what k_grow looks at, and follows the labels, not B alone (a
// block with few edges has a hashed row at B > 256), so a rebuild at the same B
// that allocates nothing may change it.  GrowSide::chunk follows the rebuild's
// total too, but any chunk is right; within one pool it differs by half at
// most.  The graph holds kernel nodes only.
int sweep_graph(usap_engine* e, int32_t batch, int32_t nb) {
  hipStream_t st = e->stream;
  if (!e->gexec || e->g_B != e->B || e->g_batch != batch || e->g_nb != nb ||
      e->g_direct != e->all_direct || e->g_epoch != e->epoch) {
    if (e->gexec) {
      std::lock_guard<std::mutex> lk(g_hip_mu);
      (void)hipGraphExecDestroy(e->gexec);
      e->gexec = nullptr;
    }
    HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    int rc = USAP_OK;
    if (!e->uni)
      k_draw<<<blocks_for(e->N, 256), 256, 0, st>>>(0, e->N, batch, e->p.seed, e->sweep, e->draws);
    for (int32_t i = 0; i < nb && rc == USAP_OK; ++i) {
      const int32_t beg = i * batch;
      const int32_t end = std::min<int64_t>((int64_t)beg + batch, e->N);
      rc = launch_batch(e, beg, end, 0);
    }
    hipGraph_t graph = nullptr;
    const hipError_t ce = hipStreamEndCapture(st, &graph);
    std::unique_lock<std::mutex> lk(g_hip_mu);
    if (rc != USAP_OK) {
      if (ce == hipSuccess && graph) (void)hipGraphDestroy(graph);
      return rc;
    }
    HIPCHK(ce);
    const hipError_t ie = hipGraphInstantiate(&e->gexec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    lk.unlock();
    if (ie != hipSuccess) {
      e->gexec = nullptr;
      return set_err(e, USAP_EHIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(ie));
    }
    e->g_B = e->B;
    e->g_batch = batch;
    e->g_nb = nb;
    e->g_direct = e->all_direct;
    e->g_epoch = e->epoch;
    e->graph_captures++;
  }
  HIPCHK(hipGraphLaunch(e->gexec, st));
  return USAP_OK;
}

// Runs the batches [first, last) of a sweep (batch nodes each) from the
// device state already in e->sweep, one host synchronisation at the end;
// rebuilds M and resumes when a batch overflowed a row slab.  Stops early
// when the sweep's convergence test fires.
constexpr int32_t kChunk = 16;  // batches per launch chunk of a sweep that may converge

int run_sweep(usap_engine* e, int32_t batch, int32_t first, int32_t last, int32_t* rebuilds) {
  hipStream_t st = e->stream;
  Sweep& hs = *e->h_sweep;
  int32_t next = first;
  for (;;) {
    bool finished = false;  // by the last batch's k_apply
    if (e->p.graphs && !e->prof && next == 0) {
      if (int rc = sweep_graph(e, batch, last)) return rc;
    } else {
      if (e->prof)
        if (int rc = prof_begin(e, (size_t)(last - next), batch)) return rc;
      // A sweep whose convergence test is active stops at a batch nobody
      // knows in advance, and the batches launched after it exit at once
      // (a few us each).  Such a sweep goes out in chunks of kChunk batches,
      // one chunk ahead of the host: before the host waits for chunk c's
      // state, chunk c + 1 is queued, so the device never idles and at most
      // one chunk is launched past the stop.
      const bool chunked = !e->prof && hs.check && last - next > 2 * kChunk;
      size_t slot = 0;
      int32_t c = 0;
      for (int32_t i0 = next; i0 < last; ++c) {
        const int32_t upto = chunked ? std::min<int32_t>(last, i0 + kChunk) : last;
        for (int32_t i = i0; i < upto; ++i, ++slot) {
          const int32_t beg = i * batch;
          const int32_t end = std::min<int64_t>((int64_t)beg + batch, e->N);
          // with every row direct nothing grows, and the flags of the chunk's
          // batches (they only report inconsistent M) are folded at its end
          const bool grow = !e->all_direct || e->prof;
          finished = !grow && !chunked && i + 1 == last;
          if (int rc = launch_batch(e, beg, end, slot, grow, finished)) return rc;
        }
        i0 = upto;
        if (!chunked) break;
        if (int rc = launch_finish(e, e->d_hchunk[c & 1])) return rc;
        HIPCHK(hipEventRecord(e->chunk_ev[c & 1], st));
        if (c > 0) {
          HIPCHK(hipEventSynchronize(e->chunk_ev[(c - 1) & 1]));
          if (e->h_chunk[(c - 1) & 1]->stop != 0) break;
        }
      }
    }
    if (!finished)
      if (int rc = launch_finish(e, e->d_hsweep)) return rc;
    if (int rc = wait_word(e, kWordSweep)) return rc;
    const int32_t executed = first + hs.done - next;  // batches run in this launch round
    if (e->prof)
      if (int rc = prof_end(e, (size_t)executed)) return rc;
    if (hs.stop == 3) return set_err(e, USAP_ESTATE, "inconsistent M during a nodal batch");
    if (hs.flags & kFlagFull) {
      if (int rc = rebuild_M(e)) return rc;
      if (rebuilds) ++*rebuilds;
    }
    if (hs.stop != 2 || first + hs.done >= last) break;
    // resume after the rebuild
    next = first + hs.done;
    hs.stop = 0;
    hs.flags = 0;
    HIPCHK(hipMemcpyAsync(e->sweep, &hs, sizeof(Sweep), hipMemcpyHostToDevice, st));
  }
  if (e->prof) {
    e->kp[USAP_K_NODAL].bytes += (double)hs.nodal_bytes;
    e->kp[USAP_K_APPLY].bytes += (double)hs.apply_bytes;
  }
  return USAP_OK;
}

void init_sweep(usap_engine* e, uint64_t stream0, double S, double mean, double thr,
                int32_t check) {
  Sweep& hs = *e->h_sweep;
  std::memset(&hs, 0, sizeof(Sweep));
  hs.stream0 = stream0;
  hs.S = S;
  hs.mean = mean;
  hs.thr = thr;
  hs.check = check;
}

}  // namespace

extern "C" {

int usap_nodal_batch(usap_engine* e, int32_t begin, int32_t end, uint64_t stream, double* dS_sum,
                     int32_t* n_moves) {
  if (int rc = check_engine(e)) return rc;
  if (begin < 0 || end > e->N || begin > end) return USAP_EINVAL;
  if (e->uni) {  // node n takes draw uni_pos + (n - begin)
    if (end - begin > e->uni_n - e->uni_pos)
      return set_err(e, USAP_ESTATE, "pre-drawn uniform stream exhausted: a nodal batch needs " +
                                         std::to_string(end - begin) + " draws, " +
                                         std::to_string(e->uni_n - e->uni_pos) + " left");
    stream = (uint64_t)(e->uni_pos - begin);
  }
  e->last_beg = begin;
  e->last_end = end;
  init_sweep(e, stream, 0.0, 0.0, 0.0, 0);
  if (begin < end) {
    // one batch of size end-begin starting at begin: index 0 of a sweep whose
    // "batch" starts at begin
    if (int rc = launch_begin(e, begin, end, end - begin, false, true)) return rc;
    if (e->prof)
      if (int rc = prof_begin(e, 1, end - begin)) return rc;
    if (int rc = launch_batch(e, begin, end, 0)) return rc;
    Sweep& hs = *e->h_sweep;
    if (int rc = launch_finish(e, e->d_hsweep)) return rc;
    if (int rc = wait_word(e, kWordSweep)) return rc;
    if (e->prof) {
      if (int rc = prof_end(e, 1)) return rc;
      e->kp[USAP_K_NODAL].bytes += (double)hs.nodal_bytes;
      e->kp[USAP_K_APPLY].bytes += (double)hs.apply_bytes;
    }
    if (hs.stop == 3) return set_err(e, USAP_ESTATE, "inconsistent M during a nodal batch");
    if (e->uni) e->uni_pos += end - begin;
    if (hs.flags & kFlagFull)
      if (int rc = rebuild_M(e)) return rc;
  }
  const Sweep& hs = *e->h_sweep;
  if (dS_sum) *dS_sum = hs.cum_inf ? -INFINITY : fx_to_double(mk128((long)hs.cum_hi, (unsigned long)hs.cum_lo));
  if (n_moves) *n_moves = (int32_t)hs.moves;
  return USAP_OK;
}

int usap_nodal_sweep(usap_engine* e, int32_t batch, uint64_t stream0, double S, double mean,
                     double thr, int32_t check, usap_sweep* out) {
  return usap::nodal_sweep(e, batch, stream0, &S, mean, thr, check, out);
}

int usap_set_uniforms(usap_engine* e, const double* u, size_t n) {
  if (!e) return USAP_EINVAL;
  if (n % 4 || (n && !u))
    return set_err(e, USAP_EINVAL, "usap_set_uniforms: n must be a multiple of 4 (four uniforms per draw)");
  std::vector<uint64_t> w(n);
  for (size_t i = 0; i < n; ++i) {
    if (!(u[i] >= 0.0 && u[i] < 1.0))
      return set_err(e, USAP_EINVAL, "usap_set_uniforms: u[" + std::to_string(i) + "] is not in [0, 1)");
    w[i] = (uint64_t)std::ldexp(u[i], 64);  // floor(u * 2^64): exact below 2^64
  }
  dfree(e, e->uni);
  e->uni_n = 0;
  e->uni_pos = 0;
  e->epoch++;  // a captured sweep holds the old pointer
  if (n) {
    if (int rc = dalloc(e, &e->uni, n)) return rc;
    HIPCHK(hipMemcpyAsync(e->uni, w.data(), sizeof(uint64_t) * n, hipMemcpyHostToDevice, e->stream));
    HIPCHK(hipStreamSynchronize(e->stream));
    e->uni_n = (int64_t)(n / 4);
  }
  return USAP_OK;
}

int usap_uniforms_used(usap_engine* e, int64_t* draws) {
  if (!e || !draws) return USAP_EINVAL;
  *draws = e->uni_pos;
  return USAP_OK;
}

}  // extern "C"

namespace usap {

// usap_nodal_sweep; with S null the sweep's starting S is the entropy of the
// current state, computed on the device between the state copy and the first
// batch (no host wait for it).
int nodal_sweep(usap_engine* e, int32_t batch, uint64_t stream0, const double* S, double mean,
                double thr, int32_t check, usap_sweep* out) {
  if (int rc = check_engine(e)) return rc;
  if (batch < 1 || !out) return USAP_EINVAL;
  double S0 = 0.0;
  if (!S && e->prof) {  // profiled: the entropy scan is timed on its own
    if (int rc = usap_entropy(e, &S0, nullptr, nullptr)) return rc;
    S = &S0;
  }
  const int32_t nb = (int32_t)(((int64_t)e->N + batch - 1) / batch);
  if (e->uni) {  // node n takes draw uni_pos + n; the sweep needs all N available
    if (e->N > e->uni_n - e->uni_pos)
      return set_err(e, USAP_ESTATE, "pre-drawn uniform stream exhausted: a nodal sweep needs " +
                                         std::to_string(e->N) + " draws, " +
                                         std::to_string(e->uni_n - e->uni_pos) + " left");
    stream0 = (uint64_t)e->uni_pos;
  }
  init_sweep(e, stream0, S ? *S : 0.0, mean, thr, check);
  if (int rc = launch_begin(e, 0, e->N, batch, !S, !(e->p.graphs && !e->prof))) return rc;
  int32_t rebuilds = 0;
  if (int rc = run_sweep(e, batch, 0, nb, &rebuilds)) return rc;
  const Sweep& hs = *e->h_sweep;
  const int32_t last = hs.done - 1;  // the last executed batch
  e->last_beg = last * batch;
  e->last_end = std::min<int64_t>((int64_t)e->last_beg + batch, e->N);
  out->batches = hs.done;
  out->proposals = std::min<int64_t>((int64_t)hs.done * batch, e->N);
  if (e->uni) e->uni_pos += out->proposals;
  out->converged = hs.stop == 1;
  out->moves = (int64_t)hs.moves;
  out->S = hs.S;
  out->dS_sum = hs.dS_last;
  out->dS_hi = (int64_t)hs.cum_hi;
  out->dS_lo = (uint64_t)hs.cum_lo;
  out->dS_inf = hs.cum_inf ? -1 : 0;
  out->rebuilds = rebuilds;
  return USAP_OK;
}

}  // namespace usap

extern "C" {

int usap_nodal_sum_fx(usap_engine* e, int64_t* hi, uint64_t* lo, int32_t* inf) {
  if (int rc = check_engine(e)) return rc;
  const Sweep& hs = *e->h_sweep;
  if (hi) *hi = (int64_t)hs.cum_hi;
  if (lo) *lo = (uint64_t)hs.cum_lo;
  if (inf) *inf = hs.cum_inf ? -1 : 0;
  return USAP_OK;
}

int usap_nodal_detail(usap_engine* e, int32_t* s, int64_t* hi, uint64_t* lo, int32_t* inf,
                      int32_t* accept) {
  if (int rc = check_engine(e)) return rc;
  const int64_t n = e->last_end - e->last_beg;
  hipStream_t st = e->stream;
  if (n > 0) {
    std::vector<Prop> p((size_t)n);
    std::vector<PropDs> d((size_t)n);
    HIPCHK(hipMemcpyAsync(p.data(), e->prop, sizeof(Prop) * n, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(d.data(), e->prop_ds, sizeof(PropDs) * n, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    for (int64_t i = 0; i < n; ++i) {
      if (s) s[i] = p[i].s;
      if (hi) hi[i] = d[i].hi;
      if (lo) lo[i] = d[i].lo;
      if (inf) inf[i] = p[i].inf;
      if (accept) accept[i] = p[i].acc;
    }
  }
  return USAP_OK;
}

int usap_profile(usap_engine* e, int32_t enable, usap_kernel_prof* out) {
  if (!e) return USAP_EINVAL;
  if (out) {
    for (int k = 0; k < USAP_NKERNELS; ++k) out[k] = e->kp[k];
    if (e->aq_acc && e->prof) {
      unsigned long long acc[3 * kAqSlots];
      HIPCHK(hipMemcpyAsync(acc, e->aq_acc, sizeof(acc), hipMemcpyDeviceToHost, e->stream));
      HIPCHK(hipStreamSynchronize(e->stream));
      for (int j = 0; j < 2 * kAqSlots; ++j) out[USAP_K_NODAL].model_bytes += (double)acc[j];
      for (int j = 0; j < kAqSlots; ++j) out[USAP_K_MERGE].model_bytes += (double)acc[2 * kAqSlots + j];
    }
  }
  if (enable == 1) {
    for (int k = 0; k < USAP_NKERNELS; ++k) e->kp[k] = usap_kernel_prof{};
    if (!e->prop_u) {
      if (int rc = dalloc(e, &e->prop_u, e->N)) return rc;
      if (int rc = dalloc(e, &e->aq_mark, e->N)) return rc;
      if (int rc = dalloc(e, &e->aq_acc, 3 * kAqSlots)) return rc;
      HIPCHK(hipMemsetAsync(e->aq_mark, 0xff, sizeof(int32_t) * e->N, e->stream));
      e->aq_stamp = 0;
    }
    HIPCHK(hipMemsetAsync(e->aq_acc, 0, 3 * kAqSlots * sizeof(unsigned long long), e->stream));
    e->prof = true;
  } else if (enable == 0) {
    e->prof = false;
  }
  return USAP_OK;
}

int usap_partition_log(usap_engine* e, int32_t cap, usap_phase* out, int32_t* n) {
  if (!e || !n) return USAP_EINVAL;
  const int32_t m = (int32_t)e->phase_log.size();
  for (int32_t i = 0; i < m && i < cap && out; ++i) out[i] = e->phase_log[i];
  *n = m;
  return USAP_OK;
}

int usap_snapshot(usap_engine* e, int32_t slot, double S) {
  if (int rc = check_engine(e)) return rc;
  if (slot < 0 || slot >= kNumSnap) return USAP_EINVAL;
  if (!e->snap_labels[slot])
    if (int rc = dalloc(e, &e->snap_labels[slot], e->N)) return rc;
  HIPCHK(hipMemcpyAsync(e->snap_labels[slot], e->labels, sizeof(int32_t) * e->N,
                        hipMemcpyDeviceToDevice, e->stream));
  e->snap_B[slot] = e->B;
  e->snap_S[slot] = S;
  return USAP_OK;
}

int usap_restore(usap_engine* e, int32_t slot) {
  if (int rc = check_engine(e)) return rc;
  if (slot < 0 || slot >= kNumSnap || !e->snap_labels[slot]) return USAP_EINVAL;
  HIPCHK(hipMemcpyAsync(e->labels, e->snap_labels[slot], sizeof(int32_t) * e->N,
                        hipMemcpyDeviceToDevice, e->stream));
  e->B = e->snap_B[slot];
  e->merge_B = -1;
  return rebuild_M(e);
}

}  // extern "C"
