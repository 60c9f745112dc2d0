// Device side of the LSM dictionary, for (uint32 key, uint32 value) rows and
// (uint64 key, uint64 value) rows.  Every kernel is a template over the row
// traits KV<K> below.
//
// Data model in HBM.  The dictionary is a stack of immutable sorted runs,
// newest first.  A run of c rows is two allocations:
//   rows[c]  rows of (key word, value): the key word holds the low B-1 bits
//            of the key with the tombstone flag in its top bit, the value
//            is 0 for a tombstone (B = key bits)
//   dir      RunMeta header (count, split, directory bits, tombstones,
//            bucket window) followed by a radix directory of 2^b + 1 u32
//            row offsets: dir[j] = first row whose key >= j << (B - b),
//            valid for j in [lo_bucket, hi_bucket + 1], the buckets of the
//            run's first and last keys; a key below that window has
//            lower bound 0, a key above it has lower bound count, so the
//            empty stretches of key space below and above the run are
//            never written.
// The top bit of a key is implied by the row position (rows >= split have
// it set), which frees it for the tombstone flag, so a row is exactly
// 2 * sizeof(K) bytes like the reference's 8-byte Row (GPULSMOpt.cuh:
// 343-377), and key and value share one cache line, so a point hit costs
// one line of rows.  Every search enters through the directory (b >= 1);
// inside one directory bucket all keys share the top bit, so comparisons
// use the low B-1 bits only.
#pragma once

#include "device_utils.hpp"
#include "radix_sort.hpp"

namespace gdict {
namespace lsm {

constexpr int kMaxRuns = 48;
constexpr u32 kMaxDirBits = 24;

struct RunMeta {
  u32 count;
  u32 split;      // rows whose key has the top bit clear
  u32 dir_bits;   // b, 1 <= b <= kMaxDirBits
  u32 tombs;      // nonzero when the run holds tombstone rows
  u32 lo_bucket;  // directory window: buckets of the first and last key
  u32 hi_bucket;  // (lo_bucket = 1, hi_bucket = 0: no rows)
};
constexpr u64 kMetaWords = sizeof(RunMeta) / sizeof(u32);
constexpr u64 kMetaBytes = 256;  // header slot in front of the directory

struct alignas(16) Row64 {
  u64 k;  // key word
  u64 v;  // value
};

// Row traits.  kSmallTile: keys a fused one-workgroup admission sorts in
// LDS; kMergeItemsMax: merge items per thread (merge tile = 256 x items),
// both sized so the LDS staging stays below 64 KB.
template <class K>
struct KV;

template <>
struct KV<u32> {
  using K = u32;
  using V = u32;
  using Row = uint2;
  static constexpr int kBits = 32;
  static constexpr K kTomb = 0x80000000u;
  static constexpr K kLow = 0x7fffffffu;
  static constexpr K kAllOnes = 0xffffffffu;
  static constexpr int kSmallTile = 4096;
  static constexpr int kMergeItemsMax = 16;
  __device__ __forceinline__ static K kw(const Row &r) { return r.x; }
  __device__ __forceinline__ static V val(const Row &r) { return r.y; }
  __device__ __forceinline__ static Row make(K kw, V v) {
    return make_uint2(kw, v);
  }
};

template <>
struct KV<u64> {
  using K = u64;
  using V = u64;
  using Row = Row64;
  static constexpr int kBits = 64;
  static constexpr K kTomb = 0x8000000000000000ull;
  static constexpr K kLow = 0x7fffffffffffffffull;
  static constexpr K kAllOnes = ~0ull;
  static constexpr int kSmallTile = 2048;
  static constexpr int kMergeItemsMax = 8;
  __device__ __forceinline__ static K kw(const Row &r) { return r.k; }
  __device__ __forceinline__ static V val(const Row &r) { return r.v; }
  __device__ __forceinline__ static Row make(K kw, V v) {
    Row r;
    r.k = kw;
    r.v = v;
    return r;
  }
};

template <class T>
struct RunView {
  const typename T::Row *rows;
  const u32 *dir;
  const RunMeta *meta;
};

template <class T>
struct RunSet {
  u32 count;
  u32 pad;
  RunView<T> run[kMaxRuns];
};

template <class T>
__device__ __forceinline__ typename T::K decode_key(typename T::K w, u32 pos,
                                                    u32 split) {
  return (w & T::kLow) | (pos >= split ? T::kTomb : typename T::K(0));
}

// Directory bits for `count` rows: about 2^rows_log rows per bucket.
__host__ __device__ __forceinline__ u32 dir_bits_for(u64 count, u32 max_bits,
                                                     u32 rows_log = 3) {
  u32 lg = 0;
  while (lg < 63 && (u64(1) << (lg + 1)) <= count) ++lg;
  u32 b = lg > rows_log ? lg - rows_log : 1;
  if (b < 1) b = 1;
  if (b > max_bits) b = max_bits;
  return b;
}

// Directory bounds [lo, hi) of the rows that may hold key x; false when x
// lies outside the run's bucket window (then lo = hi = its lower bound).
template <class T>
__device__ __forceinline__ bool dir_window(const RunView<T> &r,
                                           const RunMeta &m, typename T::K x,
                                           u32 &lo, u32 &hi) {
  const u32 bucket = static_cast<u32>(x >> (T::kBits - m.dir_bits));
  if (bucket < m.lo_bucket) {
    lo = hi = 0;
    return false;
  }
  if (bucket > m.hi_bucket) {
    lo = hi = m.count;
    return false;
  }
  u64 both;  // (one load for the two bounds)
  __builtin_memcpy(&both, r.dir + bucket, sizeof(both));
  lo = static_cast<u32>(both);
  hi = static_cast<u32>(both >> 32);
  return true;
}

// First row in [lo, hi) whose key's low bits are >= target (the rows of
// one directory bucket): bisection down to kFindWindow rows, then one batch
// of loads.
//
// A load whose 64 lanes look in 64 different places takes the L1 64 cycles, and
// searches of a thread per query are bound by those, not by their round trips:
// a window of eight rows (no bisection in most buckets) measured 353 us for
// 8,388,608 grouped lookups in 33.5 million rows, one of two 328; 1000 lookups
// take 3.4 us with either.
constexpr u32 kFindWindow = 2;

template <class T>
__device__ __forceinline__ u32 window_lower_bound(const typename T::Row *rows,
                                                  u32 lo, u32 hi,
                                                  typename T::K target) {
  while (hi - lo > kFindWindow) {
    const u32 mid = (lo + hi) >> 1;
    if ((T::kw(rows[mid]) & T::kLow) < target) lo = mid + 1;
    else hi = mid;
  }
  typename T::Row w[kFindWindow];
#pragma unroll
  for (u32 i = 0; i < kFindWindow; ++i)
    if (lo + i < hi) w[i] = rows[lo + i];
  u32 below = 0;
#pragma unroll
  for (u32 i = 0; i < kFindWindow; ++i)
    below += (lo + i < hi && (T::kw(w[i]) & T::kLow) < target) ? 1u : 0u;
  return lo + below;
}

// First row whose key is >= x.
template <class T>
__device__ __forceinline__ u32 run_lower_bound(const RunView<T> &r,
                                               const RunMeta &m,
                                               typename T::K x) {
  u32 lo, hi;
  if (!dir_window(r, m, x, lo, hi)) return lo;
  return window_lower_bound<T>(r.rows, lo, hi, x & T::kLow);
}

// First row whose key is > x.
template <class T>
__device__ __forceinline__ u32 run_upper_bound(const RunView<T> &r,
                                               const RunMeta &m,
                                               typename T::K x) {
  return x == T::kAllOnes ? m.count : run_lower_bound(r, m, x + 1);
}

// Point search; returns the row position or 0xffffffff (row in `row`).
// Keys are unique inside a run, so a binary search that meets the key
// stops there; once the directory window is down to kFindWindow rows, its
// loads are issued together (one memory round trip instead of
// log2(window) dependent ones).

template <class T>
__device__ __forceinline__ u32 run_find(const RunView<T> &r, const RunMeta &m,
                                        typename T::K key,
                                        typename T::Row &row) {
  u32 lo, hi;
  if (!dir_window(r, m, key, lo, hi)) return 0xffffffffu;
  const typename T::K target = key & T::kLow;
  while (hi - lo > kFindWindow) {
    const u32 mid = (lo + hi) >> 1;
    const typename T::Row w = r.rows[mid];
    const typename T::K km = T::kw(w) & T::kLow;
    if (km == target) {
      row = w;
      return mid;
    }
    if (km < target) lo = mid + 1;
    else hi = mid;
  }
  typename T::Row w[kFindWindow];
#pragma unroll
  for (u32 i = 0; i < kFindWindow; ++i)
    if (lo + i < hi) w[i] = r.rows[lo + i];
  u32 at = 0xffffffffu;
#pragma unroll
  for (u32 i = 0; i < kFindWindow; ++i) {
    if (lo + i < hi && (T::kw(w[i]) & T::kLow) == target) {
      at = lo + i;
      row = w[i];
    }
  }
  return at;
}

// ------------------------------------------------------------ batch runs
constexpr int kFinThreads = 512;
constexpr int kFinItems = 8;
constexpr int kFinTile = kFinThreads * kFinItems;  // 4096
constexpr int kFinWaves = kFinThreads / kWave;

enum FinalizeMode : int {
  kModeInsert = 0,
  kModeErase = 1,
  kModeMixed = 2,
};

// Turns a stably sorted batch (keys sk, input positions sp) into a run:
// keep the last occurrence of each key (the newest), gather its value and
// tombstone flag, encode, and compact with a single-pass chained scan.
// Items are striped (item j of a thread is row base + j*512 + tid), so every
// load and store of a row j is one coalesced access of the block; ballots
// give the survivors' ranks.  The run header is written without atomics:
// the tile holding the last key writes the count, the tile where keys
// first reach the top bit (or the last tile) writes the split, and tiles
// with tombstones set the tombstone flag.  The radix directory (dir_bits
// bits) is written here too: sorted position i owns the directory entries
// of the buckets in (bucket(key[i-1]), bucket(key[i])] and writes them the
// number of survivors before position i (the output row of its key).  sp: the
// sorted updates' positions or, where values is null, the values themselves
// (inserts of 32-bit values).
template <class T>
__global__ __launch_bounds__(kFinThreads) void finalize_batch_kernel(
    const typename T::K *__restrict__ sk, const u32 *__restrict__ sp, u32 n,
    const typename T::V *__restrict__ values,
    const u8 *__restrict__ erase_flags, int mode,
    typename T::Row *__restrict__ out, RunMeta *meta, u32 *__restrict__ dir,
    u32 dir_bits, u64 *status, u32 *ticket, rs::Gate gate) {
  using K = typename T::K;
  using V = typename T::V;
  if (gate.closed()) return;
  __shared__ u32 s_tile;
  __shared__ u32 s_off[kFinItems][kFinWaves];
  __shared__ u32 s_total;
  __shared__ u64 s_base;
  __shared__ u32 s_low, s_tomb;
  const u32 lane = lane_id();
  const u32 wave = threadIdx.x / kWave;
  if (threadIdx.x == 0) {
    s_tile = atomicAdd(ticket, 1u);
    s_low = 0;
    s_tomb = 0;
  }
  __syncthreads();
  const u32 tile = s_tile;
  const u64 base = u64(tile) * kFinTile;
  K key[kFinItems];
  u64 mask[kFinItems];
#pragma unroll
  for (int j = 0; j < kFinItems; ++j) {
    const u64 i = base + u64(j) * kFinThreads + threadIdx.x;
    bool keep = false;
    key[j] = 0;
    if (i < n) {
      key[j] = sk[i];
      keep = (i + 1 == n) || sk[i + 1] != key[j];
    }
    mask[j] = ballot(keep);
    if (lane == 0) s_off[j][wave] = popc64(mask[j]);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    u32 run = 0;
    for (int j = 0; j < kFinItems; ++j)
      for (int w = 0; w < kFinWaves; ++w) {
        const u32 c = s_off[j][w];
        s_off[j][w] = run;
        run += c;
      }
    s_total = run;
  }
  __syncthreads();
  const u32 tile_total = s_total;
  if (threadIdx.x < kWave) {
    const u64 ex = wave_lookback(status, tile, tile_total);
    if (threadIdx.x == 0) s_base = ex;
  }
  __syncthreads();
  const u64 out_base = s_base;
  u32 low = 0, tombs = 0;
  // (a surviving row's loads; all are issued before the first is waited for)
  V val[kFinItems];
  u32 tomb = 0;
#pragma unroll
  for (int j = 0; j < kFinItems; ++j) {
    const bool kept = (mask[j] >> lane) & 1ull;
    val[j] = kept ? V(sp[base + u64(j) * kFinThreads + threadIdx.x]) : V(0);
  }
  if (mode == kModeErase) {
    tomb = ~0u;
  } else if (values) {
#pragma unroll
    for (int j = 0; j < kFinItems; ++j) {
      if (!((mask[j] >> lane) & 1ull)) continue;
      const u32 p = static_cast<u32>(val[j]);
      if (mode == kModeMixed && erase_flags[p] != 0) tomb |= 1u << j;
      val[j] = values[p];
    }
  }
#pragma unroll
  for (int j = 0; j < kFinItems; ++j) {
    if (!((mask[j] >> lane) & 1ull)) continue;
    const u64 o = out_base + s_off[j][wave] + popc64(mask[j] & lanemask_lt());
    const bool dead = (tomb >> j) & 1u;
    out[o] = T::make((key[j] & T::kLow) | (dead ? T::kTomb : K(0)),
                     dead ? V(0) : val[j]);
    low += key[j] < T::kTomb;
    tombs += dead;
  }
  // directory entries inside the bucket window
  const u32 shift = T::kBits - dir_bits;
#pragma unroll
  for (int j = 0; j < kFinItems; ++j) {
    const u64 i = base + u64(j) * kFinThreads + threadIdx.x;
    if (i >= n) continue;
    const u32 bk = static_cast<u32>(key[j] >> shift);
    const u32 before = static_cast<u32>(out_base + s_off[j][wave] +
                                        popc64(mask[j] & lanemask_lt()));
    if (i == 0) {
      meta->lo_bucket = bk;
      dir[bk] = 0;
    } else {
      for (u32 b = static_cast<u32>(sk[i - 1] >> shift) + 1; b <= bk; ++b)
        dir[b] = before;
    }
    if (i + 1 == n) {
      meta->hi_bucket = bk;
      meta->dir_bits = dir_bits;
      dir[bk + 1] = static_cast<u32>(out_base + tile_total);
    }
  }
  low = wave_sum_u32(low);
  tombs = wave_sum_u32(tombs);
  if (lane == 0) {
    if (low) atomicAdd(&s_low, low);
    if (tombs) atomicAdd(&s_tomb, tombs);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const u64 in_end = base + kFinTile < n ? base + kFinTile : n;
    const bool last_tile = in_end == n;
    // keys before this tile are all below the top bit and some key of the
    // tile (its last) reaches it, or no key does at all
    const bool transition = (base == 0 || sk[base - 1] < T::kTomb) &&
                            (sk[in_end - 1] >= T::kTomb || last_tile);
    if (last_tile) meta->count = static_cast<u32>(out_base + tile_total);
    if (transition) meta->split = static_cast<u32>(out_base + s_low);
    if (s_tomb) meta->tombs = 1;
  }
}

// ------------------------------------------------ small batches, one launch
// A batch of at most T::kSmallTile keys becomes a run in ONE workgroup: an
// LDS LSD radix sort (the same wave64 ballot multisplit as the onesweep
// passes, with the whole batch as one tile), newest-wins dedupe, value
// gather, encode, and the radix directory.  Replaces nine launches for the
// small arrivals of a serving stream.
//
// One workgroup on an empty chip: its time is its chain of barriers and memory
// round trips.  So a short batch is spread over all eight waves (by itself 700
// keys filled two, with eight items in a row each), digits that do not vary are
// skipped, and keys, values and flags are all read before the sort.  700
// updates: 20.7 us before, 11.7 so.
constexpr int kSmallThreads = 512;
constexpr int kSmallWaves = kSmallThreads / kWave;

// Where a fused admission reads its batch: entry i's key, value and erase
// flag.  ArrayBatch reads three arrays; the serving engine's step kernels
// read the step's request buffers through its piece table instead.
template <class T>
struct ArrayBatch {
  const typename T::K *keys;
  const typename T::V *values;
  const u8 *erase_flags;
  __device__ __forceinline__ typename T::K key(u32 i) const { return keys[i]; }
  __device__ __forceinline__ typename T::V value(u32 i) const {
    return values[i];
  }
  __device__ __forceinline__ bool erased(u32 i) const {
    return erase_flags[i] != 0;
  }
};

// (the body of small_batch_run_kernel; also run by the serving engine's
// step kernels, which read the arguments from a step descriptor)
template <class T, class Batch>
__device__ __forceinline__ void small_batch_run(
    const Batch &batch, u32 n, int mode, typename T::Row *__restrict__ out,
    RunMeta *meta, u32 *__restrict__ dir, u32 max_bits, u32 rows_log) {
  using K = typename T::K;
  using V = typename T::V;
  constexpr int kTile = T::kSmallTile;
  constexpr int kItems = kTile / kSmallThreads;
  constexpr int kPasses = T::kBits / 8;
  // keys (2 x tile), 16-bit positions (2 x tile), per-wave digit counters:
  // 57 KB for 32-bit keys (4096 keys), 48 KB for 64-bit keys (2048)
  __shared__ K s_k0[kTile];
  __shared__ K s_k1[kTile];
  __shared__ unsigned short s_p0[kTile];
  __shared__ unsigned short s_p1[kTile];
  __shared__ u32 s_hist[kSmallWaves * 256];
  __shared__ u32 s_scan[kSmallWaves];
  __shared__ u32 s_misc[8];
  __shared__ K s_vary;  // the bits that vary among the keys
  constexpr u32 kSmallErased = 0x8000u;
  static_assert(kTile <= 0x8000, "positions below the erase flag");
  const u32 tid = threadIdx.x;
  const u32 lane = lane_id();
  const u32 wave = tid / kWave;
  // items per thread: a short batch is spread over all waves
  const u32 ipt = __builtin_amdgcn_readfirstlane((n + kSmallThreads - 1) /
                                                 kSmallThreads);
  const u32 wave_base = wave * (kWave * ipt);

  // everything of the batch is read here, at once: keys, erase flags (in the
  // positions' top bit) and values (item j of thread t: update j * 512 + t)
  V value[kItems];
  {
    K key[kItems];
    u32 erased = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const u32 i = j * kSmallThreads + tid;
      key[j] = 0;
      value[j] = 0;
      if (i < n) {
        key[j] = batch.key(i);
        // (an erase has no value to read)
        if (mode == kModeErase || (mode == kModeMixed && batch.erased(i)))
          erased |= 1u << j;
        else
          value[j] = batch.value(i);
      }
    }
    if (tid == 0) {
      s_k0[0] = key[0];
      s_vary = 0;
    }
    __syncthreads();
    const K first = s_k0[0];
    K vary = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const u32 i = j * kSmallThreads + tid;
      if (i < n) {
        vary |= key[j] ^ first;
        if (i) s_k0[i] = key[j];
        s_p0[i] = static_cast<unsigned short>(
            i | ((erased >> j) & 1u ? kSmallErased : 0u));
      }
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) vary |= __shfl_xor(vary, o, kWave);
    if (lane == 0 && vary) atomicOr(&s_vary, vary);
    __syncthreads();
  }
  const K vary = s_vary;
  K *src_k = s_k0, *dst_k = s_k1;
  unsigned short *src_p = s_p0, *dst_p = s_p1;
  u32 *my_hist = s_hist + wave * 256;
  for (int pass = 0; pass < kPasses; ++pass) {
    const u32 shift = 8u * pass;
    if (((vary >> shift) & K(0xff)) == 0) continue;  // (uniform)
    for (u32 i = lane; i < 256; i += kWave) lds_store(&my_hist[i], 0);
    __builtin_amdgcn_wave_barrier();
    K key[kItems];
    u32 pos[kItems], rank[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if (static_cast<u32>(j) >= ipt) continue;
      const u32 idx = wave_base + j * kWave + lane;
      const bool valid = idx < n;
      key[j] = valid ? src_k[idx] : T::kAllOnes;
      pos[j] = valid ? src_p[idx] : 0u;
      const u32 d = static_cast<u32>(key[j] >> shift) & 0xffu;
      rank[j] = count_peers(&my_hist[d], digit_peers(d, ballot(valid)), valid);
    }
    __syncthreads();
    // a digit per thread (threads 0..255): its counts in the waves, its start
    u32 c[kSmallWaves], total = 0;
    if (tid < 256) {
#pragma unroll
      for (int w = 0; w < kSmallWaves; ++w) {
        c[w] = s_hist[w * 256 + tid];
        total += c[w];
      }
    }
    const u32 inclusive = wave_inclusive_scan(total);
    if (tid < 256 && lane == kWave - 1) s_scan[wave] = inclusive;
    __syncthreads();
    if (tid < 256) {
      u32 start = inclusive - total;
      for (u32 w = 0; w < wave; ++w) start += s_scan[w];
#pragma unroll
      for (int w = 0; w < kSmallWaves; ++w) {
        s_hist[w * 256 + tid] = start;
        start += c[w];
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if (static_cast<u32>(j) >= ipt) continue;
      if (wave_base + j * kWave + lane < n) {
        const u32 d = static_cast<u32>(key[j] >> shift) & 0xffu;
        const u32 lp = my_hist[d] + rank[j];
        dst_k[lp] = key[j];
        dst_p[lp] = static_cast<unsigned short>(pos[j]);
      }
    }
    __syncthreads();
    K *tk = src_k;
    unsigned short *tp = src_p;
    src_k = dst_k;
    src_p = dst_p;
    dst_k = tk;
    dst_p = tp;
  }
  // sorted (key, position) in src_*; keep the last occurrence of each key.
  // Survivor ranks: ballots per (item row j, wave), scanned by wave 0.  The
  // values go to the array that the sort has left, by position.
  u32 *s_off = s_hist;  // reuse: kItems * kSmallWaves words
  static_assert(kItems * kSmallWaves <= kWave, "scanned by a wave");
  static_assert(sizeof(V) == sizeof(K), "values in the keys' array");
  V *s_val = reinterpret_cast<V *>(dst_k);
  u64 mask[kItems];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const u32 i = j * kSmallThreads + tid;
    const bool keep = i < n && (i + 1 == n || src_k[i + 1] != src_k[i]);
    mask[j] = ballot(keep);
    if (lane == 0) s_off[j * kSmallWaves + wave] = popc64(mask[j]);
    if (i < n) s_val[i] = value[j];
  }
  __syncthreads();
  if (wave == 0) {
    const u32 v = lane < kItems * kSmallWaves ? s_off[lane] : 0u;
    const u32 inc = wave_inclusive_scan(v);
    if (lane < kItems * kSmallWaves) s_off[lane] = inc - v;
    if (lane == kWave - 1) s_misc[0] = inc;  // count
    if (lane == 0) {
      s_misc[1] = 0;  // split
      s_misc[2] = 0;  // tombs
    }
  }
  __syncthreads();
  const u32 count = s_misc[0];
  u32 low = 0, tombs = 0;
  K kept[kItems];
  u32 at[kItems];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    at[j] = ~0u;
    if (!((mask[j] >> lane) & 1ull)) continue;
    const u32 i = j * kSmallThreads + tid;
    const u32 o = s_off[j * kSmallWaves + wave] +
                  popc64(mask[j] & lanemask_lt());
    const K k = src_k[i];
    const u32 p = src_p[i];
    const bool tomb = (p & kSmallErased) != 0;
    out[o] = T::make((k & T::kLow) | (tomb ? T::kTomb : K(0)),
                     tomb ? V(0) : s_val[p & (kSmallErased - 1)]);
    kept[j] = k;
    at[j] = o;
    low += k < T::kTomb;
    tombs += tomb;
  }
  __syncthreads();  // the values are read
  // decoded output keys go to dst_k for the directory pass
#pragma unroll
  for (int j = 0; j < kItems; ++j)
    if (at[j] != ~0u) dst_k[at[j]] = kept[j];
  low = wave_sum_u32(low);
  tombs = wave_sum_u32(tombs);
  if (lane == 0) {
    if (low) atomicAdd(&s_misc[1], low);
    if (tombs) atomicAdd(&s_misc[2], tombs);
  }
  __syncthreads();
  const u32 b = dir_bits_for(count, max_bits, rows_log);
  const u32 shift = T::kBits - b;
  if (tid == 0) {
    // count >= 1 (n >= 1)
    const u32 lo_b = static_cast<u32>(dst_k[0] >> shift);
    const u32 hi_b = static_cast<u32>(dst_k[count - 1] >> shift);
    meta->count = count;
    meta->split = s_misc[1];
    meta->tombs = s_misc[2];
    meta->dir_bits = b;
    meta->lo_bucket = lo_b;
    meta->hi_bucket = hi_b;
    dir[lo_b] = 0;
    dir[hi_b + 1] = count;
  }
  for (u32 t = 1 + tid; t < count; t += kSmallThreads) {
    const u32 bucket = static_cast<u32>(dst_k[t] >> shift);
    for (u32 j = static_cast<u32>(dst_k[t - 1] >> shift) + 1; j <= bucket;
         ++j)
      dir[j] = t;
  }
}

template <class T>
__global__ __launch_bounds__(kSmallThreads) void small_batch_run_kernel(
    const typename T::K *__restrict__ keys, u32 n,
    const typename T::V *__restrict__ values,
    const u8 *__restrict__ erase_flags, int mode,
    typename T::Row *__restrict__ out, RunMeta *meta, u32 *__restrict__ dir,
    u32 max_bits, u32 rows_log) {
  small_batch_run<T>(ArrayBatch<T>{keys, values, erase_flags}, n, mode, out,
                     meta, dir, max_bits, rows_log);
}

// Builds the radix directory of a run from its final count/split (one
// thread per row, grid-stride).
template <class T>
__global__ void build_directory_kernel(const typename T::Row *__restrict__ rows,
                                       RunMeta *meta, u32 *__restrict__ dir,
                                       u32 max_bits, u32 rows_log) {
  const u32 count = meta->count;
  const u32 split = meta->split;
  const u32 b = dir_bits_for(count, max_bits, rows_log);
  const u32 shift = T::kBits - b;
  const u64 gid = u64(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid == 0) {
    meta->dir_bits = b;
    if (count == 0) {
      meta->lo_bucket = 1;
      meta->hi_bucket = 0;
    } else {
      const u32 lo_b = static_cast<u32>(
          decode_key<T>(T::kw(rows[0]), 0, split) >> shift);
      const u32 hi_b = static_cast<u32>(
          decode_key<T>(T::kw(rows[count - 1]), count - 1, split) >> shift);
      meta->lo_bucket = lo_b;
      meta->hi_bucket = hi_b;
      dir[lo_b] = 0;
      dir[hi_b + 1] = count;
    }
  }
  const u64 stride = u64(gridDim.x) * blockDim.x;
  for (u64 t = gid + 1; t < count; t += stride) {
    const u32 pos = static_cast<u32>(t);
    const u32 bucket = static_cast<u32>(
        decode_key<T>(T::kw(rows[pos]), pos, split) >> shift);
    for (u32 j = static_cast<u32>(
                     decode_key<T>(T::kw(rows[pos - 1]), pos - 1, split) >>
                     shift) +
                 1;
         j <= bucket; ++j)
      dir[j] = pos;
  }
}

// --------------------------------------------------------------- merging
// merge workgroups: 256 or 512 threads (tile = threads x items per thread)

// LDS slot of element i of an array of E-byte elements, XOR-swizzled: the
// bits of i that select its bank inside a 128-byte line of the 32 banks are
// XORed with the line number, a bijection inside every line.  Lanes whose
// accesses start 4, 8 or 16 elements apart (a thread's merge window, its
// staged output rows) then spread over the banks as consecutive lanes do,
// instead of meeting in a few.  lds_lines rounds an array up to whole lines.
template <int E>
__host__ __device__ constexpr u32 lds_swz(u32 i) {
  constexpr u32 per = 128 / E;
  constexpr u32 gran = E >= 4 ? 1 : 4 / E;
  return i ^ ((((i / per) & 31u) * gran) & (per - 1));
}
template <int E>
__host__ __device__ constexpr u32 lds_lines(u32 n) {
  constexpr u32 per = 128 / E;
  return (n + per - 1) / per * per;
}

template <class T>
struct MergeSide {
  const typename T::Row *rows;
  const RunMeta *meta;
};

template <class T>
__device__ __forceinline__ typename T::K side_key(const MergeSide<T> &s,
                                                  u32 pos, u32 split) {
  return decode_key<T>(T::kw(s.rows[pos]), pos, split);
}

// Number of A elements among the first `diag` merged elements, where A (the
// newer run) precedes B on equal keys.
template <class T>
__device__ __forceinline__ u32 merge_path(const MergeSide<T> &a, u32 ca,
                                          u32 sa, const MergeSide<T> &b,
                                          u32 cb, u32 sb, u64 diag) {
  u64 lo = diag > cb ? diag - cb : 0;
  u64 hi = diag < ca ? diag : ca;
  while (lo < hi) {
    const u64 mid = (lo + hi) >> 1;
    const auto ka = side_key(a, static_cast<u32>(mid), sa);
    const auto kb = side_key(b, static_cast<u32>(diag - mid - 1), sb);
    if (ka <= kb) lo = mid + 1;
    else hi = mid;
  }
  return static_cast<u32>(lo);
}

// Tile split points of the merge, one wave per split point: a 64-ary
// search (every lane tests one candidate, a ballot keeps the interval that
// holds the answer), so a split over 2^26 rows costs 5 rounds of loads
// instead of 26 dependent ones.  Also clears the merge's chained-scan state
// and the output run's header (one launch instead of three).
template <class T>
__global__ void merge_partition_kernel(MergeSide<T> a, MergeSide<T> b,
                                       u32 tiles, u32 tile_rows,
                                       u32 *__restrict__ parts, u64 *status,
                                       u32 *ticket, RunMeta *out_meta,
                                       u32 dir_bits) {
  const u32 lane = lane_id();
  const u64 t = (u64(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  if (t > tiles) return;
  if (lane == 0 && t < tiles) status[t] = 0;
  if (t == 0 && lane == 0) {
    *ticket = 0;
    out_meta->count = 0;
    out_meta->split = 0;
    out_meta->dir_bits = dir_bits;
    out_meta->tombs = 0;
    out_meta->lo_bucket = 1;  // empty until the first and last input
    out_meta->hi_bucket = 0;  // element write their buckets
  }
  const u32 ca = a.meta->count, cb = b.meta->count;
  const u32 sa = a.meta->split, sb = b.meta->split;
  const u64 total = u64(ca) + cb;
  u64 diag = t * tile_rows;
  if (diag > total) diag = total;
  // answer = first m in [lo, hi) with A[m] > B[diag - m - 1], else hi
  u64 lo = diag > cb ? diag - cb : 0;
  u64 hi = diag < ca ? diag : ca;
  while (hi > lo) {
    const u64 span = hi - lo;
    const u64 m = span <= kWave ? lo + lane : lo + ((span * lane) >> 6);
    bool p = false;  // lanes past the interval vote "false"
    if (m < hi)
      p = side_key(a, static_cast<u32>(m), sa) <=
          side_key(b, static_cast<u32>(diag - m - 1), sb);
    const u64 vote = ballot(p);
    const u32 c = popc64(vote);  // the true candidates form a prefix
    if (span <= kWave) {
      lo += c;
      break;
    }
    const u64 m_prev = lo + ((span * (c ? c - 1 : 0)) >> 6);
    const u64 m_next = lo + ((span * c) >> 6);
    if (c == 0) {
      hi = lo;  // A[lo] > B[...]: the answer is lo
    } else {
      lo = m_prev + 1;
      if (c < kWave) hi = m_next;
    }
  }
  if (lane == 0) parts[t] = static_cast<u32>(lo);
}

// Merges run A (newer) with run B (older) into `out`: on equal keys the A
// row survives, and tombstones are dropped when `drop_tombstones` (the
// output becomes the oldest run, GPULSMOpt.cuh:3175-3179).  A tile is
// 256 * kMergeItems output diagonals.  The output's radix directory
// (dir_bits bits) is written here: every input element, kept or dropped,
// owns the entries of the buckets in (bucket(previous input key),
// bucket(its key)] in merged order and writes them the number of survivors
// before it, which is the output row of the first key >= those bounds.
template <class T, int kMergeItems, int kMergeThreads>
__global__ __launch_bounds__(kMergeThreads) void merge_kernel(
    MergeSide<T> a, MergeSide<T> b, const u32 *__restrict__ parts,
    typename T::Row *__restrict__ out, RunMeta *out_meta,
    u32 *__restrict__ dir, u32 dir_bits, int drop_tombstones, u64 *status,
    u32 *ticket) {
  using K = typename T::K;
  using V = typename T::V;
  using Row = typename T::Row;
  constexpr int kMergeTile = kMergeThreads * kMergeItems;
  // survivors are staged as rows over the key array, then the value array
  constexpr u32 kStageHalf = (kMergeTile + 2) / 2;
  static_assert(sizeof(Row) == 2 * sizeof(K) && sizeof(K) == sizeof(V),
                "row = key word + value");
  // LDS slots are swizzled (lds_swz) so that the lanes of a wave, whose
  // merge windows and staged outputs start kMergeItems slots apart, spread
  // over the banks
  constexpr u32 kSlots = lds_lines<sizeof(K)>(kMergeTile + 2);
  constexpr u32 kStageSlots =
      lds_lines<sizeof(Row)>(kStageHalf) * sizeof(Row) / sizeof(K);
  constexpr u32 kKeySlots = kSlots > kStageSlots ? kSlots : kStageSlots;
  auto key_slot = [](u32 i) { return lds_swz<sizeof(K)>(i); };
  auto tomb_slot = [](u32 i) { return lds_swz<1>(i); };
  auto row_slot = [](u32 i) { return lds_swz<sizeof(Row)>(i); };
  __shared__ u32 s_tile;
  // inputs: decoded key, value, tombstone flag
  __shared__ __align__(16) K s_key[kKeySlots];
  __shared__ __align__(16) V s_val[kKeySlots];
  __shared__ u8 s_tomb[lds_lines<1>(kMergeTile + 2)];
  __shared__ u32 s_scan[kMergeThreads / kWave + 1];
  __shared__ u64 s_base;
  __shared__ u32 s_low, s_tombs;
  __shared__ K s_prev_b;  // B[j0 - 1]: with A[i0 - 1], the row before the tile

  if (threadIdx.x == 0) {
    s_tile = atomicAdd(ticket, 1u);
    s_low = 0;
    s_tombs = 0;
  }
  __syncthreads();
  const u32 tile = s_tile;
  const u32 ca = a.meta->count, cb = b.meta->count;
  const u32 sa = a.meta->split, sb = b.meta->split;
  const u64 total = u64(ca) + cb;
  const u64 d0 = u64(tile) * kMergeTile;
  if (d0 >= total) return;  // every later ticket is empty too (an empty
                            // output keeps the empty bucket window)
  const u64 d1 = d0 + kMergeTile < total ? d0 + kMergeTile : total;
  const u32 i0 = parts[tile], i1 = parts[tile + 1];
  const u32 j0 = static_cast<u32>(d0 - i0), j1 = static_cast<u32>(d1 - i1);
  const u32 na = i1 - i0, nb = j1 - j0;

  // LDS layout: [0] = A[i0-1] (previous A row, for the equal-key test),
  // [1, na] = A[i0, i1), [na+1, na+nb] = B[j0, j1).  Slot t of the
  // na + 1 + nb <= kMergeTile + 1 slots is loaded by thread t % 256; every
  // load of a thread is issued before the first one is used.
  constexpr int kLoads = kMergeItems + 1;
  const u32 slots = na + 1 + nb;
  Row rr[kLoads];
#pragma unroll
  for (int r = 0; r < kLoads; ++r) {
    const u32 t = threadIdx.x + r * kMergeThreads;
    if (t < slots) {
      if (t > na) rr[r] = b.rows[j0 + (t - na - 1)];
      else if (t > 0 || i0 > 0) rr[r] = a.rows[i0 + t - 1];
    }
  }
  Row prev_b_row{};
  const bool load_prev_b = threadIdx.x == kMergeThreads - 1 && j0 > 0;
  if (load_prev_b) prev_b_row = b.rows[j0 - 1];
#pragma unroll
  for (int r = 0; r < kLoads; ++r) {
    const u32 t = threadIdx.x + r * kMergeThreads;
    if (t < slots) {
      if (t == 0 && i0 == 0) {
        s_key[0] = 0;
        s_tomb[0] = 2;  // "no previous row"
      } else {
        const bool from_a = t <= na;
        const u32 pos = from_a ? i0 + t - 1 : j0 + (t - na - 1);
        s_key[key_slot(t)] =
            decode_key<T>(T::kw(rr[r]), pos, from_a ? sa : sb);
        s_tomb[tomb_slot(t)] =
            static_cast<u8>(T::kw(rr[r]) >> (T::kBits - 1));
        s_val[key_slot(t)] = T::val(rr[r]);
      }
    }
  }
  if (threadIdx.x == kMergeThreads - 1)
    s_prev_b = load_prev_b ? decode_key<T>(T::kw(prev_b_row), j0 - 1, sb)
                           : K(0);
  __syncthreads();
  // Header fields without atomics: the tile reaching the end writes the
  // count; the first tile whose inputs reach the top key bit (or the last
  // tile) writes the split, as every row before it is below the top bit and
  // every row after it is not; tiles with surviving tombstones set the flag.
  const bool last_tile = d1 == total;
  bool transition = false;
  {
    const bool before_low = (i0 == 0 || s_key[0] < T::kTomb) &&
                            (j0 == 0 || s_prev_b < T::kTomb);
    const bool tile_high = (na && s_key[key_slot(na)] >= T::kTomb) ||
                           (nb && s_key[key_slot(na + nb)] >= T::kTomb);
    transition = before_low && (tile_high || last_tile);
  }

  // Per-thread merge path inside the tile.
  const u32 tile_len = na + nb;
  const u32 dk = threadIdx.x * kMergeItems;
  u32 ia = 0, ib = 0;
  if (dk < tile_len) {
    u32 lo = dk > nb ? dk - nb : 0;
    u32 hi = dk < na ? dk : na;
    while (lo < hi) {
      const u32 mid = (lo + hi) >> 1;
      if (s_key[key_slot(1 + mid)] <=
          s_key[key_slot(na + 1 + (dk - mid - 1))])
        lo = mid + 1;
      else hi = mid;
    }
    ia = lo;
    ib = dk - lo;
  }
  // the input element before this thread's first one, in merged order
  bool has_prev = false;
  K prev = 0;
  if (dk < tile_len) {
    if (ia > 0 || i0 > 0) {
      has_prev = true;
      prev = s_key[key_slot(ia)];  // slot ia: A[ia - 1] (A[i0 - 1] at 0)
    }
    if (ib > 0 || j0 > 0) {
      const K kb = ib > 0 ? s_key[key_slot(na + ib)] : s_prev_b;
      prev = has_prev && prev > kb ? prev : kb;
      has_prev = true;
    }
  }
  K ok[kMergeItems];
  V ov[kMergeItems];
  u8 ot[kMergeItems];
  u32 osrc[kMergeItems];  // LDS slot of each merged element
  bool okeep[kMergeItems];
  u32 kept = 0;
  const u32 steps =
      dk < tile_len ? (tile_len - dk < kMergeItems ? tile_len - dk
                                                   : u32(kMergeItems))
                    : 0u;
  // Serial merge.  Registers carry the next key of each side and the last
  // A key taken (a B row equal to it is shadowed by the newer A row), so
  // the only LDS read on the serial path is the next key of the side that
  // advanced; values and tombstone flags are read afterwards, all at once.
  {
    bool a_left = ia < na, b_left = ib < nb;
    K ka = (steps && a_left) ? s_key[key_slot(1 + ia)] : K(0);
    K kb = (steps && b_left) ? s_key[key_slot(na + 1 + ib)] : K(0);
    // LDS slot ia holds A[ia - 1] (A[i0 - 1] at 0, flag 2 when none)
    bool have_last_a = steps && s_tomb[tomb_slot(ia)] != 2;
    K last_a = steps ? s_key[key_slot(ia)] : K(0);
#pragma unroll
    for (int s = 0; s < kMergeItems; ++s) {
      okeep[s] = false;
      ok[s] = 0;
      osrc[s] = 0;
      if (static_cast<u32>(s) < steps) {
        const bool take_a = a_left && (!b_left || ka <= kb);
        const K k = take_a ? ka : kb;
        ok[s] = k;
        osrc[s] = take_a ? 1 + ia : na + 1 + ib;
        okeep[s] = take_a || !(have_last_a && last_a == k);
        if (take_a) {
          last_a = k;
          have_last_a = true;
        }
        ia += take_a;
        ib += !take_a;
        a_left = ia < na;
        b_left = ib < nb;
        const bool more = take_a ? a_left : b_left;
        const K next =
            more ? s_key[key_slot(take_a ? 1 + ia : na + 1 + ib)] : K(0);
        if (take_a) ka = next;
        else kb = next;
      }
    }
  }
#pragma unroll
  for (int s = 0; s < kMergeItems; ++s) {
    ov[s] = 0;
    ot[s] = 0;
    if (static_cast<u32>(s) < steps) {
      ot[s] = s_tomb[tomb_slot(osrc[s])];
      ov[s] = s_val[key_slot(osrc[s])];
    }
  }
#pragma unroll
  for (int s = 0; s < kMergeItems; ++s) {
    if (okeep[s] && ot[s] && drop_tombstones) okeep[s] = false;
    kept += okeep[s];
  }
  const u32 local = block_exclusive_scan<kMergeThreads>(kept, s_scan);
  const u32 tile_total = s_scan[kMergeThreads / kWave];
  // Wave 0 waits on the look-back while the other waves stage their
  // survivors at tile-local positions (the scan's barriers ordered every
  // LDS input read before these writes).
  if (threadIdx.x < kWave) {
    const u64 ex = wave_lookback(status, tile, tile_total);
    if (threadIdx.x == 0) s_base = ex;
  }
  Row *stage_lo = reinterpret_cast<Row *>(s_key);
  Row *stage_hi = reinterpret_cast<Row *>(s_val);
  u32 low = 0, tombs = 0, at = local;
#pragma unroll
  for (int s = 0; s < kMergeItems; ++s) {
    if (okeep[s]) {
      const Row r =
          T::make((ok[s] & T::kLow) | (ot[s] ? T::kTomb : K(0)), ov[s]);
      if (at < kStageHalf) stage_lo[row_slot(at)] = r;
      else stage_hi[row_slot(at - kStageHalf)] = r;
      ++at;
      low += ok[s] < T::kTomb;
      tombs += ot[s];
    }
  }
  __syncthreads();
  const u64 obase = s_base;
  for (u32 t = threadIdx.x; t < tile_total; t += kMergeThreads)
    out[obase + t] = t < kStageHalf ? stage_lo[row_slot(t)]
                                    : stage_hi[row_slot(t - kStageHalf)];
  // directory entries inside the bucket window (first to last input key)
  {
    const u32 shift = T::kBits - dir_bits;
    u32 pbk = static_cast<u32>(prev >> shift);
    u32 before = static_cast<u32>(obase) + local;
#pragma unroll
    for (int s = 0; s < kMergeItems; ++s) {
      if (static_cast<u32>(s) < steps) {
        const u32 bk = static_cast<u32>(ok[s] >> shift);
        if (s == 0 && !has_prev) {  // the first input element of the merge
          out_meta->lo_bucket = bk;
          dir[bk] = 0;
        } else {
          for (u32 j = pbk + 1; j <= bk; ++j) dir[j] = before;
        }
        pbk = bk;
        before += okeep[s];
      }
    }
    if (last_tile && steps && dk + steps == tile_len) {
      // the last input element closes the window at the row count
      out_meta->hi_bucket = pbk;
      dir[pbk + 1] = static_cast<u32>(obase + tile_total);
    }
  }
  low = wave_sum_u32(low);
  tombs = wave_sum_u32(tombs);
  if (lane_id() == 0) {
    if (low) atomicAdd(&s_low, low);
    if (tombs) atomicAdd(&s_tombs, tombs);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (last_tile) out_meta->count = static_cast<u32>(obase + tile_total);
    if (transition) out_meta->split = static_cast<u32>(obase + s_low);
    if (s_tombs) out_meta->tombs = 1;
  }
}

// --------------------------------------------------------------- queries
// Query kernels read their inputs and write their results through an IO
// policy: PlainLookup / PlainRange over contiguous arrays (the C ABI), or
// the serving engine's piece tables (one launch answers every request of a
// step straight from and into the requests' own buffers).

// A miss writes all-ones (0xFFFFFFFF for 32-bit values) without a found
// array, value 0 + found 0 with one (GPULSMOpt.cuh:4714-4806).
template <class T>
struct PlainLookup {
  const typename T::K *q;
  typename T::V *out;
  u8 *found;
  // IO policies may copy a table they search per query into LDS:
  // stage(lds) returns the policy to use after the block's next barrier
  static constexpr u32 kStageBytes = 0;
  __device__ __forceinline__ PlainLookup stage(void *) const { return *this; }
  struct Slot {
    u64 i;
  };
  __device__ __forceinline__ typename T::K load(u64 i, Slot &s) const {
    s.i = i;
    return q[i];
  }
  __device__ __forceinline__ void put(const Slot &s, bool live,
                                      typename T::V value) const {
    if (found) {
      out[s.i] = live ? value : typename T::V(0);
      found[s.i] = live ? 1 : 0;
    } else {
      out[s.i] = live ? value : T::kAllOnes;
    }
  }
};

// Newest visible version of `key`: live + value, or not live.
template <class T>
__device__ __forceinline__ bool lookup_one(const RunSet<T> &runs,
                                           typename T::K key,
                                           typename T::V &value) {
  for (u32 r = 0; r < runs.count; ++r) {
    const RunView<T> &rv = runs.run[r];
    typename T::Row row;
    const RunMeta m = *rv.meta;
    if (run_find(rv, m, key, row) != 0xffffffffu) {
      value = T::val(row);
      return !(T::kw(row) & T::kTomb);
    }
  }
  return false;
}

template <class T, class IO>
__global__ void lookup_kernel(IO io_arg, u64 n, RunSet<T> runs) {
  __shared__ __align__(16) char s_io[IO::kStageBytes ? IO::kStageBytes : 16];
  const IO io = io_arg.stage(s_io);
  __syncthreads();
  const u64 stride = u64(gridDim.x) * blockDim.x;
  for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    typename IO::Slot slot;
    const typename T::K key = io.load(i, slot);
    typename T::V value = 0;
    const bool live = lookup_one(runs, key, value);
    io.put(slot, live, value);
  }
}

// Result of a grouped lookup: value and found flag side by side, so the
// gather back to query order reads each result with one access.
template <class T>
struct alignas(2 * sizeof(typename T::V)) GroupedResult {
  typename T::V value;
  typename T::V found;
};

// Lookups over queries partitioned by their top varying key byte (qk =
// grouped keys).  Results are written in the grouped order (res_values[p],
// res_found[p]), so every store is coalesced; lookup_gather_kernel then
// brings them back to query order.  Scattering each result straight to its
// query position would dirty one cache line per query and evict the run
// rows the grouping keeps in L2.  Workgroups are dealt round-robin to the
// 8 XCDs, so block b serves the contiguous chunk (b % 8) * (G / 8) + b / 8:
// every XCD walks its own eighth of the grouped queries, i.e. its own eighth
// of the key space, and the run rows it needs stay in that XCD's L2.
// A thread carries kQ queries through each run in lock step (directory
// loads of all of them, then their row windows), so their memory round
// trips overlap; run headers are read once per workgroup into LDS.
template <class T>
__global__ __launch_bounds__(256) void lookup_grouped_kernel(
    const typename T::K *__restrict__ qk, u64 n,
    GroupedResult<T> *__restrict__ res, RunSet<T> runs) {
  using K = typename T::K;
  using V = typename T::V;
  using Row = typename T::Row;
  constexpr int kQ = 2;
  __shared__ RunMeta s_meta[kMaxRuns];
  if (threadIdx.x < runs.count) s_meta[threadIdx.x] = *runs.run[threadIdx.x].meta;
  __syncthreads();
  const u32 G = gridDim.x;  // a multiple of 8
  const u32 logical = (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u;
  const u64 chunk = (n + G - 1) / G;
  const u64 begin = u64(logical) * chunk;
  const u64 end = begin + chunk < n ? begin + chunk : n;
  for (u64 p0 = begin + threadIdx.x; p0 < end; p0 += u64(kQ) * blockDim.x) {
    K key[kQ];
    V val[kQ];
    bool open[kQ], live[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const u64 p = p0 + u64(q) * blockDim.x;
      open[q] = p < end;
      key[q] = open[q] ? qk[p] : K(0);
      live[q] = false;
      val[q] = 0;
    }
    for (u32 r = 0; r < runs.count; ++r) {
      const RunMeta m = s_meta[r];
      const RunView<T> &rv = runs.run[r];
      u32 lo[kQ], hi[kQ];
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        lo[q] = hi[q] = 0;
        if (open[q]) (void)dir_window(rv, m, key[q], lo[q], hi[q]);
      }
      bool hit[kQ];
      Row row[kQ];
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        hit[q] = false;
        // wide directory buckets (skewed keys): bisect down to the window
        const K target = key[q] & T::kLow;
        while (hi[q] - lo[q] > kFindWindow) {
          const u32 mid = (lo[q] + hi[q]) >> 1;
          const Row w = rv.rows[mid];
          const K km = T::kw(w) & T::kLow;
          if (km == target) {
            hit[q] = true;
            row[q] = w;
            lo[q] = hi[q] = mid;
          } else if (km < target) {
            lo[q] = mid + 1;
          } else {
            hi[q] = mid;
          }
        }
      }
      // the row windows: 8-byte rows are loaded in aligned pairs (one
      // 16-byte access covers two rows; row arrays carry one spare row, so
      // the pair of a window's last row stays inside the allocation)
      constexpr u32 kPair = sizeof(Row) == 8 ? 2 : 1;
      constexpr u32 kSlots = kPair == 2 ? kFindWindow + 2 : kFindWindow;
      Row w[kQ][kSlots];
      u32 first[kQ];
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        first[q] = kPair == 2 ? (lo[q] & ~1u) : lo[q];
#pragma unroll
        for (u32 i = 0; i < kSlots; i += kPair) {
          const u32 at = first[q] + i;
          if (at < hi[q]) {
            if constexpr (kPair == 2) {
              const uint4 v = *reinterpret_cast<const uint4 *>(rv.rows + at);
              w[q][i] = T::make(v.x, v.y);
              w[q][i + 1] = T::make(v.z, v.w);
            } else {
              w[q][i] = rv.rows[at];
            }
          }
        }
      }
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        const K target = key[q] & T::kLow;
#pragma unroll
        for (u32 i = 0; i < kSlots; ++i) {
          const u32 at = first[q] + i;
          if (at >= lo[q] && at < hi[q] &&
              (T::kw(w[q][i]) & T::kLow) == target) {
            hit[q] = true;
            row[q] = w[q][i];
          }
        }
        if (open[q] && hit[q]) {
          open[q] = false;
          live[q] = !(T::kw(row[q]) & T::kTomb);
          val[q] = T::val(row[q]);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const u64 p = p0 + u64(q) * blockDim.x;
      if (p < end) {
        GroupedResult<T> g;
        g.value = live[q] ? val[q] : V(0);
        g.found = live[q] ? 1 : 0;
        res[p] = g;
      }
    }
  }
}

// Result i = grouped result dest[i], written through the IO policy: dest
// (the partition pass's destination of query i) is read in query order and
// the grouped results come from 256 streams (one per key group) that each
// advance through their own segment, so reads and stores both stream.
// Blocks are dealt to the XCDs like lookup_grouped_kernel's: XCD x answers
// the x-th eighth of the queries, whose results are the x-th eighth of
// every group's segment (the partition is stable), so no result line is
// fetched into more than one XCD's L2.
template <class T, class IO>
__global__ __launch_bounds__(256) void lookup_gather_kernel(
    IO io_arg, const u32 *__restrict__ dest, u64 n,
    const GroupedResult<T> *__restrict__ res) {
  __shared__ __align__(16) char s_io[IO::kStageBytes ? IO::kStageBytes : 16];
  const IO io = io_arg.stage(s_io);
  __syncthreads();
  constexpr int kQ = 4;
  const u32 G = gridDim.x;  // a multiple of 8
  const u32 logical = (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u;
  const u64 chunk = (n + G - 1) / G;
  const u64 begin = u64(logical) * chunk;
  const u64 end = begin + chunk < n ? begin + chunk : n;
  for (u64 p0 = begin + threadIdx.x; p0 < end; p0 += u64(kQ) * blockDim.x) {
    u32 d[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const u64 i = p0 + u64(q) * blockDim.x;
      d[q] = i < end ? dest[i] : 0u;
    }
    GroupedResult<T> g[kQ];
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const u64 i = p0 + u64(q) * blockDim.x;
      if (i < end) g[q] = res[d[q]];
    }
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      const u64 i = p0 + u64(q) * blockDim.x;
      if (i < end) {
        typename IO::Slot slot;
        (void)io.load(i, slot);
        io.put(slot, g[q].found != 0, g[q].value);
      }
    }
  }
}

// Workgroups of a grouped lookup over n queries: a multiple of 8 (one
// share per XCD), two queries per thread.  (The fewer queries an XCD has in
// flight, the fewer groups' rows they touch, and the more of them its L2 holds:
// 8,388,608 lookups 373 us with four queries per thread, 355 with two.)
inline u32 grouped_lookup_blocks(u64 n) {
  const u64 g = (n + 511) / 512;
  const u64 c = g < 1 ? 1 : (g > (1u << 20) ? (1u << 20) : g);
  return static_cast<u32>((c + 7) & ~u64(7));
}

// Range sums and counts over every run.
constexpr int kRangeThreads = 256;
constexpr int kRangeWaves = kRangeThreads / kWave;

template <class T>
struct PlainRange {
  const typename T::K *lo, *hi;
  typename T::V *out;
  int count_only;
  static constexpr u32 kStageBytes = 0;
  __device__ __forceinline__ PlainRange stage(void *) const { return *this; }
  struct Slot {
    u64 q;
  };
  // bounds of query q; `count` selects count (1 per live row) or sum
  __device__ __forceinline__ void load(u64 q, Slot &s, typename T::K &a,
                                       typename T::K &z, bool &count) const {
    s.q = q;
    a = lo[q];
    z = hi[q];
    count = count_only != 0;
  }
  __device__ __forceinline__ void put(const Slot &s, typename T::V v) const {
    out[s.q] = v;
  }
};

// Queries whose bounds a wave resolves together: one lane per (query,
// run, side), at least one query.
__host__ __device__ __forceinline__ u32 range_queries_per_wave(u32 runs) {
  const u32 per = 2 * (runs ? runs : 1);
  return per >= static_cast<u32>(kWave) ? 1u : static_cast<u32>(kWave) / per;
}

// Queries per wave round of a launch of n queries: fewer than the lanes
// allow while that keeps fewer than kRangeSpread waves busy (a few thousand
// queries of a handful of runs would otherwise fill a fraction of the chip;
// with more waves, narrow queries, whose waves then resolve a few bounds each
// on mostly idle lanes, take a second turn on it).  12,000 sums of
// 2^4 to 2^24 keys' width over 7.5 million rows in 4 runs would gain from 8192
// waves (362 -> 244 us), but 8,153 of three rows over 240,860 rows in 3 runs then
// take 16.7 us instead of 11.6.
constexpr u64 kRangeSpread = 2048;
inline u32 range_round(u64 n, u32 runs) {
  const u64 most = range_queries_per_wave(runs);
  const u64 even = (n + kRangeSpread / 2) / kRangeSpread;
  return static_cast<u32>(even < 1 ? 1 : (even < most ? even : most));
}

// A query of more work than this (rows that it reads; rows of newer runs,
// which search the older ones, weigh four) is long: its workgroup's waves
// share it, in chunks of kRangeNewerStep and kRangeOldStep rows.
constexpr u32 kRangeLongWork = 1024;
constexpr u32 kRangeNewerStep = 256;
constexpr u32 kRangeOldStep = 1024;

// Rows of several runs whose newest versions a wave finds in LDS, without a
// search (range_resolve); a workgroup takes four times as many.  (A workgroup's
// registers allow four of them per CU, and so does this LDS.)
constexpr u32 kResolveRows = 512;
constexpr u32 kResolveBlockRows = kRangeWaves * kResolveRows;

// Whether that is the faster way for n ranges over so many runs: a row of a newer
// run searches the older ones one after another, two round trips each.  Sums of n
// ranges of w rows, searching and resolving: 10 equal runs, n = 1, w = 60 23.3 and
// 16.9 us, n = 10,000, w = 600 656 and 88; 40 runs 45 and 22, 9333 and 151.  4 runs
// are the edge, where few ranges are bound by the chain of one wave (falling
// sizes, n = 1025, w = 200 21.5 and 22.8) and many by the searches (n = 10,000, w =
// 600 270 and 112); over 3, n = 10,000, w = 2000 takes 247 and 271.
constexpr u32 kResolveRuns = 5;
constexpr u32 kResolveRunsMany = 4;
constexpr u64 kResolveMany = 2048;
__host__ __device__ __forceinline__ bool range_resolves(u64 n, u32 runs) {
  return runs >= (n < kResolveMany ? kResolveRuns : kResolveRunsMany);
}

// Workgroups that share the long queries of one group of queries: `size` of
// them, this one being number `rank`.  Where size > 1, acc and left (one each
// per query of the launch, zero before and after it) gather their sums.
struct RangeTeam {
  u32 size, rank;
  unsigned long long *acc;
  u32 *left;
};

// A pointer that was kept in LDS: it points to global memory, which the
// compiler cannot see by itself (it would use flat accesses, which wait for
// the LDS accesses in flight too).
template <class E>
__device__ __forceinline__ const E *as_global(const E *p) {
  return (const E *)(const __attribute__((address_space(1))) E *)
      reinterpret_cast<u64>(p);
}

// The runs' headers and pointers in LDS (a lane indexes them by its own run).
template <class T>
struct RangeRuns {
  RunMeta meta[kMaxRuns];
  const typename T::Row *rows_[kMaxRuns];
  const u32 *dir_[kMaxRuns];
  __device__ __forceinline__ const typename T::Row *rows(u32 r) const {
    return as_global(rows_[r]);
  }
  __device__ __forceinline__ const u32 *dir(u32 r) const {
    return as_global(dir_[r]);
  }
  __device__ __forceinline__ void load(const RunSet<T> &runs) {
    if (threadIdx.x < runs.count) {
      meta[threadIdx.x] = *runs.run[threadIdx.x].meta;
      rows_[threadIdx.x] = runs.run[threadIdx.x].rows;
      dir_[threadIdx.x] = runs.run[threadIdx.x].dir;
    }
  }
};

// What row idx of run r adds to its query: its own value (1 for a count, 0
// for a tombstone) less the value of the next older version of its key, which
// it shadows.  A key's versions then add up to its newest one's value, each
// older one being the next older version of exactly one row, so no row has
// to look for newer versions and the oldest run's rows, usually the most, are
// only read.  bnd = the query's bounds ([2r] lower, [2r + 1] upper): the rows
// searched in run s are the query's own, a few of them without the directory.
// (Two or four rows of a lane in lock step were measured slower.)
template <class T>
__device__ __forceinline__ u64 range_row(const RangeRuns<T> &R, const u32 *bnd,
                                         u32 r, u32 idx, u32 oldest,
                                         bool count) {
  using K = typename T::K;
  using Row = typename T::Row;
  const Row w = R.rows(r)[idx];
  u64 v = (T::kw(w) & T::kTomb) ? u64(0) : count ? u64(1) : u64(T::val(w));
  if (r >= oldest) return v;
  const K key = decode_key<T>(T::kw(w), idx, R.meta[r].split);
  const K target = key & T::kLow;
  for (u32 s = r + 1; s <= oldest; ++s) {
    u32 lo = bnd[2 * s], hi = bnd[2 * s + 1];
    if (lo >= hi) continue;
    const Row *rows = R.rows(s);
    if (hi - lo > kFindWindow) {
      const RunMeta &m = R.meta[s];
      const u32 bucket = static_cast<u32>(key >> (T::kBits - m.dir_bits));
      if (bucket < m.lo_bucket || bucket > m.hi_bucket) continue;
      const u32 *dir = R.dir(s);
      const u32 dlo = dir[bucket], dhi = dir[bucket + 1];
      lo = dlo > lo ? dlo : lo;
      hi = dhi < hi ? dhi : hi;
      // wide buckets (skewed keys): bisect; a bucket's keys share the top bit
      while (hi > lo + kFindWindow) {
        const u32 mid = (lo + hi) >> 1;
        const K km = T::kw(rows[mid]) & T::kLow;
        if (km == target) {  // one row is left
          lo = mid;
          hi = mid + 1;
        } else if (km < target) {
          lo = mid + 1;
        } else {
          hi = mid;
        }
      }
    }
    // the window; 8-byte rows in aligned pairs (row arrays carry a spare row,
    // so the pair of a window's last row is inside the allocation)
    constexpr u32 kPair = sizeof(Row) == 8 ? 2 : 1;
    constexpr u32 kSlots = kPair == 2 ? kFindWindow + 2 : kFindWindow;
    Row x[kSlots];
    const u32 at0 = kPair == 2 ? (lo & ~1u) : lo;
#pragma unroll
    for (u32 i = 0; i < kSlots; i += kPair) {
      if (at0 + i < hi) {
        if constexpr (kPair == 2) {
          const uint4 p = *reinterpret_cast<const uint4 *>(rows + at0 + i);
          x[i] = T::make(p.x, p.y);
          x[i + 1] = T::make(p.z, p.w);
        } else {
          x[i] = rows[at0 + i];
        }
      }
    }
    const u32 split = R.meta[s].split;
    bool found = false;
#pragma unroll
    for (u32 i = 0; i < kSlots; ++i) {
      const u32 at = at0 + i;
      if (at >= lo && at < hi && decode_key<T>(T::kw(x[i]), at, split) == key) {
        if (!(T::kw(x[i]) & T::kTomb)) v -= count ? u64(1) : u64(T::val(x[i]));
        found = true;
      }
    }
    if (found) break;
  }
  return v;
}

// What rows [at, at + n) of run r add to a query together (see range_row), by
// one wave whose lanes agree on everything but their rows: run by older run,
// kGroup rows per lane at a time (their directory entries in flight together),
// the runs' pointers and headers in scalar registers.  A key that lies in the
// query's range needs no check against its bounds in a run: the directory's
// rows of its bucket hold it or nothing does.
template <class T>
__device__ __forceinline__ u64 range_run_rows(const RangeRuns<T> &R,
                                              const u32 *bnd, u32 r, u32 at,
                                              u32 n, u32 oldest, bool count) {
  using K = typename T::K;
  using Row = typename T::Row;
  constexpr int kGroup = sizeof(K) == 4 ? 4 : 2;
  const u32 lane = lane_id();
  // (the builtin returns an int: widened as such, a low word with its top
  // bit set would fill the high word)
  auto uniform = [](u32 x) -> u32 { return __builtin_amdgcn_readfirstlane(x); };
  auto uniform_ptr = [&](const auto *p) {
    const u64 a = reinterpret_cast<u64>(p);
    const u64 b = u64(uniform(static_cast<u32>(a >> 32))) << 32 |
                  uniform(static_cast<u32>(a));
    return as_global(reinterpret_cast<decltype(p)>(b));
  };
  const Row *own = uniform_ptr(R.rows(r));
  const u32 own_split = uniform(R.meta[r].split);
  u64 acc = 0;
  for (u32 i0 = 0; i0 < n; i0 += kGroup * kWave) {
    Row w[kGroup];
    K key[kGroup];
    bool open[kGroup];
#pragma unroll
    for (int j = 0; j < kGroup; ++j) {
      const u32 i = i0 + j * kWave + lane;
      open[j] = i < n;
      if (open[j]) w[j] = own[at + i];
    }
#pragma unroll
    for (int j = 0; j < kGroup; ++j) {
      key[j] = 0;
      if (open[j]) {
        key[j] = decode_key<T>(T::kw(w[j]), at + i0 + j * kWave + lane,
                               own_split);
        if (!(T::kw(w[j]) & T::kTomb)) acc += count ? u64(1) : u64(T::val(w[j]));
      }
    }
    for (u32 s = r + 1; s <= oldest; ++s) {
      if (uniform(bnd[2 * s]) >= uniform(bnd[2 * s + 1])) continue;
      const Row *rows = uniform_ptr(R.rows(s));
      const u32 *dir = uniform_ptr(R.dir(s));
      const u32 shift = T::kBits - uniform(R.meta[s].dir_bits);
      const u32 lo_b = uniform(R.meta[s].lo_bucket);
      const u32 hi_b = uniform(R.meta[s].hi_bucket);
      u32 lo[kGroup], hi[kGroup];
#pragma unroll
      for (int j = 0; j < kGroup; ++j) {
        const u32 bucket = static_cast<u32>(key[j] >> shift);
        lo[j] = hi[j] = 0;
        if (open[j] && bucket >= lo_b && bucket <= hi_b) {
          lo[j] = dir[bucket];
          hi[j] = dir[bucket + 1];
        }
      }
#pragma unroll
      for (int j = 0; j < kGroup; ++j) {
        const K target = key[j] & T::kLow;
        u32 a = lo[j], z = hi[j];
        while (z - a > kFindWindow) {  // wide buckets (skewed keys)
          const u32 mid = (a + z) >> 1;
          const K km = T::kw(rows[mid]) & T::kLow;
          if (km == target) {  // one row is left
            a = mid;
            z = mid + 1;
          } else if (km < target) {
            a = mid + 1;
          } else {
            z = mid;
          }
        }
        Row x[kFindWindow];
#pragma unroll
        for (u32 k = 0; k < kFindWindow; ++k)
          if (a + k < z) x[k] = rows[a + k];
#pragma unroll
        for (u32 k = 0; k < kFindWindow; ++k) {
          if (a + k < z && (T::kw(x[k]) & T::kLow) == target) {
            if (!(T::kw(x[k]) & T::kTomb))
              acc -= count ? u64(1) : u64(T::val(x[k]));
            open[j] = false;
          }
        }
      }
    }
  }
  return acc;
}

// What chunk c of a long query adds to it: rows of the newer runs (run after
// run, kRangeNewerStep at a time), then of the oldest, by one wave.
template <class T>
__device__ __forceinline__ u64 range_chunk(const RangeRuns<T> &R,
                                           const u32 *bnd, u32 first,
                                           u32 oldest, bool count, u64 c,
                                           u64 newer_chunks) {
  u64 acc = 0;
  if (c < newer_chunks) {
    u64 off = c * kRangeNewerStep;
    u32 rest = kRangeNewerStep;
    for (u32 r = first; r < oldest && rest; ++r) {
      const u32 cnt = bnd[2 * r + 1] - bnd[2 * r];
      if (off >= cnt) {
        off -= cnt;
        continue;
      }
      const u32 take = cnt - off < rest ? static_cast<u32>(cnt - off) : rest;
      acc += range_run_rows<T>(R, bnd, r, bnd[2 * r] + static_cast<u32>(off),
                               take, oldest, count);
      rest -= take;
      off = 0;
    }
    return acc;
  }
  const u64 a = bnd[2 * oldest] + (c - newer_chunks) * kRangeOldStep;
  const u64 z = a + kRangeOldStep < bnd[2 * oldest + 1]
                    ? a + kRangeOldStep
                    : bnd[2 * oldest + 1];
  const typename T::Row *rows = R.rows(oldest);
  auto add = [&](const typename T::Row &w) {
    if (!(T::kw(w) & T::kTomb)) acc += count ? u64(1) : u64(T::val(w));
  };
  u64 i = a + lane_id();
  for (; i + 3 * kWave < z; i += 4 * kWave) {  // four rows of a lane in flight
    typename T::Row w[4];
#pragma unroll
    for (u32 j = 0; j < 4; ++j) w[j] = rows[i + j * kWave];
#pragma unroll
    for (u32 j = 0; j < 4; ++j) add(w[j]);
  }
  for (; i < z; i += kWave) add(rows[i]);
  return acc;
}

// What the `total` rows of some queries add up to, by kLanes lanes together (a
// wave, or the workgroup), each key's newest version alone: every row is read
// once, into an LDS table of the queries' keys that keeps the first row of each
// key (a query's rows come run after run, the newest first), and a row counts
// when the table kept it.  No row waits for a search, so what is left is one
// round of loads.
//
// at(f): where row f is (called for a lane's rows in ascending order): its
// address, whether it lies behind its run's split, its query, and whether that
// one counts.  span(q): query q's rows [begin, end).  add(q, v): called for each
// row that counts.
template <class T>
struct ResolveRow {
  const typename T::Row *row;
  bool top, count;
  u32 q;
};
template <class T, u32 kLanes, class At, class Span, class Add>
__device__ __forceinline__ void range_resolve(typename T::K *keys, u32 *slots,
                                              u32 total, u32 tid, At &&at,
                                              Span &&span, Add &&add) {
  using K = typename T::K;
  using V = typename T::V;
  constexpr int kItems = kResolveRows / kWave;
  constexpr int kLoads = 4;  // rows of a lane in flight
  auto sync = [] {
    if constexpr (kLanes == kWave) {
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    } else {
      __syncthreads();
    }
  };
  // (else its items' LDS addresses are worked out at the kernel's start and
  // held in registers from there)
  asm volatile("" : "+v"(tid));
  // at least two slots per row
  u32 log = 7;
  while ((1u << log) < 2 * total) ++log;
  for (u32 i = tid; i < (1u << log); i += kLanes) slots[i] = 0;
  V val[kItems];
  u32 tag[kItems];  // the query, from the search on the slot (<< 8)
#pragma unroll
  for (int j0 = 0; j0 < kItems; j0 += kLoads) {
    typename T::Row w[kLoads];
    u32 top = 0, count = 0;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const u32 f = (j0 + j) * kLanes + tid;
      tag[j0 + j] = 0;
      if (f < total) {
        const ResolveRow<T> x = at(f);
        w[j] = *x.row;
        top |= x.top ? 1u << j : 0u;
        count |= x.count ? 1u << j : 0u;
        tag[j0 + j] = x.q;
      }
    }
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const u32 f = (j0 + j) * kLanes + tid;
      if (f < total) {
        const K kw = T::kw(w[j]);
        keys[f] = (kw & T::kLow) | ((top >> j) & 1u ? T::kTomb : K(0));
        val[j0 + j] = (kw & T::kTomb) ? V(0)
                      : (count >> j) & 1u ? V(1) : T::val(w[j]);
      }
    }
  }
  sync();
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const u32 f = j * kLanes + tid;
    if (f < total) {
      const uint2 own = span(tag[j]);
      const K key = keys[f];
      u32 x = static_cast<u32>(key);
      if constexpr (sizeof(K) == 8) x ^= static_cast<u32>(key >> 32);
      u32 h = (x * 0x9E3779B1u + tag[j] * 0x85EBCA77u) >> (32 - log);
      while (true) {  // (some slot is free)
        const u32 cur = atomicCAS(&slots[h], 0u, f + 1);
        if (cur == 0) break;
        if (cur > own.x && cur <= own.y && keys[cur - 1] == key) {
          atomicMin(&slots[h], f + 1);
          break;
        }
        h = (h + 1) & ((1u << log) - 1u);
      }
      tag[j] |= h << 8;
    }
  }
  sync();
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const u32 f = j * kLanes + tid;
    if (f < total && slots[tag[j] >> 8] == f + 1) add(tag[j] & 0xffu, val[j]);
  }
}

// The range kernel's work on queries [q_begin, q_end) by the calling
// workgroup, number group of a grid of groups (the range kernel's, or the
// serving engine's step kernel taking chunks of queries), qw queries per wave
// and round.  `io` is already staged; every thread of the workgroup calls it.
//
// The lanes first resolve the bounds of a wave's queries in every run at
// once (one lane per query, run and side).  The rows of all short queries are
// then flattened over the lanes (range_row), so a round costs a few memory
// round trips however many queries it holds; a lane keeps its sum in a
// register until its next row belongs to another query.  Long queries wait
// in a list until the workgroup's waves have their short ones, and are then
// shared by all of them (and by the workgroup's team).  A count takes the rows
// of a query's oldest run from its bounds when that run has no tombstones.
// Sums are modulo 2^64 and are truncated to the value width.
//
// With `resolve` (range_resolves; kResolve: compiled for it), queries with rows of
// several runs search nothing up to kResolveBlockRows rows: a wave resolves its
// short ones in LDS, as many at a time as fit, and the workgroup's waves one of
// more than kResolveRows rows together (range_resolve).
//
// Bound by the searches, one per newer row and older run (directory entries,
// then rows), whose lines come from beyond the L2 in a dictionary of tens of
// megabytes, and by the rows read once.  A launch of 12,000 sums (or counts) of
// 2^4 to 2^24 keys' width over 6 million rows in 4 runs, a tenth tombstones: 0.72
// ms (9 ms when a wave answered each query and every row looked for newer
// versions, in LDS or, beyond 2048 of them, in global memory); 16,384 of up to 100
// rows over one run of 2^20: counts 6.5 us (9.8), sums 12 (36).  A queue of all
// long queries' chunks for a second launch made the wide ones some 30% faster,
// but every small call on a large dictionary 3 to 5 us longer.
template <class T, bool kResolve, class IO>
__device__ __forceinline__ void range_block(const IO &io, u64 q_begin,
                                            u64 q_end, const RunSet<T> &runs,
                                            u64 group, u64 groups, u32 qw,
                                            const RangeTeam &team,
                                            bool resolve) {
  using K = typename T::K;
  constexpr u32 kSlots =
      2 * kMaxRuns > kWave ? 2 * kMaxRuns : static_cast<u32>(kWave);
  constexpr u32 kQMax = kWave / 2;  // queries per wave and round
  // s_b[wave][2 * (qi * runs + r) + side]: lower (side 0) and upper (side
  // 1) bound of query qi of the round in run r
  __shared__ u32 s_b[kRangeWaves][kSlots];
  __shared__ RangeRuns<T> R;
  __shared__ typename IO::Slot s_slot[kRangeWaves][kQMax];
  // per query of the round: flags (exists, a <= z, count), plan (first |
  // oldest << 8), work offset and sum
  __shared__ u32 s_flags[kRangeWaves][kQMax];
  __shared__ u32 s_plan[kRangeWaves][kQMax];
  __shared__ u32 s_woff[kRangeWaves][kQMax];
  // rows resolved in LDS, their keys and table
  __shared__ u32 s_roff[kRangeWaves][kResolve ? kQMax + 1 : 1];
  __shared__ unsigned long long s_acc[kRangeWaves][kQMax];
  __shared__ K s_keys[kResolve ? kResolveBlockRows : 1];
  __shared__ u32 s_slots[kResolve ? 2 * kResolveBlockRows : 1];
  // the round's queries that all waves share (wave << 8 | query, kWhole: its
  // rows are resolved in LDS); round k counts in slot k % 3 and clears the next
  // one, which no wave can still be reading
  constexpr u32 kWhole = 1u << 16;
  __shared__ u32 s_list[kRangeWaves * kQMax];
  __shared__ u32 s_long[3];
  const u32 nr = runs.count;
  resolve = kResolve && resolve;
  __syncthreads();  // a previous call's readers of R are done
  R.load(runs);
  if (threadIdx.x < 3) s_long[threadIdx.x] = 0;
  __syncthreads();
  const u32 lane = lane_id();
  const u32 wave = threadIdx.x / kWave;
  const u32 per = 2 * nr;
  u32 turn = 0;
  for (u64 g0 = q_begin + group * (kRangeWaves * qw); g0 < q_end;
       g0 += groups * (kRangeWaves * qw), turn = turn == 2 ? 0 : turn + 1) {
    const u64 q0 = g0 + u64(wave) * qw;
    // every bound of the round at once, one lane each (and one per query
    // when there are no runs: every range is empty)
    const u32 step = per ? per : 1;
    for (u32 t = lane; t < qw * step; t += kWave) {
      const u64 q = q0 + t / step;
      const u32 r = (t % step) >> 1;
      u32 b = 0;
      u32 flags = 0;
      typename IO::Slot slot{};
      if (q < q_end) {
        K a, z;
        bool count_only;
        io.load(q, slot, a, z, count_only);
        flags = 1u | (a <= z ? 2u : 0u) | (count_only ? 4u : 0u);
        if (a <= z && per) {
          const RunView<T> rv{R.rows(r), R.dir(r), nullptr};
          const RunMeta m = R.meta[r];
          b = (t & 1) ? run_upper_bound(rv, m, z) : run_lower_bound(rv, m, a);
        }
      }
      if (per) s_b[wave][t] = b;
      if (t % step == 0) {
        s_slot[wave][t / step] = slot;
        s_flags[wave][t / step] = flags;
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");

    // ---- plan of query q0 + lane (lanes below qw)
    u32 work = 0, resolved = 0;
    bool is_long = false;
    if (lane < qw) {
      const u32 flags = s_flags[wave][lane];
      const u32 *bnd = &s_b[wave][lane * per];
      u32 plan = 0;
      u64 base = 0;
      if ((flags & 3u) == 3u) {
        u32 first = nr, oldest = 0;
        for (u32 r = 0; r < nr; ++r) {
          if (bnd[2 * r] < bnd[2 * r + 1]) {
            if (first == nr) first = r;
            oldest = r;
          }
        }
        if (first < nr) {
          u64 newer = 0;
          for (u32 r = first; r < oldest; ++r)
            newer += bnd[2 * r + 1] - bnd[2 * r];
          u32 old_rows = bnd[2 * oldest + 1] - bnd[2 * oldest];
          plan = first | (oldest << 8);
          const u64 all = newer + old_rows;
          const bool from_bounds = (flags & 4u) && R.meta[oldest].tombs == 0;
          is_long = 4 * newer + (from_bounds ? 0u : old_rows) > kRangeLongWork;
          // (rows that would search many runs one after another)
          const bool whole =
              resolve && newer && all > kResolveRows &&
              all <= kResolveBlockRows &&
              (is_long || newer * (oldest - first) > kResolveRows);
          if (resolve && newer && all <= kResolveRows) {
            is_long = false;
            if (team.rank == 0) resolved = static_cast<u32>(all);
          } else if (whole) {
            is_long = true;
          } else if (from_bounds) {
            base = team.rank == 0 ? old_rows : 0;
            old_rows = 0;
          }
          if (is_long)
            s_list[atomicAdd(&s_long[turn], 1u)] =
                wave << 8 | lane | (whole ? kWhole : 0u);
          else if (team.rank == 0 && !resolved)
            work = static_cast<u32>(newer + old_rows);
        }
      }
      s_plan[wave][lane] = plan;
      s_acc[wave][lane] = base;
    }
    const u32 work_inc = wave_inclusive_scan(work);
    if (lane < qw) s_woff[wave][lane] = work_inc - work;
    const u32 wend = __shfl(work_inc, kWave - 1, kWave);
    u32 rend = 0;
    if constexpr (kResolve) {
      const u32 inc = wave_inclusive_scan(resolved);
      if (lane < qw) s_roff[wave][lane + 1] = inc;
      if (lane == 0) s_roff[wave][0] = 0;
      rend = __shfl(inc, kWave - 1, kWave);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");

    // ---- the short queries whose rows are resolved in LDS, as many as fit at
    // a time
    if (kResolve && rend) {
      u32 g0 = 0;
      while (g0 < qw) {
        const u32 *off = s_roff[wave];
        const u32 from = __builtin_amdgcn_readfirstlane(off[g0]);
        // the first query whose rows end behind the group's room
        const u64 over =
            ballot(lane < qw && off[lane + 1] - from > kResolveRows &&
                   lane >= g0);
        const u32 g1 = over ? static_cast<u32>(ffs64(over)) - 1 : qw;
        const u32 total = __builtin_amdgcn_readfirstlane(off[g1]) - from;
        if (total) {
          u32 qi = g0, r = ~0u, first_row = 0;  // run r's rows start there
          range_resolve<T, kWave>(
              s_keys + wave * kResolveRows, s_slots + wave * 2 * kResolveRows,
              total, lane,
              [&](u32 f) -> ResolveRow<T> {
                const u32 at = from + f;
                while (off[qi + 1] <= at) {
                  ++qi;
                  r = ~0u;
                }
                const u32 *bnd = &s_b[wave][qi * per];
                if (r == ~0u) {
                  r = s_plan[wave][qi] & 0xffu;
                  first_row = off[qi];
                }
                while (at - first_row >= bnd[2 * r + 1] - bnd[2 * r]) {
                  first_row += bnd[2 * r + 1] - bnd[2 * r];
                  ++r;
                }
                const u32 idx = bnd[2 * r] + (at - first_row);
                return {R.rows(r) + idx, idx >= R.meta[r].split,
                        (s_flags[wave][qi] & 4u) != 0, qi};
              },
              [&](u32 q) { return make_uint2(off[q] - from, off[q + 1] - from); },
              [&](u32 q, typename T::V v) {
                if (v)
                  atomicAdd(&s_acc[wave][q], static_cast<unsigned long long>(v));
              });
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
        g0 = g1;
      }
    }

    // rows of the short queries, flattened query after query, run after run
    if (wend) {
      u32 qi = 0;
      u64 acc = 0;
      if (lane < wend) {
        u32 hi = qw;
        while (hi - qi > 1) {  // the last query whose offset is <= lane
          const u32 mid = (qi + hi) >> 1;
          if (s_woff[wave][mid] <= lane) qi = mid;
          else hi = mid;
        }
      }
      for (u32 f = lane; f < wend; f += kWave) {
        u32 next = qi;
        while (next + 1 < qw && s_woff[wave][next + 1] <= f) ++next;
        if (next != qi) {
          if (acc)
            atomicAdd(&s_acc[wave][qi], static_cast<unsigned long long>(acc));
          acc = 0;
          qi = next;
        }
        const u32 plan = s_plan[wave][qi];
        const u32 *bnd = &s_b[wave][qi * per];
        u32 r = plan & 0xffu, off = f - s_woff[wave][qi];
        while (off >= bnd[2 * r + 1] - bnd[2 * r]) {
          off -= bnd[2 * r + 1] - bnd[2 * r];
          ++r;
        }
        acc += range_row<T>(R, bnd, r, bnd[2 * r] + off, plan >> 8,
                            (s_flags[wave][qi] & 4u) != 0);
      }
      // one addition per wave when its lanes end in one query
      const u32 lead = __builtin_amdgcn_readfirstlane(qi);
      if (ballot(qi != lead && acc) == 0) {
        acc = wave_sum_u64(acc);
        if (lane == 0 && acc)
          atomicAdd(&s_acc[wave][lead], static_cast<unsigned long long>(acc));
      } else if (acc) {
        atomicAdd(&s_acc[wave][qi], static_cast<unsigned long long>(acc));
      }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (lane < qw && !is_long && team.rank == 0 && (s_flags[wave][lane] & 1u))
      io.put(s_slot[wave][lane],
             static_cast<typename T::V>(s_acc[wave][lane]));

    // ---- the workgroup's long queries, by all its waves
    if (threadIdx.x == 0) s_long[turn == 2 ? 0 : turn + 1] = 0;
    __syncthreads();
    const u32 longs = s_long[turn];
    if (!longs) continue;
    for (u32 l = 0; l < longs; ++l) {
      const u32 id = s_list[l], w = (id >> 8) & 0xffu, qi = id & 0xffu;
      const u32 *bnd = &s_b[w][qi * per];
      const u32 first = s_plan[w][qi] & 0xffu, oldest = s_plan[w][qi] >> 8;
      const bool count = (s_flags[w][qi] & 4u) != 0;
      if (kResolve && (id & kWhole)) {
        if (team.rank) continue;
        u32 total = 0;
        for (u32 r = first; r <= oldest; ++r)
          total += bnd[2 * r + 1] - bnd[2 * r];
        u32 r = first, first_row = 0;
        u64 acc = 0;
        range_resolve<T, kRangeThreads>(
            s_keys, s_slots, total, threadIdx.x,
            [&](u32 f) -> ResolveRow<T> {
              while (f - first_row >= bnd[2 * r + 1] - bnd[2 * r]) {
                first_row += bnd[2 * r + 1] - bnd[2 * r];
                ++r;
              }
              const u32 idx = bnd[2 * r] + (f - first_row);
              return {R.rows(r) + idx, idx >= R.meta[r].split, count, 0u};
            },
            [&](u32) { return make_uint2(0u, total); },
            [&](u32, typename T::V v) { acc += v; });
        acc = wave_sum_u64(acc);
        if (lane == 0 && acc)
          atomicAdd(&s_acc[w][qi], static_cast<unsigned long long>(acc));
        __syncthreads();  // the table is used again
        continue;
      }
      u64 newer = 0;
      for (u32 r = first; r < oldest; ++r) newer += bnd[2 * r + 1] - bnd[2 * r];
      const u64 old_rows = count && R.meta[oldest].tombs == 0
                               ? 0
                               : bnd[2 * oldest + 1] - bnd[2 * oldest];
      const u64 nc = (newer + kRangeNewerStep - 1) / kRangeNewerStep;
      const u64 chunks = nc + (old_rows + kRangeOldStep - 1) / kRangeOldStep;
      u64 acc = 0;
      for (u64 c = u64(team.rank) * kRangeWaves + wave; c < chunks;
           c += u64(team.size) * kRangeWaves)
        acc += range_chunk<T>(R, bnd, first, oldest, count, c, nc);
      acc = wave_sum_u64(acc);
      if (lane == 0 && acc)
        atomicAdd(&s_acc[w][qi], static_cast<unsigned long long>(acc));
    }
    __syncthreads();
    if (threadIdx.x < longs) {
      const u32 id = s_list[threadIdx.x], w = (id >> 8) & 0xffu, qi = id & 0xffu;
      u64 sum = s_acc[w][qi];
      bool last = !(id & kWhole) || team.rank == 0;
      if (team.size > 1 && !(id & kWhole)) {
        // The sum must have taken this workgroup's share before `left`
        // counts it.  The value that the addition returns is waited for
        // instead of a fence, which would write back and empty the L2.
        const u64 q = g0 + u64(w) * qw + qi;
        u64 before =
            atomicAdd(&team.acc[q], static_cast<unsigned long long>(sum));
        asm volatile("" : "+v"(before) : : "memory");
        last = atomicAdd(&team.left[q], 1u) == team.size - 1;
        if (last) {
          sum = atomicExch(&team.acc[q], 0ull);
          atomicExch(&team.left[q], 0u);
        }
      }
      if (last) io.put(s_slot[w][qi], static_cast<typename T::V>(sum));
    }
    __syncthreads();  // the next round writes the bounds and the list again
  }
}

// Teams of team.size consecutive workgroups (team.rank is set here).
template <class T, bool kResolve, class IO>
__global__ __launch_bounds__(kRangeThreads) void range_kernel(
    IO io_arg, u64 n, RunSet<T> runs, u32 qw, RangeTeam team) {
  __shared__ __align__(16) char s_io[IO::kStageBytes ? IO::kStageBytes : 16];
  const IO io = io_arg.stage(s_io);  // range_block's first barrier orders it
  team.rank = blockIdx.x % team.size;
  range_block<T, kResolve>(io, 0, n, runs, blockIdx.x / team.size,
                           gridDim.x / team.size, qw, team, kResolve);
}

// Smallest live key >= query, all-ones when there is none.
//
// A query has a group of lanes, a lane per run (1 << group_log >= the runs): each
// finds its run's first row at or above the query, and the group's smallest key
// is the candidate.  Its newest holder, the group's first lane with that key,
// decides whether it lives; if not, the lanes that hold it step to their next
// row.  A thread per query searched the runs one after another, then searched
// each again for the candidate's newest version, and started over behind a dead
// key: 3,431 queries of skewed 64-bit keys, a third of them erased, took 60 us,
// now 6; 2^20 in 6 million rows of 32 bits 332 and 213.
template <class T>
__global__ __launch_bounds__(256) void successor_kernel(
    const typename T::K *__restrict__ queries, u64 n,
    typename T::K *__restrict__ out, RunSet<T> runs, u32 group_log) {
  using K = typename T::K;
  __shared__ RangeRuns<T> R;
  if (runs.count == 0) {  // no row to load
    for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += u64(gridDim.x) * blockDim.x)
      out[i] = T::kAllOnes;
    return;
  }
  R.load(runs);
  __syncthreads();
  const u32 lane = lane_id();
  const u32 G = 1u << group_log, r = lane & (G - 1);
  const u64 group = (G == 64 ? ~u64(0) : (u64(1) << G) - 1) << (lane - r);
  const bool mine = r < runs.count;
  const u32 at = mine ? r : 0;
  const typename T::Row *rows = R.rows(at);
  const RunMeta m = R.meta[at];
  const RunView<T> rv{rows, R.dir(at), nullptr};
  const u32 per = blockDim.x >> group_log;  // queries of a workgroup's round
  for (u64 base = u64(blockIdx.x) * per; base < n;
       base += u64(gridDim.x) * per) {
    const u64 q = base + (threadIdx.x >> group_log);
    bool open = q < n;  // the same for a group's lanes
    const K query = queries[open ? q : n - 1];
    u32 p = mine ? run_lower_bound(rv, m, query) : 0u;
    K result = T::kAllOnes;
    // The loop exchanges values over the whole wave, so its lanes have to stay
    // together: a lane steps by a select and every lane loads in each round (the
    // run's first row where it did not step or has none left: few lines).  With
    // a branch around the step the compiler made an inner loop of the lanes that
    // stepped, whose exchanges then missed the other lanes' keys: wrong
    // successors.
    bool step = open && mine;
    K w = 0;
    while (ballot(open)) {
      const bool has = mine && p < m.count;
      const K x = T::kw(rows[step && has ? p : 0u]);
      w = step ? x : w;
      const K k = decode_key<T>(w, p, m.split);
      K best = has ? k : T::kAllOnes;
      for (u32 o = 1; o < G; o <<= 1) {
        const K other = __shfl_xor(best, o, kWave);
        best = other < best ? other : best;
      }
      const bool holds = has && k == best;
      const u64 holders = ballot(holds) & group;
      const u64 tombs = ballot(has && (w & T::kTomb) != 0);
      const u64 newest = holders & (~holders + 1);
      const bool live = holders && !(tombs & newest);
      result = open && live ? best : result;
      open = open && holders && !live && best != T::kAllOnes;
      step = open && holds;
      p += step ? 1u : 0u;
    }
    if (q < n && r == 0) out[q] = result;
  }
}

// Writes a tombstone-free run as plain (key, value) arrays.
template <class T>
__global__ void decode_run_kernel(const typename T::Row *__restrict__ rows,
                                  const RunMeta *meta,
                                  typename T::K *__restrict__ ok,
                                  typename T::V *__restrict__ ov) {
  const u32 count = meta->count, split = meta->split;
  const u64 stride = u64(gridDim.x) * blockDim.x;
  for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < count;
       i += stride) {
    const u32 pos = static_cast<u32>(i);
    const typename T::Row r = rows[pos];
    ok[i] = decode_key<T>(T::kw(r), pos, split);
    ov[i] = T::val(r);
  }
}

}  // namespace lsm
}  // namespace gdict
