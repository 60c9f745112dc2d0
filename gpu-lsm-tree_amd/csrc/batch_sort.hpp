// Admission of 64-bit batches in four launches instead of a radix sort's eight
// passes and a finalize launch with a gather of the values:
//
//   seg_tile_hist_kernel, seg_tile_scan_kernel (seg_admission.hpp)
//                     the batch's top varying bit h, its keys' counts by the
//                     top digit (the 8 bits up to h) and each tile's offsets
//   onesweep pass     a stable partition by the top digit, carrying the
//                     values
//   batch_local_kernel
//                     a workgroup per digit: sorts its keys in LDS by the bits
//                     that vary among them, keeps the newest of equal keys,
//                     takes its output offset from a chained scan, and writes
//                     rows, radix directory and header
//
// A batch whose most frequent digit does not fit the LDS (few dense clusters,
// keys that repeat thousands of times) is sorted by the radix passes instead.
// The device decides: both sets of launches are made, and those that the
// batch does not need return at once, so nothing waits for the host.  A batch
// that fits the LDS whole takes batch_local_kernel alone; so do 32-bit ones
// (larger ones take the segmented admission).
//
// Batches of 700,001 uniform 64-bit updates: 190 us each by radix passes, 85 so
// (histogram and scan 12, partition 17, local sort 26, the unused launches 30).
// Of a batch that takes the radix passes, those over constant digits are
// skipped, so keys of a narrow range gain too: 467,677 Zipf keys of 30 bits 150
// us instead of 185.
#pragma once

#include "radix_sort.hpp"
#include "seg_admission.hpp"

namespace gdict {
namespace bs {

using lsm::top_bit;

// Device words of one sort, cleared by its first launch.
struct Plan {
  u32 shift_top;  // shift of the top digit
  u32 largest;    // keys of the most frequent top digit
  u32 ticket;
  u32 pad;
};
constexpr u64 kPlanWords = sizeof(Plan) / sizeof(u32);
static_assert(kPlanWords % 2 == 0, "64-bit words follow");

// Where a partition pass reads its batch.  A payload policy `fn` gives input
// element idx's payload: fn(idx, key, top) (which may rewrite a key bit that
// no digit of the sort reads).
template <class K, class P, class Fn>
struct InputSource {
  const K *keys;
  Fn fn;
  __device__ __forceinline__ void load(u64 idx, bool valid, u32 top, K &key,
                                       P &val) const {
    key = valid ? keys[idx] : ~K(0);
    val = valid ? fn(idx, key, top) : P(0);
  }
};

// ------------------------------------------------------------- local sort
// Workgroup shape.  kCap: keys that it sorts in LDS.
template <class K, class P, int kThreadsArg, int kItemsArg>
struct Shape {
  static constexpr int kThreads = kThreadsArg;
  static constexpr int kItems = kItemsArg;
  static constexpr u32 kCap = kThreads * kItems;
  static constexpr int kWaves = kThreads / kWave;
  static constexpr u32 kBuckets = 4096;
  static constexpr u32 kBucketMax = 16;  // keys of a bucket that are ranked
  static_assert(kBuckets % kThreads == 0 && kWaves * 256 <= kBuckets,
                "an equal share of the buckets per thread");
  static_assert(kWaves >= 2, "the offset scan and the look-back use two waves");
  static_assert(kCap <= 65536, "16-bit positions");

  struct Shared {
    K k[kCap];
    P p[kCap];
    unsigned short at[kCap];
    u32 cnt[kBuckets];  // bucket counts, or the waves' digit counts
    u32 digit_start[256];
    u32 scan[kWaves + 1];
    u32 off[kItems][kWaves];
    u32 misc[8];
    K span[kWaves];
    u64 base;
  };
};

// OR over the workgroup.
template <class S, class K>
__device__ __forceinline__ K block_or(typename S::Shared &sh, K v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v |= __shfl_xor(v, o, kWave);
  __syncthreads();  // the previous use of sh.span is read
  if (lane_id() == 0) sh.span[threadIdx.x / kWave] = v;
  __syncthreads();
  K o = 0;
#pragma unroll
  for (int w = 0; w < S::kWaves; ++w) o |= sh.span[w];
  return o;
}

// Stable ranking of a chunk of `count` keys by the digit at `shift`, ipt per
// lane: wave w holds chunk elements [w * 64 * ipt, (w + 1) * 64 * ipt), item j
// of lane l is element w * 64 * ipt + j * 64 + l.  dst[j] = its position in
// the chunk sorted by the digit, sh.digit_start = each digit's start.
template <class S, class K>
__device__ __forceinline__ void digit_rank(typename S::Shared &sh,
                                           const K (&key)[S::kItems],
                                           u32 count, u32 ipt, u32 shift,
                                           u32 (&dst)[S::kItems]) {
  const u32 tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  const u32 wave_base = wave * kWave * ipt;
  u32 *my = sh.cnt + wave * 256;
  for (u32 i = tid; i < u32(S::kWaves) * 256; i += S::kThreads) sh.cnt[i] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < S::kItems; ++j) {
    if (static_cast<u32>(j) < ipt) {
      const bool valid = wave_base + j * kWave + lane < count;
      const u32 d = static_cast<u32>(key[j] >> shift) & 0xffu;
      dst[j] = count_peers(&my[d], digit_peers(d, ballot(valid)), valid);
    }
  }
  __syncthreads();
  u32 total = 0;
  if (tid < 256)
    for (int w = 0; w < S::kWaves; ++w) total += sh.cnt[w * 256 + tid];
  const u32 inclusive = wave_inclusive_scan(tid < 256 ? total : 0u);
  if (tid < 256 && lane == kWave - 1) sh.scan[wave] = inclusive;
  __syncthreads();
  if (tid < 256) {
    u32 start = inclusive - total;
    for (u32 w = 0; w < wave; ++w) start += sh.scan[w];
    sh.digit_start[tid] = start;
    for (int w = 0; w < S::kWaves; ++w) {
      const u32 c = sh.cnt[w * 256 + tid];
      sh.cnt[w * 256 + tid] = start;
      start += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < S::kItems; ++j)
    if (static_cast<u32>(j) < ipt)
      dst[j] += my[static_cast<u32>(key[j] >> shift) & 0xffu];
}

// Sorts sh.k / sh.p (m elements, being written) stably by the digits that vary
// (span).  Not inlined: a rare path, whose registers would otherwise be spilled
// around the common one.
template <class S, class K, class P>
__device__ __attribute__((noinline)) void digit_sort(typename S::Shared *shp,
                                                     u32 m, K span) {
  typename S::Shared &sh = *shp;
  const u32 tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  const u32 bits = span ? top_bit(span) + 1 : 0u;
  const u32 ipt = __builtin_amdgcn_readfirstlane((m + S::kThreads - 1) /
                                                 S::kThreads);
  const u32 wave_base = wave * kWave * ipt;
  for (u32 shift = 0; shift < bits; shift += 8) {
    if (((span >> shift) & K(0xff)) == 0) continue;
    __syncthreads();  // the arrays are written
    K kk[S::kItems];
    P pp[S::kItems];
    u32 dst[S::kItems];
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      const u32 i = wave_base + j * kWave + lane;
      kk[j] = ~K(0);
      if (static_cast<u32>(j) < ipt && i < m) {
        kk[j] = sh.k[i];
        pp[j] = sh.p[i];
      }
    }
    digit_rank<S, K>(sh, kk, m, ipt, shift, dst);  // (its barriers order the
                                                   // reads before the writes)
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      const u32 i = wave_base + j * kWave + lane;
      if (static_cast<u32>(j) < ipt && i < m) {
        sh.k[dst[j]] = kk[j];
        sh.p[dst[j]] = pp[j];
      }
    }
  }
  __syncthreads();
}

// Sorts m <= kCap keys (k, p: item j of thread t is element j * kThreads + t)
// into sh.k / sh.p, stably, by the bits of `order`.  One counting pass over
// the top 12 of the bits that vary among them puts about a key into each
// bucket; every key claims a slot of its bucket and takes the place that its
// (key, position) rank inside the bucket gives it.  When a bucket holds more
// than kBucketMax keys (dense or repeated keys), the keys take stable passes
// over the digits that vary instead.
template <class S, class K, class P>
__device__ __forceinline__ void local_sort(typename S::Shared &sh,
                                           const K (&k)[S::kItems],
                                           const P (&p)[S::kItems], u32 m,
                                           K order) {
  const u32 tid = threadIdx.x, lane = lane_id();
  for (u32 i = tid; i < S::kBuckets; i += S::kThreads) sh.cnt[i] = 0;
  // the bits that vary: against thread 0's first key
  __shared__ K s_first;
  if (tid == 0) {
    sh.misc[6] = 0;  // largest bucket
    s_first = k[0];
  }
  __syncthreads();
  const K first = s_first;
  K acc = 0;
#pragma unroll
  for (int j = 0; j < S::kItems; ++j)
    if (j * S::kThreads + tid < m) acc |= k[j] ^ first;
  const K span = block_or<S, K>(sh, acc & order);
  const u32 bits = span ? top_bit(span) + 1 : 0u;
  const u32 hb = bits < 12 ? bits : 12;
  const u32 lsh = bits - hb;
  const u32 bmask = (1u << hb) - 1u;
  u32 b[S::kItems];
#pragma unroll
  for (int j = 0; j < S::kItems; ++j) {
    b[j] = 0;
    if (j * S::kThreads + tid < m) {
      b[j] = static_cast<u32>((k[j] & order) >> lsh) & bmask;
      atomicAdd(&sh.cnt[b[j]], 1u);
    }
  }
  __syncthreads();
  // bucket starts: thread t owns buckets [t * kPer, (t + 1) * kPer)
  constexpr u32 kPer = S::kBuckets / S::kThreads;
  {
    u32 c[kPer], sum = 0, most = 0;
#pragma unroll
    for (u32 q = 0; q < kPer; ++q) {
      c[q] = sh.cnt[tid * kPer + q];
      sum += c[q];
      most = c[q] > most ? c[q] : most;
    }
    u32 run = block_exclusive_scan<S::kThreads>(sum, sh.scan);
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
      const u32 x = __shfl_xor(most, o, kWave);
      most = x > most ? x : most;
    }
    if (lane == 0 && most) atomicMax(&sh.misc[6], most);
#pragma unroll
    for (u32 q = 0; q < kPer; ++q) {
      sh.cnt[tid * kPer + q] = run;
      run += c[q];
    }
  }
  __syncthreads();
  if (sh.misc[6] <= S::kBucketMax) {
    u32 slot[S::kItems];
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      slot[j] = 0;
      if (j * S::kThreads + tid < m) slot[j] = atomicAdd(&sh.cnt[b[j]], 1u);
    }
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      const u32 i = j * S::kThreads + tid;
      if (i < m) {
        sh.k[slot[j]] = k[j];
        sh.at[slot[j]] = static_cast<unsigned short>(i);
      }
    }
    __syncthreads();
    // cnt[b] is now the end of bucket b
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      const u32 i = j * S::kThreads + tid;
      if (i < m) {
        const u32 end = sh.cnt[b[j]];
        const u32 beg = b[j] ? sh.cnt[b[j] - 1] : 0u;
        const K x = k[j] & order;
        u32 rank = 0;
        for (u32 y = beg; y < end; ++y) {
          const K other = sh.k[y] & order;
          rank += (other < x || (other == x && sh.at[y] < i)) ? 1u : 0u;
        }
        slot[j] = beg + rank;
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      if (j * S::kThreads + tid < m) {
        sh.k[slot[j]] = k[j];
        sh.p[slot[j]] = p[j];
      }
    }
    __syncthreads();
    return;
  }
#pragma unroll
  for (int j = 0; j < S::kItems; ++j) {
    const u32 i = j * S::kThreads + tid;
    if (i < m) {
      sh.k[i] = k[j];
      sh.p[i] = p[j];
    }
  }
  digit_sort<S, K, P>(&sh, m, span);
}

// ------------------------------------------------------ runs of the LSM
// The payload of an update: its value, nothing for an erase.  In a mixed batch
// whose keys share the top bit (top <= bits - 9, so the top digit ends below
// it) the erase flag rides in that bit; else the payload is the update's
// position, and value and flag are gathered after the sort.
template <class T>
__device__ __forceinline__ bool update_stashed(int mode, u32 top) {
  return mode == lsm::kModeMixed && top + 9 <= static_cast<u32>(T::kBits);
}

template <class T>
struct UpdatePayload {
  const typename T::V *values;
  const u8 *flags;
  int mode;
  __device__ __forceinline__ typename T::V operator()(u64 idx,
                                                      typename T::K &key,
                                                      u32 top) const {
    if (mode == lsm::kModeErase) return 0;
    if (mode == lsm::kModeMixed) {
      if (!update_stashed<T>(mode, top)) return static_cast<typename T::V>(idx);
      key = (key & T::kLow) | (flags[idx] ? T::kTomb : typename T::K(0));
    }
    return values[idx];
  }
};

// Writes the sorted batch as a run: rows, radix directory and header.  The
// last of equal keys (the newest update) stays.
template <class T>
struct LsmEmit {
  using K = typename T::K;
  using V = typename T::V;
  const V *values;
  const u8 *flags;
  int mode;
  typename T::Row *out;
  lsm::RunMeta *meta;
  u32 *dir;
  u32 dir_bits;
  // set by begin() and rows()
  bool stashed;
  K high;
  u32 low, tombs;

  __device__ __forceinline__ void begin(const K *keys, u32 top) {
    stashed = update_stashed<T>(mode, top);
    high = stashed ? keys[0] & T::kTomb : K(0);
  }
  __device__ __forceinline__ K key(K x) const {
    return stashed ? (x & T::kLow) | high : x;
  }
  // Rows and directory entries of the sorted piece (sh.k, sh.p): bit j of keep =
  // element j * kThreads + t of thread t stays, rank(j) survivors of the piece
  // come before it.  Element i owns the directory entries of the buckets in
  // (bucket of element i - 1, its bucket].
  template <class S, class Rank>
  __device__ __forceinline__ void rows(typename S::Shared &sh, u32 m, u32 keep,
                                       const Rank &rank) {
    const u32 tid = threadIdx.x;
    const K *sk = sh.k;
    const V *sp = sh.p;
    const u32 base = static_cast<u32>(sh.base);
    low = tombs = 0;
    const u32 dshift = T::kBits - dir_bits;
    const bool gathered = mode == lsm::kModeMixed && !stashed;
    V val[S::kItems];
    u32 tomb = 0;
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      const u32 i = j * S::kThreads + tid;
      const bool kept = (keep >> j) & 1u;
      val[j] = kept ? sp[i] : V(0);
      if (kept && (mode == lsm::kModeErase || (stashed && (sk[i] & T::kTomb))))
        tomb |= 1u << j;
    }
    if (gathered) {  // all items' loads before the first row is written
#pragma unroll
      for (int j = 0; j < S::kItems; ++j) {
        if ((keep >> j) & 1u) {
          const u64 at = val[j];
          tomb |= flags[at] != 0 ? 1u << j : 0u;
          val[j] = values[at];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      const u32 i = j * S::kThreads + tid;
      const u32 before = base + rank(j);
      if (i >= m) continue;
      const K k = key(sk[i]);
      const u32 b1 = static_cast<u32>(k >> dshift);
      if (i > 0)
        for (u32 b = static_cast<u32>(key(sk[i - 1]) >> dshift) + 1; b <= b1;
             ++b)
          dir[b] = before;
      if ((keep >> j) & 1u) {
        const bool dead = (tomb >> j) & 1u;
        out[before] = T::make((k & T::kLow) | (dead ? T::kTomb : K(0)),
                              dead ? V(0) : val[j]);
        low += k < T::kTomb;
        tombs += dead;
      }
    }
  }
  // The directory entries between this piece's keys and its neighbours'
  // digits (bits below `shift` cleared), and the header: the first piece
  // writes the first bucket, the last one the count and the last bucket, the
  // first one that reaches the top key bit (or the last) the split.
  template <class S>
  __device__ __forceinline__ void edges(typename S::Shared &sh, u32 m,
                                        bool has_before, K before_key,
                                        bool has_after, K after_key,
                                        u32 shift) {
    const u32 tid = threadIdx.x;
    const u32 l = wave_sum_u32(low), t = wave_sum_u32(tombs);
    if (lane_id() == 0) {
      if (l) atomicAdd(&sh.misc[1], l);
      if (t) atomicAdd(&sh.misc[2], t);
    }
    __syncthreads();
    const u32 dshift = T::kBits - dir_bits;
    const K below = (K(1) << dshift) - 1;
    const K first = key(sh.k[0]), last = key(sh.k[m - 1]);
    const u32 row0 = static_cast<u32>(sh.base), row1 = row0 + sh.misc[3];
    // the first bucket that begins at or above the digit's first key
    auto bucket_from = [&](K x) {
      const K g = x >> shift << shift;
      return static_cast<u64>(g >> dshift) + ((g & below) != 0 ? 1 : 0);
    };
    if (has_before)
      for (u64 b = bucket_from(first) + tid; b <= u64(first >> dshift);
           b += S::kThreads)
        dir[b] = row0;
    if (has_after) {
      const u64 stop = bucket_from(after_key);
      for (u64 b = u64(last >> dshift) + 1 + tid; b < stop; b += S::kThreads)
        dir[b] = row1;
    }
    if (tid == 0) {
      if (!has_before) {
        meta->dir_bits = dir_bits;
        meta->lo_bucket = static_cast<u32>(first >> dshift);
        dir[first >> dshift] = 0;
      }
      if (!has_after) {
        meta->count = row1;
        meta->hi_bucket = static_cast<u32>(last >> dshift);
        dir[(last >> dshift) + 1] = row1;
      }
      if ((!has_before || before_key < T::kTomb) &&
          (last >= T::kTomb || !has_after))
        meta->split = row0 + sh.misc[1];
      if (sh.misc[2]) meta->tombs = 1;
      else if (!has_before && !has_after) meta->tombs = 0;
    }
  }
};

// --------------------------------------------------------- host launches
// The shape of a batch's pieces: 16 waves, as many keys as 160 KB of LDS take.
template <class K, class P>
using PieceShape = Shape<K, P, 1024, sizeof(K) + sizeof(P) <= 12 ? 8 : 6>;

// One workgroup per top digit (ticket order = key order).  direct: the batch is
// one piece, read from the input; else pk / pp hold it partitioned by its top
// digit (totals: the digits' keys), and nothing is done when a digit holds more
// than kCap.  status: a chained-scan word per digit.  Emit writes the run.
//
// A workgroup has a CU to itself (100 to 130 KB of LDS) and its time is its
// chain of steps: loads, the counting pass, slots, ranks, the offset over the
// digits before it, stores.  700,001 uniform 64-bit updates: 27 us.
template <class S, class K, class P, class Fn, class Emit>
__global__ __launch_bounds__(S::kThreads) void batch_local_kernel(
    InputSource<K, P, Fn> input, bool direct, u32 n, const K *__restrict__ pk,
    const P *__restrict__ pp, Plan *plan, const u32 *__restrict__ totals,
    u64 *status, Emit emit) {
  __shared__ typename S::Shared sh;
  __shared__ u32 s_ticket;
  const u32 tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  if (!direct && plan->largest > S::kCap) return;
  if (tid == 0) s_ticket = direct ? 0u : atomicAdd(&plan->ticket, 1u);
  __syncthreads();
  const u32 tile = __builtin_amdgcn_readfirstlane(s_ticket);
  // one piece: every bit orders it, nothing rides in a key
  const u32 top = direct ? 8 * sizeof(K) - 8 : plan->shift_top;
  emit.begin(input.keys, top);
  // bits that order the batch: the bits up to the top digit's
  const K order = top + 8 >= 8 * sizeof(K) ? ~K(0) : (K(1) << (top + 8)) - 1;
  u32 start = 0, m = n;
  if (!direct) {
    const u32 mine = tid < 256 ? totals[tid] : 0u;
    const u32 ex = block_exclusive_scan<S::kThreads>(mine, sh.scan);
    if (tid == tile) {
      sh.misc[0] = ex;
      sh.misc[7] = mine;
    }
    __syncthreads();
    start = __builtin_amdgcn_readfirstlane(sh.misc[0]);
    m = __builtin_amdgcn_readfirstlane(sh.misc[7]);
    if (m == 0) {
      if (tid == 0) store_relaxed(&status[tile], kFlagAggregate);
      return;
    }
  }
  {
    K k[S::kItems];
    P p[S::kItems];
#pragma unroll
    for (int j = 0; j < S::kItems; ++j) {
      const u32 i = j * S::kThreads + tid;
      k[j] = 0;
      p[j] = 0;
      if (i < m) {
        if (direct) {
          input.load(i, true, top, k[j], p[j]);
        } else {
          k[j] = pk[start + i];
          if (pp) p[j] = pp[start + i];
        }
      }
    }
    local_sort<S, K, P>(sh, k, p, m, order);
  }
  // a neighbour's key on either side: its digit bounds this piece
  const bool has_before = start > 0, has_after = start + m < n;
  const K before_key = has_before ? emit.key(pk[start - 1]) : K(0);
  const K after_key = has_after ? emit.key(pk[start + m]) : K(0);

  // ------------------------------------- survivors: count, offset, output
  u32 keep = 0;
#pragma unroll
  for (int j = 0; j < S::kItems; ++j) {
    const u32 i = j * S::kThreads + tid;
    const bool kj =
        i < m && (i + 1 == m || ((sh.k[i + 1] ^ sh.k[i]) & order) != 0);
    keep |= kj ? 1u << j : 0u;
    const u64 mj = ballot(kj);
    if (lane == 0) sh.off[j][wave] = popc64(mj);
  }
  __syncthreads();
  if (wave == 0) {
    // exclusive scan of the (item, wave) counts in element order
    constexpr u32 kAll = S::kItems * S::kWaves;
    u32 *flat = &sh.off[0][0];
    u32 carry = 0;
#pragma unroll
    for (u32 q = 0; q < (kAll + kWave - 1) / kWave; ++q) {
      const u32 e = q * kWave + lane;
      const u32 v = e < kAll ? flat[e] : 0u;
      const u32 inc = wave_inclusive_scan(v);
      if (e < kAll) flat[e] = carry + inc - v;
      carry += __shfl(inc, kWave - 1, kWave);
    }
    // every digit publishes its survivors without waiting; one round of
    // loads then gives the sum over the digits before this one
    u64 ex = 0;
    if (!direct) {
      if (lane == 0) store_relaxed(&status[tile], kFlagAggregate | carry);
      ex = lsm::segments_before(status, tile);
    }
    if (lane == 0) {
      sh.base = ex;
      sh.misc[3] = carry;
      sh.misc[1] = sh.misc[2] = 0;
    }
  }
  __syncthreads();
  emit.template rows<S>(sh, m, keep, [&](int j) {
    return sh.off[j][wave] + popc64(ballot((keep >> j) & 1u) & lanemask_lt());
  });
  emit.template edges<S>(sh, m, has_before, before_key, has_after, after_key,
                         top);
}

// Control words of a sort of n > kCap keys: [plan | status | the radix sort's
// own (cleared with them) | its finalize state] are cleared by the first
// launch; [top totals | tile counts | tile prefixes | tile spans] are written
// whole.
template <class K>
struct Layout {
  u64 status_at, radix_at, finalize_at, cleared;
  u64 totals_at, hist_at, prefix_at, span_at, words;
  u32 tiles, finalize_tiles;
  explicit Layout(u64 n) {
    tiles = rs::tiles_for(n);
    finalize_tiles = static_cast<u32>((n + lsm::kFinTile - 1) / lsm::kFinTile);
    status_at = kPlanWords;
    radix_at = status_at + 2 * 256;
    finalize_at = radix_at + rs::control_words(n, rs::passes_for<K>());
    cleared = finalize_at + 64 + 2 * u64(finalize_tiles);
    totals_at = cleared;
    hist_at = totals_at + 256;
    prefix_at = hist_at + u64(tiles) * rs::kRadix;
    span_at = prefix_at + u64(tiles) * rs::kRadix;
    words = span_at + 2 * u64(tiles);
  }
};

// Scratch of a batch of n > kCap keys (none is needed below): partitioned keys
// and values, or the radix sort's two copies of keys and positions; and
// Layout<K>(n).words control words.
template <class T>
struct Scratch {
  typename T::K *ka, *kb;
  typename T::V *vals;
  u32 *pa, *pb, *control;
};

// Sorts a batch of n >= 1 updates (32-bit ones: at most kCap) into the run that
// `emit` describes.
template <class T>
inline hipError_t admit_batch(const typename T::K *keys, u32 n,
                              const Scratch<T> &x, const LsmEmit<T> &emit,
                              hipStream_t s, int block) {
  using K = typename T::K;
  using V = typename T::V;
  using S = PieceShape<K, V>;
  using Fn = UpdatePayload<T>;
  const InputSource<K, V, Fn> input{keys,
                                    Fn{emit.values, emit.flags, emit.mode}};
  if (n <= S::kCap) {
    batch_local_kernel<S, K, V, Fn, LsmEmit<T>><<<1, S::kThreads, 0, s>>>(
        input, true, n, nullptr, nullptr, nullptr, nullptr, nullptr, emit);
    return hipGetLastError();
  }
  if constexpr (sizeof(K) == 4) {
    return hipErrorInvalidValue;  // (the segmented admission's)
  } else {
    const Layout<K> L(n);
    u32 *c = x.control;
    Plan *plan = reinterpret_cast<Plan *>(c);
    K *span = reinterpret_cast<K *>(c + L.span_at);
    lsm::seg_tile_hist_kernel<K><<<L.tiles, rs::kThreads, 0, s>>>(
        keys, n, c + L.hist_at, span, c, L.cleared,
        reinterpret_cast<u32 *>(emit.meta), lsm::kMetaWords, nullptr, 0);
    lsm::seg_tile_scan_kernel<K><<<rs::kRadix, rs::kThreads, 0, s>>>(
        keys, n, c + L.hist_at, span, L.tiles, c + L.prefix_at, c + L.totals_at,
        &plan->shift_top, &plan->largest);
    V *vals = emit.mode == lsm::kModeErase ? nullptr : x.vals;
    rs::PassPlan top{};
    top.shift_dev = &plan->shift_top;
    top.gate = {&plan->largest, S::kCap, false};
    top.digit_totals = c + L.totals_at;
    top.tile_prefix = c + L.prefix_at;
    rs::launch_source_pass<K, V>(rs::prefix_shape<K>(n, block), input, x.ka,
                                 vals, n, top, s);
    batch_local_kernel<S, K, V, Fn, LsmEmit<T>><<<256, S::kThreads, 0, s>>>(
        input, false, n, x.ka, vals, plan, c + L.totals_at,
        reinterpret_cast<u64 *>(c + L.status_at), emit);
    // the batches that do not fit
    const rs::Gate rest{&plan->largest, S::kCap, true};
    const hipError_t e =
        rs::sort_pairs_cleared<K>(keys, n, x.ka, x.pa, x.kb, x.pb,
                                  c + L.radix_at, s, block, rest);
    if (e != hipSuccess) return e;
    u32 *fin = c + L.finalize_at;
    lsm::finalize_batch_kernel<T><<<L.finalize_tiles, lsm::kFinThreads, 0, s>>>(
        x.ka, x.pa, n, emit.values, emit.flags, emit.mode, emit.out, emit.meta,
        emit.dir, emit.dir_bits, reinterpret_cast<u64 *>(fin + 64), fin, rest);
    return hipGetLastError();
  }
}

}  // namespace bs
}  // namespace gdict
