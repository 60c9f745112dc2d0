// Stable LSD radix sort of (key, u32 payload) pairs for gfx950, 32- and 64-bit
// keys.
//
// One global-histogram launch computes the 8-bit digit histograms in a single
// read of the keys; every digit pass is then ONE launch ("onesweep"): a tile of
// 4096 or 8192 keys is ranked in registers (a multisplit: digit_peers gives
// each lane the lanes holding the same digit), tiles chain their per-digit
// offsets through a decoupled look-back, and the tile is re-ordered in LDS so
// the global stores leave as contiguous runs per digit.  The first pass writes
// payload = input position, which is what the callers need for "newest wins" (a
// stable sort keeps equal keys in input order, so the last of a run of equal
// keys is the newest update), or takes the caller's payloads.
#pragma once

#include "device_utils.hpp"

namespace gdict {
namespace rs {

constexpr int kThreads = 256;
constexpr int kRadix = 256;
constexpr int kMaxPasses = 8;
constexpr int kWaves = kThreads / kWave;

template <class K>
constexpr int passes_for() {
  return static_cast<int>(sizeof(K));
}

// Whether a launch runs at all, decided on the device: a launch with a gate
// runs only if (*value > limit) == above (an earlier launch left *value).
struct Gate {
  const u32 *value;  // null: always
  u32 limit;
  bool above;
  __device__ __forceinline__ bool closed() const {
    return value && (*value > limit) != above;
  }
};

// Digit histograms.  A block counts 16 keys per thread per round in LDS
// (the 16 loads are issued together), then adds its counts into one of
// kHistRows partial rows (row = block % kHistRows), so at most
// blocks / kHistRows atomics meet on one address; scan_kernel sums the rows.
// (Folding the scan into the histogram's last block through a done counter
// was measured slower on MI355X: every block's fence and the atomics of all
// blocks on one counter cost more than the extra launch.)
constexpr int kHistItems = 16;
constexpr int kHistRows = 32;

inline u32 hist_blocks_for(u64 n) {
  const u64 b = (n + kThreads * kHistItems - 1) / (kThreads * kHistItems);
  return static_cast<u32>(b < 1 ? 1 : (b > 4096 ? 4096 : b));
}

// rows[kHistRows][kPasses][kRadix] (zeroed) += counts of digits
// first .. first + kPasses - 1, digit p = (key >> 8p) & 0xff, by workgroup
// `block` of `blocks`.
//
// Lanes that add to one LDS word wait for each other, so neighbouring lanes count
// in copies of their own: 65,536 64-bit keys, most of them five hot ones, 12.2 ->
// 7.7 us, uniform keys as before (15,000,001 of 32 bits 24 us).
template <class K, int kPasses>
__device__ __forceinline__ void histogram_block(const K *__restrict__ keys,
                                                u32 n, u32 first,
                                                u32 *__restrict__ rows,
                                                u32 block, u32 blocks) {
  constexpr int kCopies = 4;
  __shared__ u32 s_hist[kPasses][kRadix * kCopies];
  for (int i = threadIdx.x; i < kPasses * kRadix * kCopies; i += kThreads)
    (&s_hist[0][0])[i] = 0;
  __syncthreads();
  const u32 copy = threadIdx.x % kCopies;
  const u64 round = u64(kThreads) * kHistItems;
  for (u64 base = u64(block) * round; base < n; base += u64(blocks) * round) {
    K k[kHistItems];
#pragma unroll
    for (int j = 0; j < kHistItems; ++j) {
      const u64 i = base + u64(j) * kThreads + threadIdx.x;
      k[j] = i < n ? keys[i] : K(0);
    }
#pragma unroll
    for (int j = 0; j < kHistItems; ++j) {
      if (base + u64(j) * kThreads + threadIdx.x < n) {
#pragma unroll
        for (int p = 0; p < kPasses; ++p)
          atomicAdd(&s_hist[p][(static_cast<u32>(k[j] >> (8 * (first + p))) &
                                0xffu) * kCopies + copy],
                    1u);
      }
    }
  }
  __syncthreads();
  u32 *row = rows + u64(block % kHistRows) * kPasses * kRadix;
  for (int i = threadIdx.x; i < kPasses * kRadix; i += kThreads) {
    u32 c = 0;
#pragma unroll
    for (int q = 0; q < kCopies; ++q) c += (&s_hist[0][0])[i * kCopies + q];
    if (c) atomicAdd(&row[i], c);
  }
}

template <class K, int kPasses>
static __global__ __launch_bounds__(kThreads) void histogram_kernel(
    const K *__restrict__ keys, u32 n, u32 first, u32 *__restrict__ rows,
    Gate gate) {
  if (gate.closed()) return;
  histogram_block<K, kPasses>(keys, n, first, rows, blockIdx.x, gridDim.x);
}

// Sums the kHistRows partial rows of pass p and writes the exclusive scan over
// digits -> global digit offsets, by one workgroup.  constant[p] (nullable,
// zero before) = 1 when all n keys share the pass's digit.
__device__ __forceinline__ void scan_block(const u32 *__restrict__ rows,
                                           u32 passes, u32 p,
                                           u32 *__restrict__ offsets,
                                           u32 *constant, u32 n) {
  __shared__ u32 scratch[kRadix / kWave + 1];
  u32 c[kHistRows];
#pragma unroll
  for (int r = 0; r < kHistRows; ++r)
    c[r] = rows[(u64(r) * passes + p) * kRadix + threadIdx.x];
  u32 v = 0;
#pragma unroll
  for (int r = 0; r < kHistRows; ++r) v += c[r];
  offsets[p * kRadix + threadIdx.x] = block_exclusive_scan<kRadix>(v, scratch);
  if (constant && v == n) constant[p] = 1;
}

static __global__ __launch_bounds__(kRadix) void scan_kernel(
    const u32 *__restrict__ rows, u32 passes, u32 *__restrict__ offsets,
    Gate gate = Gate{}, u32 *constant = nullptr, u32 n = 0) {
  if (gate.closed()) return;
  scan_block(rows, passes, blockIdx.x, offsets, constant, n);
}

// Payload policies of a digit pass: payload(idx, valid, key, shift)
// returns the 32-bit payload of input element idx (and may rewrite key
// bits that no digit of the sort reads).
struct PayloadIn {  // the payload array of the previous pass
  const u32 *vals;
  template <class K>
  __device__ __forceinline__ u32 operator()(u64 idx, bool valid, K &,
                                            u32) const {
    return valid ? vals[idx] : 0u;
  }
};
struct PayloadPos {  // the input position
  template <class K>
  __device__ __forceinline__ u32 operator()(u64 idx, bool, K &, u32) const {
    return static_cast<u32>(idx);
  }
};

// Keys and payloads of a pass: src.load(idx, valid, shift, key, val).
template <class K, class Payload>
struct ArraySource {
  const K *keys;
  Payload payload;
  __device__ __forceinline__ void load(u64 idx, bool valid, u32 shift, K &key,
                                       u32 &val) const {
    key = valid ? keys[idx] : ~K(0);
    val = payload(idx, valid, key, shift);
  }
};

// One digit pass: the digit and where its keys go.
struct PassPlan {
  u32 shift;               // the digit's shift, or (not null)
  const u32 *shift_dev;    // where an earlier launch left it
  // Passes compiled with a gate (kGated) may not run: when it is closed, or
  // when pair (not null) says that this pass's and its partner's digits are
  // constant, so that the two would move nothing (passes 2q and 2q + 1 leave
  // the batch in the buffer that it came in).
  Gate gate;
  const u32 *pair;
  // the digits' starts, or their totals (scanned here)
  const u32 *digit_offsets, *digit_totals;
  // per-tile digit prefixes of the input (tile_prefix[d * tiles + t]: keys of
  // digit d in tiles before t): the tiles are then independent.  Without
  // them they chain their offsets: status (tiles * kRadix words) and *ticket
  // start at zero.
  const u32 *tile_prefix;
  u64 *status;
  u32 *ticket;
  u32 *dest;               // nullable: each input element's place
};

// Workgroups go to the 8 XCDs in turn: workgroup i's tile, such that each XCD
// takes consecutive tiles.
__device__ __forceinline__ u32 xcd_tile(u32 i, u32 tiles) {
  const u32 x = i % 8, each = tiles / 8, more = tiles % 8;
  return x * each + (x < more ? x : more) + i / 8;
}

// Tiles that a look-back reads at once.
constexpr u32 kLookBack = 4;

// kBlock threads x kItems keys per tile; threads below 256 own one digit each
// for the per-digit bookkeeping.
template <class K, class V, class Source, int kItems, int kBlock, bool kGated>
__global__ __launch_bounds__(kBlock) void onesweep_kernel(
    Source src, K *__restrict__ keys_out, V *__restrict__ vals_out, u32 n,
    PassPlan plan) {
  constexpr int kTile = kBlock * kItems;
  // (an ungated pass does not spend the loads on it: 2 us of 37 at 3 million
  // 64-bit keys)
  if constexpr (kGated) {
    if (plan.gate.closed()) return;
    if (plan.pair && plan.pair[0] && plan.pair[1]) return;
  }
  const u32 *tile_prefix = plan.tile_prefix;
  const u32 shift = plan.shift_dev ? *plan.shift_dev : plan.shift;
  constexpr int kBlockWaves = kBlock / kWave;
  __shared__ u32 s_tile;
  __shared__ u32 s_wave_hist[kBlockWaves][kRadix];
  __shared__ u32 s_global_base[kRadix];
  __shared__ u32 s_scan[kBlockWaves + 1];
  __shared__ K s_keys[kTile];
  __shared__ V s_vals[kTile];

  const u32 tid = threadIdx.x;
  const u32 lane = lane_id();
  const u32 wave = tid / kWave;
  if (tid == 0) s_tile = tile_prefix ? xcd_tile(blockIdx.x, gridDim.x)
                                   : atomicAdd(plan.ticket, 1u);
  for (int i = tid; i < kBlockWaves * kRadix; i += kBlock)
    (&s_wave_hist[0][0])[i] = 0;
  __syncthreads();
  const u32 tile = s_tile;
  const u32 base = tile * kTile;  // (below n, so nothing here overflows)
  const u32 count = n - base < u32(kTile) ? n - base : u32(kTile);
  // (loaded here, before the keys' latency, not where they are used)
  u32 digit_in = 0, prefix_in = 0;
  if (tid < kRadix) {
    digit_in = plan.digit_totals ? plan.digit_totals[tid]
                                 : plan.digit_offsets[tid];
    if (tile_prefix) prefix_in = tile_prefix[u64(tid) * gridDim.x + tile];
  }

  // Places behind the input's end hold a key of the highest digit: they rank
  // behind every key of the tile and are not written.
  K key[kItems];
  V val[kItems];
  u32 rank[kItems];
  const u32 wave_at = wave * (kWave * kItems) + lane;
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const u32 i = wave_at + j * kWave;
    src.load(base + i, i < count, shift, key[j], val[j]);
  }

  // Wave-local stable ranking (item-major, then lane order == input order).
  u32 *my_hist = s_wave_hist[wave];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const u32 d = static_cast<u32>(key[j] >> shift) & 0xffu;
    rank[j] = count_peers(&my_hist[d], digit_peers(d));
  }
  __syncthreads();

  // Per digit: wave prefixes, tile total, global base via look-back.
  const u32 d = tid;
  u32 total = 0;
  u32 wave_start[kBlockWaves];
  u64 exclusive = 0;
  if (tid < kRadix) {
#pragma unroll
    for (int w = 0; w < kBlockWaves; ++w) {
      wave_start[w] = total;
      total += s_wave_hist[w][d];
    }
    // look-back: every digit owns one column of the status array
    u64 *column = plan.status;  // status[t * kRadix + d]
    if (tile_prefix) {
      exclusive = prefix_in;
    } else if (tile == 0) {
      store_relaxed(&column[d], kFlagPrefix | total);
    } else {
      store_relaxed(&column[u64(tile) * kRadix + d], kFlagAggregate | total);
      u32 t = tile;  // the tiles from t on are summed
      bool open = true;
      while (open) {
        u64 word[kLookBack];
#pragma unroll
        for (u32 q = 0; q < kLookBack; ++q)
          word[q] = q < t ? load_relaxed(&column[u64(t - 1 - q) * kRadix + d])
                          : kFlagPrefix;
        u32 ready = 0;
        bool next = true;  // every word so far was there, none a prefix
#pragma unroll
        for (u32 q = 0; q < kLookBack; ++q) {
          next = next && (word[q] >> kFlagShift) != 0;
          if (next) {
            exclusive += word[q] & kValueMask;
            ++ready;
            if (word[q] & kFlagPrefix) next = open = false;
          }
        }
        t = ready < t ? t - ready : 0;
        if (ready == 0) __builtin_amdgcn_s_sleep(4);
      }
      store_relaxed(&column[u64(tile) * kRadix + d],
                    kFlagPrefix | (exclusive + total));
    }
  }
  const u32 block_start = block_exclusive_scan<kBlock>(total, s_scan);
  // the digit's start: given, or a scan of the digit totals
  u32 digit_start = 0;
  if (plan.digit_totals) {
    __shared__ u32 s_scan2[kBlockWaves + 1];
    digit_start = block_exclusive_scan<kBlock>(digit_in, s_scan2);
  } else {
    digit_start = digit_in;
  }
  if (tid < kRadix) {
#pragma unroll
    for (int w = 0; w < kBlockWaves; ++w)
      s_wave_hist[w][d] = block_start + wave_start[w];
    s_global_base[d] = digit_start + static_cast<u32>(exclusive) - block_start;
  }
  __syncthreads();

  // Scatter into LDS in digit order.
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const u32 dj = static_cast<u32>(key[j] >> shift) & 0xffu;
    rank[j] += my_hist[dj];
    s_keys[rank[j]] = key[j];
    s_vals[rank[j]] = val[j];
  }
  // destination of each input element, written in input order
  if (plan.dest) {
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      const u32 i = wave_at + j * kWave;
      const u32 dj = static_cast<u32>(key[j] >> shift) & 0xffu;
      if (i < count) plan.dest[base + i] = s_global_base[dj] + rank[j];
    }
  }
  __syncthreads();

  // all LDS reads before the stores
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const u32 i = j * kBlock + tid;
    key[j] = s_keys[i];
    val[j] = s_vals[i];
    rank[j] = s_global_base[static_cast<u32>(key[j] >> shift) & 0xffu] + i;
  }
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    if (j * kBlock + tid < count) {
      keys_out[rank[j]] = key[j];
      if (vals_out) vals_out[rank[j]] = val[j];
    }
  }
}

// Clears a[0..na) and b[0..nb) in one launch.
static __global__ void zero_two_kernel(u32 *a, u64 na, u32 *b, u64 nb) {
  const u64 stride = u64(gridDim.x) * blockDim.x;
  for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < na + nb;
       i += stride) {
    if (i < na) a[i] = 0;
    else b[i - na] = 0;
  }
}

static __global__ void zero_u32_kernel(u32 *p, u64 n) {
  const u64 stride = u64(gridDim.x) * blockDim.x;
  for (u64 i = u64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    p[i] = 0;
}


// A pass's workgroups: `block` threads with `items` keys each, a tile per
// workgroup.
struct PassShape {
  int block, items;
  u32 tiles;
};

inline u32 tiles_for(u64 n) {
  const u64 tile = 4096;
  return static_cast<u32>((n + tile - 1) / tile);
}

// Passes over tiles of 4096 keys whose digit prefixes are known: a tile per CU
// wants many waves (up to 2^20 keys), several tiles a CU want several
// workgroups (3,000,017 32-bit keys: 20.6 us in workgroups of 1024, 17.0 of
// 512, 14.9 of 256; 64-bit keys 22.1, 18.9 and 20.4).  block != 0: as told.
template <class K>
inline PassShape prefix_shape(u64 n, int block = 0) {
  const int b = block ? block
                : n <= (u64(1) << 20) ? 1024 : sizeof(K) == 8 ? 512 : 256;
  return {b, 4096 / b, tiles_for(n)};
}

// Passes whose tiles chain their offsets: the chain costs some 15 ns a tile,
// half of a pass's time, so the tiles are 8192 keys where they still fill the
// chip (8,388,608 32-bit keys: 73 us with tiles of 4096, 61 so; 1,500,003
// 64-bit keys: 27 and 21; 300,000: 13.7 and 15.5) and where the LDS takes them.
template <class K, class V>
constexpr bool kWideTiles = sizeof(K) + sizeof(V) <= 12;
template <class K, class V>
inline PassShape chained_shape(u64 n, int block = 0) {
  if (block) return {block, 4096 / block, tiles_for(n)};
  if (n < 600000 || !kWideTiles<K, V>) return {1024, 4, tiles_for(n)};
  return {1024, 8, static_cast<u32>((n + 8191) / 8192)};
}

// Workspace (u32 words) of a sort of n keys in `passes` digit passes, not
// counting the ping-pong buffers:
//   rows    [kHistRows][passes][256]     partial histograms
//   offsets [passes][256]                global digit offsets
//   tickets [64]                         tile tickets, one per pass
//   status  u64 [passes][tiles][256]     look-back words
// Everything but the offsets starts at zero (one clearing launch).
struct Control {
  u32 *rows, *offsets, *tickets;
  u64 *status;
};

inline u64 control_words(u64 n, int passes = 4) {
  return u64(kHistRows) * passes * kRadix + u64(passes) * kRadix + 64 +
         2ull * passes * u64(tiles_for(n)) * kRadix;
}

inline Control control_layout(u32 *control, int passes) {
  Control c;
  c.rows = control;
  c.offsets = control + u64(kHistRows) * passes * kRadix;
  c.tickets = c.offsets + passes * kRadix;
  c.status = reinterpret_cast<u64 *>(c.tickets + 64);  // even word offset
  return c;
}

// Clears the control words (at least control_words(n, passes); callers may
// extend the region with their own state) and an optional second region,
// in one launch.
inline void clear_control(u32 *control, u64 words, hipStream_t stream,
                          u32 *extra = nullptr, u64 extra_words = 0) {
  const u64 total = words + extra_words;
  zero_two_kernel<<<static_cast<u32>(std::min<u64>((total + 255) / 256, 4096)),
                    256, 0, stream>>>(control, words, extra, extra_words);
}

template <bool kGated, class K, class V, class Source>
inline void launch_shaped_pass(const PassShape &h, const Source &src, K *dst_k,
                               V *dst_v, u32 n, const PassPlan &plan,
                               hipStream_t stream) {
  if constexpr (kWideTiles<K, V>) {  // tiles of 8192 keys
    if (h.block == 1024 && h.items == 8) {
      onesweep_kernel<K, V, Source, 8, 1024, kGated>
          <<<h.tiles, 1024, 0, stream>>>(src, dst_k, dst_v, n, plan);
      return;
    }
  }
  const u32 tiles = tiles_for(n);  // the others have 4096
  if (h.block == 1024) {
    onesweep_kernel<K, V, Source, 4, 1024, kGated>
        <<<tiles, 1024, 0, stream>>>(src, dst_k, dst_v, n, plan);
  } else if (h.block == 512) {
    onesweep_kernel<K, V, Source, 8, 512, kGated>
        <<<tiles, 512, 0, stream>>>(src, dst_k, dst_v, n, plan);
  } else {
    onesweep_kernel<K, V, Source, 16, 256, kGated>
        <<<tiles, 256, 0, stream>>>(src, dst_k, dst_v, n, plan);
  }
}

template <class K, class V, class Source>
inline void launch_source_pass(const PassShape &shape, const Source &src,
                               K *dst_k, V *dst_v, u32 n, const PassPlan &plan,
                               hipStream_t stream) {
  if (plan.gate.value || plan.pair)
    launch_shaped_pass<true>(shape, src, dst_k, dst_v, n, plan, stream);
  else
    launch_shaped_pass<false>(shape, src, dst_k, dst_v, n, plan, stream);
}

// A pass over an array of keys with 32-bit payloads.  With tile_prefix,
// `offsets` holds the digit totals, else the digits' starts.
template <class K, class Payload>
inline void launch_pass(const PassShape &shape, const K *src_k,
                        Payload payload, K *dst_k, u32 *dst_v, u32 n,
                        u32 shift, const u32 *offsets, u64 *status,
                        u32 *ticket, hipStream_t stream,
                        u32 *dest = nullptr,
                        const u32 *shift_dev = nullptr,
                        const u32 *tile_prefix = nullptr,
                        const Gate &gate = Gate{},
                        const u32 *pair = nullptr) {
  PassPlan plan{};
  plan.shift = shift;
  plan.shift_dev = shift_dev;
  plan.gate = gate;
  plan.pair = pair;
  (tile_prefix ? plan.digit_totals : plan.digit_offsets) = offsets;
  plan.tile_prefix = tile_prefix;
  plan.status = status;
  plan.ticket = ticket;
  plan.dest = dest;
  launch_source_pass<K, u32>(shape,
                             ArraySource<K, Payload>{src_k, payload}, dst_k,
                             dst_v, n, plan, stream);
}

// Passes from .. to - 1 of sort_pairs below, behind its clearing and counting
// launches.  constant: nullable, see scan_block; pairs of passes over constant
// digits are then skipped (64-bit keys of a narrow range, and behind a gate), but
// not the first pair, which reads the input.
template <class K>
inline hipError_t sort_passes(const K *keys_in, u32 n, K *keys_a, u32 *vals_a,
                              K *keys_b, u32 *vals_b, u32 *control,
                              hipStream_t stream, int block, const Gate &gate,
                              const u32 *constant, const u32 *vals_in,
                              int from = 0, int to = passes_for<K>()) {
  constexpr int kPasses = passes_for<K>();
  const PassShape shape = chained_shape<K, u32>(n, block);
  const Control c = control_layout(control, kPasses);
  u32 *tickets = c.tickets;
  u64 *status = c.status;
  const u32 *offsets = c.offsets;
  const K *src_k = keys_in;
  const u32 *src_v = vals_in;
  K *dst_k = keys_b;
  u32 *dst_v = vals_b;
  for (int p = 0; p < to; ++p) {
    u64 *pass_status = status + u64(p) * tiles_for(n) * kRadix;
    if (p < from) {
      // an earlier call's
    } else if (p == 0 && !vals_in) {
      launch_pass<K>(shape, src_k, PayloadPos{}, dst_k, dst_v, n, 0,
                     offsets, pass_status, tickets, stream, nullptr, nullptr,
                     nullptr, gate);
    } else {
      launch_pass<K>(shape, src_k, PayloadIn{src_v}, dst_k, dst_v, n,
                     8u * p, offsets + p * kRadix, pass_status, tickets + p,
                     stream, nullptr, nullptr, nullptr, gate,
                     constant && p >= 2 ? constant + (p & ~1) : nullptr);
    }
    src_k = dst_k;
    src_v = dst_v;
    if (dst_k == keys_b) {
      dst_k = keys_a;
      dst_v = vals_a;
    } else {
      dst_k = keys_b;
      dst_v = vals_b;
    }
  }
  return hipGetLastError();
}

// sort_pairs below, without its clearing launch and behind a gate.
template <class K>
inline hipError_t sort_pairs_cleared(const K *keys_in, u32 n, K *keys_a,
                                     u32 *vals_a, K *keys_b, u32 *vals_b,
                                     u32 *control, hipStream_t stream,
                                     int block, const Gate &gate,
                                     const u32 *vals_in = nullptr) {
  constexpr int kPasses = passes_for<K>();
  const Control c = control_layout(control, kPasses);
  u32 *constant = gate.value || kPasses > 4 ? c.tickets + 32 : nullptr;
  histogram_kernel<K, kPasses><<<hist_blocks_for(n), kThreads, 0, stream>>>(
      keys_in, n, 0, c.rows, gate);
  scan_kernel<<<kPasses, kRadix, 0, stream>>>(c.rows, kPasses, c.offsets, gate,
                                              constant, n);
  return sort_passes<K>(keys_in, n, keys_a, vals_a, keys_b, vals_b, control,
                        stream, block, gate, constant, vals_in);
}

// Sorts n (key, position) pairs stably.  keys_in is read only; the sorted
// keys and positions end in (keys_a, vals_a) (an even number of passes).
// keys_b/vals_b are scratch.  `control` holds control_words(n, passes) u32
// words.  All launches go to `stream`.
// clear_words (0 = control_words(n, passes)) words of `control` and
// extra[0..extra_words) are cleared by the first launch, so callers can
// place zero-initialised state of their own behind the sort's.  vals_in
// (nullable): payloads to carry instead of the positions.
template <class K>
inline hipError_t sort_pairs(const K *keys_in, u32 n, K *keys_a, u32 *vals_a,
                             K *keys_b, u32 *vals_b, u32 *control,
                             hipStream_t stream, int block = 0,
                             u64 clear_words = 0, u32 *extra = nullptr,
                             u64 extra_words = 0,
                             const u32 *vals_in = nullptr) {
  if (n == 0) return hipSuccess;
  clear_control(control,
                clear_words ? clear_words
                            : control_words(n, passes_for<K>()),
                stream, extra, extra_words);
  return sort_pairs_cleared<K>(keys_in, n, keys_a, vals_a, keys_b, vals_b,
                               control, stream, block, Gate{}, vals_in);
}

}  // namespace rs
}  // namespace gdict
