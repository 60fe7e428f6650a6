// Stable LSD radix sort of 64-bit keys by bits [begin_bit, end_bit), written
// for the index builds: from a few thousand to a few hundred million keys,
// sorted by 12-45 bits.
//
// Each digit pass is three launches, reduce-then-scan:
//   count   one workgroup per tile of THREADS * ITEMS keys: the tile's digit
//           histogram in LDS, stored digit-major (counts[d * tiles + t]);
//   scan    one workgroup per digit: exclusive sum over the tiles, in place,
//           and the digit's total;
//   scatter one workgroup per tile: each key's stable rank among the tile's
//           keys of its digit (ballot-matched per wave, waves in order), the
//           tile's keys regrouped by digit in LDS, then written out so that
//           consecutive lanes store consecutive positions of a digit's run.
// No look-back, no global atomics, nothing to clear between calls. The first
// pass reads its keys through a functor, so a caller whose keys are a function
// of its own arrays (an edge list) never writes and reads back an unsorted copy.
//
// What bounds it: a pass reads the keys twice and writes them once; with 8-bit
// digits at 31M keys the scatter runs at 4.5 TB/s of the 5.1 TB/s a copy
// reaches. More digits per pass split a tile's output into shorter runs: at
// 31M keys a scatter takes 110 us with 8-bit digits, 131 with 9 and 217 with
// 11, so two 11-bit passes lose to three of 8 bits (686 against 505 us).
// The count pass keeps several copies of each bin (Replicas): the last digit
// of the power-law graphs' ids is so skewed that a wave's LDS atomics met in
// one bin and serialised (31M keys: last count 107 -> 36 us, sort 563 -> 505;
// 210M keys: 697 -> 370 us, sort 4.63 -> 4.33 ms).
#pragma once

#include <algorithm>
#include <cstdint>

#include "bf_common.h"

namespace bf {
namespace sort {

constexpr int kThreads = 256;   // of the scan kernel

// Digit width: the pass count and the equal split of the bits over the passes
// with the least total cost, a pass of R-bit digits costing about kPassCost[R]
// of an 8-bit one (6M keys: 39, 41, 47, 52 us for 7 to 10 bits; 11-bit passes
// cost 1.75 and are never taken). 20 bits: two 10-bit passes, 104 us against
// 124 for three of 8; 21 bits: three 7-bit passes, 141 us against 152 (7.5M keys).
// Tile: small sorts are bound by latency and want many short tiles (14K keys:
// 18 us with 1024-key tiles, 31 with 4096), large ones long runs per digit
// (210M keys of 9-bit digits: 8192-key tiles of 256 threads 4.33 ms, 4096-key
// ones a quarter slower; 12288 keys leave one wave per SIMD). Eight waves of
// 8 keys per lane are best from 2M to 16M keys (7.5M, 8 bits: 152 us against
// 156 for four waves of 16 keys; at 31M keys 510 against 505).
// Both passes map workgroups to tiles XCD by XCD (xcd_slot), so the tiles
// that share a line of the digit-major count array meet in one L2: the
// scatter pass at 210M keys went from 1.18 to 1.03 ms with it.
constexpr int kMinRadix = 6, kMaxRadix = 10;
constexpr float kPassCost[kMaxRadix + 1] = {0, 0, 0, 0, 0, 0, 0.90f, 0.92f, 1.0f, 1.13f, 1.27f};

// The sizes past which make_plan takes larger tiles. Just past one the tiles, and with them the counts' array, are
// half as many: a plan's workspace does not grow steadily with n (workspace_bytes_max).
constexpr int64_t kTileSteps[] = {int64_t(1) << 16, int64_t(1) << 21, int64_t(1) << 22, int64_t(1) << 24,
                                  int64_t(1) << 26};

struct Tile {
  int threads, items;
  int64_t count(int64_t n) const {
    const int64_t keys = int64_t(threads) * items;
    return (n + keys - 1) / keys;
  }
};

inline Tile tile_for(int64_t n, int radix) {
  if (n <= kTileSteps[0] && radix <= 8) return {256, 4};
  if (n <= kTileSteps[1]) return {512, 4};
  if (n <= kTileSteps[radix == 10 ? 2 : 3]) return {512, 8};
  if (radix == 10) return {512, 16};
  return {256, radix == 9 && n > kTileSteps[4] ? 32 : 16};
}

struct Plan {
  int radix;
  int threads;
  int items;
  int passes;
  int64_t tiles;
};

inline Plan make_plan(int64_t n, int bits) {
  Plan p{};
  float best = 0.f;
  p.radix = kMinRadix;
  for (int passes = (bits + kMaxRadix - 1) / kMaxRadix; passes > 0 && passes <= (bits + kMinRadix - 1) / kMinRadix;
       ++passes) {
    const int r = (bits + passes - 1) / passes;
    const int radix = r < kMinRadix ? kMinRadix : r;
    const float cost = float(passes) * kPassCost[radix];
    if (p.passes == 0 || cost < best) {
      best = cost;
      p.passes = passes;
      p.radix = radix;
    }
  }
  const Tile t = tile_for(n, p.radix);
  p.threads = t.threads;
  p.items = t.items;
  p.tiles = t.count(n);
  return p;
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// The keys to sort: cap, or, with a device count, *n_dev - n_sub clamped to [0, cap] (the buffers and
// the grids are sized for cap; the tiles past the count hold nothing).
__device__ __forceinline__ int64_t live_count(int64_t cap, const int64_t* n_dev, int64_t n_sub) {
  if (!n_dev) return cap;
  const int64_t n = *n_dev - n_sub;
  return n < 0 ? 0 : (n > cap ? cap : n);
}

// The second key buffer, the per-tile counts and the digit totals.
inline size_t buffer_bytes(int64_t n, int radix, int64_t tiles) {
  const size_t digits = size_t(1) << radix;
  return align256(size_t(n > 0 ? n : 1) * 8) + align256(size_t(tiles > 0 ? tiles : 1) * digits * 4) +
         align256(digits * 4);
}

// Workspace of make_plan(n, bits).
inline size_t workspace_bytes(int64_t n, int bits) {
  const Plan p = make_plan(n, bits);
  return buffer_bytes(n, p.radix, p.tiles);
}

// The most that any sort of up to n keys needs, by any bits: a caller that knows its keys only within a capacity
// (an index's entries less the token's) sizes its workspace so.
inline size_t workspace_bytes_max(int64_t n) {
  size_t most = 0;
  for (int radix = kMinRadix; radix <= kMaxRadix; ++radix) {
    const auto at = [&](int64_t m) { most = std::max(most, buffer_bytes(m, radix, tile_for(m, radix).count(m))); };
    at(n);
    for (const int64_t step : kTileSteps)
      if (step < n) at(step);
  }
  return most;
}

// block-wide exclusive scan of one value per thread; *total gets the sum
template <int THREADS = kThreads>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* tmp /*[THREADS / 64]*/, uint32_t* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) tmp[w] = x;
  __syncthreads();
  uint32_t wbase = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < THREADS / 64; ++i) {
    const uint32_t t = tmp[i];
    if (i < w) wbase += t;
    tot += t;
  }
  __syncthreads();
  *total = tot;
  return wbase + x - v;
}

// A pass's keys by position: operator() in the count pass, last() in the scatter pass, which reads them for
// the last time. Stored keys serve every pass but the first of a sort whose caller brings its own functor.
struct StoredKeys {
  const uint64_t* keys;
  __device__ __forceinline__ uint64_t operator()(int64_t i) const { return keys[i]; }
  __device__ __forceinline__ uint64_t last(int64_t i) const { return __builtin_nontemporal_load(keys + i); }
};

// Copies of each bin in the count pass's LDS histogram: a lane adds to copy lane % kReplicas, which sits in a
// bank of its own.
template <int R>
struct Replicas {
  static constexpr int k = R <= 8 ? 16 : R == 9 ? 8 : 4;
};

template <int R, int ITEMS, int THREADS, typename Load>
__global__ __launch_bounds__(THREADS) void radix_count_kernel(Load in, int64_t cap,
                                                              const int64_t* __restrict__ n_dev, int64_t n_sub,
                                                              int shift, uint32_t mask, int64_t tiles,
                                                              uint32_t* __restrict__ counts) {
  constexpr int B = 1 << R;
  constexpr int K = Replicas<R>::k;
  constexpr int64_t TILE = int64_t(THREADS) * ITEMS;
  const int64_t n = live_count(cap, n_dev, n_sub);
  __shared__ uint32_t h[B * K];
  for (int i = threadIdx.x; i < B * K; i += THREADS) h[i] = 0;
  __syncthreads();
  const int rep = threadIdx.x & (K - 1);
  const int64_t tile = xcd_slot(blockIdx.x, gridDim.x);   // the tiles sharing a counts line on one XCD
  const int64_t t0 = tile * TILE;
  uint64_t key[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int64_t pos = t0 + i * THREADS + threadIdx.x;
    key[i] = pos < n ? in(pos) : 0;
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int64_t pos = t0 + i * THREADS + threadIdx.x;
    if (pos < n) atomicAdd(&h[(uint32_t(key[i] >> shift) & mask) * K + rep], 1u);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < B; d += THREADS) {
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) s += h[d * K + ((k + d) & (K - 1))];   // the lanes' reads in different banks
    counts[int64_t(d) * tiles + tile] = s;
  }
}

static __global__ __launch_bounds__(kThreads) void radix_scan_kernel(uint32_t* __restrict__ counts, int64_t tiles,
                                                              uint32_t* __restrict__ totals) {
  __shared__ uint32_t tmp[kThreads / 64];
  uint32_t* row = counts + int64_t(blockIdx.x) * tiles;
  uint32_t carry = 0;
  for (int64_t base = 0; base < tiles; base += kThreads * 4) {
    uint32_t v[4], s = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t t = base + threadIdx.x * 4 + u;
      v[u] = t < tiles ? row[t] : 0;
      s += v[u];
    }
    uint32_t tot;
    uint32_t e = block_excl_scan(s, tmp, &tot) + carry;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t t = base + threadIdx.x * 4 + u;
      if (t < tiles) row[t] = e;
      e += v[u];
    }
    carry += tot;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Keys of a tile sit wave-striped: wave w holds positions [w * 64 * ITEMS, (w + 1) * 64 * ITEMS) of the
// tile, item i of lane l at offset i * 64 + l, so ranking items in order and lanes in order within a wave,
// and waves in order, follows the input order (the sort is stable). The waves' running digit counts and the
// regrouped keys share one LDS buffer: a key's place in the tile is in a register before the keys go in.
template <int R, int ITEMS, int THREADS, typename Load>
__global__ __launch_bounds__(THREADS) void radix_scatter_kernel(Load in, uint64_t* __restrict__ out, int64_t cap,
                                                                const int64_t* __restrict__ n_dev, int64_t n_sub,
                                                                int shift, uint32_t mask, int64_t tiles,
                                                                const uint32_t* __restrict__ prefix,
                                                                const uint32_t* __restrict__ totals) {
  constexpr int B = 1 << R;
  constexpr int W = THREADS / 64;
  constexpr int DPT = B > THREADS ? B / THREADS : 1;   // digits per thread
  constexpr int64_t TILE = int64_t(THREADS) * ITEMS;
  static_assert(TILE <= 65536 / 2, "places in a tile fit 16 bits");
  const int64_t n = live_count(cap, n_dev, n_sub);
  const int64_t tile = xcd_slot(blockIdx.x, gridDim.x);   // as in radix_count_kernel
  if (tile * TILE >= n) return;   // a tile past the count (uniform over the block)
  constexpr size_t kCntBytes = size_t(W) * B * sizeof(uint16_t), kKeyBytes = size_t(TILE) * sizeof(uint64_t);
  __shared__ __align__(16) unsigned char buf[kCntBytes > kKeyBytes ? kCntBytes : kKeyBytes];
  __shared__ uint32_t s_scan[W];
  __shared__ uint16_t dstart[B];          // the tile's first LDS slot of each digit
  __shared__ int32_t gofs[B];             // output position of LDS slot j of digit d: gofs[d] + j
  uint16_t* const wcnt = reinterpret_cast<uint16_t*>(buf);   // per wave: counts, then offsets over the waves
  uint64_t* const skeys = reinterpret_cast<uint64_t*>(buf);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int i = tid; i < W * B / 2; i += THREADS) reinterpret_cast<uint32_t*>(buf)[i] = 0;
  const int64_t t0 = tile * TILE + int64_t(w) * (64 * ITEMS) + lane;
  uint64_t key[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const int64_t pos = t0 + i * 64;
    key[i] = pos < n ? in.last(pos) : 0;
  }
  uint32_t tv[DPT], pv[DPT], tsum = 0;
#pragma unroll
  for (int j = 0; j < DPT; ++j) {
    const int d = tid * DPT + j;
    tv[j] = d < B ? totals[d] : 0;
    pv[j] = d < B ? prefix[int64_t(d) * tiles + tile] : 0;
    tsum += tv[j];
  }
  __syncthreads();
  const uint64_t below = (uint64_t(1) << lane) - 1;
  uint16_t* const wc = wcnt + w * B;
  uint32_t place[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const bool valid = t0 + i * 64 < n;
    const uint32_t d = uint32_t(key[i] >> shift) & mask;
    // the lanes holding the same digit: R ballots narrow the valid lanes down
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < R; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const uint32_t before = __popcll(peers & below);
    const uint32_t c = valid ? wc[d] : 0u;
    place[i] = c + before;
    // the lowest lane of each digit advances its wave's count (one writer per address)
    if (valid && before == 0) wc[d] = uint16_t(c + uint32_t(__popcll(peers)));
  }
  __syncthreads();
  uint32_t tot[DPT], lsum = 0;
#pragma unroll
  for (int j = 0; j < DPT; ++j) {
    const int d = tid * DPT + j;
    uint32_t s = 0;
    if (d < B) {
#pragma unroll
      for (int ww = 0; ww < W; ++ww) {
        const uint32_t x = wcnt[ww * B + d];
        wcnt[ww * B + d] = uint16_t(s);
        s += x;
      }
    }
    tot[j] = s;
    lsum += s;
  }
  uint32_t total, gtotal;
  uint32_t ls = block_excl_scan<THREADS>(lsum, s_scan, &total);
  uint32_t gs = block_excl_scan<THREADS>(tsum, s_scan, &gtotal);
#pragma unroll
  for (int j = 0; j < DPT; ++j) {
    const int d = tid * DPT + j;
    if (d < B) {
      dstart[d] = uint16_t(ls);
      gofs[d] = int32_t(gs + pv[j]) - int32_t(ls);
    }
    ls += tot[j];
    gs += tv[j];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t d = uint32_t(key[i] >> shift) & mask;
    place[i] += uint32_t(dstart[d]) + wc[d];
  }
  __syncthreads();                        // the counts are spent: the buffer takes the keys
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    if (t0 + i * 64 < n) skeys[place[i]] = key[i];
  __syncthreads();
  const int cnt = int(total);
  for (int j = tid; j < cnt; j += THREADS) {
    const uint64_t k = skeys[j];
    const int64_t o = int64_t(gofs[uint32_t(k >> shift) & mask]) + j;
    if (o >= 0 && o < n) out[o] = k;
  }
}

// The buffers and the key count of a sort, as its passes take them.
struct Sort {
  uint64_t* out;
  uint64_t* alt;
  int64_t n;
  const int64_t* n_dev;
  int64_t n_sub;
  int begin_bit, end_bit;
  uint32_t* counts;
  uint32_t* totals;
};

template <int R, int ITEMS, int THREADS, typename Load>
int run_pass(const Plan& p, int pass, Load src, const Sort& s, hipStream_t st) {
  // the last pass writes `out`: pass k writes out when passes - 1 - k is even, alt otherwise
  uint64_t* dst = (p.passes - 1 - pass) % 2 == 0 ? s.out : s.alt;
  const int shift = s.begin_bit + pass * R;
  const int bits = s.end_bit - shift < R ? s.end_bit - shift : R;
  const uint32_t mask = (1u << bits) - 1;
  BF_LAUNCH("radix_count_kernel", (radix_count_kernel<R, ITEMS, THREADS, Load>), dim3(unsigned(p.tiles)),
            dim3(THREADS), 0, st, src, s.n, s.n_dev, s.n_sub, shift, mask, p.tiles, s.counts);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("radix_scan_kernel", radix_scan_kernel, dim3(1u << R), dim3(kThreads), 0, st, s.counts, p.tiles, s.totals);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("radix_scatter_kernel", (radix_scatter_kernel<R, ITEMS, THREADS, Load>), dim3(unsigned(p.tiles)),
            dim3(THREADS), 0, st, src, dst, s.n, s.n_dev, s.n_sub, shift, mask, p.tiles, s.counts, s.totals);
  BF_CHECK_LAUNCH();
  return BF_OK;
}

template <int R, int ITEMS, int THREADS, typename Load>
int run_passes(const Plan& p, Load in, const Sort& s, hipStream_t st) {
  BF_CHECK_OK((run_pass<R, ITEMS, THREADS>(p, 0, in, s, st)));
  for (int pass = 1; pass < p.passes; ++pass)
    BF_CHECK_OK((run_pass<R, ITEMS, THREADS>(p, pass, StoredKeys{(p.passes - pass) % 2 == 0 ? s.out : s.alt}, s, st)));
  return BF_OK;
}

template <int R, typename Load>
int run_plan(const Plan& p, Load in, const Sort& s, hipStream_t st) {
  if constexpr (R <= 8)
    if (p.threads == 256 && p.items == 4) return run_passes<R, 4, 256>(p, in, s, st);
  if (p.threads == 512) {
    if (p.items == 4) return run_passes<R, 4, 512>(p, in, s, st);
    if (p.items == 8) return run_passes<R, 8, 512>(p, in, s, st);
    if constexpr (R == 10) return run_passes<R, 16, 512>(p, in, s, st);
  }
  if constexpr (R == 9)
    if (p.items == 32) return run_passes<R, 32, 256>(p, in, s, st);
  if constexpr (R <= 9)
    return run_passes<R, 16, 256>(p, in, s, st);
  else
    return BF_ERR_INVALID;   // make_plan gives 10-bit digits eight waves
}

// Sorts the n keys in(0) .. in(n - 1) by bits [begin_bit, end_bit) into out (stable). What in reads and out
// must not overlap; the workspace holds workspace_bytes(n, end_bit - begin_bit).
// With n_dev the count is *n_dev - n_sub, read on the device (n is then a
// capacity: it sizes the grids; out[count, n) is left as it was).
template <typename Load>
inline int radix_sort(Load in, uint64_t* out, int64_t n, int begin_bit, int end_bit, void* workspace,
                      size_t workspace_bytes_given, hipStream_t st, const int64_t* n_dev = nullptr, int64_t n_sub = 0) {
  BF_CHECK_ARG(n >= 0 && n < (int64_t(1) << 31), "radix_sort: %lld keys (at most 2^31 - 1)", (long long)n);
  BF_CHECK_ARG(begin_bit >= 0 && begin_bit < end_bit && end_bit <= 64, "radix_sort: bits [%d, %d)", begin_bit,
               end_bit);
  if (n == 0) return BF_OK;
  const int bits = end_bit - begin_bit;
  const Plan p = make_plan(n, bits);
  const size_t need = workspace_bytes(n, bits);
  BF_CHECK_ARG(workspace && workspace_bytes_given >= need, "radix_sort: workspace %zu < %zu bytes",
               workspace_bytes_given, need);
  char* ws = static_cast<char*>(workspace);
  auto* alt = reinterpret_cast<uint64_t*>(ws);
  auto* counts = reinterpret_cast<uint32_t*>(ws + align256(size_t(n) * 8));
  auto* totals = reinterpret_cast<uint32_t*>(ws + align256(size_t(n) * 8) +
                                             align256(size_t(p.tiles) * (size_t(1) << p.radix) * 4));
  const Sort s{out, alt, n, n_dev, n_sub, begin_bit, end_bit, counts, totals};
  switch (p.radix) {
    case 6: return run_plan<6>(p, in, s, st);
    case 7: return run_plan<7>(p, in, s, st);
    case 8: return run_plan<8>(p, in, s, st);
    case 9: return run_plan<9>(p, in, s, st);
    default: return run_plan<10>(p, in, s, st);
  }
}

// The same for stored keys; an empty bit range copies them.
inline int radix_sort_keys(const uint64_t* in, uint64_t* out, int64_t n, int begin_bit, int end_bit,
                           void* workspace, size_t workspace_bytes_given, hipStream_t st,
                           const int64_t* n_dev = nullptr, int64_t n_sub = 0) {
  if (begin_bit == end_bit && begin_bit >= 0 && end_bit <= 64 && n > 0 && n < (int64_t(1) << 31)) {
    BF_CHECK_ARG(!n_dev, "radix_sort: an empty bit range takes a host count");
    BF_CHECK_HIP(hipMemcpyAsync(out, in, size_t(n) * 8, hipMemcpyDeviceToDevice, st));
    return BF_OK;
  }
  if (begin_bit == end_bit && n == 0) return BF_OK;
  return radix_sort(StoredKeys{in}, out, n, begin_bit, end_bit, workspace, workspace_bytes_given, st, n_dev, n_sub);
}

}  // namespace sort
}  // namespace bf
