// Edge lists (the reference's COO edge_index) to the attention index's arrays:
// the order of a list, list -> CSR, the reverse index, and the coalesced list.
//
// Every sort here is this build's radix sort (bf_sort.h) on 64-bit keys that
// hold an entry's ids in bit fields, read by the sort's first pass straight
// from the list's int64 arrays. bf_coo_order looks a list over once (ids in
// range, which orders it is in already) and the sorts take only the bits that
// the list is not yet ordered by: none for a list in row order (a coalesced
// list's own CSR), the row bits alone for one in column order (the query-major
// CSR of a coalesced list, of a typed list whose types follow each other).
// Against the former route (four torch reductions with three host reads, a
// 64-bit onesweep sort over all bits, separate passes for the ids and the row
// pointers) a 1.17M-entry list's CSR went from 430 to 190 us, host reads included.
#include "bf_common.h"
#include "bf_sort.h"

namespace bf {
namespace {

constexpr int kThreads = 256;
constexpr int kPerThread = 4;      // entries per thread of the unpacking kernels, loaded before any store

inline size_t align_up(size_t x) { return (x + 255) & ~size_t(255); }

int bits_for(uint64_t maxval) {
  int b = 1;
  while (b < 64 && (uint64_t(1) << b) <= maxval) ++b;
  return b;
}

// ---------------------------------------------------------------- the order of a list
// Each block ORs what its share of the list violates (the BF_COO_* bits), one word per block in pinned host
// memory: nothing to clear before and no atomics; the host ORs the words.
constexpr int64_t kOrderBlocks = 1024;

__global__ __launch_bounds__(kThreads) void coo_order_kernel(const int64_t* __restrict__ row,
                                                             const int64_t* __restrict__ col,
                                                             const int64_t* __restrict__ type, int64_t nnz,
                                                             int64_t n_row, int64_t n_col,
                                                             uint32_t* __restrict__ broken) {
  __shared__ uint32_t wave[kThreads / 64];
  uint32_t bad = 0;
  const int64_t stride = int64_t(gridDim.x) * kThreads;
  for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < nnz; i += stride) {
    const int64_t p = i > 0 ? i - 1 : 0;
    const int64_t r = row[i], c = col[i], rp = row[p], cp = col[p];
    int64_t t = 0, tp = 0;
    if (type) {
      t = type[i];
      tp = type[p];
      if (t < 0 || t > 1) bad |= BF_COO_TYPES;
    }
    if (r < 0 || r >= n_row || c < 0 || c >= n_col) bad |= BF_COO_IDS;
    if (i == 0) continue;
    const bool c_up = t > tp || (t == tp && c > cp), c_same = t == tp && c == cp;   // a column is (type, id)
    if (r < rp) bad |= BF_COO_BY_ROW;
    if (!c_up && !c_same) bad |= BF_COO_BY_COL;
    if (r < rp || (r == rp && !c_up && !c_same)) bad |= BF_COO_ROW_MAJOR;
    if (r < rp || (r == rp && !c_up)) bad |= BF_COO_STRICT;
    if ((!c_up && !c_same) || (c_same && r < rp)) bad |= BF_COO_COL_MAJOR;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) bad |= __shfl_xor(bad, o, 64);
  if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = bad;
  __syncthreads();
  if (threadIdx.x == 0) broken[blockIdx.x] = wave[0] | wave[1] | wave[2] | wave[3];
}

// ---------------------------------------------------------------- keys
// An entry's key: row << (cb + tb) | type << cb | col, with cb and rb the bits of the ids and tb 1 for a
// typed list (its rows are ordered by (type, col)).
struct ListKeys {
  const int64_t* row;
  const int64_t* col;
  const int64_t* type;   // NULL: untyped
  int cb, rshift;        // rshift = cb + tb
  __device__ __forceinline__ uint64_t operator()(int64_t i) const {
    const uint64_t t = type ? uint64_t(type[i]) << cb : 0;
    return (uint64_t(row[i]) << rshift) | t | uint64_t(col[i]);
  }
  __device__ __forceinline__ uint64_t last(int64_t i) const { return (*this)(i); }
};

// Coalesce's keys: src * n + dst, of the list alone or of the list and its mirror image.
struct PairKeys {
  const int64_t* src;
  const int64_t* dst;
  int64_t nnz;           // of the list; entries from nnz on are its mirror image
  uint64_t n;
  __device__ __forceinline__ uint64_t operator()(int64_t i) const {
    const bool m = i >= nnz;
    const int64_t j = m ? i - nnz : i;
    const uint64_t s = uint64_t(src[j]), d = uint64_t(dst[j]);
    return m ? d * n + s : s * n + d;
  }
  __device__ __forceinline__ uint64_t last(int64_t i) const { return (*this)(i); }
};

// Where a key's fields lie: the row pointers follow key >> row_shift, an entry's id is
// (key >> id_shift) & id_mask, its type bit (if any) the key's bit type_bit.
struct KeyFields {
  int row_shift;
  int id_shift;
  uint64_t id_mask;
  int type_bit;          // -1: none
  __device__ __forceinline__ int64_t row(uint64_t k) const { return int64_t(k >> row_shift); }
  __device__ __forceinline__ int32_t id(uint64_t k) const {
    const uint32_t x = uint32_t((k >> id_shift) & id_mask);
    return int32_t(type_bit >= 0 ? x | (uint32_t(k >> type_bit) << 31) : x);
  }
};

struct FieldBits {
  int rb, cb, tb;
};
FieldBits field_bits(int64_t n_row, int64_t n_col, bool typed) {
  return FieldBits{bits_for(uint64_t(n_row > 0 ? n_row - 1 : 0)), bits_for(uint64_t(n_col > 0 ? n_col - 1 : 0)),
                   typed ? 1 : 0};
}

// Keys in row order -> row pointers, ids (with the type in bit 31) and, when asked for, the entries' reverse
// keys col << (rb + tb) | row << tb | type. One pass: the row pointers' boundaries and the ids were two.
template <typename Load>
__global__ __launch_bounds__(kThreads) void coo_unpack_kernel(Load keys, int64_t nnz, KeyFields f, int64_t n_row,
                                                              int64_t* __restrict__ ptr, int32_t* __restrict__ ids,
                                                              uint64_t* __restrict__ rkeys, int rk_row_shift,
                                                              int rk_col_shift) {
  const int64_t base = int64_t(blockIdx.x) * (kThreads * kPerThread) + threadIdx.x;
  uint64_t cur[kPerThread], prev[kPerThread];
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const int64_t i = base + int64_t(u) * kThreads;
    cur[u] = i < nnz ? keys(i) : 0;
    prev[u] = (i > 0 && i <= nnz) ? keys(i - 1) : 0;
  }
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const int64_t i = base + int64_t(u) * kThreads;
    if (i > nnz) break;
    int64_t r_here = i < nnz ? f.row(cur[u]) : n_row;
    int64_t r_prev = i > 0 ? f.row(prev[u]) : -1;
    if (r_here > n_row) r_here = n_row;   // ids are in range: a bound for the store all the same
    if (r_prev > n_row) r_prev = n_row;
    fill_gap(r_prev, r_here, i, [&](int64_t r, int64_t v) { ptr[r] = v; });
    if (i == nnz) break;
    const int32_t id = f.id(cur[u]);
    ids[i] = id;
    if (rkeys) {
      const uint64_t t = f.type_bit >= 0 ? uint64_t(uint32_t(id) >> 31) : 0;
      const uint64_t c = uint32_t(id) & 0x7fffffffu;
      rkeys[i] = (c << rk_col_shift) | (uint64_t(r_here) << rk_row_shift) | t;
    }
  }
}

// Reverse keys of a list in its own order (a list in column order is in reverse order already).
__global__ __launch_bounds__(kThreads) void coo_reverse_keys_kernel(ListKeys in, int64_t nnz, KeyFields f,
                                                                    uint64_t* __restrict__ rkeys, int rk_row_shift,
                                                                    int rk_col_shift) {
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= nnz) return;
  const uint64_t k = in(i);
  const uint32_t id = uint32_t(f.id(k));
  const uint64_t t = f.type_bit >= 0 ? uint64_t(id >> 31) : 0;
  rkeys[i] = (uint64_t(id & 0x7fffffffu) << rk_col_shift) | (uint64_t(f.row(k)) << rk_row_shift) | t;
}

// ks of a list's reverse index: entry i of key row s names query kq[i]; its slot is where s (with the entry's
// type) sits in that query's ascending row. Equal entries of one (row, column) follow each other in both
// orders, so the k-th of them takes the k-th slot. Key rows come from a search within the block's own rows.
// Three searches an entry, where a pair sort used to carry the slots through every list's index: only a bias, factor
// or dropout needs them (COO list and layer with dropout, float32 rows of 128: 20K nodes 524 -> 382 us, 169K
// 1027 -> 836, 600K 2829 -> 2680; with a bias 580 -> 435, 1217 -> 1019, 3766 -> 3614).
__global__ __launch_bounds__(kThreads) void coo_reverse_slots_kernel(const int64_t* __restrict__ qptr,
                                                                     const int32_t* __restrict__ kv,
                                                                     const int64_t* __restrict__ kptr,
                                                                     const int32_t* __restrict__ kq, int64_t nnz,
                                                                     int64_t n_kv, int32_t* __restrict__ ks) {
  const int64_t i0 = int64_t(blockIdx.x) * kThreads;
  __shared__ int64_t bounds[2];
  if (threadIdx.x < 2) {
    const int64_t at = threadIdx.x == 0 ? i0 : (i0 + kThreads - 1 < nnz ? i0 + kThreads - 1 : nnz - 1);
    int64_t lo = 0, hi = n_kv;
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if (kptr[mid] <= at) lo = mid; else hi = mid;
    }
    bounds[threadIdx.x] = lo;
  }
  __syncthreads();
  const int64_t i = i0 + threadIdx.x;
  if (i >= nnz) return;
  int64_t lo = bounds[0], hi = bounds[1] + 1;
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) >> 1;
    if (kptr[mid] <= i) lo = mid; else hi = mid;
  }
  const int64_t s = lo;
  const uint32_t e = uint32_t(kq[i]);
  const uint32_t want = uint32_t(s) | (e & 0x80000000u);     // rows ascend as unsigned (type, id)
  const int64_t q = int64_t(e & 0x7fffffffu), beg = qptr[q];
  lo = beg;
  hi = qptr[q + 1];
  while (lo < hi) {                                           // the first slot holding `want`
    const int64_t mid = (lo + hi) >> 1;
    if (uint32_t(kv[mid]) < want) lo = mid + 1; else hi = mid;
  }
  const int64_t first = lo;
  // the first of the equal reverse entries: a key row ascends by (query, type)
  const uint64_t mine = (uint64_t(e & 0x7fffffffu) << 1) | (e >> 31);
  lo = kptr[s];
  hi = i;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    const uint32_t x = uint32_t(kq[mid]);
    if (((uint64_t(x & 0x7fffffffu) << 1) | (x >> 31)) < mine) lo = mid + 1; else hi = mid;
  }
  ks[i] = int32_t(first - beg + (i - lo));
}

// ---------------------------------------------------------------- coalesce
constexpr int kUniquePerThread = 16;
constexpr int64_t kUniqueTile = int64_t(kThreads) * kUniquePerThread;

// Bit u: sorted key u * kThreads + threadIdx.x of tile b differs from its predecessor.
__device__ __forceinline__ uint32_t unique_flags(const uint64_t* __restrict__ keys, int64_t n, int64_t t0,
                                                 uint64_t (&cur)[kUniquePerThread]) {
  uint64_t prev[kUniquePerThread];
  uint32_t f = 0;
#pragma unroll
  for (int u = 0; u < kUniquePerThread; ++u) {
    const int64_t i = t0 + int64_t(u) * kThreads;
    cur[u] = i < n ? keys[i] : 0;
    prev[u] = (i > 0 && i < n) ? keys[i - 1] : 0;
  }
#pragma unroll
  for (int u = 0; u < kUniquePerThread; ++u) {
    const int64_t i = t0 + int64_t(u) * kThreads;
    if (i < n && (i == 0 || cur[u] != prev[u])) f |= 1u << u;
  }
  return f;
}

__global__ __launch_bounds__(kThreads) void unique_count_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                                uint32_t* __restrict__ counts) {
  __shared__ uint32_t wave[kThreads / 64];
  uint64_t cur[kUniquePerThread];
  uint32_t c = __popc(unique_flags(keys, n, int64_t(blockIdx.x) * kUniqueTile + threadIdx.x, cur));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = wave[0] + wave[1] + wave[2] + wave[3];
}

// The unique keys of tile b, in order, from output position prefix[b] on: per round of kThreads keys a lane's
// place is its wave's ballot rank, after the earlier waves and rounds of the tile.
__global__ __launch_bounds__(kThreads) void unique_write_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                                const uint32_t* __restrict__ prefix, uint64_t div,
                                                                int64_t* __restrict__ out_src,
                                                                int64_t* __restrict__ out_dst) {
  __shared__ uint32_t cnt[kUniquePerThread][kThreads / 64];
  uint64_t cur[kUniquePerThread];
  const uint32_t f = unique_flags(keys, n, int64_t(blockIdx.x) * kUniqueTile + threadIdx.x, cur);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t rank[kUniquePerThread];
#pragma unroll
  for (int u = 0; u < kUniquePerThread; ++u) {
    const uint64_t m = __ballot((f >> u) & 1u);
    rank[u] = __popcll(m & ((uint64_t(1) << lane) - 1));
    if (lane == 0) cnt[u][w] = __popcll(m);
  }
  __syncthreads();
  uint32_t base = prefix[blockIdx.x];
#pragma unroll
  for (int u = 0; u < kUniquePerThread; ++u) {
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int x = 0; x < kThreads / 64; ++x) {
      const uint32_t c = cnt[u][x];
      if (x < w) before += c;
      all += c;
    }
    if ((f >> u) & 1u) {
      const uint64_t q = cur[u] / div;
      const int64_t p = int64_t(base) + before + rank[u];
      out_src[p] = int64_t(q);
      out_dst[p] = int64_t(cur[u] - q * div);
    }
    base += all;
  }
}

// ---------------------------------------------------------------- table -> list
// A table's edge list in coalesce order without its CSR: a block of kListRows table rows checks its lengths and
// ids and adds up its lengths (bf_table_list_check), writes its entries' keys id << qb | row at the places that
// follow from the blocks before it, and the keys sorted by id are the list. The virtual node's entries have
// fixed places behind them and are written with the list.
constexpr int kListRows = 512;
constexpr int kListWidth32 = 1 << 22;    // kListRows rows of at most this many slots are numbered in 32 bits

// Row lengths of block b's rows into LDS, those outside [0, width] as 0 (and counted).
__device__ __forceinline__ uint32_t list_lengths(const int32_t* __restrict__ row_len, int64_t n_rows, int width,
                                                 int32_t (&len)[kListRows]) {
  uint32_t bad = 0;
#pragma unroll
  for (int u = 0; u < kListRows / kThreads; ++u) {
    const int j = u * kThreads + threadIdx.x;
    const int64_t r = int64_t(blockIdx.x) * kListRows + j;
    int32_t l = r < n_rows ? row_len[r] : 0;
    if (l < 0 || l > width) {
      ++bad;
      l = 0;
    }
    len[j] = l;
  }
  return bad;
}

template <typename S>
__device__ __forceinline__ S block_sum(S v, S* wave /*[kThreads / 64]*/) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();                       // an earlier sum's words are read
  if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = v;
  __syncthreads();
  return wave[0] + wave[1] + wave[2] + wave[3];
}

template <typename I>   // of a slot within the block: 32 bits unless the rows are very wide
__global__ __launch_bounds__(kThreads) void table_list_check_kernel(const int32_t* __restrict__ table,
                                                                    const int32_t* __restrict__ row_len,
                                                                    int64_t n_rows, int width, int64_t id_limit,
                                                                    uint64_t* __restrict__ sums,
                                                                    uint64_t* __restrict__ bad) {
  __shared__ int32_t len[kListRows];
  __shared__ I wave[kThreads / 64];
  const uint32_t bad_len = list_lengths(row_len, n_rows, width, len);
  __syncthreads();
  I total = 0;                   // as the slots: 2^31 entries at most in a block numbered in 32 bits
  uint32_t bad_id = 0;
#pragma unroll
  for (int u = 0; u < kListRows / kThreads; ++u) total += I(len[u * kThreads + threadIdx.x]);
  const int64_t r0 = int64_t(blockIdx.x) * kListRows;
  const int rows = int(n_rows - r0 < kListRows ? n_rows - r0 : kListRows);
  const I slots = I(rows) * I(width);
  const int32_t* t = table + r0 * width;
  for (I i0 = threadIdx.x; i0 < slots; i0 += kThreads * kPerThread) {
    int32_t id[kPerThread];
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) id[u] = i0 + u * kThreads < slots ? t[i0 + u * kThreads] : 0;
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
      const I i = i0 + u * kThreads;
      if (i >= slots) break;
      const uint32_t r = uint32_t(i / I(width)), c = uint32_t(i - I(r) * I(width));
      bad_id += (int32_t(c) < len[r] && (id[u] < 0 || int64_t(id[u]) >= id_limit)) ? 1u : 0u;
    }
  }
  const I s = block_sum(total, wave), bl = block_sum(I(bad_len), wave), bi = block_sum(I(bad_id), wave);
  if (threadIdx.x == 0) {
    sums[blockIdx.x] = s;
    bad[2 * int64_t(blockIdx.x)] = bl;
    bad[2 * int64_t(blockIdx.x) + 1] = bi;
  }
}

// The blocks' sums become their first places (32 bits: a list of 2^31 entries or more is refused by the host, which
// gets the 64-bit total); out (pinned host memory) gets the entries, the bad lengths and the bad ids. One workgroup,
// and the host reads 24 bytes: copying the blocks' words (54 KB in two arrays for 2.3M rows) to add them up there
// takes 52 us, a kernel's own store of the sums 11.5 us, launch and wait included in both.
constexpr int kTotalsThreads = 1024;
__global__ __launch_bounds__(kTotalsThreads) void list_totals_kernel(uint64_t* __restrict__ sums,
                                                                     const uint64_t* __restrict__ bad, int64_t blocks,
                                                                     uint64_t* __restrict__ out) {
  __shared__ uint32_t tmp[kTotalsThreads / 64];
  __shared__ uint64_t all[3];
  if (threadIdx.x < 3) all[threadIdx.x] = 0;
  __syncthreads();
  uint32_t base_at = 0;        // the places wrap from 2^32 entries on; the total does not
  uint64_t mine[3] = {0, 0, 0};
  for (int64_t base = 0; base < blocks; base += kTotalsThreads) {
    const int64_t b = base + threadIdx.x;
    const uint64_t v = b < blocks ? sums[b] : 0;
    if (b < blocks) {
      mine[0] += v;
      mine[1] += bad[2 * b];
      mine[2] += bad[2 * b + 1];
    }
    uint32_t tot;
    const uint32_t e = sort::block_excl_scan<kTotalsThreads>(uint32_t(v), tmp, &tot);
    if (b < blocks) sums[b] = base_at + e;
    base_at += tot;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if (!__ballot(mine[i] != 0)) continue;        // the bad ones, nearly always
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mine[i] += __shfl_xor(mine[i], o, 64);
    if ((threadIdx.x & 63) == 0)                  // a wave at a time: a thread each would meet in one LDS word
      atomicAdd(reinterpret_cast<unsigned long long*>(&all[i]), (unsigned long long)mine[i]);
  }
  __syncthreads();
  if (threadIdx.x < 3) out[threadIdx.x] = all[threadIdx.x];
}

template <typename I>   // of a slot within the block: 32 bits unless the rows are very wide
__global__ __launch_bounds__(kThreads) void table_list_keys_kernel(const int32_t* __restrict__ table,
                                                                   const int32_t* __restrict__ row_len,
                                                                   int64_t n_rows, int width,
                                                                   const uint64_t* __restrict__ prefix, int qb,
                                                                   uint64_t* __restrict__ keys) {
  __shared__ int32_t len[kListRows];
  __shared__ uint32_t off[kListRows];
  __shared__ uint32_t tmp[kThreads / 64];
  list_lengths(row_len, n_rows, width, len);
  __syncthreads();
  constexpr int kRows = kListRows / kThreads;      // consecutive rows per thread
  uint32_t mine = 0, total;
#pragma unroll
  for (int u = 0; u < kRows; ++u) mine += uint32_t(len[threadIdx.x * kRows + u]);
  uint32_t at = sort::block_excl_scan<kThreads>(mine, tmp, &total) + uint32_t(prefix[blockIdx.x]);
#pragma unroll
  for (int u = 0; u < kRows; ++u) {
    off[threadIdx.x * kRows + u] = at;
    at += uint32_t(len[threadIdx.x * kRows + u]);
  }
  __syncthreads();
  const int64_t r0 = int64_t(blockIdx.x) * kListRows;
  const int rows = int(n_rows - r0 < kListRows ? n_rows - r0 : kListRows);
  const I slots = I(rows) * I(width);
  const int32_t* t = table + r0 * width;
  for (I i0 = threadIdx.x; i0 < slots; i0 += kThreads * kPerThread) {
    int32_t id[kPerThread];
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) id[u] = i0 + u * kThreads < slots ? t[i0 + u * kThreads] : 0;
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
      const I i = i0 + u * kThreads;
      if (i >= slots) break;
      const uint32_t r = uint32_t(i / I(width)), c = uint32_t(i - I(r) * I(width));
      if (int32_t(c) < len[r]) keys[off[r] + c] = (uint64_t(uint32_t(id[u])) << qb) | uint64_t(r0 + r);
    }
  }
}

// The list: out[0..total) the sources, out[total..2 total) the queries. Entry i < nnz is key i; then token_row
// entries (v + 1 -> 0), then token_col entries (0 -> token_q0 + j).
__global__ __launch_bounds__(kThreads) void list_write_kernel(const uint64_t* __restrict__ keys, int64_t nnz, int qb,
                                                              const int32_t* __restrict__ query_ids, int64_t q_lo,
                                                              int shift, int64_t token_row, int64_t token_q0,
                                                              int64_t total, int64_t* __restrict__ out) {
  const int64_t base = int64_t(blockIdx.x) * (kThreads * kPerThread) + threadIdx.x;
  uint64_t k[kPerThread];
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const int64_t i = base + int64_t(u) * kThreads;
    k[u] = i < nnz ? keys[i] : 0;
  }
#pragma unroll
  for (int u = 0; u < kPerThread; ++u) {
    const int64_t i = base + int64_t(u) * kThreads;
    if (i >= total) break;
    int64_t src, dst;
    if (i < nnz) {
      const int64_t row = int64_t(k[u] & ((uint64_t(1) << qb) - 1));
      src = int64_t(k[u] >> qb) + shift;
      dst = (query_ids ? int64_t(query_ids[row]) : q_lo + row) + shift;
    } else {
      const int64_t j = i - nnz;
      src = j < token_row ? j + 1 : 0;
      dst = j < token_row ? 0 : token_q0 + (j - token_row);
    }
    out[i] = src;
    out[total + i] = dst;
  }
}

struct Carve {            // consecutive 256-byte aligned pieces of a workspace
  char* p;
  template <typename T>
  T* take(size_t bytes) {
    T* q = reinterpret_cast<T*>(p);
    p += align_up(bytes);
    return q;
  }
};

}  // namespace
}  // namespace bf

using namespace bf;

extern "C" int bf_coo_order(const int64_t* row, const int64_t* col, const int64_t* type, int64_t nnz, int64_t n_row,
                            int64_t n_col, int32_t* holds_host, void* stream) {
  BF_CHECK_ARG(holds_host && nnz >= 0 && n_row >= 0 && n_col >= 0, "coo_order: bad arguments");
  constexpr int32_t kAll = BF_COO_IDS | BF_COO_TYPES | BF_COO_ROW_MAJOR | BF_COO_COL_MAJOR | BF_COO_STRICT |
                           BF_COO_BY_COL | BF_COO_BY_ROW;
  *holds_host = kAll;
  if (nnz == 0) return BF_OK;
  BF_CHECK_ARG(row && col, "coo_order: null tensor");
  static_assert(kHostReadBytes >= kOrderBlocks * sizeof(uint32_t), "one word per block");
  hipStream_t st = as_stream(stream);
  BF_HOST_READ(read, st);
  const int64_t want = ceil_div(nnz, int64_t(kThreads) * 4);
  const int64_t blocks = want < kOrderBlocks ? want : kOrderBlocks;
  auto* words = read.as<uint32_t>();
  BF_LAUNCH("coo_order_kernel", coo_order_kernel, dim3(unsigned(blocks)), dim3(kThreads), 0, st, row, col, type, nnz,
            n_row, n_col, words);
  BF_CHECK_LAUNCH();
  BF_CHECK_HIP(read.wait());
  uint32_t broken = 0;
  for (int64_t b = 0; b < blocks; ++b) broken |= words[b];
  *holds_host = kAll & ~int32_t(broken);
  return BF_OK;
}

extern "C" int bf_coo_to_csr_ordered_workspace_size(int64_t nnz, int64_t n_row, int64_t n_col, int32_t typed,
                                                    int32_t holds, size_t* bytes) {
  BF_CHECK_ARG(bytes && nnz >= 0 && n_row >= 0 && n_col >= 0, "coo_to_csr_ordered_workspace_size: bad arguments");
  *bytes = 256;
  if (nnz == 0 || (holds & BF_COO_ROW_MAJOR)) return BF_OK;
  const FieldBits b = field_bits(n_row, n_col, typed != 0);
  const int bits = (holds & BF_COO_BY_COL) ? b.rb : b.rb + b.cb + b.tb;
  *bytes += align_up(size_t(nnz) * 8) + sort::workspace_bytes(nnz, bits);
  return BF_OK;
}

extern "C" int bf_coo_to_csr_ordered(const int64_t* row, const int64_t* col, const int64_t* type, int64_t nnz,
                                     int64_t n_row, int64_t n_col, int32_t holds, int64_t* ptr, int32_t* ids,
                                     uint64_t* rkeys, void* workspace, size_t workspace_bytes, void* stream) {
  BF_CHECK_ARG(nnz >= 0 && n_row >= 0 && n_col > 0 && ptr, "coo_to_csr_ordered: bad arguments");
  // rows are 32-bit only in a reverse index; a key holds a row's and an id's bits, the id's at most 31
  const FieldBits b = field_bits(n_row, n_col, type != nullptr);
  BF_CHECK_ARG((!rkeys || n_row < (int64_t(1) << 31)) && b.rb + b.cb + b.tb <= 64 && n_col < (int64_t(1) << 31) &&
                   nnz < (int64_t(1) << 31),
               "coo_to_csr_ordered: sizes must fit int32");
  size_t need = 0;
  BF_CHECK_OK(bf_coo_to_csr_ordered_workspace_size(nnz, n_row, n_col, type != nullptr, holds, &need));
  BF_CHECK_ARG(workspace && workspace_bytes >= need, "coo_to_csr_ordered: workspace %zu < %zu bytes",
               workspace_bytes, need);
  hipStream_t st = as_stream(stream);
  if (nnz == 0) {
    BF_CHECK_HIP(hipMemsetAsync(ptr, 0, size_t(n_row + 1) * sizeof(int64_t), st));
    return BF_OK;
  }
  BF_CHECK_ARG(row && col && ids, "coo_to_csr_ordered: null tensor");
  const ListKeys in{row, col, type, b.cb, b.cb + b.tb};
  const KeyFields f{b.cb + b.tb, 0, (uint64_t(1) << b.cb) - 1, type ? b.cb : -1};
  const int rk_row = b.tb, rk_col = b.rb + b.tb;
  // a list in column order is its own reverse order: its reverse keys come from it, sorted
  const bool reverse_now = rkeys && (holds & BF_COO_COL_MAJOR) && !type;
  const unsigned blocks = unsigned(ceil_div(nnz + 1, int64_t(kThreads) * kPerThread));
  if (holds & BF_COO_ROW_MAJOR) {
    BF_LAUNCH("coo_unpack_kernel", coo_unpack_kernel<ListKeys>, dim3(blocks), dim3(kThreads), 0, st, in, nnz, f, n_row,
              ptr, ids, reverse_now ? nullptr : rkeys, rk_row, rk_col);
    BF_CHECK_LAUNCH();
  } else {
    Carve ws{static_cast<char*>(workspace)};
    auto* sorted = ws.take<uint64_t>(size_t(nnz) * 8);
    const int begin = (holds & BF_COO_BY_COL) ? b.cb + b.tb : 0;
    BF_CHECK_OK(sort::radix_sort(in, sorted, nnz, begin, b.rb + b.cb + b.tb, ws.p,
                                 workspace_bytes - size_t(ws.p - static_cast<char*>(workspace)), st));
    BF_LAUNCH("coo_unpack_kernel", coo_unpack_kernel<sort::StoredKeys>, dim3(blocks), dim3(kThreads), 0, st,
              sort::StoredKeys{sorted}, nnz, f, n_row, ptr, ids, reverse_now ? nullptr : rkeys, rk_row, rk_col);
    BF_CHECK_LAUNCH();
  }
  if (reverse_now) {
    BF_LAUNCH("coo_reverse_keys_kernel", coo_reverse_keys_kernel, dim3(unsigned(ceil_div(nnz, kThreads))),
              dim3(kThreads), 0, st, in, nnz, f, rkeys, rk_row, rk_col);
    BF_CHECK_LAUNCH();
  }
  return BF_OK;
}

extern "C" int bf_coo_to_csr_workspace_size(int64_t nnz, int64_t n_q, size_t* bytes) {
  BF_CHECK_ARG(bytes && nnz >= 0 && n_q >= 0, "coo_to_csr_workspace_size: bad arguments");
  *bytes = align_up(size_t(nnz > 0 ? nnz : 1) * 8) + sort::workspace_bytes_max(nnz) + 256;
  return BF_OK;
}

extern "C" int bf_coo_to_csr(const int64_t* src, const int64_t* dst, int64_t nnz, int64_t n_q, int64_t n_kv,
                             int64_t* qptr, int32_t* kv, void* workspace, size_t workspace_bytes, void* stream) {
  BF_CHECK_ARG(nnz >= 0 && n_q >= 0 && n_kv > 0 && qptr, "coo_to_csr: bad arguments");
  return bf_coo_to_csr_ordered(dst, src, nullptr, nnz, n_q, n_kv, 0, qptr, kv, nullptr, workspace, workspace_bytes,
                               stream);
}

extern "C" int bf_coo_reverse_workspace_size(int64_t nnz, int64_t n_row, int64_t n_col, int32_t typed, int32_t sorted,
                                             size_t* bytes) {
  BF_CHECK_ARG(bytes && nnz >= 0 && n_row >= 0 && n_col >= 0, "coo_reverse_workspace_size: bad arguments");
  *bytes = 256;
  if (nnz == 0 || sorted) return BF_OK;
  *bytes += align_up(size_t(nnz) * 8) + sort::workspace_bytes(nnz, field_bits(n_row, n_col, typed != 0).cb);
  return BF_OK;
}

extern "C" int bf_coo_reverse(const uint64_t* rkeys, int64_t nnz, int64_t n_row, int64_t n_col, int32_t typed,
                              int32_t sorted, int64_t* kptr, int32_t* kq, void* workspace, size_t workspace_bytes,
                              void* stream) {
  BF_CHECK_ARG(nnz >= 0 && n_row >= 0 && n_col >= 0 && kptr, "coo_reverse: bad arguments");
  BF_CHECK_ARG(n_row < (int64_t(1) << 31) && n_col < (int64_t(1) << 31) && nnz < (int64_t(1) << 31),
               "coo_reverse: sizes must fit int32");
  size_t need = 0;
  BF_CHECK_OK(bf_coo_reverse_workspace_size(nnz, n_row, n_col, typed, sorted, &need));
  BF_CHECK_ARG(workspace && workspace_bytes >= need, "coo_reverse: workspace %zu < %zu bytes", workspace_bytes, need);
  hipStream_t st = as_stream(stream);
  if (nnz == 0) {
    BF_CHECK_HIP(hipMemsetAsync(kptr, 0, size_t(n_col + 1) * sizeof(int64_t), st));
    return BF_OK;
  }
  BF_CHECK_ARG(rkeys && kq, "coo_reverse: null tensor");
  const FieldBits b = field_bits(n_row, n_col, typed != 0);
  const KeyFields f{b.rb + b.tb, b.tb, (uint64_t(1) << b.rb) - 1, typed ? 0 : -1};
  const uint64_t* keys = rkeys;
  if (!sorted) {
    Carve ws{static_cast<char*>(workspace)};
    auto* out = ws.take<uint64_t>(size_t(nnz) * 8);
    // stable over the column bits alone: each column's entries stay in CSR order
    BF_CHECK_OK(sort::radix_sort(sort::StoredKeys{rkeys}, out, nnz, b.rb + b.tb, b.rb + b.tb + b.cb, ws.p,
                                 workspace_bytes - size_t(ws.p - static_cast<char*>(workspace)), st));
    keys = out;
  }
  BF_LAUNCH("coo_unpack_kernel", coo_unpack_kernel<sort::StoredKeys>,
            dim3(unsigned(ceil_div(nnz + 1, int64_t(kThreads) * kPerThread))), dim3(kThreads), 0, st,
            sort::StoredKeys{keys}, nnz, f, n_col, kptr, kq, static_cast<uint64_t*>(nullptr), 0, 0);
  BF_CHECK_LAUNCH();
  return BF_OK;
}

extern "C" int bf_coo_reverse_slots(const int64_t* qptr, const int32_t* kv, const int64_t* kptr, const int32_t* kq,
                                    int64_t nnz, int64_t n_kv, int32_t* ks, void* stream) {
  BF_CHECK_ARG(nnz >= 0 && n_kv >= 0, "coo_reverse_slots: bad arguments");
  if (nnz == 0) return BF_OK;
  BF_CHECK_ARG(qptr && kv && kptr && kq && ks && n_kv > 0, "coo_reverse_slots: null tensor");
  BF_LAUNCH("coo_reverse_slots_kernel", coo_reverse_slots_kernel, dim3(unsigned(ceil_div(nnz, kThreads))),
            dim3(kThreads), 0, as_stream(stream), qptr, kv, kptr, kq, nnz, n_kv, ks);
  BF_CHECK_LAUNCH();
  return BF_OK;
}

extern "C" int bf_coalesce_workspace_size(int64_t nnz, size_t* bytes) {
  BF_CHECK_ARG(bytes && nnz >= 0, "coalesce_workspace_size: bad arguments");
  const int64_t tiles = ceil_div(nnz > 0 ? nnz : 1, kUniqueTile);
  *bytes = align_up(size_t(nnz > 0 ? nnz : 1) * 8) + align_up(size_t(tiles) * 4) + 256 +
           sort::workspace_bytes_max(nnz) + 256;
  return BF_OK;
}

namespace {
int coalesce_list(const PairKeys& in, int64_t total, int64_t num_nodes, int64_t* out_src, int64_t* out_dst,
                  int64_t* count_host, void* workspace, size_t workspace_bytes, hipStream_t st) {
  size_t need = 0;
  BF_CHECK_OK(bf_coalesce_workspace_size(total, &need));
  BF_CHECK_ARG(workspace && workspace_bytes >= need, "coalesce: workspace %zu < %zu bytes", workspace_bytes, need);
  const int64_t tiles = ceil_div(total, kUniqueTile);
  Carve ws{static_cast<char*>(workspace)};
  auto* keys = ws.take<uint64_t>(size_t(total) * 8);
  auto* counts = ws.take<uint32_t>(size_t(tiles) * 4);
  BF_HOST_READ(read, st);
  auto* count = read.as<uint32_t>();
  const int end_bit = bits_for(uint64_t(num_nodes) * uint64_t(num_nodes));
  BF_CHECK_OK(sort::radix_sort(in, keys, total, 0, end_bit, ws.p,
                               workspace_bytes - size_t(ws.p - static_cast<char*>(workspace)), st));
  BF_LAUNCH("unique_count_kernel", unique_count_kernel, dim3(unsigned(tiles)), dim3(kThreads), 0, st, keys, total,
            counts);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("radix_scan_kernel", sort::radix_scan_kernel, dim3(1), dim3(sort::kThreads), 0, st, counts, tiles, count);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("unique_write_kernel", unique_write_kernel, dim3(unsigned(tiles)), dim3(kThreads), 0, st, keys, total,
            counts, uint64_t(num_nodes), out_src, out_dst);
  BF_CHECK_LAUNCH();
  BF_CHECK_HIP(read.wait());
  *count_host = *count;
  return BF_OK;
}
}  // namespace

extern "C" int bf_coalesce(const int64_t* src, const int64_t* dst, int64_t nnz, int64_t num_nodes, int64_t* out_src,
                           int64_t* out_dst, int64_t* count_host, void* workspace, size_t workspace_bytes,
                           void* stream) {
  BF_CHECK_ARG(count_host && nnz >= 0 && num_nodes > 0, "coalesce: bad arguments");
  BF_CHECK_ARG(nnz < (int64_t(1) << 31) && num_nodes < (int64_t(1) << 32), "coalesce: sizes out of range");
  *count_host = 0;
  if (nnz == 0) return BF_OK;
  BF_CHECK_ARG(src && dst && out_src && out_dst, "coalesce: null tensor");
  return coalesce_list(PairKeys{src, dst, nnz, uint64_t(num_nodes)}, nnz, num_nodes, out_src, out_dst, count_host,
                       workspace, workspace_bytes, as_stream(stream));
}

extern "C" int bf_coalesce_bidirected(const int64_t* src, const int64_t* dst, int64_t nnz, int64_t num_nodes,
                                      int64_t* out_src, int64_t* out_dst, int64_t* count_host, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  BF_CHECK_ARG(count_host && nnz >= 0 && num_nodes > 0, "coalesce_bidirected: bad arguments");
  BF_CHECK_ARG(2 * nnz < (int64_t(1) << 31) && num_nodes < (int64_t(1) << 32),
               "coalesce_bidirected: sizes out of range");
  *count_host = 0;
  if (nnz == 0) return BF_OK;
  BF_CHECK_ARG(src && dst && out_src && out_dst, "coalesce_bidirected: null tensor");
  return coalesce_list(PairKeys{src, dst, nnz, uint64_t(num_nodes)}, 2 * nnz, num_nodes, out_src, out_dst, count_host,
                       workspace, workspace_bytes, as_stream(stream));
}

namespace {
int64_t list_blocks(int64_t n_rows) { return ceil_div(n_rows, int64_t(kListRows)); }
size_t list_sums_bytes(int64_t n_rows) { return align_up(size_t(list_blocks(n_rows)) * 8 + 8); }
}  // namespace

extern "C" int bf_table_list_check_workspace_size(int64_t n_rows, size_t* bytes) {
  BF_CHECK_ARG(bytes && n_rows >= 0, "table_list_check_workspace_size: bad arguments");
  *bytes = list_sums_bytes(n_rows) + align_up(size_t(list_blocks(n_rows)) * 16) + 256;
  return BF_OK;
}

extern "C" int bf_table_list_check(const int32_t* table, const int32_t* row_len, int64_t n_rows, int32_t width,
                                   int64_t id_limit, int64_t* nnz_host, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  BF_CHECK_ARG(n_rows >= 0 && width >= 0 && id_limit >= 0 && nnz_host,
               "table_list_check: bad arguments");
  *nnz_host = 0;
  if (n_rows == 0) return BF_OK;
  BF_CHECK_ARG((table || width == 0) && row_len, "table_list_check: null tensor");
  size_t need = 0;
  BF_CHECK_OK(bf_table_list_check_workspace_size(n_rows, &need));
  BF_CHECK_ARG(workspace && workspace_bytes >= need, "table_list_check: workspace %zu < %zu bytes", workspace_bytes,
               need);
  hipStream_t st = as_stream(stream);
  const int64_t blocks = list_blocks(n_rows);
  auto* sums = static_cast<uint64_t*>(workspace);
  auto* bad = reinterpret_cast<uint64_t*>(static_cast<char*>(workspace) + list_sums_bytes(n_rows));
  if (width <= kListWidth32)
    BF_LAUNCH("table_list_check_kernel", table_list_check_kernel<uint32_t>, dim3(unsigned(blocks)), dim3(kThreads), 0,
              st, table, row_len, n_rows, width, id_limit, sums, bad);
  else
    BF_LAUNCH("table_list_check_kernel", table_list_check_kernel<uint64_t>, dim3(unsigned(blocks)), dim3(kThreads), 0,
              st, table, row_len, n_rows, width, id_limit, sums, bad);
  BF_CHECK_LAUNCH();
  BF_HOST_READ(read, st);
  auto* h = read.as<uint64_t>();
  BF_LAUNCH("list_totals_kernel", list_totals_kernel, dim3(1), dim3(kTotalsThreads), 0, st, sums, bad, blocks, h);
  BF_CHECK_LAUNCH();
  BF_CHECK_HIP(read.wait());
  const int64_t nnz = int64_t(h[0]), bad_len = int64_t(h[1]), bad_id = int64_t(h[2]);
  BF_CHECK_ARG(bad_len == 0, "check_table: %lld row lengths outside [0, %d]", (long long)bad_len, width);
  BF_CHECK_ARG(bad_id == 0, "check_table: %lld table ids outside [0, %lld)", (long long)bad_id, (long long)id_limit);
  BF_CHECK_ARG(nnz < (int64_t(1) << 31), "table_list_check: %lld entries (at most 2^31 - 1)", (long long)nnz);
  *nnz_host = nnz;
  return BF_OK;
}

extern "C" int bf_table_to_list_workspace_size(int64_t nnz, int64_t id_limit, size_t* bytes) {
  BF_CHECK_ARG(bytes && nnz >= 0 && id_limit >= 0, "table_to_list_workspace_size: bad arguments");
  *bytes = 256;
  if (nnz == 0) return BF_OK;
  *bytes += 2 * align_up(size_t(nnz) * 8) +
            sort::workspace_bytes(nnz, bits_for(uint64_t(id_limit > 0 ? id_limit - 1 : 0)));
  return BF_OK;
}

extern "C" int bf_table_to_list(const int32_t* table, const int32_t* row_len, int64_t n_rows, int32_t width,
                                int64_t nnz, int64_t id_limit, const int32_t* query_ids, int64_t q_lo, int32_t shift,
                                int64_t token_row, int64_t token_q0, int64_t token_col, void* checked,
                                int64_t* out, void* workspace, size_t workspace_bytes, void* stream) {
  BF_CHECK_ARG(n_rows >= 0 && n_rows < (int64_t(1) << 31) && width >= 0 && nnz >= 0 &&
                   id_limit >= 0 && id_limit < (int64_t(1) << 31) && token_row >= 0 && token_col >= 0,
               "table_to_list: bad arguments");
  const int64_t total = nnz + token_row + token_col;
  if (total == 0) return BF_OK;
  size_t need = 0;
  BF_CHECK_OK(bf_table_to_list_workspace_size(nnz, id_limit, &need));
  BF_CHECK_ARG(out && workspace && workspace_bytes >= need, "table_to_list: workspace %zu < %zu bytes",
               workspace_bytes, need);
  hipStream_t st = as_stream(stream);
  const int qb = bits_for(uint64_t(n_rows > 0 ? n_rows - 1 : 0));
  const int ib = bits_for(uint64_t(id_limit > 0 ? id_limit - 1 : 0));
  uint64_t* sorted = nullptr;
  if (nnz > 0) {
    BF_CHECK_ARG(table && row_len && checked, "table_to_list: null tensor");
    Carve ws{static_cast<char*>(workspace)};
    auto* keys = ws.take<uint64_t>(size_t(nnz) * 8);
    sorted = ws.take<uint64_t>(size_t(nnz) * 8);
    const int64_t blocks = list_blocks(n_rows);
    const auto* sums = static_cast<const uint64_t*>(checked);    // the blocks' first places
    if (width <= kListWidth32)
      BF_LAUNCH("table_list_keys_kernel", table_list_keys_kernel<uint32_t>, dim3(unsigned(blocks)), dim3(kThreads), 0,
                st, table, row_len, n_rows, width, sums, qb, keys);
    else
      BF_LAUNCH("table_list_keys_kernel", table_list_keys_kernel<uint64_t>, dim3(unsigned(blocks)), dim3(kThreads), 0,
                st, table, row_len, n_rows, width, sums, qb, keys);
    BF_CHECK_LAUNCH();
    // stable over the id bits: each id's entries stay in row order
    BF_CHECK_OK(sort::radix_sort(sort::StoredKeys{keys}, sorted, nnz, qb, qb + ib, ws.p,
                                 workspace_bytes - size_t(ws.p - static_cast<char*>(workspace)), st));
  }
  BF_LAUNCH("list_write_kernel", list_write_kernel, dim3(unsigned(ceil_div(total, int64_t(kThreads) * kPerThread))),
            dim3(kThreads), 0, st, sorted, nnz, qb, query_ids, q_lo, shift, token_row, token_q0, total, out);
  BF_CHECK_LAUNCH();
  return BF_OK;
}
