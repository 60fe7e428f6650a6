// The node sets of an Adaptive-Budget probe (utils/fullgraph_sp_support.py:
// 1743-1821, 2261-2309): the reception cone of a probe set by breadth-first
// search over the in-neighbour CSR, and a destination filter as an ascending
// query list with what the probe build asks about it.
//
// Both keep one byte per node and read one small record back; as torch
// operators they were some sixty launches and a dozen host reads (sorts of the
// ids, a mask algebra per hop, a test for an empty frontier, minima and maxima
// of ids just made). Probe on 169K nodes: 1.60 -> 0.76 ms.
#include "bf_common.h"
#include "bf_sort.h"

namespace bf {
namespace {

constexpr int kThreads = 256;
constexpr int kGroup = 16;                          // lanes per in-neighbour row
constexpr int kRowsPerBlock = kThreads / kGroup;
constexpr int64_t kBlockRow = 512;                  // a longer row is walked by the whole workgroup
constexpr int kMarkUnroll = 8;
constexpr int kTilePerThread = 16;
constexpr int64_t kTile = int64_t(kThreads) * kTilePerThread;   // nodes per workgroup of the compaction

inline size_t align_up(size_t x) { return (x + 255) & ~size_t(255); }

// level[0, n) = 0 (n rounded up to 16 bytes in the buffer) and the words cleared, by a kernel.
__global__ __launch_bounds__(kThreads) void clear_nodes_kernel(uint4* __restrict__ level, int64_t n16,
                                                               uint32_t* __restrict__ words, int n_words) {
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i < n16) level[i] = make_uint4(0u, 0u, 0u, 0u);
  if (i < n_words) words[i] = 0u;
}

// *bound = the largest node id of any edge, plus 1: the reference sizes its mask by edge_index.max() + 1.
__global__ __launch_bounds__(kThreads) void id_bound_kernel(const int64_t* __restrict__ rowptr,
                                                            const int32_t* __restrict__ col, int64_t n, int64_t n_edges,
                                                            uint32_t* __restrict__ bound) {
  __shared__ int32_t wave[kThreads / 64];
  int32_t top = 0;
  const int64_t stride = int64_t(gridDim.x) * kThreads;
  const int64_t end = n > n_edges ? n : n_edges;
  for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < end; i += stride) {
    if (i < n_edges) top = max(top, col[i] + 1);
    if (i < n && rowptr[i + 1] > rowptr[i]) top = max(top, int32_t(i) + 1);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) top = max(top, __shfl_xor(top, o, 64));
  if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = top;
  __syncthreads();
  if (threadIdx.x == 0)
    atomicMax(bound, uint32_t(max(max(wave[0], wave[1]), max(wave[2], wave[3]))));
}

// level[id] = 1 for every id in [0, *bound); an id outside raises *outside when given.
__global__ __launch_bounds__(kThreads) void mark_ids_kernel(const int64_t* __restrict__ ids, int64_t n_ids,
                                                            int64_t n, const uint32_t* __restrict__ bound,
                                                            uint8_t* __restrict__ level,
                                                            uint32_t* __restrict__ outside) {
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n_ids) return;
  const int64_t id = ids[i], lim = bound ? (int64_t(*bound) < n ? int64_t(*bound) : n) : n;
  if (id >= 0 && id < lim)
    level[id] = 1;
  else if (outside)
    *outside = 1u;
}

// One hop: every in-neighbour of a node of level `hop` that has none yet gets level `next` (concurrent writers agree);
// *grew (if given) becomes hop_no when there is one.
// A 16-lane group walks a row; rows longer than kBlockRow are left to the whole workgroup, and a workgroup's rows
// lie gridDim.x apart, since graphs often number their hubs next to each other: with a group per row, hubs of up
// to 13K edges in one workgroup made a hop of a 169K-node graph 60 us; the workgroup on its long rows 45, the rows
// spread out as well 10.
__global__ __launch_bounds__(kThreads) void cone_hop_kernel(const int64_t* __restrict__ in_ptr,
                                                            const int32_t* __restrict__ in_src, int64_t n, int hop, int next,
                                                            uint8_t* __restrict__ level, uint32_t hop_no,
                                                            uint32_t* __restrict__ grew) {
  __shared__ int64_t long_beg[kRowsPerBlock], long_end[kRowsPerBlock];
  __shared__ int n_long;
  if (threadIdx.x == 0) n_long = 0;
  __syncthreads();
  bool marked_any = false;
  // every step-th source of [i, end), kMarkUnroll of them and then their levels in flight together
  auto mark = [&](int64_t i, int64_t end, int step) {
    for (; i < end; i += int64_t(step) * kMarkUnroll) {
      int32_t src[kMarkUnroll];
      uint8_t lev[kMarkUnroll];
#pragma unroll
      for (int u = 0; u < kMarkUnroll; ++u) {
        const int64_t j = i + int64_t(u) * step;
        src[u] = j < end ? in_src[j] : -1;
      }
#pragma unroll
      for (int u = 0; u < kMarkUnroll; ++u) lev[u] = src[u] >= 0 && src[u] < n ? level[src[u]] : uint8_t(1);
#pragma unroll
      for (int u = 0; u < kMarkUnroll; ++u)
        if (lev[u] == 0) {
          level[src[u]] = uint8_t(next);
          marked_any = true;
        }
    }
  };
  const int64_t v = int64_t(threadIdx.x / kGroup) * gridDim.x + blockIdx.x;
  const int gl = threadIdx.x % kGroup;
  if (v < n && level[v] == hop) {
    const int64_t beg = in_ptr[v], end = in_ptr[v + 1];
    if (end - beg > kBlockRow) {
      if (gl == 0) {
        const int k = atomicAdd(&n_long, 1);
        long_beg[k] = beg;
        long_end[k] = end;
      }
    } else {
      mark(beg + gl, end, kGroup);
    }
  }
  __syncthreads();
  for (int k = 0; k < n_long; ++k) mark(long_beg[k] + threadIdx.x, long_end[k], kThreads);
  if (grew && __ballot(marked_any) && (threadIdx.x & 63) == 0) *grew = hop_no;
}

// Hops between two looks at whether the cone still grows, so that one deeper than its graph ends early; a cone of up
// to this many hops takes none. 169K nodes, 400 layers: 1540 us without looks, 155 with; a chain that grows on 1050,
// 2270.
constexpr int kLookHops = 16;

// Bit u: node t0 + u of this thread's 16 consecutive nodes is marked.
__device__ __forceinline__ uint32_t marked(const uint8_t* __restrict__ level, int64_t n, int64_t t0) {
  if (t0 >= n) return 0u;
  const uint4 x = *reinterpret_cast<const uint4*>(level + t0);   // t0 is a multiple of 16, the buffer padded
  const uint32_t w[4] = {x.x, x.y, x.z, x.w};
  uint32_t f = 0;
#pragma unroll
  for (int u = 0; u < kTilePerThread; ++u)
    if ((w[u >> 2] >> (8 * (u & 3))) & 0xffu) f |= 1u << u;
  return f;
}

// Marked nodes per tile; with in_ptr also *entered = 1 when a marked node has an in-edge.
__global__ __launch_bounds__(kThreads) void mark_count_kernel(const uint8_t* __restrict__ level, int64_t n,
                                                              const int64_t* __restrict__ in_ptr,
                                                              uint32_t* __restrict__ counts,
                                                              uint32_t* __restrict__ entered) {
  __shared__ uint32_t wave[kThreads / 64];
  const int64_t t0 = int64_t(blockIdx.x) * kTile + int64_t(threadIdx.x) * kTilePerThread;
  const uint32_t f = marked(level, n, t0);
  if (in_ptr) {
    bool any = false;
    for (uint32_t rest = f; rest && !any; rest &= rest - 1) {
      const int64_t v = t0 + __ffs(int(rest)) - 1;
      any = in_ptr[v + 1] > in_ptr[v];
    }
    if (__ballot(any) && (threadIdx.x & 63) == 0) *entered = 1u;
  }
  uint32_t c = __popc(f);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = wave[0] + wave[1] + wave[2] + wave[3];
}

template <typename Id>
__global__ __launch_bounds__(kThreads) void mark_write_kernel(const uint8_t* __restrict__ level, int64_t n,
                                                              const uint32_t* __restrict__ prefix,
                                                              Id* __restrict__ out) {
  __shared__ uint32_t tmp[kThreads / 64];
  const int64_t t0 = int64_t(blockIdx.x) * kTile + int64_t(threadIdx.x) * kTilePerThread;
  const uint32_t f = marked(level, n, t0);
  uint32_t total;
  int64_t at = int64_t(prefix[blockIdx.x]) + sort::block_excl_scan<kThreads>(__popc(f), tmp, &total);
  for (uint32_t rest = f; rest; rest &= rest - 1) out[at++] = Id(t0 + __ffs(int(rest)) - 1);
}

// The hubs (ascending) that are marked, in order, and their count: one workgroup.
__global__ __launch_bounds__(kThreads) void mark_hubs_kernel(const int32_t* __restrict__ hubs, int64_t n_hubs,
                                                             const uint8_t* __restrict__ level,
                                                             int32_t* __restrict__ out, uint32_t* __restrict__ count) {
  __shared__ uint32_t tmp[kThreads / 64];
  uint32_t base = 0;
  for (int64_t i0 = 0; i0 < n_hubs; i0 += kThreads) {
    const int64_t i = i0 + threadIdx.x;
    const int32_t h = i < n_hubs ? hubs[i] : 0;
    const bool in = i < n_hubs && level[h] != 0;
    uint32_t total;
    const uint32_t at = base + sort::block_excl_scan<kThreads>(in ? 1u : 0u, tmp, &total);
    if (in) out[at] = h;
    base += total;
  }
  if (threadIdx.x == 0) *count = base;
}

// A workspace of one byte per node, the tiles' counts and a few words.
struct NodeSpace {
  uint8_t* level;
  uint32_t* counts;
  uint32_t* words;
  int64_t tiles;
};
constexpr int kWords = 8;

size_t node_space_bytes(int64_t n) {
  return align_up(size_t(n) + 16) + align_up(size_t(ceil_div(n, kTile)) * 4) + align_up(kWords * 4) + 256;
}

NodeSpace node_space(void* ws, int64_t n) {
  char* p = static_cast<char*>(ws);
  NodeSpace s;
  s.tiles = ceil_div(n, kTile);
  s.level = reinterpret_cast<uint8_t*>(p);
  p += align_up(size_t(n) + 16);
  s.counts = reinterpret_cast<uint32_t*>(p);
  p += align_up(size_t(s.tiles) * 4);
  s.words = reinterpret_cast<uint32_t*>(p);
  return s;
}

int clear_nodes(const NodeSpace& s, int64_t n, hipStream_t st) {
  const int64_t n16 = ceil_div(n, int64_t(16));
  BF_LAUNCH("clear_nodes_kernel", clear_nodes_kernel, dim3(unsigned(ceil_div(n16, int64_t(kThreads)))), dim3(kThreads),
            0, st, reinterpret_cast<uint4*>(s.level), n16, s.words, kWords);
  BF_CHECK_LAUNCH();
  return BF_OK;
}

// *any = 1 when an entry is not 0: a store by each workgroup that finds one, to pinned host memory cleared before.
__global__ __launch_bounds__(kThreads) void any_nonzero_kernel(const int32_t* __restrict__ x, int64_t n,
                                                               int32_t* __restrict__ any) {
  bool found = false;
  const int64_t stride = int64_t(gridDim.x) * kThreads;
  for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < n && !found; i += stride) found = x[i] != 0;
  if (__syncthreads_or(found) && threadIdx.x == 0) *any = 1;
}

}  // namespace
}  // namespace bf

using namespace bf;

extern "C" int bf_any_nonzero(const int32_t* x, int64_t n, int32_t* any_host, void* stream) {
  BF_CHECK_ARG(n >= 0 && any_host, "any_nonzero: bad arguments");
  *any_host = 0;
  if (n == 0) return BF_OK;
  BF_CHECK_ARG(x, "any_nonzero: null tensor");
  hipStream_t st = as_stream(stream);
  BF_HOST_READ(read, st);
  auto* any = read.as<int32_t>();
  *any = 0;
  const int64_t want = ceil_div(n, int64_t(kThreads) * 4);
  BF_LAUNCH("any_nonzero_kernel", any_nonzero_kernel, dim3(unsigned(want < 256 ? want : 256)), dim3(kThreads), 0, st,
            x, n, any);
  BF_CHECK_LAUNCH();
  BF_CHECK_HIP(read.wait());
  *any_host = *any;
  return BF_OK;
}

extern "C" int bf_node_set_workspace_size(int64_t num_nodes, size_t* bytes) {
  BF_CHECK_ARG(bytes && num_nodes >= 0, "node_set_workspace_size: bad arguments");
  *bytes = node_space_bytes(num_nodes);
  return BF_OK;
}

extern "C" int bf_reception_cone(const int64_t* rowptr, const int32_t* col, const int64_t* in_ptr,
                                 const int32_t* in_src, int64_t num_nodes, int64_t num_edges, const int64_t* probe_ids,
                                 int64_t n_probe, int32_t hops, int64_t* ids, int64_t* count_host, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  BF_CHECK_ARG(rowptr && in_ptr && num_nodes > 0 && num_nodes < (int64_t(1) << 31) && num_edges >= 0 && n_probe >= 0 &&
                   hops >= 0 && ids && count_host,
               "reception_cone: bad arguments");
  BF_CHECK_ARG((num_edges == 0 || (col && in_src)) && (n_probe == 0 || probe_ids), "reception_cone: null tensor");
  BF_CHECK_ARG((reinterpret_cast<uintptr_t>(workspace) & 15) == 0 && workspace &&
                   workspace_bytes >= node_space_bytes(num_nodes),
               "reception_cone: workspace %zu < %zu bytes", workspace_bytes, node_space_bytes(num_nodes));
  hipStream_t st = as_stream(stream);
  BF_HOST_READ(read, st);
  auto* count = read.as<uint32_t>();
  const NodeSpace s = node_space(workspace, num_nodes);
  BF_CHECK_OK(clear_nodes(s, num_nodes, st));
  const int64_t work = ceil_div(num_nodes > num_edges ? num_nodes : num_edges, int64_t(kThreads) * 8);
  BF_LAUNCH("id_bound_kernel", id_bound_kernel, dim3(unsigned(work < 2048 ? work : 2048)), dim3(kThreads), 0, st,
            rowptr, col, num_nodes, num_edges, s.words);
  BF_CHECK_LAUNCH();
  if (n_probe > 0) {
    BF_LAUNCH("mark_ids_kernel", mark_ids_kernel, dim3(unsigned(ceil_div(n_probe, int64_t(kThreads)))), dim3(kThreads),
              0, st, probe_ids, n_probe, num_nodes, s.words, s.level, static_cast<uint32_t*>(nullptr));
    BF_CHECK_LAUNCH();
  }
  // levels cycle through 1..254 to fit a byte: a node met again under an old level has no unmarked neighbour left
  uint32_t* const grew = hops > kLookHops ? s.words + 1 : nullptr;
  for (int h = 0; h < hops; ++h) {
    BF_LAUNCH("cone_hop_kernel", cone_hop_kernel, dim3(unsigned(ceil_div(num_nodes, int64_t(kRowsPerBlock)))),
              dim3(kThreads), 0, st, in_ptr, in_src, num_nodes, 1 + h % 254, 1 + (h + 1) % 254, s.level,
              uint32_t(h + 1), grew);
    BF_CHECK_LAUNCH();
    if ((h + 1) % kLookHops == 0 && h + 1 < hops) {
      BF_HOST_READ(look, st);
      BF_CHECK_HIP(hipMemcpyAsync(look.as<uint32_t>(), grew, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
      BF_CHECK_HIP(look.wait());
      if (*look.as<uint32_t>() != uint32_t(h + 1)) break;
    }
  }
  BF_LAUNCH("mark_count_kernel", mark_count_kernel, dim3(unsigned(s.tiles)), dim3(kThreads), 0, st, s.level, num_nodes,
            static_cast<const int64_t*>(nullptr), s.counts, static_cast<uint32_t*>(nullptr));
  BF_CHECK_LAUNCH();
  BF_LAUNCH("radix_scan_kernel", sort::radix_scan_kernel, dim3(1), dim3(sort::kThreads), 0, st, s.counts, s.tiles,
            count);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("mark_write_kernel", mark_write_kernel<int64_t>, dim3(unsigned(s.tiles)), dim3(kThreads), 0, st, s.level,
            num_nodes, s.counts, ids);
  BF_CHECK_LAUNCH();
  BF_CHECK_HIP(read.wait());
  *count_host = *count;
  return BF_OK;
}

extern "C" int bf_probe_queries(const int64_t* filter, int64_t n_filter, int64_t num_nodes, const int64_t* in_ptr,
                                const int32_t* hubs, int64_t n_hubs, int32_t* query_ids, int32_t* hubs_out,
                                int64_t* info_host, void* workspace, size_t workspace_bytes, void* stream) {
  BF_CHECK_ARG(n_filter >= 0 && num_nodes > 0 && num_nodes < (int64_t(1) << 31) && n_hubs >= 0 && info_host && in_ptr,
               "probe_queries: bad arguments");
  BF_CHECK_ARG((n_filter == 0 || (filter && query_ids)) && (n_hubs == 0 || (hubs && hubs_out)),
               "probe_queries: null tensor");
  BF_CHECK_ARG((reinterpret_cast<uintptr_t>(workspace) & 15) == 0 && workspace &&
                   workspace_bytes >= node_space_bytes(num_nodes),
               "probe_queries: workspace %zu < %zu bytes", workspace_bytes, node_space_bytes(num_nodes));
  for (int i = 0; i < 4; ++i) info_host[i] = 0;
  if (n_filter == 0) return BF_OK;
  hipStream_t st = as_stream(stream);
  const NodeSpace s = node_space(workspace, num_nodes);   // words: outside, entered, count, hub count
  BF_CHECK_OK(clear_nodes(s, num_nodes, st));
  BF_LAUNCH("mark_ids_kernel", mark_ids_kernel, dim3(unsigned(ceil_div(n_filter, int64_t(kThreads)))), dim3(kThreads),
            0, st, filter, n_filter, num_nodes, static_cast<const uint32_t*>(nullptr), s.level, s.words);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("mark_count_kernel", mark_count_kernel, dim3(unsigned(s.tiles)), dim3(kThreads), 0, st, s.level, num_nodes,
            in_ptr, s.counts, s.words + 1);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("radix_scan_kernel", sort::radix_scan_kernel, dim3(1), dim3(sort::kThreads), 0, st, s.counts, s.tiles,
            s.words + 2);
  BF_CHECK_LAUNCH();
  BF_LAUNCH("mark_write_kernel", mark_write_kernel<int32_t>, dim3(unsigned(s.tiles)), dim3(kThreads), 0, st, s.level,
            num_nodes, s.counts, query_ids);
  BF_CHECK_LAUNCH();
  if (n_hubs > 0) {
    BF_LAUNCH("mark_hubs_kernel", mark_hubs_kernel, dim3(1), dim3(kThreads), 0, st, hubs, n_hubs, s.level, hubs_out,
              s.words + 3);
    BF_CHECK_LAUNCH();
  }
  BF_HOST_READ(read, st);
  auto* h = read.as<uint32_t>();
  BF_CHECK_HIP(hipMemcpyAsync(h, s.words, 4 * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
  BF_CHECK_HIP(read.wait());
  info_host[0] = h[2];   // queries
  info_host[1] = h[1];   // some query has an in-edge
  info_host[2] = h[3];   // hubs among them
  info_host[3] = h[0];   // an id lies outside [0, num_nodes)
  return BF_OK;
}
