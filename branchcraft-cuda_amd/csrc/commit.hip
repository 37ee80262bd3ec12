// Accepted-path commit and copy-on-write page clone for gfx950.
//
// Reference: commit_kernel / commit_path (src/tree_attention.cu:73-89,
// 107-122) and the page clone done with cudaMemcpy D2D (src/main.cu:276-281)
// or torch copy_ (python/branchcraft_torch/transaction.py:133-134).
// bc_commit_paths commits the accepted paths of several requests in one
// launch; bc_copy_pages clones any number of pages in one launch;
// bc_write_prefix fills a request's pages from its prompt's K and V rows (the
// reference: two slice copies per page, transaction.py:64-81).
// All are bit copies of FP16 rows, moved as 16-byte vectors when every
// tensor pointer is 16-byte aligned and as single halves otherwise (the
// reference accepts any `half*`); every index is range-checked on the device
// and an out-of-range entry is skipped rather than written out of bounds
// (page ids against physical_pages when the caller gives it).
#include "bc_device.h"

namespace {

constexpr int kThreads = 256;

// One workgroup per accepted node; K and V rows of Hkv*D halves each, moved
// as `row_vec` elements of type E (uint4: eight halves, uint16_t: one).  The
// node's request is `requests[i]` when a list is given, else `request`.
template <typename E>
__global__ __launch_bounds__(kThreads) void commit_kernel(
    const E* __restrict__ draft_k, const E* __restrict__ draft_v,
    E* __restrict__ cache_k, E* __restrict__ cache_v,
    const int32_t* __restrict__ requests, const int32_t* __restrict__ path_nodes,
    const int32_t* __restrict__ dest_pages,
    const int32_t* __restrict__ dest_slots, int request, int batch, int nodes,
    int phys_pages, int row_vec) {
  const int i = blockIdx.x;
  if (requests) request = requests[i];
  const int node = path_nodes[i];
  const int page = dest_pages[i];
  const int slot = dest_slots[i];
  if (request < 0 || request >= batch || node < 0 || node >= nodes || page < 0 ||
      page >= phys_pages || slot < 0 || slot >= BC_PAGE_SIZE)
    return;
  const size_t src = ((size_t)request * nodes + node) * row_vec;
  const size_t dst = ((size_t)page * BC_PAGE_SIZE + slot) * row_vec;
  for (int x = threadIdx.x; x < row_vec; x += kThreads) {
    cache_k[dst + x] = draft_k[src + x];
    cache_v[dst + x] = draft_v[src + x];
  }
}

// grid = (count, slices): workgroup (i, s) copies slice s of page pair i,
// in elements of type E as for commit_kernel.
template <typename E>
__global__ __launch_bounds__(kThreads) void copy_pages_kernel(
    E* __restrict__ cache_k, E* __restrict__ cache_v,
    const int32_t* __restrict__ src_pages, const int32_t* __restrict__ dst_pages,
    int phys_pages, int page_vec, int slice_vec) {
  const int i = blockIdx.x;
  const int src = src_pages[i];
  const int dst = dst_pages[i];
  if (src < 0 || src >= phys_pages || dst < 0 || dst >= phys_pages || src == dst)
    return;
  const int lo = blockIdx.y * slice_vec;
  const int hi = min(lo + slice_vec, page_vec);
  const size_t s0 = (size_t)src * page_vec, d0 = (size_t)dst * page_vec;
  for (int x = lo + threadIdx.x; x < hi; x += kThreads) {
    cache_k[d0 + x] = cache_k[s0 + x];
    cache_v[d0 + x] = cache_v[s0 + x];
  }
}

// Integers carried in the kernel arguments, so that a list that lives on the
// host needs no copy: 3.5 KB of the 4 KB an argument block may hold.
constexpr int kListInts = 896;
struct IntList {
  int32_t v[kListInts];
};

// dst[i] = list.v[i], i < n: a host list into device memory without the copy
// engine.  A copy from pageable memory makes the host wait until the stream is
// idle; this is one launch.  As an index tensor from a Python list, a call in a
// stream of them: 130 entries 6.5 us (19.4 by the copy), 896 13.5 (36.4), 4096
// 54 (111), 65536 792 (1453), so that no length is better off with the copy.
__global__ __launch_bounds__(kThreads) void write_ints_kernel(int32_t* __restrict__ dst, int n,
                                                              IntList list) {
  for (int i = threadIdx.x; i < n; i += kThreads) dst[i] = list.v[i];
}

constexpr int kSliceTokens = 4;  // tokens of one page per workgroup

// grid = (pages, slices): workgroup (i, s) copies kSliceTokens of the rows
// [token, Hkv, D] that page list.v[i] takes, K and V, in elements of type E.
// A row's heads are head_vec elements each, hs apart in the source; rows are
// ts apart (both in elements, K's and V's strides each its own).
// HBM- and launch-bound: 4093 tokens of 8 heads x 128 (33.5 MB moved) take
// 7.0 us (4.8 TB/s, the rate of a large copy), against 512 slice copies of 1.6
// us each, one launch apiece; PagedTreeCache.new 3152 -> 62 us.
template <typename E>
__global__ __launch_bounds__(kThreads) void write_prefix_kernel(
    const E* __restrict__ k, const E* __restrict__ v, long long k_ts, long long k_hs,
    long long v_ts, long long v_hs, E* __restrict__ cache_k, E* __restrict__ cache_v, int tokens,
    int phys_pages, int row_vec, int head_vec, IntList list) {
  const int i = blockIdx.x;
  const int page = list.v[i];
  if (page < 0 || page >= phys_pages) return;
  const int s0 = blockIdx.y * kSliceTokens;  // first slot of the slice
  const int n = min(kSliceTokens, tokens - i * BC_PAGE_SIZE - s0) * row_vec;
  const size_t dst = ((size_t)page * BC_PAGE_SIZE + s0) * row_vec;
  const long long t0 = (long long)i * BC_PAGE_SIZE + s0;
  for (int x = threadIdx.x; x < n; x += kThreads) {
    const int t = x / row_vec, c = x - t * row_vec;
    const int h = c / head_vec, e = c - h * head_vec;
    cache_k[dst + x] = k[(t0 + t) * k_ts + h * k_hs + e];
    cache_v[dst + x] = v[(t0 + t) * v_ts + h * v_hs + e];
  }
}

bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

// Upper bound on page ids.  The reference checks no page id
// (src/tree_attention.cu:73-89); a physical_pages below 1 means the pool size
// is not given, and then only negative ids are skipped.
int pool_bound(const bc_shape& s) {
  return s.physical_pages >= 1 ? s.physical_pages : 0x7fffffff;
}

// Launches commit_kernel over `count` entries with 16-byte elements when all
// four tensors allow it, single halves otherwise.
hipError_t launch_commit(const bc_shape& s, const bc_half* draft_k, const bc_half* draft_v,
                         bc_half* cache_k, bc_half* cache_v, const int32_t* requests,
                         const int32_t* path_nodes, const int32_t* dest_pages,
                         const int32_t* dest_slots, int request, int nodes, int count,
                         hipStream_t st) {
  const int row = s.kv_heads * s.dim;  // halves per K (or V) row
  const int phys = pool_bound(s);
  if (aligned16(draft_k) && aligned16(draft_v) && aligned16(cache_k) && aligned16(cache_v))
    commit_kernel<uint4><<<dim3(count), kThreads, 0, st>>>(
        reinterpret_cast<const uint4*>(draft_k), reinterpret_cast<const uint4*>(draft_v),
        reinterpret_cast<uint4*>(cache_k), reinterpret_cast<uint4*>(cache_v), requests,
        path_nodes, dest_pages, dest_slots, request, s.batch, nodes, phys, row / 8);
  else
    commit_kernel<uint16_t><<<dim3(count), kThreads, 0, st>>>(
        draft_k, draft_v, cache_k, cache_v, requests, path_nodes, dest_pages, dest_slots,
        request, s.batch, nodes, phys, row);
  return hipGetLastError();
}

}  // namespace

extern "C" int bc_commit_path(bc_shape s, const bc_half* draft_k,
                              const bc_half* draft_v, bc_half* cache_k,
                              bc_half* cache_v, const int32_t* path_nodes,
                              const int32_t* dest_pages,
                              const int32_t* dest_slots, int request,
                              int nodes, int accepted, bc_stream_t stream) {
  // The reference's rules (src/tree_attention.cu:111-114), nothing more.
  if (!draft_k || !draft_v || !cache_k || !cache_v || !path_nodes ||
      !dest_pages || !dest_slots || request < 0 || request >= s.batch ||
      nodes < 1 || accepted < 1 || accepted > nodes)
    return BC_ERROR_INVALID_VALUE;
  if (s.dim != 64 && s.dim != 128) return BC_ERROR_INVALID_VALUE;
  if (s.kv_heads < 1) return BC_SUCCESS;  // rows of no heads: nothing to copy
  return launch_commit(s, draft_k, draft_v, cache_k, cache_v, nullptr, path_nodes,
                       dest_pages, dest_slots, request, nodes, accepted,
                       reinterpret_cast<hipStream_t>(stream));
}

extern "C" int bc_commit_paths(bc_shape s, const bc_half* draft_k,
                               const bc_half* draft_v, bc_half* cache_k,
                               bc_half* cache_v, const int32_t* requests,
                               const int32_t* path_nodes,
                               const int32_t* dest_pages,
                               const int32_t* dest_slots, int nodes, int count,
                               bc_stream_t stream) {
  if (!draft_k || !draft_v || !cache_k || !cache_v || !requests || !path_nodes ||
      !dest_pages || !dest_slots || s.batch < 1 || nodes < 1 || count < 0 ||
      (s.dim != 64 && s.dim != 128))
    return BC_ERROR_INVALID_VALUE;
  if (count == 0 || s.kv_heads < 1) return BC_SUCCESS;
  return launch_commit(s, draft_k, draft_v, cache_k, cache_v, requests, path_nodes,
                       dest_pages, dest_slots, 0, nodes, count,
                       reinterpret_cast<hipStream_t>(stream));
}

extern "C" int bc_copy_pages(bc_shape s, bc_half* cache_k, bc_half* cache_v,
                             const int32_t* src_pages,
                             const int32_t* dst_pages, int count,
                             bc_stream_t stream) {
  if (!cache_k || !cache_v || !src_pages || !dst_pages || count < 0 ||
      (s.dim != 64 && s.dim != 128))
    return BC_ERROR_INVALID_VALUE;
  if (count == 0 || s.kv_heads < 1) return BC_SUCCESS;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int page = BC_PAGE_SIZE * s.kv_heads * s.dim;  // halves per page of K (or V)
  const int phys = pool_bound(s);
  if (aligned16(cache_k) && aligned16(cache_v)) {
    const int page_vec = page / 8;
    const int slice_vec = 4 * kThreads;  // 16 KiB of K and of V per workgroup
    const int slices = (page_vec + slice_vec - 1) / slice_vec;
    copy_pages_kernel<uint4><<<dim3(count, slices), kThreads, 0, st>>>(
        reinterpret_cast<uint4*>(cache_k), reinterpret_cast<uint4*>(cache_v), src_pages,
        dst_pages, phys, page_vec, slice_vec);
  } else {
    const int slice = 16 * kThreads;  // 8 KiB of K and of V per workgroup
    copy_pages_kernel<uint16_t><<<dim3(count, (page + slice - 1) / slice), kThreads, 0, st>>>(
        cache_k, cache_v, src_pages, dst_pages, phys, page, slice);
  }
  return hipGetLastError();
}

extern "C" int bc_write_prefix(bc_shape s, const bc_half* k, const bc_half* v,
                               long long k_token_stride, long long k_head_stride,
                               long long v_token_stride, long long v_head_stride,
                               bc_half* cache_k, bc_half* cache_v, const int32_t* host_pages,
                               int tokens, bc_stream_t stream) {
  if (!k || !v || !cache_k || !cache_v || !host_pages || tokens < 0 || k_token_stride < 0 ||
      k_head_stride < 0 || v_token_stride < 0 || v_head_stride < 0 ||
      (s.dim != 64 && s.dim != 128))
    return BC_ERROR_INVALID_VALUE;
  if (s.kv_heads < 1) return BC_SUCCESS;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int phys = pool_bound(s);
  const bool vec = aligned16(k) && aligned16(v) && aligned16(cache_k) && aligned16(cache_v) &&
                   (k_token_stride | k_head_stride | v_token_stride | v_head_stride) % 8 == 0;
  IntList list;
  for (int t0 = 0; t0 < tokens; t0 += kListInts * BC_PAGE_SIZE) {
    const int n = tokens - t0 < kListInts * BC_PAGE_SIZE ? tokens - t0 : kListInts * BC_PAGE_SIZE;
    const int pages = (n + BC_PAGE_SIZE - 1) / BC_PAGE_SIZE;
    for (int i = 0; i < pages; ++i) list.v[i] = host_pages[t0 / BC_PAGE_SIZE + i];
    const dim3 grid(pages, BC_PAGE_SIZE / kSliceTokens);
    const bc_half* kt = k + (long long)t0 * k_token_stride;
    const bc_half* vt = v + (long long)t0 * v_token_stride;
    if (vec)
      write_prefix_kernel<uint4><<<grid, kThreads, 0, st>>>(
          reinterpret_cast<const uint4*>(kt), reinterpret_cast<const uint4*>(vt),
          k_token_stride / 8, k_head_stride / 8, v_token_stride / 8, v_head_stride / 8,
          reinterpret_cast<uint4*>(cache_k), reinterpret_cast<uint4*>(cache_v), n, phys,
          s.kv_heads * s.dim / 8, s.dim / 8, list);
    else
      write_prefix_kernel<uint16_t><<<grid, kThreads, 0, st>>>(
          kt, vt, k_token_stride, k_head_stride, v_token_stride, v_head_stride, cache_k, cache_v,
          n, phys, s.kv_heads * s.dim, s.dim, list);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    if (n < kListInts * BC_PAGE_SIZE) break;  // t0 + the step may overflow
  }
  return BC_SUCCESS;
}

extern "C" int bc_write_ints(int32_t* dst, const int32_t* host_values, int count,
                             bc_stream_t stream) {
  if (!dst || !host_values || count < 0) return BC_ERROR_INVALID_VALUE;
  IntList list;
  for (int at = 0; at < count; at += kListInts) {
    const int n = count - at < kListInts ? count - at : kListInts;
    for (int i = 0; i < n; ++i) list.v[i] = host_values[at + i];
    write_ints_kernel<<<dim3(1), kThreads, 0, reinterpret_cast<hipStream_t>(stream)>>>(dst + at, n,
                                                                                      list);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    if (n < kListInts) break;  // at + the step may overflow
  }
  return BC_SUCCESS;
}

extern "C" const char* bc_version(void) {
  return "branchcraft-mi355x 0.2 (gfx950)";
}
