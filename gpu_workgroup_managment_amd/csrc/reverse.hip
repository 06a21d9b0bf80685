// reverse.hip -- the in-edge CSR of a resident graph (Pannotia SSSP / BC, BFS
// bottom-up): its edges sorted by target on the device, in the order of
// parseCOO_transpose's stable sort.
#include "apps_internal.hpp"

#include <algorithm>
#include <vector>

using namespace wgm;

namespace wgm {

// Stable least-significant-digit radix sort of (target, source, weight): per
// pass the digit counts of each tile, one exclusive scan over them digit by
// digit, and the move. A wave ranks its edges of equal digits by ballots, the
// workgroup's waves by a prefix over their counts, so the order within a digit
// is kept. Bound: 28 bytes an edge and pass, written in runs of a tile's edges
// of a digit. First BFS of a graph, RMAT scale 20 (1.6e7 weighted edges, three
// passes): 174 -> 2.0 ms with all allocations (by counting on the host between
// two copies before); RMAT 17: 7.9 -> 0.40; ER 2^16 of degree 16: 3.8 -> 0.36.
constexpr int kSortWg = 1024;
constexpr int kSortPer = 16;                     // edges a thread takes in turn
constexpr int kSortTile = kSortWg * kSortPer;
constexpr int kSortBits = 8;                     // digit width, at most
constexpr int kSortBins = 1 << kSortBits;

struct SortEdges {
  int32_t* key;  // target
  int32_t* src;
  int32_t* wt;   // null: unweighted
};

// Source of every out-edge.
__global__ void k_sort_sources(const int32_t* row_ptr, int n, int64_t m, int32_t* src) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m; e += stride) src[e] = row_of(row_ptr, n, e);
}

__global__ void __launch_bounds__(kSortWg) k_sort_count(const int32_t* key, int64_t m, int shift, int mask, int* counts) {
  __shared__ int s_bin[kSortBins];
  const int tid = threadIdx.x;
  if (tid < kSortBins) s_bin[tid] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll
  for (int k = 0; k < kSortPer; k++) {
    const int64_t e = base + k * kSortWg + tid;
    if (e < m) __hip_atomic_fetch_add(&s_bin[(key[e] >> shift) & mask], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __syncthreads();
  if (tid <= mask) counts[(int64_t)tid * gridDim.x + blockIdx.x] = s_bin[tid];
}

// Exclusive prefix sums of count (a multiple of 4) integers, by one workgroup.
__global__ void __launch_bounds__(kSortWg) k_sort_scan(int* counts, int64_t count) {
  __shared__ int s_wave[17];
  int carry = 0;
  for (int64_t b = 0; b < count / 4; b += kSortWg) {
    const int64_t i = b + threadIdx.x;
    int4 c = i < count / 4 ? ((int4*)counts)[i] : int4{0, 0, 0, 0};
    int total;
    int at = carry + wg_exclusive_scan(c.x + c.y + c.z + c.w, s_wave, &total);
    const int4 o{at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z};
    if (i < count / 4) ((int4*)counts)[i] = o;
    carry += total;
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kSortWg) k_sort_move(SortEdges in, SortEdges out, int64_t m, int shift, int bits,
                                                      const int* counts) {
  __shared__ int s_base[kSortBins];
  __shared__ int s_wave[kSortWg / 64][kSortBins];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, bins = 1 << bits;
  if (tid < bins) s_base[tid] = counts[(int64_t)tid * gridDim.x + blockIdx.x];
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
  for (int k = 0; k < kSortPer; k++) {
    for (int i = tid; i < kSortWg / 64 * kSortBins; i += kSortWg) (&s_wave[0][0])[i] = 0;
    const int64_t e = base + k * kSortWg + tid;
    const bool on = e < m;
    const int key = on ? in.key[e] : 0, src = on ? in.src[e] : 0, wt = on && in.wt ? in.wt[e] : 0;
    const int bin = (key >> shift) & (bins - 1);
    unsigned long long peers = __ballot(on);
    for (int b = 0; b < bits; b++) {
      const bool set = (bin >> b) & 1;
      const unsigned long long have = __ballot(set);
      peers &= set ? have : ~have;
    }
    const int rank = __popcll(peers & ((1ull << lane) - 1ull));
    __syncthreads();
    if (on && rank == 0) s_wave[wave][bin] = __popcll(peers);
    __syncthreads();
    if (tid < bins) {
      int at = s_base[tid];
#pragma unroll
      for (int w = 0; w < kSortWg / 64; w++) {
        const int c = s_wave[w][tid];
        s_wave[w][tid] = at;
        at += c;
      }
      s_base[tid] = at;
    }
    __syncthreads();
    if (on) {
      const int at = s_wave[wave][bin] + rank;
      out.key[at] = key;
      out.src[at] = src;
      if (in.wt) out.wt[at] = wt;
    }
    __syncthreads();
  }
}

// Row starts by search in the sorted targets, and the weights' padding.
__global__ void k_sort_rows(const int32_t* key, int64_t m, int n, int32_t* rrow, int32_t* rwt, int64_t padded) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  for (int64_t v = tid; v <= n; v += stride) {
    int64_t lo = 0, hi = m;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (key[mid] < v) lo = mid + 1;
      else hi = mid;
    }
    rrow[v] = (int32_t)lo;
  }
  for (int64_t e = m + tid; rwt && e < padded; e += stride) rwt[e] = 0;
}

// Whether a vertex has an in-edge (and zeros up to `padded`), to be summed.
__global__ void k_row_flags(const int32_t* rrow, int n, int64_t padded, int32_t* id) {
  for (int64_t v = blockIdx.x * blockDim.x + threadIdx.x; v < padded; v += gridDim.x * blockDim.x)
    id[v] = v < n && rrow[v + 1] > rrow[v] ? 1 : 0;
}
__global__ void k_row_ids(const int32_t* rrow, int n, int32_t* id) {
  for (Span mine{blockIdx.x * blockDim.x + threadIdx.x, (uint32_t)n}; mine.has(); mine.next(gridDim.x * blockDim.x))
    if (rrow[mine.at + 1] == rrow[mine.at]) id[mine.at] = -1;
}

}  // namespace wgm

#define HIPCHK WGM_HIPCHK

namespace {

// On the host, by counting: graphs whose sort buffers (16 bytes an edge) find
// no room. (Slower at every size: first BFS of a graph of 1024 edges 160 us, 110
// with the sort.)
int reverse_on_host(wgm_graph* g, int32_t* rrow_out, int32_t* rcol_out, int32_t* rwt_out, size_t padded) {
  wgm_runtime* rt = g->rt;
  const int32_t n = g->n;
  const int64_t m = g->m;
  std::vector<int32_t> rp((size_t)n + 1), col((size_t)m), wt(g->wt ? (size_t)m : 0);
  HIPCHK(rt, hipMemcpy(rp.data(), g->row_ptr, sizeof(int32_t) * ((size_t)n + 1), hipMemcpyDeviceToHost));
  if (m) HIPCHK(rt, hipMemcpy(col.data(), g->col, sizeof(int32_t) * (size_t)m, hipMemcpyDeviceToHost));
  if (g->wt && m) HIPCHK(rt, hipMemcpy(wt.data(), g->wt, sizeof(int32_t) * (size_t)m, hipMemcpyDeviceToHost));
  std::vector<int32_t> rrow((size_t)n + 1, 0), rcol((size_t)m), rwt(g->wt ? padded : 0);
  for (int64_t e = 0; e < m; e++) rrow[(size_t)col[(size_t)e] + 1]++;
  for (int32_t v = 0; v < n; v++) rrow[(size_t)v + 1] += rrow[(size_t)v];
  std::vector<int32_t> pos(rrow.begin(), rrow.end() - 1);
  for (int32_t u = 0; u < n; u++)
    for (int32_t e = rp[(size_t)u]; e < rp[(size_t)u + 1]; e++) {
      const int32_t p = pos[(size_t)col[(size_t)e]]++;
      rcol[(size_t)p] = u;
      if (g->wt) rwt[(size_t)p] = wt[(size_t)e];
    }
  HIPCHK(rt, hipMemcpy(rrow_out, rrow.data(), sizeof(int32_t) * ((size_t)n + 1), hipMemcpyHostToDevice));
  if (m) HIPCHK(rt, hipMemcpy(rcol_out, rcol.data(), sizeof(int32_t) * (size_t)m, hipMemcpyHostToDevice));
  if (g->wt && m) HIPCHK(rt, hipMemcpy(rwt_out, rwt.data(), sizeof(int32_t) * rwt.size(), hipMemcpyHostToDevice));
  return WGM_OK;
}

// Sorts into rcol, rwt and rrow; false if there is no room for the buffers.
bool reverse_on_device(wgm_graph* g, int32_t* rrow, int32_t* rcol, int32_t* rwt, size_t padded, hipError_t* e) {
  hipStream_t st = g->rt->stream;
  const int32_t n = g->n;
  const int64_t m = g->m;
  int bits = 1;
  while (bits < 31 && (1ll << bits) < n) bits++;
  const int passes = (bits + kSortBits - 1) / kSortBits, digit = (bits + passes - 1) / passes;
  const int nb = (int)(((m + kSortTile - 1) / kSortTile + 3) / 4 * 4);  // whole int4 per digit
  int32_t* buf = nullptr;
  const size_t words = (size_t)m * (g->wt ? 4 : 3) + 16, cwords = (size_t)nb << digit;
  *e = hipSuccess;
  if (hipMalloc((void**)&buf, sizeof(int32_t) * (words + cwords)) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  int* counts = buf;
  int32_t* p = buf + cwords;
  // the last pass writes to a, the one before it to b, and so on in turn; the
  // sources of the first lie where the second writes
  SortEdges a{p, rcol, rwt}, b{p + m, p + 2 * m, g->wt ? p + 3 * m : nullptr};
  SortEdges in{g->col, passes % 2 ? b.src : a.src, g->wt}, out = passes % 2 ? a : b;
  hipLaunchKernelGGL(k_sort_sources, dim3(4096), dim3(256), 0, st, g->row_ptr, n, m, in.src);
  for (int k = 0; k < passes; k++) {
    const int shift = k * digit;
    hipLaunchKernelGGL(k_sort_count, dim3(nb), dim3(kSortWg), 0, st, in.key, m, shift, (1 << digit) - 1, counts);
    hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(kSortWg), 0, st, counts, (int64_t)cwords);
    hipLaunchKernelGGL(k_sort_move, dim3(nb), dim3(kSortWg), 0, st, in, out, m, shift, digit, counts);
    in = out;
    out = in.key == a.key ? b : a;
  }
  hipLaunchKernelGGL(k_sort_rows, dim3(1024), dim3(256), 0, st, a.key, m, n, rrow, rwt, (int64_t)padded);
  *e = hipGetLastError();
  if (*e == hipSuccess) *e = hipStreamSynchronize(st);
  (void)hipFree(buf);
  return true;
}

}  // namespace

// The graph's in-edge CSR (sources ascending within a row), built on first use
// and kept resident; the weights padded with zeros to a multiple of kRwtPad.
int wgm_graph_in_edges(wgm_graph* g) {
  if (g->rrow) return WGM_OK;
  wgm_runtime* rt = g->rt;
  const size_t n = (size_t)g->n, m = (size_t)g->m, padded = (m + kRwtPad - 1) / kRwtPad * kRwtPad;
  int32_t *rrow = nullptr, *rcol = nullptr, *rwt = nullptr;
  auto alloc = [&](int32_t** p, size_t count) { return hipMalloc((void**)p, sizeof(int32_t) * std::max<size_t>(count, 1)); };
  hipError_t e = alloc(&rrow, n + 1);
  if (e == hipSuccess) e = alloc(&rcol, m);
  if (e == hipSuccess && g->wt) e = alloc(&rwt, padded);
  int rc = e == hipSuccess ? WGM_OK : wgm_hip_fail(rt, e, "hipMalloc(in-edge CSR)");
  if (!rc) {
    if (g->m > 0 && reverse_on_device(g, rrow, rcol, rwt, padded, &e)) {
      if (e != hipSuccess) rc = wgm_hip_fail(rt, e, "in-edge sort");
    } else {
      rc = reverse_on_host(g, rrow, rcol, rwt, padded);
    }
  }
  if (rc) {
    for (int32_t* p : {rrow, rcol, rwt})
      if (p) (void)hipFree(p);
    return rc;
  }
  g->rrow = rrow;
  g->rcol = rcol;
  g->rwt = rwt;
  return WGM_OK;
}

// Numbers the vertices with an in-edge in order: id[v], -1 for the others (id
// holds wgm_row_id_words(n) integers); *rows: how many.
size_t wgm_row_id_words(int32_t n) { return ((size_t)n + 4) / 4 * 4; }
int wgm_row_ids(wgm_graph* g, int32_t* id, int32_t* rows) {
  wgm_runtime* rt = g->rt;
  const int64_t padded = (int64_t)wgm_row_id_words(g->n);
  hipLaunchKernelGGL(k_row_flags, dim3(1024), dim3(256), 0, rt->stream, g->rrow, g->n, padded, id);
  hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(kSortWg), 0, rt->stream, id, padded);
  hipLaunchKernelGGL(k_row_ids, dim3(1024), dim3(256), 0, rt->stream, g->rrow, g->n, id);
  HIPCHK(rt, hipGetLastError());
  HIPCHK(rt, hipMemcpyAsync(rows, id + g->n, sizeof(int32_t), hipMemcpyDeviceToHost, rt->stream));
  HIPCHK(rt, hipStreamSynchronize(rt->stream));
  return WGM_OK;
}
