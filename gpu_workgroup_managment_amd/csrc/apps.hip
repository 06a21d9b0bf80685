// apps.hip -- device-resident graphs and the standalone persistent apps.
//
// Plays the role of the reference's persistent-app plugins plus run_persistent:
// init_persistent_app_for_occupancy uploads the graph, reset_persistent_task
// re-initialises state, the driver launches the standalone kernel, waits on the
// handshake and check_persistent_task reads the result back
// (src/lonestar/graph_apps/bfs/bfs.h:209-370, src/pannotia/graph_apps/color/color.h:41-195,
// src/pannotia/graph_apps/mis/mis.h:40-202, src/host_skeleton/skel.cpp:250-385).
// Unlike the reference, a reset never re-uploads the graph: graph arrays stay
// resident and only the per-run state is re-initialised on the device.

#include "apps_internal.hpp"
#include "low_degree.hpp"

#include <algorithm>
#include <cstring>
#include <utility>

using namespace wgm;

namespace wgm {

// ====================================================== standalone kernels
// Shape of each (standalone.cl, e.g. src/lonestar/graph_apps/bfs/device/standalone.cl:247-320):
// discovery; host handshake; barrier; the application loop with global
// barriers (here the XCD-aware two-level barrier); retire.

// Band widths of the standalone SSSP's near-far bands for weights in
// [1, 255]: wide on graphs of out-degree <= 4 (long, narrow traversals: fewer
// levels), narrower on the others (short, wide ones: less rework). Measured on
// RMAT scale 20 (ef 16), push direction, 1024 x 64 workgroups, four edges per
// thread per pass and the heavy entries claimed as one list: 3.32 ms at 12
// (78 levels), 3.09 at 16, 2.83 at 32, 2.76 at 48, 2.66 at 96, 2.65 at 128
// (18 levels), 2.70 at 192 and 256, 2.67 at 512. With one edge per pass and
// the heavy entries claimed one by one, 16 had been best (6.32 ms at 256
// workgroups; 7.21 at 64, 8.24 at 1024): wide levels then cost more.
constexpr uint32_t kStandaloneDelta = 1024;
constexpr uint32_t kStandaloneDeltaHighDegree = 128;

// BFS / SSSP over the whole grid as one team (run_team): state shared through
// agent-scope atomics, so the per-level two-level barrier skips its L2
// write-back and invalidation (which would refetch the graph every level);
// SSSP queue entries carry distance tags and run in near-far bands.
template <bool SSSP>
__global__ void __launch_bounds__(1024) k_frontier(Ctl c, GraphDev g, FrontierDev s, NearFar nf, int src,
                                                   int* iters_out) {
  extern __shared__ int lds[];
  Team t;
  if (!standalone_begin(c, t)) return;
  run_team<SSSP, SSSP ? kEdgeSlots : 1, true>(g, s, nf, src, t.id, t.n, lds, iters_out,
                                              [&]() { xcd_barrier<false>(c, t); },
                                              lds + standalone_pass_lds_bytes(SSSP, blockDim.x) / 4);
  clock_end(c, t.id);
  standalone_retire(c);
}

// BFS / push SSSP on a low-degree graph of narrow levels (a mesh or road
// network of up to kLowMaxN vertices): one workgroup runs the degree-bounded
// step of the batched launch, its queues, visited or far bits and combine
// tables in LDS, on packed rows (k_low_rows). A team's cross-workgroup barrier
// costs more than a narrow level's work. Bound: two dependent loads and one or
// two workgroup barriers a level (1.1 us BFS, 2.2 us SSSP).
// Rule: no edge spans more than kLowSpan places of the (circular) vertex
// order, so that k levels reach at most 2 k kLowSpan + 1 vertices; or the whole
// graph is small. Kernel times, team -> one workgroup, 64 x 512: 361 x 415 grid
// BFS 3508 -> 604 us, SSSP 7293 -> 2193; 10^5 vertices of 4 random edges within
// span 300: 2608 -> 408 and 6428 -> 1455, span 1000: 502 -> 243 and 1392 ->
// 1422, so the line lies at 768; random targets, 8192 vertices: 75 -> 32 and
// 209 -> 122, 16384: 93 -> 50 and 254 -> 237, 20000: SSSP 272 -> 300 and more,
// so it lies at 16384. Whole calls, 361 x 415 SSSP: 8093 -> 2507 us.
constexpr int32_t kLowSpan = 768;
constexpr int32_t kLowAnySpan = 16384;
constexpr int32_t kLowMaxN = 32 * kFarBitWords;
// Band width of the low-degree SSSP (weights in [0, 255]), as in the batched
// launch.
constexpr uint32_t kLowDelta = 512;

template <bool SSSP>
__global__ void __launch_bounds__(1024) k_low(Ctl c, GraphDev g, FrontierDev s, NearFar nf, int src,
                                              const uint32_t* ell, int* iters_out) {
  extern __shared__ __attribute__((aligned(16))) int lds_low[];  // the combine tables hold 64-bit words
  __shared__ int s_cnt[3];
  Team t;
  if (!standalone_begin(c, t)) return;
  if (t.id == 0) {
    nf.delta = SSSP ? kLowDelta : 0u;
    if constexpr (SSSP) run_low_comb(g, s, nf, src, lds_low, s_cnt, iters_out, ell);
    else run_low<false, kLowDegree, kLowSlots, true>(g, s, nf, src, lds_low, s_cnt, iters_out, true, ell);
    __syncthreads();
    if (threadIdx.x == 0) clock_end(c, 0);
  }
  standalone_retire(c);
}

// Packed rows of a low-degree graph: kLowDegree words a vertex, (target << 8) |
// weight, kEllNone past the degree. *flags: bit 0 where an edge spans more than
// kLowSpan of more than kLowAnySpan vertices, bit 1 where a weight does not fit.
__global__ void k_low_rows(GraphDev g, uint32_t* ell, int* flags) {
  int bad = 0;
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < g.n; v += gridDim.x * blockDim.x) {
    const int beg = g.row_ptr[v], deg = g.row_ptr[v + 1] - beg;
#pragma unroll
    for (int k = 0; k < kLowDegree; k++) {
      const int u = k < deg ? g.col[beg + k] : v, d = u > v ? u - v : v - u;
      const uint32_t w = k < deg && g.wt ? (uint32_t)g.wt[beg + k] : 0u;
      bad |= (g.n > kLowAnySpan && min(d, g.n - d) > kLowSpan ? 1 : 0) | (w > 255u ? 2 : 0);
      ell[(size_t)v * kLowDegree + k] = k < deg ? ((uint32_t)u << 8) | (w & 255u) : kEllNone;
    }
  }
  if (bad) __hip_atomic_fetch_or(flags, bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Colouring without rounds. The rounds give a vertex the colour 1 + the
// largest colour among its neighbours of priority not below its own (1
// without one, or with exactly one neighbour), whenever each is reached, so
// the workgroups sweep their open vertices on their own until none is left:
// a vertex takes its colour once its last blocker has one, and colours travel
// through agent-scope accesses, which need no barrier. Two barriers remain:
// after the first pass, which writes every state, and before the round count,
// which is what the rounds' stop flag gives -- the largest colour R, or R + 1
// where a vertex coloured last, with more than one neighbour, has a neighbour
// coloured last too (possible where an edge has no reverse).
// Every participant is resident and the highest open vertex is never blocked,
// so the sweeps end.
// Bound: the first pass by the graph's bytes, then the longest chain of
// dependent colours (one trip beyond the L2 each) and the sweeps' list
// traffic. 2048^2 grid, 14 colours, 256 x 1024, kernel: 410 us in rounds (of
// about 12 us each for draining the stores, the slowest workgroup and the
// barrier), 285 us here.
// wl: two lists of n entries (16 bytes with LONG, the graphs with rows of more
// than kTopoEdges edges, 8 without); a workgroup uses [lo, hi) of each.
template <bool LONG>
__global__ void __launch_bounds__(1024) k_color(Ctl c, GraphDev g, int32_t* color, void* wl, int* iters_out) {
  extern __shared__ int lds[];
  __shared__ int s_cnt[2];
  __shared__ int s_n[2];
  __shared__ int s_top;
  Team t;
  if (!standalone_begin(c, t)) return;
  int lo, hi;
  if (LONG) balanced_range(g, t.id, t.n, s_n, &lo, &hi);
  else block_range(g.n, t.id, t.n, &lo, &hi);
  if (threadIdx.x == 0) s_cnt[0] = s_cnt[1] = s_top = 0;
  __syncthreads();
  const size_t half = (size_t)g.n * (LONG ? sizeof(int4) : sizeof(int2));
  int top = 0;  // largest colour this thread gave
  auto decide = [&](int v, int acc) {
    st_agent(&color[v], acc + 1);
    top = max(top, acc + 1);
  };
  auto keep = [&](int v) { st_agent(&color[v], -1); };
  open_pass<LONG>(g, FirstProbe<true>{g.prio}, true, lo, hi - lo, nullptr, wl, &s_cnt[0], lds, s_n, decide, keep);
  xcd_barrier<false>(c, t);
  int which = 0, cnt = __builtin_amdgcn_readfirstlane(s_cnt[0]);
  while (cnt > 0) {  // list `which` to the other, whose count was cleared a sweep ago
    open_pass<LONG>(g, ColorProbe{color, g.prio}, true, lo, cnt, (char*)wl + which * half,
                    (char*)wl + (1 - which) * half, &s_cnt[1 - which], lds, s_n, decide, keep);
    __syncthreads();
    const int left = __builtin_amdgcn_readfirstlane(s_cnt[1 - which]);
    if (threadIdx.x == 0) s_cnt[which] = 0;
    __syncthreads();
    if (left == cnt) spin_pause();
    cnt = left;
    which = 1 - which;
  }
  // the round count
  for (int o = 32; o > 0; o >>= 1) top = max(top, __shfl_xor(top, o, 64));
  if ((threadIdx.x & 63) == 0)
    __hip_atomic_fetch_max(&s_top, top, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  __syncthreads();
  int* largest = &c.lines[0];
  int* again = &c.lines[kLine];
  const int mine = s_top;
  if (threadIdx.x == 0) __hip_atomic_fetch_max(largest, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  xcd_barrier<false>(c, t);
  const int last = ld_relaxed(largest);
  if (mine == last) {
    const int lane = (int)threadIdx.x & 63;
    for (Span mine{(uint32_t)lo + (threadIdx.x & ~63u), (uint32_t)hi}; mine.has(); mine.next(blockDim.x)) {
      unsigned long long m = __ballot(ld_agent(&color[mine.until(lane + 1) - 1]) == last && mine.has(lane));
      for (; m; m &= m - 1) {  // the wave walks each row
        const int v = (int)mine.at + __ffsll((long long)m) - 1;
        const int beg = g.row_ptr[v], end = g.row_ptr[v + 1];
        if (end - beg == 1) continue;
        bool hit = false;
        for (Span row{(uint32_t)beg + lane, (uint32_t)end}; row.has(); row.next(64))
          hit |= ld_agent(&color[g.col[row.at]]) == last;
        if (hit) st_relaxed(again, 1);
      }
    }
  }
  xcd_barrier<false>(c, t);
  clock_end(c, t.id);
  if (t.id == 0 && threadIdx.x == 0) *iters_out = last + ld_relaxed(again);
  standalone_retire(c);
}

// Phase A moves the open vertices from the first list to the second, phase B
// those that stay open back to the first (first round: the whole range). Their
// counts are s_a and s_b, each cleared in the other phase.
template <bool LONG>
__global__ void __launch_bounds__(1024) k_mis(Ctl c, GraphDev g, int32_t* st, int32_t* s_out, void* wl,
                                             int* iters_out) {
  extern __shared__ int lds[];
  __shared__ int s_a, s_b;
  __shared__ int s_n[2];
  Team t;
  if (!standalone_begin(c, t)) return;
  int lo, hi;
  if (LONG) balanced_range(g, t.id, t.n, s_n, &lo, &hi);
  else block_range(g.n, t.id, t.n, &lo, &hi);
  if (threadIdx.x == 0) s_a = s_b = 0;
  __syncthreads();
  void* la = wl;
  void* lb = (char*)wl + (size_t)g.n * (LONG ? sizeof(int4) : sizeof(int2));
  int* flags = c.lines;
  int round = 1, cnt = hi - lo;
  for (;; round++) {
    // a vertex is open: not the last round
    if (cnt > 0 && threadIdx.x == 0) st_relaxed(&flags[(round % 3) * kLine], 1);
    mis_phase_a_wl<LONG>(g, st, s_out, round, lo, cnt, round == 1 ? nullptr : la, lb, &s_a, lds, s_n);
    if (t.id == 0 && threadIdx.x == 0) st_relaxed(&flags[((round + 1) % 3) * kLine], 0);
    xcd_barrier(c, t);
    if (ld_relaxed(&flags[(round % 3) * kLine]) == 0) break;
    const int left = __builtin_amdgcn_readfirstlane(s_a);  // scalar: the passes' loops hold barriers
    if (threadIdx.x == 0) s_b = 0;
    __syncthreads();
    if (LONG) mis_phase_b_long(g, st, round, lo, left, (const int4*)lb, (int4*)la, &s_b, lds, s_n);
    else mis_phase_b_low(g, st, round, lo, left, (const int2*)lb, (int2*)la, &s_b);
    xcd_barrier(c, t);
    cnt = __builtin_amdgcn_readfirstlane(s_b);
    if (threadIdx.x == 0) s_a = 0;
    __syncthreads();
  }
  clock_end(c, t.id);
  if (t.id == 0 && threadIdx.x == 0) *iters_out = round;
  standalone_retire(c);
}

// LONG: the graph has rows of more than kTopoEdges edges, which go on lists. A
// workgroup whose range's row starts, columns and lists fit `words` words of
// dynamic LDS holds them there for all iterations (a barrier leaves nothing of
// them in the caches, and each was a load that the next waited for); the
// others read them from memory, the lists from wl, two of n entries. Whole
// calls of 50 iterations, memory -> LDS: symmetrised RMAT scale 17 ef 16, 512 x
// 1024, 1255 -> 1098 us; ER n = 131072 of degree 8, 64 x 1024, 1127 -> 833; RMAT
// scale 19, whose ranges do not fit, 4054 -> 3994. Both forms
// share one resource class (64 VGPRs, no scratch): the grid is sized on the form
// without.
template <bool LONG>
__global__ void __launch_bounds__(1024, 8) k_pagerank(Ctl c, GraphDev g, float* c0, float* c1, float* rank,
                                                   float damping, float base, float r0, int iters, int32_t* wl,
                                                   int words, int* iters_out) {
  extern __shared__ __attribute__((aligned(16))) int lds_pr[];
  __shared__ int s_range[2];
  __shared__ int s_cnt[3];
  __shared__ float s_seg[kPrSegs];
  Team t;
  if (!standalone_begin(c, t)) return;
  int lo, hi;
  if (LONG) {
    if (threadIdx.x < 3) s_cnt[threadIdx.x] = 0;
    balanced_range(g, t.id, t.n, s_range, &lo, &hi);
  } else {
    block_range(g.n, t.id, t.n, &lo, &hi);
  }
  auto run = [&](const auto& rows) {
    xcd_barrier(c, t);
    for (int it = 0; it < iters; it++) {
      const float* cin = (it & 1) ? c1 : c0;
      float* cout = (it & 1) ? c0 : c1;
      pagerank_pass<LONG>(rows, cin, cout, rank, damping, base, it == iters - 1, lo, hi, s_cnt, s_seg);
      xcd_barrier(c, t);
    }
  };
  pagerank_init(g, c0, r0, lo, hi);
  if constexpr (LONG) {
    const int nr = hi - lo;
    const int e0 = __builtin_amdgcn_readfirstlane(g.row_ptr[lo]);
    const int ne = __builtin_amdgcn_readfirstlane(g.row_ptr[hi]) - e0;
    const int n2 = ne / kPrSeg;  // rows of more than kPrSeg edges at most
    if ((long long)ne + 2 * (long long)nr + 1 + n2 <= words) {
      lds_i32* mem = (lds_i32*)lds_pr;
      const PrRows<lds_i32*> rows{mem + ne, mem, mem + ne + nr + 1, mem + ne + 2 * nr + 1, lo, 0};
      const int bd = blockDim.x;
#pragma unroll 4
      for (int i = threadIdx.x; i < ne; i += bd) mem[i] = g.col[e0 + i];
      for (int i = threadIdx.x; i <= nr; i += bd) rows.row_ptr[i] = g.row_ptr[lo + i] - e0;
      __syncthreads();
      pagerank_lists(rows, lo, hi, s_cnt);
      run(rows);
    } else {
      const PrRows<int32_t*> rows{(int32_t*)g.row_ptr, (int32_t*)g.col, wl, wl + g.n, 0, lo};
      pagerank_lists(rows, lo, hi, s_cnt);
      run(rows);
    }
  } else {
    run(PrRows<const int32_t*>{g.row_ptr, g.col, nullptr, nullptr, 0, 0});
  }
  clock_end(c, t.id);
  if (t.id == 0 && threadIdx.x == 0) *iters_out = iters;
  standalone_retire(c);
}

// PageRank of a graph of out-degree <= 4 whose edges span less than 2^15 places
// of the vertex order (a mesh): the rows as four 16-bit steps from the vertex,
// kNearNone past the degree. Bound of the CSR form: 28 bytes a vertex and
// iteration, 20 of them the unchanging rows (2048 x 2048 grid, 512 x 1024: 27.5
// us an iteration at 4.3 TB/s). The first `held` rows of a workgroup's range
// stay in LDS for all iterations, the others are 8 bytes: 15.2 us an iteration,
// about a third of it the barrier with the write-back of the contributions (50
// iterations, kernel: 1395 -> 790 us; 64 x 1024, where the LDS holds a third of the
// rows: 4919 -> 2646). The sums and their order are the CSR form's, bit for bit.
constexpr int kNearNone = -32768;
__global__ void k_near_rows(GraphDev g, uint2* rows, int* far) {
  bool bad = false;
  for (Span mine{blockIdx.x * blockDim.x + threadIdx.x, (uint32_t)g.n}; mine.has(); mine.next(gridDim.x * blockDim.x)) {
    const int v = (int)mine.at, beg = g.row_ptr[v], deg = g.row_ptr[v + 1] - beg;
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int step = k < deg ? g.col[beg + k] - v : kNearNone;
      bad |= k < deg && (step <= kNearNone || step > 32767);
      w[k] = (uint32_t)step & 0xffffu;
    }
    rows[v] = make_uint2(w[0] | w[1] << 16, w[2] | w[3] << 16);
  }
  if (bad) st_relaxed(far, 1);
}

__global__ void __launch_bounds__(1024, 8) k_pagerank_near(Ctl c, GraphDev g, const uint2* rows, int held, float* c0,
                                                        float* c1, float* rank, float damping, float base, float r0,
                                                        int iters, int* iters_out) {
  extern __shared__ __attribute__((aligned(16))) int lds_rows[];
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
  lds_u32x2* mine = (lds_u32x2*)lds_rows;
  Team t;
  if (!standalone_begin(c, t)) return;
  int lo, hi;
  block_range(g.n, t.id, t.n, &lo, &hi);
  const int bd = blockDim.x;
  held = min(held, hi - lo);
  for (int i = threadIdx.x; i < held; i += bd) mine[i] = ((const u32x2*)rows)[lo + i];
  pagerank_init(g, c0, r0, lo, hi);
  xcd_barrier(c, t);
  constexpr int U = 4;
  for (int it = 0; it < iters; it++) {
    const float* cin = (it & 1) ? c1 : c0;
    float* cout = it == iters - 1 ? rank : (it & 1) ? c0 : c1;
    const bool last = it == iters - 1;
    auto rows_of = [&](int a, int z, auto&& row) {
      for (Span place{(uint32_t)a + threadIdx.x, (uint32_t)z}; place.has(); place.next(U * bd)) {
        uint32_t i[U];  // beyond the range: its last row
#pragma unroll
        for (int k = 0; k < U; k++) i[k] = min(place.at + k * bd, place.stop - 1u);
        u32x2 r[U];
#pragma unroll
        for (int k = 0; k < U; k++) r[k] = row(i[k]);
        float cu[U][4];
#pragma unroll
        for (int k = 0; k < U; k++)
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const int step = (int)(int16_t)(r[k][j >> 1] >> (16 * (j & 1)));
            cu[k][j] = step != kNearNone ? cin[lo + i[k] + step] : 0.0f;
          }
#pragma unroll
        for (int k = 0; k < U; k++) {
          float sum = 0.0f;
          int deg = 0;
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const bool edge = ((r[k][j >> 1] >> (16 * (j & 1))) & 0xffffu) != 0x8000u;
            sum = edge ? sum + cu[k][j] : sum;
            deg += edge ? 1 : 0;
          }
          const float x = __builtin_fmaf(damping, sum, base);
          if (place.has(k * bd)) cout[lo + i[k]] = last ? x : deg > 0 ? x / (float)deg : 0.0f;
        }
      }
    };
    rows_of(0, held, [&](uint32_t i) { return mine[i]; });
    rows_of(held, hi - lo, [&](uint32_t i) { return ((const u32x2*)rows)[lo + i]; });
    xcd_barrier(c, t);
  }
  clock_end(c, t.id);
  if (t.id == 0 && threadIdx.x == 0) *iters_out = iters;
  standalone_retire(c);
}

}  // namespace wgm


#define fail wgm_fail
#define HIPCHK WGM_HIPCHK

namespace {

template <typename T>
int dev_alloc(wgm_runtime* rt, T** p, size_t count) {
  if (*p) return WGM_OK;
  hipError_t e = hipMalloc((void**)p, (count ? count : 1) * sizeof(T));
  if (e != hipSuccess) {
    *p = nullptr;
    return wgm_hip_fail(rt, e, "hipMalloc(graph state)");
  }
  return WGM_OK;
}

// Words of the graph's worklists: two lists of n entries of 16 bytes on graphs
// with rows of more than kTopoEdges edges (PageRank takes the first 2 n
// words), 8 bytes on the others.
size_t wl_words(const wgm_graph* g) { return (g->maxdeg > kTopoEdges ? 8 : 4) * (size_t)g->n; }

int launch_prologue(wgm_runtime* rt, int kernel, const wgm_launch* lc, int* grid, int* wg) {
  wgm_launch def{256, 0, 0, 0};
  const wgm_launch& l = lc ? *lc : def;
  *wg = l.wg_size > 0 ? l.wg_size : 256;
  int rc = wgm_resolve_resident(rt, kernel, *wg, l.num_wgs, grid);
  if (rc) return rc;
  rc = wgm_reset_ctl(rt, 0, l.handshake ? 1 : 0);
  if (rc) return rc;
  HIPCHK(rt, hipEventRecord(rt->ev0, rt->stream));
  return WGM_OK;
}

// The finish of an app whose result is n elements from `src`.
template <typename T>
int launch_epilogue(wgm_runtime* rt, const wgm_launch* lc, wgm_graph* g, const T* src, T* dst, wgm_run_stats* st) {
  HIPCHK(rt, hipGetLastError());
  AppOut out;
  out.iters = g->iters;
  out.src = src;
  out.dst = dst;
  out.bytes = sizeof(T) * (size_t)g->n;
  return wgm_finish_app(rt, lc ? lc->handshake : 0, out, st);
}

}  // namespace

GraphDev wgm_graph_view(const wgm_graph* g) {
  GraphDev v{};
  v.row_ptr = g->row_ptr;
  v.col = g->col;
  v.wt = g->wt;
  v.prio = g->prio;
  v.n = g->n;
  v.m = (int32_t)g->m;
  return v;
}

int wgm_graph_frontier_state(wgm_graph* g, bool sssp, FrontierDev* s) {
  wgm_runtime* rt = g->rt;
  int rc = dev_alloc(rt, &g->dist, g->n);
  if (!rc) rc = dev_alloc(rt, &g->q0, g->n + 1);
  if (!rc) rc = dev_alloc(rt, &g->q1, g->n + 1);
  if (!rc) rc = dev_alloc(rt, &g->counts, 3 * kLine);
  if (!rc && sssp) rc = dev_alloc(rt, &g->stamp, g->n);
  if (rc) return rc;
  s->dist = g->dist;
  s->stamp = sssp ? g->stamp : nullptr;
  s->q0 = g->q0;
  s->q1 = g->q1;
  s->counts = g->counts;
  return WGM_OK;
}

int wgm_graph_app_state(wgm_graph* g, int app) {
  wgm_runtime* rt = g->rt;
  int rc = WGM_OK;
  if (app == 1 || app == 2) rc = dev_alloc(rt, &g->i32a, g->n);
  if (!rc && app == 2) rc = dev_alloc(rt, &g->i32b, g->n);
  if (!rc && app == 3) rc = dev_alloc(rt, &g->f0, g->n);
  if (!rc && app == 3) rc = dev_alloc(rt, &g->f1, g->n);
  if (!rc && app == 3) rc = dev_alloc(rt, &g->f2, g->n);
  return rc;
}

// State of the standalone team traversal: queues of max(n, m) + 1 entries
// with distance tags for SSSP (a level queues at most one entry per
// relaxation), n + 1 for BFS; claim counters; near-far queues and flags.
static int team_frontier_state(wgm_graph* g, bool sssp, FrontierDev* s, NearFar* nf) {
  wgm_runtime* rt = g->rt;
  const int64_t cap = (sssp ? std::max<int64_t>(g->n, g->m) : (int64_t)g->n) + 1;
  if (g->tcap < cap) {  // a BFS-sized pair of queues cannot serve SSSP
    (void)hipFree(g->tq);
    (void)hipFree(g->tqa);
    g->tq = nullptr;
    g->tqa = nullptr;
    g->tcap = 0;
  }
  int rc = dev_alloc(rt, &g->dist, g->n);
  if (!rc) rc = dev_alloc(rt, &g->tq, 2 * (size_t)cap);
  if (!rc && sssp) rc = dev_alloc(rt, &g->tqa, 2 * (size_t)std::max<int64_t>(cap, g->tcap));
  if (!rc) rc = dev_alloc(rt, &g->counts, 3 * kLine);
  if (!rc) rc = dev_alloc(rt, &g->claims, 3 * kLine);
  if (!rc && sssp) rc = dev_alloc(rt, &g->far, 2 * ((size_t)g->n + 1));
  if (!rc && sssp) rc = dev_alloc(rt, &g->in_far, (size_t)g->n);
  if (!rc && sssp) rc = dev_alloc(rt, &g->fcnt, 3 * kLine);
  const size_t hcap = (size_t)(g->m / kHeavyMin) + 2;
  if (!rc) rc = dev_alloc(rt, &g->hv, hcap);
  if (!rc) rc = dev_alloc(rt, &g->hdu, hcap);
  if (!rc) rc = dev_alloc(rt, &g->hclaim, hcap);
  if (!rc) rc = dev_alloc(rt, &g->hcnt, 3 * kLine);
  if (rc) return rc;
  if (g->tcap < cap) g->tcap = cap;
  *s = FrontierDev{};
  s->dist = g->dist;
  s->q0 = g->tq;
  s->q1 = g->tq + g->tcap;
  s->qa0 = sssp ? g->tqa : nullptr;
  s->qa1 = sssp ? g->tqa + g->tcap : nullptr;
  s->counts = g->counts;
  s->claims = g->claims;
  s->hv = g->hv;
  s->hdu = g->hdu;
  s->hclaim = g->hclaim;
  s->hcnt = g->hcnt;
  s->fine = g->maxdeg > kFineDegree ? 1 : 0;
  *nf = NearFar{};
  if (sssp) {
    nf->q[0] = g->far;
    nf->q[1] = g->far + g->n + 1;
    nf->flag = g->in_far;
    nf->cnt = g->fcnt;
    nf->delta = wgm_standalone_delta(g->maxdeg);
  }
  return WGM_OK;
}

// Both forms of the colour and MIS kernels are launched with the long-row
// form's LDS, so that the grid found for one holds for the other.
template <bool SSSP>
static int frontier_lds(int wg) { return standalone_frontier_lds_bytes(SSSP, wg); }
static int scan_lds(int wg) { return scan_lds_bytes(wg); }

bool wgm_app_kernel_info(int kernel, KernelInfo* out) {
  switch (kernel) {
    case WGM_K_BFS: *out = KernelInfo{(const void*)&k_frontier<false>, frontier_lds<false>}; return true;
    case WGM_K_SSSP: *out = KernelInfo{(const void*)&k_frontier<true>, frontier_lds<true>}; return true;
    case WGM_K_COLOR: *out = KernelInfo{(const void*)&k_color<false>, scan_lds}; return true;
    case WGM_K_MIS: *out = KernelInfo{(const void*)&k_mis<false>, scan_lds}; return true;
    case WGM_K_PAGERANK: *out = KernelInfo{(const void*)&k_pagerank<false>, nullptr}; return true;
    default: return wgm_pannotia_kernel_info(kernel, out);
  }
}

// Discovery probe with the app kernel itself (im_exit set: every workgroup
// returns right after discovery and never reads its other arguments).
int wgm_app_probe(wgm_runtime* rt, int kernel, int grid, int wg_size) {
  const size_t lds = wgm_kernel_lds(kernel, wg_size);
  switch (kernel) {
    case WGM_K_BFS:
      hipLaunchKernelGGL(k_frontier<false>, dim3(grid), dim3(wg_size), lds, rt->stream, rt->ctl, GraphDev{},
                         FrontierDev{}, NearFar{}, 0, (int*)nullptr);
      return WGM_OK;
    case WGM_K_SSSP:
      hipLaunchKernelGGL(k_frontier<true>, dim3(grid), dim3(wg_size), lds, rt->stream, rt->ctl, GraphDev{},
                         FrontierDev{}, NearFar{}, 0, (int*)nullptr);
      return WGM_OK;
    case WGM_K_COLOR:
      hipLaunchKernelGGL(k_color<false>, dim3(grid), dim3(wg_size), lds, rt->stream, rt->ctl, GraphDev{},
                         (int32_t*)nullptr, (void*)nullptr, (int*)nullptr);
      return WGM_OK;
    case WGM_K_MIS:
      hipLaunchKernelGGL(k_mis<false>, dim3(grid), dim3(wg_size), lds, rt->stream, rt->ctl, GraphDev{},
                         (int32_t*)nullptr, (int32_t*)nullptr, (void*)nullptr, (int*)nullptr);
      return WGM_OK;
    case WGM_K_PAGERANK:
      hipLaunchKernelGGL(k_pagerank<false>, dim3(grid), dim3(wg_size), 0, rt->stream, rt->ctl, GraphDev{}, (float*)nullptr,
                         (float*)nullptr, (float*)nullptr, 0.f, 0.f, 0.f, 0, (int32_t*)nullptr, 0, (int*)nullptr);
      return WGM_OK;
    default:
      return wgm_pannotia_probe(rt, kernel, grid, wg_size);
  }
}

extern "C" {

int wgm_graph_create(wgm_runtime* rt, const wgm_csr* h, const uint32_t* prio, wgm_graph** out) {
  if (!rt || !h || !out) return fail(rt, WGM_ERR_INVALID, "NULL argument");
  if (h->n < 1 || h->m < 0 || h->m > INT32_MAX || !h->row_ptr || (h->m > 0 && !h->col))
    return fail(rt, WGM_ERR_INVALID, "bad CSR shape n=%d m=%lld", h->n, (long long)h->m);
  if (h->row_ptr[0] != 0 || h->row_ptr[h->n] != h->m)
    return fail(rt, WGM_ERR_INVALID, "row_ptr must start at 0 and end at m");
  int32_t maxdeg = 0;
  for (int32_t v = 0; v < h->n; v++) {
    if (h->row_ptr[v + 1] < h->row_ptr[v]) return fail(rt, WGM_ERR_INVALID, "row_ptr not monotone at %d", v);
    maxdeg = std::max(maxdeg, h->row_ptr[v + 1] - h->row_ptr[v]);
  }
  for (int64_t e = 0; e < h->m; e++)
    if (h->col[e] < 0 || h->col[e] >= h->n) return fail(rt, WGM_ERR_INVALID, "col[%lld] out of range", (long long)e);
  wgm_graph* g = new wgm_graph();
  g->rt = rt;
  g->n = h->n;
  g->m = h->m;
  g->maxdeg = maxdeg;
  auto bail = [&](int rc) { wgm_graph_destroy(g); return rc; };
  int rc = dev_alloc(rt, &g->row_ptr, (size_t)h->n + 1);
  if (!rc) rc = dev_alloc(rt, &g->col, (size_t)h->m);
  if (!rc && h->wt) rc = dev_alloc(rt, &g->wt, (size_t)h->m);
  if (!rc && prio) rc = dev_alloc(rt, &g->prio, (size_t)h->n);
  if (!rc) rc = dev_alloc(rt, &g->iters, 4);
  if (rc) return bail(rc);
  hipError_t e = hipMemcpy(g->row_ptr, h->row_ptr, sizeof(int32_t) * ((size_t)h->n + 1), hipMemcpyHostToDevice);
  if (e == hipSuccess && h->m) e = hipMemcpy(g->col, h->col, sizeof(int32_t) * (size_t)h->m, hipMemcpyHostToDevice);
  if (e == hipSuccess && h->wt && h->m) e = hipMemcpy(g->wt, h->wt, sizeof(int32_t) * (size_t)h->m, hipMemcpyHostToDevice);
  if (e == hipSuccess && prio) e = hipMemcpy(g->prio, prio, sizeof(uint32_t) * (size_t)h->n, hipMemcpyHostToDevice);
  if (e != hipSuccess) return bail(wgm_hip_fail(rt, e, "graph upload"));
  *out = g;
  return WGM_OK;
}

int wgm_graph_destroy(wgm_graph* g) {
  if (!g) return WGM_OK;
  wgm_pannotia_release(g);
  void* ptrs[] = {g->row_ptr, g->col, g->wt, g->prio, g->dist, g->stamp, g->q0, g->q1, g->counts,
                  g->i32a, g->i32b, g->f0, g->f1, g->f2, g->iters, g->tq, g->tqa, g->claims, g->far,
                  g->in_far, g->fcnt, g->hv, g->hdu, g->hclaim, g->hcnt, g->wl, g->ell, g->near_rows};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  delete g;
  return WGM_OK;
}

// Every array that the graph holds: itself, the layouts made from it and the
// apps' state.
int64_t wgm_graph_bytes(const wgm_graph* g) {
  if (!g) return 0;
  const int64_t n = g->n, m = g->m, heavy = m / kHeavyMin + 2;
  const std::pair<const void*, int64_t> arrays[] = {
      {g->row_ptr, 4 * (n + 1)}, {g->col, 4 * m}, {g->wt, 4 * m}, {g->prio, 4 * n}, {g->iters, 16},
      {g->near_rows, 8 * n}, {g->ell, 4 * kLowDegree * n},
      // frontier state
      {g->dist, 4 * n}, {g->stamp, 4 * n}, {g->q0, 4 * (n + 1)}, {g->q1, 4 * (n + 1)}, {g->counts, 12 * kLine},
      {g->tq, 8 * g->tcap}, {g->tqa, 8 * g->tcap}, {g->claims, 12 * kLine}, {g->far, 8 * (n + 1)}, {g->in_far, 4 * n},
      {g->fcnt, 12 * kLine}, {g->hv, 4 * heavy}, {g->hdu, 4 * heavy}, {g->hclaim, 4 * heavy}, {g->hcnt, 12 * kLine},
      // colour, MIS, PageRank
      {g->i32a, 4 * n}, {g->i32b, 4 * n}, {g->f0, 4 * n}, {g->f1, 4 * n}, {g->f2, 4 * n}, {g->wl, 4 * (int64_t)wl_words(g)}};
  int64_t b = wgm_pannotia_bytes(g);
  for (const auto& [p, bytes] : arrays)
    if (p) b += bytes;
  return b;
}

}  // extern "C"

uint32_t wgm_standalone_delta(int maxdeg) { return maxdeg > 4 ? kStandaloneDeltaHighDegree : kStandaloneDelta; }

// Enqueue the standalone frontier kernel (no wait, nothing allocated): chunked
// claims of one workgroup's width, heavy entries above heavy_threshold(wg);
// *iters_dev is the device cell the kernel writes its level count to.
int wgm_enqueue_frontier(wgm_runtime* rt, const GraphDev& g, FrontierDev s, const NearFar& nf, bool sssp, int src,
                         int grid, int wg, int* iters_dev) {
  s.chunk = wg;  // frontier entries a workgroup claims at a time
  s.heavy = heavy_threshold(wg);
  const size_t lds = standalone_frontier_lds_bytes(sssp, wg);
  if (sssp)
    hipLaunchKernelGGL(k_frontier<true>, dim3(grid), dim3(wg), lds, rt->stream, rt->ctl, g, s, nf, src, iters_dev);
  else
    hipLaunchKernelGGL(k_frontier<false>, dim3(grid), dim3(wg), lds, rt->stream, rt->ctl, g, s, nf, src, iters_dev);
  HIPCHK(rt, hipGetLastError());
  return WGM_OK;
}

int wgm_launch_frontier(wgm_runtime* rt, const GraphDev& g, FrontierDev s, const NearFar& nf, bool sssp, int src,
                        int grid, int wg, int handshake, const AppOut& out, wgm_run_stats* st) {
  int rc = wgm_reset_ctl(rt, 0, handshake ? 1 : 0);
  if (rc) return rc;
  HIPCHK(rt, hipEventRecord(rt->ev0, rt->stream));
  rc = wgm_enqueue_frontier(rt, g, s, nf, sssp, src, grid, wg, (int*)out.iters);
  return rc ? rc : wgm_finish_app(rt, handshake, out, st);
}

// The packed rows of a low-degree graph, laid out once, and whether BFS and the
// push SSSP take them (g->low, g->low_weights).
static int low_rows(wgm_runtime* rt, wgm_graph* g) {
  if (g->low_known) return WGM_OK;
  if (g->maxdeg > kLowDegree || g->n > kLowMaxN) {
    g->low_known = true;
    return WGM_OK;
  }
  int rc = dev_alloc(rt, &g->ell, (size_t)kLowDegree * (size_t)g->n);
  if (rc) return rc;
  int flags = 0;
  HIPCHK(rt, hipMemcpyAsync(g->iters, &flags, sizeof(int), hipMemcpyHostToDevice, rt->stream));
  hipLaunchKernelGGL(k_low_rows, dim3(256), dim3(256), 0, rt->stream, wgm_graph_view(g), g->ell, g->iters);
  HIPCHK(rt, hipMemcpyAsync(&flags, g->iters, sizeof(int), hipMemcpyDeviceToHost, rt->stream));
  HIPCHK(rt, hipStreamSynchronize(rt->stream));
  g->low = !(flags & 1);
  g->low_weights = !flags && g->wt;
  g->low_known = true;
  if (!g->low) {
    (void)hipFree(g->ell);
    g->ell = nullptr;
  }
  return WGM_OK;
}

// Workgroups where the caller leaves the number open, of the `fit` that can be
// resident. A barrier costs 6 us with 512 workgroups, 4 with 256, 2.5 with 64, and
// a pass over a small graph little else: a thread for every `each` units of cost
// (edges and rows (kRowCost), vertices for k_pagerank_near), from 65536 threads to
// 1024 a CU. (BFS and MIS hold no more than those in workgroups of 1024, in smaller
// ones up to 1.75 times as many.)
// Whole calls, all that fit -> by the rule:
// BFS, 1024 threads: ER n = 4097 of degree 8, 102 -> 94 us, RMAT 131072 ef 16, 148 ->
// 142; 512 threads: RMAT scale 20 ef 16, 374 -> 342, 1201 x 1303 grid, 24.4 -> 19.8
// ms; 256 threads: ER n = 4097, 214 -> 101.
// MIS, 1024 threads: ER n = 60001 of degree 8, 175 -> 139, 401^2 grid 170 -> 135, 801^2
// 254 -> 238; 256 threads: ER n = 60001, 395 -> 173, 524288 of 16, 656 -> 589, 2047^2
// grid 968 -> 894.
// PageRank, 50 iterations, 1024 threads: ER n = 4097 of degree 8, 434 -> 246, 30001
// of 16, 489 -> 365, 131072 of 8, 638 -> 542; four random edges a vertex, n = 5001,
// 421 -> 233; meshes, 401^2, 478 -> 299; 256 threads, ER 16001 of degree 8, 1161 ->
// 369.
constexpr int kFitBfs = 16;
constexpr int kFitMis = 32;
constexpr int kFitPr = 4;
static int fitted_grid(const wgm_runtime* rt, const wgm_launch* lc, int64_t cost, int each, int fit, int wg) {
  if (lc && lc->num_wgs > 0) return fit;
  const int64_t most = (int64_t)rt->info.num_cus * 1024;
  const int64_t threads = std::min(most, std::max<int64_t>(65536, cost / each));
  return (int)std::min<int64_t>(fit, (threads + wg - 1) / wg);
}
static int64_t rows_and_edges(const wgm_graph* g) { return g->m + kRowCost * (int64_t)g->n; }

// Enqueue k_low: the threads asked for, in workgroups of up to 1024 (one fits a
// CU beside its LDS).
static int enqueue_low(wgm_runtime* rt, const wgm_graph* g, const FrontierDev& s, const NearFar& nf, bool sssp, int src,
                       int grid, int wg) {
  const GraphDev view = wgm_graph_view(g);
  const long long threads = (long long)grid * wg;
  const int lwg = (int)std::min<long long>(1024, threads);
  const int lgrid = (int)std::min<long long>(threads / lwg, rt->info.num_cus);
  const size_t lds = sssp ? (size_t)kLowSsspLds : (size_t)low_bfs_lds_bytes(lwg);
  if (sssp)
    hipLaunchKernelGGL(k_low<true>, dim3(lgrid), dim3(lwg), lds, rt->stream, rt->ctl, view, s, nf, src, g->ell, g->iters);
  else
    hipLaunchKernelGGL(k_low<false>, dim3(lgrid), dim3(lwg), lds, rt->stream, rt->ctl, view, s, nf, src, g->ell, g->iters);
  HIPCHK(rt, hipGetLastError());
  return WGM_OK;
}

extern "C" {

static int run_frontier(wgm_runtime* rt, wgm_graph* g, int32_t src, const wgm_launch* lc, uint32_t* dist_out,
                        wgm_run_stats* st, bool sssp) {
  if (!rt || !g || g->rt != rt) return fail(rt, WGM_ERR_INVALID, "bad runtime/graph");
  if (src < 0 || src >= g->n) return fail(rt, WGM_ERR_INVALID, "source %d out of range", src);
  if (sssp && !g->wt) return fail(rt, WGM_ERR_INVALID, "SSSP needs edge weights");
  const int mode = lc ? lc->mode : WGM_SSSP_AUTO;
  if (mode < WGM_SSSP_AUTO || mode > WGM_SSSP_PULL) return fail(rt, WGM_ERR_INVALID, "unknown SSSP mode %d", mode);
  if (sssp && (mode == WGM_SSSP_PULL || (mode == WGM_SSSP_AUTO && g->maxdeg > 4))) {
    return wgm_sssp_pull(rt, g, src, lc, dist_out, st);
  }
  FrontierDev s{};
  NearFar nf{};
  int rc = team_frontier_state(g, sssp, &s, &nf);
  if (rc) return rc;
  const int kernel = sssp ? WGM_K_SSSP : WGM_K_BFS;
  const int wg = lc && lc->wg_size > 0 ? lc->wg_size : 256;
  int grid = 0;
  rc = wgm_resolve_resident(rt, kernel, wg, lc ? lc->num_wgs : 0, &grid);
  if (rc) return rc;
  rc = low_rows(rt, g);
  if (rc) return rc;
  const bool low = sssp ? g->low_weights : g->low;
  if (!sssp && !low) grid = fitted_grid(rt, lc, rows_and_edges(g), kFitBfs, grid, wg);
  GraphDev view = wgm_graph_view(g);
  if (!sssp && !low) {
    // BFS takes its wide levels bottom-up over the in-edges
    rc = wgm_graph_in_edges(g);
    if (rc) return rc;
    view.rrow = g->rrow;
    view.rcol = g->rcol;
  }
  const int handshake = lc ? lc->handshake : 0;
  AppOut out;
  out.iters = g->iters;
  out.reached = g->dist;
  out.g = view;
  out.src = g->dist;
  out.dst = dist_out;
  out.bytes = sizeof(uint32_t) * (size_t)g->n;
  if (!low) return wgm_launch_frontier(rt, view, s, nf, sssp, src, grid, wg, handshake, out, st);
  rc = wgm_reset_ctl(rt, 0, handshake ? 1 : 0);
  if (rc) return rc;
  HIPCHK(rt, hipEventRecord(rt->ev0, rt->stream));
  rc = enqueue_low(rt, g, s, nf, sssp, src, grid, wg);
  return rc ? rc : wgm_finish_app(rt, handshake, out, st);
}

int wgm_bfs(wgm_runtime* rt, wgm_graph* g, int32_t src, const wgm_launch* lc, uint32_t* dist_out,
            wgm_run_stats* st) {
  return run_frontier(rt, g, src, lc, dist_out, st, false);
}

int wgm_sssp(wgm_runtime* rt, wgm_graph* g, int32_t src, const wgm_launch* lc, uint32_t* dist_out,
             wgm_run_stats* st) {
  return run_frontier(rt, g, src, lc, dist_out, st, true);
}

int wgm_color(wgm_runtime* rt, wgm_graph* g, const wgm_launch* lc, int32_t* color_out, wgm_run_stats* st) {
  if (!rt || !g || g->rt != rt) return fail(rt, WGM_ERR_INVALID, "bad runtime/graph");
  if (!g->prio) return fail(rt, WGM_ERR_INVALID, "colouring needs vertex priorities");
  int rc = dev_alloc(rt, &g->i32a, g->n);
  if (!rc) rc = dev_alloc(rt, &g->wl, wl_words(g));
  if (rc) return rc;
  int grid = 0, wg = 0;
  rc = launch_prologue(rt, WGM_K_COLOR, lc, &grid, &wg);
  if (rc) return rc;
  hipLaunchKernelGGL(g->maxdeg > kTopoEdges ? k_color<true> : k_color<false>, dim3(grid), dim3(wg), scan_lds_bytes(wg),
                     rt->stream, rt->ctl, wgm_graph_view(g), g->i32a, (void*)g->wl, g->iters);
  return launch_epilogue(rt, lc, g, g->i32a, color_out, st);
}

int wgm_mis(wgm_runtime* rt, wgm_graph* g, const wgm_launch* lc, int32_t* s_out, wgm_run_stats* st) {
  if (!rt || !g || g->rt != rt) return fail(rt, WGM_ERR_INVALID, "bad runtime/graph");
  if (!g->prio) return fail(rt, WGM_ERR_INVALID, "MIS needs vertex priorities");
  int rc = dev_alloc(rt, &g->i32a, g->n);
  if (!rc) rc = dev_alloc(rt, &g->i32b, g->n);
  if (!rc) rc = dev_alloc(rt, &g->wl, wl_words(g));
  if (rc) return rc;
  int grid = 0, wg = 0;
  rc = launch_prologue(rt, WGM_K_MIS, lc, &grid, &wg);
  if (rc) return rc;
  grid = fitted_grid(rt, lc, rows_and_edges(g), kFitMis, grid, wg);
  hipLaunchKernelGGL(g->maxdeg > kTopoEdges ? k_mis<true> : k_mis<false>, dim3(grid), dim3(wg), scan_lds_bytes(wg),
                     rt->stream, rt->ctl, wgm_graph_view(g), g->i32a, g->i32b, (void*)g->wl, g->iters);
  return launch_epilogue(rt, lc, g, g->i32b, s_out, st);
}

// The 16-bit rows, laid out once per graph (g->near: 1 there, -1 none).
static int near_rows(wgm_runtime* rt, wgm_graph* g) {
  if (g->near) return WGM_OK;
  if (g->maxdeg > 4) {
    g->near = -1;
    return WGM_OK;
  }
  int rc = dev_alloc(rt, &g->near_rows, (size_t)g->n);
  if (rc) return rc;
  int far = 0;
  HIPCHK(rt, hipMemcpyAsync(g->iters, &far, sizeof(int), hipMemcpyHostToDevice, rt->stream));
  hipLaunchKernelGGL(k_near_rows, dim3(1024), dim3(256), 0, rt->stream, wgm_graph_view(g), g->near_rows, g->iters);
  HIPCHK(rt, hipMemcpyAsync(&far, g->iters, sizeof(int), hipMemcpyDeviceToHost, rt->stream));
  HIPCHK(rt, hipStreamSynchronize(rt->stream));
  if (far) {
    (void)hipFree(g->near_rows);
    g->near_rows = nullptr;
  }
  g->near = far ? -1 : 1;
  return WGM_OK;
}

// LDS of a workgroup where 2048 threads of a CU stay resident, or the one
// workgroup that each CU has.
static int lds_share(const wgm_runtime* rt, int grid, int wg) {
  return grid > rt->info.num_cus ? (160 << 10) / (2048 / wg) : 160 << 10;
}

// Rows that a workgroup holds in LDS: its range, within the share of a CU's 160
// KB that leaves 2048 threads (or the workgroup each CU has) resident.
static int near_held(const wgm_runtime* rt, int n, int grid, int wg) {
  return (int)std::min<int64_t>((lds_share(rt, grid, wg) - 1536) / 8, ((int64_t)n + grid - 1) / grid);
}

// Words of dynamic LDS of k_pagerank<LONG>, for a range's rows.
static int held_words(const wgm_runtime* rt, int grid, int wg) { return (lds_share(rt, grid, wg) - 3072) / 4; }

// Workgroups of PageRank where left open: by fitted_grid, or all that fit. By
// measurement of both (whole calls, 50 iterations, few / all, us):
// Meshes: few up to 12 vertices a thread of theirs; 1024 threads, 1801 x 1701, 981 /
// 1073, 2047^2, 1280 / 1254. Four random edges a vertex: few; 1024 threads, n =
// 700001, 1097 / 1182, 4000001, 11310 / 11500.
// With longer rows it is whether an average range's rows fit the LDS: ER n =
// 524288, 1024 threads, of degree 16 (they do), 2099 / 2166, 512 threads, of degree 8
// (only with all), 1898 / 1588; symmetrised RMAT scale 18, 1024 threads, ef 32 (with
// neither), 4063 / 3100. Many rows of more than kPrSeg edges in a workgroup, which
// sums them one after another, make all the better choice, if the longest fits
// then (scale 18 ef 8, 1306 / 1242, scale 19 ef 4, 1597 / 1415) or the largest ranges,
// up to 1.3 times the average there, do not with few (scale 19 ef 8, 2437 / 2302),
// against scale 18 ef 16, 1566 / 1742, and scale 17 ef 32, 1198 / 1398. (How many meet
// is an estimate: scale 17 ef 4, 841 / 745 and few taken.)
// The barrier of more than four workgroups a CU costs too much, short of huge
// graphs with longer rows: 256 threads, 3001 x 2903 mesh, 3793 / 3927, scale 18 ef 8,
// 1580 / 1944, ER n = 2^20 of degree 32, 10190 / 11420, RMAT scale 20 ef 32, 15590 /
// 15180.
static int pagerank_grid(const wgm_runtime* rt, const wgm_launch* lc, const wgm_graph* g, int fit, int wg) {
  const int64_t cus = rt->info.num_cus, cost = rows_and_edges(g);
  const int few = fitted_grid(rt, lc, g->near == 1 ? g->n : cost, kFitPr, fit, wg);
  if (g->near == 1) return fit <= 4 * cus && g->n > 12 * 1024 * cus ? fit : few;
  if (g->maxdeg <= kTopoEdges) return few;
  if (fit > 4 * cus) return cost > 192 * 1024 * cus ? fit : few;
  const int64_t average = (g->m + 2 * (int64_t)g->n) / few;
  if (g->maxdeg > kPrSeg && cost / few >= 9 * kPrSeg)
    return g->maxdeg <= held_words(rt, fit, wg) || average + average / 4 > held_words(rt, few, wg) ? fit : few;
  return average < held_words(rt, few, wg) ? few : fit;
}

int wgm_pagerank(wgm_runtime* rt, wgm_graph* g, float damping, int32_t iterations, const wgm_launch* lc,
                 float* rank_out, wgm_run_stats* st) {
  if (!rt || !g || g->rt != rt) return fail(rt, WGM_ERR_INVALID, "bad runtime/graph");
  if (iterations < 1 || !(damping >= 0.0f && damping <= 1.0f))
    return fail(rt, WGM_ERR_INVALID, "need iterations >= 1 and damping in [0, 1]");
  int rc = dev_alloc(rt, &g->f0, g->n);
  if (!rc) rc = dev_alloc(rt, &g->f1, g->n);
  if (!rc) rc = dev_alloc(rt, &g->f2, g->n);
  if (!rc && g->maxdeg > kTopoEdges) rc = dev_alloc(rt, &g->wl, wl_words(g));
  if (!rc) rc = near_rows(rt, g);
  if (rc) return rc;
  const float nf = (float)g->n;
  const float base = (1.0f - damping) / nf;
  const float r0 = 1.0f / nf;
  int grid = 0, wg = 0;
  rc = launch_prologue(rt, WGM_K_PAGERANK, lc, &grid, &wg);
  if (rc) return rc;
  grid = pagerank_grid(rt, lc, g, grid, wg);
  if (g->near == 1)
    hipLaunchKernelGGL(k_pagerank_near, dim3(grid), dim3(wg), 8 * (size_t)near_held(rt, g->n, grid, wg), rt->stream, rt->ctl,
                       wgm_graph_view(g), g->near_rows, near_held(rt, g->n, grid, wg), g->f0, g->f1, g->f2, damping, base,
                       r0, iterations, g->iters);
  else if (g->maxdeg > kTopoEdges) {
    const int words = held_words(rt, grid, wg);
    hipLaunchKernelGGL(k_pagerank<true>, dim3(grid), dim3(wg), 4 * (size_t)words, rt->stream, rt->ctl, wgm_graph_view(g),
                       g->f0, g->f1, g->f2, damping, base, r0, iterations, g->wl, words, g->iters);
  } else
    hipLaunchKernelGGL(k_pagerank<false>, dim3(grid), dim3(wg), 0, rt->stream, rt->ctl, wgm_graph_view(g), g->f0, g->f1,
                       g->f2, damping, base, r0, iterations, (int32_t*)nullptr, 0, g->iters);
  return launch_epilogue(rt, lc, g, g->f2, rank_out, st);
}

}  // extern "C"
