// pannotia.hip -- the Pannotia SSSP and BC persistent apps.
//
// Pannotia SSSP (sssp_combined, src/pannotia/graph_apps/sssp/device/sssp.cl:11-92,
// plugin src/pannotia/graph_apps/sssp/sssp.h:40-176): min-plus sweeps over the
// in-edges, y[v] = min(x[v], min_j w_j + x[src_j]), until a sweep changes
// nothing. The reference runs Jacobi sweeps with three barriers each (copy,
// relax, compare). Here one sweep relaxes in place and flags any decrease, with
// one barrier per sweep: values only decrease and every one stays an upper
// bound, so the sweeps reach the same unique fixpoint (the shortest
// distances; BIG_NUM where unreached) in at most as many sweeps. A sweep follows
// only the edges whose source the last one lowered; the in-edges lie in blocks of
// 256, so a hub's row is shared by several waves and meets at one atomic min.
//
// Pannotia BC (bc_combined, src/pannotia/graph_apps/bc/device/bc.cl:186-235,
// plugin src/pannotia/graph_apps/bc/bc.h): Brandes' betweenness. The reference
// runs one source at a time over all workgroups with global barriers per BFS
// level (two per level forward, one per level backward) and float atomics for
// the path counts and dependencies, which makes its sums order-dependent.
// Here each workgroup takes a whole source: BFS levels with a workgroup queue,
// path counts pulled over in-edges in in-edge order, dependencies pulled over
// out-edges in CSR order, all in FP64 with no atomics on the sums. The
// dependencies of a batch of sources land in a row each; after one barrier the
// rows are added to bc in source order. The result does not depend on the grid and
// equals the FP64 oracle bit for bit.

#include "apps_internal.hpp"

#include <algorithm>
#include <utility>

using namespace wgm;

namespace wgm {

constexpr int32_t kBigNum = WGM_BIG_NUM;
// Cap on BC's per-slot state (28 bytes a vertex per slot, its row included): the
// grid shrinks to fit.
constexpr unsigned long long kBcSlotBytes = 8ull << 30;

// Min-plus graph: the vertices with an in-edge ("rows") numbered in order, the
// in-edges in row order in blocks of 256, the last one padded.
constexpr int kMpBlock = kRwtPad;
struct MinplusDev {
  const int32_t* sid;    // row of an edge's source; none: a vertex without in-edges, or padding
  const int32_t* wt;
  const uint8_t* roff;   // row of an edge less the block's first
  const int32_t* bstart; // [nblk + 1] first row of a block; the last one: nrows
  const int32_t* cid;    // [n] row of a vertex, -1: none
  const int32_t* row_ptr;
  const int32_t* col;
  const int32_t* owt;    // weights of the out-edges
  int32_t nblk;
  int32_t nrows;
  int32_t none;          // a row number whose bit of the LDS map no row shares (mp_none)
  int32_t n;
  int32_t src;
  int32_t big;           // distance of an unreached vertex
  int32_t all;           // the first sweep follows every vertex's edges (minplus_first)
  int32_t max_sweeps;    // n + 1 sweeps settle any graph without a negative cycle
  int32_t shift;         // rows per bit of the LDS map: 1 << shift
  int32_t map_words;
  int32_t bit_words;     // words of one bit set
  int32_t* d;            // [nrows + 1] distances of the rows; the last one stays at big (a block's end is read there)
  uint32_t* bits;        // three bit sets: rows lowered in sweep s in set s % 3
  int32_t* dist;         // [n] result
  unsigned long long* first_edges;  // edges that the first sweep follows
};

typedef __attribute__((address_space(3))) int lds_i32;
typedef int i32x4 __attribute__((ext_vector_type(4)));

// Marks the lowered rows row0 + i (bit i of mask) for the next sweep.
__device__ __forceinline__ void mp_mark(uint32_t* next, int row0, unsigned long long mask) {
  if (!mask) return;
  const int lane = (int)threadIdx.x & 63, sh = row0 & 31;
  const unsigned long long lo = mask << sh, hi = sh ? mask >> (64 - sh) : 0ull;
  const uint32_t w = lane == 0 ? (uint32_t)lo : lane == 1 ? (uint32_t)(lo >> 32) : lane == 2 ? (uint32_t)hi : 0u;
  if (w) __hip_atomic_fetch_or(&next[(row0 >> 5) + lane], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The bit set into the LDS map: bit j of the map is the union of the bits
// j << shift .. ((j + 1) << shift) - 1. (Sets and map are whole 16-byte units.)
__device__ __forceinline__ void mp_load_map(const MinplusDev& p, const uint32_t* set, lds_u32* map) {
  if (p.shift == 0) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
#pragma unroll 4
    for (int i = (int)threadIdx.x; i < p.map_words / 4; i += blockDim.x) ((lds_u32x4*)map)[i] = ((const u32x4*)set)[i];
    return;
  }
  for (int i = (int)threadIdx.x; i < p.map_words; i += blockDim.x) {
    uint32_t out = 0;
    for (int b = 0; b < 32; b++) {
      const long long r0 = (32ll * i + b) << p.shift, r1 = r0 + (1ll << p.shift);
      uint32_t any = 0;
      if (p.shift < 5) {
        if ((r0 >> 5) < p.bit_words) any = (set[r0 >> 5] >> (r0 & 31)) & ((1u << (1 << p.shift)) - 1u);
      } else {
        for (long long w = r0 >> 5; w < min(r1 >> 5, (long long)p.bit_words); w++) any |= set[w];
      }
      out |= any ? 1u << b : 0u;
    }
    map[i] = out;
  }
}

// The first sweep: from a cleared state only the source's edges lower
// anything, unless a weight is negative or so large that it wraps (p.all).
__device__ __forceinline__ bool minplus_first(const MinplusDev& p, int id, int nteam) {
  uint32_t* next = p.bits + p.bit_words;
  const uint32_t tid = (uint32_t)id * blockDim.x + threadIdx.x, stride = (uint32_t)nteam * blockDim.x;
  bool any = false;
  auto relax = [&](int e, int du) {
    const int c = p.cid[p.col[e]], cand = (int)((uint32_t)du + (uint32_t)p.owt[e]);
    if (cand < p.big && cand < __hip_atomic_fetch_min(&p.d[c], cand, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
      __hip_atomic_fetch_or(&next[c >> 5], 1u << (c & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      any = true;
    }
  };
  if (p.all) {
    for (Span mine{tid, (uint32_t)p.n}; mine.has(); mine.next(stride))
      for (int u = (int)mine.at, e = p.row_ptr[u]; e < p.row_ptr[u + 1]; e++) relax(e, u == p.src ? 0 : p.big);
  } else {
    Span row{(uint32_t)p.row_ptr[p.src] + tid, (uint32_t)p.row_ptr[p.src + 1]};
    for (; row.has(); row.next(stride)) relax((int)row.at, 0);
  }
  return any;
}

// A step of a sweep: the blocks [b, b1), kMpU at most, by one wave, which
// follows the edges whose source is set in `map`. A block's candidates meet in
// the wave's LDS table, an entry per row of the block; a row that goes on in
// the next block is carried there. All rows but those at the step's ends are
// this wave's alone, so they are lowered by plain stores; a row at an end by an
// atomic minimum, and each wave that lowers it below what it was before the
// sweep marks it. The blocks' loads are in flight together.
constexpr int kMpU = 4;
__device__ __forceinline__ bool minplus_step(const MinplusDev& p, int b, int b1, lds_i32* tab, const lds_u32* map,
                                             uint32_t* next) {
  const int lane = (int)threadIdx.x & 63;
  i32x4 s[kMpU];
  int c0[kMpU + 1];
#pragma unroll
  for (int u = 0; u < kMpU; u++)
    s[u] = b + u < b1 ? ((const i32x4*)p.sid)[(size_t)(b + u) * 64 + lane] : i32x4{p.none, p.none, p.none, p.none};
#pragma unroll
  for (int u = 0; u <= kMpU; u++) c0[u] = p.bstart[min(b + u, b1)];
  const int first = c0[0], last = c0[kMpU];  // rows that other waves may lower too
  unsigned hit[kMpU], some = 0;
#pragma unroll
  for (int u = 0; u < kMpU; u++) {
    const int id[4] = {s[u].x, s[u].y, s[u].z, s[u].w};
    hit[u] = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const unsigned r = (unsigned)id[j] >> p.shift;
      hit[u] |= ((map[r >> 5] >> (r & 31)) & 1u) << j;
    }
    some |= hit[u];
  }
  if (!__ballot(some != 0)) return false;
  i32x4 w[kMpU];
  int du[kMpU][4], dv[kMpU][4];
  uint32_t ro[kMpU];
#pragma unroll
  for (int u = 0; u < kMpU; u++) {
    w[u] = i32x4{0, 0, 0, 0};
    ro[u] = 0;
    if (hit[u]) {
      w[u] = ((const i32x4*)p.wt)[(size_t)(b + u) * 64 + lane];
      ro[u] = ((const uint32_t*)p.roff)[(size_t)(b + u) * 64 + lane];
    }
    const int id[4] = {s[u].x, s[u].y, s[u].z, s[u].w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      du[u][j] = 0;
      if ((hit[u] >> j) & 1u) du[u][j] = __hip_atomic_load(&p.d[id[j]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      dv[u][q] = 0;
      if (c0[u + 1] - c0[u] >= 64 * q)
        dv[u][q] = __hip_atomic_load(&p.d[min((uint32_t)c0[u] + 64 * q + lane, (uint32_t)p.nrows)], __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  bool any = false;
  int carry = INT32_MAX;
#pragma unroll
  for (int u = 0; u < kMpU; u++) {
    if (b + u >= b1) break;
    if (!__ballot(hit[u] != 0) && carry == INT32_MAX) continue;
    // a lane's candidates of one row, which is the ordinary case, go in as one
    const int wj[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
    int best = INT32_MAX;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if ((hit[u] >> j) & 1u) best = min(best, (int)((uint32_t)wj[j] + (uint32_t)du[u][j]));
      const unsigned row = (ro[u] >> (8 * j)) & 255u;
      if (best != INT32_MAX && (j == 3 || row != ((ro[u] >> (8 * j + 8)) & 255u))) {
        __hip_atomic_fetch_min(&tab[row], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        best = INT32_MAX;
      }
    }
    // entry `rows` (if there is one) is the row that the next block begins in
    const int rows = c0[u + 1] - c0[u];
    const bool on = u + 1 < kMpU && b + u + 1 < b1;
    int carried = INT32_MAX;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (rows < 64 * q) break;
      const int i = 64 * q + lane, c = c0[u] + i;
      int val = INT32_MAX;
      if (i <= rows) {
        val = __hip_atomic_load(&tab[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (val != INT32_MAX) __hip_atomic_store(&tab[i], INT32_MAX, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      if (i == 0) val = min(val, carry);
      if (on && rows < 64 * (q + 1)) {
        carried = __builtin_amdgcn_readlane(val, rows & 63);
        if (i == rows) val = INT32_MAX;
      }
      const bool lower = val < dv[u][q];
      if (lower) {
        if (c == first || c == last)
          __hip_atomic_fetch_min(&p.d[c], val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
          __hip_atomic_store(&p.d[c], val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      any |= lower;
      mp_mark(next, c0[u] + 64 * q, __ballot(lower));
    }
    carry = carried;
  }
  return any;
}

// Bound: in the sweeps that follow most edges the L1's limit of lines on their
// way (55 a CU measured, 450 cycles each), which the gathers of sources'
// distances take; elsewhere the barrier and three dependent loads a sweep. A
// sweep over all edges read 8 bytes and gathered a distance an edge, though
// over the 11 sweeps of RMAT scale 20 (ef 16) a source is lowered 3.3 times:
// 1575 -> 590 us (kernel, 512 x 1024 asked); RMAT 17, 64 x 1024: 620 -> 256;
// ER 2^18 of degree 16: 1001 -> 553; ER 4096 of degree 8, 64 x 512: 116 -> 100.
// Not better: steps dealt out over all workgroups (613 us: several XCDs then
// write a line of distances), rows in the order of their out-degree (610).
__global__ void __launch_bounds__(1024) k_minplus(Ctl c, MinplusDev p, int* iters_out) {
  extern __shared__ __attribute__((aligned(16))) int lds_mp[];
  Team t;
  if (!standalone_begin(c, t)) return;
  const int wave = (int)threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
  lds_i32* tab = (lds_i32*)lds_mp + wave * kMpBlock;
  lds_u32* map = (lds_u32*)lds_mp + nw * kMpBlock;
  for (int i = (int)threadIdx.x & 63; i < kMpBlock; i += 64) tab[i] = INT32_MAX;
  // a workgroup's blocks, in steps that its waves take in turn
  int lo, hi;
  block_range(p.nblk, t.id, t.n, &lo, &hi);
  const int per = min(kMpU, max(1, (hi - lo) / nw));
  const int b0 = __builtin_amdgcn_readfirstlane(lo + wave * per);
  int clo, chi;
  block_range(p.bit_words, t.id, t.n, &clo, &chi);
  int* flags = c.lines;
  int sweep = 1;
  for (;; sweep++) {
    bool any;
    uint32_t* next = p.bits + (size_t)(sweep % 3) * p.bit_words;
    if (sweep == 1) {
      any = minplus_first(p, t.id, t.n);
    } else {
      mp_load_map(p, p.bits + (size_t)((sweep - 1) % 3) * p.bit_words, map);
      __syncthreads();
      any = false;
      for (int b = b0; b < hi; b += nw * per) any |= minplus_step(p, b, min(b + per, hi), tab, map, next);
    }
    uint32_t* clear = p.bits + (size_t)((sweep + 1) % 3) * p.bit_words;
    for (int i = clo + (int)threadIdx.x; i < chi; i += blockDim.x) clear[i] = 0u;
    if (__syncthreads_or(any) && threadIdx.x == 0) st_relaxed(&flags[(sweep % 3) * kLine], 1);
    if (t.id == 0 && threadIdx.x == 0) st_relaxed(&flags[((sweep + 1) % 3) * kLine], 0);
    xcd_barrier(c, t);
    if (ld_relaxed(&flags[(sweep % 3) * kLine]) == 0) break;
    if (sweep == p.max_sweeps) {  // still changing: a negative cycle; every workgroup stops here
      sweep = -1;
      break;
    }
  }
  for (Span mine{t.id * blockDim.x + threadIdx.x, (uint32_t)p.n}; mine.has(); mine.next(t.n * blockDim.x)) {
    const int v = (int)mine.at, r = p.cid[v];
    p.dist[v] = r >= 0 ? p.d[r] : v == p.src ? 0 : p.big;
  }
  clock_end(c, t.id);
  if (t.id == 0 && threadIdx.x == 0) *iters_out = sweep;
  standalone_retire(c);
}

// Distances of the rows (unreached ones at `big`: BIG_NUM for Pannotia SSSP,
// MYINFINITY for Lonestar SSSP's pull direction), the bit sets, and how many edges
// the first sweep follows.
__global__ void k_minplus_init(MinplusDev p) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  const int s = p.cid[p.src];
  for (Span rows{(uint32_t)tid, (uint32_t)p.nrows + 1u}; rows.has(); rows.next(stride))
    p.d[rows.at] = (int)rows.at == s ? 0 : p.big;
  for (int i = tid; i < 3 * p.bit_words; i += stride) p.bits[i] = 0u;
  if (tid == 0)
    *p.first_edges = (unsigned long long)(p.all ? p.row_ptr[p.n] : p.row_ptr[p.src + 1] - p.row_ptr[p.src]);
}

// First rows of the blocks; one wave a vertex.
__global__ void k_minplus_starts(const int32_t* rrow, const int32_t* cid, int n, int nblk, int nrows, int32_t* bstart) {
  const int waves = (int)(gridDim.x * blockDim.x) >> 6, lane = (int)threadIdx.x & 63;
  for (Span mine{(blockIdx.x * blockDim.x + threadIdx.x) >> 6, (uint32_t)n}; mine.has(); mine.next(waves)) {
    const int v = (int)mine.at;
    for (long long b = ((long long)rrow[v] + kMpBlock - 1) / kMpBlock + lane; b * kMpBlock < rrow[v + 1]; b += 64)
      bstart[b] = cid[v];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) bstart[nblk] = nrows;
}

// Rows of the edges and of their sources, padding included. *wild: 1 where a
// weight is negative, or wraps when added to an unreached distance.
__global__ void k_minplus_edges(const int32_t* rrow, const int32_t* rcol, const int32_t* rwt, const int32_t* cid,
                                const int32_t* bstart, int n, int nblk, int none, int32_t* sid, uint8_t* roff,
                                int* wild) {
  bool bad = false;
  const int64_t m = rrow[n], stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < (int64_t)nblk * kMpBlock; e += stride) {
    const int c = e < m ? cid[rcol[e]] : -1;
    sid[e] = c < 0 ? none : c;
    roff[e] = e < m ? (uint8_t)(cid[row_of(rrow, n, e)] - bstart[e / kMpBlock]) : 0;
    bad |= e < m && (uint32_t)rwt[e] > (uint32_t)(INT32_MAX - (int32_t)kInf);
  }
  if (bad) st_relaxed(wild, 1);
}

struct BcDev {
  const int32_t* row_ptr;
  const int32_t* col;
  const int32_t* rrow;
  const int32_t* rcol;
  int32_t n;
  int32_t nsrc;
  int32_t slots;     // per-slot arrays allocated (>= participants)
  int32_t* d;        // [slots][n] BFS level, -1 unreached
  double* sig;       // [slots][n] shortest-path counts
  double* del;       // [rows][n] dependencies, a row per source of a batch
  int32_t rows;      // sources per batch
  const int32_t* srcs;  // [nsrc] sources with an out-edge; [nsrc]: their count
  int32_t* q;        // [slots][n] vertices in level order
  int32_t* lvl;      // [slots][n + 2] level starts in q
  double* bc;        // [n]
  unsigned long long* levels;  // total BFS levels over all sources
};

__device__ __forceinline__ int wg_ld(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// State of one source. In global memory: levels in d. In LDS, for graphs that
// fit: level membership as bitmaps, of which three levels' are kept in turn
// (bit set l % 3 is cleared while level l + 1 is the current one of the
// forward pass, or level l - 2 of the backward pass), since a pass only asks
// for the levels next to its own; 18 bytes a vertex, two workgroups per CU up
// to 4300 vertices.
struct BcGlobal {
  static constexpr int kRow = 16;
  int32_t* d;
  double* sig;
  double* del;
  int32_t* q;
  __device__ __forceinline__ void init(int n) const {
    for (int v = (int)threadIdx.x; v < n; v += blockDim.x) {
      d[v] = -1;
      del[v] = 0.0;
    }
  }
  __device__ __forceinline__ void set(int v, int l) const { d[v] = l; }
  __device__ __forceinline__ bool fresh(int w) const { return wg_ld(&d[w]) == -1; }
  __device__ __forceinline__ bool claim(int w, int l) const {
    int expect = -1;
    return __hip_atomic_compare_exchange_strong(&d[w], &expect, l, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ bool at(int v, int l) const { return wg_ld(&d[v]) == l; }
  __device__ __forceinline__ void mark(int, int) const {}
  __device__ __forceinline__ void clear(int) const {}
};

typedef __attribute__((address_space(3))) double lds_f64;
typedef __attribute__((address_space(3))) uint16_t lds_u16;

struct BcLds {
  static constexpr int kRow = 8;
  lds_f64* sig;
  lds_f64* del;
  lds_u16* q;
  lds_u32* seen;
  lds_u32* bits;  // three bit sets
  int words;
  __device__ __forceinline__ void init(int n) const {
    for (int v = (int)threadIdx.x; v < n; v += blockDim.x) del[v] = 0.0;
    for (int i = (int)threadIdx.x; i < words; i += blockDim.x) seen[i] = bits[i] = bits[words + i] = bits[2 * words + i] = 0u;
  }
  __device__ __forceinline__ void set(int v, int l) const {
    seen[v >> 5] = 1u << (v & 31);
    bits[(l % 3) * words + (v >> 5)] = 1u << (v & 31);
  }
  __device__ __forceinline__ bool fresh(int w) const { return !((seen[w >> 5] >> (w & 31)) & 1u); }
  __device__ __forceinline__ bool claim(int w, int l) const {
    const uint32_t bit = 1u << (w & 31);
    if (__hip_atomic_fetch_or(&seen[w >> 5], bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & bit) return false;
    mark(w, l);
    return true;
  }
  __device__ __forceinline__ bool at(int v, int l) const {
    return (bits[(l % 3) * words + (v >> 5)] >> (v & 31)) & 1u;
  }
  __device__ __forceinline__ void mark(int v, int l) const {
    __hip_atomic_fetch_or(&bits[(l % 3) * words + (v >> 5)], 1u << (v & 31), __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ void clear(int l) const {
    for (int i = (int)threadIdx.x; i < words; i += blockDim.x) bits[((l + 3) % 3) * words + i] = 0u;
  }
};

__host__ __device__ constexpr int bc_words(int n) { return (n + 31) / 32; }
__host__ __device__ constexpr long long bc_lds_bytes(long long n) {
  return 16 * n + (2 * n + 3) / 4 * 4 + 4 * 4 * ((n + 31) / 32);
}

// Rows of up to State::kRow edges are walked by one thread, all its edges in
// flight; up to kBcMid by 16 lanes (one DPP row), four rows a wave at a time;
// longer ones by the wave. (kRow: 16 where an edge's lookups go to memory and
// want to be many in flight, 8 where they stay in LDS and the kernel is to fit
// 64 VGPRs.)
constexpr int kBcMid = 64;

// The rows of the wave's lanes in `m`, 16 lanes a row: the groups take the
// rows in turn, 16 edges a step, step(v, this lane's target or -1, first step,
// last step). The next step's targets are loaded before a step is taken.
template <class Step>
__device__ __forceinline__ void bc_mid(unsigned long long m, int v, int beg, int end, const int32_t* col,
                                       const Step& step) {
  if (!m) return;
  const int lane = (int)threadIdx.x & 63, sub = lane & 15;
  const int count = __popcll(m);
  // lane k: the lane of the k-th row
  const int rank = __popcll(m & ((1ull << lane) - 1ull));
  const bool mine = (m >> lane) & 1ull;
  const int from = __builtin_amdgcn_ds_permute(4 * (mine ? rank : count + lane - rank), lane);
  auto open = [&](int k, int& vv, Span& row) {
    const int src = __shfl(from, k & 63, 64);
    vv = __shfl(v, src, 64);
    row.at = (uint32_t)__shfl(beg, src, 64);
    row.stop = (uint32_t)__shfl(end, src, 64);
    if (k >= count) row = Span{0u, 0u};
  };
  int k = lane >> 4;  // this group's row, and its next one
  int vv, ov;
  Span row, ahead;
  open(k, vv, row);
  int w = row.has(sub) ? col[row.at + sub] : -1;
  open(k + 4, ov, ahead);
  bool first = true;
  while (__ballot(row.has())) {  // every lane takes part in the moves between lanes
    const bool last = !row.has(16);
    const int cv = vv, cw = w;
    const bool live = row.has();
    vv = last ? ov : vv;
    row.at = last ? ahead.at : row.at + 16;
    row.stop = last ? ahead.stop : row.stop;
    k = last ? k + 4 : k;
    w = row.has(sub) ? col[row.at + sub] : -1;
    if (__ballot(last)) open(k + 4, ov, ahead);
    if (live) step(cv, cw, first, last);
    first = last;
  }
}

// The rows of the wave's lanes in `m`, one after the other, 64 edges a step:
// step(lane of the row, this lane's target or -1, first step, last step). The
// next step's targets are loaded before a step is taken.
template <class Step>
__device__ __forceinline__ void bc_wide(unsigned long long m, int beg, int end, const int32_t* col, const Step& step) {
  if (!m) return;
  const int lane = (int)threadIdx.x & 63;
  int l = __ffsll((long long)m) - 1;
  Span row{(uint32_t)__builtin_amdgcn_readlane(beg, l), (uint32_t)__builtin_amdgcn_readlane(end, l)};
  int w = row.has(lane) ? col[row.at + lane] : -1;
  bool first = true;
  while (true) {
    const int cl = l, cw = w;
    const bool last = !row.has(64);
    row.next(64);
    if (last) {
      m &= m - 1;
      if (m) {
        l = __ffsll((long long)m) - 1;
        row.at = (uint32_t)__builtin_amdgcn_readlane(beg, l);
        row.stop = (uint32_t)__builtin_amdgcn_readlane(end, l);
      }
    }
    w = m && row.has(lane) ? col[row.at + lane] : -1;
    step(cl, cw, first, last);
    if (!m) break;
    first = last;
  }
}

// acc plus the wave's terms in lane order (lanes outside h have none).
__device__ __forceinline__ double bc_add_wave(double acc, double t, unsigned long long h) {
  const long long bits = __double_as_longlong(t);
  const int tl = (int)bits, th = (int)(bits >> 32);
  auto lane_value = [&](int k) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane(tl, k), hi = (unsigned)__builtin_amdgcn_readlane(th, k);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
  };
  if (__popcll(h) < 24) {
    for (; h; h &= h - 1) acc += lane_value(__ffsll((long long)h) - 1);
  } else {
#pragma unroll
    for (int k = 0; k < 64; k++) acc += lane_value(k);  // a lane without a term adds zero
  }
  return acc;
}

// acc plus the terms of the 16 lanes of this lane's DPP row, in lane order.
template <int K = 0>
__device__ __forceinline__ double bc_add_row(double acc, double t) {
  if constexpr (K < 16) {
    const long long bits = __double_as_longlong(t);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)bits, 0x150 + K, 0xf, 0xf, false);  // row_newbcast:K
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(bits >> 32), 0x150 + K, 0xf, 0xf, false);
    return bc_add_row<K + 1>(
        acc + __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo)), t);
  } else {
    return acc;
  }
}

// For every vertex v of q[a, z): the terms of its row's edges that have one
// (term(v, w, &t), never negative), added in edge order whoever computes them
// (an edge without a term adds zero), then put(v, sum). Consecutive entries go
// to different waves, so that the hubs, which are found early in a level,
// spread over the workgroup.
template <class State, class Term, class Put>
__device__ __forceinline__ void bc_rows(const State& st, const int32_t* row, const int32_t* col, int a, int z,
                                        const Term& term, const Put& put) {
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
  for (int base = a; base < z; base += blockDim.x) {
    const int i = base + lane * nw + wave;
    const bool in = i < z;
    const int v = in ? (int)st.q[i] : 0;
    const int beg = in ? row[v] : 0, end = in ? row[v + 1] : 0;
    const int deg = end - beg;
    int w[State::kRow];
#pragma unroll
    for (int k = 0; k < State::kRow; k++) w[k] = deg <= State::kRow && k < deg ? col[beg + k] : -1;
    if (in && deg <= State::kRow) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < State::kRow; k++) {
        double t;
        if (w[k] >= 0 && term(v, w[k], &t)) acc += t;
      }
      put(v, acc);
    }
    double acc = 0.0;
    bc_wide(__ballot(deg > kBcMid), beg, end, col, [&](int l, int u, bool first, bool last) {
      const int vv = __builtin_amdgcn_readlane(v, l);
      double t = 0.0;
      const bool has = u >= 0 && term(vv, u, &t);
      acc = bc_add_wave(first ? 0.0 : acc, has ? t : 0.0, __ballot(has));
      if (last && lane == 0) put(vv, acc);
    });
    bc_mid(__ballot(deg > State::kRow && deg <= kBcMid), v, beg, end, col, [&](int vv, int u, bool first, bool last) {
      double t = 0.0;
      if (u < 0 || !term(vv, u, &t)) t = 0.0;
      acc = bc_add_row(first ? 0.0 : acc, t);
      if (last && (lane & 15) == 0) put(vv, acc);
    });
  }
}

// One source on one workgroup; returns its number of BFS levels.
template <class State>
__device__ __forceinline__ int bc_source(const BcDev& b, int s, const State& st, int32_t* lvl, int* s_tail) {
  st.init(b.n);
  __syncthreads();
  if (threadIdx.x == 0) {
    st.set(s, 0);
    st.sig[s] = 1.0;
    st.q[0] = s;
    lvl[0] = 0;
    lvl[1] = 1;
    *s_tail = 1;
  }
  __syncthreads();
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
  int L = 0, lo = 0, hi = 1;
  while (lo < hi) {
    // discover level L + 1 (mega_bfs_kernel_func, bc.cl:17-104)
    auto reach = [&](int w) {
      if (st.claim(w, L + 1)) st.q[atomicAdd(s_tail, 1)] = w;
    };
    st.clear(L - 1);
    for (int base = lo; base < hi; base += blockDim.x) {
      const int i = base + lane * nw + wave;
      const bool in = i < hi;
      const int v = in ? (int)st.q[i] : 0;
      const int beg = in ? b.row_ptr[v] : 0, end = in ? b.row_ptr[v + 1] : 0;
      const int deg = end - beg;
      int w[State::kRow];
      bool open[State::kRow];
#pragma unroll
      for (int k = 0; k < State::kRow; k++) w[k] = deg <= State::kRow && k < deg ? b.col[beg + k] : -1;
#pragma unroll
      for (int k = 0; k < State::kRow; k++) open[k] = w[k] >= 0 && st.fresh(w[k]);
#pragma unroll
      for (int k = 0; k < State::kRow; k++)
        if (open[k]) reach(w[k]);
      bc_wide(__ballot(deg > kBcMid), beg, end, b.col, [&](int, int u, bool, bool) {
        if (u >= 0 && st.fresh(u)) reach(u);
      });
      bc_mid(__ballot(deg > State::kRow && deg <= kBcMid), v, beg, end, b.col, [&](int, int u, bool, bool) {
        if (u >= 0 && st.fresh(u)) reach(u);
      });
    }
    __syncthreads();
    // the same for every lane: keep the level loop's control uniform
    const int tail = __builtin_amdgcn_readfirstlane(*s_tail);
    // path counts of level L + 1, pulled over in-edges in order
    bc_rows(
        st, b.rrow, b.rcol, hi, tail,
        [&](int, int u, double* t) {
          if (!st.at(u, L)) return false;
          *t = st.sig[u];
          return true;
        },
        [&](int w, double acc) { st.sig[w] = acc; });
    if (threadIdx.x == 0) lvl[L + 2] = tail;
    __syncthreads();
    lo = hi;
    hi = tail;
    L++;
  }
  // dependencies, deepest level first (mega_backtrack_kernel_func, bc.cl:106-183);
  // the last level's are zero, as initialised
  for (int l = L - 2; l >= 0; l--) {
    const int a = __builtin_amdgcn_readfirstlane(lvl[l]), z = __builtin_amdgcn_readfirstlane(lvl[l + 1]);
    st.clear(l - 1);
    bc_rows(
        st, b.row_ptr, b.col, a, z,
        [&](int v, int w, double* t) {
          if (!st.at(w, l + 1)) return false;
          *t = st.sig[v] / st.sig[w] * (1.0 + st.del[w]);
          return true;
        },
        [&](int v, double acc) {
          if (v != s) st.del[v] = acc;
          st.mark(v, l);
        });
    __syncthreads();
  }
  return L;
}

// The sources that reach something (an out-edge), in order, by one workgroup;
// the others have one level and no dependencies. out[nsrc] = their count.
__global__ void __launch_bounds__(1024) k_bc_sources(const int32_t* row_ptr, int nsrc, int32_t* out) {
  __shared__ int s_wave[17];
  int total = 0;
  for (int base = 0; base < nsrc; base += blockDim.x) {
    const int s = base + (int)threadIdx.x;
    const bool take = s < nsrc && row_ptr[s + 1] > row_ptr[s];
    int cnt;
    const int at = wg_exclusive_scan(take ? 1 : 0, s_wave, &cnt);
    if (take) out[total + at] = s;
    total += cnt;
  }
  if (threadIdx.x == 0) out[nsrc] = total;
}

// The workgroups claim sources one by one and leave each one's dependencies in
// its row; after a barrier the rows are added to bc in source order, 64
// vertices a workgroup: every wave stages kBcAhead rows in LDS, one wave adds
// them. As many sources share a barrier as the rows hold (one row per source
// where memory allows).
// Bound: RMAT 12 (ef 8, 4096 sources): the rows' dependent loads and ordered
// additions in a workgroup. One thread a row, the state in global memory, a
// barrier per source and workgroup, and the rows added with one load in
// flight: 11.3 ms a call (1024 x 256), 1.35 ms here.
constexpr int kBcAhead = 8;
__host__ __device__ constexpr long long bc_stage_bytes(int wg) { return (long long)wg * kBcAhead * 8; }

template <bool LDS>
__global__ void __launch_bounds__(1024, LDS ? 8 : 4) k_bc(Ctl c, BcDev b, int* iters_out) {
  extern __shared__ double lds_bc[];
  __shared__ int s_tail, s_claim;
  Team t;
  if (!standalone_begin(c, t)) return;
  const size_t off = (size_t)t.id * (size_t)b.n;
  int32_t* lvl = b.lvl + (size_t)t.id * ((size_t)b.n + 2);
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
  const int count = __builtin_amdgcn_readfirstlane(b.srcs[b.nsrc]);
  unsigned long long levels = t.id == 0 ? (unsigned long long)(b.nsrc - count) : 0;
  int batches = 0;
  for (int base = 0; base < count; base += b.rows, batches++) {
    const int stop = min(count, base + b.rows);
    int* claim = &c.lines[(batches & 1) * kLine];  // the other one is cleared for the next batch
    while (t.id < b.slots) {
      if (threadIdx.x == 0) s_claim = add_relaxed(claim, 1);
      __syncthreads();
      const int k = base + __builtin_amdgcn_readfirstlane(s_claim);
      if (k >= stop) break;
      const int s = __builtin_amdgcn_readfirstlane(b.srcs[k]);
      double* del = b.del + (size_t)(k - base) * (size_t)b.n;
      if constexpr (LDS) {
        lds_f64* p = (lds_f64*)lds_bc;
        lds_u16* q = (lds_u16*)(p + 2 * b.n);
        lds_u32* w = (lds_u32*)q + (b.n + 1) / 2;
        const int words = bc_words(b.n);
        const BcLds st{p, p + b.n, q, w, w + words, words};
        levels += (unsigned long long)bc_source(b, s, st, lvl, &s_tail);
        for (int v = (int)threadIdx.x; v < b.n; v += blockDim.x) del[v] = st.del[v];
      } else {
        const BcGlobal st{b.d + off, b.sig + off, del, b.q + off};
        levels += (unsigned long long)bc_source(b, s, st, lvl, &s_tail);
      }
      __syncthreads();
    }
    if (t.id == 0 && threadIdx.x == 0) st_relaxed(&c.lines[((batches + 1) & 1) * kLine], 0);
    xcd_barrier(c, t);
    double* stage = lds_bc;  // [nw * kBcAhead][64]
    for (int v0 = t.id * 64; v0 < b.n; v0 += t.n * 64) {
      const int v = v0 + lane;
      double acc = wave == 0 && v < b.n ? b.bc[v] : 0.0;
      for (int j0 = base; j0 < stop; j0 += nw * kBcAhead) {
        const int j = j0 + wave * kBcAhead;
        const double* x = b.del + (size_t)(j - base) * (size_t)b.n + v;
        double y[kBcAhead];
#pragma unroll
        for (int k = 0; k < kBcAhead; k++) y[k] = j + k < stop && v < b.n ? x[(size_t)k * (size_t)b.n] : 0.0;
        __syncthreads();  // the last round's sums are done
#pragma unroll
        for (int k = 0; k < kBcAhead; k++) stage[(wave * kBcAhead + k) * 64 + lane] = y[k];
        __syncthreads();
        if (wave == 0)
          for (int k = 0; k < nw * kBcAhead; k++) acc += stage[k * 64 + lane];  // rows past the end add zero
      }
      if (wave == 0 && v < b.n) b.bc[v] = acc;
      __syncthreads();
    }
    xcd_barrier(c, t);
  }
  if (threadIdx.x == 0 && levels) atomicAdd(b.levels, levels);
  clock_end(c, t.id);
  if (t.id == 0 && threadIdx.x == 0) *iters_out = batches;
  standalone_retire(c);
}

}  // namespace wgm

#define fail wgm_fail
#define HIPCHK WGM_HIPCHK

namespace {

// Rows per bit of the sweeps' LDS map, as a shift: one up to kMpMapBytes, above
// that 2, 4, ...
constexpr long long kMpMapBytes = 128 << 10;
int mp_shift(int32_t rows) {
  int shift = 0;
  while (4ll * ((rows >> shift) / 32 + 4) > kMpMapBytes) shift++;
  return shift;
}
// The row number for sources without in-edges: the first whose bit no row
// shares. A bit's rows are followed when any of them was lowered, and such a
// source's edges, followed from the unreached distance, would go wrong where a
// weight wraps. (Unsigned: up to 2^31.)
uint32_t mp_none(int32_t rows) {
  const uint32_t per = 1u << mp_shift(rows);
  return ((uint32_t)rows + per - 1u) / per * per;
}

// Edges of the min-plus graph, padding included.
int64_t mp_edges(int64_t m) { return (m + kMpBlock - 1) / kMpBlock * kMpBlock; }

// Launch of a standalone persistent kernel whose first argument is the
// control block (*ctl, refreshed after the reset), as the apps launch theirs:
// grid from the occupancy of `kernel` (capped at max_grid), optional host
// handshake, bounded wait.
int launch_standalone_app(wgm_runtime* rt, int kernel, const void* fn, const wgm_launch* lc, Ctl* ctl, void** args,
                          int max_grid, const AppOut& out, wgm_run_stats* st, size_t lds,
                          unsigned long long* extra = nullptr) {
  wgm_launch def{256, 0, 0, 0};
  const wgm_launch& l = lc ? *lc : def;
  const int wg = l.wg_size > 0 ? l.wg_size : 256;
  int grid = 0;
  int rc = wgm_resolve_grid(rt, kernel, wg, l.num_wgs, &grid);
  if (rc) return rc;
  if (max_grid > 0 && grid > max_grid) grid = max_grid;
  rc = wgm_reset_ctl(rt, 0, l.handshake ? 1 : 0);
  if (rc) return rc;
  *ctl = rt->ctl;
  HIPCHK(rt, hipEventRecord(rt->ev0, rt->stream));
  HIPCHK(rt, hipLaunchKernel(fn, dim3(grid), dim3(wg), args, lds, rt->stream));
  return wgm_finish_app(rt, l.handshake, out, st, extra);
}

// The min-plus graph, built once from the in-edge CSR and kept resident.
int minplus_rows(wgm_graph* g) {
  int rc = wgm_graph_in_edges(g);
  if (rc || g->mp_sid) return rc;
  wgm_runtime* rt = g->rt;
  const int32_t n = g->n;
  const size_t edges = (size_t)mp_edges(g->m);
  const int32_t nblk = (int32_t)(edges / kMpBlock);
  auto alloc = [&](auto** p, size_t count) {
    if (*p) return hipSuccess;  // of an earlier try
    return hipMalloc((void**)p, sizeof(**p) * std::max<size_t>(count, 1));
  };
  int32_t* sid = nullptr;
  hipError_t e = alloc(&g->mp_cid, wgm_row_id_words(n));
  if (e != hipSuccess) return wgm_hip_fail(rt, e, "min-plus graph");
  int32_t rows = 0;
  rc = wgm_row_ids(g, g->mp_cid, &rows);
  if (rc) return rc;
  g->mp_rows = rows;
  g->mp_words = (rows / 32 + 4) / 4 * 4;
  e = alloc(&g->mp_start, (size_t)nblk + 1);
  if (e == hipSuccess) e = alloc(&g->mp_roff, edges);
  if (e == hipSuccess) e = alloc(&g->mp_d, (size_t)rows + 1);
  if (e == hipSuccess) e = alloc(&g->mp_bits, 3 * (size_t)g->mp_words);
  if (e == hipSuccess) e = alloc(&sid, edges);
  if (e != hipSuccess) return wgm_hip_fail(rt, e, "min-plus graph");
  int wild = 0;
  e = hipMemcpyAsync(g->iters, &wild, sizeof(int), hipMemcpyHostToDevice, rt->stream);
  hipLaunchKernelGGL(k_minplus_starts, dim3(1024), dim3(256), 0, rt->stream, g->rrow, g->mp_cid, n, nblk, rows, g->mp_start);
  hipLaunchKernelGGL(k_minplus_edges, dim3(4096), dim3(256), 0, rt->stream, g->rrow, g->rcol, g->rwt, g->mp_cid,
                     g->mp_start, n, nblk, (int32_t)mp_none(rows), sid, g->mp_roff, g->iters);
  if (e == hipSuccess) e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(&wild, g->iters, sizeof(int), hipMemcpyDeviceToHost, rt->stream);
  const hipError_t done = hipStreamSynchronize(rt->stream);
  if (e == hipSuccess) e = done;
  if (e != hipSuccess) {
    (void)hipFree(sid);
    return wgm_hip_fail(rt, e, "min-plus graph");
  }
  g->wild_weights = wild != 0;
  g->mp_sid = sid;
  return WGM_OK;
}

int minplus_tables(int wg) { return wg / 64 * kMpBlock * 4; }

// LDS a BC workgroup may use, and what it takes besides its state (statics and
// allocation granularity, rounded up).
constexpr long long kBcLds = 160 << 10;
constexpr long long kBcLdsFixed = 1536;
constexpr int kCuThreads = 2048;  // 32 waves
constexpr size_t kBcRowBytes = 1ull << 30;

// Whether a source's state fits LDS: 18 bytes a vertex, up to about 8900
// vertices. Below that the state is always in LDS, also where only one
// workgroup then fits a CU (RMAT 13, ef 8, 1500 sources, kernel: 1.28 ms; 3.14
// ms in global memory at 1024 x 256, 2.27 at 256 x 1024).
bool bc_in_lds(const wgm_graph* g) { return bc_lds_bytes(g->n) + kBcLdsFixed <= kBcLds; }
long long bc_lds(const wgm_graph* g, int wg) {
  return std::max(bc_stage_bytes(wg), bc_in_lds(g) ? bc_lds_bytes(g->n) : 0ll);
}

// Grid of the BC launch: the occupancy grid, capped so the per-slot state
// stays within kBcSlotBytes. With the state in LDS, which then bounds the
// workgroups on a CU, the threads asked for are taken in as many larger
// workgroups as fit (RMAT 12, 1024 x 256 asked, kernel: 1.73 ms as 512 x 256,
// 1.25 ms as 512 x 512).
int bc_grid(wgm_runtime* rt, const wgm_graph* g, const wgm_launch* lc, int* grid, int* wg) {
  wgm_launch def{256, 0, 0, 0};
  const wgm_launch& l = lc ? *lc : def;
  int rc = wgm_resolve_grid(rt, WGM_K_BC, l.wg_size > 0 ? l.wg_size : 256, l.num_wgs, grid);
  if (rc) return rc;
  const size_t per_slot = (size_t)g->n * 28 + 8;
  const size_t cap = (size_t)kBcSlotBytes / per_slot;
  if (cap < 1) return fail(rt, WGM_ERR_NOMEM, "one BC slot needs %zu bytes", per_slot);
  if ((size_t)*grid > cap) *grid = (int)cap;
  *wg = l.wg_size > 0 ? l.wg_size : 256;
  if (bc_in_lds(g)) {
    const int per_cu = (int)std::min(kBcLds / (bc_lds(g, *wg) + kBcLdsFixed), (long long)kCuThreads / *wg);
    const int fit = std::max(per_cu, 1) * rt->info.num_cus;
    if (*grid > fit) {
      *wg = std::min({1024, *wg * (*grid / fit), kCuThreads / std::max(per_cu, 1) / 64 * 64});
      *grid = fit;
    }
  } else {  // more than can be resident would only cost the discovery window
    int per_cu = 0;
    rc = wgm_occupancy(rt, WGM_K_BC, *wg, &per_cu);
    if (rc) return rc;
    *grid = std::min(*grid, std::max(per_cu, 1) * rt->info.num_cus);
  }
  return WGM_OK;
}

// Min-plus sweeps from src into dist (device, n entries; `big` where
// unreached). The LDS map takes a CU for a workgroup: more workgroups than that
// are taken as one larger one on each CU, which also shortens the barrier.
int run_minplus(wgm_runtime* rt, wgm_graph* g, int32_t src, int32_t big, const wgm_launch* lc, int32_t* dist,
                bool reached, void* dst, wgm_run_stats* st) {
  int rc = minplus_rows(g);
  if (rc) return rc;
  MinplusDev p{};
  p.sid = g->mp_sid;
  p.wt = g->rwt;
  p.roff = g->mp_roff;
  p.bstart = g->mp_start;
  p.cid = g->mp_cid;
  p.row_ptr = g->row_ptr;
  p.col = g->col;
  p.owt = g->wt;
  p.nblk = (int32_t)(mp_edges(g->m) / kMpBlock);
  p.nrows = g->mp_rows;
  p.n = g->n;
  p.src = src;
  p.big = big;
  p.all = g->wild_weights ? 1 : 0;
  p.max_sweeps = std::min(g->n, INT32_MAX - 1) + 1;
  p.none = (int32_t)mp_none(p.nrows);
  p.shift = mp_shift(p.nrows);
  p.map_words = (int32_t)((mp_none(p.nrows) >> p.shift) / 32 + 4) / 4 * 4;
  p.bit_words = g->mp_words;
  p.d = g->mp_d;
  p.bits = g->mp_bits;
  p.dist = dist;
  p.first_edges = wgm_graph_extra(g);
  wgm_launch shape{256, 0, 0, 0};
  if (lc) shape = *lc;
  if (shape.wg_size <= 0) shape.wg_size = 256;
  int grid = 0;
  rc = wgm_resolve_grid(rt, WGM_K_MINPLUS, shape.wg_size, shape.num_wgs, &grid);
  if (rc) return rc;
  if (grid > rt->info.num_cus) {
    shape.wg_size = std::min(1024, shape.wg_size * ((grid + rt->info.num_cus - 1) / rt->info.num_cus));
    grid = rt->info.num_cus;
  }
  // Small graphs: every further workgroup lengthens each sweep's barrier, more
  // waves its reductions. Eight waves with a block each on up to 64 workgroups,
  // more of them only where a wave has four (kernel, 128 blocks asked as 1024
  // threads on a workgroup a CU: 169 -> 102 us; 2048 blocks: 328 -> 231).
  const auto wanted = [&](int wg) {
    const int waves = wg / 64, one = (p.nblk + waves - 1) / waves;
    return std::max({std::min(64, one), (one + 3) / 4, g->n / (8 * wg) + 1});
  };
  const int few = std::min(512, shape.wg_size);
  if (wanted(few) <= grid) shape.wg_size = few;
  grid = std::min(grid, wanted(shape.wg_size));
  shape.num_wgs = grid;
  hipLaunchKernelGGL(k_minplus_init, dim3(256), dim3(256), 0, rt->stream, p);
  Ctl ctl{};
  void* args[] = {&ctl, &p, &g->iters};
  AppOut out;
  out.iters = g->iters;
  out.extra = reached ? nullptr : p.first_edges;
  out.g = wgm_graph_view(g);
  out.reached = reached ? (const uint32_t*)dist : nullptr;
  out.src = dist;
  out.dst = dst;
  out.bytes = sizeof(int32_t) * (size_t)g->n;
  wgm_run_stats local{};
  unsigned long long first = 0;
  rc = launch_standalone_app(rt, WGM_K_MINPLUS, (const void*)&k_minplus, &shape, &ctl, args, 0, out, &local,
                             (size_t)minplus_tables(shape.wg_size) + 4 * (size_t)p.map_words, &first);
  if (rc) return rc;
  if (local.iterations < 0)
    return fail(rt, WGM_ERR_INVALID, "distances still fall after %d sweeps: negative cycle", g->n + 1);
  // every sweep after the first passes every in-edge
  if (!reached) local.edges_scanned = (int64_t)first + (local.iterations - 1) * g->m;
  if (st) *st = local;
  return WGM_OK;
}

}  // namespace

static int bc_stage(int wg) { return (int)bc_stage_bytes(wg); }

bool wgm_pannotia_kernel_info(int kernel, KernelInfo* out) {
  switch (kernel) {
    case WGM_K_MINPLUS: *out = KernelInfo{(const void*)&k_minplus, minplus_tables}; return true;
    case WGM_K_BC: *out = KernelInfo{(const void*)&k_bc<false>, bc_stage}; return true;
    default: return false;
  }
}

int wgm_pannotia_probe(wgm_runtime* rt, int kernel, int grid, int wg_size) {
  switch (kernel) {
    case WGM_K_MINPLUS:
      hipLaunchKernelGGL(k_minplus, dim3(grid), dim3(wg_size), (size_t)minplus_tables(wg_size), rt->stream, rt->ctl,
                         MinplusDev{}, (int*)nullptr);
      return WGM_OK;
    case WGM_K_BC:
      hipLaunchKernelGGL(k_bc<false>, dim3(grid), dim3(wg_size), (size_t)bc_stage_bytes(wg_size), rt->stream, rt->ctl, BcDev{}, (int*)nullptr);
      return WGM_OK;
    default:
      return WGM_ERR_INVALID;
  }
}

void wgm_pannotia_release(wgm_graph* g) {
  void* ptrs[] = {g->rrow, g->rcol, g->rwt, g->mp_sid, g->mp_roff, g->mp_start, g->mp_cid, g->mp_d, g->mp_bits, g->bc_d, g->bc_sig, g->bc_del, g->bc_q, g->bc_lvl, g->bc_sum, g->bc_srcs};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
}

int64_t wgm_pannotia_bytes(const wgm_graph* g) {
  const int64_t n = g->n, m = g->m, edges = mp_edges(m), slots = g->bc_slots;
  const std::pair<const void*, int64_t> arrays[] = {
      {g->rrow, 4 * (n + 1)}, {g->rcol, 4 * m}, {g->rwt, 4 * edges},
      {g->mp_sid, 4 * edges}, {g->mp_roff, edges}, {g->mp_start, 4 * (edges / kMpBlock + 1)},
      {g->mp_cid, 4 * (int64_t)wgm_row_id_words(g->n)}, {g->mp_d, 4 * ((int64_t)g->mp_rows + 1)}, {g->mp_bits, 12 * (int64_t)g->mp_words},
      {g->bc_d, 4 * slots * n}, {g->bc_sig, 8 * slots * n}, {g->bc_del, 8 * g->bc_rows * n}, {g->bc_q, 4 * slots * n},
      {g->bc_lvl, 4 * slots * (n + 2)}, {g->bc_sum, 8 * (n + 1)}, {g->bc_srcs, 4 * (n + 1)}};
  int64_t b = 0;
  for (const auto& [p, bytes] : arrays)
    if (p) b += bytes;
  return b;
}

extern "C" {

int wgm_sssp_minplus(wgm_runtime* rt, wgm_graph* g, int32_t src, const wgm_launch* lc, int32_t* dist_out,
                     wgm_run_stats* st) {
  if (!rt || !g || g->rt != rt) return fail(rt, WGM_ERR_INVALID, "bad runtime/graph");
  if (src < 0 || src >= g->n) return fail(rt, WGM_ERR_INVALID, "source %d out of range", src);
  if (!g->wt) return fail(rt, WGM_ERR_INVALID, "SSSP needs edge weights");
  if (!g->i32a) HIPCHK(rt, hipMalloc((void**)&g->i32a, sizeof(int32_t) * (size_t)g->n));
  return run_minplus(rt, g, src, kBigNum, lc, g->i32a, false, dist_out, st);
}

}  // extern "C"

// Lonestar SSSP in the pull direction: the min-plus sweeps above on the
// graph's own distance array with MYINFINITY for unreached vertices, so the
// result is wgm_sssp's uint32 distances.
int wgm_sssp_pull(wgm_runtime* rt, wgm_graph* g, int32_t src, const wgm_launch* lc, uint32_t* dist_out,
                  wgm_run_stats* st) {
  if (!g->dist) HIPCHK(rt, hipMalloc((void**)&g->dist, sizeof(uint32_t) * (size_t)g->n));
  return run_minplus(rt, g, src, (int32_t)kInf, lc, (int32_t*)g->dist, true, dist_out, st);
}

extern "C" {

int wgm_bc(wgm_runtime* rt, wgm_graph* g, int32_t num_sources, const wgm_launch* lc, double* bc_out,
           wgm_run_stats* st) {
  if (!rt || !g || g->rt != rt) return fail(rt, WGM_ERR_INVALID, "bad runtime/graph");
  if (num_sources > g->n) return fail(rt, WGM_ERR_INVALID, "%d sources for %d vertices", num_sources, g->n);
  const int32_t nsrc = num_sources > 0 ? num_sources : g->n;
  int rc = wgm_graph_in_edges(g);
  if (rc) return rc;
  int grid = 0, wg = 0;
  rc = bc_grid(rt, g, lc, &grid, &wg);
  if (rc) return rc;
  // a row per source where kBcRowBytes hold them, at least one per workgroup
  const int32_t rows = (int32_t)std::min<size_t>((size_t)nsrc, std::max<size_t>((size_t)grid, kBcRowBytes / (8 * (size_t)g->n)));
  if (g->bc_slots < grid || g->bc_rows < rows) {
    void* old[] = {g->bc_d, g->bc_sig, g->bc_del, g->bc_q, g->bc_lvl};
    for (void* p : old)
      if (p) (void)hipFree(p);
    g->bc_d = g->bc_q = g->bc_lvl = nullptr;
    g->bc_sig = g->bc_del = nullptr;
    const int32_t slots = std::max(g->bc_slots, grid), nrows = std::max(g->bc_rows, rows);
    g->bc_slots = g->bc_rows = 0;
    const size_t sn = (size_t)slots * (size_t)g->n;
    hipError_t e = hipMalloc((void**)&g->bc_del, sizeof(double) * (size_t)nrows * (size_t)g->n);
    if (e == hipSuccess) e = hipMalloc((void**)&g->bc_lvl, sizeof(int32_t) * (size_t)slots * ((size_t)g->n + 2));
    if (!bc_in_lds(g)) {
      if (e == hipSuccess) e = hipMalloc((void**)&g->bc_d, sizeof(int32_t) * sn);
      if (e == hipSuccess) e = hipMalloc((void**)&g->bc_sig, sizeof(double) * sn);
      if (e == hipSuccess) e = hipMalloc((void**)&g->bc_q, sizeof(int32_t) * sn);
    }
    if (e != hipSuccess) return wgm_hip_fail(rt, e, "hipMalloc(BC slots)");
    g->bc_slots = slots;
    g->bc_rows = nrows;
  }
  if (!g->bc_srcs) HIPCHK(rt, hipMalloc((void**)&g->bc_srcs, sizeof(int32_t) * ((size_t)g->n + 1)));
  if (!g->bc_sum) HIPCHK(rt, hipMalloc((void**)&g->bc_sum, sizeof(double) * ((size_t)g->n + 1)));
  unsigned long long* levels = (unsigned long long*)(g->bc_sum + g->n);
  HIPCHK(rt, hipMemsetAsync(g->bc_sum, 0, sizeof(double) * ((size_t)g->n + 1), rt->stream));
  BcDev b{g->row_ptr, g->col, g->rrow, g->rcol, g->n, nsrc, g->bc_slots, g->bc_d, g->bc_sig, g->bc_del,
          rows, g->bc_srcs, g->bc_q, g->bc_lvl, g->bc_sum, levels};
  hipLaunchKernelGGL(k_bc_sources, dim3(1), dim3(1024), 0, rt->stream, g->row_ptr, nsrc, g->bc_srcs);
  Ctl ctl{};
  void* args[] = {&ctl, &b, &g->iters};
  wgm_run_stats local{};
  const wgm_launch shape{wg, grid, lc ? lc->handshake : 0, 0};
  AppOut out;
  out.iters = g->iters;
  out.extra = levels;
  out.src = g->bc_sum;
  out.dst = bc_out;
  out.bytes = sizeof(double) * (size_t)g->n;
  unsigned long long lv = 0;
  rc = launch_standalone_app(rt, WGM_K_BC, bc_in_lds(g) ? (const void*)&k_bc<true> : (const void*)&k_bc<false>, &shape, &ctl, args, grid,
                             out, &local, (size_t)bc_lds(g, wg), &lv);
  if (rc) return rc;
  local.iterations = (int32_t)std::min<unsigned long long>(lv, INT32_MAX);  // BFS levels over all sources
  // TEPS convention for BC: each source traverses every edge once forward
  local.edges_scanned = (int64_t)nsrc * g->m;
  if (st) *st = local;
  return WGM_OK;
}

}  // extern "C"
