// team_frontier.hpp -- BFS / SSSP over one graph by a team of workgroups
// that share state through agent-scope atomics (the batched launch's teams
// and the standalone frontier apps).
#pragma once

#include "graph_apps.hpp"

namespace wgm {

// Wave-aggregated push of `item` (and its distance tag into qa, when given)
// where `want`, one counter atomic per wave.
template <bool COH>
__device__ __forceinline__ void push_item(bool want, int item, int32_t* q, int* cnt, int scope,
                                          uint32_t* qa = nullptr, uint32_t tag = 0) {
  const unsigned long long mask = __ballot(want);
  if (!mask) return;
  const int lane = threadIdx.x & 63;
  const int leader = __ffsll((long long)mask) - 1;
  int base = 0;
  if (lane == leader) {
    base = scope == __HIP_MEMORY_SCOPE_WORKGROUP
               ? __hip_atomic_fetch_add(cnt, __popcll(mask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)
               : __hip_atomic_fetch_add(cnt, __popcll(mask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  base = __builtin_amdgcn_readlane(base, leader);  // leader is wave-uniform: no LDS round trip
  if (want) {
    const int pos = base + __popcll(mask & ((1ull << lane) - 1ull));
    if (COH) {
      __hip_atomic_store(&q[pos], item, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (qa) __hip_atomic_store(&qa[pos], tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      q[pos] = item;
      if (qa) qa[pos] = tag;
    }
  }
}

__device__ __forceinline__ int wave_min_int(int x) {
  for (int off = 32; off > 0; off >>= 1) x = min(x, __shfl_xor(x, off, 64));
  return x;
}

// Counter barrier of a team of k workgroups (k small). Arrival is a fetch_add
// on a monotonic counter; the arrival that completes epoch e publishes
// generation e. Everything the team shares is accessed with agent-scope
// atomics (frontier_batch<..., COH>), so the barrier only has to drain this
// workgroup's outstanding accesses before arriving: no L2 write-back or
// invalidation, which would also evict every other job's cached graph on the
// XCD.
__device__ __forceinline__ void team_barrier(int* cnt, int* gen, int k, int& epoch) {
  drain_vmem();
  __syncthreads();
  epoch++;
  if (threadIdx.x == 0) {
    const int old = add_relaxed(cnt, 1);
    if (old == epoch * k - 1) {
      st_relaxed(gen, epoch);
    } else {
      while (ld_relaxed(gen) < epoch) {
      }
    }
  }
  __syncthreads();
}

// LDS of the standalone frontier kernels: a frontier pass (frontier_batch) or, of
// BFS, a bottom-up pass (the scan queues and its found vertices), then
// kStandaloneWords words that outlast a pass.
constexpr int kStandaloneWords = 4;
__host__ __device__ constexpr int bottom_up_lds_bytes(int bd) { return scan_lds_bytes(bd) + kScanU * bd * 4; }
__host__ __device__ constexpr int standalone_pass_lds_bytes(bool sssp, int bd) {
  return sssp || frontier_lds_bytes(bd) > bottom_up_lds_bytes(bd) ? frontier_lds_bytes(bd) : bottom_up_lds_bytes(bd);
}
__host__ __device__ constexpr int standalone_frontier_lds_bytes(bool sssp, int bd) {
  return standalone_pass_lds_bytes(sssp, bd) + 4 * kStandaloneWords;
}

// Frontier membership (bottom-up): a vertex of distance `level`.
struct FrontProbe {
  static constexpr bool kPrio = false;
  const uint32_t* dist;
  uint32_t level;
  __device__ __forceinline__ bool test(int u, uint32_t, bool valid, int&) const {
    return valid & (ld_agent(&dist[u]) == level);
  }
};

// A BFS level taken bottom-up (direction-optimizing BFS, Beamer et al.,
// SC 2012): every unvisited vertex of the member's range looks for an
// in-neighbour in the frontier (dist == level) and if it finds one takes
// level + 1 and queues itself. The first four in-edges are the thread's; the
// rows still open then go on in LDS queues, eight lanes a row, then a wave
// (scan_queued): a few vertices whose long rows meet no frontier would
// otherwise hold back their waves, edge after edge. The vertices found are
// gathered in LDS and queued with one counter atomic per chunk. A vertex is
// written only by its own workgroup, so no atomic on dist is needed; the
// distances are read and written with agent-scope accesses (coherent across
// the XCDs' L2s, as the top-down step's). The set of vertices it discovers is
// the top-down level's: the unvisited vertices with an in-edge from the
// frontier. The level's counters are rotated as frontier_level rotates them.
// s_n: four LDS words, the first three zero at the call and at the return.
// A level runs bottom-up while the frontier holds more than n / kBottomUpDiv
// vertices, or more than the vertices not yet reached (the tail of a BFS,
// where a few unvisited vertices scan their in-edges instead of the frontier
// its out-edges), or where a smaller one has so many out-edges that scanning
// is cheaper (bottom_up_pays).
constexpr int kBottomUpDiv = 16;

__device__ __forceinline__ void frontier_bottom_up(const GraphDev& g, const FrontierDev& s, int level, int rank,
                                                   int nteam, int* lds, int* s_n) {
  const int bd = blockDim.x, tid = threadIdx.x;
  int32_t* out_q = (level & 1) ? s.q0 : s.q1;
  int* out_cnt = &s.counts[((level + 1) % 3) * kLine];
  const uint32_t next = (uint32_t)level + 1u;
  const FrontProbe probe{s.dist, (uint32_t)level};
  GraphDev in = g;  // rows of in-edges
  in.row_ptr = g.rrow;
  in.col = g.rcol;
  int* s_found = lds + scan_lds_bytes(bd) / 4;
  int lo, hi;
  block_range(g.n, rank, nteam, &lo, &hi);
  for (Span chunk{(uint32_t)lo, (uint32_t)hi}; chunk.has(); chunk.next(kScanU * bd)) {
    if (chunk.at > (uint32_t)lo) __syncthreads();  // the last chunk's found vertices are stored
    int v[kScanU], e[kScanU], end[kScanU], u[kScanU][4], none = 0;
    bool open[kScanU], hit[kScanU][4];
#pragma unroll
    for (int k = 0; k < kScanU; k++) {
      v[k] = (int)min(chunk.at + k * bd + tid, chunk.stop - 1u);
      open[k] = chunk.has(k * bd + tid) && ld_agent(&s.dist[v[k]]) == kInf;
    }
#pragma unroll
    for (int k = 0; k < kScanU; k++) {
      e[k] = open[k] ? in.row_ptr[v[k]] : 0;
      end[k] = open[k] ? in.row_ptr[v[k] + 1] : 0;
    }
#pragma unroll
    for (int k = 0; k < kScanU; k++)
#pragma unroll
      for (int j = 0; j < 4; j++) u[k][j] = j < end[k] - e[k] ? in.col[e[k] + j] : -1;
#pragma unroll
    for (int k = 0; k < kScanU; k++)
#pragma unroll
      for (int j = 0; j < 4; j++) hit[k][j] = u[k][j] >= 0 && probe.test(max(u[k][j], 0), 0u, true, none);
#pragma unroll
    for (int k = 0; k < kScanU; k++) {
      const bool found = hit[k][0] || hit[k][1] || hit[k][2] || hit[k][3];
      const bool more = !found && end[k] - e[k] > 4;
      const int fs = wl_slot(found, &s_n[2]);
      if (found) s_found[fs] = v[k];
      const int qs = wl_slot(more, &s_n[0]);
      if (more) {
        lds[qs] = v[k];
        lds[kScanU * bd + qs] = e[k] + 4;
        lds[2 * kScanU * bd + qs] = 0;
      }
    }
    scan_queued(
        in, lds, s_n, probe, [&](int id) { return id; },
        [&](int, int w, int edge, int, int) {
          if (edge >= 0) s_found[wl_slot1(&s_n[2])] = w;
        });
    // scan_queued passed a barrier after the last use of what is read here, and
    // every thread reads the count before the barrier below
    const int nf = __builtin_amdgcn_readfirstlane(s_n[2]);
    if (tid == 0) s_n[0] = s_n[1] = 0;
    if (nf > 0) {
      if (tid == 0) s_n[3] = add_relaxed(out_cnt, nf);
      __syncthreads();
      if (tid == 0) s_n[2] = 0;
      const int at = __builtin_amdgcn_readfirstlane(s_n[3]);
      for (int i = tid; i < nf; i += bd) {
        const int w = s_found[i];
        st_agent(&s.dist[w], next);
        st_agent(&out_q[at + i], w);
      }
    }
  }
  if (rank == 0 && tid == 0) {
    st_relaxed(&s.counts[((level + 2) % 3) * kLine], 0);
    if (s.chunk > 0 && s.claims) st_relaxed(&s.claims[((level + 2) % 3) * kLine], 0);
    if (s.heavy > 0) st_relaxed(&s.hcnt[((level + 1) % 3) * kLine], 0);
  }
}

// Out-edges of the frontier q[0, in_n), estimated from kSamples of its entries,
// evenly spaced, by the first wave: every member reads the same entries and
// gets the same sum, so none has to be told. word: an LDS word.
constexpr int kSamples = 256;
__device__ __forceinline__ float front_edges(const GraphDev& g, const int32_t* q, int in_n, int* word) {
  const int samples = min(kSamples, in_n);
  if (threadIdx.x < 64) {
    int v[kSamples / 64], deg = 0;
#pragma unroll
    for (int k = 0; k < kSamples / 64; k++) {
      const int i = (int)threadIdx.x + 64 * k;
      v[k] = i < samples ? ld_agent(&q[(int)((long long)i * in_n / samples)]) : -1;
    }
#pragma unroll
    for (int k = 0; k < kSamples / 64; k++) deg += v[k] >= 0 ? g.row_ptr[v[k] + 1] - g.row_ptr[v[k]] : 0;
    for (int o = 32; o > 0; o >>= 1) deg += __shfl_xor(deg, o, 64);
    if (threadIdx.x == 0) *word = deg;
  }
  __syncthreads();
  const float sum = (float)__builtin_amdgcn_readfirstlane(*word);
  return sum * ((float)in_n / (float)samples);
}

// Whether a level of `edges` frontier edges is cheaper bottom-up: there the
// unreached vertices scan until they meet the frontier, about m / edges edges
// each, if they have so many. A frontier edge is taken at kFrontierEdge
// scanned ones (its claim is performed beyond the L2). Asked on graphs of
// skewed degrees (FrontierDev.fine) for frontiers of more than n / kSampleDiv
// vertices: elsewhere edges go with vertices, and the question's two dependent
// loads (2 us) would only cost (ER 2^16, 64 x 512: 97 -> 100 us). RMAT scale
// 20 (ef 16), 512 x 1024, kernel: the second level, 1.5 to 5% of the vertices
// with 41% of the edges, took 1.3 of the BFS's 1.72 ms top-down; 0.16 ms in
// all with it bottom-up.
constexpr int kSampleDiv = 128;
constexpr float kFrontierEdge = 2.0f;
__device__ __forceinline__ bool bottom_up_pays(const GraphDev& g, float edges, int unreached) {
  const float m = (float)g.m;
  return (float)unreached * fminf(m / (float)g.n, m / fmaxf(edges, 1.0f)) < kFrontierEdge * edges;
}

// A graph served by a team of k workgroups (rank 0..k-1). Everything the
// team shares -- queue entries and their distance tags, a frontier vertex's
// distance, counters -- goes through agent-scope atomics, so `bar` (the
// team's barrier) only has to drain, never to write back or invalidate an
// L2. SSSP runs near-far bands of width nf.delta (0: frontier
// Bellman-Ford), with the far counters and band minimum in device lines.
// U: edges per thread per frontier pass (frontier_batch). HEAVY: teams whose
// FrontierDev sets heavy > 0 (the standalone kernels) run the heavy-entry
// pass; the batched kernel's teams (heavy = 0) are built without it. s_words:
// kStandaloneWords LDS words (with HEAVY).
// Reference: drelax2 (src/lonestar/graph_apps/bfs/device/bfs.cl:214-302,
// src/lonestar/graph_apps/sssp/device/sssp.cl:262-318).
template <bool SSSP, int U = 1, bool HEAVY = false, class Barrier>
__device__ void run_team(const GraphDev& g, const FrontierDev& s, const NearFar& nf, int src, int rank, int k,
                         int* lds, int* iters_out, Barrier&& bar, int* s_words = nullptr) {
  const bool near_far = SSSP && nf.delta > 0;
  int lo, hi;
  block_range(g.n, rank, k, &lo, &hi);
  // initial state through the coherent path (other members' atomics see it)
  for (int v = lo + (int)threadIdx.x; v < hi; v += blockDim.x) {
    __hip_atomic_store(&s.dist[v], (v == src) ? 0u : kInf, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (near_far) __hip_atomic_store(&nf.flag[v], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (rank == 0 && threadIdx.x == 0) {
    __hip_atomic_store(&s.q0[0], src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (SSSP) __hip_atomic_store(&s.qa0[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    st_relaxed(&s.counts[0], 1);
    st_relaxed(&s.counts[kLine], 0);
    st_relaxed(&s.counts[2 * kLine], 0);
    for (int l = 0; l < 3; l++) {
      st_relaxed(&s.claims[l * kLine], 0);
      if (s.heavy > 0) st_relaxed(&s.hcnt[l * kLine], 0);
    }
    if (near_far) {
      st_relaxed(&nf.cnt[0], 0);
      st_relaxed(&nf.cnt[kLine], 0);
      st_relaxed(&nf.cnt[2 * kLine], INT32_MAX);
    }
  }
  if (HEAVY && threadIdx.x < kStandaloneWords) s_words[threadIdx.x] = 0;
  bar();
  const int bd = blockDim.x;
  int level = 0, fi = 0;
  int seen = 0;  // BFS: vertices reached so far, this level's frontier included
  uint32_t thr = near_far ? nf.delta : 0xffffffffu;
  while (true) {
    int in_n;
    while ((in_n = ld_relaxed(&s.counts[(level % 3) * kLine])) != 0) {
      // every member read the same counts after the barriers: the same choice
      seen += in_n;
      bool up = !SSSP && HEAVY && g.rrow && (in_n > g.n / kBottomUpDiv || in_n > g.n - seen);
      if (!SSSP && HEAVY && g.rrow && s.fine && !up && in_n > g.n / kSampleDiv)
        up = bottom_up_pays(g, front_edges(g, (level & 1) ? s.q1 : s.q0, in_n, s_words + 3), g.n - seen);
      if (up)
        frontier_bottom_up(g, s, level, rank, k, lds, s_words);
      else
        frontier_level<SSSP, true, SSSP, U>(g, s, level, rank, k, lds, thr, near_far ? nf.far(fi) : nullptr,
                                            &nf.cnt[fi * kLine], nf.flag);
      bar();
      // heavy entries deferred by the pass (read after the barrier: every
      // member sees the same count and takes the same number of barriers)
      if (HEAVY && s.heavy > 0 && ld_relaxed(&s.hcnt[(level % 3) * kLine]) != 0) {
        frontier_heavy<SSSP, SSSP>(g, s, level, lds, thr, near_far ? nf.far(fi) : nullptr, &nf.cnt[fi * kLine],
                                   nf.flag);
        bar();
      }
      level++;
    }
    if (!near_far) break;
    const int fn = ld_relaxed(&nf.cnt[fi * kLine]);
    if (fn == 0) break;
    int mn = INT32_MAX;
    const uint32_t t_old = thr;  // far entries below it were relaxed in the band (dropped)
    for (int i = rank * bd + (int)threadIdx.x; i < fn; i += k * bd) {
      const int v = __hip_atomic_load(&nf.far(fi)[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t d = __hip_atomic_load(&s.dist[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d >= t_old) mn = min(mn, (int)d);
    }
    mn = wave_min_int(mn);
    if ((threadIdx.x & 63) == 0 && mn != INT32_MAX)
      __hip_atomic_fetch_min(&nf.cnt[2 * kLine], mn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bar();
    thr = (uint32_t)ld_relaxed(&nf.cnt[2 * kLine]) + nf.delta;
    int32_t* lq = (level & 1) ? s.q1 : s.q0;  // this level's (empty) queue
    uint32_t* lqa = (level & 1) ? s.qa1 : s.qa0;
    for (int base = rank * bd; base < fn; base += k * bd) {
      const int i = base + (int)threadIdx.x;
      bool to_near = false, to_far = false;
      int v = 0;
      uint32_t dv = 0;
      if (i < fn) {
        v = __hip_atomic_load(&nf.far(fi)[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        dv = __hip_atomic_load(&s.dist[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (dv < thr) {
          __hip_atomic_store(&nf.flag[v], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          to_near = dv >= t_old;
        } else {
          to_far = true;
        }
      }
      push_item<true>(to_near, v, lq, &s.counts[(level % 3) * kLine], __HIP_MEMORY_SCOPE_AGENT, lqa, dv);
      push_item<true>(to_far, v, nf.far(1 - fi), &nf.cnt[(1 - fi) * kLine], __HIP_MEMORY_SCOPE_AGENT);
    }
    bar();
    // every member has read q[fi] and the minimum; the next split follows at
    // least one more team barrier (the minimum moved to the near queue)
    if (rank == 0 && threadIdx.x == 0) {
      st_relaxed(&nf.cnt[fi * kLine], 0);
      st_relaxed(&nf.cnt[2 * kLine], INT32_MAX);
    }
    fi = 1 - fi;
  }
  if (rank == 0 && threadIdx.x == 0) *iters_out = level;
}

}  // namespace wgm
