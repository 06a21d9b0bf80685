// low_degree.hpp -- BFS / SSSP over one low-degree graph on one workgroup (the
// batched launch's small graphs and the standalone apps' narrow ones).
#pragma once

#include <type_traits>

#include "team_frontier.hpp"

namespace wgm {

// Low-degree graphs (out-degree <= kLowDegree: grids, meshes, road-like)
// traverse thousands of narrow levels, each a chain of memory round trips:
// they take the degree-bounded frontier step, and a team's cross-workgroup
// barrier would add to every level, so one workgroup serves them up to
// kLowDegreeSingle edges. Measured on the 512-query batch: with 2-workgroup
// teams for the 1M-edge grids the batch took 17.4 ms instead of 10.2 ms.
constexpr int kLowDegree = 4;
constexpr long long kLowDegreeSingle = 1ll << 22;
// Frontier entries per thread group in flight together. A narrow level's
// cost is instruction issue, and each unrolled slot adds its scalar checks
// to every level: on the 512-query batch, 4 slots took 8.99 ms per step,
// 2 took 8.75 and 1 took 8.64 (levels past bd / K entries take more passes).
constexpr int kLowSlots = 1;

// The low-degree step keeps the first low_lds_cap(bd) entries of each of its
// two frontier queues (vertex, row info, distance tag) in LDS behind the
// frontier step's own LDS; entries past that spill to the HBM queues at the
// same index. A level then reads its entries from LDS and ends without
// waiting on queue stores to reach L2. 2 * bd entries keep a 1024-thread
// workgroup under 64 KB of LDS, and two such workgroups fit one CU.
__host__ __device__ constexpr int low_lds_cap(int bd) { return 2 * bd; }
// A 1024-thread workgroup is alone on its CU (its register and wave counts
// allow one), so it may also hold the far flags of a low-degree SSSP job
// as an LDS bitmap of kFarBitWords words (graphs up to 2^18 vertices):
// setting a far flag is then an LDS atomic instead of a round trip to L2.
constexpr int kFarBitWords = 8192;
__host__ __device__ constexpr int batch_far_bits_bytes(int bd) { return bd >= 1024 ? 4 * kFarBitWords : 0; }

// Packed rows of low-degree graphs: kLowDegree words per vertex, (target << 8)
// | weight, kEllNone past the degree. A graph gets them when every weight fits
// 8 bits and its vertex ids fit 24 (kEllNone is no valid word then).
constexpr uint32_t kEllNone = 0xffffffffu;
constexpr int32_t kEllMaxN = (1 << 24) - 1;
// Distances kept in the L2 (low_ell == 2): a low-degree SSSP query on one
// 1024-thread workgroup updates its distances with plain loads and stores,
// which stay in its XCD's L2, instead of atomics, which are all performed
// beyond it. Each pass first folds its candidates per target in an LDS hash
// table of kCombSlots 64-bit words, (distance << 32) | (target << 11) |
// candidate (slot and thread, so that words are unique and the minimum has
// one owner), open addressing with linear probes. A pass takes kCombU
// entries per 4-lane group, at most kCombU * blockDim.x <= 2048 candidates,
// so a table is at most half full and every probe sequence ends.
// Three tables serve consecutive passes in turn: the winner of a slot clears
// it after the next pass's barrier, when every reader of the slot is past it,
// and the pass after that (the slot's next user) starts after the clear.
// Passes are the cost of a level (each is two memory round trips and two
// barriers): two entries per group halve the passes of the levels wider than
// blockDim.x / 4 entries.
constexpr int kCombBits = 12;
constexpr int kCombSlots = 1 << kCombBits;
constexpr int kCombU = 2;
constexpr unsigned long long kCombEmpty = ~0ull;
// Its own LDS layout: two frontier queues of kCombCap (vertex, tag) entries,
// the far bitmap, the three tables (152 KB at 1024 threads).
constexpr int kCombCap = 1536;
__host__ __device__ constexpr int comb_lds_bytes(int bd) {
  return bd >= 1024 ? 2 * 2 * 4 * kCombCap + 4 * kFarBitWords + 3 * kCombSlots * 8 : 0;
}
__host__ __device__ constexpr int batch_lds_bytes(int bd) {
  return frontier_lds_bytes(bd) + 2 * 3 * 4 * low_lds_cap(bd) + batch_far_bits_bytes(bd) > comb_lds_bytes(bd)
             ? frontier_lds_bytes(bd) + 2 * 3 * 4 * low_lds_cap(bd) + batch_far_bits_bytes(bd)
             : comb_lds_bytes(bd);
}
typedef __attribute__((address_space(3))) unsigned long long lds_u64;

// The per-vertex bitmap: batch_far_bits_bytes(bd) after the low-degree queues.
__device__ __forceinline__ lds_u32* batch_bits(int* lds) {
  return (lds_u32*)(reinterpret_cast<uint32_t*>(lds) +
                    (frontier_lds_bytes((int)blockDim.x) + 2 * 3 * 4 * low_lds_cap((int)blockDim.x)) / 4);
}
// The combine layout's far bitmap and tables.
__device__ __forceinline__ lds_u32* comb_bits(int* lds) { return (lds_u32*)lds + 2 * 2 * kCombCap; }
__device__ __forceinline__ lds_u64* batch_comb(int* lds) { return (lds_u64*)(comb_bits(lds) + kFarBitWords); }

__device__ __forceinline__ unsigned long long comb_word(int u, uint32_t alt, int cand) {
  return ((unsigned long long)alt << 32) | ((unsigned long long)(uint32_t)u << 11) | (uint32_t)cand;
}
// Slot of target u (< 2^21) in a combine table, where its word is folded in
// by a minimum: the first candidate of u claims an empty slot, later ones
// find u there. -1 only if the table were full, which a pass cannot make it.
__device__ __forceinline__ int comb_insert(lds_u64* t, int u, unsigned long long mine) {
  int h = (int)(((uint32_t)u * 2654435761u) >> (32 - kCombBits));
  for (int probe = 0; probe < kCombSlots; probe++) {
    unsigned long long old = kCombEmpty;
    if (__hip_atomic_compare_exchange_strong(&t[h], &old, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP))
      return h;
    if (((uint32_t)old >> 11) == (uint32_t)u) {
      __hip_atomic_fetch_min(&t[h], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      return h;
    }
    h = (h + 1) & (kCombSlots - 1);
  }
  return -1;
}

// Workgroup barrier that orders LDS only: memory loads stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Row start and out-degree of v packed into one queue word (row start
// < 2^29, degree <= 7), loaded by the producer alongside its atomic so the
// consumer skips a dependent round trip.
__device__ __forceinline__ uint32_t row_info(const GraphDev& g, int v) {
  const int rs = g.row_ptr[v];
  return ((uint32_t)rs << 3) | (uint32_t)(g.row_ptr[v + 1] - rs);
}

// Frontier queues of the low-degree step: entry i of queue p (0 or 1) in
// LDS below cap, in the HBM queue at index i above.
// LDS-typed (lds_u32), so that the two paths of load/store stay ds_* and
// global_* instructions: through a generic pointer the compiler merges them
// into one flat access, which then waits on both the LDS and the memory
// counters.

struct LowQueues {
  lds_u32* lds;  // [queue][vertex, row info, tag][cap]; F = 2: [queue][vertex, tag][cap] (no row info)
  int cap;
  const FrontierDev* s;
  int F;
  // rows: the entry carries row_info (CSR rows; packed rows need none)
  __device__ __forceinline__ void load(int p, int i, int& v, uint32_t& ri, uint32_t& du, bool tag,
                                       bool rows = true) const {
    ri = 0u;
    if (i < cap) {
      const lds_u32* b = lds + p * F * cap;
      v = (int)b[i];
      if (rows) ri = b[cap + i];
      du = tag ? b[(F - 1) * cap + i] : 0u;
    } else {
      v = (p ? s->q1 : s->q0)[i];
      if (rows) ri = (p ? s->qr1 : s->qr0)[i];
      du = tag ? (p ? s->qa1 : s->qa0)[i] : 0u;
    }
  }
  __device__ __forceinline__ void store(int p, int i, int v, uint32_t ri, uint32_t du, bool tag,
                                        bool rows = true) const {
    if (i < cap) {
      lds_u32* b = lds + p * F * cap;
      b[i] = (uint32_t)v;
      if (rows) b[cap + i] = ri;
      if (tag) b[(F - 1) * cap + i] = du;
    } else {
      (p ? s->q1 : s->q0)[i] = v;
      if (rows) (p ? s->qr1 : s->qr0)[i] = ri;
      if (tag) (p ? s->qa1 : s->qa0)[i] = du;
    }
  }
};

// A low-degree graph (out-degree <= K) on one workgroup: K threads per
// frontier entry, one edge each, and entries that carry what the consumer
// would otherwise fetch in sequence: the vertex, its row (row_info) and, for
// SSSP, the distance it was queued with. With the queues in LDS a pass over
// entries is two dependent HBM round trips -- edge (+ the vertex's current
// distance); atomic (+ the target's row) -- and each thread keeps U entries'
// round trips in flight together, so a level of up to U * bd / K entries is
// one pass and one barrier. An SSSP entry whose vertex has since dropped
// lower is skipped (its newer entry carries the lower distance). Near-far
// bands as in run_single; a far queue of at most bd entries is split in one
// pass that keeps each entry's distance and row in registers across the
// band minimum.
// ELL: the graph is read from packed rows instead of the CSR -- K words per
// vertex, word k = (target << 8) | weight of its k-th edge, kEllNone past its
// degree -- so the K threads of an entry load one 4K-byte row together, an
// entry needs no row_info, and the second round trip is the atomic alone.
template <bool SSSP, int K, int U, bool ELL>
__device__ void run_low(const GraphDev& g, const FrontierDev& s, const NearFar& nf, int src, int* lds, int* s_cnt,
                        int* iters_out, bool lds_flags, const uint32_t* ell) {
  const bool near_far = SSSP && nf.delta > 0;
  __shared__ int s_far[3];  // far counts of q[0], q[1]; band minimum
  const LowQueues lq{(lds_u32*)(reinterpret_cast<uint32_t*>(lds) + frontier_lds_bytes((int)blockDim.x) / 4),
                     low_lds_cap((int)blockDim.x), &s, 3};
  // one bit per vertex in LDS (lds_flags): SSSP's far flags (else a word per
  // vertex in HBM); BFS's visited marks, which then replace the atomic on
  // dist (else the atomic minimum decides the discovery)
  lds_u32* fbits = batch_bits(lds);
  const bool bits = near_far && lds_flags;
  const bool vis = !SSSP && lds_flags;
  for (int v = threadIdx.x; v < g.n; v += blockDim.x) {
    s.dist[v] = (v == src) ? 0u : kInf;
    if (near_far && !bits) nf.flag[v] = 0u;
  }
  if (bits || vis)
    for (int w = threadIdx.x; w < (g.n + 31) / 32; w += blockDim.x)
      fbits[w] = vis && w == (src >> 5) ? 1u << (src & 31) : 0u;
  if (threadIdx.x == 0) {
    lq.store(0, 0, src, ELL ? 0u : row_info(g, src), 0u, SSSP, !ELL);
    s_cnt[0] = 1;
    s_cnt[1] = 0;
    s_cnt[2] = 0;
    s_far[0] = 0;
    s_far[1] = 0;
    s_far[2] = INT32_MAX;
  }
  __syncthreads();
  const int bd = blockDim.x, per = bd / K;
  const int slot = (int)threadIdx.x / K, k = (int)threadIdx.x % K;
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  int level = 0, fi = 0;
  uint32_t thr = near_far ? nf.delta : 0xffffffffu;
  uint32_t nrel = 0;  // edges this thread relaxed (live entries' edges)
  while (true) {
    for (;; level++) {
      const int in_n = __builtin_amdgcn_readfirstlane(s_cnt[level % 3]);
      if (in_n == 0) break;
      // counter (level + 2) % 3 was last read at the start of level - 1
      if (threadIdx.x == 0) s_cnt[(level + 2) % 3] = 0;
      const int p = level & 1;  // in queue; 1 - p is the out queue
      int* out_cnt = &s_cnt[(level + 1) % 3];
      const uint32_t next = (uint32_t)level + 1u;
      for (int a = 0; a < in_n; a += per * U) {
        // slot x holds entries of this wave only while a + x per + its first
        // slot < in_n: a scalar test, so a wave runs no code for empty slots
        // (most levels fill one slot, and only some waves of it) -- issue
        // time, not memory, bounds a narrow level.
        const int wslot = __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~63) / K;
        if (a + wslot >= in_n) continue;
        bool lv[U];
#pragma unroll
        for (int x = 0; x < U; x++) lv[x] = a + x * per + wslot < in_n;
        int v[U], e[U];
        uint32_t du[U];
        bool ok[U];
#pragma unroll
        for (int x = 0; x < U; x++) {
          const int i = a + x * per + slot;
          uint32_t ri = 0;
          v[x] = 0;
          du[x] = 0;
          if (lv[x] && i < in_n) lq.load(p, i, v[x], ri, du[x], SSSP, !ELL);
          ok[x] = ELL ? (lv[x] && i < in_n) : (int)(ri & 7u) > k;
          e[x] = ELL ? v[x] * K + k : (int)(ri >> 3) + k;
        }
        // round trip 1, every slot in flight: the edge and the entry's distance
        int u[U];
        uint32_t w[U], dv[U];
#pragma unroll
        for (int x = 0; x < U; x++) {
          u[x] = 0;
          w[x] = 0u;
          dv[x] = 0u;
          if (!lv[x]) continue;
          if (ELL) {
            const uint32_t word = ok[x] ? ell[e[x]] : kEllNone;
            dv[x] = SSSP && ok[x] ? s.dist[v[x]] : 0u;
            ok[x] = word != kEllNone;
            u[x] = ok[x] ? (int)(word >> 8) : 0;
            w[x] = word & 255u;
          } else {
            u[x] = ok[x] ? g.col[e[x]] : 0;
            w[x] = SSSP && ok[x] ? (uint32_t)g.wt[e[x]] : 0u;
            dv[x] = SSSP && ok[x] ? s.dist[v[x]] : 0u;
          }
        }
        // round trip 2, every slot in flight: the atomic and the target's row.
        // Only the memory operations sit under each slot's condition; what
        // reads their results comes after every slot has issued.
        uint32_t alt[U], old[U], r0[U], r1[U];
#pragma unroll
        for (int x = 0; x < U; x++) {
          const bool live = ok[x] && (!SSSP || dv[x] == du[x]);
          nrel += live ? 1u : 0u;
          alt[x] = SSSP ? du[x] + w[x] : next;
          // the row loads are unconditional (a dead slot reads row 0, which
          // every graph has): only the atomic needs the slot's condition
          r0[x] = 0u;
          r1[x] = 0u;
          old[x] = 0u;  // not live: never an improvement, never kInf
          if (!lv[x]) continue;
          if (!ELL) {
            int uu = live ? u[x] : 0;
            opaque(uu);  // one unconditional load pair, not one per arm of live
            r0[x] = (uint32_t)g.row_ptr[uu];
            r1[x] = (uint32_t)g.row_ptr[uu + 1];
          }
          if (live) {
            if (vis) {
              // BFS with visited bits: the first to set u's bit discovers it
              const uint32_t bit = 1u << (u[x] & 31);
              old[x] = (__hip_atomic_fetch_or(&fbits[u[x] >> 5], bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) &
                        bit) ? 0u : kInf;
            } else {
              // BFS: every distance set so far is <= level + 1 = alt, so the
              // minimum changes only kInf and old == kInf marks the discovery
              // (a compare-and-swap without its compare inside the block)
              old[x] = __hip_atomic_fetch_min(&s.dist[u[x]], alt[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
          }
        }
#pragma unroll
        for (int x = 0; x < U; x++) {
          opaque(old[x]);
          opaque(r0[x]);
          opaque(r1[x]);
        }
        bool want[U], far_cand[U];
        uint32_t ru[U];
#pragma unroll
        for (int x = 0; x < U; x++) {
          ru[x] = (r0[x] << 3) | (r1[x] - r0[x]);
          const bool better = SSSP ? alt[x] < old[x] : old[x] == kInf;
          want[x] = better && (!SSSP || alt[x] < thr);
          far_cand[x] = SSSP && better && alt[x] >= thr;
          // the discoverer writes the level: nothing reads dist during a BFS
          if (vis && want[x]) s.dist[u[x]] = alt[x];
        }
#pragma unroll
        for (int x = 0; x < U; x++) {
          if (!lv[x]) continue;
          // the far flag's exchange is issued first, so that its round trip
          // overlaps the near queue's counter atomic below
          bool far_want = false;
          if (SSSP) {
            if (bits) {
              const uint32_t bit = 1u << (u[x] & 31);
              far_want = far_cand[x] && (__hip_atomic_fetch_or(&fbits[u[x] >> 5], bit, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_WORKGROUP) & bit) == 0u;
            } else {
              far_want = far_cand[x] && __hip_atomic_exchange(&nf.flag[u[x]], 1u, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_WORKGROUP) == 0u;
            }
          }
          const unsigned long long mask = __ballot(want[x]);
          if (mask) {
            const int leader = __ffsll((long long)mask) - 1;
            int base = 0;
            if (lane == leader)
              base = __hip_atomic_fetch_add(out_cnt, __popcll(mask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            base = __builtin_amdgcn_readlane(base, leader);  // leader is wave-uniform: no LDS round trip
            if (want[x]) lq.store(1 - p, base + __popcll(mask & below), u[x], ru[x], alt[x], SSSP, !ELL);
          }
          if (SSSP) push_item<false>(far_want, u[x], nf.far(fi), &s_far[fi], __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
      __syncthreads();
    }
    if (!near_far) break;
    // uniform: read after the level's barrier (scalar, so the branches
    // around the barriers below stay uniform for the compiler too)
    const int fn = __builtin_amdgcn_readfirstlane(s_far[fi]);
    if (fn == 0) break;
    const int p = level & 1;  // this level's (empty) queue
    // move a far entry below the new threshold to the near queue, else to the other far queue
    const uint32_t t_old = thr;  // far entries below it were relaxed in the band (dropped)
    auto split = [&](bool in, int v, uint32_t dv, uint32_t rv) {
      bool to_near = false, to_far = false;
      if (in) {
        if (dv < thr) {
          // each deferred vertex is in one far queue once: it moves once
          if (bits) __hip_atomic_fetch_and(&fbits[v >> 5], ~(1u << (v & 31)), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
          else nf.flag[v] = 0u;
          to_near = dv >= t_old;
        } else {
          to_far = true;  // stays flagged in the other far queue
        }
      }
      const unsigned long long mask = __ballot(to_near);
      if (mask) {
        const int leader = __ffsll((long long)mask) - 1;
        int nb = 0;
        if (lane == leader)
          nb = __hip_atomic_fetch_add(&s_cnt[level % 3], __popcll(mask), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_WORKGROUP);
        nb = __builtin_amdgcn_readlane(nb, leader);
        if (to_near) lq.store(p, nb + __popcll(mask & below), v, rv, dv, true, !ELL);
      }
      push_item<false>(to_far, v, nf.far(1 - fi), &s_far[1 - fi], __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    if (fn <= bd) {
      const bool in = (int)threadIdx.x < fn;
      int v = 0;
      uint32_t dv = 0, rv = 0;
      if (in) {
        v = nf.far(fi)[threadIdx.x];
        dv = s.dist[v];
        rv = ELL ? 0u : row_info(g, v);
      }
      const int mn = wave_min_int(in && dv >= t_old ? (int)dv : INT32_MAX);
      if (lane == 0) atomicMin(&s_far[2], mn);
      __syncthreads();
      thr = (uint32_t)__builtin_amdgcn_readfirstlane(s_far[2]) + nf.delta;
      split(in, v, dv, rv);
    } else {
      int mn = INT32_MAX;
      for (int i = threadIdx.x; i < fn; i += bd) {
        const uint32_t d = s.dist[nf.far(fi)[i]];
        if (d >= t_old) mn = min(mn, (int)d);
      }
      mn = wave_min_int(mn);
      if (lane == 0) atomicMin(&s_far[2], mn);
      __syncthreads();
      thr = (uint32_t)__builtin_amdgcn_readfirstlane(s_far[2]) + nf.delta;
      for (int base = 0; base < fn; base += bd) {
        const int i = base + threadIdx.x;
        const bool in = i < fn;
        int v = 0;
        uint32_t dv = 0, rv = 0;
        if (in) {
          v = nf.far(fi)[i];
          dv = s.dist[v];
          rv = ELL ? 0u : row_info(g, v);
        }
        split(in, v, dv, rv);
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      s_far[fi] = 0;
      s_far[2] = INT32_MAX;
    }
    fi = 1 - fi;
    __syncthreads();
  }
  for (int d = 32; d > 0; d >>= 1) nrel += __shfl_down(nrel, d, 64);
  if ((threadIdx.x & 63) == 0 && nrel && s.relaxed) atomicAdd(s.relaxed, (unsigned long long)nrel);
  if (threadIdx.x == 0) *iters_out = level;
}

// SSSP on packed rows with everything but the graph and the distances in LDS
// (the combine layout): no atomic on dist at all. A pass loads each candidate
// target's distance with a plain load and folds its candidates per target in
// an LDS combine table (comb_insert); after an LDS barrier the one winner of
// each slot, if below the loaded distance, stores it and queues the target.
// The workgroup is the only writer of the graph's distances, so its L2 holds
// them. Entry, bands and far queues are run_low's, four lanes an entry. A level
// of up to blockDim.x / 4 entries is one pass of a slot per lane group, a wider
// one takes passes of two, with a barrier between the stores of one pass and
// the loads of the next. Only a level of several passes can queue a vertex
// twice, so only the entries after one are compared with their vertices'
// distances.
// Bound: the chain of a level -- its entries from LDS, their rows and their
// targets' distances from the L2, the table, the queue -- 2.2 us at 200 entries.
// As a case of run_low, whose queue reads may also come from memory, every level
// waited for the stores of the one before (361 x 415 grid, kernel: 2720 us; 2270
// here). A queued target's row is not fetched ahead: wherever its register or LDS
// word lay, a wait for it came before the level's end (2440 us).
__device__ void run_low_comb(const GraphDev& g, const FrontierDev& s, const NearFar& nf, int src, int* lds, int* s_cnt,
                             int* iters_out, const uint32_t* ell) {
  constexpr int K = kLowDegree;
  __shared__ int s_far[3];  // far counts of q[0], q[1]; band minimum
  // uniform values in scalar registers: the loops and the barriers in them stay
  // uniform for the compiler
  const int bd = __builtin_amdgcn_readfirstlane((int)blockDim.x), per = bd / K;
  const LowQueues lq{(lds_u32*)lds, kCombCap, &s, 2};
  lds_u32* fbits = comb_bits(lds);
  lds_u64* comb = batch_comb(lds);
  for (int v = threadIdx.x; v < g.n; v += bd) s.dist[v] = (v == src) ? 0u : kInf;
  for (int w = threadIdx.x; w < (g.n + 31) / 32; w += bd) fbits[w] = 0u;
  for (int i = threadIdx.x; i < 3 * kCombSlots; i += bd) comb[i] = kCombEmpty;
  if (threadIdx.x == 0) {
    lq.store(0, 0, src, 0u, 0u, true, false);
    s_cnt[0] = 1;
    s_cnt[1] = 0;
    s_cnt[2] = 0;
    s_far[0] = 0;
    s_far[1] = 0;
    s_far[2] = INT32_MAX;
  }
  __syncthreads();
  const int lane = (int)threadIdx.x & 63, slot = (int)threadIdx.x / K, k = (int)threadIdx.x % K;
  const int wslot = __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~63) / K;  // the wave's first slot
  const unsigned long long below = (1ull << lane) - 1ull;
  int level = 0, fi = 0, tcur = 0;
  uint32_t thr = nf.delta, nrel = 0;
  bool twice = false;         // the level's queue may hold a vertex twice
  int clr[kCombU];            // slots this thread won in the previous pass, cleared after this pass's barrier
#pragma unroll
  for (int x = 0; x < kCombU; x++) clr[x] = -1;

  auto pass = [&](auto slots, int a, int in_n, int p, int* out_cnt) {
    constexpr int N = decltype(slots)::value;
    tcur = __builtin_amdgcn_readfirstlane(tcur);
    lds_u64* tb = comb + tcur * kCombSlots;
    lds_u64* tp = comb + (tcur == 0 ? 2 : tcur - 1) * kCombSlots;
    uint32_t du[N], word[N], dv[N], alt[N], old[N];
    int v[N], u[N], hs[N];
    bool on[N], ok[N];
#pragma unroll
    for (int x = 0; x < N; x++) {
      on[x] = a + x * per + wslot < in_n;  // scalar: this wave has entries in the slot
      ok[x] = false;
      hs[x] = -1;
    }
    if (on[0]) {
#pragma unroll
      for (int x = 0; x < N; x++) {
        const int i = a + x * per + slot;
        ok[x] = i < in_n;
        uint32_t none;
        v[x] = 0;
        du[x] = 0;
        if (in_n <= kCombCap) {  // scalar: the queue is in LDS as a whole
          const lds_u32* q = lq.lds + p * 2 * kCombCap + min(i, in_n - 1);
          v[x] = (int)q[0];
          du[x] = q[kCombCap];
        } else if (ok[x]) {
          lq.load(p, i, v[x], none, du[x], true, false);
        }
      }
      // round trip 1: the edges (and the entries' distances)
#pragma unroll
      for (int x = 0; x < N; x++) word[x] = ell[(uint32_t)v[x] * K + k];
#pragma unroll
      for (int x = 0; x < N; x++) dv[x] = twice ? s.dist[v[x]] : du[x];
      // round trip 2: the targets' distances, in flight across the barrier
#pragma unroll
      for (int x = 0; x < N; x++) {
        ok[x] = ok[x] && word[x] != kEllNone && dv[x] == du[x];
        u[x] = ok[x] ? (int)(word[x] >> 8) : 0;
        alt[x] = du[x] + (word[x] & 255u);
        nrel += ok[x] ? 1u : 0u;
      }
#pragma unroll
      for (int x = 0; x < N; x++) old[x] = s.dist[u[x]];
#pragma unroll
      for (int x = 0; x < N; x++)
        if (ok[x]) hs[x] = comb_insert(tb, u[x], comb_word(u[x], alt[x], x * bd + (int)threadIdx.x));
    }
    lds_barrier();
    // every candidate is in the table; the slot's word is the minimum over its
    // target's candidates, and the candidate whose word it is wins it (the
    // thread bits break ties)
#pragma unroll
    for (int x = 0; x < kCombU; x++) {
      if (clr[x] >= 0) tp[clr[x]] = kCombEmpty;
      clr[x] = -1;
    }
    tcur = tcur == 2 ? 0 : tcur + 1;
    if (!on[0]) return;
    bool won[N];
#pragma unroll
    for (int x = 0; x < N; x++) {
      won[x] = false;
      if (hs[x] >= 0) {
        won[x] = tb[hs[x]] == comb_word(u[x], alt[x], x * bd + (int)threadIdx.x);
        if (won[x]) clr[x] = hs[x];
      }
    }
#pragma unroll
    for (int x = 0; x < N; x++) {
      const bool better = won[x] && alt[x] < old[x];
      if (!__ballot(better)) continue;
      const bool near = better && alt[x] < thr, far = better && alt[x] >= thr;
      if (better) s.dist[u[x]] = alt[x];
      const unsigned long long mask = __ballot(near);
      if (mask) {
        const int leader = __ffsll((long long)mask) - 1, count = __popcll(mask);
        int base = 0;
        // (opaque: one lane's addition, which needs no combining over the wave)
        int at = 0;
        opaque(at);
        if (lane == leader)
          base = __hip_atomic_fetch_add(out_cnt + at, count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        base = __builtin_amdgcn_readlane(base, leader);
        const int i = base + __popcll(mask & below);
        if (base + count <= kCombCap) {  // scalar
          lds_u32* q = lq.lds + (1 - p) * 2 * kCombCap + i;
          if (near) {
            q[0] = (uint32_t)u[x];
            q[kCombCap] = alt[x];
          }
        } else if (near) {
          lq.store(1 - p, i, u[x], 0u, alt[x], true, false);
        }
      }
      if (__ballot(far)) {
        const uint32_t bit = 1u << (u[x] & 31);
        const bool fresh = far && (__hip_atomic_fetch_or(&fbits[u[x] >> 5], bit, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_WORKGROUP) & bit) == 0u;
        push_item<false>(fresh, u[x], nf.far(fi), &s_far[fi], __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  };

  while (true) {
    for (;; level++) {
      const int in_n = __builtin_amdgcn_readfirstlane(s_cnt[level % 3]);
      if (in_n == 0) break;
      // counter (level + 2) % 3 was last read at the start of level - 1
      if (threadIdx.x == 0) s_cnt[(level + 2) % 3] = 0;
      int* out_cnt = &s_cnt[(level + 1) % 3];
      const int p = level & 1;  // in queue; 1 - p is the out queue
      if (in_n <= per) {
        pass(std::integral_constant<int, 1>{}, 0, in_n, p, out_cnt);
        twice = false;
      } else {
        for (int a = 0; a < in_n; a += kCombU * per) {
          if (a > 0) __syncthreads();  // the last pass's stores before this pass's loads
          pass(std::integral_constant<int, kCombU>{}, a, in_n, p, out_cnt);
        }
        twice = in_n > kCombU * per;
      }
      __syncthreads();
    }
    // uniform: read after the level's barrier (scalar, so the branches
    // around the barriers below stay uniform for the compiler too)
    const int fn = __builtin_amdgcn_readfirstlane(s_far[fi]);
    if (fn == 0) break;
    const int p = level & 1;  // this level's (empty) queue
    // move a far entry below the new threshold to the near queue, else to the other far queue
    const uint32_t t_old = thr;  // far entries below it were relaxed in the band (dropped)
    twice = false;
    auto split = [&](bool in, int v, uint32_t dv) {
      bool to_near = false, to_far = false;
      if (in) {
        if (dv < thr) {
          // each deferred vertex is in one far queue once: it moves once
          __hip_atomic_fetch_and(&fbits[v >> 5], ~(1u << (v & 31)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          to_near = dv >= t_old;
        } else {
          to_far = true;  // stays flagged in the other far queue
        }
      }
      const unsigned long long mask = __ballot(to_near);
      if (mask) {
        const int leader = __ffsll((long long)mask) - 1;
        int nb = 0;
        if (lane == leader)
          nb = __hip_atomic_fetch_add(&s_cnt[level % 3], __popcll(mask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        nb = __builtin_amdgcn_readlane(nb, leader);
        if (to_near) lq.store(p, nb + __popcll(mask & below), v, 0u, dv, true, false);
      }
      push_item<false>(to_far, v, nf.far(1 - fi), &s_far[1 - fi], __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    if (fn <= bd) {
      const bool in = (int)threadIdx.x < fn;
      int v = 0;
      uint32_t dv = 0;
      if (in) {
        v = nf.far(fi)[threadIdx.x];
        dv = s.dist[v];
      }
      const int mn = wave_min_int(in && dv >= t_old ? (int)dv : INT32_MAX);
      if (lane == 0) atomicMin(&s_far[2], mn);
      __syncthreads();
      thr = (uint32_t)__builtin_amdgcn_readfirstlane(s_far[2]) + nf.delta;
      split(in, v, dv);
    } else {
      int mn = INT32_MAX;
      for (int i = threadIdx.x; i < fn; i += bd) {
        const uint32_t d = s.dist[nf.far(fi)[i]];
        if (d >= t_old) mn = min(mn, (int)d);
      }
      mn = wave_min_int(mn);
      if (lane == 0) atomicMin(&s_far[2], mn);
      __syncthreads();
      thr = (uint32_t)__builtin_amdgcn_readfirstlane(s_far[2]) + nf.delta;
      for (int base = 0; base < fn; base += bd) {
        const int i = base + (int)threadIdx.x;
        const bool in = i < fn;
        int v = 0;
        uint32_t dv = 0;
        if (in) {
          v = nf.far(fi)[i];
          dv = s.dist[v];
        }
        split(in, v, dv);
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      s_far[fi] = 0;
      s_far[2] = INT32_MAX;
    }
    fi = 1 - fi;
    __syncthreads();
  }
  for (int d = 32; d > 0; d >>= 1) nrel += __shfl_down(nrel, d, 64);
  if ((threadIdx.x & 63) == 0 && nrel && s.relaxed) atomicAdd(s.relaxed, (unsigned long long)nrel);
  if (threadIdx.x == 0) *iters_out = level;
}

// Standalone low-degree kernels: LDS of the form with bits (BFS) or of the
// combine form (SSSP) at any workgroup size.
__host__ __device__ constexpr int low_bfs_lds_bytes(int bd) {
  return frontier_lds_bytes(bd) + 2 * 3 * 4 * low_lds_cap(bd) + 4 * kFarBitWords;
}
constexpr int kLowSsspLds = 2 * 2 * 4 * kCombCap + 4 * kFarBitWords + 3 * kCombSlots * 8;

}  // namespace wgm
