// apps_internal.hpp -- device-resident graph object shared by the .hip units.
#pragma once

#include "runtime_internal.hpp"

struct wgm_graph {
  wgm_runtime* rt = nullptr;
  int32_t n = 0;
  int64_t m = 0;
  int32_t maxdeg = 0;  // largest out-degree
  int32_t* row_ptr = nullptr;
  int32_t* col = nullptr;
  int32_t* wt = nullptr;
  uint32_t* prio = nullptr;
  // per-run state, allocated on first use and kept resident
  uint32_t* dist = nullptr;
  uint32_t* stamp = nullptr;
  int32_t* q0 = nullptr;
  int32_t* q1 = nullptr;
  int* counts = nullptr;
  int32_t* i32a = nullptr;
  int32_t* i32b = nullptr;
  float* f0 = nullptr;
  float* f1 = nullptr;
  float* f2 = nullptr;
  int* iters = nullptr;   // the run's levels / rounds / sweeps; a 64-bit count at wgm_graph_extra
  int32_t* wl = nullptr;  // colour / MIS worklists, PageRank's long rows (wl_words in apps.hip)
  // low-degree graphs (k_low), looked at on first use: BFS may run on one
  // workgroup; the weights also fit the packed rows; the rows
  bool low_known = false;
  bool low = false;
  bool low_weights = false;
  uint32_t* ell = nullptr;
  // PageRank's 16-bit rows (k_near_rows): 0 not looked at yet, 1 there, -1 none
  int near = 0;
  uint2* near_rows = nullptr;
  // standalone BFS / SSSP (one team of every participant): two queues of
  // tcap entries with distance tags (SSSP), claim counters, near-far queues
  // and flags
  int32_t* tq = nullptr;
  uint32_t* tqa = nullptr;
  int64_t tcap = 0;
  int* claims = nullptr;
  int32_t* far = nullptr;
  uint32_t* in_far = nullptr;
  int* fcnt = nullptr;
  int32_t* hv = nullptr;  // heavy lists: m / kHeavyMin + 2 entries
  uint32_t* hdu = nullptr;
  int32_t* hclaim = nullptr;
  int* hcnt = nullptr;    // 3 lines
  // in-edge CSR, built on first use
  int32_t* rrow = nullptr;
  int32_t* rcol = nullptr;
  int32_t* rwt = nullptr;
  // min-plus graph (MinplusDev in pannotia.hip) and its state, on first use
  int32_t* mp_sid = nullptr;
  uint8_t* mp_roff = nullptr;
  int32_t* mp_start = nullptr;
  int32_t* mp_cid = nullptr;
  int32_t* mp_d = nullptr;
  uint32_t* mp_bits = nullptr;
  int32_t mp_rows = 0;
  int32_t mp_words = 0;
  bool wild_weights = false;  // a weight is negative, or wraps when added to an unreached distance
  // BC per-slot state and the result
  int32_t bc_slots = 0;
  int32_t bc_rows = 0;  // dependency rows in bc_del
  int32_t* bc_srcs = nullptr;
  int32_t* bc_d = nullptr;
  double* bc_sig = nullptr;
  double* bc_del = nullptr;
  int32_t* bc_q = nullptr;
  int32_t* bc_lvl = nullptr;
  double* bc_sum = nullptr;
};

wgm::GraphDev wgm_graph_view(const wgm_graph* g);
inline unsigned long long* wgm_graph_extra(const wgm_graph* g) { return (unsigned long long*)(g->iters + 2); }
// defined by the Pannotia unit (pannotia.hip)
bool wgm_pannotia_kernel_info(int kernel, KernelInfo* out);
int wgm_pannotia_probe(wgm_runtime* rt, int kernel, int grid, int wg_size);
void wgm_pannotia_release(wgm_graph* g);
int64_t wgm_pannotia_bytes(const wgm_graph* g);
int wgm_graph_frontier_state(wgm_graph* g, bool sssp, wgm::FrontierDev* s);
// per-run arrays of a topology-driven app: 1 colour (i32a), 2 MIS (i32a,
// i32b), 3 PageRank (f0, f1, f2); 0 nothing
int wgm_graph_app_state(wgm_graph* g, int app);
int wgm_launch_frontier(wgm_runtime* rt, const wgm::GraphDev& g, wgm::FrontierDev s, const wgm::NearFar& nf, bool sssp,
                        int src, int grid, int wg, int handshake, const AppOut& out, wgm_run_stats* st);
int wgm_enqueue_frontier(wgm_runtime* rt, const wgm::GraphDev& g, wgm::FrontierDev s, const wgm::NearFar& nf, bool sssp,
                         int src, int grid, int wg, int* iters_dev);
uint32_t wgm_standalone_delta(int maxdeg);
int wgm_sssp_pull(wgm_runtime* rt, wgm_graph* g, int32_t src, const wgm_launch* lc, uint32_t* dist_out,
                  wgm_run_stats* st);
// the graph's in-edge CSR (g->rrow, g->rcol, g->rwt), built once and kept
// resident (reverse.hip); the weights padded with zeros to a multiple of kRwtPad
constexpr int kRwtPad = 256;
int wgm_graph_in_edges(wgm_graph* g);
size_t wgm_row_id_words(int32_t n);
int wgm_row_ids(wgm_graph* g, int32_t* id, int32_t* rows);
