// C ABI of one device-resident CA domain (include/amca3d.h).
//
// The reference keeps the grid as raw host arrays owned by
// CellularAutomataManager (CellularAutomataManager.cpp:303-326) and one heap
// Grain per solid cell.  Here the grid and the per-cell envelopes live in HBM
// for the lifetime of the handle, a step is a fixed sequence of six or twelve
// kernel launches that reads every scalar it needs from device memory, and the host
// only reads the counters back between batches of steps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/amca3d.h"
#include "env.h"
#include "plain_step.h"

namespace {

constexpr long long kFusedCells = 1ll << 24;

// When a domain that may take the short step takes the long one: while its wave-1
// grains in steps with a wave-1 claim (DevCounters::w1_walk) are more than kWalkShort
// a step.  In the short step k_tail's one work-group walks them, about 4 us for every
// thousand, against some 18 us a step saved by the shorter form.  How many there are
// depends on the growth per step, the truncation and the density of the grains, so
// it is measured as the run goes.  Short against long form, us a step (walked grains a
// step): 128^3 68.7 / 74.4 (2925), 102 / 94 (7489); 160^3 66.1 / 76.6 (2813), 103 / 89
// (9347); 200^3 71.8 / 84.2 (2343), 97 / 87 (8538); 256^3 93 / 100 (2863), 102 / 102
// (4510), 128 / 106 (10600), 372 / 152 (61145).  They break even near 5000; claims come
// singly at first, and a limit that a few of them within one look pass makes the form
// change for nothing (256^3 at factor 0.1, ms a run at limits of 4500, 6000 and 9000:
// 60.4, 59.5, 58.8, short throughout 58.3; at factor 0.25 38.2, 38.1, 40.4 and 42.8).
// In a batch the launches are shared (4 to 8 us a step between the forms) and any
// member's walk holds up the rest, so kWalkBatch is the limit for the members' sum: 8
// domains of 160^3 58.1 ms a run, short or long throughout 59.3 and 60.4; 4 of 256^3
// 94.0, 112 and 92.9.
constexpr long long kWalkShort = 7000, kWalkBatch = 2000;
constexpr long long kFormSteps = 8;  // steps between looks at w1_walk, at least
// More than kBurstSites live sites in more than kBurstCells cells may nucleate in a burst
// of a few tens of steps, over before a look can answer it, so such a domain takes the
// long step from the start until an eighth of kBurstSites is left.  256^3 with 2.7e5
// sites: 50 ms a run by the walk alone, 37 with the long step from the start; 160^3 with
// 3.3e4: 20.6 and 21.6, but at 1 K a step, where they all nucleate within ten steps, 19.5
// and 10.0; 200^3 with 1.9e4: 27.8 and 29.7, at 1 K a step 22.7 and 18.5; 240^3 with 1.1e4:
// 33.3 and 37.6, 25.7 and 26.5.
constexpr int kBurstSites = 24000;
constexpr long long kBurstCells = 1ll << 21;

thread_local std::string g_last_error;

amca_status fail(amca_status st, const std::string& msg) {
  g_last_error = msg;
  return st;
}

#define HIP_TRY(expr)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (expr);                                                             \
    if (e_ != hipSuccess)                                                               \
      return fail(AMCA_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));     \
  } while (0)

enum KernelId {
  K_NUCLEATE = 0, K_CLAIM, K_RESOLVE, K_EMIT, K_TAIL, K_IDSCAN, K_COMPACT, K_CNT, K_COUNT
};
// named as the kernels are, so event times line up with a kernel trace (the short
// step's k_wake_claim counts as k_claim)
const char* kKernelNames[K_COUNT] = {"k_nucleate", "k_claim",   "k_resolve", "k_emit",
                                     "k_tail",     "k_idscan",  "k_compact", "k_count"};

}  // namespace

struct amca_domain {
  int device = 0;
  hipStream_t stream = nullptr;
  amca_domain_desc desc{};
  amca::DevParams P{};
  amca::DevBuffers B{};
  int site_cap = 0;
  int orient_pushed = 0;
  int nuc_blocks = 1;
  int list_blocks = 1;
  int emit_blocks = 1;
  int ids_blocks = 1;
  bool timing = false;
  // event pairs recorded around timed launches, resolved when times are read
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<int, size_t>> ev_pending;  // (kernel id, index of first event)
  size_t ev_used = 0;
  double kernel_ms[K_COUNT] = {};
  int64_t kernel_launches[K_COUNT] = {};
  std::vector<void*> allocs;
  // graph_steps steps captured once and replayed by run / run_fixed when
  // kernel timing is off; dropped whenever a launch argument changes.
  // AMCA_DOMAIN_GRAPH_STEPS sets the count (0: no graphs, every step launched
  // on its own, for tools that do not follow graph launches).
  int graph_steps = 16;
  hipGraph_t graph[2] = {nullptr, nullptr};  // by step form (P.fused)
  hipGraphExec_t gexec[2] = {nullptr, nullptr};
  // step form: whether the short one may be taken, compaction blocks by form, and the
  // counters at the last look at w1_walk
  bool may_fuse = false, walk_ok = true, many_sites = false;
  int cmp_blocks[2] = {1, 1};
  long long seen_step = 0, seen_walk = 0;
  // room of the lists that only a running step holds anything in
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  // counters copied behind a stretch of queued steps (pinned) and the event behind
  // the copy, for two stretches in flight (run_steps)
  amca::DevCounters* look[2] = {nullptr, nullptr};
  hipEvent_t looked[2] = {nullptr, nullptr};

  void set_form(int fused) {
    P.fused = fused;
    P.cmp_blocks = cmp_blocks[fused];
  }

  void drop_graph() {
    for (int f = 0; f < 2; f++) {
      if (gexec[f]) (void)hipGraphExecDestroy(gexec[f]);
      if (graph[f]) (void)hipGraphDestroy(graph[f]);
      gexec[f] = nullptr;
      graph[f] = nullptr;
    }
  }

  template <class T>
  amca_status alloc(T** p, size_t count) {
    void* q = nullptr;
    size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
    hipError_t e = hipMalloc(&q, bytes);
    if (e != hipSuccess)
      return fail(AMCA_ERR_HIP, std::string("hipMalloc(") + std::to_string(bytes) +
                                    "): " + hipGetErrorString(e));
    allocs.push_back(q);
    *p = static_cast<T*>(q);
    return AMCA_OK;
  }

  ~amca_domain() {
    if (stream) (void)hipStreamSynchronize(stream);
    drop_graph();
    for (void* p : allocs) (void)hipFree(p);
    for (auto& e : ev_pool)
      if (e) (void)hipEventDestroy(e);
    for (auto& e : looked)
      if (e) (void)hipEventDestroy(e);
    for (auto& p : look)
      if (p) (void)hipHostFree(p);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

#define AMCA_TRY(expr)                  \
  do {                                  \
    amca_status s_ = (expr);            \
    if (s_ != AMCA_OK) return s_;       \
  } while (0)

amca_status read_counters(amca_domain* d, amca::DevCounters* c) {
  HIP_TRY(hipMemcpyAsync(c, d->B.ctr, sizeof(*c), hipMemcpyDeviceToHost, d->stream));
  HIP_TRY(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

void fill_counters(const amca_domain* d, const amca::DevCounters& c, amca_counters* out) {
  if (!out) return;
  out->step = c.step;
  out->time = c.t;
  out->dt = c.dt;
  out->n_liquid = d->P.N - c.n_solid;
  out->n_grains = c.n_grains;
  out->n_orient = c.n_orient;
  out->n_active = c.nA_in;
  out->n_sites = c.n_sites;
  out->done = (c.done || !(c.t < d->desc.final_time)) ? 1 : 0;
  out->max_wave = c.max_wave;
}

amca_status resolve_events(amca_domain* d) {
  if (d->ev_pending.empty()) return AMCA_OK;
  HIP_TRY(hipStreamSynchronize(d->stream));
  for (auto& p : d->ev_pending) {
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, d->ev_pool[p.second], d->ev_pool[p.second + 1]));
    d->kernel_ms[p.first] += ms;
    d->kernel_launches[p.first] += 1;
  }
  d->ev_pending.clear();
  d->ev_used = 0;
  return AMCA_OK;
}

template <class F>
amca_status timed(amca_domain* d, int k, F&& launch) {
  if (!d->timing) {
    HIP_TRY(launch());
    return AMCA_OK;
  }
  if (d->ev_used + 2 > d->ev_pool.size()) {
    if (d->ev_pool.size() >= 1u << 16) AMCA_TRY(resolve_events(d));
    while (d->ev_used + 2 > d->ev_pool.size()) {
      hipEvent_t e;
      HIP_TRY(hipEventCreate(&e));
      d->ev_pool.push_back(e);
    }
  }
  const size_t i = d->ev_used;
  d->ev_used += 2;
  HIP_TRY(hipEventRecord(d->ev_pool[i], d->stream));
  HIP_TRY(launch());
  HIP_TRY(hipEventRecord(d->ev_pool[i + 1], d->stream));
  d->ev_pending.emplace_back(k, i);
  return AMCA_OK;
}

// The fixed launch sequence of one step.
amca_status enqueue_step(amca_domain* d) {
  const amca::DevParams& P = d->P;
  const amca::DevBuffers& B = d->B;
  hipStream_t s = d->stream;
  AMCA_TRY(timed(d, K_NUCLEATE, [&] { return amca::launch_nucleate(P, B, d->nuc_blocks, s); }));
  if (P.fused) {
    AMCA_TRY(timed(d, K_CLAIM, [&] { return amca::launch_wake_claim(P, B, s); }));
    AMCA_TRY(timed(d, K_RESOLVE, [&] { return amca::launch_resolve(P, B, 0, P.cmp_blocks, s); }));
    AMCA_TRY(timed(d, K_IDSCAN, [&] { return amca::launch_idscan(P, B, 0, P.cmp_blocks, s); }));
    AMCA_TRY(timed(d, K_EMIT, [&] { return amca::launch_emit(P, B, 0, P.cmp_blocks, s); }));
    AMCA_TRY(timed(d, K_TAIL, [&] { return amca::launch_tail(P, B, s); }));
    return AMCA_OK;
  }
  AMCA_TRY(timed(d, K_CNT, [&] { return amca::launch_count(P, B, P.cmp_blocks, s); }));
  AMCA_TRY(timed(d, K_COMPACT, [&] { return amca::launch_compact(P, B, P.cmp_blocks, s); }));
  for (int wave = 0; wave < 2; wave++) {
    AMCA_TRY(timed(d, K_CLAIM, [&] { return amca::launch_claim(P, B, wave, d->list_blocks, s); }));
    AMCA_TRY(timed(d, K_RESOLVE,
                   [&] { return amca::launch_resolve(P, B, wave, d->emit_blocks, s); }));
    AMCA_TRY(timed(d, K_IDSCAN,
                   [&] { return amca::launch_idscan(P, B, wave, d->emit_blocks, s); }));
    AMCA_TRY(timed(d, K_EMIT, [&] { return amca::launch_emit(P, B, wave, d->emit_blocks, s); }));
  }
  AMCA_TRY(timed(d, K_TAIL, [&] { return amca::launch_tail(P, B, s); }));
  return AMCA_OK;
}

amca_status capture_steps(amca_domain* d) {
  HIP_TRY(hipStreamBeginCapture(d->stream, hipStreamCaptureModeThreadLocal));
  amca_status st = AMCA_OK;
  for (int q = 0; q < d->graph_steps && st == AMCA_OK; q++) st = enqueue_step(d);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(d->stream, &g);
  if (st != AMCA_OK || e != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return st != AMCA_OK ? st : fail(AMCA_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(e));
  }
  const int f = d->P.fused;
  if (d->graph[f]) (void)hipGraphDestroy(d->graph[f]);
  d->graph[f] = g;
  HIP_TRY(hipGraphInstantiate(&d->gexec[f], g, nullptr, nullptr, 0));
  return AMCA_OK;
}

// The step form for the coming steps, from the live sites and the walk of the steps
// since the last look.  Every step leaves the same state in either form.
void choose_form(amca_domain* d, const amca::DevCounters& c) {
  if (!d->may_fuse) return;
  const long long steps = c.step - d->seen_step;
  if (steps >= kFormSteps) {
    d->walk_ok = c.w1_walk - d->seen_walk <= kWalkShort * steps;
    d->seen_step = c.step;
    d->seen_walk = c.w1_walk;
  }
  d->many_sites = d->P.N > kBurstCells && c.n_sites > (d->many_sites ? kBurstSites / 8 : kBurstSites);
  d->set_form(d->walk_ok && !d->many_sites ? 1 : 0);
}

// n steps: whole graphs of graph_steps steps, then single launches (every
// launch is single, with its events, when kernel timing is on).  Steps past
// termination do nothing, so a graph may run beyond the last live step.
amca_status enqueue_steps(amca_domain* d, long long n) {
  if (!d->timing && d->graph_steps > 0) {
    for (; n >= d->graph_steps; n -= d->graph_steps) {
      if (!d->gexec[d->P.fused]) AMCA_TRY(capture_steps(d));
      HIP_TRY(hipGraphLaunch(d->gexec[d->P.fused], d->stream));
    }
  }
  for (; n > 0; n--) AMCA_TRY(enqueue_step(d));
  return AMCA_OK;
}

// Up to `most` steps (negative: no limit), until the run is over if `to_end`; *c holds
// the counters before and after.  Two stretches of steps are in flight, so that the
// look at one stretch's counters costs the GPU no more than the copy; 16 steps each
// where the form, which follows the look a stretch late, may cost more than the copies
// (128^3 with 8.3e4 sites 19.7 ms in stretches of 32, 17.7 of 16; 60^3 0.9 % slower in
// those), else 32 (the steps queued past the end of a run do nothing, but 512^3 takes
// 30 us for each), or a graph's length where that was set longer.
amca_status run_steps(amca_domain* d, long long most, bool to_end, amca::DevCounters* c) {
  for (int q = 0; q < 2; q++) {
    if (!d->look[q]) HIP_TRY(hipHostMalloc(&d->look[q], sizeof(amca::DevCounters)));
    if (!d->looked[q]) HIP_TRY(hipEventCreateWithFlags(&d->looked[q], hipEventDisableTiming));
  }
  const long long graph = to_end ? std::min(d->graph_steps, 64) : d->graph_steps;
  const long long longest = std::max(d->may_fuse && d->P.N > (1ll << 20) ? 16LL : 32LL, graph);
  long long len = 8, queued = 0;
  long long made = 0, seen = 0;  // stretches queued and looked at
  while (true) {
    const bool over = c->err || (to_end && (c->done || !(c->t < d->desc.final_time)));
    for (; !over && made - seen < 2 && (most < 0 || queued < most); made++) {
      const long long k = most < 0 ? len : std::min(len, most - queued);
      choose_form(d, *c);
      AMCA_TRY(enqueue_steps(d, k));
      HIP_TRY(hipMemcpyAsync(d->look[made & 1], d->B.ctr, sizeof(amca::DevCounters),
                             hipMemcpyDeviceToHost, d->stream));
      HIP_TRY(hipEventRecord(d->looked[made & 1], d->stream));
      queued += k;
      len = std::min(2 * len, longest);
    }
    if (made == seen) return AMCA_OK;
    HIP_TRY(hipEventSynchronize(d->looked[seen & 1]));
    *c = *d->look[seen++ & 1];
  }
}

// Every live site can nucleate once and takes the next orientation row, so a
// run may start only when the pushed rows cover the orientations in use plus
// one per live site.  The kernels never read a row that was not pushed.
amca_status check_rows(amca_domain* d, const amca::DevCounters& c) {
  if ((long long)c.n_orient + c.n_sites > d->orient_pushed)
    return fail(AMCA_ERR_CAPACITY,
                "orientation rows pushed (" + std::to_string(d->orient_pushed) +
                    ") do not cover the orientations in use plus one per live site (" +
                    std::to_string((long long)c.n_orient + c.n_sites) +
                    "): push more rows with amca_domain_push_orientations");
  return AMCA_OK;
}

amca_status check_err(amca_domain* d, const amca::DevCounters& c) {
  if (c.err)
    return fail(AMCA_ERR_CAPACITY,
                "orientation table exhausted: push more rows with amca_domain_push_orientations");
  return AMCA_OK;
}

}  // namespace

namespace {
template <class F>
struct ScopeExit {
  F f;
  ~ScopeExit() { f(); }
};
template <class F>
ScopeExit<F> on_scope_exit(F f) {
  return {f};
}
}  // namespace

extern "C" {

const char* amca_last_error(void) { return g_last_error.c_str(); }
const char* amca_version(void) { return "amca3d-mi355x 0.1 (gfx950)"; }

amca_status amca_domain_create(const amca_domain_desc* desc, int32_t orient_capacity,
                               amca_domain** out) {
  if (!desc || !out) return fail(AMCA_ERR_INVALID, "null argument");
  *out = nullptr;
  if (desc->nx < 1 || desc->ny < 1 || desc->nz < 1)
    return fail(AMCA_ERR_INVALID, "domain needs at least one cell per axis");
  const long long nxG = desc->nx + 2LL, nyG = desc->ny + 2LL, nzG = desc->nz + 2LL;
  const long long NG = nxG * nyG * nzG;
  if (NG > (long long)INT_MAX)
    return fail(AMCA_ERR_INVALID, "ghosted grid exceeds 2^31-1 cells (int32 cell index)");
  if (!(desc->h > 0)) return fail(AMCA_ERR_INVALID, "cell size must be positive");
  if (orient_capacity < 0) return fail(AMCA_ERR_INVALID, "negative orientation capacity");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return fail(AMCA_ERR_NO_DEVICE, "no HIP device visible");

  auto* d = new amca_domain();
  HIP_TRY(hipGetDevice(&d->device));
  HIP_TRY(hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking));
  d->desc = *desc;
  amca::DevParams& P = d->P;
  P.nx = desc->nx; P.ny = desc->ny; P.nz = desc->nz;
  P.nxG = (int)nxG; P.nyG = (int)nyG; P.nzG = (int)nzG;
  P.nxyG = (int)(nxG * nyG);
  P.NG = (int)NG;
  P.nbX = (int)((nxG + 3) / 4);
  P.nbY = (int)((nyG + 3) / 4);
  P.nbZ = (int)((nzG + 3) / 4);
  P.fdX = amca::make_fastdiv((unsigned)P.nbX);
  P.fdY = amca::make_fastdiv((unsigned)P.nbY);
  P.N = (long long)desc->nx * desc->ny * desc->nz;
  const long long nB = (long long)P.nbX * P.nbY * P.nbZ;
  if (64 * nB > (long long)INT_MAX) {
    delete d;
    return fail(AMCA_ERR_INVALID, "grid exceeds 2^31-1 brick slots (int32 slot index)");
  }
  P.h = desc->h; P.x0 = desc->x0; P.y0 = desc->y0; P.z0 = desc->z0;
  P.T0 = desc->T0; P.Tm = desc->Tm; P.Tdot = desc->Tdot;
  P.a1 = desc->a1; P.a2 = desc->a2; P.a3 = desc->a3;
  P.trunc = desc->trunc;
  P.tsf = desc->time_step_factor;
  P.max_dt = desc->max_dt;
  P.final_time = desc->final_time;
  P.sqrt2f = (double)sqrtf(2.0f);
  P.orient_cap = orient_capacity;
  {
    int s = 0;
    for (int dk = -1; dk <= 1; dk++)
      for (int dj = -1; dj <= 1; dj++)
        for (int di = -1; di <= 1; di++) {
          if (!dk && !dj && !di) continue;
          P.off[s++] = dk * P.nxyG + dj * P.nxG + di;
        }
  }
  amca::DevBuffers& B = d->B;
  const size_t N = (size_t)P.N;
  // One allocation for everything whose size the grid fixes: a domain made and
  // dropped per run (a batch of 16: 560 allocations) otherwise spends tens of
  // milliseconds on them.
  struct Part {
    void** p;
    size_t bytes;
  };
  std::vector<Part> parts;
  const auto want_buf = [&](auto** p, size_t n) {
    parts.push_back({reinterpret_cast<void**>(p), (std::max<size_t>(n, 1) * sizeof(**p) + 255) / 256 * 256});
  };
  want_buf(&B.gid, (size_t)NG);
  want_buf(&B.oid, (size_t)NG);
  want_buf(&B.claim, 64 * (size_t)nB);  // brick order (claim_index)
  want_buf(&B.bmap, 2 * (size_t)nB);
  want_buf(&B.amap, (size_t)nB);
  want_buf(&B.rec, 64 * (size_t)nB);
  want_buf(&B.wake, 64 * (size_t)nB);
  want_buf(&B.inc, amca::kRing);
  want_buf(&B.cl1, (size_t)nB);
  want_buf(&B.awk, (size_t)nB);
  want_buf(&B.genv, N);
  want_buf(&B.alist, 64 * (size_t)nB);  // from here to masks: of a step, `scratch` between steps
  want_buf(&B.plist, 64 * (size_t)nB);
  want_buf(&B.masks, 64 * (size_t)nB);
  want_buf(&B.cnt, N + 64);  // the id scan reads whole 16-byte groups past the last id
  want_buf(&B.coff, N);
  want_buf(&B.idtot, amca::kMaxIdsBlocks);
  want_buf(&B.cmptot, amca::kMaxBlocks);
  want_buf(&B.listW[1], N);
  want_buf(&B.l2g, 9 * (size_t)std::max(orient_capacity, 1));
  want_buf(&B.lb_flag, (size_t)amca::kLbSites * amca::kMaxBlocks);
  want_buf(&B.lb_agg, (size_t)amca::kLbSites * amca::kMaxBlocks);
  want_buf(&B.lb_pref, (size_t)amca::kLbSites * amca::kMaxBlocks);
  want_buf(&B.ctr, 1);
  want_buf(&B.site_cell[0], 1);
  want_buf(&B.site_cell[1], 1);
  want_buf(&B.site_dt[0], 1);
  want_buf(&B.site_dt[1], 1);
  size_t total = 0;
  for (const Part& q : parts) total += q.bytes;
  char* arena = nullptr;
  const amca_status st = d->alloc(&arena, total);
  if (st != AMCA_OK) {
    delete d;
    return st;
  }
  for (const Part& q : parts) {
    *q.p = arena;
    arena += q.bytes;
  }
  // Shared room (12 bytes a cell, 1.6 of 22 GB at 512^3: the driver clears what a
  // domain gives back, 0.45 s for 22 GB, and a program that makes large domains one
  // after another waits for it).  Wave 0's list is last read by its k_resolve, and its
  // k_emit then writes wave 1's; the parent list holds nothing between steps, when a
  // download writes the (cell, orientation) pairs.
  B.listW[0] = B.alist;
  B.gco = reinterpret_cast<int2*>(B.plist);
  d->scratch = B.alist;
  d->scratch_bytes = reinterpret_cast<char*>(B.masks + 64 * (size_t)nB) - reinterpret_cast<char*>(B.alist);
  B.log = nullptr;
  d->site_cap = 1;
  HIP_TRY(hipMemsetAsync(B.lb_flag, 0, sizeof(unsigned) * amca::kLbSites * amca::kMaxBlocks, d->stream));
  HIP_TRY(hipMemsetAsync(B.cnt, 0, N + 64, d->stream));
  amca::DevCounters c{};
  c.t = 0.0;
  HIP_TRY(hipMemcpyAsync(B.ctr, &c, sizeof(c), hipMemcpyHostToDevice, d->stream));
  HIP_TRY(amca::launch_init_grid(P, B, d->stream));
  // Grid sizes.  The list kernels hold four blocks on a CU (their registers), and an
  // entry is a chain of dependent loads, so they take as many blocks as the card
  // holds at once, each with its share of the list: 512^3, claim / resolve / emit of
  // wave 0 in us at 16, 12, 8 and 4 blocks per CU: 88 / 92 / 60, 86 / 88 / 56,
  // 83 / 84 / 53, 80 / 80 / 50; at 3 and 2, claim / emit 85 / 52 and 97 / 57.
  int cus = 256;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, d->device) == hipSuccess && prop.multiProcessorCount > 0)
    cus = prop.multiProcessorCount;
  long long want = (P.N + amca::kBlock - 1) / amca::kBlock;
  d->list_blocks = (int)std::max(8LL, std::min<long long>((want + 7) / 8 * 8, 4LL * cus));
  d->emit_blocks = (int)std::max(8LL, std::min<long long>((want + 7) / 8 * 8, std::min(4LL * cus, (long long)amca::kMaxBlocks)));
  d->nuc_blocks = 1;
  // id scan: eight blocks per CU at most (each block's tiles run one after
  // another), at least 32 K ids per block
  d->ids_blocks = (int)std::max(1LL, std::min<long long>((P.N + 32767) / 32768,
                                                         std::min(8LL * cus, (long long)amca::kMaxIdsBlocks)));
  P.ids_blocks = d->ids_blocks;
  // The short step (see plain_step.hip) may be taken on grids of up to kFusedCells
  // whose grains grow at most a quarter of a cell per step (dt <= time_step_factor
  // h / v): there captures by wave 1's fresh envelopes, which k_tail takes with one
  // work-group, are rare unless the grains are dense or the truncation is large
  // (choose_form).  Short against long form, us a step, at 5e13 sites a cubic metre:
  // 64^3 39 / 53, 128^3 50 / 67, 200^3 64 / 85, 256^3 93 / 100, 320^3 152 / 129.
  d->may_fuse = P.N <= kFusedCells && desc->time_step_factor <= 0.25;
  // compaction and retirement: the 64-brick pieces of the grid over at most eight
  // blocks per CU; two for the short step, whose wave-0 kernels all have these blocks
  // and each of them starts up for a few dozen entries (256^3: 113, 101 and 98 us a
  // step at 8, 4 and 2 per CU; 512^3 long form: 347, 346, 381)
  for (int f = 0; f < 2; f++)
    d->cmp_blocks[f] = (int)std::max(1LL, std::min<long long>((nB + 63) / 64,
                                                              std::min((f ? 2LL : 8LL) * cus,
                                                                       (long long)amca::kMaxBlocks)));
  d->set_form(d->may_fuse ? 1 : 0);
  if (amca::env_int("AMCA_DOMAIN_GRAPH_STEPS", 0, 1024, &d->graph_steps) < 0) {
    delete d;
    return fail(AMCA_ERR_INVALID, "AMCA_DOMAIN_GRAPH_STEPS must be an integer in [0, 1024]");
  }
  HIP_TRY(hipStreamSynchronize(d->stream));
  *out = d;
  return AMCA_OK;
}

amca_status amca_domain_destroy(amca_domain* d) {
  if (!d) return AMCA_OK;
  (void)hipStreamSynchronize(d->stream);  // the handle goes either way
  delete d;
  return AMCA_OK;
}

amca_status amca_domain_set_sites(amca_domain* d, int32_t n, const int32_t* cell,
                                  const double* dT_crit) {
  if (!d || n < 0 || (n > 0 && (!cell || !dT_crit))) return fail(AMCA_ERR_INVALID, "bad sites");
  for (int i = 0; i < n; i++) {
    if (cell[i] < 0 || cell[i] >= d->P.NG) return fail(AMCA_ERR_INVALID, "site cell out of range");
    if (i > 0 && cell[i] <= cell[i - 1])
      return fail(AMCA_ERR_INVALID, "sites must be strictly ascending by cell");
  }
  HIP_TRY(hipStreamSynchronize(d->stream));
  d->drop_graph();  // site buffers and the nucleation grid may change
  int cap = std::max(n, 1);
  if (cap > d->site_cap) {
    for (int b = 0; b < 2; b++) {
      for (auto& p : d->allocs) {
        if (p == d->B.site_cell[b] || p == d->B.site_dt[b]) {
          (void)hipFree(p);
          p = nullptr;
        }
      }
    }
    d->allocs.erase(std::remove(d->allocs.begin(), d->allocs.end(), nullptr), d->allocs.end());
    for (int b = 0; b < 2; b++) {
      AMCA_TRY(d->alloc(&d->B.site_cell[b], (size_t)cap));
      AMCA_TRY(d->alloc(&d->B.site_dt[b], (size_t)cap));
    }
    d->site_cap = cap;
  }
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  if (n > 0) {
    HIP_TRY(hipMemcpyAsync(d->B.site_cell[c.site_sel], cell, sizeof(int32_t) * n,
                           hipMemcpyHostToDevice, d->stream));
    HIP_TRY(hipMemcpyAsync(d->B.site_dt[c.site_sel], dT_crit, sizeof(double) * n,
                           hipMemcpyHostToDevice, d->stream));
  }
  c.n_sites = n;
  HIP_TRY(hipMemcpyAsync(d->B.ctr, &c, sizeof(c), hipMemcpyHostToDevice, d->stream));
  long long want = ((long long)n + amca::kBlock - 1) / amca::kBlock;
  d->nuc_blocks = (int)std::max(1LL, std::min<long long>(want, amca::kMaxBlocks));
  HIP_TRY(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

amca_status amca_domain_push_orientations(amca_domain* d, int32_t n, const double* euler3,
                                          const double* l2g9) {
  (void)euler3;
  if (!d || n < 0 || (n > 0 && !l2g9)) return fail(AMCA_ERR_INVALID, "bad orientation rows");
  if (d->orient_pushed + n > d->P.orient_cap)
    return fail(AMCA_ERR_CAPACITY, "orientation table capacity exceeded");
  if (n > 0)
    HIP_TRY(hipMemcpyAsync(d->B.l2g + 9 * (size_t)d->orient_pushed, l2g9, sizeof(double) * 9 * n,
                           hipMemcpyHostToDevice, d->stream));
  d->orient_pushed += n;
  HIP_TRY(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

amca_status amca_domain_step(amca_domain* d, amca_counters* out) {
  if (!d) return fail(AMCA_ERR_INVALID, "null domain");
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  AMCA_TRY(check_rows(d, c));
  choose_form(d, c);
  AMCA_TRY(enqueue_step(d));
  AMCA_TRY(read_counters(d, &c));
  fill_counters(d, c, out);
  return check_err(d, c);
}

amca_status amca_domain_run(amca_domain* d, int64_t max_steps, amca_counters* out) {
  if (!d) return fail(AMCA_ERR_INVALID, "null domain");
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  AMCA_TRY(check_rows(d, c));
  AMCA_TRY(run_steps(d, max_steps, true, &c));
  fill_counters(d, c, out);
  return check_err(d, c);
}

amca_status amca_domain_run_fixed(amca_domain* d, int64_t n_steps) {
  if (!d || n_steps < 0) return fail(AMCA_ERR_INVALID, "bad arguments");
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  AMCA_TRY(check_rows(d, c));
  if (d->may_fuse) return run_steps(d, n_steps, false, &c);
  AMCA_TRY(enqueue_steps(d, n_steps));
  HIP_TRY(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

amca_status amca_domain_counters(amca_domain* d, amca_counters* out) {
  if (!d || !out) return fail(AMCA_ERR_INVALID, "null argument");
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  fill_counters(d, c, out);
  return check_err(d, c);
}

amca_status amca_domain_enable_log(amca_domain* d, int32_t capacity) {
  if (!d || capacity < 0) return fail(AMCA_ERR_INVALID, "bad arguments");
  HIP_TRY(hipStreamSynchronize(d->stream));
  d->drop_graph();  // the log pointer is a launch argument
  if (d->B.log) {
    for (auto& p : d->allocs)
      if (p == d->B.log) {
        (void)hipFree(p);
        p = nullptr;
      }
    d->allocs.erase(std::remove(d->allocs.begin(), d->allocs.end(), nullptr), d->allocs.end());
    d->B.log = nullptr;
  }
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  c.log_cap = capacity;
  if (capacity > 0) AMCA_TRY(d->alloc(&d->B.log, (size_t)capacity));
  HIP_TRY(hipMemcpyAsync(d->B.ctr, &c, sizeof(c), hipMemcpyHostToDevice, d->stream));
  HIP_TRY(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

amca_status amca_domain_read_log(amca_domain* d, int32_t cap, amca_step_record* rows,
                                 int32_t* n_rows) {
  if (!d || !n_rows) return fail(AMCA_ERR_INVALID, "null argument");
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  const long long avail = std::min<long long>(c.step, c.log_cap);
  *n_rows = (int32_t)avail;  // rows available; at most `cap` are copied
  const long long n = std::min<long long>(avail, std::max(cap, 0));
  if (n > 0 && rows && d->B.log) {
    std::vector<amca::StepLogRow> tmp((size_t)n);
    HIP_TRY(hipMemcpy(tmp.data(), d->B.log, sizeof(amca::StepLogRow) * n, hipMemcpyDeviceToHost));
    for (long long i = 0; i < n; i++) {
      rows[i].time_before = tmp[i].time_before;
      rows[i].dt = tmp[i].dt;
      rows[i].n_nucleated = tmp[i].n_nucleated;
      rows[i].n_active_before = tmp[i].n_active_before;
      rows[i].n_captured = tmp[i].n_captured;
      rows[i].n_active_after = tmp[i].n_active_after;
      rows[i].n_liquid = tmp[i].n_liquid;
      rows[i].n_wave1 = tmp[i].n_wave1;
      rows[i].max_wave = tmp[i].max_wave;
      rows[i].n_sites = tmp[i].n_sites;
    }
  }
  return AMCA_OK;
}

amca_status amca_domain_download(amca_domain* d, int32_t* orient, int32_t* grain, double* env,
                                 int32_t site_cap, int32_t* site_cell, double* site_dt,
                                 int32_t* n_sites) {
  if (!d) return fail(AMCA_ERR_INVALID, "null domain");
  const size_t NG = (size_t)d->P.NG;
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  // the grain-ID fields, materialized from the slots
  if (orient || grain) {
    HIP_TRY(amca::launch_materialize(d->P, d->B, amca::kMatFields, d->stream));
    HIP_TRY(hipStreamSynchronize(d->stream));
  }
  if (orient) HIP_TRY(hipMemcpy(orient, d->B.oid, sizeof(int32_t) * NG, hipMemcpyDeviceToHost));
  if (grain) HIP_TRY(hipMemcpy(grain, d->B.gid, sizeof(int32_t) * NG, hipMemcpyDeviceToHost));
  if (env) {
    // laid out by cell on the device, a piece of up to 64 MB at a time (the host's
    // memset and scatter of the records took longer than the run of a small grid), in
    // the room of a step's lists: no allocation that could fail or be waited for
    const size_t piece = std::min<size_t>({NG, d->scratch_bytes / sizeof(double4), (size_t)1 << 21});
    double4* buf = static_cast<double4*>(d->scratch);
    for (size_t c0 = 0; c0 < NG; c0 += piece) {
      const int n = (int)std::min(piece, NG - c0);
      HIP_TRY(amca::launch_cell_env(d->P, d->B, (long long)c0, n, buf, d->stream));
      HIP_TRY(hipMemcpyAsync(env + 4 * c0, buf, sizeof(double4) * n, hipMemcpyDeviceToHost, d->stream));
      HIP_TRY(hipStreamSynchronize(d->stream));
    }
  }
  if (n_sites) *n_sites = c.n_sites;
  int m = std::min(c.n_sites, site_cap);
  if (m > 0 && site_cell)
    HIP_TRY(hipMemcpy(site_cell, d->B.site_cell[c.site_sel], sizeof(int32_t) * m, hipMemcpyDeviceToHost));
  if (m > 0 && site_dt)
    HIP_TRY(hipMemcpy(site_dt, d->B.site_dt[c.site_sel], sizeof(double) * m, hipMemcpyDeviceToHost));
  return AMCA_OK;
}

amca_status amca_domain_download_grains(amca_domain* d, int32_t cap, double* env4, int32_t* cell,
                                        int32_t* orient, int32_t* n_grains) {
  if (!d || !n_grains) return fail(AMCA_ERR_INVALID, "null argument");
  amca::DevCounters c;
  AMCA_TRY(read_counters(d, &c));
  *n_grains = c.n_grains;
  const size_t m = (size_t)std::max(0, std::min(cap, c.n_grains));
  if (m == 0) return AMCA_OK;
  HIP_TRY(amca::launch_materialize(d->P, d->B, amca::kMatGrains, d->stream));
  HIP_TRY(hipStreamSynchronize(d->stream));
  if (env4) {
    HIP_TRY(hipMemcpy(env4, d->B.genv, sizeof(double) * 4 * m, hipMemcpyDeviceToHost));
  }
  if (cell || orient) {
    std::vector<int32_t> co(2 * m);
    HIP_TRY(hipMemcpy(co.data(), d->B.gco, sizeof(int32_t) * 2 * m, hipMemcpyDeviceToHost));
    for (size_t g = 0; g < m; g++) {
      if (cell) cell[g] = co[2 * g];
      if (orient) orient[g] = co[2 * g + 1];
    }
  }
  return AMCA_OK;
}

amca_status amca_domain_device_fields(amca_domain* d, void** orient, void** grain, void** env,
                                      void** stream) {
  if (!d) return fail(AMCA_ERR_INVALID, "null domain");
  if (orient || grain || env) {
    HIP_TRY(amca::launch_materialize(d->P, d->B, amca::kMatDevice, d->stream));
    HIP_TRY(hipStreamSynchronize(d->stream));
  }
  if (orient) *orient = d->B.oid;
  if (grain) *grain = d->B.gid;
  if (env) *env = d->B.genv;
  if (stream) *stream = d->stream;
  return AMCA_OK;
}

amca_status amca_domain_enable_timing(amca_domain* d, int32_t on) {
  if (!d) return fail(AMCA_ERR_INVALID, "null domain");
  AMCA_TRY(resolve_events(d));
  d->timing = on != 0;
  for (int k = 0; k < K_COUNT; k++) {
    d->kernel_ms[k] = 0.0;
    d->kernel_launches[k] = 0;
  }
  return AMCA_OK;
}

int32_t amca_kernel_count(void) { return K_COUNT; }

const char* amca_kernel_name(int32_t i) {
  if (i < 0 || i >= K_COUNT) return "";
  return kKernelNames[i];
}

amca_status amca_domain_kernel_times(amca_domain* d, double* ms, int64_t* launches) {
  if (!d) return fail(AMCA_ERR_INVALID, "null domain");
  AMCA_TRY(resolve_events(d));
  for (int k = 0; k < K_COUNT; k++) {
    if (ms) ms[k] = d->kernel_ms[k];
    if (launches) launches[k] = d->kernel_launches[k];
  }
  return AMCA_OK;
}

amca_status amca_envelope_selftest(int32_t n, const double* env4, const double* l2g9,
                                   const double* cell3, double h, double trunc,
                                   int32_t* inside, double* child4) {
  if (n < 0 || (n > 0 && (!env4 || !l2g9 || !cell3 || !inside || !child4)))
    return fail(AMCA_ERR_INVALID, "bad arguments");
  if (n == 0) return AMCA_OK;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return fail(AMCA_ERR_NO_DEVICE, "no HIP device visible");
  double *de = nullptr, *dr = nullptr, *dc = nullptr, *dout = nullptr;
  int* din = nullptr;
  // device buffers freed on every path, the early error returns included
  const auto release = on_scope_exit([&] {
    for (void* q : {(void*)de, (void*)dr, (void*)dc, (void*)dout, (void*)din})
      if (q) (void)hipFree(q);
  });
  HIP_TRY(hipMalloc(&de, sizeof(double) * 4 * n));
  HIP_TRY(hipMalloc(&dr, sizeof(double) * 9 * n));
  HIP_TRY(hipMalloc(&dc, sizeof(double) * 3 * n));
  HIP_TRY(hipMalloc(&dout, sizeof(double) * 4 * n));
  HIP_TRY(hipMalloc(&din, sizeof(int) * n));
  HIP_TRY(hipMemcpy(de, env4, sizeof(double) * 4 * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(dr, l2g9, sizeof(double) * 9 * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(dc, cell3, sizeof(double) * 3 * n, hipMemcpyHostToDevice));
  HIP_TRY(amca::launch_envelope_selftest(n, de, dr, dc, h, trunc, (double)sqrtf(2.0f), din, dout, 0));
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(inside, din, sizeof(int) * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(child4, dout, sizeof(double) * 4 * n, hipMemcpyDeviceToHost));
  return AMCA_OK;
}

}  // extern "C"

// ===========================================================================
// Batches: many independent plain domains stepped together.  Every kernel of
// a step is launched once for the whole batch; its blocks are split among the
// domains by a per-kernel (domain, block, count) map, so small domains that
// could not fill the device alone share it.  The steps are captured in a HIP
// graph of `steps_per_graph` steps that is replayed until every domain has
// finished; a finished domain's kernels return at once.  Results per domain
// do not depend on the block split (every kernel's result is independent of
// its block count), so each domain stays identical to its own run.

struct amca_batch {
  std::vector<amca_domain*> doms;
  std::vector<amca::DevParams> P;  // the domains' parameters with the batch's step form and grids
  // step form: whether every domain may take the short step, whether a nucleation burst
  // is still to come, and the form of the next replay; the domains' walks (w1_walk, low
  // 31 bits) when they were last looked at and the steps run since
  bool may_fuse = false, burst = false;
  int form = 0;
  std::vector<int> walk0;
  long long walk_steps = 0;
  int device = 0;
  hipStream_t stream = nullptr;
  amca::DevParams* dP = nullptr;  // by step form, n each
  amca::DevBuffers* dB = nullptr;
  int4* maps = nullptr;  // nuc | list | emit | tail | ids by form | compaction, back to back
  int4* status = nullptr;
  int4* hstatus = nullptr;  // pinned: two slots of n statuses, one per replay in flight
  hipEvent_t hready[2] = {nullptr, nullptr};
  amca::BatchLaunch L[2] = {};  // by step form
  amca_batch_schedule sched{};
  hipGraph_t graph[2] = {nullptr, nullptr};
  hipGraphExec_t exec[2] = {nullptr, nullptr};
  int graph_steps = 0;  // of both graphs
  bool use_graph = true;  // false: every replay launches its kernels one by one
  int cus = 256;
  double last_ms_per_step = 0.0;
  // domains still running when the maps were last built (finished domains get
  // no blocks) and the finished count then
  std::vector<char> active;
  int mapped_finished = 0;

  void drop_graph() {
    for (int f = 0; f < 2; f++) {
      if (exec[f]) (void)hipGraphExecDestroy(exec[f]);
      if (graph[f]) (void)hipGraphDestroy(graph[f]);
      exec[f] = nullptr;
      graph[f] = nullptr;
    }
    graph_steps = 0;
  }
  ~amca_batch() {
    if (stream) (void)hipStreamSynchronize(stream);
    drop_graph();
    if (dP) (void)hipFree(dP);
    if (dB) (void)hipFree(dB);
    if (maps) (void)hipFree(maps);
    if (status) (void)hipFree(status);
    if (hstatus) (void)hipHostFree(hstatus);
    for (auto& e : hready)
      if (e) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

// The blocks that a budget stands for: all of it up to four per CU, which are
// resident at once, then four per CU until a quarter of it is more.  Only awake
// grains are in the lists, so more blocks than that mostly start up for a
// fraction of a tile each, and far fewer leave the last ones to carry the run.
// A run's ms at 2, 4, 8 and 16 blocks per CU: 16 uneven domains, short step 83, 68,
// 70, 87, long step 86, 73, 76, 91; 64 of 32^3, long step 29, 34, 44, 49; 8 of 160^3,
// long step 63, 61, 64, 71; 4 of 256^3, long step 106, 94, 98, 106.
int budget_blocks(const amca_batch* b, int budget) {
  return std::max(budget / 4, std::min(budget, 4 * b->cus));
}

// Per-domain block counts of the list kernels under a schedule: the budget of
// `list_blocks` blocks (and emit_blocks for resolve/emit) shared in proportion
// to the domains' cell counts, at least `min_blocks` each, capped by what a
// domain can use (one block per 256 cells of its grid, kMaxBlocks for the
// scanned kernels).
void batch_geometry(const amca_batch* b, std::vector<int>& nl, std::vector<int>& ne) {
  const size_t n = b->doms.size();
  const int list = budget_blocks(b, b->sched.list_blocks);
  const int emit = budget_blocks(b, b->sched.emit_blocks);
  double total = 0.0;
  for (size_t i = 0; i < n; i++)
    if (b->active[i]) total += (double)b->doms[i]->P.N;
  nl.assign(n, 0);
  ne.assign(n, 0);
  for (size_t i = 0; i < n; i++) {
    if (!b->active[i]) continue;
    const double share = (double)b->doms[i]->P.N / total;
    const long long cap = std::max(1LL, (b->doms[i]->P.N + amca::kBlock - 1) / amca::kBlock);
    long long l = (long long)std::llround(share * list);
    long long e = (long long)std::llround(share * emit);
    l = std::max<long long>(b->sched.min_blocks, std::min(l, cap));
    // resolve / emit blocks keep per-block stats in kMaxBlocks slots
    e = std::min(std::max<long long>(b->sched.min_blocks, std::min(e, cap)), (long long)amca::kMaxBlocks);
    nl[i] = (int)std::max(1LL, l);
    ne[i] = (int)std::max(1LL, e);
  }
}

// Block order within one launch: domain-major in the given domain order
// (`interleave` = 0), or round-robin over domains so that every domain's
// blocks are spread over the whole launch (`interleave` = 1).
void build_map(const std::vector<int>& order, const std::vector<int>& cnt, int interleave,
               std::vector<int4>& out) {
  out.clear();
  if (!interleave) {
    for (int d : order)
      for (int k = 0; k < cnt[d]; k++) out.push_back(make_int4(d, k, cnt[d], 0));
    return;
  }
  int left = 1;
  for (int k = 0; left; k++) {
    left = 0;
    for (int d : order)
      if (k < cnt[d]) {
        out.push_back(make_int4(d, k, cnt[d], 0));
        left = 1;
      }
  }
}

amca_status batch_apply_schedule(amca_batch* b) {
  const int n = (int)b->doms.size();
  std::vector<int> nl, ne, nn(n), one(n, 1), ni(n), nc(n);
  batch_geometry(b, nl, ne);
  for (int i = 0; i < n; i++) {
    // a finished domain gets no blocks (its kernels would return at once)
    nn[i] = b->active[i] ? b->doms[i]->nuc_blocks : 0;
    ni[i] = b->active[i] ? b->doms[i]->ids_blocks : 0;
    // bricks over blocks as the resolve / emit budget has it, whole 64-brick pieces
    const amca::DevParams& P = b->doms[i]->P;
    const long long pieces = ((long long)P.nbX * P.nbY * P.nbZ + 63) / 64;
    nc[i] = b->active[i] ? (int)std::max(1LL, std::min<long long>({(long long)ne[i], pieces,
                                                                   (long long)amca::kMaxBlocks}))
                         : 0;
    b->P[i].cmp_blocks = std::max(1, nc[i]);
    one[i] = b->active[i] ? 1 : 0;
  }
  std::vector<int> order(n);
  for (int i = 0; i < n; i++) order[i] = i;
  // larger domains first: their blocks start earliest
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int c) { return b->doms[a]->P.N > b->doms[c]->P.N; });
  std::vector<int4> mn, ml, me, ms, mi[2], mc;
  build_map(order, nn, b->sched.interleave, mn);
  // the id scan sums the domain's k_resolve blocks (short step: of wave 0 only)
  for (int f = 0; f < 2; f++) {
    build_map(order, ni, b->sched.interleave, mi[f]);
    for (auto& m : mi[f]) m.w = f ? nc[m.x] : ne[m.x];
  }
  build_map(order, nc, b->sched.interleave, mc);
  build_map(order, nl, b->sched.interleave, ml);
  build_map(order, ne, b->sched.interleave, me);
  build_map(order, one, 0, ms);
  const size_t total =
      mn.size() + ml.size() + me.size() + ms.size() + 2 * mi[0].size() + mc.size();
  if (b->maps) HIP_TRY(hipFree(b->maps));
  b->maps = nullptr;
  HIP_TRY(hipMalloc(&b->maps, sizeof(int4) * total));
  std::vector<int4> all;
  all.insert(all.end(), mn.begin(), mn.end());
  all.insert(all.end(), ml.begin(), ml.end());
  all.insert(all.end(), me.begin(), me.end());
  all.insert(all.end(), ms.begin(), ms.end());
  for (int f = 0; f < 2; f++) all.insert(all.end(), mi[f].begin(), mi[f].end());
  all.insert(all.end(), mc.begin(), mc.end());
  HIP_TRY(hipMemcpy(b->maps, all.data(), sizeof(int4) * total, hipMemcpyHostToDevice));
  for (int f = 0; f < 2; f++) {
    for (auto& p : b->P) p.fused = f;
    HIP_TRY(hipMemcpy(b->dP + (size_t)f * n, b->P.data(), sizeof(amca::DevParams) * n,
                      hipMemcpyHostToDevice));
    amca::BatchLaunch& L = b->L[f];
    L.P = b->dP + (size_t)f * n;
    L.B = b->dB;
    L.fused = f;
    L.map_nuc = b->maps;
    L.map_list = L.map_nuc + mn.size();
    L.map_emit = L.map_list + ml.size();
    L.map_one = L.map_emit + me.size();
    L.map_ids = L.map_one + ms.size() + (size_t)f * mi[0].size();
    L.map_cmp = L.map_one + ms.size() + 2 * mi[0].size();
    L.n_nuc = (int)mn.size();
    L.n_list = (int)ml.size();
    L.n_emit = (int)me.size();
    L.n_one = (int)ms.size();
    L.n_ids = (int)mi[f].size();
    L.n_cmp = (int)mc.size();
  }
  b->drop_graph();
  return AMCA_OK;
}

// The graph of the batch's form; both are of the schedule's steps_per_graph.
amca_status batch_capture(amca_batch* b) {
  const int steps = b->sched.steps_per_graph, f = b->form;
  if (b->graph_steps != steps) b->drop_graph();
  if (b->exec[f]) return AMCA_OK;
  HIP_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  hipError_t e = hipSuccess;
  for (int q = 0; q < steps && e == hipSuccess; q++) e = amca::launch_batch_step(b->L[f], b->stream);
  if (e == hipSuccess)
    e = amca::launch_batch_status(b->L[f], (int)b->doms.size(), b->status, b->stream);
  hipGraph_t g = nullptr;
  const hipError_t e2 = hipStreamEndCapture(b->stream, &g);
  if (e != hipSuccess || e2 != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    return fail(AMCA_ERR_HIP, std::string("graph capture: ") +
                                  hipGetErrorString(e != hipSuccess ? e : e2));
  }
  if (b->graph[f]) (void)hipGraphDestroy(b->graph[f]);
  b->graph[f] = g;
  b->graph_steps = steps;
  HIP_TRY(hipGraphInstantiate(&b->exec[f], g, nullptr, nullptr, 0));
  return AMCA_OK;
}

// Replays the graph until every domain has finished or `max_graphs` replays
// ran; returns the number of finished domains and the elapsed time.  Each
// replay ends with a status kernel whose output is copied to a pinned slot;
// replay r + 1 is queued before the host reads replay r's slot, so the GPU
// does not wait for the host's check.  A replay queued after every domain
// finished runs steps that all skip.  With `remap`, once max(4, n/8) more
// domains have finished the maps are rebuilt over the domains still running,
// so that the budgets of the list kernels go to them alone (a finished
// domain's kernels return at once, so leaving it out changes no result), and the
// step form of the next replay follows the walk of the last ones.
amca_status batch_replay(amca_batch* b, long long max_graphs, int* finished, double* ms,
                         long long* replays, bool remap) {
  const int n = (int)b->doms.size();
  struct Events {  // destroyed on every return
    hipEvent_t e0 = nullptr, e1 = nullptr;
    ~Events() {
      if (e0) (void)hipEventDestroy(e0);
      if (e1) (void)hipEventDestroy(e1);
    }
  } ev;
  HIP_TRY(hipEventCreate(&ev.e0));
  HIP_TRY(hipEventCreate(&ev.e1));
  auto queue = [&](long long r) -> amca_status {
    const amca::BatchLaunch& L = b->L[b->form];
    if (b->use_graph) {
      AMCA_TRY(batch_capture(b));
      HIP_TRY(hipGraphLaunch(b->exec[b->form], b->stream));
    } else {
      for (int q = 0; q < b->sched.steps_per_graph; q++)
        HIP_TRY(amca::launch_batch_step(L, b->stream));
      HIP_TRY(amca::launch_batch_status(L, n, b->status, b->stream));
    }
    HIP_TRY(hipMemcpyAsync(b->hstatus + (r & 1) * n, b->status, sizeof(int4) * n,
                           hipMemcpyDeviceToHost, b->stream));
    HIP_TRY(hipEventRecord(b->hready[r & 1], b->stream));
    return AMCA_OK;
  };
  // the form by the walk of the steps since the last look (every step leaves the same
  // state in either); the autotuner's trials keep theirs
  auto look = [&](const int4* st, long long steps) {
    b->walk_steps += steps;
    if (b->walk_steps < kFormSteps) return;
    long long walk = 0;
    for (int i = 0; i < n; i++) {
      walk += (st[i].w - b->walk0[i]) & 0x7fffffff;
      b->walk0[i] = st[i].w;
    }
    const bool light = walk <= kWalkBatch * b->walk_steps;
    b->walk_steps = 0;
    if (!light) b->burst = false;  // it has begun, and its walk decides from here on
    if (remap) b->form = b->may_fuse && light && !b->burst ? 1 : 0;
  };
  if (b->use_graph) AMCA_TRY(batch_capture(b));
  HIP_TRY(hipEventRecord(ev.e0, b->stream));
  long long r = 0, queued = 0;
  int fin = 0;
  if (max_graphs != 0) {
    AMCA_TRY(queue(0));
    queued = 1;
  }
  while (r < queued) {
    if (max_graphs < 0 || queued < max_graphs) {
      AMCA_TRY(queue(queued));
      queued++;
    }
    HIP_TRY(hipEventSynchronize(b->hready[r & 1]));
    const int4* st = b->hstatus + (r & 1) * n;
    r++;
    fin = 0;
    for (int i = 0; i < n; i++) {
      if (st[i].y) {
        (void)hipStreamSynchronize(b->stream);
        return fail(AMCA_ERR_CAPACITY, "orientation table exhausted in domain " + std::to_string(i));
      }
      fin += st[i].x;
    }
    if (fin == n) break;
    look(st, b->sched.steps_per_graph);
    if (remap && fin - b->mapped_finished >= std::max(4, n / 8)) {
      // rebuild the maps over the running domains: wait for the queued replay,
      // take the finished set from its status, and capture a new graph
      HIP_TRY(hipStreamSynchronize(b->stream));
      const int4* last = b->hstatus + ((queued - 1) & 1) * n;
      fin = 0;
      for (int i = 0; i < n; i++) {
        if (last[i].y)
          return fail(AMCA_ERR_CAPACITY, "orientation table exhausted in domain " + std::to_string(i));
        fin += last[i].x;
        b->active[i] = last[i].x ? 0 : 1;
      }
      if (queued > r) look(last, b->sched.steps_per_graph * (queued - r));
      r = queued;
      if (fin == n) break;
      b->mapped_finished = fin;
      b->burst = false;
      AMCA_TRY(batch_apply_schedule(b));
      if (max_graphs < 0 || queued < max_graphs) {
        AMCA_TRY(queue(queued));
        queued++;
      }
    }
  }
  HIP_TRY(hipEventRecord(ev.e1, b->stream));
  HIP_TRY(hipEventSynchronize(ev.e1));
  float t = 0.f;
  HIP_TRY(hipEventElapsedTime(&t, ev.e0, ev.e1));
  r = queued;
  if (finished) *finished = fin;
  if (ms) *ms = t;
  if (replays) *replays = r;
  return AMCA_OK;
}

}  // namespace

extern "C" {

amca_status amca_batch_create(amca_domain* const* doms, int32_t n, amca_batch** out) {
  if (!doms || n < 1 || !out) return fail(AMCA_ERR_INVALID, "need at least one domain");
  *out = nullptr;
  auto* b = new amca_batch();
  bool many_sites = false;
  for (int i = 0; i < n; i++) {
    if (!doms[i]) {
      delete b;
      return fail(AMCA_ERR_INVALID, "null domain in batch");
    }
    if (doms[i]->timing) {
      delete b;
      return fail(AMCA_ERR_INVALID, "disable per-kernel timing before batching a domain");
    }
    amca::DevCounters c;
    amca_status rows = read_counters(doms[i], &c);
    if (rows == AMCA_OK) rows = check_rows(doms[i], c);
    if (rows != AMCA_OK) {
      delete b;
      return rows;
    }
    b->doms.push_back(doms[i]);
    b->walk0.push_back((int)(c.w1_walk & 0x7fffffffll));
    choose_form(doms[i], c);
    many_sites |= doms[i]->many_sites;
  }
  amca_status st = AMCA_OK;
  do {
    if (hipGetDevice(&b->device) != hipSuccess) { st = fail(AMCA_ERR_HIP, "hipGetDevice"); break; }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, b->device) == hipSuccess && prop.multiProcessorCount > 0)
      b->cus = prop.multiProcessorCount;
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
      st = fail(AMCA_ERR_HIP, "stream creation failed");
      break;
    }
    std::vector<amca::DevParams>& P = b->P;
    P.resize(n);
    std::vector<amca::DevBuffers> B(n);
    for (int i = 0; i < n; i++) {
      // every domain's own queued work must be done before the batch stream takes over
      if (hipStreamSynchronize(b->doms[i]->stream) != hipSuccess) { st = fail(AMCA_ERR_HIP, "sync"); break; }
      P[i] = b->doms[i]->P;
      B[i] = b->doms[i]->B;
      b->may_fuse = (i == 0 || b->may_fuse) && b->doms[i]->may_fuse;
    }
    if (st != AMCA_OK) break;
    // one launch sequence for the batch: the short one if every domain may take it,
    // as long as their sites and walks allow (batch_replay)
    b->burst = many_sites;
    b->form = b->may_fuse && !b->burst ? 1 : 0;
    if (hipMalloc(&b->dP, sizeof(amca::DevParams) * 2 * n) != hipSuccess ||
        hipMalloc(&b->dB, sizeof(amca::DevBuffers) * n) != hipSuccess ||
        hipMalloc(&b->status, sizeof(int4) * n) != hipSuccess ||
        hipHostMalloc(&b->hstatus, sizeof(int4) * 2 * n) != hipSuccess ||
        hipEventCreateWithFlags(&b->hready[0], hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&b->hready[1], hipEventDisableTiming) != hipSuccess) {
      st = fail(AMCA_ERR_HIP, "batch allocation failed");
      break;
    }
    if (hipMemcpy(b->dB, B.data(), sizeof(amca::DevBuffers) * n, hipMemcpyHostToDevice) != hipSuccess) {
      st = fail(AMCA_ERR_HIP, "batch upload failed");
      break;
    }
    b->sched.list_blocks = 16 * b->cus;
    b->sched.emit_blocks = 16 * b->cus;
    b->sched.min_blocks = 1;
    b->sched.interleave = 0;
    b->sched.steps_per_graph = 16;
    b->active.assign(n, 1);
    int g = 1;
    if (amca::env_int("AMCA_BATCH_GRAPHS", 0, 1, &g) < 0) {
      st = fail(AMCA_ERR_INVALID, "AMCA_BATCH_GRAPHS must be 0 or 1");
      break;
    }
    b->use_graph = g != 0;
    st = batch_apply_schedule(b);
  } while (0);
  if (st != AMCA_OK) {
    delete b;
    return st;
  }
  *out = b;
  return AMCA_OK;
}

amca_status amca_batch_destroy(amca_batch* b) {
  delete b;
  return AMCA_OK;
}

amca_status amca_batch_set_schedule(amca_batch* b, const amca_batch_schedule* s) {
  if (!b || !s || s->list_blocks < 1 || s->emit_blocks < 1 || s->min_blocks < 1 ||
      s->min_blocks > amca::kMaxBlocks || s->steps_per_graph < 1 || s->steps_per_graph > 4096)
    return fail(AMCA_ERR_INVALID, "bad schedule (budgets >= 1, min_blocks in [1, 4096], "
                                  "steps_per_graph in [1, 4096])");
  HIP_TRY(hipStreamSynchronize(b->stream));
  b->sched = *s;
  return batch_apply_schedule(b);
}

amca_status amca_batch_get_schedule(amca_batch* b, amca_batch_schedule* s) {
  if (!b || !s) return fail(AMCA_ERR_INVALID, "null argument");
  *s = b->sched;
  return AMCA_OK;
}

amca_status amca_batch_run(amca_batch* b, int64_t max_graphs, int32_t* n_finished, double* ms,
                           int64_t* replays) {
  if (!b) return fail(AMCA_ERR_INVALID, "null batch");
  int fin = 0;
  double t = 0.0;
  long long r = 0;
  AMCA_TRY(batch_replay(b, max_graphs, &fin, &t, &r, true));
  if (n_finished) *n_finished = fin;
  if (ms) *ms = t;
  if (replays) *replays = r;
  return AMCA_OK;
}

// The autotuner runs the real batch: each candidate schedule takes
// `trial_graphs` replays of a short graph (kTrialSteps steps, or the
// schedule's own length if shorter) in turn, for `rounds` rounds, and the
// schedule with the least mean time per step wins.  The batch's work per step
// drifts while the trials run, so odd rounds visit the candidates in reverse
// order, which cancels a steady drift over each pair of rounds.  Stage 1 tries
// one block budget for all list kernels (2, 16, 64 blocks per CU: 4 would stand for
// the same blocks as 16) in both block orders; stage 2 sizes the claim grid and the
// resolve / emit grid apart, a factor 4 up and down from the stage-1 choice, where
// that is another number of blocks (the short step has one grid for both, of
// emit_blocks).  Schedules do not change results, so the trial steps are ordinary
// steps of the run.
amca_status amca_batch_autotune(amca_batch* b, int32_t trial_graphs, int32_t rounds,
                                amca_batch_schedule* chosen) {
  if (!b || trial_graphs < 1 || rounds < 1) return fail(AMCA_ERR_INVALID, "bad arguments");
  constexpr int kTrialSteps = 4;
  const int run_steps = b->sched.steps_per_graph;
  const int trial_steps = std::min(run_steps, kTrialSteps);
  // the schedule as it was, restored if a trial fails
  const amca_batch_schedule before = b->sched;
  struct Restore {
    amca_batch* b;
    const amca_batch_schedule* s;
    bool armed = true;
    ~Restore() {
      if (!armed) return;
      (void)hipStreamSynchronize(b->stream);
      b->sched = *s;
      (void)batch_apply_schedule(b);
    }
  } restore{b, &before};
  const int emit_cap = (int)amca::kMaxBlocks * 8;
  auto make = [&](int list_budget, int emit_budget, int inter) {
    amca_batch_schedule s = b->sched;
    s.list_blocks = list_budget * b->cus;
    s.emit_blocks = std::min(emit_budget * b->cus, emit_cap);
    s.min_blocks = 1;
    s.interleave = inter;
    return s;
  };
  bool all_done = false;
  // mean ms per step of each candidate over `rounds` passes; the best index
  auto pick = [&](const std::vector<amca_batch_schedule>& cand, size_t* best) -> amca_status {
    std::vector<double> tot(cand.size(), 0.0);
    std::vector<int> runs(cand.size(), 0);
    for (int r = 0; r < rounds && !all_done; r++)
      for (size_t u = 0; u < cand.size() && !all_done; u++) {
        const size_t c = (r & 1) ? cand.size() - 1 - u : u;
        b->sched.list_blocks = cand[c].list_blocks;
        b->sched.emit_blocks = cand[c].emit_blocks;
        b->sched.min_blocks = cand[c].min_blocks;
        b->sched.interleave = cand[c].interleave;
        b->sched.steps_per_graph = trial_steps;
        AMCA_TRY(batch_apply_schedule(b));
        int fin = 0;
        double ms = 0.0;
        long long rep = 0;
        AMCA_TRY(batch_replay(b, trial_graphs, &fin, &ms, &rep, false));
        tot[c] += ms / (double)(std::max(1LL, rep) * trial_steps);
        runs[c]++;
        if (fin == (int)b->doms.size()) all_done = true;
      }
    size_t k = 0;
    for (size_t c = 1; c < cand.size(); c++)
      if (runs[c] > 0 && (runs[k] == 0 || tot[c] / runs[c] < tot[k] / runs[k])) k = c;
    *best = k;
    return AMCA_OK;
  };
  // stage 1: one budget for every list kernel, both block orders
  std::vector<amca_batch_schedule> cand;
  for (int budget : {2, 16, 64})
    for (int inter : {0, 1}) cand.push_back(make(budget, budget, inter));
  size_t best = 0;
  AMCA_TRY(pick(cand, &best));
  amca_batch_schedule win = cand[best];
  // stage 2: the claim kernel's grid and the resolve / emit grid apart, a
  // factor 4 either way from the stage-1 choice
  if (!all_done) {
    const int lb = win.list_blocks / b->cus, eb = std::max(1, win.emit_blocks / b->cus);
    std::vector<amca_batch_schedule> c2 = {win};
    for (int f : {4, -4}) {
      const int l2 = f > 0 ? lb * f : std::max(1, lb / -f);
      const int e2 = f > 0 ? eb * f : std::max(1, eb / -f);
      const auto other = [&](int p, int q) {
        return budget_blocks(b, p * b->cus) != budget_blocks(b, q * b->cus);
      };
      if (!b->form && other(l2, lb)) c2.push_back(make(l2, eb, win.interleave));
      if (other(e2, eb)) c2.push_back(make(lb, e2, win.interleave));
    }
    AMCA_TRY(pick(c2, &best));
    win = c2[best];
  }
  b->sched.list_blocks = win.list_blocks;
  b->sched.emit_blocks = win.emit_blocks;
  b->sched.min_blocks = win.min_blocks;
  b->sched.interleave = win.interleave;
  b->sched.steps_per_graph = run_steps;
  restore.armed = false;
  AMCA_TRY(batch_apply_schedule(b));
  if (chosen) *chosen = b->sched;
  return AMCA_OK;
}

}  // extern "C"
