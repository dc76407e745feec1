// C ABI of a coupled CA-FE (remelting) domain (include/amca3d.h, amca_remelt_*).
//
// The reference's CafeSolver owns a FiniteElementManager that streams text
// frames and a MapVoxelManager that interpolates them per cell every step
// (CafeSolver.cpp:159-219).  Here the FE frames, the voxel map and the whole CA
// state are resident in HBM; the host only maps voxels once, refills the
// orientation rows it draws from the rand() stream, and reads counters back
// between batches of steps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/amca3d.h"
#include "host/fe_text.h"
#include "host/generators.h"
#include "host/sites.h"
#include "host/voxel_map.h"
#include "env.h"
#include "libm_pow.h"
#include "plain_step.h"
#include "remelt_step.h"
#include "surrogate.h"

namespace {

thread_local std::string g_rm_error;

amca_status rm_fail(amca_status st, const std::string& msg) {
  g_rm_error = msg;
  return st;
}

#define RM_HIP(expr)                                                                      \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess)                                                                 \
      return rm_fail(AMCA_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));    \
  } while (0)

#define RM_TRY(expr)              \
  do {                            \
    amca_status s_ = (expr);      \
    if (s_ != AMCA_OK) return s_; \
  } while (0)

}  // namespace

struct amca_remelt {
  hipStream_t stream = nullptr;
  amca_remelt_desc desc{};
  amca::RmParams P{};
  amca::RmBuffers B{};
  std::vector<void*> allocs;
  bool fe_ready = false, state_ready = false;
  int site_blocks = 1;
  int rows_pushed = 0;
  amca_orientation_source source = nullptr;
  void* source_user = nullptr;
  std::unique_ptr<amca_host::GlibcRand> rng;  // the rand() stream after amca_remelt_draw_sites
  std::vector<int32_t> site_cells;            // nucleation sites as last set
  std::vector<double> site_dts;
  std::vector<double> euler;                  // Euler angles of every row, 3 per row
  size_t grain_cap = 0;  // records genv/gco can hold
  std::vector<double> node_xyz;
  // per-kernel event timing (off by default)
  bool timing = false;
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<int, size_t>> ev_pending;
  size_t ev_used = 0;
  double kernel_ms[amca::kRmKernels] = {};
  int64_t kernel_launches[amca::kRmKernels] = {};

  template <class T>
  amca_status alloc(T** p, size_t count) {
    void* q = nullptr;
    const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
    hipError_t e = hipMalloc(&q, bytes);
    if (e != hipSuccess)
      return rm_fail(AMCA_ERR_HIP, "hipMalloc(" + std::to_string(bytes) + "): " + hipGetErrorString(e));
    allocs.push_back(q);
    *p = static_cast<T*>(q);
    return AMCA_OK;
  }
  void release(void* p) {
    if (!p) return;
    for (auto& a : allocs)
      if (a == p) {
        (void)hipFree(a);
        a = nullptr;
      }
    allocs.erase(std::remove(allocs.begin(), allocs.end(), nullptr), allocs.end());
  }
  // kGraphSteps steps captured as one HIP graph, valid while the kernels'
  // arguments (parameters, buffers, site blocks) are the ones captured
  int graph_steps = 8;  // 0: every kernel launched on the stream
  int row_reserve = 4096;  // orientation rows drawn ahead of the rows in use
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  std::vector<unsigned char> graph_sig;

  void drop_graph() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph) (void)hipGraphDestroy(graph);
    graph_exec = nullptr;
    graph = nullptr;
    graph_sig.clear();
  }
  std::vector<unsigned char> launch_sig() const {
    std::vector<unsigned char> v(sizeof(P) + sizeof(B) + sizeof(int));
    std::memcpy(v.data(), &P, sizeof(P));
    std::memcpy(v.data() + sizeof(P), &B, sizeof(B));
    std::memcpy(v.data() + sizeof(P) + sizeof(B), &site_blocks, sizeof(int));
    return v;
  }
  ~amca_remelt() {
    if (stream) (void)hipStreamSynchronize(stream);
    drop_graph();
    for (hipEvent_t e : ev_pool) (void)hipEventDestroy(e);
    for (void* p : allocs) (void)hipFree(p);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

amca_status rm_counters(amca_remelt* d, amca::RmCounters* c) {
  RM_HIP(hipMemcpyAsync(c, d->B.ctr, sizeof(*c), hipMemcpyDeviceToHost, d->stream));
  RM_HIP(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

amca_status rm_put_counters(amca_remelt* d, const amca::RmCounters& c) {
  RM_HIP(hipMemcpyAsync(d->B.ctr, &c, sizeof(c), hipMemcpyHostToDevice, d->stream));
  RM_HIP(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

// the next step runs over the whole grid and restarts the box bookkeeping
void rm_restart_box(amca::RmCounters& c) {
  for (int q = 0; q < 2; q++) {
    for (int r = 0; r < 3; r++)
      for (int a = 0; a < 3; a++) {
        c.acc[q][r].lo[a] = INT_MAX;
        c.acc[q][r].hi[a] = INT_MIN;
      }
  }
  c.force_full = 1;
}

void rm_fill(const amca_remelt* d, const amca::RmCounters& c, amca_remelt_counters* o) {
  if (!o) return;
  o->step = c.step;
  o->time = c.t;
  o->time_fe = c.time_fe;
  o->dt = c.dt;
  o->max_dt = c.max_dt;
  o->n_grains = c.n_grains;
  o->n_orient = c.n_orient;
  o->frames_exhausted = c.exhausted;
  o->done = (c.exhausted || !(c.tcafe < d->desc.final_time)) ? 1 : 0;
}

amca_status push_rows(amca_remelt* d, int n, const double* l2g9) {
  if (d->rows_pushed + n > d->P.orient_cap)
    return rm_fail(AMCA_ERR_CAPACITY, "orientation table capacity exceeded");
  if (n > 0)
    RM_HIP(hipMemcpyAsync(d->B.l2g + 9 * (size_t)d->rows_pushed, l2g9, sizeof(double) * 9 * n,
                          hipMemcpyHostToDevice, d->stream));
  d->rows_pushed += n;
  // the device runs a step only when its armed sites fit in the pushed rows
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  c.rows_avail = d->rows_pushed;
  RM_TRY(rm_put_counters(d, c));
  RM_HIP(hipStreamSynchronize(d->stream));
  return AMCA_OK;
}

// make sure `need` rows exist, pulling from the orientation source
amca_status ensure_rows(amca_remelt* d, long long need) {
  if (need <= d->rows_pushed) return AMCA_OK;
  if (!d->source && !d->rng)
    return rm_fail(AMCA_ERR_CAPACITY, "orientation rows exhausted and no orientation source set");
  need = std::min<long long>(need, d->P.orient_cap);
  const int n = (int)(need - d->rows_pushed);
  if (n <= 0) return AMCA_OK;
  std::vector<double> eu(3 * (size_t)n), r(9 * (size_t)n);
  if (d->rng) {
    for (int q = 0; q < n; q++) {
      amca_host::random_orientation(*d->rng, &eu[3 * (size_t)q]);
      amca_host::rotation_from_euler(&eu[3 * (size_t)q], &r[9 * (size_t)q]);
    }
  } else if (d->source(d->source_user, n, eu.data(), r.data()) != 0) {
    return rm_fail(AMCA_ERR_INVALID, "orientation source failed");
  }
  d->euler.insert(d->euler.end(), eu.begin(), eu.end());
  return push_rows(d, n, r.data());
}

amca_status rm_resolve_events(amca_remelt* d) {
  RM_HIP(hipStreamSynchronize(d->stream));
  for (auto& p : d->ev_pending) {
    float ms = 0.f;
    RM_HIP(hipEventElapsedTime(&ms, d->ev_pool[p.second], d->ev_pool[p.second + 1]));
    d->kernel_ms[p.first] += ms;
    d->kernel_launches[p.first] += 1;
  }
  d->ev_pending.clear();
  d->ev_used = 0;
  return AMCA_OK;
}

// k steps without per-kernel timing: whole graphs of graph_steps steps, then
// single steps for the rest
amca_status rm_enqueue_steps(amca_remelt* d, long long k) {
  const int G = d->graph_steps > 0 ? d->graph_steps : 1;
  if (d->graph_steps > 0 && k >= G) {
    std::vector<unsigned char> sig = d->launch_sig();
    if (!d->graph_exec || sig != d->graph_sig) {
      d->drop_graph();
      RM_HIP(hipStreamBeginCapture(d->stream, hipStreamCaptureModeThreadLocal));
      hipError_t e = hipSuccess;
      for (int q = 0; q < G && e == hipSuccess; q++)
        e = amca::rm_launch_step(d->P, d->B, d->site_blocks, d->stream);
      hipGraph_t g = nullptr;
      const hipError_t e2 = hipStreamEndCapture(d->stream, &g);
      if (e != hipSuccess || e2 != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return rm_fail(AMCA_ERR_HIP, std::string("graph capture: ") +
                                         hipGetErrorString(e != hipSuccess ? e : e2));
      }
      d->graph = g;
      RM_HIP(hipGraphInstantiate(&d->graph_exec, g, nullptr, nullptr, 0));
      d->graph_sig = std::move(sig);
    }
    for (long long q = 0; q < k / G; q++) RM_HIP(hipGraphLaunch(d->graph_exec, d->stream));
  }
  const long long rest = d->graph_steps > 0 ? k % G : k;
  for (long long q = 0; q < rest; q++)
    RM_HIP(amca::rm_launch_step(d->P, d->B, d->site_blocks, d->stream));
  return AMCA_OK;
}

// one step; with timing on, each kernel sits between two events on the stream
amca_status rm_enqueue_step(amca_remelt* d) {
  if (!d->timing) {
    RM_HIP(amca::rm_launch_step(d->P, d->B, d->site_blocks, d->stream));
    return AMCA_OK;
  }
  for (int q = 0; q < amca::kRmKernels; q++) {
    if (d->ev_used + 2 > d->ev_pool.size()) {
      if (d->ev_pool.size() >= (1u << 16)) RM_TRY(rm_resolve_events(d));
      while (d->ev_used + 2 > d->ev_pool.size()) {
        hipEvent_t e;
        RM_HIP(hipEventCreate(&e));
        d->ev_pool.push_back(e);
      }
    }
    const size_t i = d->ev_used;
    d->ev_used += 2;
    RM_HIP(hipEventRecord(d->ev_pool[i], d->stream));
    RM_HIP(amca::rm_launch_kernel(q, d->P, d->B, d->site_blocks, d->stream));
    RM_HIP(hipEventRecord(d->ev_pool[i + 1], d->stream));
    d->ev_pending.emplace_back(q, i);
  }
  return AMCA_OK;
}

}  // namespace

extern "C" {

const char* amca_remelt_last_error(void) { return g_rm_error.c_str(); }

amca_status amca_remelt_enable_timing(amca_remelt* d, int32_t on) {
  if (!d) return rm_fail(AMCA_ERR_INVALID, "null domain");
  RM_TRY(rm_resolve_events(d));
  d->timing = on != 0;
  for (int q = 0; q < amca::kRmKernels; q++) {
    d->kernel_ms[q] = 0.0;
    d->kernel_launches[q] = 0;
  }
  return AMCA_OK;
}

int32_t amca_remelt_kernel_count(void) { return amca::kRmKernels; }

const char* amca_remelt_kernel_name(int32_t i) {
  return (i >= 0 && i < amca::kRmKernels) ? amca::kRmKernelNames[i] : "";
}

amca_status amca_remelt_kernel_times(amca_remelt* d, double* ms, int64_t* launches) {
  if (!d || !ms || !launches) return rm_fail(AMCA_ERR_INVALID, "null argument");
  RM_TRY(rm_resolve_events(d));
  for (int q = 0; q < amca::kRmKernels; q++) {
    ms[q] = d->kernel_ms[q];
    launches[q] = d->kernel_launches[q];
  }
  return AMCA_OK;
}

amca_status amca_remelt_create(const amca_remelt_desc* desc, int32_t orient_capacity,
                               amca_remelt** out) {
  if (!desc || !out) return rm_fail(AMCA_ERR_INVALID, "null argument");
  *out = nullptr;
  if (desc->nx < 1 || desc->ny < 1 || desc->nz < 1 || !(desc->h > 0))
    return rm_fail(AMCA_ERR_INVALID, "bad grid");
  for (double b : {desc->b1, desc->b2, desc->b3})
    if (!amca_libm::pow_exponent_supported(b))
      return rm_fail(AMCA_ERR_INVALID,
                     "kinetics exponents b1, b2, b3 must be 0 or of magnitude in [2^-65, 2^63)");
  const long long nxG = desc->nx + 2LL, nyG = desc->ny + 2LL, nzG = desc->nz + 2LL;
  const long long NG = nxG * nyG * nzG;
  if (NG > (long long)INT_MAX) return rm_fail(AMCA_ERR_INVALID, "grid exceeds int32 cell indices");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return rm_fail(AMCA_ERR_NO_DEVICE, "no HIP device visible");
  auto* d = new amca_remelt();
  d->desc = *desc;
  if (amca::env_int("AMCA_REMELT_GRAPH_STEPS", 0, 1024, &d->graph_steps) < 0) {
    delete d;
    return rm_fail(AMCA_ERR_INVALID, "AMCA_REMELT_GRAPH_STEPS must be an integer in [0, 1024]");
  }
  if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) {
    delete d;
    return rm_fail(AMCA_ERR_HIP, "stream creation failed");
  }
  amca::RmParams& P = d->P;
  P.nx = desc->nx; P.ny = desc->ny; P.nz = desc->nz;
  P.nxG = (int)nxG; P.nyG = (int)nyG; P.nzG = (int)nzG;
  P.nxyG = (int)(nxG * nyG);
  P.NG = (int)NG;
  P.N = (long long)desc->nx * desc->ny * desc->nz;
  P.h = desc->h; P.x0 = desc->x0; P.y0 = desc->y0; P.z0 = desc->z0;
  P.Tm = desc->Tm; P.Ts = desc->Ts; P.Tmin_nuc = desc->Tmin_nuc;
  P.a1 = desc->a1; P.a2 = desc->a2; P.a3 = desc->a3;
  P.b1 = desc->b1; P.b2 = desc->b2; P.b3 = desc->b3;
  P.trunc = desc->trunc;
  P.tsf = desc->time_step_factor;
  P.sqrt2f = (double)sqrtf(2.0f);
  P.cutoff = desc->cutoff_factor * desc->h;  // cellGrainLegnthCutoff_ *= h_
  P.final_time = desc->final_time;
  P.void_temp = desc->void_temperature;
  P.orient_cap = orient_capacity;
  // A part takes the cells of every kRmParts-th of n blocks, each walking its 256
  // threads through up to NG cells in strides of 256 n: at most
  // 256 (NG / (256 n) + 1) (n / kRmParts + 1) cells, with n at most 16384 and at least
  // 512 or NG / 256.
  P.flist_cap = (int)std::min<long long>(
      INT_MAX, NG / amca::kRmParts + NG / 512 + 256 * (16384 / amca::kRmParts + 3));
  if (P.flist_cap > P.N) P.flist_cap = (int)P.N;  // one entry per interior cell
  P.window = 1;
  P.hot_margin = 1.0;
  P.sur_hot[0] = 1;
  P.sur_hot[1] = 0;
  {
    int s = 0;
    for (int dk = -1; dk <= 1; dk++)
      for (int dj = -1; dj <= 1; dj++)
        for (int di = -1; di <= 1; di++) {
          if (!dk && !dj && !di) continue;
          P.off[s++] = dk * P.nxyG + dj * P.nxG + di;
        }
  }
  amca::RmBuffers& B = d->B;
  const size_t ng = (size_t)NG, nc = (size_t)P.N + 1;
  amca_status st = AMCA_OK;
  auto A = [&](auto** p, size_t n) {
    if (st == AMCA_OK) st = d->alloc(p, n);
  };
  A(&B.gid, ng);
  A(&B.oid, ng);
  A(&B.T, ng);
  A(&B.cooling, ng);
  A(&B.melted, ng);
  A(&B.flag, ng);
  A(&B.tag, ng);
  A(&B.par, 3 * ng);
  A(&B.claim, ng);
  A(&B.msk, ng);
  A(&B.flist, (size_t)amca::kRmParts * P.flist_cap);
  A(&B.clist, (size_t)P.N);
  A(&B.genv, nc);
  A(&B.gco, nc);
  d->grain_cap = nc;
  A(&B.l2g, 9 * (size_t)std::max(orient_capacity, 1));
  A(&B.rowcnt, (size_t)P.nx * P.ny);
  A(&B.rowoff, (size_t)P.nx * P.ny);
  A(&B.lb_flag, (size_t)amca::kMaxBlocks);
  A(&B.lb_agg, (size_t)amca::kMaxBlocks);
  A(&B.lb_pref, (size_t)amca::kMaxBlocks);
  A(&B.ctr, 1);
  A(&B.blk_box, 6 * 16384);
  A(&B.site_cell, 1);
  A(&B.site_dt, 1);
  if (st != AMCA_OK) {
    delete d;
    return st;
  }
  B.log = nullptr;
  B.frames = nullptr;
  B.frame_time = nullptr;
  B.theta = nullptr;
  // every cell liquid without a grain until a state is loaded
  (void)hipMemsetAsync(B.gid, 0xff, sizeof(int) * ng, d->stream);
  (void)hipMemsetAsync(B.oid, 0xff, sizeof(int) * ng, d->stream);
  (void)hipMemsetAsync(B.melted, desc->initial_melted ? 1 : 0, ng, d->stream);
  (void)hipMemsetAsync(B.lb_flag, 0, sizeof(unsigned) * amca::kMaxBlocks, d->stream);
  (void)hipMemsetAsync(B.rowcnt, 0, sizeof(int) * (size_t)P.nx * P.ny, d->stream);
  amca::RmCounters c{};
  for (int q = 0; q < 64; q++) c.min_t_keys[q] = ~0ull;
  c.last_step = -1;
  for (int q = 0; q < 2; q++) {
    c.box[q].lo[0] = c.box[q].lo[1] = c.box[q].lo[2] = 0;
    c.box[q].hi[0] = P.nxG - 1;
    c.box[q].hi[1] = P.nyG - 1;
    c.box[q].hi[2] = P.nzG - 1;
  }
  rm_restart_box(c);
  // the velocity at Ts + 0.01 K, through the step's own kinetics code
  P.vts = 0.0;
  double* vts_dev = nullptr;
  const bool ok = hipMalloc(&vts_dev, sizeof(double)) == hipSuccess &&
                  hipMemcpyAsync(B.ctr, &c, sizeof(c), hipMemcpyHostToDevice, d->stream) == hipSuccess &&
                  amca::rm_launch_init(P, B, d->stream) == hipSuccess &&
                  amca::rm_launch_vts(P, vts_dev, d->stream) == hipSuccess &&
                  hipMemcpyAsync(&P.vts, vts_dev, sizeof(double), hipMemcpyDeviceToHost,
                                 d->stream) == hipSuccess &&
                  hipStreamSynchronize(d->stream) == hipSuccess;
  if (vts_dev) (void)hipFree(vts_dev);
  if (!ok) {
    delete d;
    return rm_fail(AMCA_ERR_HIP, "initialisation failed");
  }
  *out = d;
  return AMCA_OK;
}

amca_status amca_remelt_destroy(amca_remelt* d) {
  delete d;
  return AMCA_OK;
}

namespace {

// device memory of one call, freed on every return
struct DeviceTemp {
  void* p = nullptr;
  ~DeviceTemp() {
    if (p) (void)hipFree(p);
  }
  hipError_t get(size_t bytes) { return hipMalloc(&p, std::max<size_t>(bytes, 16)); }
};

// tag_voxels on the device: one thread per CA cell (ghosts included), the
// arithmetic of the host mapper (voxel_math.h), so tags and parametric
// coordinates equal the host's bit for bit; *any is set when a cell has an element
__global__ void k_map_voxels(amca_vox::MeshView M, amca_vox::VoxelGrid G,
                             const int* __restrict__ bin_start, const int* __restrict__ bin_elems,
                             long long NG, double tol, int max_iter, int32_t* __restrict__ tag,
                             double* __restrict__ par, int* any) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  int found = 0;
  for (long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x; v < NG; v += stride) {
    double pc[3];
    const int e = amca_vox::tag_voxel(M, G, bin_start, bin_elems, v, tol, max_iter, pc);
    tag[v] = e;
    for (int q = 0; q < 3; q++) par[3 * v + q] = e >= 0 ? pc[q] : -2.0;
    found |= e >= 0 ? 1 : 0;
  }
  if (__syncthreads_or(found) && threadIdx.x == 0 &&
      !__hip_atomic_load(any, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    __hip_atomic_store(any, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// map_voxels on the device into tag[NG], par[3 NG] (device memory): the plan
// (search box, bins) on the host, the per-cell search in k_map_voxels.  any:
// whether a cell found an element.
amca_status map_voxels_device(const amca_host::FeMesh& mesh, const amca_host::VoxelMapParams& vp,
                              int32_t* tag, double* par, hipStream_t s, bool& any) {
  amca_host::VoxelPlan plan;
  amca_host::plan_voxels(mesh, vp, plan);
  const amca_vox::VoxelGrid& G = plan.grid;
  const long long NG = (long long)G.nxG * G.nyG * G.nzG;
  if (plan.bin_elems.empty()) plan.bin_elems.push_back(0);  // a valid pointer; no bin reads it
  DeviceTemp dxyz, dbs, dbe, dany;
  RM_HIP(dxyz.get(sizeof(double) * mesh.xyz.size()));
  RM_HIP(dbs.get(sizeof(int) * plan.bin_start.size()));
  RM_HIP(dbe.get(sizeof(int) * plan.bin_elems.size()));
  RM_HIP(dany.get(sizeof(int)));
  int found = 0;
  RM_HIP(hipMemcpyAsync(dxyz.p, mesh.xyz.data(), sizeof(double) * mesh.xyz.size(),
                        hipMemcpyHostToDevice, s));
  RM_HIP(hipMemcpyAsync(dbs.p, plan.bin_start.data(), sizeof(int) * plan.bin_start.size(),
                        hipMemcpyHostToDevice, s));
  RM_HIP(hipMemcpyAsync(dbe.p, plan.bin_elems.data(), sizeof(int) * plan.bin_elems.size(),
                        hipMemcpyHostToDevice, s));
  RM_HIP(hipMemcpyAsync(dany.p, &found, sizeof(int), hipMemcpyHostToDevice, s));
  const amca_vox::MeshView mv{static_cast<double*>(dxyz.p), mesh.fnx, mesh.fny, mesh.fnz};
  long long blocks = (NG + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_map_voxels, dim3((unsigned)blocks), dim3(256), 0, s, mv, G,
                     static_cast<int*>(dbs.p), static_cast<int*>(dbe.p), NG, vp.tol, vp.max_iter,
                     tag, par, static_cast<int*>(dany.p));
  RM_HIP(hipGetLastError());
  RM_HIP(hipMemcpyAsync(&found, dany.p, sizeof(int), hipMemcpyDeviceToHost, s));
  RM_HIP(hipStreamSynchronize(s));
  any = found != 0;
  return AMCA_OK;
}

// ---- boxes for the active box (amca_remelt_set_fe) --------------------------
// Per element the box of its cells; per frame the union over the elements with a
// hot node (at or above Tm - hot_margin), and the union over the elements with a
// node whose void state can change between frames.  On the host these loops and
// the copies of the voxel map down and up again were most of the call (72 ms at
// 400 x 160 x 80 cells and 100 frames).

__global__ void k_box_clear(long long n, int* __restrict__ b) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) b[q] = (q % 6) < 3 ? INT_MAX : INT_MIN;
}

__global__ void k_elem_boxes(amca::RmParams P, const int32_t* __restrict__ tag, int* ebox) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < P.NG; c += stride) {
    const int e = tag[c];
    if (e < 0) continue;
    const int k = (int)c / P.nxyG, r = (int)c - k * P.nxyG, j = r / P.nxG, i = r - j * P.nxG;
    int* b = ebox + 6 * (size_t)e;
    const int v[3] = {i, j, k};
    // most cells change nothing: a plain read first (a stale one only costs an atomic)
    for (int a = 0; a < 3; a++) {
      if (v[a] < b[a]) atomicMin(&b[a], v[a]);
      if (v[a] > b[3 + a]) atomicMax(&b[3 + a], v[a]);
    }
  }
}

// a node near the void temperature in some frame may change between void and
// material: the field is void_temp where a frame is at or below it, and is
// compared with void_temp + 1e-5
__global__ void k_void_nodes(const double* __restrict__ frames, int n_frames, int nodes,
                             double void_temp, unsigned char* __restrict__ out) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nodes) return;
  const double nm = void_temp + 0.00001;
  bool maybe = false, always = true;
  for (int f = 0; f < n_frames; f++) {
    const double v = frames[(size_t)f * nodes + n];
    maybe |= !(v > nm + 1e-6);
    always &= v <= void_temp;
  }
  out[n] = maybe && !always ? 1 : 0;
}

// box blockIdx.y: the union of the boxes of the elements with a marked node --
// frame blockIdx.y's nodes at or above `hot`, or with `mark` the marked ones
__global__ void __launch_bounds__(256)
k_union_boxes(amca::RmParams P, const double* __restrict__ frames, double hot,
              const unsigned char* __restrict__ mark, const int* __restrict__ ebox,
              int* __restrict__ out) {
  const int ncx = P.fnx - 1, ncy = P.fny - 1, nxy = P.fnx * P.fny;
  const long long ne = (long long)ncx * ncy * (P.fnz - 1);
  const double* v = frames + (size_t)blockIdx.y * P.nodes;
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
  for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < ne;
       e += (long long)gridDim.x * blockDim.x) {
    const int ei = (int)(e % ncx), ej = (int)((e / ncx) % ncy), ek = (int)(e / ((long long)ncx * ncy));
    const int n0 = nxy * ek + P.fnx * ej + ei;
    const int nid[8] = {n0, n0 + 1, n0 + P.fnx, n0 + P.fnx + 1, n0 + nxy, n0 + nxy + 1,
                        n0 + nxy + P.fnx, n0 + nxy + P.fnx + 1};
    bool any = false;
#pragma unroll
    for (int m = 0; m < 8; m++) any |= mark ? mark[nid[m]] != 0 : v[nid[m]] >= hot;
    if (!any) continue;
    const int* b = ebox + 6 * e;
    for (int a = 0; a < 3; a++) {
      lo[a] = min(lo[a], b[a]);
      hi[a] = max(hi[a], b[3 + a]);
    }
  }
  __shared__ int s_b[6];
  if (threadIdx.x < 6) s_b[threadIdx.x] = threadIdx.x < 3 ? INT_MAX : INT_MIN;
  __syncthreads();
#pragma unroll
  for (int a = 0; a < 3; a++) {
    for (int o = 32; o > 0; o >>= 1) {
      lo[a] = min(lo[a], __shfl_xor(lo[a], o, 64));
      hi[a] = max(hi[a], __shfl_xor(hi[a], o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
      atomicMin(&s_b[a], lo[a]);
      atomicMax(&s_b[3 + a], hi[a]);
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    int* q = out + 6 * (size_t)blockIdx.y + threadIdx.x;
    if (threadIdx.x < 3 && s_b[threadIdx.x] < INT_MAX) atomicMin(q, s_b[threadIdx.x]);
    if (threadIdx.x >= 3 && s_b[threadIdx.x] > INT_MIN) atomicMax(q, s_b[threadIdx.x]);
  }
}

unsigned grid_for(long long n, int cap = 65536) {
  return (unsigned)std::max(1LL, std::min<long long>((n + 255) / 256, cap));
}

}  // namespace

amca_status amca_remelt_set_fe(amca_remelt* d, int32_t fnx, int32_t fny, int32_t fnz,
                               const double* node_xyz, int32_t n_frames, const double* frame_time,
                               const double* frame_theta) {
  if (!d || fnx < 2 || fny < 2 || fnz < 2 || !node_xyz || n_frames < 2 || !frame_time ||
      !frame_theta)
    return rm_fail(AMCA_ERR_INVALID, "FE mesh needs >= 2 nodes per axis and >= 2 frames");
  amca::RmParams& P = d->P;
  amca_host::FeMesh mesh;
  mesh.fnx = fnx;
  mesh.fny = fny;
  mesh.fnz = fnz;
  const size_t nodes = (size_t)fnx * fny * fnz;
  mesh.xyz.assign(node_xyz, node_xyz + 3 * nodes);
  d->node_xyz = mesh.xyz;
  amca_host::VoxelMapParams vp;
  vp.nx = P.nx; vp.ny = P.ny; vp.nz = P.nz;
  vp.h = P.h; vp.x0 = P.x0; vp.y0 = P.y0; vp.z0 = P.z0;
  for (int q = 0; q < 3; q++) vp.bin[q] = d->desc.bin[q] > 0 ? d->desc.bin[q] : 10;
  vp.tol = d->desc.tolerance;
  vp.max_iter = d->desc.max_iterations;
  bool any = false;
  // a new map next to the one in use, which stays if the mesh holds no cell
  int32_t* tag = nullptr;
  double* par = nullptr;
  RM_TRY(d->alloc(&tag, (size_t)P.NG));
  amca_status st = d->alloc(&par, 3 * (size_t)P.NG);
  if (st == AMCA_OK) st = map_voxels_device(mesh, vp, tag, par, d->stream, any);
  if (st == AMCA_OK && !any) st = rm_fail(AMCA_ERR_INVALID, "no CA cell lies in the FE mesh");
  if (st != AMCA_OK) {
    d->release(tag);
    d->release(par);
    return st;
  }
  d->release(d->B.tag);
  d->release(d->B.par);
  d->B.tag = tag;
  d->B.par = par;
  P.fnx = fnx;
  P.fny = fny;
  P.fnz = fnz;
  P.nodes = (int)nodes;
  P.ncx = fnx - 1;
  P.ncy = fny - 1;
  P.n_frames = n_frames;
  d->release((void*)d->B.frames);
  d->release((void*)d->B.frame_time);
  d->release(d->B.theta);
  d->release(const_cast<int*>(d->B.frame_hot));
  d->B.frames = d->B.frame_time = nullptr;
  d->B.theta = nullptr;
  d->B.frame_hot = nullptr;
  d->fe_ready = false;  // until all of it is set
  double *fr = nullptr, *ft = nullptr, *th = nullptr;
  int* fh = nullptr;
  RM_TRY(d->alloc(&fr, nodes * (size_t)n_frames));
  RM_TRY(d->alloc(&ft, (size_t)n_frames));
  RM_TRY(d->alloc(&th, nodes));
  RM_TRY(d->alloc(&fh, 6 * (size_t)n_frames));
  RM_HIP(hipMemcpyAsync(fr, frame_theta, sizeof(double) * nodes * n_frames, hipMemcpyHostToDevice, d->stream));
  {
    const long long ne = (long long)(fnx - 1) * (fny - 1) * (fnz - 1);
    DeviceTemp ebox, mark, vbox;
    RM_HIP(ebox.get(sizeof(int) * 6 * (size_t)ne));
    RM_HIP(mark.get(nodes));
    RM_HIP(vbox.get(sizeof(int) * 6));
    int* eb = static_cast<int*>(ebox.p);
    int* vb = static_cast<int*>(vbox.p);
    unsigned char* mk = static_cast<unsigned char*>(mark.p);
    const auto clear = [&](long long n, int* b) {
      hipLaunchKernelGGL(k_box_clear, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, d->stream, n, b);
    };
    clear(6 * ne, eb);
    clear(6, vb);
    clear(6LL * n_frames, fh);
    hipLaunchKernelGGL(k_elem_boxes, dim3(grid_for(P.NG, 16384)), dim3(256), 0, d->stream, P, tag, eb);
    hipLaunchKernelGGL(k_void_nodes, dim3((unsigned)((nodes + 255) / 256)), dim3(256), 0, d->stream,
                       fr, n_frames, (int)nodes, P.void_temp, mk);
    for (int f = 0; f < n_frames; f += 32768)  // frames on the grid's y axis (65535 at most)
      hipLaunchKernelGGL(k_union_boxes, dim3(grid_for(ne, 64), std::min(32768, n_frames - f)),
                         dim3(256), 0, d->stream, P, fr + (size_t)f * nodes, P.Tm - P.hot_margin,
                         (const unsigned char*)nullptr, eb, fh + 6 * (size_t)f);
    hipLaunchKernelGGL(k_union_boxes, dim3(grid_for(ne, 256)), dim3(256), 0, d->stream, P, fr, 0.0,
                       mk, eb, vb);
    RM_HIP(hipGetLastError());
    RM_HIP(hipMemcpyAsync(P.void_box, vb, sizeof(int) * 6, hipMemcpyDeviceToHost, d->stream));
    RM_HIP(hipStreamSynchronize(d->stream));
  }
  std::vector<double> rel(n_frames);
  for (int f = 0; f < n_frames; f++) rel[f] = frame_time[f] - frame_time[0];  // inTimeOffset_
  RM_HIP(hipMemcpyAsync(ft, rel.data(), sizeof(double) * n_frames, hipMemcpyHostToDevice, d->stream));
  // thetaArray_ starts as theta_[1], the first frame
  RM_HIP(hipMemcpyAsync(th, fr, sizeof(double) * nodes, hipMemcpyDeviceToDevice, d->stream));
  d->B.frames = fr;
  d->B.frame_time = ft;
  d->B.theta = th;
  d->B.frame_hot = fh;
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  // the coming step's field is the first frame as loaded
  c.fs[c.step % 3] = amca::RmField{0, 1, 0.0};
  rm_restart_box(c);
  c.frame = 1;
  c.in_t1 = rel[0];
  c.in_t0 = rel[1];
  c.time_fe = 0.0;
  c.max_dt = c.in_t0 - c.in_t1;  // get_output_time_step_from_txt_file
  RM_TRY(rm_put_counters(d, c));
  d->fe_ready = true;
  return AMCA_OK;
}

amca_status amca_remelt_voxel_map(amca_remelt* d, int32_t* tag, double* par) {
  if (!d || !d->fe_ready) return rm_fail(AMCA_ERR_INVALID, "FE mesh not set");
  RM_HIP(hipStreamSynchronize(d->stream));
  if (tag) RM_HIP(hipMemcpy(tag, d->B.tag, sizeof(int32_t) * d->P.NG, hipMemcpyDeviceToHost));
  if (par)
    RM_HIP(hipMemcpy(par, d->B.par, sizeof(double) * 3 * (size_t)d->P.NG, hipMemcpyDeviceToHost));
  return AMCA_OK;
}

amca_status amca_fe_map_voxels(int32_t nx, int32_t ny, int32_t nz, double h, double x0, double y0,
                               double z0, const int32_t* bin, double tolerance,
                               int32_t max_iterations, int32_t fnx, int32_t fny, int32_t fnz,
                               const double* node_xyz, int32_t* tag, double* par) {
  if (nx < 1 || ny < 1 || nz < 1 || fnx < 2 || fny < 2 || fnz < 2 || !node_xyz || !tag || !par)
    return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  amca_host::FeMesh mesh;
  mesh.fnx = fnx;
  mesh.fny = fny;
  mesh.fnz = fnz;
  mesh.xyz.assign(node_xyz, node_xyz + 3 * (size_t)fnx * fny * fnz);
  amca_host::VoxelMapParams vp;
  vp.nx = nx; vp.ny = ny; vp.nz = nz;
  vp.h = h; vp.x0 = x0; vp.y0 = y0; vp.z0 = z0;
  for (int q = 0; q < 3; q++) vp.bin[q] = (bin && bin[q] > 0) ? bin[q] : 10;
  vp.tol = tolerance;
  vp.max_iter = max_iterations;
  std::vector<int32_t> t;
  std::vector<double> p;
  const bool any = amca_host::map_voxels(mesh, vp, t, p);
  std::memcpy(tag, t.data(), sizeof(int32_t) * t.size());
  std::memcpy(par, p.data(), sizeof(double) * p.size());
  return any ? AMCA_OK : rm_fail(AMCA_ERR_INVALID, "no CA cell lies in the FE mesh");
}

amca_status amca_fe_map_voxels_device(int32_t nx, int32_t ny, int32_t nz, double h, double x0,
                                      double y0, double z0, const int32_t* bin, double tolerance,
                                      int32_t max_iterations, int32_t fnx, int32_t fny,
                                      int32_t fnz, const double* node_xyz, int32_t* tag,
                                      double* par) {
  if (nx < 1 || ny < 1 || nz < 1 || fnx < 2 || fny < 2 || fnz < 2 || !node_xyz || !tag || !par)
    return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  amca_host::FeMesh mesh;
  mesh.fnx = fnx;
  mesh.fny = fny;
  mesh.fnz = fnz;
  mesh.xyz.assign(node_xyz, node_xyz + 3 * (size_t)fnx * fny * fnz);
  amca_host::VoxelMapParams vp;
  vp.nx = nx; vp.ny = ny; vp.nz = nz;
  vp.h = h; vp.x0 = x0; vp.y0 = y0; vp.z0 = z0;
  for (int q = 0; q < 3; q++) vp.bin[q] = (bin && bin[q] > 0) ? bin[q] : 10;
  vp.tol = tolerance;
  vp.max_iter = max_iterations;
  const size_t NG = (size_t)(nx + 2) * (ny + 2) * (nz + 2);
  DeviceTemp dtag, dpar;
  RM_HIP(dtag.get(sizeof(int32_t) * NG));
  RM_HIP(dpar.get(sizeof(double) * 3 * NG));
  bool any = false;
  RM_TRY(map_voxels_device(mesh, vp, static_cast<int32_t*>(dtag.p), static_cast<double*>(dpar.p), 0,
                           any));
  RM_HIP(hipMemcpy(tag, dtag.p, sizeof(int32_t) * NG, hipMemcpyDeviceToHost));
  RM_HIP(hipMemcpy(par, dpar.p, sizeof(double) * 3 * NG, hipMemcpyDeviceToHost));
  return any ? AMCA_OK : rm_fail(AMCA_ERR_INVALID, "no CA cell lies in the FE mesh");
}

namespace {

// ---- loading a state (amca_remelt_set_state) --------------------------------
// The checks and the layout of a loaded state, from the caller's arrays as they
// are: one upload of 9 bytes per cell and 8 per record, then kernels.  The host
// loops over cells and records took 89 ms at 400 x 160 x 80 cells.

// smallest key of a failed check, per pass: cell or record index, and what failed
struct StateErr {
  unsigned long long record_orient, cell, no_record, record_cell;  // ~0: none
  unsigned long long grainless;
};
enum : unsigned { kBadOrient = 0, kBadGrain = 1, kShared = 2 };

__device__ __forceinline__ bool state_interior(const amca::RmParams& P, long long c) {
  const int k = (int)c / P.nxyG, r = (int)c - k * P.nxyG, j = r / P.nxG, i = r - j * P.nxG;
  return !(i == 0 || j == 0 || k == 0 || i == P.nxG - 1 || j == P.nyG - 1 || k == P.nzG - 1);
}

__global__ void k_state_records(amca::RmParams P, int n_orient, int n_grains,
                                const int* __restrict__ gcell, const int* __restrict__ gorient,
                                int* __restrict__ owner, StateErr* err) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < n_grains; g += stride) {
    owner[g] = INT_MAX;
    if (gorient[g] < 0 || gorient[g] >= n_orient)
      atomicMin(&err->record_orient, (unsigned long long)g);
    if (gcell[g] < 0 || gcell[g] >= P.NG) atomicMin(&err->record_cell, (unsigned long long)g);
  }
}

// the first cell of every record, the cells' own checks and the grainless count
__global__ void __launch_bounds__(256)
k_state_cells(amca::RmParams P, int n_orient, int n_grains, const int* __restrict__ orient,
              const int* __restrict__ grain, int* __restrict__ owner, StateErr* err) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  unsigned less = 0;
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < P.NG; c += stride) {
    if (!state_interior(P, c)) continue;
    const int g = grain[c], o = orient[c];
    if (o < -1 || o >= n_orient)
      atomicMin(&err->cell, 4ull * (unsigned long long)c + kBadOrient);
    else if (g >= n_grains)
      atomicMin(&err->cell, 4ull * (unsigned long long)c + kBadGrain);
    if (g < 0) {
      less++;
      if (o <= -1) atomicMin(&err->no_record, (unsigned long long)c);
    } else if (g < n_grains) {
      atomicMin(&owner[g], (int)c);
    }
  }
  for (int o = 32; o > 0; o >>= 1) less += __shfl_xor(less, o, 64);
  if ((threadIdx.x & 63) == 0 && less) atomicAdd(&err->grainless, (unsigned long long)less);
}

__global__ void k_state_shared(amca::RmParams P, int n_grains, const int* __restrict__ grain,
                               const int* __restrict__ owner, StateErr* err) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < P.NG; c += stride) {
    if (!state_interior(P, c)) continue;
    const int g = grain[c];
    if (g >= 0 && g < n_grains && owner[g] != (int)c)
      atomicMin(&err->cell, 4ull * (unsigned long long)c + kShared);
  }
}

// retrieve_grain_information_before_simulation (:312-332): ghosts liquid, other
// cells without an orientation take their grain's; grain records with the centre
// reset to the cell centre and zero length (:282-300)
__global__ void k_state_load(amca::RmParams P, amca::RmBuffers B, int n_grains,
                             const int* __restrict__ orient, const int* __restrict__ grain,
                             const unsigned char* __restrict__ melted,
                             const int* __restrict__ gcell, const int* __restrict__ gorient) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  const long long t0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  for (long long c = t0; c < P.NG; c += stride) {
    int o = -1;
    if (state_interior(P, c)) {
      o = orient[c];
      if (o <= -1) o = gorient[grain[c]];
    }
    B.oid[c] = o;
    B.gid[c] = grain[c];
    B.melted[c] = melted[c];
  }
  for (long long g = t0; g < n_grains; g += stride) {
    const int c = gcell[g];
    const int k = c / P.nxyG, r = c - k * P.nxyG, j = r / P.nxG, i = r - j * P.nxG;
    B.genv[g] = make_double4(P.x0 + P.h * (i - 0.5), P.y0 + P.h * (j - 0.5), P.z0 + P.h * (k - 0.5),
                             0.0);
    B.gco[g] = make_int2(c, gorient[g]);
  }
}

}  // namespace

amca_status amca_remelt_set_state(amca_remelt* d, const int32_t* orient, const int32_t* grain,
                                  const uint8_t* melted, int32_t n_orient, int32_t n_grains,
                                  const int32_t* grain_cell, const int32_t* grain_orient) {
  if (!d || !orient || !grain || !melted || n_grains < 0 || (n_grains > 0 && (!grain_cell || !grain_orient)))
    return rm_fail(AMCA_ERR_INVALID, "bad state arrays");
  amca::RmParams& P = d->P;
  if (n_orient < 0 || n_orient > d->rows_pushed)
    return rm_fail(AMCA_ERR_INVALID, "push the loaded orientation rows before the state");
  // Every interior cell owns at most one grain record and no record is shared:
  // the device grows a record once per flagged cell, as the reference does when
  // each cell carries its own grain.  Records for grainless cells are added by
  // captures and nucleation, so the table needs n_grains + (grainless cells).
  const size_t NG = (size_t)P.NG, ng = (size_t)n_grains;
  const auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t cells = up(sizeof(int32_t) * NG), recs = up(sizeof(int32_t) * std::max<size_t>(ng, 1));
  DeviceTemp tmp;
  RM_HIP(tmp.get(2 * cells + up(NG) + 3 * recs + sizeof(StateErr)));
  char* p = static_cast<char*>(tmp.p);
  int* d_orient = reinterpret_cast<int*>(p);
  int* d_grain = reinterpret_cast<int*>(p + cells);
  unsigned char* d_melted = reinterpret_cast<unsigned char*>(p + 2 * cells);
  int* d_gcell = reinterpret_cast<int*>(p + 2 * cells + up(NG));
  int* d_gorient = reinterpret_cast<int*>(p + 2 * cells + up(NG) + recs);
  int* d_owner = reinterpret_cast<int*>(p + 2 * cells + up(NG) + 2 * recs);
  StateErr* d_err = reinterpret_cast<StateErr*>(p + 2 * cells + up(NG) + 3 * recs);
  StateErr err{~0ull, ~0ull, ~0ull, ~0ull, 0ull};
  hipStream_t s = d->stream;
  RM_HIP(hipMemcpyAsync(d_err, &err, sizeof(err), hipMemcpyHostToDevice, s));
  RM_HIP(hipMemcpyAsync(d_orient, orient, sizeof(int32_t) * NG, hipMemcpyHostToDevice, s));
  RM_HIP(hipMemcpyAsync(d_grain, grain, sizeof(int32_t) * NG, hipMemcpyHostToDevice, s));
  RM_HIP(hipMemcpyAsync(d_melted, melted, NG, hipMemcpyHostToDevice, s));
  if (ng) {
    RM_HIP(hipMemcpyAsync(d_gcell, grain_cell, sizeof(int32_t) * ng, hipMemcpyHostToDevice, s));
    RM_HIP(hipMemcpyAsync(d_gorient, grain_orient, sizeof(int32_t) * ng, hipMemcpyHostToDevice, s));
  }
  const dim3 grid(grid_for(P.NG, 16384)), block(256);
  hipLaunchKernelGGL(k_state_records, dim3(grid_for(n_grains, 16384)), block, 0, s, P, n_orient,
                     n_grains, d_gcell, d_gorient, d_owner, d_err);
  hipLaunchKernelGGL(k_state_cells, grid, block, 0, s, P, n_orient, n_grains, d_orient, d_grain,
                     d_owner, d_err);
  hipLaunchKernelGGL(k_state_shared, grid, block, 0, s, P, n_grains, d_grain, d_owner, d_err);
  RM_HIP(hipGetLastError());
  RM_HIP(hipMemcpyAsync(&err, d_err, sizeof(err), hipMemcpyDeviceToHost, s));
  RM_HIP(hipStreamSynchronize(s));
  if (err.record_orient != ~0ull) return rm_fail(AMCA_ERR_INVALID, "grain orientation out of range");
  if (err.cell != ~0ull)
    return rm_fail(AMCA_ERR_INVALID, (err.cell & 3u) == kBadOrient ? "cell orientation out of range"
                                     : (err.cell & 3u) == kBadGrain
                                         ? "cell grain id out of range"
                                         : "a grain record is shared by two cells");
  if (err.no_record != ~0ull)
    return rm_fail(AMCA_ERR_INVALID, "a cell without orientation has no grain record");
  if (err.record_cell != ~0ull) return rm_fail(AMCA_ERR_INVALID, "grain cell out of range");
  const size_t need = ng + (size_t)err.grainless;
  if (need > d->grain_cap) {
    d->release(d->B.genv);
    d->release(d->B.gco);
    d->B.genv = nullptr;
    d->B.gco = nullptr;
    d->grain_cap = 0;
    RM_TRY(d->alloc(&d->B.genv, need));
    RM_TRY(d->alloc(&d->B.gco, need));
    d->grain_cap = need;
  }
  hipLaunchKernelGGL(k_state_load, grid, block, 0, s, P, d->B, n_grains, d_orient, d_grain, d_melted,
                     d_gcell, d_gorient);
  RM_HIP(hipGetLastError());
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  c.n_grains = n_grains;
  c.n_orient = n_orient;
  rm_restart_box(c);
  RM_TRY(rm_put_counters(d, c));
  d->state_ready = true;
  return AMCA_OK;
}

amca_status amca_remelt_push_orientations(amca_remelt* d, int32_t n, const double* euler3,
                                          const double* l2g9) {
  if (!d || n < 0 || (n > 0 && !l2g9 && !euler3)) return rm_fail(AMCA_ERR_INVALID, "bad rows");
  if (!l2g9 && n > 0) {
    // Octahedron::set_coordinate_transformation_matrix on the host (glibc cos/sin)
    std::vector<double> r(9 * (size_t)n);
    for (int q = 0; q < n; q++) amca_host::rotation_from_euler(euler3 + 3 * q, &r[9 * (size_t)q]);
    RM_TRY(push_rows(d, n, r.data()));
  } else {
    RM_TRY(push_rows(d, n, l2g9));
  }
  for (int q = 0; q < 3 * n; q++) d->euler.push_back(euler3 ? euler3[q] : 0.0);
  return AMCA_OK;
}

amca_status amca_remelt_set_orientation_source(amca_remelt* d, amca_orientation_source src,
                                               void* user) {
  if (!d) return rm_fail(AMCA_ERR_INVALID, "null domain");
  d->source = src;
  d->source_user = user;
  d->rng.reset();
  return AMCA_OK;
}

amca_status amca_remelt_draw_sites_after(amca_remelt* d, uint32_t seed, int64_t skip_draws,
                                         double ns, double dTs_mean, double dTs_sd, double nv,
                                         double dTv_mean, double dTv_sd, int32_t* n_surface_new,
                                         int32_t* n_bulk_new) {
  if (!d || skip_draws < 0) return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  amca_host::Grid g{d->P.nx, d->P.ny, d->P.nz};
  auto rng = std::make_unique<amca_host::GlibcRand>(seed);
  for (int64_t q = 0; q < skip_draws; q++) (void)rng->next();
  // create_nucleation_sites merges into the list already held (the seeds of a
  // loaded microstructure file): a draw on a listed cell only lowers its value
  std::unordered_map<int, double> cell_dt;
  std::vector<int> sites;
  for (size_t q = 0; q < d->site_cells.size(); q++) {
    if (!cell_dt.emplace(d->site_cells[q], d->site_dts[q]).second || d->site_dts[q] < 0)
      return rm_fail(AMCA_ERR_INVALID, "sites to merge with must be distinct cells with undercooling >= 0");
    sites.push_back(d->site_cells[q]);
  }
  const double h = d->P.h;
  amca_host::SiteDraw ds, db;
  {
    std::vector<int> ids;
    amca_host::surface_cells(g, amca_host::SurfaceFaces::kReferenceSix, ids);
    ds = amca_host::create_nucleation_sites((int)ids.size(), [&](int i) { return ids[i]; }, h * h,
                                            ns, dTs_mean, dTs_sd, *rng, cell_dt, sites);
  }
  db = amca_host::create_nucleation_sites((int)(g.nx * (long long)g.ny * g.nz),
                                          amca_host::BulkCellAt{g}, h * h * h, nv, dTv_mean,
                                          dTv_sd, *rng, cell_dt, sites);
  std::vector<double> dts(sites.size());
  for (size_t q = 0; q < sites.size(); q++) dts[q] = cell_dt[sites[q]];
  RM_TRY(amca_remelt_set_sites(d, (int32_t)sites.size(), sites.data(), dts.data()));
  d->source = nullptr;
  d->source_user = nullptr;
  d->rng = std::move(rng);
  if (n_surface_new) *n_surface_new = ds.n_new;
  if (n_bulk_new) *n_bulk_new = db.n_new;
  return AMCA_OK;
}

amca_status amca_remelt_draw_sites(amca_remelt* d, uint32_t seed, double ns, double dTs_mean,
                                   double dTs_sd, double nv, double dTv_mean, double dTv_sd,
                                   int32_t* n_sites) {
  int32_t a = 0, b = 0;
  RM_TRY(amca_remelt_draw_sites_after(d, seed, 0, ns, dTs_mean, dTs_sd, nv, dTv_mean, dTv_sd, &a,
                                      &b));
  if (n_sites) *n_sites = (int32_t)d->site_cells.size();
  return AMCA_OK;
}

amca_status amca_remelt_sites(amca_remelt* d, int32_t cap, int32_t* cell, double* dT_crit,
                              int32_t* n) {
  if (!d || !n) return rm_fail(AMCA_ERR_INVALID, "null argument");
  *n = (int32_t)d->site_cells.size();
  const int m = std::max(0, std::min(cap, *n));
  if (m > 0 && cell) std::memcpy(cell, d->site_cells.data(), sizeof(int32_t) * m);
  if (m > 0 && dT_crit) std::memcpy(dT_crit, d->site_dts.data(), sizeof(double) * m);
  return AMCA_OK;
}

amca_status amca_remelt_euler(amca_remelt* d, int32_t cap, double* euler3, int32_t* n) {
  if (!d || !n) return rm_fail(AMCA_ERR_INVALID, "null argument");
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  *n = c.n_orient;
  const int m = std::max(0, std::min(std::min(cap, c.n_orient), (int)(d->euler.size() / 3)));
  if (euler3 && m > 0) std::memcpy(euler3, d->euler.data(), sizeof(double) * 3 * m);
  return AMCA_OK;
}

amca_status amca_rosenthal_frames(int64_t n_nodes, const double* node_xyz, int32_t n_frames,
                                  double t0, double dt, double P, double eta, double v, double k,
                                  double alpha, double T0, double x_start, double y_c,
                                  double z_top, double r_min, double* out) {
  if (n_nodes < 1 || n_frames < 1 || !node_xyz || !out || !(k > 0) || !(alpha > 0))
    return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  amca_host::RosenthalParams p{P, eta, v, k, alpha, T0, x_start, y_c, z_top, r_min};
  amca_host::rosenthal_frames(n_nodes, node_xyz, n_frames, t0, dt, p, out);
  return AMCA_OK;
}

amca_status amca_write_fe_frames(const char* path, int32_t title_lines, int32_t fnx, int32_t fny,
                                 int32_t fnz, const double* node_xyz, int32_t n_frames,
                                 const double* times, const double* theta) {
  if (!path || title_lines < 0 || fnx < 2 || fny < 2 || fnz < 2 || n_frames < 1 || !node_xyz ||
      !times || !theta)
    return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  if ((long long)fnx * fny * fnz > INT_MAX) return rm_fail(AMCA_ERR_INVALID, "mesh too large");
  try {
    amca_host::write_fe_text(path, title_lines, fnx, fny, fnz, node_xyz, n_frames, times, theta);
  } catch (const std::exception& e) {
    return rm_fail(AMCA_ERR_IO, std::string(path) + ": " + e.what());
  }
  return AMCA_OK;
}

amca_status amca_voronoi_substrate(int32_t nx, int32_t ny, int32_t nz, double h, double x0,
                                   double y0, double z0, int32_t n_seeds, uint64_t seed,
                                   int32_t* label, double* euler3) {
  if (nx < 1 || ny < 1 || nz < 1 || n_seeds < 1 || !label || !euler3 || !(h > 0))
    return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  amca_host::voronoi_labels(nx, ny, nz, h, x0, y0, z0, n_seeds, seed, label, euler3);
  return AMCA_OK;
}

amca_status amca_remelt_set_sites(amca_remelt* d, int32_t n, const int32_t* cell,
                                  const double* dT_crit) {
  if (!d || n < 0 || (n > 0 && (!cell || !dT_crit))) return rm_fail(AMCA_ERR_INVALID, "bad sites");
  for (int i = 0; i < n; i++) {
    if (cell[i] < 0 || cell[i] >= d->P.NG) return rm_fail(AMCA_ERR_INVALID, "site out of range");
    if (i > 0 && cell[i] <= cell[i - 1]) return rm_fail(AMCA_ERR_INVALID, "sites must ascend");
  }
  d->site_cells.assign(cell, cell + n);
  d->site_dts.assign(dT_crit, dT_crit + n);
  d->release(d->B.site_cell);
  d->release(d->B.site_dt);
  RM_TRY(d->alloc(&d->B.site_cell, (size_t)std::max(n, 1)));
  RM_TRY(d->alloc(&d->B.site_dt, (size_t)std::max(n, 1)));
  if (n > 0) {
    RM_HIP(hipMemcpyAsync(d->B.site_cell, cell, sizeof(int32_t) * n, hipMemcpyHostToDevice, d->stream));
    RM_HIP(hipMemcpyAsync(d->B.site_dt, dT_crit, sizeof(double) * n, hipMemcpyHostToDevice, d->stream));
  }
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  c.n_sites = n;
  RM_TRY(rm_put_counters(d, c));
  d->site_blocks = std::max(1, std::min((n + 255) / 256, (int)amca::kMaxBlocks));
  return AMCA_OK;
}

amca_status amca_remelt_enable_log(amca_remelt* d, int32_t capacity) {
  if (!d || capacity < 0) return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  RM_HIP(hipStreamSynchronize(d->stream));
  d->release(d->B.log);
  d->B.log = nullptr;
  if (capacity > 0) RM_TRY(d->alloc(&d->B.log, (size_t)capacity));
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  c.log_cap = capacity;
  return rm_put_counters(d, c);
}

amca_status amca_remelt_read_log(amca_remelt* d, int32_t cap, amca_remelt_step_record* rows,
                                 int32_t* n_rows) {
  if (!d || !n_rows) return rm_fail(AMCA_ERR_INVALID, "null argument");
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  const long long avail = std::min<long long>(c.step, c.log_cap);
  *n_rows = (int32_t)avail;
  const long long n = std::min<long long>(avail, std::max(cap, 0));
  if (n > 0 && rows && d->B.log) {
    std::vector<amca::RmLogRow> tmp((size_t)n);
    RM_HIP(hipMemcpy(tmp.data(), d->B.log, sizeof(amca::RmLogRow) * n, hipMemcpyDeviceToHost));
    for (long long i = 0; i < n; i++) {
      rows[i].time_before = tmp[i].time_before;
      rows[i].dt = tmp[i].dt;
      rows[i].n_nucleated = tmp[i].n_nucleated;
      rows[i].n_captured = tmp[i].n_captured;
      rows[i].n_fresh = tmp[i].n_fresh;
      rows[i].n_flagged = tmp[i].n_flagged;
      rows[i].n_fallback = tmp[i].n_fallback;
      rows[i].n_box = tmp[i].n_box;
    }
  }
  return AMCA_OK;
}

amca_status amca_pow_selftest(int64_t n, const double* x, double y, double* out) {
  if (n < 0 || (n > 0 && (!x || !out))) return rm_fail(AMCA_ERR_INVALID, "bad arguments");
  if (!amca_libm::pow_exponent_supported(y))
    return rm_fail(AMCA_ERR_INVALID, "exponent outside [2^-65, 2^63) in magnitude");
  for (int64_t i = 0; i < n; i++)
    if (!(x[i] > 0) || !(x[i] < HUGE_VAL))
      return rm_fail(AMCA_ERR_INVALID, "bases must be finite and positive");
  if (n == 0) return AMCA_OK;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return rm_fail(AMCA_ERR_NO_DEVICE, "no HIP device visible");
  double *dx = nullptr, *dout = nullptr;
  hipError_t e = hipMalloc(&dx, sizeof(double) * n);
  if (e == hipSuccess) e = hipMalloc(&dout, sizeof(double) * n);
  if (e == hipSuccess) e = hipMemcpy(dx, x, sizeof(double) * n, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = amca::launch_pow_selftest(n, dx, y, dout, 0);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(out, dout, sizeof(double) * n, hipMemcpyDeviceToHost);
  if (dx) (void)hipFree(dx);
  if (dout) (void)hipFree(dout);
  if (e != hipSuccess) return rm_fail(AMCA_ERR_HIP, std::string("pow self-test: ") + hipGetErrorString(e));
  return AMCA_OK;
}

}  // extern "C"

namespace {

// One domain's run, in rounds: plan (the next batch of steps, after any rows
// a stopped step asked for), enqueue, collect the counters.
struct RunState {
  long long start = 0, batch = 4, k = 0;
  bool done = false;
  amca::RmCounters c{};
};

amca_status run_begin(amca_remelt* d, RunState& st) {
  if (!d || !d->fe_ready) return rm_fail(AMCA_ERR_INVALID, "FE mesh not set");
  RM_TRY(rm_counters(d, &st.c));
  st.start = st.c.step;
  return AMCA_OK;
}

amca_status run_plan(amca_remelt* d, RunState& st, int64_t max_steps) {
  amca::RmCounters& c = st.c;
  st.k = 0;
  if (c.err == 1) return rm_fail(AMCA_ERR_CAPACITY, "orientation table exhausted");
  if (c.err == 2) return rm_fail(AMCA_ERR_INVALID, "FE time ratio below zero");
  const long long taken = c.step - st.start;
  if (c.exhausted || !(c.tcafe < d->desc.final_time) || (max_steps >= 0 && taken >= max_steps)) {
    st.done = true;
    return AMCA_OK;
  }
  if (c.need_rows) {
    // a step stopped: its armed sites could need more rows than were pushed
    const long long want = (long long)c.n_orient + c.armed[c.step & 1];
    if (want > d->P.orient_cap) return rm_fail(AMCA_ERR_CAPACITY, "orientation table exhausted");
    RM_TRY(ensure_rows(d, want + d->row_reserve));
    if (d->rows_pushed < want)
      return rm_fail(AMCA_ERR_CAPACITY, "orientation rows exhausted and no orientation source set");
    RM_TRY(rm_counters(d, &c));
    c.need_rows = 0;
    c.armed[c.step & 1] = 0;
    RM_TRY(rm_put_counters(d, c));
  }
  st.k = st.batch;
  if (max_steps >= 0) st.k = std::min<long long>(st.k, max_steps - taken);
  if (c.n_sites > 0 && (d->source || d->rng))
    RM_TRY(ensure_rows(d, (long long)c.n_orient + d->row_reserve));
  return AMCA_OK;
}

amca_status run_enqueue(amca_remelt* d, RunState& st) {
  if (st.k <= 0) return AMCA_OK;
  if (d->timing) {
    for (long long q = 0; q < st.k; q++) RM_TRY(rm_enqueue_step(d));
  } else {
    RM_TRY(rm_enqueue_steps(d, st.k));
  }
  return AMCA_OK;
}

amca_status run_collect(amca_remelt* d, RunState& st) {
  if (st.k <= 0) return AMCA_OK;
  RM_TRY(rm_counters(d, &st.c));
  st.batch = std::min<long long>(st.batch * 2, 64);
  return AMCA_OK;
}

amca_status run_end(amca_remelt* d, RunState& st, amca_remelt_counters* out) {
  // cells outside the last step's box take that step's T and cooling
  if (st.c.step > st.start) {
    RM_HIP(amca::rm_launch_complete(d->P, d->B, d->stream));
    RM_HIP(hipStreamSynchronize(d->stream));
  }
  rm_fill(d, st.c, out);
  return AMCA_OK;
}

}  // namespace

extern "C" {

amca_status amca_remelt_run(amca_remelt* d, int64_t max_steps, amca_remelt_counters* out) {
  RunState st;
  RM_TRY(run_begin(d, st));
  while (true) {
    RM_TRY(run_plan(d, st, max_steps));
    if (st.done) break;
    RM_TRY(run_enqueue(d, st));
    RM_TRY(run_collect(d, st));
  }
  return run_end(d, st, out);
}

amca_status amca_remelt_run_many(amca_remelt* const* ds, int32_t n, int64_t max_steps,
                                 amca_remelt_counters* outs) {
  if (!ds || n < 1) return rm_fail(AMCA_ERR_INVALID, "no domains");
  for (int i = 0; i < n; i++)
    for (int j = 0; j < i; j++)
      if (ds[i] == ds[j]) return rm_fail(AMCA_ERR_INVALID, "a domain is listed twice");
  std::vector<RunState> st((size_t)n);
  for (int i = 0; i < n; i++) RM_TRY(run_begin(ds[i], st[i]));
  while (true) {
    int live = 0;
    // every domain's next batch is queued on its own stream before any is waited for
    for (int i = 0; i < n; i++) {
      if (st[i].done) continue;
      RM_TRY(run_plan(ds[i], st[i], max_steps));
      if (st[i].done) continue;
      RM_TRY(run_enqueue(ds[i], st[i]));
      live++;
    }
    if (!live) break;
    for (int i = 0; i < n; i++)
      if (!st[i].done) RM_TRY(run_collect(ds[i], st[i]));
  }
  for (int i = 0; i < n; i++) RM_TRY(run_end(ds[i], st[i], outs ? &outs[i] : nullptr));
  return AMCA_OK;
}

amca_status amca_remelt_set_window(amca_remelt* d, int32_t on) {
  if (!d) return rm_fail(AMCA_ERR_INVALID, "null domain");
  d->P.window = on ? 1 : 0;
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  rm_restart_box(c);
  RM_TRY(rm_put_counters(d, c));
  return AMCA_OK;
}

amca_status amca_remelt_set_row_reserve(amca_remelt* d, int32_t rows) {
  if (!d || rows < 0) return rm_fail(AMCA_ERR_INVALID, "bad row reserve");
  d->row_reserve = rows;
  return AMCA_OK;
}

amca_status amca_remelt_set_graph_steps(amca_remelt* d, int32_t steps) {
  if (!d || steps < 0 || steps > 1024) return rm_fail(AMCA_ERR_INVALID, "bad graph step count");
  RM_HIP(hipStreamSynchronize(d->stream));
  d->drop_graph();
  d->graph_steps = steps;
  return AMCA_OK;
}

amca_status amca_remelt_last_box(amca_remelt* d, int32_t* box6) {
  if (!d || !box6) return rm_fail(AMCA_ERR_INVALID, "null argument");
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  if (c.last_step < 0) return rm_fail(AMCA_ERR_INVALID, "no step has run");
  const amca::RmBox& b = c.box[c.last_step & 1];
  for (int a = 0; a < 3; a++) {
    box6[a] = b.lo[a];
    box6[3 + a] = b.hi[a];
  }
  return AMCA_OK;
}

amca_status amca_remelt_get_counters(amca_remelt* d, amca_remelt_counters* out) {
  if (!d || !out) return rm_fail(AMCA_ERR_INVALID, "null argument");
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  rm_fill(d, c, out);
  return AMCA_OK;
}

namespace {
// Up to here one copy of the (cell, orientation) pairs and a host loop take less than the
// kernel and the second copy.  A download, ms, split on the host and on the device: 96 K
// records 0.39 / 0.45, 640 K 2.35 / 2.23, 1.28 M 6.4 / 6.0.
constexpr size_t kHostSplit = 1 << 18;

__global__ void k_split_pairs(long long n, const int2* __restrict__ in, int* __restrict__ x,
                              int* __restrict__ y) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int2 v = in[i];
    x[i] = v.x;
    y[i] = v.y;
  }
}
}  // namespace

amca_status amca_remelt_download(amca_remelt* d, int32_t* orient, int32_t* grain, double* T,
                                 uint8_t* melted, uint8_t* cooling, int32_t grain_cap,
                                 double* genv, int32_t* gcell, int32_t* gorient, int32_t* n_grains) {
  if (!d) return rm_fail(AMCA_ERR_INVALID, "null domain");
  const size_t ng = (size_t)d->P.NG;
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  if (orient) RM_HIP(hipMemcpy(orient, d->B.oid, sizeof(int32_t) * ng, hipMemcpyDeviceToHost));
  if (grain) RM_HIP(hipMemcpy(grain, d->B.gid, sizeof(int32_t) * ng, hipMemcpyDeviceToHost));
  if (T) RM_HIP(hipMemcpy(T, d->B.T, sizeof(double) * ng, hipMemcpyDeviceToHost));
  if (melted) RM_HIP(hipMemcpy(melted, d->B.melted, ng, hipMemcpyDeviceToHost));
  if (cooling) RM_HIP(hipMemcpy(cooling, d->B.cooling, ng, hipMemcpyDeviceToHost));
  if (n_grains) *n_grains = c.n_grains;
  const size_t m = (size_t)std::max(0, std::min(grain_cap, c.n_grains));
  if (m > 0) {
    if (genv) RM_HIP(hipMemcpy(genv, d->B.genv, sizeof(double) * 4 * m, hipMemcpyDeviceToHost));
    if ((gcell || gorient) && m <= kHostSplit) {
      std::vector<int32_t> co(2 * m);
      RM_HIP(hipMemcpy(co.data(), d->B.gco, sizeof(int32_t) * 2 * m, hipMemcpyDeviceToHost));
      for (size_t g = 0; g < m; g++) {
        if (gcell) gcell[g] = co[2 * g];
        if (gorient) gorient[g] = co[2 * g + 1];
      }
    } else if (gcell || gorient) {
      // split in the list of captures, which holds nothing between steps and room for
      // one pair per cell: a piece at a time, cells, then orientations
      const size_t piece = (size_t)d->P.N;
      int* q = reinterpret_cast<int*>(d->B.clist);
      for (size_t g0 = 0; g0 < m; g0 += piece) {
        const size_t n = std::min(piece, m - g0);
        hipLaunchKernelGGL(k_split_pairs, dim3(grid_for((long long)n, 16384)), dim3(256), 0,
                           d->stream, (long long)n, d->B.gco + g0, q, q + n);
        RM_HIP(hipGetLastError());
        if (gcell)
          RM_HIP(hipMemcpyAsync(gcell + g0, q, sizeof(int32_t) * n, hipMemcpyDeviceToHost, d->stream));
        if (gorient)
          RM_HIP(hipMemcpyAsync(gorient + g0, q + n, sizeof(int32_t) * n, hipMemcpyDeviceToHost,
                                d->stream));
        RM_HIP(hipStreamSynchronize(d->stream));
      }
    }
  }
  return AMCA_OK;
}

amca_status amca_remelt_use_surrogate(amca_remelt* d, amca_mlp* m, const amca_surrogate_desc* sd,
                                      const amca_scan* scan, double band, double resid) {
  if (!d || !d->fe_ready) return rm_fail(AMCA_ERR_INVALID, "FE mesh not set");
  if (!m || !sd || !scan || !(band >= 0) || !(resid >= 0))
    return rm_fail(AMCA_ERR_INVALID, "bad surrogate arguments");
  amca::RmParams& P = d->P;
  if (sd->fnx != P.fnx || sd->fny != P.fny || sd->fnz != P.fnz)
    return rm_fail(AMCA_ERR_INVALID, "surrogate mesh differs from the domain's FE mesh");
  // the FE mesh must be the uniform lattice the description names
  for (int n = 0; n < P.nodes; n++) {
    const int i = n % P.fnx, j = (n / P.fnx) % P.fny, k = n / (P.fnx * P.fny);
    const double e[3] = {sd->fx0 + i * sd->fdx, sd->fy0 + j * sd->fdx, sd->fz0 + k * sd->fdx};
    for (int q = 0; q < 3; q++)
      if (std::fabs(d->node_xyz[3 * (size_t)n + q] - e[q]) > 1e-9 * sd->fdx)
        return rm_fail(AMCA_ERR_INVALID, "the FE mesh is not the uniform lattice of the description");
  }
  RM_HIP(hipStreamSynchronize(d->stream));
  // time span of the frames
  std::vector<double> ft(P.n_frames);
  RM_HIP(hipMemcpy(ft.data(), d->B.frame_time, sizeof(double) * P.n_frames, hipMemcpyDeviceToHost));
  const double tmax = ft.back();
  const double h = P.h;
  const double xlo = std::min(P.x0 - 1.0 * h, sd->fx0), xhi = std::max(P.x0 + (P.nx + 1) * h, sd->fx0 + (P.fnx - 1) * sd->fdx);
  const double a = xlo - scan->x_start - std::max(0.0, scan->v) * tmax - 2 * h;
  const double b = xhi - scan->x_start - std::min(0.0, scan->v) * tmax + 2 * h;
  const int nxi = (int)std::ceil((b - a) / h) + 2;
  d->release(const_cast<float*>(d->B.sur_cell));
  d->release(const_cast<float*>(d->B.sur_node));
  d->release(d->B.node_bad);
  d->release(d->B.elem_fb);
  d->release(d->B.sur_stats);
  d->release(d->B.fb_slots);
  float *tc = nullptr, *tn = nullptr;
  unsigned char *nb = nullptr, *eb = nullptr;
  double* stats = nullptr;
  RM_TRY(d->alloc(&tc, (size_t)nxi * P.nyG * P.nzG));
  RM_TRY(d->alloc(&tn, (size_t)nxi * P.fny * P.fnz));
  RM_TRY(d->alloc(&nb, (size_t)P.nodes));
  RM_TRY(d->alloc(&eb, 2 * (size_t)(P.fnx - 1) * (P.fny - 1) * (P.fnz - 1)));
  RM_TRY(d->alloc(&stats, 8));
  int* slots = nullptr;
  RM_TRY(d->alloc(&slots, 256));
  RM_HIP(hipMemset(slots, 0, sizeof(int) * 256));
  // cell lattice: y, z at the cell centres (ghosts included); node lattice at the nodes
  SurLattice gc{a, h, nxi, P.y0 - 0.5 * h, h, P.nyG, P.z0 - 0.5 * h, h, P.nzG};
  SurLattice gn{a, h, nxi, sd->fy0, sd->fdx, P.fny, sd->fz0, sd->fdx, P.fnz};
  amca_status st = surrogate_eval_lattice(m, *sd, *scan, gc, tc);
  if (st == AMCA_OK) st = surrogate_eval_lattice(m, *sd, *scan, gn, tn);
  if (st != AMCA_OK) return rm_fail(st, std::string("surrogate evaluation: ") + surrogate_error());
  d->B.sur_cell = tc;
  d->B.sur_node = tn;
  d->B.node_bad = nb;
  d->B.elem_fb = eb;
  d->B.sur_stats = stats;
  d->B.fb_slots = slots;
  P.sur = 1;
  P.sur_xi0 = a;
  P.sur_dxi = h;
  P.sur_nxi = nxi;
  P.sur_nxi_nodes = nxi;
  P.sur_x_start = scan->x_start;
  P.sur_v = scan->v;
  P.sur_band = band;
  P.sur_resid = resid;
  P.fx0 = sd->fx0;
  P.fy0 = sd->fy0;
  P.fz0 = sd->fz0;
  P.fdx = sd->fdx;
  // hot region of the cell table (xi index, j, k), for the active box
  {
    int* hb = nullptr;
    RM_TRY(d->alloc(&hb, 6));
    const int init[6] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN};
    RM_HIP(hipMemcpy(hb, init, sizeof(init), hipMemcpyHostToDevice));
    RM_HIP(amca::rm_launch_sur_hot(P, d->B, hb, d->stream));
    int got[6];
    RM_HIP(hipMemcpyAsync(got, hb, sizeof(got), hipMemcpyDeviceToHost, d->stream));
    RM_HIP(hipStreamSynchronize(d->stream));
    d->release(hb);
    P.sur_hot[0] = got[0];
    P.sur_hot[1] = got[3];
    P.sur_hot[2] = got[1];
    P.sur_hot[3] = got[4];
    P.sur_hot[4] = got[2];
    P.sur_hot[5] = got[5];
  }
  amca::RmCounters c;
  RM_TRY(rm_counters(d, &c));
  rm_restart_box(c);
  RM_TRY(rm_put_counters(d, c));
  return AMCA_OK;
}

amca_status amca_remelt_surrogate_error(amca_remelt* d, double* out6) {
  if (!d || !out6 || !d->P.sur) return rm_fail(AMCA_ERR_INVALID, "no surrogate in use");
  RM_HIP(hipMemsetAsync(d->B.sur_stats, 0, sizeof(double) * 8, d->stream));
  RM_HIP(amca::rm_launch_sur_error(d->P, d->B, d->stream));
  double s[8];
  RM_HIP(hipMemcpyAsync(s, d->B.sur_stats, sizeof(s), hipMemcpyDeviceToHost, d->stream));
  RM_HIP(hipStreamSynchronize(d->stream));
  out6[0] = s[1] > 0 ? std::sqrt(s[0] / s[1]) : 0.0;  // RMS over all cells with material
  out6[1] = s[1];
  out6[2] = s[3] > 0 ? std::sqrt(s[2] / s[3]) : 0.0;  // RMS over the cells the surrogate serves
  out6[3] = s[3];
  out6[4] = s[4];                                     // max |error| over those cells
  out6[5] = s[5];                                     // cells on the FE path
  return AMCA_OK;
}

amca_status amca_remelt_theta(amca_remelt* d, double* theta) {
  if (!d || !d->fe_ready || !theta) return rm_fail(AMCA_ERR_INVALID, "FE mesh not set");
  RM_HIP(hipStreamSynchronize(d->stream));
  RM_HIP(hipMemcpy(theta, d->B.theta, sizeof(double) * d->P.nodes, hipMemcpyDeviceToHost));
  return AMCA_OK;
}

}  // extern "C"
