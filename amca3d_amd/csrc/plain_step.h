// Device-side state of one CA domain and the kernels of the plain step.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace amca {

// Division by a fixed 32-bit divisor d as a multiply and shifts (the
// round-up method of Granlund and Montgomery, exact for every 32-bit n):
// t = mulhi(m, n), n / d = (t + ((n - t) >> s1)) >> s2.
struct FastDiv {
  unsigned m;
  int s1, s2;
};

// Constant description of a domain, passed by value to every kernel.
struct DevParams {
  int nx, ny, nz;
  int nxG, nyG, nzG;
  int nxyG;
  int NG;                 // ghosted cell count
  long long N;            // interior cell count
  double h, x0, y0, z0;
  double T0, Tm, Tdot, a1, a2, a3;
  double trunc, tsf, max_dt, final_time;
  double sqrt2f;          // (double)sqrtf(2), Octahedron.cpp:260
  int off[26];            // 26-neighbour offsets in the reference's k,j,i order
  int orient_cap;
  int nbX, nbY, nbZ;      // 4x4x4-cell bricks per axis of the liquid / claimed map
  FastDiv fdX, fdY;       // division by nbX and by nbY
  int ids_blocks;         // blocks of the id scan (k_idscan)
  int cmp_blocks;         // blocks of k_count / k_compact, and of the retirement in k_resolve
  int fused;              // the short step: k_wake_claim instead of k_count, k_compact and wave 0's
                          // k_claim, no other kernels for wave 1, its captures in k_tail
};

// Mutable scalars that live on the device, so that a whole step (or many
// steps) runs without a host round trip.
struct DevCounters {
  double t;               // time_
  double dt;              // dT_ of the current step
  double v;               // growth velocity of the current step
  long long step;         // iStep_
  long long n_solid;      // solid interior cells
  int skip;               // 1: this step is past termination, every kernel returns
  int done;               // no liquid cell left
  int site_sel;           // which site buffer holds the live sites
  int n_grains, n_orient;
  int nA_in, nA_out;      // active list lengths (input / survivors)
  double S;               // growth since the last refresh step, the running step's included
  int Sq;                 // S in kWakeUnits per cell, rounded down, at most kWakeLate
  int force;              // the running step is a refresh step: every active grain is awake
  int n_awake;            // length of wave 0's list
  int nW[2];              // capture-wave list lengths
  int n_sites;
  int step_nuc, step_cap, step_nA0;
  int step_sites;         // live sites at the running step's start
  int max_wave;
  int step_wave;          // deepest capturing wave of the running step
  int wave_gbase;         // first new grain id of the running wave
  int w1_lo, w1_n;        // ids of wave 1's entries (wave 0's children)
  int err;                // 1: orientation table exhausted
  int log_cap;
  unsigned tickets[8];    // block tickets of the look-back kernels
  // ids of wave 0's claiming grains (min, max), spread over 64 slots by k_claim
  // block so that blocks rarely meet at one address
  int claim_lo[64], claim_hi[64];
  // wave 1: whether any of its grains claimed a cell, and its grains without a
  // liquid neighbour, spread over 64 slots
  int w1_claims;
  int w1_ret[64];
  // wave-1 grains of the steps in which one of them claimed a cell, since the domain
  // was made: what k_tail's one work-group walks in the short step
  long long w1_walk;
};

struct StepLogRow {
  double time_before, dt;
  int n_nucleated, n_active_before, n_captured, n_active_after;
  long long n_liquid;
  int n_wave1, max_wave;
  int n_sites;
};

// The grain in a cell's slot: its centre, its half-diagonal L before the growth
// of step `stamp` and later ones, id and orientation: half a 128-byte line, all
// that its tests, its children and its end read or write.
struct alignas(64) SlotRec {
  double x, y, z, L;
  int id, o, stamp, pad;
  double spare[2];
};

// Device buffers of one domain (all owned by the handle).
//
// The grid is cut into 4x4x4-cell bricks (x fastest); cell (i, j, k) is lane
// ((k&3)*16 + (j&3)*4 + (i&3)) of brick b, and its "slot" is 64 b + lane
// (claim_index).  Per brick: two 64-bit words of the 1-bit maps, [2b] liquid
// and [2b+1] claimed, and the active word (a grain whose cell has the bit set
// is on the reference's active list).  Per slot: the grain occupying the cell
// (its record) and the claim word of the capture waves.  Steps read and write
// only these: wave 0 walks the awake slots in brick order, so neighbouring
// entries share map words; wave 1's list holds slots in its parents' brick order,
// the lists of waves >= 2 in grain-id order.  The reference's layouts (cellGrainID_ / cellOrientationID_ on the
// ghosted grid, x fastest; records by grain id) are materialized from the slots
// when a download asks for them.
//
// Sleep.  Every active grain grows by the same increment in a step, so the growth
// it needs to enclose its nearest liquid neighbour is known when it is tested:
// the growth clock S (DevCounters) at which it can next capture goes to `wake`,
// and until then a step does not touch it (about one active grain in five is
// awake in a step).  Its L is worked out when it wakes, retires or is downloaded,
// by adding the increments of the steps since `stamp` one by one, in order: the
// additions of Grain::grow, so the same value to the bit.  The liquid set only
// shrinks, so a sleeping grain can never capture earlier than its clock says.
// At a refresh step (every kRefresh steps, or when S nears its range) all active
// grains are awake and take their L anew, and S restarts from zero, so no replay
// outlasts the ring of increments.
struct DevBuffers {
  int* gid;               // cellGrainID_ [NG], materialized for downloads
  int* oid;               // cellOrientationID_ [NG], materialized for downloads
  int* claim;             // smallest claiming grain id per slot, INT_MAX when free [64 nB]
  unsigned long long* bmap;  // brick words: liquid, claimed [2 nB]
  unsigned long long* amap;  // brick words: active grains [nB]
  SlotRec* rec;           // the grain in each slot [64 nB]
  unsigned short* wake;   // growth clock (kWakeUnits per cell, rounded down) from which the
                          // active grain in the slot may capture a cell [64 nB]
  double* inc;            // growth increments of the last kRing steps, by step [kRing]
  unsigned long long* cl1;  // brick words: cells claimed in wave 1 [nB]
  unsigned long long* awk;  // brick words: active grains awake in the running step [nB]
  double4* genv;          // envelope by grain id, materialized for downloads [N]
  int2* gco;              // grain -> (cell, orientation), materialized for downloads into the
                          // room of plist [N]
  int* alist;             // wave-0 list: awake slots in brick order (short step: one segment per
                          // k_wake_claim block, from the block's first slot) [64 nB]
  int4* plist;            // wave-0 capturing grains: (id, slot, captured slots), one segment
                          // per k_resolve block from its first list entry [64 nB]
  unsigned char* cnt;     // captures per grain id, nonzero only inside a wave-0 step [N]
  int* coff;              // first child (wave-relative) per capturing grain id [N]
  unsigned* idtot;        // wave-0 captures per id-scan block [kMaxIdsBlocks]
  unsigned* cmptot;       // awake grains per compaction block [kMaxBlocks]
  int* listW[2];          // capture-wave lists (slots): [0] wave 1, in its parents' brick order
                          // and in the room of alist, then alternately the waves >= 2, in
                          // grain-id order [N]
  unsigned long long* masks;  // per wave entry: inside bits << 32 | grain id (wave 0) or liquid
                              // bits (waves >= 1) [64 nB]
  int* site_cell[2];      // live nucleation sites, ascending cell, ping-pong
  double* site_dt[2];
  double* l2g;            // orientation table, 9 doubles per row
  unsigned* lb_flag;      // look-back state: epoch<<2 | state; from kStatBase the grains retired
                          // per block [kLbSites * kMaxBlocks]
  unsigned long long* lb_agg;
  unsigned long long* lb_pref;
  StepLogRow* log;
  DevCounters* ctr;
};

constexpr int kBlock = 256;       // threads per block of the list kernels
constexpr int kMaxBlocks = 4096;  // blocks of a look-back kernel
constexpr int kLbSites = 2;       // look-back arrays: [0] k_nucleate's look-back, [1] k_resolve's
                                  // per-block statistics (lb_agg, lb_pref at kStatBase + block)
constexpr int kStatBase = kMaxBlocks;
constexpr int kRefresh = 2048;    // most steps between refresh steps
constexpr int kRing = 2 * kRefresh;  // growth increments kept
// Wake clocks: 1/1024 of a cell (a step's growth is some thousandths to a fifth of
// a cell, so rounding down wakes a grain about a step early at most); S is
// restarted from kWakeSpan cells, within the 16 bits.
constexpr int kWakeUnits = 1024, kWakeSpan = 60;
constexpr int kWakeLate = 65534, kWakeNever = 65535;
constexpr int kMaxIdsBlocks = 2048;  // blocks of the id scan (a k_resolve block keeps one count each)

inline FastDiv make_fastdiv(unsigned d) {
  int l = 0;
  while ((1ull << l) < d) l++;  // ceil(log2 d)
  FastDiv f;
  f.m = (unsigned)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
  f.s1 = l < 1 ? l : 1;
  f.s2 = l > 1 ? l - 1 : 0;
  return f;
}

// Kernel launchers (plain_step.hip).  Each returns hipGetLastError().
hipError_t launch_init_grid(const DevParams& P, const DevBuffers& B, hipStream_t s);
hipError_t launch_nucleate(const DevParams& P, const DevBuffers& B, int blocks, hipStream_t s);
hipError_t launch_claim(const DevParams& P, const DevBuffers& B, int wave, int blocks,
                        hipStream_t s);
// Waves 0 and 1: k_claim, k_resolve, k_idscan and k_emit in that order (k_emit of
// wave 0 makes wave 1's claims);
// k_resolve and k_emit with the same `blocks` (<= kMaxBlocks list chunks)
hipError_t launch_resolve(const DevParams& P, const DevBuffers& B, int wave, int blocks,
                          hipStream_t s);
// wave 0's list: the awake slots in brick order (k_count: awake grains per
// block of bricks, then k_compact over the same blocks)
hipError_t launch_count(const DevParams& P, const DevBuffers& B, int blocks, hipStream_t s);
hipError_t launch_compact(const DevParams& P, const DevBuffers& B, int blocks, hipStream_t s);
// the short step's list and claims of wave 0 (P.cmp_blocks blocks, as its
// k_resolve and k_emit of wave 0)
hipError_t launch_wake_claim(const DevParams& P, const DevBuffers& B, hipStream_t s);
// child offsets of a wave's capturing grains, an exclusive scan over their
// ids (P.ids_blocks blocks; `nres` = blocks of the wave's k_resolve, whose
// statistics words it reads)
hipError_t launch_idscan(const DevParams& P, const DevBuffers& B, int wave, int nres,
                         hipStream_t s);
// from the slots: gid / oid on the ghosted grid (kMatFields), genv / gco by grain id
// (kMatGrains), or gid / oid and genv (kMatDevice)
enum { kMatFields, kMatGrains, kMatDevice };
hipError_t launch_materialize(const DevParams& P, const DevBuffers& B, int what, hipStream_t s);
// envelopes by cell of the n ghosted cells from c0 on
hipError_t launch_cell_env(const DevParams& P, const DevBuffers& B, long long c0, int n, double4* out,
                           hipStream_t s);
hipError_t launch_emit(const DevParams& P, const DevBuffers& B, int wave, int blocks,
                       hipStream_t s);
hipError_t launch_tail(const DevParams& P, const DevBuffers& B, hipStream_t s);

// One step of many domains in one launch per kernel (device arrays of the
// domains' parameters and buffers; per-block (domain, block, count) maps).
struct BatchLaunch {
  const DevParams* P;
  const DevBuffers* B;
  const int4* map_nuc;   // nucleation geometry per domain
  const int4* map_list;  // claim geometry
  const int4* map_emit;  // resolve / emit geometry
  const int4* map_one;   // one block per domain (tail)
  const int4* map_ids;   // id-scan geometry
  const int4* map_cmp;   // compaction geometry (k_count and k_compact)
  int n_nuc, n_list, n_emit, n_one, n_ids, n_cmp;
  int fused;             // the domains take the short step
};
hipError_t launch_batch_step(const BatchLaunch& L, hipStream_t s);
// out[d] = (finished, error, step, w1_walk), the last two their low 31 bits, for each
// of n domains
hipError_t launch_batch_status(const BatchLaunch& L, int n, int4* out, hipStream_t s);
hipError_t launch_envelope_selftest(int n, const double* env4, const double* l2g9,
                                    const double* cell3, double h, double trunc, double sqrt2f,
                                    int* inside, double* child4, hipStream_t s);

}  // namespace amca
