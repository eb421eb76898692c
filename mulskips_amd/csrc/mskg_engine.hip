// mskg_engine.hip -- MI355X KMC event engine: kernels and the C ABI of
// include/mskg.h.
//
// Kernels
//   k_rate_sweep   Get_Prob over every lattice point (HBM-bound stream of the
//                  packed words + neighbour gathers); the rate-update sweep.
//   k_replay       applies a logged event sequence with the reference's
//                  update rules (one wave; events are strictly ordered).
//   k_build_lists  per-tile candidate lists from the classes (after an upload,
//                  a rate sweep or a replay); k_tile_rates: their rate totals.
//   k_pass         one colour of the synchronous-sublattice sweep: each
//                  workgroup (one 64-wide wave) runs rejection-free KMC inside
//                  one tile for the window tau, selecting events with a
//                  wavefront prefix scan over the tile's FP32 rates held in
//                  LDS, FP64 partial sums and Philox-4x32-10 draws.
//   k_sweep        the eight colours of a sweep in one launch, each tile
//                  starting when its lower-colour neighbours are done (same
//                  result as eight k_pass launches, without their barriers);
//   k_sweep_xcd    the same on one XCD, for small lattices.
//   k_sweep_end    fixed-order FP64 sum of the tile rate totals -> next tau
//                  and the clock.
//   k_serial       serial BKL over a batch of lattices (one wave each).
//   k_adjoint      log replay with per-class likelihood statistics.
//   k_build_slab, k_frame_count / k_frame_scan / k_frame_write: device builder,
//                  frame records.
//   k_words_in / k_words_out / k_lists_in / k_state_write: LattCoo and the
//                  particle lists in and out.
// The event kernels are templates on the rate model (laser annealing,
// coverage species), chosen at launch from the tables.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstdarg>
#include <cstring>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/mskg.h"
#include "mskg_events.h"

using namespace mskg;

namespace {

constexpr int WAVE = 64;

// Per-sweep accumulators, striped over slots so that thousands of tile
// waves do not serialise on one address; k_sweep_end folds them.
constexpr int NSLOT = 128;
// Device-side stop at the run's event or time limit (reported as MSKG_STOP_LIMIT).
constexpr int STOP_AT_LIMIT = 100;
// Events one tile may execute in one window (a bound on the wave's work).
constexpr int PASS_EVENT_CAP = 1 << 16;
// With only the bottom planes stored (stored_len_z), an event's site stays
// this many planes below the top stored plane (Lattice::ztop): an event
// reads at most 12 planes and writes at most 6 planes away from its site.
constexpr int TOP_MARGIN = 24;
struct Slot {
  unsigned long long rmax;  // bit pattern of the largest (non-negative) tile rate
  unsigned long long n, tiles, events, counts[8];
};
// The FP64 total rate is summed without atomics, in a fixed order: every
// tile keeps its total (Lattice::tile_r), k_sweep_end sums NPART fixed chunks
// of tiles and then the NPART partials.  A rerun with
// the same seed therefore repeats the same windows.
constexpr int NPART = 2 * NSLOT;

// Device-resident run state (one per engine).
struct RunState {
  double tau;            // current window
  double clock;          // KMC time (FP64)
  double rtot;           // total rate estimate (isolated-atom rule)
  double rmax;           // largest tile rate of the last sweep
  double events_per_pass;
  int tau_policy;        // 0: tau = k / max tile rate; 1: tau = k * active tiles / total rate
  unsigned long long events;
  unsigned long long counts[8];
  unsigned long long sweeps;      // sweep counter (RNG stream position)
  unsigned long long sweeps_run;  // sweeps that advanced the clock
  long long n_mc;                 // MC particles at the end of the last sweep
  unsigned long long log_n;
  double max_time;                  // the run's limits: the sweep that reaches one stops the run
  unsigned long long max_events;
  int err;
  int err_site[3];
  int stop;
  // the laser-annealing build's crystal counts (la_variant): CountCrystal,
  // InitCountCrystal, the CountLiquid the rates read (refreshed per event in
  // a replay, per sweep in the parallel engine) and a sweep's changes
  int la_variant;
  long long cc[3], cinit[3], cl[3];
  unsigned long long dcc[3];
  unsigned long long desorbed[3];  // desorptions by coverage slot (CountCov)
  int final_sweep;                 // the window was shortened to end at max_time
  unsigned long long guard_exits;  // tile windows cut short by the per-window event cap
  int ever_lo, ever_hi;            // the first / last tile layer any of the run's sweeps could visit
  // the sweep's working sums, last: the host reads and writes only the
  // fields before them (RS_HEAD bytes)
  Slot slot[NSLOT];
};
constexpr size_t RS_HEAD = offsetof(RunState, slot);
// What the host asks of many engines' states at once.
struct RunHead {
  double clock, rtot;
  unsigned long long events, log_n;
  int err, stop, list_err;
  int ever_lo, ever_hi;
};
// A run state's start: `words` words to clear (the state, or its slots alone)
// by one small block, which takes the place of copies of 15 KB from the host.
__device__ inline void clear_words(unsigned int *w, int words) {
  for (int i = threadIdx.x; i < words; i += blockDim.x) w[i] = 0u;
}
__global__ void __launch_bounds__(256) k_state_new(RunState *st, double events_per_pass, double rtot,
                                                   unsigned long long *atoms, int *err) {
  clear_words((unsigned int *)st, (int)(sizeof(RunState) / 4));
  __syncthreads();
  if (threadIdx.x != 0) return;
  st->events_per_pass = events_per_pass;
  st->rtot = rtot;
  atoms[0] = atoms[1] = 0ull;
  *err = 0;
}
// The heads of n engines' states (ptr: their states, then their list errors).
__global__ void __launch_bounds__(64) k_heads(const void *const *ptr, int n, RunHead *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const RunState *const st = (const RunState *)ptr[i];
  RunHead h;
  h.clock = st->clock; h.rtot = st->rtot;
  h.events = st->events; h.log_n = st->log_n;
  h.err = st->err; h.stop = st->stop;
  h.list_err = *(const int *)ptr[n + i];
  h.ever_lo = st->ever_lo; h.ever_hi = st->ever_hi;
  out[i] = h;
}

struct PassParams {
  Lattice L;
  RunState *st;
  mskg_event *log;          // optional event log (valid serialisation of the run)
  unsigned long long log_cap;
  int ntz;
  int cap;
  uint32_t key0, key1;
  int colour;
  int rsum_chunk;           // tiles a chunk of the fixed-order tile sum (chunk_sum)
  // dependency-scheduled sweep: per-tile completion stamps, and sched[0]
  // the sweep's stamp, [1] queue head, [2] abort flag, [3] / [4] the first /
  // last tile layer holding candidates when the sweep starts
  unsigned int *done;
  unsigned int *sched;
};

// Between the lanes of a workgroup of one wave: what one has written the
// others read from here on.  The hardware takes a wave's LDS and its vector
// memory instructions in order, so nothing is waited for; a workgroup barrier
// waits until every store has returned, a round trip on every event (whole
// passes with it and without: CVD 95.0, 93.7 ms; 512^3 SiC 48.2, 47.6).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
  return v;
}
__device__ inline double wave_incl_scan(double v, int lane) {
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    double t = __shfl_up(v, off, WAVE);
    if (lane >= off) v += t;
  }
  return v;
}

// The value of v in another lane of the row (DPP, both halves of the
// double moved by the same control); lanes the control gives no source, and
// rows outside ROW_MASK, get 0.0.  Every lane of the wave must be active.
template <int CTRL, int ROW_MASK>
__device__ inline double dpp_take(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROW_MASK, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROW_MASK, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// Inclusive prefix sum over the wave's lanes in registers: prefix sums
// within each row of 16 lanes (row_shr 1, 2, 4, 8), then row 0's total into
// row 1 and row 2's into row 3 (row_bcast:15), then rows 0-1's total into
// rows 2 and 3 (row_bcast:31).  Every lane of the wave must be active.
__device__ inline double wave_incl_scan_dpp(double v) {
  v += dpp_take<0x111, 0xf>(v);  // row_shr:1
  v += dpp_take<0x112, 0xf>(v);  // row_shr:2
  v += dpp_take<0x114, 0xf>(v);  // row_shr:4
  v += dpp_take<0x118, 0xf>(v);  // row_shr:8
  v += dpp_take<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_take<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
// v of lane l (l the same in every lane).
__device__ inline double read_lane(double v, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// A pointer read from device memory (a replica's parameters, a descriptor) is
// a generic pointer to the compiler, and every access through it a flat
// instruction, which waits on both the vector-memory and the LDS counters.
// Every pointer of a lattice is to global memory; the rate tables and the
// geometry are constant while a kernel runs, so that reads of one value by
// the whole wave are scalar loads.  A round trip through the address space
// states that (through an integer: a direct cast there and back folds away).
template <typename T>
__device__ inline const T *as_constant(const T *p) {
  const __attribute__((address_space(4))) T *c = (const __attribute__((address_space(4))) T *)(uintptr_t)p;
  return (const T *)c;
}
__device__ inline void to_global(Lattice &L) {
  L.site = as_global(L.site); L.rate = as_global(L.rate); L.cls = as_global(L.cls);
  L.inlist = as_global(L.inlist); L.tl_idx = as_global(L.tl_idx); L.tl_n = as_global(L.tl_n);
  L.tl_own = as_global(L.tl_own); L.tile_r = as_global(L.tile_r); L.list_err = as_global(L.list_err);
  L.win = as_global(L.win); L.geo = as_constant(L.geo); L.tab = as_constant(L.tab); L.key = as_global(L.key);
  L.cl = as_global(L.cl);
}
__device__ inline void slot_add(RunState *st, int b, double r, unsigned long long n) {
  Slot &sl = st->slot[b & (NSLOT - 1)];
  if (!n) return;
  const unsigned long long rb = (unsigned long long)__double_as_longlong(r);
  if (rb > sl.rmax) atomicMax(&sl.rmax, rb);
  atomicAdd(&sl.n, n);
  atomicAdd(&sl.tiles, 1ull);
}

// The reference event's counter (RunState::counts).
__device__ inline int count_slot(int itrans) {
  return itrans <= 3 ? itrans - 1 : (itrans == 4 ? 3 : (itrans == 5 ? 4 : itrans - 1));
}

struct TileGeom {
  int tx, ty, tz, z0, nz, half;
  int64_t npt;
};
__device__ inline TileGeom tile_geom(int t, int T, int ntx, int nty, int lz) {
  TileGeom g;
  g.tx = t % ntx;
  g.ty = (t / ntx) % nty;
  g.tz = t / (ntx * nty);
  g.z0 = g.tz * T;
  g.nz = min(T, lz + 1 - g.z0);
  g.half = T / 2;
  g.npt = (int64_t)g.half * g.half * g.nz;
  return g;
}
// The point of a packed tile offset (tile_pack).
__device__ inline P3 tile_point(const Box &b, const TileGeom &g, int T, int k) {
  P3 p;
  p.z = g.z0 + (k >> 14);
  const int par = p.z & 1;
  p.x = g.tx * T + 2 * (k & 127) + par;
  p.y = g.ty * T + 2 * ((k >> 7) & 127) + par;
  p.i = pidx(b, p.x, p.y, p.z);
  return p;
}
// The packed offset of the k-th point of a tile in (z, y, x) order.
__device__ inline int tile_nth(const TileGeom &g, int k) {
  const int pp = g.half * g.half;
  const int zl = k / pp, r = k - zl * pp;
  const int j = r / g.half, i = r - j * g.half;
  return (zl << 14) | (j << 7) | i;
}
// The packed offset of p in tile g, -1 when p is outside the tile.
__device__ inline int tile_local(const TileGeom &g, int T, const P3 &p) {
  if (p.i < 0) return -1;
  const int xl = p.x - g.tx * T, yl = p.y - g.ty * T, zl = p.z - g.z0;
  if ((unsigned)xl >= (unsigned)T || (unsigned)yl >= (unsigned)T || (unsigned)zl >= (unsigned)g.nz) return -1;
  return tile_pack(zl, yl, xl);
}

// ---- rate-update sweep ----------------------------------------------------
// Every point: an MC particle is an empty or coverage site with coordination
// 1..3 or an atom with coordination <= 3 (Get_Prob.f:54-331 is evaluated for
// it); everything else gets class 0.
// With atoms_only, only atoms of coordination 1..3 are re-evaluated and every
// other point keeps its rate (used after the device slab builder, whose
// atoms need the second-neighbour factor).
//
// Each thread takes four consecutive points: four 16-byte record loads in
// flight, one 16-byte store of the rates and one 4-byte store of the
// classes.  Nearly every point is not an MC particle (a few per cent of the
// stored points are), so the Get_Prob branch is rare.
// Whether a record is an MC particle's; keep: atoms_only leaves the point alone.
__device__ inline bool sweep_mc(uint32_t w, int atoms_only, bool &keep) {
  const int kind = w & 7, coor = (w >> 3) & 7;
  keep = atoms_only && !(kind_species(kind) && coor >= 1 && coor <= 3);
  return !keep && ((kind == KIND_EMPTY && coor >= 1 && coor <= 3) || (kind >= KIND_COV0 && coor <= 3) ||
                   (kind_species(kind) && coor <= 3));
}

// LA, COV: the rate model's laser-annealing and coverage branches are compiled in.
// Four consecutive points from p0, or the points p0..n-1 at the end.  One
// instance of Get_Prob: the group's MC particles are taken in turn and their
// records read again (from the cache), so that the stream itself holds few
// registers -- 44 with 7 waves per SIMD, against 128 and 4 with Get_Prob
// inlined for each of the four records.
template <bool LA, bool COV>
__device__ inline void sweep_group(const Lattice &L, double rtot, int *err, int atoms_only, int64_t p0, int64_t n) {
  const int m = p0 + 4 <= n ? 4 : (int)(n - p0);
  uint32_t w[4];
  if (m == 4) {
    Rec sp[4];
    for (int k = 0; k < 4; k++) sp[k] = load_rec(L, p0 + k);
    for (int k = 0; k < 4; k++) w[k] = sp[k].w;
  } else {
    for (int k = 0; k < 4; k++) w[k] = k < m ? load_rec(L, p0 + k).w : 0u;
  }
  float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  uint32_t c = 0;
  unsigned mc = 0, kept = 0;
  for (int k = 0; k < 4; k++) {
    bool keep;
    mc |= sweep_mc(w[k], atoms_only, keep) && k < m ? 1u << k : 0u;
    kept |= keep ? 1u << k : 0u;
    if (L.key && !keep && k < m) L.key[p0 + k] = -1;
  }
#pragma unroll 1
  for (; mc; mc &= mc - 1u) {
    const int k = __ffs((int)mc) - 1;
    P3 pt;
    pt.i = p0 + k;
    pxyz(L.box, pt.i, pt.x, pt.y, pt.z);
    int e = ERR_NONE, cls = 0, key = -1;
    double rd = 0.0;
    get_prob<LA, COV>(L, rtot, pt, load_rec(L, pt.i), cls, rd, e, key);
    if (e) atomicExch(err, e);
    const float rf = cls ? (float)rd : 0.0f;
    if (k == 0) r.x = rf;
    if (k == 1) r.y = rf;
    if (k == 2) r.z = rf;
    if (k == 3) r.w = rf;
    c |= (uint32_t)cls << (8 * k);
    if (L.key && cls) L.key[pt.i] = key;
  }
  if (m == 4 && !kept) {
    *(float4 *)(L.rate + p0) = r;
    *(uint32_t *)(L.cls + p0) = c;
  } else {
    for (int k = 0; k < 4; k++)
      if (k < m && !((kept >> k) & 1u)) {
        L.rate[p0 + k] = k == 0 ? r.x : (k == 1 ? r.y : (k == 2 ? r.z : r.w));
        L.cls[p0 + k] = (uint8_t)(c >> (8 * k));
      }
  }
}

template <bool LA, bool COV>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_rate_sweep(Lattice L, const double *rtot_at, int *err, int atoms_only) {
  L.tab = as_constant(L.tab);
  const double rtot = rtot_at ? *rtot_at : 0.0;
  const int64_t n = L.box.npts;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x * 4;
  for (int64_t p0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; p0 < n; p0 += stride)
    sweep_group<LA, COV>(L, rtot, err, atoms_only, p0, n);
}

// The same over the points [first, end) of the stored order (first a
// multiple of 4), in groups of four counted in 32 bits (the largest lattice
// holds fewer than 2^31 groups).
template <bool LA, bool COV>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_rate_sweep_range(Lattice L, const double *rtot_at, int *err, int atoms_only, int64_t first, int64_t end) {
  L.tab = as_constant(L.tab);
  const double rtot = rtot_at ? *rtot_at : 0.0;
  const int g_first = (int)(first >> 2), g_end = (int)((end + 3) >> 2);
  const int gstride = gridDim.x * blockDim.x;
  for (int g = g_first + blockIdx.x * blockDim.x + threadIdx.x; g < g_end; g += gstride)
    sweep_group<LA, COV>(L, rtot, err, atoms_only, (int64_t)g * 4, end);
}

// Class and rate of given sites.  Few sites are asked for of a large lattice,
// so they are gathered here: what bounds it is the round trip of a launch and
// the copies of 20 bytes a site (the host read every point's 5 bytes for it:
// 16384 sites of 768x768x384, 67.7 ms, now 0.2).  bad: the first site that is
// no lattice point.
__global__ void __launch_bounds__(256) k_site_rates(Lattice L, int64_t n, const int32_t *xyz, int32_t *cls,
                                                    float *rate, unsigned int *bad) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t p = pidx_checked(L.box, xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]);
  if (p < 0) {
    atomicMin(bad, (unsigned int)i);
    return;
  }
  cls[i] = L.cls[p];
  rate[i] = L.rate[p];
}

// ---- event-log replay -------------------------------------------------------
template <bool LA, bool COV>
__global__ void __launch_bounds__(WAVE) k_replay(Lattice L, const mskg_event *log, int64_t n, int clock_mode,
                                                 RunState *st) {
  __shared__ TabLds tabs;
  const int lane = threadIdx.x;
  L.geo = as_constant(L.geo);
  L.tab = as_constant(L.tab);
  load_tables<LA>(*L.tab, tabs, lane);
  wave_sync();
  double clock = st->clock;
  int bad = 0;
  P3 s;
  s.x = s.y = s.z = 0;
  int64_t k = 0;
  for (; k < n; k++) {
    const mskg_event ev = log[k];
    s = at(L, __builtin_amdgcn_readfirstlane(ev.site[0]), __builtin_amdgcn_readfirstlane(ev.site[1]),
           __builtin_amdgcn_readfirstlane(ev.site[2]));
    const int itrans = __builtin_amdgcn_readfirstlane(ev.itrans);
    if (s.i < 0 || __builtin_amdgcn_readfirstlane((int)L.cls[s.i]) == 0) {
      bad = ERR_NOT_MC;
      break;
    }
    if (clock_mode == 0) clock = clock + 1.0 / ev.rtot;
    Choice ch;
    ch.arm = __builtin_amdgcn_readfirstlane(ev.arm);
    ch.u_arm = 0.0;
    EvOut o;
    execute<LA, COV>(L, tabs, ev.rtot, s, uniform_rec(load_rec(L, s.i)), itrans, ch, o, lane);
    bad = __builtin_amdgcn_readfirstlane(o.err);
    if (bad) break;
    if (lane == 0) {
      const int slot = count_slot(itrans);
      if (slot >= 0 && slot < 8) st->counts[slot]++;
      if (COV && itrans == 5 && o.species) st->desorbed[o.species - 1]++;
      if (LA && L.cl && o.species && itrans <= 4) {  // CountCrystal, then the next iteration's CountLiquid
        st->cc[o.species - 1] += itrans <= 3 ? 1 : -1;
        for (int q = 0; q < 3; q++) st->cl[q] = st->cinit[q] - st->cc[q];
      }
    }
    wave_sync();  // the next event reads this one's records, rates and counts
  }
  if (lane != 0) return;
  if (bad) {
    st->err = bad;
    st->err_site[0] = s.x; st->err_site[1] = s.y; st->err_site[2] = s.z;
    st->events = (unsigned long long)k;
  } else {
    st->events += (unsigned long long)n;
    st->clock = clock;
  }
}

// ---- synchronous sublattice -------------------------------------------------
// Build every tile's candidate list from the classes (after a state upload,
// a rate sweep or a replay).  One wave per tile, four of its points a lane in
// flight.  Points outside the planes [zlo, zhi] are no MC particles and have no
// list flag, which the caller knows of a slab (touched_planes): only the planes
// [zlo, zhi] are looked at, by the first `full` blocks, which take the tiles
// from t0 on that hold such planes; a thread of the others empties the list of
// a tile outside (a wave each for those cost 80 us at 83000 tiles).
// zeroed: no list flag is set anywhere, and none needs clearing (a store for
// every eight points of a tile's row, otherwise).
__global__ void __launch_bounds__(256) k_build_lists(Lattice L, int ntiles, int zlo, int zhi, int t0, int t1,
                                                     int full, int zeroed) {
  int lane = threadIdx.x & (WAVE - 1);
  if ((int)blockIdx.x >= full) {
    int q = ((int)blockIdx.x - full) * 256 + (int)threadIdx.x;
    if (q >= t0) q += t1 - t0;
    if (q >= ntiles) return;
    L.tl_n[q] = 0;
    L.tl_own[q] = 0;
    return;
  }
  int t = t0 + blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
  if (t >= t1) return;
  TileGeom g = tile_geom(t, L.tile, L.ntx, L.nty, L.box.lz);
  int n = 0;
  {
    const int pp = g.half * g.half;
    const int first = max(zlo - g.z0, 0) * pp, end = min(zhi + 1 - g.z0, g.nz) * pp;
    for (int k0 = first; k0 < end; k0 += 4 * WAVE) {
      int kp[4];
      int64_t pi[4];
      uint8_t c[4];
      for (int u = 0; u < 4; u++) {
        const int k = k0 + u * WAVE + lane;
        const bool in = k < end;
        kp[u] = tile_nth(g, in ? k : 0);
        pi[u] = tile_point(L.box, g, L.tile, kp[u]).i;
        c[u] = in ? L.cls[pi[u]] : (uint8_t)0;
        if (!in) pi[u] = -1;
      }
      for (int u = 0; u < 4; u++) {
        const bool on = c[u] != 0;
        if (pi[u] >= 0 && (on || !zeroed)) L.inlist[pi[u]] = on ? 1 : 0;
        const unsigned long long m = __ballot(on);
        const int slot = n + __popcll(m & ((1ull << lane) - 1ull));
        if (on) {
          if (slot < L.capg) L.tl_idx[(int64_t)t * L.capg + slot] = kp[u];
          else *L.list_err = ERR_TILE_LIST;
        }
        n += __popcll(m);
      }
    }
  }
  if (lane == 0) {
    L.tl_n[t] = n;
    L.tl_own[t] = min(n, L.capg);
  }
}

// Windows of tile layers from the lists: a block a layer (from layer l0 on),
// which finds the colours that hold any and widens their windows once.  (Every
// tile had widened its colour's itself: all of them at once, against windows
// still empty, 100 us of atomics on one word at 18000 tiles.)
__global__ void __launch_bounds__(1024) k_list_window(Lattice L, int l0) {
  __shared__ unsigned int found;
  const int tz = l0 + blockIdx.x, layer = L.ntx * L.nty;
  if (threadIdx.x == 0) found = 0u;
  __syncthreads();
  unsigned int mine = 0u;
  for (int i = threadIdx.x; i < layer; i += blockDim.x)
    if (L.tl_n[tz * layer + i] > 0) mine |= 1u << tile_colour(i % L.ntx, i / L.ntx, tz);
  for (int off = 32; off > 0; off >>= 1) mine |= __shfl_xor(mine, off, WAVE);
  if ((threadIdx.x & (WAVE - 1)) == 0 && mine) atomicOr(&found, mine);
  __syncthreads();
  if (threadIdx.x < 8 && ((found >> threadIdx.x) & 1u)) widen_window(L.win, threadIdx.x, tz);
}

// A run's start, by one block: empty windows, empty slots, the run's limits and
// a zero window tau in the state (k_sweep_end then sets the first).
__global__ void __launch_bounds__(256) k_run_start(RunState *st, int *win, int *list_err, int lists, int tau_policy,
                                                   double events_per_pass, double max_time,
                                                   unsigned long long max_events) {
  const int i = threadIdx.x;
  if (i < 32) win[i] = i & 1 ? -1 : 0x7fffffff;
  if (i == 32 && lists) *list_err = 0;
  clear_words((unsigned int *)st->slot, (int)(sizeof st->slot / 4));
  if (i != 0) return;
  st->tau = 0.0;
  st->stop = 0;
  st->final_sweep = 0;
  st->tau_policy = tau_policy;
  st->events_per_pass = events_per_pass;
  st->max_time = max_time;
  st->max_events = st->events + max_events;
  st->ever_lo = 0x7fffffff;
  st->ever_hi = -1;
}

// Rate total (without isolated atoms) and population of every tile's list; the
// tiles outside [t0, t1) have none (k_build_lists).
__global__ void __launch_bounds__(256) k_tile_rates(Lattice L, int ntiles, RunState *st, int t0, int t1, int full) {
  int lane = threadIdx.x & (WAVE - 1);
  if ((int)blockIdx.x >= full) {
    int q = ((int)blockIdx.x - full) * 256 + (int)threadIdx.x;
    if (q >= t0) q += t1 - t0;
    if (q < ntiles) L.tile_r[q] = 0.0;
    return;
  }
  int t = t0 + blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
  if (t >= t1) return;
  const int m = min(L.tl_n[t], L.capg);
  if (m <= 0) {  // most tiles of a box
    if (lane == 0) L.tile_r[t] = 0.0;
    return;
  }
  TileGeom g = tile_geom(t, L.tile, L.ntx, L.nty, L.box.lz);
  double acc = 0.0;
  int cnt = 0;
  for (int j = lane; j < m; j += WAVE) {
    P3 p = tile_point(L.box, g, L.tile, L.tl_idx[(int64_t)t * L.capg + j]);
    uint8_t c = L.cls[p.i];
    if (c) cnt++;
    if (c && c != CLS_ISOLATED) acc += (double)L.rate[p.i];
  }
  acc = wave_sum(acc);
  for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, WAVE);
  if (lane == 0) {
    L.tile_r[t] = cnt ? acc : 0.0;
    if (cnt) slot_add(st, t, acc, (unsigned long long)cnt);
  }
}

// Sorts lk/lr/lc[lo, hi) by offset (the offsets are distinct): up to 64
// entries by rank, each lane counting the smaller ones (a handful: the
// appends from other tiles between two passes), odd-even transposition rounds
// beyond.
__device__ inline void sort_by_offset(int32_t *lk, float *lr, uint8_t *lc, int lo, int hi, int lane) {
  const int m = hi - lo;
  if (m <= 1) return;
  if (m <= WAVE) {
    int key = 0, rank = 0;
    float r = 0.0f;
    uint8_t c = 0;
    if (lane < m) {
      key = lk[lo + lane];
      r = lr[lo + lane];
      c = lc[lo + lane];
    }
#pragma unroll 1
    for (int q = 0; q < m; q++) rank += __builtin_amdgcn_readlane(key, q) < key ? 1 : 0;
    wave_sync();
    if (lane < m) {
      lk[lo + rank] = key;
      lr[lo + rank] = r;
      lc[lo + rank] = c;
    }
    wave_sync();
    return;
  }
  for (int round = 0; round < m; round++) {
    for (int i = lo + 2 * lane + (round & 1); i + 1 < hi; i += 2 * WAVE)
      if (lk[i] > lk[i + 1]) {
        const int tk = lk[i];
        lk[i] = lk[i + 1];
        lk[i + 1] = tk;
        const float tr = lr[i];
        lr[i] = lr[i + 1];
        lr[i + 1] = tr;
        const uint8_t tc = lc[i];
        lc[i] = lc[i + 1];
        lc[i + 1] = tc;
      }
    wave_sync();
  }
}

// The sum of v over the wave, added as an exchange with the lane 32, 16, 8,
// 4, 2 and 1 apart adds it (every lane the same bits): the first two steps by
// lane swaps, the others by rotations within a row of 16, whose operands the
// steps before made periodic.
__device__ inline double swap_add(double v, bool rows) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
  unsigned l0, l1, h0, h1;
  if (rows) {
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    l0 = l[0]; l1 = l[1]; h0 = h[0]; h1 = h[1];
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    l0 = l[0]; l1 = l[1]; h0 = h[0]; h1 = h[1];
  }
  return __longlong_as_double((long long)(((unsigned long long)h0 << 32) | l0)) +
         __longlong_as_double((long long)(((unsigned long long)h1 << 32) | l1));
}
__device__ inline double wave_sum_dpp(double v) {
  v = swap_add(v, true);
  v = swap_add(v, false);
  v += dpp_take<0x128, 0xf>(v);  // row_ror:8
  v += dpp_take<0x124, 0xf>(v);  // row_ror:4
  v += dpp_take<0x122, 0xf>(v);  // row_ror:2
  v += dpp_take<0x121, 0xf>(v);  // row_ror:1
  return v;
}

// The parameters of a kernel whose only argument they are, in its argument segment.
__device__ inline const PassParams *kernel_params() {
  return as_constant((const PassParams *)__builtin_amdgcn_kernarg_segment_ptr());
}
// The fields an event needs of the lattice in pp; the others are read where
// they are used.
__device__ inline Lattice event_part(const PassParams *pp) {
  Lattice L = pp->L;
  to_global(L);
  L.cold = &pp->L;
  return L;
}

// One tile's share of a colour pass: its candidate list into LDS, rejection-
// free KMC inside the tile for the window tau, the list back.  Returns the
// error that ends the wave's work (0: none).  The selected site, its record
// and the event type are kept in scalar registers: the event's addresses and
// branches are then scalar too.
// pp: the parameters in constant memory, read where they are needed (read_here);
// L: the fields an event needs.  fresh: the wave's tables are to be loaded.
template <bool LA, bool COV>
__device__ inline int pass_tile(const PassParams *pp, Lattice &L, RunState *st, const double tau, const int t,
                                const int colour, TabLds &tabs, const bool fresh, unsigned char *smem,
                                const int lane) {
  const int cap = pp->cap;
  int32_t *const lk = (int32_t *)smem;        // tile-local point offsets
  float *const lr = (float *)(lk + cap);      // rates
  uint8_t *const lc = (uint8_t *)(lr + cap);  // classes
  TileGeom g;
  int n = 0;
  unsigned long long sweeps;
  double rtot;
  {
  const PassParams &P = *read_here(pp);
  int32_t *const tl_n = as_global(P.L.tl_n);
  const int32_t *const idx = as_global(P.L.tl_idx) + (int64_t)t * P.L.capg;
  uint8_t *const inlist = as_global(P.L.inlist);
  // The tile's first loads leave together, in one round trip: its list
  // length and own count, the first WAVE list entries (read whatever the
  // length; a lane uses its entry only below it, and the index stays in the
  // tile's list storage), and the run state the window needs.
  TabRegs tr;
  if (fresh) fetch_tables<LA>(*L.tab, tr, lane);
  const int n_raw = tl_n[t], own_raw = as_global(P.L.tl_own)[t];
  const int k_first = idx[min(lane, P.L.capg - 1)];
  rtot = st->rtot;
  sweeps = st->sweeps;
  if (fresh) put_tables<LA>(tr, tabs, lane);
  const int n_in = __builtin_amdgcn_readfirstlane(n_raw), own = __builtin_amdgcn_readfirstlane(own_raw);
  if (n_in == 0) return 0;
  g = tile_geom(t, L.tile, P.L.ntx, P.L.nty, L.box.lz);
  L.cur_tile = t;
  L.cx = g.tx * L.tile;
  L.cy = g.ty * L.tile;
  L.cz = g.z0;

  // 1. the tile's candidate list -> LDS, dropping entries no longer active;
  // the entries other tiles appended since the tile's last pass (an order
  // that depends on timing) are then sorted by offset
  const int m_in = min(n_in, P.L.capg);
  int nh = 0;
  for (int j0 = 0; j0 < m_in; j0 += WAVE) {
    int j = j0 + lane;
    uint8_t c = 0;
    float r = 0.0f;
    int k = 0;
    if (j < m_in) {
      k = j0 == 0 ? k_first : idx[j];
      P3 p = tile_point(L.box, g, L.tile, k);
      // class and rate in one round trip (the rate is used only with a class)
      c = L.cls[p.i];
      r = L.rate[p.i];
      if (!c) inlist[p.i] = 0;
    }
    unsigned long long m = __ballot(c != 0);
    int slot = n + __popcll(m & ((1ull << lane) - 1ull));
    if (c && slot < cap) {
      lk[slot] = k;
      lr[slot] = r;
      lc[slot] = c;
    }
    n += __popcll(m);
    nh += __popcll(__ballot(c != 0 && j < own));
  }
  if (n > cap) {
    if (lane == 0) {
      st->err = ERR_CAPACITY;
      P3 p = tile_point(L.box, g, L.tile, 0);
      st->err_site[0] = p.x; st->err_site[1] = p.y; st->err_site[2] = p.z;
    }
    return ERR_CAPACITY;
  }
  wave_sync();
  sort_by_offset(lk, lr, lc, nh, n, lane);
  }

  // 2. rejection-free KMC inside the tile for the window tau
  double tloc = 0.0;
  unsigned int nev = 0;
  unsigned int my_cnt = 0, my_des = 0;  // lane l + 4: events of counter l; lane l: desorptions of coverage slot l + 1
  int my_dcc = 0;                       // lane l: change of CountCrystal(l + 1) (laser-annealing build's form)
  U4 d;              // lane l: the Philox block of draw 64 b + l, b the current batch
  double wait = 0.0;  // ... and -ln of its first uniform
  int err = 0;
  const bool logging = pp->log != nullptr;
  pin(L.site); pin(L.rate); pin(L.cls);
  // every wave ends its pass: the window tau bounds the expected number of
  // events, and this cap bounds the worst case (a window cut short by it is
  // counted in RunState::guard_exits and reported by the run)
  int guard = 0;
  for (; guard < PASS_EVENT_CAP; guard++) {
    pin(L.box);
    // one Philox block per event: waiting time, selection, event type and
    // stacking choice, 32 random bits each (the reference's ran3 has fewer).
    // The block depends on the draw's number only, so the wave makes 64 of
    // them, and their FP64 logarithms, at once.
    const int dl = guard & (WAVE - 1);
    if (dl == 0) {
      U4 ctr;
      ctr.x = (uint32_t)t;
      ctr.y = (uint32_t)sweeps;
      ctr.z = (uint32_t)(sweeps >> 32) ^ ((uint32_t)colour << 29);
      ctr.w = (uint32_t)(guard + lane);
      const PassParams &P = *read_here(pp);
      d = philox4x32_10(ctr, P.key0, P.key1);
      wait = -log(u01_32(d.x));
    }
    // lane-major order: lane l owns entries l, l + 64, ...; one wave scan of
    // the lanes' partial sums gives the total and the lane that holds the pick
    double part = 0.0;
    for (int j = lane; j < n; j += WAVE) part += (double)lr[j];
    const double inc = wave_incl_scan_dpp(part);
    const double R = read_lane(inc, WAVE - 1);
    if (!(R > 0.0)) break;
    const double target = u01_32((uint32_t)__builtin_amdgcn_readlane((int)d.y, dl)) * R;
    // the first lane whose inclusive prefix exceeds target (the last lane
    // with a rate when rounding leaves target at the top end), then the
    // first of its entries whose running prefix exceeds target
    const unsigned long long nzl = __ballot(part > 0.0);
    const unsigned long long hit = __ballot(part > 0.0 && inc > target);
    if (!nzl) break;
    const int owner = hit ? __ffsll((long long)hit) - 1 : 63 - __clzll((long long)nzl);
    int sel = owner;  // up to 64 entries: the lane's only one
    if (n > WAVE) {
      sel = -1;
      if (lane == owner) {
        double acc = inc - part;
        int last = -1;
        for (int j = lane; j < n; j += WAVE) {
          const double v = (double)lr[j];
          if (v > 0.0) {
            last = j;
            acc += v;
            if (acc > target) {
              sel = j;
              break;
            }
          }
        }
        if (sel < 0) sel = last;
      }
      sel = __builtin_amdgcn_readlane(sel, owner);
      if (sel < 0) break;
    }
    const P3 s = tile_point(L.box, g, L.tile, __builtin_amdgcn_readfirstlane(lk[sel]));
    // the site's record is on its way while the waiting time is taken: the
    // event may lie beyond the window
    const Rec srec_v = load_rec(L, s.i);
    const double dt = read_lane(wait, dl) / R;  // FP64 waiting time
    if (tloc + dt > tau) break;
    tloc += dt;
    const Rec srec = uniform_rec(srec_v);
    const int cls = __builtin_amdgcn_readfirstlane((int)lc[sel]);
    Choice ch;
    ch.arm = -1;
    ch.u_arm = u01_32((uint32_t)__builtin_amdgcn_readlane((int)d.w, dl));
    const int coor0 = r_coor(srec);
    const int itrans = __builtin_amdgcn_readfirstlane(la_swap<LA>(
        L, pick_itrans<LA, COV>(L, TabEv<COV>{*L.tab, tabs}, coor0, r_temp(srec), cls,
                                u01_32((uint32_t)__builtin_amdgcn_readlane((int)d.z, dl)))));
    EvOut o;
    execute<LA, COV>(L, tabs, rtot, s, srec, itrans, ch, o, lane);
    err = __builtin_amdgcn_readfirstlane(o.err);
    if (logging && lane == 0) {
      const PassParams &P = *read_here(pp);
      mskg_event *const out = as_global(P.log);
      const unsigned long long li = atomicAdd(&st->log_n, 1ull);
      if (li < P.log_cap) {
        mskg_event ev;
        ev.iter = (int64_t)li + 1;
        ev.site[0] = s.x; ev.site[1] = s.y; ev.site[2] = s.z;
        ev.itrans = itrans;
        ev.arm = o.arm;
        ev.coor = coor0;
        ev.rtot = rtot;
        ev.time = st->clock + tloc;
        out[li] = ev;
      }
    }
    if (lane == count_slot(itrans) + 4) my_cnt++;
    if (LA && o.species && itrans <= 4 && lane == o.species - 1) my_dcc += itrans <= 3 ? 1 : -1;
    if (COV && itrans == 5 && o.species && lane == o.species - 1) my_des++;
    nev++;
    if (err) break;
    // refresh the on-chip list with the touched points' new rates, which
    // execute() left a lane each: each such lane inside the tile looks its
    // offset up in the list, four entries a read (the offsets are distinct;
    // what lies behind the list's end is not taken)
    const int kl = o.set ? tile_local(g, L.tile, o.p) : -1;
    float tr = o.rate;
    int tc = o.cls;
    int found = -1;
    for (int j0 = (n - 1) & ~3; j0 >= 0; j0 -= 4) {
      const int4 v = *(const int4 *)(lk + j0);
      found = v.w == kl ? j0 + 3 : found;
      found = v.z == kl ? j0 + 2 : found;
      found = v.y == kl ? j0 + 1 : found;
      found = v.x == kl ? j0 : found;
    }
    if (found >= n) found = -1;
    // repeated list entries: the rates are in memory, and a point touched
    // twice joins the list once
    bool dup = false;
    if (__ballot(o.set == 2)) {
      if (o.set == 2 && kl >= 0) {
        tr = L.rate[o.p.i];
        tc = L.cls[o.p.i];
      }
      // the loads are waited for here, in this seldom taken branch: where it
      // joins the others they would make every event wait for its stores
      asm volatile("" : "+v"(tr), "+v"(tc));
      for (unsigned long long tm = __ballot(kl >= 0); tm; tm &= tm - 1ull) {
        const int q = __ffsll((long long)tm) - 1;
        if (q < lane && __builtin_amdgcn_readlane(kl, q) == kl) dup = true;
      }
    }
    // ... updates in place, and appends the new MC particles (first
    // occurrence of each) after the list in touched order
    bool app = false;
    if (kl >= 0) {
      if (found >= 0) {
        lr[found] = tr;
        lc[found] = (uint8_t)tc;
      } else if (tc) {
        app = !dup;
      }
    }
    const unsigned long long am = __ballot(app);
    if (am) {
      if (app) {
        const int slot = n + __popcll(am & ((1ull << lane) - 1ull));
        if (slot < cap) {
          lk[slot] = kl;
          lr[slot] = tr;
          lc[slot] = (uint8_t)tc;
        }
      }
      if (n + __popcll(am) > cap) {  // the list keeps its first cap entries
        err = ERR_CAPACITY;
        break;
      }
      n += __popcll(am);
    }
    wave_sync();  // the next event reads this one's records and list entries
  }
  if (guard >= PASS_EVENT_CAP && lane == 0) atomicAdd(&st->guard_exits, 1ull);
  // 3. write the list back (active entries only), tile totals, counters
  const PassParams &P = *read_here(pp);
  // the values the counters are compared with before an atomic (they change
  // seldom), on their way with the list
  Slot &sl = st->slot[t & (NSLOT - 1)];
  int *const win = as_global(P.L.win) + 4 * colour;
  const unsigned long long rmax = sl.rmax;
  const int win_lo = win[2], win_hi = win[3];
  int32_t *const idx = as_global(P.L.tl_idx) + (int64_t)t * P.L.capg;
  uint8_t *const inlist = as_global(P.L.inlist);
  double part = 0.0;
  int nout = 0;
  for (int j0 = 0; j0 < n; j0 += WAVE) {
    int j = j0 + lane;
    bool keep = j < n && lc[j] != 0;
    if (j < n) inlist[tile_point(L.box, g, L.tile, lk[j]).i] = keep ? 1 : 0;
    if (keep && lc[j] != CLS_ISOLATED) part += (double)lr[j];
    unsigned long long m = __ballot(keep);
    int slot = nout + __popcll(m & ((1ull << lane) - 1ull));
    if (keep) idx[slot] = lk[j];
    nout += __popcll(m);
  }
  const double R = wave_sum_dpp(part);
  {
    // the slot's sums in one atomic instruction, a lane each: n, tiles, events, counts
    static_assert(offsetof(Slot, n) == 8 && offsetof(Slot, tiles) == 16 && offsetof(Slot, events) == 24 &&
                  offsetof(Slot, counts) == 32, "Slot's words by lane");
    const unsigned int v = lane == 1 ? (unsigned)nout : (lane == 2 ? (nout ? 1u : 0u) : (lane == 3 ? nev : my_cnt));
    if (lane >= 1 && lane < 12 && v) atomicAdd(&sl.rmax + lane, (unsigned long long)v);
  }
  if (LA && L.cl && my_dcc) atomicAdd(&st->dcc[lane], (unsigned long long)(long long)my_dcc);
  if (COV && my_des) atomicAdd(&st->desorbed[lane], (unsigned long long)my_des);
  if (lane == 0) {
    as_global(P.L.tl_n)[t] = nout;
    as_global(P.L.tl_own)[t] = nout;
    as_global(P.L.tile_r)[t] = R;
    if (nout) {
      const unsigned long long rb = (unsigned long long)__double_as_longlong(R);
      if (rb > rmax) atomicMax(&sl.rmax, rb);
      if (g.tz < win_lo) atomic_min_i32(&win[2], g.tz);
      if (g.tz > win_hi) atomic_max_i32(&win[3], g.tz);
    }
    if (err) {
      st->err = err;
      P3 p = tile_point(L.box, g, L.tile, 0);
      st->err_site[0] = p.x; st->err_site[1] = p.y; st->err_site[2] = p.z;
    }
  }
  if (err) return err;
  wave_sync();
  return 0;
}

// The tiles of `colour` in the colour's window of tile layers [lo, hi] that
// hold candidates (win[4c], win[4c+1], fixed during a sweep): their number, and
// zfirst, the lowest of those layers with the colour's layer parity.
__device__ inline int colour_tiles(const Lattice &L, int ntz, int colour, int lo, int hi, int &zfirst) {
  const int c2 = (colour >> 2) & 1;
  const int zlo = max(lo, 0), zhi = min(hi, ntz - 1);
  zfirst = 0;
  if (zlo > zhi) return 0;  // no tile of this colour holds candidates
  zfirst = zlo + ((c2 - zlo) & 1);
  const int nlayers = zfirst <= zhi ? (zhi - zfirst) / 2 + 1 : 0;
  return nlayers * (L.ntx / 2) * (L.nty / 2);
}
// The wi-th of those tiles: layer by layer, y then x.
__device__ inline int colour_tile(const Lattice &L, int colour, int zfirst, int wi) {
  const int c0 = colour & 1, c1 = (colour >> 1) & 1;
  const int hx = L.ntx / 2, per_layer = hx * (L.nty / 2);
  const int layer = wi / per_layer, rr = wi - layer * per_layer;
  return ((zfirst + 2 * layer) * L.nty + 2 * (rr / hx) + c1) * L.ntx + 2 * (rr % hx) + c0;
}

// One colour pass: the tiles of `colour` in the window of tile layers that
// hold candidates, each workgroup (one wave) striding over them.  Three
// waves per SIMD (157 VGPRs, no spills): 3072 tiles in flight on 256 CUs.
// Measured on 8e6 events at 512^3 SiC (before the scalar registers were
// relieved): 69.1 ms; with two waves 74.9, with four (128 VGPRs, spilled) 76.0.
// The laser-annealing kernels hold exp and erf: two waves (223 VGPRs), 55.3 ms
// on two exchanges of 3e4 events at 264x264x384, against 60.4 with three (184
// bytes a lane spilled) and 79.4 with four (before the exponentials of the
// deposition rates went to the tables).
template <bool LA, bool COV>
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(LA ? 2 : 3, LA ? 2 : 3))) k_pass(PassParams P) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ TabLds tabs;
  const int lane = threadIdx.x;
  const PassParams *const pp = kernel_params();
  RunState *const st = P.st;
  // the run state and the colour's window in one round trip
  const double tau = st->tau;
  const int idle = st->err | st->stop, lo = P.L.win[4 * P.colour], hi = P.L.win[4 * P.colour + 1];
  if (!(tau > 0.0) || idle) return;
  int zfirst;
  const int nwin = colour_tiles(P.L, P.ntz, P.colour, lo, hi, zfirst);
  Lattice L = event_part(pp);
  bool fresh = true;
  for (int wi = blockIdx.x; wi < nwin; wi += gridDim.x) {
    const int t = colour_tile(P.L, P.colour, zfirst, wi);
    if (pass_tile<LA, COV>(pp, L, st, tau, t, P.colour, tabs, fresh, smem, lane)) return;
    fresh = false;
  }
}

// ---- a sweep scheduled by tile dependencies ------------------------------
// The eight colour passes of a sweep in one launch without a barrier
// between colours: a tile's pass starts as soon as its neighbour tiles of
// the lower colours have finished theirs in this sweep (tiles of the higher
// colours finished theirs in the previous launch).  A tile's events read
// and write only its own tile and the 24-unit shell of its 26 neighbour
// tiles, so every tile sees exactly the state it sees with a barrier after
// each colour, and the sweep's result -- lattice, lists, totals, random
// streams -- is the same bit for bit.  Tiles that do not neighbour each
// other (same colour, or farther apart) run concurrently as before.
//
// Work distribution: a queue of the sweep's tiles in colour order; every
// wave takes the next entry with one atomic, waits for the entry's lower-
// colour neighbours, runs the tile and publishes its completion.  A wave
// only waits on entries of lower colours, which were taken earlier by waves
// that are running, so the queue always drains.  The completion flag of a
// tile is the sweep's stamp (sched[0], advanced by k_sweep_end), stored
// with agent-scope release after the tile's writes; a waiting wave loads it
// at agent scope and takes an agent-scope acquire before it reads the
// neighbours' records, so the tiles' records travel between XCDs.  The release
// writes the XCD's L2 back and the acquire invalidates it for all of its waves,
// which costs more than the barriers they replace (512^3 SiC: 39.8 against 75.3
// M events/s).
//
// The same sweep on one XCD (LOCAL): the waves of one XCD, whichever the
// first wave to start is on, take all of the queue, and the others leave.
// They share its L2, so that a tile's writes are released when the L2 has them
// (its stores have returned), without the write-back.  The acquire is the same
// agent-scope invalidate (a workgroup's would do for the L1, but outside
// threadgroup-split mode its loads and invalidates leave other CUs' writes
// unseen); a few dozen waves can afford its refetches.
// What bounds a sweep of a small lattice is the chain of its slowest tiles,
// a few events of about 5 us each a colour, with a launch of 4.5 us after
// every colour, whether it has tiles or not: a film in one tile layer has
// tiles in four of the eight.

// The tile layers of colours with layer parity `odd` that a sweep's queue
// holds, for candidates in layers [zlo, zhi] when the sweep starts: the
// even colours (0-3) run first, so their layers outside the window stay
// empty until they have run; the odd colours (4-7) run after the even
// layers next to them, whose events can enlist points one layer out.
__device__ inline void queue_layers(int zlo, int zhi, int odd, int ntz, int &first, int &count) {
  const int lo = max(odd ? zlo - 1 : zlo, 0), hi = min(odd ? zhi + 1 : zhi, ntz - 1);
  first = lo + ((odd - lo) & 1);
  count = first <= hi ? (hi - first) / 2 + 1 : 0;
}

// A wave polls at most this often for its neighbour tiles (a preempted wave does
// not poll); the run then stops with ERR_SCHED instead of hanging.  The longest
// wait of a correct run is the chain of the seven colours below a tile's, each
// tile with PASS_EVENT_CAP events in its window.  An event takes 5 us in a short
// list, 38 in one of 1460 entries and about 80 in one of 3400 (laser annealing,
// whose events are the slowest; a list holds at most 6144), and a poll 0.5 us at
// least: 512 polls an event are 256 us or more, two minutes in all.  (With 2^22
// polls, 2.2 s, a laser-annealing run of 48-wide tiles whose windows reach the
// cap stopped with the error, where the colour passes finish.)
constexpr int EVENT_POLLS = 512;
constexpr int SCHED_POLLS = 7 * PASS_EVENT_CAP * EVENT_POLLS;

// A word another CU of the same XCD has written, read at agent scope (past the
// L1), the load and its wait in one block.
__device__ inline unsigned int load_xcd(const unsigned int *p) {
  unsigned int v;
  asm volatile("global_load_dword %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(v) : "v"(p) : "memory");
  return v;
}
template <bool LOCAL>
__device__ inline unsigned int load_flag(const unsigned int *p) {
  return LOCAL ? load_xcd(p) : __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool LOCAL>
__device__ inline void sweep_acquire() {
  if (LOCAL) asm volatile("buffer_inv sc1" ::: "memory");
  else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}
template <bool LOCAL>
__device__ inline void sweep_release() {
  if (LOCAL) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
}
// Is this wave on the XCD that runs the sweep `stamp`?  The first wave to ask
// settles it (sched[5]: 4 bits of XCD below 28 of the stamp), so at least one
// wave runs, and any number of waves drains the queue.
__device__ inline bool on_sweeps_xcd(unsigned int *word, unsigned int stamp) {
  const unsigned int xcc = (unsigned int)__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 15u;  // HW_REG_XCC_ID, bits 0..3
  const unsigned int mine = (stamp << 4) | xcc;
  unsigned int v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (__builtin_amdgcn_readfirstlane((int)((v ^ mine) >> 4)) != 0) {  // an earlier sweep's
    unsigned int seen = v;
    if (threadIdx.x == 0 && __hip_atomic_compare_exchange_strong(word, &seen, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT))
      seen = mine;
    v = seen;
  }
  return __builtin_amdgcn_readfirstlane((int)v) == (int)mine;
}

template <bool LA, bool COV, bool LOCAL>
__device__ inline void sweep_tiles(const PassParams &P, const PassParams *const pp, TabLds &tabs, unsigned char *smem) {
  const int lane = threadIdx.x;
  if (LOCAL && !on_sweeps_xcd(P.sched + 5, P.sched[0])) return;
  Lattice L = event_part(pp);
  RunState *st = P.st;
  const double tau = st->tau;
  if (!(tau > 0.0) || st->err || st->stop) return;
  // the window as the sweep starts (L.win's first words widen during it)
  const int zlo = (int)P.sched[3], zhi = (int)P.sched[4];
  if (zlo > zhi) return;
  load_tables<LA>(*L.tab, tabs, lane);
  int first[2], count[2];
  queue_layers(zlo, zhi, 0, P.ntz, first[0], count[0]);
  queue_layers(zlo, zhi, 1, P.ntz, first[1], count[1]);
  const int hx = L.ntx / 2, per_layer = hx * (L.nty / 2);
  const int per_even = count[0] * per_layer, per_odd = count[1] * per_layer;
  const int total = 4 * (per_even + per_odd);
  const unsigned int stamp = P.sched[0];
  unsigned int *const head = P.sched + 1;
  // neighbour k of 26 (lanes 0..25): offsets -1..1 along each axis
  const int kk = lane + (lane >= 13 ? 1 : 0);
  const int ndx = kk % 3 - 1, ndy = (kk / 3) % 3 - 1, ndz = kk / 9 - 1;
  const int nflip = (ndx & 1) | ((ndy & 1) << 1) | ((ndz & 1) << 2);
  // Every decision of this loop is wave-uniform by construction (scalar
  // values from readfirstlane / ballot) and no memory access sits under a
  // lane-dependent branch: the compiler may otherwise restructure the loop
  // so that lane 0, which would own such accesses, runs a different
  // iteration than the other lanes.
  for (;;) {
    // the next entry: every lane adds 1 (one atomic of 64 for the wave), so
    // the head counts entries in units of 64
    const unsigned int took = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int q = __builtin_amdgcn_readfirstlane((int)(took >> 6));
    if (q >= total) break;
    // entry -> colour, tile
    int colour, wi;
    if (q < 4 * per_even) {
      colour = q / per_even;
      wi = q - colour * per_even;
    } else {
      const int r = q - 4 * per_even;
      colour = 4 + r / per_odd;
      wi = r - (colour - 4) * per_odd;
    }
    const int odd = colour >> 2;
    const int layer = wi / per_layer, rr = wi - layer * per_layer;
    const int tz = first[odd] + 2 * layer, ty = 2 * (rr / hx) + ((colour >> 1) & 1), tx = 2 * (rr % hx) + (colour & 1);
    const int t = (tz * L.nty + ty) * L.ntx + tx;
    // the neighbours of lower colours that this sweep's queue holds
    bool dep = false;
    int n = 0;
    if (lane < 26) {
      const int nc = colour ^ nflip, nz = tz + ndz;
      if (nc < colour && nz >= 0 && nz < P.ntz) {
        const int nodd = nc >> 2;
        const int rel = nz - first[nodd];
        if (rel >= 0 && rel < 2 * count[nodd]) {
          int nx = tx + ndx, ny = ty + ndy;
          nx += nx < 0 ? L.ntx : (nx >= L.ntx ? -L.ntx : 0);
          ny += ny < 0 ? L.nty : (ny >= L.nty ? -L.nty : 0);
          n = (nz * L.nty + ny) * L.ntx + nx;
          dep = true;
        }
      }
    }
    // lane 26 reads the abort flag with them; a lane without a neighbour reads its own tile's
    const unsigned int *const flag = lane == 26 ? P.sched + 2 : P.done + (dep ? n : t);
    bool abort = false;
    if (__ballot(dep) != 0ull) {
      for (int polls = 0;; polls++) {
        const unsigned int f = load_flag<LOCAL>(flag);
        if (__ballot(dep && f != stamp) == 0ull) break;
        const bool late = polls >= SCHED_POLLS;
        if (__builtin_amdgcn_readlane((int)f, 26) != 0 || late) {
          if (late) {  // every lane stores the same values
            __hip_atomic_store(&P.sched[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            atomicCAS(&st->err, 0, ERR_SCHED);
          }
          abort = true;
          break;
        }
        // a waiting wave's polls delay the tiles' own loads: with more than 64 of
        // them about 1 us between two polls (40 x 64 cycles), else 0.3 us (edge
        // 384: 6.0 against 6.1 ms, edge 96: 4.4 against 4.4)
        if (LOCAL && gridDim.x > 8 * 64) __builtin_amdgcn_s_sleep(40);
        else __builtin_amdgcn_s_sleep(LOCAL ? 12 : 2);
      }
    }
    // many tiles of the queue are empty: their length (and the run's error)
    // alone is read past the caches, and only a tile with candidates pays for
    // the acquire
    const int now = (int)load_flag<LOCAL>(lane == 0 ? (const unsigned int *)L.tl_n + t : (const unsigned int *)&st->err);
    const int n_in = __builtin_amdgcn_readlane(now, 0), err_now = __builtin_amdgcn_readlane(now, 1);
    if (!abort && !err_now && n_in > 0) {
      if (__ballot(dep) != 0ull) sweep_acquire<LOCAL>();
      pass_tile<LA, COV>(pp, L, st, tau, t, colour, tabs, false, smem, lane);
      sweep_release<LOCAL>();  // the tile's writes before its flag
    }
    // every lane stores the same stamp
    __hip_atomic_store(&P.done[t], stamp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <bool LA, bool COV>
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(LA ? 2 : 3, LA ? 2 : 3))) k_sweep(PassParams P) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ TabLds tabs;
  sweep_tiles<LA, COV, false>(P, kernel_params(), tabs, smem);
}
template <bool LA, bool COV>
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(LA ? 2 : 3, LA ? 2 : 3))) k_sweep_xcd(PassParams P) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ TabLds tabs;
  sweep_tiles<LA, COV, true>(P, kernel_params(), tabs, smem);
}

// The fixed-order sum of the tile totals: chunk b of `chunk` tiles into
// part[b], in the order of 256 threads with a stride of 256 and a binary tree
// over them, which a wave keeps with four of those threads a lane.  Only
// chunks with a tile in the layers [zlo, zhi] are read: a tile outside the
// windows has no list and a total of zero.
__device__ inline double chunk_sum(const double *tile_r, int lo, int hi, int lane) {
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int t = lo + lane; t < hi; t += 4 * 256) {
    double v[4][4];
    for (int r = 0; r < 4; r++)
      for (int u = 0; u < 4; u++) {
        const int k = t + 256 * r + 64 * u;
        v[r][u] = k < hi ? tile_r[k] : 0.0;
      }
    for (int r = 0; r < 4; r++)
      for (int u = 0; u < 4; u++) acc[u] += v[r][u];
  }
  double x = (acc[0] + acc[2]) + (acc[1] + acc[3]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, WAVE);
  return x;
}

constexpr int END_THREADS = 1024;
constexpr int SLOT_WORDS = (int)(sizeof(Slot) / 8);
static_assert(SLOT_WORDS == 12 && offsetof(Slot, rmax) == 0 && offsetof(Slot, counts) == 32, "a wave a word of Slot");
static_assert(RS_HEAD % 4 == 0, "RunState's head in words");
struct SweepEndLds {
  double part[NPART];
  unsigned long long sum[SLOT_WORDS];  // Slot's words: the largest rmax, the others summed
  __align__(8) unsigned int head[RS_HEAD / 4];
  int win[32];
  int list_err, zlo, zhi;
  unsigned int sched0;
};
// One thread's part: the state after the sweep, from its head's copy st.
__device__ inline void sweep_end_state(const PassParams &P, SweepEndLds &E, RunState *st, const double rsum) {
  int *const win = P.L.win;
  unsigned int *const sched = P.sched;
  const double rmax = __longlong_as_double((long long)E.sum[0]);
  const long long nmc = (long long)E.sum[1];
  st->events += E.sum[3];
  for (int q = 0; q < 8; q++) st->counts[q] += E.sum[4 + q];
  if (st->la_variant)  // CountLiquid for the next sweep (main.f:637 of the laser-annealing build)
    for (int k = 0; k < 3; k++) {
      st->cc[k] += (long long)st->dcc[k];
      st->dcc[k] = 0ull;
      st->cl[k] = st->cinit[k] - st->cc[k];
    }
  // the passes of the next sweep visit the layers that held candidates; a
  // sweep whose passes were skipped (the run had stopped) collected none,
  // and the windows stay those of the last sweep that ran
  const bool passes_ran = !st->stop;
  int zlo = 0x7fffffff, zhi = -1;
  for (int c = 0; c < 8; c++) {
    if (passes_ran) {
      win[4 * c] = E.win[4 * c] = E.win[4 * c + 2];
      win[4 * c + 1] = E.win[4 * c + 1] = E.win[4 * c + 3];
      win[4 * c + 2] = 0x7fffffff;
      win[4 * c + 3] = -1;
    }
    zlo = min(zlo, E.win[4 * c]);
    zhi = max(zhi, E.win[4 * c + 1]);
  }
  st->ever_lo = min(st->ever_lo, zlo);
  st->ever_hi = max(st->ever_hi, zhi);
  // the dependency-scheduled sweep: a new stamp, an empty queue, the window
  sched[0] = E.sched0 + 1u;
  sched[1] = 0u;
  sched[2] = 0u;
  sched[3] = (unsigned int)zlo;
  sched[4] = (unsigned int)zhi;
  if (E.list_err && !st->err) st->err = E.list_err;
  if (st->tau > 0.0 && !st->err && !st->stop) {
    // a window shortened to end at the time limit lands on it exactly
    st->clock = st->final_sweep ? st->max_time : st->clock + st->tau;
    st->sweeps_run++;
  }
  st->final_sweep = 0;
  st->sweeps++;
  st->rmax = rmax;
  st->n_mc = nmc;
  if (rsum > 0.0) st->rtot = rsum;
  if (st->tau_policy == 1)
    st->tau = rsum > 0.0 ? st->events_per_pass * (double)E.sum[2] / rsum : 0.0;
  else
    st->tau = rmax > 0.0 ? st->events_per_pass / rmax : 0.0;
  if (!st->stop) {
    if (nmc <= 20) st->stop = MSKG_STOP_FEW_MC;
    else if (!(rmax > 0.0)) st->stop = MSKG_STOP_NO_EVENTS;
    else if (st->clock >= st->max_time || st->events >= st->max_events) st->stop = STOP_AT_LIMIT;
  }
  // the last window of a run to a time limit ends at that limit: every tile
  // stops at max_time, as the serial loop stops at the first event past it
  if (!st->stop && st->tau > 0.0 && st->clock + st->tau >= st->max_time) {
    st->tau = st->max_time - st->clock;
    st->final_sweep = 1;
  }
}

// After the eight colour passes: the clock advances by the window just used
// (operator splitting of the master equation over the colours), the next
// window is events_per_pass / (largest tile rate), and the reference's
// early stop applies when at most 20 MC particles remain (main.f:307-310).
//
// One block of END_THREADS: what it needs leaves memory in two round trips --
// a wave a word of the slots, one the windows, two the state's head; then a
// wave a chunk of tiles -- and one thread works on the copy in LDS and writes
// the state.  What bounds it: the launch and those round trips (the tile sums
// had a launch of their own, and the slots a tree of barriers: 10 us a sweep,
// 16.5 at 512^3 SiC).
__device__ inline void sweep_end(const PassParams &P, SweepEndLds &E) {
  int *const win = P.L.win;
  unsigned int *const sched = P.sched;
  const int i = threadIdx.x, lane = i & (WAVE - 1), w = i / WAVE;
  if (i < NPART) E.part[i] = 0.0;
  if (w < SLOT_WORDS) {
    unsigned long long *const a = (unsigned long long *)P.st->slot + (size_t)lane * SLOT_WORDS + w;
    static_assert(NSLOT == 2 * WAVE, "two slots a lane");
    unsigned long long v = a[0], o = a[WAVE * SLOT_WORDS];
    a[0] = 0ull;
    a[WAVE * SLOT_WORDS] = 0ull;
    for (int off = WAVE; off > 0; off >>= 1) {  // the lane's other slot first, then the other lanes
      if (off < WAVE) o = __shfl_xor(v, off, WAVE);
      v = w == 0 ? (v > o ? v : o) : v + o;
    }
    if (lane == 0) E.sum[w] = v;
  } else if (w == SLOT_WORDS) {
    const int v = win[lane & 31];
    if (lane < 32) E.win[lane] = v;
    // the windows of this sweep and of the next: tiles outside hold no rate
    int lo = lane < 32 && !(lane & 1) ? v : 0x7fffffff, hi = lane < 32 && (lane & 1) ? v : -1;
    for (int off = 32; off > 0; off >>= 1) {
      lo = min(lo, __shfl_xor(lo, off, WAVE));
      hi = max(hi, __shfl_xor(hi, off, WAVE));
    }
    if (lane == 0) {
      E.zlo = max(lo, 0);
      E.zhi = min(hi, P.ntz - 1);
    }
  } else if (w == SLOT_WORDS + 1) {
    const unsigned int *const h = (const unsigned int *)P.st;
    for (int k = lane; k < (int)(RS_HEAD / 4); k += WAVE) E.head[k] = h[k];
  } else if (w == SLOT_WORDS + 2 && lane == 0) {
    E.list_err = *P.L.list_err;
    E.sched0 = sched[0];
  }
  __syncthreads();
  if (E.zlo <= E.zhi) {
    const int layer = P.L.ntx * P.L.nty, ntiles = layer * P.ntz, chunk = P.rsum_chunk;
    const int last = min(((E.zhi + 1) * layer - 1) / chunk, NPART - 1);
    for (int b = E.zlo * layer / chunk + w; b <= last; b += END_THREADS / WAVE) {
      const double x = chunk_sum(P.L.tile_r, b * chunk, min(b * chunk + chunk, ntiles), lane);
      if (lane == 0) E.part[b] = x;
    }
  }
  __syncthreads();
  if (w != 0) return;
  double rs = (E.part[lane] + E.part[lane + NSLOT]) + (E.part[lane + WAVE] + E.part[lane + WAVE + NSLOT]);
  for (int off = 32; off > 0; off >>= 1) rs += __shfl_down(rs, off, WAVE);
  RunState *const st = (RunState *)E.head;  // the copy: its head only
  if (i == 0) sweep_end_state(P, E, st, rs);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  unsigned int *const h = (unsigned int *)P.st;
  for (int k = lane; k < (int)(RS_HEAD / 4); k += WAVE) h[k] = E.head[k];
}
__global__ void __launch_bounds__(END_THREADS) k_sweep_end(PassParams P) {
  __shared__ SweepEndLds E;
  sweep_end(P, E);
}

// ---- the batched ensemble: one sweep over many lattices ------------------------
// Every replica keeps its own lattice, lists, windows, run state and random
// stream; a colour pass is one launch over that colour's tiles of all the
// replicas still running.  Before each colour pass a plan lays that
// colour's tiles of the replicas end to end -- made just before the pass,
// as k_pass reads its window when it starts, because the passes of the
// earlier colours widen the windows of the later ones when they enlist
// points in a new tile layer:
//   plan[c * (n + 1) + r]      c = 0..7, r = 0..n: tiles of colour c in the
//                              windows of replicas 0..r-1 (replicas that do
//                              not run hold none)
//   plan[8 * (n + 1) + c]      queue head of colour c, in units of 64
//   plan[8 * (n + 1) + 8]      replicas running the coming sweep
//   plan[8 * (n + 1) + 9 + r]  replica r runs the coming sweep
// The plan of colour 0 (start = 1) comes after the sweep's end and also
// decides which replicas run the next sweep.  Persistent waves take the
// entries of a colour's queue one at a time, so the tiles of large and
// small replicas share the GPU and the slowest tiles of a pass overlap
// other tiles' work instead of idling the rest.
constexpr int ENS_MAX = 1024;
static inline int64_t ens_plan_words(int n) { return 8 * (int64_t)(n + 1) + 9 + n; }

__global__ void __launch_bounds__(ENS_MAX) k_ens_plan(const PassParams *__restrict__ reps, int n, int *plan,
                                                      int colour, int start) {
  __shared__ int sc[ENS_MAX];
  __shared__ int nrun;
  const int r = threadIdx.x;
  int cnt = 0, run = 0;
  if (r == 0) nrun = 0;
  if (r < n) {
    const PassParams &P = reps[r];
    const RunState *st = P.st;
    if (start) {
      run = st->tau > 0.0 && !st->err && !st->stop;
      plan[8 * (n + 1) + 9 + r] = run;
    } else {
      run = plan[8 * (n + 1) + 9 + r];
    }
    // k_pass's condition, checked as its colour pass starts
    if (run && !st->err) {
      int zf;
      cnt = colour_tiles(P.L, P.ntz, colour, P.L.win[4 * colour], P.L.win[4 * colour + 1], zf);
    }
  }
  __syncthreads();
  if (start && run) atomicAdd(&nrun, 1);
  // inclusive scan over the replicas, in replica order
  sc[r] = cnt;
  __syncthreads();
  for (int off = 1; off < ENS_MAX; off <<= 1) {
    const int v = r >= off ? sc[r - off] : 0;
    __syncthreads();
    sc[r] += v;
    __syncthreads();
  }
  if (r < n) plan[colour * (n + 1) + r + 1] = sc[r];
  if (r == 0) {
    plan[colour * (n + 1)] = 0;
    plan[8 * (n + 1) + colour] = 0;
    if (start) plan[8 * (n + 1) + 8] = nrun;
  }
}

// The replica whose tiles hold entry q of colour pc's queue: the last r with
// pc[r] <= q (pc is the colour's prefix, pc[n] > q), 64 prefixes at a time.
__device__ inline int ens_replica(const int *pc, int n, int q, int lane) {
  const int j1 = 64 * lane;
  const int v1 = pc[min(j1, n)];  // every lane loads (an index clamped to the prefix)
  const int b = __popcll(__ballot(j1 <= n && v1 <= q)) - 1;  // pc[0] = 0 <= q: b >= 0
  const int j2 = 64 * b + lane;
  const int v2 = pc[min(j2, n)];
  return 64 * b + __popcll(__ballot(j2 <= n && v2 <= q)) - 1;
}

template <bool LA, bool COV>
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(LA ? 2 : 3, LA ? 2 : 3)))
k_pass_ens(const PassParams *__restrict__ reps, int n, int *plan, int colour) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ TabLds tabs;
  const int lane = threadIdx.x;
  const int *pc = plan + colour * (n + 1);
  const int total = __builtin_amdgcn_readfirstlane(pc[n]);
  unsigned int *const head = (unsigned int *)(plan + 8 * (n + 1) + colour);
  // the replica of the last entry: its entries [lo, hi) of the queue, its
  // lattice and run state, the window's first layer and the window tau
  int r = -1, lo = 0, hi = 0, zfirst = 0, failed = 0;
  double tau = 0.0;
  bool fresh = false;
  const PassParams *pp = as_constant(reps);
  Lattice L = event_part(pp);
  RunState *st = nullptr;
  // Every decision of this loop is wave-uniform (readfirstlane / ballot)
  // and no memory access sits under a lane-dependent branch.  A wave's
  // first entry is its own (blockIdx.x), so that the waves do not all meet
  // at the queue head when the pass starts (same-address atomics are
  // served one after another), and an empty pass takes no atomic at all;
  // the entries from gridDim.x on are taken from the queue.
  int q = blockIdx.x;
  for (;;) {
    if (q >= total) break;
    if (q < lo || q >= hi) {
      r = __builtin_amdgcn_readfirstlane(ens_replica(pc, n, q, lane));
      lo = __builtin_amdgcn_readfirstlane(pc[r]);
      hi = __builtin_amdgcn_readfirstlane(pc[r + 1]);
      pp = as_constant(reps + r);
      L = event_part(pp);
      fresh = true;
      st = as_global(pp->st);
      // a replica that has failed in this sweep runs no further tiles here
      // (k_pass checks at the start of each colour pass)
      failed = __builtin_amdgcn_readfirstlane(__hip_atomic_load(&st->err, __ATOMIC_RELAXED,
                                                                __HIP_MEMORY_SCOPE_AGENT));
      tau = st->tau;
      const int *const win = as_global(pp->L.win) + 4 * colour;
      colour_tiles(pp->L, pp->ntz, colour, win[0], win[1], zfirst);
    }
    if (!failed) {
      const int t = colour_tile(pp->L, colour, zfirst, q - lo);
      // a wave stops its tiles of a replica whose tile failed (as k_pass's wave returns)
      failed = __builtin_amdgcn_readfirstlane(
          pass_tile<LA, COV>(pp, L, st, tau, t, colour, tabs, fresh, smem, lane));
      fresh = false;
    }
    // the next entry: every lane adds 1 (one atomic of 64 for the wave)
    const unsigned int took = __hip_atomic_fetch_add(head, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    q = (int)gridDim.x + __builtin_amdgcn_readfirstlane((int)(took >> 6));
  }
}

// The sweep's end for every replica that ran the sweep (the same per-replica
// work as k_sweep_end, so the replica's window, clock and stop are those it
// gets alone).
__global__ void __launch_bounds__(END_THREADS) k_sweep_end_ens(const PassParams *__restrict__ reps, int n,
                                                               const int *plan) {
  __shared__ SweepEndLds E;
  const int r = blockIdx.x;
  if (!plan[8 * (n + 1) + 9 + r]) return;
  sweep_end(reps[r], E);
}

// ---- device-side initial state ----------------------------------------------
// Diamond sites of the reference grid: x, y, z multiples of 3 whose thirds
// have equal parity; (x+y+z)/3 = 0 (mod 4) is fcc sublattice A (bonds
// JumpDia(:,1:4)), = 3 (mod 4) sublattice B (JumpDia(:,5:8))
// (initial/SetSi.f:36-45, modules/defsystem.f:112-113).
__device__ inline int dia_type(int x, int y, int z) {
  if (x % 3 || y % 3 || z % 3) return 0;
  int x1 = x / 3, y1 = y / 3, z1 = z / 3;
  if ((x1 & 1) != (y1 & 1) || (x1 & 1) != (z1 & 1)) return 0;
  int m = (x1 + y1 + z1) & 3;
  return m == 0 ? 1 : (m == 3 ? 2 : 0);
}
__constant__ int c_jump_dia[8][3] = {{3, 3, 3}, {3, -3, -3}, {-3, -3, 3}, {-3, 3, -3},
                                     {3, 3, -3}, {3, -3, 3}, {-3, -3, -3}, {-3, 3, 3}};

// A block's threads' atoms of species 1 and 2 into atoms[].
__device__ inline void count_atoms(const unsigned int mine[2], unsigned long long *atoms) {
  __shared__ unsigned int sum[2];
  if (threadIdx.x < 2) sum[threadIdx.x] = 0u;
  __syncthreads();
  for (int k = 0; k < 2; k++) {
    unsigned int v = mine[k];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0 && v) atomicAdd(&sum[k], v);
  }
  __syncthreads();
  if (threadIdx.x < 2 && sum[threadIdx.x]) atomicAdd(&atoms[threadIdx.x], (unsigned long long)sum[threadIdx.x]);
}

// The flat (001) slab of SetSi.f:25-220 (sic=0: Si on both sublattices,
// wall layers z=0..5 and LenZ-6..LenZ-1) or SetSiC3C.f:25-198 (sic=1: Si on
// A, C on B, no walls): bulk below len-3, the top atomic layer as MC
// particles with PTransE(s,2,0,...), the empty sites above with
// coordination 2 and their deposition rate.  Every point is written, and its
// list flag cleared; `atoms` takes the atoms by species.
//
// What bounds it: 22 bytes written a point.  Walls and the planes above the
// slab or off the diamond planes hold one value, known from the point's z;
// only every sixth point of every third plane of the slab is computed.  The
// atoms are counted here, where they are placed (a census of the lattice
// read its 16 bytes a point again), and after it only the planes of the surface
// are swept for rates and searched for list entries.  Whole passes with those
// three reading every point, and now: 512^3 SiC 52.4, 49.5 ms; 24 SiGe
// replicas 36.1, 30.0; likelihood of 128 trajectories 34.5, 30.4; 64 serial
// trajectories 51.7, 48.1; Si PVD 50.5, 49.3.
__global__ void __launch_bounds__(256) k_build_slab(Lattice L, int len, int sic, double fraction, uint32_t key0,
                                                   uint32_t key1, int top_lz, unsigned long long *atoms) {
  const Tables &t = *L.tab;
  const int64_t n = L.box.npts;
  unsigned int mine[2] = {0u, 0u};
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
    int z = (int)div_by(p, L.box.plane, L.box.inv_plane);
    Site s;
    for (int a = 0; a < 4; a++) s.d[a][0] = s.d[a][1] = s.d[a][2] = 0;
    s.kc = 0; s.valid = 0; s.temp = 0;
    int cls = CLS_NONE;
    double r = 0.0;
    // top_lz: LenZ of the whole box (the top wall planes lie above the stored ones when only the bottom planes are stored)
    const bool wall = sic != 1 && ((z >= 0 && z <= 5) || (z >= top_lz - 6 && z <= top_lz - 1));
    int x = 0, y = 0, ty = 0;
    if (!wall && z <= len && z % 3 == 0) {
      pxyz(L.box, p, x, y, z);
      ty = dia_type(x, y, z);
    }
    if (wall) {
      s.kc = KIND_WALL;
    } else if (ty) {
      int sp = (sic == 1 && ty == 2) ? 2 : 1;
      if (sic == 2) {  // random substitutional alloy: species 2 with probability `fraction`
        U4 c;
        c.x = (uint32_t)p; c.y = (uint32_t)(p >> 32); c.z = 0x5e6e0001u; c.w = 0;
        const U4 d = philox4x32_10(c, key0, key1);
        if (u01_open(d.x, d.y) < fraction) sp = 2;
      }
      NL l;
      for (int i = 0; i < 4; i++) {
        const int *j = c_jump_dia[(ty == 1 ? 0 : 4) + i];
        l.x[i] = x + j[0]; l.y[i] = y + j[1]; l.z[i] = z + j[2];
        if (l.x[i] >= L.box.lx) l.x[i] -= L.box.lx;
        if (l.x[i] < 0) l.x[i] += L.box.lx;
        if (l.y[i] >= L.box.ly) l.y[i] -= L.box.ly;
        if (l.y[i] < 0) l.y[i] += L.box.ly;
      }
      set_list(L.box, s, x, y, z, l);
      if (z <= len - 4) {
        s.kc = (uint8_t)(sp | (4 << 3));
      } else if (z <= len - 1) {
        s.kc = (uint8_t)(sp | (2 << 3));
        if (z >= t.frozen_below_z) {
          cls = CLS_EVAP;
          r = t.pe[pe_flat(sp, 2, 0, 0, 0, 0, 0)];
        }
      } else {
        s.kc = (uint8_t)(KIND_EMPTY | (2 << 3));
        cls = CLS_ADSORB;
        double pd[3];
        pd_of<true>(TabSrc{t}, 2, 0, nullptr, pd);
        r = pd[0] + pd[1] + pd[2] +
            t.pabs[0 + 6] + t.pabs[1 + 6] + t.pabs[2 + 6];
      }
      if (z <= len - 1) mine[sp - 1]++;
    }
    L.site[p] = s;
    L.rate[p] = cls ? (float)r : 0.0f;
    L.cls[p] = (uint8_t)cls;
    L.inlist[p] = 0;
  }
  count_atoms(mine, atoms);
}

// ---- the shaped initial states (main.f:224-294) ----------------------------------
// SetNC / SetNCSp / SetInvPOff / SetSiFINFET / SetCAD all place atoms and
// walls first, then run one coordination pass (an atom with no occupied
// neighbour is removed) and one probability pass that fills the lists.  On
// the device: k_shape_place writes every stored point's kind from the
// builder's geometry, k_shape_isolated removes the isolated atoms,
// k_shape_records gives every site its coordination and neighbour list,
// and the rate sweep evaluates the MC particles.  An isolated atom's
// neighbours are all empty, so no removal changes a coordination another
// removal reads, and the result does not depend on the order of the
// reference's sequential pass.
enum : int { SHAPE_BOX = 0, SHAPE_SPHERE = 1, SHAPE_INVP = 2, SHAPE_FINFET = 3, SHAPE_CAD = 4 };
struct ShapeSpec {
  int shape;
  int l1, l2, l3, l4;   // Len1..Len4 as the builder takes them
  int cx, cy, cz;       // SetNC / SetNCSp centre (LenX/2, LenY/2, LenZ/2)
  int lz;               // LenZ
  int xa, xb;           // SetSiFINFET: the fin lies in xa <= x < xb
  int zfix;             // SetInvPOff: atoms at z <= zfix are bulk of coordination 4 (-1: none)
  int walls;            // an empty site's coordination leaves walls out
  const int8_t *ids;    // SetCAD geometry ids, [z][y][x] for z < LenZ
  double fraction;      // SetCAD: species 2 with this probability (Philox)
  uint32_t key0, key1;
};

// The builder's content of grid point (x, y, z): KIND_WALL, a species, or
// KIND_EMPTY.  Walls lie on every grid point of their region, atoms on the
// diamond sites of theirs (SetNC.f, SetNCSp.f, SetInvPOff.f:21-286,
// SetSiFINFET.f:25-312, SetCAD.f:84-190).
__device__ inline int shape_content(const ShapeSpec &S, int x, int y, int z, int lx, int ly, int64_t p) {
  const int t = dia_type(x, y, z);
  switch (S.shape) {
    case SHAPE_BOX:
    case SHAPE_SPHERE: {
      const int l2 = S.shape == SHAPE_BOX ? S.l2 : S.l1, l3 = S.shape == SHAPE_BOX ? S.l3 : S.l1;
      if (!t || x < S.cx - S.l1 / 2 || x > S.cx + S.l1 / 2 - 1 || y < S.cy - l2 / 2 || y > S.cy + l2 / 2 - 1 ||
          z < S.cz - l3 / 2 || z > S.cz + l3 / 2 - 1)
        return KIND_EMPTY;
      if (S.shape == SHAPE_SPHERE) {
        const int d2 = (x - S.cx) * (x - S.cx) + (y - S.cy) * (y - S.cy) + (z - S.cz) * (z - S.cz);
        if (!(d2 <= S.l1 * S.l1 / 4)) return KIND_EMPTY;
      }
      return t == 1 ? 1 : 2;
    }
    case SHAPE_INVP: {  // l1: Len (pyramid size), l2: Len3 (substrate top)
      if (!t) return KIND_EMPTY;
      if (z <= 20) return t == 1 ? 1 : 2;
      if (z > S.l2 - 1) return KIND_EMPTY;
      // the reference's single-precision test: integer sums minus
      // 1.10*(z-Len3) in REAL(4) against REAL(4) Len
      const int lenh = lx / 2 - 1;
      const float dz = 1.10f * (float)(z - S.l2), fl = (float)S.l1;
      const bool hole = ((float)(abs(x - lenh) + abs(y - lenh)) - dz <= fl) ||
                        ((float)(abs(x) + abs(y)) - dz <= fl) || ((float)(abs(x - lx) + abs(y)) - dz <= fl) ||
                        ((float)(abs(x) + abs(y - ly)) - dz <= fl) ||
                        ((float)(abs(x - lx) + abs(y - ly)) - dz <= fl);
      return hole ? KIND_EMPTY : (t == 1 ? 1 : 2);
    }
    case SHAPE_FINFET: {  // l1: Len (Si top), l2: wall bottom, l3: wall top
      const bool wall = z <= 5 || (z >= S.lz - 6 && z <= S.lz - 1) || (z >= S.l3 && z <= S.lz - 7) ||
                        (z >= S.l2 && z <= S.lz - 7 && (x < S.xa || x >= S.xb));
      if (wall) return KIND_WALL;
      return (t && z >= 6 && z <= S.l1 - 1) ? 1 : KIND_EMPTY;
    }
    default: {  // SHAPE_CAD
      if (z <= 3 || (z >= S.lz - 4 && z <= S.lz - 1)) return KIND_WALL;
      if (z > S.lz - 5) return KIND_EMPTY;
      const int id = S.ids[(int64_t)x + (int64_t)lx * ((int64_t)y + (int64_t)ly * z)];
      if (id == 10) return KIND_WALL;
      if (id != 1 || !t) return KIND_EMPTY;
      if (S.fraction > 0.0) {  // the reference's RAND() < alloyfraction, from the engine's stream
        U4 c;
        c.x = (uint32_t)p; c.y = (uint32_t)(p >> 32); c.z = 0x5e6e0002u; c.w = 0;
        const U4 d = philox4x32_10(c, S.key0, S.key1);
        if (u01_open(d.x, d.y) < S.fraction) return 2;
      }
      return 1;
    }
  }
}

__global__ void __launch_bounds__(256) k_shape_place(Lattice L, ShapeSpec S) {
  const int64_t n = L.box.npts;
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
    int x, y, z;
    pxyz(L.box, p, x, y, z);
    Site s;
    for (int a = 0; a < 4; a++) s.d[a][0] = s.d[a][1] = s.d[a][2] = 0;
    s.valid = 0;
    s.temp = L.site[p].temp;  // a temperature set before the build stays (SetCAD.f:62-65)
    s.kc = (uint8_t)shape_content(S, x, y, z, L.box.lx, L.box.ly, p);
    L.site[p] = s;
    L.rate[p] = 0.0f;
    L.cls[p] = 0;
    L.inlist[p] = 0;
  }
}

// The four neighbour sites of diamond site (x, y, z) of type t, x and y
// wrapped once (the builders' JumpDia lists).
__device__ inline NL dia_list(const Box &b, int t, int x, int y, int z) {
  NL l;
  for (int i = 0; i < 4; i++) {
    const int *j = c_jump_dia[(t == 1 ? 0 : 4) + i];
    l.x[i] = x + j[0]; l.y[i] = y + j[1]; l.z[i] = z + j[2];
    if (l.x[i] >= b.lx) l.x[i] -= b.lx;
    if (l.x[i] < 0) l.x[i] += b.lx;
    if (l.y[i] >= b.ly) l.y[i] -= b.ly;
    if (l.y[i] < 0) l.y[i] += b.ly;
  }
  return l;
}
__device__ inline int kind_at(const Lattice &L, int x, int y, int z) {
  const int64_t q = pidx_checked(L.box, x, y, z);
  return q < 0 ? KIND_EMPTY : s_kind(L.site[q]);
}

// An atom none of whose four neighbours is occupied (an atom or a wall) is
// removed (SetCAD.f:229-246, SetNC.f's same pass); atoms of a fixed bulk
// region are left alone.
__global__ void __launch_bounds__(256) k_shape_isolated(Lattice L, ShapeSpec S) {
  const int64_t n = L.box.npts;
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
    const Site sp = L.site[p];
    if (!kind_species(s_kind(sp))) continue;
    int x, y, z;
    pxyz(L.box, p, x, y, z);
    if (z <= S.zfix) continue;
    const int t = dia_type(x, y, z);
    if (!t) continue;
    const NL l = dia_list(L.box, t, x, y, z);
    int occ = 0;
    for (int i = 0; i < 4; i++) occ += kind_occupied(kind_at(L, l.x[i], l.y[i], l.z[i]));
    if (!occ) {
      Site e = sp;
      e.kc = KIND_EMPTY;  // LattCoo = 0, the temperature kept
      L.site[p] = e;
    }
  }
}

// Coordination and neighbour list of every diamond site (SetCAD.f:194-416):
// an atom counts its occupied neighbours (walls included), an empty site
// its atoms (with walls = 1; every occupied neighbour otherwise); an empty
// site of coordination 1 keeps only that neighbour, in entry 1.  Atoms and
// empty sites of coordination >= 1 get their list; walls and the empty
// sites of coordination 0 keep a bare record.  The atoms are final here and
// counted on the way (a census read every record once more: 218 us at
// 768x768x384).
__global__ void __launch_bounds__(256) k_shape_records(Lattice L, ShapeSpec S, int *err, unsigned long long *atoms) {
  const int64_t n = L.box.npts;
  unsigned int mine[2] = {0u, 0u};
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
    Site s = L.site[p];
    const int kind = s_kind(s);
    if (kind == KIND_WALL) continue;
    if (kind_species(kind)) mine[kind - 1]++;  // the builders place species 1 and 2
    int x, y, z;
    pxyz(L.box, p, x, y, z);
    const int t = dia_type(x, y, z);
    if (!t) continue;
    NL l = dia_list(L.box, t, x, y, z);
    int coor = 0, last = -1;
    for (int i = 0; i < 4; i++) {
      const int k = kind_at(L, l.x[i], l.y[i], l.z[i]);
      if (kind_species(kind) ? kind_occupied(k) : (S.walls ? kind_species(k) : kind_occupied(k))) {
        coor++;
        last = i;
      }
    }
    if (kind_species(kind) && z <= S.zfix) coor = 4;
    if (!kind_species(kind) && coor == 0) continue;
    if (!kind_species(kind) && coor == 1) {
      // the NBuff compaction of SetCAD.f:316-327: entry 1 the one atom, the rest unfixed
      const int lx0 = l.x[last], ly0 = l.y[last], lz0 = l.z[last];
      for (int i = 0; i < 4; i++) l.x[i] = l.y[i] = l.z[i] = 0;
      l.x[0] = lx0; l.y[0] = ly0; l.z[0] = lz0;
    }
    s_set_coor(s, coor);
    if (!set_list(L.box, s, x, y, z, l)) atomicExch(err, ERR_GEOM);
    L.site[p] = s;
  }
  count_atoms(mine, atoms);
}

// The placeholder deposition rate of an initial state is Get_Prob_Ini's
// REAL(4) 1.e-6 (Get_Prob_Ini.f:104), not Get_Prob's 1.e-8.
__global__ void __launch_bounds__(256) k_initial_placeholders(Lattice L) {
  const int64_t n = L.box.npts;
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x)
    if (L.cls[p] == CLS_PLACEHOLDER) L.rate[p] = (float)(double)1.e-6f;
}

// Walls on the grid points off the stored lattice, one bit per grid point
// (what the phase maps report): a lane takes four consecutive grid points (of
// one row: LenX is a multiple of 12), eight lanes a word.  A position costs
// two divisions by the FP64 reciprocals for four points, and a lane's reads of
// their geometry ids are in flight together (a thread a word of 32 points took
// six 64-bit remainders a point, a wave 64 points at a time one read at a
// time: 519 and 612 us at 768x768x384).
__global__ void __launch_bounds__(256) k_shape_offwall(Lattice L, ShapeSpec S, uint32_t *bits, int64_t words) {
  const int lx = L.box.lx, ly = L.box.ly;
  const int64_t face = (int64_t)lx * ly, lanes = words * 8;
  const double inv_face = 1.0 / (double)face, inv_lx = 1.0 / (double)lx;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t rounds = (lanes + stride - 1) / stride;  // the same for every lane: all of a word's take part
  for (int64_t r = 0; r < rounds; r++) {
    const int64_t q = r * stride + (int64_t)blockIdx.x * blockDim.x + threadIdx.x, g = 4 * q;
    const int64_t z = div_by(g, face, inv_face), f = g - z * face;
    const int y = (int)div_by(f, lx, inv_lx), x = (int)(f - (int64_t)y * lx);
    uint32_t m = 0;
    if (q < lanes && z <= L.box.lz)
      for (int k = 0; k < 4; k++)
        if (!valid_parity(x + k, y, (int)z) && shape_content(S, x + k, y, (int)z, lx, ly, 0) == KIND_WALL) m |= 1u << k;
    m <<= 4 * (threadIdx.x & 7);
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xb1, 0xf, 0xf, false);   // lanes 1 0 3 2
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4e, 0xf, 0xf, false);   // lanes 2 3 0 1
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xf, 0xf, false);  // row_half_mirror: the other four
    if (q < lanes && (threadIdx.x & 7) == 0) bits[q >> 3] = m;
  }
}

// ---- serial BKL over a batch of independent lattices --------------------------
// One workgroup (one wave) per replica runs the reference's serial algorithm:
// every event picks one MC particle of the whole lattice with probability
// rate/R (R the FP64 total) and advances the clock by -ln(u)/R.  The rates
// are organised as a three-level sum: the FP32 rates of each tile's
// candidate list, FP64 tile sums, and FP64 sums of 64 consecutive tiles; an
// event rescans only the lists of the tiles it touched.
struct SerialDesc {
  Lattice L;
  double *tsum;   // [ntiles]
  double *bsum;   // [nblk]
  RunState *st;
  mskg_event *log;
  unsigned long long log_cap;
  long long max_events;
  double max_time;
  uint32_t key0, key1;
  int ntiles, nblk, replica;
};

// Rate sum of one tile's list (every class); entries whose class fell to 0
// leave the list.  The compaction is in place: an entry moves only to a
// position at or before the one it was read from in the same step.
__device__ inline double tile_sum_compact(const Lattice &L, int t, int lane) {
  const TileGeom g = tile_geom(t, L.tile, L.ntx, L.nty, L.box.lz);
  const int m = min(L.tl_n[t], L.capg);
  int32_t *idx = L.tl_idx + (int64_t)t * L.capg;
  double part = 0.0;
  int nout = 0;
  for (int j0 = 0; j0 < m; j0 += WAVE) {
    const int j = j0 + lane;
    int k = 0;
    bool keep = false;
    if (j < m) {
      k = idx[j];
      const P3 p = tile_point(L.box, g, L.tile, k);
      const uint8_t c = L.cls[p.i];  // class and rate in one round trip
      const float r = L.rate[p.i];
      keep = c != 0;
      if (keep) part += (double)r;
      else L.inlist[p.i] = 0;
    }
    const unsigned long long msk = __ballot(keep);
    const int slot = nout + __popcll(msk & ((1ull << lane) - 1ull));
    if (keep) idx[slot] = k;
    nout += __popcll(msk);
  }
  part = wave_sum_dpp(part);
  if (lane == 0) L.tl_n[t] = nout;
  return part;
}
// The same for four tiles at once, a row of 16 lanes each (t: the row's tile,
// -1: none): one chain of reads for all of them.  The additions are those of
// the whole wave, whose lanes 16..63 hold zeros.  False, with nothing
// changed, when a list is longer than a row.
__device__ inline bool tile_sum_rows(const Lattice &L, int t, int lane, double &sum) {
  const int rl = lane & 15;
  const int tt = max(t, 0);
  const int raw = L.tl_n[tt];
  int32_t *const idx = L.tl_idx + (int64_t)tt * L.capg;
  const int k = idx[min(rl, L.capg - 1)];  // read whatever the length, used only below it
  const int m = t >= 0 ? min(raw, L.capg) : 0;
  if (__ballot(m > 16)) return false;
  double part = 0.0;
  bool keep = false;
  if (rl < m) {
    const TileGeom g = tile_geom(tt, L.tile, L.ntx, L.nty, L.box.lz);
    const P3 p = tile_point(L.box, g, L.tile, k);
    const uint8_t c = L.cls[p.i];
    const float r = L.rate[p.i];
    keep = c != 0;
    if (keep) part = (double)r;
    else L.inlist[p.i] = 0;
  }
  const unsigned mask = (unsigned)(__ballot(keep) >> (lane & 48)) & 0xffffu;
  const int slot = __popc(mask & ((1u << rl) - 1u));
  if (keep && slot != rl) idx[slot] = k;
  if (t >= 0 && rl == 0 && __popc(mask) != raw) L.tl_n[t] = __popc(mask);
  part += dpp_take<0x128, 0xf>(part);  // row_ror:8
  part += dpp_take<0x124, 0xf>(part);  // row_ror:4
  part += dpp_take<0x122, 0xf>(part);  // row_ror:2
  part += dpp_take<0x121, 0xf>(part);  // row_ror:1
  sum = part;
  return true;
}
// wave_incl_scan of values that lanes 16..63 hold none of, for the lanes
// 0..15: the same additions in one row.
__device__ inline double row_incl_scan(double v) {
  v += dpp_take<0x111, 0xf>(v);  // row_shr:1
  v += dpp_take<0x112, 0xf>(v);  // row_shr:2
  v += dpp_take<0x114, 0xf>(v);  // row_shr:4
  v += dpp_take<0x118, 0xf>(v);  // row_shr:8
  return v;
}

// Index of the first element of v[0..n) (FP64, read from memory) whose
// inclusive prefix exceeds target; *below receives the prefix before it.
// Rounding at the top end falls back to the last positive element.
__device__ int scan_pick(const double *v, int n, double target, int lane, double *below) {
  double acc = 0.0;
  int last_nz = -1;
  double acc_last = 0.0;
  for (int base = 0; base < n; base += WAVE) {
    const int j = base + lane;
    const double x = j < n ? v[j] : 0.0;
    const double inc = (n <= 16 ? row_incl_scan(x) : wave_incl_scan(x, lane)) + acc;
    const unsigned long long nzm = __ballot(x > 0.0);
    if (nzm) {
      const int hi = 63 - __clzll((long long)nzm);
      last_nz = base + hi;
      acc_last = __shfl(inc - x, hi, WAVE);
    }
    const unsigned long long hit = __ballot(j < n && x > 0.0 && inc > target);
    if (hit) {
      const int l = __ffsll((long long)hit) - 1;
      *below = __shfl(inc - x, l, WAVE);
      return base + l;
    }
    acc = __shfl(inc, WAVE - 1, WAVE);
  }
  *below = acc_last;
  return last_nz;
}

// Replicas of up to SERIAL_LDS_TILES tiles keep their tile and block sums on
// chip; larger ones use the engine's global arrays.
constexpr int SERIAL_LDS_TILES = 4096;
//
// What bounds it: one wave's chain of an event's reads and instructions, about
// 7.5 us an event, of which the event itself 3.5.  Draws and logarithms are made
// 64 at once; the tiles an event touched are rescanned four at a time, a row
// of 16 lanes each; lists and levels of up to 16 entries are scanned in one
// row.  64 lattices of 144^3, 3000 events each: 27.1 ms with one after the other, now 22.6.
template <bool LA, bool COV>
__global__ void __launch_bounds__(WAVE) k_serial(const SerialDesc *descs) {
  __shared__ TabLds tabs;
  __shared__ double s_tsum[SERIAL_LDS_TILES], s_bsum[SERIAL_LDS_TILES / WAVE];
  const int lane = threadIdx.x;
  const SerialDesc D = descs[blockIdx.x];
  Lattice L = D.L;
  to_global(L);
  L.cold = as_constant(&descs[blockIdx.x].L);
  RunState *st = as_global(D.st);
  load_tables<LA>(*L.tab, tabs, lane);
  if (st->err) return;
  const bool on_chip = D.ntiles <= SERIAL_LDS_TILES;
  double *tsum = on_chip ? s_tsum : D.tsum;
  double *bsum = on_chip ? s_bsum : D.bsum;
  unsigned long long my_cnt = 0;  // lane l: events of counter l
  // initial sums
  for (int t = 0; t < D.ntiles; t++) {
    const double ts = tile_sum_compact(L, t, lane);
    if (lane == 0) tsum[t] = ts;
  }
  wave_sync();
  for (int b = 0; b < D.nblk; b++) {
    const int t = b * WAVE + lane;
    const double v = wave_sum_dpp(t < D.ntiles ? tsum[t] : 0.0);
    if (lane == 0) bsum[b] = v;
  }
  wave_sync();
  double clock = st->clock;
  unsigned long long events = st->events, nev = 0;
  int stop = MSKG_STOP_LIMIT, err = 0;
  const unsigned long long log_n = st->log_n;
  U4 draw;           // lane l: the Philox block of event 64 b + l of this call, b the current batch
  double wait = 0.0;  // ... and -ln of its first uniform
  while ((long long)nev < D.max_events && clock < D.max_time) {
    // one Philox block per event: waiting time, selection, event type and
    // stacking choice, 32 random bits each
    const int dl = (int)(nev & (WAVE - 1));
    if (dl == 0) {
      U4 ctr;
      ctr.x = 0x5e71a1u;  // the stream depends on the engine's seed only, not on its place in the batch
      ctr.y = (uint32_t)(events + lane);
      ctr.z = (uint32_t)((events + lane) >> 32);
      ctr.w = 0;
      draw = philox4x32_10(ctr, D.key0, D.key1);
      wait = -log(u01_32(draw.x));
    }
    double part = 0.0;
    for (int b = lane; b < D.nblk; b += WAVE) part += bsum[b];
    const double R = wave_sum_dpp(part);
    if (!(R > 0.0)) { stop = MSKG_STOP_NO_EVENTS; break; }
    const double dt = read_lane(wait, dl) / R;
    double target = u01_32((uint32_t)__builtin_amdgcn_readlane((int)draw.y, dl)) * R, below = 0.0;
    // block -> tile -> list entry
    const int b = scan_pick(bsum, D.nblk, target, lane, &below);
    if (b < 0) { stop = MSKG_STOP_NO_EVENTS; break; }
    target -= below;
    const int t0 = b * WAVE;
    const int tl = scan_pick(tsum + t0, min(WAVE, D.ntiles - t0), target, lane, &below);
    if (tl < 0) { err = ERR_SUMS; break; }
    const int t = t0 + tl;
    target -= below;
    const TileGeom g = tile_geom(t, L.tile, L.ntx, L.nty, L.box.lz);
    const int m = min(L.tl_n[t], L.capg);
    const int32_t *idx = L.tl_idx + (int64_t)t * L.capg;
    double acc = 0.0;
    int sel = -1, last_nz = -1;
    for (int base = 0; base < m; base += WAVE) {
      const int j = base + lane;
      double v = 0.0;
      if (j < m) {
        const P3 p = tile_point(L.box, g, L.tile, idx[j]);
        const uint8_t c = L.cls[p.i];
        const float r = L.rate[p.i];
        if (c) v = (double)r;
      }
      const unsigned long long nzm = __ballot(v > 0.0);
      if (nzm) last_nz = base + 63 - __clzll((long long)nzm);
      const double inc = (m <= 16 ? row_incl_scan(v) : wave_incl_scan(v, lane)) + acc;
      const unsigned long long hit = __ballot(j < m && v > 0.0 && inc > target);
      if (hit) { sel = base + __ffsll((long long)hit) - 1; break; }
      acc = __shfl(inc, WAVE - 1, WAVE);
    }
    if (sel < 0) sel = last_nz;
    if (sel < 0) { err = ERR_SUMS; break; }
    const P3 s = tile_point(L.box, g, L.tile, __builtin_amdgcn_readfirstlane(idx[sel]));
    Choice ch;
    ch.arm = -1;
    ch.u_arm = u01_32((uint32_t)__builtin_amdgcn_readlane((int)draw.w, dl));
    const Rec srec = uniform_rec(load_rec(L, s.i));
    const int coor0 = r_coor(srec);
    const int itrans = __builtin_amdgcn_readfirstlane(pick_itrans<LA, COV>(
        L, TabEv<COV>{*L.tab, tabs}, coor0, r_temp(srec), __builtin_amdgcn_readfirstlane((int)L.cls[s.i]),
        u01_32((uint32_t)__builtin_amdgcn_readlane((int)draw.z, dl))));
    EvOut o;
    execute<LA, COV>(L, tabs, R, s, srec, itrans, ch, o, lane);
    clock += dt;
    if (lane == 0) {
      if (D.log) {
        const unsigned long long li = log_n + nev;
        if (li < D.log_cap) {
          mskg_event ev;
          ev.iter = (int64_t)(events + 1);
          ev.site[0] = s.x; ev.site[1] = s.y; ev.site[2] = s.z;
          ev.itrans = itrans;
          ev.arm = o.arm;
          ev.coor = coor0;
          ev.rtot = R;
          ev.time = clock;
          D.log[li] = ev;
        }
      }
      if (COV && itrans == 5 && o.species) st->desorbed[o.species - 1]++;
    }
    if (lane == count_slot(itrans)) my_cnt++;
    wave_sync();
    events++;
    nev++;
    err = __builtin_amdgcn_readfirstlane(o.err);
    if (err) break;
    // the tiles of the points that got a new rate, each rescanned once; then
    // the blocks of those tiles
    const int tq = o.set ? tile_of(L, o.p) : -1;
    const unsigned long long tm = __ballot(o.set != 0);
    for (unsigned long long m2 = tm; m2;) {
      int four[4];
      for (int q = 0; q < 4; q++) {
        four[q] = -1;
        if (m2) {
          four[q] = __builtin_amdgcn_readlane(tq, __ffsll((long long)m2) - 1);
          m2 &= ~__ballot(tq == four[q]);
        }
      }
      const int mine = lane < 32 ? (lane < 16 ? four[0] : four[1]) : (lane < 48 ? four[2] : four[3]);
      double ts;
      if (tile_sum_rows(L, mine, lane, ts)) {
        if ((lane & 15) == 0 && mine >= 0) tsum[mine] = ts;
      } else {
        for (int q = 0; q < 4; q++) {
          if (four[q] < 0) continue;
          ts = tile_sum_compact(L, four[q], lane);
          if (lane == 0) tsum[four[q]] = ts;
        }
      }
    }
    wave_sync();
    const int bq = o.set ? tq / WAVE : -1;
    for (unsigned long long m2 = tm; m2;) {
      const int bb = __builtin_amdgcn_readlane(bq, __ffsll((long long)m2) - 1);
      m2 &= ~__ballot(bq == bb);
      const int tt = bb * WAVE + lane;
      const double v = wave_sum_dpp(tt < D.ntiles ? tsum[tt] : 0.0);
      if (lane == 0) bsum[bb] = v;
    }
    wave_sync();
  }
  if (lane == 0) {
    st->clock = clock;
    st->events = events;
    st->log_n += nev;
    st->stop = stop;
    if (err) st->err = err;
  }
  if (lane < 8) st->counts[lane] += my_cnt;
}

// ---- adjoint: replay with per-class accounting ---------------------------------
// For a recorded trajectory {(event k, dt_k)} the log-likelihood is
//   sum_k [ log r(event k) - R_k dt_k ]  with R_k = sum_c n_c(k) r_c,
// where n_c(k) is the number of points whose rate comes from class c before
// event k.  Replaying the log, this kernel accumulates S_c (selections of
// class c) and A_c = sum_k n_c(k) dt_k; the likelihood and its gradient with
// respect to any parameter of the rate tables follow on the host as
// sum_c S_c log r_c - A_c r_c.  A_c is accumulated lazily per class in LDS
// (A_c += n_c (t - tau_c) whenever n_c changes) on a clock that restarts
// every ADJ_EPOCH events, so that the interval lengths keep full precision.
constexpr int ADJ_EPOCH = 1024;
constexpr int ADJ_NS = KEY_N + 9;  // + deposition of species s at coordination c
struct AdjDesc {
  Lattice L;                 // L.key set
  int32_t *key_seen;         // key each point was last accounted under
  float *rate_seen;          // its rate then (isolated atoms)
  const mskg_event *log;
  const double *dt;
  long long n;
  int *cnt0;                 // [KEY_N + 1] initial class populations, then the unsupported points
  double *iso0;              // initial sum of isolated-atom rates
  int *sweep_err;            // the rate sweep's error flag (the engine's)
  int fresh;                 // the keys are not current: a rate sweep first
  double *S;                 // [ADJ_NS]
  double *A;                 // [KEY_N]
  double *scal;              // [4]: sum dt, integral of isolated rates, sum of their log rates, events
  RunState *st;
  int32_t *hist;             // may be null: [n / every][KEY_N] class populations after every `every` events
  long long every;
  double *acc;               // [2][KEY_N]: each class's population integral, then the time of its last change
};

__global__ void __launch_bounds__(WAVE) k_adjoint(const AdjDesc *descs) {
  extern __shared__ unsigned char smem[];
  int *cnt = (int *)smem;                 // [KEY_N] class populations
  __shared__ TabLds tabs;
  const int lane = threadIdx.x;
  AdjDesc D = descs[blockIdx.x];
  D.key_seen = as_global(D.key_seen);
  D.rate_seen = as_global(D.rate_seen);
  D.log = as_global(D.log);
  D.dt = as_global(D.dt);
  D.S = as_global(D.S);
  D.acc = as_global(D.acc);
  Lattice L = D.L;
  to_global(L);
  load_tables<false>(*L.tab, tabs, lane);
  // the per-class integrals and change times in the segment's own device
  // memory (LDS holds the populations only, so that more waves fit a CU)
  double *const A = D.acc, *const tau = D.acc + KEY_N;
  for (int c = lane; c < KEY_N; c += WAVE) {
    A[c] = 0.0;
    tau[c] = 0.0;
    cnt[c] = D.cnt0[c];
  }
  for (int c = lane; c < ADJ_NS; c += WAVE) D.S[c] = 0.0;
  wave_sync();
  double t = 0.0, ttot = 0.0, r_iso = *D.iso0, tau_iso = 0.0, iso_int = 0.0, iso_log = 0.0;
  int err = 0;
  long long k = 0;
  // the log is read one event ahead: its loads overlap the event before
  mskg_event ev_next;
  double dt_next = 0.0;
  if (D.n > 0) {
    ev_next = D.log[0];
    dt_next = D.dt[0];
  }
  for (; k < D.n; k++) {
    const mskg_event ev = ev_next;
    const double dtk = dt_next;
    if (k + 1 < D.n) {
      ev_next = D.log[k + 1];
      dt_next = D.dt[k + 1];
    }
    t += dtk;
    ttot += dtk;
    const P3 s = at(L, __builtin_amdgcn_readfirstlane(ev.site[0]), __builtin_amdgcn_readfirstlane(ev.site[1]),
                    __builtin_amdgcn_readfirstlane(ev.site[2]));
    const int itrans = __builtin_amdgcn_readfirstlane(ev.itrans);
    if (s.i < 0) { err = ERR_NOT_MC; break; }
    // the site's class, key and record in one round trip
    const int cs = L.cls[s.i], ks = __builtin_amdgcn_readfirstlane(D.key_seen[s.i]);
    const Rec srec = uniform_rec(load_rec(L, s.i));
    if (__builtin_amdgcn_readfirstlane(cs) == 0) err = ERR_NOT_MC;
    else if (ks < 0) err = ERR_COVERAGE;  // a rate class the likelihood does not cover
    else if (ks >= KEY_ADS && ks < KEY_PH && (itrans < 1 || itrans > 3)) err = ERR_NOT_MC;
    if (err) break;
    if (lane == 0) {
      // the selections by class: no return value, the wave does not wait
      const int sk = ks >= KEY_ADS && ks < KEY_PH ? KEY_N + (itrans - 1) * 3 + (ks - KEY_ADS) : ks;
      atomicAdd(&D.S[sk], 1.0);
      if (ks == KEY_ISO) iso_log += log((double)D.rate_seen[s.i]);
    }
    Choice ch;
    ch.arm = __builtin_amdgcn_readfirstlane(ev.arm);
    ch.u_arm = 0.0;
    EvOut out;
    execute<false, false>(L, tabs, ev.rtot, s, srec, itrans, ch, out, lane);  // the likelihood excludes LA and coverage tables
    wave_sync();
    // the touched points' keys and rates, before and after, a lane each (a
    // point listed twice is taken once); every class change of the event
    // happens at time t, so the accounting below does not depend on order
    int o = -3, nw = -1;  // o = -3: a point an earlier lane holds (or none)
    float ro = 0.0f, rn = 0.0f;
    if (out.set) {
      o = D.key_seen[out.p.i];
      nw = L.key[out.p.i];
      ro = D.rate_seen[out.p.i];
      rn = L.rate[out.p.i];
    }
    if (__ballot(out.set == 2)) {  // repeated list entries, or the site among them
      bool dup = false;
      for (int q = -1; q < 4; q++) {
        const int l = q < 0 ? 0 : 4 * q + 1;
        const int lo = __builtin_amdgcn_readlane((int)(uint32_t)out.p.i, l);
        const int hi = __builtin_amdgcn_readlane((int)(out.p.i >> 32), l);
        const int on = __builtin_amdgcn_readlane(out.set, l);
        dup |= on && l < lane && lo == (int)(uint32_t)out.p.i && hi == (int)(out.p.i >> 32);
      }
      if (dup) o = -3;
    }
    if (out.set && o != -3) {
      D.key_seen[out.p.i] = nw;
      D.rate_seen[out.p.i] = rn;
    }
    int bad = __builtin_amdgcn_readfirstlane(out.err);
    if (!bad && __ballot(o != -3 && nw == KEY_UNSUPPORTED)) bad = ERR_COVERAGE;
    if (!bad) {
      // Every class change of the event happens at time t: a class's
      // integral takes its population up to t once (a second change at t
      // adds population x 0), so the earliest lane holding a class, as old
      // or new class in touched order, updates it with the population before
      // the event, and the populations then change by atomics.
      const bool chg = o != -3 && o != nw;
      const int co = chg && o >= 0 ? o : -1, cn = chg && nw >= 0 ? nw : -1;
      bool do_o = co >= 0, do_n = cn >= 0;
      for (unsigned long long cm = __ballot(chg); cm; cm &= cm - 1ull) {
        const int q = __ffsll((long long)cm) - 1;
        const int qo = __builtin_amdgcn_readlane(co, q), qn = __builtin_amdgcn_readlane(cn, q);
        if (q < lane) {
          if (qo == co || qn == co) do_o = false;
          if (qo == cn || qn == cn) do_n = false;
        }
      }
      if (do_o) { A[co] += cnt[co] * (t - tau[co]); tau[co] = t; }
      if (do_n) { A[cn] += cnt[cn] * (t - tau[cn]); tau[cn] = t; }
      wave_sync();  // every first update has read its population
      if (co >= 0) atomicAdd(&cnt[co], -1);
      if (cn >= 0) atomicAdd(&cnt[cn], 1);
      // the isolated-atom rate sum changes in touched order (rare)
      const double roq = o == KEY_ISO ? (double)ro : 0.0, rnq = nw == KEY_ISO ? (double)rn : 0.0;
      for (unsigned long long im = __ballot(o != -3 && roq != rnq); im; im &= im - 1ull) {
        const int q = __ffsll((long long)im) - 1;
        iso_int += r_iso * (t - tau_iso);
        tau_iso = t;
        r_iso += read_lane(rnq, q) - read_lane(roq, q);
      }
    }
    wave_sync();
    if (bad) { err = bad; k++; break; }
    if (D.hist && (k + 1) % D.every == 0) {  // checkpoint: the class populations after event k
      int32_t *row = D.hist + ((k + 1) / D.every - 1) * KEY_N;
      for (int c = lane; c < KEY_N; c += WAVE) row[c] = cnt[c];
    }
    if ((k + 1) % ADJ_EPOCH == 0) {  // restart the accounting clock
      for (int c = lane; c < KEY_N; c += WAVE) {
        A[c] += cnt[c] * (t - tau[c]);
        tau[c] = 0.0;
      }
      iso_int += r_iso * (t - tau_iso);
      tau_iso = 0.0;
      t = 0.0;
      wave_sync();
    }
  }
  for (int c = lane; c < KEY_N; c += WAVE) D.A[c] = A[c] + cnt[c] * (t - tau[c]);
  if (lane == 0) {
    iso_int += r_iso * (t - tau_iso);
    D.scal[0] = ttot;
    D.scal[1] = iso_int;
    D.scal[2] = iso_log;
    D.scal[3] = (double)k;
    if (err) D.st->err = err;
  }
}

// Before the replay: each segment's rate-sweep error and unsupported-point
// count (out[2i], out[2i + 1]); after it: each replica's run error (out[i]).
__global__ void __launch_bounds__(256) k_adj_check(const AdjDesc *descs, int n, int *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[2 * i] = descs[i].sweep_err[0];
  out[2 * i + 1] = descs[i].cnt0[KEY_N];
}
__global__ void __launch_bounds__(256) k_adj_errs(const AdjDesc *descs, int n, int *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = descs[i].st->err;
}

// Every segment's start in one launch (block row y: segment y): the rates and
// keys where they are not current, the class populations and isolated-rate
// sum, and the keys and rates as first seen, four points a thread.  What
// bounds it: the records' bytes where a sweep is needed (21 and 16 more a
// point); a launch and two copies a segment had left most of the chip idle
// (128 lattices of 144^3: 3.1 ms of device time and 640 calls).
__global__ void __launch_bounds__(64) k_adj_clear(const AdjDesc *descs, int n) {
  const int i = blockIdx.x;
  for (int c = threadIdx.x; c < KEY_N + 1; c += blockDim.x) descs[i].cnt0[c] = 0;
  if (threadIdx.x == 0) {
    *descs[i].iso0 = 0.0;
    *descs[i].sweep_err = 0;
  }
}
template <bool LA, bool COV>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_adj_start(const AdjDesc *descs) {
  const AdjDesc &D = descs[blockIdx.y];
  Lattice L = D.L;
  to_global(L);
  const double rtot = D.st->rtot;
  const int64_t n = L.box.npts, stride = (int64_t)gridDim.x * blockDim.x * 4;
  for (int64_t p0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4; p0 < n; p0 += stride) {
    if (D.fresh) sweep_group<LA, COV>(L, rtot, D.sweep_err, 0, p0, n);
    for (int64_t p = p0; p < n && p < p0 + 4; p++) {
      const int k = L.key[p];
      const float r = L.rate[p];
      D.key_seen[p] = k;
      D.rate_seen[p] = r;
      if (k == KEY_ISO) atomicAdd(D.iso0, (double)r);
      if (k >= 0) atomicAdd(&D.cnt0[k], 1);
      else if (k == KEY_UNSUPPORTED) atomicAdd(&D.cnt0[KEY_N], 1);
    }
  }
}

// ---- frame compaction (the xyz output of inpout/WriteMolMolXYZFile.f) --------
// Ordered record lists in the reference's grid order (z, then y, then x; the
// stored-point order restricted to one z plane is the same), z <= LenZ-1.
// FRAME_MAIN, the main and _d frames:
//   list 0 the points the main frame lists: coverage species and atoms of
//     coordination <= 3 (WriteMolMolXYZFile.f:131-166);
//   list 1 vacancies (empty, coordination 4);
//   list 2 non-epitaxial bulk atoms: coordination 4 off the cubic diamond
//     sites (the _d frame, :77-121);
//   and two header counts over z = 1..LenZ-1 (:93-110): atoms of
//   coordination <= 3, covered points.
// FRAME_DEFECTS, the SiC defect frames:
//   list 0 vacancies with the species sum of their four listed neighbours
//     (the _v frame's classification, :222-260);
//   list 1 the _w frame (:264-398): bulk atoms with z = 1..LenZ-1 and three
//     first neighbours of the other species (Si around C, C around Si), read
//     while the isolated wrong atoms -- bulk atoms with no such neighbour --
//     are flipped to the other species; code = the species as flipped.
//     k_wrong_set marks those flips (bit 7 of the record's `valid` byte,
//     which the neighbour lists leave unused) and clears the marks after.
// Each wave owns a contiguous segment of points: k_frame_count counts it and
// leaves a bit a point for the points that have a record, k_frame_scan turns
// the counts into offsets, k_frame_write writes in order.
//
// What bounds it: the records' bytes, read once, by the count; the write
// reads a bit a point and the records of the few points that have one.  A
// lattice a slab builder made and runs have changed since is read only over
// the planes those runs could have touched (touched_planes).  With every
// stored plane read by the count and again by the write, 65536 points a block
// whatever the lattice, and a sizing call before each frame, a whole pass
// (build, run, frames) took 63.6 ms at 512^3 SiC, now 52.4; Si PVD 768^2 x
// 1536 53.0, now 50.5; 24 SiGe replicas 54.8, now 36.1; the smallest box 8.7,
// now 8.2.
constexpr int FRAME_THREADS = 256;
constexpr uint32_t NO_POINT = 0xffffffffu;  // in the place of a record's last word (whose temperature has 13 bits)
constexpr int FRAME_GROUPS = 64;  // groups of 64 points a wave takes at a time: a lane's bits each
enum : int { FRAME_MAIN = 0, FRAME_DEFECTS = 1, FRAME_STATE = 2 };
template <int MODE> struct FrameShape;
template <> struct FrameShape<FRAME_MAIN> { static constexpr int NLIST = 3, NCNT = 5; };
template <> struct FrameShape<FRAME_DEFECTS> { static constexpr int NLIST = 2, NCNT = 2; };
template <> struct FrameShape<FRAME_STATE> { static constexpr int NLIST = 3, NCNT = 3; };
constexpr uint8_t WRONG_FLIP = 0x80;

// Species of a record as the _w analysis sees it: the wrong-site flip swaps
// Si (1) and C (2).
__device__ inline int flipped_species(const Site &s) {
  const int k = s_kind(s);
  return (s.valid & WRONG_FLIP) ? 3 - k : k;
}
// NCoorCorr (WriteMolMolXYZFile.f:284-296) of a bulk atom: its listed
// neighbours carrying the other species' bit (the C bit around Si, the Si
// bit around C), with the flips marked or not.
__device__ inline int wrong_corr(const Lattice &L, const P3 &pt, const Site &sp, bool flips) {
  const int k = flips ? flipped_species(sp) : s_kind(sp);
  const NL l = list_of(L, pt, sp);
  int corr = 0;
  for (int i = 0; i < 4; i++) {
    const Site q = rd(L, entry(L, l, i).i);
    int kq = s_kind(q);
    if (!kind_species(kq)) continue;
    if (flips) kq = flipped_species(q);
    corr += (k == 1) ? ((kq >> 1) & 1) : (k == 2 ? (kq & 1) : 0);
  }
  return corr;
}

// Membership of point p, whose record's last word is w, in the lists of a
// frame, the code per list and the header counts.
template <int MODE>
__device__ inline void frame_point(const Lattice &L, int64_t p, uint32_t w, int sic, bool in[], int code[],
                                   unsigned int cnt[]) {
  const int kind = w & 7, coor = (w >> 3) & 7;
  for (int k = 0; k < FrameShape<MODE>::NLIST; k++) {
    in[k] = false;
    code[k] = 0;
  }
  const bool atom = kind_species(kind), covered = kind >= KIND_COV0;
  const bool below = p < L.box.plane * L.box.lz;  // z <= LenZ-1
  if (w == NO_POINT) return;
  if (MODE == FRAME_STATE) {
    // the reference's lists: an atom of coordination <= 3 is an MC particle
    // even when it has no rate (a frozen-substrate atom)
    in[0] = (atom && coor <= 3) || L.cls[p] != 0;
    in[1] = !in[0] && atom;
    in[2] = !in[0] && !atom && kind != KIND_WALL && coor == 4;
  } else if (MODE == FRAME_MAIN) {
    if (!below) return;
    const bool inner = p >= L.box.plane;  // z >= 1
    in[0] = covered || (atom && coor <= 3);  // a covered vacancy is also listed in the main frame
    in[1] = coor == 4 && (covered || kind == KIND_EMPTY);
    if (atom && coor > 3) {
      int x, y, z;
      pxyz(L.box, p, x, y, z);
      in[2] = !dia_type(x, y, z);
    }
    code[0] = covered ? -kind_cov_slot(kind) : kind;  // the host maps a coverage slot to ListCov
    code[2] = kind;
    cnt[3] += in[0] && atom && inner;
    cnt[4] += covered && inner;
  } else if (below && coor == 4 && kind != KIND_WALL) {
    P3 pt;
    pt.i = p;
    pxyz(L.box, p, pt.x, pt.y, pt.z);
    if (!atom) {  // a vacancy: the species sum of its neighbours
      const NL l = list_of(L, pt, L.site[p]);
      int sum = 0;
      for (int i = 0; i < 4; i++) {
        const int kq = s_kind(rd(L, entry(L, l, i).i));
        sum += kind_species(kq) ? kq : 0;
      }
      in[0] = true;
      code[0] = sum;
    } else if (sic && pt.z >= 1) {
      const Site sp = L.site[p];
      in[1] = wrong_corr(L, pt, sp, true) == 3;
      code[1] = flipped_species(sp);
    }
  }
  for (int k = 0; k < FrameShape<MODE>::NLIST; k++) cnt[k] += in[k];
}

// The groups of 64 points from g0 (at most FRAME_GROUPS of them, below end):
// lane g gets the bits of group g's points that are in a list; cnt counts.
// Four records' words in flight a lane.
template <int MODE>
__device__ inline unsigned long long frame_bits(const Lattice &L, int64_t g0, int64_t end, int groups, int sic,
                                                unsigned int cnt[], int lane) {
  unsigned long long mine = 0ull;
  for (int g = 0; g < groups && g0 + g * WAVE < end; g += 4) {
    uint32_t w[4];
    for (int u = 0; u < 4; u++) {
      const int64_t p = g0 + (int64_t)(g + u) * WAVE + lane;
      w[u] = g + u < groups && p < end ? ((const uint32_t *)(L.site + p))[3] : NO_POINT;
    }
    for (int u = 0; u < 4; u++) {
      bool in[FrameShape<MODE>::NLIST];
      int code[FrameShape<MODE>::NLIST];
      frame_point<MODE>(L, g0 + (int64_t)(g + u) * WAVE + lane, w[u], sic, in, code, cnt);
      bool any = false;
      for (int k = 0; k < FrameShape<MODE>::NLIST; k++) any |= in[k];
      const unsigned long long m = __ballot(any);
      if (lane == g + u) mine = m;
    }
  }
  return mine;
}

// The isolated wrong atoms of the SiC analysis (WriteMolMolXYZFile.f:269-299).
// The reference visits the bulk atoms in grid order and flips each one with
// no neighbour of the other species on the spot, so a flip is seen by the
// atoms visited after it.  A flip only raises its neighbours' counts (its
// neighbours share its species until it flips), so an atom flips iff it has
// no neighbour of the other species to begin with (a candidate) and no
// candidate neighbour before it in grid order flips: the candidates are few,
// k_wrong_cand lists them with their neighbours, the host resolves that
// order, and k_wrong_set marks (or unmarks) the flips.
__global__ void __launch_bounds__(256) k_wrong_cand(Lattice L, int64_t first, int64_t end, int64_t cap,
                                                    unsigned long long *n, int4 *out) {
  for (int64_t p = first + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < end;
       p += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t w = ((const uint32_t *)(L.site + p))[3];
    const int kind = w & 7;
    if (!(kind == 1 || kind == 2) || ((w >> 3) & 7) != 4) continue;
    const Site sp = L.site[p];
    P3 pt;
    pt.i = p;
    pxyz(L.box, p, pt.x, pt.y, pt.z);
    if (pt.z < 1 || pt.z > L.box.lz - 1 || wrong_corr(L, pt, sp, false) != 0) continue;
    const unsigned long long i = atomicAdd(n, 1ull);
    if ((int64_t)i >= cap) continue;  // counted; the host grows the list and asks again
    const NL l = list_of(L, pt, sp);
    out[5 * i] = make_int4(pt.x, pt.y, pt.z, 0);
    for (int k = 0; k < 4; k++) out[5 * i + 1 + k] = make_int4(l.x[k], l.y[k], l.z[k], 0);
  }
}
__global__ void __launch_bounds__(256) k_wrong_set(Lattice L, const int4 *pos, int64_t n, int set) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = pidx(L.box, pos[i].x, pos[i].y, pos[i].z);
    const uint8_t v = L.site[p].valid;
    L.site[p].valid = (uint8_t)(set ? (v | WRONG_FLIP) : (v & ~WRONG_FLIP));
  }
}

// The points of a frame's kernels and how its waves share them: segment i is
// the points [first + i * rounds * groups * 64, ...) below end, `rounds`
// times `groups` groups of 64 points.
struct FramePlan {
  int64_t first, end;
  int groups, rounds;
  int nseg;
  int sic;
};

// counts: [NCNT][nseg]; bits: a word a group of 64 points, null: not kept.
template <int MODE>
__global__ void __launch_bounds__(FRAME_THREADS) k_frame_count(Lattice L, FramePlan F, uint32_t *counts,
                                                               unsigned long long *bits) {
  constexpr int NC = FrameShape<MODE>::NCNT;
  const int lane = threadIdx.x & (WAVE - 1);
  const int seg = blockIdx.x * (FRAME_THREADS / WAVE) + threadIdx.x / WAVE;
  if (seg >= F.nseg) return;
  unsigned int c[NC];
  for (int k = 0; k < NC; k++) c[k] = 0u;
  for (int r = 0; r < F.rounds; r++) {
    const int64_t grp = ((int64_t)seg * F.rounds + r) * F.groups, g0 = F.first + grp * WAVE;
    if (g0 >= F.end) break;
    const unsigned long long mine = frame_bits<MODE>(L, g0, F.end, F.groups, F.sic, c, lane);
    if (bits && lane < F.groups && g0 + (int64_t)lane * WAVE < F.end) bits[grp + lane] = mine;
  }
  for (int k = 0; k < NC; k++) {
    unsigned int v = c[k];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
    if (lane == 0) counts[(int64_t)k * F.nseg + seg] = v;
  }
}

// Calls put(list, place, point, x, y, z, code) for every record of a wave's
// segment.  The groups are taken a lane each: a lane reads its group's listed
// points one after the other, once to count them by list and once to write.
template <int MODE, class Put>
__device__ inline void frame_put(const Lattice &L, const FramePlan &F, const unsigned long long *bits,
                                 const unsigned long long *offs, Put put) {
  constexpr int NL_ = FrameShape<MODE>::NLIST, NC = FrameShape<MODE>::NCNT;
  const int lane = threadIdx.x & (WAVE - 1);
  const int seg = blockIdx.x * (FRAME_THREADS / WAVE) + threadIdx.x / WAVE;
  if (seg >= F.nseg) return;
  unsigned long long base[NL_];
  for (int k = 0; k < NL_; k++) base[k] = offs[(int64_t)k * F.nseg + seg];
  for (int r = 0; r < F.rounds; r++) {
    const int64_t grp = ((int64_t)seg * F.rounds + r) * F.groups, g0 = F.first + grp * WAVE;
    if (g0 >= F.end) break;
    unsigned long long mine = 0ull;
    unsigned int dummy[NC];
    for (int k = 0; k < NC; k++) dummy[k] = 0u;
    if (!bits) mine = frame_bits<MODE>(L, g0, F.end, F.groups, F.sic, dummy, lane);
    else if (lane < F.groups && g0 + (int64_t)lane * WAVE < F.end) mine = bits[grp + lane];
    if (!__ballot(mine != 0ull)) continue;
    const int64_t pl = g0 + (int64_t)lane * WAVE;
    bool in[NL_];
    int code[NL_];
    unsigned int n[NC];
    for (int k = 0; k < NC; k++) n[k] = 0u;
    for (unsigned long long m = mine; m; m &= m - 1ull) {
      const int64_t p = pl + __ffsll((long long)m) - 1;
      frame_point<MODE>(L, p, ((const uint32_t *)(L.site + p))[3], F.sic, in, code, n);
    }
    unsigned long long at[NL_];
    for (int k = 0; k < NL_; k++) {
      unsigned int inc = n[k];
      for (int off = 1; off < WAVE; off <<= 1) {
        const unsigned int t = __shfl_up(inc, off, WAVE);
        if (lane >= off) inc += t;
      }
      at[k] = base[k] + inc - n[k];
      base[k] += __shfl(inc, WAVE - 1, WAVE);
    }
    for (unsigned long long m = mine; m; m &= m - 1ull) {
      const int64_t p = pl + __ffsll((long long)m) - 1;
      frame_point<MODE>(L, p, ((const uint32_t *)(L.site + p))[3], F.sic, in, code, dummy);
      int x, y, z;
      pxyz(L.box, p, x, y, z);
      for (int k = 0; k < NL_; k++)
        if (in[k]) {
          put(k, at[k], p, x, y, z, code[k]);
          at[k]++;
        }
    }
  }
}
template <int MODE>
__global__ void __launch_bounds__(FRAME_THREADS) k_frame_write(Lattice L, FramePlan F, const unsigned long long *bits,
                                                               const unsigned long long *offs, int4 *out0,
                                                               int4 *out1, int4 *out2, int64_t cap0, int64_t cap1,
                                                               int64_t cap2) {
  int4 *const outs[3] = {out0, out1, out2};
  const unsigned long long caps[3] = {(unsigned long long)cap0, (unsigned long long)cap1, (unsigned long long)cap2};
  frame_put<MODE>(L, F, bits, offs, [&](int k, unsigned long long at, int64_t, int x, int y, int z, int code) {
    if (at < caps[k]) outs[k][at] = make_int4(x, y, z, code);
  });
}

// The segments' offsets of a frame from their counts, and the totals (NCNT
// of them): a block a count, which scans its segments 4096 at a time.
constexpr int SCAN_THREADS = 1024;
template <int MODE>
__global__ void __launch_bounds__(SCAN_THREADS) k_frame_scan(const uint32_t *counts, int nseg,
                                                             unsigned long long *offs, int64_t *totals) {
  __shared__ unsigned long long wsum[SCAN_THREADS / WAVE];
  const int k = blockIdx.x, lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const uint32_t *const c = counts + (int64_t)k * nseg;
  unsigned long long *const o = k < FrameShape<MODE>::NLIST ? offs + (int64_t)k * nseg : nullptr;
  unsigned long long base = 0ull;
  for (int s0 = 0; s0 < nseg; s0 += 4 * SCAN_THREADS) {
    const int i0 = s0 + 4 * (int)threadIdx.x;
    uint32_t v[4];
    for (int u = 0; u < 4; u++) v[u] = i0 + u < nseg ? c[i0 + u] : 0u;
    const unsigned long long mine = (unsigned long long)v[0] + v[1] + v[2] + v[3];
    unsigned long long inc = mine;
    for (int off = 1; off < WAVE; off <<= 1) {
      const unsigned long long t = __shfl_up(inc, off, WAVE);
      if (lane >= off) inc += t;
    }
    if (lane == WAVE - 1) wsum[w] = inc;
    __syncthreads();
    unsigned long long before = base, all = 0ull;
    for (int q = 0; q < SCAN_THREADS / WAVE; q++) {
      if (q < w) before += wsum[q];
      all += wsum[q];
    }
    unsigned long long at = before + inc - mine;
    for (int u = 0; u < 4; u++) {
      if (o && i0 + u < nseg) o[i0 + u] = at;
      at += v[u];
    }
    base += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) totals[k] = (int64_t)base;
}

// Scratch of the allocation-free frame entry point (mskg_frame_device): the
// counts (5 a segment, 32 bits) and offsets (3 a segment) of one frame.  Every
// GPU the library runs on holds its own copy until the process ends; host
// code reaches it only through the address hipGetSymbolAddress gives for the
// device (noalloc_scratch), never through the array's name.
constexpr int NOALLOC_FRAME_BLOCKS = 16384;       // segments at most
constexpr int64_t NOALLOC_MAX_CHUNK = 1ll << 30;  // lattice points a segment
static __device__ __align__(256) unsigned long long scratch[NOALLOC_FRAME_BLOCKS * 8];

// ---- the host's arrays: LattCoo words and particle lists ------------------------
// The reference's lists out of the lattice (xyz, NextNXYZ; of MC particles
// also Ind_Event and ProbTrans), and LattCoo's words in and out.  The device
// reads and writes the records; the host copies 4 bytes a lattice point and
// the lists, where it had copied every point's 21 bytes and gone through them
// point by point: the whole exchange (load, 1e5 events, store) of CVD at
// 240x240x760 took 346 ms, now 70.
struct StateOut {
  int32_t *xyz[3], *nn[3];
  int32_t *event;
  double *prob;
};
__global__ void __launch_bounds__(FRAME_THREADS) k_state_write(Lattice L, FramePlan F, const unsigned long long *bits,
                                                               const unsigned long long *offs, StateOut O) {
  frame_put<FRAME_STATE>(L, F, bits, offs, [&](int k, unsigned long long at, int64_t p, int x, int y, int z, int) {
    int32_t *const q = O.xyz[k] + 3 * at, *const w = O.nn[k] + 12 * at;
    q[0] = x; q[1] = y; q[2] = z;
    const NL l = site_list(L.box, L.site[p], x, y, z);
    for (int i = 0; i < 4; i++) {
      w[3 * i] = l.x[i];
      w[3 * i + 1] = l.y[i];
      w[3 * i + 2] = l.z[i];
    }
    if (k == 0) {
      const int c = L.cls[p];
      O.event[at] = (c == CLS_EVAP || c == CLS_ISOLATED || !c) ? 4 : c == CLS_DESORB ? 5 : 1;
      O.prob[at] = (double)L.rate[p];
    }
  });
}

// LattCoo's coverage indices by slot.
struct CovList {
  int n, index[3];
};
// The content of a LattCoo word; < 0: not representable.
MSKG_HD int word_kind(const CovList &C, int32_t v) {
  const int cov = v & 255, occ = (v >> 23) & 1, sic = (v >> 27) & 7;
  if (cov == 113) return KIND_WALL;
  if (cov != 0) {
    if (occ) return -1;
    for (int k = 0; k < C.n; k++)
      if (C.index[k] == cov) return KIND_COV0 + k;
    return -2;
  }
  if (occ) return sic < 1 || sic > 3 ? -3 : sic;
  return sic ? -4 : KIND_EMPTY;
}
__global__ void __launch_bounds__(256) k_words_out(Lattice L, CovList C, int64_t first, int64_t end, int32_t *out) {
  for (int64_t p = first + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < end;
       p += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t w = ((const uint32_t *)(L.site + p))[3];
    const int kind = w & 7;
    uint32_t v = 0u;
    if (kind == KIND_WALL) v = (1u << 23) | 113u;
    else if (kind_species(kind)) v = (1u << 23) | ((uint32_t)kind << 27);
    else if (kind >= KIND_COV0) v = (uint32_t)C.index[kind - KIND_COV0];
    v |= ((w >> 3) & 7u) << 24;
    v |= (w >> 16) << 9;
    out[p - first] = (int32_t)v;
  }
}
// What a piece of LattCoo (grid points g0..g0+n-1) holds that matters before
// any of it is taken: out[0] the first lattice point that is no site state,
// out[1] whether there are walls off the lattice.
__global__ void __launch_bounds__(256) k_words_check(Box b, CovList C, const int32_t *latt, int64_t g0, int64_t n,
                                                     unsigned long long *out) {
  const int64_t face = (int64_t)b.lx * b.ly;
  const double inv_face = 1.0 / (double)face, inv_lx = 1.0 / (double)b.lx;
  bool walls = false;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t v = latt[i];
    if (v == 0) continue;
    const int64_t g = g0 + i, z = div_by(g, face, inv_face), r = g - z * face;
    const int y = (int)div_by(r, b.lx, inv_lx), x = (int)(r - (int64_t)y * b.lx);
    if (valid_parity(x, y, (int)z)) {
      if (word_kind(C, v) < 0) atomicMin(&out[0], (unsigned long long)g);
    } else {
      walls |= (v & 255) == 113;
    }
  }
  if (__ballot(walls) && (threadIdx.x & (WAVE - 1)) == 0) atomicOr(&out[1], 1ull);
}
// The records of the lattice points first..end-1 from their words (latt: from
// grid point g0 on): no list, no rate.
__global__ void __launch_bounds__(256) k_words_in(Lattice L, CovList C, const int32_t *latt, int64_t g0, int64_t first,
                                                  int64_t end) {
  for (int64_t p = first + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < end;
       p += (int64_t)gridDim.x * blockDim.x) {
    int x, y, z;
    pxyz(L.box, p, x, y, z);
    const uint32_t v = (uint32_t)latt[(int64_t)x + (int64_t)L.box.lx * ((int64_t)y + (int64_t)L.box.ly * z) - g0];
    const uint32_t w = (uint32_t)word_kind(C, (int32_t)v) | (((v >> 24) & 7u) << 3) | (((v >> 9) & 0x1fffu) << 16);
    store_rec(L, p, make_rec(0u, 0u, 0u, w));
    L.rate[p] = 0.0f;
    L.cls[p] = 0;
  }
}
// The walls off the lattice of that piece, one bit per grid point (g0 and, but
// at the grid's end, n multiples of 32): a wave 64 points at a time.
__global__ void __launch_bounds__(256) k_words_offwall(Box b, const int32_t *latt, int64_t g0, int64_t n,
                                                       uint32_t *bits) {
  const int64_t face = (int64_t)b.lx * b.ly, words = (n + 31) / 32, pairs = (words + 1) / 2;
  const double inv_face = 1.0 / (double)face, inv_lx = 1.0 / (double)b.lx;
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
  for (int64_t q = wave; q < pairs; q += (int64_t)gridDim.x * (blockDim.x / WAVE)) {
    const int64_t i = q * WAVE + lane, g = g0 + i;
    bool wall = i < n && (latt[i] & 255) == 113;
    if (wall) {
      const int64_t z = div_by(g, face, inv_face), r = g - z * face;
      const int y = (int)div_by(r, b.lx, inv_lx), x = (int)(r - (int64_t)y * b.lx);
      wall = !valid_parity(x, y, (int)z);
    }
    const unsigned long long m = __ballot(wall);
    if (lane < 2 && 2 * q + lane < words) bits[g0 / 32 + 2 * q + lane] = (uint32_t)(m >> (32 * lane));
  }
}
// A listed particle: its neighbour list, and with cls >= 0 its class and rate.
struct StateRec {
  int64_t p;
  uint32_t x, y, z, valid;
  float rate;
  int cls;
};
__global__ void __launch_bounds__(256) k_lists_in(Lattice L, const StateRec *rec, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const StateRec r = rec[i];
  Rec s = load_rec(L, r.p);
  s.x = r.x;
  s.y = r.y;
  s.z = r.z;
  s.w = (s.w & ~0xff00u) | (r.valid << 8);
  store_rec(L, r.p, s);
  if (r.cls >= 0) {
    L.rate[r.p] = r.rate;
    L.cls[r.p] = (uint8_t)r.cls;
  }
}

// ---- census: atoms by species and covered points by coverage slot ---------
// Every deposition adds one atom of its species and every evaporation
// removes one (absorption / desorption likewise for coverage), so the
// evaporations and desorptions by species since a state was loaded follow
// from the depositions and absorptions counted by the events and the
// census then and now, with no per-event work.
__global__ void __launch_bounds__(256) k_census(Lattice L, unsigned long long *out) {
  __shared__ unsigned long long s[6];
  if (threadIdx.x < 6) s[threadIdx.x] = 0ull;
  __syncthreads();
  unsigned long long c[6] = {0ull, 0ull, 0ull, 0ull, 0ull, 0ull};
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < L.box.npts;
       p += (int64_t)gridDim.x * blockDim.x) {
    const int k = s_kind(L.site[p]);
    if (kind_species(k)) c[k - 1]++;
    else if (kind_cov_slot(k)) c[2 + kind_cov_slot(k)]++;
  }
  for (int q = 0; q < 6; q++) {
    unsigned long long v = c[q];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
    if ((threadIdx.x & (WAVE - 1)) == 0 && v) atomicAdd(&s[q], v);
  }
  __syncthreads();
  if (threadIdx.x < 6 && s[threadIdx.x]) atomicAdd(&out[threadIdx.x], s[threadIdx.x]);
}

// ---- laser-annealing coupling: temperature map in, phase maps out ----------
// The laser-annealing build exchanges whole-grid int32 maps with its FEM
// driver: the temperature map b and the phase maps c (coordination) and d
// (species), DIMENSION(LenZ, LenX*LenY) (mulskips-source-LaserAnnealing/
// modules/defsystem.f:88-91), or the temperature file's planes
// (mulskips-source-LaserAnnealing/initial/SetT.f:56-66).  Both are read and
// written here on the device, so a cycle moves 4 B per grid point over PCIe
// instead of the lattice.
enum : int { FIELD_LATTCOO = 2 };  // x fastest over the LenZ+1 planes of LattCoo
MSKG_HD int64_t field_index(const Box &b, int layout, int x, int y, int z) {
  if (layout == MSKG_FIELD_SOCKET) return z + (int64_t)b.lz * (x + (int64_t)b.lx * y);
  return x + (int64_t)b.lx * (y + (int64_t)b.ly * z);
}

// Range check of a strict temperature map at the stored points (the 13 bits
// of LattCoo's T field), before anything is written.
__global__ void __launch_bounds__(256) k_check_field(Lattice L, const int32_t *f, int layout, int *err) {
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < L.box.npts;
       p += (int64_t)gridDim.x * blockDim.x) {
    int x, y, z;
    pxyz(L.box, p, x, y, z);
    const int32_t v = f[field_index(L.box, layout, x, y, z)];
    if (v < 0 || v > 8191) atomicExch(err, 1);
  }
}

// SetT.f:38-48 (the laser-annealing build): every point of the planes
// 0..LenZ-1 takes the low LenT = 13 bits of its map value (MVBITS), except
// where the value is 10, the FEM side's wall marker, which leaves the point
// as it is.  strict: the map
// covers LattCoo's LenZ+1 planes and every value is taken as it is (range
// checked before).  One thread per stored point, records read and written
// whole.
__global__ void __launch_bounds__(256) k_set_temperature(Lattice L, const int32_t *f, int layout, int strict) {
  const int64_t n = L.box.npts;
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
    int x, y, z;
    pxyz(L.box, p, x, y, z);
    if (!strict && z >= L.box.lz) continue;
    const int32_t v = f[field_index(L.box, layout, x, y, z)];
    if (!strict && v == 10) continue;
    Site s = L.site[p];
    s.temp = (uint16_t)(v & 8191);
    L.site[p] = s;
  }
}

// main.f:796-818 of the laser-annealing build: for the points of planes
// 0..LenZ-1, c = coordination and d = species of an occupied point, 10 and
// 10 on a wall (index 113), 0 and 0 elsewhere (grid points off the diamond
// super-lattice are never occupied).  Rows of the map (a z column of the
// socket layout, an x row of the plane layout) are strided over the grid;
// writes are in map order.
__global__ void __launch_bounds__(256) k_phases(Lattice L, int layout, const uint32_t *offwall, int wall_planes,
                                               int32_t *c, int32_t *d) {
  const Box &b = L.box;
  const int64_t rows = layout == MSKG_FIELD_SOCKET ? (int64_t)b.lx * b.ly : (int64_t)b.ly * b.lz;
  const int len = layout == MSKG_FIELD_SOCKET ? b.lz : b.lx;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    int x = 0, y = 0, z = 0;
    if (layout == MSKG_FIELD_SOCKET) {
      x = (int)(r % b.lx);
      y = (int)(r / b.lx);
    } else {
      y = (int)(r % b.ly);
      z = (int)(r / b.ly);
    }
    for (int k = threadIdx.x; k < len; k += blockDim.x) {
      if (layout == MSKG_FIELD_SOCKET) z = k;
      else x = k;
      int32_t cv = 0, dv = 0;
      if (valid_parity(x, y, z)) {
        const Site s = L.site[pidx(b, x, y, z)];
        const int kind = s_kind(s);
        if (kind == KIND_WALL) {
          cv = dv = 10;
        } else if (kind_species(kind)) {
          cv = s_coor(s);
          dv = kind;
        }
      } else {
        const int64_t g = x + (int64_t)b.lx * (y + (int64_t)b.ly * z);
        const bool wall = (offwall && ((offwall[g >> 5] >> (g & 31)) & 1)) ||
                          (wall_planes && (z <= 5 || (z >= b.lz - 6 && z <= b.lz - 1)));
        if (wall) cv = dv = 10;
      }
      const int64_t o = r * len + k;
      if (c) c[o] = cv;
      if (d) d[o] = dv;
    }
  }
}

// The kernel instance for a rate model (all four share one signature).
template <class F>
F pick_variant(bool la, bool cov, F tt, F tf, F ft, F ff) {
  return la ? (cov ? tt : tf) : (cov ? ft : ff);
}
#define MSKG_VARIANT(K, la, cov) pick_variant((la) != 0, (cov) != 0, K<true, true>, K<true, false>, K<false, true>, K<false, false>)

// ---- host side ---------------------------------------------------------------
#define HIPCHK(e, x)                                                                  \
  do {                                                                                \
    hipError_t _r = (x);                                                              \
    if (_r != hipSuccess) return fail_((e), MSKG_EDEVICE, "%s: %s", #x, hipGetErrorString(_r)); \
  } while (0)

}  // namespace

// Until a caller sets a schedule: one XCD's sweep where the rule says so
// (xcd_waves), else the colour passes.
constexpr int SCHEDULE_AUTO = -1;

struct mskg_engine {
  mskg_config cfg;
  bool cov_model = true;  // the kernels with the coverage-species branches
  Box box;               // the stored planes (all of them unless cfg.stored_len_z)
  int logical_lz = 0;    // the reference's LenZ
  bool windowed = false; // only the bottom planes are stored
  Geometry geo;
  Tables tab;
  int ncrystal, ncov, list_cov[3];
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // device memory
  Site *d_site = nullptr;
  float *d_rate = nullptr;
  uint8_t *d_cls = nullptr;
  uint8_t *d_inlist = nullptr;
  int32_t *d_tl_idx = nullptr;
  int32_t *d_tl_n = nullptr;
  int32_t *d_tl_own = nullptr;
  double *d_tile_r = nullptr;
  int32_t *d_field[2] = {nullptr, nullptr};  // grid-sized maps of the laser-annealing coupling (on first use)
  // walls on grid points off the diamond super-lattice (the reference's
  // builders fill whole wall regions), which only the phase maps report:
  // one bit per grid point from mskg_load_state (null: none), or the wall
  // planes of the device builders
  uint32_t *d_offwall = nullptr;
  bool offwall_planes = false;
  // InitSt 'ST' reference tables (one allocation: temperatures, then the tables)
  void *d_st_tables = nullptr;
  // census (atoms by species, covered points by slot) of the state as loaded
  int64_t census0[6] = {0, 0, 0, 0, 0, 0};
  int *d_list_err = nullptr;
  int *d_win = nullptr;
  // per-tile completion stamps of the dependency-scheduled sweep, then its
  // stamp / queue / window words (PassParams::done, ::sched)
  unsigned int *d_done = nullptr;
  int schedule = SCHEDULE_AUTO;
  Geometry *d_geo = nullptr;
  Tables *d_tab = nullptr;
  RunState *d_st = nullptr;
  int *d_err = nullptr;
  int device = 0;          // the HIP device the engine lives on
  int tile = 0, ntx = 0, nty = 0, ntz = 0, ntiles = 0, cap = 1024, capg = 512;
  int rsum_chunk = 1;      // tiles per block of the fixed-order tile sum
  bool lists_dirty = true;
  int pass_grid = 4096;  // workgroups per colour pass (they stride over the window)
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  mskg_event *d_log = nullptr;
  int64_t log_cap = 0;
  // serial mode: tile and block rate sums
  double *d_tsum = nullptr, *d_bsum = nullptr;
  // likelihood accounting: class key of every point, and as last accounted
  int32_t *d_key = nullptr, *d_key_seen = nullptr;
  float *d_rate_seen = nullptr;
  bool track = false;       // keep every point's class key current through runs
  bool keys_valid = false;  // d_key matches the rates (a keyed sweep or a tracked run since)
  double run_ms = 0, sweep_ms = 0;
  int64_t sweep_points = 0, sweeps_done = 0;
  bool loaded = false;
  // The planes [slab_z0, slab_z1] that may differ from the flat slab the
  // device builder wrote (slab: its mode; -1: some other state, of which
  // nothing is known): its surface, and 12 planes around every tile layer
  // that a run's sweeps could visit since.  An event's site lies in such a
  // layer, and it writes at most 6 planes from it.
  int slab = -1, slab_z0 = 0, slab_z1 = 0;
  bool flags_zero = false;   // no list flag is set at all: a slab was built, and no lists since
  bool flags_clean = false;  // no list flag outside the touched planes (d_inlist), while they are known
  // workspaces of the frames and of the exchange: kept while they are small (work_keep)
  void *d_work[2] = {nullptr, nullptr};
  size_t work_n[2] = {0, 0};
  std::string err;
};

static int fail_(mskg_engine *e, int code, const char *fmt, ...) {
  if (e) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    e->err = buf;
  }
  return code;
}

// cos/sin of DFLOAT(2*irot)*pi/3. with the REAL(4) pi of FIND_NN.f:27,
// evaluated with the host C library like the reference; the device uses
// these values rather than its own cos/sin.
static void build_geometry(Geometry &g) {
  const double pi = (double)3.14159265358979323f;
  for (int irot = 1; irot <= 2; irot++) {
    double ang = (double)(2 * irot) * pi / (double)3.0f;
    g.cth[irot - 1] = std::cos(ang);
    g.sth[irot - 1] = std::sin(ang);
  }
  g.arm_shift = (double)8.6602254037f;
}

static Lattice make_lattice(mskg_engine *e) {
  Lattice L;
  L.site = e->d_site;
  L.rate = e->d_rate;
  L.cls = e->d_cls;
  L.inlist = e->d_inlist;
  L.tl_idx = e->d_tl_idx;
  L.tl_n = e->d_tl_n;
  L.tl_own = e->d_tl_own;
  L.tile_r = e->d_tile_r;
  L.list_err = e->d_list_err;
  L.win = e->d_win;
  L.capg = e->capg;
  L.cur_tile = -1;
  L.cx = L.cy = L.cz = 0;
  L.cold = nullptr;
  L.box = e->box;
  L.geo = e->d_geo;
  L.tab = e->d_tab;
  L.tile = e->tile;
  L.inv_tile = 1.0f / (float)e->tile;
  L.ntx = e->ntx;
  L.nty = e->nty;
  L.key = e->track ? e->d_key : nullptr;
  L.cl = e->tab.la_variant ? (const long long *)((const char *)e->d_st + offsetof(RunState, cl)) : nullptr;
  L.ztop = e->windowed ? e->box.lz - TOP_MARGIN : 0x7fffffff;
  return L;
}

// The captured sweep holds the k_pass variant (InitSt 'ST' tables on or off)
// and what make_lattice gave at capture (CountLiquid, class keys) and the
// event log: a change to any of these needs a new capture at the next run.
static void drop_graph(mskg_engine *e) {
  if (e->graph_exec) { hipGraphExecDestroy(e->graph_exec); e->graph_exec = nullptr; }
  if (e->graph) { hipGraphDestroy(e->graph); e->graph = nullptr; }
}

// Same-colour tiles are one tile apart, so two concurrent events are at
// least tile+1 grid units apart along some axis.  An event writes records
// and rates at most 3 units from its site per axis (6 with the
// second-neighbour term, which refreshes the second neighbours) and reads at
// most 6 (12) units away, so a tile edge of 16 (24) keeps what one event
// writes out of what any other reads, with room for the rare neighbour
// entries that are not bond vectors.
static int choose_tile(int lx, int ly, int want, int min_tile) {
  auto ok = [&](int t) {
    return t >= min_tile && t <= 254 && t % 2 == 0 && lx % t == 0 && ly % t == 0 && (lx / t) % 2 == 0 &&
           (ly / t) % 2 == 0;
  };
  if (want) return ok(want) ? want : -1;
  const int pref[] = {24, 20, 18, 28, 30, 32, 36, 40, 42, 48, 16, 22, 26, 34, 38, 44, 46};
  for (int t : pref)
    if (ok(t)) return t;
  for (int t = min_tile; t <= std::min(lx, ly) / 2; t += 2)
    if (ok(t)) return t;
  return -1;
}

static const char *err_name(int c) {
  switch (c) {
    case ERR_COORD: return "coordination inconsistent with neighbour counts (Get_Prob.f:293-298)";
    case ERR_GEOM: return "neighbour displacement does not fit the site record";
    case ERR_NOT_MC: return "logged event on a site that is not an MC particle";
    case ERR_COVERAGE: return "coverage species not in ListCov";
    case ERR_CAPACITY: return "tile holds more MC particles than tile_capacity";
    case ERR_TEMPERATURE: return "zero temperature in laser-annealing mode";
    case ERR_TILE_LIST: return "a tile's candidate list overflowed tile_capacity";
    case ERR_SUMS: return "serial selection found no event inside a positive rate sum";
    case ERR_LIQUID: return "a species' CountLiquid is negative: its solidification rate would be negative";
    case ERR_ST_RANGE: return "a site's temperature lies outside the InitSt 'ST' reference temperatures";
    case ERR_SCHED: return "a tile waited too long (some minutes) for its neighbour tiles in a dependency-scheduled sweep";
    case ERR_TOP:
      return "an event site within 24 planes of the top of the stored planes (stored_len_z): store more planes";
    default: return "unknown";
  }
}

static int la_variant_off(mskg_engine *e);
static int census(mskg_engine *e, int64_t out[6]);
// The planes [z0, z1] outside which the state is the pristine slab: walls,
// bulk atoms on diamond sites, empty points of coordination 0.
static void touched_planes(const mskg_engine *e, int &z0, int &z1) {
  z0 = e->slab < 0 ? 0 : std::max(0, e->slab_z0);
  z1 = e->slab < 0 ? e->box.lz : std::min(e->box.lz, e->slab_z1);
}
// A run starts: until it has ended well, nothing is known of its state
// (returned: what was known).  run_over puts it back, wider.
static int run_touches(mskg_engine *e) {
  const int slab = e->slab;
  e->slab = -1;
  return slab;
}
static void run_over(mskg_engine *e, int slab, int lo, int hi) {
  e->slab = slab;
  if (slab < 0 || lo > hi) return;
  e->slab_z0 = std::min(e->slab_z0, lo * e->tile - 12);
  e->slab_z1 = std::max(e->slab_z1, (hi + 1) * e->tile - 1 + 12);
}
// A workspace of at least n bytes, null when there is no memory for it; a
// call that took one larger than work_keep gives it back at its end.  What is
// kept follows the lattice (a fifth of its records, rates and classes, which is
// what the words of a small one take on their way out; 8 MB at most): a scan over
// hundreds of small lattices keeps little beside them.
static size_t work_keep(const mskg_engine *e) {
  const int64_t lattice = e->box.npts * (int64_t)(sizeof(Site) + sizeof(float) + 1);
  return (size_t)std::min<int64_t>(8 << 20, std::max<int64_t>(lattice / 5, 1 << 16));
}
static void *work_take(mskg_engine *e, int k, size_t n) {
  if (e->work_n[k] < n) {
    hipFree(e->d_work[k]);
    e->d_work[k] = nullptr;
    e->work_n[k] = 0;
    n = std::max<size_t>(n, 1 << 16);
    if (hipMalloc(&e->d_work[k], n) != hipSuccess) {
      (void)hipGetLastError();
      e->d_work[k] = nullptr;
      return nullptr;
    }
    e->work_n[k] = n;
  }
  return e->d_work[k];
}
static void work_done(mskg_engine *e) {
  for (int k = 0; k < 2; k++)
    if (e->work_n[k] > work_keep(e)) {
      hipFree(e->d_work[k]);
      e->d_work[k] = nullptr;
      e->work_n[k] = 0;
    }
}
// The run state's fields before the sweep sums (slot: left as it is in st).
static int read_state(mskg_engine *e, RunState &st) {
  HIPCHK(e, hipMemcpyAsync(&st, e->d_st, RS_HEAD, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  return MSKG_OK;
}
// ... and back (the device's sweep sums kept).
static int write_state_head(mskg_engine *e, const RunState &st) {
  HIPCHK(e, hipMemcpyAsync(e->d_st, &st, RS_HEAD, hipMemcpyHostToDevice, e->stream));
  return MSKG_OK;
}

// The segments of a frame's kernels over the planes [z0, z1]: small enough
// that a small lattice still fills the chip, at most max_seg of them (0: any
// number, of FRAME_GROUPS groups at most).
static FramePlan frame_plan(const mskg_engine *e, int z0, int z1, int sic, int max_seg) {
  FramePlan F;
  F.first = z0 * e->box.plane;
  F.end = (z1 + 1) * e->box.plane;
  F.sic = sic;
  const int64_t ng = std::max<int64_t>(1, (F.end - F.first + WAVE - 1) / WAVE);
  F.groups = 4;
  while (F.groups < FRAME_GROUPS && ng / F.groups > 8192) F.groups *= 2;
  F.rounds = 1;
  if (max_seg) F.rounds = (int)((ng + (int64_t)F.groups * max_seg - 1) / ((int64_t)F.groups * max_seg));
  F.nseg = (int)((ng + (int64_t)F.groups * F.rounds - 1) / ((int64_t)F.groups * F.rounds));
  return F;
}

// Page-locked buffers of two halves for the host's data on its way, taken by a
// call and given back at its end (nothing of the call's is in flight then).
// The process keeps up to PINNED_IDLE that no call holds, for whichever engine
// and thread is next, until its last engine is destroyed: an allocation of one
// costs milliseconds, and a buffer an engine is memory that a scan over
// hundreds of engines does not get back.
constexpr int64_t PINNED_HALF = 4 << 20;  // bytes
constexpr int PINNED_IDLE = 2;
static std::mutex g_pinned_mu;  // guards the three below
static char *g_pinned_idle[PINNED_IDLE];
static int g_pinned_n = 0;
static int g_engines = 0;  // engines alive
struct Pinned {
  char *buf = nullptr;
  hipError_t take() {
    {
      std::lock_guard<std::mutex> lock(g_pinned_mu);
      if (g_pinned_n > 0) {
        buf = g_pinned_idle[--g_pinned_n];
        return hipSuccess;
      }
    }
    const hipError_t ce = hipHostMalloc((void **)&buf, 2 * PINNED_HALF, hipHostMallocPortable);
    if (ce != hipSuccess) buf = nullptr;
    return ce;
  }
  char *half(int64_t i) const { return buf + (i & 1) * PINNED_HALF; }
  ~Pinned() {
    if (!buf) return;
    {
      std::lock_guard<std::mutex> lock(g_pinned_mu);
      if (g_engines > 0 && g_pinned_n < PINNED_IDLE) {
        g_pinned_idle[g_pinned_n++] = buf;
        return;
      }
    }
    (void)hipHostFree(buf);
  }
};
static void engine_born() {
  std::lock_guard<std::mutex> lock(g_pinned_mu);
  g_engines++;
}
static void engine_gone() {
  char *idle[PINNED_IDLE];
  int n = 0;
  {
    std::lock_guard<std::mutex> lock(g_pinned_mu);
    if (--g_engines == 0)
      while (g_pinned_n > 0) idle[n++] = g_pinned_idle[--g_pinned_n];
  }
  while (n > 0) (void)hipHostFree(idle[--n]);
}

// Host pieces into device memory at dst + off (offsets increasing), through
// the two halves of a page-locked buffer: one copy for many small pieces, the
// next half filled while the last is on its way.
struct HostPiece {
  size_t off;
  const void *src;
  size_t n;
};
static hipError_t stage_in(mskg_engine *e, hipStream_t sm, char *dst, const std::vector<HostPiece> &pieces) {
  Pinned pin;
  hipError_t ce = pin.take();
  size_t begin = 0, fill = 0;  // the half holds [begin, begin + fill)
  int half = 0;
  bool used[2] = {false, false};
  auto flush = [&]() {
    if (!fill || ce != hipSuccess) return;
    ce = hipMemcpyAsync(dst + begin, pin.half(half), fill, hipMemcpyHostToDevice, sm);
    if (ce == hipSuccess) ce = hipEventRecord(half ? e->ev1 : e->ev0, sm);
    used[half] = true;
    half ^= 1;
    fill = 0;
  };
  for (const HostPiece &p : pieces)
    for (size_t done = 0; done < p.n && ce == hipSuccess;) {
      const size_t off = p.off + done;
      if (fill && off - begin >= (size_t)PINNED_HALF) flush();
      if (!fill) {
        begin = off;
        if (used[half] && ce == hipSuccess) ce = hipEventSynchronize(half ? e->ev1 : e->ev0);
      }
      if (ce != hipSuccess) break;
      const size_t m = std::min(p.n - done, (size_t)PINNED_HALF - (off - begin));
      memcpy(pin.half(half) + (off - begin), (const char *)p.src + done, m);
      fill = off - begin + m;
      done += m;
      if (fill == (size_t)PINNED_HALF) flush();
    }
  flush();
  // the buffer is the next caller's when this returns
  const hipError_t cs = hipStreamSynchronize(sm);
  return ce == hipSuccess ? cs : ce;
}

// The heads of n engines' run states in one exchange, once their own streams
// are idle (an exchange each had cost about 20 us an engine).
static int read_heads(mskg_engine *const *engines, int n, std::vector<RunHead> &out) {
  mskg_engine *e0 = engines[0];
  out.resize(n);
  std::vector<const void *> ptr(2 * (size_t)n);
  for (int i = 0; i < n; i++) {
    HIPCHK(engines[i], hipStreamSynchronize(engines[i]->stream));
    ptr[i] = engines[i]->d_st;
    ptr[n + i] = engines[i]->d_list_err;
  }
  char *w = (char *)work_take(e0, 0, (size_t)n * (2 * sizeof(void *) + sizeof(RunHead)));
  if (!w) return fail_(e0, MSKG_ENOMEM, "no device memory for the states of %d engines", n);
  const void **d_ptr = (const void **)w;
  RunHead *d_out = (RunHead *)(w + 2 * (size_t)n * sizeof(void *));
  HIPCHK(e0, hipMemcpyAsync(d_ptr, ptr.data(), ptr.size() * sizeof(void *), hipMemcpyHostToDevice, e0->stream));
  hipLaunchKernelGGL(k_heads, dim3((n + 63) / 64), dim3(64), 0, e0->stream, d_ptr, n, d_out);
  HIPCHK(e0, hipGetLastError());
  HIPCHK(e0, hipMemcpyAsync(out.data(), d_out, (size_t)n * sizeof(RunHead), hipMemcpyDeviceToHost, e0->stream));
  HIPCHK(e0, hipStreamSynchronize(e0->stream));
  return MSKG_OK;
}

// The ordered record lists of one frame mode (k_frame_count / k_frame_write):
// hosts[k] receives list k (caps[k] records), counts the NCNT totals.  A call
// with too small capacities only sizes the lists (MSKG_ECAPACITY when it
// brought buffers).
template <int MODE>
static int frame_lists(mskg_engine *e, int sic, int32_t *const hosts[], const int64_t caps[], int64_t counts[]) {
  constexpr int NL_ = FrameShape<MODE>::NLIST, NC = FrameShape<MODE>::NCNT;
  // outside the touched planes a slab has no record: its atoms there have
  // coordination 4 and lie on diamond sites, its empty points coordination 0,
  // and in the SiC slab every atom's neighbours are of the other species (an
  // alloy's or a one-species slab's are not: every plane is read)
  int z0 = 0, z1 = e->box.lz;
  if (MODE == FRAME_MAIN || !sic || e->slab == 1) touched_planes(e, z0, z1);
  const FramePlan F = frame_plan(e, z0, z1, sic, 0);
  const int nblk = (F.nseg + FRAME_THREADS / WAVE - 1) / (FRAME_THREADS / WAVE);
  Lattice L = make_lattice(e);
  const size_t n_bits = (size_t)F.nseg * F.groups * 8, n_offs = (size_t)F.nseg * NL_ * 8, n_cnt = (size_t)F.nseg * NC * 4;
  // totals, offsets, counts, then the bits (left out when there is no memory for them)
  unsigned long long *bits = nullptr;
  char *w = (char *)work_take(e, 0, 64 + n_offs + n_cnt + 8 + n_bits);
  if (w) bits = (unsigned long long *)(w + 64 + n_offs + (n_cnt + 7) / 8 * 8);
  else w = (char *)work_take(e, 0, 64 + n_offs + n_cnt);
  if (!w) return fail_(e, MSKG_ENOMEM, "frame: no device memory for the block counts");
  int64_t *d_tot = (int64_t *)w;
  unsigned long long *d_offs = (unsigned long long *)(w + 64);
  uint32_t *d_counts = (uint32_t *)(w + 64 + n_offs);
  hipLaunchKernelGGL(k_frame_count<MODE>, dim3(nblk), dim3(FRAME_THREADS), 0, e->stream, L, F, d_counts, bits);
  hipLaunchKernelGGL(k_frame_scan<MODE>, dim3(NC), dim3(SCAN_THREADS), 0, e->stream, d_counts, F.nseg, d_offs, d_tot);
  int64_t tot[NC];
  hipError_t ce = hipGetLastError();
  if (ce == hipSuccess) ce = hipMemcpyAsync(tot, d_tot, sizeof tot, hipMemcpyDeviceToHost, e->stream);
  if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
  if (ce != hipSuccess) {
    work_done(e);
    return fail_(e, MSKG_EDEVICE, "frame count: %s", hipGetErrorString(ce));
  }
  bool fits = true, brought = false;
  int64_t all = 0;
  for (int k = 0; k < NC; k++) counts[k] = tot[k];
  for (int k = 0; k < NL_; k++) {
    fits &= tot[k] <= caps[k];
    brought |= hosts[k] && caps[k];
    all += tot[k];
  }
  if (!fits) {
    work_done(e);
    if (brought) return fail_(e, MSKG_ECAPACITY, "frame: the records do not fit the buffers given");
    return MSKG_OK;  // sizing call
  }
  if (all) {
    int4 *d_rec = (int4 *)work_take(e, 1, (size_t)all * sizeof(int4));
    if (!d_rec) {
      work_done(e);
      return fail_(e, MSKG_ENOMEM, "frame: no device memory for the records");
    }
    int4 *d_out[3] = {d_rec, d_rec + tot[0], d_rec + tot[0] + tot[1]};
    hipLaunchKernelGGL(k_frame_write<MODE>, dim3(nblk), dim3(FRAME_THREADS), 0, e->stream, L, F, bits, d_offs,
                       d_out[0], d_out[1], d_out[2], tot[0], tot[1], NL_ > 2 ? tot[2] : (int64_t)0);
    ce = hipGetLastError();
    for (int k = 0; k < NL_ && ce == hipSuccess; k++)
      if (tot[k] && hosts[k])
        ce = hipMemcpyAsync(hosts[k], d_out[k], tot[k] * sizeof(int4), hipMemcpyDeviceToHost, e->stream);
    if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
  }
  work_done(e);
  if (ce != hipSuccess) return fail_(e, MSKG_EDEVICE, "frame write: %s", hipGetErrorString(ce));
  return MSKG_OK;
}

static CovList cov_list(const mskg_engine *e) {
  CovList C;
  C.n = e->ncov;
  for (int k = 0; k < 3; k++) C.index[k] = e->list_cov[k];
  return C;
}
// One record a site: the neighbour list its last record gives, the class and
// rate of its last MC record.
static void merge_listed(std::vector<StateRec> &recs) {
  std::unordered_map<int64_t, size_t> at;
  std::vector<StateRec> one;
  for (const StateRec &r : recs) {
    const auto it = at.find(r.p);
    if (it == at.end()) {
      at.emplace(r.p, one.size());
      one.push_back(r);
      continue;
    }
    StateRec &o = one[it->second];
    const float rate = o.rate;
    const int cls = o.cls;
    o = r;
    if (r.cls < 0) {
      o.cls = cls;
      o.rate = rate;
    }
  }
  recs.swap(one);
}
// A piece of a state's exchange: the points of whole planes, about this many.
constexpr int64_t STATE_PIECE = 1ll << 24;

// The three particle lists in grid order: tot their lengths, the first cap[k]
// records of each to the arrays that are given.
static int state_lists(mskg_engine *e, const int64_t cap[3], int32_t *const xyz[3], int32_t *const nn[3],
                       int32_t *event, double *prob, int64_t tot[3]) {
  Lattice L = make_lattice(e);
  const int step = (int)std::max<int64_t>(1, STATE_PIECE / e->box.plane);
  for (int z = 0; z <= e->box.lz; z += step) {
    const FramePlan F = frame_plan(e, z, std::min(z + step - 1, e->box.lz), 0, 0);
    const int nblk = (F.nseg + FRAME_THREADS / WAVE - 1) / (FRAME_THREADS / WAVE);
    const size_t n_offs = (size_t)F.nseg * 3 * 8, n_cnt = ((size_t)F.nseg * 3 * 4 + 7) / 8 * 8;
    char *w = (char *)work_take(e, 0, 64 + n_offs + n_cnt + (size_t)F.nseg * F.groups * 8);
    if (!w) return fail_(e, MSKG_ENOMEM, "store: no device memory for the list counts");
    int64_t *d_tot = (int64_t *)w, n[3];
    unsigned long long *d_offs = (unsigned long long *)(w + 64), *bits = (unsigned long long *)(w + 64 + n_offs + n_cnt);
    uint32_t *d_counts = (uint32_t *)(w + 64 + n_offs);
    hipLaunchKernelGGL(k_frame_count<FRAME_STATE>, dim3(nblk), dim3(FRAME_THREADS), 0, e->stream, L, F, d_counts, bits);
    hipLaunchKernelGGL(k_frame_scan<FRAME_STATE>, dim3(3), dim3(SCAN_THREADS), 0, e->stream, d_counts, F.nseg, d_offs,
                       d_tot);
    HIPCHK(e, hipGetLastError());
    HIPCHK(e, hipMemcpyAsync(n, d_tot, sizeof n, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    int64_t take[3], all = n[0] + n[1] + n[2];
    bool any = false;
    for (int k = 0; k < 3; k++) {
      take[k] = std::max<int64_t>(0, std::min(n[k], cap[k] - tot[k]));
      any |= take[k] > 0 && (xyz[k] || nn[k] || (k == 0 && (event || prob)));
    }
    if (any) {
      char *r = (char *)work_take(e, 1, (size_t)all * 60 + (size_t)n[0] * 12);
      if (!r) return fail_(e, MSKG_ENOMEM, "store: no device memory for the lists");
      StateOut O;
      O.prob = (double *)r;
      int32_t *q = (int32_t *)(O.prob + n[0]);
      for (int k = 0; k < 3; k++) {
        O.xyz[k] = q;
        O.nn[k] = q + 3 * n[k];
        q += 15 * n[k];
      }
      O.event = q;
      hipLaunchKernelGGL(k_state_write, dim3(nblk), dim3(FRAME_THREADS), 0, e->stream, L, F, bits, d_offs, O);
      HIPCHK(e, hipGetLastError());
      auto out = [&](void *host, const void *dev, int64_t bytes) {
        return host && bytes ? hipMemcpyAsync(host, dev, (size_t)bytes, hipMemcpyDeviceToHost, e->stream) : hipSuccess;
      };
      for (int k = 0; k < 3; k++) {
        HIPCHK(e, out(xyz[k] ? xyz[k] + 3 * tot[k] : nullptr, O.xyz[k], take[k] * 12));
        HIPCHK(e, out(nn[k] ? nn[k] + 12 * tot[k] : nullptr, O.nn[k], take[k] * 48));
      }
      HIPCHK(e, out(event ? event + tot[0] : nullptr, O.event, take[0] * 4));
      HIPCHK(e, out(prob ? prob + tot[0] : nullptr, O.prob, take[0] * 8));
      HIPCHK(e, hipStreamSynchronize(e->stream));
    }
    for (int k = 0; k < 3; k++) tot[k] += n[k];
  }
  return MSKG_OK;
}

// LattCoo's words at the lattice points (the others are left as the caller
// has them).  The words come through two halves of a page-locked buffer, the
// next on its way while the last is laid out; a word that is there already is
// not written again (most of a box is vacuum, and so is a fresh array).
static int state_words(mskg_engine *e, int32_t *latt) {
  const Box &b = e->box;
  constexpr int64_t HALF = PINNED_HALF / 4;  // words
  Pinned pin;
  HIPCHK(e, pin.take());
  int32_t *d = (int32_t *)work_take(e, 1, b.npts <= HALF ? b.npts * 4 : 2 * HALF * 4);  // one piece, or two in turn
  if (!d) return fail_(e, MSKG_ENOMEM, "store: no device memory for LattCoo's words");
  Lattice L = make_lattice(e);
  const CovList C = cov_list(e);
  const int64_t pieces = (b.npts + HALF - 1) / HALF;
  auto fetch = [&](int64_t i) -> hipError_t {
    const int64_t p0 = i * HALF, p1 = std::min(p0 + HALF, b.npts);
    int32_t *const dst = d + (i & 1) * HALF;
    hipLaunchKernelGGL(k_words_out, dim3((unsigned)((p1 - p0 + 255) / 256)), dim3(256), 0, e->stream, L, C, p0, p1, dst);
    hipError_t ce = hipGetLastError();
    if (ce == hipSuccess)
      ce = hipMemcpyAsync(pin.half(i), dst, (size_t)(p1 - p0) * 4, hipMemcpyDeviceToHost, e->stream);
    if (ce == hipSuccess) ce = hipEventRecord(i & 1 ? e->ev1 : e->ev0, e->stream);
    return ce;
  };
  hipError_t ce = fetch(0);
  for (int64_t i = 0; i < pieces && ce == hipSuccess; i++) {
    if (i + 1 < pieces) ce = fetch(i + 1);
    if (ce == hipSuccess) ce = hipEventSynchronize(i & 1 ? e->ev1 : e->ev0);
    if (ce != hipSuccess) break;
    const int32_t *src = (const int32_t *)pin.half(i);
    const int64_t p1 = std::min((i + 1) * HALF, b.npts);
    for (int64_t p = i * HALF; p < p1;) {  // row by row
      const int64_t row = p / b.hx, end = std::min(p1, (row + 1) * b.hx);
      const int y2 = (int)(row % b.hy), z = (int)(row / b.hy), par = z & 1;
      int32_t *g = latt + (int64_t)b.lx * ((int64_t)(2 * y2 + par) + (int64_t)b.ly * z) + par + 2 * (p - row * b.hx);
      for (; p < end; p++, g += 2) {
        const int32_t v = *src++;
        if (*g != v) *g = v;
      }
    }
  }
  const hipError_t cs = hipStreamSynchronize(e->stream);
  if (ce == hipSuccess) ce = cs;
  if (ce != hipSuccess) return fail_(e, MSKG_EDEVICE, "store: %s", hipGetErrorString(ce));
  return MSKG_OK;
}

// The flips of the SiC wrong-site analysis in the reference's grid order
// (see k_wrong_cand): the positions of the atoms that flip.
static int wrong_flips(mskg_engine *e, std::vector<int4> &flips) {
  flips.clear();
  Lattice L = make_lattice(e);
  int z0 = 0, z1 = e->box.lz;
  if (e->slab == 1) touched_planes(e, z0, z1);  // every atom of the SiC slab has neighbours of the other species
  const int64_t first = z0 * e->box.plane, end = (z1 + 1) * e->box.plane;
  const int blocks = (int)std::min<int64_t>((end - first + 255) / 256, 256 * 64);
  int64_t cap = 1 << 16;
  for (;;) {
    unsigned long long *d_n = nullptr;
    int4 *d_c = nullptr;
    if (hipMalloc(&d_n, sizeof(unsigned long long)) != hipSuccess ||
        hipMalloc(&d_c, (size_t)cap * 5 * sizeof(int4)) != hipSuccess) {
      hipFree(d_n);
      return fail_(e, MSKG_ENOMEM, "frame: no device memory for the wrong-site candidates");
    }
    unsigned long long n = 0;
    std::vector<int4> c;
    hipError_t ce = hipMemsetAsync(d_n, 0, sizeof n, e->stream);
    if (ce == hipSuccess) {
      hipLaunchKernelGGL(k_wrong_cand, dim3(blocks), dim3(256), 0, e->stream, L, first, end, cap, d_n,
                         d_c);
      ce = hipGetLastError();
    }
    if (ce == hipSuccess) ce = hipMemcpyAsync(&n, d_n, sizeof n, hipMemcpyDeviceToHost, e->stream);
    if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
    if (ce == hipSuccess && (int64_t)n <= cap) {
      c.resize((size_t)n * 5);
      if (n) ce = hipMemcpy(c.data(), d_c, c.size() * sizeof(int4), hipMemcpyDeviceToHost);
    }
    hipFree(d_n);
    hipFree(d_c);
    if (ce != hipSuccess) return fail_(e, MSKG_EDEVICE, "frame wrong-site candidates: %s", hipGetErrorString(ce));
    if ((int64_t)n > cap) {
      cap = (int64_t)n;
      continue;
    }
    // grid order (z, then y, then x); a candidate flips unless a candidate
    // neighbour before it did
    const Box &b = e->box;
    auto key = [&](const int4 &q) { return ((int64_t)q.z * b.ly + q.y) * b.lx + q.x; };
    std::vector<size_t> order(n);
    for (size_t i = 0; i < n; i++) order[i] = i;
    std::sort(order.begin(), order.end(), [&](size_t a, size_t bb) { return key(c[5 * a]) < key(c[5 * bb]); });
    std::vector<int64_t> flipped_keys;
    for (size_t oi = 0; oi < n; oi++) {
      const size_t i = order[oi];
      bool flip = true;
      for (int k = 0; k < 4 && flip; k++) {
        const int64_t q = key(c[5 * i + 1 + k]);
        flip = !std::binary_search(flipped_keys.begin(), flipped_keys.end(), q);
      }
      if (flip) {
        flipped_keys.push_back(key(c[5 * i]));  // keys arrive in increasing order
        flips.push_back(c[5 * i]);
      }
    }
    return MSKG_OK;
  }
}

static int set_wrong_marks(mskg_engine *e, const std::vector<int4> &flips, int set) {
  if (flips.empty()) return MSKG_OK;
  int4 *d = nullptr;
  HIPCHK(e, hipMalloc(&d, flips.size() * sizeof(int4)));
  hipError_t ce = hipMemcpyAsync(d, flips.data(), flips.size() * sizeof(int4), hipMemcpyHostToDevice, e->stream);
  if (ce == hipSuccess) {
    const int blocks = (int)std::min<size_t>((flips.size() + 255) / 256, 4096);
    hipLaunchKernelGGL(k_wrong_set, dim3(blocks), dim3(256), 0, e->stream, make_lattice(e), d,
                       (int64_t)flips.size(), set);
    ce = hipGetLastError();
  }
  if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
  hipFree(d);
  if (ce != hipSuccess) return fail_(e, MSKG_EDEVICE, "frame wrong-site marks: %s", hipGetErrorString(ce));
  return MSKG_OK;
}

// The device address of `scratch` on each device, taken once per device
// with that device current (mskg_create).
constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static unsigned long long *g_scratch[MAX_DEVICES] = {};

static int noalloc_scratch_init(mskg_engine *e) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (e->device < 0 || e->device >= MAX_DEVICES)
    return fail_(e, MSKG_EDEVICE, "device %d beyond the %d the library tracks", e->device, MAX_DEVICES);
  if (g_scratch[e->device]) return MSKG_OK;
  void *ptr = nullptr;
  const hipError_t rc = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (rc != hipSuccess || !ptr)
    return fail_(e, MSKG_EDEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(rc));
  g_scratch[e->device] = (unsigned long long *)ptr;
  return MSKG_OK;
}

extern "C" {

const char *mskg_last_error(const mskg_engine *e) { return e ? e->err.c_str() : "null engine"; }

int mskg_create(const mskg_config *cfg, mskg_engine **out) {
  if (!cfg || !out) return MSKG_EINVAL;
  *out = nullptr;
  mskg_engine *e = new (std::nothrow) mskg_engine();
  if (!e) return MSKG_ENOMEM;
  engine_born();
  *out = e;
  e->cfg = *cfg;
  if (cfg->len_x <= 0 || cfg->len_y <= 0 || cfg->len_z <= 0 || cfg->len_x % 12 || cfg->len_y % 12)
    return fail_(e, MSKG_EINVAL, "box %d x %d x %d: len_x and len_y must be positive multiples of 12", cfg->len_x,
                 cfg->len_y, cfg->len_z);
  if (cfg->len_z > 8190) return fail_(e, MSKG_EINVAL, "len_z must be <= 8190");
  if (cfg->stored_len_z < 0 || cfg->stored_len_z > cfg->len_z + 1 ||
      (cfg->stored_len_z > 0 && cfg->stored_len_z < 2 * TOP_MARGIN))
    return fail_(e, MSKG_EINVAL, "stored_len_z %d: 0 (all planes) or %d..%d", cfg->stored_len_z, 2 * TOP_MARGIN,
                 cfg->len_z + 1);
  if (cfg->n_crystal < 1 || cfg->n_crystal > 3 || cfg->n_cov < 0 || cfg->n_cov > 3)
    return fail_(e, MSKG_EINVAL, "n_crystal must be 1..3 and n_cov 0..3");
  if (!cfg->ptrans_e || !cfg->ptrans_d) return fail_(e, MSKG_EINVAL, "ptrans_e and ptrans_d are required");
  if (cfg->n_cov > 0 && (!cfg->ptrans_abs || !cfg->ptrans_des))
    return fail_(e, MSKG_EINVAL, "ptrans_abs and ptrans_des are required when n_cov > 0");
  e->logical_lz = cfg->len_z;
  e->windowed = cfg->stored_len_z > 0 && cfg->stored_len_z < cfg->len_z + 1;
  e->box = make_box(cfg->len_x, cfg->len_y, e->windowed ? cfg->stored_len_z - 1 : cfg->len_z);
  e->ncrystal = cfg->n_crystal;
  e->ncov = cfg->n_cov;
  for (int i = 0; i < 3; i++) e->list_cov[i] = cfg->list_cov[i];
  memset(&e->tab, 0, sizeof e->tab);
  memcpy(e->tab.pe, cfg->ptrans_e, sizeof e->tab.pe);
  memcpy(e->tab.pd, cfg->ptrans_d, sizeof e->tab.pd);
  if (cfg->ptrans_abs) memcpy(e->tab.pabs, cfg->ptrans_abs, sizeof e->tab.pabs);
  if (cfg->ptrans_des) memcpy(e->tab.pdes, cfg->ptrans_des, sizeof e->tab.pdes);
  e->tab.ptrans_zig = cfg->ptrans_zig;
  e->tab.ncrystal = cfg->n_crystal;
  e->tab.ncov = cfg->n_cov;
  e->tab.la_mode = cfg->la_mode;
  e->cov_model = cfg->n_cov > 0;  // coverage species, or absorption / desorption rates in the tables
  for (int i = 0; i < 12; i++) e->cov_model |= e->tab.pabs[i] != 0.0 || e->tab.pdes[i] != 0.0;
  e->tab.p0 = cfg->p0;
  e->tab.tm = cfg->tm;
  e->tab.sigma = cfg->sigma;
  e->tab.tflex = cfg->tflex;
  e->tab.frozen_below_z = cfg->frozen_below_z;
  e->tab.use_f2 = cfg->second_factor != nullptr;
  if (cfg->second_factor)
    for (int i = 0; i < 13; i++) {
      e->tab.f2[i] = cfg->second_factor[i];
      if (!(e->tab.f2[i] > 0.0) || !std::isfinite(e->tab.f2[i]))
        return fail_(e, MSKG_EINVAL, "second_factor[%d] must be positive and finite", i);
    }
  build_geometry(e->geo);
  const int min_tile = e->tab.use_f2 ? 24 : 16;
  e->tile = choose_tile(cfg->len_x, cfg->len_y, cfg->tile, min_tile);
  if (e->tile < 0)
    return fail_(e, MSKG_EINVAL,
                 "no valid tile edge for box %d x %d (requested %d): need an even tile >= %d with an even "
                 "number of tiles along x and y",
                 cfg->len_x, cfg->len_y, cfg->tile, min_tile);
  // the pass kernel holds a tile's list in LDS at 9 B per entry: at most
  // 6144 entries (55 KB) keep one wave's LDS under 64 KB
  if (cfg->tile_capacity < 0 || cfg->tile_capacity > 6144)
    return fail_(e, MSKG_EINVAL, "tile_capacity %d: 0 (1024) or 1..6144", cfg->tile_capacity);
  e->cap = cfg->tile_capacity > 0 ? cfg->tile_capacity : 1024;
  e->capg = e->cap;
  e->ntx = cfg->len_x / e->tile;
  e->nty = cfg->len_y / e->tile;
  e->ntz = (e->box.lz + 1 + e->tile - 1) / e->tile;
  e->ntiles = e->ntx * e->nty * e->ntz;
  // the tile sums are taken in chunks of the full box's tiles, so that a
  // box storing only its bottom planes sums the same values in the same
  // order (the tiles it does not store hold no rates)
  e->rsum_chunk = (e->ntx * e->nty * ((cfg->len_z + 1 + e->tile - 1) / e->tile) + NPART - 1) / NPART;

  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail_(e, MSKG_EDEVICE, "no HIP device available");
  HIPCHK(e, hipGetDevice(&e->device));
  if (int rc = noalloc_scratch_init(e)) return rc;
  HIPCHK(e, hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
  HIPCHK(e, hipEventCreate(&e->ev0));
  HIPCHK(e, hipEventCreate(&e->ev1));
  const int64_t n = e->box.npts;
  HIPCHK(e, hipMalloc(&e->d_site, n * sizeof(Site)));
  HIPCHK(e, hipMalloc(&e->d_rate, n * sizeof(float)));
  HIPCHK(e, hipMalloc(&e->d_cls, n * sizeof(uint8_t)));
  HIPCHK(e, hipMalloc(&e->d_inlist, n));
  HIPCHK(e, hipMalloc(&e->d_tl_idx, (size_t)e->ntiles * e->capg * sizeof(int32_t)));
  HIPCHK(e, hipMalloc(&e->d_tl_n, e->ntiles * sizeof(int32_t)));
  HIPCHK(e, hipMalloc(&e->d_tl_own, e->ntiles * sizeof(int32_t)));
  HIPCHK(e, hipMalloc(&e->d_tile_r, e->ntiles * sizeof(double)));
  HIPCHK(e, hipMalloc(&e->d_list_err, sizeof(int)));
  HIPCHK(e, hipMalloc(&e->d_win, 32 * sizeof(int)));
  HIPCHK(e, hipMalloc(&e->d_done, ((size_t)e->ntiles + 8) * sizeof(unsigned int)));
  HIPCHK(e, hipMalloc(&e->d_geo, sizeof(Geometry)));
  HIPCHK(e, hipMalloc(&e->d_tab, sizeof(Tables)));
  HIPCHK(e, hipMalloc(&e->d_st, sizeof(RunState)));
  HIPCHK(e, hipMalloc(&e->d_err, sizeof(int)));
  HIPCHK(e, hipMemcpyAsync(e->d_geo, &e->geo, sizeof(Geometry), hipMemcpyHostToDevice, e->stream));
  HIPCHK(e, hipMemcpyAsync(e->d_tab, &e->tab, sizeof(Tables), hipMemcpyHostToDevice, e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_site, 0, n * sizeof(Site), e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_rate, 0, n * sizeof(float), e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_cls, 0, n, e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_inlist, 0, n, e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_tl_n, 0, e->ntiles * sizeof(int32_t), e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_tl_own, 0, e->ntiles * sizeof(int32_t), e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_tile_r, 0, e->ntiles * sizeof(double), e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_list_err, 0, sizeof(int), e->stream));
  {  // empty windows: lists built before any run widen them
    int w0[32];
    for (int c = 0; c < 8; c++) {
      w0[4 * c] = w0[4 * c + 2] = 0x7fffffff;
      w0[4 * c + 1] = w0[4 * c + 3] = -1;
    }
    HIPCHK(e, hipMemcpyAsync(e->d_win, w0, sizeof w0, hipMemcpyHostToDevice, e->stream));
  }
  // completion stamps: 0 is no sweep's (the first k_sweep_end makes it 1)
  HIPCHK(e, hipMemsetAsync(e->d_done, 0, ((size_t)e->ntiles + 8) * sizeof(unsigned int), e->stream));
  RunState st;
  memset(&st, 0, sizeof st);
  HIPCHK(e, hipMemcpyAsync(e->d_st, &st, sizeof st, hipMemcpyHostToDevice, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  return MSKG_OK;
}

void mskg_destroy(mskg_engine *e) {
  if (!e) return;
  if (e->stream) hipStreamSynchronize(e->stream);
  hipFree(e->d_site); hipFree(e->d_rate); hipFree(e->d_cls);
  if (e->graph_exec) hipGraphExecDestroy(e->graph_exec);
  if (e->graph) hipGraphDestroy(e->graph);
  hipFree(e->d_inlist); hipFree(e->d_tl_idx); hipFree(e->d_tl_n); hipFree(e->d_tl_own); hipFree(e->d_tile_r); hipFree(e->d_list_err);
  hipFree(e->d_field[0]); hipFree(e->d_field[1]); hipFree(e->d_offwall); hipFree(e->d_st_tables); hipFree(e->d_win);
  hipFree(e->d_done);
  for (int k = 0; k < 2; k++) hipFree(e->d_work[k]);
  hipFree(e->d_geo); hipFree(e->d_tab); hipFree(e->d_st); hipFree(e->d_err); hipFree(e->d_log);
  hipFree(e->d_tsum); hipFree(e->d_bsum); hipFree(e->d_key); hipFree(e->d_key_seen); hipFree(e->d_rate_seen);
  if (e->ev0) hipEventDestroy(e->ev0);
  if (e->ev1) hipEventDestroy(e->ev1);
  if (e->stream) hipStreamDestroy(e->stream);
  delete e;
  engine_gone();
}

int mskg_load_state(mskg_engine *e, const int32_t *latt, int32_t n_ad, const int32_t *ad_xyz, const int32_t *ad_nn,
                    const int32_t *ad_event, const double *ad_prob, int32_t n_bulk, const int32_t *bulk_xyz,
                    const int32_t *bulk_nn, int32_t n_void, const int32_t *void_xyz, const int32_t *void_nn,
                    double kmc_time) {
  if (!e || !latt) return MSKG_EINVAL;
  if (!e->d_site) return fail_(e, MSKG_EINVAL, "engine not created");
  const Box &b = e->box;
  const CovList C = cov_list(e);
  const int64_t face = (int64_t)b.lx * b.ly, grid = face * (b.lz + 1);
  // LattCoo goes to the device whole when that takes at most WORDS_WHOLE
  // bytes, else in pieces of planes, once to be checked and once to be taken
  // (an even number of planes: whole words of wall bits)
  constexpr int64_t WORDS_WHOLE = 2ll << 30;
  int64_t planes = b.lz + 1;
  if (grid * 4 > WORDS_WHOLE) planes = std::max<int64_t>(2, (WORDS_WHOLE / 8) / (face * 4) / 2 * 2);
  char *w = nullptr;
  for (;; planes = std::max<int64_t>(2, planes / 4 * 2)) {  // smaller pieces when memory is short
    planes = std::min<int64_t>(planes, b.lz + 1);
    if ((w = (char *)work_take(e, 1, 16 + (size_t)(planes * face) * 4))) break;
    if (planes <= 2) return fail_(e, MSKG_ENOMEM, "load: no device memory for a piece of LattCoo");
  }
  struct Done {  // the workspaces go back however the call ends
    mskg_engine *e;
    ~Done() { work_done(e); }
  } at_end{e};
  (void)at_end;
  unsigned long long *d_out = (unsigned long long *)w;
  int32_t *d_words = (int32_t *)(w + 16);
  const bool whole = planes == b.lz + 1;
  unsigned long long found[2] = {~0ull, 0ull};
  HIPCHK(e, hipMemcpyAsync(d_out, found, sizeof found, hipMemcpyHostToDevice, e->stream));
  auto blocks_of = [](int64_t n) { return dim3((unsigned)std::min<int64_t>((n + 255) / 256, 256 * 64)); };
  for (int64_t z = 0; z <= b.lz; z += planes) {
    const int64_t g0 = z * face, n = std::min(planes, b.lz + 1 - z) * face;
    HIPCHK(e, hipMemcpyAsync(d_words, latt + g0, (size_t)n * 4, hipMemcpyHostToDevice, e->stream));
    hipLaunchKernelGGL(k_words_check, blocks_of(n), dim3(256), 0, e->stream, b, C, d_words, g0, n, d_out);
    HIPCHK(e, hipGetLastError());
  }
  HIPCHK(e, hipMemcpyAsync(found, d_out, sizeof found, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  if (found[0] != ~0ull) {
    const int64_t g = (int64_t)found[0];
    return fail_(e, MSKG_ESTATE, "LattCoo(%d,%d,%d)=0x%08x is not a representable site state", (int)(g % b.lx),
                 (int)(g / b.lx % b.ly), (int)(g / face), latt[g]);
  }
  // planes above the stored ones: vacuum or walls only, which no event reaches
  for (int z = b.lz + 1; z <= e->logical_lz; z++)
    for (int y = 0; y < b.ly; y++)
      for (int x = 0; x < b.lx; x++) {
        const int32_t v = latt[(int64_t)x + (int64_t)b.lx * ((int64_t)y + (int64_t)b.ly * z)];
        if (v != 0 && (v & 255) != 113)
          return fail_(e, MSKG_ESTATE, "LattCoo(%d,%d,%d)=0x%08x lies above the %d stored planes", x, y, z, v,
                       b.lz + 1);
      }
  // the lists: checked, and every record as the device takes it
  std::vector<StateRec> recs;
  recs.reserve((size_t)std::max(n_ad, 0) + std::max(n_bulk, 0) + std::max(n_void, 0));
  std::vector<bool> listed((size_t)b.npts, false);
  bool again = false;  // a site is listed more than once
  double rsum = 0.0;
  auto put = [&](int which, int32_t n, const int32_t *xyz, const int32_t *nn) -> int {
    for (int32_t i = 0; i < n; i++) {
      const int32_t *s = xyz + 3 * i;
      int64_t p = pidx_checked(b, s[0], s[1], s[2]);
      if (p < 0)
        return fail_(e, MSKG_ESTATE, "list %d record %d: site (%d,%d,%d) is not a lattice point of the box", which, i,
                     s[0], s[1], s[2]);
      if (which == 0 && e->windowed && s[2] > b.lz - TOP_MARGIN)
        return fail_(e, MSKG_ESTATE, "MC record %d at (%d,%d,%d) lies within %d planes of the stored top (%d)", i,
                     s[0], s[1], s[2], TOP_MARGIN, b.lz);
      NL l;
      for (int k = 0; k < 4; k++) {
        l.x[k] = nn[12 * i + 3 * k];
        l.y[k] = nn[12 * i + 3 * k + 1];
        l.z[k] = nn[12 * i + 3 * k + 2];
      }
      union {
        Site site;
        uint32_t word[4];
      } u;
      memset(&u, 0, sizeof u);
      if (!set_list(b, u.site, s[0], s[1], s[2], l))
        return fail_(e, MSKG_ESTATE, "list %d record %d at (%d,%d,%d): a NextNXYZ entry is too far away", which, i,
                     s[0], s[1], s[2]);
      StateRec r;
      r.p = p;
      r.x = u.word[0];
      r.y = u.word[1];
      r.z = u.word[2];
      r.valid = u.site.valid;
      r.rate = 0.0f;
      r.cls = -1;
      if (which == 0) {
        const int32_t v = latt[(int64_t)s[0] + (int64_t)b.lx * ((int64_t)s[1] + (int64_t)b.ly * s[2])];
        int ev = ad_event ? ad_event[i] : 1;
        double pr = ad_prob ? ad_prob[i] : 0.0;
        int kind = word_kind(C, v), coor = (v >> 24) & 7;
        int c;
        if (ev == 4) c = (kind_species(kind) && coor == 0) ? CLS_ISOLATED : CLS_EVAP;
        else if (ev == 5) c = CLS_DESORB;
        else if (kind == KIND_EMPTY && coor == 1 && (pr == (double)1.e-8f || pr == (double)1.e-6f)) c = CLS_PLACEHOLDER;
        else c = CLS_ADSORB;
        if (!(pr > 0.0)) return fail_(e, MSKG_ESTATE, "MC record %d has a non-positive rate", i);
        r.cls = c;
        r.rate = (float)pr;
        rsum += pr;
      }
      again |= listed[(size_t)p];
      listed[(size_t)p] = true;
      recs.push_back(r);
    }
    return 0;
  };
  int rc;
  if ((rc = put(0, n_ad, ad_xyz, ad_nn))) return rc;
  if ((rc = put(1, n_bulk, bulk_xyz, bulk_nn))) return rc;
  if ((rc = put(2, n_void, void_xyz, void_nn))) return rc;
  if (again) merge_listed(recs);
  StateRec *d_recs = nullptr;
  if (!recs.empty()) {
    d_recs = (StateRec *)work_take(e, 0, recs.size() * sizeof(StateRec));
    if (!d_recs) return fail_(e, MSKG_ENOMEM, "load: no device memory for the lists");
  }
  // from here on the state changes
  e->slab = -1;
  hipFree(e->d_offwall);
  e->d_offwall = nullptr;
  e->offwall_planes = false;
  if (found[1]) HIPCHK(e, hipMalloc(&e->d_offwall, (size_t)((grid + 31) / 32) * sizeof(uint32_t)));
  Lattice L = make_lattice(e);
  for (int64_t z = 0; z <= b.lz; z += planes) {
    const int64_t nz = std::min(planes, b.lz + 1 - z), g0 = z * face, n = nz * face;
    if (!whole) HIPCHK(e, hipMemcpyAsync(d_words, latt + g0, (size_t)n * 4, hipMemcpyHostToDevice, e->stream));
    hipLaunchKernelGGL(k_words_in, blocks_of(nz * b.plane), dim3(256), 0, e->stream, L, C, d_words, g0, z * b.plane,
                       (z + nz) * b.plane);
    if (found[1])
      hipLaunchKernelGGL(k_words_offwall, blocks_of(n), dim3(256), 0, e->stream, b, d_words, g0, n, e->d_offwall);
    HIPCHK(e, hipGetLastError());
  }
  if (d_recs) {
    HIPCHK(e, hipMemcpyAsync(d_recs, recs.data(), recs.size() * sizeof(StateRec), hipMemcpyHostToDevice, e->stream));
    hipLaunchKernelGGL(k_lists_in, dim3((unsigned)((recs.size() + 255) / 256)), dim3(256), 0, e->stream, L, d_recs,
                       (int64_t)recs.size());
    HIPCHK(e, hipGetLastError());
  }
  RunState st;
  memset(&st, 0, sizeof st);
  st.clock = kmc_time;
  st.rtot = rsum;
  st.events_per_pass = e->cfg.events_per_pass > 0 ? e->cfg.events_per_pass : 1.0;
  HIPCHK(e, hipMemcpyAsync(e->d_st, &st, sizeof st, hipMemcpyHostToDevice, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  if (int rc_la = la_variant_off(e)) return rc_la;  // a new state: the counts are the caller's to give again
  if (int rc_c = census(e, e->census0)) return rc_c;
  e->loaded = true;
  e->lists_dirty = true;
  e->keys_valid = false;
  return MSKG_OK;
}

// A grid-sized device map of the coupling (LenX * LenY * (LenZ+1) int32).
static int32_t *field_buffer(mskg_engine *e, int k) {
  if (!e->d_field[k]) {
    const Box &b = e->box;
    if (hipMalloc(&e->d_field[k], (size_t)b.lx * b.ly * (b.lz + 1) * sizeof(int32_t)) != hipSuccess) {
      e->d_field[k] = nullptr;
      fail_(e, MSKG_ENOMEM, "no device memory for a %d x %d x %d map", b.lx, b.ly, b.lz + 1);
    }
  }
  return e->d_field[k];
}

static int set_temperature_map(mskg_engine *e, const int32_t *map, int layout, int on_device) {
  const Box &b = e->box;
  const bool strict = layout == FIELD_LATTCOO;
  const int64_t n = (int64_t)b.lx * b.ly * (strict ? b.lz + 1 : b.lz);
  const int32_t *f = map;
  if (!on_device) {
    int32_t *buf = field_buffer(e, 0);
    if (!buf) return MSKG_ENOMEM;
    HIPCHK(e, hipMemcpyAsync(buf, map, n * sizeof(int32_t), hipMemcpyHostToDevice, e->stream));
    f = buf;
  }
  const int blocks = (int)std::min<int64_t>((std::max<int64_t>(n, b.npts) + 255) / 256, 256 * 64);
  if (strict) {
    int bad = 0;
    HIPCHK(e, hipMemsetAsync(e->d_err, 0, sizeof(int), e->stream));
    hipLaunchKernelGGL(k_check_field, dim3(blocks), dim3(256), 0, e->stream, make_lattice(e), f, layout, e->d_err);
    HIPCHK(e, hipGetLastError());
    HIPCHK(e, hipMemcpyAsync(&bad, e->d_err, sizeof(int), hipMemcpyDeviceToHost, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    if (bad) return fail_(e, MSKG_EINVAL, "a temperature is out of the 13-bit range 0..8191 K");
  }
  hipLaunchKernelGGL(k_set_temperature, dim3(blocks), dim3(256), 0, e->stream, make_lattice(e), f, layout,
                     strict ? 1 : 0);
  HIPCHK(e, hipGetLastError());
  HIPCHK(e, hipStreamSynchronize(e->stream));
  return MSKG_OK;
}

// The laser-annealing maps and forms cover the whole grid: they need every plane stored.
static int whole_grid(mskg_engine *e, const char *what) {
  if (e->windowed)
    return fail_(e, MSKG_EINVAL, "%s needs every grid plane stored (stored_len_z %d of %d)", what, e->box.lz + 1,
                 e->logical_lz + 1);
  return MSKG_OK;
}

int mskg_set_temperature(mskg_engine *e, const int32_t *temp_k) {
  if (!e || !temp_k) return MSKG_EINVAL;
  if (!e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  if (int rc = whole_grid(e, "the temperature map")) return rc;
  return set_temperature_map(e, temp_k, FIELD_LATTCOO, 0);
}

int mskg_set_temperature_field(mskg_engine *e, const int32_t *field, int32_t layout, int32_t on_device) {
  if (!e || !field) return MSKG_EINVAL;
  if (!e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  if (int rc = whole_grid(e, "the temperature map")) return rc;
  if (layout != MSKG_FIELD_SOCKET && layout != MSKG_FIELD_PLANES)
    return fail_(e, MSKG_EINVAL, "field layout %d: 0 (socket) or 1 (planes)", layout);
  return set_temperature_map(e, field, layout, on_device);
}

int mskg_phases(mskg_engine *e, int32_t *coor, int32_t *species, int32_t layout, int32_t on_device) {
  if (!e) return MSKG_EINVAL;
  if (!e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  if (int rc = whole_grid(e, "the phase maps")) return rc;
  if (layout != MSKG_FIELD_SOCKET && layout != MSKG_FIELD_PLANES)
    return fail_(e, MSKG_EINVAL, "phase map layout %d: 0 (socket) or 1 (planes)", layout);
  if (!coor && !species) return MSKG_OK;
  const Box &b = e->box;
  const int64_t n = (int64_t)b.lx * b.ly * b.lz;
  int32_t *out[2] = {coor, species};
  if (!on_device)
    for (int k = 0; k < 2; k++)
      if (out[k] && !(out[k] = field_buffer(e, k))) return MSKG_ENOMEM;
  const int64_t rows = layout == MSKG_FIELD_SOCKET ? (int64_t)b.lx * b.ly : (int64_t)b.ly * b.lz;
  const int blocks = (int)std::min<int64_t>(rows, 256 * 64);
  hipLaunchKernelGGL(k_phases, dim3(blocks), dim3(256), 0, e->stream, make_lattice(e), (int)layout, e->d_offwall,
                     e->offwall_planes ? 1 : 0, out[0], out[1]);
  HIPCHK(e, hipGetLastError());
  if (!on_device) {
    if (coor) HIPCHK(e, hipMemcpyAsync(coor, out[0], n * sizeof(int32_t), hipMemcpyDeviceToHost, e->stream));
    if (species) HIPCHK(e, hipMemcpyAsync(species, out[1], n * sizeof(int32_t), hipMemcpyDeviceToHost, e->stream));
  }
  HIPCHK(e, hipStreamSynchronize(e->stream));
  return MSKG_OK;
}

// Back to the main build's laser-annealing form (a new state was loaded).
static int la_variant_off(mskg_engine *e) {
  if (!e->tab.la_variant) return MSKG_OK;
  e->tab.la_variant = 0;
  drop_graph(e);
  HIPCHK(e, hipMemcpyAsync(e->d_tab, &e->tab, sizeof(Tables), hipMemcpyHostToDevice, e->stream));
  return MSKG_OK;
}

int mskg_set_la_variant(mskg_engine *e, const double p0[3], const double tm[3], const double sigma[3],
                        const double tflex[3], const int64_t init_count[3], const int64_t count[3]) {
  if (!e || !p0 || !tm || !sigma || !tflex || !init_count || !count) return MSKG_EINVAL;
  if (!e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  if (!e->tab.la_mode) return fail_(e, MSKG_EINVAL, "the laser-annealing build's form needs la_mode");
  if (int rc = whole_grid(e, "the laser-annealing build's form")) return rc;
  for (int k = 0; k < 3; k++)
    if (k < e->ncrystal && !(sigma[k] != 0.0))
      return fail_(e, MSKG_EINVAL, "sigma of species %d is zero", k + 1);
  e->tab.la_variant = 1;
  drop_graph(e);
  e->tab.la_swap = e->ncrystal == 2 && e->cfg.list_crystal[0] == 14 && e->cfg.list_crystal[1] == 32;
  for (int k = 0; k < 3; k++) {
    e->tab.la_p0[k] = p0[k];
    e->tab.la_tm[k] = tm[k];
    e->tab.la_sigma[k] = k < e->ncrystal ? sigma[k] : 1.0;
    e->tab.la_tflex[k] = tflex[k];
  }
  HIPCHK(e, hipMemcpyAsync(e->d_tab, &e->tab, sizeof(Tables), hipMemcpyHostToDevice, e->stream));
  RunState st;
  int rc = read_state(e, st);
  if (rc) return rc;
  st.la_variant = 1;
  for (int k = 0; k < 3; k++) {
    st.cinit[k] = init_count[k];
    st.cc[k] = count[k];
    st.dcc[k] = 0ull;
    st.cl[k] = st.cinit[k] - st.cc[k];
  }
  if (int rc2 = write_state_head(e, st)) return rc2;
  HIPCHK(e, hipStreamSynchronize(e->stream));
  e->lists_dirty = true;
  return MSKG_OK;
}

int mskg_set_st_tables(mskg_engine *e, int32_t ntemp, const int32_t *temps, const double *pe, const double *pd,
                       const double *pabs, const double *pdes) {
  if (!e || ntemp < 0 || (ntemp > 0 && (!temps || !pe || !pd || !pabs || !pdes))) return MSKG_EINVAL;
  if (!e->d_tab) return fail_(e, MSKG_EINVAL, "engine not created");
  if (ntemp > 0 && e->tab.la_mode) return fail_(e, MSKG_EINVAL, "InitSt 'ST' tables and la_mode exclude each other");
  for (int k = 0; k < ntemp; k++) {
    if (temps[k] <= 0 || temps[k] > 8191) return fail_(e, MSKG_EINVAL, "reference temperature %d K out of range", temps[k]);
    if (k && temps[k] <= temps[k - 1])
      return fail_(e, MSKG_EINVAL, "reference temperatures must increase (InterpProbFromField.f:39 assumes it)");
  }
  HIPCHK(e, hipStreamSynchronize(e->stream));
  drop_graph(e);
  hipFree(e->d_st_tables);
  e->d_st_tables = nullptr;
  e->tab.st_n = 0;
  e->tab.st_temp = nullptr;
  e->tab.st_pe = e->tab.st_pd = e->tab.st_pabs = e->tab.st_pdes = nullptr;
  if (ntemp > 0) {
    const size_t n = (size_t)ntemp, off_pe = 256 * ((n * sizeof(int32_t) + 255) / 256);
    const size_t npe = n * 3 * 4096, npd = n * 9, nab = n * 12;
    const size_t bytes = off_pe + (npe + npd + 2 * nab) * sizeof(double);
    HIPCHK(e, hipMalloc(&e->d_st_tables, bytes));
    char *base = (char *)e->d_st_tables;
    double *dpe = (double *)(base + off_pe), *dpd = dpe + npe, *dab = dpd + npd, *dde = dab + nab;
    HIPCHK(e, hipMemcpyAsync(base, temps, n * sizeof(int32_t), hipMemcpyHostToDevice, e->stream));
    HIPCHK(e, hipMemcpyAsync(dpe, pe, npe * sizeof(double), hipMemcpyHostToDevice, e->stream));
    HIPCHK(e, hipMemcpyAsync(dpd, pd, npd * sizeof(double), hipMemcpyHostToDevice, e->stream));
    HIPCHK(e, hipMemcpyAsync(dab, pabs, nab * sizeof(double), hipMemcpyHostToDevice, e->stream));
    HIPCHK(e, hipMemcpyAsync(dde, pdes, nab * sizeof(double), hipMemcpyHostToDevice, e->stream));
    e->tab.st_n = ntemp;
    e->tab.st_temp = (const int *)base;
    e->tab.st_pe = dpe;
    e->tab.st_pd = dpd;
    e->tab.st_pabs = dab;
    e->tab.st_pdes = dde;
  }
  HIPCHK(e, hipMemcpyAsync(e->d_tab, &e->tab, sizeof(Tables), hipMemcpyHostToDevice, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  e->lists_dirty = true;
  return MSKG_OK;
}

int mskg_la_counts(mskg_engine *e, int64_t count[3], int64_t liquid[3]) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  RunState st;
  int rc = read_state(e, st);
  if (rc) return rc;
  for (int k = 0; k < 3; k++) {
    if (count) count[k] = st.cc[k] + (long long)st.dcc[k];
    if (liquid) liquid[k] = st.cinit[k] - (st.cc[k] + (long long)st.dcc[k]);
  }
  return MSKG_OK;
}

// The rate sweep over the stored points [first, end).
// A sweep of the whole lattice recomputes the classes from the records, so
// the tile lists are rebuilt at the next run; a sweep of the layers that
// hold the MC particles of engine-kept lists changes rates only (a point's
// class is zero exactly when its record makes it no MC particle, which a
// sweep does not change), so the lists stay.
static int refresh_range(mskg_engine *e, int64_t first, int64_t end, bool lists_stay) {
  HIPCHK(e, hipMemsetAsync(e->d_err, 0, sizeof(int), e->stream));
  Lattice L = make_lattice(e);
  if (!lists_stay) e->lists_dirty = true;
  HIPCHK(e, hipEventRecord(e->ev0, e->stream));
  const bool la = e->tab.la_mode || e->tab.st_n;
  if (first == 0 && end == e->box.npts) {
    const int blocks = (int)std::min<int64_t>((e->box.npts + 255) / 256, 256 * 64);
    hipLaunchKernelGGL(MSKG_VARIANT(k_rate_sweep, la, e->cov_model), dim3(blocks), dim3(256), 0, e->stream, L,
                       &e->d_st->rtot, e->d_err, 0);
    HIPCHK(e, hipGetLastError());
  } else if (end > first) {
    // one group of four points per thread up to 65536 blocks: the range of
    // the active layers (~57 M points at 512^3) runs in a single round of
    // groups (0.671 of HBM peak, against 0.647-0.650 at 16384 or 4096
    // blocks with several groups per thread)
    const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>((end - first + 1023) / 1024, 65536));
    hipLaunchKernelGGL(MSKG_VARIANT(k_rate_sweep_range, la, e->cov_model), dim3(blocks), dim3(256), 0, e->stream, L,
                       &e->d_st->rtot, e->d_err, 0, first, end);
    HIPCHK(e, hipGetLastError());
  }
  HIPCHK(e, hipEventRecord(e->ev1, e->stream));
  int err = 0;
  HIPCHK(e, hipMemcpyAsync(&err, e->d_err, sizeof(int), hipMemcpyDeviceToHost, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  float ms = 0;
  HIPCHK(e, hipEventElapsedTime(&ms, e->ev0, e->ev1));
  e->sweep_ms = ms;
  e->sweep_points = end - first;
  if (err) return fail_(e, MSKG_ESTATE, "rate sweep: %s", err_name(err));
  return MSKG_OK;
}

int mskg_refresh_rates(mskg_engine *e) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  const int rc = refresh_range(e, 0, e->box.npts, false);
  if (!rc && e->track) e->keys_valid = true;
  return rc;
}

int mskg_refresh_active(mskg_engine *e) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  // the tile layers that hold MC particles: every tile layer that held a
  // list entry since the lists were built is in the window of some colour
  // (windows only widen between sweeps, and a sweep keeps the layers its
  // tiles and their appends touched).  With lists that are not current (an
  // upload, a replay, a whole-lattice sweep since) every point is swept.
  if (e->lists_dirty) return mskg_refresh_rates(e);
  int zlo = 0, zhi = e->ntz - 1;
  {
    int w[32];
    HIPCHK(e, hipMemcpyAsync(w, e->d_win, sizeof w, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    zlo = 0x7fffffff;
    zhi = -1;
    for (int c = 0; c < 8; c++) {
      zlo = std::min(zlo, w[4 * c]);
      zhi = std::max(zhi, w[4 * c + 1]);
    }
    if (zlo > zhi) zlo = 0, zhi = -1;  // no MC particle
    zlo = std::max(zlo, 0);
    zhi = std::min(zhi, e->ntz - 1);
  }
  const Box &b = e->box;
  const int64_t z0 = (int64_t)zlo * e->tile, z1 = zhi < zlo ? z0 : std::min<int64_t>((int64_t)(zhi + 1) * e->tile, b.lz + 1);
  return refresh_range(e, z0 * b.plane, z1 * b.plane, true);
}

int mskg_replay(mskg_engine *e, const mskg_event *log, int64_t n, int32_t clock_mode) {
  if (!e || !e->loaded || (n > 0 && !log)) return fail_(e, MSKG_EINVAL, "replay: no state or no log");
  if (n == 0) return MSKG_OK;
  e->slab = -1;  // the log's sites may lie anywhere
  mskg_event *d_log = nullptr;
  HIPCHK(e, hipMalloc(&d_log, n * sizeof(mskg_event)));
  hipError_t ce = hipMemcpyAsync(d_log, log, n * sizeof(mskg_event), hipMemcpyHostToDevice, e->stream);
  if (ce != hipSuccess) {
    hipFree(d_log);
    return fail_(e, MSKG_EDEVICE, "replay upload: %s", hipGetErrorString(ce));
  }
  Lattice L = make_lattice(e);
  e->lists_dirty = true;
  hipLaunchKernelGGL(MSKG_VARIANT(k_replay, e->tab.la_mode || e->tab.st_n, e->cov_model), dim3(1), dim3(WAVE), 0, e->stream, L, d_log, n, clock_mode, e->d_st);
  hipError_t le = hipGetLastError();
  RunState st;
  int rc = read_state(e, st);
  hipFree(d_log);
  if (le != hipSuccess) return fail_(e, MSKG_EDEVICE, "k_replay launch: %s", hipGetErrorString(le));
  if (rc) return rc;
  if (st.err)
    return fail_(e, MSKG_ESTATE, "replay stopped at event %llu, site (%d,%d,%d): %s", st.events, st.err_site[0],
                 st.err_site[1], st.err_site[2], err_name(st.err));
  return MSKG_OK;
}

// The pass kernels' parameters of an engine (colour 0).
static PassParams pass_params(mskg_engine *e) {
  PassParams P;
  P.L = make_lattice(e);
  P.st = e->d_st;
  P.log = e->d_log;
  P.log_cap = (unsigned long long)e->log_cap;
  P.ntz = e->ntz;
  P.cap = e->cap;
  P.key0 = (uint32_t)e->cfg.seed;
  P.key1 = (uint32_t)(e->cfg.seed >> 32);
  P.colour = 0;
  P.rsum_chunk = e->rsum_chunk;
  P.done = e->d_done;
  P.sched = e->d_done + e->ntiles;
  return P;
}

// The planes and tiles that may hold list entries: of a slab whose list flags
// were cleared when it was built (flags_clean), the touched planes.
struct TouchedTiles {
  int z0, z1;      // planes
  int t0, t1;      // tiles of their layers
  int full, rest;  // blocks: a wave a tile for those, a thread a tile for the others
};
static TouchedTiles touched_tiles(const mskg_engine *e) {
  TouchedTiles T;
  T.z0 = 0;
  T.z1 = e->box.lz;
  if (e->flags_clean) touched_planes(e, T.z0, T.z1);
  const int layer = e->ntx * e->nty;
  T.t0 = T.z0 / e->tile * layer;
  T.t1 = (T.z1 / e->tile + 1) * layer;
  T.full = (T.t1 - T.t0 + 3) / 4;
  T.rest = (e->ntiles - (T.t1 - T.t0) + 255) / 256;
  return T;
}
// The windows of tile layers of the present lists.
static void list_windows(mskg_engine *e, const Lattice &L) {
  const TouchedTiles T = touched_tiles(e);
  const int l0 = T.z0 / e->tile, layers = T.z1 / e->tile - l0 + 1;
  hipLaunchKernelGGL(k_list_window, dim3(layers), dim3(1024), 0, e->stream, L, l0);
}
// The tile lists of the present classes, and their windows.
static int build_lists(mskg_engine *e, const Lattice &L) {
  const TouchedTiles T = touched_tiles(e);
  hipLaunchKernelGGL(k_build_lists, dim3(T.full + T.rest), dim3(256), 0, e->stream, L, e->ntiles, T.z0, T.z1, T.t0, T.t1,
                     T.full, e->flags_zero ? 1 : 0);
  e->flags_zero = false;
  list_windows(e, L);
  HIPCHK(e, hipGetLastError());
  e->lists_dirty = false;
  return MSKG_OK;
}

// The start of a synchronous-sublattice run, on the engine's stream: tile
// lists current, the run's limits in the run state, the tile totals of the
// current rates and the first window (k_sweep_end with tau = 0).  st: the
// run state before it.
static int run_begin(mskg_engine *e, int64_t max_events, double max_time, RunState &st) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  if (max_events < 0) return fail_(e, MSKG_EINVAL, "max_events < 0");
  Lattice L = make_lattice(e);
  int rc = read_state(e, st);
  if (rc) return rc;
  if (st.err) return fail_(e, MSKG_ESTATE, "engine is in an error state: %s", err_name(st.err));
  hipLaunchKernelGGL(k_run_start, dim3(1), dim3(256), 0, e->stream, e->d_st, e->d_win, e->d_list_err,
                     e->lists_dirty ? 1 : 0, (int)e->cfg.tau_policy,
                     e->cfg.events_per_pass > 0 ? e->cfg.events_per_pass : 1.0, max_time,
                     (unsigned long long)max_events);
  if (e->lists_dirty) {
    if (int rc2 = build_lists(e, L)) return rc2;
  } else {
    list_windows(e, L);
  }
  // tile totals of the current rates, then the first window
  // (the touched tiles hold every list, also of a run before this one)
  const TouchedTiles T = touched_tiles(e);
  hipLaunchKernelGGL(k_tile_rates, dim3(T.full + T.rest), dim3(256), 0, e->stream, L, e->ntiles, e->d_st, T.t0, T.t1,
                     T.full);
  HIPCHK(e, hipGetLastError());
  hipLaunchKernelGGL(k_sweep_end, dim3(1), dim3(END_THREADS), 0, e->stream, pass_params(e));
  HIPCHK(e, hipGetLastError());
  return MSKG_OK;
}

// The waves a sweep on one XCD takes, 0: the lattice is too large for it.
// A film in one tile layer keeps a colour's tiles of that layer busy, so about
// as many waves are wanted (a wave that finds no tile free polls memory); an
// XCD has 128 SIMDs, and past that its waves share issue slots that seven
// other XCDs have idle.
// Where the line lies: a sweep's time over the colour passes', SiC, Si, CVD and
// laser annealing in tiles of 16 to 48, films in one tile layer and in two, with
// 64, 81 and 100 tiles a colour and layer.  Windows of four events a tile
// (policy 1): 0.70-0.91, 0.66-0.89 (one of 1.11), 0.70-0.90; of one: 0.69-0.90,
// 0.64-1.00, 0.69-0.96; the shortest (policy 0, k = 1, where the queue's own
// cost, an entry a tile with events or without, counts most) in tiles of 32
// and more: 0.72-0.81, 0.75-0.96, 0.77-1.06, in smaller ones: 0.73-1.03 (mean
// 0.86), 0.78-1.12 (0.93), 0.83-1.27 (1.02).  So 100 is the break-even of the
// shortest windows in small tiles.  Above it longer windows and tiles of 16
// would still gain (121 tiles of 24, k = 4: 7.2, 6.7 ms a run; 144 of 16: 4.8,
// 3.9): the rule does not look at either.
constexpr int XCD_TILES = 100;
static int xcd_waves(const mskg_engine *e) {
  const int colour = e->ntx * e->nty / 4;
  return colour > XCD_TILES ? 0 : (colour + 15) / 8 * 8;
}

int mskg_run(mskg_engine *e, int64_t max_events, double max_time, int64_t *events_done, double *kmc_time,
             int32_t *stop_reason) {
  RunState st;
  int rc = run_begin(e, max_events, max_time, st);
  if (rc) return rc;
  const int slab = run_touches(e);
  const unsigned long long ev_start = st.events;
  const size_t shm = (size_t)e->cap * (4 + 4 + 1) + 16;
  // one sweep = eight colour passes (or one dependency-scheduled launch) +
  // the window/clock update, captured once as a graph and replayed
  if (!e->graph_exec) {
    PassParams P = pass_params(e);
    const bool la = e->tab.la_mode || e->tab.st_n;
    int grid = std::max(1, std::min(e->ntiles / 8 + 1, e->pass_grid));
    const int local = e->schedule == MSKG_SCHEDULE_COLOURS ? 0 : xcd_waves(e);
    if (local) {
      grid = 8 * local;  // workgroups go to the eight XCDs in turn
    } else if (e->schedule == MSKG_SCHEDULE_TILES) {
      // every wave the device holds at once: the waves take tiles from the
      // sweep's queue until it is empty
      int per_cu = 0, cus = 0;
      HIPCHK(e, hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &per_cu, reinterpret_cast<const void *>(MSKG_VARIANT(k_sweep, la, e->cov_model)), WAVE, shm));
      HIPCHK(e, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, e->device));
      grid = std::max(1, per_cu * cus);
    }
    HIPCHK(e, hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
    if (local) {
      hipLaunchKernelGGL(MSKG_VARIANT(k_sweep_xcd, la, e->cov_model), dim3(grid), dim3(WAVE), shm, e->stream, P);
    } else if (e->schedule == MSKG_SCHEDULE_TILES) {
      hipLaunchKernelGGL(MSKG_VARIANT(k_sweep, la, e->cov_model), dim3(grid), dim3(WAVE), shm, e->stream, P);
    } else {
      for (int c = 0; c < 8; c++) {
        P.colour = c;
        hipLaunchKernelGGL(MSKG_VARIANT(k_pass, la, e->cov_model), dim3(grid), dim3(WAVE), shm, e->stream, P);
      }
    }
    hipLaunchKernelGGL(k_sweep_end, dim3(1), dim3(END_THREADS), 0, e->stream, P);
    HIPCHK(e, hipStreamEndCapture(e->stream, &e->graph));
    HIPCHK(e, hipGraphInstantiate(&e->graph_exec, e->graph, nullptr, nullptr, 0));
  }
  int32_t stop = MSKG_STOP_LIMIT;
  HIPCHK(e, hipEventRecord(e->ev0, e->stream));
  int64_t sweeps = 0;
  int batch = 1;
  for (;;) {
    for (int sb = 0; sb < batch; sb++) HIPCHK(e, hipGraphLaunch(e->graph_exec, e->stream));
    sweeps += batch;
    rc = read_state(e, st);
    if (rc) return rc;
    if (st.err) break;
    int64_t done = (int64_t)(st.events - ev_start);
    if (st.stop) { stop = st.stop == STOP_AT_LIMIT ? MSKG_STOP_LIMIT : st.stop; break; }
    if (done >= max_events || st.clock >= max_time) break;
    // size the next batch of sweeps from the observed events per sweep, at
    // most doubling the sweeps run so far: sweeps queued past the stop
    // still cost a launch each
    double per = (double)done / (double)sweeps;
    int64_t want = per > 0 ? (int64_t)((double)(max_events - done) / per * 0.9) : 16;
    batch = (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(want, 512), sweeps));
  }
  HIPCHK(e, hipEventRecord(e->ev1, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  float ms = 0;
  HIPCHK(e, hipEventElapsedTime(&ms, e->ev0, e->ev1));
  run_over(e, slab, st.ever_lo, st.ever_hi);
  e->run_ms = ms;
  e->sweeps_done = sweeps;
  if (events_done) *events_done = (int64_t)(st.events - ev_start);
  if (kmc_time) *kmc_time = st.clock;
  if (stop_reason) *stop_reason = stop;
  if (st.err)
    return fail_(e, MSKG_ESTATE, "run stopped in the tile at (%d,%d,%d): %s", st.err_site[0], st.err_site[1],
                 st.err_site[2], err_name(st.err));
  return MSKG_OK;
}

int mskg_store_state(mskg_engine *e, int32_t *latt, int32_t cap_ad, int32_t *n_ad, int32_t *ad_xyz, int32_t *ad_nn,
                     int32_t *ad_event, double *ad_prob, int32_t cap_bulk, int32_t *n_bulk, int32_t *bulk_xyz,
                     int32_t *bulk_nn, int32_t cap_void, int32_t *n_void, int32_t *void_xyz, int32_t *void_nn) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  int64_t tot[3] = {0, 0, 0};
  const int64_t cap[3] = {cap_ad, cap_bulk, cap_void};
  int32_t *const xyz[3] = {ad_xyz, bulk_xyz, void_xyz}, *const nn[3] = {ad_nn, bulk_nn, void_nn};
  const int rc = state_lists(e, cap, xyz, nn, ad_event, ad_prob, tot);
  int rc2 = MSKG_OK;
  if (!rc && latt) rc2 = state_words(e, latt);
  work_done(e);
  if (rc || rc2) return rc ? rc : rc2;
  const int32_t na = (int32_t)tot[0], nb = (int32_t)tot[1], nv = (int32_t)tot[2];
  if (n_ad) *n_ad = na;
  if (n_bulk) *n_bulk = nb;
  if (n_void) *n_void = nv;
  if (tot[0] > std::max<int64_t>(cap_ad, 0) || tot[1] > std::max<int64_t>(cap_bulk, 0) ||
      tot[2] > std::max<int64_t>(cap_void, 0))
    return fail_(e, MSKG_ECAPACITY, "list capacity too small (need %d MC, %d bulk, %d void)", na, nb, nv);
  return MSKG_OK;
}

int mskg_site_rates(mskg_engine *e, int64_t n, const int32_t *xyz, int32_t *cls_out, float *rate_out) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  if (n <= 0) return MSKG_OK;
  // the sites in pieces of up to 1M, through one workspace: first bad site,
  // then positions, classes and rates (20 bytes a site)
  constexpr int64_t PIECE = 1 << 20;
  const int64_t cap = std::min(n, PIECE);
  char *w = (char *)work_take(e, 0, 16 + (size_t)cap * 20);
  if (!w) return fail_(e, MSKG_ENOMEM, "site rates: no device memory for %lld sites", (long long)cap);
  unsigned int *d_bad = (unsigned int *)w;
  int32_t *d_xyz = (int32_t *)(w + 16), *d_cls = d_xyz + 3 * cap;
  float *d_rate = (float *)(d_cls + cap);
  int rc = MSKG_OK;
  for (int64_t i0 = 0; i0 < n && !rc; i0 += cap) {
    const int64_t m = std::min(cap, n - i0);
    unsigned int bad = 0xffffffffu;
    hipError_t ce = hipMemsetAsync(d_bad, 0xff, sizeof bad, e->stream);
    if (ce == hipSuccess)
      ce = hipMemcpyAsync(d_xyz, xyz + 3 * i0, (size_t)m * 12, hipMemcpyHostToDevice, e->stream);
    if (ce == hipSuccess) {
      hipLaunchKernelGGL(k_site_rates, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, e->stream, make_lattice(e), m,
                         d_xyz, d_cls, d_rate, d_bad);
      ce = hipGetLastError();
    }
    if (ce == hipSuccess) ce = hipMemcpyAsync(&bad, d_bad, sizeof bad, hipMemcpyDeviceToHost, e->stream);
    if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
    // the sites before the first that is no lattice point are given
    const int64_t good = std::min<int64_t>(m, bad);
    if (ce == hipSuccess && good)
      ce = hipMemcpyAsync(cls_out + i0, d_cls, (size_t)good * 4, hipMemcpyDeviceToHost, e->stream);
    if (ce == hipSuccess && good)
      ce = hipMemcpyAsync(rate_out + i0, d_rate, (size_t)good * 4, hipMemcpyDeviceToHost, e->stream);
    if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
    if (ce != hipSuccess) {
      rc = fail_(e, MSKG_EDEVICE, "site rates: %s", hipGetErrorString(ce));
    } else if (good < m) {
      const int32_t *s = xyz + 3 * (i0 + good);
      rc = fail_(e, MSKG_EINVAL, "site %lld (%d,%d,%d) is not a lattice point", (long long)(i0 + good), s[0], s[1], s[2]);
    }
  }
  work_done(e);
  return rc;
}

static int census(mskg_engine *e, int64_t out[6]) {
  unsigned long long *d = nullptr;
  if (hipMalloc(&d, 6 * sizeof(unsigned long long)) != hipSuccess)
    return fail_(e, MSKG_ENOMEM, "census: no device memory");
  unsigned long long h[6];
  hipError_t ce = hipMemsetAsync(d, 0, 6 * sizeof(unsigned long long), e->stream);
  if (ce == hipSuccess) {
    const int blocks = (int)std::min<int64_t>((e->box.npts + 255) / 256, 256 * 64);
    hipLaunchKernelGGL(k_census, dim3(blocks), dim3(256), 0, e->stream, make_lattice(e), d);
    ce = hipGetLastError();
  }
  if (ce == hipSuccess) ce = hipMemcpyAsync(h, d, sizeof h, hipMemcpyDeviceToHost, e->stream);
  if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
  hipFree(d);
  if (ce != hipSuccess) return fail_(e, MSKG_EDEVICE, "census: %s", hipGetErrorString(ce));
  for (int q = 0; q < 6; q++) out[q] = (int64_t)h[q];
  return MSKG_OK;
}

int mskg_species_counts(mskg_engine *e, int64_t evaporated[3], int64_t desorbed[3]) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  RunState st;
  int rc = read_state(e, st);
  if (rc) return rc;
  int64_t now[6];
  if ((rc = census(e, now))) return rc;
  for (int k = 0; k < 3; k++) {
    if (evaporated) evaporated[k] = (int64_t)st.counts[k] - (now[k] - e->census0[k]);
    if (desorbed) desorbed[k] = (int64_t)st.desorbed[k];
  }
  return MSKG_OK;
}

int mskg_counters(mskg_engine *e, int64_t counts[8], double *kmc_time, int64_t *n_adatom, int64_t *n_atoms,
                  int64_t *n_voids) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  RunState st;
  int rc = read_state(e, st);
  if (rc) return rc;
  if (counts)
    for (int i = 0; i < 8; i++) counts[i] = (int64_t)st.counts[i];
  if (kmc_time) *kmc_time = st.clock;
  if (n_adatom || n_atoms || n_voids) {
    int32_t na = 0, nb = 0, nv = 0;
    rc = mskg_store_state(e, nullptr, 0, &na, nullptr, nullptr, nullptr, nullptr, 0, &nb, nullptr, nullptr, 0, &nv,
                          nullptr, nullptr);
    if (rc && rc != MSKG_ECAPACITY) return rc;
    e->err.clear();
    if (n_adatom) *n_adatom = na;
    if (n_atoms) *n_atoms = nb;
    if (n_voids) *n_voids = nv;
  }
  return MSKG_OK;
}

int mskg_last_timing(mskg_engine *e, double *run_ms, double *sweep_ms, int64_t *sweep_points, int64_t *sweeps_done) {
  if (!e) return MSKG_EINVAL;
  if (run_ms) *run_ms = e->run_ms;
  if (sweep_ms) *sweep_ms = e->sweep_ms;
  if (sweep_points) *sweep_points = e->sweep_points;
  if (sweeps_done) *sweeps_done = e->sweeps_done;
  return MSKG_OK;
}

int mskg_set_schedule(mskg_engine *e, int32_t schedule) {
  if (!e) return MSKG_EINVAL;
  if (schedule != MSKG_SCHEDULE_TILES && schedule != MSKG_SCHEDULE_COLOURS)
    return fail_(e, MSKG_EINVAL, "schedule %d: MSKG_SCHEDULE_TILES (1) or MSKG_SCHEDULE_COLOURS (0)", schedule);
  if (schedule != e->schedule) {
    HIPCHK(e, hipStreamSynchronize(e->stream));
    drop_graph(e);
    e->schedule = schedule;
  }
  return MSKG_OK;
}

int mskg_run_diagnostics(mskg_engine *e, int64_t *guard_exits, int64_t *sweeps, double *tau, int64_t *n_mc) {
  if (!e || !e->loaded) return fail_(e, MSKG_EINVAL, "no state loaded");
  RunState st;
  int rc = read_state(e, st);
  if (rc) return rc;
  if (guard_exits) *guard_exits = (int64_t)st.guard_exits;
  if (sweeps) *sweeps = (int64_t)st.sweeps_run;
  if (tau) *tau = st.tau;
  if (n_mc) *n_mc = (int64_t)st.n_mc;
  return MSKG_OK;
}

static int build_slab(mskg_engine *e, int32_t mode, int32_t len, double fraction);

int mskg_build_slab(mskg_engine *e, int32_t mode, int32_t len) {
  if (!e || !e->d_site) return MSKG_EINVAL;
  if (mode != 0 && mode != 1) return fail_(e, MSKG_EINVAL, "mode must be 0 (SetSi) or 1 (SetSiC3C)");
  return build_slab(e, mode, len, 0.0);
}

int mskg_build_alloy_slab(mskg_engine *e, int32_t len, double fraction) {
  if (!e || !e->d_site) return MSKG_EINVAL;
  if (!(fraction >= 0.0 && fraction <= 1.0)) return fail_(e, MSKG_EINVAL, "alloy fraction must be in [0, 1]");
  if (e->ncrystal < 2) return fail_(e, MSKG_EINVAL, "an alloy needs n_crystal >= 2");
  return build_slab(e, 2, len, fraction);
}

static int build_slab(mskg_engine *e, int32_t mode, int32_t len, double fraction) {
  if (len < 6 || len > e->logical_lz - (mode != 1 ? 7 : 1) || len % 3)
    return fail_(e, MSKG_EINVAL, "slab height %d does not fit the box height %d", len, e->logical_lz);
  if (e->windowed && len + 6 > e->box.lz - TOP_MARGIN)
    return fail_(e, MSKG_EINVAL, "slab height %d: the stored planes (stored_len_z %d) need %d more above it", len,
                 e->box.lz + 1, TOP_MARGIN + 6);
  Lattice L = make_lattice(e);
  e->slab = -1;
  const int blocks = (int)std::min<int64_t>((e->box.npts + 255) / 256, 4096);
  unsigned long long *d_atoms = (unsigned long long *)work_take(e, 0, 2 * sizeof(unsigned long long));
  if (!d_atoms) return fail_(e, MSKG_ENOMEM, "slab: no device memory for the census");
  // the total rate of the initial population seeds the isolated-atom rule
  const double nsurf = (double)e->box.lx * e->box.ly / 36.0;  // 2 atoms per (6x6) surface cell per layer
  const Tables &t = e->tab;
  const double rtot = nsurf * (mode ? 0.5 * (t.pe[0 + 3 * 2] + t.pe[1 + 3 * 2]) : t.pe[0 + 3 * 2]) +
                      nsurf * (t.pd[0 + 3] + t.pd[1 + 3] + t.pd[2 + 3]);
  hipLaunchKernelGGL(k_state_new, dim3(1), dim3(256), 0, e->stream, e->d_st,
                     e->cfg.events_per_pass > 0 ? e->cfg.events_per_pass : 1.0, rtot, d_atoms, e->d_err);
  hipLaunchKernelGGL(k_build_slab, dim3(blocks), dim3(256), 0, e->stream, L, len, mode, fraction,
                     (uint32_t)e->cfg.seed, (uint32_t)(e->cfg.seed >> 32), e->logical_lz, d_atoms);
  HIPCHK(e, hipGetLastError());
  if (e->d_offwall) hipFree(e->d_offwall);  // the SetSi builders fill their wall planes at every grid point
  e->d_offwall = nullptr;
  e->offwall_planes = mode != 1;
  if (e->tab.use_f2 || mode == 2) {
    // the surface atoms' rates from their neighbours (species, second shell):
    // every atom of coordination 1..3 lies in the planes len-3..len-1
    const int64_t first = (len - 3) * e->box.plane, end = len * e->box.plane;
    const int sb = (int)std::max<int64_t>(1, std::min<int64_t>((end - first + 1023) / 1024, 65536));
    hipLaunchKernelGGL(MSKG_VARIANT(k_rate_sweep_range, e->tab.la_mode || e->tab.st_n, e->cov_model), dim3(sb), dim3(256),
                       0, e->stream, L, (const double *)nullptr, e->d_err, 1, first, end);
    HIPCHK(e, hipGetLastError());
  }
  unsigned long long atoms[2];
  HIPCHK(e, hipMemcpyAsync(atoms, d_atoms, sizeof atoms, hipMemcpyDeviceToHost, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  if (int rc_la = la_variant_off(e)) return rc_la;  // a new state: the counts are the caller's to give again
  for (int k = 0; k < 6; k++) e->census0[k] = k < 2 ? (int64_t)atoms[k] : 0;
  e->loaded = true;
  e->lists_dirty = true;
  e->keys_valid = false;
  e->flags_clean = e->flags_zero = true;
  e->slab = mode;
  e->slab_z0 = len - 3;  // the surface atoms ...
  e->slab_z1 = len;      // ... and the empty sites above them
  return MSKG_OK;
}

// A shaped initial state built on the device (k_shape_place ->
// k_shape_isolated -> k_shape_records -> rate sweep), and the off-lattice
// wall bits of the builders that fill wall regions.
static int build_shape(mskg_engine *e, ShapeSpec S, bool walls_off_lattice) {
  if (e->windowed)
    return fail_(e, MSKG_EINVAL, "the shaped builders fill the whole box: every plane must be stored");
  S.lz = e->logical_lz;
  S.key0 = (uint32_t)e->cfg.seed;
  S.key1 = (uint32_t)(e->cfg.seed >> 32);
  S.cx = e->box.lx / 2;
  S.cy = e->box.ly / 2;
  S.cz = e->logical_lz / 2;
  e->slab = -1;
  Lattice L = make_lattice(e);
  L.key = nullptr;
  const int blocks = (int)std::min<int64_t>((e->box.npts + 255) / 256, 256 * 64);
  unsigned long long *d_atoms = (unsigned long long *)work_take(e, 0, 2 * sizeof(unsigned long long));
  if (!d_atoms) return fail_(e, MSKG_ENOMEM, "builder: no device memory for the census");
  HIPCHK(e, hipMemsetAsync(d_atoms, 0, 2 * sizeof(unsigned long long), e->stream));
  HIPCHK(e, hipMemsetAsync(e->d_err, 0, sizeof(int), e->stream));
  hipLaunchKernelGGL(k_shape_place, dim3(blocks), dim3(256), 0, e->stream, L, S);
  hipLaunchKernelGGL(k_shape_isolated, dim3(blocks), dim3(256), 0, e->stream, L, S);
  hipLaunchKernelGGL(k_shape_records, dim3(blocks), dim3(256), 0, e->stream, L, S, e->d_err,
                     d_atoms);
  hipLaunchKernelGGL(MSKG_VARIANT(k_rate_sweep, e->tab.la_mode || e->tab.st_n, e->cov_model), dim3(blocks),
                     dim3(256), 0, e->stream, L, (const double *)nullptr, e->d_err, 0);
  hipLaunchKernelGGL(k_initial_placeholders, dim3(blocks), dim3(256), 0, e->stream, L);
  HIPCHK(e, hipGetLastError());
  if (!walls_off_lattice) {
    hipFree(e->d_offwall);
    e->d_offwall = nullptr;
  }
  e->offwall_planes = false;
  if (walls_off_lattice) {
    const int64_t words = (e->box.lx * (int64_t)e->box.ly * (e->box.lz + 1) + 31) / 32;
    if (!e->d_offwall) HIPCHK(e, hipMalloc(&e->d_offwall, words * sizeof(uint32_t)));
    const int wb = (int)std::min<int64_t>((words * 8 + 255) / 256, 256 * 64);
    hipLaunchKernelGGL(k_shape_offwall, dim3(wb), dim3(256), 0, e->stream, L, S, e->d_offwall, words);
    HIPCHK(e, hipGetLastError());
  }
  int err = 0;
  HIPCHK(e, hipMemcpyAsync(&err, e->d_err, sizeof(int), hipMemcpyDeviceToHost, e->stream));
  unsigned long long atoms[2];
  HIPCHK(e, hipMemcpyAsync(atoms, d_atoms, sizeof atoms, hipMemcpyDeviceToHost, e->stream));
  // the new run state only now: the rates above go by the liquid counts of the state before
  RunState st;
  memset(&st, 0, sizeof st);
  st.events_per_pass = e->cfg.events_per_pass > 0 ? e->cfg.events_per_pass : 1.0;
  HIPCHK(e, hipMemcpyAsync(e->d_st, &st, sizeof st, hipMemcpyHostToDevice, e->stream));
  HIPCHK(e, hipStreamSynchronize(e->stream));
  e->loaded = true;  // the state is the builder's, whatever follows
  e->lists_dirty = true;
  e->keys_valid = false;
  if (err) {
    e->loaded = false;
    return fail_(e, MSKG_ESTATE, "shaped builder: %s", err_name(err));
  }
  if (int rc_la = la_variant_off(e)) return rc_la;
  for (int k = 0; k < 6; k++) e->census0[k] = k < 2 ? (int64_t)atoms[k] : 0;
  return MSKG_OK;
}

int mskg_build_shape(mskg_engine *e, const char *init_st, const int32_t lens[4]) {
  if (!e || !e->d_site || !init_st || !lens) return MSKG_EINVAL;
  const std::string is(init_st);
  if (is == "F" || is == "FS") return mskg_build_slab(e, is == "F" ? 1 : 0, lens[0] - lens[0] % 24);
  ShapeSpec S;
  memset(&S, 0, sizeof S);
  S.zfix = -1;
  S.l1 = lens[0]; S.l2 = lens[1]; S.l3 = lens[2]; S.l4 = lens[3];
  if (is == "C" || is == "S") {  // SetNC.f:25-235, SetNCSp.f:25-237
    S.shape = is == "C" ? SHAPE_BOX : SHAPE_SPHERE;
    if (S.l1 <= 0 || (is == "C" && (S.l2 <= 0 || S.l3 <= 0)))
      return fail_(e, MSKG_EINVAL, "InitSt %s: the shape's lengths must be positive", init_st);
    return build_shape(e, S, false);
  }
  if (is == "I") {  // SetInvPOff.f:21-286: Len1 the pyramid, Len2 the substrate top
    S.shape = SHAPE_INVP;
    S.zfix = 20;
    if (S.l2 <= 21 || S.l2 + 10 > e->logical_lz)
      return fail_(e, MSKG_EINVAL, "InitSt I: Len2 %d must lie in 22..LenZ-10", S.l2);
    return build_shape(e, S, false);
  }
  if (is == "FF") {  // SetSiFINFET.f:25-312 with main.f:281-285's reductions
    S.shape = SHAPE_FINFET;
    S.l1 -= S.l1 % 24; S.l2 -= S.l2 % 24; S.l3 -= S.l3 % 24; S.l4 -= S.l4 % 24;
    if (S.l1 < 6 || S.l3 + 10 > e->logical_lz)
      return fail_(e, MSKG_EINVAL, "InitSt FF: lengths %d %d %d %d do not fit the box", S.l1, S.l2, S.l3, S.l4);
    S.xa = (int)(0.5f * (float)(e->box.lx - S.l4));
    S.xb = (int)(0.5f * (float)(e->box.lx + S.l4));
    S.walls = 1;
    return build_shape(e, S, true);
  }
  return fail_(e, MSKG_EINVAL, "InitSt '%s': the device builds F, FS, C, S, I, FF (and IN with mskg_build_cad)",
               init_st);
}

int mskg_build_cad(mskg_engine *e, const int8_t *ids, int32_t on_device, double alloy_fraction) {
  if (!e || !e->d_site || !ids) return MSKG_EINVAL;
  if (!(alloy_fraction >= 0.0 && alloy_fraction <= 1.0))
    return fail_(e, MSKG_EINVAL, "alloy fraction must be in [0, 1]");
  if (alloy_fraction > 0.0 && e->ncrystal < 2) return fail_(e, MSKG_EINVAL, "an alloy needs n_crystal >= 2");
  if (e->logical_lz < 10) return fail_(e, MSKG_EINVAL, "SetCAD needs LenZ >= 10");
  if (e->windowed)
    return fail_(e, MSKG_EINVAL, "the shaped builders fill the whole box: every plane must be stored");
  ShapeSpec S;
  memset(&S, 0, sizeof S);
  S.shape = SHAPE_CAD;
  S.zfix = -1;
  S.walls = 1;
  S.fraction = alloy_fraction;
  int8_t *d_ids = nullptr;
  const size_t nb = (size_t)e->box.lx * e->box.ly * e->logical_lz;
  if (on_device) {
    S.ids = ids;
  } else {
    HIPCHK(e, hipMalloc(&d_ids, nb));
    hipError_t ce = hipMemcpyAsync(d_ids, ids, nb, hipMemcpyHostToDevice, e->stream);
    if (ce != hipSuccess) {
      hipFree(d_ids);
      return fail_(e, MSKG_EDEVICE, "geometry upload: %s", hipGetErrorString(ce));
    }
    S.ids = d_ids;
  }
  const int rc = build_shape(e, S, true);
  hipStreamSynchronize(e->stream);
  hipFree(d_ids);
  return rc;
}

int mskg_track_classes(mskg_engine *e, int32_t on) {
  if (!e || !e->d_site) return MSKG_EINVAL;
  if (!on) {
    if (e->track) drop_graph(e);
    e->track = false;
    e->keys_valid = false;
    return MSKG_OK;
  }
  if (e->tab.ncov || e->tab.la_mode)
    return fail_(e, MSKG_EINVAL, "class keys cover models without coverage species and without LA rates");
  const int64_t np = e->box.npts;
  if (!e->d_key) {
    HIPCHK(e, hipMalloc(&e->d_key, np * sizeof(int32_t)));
    HIPCHK(e, hipMalloc(&e->d_key_seen, np * sizeof(int32_t)));
    HIPCHK(e, hipMalloc(&e->d_rate_seen, np * sizeof(float)));
  }
  if (!e->track) drop_graph(e);
  e->track = true;
  e->keys_valid = false;
  if (!e->loaded) return MSKG_OK;
  return mskg_refresh_rates(e);  // a keyed sweep: rates and keys from the state
}

int mskg_copy_state(mskg_engine *dst, const mskg_engine *src) {
  if (!dst || !src || !src->loaded) return MSKG_EINVAL;
  if (dst == src) return MSKG_OK;
  if (dst->box.lx != src->box.lx || dst->box.ly != src->box.ly || dst->box.lz != src->box.lz ||
      dst->logical_lz != src->logical_lz ||
      dst->tile != src->tile)
    return fail_(dst, MSKG_EINVAL, "copy_state: engines differ in box or tile");
  const int64_t np = dst->box.npts;
  dst->slab = -1;
  dst->flags_clean = dst->flags_zero = false;
  HIPCHK(dst, hipStreamSynchronize(src->stream));
  HIPCHK(dst, hipMemcpyAsync(dst->d_site, src->d_site, np * sizeof(Site), hipMemcpyDeviceToDevice, dst->stream));
  HIPCHK(dst, hipMemcpyAsync(dst->d_rate, src->d_rate, np * sizeof(float), hipMemcpyDeviceToDevice, dst->stream));
  HIPCHK(dst, hipMemcpyAsync(dst->d_cls, src->d_cls, np, hipMemcpyDeviceToDevice, dst->stream));
  dst->keys_valid = false;
  hipFree(dst->d_offwall);
  dst->d_offwall = nullptr;
  dst->offwall_planes = src->offwall_planes;
  if (src->d_offwall) {
    const size_t words = (size_t)((src->box.lx * (int64_t)src->box.ly * (src->box.lz + 1) + 31) / 32);
    HIPCHK(dst, hipMalloc(&dst->d_offwall, words * sizeof(uint32_t)));
    HIPCHK(dst, hipMemcpyAsync(dst->d_offwall, src->d_offwall, words * sizeof(uint32_t), hipMemcpyDeviceToDevice,
                               dst->stream));
  }
  if (dst->track && src->track && src->keys_valid) {
    HIPCHK(dst, hipMemcpyAsync(dst->d_key, src->d_key, np * sizeof(int32_t), hipMemcpyDeviceToDevice, dst->stream));
    dst->keys_valid = true;
  }
  RunState st;
  HIPCHK(dst, hipMemcpyAsync(&st, src->d_st, sizeof st, hipMemcpyDeviceToHost, dst->stream));
  HIPCHK(dst, hipStreamSynchronize(dst->stream));
  RunState s0;
  memset(&s0, 0, sizeof s0);
  s0.clock = st.clock;
  s0.rtot = st.rtot;
  s0.events_per_pass = dst->cfg.events_per_pass > 0 ? dst->cfg.events_per_pass : 1.0;
  s0.la_variant = dst->tab.la_variant;
  for (int k = 0; k < 3; k++) {
    s0.cc[k] = st.cc[k] + (long long)st.dcc[k];
    s0.cinit[k] = st.cinit[k];
    s0.cl[k] = s0.cinit[k] - s0.cc[k];
  }
  HIPCHK(dst, hipMemcpyAsync(dst->d_st, &s0, sizeof s0, hipMemcpyHostToDevice, dst->stream));
  HIPCHK(dst, hipStreamSynchronize(dst->stream));
  if (int rc = census(dst, dst->census0)) return rc;  // the event counters restart here
  dst->loaded = true;
  dst->lists_dirty = true;
  dst->slab = src->slab;
  dst->slab_z0 = src->slab_z0;
  dst->slab_z1 = src->slab_z1;
  return MSKG_OK;
}

int mskg_set_event_log(mskg_engine *e, int64_t capacity) {
  if (!e || capacity < 0) return MSKG_EINVAL;
  if (e->d_log) { HIPCHK(e, hipFree(e->d_log)); e->d_log = nullptr; }
  e->log_cap = 0;
  if (capacity > 0) {
    HIPCHK(e, hipMalloc(&e->d_log, capacity * sizeof(mskg_event)));
    e->log_cap = capacity;
  }
  drop_graph(e);
  if (e->loaded) {
    RunState st;
    int rc = read_state(e, st);
    if (rc) return rc;
    st.log_n = 0;
    if (int rc2 = write_state_head(e, st)) return rc2;
    HIPCHK(e, hipStreamSynchronize(e->stream));
  }
  return MSKG_OK;
}

int mskg_get_event_log(mskg_engine *e, mskg_event *out, int64_t cap, int64_t *n) {
  if (!e || !n) return MSKG_EINVAL;
  RunState st;
  int rc = read_state(e, st);
  if (rc) return rc;
  *n = (int64_t)st.log_n;
  if (st.log_n > (unsigned long long)e->log_cap)
    return fail_(e, MSKG_ECAPACITY, "event log overflowed: %lld events, capacity %lld", (long long)st.log_n,
                 (long long)e->log_cap);
  int64_t m = std::min<int64_t>(*n, cap);
  if (m > 0 && out) {
    HIPCHK(e, hipMemcpyAsync(out, e->d_log, m * sizeof(mskg_event), hipMemcpyDeviceToHost, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
  }
  return MSKG_OK;
}

int mskg_geometry_find_nn(const int32_t s1[3], const int32_t s2[3], const int32_t sc[3], int32_t len_x, int32_t len_y,
                          int32_t out[6]) {
  Geometry g;
  build_geometry(g);
  int a[3] = {s1[0], s1[1], s1[2]}, b[3] = {s2[0], s2[1], s2[2]}, c[3] = {sc[0], sc[1], sc[2]}, o[2][3];
  find_nn(g, len_x, len_y, a, b, c, o);
  for (int r = 0; r < 2; r++)
    for (int k = 0; k < 3; k++) out[3 * r + k] = o[r][k];
  return MSKG_OK;
}

int mskg_geometry_find_sn(const int32_t site[3], const int32_t sitec[3], const int32_t sn[9], int32_t len_x,
                          int32_t len_y, int32_t zig[9], int32_t arm[9]) {
  Geometry g;
  build_geometry(g);
  int s[3] = {site[0], site[1], site[2]}, c[3] = {sitec[0], sitec[1], sitec[2]}, n[3][3], zz[3][3], aa[3][3];
  for (int i = 0; i < 3; i++)
    for (int k = 0; k < 3; k++) n[i][k] = sn[3 * i + k];
  find_sn(g, len_x, len_y, s, c, n, zz, aa);
  for (int i = 0; i < 3; i++)
    for (int k = 0; k < 3; k++) {
      zig[3 * i + k] = zz[i][k];
      arm[3 * i + k] = aa[i][k];
    }
  return MSKG_OK;
}

int mskg_run_serial(mskg_engine *const *engines, int32_t n, const int64_t *max_events, const double *max_time,
                    int64_t *events_done, double *kmc_time, int32_t *stop_reason) {
  if (!engines || n <= 0 || !max_events || !max_time) return MSKG_EINVAL;
  mskg_engine *e0 = engines[0];
  if (!e0) return MSKG_EINVAL;
  std::vector<SerialDesc> descs(n);
  std::vector<unsigned long long> ev0(n);
  bool any_la = false, any_cov = false;
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    if (!e || !e->loaded) return fail_(e0, MSKG_EINVAL, "serial run: replica %d has no state loaded", i);
    any_la |= e->tab.la_mode != 0 || e->tab.st_n > 0;
    if (e->tab.la_variant)
      return fail_(e0, MSKG_EINVAL, "serial run: replica %d uses the laser-annealing build's rate form", i);
    any_cov |= e->cov_model;
    if (max_events[i] < 0) return fail_(e, MSKG_EINVAL, "max_events < 0");
    for (int j = 0; j < i; j++)
      if (engines[j] == e) return fail_(e0, MSKG_EINVAL, "serial run: replica %d appears twice", i);
    const int nblk = (e->ntiles + WAVE - 1) / WAVE;
    if (!e->d_tsum) {
      HIPCHK(e, hipMalloc(&e->d_tsum, e->ntiles * sizeof(double)));
      HIPCHK(e, hipMalloc(&e->d_bsum, nblk * sizeof(double)));
    }
    Lattice L = make_lattice(e);
    if (e->lists_dirty) {
      HIPCHK(e, hipMemsetAsync(e->d_list_err, 0, sizeof(int), e->stream));
      if (int rc2 = build_lists(e, L)) return rc2;
    }
    e->slab = -1;  // the serial run keeps no record of the layers it visits
    SerialDesc &D = descs[i];
    D.L = L;
    D.tsum = e->d_tsum;
    D.bsum = e->d_bsum;
    D.st = e->d_st;
    D.log = e->d_log;
    D.log_cap = (unsigned long long)e->log_cap;
    D.max_events = max_events[i];
    D.max_time = max_time[i];
    D.key0 = (uint32_t)e->cfg.seed;
    D.key1 = (uint32_t)(e->cfg.seed >> 32) ^ 0x5e1a1u;  // a stream apart from the sublattice passes
    D.ntiles = e->ntiles;
    D.nblk = nblk;
    D.replica = i;
  }
  std::vector<RunHead> head;
  if (int rc = read_heads(engines, n, head)) return rc;
  for (int i = 0; i < n; i++) {
    if (head[i].err)
      return fail_(engines[i], MSKG_ESTATE, "engine is in an error state: %s", err_name(head[i].err));
    if (head[i].list_err) return fail_(engines[i], MSKG_ECAPACITY, "a tile holds more MC particles than tile_capacity");
    ev0[i] = head[i].events;
  }
  SerialDesc *d_descs = nullptr;
  HIPCHK(e0, hipMalloc(&d_descs, n * sizeof(SerialDesc)));
  hipError_t ce = hipMemcpyAsync(d_descs, descs.data(), n * sizeof(SerialDesc), hipMemcpyHostToDevice, e0->stream);
  if (ce == hipSuccess) {
    HIPCHK(e0, hipEventRecord(e0->ev0, e0->stream));
    hipLaunchKernelGGL(MSKG_VARIANT(k_serial, any_la, any_cov), dim3(n), dim3(WAVE), 0, e0->stream, d_descs);
    ce = hipGetLastError();
    if (ce == hipSuccess) ce = hipEventRecord(e0->ev1, e0->stream);
    if (ce == hipSuccess) ce = hipStreamSynchronize(e0->stream);
  }
  hipFree(d_descs);
  if (ce != hipSuccess) return fail_(e0, MSKG_EDEVICE, "k_serial: %s", hipGetErrorString(ce));
  float ms = 0;
  HIPCHK(e0, hipEventElapsedTime(&ms, e0->ev0, e0->ev1));
  if (int rc = read_heads(engines, n, head)) return rc;
  int rc_all = MSKG_OK;
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    const RunHead &st = head[i];
    e->run_ms = ms;
    e->lists_dirty = false;
    if (events_done) events_done[i] = (int64_t)(st.events - ev0[i]);
    if (kmc_time) kmc_time[i] = st.clock;
    if (stop_reason) stop_reason[i] = st.stop;
    if (st.err && rc_all == MSKG_OK)
      rc_all = fail_(e, MSKG_ESTATE, "serial run of replica %d stopped: %s", i, err_name(st.err));
    if (e->d_log && st.log_n > (unsigned long long)e->log_cap && rc_all == MSKG_OK)
      rc_all = fail_(e, MSKG_ECAPACITY, "event log of replica %d overflowed", i);
  }
  return rc_all;
}

int mskg_run_ensemble(mskg_engine *const *engines, int32_t n, const int64_t *max_events, const double *max_time,
                      int64_t *events_done, double *kmc_time, int32_t *stop_reason) {
  if (!engines || n <= 0 || !max_events || !max_time) return MSKG_EINVAL;
  mskg_engine *e0 = engines[0];
  if (!e0) return MSKG_EINVAL;
  if (n > ENS_MAX) return fail_(e0, MSKG_EINVAL, "ensemble of %d replicas: at most %d", n, ENS_MAX);
  const bool la = e0->tab.la_mode || e0->tab.st_n;
  const bool cov = e0->cov_model;
  int cap = 0;
  int64_t queue_bound = 0;
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    if (!e) return fail_(e0, MSKG_EINVAL, "ensemble: replica %d is null", i);
    for (int j = 0; j < i; j++)
      if (engines[j] == e) return fail_(e0, MSKG_EINVAL, "ensemble: replica %d appears twice", i);
    if (e->device != e0->device) return fail_(e0, MSKG_EINVAL, "ensemble: replica %d lives on another device", i);
    if ((bool)(e->tab.la_mode || e->tab.st_n) != la || e->cov_model != cov)
      return fail_(e0, MSKG_EINVAL, "ensemble: replica %d needs another rate-model kernel than replica 0", i);
    cap = std::max(cap, e->cap);
    queue_bound += (int64_t)(e->ntx / 2) * (e->nty / 2) * ((e->ntz + 1) / 2);  // a colour's tiles at most
  }
  // a colour's queue head counts entries in units of 64 in 32 bits
  if (queue_bound > (1ll << 25)) return fail_(e0, MSKG_EINVAL, "ensemble: too many tiles per colour pass");
  std::vector<PassParams> reps(n);
  std::vector<unsigned long long> ev0(n);
  std::vector<int> slab(n);
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    RunState st;
    if (int rc = run_begin(e, max_events[i], max_time[i], st)) {
      if (e != e0) fail_(e0, rc, "ensemble replica %d: %s", i, e->err.c_str());
      return rc;
    }
    ev0[i] = st.events;
    reps[i] = pass_params(e);
  }
  for (int i = 0; i < n; i++) HIPCHK(engines[i], hipStreamSynchronize(engines[i]->stream));
  for (int i = 0; i < n; i++) slab[i] = run_touches(engines[i]);
  hipStream_t sm = e0->stream;
  PassParams *d_reps = nullptr;
  int *d_plan = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  const int64_t pw = ens_plan_words(n);
  const size_t shm = (size_t)cap * (4 + 4 + 1) + 16;
  int nrun = 0;
  int64_t sweeps = 0;
  float ms = 0;
  auto kpass = MSKG_VARIANT(k_pass_ens, la, cov);
  hipError_t ce = hipMalloc(&d_reps, n * sizeof(PassParams));
  if (ce == hipSuccess) ce = hipMalloc(&d_plan, pw * sizeof(int));
  if (ce == hipSuccess) ce = hipMemcpyAsync(d_reps, reps.data(), n * sizeof(PassParams), hipMemcpyHostToDevice, sm);
  int grid = 0;
  if (ce == hipSuccess) {
    // persistent waves: as many as the device holds at once
    int per_cu = 0, cus = 0;
    ce = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(kpass), WAVE, shm);
    if (ce == hipSuccess) ce = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, e0->device);
    grid = std::max(1, per_cu * cus);
  }
  if (ce == hipSuccess) {
    hipLaunchKernelGGL(k_ens_plan, dim3(1), dim3(ENS_MAX), 0, sm, d_reps, n, d_plan, 0, 1);
    ce = hipGetLastError();
  }
  // one sweep of every running replica: the eight colour passes, the tile
  // sums and sweep ends, the next sweep's plan
  if (ce == hipSuccess) ce = hipStreamBeginCapture(sm, hipStreamCaptureModeThreadLocal);
  if (ce == hipSuccess) {
    for (int c = 0; c < 8; c++) {
      if (c) hipLaunchKernelGGL(k_ens_plan, dim3(1), dim3(ENS_MAX), 0, sm, d_reps, n, d_plan, c, 0);
      hipLaunchKernelGGL(kpass, dim3(grid), dim3(WAVE), shm, sm, d_reps, n, d_plan, c);
    }
    hipLaunchKernelGGL(k_sweep_end_ens, dim3(n), dim3(END_THREADS), 0, sm, d_reps, n, d_plan);
    hipLaunchKernelGGL(k_ens_plan, dim3(1), dim3(ENS_MAX), 0, sm, d_reps, n, d_plan, 0, 1);
    ce = hipStreamEndCapture(sm, &graph);
  }
  if (ce == hipSuccess) ce = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  if (ce == hipSuccess) ce = hipEventRecord(e0->ev0, sm);
  int batch = 1;
  while (ce == hipSuccess) {
    for (int b = 0; b < batch && ce == hipSuccess; b++) ce = hipGraphLaunch(exec, sm);
    if (ce != hipSuccess) break;
    sweeps += batch;
    ce = hipMemcpyAsync(&nrun, d_plan + 8 * (n + 1) + 8, sizeof(int), hipMemcpyDeviceToHost, sm);
    if (ce == hipSuccess) ce = hipStreamSynchronize(sm);
    if (ce != hipSuccess || nrun == 0) break;
    // a sweep queued after every replica has stopped still costs its
    // launches: batches grow with the sweeps run, up to 32
    batch = (int)std::max<int64_t>(1, std::min<int64_t>(sweeps / 4, 32));
  }
  if (ce == hipSuccess) ce = hipEventRecord(e0->ev1, sm);
  // whatever happened, nothing queued may still use the plan or the
  // parameters when they are freed
  const hipError_t cs = hipStreamSynchronize(sm);
  if (ce == hipSuccess) ce = cs;
  if (ce == hipSuccess) ce = hipEventElapsedTime(&ms, e0->ev0, e0->ev1);
  if (exec) hipGraphExecDestroy(exec);
  if (graph) hipGraphDestroy(graph);
  hipFree(d_reps);
  hipFree(d_plan);
  if (ce != hipSuccess) return fail_(e0, MSKG_EDEVICE, "ensemble run: %s", hipGetErrorString(ce));
  int rc_all = MSKG_OK;
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    e->run_ms = ms;
    e->sweeps_done = sweeps;
    RunState st;
    if (int rc = read_state(e, st)) return rc;
    run_over(e, slab[i], st.ever_lo, st.ever_hi);
    if (events_done) events_done[i] = (int64_t)(st.events - ev0[i]);
    if (kmc_time) kmc_time[i] = st.clock;
    if (stop_reason) stop_reason[i] = st.stop == STOP_AT_LIMIT || !st.stop ? MSKG_STOP_LIMIT : st.stop;
    if (st.err && rc_all == MSKG_OK) {
      rc_all = fail_(e, MSKG_ESTATE, "run stopped in the tile at (%d,%d,%d): %s", st.err_site[0], st.err_site[1],
                     st.err_site[2], err_name(st.err));
      if (e != e0) fail_(e0, rc_all, "ensemble replica %d: %s", i, e->err.c_str());
    }
  }
  return rc_all;
}

int mskg_adjoint(mskg_engine *const *engines, int32_t n, const mskg_event *const *logs, const double *const *dts,
                 const int64_t *n_events, double *S, double *A, double *scalars) {
  return mskg_adjoint_checkpointed(engines, n, logs, dts, n_events, S, A, scalars, 0, nullptr);
}

int mskg_adjoint_checkpointed(mskg_engine *const *engines, int32_t n, const mskg_event *const *logs,
                              const double *const *dts, const int64_t *n_events, double *S, double *A, double *scalars,
                              int64_t every, int32_t *const *hist) {
  if (!engines || n <= 0 || !logs || !dts || !n_events || !S || !A || !scalars) return MSKG_EINVAL;
  if (every < 0 || (every > 0 && !hist) || (every == 0 && hist)) return fail_(engines[0], MSKG_EINVAL, "checkpoints: every %lld", (long long)every);
  mskg_engine *e0 = engines[0];
  if (!e0) return MSKG_EINVAL;
  // every replica's state is checked and its key arrays exist before anything is queued
  std::vector<char> fresh(n);
  std::vector<int64_t> rows(n);
  bool any_la = false, any_cov = false;
  int64_t most = 0;
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    if (!e || !e->loaded) return fail_(e0, MSKG_EINVAL, "adjoint: replica %d has no state loaded", i);
    for (int j = 0; j < i; j++)
      if (engines[j] == e) return fail_(e0, MSKG_EINVAL, "adjoint: replica %d appears twice", i);
    if (e->tab.ncov || e->tab.la_mode)
      return fail_(e, MSKG_EINVAL, "the likelihood covers models without coverage species and without LA rates");
    if (n_events[i] < 0 || (n_events[i] > 0 && (!logs[i] || !dts[i]))) return fail_(e, MSKG_EINVAL, "bad log");
    const int64_t np = e->box.npts;
    if (!e->d_key) {
      if (hipMalloc(&e->d_key, np * sizeof(int32_t)) != hipSuccess ||
          hipMalloc(&e->d_key_seen, np * sizeof(int32_t)) != hipSuccess ||
          hipMalloc(&e->d_rate_seen, np * sizeof(float)) != hipSuccess)
        return fail_(e, MSKG_ENOMEM, "adjoint: no device memory for the class keys");
    }
    any_la |= e->tab.la_mode || e->tab.st_n;
    any_cov |= e->cov_model;
    most = std::max(most, np);
    // the trajectory starts from the engine's rates: a tracked engine's keys
    // are current; otherwise a sweep refreshes the rates and assigns the keys
    fresh[i] = !(e->track && e->keys_valid);
    rows[i] = every > 0 ? n_events[i] / every : 0;
  }
  std::vector<RunHead> head;
  if (int rc = read_heads(engines, n, head)) return rc;  // also: nothing of their own streams is still running
  for (int i = 0; i < n; i++)
    if (head[i].err) return fail_(engines[i], MSKG_ESTATE, "engine is in an error state: %s", err_name(head[i].err));
  // One device block for every segment, in regions of one kind each so that
  // the results come back in one copy per kind: the logs and waiting times,
  // the initial class counts (+ the unsupported points) and isolated-rate
  // sums, S, A and the scalars in the caller's layouts, the checkpoints, the
  // check words, the descriptors, the replay's per-class integrals.
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  std::vector<size_t> log_off(n), dt_off(n), hist_off(n);
  size_t lb = 0, db = 0, hb = 0;
  for (int i = 0; i < n; i++) {
    const size_t ne = (size_t)std::max<int64_t>(1, n_events[i]);
    log_off[i] = lb; lb += up(ne * sizeof(mskg_event));
    dt_off[i] = db; db += up(ne * sizeof(double));
    hist_off[i] = hb; hb += (size_t)rows[i] * KEY_N * sizeof(int32_t);
  }
  const size_t cnt_b = up((size_t)n * (KEY_N + 1) * sizeof(int)), iso_b = up((size_t)n * sizeof(double)),
               s_b = up((size_t)n * ADJ_NS * sizeof(double)), a_b = up((size_t)n * KEY_N * sizeof(double)),
               sc_b = up((size_t)n * 4 * sizeof(double)), h_b = up(std::max<size_t>(hb, 1)),
               chk_b = up((size_t)n * 2 * sizeof(int)), d_b = up((size_t)n * sizeof(AdjDesc)),
               acc_b = up((size_t)n * 2 * KEY_N * sizeof(double));
  const size_t o_dt = lb, o_cnt = o_dt + db, o_iso = o_cnt + cnt_b, o_s = o_iso + iso_b, o_a = o_s + s_b,
               o_sc = o_a + a_b, o_h = o_sc + sc_b, o_chk = o_h + h_b, o_d = o_chk + chk_b, o_acc = o_d + d_b,
               total = o_acc + acc_b;
  char *arena = nullptr;
  if (hipMalloc(&arena, total) != hipSuccess) return fail_(e0, MSKG_ENOMEM, "adjoint: no device memory for the logs");
  int *const d_cnt = (int *)(arena + o_cnt);
  double *const d_iso = (double *)(arena + o_iso);
  int *const d_chk = (int *)(arena + o_chk);
  AdjDesc *const d_descs = (AdjDesc *)(arena + o_d);
  std::vector<AdjDesc> descs(n);
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    Lattice L = make_lattice(e);
    L.key = e->d_key;
    AdjDesc &D = descs[i];
    D.L = L;
    D.key_seen = e->d_key_seen;
    D.rate_seen = e->d_rate_seen;
    D.log = (const mskg_event *)(arena + log_off[i]);
    D.dt = (const double *)(arena + o_dt + dt_off[i]);
    D.n = n_events[i];
    D.cnt0 = d_cnt + (size_t)i * (KEY_N + 1);
    D.iso0 = d_iso + i;
    D.sweep_err = e->d_err;
    D.fresh = fresh[i];
    D.S = (double *)(arena + o_s) + (size_t)i * ADJ_NS;
    D.A = (double *)(arena + o_a) + (size_t)i * KEY_N;
    D.scal = (double *)(arena + o_sc) + (size_t)i * 4;
    D.st = e->d_st;
    D.hist = rows[i] > 0 ? (int32_t *)(arena + o_h + hist_off[i]) : nullptr;
    D.every = every > 0 ? every : 1;
    D.acc = (double *)(arena + o_acc) + (size_t)i * 2 * KEY_N;
  }
  hipStream_t sm = e0->stream;
  auto done = [&](int rc) {
    hipStreamSynchronize(sm);  // nothing queued may still use the block when it is freed
    hipFree(arena);
    return rc;
  };
  // the copies from host memory first, while the stream is still idle (a
  // copy from pageable memory returns only when done)
  hipError_t ce = hipMemcpyAsync(d_descs, descs.data(), n * sizeof(AdjDesc), hipMemcpyHostToDevice, sm);
  std::vector<HostPiece> logs_in;
  for (int i = 0; i < n; i++)
    if (n_events[i] > 0) logs_in.push_back({log_off[i], logs[i], (size_t)n_events[i] * sizeof(mskg_event)});
  for (int i = 0; i < n; i++)
    if (n_events[i] > 0) logs_in.push_back({o_dt + dt_off[i], dts[i], (size_t)n_events[i] * sizeof(double)});
  if (ce == hipSuccess) ce = stage_in(e0, sm, arena, logs_in);
  // each segment's initial classes
  if (ce == hipSuccess) {
    hipLaunchKernelGGL(k_adj_clear, dim3(n), dim3(64), 0, sm, d_descs, n);
    const int blocks = (int)std::min<int64_t>((most + 1023) / 1024, 256 * 16);
    for (int i0 = 0; i0 < n; i0 += 65535)
      hipLaunchKernelGGL(MSKG_VARIANT(k_adj_start, any_la, any_cov), dim3(blocks, std::min(n - i0, 65535)), dim3(256), 0,
                         sm, d_descs + i0);
    ce = hipGetLastError();
  }
  for (int i = 0; i < n; i++) {
    engines[i]->lists_dirty = true;
    engines[i]->slab = -1;
  }
  const int cblocks = (n + 255) / 256;
  std::vector<int> chk(2 * (size_t)n);
  if (ce == hipSuccess) {
    hipLaunchKernelGGL(k_adj_check, dim3(cblocks), dim3(256), 0, sm, d_descs, n, d_chk);
    ce = hipGetLastError();
  }
  if (ce == hipSuccess) ce = hipMemcpyAsync(chk.data(), d_chk, 2 * (size_t)n * sizeof(int), hipMemcpyDeviceToHost, sm);
  if (ce == hipSuccess) ce = hipStreamSynchronize(sm);
  if (ce != hipSuccess) return done(fail_(e0, MSKG_EDEVICE, "adjoint setup: %s", hipGetErrorString(ce)));
  for (int i = 0; i < n; i++) {
    if (chk[2 * i]) return done(fail_(engines[i], MSKG_ESTATE, "rate sweep: %s", err_name(chk[2 * i])));
    if (chk[2 * i + 1])
      return done(fail_(engines[i], MSKG_EINVAL, "%d points have rates the likelihood does not cover", chk[2 * i + 1]));
  }
  const size_t shm = (size_t)KEY_N * sizeof(int);
  ce = hipEventRecord(e0->ev0, sm);
  if (ce == hipSuccess) {
    hipLaunchKernelGGL(k_adjoint, dim3(n), dim3(WAVE), shm, sm, d_descs);
    ce = hipGetLastError();
  }
  if (ce == hipSuccess) ce = hipEventRecord(e0->ev1, sm);
  if (ce == hipSuccess) {
    hipLaunchKernelGGL(k_adj_errs, dim3(cblocks), dim3(256), 0, sm, d_descs, n, d_chk);
    ce = hipGetLastError();
  }
  // the results, one copy per kind (the checkpoints through a host buffer)
  std::vector<int32_t> hall(hb / sizeof(int32_t));
  if (ce == hipSuccess) ce = hipMemcpyAsync(S, arena + o_s, (size_t)n * ADJ_NS * sizeof(double), hipMemcpyDeviceToHost, sm);
  if (ce == hipSuccess) ce = hipMemcpyAsync(A, arena + o_a, (size_t)n * KEY_N * sizeof(double), hipMemcpyDeviceToHost, sm);
  if (ce == hipSuccess) ce = hipMemcpyAsync(scalars, arena + o_sc, (size_t)n * 4 * sizeof(double), hipMemcpyDeviceToHost, sm);
  if (ce == hipSuccess) ce = hipMemcpyAsync(chk.data(), d_chk, (size_t)n * sizeof(int), hipMemcpyDeviceToHost, sm);
  if (ce == hipSuccess && hb) ce = hipMemcpyAsync(hall.data(), arena + o_h, hb, hipMemcpyDeviceToHost, sm);
  if (ce == hipSuccess) ce = hipStreamSynchronize(sm);
  if (ce != hipSuccess) return done(fail_(e0, MSKG_EDEVICE, "k_adjoint: %s", hipGetErrorString(ce)));
  float ms = 0;
  hipEventElapsedTime(&ms, e0->ev0, e0->ev1);
  int rc_all = MSKG_OK;
  for (int i = 0; i < n; i++) {
    mskg_engine *e = engines[i];
    e->run_ms = ms;
    if (rows[i] > 0)
      memcpy(hist[i], hall.data() + hist_off[i] / sizeof(int32_t), (size_t)rows[i] * KEY_N * sizeof(int32_t));
    if (chk[i] && rc_all == MSKG_OK)
      rc_all = fail_(e, MSKG_ESTATE, "adjoint replay of replica %d stopped after %lld events: %s", i,
                     (long long)scalars[(size_t)i * 4 + 3], err_name(chk[i]));
  }
  return done(rc_all);
}

int mskg_frame(mskg_engine *e, int32_t *main_rec, int64_t cap_main, int32_t *void_rec, int64_t cap_void,
               int32_t *noepi_rec, int64_t cap_noepi, int64_t counts[5]) {
  if (!e || !e->loaded || !counts) return fail_(e, MSKG_EINVAL, "frame: no state loaded");
  int32_t *const hosts[3] = {main_rec, void_rec, noepi_rec};
  const int64_t caps[3] = {cap_main, cap_void, cap_noepi};
  return frame_lists<FRAME_MAIN>(e, 0, hosts, caps, counts);
}

int mskg_frame_device(mskg_engine *e, int32_t *main_rec, int64_t cap_main, int32_t *void_rec, int64_t cap_void,
                      int32_t *noepi_rec, int64_t cap_noepi, int64_t *counts) {
  if (!e || !e->loaded || !counts) return fail_(e, MSKG_EINVAL, "frame_device: no state loaded or no counts");
  if (cap_main < 0 || cap_void < 0 || cap_noepi < 0) return fail_(e, MSKG_EINVAL, "frame_device: negative capacity");
  const int64_t n = e->box.npts;
  if ((n + NOALLOC_FRAME_BLOCKS - 1) / NOALLOC_FRAME_BLOCKS > NOALLOC_MAX_CHUNK)
    return fail_(e, MSKG_EINVAL, "frame_device: %lld lattice points exceed the scratch's %d blocks of %lld points",
                 (long long)n, NOALLOC_FRAME_BLOCKS, (long long)NOALLOC_MAX_CHUNK);
  unsigned long long *sc = g_scratch[e->device];
  if (!sc) return fail_(e, MSKG_EDEVICE, "frame_device: the device's scratch is not set up");
  int z0, z1;
  touched_planes(e, z0, z1);
  const FramePlan F = frame_plan(e, z0, z1, 0, NOALLOC_FRAME_BLOCKS);
  const int nblk = (F.nseg + FRAME_THREADS / WAVE - 1) / (FRAME_THREADS / WAVE);
  unsigned long long *d_offs = sc;
  uint32_t *d_counts = (uint32_t *)(sc + (size_t)F.nseg * FrameShape<FRAME_MAIN>::NLIST);
  Lattice L = make_lattice(e);
  // no bits kept between the two passes: the write reads the records again
  hipLaunchKernelGGL(k_frame_count<FRAME_MAIN>, dim3(nblk), dim3(FRAME_THREADS), 0, e->stream, L, F, d_counts,
                     (unsigned long long *)nullptr);
  hipLaunchKernelGGL(k_frame_scan<FRAME_MAIN>, dim3(FrameShape<FRAME_MAIN>::NCNT), dim3(SCAN_THREADS), 0, e->stream,
                     d_counts, F.nseg, d_offs, counts);
  hipLaunchKernelGGL(k_frame_write<FRAME_MAIN>, dim3(nblk), dim3(FRAME_THREADS), 0, e->stream, L, F,
                     (const unsigned long long *)nullptr, d_offs, (int4 *)main_rec, (int4 *)void_rec,
                     (int4 *)noepi_rec, cap_main, cap_void, cap_noepi);
  hipError_t ce = hipGetLastError();
  if (ce == hipSuccess) ce = hipStreamSynchronize(e->stream);
  if (ce != hipSuccess) return fail_(e, MSKG_EDEVICE, "frame_device: %s", hipGetErrorString(ce));
  return MSKG_OK;
}

int mskg_frame_defects(mskg_engine *e, int32_t *vac_rec, int64_t cap_vac, int32_t *wrong_rec, int64_t cap_wrong,
                       int64_t counts[2]) {
  if (!e || !e->loaded || !counts) return fail_(e, MSKG_EINVAL, "frame: no state loaded");
  // the wrong-occupation analysis runs for two crystal species one of which is C
  const int sic = e->ncrystal == 2 &&
                  (e->cfg.list_crystal[0] == 6 || e->cfg.list_crystal[1] == 6 || e->cfg.list_crystal[2] == 6);
  std::vector<int4> flips;
  if (sic) {
    if (int rc = wrong_flips(e, flips)) return rc;
    if (int rc = set_wrong_marks(e, flips, 1)) return rc;
  }
  int32_t *const hosts[2] = {vac_rec, wrong_rec};
  const int64_t caps[2] = {cap_vac, cap_wrong};
  const int rc = frame_lists<FRAME_DEFECTS>(e, sic, hosts, caps, counts);
  if (sic) {
    const std::string msg = e->err;
    if (int rc2 = set_wrong_marks(e, flips, 0)) return rc2;  // the lattice is left as it was
    e->err = msg;
  }
  return rc;
}

}  // extern "C"
