// mskg_events.h -- per-site rate evaluation and event execution on the
// device-resident lattice.  Each routine follows the reference routine named
// in its comment (paths relative to the reference repository root) and keeps
// its update order, its absolute-coordinate comparisons and its rule for
// which sites get a fresh rate, so that a replayed event log reproduces the
// reference state bit for bit.
//
// The reference keeps three particle lists and a sum tree; here a site's
// neighbour list lives in its own record and its rate/class beside it, so
// AddMC/EraseMC/AddBulk/AddVoid become "set rate/class" or "clear rate".
#pragma once

#include "mskg_lattice.h"

namespace mskg {

enum : int {
  ERR_NONE = 0,
  ERR_COORD = 1,      // N_Si+N_C+N_B+N_wall != Coor (Get_Prob.f:293-298)
  ERR_GEOM = 2,       // a neighbour displacement that does not fit the record
  ERR_NOT_MC = 3,     // replayed event on a site that is not an MC particle
  ERR_COVERAGE = 4,   // coverage index not in ListCov
  ERR_CAPACITY = 5,   // tile candidate list overflow
  ERR_TEMPERATURE = 6, // zero temperature in LA mode
  ERR_TILE_LIST = 7,   // a tile's candidate list overflowed
  ERR_SUMS = 8,        // serial selection: the rate sums disagree with the lists
  ERR_LIQUID = 9,      // negative CountLiquid (laser-annealing build's form)
  ERR_ST_RANGE = 10,   // a temperature outside the interpolation tables (InitSt 'ST')
  ERR_SCHED = 11,      // a tile waited too long for its neighbour tiles (dependency-scheduled sweep)
  ERR_TOP = 12         // an event within 24 planes of the top of the stored planes (stored_len_z)
};

// Per-tile candidate lists (synchronous-sublattice mode): every MC particle
// of a tile is listed once (inlist[p] = 1) as its tile-local offset; entries
// whose class has dropped to 0 are removed when the tile is next processed.
struct Lattice {
  Site *site;
  float *rate;
  uint8_t *cls;
  uint8_t *inlist;        // may be null (no list maintenance)
  int32_t *tl_idx;        // [ntiles][capg] tile-local offsets
  int32_t *tl_n;          // [ntiles] entries used
  int32_t *tl_own;        // [ntiles] entries the tile itself wrote (the rest were appended by others)
  double *tile_r;         // [ntiles] FP64 rate total of the tile's list (isolated atoms excluded)
  int *list_err;          // set on overflow
  int *win;               // [8][4] per colour: tile-layer window lo, hi (read by that colour's
                          // pass), next lo, next hi (collected for the next sweep)
  Box box;
  const Geometry *geo;
  const Tables *tab;
  int tile, ntx, nty, capg;
  int cur_tile;           // the tile whose pass is running: its list lives on chip
  int cx, cy, cz;         // its lowest corner (when cur_tile >= 0)
  float inv_tile;         // 1 / tile
  int32_t *key;           // may be null: rate-class key of every point (likelihood accounting)
  const long long *cl;    // may be null: CountLiquid(1..3) the laser-annealing build's rates read
  const Lattice *cold;    // in a kernel that keeps lists: this lattice in constant memory, for
                          // the fields an event seldom needs (enlist); null: no lists to keep
  int ztop;               // highest z of an event's site: an event reads at most 12 and writes at
                          // most 6 planes from its site, so with only the bottom planes stored an
                          // event above this would reach past them (INT_MAX: every plane stored)
};

// Rate-class keys for the trajectory likelihood (models without coverage
// species).  A key names the table entry a point's rate comes from:
//   evaporation  (species-1) + 3*(n_Si+n_wall + 4*(n_C + 4*n_B)) + 192*n2
//                (n2 = occupied second-neighbour positions, 0 without that term)
//   adsorption site of coordination c       KEY_ADS + c - 1
//   placeholder deposition (1e-8)           KEY_PH
//   isolated atom (1e5*R, per point)        KEY_ISO
// and -1 for no rate.
enum : int { KEY_EVAP_N = 192 * 13, KEY_ADS = KEY_EVAP_N, KEY_PH = KEY_ADS + 3, KEY_ISO = KEY_PH + 1,
             KEY_N = KEY_ISO + 1, KEY_UNSUPPORTED = -2 };

struct P3 {
  int x, y, z;
  int64_t i;  // -1 outside the box
};

MSKG_HD P3 at(const Lattice &L, int x, int y, int z) {
  P3 p;
  p.x = x; p.y = y; p.z = z;
  p.i = pidx_checked(L.box, x, y, z);
  return p;
}
MSKG_HD P3 entry(const Lattice &L, const NL &l, int i) { return at(L, l.x[i], l.y[i], l.z[i]); }
MSKG_HD Site rd(const Lattice &L, int64_t i) {
  if (i < 0) {
    Site z;
    for (int a = 0; a < 4; a++) z.d[a][0] = z.d[a][1] = z.d[a][2] = 0;
    z.kc = 0; z.valid = 0; z.temp = 0;
    return z;
  }
  return L.site[i];
}
MSKG_HD NL list_of(const Lattice &L, const P3 &p, const Site &s) { return site_list(L.box, s, p.x, p.y, p.z); }

// x / tile for 0 <= x < 2^20: the FP32 quotient is off by at most one.
MSKG_HD int tdiv(const Lattice &L, int x) {
  int q = (int)((float)x * L.inv_tile);
  const int r = x - q * L.tile;
  if (r < 0) q--;
  else if (r >= L.tile) q++;
  return q;
}
MSKG_HD int tile_of(const Lattice &L, const P3 &p) {
  return (tdiv(L, p.z) * L.nty + tdiv(L, p.y)) * L.ntx + tdiv(L, p.x);
}
// A point's offset inside its tile, packed as (z << 14) | ((y / 2) << 7) |
// (x / 2) in tile-local coordinates (tile edge <= 254), so that decoding
// needs no division; offsets sort like the points' (z, y, x) order.
MSKG_HD int tile_pack(int zl, int yl, int xl) { return (zl << 14) | ((yl >> 1) << 7) | (xl >> 1); }
MSKG_HD int atomic_add_i32(int32_t *a, int v) {
#ifdef __HIP_DEVICE_COMPILE__
  return atomicAdd(a, v);
#else
  int o = *a;
  *a += v;
  return o;
#endif
}
MSKG_HD void atomic_min_i32(int *a, int v) {
#ifdef __HIP_DEVICE_COMPILE__
  atomicMin(a, v);
#else
  if (v < *a) *a = v;
#endif
}
MSKG_HD void atomic_max_i32(int *a, int v) {
#ifdef __HIP_DEVICE_COMPILE__
  atomicMax(a, v);
#else
  if (v > *a) *a = v;
#endif
}
MSKG_HD int tile_colour(int tx, int ty, int tz) { return (tx & 1) | ((ty & 1) << 1) | ((tz & 1) << 2); }
// A tile layer that holds candidates joins the window of layers its colour's
// pass visits.  A colour's window is only widened by passes of the other
// colours (same-colour tiles never touch each other), so it is constant
// while its own pass runs.
MSKG_HD void widen_window(int *win, int colour, int tz) {
  int *w = win + 4 * colour;
  // read first: the window rarely changes, and atomics on one word serialise
  if (tz < w[0]) atomic_min_i32(&w[0], tz);
  if (tz > w[1]) atomic_max_i32(&w[1], tz);
  if (tz < w[2]) atomic_min_i32(&w[2], tz);
  if (tz > w[3]) atomic_max_i32(&w[3], tz);
}
// A pointer to constant memory, read here: the compiler may not load what is
// behind it earlier and carry it in registers.  An event's loop has more
// values the same in every lane than scalar registers (it spilled about 80 of
// them to vector lanes and read them back on every event).
template <typename T>
__device__ inline const T *read_here(const T *p) {
  uint64_t v = (uint64_t)(uintptr_t)p;
  asm volatile("" : "+s"(v));
  const __attribute__((address_space(4))) T *c = (const __attribute__((address_space(4))) T *)(uintptr_t)v;
  return (const T *)c;
}
template <typename T>
__device__ inline T *as_global(T *p) {
  __attribute__((address_space(1))) T *g = (__attribute__((address_space(1))) T *)(uintptr_t)p;
  return (T *)g;
}
// A value that is the same in every lane, held in a scalar register from here
// on: the compiler may neither load it again nor carry in registers what
// could be computed from it before this point.
__device__ inline void pin(int &v) {
  v = __builtin_amdgcn_readfirstlane(v);
  asm volatile("" : "+s"(v));
}
__device__ inline void pin(uint32_t &v) {
  int i = (int)v;
  pin(i);
  v = (uint32_t)i;
}
__device__ inline void pin(int64_t &v) {
  int lo = (int)(uint32_t)v, hi = (int)(v >> 32);
  pin(lo);
  pin(hi);
  v = (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
template <typename T>
__device__ inline void pin(T *&p) {
  int64_t v = (int64_t)(uintptr_t)p;
  pin(v);
  p = as_global((T *)(uintptr_t)v);
}
__device__ inline void pin(Box &b) {
  pin(b.lx); pin(b.ly); pin(b.lz); pin(b.hx); pin(b.hy); pin(b.plane);
}
// A site that becomes an MC particle joins its tile's list (once).
__device__ inline void enlist(const Lattice &L, const P3 &p) {
  if (!L.cold) return;
  // the running tile keeps its list on chip and flags it on write-back
  if (L.cur_tile >= 0 && (unsigned)(p.x - L.cx) < (unsigned)L.tile && (unsigned)(p.y - L.cy) < (unsigned)L.tile &&
      (unsigned)(p.z - L.cz) < (unsigned)L.tile)
    return;
  const Lattice &C = *read_here(L.cold);
  uint8_t *const inlist = as_global(C.inlist);
  if (inlist[p.i]) return;
  inlist[p.i] = 1;
  const int tx = tdiv(C, p.x), ty = tdiv(C, p.y), tz = tdiv(C, p.z);
  const int t = (tz * C.nty + ty) * C.ntx + tx;
  widen_window(as_global(C.win), tile_colour(tx, ty, tz), tz);
  const int slot = atomic_add_i32(as_global(C.tl_n) + t, 1);
  if (slot < C.capg)
    as_global(C.tl_idx)[(int64_t)t * C.capg + slot] = tile_pack(p.z - tz * C.tile, p.y - ty * C.tile, p.x - tx * C.tile);
  else *as_global(C.list_err) = ERR_TILE_LIST;
}

// ---- rates ---------------------------------------------------------------
// The reference's kb (Get_Prob.f:70).
#define MSKG_KB 0.00008617330350
// Where a rate evaluation takes the tables from: all of them in device
// memory (the sweep), or an event wave's copy in LDS.
struct TabSrc {
  const Tables &t;
  MSKG_HD double pe(int i) const { return t.pe[i]; }
  MSKG_HD double pd(int i) const { return t.pd[i]; }
  MSKG_HD double pabs(int i) const { return t.pabs[i]; }
  MSKG_HD double pdes(int i) const { return t.pdes[i]; }
  MSKG_HD double f2(int i) const { return t.f2[i]; }
  // the Boltzmann factor of laser-annealing deposition entry i (species i % 3)
  // at the species' melting temperature
  MSKG_HD double ex(int i, bool variant) const {
    return exp(-t.pd[i] / (MSKG_KB * (variant ? t.la_tm[i % 3] : t.tm)));
  }
  MSKG_HD double ads(int coor) const {
    return t.pd[3 * (coor - 1)] + t.pd[1 + 3 * (coor - 1)] + t.pd[2 + 3 * (coor - 1)] +
           (t.pabs[3 * coor] + t.pabs[1 + 3 * coor] + t.pabs[2 + 3 * coor]);
  }
};
// The tables an event reads, 2 KB of LDS a wave: a lookup is the last of an
// event's chain of dependent reads, and from memory it cost a round trip of
// its own.  PTransE's entries without covered neighbours are the first 192
// of the full table; with coverage species the full table stays in memory.
constexpr int PE_PLAIN = 192;
struct TabLds {
  double pe[PE_PLAIN], pd[9], pabs[12], pdes[12], f2[13];
  double ads[4];  // an adsorption site's rate by coordination (without laser annealing): PTransD + PTransAbs
  double ex[10];  // laser annealing: TabSrc::ex, nine exponentials a wave instead of three a rate
};
// A tile's list lies behind the tables and is read 16 bytes at a time (with
// 8 bytes less here the passes took 1-2% longer: CVD 96.3 against 94.1 ms).
static_assert(sizeof(TabLds) % 16 == 0, "the list behind the tables is read 16 bytes at a time");
template <bool COV>
struct TabEv {
  const Tables &t;
  const TabLds &l;
  MSKG_HD double pe(int i) const { return COV ? t.pe[i] : l.pe[i]; }
  MSKG_HD double pd(int i) const { return l.pd[i]; }
  MSKG_HD double pabs(int i) const { return l.pabs[i]; }
  MSKG_HD double pdes(int i) const { return l.pdes[i]; }
  MSKG_HD double f2(int i) const { return l.f2[i]; }
  MSKG_HD double ads(int coor) const { return l.ads[coor]; }
  MSKG_HD double ex(int i, bool) const { return l.ex[i]; }  // laser-annealing kernels only
};
// The copy in two halves, so that its loads can leave with a tile's first ones.
struct TabRegs {
  double pe[PE_PLAIN / 64], rest, ads, ex;
};
template <bool LA>
__device__ inline void fetch_tables(const Tables &t, TabRegs &r, int lane) {
  for (int k = 0; k < PE_PLAIN / 64; k++) r.pe[k] = t.pe[lane + 64 * k];
  // pd (9), pabs (12), pdes (12), f2 (13): a lane each
  const double *src = lane < 9 ? t.pd + lane : (lane < 21 ? t.pabs + (lane - 9) : (lane < 33 ? t.pdes + (lane - 21)
                                                                                              : t.f2 + min(lane - 33, 12)));
  r.rest = *src;
  const int c = min(max(lane, 1), 3);
  r.ads = TabSrc{t}.ads(c);
  if (LA) r.ex = t.la_mode ? TabSrc{t}.ex(min(lane, 8), t.la_variant != 0) : 0.0;
}
template <bool LA>
__device__ inline void put_tables(const TabRegs &r, TabLds &l, int lane) {
  for (int k = 0; k < PE_PLAIN / 64; k++) l.pe[lane + 64 * k] = r.pe[k];
  if (lane < 9) l.pd[lane] = r.rest;
  else if (lane < 21) l.pabs[lane - 9] = r.rest;
  else if (lane < 33) l.pdes[lane - 21] = r.rest;
  else if (lane < 46) l.f2[lane - 33] = r.rest;
  if (lane < 4) l.ads[lane] = r.ads;
  if (LA && lane < 9) l.ex[lane] = r.ex;
}
template <bool LA>
__device__ inline void load_tables(const Tables &t, TabLds &l, int lane) {
  TabRegs r;
  fetch_tables<LA>(t, r, lane);
  put_tables<LA>(r, l, lane);
}
// The deposition rates of the three species at a site of coordination coor.
// LA = false compiles the laser-annealing branches out (tables with la_mode 0).
template <bool LA, class Src>
MSKG_HD void pd_of(const Src &S, int coor, int temperature, const long long *cl, double p[3]) {
  const Tables &t = S.t;
  double e[3];
  for (int k = 0; k < 3; k++) p[k] = e[k] = S.pd(k + 3 * (coor - 1));
  if (!LA || !t.la_mode) return;
  if (t.la_variant && cl) {
    // LaserAnnealing Get_Prob.f:148-151, evaluated left to right: 0.5d0 *
    // P0(k) * FLOAT(CountLiquid(k)) / SUM(CountLiquid) * EXP(..) * (1 + ERF(..)),
    // FLOAT the REAL(4) conversion.  With no liquid left (the reference
    // divides by zero) solidification stops.
    const long long sum = cl[0] + cl[1] + cl[2];
    for (int k = 0; k < 3; k++)
      p[k] = sum <= 0 || k >= t.ncrystal ? 0.0  // PD(k,:) is set for k <= NCrystal only
                                         : 0.5 * t.la_p0[k] * (double)(float)(int)cl[k] / (double)sum *
                                               S.ex(k + 3 * (coor - 1), true) *
                                               (1.0 + erf((temperature - t.la_tflex[k]) / t.la_sigma[k])) *
                                               (e[k] != 0.0 ? 1.0 : 0.0);
    return;
  }
  const double step = 1.0 + erf((temperature - t.tflex) / t.sigma);
  for (int k = 0; k < 3; k++)
    p[k] = 0.5 * t.p0 * S.ex(k + 3 * (coor - 1), false) * step * (e[k] != 0.0 ? 1.0 : 0.0);
}
MSKG_HD int pe_flat(int sp, int a, int b, int c, int d, int e, int f) {
  return (sp - 1) + 3 * (a + 4 * (b + 4 * (c + 4 * (d + 4 * (e + 4 * f)))));
}
template <bool LA, class Src>
MSKG_HD double pe_of(const Src &S, int sp, int idx, int temperature) {
  const Tables &t = S.t;
  double v = S.pe(idx);
  if (!LA || !t.la_mode) return v;
  const double p0 = t.la_variant ? t.la_p0[sp - 1] : t.p0;  // LaserAnnealing Get_Prob.f:144-146
  return p0 * exp(-v / (MSKG_KB * temperature)) * (v != 0.0 ? 1.0 : 0.0);
}
// The laser-annealing build's SiGe rule (its main.f:676-681): a deposition of
// a species whose liquid is used up (CountCrystal >= InitCountCrystal, i.e.
// CountLiquid <= 0) deposits the other species.
template <bool LA = true>
MSKG_HD int la_swap(const Lattice &L, int itrans) {
  if (LA && L.cl && L.tab->la_mode && L.tab->la_variant && L.tab->la_swap && (itrans == 1 || itrans == 2) &&
      L.cl[itrans - 1] <= 0)
    return itrans % 2 + 1;
  return itrans;
}

// InterpProbFromField.f:28-54: the tables at temperature T are reference
// table iu when T equals its temperature (the first such), else the blend
// of tables il = iu - 1 and iu, iu the first of the smallest positive
// (reference temperature - T), with integer weights wl = |T_iu - T| on il
// and wu = |T_il - T| on iu.  False when T lies outside the references (the
// reference indexes out of its arrays there).
struct STW {
  int il, iu, wl, wu, exact;
};
MSKG_HD bool st_weights(const Tables &t, int temperature, STW &w) {
  int best = -1;
  w.exact = 0;
  for (int k = 0; k < t.st_n; k++) {
    const int diff = t.st_temp[k] - temperature;
    if (diff == 0) {
      w.exact = 1;
      w.il = w.iu = k;
      w.wl = w.wu = 0;
      return true;
    }
    if (diff > 0 && (best < 0 || diff < t.st_temp[best] - temperature)) best = k;
  }
  if (best <= 0) return false;
  w.iu = best;
  w.il = best - 1;
  const int dl = t.st_temp[w.iu] - temperature, du = t.st_temp[w.il] - temperature;
  w.wl = dl < 0 ? -dl : dl;
  w.wu = du < 0 ? -du : du;
  return true;
}
// One interpolated table entry: (wl * ref(il) + wu * ref(iu)) / (wl + wu),
// the integer weights converted as Fortran does.
MSKG_HD double st_entry(const double *ref, int stride, int idx, const STW &w) {
  if (w.exact) return ref[(int64_t)w.iu * stride + idx];
  return ((double)w.wl * ref[(int64_t)w.il * stride + idx] + (double)w.wu * ref[(int64_t)w.iu * stride + idx]) /
         (double)(w.wl + w.wu);
}
// What a rate depends on besides the point's own record, packed so that the
// lanes looking at a point's neighbours add up in one word: reciprocal
// neighbours of species 1..3 (bits 0, 4, 8), walls (12), reciprocal covered
// neighbours by slot (16, 20, 24), occupied second-neighbour positions (28).
MSKG_HD uint32_t neighbour_count(int kq, bool lists) {
  // kinds 1..3, wall and covered 5..7 count at bit 4 (kind - 1)
  return kq != KIND_EMPTY && (lists || kq == KIND_WALL) ? 1u << ((4 * kq - 4) & 31) : 0u;
}

// Get_Prob, Get_Prob.f:54-331, evaluated for a point at height z of this
// kind, temperature and coordination (Evaporation.f:121 evaluates with a
// stale list copy: the counts are those of the list the caller went by).
// c0: the coordination of its first listed neighbour (read for an empty point
// of coordination 1); cnt: neighbour_count summed over its list (read for an
// atom).  rtot is the total rate R used by the isolated-atom rule.  No random
// number is drawn: the deposition species / absorbed coverage is drawn when
// the event executes (class CLS_ADSORB).
// COV = false compiles the coverage-species branches out (tables without
// coverage species and without absorption or desorption rates).
template <bool LA, bool COV, class Src>
MSKG_HD void rate_of(const Src &S, const long long *cl, double rtot, int z, int kind, int temp, int coor, int c0,
                     uint32_t cnt, int &cls, double &rate, int &err, int &key) {
  const Tables &t = S.t;
  key = -1;
  cls = CLS_NONE;
  rate = 0.0;
  int temperature = 0;
  STW w;
  const bool st = LA && t.st_n > 0;  // Get_Prob.f:77-90: tables at the site's temperature
  if (LA && (t.la_mode || st)) {
    temperature = temp;
    if (temperature == 0) { err = ERR_TEMPERATURE; return; }
    if (st && !st_weights(t, temperature, w)) { err = ERR_ST_RANGE; return; }
  }
  if (!COV && kind >= KIND_COV0) { err = ERR_COVERAGE; return; }
  const int slot = COV ? kind_cov_slot(kind) : 0;
  if (slot) {  // desorption, :93-123
    if (slot > t.ncov) { err = ERR_COVERAGE; return; }
    if (coor <= 3) {
      cls = CLS_DESORB;
      rate = st ? st_entry(t.st_pdes, 12, (slot - 1) + 3 * coor, w) : S.pdes((slot - 1) + 3 * coor);
      key = KEY_UNSUPPORTED;
    }
    return;
  }
  if (kind == KIND_EMPTY) {  // :155-214
    if (LA && t.la_mode && t.la_variant && cl && (cl[0] < 0 || cl[1] < 0 || cl[2] < 0)) {
      // a negative solidification rate, which a sum tree cannot hold (the
      // reference's selection goes wrong there, or UpdateTree.f:37-41 stops
      // on a rate that cancels to zero): the engine stops with an error
      err = ERR_LIQUID;
      return;
    }
    if (coor >= 1 && coor <= 3) {
      if (coor > 1 || c0 >= 2) {
        double pdep = 0.0, pabs = 0.0;
        if (!LA) {
          pdep = S.ads(coor);
        } else if (st) {
          pdep = st_entry(t.st_pd, 9, 3 * (coor - 1), w) + st_entry(t.st_pd, 9, 1 + 3 * (coor - 1), w) +
                 st_entry(t.st_pd, 9, 2 + 3 * (coor - 1), w);
          pabs = COV ? st_entry(t.st_pabs, 12, 3 * coor, w) + st_entry(t.st_pabs, 12, 1 + 3 * coor, w) +
                           st_entry(t.st_pabs, 12, 2 + 3 * coor, w)
                     : 0.0;
        } else {
          double p[3];
          pd_of<LA>(S, coor, temperature, cl, p);
          pdep = p[0] + p[1] + p[2];
          pabs = COV ? S.pabs(0 + 3 * coor) + S.pabs(1 + 3 * coor) + S.pabs(2 + 3 * coor) : 0.0;
        }
        cls = CLS_ADSORB;
        rate = pdep + pabs;
        key = (t.ncov || st) ? KEY_UNSUPPORTED : KEY_ADS + coor - 1;
      } else {
        cls = CLS_PLACEHOLDER;
        rate = (double)1.e-8f;  // REAL(4) literal, Get_Prob.f:183
        key = KEY_PH;
      }
    }
    return;  // Coor 0 leaves the reference's outputs unassigned; Coor 4 is a vacancy
  }
  // evaporation, :215-324
  if (z < t.frozen_below_z) return;  // frozen substrate (engine option, no reference counterpart)
  const int n_si = cnt & 15, n_c = (cnt >> 4) & 15, n_b = (cnt >> 8) & 15, n_wall = (cnt >> 12) & 15;
  const int tot = n_si + n_c + n_b + n_wall;
  if (tot != coor) { err = ERR_COORD; return; }
  if (tot > 3) return;
  if (tot == 0) {
    cls = CLS_ISOLATED;
    rate = (double)100000.0f * rtot;
    key = KEY_ISO;
    return;
  }
  const int c1 = COV ? (cnt >> 16) & 15 : 0, c2 = COV ? (cnt >> 20) & 15 : 0, c3 = COV ? (cnt >> 24) & 15 : 0;
  const int idx = pe_flat(kind, n_si + n_wall, n_c, n_b, c1, c2, c3);
  cls = CLS_EVAP;
  rate = st ? st_entry(t.st_pe, 3 * 4096, idx, w) : pe_of<LA>(S, kind, idx, temperature);
  const int n2 = t.use_f2 ? (int)(cnt >> 28) : 0;
  if (t.use_f2) rate *= S.f2(n2);
  key = (t.ncov || t.la_mode || st) ? KEY_UNSUPPORTED : (kind - 1) + 3 * (n_si + n_wall + 4 * (n_c + 4 * n_b)) + 192 * n2;
}

// The 12 second-neighbour positions of a diamond super-lattice site (the
// fcc shell: (+-6,+-6,0) and permutations), for the optional
// second-neighbour energy term; no reference counterpart.
MSKG_HD void second_vec(int k, int &dx, int &dy, int &dz) {
  const int a = (k & 2) ? -6 : 6, b = (k & 1) ? -6 : 6, g = k >> 2;
  dx = g == 2 ? 0 : a;
  dy = g == 0 ? b : (g == 1 ? 0 : a);
  dz = g == 0 ? 0 : b;
}
MSKG_HD uint32_t shell_disp(int k) {
  int dx, dy, dz;
  second_vec(k, dx, dy, dz);
  return (uint32_t)(dx & 255) | ((uint32_t)(dy & 255) << 8) | ((uint32_t)(dz & 255) << 16);
}
// p shifted by a small vector, with one x/y wrap.
MSKG_HD P3 shifted(const Lattice &L, const P3 &p, int dx, int dy, int dz) {
  int x = p.x + dx, y = p.y + dy;
  if (x >= L.box.lx) x -= L.box.lx;
  if (x < 0) x += L.box.lx;
  if (y >= L.box.ly) y -= L.box.ly;
  if (y < 0) y += L.box.ly;
  return at(L, x, y, p.z + dz);
}

// Where a stochastic choice of the reference comes from: the log (replay)
// or the engine's RNG.
struct Choice {
  int arm;       // 0/1 forced arm-chair choice, -1 draw
  double u_arm;  // uniform used when the arm/zig coordination sums tie
};

// The reference event an MC particle of class `cls`, whose record is ss,
// executes.  For an adsorption site this draws the species / coverage as
// Get_Prob.f:160-176 and IndexEvent_Abs (Get_Prob.f:22-52) do, with the draw
// taken at execution instead of at rate-update time (same distribution: the
// class is refreshed whenever the coordination changes).  Returns itrans in
// the reference's numbering (1..3 deposit, 4 evaporate, 5 desorb, 6.. absorb).
template <bool LA, bool COV, class Src>
MSKG_HD int pick_itrans(const Lattice &L, const Src &S, int coor, int temp, int cls, double u) {
  const Tables &t = S.t;
  if (cls == CLS_PLACEHOLDER) return 1;
  if (cls == CLS_EVAP || cls == CLS_ISOLATED) return 4;
  if (cls == CLS_DESORB) return 5;
  int temperature = (LA && t.la_mode) ? temp : 0;
  STW w;
  // InitSt 'ST': the tables at the site's temperature (its rate was evaluated
  // with them, so the temperature lies inside the references)
  const bool st = LA && t.st_n > 0 && st_weights(t, temp, w);
  auto pabs_of = [&](int i) { return st ? st_entry(t.st_pabs, 12, i + 3 * coor, w) : S.pabs(i + 3 * coor); };
  double p1, p2, p3;
  if (st) {
    p1 = st_entry(t.st_pd, 9, 3 * (coor - 1), w);
    p2 = st_entry(t.st_pd, 9, 1 + 3 * (coor - 1), w);
    p3 = st_entry(t.st_pd, 9, 2 + 3 * (coor - 1), w);
  } else {
    double p[3];
    pd_of<LA>(S, coor, temperature, L.cl, p);
    p1 = p[0];
    p2 = p[1];
    p3 = p[2];
  }
  double pdep = p1 + p2 + p3;
  double pabs = COV ? pabs_of(0) + pabs_of(1) + pabs_of(2) : 0.0;
  double pcurr = u * (pdep + pabs);
  if (!COV || pcurr <= pdep) {
    if (pcurr <= p1) return 1;
    if (pcurr > p1 + p2) return 3;
    return 2;
  }
  if (t.ncov == 1) return 6;
  int r = 6;
  double lo = pdep;
  for (int i = 1; i <= t.ncov; i++) {
    double hi = lo + pabs_of(i - 1);
    if (pcurr > lo && pcurr <= hi) r = 5 + i;
    lo = hi;
  }
  return r;
}

// ---- event execution -------------------------------------------------------
// One 64-wide wave executes an event, every lane in step: sixteen quads of
// four lanes, each quad one point the event looks at, each lane of a quad one
// entry of that point's neighbour list.
//   quads 0..3    the site's four listed neighbours
//   quads 4..15   with the second-neighbour term, the site's second shell
// The event is then three dependent gathers (the site's record, the sixteen
// points' records, their 64 listed neighbours' records) whatever its type,
// and one rate evaluation for all of the points and the site itself.
//
// What bounds it: a wave issues one instruction every four cycles or more and
// waits for each gather, and the waves of a pass are few and uneven, so the
// length of one wave's instruction stream is the time of an event.  With a
// lane a point (each lane walking its point's four neighbours and twelve
// second neighbours in turn, 13 lanes busy) an event was about 3400
// instructions; counts are now sums over a quad by DPP, and nothing passes
// through LDS.  Passes before and after: 8e6 events at 512^3 SiC 92 -> 42 ms,
// 5e5 events of SiC on 480^3 132 -> 56 ms, 2e5 of CVD on 240x240x760
// 252 -> 116 ms, k_serial on 64 lattices of 144^3 55.6 -> 25 ms.
//
// The reference visits the neighbours one after the other, but each
// neighbour's update writes only that neighbour's record and reads only
// records the other neighbour updates do not write (two neighbours of a
// site are never neighbours of each other), so the concurrent updates give
// the sequential result.  When two list entries resolve to the same point
// the neighbours are visited in order, a round each.  The site's own record
// is written last, and before each round that has another after it; lanes
// whose gather meets the site take it from registers.

// A site record as it lies in memory (struct Site), in four words.
typedef uint32_t Rec __attribute__((ext_vector_type(4)));
__device__ inline Rec make_rec(uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
  Rec r = {x, y, z, w};
  return r;
}
__device__ inline int r_kind(const Rec &r) { return r.w & 7; }
__device__ inline int r_coor(const Rec &r) { return (r.w >> 3) & 7; }
__device__ inline int r_temp(const Rec &r) { return r.w >> 16; }
__device__ inline uint32_t w_kind(uint32_t w, int k) { return (w & ~7u) | (uint32_t)k; }
__device__ inline uint32_t w_coor(uint32_t w, int c) { return (w & ~0x38u) | (((uint32_t)c & 7u) << 3); }
__device__ inline Rec load_rec(const Lattice &L, int64_t i) { return *(const Rec *)(L.site + i); }
__device__ inline void store_rec(const Lattice &L, int64_t i, const Rec &r) { *(Rec *)(L.site + i) = r; }
// Entry j's displacement, its three bytes in one word, and whether it is one.
__device__ inline uint32_t rec_disp(const Rec &r, int j) {
  const uint32_t lo = j < 2 ? r.x : (j == 2 ? r.y : r.z), hi = j < 2 ? r.y : r.z;
  return __builtin_amdgcn_alignbyte(hi, lo, (4 - j) & 3) & 0xffffffu;
}
// The same for an entry known when compiled (scalar shifts for a record in scalar registers).
template <int J>
__device__ inline uint32_t rec_disp_at(const Rec &r) {
  const uint32_t lo = J < 2 ? r.x : (J == 2 ? r.y : r.z), hi = J < 2 ? r.y : r.z;
  const int sh = J == 0 ? 0 : (J == 1 ? 24 : (J == 2 ? 16 : 8));
  return (uint32_t)((((uint64_t)hi << 32) | lo) >> sh) & 0xffffffu;
}
__device__ inline bool rec_has(const Rec &r, int j) { return (r.w >> (8 + j)) & 1; }
// The position of a displacement from p (the absolute point (0,0,0) when it is none).
__device__ inline P3 disp_point(const Lattice &L, const P3 &p, uint32_t d, bool has) {
  int x = p.x + (int)(int8_t)d, y = p.y + (int)(int8_t)(d >> 8);
  const int z = p.z + (int)(int8_t)(d >> 16);
  if (x >= L.box.lx) x -= L.box.lx;
  if (x < 0) x += L.box.lx;
  if (y >= L.box.ly) y -= L.box.ly;
  if (y < 0) y += L.box.ly;
  return at(L, has ? x : 0, has ? y : 0, has ? z : 0);
}
__device__ inline P3 rec_entry(const Lattice &L, const Rec &r, const P3 &p, int j) {
  return disp_point(L, p, rec_disp(r, j), rec_has(r, j));
}
// set_list for one entry: position o as a displacement from p (the point
// (0,0,0) is no displacement); ok: it fits the record.
__device__ inline uint32_t pack_disp(const Box &b, const P3 &p, const P3 &o, bool &has, bool &ok) {
  has = (o.x | o.y | o.z) != 0;
  ok = true;
  if (!has) return 0u;
  int dx = o.x - p.x, dy = o.y - p.y, dz = o.z - p.z;
  if (dx > b.lx / 2) dx -= b.lx;
  if (dx < -b.lx / 2) dx += b.lx;
  if (dy > b.ly / 2) dy -= b.ly;
  if (dy < -b.ly / 2) dy += b.ly;
  ok = (unsigned)(dx + 128) < 256u && (unsigned)(dy + 128) < 256u && (unsigned)(dz + 128) < 256u;
  return (uint32_t)(dx & 255) | ((uint32_t)(dy & 255) << 8) | ((uint32_t)(dz & 255) << 16);
}
// The displacement back: minus each byte.
__device__ inline uint32_t disp_back(uint32_t d) {
  return ((0x808080u - (d & 0x7f7f7fu)) ^ (~d & 0x808080u)) & 0xffffffu;
}
// Does the record list the point at displacement w from it, which is not the
// origin?  An entry that is no displacement holds zero, which w, of another
// point, is not; it stands for the origin, which rec_lists looks for.
__device__ inline bool rec_lists_disp(const Rec &r, uint32_t w) {
  const uint32_t a = rec_disp_at<0>(r) ^ w, b = rec_disp_at<1>(r) ^ w, c = rec_disp_at<2>(r) ^ w,
                 d = rec_disp_at<3>(r) ^ w;
  return min(min(a, b), min(c, d)) == 0u;
}
// Does the record r of point q list position p?  The reference's Recipr loops
// (q's list contains p) on the stored displacements: a valid entry holds p - q
// wrapped as set_list wraps it, an entry that is no displacement stands for the
// origin.  For a displacement that may not fit the record or a p that may be
// the origin; rec_lists_disp does for the others.
__device__ inline bool rec_lists(const Box &b, const P3 &q, const Rec &r, const P3 &p) {
  bool has, ok;
  const uint32_t w = pack_disp(b, q, p, has, ok);
  return has ? ok && rec_lists_disp(r, w) : ((r.w >> 8) & 15u) != 15u;
}

// Get_Prob of point p by one thread, from its record: the sweep.  Few of a
// sweep's points are MC particles, so what counts here is that the branch
// holds few registers: the neighbours are taken two at a time, the second
// shell four.
template <bool LA, bool COV>
__device__ inline void get_prob(const Lattice &L, double rtot, const P3 &p, const Rec &r, int &cls, double &rate,
                                int &err, int &key) {
  const Tables &t = *L.tab;
  const int kind = r_kind(r), coor = r_coor(r);
  int c0 = 0;
  uint32_t cnt = 0;
  if (kind == KIND_EMPTY) {
    if (coor == 1) {
      const int64_t i0 = rec_entry(L, r, p, 0).i;
      c0 = i0 < 0 ? 0 : (L.site[i0].kc >> 3) & 7;
    }
  } else if (kind_species(kind) && p.z >= t.frozen_below_z) {
    const bool origin = p.i == 0;
#pragma unroll 2
    for (int i = 0; i < 4; i++) {
      const P3 q = rec_entry(L, r, p, i);
      Rec sq = make_rec(0u, 0u, 0u, 0u);
      if (q.i >= 0) sq = load_rec(L, q.i);
      const int kq = r_kind(sq);
      const bool lists = kq != KIND_EMPTY && kq != KIND_WALL &&
                         (rec_has(r, i) && !origin ? rec_lists_disp(sq, disp_back(rec_disp(r, i)))
                                                   : rec_lists(L.box, q, sq, p));
      if (COV && lists && kind_cov_slot(kq) > t.ncov) err = ERR_COVERAGE;
      cnt += neighbour_count(kq, lists);
    }
    if (t.use_f2) {
#pragma unroll 1
      for (int g = 0; g < 3; g++)
        for (int k = 0; k < 4; k++) {
          int dx, dy, dz;
          second_vec(4 * g + k, dx, dy, dz);
          const int64_t i2 = shifted(L, p, dx, dy, dz).i;
          const int kq = i2 < 0 ? 0 : L.site[i2].kc & 7;
          cnt += kind_species(kq) ? 1u << 28 : 0u;
        }
    }
    if (COV && err) { cls = CLS_NONE; rate = 0.0; key = -1; return; }
  }
  rate_of<LA, COV>(TabSrc{t}, L.cl, rtot, p.z, kind, r_temp(r), coor, c0, cnt, cls, rate, err, key);
}

// A value of lane J of the quad; sums and ORs over the quad.  Every lane of
// the wave must be active.
template <int J>
__device__ inline int quad_take(int v) {
  return __builtin_amdgcn_update_dpp(0, v, J * 0x55, 0xf, 0xf, false);
}
__device__ inline uint32_t quad_sum(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, false);  // lanes 1 0 3 2
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, false);  // lanes 2 3 0 1
  return v;
}
__device__ inline uint32_t quad_or(uint32_t v) {
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, false);
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, false);
  return v;
}
// The record of a quad's four entries (e, has: this lane's).
__device__ inline void quad_list(Rec &r, uint32_t e, bool has, int j) {
  const uint32_t e0 = quad_take<0>((int)e), e1 = quad_take<1>((int)e), e2 = quad_take<2>((int)e),
                 e3 = quad_take<3>((int)e);
  r.x = e0 | (e1 << 24);
  r.y = (e1 >> 8) | (e2 << 16);
  r.z = (e2 >> 16) | (e3 << 8);
  r.w = (r.w & ~0xff00u) | (quad_or(has ? 1u << j : 0u) << 8);
}
__device__ inline Rec uniform_rec(const Rec &r) {
  return make_rec((uint32_t)__builtin_amdgcn_readfirstlane((int)r.x), (uint32_t)__builtin_amdgcn_readfirstlane((int)r.y),
                    (uint32_t)__builtin_amdgcn_readfirstlane((int)r.z), (uint32_t)__builtin_amdgcn_readfirstlane((int)r.w));
}

// What an event leaves in the wave's registers: the points whose rate may
// have changed, on lane 0 the site, on lane 4 i + 1 neighbour i, on lane
// 17 + 4 k second-shell point k -- in lane order, the order the lists take
// new particles in.
struct EvOut {
  P3 p;        // this lane's point
  float rate;  // its new rate and class as stored, when set is 1
  int cls;
  int set;     // 0: no point here, or one that got no new rate; 2: read both from memory
               // (a list with repeated entries, whose points take several rates in turn)
  // the same in every lane
  int arm;      // stacking choice made (-1 none)
  int err;
  int species;  // deposited or evaporated species (1..3), desorbed coverage slot (1..3), 0 otherwise
};

// The stacking of a deposition at coordination 1 (deposition.f:40-74,
// FIND_SN + IF_Arm_Choice): lanes 0..2 the arm-chair and lanes 4..6 the
// zig-zag candidates; S takes the chosen list.
__device__ inline void ev_stacking(const Lattice &L, const P3 &s, Rec &S, const Choice &ch, EvOut &o, int lane) {
  const int j = lane & 3;
  const P3 c = rec_entry(L, S, s, 0);
  Rec cr = make_rec(0u, 0u, 0u, 0u);
  if (c.i >= 0) cr = load_rec(L, c.i);
  // the back bonds' ends: the first three entries of c's list that are not s
  const P3 le = rec_entry(L, cr, c, j);
  const unsigned m0 = (unsigned)__ballot(!(le.x == s.x && le.y == s.y && le.z == s.z)) & 15u;
  const unsigned m1 = m0 & (m0 - 1u), m2 = m1 & (m1 - 1u);
  const int src = __ffs((int)(j == 0 ? m0 : (j == 1 ? m1 : m2))) - 1;
  int sn[3] = {__shfl(le.x, src & 3, 64), __shfl(le.y, src & 3, 64), __shfl(le.z, src & 3, 64)};
  if (src < 0) sn[0] = sn[1] = sn[2] = 0;
  const int site[3] = {s.x, s.y, s.z}, cc[3] = {c.x, c.y, c.z};
  int cand[3];
  find_sn_one(*L.geo, L.box.lx, L.box.ly, site, cc, sn, (lane & 4) != 0, cand);
  const P3 cp = at(L, cand[0], cand[1], cand[2]);
  int cco = 0;
  if (lane < 8 && j < 3 && cp.i >= 0) cco = r_coor(load_rec(L, cp.i));
  const int csum = (int)quad_sum((uint32_t)cco);
  const int carm = __builtin_amdgcn_readlane(csum, 0), czig = __builtin_amdgcn_readlane(csum, 4);
  int is_arm = 1;  // IF_Arm_Choice.f:35-54
  if (ch.arm >= 0) is_arm = ch.arm;
  else if (czig > carm) is_arm = 0;
  else if (czig == carm) is_arm = (ch.u_arm <= L.tab->ptrans_zig) ? 0 : 1;
  is_arm = __builtin_amdgcn_readfirstlane(is_arm);
  o.arm = is_arm;
  const int from = (is_arm ? 0 : 4) + (j > 0 ? j - 1 : 0);
  P3 e;
  e.x = __shfl(cand[0], from, 64);
  e.y = __shfl(cand[1], from, 64);
  e.z = __shfl(cand[2], from, 64);
  if (j == 0) { e.x = c.x; e.y = c.y; e.z = c.z; }
  bool has, ok;
  const uint32_t d = pack_disp(L.box, s, e, has, ok);
  if (__ballot(!ok)) o.err = ERR_GEOM;
  quad_list(S, d, has, j);
  S = uniform_rec(S);
}

// Execute one event of type itrans at site s, whose record is S.  Called by
// every lane of the wave with the same arguments.
template <bool LA, bool COV>
__device__ inline void execute(const Lattice &L, const TabLds &tabs, double rtot, const P3 &s_in, Rec S, int itrans,
                               const Choice &ch, EvOut &o, const int lane) {
  const TabEv<COV> T{*L.tab, tabs};
  const Tables &t = T.t;
  const P3 s = s_in;
  const bool f2 = t.use_f2 != 0, s_origin = (s.x | s.y | s.z) == 0;
  const int frozen = t.frozen_below_z;
  const int grp = lane >> 2, j = lane & 3;
  o.p = s;
  o.rate = 0.0f;
  o.cls = CLS_NONE;
  o.set = 0;
  o.arm = -1;
  o.err = ERR_NONE;
  o.species = 0;
  if (s.z > L.ztop) {  // before anything changes: the run stops with the state as it was
    o.err = ERR_TOP;
    return;
  }
  if (!COV && itrans > 4) {
    o.err = ERR_COVERAGE;
    return;
  }
  const bool dep = itrans <= 3, evap = itrans == 4, absorb = itrans >= 6;
  const int old_kind = r_kind(S), coor_old = r_coor(S);
  // the site: deposition.f:24-74, Evaporation.f:25-35, absorption.f:25-78 and
  // desorption.f:25-117 (at coordination 1 desorption visits only the first neighbour)
  const int new_kind = dep ? itrans : (evap || itrans == 5 ? KIND_EMPTY : KIND_COV0 + itrans - 6);
  S.w = w_kind(S.w, new_kind);
  o.species = dep ? itrans : (evap && kind_species(old_kind) ? old_kind : 0);
  if (COV && itrans == 5) o.species = kind_cov_slot(old_kind);  // the coverage desorbed
  if (dep && coor_old == 1) {
    ev_stacking(L, s, S, ch, o, lane);
    if (o.err) return;
  }
  const int nvisit = COV && itrans == 5 && coor_old == 1 ? 1 : 4;
  // the quads' points, as displacements from the site; an entry that is no
  // displacement is the origin
  uint32_t pd = rec_disp(S, grp & 3);
  bool phas = rec_has(S, grp & 3);
  if (grp >= 4) {
    pd = shell_disp(grp - 4);
    phas = true;
  }
  const P3 p = disp_point(L, s, pd, phas);
  // the site's displacement from its point
  uint32_t to_s = disp_back(pd);
  if (((S.w >> 8) & 15u) != 15u && !phas) {
    bool has, ok;
    to_s = pack_disp(L.box, p, s, has, ok);
    if (!has || !ok) to_s = 1u << 24;  // no entry is the site
  }
  // repeated list entries (no displacement: zero), or a zero one, which may be
  // the site itself: an atom deposited on an unfixed site whose one neighbour is
  // the origin, with no list there, takes the site for its zig-zag candidates,
  // and the origin lists itself with an entry that is no displacement
  const uint32_t s0 = rec_disp_at<0>(S), s1 = rec_disp_at<1>(S), s2 = rec_disp_at<2>(S), s3 = rec_disp_at<3>(S);
  const bool twice = nvisit == 4 && ((s0 == s1) | (s0 == s2) | (s0 == s3) | (s1 == s2) | (s1 == s3) | (s2 == s3) |
                                     (min(min(s0, s1), min(s2, s3)) == 0u));
  // absorption and desorption change no neighbour's record: visits of one
  // point give it one rate, in whatever order (a covered site of coordination
  // 1 lists the origin three times)
  const bool seq = twice && (dep || evap);
  const bool shell = f2 && (dep || evap);
  Rec S_in = S;
  // The rounds: all quads at once; with repeated entries a round for each
  // neighbour and a last one for the second shell; with coverage species and
  // a second shell the neighbours first, since a covered neighbour's new list
  // counts for the shell.  Each round reads what the one before wrote.
  const int lead = seq ? nvisit : (COV && shell ? 1 : 0);  // rounds before the last
  int coor = coor_old;
  P3 nbuff;  // Evaporation.f's NBuff, carried over the neighbours
  nbuff.x = nbuff.y = nbuff.z = 0;
  nbuff.i = 0;
#pragma unroll 1
  for (int round = 0; round <= lead; round++) {
    const bool last = round == lead;
    // nearly always the only round: nothing of it is to be computed ahead of
    // the loop for branches that are seldom taken (about 240 instructions)
    P3 s = s_in;
    Rec S = S_in;
    pin(s.x); pin(s.y); pin(s.z); pin(s.i);
    {
      uint32_t a = S.x, b = S.y, c = S.z, d = S.w;
      pin(a); pin(b); pin(c); pin(d);
      S = make_rec(a, b, c, d);
    }
    if (!last) {
      if (lane == 0) store_rec(L, s.i, S);
      __threadfence_block();
    }
    const unsigned nbm = (1u << nvisit) - 1u;
    const unsigned M = (seq ? (last ? 0u : 1u << round) : (round == 0 ? nbm : 0u)) | (last && shell ? 0xfff0u : 0u);
    const bool act = (M >> grp) & 1u;
    const bool nb = act && grp < 4;
    Rec r = make_rec(0u, 0u, 0u, 0u);
    if ((act || (last && lead && grp < 4)) && p.i >= 0) r = load_rec(L, p.i);
    const int kind = r_kind(r), coornn = r_coor(r);
    const bool wall = kind == KIND_WALL, atom = kind_species(kind), empty = !atom && !wall;  // empty or covered
    // this lane's entry of its point's list
    uint32_t e = rec_disp(r, j);
    bool ehas = rec_has(r, j);
    P3 q = disp_point(L, p, e, ehas);
    // the list holds the site (the site at the origin: an entry that is no displacement)
    const bool back = quad_or((ehas ? e == to_s : s_origin) ? 1u : 0u) != 0u;
    // what happens to the point
    bool need = act & (grp >= 4) & atom & (coornn >= 1) & (coornn <= 3);  // a second-shell atom: a fresh rate
    bool first = false, second = false, erase = false, unfix = false, bad = false;
    int inc = 0, cn = coornn;
    if (dep) {  // deposition.f:78-235
      const bool more = nb & back & ((atom & (coornn <= 3)) | (empty & ((coornn & 6) == 2)));
      first = nb & empty & (coornn == 0);
      inc = ((nb & wall) | (more & atom & (coor_old == 1) & (grp >= 1))) ? 1 : 0;
      cn = coornn + ((more | first) ? 1 : 0);
      need |= more | first;
      if (__ballot(nb & empty & (coornn == 1))) {
        // a second fixed neighbour: the two others follow when the first is
        // a second neighbour of the site (FIND_NN.f, a lane each)
        const int ax = quad_take<0>(q.x), ay = quad_take<0>(q.y), az = quad_take<0>(q.z);
        int dx = ax - s.x, dy = ay - s.y;
        const int dz = az - s.z;
        dx = dx < 0 ? -dx : dx;
        dx = dx < L.box.lx - dx ? dx : L.box.lx - dx;
        dy = dy < 0 ? -dy : dy;
        dy = dy < L.box.ly - dy ? dy : L.box.ly - dy;
        second = nb && empty && coornn == 1 && dx * dx + dy * dy + dz * dz == 72;
        if (second) {
          cn = 2;
          need = true;
          if (j == 1) q = s;
          if (j >= 2) {
            const int a1[3] = {ax, ay, az}, a2[3] = {s.x, s.y, s.z}, pc[3] = {p.x, p.y, p.z};
            int ns[3];
            find_nn_one(*L.geo, L.box.lx, L.box.ly, a1, a2, pc, j - 2, ns);
            q = at(L, ns[0], ns[1], ns[2]);
          }
          bool ok;
          e = pack_disp(L.box, p, q, ehas, ok);
          bad = !ok;
        }
      }
      if (first) {  // its list starts with the site
        ehas = j == 0 && !s_origin;
        e = ehas ? to_s & 0xffffffu : 0u;
        bad = to_s >> 24 && !s_origin;
        q = s;
      }
    } else if (evap) {  // Evaporation.f:36-208
      const bool hit = nb & back & (atom | (empty & (coornn >= 1) & (coornn <= 4)));
      inc = (nb & wall) ? -1 : 0;
      erase = hit & empty & (coornn == 1);  // EraseMC + LattCoo=0, keeping the temperature bits
      need |= hit & !erase;
      unfix = hit & empty & (coornn == 2);  // the list keeps the reciprocal partner (NBuff)
      cn = coornn - ((hit & !erase) ? 1 : 0);  // coordination 4 -> 3 is EraseBulk/EraseVoid + AddMC
    } else if (COV) {  // an atom bonded back to the site (absorption.f:45-60, desorption.f:45-105)
      need |= nb & atom & (!absorb | (coornn <= 3)) & back;
    }
    // the listed neighbours' records (the rate of an unfixed point comes from
    // its old list, Evaporation.f:121)
    const bool count = need & atom & (p.z >= frozen);
    const bool look = count | unfix | (second & (j >= 2)) | (need & empty & (cn == 1) & (j == 0));
    Rec er = make_rec(0u, 0u, 0u, 0u);
    uint32_t k2 = 0;
    if (look && q.i >= 0) er = load_rec(L, q.i);
    if (f2 && count) {
      // four second neighbours a lane in three steps; at least 6 units from
      // every face they are at fixed index steps
      const int a = (j & 2) ? -6 : 6, b = (j & 1) ? -6 : 6;
      const Box &B = L.box;
      int64_t i0, i1, i2;
      if (shell_inside(B, p.x, p.y, p.z)) {
        i0 = p.i + (a / 2 + (b / 2) * B.hx);
        i1 = p.i + (b * B.plane + a / 2);
        i2 = p.i + (b * B.plane + (a / 2) * B.hx);
      } else {
        i0 = shifted(L, p, a, b, 0).i;
        i1 = shifted(L, p, a, 0, b).i;
        i2 = shifted(L, p, 0, a, b).i;
      }
      // every lane loads all three (outside the box: point 0, not used): a load
      // under a condition of its own is waited for before the next leaves
      const int r0 = L.site[i0 < 0 ? 0 : i0].kc, r1 = L.site[i1 < 0 ? 0 : i1].kc, r2 = L.site[i2 < 0 ? 0 : i2].kc;
      const int k0 = i0 == s.i ? new_kind : (i0 < 0 ? 0 : r0 & 7);
      const int k1 = i1 == s.i ? new_kind : (i1 < 0 ? 0 : r1 & 7);
      const int kk = i2 == s.i ? new_kind : (i2 < 0 ? 0 : r2 & 7);
      k2 = ((uint32_t)kind_species(k0) + (uint32_t)kind_species(k1) + (uint32_t)kind_species(kk)) << 28;
    }
    if (q.i == s.i) er = S;
    const int kq = r_kind(er);
    bool lists = rec_lists_disp(er, disp_back(e));
    // ... for a neighbour or a point at the origin by the form its position has in a list
    const bool origin = !ehas | (p.i == 0);
    if (__ballot(look & origin & (kq != KIND_EMPTY)) && look && origin) lists = rec_lists(L.box, q, er, p);
    lists &= look & (kq != KIND_EMPTY) & (kq != KIND_WALL);
    int err = ERR_NONE;
    if (COV) {
      if (quad_or((count & lists & (kind_cov_slot(kq) > t.ncov)) ? 1u : 0u)) err = ERR_COVERAGE;
    }
    uint32_t cnt = quad_sum((count ? neighbour_count(kq, lists) : 0u) + k2);
    const bool partner = lists & kind_species(kq) & (r_coor(er) <= 3);
    const unsigned pm = quad_or(partner ? 1u << j : 0u);  // reciprocal partners by entry
    const int c0 = quad_take<0>(r_coor(er));
    if (second) cn += __popc(pm >> 2);
    // the point's new record
    Rec nr = r;
    nr.w = w_coor(r.w, cn);
    if (erase) nr = make_rec(0u, 0u, 0u, r.w & 0xffff0000u);
    if (__ballot(first | second)) {
      Rec lr = nr;
      bad = quad_or(bad ? 1u : 0u) != 0u;
      quad_list(lr, e, ehas, j);
      if (first | second) {
        if (bad) {
          err = ERR_GEOM;
          need = false;
          nr = r;
        } else {
          nr = lr;
        }
      }
    }
    const unsigned um = (unsigned)((__ballot(unfix) >> 1) & 0x1111ull);  // unfixed neighbours, bit 4 i
    if (um) {
      const int jb = pm ? 31 - __clz((int)pm) : 0;  // the last partner
      const uint32_t pe = rec_disp(r, jb);
      if (unfix) {  // one entry; none for no partner, or a partner at the origin
        const bool keep = pm != 0u && rec_has(r, jb);
        nr.x = keep ? pe : 0u;
        nr.y = nr.z = 0u;
        nr.w = (nr.w & ~0xff00u) | (keep ? 0x100u : 0u);
      }
      // NBuff over the neighbours in order: one that found no partner gets
      // the last one found before it (or the initial (0,0,0): none).  Every
      // neighbour with a partner needs only the last such.
      const unsigned fm = um & (unsigned)(__ballot(pm != 0u) >> 1);
      const P3 pp = disp_point(L, p, pe, rec_has(r, jb));
      for (int i = fm == um ? (31 - __clz((int)um)) >> 2 : 0; i < 4; i++) {
        if (!((um >> (4 * i)) & 1u)) continue;
        if ((fm >> (4 * i)) & 1u) {
          nbuff.x = __builtin_amdgcn_readlane(pp.x, 4 * i + 1);
          nbuff.y = __builtin_amdgcn_readlane(pp.y, 4 * i + 1);
          nbuff.z = __builtin_amdgcn_readlane(pp.z, 4 * i + 1);
        } else if (nbuff.x | nbuff.y | nbuff.z) {
          bool has, ok;
          const uint32_t d = pack_disp(L.box, p, nbuff, has, ok);
          if (grp == i) {
            if (!ok) err = ERR_GEOM;
            else { nr.x = d; nr.w |= 0x100u; }
          }
        }
      }
    }
    coor += __popcll(__ballot(inc > 0 && j == 1)) - __popcll(__ballot(inc < 0 && j == 1));
    bool put = nb && (dep || evap) && (need || erase) && j == 1;  // this lane stores its point's record
    bool set = (need || erase) && j == 1;
    // what the rate evaluation below takes: the quad's point, or on lane 0
    // the site with its final coordination and neighbours
    int ek = kind, ecoor = cn, ec0 = c0, et = r_temp(r), ez = p.z;
    bool eval = need;
    int64_t wi = p.i;
    if (last) {
      const bool sn = lane < 16 && j == 1;  // a lane a neighbour
      const int fk = r_kind(nr), fc = r_coor(nr);
      const bool rem = evap && coor == 0;  // EraseMC zeroes the record
      uint32_t scnt = 0;
      if (dep || (evap && coor == 1)) {
        bool sl = s_origin ? ((nr.w >> 8) & 15u) != 15u : rec_lists_disp(nr, to_s);
        sl &= sn & (fk != KIND_EMPTY) & (fk != KIND_WALL);
        if (dep) {
          const uint32_t c1 = sn ? neighbour_count(fk, sl) : 0u;
          if (COV && __ballot(sl && kind_cov_slot(fk) > t.ncov)) { if (lane == 0) err = ERR_COVERAGE; }
          scnt = (uint32_t)(__builtin_amdgcn_readlane((int)c1, 1) + __builtin_amdgcn_readlane((int)c1, 5) +
                            __builtin_amdgcn_readlane((int)c1, 9) + __builtin_amdgcn_readlane((int)c1, 13));
          if (f2) scnt += (uint32_t)__popcll(__ballot(lane >= 16 && j == 1 && atom)) << 28;
        } else {  // the site keeps one reciprocal bond (NBuff)
          const unsigned long long sp = __ballot(sl && kind_species(fk) && fc <= 3);
          if (sp) {
            const int l = 63 - __clzll((long long)sp);
            nbuff.x = __builtin_amdgcn_readlane(p.x, l);
            nbuff.y = __builtin_amdgcn_readlane(p.y, l);
            nbuff.z = __builtin_amdgcn_readlane(p.z, l);
          }
        }
      }
      const uint32_t old_w = S.w;
      if (!dep || coor != coor_old) S.w = w_coor(S.w, coor);  // deposition.f:236 writes a changed one only
      if (rem) S = make_rec(0u, 0u, 0u, S.w & 0xffff0000u);
      const int sc0 = __builtin_amdgcn_readlane(fc, 1);
      if (lane == 0) {
        ek = new_kind;
        ecoor = coor;
        ec0 = sc0;
        cnt = scnt;
        et = old_w >> 16;
        ez = s.z;
        eval = !rem && !err;
        set = true;
        put = true;
        wi = s.i;
      }
      if (evap && coor == 1) {
        bool has, ok;
        const uint32_t d = pack_disp(L.box, s, nbuff, has, ok);
        if (ok) S = make_rec(d, 0u, 0u, (S.w & ~0xff00u) | (has ? 0x100u : 0u));
        else if (lane == 0) err = ERR_GEOM;
      }
      if (lane == 0) nr = S;
    }
    int cls = CLS_NONE, key = -1;
    double rate = 0.0;
    if (eval && !err) rate_of<LA, COV>(T, L.cl, rtot, ez, ek, et, ecoor, ec0, cnt, cls, rate, err, key);
    if (first && !cls && lane != 0) {  // AddMC stores the list with the rate only (lane 0 holds the site)
      nr.x = r.x;
      nr.y = r.y;
      nr.z = r.z;
      nr.w = (nr.w & ~0xff00u) | (r.w & 0xff00u);
    }
    if (put && wi >= 0) store_rec(L, wi, nr);
    const unsigned long long em = __ballot(err != ERR_NONE);
    if (em) o.err = __builtin_amdgcn_readlane(err, 63 - __clzll((long long)em));
    if (set && wi >= 0) {
      const float rf = cls ? (float)rate : 0.0f;
      L.rate[wi] = rf;
      L.cls[wi] = (uint8_t)cls;
      if (L.key) L.key[wi] = cls ? key : -1;
      const P3 sp = lane == 0 ? s : p;
      if (cls) enlist(L, sp);
      o.p = sp;
      o.rate = rf;
      o.cls = cls;
      o.set = twice && lane != 0 && grp < 4 ? 2 : 1;
    }
    if (!last) {  // the next round reads this one's records, the site's too where it lists itself
      __threadfence_block();
      S_in = uniform_rec(load_rec(L, s.i));
    }
  }
}

}  // namespace mskg
