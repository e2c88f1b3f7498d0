// dev_common.h -- types, layout helpers and host-side declarations shared by
// the HIP translation units of libsrs_amd (device.hip: the step kernels and the
// context; linescan.hip: the line-scan operator; adjoint.hip: recording,
// replayed segments and the adjoint).  Not part of the ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cstddef>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <numeric>
#include <thread>
#include <vector>

#include "kinetics.h"
#include "philox.h"
#include "srs_internal.h"

#pragma clang fp contract(off)

namespace srs_dev {

constexpr int MAX_TILE = 512;  // largest k_sweep workgroup (elements per workgroup)
constexpr int GATE_THREADS = 256;
constexpr int MAX_RYR = 1024;  // the reference GPU path launches <<<1, N_RyR>>>
constexpr int MAX_LCC = 1024;
constexpr int NXCD = 8;        // MI355X: 8 XCDs, workgroups dispatched round-robin

enum : uint8_t { F_JSR = 1, F_TROPC = 2, F_SL = 4, F_BR = 8, F_CHAN = 16 };
// What holds for every element of a 64-element block (the elements of one
// wavefront of a sweep), read with one scalar load per wavefront.
enum : uint32_t {
  BLK_PLAIN = 1,  // every element is plain cytosol with troponin (F_TROPC and nothing else)
};

// State layout of one realization (6*np doubles): the four diffusing species
// of QB elements form a block of two halves, QB pairs (Ca, ATP) and then QB
// pairs (CaM, Fluo); then the TnC and CSQ planes, which are never gathered.
//  QB = 64: each of a wavefront's 16-byte loads and stores of consecutive
//    elements covers 1 KB without gaps.  With the four species side by side
//    every access covered half of each cache line it touched: a plain copy in
//    that form ran at 5.7 TB/s against 6.3, and the write requests to L2 were
//    72 per wavefront instead of 40 (48-member ensemble: 175.7 -> 171.8 us per
//    step; with non-temporal stores, which that form had made slower, 154 us).
//  QB = 1: an element's four species side by side (32 B), for element orders
//    whose neighbours lie scattered.  A neighbour with no other of the tile's
//    near it costs one cache line here and two there (quad_block_for).
template <int QB>
struct Quads {
  __host__ __device__ static constexpr uint32_t half() { return QB; }  // pairs from an element's first to its second
  // element e's first pair (pairs of 2^31 elements still count in 32 bits)
  __host__ __device__ static uint32_t at(uint32_t e) { return e + (e & ~(uint32_t)(QB - 1)); }
  // offsets of its Ca and its Fluo in doubles
  __host__ __device__ static size_t ca(uint32_t e) { return 2 * (size_t)at(e); }
  __host__ __device__ static size_t fluo(uint32_t e) { return ca(e) + 2 * QB + 1; }
};
// The same for a layout that is known at run time only (RealDesc::qb).
struct QuadsOf {
  uint32_t qb;
  __host__ __device__ uint32_t half() const { return qb; }
  __host__ __device__ uint32_t at(uint32_t e) const { return e + (e & ~(qb - 1)); }
  __host__ __device__ size_t ca(uint32_t e) const { return 2 * (size_t)at(e); }
  __host__ __device__ size_t fluo(uint32_t e) const { return ca(e) + 2 * qb + 1; }
};
__host__ __device__ inline size_t xoff(QuadsOf lay, int s, size_t e, size_t np) {
  if (s == srs::TRPN) return 4 * np + e;
  if (s == srs::CSQN) return 5 * np + e;
  const size_t q = lay.ca((uint32_t)e), f = lay.fluo((uint32_t)e);
  return s == srs::CA ? q : s == srs::ATP ? q + 1 : s == srs::CMDN ? f - 1 : f;
}
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));

// One channel of an element that carries channel flux, in the reference's order.
struct ChanEntry {
  int32_t code;      // >=0: 2*ryr + side (0 cleft, 1 jSR); <0: -(lcc+1)
  int32_t jsr, cyt;  // a RyR's two elements
  int32_t sl;        // bit 0: jsr has F_SL, bit 1: cyt has
};
// Everything about a channel-flux element that is fixed, in one record, for
// the workgroup that gates and then updates these elements (sweep_gated).
struct ChanElem {
  double a[5], v0, tt;
  int32_t j, nb[4], e0, e1;  // the element, its neighbours, its run of centry
  uint32_t f;
  ChanEntry first;  // centry[e0]
};

// Immutable per-realization descriptor (read with scalar loads).
struct RealDesc {
  const uint32_t* nbr;    // [np][4] neighbour indices (IDX_SL)
  // tile map of the sweep (TileMap): where each element's neighbours are among
  // its tile's staged quads
  const uint16_t* loc;    // [np][4]
  const uint32_t* hal;    // halo elements (IDX_SL), tile by tile
  const int32_t* hoff;    // [tiles + 1] the tiles' runs in hal
  int32_t qcap;           // quads a tile stages at most
  int32_t qb;             // the state layout's block (Quads)
  const double* coef;     // [5][np] (plain rows)
  const uint32_t* row;    // class rows: [np][3] words, the row's class and five deltas (int16 each)
  const double* tab;      // class rows: [n_class][5] class values
  const uint32_t* blk;    // [np / 64] flags of each 64-element block (BLK_*)
  int32_t n_class;
  const uint8_t* flags;   // [np]
  const double* V0;       // [np]
  const double* tt;       // [np]
  const double* br;       // [4][np] Ca, Fluo, ATP, CaM boundary rates at this realization's D, or null
  const double* br_mesh;  // [4][np] the mesh's boundary rates, built with the D in brd
  double brd[4];          // the D_Ca, D_Fluo, D_ATP, D_CaM the mesh's boundary rates were built with
  double* X[2];           // [6][np] ping-pong state
  int32_t n, np;
  int32_t n_ryr, n_lcc;
  const int32_t* ryr_ele;
  const int32_t* ryr_jsr;
  const int32_t* ryr_nb;
  int32_t* ryr_state;
  const int32_t* lcc_ele;
  int32_t* lcc_state;
  int32_t* lccv_state;
  double* R;
  int32_t n_celem;
  const int32_t* celem;   // sorted element indices that carry channel flux
  const int32_t* cstart;  // [n_celem+1]
  const ChanEntry* centry;
  const ChanElem* crec;   // [n_celem] what an element of celem is updated from
  int32_t* sched;         // replay or recorded schedule [n_sched][n_ryr] or null
  int64_t n_sched;
  int64_t rec_step0;      // the step that row 0 of a recorded schedule is before
  float* rec;
  int32_t rec_cap, rec_len, ryr_out, gpu_layout;
  uint64_t key, stream;
  // model extensions (srs_extensions): Ca diffusion with D_CAJSR in jSR
  // elements, SR-site rapid buffer (b_sr uM, dissociation constant k_sr uM)
  int32_t jsr_diff;
  double b_sr, k_sr;
  double P[SRS_N_REAL];
  int32_t I[SRS_N_INT];
};

// A boundary rate at a realization's current D.  The mesh's planes hold
// D_b Face_C b / V0 summed over an element's bound faces
// (cpu/InitFuncs.cpp:1019-1024), with D_b the coefficient they were built
// with (brd); the rate is linear in D, so a realization whose D has since been
// changed (srs_params_set) gets planes of its own scaled by D / D_b, and one
// whose D is unchanged uses the mesh's bits as they are.
__host__ __device__ inline double br_scaled(double v, double D, double D_b) {
  return (D == D_b || D_b == 0.0) ? v : v / D_b * D;
}
// The D-free part Face_C b / V0 of a boundary rate (its derivative in D).
__host__ __device__ inline double br_unit(double v, double D_b) { return D_b == 0.0 ? 0.0 : v / D_b; }

// Mutable per-realization loop state.
struct RealLive {
  double t, dt_last, vm, ca_nsr, t_lcc_close, ca_max_last;
  // CaNSR-dependent SERCA subexpressions of cpu/RunSimulation.cpp:85-88, the
  // same for every element: 0.104217 + 17.923 K_sr, 1.75583e6 + K_sr 7.61673e6,
  // 6.08463e11 + K_sr 4.50544e11, 9.17846e6 - 11478.2 K_sr, 0.329904 K_sr
  double serca[5];
  int64_t step;
  int64_t sched_base;
  int32_t done, lcc_open, n_open_last, cur, rec_count, rec_overflow;
  int32_t ffwd;  // gating-only phase of flag_ffwd: the sweep skips this realization
};

enum : uint32_t {
  G_AFTER_SWEEP = 1,  // new state is X[1-cur]; flip cur afterwards
  G_PROTOCOL = 2,     // run the loop body for the next time
  G_NO_GATING = 4,    // skip gating regardless of the parameter flag
  G_REPLAY = 8,       // load RyR states for the next step from the schedule
  G_RECORD = 16,      // write RyR states for the next step to the schedule
};

__device__ __forceinline__ int xcd_tile(int bid, int grid) {
  // Consecutive tiles of a realization land on one XCD, so neighbour gathers
  // that cross a tile boundary hit that XCD's L2.
  return (bid % NXCD) * (grid / NXCD) + bid / NXCD;
}

// Sum of v over the 64 lanes of a wavefront, left in lane 63, by DPP lane
// moves (no LDS traffic): sums within quads, then within each row of 16
// lanes (row_shr 4 and 8 leave the row's sum in its lane 15), then row 0
// into row 1 and rows 0-1 into rows 2-3 by row broadcasts.  Every lane must
// be active.  A fixed order, so the result is deterministic.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
  return __hiloint2double(hi, lo);
}
// The first four steps alone: each row's sum in its lane 15.
__device__ __forceinline__ double row_sum_dpp(double v) {
  v += dpp_f64<0xb1, 0xf>(v);   // quad_perm [1,0,3,2]
  v += dpp_f64<0x4e, 0xf>(v);   // quad_perm [2,3,0,1]
  v += dpp_f64<0x114, 0xf>(v);  // row_shr:4
  v += dpp_f64<0x118, 0xf>(v);  // row_shr:8
  return v;
}
__device__ __forceinline__ double wave_sum_dpp(double v) {
  v = row_sum_dpp(v);
  v += dpp_f64<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_f64<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Pointers read from the descriptor are generic; casting them to the global
// address space lets the compiler use global (not flat) memory instructions.
#define SRS_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ const SRS_GLOBAL T* gp(const T* p) { return (const SRS_GLOBAL T*)p; }
template <class T>
__device__ __forceinline__ SRS_GLOBAL T* gpw(T* p) { return (SRS_GLOBAL T*)p; }

template <bool NT, class T>
__device__ __forceinline__ void stg(SRS_GLOBAL T* p, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// The diffusing species (Ca, ATP, CaM, Fluo) of element e in a state or
// adjoint buffer.
template <class Lay>
__device__ __forceinline__ d4 ld_quad(const SRS_GLOBAL double* X, const Lay lay, uint32_t e) {
  const SRS_GLOBAL d2* p = (const SRS_GLOBAL d2*)X + lay.at(e);
  const d2 a = p[0], b = p[lay.half()];
  return d4{a.x, a.y, b.x, b.y};
}
template <bool NT, class Lay>
__device__ __forceinline__ void st_quad(SRS_GLOBAL double* X, const Lay lay, uint32_t e, const d4 m) {
  SRS_GLOBAL d2* p = (SRS_GLOBAL d2*)X + lay.at(e);
  stg<NT>(p, d2{m.x, m.y});
  stg<NT>(p + lay.half(), d2{m.z, m.w});
}
typedef int i2 __attribute__((ext_vector_type(2)));
typedef int i4 __attribute__((ext_vector_type(4)));
typedef int i3 __attribute__((ext_vector_type(3), aligned(4)));

// A tile's quads in LDS: its own elements' first, then its halo's (the
// elements outside the tile that its elements neighbour, each once), as two
// arrays of pairs (consecutive lanes read consecutive 16 B).
struct QuadTile {
  d2 *a, *b;
  __device__ __forceinline__ QuadTile(void* lds, int cap) : a((d2*)lds), b((d2*)lds + cap) {}
  __device__ __forceinline__ void put(int k, const d4 m) const {
    a[k] = d2{m.x, m.y};
    b[k] = d2{m.z, m.w};
  }
  __device__ __forceinline__ d4 get(int k) const { return d4{a[k].x, a[k].y, b[k].x, b[k].y}; }
};

// Read-only data at a wavefront-uniform address: a scalar load.
template <class T>
__device__ __forceinline__ T sld(const T* p) { return *(const __attribute__((address_space(4))) T*)p; }

// An element index with bit 31 set where the element has F_SL, as the halo
// lists and the neighbour table hold them.
constexpr uint32_t IDX_SL = 0x80000000u;
__host__ __device__ __forceinline__ uint32_t idx_of(uint32_t e) { return e & ~IDX_SL; }

// A tile's run of the halo list, and the entries of a thread: the first HPRE
// of them are loaded ahead of everything that does not depend on them.
constexpr int HPRE = 2;
struct Halo {
  int s, n;
  uint32_t e[HPRE];
};
template <int BS>
__device__ __forceinline__ Halo load_halo(const uint32_t* hal, const int32_t* hoff, const int t) {
  Halo h;
  h.s = sld(hoff + t);
  h.n = sld(hoff + t + 1) - h.s;
#pragma unroll
  for (int q = 0; q < HPRE; ++q) {
    const int k = (int)threadIdx.x + q * BS;
    h.e[q] = k < h.n ? gp(hal)[h.s + k] : 0u;
  }
  return h;
}
// put(i, e) for each of the thread's halo entries e, i its place in the halo.
template <int BS, class F>
__device__ __forceinline__ void each_halo(const uint32_t* hal, const Halo& h, F put) {
#pragma unroll
  for (int q = 0; q < HPRE; ++q)
    if ((int)threadIdx.x + q * BS < h.n) put((int)threadIdx.x + q * BS, h.e[q]);
  for (int k = (int)threadIdx.x + HPRE * BS; k < h.n; k += BS) put(k, gp(hal)[h.s + k]);
}

// TnC has a nonzero rate only in cytosol elements with troponin, CSQ only in
// the jSR (cpu/RunSimulation.cpp:45-46 reset both rates to zero).  A zero rate
// leaves the value unchanged, and both state buffers hold the same value, so
// those planes are neither read nor written elsewhere.
__device__ __forceinline__ bool lives_tr(const uint8_t f) { return (f & (F_JSR | F_TROPC)) == F_TROPC; }
__device__ __forceinline__ bool lives_cs(const uint8_t f) { return (f & F_JSR) != 0; }

// Operator row of one element: coefficients (diagonal first), its neighbours'
// places among the tile's staged quads, and flags.  Mesh-level data, shared
// by every realization of the mesh.
struct Geo {
  double a0, a1, a2, a3, a4;
  int l1, l2, l3, l4;
  uint8_t f;
};

// A class row's coefficient: the class value with its bit pattern moved by
// the element's delta.
__device__ __forceinline__ double ulps_from(const double t, const int delta) {
  return __longlong_as_double(__double_as_longlong(t) + (long long)delta);
}
template <bool CLASS>
__device__ __forceinline__ void load_coef(const RealDesc& d, const int j, Geo& g) {
  if constexpr (CLASS) {
    // reproduces the assembled FP64 values exactly (every row was checked
    // when the mesh was added)
    const i3 r = *(const SRS_GLOBAL i3*)(gp(d.row) + 3 * (size_t)j);
    const SRS_GLOBAL double* t = gp(d.tab) + 5 * (r.x & 0xffff);
    g.a0 = ulps_from(t[0], r.x >> 16);
    g.a1 = ulps_from(t[1], (int16_t)r.y);
    g.a2 = ulps_from(t[2], r.y >> 16);
    g.a3 = ulps_from(t[3], (int16_t)r.z);
    g.a4 = ulps_from(t[4], r.z >> 16);
  } else {
    const size_t np = d.np;
    const SRS_GLOBAL double* cf = gp(d.coef);
    g.a0 = cf[j]; g.a1 = cf[np + j]; g.a2 = cf[2 * np + j]; g.a3 = cf[3 * np + j]; g.a4 = cf[4 * np + j];
  }
}
// The row of an element of the workgroup's tile.  b: the flags of the
// element's block; in a plain block no element flags are loaded.  A row is two
// wide loads (places 8 B, class row 12 B).
template <bool CLASS>
__device__ __forceinline__ Geo load_geo(const RealDesc& d, const uint16_t* loc, const int j, const uint32_t b) {
  Geo g;
  g.f = (b & BLK_PLAIN) ? (uint8_t)F_TROPC : gp(d.flags)[j];
  const i2 q = ((const SRS_GLOBAL i2*)loc)[j];
  g.l1 = q.x & 0xffff; g.l2 = (uint32_t)q.x >> 16;
  g.l3 = q.y & 0xffff; g.l4 = (uint32_t)q.y >> 16;
  load_coef<CLASS>(d, j, g);
  return g;
}
// The row of any element, with neighbour indices (IDX_SL) in place of tile places.
template <bool CLASS>
__device__ __forceinline__ Geo load_geo_nbr(const RealDesc& d, const int j) {
  Geo g;
  g.f = gp(d.flags)[j];
  const i4 q = ((const SRS_GLOBAL i4*)d.nbr)[j];
  g.l1 = q.x; g.l2 = q.y; g.l3 = q.z; g.l4 = q.w;
  load_coef<CLASS>(d, j, g);
  return g;
}
// The operator row applied to an element's own and its neighbours' quads, in
// the reference's order (cpu/RunSimulation.cpp:61-71).
__device__ __forceinline__ d4 row_sum(const Geo& g, const d4& m0, const d4& m1, const d4& m2, const d4& m3,
                                      const d4& m4) {
  return m0 * g.a0 + m1 * g.a1 + m2 * g.a2 + m3 * g.a3 + m4 * g.a4;
}

// Index in celem of each F_CHAN lane's element (chan: those lanes, j the
// lane's element, consecutive across a wavefront of 64 active lanes), -1 where
// the element is another realization's.  The records of a wavefront's
// elements follow each other, so one round of loads counts those before them
// and the flags below a lane give its place; on a mesh shared with other
// clusters, a search.
__device__ __forceinline__ int chan_place(const RealDesc& d, const int j, const uint64_t chan) {
  const int lane = threadIdx.x & 63, j0 = j - lane;
  int before = 0;
  for (int k = 0; k < d.n_celem; k += 64)
    before += __builtin_popcountll(
        __builtin_amdgcn_ballot_w64(k + lane < d.n_celem && d.celem[min(k + lane, d.n_celem - 1)] < j0));
  if (!(chan >> lane & 1)) return -1;
  const int own = before + __builtin_popcountll(chan & ((1ull << lane) - 1));
  if (own < d.n_celem && d.celem[own] == j) return own;
  int lo = before, hi = min(own, d.n_celem);
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (d.celem[mid] < j) lo = mid + 1; else hi = mid;
  }
  return lo < d.n_celem && d.celem[lo] == j ? lo : -1;
}

// The flags of the block of element j, j consecutive across the wavefront from
// a multiple of 64.
__device__ __forceinline__ uint32_t block_flags(const RealDesc& d, const int j) {
  return sld(d.blk + (__builtin_amdgcn_readfirstlane(j) >> 6));
}

// --------------------------------------------- line-scan geometry and sizes
// linescan/main.cpp:195-249.  The blurred fluorescence of scan point i is
// sum_j V0_j CaF_j w(c_j - p_i) over cells with |c_j - p_i|^2 < 1, with the
// Gaussian PSF w of linescan/parameters.h:60-62.  Mesh cells are summed on the
// device, one partial sum per workgroup and point, then the partials in
// workgroup order; the padding cells' part is a per-point constant.
//
// Along the line only the axis term of the PSF's exponent changes, by a
// quadratic in the point index, so k points from a point of weight w0 and
// ratio r0 = w(1) / w0 a cell's weight is w0 r0^k q^(k (k - 1) / 2) upwards and
// w0 r0^-k q^(k (k + 1) / 2) downwards, q = exp(-res^2 / s_a^2): one product
// per point and cell instead of an exponential, and the powers of q are factors
// of a point's whole sum.  Points go in segments of SCAN_SEG, with the closed
// form at the middle one (two exponentials per segment and cell), which keeps
// the rounding of a weight within a few tens of ulps.  PSFs so narrow that a
// middle weight could underflow while its segment holds a weight above
// exp(-260), or a power of the ratio overflow, within a cell's reach take the
// closed form at every point (walk = 0).
constexpr int SCAN_SEG = 16, SCAN_HALF = SCAN_SEG / 2;

struct ScanGeo {
  double base[3];   // scan line point with the axis coordinate zero
  int axis;
  double x_min, res;
  double sx, sy, sz, alpha;
  double inv[3];    // 1 / s^2 per coordinate (s = sx, sy, sz)
  double ia;        // inv[axis] (device code indexes no array by axis: the
                    // struct then stays in scalar registers)
  double kw;        // alpha / (sx sy sz)
  double pw[SCAN_HALF + 1];  // q^(k (k + 1) / 2), q = exp(-res^2 inv[axis])
  int walk;         // 1: the recurrence above; 0: the closed form everywhere
};

// One cell's terms of the walk: its axis coordinate, the perpendicular
// squares in the reference's summation order (distance^2 = (da^2 + u) + v,
// da the axis difference) and the perpendicular part of the PSF exponent.
struct ScanCell {
  double ca, u, v, eperp;
};
__device__ __forceinline__ ScanCell scan_cell(const ScanGeo& g, double cx, double cy, double cz) {
  const double r0 = cx - g.base[0], r1 = cy - g.base[1], r2 = cz - g.base[2];
  const double t0 = r0 * r0, t1 = r1 * r1, t2 = r2 * r2;
  ScanCell c;
  if (g.axis == 0) { c.ca = cx; c.u = t1; c.v = t2; c.eperp = t1 * g.inv[1] + t2 * g.inv[2]; }
  else if (g.axis == 1) { c.ca = cy; c.u = t0; c.v = t2; c.eperp = t0 * g.inv[0] + t2 * g.inv[2]; }
  else { c.ca = cz; c.u = t0 + t1; c.v = 0.0; c.eperp = t0 * g.inv[0] + t1 * g.inv[1]; }
  return c;
}
// Axis coordinate of scan point i (linescan/main.cpp:199-200).
__device__ __forceinline__ double scan_pa(const ScanGeo& g, int i) { return g.x_min + i * g.res; }
// The reference's distance^2 between the cell and point i, bit for bit.
__device__ __forceinline__ double scan_dist2(const ScanCell& c, double pa) {
  const double da = c.ca - pa;
  return (da * da + c.u) + c.v;
}
// Weight at point i from the closed form and the ratio to point i + 1.
__device__ __forceinline__ void scan_anchor(const ScanGeo& g, const ScanCell& c, double pa, double* w, double* r) {
  const double da = c.ca - pa, ia = g.ia;
  *w = g.kw * exp(-0.5 * (da * da * ia + c.eperp));
  *r = exp(g.res * (da - 0.5 * g.res) * ia);
}
// The points within the reference's exact cut-off of a cell, [lo, hi] (none
// if lo > hi), inside a superset [lo, hi] (scan_point_range).  The point
// coordinate x_min + i res rises with i and every rounding step is monotonic,
// so the distance^2 falls and then rises along the line: the points that pass
// are one run, found by testing its ends, and the callers' per-point test
// becomes a range check (the same points, the same bits).
__device__ __forceinline__ void scan_exact_range(const ScanGeo& g, const ScanCell& c, int* lo, int* hi) {
  while (*lo <= *hi && !(scan_dist2(c, scan_pa(g, *lo)) < 1.0)) ++*lo;
  while (*hi >= *lo && !(scan_dist2(c, scan_pa(g, *hi)) < 1.0)) --*hi;
}
// The reciprocal of a ratio in the normal range, to the last bit or so.
__device__ __forceinline__ double scan_rcp(double r) {
  double x = __builtin_amdgcn_rcp(r);
  x = __builtin_fma(x, __builtin_fma(-r, x, 1.0), x);
  return __builtin_fma(x, __builtin_fma(-r, x, 1.0), x);
}
// f(m, t) at the points base + m of a segment that use(first, last) asks for,
// half by half: t times scan_power(m) is scale times the cell's weight there.
template <bool WALK, class U, class F>
__device__ __forceinline__ void scan_walk(const ScanGeo& g, const ScanCell& c, int base, double scale, U use, F f) {
  if constexpr (WALK) {
    double w0, r0;
    scan_anchor(g, c, scan_pa(g, base + SCAN_HALF), &w0, &r0);
    w0 *= scale;
    if (use(SCAN_HALF, SCAN_SEG - 1)) {
      double t = w0;
#pragma unroll
      for (int k = 0; k < SCAN_HALF; ++k) {
        f(SCAN_HALF + k, t);
        t *= r0;
      }
    }
    if (use(0, SCAN_HALF - 1)) {
      const double rd = scan_rcp(r0);
      double t = w0;
#pragma unroll
      for (int k = 1; k <= SCAN_HALF; ++k) {
        t *= rd;
        f(SCAN_HALF - k, t);
      }
    }
  } else {
    for (int m = 0; m < SCAN_SEG; ++m) {
      double w, r;
      scan_anchor(g, c, scan_pa(g, base + m), &w, &r);
      f(m, scale * w);
    }
  }
}
template <bool WALK>
__device__ __forceinline__ double scan_power(const ScanGeo& g, int m) {
  return !WALK ? 1.0 : m >= SCAN_HALF ? g.pw[m > SCAN_HALF ? m - SCAN_HALF - 1 : 0] : g.pw[SCAN_HALF - m];
}
// First point of the segment that holds point i.
__device__ __forceinline__ int scan_seg(int i) { return i & ~(SCAN_SEG - 1); }

// The scan points a cell at (cx, cy, cz) can reach (distance < 1 um): none
// (lo > hi) when its distance to the line is 1 um or more, else those whose
// axis coordinate lies within sqrt(1 - t^2) of the cell's, t the distance to
// the line, widened by one point each way and by 1e-9 on t^2 against the
// rounding of the exact test, which the callers still apply.
__device__ __forceinline__ void scan_point_range(const ScanGeo& g, int n_f, double cx, double cy, double cz, int* lo,
                                                 int* hi) {
  const double ca = g.axis == 0 ? cx : g.axis == 1 ? cy : cz;
  double t2 = 0.0;
  if (g.axis != 0) t2 += (cx - g.base[0]) * (cx - g.base[0]);
  if (g.axis != 1) t2 += (cy - g.base[1]) * (cy - g.base[1]);
  if (g.axis != 2) t2 += (cz - g.base[2]) * (cz - g.base[2]);
  if (!(t2 < 1.0 + 1e-9)) {
    *lo = n_f;
    *hi = -1;
    return;
  }
  const double half = sqrt(1.0 + 1e-9 - t2);
  *lo = max(0, (int)floor((ca - half - g.x_min) / g.res) - 1);
  *hi = min(n_f - 1, (int)ceil((ca + half - g.x_min) / g.res) + 1);
}

constexpr int SCAN_BS = 256;
constexpr int SCAN_MAX_POINTS = 1024;
constexpr int SCAN_CELLS_PER_THREAD = 4;

// LDS of the blur's workgroup, its wavefronts' sums per point, and the
// workgroups of the final sum, a wavefront per point.
inline size_t scan_lds(int n_f) { return sizeof(double) * (SCAN_BS / 64) * (size_t)n_f; }
inline unsigned scan_final_blocks(int n_f) { return (unsigned)std::max(1, (n_f + SCAN_BS / 64 - 1) / (SCAN_BS / 64)); }

// Realization of workgroup row blockIdx.y in a batched launch: rid[blockIdx.y],
// or r when there is no table (a launch for one realization).
__device__ __forceinline__ int batch_real(const int32_t* __restrict__ rid, int r) { return rid ? rid[blockIdx.y] : r; }

// ----------------------------------------------------------- host-side state

#define HIPCHK(expr)                                                                  \
  do {                                                                                \
    hipError_t _e = (expr);                                                           \
    if (_e != hipSuccess) return srs::fail(SRS_E_HIP, "%s: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, __LINE__); \
  } while (0)

struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
};

// body(i) for i in [0, n), on up to eight threads for long work; false if a
// body threw.
template <class F>
bool each_chunk(int n, F body) {
  std::atomic<int> next{0};
  std::atomic<bool> ok{true};
  auto work = [&] {
    try {
      for (int i; (i = next.fetch_add(1)) < n && ok;) body(i);
    } catch (...) {
      ok = false;
    }
  };
  std::vector<std::thread> th;
  try {
    const int helpers = std::min({n - 1, 7, (int)std::thread::hardware_concurrency() - 1});
    for (int k = 0; k < helpers; ++k) th.emplace_back(work);
  } catch (...) {  // fewer threads than asked for
  }
  work();
  for (std::thread& t : th) t.join();
  return ok;
}

// Where the neighbours of a tile's elements are once the tile is staged: place
// k < tile is the tile's own element k, place tile + i the i-th of its halo.
struct TileMap {
  int tile = 0;       // elements per tile; 0: not built
  int32_t qcap = 0;   // the most quads a tile stages (its elements and its halo)
  int32_t n_halo = 0; // elements of all halos
  uint16_t* d_loc = nullptr;
  uint32_t* d_hal = nullptr;
  int32_t* d_hoff = nullptr;
};

struct HostMesh {
  int32_t n = 0, np = 0;
  std::vector<int32_t> perm;  // dev -> ref
  std::vector<int32_t> inv;   // ref -> dev
  std::vector<uint32_t> nbr;  // [np][4] dev numbering (IDX_SL)
  std::vector<double> coef;   // [5][np]
  std::vector<uint8_t> flags;
  std::vector<double> V0, tt, br;  // br [4][np] or empty
  // The D of the four diffusing species that br was built with
  // (D Face_C b / V0, cpu/InitFuncs.cpp:1019-1024): those of the first
  // realization added on the mesh, which every later one must share.
  double br_d[4] = {0, 0, 0, 0};
  bool br_d_set = false;
  TileMap map;                      // of the sweep's tiles
  // compact operator layout
  bool class_rows = false;          // row and tab reproduce every coefficient
  std::vector<uint32_t> row;        // [np][3]
  std::vector<double> tab;
  int32_t n_class = 0;
  uint32_t* d_nbr = nullptr;
  int32_t* d_inv = nullptr;
  double *d_coef = nullptr, *d_V0 = nullptr, *d_tt = nullptr, *d_br = nullptr, *d_tab = nullptr;
  uint8_t* d_flags = nullptr;
  uint32_t *d_blk = nullptr, *d_row = nullptr;
};

struct HostReal {
  int32_t mesh = 0;
  double* d_br_own = nullptr;  // boundary rates rescaled to this realization's D (srs_params_set)
  srs_extensions ext{0, 0.0, 0.6};
  std::vector<int32_t> ryr_ele, ryr_jsr, ryr_nb, lcc_ele;  // dev numbering
  std::vector<int32_t> celem, cstart;
  std::vector<ChanEntry> centry;
  int32_t ints[SRS_N_INT];
  double reals[SRS_N_REAL];
  uint64_t key = 0, stream = 0;
  int32_t band = 0;   // index into srs_ctx::bands
  RealDesc desc{};
};

struct HostScan {
  int32_t mesh = 0, n_f = 0, n_ca = 0, n_blocks = 0;
  srs_scan_desc desc{};
  ScanGeo geo{};
  double *d_cen = nullptr, *d_pad = nullptr, *d_part = nullptr, *d_out = nullptr;
  int32_t *d_near_f = nullptr, *d_near_ca = nullptr;
};

// cpu/RunSimulation.cpp:85-88, the parts that depend on CaNSR only.
void serca_terms(double nsr, const double* P, double* out);

}  // namespace srs_dev

using namespace srs_dev;

struct srs_ctx {
  int device = 0;
  int tile_set = 0;      // SRS_TUNE_TILE, 0: chosen by srs_ctx_finalize
  int tile = 0;          // elements per k_sweep workgroup
  size_t sweep_lds = 0;  // LDS bytes of a sweep workgroup (staged quads)
  int quad_block = 64;   // the state layout's block (Quads), chosen by srs_ctx_finalize
  int nt_state = -1;     // non-temporal stores of the new state; -1: chosen by srs_ctx_finalize
  int plane_pad = 0;     // extra elements per SoA plane
  int compact = 1;       // compress operator rows when a mesh allows it
  int occ = 0;           // gated sweep's register budget: 0 by size, else six wavefronts per SIMD
  int group = 1;         // SRS_TUNE_GROUP
  int drop_finished = 1; // sweep without the tiles of finished realizations
  int gated = 1;         // fold each step's gating into the next step's sweep (k_sweep_gated) where it applies
  int alt_order = 0;      // single-realization gated sweep: tiles in reverse order on alternate steps
  int gpu_layout = 0;     // states records in the GPU program's layout (Ca_cyt at each RyR appended)
  int adj_levels = 0;     // adjoint checkpoint levels, 0: the fewest that fit the sub-batch
  int adj_last_levels = 0, adj_last_batch = 0;  // the plan of the last loss/gradient call
  int64_t adj_last_strides[6] = {};
  bool class_all = false;  // class rows on every mesh
  bool layout_fixed = false;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  bool finalized = false;
  std::vector<std::unique_ptr<HostMesh>> meshes;
  std::vector<HostReal> reals;
  std::vector<void*> allocs;
  RealDesc* d_desc = nullptr;
  RealLive* d_live = nullptr;
  int2* d_tiles = nullptr;   // {realization, tile} of the sweep
  int n_tiles = 0, grid_sweep = 0;
  // Every realization's tiles; when the finished ones hold enough of them, the
  // sweep runs over a list without them (d_tiles_live).
  std::vector<int2> tiles_all;
  int2* d_tiles_all = nullptr;
  std::vector<int2> tiles_cur;    // host copy of the tile list the sweep runs over (d_tiles)
  // Realization subsets (SRS_TUNE_SUBSET_MB): consecutive bands of the tile
  // list whose state takes at most subset_mb MB, each stepped through a
  // whole block of steps before the next, so that its state stays in the
  // last-level cache between steps.
  struct Subset { int t0, nt, r0, nr; };
  int subset_mb = 0;
  std::vector<Subset> subsets;
  bool subsets_valid = false;
  int32_t* d_sub_rids = nullptr;  // realization ids of the subsets, concatenated
  int2* d_tiles_live = nullptr;
  bool tiles_compacted = false;
  std::vector<std::vector<int32_t>> bands;  // realizations of one mesh whose tiles are side by side in the list
  double* stage[2] = {};         // pinned buffers of state transfers (state_xfer), stage_len doubles each, one allocation
  size_t stage_len = 0;
  hipEvent_t ev_stage[2] = {};
  double last_total_ms = 0, last_sweep_ms = 0;
  // captured step blocks, keyed by (steps, gate mode)
  std::map<std::pair<int64_t, uint32_t>, hipGraphExec_t> graphs;
  std::vector<HostScan> scans;
};

namespace srs_dev {

template <class T>
int dev_alloc(srs_ctx* c, T** p, size_t count) {
  *p = nullptr;
  if (count == 0) return SRS_OK;
  HIPCHK(hipMalloc((void**)p, count * sizeof(T)));
  c->allocs.push_back((void*)*p);
  return SRS_OK;
}

template <class T>
int dev_upload(srs_ctx* c, T** p, const std::vector<T>& v) {
  int rc = dev_alloc(c, p, v.size());
  if (rc) return rc;
  if (!v.empty()) HIPCHK(hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return SRS_OK;
}

// Temporary device buffers freed when the call returns.
struct DevMem {
  std::vector<void*> ptrs;
  ~DevMem() { for (void* p : ptrs) (void)hipFree(p); }
  template <class T>
  hipError_t alloc(T** p, size_t count) {
    hipError_t e = hipMalloc((void**)p, std::max<size_t>(count, 1) * sizeof(T));
    if (e == hipSuccess) ptrs.push_back((void*)*p);
    return e;
  }
};

// Context helpers (device.hip).
int check_real(srs_ctx* c, int32_t r);
void launch_sweep(srs_ctx* c);
int launch_step(srs_ctx* c, uint32_t gmode);
// m steps of a single-realization context through the gated sweep, starting
// from live state index cur, ending with the gating of the last step
void launch_gated_block(srs_ctx* c, int64_t m, int cur, uint32_t gmode);
// One replayed step of the tile list from schedule row `row` (ReplayAt), and m of
// them with the live state of the listed realizations moved on
void launch_replay(srs_ctx* c, int64_t row, int par, const double* xo = nullptr, double* xn = nullptr,
                   size_t stride = 0, int n_tiles = 1);
void launch_replay_block(srs_ctx* c, int64_t m, int64_t row, const int32_t* rid, int n_rid);
// One step through the single-realization gated sweep; xo_at/xn_at (both or
// neither) replace X[cur] -> X[cur ^ 1] as the step's state buffers.
void launch_gated(srs_ctx* c, int cur, uint32_t gmode, bool proto, const double* xo_at = nullptr,
                  double* xn_at = nullptr);
void launch_gate_single(srs_ctx* c, uint32_t gmode);
int drop_graphs(srs_ctx* c);
int tiles_full(srs_ctx* c);
int tiles_compact(srs_ctx* c);
int plan_subsets(srs_ctx* c);
void launch_subset_block(srs_ctx* c, int64_t m, uint32_t gmode);
int gated_start(srs_ctx* c, bool* ok, int* cur);
void launch_steps(srs_ctx* c, int64_t n_steps, uint32_t gmode, bool gated, int cur);
int live_rw(srs_ctx* c, int32_t r, RealLive* lv, bool write);
int state_xfer(srs_ctx* c, int32_t r, double* host, bool to_dev);

// The line-scan kernels (linescan.hip), also launched by the adjoint.
__global__ void k_scan_blur(const RealDesc* __restrict__ D, const RealLive* __restrict__ L, int r,
                            const int32_t* __restrict__ rid, const double* __restrict__ cen, ScanGeo g, int n_f,
                            double* __restrict__ part);
__global__ void k_scan_final(const RealDesc* __restrict__ D, const RealLive* __restrict__ L, int r,
                             const int32_t* __restrict__ rid, int n_blocks, int n_f, int n_ca,
                             const double* __restrict__ part, const double* __restrict__ pad,
                             const int32_t* __restrict__ near_f, const int32_t* __restrict__ near_ca, double f0,
                             double c0, double* __restrict__ out, int out_stride);

}  // namespace srs_dev
