// device.hip -- gfx950 kernels and the device half of the C ABI.
//
// One spark time-step (cpu/RunSimulation.cpp:591-654) is two kernels:
//   k_sweep : every element of every live realization, fused: 5-point ELL
//             diffusion of Ca/Fluo/ATP/CaM, binding reactions, SERCA, jSR
//             refill, RyR/LCC flux injection, rapid SL buffer and the forward
//             Euler update, old state -> new state (ping-pong buffers).
//   k_gate  : one workgroup per realization: RyR and LCC Markov gating on the
//             new Ca (integrated-hazard residuals, Philox draws), then,
//             optionally, the RunSimulation loop body for the next time
//             (while-condition, LCC trigger, voltage clamp, RyR hold,
//             states-record output).
// A single realization runs each step as one launch instead, k_sweep_gated:
// its workgroup 0 runs k_gate's body for the previous step beside the channel
// elements' update.
// The reference runs the same step as nine kernels with a state-sized rate
// buffer (gpu/RunSimulation.cu:781-852); here the rates never leave registers.
//
// Arithmetic keeps the reference's operation order and this file is compiled
// without FP contraction, so the field update is bit-identical to the
// reference CPU path for the same row order of each element's neighbours.
// The line-scan operator is in linescan.hip, recording and the adjoint in
// adjoint.hip; the shared types are in dev_common.h.
#include "dev_common.h"

#ifndef SRS_UNIT
#define SRS_UNIT 0
#endif

#include <functional>
#include <mutex>
#include <unordered_map>

namespace srs_dev {

// The state of one element of one realization: its own diffusing quad, the
// operator row applied to each diffusing species, TnC and CSQ where they are
// live.
struct Loc {
  d4 m0, s;
  double c_tr, c_cs;
};

// A realization's state buffers for one step: read X[cur], write X[cur ^ 1].
// Both pointers are loaded and one is selected, so that the live index and
// the pointers arrive in the same round of scalar loads.
struct Bufs {
  const SRS_GLOBAL double* xo;
  SRS_GLOBAL double* xn;
};
__device__ __forceinline__ Bufs bufs(double* x0, double* x1, int cur) {
  return cur ? Bufs{gp(x1), gpw(x0)} : Bufs{gp(x0), gpw(x1)};
}

// Pins uniform values to this point of the program: the scalar loads that
// produce them are issued as one batch ahead of the branches that follow,
// instead of one memory round trip after another where each is first used.
// The values are folded into one operand of an empty asm statement.
template <typename T>
__device__ __forceinline__ uint64_t fold_bits(const T v) {
  if constexpr (std::is_pointer<T>::value) return (uint64_t)(uintptr_t)v;
  else return (uint64_t)(int64_t)v;
}
template <typename... T>
__device__ __forceinline__ uint64_t fold(const T... v) {
  return (fold_bits(v) ^ ...);
}
__device__ __forceinline__ void scalars_here(const uint64_t folded) { __asm__ volatile("" ::"s"(folded)); }

// An element's rates without the channel fluxes, and the divisor of the rapid
// buffers (B, used where `div`).
struct Rates {
  double ca, dy, at, cm, tr, cs, B;
  bool div;
};

// In the reference's operation order (cpu/RunSimulation.cpp:591-618).  ttj, v0j:
// the TT area and volume of an element with F_SL.
template <int FK>
__device__ __forceinline__ Rates elem_rates(const RealDesc& d, const RealLive& l, const int j, const uint8_t flags,
                                            const Loc& c, const double ttj, const double v0j) {
  const size_t np = d.np;
  const double* P = d.P;
  const uint8_t f = FK >= 0 ? (uint8_t)FK : flags;
  const double c_ca = c.m0.x, c_at = c.m0.y, c_cm = c.m0.z, c_dy = c.m0.w;
  const double c_tr = c.c_tr, c_cs = c.c_cs;
  const bool live_cs = lives_cs(f);

  double br_ca = 0.0, br_dy = 0.0, br_at = 0.0, br_cm = 0.0;
  if (f & F_BR) {
    const SRS_GLOBAL double* br = gp(d.br);
    br_ca = br[j];
    br_dy = br[np + j];
    br_at = br[2 * np + j];
    br_cm = br[3 * np + j];
  }
  // cpu/RunSimulation.cpp:61-71 (Ca uses D_CA in both domains; with the jSR
  // diffusion extension, D_CAJSR in jSR elements)
  const double d_ca = (live_cs && d.jsr_diff) ? P[SRS_R_D_CA_JSR] : P[SRS_R_D_CA];
  Rates r;
  r.ca = d_ca * c.s.x + br_ca;
  r.dy = P[SRS_R_D_DYE] * c.s.w + br_dy;
  r.at = P[SRS_R_D_ATP] * c.s.y + br_at;
  r.cm = P[SRS_R_D_CMDN] * c.s.z + br_cm;
  r.tr = r.cs = 0.0;

  if (!(f & F_JSR)) {
    if (f & F_TROPC) {  // :75-91
      const double q = P[SRS_R_K_ON_TRPN] * (P[SRS_R_B_TOT_TRPN] - c_tr) * c_ca - P[SRS_R_K_OFF_TRPN] * c_tr;
      r.ca += -q;
      r.tr = q;
      double K_i = c_ca / P[SRS_R_K_D_I];
      K_i = K_i * K_i;
      const double D_cycle = l.serca[0] + K_i * l.serca[1] + K_i * K_i * l.serca[2];
      const double v_cycle = (K_i * K_i * 3.24873e12 + K_i * l.serca[3] - l.serca[4]) / D_cycle;
      const double d_serca = (2e-3) * v_cycle * P[SRS_R_A_P];
      r.ca -= d_serca;
    }
    double q = P[SRS_R_K_ON_DYE] * (P[SRS_R_B_TOT_DYE] - c_dy) * c_ca - P[SRS_R_K_OFF_DYE] * c_dy;
    r.ca += -q;
    r.dy += q;
    q = P[SRS_R_K_ON_ATP] * (P[SRS_R_B_TOT_ATP] - c_at) * c_ca - P[SRS_R_K_OFF_ATP] * c_at;
    r.ca += -q;
    r.at += q;
    q = P[SRS_R_K_ON_CMDN] * (P[SRS_R_B_TOT_CMDN] - c_cm) * c_ca - P[SRS_R_K_OFF_CMDN] * c_cm;
    r.ca += -q;
    r.cm += q;
  } else {  // :113-121
    const double q = P[SRS_R_K_ON_CSQN] * (P[SRS_R_B_T_JSR] - c_cs) * c_ca - P[SRS_R_K_OFF_CSQN] * c_cs;
    r.ca += -q;
    r.cs = q;
    r.ca += (l.ca_nsr - c_ca) * P[SRS_R_V_REFILL];
  }

  // SR-site rapid buffer of the cytosol (extension; b_sr == 0 in the reference model)
  const bool sr = !live_cs && d.b_sr != 0.0;
  r.B = 1.0;
  r.div = (f & F_SL) || sr;
  if (r.div) {
    if (f & F_SL) {  // :15-22; B == 1 exactly where the TT area is zero
      const double btothi = ttj * P[SRS_R_B_TOT_SL_HI] / (v0j * (1e-15));
      const double btotlo = ttj * P[SRS_R_B_TOT_SL_LO] / (v0j * (1e-15));
      const double kh = P[SRS_R_K_D_SL_HI], kl = P[SRS_R_K_D_SL_LO];
      r.B = 1 + (btothi * kh / ((kh + c_ca) * (kh + c_ca))) + (btotlo * kl / ((kl + c_ca) * (kl + c_ca)));
    }
    if (sr) r.B = r.B + d.b_sr * d.k_sr / ((d.k_sr + c_ca) * (d.k_sr + c_ca));
  }
  return r;
}

// Adds one channel's flux to an element's Ca rate (cpu/RunSimulation.cpp:619-632).
// dc: Ca of a RyR's jSR element less its cleft element's.
__device__ __forceinline__ void chan_flux(const RealDesc& d, const RealLive& l, const int code, const bool open,
                                          const double dc, const double c_ca, const double v0, double& rca) {
  const double* P = d.P;
  if (!open) return;
  if (code >= 0) {
    const double J = P[SRS_R_V_RYR] * dc * P[SRS_R_V_CELL];
    if (code & 1) rca -= J / v0; else rca += J / v0;
  } else {
    rca += srs_lcc_flux_raw(l.vm, c_ca, P[SRS_R_CA_0]) / v0;
  }
}

// Division by the rapid buffers and forward Euler (:633-644).
template <bool NTS, int QB, int FK>
__device__ __forceinline__ void elem_store(const RealDesc& d, const Bufs bf, const int j, const uint8_t flags,
                                           const Loc& c, const Rates& r) {
  const size_t np = d.np;
  const uint8_t f = FK >= 0 ? (uint8_t)FK : flags;
  const double dt = d.P[SRS_R_T_STEP];
  SRS_GLOBAL double* __restrict__ Xn = bf.xn;
  const double rca = r.div ? r.ca / r.B : r.ca;
  st_quad<NTS>(Xn, Quads<QB>(), j,
               d4{c.m0.x + rca * dt, c.m0.y + r.at * dt, c.m0.z + r.cm * dt, c.m0.w + r.dy * dt});
  if (lives_tr(f)) stg<NTS>(Xn + 4 * np + j, c.c_tr + r.tr * dt);
  if (lives_cs(f)) stg<NTS>(Xn + 5 * np + j, c.c_cs + r.cs * dt);
}

// The fused step of one element of one realization, from its loaded row and
// state, in the reference's operation order (cpu/RunSimulation.cpp:591-648).
// ryr: the RyR states that the fluxes read.
template <bool NTS, int QB, int FK>
__device__ __forceinline__ void step_elem(const RealDesc& d, const RealLive& l, const Bufs bf, const int j,
                                          const uint8_t flags, const Loc& c, const int32_t* ryr) {
  const uint8_t f = FK >= 0 ? (uint8_t)FK : flags;
  const bool sl = (f & F_SL) != 0;
  Rates r = elem_rates<FK>(d, l, j, f, c, sl ? gp(d.tt)[j] : 0.0, sl ? gp(d.V0)[j] : 1.0);
  if (f & F_CHAN) {  // contributions in the reference's channel order
    int lo = 0, hi = d.n_celem;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (d.celem[mid] < j) lo = mid + 1; else hi = mid;
    }
    if (lo < d.n_celem && d.celem[lo] == j) {
      const double v0 = d.V0[j];
      for (int e = d.cstart[lo]; e < d.cstart[lo + 1]; ++e) {
        const ChanEntry en = d.centry[e];
        const int i = en.code >= 0 ? en.code >> 1 : -en.code - 1;
        const bool open = en.code >= 0 ? ryr[i] != 0 : srs_lcc_open(d.lcc_state[i], d.lccv_state[i]);
        const double dc = open && en.code >= 0 ? bf.xo[Quads<QB>::ca(en.jsr)] - bf.xo[Quads<QB>::ca(en.cyt)] : 0.0;
        chan_flux(d, l, en.code, open, dc, c.m0.x, v0, r.ca);
      }
    }
  }
  elem_store<NTS, QB, FK>(d, bf, j, f, c, r);
}

// The sizes and mesh pointers of a tile's rows and halo, folded for scalars_here.
template <bool CLASS>
__device__ __forceinline__ uint64_t geo_fold(const RealDesc& d) {
  const uint64_t m = fold(d.n, d.np, d.flags, d.blk, d.loc, d.hal, d.hoff, d.qcap);
  if constexpr (CLASS) return m ^ fold(d.row, d.tab);
  else return m ^ fold(d.coef);
}

extern __shared__ double dyn_lds[];

// One tile of one realization.  The tile's quads and its halo's are staged in
// LDS (every lane's own by consecutive loads, the halo's by the tile's sorted
// list, each element once) and each element reads its neighbours from there.
// Bound by the memory system, not by arithmetic (with the reactions left out
// the step takes as long): a 48-member ensemble (6.68M elements) moves 110 B
// per element-step at 5.5 TB/s, a copy of the same shape runs at 5.5.  When each
// element gathered its out-of-tile neighbours itself, a neighbour of several
// elements was fetched for each of them, and every wavefront held four quads
// in flight in registers: 84 VGPRs against 64, 175 us against 160 us per step of
// that ensemble with 512-element tiles, 71.4 against 66.8 us (separate gating,
// 3M-element dyad).
// A wavefront whose elements are all plain cytosol with troponin (the bulk of
// a mesh, known from its block's flags) runs the specialisation with the flags
// known at compile time.
template <int BS, bool NTS, bool CLASS, int QB, bool SKIP_CHAN>
__device__ __forceinline__ void sweep_tile(const RealDesc& d, const RealLive& l, const Bufs bf, const int t,
                                           const int32_t* ryr) {
  const QuadTile tq(dyn_lds, d.qcap);
  const Halo h = load_halo<BS>(d.hal, d.hoff, t);
  const int j = t * BS + (int)threadIdx.x;
  // rows and states are padded to whole tiles, so the last tile's lanes past
  // the mesh load (and discard) zeros
  const uint32_t b = block_flags(d, j);
  const Geo g = load_geo<CLASS>(d, d.loc, j, b);
  const SRS_GLOBAL double* Xo = bf.xo;
  const size_t np = d.np, pl = 4 * np + (size_t)j;
  auto quad = [&](int e) { return ld_quad(Xo, Quads<QB>(), e); };
  Loc c;
  c.m0 = quad(j);
  // the element's TnC is loaded with its quad, before its flags are known (it
  // is live in all but jSR and troponin-free cytosol elements)
  c.c_tr = Xo[pl];
  tq.put(threadIdx.x, c.m0);
  each_halo<BS>(d.hal, h, [&](int i, uint32_t e) { tq.put(BS + i, quad((int)idx_of(e))); });
  __syncthreads();
  if (j >= d.n || (SKIP_CHAN && (g.f & F_CHAN))) return;
  c.s = row_sum(g, c.m0, tq.get(g.l1), tq.get(g.l2), tq.get(g.l3), tq.get(g.l4));
  if (b & BLK_PLAIN) {
    step_elem<NTS, QB, F_TROPC>(d, l, bf, j, g.f, c, ryr);
  } else {
    if (!lives_tr(g.f)) c.c_tr = 0.0;
    c.c_cs = lives_cs(g.f) ? Xo[pl + np] : 0.0;
    step_elem<NTS, QB, -1>(d, l, bf, j, g.f, c, ryr);
  }
}

// A replayed step: the RyR states of schedule row `row`, from X[cur ^ par] (or,
// with xo, realization y of the tile list's from xo + y stride to xn + y
// stride, each with n_tiles tiles in turn).
struct ReplayAt {
  int64_t row;
  const double* xo;
  double* xn;
  size_t stride;
  int par, n_tiles;
};

// REPLAY: the step takes its RyR states from the schedule itself, so that no
// gating launch lies between replayed steps and nothing but the fields changes
// until k_replay_end: fitting call of three 90,540-element members, 724 steps,
// 35.0 -> 29.0 ms (a step was sweep and gating forward, and those two and an
// update of the state pointers when recomputed), of eight of 927,816, 39.5 ->
// 39.1.  A single realization's replay is faster through the gated sweep (call
// of 56,250 elements, 39.3 against 42.9 ms: its channel elements are the longest
// chain there).
template <int BS, bool NTS, bool CLASS, int QB, bool REPLAY>
__global__ __launch_bounds__(BS) void k_sweep(const RealDesc* __restrict__ D, const RealLive* __restrict__ L,
                                              const int2* __restrict__ tiles, int n_tiles, int single, ReplayAt at) {
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  if (b >= n_tiles) return;
  const int2 tl = single ? make_int2(0, b) : tiles[b];  // {realization, tile}
  const RealDesc& d = D[tl.x];
  const RealLive& l = L[tl.x];
  // a finished realization (done) or one in the gating-only ffwd phase keeps
  // its fields
  const int skip = l.done | l.ffwd;
  Bufs bf = bufs(d.X[0], d.X[1], REPLAY ? l.cur ^ at.par : l.cur);
  if (REPLAY && at.xo) {
    const size_t y = (size_t)(b / at.n_tiles) * at.stride;
    bf = Bufs{gp(at.xo + y), gpw(at.xn + y)};
  }
  const int32_t* ryr = REPLAY ? d.sched + at.row * d.n_ryr : d.ryr_state;
  scalars_here(fold(skip, bf.xo, bf.xn) ^ geo_fold<CLASS>(d));
  if (skip) return;
  sweep_tile<BS, NTS, CLASS, QB, false>(d, l, bf, tl.y, ryr);
}

template <class Lay>
__device__ void write_record(const RealDesc& d, RealLive& l, const double* Ca, const Lay lay, double t) {
  // Called by one thread: sums run sequentially, in the reference's order.
  if (l.rec_count >= d.rec_cap) { l.rec_overflow = 1; return; }
  float* rec = d.rec + (size_t)l.rec_count * d.rec_len;
  int k = 0;
  rec[k++] = (float)t;
  double i_ryr = 0;
  for (int i = 0; i < d.n_ryr; ++i)
    i_ryr += d.ryr_state[i] * d.P[SRS_R_V_RYR] * (Ca[lay.ca(d.ryr_jsr[i])] - Ca[lay.ca(d.ryr_ele[i])]) * (d.P[SRS_R_V_CELL]) * 96485 *
             2 * (1e-6);
  rec[k++] = (float)i_ryr;
  int n_open = 0;
  for (int i = 0; i < d.n_ryr; ++i) n_open += d.ryr_state[i];
  rec[k++] = (float)n_open;
  int n_open_lcc = 0;
  for (int i = 0; i < d.n_lcc; ++i)
    if (d.lccv_state[i] == 2 && (d.lcc_state[i] == 6 || d.lcc_state[i] == 12)) n_open_lcc++;
  rec[k++] = (float)n_open_lcc;
  double i_lcc = 0;
  for (int i = 0; i < d.n_lcc; ++i)
    if (srs_lcc_open(d.lcc_state[i], d.lccv_state[i]))
      i_lcc += srs_lcc_flux_raw(l.vm, Ca[lay.ca(d.lcc_ele[i])], d.P[SRS_R_CA_0]) * 96485 * 2 * (1e-6);
  rec[k++] = (float)i_lcc;
  double m = 0;
  for (int i = 0; i < d.n_ryr; ++i) m += Ca[lay.ca(d.ryr_jsr[i])];
  m /= d.n_ryr;
  rec[k++] = (float)m;
  m = 0;
  for (int i = 0; i < d.n_ryr; ++i) m += Ca[lay.ca(d.ryr_ele[i])];
  m /= d.n_ryr;
  rec[k++] = (float)m;
  if (d.gpu_layout)
    for (int i = 0; i < d.n_ryr; ++i) rec[k++] = (float)Ca[lay.ca(d.ryr_ele[i])];
  if (d.ryr_out)
    for (int i = 0; i < d.n_ryr; ++i) rec[k++] = (float)d.ryr_state[i];
  l.rec_count++;
}

constexpr int GATE_RYR = 3 * MAX_RYR, GATE_LCC = 4 * MAX_RYR;
constexpr size_t GATE_LDS = (GATE_LCC + MAX_LCC) * sizeof(int);
// Where a step does not gate: the LCCs as they are.
template <int NT>
__device__ __forceinline__ void held_lccs(const RealDesc& d, int* smem) {
  for (int i = NT - 1 - threadIdx.x; i < d.n_lcc; i += NT)
    smem[GATE_LCC + i] = srs_lcc_open(d.lcc_state[i], d.lccv_state[i]);
}

// The gating and loop body of realization r by one workgroup of NT threads.
// PROTO = false leaves out the loop body (callers that never pass G_PROTOCOL).
// smem: GATE_LDS bytes; from GATE_RYR its ints end as the RyR states, from
// GATE_LCC as whether the LCCs are open.  mid() runs once, by every thread,
// after the first barrier: work of other wavefronts than the first and the
// last, which mostly gate no channel, done while those two are at theirs.
struct NoMid { __device__ void operator()() const {} };
template <int NT, bool PROTO = true, class Lay, class Mid = NoMid>
__device__ __forceinline__ void gate_workgroup(const RealDesc* __restrict__ D, RealLive* __restrict__ L, const int r,
                                               const uint32_t mode, int* smem, const Lay lay, Mid mid = NoMid()) {
  static_assert(MAX_RYR % NT == 0 && MAX_LCC % NT == 0, "channel slots per thread");
  const RealDesc& d = D[r];
  RealLive& l = L[r];
  if (l.done) return;
  int *s_old = smem, *s_a = smem + MAX_RYR, *s_b = smem + 2 * MAX_RYR, *s_fin = smem + GATE_RYR;
  int* s_lcc = smem + GATE_LCC;
  const int tid = threadIdx.x;
  const int cur = l.cur;
  // In the flag_ffwd phase the sweep skipped this realization: the fields are
  // unchanged and only the channels gate (cpu/RunSimulation.cpp:474-476).
  const bool ff = l.ffwd != 0;
  const bool swept = (mode & G_AFTER_SWEEP) && !ff;
  const double* Xn = swept ? d.X[cur ^ 1] : d.X[cur];
  const double* Ca = Xn;  // Ca of element e at Ca[lay.ca(e)]
  const double* P = d.P;
  const double dt = P[SRS_R_T_STEP];
  const int64_t step = l.step;
  // read by every thread before the first barrier: thread 0 rewrites the
  // live state at the end, and the time decides below whether the whole
  // workgroup takes part in the loop-body counts
  const double t = l.t + dt;  // cpu/RunSimulation.cpp:572-573 (ffwd: :477-478)
  // ExplicitStep honours flag_nogating; the ffwd loop calls
  // UpdateChannelGating directly (cpu/RunSimulation.cpp:476, 650-652).
  const bool gating = !(mode & G_NO_GATING) && (ff || !d.I[SRS_I_FLAG_NO_GATING]);
  const int nr = d.n_ryr;

  if (gating) {
    // Everything a channel's update reads is loaded before the first barrier
    // (RyR i by thread i mod NT, LCC i by thread NT - 1 - i mod NT, so RyRs and
    // LCCs are updated side by side), leaving one memory round trip in front
    // of the arithmetic.  Channels beyond the workgroup's threads are loaded
    // when their turn comes: holding two of each per thread cost the kernel
    // this is folded into half of its registers.
    double ca_c = 0.0, ca_j = 0.0, Rr = 0.0;
    auto load_ryr = [&](const int i) {
      ca_c = Ca[lay.ca(d.ryr_ele[i])];
      ca_j = Ca[lay.ca(d.ryr_jsr[i])];
      Rr = d.R[i];
    };
    for (int i = tid; i < nr; i += NT) s_old[i] = s_a[i] = d.ryr_state[i];
    if (tid < nr) load_ryr(tid);
    int ls = 0, lvs = 0;
    double ca_l = 0.0, Rl = 0.0;
    auto load_lcc = [&](const int i) {
      ls = d.lcc_state[i];
      lvs = d.lccv_state[i];
      ca_l = Ca[lay.ca(d.lcc_ele[i])];
      Rl = d.R[nr + i];
    };
    const int l0 = NT - 1 - tid;
    if (l0 < d.n_lcc) load_lcc(l0);
    __syncthreads();
    mid();
    // LCCs, cpu/RunSimulation.cpp:229-400; first, so that their wavefronts work
    // while the RyRs' do
#pragma unroll 1
    for (int i = l0; i < d.n_lcc; i += NT) {
      if (i != l0) load_lcc(i);
      const int s = ls, vs = lvs;
      double tr[3];
      int32_t tg[3];
      const double lr = srs_lcc_rates(s, vs, l.vm, ca_l, tr, tg);
      const int ic = nr + i;
      double Rn = Rl + (tr[0] + tr[1] + tr[2] + lr) * dt;
      int sn = s, vn = vs;
      if (Rn > 0) {
        uint64_t o[4];
        srs_philox4x64_10((uint64_t)step, (uint64_t)ic, d.stream, SRS_PURPOSE_GATING, d.key, SRS_PHILOX_KEY1, o);
        Rn = log(srs_open01(o[0]));
        const double u = srs_open01(o[1]) * (tr[0] + tr[1] + tr[2] + lr);
        if (u < tr[0]) sn = tg[0];
        else if (u < tr[0] + tr[1]) sn = tg[1];
        else if (u < tr[0] + tr[1] + tr[2]) sn = tg[2];
        else vn = (vs == 1) ? 2 : 1;
        d.lcc_state[i] = sn;
        d.lccv_state[i] = vn;
      }
      s_lcc[i] = srs_lcc_open(sn, vn);
      d.R[ic] = Rn;
    }
    // RyRs: the reference updates them one after another (later RyRs see
    // earlier flips through the neighbour counts, cpu/RunSimulation.cpp:661-666).
    // Each sweep below recomputes every RyR with lower-index neighbours taken
    // from the previous sweep's result and higher-index ones from the old
    // states; the first sweep that changes nothing is the sequential result.
    // (For uncoupled RyRs the neighbour counts do not enter the rate, A* = 0
    // gives X = 1.)  A rate is some 250 dependent instructions, 0.9 us: with at
    // most one RyR per thread the last sweep's values are committed as they are
    // instead of being computed once more.
    const bool coupled = P[SRS_R_RYR_A_STAR] != 0.0;
    int* prev = s_a;
    int* next = s_b;
    double Rn = 0.0;
    int ns = 0;
    auto update = [&](const int i) {
      if (nr > NT) load_ryr(i);
      int no = 0, ncl = 0;
      if (coupled) {
        for (int q = 0; q < 4; ++q) {
          const int nb = d.ryr_nb[4 * i + q];
          if (nb >= 0) {
            const int s = (nb < i) ? prev[nb] : s_old[nb];
            if (s) no++; else ncl++;
          }
        }
      }
      Rn = Rr + srs_ryr_rate(s_old[i], no, ncl, ca_c, ca_j, P) * dt;
      ns = (Rn > 0) ? (s_old[i] == 1 ? 0 : 1) : s_old[i];
    };
    if (coupled) {
      for (int it = 0; it <= nr; ++it) {
        int changed = 0;
#pragma unroll 1
        for (int i = tid; i < nr; i += NT) {
          update(i);
          next[i] = ns;
          changed |= (ns != prev[i]);
        }
        changed = __syncthreads_or(changed);
        int* tmp = prev; prev = next; next = tmp;
        if (!changed) break;
      }
    }
    // commit
#pragma unroll 1
    for (int i = tid; i < nr; i += NT) {
      if (!coupled || nr > NT) update(i);
      if (Rn > 0) {
        uint64_t o[4];
        srs_philox4x64_10((uint64_t)step, (uint64_t)i, d.stream, SRS_PURPOSE_GATING, d.key, SRS_PHILOX_KEY1, o);
        Rn = log(srs_open01(o[0]));
      }
      d.R[i] = Rn;
      d.ryr_state[i] = ns;
      s_fin[i] = ns;
    }
  }
  else {
    // a replay (never with gating) takes the row of the next step, if there is one
    const int64_t k = step + 1 - l.sched_base;
    if ((mode & G_REPLAY) && k < d.n_sched)
      for (int i = tid; i < nr; i += NT) s_fin[i] = d.ryr_state[i] = d.sched[k * nr + i];
    else
      for (int i = tid; i < nr; i += NT) s_fin[i] = d.ryr_state[i];
    held_lccs<NT>(d, smem);
    mid();
  }
  __syncthreads();

  if (mode & G_RECORD) {  // a launch of its own after each step took 4.7 us
    const int64_t k = step + 1 - d.rec_step0;
    if (k < d.n_sched)
      for (int i = tid; i < nr; i += NT) d.sched[k * nr + i] = s_fin[i];
  }

  const double iv = P[SRS_R_OUTPUT_STATES_INTERVAL];
  const bool out_due = floor(t / iv) > floor((t - dt) / iv);
  // The loop body's counts (open RyRs, open LCCs, the largest cleft Ca over
  // the RyRs) are needed in the ffwd phase and at states outputs.  The
  // workgroup reduces them with wavefront ballots and a cross-lane max
  // (exact: integer counts and a maximum, so any order gives the sequential
  // result).  Each thread reads the channel entries it wrote itself above.
  int n_open_all = 0, n_lcc_all = 0;
  double cmax_all = 0.0;
  if (PROTO && (mode & G_PROTOCOL) && (ff || out_due)) {
    __shared__ int s_cnt[2][NT / 64];
    __shared__ double s_max[NT / 64];
    int cr = 0, cl = 0;
    double m = 0.0;
    for (int b = 0; b < nr; b += NT) {
      const int i = b + tid;
      const bool open = i < nr && d.ryr_state[i] != 0;
      cr += __builtin_popcountll(__builtin_amdgcn_ballot_w64(open));
      if (i < nr) {
        const double c = Ca[lay.ca(d.ryr_ele[i])];
        if (c > m) m = c;
      }
    }
    for (int b = 0; b < d.n_lcc; b += NT) {
      const int i = b + (NT - 1 - tid);
      const bool open = i < d.n_lcc && d.lccv_state[i] == 2 && (d.lcc_state[i] == 6 || d.lcc_state[i] == 12);
      cl += __builtin_popcountll(__builtin_amdgcn_ballot_w64(open));
    }
    for (int o = 32; o > 0; o >>= 1) {
      const double v = __shfl_xor(m, o);
      if (v > m) m = v;
    }
    const int wave = tid >> 6;
    if ((tid & 63) == 0) {
      s_cnt[0][wave] = cr;
      s_cnt[1][wave] = cl;
      s_max[wave] = m;
    }
    __syncthreads();
    if (tid == 0)
      for (int w = 0; w < NT / 64; ++w) {
        n_open_all += s_cnt[0][w];
        n_lcc_all += s_cnt[1][w];
        if (s_max[w] > cmax_all) cmax_all = s_max[w];
      }
  }

  if (tid != 0) return;
  if (swept) l.cur = cur ^ 1;
  l.step = step + 1;
  l.t = t;
  l.dt_last = dt;
  if (!PROTO || !(mode & G_PROTOCOL)) return;

  if (ff) {  // the rest of the ffwd loop body, cpu/RunSimulation.cpp:480-518
    const int n_open = n_open_all, n_open_lcc = n_lcc_all;
    const bool stop = n_open > 0 || n_open_lcc > 0 || t > P[SRS_R_T_FINAL];
    if (!stop && out_due) write_record(d, l, Ca, lay, t);
    if (d.I[SRS_I_FLAG_V_CLAMP]) l.vm = (t <= P[SRS_R_T_CLAMP]) ? P[SRS_R_V_CLAMP] : P[SRS_R_DEFAULT_VM];
    if (!stop) return;
    // The main loop starts at this t with N_RyR_Open from the last ffwd
    // count; ca_ss_max keeps its initial value.
    l.ffwd = 0;
    l.n_open_last = n_open;
  }

  // While-condition at the top of the next iteration (:522).
  const bool fid = d.I[SRS_I_FLAG_FIDELITY_SIM] != 0;
  const bool cont = t <= P[SRS_R_T_FINAL] &&
                    (!fid || ((l.lcc_open || l.n_open_last > 0 || l.ca_max_last > P[SRS_R_C_MIN]) &&
                              l.n_open_last < d.I[SRS_I_N_RYR_FIDELITY]));
  if (!cont) {
    l.done = 1;
    write_record(d, l, Ca, lay, t);  // final states output, :584
    return;
  }
  if (d.I[SRS_I_FLAG_LCC] && l.lcc_open && t >= l.t_lcc_close) {  // :525-528
    l.lcc_open = 0;
    d.lcc_state[d.I[SRS_I_LCC_INDEX]] = 1;
    s_lcc[d.I[SRS_I_LCC_INDEX]] = 0;
  }
  if (d.I[SRS_I_FLAG_V_CLAMP]) l.vm = (t <= P[SRS_R_T_CLAMP]) ? P[SRS_R_V_CLAMP] : P[SRS_R_DEFAULT_VM];  // :531-537
  const int ir = d.I[SRS_I_INIT_RYR];
  if (ir != -1 && t < P[SRS_R_INIT_RYR_HOLD] && !d.ryr_state[ir]) {  // :540-542
    d.ryr_state[ir] = s_fin[ir] = 1;
    ++n_open_all;  // counted closed above
  }
  if (out_due) {  // :552-566
    l.n_open_last = n_open_all;
    l.ca_max_last = cmax_all;
    write_record(d, l, Ca, lay, t);
  }
}

#if SRS_UNIT == 0
__global__ __launch_bounds__(GATE_THREADS) void k_gate(const RealDesc* __restrict__ D, RealLive* __restrict__ L,
                                                       uint32_t mode) {
  __shared__ int smem[GATE_LDS / sizeof(int)];
  gate_workgroup<GATE_THREADS>(D, L, blockIdx.x, mode, smem, QuadsOf{(uint32_t)D[blockIdx.x].qb});
}
// The gating of the realizations of a list (one subset of the context).
__global__ __launch_bounds__(GATE_THREADS) void k_gate_list(const RealDesc* __restrict__ D, RealLive* __restrict__ L,
                                                            const int32_t* __restrict__ rids, uint32_t mode) {
  __shared__ int smem[GATE_LDS / sizeof(int)];
  const int r = rids[blockIdx.x];
  gate_workgroup<GATE_THREADS>(D, L, r, mode, smem, QuadsOf{(uint32_t)D[r].qb});
}
#endif

// One step of a single-realization context with the previous step's gating
// folded in (cpu/RunSimulation.cpp:650-652 then :591-648).  Workgroup 0 gates
// on the state this step reads, which is the previous step's result, exactly
// as k_gate would after that step, then updates the elements that carry
// channel flux: only their rates read the channel states.  The other
// workgroups sweep the tiles without those elements.  cur, the state buffer
// this step reads, is an argument because workgroup 0 flips the live index
// while the others run.  With the loop body (PROTO, G_PROTOCOL) workgroup 0
// also changes Vm and channel states, which only the channel elements read,
// and may finish the realization: workgroups that see `done` skip their
// tile, the others write the buffer the finished realization never reads
// again.  A block starts only outside the ffwd phase, which the loop body
// can leave but not enter, so every step of it flips the live index.
// gmode 0 skips the gating (the first step of a block).
// curx: the live state index in bit 0; bit 1 set sweeps the tiles in the
// reverse order when the index is 1 (alternate steps), so that a step first
// reads the tiles the step before wrote last, while they may still be in the
// last-level cache.  The order changes no result.
template <int BS, bool NTS, bool CLASS, int QB, bool PROTO, bool PRE>
__device__ __forceinline__ void sweep_gated(const RealDesc* __restrict__ D, RealLive* __restrict__ L, int n_tiles,
                                            int curx, uint32_t gmode, const double* xo_at, double* xn_at) {
  const int cur = curx & 1;
  constexpr Quads<QB> lay;
  int b = xcd_tile(blockIdx.x, gridDim.x);
  if (b > n_tiles) return;  // b = 0: the gating workgroup; b = 1..n_tiles: tile b - 1
  if (b > 0 && curx == 3) b = n_tiles + 1 - b;
  const RealDesc& d = D[0];
  const RealLive& l = L[0];
  const int skip = l.done | l.ffwd;
  // the state buffers: X[cur] -> X[cur ^ 1], or the caller's (xo_at, xn_at)
  // (a replayed segment whose steps each have a slot of their own)
  const Bufs bf = xo_at ? Bufs{gp(xo_at), gpw(xn_at)} : bufs(d.X[0], d.X[1], cur);
  scalars_here(fold(skip, bf.xo, bf.xn) ^ geo_fold<CLASS>(d));
  if (b == 0) {
    // The channel elements: all that does not depend on the gating (every
    // species but Ca, and Ca's rate without the fluxes) is loaded, computed and
    // stored beside the gating, by wavefronts that mostly gate no channel; a
    // channel-flux element is one record instead of a search and six tables.
    // This workgroup's chain is the step of a small mesh (the tiles alone take
    // 4.7 us on 56,250 elements, an empty launch 1.6): 9.2 us with everything
    // after the gating, 6.5 with the first half ahead of the gating's first
    // barrier, which then waits for it, 5.3 with it behind that barrier; 10.1,
    // 7.8 and 7.4 on 172,494 elements.  Only its loads ahead of the barrier is no
    // faster and spills in the four-wavefront variant (5.5 and 11.9).
    int* smem = (int*)dyn_lds;
    constexpr int FIRST = BS / 4;  // the thread of channel element 0
    struct Raw { d4 m0, m1, m2, m3, m4; double tr, cs, xj, xc, a[5], v0, tt; int code, j, e0, e1; uint8_t f; };
    struct Pending { double rca, ca, B, dc, v0; int code, j, e0, e1; };
    auto load = [&](int k) -> Raw {
      const ChanElem* r = d.crec + k;
      const SRS_GLOBAL double* Xo = bf.xo;
      const size_t np = d.np;
      Raw w;
      w.f = (uint8_t)r->f;
      w.j = r->j;
      w.e0 = r->e0;
      w.e1 = r->e1;
      w.v0 = r->v0;
      w.tt = r->tt;
      w.code = r->first.code;
      for (int q = 0; q < 5; ++q) w.a[q] = r->a[q];
      w.m0 = ld_quad(Xo, lay, w.j);
      w.m1 = ld_quad(Xo, lay, r->nb[0]), w.m2 = ld_quad(Xo, lay, r->nb[1]);
      w.m3 = ld_quad(Xo, lay, r->nb[2]), w.m4 = ld_quad(Xo, lay, r->nb[3]);
      w.tr = lives_tr(w.f) ? Xo[4 * np + w.j] : 0.0;
      w.cs = lives_cs(w.f) ? Xo[5 * np + w.j] : 0.0;
      w.xj = w.xc = 0.0;
      if (w.code >= 0) w.xj = Xo[lay.ca(r->first.jsr)], w.xc = Xo[lay.ca(r->first.cyt)];
      return w;
    };
    auto half = [&](const Raw& w) -> Pending {
      Pending p{0.0, w.m0.x, 0.0, w.xj - w.xc, w.v0, w.code, w.j, w.e0, w.e1};
      Loc c;
      c.m0 = w.m0;
      c.c_tr = w.tr;
      c.c_cs = w.cs;
      c.s = w.m0 * w.a[0] + w.m1 * w.a[1] + w.m2 * w.a[2] + w.m3 * w.a[3] + w.m4 * w.a[4];
      const Rates q = elem_rates<-1>(d, l, w.j, w.f, c, w.tt, w.v0);
      elem_store<NTS, QB, -1>(d, bf, w.j, w.f, c, q);  // Ca without its fluxes: replaced by finish
      p.rca = q.ca;
      p.B = q.B;  // 1 where nothing divides
      return p;
    };
    auto is_open = [&](int code) { return code >= 0 ? smem[GATE_RYR + (code >> 1)] : smem[GATE_LCC - code - 1]; };
    auto finish = [&](const Pending& p) {
      double rca = p.rca;
      chan_flux(d, l, p.code, is_open(p.code), p.dc, p.ca, p.v0, rca);
      for (int i = p.e0 + 1; i < p.e1; ++i) {
        const ChanEntry en = d.centry[i];
        const bool open = is_open(en.code);
        const double dc = open && en.code >= 0 ? bf.xo[lay.ca(en.jsr)] - bf.xo[lay.ca(en.cyt)] : 0.0;
        chan_flux(d, l, en.code, open, dc, p.ca, p.v0, rca);
      }
      rca /= p.B;
      bf.xn[lay.ca(p.j)] = p.ca + rca * d.P[SRS_R_T_STEP];
    };
    const int k0 = ((int)threadIdx.x + BS - FIRST) % BS;
    const bool pre = PRE && !skip && k0 < d.n_celem;
    Pending p0;
    auto mid = [&] {
      if (pre) p0 = half(load(k0));
    };
    if (gmode) {
      gate_workgroup<BS, PROTO>(D, L, 0, gmode, smem, lay, mid);
    } else {
      for (int i = threadIdx.x; i < d.n_ryr; i += BS) smem[GATE_RYR + i] = d.ryr_state[i];
      held_lccs<BS>(d, smem);
      mid();
    }
    __syncthreads();  // the new channel states, written by this workgroup, before the flux reads them
    if (skip) return;
    if (pre) finish(p0);
    for (int k = PRE ? k0 + BS : k0; k < d.n_celem; k += BS) finish(half(load(k)));
    return;
  }
  if (skip) return;
  sweep_tile<BS, NTS, CLASS, QB, true>(d, l, bf, b - 1, nullptr);
}
// W: the register budget, at least W wavefronts per SIMD.
template <int BS, bool NTS, bool CLASS, int QB, bool PROTO, bool PRE, int W>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(W))) void k_sweep_gated(
    const RealDesc* __restrict__ D, RealLive* __restrict__ L, int n_tiles, int cur, uint32_t gmode,
    const double* xo_at, double* xn_at) {
  sweep_gated<BS, NTS, CLASS, QB, PROTO, PRE>(D, L, n_tiles, cur, gmode, xo_at, xn_at);
}

// ------------------------------------------------------------ kernel choice
// The sweep kernels are instantiated in five compilation units of this file
// (SRS_UNIT 0: host code and the gating kernel; 1: the sweeps; 2, 3, 4: the
// gated sweeps of 128-, 256- and 512-element tiles), which the build
// compiles in parallel.

using SweepFn = void (*)(const RealDesc*, const RealLive*, const int2*, int, int, ReplayAt);
using GatedFn = void (*)(const RealDesc*, RealLive*, int, int, uint32_t, const double*, double*);
SweepFn pick_sweep(const srs_ctx* c, bool replay = false);
template <int BS>
GatedFn pick_gated_bs(const srs_ctx* c, bool proto);

#if SRS_UNIT == 1
template <int BS, bool CMP, bool REPLAY>
SweepFn pick_nt(const srs_ctx* c) {
  if (c->quad_block == 1) return c->nt_state ? k_sweep<BS, true, CMP, 1, REPLAY> : k_sweep<BS, false, CMP, 1, REPLAY>;
  return c->nt_state ? k_sweep<BS, true, CMP, 64, REPLAY> : k_sweep<BS, false, CMP, 64, REPLAY>;
}

template <bool CMP, bool REPLAY>
SweepFn pick_tile(const srs_ctx* c) {
  switch (c->tile) {
    case 128: return pick_nt<128, CMP, REPLAY>(c);
    case 256: return pick_nt<256, CMP, REPLAY>(c);
    default: return pick_nt<512, CMP, REPLAY>(c);
  }
}

SweepFn pick_sweep(const srs_ctx* c, bool replay) {
  if (replay) return c->class_all ? pick_tile<true, true>(c) : pick_tile<false, true>(c);
  return c->class_all ? pick_tile<true, false>(c) : pick_tile<false, false>(c);
}
#endif  // SRS_UNIT == 1

#if SRS_UNIT >= 2
template <int BS, bool CMP, bool PROTO, bool PRE, int W>
GatedFn pick_gated_nt(const srs_ctx* c) {
  if (c->quad_block == 1)
    return c->nt_state ? k_sweep_gated<BS, true, CMP, 1, PROTO, PRE, W> : k_sweep_gated<BS, false, CMP, 1, PROTO, PRE, W>;
  return c->nt_state ? k_sweep_gated<BS, true, CMP, 64, PROTO, PRE, W> : k_sweep_gated<BS, false, CMP, 64, PROTO, PRE, W>;
}

// How much the registers of the gating workgroup may cost the tiles.  With no
// more tiles than CUs (256), each workgroup has a CU to itself: no budget
// (56,250 elements: 5.3 us per step).  Then four wavefronts, with the first half
// of its channel elements behind the gating's first barrier, while the gating
// workgroup is the longest one; beyond, the tiles' own wavefronts decide: six,
// the gating's registers spilled and its channel elements updated after it.  us
// per step with four / six, RCM, block and Morton order: 354,816 elements
// 12.5 / 13.2, -, 10.3 / 13.3; 638,262 18.8 / 17.4, 17.2 / 16.2, 15.9 / 16.8;
// 703,452 19.9 / 18.5, 18.4 / 17.2, 17.2 / 17.1; 750,708 20.7 / 19.3, 19.1 /
// 17.8, 17.5 / 17.5; with rows that all differ 704,184 22.1 / 20.7, 21.0 / 19.6,
// 19.6 / 18.5.  The line is where six are slower in no order.
template <int BS, bool CMP, bool PROTO>
GatedFn pick_gated_w(const srs_ctx* c) {
  if (c->occ || (int64_t)c->n_tiles * BS >= 700000) return pick_gated_nt<BS, CMP, PROTO, false, 6>(c);
  return c->n_tiles <= 256 ? pick_gated_nt<BS, CMP, PROTO, true, 2>(c)
                           : pick_gated_nt<BS, CMP, PROTO, true, 4>(c);
}

template <int BS>
GatedFn pick_gated_bs(const srs_ctx* c, bool proto) {
  if (c->class_all) return proto ? pick_gated_w<BS, true, true>(c) : pick_gated_w<BS, true, false>(c);
  return proto ? pick_gated_w<BS, false, true>(c) : pick_gated_w<BS, false, false>(c);
}
// one tile size per unit: 128 in unit 2, 256 in unit 3, 512 in unit 4
template GatedFn pick_gated_bs<SRS_UNIT == 2 ? 128 : SRS_UNIT == 3 ? 256 : 512>(const srs_ctx*, bool);
#endif  // SRS_UNIT >= 2

#if SRS_UNIT == 0
// Ends a block of m replayed steps of the listed realizations from schedule row
// `row`: time, step and live index, and the RyR states of the row after it, as m
// gating launches leave them.
__global__ __launch_bounds__(64) void k_replay_end(const RealDesc* __restrict__ D, RealLive* __restrict__ L,
                                                   const int32_t* __restrict__ rid, int64_t m, int64_t row) {
  const int r = rid[blockIdx.x];
  const RealDesc& d = D[r];
  RealLive& l = L[r];
  const int64_t k = row + m < d.n_sched ? row + m : d.n_sched - 1;
  for (int i = threadIdx.x; i < d.n_ryr; i += 64) d.ryr_state[i] = d.sched[k * d.n_ryr + i];
  if (threadIdx.x != 0) return;
  const double dt = d.P[SRS_R_T_STEP];
  double t = l.t;
  for (int64_t q = 0; q < m; ++q) t += dt;
  l.t = t;
  l.dt_last = dt;
  l.step += m;
  l.cur ^= (int)(m & 1);
}

// Gathers Ca at the channel elements of one realization.
__global__ void k_channel_ca(const RealDesc* __restrict__ D, const RealLive* __restrict__ L, int r, double* out) {
  const RealDesc& d = D[r];
  const double* Ca = d.X[L[r].cur];  // Ca of element e at Ca[lay.ca(e)]
  const QuadsOf lay{(uint32_t)d.qb};
  for (int i = threadIdx.x; i < d.n_ryr; i += blockDim.x) {
    out[i] = Ca[lay.ca(d.ryr_ele[i])];
    out[d.n_ryr + i] = Ca[lay.ca(d.ryr_jsr[i])];
  }
  for (int i = threadIdx.x; i < d.n_lcc; i += blockDim.x) out[2 * d.n_ryr + i] = Ca[lay.ca(d.lcc_ele[i])];
}


// Moves a run [t0, t0 + cnt) of one realization's fields between its state
// buffers and a staging buffer in the caller's layout, [6][n] in the reference
// numbering (inv: reference -> device position).  to_dev writes both
// ping-pong buffers; otherwise the live one is read.  Bound by the host link:
// the kernel's scattered side is the elements' pairs (each read for two of the
// six species, the repeats from L2), the staging side is contiguous.
__global__ __launch_bounds__(256) void k_state_xfer(const RealDesc* __restrict__ D, const RealLive* __restrict__ L,
                                                    int r, const int32_t* __restrict__ inv, double* __restrict__ stage,
                                                    size_t t0, size_t cnt, int to_dev) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= cnt) return;
  const RealDesc& d = D[r];
  const size_t t = t0 + i, n = d.n;
  const int s = (int)(t / n);
  const size_t x = xoff(QuadsOf{(uint32_t)d.qb}, s, inv[t - s * n], d.np);
  if (to_dev) {
    const double v = stage[i];
    d.X[0][x] = v;
    d.X[1][x] = v;
  } else {
    stage[i] = d.X[L[r].cur][x];
  }
}

// ----------------------------------------------------------------- host side

// Rounds the significand to 40 bits, ties to even (class key of a coefficient).
double quantize(double a) {
  uint64_t u;
  memcpy(&u, &a, 8);
  const uint64_t e = u >> 52 & 0x7ff;
  if (e != 0 && e < 0x7fe) {  // normal, and so after a carry: 13 bits go
    u = (u + 0xfff + (u >> 13 & 1)) & ~(uint64_t)0x1fff;
    memcpy(&a, &u, 8);
    return a;
  }
  if (a == 0.0 || !std::isfinite(a)) return a;
  int x;
  const double m = std::frexp(a, &x);
  return std::ldexp(std::nearbyint(std::ldexp(m, 40)), x - 40);
}

// Each coefficient row as a class row plus int16 deltas of the bit patterns.
// class_rows stays false unless every row of the mesh is reproduced exactly,
// and where classes are hardly fewer than rows (an irregular mesh), so that
// the table would be as much to read as the rows.
void build_class_rows(HostMesh& hm) {
  const int n = hm.n, np = hm.np;
  struct Hash {
    size_t operator()(const std::array<double, 5>& k) const {
      uint64_t h = 0;
      for (double v : k) {
        uint64_t u;
        memcpy(&u, &v, 8);
        h = (h ^ u) * 0x9E3779B97F4A7C15ull;
        h ^= h >> 32;
      }
      return h;
    }
  };
  std::unordered_map<std::array<double, 5>, int, Hash> classes;
  std::vector<uint32_t> row(3 * (size_t)np + 1, 0);
  // A regular mesh's few classes are found again without rounding and comparing: a
  // value less than half a rounding interval from a class's (12 bits; equal to a
  // zero) rounds to it.
  struct Seen { int64_t t[5], tol[5]; int id; };
  std::vector<Seen> seen(512, Seen{{}, {}, -1});
  for (int k = 0; k < n; ++k) {
    int64_t u[5], d[5];
    for (int q = 0; q < 5; ++q) memcpy(&u[q], &hm.coef[(size_t)q * np + k], 8);
    uint64_t h = 0;
    for (int q = 0; q < 5; ++q) h += (((uint64_t)u[q] + 4096) >> 13) * (2 * q + 1);
    Seen& sn = seen[h * 0x9E3779B97F4A7C15ull >> 55];
    int id = sn.id;
    bool same = id >= 0;
    for (int q = 0; q < 5; ++q) {
      d[q] = (int64_t)((uint64_t)u[q] - (uint64_t)sn.t[q]);  // as the kernel adds it back, for any pair of patterns
      same &= (uint64_t)d[q] + (uint64_t)sn.tol[q] <= 2 * (uint64_t)sn.tol[q];
    }
    if (!same) {
      std::array<double, 5> key;
      Seen cls;
      bool normal = true;
      for (int q = 0; q < 5; ++q) {
        const double a = hm.coef[(size_t)q * np + k];
        if (!std::isfinite(a) || (a == 0.0 && std::signbit(a))) return;  // the classes are keyed by value
        key[q] = quantize(a);
        memcpy(&cls.t[q], &key[q], 8);
        d[q] = u[q] - cls.t[q];
        if (d[q] < -32768 || d[q] > 32767) return;
        const int e = (int)(cls.t[q] >> 52 & 0x7ff);
        cls.tol[q] = cls.t[q] == 0 ? 0 : 4095;
        normal &= cls.t[q] == 0 || (e != 0 && e < 0x7fe);
      }
      auto it = classes.find(key);
      if (it == classes.end()) {
        if (classes.size() >= 65535 || (classes.size() >= 8192 && 2 * classes.size() > (size_t)k)) return;
        it = classes.emplace(key, (int)classes.size()).first;
      }
      cls.id = id = it->second;
      if (normal) sn = cls;
    }
    auto w = [](int64_t v) { return (uint32_t)(uint16_t)v; };
    row[3 * (size_t)k] = (uint32_t)id | w(d[0]) << 16;
    row[3 * (size_t)k + 1] = w(d[1]) | w(d[2]) << 16;
    row[3 * (size_t)k + 2] = w(d[3]) | w(d[4]) << 16;
  }
  hm.n_class = (int)classes.size();
  hm.tab.resize(5 * (size_t)hm.n_class);
  for (auto& kv : classes)
    for (int q = 0; q < 5; ++q) hm.tab[5 * (size_t)kv.second + q] = kv.first[q];
  hm.row.swap(row);
  hm.class_rows = true;
}

// Where the neighbours of a mesh's elements are, for `tile` elements per tile,
// on the host.
struct HostMap {
  int tile = 0, qcap = 0;      // as in TileMap
  std::vector<uint32_t> hal;
  std::vector<uint16_t> loc;
  std::vector<int32_t> hoff;
  // Cache lines that the halos cost more with blocks of 64 (two for up to eight
  // neighbours that follow each other, one in each half) than with an element's
  // species side by side (one for up to four), of all tiles.
  int64_t lines = 0;
};

// Halos are sorted, so that a wavefront's loads of them fall in runs.  The
// elements that a tile needs are bits of a bitmap, its own all set, and an
// element's place is the rank of its bit: no branch per neighbour.  From 128k
// elements up, runs of tiles on several threads (below, a thread costs more to
// start than its tiles take).
int make_map(const HostMesh& hm, int tile, HostMap* m) {
  const int n = hm.n, np = hm.np, nt = (n + tile - 1) / tile;
  const int n_run = n < 1 << 17 ? 1 : std::min(nt, 32);
  m->tile = tile;
  m->lines = 0;
  m->loc.assign(4 * (size_t)np, 0);
  m->hoff.assign(nt + 1, 0);
  std::vector<std::vector<uint32_t>> halos(n_run);
  std::vector<int64_t> lines(n_run, 0);
  static_assert(MAX_TILE % 64 == 0, "tiles are whole words of the bitmap");
  const bool ok = each_chunk(n_run, [&](int q) {
    std::vector<uint32_t>& hal = halos[q];
    std::vector<uint64_t> bits((size_t)np / 64, 0);
    std::vector<int32_t> rank(bits.size()), words;
    int64_t more = 0;
    const int t0 = (int)((int64_t)nt * q / n_run), t1 = (int)((int64_t)nt * (q + 1) / n_run);
    for (int t = t0; t < t1; ++t) {
      const int j0 = t * tile, j1 = std::min(n, j0 + tile);
      const int w0 = j0 / 64, w1 = std::min(w0 + tile / 64, np / 64);
      for (int w = w0; w < w1; ++w) {
        bits[w] = ~0ull;
        rank[w] = 64 * (w - w0);
      }
      words.clear();
      const uint32_t *nb0 = hm.nbr.data() + 4 * (size_t)j0, *nb1 = hm.nbr.data() + 4 * (size_t)j1;
      for (const uint32_t* p = nb0; p < nb1; ++p) {
        const uint32_t e = idx_of(*p);
        uint64_t& w = bits[e >> 6];
        if (!w) words.push_back((int32_t)(e >> 6));
        w |= 1ull << (e & 63);
      }
      std::sort(words.begin(), words.end());
      const size_t h0 = hal.size();
      for (int w : words) {
        rank[w] = tile + (int)(hal.size() - h0);
        uint64_t four = bits[w] | bits[w] >> 1;
        four = (four | four >> 2) & 0x1111111111111111ull;  // any of four neighbours in a row
        more += 2 * __builtin_popcountll((four | four >> 4) & 0x0101010101010101ull) - __builtin_popcountll(four);
        for (uint64_t b = bits[w]; b; b &= b - 1) {
          const int e = 64 * w + __builtin_ctzll(b);
          hal.push_back((uint32_t)e | ((hm.flags[e] & F_SL) ? IDX_SL : 0u));
        }
      }
      m->hoff[t + 1] = (int32_t)(hal.size() - h0);
      uint16_t* loc = m->loc.data() + 4 * (size_t)j0;
      for (const uint32_t* p = nb0; p < nb1; ++p) {
        const uint32_t e = idx_of(*p);
        *loc++ = (uint16_t)(rank[e >> 6] + __builtin_popcountll(bits[e >> 6] & ((1ull << (e & 63)) - 1)));
      }
      for (int w : words) bits[w] = 0;
      for (int w = w0; w < w1; ++w) bits[w] = 0;
    }
    lines[q] = more;
  });
  if (!ok) return srs::fail(SRS_E_STATE, "out of host memory for the tile map");
  int64_t total = 0;
  int h_max = 0;
  for (int t = 0; t < nt; ++t) {
    h_max = std::max(h_max, (int)m->hoff[t + 1]);
    total += m->hoff[t + 1];
    if (total > INT32_MAX) return srs::fail(SRS_E_ARG, "mesh too large for its halo lists");
    m->hoff[t + 1] = (int32_t)total;
  }
  m->hal.clear();
  if (n_run == 1) m->hal.swap(halos[0]);
  else {
    m->hal.reserve(total + 1);
    for (const auto& h : halos) m->hal.insert(m->hal.end(), h.begin(), h.end());
  }
  if (m->hal.empty()) m->hal.push_back(0);
  for (int64_t l : lines) m->lines += l;
  m->qcap = tile + h_max;
  return SRS_OK;
}

// The maps of every mesh for the context's tile, which is chosen here with the
// state layout unless SRS_TUNE_TILE gave one.
//
// Layout: blocks of 64, or an element's species side by side where the halos of
// an average element cost half a cache line less with it.  us per step, blocks of
// 64 / 1 (lines): 927,816 elements in Morton order 20.4 / 22.5 (0.17), with 5% of
// the elements anywhere 25.5 / 25.3 (0.41), 8% 29.2 / 26.8 (0.55), 10% 32.1 / 27.7
// (0.65), in shuffled runs of 32 41.7 / 34.7 (0.58); 2,952,000 with 5% 76.0 / 83.5
// (0.41), 8% 87.0 / 87.5 (0.56), 10% 96.2 / 90.1, all 436 / 250, runs of 32 127 /
// 102; four members of 56,250 with 5% 14.9 / 13.4, 10% 16.8 / 14.0, runs of 32
// 18.2 / 16.1; eight of 15,360 with 15% 13.6 / 10.9.  One realization of up to
// 32,768 elements, whose states stay in the L2s, gains later: 15,360 with 15% 5.8 /
// 6.5 (0.59), 30% 6.6 / 6.5 (1.01), all 7.0 / 6.6; 28,800 with 15% 6.3 / 6.5 (0.73),
// 30% 7.1 / 6.5 (1.28).
//
// Tile: 512 elements share the most neighbours inside a tile (halos of 1.4
// elements per element in the block order, 0.6 in the Morton order, 2.0 in RCM;
// 1.9, 0.8 and 2.1 with 256) and are the fastest while three workgroups share a
// CU: 2,952,000 elements 61.6 us per step in the block order, 64.2 with 256, 59.2
// and 60.8 in the Morton order; a hundred 56,250-element members 111 and 128.
// The staged quads of the worst tile decide that.  In a breadth-first order of
// the 2,952,000 they pass a third of the LDS, and 256 elements take 70.3 us
// against 77.0 (rows that all differ: 77.7 against 86.1), of 3,930,960 93.8
// against 102.6; with runs of 64 elements of the block order shuffled, 927,816
// take 38.6 against 47.9.
// Several realizations with no more tiles than CUs (256) take the smallest such
// tile: each has a CU to itself, and what it waits for is its own chain of loads
// and barriers.  us per step with 128 / 256 / 512: two members of 3,600 elements
// 10.3 / 10.9 / 11.5, eight 10.6 / 11.0 / 11.7, eight of 8,112 (512, 256 and 128
// tiles) 10.9 / 10.9 / 11.3, of 15,360 (960, 480, 240) 11.2 / 11.4 / 11.3.
// Scattered orders have no neighbours to share: there 128 is the fastest (us per
// step with 128 / 512 elements shuffled: 2,952,000 250 / 290, sixteen members of
// 172,494 131 / 144, 172,494 13.7 / 15.3).
int plan_tiles(srs_ctx* c, std::vector<HostMap>* maps) {
  maps->resize(c->meshes.size());
  auto make = [&](int tile) {
    c->tile = tile;
    for (size_t k = 0; k < maps->size(); ++k)
      if (int rc = make_map(*c->meshes[k], tile, &(*maps)[k])) return rc;
    return (int)SRS_OK;
  };
  auto one_each = [&](int tile) {
    int64_t nt = 0;
    for (const HostReal& hr : c->reals) nt += (c->meshes[hr.mesh]->n + tile - 1) / tile;
    return c->reals.size() > 1 && nt <= 256;
  };
  int rc = make(c->tile_set ? c->tile_set : one_each(128) ? 128 : one_each(256) ? 256 : 512);
  if (rc) return rc;
  double lines = 0.0, n = 0.0;
  int qcap = 0;
  for (const HostReal& hr : c->reals) {
    lines += (double)(*maps)[hr.mesh].lines;
    n += c->meshes[hr.mesh]->n;
  }
  for (const HostMap& m : *maps) qcap = std::max(qcap, m.qcap);
  c->quad_block = lines > (c->reals.size() == 1 && n <= 1 << 15 ? 1.0 : 0.5) * n ? 1 : 64;
  if (c->tile_set || c->tile == 128) return SRS_OK;
  if (c->quad_block == 1) return make(128);
  // a CU's 160 KB in granules of 1280 B, 42 for each of three workgroups; the
  // gated sweep has 256 or 384 B of its own
  const size_t lds = 4 * sizeof(double) * (size_t)qcap + (c->reals.size() == 1 && c->gated ? 384 : 0);
  return c->tile == 512 && lds > 42 * 1280 ? make(256) : (int)SRS_OK;
}

// Small tables in one device allocation and one copy (an allocation and a copy
// of each took 10 us); larger ones get their own.  The pointers are set by
// upload().
class Pack {
 public:
  explicit Pack(srs_ctx* c) : c_(c) {}
  template <class T>
  int add(T** p, const std::vector<T>& v) {
    const size_t bytes = v.size() * sizeof(T), at = (host_.size() + 255) / 256 * 256;
    if (bytes == 0 || bytes > (size_t)1 << 18) return dev_upload(c_, p, v);
    host_.resize(at + bytes);
    memcpy(host_.data() + at, v.data(), bytes);
    set_.push_back([p, at](char* base) { *p = (T*)(base + at); });
    return SRS_OK;
  }
  int upload() {
    char* base;
    if (int rc = dev_upload(c_, &base, host_)) return rc;
    for (const auto& s : set_) s(base);
    return SRS_OK;
  }

 private:
  srs_ctx* c_;
  std::vector<char> host_;
  std::vector<std::function<void(char*)>> set_;
};

// The tables of a mesh on the device.
int upload_mesh(srs_ctx* c, HostMesh& hm, const HostMap& m) {
  // the meshes' channel flags were set by add_realization: what blocks hold
  std::vector<uint32_t> blk(hm.np / 64, 0);
  for (size_t b = 0; b < blk.size(); ++b) {
    bool plain = true;
    for (size_t k = 64 * b; k < std::min<size_t>(64 * b + 64, hm.n); ++k) plain &= hm.flags[k] == F_TROPC;
    if (plain) blk[b] |= BLK_PLAIN;
  }
  TileMap& t = hm.map;
  t.tile = m.tile;
  t.qcap = m.qcap;
  t.n_halo = m.hoff.back();
  Pack pk(c);
  int rc;
  if ((rc = pk.add(&hm.d_nbr, hm.nbr)) || (rc = pk.add(&hm.d_blk, blk)) || (rc = pk.add(&t.d_loc, m.loc)) ||
      (rc = pk.add(&t.d_hal, m.hal)) || (rc = pk.add(&t.d_hoff, m.hoff)))
    return rc;
  if (c->class_all ? (rc = pk.add(&hm.d_row, hm.row)) || (rc = pk.add(&hm.d_tab, hm.tab))
                   : (rc = pk.add(&hm.d_coef, hm.coef)))
    return rc;
  if ((rc = pk.add(&hm.d_flags, hm.flags)) || (rc = pk.add(&hm.d_inv, hm.inv)) || (rc = pk.add(&hm.d_V0, hm.V0)) ||
      (rc = pk.add(&hm.d_tt, hm.tt)) || (rc = pk.add(&hm.d_br, hm.br)))
    return rc;
  return pk.upload();
}

// cpu/RunSimulation.cpp:85-88, the parts that depend on CaNSR only.
void serca_terms(double nsr, const double* P, double* out) {
  double K_sr = nsr / P[SRS_R_K_D_SR];
  K_sr = K_sr * K_sr;
  out[0] = 0.104217 + 17.923 * K_sr;
  out[1] = 1.75583e6 + K_sr * 7.61673e6;
  out[2] = 6.08463e11 + K_sr * 4.50544e11;
  out[3] = 9.17846e6 - 11478.2 * K_sr;
  out[4] = 0.329904 * K_sr;
}

int check_real(srs_ctx* c, int32_t r) {
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (!c->finalized) return srs::fail(SRS_E_STATE, "context not finalized");
  if (r < 0 || r >= (int32_t)c->reals.size()) return srs::fail(SRS_E_ARG, "realization %d out of range", r);
  return SRS_OK;
}

void launch_sweep(srs_ctx* c) {
  if (c->grid_sweep == 0) return;  // every realization has finished
  // one realization: tile b is tile b of realization 0, no table lookups
  const int single = c->reals.size() == 1 ? 1 : 0;
  hipLaunchKernelGGL(pick_sweep(c), dim3(c->grid_sweep), dim3(c->tile), c->sweep_lds, c->stream, c->d_desc, c->d_live,
                     c->d_tiles, c->n_tiles, single, ReplayAt{});
}

// One replayed step of the tile list (ReplayAt), and m of them with the live
// state brought up to date.
void launch_replay(srs_ctx* c, int64_t row, int par, const double* xo, double* xn, size_t stride, int n_tiles) {
  if (c->grid_sweep == 0) return;
  hipLaunchKernelGGL(pick_sweep(c, true), dim3(c->grid_sweep), dim3(c->tile), c->sweep_lds, c->stream, c->d_desc,
                     c->d_live, c->d_tiles, c->n_tiles, c->reals.size() == 1 ? 1 : 0,
                     (ReplayAt{row, xo, xn, stride, par, n_tiles}));
}
void launch_replay_block(srs_ctx* c, int64_t m, int64_t row, const int32_t* rid, int n_rid) {
  for (int64_t k = 0; k < m; ++k) launch_replay(c, row + k, (int)(k & 1));
  hipLaunchKernelGGL(k_replay_end, dim3(n_rid), dim3(64), 0, c->stream, c->d_desc, c->d_live, rid, m, row);
}

// m steps of every subset, one subset after another: the sweep over the
// subset's run of tiles and the gating of its realizations, m times.
// Realizations are independent and each one's Philox counters follow its own
// step count, so the order changes no result.
void launch_subset_block(srs_ctx* c, int64_t m, uint32_t gmode) {
  for (const srs_ctx::Subset& sb : c->subsets)
    for (int64_t k = 0; k < m; ++k) {
      if (sb.nt > 0)
        hipLaunchKernelGGL(pick_sweep(c), dim3((sb.nt + NXCD - 1) / NXCD * NXCD), dim3(c->tile), c->sweep_lds, c->stream,
                           c->d_desc, c->d_live, c->d_tiles + sb.t0, sb.nt, 0, ReplayAt{});
      hipLaunchKernelGGL(k_gate_list, dim3((unsigned)sb.nr), dim3(GATE_THREADS), 0, c->stream, c->d_desc, c->d_live,
                         (const int32_t*)c->d_sub_rids + sb.r0, gmode);
    }
}

// Splits the current tile list into subsets: runs of whole bands (in list
// order) whose realizations' state buffers (two of 48 B per element each)
// take at most subset_mb MB; realizations whose bands have no tile left
// (all finished) are gated with the last subset, as k_gate would.
int plan_subsets(srs_ctx* c) {
  c->subsets.clear();
  c->subsets_valid = true;
  if (c->subset_mb <= 0 || c->reals.size() < 2) return SRS_OK;
  const size_t budget = (size_t)c->subset_mb << 20;
  auto band_of = [&](int t) { return c->reals[c->tiles_cur[t].x].band; };
  std::vector<int32_t> rids;
  std::vector<char> listed(c->reals.size(), 0);
  srs_ctx::Subset cur{0, 0, 0, 0};
  size_t bytes = 0;
  const int n = (int)c->tiles_cur.size();
  for (int t = 0; t < n;) {
    const int g = band_of(t);
    int t1 = t;
    while (t1 < n && band_of(t1) == g) ++t1;
    size_t gb = 0;
    for (int r : c->bands[g]) gb += 2 * 48 * (size_t)c->meshes[c->reals[r].mesh]->np;
    if (cur.nt > 0 && bytes + gb > budget) {
      c->subsets.push_back(cur);
      cur = srs_ctx::Subset{t, 0, (int)rids.size(), 0};
      bytes = 0;
    }
    for (int r : c->bands[g])
      if (!listed[r]) {
        listed[r] = 1;
        rids.push_back(r);
        cur.nr++;
      }
    cur.nt += t1 - t;
    bytes += gb;
    t = t1;
  }
  for (size_t r = 0; r < c->reals.size(); ++r)
    if (!listed[r]) {
      rids.push_back((int32_t)r);
      cur.nr++;
    }
  if (cur.nt > 0 || cur.nr > 0) c->subsets.push_back(cur);
  if (c->subsets.size() < 2) {  // one subset is the whole context: the plain step is the same launches
    c->subsets.clear();
    return SRS_OK;
  }
  HIPCHK(hipMemcpy(c->d_sub_rids, rids.data(), rids.size() * sizeof(int32_t), hipMemcpyHostToDevice));
  return SRS_OK;
}

int launch_step(srs_ctx* c, uint32_t gmode) {
  launch_sweep(c);
  hipLaunchKernelGGL(k_gate, dim3((unsigned)c->reals.size()), dim3(GATE_THREADS), 0, c->stream, c->d_desc,
                     c->d_live, gmode);
  return SRS_OK;
}

// One step through k_sweep_gated: tile b - 1 in workgroup b, workgroup 0
// gates (gmode) and updates the channel elements.  proto picks the kernel
// with the loop body.
void launch_gated(srs_ctx* c, int cur, uint32_t gmode, bool proto, const double* xo_at, double* xn_at) {
  const GatedFn f = c->tile == 128 ? pick_gated_bs<128>(c, proto)
                    : c->tile == 512 ? pick_gated_bs<512>(c, proto) : pick_gated_bs<256>(c, proto);
  const int grid = (c->n_tiles + 1 + NXCD - 1) / NXCD * NXCD;
  hipLaunchKernelGGL(f, dim3(grid), dim3(c->tile), std::max(c->sweep_lds, GATE_LDS), c->stream, c->d_desc, c->d_live, c->n_tiles,
                     cur | (c->alt_order ? 2 : 0), gmode, xo_at, xn_at);
}

// The gating of a single realization's last gated step (k_gate alone).
void launch_gate_single(srs_ctx* c, uint32_t gmode) {
  hipLaunchKernelGGL(k_gate, dim3(1), dim3(GATE_THREADS), 0, c->stream, c->d_desc, c->d_live, gmode);
}

// m steps through k_sweep_gated: the first without gating (nothing is
// pending when a block starts), each later one gating the step before it,
// then k_gate for the last step, so that a block leaves no gating pending.
// cur is the live state index when the block starts; gmode is the step's
// gating mode (G_AFTER_SWEEP, with G_PROTOCOL for the loop body).
void launch_gated_block(srs_ctx* c, int64_t m, int cur, uint32_t gmode) {
  const bool proto = (gmode & G_PROTOCOL) != 0;
  for (int64_t k = 0; k < m; ++k) launch_gated(c, cur ^ (int)(k & 1), k ? gmode : 0u, proto);
  launch_gate_single(c, gmode);
}

// Captured step blocks hold the sweep's tile list and grid; they are dropped
// when either changes.
int drop_graphs(srs_ctx* c) {
  HIPCHK(hipStreamSynchronize(c->stream));
  for (auto& kv : c->graphs) (void)hipGraphExecDestroy(kv.second);
  c->graphs.clear();
  return SRS_OK;
}

void set_tiles(srs_ctx* c, int2* d, int n) {
  c->d_tiles = d;
  c->n_tiles = n;
  c->grid_sweep = (n + NXCD - 1) / NXCD * NXCD;
  c->subsets_valid = false;
}

// The full tile list again, before the host changes live state (a finished
// realization may be restarted).
int tiles_full(srs_ctx* c) {
  if (!c->tiles_compacted) return SRS_OK;
  int rc = drop_graphs(c);
  if (rc) return rc;
  set_tiles(c, c->d_tiles_all, (int)c->tiles_all.size());
  c->tiles_cur = c->tiles_all;
  c->tiles_compacted = false;
  return SRS_OK;
}

// A tile whose realizations have all finished still costs the sweep about
// what a live one does (its workgroup is dispatched, reads the tile table and
// the done flags, and exits), so once such tiles make up an eighth of the
// list the sweep gets a list without them.  A finished realization stays
// finished until the host changes its live state, which puts the full list
// back (tiles_full).
int tiles_compact(srs_ctx* c) {
  const int n_real = (int)c->reals.size();
  if (n_real < 2 || !c->drop_finished) return SRS_OK;
  HIPCHK(hipStreamSynchronize(c->stream));
  std::vector<RealLive> lv(n_real);
  HIPCHK(hipMemcpy(lv.data(), c->d_live, n_real * sizeof(RealLive), hipMemcpyDeviceToHost));
  std::vector<int2> t;
  for (const int2& x : c->tiles_all)
    if (!lv[x.x].done) t.push_back(x);
  if ((int64_t)t.size() == c->n_tiles || (int64_t)t.size() * 8 > (int64_t)c->n_tiles * 7) return SRS_OK;
  int rc = drop_graphs(c);
  if (rc) return rc;
  if (!t.empty()) HIPCHK(hipMemcpy(c->d_tiles_live, t.data(), t.size() * sizeof(int2), hipMemcpyHostToDevice));
  set_tiles(c, c->d_tiles_live, (int)t.size());
  c->tiles_cur = t;
  c->tiles_compacted = true;
  return SRS_OK;
}


// Host copies of a transfer's parts by several threads: one thread's copy into
// fresh pages, not the link, bounded a transfer (15 GB/s).  The threads live
// for one transfer; with none (too small a transfer, or none to be had) the
// caller copies alone.
class CopyTeam {
 public:
  explicit CopyTeam(int helpers) {
    try {
      for (int k = 0; k < helpers; ++k) th_.emplace_back([this, k] { work(k + 1); });
    } catch (...) {  // fewer threads than asked for
    }
    n_ = (int)th_.size();
  }
  ~CopyTeam() {
    stop_ = true;
    go_.fetch_add(1, std::memory_order_release);
    for (std::thread& t : th_) t.join();
  }
  CopyTeam(const CopyTeam&) = delete;
  CopyTeam& operator=(const CopyTeam&) = delete;
  void copy(void* dst, const void* src, size_t bytes) {
    dst_ = (char*)dst;
    src_ = (const char*)src;
    bytes_ = bytes;
    parts_ = n_ + 1;
    left_.store(n_, std::memory_order_relaxed);
    go_.fetch_add(1, std::memory_order_release);
    slice(0);
    while (left_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
  }

 private:
  void slice(int k) {
    const size_t lo = bytes_ / 64 * k / parts_ * 64, hi = k + 1 == parts_ ? bytes_ : bytes_ / 64 * (k + 1) / parts_ * 64;
    memcpy(dst_ + lo, src_ + lo, hi - lo);
  }
  void work(int k) {
    for (unsigned seen = 0;;) {
      unsigned g;
      while ((g = go_.load(std::memory_order_acquire)) == seen) std::this_thread::yield();
      seen = g;
      if (stop_) return;
      slice(k);
      left_.fetch_sub(1, std::memory_order_release);
    }
  }
  std::vector<std::thread> th_;
  int n_ = 0, parts_ = 1;
  std::atomic<unsigned> go_{0};
  std::atomic<int> left_{0};
  std::atomic<bool> stop_{false};
  char* dst_ = nullptr;
  const char* src_ = nullptr;
  size_t bytes_ = 0;
};

// Copies one realization's fields between the caller's array ([6][n], reference
// numbering) and its state buffers in parts, through two pinned host buffers
// that the reordering kernel writes (or reads) over the link while the host
// copies the part before.  On the 3M-element dyad a host loop over the same
// elements, with its own 142 MB copy of the fields, took 75 ms to read and 70
// ms to set; one device staging buffer and plain copies 9.4 and 5.4; this 4.3
// and 3.2.
int state_xfer(srs_ctx* c, int32_t r, double* host, bool to_dev) {
  const HostMesh& hm = *c->meshes[c->reals[r].mesh];
  const size_t total = 6 * (size_t)hm.n, part = c->stage_len;
  const int n_parts = (int)((total + part - 1) / part);
  // helper threads from 4 MB up (3M-element dyad, read: none 6.8 ms, one 4.6,
  // three 4.3, five 4.4)
  CopyTeam team(total >= (size_t)1 << 19 ? 3 : 0);
  auto len = [&](int i) { return std::min(part, total - part * (size_t)i); };
  auto launch = [&](int i) -> int {
    hipLaunchKernelGGL(k_state_xfer, dim3((unsigned)((len(i) + 255) / 256)), dim3(256), 0, c->stream, c->d_desc,
                       c->d_live, r, hm.d_inv, c->stage[i & 1], part * (size_t)i, len(i), to_dev ? 1 : 0);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->ev_stage[i & 1], c->stream));
    return SRS_OK;
  };
  int rc;
  if (to_dev) {
    for (int i = 0; i < n_parts; ++i) {
      if (i >= 2) HIPCHK(hipEventSynchronize(c->ev_stage[i & 1]));  // part i - 2 has left its buffer
      team.copy(c->stage[i & 1], host + part * (size_t)i, len(i) * sizeof(double));
      if ((rc = launch(i))) return rc;
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    return SRS_OK;
  }
  if ((rc = launch(0))) return rc;
  for (int i = 0; i < n_parts; ++i) {
    if (i + 1 < n_parts && (rc = launch(i + 1))) return rc;
    HIPCHK(hipEventSynchronize(c->ev_stage[i & 1]));
    team.copy(host + part * (size_t)i, c->stage[i & 1], len(i) * sizeof(double));
  }
  return SRS_OK;
}

int live_rw(srs_ctx* c, int32_t r, RealLive* lv, bool write) {
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  if (write) {
    int rc = tiles_full(c);
    if (rc) return rc;
  }
  if (write) HIPCHK(hipMemcpy(c->d_live + r, lv, sizeof(*lv), hipMemcpyHostToDevice));
  else HIPCHK(hipMemcpy(lv, c->d_live + r, sizeof(*lv), hipMemcpyDeviceToHost));
  return SRS_OK;
}

// Whether steps run through k_sweep_gated, and the live state index they
// start from: single-realization contexts while the realization is neither
// finished nor in the ffwd phase.  Reading the live state waits for the
// stream.
int gated_start(srs_ctx* c, bool* ok, int* cur) {
  *ok = false;
  if (!c->gated || c->reals.size() != 1) return SRS_OK;
  RealLive lv;
  int rc = live_rw(c, 0, &lv, false);
  if (rc) return rc;
  if (lv.done || lv.ffwd || c->n_tiles == 0) return SRS_OK;
  *ok = true;
  *cur = lv.cur;
  return SRS_OK;
}

// n_steps steps launched one by one, through the gated sweep from live index
// cur or as sweep and gating.
void launch_steps(srs_ctx* c, int64_t n_steps, uint32_t gmode, bool gated, int cur) {
  if (gated) launch_gated_block(c, n_steps, cur, gmode);
  else
    for (int64_t k = 0; k < n_steps; ++k) launch_step(c, gmode);
}

#endif  // SRS_UNIT == 0

}  // namespace srs_dev

#if SRS_UNIT == 0
// Replay schedules of srs_explicit_step_replay_static: file-scope device
// memory that every GPU the library runs on holds until the process ends
// (8 MiB: 2,097,152 RyR states, steps x RyRs).  In host code `scratch` names
// a host-side stand-in; the device address of each GPU's copy comes from
// hipGetSymbolAddress with that GPU current and is the only form used.
constexpr size_t kStaticSchedInts = (size_t)1 << 21;
static __device__ __align__(256) int32_t scratch[kStaticSchedInts];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
int32_t* g_scratch_ptr[kMaxDevices] = {};

// Once per device, with that device current (srs_ctx_create sets it).
int scratch_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return srs::fail(SRS_E_ARG, "device %d beyond %d", device, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return SRS_OK;
  void* p = nullptr;
  HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = (int32_t*)p;
  return SRS_OK;
}

int32_t* scratch_ptr(int device) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return device >= 0 && device < kMaxDevices ? g_scratch_ptr[device] : nullptr;
}
}  // namespace

extern "C" {

int srs_ctx_create(int device, srs_ctx** out) {
  srs::clear_error();
  if (!out) return srs::fail(SRS_E_ARG, "null out");
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return srs::fail(SRS_E_NODEV, "no HIP device");
  if (device < 0 || device >= n) return srs::fail(SRS_E_ARG, "device %d out of range (%d)", device, n);
  hipDeviceProp_t prop;
  HIPCHK(hipGetDeviceProperties(&prop, device));
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return srs::fail(SRS_E_NODEV, "device %d is %s; this library is built for gfx950", device, prop.gcnArchName);
  HIPCHK(hipSetDevice(device));
  int rc = scratch_setup(device);
  if (rc) return rc;
  auto c = new srs_ctx();
  c->device = device;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
    delete c;
    return srs::fail(SRS_E_HIP, "stream/event creation failed");
  }
  *out = c;
  return SRS_OK;
}

int srs_ctx_tune(srs_ctx* c, int32_t key, int32_t value) {
  srs::clear_error();
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  switch (key) {
    case SRS_TUNE_TILE:
      if (value != 128 && value != 256 && value != 512) return srs::fail(SRS_E_ARG, "tile must be 128, 256 or 512");
      if (c->finalized) return srs::fail(SRS_E_STATE, "tile must be set before srs_ctx_finalize");
      c->tile_set = value;
      return SRS_OK;
    case SRS_TUNE_PLANE_PAD:
      if (value < 0 || value % 64 || value > 1 << 20) return srs::fail(SRS_E_ARG, "plane pad must be a multiple of 64");
      if (c->layout_fixed) return srs::fail(SRS_E_STATE, "plane pad must be set before the first mesh");
      c->plane_pad = value;
      return SRS_OK;
    case SRS_TUNE_COMPACT:
      if (c->layout_fixed) return srs::fail(SRS_E_STATE, "compact layout must be chosen before the first mesh");
      c->compact = value != 0;
      return SRS_OK;
    // kernel keys: captured step graphs hold the old kernels, so they are dropped
    case SRS_TUNE_NT_GEOMETRY: return SRS_OK;  // rows are read through the caches
    case SRS_TUNE_OCCUPANCY:
      if (value != 0 && value != 6 && value != 8) return srs::fail(SRS_E_ARG, "occupancy must be 0, 6 or 8");
      c->occ = value;
      return c->finalized ? drop_graphs(c) : SRS_OK;
    case SRS_TUNE_NT_STATE:
      c->nt_state = value != 0;
      return c->finalized ? drop_graphs(c) : SRS_OK;
    case SRS_TUNE_LDS: return SRS_OK;  // tiles are always staged
    case SRS_TUNE_GATED_SWEEP:
      c->gated = value != 0;
      return c->finalized ? drop_graphs(c) : SRS_OK;
    case SRS_TUNE_DROP_FINISHED:
      c->drop_finished = value != 0;
      return c->finalized ? tiles_full(c) : SRS_OK;
    case SRS_TUNE_ADJ_WAVES:
      if (value != 0 && value != 4) return srs::fail(SRS_E_ARG, "adjoint register budget must be 0 or 4");
      return SRS_OK;  // four wavefronts per SIMD either way
    case SRS_TUNE_ADJ_W:
      if (value < 0 || value > 2) return srs::fail(SRS_E_ARG, "adjoint w form must be 0, 1 or 2");
      return SRS_OK;  // the gather reads the stored adjoint: no w
    case SRS_TUNE_ALT_ORDER:
      c->alt_order = value != 0;
      return c->finalized ? drop_graphs(c) : SRS_OK;
    case SRS_TUNE_SUBSET_MB:
      if (value < 0 || value > (1 << 20)) return srs::fail(SRS_E_ARG, "subset size must be 0..2^20 MB");
      c->subset_mb = value;
      c->subsets_valid = false;
      return c->finalized ? drop_graphs(c) : SRS_OK;
    case SRS_TUNE_ADJ_LEVELS:
      if (value < 0 || value > 6) return srs::fail(SRS_E_ARG, "adjoint checkpoint levels must be 0..6");
      c->adj_levels = value;
      return SRS_OK;
    case SRS_TUNE_GROUP:
      if (value != 1 && value != 2 && value != 4) return srs::fail(SRS_E_ARG, "group must be 1, 2 or 4");
      if (c->finalized) return srs::fail(SRS_E_STATE, "group must be set before srs_ctx_finalize");
      c->group = value;
      return SRS_OK;
    default: return srs::fail(SRS_E_ARG, "unknown tuning key %d", key);
  }
}

int srs_ctx_record_layout(srs_ctx* c, int32_t gpu_layout) {
  srs::clear_error();
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (c->finalized) return srs::fail(SRS_E_STATE, "the record layout is fixed at srs_ctx_finalize");
  if (gpu_layout != 0 && gpu_layout != 1) return srs::fail(SRS_E_ARG, "gpu_layout must be 0 or 1");
  c->gpu_layout = gpu_layout;
  return SRS_OK;
}

int srs_ctx_extensions(srs_ctx* c, int32_t r, const srs_extensions* e) {
  srs::clear_error();
  if (!c || !e) return srs::fail(SRS_E_ARG, "null argument");
  if (r < 0 || r >= (int32_t)c->reals.size()) return srs::fail(SRS_E_ARG, "realization %d out of range", r);
  if (e->jsr_diffusion != 0 && e->jsr_diffusion != 1) return srs::fail(SRS_E_ARG, "jsr_diffusion must be 0 or 1");
  if (!(e->b_sr_sites >= 0.0) || (e->b_sr_sites > 0.0 && !(e->k_d_sr_sites > 0.0)))
    return srs::fail(SRS_E_ARG, "SR sites need b >= 0 and, when b > 0, a dissociation constant > 0");
  HostReal& hr = c->reals[r];
  hr.ext = *e;
  if (!c->finalized) return SRS_OK;
  hr.desc.jsr_diff = e->jsr_diffusion;
  hr.desc.b_sr = e->b_sr_sites;
  hr.desc.k_sr = e->k_d_sr_sites;
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(c->d_desc + r, &hr.desc, sizeof(hr.desc), hipMemcpyHostToDevice));
  return SRS_OK;
}

static void release_stage(srs_ctx* c) {
  if (c->stage[0]) (void)hipHostFree(c->stage[0]);
  for (int k = 0; k < 2; ++k) {
    if (c->ev_stage[k]) (void)hipEventDestroy(c->ev_stage[k]);
    c->stage[k] = nullptr;
    c->ev_stage[k] = nullptr;
  }
  c->stage_len = 0;
}

int srs_ctx_destroy(srs_ctx* c) {
  if (!c) return SRS_OK;
  (void)hipSetDevice(c->device);
  (void)hipStreamSynchronize(c->stream);
  for (auto& kv : c->graphs) (void)hipGraphExecDestroy(kv.second);
  for (void* p : c->allocs) (void)hipFree(p);
  release_stage(c);
  (void)hipEventDestroy(c->ev0);
  (void)hipEventDestroy(c->ev1);
  (void)hipStreamDestroy(c->stream);
  delete c;
  return SRS_OK;
}

int srs_ctx_add_mesh(srs_ctx* c, const srs_mesh_desc* m, int32_t* mesh_id) {
  srs::clear_error();
  if (!c || !m || !mesh_id) return srs::fail(SRS_E_ARG, "null argument");
  if (c->finalized) return srs::fail(SRS_E_STATE, "context already finalized");
  const int32_t n = m->n_ele;
  if (n <= 0 || !m->aij || !m->nij || !m->domain || !m->tropc || !m->V0 || !m->tt_area)
    return srs::fail(SRS_E_ARG, "mesh descriptor incomplete");
  for (int64_t k = 0; k < 4LL * n; ++k)
    if (m->nij[k] < 0 || m->nij[k] >= n) return srs::fail(SRS_E_ARG, "nij[%lld] = %d out of range", (long long)k, m->nij[k]);
  auto hm = std::make_unique<HostMesh>();
  hm->n = n;
  c->layout_fixed = true;
  hm->np = (n + MAX_TILE - 1) / MAX_TILE * MAX_TILE + c->plane_pad;
  const int np = hm->np;
  // element order inside the context
  if (m->order == SRS_ORDER_RCM) {
    srs::rcm_order(n, m->nij, hm->perm);
  } else if (m->order == SRS_ORDER_CUSTOM) {
    if (!m->perm) return srs::fail(SRS_E_ARG, "SRS_ORDER_CUSTOM needs a permutation");
    hm->perm.assign(m->perm, m->perm + n);
    std::vector<uint8_t> seen(n, 0);
    for (int i = 0; i < n; ++i) {
      if (hm->perm[i] < 0 || hm->perm[i] >= n || seen[hm->perm[i]]) return srs::fail(SRS_E_ARG, "perm is not a permutation");
      seen[hm->perm[i]] = 1;
    }
  } else {
    hm->perm.resize(n);
    std::iota(hm->perm.begin(), hm->perm.end(), 0);
  }
  hm->inv.assign(n, 0);
  for (int i = 0; i < n; ++i) hm->inv[hm->perm[i]] = i;
  hm->nbr.assign(4 * (size_t)np, 0);
  hm->coef.assign(5 * (size_t)np, 0.0);
  hm->flags.assign(np, 0);
  hm->V0.assign(np, 1.0);
  hm->tt.assign(np, 0.0);
  bool any_br = false;
  if (m->br)
    for (int s : {srs::CA, srs::DYE, srs::ATP, srs::CMDN})
      for (int i = 0; i < n; ++i) any_br |= (m->br[(size_t)s * n + i] != 0.0);
  if (any_br) hm->br.assign(4 * (size_t)np, 0.0);
  for (int k = 0; k < np; ++k) {
    if (k >= n) {  // padding rows point at themselves
      for (int q = 0; q < 4; ++q) hm->nbr[4 * (size_t)k + q] = 0;
      continue;
    }
    const int i = hm->perm[k];
    for (int q = 0; q < 5; ++q) hm->coef[(size_t)q * np + k] = m->aij[5 * (size_t)i + q];
    for (int q = 0; q < 4; ++q) {
      const int32_t nb = m->nij[4 * (size_t)i + q];
      hm->nbr[4 * (size_t)k + q] = (uint32_t)hm->inv[nb] | (m->tt_area[nb] != 0.0 ? IDX_SL : 0u);
    }
    uint8_t f = 0;
    if (m->domain[i] != 0) f |= F_JSR;
    if (m->tropc[i]) f |= F_TROPC;
    if (m->tt_area[i] != 0.0) f |= F_SL;
    hm->V0[k] = m->V0[i];
    hm->tt[k] = m->tt_area[i];
    if (any_br) {
      const int sp[4] = {srs::CA, srs::DYE, srs::ATP, srs::CMDN};
      bool nz = false;
      for (int q = 0; q < 4; ++q) {
        const double v = m->br[(size_t)sp[q] * n + i];
        hm->br[(size_t)q * np + k] = v;
        nz |= (v != 0.0);
      }
      if (nz) f |= F_BR;
    }
    hm->flags[k] = f;
  }
  if (c->compact) build_class_rows(*hm);
  *mesh_id = (int32_t)c->meshes.size();
  c->meshes.push_back(std::move(hm));
  return SRS_OK;
}

int srs_ctx_add_realization(srs_ctx* c, int32_t mesh_id, const srs_chan_desc* ch, const int32_t ints[SRS_N_INT],
                            const double reals[SRS_N_REAL], uint64_t seed_key, uint64_t stream, int32_t* real_id) {
  srs::clear_error();
  if (!c || !ch || !ints || !reals || !real_id) return srs::fail(SRS_E_ARG, "null argument");
  if (c->finalized) return srs::fail(SRS_E_STATE, "context already finalized");
  if (mesh_id < 0 || mesh_id >= (int32_t)c->meshes.size()) return srs::fail(SRS_E_ARG, "bad mesh id %d", mesh_id);
  HostMesh& hm = *c->meshes[mesh_id];
  if (ch->n_ryr < 0 || ch->n_ryr > MAX_RYR || ch->n_lcc < 0 || ch->n_lcc > MAX_LCC)
    return srs::fail(SRS_E_ARG, "channel counts %d/%d exceed %d/%d", ch->n_ryr, ch->n_lcc, MAX_RYR, MAX_LCC);
  if (!(reals[SRS_R_T_STEP] > 0)) return srs::fail(SRS_E_ARG, "t_step must be > 0");
  HostReal hr;
  hr.mesh = mesh_id;
  memcpy(hr.ints, ints, sizeof(hr.ints));
  memcpy(hr.reals, reals, sizeof(hr.reals));
  hr.key = seed_key;
  hr.stream = stream;
  std::vector<std::pair<int32_t, ChanEntry>> entries;  // (dev element, channel) in reference order
  for (int i = 0; i < ch->n_ryr; ++i) {
    const int ce = ch->ryr_ele[i], je = ch->ryr_jsr[i];
    if (ce < 0 || ce >= hm.n || je < 0 || je >= hm.n) return srs::fail(SRS_E_ARG, "RyR %d element out of range", i);
    hr.ryr_ele.push_back(hm.inv[ce]);
    hr.ryr_jsr.push_back(hm.inv[je]);
    for (int q = 0; q < 4; ++q) {
      const int nb = ch->ryr_nb ? ch->ryr_nb[4 * i + q] : -1;
      if (nb >= ch->n_ryr || nb < -1) return srs::fail(SRS_E_ARG, "RyR %d neighbour %d out of range", i, nb);
      hr.ryr_nb.push_back(nb);
    }
    entries.push_back({hm.inv[ce], {2 * i, hm.inv[je], hm.inv[ce], 0}});
    entries.push_back({hm.inv[je], {2 * i + 1, hm.inv[je], hm.inv[ce], 0}});
  }
  for (int i = 0; i < ch->n_lcc; ++i) {
    const int e = ch->lcc_ele[i];
    if (e < 0 || e >= hm.n) return srs::fail(SRS_E_ARG, "LCC %d element out of range", i);
    hr.lcc_ele.push_back(hm.inv[e]);
    entries.push_back({hm.inv[e], {-(i + 1), 0, 0, 0}});
  }
  if (ints[SRS_I_INIT_RYR] != -1 && (ints[SRS_I_INIT_RYR] < 0 || ints[SRS_I_INIT_RYR] >= ch->n_ryr))
    return srs::fail(SRS_E_ARG, "ryr_open_init %d must be -1 or in [0, %d)", ints[SRS_I_INIT_RYR], ch->n_ryr);
  if (ints[SRS_I_FLAG_LCC] && (ints[SRS_I_LCC_INDEX] < 0 || ints[SRS_I_LCC_INDEX] >= ch->n_lcc))
    return srs::fail(SRS_E_ARG, "LCC index %d out of range", ints[SRS_I_LCC_INDEX]);
  std::stable_sort(entries.begin(), entries.end(),
                   [](const std::pair<int32_t, ChanEntry>& a, const std::pair<int32_t, ChanEntry>& b) {
                     return a.first < b.first;
                   });
  for (size_t k = 0; k < entries.size(); ++k) {
    if (k == 0 || entries[k].first != entries[k - 1].first) {
      hr.celem.push_back(entries[k].first);
      hr.cstart.push_back((int32_t)k);
      hm.flags[entries[k].first] |= F_CHAN;
    }
    hr.centry.push_back(entries[k].second);
  }
  hr.cstart.push_back((int32_t)entries.size());
  if (!hm.br.empty()) {
    // The mesh's boundary rates were built with one set of D; every
    // realization on the mesh must start from it (srs_params_set may move it
    // later, and the rates follow).
    const double D[4] = {reals[SRS_R_D_CA], reals[SRS_R_D_DYE], reals[SRS_R_D_ATP], reals[SRS_R_D_CMDN]};
    if (!hm.br_d_set) {
      std::copy(D, D + 4, hm.br_d);
      hm.br_d_set = true;
    } else if (!std::equal(D, D + 4, hm.br_d)) {
      return srs::fail(SRS_E_ARG, "realizations on a mesh with boundary rates must share the D the rates were "
                                  "built with (D_Ca %g, D_Fluo %g, D_ATP %g, D_CaM %g)", hm.br_d[0], hm.br_d[1],
                       hm.br_d[2], hm.br_d[3]);
    }
  }
  *real_id = (int32_t)c->reals.size();
  c->reals.push_back(std::move(hr));
  return SRS_OK;
}

int srs_ctx_finalize(srs_ctx* c, int32_t record_capacity) {
  srs::clear_error();
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (c->finalized) return srs::fail(SRS_E_STATE, "already finalized");
  if (c->reals.empty()) return srs::fail(SRS_E_STATE, "no realizations");
  HIPCHK(hipSetDevice(c->device));
  int rc;
  // nothing of a call that failed part way stays: it may be repeated
  c->bands.clear();
  c->sweep_lds = 0;
  release_stage(c);
  std::vector<HostMap> maps;
  if ((rc = plan_tiles(c, &maps))) return rc;
  c->class_all = !c->meshes.empty();
  for (auto& hmp : c->meshes) c->class_all &= hmp->class_rows;
  for (size_t k = 0; k < c->meshes.size(); ++k) {
    if ((rc = upload_mesh(c, *c->meshes[k], maps[k]))) return rc;
    c->sweep_lds = std::max(c->sweep_lds, 4 * sizeof(double) * (size_t)maps[k].qcap);
  }
  maps.clear();
  std::vector<RealDesc> descs;
  std::vector<RealLive> lives;
  std::vector<int2> tiles;
  // bytes a step works on: the state buffers, and rows and halo lists
  double ws = 0.0;
  for (const HostReal& hr : c->reals) ws += 2.0 * 48.0 * c->meshes[hr.mesh]->n;
  for (auto& hmp : c->meshes) ws += (double)hmp->n * ((c->class_all ? 12 : 40) + 9) + 4.0 * hmp->map.n_halo;
  // Tile order.  Up to four realizations of a mesh form a band whose tiles lie
  // side by side, so that rows and halo lists come from the L2 for all but the
  // first, while everything a step touches fits the 256 MB last-level cache (us
  // per step in bands of one / four: 14-member ensemble, 207 MB, 40.9 / 37.8;
  // 16 members, 237 MB, 45.2 / 43.4; two 928k-element dyads, 200 MB, 40.4 /
  // 38.5).  Beyond it four state streams at a time cost more than the rows (18
  // members, 266 MB, 52.7 / 56.6; 48, 137 / 142; twelve 214k-element dyads, 241
  // MB, 53.7 / 48.5 in one run and 57.4 in another).  Nor with scattered orders,
  // whose halos fill the L2 (four members of 56,250 elements 19.0 / 21.6, of
  // 172,494, recording, 45 / 58).
  const int width = ws > 220e6 || c->quad_block == 1 ? 1 : 4;
  for (size_t m = 0; m < c->meshes.size(); ++m) {
    for (size_t r = 0, fill = width; r < c->reals.size(); ++r) {
      if (c->reals[r].mesh != (int)m) continue;
      if (fill == (size_t)width) {
        c->bands.emplace_back();
        fill = 0;
      }
      c->bands.back().push_back((int32_t)r);
      c->reals[r].band = (int32_t)c->bands.size() - 1;
      ++fill;
    }
  }
  for (const auto& band : c->bands) {
    const HostMesh& hm = *c->meshes[c->reals[band[0]].mesh];
    const int nt = (hm.n + c->tile - 1) / c->tile;
    for (int t = 0; t < nt; ++t)
      for (int r : band) tiles.push_back(make_int2(r, t));
  }
  for (size_t r = 0; r < c->reals.size(); ++r) {
    HostReal& hr = c->reals[r];
    HostMesh& hm = *c->meshes[hr.mesh];
    RealDesc d{};
    d.nbr = hm.d_nbr; d.coef = hm.d_coef; d.flags = hm.d_flags; d.V0 = hm.d_V0; d.tt = hm.d_tt; d.br = hm.d_br;
    d.br_mesh = hm.d_br;
    std::copy(hm.br_d, hm.br_d + 4, d.brd);
    d.loc = hm.map.d_loc; d.hal = hm.map.d_hal; d.hoff = hm.map.d_hoff; d.qcap = hm.map.qcap;
    d.qb = c->quad_block;
    d.row = hm.d_row; d.tab = hm.d_tab; d.blk = hm.d_blk;
    d.n_class = hm.n_class;
    d.n = hm.n; d.np = hm.np;
    for (int k = 0; k < 2; ++k) {
      if ((rc = dev_alloc(c, &d.X[k], 6 * (size_t)hm.np))) return rc;
      HIPCHK(hipMemset(d.X[k], 0, 6 * (size_t)hm.np * sizeof(double)));
    }
    d.n_ryr = (int32_t)hr.ryr_ele.size();
    d.n_lcc = (int32_t)hr.lcc_ele.size();
    for (ChanEntry& en : hr.centry)
      if (en.code >= 0) en.sl = (hm.flags[en.jsr] & F_SL ? 1 : 0) | (hm.flags[en.cyt] & F_SL ? 2 : 0);
    std::vector<ChanElem> crec(hr.celem.size());
    for (size_t k = 0; k < crec.size(); ++k) {
      ChanElem& e = crec[k];
      e.j = hr.celem[k];
      for (int q = 0; q < 5; ++q) e.a[q] = hm.coef[(size_t)q * hm.np + e.j];
      for (int q = 0; q < 4; ++q) e.nb[q] = (int32_t)idx_of(hm.nbr[4 * (size_t)e.j + q]);
      e.v0 = hm.V0[e.j];
      e.tt = hm.tt[e.j];
      e.e0 = hr.cstart[k];
      e.e1 = hr.cstart[k + 1];
      e.f = hm.flags[e.j];
      e.first = hr.centry[e.e0];
    }
    d.n_celem = (int32_t)hr.celem.size();
    struct { int32_t *ryr_ele, *ryr_jsr, *ryr_nb, *lcc_ele, *celem, *cstart; ChanEntry* centry; ChanElem* crec; } t{};
    const std::vector<int32_t> closed(d.n_ryr, 0), ones(d.n_lcc, 1), twos(d.n_lcc, 2);
    const std::vector<double> resid(d.n_ryr + d.n_lcc, -1.0);
    Pack pk(c);
    if ((rc = pk.add(&t.ryr_ele, hr.ryr_ele)) || (rc = pk.add(&t.ryr_jsr, hr.ryr_jsr)) ||
        (rc = pk.add(&t.ryr_nb, hr.ryr_nb)) || (rc = pk.add(&t.lcc_ele, hr.lcc_ele)) ||
        (rc = pk.add(&t.celem, hr.celem)) || (rc = pk.add(&t.cstart, hr.cstart)) ||
        (rc = pk.add(&t.centry, hr.centry)) || (rc = pk.add(&t.crec, crec)) || (rc = pk.add(&d.ryr_state, closed)) ||
        (rc = pk.add(&d.lcc_state, ones)) || (rc = pk.add(&d.lccv_state, twos)) || (rc = pk.add(&d.R, resid)) ||
        (rc = pk.upload()))
      return rc;
    d.ryr_ele = t.ryr_ele; d.ryr_jsr = t.ryr_jsr; d.ryr_nb = t.ryr_nb; d.lcc_ele = t.lcc_ele;
    d.celem = t.celem; d.cstart = t.cstart; d.centry = t.centry; d.crec = t.crec;
    d.ryr_out = hr.ints[SRS_I_FLAG_RYR_OUT] ? 1 : 0;
    d.gpu_layout = c->gpu_layout;
    d.rec_len = 7 + (d.gpu_layout ? d.n_ryr : 0) + (d.ryr_out ? d.n_ryr : 0);
    if (record_capacity > 0 && d.rec_len > 255)  // cpu/OutputFuncs.cpp:441-444
      return srs::fail(SRS_E_ARG, "states record of %d floats exceeds the 255-float record limit", d.rec_len);
    d.rec_cap = record_capacity;
    if (record_capacity > 0) {
      float* fr;
      if ((rc = dev_alloc(c, &fr, (size_t)record_capacity * d.rec_len))) return rc;
      d.rec = fr;
    }
    d.key = hr.key;
    d.stream = hr.stream;
    d.jsr_diff = hr.ext.jsr_diffusion;
    d.b_sr = hr.ext.b_sr_sites;
    d.k_sr = hr.ext.k_d_sr_sites;
    memcpy(d.P, hr.reals, sizeof(d.P));
    memcpy(d.I, hr.ints, sizeof(d.I));
    hr.desc = d;
    descs.push_back(d);
    RealLive lv{};
    lv.vm = hr.reals[SRS_R_DEFAULT_VM];
    lv.ca_nsr = hr.reals[SRS_R_DEFAULT_CA_NSR];
    serca_terms(lv.ca_nsr, hr.reals, lv.serca);
    lives.push_back(lv);
  }
  // Cache hints.  A step reads and writes every state buffer in turn with the
  // one before, so while the buffers and the meshes' rows fit the 256 MB
  // last-level cache nothing is hinted past it (us per step without hints /
  // non-temporal stores / non-temporal row loads: 928k-element dyad, 114 MB,
  // 21.5 / 25.9 / 24.8; 18-member ensemble, 266 MB, 53.6 / 60.8 / 61.2; 20
  // members, 295 MB, 62.0 / 62.5 / -).  Beyond it plain stores
  // evict what the next step could still have found (24 members, 351 MB, 78.6 /
  // 74.9 / 77.4; 3M-element dyad, 362 MB, 69.4 / 61.1 / 61.2; 48 members, 147 /
  // 138 / 160).  The line lies between 295 and 351 MB.  Row loads are never
  // hinted: nowhere faster than the better of the other two.
  const int nt_state = c->nt_state < 0 ? ws > 330e6 : c->nt_state;
  c->n_tiles = (int)tiles.size();
  c->grid_sweep = (c->n_tiles + NXCD - 1) / NXCD * NXCD;
  // State transfers: up to 4 MB of fields in parts of 0.5 MB, larger ones in
  // halves of at most 8 MB, one part copied while one moves.  A pinned page costs
  // 0.75 us when it is first touched: with two halves of 1.3 MB the first fields
  // set of 56,250 elements took 1.0 ms against 0.4, later ones no less (read 0.17
  // against 0.13).  Eight parts of 1.3 MB, each with its launch, wait and
  // helpers, read 219,000 elements 0.07 ms slower than halves.
  size_t fields = 0;
  for (const HostReal& hr : c->reals) fields = std::max(fields, 6 * (size_t)c->meshes[hr.mesh]->n);
  c->stage_len = fields <= (size_t)1 << 19 ? std::min(fields, (size_t)1 << 16)
                                           : std::min((fields + 1) / 2, (size_t)1 << 20);
  c->stage_len = (c->stage_len + 511) / 512 * 512;  // the second buffer on a page
  HIPCHK(hipHostMalloc((void**)&c->stage[0], 2 * c->stage_len * sizeof(double), hipHostMallocDefault));
  c->stage[1] = c->stage[0] + c->stage_len;
  for (int k = 0; k < 2; ++k) HIPCHK(hipEventCreateWithFlags(&c->ev_stage[k], hipEventDisableTiming));
  if ((rc = dev_upload(c, &c->d_desc, descs))) return rc;
  if ((rc = dev_upload(c, &c->d_live, lives))) return rc;
  if ((rc = dev_upload(c, &c->d_tiles, tiles))) return rc;
  c->tiles_all = tiles;
  c->tiles_cur = tiles;
  c->d_tiles_all = c->d_tiles;
  if (c->reals.size() > 1 && (rc = dev_alloc(c, &c->d_sub_rids, c->reals.size()))) return rc;
  if (c->reals.size() > 1 && (rc = dev_alloc(c, &c->d_tiles_live, tiles.size()))) return rc;
  HIPCHK(hipDeviceSynchronize());
  c->nt_state = nt_state;
  c->finalized = true;
  return SRS_OK;
}


int srs_state_set(srs_ctx* c, int32_t r, const double* X) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (!X) return srs::fail(SRS_E_ARG, "null state");
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  return state_xfer(c, r, const_cast<double*>(X), true);
}

int srs_state_get(srs_ctx* c, int32_t r, double* X) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (!X) return srs::fail(SRS_E_ARG, "null state");
  HIPCHK(hipSetDevice(c->device));
  return state_xfer(c, r, X, false);
}

int srs_channels_set(srs_ctx* c, int32_t r, const int32_t* ryr_state, const int32_t* lcc_state,
                     const int32_t* lccv_state, const double* R) {
  int rc = check_real(c, r);
  if (rc) return rc;
  const RealDesc& d = c->reals[r].desc;
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  if (ryr_state && d.n_ryr) HIPCHK(hipMemcpy(d.ryr_state, ryr_state, d.n_ryr * sizeof(int32_t), hipMemcpyHostToDevice));
  if (lcc_state && d.n_lcc) HIPCHK(hipMemcpy(d.lcc_state, lcc_state, d.n_lcc * sizeof(int32_t), hipMemcpyHostToDevice));
  if (lccv_state && d.n_lcc) HIPCHK(hipMemcpy(d.lccv_state, lccv_state, d.n_lcc * sizeof(int32_t), hipMemcpyHostToDevice));
  if (R && d.n_ryr + d.n_lcc) HIPCHK(hipMemcpy(d.R, R, (d.n_ryr + d.n_lcc) * sizeof(double), hipMemcpyHostToDevice));
  return SRS_OK;
}

int srs_channels_get(srs_ctx* c, int32_t r, int32_t* ryr_state, int32_t* lcc_state, int32_t* lccv_state, double* R) {
  int rc = check_real(c, r);
  if (rc) return rc;
  const RealDesc& d = c->reals[r].desc;
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  if (ryr_state && d.n_ryr) HIPCHK(hipMemcpy(ryr_state, d.ryr_state, d.n_ryr * sizeof(int32_t), hipMemcpyDeviceToHost));
  if (lcc_state && d.n_lcc) HIPCHK(hipMemcpy(lcc_state, d.lcc_state, d.n_lcc * sizeof(int32_t), hipMemcpyDeviceToHost));
  if (lccv_state && d.n_lcc) HIPCHK(hipMemcpy(lccv_state, d.lccv_state, d.n_lcc * sizeof(int32_t), hipMemcpyDeviceToHost));
  if (R && d.n_ryr + d.n_lcc) HIPCHK(hipMemcpy(R, d.R, (d.n_ryr + d.n_lcc) * sizeof(double), hipMemcpyDeviceToHost));
  return SRS_OK;
}


int srs_globals_set(srs_ctx* c, int32_t r, double vm, double ca_nsr) {
  int rc = check_real(c, r);
  if (rc) return rc;
  RealLive lv;
  if ((rc = live_rw(c, r, &lv, false))) return rc;
  lv.vm = vm;
  lv.ca_nsr = ca_nsr;
  serca_terms(ca_nsr, c->reals[r].reals, lv.serca);
  return live_rw(c, r, &lv, true);
}

int srs_globals_get(srs_ctx* c, int32_t r, double* vm, double* ca_nsr) {
  int rc = check_real(c, r);
  if (rc) return rc;
  RealLive lv;
  if ((rc = live_rw(c, r, &lv, false))) return rc;
  if (vm) *vm = lv.vm;
  if (ca_nsr) *ca_nsr = lv.ca_nsr;
  return SRS_OK;
}

int srs_loop_set(srs_ctx* c, int32_t r, const srs_loop_state* ls) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (!ls) return srs::fail(SRS_E_ARG, "null loop state");
  RealLive lv;
  if ((rc = live_rw(c, r, &lv, false))) return rc;
  lv.t = ls->t; lv.dt_last = ls->dt_last; lv.step = ls->step; lv.done = ls->done; lv.lcc_open = ls->lcc_open;
  lv.t_lcc_close = ls->t_lcc_close; lv.n_open_last = ls->n_ryr_open_last; lv.ca_max_last = ls->ca_ss_max_last;
  lv.ffwd = ls->ffwd ? 1 : 0;
  return live_rw(c, r, &lv, true);
}

int srs_loop_get(srs_ctx* c, int32_t r, srs_loop_state* ls) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (!ls) return srs::fail(SRS_E_ARG, "null loop state");
  RealLive lv;
  if ((rc = live_rw(c, r, &lv, false))) return rc;
  ls->t = lv.t; ls->dt_last = lv.dt_last; ls->step = lv.step; ls->done = lv.done; ls->lcc_open = lv.lcc_open;
  ls->t_lcc_close = lv.t_lcc_close; ls->n_ryr_open_last = lv.n_open_last; ls->ca_ss_max_last = lv.ca_max_last;
  ls->ffwd = lv.ffwd;
  return SRS_OK;
}

// ---------------------------------------------------------- checkpoints
// Layout of a realization's checkpoint: header, fields in the reference
// numbering ([6][n_ele] FP64, as srs_state_get), RyR states, LCC states, LCC
// voltage-gate states (int32, padded to 8 bytes), residuals, then the loop
// state.
namespace {
struct CkHeader {
  char magic[8];
  int32_t version, n_ele, n_ryr, n_lcc;
  uint64_t key, stream;
};
struct CkLive {
  double t, dt_last, vm, ca_nsr, t_lcc_close, ca_max_last;
  int64_t step;
  int32_t done, lcc_open, n_open_last, ffwd;
};
constexpr char kCkMagic[8] = {'S', 'R', 'S', 'C', 'K', 'P', 'T', '1'};

size_t ck_int_bytes(size_t nr, size_t nl) { return (sizeof(int32_t) * (nr + 2 * nl) + 7) / 8 * 8; }

size_t ck_bytes(const HostReal& hr, int32_t n_ele) {
  const size_t nr = hr.ryr_ele.size(), nl = hr.lcc_ele.size();
  return sizeof(CkHeader) + 6 * sizeof(double) * (size_t)n_ele + ck_int_bytes(nr, nl) + sizeof(double) * (nr + nl) +
         sizeof(CkLive);
}
}  // namespace

int srs_checkpoint_size(srs_ctx* c, int32_t r, size_t* bytes) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (!bytes) return srs::fail(SRS_E_ARG, "null size");
  *bytes = ck_bytes(c->reals[r], c->meshes[c->reals[r].mesh]->n);
  return SRS_OK;
}

int srs_checkpoint_save(srs_ctx* c, int32_t r, void* buf, size_t bytes) {
  int rc = check_real(c, r);
  if (rc) return rc;
  const HostReal& hr = c->reals[r];
  const int32_t n = c->meshes[hr.mesh]->n;
  if (!buf || bytes < ck_bytes(hr, n)) return srs::fail(SRS_E_ARG, "checkpoint buffer smaller than srs_checkpoint_size");
  const size_t nr = hr.ryr_ele.size(), nl = hr.lcc_ele.size();
  char* p = (char*)buf;
  CkHeader h{};
  memcpy(h.magic, kCkMagic, 8);
  h.version = 1;
  h.n_ele = n;
  h.n_ryr = (int32_t)nr;
  h.n_lcc = (int32_t)nl;
  h.key = hr.key;
  h.stream = hr.stream;
  memcpy(p, &h, sizeof h);
  p += sizeof h;
  if ((rc = srs_state_get(c, r, (double*)p))) return rc;
  p += 6 * sizeof(double) * (size_t)n;
  int32_t* rs = (int32_t*)p;
  int32_t* ls = rs + nr;
  int32_t* lv = ls + nl;
  memset(lv + nl, 0, ck_int_bytes(nr, nl) - sizeof(int32_t) * (nr + 2 * nl));
  double* R = (double*)(p + ck_int_bytes(nr, nl));
  if ((rc = srs_channels_get(c, r, rs, ls, lv, R))) return rc;
  p = (char*)(R + nr + nl);
  RealLive L;
  if ((rc = live_rw(c, r, &L, false))) return rc;
  const CkLive k{L.t, L.dt_last, L.vm, L.ca_nsr, L.t_lcc_close, L.ca_max_last, L.step,
                 L.done, L.lcc_open, L.n_open_last, L.ffwd};
  memcpy(p, &k, sizeof k);
  return SRS_OK;
}

int srs_checkpoint_load(srs_ctx* c, int32_t r, const void* buf, size_t bytes) {
  int rc = check_real(c, r);
  if (rc) return rc;
  const HostReal& hr = c->reals[r];
  const int32_t n = c->meshes[hr.mesh]->n;
  const size_t need = ck_bytes(hr, n);
  if (!buf || bytes < sizeof(CkHeader)) return srs::fail(SRS_E_ARG, "checkpoint buffer too small");
  const char* p = (const char*)buf;
  CkHeader h;
  memcpy(&h, p, sizeof h);
  if (memcmp(h.magic, kCkMagic, 8) || h.version != 1) return srs::fail(SRS_E_IO, "not an srs checkpoint (version 1)");
  if (h.n_ele != n || h.n_ryr != (int32_t)hr.ryr_ele.size() || h.n_lcc != (int32_t)hr.lcc_ele.size())
    return srs::fail(SRS_E_ARG, "checkpoint of %d elements, %d RyR, %d LCC does not fit this realization", h.n_ele,
                     h.n_ryr, h.n_lcc);
  if (h.key != hr.key || h.stream != hr.stream)
    return srs::fail(SRS_E_ARG, "checkpoint of another seed or stream: its gating would not continue the same run");
  if (bytes < need) return srs::fail(SRS_E_ARG, "checkpoint buffer truncated");
  p += sizeof h;
  const size_t nr = h.n_ryr, nl = h.n_lcc;
  const double* X = (const double*)p;
  const int32_t* rs = (const int32_t*)(X + 6 * (size_t)n);
  const int32_t* ls = rs + nr;
  const int32_t* lv = ls + nl;
  const double* R = (const double*)((const char*)rs + ck_int_bytes(nr, nl));
  CkLive k;
  memcpy(&k, R + nr + nl, sizeof k);
  if ((rc = srs_state_set(c, r, X))) return rc;
  if ((rc = srs_channels_set(c, r, rs, ls, lv, R))) return rc;
  RealLive L;
  if ((rc = live_rw(c, r, &L, false))) return rc;
  L.t = k.t; L.dt_last = k.dt_last; L.vm = k.vm; L.ca_nsr = k.ca_nsr; L.t_lcc_close = k.t_lcc_close;
  L.ca_max_last = k.ca_max_last; L.step = k.step; L.sched_base = k.step;
  L.done = k.done; L.lcc_open = k.lcc_open; L.n_open_last = k.n_open_last; L.ffwd = k.ffwd;
  L.rec_count = 0;
  L.rec_overflow = 0;
  serca_terms(L.ca_nsr, hr.reals, L.serca);
  return live_rw(c, r, &L, true);
}

// The captured block of `block` steps in gate mode `gmode` (made on first use
// and cached; tiles_compact and tiles_full drop the cache).
// Graph-cache key bits of the gated blocks (host only, never passed to a kernel).
constexpr uint32_t G_KEY_GATED = 1u << 8, G_KEY_CUR1 = 1u << 9, G_KEY_SUBSETS = 1u << 10;

static int graph_cached(srs_ctx* c, int64_t block, uint32_t key_mode, const std::function<void()>& capture,
                        hipGraphExec_t* out) {
  auto key = std::make_pair(block, key_mode);
  auto it = c->graphs.find(key);
  if (it == c->graphs.end()) {
    hipGraph_t g;
    HIPCHK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    capture();
    HIPCHK(hipStreamEndCapture(c->stream, &g));
    hipGraphExec_t ge;
    HIPCHK(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
    HIPCHK(hipGraphDestroy(g));
    it = c->graphs.emplace(key, ge).first;
  }
  *out = it->second;
  return SRS_OK;
}

static int graph_for(srs_ctx* c, int64_t block, uint32_t gmode, hipGraphExec_t* out) {
  if (!c->subsets.empty())
    return graph_cached(c, block, gmode | G_KEY_SUBSETS, [&] { launch_subset_block(c, block, gmode); }, out);
  return graph_cached(c, block, gmode, [&] { for (int64_t k = 0; k < block; ++k) launch_step(c, gmode); }, out);
}

// A block of steps through k_sweep_gated starting from live state index cur.
static int graph_gated(srs_ctx* c, int64_t block, int cur, uint32_t gmode, hipGraphExec_t* out) {
  return graph_cached(c, block, gmode | G_KEY_GATED | (cur ? G_KEY_CUR1 : 0u),
                      [&] { launch_gated_block(c, block, cur, gmode); }, out);
}

constexpr int64_t kGraphBlock = 128, kGraphMin = 16;
static_assert(kGraphBlock % 2 == 0, "a full gated block returns the live state index to where it started");

int srs_explicit_step_prepare(srs_ctx* c, int64_t n_steps, uint32_t flags) {
  srs::clear_error();
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (!c->finalized) return srs::fail(SRS_E_STATE, "context not finalized");
  if (n_steps < 0) return srs::fail(SRS_E_ARG, "negative step count");
  HIPCHK(hipSetDevice(c->device));
  const uint32_t gmode = G_AFTER_SWEEP | ((flags & SRS_STEP_PROTOCOL) ? G_PROTOCOL : 0u);
  int rc = tiles_compact(c);
  if (rc) return rc;
  if (!c->subsets_valid && (rc = plan_subsets(c))) return rc;
  hipGraphExec_t ge;
  bool gated;
  int cur;
  if ((rc = gated_start(c, &gated, &cur))) return rc;
  if (gated) {
    // both starting live indices: the one a later call starts from is not known here
    for (int p = 0; p < 2; ++p) {
      if (n_steps >= kGraphBlock && (rc = graph_gated(c, kGraphBlock, p, gmode, &ge))) return rc;
      if (n_steps % kGraphBlock >= kGraphMin && (rc = graph_gated(c, n_steps % kGraphBlock, p, gmode, &ge)))
        return rc;
    }
    return SRS_OK;
  }
  if (n_steps >= kGraphBlock && (rc = graph_for(c, kGraphBlock, gmode, &ge))) return rc;
  if (n_steps % kGraphBlock >= kGraphMin && (rc = graph_for(c, n_steps % kGraphBlock, gmode, &ge))) return rc;
  return SRS_OK;
}

int srs_explicit_step(srs_ctx* c, int64_t n_steps, uint32_t flags) {
  srs::clear_error();
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (!c->finalized) return srs::fail(SRS_E_STATE, "context not finalized");
  if (n_steps < 0) return srs::fail(SRS_E_ARG, "negative step count");
  HIPCHK(hipSetDevice(c->device));
  const uint32_t gmode = G_AFTER_SWEEP | ((flags & SRS_STEP_PROTOCOL) ? G_PROTOCOL : 0u);
  int rc = tiles_compact(c);
  if (rc) return rc;
  if (!c->subsets_valid && (rc = plan_subsets(c))) return rc;
  bool gated = false;
  int cur = 0;
  if (n_steps > 0 && (rc = gated_start(c, &gated, &cur))) return rc;
  HIPCHK(hipEventRecord(c->ev0, c->stream));
  int64_t done = 0;
  if (flags & SRS_STEP_GRAPH) {
    // 128-step blocks, then the rest as one block of its own when it is long enough
    hipGraphExec_t ge;
    if (n_steps >= kGraphBlock) {
      if ((rc = gated ? graph_gated(c, kGraphBlock, cur, gmode, &ge) : graph_for(c, kGraphBlock, gmode, &ge)))
        return rc;
      for (; n_steps - done >= kGraphBlock; done += kGraphBlock) HIPCHK(hipGraphLaunch(ge, c->stream));
    }
    if (n_steps - done >= kGraphMin) {
      const int64_t m = n_steps - done;
      if ((rc = gated ? graph_gated(c, m, cur, gmode, &ge) : graph_for(c, m, gmode, &ge))) return rc;
      HIPCHK(hipGraphLaunch(ge, c->stream));
      cur ^= (int)(m & 1);
      done = n_steps;
    }
  }
  if (gated) {
    if (done < n_steps) launch_gated_block(c, n_steps - done, cur, gmode);
  } else if (!c->subsets.empty()) {
    if (done < n_steps) launch_subset_block(c, n_steps - done, gmode);
  } else {
    for (; done < n_steps; ++done) launch_step(c, gmode);
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipEventRecord(c->ev1, c->stream));
  HIPCHK(hipEventSynchronize(c->ev1));
  float ms = 0;
  HIPCHK(hipEventElapsedTime(&ms, c->ev0, c->ev1));
  c->last_total_ms = ms;
  return SRS_OK;
}

int srs_channel_gating(srs_ctx* c) {
  srs::clear_error();
  if (!c || !c->finalized) return srs::fail(SRS_E_STATE, "context not finalized");
  HIPCHK(hipSetDevice(c->device));
  hipLaunchKernelGGL(k_gate, dim3((unsigned)c->reals.size()), dim3(GATE_THREADS), 0, c->stream, c->d_desc, c->d_live,
                     0u);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(c->stream));
  return SRS_OK;
}

// n_steps replayed steps with the schedule already in device memory at ds
// (null when the realization has no RyRs).
static int replay_from(srs_ctx* c, int32_t r, int64_t n_steps, const int32_t* schedule, int32_t* ds) {
  HostReal& hr = c->reals[r];
  const int nr = (int)hr.ryr_ele.size();
  if (nr) HIPCHK(hipMemcpy(hr.desc.ryr_state, schedule, nr * sizeof(int32_t), hipMemcpyHostToDevice));
  RealDesc d = hr.desc;
  d.sched = ds;
  d.n_sched = n_steps;
  HIPCHK(hipMemcpy(c->d_desc + r, &d, sizeof(d), hipMemcpyHostToDevice));
  RealLive lv;
  HIPCHK(hipMemcpy(&lv, c->d_live + r, sizeof(lv), hipMemcpyDeviceToHost));
  lv.sched_base = lv.step;
  HIPCHK(hipMemcpy(c->d_live + r, &lv, sizeof(lv), hipMemcpyHostToDevice));
  const uint32_t gmode = G_AFTER_SWEEP | G_NO_GATING | G_REPLAY;
  // through the gated sweep, a launch per step with the replay of the step
  // before in its workgroup 0: 400 steps of 124,146 elements 3.3 ms, 4.8 with
  // two launches
  bool gated;
  int cur;
  const int rc = gated_start(c, &gated, &cur);
  if (rc == SRS_OK) launch_steps(c, n_steps, gmode, gated, cur);
  hipError_t e = hipGetLastError();
  (void)hipStreamSynchronize(c->stream);
  HIPCHK(hipMemcpy(c->d_desc + r, &hr.desc, sizeof(hr.desc), hipMemcpyHostToDevice));
  if (e != hipSuccess) return srs::fail(SRS_E_HIP, "replay launch: %s", hipGetErrorString(e));
  return rc;
}

static int replay_check(srs_ctx* c, int32_t r, int64_t n_steps, const int32_t* schedule) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (c->reals.size() != 1) return srs::fail(SRS_E_ARG, "replay needs a single-realization context");
  if (n_steps < 0) return srs::fail(SRS_E_ARG, "negative step count");
  if (!schedule && n_steps > 0 && !c->reals[r].ryr_ele.empty()) return srs::fail(SRS_E_ARG, "null schedule");
  return SRS_OK;
}

int srs_explicit_step_replay(srs_ctx* c, int32_t r, int64_t n_steps, const int32_t* schedule) {
  int rc = replay_check(c, r, n_steps, schedule);
  if (rc || n_steps == 0) return rc;
  const int nr = (int)c->reals[r].ryr_ele.size();
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  int32_t* ds = nullptr;
  if (nr) {
    HIPCHK(hipMalloc(&ds, (size_t)n_steps * nr * sizeof(int32_t)));
    hipError_t e = hipMemcpy(ds, schedule, (size_t)n_steps * nr * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      (void)hipFree(ds);
      return srs::fail(SRS_E_HIP, "replay schedule copy: %s", hipGetErrorString(e));
    }
  }
  rc = replay_from(c, r, n_steps, schedule, ds);
  if (ds) (void)hipFree(ds);
  return rc;
}

int srs_explicit_step_replay_static(srs_ctx* c, int32_t r, int64_t n_steps, const int32_t* schedule) {
  int rc = replay_check(c, r, n_steps, schedule);
  if (rc || n_steps == 0) return rc;
  const size_t nr = c->reals[r].ryr_ele.size();
  if (nr && (size_t)n_steps > kStaticSchedInts / nr)
    return srs::fail(SRS_E_ARG, "replay of %lld steps x %zu RyRs exceeds the static schedule buffer of %zu RyR states",
                     (long long)n_steps, nr, kStaticSchedInts);
  int32_t* ds = scratch_ptr(c->device);
  if (!ds) return srs::fail(SRS_E_STATE, "no static schedule buffer on device %d", c->device);
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  if (nr) HIPCHK(hipMemcpy(ds, schedule, (size_t)n_steps * nr * sizeof(int32_t), hipMemcpyHostToDevice));
  return replay_from(c, r, n_steps, schedule, nr ? ds : nullptr);
}

int srs_channel_ca(srs_ctx* c, int32_t r, double* ca_ryr_cyt, double* ca_ryr_jsr, double* ca_lcc) {
  int rc = check_real(c, r);
  if (rc) return rc;
  const RealDesc& d = c->reals[r].desc;
  const int n = 2 * d.n_ryr + d.n_lcc;
  if (n == 0) return SRS_OK;
  HIPCHK(hipSetDevice(c->device));
  double* tmp;
  HIPCHK(hipMalloc(&tmp, n * sizeof(double)));
  hipLaunchKernelGGL(k_channel_ca, dim3(1), dim3(256), 0, c->stream, c->d_desc, c->d_live, r, tmp);
  std::vector<double> h(n);
  hipError_t e = hipStreamSynchronize(c->stream);
  if (e == hipSuccess) e = hipMemcpy(h.data(), tmp, n * sizeof(double), hipMemcpyDeviceToHost);
  (void)hipFree(tmp);
  if (e != hipSuccess) return srs::fail(SRS_E_HIP, "channel Ca: %s", hipGetErrorString(e));
  if (ca_ryr_cyt) memcpy(ca_ryr_cyt, h.data(), d.n_ryr * sizeof(double));
  if (ca_ryr_jsr) memcpy(ca_ryr_jsr, h.data() + d.n_ryr, d.n_ryr * sizeof(double));
  if (ca_lcc) memcpy(ca_lcc, h.data() + 2 * d.n_ryr, d.n_lcc * sizeof(double));
  return SRS_OK;
}

int srs_records_read(srs_ctx* c, int32_t r, float* out, int32_t max_records, int32_t* n_records, int32_t* rec_len) {
  int rc = check_real(c, r);
  if (rc) return rc;
  const RealDesc& d = c->reals[r].desc;
  RealLive lv;
  if ((rc = live_rw(c, r, &lv, false))) return rc;
  if (rec_len) *rec_len = d.rec_len;
  if (lv.rec_overflow) return srs::fail(SRS_E_STATE, "device record buffer overflowed (capacity %d)", d.rec_cap);
  const int n = std::min(lv.rec_count, max_records);
  if (n > 0 && out) HIPCHK(hipMemcpy(out, d.rec, (size_t)n * d.rec_len * sizeof(float), hipMemcpyDeviceToHost));
  if (n_records) *n_records = n;
  // keep any records that did not fit
  const int rest = lv.rec_count - n;
  if (n == 0) return SRS_OK;
  if (rest > 0) {
    std::vector<float> tail((size_t)rest * d.rec_len);
    HIPCHK(hipMemcpy(tail.data(), d.rec + (size_t)n * d.rec_len, tail.size() * sizeof(float), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(d.rec, tail.data(), tail.size() * sizeof(float), hipMemcpyHostToDevice));
  }
  // Only the record count changes: a finished realization whose records
  // are drained stays finished, so the sweep's tile list and the captured
  // graphs remain valid (a full live-state write would restore the tile
  // list and drop them).
  const int32_t cnt = rest;
  HIPCHK(hipMemcpy((char*)(c->d_live + r) + offsetof(RealLive, rec_count), &cnt, sizeof cnt, hipMemcpyHostToDevice));
  return SRS_OK;
}

int srs_ctx_sync(srs_ctx* c) {
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  return SRS_OK;
}

int srs_real_info(srs_ctx* c, int32_t r, int32_t* n_ele, int32_t* n_ryr, int32_t* n_lcc) {
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (r < 0 || r >= (int32_t)c->reals.size()) return srs::fail(SRS_E_ARG, "realization %d out of range", r);
  const HostReal& hr = c->reals[r];
  if (n_ele) *n_ele = c->meshes[hr.mesh]->n;
  if (n_ryr) *n_ryr = (int32_t)hr.ryr_ele.size();
  if (n_lcc) *n_lcc = (int32_t)hr.lcc_ele.size();
  return SRS_OK;
}

int srs_last_timing(srs_ctx* c, double* total_ms, double* sweep_ms) {
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (total_ms) *total_ms = c->last_total_ms;
  if (sweep_ms) *sweep_ms = c->last_sweep_ms;
  return SRS_OK;
}

int srs_time_sweep(srs_ctx* c, int32_t reps, double* sweep_ms, double* gating_ms) {
  // Real steps (sweep + gating, state advances), with HIP events on the
  // context's stream bracketing each kernel separately.
  srs::clear_error();
  if (!c || !c->finalized) return srs::fail(SRS_E_STATE, "context not finalized");
  if (reps <= 0) return srs::fail(SRS_E_ARG, "reps must be > 0");
  HIPCHK(hipSetDevice(c->device));
  bool gated;
  int cur;
  int rc = gated_start(c, &gated, &cur);
  if (rc) return rc;
  std::vector<hipEvent_t> ev(3 * reps);
  for (auto& e : ev) HIPCHK(hipEventCreate(&e));
  const uint32_t gmode = G_AFTER_SWEEP;
  for (int k = 0; k < reps; ++k) {
    HIPCHK(hipEventRecord(ev[3 * k], c->stream));
    // the kernels srs_explicit_step runs: with the gated sweep, each launch
    // also gates the step before it, and the gating after the last one is
    // the whole gating time of the reps
    if (gated) launch_gated(c, cur ^ (k & 1), k ? gmode : 0u, false);
    else launch_sweep(c);
    HIPCHK(hipEventRecord(ev[3 * k + 1], c->stream));
    if (!gated || k == reps - 1) {
      hipLaunchKernelGGL(k_gate, dim3((unsigned)c->reals.size()), dim3(GATE_THREADS), 0, c->stream, c->d_desc,
                         c->d_live, gmode);
      HIPCHK(hipEventRecord(ev[3 * k + 2], c->stream));
    }
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(c->stream));
  double s = 0, g = 0;
  for (int k = 0; k < reps; ++k) {
    float a = 0, b = 0;
    HIPCHK(hipEventElapsedTime(&a, ev[3 * k], ev[3 * k + 1]));
    if (!gated || k == reps - 1) HIPCHK(hipEventElapsedTime(&b, ev[3 * k + 1], ev[3 * k + 2]));
    s += a;
    g += b;
  }
  for (auto& e : ev) (void)hipEventDestroy(e);
  c->last_sweep_ms = s / reps;
  if (sweep_ms) *sweep_ms = s / reps;
  if (gating_ms) *gating_ms = g / reps;
  return SRS_OK;
}

}  // extern "C"
#endif  // SRS_UNIT == 0
