// adjoint.hip -- schedule recording, replayed segments and the adjoint of
// the frozen-channel step for line-scan fitting (single realizations and
// batches).  No reference counterpart.
#include "dev_common.h"

#include <functional>

namespace srs_dev {

// Reverse mode of the explicit step with the channel trajectory frozen
// (RyR states from a recorded schedule, LCC states held): for
// X_{n+1} = X_n + dt r(X_n; theta), lambda_n = lambda_{n+1} + dt J^T lambda_{n+1}
// and dL/dtheta += dt (dr/dtheta)^T lambda_{n+1}.  The diffusion operator
// satisfies V_i A_ij = V_j A_ji (both equal the face coefficient), so
// (A^T y)_j = V_j (A (y / V))_j: the transpose is another gather over the same
// rows.  The stored adjoint is m = lambda / V0, so that this gather reads it as
// it is (divided by the SL buffer's beta in the few SL elements); within an
// element the recursion is linear in lambda and keeps its form, and the
// gradient terms take one factor V0.  Single-realization layout (quads, then
// the TnC and CSQ planes); a launch covers the realizations of a table, one
// workgroup row (blockIdx.y) each, with row y's adjoint and state arrays at y
// times their size.
constexpr int ADJ_NT = 13;   // D_CA, D_DYE, kon/koff of CaM, TnC, ATP, Fluo, V_RYR, A_P, K_D_SL_HI
constexpr int ADJ_BS = 256;
__constant__ const int kAdjTheta[ADJ_NT] = {SRS_R_D_CA,     SRS_R_D_DYE,     SRS_R_K_ON_CMDN, SRS_R_K_OFF_CMDN,
                                            SRS_R_K_ON_TRPN, SRS_R_K_OFF_TRPN, SRS_R_K_ON_ATP, SRS_R_K_OFF_ATP,
                                            SRS_R_K_ON_DYE, SRS_R_K_OFF_DYE, SRS_R_V_RYR,     SRS_R_A_P,
                                            SRS_R_K_D_SL_HI};

// 1 / beta of the rapid SL buffer (cpu/RunSimulation.cpp:15-22) at an element
// with F_SL, beta = 1 + q (B_hi K_hi / (K_hi + c)^2 + B_lo K_lo / (K_lo + c)^2),
// q = TT area / (V0 1e-15): over the common denominator, one division instead
// of six (a neighbour's w is on the step's critical path).
__device__ __forceinline__ double sl_inv_beta(const double* P, double tt, double v0, double c) {
  const double kh = P[SRS_R_K_D_SL_HI], kl = P[SRS_R_K_D_SL_LO];
  const double eh = kh + c, el = kl + c, eh2 = eh * eh, el2 = el * el;
  const double D = eh2 * el2 * (v0 * 1e-15);
  return D / (D + tt * (P[SRS_R_B_TOT_SL_HI] * kh * el2 + P[SRS_R_B_TOT_SL_LO] * kl * eh2));
}
// Derivatives of beta in c and in K_D_SL_HI.
struct SlDer { double dc, dkh; };
__device__ __forceinline__ SlDer sl_derivs(const double* P, double tt, double v0, double c) {
  const double q = tt / (v0 * 1e-15), kh = P[SRS_R_K_D_SL_HI], kl = P[SRS_R_K_D_SL_LO];
  const double eh = kh + c, el = kl + c, r = 1.0 / (eh * el), ih = r * el, il = r * eh;
  const double hi = q * P[SRS_R_B_TOT_SL_HI] * ih * ih * ih, lo = q * P[SRS_R_B_TOT_SL_LO] * il * il * il;
  return SlDer{-2.0 * (hi * kh + lo * kl), hi * (c - kh)};
}

// The loss source of one scan sample at element j: sum_i gcoef_i w(c_j - p_i)
// over points within 1 um (the blur's PSF, linescan/parameters.h:60-62), with
// the blur's own points and weights (the cell's run of points within the
// cut-off).  Every lane of the wavefront calls it (valid false: no element,
// sum zero).  The loop runs over the points any lane can reach, the same for
// the whole wavefront, so gcoef_i is one uniform load per point (a weight
// outside a lane's own run is never used, so it may be anything).
template <bool WALK>
__device__ __forceinline__ double scan_adj_run(const ScanGeo& g, const ScanCell& c, int n_f,
                                               const double* __restrict__ gcoef, int lo, int hi, int i_lo, int i_hi) {
  double s = 0.0;
  for (int base = scan_seg(lo); base <= hi; base += SCAN_SEG)
    scan_walk<WALK>(g, c, base, 1.0, [&](int a, int b) { return base + a <= hi && base + b >= lo; },
                    [&](int m, double t) {
                      const int i = base + m;
                      const double gi = gcoef[min(i, n_f - 1)] * scan_power<WALK>(g, m);
                      if (i >= i_lo && i <= i_hi) s += gi * t;
                    });
  return s;
}

__device__ __forceinline__ double scan_adj_sum(const double* __restrict__ cen, const ScanGeo& g, int n_f,
                                               const double* __restrict__ gcoef, size_t np, int j, bool valid) {
  int i_lo = n_f, i_hi = -1;
  ScanCell c{0.0, 0.0, 0.0, 0.0};
  if (valid) {
    const double cx = cen[j], cy = cen[np + j], cz = cen[2 * np + j];
    scan_point_range(g, n_f, cx, cy, cz, &i_lo, &i_hi);
    c = scan_cell(g, cx, cy, cz);
    scan_exact_range(g, c, &i_lo, &i_hi);
  }
  int lo = i_lo <= i_hi ? i_lo : n_f, hi = i_lo <= i_hi ? i_hi : -1;
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
  }
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  if (lo > hi) return 0.0;
  return g.walk ? scan_adj_run<true>(g, c, n_f, gcoef, lo, hi, i_lo, i_hi)
                : scan_adj_run<false>(g, c, n_f, gcoef, lo, hi, i_lo, i_hi);
}

// The loss source of a scan sample taken after n steps (SCAN), added to
// lambda_n.
struct AdjScan {
  const double* cen;    // scan cell centres [3][np]
  const double* gcoef;  // the sample's loss coefficients per point
  ScanGeo g;
  int n_f, gstride;
};

// The tiles of each chiplet's workgroups lie next to each other (the grid's
// remainder modulo eight keeps its place): its L2 then holds most neighbours
// (8.5 against 9.2 us per step on the 56,250-element mesh when it was measured,
// the same on eight 927,816-element members).
__device__ __forceinline__ int xcd_run(int bid, int grid) {
  const int whole = grid / NXCD * NXCD;
  return bid < whole ? xcd_tile(bid, whole) : bid;
}

// m_n (lambda_n / V0) and the theta-gradient partials of one step.  The
// transposed diffusion gathers w = (m_Ca / beta, m_ATP, m_CaM, m_Fluo) of
// m_{n+1} and this step's state, each element its neighbours' itself.
// Bound by memory traffic and the gathers' lines: m, X and the rows in and m
// out are 1.16 GB per step of eight 927,816-element members, 211 us at the
// 5.5 TB/s that a launch of this mix of reads and writes reaches; the step
// takes 229 us, and 309 with lambda itself stored, whose gather read 1/V0 as
// well or w written by a pass of its own.  The neighbours staged in LDS with the sweep's halo lists are
// slower (251 us, and 9.9 against 9.2 us on the 56,250-element mesh): the
// registers that hold the gradient sums leave four wavefronts per SIMD, too
// few to cover a barrier, and the second copy of m fits the cache.
template <bool CLASS, bool SCAN, bool NTS, int QB>
__device__ __forceinline__ void adj_step(const RealDesc* __restrict__ D, const RealLive* __restrict__ L,
                                         const int32_t* __restrict__ rid, const double* __restrict__ X,
                                         const double* __restrict__ lam, int64_t step, double* __restrict__ lam_out,
                                         double* __restrict__ gpart, const AdjScan& sc) {
  constexpr Quads<QB> lay;
  __shared__ double red[ADJ_BS / 64][ADJ_NT][16];  // gradient partials per wavefront and lane modulo 16
  const int r = rid[blockIdx.y];
  const RealDesc& d = D[r];
  const RealLive& l = L[r];
  const int tile = xcd_run(blockIdx.x, gridDim.x);
  const int j = tile * ADJ_BS + threadIdx.x;
  const size_t np = d.np;
  X += blockIdx.y * 6 * np;
  lam += blockIdx.y * 6 * np;
  lam_out += blockIdx.y * 6 * np;
  // the tile's running partials (16 threads per component), loaded now so the
  // final update waits on no load
  const bool sums = threadIdx.x < ADJ_NT * 16;
  double* gsum = gpart + ((size_t)blockIdx.y * gridDim.x + tile) * ADJ_NT + (threadIdx.x >> 4);
  const double gp_old = sums ? *gsum : 0.0;
  // RyR states during this step: row `step` of the frozen schedule
  const int32_t* ryr = d.n_ryr ? d.sched + step * d.n_ryr : nullptr;
  double gr[ADJ_NT];
#pragma unroll
  for (int k = 0; k < ADJ_NT; ++k) gr[k] = 0.0;
  // the element's operator row, state, m_{n+1} and its neighbours' w
  const bool in = j < d.n;
  Geo g{};
  d4 m0 = {0.0, 0.0, 0.0, 0.0}, mu = {0.0, 0.0, 0.0, 0.0};
  double V0 = 1.0, u = 0.0, ttj = 0.0, inv_beta = 1.0;
  if (in) {
    g = load_geo_nbr<CLASS>(d, j);
    m0 = ld_quad(gp(X), lay, j);
    mu = ld_quad(gp(lam), lay, j);
    V0 = gp(d.V0)[j];
    u = mu.x;
    if (g.f & F_SL) {
      ttj = gp(d.tt)[j];
      inv_beta = sl_inv_beta(d.P, ttj, V0, m0.x);
      u = mu.x * inv_beta;
    }
  }
  auto w_at = [&](uint32_t e) -> d4 {
    const uint32_t i = idx_of(e);
    d4 w = ld_quad(gp(lam), lay, i);
    if (e & IDX_SL) w.x *= sl_inv_beta(d.P, gp(d.tt)[i], gp(d.V0)[i], X[lay.ca(i)]);
    return w;
  };
  d4 w1{}, w2{}, w3{}, w4{};
  if (in) w1 = w_at(g.l1), w2 = w_at(g.l2), w3 = w_at(g.l3), w4 = w_at(g.l4);
  // The realization's record of a channel element.  A binary search and the
  // tables it led to were ten loads in a chain: 8.5 -> 7.6 us per step of the
  // 56,250-element mesh, with one division per SL neighbour instead of six.
  int own = -1;
  ChanElem ce{};
  const uint64_t chan = __builtin_amdgcn_ballot_w64(in && (g.f & F_CHAN));
  if (chan) {
    own = chan_place(d, j, chan);
    if (own >= 0) ce = d.crec[own];
  }
  // the scan sample's loss source (all lanes of the wavefront take part)
  const double src =
      SCAN ? scan_adj_sum(sc.cen, sc.g, sc.n_f, sc.gcoef + (size_t)blockIdx.y * sc.gstride, np, j, in) : 0.0;
  if (in) {
    const double* P = d.P;
    const double dt = P[SRS_R_T_STEP], dv0 = dt * V0;
    const uint8_t f = g.f;
    const d4 aw = row_sum(g, d4{u, mu.y, mu.z, mu.w}, w1, w2, w3, w4);
    const bool live_tr = lives_tr(f), live_cs = lives_cs(f);
    const double bT = live_tr ? X[4 * np + j] : 0.0, bC = live_cs ? X[5 * np + j] : 0.0;
    // the TnC and CSQ adjoints change only where the buffer lives (troponin
    // cytosol, jSR); both adjoint buffers start at zero, so elsewhere they stay
    // zero and those planes are neither read nor written
    const double muT = live_tr ? lam[4 * np + j] : 0.0, muC = live_cs ? lam[5 * np + j] : 0.0;
    const double c = m0.x, bA = m0.y, bM = m0.z, bD = m0.w;

    // transposed diffusion: dt D_s (A w_s)_j
    double lc = mu.x + dt * P[SRS_R_D_CA] * aw.x;
    double la = mu.y + dt * P[SRS_R_D_ATP] * aw.y;
    double lm = mu.z + dt * P[SRS_R_D_CMDN] * aw.z;
    double ld = mu.w + dt * P[SRS_R_D_DYE] * aw.w;
    double lT = muT, lC = muC;

    // The D gradients sum V0_j u_j (A c)_j and V0_j m_Fluo,j (A b_Fluo)_j over the
    // mesh; V_i A_ij = V_j A_ji turns those sums into sum_j c_j V0_j (A w_Ca)_j and
    // sum_j b_Fluo,j V0_j (A w_Fluo)_j, terms of the element alone.  So the
    // neighbours' states are gathered only for an SL element, whose SL terms
    // need its full Ca rate before the division (rca; unused elsewhere).
    double ac = 0.0;
    if (f & F_SL) {
      auto ca_at = [&](uint32_t e) { return X[lay.ca(idx_of(e))]; };
      ac = c * g.a0 + ca_at(g.l1) * g.a1 + ca_at(g.l2) * g.a2 + ca_at(g.l3) * g.a3 + ca_at(g.l4) * g.a4;
    }
    // boundary rates are D times a D-free plane: they enter the D gradients
    const double bu_c = (f & F_BR) ? br_unit(d.br_mesh[j], d.brd[0]) : 0.0;
    const double bu_d = (f & F_BR) ? br_unit(d.br_mesh[np + j], d.brd[1]) : 0.0;
    double rca = P[SRS_R_D_CA] * ac + ((f & F_BR) ? d.br[j] : 0.0);
    gr[0] += dv0 * (c * aw.x + u * bu_c);       // D_CA
    gr[1] += dv0 * (bD * aw.w + mu.w * bu_d);   // D_DYE
    if (!(f & F_JSR)) {
      if (f & F_TROPC) {
        const double kon = P[SRS_R_K_ON_TRPN], koff = P[SRS_R_K_OFF_TRPN], B = P[SRS_R_B_TOT_TRPN];
        const double r = kon * (B - bT) * c - koff * bT;
        rca -= r;
        lc += dt * (muT - u) * kon * (B - bT);
        lT += dt * (muT - u) * (-kon * c - koff);
        gr[4] += dv0 * (muT - u) * (B - bT) * c;
        gr[5] += dv0 * (muT - u) * (-bT);
        // SERCA, cpu/RunSimulation.cpp:82-90
        const double kdi = P[SRS_R_K_D_I];
        double K = c / kdi;
        K = K * K;
        const double dK = 2.0 * (c / kdi) / kdi;
        const double Nn = K * K * 3.24873e12 + K * l.serca[3] - l.serca[4];
        const double Dn = l.serca[0] + K * l.serca[1] + K * K * l.serca[2];
        const double v = Nn / Dn;
        const double dv = ((2 * K * 3.24873e12 + l.serca[3]) * Dn - Nn * (l.serca[1] + 2 * K * l.serca[2])) / (Dn * Dn);
        rca -= (2e-3) * v * P[SRS_R_A_P];
        lc += dt * (-u) * (2e-3) * P[SRS_R_A_P] * dv * dK;
        gr[11] += dv0 * u * (-(2e-3) * v);
      }
      const double konD = P[SRS_R_K_ON_DYE], koffD = P[SRS_R_K_OFF_DYE], BD = P[SRS_R_B_TOT_DYE];
      const double rD = konD * (BD - bD) * c - koffD * bD;
      rca -= rD;
      lc += dt * (mu.w - u) * konD * (BD - bD);
      ld += dt * (mu.w - u) * (-konD * c - koffD);
      gr[8] += dv0 * (mu.w - u) * (BD - bD) * c;
      gr[9] += dv0 * (mu.w - u) * (-bD);
      const double konA = P[SRS_R_K_ON_ATP], koffA = P[SRS_R_K_OFF_ATP], BA = P[SRS_R_B_TOT_ATP];
      const double rA = konA * (BA - bA) * c - koffA * bA;
      rca -= rA;
      lc += dt * (mu.y - u) * konA * (BA - bA);
      la += dt * (mu.y - u) * (-konA * c - koffA);
      gr[6] += dv0 * (mu.y - u) * (BA - bA) * c;
      gr[7] += dv0 * (mu.y - u) * (-bA);
      const double konM = P[SRS_R_K_ON_CMDN], koffM = P[SRS_R_K_OFF_CMDN], BM = P[SRS_R_B_TOT_CMDN];
      const double rM = konM * (BM - bM) * c - koffM * bM;
      rca -= rM;
      lc += dt * (mu.z - u) * konM * (BM - bM);
      lm += dt * (mu.z - u) * (-konM * c - koffM);
      gr[2] += dv0 * (mu.z - u) * (BM - bM) * c;
      gr[3] += dv0 * (mu.z - u) * (-bM);
    } else {
      const double kon = P[SRS_R_K_ON_CSQN], koff = P[SRS_R_K_OFF_CSQN], B = P[SRS_R_B_T_JSR];
      const double r = kon * (B - bC) * c - koff * bC;
      rca -= r;
      rca += (l.ca_nsr - c) * P[SRS_R_V_REFILL];
      lc += dt * ((muC - u) * kon * (B - bC) - u * P[SRS_R_V_REFILL]);
      lC += dt * (muC - u) * (-kon * c - koff);
    }
    if (own >= 0) {
      const double a = P[SRS_R_V_RYR] * P[SRS_R_V_CELL];
      ChanEntry en = ce.first;
      for (int e = ce.e0;;) {
        const int ch = en.code;
        if (ch >= 0) {
          const int p = (ch & 1) ? en.cyt : en.jsr;  // the partner element
          if (ryr[ch >> 1]) {
            const double xj = X[lay.ca(en.jsr)], xc = X[lay.ca(en.cyt)];
            double up = lam[lay.ca(p)];
            if (en.sl & ((ch & 1) ? 2 : 1))
              up *= sl_inv_beta(P, gp(d.tt)[p], gp(d.V0)[p], (ch & 1) ? xc : xj);
            const double dc = xj - xc;
            const double J = a * dc;
            lc += dt * (a / V0) * (up - u);
            if (ch & 1) {  // jSR side: r -= J / V0_jsr
              rca -= J / V0;
            } else {       // cleft side: r += J / V0_cyt
              rca += J / V0;
              gr[10] += dt * P[SRS_R_V_CELL] * dc * (u - up);
            }
          }
        } else {
          const int i = -ch - 1;
          if (srs_lcc_open(d.lcc_state[i], d.lccv_state[i])) {
            rca += srs_lcc_flux_raw(l.vm, c, P[SRS_R_CA_0]) / V0;
            lc += dt * u * srs_lcc_flux_raw(l.vm, 1.0, 0.0) / V0;
          }
        }
        if (++e >= ce.e1) break;
        en = d.centry[e];
      }
    }
    if (f & F_SL) {
      const SlDer sd = sl_derivs(P, ttj, V0, c);
      const double k = mu.x * (-rca * inv_beta * inv_beta);
      lc += dt * k * sd.dc;
      gr[12] += dv0 * k * sd.dkh;
    }
    if (SCAN) ld += src;
    st_quad<NTS>(gpw(lam_out), lay, j, d4{lc, la, lm, ld});
    if (live_tr) stg<NTS>(gpw(lam_out) + 4 * np + j, lT);
    if (live_cs) stg<NTS>(gpw(lam_out) + 5 * np + j, lC);
  }
  // block reduction of the gradient partials, accumulated per block, in a fixed
  // order.  A matrix instruction with a matrix of ones adds the four lanes l,
  // l + 16, l + 32, l + 48 of a wavefront in FP64, on the matrix cores instead
  // of twelve lane moves and additions per component; the rest goes through
  // LDS, 16 sums per wavefront and component.  A channel or SL component that
  // is zero in every lane is not summed.
  typedef double v4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < ADJ_NT; ++k) {
    double v = 0.0;
    if ((k != 10 && k != 12) || __builtin_amdgcn_ballot_w64(gr[k] != 0.0)) {
      const v4 z = {0.0, 0.0, 0.0, 0.0};
      v = __builtin_amdgcn_mfma_f64_16x16x4f64(1.0, gr[k], z, 0, 0, 0)[0];
    }
    if (lane < 16) red[wave][k][lane] = v;
  }
  __syncthreads();
  if (sums) {
    const int k = threadIdx.x >> 4, q = threadIdx.x & 15;
    double s = red[0][k][q];
#pragma unroll
    for (int w = 1; w < ADJ_BS / 64; ++w) s += red[w][k][q];
    s = row_sum_dpp(s);
    if (q == 15) *gsum = gp_old + s;
  }
}

// At most 128 VGPRs: four wavefronts per SIMD (a budget of five spills 116 B
// per lane: 366 against 280 us per step of eight 927,816-element members).
template <bool CLASS, bool SCAN, bool NTS, int QB>
__global__ __launch_bounds__(ADJ_BS) __attribute__((amdgpu_waves_per_eu(4))) void k_adj_step(
    const RealDesc* __restrict__ D, const RealLive* __restrict__ L, const int32_t* __restrict__ rid,
    const double* __restrict__ X, const double* __restrict__ lam, int64_t step, double* __restrict__ lam_out,
    double* __restrict__ gpart, AdjScan sc) {
  adj_step<CLASS, SCAN, NTS, QB>(D, L, rid, X, lam, step, lam_out, gpart, sc);
}

using AdjStepFn = void (*)(const RealDesc*, const RealLive*, const int32_t*, const double*, const double*, int64_t,
                           double*, double*, AdjScan);
template <bool CLASS, int QB>
static AdjStepFn adj_step_fn(bool scan, bool nts) {
  if (scan) return nts ? k_adj_step<CLASS, true, true, QB> : k_adj_step<CLASS, true, false, QB>;
  return nts ? k_adj_step<CLASS, false, true, QB> : k_adj_step<CLASS, false, false, QB>;
}
static AdjStepFn adj_step_fn(const srs_ctx* c, bool scan, bool nts) {
  if (c->quad_block == 1) return c->class_all ? adj_step_fn<true, 1>(scan, nts) : adj_step_fn<false, 1>(scan, nts);
  return c->class_all ? adj_step_fn<true, 64>(scan, nts) : adj_step_fn<false, 64>(scan, nts);
}

// The loss gradient of one scan sample in the Fluo adjoint:
// lambda_Fluo,j += V0_j sum_i gcoef_i w(c_j - p_i) over points within 1 um
// (m = lambda / V0).
__global__ __launch_bounds__(ADJ_BS) void k_scan_adj(const RealDesc* __restrict__ D, const int32_t* __restrict__ rid,
                                                     const double* __restrict__ cen, ScanGeo g, int n_f,
                                                     const double* __restrict__ gcoef, int gstride,
                                                     double* __restrict__ lam) {
  const RealDesc& d = D[rid[blockIdx.y]];
  const int j = blockIdx.x * ADJ_BS + threadIdx.x;
  const size_t np = d.np;
  const double s = scan_adj_sum(cen, g, n_f, gcoef + (size_t)blockIdx.y * gstride, np, j, j < d.n);
  if (j >= d.n) return;
  lam += blockIdx.y * 6 * np;
  lam[QuadsOf{(uint32_t)d.qb}.fluo(j)] += s;
}

// Copies the current state (X[cur]) of each realization of a table to slot y
// of a contiguous buffer (to_buf) or back.
__global__ void k_batch_state(const RealDesc* __restrict__ D, const RealLive* __restrict__ L,
                              const int32_t* __restrict__ rid, double* __restrict__ buf, int to_buf) {
  const int r = rid[blockIdx.y];
  const RealDesc& d = D[r];
  const size_t n6 = 6 * (size_t)d.np;
  double* X = d.X[L[r].cur];
  double* B = buf + blockIdx.y * n6;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n6; i += (size_t)gridDim.x * blockDim.x) {
    if (to_buf) B[i] = X[i];
    else X[i] = B[i];
  }
}

// Starts a replayed segment at `step` for each realization of a table: the
// step counter, schedule rows counted from zero, RyR states of row `step`.
__global__ void k_seg_start(const RealDesc* __restrict__ D, RealLive* __restrict__ L, const int32_t* __restrict__ rid,
                            int64_t step) {
  const int r = rid[blockIdx.x];
  const RealDesc& d = D[r];
  for (int i = threadIdx.x; i < d.n_ryr; i += blockDim.x) d.ryr_state[i] = d.sched[step * d.n_ryr + i];
  if (threadIdx.x == 0) {
    L[r].step = step;
    L[r].sched_base = 0;
  }
}

// Row 0 of each realization's recorded schedule: its RyR states now.
__global__ void k_sched_first(const RealDesc* __restrict__ D) {
  const RealDesc& d = D[blockIdx.x];
  for (int i = threadIdx.x; i < d.n_ryr; i += blockDim.x) d.sched[i] = d.ryr_state[i];
}

}  // namespace srs_dev

extern "C" {

int srs_adjoint_theta(int32_t* idx) {
  srs::clear_error();
  if (!idx) return srs::fail(SRS_E_ARG, "null output");
  const int t[ADJ_NT] = {SRS_R_D_CA,     SRS_R_D_DYE,     SRS_R_K_ON_CMDN, SRS_R_K_OFF_CMDN, SRS_R_K_ON_TRPN,
                         SRS_R_K_OFF_TRPN, SRS_R_K_ON_ATP, SRS_R_K_OFF_ATP, SRS_R_K_ON_DYE,  SRS_R_K_OFF_DYE,
                         SRS_R_V_RYR,     SRS_R_A_P,       SRS_R_K_D_SL_HI};
  for (int k = 0; k < ADJ_NT; ++k) idx[k] = t[k];
  return SRS_N_THETA == ADJ_NT ? SRS_OK : srs::fail(SRS_E_STATE, "theta count mismatch");
}

int srs_params_set(srs_ctx* c, int32_t r, const double* reals) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (!reals) return srs::fail(SRS_E_ARG, "null parameters");
  HostReal& hr = c->reals[r];
  memcpy(hr.reals, reals, sizeof(hr.reals));
  memcpy(hr.desc.P, reals, sizeof(hr.desc.P));
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  const HostMesh& hm = *c->meshes[hr.mesh];
  if (!hm.br.empty()) {
    // boundary rates are D Face_C b / V0: at a D other than the one the
    // mesh's rates were built with, the realization steps with rates of its own
    const double D[4] = {reals[SRS_R_D_CA], reals[SRS_R_D_DYE], reals[SRS_R_D_ATP], reals[SRS_R_D_CMDN]};
    if (std::equal(D, D + 4, hm.br_d)) {
      hr.desc.br = hm.d_br;
    } else {
      if (!hr.d_br_own && (rc = dev_alloc(c, &hr.d_br_own, hm.br.size()))) return rc;
      std::vector<double> own(hm.br.size());
      const size_t np = hm.np;
      for (int q = 0; q < 4; ++q)
        for (size_t k = 0; k < np; ++k) own[q * np + k] = br_scaled(hm.br[q * np + k], D[q], hm.br_d[q]);
      HIPCHK(hipMemcpy(hr.d_br_own, own.data(), own.size() * sizeof(double), hipMemcpyHostToDevice));
      hr.desc.br = hr.d_br_own;
    }
  }
  HIPCHK(hipMemcpy(c->d_desc + r, &hr.desc, sizeof(hr.desc), hipMemcpyHostToDevice));
  RealLive lv;
  if ((rc = live_rw(c, r, &lv, false))) return rc;
  serca_terms(lv.ca_nsr, hr.reals, lv.serca);
  return live_rw(c, r, &lv, true);
}

static int single_real(srs_ctx* c, int32_t r) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if (c->reals.size() != 1 || c->group != 1)
    return srs::fail(SRS_E_ARG, "this call needs a context with one realization and group size 1");
  return SRS_OK;
}

// n_steps gated steps of the whole context, recording every realization's RyR
// states per step: realization r's n_steps x n_ryr rows at out + off[r].
static int record_run(srs_ctx* c, int64_t n_steps, int32_t* out_host) {
  const int n_real = (int)c->reals.size();
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  std::vector<RealLive> lv(n_real);
  HIPCHK(hipMemcpy(lv.data(), c->d_live, n_real * sizeof(RealLive), hipMemcpyDeviceToHost));
  std::vector<size_t> off(n_real + 1, 0);
  for (int r = 0; r < n_real; ++r) {
    if (lv[r].done) return srs::fail(SRS_E_ARG, "record schedule: realization %d has finished its protocol", r);
    off[r + 1] = off[r] + (size_t)n_steps * c->reals[r].ryr_ele.size();
  }
  bool gated;
  int cur;
  int rc = gated_start(c, &gated, &cur);
  if (rc) return rc;
  DevMem M;
  int32_t* d_out = nullptr;
  HIPCHK(M.alloc(&d_out, off[n_real]));
  // the gating writes each step's row to the descriptors' schedules
  std::vector<RealDesc> own(n_real), rec(n_real);
  for (int r = 0; r < n_real; ++r) {
    own[r] = rec[r] = c->reals[r].desc;
    rec[r].sched = d_out + off[r];
    rec[r].n_sched = n_steps;
    rec[r].rec_step0 = lv[r].step;
  }
  HIPCHK(hipMemcpy(c->d_desc, rec.data(), n_real * sizeof(RealDesc), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_sched_first, dim3(n_real), dim3(256), 0, c->stream, c->d_desc);
  hipError_t e = hipGetLastError();
  for (int64_t k = 0; k < n_steps && e == hipSuccess; k += 1024) {
    const int64_t m = std::min<int64_t>(1024, n_steps - k);
    launch_steps(c, m, G_AFTER_SWEEP | G_RECORD, gated, cur);  // an even count leaves cur as it was
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  }
  (void)hipStreamSynchronize(c->stream);
  if (e == hipSuccess) e = hipMemcpy(out_host, d_out, off[n_real] * sizeof(int32_t), hipMemcpyDeviceToHost);
  const hipError_t e2 = hipMemcpy(c->d_desc, own.data(), n_real * sizeof(RealDesc), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = e2;
  if (e != hipSuccess) return srs::fail(SRS_E_HIP, "record schedule: %s", hipGetErrorString(e));
  return SRS_OK;
}

int srs_record_schedule(srs_ctx* c, int32_t r, int64_t n_steps, int32_t* schedule) {
  int rc = single_real(c, r);
  if (rc) return rc;
  if (n_steps <= 0) return SRS_OK;
  if (c->reals[r].ryr_ele.empty()) return srs::fail(SRS_E_ARG, "realization has no RyRs");
  if (!schedule) return srs::fail(SRS_E_ARG, "null schedule");
  return record_run(c, n_steps, schedule);
}

int srs_record_schedules(srs_ctx* c, int64_t n_steps, int32_t* schedules) {
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (!c->finalized) return srs::fail(SRS_E_STATE, "context not finalized");
  if (n_steps <= 0) return SRS_OK;
  if (!schedules) return srs::fail(SRS_E_ARG, "null schedules");
  return record_run(c, n_steps, schedules);
}

// Checkpoint plan of the adjoint: L levels of stored states with strides
// K[0] > K[1] > ... > K[L-1], the last being the length of a recomputed
// segment whose every state is kept.  The forward run keeps the state every
// K[0] steps; going backward, each level-l segment is recomputed from its
// checkpoint keeping the states every K[l+1] steps, down to the segments of
// the last level.  A member holds slots[0] + ... + slots[L-1] + K[L-1]
// states, about (L + 1) n^(1/(L+1)) for equal ratios, and every level below
// the first costs one more forward pass.  Each recomputation replays the same
// kernels from the same state, so the plan changes memory and time, never a
// bit of the losses or gradients.
constexpr int ADJ_MAX_LEVELS = 6;
struct AdjPlan {
  int L = 1;
  int64_t K[ADJ_MAX_LEVELS] = {};
  int64_t slots[ADJ_MAX_LEVELS] = {};
  int64_t kept() const {
    int64_t s = 0;
    for (int l = 0; l < L; ++l) s += slots[l];
    return s;
  }
};
// leaf: the recomputed segment's length, 0 = (n_steps)^(1/(L+1)) rounded up.
static AdjPlan adj_plan(int64_t n_steps, int64_t leaf, int L) {
  AdjPlan p;
  p.L = L;
  const double n = (double)std::max<int64_t>(n_steps, 1);
  if (leaf <= 0) leaf = (int64_t)std::ceil(std::pow(n, 1.0 / (L + 1)) - 1e-9);
  leaf = std::max<int64_t>(1, std::min<int64_t>(leaf, std::max<int64_t>(n_steps, 1)));
  p.K[L - 1] = leaf;
  const int64_t r = L > 1 ? std::max<int64_t>(2, (int64_t)std::ceil(std::pow(n / leaf, 1.0 / L) - 1e-9)) : 0;
  for (int l = L - 2; l >= 0; --l) p.K[l] = p.K[l + 1] * r;
  p.slots[0] = (std::max<int64_t>(n_steps, 1) + p.K[0] - 1) / p.K[0];
  for (int l = 1; l < L; ++l) p.slots[l] = (p.K[l - 1] + p.K[l] - 1) / p.K[l];
  return p;
}

// Line-scan loss and adjoint gradient of the realizations `ids` (all on the
// scan's mesh, group size 1; arguments already checked).  Members run in
// sub-batches of at most `max_batch` that step together; every other
// realization is held (done) meanwhile, and all are left as they were.
// Schedules are each member's n_steps x n_ryr rows, concatenated in member
// order; targets are [member][sample][point].
static int loss_grad_run(srs_ctx* c, const std::vector<int32_t>& ids, int32_t scan_id, int64_t n_steps,
                         const int32_t* schedules, int32_t n_samples, const int64_t* sample_steps,
                         const double* targets, int32_t ckpt, int32_t max_batch, double* losses, double* grads,
                         double* scans) {
  const HostScan& S = c->scans[scan_id];
  const HostMesh& hm = *c->meshes[S.mesh];
  const size_t np = hm.np, n6 = 6 * np;
  const int nf = S.n_f, nca = S.n_ca, nout = nca + 2 * nf;
  const int n_mem = (int)ids.size(), n_real = (int)c->reals.size();
  const bool want_grad = grads != nullptr;
  const int nblk = (hm.n + ADJ_BS - 1) / ADJ_BS;
  std::vector<size_t> soff(n_mem + 1, 0);
  size_t max_sched = 0;
  for (int m = 0; m < n_mem; ++m) {
    const size_t k = (size_t)n_steps * c->reals[ids[m]].ryr_ele.size();
    soff[m + 1] = soff[m] + k;
    max_sched = std::max(max_sched, k);
  }
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  size_t mem_free = 0, mem_total = 0;
  HIPCHK(hipMemGetInfo(&mem_free, &mem_total));
  const size_t budget = mem_free / 10 * 9;
  // device bytes per member of a sub-batch under a plan (a loss alone keeps
  // only the start state)
  auto per_member = [&](const AdjPlan& p) {
    return 8 * n6 * (size_t)(want_grad ? p.kept() + p.K[p.L - 1] + 2 : 1) +
           8 * (size_t)n_samples * nout + 8 * (size_t)S.n_blocks * nf + 8 * (size_t)nblk * ADJ_NT +
           8 * (size_t)n_samples * nf + 4 * max_sched + 64;
  };
  // the plan: the tuned number of levels, or the fewest levels (least
  // recomputation) with which the wanted sub-batch fits
  const int want = max_batch > 0 ? std::min(max_batch, n_mem) : 1;
  AdjPlan plan = adj_plan(n_steps, ckpt, std::max(1, c->adj_levels));
  if (want_grad && c->adj_levels == 0) {
    for (int L = 1; L <= ADJ_MAX_LEVELS; ++L) {
      const AdjPlan p = adj_plan(n_steps, L == 1 ? ckpt : 0, L);
      if (L == 1 || budget / per_member(p) > budget / per_member(plan)) plan = p;
      if (budget / per_member(p) >= (size_t)want) {
        plan = p;
        break;
      }
    }
  }
  const size_t per = per_member(plan);
  int bs = max_batch > 0 ? std::min(max_batch, n_mem) : n_mem;
  bs = (int)std::min<size_t>((size_t)bs, budget / per);
  if (bs < 1)
    return srs::fail(SRS_E_ARG, "checkpoint plan (%d level(s), segments of %lld steps) needs %.3g GB per "
                     "realization, %.3g GB free", plan.L, (long long)plan.K[plan.L - 1], per / 1e9, mem_free / 1e9);
  const int64_t K0 = plan.K[0];
  const int64_t n_ck_kept = want_grad ? plan.slots[0] : 1;
  const int64_t leaf = plan.K[plan.L - 1];
  c->adj_last_levels = plan.L;
  for (int l = 0; l < ADJ_MAX_LEVELS; ++l) c->adj_last_strides[l] = l < plan.L ? plan.K[l] : 0;
  c->adj_last_batch = bs;

  // the reverse step's new lambda past the caches once a step's states no longer
  // fit them (eight 927,816-element members, 1.07 GB: 238 -> 234 us per step)
  const bool nts = 8.0 * n6 * bs * 3 > 330e6;

  // everything restored at the end
  std::vector<RealLive> live0(n_real);
  HIPCHK(hipMemcpy(live0.data(), c->d_live, n_real * sizeof(RealLive), hipMemcpyDeviceToHost));
  std::vector<std::vector<int32_t>> ryr0(n_mem);
  for (int m = 0; m < n_mem; ++m) {
    const HostReal& hr = c->reals[ids[m]];
    ryr0[m].resize(hr.ryr_ele.size());
    if (!ryr0[m].empty())
      HIPCHK(hipMemcpy(ryr0[m].data(), hr.desc.ryr_state, ryr0[m].size() * sizeof(int32_t), hipMemcpyDeviceToHost));
  }

  DevMem M;
  double *ck = nullptr, *samp = nullptr, *part = nullptr, *dg = nullptr, *gpart = nullptr;
  double *lam0 = nullptr, *lam1 = nullptr, *seg = nullptr;
  std::vector<double*> ckl(plan.L, nullptr);  // checkpoint levels; ckl[0] = ck, the forward's
  int32_t *d_sched = nullptr, *d_rid = nullptr;
  int2* d_sub_tiles = nullptr;
  const int nt_mesh = (hm.n + c->tile - 1) / c->tile;
  HIPCHK(M.alloc(&ck, (size_t)n_ck_kept * bs * n6));
  ckl[0] = ck;
  HIPCHK(M.alloc(&d_sub_tiles, (size_t)bs * nt_mesh));
  HIPCHK(M.alloc(&samp, (size_t)n_samples * bs * nout));
  HIPCHK(M.alloc(&part, (size_t)bs * S.n_blocks * nf));
  HIPCHK(M.alloc(&d_sched, std::max<size_t>(1, (size_t)bs * max_sched)));
  HIPCHK(M.alloc(&d_rid, (size_t)bs));
  if (want_grad) {
    HIPCHK(M.alloc(&lam0, (size_t)bs * n6));
    HIPCHK(M.alloc(&lam1, (size_t)bs * n6));
    HIPCHK(M.alloc(&seg, (size_t)leaf * bs * n6));
    for (int l = 1; l < plan.L; ++l) HIPCHK(M.alloc(&ckl[l], (size_t)plan.slots[l] * bs * n6));
    HIPCHK(M.alloc(&gpart, (size_t)bs * nblk * ADJ_NT));
    HIPCHK(M.alloc(&dg, (size_t)bs * n_samples * nf));
  }
  const uint32_t gmode = G_AFTER_SWEEP | G_NO_GATING | G_REPLAY;
  const unsigned cp_blocks = (unsigned)std::min<size_t>((n6 + 255) / 256, 2048);
  std::vector<double> sh, gco, gp;
  std::vector<RealLive> lv(n_real);
  std::vector<int2> sub_tiles;
  // the sweep visits only the members' tiles (a held realization's tiles would
  // still cost a dispatch each); the context's own list is put back on every
  // return, before the buffers above are freed
  struct TileRestore {
    srs_ctx* c;
    int2* tiles;
    int n_tiles, grid;
    ~TileRestore() { c->d_tiles = tiles; c->n_tiles = n_tiles; c->grid_sweep = grid; }
  } tile_restore{c, c->d_tiles, c->n_tiles, c->grid_sweep};
  hipError_t e = hipSuccess;
  const int rc = [&]() -> int {
  for (int m0 = 0; m0 < n_mem; m0 += bs) {
    const int nb = std::min(bs, n_mem - m0);
    const dim3 g_adj(nblk, nb), g_cp(cp_blocks, nb);
    if (n_real > 1) {
      sub_tiles.clear();
      for (int y = 0; y < nb; ++y)
        for (int t = 0; t < nt_mesh; ++t) sub_tiles.push_back(make_int2(ids[m0 + y], t));
      HIPCHK(hipMemcpy(d_sub_tiles, sub_tiles.data(), sub_tiles.size() * sizeof(int2), hipMemcpyHostToDevice));
      c->d_tiles = d_sub_tiles;
      c->n_tiles = (int)sub_tiles.size();
      c->grid_sweep = (c->n_tiles + NXCD - 1) / NXCD * NXCD;
    }
    // members replay their schedules from row 0; the rest are held
    for (int q = 0; q < n_real; ++q) {
      lv[q] = live0[q];
      lv[q].done = 1;
    }
    for (int y = 0; y < nb; ++y) {
      const int r = ids[m0 + y];
      lv[r].done = 0;
      lv[r].ffwd = 0;
      lv[r].step = 0;
      lv[r].sched_base = 0;
      HostReal& hr = c->reals[r];
      RealDesc dsc = hr.desc;
      dsc.sched = d_sched + (size_t)y * max_sched;
      dsc.n_sched = n_steps;
      HIPCHK(hipMemcpy(d_sched + (size_t)y * max_sched, schedules + soff[m0 + y],
                       (soff[m0 + y + 1] - soff[m0 + y]) * sizeof(int32_t), hipMemcpyHostToDevice));
      HIPCHK(hipMemcpy(c->d_desc + r, &dsc, sizeof(dsc), hipMemcpyHostToDevice));
    }
    HIPCHK(hipMemcpy(c->d_live, lv.data(), n_real * sizeof(RealLive), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(d_rid, ids.data() + m0, nb * sizeof(int32_t), hipMemcpyHostToDevice));
    auto scan_into = [&](double* out) {
      hipLaunchKernelGGL(k_scan_blur, dim3(S.n_blocks, nb), dim3(SCAN_BS), scan_lds(nf), c->stream, c->d_desc, c->d_live, 0,
                         d_rid, S.d_cen, S.geo, nf, part);
      hipLaunchKernelGGL(k_scan_final, dim3(scan_final_blocks(nf), nb), dim3(SCAN_BS), 0, c->stream, c->d_desc, c->d_live, 0, d_rid,
                         S.n_blocks, nf, nca, part, S.d_pad, S.d_near_f, S.d_near_ca, S.desc.f0, S.desc.c0, out, nout);
    };
    auto ck_at = [&](int l, int64_t k) { return ckl[l] + (size_t)k * nb * n6; };

    // forward, with checkpoints and scan samples; the steps between two of those
    // are one launch each: a single realization's through the gated sweep (whose
    // workgroup 0 replays the step before), several through sweeps that read the
    // schedules
    const bool gated = c->gated && n_real == 1;
    int cur = lv[ids[m0]].cur;
    auto replay_block = [&](int64_t m, int64_t n) {
      if (gated) launch_gated_block(c, m, cur, gmode);
      else launch_replay_block(c, m, n, d_rid, nb);
      cur ^= (int)(m & 1);
    };
    hipLaunchKernelGGL(k_seg_start, dim3(nb), dim3(256), 0, c->stream, c->d_desc, c->d_live, d_rid, (int64_t)0);
    int ks = 0;
    for (int64_t n = 0; n < n_steps && e == hipSuccess;) {
      if (n % K0 == 0 && n / K0 < n_ck_kept)
        hipLaunchKernelGGL(k_batch_state, g_cp, dim3(256), 0, c->stream, c->d_desc, c->d_live, d_rid,
                           ck_at(0, n / K0), 1);
      int64_t next = std::min<int64_t>(n_steps, (n / K0 + 1) * K0);
      if (ks < n_samples && sample_steps[ks] > n) next = std::min<int64_t>(next, sample_steps[ks]);
      const int64_t m = std::min<int64_t>(4096, std::max<int64_t>(1, next - n));
      replay_block(m, n);
      n += m;
      if (ks < n_samples && sample_steps[ks] == n) scan_into(samp + (size_t)(ks++) * nb * nout);
      e = hipGetLastError();
      if (e == hipSuccess && n / 4096 != (n - m) / 4096) e = hipStreamSynchronize(c->stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return srs::fail(SRS_E_HIP, "adjoint forward: %s", hipGetErrorString(e));
    sh.resize((size_t)n_samples * nb * nout);
    if ((e = hipMemcpy(sh.data(), samp, sh.size() * sizeof(double), hipMemcpyDeviceToHost)) != hipSuccess)
      return srs::fail(SRS_E_HIP, "adjoint forward: %s", hipGetErrorString(e));
    // losses and their gradients in the blurred fluorescence
    gco.assign((size_t)nb * n_samples * nf, 0.0);
    const double f0 = S.desc.f0;
    for (int y = 0; y < nb; ++y) {
      const double* tg = targets + (size_t)(m0 + y) * n_samples * nf;
      double Ls = 0.0;
      for (int k = 0; k < n_samples; ++k)
        for (int i = 0; i < nf; ++i) {
          const double dff = sh[((size_t)k * nb + y) * nout + nca + nf + i] / f0 - 1.0;
          const double res = dff - tg[(size_t)k * nf + i];
          Ls += res * res;
          gco[((size_t)y * n_samples + k) * nf + i] = 2.0 * res / f0;
          if (scans) scans[((size_t)(m0 + y) * n_samples + k) * nf + i] = dff;
        }
      losses[m0 + y] = Ls;
    }

    if (want_grad) {
      e = hipMemcpy(dg, gco.data(), gco.size() * sizeof(double), hipMemcpyHostToDevice);
      if (e == hipSuccess) e = hipMemsetAsync(lam0, 0, (size_t)nb * n6 * sizeof(double), c->stream);
      if (e == hipSuccess) e = hipMemsetAsync(lam1, 0, (size_t)nb * n6 * sizeof(double), c->stream);
      if (e == hipSuccess) e = hipMemsetAsync(gpart, 0, (size_t)nb * nblk * ADJ_NT * sizeof(double), c->stream);
      double* lam = lam0;   // lambda_{n+1}
      double* lout = lam1;  // lambda_n
      ks = n_samples - 1;
      // the loss source of a sample after the last step; the step kernel
      // adds the others to the lambda it produces
      if (sample_steps[ks] == n_steps) {
        hipLaunchKernelGGL(k_scan_adj, g_adj, dim3(ADJ_BS), 0, c->stream, c->d_desc, d_rid, S.d_cen, S.geo, nf,
                           dg + (size_t)ks * nf, n_samples * nf, lam);
        --ks;
      }
      // a segment of the last level: recompute it from its checkpoint, the
      // sweep writing each state into its slot of the segment, then step
      // backward through it
      auto leaf_back = [&](int64_t s0, int64_t s1, const double* ckq) -> hipError_t {
        hipLaunchKernelGGL(k_seg_start, dim3(nb), dim3(256), 0, c->stream, c->d_desc, c->d_live, d_rid, s0);
        hipError_t e2 = hipMemcpyAsync(seg, ckq, (size_t)nb * n6 * sizeof(double), hipMemcpyDeviceToDevice,
                                       c->stream);
        for (int64_t n = s0; n < s1 - 1 && e2 == hipSuccess; ++n) {
          // from slot n - s0 into slot n - s0 + 1
          const double* from = seg + (size_t)(n - s0) * nb * n6;
          double* to = seg + (size_t)(n - s0 + 1) * nb * n6;
          if (gated) launch_gated(c, 0, n > s0 ? gmode : 0u, false, from, to);
          else launch_replay(c, n, 0, from, to, n6, nt_mesh);
          e2 = hipGetLastError();
        }
        if (gated && s1 - 1 > s0 && e2 == hipSuccess) {
          launch_gate_single(c, gmode);  // moves the live index on
          cur ^= (int)((s1 - 1 - s0) & 1);
          e2 = hipGetLastError();
        }
        for (int64_t n = s1 - 1; n >= s0 && e2 == hipSuccess; --n) {
          const double* Xn = seg + (size_t)(n - s0) * nb * n6;
          const bool scan = ks >= 0 && sample_steps[ks] == n;
          const AdjScan sc{S.d_cen, scan ? dg + (size_t)ks * nf : nullptr, S.geo, nf, n_samples * nf};
          if (scan) --ks;
          const AdjStepFn kern = adj_step_fn(c, scan, nts);
          hipLaunchKernelGGL(kern, g_adj, dim3(ADJ_BS), 0, c->stream, c->d_desc, c->d_live, d_rid, Xn, lam, n, lout,
                             gpart, sc);
          std::swap(lam, lout);
          e2 = hipGetLastError();
        }
        if (e2 == hipSuccess) e2 = hipStreamSynchronize(c->stream);
        return e2;
      };
      // the level-l segments of [a, b), last first; the states at a + q K[l]
      // are in slot q of level l
      std::function<hipError_t(int, int64_t, int64_t)> back = [&](int l, int64_t a, int64_t b) -> hipError_t {
        const int64_t K = plan.K[l];
        hipError_t e2 = hipSuccess;
        for (int64_t q = (b - a + K - 1) / K - 1; q >= 0 && e2 == hipSuccess; --q) {
          const int64_t s0 = a + q * K, s1 = std::min<int64_t>(b, s0 + K);
          if (l == plan.L - 1) {
            e2 = leaf_back(s0, s1, ck_at(l, q));
            continue;
          }
          // recompute [s0, s1) in the members' own state buffers, keeping the
          // next level's checkpoints
          hipLaunchKernelGGL(k_seg_start, dim3(nb), dim3(256), 0, c->stream, c->d_desc, c->d_live, d_rid, s0);
          hipLaunchKernelGGL(k_batch_state, g_cp, dim3(256), 0, c->stream, c->d_desc, c->d_live, d_rid,
                             (double*)ck_at(l, q), 0);
          const int64_t K1 = plan.K[l + 1];
          int64_t queued = 0;
          for (int64_t n = s0; n < s1 && e2 == hipSuccess; n += K1) {
            hipLaunchKernelGGL(k_batch_state, g_cp, dim3(256), 0, c->stream, c->d_desc, c->d_live, d_rid,
                               ck_at(l + 1, (n - s0) / K1), 1);
            replay_block(std::min<int64_t>(K1, s1 - n), n);
            e2 = hipGetLastError();
            queued += K1;
            if (e2 == hipSuccess && queued >= 4096) {
              e2 = hipStreamSynchronize(c->stream);
              queued = 0;
            }
          }
          if (e2 == hipSuccess) e2 = back(l + 1, s0, s1);
        }
        return e2;
      };
      if (e == hipSuccess) e = back(0, 0, n_steps);
      if (e == hipSuccess) {
        gp.resize((size_t)nb * nblk * ADJ_NT);
        e = hipMemcpy(gp.data(), gpart, gp.size() * sizeof(double), hipMemcpyDeviceToHost);
      }
      if (e != hipSuccess) return srs::fail(SRS_E_HIP, "adjoint backward: %s", hipGetErrorString(e));
      for (int y = 0; y < nb; ++y)
        for (int k = 0; k < ADJ_NT; ++k) {
          double sum = 0.0;
          for (int b = 0; b < nblk; ++b) sum += gp[((size_t)y * nblk + b) * ADJ_NT + k];
          grads[(size_t)(m0 + y) * ADJ_NT + k] = sum;
        }
    }
    // the members' states as they were: descriptors (their schedules were this
    // call's) and live state (it names the current buffer) first, then the start
    // state into that buffer
    for (int y = 0; y < nb; ++y) {
      const HostReal& hr = c->reals[ids[m0 + y]];
      HIPCHK(hipMemcpy(c->d_desc + ids[m0 + y], &hr.desc, sizeof(hr.desc), hipMemcpyHostToDevice));
    }
    HIPCHK(hipMemcpy(c->d_live, live0.data(), n_real * sizeof(RealLive), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_batch_state, g_cp, dim3(256), 0, c->stream, c->d_desc, c->d_live, d_rid, ck_at(0, 0), 0);
    HIPCHK(hipStreamSynchronize(c->stream));
  }
  return SRS_OK;
  }();
  // restore descriptors, live state and RyR states (also after a failure)
  for (int m = 0; m < n_mem; ++m) {
    const HostReal& hr = c->reals[ids[m]];
    (void)hipMemcpy(c->d_desc + ids[m], &hr.desc, sizeof(hr.desc), hipMemcpyHostToDevice);
    if (!ryr0[m].empty())
      (void)hipMemcpy(hr.desc.ryr_state, ryr0[m].data(), ryr0[m].size() * sizeof(int32_t), hipMemcpyHostToDevice);
  }
  (void)hipMemcpy(c->d_live, live0.data(), n_real * sizeof(RealLive), hipMemcpyHostToDevice);
  e = hipDeviceSynchronize();
  if (rc == SRS_OK && e != hipSuccess) return srs::fail(SRS_E_HIP, "adjoint restore: %s", hipGetErrorString(e));
  return rc;
}

static int loss_grad_check(srs_ctx* c, int32_t scan_id, int64_t n_steps, int32_t n_samples,
                           const int64_t* sample_steps, const double* target, int32_t ckpt, const void* loss,
                           bool auto_ckpt = false) {
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (!c->finalized) return srs::fail(SRS_E_STATE, "context not finalized");
  if (c->group != 1) return srs::fail(SRS_E_ARG, "the adjoint needs realization groups of size 1");
  if (scan_id < 0 || scan_id >= (int)c->scans.size()) return srs::fail(SRS_E_ARG, "bad scan id %d", scan_id);
  if (c->scans[scan_id].n_f <= 0) return srs::fail(SRS_E_ARG, "the scan has no fluorescence points");
  if (n_steps <= 0 || n_samples <= 0 || !sample_steps || !target || !loss) return srs::fail(SRS_E_ARG, "bad arguments");
  if ((ckpt <= 0 && !(auto_ckpt && ckpt == 0)) || ckpt > 65536)
    return srs::fail(SRS_E_ARG, "checkpoint interval must be 1..65536%s", auto_ckpt ? " or 0" : "");
  for (int k = 0; k < n_samples; ++k)
    if (sample_steps[k] < 1 || sample_steps[k] > n_steps || (k && sample_steps[k] <= sample_steps[k - 1]))
      return srs::fail(SRS_E_ARG, "sample steps must increase within 1..n_steps");
  return SRS_OK;
}

int srs_linescan_loss_grad(srs_ctx* c, int32_t r, int32_t scan_id, int64_t n_steps, const int32_t* schedule,
                           int32_t n_samples, const int64_t* sample_steps, const double* target, int32_t ckpt,
                           double* loss, double* grad) {
  int rc = check_real(c, r);
  if (rc) return rc;
  if ((rc = loss_grad_check(c, scan_id, n_steps, n_samples, sample_steps, target, ckpt, loss))) return rc;
  if (c->reals[r].mesh != c->scans[scan_id].mesh) return srs::fail(SRS_E_ARG, "realization is not on the scan's mesh");
  if (c->reals[r].ext.jsr_diffusion || c->reals[r].ext.b_sr_sites != 0.0)
    return srs::fail(SRS_E_ARG, "realization %d has a model extension on; the adjoint covers the reference model", r);
  if (!c->reals[r].ryr_ele.empty() && !schedule) return srs::fail(SRS_E_ARG, "null schedule");
  return loss_grad_run(c, {r}, scan_id, n_steps, schedule, n_samples, sample_steps, target, ckpt, 1, loss, grad,
                       nullptr);
}

int srs_linescan_loss_grad_batch(srs_ctx* c, int32_t n_real, const int32_t* real_ids, int32_t scan_id,
                                 int64_t n_steps, const int32_t* schedules, int32_t n_samples,
                                 const int64_t* sample_steps, const double* targets, int32_t ckpt, int32_t max_batch,
                                 double* losses, double* grads, double* scans) {
  int rc = c ? SRS_OK : srs::fail(SRS_E_ARG, "null context");
  if (rc) return rc;
  if (n_real <= 0 || !real_ids) return srs::fail(SRS_E_ARG, "no realizations");
  if ((rc = loss_grad_check(c, scan_id, n_steps, n_samples, sample_steps, targets, ckpt, losses, true))) return rc;
  std::vector<int32_t> ids(real_ids, real_ids + n_real);
  std::vector<char> seen(c->reals.size(), 0);
  bool any_ryr = false;
  for (int32_t r : ids) {
    if ((rc = check_real(c, r))) return rc;
    if (seen[r]++) return srs::fail(SRS_E_ARG, "realization %d listed twice", r);
    if (c->reals[r].mesh != c->scans[scan_id].mesh)
      return srs::fail(SRS_E_ARG, "realization %d is not on the scan's mesh", r);
    if (c->reals[r].ext.jsr_diffusion || c->reals[r].ext.b_sr_sites != 0.0)
      return srs::fail(SRS_E_ARG, "realization %d has a model extension on; the adjoint covers the reference model", r);
    any_ryr |= !c->reals[r].ryr_ele.empty();
  }
  if (any_ryr && !schedules) return srs::fail(SRS_E_ARG, "null schedules");
  return loss_grad_run(c, ids, scan_id, n_steps, schedules, n_samples, sample_steps, targets, ckpt, max_batch, losses,
                       grads, scans);
}

int srs_adjoint_last_plan(srs_ctx* c, int32_t* levels, int64_t* strides, int32_t* sub_batch) {
  srs::clear_error();
  if (!c) return srs::fail(SRS_E_ARG, "null context");
  if (levels) *levels = c->adj_last_levels;
  if (strides)
    for (int l = 0; l < ADJ_MAX_LEVELS; ++l) strides[l] = c->adj_last_strides[l];
  if (sub_batch) *sub_batch = c->adj_last_batch;
  return SRS_OK;
}


}  // extern "C"
