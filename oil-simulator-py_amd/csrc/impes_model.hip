// IMPES step kernels and their host orchestration.
#include "fgmres_dev.h"
#include "impes_model.h"
#include "model_dev.h"

#include <cstring>

#include <algorithm>
#include <cmath>

// Products and sums are rounded separately (no fused multiply-add), as in the
// numpy restatement: the substep count is a ceil() of a global maximum that can
// sit exactly on an integer (a choked well filling its saturation window).
#pragma clang fp contract(off)

namespace impes {

namespace {
using namespace model_dev;
// Sums of NV values (a power of two) over the workgroup, in a fixed order: a wave folds
// all its values by halving (wave_fold), LDS joins the waves. Thread q < NV returns the
// sum of value q. `lds`: NV slots per wave.
template <int NV>
__device__ __forceinline__ double block_fold(double (&v)[NV], double* lds) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const double s = wave_fold(v);
  if (lane % (kWave / NV) == 0) lds[wid * NV + fold_index<NV>(lane)] = s;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x < NV)
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) r += lds[w * NV + threadIdx.x];
  return r;
}

constexpr int kLedgerQ = 10;  // mass(6) + volume dV_w, dV_g, clamp_w, clamp_g
constexpr int kFoldQ = 16;    // their slots in a fold (a power of two)

// ---------------------------------------------------------------- transmissibility
// simulation.py:52-74: T = 2 k1 k2/(k1 + k2 + 1e-15) * area / distance
__global__ void k_trans(GridDev G, const double* __restrict__ kx, const double* __restrict__ ky,
                        const double* __restrict__ kz, const double* __restrict__ pv_in, double* __restrict__ tx,
                        double* __restrict__ ty, double* __restrict__ tz, double* __restrict__ pv) {
  const long long n = (long long)G.nx * G.ny * G.nz;
  CELL_LOOP(c, n) {
    int i, j, k;
    ijk(G, c, i, j, k);
    double t = 0.0;
    // no face between two stacked reservoirs (their last and first x-layers)
    if (i < G.nx - 1 && !(G.env_nx > 0 && (i + 1) % G.env_nx == 0)) {
      const double a = kx[c], b = kx[c + G.sx];
      t = 2 * a * b / (a + b + 1e-15) * G.dy * G.dz / G.dx;
    }
    tx[c] = t;
    t = 0.0;
    if (j < G.ny - 1) {
      const double a = ky[c], b = ky[c + G.sy];
      t = 2 * a * b / (a + b + 1e-15) * G.dx * G.dz / G.dy;
    }
    ty[c] = t;
    t = 0.0;
    if (k < G.nz - 1) {
      const double a = kz[c], b = kz[c + 1];
      t = 2 * a * b / (a + b + 1e-15) * G.dx * G.dy / G.dz;
    }
    tz[c] = t;
    pv[c] = pv_in[c];
  }
}

// ---------------------------------------------------------------- pressure step
// simulation.py:871-882 + fluid properties at the previous pressure
// acc and mt always; grav = mw rw + mo ro + mg rg and pc, mo are what the assembly
// reads (with gravity, with capillarity); the phases' own mobilities and densities only
// where they are asked for (the reverse sweep; nullptr otherwise). At 1M
// cells 42 us; 61 us with all of them written and one table search after the other.
struct PressureProps {
  double *mt, *acc, *grav, *pc, *mo;
  double *mw, *mg, *rw, *ro, *rg;
};
__global__ __launch_bounds__(kBlock) void k_props_pressure(GridDev G, FluidParams F, PvtDev T, double dt,
                                                           const double* __restrict__ p,
                                                           const double* __restrict__ sw,
                                                           const double* __restrict__ sg,
                                                           const double* __restrict__ pv, PressureProps Q) {
  const long long n = (long long)G.nx * G.ny * G.nz;
  CELL_LOOP(c, n) {
    const double pp = p[c], s_w = sw[c], s_g = sg[c];
    double kro, krw, krg, muo, muw, mug;
    relperms(F, s_w, s_g, kro, krw, krg);
    PvtAt at[4] = {};
    if (T.n > 0) {
      double q[4], ct[3];
      ct_pressures(pp, ct);
      q[0] = pp;
      for (int i = 0; i < 3; ++i) q[i + 1] = ct[i];
      pvt_locate(T, q, at);
    }
    viscosities(F, T, pp, muo, muw, mug, at);
    const double a = krw / muw, o = kro / muo, g = krg / mug;
    Q.mt[c] = a + o + g;
    if (Q.mo) Q.mo[c] = o;
    if (Q.mw) {
      Q.mw[c] = a;
      Q.mg[c] = g;
    }
    if (G.gravity) {
      double r1, r2, r3;
      densities(F, T, pp, r1, r2, r3, at);
      Q.grav[c] = a * r1 + o * r2 + g * r3;
      if (Q.rw) {
        Q.rw[c] = r1;
        Q.ro[c] = r2;
        Q.rg[c] = r3;
      }
    }
    if (F.pc_scale > 0.0) Q.pc[c] = pc_ow(F, s_w);
    Q.acc[c] = pv[c] * total_compressibility(F, T, pp, s_w, s_g, at + 1) / dt;
  }
}

// _build_pressure_matrix_vectorized (:1546-1580) + _build_pressure_rhs (:1582-1620) in face form:
// each cell visits its six faces (coefficients recomputed on both sides, no atomics).
// Every load is made whether its face exists or not (a missing neighbour reads the cell
// itself), so that a wave waits for them once and not face after face; each XCD takes
// one run of cells. At 1M cells 31 us; 52 us with a wait per face.
__global__ __launch_bounds__(kBlock) void k_assemble(
    GridDev G, FluidParams F, const double* __restrict__ p, const double* __restrict__ tx,
    const double* __restrict__ ty, const double* __restrict__ tz, const double* __restrict__ mt,
    const double* __restrict__ grav, const double* __restrict__ mo, const double* __restrict__ pc,
    const double* __restrict__ acc, double* __restrict__ diag, double* __restrict__ ox, double* __restrict__ oy,
    double* __restrict__ oz, double* __restrict__ b, double* __restrict__ extra, double* __restrict__ dinv) {
  const long long n = (long long)G.nx * G.ny * G.nz;
  const bool with_pc = F.pc_scale > 0.0, with_g = G.gravity != 0;
  for (long long c = xcd_block() * kBlock + threadIdx.x; c < n; c += (long long)gridDim.x * kBlock) {
    int i, j, k;
    ijk(G, c, i, j, k);
    const bool up[3] = {i < G.nx - 1, j < G.ny - 1, k < G.nz - 1}, dn[3] = {i > 0, j > 0, k > 0};
    const long long st[3] = {G.sx, G.sy, 1};
    const double* const T[3] = {tx, ty, tz};
    // face f: axis f / 2, to the upper (even) or the lower (odd) neighbour
    double pn[6], tn[6], mn[6], on[6], cn[6], gn[2] = {0.0, 0.0}, gc = 0.0;
    const double pcc = p[c], mc = mt[c], a = acc[c];
    const double oc = with_pc ? mo[c] : 0.0, cc = with_pc ? pc[c] : 0.0;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const int ax = f >> 1;
      const long long o = f & 1 ? (dn[ax] ? c - st[ax] : c) : (up[ax] ? c + st[ax] : c);
      pn[f] = p[o];
      mn[f] = mt[o];
      tn[f] = T[ax][f & 1 ? o : c];
      on[f] = with_pc ? mo[o] : 0.0;
      cn[f] = with_pc ? pc[o] : 0.0;
    }
    if (with_g) {
      gc = grav[c];
      gn[0] = grav[up[2] ? c + 1 : c];
      gn[1] = grav[dn[2] ? c - 1 : c];
    }
    double d = 0.0, qg = 0.0, qpc = 0.0;
    double o_plus[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const int ax = f >> 1;
      const bool low = f & 1;
      if (!(low ? dn[ax] : up[ax])) continue;
      // the flow leaves this cell: over its upper face, or not in over its lower one
      const bool self = low ? !((pn[f] - pcc) > 0) : (pcc - pn[f]) > 0;
      const double tl = tn[f] * (self ? mc : mn[f]);
      if (!low) o_plus[ax] = -tl;
      d += tl;
      if (ax == 2 && with_g) {
        const double q = tn[f] * F.g * G.dz * (self ? gc : gn[f & 1]);
        qg = low ? qg + q : qg - q;
      }
      if (with_pc) {
        const double q = tn[f] * (self ? oc : on[f]) * (low ? cc - cn[f] : cn[f] - cc);
        qpc = low ? qpc + q : qpc - q;
      }
    }
    ox[c] = o_plus[0];
    oy[c] = o_plus[1];
    oz[c] = o_plus[2];
    const double dd = d + a;
    diag[c] = dd;
    dinv[c] = 1.0 / dd;
    const double e = qg + qpc;
    extra[c] = e;
    b[c] = a * pcc + e;
  }
}

// Wells of one cell form a chain: link[2 w] is the cell's first well, link[2 w + 1] the
// next one after w (-1: none). Several wells of a cell add to it in well order (the
// serial loop's accumulation, bit for bit), by the thread of the first; wells of
// different cells are independent, so nothing else is serial.
__device__ __forceinline__ bool well_lone(const int* __restrict__ link, int w) {
  return link[2 * w] == w && link[2 * w + 1] < 0;
}

// _calculate_well_terms (:1622-1660). One thread per well computes its diagonal and
// right-hand-side increments and report slots and, where the well has its cell to
// itself (every well unless `shared`), adds them; the others leave them in
// ws[2 w], ws[2 w + 1] for the first well's thread. One workgroup: latency is all it
// costs (a serial thread over the wells took 128 us for 256 wells, 3.2 us).
__global__ __launch_bounds__(256) void k_wells_pressure(FluidParams F, int nw, const WellDesc* __restrict__ W,
                                                        const double* __restrict__ p, const double* __restrict__ mt,
                                                        double* __restrict__ diag, double* __restrict__ b,
                                                        double* __restrict__ dinv, double* __restrict__ rep,
                                                        double* __restrict__ ws, const int* __restrict__ link,
                                                        int shared) {
  for (int w = threadIdx.x; w < nw; w += blockDim.x) {
    double* R = rep + kReportHead + kWellSlots * w;
    const WellDesc& d = W[w];
    const int c = d.cell;
    double dd = 0.0, db = 0.0;
    R[kWMode] = -1.0;
    R[kWTerm] = 0.0;
    R[kWQRate] = 0.0;
    if (d.control == 0) {
      const double rate = (d.value * F.rate_scale) / kDay * (d.producer ? -1.0 : 1.0);
      bool bhp = false;
      if (d.producer && d.has_bhp_min) {
        const double denom = d.wi * mt[c] + 1e-12;
        const double preq = p[c] - rate / denom;
        const double pmin = d.bhp_min * 1e6;
        if (preq < pmin) {
          const double term = d.wi * mt[c];
          R[kWMode] = 1.0;
          R[kWTerm] = term;
          dd = term;
          db = term * pmin;
          bhp = true;
        }
      }
      if (!bhp) {
        R[kWMode] = 0.0;
        R[kWQRate] = rate;
        db = rate;
      }
    } else if (d.control == 1) {
      const double term = d.wi * mt[c];
      R[kWTerm] = term;
      dd = term;
      db = term * (d.value * 1e6);
    }
    if (!shared || well_lone(link, w)) {
      const double a = diag[c] + dd;
      diag[c] = a;
      b[c] += db;
      dinv[c] = 1.0 / a;
    } else {
      ws[2 * w] = dd;
      ws[2 * w + 1] = db;
    }
  }
  if (!shared) return;
  __syncthreads();
  for (int w = threadIdx.x; w < nw; w += blockDim.x) {
    if (link[2 * w] != w || link[2 * w + 1] < 0) continue;
    const int c = W[w].cell;
    double a = diag[c], r = b[c];
    for (int v = w; v >= 0; v = link[2 * v + 1]) {
      a += ws[2 * v];
      r += ws[2 * v + 1];
    }
    diag[c] = a;
    b[c] = r;
    dinv[c] = 1.0 / a;
  }
}

// ---------------------------------------------------------------- transport
// Sum over BHP-type wells of WI*lambda*(p_bhp - p_cell) from the pressure-equation
// row of cell c (well terms excluded).
__device__ double row_balance(const SatWellCtx& X, int c, double q_rate) {
  const GridDev& G = X.G;
  int i, j, k;
  ijk(G, c, i, j, k);
  const double pc = X.p[c];
  double f = 0.0;
  if (i < G.nx - 1) f += -X.ox[c] * (pc - X.p[c + G.sx]);
  if (i > 0) f += -X.ox[c - G.sx] * (pc - X.p[c - G.sx]);
  if (j < G.ny - 1) f += -X.oy[c] * (pc - X.p[c + G.sy]);
  if (j > 0) f += -X.oy[c - G.sy] * (pc - X.p[c - G.sy]);
  if (k < G.nz - 1) f += -X.oz[c] * (pc - X.p[c + 1]);
  if (k > 0) f += -X.oz[c - 1] * (pc - X.p[c - 1]);
  return f + X.acc[c] * (pc - X.p_prev[c]) - q_rate - X.extra[c];
}

// The per-well loop of the transport step (simulation.py:1051-1347). Each well's
// terms depend only on its cell's state and on the pressure step's report, so one
// thread per well computes them: the increments of qw, qg, qo go to the cell (or, for
// wells that share one, through the scratch row ws[3 w ..] to the first well's thread,
// which adds them in well order), and the oil in/out, gas in/out and volume sums are
// folded over the workgroup in a fixed order. One workgroup: latency is all it costs (a
// serial thread adding up 256 wells took 125 us, this 12 us: dependent loads that miss),
// which is hidden: the workgroup runs beside those of the cells (k_props_wells), so the
// mobilities of the well cells are formed here and not read.
__device__ void wells_sat(const SatWellCtx& X, double* __restrict__ qw, double* __restrict__ qg,
                          double* __restrict__ qo, double* __restrict__ rep, double* __restrict__ ws,
                          double* lds) {
  const FluidParams& F = X.F;
  const bool pvt = X.T.n > 0;
  const double dt = X.dt;
  const int* __restrict__ link = X.link;
  // oil in, oil out, gas in, gas out, sums of qw and qg (a power of two of slots)
  double tot[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int w = threadIdx.x; w < X.nw; w += blockDim.x) {
    double dqw = 0.0, dqg = 0.0, dqo = 0.0;
    double oil_in = 0.0, oil_out = 0.0, gas_in = 0.0, gas_out = 0.0, sum_qw = 0.0, sum_qg = 0.0;
    const WellDesc& d = X.W[w];
    double* R = rep + kReportHead + kWellSlots * w;
    R[kWHasQ] = 0.0;
    R[kWBal] = NAN;
    R[kWObs + 0] = R[kWObs + 1] = R[kWObs + 2] = 0.0;
    const int c = d.cell;
    const double P = X.p[c];
    const PvtAt atP = pvt ? pvt_locate(X.T, P) : PvtAt{};  // every lookup below is at P
    const double sw = X.sw[c], sg = X.sg[c];
    double kro, krw, krg, muo, muw, mug;
    relperms(F, sw, sg, kro, krw, krg);
    viscosities(F, X.T, P, muo, muw, mug, &atP);
    const double mwc = krw / muw, moc = kro / muo, mgc = krg / mug;
    const double mtc = mwc + moc + mgc;
    const double fw = mwc / (mtc + 1e-10), fg = mgc / (mtc + 1e-10), fo = moc / (mtc + 1e-10);
    const double pvc = X.pv[c];
    if (d.control == 0) {
      const double q_base = (d.value * F.rate_scale) / kDay;
      double q;
      if (!d.producer && d.surface && pvt) q = q_base * pvt_at(X.T, d.gas ? kBg : kBw, atP);
      else q = q_base;
      q *= d.producer ? -1.0 : 1.0;
      if (!d.producer) {
        double up, dn;
        if (d.gas) { up = fmax(0.0, (1.0 - F.so_r - sw) - sg); dn = sg - F.sg_cr; }
        else { up = fmax(0.0, (1.0 - F.so_r - sg) - sw); dn = sw - F.sw_cr; }
        const double dS = (dt / mx12(pvc)) * q;
        double alpha = 1.0;
        alpha = (dS > 0.0) ? fmin(alpha, up / mx12(dS)) : fmin(alpha, dn / mx12(fabs(dS)));
        q *= fmax(0.0, fmin(1.0, alpha));
        if (d.gas) {
          dqg += q;
          sum_qg += q;
          if (pvt) {
            const double bg = pvt_at(X.T, kBg, atP), rv = pvt_at(X.T, kRv, atP);
            const double qs = fmax(q, 0.0) / mx12(bg) * kDay;
            gas_in += qs * (dt / kDay);
            oil_in += rv * qs * (dt / kDay);
          }
        } else {
          dqw += q;
          sum_qw += q;
        }
      } else {
        const bool surface = d.surface && pvt;
        if (surface || pvt) {
          const double bo = pvt_at(X.T, kBo, atP), bw = pvt_at(X.T, kBw, atP), bg = pvt_at(X.T, kBg, atP);
          const double rs = pvt_at(X.T, kRs, atP), rv = pvt_at(X.T, kRv, atP);
          if (surface) {
            if (d.surface_phase == 0) q = -(q_base / mx12(fo / mx12(bo) + fg * rv / mx12(bg)));
            else if (d.surface_phase == 1) q = -(q_base * bw) / fmax(fw, 1e-8);
            else if (d.surface_phase == 2) q = -(q_base / mx12(fg / mx12(bg) + fo * rs / mx12(bo)));
            else q = -(q_base / mx12(fo / mx12(bo) + fg * rv / mx12(bg) + fw / mx12(bw)));
          }
          const double sw_up = fmax(0.0, (1.0 - F.so_r - sg) - sw), sw_dn = fmax(0.0, sw - F.sw_cr);
          const double sg_up = fmax(0.0, (1.0 - F.so_r - sw) - sg), sg_dn = fmax(0.0, sg - F.sg_cr);
          const double dSw = (dt / mx12(pvc)) * (q * fw), dSg = (dt / mx12(pvc)) * (q * fg);
          double alpha = 1.0;
          alpha = (dSw > 0.0) ? fmin(alpha, sw_up / mx12(dSw)) : fmin(alpha, sw_dn / mx12(fabs(dSw)));
          alpha = (dSg > 0.0) ? fmin(alpha, sg_up / mx12(dSg)) : fmin(alpha, sg_dn / mx12(fabs(dSg)));
          q *= fmax(0.0, fmin(1.0, alpha));
          if (d.lim_mask) {
            const double d_o = fo / mx12(bo) + fg * rv / mx12(bg);
            const double d_w = fw / mx12(bw);
            const double d_g = fg / mx12(bg) + fo * rs / mx12(bo);
            const double d_l = d_o + d_w;
            double m = INFINITY;
            bool any = false;
            if ((d.lim_mask & 1) && d_o > 0) { m = fmin(m, (d.lim[0] / kDay) / d_o); any = true; }
            if ((d.lim_mask & 2) && d_w > 0) { m = fmin(m, (d.lim[1] / kDay) / d_w); any = true; }
            if ((d.lim_mask & 4) && d_g > 0) { m = fmin(m, (d.lim[2] / kDay) / d_g); any = true; }
            if ((d.lim_mask & 8) && d_l > 0) { m = fmin(m, (d.lim[3] / kDay) / d_l); any = true; }
            if (any && fabs(q) > m) q = -m;
          }
          const double os = fabs(q) * (fo / mx12(bo) + fg * rv / mx12(bg)) * kDay;
          const double ws = fabs(q) * (fw / mx12(bw)) * kDay;
          const double gs = fabs(q) * (fg / mx12(bg) + fo * rs / mx12(bo)) * kDay;
          R[kWHasQ] = 1.0;
          R[kWQTotal] = q;
          R[kWSurf + 0] = os;
          R[kWSurf + 1] = ws;
          R[kWSurf + 2] = gs;
          R[kWSurf + 3] = os + ws;
          R[kWObs + 0] = os;
          R[kWObs + 1] = ws;
          R[kWObs + 2] = gs;
          const double qo_res = -q * fo, qg_res = -q * fg;
          oil_out += dt * (fmax(qo_res, 0.0) / mx12(bo) + rv * fmax(qg_res, 0.0) / mx12(bg));
          gas_out += dt * (fmax(qg_res, 0.0) / mx12(bg) + rs * fmax(qo_res, 0.0) / mx12(bo));
        } else {
          R[kWObs + 0] = fabs(q) * fo * kDay;
          R[kWObs + 1] = fabs(q) * fw * kDay;
          R[kWObs + 2] = fabs(q) * fg * kDay;
        }
        dqw += q * fw;
        dqg += q * fg;
        dqo += q * fo;
        sum_qw += q * fw;
        sum_qg += q * fg;
      }
    } else if (d.control == 1) {
      // WI*mob_t*(p_cell - p_bhp) through the row balance when this is the only
      // well with a pressure-equation diagonal term in the cell
      int nterm = 0;
      double q_rate = 0.0;
      for (int v = link[2 * w]; v >= 0; v = link[2 * v + 1]) {
        const double* Rv = rep + kReportHead + kWellSlots * v;
        if (Rv[kWTerm] != 0.0) ++nterm;
        q_rate += Rv[kWQRate];
      }
      double q;
      if (nterm == 1) {
        const double B = row_balance(X, c, q_rate);
        R[kWBal] = B;
        q = -B * mtc / X.mt_pres[c];
      } else {
        q = d.wi * mtc * (P - d.value * 1e6);
      }
      if (!d.producer) {
        if (d.gas) {
          dqg += -q;
          sum_qg += -q;
          if (pvt) {
            const double bg = pvt_at(X.T, kBg, atP), rv = pvt_at(X.T, kRv, atP);
            const double qs = fmax(-q, 0.0) / mx12(bg) * kDay;
            gas_in += qs * (dt / kDay);
            oil_in += rv * qs * (dt / kDay);
          }
        } else {
          dqw += -q;
          sum_qw += -q;
        }
      } else {
        dqw += -q * fw;
        dqg += -q * fg;
        dqo += -q * fo;
        sum_qw += -q * fw;
        sum_qg += -q * fg;
        const double qa = fabs(q);
        if (pvt) {
          const double bo = pvt_at(X.T, kBo, atP), bg = pvt_at(X.T, kBg, atP);
          const double rs = pvt_at(X.T, kRs, atP), rv = pvt_at(X.T, kRv, atP), bw = pvt_at(X.T, kBw, atP);
          const double qo_res = qa * fo, qg_res = qa * fg;
          oil_out += dt * (qo_res / mx12(bo) + rv * qg_res / mx12(bg));
          gas_out += dt * (qg_res / mx12(bg) + rs * qo_res / mx12(bo));
          R[kWObs + 0] = qa * (fo / mx12(bo) + fg * rv / mx12(bg)) * kDay;
          R[kWObs + 1] = qa * (fw / mx12(bw)) * kDay;
          R[kWObs + 2] = qa * (fg / mx12(bg) + fo * rs / mx12(bo)) * kDay;
        } else {
          R[kWObs + 0] = qa * fo * kDay;
          R[kWObs + 1] = qa * fw * kDay;
          R[kWObs + 2] = qa * fg * kDay;
        }
      }
    }
    if (!X.shared || well_lone(link, w)) {
      qw[c] += dqw;
      qg[c] += dqg;
      qo[c] += dqo;
    } else {
      double* r = ws + (long long)kWellScratch * w;
      r[0] = dqw;
      r[1] = dqg;
      r[2] = dqo;
    }
    tot[0] += oil_in;
    tot[1] += oil_out;
    tot[2] += gas_in;
    tot[3] += gas_out;
    tot[4] += sum_qw;
    tot[5] += sum_qg;
  }
  const double f = block_fold(tot, lds);  // also the barrier before the rows of ws are read
  if (X.shared) {
    for (int w = threadIdx.x; w < X.nw; w += blockDim.x) {
      if (link[2 * w] != w || link[2 * w + 1] < 0) continue;
      const int c = X.W[w].cell;
      double a = qw[c], g = qg[c], o = qo[c];
      for (int v = w; v >= 0; v = link[2 * v + 1]) {
        const double* r = ws + (long long)kWellScratch * v;
        a += r[0];
        g += r[1];
        o += r[2];
      }
      qw[c] = a;
      qg[c] = g;
      qo[c] = o;
    }
  }
  const int t = threadIdx.x;
  if (t < 4) rep[kCompOIn + t] = f;
  else if (t < 6) rep[kVolQW + t - 4] = dt * f;
}

// simulation.py:973-1006: mobilities at the new pressure, densities, o-g capillarity,
// and, in the first workgroup, the wells. mo: nullptr where nobody reads the oil
// mobility (the reverse sweep does). A streaming pass: at 1M cells 24 MB read, 32 MB
// (40 with mo) written, 22 us; as two launches 26 + 15 us and their gap (34.5 us as one
// with a branch per table lookup).
__global__ __launch_bounds__(kBlock) void k_props_wells(SatWellCtx X, double* __restrict__ mw,
                                                        double* __restrict__ mo, double* __restrict__ mg,
                                                        double* __restrict__ rw, double* __restrict__ rg,
                                                        double* __restrict__ pcog, double* __restrict__ qw,
                                                        double* __restrict__ qg, double* __restrict__ qo,
                                                        double* __restrict__ rep, double* __restrict__ ws) {
  __shared__ double lds[8 * (kBlock / kWave)];
  if (blockIdx.x == 0) {
    wells_sat(X, qw, qg, qo, rep, ws, lds);
    return;
  }
  const GridDev& G = X.G;
  const FluidParams& F = X.F;
  const PvtDev& T = X.T;
  const double* __restrict__ p = X.p;
  const double* __restrict__ sw = X.sw;
  const double* __restrict__ sg = X.sg;
  const long long n = (long long)G.nx * G.ny * G.nz;
  for (long long c = (blockIdx.x - 1) * (long long)kBlock + threadIdx.x; c < n;
       c += (gridDim.x - 1) * (long long)kBlock) {
    const double pp = p[c];
    double kro, krw, krg, muo, muw, mug;
    relperms(F, sw[c], sg[c], kro, krw, krg);
    PvtAt at{};
    if (T.n > 0) at = pvt_locate(T, pp);
    viscosities(F, T, pp, muo, muw, mug, &at);
    mw[c] = krw / muw;
    if (mo) mo[c] = kro / muo;
    mg[c] = krg / mug;
    if (G.gravity) {
      double r1, r2, r3;
      densities(F, T, pp, r1, r2, r3, &at);
      rw[c] = r1;
      rg[c] = r3;
    }
    if (F.pcog_scale > 0.0) pcog[c] = pc_og(F, sg[c]);
  }
}

// NaN/inf-propagating max (torch.max semantics)
__device__ __forceinline__ double nmax(double a, double b) {
  if (a != a || b != b) return NAN;
  return a > b ? a : b;
}

// the well cells' sources back to zero, by one workgroup
__device__ __forceinline__ void reset_wells(int nw, const WellDesc* __restrict__ W, double* __restrict__ qw,
                                            double* __restrict__ qg, double* __restrict__ qo) {
  for (int w = threadIdx.x; w < nw; w += blockDim.x) {
    const int c = W[w].cell;
    qw[c] = 0.0;
    qg[c] = 0.0;
    qo[c] = 0.0;
  }
}

// NaN-propagating max of the block's values (order-independent), on every thread
__device__ double block_nmax(double m, double* lds) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  for (int off = kWave / 2; off > 0; off >>= 1) m = nmax(m, __shfl_xor(m, off, kWave));
  if (lane == 0) lds[wid] = m;
  __syncthreads();
  double r = lds[0];
  for (int q = 1; q < (int)(blockDim.x / kWave); ++q) r = nmax(r, lds[q]);
  return r;
}

// The transport kernels below give each workgroup one run of `per` x kBlock cells, and
// each XCD one run of workgroups, so that a cell's neighbours mostly sit in the L2 that
// read them.
constexpr int kTransBlocks = 2048;  // workgroups (and partials) at most
inline int trans_per(long long n) {
  return (int)((n + (long long)kTransBlocks * kBlock - 1) / ((long long)kTransBlocks * kBlock));
}
inline int trans_blocks(long long n) {
  const long long run = (long long)trans_per(n) * kBlock;
  return (int)((n + run - 1) / run);
}

// simulation.py:985-1042 and :1352-1373: upwind phase fluxes (upwind by the pressure
// difference only), gravity potential with arithmetic-mean densities, o-g capillarity
// on gas; their divergence; the saturation increments and the per-cell substep demand
// (its maximum per workgroup in part, and per cell in rat when the grid holds several
// reservoirs).
// One pass, so the divergences stay in registers; and every load is made whether its
// face exists or not (a missing neighbour reads the cell itself), both sides of an
// upwind choice included, so that a wave waits for them once and not face after face.
// At 1M cells 27 us; 29.9 us (fluxes) + 16.0 us (increments) as two passes with a
// wait per face.
__global__ __launch_bounds__(kBlock) void k_flux_rat(
    GridDev G, FluidParams F, double dt, int per, const double* __restrict__ p, const double* __restrict__ tx,
    const double* __restrict__ ty, const double* __restrict__ tz, const double* __restrict__ mw,
    const double* __restrict__ mg, const double* __restrict__ rw, const double* __restrict__ rg,
    const double* __restrict__ pcog, const double* __restrict__ sw, const double* __restrict__ sg,
    const double* __restrict__ pv, const double* __restrict__ qw, const double* __restrict__ qg,
    double* __restrict__ dsw, double* __restrict__ dsg, double* __restrict__ part, double* __restrict__ rat) {
  __shared__ double lds[kBlock / kWave];
  const long long n = (long long)G.nx * G.ny * G.nz;
  const bool with_pcog = F.pcog_scale > 0.0, grav = G.gravity != 0;
  const double eps = 1e-12;
  const long long b = xcd_block();
  double m = 0.0;
  for (int t = 0; t < per; ++t) {
    const long long c = (b * per + t) * kBlock + threadIdx.x;
    if (c >= n) break;
    int i, j, k;
    ijk(G, c, i, j, k);
    const bool up[3] = {i < G.nx - 1, j < G.ny - 1, k < G.nz - 1}, dn[3] = {i > 0, j > 0, k > 0};
    const long long st[3] = {G.sx, G.sy, 1};
    const double* const T[3] = {tx, ty, tz};
    double pn[6], tn[6], wn[6], gn[6], cn[6];
    const double pc = p[c], wc = mw[c], gc = mg[c], cc = with_pcog ? pcog[c] : 0.0;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const int ax = f >> 1;
      const long long o = f & 1 ? (dn[ax] ? c - st[ax] : c) : (up[ax] ? c + st[ax] : c);
      pn[f] = p[o];
      wn[f] = mw[o];
      gn[f] = mg[o];
      cn[f] = with_pcog ? pcog[o] : 0.0;
      tn[f] = T[ax][f & 1 ? o : c];
    }
    double rwc = 0.0, rgc = 0.0, rwn[2] = {0.0, 0.0}, rgn[2] = {0.0, 0.0};
    if (grav) {
      const long long hi = up[2] ? c + 1 : c, lo = dn[2] ? c - 1 : c;
      rwc = rw[c];
      rgc = rg[c];
      rwn[0] = rw[hi];
      rgn[0] = rg[hi];
      rwn[1] = rw[lo];
      rgn[1] = rg[lo];
    }
    const double s_w = sw[c], s_g = sg[c], v = pv[c], q_w = qw[c], q_g = qg[c];
    double dw = 0.0, dg = 0.0;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const int ax = f >> 1;
      const bool low = f & 1;  // face to the lower neighbour: this cell is the upper one
      const double dp = low ? pn[f] - pc : pc - pn[f];
      const bool from_c = (dp > 0) != low;
      double pot_w = dp, pot_g = dp;
      if (ax == 2 && grav) {
        const int q = f & 1;
        pot_w = dp + F.g * (0.5 * (rwc + rwn[q])) * G.dz;
        pot_g = dp + F.g * (0.5 * (rgc + rgn[q])) * G.dz;
      }
      const double t = tn[f];
      const double fw = t * (from_c ? wc : wn[f]) * pot_w;
      const double mgu = from_c ? gc : gn[f];
      const double fg = with_pcog ? t * mgu * (pot_g - (low ? cc - cn[f] : cn[f] - cc)) : t * mgu * pot_g;
      if (low ? dn[ax] : up[ax]) {
        dw = low ? dw - fw : dw + fw;
        dg = low ? dg - fg : dg + fg;
      }
    }
    const double kk = dt / v;
    const double a = kk * (q_w - dw);
    const double g = kk * (q_g - dg);
    dsw[c] = a;
    dsg[c] = g;
    const double sw_up = fmax(1.0 - F.so_r - s_g - s_w, 0.0), sw_dn = fmax(s_w - F.sw_cr, 0.0);
    const double sg_up = fmax(1.0 - F.so_r - s_w - s_g, 0.0), sg_dn = fmax(s_g - F.sg_cr, 0.0);
    const double ra = a > 0 ? a / fmax(sw_up, eps) : (-a) / fmax(sw_dn, eps);
    const double rb = g > 0 ? g / fmax(sg_up, eps) : (-g) / fmax(sg_dn, eps);
    const double rl = nmax(fabs(a) / F.max_ds, fabs(g) / F.max_ds);
    const double rc = nmax(nmax(ra, rb), rl);
    if (rat) rat[c] = rc;
    m = nmax(m, rc);
  }
  const double r = block_nmax(m, lds);
  if (threadIdx.x == 0) part[b] = r;
}

// Substep count from the largest demand (simulation.py:1352-1377)
__device__ __forceinline__ double substep_count(const FluidParams& F, double& r) {
  if (!isfinite(r)) r = 0.0;  // nan_to_num(nan=0, posinf=0, neginf=0)
  double N = ceil(r);
  if (N < 1) N = 1;
  if (N > F.max_substeps) N = F.max_substeps;
  return N;
}

// The count alone, for the reverse sweep (k_substeps forms its own), and the well cells'
// sources back to zero. One workgroup.
__global__ void k_nsub(int nb, FluidParams F, const double* __restrict__ part, double* __restrict__ rep, int nw,
                       const WellDesc* __restrict__ W, double* __restrict__ qw, double* __restrict__ qg,
                       double* __restrict__ qo) {
  __shared__ double lds[kBlock / kWave];
  double m = 0.0;
  for (int q = threadIdx.x; q < nb; q += blockDim.x) m = nmax(m, part[q]);
  double r = block_nmax(m, lds);
  reset_wells(nw, W, qw, qg, qo);
  if (threadIdx.x != 0) return;
  rep[kNSub] = substep_count(F, r);
  rep[kRatMax] = r;
}

// Substep count of each stacked reservoir (over its own cells, which are contiguous:
// env e holds cells [e*cells, (e+1)*cells)). One block per reservoir; nsub[e] also
// lands in the report tail.
__global__ void k_nsub_env(long long cells, FluidParams F, const double* __restrict__ rat, double* __restrict__ nsub,
                           double* __restrict__ rep_tail) {
  __shared__ double lds[kBlock / kWave];
  const long long c0 = (long long)blockIdx.x * cells;
  double m = 0.0;
  for (long long c = threadIdx.x; c < cells; c += blockDim.x) m = nmax(m, rat[c0 + c]);
  double r = block_nmax(m, lds);
  if (threadIdx.x != 0) return;
  const double N = substep_count(F, r);
  nsub[blockIdx.x] = N;
  rep_tail[blockIdx.x] = N;
}

// one substep of simulation.py:1385-1394 (shared by the field kernel and the ledger kernel)
__device__ __forceinline__ void substep(const FluidParams& F, double dsw_sub, double dsg_sub, double& s_w, double& s_g,
                                        double& cw, double& cg) {
  const double wu = s_w + dsw_sub;
  const double gu = s_g + dsg_sub;
  const double w = fmin(fmax(wu, F.sw_cr), 1.0 - F.so_r - gu);
  const double g = fmin(fmax(gu, F.sg_cr), 1.0 - F.so_r - w);
  cw = w - wu;
  cg = g - gu;
  s_w = w;
  s_g = g;
}

// Substeps, write-back and the ledgers (simulation.py:1385-1525): mass ledger at the
// new pressure and the volume ledger sum PV dS vs dt sum q + clamp corrections. Every
// workgroup first folds the demand's partials into the substep count by itself: about
// 1 us, where a launch for it took 4.5 us and its gap. At 1M cells (48 MB read, 24 MB
// written) 33 us; 49 us with 512 workgroups, two per CU, and ten block sums at the
// end.
__global__ __launch_bounds__(kBlock) void k_substeps(
    GridDev G, FluidParams F, PvtDev T, int per, double* __restrict__ rep, int n_rat,
    const double* __restrict__ part_rat, const double* __restrict__ p, const double* __restrict__ sw,
    const double* __restrict__ sg, const double* __restrict__ pv, const double* __restrict__ dsw,
    const double* __restrict__ dsg, double* __restrict__ sw_out, double* __restrict__ sg_out,
    double* __restrict__ so_out, double* __restrict__ part, const double* __restrict__ nsub, long long env_cells) {
  __shared__ double lds[kFoldQ * (kBlock / kWave)];
  const long long n = (long long)G.nx * G.ny * G.nz, blk = xcd_block();
  double m = 0.0;
  for (int q = threadIdx.x; q < n_rat; q += kBlock) m = nmax(m, part_rat[q]);
  double r = block_nmax(m, lds);
  const double Nd = substep_count(F, r);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    rep[kRatMax] = r;
    rep[kNSub] = Nd;
  }
  const int N_all = (int)Nd;
  const double r_all = 1.0 / N_all;
  double acc[kFoldQ];
#pragma unroll
  for (int q = 0; q < kFoldQ; ++q) acc[q] = 0.0;
  for (int t = 0; t < per; ++t) {
    const long long c = (blk * per + t) * kBlock + threadIdx.x;
    if (c >= n) break;
    const int N = nsub ? (int)nsub[c / env_cells] : N_all;  // this cell's reservoir
    const double w0 = sw[c], g0 = sg[c];
    const double rN = nsub ? 1.0 / N : r_all;
    const double a = div_by(dsw[c], N, rN), b = div_by(dsg[c], N, rN);
    double w = w0, g = g0, cw = 0.0, cg = 0.0;
    const double v = pv[c];
    for (int s = 0; s < N; ++s) {
      double c1, c2;
      substep(F, a, b, w, g, c1, c2);
      cw += v * c1;
      cg += v * c2;
    }
    sw_out[c] = w;
    sg_out[c] = g;
    if (so_out) so_out[c] = 1.0 - w - g;
    double rw, ro, rg;
    densities(F, T, p[c], rw, ro, rg);
    const double dw = w - w0, dg = g - g0;
    const double mw = dw * v * rw, mg = dg * v * rg, mo = (-(dw + dg)) * v * ro;
    acc[0] += fmax(mw, 0.0);
    acc[1] += -fmin(mw, 0.0);
    acc[2] += fmax(mo, 0.0);
    acc[3] += -fmin(mo, 0.0);
    acc[4] += fmax(mg, 0.0);
    acc[5] += -fmin(mg, 0.0);
    acc[6] += v * dw;
    acc[7] += v * dg;
    acc[8] += cw;
    acc[9] += cg;
  }
  __syncthreads();  // lds still holds the demand
  const double f = block_fold(acc, lds);
  if (threadIdx.x < kLedgerQ) part[threadIdx.x * (long long)gridDim.x + blk] = f;
}

// Component ledger of the substeps (simulation.py:1396-1503), well cells only. One
// thread per (well, substep) pair: it replays the cell's clamped substeps up to its own
// and adds that substep's surface in/out terms; a fixed-order fold keeps the result
// independent of timing.
__device__ void substep_ledger(const SatWellCtx& X, const double* __restrict__ dsw, const double* __restrict__ dsg,
                               double* __restrict__ rep, const double* __restrict__ nsub, long long env_cells,
                               double* lds) {
  const FluidParams& F = X.F;
  const int N_all = (int)rep[kNSub];
  // stacked reservoirs: each well uses its own reservoir's count, at most max_substeps
  const int Nb = nsub ? (int)F.max_substeps : N_all;
  double oil_in = 0.0, oil_out = 0.0, gas_in = 0.0, gas_out = 0.0;
  for (int t = threadIdx.x; t < X.nw * Nb; t += blockDim.x) {
    const int w = t / Nb, sub = t % Nb;
    const WellDesc& d = X.W[w];
    const int N = nsub ? (int)nsub[d.cell / env_cells] : N_all;
    if (sub >= N) continue;
    const double dt_sub = X.dt / N;
    if (d.control != 0 && d.control != 1) continue;
    const double* R = rep + kReportHead + kWellSlots * w;
    const int c = d.cell;
    const double P = X.p[c];
    const PvtAt atP = pvt_locate(X.T, P);  // every lookup below is at P
    const double muw = pvt_at(X.T, kMuW, atP), muo = pvt_at(X.T, kMuO, atP), mug = pvt_at(X.T, kMuG, atP);
    const double bo = pvt_at(X.T, kBo, atP), bw = pvt_at(X.T, kBw, atP), bg = pvt_at(X.T, kBg, atP);
    const double rs = pvt_at(X.T, kRs, atP), rv = pvt_at(X.T, kRv, atP);
    const double a = dsw[c] / N, b = dsg[c] / N;
    double s_w = X.sw[c], s_g = X.sg[c];
    for (int q = 0; q <= sub; ++q) {
      double c1, c2;
      substep(F, a, b, s_w, s_g, c1, c2);
    }
    const double q_base = (d.value * F.rate_scale) / kDay;
    double kro, krw, krg;
    relperms(F, s_w, s_g, kro, krw, krg);
    const double mw = krw / (muw + 1e-12), mo = kro / (muo + 1e-12), mg = krg / (mug + 1e-12);
    const double mt = mw + mo + mg;
    const double fw = mw / (mt + 1e-12), fg = mg / (mt + 1e-12), fo = mo / (mt + 1e-12);
    if (d.control == 0) {
      if (!d.producer) {
        if (d.gas) {
          const double q = d.surface ? q_base * bg : q_base;
          const double qs = fmax(q, 0.0) / mx12(bg) * kDay;
          gas_in += qs * (dt_sub / kDay);
          oil_in += rv * qs * (dt_sub / kDay);
        }
      } else {
        double q;
        if (d.surface) {
          if (d.surface_phase == 0) q = -(q_base / mx12(fo / mx12(bo) + fg * rv / mx12(bg)));
          else if (d.surface_phase == 1) q = -(q_base * bw) / mx12(fw);
          else if (d.surface_phase == 2) q = -(q_base / mx12(fg / mx12(bg) + fo * rs / mx12(bo)));
          else q = -(q_base / mx12(fo / mx12(bo) + fg * rv / mx12(bg) + fw / mx12(bw)));
        } else {
          q = -q_base;
        }
        const double qo_res = fmax(-q * fo, 0.0), qg_res = fmax(-q * fg, 0.0);
        oil_out += dt_sub * (qo_res / mx12(bo) + rv * qg_res / mx12(bg));
        gas_out += dt_sub * (qg_res / mx12(bg) + rs * qo_res / mx12(bo));
      }
    } else {
      const double bal = R[kWBal];
      const double q = (bal == bal) ? -bal * mt / X.mt_pres[c] : d.wi * mt * (P - d.value * 1e6);
      if (!d.producer) {
        if (d.gas) {
          const double qs = fmax(-q, 0.0) / mx12(bg) * kDay;
          gas_in += qs * (dt_sub / kDay);
          oil_in += rv * qs * (dt_sub / kDay);
        }
      } else {
        const double qa = fabs(q);
        const double qo_res = qa * fo, qg_res = qa * fg;
        oil_out += dt_sub * (qo_res / mx12(bo) + rv * qg_res / mx12(bg));
        gas_out += dt_sub * (qg_res / mx12(bg) + rs * qo_res / mx12(bo));
      }
    }
  }
  double tot[4] = {oil_in, oil_out, gas_in, gas_out};
  const double f = block_fold(tot, lds);
  if (threadIdx.x < 4) rep[kCompOIn + threadIdx.x] += f;
}

// The end of a step: workgroups 0..9 fold a ledger each, the last one integrates the
// component ledger over the wells' substeps, zeroes the wells' sources and hands the
// report out. Report and ledgers are written to `host` (mapped host memory) as well:
// the caller waits for the stream and reads them there, with no copy to queue (at 1M
// cells and 9 wells 9 us in all; the three launches it replaces took 22 us, the copy
// on top).
__global__ __launch_bounds__(kBlock) void k_step_end(SatWellCtx X, int nb, const double* __restrict__ part,
                                                     const double* __restrict__ dsw, const double* __restrict__ dsg,
                                                     double* __restrict__ qw, double* __restrict__ qg,
                                                     double* __restrict__ qo, double* __restrict__ rep, int len,
                                                     double* __restrict__ host, const double* __restrict__ nsub,
                                                     long long env_cells) {
  __shared__ double lds[4 * (kBlock / kWave)];
  constexpr int slot[kLedgerQ] = {kMassWIn, kMassWOut, kMassOIn, kMassOOut, kMassGIn, kMassGOut,
                                  kVolDW, kVolDG, kVolCW, kVolCG};
  const int q = blockIdx.x;
  if (q < kLedgerQ) {
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += kBlock) s += part[(long long)q * nb + b];
    s = block_sum(s, lds);
    if (threadIdx.x == 0) {
      rep[slot[q]] = s;
      host[slot[q]] = s;
    }
    return;
  }
  if (X.T.n > 0 && X.nw > 0) substep_ledger(X, dsw, dsg, rep, nsub, env_cells, lds);
  reset_wells(X.nw, X.W, qw, qg, qo);
  __syncthreads();  // the component ledgers are in rep
  for (int i = threadIdx.x; i < len; i += kBlock) {
    bool mine = true;
#pragma unroll
    for (int l = 0; l < kLedgerQ; ++l) mine = mine && i != slot[l];
    if (mine) host[i] = rep[i];
  }
}

__global__ void k_eval_props(FluidParams F, PvtDev T, long long n, const double* __restrict__ p,
                             const double* __restrict__ sw, const double* __restrict__ sg, double* __restrict__ out) {
  CELL_LOOP(c, n) {
    double kro, krw, krg, mo, mw, mg, rw, ro, rg;
    relperms(F, sw[c], sg[c], kro, krw, krg);
    viscosities(F, T, p[c], mo, mw, mg);
    densities(F, T, p[c], rw, ro, rg);
    const double v[12] = {kro, krw, krg, pc_ow(F, sw[c]), pc_og(F, sg[c]), total_compressibility(F, T, p[c], sw[c], sg[c]),
                          rw, ro, rg, mo, mw, mg};
    for (int q = 0; q < 12; ++q) out[q * n + c] = v[q];
  }
}

__global__ void k_eval_pvt(PvtDev T, int key, long long n, const double* __restrict__ p, double* __restrict__ out) {
  CELL_LOOP(c, n) out[c] = pvt_eval(T, key, p[c]);
}

}  // namespace

// ---------------------------------------------------------------- Model
Model::Model(const Grid& g, const FluidParams& f, int pvt_n, const double* pvt_host, const std::vector<WellDesc>& w)
    : grid(g), F(f) {
  IMPES_REQUIRE(g.nx >= 1 && g.ny >= 1 && g.nz >= 1, "model: bad grid");
  N_ = (long long)g.nx * g.ny * g.nz;
  IMPES_REQUIRE(N_ < (1LL << 30), "model: grid too large for int32 indexing");
  env_cells_ = N_;
  gravity_ = g.dz > 0 && g.nz > 1;  // simulation.py:999,1594
  if (pvt_n > 0) {
    IMPES_REQUIRE(pvt_n >= 2 && pvt_host, "model: PVT table needs >= 2 rows");
    std::vector<double> P(pvt_host, pvt_host + pvt_n), cols(pvt_host + pvt_n, pvt_host + 9 * pvt_n);
    for (int i = 0; i + 1 < pvt_n; ++i) IMPES_REQUIRE(P[i + 1] > P[i], "model: PVT pressures must increase");
    std::vector<double2> tab(8 * (size_t)(pvt_n + 1));
    for (int k = 0; k < 8; ++k) {
      const double* col = cols.data() + k * pvt_n;
      for (int i = 0; i + 1 < pvt_n; ++i) tab[8 * i + k] = double2{(col[i + 1] - col[i]) / (P[i + 1] - P[i]), col[i]};
      tab[8 * (pvt_n - 1) + k] = double2{0.0, col[pvt_n - 1]};
      tab[8 * pvt_n + k] = double2{0.0, col[0]};
    }
    pvt_P_.alloc(pvt_n);
    pvt_tab_.alloc(tab.size());
    // not hipMemcpy, which ends captures of other threads
    IMPES_HIP_CHECK(hipMemcpyAsync(pvt_P_.p, P.data(), sizeof(double) * pvt_n, hipMemcpyHostToDevice, nullptr));
    IMPES_HIP_CHECK(
        hipMemcpyAsync(pvt_tab_.p, tab.data(), sizeof(double2) * tab.size(), hipMemcpyHostToDevice, nullptr));
    IMPES_HIP_CHECK(hipStreamSynchronize(nullptr));
    pvt.n = pvt_n;
    pvt.P = pvt_P_.p;
    pvt.tab = pvt_tab_.p;
  }
  const long long n = N_;
  for (auto* b : {&tx, &ty, &tz, &pv, &diag, &ox, &oy, &oz, &this->b, &dinv, &acc, &extra, &mob_t}) b->alloc(n);
  for (auto* b : {&mob_w_, &mob_o_, &mob_g_, &dsw_, &dsg_, &qw_, &qg_, &qo_}) b->alloc(n);
  if (gravity_) for (auto* b : {&rho_w_, &rho_o_, &rho_g_, &grav_}) b->alloc(n);
  if (F.pc_scale > 0.0) pc_.alloc(n);
  if (F.pcog_scale > 0.0) pcog_.alloc(n);
  for (auto* b : {&qw_, &qg_, &qo_}) launch_fill_f64(b->p, 0.0, n, nullptr);
  part_.alloc((size_t)kTransBlocks * (kLedgerQ + 1));  // the demand's partials and the ledgers'
  set_wells(w, nullptr);
  IMPES_HIP_CHECK(hipStreamSynchronize(nullptr));
}

void Model::HostReport::reserve(size_t n) {
  if (cap >= n) return;
  if (p) IMPES_HIP_CHECK(hipHostFree(p));  // every step that writes it has been waited for
  p = dev = nullptr;
  cap = 0;
  IMPES_HIP_CHECK(hipHostMalloc((void**)&p, sizeof(double) * n, hipHostMallocMapped));
  IMPES_HIP_CHECK(hipHostGetDevicePointer((void**)&dev, p, 0));
  cap = n;
}

Model::HostReport::~HostReport() {
  if (p) (void)hipHostFree(p);
}

Model::Staging::~Staging() {
  if (ev) {
    (void)hipEventSynchronize(ev);
    (void)hipEventDestroy(ev);
  }
  if (p) (void)hipHostFree(p);
}

namespace {
// Chains of the wells that share a cell (k_wells_pressure); returns whether one does.
int link_wells(const std::vector<WellDesc>& w, int* link) {
  const int n = (int)w.size();
  std::vector<int> order(n);
  for (int i = 0; i < n; ++i) {
    order[i] = link[2 * i] = i;
    link[2 * i + 1] = -1;
  }
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return w[a].cell < w[b].cell; });
  int shared = 0;
  for (int i = 1; i < n; ++i) {
    const int a = order[i - 1], b = order[i];
    if (w[a].cell != w[b].cell) continue;
    link[2 * a + 1] = b;
    link[2 * b] = link[2 * a];
    shared = 1;
  }
  return shared;
}
}  // namespace

void Model::set_wells(const std::vector<WellDesc>& w, hipStream_t s) {
  for (const auto& d : w) IMPES_REQUIRE(d.cell >= 0 && d.cell < N_, "model: well outside the grid");
  nw_ = (int)w.size();
  if (nw_ > 0) {
    wells_.reserve(nw_);
    well_link_.reserve(2 * (size_t)nw_);
    well_sc_.reserve((size_t)kWellScratch * nw_);
    if (!stage_.ev) IMPES_HIP_CHECK(hipEventCreateWithFlags(&stage_.ev, hipEventDisableTiming));
    IMPES_HIP_CHECK(hipEventSynchronize(stage_.ev));  // the last upload has left the staging
    if (stage_.cap < (size_t)nw_) {
      if (stage_.p) IMPES_HIP_CHECK(hipHostFree(stage_.p));
      stage_.p = nullptr;
      stage_.cap = 0;
      IMPES_HIP_CHECK(hipHostMalloc((void**)&stage_.p, (sizeof(WellDesc) + 2 * sizeof(int)) * nw_,
                                    hipHostMallocDefault));
      stage_.cap = nw_;
    }
    std::memcpy(stage_.p, w.data(), sizeof(WellDesc) * nw_);
    int* link = reinterpret_cast<int*>(stage_.p + nw_);
    wells_shared_ = link_wells(w, link);
    IMPES_HIP_CHECK(hipMemcpyAsync(wells_.p, stage_.p, sizeof(WellDesc) * nw_, hipMemcpyHostToDevice, s));
    IMPES_HIP_CHECK(hipMemcpyAsync(well_link_.p, link, 2 * sizeof(int) * nw_, hipMemcpyHostToDevice, s));
    IMPES_HIP_CHECK(hipEventRecord(stage_.ev, s));
  }
  report_.reserve(report_len());
  report_host_.reserve(report_len());
  launch_fill_f64(report_.p, 0.0, report_len(), s);
}

void Model::set_envs(int env_nx, hipStream_t s) {
  IMPES_REQUIRE(env_nx >= 0, "model: env_nx must be >= 0");
  if (env_nx == 0 || env_nx == grid.nx) {
    env_nx_ = 0;
    n_env_ = 1;
  } else {
    IMPES_REQUIRE(grid.nx % env_nx == 0, "model: nx must be a multiple of env_nx");
    env_nx_ = env_nx;
    n_env_ = grid.nx / env_nx;
    rat_.alloc(N_);
    nsub_.alloc(n_env_);
  }
  env_cells_ = (long long)(env_nx_ > 0 ? env_nx_ : grid.nx) * grid.ny * grid.nz;
  amg_.reset();  // the operator's pattern loses the faces between reservoirs
  report_.reserve(report_len());
  report_host_.reserve(report_len());
  launch_fill_f64(report_.p, 0.0, report_len(), s);
}

void Model::set_rock(const double* kx, const double* ky, const double* kz, const double* pv_in, hipStream_t s) {
  GridDev G = grid_dev(grid, gravity_, env_nx_);
  k_trans<<<grid_for(N_, kBlock, 1 << 16), kBlock, 0, s>>>(G, kx, ky, kz, pv_in, tx.p, ty.p, tz.p, pv.p);
  IMPES_LAUNCH_CHECK();
}

void Model::assemble(double dt, const double* p, const double* sw, const double* sg, hipStream_t s) {
  IMPES_REQUIRE(dt > 0.0, "assemble: dt must be positive");
  dt_ = dt;
  GridDev G = grid_dev(grid, gravity_, env_nx_);
  const int gr = grid_for(N_, kBlock, 1 << 16);
  // the mobility of the oil is read for the capillary fluxes alone
  const PressureProps Q{mob_t.p, acc.p, grav_.p, pc_.p, F.pc_scale > 0.0 ? mob_o_.p : nullptr,
                        nullptr, nullptr, nullptr, nullptr, nullptr};
  k_props_pressure<<<gr, kBlock, 0, s>>>(G, F, pvt, dt, p, sw, sg, pv.p, Q);
  IMPES_LAUNCH_CHECK();
  k_assemble<<<gr, kBlock, 0, s>>>(G, F, p, tx.p, ty.p, tz.p, mob_t.p, grav_.p, mob_o_.p, pc_.p, acc.p, diag.p, ox.p,
                                   oy.p, oz.p, b.p, extra.p, dinv.p);
  IMPES_LAUNCH_CHECK();
  if (nw_ > 0) {
    k_wells_pressure<<<1, 256, 0, s>>>(F, nw_, wells_.p, p, mob_t.p, diag.p, b.p, dinv.p, report_.p, well_sc_.p,
                                       well_link_.p, wells_shared_);
    IMPES_LAUNCH_CHECK();
  }
}

void Model::solve(int precision, double rtol, int restart, int maxit, double* p_new, SolveStats& st, hipStream_t s) {
  if (!amg_) {
    auto h = std::make_unique<Hierarchy>(amg_prm_);
    h->setup_stencil(grid.nx, grid.ny, grid.nz, diag.p, ox.p, oy.p, oz.p, s);
    amg_ = std::move(h);  // a setup that fails is tried again by the next solve
  } else {
    amg_->update_stencil(diag.p, ox.p, oy.p, oz.p, s);
  }
  Operator A;
  A.stencil = true;
  A.st = Stencil7<double>{grid.nx, grid.ny, grid.nz, diag.p, ox.p, oy.p, oz.p};
  A.dinv = dinv.p;
  A.n = N_;
  fgmres_.solve(A, amg_.get(), precision, b.p, p_new, true, rtol, restart, maxit, st, s);
}

bool Model::solve_cg(double tol, int maxit, double* x, int& its, hipStream_t s) {
  const long long n = N_;
  cg_r_.reserve(n); cg_z_.reserve(n); cg_p_.reserve(n); cg_ap_.reserve(n);
  cg_s_.reserve(kRedBlocks + 8);
  double* work = cg_s_.p;
  double* sc = cg_s_.p + kRedBlocks;
  Stencil7<double> S{grid.nx, grid.ny, grid.nz, diag.p, ox.p, oy.p, oz.p};
  double hbuf = 0.0;
  auto read = [&](const double* dev) {
    IMPES_HIP_CHECK(hipMemcpyAsync(&hbuf, dev, sizeof(double), hipMemcpyDeviceToHost, s));
    IMPES_HIP_CHECK(hipStreamSynchronize(s));
    return hbuf;
  };
  launch_fill_f64(x, 0.0, n, s);
  launch_copy_f64(cg_r_.p, b.p, n, s);
  launch_scale_f64(cg_z_.p, dinv.p, cg_r_.p, n, s);
  launch_copy_f64(cg_p_.p, cg_z_.p, n, s);
  launch_dot_f64(cg_r_.p, cg_z_.p, n, sc, work, s);
  double rs_old = read(sc);
  its = 0;
  if (rs_old < 1e-10) return true;
  for (int it = 0; it < maxit; ++it) {
    launch_st7_spmv_f64(S, cg_p_.p, cg_ap_.p, s);
    launch_dot_f64(cg_p_.p, cg_ap_.p, n, sc + 1, work, s);
    const double alpha = rs_old / read(sc + 1);
    launch_axpy_f64(x, alpha, cg_p_.p, n, s);
    launch_axpy_f64(cg_r_.p, -alpha, cg_ap_.p, n, s);
    launch_scale_f64(cg_z_.p, dinv.p, cg_r_.p, n, s);
    launch_dot_f64(cg_r_.p, cg_z_.p, n, sc + 2, work, s);
    const double rs_new = read(sc + 2);
    its = it + 1;
    if (std::sqrt(rs_new) < tol) return true;
    launch_xpby_f64(cg_p_.p, cg_z_.p, rs_new / rs_old, n, s);
    rs_old = rs_new;
  }
  return false;
}

SatWellCtx Model::sat_ctx(double dt, const double* p_prev, const double* p_new, const double* sw,
                          const double* sg) const {
  return SatWellCtx{grid_dev(grid, gravity_, env_nx_), F, pvt, dt, nw_, wells_.p, well_link_.p, wells_shared_, p_prev,
                    p_new, sw, sg, pv.p, mob_t.p, ox.p, oy.p, oz.p, acc.p, extra.p};
}

// the transport up to the saturation increments and the demand's partials; returns
// how many there are
int Model::transport_increments(const SatWellCtx& X, double* mo, double* rat, hipStream_t s) {
  k_props_wells<<<1 + grid_for(N_, kBlock, 1 << 16), kBlock, 0, s>>>(X, mob_w_.p, mo, mob_g_.p, rho_w_.p, rho_g_.p,
                                                                     pcog_.p, qw_.p, qg_.p, qo_.p, report_.p,
                                                                     well_sc_.p);
  IMPES_LAUNCH_CHECK();
  const int nb = trans_blocks(N_);
  k_flux_rat<<<nb, kBlock, 0, s>>>(X.G, F, X.dt, trans_per(N_), X.p, tx.p, ty.p, tz.p, mob_w_.p, mob_g_.p, rho_w_.p,
                                   rho_g_.p, pcog_.p, X.sw, X.sg, pv.p, qw_.p, qg_.p, dsw_.p, dsg_.p, part_.p, rat);
  IMPES_LAUNCH_CHECK();
  return nb;
}

void Model::saturation(double dt, const double* p_prev, const double* p_new, const double* sw, const double* sg,
                       double* sw_out, double* sg_out, double* so_out, double* host_report, hipStream_t s) {
  const SatWellCtx X = sat_ctx(dt, p_prev, p_new, sw, sg);
  const bool envs = n_env_ > 1;
  const int nb = transport_increments(X, nullptr, envs ? rat_.p : nullptr, s);
  if (envs) {
    k_nsub_env<<<n_env_, kBlock, 0, s>>>(env_cells_, F, rat_.p, nsub_.p, report_.p + report_len() - n_env_);
    IMPES_LAUNCH_CHECK();
  }
  double* part = part_.p + kTransBlocks;
  k_substeps<<<nb, kBlock, 0, s>>>(X.G, F, pvt, trans_per(N_), report_.p, nb, part_.p, p_new, sw, sg, pv.p, dsw_.p,
                                   dsg_.p, sw_out, sg_out, so_out, part, envs ? nsub_.p : nullptr, env_cells_);
  IMPES_LAUNCH_CHECK();
  k_step_end<<<kLedgerQ + 1, kBlock, 0, s>>>(X, nb, part, dsw_.p, dsg_.p, qw_.p, qg_.p, qo_.p, report_.p,
                                             report_len(), report_host_.dev, envs ? nsub_.p : nullptr, env_cells_);
  IMPES_LAUNCH_CHECK();
  IMPES_HIP_CHECK(hipStreamSynchronize(s));
  std::memcpy(host_report, report_host_.p, sizeof(double) * report_len());
}

void Model::transport_forward(double dt, const double* p_prev, const double* p_new, const double* sw,
                              const double* sg, hipStream_t s) {
  const int nb = transport_increments(sat_ctx(dt, p_prev, p_new, sw, sg), mob_o_.p, nullptr, s);
  k_nsub<<<1, kBlock, 0, s>>>(nb, F, part_.p, report_.p, nw_, wells_.p, qw_.p, qg_.p, qo_.p);
  IMPES_LAUNCH_CHECK();
}

void Model::pressure_props(double dt, const double* p, const double* sw, const double* sg, hipStream_t s) {
  GridDev G = grid_dev(grid, gravity_, env_nx_);
  const PressureProps Q{mob_t.p, acc.p, grav_.p, pc_.p, mob_o_.p, mob_w_.p, mob_g_.p, rho_w_.p, rho_o_.p, rho_g_.p};
  k_props_pressure<<<grid_for(N_, kBlock, 1 << 16), kBlock, 0, s>>>(G, F, pvt, dt, p, sw, sg, pv.p, Q);
  IMPES_LAUNCH_CHECK();
}

void Model::eval_props(long long n, const double* p, const double* sw, const double* sg, double* out, hipStream_t s) {
  if (n <= 0) return;
  k_eval_props<<<grid_for(n, kBlock, 1 << 16), kBlock, 0, s>>>(F, pvt, n, p, sw, sg, out);
  IMPES_LAUNCH_CHECK();
}

void Model::eval_pvt(int key, long long n, const double* p, double* out, hipStream_t s) {
  IMPES_REQUIRE(pvt.n > 0, "no PVT table loaded");
  IMPES_REQUIRE(key >= 0 && key < 8, "bad PVT key");
  if (n <= 0) return;
  k_eval_pvt<<<grid_for(n, kBlock, 1 << 16), kBlock, 0, s>>>(pvt, key, n, p, out);
  IMPES_LAUNCH_CHECK();
}

}  // namespace impes
