// Device-side black-oil physics of the IMPES step (FP64), restating
// src/simulator/fluid.py and src/simulator/pvt.py of the reference.
#pragma once

#include "common.h"

namespace impes {

enum PvtKey { kBo = 0, kBw = 1, kBg = 2, kMuO = 3, kMuW = 4, kMuG = 5, kRs = 6, kRv = 7, kPvtKeys = 8 };

// Fluid / rock / scheme parameters (fluid.py:26-110, simulation.py:826-828,1354,1377).
struct FluidParams {
  int stone2;
  double nw, no, ng, ko_end_w, ko_end_g, now_, nog;
  double sw_cr, so_r, sg_cr;
  double mu_o, mu_w, mu_g;            // Pa s (no PVT table)
  double rho_o_ref, rho_w_ref, rho_g_ref;
  double c_o, c_w, c_g, c_r, cf;      // 1/Pa
  double pc_scale, pc_exp, pcog_scale, pcog_exp;
  double g;                           // 9.81
  double max_ds;                      // max_saturation_change
  int max_substeps;
  double rate_scale;                  // global_rate_scale
};

// PVT table (pvt.py): pressure in MPa, 8 columns. Row r < n of tab holds, for every
// column, the slope of the segment above node r and the value at the node (row n - 1:
// slope 0), row n slope 0 and the value at node 0: one 128-byte line for all the
// columns of a pressure, and no case split for pressures outside the table.
struct PvtDev {
  int n = 0;
  const double* P = nullptr;
  const double2* tab = nullptr;  // (n + 1) x 8, {slope, value}
};

// One well (well.py:10-55 + the branch flags of simulation.py:1051-1347,1622-1660).
struct WellDesc {
  int cell;                // z-fastest flat index (simulation.py:816)
  int producer;            // 0 injector, 1 producer
  int control;             // 0 rate, 1 bhp, 2 other (ignored)
  int gas;                 // injected phase: 0 water, 1 gas
  int surface;             // rate_type == "surface"
  int surface_phase;       // 0 oil, 1 water, 2 gas, 3 liquid
  int has_bhp_min;
  int lim_mask;            // bit0 wopr, bit1 wlpr, bit2 wgpr, bit3 liqr
  double value;            // m3/day or MPa
  double wi;               // Peaceman index (non-SI, well.py:44-51)
  double bhp_min;          // MPa
  double lim[4];           // m3/day
};

// x / d, correctly rounded, from r = 1/d (rounded): Markstein's quotient correction
// (P. W. Markstein, IBM J. Res. Dev. 34, 1990). 3 operations where the general division
// takes about 10; x = +-inf keeps its quotient.
__device__ __forceinline__ double div_by(double x, double d, double r) {
  const double q = x * r;
  const double e = fma(-q, d, x);
  return e == e ? fma(e, r, q) : q;
}
__device__ __forceinline__ double mega(double p_pa) { return div_by(p_pa, 1e6, 1.0 / 1e6); }

// np.interp(p/1e6, P, col, left=col[0], right=col[-1]); products and sums are
// rounded separately, as numpy does. The table row depends only on the pressure, so it
// is located once (pvt_locate) and read for every column that pressure needs
// (pvt_at): one search per pressure instead of one per property.
struct PvtAt {
  double dx;  // p / 1e6 less its node (0 outside the table, NaN for a NaN)
  int row;    // of PvtDev::tab
};

// K pressures at once: each step of the searches is one load and no branch (the number
// of steps depends on the table alone), and the K chains of dependent loads overlap.
template <int K>
__device__ __forceinline__ void pvt_locate(const PvtDev& T, const double (&p_pa)[K], PvtAt (&a)[K]) {
  const double* __restrict__ xp = T.P;
  const int n = T.n;
  const double first = xp[0], last = xp[n - 1];
  double x[K], node[K];
  int lo[K];
#pragma unroll
  for (int q = 0; q < K; ++q) {
    x[q] = mega(p_pa[q]);
    lo[q] = 0;
    node[q] = first;
  }
  for (int len = n - 1; len > 1;) {
    const int half = len >> 1;
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const double v = xp[lo[q] + half];
      const bool up = v <= x[q];
      lo[q] = up ? lo[q] + half : lo[q];
      node[q] = up ? v : node[q];
    }
    len -= half;
  }
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const bool below = x[q] < first, above = x[q] >= last;
    a[q].row = below ? n : above ? n - 1 : lo[q];
    a[q].dx = below || above ? 0.0 : x[q] - node[q];
  }
}
__device__ __forceinline__ PvtAt pvt_locate(const PvtDev& T, double p_pa) {
  const double p[1] = {p_pa};
  PvtAt a[1];
  pvt_locate(T, p, a);
  return a[0];
}

__device__ __forceinline__ double pvt_at(const PvtDev& T, int key, const PvtAt& a) {
#pragma clang fp contract(off)
  const double2 e = T.tab[a.row * kPvtKeys + key];
  return e.x * a.dx + e.y;
}

__device__ __forceinline__ double pvt_eval(const PvtDev& T, int key, double p_pa) {
  return pvt_at(T, key, pvt_locate(T, p_pa));
}

__device__ __forceinline__ double clamp01(double x) { return fmin(fmax(x, 0.0), 1.0); }

// x^e for the curve exponents: the common Corey exponents 2 and 1 as the exact
// product (pow goes through log and exp in FP64); the branch is uniform (e is a
// fluid constant)
__device__ __forceinline__ double powe(double x, double e) {
  if (e == 2.0) return x * x;
  if (e == 1.0) return x;
  return pow(x, e);
}

// fluid.py:231-248, 377-435 -> kro, krw, krg
__device__ __forceinline__ void relperms(const FluidParams& F, double sw, double sg, double& kro, double& krw,
                                         double& krg) {
  const double denom = 1.0 - F.sw_cr - F.so_r;
  const double sn = clamp01((sw - F.sw_cr) / denom);
  krw = powe(sn, F.nw);
  if (F.stone2) {
    const double swn = clamp01((sw - F.sw_cr) / (denom + 1e-12));
    const double dg = 1.0 - F.sg_cr - F.so_r;
    const double sgn = clamp01((sg - F.sg_cr) / (dg + 1e-12));
    const double k = F.ko_end_w * powe(1.0 - swn, F.now_) + F.ko_end_g * powe(1.0 - sgn, F.nog) -
                     fmin(F.ko_end_w, F.ko_end_g);
    kro = fmax(k, 0.0);
  } else {
    kro = powe(1.0 - sn, F.no);
  }
  const double sg2 = clamp01(sg / (1.0 - F.sw_cr - F.so_r + 1e-10));
  krg = powe(sg2, F.ng);
}

// fluid.py:273-287
__device__ __forceinline__ double pc_ow(const FluidParams& F, double sw) {
  if (F.pc_scale == 0.0) return 0.0;
  const double sn = clamp01((sw - F.sw_cr) / (1.0 - F.sw_cr - F.so_r));
  return F.pc_scale * pow(1.0 - sn + 1e-6, -F.pc_exp);
}

// fluid.py:288-296
__device__ __forceinline__ double pc_og(const FluidParams& F, double sg) {
  if (F.pcog_scale == 0.0) return 0.0;
  const double d = 1.0 - F.sw_cr - F.so_r;
  const double sn = clamp01(sg / (d + 1e-12));
  return F.pcog_scale * pow(1.0 - sn + 1e-6, -F.pcog_exp);
}

// phase viscosities in Pa s (simulation.py:875-877)
// `at`: the located pressure p (pvt_locate(T, p)) when the caller has it
__device__ __forceinline__ void viscosities(const FluidParams& F, const PvtDev& T, double p, double& mo, double& mw,
                                            double& mg, const PvtAt* at = nullptr) {
  if (T.n > 0) {
    const PvtAt a = at ? *at : pvt_locate(T, p);
    mo = pvt_at(T, kMuO, a) * 1e-3;
    mw = pvt_at(T, kMuW, a) * 1e-3;
    mg = pvt_at(T, kMuG, a) * 1e-3;
  } else {
    mo = F.mu_o;
    mw = F.mu_w;
    mg = F.mu_g;
  }
}

// The pressures whose formation volume factors the compressibility takes: its own and
// the two +-0.1 MPa away (fluid.py:190-222).
__device__ __forceinline__ void ct_pressures(double p, double (&q)[3]) {
  const double pm = mega(p);
  q[0] = pm * 1e6;
  q[1] = (pm + 0.1) * 1e6;
  q[2] = (pm - 0.1) * 1e6;
}

// fluid.py:190-222 (central difference of B over +-0.1 MPa); fluid.py:47-48 without PVT.
// `at`: the located ct_pressures when the caller has them
__device__ __forceinline__ double total_compressibility(const FluidParams& F, const PvtDev& T, double p, double sw,
                                                        double sg, const PvtAt* at = nullptr) {
  if (T.n == 0) return F.cf;
  PvtAt a[3];
  if (at) {
    for (int q = 0; q < 3; ++q) a[q] = at[q];
  } else {
    double pq[3];
    ct_pressures(p, pq);
    pvt_locate(T, pq, a);
  }
  double c[3];
  const int keys[3] = {kBw, kBo, kBg};
  for (int q = 0; q < 3; ++q) {
    const double b0 = pvt_at(T, keys[q], a[0]);
    const double bp = pvt_at(T, keys[q], a[1]);
    const double bm = pvt_at(T, keys[q], a[2]);
    const double dB = div_by(bp - bm, 2 * 0.1, 1.0 / (2 * 0.1));
    c[q] = mega(-(dB / (b0 + 1e-12)));
  }
  const double so = 1.0 - sw - sg;
  return F.c_r + sw * c[0] + so * c[1] + sg * c[2];
}

// fluid.py:129-158, 330-375
__device__ __forceinline__ void densities(const FluidParams& F, const PvtDev& T, double p, double& rw, double& ro,
                                          double& rg, const PvtAt* at = nullptr) {
  if (T.n == 0) {
    rw = F.rho_w_ref * (1.0 + F.c_w * (p - 1e5));
    ro = F.rho_o_ref * (1.0 + F.c_o * (p - 1e5));
    rg = F.rho_g_ref * (1.0 + F.c_g * (p - 1e5));
    return;
  }
  const PvtAt a = at ? *at : pvt_locate(T, p);
  const double bw = pvt_at(T, kBw, a), bo = pvt_at(T, kBo, a), rs = pvt_at(T, kRs, a);
  const double bg = pvt_at(T, kBg, a), rv = pvt_at(T, kRv, a);
  rw = F.rho_w_ref / (bw + 1e-12);
  ro = (F.rho_o_ref + rs * F.rho_g_ref) / (bo + 1e-12);
  rg = (F.rho_g_ref + rv * F.rho_o_ref) / (bg + 1e-12);
}

}  // namespace impes
