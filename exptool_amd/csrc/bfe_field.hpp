// Point evaluation of folded SL and EOF tables (device side).
//
// "Folded" tables hold sum_n a_n T_n per table node for a fixed coefficient
// set (an exact linear rewrite of the reference sums over n, whose only effect
// is rounding), so evaluation gathers (2 mmax + 1) values per EOF node and
// (lmax + 1)^2 per SL node instead of norder / nmax times that.
#pragma once

#include "bfe_internal.hpp"

namespace bfe {

struct SLOut {
  double den0, den1, pot0, pot1, potr, pott, potp;
  double pot;   // pot0 + pot1
};

struct EOFOut {
  double p0, p, fr, fp, fz, d0, d;
  double fr0, fz0;   // the m = 0 parts of fr and fz (eof.force_eval perturb=True)
};

// Folded table layouts (float32, streamed as float4):
//  SL : per radial node i, one 8-float block per (l, m) pair in m-major order
//       (m = 0..L, l = m..L):
//         [E_c(i), E_s(i), dE_c(i), dE_s(i), D1_c, D1_s, D2_c, D2_s]
//       with dE(i) = E(i+1) - E(i), so that E at x2 is E(i) + x2 dE(i)
//       with D1, D2 at the stencil centre c = max(i, 1); after the numr
//       nodes of these, the density blocks per node and pair:
//         [Dn_c(i), Dn_s(i), Dn_c(i+1), Dn_s(i+1)].
//       E = sum_n a N_lm ef/sqrt(ev), Dn = sum_n a N_lm ef sqrt(ev),
//       D1 = (G_{c+1} - G_{c-1})/2, D2 = G_{c-1} - 2 G_c + G_{c+1},
//       G = sum_n a N_lm ef p0/sqrt(ev)   (S entries are 0 for m = 0).
//       Forces read two float4 per pair, both from node i.
//  EOF: per grid node, one 8-float block per m = 0..M:
//       [potC, rforceC, zforceC, densC, potS, rforceS, zforceS, densS];
//       then, in float64, the m = 0 cos block of each edge node
//       (eof_edge_index): [pot, rforce, zforce, dens].
// SL table values are interpolated in float32 (they are stored in float32;
// the weights are convex) and combined in float64.  EOF values are
// interpolated in float64: far from the disc plane the mapped grid cells are
// wide and the force is small against the corner values, where float32
// interpolation gave force errors of 3e-5.
__host__ __device__ inline int sl_npairs(int L) { return (L + 1) * (L + 2) / 2; }
// index of (l, m) in m-major order
__host__ __device__ inline int sl_pair(int l, int m, int L) {
  return m * (L + 1) - m * (m - 1) / 2 + (l - m);
}

// SL evaluation at (r, cos theta, phi): get_halo_dens_pot_force
// (spheresl.py:106-160) and the l,m sums of all_eval_particles / force_eval
// (spheresl.py:1276-1341, :1199-1228) with N_lm and the coefficients folded in.
// The associated Legendre functions are generated column by column (m outer,
// l inner) with the recurrences of legendre_R / dlegendre_R
// (spheresl.py:664-770), in the order the table is stored.
//   flags: BFE_COMPAT_SL_EDGE  first-cell stencil one cell outward (:150-153)
//          BFE_COMPAT_SL_COS_L cos/sin(l phi) for 0 < m (:1222-1225)
//          BFE_COMPAT_SL_DENS  den1 uses P_1^0 for m = 0 (:1323)
// LDS view of staged float4 data: reads through it are LDS instructions, not
// flat ones (which would pass through the vector-memory address path).
typedef float F4v __attribute__((ext_vector_type(4)));
typedef const F4v __attribute__((address_space(3)))* LdsF4;
__device__ __forceinline__ float4 ld4(LdsF4 p, int k) {
  const F4v v = p[k];
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float4 ld4(const float4* __restrict__ p, int k) { return p[k]; }

// Steps of the angular sums, shared by the one-lane and the split evaluation
// (field_eval_point, field_eval_split), with every fused multiply-add
// spelled out so that both give the same bits.
// P_l^m from P_{l-1}^m (pl) and P_{l-2}^m (plm1) at x (A, B of sl_lmc)
__device__ __forceinline__ double sl_next(double A, double B, double x, double pl, double plm1) {
  return fma(x * A, pl, -(B * plm1));
}
// (x^2 - 1) dP_l^m/dx (dl = l, ds = l + m)
__device__ __forceinline__ double sl_dnum(double dl, double ds, double xc, double pl,
                                          double plm1) {
  return fma(xc * dl, pl, -(ds * plm1));
}
// cos/sin(m phi) one order up (m = 1 gives c1, s1 exactly from 1, 0, c1, -s1)
__device__ __forceinline__ void cheb_next(double c1, double& c, double& s, double& cp,
                                          double& sp) {
  const double cn = fma(2.0 * c1, c, -cp), sn = fma(2.0 * c1, s, -sp);
  cp = c; sp = s; c = cn; s = sn;
}
// the m sums Pc.. of one column combined with cos/sin(m phi)
__device__ __forceinline__ double cs_sum(double c, double a, double s, double b) {
  return fma(c, a, s * b);
}

// Angular sums of sl_eval_folded.  The azimuthal factors cos/sin(m phi) do
// not depend on l, so the l sums are taken per m first (sum_l P_l^m E,
// sum_l P_l^m D, sum_l dP_l^m E for cos and sin) and combined with the
// factors once per m.  The l loops are branch-free: m = 0 runs alone (l = 0
// peeled) and each m > 0 peels l = m, so no accumulator passes through a
// per-lane or per-iteration branch.  A NaN cos(theta) is replaced by 0 for
// the recurrences and its l > 0 sums are zeroed at the end, which is what
// skipping them term by term gives.
template <bool DENS, typename PA>
__device__ __forceinline__ void sl_angular(const SLGeom& g, PA A, const float4* __restrict__ Nd,
                                           int L, float x1f, float x2f, float ps, double x,
                                           double c1, double s1, bool dq, double* acc) {
  const bool good = (x == x);
  const double xs = good ? x : 0.0;
  double xc = xs;   // dlegendre_R clamps x for the derivative only
  if (1.0 - fabs(xc) < 1.e-8) xc = (xc > 0) ? 1.0 - 1.e-8 : -(1.0 - 1.e-8);
  const double somx2d = 1.0 / (xc * xc - 1.0);
  const double somx2 = sqrt((1.0 - xs) * (1.0 + xs));
  // m = 0, l = 0
  const float4 a0 = ld4(A, 0), b0 = ld4(A, 1);
  const double pot0 = (double)fmaf(x2f, a0.z, a0.x);
  const double potr0 = (double)fmaf(ps, b0.z, b0.x);
  double den0 = 0.0;
  if (DENS) {
    const float4 nd = Nd[0];
    den0 = (double)fmaf(x2f, nd.z, x1f * nd.x);
  }
  double pot1 = 0, potr = 0, pott = 0, potp = 0, den1 = 0;
  // m = 0, l >= 1
  {
    double plm1 = 0.0, pl = 1.0;
#pragma unroll 2
    for (int l = 1; l <= L; ++l) {
      const int lm = lm_index(l, 0);
      const double pn = sl_next(g.lmc[kLmcA + lm], g.lmc[kLmcB + lm], xs, pl, plm1);
      plm1 = pl;
      pl = pn;
      const float4 a = ld4(A, 2 * l), b = ld4(A, 2 * l + 1);
      const double ec = (double)fmaf(x2f, a.z, a.x);
      const double dc = (double)fmaf(ps, b.z, b.x);
      // dP/dx without its factor 1/(x^2 - 1), applied once to pott below
      const double dpl = sl_dnum(g.lmc[kLmcL + lm], g.lmc[kLmcS + lm], xc, pl, plm1);
      pot1 = fma(pl, ec, pot1);
      potr = fma(pl, dc, potr);
      pott = fma(dpl, ec, pott);
      if (DENS) {
        const float4 nd = Nd[l];
        den1 += (dq ? xs : pl) * (double)fmaf(x2f, nd.z, x1f * nd.x);
      }
    }
  }
  double pmm = 1.0, fact = 1.0;
  double cmm = 1.0, smm = 0.0, cmm1 = c1, smm1 = -s1;
  int p = L + 1;
#pragma unroll 1
  for (int m = 1; m <= L; ++m) {
    pmm *= -fact * somx2;
    fact += 2.0;
    cheb_next(c1, cmm, smm, cmm1, smm1);
    double Pc = 0, Ps = 0, Rc = 0, Rs = 0, Tc = 0, Ts = 0, Nc = 0, Ns = 0;
    auto term = [&](int q, int lm, double pl, double plm1) {
      const float4 a = ld4(A, 2 * q), b = ld4(A, 2 * q + 1);
      const double ec = (double)fmaf(x2f, a.z, a.x);
      const double dc = (double)fmaf(ps, b.z, b.x);
      const double es = (double)fmaf(x2f, a.w, a.y);
      const double ds = (double)fmaf(ps, b.w, b.y);
      const double dpl = sl_dnum(g.lmc[kLmcL + lm], g.lmc[kLmcS + lm], xc, pl, plm1);
      Pc = fma(pl, ec, Pc);
      Ps = fma(pl, es, Ps);
      Rc = fma(pl, dc, Rc);
      Rs = fma(pl, ds, Rs);
      Tc = fma(dpl, ec, Tc);
      Ts = fma(dpl, es, Ts);
      if (DENS) {
        const float4 nd = Nd[q];
        Nc += pl * (double)fmaf(x2f, nd.z, x1f * nd.x);
        Ns += pl * (double)fmaf(x2f, nd.w, x1f * nd.y);
      }
    };
    double plm1 = 0.0, pl = pmm;
    term(p, lm_index(m, m), pl, plm1);
    ++p;
#pragma unroll 2
    for (int l = m + 1; l <= L; ++l, ++p) {
      const int lm = lm_index(l, m);
      const double pn = sl_next(g.lmc[kLmcA + lm], g.lmc[kLmcB + lm], xs, pl, plm1);
      plm1 = pl;
      pl = pn;
      term(p, lm, pl, plm1);
    }
    pot1 += cs_sum(cmm, Pc, smm, Ps);
    potr += cs_sum(cmm, Rc, smm, Rs);
    pott += cs_sum(cmm, Tc, smm, Ts);
    potp = fma((double)m, cs_sum(cmm, Ps, -smm, Pc), potp);
    if (DENS) den1 += cmm * Nc + smm * Ns;
  }
  pott *= somx2d;
  if (!good) {   // P_l^m = 0 for l > 0 when cos(theta) is NaN (spheresl.py:698)
    pot1 = potr = pott = potp = den1 = 0.0;
  }
  acc[0] = pot0;
  acc[1] = potr0 + potr;
  acc[2] = den0;
  acc[3] = pot1;
  acc[4] = pott;
  acc[5] = potp;
  acc[6] = den1;
}

// The sums with BFE_COMPAT_SL_COS_L: the azimuthal factor of term (l, m > 0)
// is cos/sin(l phi), so it enters per term.  Same recurrences as sl_angular.
template <bool DENS, typename PA>
__device__ __forceinline__ void sl_angular_cosl(const SLGeom& g, PA A,
                                                const float4* __restrict__ Nd, int L, float x1f,
                                                float x2f, float ps, double x, double c1,
                                                double s1, bool dq, double* acc) {
  const bool good = (x == x);
  double xc = x;
  if (good && 1.0 - fabs(xc) < 1.e-8) xc = (xc > 0) ? 1.0 - 1.e-8 : -(1.0 - 1.e-8);
  const double somx2d = 1.0 / (xc * xc - 1.0);
  const double somx2 = good ? sqrt((1.0 - x) * (1.0 + x)) : 0.0;
  double pot0 = 0, potr0 = 0, den0 = 0, pot1 = 0, potr = 0, pott = 0, potp = 0, den1 = 0;
  double pmm = 1.0, fact = 1.0;
  double cmm = 1.0, smm = 0.0, cmm1 = c1, smm1 = -s1;
  int p = 0;
#pragma unroll 1
  for (int m = 0; m <= L; ++m) {
    if (m > 0) {
      pmm *= -fact * somx2;
      fact += 2.0;
      const double cn = 2.0 * c1 * cmm - cmm1, sn = 2.0 * c1 * smm - smm1;
      cmm1 = cmm; smm1 = smm; cmm = cn; smm = sn;
    }
    double plm1 = 0.0, pl = pmm;
    double cl = cmm, sl = smm, clm1 = cmm1, slm1 = smm1;
#pragma unroll 1
    for (int l = m; l <= L; ++l, ++p) {
      const int lm = lm_index(l, m);
      if (l > m) {
        const double pn = x * g.lmc[kLmcA + lm] * pl - g.lmc[kLmcB + lm] * plm1;
        plm1 = pl;
        pl = pn;
        const double cn = 2.0 * c1 * cl - clm1, sn = 2.0 * c1 * sl - slm1;
        clm1 = cl; slm1 = sl; cl = cn; sl = sn;
      }
      const float4 a = ld4(A, 2 * p), b = ld4(A, 2 * p + 1);
      const double ec = (double)fmaf(x2f, a.z, a.x);
      const double dc = (double)fmaf(ps, b.z, b.x);
      if (l == 0) {
        pot0 = ec;
        potr0 = dc;
        if (DENS) {
          const float4 nd = Nd[p];
          den0 = (double)fmaf(x2f, nd.z, x1f * nd.x);
        }
        continue;
      }
      if (!good) continue;  // P_l^m = 0 for l > 0 when cos(theta) is NaN (spheresl.py:698)
      const double dpl = somx2d * (xc * g.lmc[kLmcL + lm] * pl - g.lmc[kLmcS + lm] * plm1);
      if (m == 0) {
        pot1 += pl * ec;
        potr += pl * dc;
        pott += dpl * ec;
        if (DENS) {
          const float4 nd = Nd[p];
          den1 += (dq ? x : pl) * (double)fmaf(x2f, nd.z, x1f * nd.x);
        }
        continue;
      }
      const double es = (double)fmaf(x2f, a.w, a.y);
      const double ds = (double)fmaf(ps, b.w, b.y);
      const double pa = ec * cl + es * sl;
      pot1 += pl * pa;
      potr += pl * (dc * cl + ds * sl);
      pott += dpl * pa;
      potp += pl * m * (-ec * sl + es * cl);
      if (DENS) {
        const float4 nd = Nd[p];
        const double nc = (double)fmaf(x2f, nd.z, x1f * nd.x);
        const double ns = (double)fmaf(x2f, nd.w, x1f * nd.y);
        den1 += pl * (nc * cl + ns * sl);
      }
    }
  }
  acc[0] = pot0;
  acc[1] = potr0 + potr;
  acc[2] = den0;
  acc[3] = pot1;
  acc[4] = pott;
  acc[5] = potp;
  acc[6] = den1;
}

// What a point's radial cell gives beside its weights: the background
// potential P0 the sums are scaled by, the scale fac of the radial derivative
// sums and the stencil offset ps of the potential derivative (spheresl.py:
// 141-157).
struct SLRadial {
  double P0, fac;
  float ps;
};
__device__ __forceinline__ SLRadial sl_radial(const SLGeom& g, const SLCell& cell,
                                              uint32_t flags) {
  const int i = cell.i;
  SLRadial q;
  q.P0 = fma(cell.x1, g.p0[i], cell.x2 * g.p0[i + 1]);
  q.fac = (g.cmap == 1) ? (1.0 - cell.x) * (1.0 - cell.x) * g.dfac
                        : d_xi_to_r(cell.x, g.cmap, g.scale) * g.idxi;
  q.ps = (float)((i == 0) ? ((flags & BFE_COMPAT_SL_EDGE) ? cell.x2 : cell.x2 - 1.0) : cell.x2);
  return q;
}

// The sums of sl_eval_folded in cell `cell` from its node's blocks: A (2 np
// float4, in global memory or LDS) and the density block Nd.
template <bool DENS, typename PA>
__device__ __forceinline__ void sl_eval_cell(const SLGeom& g, PA A, const float4* __restrict__ Nd,
                                             int L, const SLCell& cell, double costh, double c1,
                                             double s1, uint32_t flags, SLOut& o) {
  const int i = cell.i;
  const double x1 = cell.x1, x2 = cell.x2;
  const SLRadial rad = sl_radial(g, cell, flags);
  const double P0 = rad.P0;
  const double D0 = DENS ? x1 * g.d0[i] + x2 * g.d0[i + 1] : 0.0;
  const float ps = rad.ps;
  const bool dq = (flags & BFE_COMPAT_SL_DENS) != 0;
  double acc[7];
  if (flags & BFE_COMPAT_SL_COS_L)
    sl_angular_cosl<DENS>(g, A, Nd, L, (float)x1, (float)x2, ps, costh, c1, s1, dq, acc);
  else
    sl_angular<DENS>(g, A, Nd, L, (float)x1, (float)x2, ps, costh, c1, s1, dq, acc);
  o.pot0 = acc[0] * P0;
  o.pot = fma(acc[3], P0, acc[0] * P0);
  o.potr = acc[1] * rad.fac;
  o.den0 = acc[2] * D0;
  o.pot1 = acc[3] * P0;
  o.pott = acc[4] * P0;
  o.potp = acc[5] * P0;
  o.den1 = acc[6] * D0;
}

// pcell: the radial cell of r when the caller has located it already.
// STAGED: node i's force blocks are read from the LDS copy Abase at
// (i - ibase) * 2 np float4 (a block stages its nodes there); otherwise from
// the folded table itself.
template <bool DENS, bool STAGED = false>
__device__ __forceinline__ void sl_eval_folded(const SLGeom& g, const float* __restrict__ F,
                                               int L, double r, double costh, double c1,
                                               double s1, uint32_t flags, SLOut& o,
                                               const SLCell* pcell = nullptr,
                                               const float4* Abase = nullptr, int ibase = 0) {
  const SLCell cell = pcell ? *pcell : sl_locate(r, g.cmap, g.scale, g.xi, g.numr, g.idxi, g.xi0, g.xin);
  const int i = cell.i;
  const int np = sl_npairs(L);
  const float4* __restrict__ Nd =
      reinterpret_cast<const float4*>(F + (size_t)g.numr * np * 8) + (size_t)i * np;
  if (STAGED) {
    const LdsF4 A = (LdsF4)Abase + (size_t)(i - ibase) * 2 * np;
    sl_eval_cell<DENS>(g, A, Nd, L, cell, costh, c1, s1, flags, o);
  } else {
    const float4* __restrict__ A = reinterpret_cast<const float4*>(F) + (size_t)i * 2 * np;
    sl_eval_cell<DENS>(g, A, Nd, L, cell, costh, c1, s1, flags, o);
  }
}

// m = 0 corner values [pot, rforce, zforce, dens] of a cell: from the float64
// edge blocks in the last grid column or row, else from the float32 table.
struct EOFCorners0 {
  double4 a, b, c, e;   // (ix, iy), (ix, iy+1), (ix+1, iy), (ix+1, iy+1)
};
__device__ __forceinline__ EOFCorners0 eof_corners0(const EOFGeom& g, const float* __restrict__ F,
                                                    const EOFCell& cell, const float4& a,
                                                    const float4& b, const float4& c,
                                                    const float4& e) {
  EOFCorners0 q;
  if (cell.ix == g.numx - 1 || cell.iy == g.numy - 1) {
    const double4* __restrict__ E =
        reinterpret_cast<const double4*>(F + eof_fold32_floats(g.numx, g.numy, g.mmax));
    const int x0 = cell.ix, y0 = cell.iy;
    q.a = E[eof_edge_index(x0, y0, g.numx, g.numy)];
    q.b = E[eof_edge_index(x0, y0 + 1, g.numx, g.numy)];
    q.c = E[eof_edge_index(x0 + 1, y0, g.numx, g.numy)];
    q.e = E[eof_edge_index(x0 + 1, y0 + 1, g.numx, g.numy)];
  } else {
    q.a = make_double4(a.x, a.y, a.z, a.w);
    q.b = make_double4(b.x, b.y, b.z, b.w);
    q.c = make_double4(c.x, c.y, c.z, c.w);
    q.e = make_double4(e.x, e.y, e.z, e.w);
  }
  return q;
}
__device__ __forceinline__ double eof_bil0(const EOFCell& w, double a, double c, double b,
                                           double e) {
  return fma(w.c11, e, fma(w.c01, b, fma(w.c10, c, w.c00 * a)));
}
// One order m > 0: the corners (a, b, c, e cos, a2.. sin blocks as
// EOFCorners0) interpolated in float32, combined with cm, sm = cos/sin(m phi)
// in float64.  t: the terms of p, fr, fz, and of fp without its factor m.
struct EOFWeights32 {
  float v00, v10, v01, v11;
};
__device__ __forceinline__ double eof_bil(const EOFWeights32& v, float a, float c, float b,
                                          float e) {
  return (double)fmaf(v.v11, e, fmaf(v.v01, b, fmaf(v.v10, c, v.v00 * a)));
}
__device__ __forceinline__ void eof_term(const EOFWeights32& v, const float4& a, const float4& b,
                                         const float4& c, const float4& e, const float4& a2,
                                         const float4& b2, const float4& c2, const float4& e2,
                                         double cm, double sm, double t[4]) {
  const double pc = eof_bil(v, a.x, c.x, b.x, e.x), ps = eof_bil(v, a2.x, c2.x, b2.x, e2.x);
  const double rc = eof_bil(v, a.y, c.y, b.y, e.y), rs = eof_bil(v, a2.y, c2.y, b2.y, e2.y);
  const double zc = eof_bil(v, a.z, c.z, b.z, e.z), zs = eof_bil(v, a2.z, c2.z, b2.z, e2.z);
  t[0] = cs_sum(cm, pc, sm, ps);
  t[1] = cs_sum(cm, rc, sm, rs);
  t[2] = cs_sum(cm, zc, sm, zs);
  t[3] = cs_sum(sm, pc, -cm, ps);
}

// The sums of eof_eval_folded from the cell's four node blocks A (ix, iy), B (ix,
// iy + 1), C (ix + 1, iy), D (ix + 1, iy + 1).
template <bool DENS, int MU = 1>
__device__ __forceinline__ void eof_eval_corners(const EOFCell& cell, int M, const EOFCorners0& q0,
                                                 const float4* __restrict__ A,
                                                 const float4* __restrict__ B,
                                                 const float4* __restrict__ C,
                                                 const float4* __restrict__ D, double c1, double s1,
                                                 EOFOut& o) {
  const double p0 = eof_bil0(cell, q0.a.x, q0.c.x, q0.b.x, q0.e.x);
  const double fr0 = eof_bil0(cell, q0.a.y, q0.c.y, q0.b.y, q0.e.y);
  const double fz0 = eof_bil0(cell, q0.a.z, q0.c.z, q0.b.z, q0.e.z);
  const double d0 = DENS ? eof_bil0(cell, q0.a.w, q0.c.w, q0.b.w, q0.e.w) : 0.0;
  double fr = fr0, fz = fz0, p = 0, fp = 0, d = 0;
  double cm = 1.0, sm = 0.0, cm1 = c1, sm1 = -s1;
  // m > 0: the corners of the float32 table interpolated in float32 (one
  // conversion per value instead of four), the sums over m in float64
  const EOFWeights32 v{(float)cell.c00, (float)cell.c10, (float)cell.c01, (float)cell.c11};
#pragma unroll MU
  for (int m = 1; m <= M; ++m) {
    cheb_next(c1, cm, sm, cm1, sm1);
    const float4 a = A[2 * m], b = B[2 * m], c = C[2 * m], e = D[2 * m];
    const float4 a2 = A[2 * m + 1], b2 = B[2 * m + 1], c2 = C[2 * m + 1], e2 = D[2 * m + 1];
    double t[4];
    eof_term(v, a, b, c, e, a2, b2, c2, e2, cm, sm, t);
    p += t[0];
    fr += t[1];
    fz += t[2];
    fp = fma((double)m, t[3], fp);
    if (DENS)
      d += cs_sum(cm, eof_bil(v, a.w, c.w, b.w, e.w), sm, eof_bil(v, a2.w, c2.w, b2.w, e2.w));
  }
  o.p0 = p0;
  o.p = p;
  o.fr = fr;
  o.fz = fz;
  o.fp = fp;
  o.d0 = d0;
  o.d = d;
  o.fr0 = fr0;
  o.fz0 = fz0;
}

// EOF evaluation at planar radius R, height z, angle phi from the folded
// table (8-float block per m).  Bilinear weights as eof.py:443-451; sums as
// force_eval (eof.py:842-870) and accumulated_eval_particles (:1092-1138):
// fp = sum m (C sin m phi potC - S cos m phi potS) = -dPhi/dphi.  MU: unroll
// count of the m loop (2 measured 7 % faster in the RK4 kernel, slower in
// the leapfrog one).  Cells of the last grid column or row take their m = 0
// corner values from the float64 edge blocks that follow the float32 table:
// past the outer edges the weights extrapolate linearly (eof.py:414-415) and
// grow without bound, and with them the rounding of the table values; the
// m = 0 terms carry the largest values.  The m > 0 terms stay float32.
template <bool DENS, int MU = 1>
__device__ __forceinline__ void eof_eval_folded(const EOFGeom& g, const float* __restrict__ F,
                                                double R, double z, double c1, double s1,
                                                EOFOut& o) {
  const EOFCell cell = eof_locate(R, z, g.cmap, g.ascale, g.ihscale, g.xmin, g.idx, g.ymin, g.idy,
                                  g.numx, g.numy);
  const int ny1 = g.numy + 1;
  const int ns4 = 2 * (g.mmax + 1);
  const size_t n00 = (size_t)cell.ix * ny1 + cell.iy;
  const float4* __restrict__ A = reinterpret_cast<const float4*>(F) + n00 * ns4;  // (ix, iy)
  const float4* __restrict__ B = A + ns4;                                          // (ix, iy+1)
  const float4* __restrict__ C = A + (size_t)ny1 * ns4;                            // (ix+1, iy)
  const float4* __restrict__ D = C + ns4;                                          // (ix+1, iy+1)
  // m = 0: [pot, rforce, zforce, dens] of the four corners
  const EOFCorners0 q0 = eof_corners0(g, F, cell, A[0], B[0], C[0], D[0]);
  eof_eval_corners<DENS, MU>(cell, g.mmax, q0, A, B, C, D, c1, s1, o);
}

// The SL radial cell field_eval_point locates for the point (x, y, z).
__device__ __forceinline__ SLCell field_sl_cell(const SLGeom& g, double x, double y, double z) {
  const double r2 = sqrt(fma(x, x, y * y)) + 1.e-15;
  const double r3 = sqrt(fma(r2, r2, z * z)) + 1.e-15;
  return sl_locate(r3, g.cmap, g.scale, g.xi, g.numr, g.idxi, g.xi0, g.xin);
}

// Frozen disc + halo field at a Cartesian point, Fields.return_forces_cart
// (potential.py:445-497).  comp receives the 8 reference outputs.
struct FieldTables {
  SLGeom slg;
  EOFGeom eg;
  const float* slF;
  const float* eofF;
  int lmax;          // folded SL layout size (table lmax)
  uint32_t flags;
  double ximin;      // min(xi_halo) for the azimuthal-force guard (:483-485)
  double crot, srot; // cos/sin of rotpos
};

// Radii, reciprocals and angles of a point (potential.py:449-463).
struct FieldGeom {
  double r2, r3, ir2, ir3, costh;
  double c1, s1;   // cos/sin(phi + rotpos)
};
__device__ __forceinline__ FieldGeom field_geom(const FieldTables& T, double x, double y,
                                                double z) {
  FieldGeom q;
  const double rho = sqrt(fma(x, x, y * y));
  q.r2 = rho + 1.e-15;
  q.r3 = sqrt(fma(q.r2, q.r2, z * z)) + 1.e-15;
  // reciprocals once; the force combination multiplies by them
  q.ir2 = 1.0 / q.r2;
  q.ir3 = 1.0 / q.r3;
  q.costh = z * q.ir3;
  double c0, s0;
  planar_angle(x, y, rho, c0, s0);
  q.c1 = fma(c0, T.crot, -(s0 * T.srot));
  q.s1 = fma(s0, T.crot, c0 * T.srot);
  return q;
}

// The 8 outputs of return_forces_cart from the disc terms (fr, fz, fp and the
// potential) and the halo terms (dPhi/dr, dPhi/dcos(theta), dPhi/dphi and the
// potential).
__device__ __forceinline__ void field_combine(const FieldTables& T, const FieldGeom& q, double x,
                                              double y, double z, double dfr, double dfz,
                                              double dfp, double dp, double hfr, double hft,
                                              double hfp, double hp, double comp[8]) {
  if (q.r3 < T.ximin) {
    hfp = 0.0;
    dfp = 0.0;
  }
  const double r2sq = q.r2 * q.r2, ir2sq = q.ir2 * q.ir2, ir3cu = q.ir3 * q.ir3 * q.ir3;
  const double yi = y * ir2sq, xi = x * ir2sq;
  comp[0] = fma(dfr, x * q.ir2, -(dfp * yi));
  comp[1] = fma(hfp, yi, -fma(hfr, x * q.ir3, -(hft * (x * z * ir3cu))));
  comp[2] = fma(dfr, y * q.ir2, dfp * xi);
  comp[3] = -fma(hfp, xi, fma(hfr, y * q.ir3, -(hft * (y * z * ir3cu))));
  comp[4] = dfz;
  comp[5] = -fma(hfr, z * q.ir3, hft * (r2sq * ir3cu));
  comp[6] = dp;
  comp[7] = hp;
}

// pcell/slA/slbase: the point's SL cell (field_sl_cell) and SL node blocks
// staged by the caller in LDS (STAGED, see sl_eval_folded).  MU: unroll count
// of the EOF m loop (eof_eval_folded).
template <bool STAGED = false, int MU = 1>
__device__ __forceinline__ void field_eval_point(const FieldTables& T, double x, double y,
                                                 double z, double comp[8],
                                                 const SLCell* pcell = nullptr,
                                                 const float4* slA = nullptr, int slbase = 0) {
  const FieldGeom q = field_geom(T, x, y, z);
  EOFOut d;
  eof_eval_folded<false, MU>(T.eg, T.eofF, q.r2, z, q.c1, q.s1, d);
  SLOut h;
  sl_eval_folded<false, STAGED>(T.slg, T.slF, T.lmax, q.r3, q.costh, q.c1, q.s1, T.flags, h, pcell,
                                slA, slbase);
  field_combine(T, q, x, y, z, d.fr, d.fz, d.fp, d.p + d.p0, h.potr, h.pott, h.potp, h.pot, comp);
}

// LDS a block may fill with SL node force blocks (2 np float4 per node): 40
// nodes of lmax 6 (35 KB, four blocks per CU); measured on the workload,
// 16, 32, 40 and 48 nodes gave 243, 222, 219 and 230 us.
constexpr int kStageFloat4 = 40 * 56;

// Block-wide minimum and maximum of v (all 256 threads call it).
__device__ __forceinline__ void block_minmax(int v_min, int v_max, int* smin, int* smax,
                                             int& out_min, int& out_max) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    v_min = min(v_min, __shfl_xor(v_min, o, 64));
    v_max = max(v_max, __shfl_xor(v_max, o, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    smin[threadIdx.x >> 6] = v_min;
    smax[threadIdx.x >> 6] = v_max;
  }
  __syncthreads();
  out_min = min(min(smin[0], smin[1]), min(smin[2], smin[3]));
  out_max = max(max(smax[0], smax[1]), max(smax[2], smax[3]));
}

// Copies the force blocks of the SL nodes used by the block's points to
// stage when they fit (all 256 threads call it; live: the thread has a
// point, node: its SL node).  Returns whether they were staged; imin is then
// the first staged node.  Ends with a barrier.
__device__ __forceinline__ bool stage_sl_nodes(const FieldTables& T, bool live, int node,
                                               float4* stage, int* smin, int* smax, int& imin) {
  const int np2 = sl_npairs(T.lmax) * 2;   // float4 per SL node
  int imax;
  block_minmax(live ? node : 0x7fffffff, live ? node : -1, smin, smax, imin, imax);
  bool staged = false;
  if (imax >= imin && (imax - imin + 1) * np2 <= kStageFloat4) {
    const float4* src = reinterpret_cast<const float4*>(T.slF) + (size_t)imin * np2;
    const int cnt = (imax - imin + 1) * np2;
    for (int k = threadIdx.x; k < cnt; k += 256) stage[k] = src[k];
    staged = true;
  }
  __syncthreads();
  return staged;
}

// ---------------------------------------------------------------------------
// Split evaluation: 64 points per block of eight waves
// ---------------------------------------------------------------------------
// One lane per point leaves the chip idle when there are few points, and a
// lane's ~1 700 instructions, two gather rounds per order and pair, are then
// one latency chain (one orbit: 7.9 us a step; 12 800 orbits, 200 waves:
// 14.6 us).  Here lane q of all eight waves holds point q of the block, and
// the waves share the orders: wave e < 4 takes the EOF orders m = e, e + 4,
// .., wave 4 + s the SL columns m = s, 7 - s, 8 + s, 15 - s, .. (the columns
// get shorter with m, so a long one is paired with a short one: for lmax 6
// each wave has seven (l, m) pairs).  The
// orders are wave-uniform, so their constants stay scalar and no lane
// diverges.  Each wave leaves its terms per order in LDS; after a barrier
// wave w sums component w (EOF pot, fr, fz, fp; SL pot, dr, dcos, dphi) over
// the orders in the order field_eval_point adds them, and after another
// every wave has the eight sums and combines them.  The results are those of
// field_eval_point bit for bit.
constexpr int kSplitPts = 64;
constexpr int kSplitThreads = 512;
constexpr int kSplitChunk = 8;   // SL pairs whose table reads are in flight together
// doubles of LDS: EOF terms [M + 1][4][64], SL terms [L + 2][4][64], sums [8][64]
__host__ __device__ constexpr int split_lds_doubles(int M, int L) {
  return (4 * (M + 1) + 4 * (L + 2) + 8) * kSplitPts;
}

struct SplitWave {
  int lane, wave;
};
__device__ __forceinline__ SplitWave split_wave() {
  return SplitWave{(int)(threadIdx.x & 63), __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)};
}

// A wave-uniform value, kept in a scalar register.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The SL columns of wave s after column m: s -> 7 - s -> 8 + s -> 15 - s -> ..
__host__ __device__ constexpr int split_next_column(int m, int s) {
  return (m | 3) + ((m & 4) ? 1 + s : 4 - s);
}

// What a point's SL waves share: the radial cell, cos(theta) for the sums and
// clamped for the derivative (legendre_R, dlegendre_R), sin(theta).
struct SplitSL {
  SLCell cell;
  double xs, xc, somx2;
  bool good;
};
__device__ __forceinline__ SplitSL split_sl_point(const FieldTables& T, const FieldGeom& q) {
  SplitSL o;
  o.cell = sl_cell_index(q.r3, T.slg.cmap, T.slg.scale, T.slg.numr, T.slg.idxi, T.slg.xi0,
                         T.slg.xin);
  o.good = (q.costh == q.costh);
  o.xs = o.good ? q.costh : 0.0;
  o.xc = o.xs;
  if (1.0 - fabs(o.xc) < 1.e-8) o.xc = (o.xc > 0) ? 1.0 - 1.e-8 : -(1.0 - 1.e-8);
  o.somx2 = sqrt((1.0 - o.xs) * (1.0 + o.xs));
  return o;
}

// P_m^m and cos/sin(m phi), taken up from order to order.
struct SplitOrder {
  double pmm = 1.0, fact = 1.0, c = 1.0, s = 0.0, cp, sp;
  __device__ __forceinline__ SplitOrder(double c1, double s1) : cp(c1), sp(-s1) {}
  __device__ __forceinline__ void next(double c1, double somx2) {
    pmm *= -fact * somx2;
    fact += 2.0;
    cheb_next(c1, c, s, cp, sp);
  }
};

// The l sums of one column.
struct SplitColumn {
  double pl, plm1 = 0.0, Pc = 0.0, Ps = 0.0, Rc = 0.0, Rs = 0.0, Tc = 0.0, Ts = 0.0;
  __device__ __forceinline__ explicit SplitColumn(double p) : pl(p) {}
  __device__ __forceinline__ void step(const double2& ab, double xs) {
    const double pn = sl_next(ab.x, ab.y, xs, pl, plm1);
    plm1 = pl;
    pl = pn;
  }
  __device__ __forceinline__ void term(const float4& a, const float4& b, float x2f, float ps,
                                       double dl, double dlm, double xc) {
    const double ec = (double)fmaf(x2f, a.z, a.x), es = (double)fmaf(x2f, a.w, a.y);
    const double dc = (double)fmaf(ps, b.z, b.x), ds = (double)fmaf(ps, b.w, b.y);
    const double dpl = sl_dnum(dl, dlm, xc, pl, plm1);
    Pc = fma(pl, ec, Pc);
    Ps = fma(pl, es, Ps);
    Rc = fma(pl, dc, Rc);
    Rs = fma(pl, ds, Rs);
    Tc = fma(dpl, ec, Tc);
    Ts = fma(dpl, es, Ts);
  }
  // the column's terms (pot, dr, dcos, and dphi without its factor m)
  __device__ __forceinline__ void store(double* o, const SplitOrder& t, bool good) const {
    o[0] = good ? cs_sum(t.c, Pc, t.s, Ps) : 0.0;
    o[kSplitPts] = good ? cs_sum(t.c, Rc, t.s, Rs) : 0.0;
    o[2 * kSplitPts] = good ? cs_sum(t.c, Tc, t.s, Ts) : 0.0;
    o[3 * kSplitPts] = good ? cs_sum(t.c, Ps, -t.s, Pc) : 0.0;
  }
};

// SL terms of wave s's columns into slot[4 (m + 1) + j] (j as the column's
// store; m = 0 without l = 0), the l = 0 pot and dr into slot[0], slot[1].
// Any lmax: the wave's (l, m) pairs in a row, kSplitChunk at a time with
// their table and constant reads first (pairs past the last re-read pair 0;
// a wave past lmax makes one idle round, for rad).
__device__ __forceinline__ void split_sl_terms(const FieldTables& T, const FieldGeom& q,
                                               SplitSL& p, SLRadial& rad, int s, int L, int lane,
                                               double* __restrict__ slot) {
  const SLGeom& g = T.slg;
  const float4* __restrict__ A =
      reinterpret_cast<const float4*>(T.slF) + (size_t)p.cell.i * 2 * sl_npairs(L);
  const double2* __restrict__ ABc = reinterpret_cast<const double2*>(g.lmc + kLmcAB);
  SplitOrder t(q.c1, q.s1);
  SplitColumn u(1.0);
  int k = 0;   // order of t
  int m = s, l = s;
#pragma unroll 1
  do {
    float4 a[kSplitChunk], b[kSplitChunk];
    double2 ab[kSplitChunk];
    int l2 = l, m2 = m;
#pragma unroll
    for (int j = 0; j < kSplitChunk; ++j) {
      const int o = m2 <= L ? sl_pair(l2, m2, L) : 0;
      a[j] = A[2 * o];
      b[j] = A[2 * o + 1];
      ab[j] = ABc[m2 <= L ? sl_pair(l2, m2, kMaxL) : 0];
      const bool end = l2 >= L;
      m2 = uni(end ? split_next_column(m2, s) : m2);
      l2 = uni(end ? m2 : l2 + 1);
    }
    // the weights' reads follow the table's: they are waited for together
    sl_cell_weights(p.cell, g.xi, g.idxi);
    rad = sl_radial(g, p.cell, T.flags);
    const float x2f = (float)p.cell.x2;
#pragma unroll
    for (int j = 0; j < kSplitChunk; ++j)
      if (m <= L) {
        if (l == m) {
          for (; k < m; ++k) t.next(q.c1, p.somx2);
          u = SplitColumn(t.pmm);
        } else {
          u.step(ab[j], p.xs);
        }
        if (l == 0) {
          slot[lane] = (double)fmaf(x2f, a[j].z, a[j].x);
          slot[kSplitPts + lane] = (double)fmaf(rad.ps, b[j].z, b[j].x);
        } else {
          u.term(a[j], b[j], x2f, rad.ps, (double)l, (double)(l + m), p.xc);
        }
        if (l == L) {
          u.store(slot + 4 * (m + 1) * kSplitPts + lane, t, p.good);
          m = uni(split_next_column(m, s));
          l = m;
        } else {
          l = uni(l + 1);
        }
      }
  } while (m <= L);
}

// The same with lmax L and the wave S fixed at compile time: no branch and no
// index arithmetic, about a third of the instructions (a wave here is bound
// by its own instruction stream: one orbit 4.4 -> 2.8 us a step).
template <int L, int S>
__device__ __forceinline__ void split_sl_fixed(const FieldTables& T, const FieldGeom& q,
                                               SplitSL& p, SLRadial& rad, int lane,
                                               double* __restrict__ slot) {
  const SLGeom& g = T.slg;
  constexpr int np = (L + 1) * (L + 2) / 2;
  const float4* __restrict__ A =
      reinterpret_cast<const float4*>(T.slF) + (size_t)(unsigned)p.cell.i * (2 * np);
  const double2* __restrict__ ABc = reinterpret_cast<const double2*>(g.lmc + kLmcAB);
  float4 a[np], b[np];
  double2 ab[np];
#pragma unroll
  for (int m = S; m <= L; m = split_next_column(m, S))
#pragma unroll
    for (int l = m; l <= L; ++l) {
      const int o = sl_pair(l, m, L);
      a[o] = A[2 * o];
      b[o] = A[2 * o + 1];
      ab[o] = ABc[sl_pair(l, m, kMaxL)];
    }
  sl_cell_weights(p.cell, g.xi, g.idxi);
  rad = sl_radial(g, p.cell, T.flags);
  const float x2f = (float)p.cell.x2;
  SplitOrder t(q.c1, q.s1);
  int k = 0;
#pragma unroll
  for (int m = S; m <= L; m = split_next_column(m, S)) {
    for (; k < m; ++k) t.next(q.c1, p.somx2);
    SplitColumn u(t.pmm);
#pragma unroll
    for (int l = m; l <= L; ++l) {
      const int o = sl_pair(l, m, L);
      if (l > m) u.step(ab[o], p.xs);
      if (l == 0) {
        slot[lane] = (double)fmaf(x2f, a[o].z, a[o].x);
        slot[kSplitPts + lane] = (double)fmaf(rad.ps, b[o].z, b[o].x);
      } else {
        u.term(a[o], b[o], x2f, rad.ps, (double)l, (double)(l + m), p.xc);
      }
    }
    u.store(slot + 4 * (m + 1) * kSplitPts + lane, t, p.good);
  }
}

// EOF terms of the orders m = e, e + 4, .. <= M into slot[4 m + j] (j: pot, fr,
// fz, and fp without its factor m).  M, E >= 0: mmax and the wave fixed at
// compile time; E < 0: any.
template <int M, int E>
__device__ __forceinline__ void split_eof_terms(const FieldTables& T, const FieldGeom& q, double z,
                                                int ee, int mm, int lane,
                                                double* __restrict__ slot) {
  const EOFGeom& g = T.eg;
  const int e = E >= 0 ? E : ee, mmax = E >= 0 ? M : mm;
  const EOFCell cell = eof_locate(q.r2, z, g.cmap, g.ascale, g.ihscale, g.xmin, g.idx, g.ymin,
                                  g.idy, g.numx, g.numy);
  const int ns4 = 2 * (mmax + 1), ny1 = g.numy + 1;
  const float4* __restrict__ A =
      reinterpret_cast<const float4*>(T.eofF) + ((size_t)cell.ix * ny1 + cell.iy) * ns4;
  const float4* __restrict__ C = A + (size_t)ny1 * ns4;
  const EOFWeights32 v{(float)cell.c00, (float)cell.c10, (float)cell.c01, (float)cell.c11};
  double cm = 1.0, sm = 0.0, cm1 = q.c1, sm1 = -q.s1;
  int k = 0;
  // two orders' reads in flight together (an order past mmax re-reads the last)
  for (int m0 = e; m0 <= mmax; m0 += 8) {
    const bool two = m0 + 4 <= mmax;
    const int m1 = two ? m0 + 4 : m0;
    float4 a[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int m = h ? m1 : m0;
      a[h][0] = A[2 * m];
      a[h][1] = A[ns4 + 2 * m];
      a[h][2] = C[2 * m];
      a[h][3] = C[ns4 + 2 * m];
      a[h][4] = A[2 * m + 1];
      a[h][5] = A[ns4 + 2 * m + 1];
      a[h][6] = C[2 * m + 1];
      a[h][7] = C[ns4 + 2 * m + 1];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int m = h ? m1 : m0;
      if (h && !two) break;
      double t[4];
      if (m == 0) {
        const EOFCorners0 o = eof_corners0(g, T.eofF, cell, a[0][0], a[0][1], a[0][2], a[0][3]);
        t[0] = eof_bil0(cell, o.a.x, o.c.x, o.b.x, o.e.x);
        t[1] = eof_bil0(cell, o.a.y, o.c.y, o.b.y, o.e.y);
        t[2] = eof_bil0(cell, o.a.z, o.c.z, o.b.z, o.e.z);
        t[3] = 0.0;
      } else {
        for (; k < m; ++k) cheb_next(q.c1, cm, sm, cm1, sm1);
        eof_term(v, a[h][0], a[h][1], a[h][2], a[h][3], a[h][4], a[h][5], a[h][6], a[h][7], cm, sm,
                 t);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) slot[(4 * m + j) * kSplitPts + lane] = t[j];
    }
  }
}

// v0 + the slots of orders 1..last in turn (dphi: each with its factor m).
template <int LAST>
__device__ __forceinline__ double split_sum(const double* __restrict__ o, double v, bool dphi,
                                            int last) {
  if constexpr (LAST >= 0) {
    double u[LAST + 1];
#pragma unroll
    for (int m = 1; m <= LAST; ++m) u[m] = o[4 * m * kSplitPts];
    if (dphi) {
#pragma unroll
      for (int m = 1; m <= LAST; ++m) v = fma((double)m, u[m], v);
    } else {
#pragma unroll
      for (int m = 1; m <= LAST; ++m) v += u[m];
    }
  } else if (dphi) {
    for (int m = 1; m <= last; ++m) v = fma((double)m, o[4 * m * kSplitPts], v);
  } else {
    for (int m = 1; m <= last; ++m) v += o[4 * m * kSplitPts];
  }
  return v;
}

// Fields.return_forces_cart at the point (x, y, z) of lane q of the block
// (the same in all eight waves; every thread calls it, lanes without a point
// with any finite one).  sm: split_lds_doubles(mmax, lmax) doubles of LDS.
// LM, MM: lmax and mmax at compile time, or -1 and any.
// BFE_COMPAT_SL_COS_L is not handled here (split_ok).
template <int LM, int MM>
__device__ __forceinline__ void field_eval_split(const FieldTables& T, double x, double y,
                                                 double z, const SplitWave& w, double* sm,
                                                 double comp[8]) {
  const int mm = MM >= 0 ? MM : uni(T.eg.mmax), ll = LM >= 0 ? LM : uni(T.lmax);
  double* se = sm;
  double* ss = se + 4 * (mm + 1) * kSplitPts;
  double* tot = ss + 4 * (ll + 2) * kSplitPts;
  const int lane = w.lane;
  const FieldGeom q = field_geom(T, x, y, z);
  const bool eof = w.wave < 4;
  const int c = w.wave & 3;   // component the wave sums
  SLRadial rad{0.0, 0.0, 0.f};
  SplitSL p;
  p.xc = 0.0;
  if (eof) {
    if constexpr (MM >= 0) {
      if (c == 0) split_eof_terms<MM, 0>(T, q, z, 0, mm, lane, se);
      else if (c == 1) split_eof_terms<MM, 1>(T, q, z, 1, mm, lane, se);
      else if (c == 2) split_eof_terms<MM, 2>(T, q, z, 2, mm, lane, se);
      else split_eof_terms<MM, 3>(T, q, z, 3, mm, lane, se);
    } else {
      split_eof_terms<-1, -1>(T, q, z, c, mm, lane, se);
    }
  } else {
    p = split_sl_point(T, q);
    if constexpr (LM >= 0) {
      if (c == 0) split_sl_fixed<LM, 0>(T, q, p, rad, lane, ss);
      else if (c == 1) split_sl_fixed<LM, 1>(T, q, p, rad, lane, ss);
      else if (c == 2) split_sl_fixed<LM, 2>(T, q, p, rad, lane, ss);
      else split_sl_fixed<LM, 3>(T, q, p, rad, lane, ss);
    } else {
      split_sl_terms(T, q, p, rad, c, ll, lane, ss);
    }
  }
  __syncthreads();
  // over the orders, in field_eval_point's sequence: EOF m = 0 first for fr
  // and fz, last for the potential
  double v;
  if (eof) {
    const double* o = se + c * kSplitPts + lane;
    const double v0 = o[0];
    v = split_sum<MM>(o, c == 0 ? 0.0 : v0, c == 3, mm);
    if (c == 0) v += v0;
  } else {
    const double* o = ss + (4 + c) * kSplitPts + lane;
    v = split_sum<LM>(o, o[0], c == 3, ll);
    if (c == 0) v = fma(v, rad.P0, ss[lane] * rad.P0);
    else if (c == 1) v = (ss[kSplitPts + lane] + v) * rad.fac;
    else if (c == 2) v = v * (1.0 / (p.xc * p.xc - 1.0)) * rad.P0;
    else v *= rad.P0;
  }
  tot[w.wave * kSplitPts + lane] = v;
  __syncthreads();
  const double dp = tot[lane], dfr = tot[kSplitPts + lane], dfz = tot[2 * kSplitPts + lane];
  const double dfp = tot[3 * kSplitPts + lane], hp = tot[4 * kSplitPts + lane];
  const double hfr = tot[5 * kSplitPts + lane], hft = tot[6 * kSplitPts + lane];
  const double hfp = tot[7 * kSplitPts + lane];
  field_combine(T, q, x, y, z, dfr, dfz, dfp, dp, hfr, hft, hfp, hp, comp);
}

// Whether the split kernels take this field: term slots within the default
// 64 KiB of LDS, and the azimuthal factors per order (not per (l, m)).
inline bool split_ok(const FieldTables& T) {
  return (size_t)split_lds_doubles(T.eg.mmax, T.lmax) * sizeof(double) <= 64 * 1024 &&
         !(T.flags & BFE_COMPAT_SL_COS_L);
}

}  // namespace bfe
