// spx_sph.hpp -- the SPH derivative pass (mixed precision and FP64) and the compatible-energy full
// update.
#pragma once

#include "spx_kernels.hpp"

namespace spx {

// Neighbour record at the midpoint state, image-transformed.
template <int D, typename R>
struct Nbr {
  double x[D], v[D];     // positions and velocities stay double: differences are formed before rounding to R
  R m, rho, cs, h, prho, irho;
};

// A neighbour's midpoint record as loaded (no image transform yet), so the loads of the
// next neighbour can be issued before the current pair is evaluated.
template <int D>
struct NbrRaw {
  double x[D], v[D], m, rho, cs, h, prho, irho;
};
template <int D>
__device__ __forceinline__ void load_raw(const Fields& f, int j, NbrRaw<D>& q) {
  const double2* X = reinterpret_cast<const double2*>(f.xhm) + 2*(size_t)j;
  const double2* P = reinterpret_cast<const double2*>(f.pkm) + 4*(size_t)j;
  const double2 a = X[0], b = X[1], c = P[0], d = P[1], e = P[2], p = P[3];
  q.x[0] = a.x;
  if (D >= 2) q.x[1 % D] = a.y;
  if (D >= 3) q.x[2 % D] = b.x;
  q.h = b.y;
  q.v[0] = c.x;
  if (D >= 2) q.v[1 % D] = c.y;
  if (D >= 3) q.v[2 % D] = d.x;
  q.m = d.y;
  q.rho = e.x;
  q.cs = e.y;
  q.prho = p.x;
  q.irho = p.y;
}
// Image-transformed neighbour record in the pair arithmetic type.
template <int D, typename R>
__device__ __forceinline__ void finish_mid(const Geo& g, int code, const NbrRaw<D>& r, Nbr<D, R>& q) {
#pragma unroll
  for (int a = 0; a < D; ++a) { q.x[a] = r.x[a]; q.v[a] = r.v[a]; }
  if (code) {
    image_pos<D>(g, code, q.x);
#pragma unroll
    for (int a = 0; a < D; ++a) q.v[a] *= refl_sign<D>(g, code, a);
  }
  q.m = (R)r.m;
  q.rho = (R)r.rho;
  q.cs = (R)r.cs;
  q.h = (R)r.h;
  q.prho = (R)r.prho;
  q.irho = (R)r.irho;
}
template <int D, typename R>
__device__ __forceinline__ void load_self(const Fields& f, int i, Nbr<D, R>& s) {
#pragma unroll
  for (int a = 0; a < D; ++a) { s.x[a] = f.xm[a][i]; s.v[a] = f.vm[a][i]; }
  s.m = (R)f.m[i];
  s.rho = (R)f.rhom[i];
  s.cs = (R)f.csm[i];
  s.h = (R)f.hinvm[i];
  s.prho = (R)f.prhom[i];
  s.irho = (R)reinterpret_cast<const double2*>(f.pkm)[4*(size_t)i + 3].y;   // the value partners read
}

// Pair quantities of SPH::evaluateDerivativesImpl (SPH/SPH.cc:362-430) and
// MonaghanGingoldViscosity::QPiij (MonaghanGingoldViscosity.cc:64-100), evaluated
// from the gathering node s toward its neighbour o (r = r_s - r_o).  The canonical
// pair (a, b) of the reference has a = s when aFirst, else a = o.
//
// With isotropic H (H = h^-1 I) each side's kernel gradient H etaUnit dW is parallel to r:
// gradW_s = ks r with ks = (dW_s h_s^-1)(h_s^-1 / |eta_s|), and the Q's tensor is a scalar times
// the identity, so the pairwise acceleration (SPH.cc:428) is one scalar times r:
//   pacc_ab / (-m_b) = C r_ab,   C = ((P_a k_a + P_b k_b) + Q_a k_a / 2) + Q_b k_b / 2
// (P = safeInv(Omega) P / rho^2, Q = the Q's QPi).  C is formed in that canonical order from
// quantities both lanes compute on the same operands (r and the velocity jump change sign exactly),
// so without viscosity both lanes hold the same C bits and each lane's C*r_lane is the exact negation
// of the other's.  The Q's own term is fused the one way and the partner's the other (the results
// programs have had are held to the bit), so an approaching pair's two C differ by FP32 rounding: the
// momentum rate of a Gresho vortex is 2e-9 of the sum of m|a|, of KH 4096 with random velocities 1e-10.
// (FP64 forms C by operations that commute in the two nodes, sph_node64.)  C per neighbour entry is all the
// compatible-energy update needs besides the positions, which it re-forms with the same operations.
//
// Sums whose contraction the compiler may choose are spelled out here, in kernel_wgw_c and in the
// accumulations of sph_node: sph_node4, chosen by the count of active nodes, has the same bits.
template <int D, typename R>
struct PairS {
  R r[D], vso[D], gs[D], es[D];
  R C, Ws, Qs, workQs, vdg, etaMagS, wsphS;
};

// LimitedMonaghanGingoldViscosity's velocity jump dotted with r (LimitedMonaghanGingoldViscosity.cc:
// 160-195): the jump at the pair's midpoint, extrapolated with the nodes' velocity gradients TS, TO
// (row-major D x D, the partner's already image-transformed) scaled by the limiter.
template <int D, typename R>
__device__ __forceinline__ R limited_jump(const Phys& ph, const R* r, const double* vS, const double* vO, R etaS, R etaO,
                                          const R* TS, const R* TO) {
  // van Leer limiter on the ratio of the gradients' projections along the half separation,
  // phased back toward the full Q when the pair is closer than etaCrit
  R xij[D], gi = (R)0, gj = (R)0;
#pragma unroll
  for (int c = 0; c < D; ++c) xij[c] = (R)0.5*r[c];
#pragma unroll
  for (int a = 0; a < D; ++a) {
    R s1 = TS[a*D]*xij[0], s2 = TO[a*D]*xij[0];
#pragma unroll
    for (int b = 1; b < D; ++b) { s1 += TS[a*D + b]*xij[b]; s2 += TO[a*D + b]*xij[b]; }
    gi = a == 0 ? s1*xij[0] : gi + s1*xij[a];
    gj = a == 0 ? s2*xij[0] : gj + s2*xij[a];
  }
  const R tiny30 = sizeof(R) == sizeof(double) ? (R)1.0e-30 : (R)1.0e-30f;
  const R ri = gi/((gj < (R)0 ? (R)-1 : (R)1)*fmax(tiny30, fabs(gj)));
  const R rj = gj/((gi < (R)0 ? (R)-1 : (R)1)*fmax(tiny30, fabs(gi)));
  const R rmin = fmin(ri, rj);
  R phi = rmin > (R)0 ? (R)2/((R)1 + rmin)*(R)2*rmin/((R)1 + rmin) : (R)0;
  const R etaij = fmin(etaS, etaO), ec = (R)ph.etaCrit;
  if (etaij < ec) { const R q = (etaij - ec)/(R)ph.etaFold; phi *= exp(-(q*q)); }
  // (phi*T).xij: the product with the scaled tensor, as the reference forms it
  R vqr = (R)0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    R s1 = (phi*TS[a*D])*xij[0], s2 = (phi*TO[a*D])*xij[0];
#pragma unroll
    for (int b = 1; b < D; ++b) { s1 += (phi*TS[a*D + b])*xij[b]; s2 += (phi*TO[a*D + b])*xij[b]; }
    const R vq = (R)((vS[a] - (double)s1) - (vO[a] + (double)s2));
    vqr += vq*r[a];
  }
  return vqr;
}

// coef: the kernel table's coefficients in arithmetic R (global, or the block's LDS copy).
// LQ: LimitedMonaghanGingoldViscosity::QPiij (LimitedMonaghanGingoldViscosity.cc:160-195) in
// place of the plain Q; TS, TO are the two nodes' velocity gradients as the Q holds them
// (row-major D x D, the partner's already image-transformed).
template <int D, typename R, bool LQ = false, typename CP>
__device__ __forceinline__ void pair_eval(const DevTable& tab, CP coef, const Phys& ph, const Nbr<D, R>& S,
                                          const Nbr<D, R>& O, bool aFirst, PairS<D, R>& e,
                                          const R* TS = nullptr, const R* TO = nullptr) {
  R eo[D];
#pragma unroll
  for (int c = 0; c < D; ++c) {
    e.r[c] = (R)(S.x[c] - O.x[c]);
    e.es[c] = S.h*e.r[c];
    eo[c] = O.h*e.r[c];
    e.vso[c] = (R)(S.v[c] - O.v[c]);
  }
  const R e2s = norm2<D>(e.es), e2o = norm2<D>(eo);
  // |eta| and safeInvVar(|eta|) = 1/max(1e-30, |eta|) from one reciprocal square root each
  const R tiny = (R)1.0e-30f;
  const R is = e2s > tiny*tiny ? rsqrt(e2s) : (R)1/tiny, io = e2o > tiny*tiny ? rsqrt(e2o) : (R)1/tiny;
  e.etaMagS = e2s*is;
  const R etaMagO = e2o*io;
  R gws, gwo, graws, grawo, Wo;
  kernel_wgw_c<R>(coef, tab, e.etaMagS, hdet_iso<D, R>(S.h), e.Ws, gws, graws);
  kernel_wgw_c<R>(coef, tab, etaMagO, hdet_iso<D, R>(O.h), Wo, gwo, grawo);
  e.wsphS = fabs(graws);                                      // kernelValueSPH(etaMagS)
  const R ks = (gws*S.h)*(S.h*is), ko = (gwo*O.h)*(O.h*io);  // gradW = k r
  R vsr = (R)0;
#pragma unroll
  for (int c = 0; c < D; ++c) {
    e.gs[c] = ks*e.r[c];
    vsr = fused(e.vso[c], e.r[c], vsr);
  }
  // velocity jump the Q sees: the plain difference, or the limited midpoint extrapolation
  R vqr = vsr;
  if (LQ) {
    vqr = limited_jump<D, R>(ph, e.r, S.v, O.v, e.etaMagS, etaMagO, TS, TO);
  }
  // mu = (vq . eta)/(eta^2 + eps^2) with eta = h^-1 r on each side
  const R mus = (S.h*vqr)/(e2s + (R)1.0e-2), muo = (O.h*vqr)/(e2o + (R)1.0e-2);
  const R mms = fmin((R)0, mus), mmo = fmin((R)0, muo);
  const R Cl = (R)ph.Cl, Cq = (R)ph.Cq;
  const R es_ = fused(-Cl*S.cs, mms, Cq*(mms*mms));
  const R eo_ = fused(Cq, mmo*mmo, -(Cl*O.cs*mmo));
  const R QPs = es_*S.irho, QPo = eo_*O.irho;
  e.Qs = S.rho*es_;
  const R p1 = aFirst ? S.prho : O.prho, p2 = aFirst ? O.prho : S.prho;
  const R k1 = aFirst ? ks : ko, k2 = aFirst ? ko : ks;
  const R q1 = aFirst ? QPs : QPo, q2 = aFirst ? QPo : QPs;
  e.C = fused((R)0.5, q2*k2, fused((R)0.5, q1*k1, fused(p1, k1, p2*k2)));
  e.vdg = ks*vsr;                                            // v_so . gradW_s
  e.workQs = (R)0.5*(QPs*e.vdg);                             // v_so . (QPi_s gradW_s / 2)
}

// ---------------------------------------------------------------------------
// SPH::evaluateDerivatives + SPHSmoothingScale::evaluateDerivatives on the midpoint
// state (SPH/SPH.cc:271-551, SmoothingScale/SPHSmoothingScale.cc:154-245), gather form.
// FULL also produces the outputs the integration does not consume (sum density,
// normalisation, effective Q, density gradient, first moment, M).
// ---------------------------------------------------------------------------
// ldsTable != 0: the table's coefficients are staged in the block's dynamic LDS first (the
// pair loop makes three lookups per pair at scattered intervals).  sc != nullptr (the step):
// the node's half-step velocity record for the compatible-energy update is written too (as
// k_v12 would, with the run's dt/2).

// A node's sums over its pairs.
template <int D>
struct SphSums {
  double dvdt[D], dvdx[D*D], M[D*D], depsdt, maxq, m0;
  double rhosum, nrm, effq, grho[D], m1[D];              // FULL
};

// The node's derivatives and ideal H from its sums (SPH.cc:480-551, SPHSmoothingScale.cc:228-245),
// double precision, and its partition record.
template <int D, bool FULL>
__device__ __forceinline__ void sph_finalize(const Fields& f, const Phys& ph, const DevTable& tab, int i, int nn,
                                             SphSums<D>& q, const Scalars* sc) {
  const size_t ld = (size_t)f.ld;
  const double Sm = f.m[i], Srho = f.rhom[i], Sh = f.hinvm[i];
  const double hdet = hdet_iso<D>(Sh);
  double det;
  if (D == 1) det = q.M[0];
  else if (D == 2) det = q.M[0]*q.M[3] - q.M[1]*q.M[2];
  else det = (q.M[0]*q.M[4]*q.M[8] + q.M[1]*q.M[5]*q.M[6] + q.M[2]*q.M[3]*q.M[7] -
              q.M[0]*q.M[5]*q.M[7] - q.M[1]*q.M[3]*q.M[8] - q.M[2]*q.M[4]*q.M[6]);
  const double pow2d = D == 1 ? 2.0 : (D == 2 ? 4.0 : 8.0);
  double G[D*D];
  if (ph.correctVG && fabs(det) > 1.0e-10 && (double)nn > pow2d) {
    double Mi[D*D];
    if (D == 1) {
      Mi[0] = 1.0/q.M[0];
    } else if (D == 2) {
      const double r = 1.0/det;
      Mi[0] = q.M[3]*r; Mi[1] = -q.M[1]*r; Mi[2] = -q.M[2]*r; Mi[3] = q.M[0]*r;
    } else {
      const double r = 1.0/det;
      const double xx = q.M[0], xy = q.M[1], xz = q.M[2], yx = q.M[3], yy = q.M[4], yz = q.M[5], zx = q.M[6], zy = q.M[7], zz = q.M[8];
      Mi[0] = (yy*zz - yz*zy)*r; Mi[1] = (xz*zy - xy*zz)*r; Mi[2] = (xy*yz - xz*yy)*r;
      Mi[3] = (yz*zx - yx*zz)*r; Mi[4] = (xx*zz - xz*zx)*r; Mi[5] = (xz*yx - xx*yz)*r;
      Mi[6] = (yx*zy - yy*zx)*r; Mi[7] = (xy*zx - xx*zy)*r; Mi[8] = (xx*yy - xy*yx)*r;
    }
#pragma unroll
    for (int a = 0; a < D; ++a)
#pragma unroll
      for (int b = 0; b < D; ++b) {
        double s = 0.0;
#pragma unroll
        for (int k2 = 0; k2 < D; ++k2) s += q.dvdx[a*D + k2]*Mi[k2*D + b];
        G[a*D + b] = s;
      }
    if (FULL) {
#pragma unroll
      for (int a = 0; a < D*D; ++a) q.M[a] = Mi[a];
    }
  } else {
#pragma unroll
    for (int a = 0; a < D*D; ++a) G[a] = rdiv<D>(q.dvdx[a], Srho);
  }
  double tr = 0.0;
#pragma unroll
  for (int a = 0; a < D; ++a) tr += G[a*D + a];
#pragma unroll
  for (int a = 0; a < D*D; ++a) f.DvDx[a*ld + i] = G[a];
#pragma unroll
  for (int a = 0; a < D; ++a) { f.DvDt[a][i] = q.dvdt[a]; f.DxDt[a][i] = f.vm[a][i]; }
  f.DepsDt[i] = q.depsdt;
  {
    // the partition record: this evaluation's positions (the pair coefficients' r) always; the
    // half-step velocities and DepsDt in the step (otherwise k_v12 writes them)
    double2* PV = reinterpret_cast<double2*>(f.pkv) + 4*(size_t)i;
    double xs[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < D; ++a) xs[a] = f.xm[a][i];
    if (sc) {
      const double hdt = 0.5*sc[f.run[i]].dt;
      double w[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int a = 0; a < D; ++a) w[a] = f.v[a][i] + q.dvdt[a]*hdt;
      PV[0] = make_double2(w[0], w[1]);
      PV[1] = make_double2(w[2], q.depsdt);
    }
    PV[2] = make_double2(Sm, xs[0]);
    PV[3] = make_double2(xs[1], xs[2]);
  }
  f.DrhoDt[i] = -Srho*tr;
  f.maxQ[i] = q.maxq;
  // ---- SPHSmoothingScale finalize (SPHSmoothingScale.cc:228-245)
  const double m0 = rootnu<D>(fmax(0.0, q.m0));
  f.m0[i] = m0;
  f.DHDt[i] = rdiv<D>(-Sh, double(D))*tr;
  const double cur = (fabs(m0) <= 1.0e-15*fmax(1.0, fabs(m0))) ? 0.5*ph.nperh : nperh_lookup(tab, m0);
  const double s = fmin(4.0, fmax(0.25, ph.nperh/(cur + 1.0e-30)));
  const double aa = s < 1.0 ? 0.4*(1.0 + s*s) : 0.4*(1.0 + 1.0/(s*s*s));
  const double hi0 = 1.0/Sh;
  const double hi1 = fmin(ph.hmax, fmax(ph.hmin, hi0*(1.0 - aa + aa*s)));
  f.Hideal[i] = 1.0/hi1;
  if (FULL) {
    f.rhoSum[i] = q.rhosum + Sm*tab.W0*hdet;
    f.norm[i] = q.nrm + Sm/Srho*tab.W0*hdet;
    f.effQ[i] = q.effq;
#pragma unroll
    for (int c = 0; c < D; ++c) { f.gradRho[c][i] = rdiv<D>(q.grho[c], Srho); f.m1[c][i] = q.m1[c]; }
#pragma unroll
    for (int a = 0; a < D*D; ++a) f.Mcorr[a*ld + i] = q.M[a];
  }
}

template <int D, bool FULL, bool LQ, typename CP>
__device__ __forceinline__ void sph_node(const Fields& f, const Geo& g, const Phys& ph, const DevTable& tab,
                                         CP coef, int n, const Scalars* sc) {
  using R = float;
  constexpr int L = 2;
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int i = gl >> 1, sub = gl & 1;
  // both lanes of a pair share i: they leave together
  if (i >= n) return;
  const size_t ld = (size_t)f.ld;
  R* pdd = (R*)f.pdd;
  Nbr<D, R> S;
  load_self<D, R>(f, i, S);
  const double Sm = f.m[i], Srho = f.rhom[i], Sh = f.hinvm[i];

  double dvdt[D], dvdx[D*D], Mc[D*D], depsdt = 0.0, m0 = 0.0;
  R maxqr = (R)0;
  double rhosum = 0.0, nrm = 0.0, effq = 0.0, grho[D], m1[D];
#pragma unroll
  for (int a = 0; a < D; ++a) { dvdt[a] = 0.0; grho[a] = 0.0; m1[a] = 0.0; }
#pragma unroll
  for (int a = 0; a < D*D; ++a) { dvdx[a] = 0.0; Mc[a] = 0.0; }

  R TS[LQ ? D*D : 1];
  if (LQ) {
#pragma unroll
    for (int a = 0; a < D*D; ++a) TS[a] = (R)f.DvDxQ[a*ld + i];
  }
  const int nn = f.cnt[i];
  // A neighbour's record is fetched one pair ahead, and its ELL entry two: the record's address is
  // at hand when its turn comes, instead of a wait for the entry (and all before it) in every pair.
  uint32_t en = 0, en2 = 0;
  NbrRaw<D> rn;
  if (sub < nn) {
    en = f.nbr[ell_at(sub, i, ld)];
    if (sub + L < nn) en2 = f.nbr[ell_at(sub + L, i, ld)];
    load_raw<D>(f, (int)(en & kIdxMask), rn);
  }
  for (int k = sub; k < nn; k += L) {
    const uint32_t ent = en;
    const NbrRaw<D> rc = rn;
    en = en2;
    if (k + 2*L < nn) en2 = f.nbr[ell_at(k + 2*L, i, ld)];
    if (k + L < nn) load_raw<D>(f, (int)(en & kIdxMask), rn);
    const int j = (int)(ent & kIdxMask);
    const int code = (int)(ent >> kImgShift);
    Nbr<D, R> O;
    finish_mid<D, R>(g, code, rc, O);
    PairS<D, R> e;
    if (LQ) {
      // the partner's gradient: ghosts carry the tensor image (reflected axes flip sign per
      // index) when boundaries were applied after the Q's copy; otherwise the zero the cycle's
      // ghost rebuild left (ArtificialViscosityHandle.cc:168-183, Integrator.cc:254-271)
      R TO[D*D];
      const bool img = code != 0;
#pragma unroll
      for (int a = 0; a < D; ++a)
#pragma unroll
        for (int b = 0; b < D; ++b) {
          const double t = f.DvDxQ[(size_t)(a*D + b)*ld + j];
          TO[a*D + b] = img ? (ph.qImages ? (R)(refl_sign<D>(g, code, a)*refl_sign<D>(g, code, b)*t) : (R)0) : (R)t;
        }
      pair_eval<D, R, true>(tab, coef, ph, S, O, code != 0 || i < j, e, TS, TO);
    } else {
      pair_eval<D, R>(tab, coef, ph, S, O, code != 0 || i < j, e);
    }
    pdd[(size_t)k*ld + i] = e.C;
    const double mo = rc.m;
#pragma unroll
    for (int c = 0; c < D; ++c) {
      dvdt[c] = fused(-mo, (double)(e.C*e.r[c]), dvdt[c]);
      const double mv = mo*(double)e.vso[c], mr = mo*(double)e.r[c];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        dvdx[c*D + d] = fused(-mv, (double)e.gs[d], dvdx[c*D + d]);
        // (the FP32 pair terms round r_c g_d and r_d g_c differently: all of M is accumulated)
        Mc[c*D + d] = fused(-mr, (double)e.gs[d], Mc[c*D + d]);
      }
    }
    depsdt = fused(mo, (double)fused(S.prho, e.vdg, e.workQs), depsdt);
    maxqr = fmax(maxqr, e.Qs);
    const R wsph = e.wsphS;
    m0 += (double)wsph;
    if (FULL) {
      const double orho = rc.rho;
      rhosum += mo*(double)e.Ws;
      nrm += Sm/Srho*(double)e.Ws;
      effq += mo*(double)e.Qs*(double)e.Ws/orho;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        grho[c] += mo*(orho - Srho)*(double)e.gs[c];
        m1[c] -= (double)(wsph*e.es[c]);
      }
    }
  }

  double maxq = (double)maxqr;
  {
    // the pair's partial sums: each lane forms (own + partner's), the same bits on both
#pragma unroll
    for (int a = 0; a < D; ++a) dvdt[a] += quad_swap<0xB1>(dvdt[a]);
#pragma unroll
    for (int c = 0; c < D; ++c)
#pragma unroll
      for (int d = 0; d < D; ++d) {
        dvdx[c*D + d] += quad_swap<0xB1>(dvdx[c*D + d]);
        Mc[c*D + d] += quad_swap<0xB1>(Mc[c*D + d]);
      }
    depsdt += quad_swap<0xB1>(depsdt);
    m0 += quad_swap<0xB1>(m0);
    maxq = fmax(maxq, quad_swap<0xB1>(maxq));
    if (FULL) {
      rhosum += quad_swap<0xB1>(rhosum);
      nrm += quad_swap<0xB1>(nrm);
      effq += quad_swap<0xB1>(effq);
#pragma unroll
      for (int a = 0; a < D; ++a) { grho[a] += quad_swap<0xB1>(grho[a]); m1[a] += quad_swap<0xB1>(m1[a]); }
    }
    if (sub != 0) return;
  }
  SphSums<D> q;
#pragma unroll
  for (int a = 0; a < D; ++a) { q.dvdt[a] = dvdt[a]; q.grho[a] = grho[a]; q.m1[a] = m1[a]; }
#pragma unroll
  for (int a = 0; a < D*D; ++a) { q.dvdx[a] = dvdx[a]; q.M[a] = Mc[a]; }
  q.depsdt = depsdt; q.maxq = maxq; q.m0 = m0;
  q.rhosum = rhosum; q.nrm = nrm; q.effq = effq;
  sph_finalize<D, FULL>(f, ph, tab, i, nn, q, sc);
}

// ---------------------------------------------------------------------------
// The FP64 pass: L lanes per node, each over the entries k = sub, sub + L, ...; the lanes' sums are
// joined by DPP and left in LDS, and the block's first threads finalize its nodes.
//
// Everything both sides of a pair must agree on (C and what it is made of) is formed from r^2, the
// two supports and the two records by operations that commute in the two nodes, each rounded as
// written (no contraction the compiler could choose differently on the two sides): t_x = k_x (P_x +
// Q_x/2), C = t_s + t_o has the same bits in both lanes, so C r is exactly antisymmetric without
// selecting a canonical order.  An image partner's position is rounded on each side by itself, as
// the reference's ghost is.
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ double h_power(double h) {   // h^(D + 1): k = dW/deta h^(D + 1) / |r|
  if (D == 1) return rounded_product(h, h);
  if (D == 2) return rounded_product(rounded_product(h, h), h);
  const double h2 = rounded_product(h, h);
  return rounded_product(h2, h2);
}
// A node's viscous term rho^-1 Q (before the division by rho^2's other half): Cq mu^2 - Cl cs mu.
__device__ __forceinline__ double mg_term(const Phys& ph, double clcs, double mu) {
  return rounded_product(mu, fused(ph.Cq, mu, -clcs));
}

// Sums of a node: DvDt, DvDx, M's upper triangle, DepsDt, the zeroth moment, the largest Q; with FULL
// also the sum density, normalisation, effective Q, density gradient and first moment.
constexpr int sph_sums(int D, bool full) { return D + D*D + D*(D + 1)/2 + 3 + (full ? 3 + 2*D : 0); }
template <int D, bool FULL, bool LQ, int L, typename CP>
__device__ __forceinline__ void sph_node64(const Fields& f, const Geo& g, const Phys& ph, const DevTable& tab, CP coef,
                                           int n, const Scalars* sc, double (&sums)[sph_sums(D, FULL)][kBlock/L]) {
  constexpr int NB = kBlock/L;
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int i = gl/L, sub = gl & (L - 1);
  const size_t ld = (size_t)f.ld;
  double* pdd = (double*)f.pdd;
  double dvdt[D], dvdx[D*D], M[D*D], depsdt = 0.0, maxe = 0.0, m0 = 0.0;
  double rhosum = 0.0, nrm = 0.0, effq = 0.0, grho[D], m1[D];
#pragma unroll
  for (int a = 0; a < D; ++a) { dvdt[a] = 0.0; grho[a] = 0.0; m1[a] = 0.0; }
#pragma unroll
  for (int a = 0; a < D*D; ++a) { dvdx[a] = 0.0; M[a] = 0.0; }
  double Srho = 0.0;
  if (i < n) {
    NbrRaw<D> S;
    load_raw<D>(f, i, S);
    Srho = S.rho;
    const double SA = h_power<D>(S.h), Sclcs = rounded_product(ph.Cl, S.cs);
    double TS[LQ ? D*D : 1];
    if (LQ) {
#pragma unroll
      for (int a = 0; a < D*D; ++a) TS[a] = f.DvDxQ[a*ld + i];
    }
    const int nn = f.cnt[i];
    // the neighbour's record is fetched one pair ahead, its entry two (sph_node)
    uint32_t en = 0, en2 = 0;
    NbrRaw<D> rn;
    if (sub < nn) {
      en = f.nbr[ell_at(sub, i, ld)];
      if (sub + L < nn) en2 = f.nbr[ell_at(sub + L, i, ld)];
      load_raw<D>(f, (int)(en & kIdxMask), rn);
    }
    for (int k = sub; k < nn; k += L) {
      const uint32_t ent = en;
      NbrRaw<D> O = rn;
      en = en2;
      if (k + 2*L < nn) en2 = f.nbr[ell_at(k + 2*L, i, ld)];
      if (k + L < nn) load_raw<D>(f, (int)(en & kIdxMask), rn);
      const int code = (int)(ent >> kImgShift);
      if (code) {
        image_pos<D>(g, code, O.x);
#pragma unroll
        for (int c = 0; c < D; ++c) O.v[c] *= refl_sign<D>(g, code, c);
      }
      double r[D], dv[D];
#pragma unroll
      for (int c = 0; c < D; ++c) { r[c] = S.x[c] - O.x[c]; dv[c] = S.v[c] - O.v[c]; }
      const double r2 = norm2<D>(r);
      const double rinv = r2 > 1.0e-290 ? fast_rsqrt(r2) : 0.0;
      const double d = rounded_product(r2, rinv);
      const double etas = rounded_product(S.h, d), etao = rounded_product(O.h, d);
      double grs, gro, Ws = 0.0;
      if (FULL) {
        double gw;
        kernel_wgw_c<double>(coef, tab, etas, hdet_iso<D, double>(S.h), Ws, gw, grs);
        gro = kernel_graw<6, double>(coef + 3, tab, etao);
      } else {
        grs = kernel_graw<3, double>(coef, tab, etas);
        gro = kernel_graw<3, double>(coef, tab, etao);
      }
      const double ks = rounded_product(rounded_product(grs, SA), rinv);             // gradW = k r
      const double ko = rounded_product(rounded_product(gro, h_power<D>(O.h)), rinv);
      double vsr = rounded_product(dv[0], r[0]);
#pragma unroll
      for (int c = 1; c < D; ++c) vsr = fused(dv[c], r[c], vsr);
      double vqr = vsr;
      if (LQ) {
        // the limited velocity jump (pair_eval's, FP64)
        const int j = (int)(ent & kIdxMask);
        double TO[D*D];
#pragma unroll
        for (int a = 0; a < D; ++a)
#pragma unroll
          for (int b = 0; b < D; ++b) {
            const double t = f.DvDxQ[(size_t)(a*D + b)*ld + j];
            TO[a*D + b] = code ? (ph.qImages ? refl_sign<D>(g, code, a)*refl_sign<D>(g, code, b)*t : 0.0) : t;
          }
        vqr = limited_jump<D, double>(ph, r, S.v, O.v, etas, etao, TS, TO);
      }
      // mu = (vq . eta)/(eta^2 + eps^2) on each side, one reciprocal for both
      const double ps = fused(etas, etas, 1.0e-2), po = fused(etao, etao, 1.0e-2);
      const double inv = fast_rcp(rounded_product(ps, po));
      const double mus = rounded_product(rounded_product(S.h, vqr), rounded_product(inv, po));
      const double muo = rounded_product(rounded_product(O.h, vqr), rounded_product(inv, ps));
      const double es = mg_term(ph, Sclcs, fmin(0.0, mus));
      const double eo = mg_term(ph, rounded_product(ph.Cl, O.cs), fmin(0.0, muo));
      const double us = fused(0.5, rounded_product(es, S.irho), S.prho);
      const double uo = fused(0.5, rounded_product(eo, O.irho), O.prho);
      const double C = rounded_product(ks, us) + rounded_product(ko, uo);
      pdd[(size_t)k*ld + i] = C;
      const double mC = O.m*C, w = O.m*ks;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        dvdt[c] -= mC*r[c];
        const double wr = w*r[c];
#pragma unroll
        for (int b = 0; b < D; ++b) {
          dvdx[b*D + c] -= dv[b]*wr;
          // with isotropic H the gradient is parallel to r: M = sum m r (x) gradW is symmetric and
          // only its upper triangle is summed
          if (b <= c) M[b*D + c] -= r[b]*wr;
        }
      }
      depsdt += w*vsr*us;
      maxe = fmax(maxe, es);
      m0 += fabs(grs);
      if (FULL) {
        rhosum += O.m*Ws;
        nrm += S.m/S.rho*Ws;
        effq += O.m*(S.rho*es)*Ws/O.rho;
#pragma unroll
        for (int c = 0; c < D; ++c) {
          grho[c] += O.m*(O.rho - S.rho)*(ks*r[c]);
          m1[c] -= fabs(grs)*(S.h*r[c]);
        }
      }
    }
  }
  auto join = [&](double v) {
    if (L >= 2) v += quad_swap<0xB1>(v);
    if (L >= 4) v += quad_swap<0x4E>(v);
    return v;
  };
  const int slot = threadIdx.x/L;
  int q = 0;
  auto put = [&](double v) {
    v = join(v);
    if (sub == 0) sums[q][slot] = v;
    ++q;
  };
#pragma unroll
  for (int a = 0; a < D; ++a) put(dvdt[a]);
#pragma unroll
  for (int a = 0; a < D*D; ++a) put(dvdx[a]);
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int b = a; b < D; ++b) put(M[a*D + b]);
  put(depsdt);
  put(m0);
  {
    double e = maxe;
    if (L >= 2) e = fmax(e, quad_swap<0xB1>(e));
    if (L >= 4) e = fmax(e, quad_swap<0x4E>(e));
    if (sub == 0) sums[q][slot] = Srho*e;                // the largest rho^2 Q of the node
    ++q;
  }
  if (FULL) {
    put(rhosum);
    put(nrm);
    put(effq);
#pragma unroll
    for (int a = 0; a < D; ++a) { put(grho[a]); put(m1[a]); }
  }
  __syncthreads();
  if ((int)threadIdx.x >= NB) return;
  const int j = xcd_block()*NB + threadIdx.x;
  if (j >= n) return;
  SphSums<D> t;
  q = 0;
  auto get = [&] { return sums[q++][threadIdx.x]; };
#pragma unroll
  for (int a = 0; a < D; ++a) t.dvdt[a] = get();
#pragma unroll
  for (int a = 0; a < D*D; ++a) t.dvdx[a] = get();
#pragma unroll
  for (int a = 0; a < D; ++a)
#pragma unroll
    for (int b = a; b < D; ++b) t.M[a*D + b] = t.M[b*D + a] = get();
  t.depsdt = get();
  t.m0 = get();
  t.maxq = get();
  if (FULL) {
    t.rhosum = get();
    t.nrm = get();
    t.effq = get();
#pragma unroll
    for (int a = 0; a < D; ++a) { t.grho[a] = get(); t.m1[a] = get(); }
  }
  sph_finalize<D, FULL>(f, ph, tab, j, f.cnt[j], t, sc);
}

// The mixed-precision pass of a step on four lanes per node, with the two-lane pass's bits (above):
// lanes 0 and 2 form the pairs k = 0, 4, .. and 2, 6, .., lanes 1 and 3 the odd ones, and the sums
// of the even and of the odd pairs are accumulated in order of k.  To that end each of the two lanes
// of a parity adds both lanes' terms, but only to half of the sums: the lower to DvDx and DvDt, the
// upper to M, DepsDt and the zeroth moment.  The pairs' values pass by DPP, 32 exchanges and 12
// selects per pair; twice the lanes per node halve a node's chain of pairs, which is what a small
// run waits for.
template <int D, typename CP>
__device__ __forceinline__ void sph_node4(const Fields& f, const Geo& g, const Phys& ph, const DevTable& tab, CP coef,
                                          int n, const Scalars* sc) {
  using R = float;
  constexpr int L = 4, LOW = 0x44, UP = 0xEE;       // quad_perm [0,1,0,1] and [2,3,2,3]
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int i = gl >> 2, sub = gl & 3;
  if (i >= n) return;
  const bool upper = sub >= 2;
  const size_t ld = (size_t)f.ld;
  R* pdd = (R*)f.pdd;
  Nbr<D, R> S;
  load_self<D, R>(f, i, S);
  double acc[D*D], ext[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int a = 0; a < D*D; ++a) acc[a] = 0.0;
  R maxqr = (R)0;
  const int nn = f.cnt[i];
  uint32_t en = 0, en2 = 0;
  NbrRaw<D> rn;
  if (sub < nn) {
    en = f.nbr[ell_at(sub, i, ld)];
    if (sub + L < nn) en2 = f.nbr[ell_at(sub + L, i, ld)];
    load_raw<D>(f, (int)(en & kIdxMask), rn);
  }
  for (int k = sub; k - sub < nn; k += L) {
    const uint32_t ent = en;
    const NbrRaw<D> rc = rn;
    en = en2;
    if (k + 2*L < nn) en2 = f.nbr[ell_at(k + 2*L, i, ld)];
    if (k + L < nn) load_raw<D>(f, (int)(en & kIdxMask), rn);
    double mo = 0.0;
    R vso[D], r[D], gs[D], cr[D], dep = (R)0, wsph = (R)0;
#pragma unroll
    for (int c = 0; c < D; ++c) vso[c] = r[c] = gs[c] = cr[c] = (R)0;
    if (k < nn) {
      const int j = (int)(ent & kIdxMask), code = (int)(ent >> kImgShift);
      Nbr<D, R> O;
      finish_mid<D, R>(g, code, rc, O);
      PairS<D, R> e;
      pair_eval<D, R>(tab, coef, ph, S, O, code != 0 || i < j, e);
      pdd[(size_t)k*ld + i] = e.C;
      mo = rc.m;
#pragma unroll
      for (int c = 0; c < D; ++c) { vso[c] = e.vso[c]; r[c] = e.r[c]; gs[c] = e.gs[c]; cr[c] = rounded_product(e.C, e.r[c]); }
      dep = fused(S.prho, e.vdg, e.workQs);
      wsph = e.wsphS;
      maxqr = fmax(maxqr, e.Qs);
    }
    auto add = [&](auto from) {
      const double m = quad_swap<from>(mo);
      double gd[D];
#pragma unroll
      for (int c = 0; c < D; ++c) gd[c] = (double)quad_swap<from>(gs[c]);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        const R v = quad_swap<from>(vso[c]), x = quad_swap<from>(r[c]);
        const double w = rounded_product(m, (double)(upper ? x : v));
#pragma unroll
        for (int d = 0; d < D; ++d) acc[c*D + d] = fused(-w, gd[d], acc[c*D + d]);
      }
      // lower: DvDt -= m C r; upper: DepsDt += m dep, m0 += wsph
      const R de = quad_swap<from>(dep), ws = quad_swap<from>(wsph);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        const R q = quad_swap<from>(cr[c]);
        if (c == 0) ext[0] = fused(-m, (double)(upper ? -de : q), ext[0]);
        else if (c == 1) ext[1] = fused(upper ? -1.0 : -m, (double)(upper ? -ws : q), ext[1]);
        else ext[2] = fused(-m, (double)q, ext[2]);
      }
      if (D == 1) ext[1] = fused(-1.0, (double)(upper ? -ws : (R)0), ext[1]);
    };
    add(std::integral_constant<int, LOW>{});
    add(std::integral_constant<int, UP>{});
  }
  // even + odd, then the upper lanes' half to the lower ones
  double maxq = (double)maxqr;
  maxq = fmax(maxq, quad_swap<0xB1>(maxq));
  maxq = fmax(maxq, quad_swap<0x4E>(maxq));
  SphSums<D> q;
#pragma unroll
  for (int a = 0; a < D*D; ++a) {
    acc[a] += quad_swap<0xB1>(acc[a]);
    q.dvdx[a] = acc[a];
    q.M[a] = quad_swap<0x4E>(acc[a]);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) ext[a] += quad_swap<0xB1>(ext[a]);
  q.depsdt = quad_swap<0x4E>(ext[0]);
  q.m0 = quad_swap<0x4E>(ext[1]);
  if (sub != 0) return;
#pragma unroll
  for (int a = 0; a < D; ++a) { q.dvdt[a] = ext[a]; q.grho[a] = 0.0; q.m1[a] = 0.0; }
  q.maxq = maxq;
  q.rhosum = q.nrm = q.effq = 0.0;
  sph_finalize<D, false>(f, ph, tab, i, nn, q, sc);
}

// Lanes per node of the SPH pass.  The choice depends only on the configuration (dimension,
// precision), so a run gives the same bits in any batch; k_sph_wide, which a mixed-precision step takes
// by the particle count, has the two-lane pass's bits.  FP64, us per
// pass with 1 / 2 / 4 lanes: Sod 1-D 400 9.2 / 7.5 / 6.5, Noh 1-D 100 14.3 / 10.4 / 7.8, KH 2-D 65536
// 71.9 / 46.7 / 41.5, Taylor-Green 37^3 56.4 / 39.8 / 41.8, 128^3 1451 / 1309 / 1385; with the list
// entries read two pairs ahead 6.3, 7.5, 40.2, 37.7 and 1269 (before, with two
// sides' divisions, two reciprocal square roots and canonical-order selects per pair: 8.0, 10.6,
// 53.8, 64 and 1406).  On large 3-D runs the pass is bound by the records' gathers: 96 bytes per
// neighbour, 9 GB through the L1s of which most misses them.
template <int D>
constexpr int kSphLanes64 = D == 3 ? 2 : 4;
constexpr int kSphLanesMixed = 2;
template <int D>
__global__ void __launch_bounds__(kBlock, 3) k_sph_wide(Fields f, Geo g, Phys ph, DevTable tab, int n, int ldsTable,
                                                        const Scalars* sc) {
  with_table<float>(tab, ldsTable, [&](auto coef) { sph_node4<D>(f, g, ph, tab, coef, n, sc); });
}
// Wavefronts per SIMD that a variant's registers are cut for: three (168 VGPRs), or two where three
// spill and two measured faster.  Three / two: evaluate_derivatives with the Limited Q, Taylor-Green
// 48^3 mixed 449 / 231 us, FP64 679 / 218, 96^3 2540 / 1450 and 4810 / 1380, without it 713 / 659
// and 801 / 764, KH 65536 FP64 with it 143 / 119; the step's 3-D FP64 pass with it 48^3 414 / 160,
// 96^3 2540 / 1145.  The step's other variants with the Limited Q (2-D FP64: 8 spilled, 3-D mixed:
// 38) stay at three: KH 262144 190 / 196, Taylor-Green 96^3 1135 / 1334.
constexpr int sph_waves(int D, bool full, bool fp64, bool lq) {
  return (D == 3 && (full || (fp64 && lq))) || (D == 2 && full && fp64 && lq) ? 2 : 3;
}
template <int D, bool FULL, typename R, bool LQ = false>
__global__ void __launch_bounds__(kBlock, (sph_waves(D, FULL, sizeof(R) == sizeof(double), LQ))) k_sph(Fields f, Geo g, Phys ph, DevTable tab, int n, int ldsTable,
                                                   const Scalars* sc) {
  if constexpr (sizeof(R) == sizeof(float)) {
    with_table<float>(tab, ldsTable, [&](auto coef) { sph_node<D, FULL, LQ>(f, g, ph, tab, coef, n, sc); });
  } else {
    __shared__ double sums[sph_sums(D, FULL)][kBlock/kSphLanes64<D>];
    auto body = [&](auto coef) { sph_node64<D, FULL, LQ, kSphLanes64<D>>(f, g, ph, tab, coef, n, sc, sums); };
    if constexpr (FULL) with_table<double>(tab, ldsTable, body);
    else with_gradient_table(tab, ldsTable, body);
  }
}

// ---------------------------------------------------------------------------
// SpecificThermalEnergyPolicy::update's partition of the pair work (Hydro/
// SpecificThermalEnergyPolicy.cc:79-144): node i's specific thermal energy rate from the pair
// coefficients C the SPH pass stored per ELL entry and the partition records (Fields::pkv: the
// half-step velocity, DepsDt, m and the evaluation's position).  The pairwise acceleration is
// re-formed as C*r with r computed from the evaluation's positions by the SPH pass's own
// operations, so it is the same bits the SPH pass summed into DvDt.
//
// FP64 forms a pair's share from node i's own side: with q = (v_o - v_i)^{1/2} . (C r) it is
// w (-m_o q), w = w_i/(w_i + w_o), w_x = max(eps, DepsDt_x sgn(-m q)).  q has the same bits from
// both sides (both factors change sign exactly), so both sides take the same branch and the two
// shares add up to the pair's work; one reciprocal instead of two divisions.  Mixed precision keeps
// the canonical (a, b) form.  Every lane of the quad returns the node's rate.
// ---------------------------------------------------------------------------
template <int D, typename R, int U>
__device__ __forceinline__ double compatible_rate(const Fields& f, const Geo& g, int i, int sub) {
  constexpr int L = kNodeLanes;
  const size_t ld = (size_t)f.ld;
  const R* pdd = (const R*)f.pdd;       // pair coefficients in the pair arithmetic; the partition is FP64
  const double ms = f.m[i];
  double v12s[D], xs[D];
  const double2* PV = reinterpret_cast<const double2*>(f.pkv);
  {
    const double2 a = PV[4*(size_t)i], b = PV[4*(size_t)i + 1], c = PV[4*(size_t)i + 2], d = PV[4*(size_t)i + 3];
    v12s[0] = a.x;
    if (D >= 2) v12s[1 % D] = a.y;
    if (D >= 3) v12s[2 % D] = b.x;
    xs[0] = c.y;
    if (D >= 2) xs[1 % D] = d.x;
    if (D >= 3) xs[2 % D] = d.y;
  }
  const double de0s = f.DepsDt[i];
  const double epsm = 2.220446049250313e-16;
  NodeSum<L, sizeof(R) == sizeof(float)> du(0.0, sub);
  const int nn = f.cnt[i];
  for (int k0 = 0; k0 < nn; k0 += U*L) {
    int js[U], codes[U];
    bool in[U];
    lane_entries<U, L>(f.nbr, ld, k0, sub, i, nn, js, codes, in);
    double vo[U][D], xo[U][D], mo[U], deo[U];
    R C[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = js[u];
      const double2 a = PV[4*(size_t)j], b = PV[4*(size_t)j + 1], c = PV[4*(size_t)j + 2], d = PV[4*(size_t)j + 3];
      vo[u][0] = a.x;
      if (D >= 2) vo[u][1 % D] = a.y;
      if (D >= 3) vo[u][2 % D] = b.x;
      deo[u] = b.y;
      mo[u] = c.x;
      xo[u][0] = c.y;
      if (D >= 2) xo[u][1 % D] = d.x;
      if (D >= 3) xo[u][2 % D] = d.y;
      C[u] = pdd[(size_t)(in[u] ? k0 + u*L + sub : 0)*ld + i];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      double t = 0.0;
      if (in[u]) {
        const int j = js[u], code = codes[u];
        if (code) {
          image_pos<D>(g, code, xo[u]);
#pragma unroll
          for (int c = 0; c < D; ++c) vo[u][c] *= refl_sign<D>(g, code, c);
        }
        if (sizeof(R) == sizeof(double)) {
          double q = 0.0;
#pragma unroll
          for (int c = 0; c < D; ++c)
            q += (vo[u][c] - v12s[c])*(double)(C[u]*(R)(xs[c] - xo[u][c]));     // the SPH pass's C*r
          const double e = -mo[u]*q;
          const double sgn = e < 0.0 ? -1.0 : 1.0;
          const double wi = fmax(epsm, de0s*sgn), wo = fmax(epsm, deo[u]*sgn);
          t = wi*fast_rcp(wi + wo)*e;
        } else {
          // canonical: pacc_ab = (-m_b) C r_ab ; du_ab = (v_b^{1/2} - v_a^{1/2}) . pacc_ab
          const bool aFirst = code != 0 || i < j;
          const double mb = aFirst ? mo[u] : ms, ma = aFirst ? ms : mo[u];
          double duab = 0.0;
#pragma unroll
          for (int c = 0; c < D; ++c) {
            const double dd = (double)(C[u]*(R)(xs[c] - xo[u][c]));     // the SPH pass's C*r, this lane's side
            const double va = aFirst ? v12s[c] : vo[u][c], vb = aFirst ? vo[u][c] : v12s[c];
            const double ddc = aFirst ? dd : -dd;
            const double ac = (-mb)*ddc;
            duab = c == 0 ? rounded_product(vb - va, ac) : fused(vb - va, ac, duab);
          }
          const double sgn = duab < 0.0 ? -1.0 : 1.0;
          const double wa = fmax(epsm, (aFirst ? de0s : deo[u])*sgn), wb = fmax(epsm, (aFirst ? deo[u] : de0s)*sgn);
          const double w = wa/(wa + wb);
          t = aFirst ? w*duab : (1.0 - w)*duab*ma/mb;
        }
      }
      du.add(t);
    }
  }
  return du.total();
}

// ---------------------------------------------------------------------------
// Full step from the start-of-step state with the midpoint derivatives
// (CheapSynchronousRK2.cc:106-109, SynchronousRK2.cc:115-118): the compatible energy
// partition (compatible_rate), then the increment and replace policies and the EOS.  v0 is
// read from f.v, the new velocity goes to f.v1.  The step variant also measures, per run, how far nodes have moved and h
// grown since the candidate list was built (see k_candidates).  ENERGY_ONLY: the
// package-level policy call (eps only).
// ---------------------------------------------------------------------------
template <int D, bool ENERGY_ONLY, typename R, int U>
__global__ void __launch_bounds__(kBlock) k_full_update(Fields f, Geo g, Phys ph, Scalars* sc, double multiplier,
                                                        int n) {
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int i = gl/kNodeLanes, sub = gl & (kNodeLanes - 1);
  const bool valid = i < n && sub == 0;
  int skr = 0;                       // candidate-list check: how far the run has used up its skin
  double skd = 0.0, skg = 0.0;
  double du = 0.0;
  if (i < n) du = compatible_rate<D, R, U>(f, g, i, sub);
  if (valid) {
  const double dt = ENERGY_ONLY ? multiplier : sc[f.run[i]].dt;
  const double eps1 = f.eps[i] + du*dt;
  f.eps[i] = eps1;
  if (ENERGY_ONLY) return;
  double x1[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    x1[a] = f.x[a][i] + dt*f.DxDt[a][i];
    f.x[a][i] = x1[a];
    double va = f.v[a][i] + dt*f.DvDt[a][i];
    if (ph.gravity) va = va + dt*f.DvDtG[a][i];
    f.v1[a][i] = va;
  }
  const double rho1 = fmin(ph.rho_max, fmax(ph.rho_min, f.rho[i] + dt*f.DrhoDt[i]));
  f.rho[i] = rho1;
  const double h1 = fmin(ph.hminInv, fmax(ph.hmaxInv, f.Hideal[i]));
  f.hinv[i] = h1;
  // end-of-step position and h^-1 for the grad-h pass that follows
  double2* PK = reinterpret_cast<double2*>(f.xh) + 2*(size_t)i;
  PK[0] = make_double2(x1[0], x1[1]);
  PK[1] = make_double2(x1[2], h1);
  // displacement and support growth since the run's candidate list was built
  skr = f.run[i];
  double d2 = 0.0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    double d = x1[a] - f.xb[a][i];
    if ((g.permask >> a) & 1) {
      const double box = g.xmax[a] - g.xmin[a];
      d = fabs(d);
      d = fmin(d, fabs(box - d));
    }
    d2 += d*d;
  }
  const double hb = f.hb[i];
  skd = sqrt(d2)*hb/ph.ext;
  skg = hb/h1;
  f.P[i] = ph.g1*rho1*eps1;
  f.cs[i] = sqrt(fmax(0.0, ph.gamma*ph.g1*eps1));
  }
  if (!ENERGY_ONLY) {
    const size_t stride = sizeof(Scalars)/sizeof(unsigned long long);
    run_max_bits(&sc[0].skinD, stride, skr, ord_bits(skd), valid);
    run_max_bits(&sc[0].skinG, stride, skr, ord_bits(skg), valid);
  }
}

// SynchronousRK2's trial half step (SynchronousRK2.cc:67-68: state.update with multiplier dt/2):
// the full policies, not timeAdvanceOnly -- the compatible energy partition of the start-of-step
// pair accelerations, the increments, H replaced by the ideal H (ReplaceBoundedState) and the
// EOS -- written to the midpoint arrays and position record; the start-of-step state stays.
template <int D, typename R, int U>
__global__ void __launch_bounds__(kBlock) k_half_update(Fields f, Geo g, Phys ph, const Scalars* sc, int n) {
  const int gl = xcd_block()*blockDim.x + threadIdx.x;
  const int i = gl/kNodeLanes, sub = gl & (kNodeLanes - 1);
  if (i >= n) return;
  const double du = compatible_rate<D, R, U>(f, g, i, sub);
  if (sub) return;
  const double hdt = sc[f.run[i]].hdt;
  const double eps = f.eps[i] + du*hdt;
  double xm[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    xm[a] = f.x[a][i] + hdt*f.DxDt[a][i];
    f.xm[a][i] = xm[a];
    double va = f.v[a][i] + hdt*f.DvDt[a][i];
    if (ph.gravity) va = va + hdt*f.DvDtG[a][i];
    f.vm[a][i] = va;
  }
  const double rho = fmin(ph.rho_max, fmax(ph.rho_min, f.rho[i] + hdt*f.DrhoDt[i]));
  const double h = fmin(ph.hminInv, fmax(ph.hmaxInv, f.Hideal[i]));
  f.rhom[i] = rho;
  f.epsm[i] = eps;
  f.hinvm[i] = h;
  f.Pm[i] = ph.g1*rho*eps;
  f.csm[i] = sqrt(fmax(0.0, ph.gamma*ph.g1*eps));
  double2* P = reinterpret_cast<double2*>(f.xhm) + 2*(size_t)i;
  P[0] = make_double2(xm[0], xm[1]);
  P[1] = make_double2(xm[2], h);
}

// Half-step velocity of the compatible-energy partition, v^{1/2} = v + a*multiplier/2 with the
// evaluation's hydro acceleration (SpecificThermalEnergyPolicy.cc:97-99), packed with DepsDt and
// m (Fields::pkv).  sc == nullptr: hdt is the fixed multiplier/2; otherwise hdt is the fraction
// of each run's dt (1/4 for SynchronousRK2's trial half step, whose multiplier is dt/2).
template <int D>
__global__ void __launch_bounds__(kBlock) k_v12(Fields f, const Scalars* sc, double hdtScale, int n) {
  const int i = blockIdx.x*blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double hdt = sc ? hdtScale*sc[f.run[i]].dt : hdtScale;
  double w[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int a = 0; a < D; ++a) w[a] = f.v[a][i] + f.DvDt[a][i]*hdt;
  double2* P = reinterpret_cast<double2*>(f.pkv) + 4*(size_t)i;
  P[0] = make_double2(w[0], w[1]);
  P[1] = make_double2(w[2], f.DepsDt[i]);
}


}  // namespace spx
