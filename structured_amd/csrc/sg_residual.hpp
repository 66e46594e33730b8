// Fused finite-volume residual on LDS tiles (one pass per tile):
// primitive recovery + ghost boundary cells -> power-law mu/k (+ SA eddy
// viscosity) -> MUSCL/van-Albada-type reconstruction -> Roe or AUSM face flux
// -> Green-Gauss face gradients and viscous flux -> SA source -> assembly /V,
// with the per-block partial sums of R^2 for the L2 norm.
//
// Follows EulerEquation::calc_residual (src/model/eulerequation.cpp:202-232)
// and the kernels it calls: FluidModel::primvars (src/model/fluid.cpp:50-67),
// BoundaryContainer::apply (src/model/bc.cpp:430-433), ReconstructionSecondOrder
// (src/model/reconstruction.cpp:55-154), ConvectiveFluxRoe (src/model/flux.cpp:51-146),
// ConvectiveFluxAUSM (:149-224), Mesh::calc_gradient / calc_face
// (src/utils/mesh.cpp:8-131) and DiffusiveFluxGreenGauss (src/model/flux.cpp:12-48).
//
// Tiling.  A block of TX x TY threads (32 x 8 or 32 x 16) is a grid of face
// owners: thread (tx, ty) computes the chi face i0+tx on row j0+ty and the eta
// face j0+ty on column i0+tx, so every thread evaluates exactly two faces.
// The block then assembles the (TX - 1) x (TY - 1) cells whose four faces it
// owns, so one column and one row of faces per tile are computed twice.  The
// cell data of the tile plus its halo (two cells along each face normal for
// MUSCL, one cell around for the viscous stencil) is staged once in LDS as
// primitives and transport properties.
//
// Bound.  FP64 issue on large grids (two thirds of the vector instructions are
// FP64, the rest address, select and move), the chain load - stage - barrier -
// faces - barrier - cell - norms on small ones.  Both want few branches: the
// ends of grid lines are handled by clamped indices and selects, where a
// branch per variable and per kind of face kept the loads of a face behind one
// another and cost a third of the instructions that are not FP64; ghost cells
// are evaluated once, by threads of their own.  With it, a finaliser that waits
// on slots instead of counting arrivals, and metrics loaded just ahead of their
// use so that nothing spills, SA at 545x385 24.0 -> 20.2 us, 1409x641 77 -> 61,
// laminar 97x65 16.4 -> 9.2; J.v at 705x321 41.5 -> 32.4.
#pragma once
#include "sg_closure.hpp"
#include "sg_device.hpp"
#include "sg_scalar.hpp"

namespace sg {

constexpr int RW = TX + 3;           // LDS region, origin (i0-2, j0-2)
template <class S>
struct Prim {
  S r, u, v, p, T, n;
};

// Primitives from the conservative values (rho, rho u, rho v, rho E[, rho nu~]).
template <class S, bool SA>
__device__ __forceinline__ Prim<S> prim_from_cons(const S* qc, const DevPhys& ph) {
  Prim<S> P;
  P.r = qc[0];
  const S ir = srcp(P.r);
  P.u = qc[1] * ir;
  P.v = qc[2] * ir;
  P.p = (qc[3] - 0.5 * P.r * (P.u * P.u + P.v * P.v)) * (kGamma - 1.0);
  P.T = P.p * ir * ph.iR;
  if (SA) P.n = qc[4] * ir;
  else P.n = S(0.0);
  return P;
}

template <class S, bool SA, class F>
__device__ __forceinline__ Prim<S> prim_interior(const F& q, const DevGeom& g, const DevPhys& ph, int ci, int cj) {
  const size_t idx = (size_t)cj * g.ldi + ci;
  S qc[5];
#pragma unroll
  for (int k = 0; k < (SA ? 5 : 4); ++k) qc[k] = q.at(k, g.plane, idx, ci, cj);
  return prim_from_cons<S, SA>(qc, ph);
}

// src/model/bc.cpp: freestream :25-60, slipwall :77-128, wall :149-204,
// outflow :283-311, periodic/wake copies :223-263,328-365, isothermal :387-427.
template <class S>
__device__ __forceinline__ Prim<S> apply_op(const BcNode& nd, const Prim<S>& A, const Prim<S>& B, const DevPhys& ph) {
  Prim<S> o;
  switch (nd.op) {
    case OP_FREESTREAM:
      o.r = S(ph.rho_inf); o.u = S(ph.u_inf); o.v = S(ph.v_inf); o.p = S(ph.p_inf);
      o.T = sdiv(o.p, o.r) * ph.iR; o.n = S(ph.nut_inf);
      break;
    case OP_SLIP: {
      const double nx = nd.c0, ny = nd.c1, ids = frcp(nx * nx + ny * ny);
      o.p = 1.5 * A.p - 0.5 * B.p;
      o.r = 1.5 * A.r - 0.5 * B.r;
      S un = A.u * nx + A.v * ny;
      o.u = A.u - 2.0 * un * nx * ids;
      o.v = A.v - 2.0 * un * ny * ids;
      o.T = sdiv(o.p, o.r) * ph.iR;
      o.n = 1.5 * A.n - 0.5 * B.n;
    } break;
    case OP_WALL:
      o.T = 1.5 * A.T - 0.5 * B.T;
      o.r = 1.5 * A.r - 0.5 * B.r;
      o.u = 2.0 * nd.c0 - (1.5 * A.u - 0.5 * B.u);
      o.v = 2.0 * nd.c1 - (1.5 * A.v - 0.5 * B.v);
      o.p = o.r * ph.R * o.T;
      o.n = -(1.5 * A.n - 0.5 * B.n);
      break;
    case OP_ISO:
      o.p = 1.5 * A.p - 0.5 * B.p;
      o.u = 2.0 * nd.c0 - (1.5 * A.u - 0.5 * B.u);
      o.v = 2.0 * nd.c1 - (1.5 * A.v - 0.5 * B.v);
      o.T = S(nd.c2);
      o.r = sdiv(o.p, o.T) * ph.iR;
      o.n = -(1.5 * A.n - 0.5 * B.n);
      break;
    case OP_OUTFLOW:
      o.r = A.r; o.u = A.u; o.v = A.v; o.p = S(ph.p_inf);
      o.T = sdiv(o.p, o.r) * ph.iR; o.n = A.n;
      break;
    default:  // OP_COPY
      o = A;
      break;
  }
  return o;
}

template <class S, bool SA, class F>
__device__ __forceinline__ Prim<S> ref_leaf(int ref, const F& q, const DevGeom& g, const DevPhys& ph) {
  return prim_interior<S, SA>(q, g, ph, ref % g.nic, ref / g.nic);
}

// Node whose operands are interior cells.
template <class S, bool SA, class F>
__device__ Prim<S> eval_leaf_node(const BcNode& nd, const F& q, const DevGeom& g, const DevPhys& ph) {
  Prim<S> A, B;
  if (nd.op != OP_FREESTREAM) A = ref_leaf<S, SA>(nd.ra, q, g, ph);
  if (nd.op == OP_SLIP || nd.op == OP_WALL || nd.op == OP_ISO) B = ref_leaf<S, SA>(nd.rb, q, g, ph);
  return apply_op<S>(nd, A, B, ph);
}

// Node whose operands are interior cells or leaf nodes (depth <= 2 is
// guaranteed by the host-side boundary compiler).
template <class S, bool SA, class F>
__device__ Prim<S> eval_node(int id, const DevBc& bc, const F& q, const DevGeom& g, const DevPhys& ph) {
  const BcNode nd = bc.nodes[id];
  Prim<S> A, B;
  if (nd.op != OP_FREESTREAM) {
    A = nd.ra >= 0 ? ref_leaf<S, SA>(nd.ra, q, g, ph) : eval_leaf_node<S, SA>(bc.nodes[-(nd.ra + 1)], q, g, ph);
  }
  if (nd.op == OP_SLIP || nd.op == OP_WALL || nd.op == OP_ISO) {
    B = nd.rb >= 0 ? ref_leaf<S, SA>(nd.rb, q, g, ph) : eval_leaf_node<S, SA>(bc.nodes[-(nd.rb + 1)], q, g, ph);
  }
  return apply_op<S>(nd, A, B, ph);
}

__device__ __forceinline__ int ghost_index(int ci, int cj, int nic, int njc) {
  const int gi = ci + 1, gj = cj + 1;
  if (gj == 0) return gi;
  if (gj == njc + 1) return (nic + 2) + gi;
  if (gi == 0) return 2 * (nic + 2) + gj - 1;
  return 2 * (nic + 2) + njc + gj - 1;
}

// A pure tangent (value 0) for the dual, nothing for plain doubles.
template <class S>
__device__ __forceinline__ S beta_tangent(double t);
template <>
__device__ __forceinline__ double beta_tangent<double>(double) { return 0.0; }
template <>
__device__ __forceinline__ Dual beta_tangent<Dual>(double t) { return Dual(0.0, t); }

// LDS slots of the staged cell data.
enum { L_R = 0, L_U, L_V, L_P, L_T, L_MU, L_K, L_N, L_ETA, L_ML, L_MAX };

// MUSCL left/right states, src/model/reconstruction.cpp:142-219.
// Left state of a face from cell c with neighbours cm (behind) and cp (ahead):
//   dm = c - cm, dp = cp - c, s = 0.25 (3 dp dm + eps) / (2 (dp - dm)^2 + 3 dp dm + eps)
//   left  = c + s (2/3 dm + 4/3 dp);   right = c - s (4/3 dm + 2/3 dp)
template <class S>
__device__ __forceinline__ S muscl_left(S cm, S c, S cp, double eps) {
  const double thm = 2.0 / 3.0, thp = 4.0 / 3.0;
  S dm = c - cm, dp = cp - c;
  S a1 = 3.0 * dp * dm;
  S a2 = 2.0 * (dp - dm) * (dp - dm) + a1;
  S s = 0.25 * sdiv(a1 + eps, a2 + eps);
  return c + s * (thm * dm + thp * dp);
}
template <class S>
__device__ __forceinline__ S muscl_right(S cm, S c, S cp, double eps) {
  const double thm = 2.0 / 3.0, thp = 4.0 / 3.0;
  S dm = c - cm, dp = cp - c;
  S a1 = 3.0 * dp * dm;
  S a2 = 2.0 * (dp - dm) * (dp - dm) + a1;
  S s = 0.25 * sdiv(a1 + eps, a2 + eps);
  return c - s * (thp * dm + thm * dp);
}

// Roe flux without entropy fix, src/model/flux.cpp:51-146; with SA the
// rho*nu~ transport is first-order upwind on the Roe mass flux.
template <class S, bool SA>
__device__ __forceinline__ void roe_flux(double nx, double ny, S rl, S ul, S vl, S pl, S rr, S ur, S vr, S pr, S ntl,
                                         S ntr, S* f) {
  const double gm1 = kGamma - 1.0, ogm1 = 1.0 / gm1;
  S rli = srcp(rl), rul = rl * ul, rvl = rl * vl, uvl = 0.5 * (ul * ul + vl * vl);
  S el = pl * ogm1 + rl * uvl, hl = (el + pl) * rli;
  S rri = srcp(rr), rur = rr * ur, rvr = rr * vr, uvr = 0.5 * (ur * ur + vr * vr);
  S er = pr * ogm1 + rr * uvr, hr = (er + pr) * rri;
  S rat = ssqrt(rr * rli), rati = srcp(rat + 1.0);
  S rav = rat * rl, uav = (rat * ur + ul) * rati, vav = (rat * vr + vl) * rati, hav = (rat * hr + hl) * rati;
  S uv = 0.5 * (uav * uav + vav * vav);
  S cav = ssqrt(gm1 * (hav - uv));
  S d1 = rr - rl, d2 = ur - ul, d3 = vr - vl, d4 = pr - pl;
  const double dr = fsqrt(nx * nx + ny * ny), idr = frcp(dr), r1 = nx * idr, r2 = ny * idr;
  S uu = r1 * uav + r2 * vav, c2 = cav * cav, c2i = srcp(c2);
  S auu = sabs(uu), aupc = sabs(uu + cav), aumc = sabs(uu - cav);
  S uul = r1 * ul + r2 * vl, uur = r1 * ur + r2 * vr;
  S rcav = rav * cav, aquu = uur - uul, c2ih = 0.5 * c2i, ruuav = auu * rav;
  S b1 = auu * (d1 - c2i * d4);
  S b2 = c2ih * aupc * (d4 + rcav * aquu);
  S b3 = c2ih * aumc * (d4 - rcav * aquu);
  S b4 = b1 + b2 + b3, b5 = cav * (b2 - b3);
  S b6 = ruuav * (d2 - r1 * aquu), b7 = ruuav * (d3 - r2 * aquu);
  S a2 = uav * b4 + r1 * b5 + b6, a3 = vav * b4 + r2 * b5 + b7;
  S a4 = hav * b4 + uu * b5 + uav * b6 + vav * b7 - c2 * b1 * ogm1;
  const double aj = 0.5 * dr;
  S plar = pl + pr, epl = el + pl, epr = er + pr;
  f[0] = aj * (rl * uul + rr * uur - b4);
  f[1] = aj * (rul * uul + rur * uur + r1 * plar - a2);
  f[2] = aj * (rvl * uul + rvr * uur + r2 * plar - a3);
  f[3] = aj * (epl * uul + epr * uur - a4);
  if (SA) f[4] = 0.5 * (f[0] * (ntl + ntr) - sabs(f[0]) * (ntr - ntl));
}

// AUSM flux (Liou-Steffen), src/model/flux.cpp:149-224: split Mach numbers
// M+-(M) = +-(M +- 1)^2 / 4 and pressures P+-(M) = p (M +- 1)^2 (2 -+ M) / 4
// for |M| <= 1, otherwise the upwind values (M+ = M, P+ = p for M > 1 and 0
// for M < -1; mirrored for M-P-); the interface Mach number picks the side
// whose rho a (1, u, v, h) is convected.  With SA, rho*nu~ is carried
// first-order upwind by the AUSM mass flux, as for Roe.
template <class S, bool SA>
__device__ __forceinline__ void ausm_flux(double nx, double ny, S rl, S ul, S vl, S pl, S rr, S ur, S vr, S pr, S ntl,
                                          S ntr, S* f) {
  const double ds = fsqrt(nx * nx + ny * ny), ids = frcp(ds), gg = kGamma / (kGamma - 1.0);
  S rli = srcp(rl), rri = srcp(rr);
  S al = ssqrt(kGamma * pl * rli), ar = ssqrt(kGamma * pr * rri);
  S Ml = (ul * nx + vl * ny) * ids * srcp(al), Mr = (ur * nx + vr * ny) * ids * srcp(ar);
  S mp, pp, mm, pm;
  if (fabs(val(Ml)) <= 1.0) {
    S a = Ml + 1.0, a2 = 0.25 * a * a;
    mp = a2; pp = pl * a2 * (2.0 - Ml);
  } else if (val(Ml) > 0.0) {
    mp = Ml; pp = pl;
  } else {
    mp = S(0.0); pp = S(0.0);
  }
  if (fabs(val(Mr)) <= 1.0) {
    S b = Mr - 1.0, b2 = 0.25 * b * b;
    mm = -b2; pm = pr * b2 * (2.0 + Mr);
  } else if (val(Mr) < 0.0) {
    mm = Mr; pm = pr;
  } else {
    mm = S(0.0); pm = S(0.0);
  }
  S mh = mp + mm, ph = pp + pm;
  const bool up = val(mh) >= 0.0;
  S r = up ? rl : rr, a = up ? al : ar, u = up ? ul : ur, v = up ? vl : vr;
  S h = gg * (up ? pl * rli : pr * rri) + 0.5 * (u * u + v * v);
  S m = r * a * mh * ds;
  f[0] = m;
  f[1] = m * u + ph * nx;
  f[2] = m * v + ph * ny;
  f[3] = m * h;
  if (SA) f[4] = 0.5 * (f[0] * (ntl + ntr) - sabs(f[0]) * (ntr - ntl));
}

template <class S, bool SA>
__device__ __forceinline__ void conv_flux(int kind, double nx, double ny, S rl, S ul, S vl, S pl, S rr, S ur, S vr,
                                          S pr, S ntl, S ntr, S* f) {
  if (kind == FLUX_AUSM) ausm_flux<S, SA>(nx, ny, rl, ul, vl, pl, rr, ur, vr, pr, ntl, ntr, f);
  else roe_flux<S, SA>(nx, ny, rl, ul, vl, pl, rr, ur, vr, pr, ntl, ntr, f);
}

template <class S>
struct FaceGeo {
  double tx, ty, bx, by, lx, ly, rx, ry, ivol;  // top/bottom/left/right normals, 1/auxiliary volume
};

// Green-Gauss face gradient (src/utils/mesh.cpp:34-131) of one variable from
// the face's left/right cells and its top/bottom 4-cell averages.
template <class S>
__device__ __forceinline__ void gg_grad(const FaceGeo<S>& G, S qt, S qb, S ql, S qr, S* out) {
  out[0] = (G.tx * qt - G.bx * qb + G.rx * qr - G.lx * ql) * G.ivol;
  out[1] = (G.ty * qt - G.by * qb + G.ry * qr - G.ly * ql) * G.ivol;
}

// DiffusiveFluxGreenGauss::evaluate, src/model/flux.cpp:12-48 (+ SA nu~ diffusion).
template <class S, bool SA>
__device__ __forceinline__ void visc_flux(double nx, double ny, const S* gu, const S* gv, const S* gT, S ub, S vb, S m,
                                          S k, const S* gn, S et, S* f) {
  S txy = m * (gu[1] + gv[0]);
  S txx = m * (2.0 * gu[0] - 2.0 / 3.0 * (gu[0] + gv[1]));
  S tyy = m * (2.0 * gv[1] - 2.0 / 3.0 * (gu[0] + gv[1]));
  S qx = -k * gT[0], qy = -k * gT[1];
  f[1] = txx * nx + txy * ny;
  f[2] = txy * nx + tyy * ny;
  f[3] = (ub * txx + vb * txy - qx) * nx + (ub * txy + vb * tyy - qy) * ny;
  if (SA) f[4] = (1.0 / kSigma) * et * (gn[0] * nx + gn[1] * ny);
}

template <class S, bool SA>
__device__ __forceinline__ void transport(const Prim<S>& P, const DevPhys& ph, S* slot) {
  S ml = ph.mu_inf * spow23(P.T * ph.iTinf);
  if (!SA) {
    slot[L_MU] = ml;
    slot[L_K] = ml * ph.cp * ph.ipr;
    return;
  }
  S rn = P.r * P.n;
  S chi = sdiv(rn, ml), chi3 = chi * chi * chi;
  S mut(0.0), fn(1.0);
  if (val(P.n) >= 0.0) mut = rn * sdiv(chi3, chi3 + kCv1 * kCv1 * kCv1);
  else fn = sdiv(kCn1 + chi3, kCn1 - chi3);
  slot[L_MU] = ml + mut;
  slot[L_K] = ph.cp * (ml * ph.ipr + mut * (1.0 / kPrt));
  slot[L_ETA] = ml + rn * fn;
  slot[L_ML] = ml;
}

// SA-noft2 source (production * beta - destruction + cb2 and density-gradient
// diffusion terms, NASA TMR compressible form) at one cell; the cell
// gradients are Green-Gauss over its four faces with arithmetic face means.
// Split as src = beta * P1 - D + rest so that a closure can supply beta.
template <class S>
struct SaTerms {
  S P1, D, rest;
};
template <class S>
__device__ __forceinline__ SaTerms<S> sa_terms(S r, S n, S ml, const S* gu, const S* gv, const S* gn, const S* gr,
                                               double d) {
  const double cw1 = kCb1 / (kKappa * kKappa) + (1.0 + kCb2) / kSigma;
  S nu = sdiv(ml, r);
  S omega = sabs(gv[0] - gu[1]);
  const double k2d2 = kKappa * kKappa * d * d, ik2d2 = frcp(k2d2), id = frcp(d);
  SaTerms<S> t;
  if (val(n) >= 0.0) {
    S chi = sdiv(n, nu), chi3 = chi * chi * chi;
    S fv1 = sdiv(chi3, chi3 + kCv1 * kCv1 * kCv1);
    S fv2 = 1.0 - sdiv(chi, 1.0 + chi * fv1);
    S sbar = n * fv2 * ik2d2;
    S stil = (val(sbar) >= -kCv2 * val(omega))
                 ? omega + sbar
                 : omega + sdiv(omega * (kCv2 * kCv2 * omega + kCv3 * sbar), (kCv3 - 2.0 * kCv2) * omega - sbar);
    S rr = (val(stil) > 0.0) ? smin(sdiv(n, stil * k2d2), 10.0) : S(10.0);
    S r2 = rr * rr, r6 = r2 * r2 * r2;
    S gg = rr + kCw2 * (r6 - rr);
    S g2 = gg * gg, g6 = g2 * g2 * g2;
    const double cw3_6 = kCw3 * kCw3 * kCw3 * kCw3 * kCw3 * kCw3;
    S fw = gg * spow16(sdiv(S(1.0 + cw3_6), g6 + cw3_6));
    t.P1 = kCb1 * stil * r * n;
    t.D = cw1 * fw * r * (n * id) * (n * id);
  } else {
    t.P1 = kCb1 * (1.0 - kCt3) * omega * r * n;
    t.D = -cw1 * r * (n * id) * (n * id);
  }
  S cb2t = (kCb2 / kSigma) * r * (gn[0] * gn[0] + gn[1] * gn[1]);
  S cross = -(1.0 / kSigma) * (nu + n) * (gr[0] * gn[0] + gr[1] * gn[1]);
  t.rest = cb2t + cross;
  return t;
}

// Fused norm output.  With slots set the launch has one more block, the last,
// which waits for every tile's partial sums, adds them in a fixed order and
// empties the slots for the next launch.  A slot is one 64-bit atomic that
// holds either a partial sum or kNoValue, so nothing has to be ordered between
// slots.  The tiles depend on nothing, so the wait ends; see SlotHead for one that
// gives up.
struct NormOut {
  unsigned long long* slots = nullptr;  // 2 NV per tile, component-major, after their head
  double* l2 = nullptr;                 // ||R_k||_2 (k < NV), then ||V R_k||_2 (NV <= k < 2 NV)
  int count = 0;                        // entries of l2 written: NV (caller's buffer) or 2 NV
};

template <int NT, int NV2>
__device__ __forceinline__ void finalise_norms(const NormOut& no, int ntile, double (*red)[NV2]) {
  const int tid = threadIdx.x;
  const SlotHead head = slot_head(no.slots);
  double acc[NV2];
#pragma unroll
  for (int k = 0; k < NV2; ++k) acc[k] = 0.0;
  unsigned long long polls = 0;
  for (int b = tid; b < ntile; b += NT) {
    unsigned long long v[NV2];
    bool wait = true;
    while (wait) {  // every sum of the tile again, all loads in flight together
#pragma unroll
      for (int k = 0; k < NV2; ++k) v[k] = k < no.count ? slot_load(no.slots + (size_t)k * ntile + b) : 0ull;
      wait = false;
#pragma unroll
      for (int k = 0; k < NV2; ++k) wait = wait || v[k] == kNoValue;
      if (wait && ++polls > head.polls) break;
    }
#pragma unroll
    for (int k = 0; k < NV2; ++k) {
      if (k < no.count) slot_store(no.slots + (size_t)k * ntile + b, kNoValue);
      acc[k] += wait ? __builtin_nan("") : __longlong_as_double((long long)v[k]);
    }
  }
  if (polls > head.polls) slots_lost(no.slots);
  if (head.state != kNoValue) {
#pragma unroll
    for (int k = 0; k < NV2; ++k) acc[k] = __builtin_nan("");
  }
#pragma unroll
  for (int k = 0; k < NV2; ++k) acc[k] = wave_sum_lane63(acc[k]);
  if ((tid & 63) == 63) {
#pragma unroll
    for (int k = 0; k < NV2; ++k) red[tid >> 6][k] = acc[k];
  }
  __syncthreads();
  if (tid < no.count) {
    double s = 0.0;
    for (int w = 0; w < NT / 64; ++w) s += red[w][tid];
    no.l2[tid] = sqrt(s);
  }
}

// CL: closure kind of beta (ClosureKind); CLOSURE_MLP stages the hidden
// layer of the network (and its tangent) in the same LDS area.  F and O: where
// the state comes from and the result goes (Field and OutField, or SeedField
// and OutBlocks for Jacobian blocks).
template <int TY, class I, class S, bool SA, int CL, class F, class O>
__global__ __launch_bounds__(TX * TY, sizeof(S) == sizeof(double) ? 4 : 2) void residual_kernel(
    DevGeom g, DevPhys ph, DevBc bc, F q, O out, const double* beta_dot, DevClosure clo, NormOut nout) {
  constexpr int NT = TX * TY, OY = TY - 1, RH = TY + 3, NPOS = RW * RH;
  constexpr int NL = SA ? L_MAX : (L_K + 1);
  constexpr int NV = SA ? 5 : 4;
  constexpr int NLDS0 = NL * NPOS > 2 * NV * (NT + 16) ? NL * NPOS : 2 * NV * (NT + 16);  // cells, then fluxes, then sums
  constexpr int NLDS_D = NLDS0 * (int)(sizeof(S) / sizeof(double));
  constexpr bool TAN = sizeof(S) > sizeof(double);
  constexpr int NMLP_D = (CL == CLOSURE_MLP) ? (TAN ? 2 : 1) * (NT / 64) * 64 * kHld / 4 : 0;
  __shared__ double lds_raw[NLDS_D > NMLP_D ? NLDS_D : NMLP_D];
  S* lds = reinterpret_cast<S*>(lds_raw);
  __shared__ double red[NT / 64][2 * NV];

  const int ncol = (g.nic + OX - 1) / OX, ntile = residual_tiles(g, TY);
  int tile = blockIdx.x;
  if (tile == ntile) {
    finalise_norms<NT, 2 * NV>(nout, ntile, red);
    return;
  }
  const int bid = tile;
  q.begin(blockIdx.z);
  out.begin(blockIdx.z);
  const int tid = threadIdx.x;
  const int tx = tid % TX, ty = tid / TX;
  // XCD-aware tile order: work-groups are handed to the 8 XCDs round-robin in
  // linear order, so XCD x's k-th group takes the k-th tile of the x-th
  // contiguous run of tiles; neighbouring tiles then share their halo rows in
  // the same L2.  The map is a bijection on the tiles for any tile count.
  {
    const int x = tile & 7, k = tile >> 3, qn = ntile >> 3, rn = ntile & 7;
    tile = (x < rn) ? x * (qn + 1) + k : rn * (qn + 1) + (x - rn) * qn + k;
  }
  const int trow = tile / ncol, i0 = (tile - trow * ncol) * OX, j0 = trow * OY;
  const int nic = g.nic, njc = g.njc;

  const int jo = max(j0 - 2, 0), io = max(i0 - 2, 0);

  // ---- ghost cells of the ring around the grid that lie in this tile's
  // region: at most RW on a row and RH on a column, one thread each.  The
  // threads counted from the end take them, since the first waves have the
  // second pass of the staging.  The boundary node is asked for first; what it
  // reads is two dependent loads away.
  static_assert(2 * (RW + RH) <= NT, "a thread per ghost cell");
  int gp = -1, node = -1;
  {
    const int t = NT - 1 - tid;
    int lx, ly;
    if (t < 2 * RW) { lx = t < RW ? t : t - RW; ly = t < RW ? 1 - j0 : njc - j0 + 2; }
    else { const int u = t - 2 * RW; ly = u < RH ? u : u - RH; lx = u < RH ? 1 - i0 : nic - i0 + 2; }
    const int ci = i0 - 2 + lx, cj = j0 - 2 + ly;
    // a corner belongs to the row
    if (t < 2 * (RW + RH) && lx >= 0 && lx < RW && ly >= 0 && ly < RH && ci >= -1 && ci <= nic && cj >= -1 && cj <= njc &&
        (t < 2 * RW || (cj >= 0 && cj < njc))) {
      gp = ly * RW + lx;
      node = bc.ghost_map[ghost_index(ci, cj, nic, njc)];
    }
  }

  // ---- stage primitives (+ transport properties) of tile + halo in LDS.
  // A thread stages at most NPASS positions; the conservative values of its
  // interior positions are loaded first, all in flight together, and only
  // then converted.
  constexpr int NPASS = (NPOS + NT - 1) / NT;
  constexpr int NQ = SA ? 5 : 4;
  auto stage = [&](int p, int lx, int ly, const Prim<S>& P) {
    lds[L_R * NPOS + p] = P.r; lds[L_U * NPOS + p] = P.u; lds[L_V * NPOS + p] = P.v; lds[L_P * NPOS + p] = P.p;
    lds[L_T * NPOS + p] = P.T;
    if (SA) lds[L_N * NPOS + p] = P.n;
    // the viscous stencil reads transport properties one cell around only
    if (ph.viscous && lx >= 1 && lx < RW - 1 && ly >= 1 && ly < RH - 1) {
      S slot[L_MAX];
      transport<S, SA>(P, ph, slot);
      lds[L_MU * NPOS + p] = slot[L_MU]; lds[L_K * NPOS + p] = slot[L_K];
      if (SA) { lds[L_ETA * NPOS + p] = slot[L_ETA]; lds[L_ML * NPOS + p] = slot[L_ML]; }
    }
  };
  S qraw[NPASS][NQ];
#pragma unroll
  for (int pass = 0; pass < NPASS; ++pass) {
    const int p = tid + pass * NT;
    const int ci = i0 - 2 + p % RW, cj = j0 - 2 + p / RW;
    // positions outside the grid load the nearest cell and do not use it
    const int cc = min(max(ci, 0), nic - 1), cr = min(max(cj, 0), njc - 1);
    if (p < NPOS) q.template load<NQ, I>(qraw[pass], g.plane, g.ldi, jo, io, cc, cr);
  }
#pragma unroll
  for (int pass = 0; pass < NPASS; ++pass) {
    const int p = tid + pass * NT;
    if (p >= NPOS) break;
    const int lx = p % RW, ly = p / RW;
    const int ci = i0 - 2 + lx, cj = j0 - 2 + ly;
    if (ci < 0 || ci >= nic || cj < 0 || cj >= njc) continue;
    stage(p, lx, ly, prim_from_cons<S, SA>(qraw[pass], ph));
  }
  if (gp >= 0) {
    const S nan(__builtin_nan(""));
    Prim<S> P{nan, nan, nan, nan, nan, nan};
    if (node >= 0) P = eval_node<S, SA>(node, bc, q, g, ph);
    stage(gp, gp % RW, gp / RW, P);
  }
  // ---- metrics of this thread's two faces and cell, loaded where they are used.
  // Loaded together ahead of the reconstruction, the 128 registers did not hold
  // them: the spills were 10 of 40 MB that a launch moved at 545x385, and cost 1 us
  // there, 6 at 1409x641.  The other waves cover the wait.  At the ends of a grid
  // line the neighbour index is clamped: the mean of a face's normal (a cell's
  // volume) with itself is the one-sided value that belongs there, and a thread
  // without a face computes one that nothing reads.
  const int fi = i0 + tx, cj = j0 + ty;  // the chi face's row is the eta face's upper cell
  double2 C0, CL_, CR, Cb, CRb, E0, EL, Et, ELt, Eb;
  double V0, VL, VB;
  const int f0 = min(fi, nic), fr = min(f0 + 1, nic), c0 = min(fi, nic - 1);
  const int e0 = min(cj, njc), eb = max(e0 - 1, 0);
  auto nc = [&](int f, int r) { return double2{tile_at<I>(g.ncx, g.ldf, jo, io, f, r), tile_at<I>(g.ncy, g.ldf, jo, io, f, r)}; };
  auto ne = [&](int c, int r) { return double2{tile_at<I>(g.nex, g.ldi, jo, io, c, r), tile_at<I>(g.ney, g.ldi, jo, io, c, r)}; };
  auto vol = [&](int c, int r) { return tile_at<I>(g.vol, g.ldi, jo, io, c, r); };
  const int fl = max(f0 - 1, 0), cl = min(fl, c0), r0 = min(cj, njc - 1), et = min(e0 + 1, njc);
  C0 = nc(f0, r0);
  __syncthreads();

  auto at = [&](int k, int lx, int ly) -> S { return lds[k * NPOS + ly * RW + lx]; };

  S hc[NV], he[NV];

  // ---- chi face fi on row cj (between cells fi-1 and fi)
  {
    const int xl = tx + 1, xr = tx + 2, y = ty + 2;  // LDS coords of the left/right cells
    S st[2][4];
    const bool sl = fi >= 1, sr = fi <= nic - 1;  // first order from a ghost cell
    if (ph.order == 2) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const S a = at(L_R + k, xl, y), b = at(L_R + k, xr, y);
        st[0][k] = ssel(sl, muscl_left(at(L_R + k, xl - 1, y), a, b, ph.eps_chi), a);
        st[1][k] = ssel(sr, muscl_right(a, b, at(L_R + k, xr + 1, y), ph.eps_chi), b);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) { st[0][k] = at(L_R + k, xl, y); st[1][k] = at(L_R + k, xr, y); }
    }
    S ntl(0.0), ntr(0.0);
    if (SA) { ntl = at(L_N, xl, y); ntr = at(L_N, xr, y); }
    conv_flux<S, SA>(ph.flux, C0.x, C0.y, st[0][0], st[0][1], st[0][2], st[0][3], st[1][0], st[1][1], st[1][2], st[1][3],
                     ntl, ntr, hc);
    CL_ = nc(fl, r0); CR = nc(fr, r0);
    E0 = ne(c0, e0); EL = ne(cl, e0); Et = ne(c0, et); ELt = ne(cl, et);
    V0 = vol(c0, r0); VL = vol(cl, r0);
    if (ph.viscous) {
      FaceGeo<S> G;
      G.tx = 0.5 * (Et.x + ELt.x); G.ty = 0.5 * (Et.y + ELt.y);
      G.bx = 0.5 * (E0.x + EL.x); G.by = 0.5 * (E0.y + EL.y);
      G.rx = 0.5 * (C0.x + CR.x); G.ry = 0.5 * (C0.y + CR.y);
      G.lx = 0.5 * (C0.x + CL_.x); G.ly = 0.5 * (C0.y + CL_.y);
      G.ivol = frcp(0.5 * (V0 + VL));
      // left/right cells and their north/south neighbours
      auto grad_avg = [&](int k, S* gr, S* avg) {
        S a = at(k, xl, y), b = at(k, xr, y);
        S qt = 0.25 * (a + b + at(k, xl, y + 1) + at(k, xr, y + 1));
        S qb = 0.25 * (a + b + at(k, xl, y - 1) + at(k, xr, y - 1));
        if (gr) gg_grad(G, qt, qb, a, b, gr);
        if (avg) *avg = 0.25 * (a + b + qt + qb);
      };
      S gu[2], gv[2], gT[2], gn[2] = {S(0.0), S(0.0)}, ub, vb, mb, kb, eb(0.0);
      grad_avg(L_U, gu, &ub);
      grad_avg(L_V, gv, &vb);
      grad_avg(L_T, gT, nullptr);
      grad_avg(L_MU, nullptr, &mb);
      grad_avg(L_K, nullptr, &kb);
      if (SA) { grad_avg(L_N, gn, nullptr); grad_avg(L_ETA, nullptr, &eb); }
      S fv[5];
      visc_flux<S, SA>(C0.x, C0.y, gu, gv, gT, ub, vb, mb, kb, gn, eb, fv);
#pragma unroll
      for (int k = 1; k < NV; ++k) hc[k] = hc[k] - fv[k];
    }
  }

  // ---- eta face fj on column ci (between cells fj-1 and fj)
  {
    const int x = tx + 2, ys = ty + 1, yn = ty + 2;
    S st[2][4];
    const bool sl = cj >= 1, sr = cj <= njc - 1;  // first order from a ghost cell
    if (ph.order == 2) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const S cl = at(L_R + k, x, ys), cr = at(L_R + k, x, yn);
        st[0][k] = ssel(sl, muscl_left(at(L_R + k, x, ys - 1), cl, cr, ph.eps_eta), cl);
        st[1][k] = ssel(sr, muscl_right(cl, cr, at(L_R + k, x, yn + 1), ph.eps_eta), cr);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) { st[0][k] = at(L_R + k, x, ys); st[1][k] = at(L_R + k, x, yn); }
    }
    S nts(0.0), ntn(0.0);
    if (SA) { nts = at(L_N, x, ys); ntn = at(L_N, x, yn); }
    conv_flux<S, SA>(ph.flux, E0.x, E0.y, st[0][0], st[0][1], st[0][2], st[0][3], st[1][0], st[1][1], st[1][2], st[1][3],
                     nts, ntn, he);
    Cb = nc(f0, eb); CRb = nc(fr, eb); Eb = ne(c0, eb); VB = vol(c0, eb);
    if (ph.viscous) {
      FaceGeo<S> G;
      G.tx = 0.5 * (E0.x + Et.x); G.ty = 0.5 * (E0.y + Et.y);
      G.bx = 0.5 * (E0.x + Eb.x); G.by = 0.5 * (E0.y + Eb.y);
      G.lx = 0.5 * (C0.x + Cb.x); G.ly = 0.5 * (C0.y + Cb.y);
      G.rx = 0.5 * (CR.x + CRb.x); G.ry = 0.5 * (CR.y + CRb.y);
      G.ivol = frcp(0.5 * (V0 + VB));
      auto grad_avg = [&](int k, S* gr, S* avg) {
        S t = at(k, x, yn), b = at(k, x, ys);
        S l = 0.25 * (t + b + at(k, x - 1, yn) + at(k, x - 1, ys));
        S r = 0.25 * (t + b + at(k, x + 1, yn) + at(k, x + 1, ys));
        if (gr) gg_grad(G, t, b, l, r, gr);
        if (avg) *avg = 0.25 * (l + r + t + b);
      };
      S gu[2], gv[2], gT[2], gn[2] = {S(0.0), S(0.0)}, ub, vb, mb, kb, eb(0.0);
      grad_avg(L_U, gu, &ub);
      grad_avg(L_V, gv, &vb);
      grad_avg(L_T, gT, nullptr);
      grad_avg(L_MU, nullptr, &mb);
      grad_avg(L_K, nullptr, &kb);
      if (SA) { grad_avg(L_N, gn, nullptr); grad_avg(L_ETA, nullptr, &eb); }
      S fv[5];
      visc_flux<S, SA>(E0.x, E0.y, gu, gv, gT, ub, vb, mb, kb, gn, eb, fv);
#pragma unroll
      for (int k = 1; k < NV; ++k) he[k] = he[k] - fv[k];
    }
  }

  // ---- SA source of the owned output cell (needs the staged cells)
  const int ci = i0 + tx;
  const bool owns = tx < OX && ty < OY && ci < nic && cj < njc;
  S src(0.0);
  if (SA && ph.viscous) {  // uniform over the block
    const size_t cidx = (size_t)cj * g.ldi + ci;
    SaTerms<S> st{S(0.0), S(0.0), S(0.0)};
    S feat[kNFeat];
    if (owns) {
      const int x = tx + 2, y = ty + 2;
      const double iV = frcp(V0);
      auto cgrad = [&](int k, S* o) {
        S c = at(k, x, y);
        S fe = 0.5 * (c + at(k, x + 1, y)), fw = 0.5 * (c + at(k, x - 1, y));
        S fn = 0.5 * (c + at(k, x, y + 1)), fs = 0.5 * (c + at(k, x, y - 1));
        o[0] = (fe * CR.x - fw * C0.x + fn * Et.x - fs * E0.x) * iV;
        o[1] = (fe * CR.y - fw * C0.y + fn * Et.y - fs * E0.y) * iV;
      };
      S gu[2], gv[2], gn[2], gr[2];
      cgrad(L_U, gu); cgrad(L_V, gv); cgrad(L_N, gn); cgrad(L_R, gr);
      const S r = at(L_R, x, y), n = at(L_N, x, y), ml = at(L_ML, x, y);
      st = sa_terms<S>(r, n, ml, gu, gv, gn, gr, g.wd[cidx]);
      if (CL != CLOSURE_FIELD || clo.aux) {
        S gp[2];
        cgrad(L_P, gp);
        sa_features<S>(r, at(L_U, x, y), at(L_V, x, y), n, sdiv(ml, r), gu, gv, gp, g.wd[cidx], st.P1, st.D, ph, feat);
      }
    }
    S bcell(1.0);
    if (CL == CLOSURE_FIELD) {
      if (owns) {
        bcell = S(g.beta[cidx]);
        if (beta_dot) bcell = bcell + beta_tangent<S>(beta_dot[cidx]);
      }
    } else if (CL == CLOSURE_ANALYTIC) {
      if (owns) bcell = closure_analytic<S>(clo, feat);
    } else {
      float xv[kNFeat], xt[kNFeat];
#pragma unroll
      for (int k = 0; k < kNFeat; ++k) {
        xv[k] = owns ? (float)val(feat[k]) : 0.f;
        xt[k] = owns ? (float)tan_(feat[k]) : 0.f;
      }
      __syncthreads();  // staged cells no longer read: reuse LDS for the hidden layer
      __bf16* hs = reinterpret_cast<__bf16*>(lds_raw) + (tid >> 6) * 64 * kHld;
      __bf16* ht = hs + (NT / 64) * 64 * kHld;
      float y, yt;
      mlp_wave<TAN>(clo.params, reinterpret_cast<const __bf16*>(clo.w2), xv, xt, hs, ht, y, yt);
      bcell = S(1.0 + (double)y);
      if (TAN) bcell = bcell + beta_tangent<S>((double)yt);
    }
    if (owns) {
      src = bcell * st.P1 - st.D + st.rest;
      if (clo.aux) {
#pragma unroll
        for (int k = 0; k < kNFeat; ++k) clo.aux[k * g.plane + cidx] = val(feat[k]);
        clo.aux[kNFeat * g.plane + cidx] = val(bcell);
      }
    }
  }

  // ---- exchange face fluxes through LDS (reusing the staging area)
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    lds[k * NT + tid] = hc[k];
    lds[(NV + k) * NT + tid] = he[k];
  }
  __syncthreads();

  double sq[2 * NV];  // R^2 (reference norm) and (V R)^2 (flux-balance norm)
  S res[NV];
  const size_t oidx = (size_t)cj * g.ldi + ci;
#pragma unroll
  for (int k = 0; k < 2 * NV; ++k) sq[k] = 0.0;
  if (owns) {
    const double V = V0, iV = frcp(V);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      S hw = lds[k * NT + tid], hE = lds[k * NT + tid + 1];
      S hs = lds[(NV + k) * NT + tid], hn = lds[(NV + k) * NT + tid + TX];
      S r = S(0.0) - (hn - hs);
      r = r - (hE - hw);
      if (k == 1) r = r + (-ph.dpdx * V);
      if (k == 2) r = r + (-ph.dpdy * V);
      if (SA && k == 4) r = r + V * src;
      r = r * iV;
      res[k] = r;
      sq[k] = val(r) * val(r);
      sq[NV + k] = sq[k] * V * V;
    }
  }
  if (owns) {
    out.template put<NV>(g.plane, oidx, ci, cj, res);
  }
  // ---- the tile's sums of R^2, in a fixed order: 16 threads per norm add 16
  // values each from LDS, then one another's by DPP (a wavefront sum per norm,
  // 18 instructions each, was 5% of the kernel's)
  if (nout.slots) {
    constexpr int LD = NT + 16;  // a norm's row: 16 doubles on, so that four rows read different banks
    double* sums = lds_raw;
    const int nsum = nout.count;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2 * NV; ++k)
      if (k < nsum) sums[k * LD + tid] = sq[k];
    __syncthreads();
    const int k = tid >> 4, l = tid & 15;
    if (k < nsum) {
      double a = 0.0;
#pragma unroll
      for (int m = 0; m < NT / 16; ++m) a += sums[k * LD + m * 16 + l];
      a = row_sum(a);
      if (l == 0)
        slot_store(nout.slots + (size_t)k * ntile + bid, (unsigned long long)__double_as_longlong(a));
    }
  }
}

}  // namespace sg
