// sd2d_adj.hpp - device kernels of the adjoint (vector-Jacobian product)
// of the residual evaluation and of the wall-drag objective.
//
// For a residual evaluation R(Q; c_h, free stream) on the inviscid path
// (compresid.f90:1-80 with the fluxes of compflux.f90:35-104,
// interfaceflux_all.f90:1-112, cyclocflux_all.f90:1-112, bcflux.f90:1-377)
// and a cotangent Rbar, the kernels accumulate
//   Qbar += (dR/dQ)^T Rbar,  and the partial sums of
//   c_hbar = (dR/dc_h)^T Rbar and pbar = (dR/d free stream)^T Rbar.
// adj_stage_kernel does the whole reverse sweep of one evaluation in one pass
// over the tiles, written by hand over the structure of the forward kernel:
//   - per solution point, resid = -(dF/dxi + dG/deta)/J - Powell(divB) -
//     alpha psi reversed: the cotangent of the flux derivatives
//     Dbar = -Rbar/J, that of the divB weight wbar = (dR/d divB)^T Rbar / J,
//     and the direct (pointwise) part of Qbar;
//   - per grid line and flux point, the cotangent of the flux there
//     (Mmat^T Dbar along the line) through the transposed Jacobian of the
//     interior flux, of the Rusanov flux at faces (with the neighbour's own
//     cotangent of the same face flux, formed from its line, so each cell
//     updates only its own Qbar) or of the boundary flux with its ghost
//     state; the divB weights of the averaged face states likewise; the
//     trace cotangents go back to the line's points through Lmat^T.
// With Rbar = rscale * (cotangent of the stage's output) it is also the
// reverse of the Runge-Kutta stage Qout = cin Qin + ca Qaux + b dt R(Qin).
// The running maxima behind c_h are differentiated by adj_tail_kernel with
// the forward's physics on dual numbers (sd2d_dual.hpp), one input direction
// per lane.  The AV sensor does not act on the state and has no adjoint.
#pragma once
#include "sd2d_dual.hpp"
#include "sd2d_stage.hpp"

namespace sd2d {

struct AdjArgs {
  const double *q;         // state the residual is taken of (tile layout)
  const double *rbar;      // cotangent of the stage's output (tile layout)
  double rscale;           // that of the residual is rscale * rbar
  double cin, ca;          // qbar gets cin * rbar besides, abar ca * rbar
  const double *divb;      // divB of q per solution point [tile][p][ci]
  const double *met;
  int mcomp;               // as StageArgs
  const int *ftab;
  const int *tinfo;        // per tile: member << 6 | TI_FIRST | valid cells
  const Phys *phm;         // free stream
  const unsigned long long *gm;   // the maxima that the evaluation's c_h came from (a set)
  double *qbar, *abar;     // cotangents of Qin and Qaux (abar may be null)
  int qadd, aadd;          // add to what they hold (else overwrite it)
  double *part;            // per tile: c_hbar, pbar[6] (rinf pinf uinf vinf bx by)
  double alpha;
  int ntile;
};

constexpr int ADJ_NPART = 7;

// LDS (in doubles): the tile's state and Rbar (qo layout), after the line
// sweeps the cotangents the families hand each other (variables 0-3 for the
// xi-lines, 4-8 for the eta-lines), and the reduction slots.
template <int N> struct AdjLds {
  static constexpr int T = Geo<N>::CPW, N2 = N * N;
  static constexpr int Q0 = 0, R0 = 9 * N2 * T;
  static constexpr int XA = 0, XB = 5 * N2 * T;
  static constexpr int RED = 18 * N2 * T;
  static constexpr int TOTAL = RED + ADJ_NPART * (STAGE_THREADS / 64);
};

// The operators copied to LDS, where the reverse sweeps index their rows
// with run-time flux-point numbers.
template <int OFF>
__device__ __forceinline__ const Ops &ops_to_lds(double *lds, const Ops &ops) {
  Ops *o = reinterpret_cast<Ops *>(lds + OFF);
  const double *src = reinterpret_cast<const double *>(&ops);
  for (int i = threadIdx.x; i < (int)(sizeof(Ops) / sizeof(double)); i += blockDim.x)
    reinterpret_cast<double *>(o)[i] = src[i];
  __syncthreads();
  return *o;
}

template <int N>
constexpr size_t adj_lds_bytes() { return sizeof(double) * AdjLds<N>::TOTAL; }

// Trace of the 9 variables along the line through point p0 (stride ps) of
// the slot `base` = tile * QT + ci (the face-table encoding) of the
// state-layout array q.
template <int N>
__device__ __forceinline__ void adj_trace(const double *q, int base, int p0, int ps,
                                          const double *Lr, double *t) {
  constexpr int QT = Geo<N>::QT;
  const int nt = base / QT, ci = base - nt * QT;
  const double *qt = q + (size_t)nt * QT;
#pragma unroll
  for (int v = 0; v < 9; ++v) {
    double vals[N];
#pragma unroll
    for (int s = 0; s < N; ++s) vals[s] = qt[qo<N>(v, p0 + ps * s, ci)];
    t[v] = line_trace<N, double>(vals, Lr);
  }
}

// ---- reverse sweeps of the pointwise fluxes (FP64) -------------------------------
// With Fb the cotangent of a flux, these accumulate (dF/dq)^T Fb and
// (dF/dc_h)^T Fb, the forward values being formed as iflux_n / rusanov
// form them.  Derivatives of |x| take the sign of x (+1 at 0), of sqrt(x)
// 1/(2 sqrt(x)), as the dual numbers of sd2d_dual.hpp do; the running
// maxima outputs are not differentiated here (adj_tail_kernel).

// iflux_n (getrusanov.f90:127-193 contracted with (sx, sy))
__device__ __forceinline__ void iflux_n_vjp(const double *q, double c_h, double sx, double sy,
                                            const double *Fb, double *qb, double &chb) {
  constexpr double g1 = GAM - 1.0;
  const double rho = q[0], rhou = q[1], rhov = q[2], rhow = q[3], rhoE = q[4];
  const double Bx = q[5], By = q[6], Bz = q[7], psi = q[8];
  const double ri = rcp(rho);
  const double u = rhou * ri, v = rhov * ri, w = rhow * ri;
  const double B2 = Bx * Bx + By * By + Bz * Bz;
  const double pr = g1 * (rhoE - 0.5 * (rhou * u + rhov * v + rhow * w) - 0.5 * B2 - 0.5 * psi * psi);
  const double pt = pr + 0.5 * B2;
  const double uB = u * Bx + v * By + w * Bz;
  const double ef = rhoE - 0.5 * psi * psi + pt;
  const double un = u * sx + v * sy;
  const double bn = Bx * sx + By * sy;
  const double cp = c_h * psi;
  // the nine outputs (iflux_n), backwards
  double rhob = 0.0, rhoub = Fb[0] * sx + Fb[1] * un, rhovb = Fb[0] * sy + Fb[2] * un;
  double rhowb = Fb[3] * un, rhoEb = 0.0, psib = 0.0;
  double Bxb = -Fb[1] * bn, Byb = -Fb[2] * bn, Bzb = -Fb[3] * bn + Fb[7] * un;
  double ub = 0.0, vb = 0.0, wb = -Fb[7] * bn;
  double unb = Fb[1] * rhou + Fb[2] * rhov + Fb[3] * rhow + Fb[4] * ef + Fb[7] * Bz;
  double ptb = Fb[1] * sx + Fb[2] * sy;
  double bnb = -Fb[1] * Bx - Fb[2] * By - Fb[3] * Bz + Fb[4] * (cp - uB) - Fb[7] * w + Fb[8] * c_h;
  const double efb = Fb[4] * un;
  const double uBb = -Fb[4] * bn;
  const double cpb = Fb[4] * bn + Fb[5] * sx + Fb[6] * sy;
  const double xb = Fb[5] * sy - Fb[6] * sx;        // x = v*Bx - u*By
  double ch = Fb[8] * bn;
  // intermediates, backwards
  vb += xb * Bx; Bxb += xb * v; ub -= xb * By; Byb -= xb * u;
  ch += cpb * psi; psib += cpb * c_h;
  Bxb += bnb * sx; Byb += bnb * sy;
  ub += unb * sx; vb += unb * sy;
  rhoEb += efb; psib -= efb * psi; ptb += efb;
  ub += uBb * Bx; Bxb += uBb * u; vb += uBb * By; Byb += uBb * v; wb += uBb * Bz; Bzb += uBb * w;
  const double prb = ptb;
  double B2b = 0.5 * ptb;
  rhoEb += g1 * prb;
  rhoub -= 0.5 * g1 * prb * u; ub -= 0.5 * g1 * prb * rhou;
  rhovb -= 0.5 * g1 * prb * v; vb -= 0.5 * g1 * prb * rhov;
  rhowb -= 0.5 * g1 * prb * w; wb -= 0.5 * g1 * prb * rhow;
  B2b -= 0.5 * g1 * prb; psib -= g1 * prb * psi;
  Bxb += 2.0 * Bx * B2b; Byb += 2.0 * By * B2b; Bzb += 2.0 * Bz * B2b;
  rhoub += ub * ri; rhovb += vb * ri; rhowb += wb * ri;
  rhob -= (ub * rhou + vb * rhov + wb * rhow) * ri * ri;
  qb[0] = rhob; qb[1] = rhoub; qb[2] = rhovb; qb[3] = rhowb; qb[4] = rhoEb;
  qb[5] = Bxb; qb[6] = Byb; qb[7] = Bzb; qb[8] = psib;
  chb += ch;
}

// one side's physical flux of rusanov (Fl or Fr) backwards, with Fb its
// cotangent and pgb / Vnb the cotangents its gas pressure and normal
// velocity receive from the wave speed; accumulates into Qb and chb
__device__ __forceinline__ void rusanov_side_vjp(const double *Q, double ux, double uy, double c_h,
                                                 const double *Fb, double pgb, double Vnb,
                                                 double *Qb, double &chb) {
  constexpr double g1 = GAM - 1.0;
  const double ri = rcp(Q[0]);
  const double u = ri * Q[1], v = ri * Q[2], w = ri * Q[3];
  const double B2 = Q[5] * Q[5] + Q[6] * Q[6] + Q[7] * Q[7];
  const double pg = g1 * (Q[4] - 0.5 * Q[0] * (u * u + v * v + w * w) - B2 * 0.5 - 0.5 * Q[8] * Q[8]);
  const double pt = pg + 0.5 * B2;
  const double Vn = u * ux + v * uy;
  const double Bn = Q[5] * ux + Q[6] * uy;
  const double e = Q[4] - 0.5 * Q[8] * Q[8] + pt;
  const double uB = u * Q[5] + v * Q[6] + w * Q[7];
  Vnb += Fb[0] * Q[0] + Fb[1] * Q[1] + Fb[2] * Q[2] + Fb[3] * Q[3] + Fb[4] * e + Fb[7] * Q[7];
  Qb[0] += Fb[0] * Vn; Qb[1] += Fb[1] * Vn; Qb[2] += Fb[2] * Vn; Qb[3] += Fb[3] * Vn;
  Qb[7] += Fb[7] * Vn;
  double ptb = Fb[1] * ux + Fb[2] * uy;
  const double eb = Fb[4] * Vn;
  Qb[4] += eb; Qb[8] -= eb * Q[8]; ptb += eb;
  const double Bnb = -Fb[1] * Q[5] - Fb[2] * Q[6] - Fb[3] * Q[7] - Fb[4] * uB + Fb[4] * c_h * Q[8] -
                     Fb[7] * w + Fb[8] * c_h;
  Qb[5] -= Fb[1] * Bn; Qb[6] -= Fb[2] * Bn; Qb[7] -= Fb[3] * Bn;
  const double uBb = -Fb[4] * Bn;
  chb += Fb[4] * Q[8] * Bn + Fb[5] * Q[8] * ux + Fb[6] * Q[8] * uy + Fb[8] * Bn;
  Qb[8] += Fb[4] * c_h * Bn + Fb[5] * c_h * ux + Fb[6] * c_h * uy;
  const double xb = Fb[5] * uy - Fb[6] * ux;        // x = v*Q5 - u*Q6
  double ub = 0.0, vb = 0.0, wb = -Fb[7] * Bn;
  vb += xb * Q[5]; Qb[5] += xb * v; ub -= xb * Q[6]; Qb[6] -= xb * u;
  ub += uBb * Q[5]; Qb[5] += uBb * u; vb += uBb * Q[6]; Qb[6] += uBb * v;
  wb += uBb * Q[7]; Qb[7] += uBb * w;
  Qb[5] += Bnb * ux; Qb[6] += Bnb * uy;
  ub += Vnb * ux; vb += Vnb * uy;
  pgb += ptb;
  double B2b = 0.5 * ptb;
  Qb[4] += g1 * pgb;
  Qb[0] -= 0.5 * g1 * pgb * (u * u + v * v + w * w);
  ub -= g1 * pgb * Q[0] * u; vb -= g1 * pgb * Q[0] * v; wb -= g1 * pgb * Q[0] * w;
  B2b -= 0.5 * g1 * pgb; Qb[8] -= g1 * pgb * Q[8];
  Qb[5] += 2.0 * Q[5] * B2b; Qb[6] += 2.0 * Q[6] * B2b; Qb[7] += 2.0 * Q[7] * B2b;
  Qb[1] += ub * ri; Qb[2] += vb * ri; Qb[3] += wb * ri;
  Qb[0] -= (ub * Q[1] + vb * Q[2] + wb * Q[3]) * ri * ri;
}

// rusanov (getrusanov.f90:1-125): Fn = sc (Fl + Fr - ev (QR - QL)) with the
// fast magneto-acoustic speed ev of the averaged state.  The cotangent of
// one side, or with BOTH of both: Qa is the side wanted (the left state when
// aleft), Qb the other; Fnb is the cotangent of Fn.  chb receives the c_h
// part of the sides that are formed.
template <bool BOTH>
__device__ __forceinline__ void rusanov_vjp(const double *Qa, const double *Qb, bool aleft,
                                            double nx, double ny, int sign_l, double c_h,
                                            const double *Fnb, double *Qab, double *Qbb,
                                            double &chb) {
  constexpr double g1 = GAM - 1.0;
  const double mag = sqrt(nx * nx + ny * ny);
  const double im = double(sign_l) * rcp(mag);
  const double ux = nx * im, uy = ny * im;
  const double ria = rcp(Qa[0]), rib = rcp(Qb[0]);
  const double ua = ria * Qa[1], va = ria * Qa[2], wa = ria * Qa[3];
  const double ub = rib * Qb[1], vb = rib * Qb[2], wb = rib * Qb[3];
  const double B2a = Qa[5] * Qa[5] + Qa[6] * Qa[6] + Qa[7] * Qa[7];
  const double B2b = Qb[5] * Qb[5] + Qb[6] * Qb[6] + Qb[7] * Qb[7];
  const double pga = g1 * (Qa[4] - 0.5 * Qa[0] * (ua * ua + va * va + wa * wa) - B2a * 0.5 -
                           0.5 * Qa[8] * Qa[8]);
  const double pgb = g1 * (Qb[4] - 0.5 * Qb[0] * (ub * ub + vb * vb + wb * wb) - B2b * 0.5 -
                           0.5 * Qb[8] * Qb[8]);
  const double sV = (ua * ux + va * uy) + (ub * ux + vb * uy);
  const double bx = 0.5 * (Qa[5] + Qb[5]), by = 0.5 * (Qa[6] + Qb[6]), bz = 0.5 * (Qa[7] + Qb[7]);
  const double irs = rcp(Qa[0] + Qb[0]);
  const double ca = GAM * (pga + pgb) * irs;
  const double bb = bx * bx + by * by + bz * bz;
  const double cd = 2.0 * bb * irs;
  const double bn = bx * ux + by * uy;
  const double cn = 2.0 * bn * bn * irs;
  const double cad = ca + cd;
  const double ct = sqrt(cad * cad - 4.0 * ca * cn);
  const double cf = sqrt(0.5 * (cad + ct));
  const double ev = 0.5 * fabs(sV) + cf;
  const double sc = 0.5 * mag * double(sign_l);
  // QR - QL is sg (Qb - Qa)
  const double sg = aleft ? 1.0 : -1.0;
  double G[9], evb = 0.0;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    G[k] = sc * Fnb[k];
    evb -= G[k] * (Qb[k] - Qa[k]);
    Qab[k] = sg * G[k] * ev;
    if (BOTH) Qbb[k] = -sg * G[k] * ev;
  }
  evb *= sg;
  // ev = |Vn_l + Vn_r|/2 + cf, cf = sqrt((cad + ct)/2), ct = sqrt(cad^2 - 4 ca cn)
  const double sb = 0.5 * (sV < 0.0 ? -evb : evb);
  const double yb = 0.5 * evb * rcp(cf);
  double cadb = 0.5 * yb;
  const double ctb = 0.5 * yb;
  const double zb = ctb / (2.0 * ct);
  cadb += 2.0 * cad * zb;
  const double cab = -4.0 * cn * zb + cadb;
  const double cnb = -4.0 * ca * zb;
  const double cdb = cadb;
  const double bnb = 4.0 * bn * irs * cnb;
  const double irsb = 2.0 * bn * bn * cnb + 2.0 * bb * cdb + GAM * (pga + pgb) * cab;
  const double h5 = 0.5 * (bnb * ux + 4.0 * bx * irs * cdb);
  const double h6 = 0.5 * (bnb * uy + 4.0 * by * irs * cdb);
  const double h7 = 0.5 * (4.0 * bz * irs * cdb);
  const double pb = GAM * irs * cab;
  const double d0 = -irs * irs * irsb;
  Qab[0] += d0; Qab[5] += h5; Qab[6] += h6; Qab[7] += h7;
  rusanov_side_vjp(Qa, ux, uy, c_h, G, pb, sb, Qab, chb);
  if (BOTH) {
    Qbb[0] += d0; Qbb[5] += h5; Qbb[6] += h6; Qbb[7] += h7;
    rusanov_side_vjp(Qb, ux, uy, c_h, G, pb, sb, Qbb, chb);
  }
}

// The ghost state of a boundary face (bc_ghost_p with vismode 1) backwards:
// the ghost's cotangent gb goes to the own trace t (added to ob) and to the
// free stream pb[6] (rinf pinf uinf vinf bx by).
__device__ __forceinline__ void bc_ghost_vjp(int bc, const double *t, double nx, double ny,
                                             const Phys &ph, const double *gb, double *ob,
                                             double *pb) {
  constexpr double ig1 = 1.0 / (GAM - 1.0);
  const double ri = rcp(t[0]);
  const double uw = t[1] * ri, vw = t[2] * ri, ww = t[3] * ri;
  if (bc == FT_INLE) {
    pb[0] += gb[0] + gb[1] * ph.uinf + gb[2] * ph.vinf +
             gb[4] * 0.5 * (ph.uinf * ph.uinf + ph.vinf * ph.vinf);
    pb[2] += ph.rinf * (gb[1] + gb[4] * ph.uinf);
    pb[3] += ph.rinf * (gb[2] + gb[4] * ph.vinf);
    ob[8] += gb[8] + gb[4] * t[8];
  } else if (bc == FT_OUTL) {
    ob[0] += gb[0] - gb[4] * 0.5 * (uw * uw + vw * vw);
    ob[1] += gb[1] + gb[4] * uw;
    ob[2] += gb[2] + gb[4] * vw;
    ob[8] += gb[4] * t[8];
  } else if (bc == FT_WALL) {
    ob[0] += gb[0]; ob[1] -= gb[1]; ob[2] -= gb[2]; ob[3] -= gb[3]; ob[4] += gb[4];
    ob[5] -= gb[5]; ob[6] -= gb[6]; ob[7] -= gb[7]; ob[8] += gb[8];
  } else if (bc == FT_SYMP) {
    const double im = rcp(sqrt(nx * nx + ny * ny)), ex = nx * im, ey = ny * im;
    const double vn = uw * ex + vw * ey;
    const double ur = uw - 2.0 * vn * ex, vr = vw - 2.0 * vn * ey;
    const double rs = 2.0 * ph.rinf - t[0];
    // ghost momenta rs (ur, vr, -ww) and energy with |m|^2 / (2 rs)
    const double m1 = gb[1] + gb[4] * ur, m2 = gb[2] + gb[4] * vr, m3 = gb[3] - gb[4] * ww;
    const double rsb = gb[0] - 0.5 * gb[4] * (ur * ur + vr * vr + ww * ww) + m1 * ur + m2 * vr -
                       m3 * ww;
    const double urb = m1 * rs, vrb = m2 * rs, wwb = -m3 * rs;
    const double nb = 2.0 * (urb * ex + vrb * ey);   // the reflection is symmetric
    const double uwb = urb - nb * ex, vwb = vrb - nb * ey;
    ob[0] += -rsb - (uwb * uw + vwb * vw + wwb * ww) * ri;
    ob[1] += uwb * ri;
    ob[2] += vwb * ri;
    ob[3] += wwb * ri;
    ob[7] += gb[4] * t[7] - gb[7];
    ob[8] += gb[8] + gb[4] * t[8];
    pb[0] += 2.0 * rsb;
  } else {   // FREE
#pragma unroll
    for (int v = 0; v < 9; ++v) ob[v] += gb[v];
  }
  if (bc == FT_INLE || bc == FT_OUTL || bc == FT_SYMP) {
    pb[1] += gb[4] * ig1;
    pb[4] += gb[5] + gb[4] * ph.bxinf;
    pb[5] += gb[6] + gb[4] * ph.byinf;
  }
}

// Cotangent of divB at a point, (dR/d divB)^T rb: the Powell source backwards.
__device__ __forceinline__ double adj_divb_cot(const double *q, const double *rb) {
  const double ri = rcp(q[0]);
  const double ux = q[1] * ri, uy = q[2] * ri, uz = q[3] * ri;
  return -(rb[1] * q[5] + rb[2] * q[6] + rb[3] * q[7] +
           rb[4] * (ux * q[5] + uy * q[6] + uz * q[7]) + rb[5] * ux + rb[6] * uy + rb[7] * uz);
}

// (is, js) of a solution point
template <int N> __device__ __forceinline__ int pt_is(int p) { return p % N; }
template <int N> __device__ __forceinline__ int pt_js(int p) { return p / N; }

// From the line of another cell through a shared face point (points p0 + ps*s
// of slot ci, state q and cotangent r in qo layout, 1/J at ji): the state's
// trace t with row Lr, and the cotangents of that cell's flux and divB weight
// there, Mr^T Dbar and Mr^T wbar.
template <int N>
__device__ __forceinline__ void adj_far_line(const double *q, const double *r, const double *ji,
                                             int p0, int ps, int ci, const double *Lr,
                                             const double *Mr, double rscale, double *t,
                                             double *Fb, double &Wb) {
  constexpr int T = Geo<N>::CPW;
#pragma unroll
  for (int v = 0; v < 9; ++v) t[v] = Fb[v] = 0.0;
  Wb = 0.0;
#pragma unroll
  for (int s = 0; s < N; ++s) {
    const int p = p0 + ps * s;
    double a[9], b[9];
    load_vars<N, 0, 9>(q, p, ci, a);
    load_vars<N, 0, 9>(r, p, ci, b);
    const double c = rscale * ji[(pt_js<N>(p) + N * pt_is<N>(p)) * T] * Mr[s];
    Wb = fma(c, adj_divb_cot(a, b), Wb);
#pragma unroll
    for (int v = 0; v < 9; ++v) {
      t[v] = fma(a[v], Lr[s], t[v]);
      Fb[v] = fma(-c, b[v], Fb[v]);
    }
  }
}

// ---- one evaluation backwards ------------------------------------------------
// One 128-thread workgroup per tile, one thread per grid line, one family per
// wavefront, as in the stage kernel.  The state and Rbar of the tile are staged
// in LDS (one wave each); the first end face of a line whose neighbour lies in
// another tile is gathered meanwhile.  Every flux point's trace cotangent is
// folded straight into the line's Qbar accumulators through Lmat^T; then the
// pointwise parts and the Runge-Kutta terms are added (xi-lines variables 0-3,
// eta-lines 4-8) and the families exchange their halves through the staging
// area.
// 256 VGPRs and 26-62 AGPRs (the 9 N accumulators beside the Rusanov sweep),
// so one wave per SIMD; bound by the latency of its loads, then by FP64 issue.
// 128 x 256 cells, N = 4: 79 us.  It replaces a point kernel, a line kernel
// that read every flux point's lines from memory and the RK combinations
// (31 + 150 + 2 x 19 us and a clear of the cotangent).  Held to two waves per
// SIMD it spills (108-284 bytes a lane): 89 us at N = 4, 50 against 47 us at
// N = 5 (64 x 128 cells), 22 against 17 us at N = 3.
template <int N>
__global__ __launch_bounds__(STAGE_THREADS, 1) void adj_stage_kernel(AdjArgs a, Ops ops) {
  using G = Geo<N>;
  using LD = AdjLds<N>;
  constexpr int T = G::CPW, N2 = G::N2, NF = N + 1, QT = G::QT;
  static_assert(N * T <= 64 && STAGE_THREADS == 128, "one wavefront per line family");
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const int tile = tile_of_block(blockIdx.x, a.ntile, 0);
  const int fam = tid >> 6, line = (tid & 63) / T, ci = (tid & 63) % T;
  int nb0, nbN, info0, infoN;
  face_words<N>(a, tile, ci, fam, line, 0, nb0, info0);
  face_words<N>(a, tile, ci, fam, line, N, nbN, infoN);
  const int ti = a.tinfo[tile];
  {   // the xi wave stages the state, the eta wave Rbar
    constexpr int NV2 = QT / 2, NSW = (NV2 + 63) / 64;
    const double2 *src = reinterpret_cast<const double2 *>((fam ? a.rbar : a.q) + (size_t)tile * QT);
    double2 *dst = reinterpret_cast<double2 *>(lds + (fam ? LD::R0 : LD::Q0));
    const int l = tid & 63;
    double2 st[NSW];
#pragma unroll
    for (int k = 0; k < NSW; ++k) {
      const int i = l + k * 64;
      st[k] = src[(k < NSW - 1 || i < NV2) ? i : 0];
    }
#pragma unroll
    for (int k = 0; k < NSW - 1; ++k) dst[l + k * 64] = st[k];
    if (l + (NSW - 1) * 64 < NV2) dst[l + (NSW - 1) * 64] = st[NSW - 1];
  }
  const bool valid = line < N && ci < (ti & TI_VALID);
  const MetLine<N, double> ml(a.met, a.mcomp, tile, ci, fam, line);
  const int p0 = fam ? line : N * line, ps = fam ? N : 1;
  const bool i0 = ((info0 >> 3) & 7) == FT_INTERIOR, iN = ((infoN >> 3) & 7) == FT_INTERIOR;
  const bool far0 = i0 && nb0 / QT != tile, farN = iN && nbN / QT != tile;
  const bool nfirst = farN && !far0;   // the end whose traces are gathered first
  double tn[9], Fn[9], Wn = 0.0;       // neighbour's trace and cotangents at an end
  int sgn = 0;                         // whether its stored normal is the negative
  auto other_side = [&](bool atN, bool staged) __attribute__((always_inline)) {
    const int rfp = atN ? N : 0, nb = atN ? nbN : nb0, info = atN ? infoN : info0;
    const int nt = nb / QT, nci = nb - nt * QT, kn = info & 3;
    int k, nfp, np0, nst;
    bool endN;
    end_face<N>(fam, line, rfp, k, nfp);
    neighbour_line<N>(kn, nfp, np0, nst, endN);
    double Lr[N], Mr[N];
#pragma unroll
    for (int s = 0; s < N; ++s) {
      Lr[s] = endN ? ops.L[N][s] : ops.L[0][s];
      Mr[s] = endN ? ops.M[N][s] : ops.M[0][s];
    }
    const double *ji = MetLine<N, double>(a.met, a.mcomp, nt, nci, 0, 0).ji;
    sgn = a.ftab[((size_t)nt * 8 + kn * 2 + 1) * T + nci];
    if (staged)
      adj_far_line<N>(lds + LD::Q0, lds + LD::R0, ji, np0, nst, nci, Lr, Mr, a.rscale, tn, Fn, Wn);
    else
      adj_far_line<N>(a.q + (size_t)nt * QT, a.rbar + (size_t)nt * QT, ji, np0, nst, nci, Lr, Mr,
                      a.rscale, tn, Fn, Wn);
  };
  double ji[N], msx[NF], msy[NF];
  if (valid) {
    if (far0 || farN) other_side(nfirst, false);
#pragma unroll
    for (int s = 0; s < N; ++s) ji[s] = ml.ji[((fam ? s : line) + N * (fam ? line : s)) * T];
#pragma unroll
    for (int r = 0; r < NF; ++r) {
      msx[r] = ml.x[r * T];
      msy[r] = ml.y[r * T];
    }
  }
  double ge, gu;
  set_pair(a.gm, ge, gu);
  const double c_h = sqrt(ge * (ge - gu));   // as the forward forms it (compflux.f90:6)
  const Phys &ph = a.phm[0];
  double chb = 0.0, pb[6] = {0, 0, 0, 0, 0, 0};
  __syncthreads();
  double A[N][9];   // the line's part of Qbar at its points
  const double *qs = lds + LD::Q0, *rs = lds + LD::R0;
  if (valid) {
    double c[N], wb[N];   // Dbar = c * rbar and wbar at the line's points
#pragma unroll
    for (int s = 0; s < N; ++s) {
      double q[9], b[9];
      load_vars<N, 0, 9>(qs, p0 + ps * s, ci, q);
      load_vars<N, 0, 9>(rs, p0 + ps * s, ci, b);
      c[s] = -a.rscale * ji[s];
      wb[s] = -c[s] * adj_divb_cot(q, b);
    }
    // trace, flux cotangent and divB-weight cotangent at a flux point
    auto point = [&](const double *Lr, const double *Mr, double *t, double *Fb, double &Wb) __attribute__((always_inline)) {
      double m[N];
      Wb = 0.0;
#pragma unroll
      for (int s = 0; s < N; ++s) {
        m[s] = Mr[s] * c[s];
        Wb = fma(Mr[s], wb[s], Wb);
      }
      line_vals<N, double>(qs, p0, ps, ci, [&](int v, const double *x) {
        t[v] = line_trace<N, double>(x, Lr);
      });
      line_vals<N, double>(rs, p0, ps, ci, [&](int v, const double *x) {
        Fb[v] = line_trace<N, double>(x, m);
      });
    };
    auto end_point = [&](bool atN, bool gathered, double *Qt) __attribute__((always_inline)) {
      const int info = atN ? infoN : info0;
      const int k = fam == 0 ? (atN ? 1 : 3) : (atN ? 2 : 0);
      const bool inter = atN ? iN : i0, far = atN ? farN : far0;
      const double sx = atN ? msx[N] : msx[0], sy = atN ? msy[N] : msy[0];
      if (inter && !far) other_side(atN, true);
      else if (far && !gathered) other_side(atN, false);
      double Lo[N], Mo[N], t[9], Fb[9], Wb;
#pragma unroll
      for (int s = 0; s < N; ++s) {
        Lo[s] = atN ? ops.L[N][s] : ops.L[0][s];
        Mo[s] = atN ? ops.M[N][s] : ops.M[0][s];
      }
      point(Lo, Mo, t, Fb, Wb);
      const int own_sl = (k == 0 || k == 3) ? -1 : 1;
      if (inter) {
        // the face as interfaceflux / CYCLOCFLUX evaluate it, with the
        // neighbour's cotangent of its own copy of the face flux
        const int kn = info & 3, left = (info >> 2) & 1, sneg = (info >> 6) & 1;
        const int sl = left ? own_sl : ((kn == 0 || kn == 3) ? -1 : 1);
        const int sr = left ? ((kn == 1 || kn == 2) ? -1 : 1) : ((k == 1 || k == 2) ? -1 : 1);
        const double nsg = (left || !sneg) ? 1.0 : -1.0;
        const double fo = left ? 1.0 : double(sl * sr), fn = left ? double(sl * sr) : 1.0;
        // the neighbour's own metric at the point is sig times this cell's
        const double sig = (left ? (sgn >> 6) & 1 : sneg) ? -1.0 : 1.0;
        const double wq = 0.5 * (Wb + sig * Wn);
#pragma unroll
        for (int v = 0; v < 9; ++v) Fb[v] = fo * Fb[v] + fn * Fn[v];
        rusanov_vjp<false>(t, tn, left, nsg * sx, nsg * sy, sl, c_h, Fb, Qt, nullptr, chb);
        // divB weights of the averaged state (QL + QR)/2 seen by both cells
        Qt[5] += wq * sx;
        Qt[6] += wq * sy;
      } else {
        const int bc = (info >> 3) & 7;
        double g[9], gb[9];
        bc_ghost<double>(bc, t, sx, sy, ph, g);
        rusanov_vjp<true>(t, g, true, sx, sy, own_sl, c_h, Fb, Qt, gb, chb);
        const double hx = 0.5 * Wb * sx, hy = 0.5 * Wb * sy;
        Qt[5] += hx; Qt[6] += hy;
        gb[5] += hx; gb[6] += hy;
        bc_ghost_vjp(bc, t, sx, sy, ph, gb, Qt, pb);
      }
    };
    {
      double QA[9], QB[9];
      end_point(nfirst, true, QA);
      __builtin_amdgcn_sched_barrier(0);
      end_point(!nfirst, false, QB);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < N; ++s) {
        const double LA = nfirst ? ops.L[N][s] : ops.L[0][s], LB = nfirst ? ops.L[0][s] : ops.L[N][s];
#pragma unroll
        for (int v = 0; v < 9; ++v) A[s][v] = fma(QB[v], LB, QA[v] * LA);
      }
    }
    // interior flux points (compflux.f90:53-104) and the divB weight of the trace
#pragma unroll
    for (int r = 1; r < N; ++r) {
      double t[9], Fb[9], Wb, Qt[9];
      point(ops.L[r], ops.M[r], t, Fb, Wb);
      iflux_n_vjp(t, c_h, msx[r], msy[r], Fb, Qt, chb);
      Qt[5] = fma(Wb, msx[r], Qt[5]);
      Qt[6] = fma(Wb, msy[r], Qt[6]);
#pragma unroll
      for (int s = 0; s < N; ++s)
#pragma unroll
        for (int v = 0; v < 9; ++v) A[s][v] = fma(Qt[v], ops.L[r][s], A[s][v]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the points' direct part (Powell source and GLM damping), cin * rbar, and
    // the auxiliary register's cotangent, for the variables this family finishes
    const double *dv = a.divb + (size_t)tile * N2 * T + ci;
    auto direct = [&](auto v0c, auto v1c) __attribute__((always_inline)) {
      constexpr int V0 = decltype(v0c)::value, V1 = decltype(v1c)::value;
#pragma unroll
      for (int s = 0; s < N; ++s) {
        const int p = p0 + ps * s;
        double q[9], b[9], d[9];
        load_vars<N, 0, 8>(qs, p, ci, q);
        load_vars<N, 0, 9>(rs, p, ci, b);
        const double w = -a.rscale * dv[p * T];   // the residual's cotangent is rscale * b
        const double ri = rcp(q[0]);
        const double ux = q[1] * ri, uy = q[2] * ri, uz = q[3] * ri;
        const double ubx = w * (b[4] * q[5] + b[5]), uby = w * (b[4] * q[6] + b[6]),
                     ubz = w * (b[4] * q[7] + b[7]);
        d[0] = -(ubx * ux + uby * uy + ubz * uz) * ri;
        d[1] = ubx * ri;
        d[2] = uby * ri;
        d[3] = ubz * ri;
        d[4] = 0.0;
        d[5] = w * (b[1] + b[4] * ux);
        d[6] = w * (b[2] + b[4] * uy);
        d[7] = w * (b[3] + b[4] * uz);
        d[8] = -a.alpha * a.rscale * b[8];
#pragma unroll
        for (int v = V0; v < V1; ++v) A[s][v] += d[v] + a.cin * b[v];
        if (a.abar) {
          double *ab = a.abar + (size_t)tile * QT;
          double x[V1 - V0];
          if (a.aadd) {
            load_vars<N, V0, V1>(ab, p, ci, x);
#pragma unroll
            for (int v = V0; v < V1; ++v) x[v - V0] = fma(a.ca, b[v], x[v - V0]);
          } else {
#pragma unroll
            for (int v = V0; v < V1; ++v) x[v - V0] = a.ca * b[v];
          }
          store_vars<N, V0, V1>(ab, p, ci, x);
        }
      }
    };
    if (fam == 0) direct(std::integral_constant<int, 0>{}, std::integral_constant<int, 4>{});
    else direct(std::integral_constant<int, 4>{}, std::integral_constant<int, 9>{});
  }
  {   // partial sums of the block
    const int w = tid >> 6, l = tid & 63;
    double x[ADJ_NPART] = {chb, pb[0], pb[1], pb[2], pb[3], pb[4], pb[5]};
#pragma unroll
    for (int j = 0; j < ADJ_NPART; ++j) {
      x[j] = wave_sum(x[j]);
      if (l == 0) lds[LD::RED + j * (STAGE_THREADS / 64) + w] = x[j];
    }
  }
  __syncthreads();   // every read of the staged tile is done
  if (tid < ADJ_NPART)
    a.part[(size_t)tile * ADJ_NPART + tid] = lds[LD::RED + 2 * tid] + lds[LD::RED + 2 * tid + 1];
  if (valid) {
#pragma unroll
    for (int s = 0; s < N; ++s) {
      if (fam) xput<N, 4>(lds + LD::XA, p0 + ps * s, ci, A[s]);
      else xput<N, 5>(lds + LD::XB, p0 + ps * s, ci, A[s] + 4);
    }
  }
  __syncthreads();
  if (!valid) return;
  double *qb = a.qbar + (size_t)tile * QT;
  auto finish = [&](auto v0c, auto v1c) __attribute__((always_inline)) {
    constexpr int V0 = decltype(v0c)::value, V1 = decltype(v1c)::value;
#pragma unroll
    for (int s = 0; s < N; ++s) {
      const int p = p0 + ps * s;
      xadd<N, V1 - V0>(lds + (fam ? LD::XB : LD::XA), p, ci, A[s] + V0);
      if (a.qadd) {
        double x[V1 - V0];
        load_vars<N, V0, V1>(qb, p, ci, x);
#pragma unroll
        for (int v = V0; v < V1; ++v) A[s][v] += x[v - V0];
      }
      store_vars<N, V0, V1>(qb, p, ci, A[s] + V0);
    }
  };
  if (fam == 0) finish(std::integral_constant<int, 0>{}, std::integral_constant<int, 4>{});
  else finish(std::integral_constant<int, 4>{}, std::integral_constant<int, 9>{});
}

// ---- wall drag ------------------------------------------------------------------
// D = sum over WALL faces and their N points of w_i * p * (outward S)_x,
// p = (gamma-1)(E - |m|^2/(2 rho) - |B|^2/2 - psi^2/2) of the cell's own
// trace, S the cell's metric vector at the point (S1(1,:) or S2(2,:),
// whose length is the face's arc length per unit reference coordinate),
// signed outwards, and w_i the weights of the interpolatory quadrature on
// the solution-point positions Xs of the face.  One wave per tile, one lane
// per line of a cell, the four faces one after the other: the drag per tile,
// and with qbar set, Qbar += scale * dD/dQ (the lines of one face share no
// point; a cell's next wall face comes after the barrier).
template <int N>
__global__ __launch_bounds__(64) void drag_kernel(const double *q, const int *ftab,
                                                  const double *met, int mcomp, const double *wq, Ops ops,
                                                  double *dtile, double *qbar, double scale) {
  using G = Geo<N>;
  constexpr int T = G::CPW, NF = N + 1;
  static_assert(N * T <= 64, "one lane per line");
  const int tile = blockIdx.x, line = threadIdx.x / T, ci = threadIdx.x % T;
  const bool on = line < N;
  double d = 0.0;
  int bc[4];
  bool any = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) {   // (a padding slot has no wall face)
    const int info = ftab[((size_t)tile * 8 + k * 2 + 1) * T + ci];
    bc[k] = (info >> 3) & 7;
    any |= bc[k] == FT_WALL;
  }
  if (__syncthreads_or(any)) {
    const double *qc = q + (size_t)tile * G::QT;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (on && bc[k] == FT_WALL) {
        // the face's points: own lines of the family crossing it
        const int fam = (k == 1 || k == 3) ? 0 : 1;
        const int rfp = (k == 0 || k == 3) ? 0 : N;
        const double sgn = (k == 0 || k == 3) ? -1.0 : 1.0;
        const MetLine<N, double> ml(met, mcomp, tile, ci, fam, line);
        const int p0 = fam ? line : N * line, ps = fam ? N : 1;
        double t[9];
        line_vals<N, double>(qc, p0, ps, ci, [&](int v, const double *x) {
          t[v] = line_trace<N, double>(x, ops.L[rfp]);
        });
        const double g1 = GAM - 1.0;
        const double ke = 0.5 * (t[1] * t[1] + t[2] * t[2] + t[3] * t[3]) / t[0];
        const double pr = g1 * (t[4] - ke - 0.5 * (t[5] * t[5] + t[6] * t[6] + t[7] * t[7]) -
                                0.5 * t[8] * t[8]);
        const double nx = sgn * ml.x[rfp * T];
        d += wq[line] * pr * nx;
        if (qbar) {
          const double c = scale * wq[line] * nx * g1;
          const double pt[9] = {c * ke / t[0], -c * t[1] / t[0], -c * t[2] / t[0],
                                -c * t[3] / t[0], c, -c * t[5], -c * t[6], -c * t[7], -c * t[8]};
          double *qb = qbar + (size_t)tile * G::QT;
#pragma unroll
          for (int s = 0; s < N; ++s) {
            double x[9];
            load_vars<N, 0, 9>(qb, p0 + ps * s, ci, x);
#pragma unroll
            for (int v = 0; v < 9; ++v) x[v] += pt[v] * ops.L[rfp][s];
            store_vars<N, 0, 9>(qb, p0 + ps * s, ci, x);
          }
        }
      }
      if (qbar) __syncthreads();
    }
  }
  d = wave_sum(d);
  if (threadIdx.x == 0) dtile[tile] = d;
}

// ---- the running maxima behind c_h -------------------------------------------------
// c_h of an evaluation is formed from the running maxima of eigvmax and
// umax over all earlier evaluations (compflux.f90:6; getrusanov.f90:116-123,
// 184-191).  Where an evaluation raised a maximum, the cotangent of the
// maximum goes to the wave speed of the one flux point that attained it.
// Location code of a flux point: ((slot*2 + fam)*N + line)*(N+1) + rfp.

// wave speed eig (face points) and velocity bound um of flux point r of a
// line, with the forward's arithmetic; T is double or Dual, with the own
// trace t and the neighbour trace qn (interior faces) as inputs
template <int N, typename R>
__device__ __forceinline__ void adj_point_speeds(const AdjArgs &a, int info, int k, int r,
                                                 bool face, double sx, double sy,
                                                 const R *t, const R *qn, R &eig, R &um) {
  eig = R(0.0);
  um = R(0.0);
  if (!face) {
    R F[9];
    iflux_n<R>(t, R(0.0), R(sx), R(sy), F, um);
    return;
  }
  const int bc = (info >> 3) & 7;
  const int own_sl = (k == 0 || k == 3) ? -1 : 1;
  R F[9];
  if (bc == FT_INTERIOR) {
    const int kn = info & 3, left = (info >> 2) & 1, sneg = (info >> 6) & 1;
    R QL[9], QR[9];
#pragma unroll
    for (int v = 0; v < 9; ++v) { QL[v] = left ? t[v] : qn[v]; QR[v] = left ? qn[v] : t[v]; }
    const int sl = left ? own_sl : ((kn == 0 || kn == 3) ? -1 : 1);
    const double nsg = (left || !sneg) ? 1.0 : -1.0;
    rusanov<R>(QL, QR, R(nsg * sx), R(nsg * sy), sl, R(0.0), F, eig, um);
  } else {
    const Phys &ph = a.phm[0];
    R QR[9];
    bc_ghost_p<R>(bc, t, R(sx), R(sy), R(ph.rinf), R(ph.pinf), R(ph.uinf), R(ph.vinf),
                  R(ph.bxinf), R(ph.byinf), ph.vismode, QR);
    rusanov<R>(t, QR, R(sx), R(sy), own_sl, R(0.0), F, eig, um);
  }
}

// the geometry of flux point r of a line: metric, face word and the
// neighbour's line (for a face point of an interior face)
template <int N>
__device__ __forceinline__ void adj_point_geom(const AdjArgs &a, const Ops &ops, int tile, int ci,
                                               int fam, int line, int r, double &sx, double &sy,
                                               int &info, int &k, int &nbase, int &np0, int &nst,
                                               bool &endN) {
  using G = Geo<N>;
  constexpr int T = G::CPW, NF = N + 1;
  const MetLine<N, double> ml(a.met, a.mcomp, tile, ci, fam, line);
  sx = ml.x[r * T];
  sy = ml.y[r * T];
  info = 0; k = 0; nbase = 0; np0 = 0; nst = 1; endN = false;
  if (r != 0 && r != N) return;
  int nfp;
  end_face<N>(fam, line, r, k, nfp);
  const int *ft = a.ftab + ((size_t)tile * 8 + k * 2) * T + ci;
  nbase = ft[0];
  info = ft[T];
  if (((info >> 3) & 7) == FT_INTERIOR) neighbour_line<N>(info & 3, nfp, np0, nst, endN);
}

// Qbar += w * d(speed)/dQ at flux point `loc` (kind 0: eig, 1: um), called by
// one block: lane kk < 9 takes variable kk of the cell's own trace, lane
// 9 + v variable v of the neighbour's, after a barrier (on a one-cell wide
// periodic mesh the two lines may share points).
template <int N>
__device__ __forceinline__ void adj_speed_apply(const AdjArgs &a, const Ops &ops, int loc, int kind,
                                                double w) {
  constexpr int T = Geo<N>::CPW, NF = N + 1, QT = Geo<N>::QT;
  const int kk = threadIdx.x;
  const int r = loc % NF, line = (loc / NF) % N, fam = (loc / (NF * N)) % 2;
  const int slot = loc / (NF * N * 2), tile = slot / T, ci = slot % T;
  const int p0 = fam ? line : N * line, ps = fam ? N : 1;
  double sx, sy;
  int info, k, nbase, np0, nst;
  bool endN;
  adj_point_geom<N>(a, ops, tile, ci, fam, line, r, sx, sy, info, k, nbase, np0, nst, endN);
  const bool face = r == 0 || r == N;
  const bool nbr = face && ((info >> 3) & 7) == FT_INTERIOR;
  const int nbt = nbase / QT, nbc = nbase - nbt * QT;
  double d = 0.0;
  if (kk < (nbr ? 18 : 9)) {
    double Lr[N], Ln[N], t[9], qn[9];
    for (int s = 0; s < N; ++s) {
      Lr[s] = ops.L[r][s];
      Ln[s] = endN ? ops.L[N][s] : ops.L[0][s];
    }
    adj_trace<N>(a.q, tile * QT + ci, p0, ps, Lr, t);
    if (nbr) adj_trace<N>(a.q, nbase, np0, nst, Ln, qn);
    Dual td[9], nd[9], e, u;
#pragma unroll
    for (int v = 0; v < 9; ++v) {
      td[v] = Dual(t[v], kk == v ? 1.0 : 0.0);
      nd[v] = Dual(nbr ? qn[v] : 0.0, kk == 9 + v ? 1.0 : 0.0);
    }
    adj_point_speeds<N, Dual>(a, info, k, r, face, sx, sy, td, nd, e, u);
    d = w * (kind == 0 ? e.d : u.d);
  }
  if (kk < 9)
    for (int s = 0; s < N; ++s)
      a.qbar[(size_t)tile * QT + qo<N>(kk, p0 + ps * s, ci)] += d * ops.L[r][s];
  __syncthreads();
  if (nbr && kk >= 9 && kk < 18)
    for (int s = 0; s < N; ++s)
      a.qbar[(size_t)nbt * QT + qo<N>(kk - 9, np0 + nst * s, nbc)] +=
          d * (endN ? ops.L[N][s] : ops.L[0][s]);
  __syncthreads();
}

// What the reverse pass carries from one evaluation to the next, on the
// device: the pending cotangents of the running maxima, the free stream's, and
// whether a maximum's flux point was not found.
struct AdjCarry {
  double PE, PU, p[6];
  int missed;
};

// After adj_stage_kernel of one evaluation (one block): the tiles' partial
// sums in a fixed order; where a flux point of this evaluation exceeded a
// running maximum the pending cotangent of the later evaluations' c_h goes to
// the point that attained the new one (the smallest location code on a tie); and
// this evaluation's own c_h = sqrt(E (E - U)) is passed on to the maxima before
// it.  Where no point exceeded it, the pending cotangent goes on to the earlier
// evaluations, unless the maximum is another value than the one this c_h was
// formed from: then it is the caller's (sd2d_set_state with eigvmax apart from
// eigvmax_g), a constant, and the cotangent ends here.
// 128 x 256 cells, N = 4: 13 us; it replaces two searches over all flux points
// (71 us each), a single-thread evaluation of the 18 directions (106 us) and
// the copy of the partial sums to the host, which waited for every stage.
constexpr int ADJ_TAIL_THREADS = 512;
template <int N>
__global__ __launch_bounds__(ADJ_TAIL_THREADS) void adj_tail_kernel(AdjArgs a, Ops ops_arg,
                                                                    const double *tmax,
                                                                    const int *tloc,
                                                                    const unsigned long long *m1,
                                                                    AdjCarry *cy, double *chbar) {
  constexpr int NT = ADJ_TAIL_THREADS;
  __shared__ double so[sizeof(Ops) / sizeof(double)];
  __shared__ double sum[ADJ_NPART][NT / 64], mv[2][NT / 64];
  __shared__ int ml[2][NT / 64];
  const Ops &ops = ops_to_lds<0>(so, ops_arg);
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  const int none = 0x7fffffff;
  double E, U, g1[2];
  set_pair(a.gm, E, U);
  set_pair(m1, g1[0], g1[1]);
  const double PE = cy->PE, PU = cy->PU;
  const bool raised[2] = {g1[0] > __longlong_as_double((long long)a.gm[0]),
                          g1[1] > __longlong_as_double((long long)a.gm[1])};
  double x[ADJ_NPART] = {0, 0, 0, 0, 0, 0, 0}, best[2] = {0.0, 0.0};
  int loc[2] = {none, none};
  for (int i = t; i < a.ntile; i += NT) {
#pragma unroll
    for (int j = 0; j < ADJ_NPART; ++j) x[j] += a.part[(size_t)i * ADJ_NPART + j];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (!raised[j]) continue;
      const double v = tmax[2 * (size_t)i + j];
      const int c = tloc[2 * (size_t)i + j];
      if (v > best[j] || (v == best[j] && c < loc[j])) { best[j] = v; loc[j] = c; }
    }
  }
#pragma unroll
  for (int j = 0; j < ADJ_NPART; ++j) {
    x[j] = wave_sum(x[j]);
    if (l == 0) sum[j][w] = x[j];
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    for (int o = 32; o > 0; o >>= 1) {
      const double v = __shfl_xor(best[j], o, 64);
      const int c = __shfl_xor(loc[j], o, 64);
      if (v > best[j] || (v == best[j] && c < loc[j])) { best[j] = v; loc[j] = c; }
    }
    if (l == 0) { mv[j][w] = best[j]; ml[j][w] = loc[j]; }
  }
  __syncthreads();
  for (int j = 0; j < 2; ++j) {
    const double p = j == 0 ? PE : PU;
    if (!raised[j] || p == 0.0) continue;   // uniform over the block
    double v = mv[j][0];
    int c = ml[j][0];
    for (int k = 1; k < NT / 64; ++k)
      if (mv[j][k] > v || (mv[j][k] == v && ml[j][k] < c)) { v = mv[j][k]; c = ml[j][k]; }
    if (c == none || v != g1[j]) {
      if (t == 0) cy->missed = 1;
      continue;
    }
    adj_speed_apply<N>(a, ops, c, j, p);
  }
  if (t < ADJ_NPART) {
    double s = 0.0;
    for (int k = 0; k < NT / 64; ++k) s += sum[t][k];
    if (t > 0) cy->p[t - 1] += s;
    else {
      const double ch = sqrt(E * (E - U));
      double pe = raised[0] || g1[0] != E ? 0.0 : PE, pu = raised[1] || g1[1] != U ? 0.0 : PU;
      if (ch > 0.0) {
        pe += s * (2.0 * E - U) / (2.0 * ch);
        pu += s * (-E) / (2.0 * ch);
      }
      cy->PE = pe;
      cy->PU = pu;
      *chbar = s;
    }
  }
}

// The drag of one state added to *J, summed in a fixed order (one block).
__global__ __launch_bounds__(1024) void k_drag_sum(const double *__restrict__ dtile, int n,
                                                   double *__restrict__ J) {
  __shared__ double s[16];
  double x = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) x += dtile[i];
  x = wave_sum(x);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int k = 0; k < 16; ++k) t += s[k];
    *J += t;
  }
}

}  // namespace sd2d
