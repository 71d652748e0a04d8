// sd2d_visc.hpp - the viscous and resistive fluxes of the residual
// (vismode = 1 with mu or eta0 non-zero), in two kernels that run before
// the stage kernel of every residual evaluation:
//
//   vis_grad_kernel   BR1 gradient of all nine variables at the solution
//                     points from the averaged face states (nablaQsp,
//                     compflux.f90:107-157) and, on a mesh with walls, the
//                     computational derivatives of the internal energy
//                     (comp_grad_internal_energy, compflux.f90:260-299);
//   vis_flux_kernel   the gradient at every flux point (interpolated inside
//                     the cell, nablaQ_interior_FP, compflux.f90:159-196;
//                     averaged with the neighbour's trace on interior and
//                     periodic faces, interfaceflux_all.f90:114-195 and
//                     cyclocflux_all.f90:114-204; boundary gradient ghosts
//                     with the adiabatic-wall energy gradient,
//                     bcflux.f90:380-666), the viscous/resistive flux normal
//                     to the point's metric vector (getVfluxvectors,
//                     getrusanov.f90:197-294; comp_viscous_flux,
//                     compflux.f90:198-258) and its divergence dFv + dGv at
//                     the solution points, which the stage kernel adds to
//                     the residual before the Jacobian scaling
//                     (compresid.f90:43-46).
//
// Both use the stage kernel's thread layout: one workgroup per tile of cells, one
// family per wavefront, one thread per grid line (vis_flux_kernel: two).  The
// gradient (18 values per point) lives in HBM between the two kernels in
// tiles of twice the size of a state.
//
// The artificial-viscosity part of comp_viscous_flux adds
// getVfluxvectors_AV with mu_art = eta_art = 0 (getrusanov.f90:325-328),
// which is zero for finite gradients, and is not formed.
#pragma once
#include "sd2d_stage.hpp"

namespace sd2d {

constexpr double LAMBDA_V = -2.0 / 3.0;   // setup2d.f90:69
constexpr double PRANDTL = 0.72;          // setup2d.f90:70

struct VisArgs {
  const double *qin;       // state (tile layout)
  const int *ftab;         // per-cell face table (tile layout)
  const double *met;       // metrics (tile layout)
  int mcomp;               // as StageArgs
  const double *metw;      // other-family metrics at the line ends, for walls
  double *gq;              // gradient (go layout)
  double *dei;             // d(e)/dxi, d(e)/deta [tile][k*N2 + p][ci] (walls)
  double *visres;          // dFv + dGv of variables 0-7, state tile layout (qo)
  const int *tinfo;        // per tile: member << 6 | TI_FIRST | valid cells
  double mu, eta0;
  int ntile, walls;
  int rev, sfam;           // as StageArgs
};

// Slots of the other-family metric table metw, per cell: for each family,
// line end (0: rfp = 0, 1: rfp = N), component and line, S1(2,c,rfp,js)
// on xi-lines and S2(1,c,is,rfp) on eta-lines (bcflux.f90:547-571).
template <int N> struct VisGeo {
  static constexpr int NW = 8 * N;
  static __host__ __device__ constexpr int slot(int fam, int end, int comp, int line) {
    return fam * 4 * N + end * 2 * N + comp * N + line;
  }
};

// Element (v, p, ci) of a gradient tile: d(q_v)/dx and d(q_v)/dy of a point
// of a cell are one 16-byte word.
template <int N>
__host__ __device__ constexpr int go(int v, int p, int ci) {
  return ((v * N * N + p) * cpw_of(N) + ci) * 2;
}

// LDS of vis_grad_kernel (in doubles): the staged state (qo layout); two
// exchange areas of one variable's gradient [p][ci]{x, y}, which on a tile
// with walls then hold the internal energy at the flux points
// [fam][line][rfp][ci]; the wall flag.
template <int N> struct VisGradLds {
  static constexpr int T = Geo<N>::CPW, N2 = N * N, NF = N + 1;
  static constexpr int XA = 9 * N2 * T;          // handed to the xi-lines
  static constexpr int XB = XA + 2 * N2 * T;     // handed to the eta-lines
  static constexpr int EF = XA;
  static constexpr int FLAG = XB + 2 * N2 * T;
  static constexpr int TOTAL = FLAG + 2;
  static_assert(2 * N * NF <= 4 * N2, "the internal energy fits the exchange areas");
};

// LDS of vis_flux_kernel (in doubles): the tile's gradient (go layout), then
// the accumulators handed over, 2 x 7 values per point.
template <int N> struct VisFluxLds {
  static constexpr int TOTAL = 18 * N * N * Geo<N>::CPW;
};

// The averaged state at end rfp of a line (BR1: interfaceflux_all.f90:79-91,
// bcflux.f90 with vismode = 1): own trace t, neighbour trace qn.
__device__ __forceinline__ void vis_end_state(int info, const Phys &ph, const double *t,
                                              const double *qn, double sx, double sy,
                                              double *Qv) {
  const int bc = (info >> 3) & 7;
  if (bc == FT_INTERIOR) {
    const int left = (info >> 2) & 1;
#pragma unroll
    for (int v = 0; v < 9; ++v) {
      const double QL = left ? t[v] : qn[v], QR = left ? qn[v] : t[v];
      Qv[v] = 0.5 * QL + 0.5 * QR;
    }
  } else {
    double QR[9];
    bc_ghost<double>(bc, t, sx, sy, ph, QR);
#pragma unroll
    for (int v = 0; v < 9; ++v) Qv[v] = 0.5 * t[v] + 0.5 * QR[v];
  }
}

// Internal energy of a flux-point state as comp_grad_internal_energy forms
// it (compflux.f90:275-280).
__device__ __forceinline__ double enei_of(const double *q) {
  const double ri = rcp(q[0]);
  const double u = quot(q[1], q[0], ri), v = quot(q[2], q[0], ri), w = quot(q[3], q[0], ri);
  return (((quot(q[4], q[0], ri) - 0.5 * (u * u)) - 0.5 * (v * v)) - 0.5 * (w * w)) -
         quot(0.5 * (((q[5] * q[5] + q[6] * q[6]) + q[7] * q[7]) + q[8] * q[8]), q[0], ri);
}

// nablaQsp (compflux.f90:107-157) and, on tiles with walls,
// comp_grad_internal_energy (compflux.f90:260-299).
//
// One thread per grid line as in the stage kernel, and the same start: face
// words, the tile's state staged in LDS, the neighbours' traces gathered in
// as few passes as the wave needs, the averaged end states in registers.
// Then one variable per family and round: a thread forms the line's
// contribution to the gradient at its N points of the variable the other
// family finishes (into LDS) and of the one its own finishes (kept), and
// after the barrier adds the two, scales by 1/J and stores both components
// as one 16-byte word.  The xi-lines finish variables 0-3 and d(psi)/dx, the
// eta-lines 4-7 and d(psi)/dy, so both waves store half.
// Bound by the L2 and the loads in flight (2 waves per SIMD, 3 at N = 3: 158-210
// VGPRs, 31-41 KB of LDS).  128 x 256 cells, N = 5: 62 us, 3.1 TB/s of its compulsory
// 232 bytes a point; N = 4: 33 us, N = 3: 21 us.  The form before it, which read every
// flux point's line and neighbour from memory (12 reads of the tile, one
// 8-byte word at a time) and let one family store everything: 259 and 115 us.
template <int N>
__global__ __launch_bounds__(STAGE_THREADS, 2) void vis_grad_kernel(VisArgs va, Ops ops, Phys ph) {
  using G = Geo<N>;
  using LD = VisGradLds<N>;
  constexpr int T = G::CPW, N2 = G::N2, NF = N + 1;
  static_assert(N * T <= 64 && STAGE_THREADS == 128, "one wavefront per line family");
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const int tile = tile_of_block(blockIdx.x, va.ntile, va.rev);
  const int fam = wave_uniform(tid >> 6), line = (tid & 63) / T, ci = (tid & 63) % T;
  int nb0, nbN, info0, infoN;
  face_words<N>(va, tile, ci, fam, line, 0, nb0, info0);
  face_words<N>(va, tile, ci, fam, line, N, nbN, infoN);
  const int ti = va.tinfo[tile];
  if (fam == va.sfam) {
    constexpr int NV2 = 9 * N2 * T / 2, NSW = (NV2 + 63) / 64;
    const double2 *src = reinterpret_cast<const double2 *>(va.qin + (size_t)tile * G::QT);
    double2 *dst = reinterpret_cast<double2 *>(lds);
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
  if (tid == 0) lds[LD::FLAG] = 0.0;
  const bool valid = line < N && ci < (ti & TI_VALID);
  const MetLine<N, double> ml(va.met, va.mcomp, tile, ci, fam, line);
  const int p0 = fam ? line : N * line, ps = fam ? N : 1;
  double qn0[9], qnN[9];
  int lci0 = -1, lciN = -1;
  double msx[NF], msy[NF], ji[N];
  if (valid) {
    face_gather_pair<N, double>(va, ops, tile, fam, line, nb0, info0, nbN, infoN, qn0, qnN, lci0,
                                lciN);
#pragma unroll
    for (int r = 0; r < NF; ++r) {
      msx[r] = ml.x[r * T];
      msy[r] = ml.y[r * T];
    }
#pragma unroll
    for (int s = 0; s < N; ++s)
      ji[s] = ml.ji[((fam ? s : line) + N * (fam ? line : s)) * T];
  }
  __syncthreads();
  const bool wall0 = valid && ((info0 >> 3) & 7) == FT_WALL;
  const bool wallN = valid && ((infoN >> 3) & 7) == FT_WALL;
  if (va.walls && (wall0 || wallN)) lds[LD::FLAG] = 1.0;   // (every writer stores the same)
  double qe0[9], qeN[9];                 // averaged states of the line's two ends
  if (valid) {
    if (lci0 >= 0) face_trace_lds<N, double>(lds, ops, info0, fam, line, 0, lci0, qn0);
    if (lciN >= 0) face_trace_lds<N, double>(lds, ops, infoN, fam, line, N, lciN, qnN);
    double t0[9], tN[9];
    line_vals<N, double>(lds, p0, ps, ci, [&](int v, const double *vals) {
      t0[v] = line_trace<N, double>(vals, ops.L[0]);
      tN[v] = line_trace<N, double>(vals, ops.L[N]);
    });
    vis_end_state(info0, ph, t0, qn0, msx[0], msy[0], qe0);
    vis_end_state(infoN, ph, tN, qnN, msx[N], msy[N], qeN);
  }
  // the line's contribution to the gradient of variable v at its points
  auto contrib = [&](int v, double e0, double eN, double *gx, double *gy) {
    double vals[N], q[NF];
#pragma unroll
    for (int s = 0; s < N; ++s) vals[s] = lds[qo<N>(v, p0 + ps * s, ci)];
    q[0] = e0;
    q[N] = eN;
#pragma unroll
    for (int r = 1; r < N; ++r) q[r] = line_trace<N, double>(vals, ops.L[r]);
#pragma unroll
    for (int s = 0; s < N; ++s) gx[s] = gy[s] = 0.0;
#pragma unroll
    for (int r = 0; r < NF; ++r) {
      const double tx = q[r] * msx[r], ty = q[r] * msy[r];
#pragma unroll
      for (int s = 0; s < N; ++s) {
        gx[s] = fma(tx, ops.M[r][s], gx[s]);
        gy[s] = fma(ty, ops.M[r][s], gy[s]);
      }
    }
  };
  double *gq = va.gq + (size_t)tile * 2 * G::QT;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    // rounds 0-3: variable k for the xi-lines, 4 + k for the eta-lines; round
    // 4: psi, its x part for the xi-lines, its y part for the eta-lines
    const int vx = k < 4 ? k : 8, ve = k < 4 ? 4 + k : 8;
    double ox[N], oy[N];
    if (valid) {
      const int vo = fam ? ve : vx, vg = fam ? vx : ve;   // own, given away
      const double eo0 = fam ? qe0[ve] : qe0[vx], eoN = fam ? qeN[ve] : qeN[vx];
      if (k < 4) {
        const double eg0 = fam ? qe0[vx] : qe0[ve], egN = fam ? qeN[vx] : qeN[ve];
        double gx[N], gy[N];
        contrib(vg, eg0, egN, gx, gy);
        double *x = lds + (fam ? LD::XA : LD::XB);
#pragma unroll
        for (int s = 0; s < N; ++s)
          *reinterpret_cast<double2 *>(x + 2 * ((p0 + ps * s) * T + ci)) = double2{gx[s], gy[s]};
      }
      contrib(vo, eo0, eoN, ox, oy);
      if (k == 4) {
        double *x = lds + (fam ? LD::XA : LD::XB);
#pragma unroll
        for (int s = 0; s < N; ++s) x[(p0 + ps * s) * T + ci] = fam ? ox[s] : oy[s];
      }
    }
    __syncthreads();
    if (valid) {
      const double *x = lds + (fam ? LD::XB : LD::XA);
#pragma unroll
      for (int s = 0; s < N; ++s) {
        const int p = p0 + ps * s;
        if (k < 4) {
          const double2 d = *reinterpret_cast<const double2 *>(x + 2 * (p * T + ci));
          const double2 g = {(ox[s] + d.x) * ji[s], (oy[s] + d.y) * ji[s]};
          *reinterpret_cast<double2 *>(gq + go<N>(fam ? ve : vx, p, ci)) = g;
        } else {
          gq[go<N>(8, p, ci) + fam] = ((fam ? oy[s] : ox[s]) + x[p * T + ci]) * ji[s];
        }
      }
    }
    __syncthreads();
  }
  // internal-energy derivatives for the adiabatic wall's gradient ghost
  // (bcflux.f90:547-571), on the few tiles that hold a wall face
  if (!va.walls || lds[LD::FLAG] == 0.0) return;
  if (valid) {
    double *ef = lds + LD::EF + (fam * N + line) * NF * T + ci;
    ef[0] = enei_of(qe0);
    ef[N * T] = enei_of(qeN);
#pragma unroll
    for (int r = 1; r < N; ++r) {
      double t[9];
      line_vals<N, double>(lds, p0, ps, ci, [&](int v, const double *vals) {
        t[v] = line_trace<N, double>(vals, ops.L[r]);
      });
      ef[r * T] = enei_of(t);
    }
  }
  __syncthreads();
  if (valid) {
    // a xi-line thread stores d(e)/dxi at its points, an eta-line d(e)/deta
    const double *ef = lds + LD::EF + (fam * N + line) * NF * T + ci;
    double *o = va.dei + ((size_t)tile * 2 + fam) * N2 * T + ci;
#pragma unroll
    for (int s = 0; s < N; ++s) {
      double d = 0.0;
#pragma unroll
      for (int r = 0; r < NF; ++r) d = fma(ef[r * T], ops.M[r][s], d);
      o[(size_t)(p0 + ps * s) * T] = d;
    }
  }
}

// getVfluxvectors (getrusanov.f90:197-294) contracted with the metric
// vector (sx, sy): Fn[k] = Fv[k+1]*sx + Gv[k+1]*sy for variables 1-7 (the
// fluxes of rho and psi are zero; compflux.f90:215-216,243-244).
// g[2v] is d(q_v)/dx, g[2v+1] is d(q_v)/dy.
// The quotients by rho share one reciprocal and are corrected (quot): plain
// products with it put the momentum components 8-11 % further from the exact flux
// than divisions do (rms over random states) and saved at most 1 % of a step.
__device__ __forceinline__ void vflux_n(const double *Qv, const double *g, double mu,
                                        double eta, double sx, double sy, double *Fn) {
  const double rho = Qv[0], rhoE = Qv[4];
  const double Bx = Qv[5], By = Qv[6], Bz = Qv[7], psi = Qv[8];
  const double ri = rcp(rho);
  const double u = quot(Qv[1], rho, ri), v = quot(Qv[2], rho, ri), w = quot(Qv[3], rho, ri);
  const double nu = u * u + v * v + w * w;
  const double nb = Bx * Bx + By * By + Bz * Bz;
  const double inte = quot(rhoE - 0.5 * nu * rho - 0.5 * nb - 0.5 * (psi * psi), rho, ri);
  double du[2], dv[2], dw[2], de[2];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const double dr = g[d];
    du[d] = quot(g[2 + d] - dr * u, rho, ri);
    dv[d] = quot(g[4 + d] - dr * v, rho, ri);
    dw[d] = quot(g[6 + d] - dr * w, rho, ri);
    const double dke = 0.5 * nu * dr + rho * (u * du[d] + v * dv[d] + w * dw[d]);
    const double dpb = Bx * g[10 + d] + By * g[12 + d] + Bz * g[14 + d];
    de[d] = quot(g[8 + d] - dke - dpb - dr * inte - psi * g[16 + d], rho, ri);
  }
  const double ux = du[0], uy = du[1], vx = dv[0], vy = dv[1], wx = dw[0], wy = dw[1];
  constexpr double KP = GAM / PRANDTL;
  const double txx = mu * (2.0 * ux + LAMBDA_V * (ux + vy));
  const double tyy = mu * (2.0 * vy + LAMBDA_V * (ux + vy));
  const double txy = mu * (vx + uy), txz = mu * wx, tyz = mu * wy;
  // J = curl B in 2-D (getrusanov.f90:271-292), times the resistivity
  const double Jx = eta * g[15], Jy = -eta * g[14], Jz = eta * (g[12] - g[11]);
  const double F4 = u * txx + v * txy + w * txz + mu * KP * de[0] + Jz * By - Jy * Bz;
  const double G4 = u * txy + v * tyy + w * tyz + mu * KP * de[1] - Jz * Bx + Jx * Bz;
  Fn[0] = txx * sx + txy * sy;
  Fn[1] = txy * sx + tyy * sy;
  Fn[2] = txz * sx + tyz * sy;
  Fn[3] = F4 * sx + G4 * sy;
  Fn[4] = -Jz * sy;
  Fn[5] = Jz * sx;
  Fn[6] = Jx * sy - Jy * sx;
}

// Energy rows of the gradient ghost of the adiabatic wall (bcflux.f90:484-571)
// for the wall trace Qo of the state, the own gradient trace gl (layout of
// vflux_n), the internal-energy derivative across the wall family dface
// (dedeta on xi-lines, dedxi on eta-lines) and the other-family metric
// (ox, oy): gr4[d].  The other rows are the own trace's.  The second
// direction reuses the first direction's magnetic term, as the reference
// does (bcflux.f90:563).
__device__ __forceinline__ void wall_grad_ghost(const double *Qo, const double *gl, double dface,
                                                double ox, double oy, double *gr4) {
  const double ri = rcp(Qo[0]);
  const double ur = quot(Qo[1], Qo[0], ri), vr = quot(Qo[2], Qo[0], ri),
               wr = quot(Qo[3], Qo[0], ri);
  const double inte = enei_of(Qo);
  const double dBp = ((Qo[5] * gl[10] + Qo[6] * gl[12]) + Qo[7] * gl[14]) + Qo[8] * gl[16];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const double dur = quot(gl[2 + d] - ur * gl[d], Qo[0], ri);
    const double dvr = quot(gl[4 + d] - vr * gl[d], Qo[0], ri);
    const double dwr = quot(gl[6 + d] - wr * gl[d], Qo[0], ri);
    const double dKE = 0.5 * ((ur * ur + vr * vr) + wr * wr) * gl[d] +
                       Qo[0] * ((ur * dur + vr * dvr) + wr * dwr);
    gr4[d] = (((-gl[8 + d] + 2.0 * inte * gl[d]) + 2.0 * dKE) + dBp) +
             2.0 * dface * (d == 0 ? ox : oy) * Qo[0];
  }
}

// f(v, vals) for v = 0..8 with vals[2s + d] = d(q_v)/dx_d at point p0 + ps*s
// of slot ci of the gradient tile g (go layout).
template <int N, typename F>
__device__ __forceinline__ void grad_vals(const double *g, int p0, int ps, int ci, F &&f) {
#pragma unroll
  for (int v = 0; v < 9; ++v) {
    double vals[2 * N];
#pragma unroll
    for (int s = 0; s < N; ++s) {
      const double2 d = *reinterpret_cast<const double2 *>(g + go<N>(v, p0 + ps * s, ci));
      vals[2 * s] = d.x;
      vals[2 * s + 1] = d.y;
    }
    f(v, vals);
  }
}

// The gradient trace at a flux point from grad_vals, with operator row Lr.
template <int N>
__device__ __forceinline__ void grad_trace(const double *vals, const double *Lr, double *out) {
  double a = 0.0, b = 0.0;
#pragma unroll
  for (int s = 0; s < N; ++s) {
    a = fma(vals[2 * s], Lr[s], a);
    b = fma(vals[2 * s + 1], Lr[s], b);
  }
  out[0] = a;
  out[1] = b;
}

// Viscous flux divergence dFv + dGv at the solution points (variables 1-7).
//
// Four waves per tile, two threads per grid line: wave 2*fam + half, where half
// 0 takes the flux points 0 .. N/2 of the line, half 1 the others from N down.
// The tile's gradient (18 values a point) is staged in LDS.  Before the
// barrier a thread forms the state traces of its flux points and, where its
// end face's neighbour lies in another tile, gathers that neighbour's gradient
// trace (from the staged gradient after it otherwise); the end's traces are
// averaged (BR1, interfaceflux_all.f90:140-190; boundary ghosts: a copy, or
// the adiabatic wall, bcflux.f90:380-666).  Each flux point's seven fluxes are
// folded into the thread's derivative accumulators; half 1 hands its
// accumulators to half 0 through the LDS the gradient occupied, then the
// families exchange: the xi-lines finish variables 1-3, the eta-lines 4-7.
// Two waves per SIMD (193-254 VGPRs, 26-43 KB of LDS); bound by the vector
// memory and LDS pipes together (95 16-byte loads and 180 LDS reads a thread
// at N = 5), then by FP64 issue.  128 x 256 cells, N = 5: 109 us; with one
// thread per line (both ends and all interior points: 376 registers, one wave
// per SIMD) 133 us; when every flux point read its lines from memory, 406 us.
// N = 4 (151 x 90): 35 / 35 / 108 us, N = 3 (128 x 256): 47 / 44 / 153 us
// (this form with uncorrected quotients: 111, 34 and 46 us).
// All flux points' gradient traces in one pass over LDS spill (660 bytes a
// lane at N = 5).
constexpr int VIS_FLUX_THREADS = 256;
template <int N>
__global__ __launch_bounds__(VIS_FLUX_THREADS, 2) void vis_flux_kernel(VisArgs va, Ops ops,
                                                                       Phys ph) {
  using G = Geo<N>;
  constexpr int T = G::CPW, N2 = G::N2, QT = G::QT;
  static_assert(N * T <= 64, "one wavefront per line family and half");
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const int tile = tile_of_block(blockIdx.x, va.ntile, va.rev);
  // (uniform, so that each half runs its own code with a barrier of its own)
  const int wv = wave_uniform(tid >> 6), fam = wv >> 1, half = wv & 1;
  const int line = (tid & 63) / T, ci = (tid & 63) % T;
  int nb, info;
  face_words<N>(va, tile, ci, fam, line, half ? N : 0, nb, info);
  const int ti = va.tinfo[tile];
  {
    constexpr int NV2 = 9 * N2 * T, NR = (NV2 + VIS_FLUX_THREADS - 1) / VIS_FLUX_THREADS;
    const double2 *src = reinterpret_cast<const double2 *>(va.gq + (size_t)tile * 2 * QT);
    double2 *dst = reinterpret_cast<double2 *>(lds);
    double2 st[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int i = tid + k * VIS_FLUX_THREADS;
      st[k] = src[(k < NR - 1 || i < NV2) ? i : 0];
    }
#pragma unroll
    for (int k = 0; k < NR - 1; ++k) dst[tid + k * VIS_FLUX_THREADS] = st[k];
    if (tid + (NR - 1) * VIS_FLUX_THREADS < NV2) dst[tid + (NR - 1) * VIS_FLUX_THREADS] = st[NR - 1];
  }
  const bool valid = line < N && ci < (ti & TI_VALID);
  const MetLine<N, double> ml(va.met, va.mcomp, tile, ci, fam, line);
  const int p0 = fam ? line : N * line, ps = fam ? N : 1;
  const double *qt = va.qin + (size_t)tile * QT;
  const bool inter = ((info >> 3) & 7) == FT_INTERIOR, far = inter && nb / QT != tile;
  // the neighbour's line through the end face's shared point
  int np0 = 0, nst = 0, nci = 0;
  bool endN;
  {
    int k, nfp;
    end_face<N>(fam, line, half ? N : 0, k, nfp);
    neighbour_line<N>(info & 3, nfp, np0, nst, endN);
  }
  auto row = [&](int s) { return endN ? ops.L[N][s] : ops.L[0][s]; };
  double D[N][7];
  // a half's flux points: the end face (row RE) and NI interior points from R1
  // in steps of DR
  auto fluxes = [&](auto hc) __attribute__((always_inline)) {
    constexpr int H = decltype(hc)::value;
    constexpr int RE = H ? N : 0, R1 = H ? N - 1 : 1, DR = H ? -1 : 1;
    constexpr int NI = H ? N - 1 - N / 2 : N / 2;
    double Qv[9], t[NI][9], g1[18], sx[NI + 1], sy[NI + 1];
    if (valid) {
      double qn[9];
      if (inter) {
        const int nt = nb / QT;
        nci = nb - nt * QT;
        double Lr[N];
#pragma unroll
        for (int s = 0; s < N; ++s) Lr[s] = row(s);
        if (far)
          grad_vals<N>(va.gq + (size_t)nt * 2 * QT, np0, nst, nci, [&](int v, const double *x) {
            grad_trace<N>(x, Lr, g1 + 2 * v);
          });
        line_vals<N, double>(va.qin + (size_t)nt * QT, np0, nst, nci, [&](int v, const double *x) {
          qn[v] = line_trace<N, double>(x, Lr);
        });
      }
      sx[NI] = ml.x[RE * T];
      sy[NI] = ml.y[RE * T];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        sx[i] = ml.x[(R1 + DR * i) * T];
        sy[i] = ml.y[(R1 + DR * i) * T];
      }
      double te[9];
      line_vals<N, double>(qt, p0, ps, ci, [&](int v, const double *x) {
        te[v] = line_trace<N, double>(x, ops.L[RE]);
#pragma unroll
        for (int i = 0; i < NI; ++i) t[i][v] = line_trace<N, double>(x, ops.L[R1 + DR * i]);
      });
      vis_end_state(info, ph, te, qn, sx[NI], sy[NI], Qv);
    }
    __syncthreads();
    if (!valid) return;
    {
      double g[18], F[7];
      grad_vals<N>(lds, p0, ps, ci, [&](int v, const double *x) {
        grad_trace<N>(x, ops.L[RE], g + 2 * v);
      });
      if (inter) {
        if (!far) {   // an in-tile neighbour: its gradient is staged
          double Lr[N];
#pragma unroll
          for (int s = 0; s < N; ++s) Lr[s] = row(s);
          grad_vals<N>(lds, np0, nst, nci, [&](int v, const double *x) {
            grad_trace<N>(x, Lr, g1 + 2 * v);
          });
        }
#pragma unroll
        for (int c = 0; c < 18; ++c) g[c] = 0.5 * g[c] + 0.5 * g1[c];
      } else if (((info >> 3) & 7) == FT_WALL) {
        // d(e)/deta along a xi-line, d(e)/dxi along an eta-line
        const double *de = va.dei + ((size_t)tile * 2 + (1 - fam)) * N2 * T + ci;
        double dface = 0.0, to[9];
#pragma unroll
        for (int s = 0; s < N; ++s) dface = fma(de[(size_t)(p0 + ps * s) * T], ops.L[RE][s], dface);
        line_vals<N, double>(qt, p0, ps, ci, [&](int v, const double *x) {
          to[v] = line_trace<N, double>(x, ops.L[RE]);
        });
        const double *mw = va.metw + (size_t)tile * VisGeo<N>::NW * T + ci;
        double gr4[2];
        wall_grad_ghost(to, g, dface, mw[VisGeo<N>::slot(fam, H, 0, line) * T],
                        mw[VisGeo<N>::slot(fam, H, 1, line) * T], gr4);
        g[8] = 0.5 * g[8] + 0.5 * gr4[0];
        g[9] = 0.5 * g[9] + 0.5 * gr4[1];
      }
      vflux_n(Qv, g, va.mu, va.eta0, sx[NI], sy[NI], F);
#pragma unroll
      for (int s = 0; s < N; ++s)
#pragma unroll
        for (int c = 0; c < 7; ++c) D[s][c] = F[c] * ops.M[RE][s];
    }
    // interior flux points (compflux.f90:198-258)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      double g[18], F[7];
      grad_vals<N>(lds, p0, ps, ci, [&](int v, const double *x) {
        grad_trace<N>(x, ops.L[R1 + DR * i], g + 2 * v);
      });
      vflux_n(t[i], g, va.mu, va.eta0, sx[i], sy[i], F);
#pragma unroll
      for (int s = 0; s < N; ++s)
#pragma unroll
        for (int c = 0; c < 7; ++c) D[s][c] = fma(F[c], ops.M[R1 + DR * i][s], D[s][c]);
    }
  };
  if (half) fluxes(std::integral_constant<int, 1>{});
  else fluxes(std::integral_constant<int, 0>{});
  // half 1's accumulators to half 0, [fam][c][p][ci]
  double *own = lds + fam * 7 * N2 * T, *other = lds + (1 - fam) * 7 * N2 * T;
  auto at = [&](int c, int s) { return (c * N2 + p0 + ps * s) * T + ci; };
  __syncthreads();   // every read of the staged gradient is done
  if (valid && half) {
#pragma unroll
    for (int s = 0; s < N; ++s)
#pragma unroll
      for (int c = 0; c < 7; ++c) own[at(c, s)] = D[s][c];
  }
  __syncthreads();
  // the sums of a line; what the other family finishes goes back to where
  // this thread read it
  if (valid && !half) {
#pragma unroll
    for (int s = 0; s < N; ++s)
#pragma unroll
      for (int c = 0; c < 7; ++c) {
        D[s][c] += own[at(c, s)];
        if ((c < 3) == (fam == 1)) own[at(c, s)] = D[s][c];
      }
  }
  __syncthreads();
  if (!valid || half) return;
  double *o = va.visres + (size_t)tile * QT;
#pragma unroll
  for (int s = 0; s < N; ++s) {
    const int p = p0 + ps * s;
    double w[4];
    if (fam) {
#pragma unroll
      for (int c = 0; c < 4; ++c) w[c] = D[s][3 + c] + other[at(3 + c, s)];
      store_vars<N, 4, 8>(o, p, ci, w);
    } else {
      w[0] = 0.0;   // rho has no viscous flux
#pragma unroll
      for (int c = 0; c < 3; ++c) w[1 + c] = D[s][c] + other[at(c, s)];
      store_vars<N, 0, 4>(o, p, ci, w);
    }
  }
}

template <int N>
constexpr size_t vis_grad_lds_bytes() { return sizeof(double) * VisGradLds<N>::TOTAL; }
template <int N>
constexpr size_t vis_flux_lds_bytes() { return sizeof(double) * VisFluxLds<N>::TOTAL; }

}  // namespace sd2d
