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
// Both use the stage kernel's thread layout: one 128-thread workgroup per
// tile of cells, one thread per grid line, one family per wavefront.  The
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

// LDS of vis_flux_kernel (in doubles): the tile's gradient (go layout); after
// the fluxes, the derivatives the families hand each other: variables 1-3 for
// the xi-lines, 4-7 for the eta-lines, [k][p][ci].
template <int N> struct VisFluxLds {
  static constexpr int T = Geo<N>::CPW, N2 = N * N;
  static constexpr int XA = 0, XB = 3 * N2 * T;
  static constexpr int TOTAL = 18 * N2 * T;
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
  const double u = q[1] * ri, v = q[2] * ri, w = q[3] * ri;
  return (((q[4] * ri - 0.5 * (u * u)) - 0.5 * (v * v)) - 0.5 * (w * w)) -
         0.5 * (((q[5] * q[5] + q[6] * q[6]) + q[7] * q[7]) + q[8] * q[8]) * ri;
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
// Bound by the L2 and the loads in flight (2 waves per SIMD: 184-216 VGPRs,
// 31-41 KB of LDS).  128 x 256 cells, N = 5: 69 us, 3.1 TB/s of its compulsory
// 262 bytes a point; N = 4: 35 us.  The form before it, which read every
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
  const int fam = tid >> 6, line = (tid & 63) / T, ci = (tid & 63) % T;
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
__device__ __forceinline__ void vflux_n(const double *Qv, const double *g, double mu,
                                        double eta, double sx, double sy, double *Fn) {
  const double rho = Qv[0], rhoE = Qv[4];
  const double Bx = Qv[5], By = Qv[6], Bz = Qv[7], psi = Qv[8];
  const double ri = rcp(rho);
  const double u = Qv[1] * ri, v = Qv[2] * ri, w = Qv[3] * ri;
  const double nu = u * u + v * v + w * w;
  const double nb = Bx * Bx + By * By + Bz * Bz;
  const double inte = (rhoE - 0.5 * nu * rho - 0.5 * nb - 0.5 * (psi * psi)) * ri;
  double du[2], dv[2], dw[2], de[2];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const double dr = g[d];
    du[d] = (g[2 + d] - dr * u) * ri;
    dv[d] = (g[4 + d] - dr * v) * ri;
    dw[d] = (g[6 + d] - dr * w) * ri;
    const double dke = 0.5 * nu * dr + rho * (u * du[d] + v * dv[d] + w * dw[d]);
    const double dpb = Bx * g[10 + d] + By * g[12 + d] + Bz * g[14 + d];
    de[d] = (g[8 + d] - dke - dpb - dr * inte - psi * g[16 + d]) * ri;
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
  const double ur = Qo[1] * ri, vr = Qo[2] * ri, wr = Qo[3] * ri;
  const double inte = enei_of(Qo);
  const double dBp = ((Qo[5] * gl[10] + Qo[6] * gl[12]) + Qo[7] * gl[14]) + Qo[8] * gl[16];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const double dur = (gl[2 + d] - ur * gl[d]) * ri;
    const double dvr = (gl[4 + d] - vr * gl[d]) * ri;
    const double dwr = (gl[6 + d] - wr * gl[d]) * ri;
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
// One thread per grid line; the tile's gradient (18 values a point) is staged
// in LDS by both waves, the line's own state stays in registers.  The
// neighbours' state and gradient traces of the two end faces are gathered
// before the barrier where the neighbour lies in another tile (from the
// staged gradient after it otherwise) and averaged with the own ones (BR1,
// interfaceflux_all.f90:140-190; boundary ghosts: a copy, or the adiabatic
// wall, bcflux.f90:380-666).  Each flux point's seven fluxes are folded into
// the line's derivative accumulators, and the families exchange half of them
// through the LDS the gradient occupied: the xi-lines finish variables 1-3,
// the eta-lines 4-7.
// 256 VGPRs and 40-152 AGPRs (the line's 9 N state values, 7 N accumulators,
// the gathered traces), so one wave per SIMD; bound by the latency of its
// loads, which nothing overlaps, then by FP64 issue.  128 x 256 cells, N = 5:
// 136 us (406 us when every flux point read its lines from memory); N = 4:
// 65 us (216).  Held to two waves per SIMD the kernel spills (250-370
// bytes a lane) and takes 207 us at N = 5, with the state re-read from memory
// per point 152 us; both lose at N = 3 and 4 as well.
template <int N>
__global__ __launch_bounds__(STAGE_THREADS, 1) void vis_flux_kernel(VisArgs va, Ops ops, Phys ph) {
  using G = Geo<N>;
  using LD = VisFluxLds<N>;
  constexpr int T = G::CPW, N2 = G::N2, NF = N + 1, QT = G::QT;
  static_assert(N * T <= 64 && STAGE_THREADS == 128, "one wavefront per line family");
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const int tile = tile_of_block(blockIdx.x, va.ntile, va.rev);
  const int fam = tid >> 6, line = (tid & 63) / T, ci = (tid & 63) % T;
  int nb0, nbN, info0, infoN;
  face_words<N>(va, tile, ci, fam, line, 0, nb0, info0);
  face_words<N>(va, tile, ci, fam, line, N, nbN, infoN);
  const int ti = va.tinfo[tile];
  {
    constexpr int NV2 = 9 * N2 * T, NR = (NV2 + STAGE_THREADS - 1) / STAGE_THREADS;
    const double2 *src = reinterpret_cast<const double2 *>(va.gq + (size_t)tile * 2 * QT);
    double2 *dst = reinterpret_cast<double2 *>(lds);
    double2 st[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int i = tid + k * STAGE_THREADS;
      st[k] = src[(k < NR - 1 || i < NV2) ? i : 0];
    }
#pragma unroll
    for (int k = 0; k < NR - 1; ++k) dst[tid + k * STAGE_THREADS] = st[k];
    if (tid + (NR - 1) * STAGE_THREADS < NV2) dst[tid + (NR - 1) * STAGE_THREADS] = st[NR - 1];
  }
  const bool valid = line < N && ci < (ti & TI_VALID);
  const MetLine<N, double> ml(va.met, va.mcomp, tile, ci, fam, line);
  const int p0 = fam ? line : N * line, ps = fam ? N : 1;
  const double *qt = va.qin + (size_t)tile * QT;
  double q[N][9];
  double msx[NF], msy[NF];
  const bool i0 = ((info0 >> 3) & 7) == FT_INTERIOR, iN = ((infoN >> 3) & 7) == FT_INTERIOR;
  const bool far0 = i0 && nb0 / QT != tile, farN = iN && nbN / QT != tile;
  // the neighbour's gradient line through the shared point of an end face
  auto grad_line = [&](int rfp, int info, int &np0, int &nst, double *Lr) {
    int k, nfp;
    end_face<N>(fam, line, rfp, k, nfp);
    bool endN;
    neighbour_line<N>(info & 3, nfp, np0, nst, endN);
#pragma unroll
    for (int s = 0; s < N; ++s) Lr[s] = endN ? ops.L[N][s] : ops.L[0][s];
  };
  // the traces of the line's first end whose neighbour lies in another tile,
  // gathered now; a second such end waits until its flux is formed
  double q1[9], g1[18];
  auto far_traces = [&](int rfp, int nb, int info, double *qn, double *gn) {
    const int nt = nb / QT, nci = nb - nt * QT;
    int np0, nst;
    double Lr[N];
    grad_line(rfp, info, np0, nst, Lr);
    line_vals<N, double>(va.qin + (size_t)nt * QT, np0, nst, nci, [&](int v, const double *vals) {
      qn[v] = line_trace<N, double>(vals, Lr);
    });
    grad_vals<N>(va.gq + (size_t)nt * 2 * QT, np0, nst, nci, [&](int v, const double *vals) {
      grad_trace<N>(vals, Lr, gn + 2 * v);
    });
  };
  if (valid) {
    if (far0 || farN)
      far_traces(far0 ? 0 : N, far0 ? nb0 : nbN, far0 ? info0 : infoN, q1, g1);
#pragma unroll
    for (int s = 0; s < N; ++s) load_vars<N, 0, 9>(qt, p0 + ps * s, ci, q[s]);
#pragma unroll
    for (int r = 0; r < NF; ++r) {
      msx[r] = ml.x[r * T];
      msy[r] = ml.y[r * T];
    }
  }
  __syncthreads();
  double D[N][7];
  if (valid) {
    auto state_trace = [&](const double *Lr, double *t) {
#pragma unroll
      for (int v = 0; v < 9; ++v) {
        double a = 0.0;
#pragma unroll
        for (int s = 0; s < N; ++s) a = fma(q[s][v], Lr[s], a);
        t[v] = a;
      }
    };
    // The two end faces, the one whose traces are at hand first: end N where
    // only that one gathered, so the order is a value of the lane and the
    // wave runs two passes, not three.
    auto end_flux = [&](bool atN, bool gathered, double *F) {
      const int rfp = atN ? N : 0, nb = atN ? nbN : nb0, info = atN ? infoN : info0;
      const bool inter = atN ? iN : i0, far = atN ? farN : far0;
      double Lo[N];
#pragma unroll
      for (int s = 0; s < N; ++s) Lo[s] = atN ? ops.L[N][s] : ops.L[0][s];
      const double sx = atN ? msx[N] : msx[0], sy = atN ? msy[N] : msy[0];
      if (inter && !far) {   // an in-tile neighbour: its gradient is staged
        int np0, nst;
        double Lr[N];
        grad_line(rfp, info, np0, nst, Lr);
        line_vals<N, double>(qt, np0, nst, nb - tile * QT, [&](int v, const double *vals) {
          q1[v] = line_trace<N, double>(vals, Lr);
        });
        grad_vals<N>(lds, np0, nst, nb - tile * QT, [&](int v, const double *vals) {
          grad_trace<N>(vals, Lr, g1 + 2 * v);
        });
      } else if (far && !gathered) {
        far_traces(rfp, nb, info, q1, g1);
      }
      double t[9], Qv[9], g[18];
      state_trace(Lo, t);
      vis_end_state(info, ph, t, q1, sx, sy, Qv);
      grad_vals<N>(lds, p0, ps, ci, [&](int v, const double *vals) {
        grad_trace<N>(vals, Lo, g + 2 * v);
      });
      if (inter) {
#pragma unroll
        for (int c = 0; c < 18; ++c) g[c] = 0.5 * g[c] + 0.5 * g1[c];
      } else if (((info >> 3) & 7) == FT_WALL) {
        // d(e)/deta along a xi-line, d(e)/dxi along an eta-line
        const double *de = va.dei + ((size_t)tile * 2 + (1 - fam)) * N2 * T + ci;
        double dface = 0.0;
#pragma unroll
        for (int s = 0; s < N; ++s) dface = fma(de[(size_t)(p0 + ps * s) * T], Lo[s], dface);
        const double *mw = va.metw + (size_t)tile * VisGeo<N>::NW * T + ci;
        double gr4[2];
        wall_grad_ghost(t, g, dface, mw[VisGeo<N>::slot(fam, atN, 0, line) * T],
                        mw[VisGeo<N>::slot(fam, atN, 1, line) * T], gr4);
        g[8] = 0.5 * g[8] + 0.5 * gr4[0];
        g[9] = 0.5 * g[9] + 0.5 * gr4[1];
      }
      vflux_n(Qv, g, va.mu, va.eta0, sx, sy, F);
    };
    {
      double FA[7], FB[7];
      const bool nfirst = farN && !far0;
      end_flux(nfirst, true, FA);
      __builtin_amdgcn_sched_barrier(0);
      end_flux(!nfirst, false, FB);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < N; ++s) {
        const double MA = nfirst ? ops.M[N][s] : ops.M[0][s], MB = nfirst ? ops.M[0][s] : ops.M[N][s];
#pragma unroll
        for (int k = 0; k < 7; ++k) D[s][k] = fma(FB[k], MB, FA[k] * MA);
      }
    }
    // interior flux points two at a time (compflux.f90:198-258)
    auto point = [&](int r, const double *g) {
      double t[9], F[7];
      state_trace(ops.L[r], t);
      vflux_n(t, g, va.mu, va.eta0, msx[r], msy[r], F);
#pragma unroll
      for (int s = 0; s < N; ++s)
#pragma unroll
        for (int k = 0; k < 7; ++k) D[s][k] = fma(F[k], ops.M[r][s], D[s][k]);
    };
#pragma unroll
    for (int r = 1; r < N; r += 2) {
      const bool two = r + 1 < N;
      double ga[18], gb[18];
      grad_vals<N>(lds, p0, ps, ci, [&](int v, const double *vals) {
        grad_trace<N>(vals, ops.L[r], ga + 2 * v);
        if (two) grad_trace<N>(vals, ops.L[r + 1], gb + 2 * v);
      });
      point(r, ga);
      if (two) point(r + 1, gb);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();   // every read of the staged gradient is done
  if (valid) {
#pragma unroll
    for (int s = 0; s < N; ++s) {
      const int p = p0 + ps * s;
      if (fam) {
#pragma unroll
        for (int k = 0; k < 3; ++k) lds[LD::XA + (k * N2 + p) * T + ci] = D[s][k];
      } else {
#pragma unroll
        for (int k = 3; k < 7; ++k) lds[LD::XB + ((k - 3) * N2 + p) * T + ci] = D[s][k];
      }
    }
  }
  __syncthreads();
  if (!valid) return;
  double *o = va.visres + (size_t)tile * QT;
#pragma unroll
  for (int s = 0; s < N; ++s) {
    const int p = p0 + ps * s;
    double w[4];
    if (fam) {
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = D[s][3 + k] + lds[LD::XB + (k * N2 + p) * T + ci];
      store_vars<N, 4, 8>(o, p, ci, w);
    } else {
      w[0] = 0.0;   // rho has no viscous flux
#pragma unroll
      for (int k = 0; k < 3; ++k) w[1 + k] = D[s][k] + lds[LD::XA + (k * N2 + p) * T + ci];
      store_vars<N, 0, 4>(o, p, ci, w);
    }
  }
}

template <int N>
constexpr size_t vis_grad_lds_bytes() { return sizeof(double) * VisGradLds<N>::TOTAL; }
template <int N>
constexpr size_t vis_flux_lds_bytes() { return sizeof(double) * VisFluxLds<N>::TOTAL; }

}  // namespace sd2d
