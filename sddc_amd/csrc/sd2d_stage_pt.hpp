// sd2d_stage_pt.hpp - the stage kernel of meshes too small to fill the chip.
//
// The same tiles and arithmetic as stage_kernel, and the same state, maxima and
// sensor bit for bit (a run made alone and as a member of a large ensemble agree;
// the norms are summed in another order), split finer: one
// wavefront per (line family, flux-point number), so a thread forms the flux of
// one flux point of one line, then one thread per solution point and half of
// its variables.  With less than one tile per CU the line
// kernel leaves half the SIMDs idle and each busy one issues a whole line (two
// Rusanov fluxes and N-1 interior ones) from one wavefront; here a tile's four
// face wavefronts sit on four SIMDs and the interior points run between their
// dependent FP64 instructions.
//
// The fluxes go to the solution points through LDS instead of the derivatives:
// every point sums its 2(N+1) fluxes in the line kernel's order.  That is three
// times the line kernel's LDS traffic and one tile takes 52-88 KB, which is
// why a full chip keeps the line kernel.
// Bound by the chain launch - face words - neighbour line - flux - update.
// One stage, this kernel against the line kernel, us: 16 x 32 cells, N = 3, 4, 5:
// 8.2 / 9.2 / 10.2 against 10.9 / 10.1 / 11.8; 32 x 64, N = 4 (128 tiles): 9.4
// against 10.2; 64 x 64, N = 4 (256 tiles, one per CU): 9.8 against 10.8.  With
// more than one tile per CU it loses: 342 tiles, N = 5: 19.0 against 16.3; 512
// tiles, N = 4: 16.7 against 14.8; 8192 tiles, N = 4: 236 against 127.
// 20 steps of 32 x 64 cells, N = 4, with the state's download: 1384 -> 1276 us; a
// step of 13 x 9 cells, N = 3, by host stages and downloads: 140 us.
#pragma once
#include "sd2d_stage.hpp"

namespace sd2d {

template <int N> constexpr int PT_THREADS = 64 * 2 * (N + 1);

// the modes with this form: inviscid stepping that stores nothing but the state,
// the residual register, the norms and the sensor
constexpr bool pt_mode(int mode) {
  return (mode & M_RK) != 0 && (mode & (M_COMPAT | M_VIS | M_DIVB | M_TRACE)) == 0;
}

// LDS of one workgroup (in doubles): the tile's state (qo layout); the flux
// points' values in pairs (variables 0-1, 2-3, 4-5, 6-7, then psi and the divB
// weight), [pair][fam][r][line][ci]{2}, and (AV) their Jz weights; (AV) Jz^2 of
// the points, then the sensor's line sums; the differentiation matrix
// [r][s]; reduction slots.
template <int N, int MODE> struct StagePtLds {
  static constexpr int T = Geo<N>::CPW, N2 = N * N, NF = N + 1, NW = 2 * NF;
  static constexpr bool AV = (MODE & M_AV) != 0, NORMS = (MODE & M_NORMS) != 0;
  static constexpr int NP = 2 * NF * N * T;    // flux points of the tile
  static constexpr int F = 9 * N2 * T;
  static constexpr int FJ = F + 10 * NP;
  static constexpr int XJ = FJ + (AV ? NP : 0);
  static constexpr int OM = XJ + (AV ? N2 * T : 0);
  static constexpr int RED = OM + NF * N;
  static constexpr int TOTAL = RED + (NORMS ? 2 * NW : 0);
  static_assert(F % 2 == 0, "pairs on 16-byte boundaries");
  static_assert(2 * N <= N2, "the AV line sums fit the Jz area");
  static constexpr int at(int pair, int pt) { return F + 2 * (pair * NP + pt); }
};

template <int N, int MODE>
constexpr size_t stage_pt_lds_bytes() { return sizeof(double) * StagePtLds<N, MODE>::TOTAL; }

template <int N, int MODE>
__global__ __launch_bounds__(PT_THREADS<N>) void stage_pt_kernel(StageArgs a, Ops ops) {
#pragma clang fp contract(on)   // as iflux_n<double>
  using G = Geo<N>;
  using LD = StagePtLds<N, MODE>;
  constexpr int T = G::CPW, N2 = G::N2, NF = N + 1, QT = G::QT, NT = PT_THREADS<N>;
  constexpr bool AV = (MODE & M_AV) != 0, NORMS = (MODE & M_NORMS) != 0;
  constexpr int NAUX = (MODE & M_AUX4) ? 4 : ((MODE & M_AUX1) ? 1 : 0);
  constexpr bool RSTORE = (MODE & M_RSTORE) != 0;
  constexpr int VS = 4;                        // variables 0..VS-1 | VS..8 of a point
  constexpr int PW = (N2 * T + 63) / 64;       // wavefronts of each half
  // the RK register is loaded with the first loads where 168 VGPRs hold it (3 waves
  // per SIMD)
  constexpr bool EARLY = N < 5 || !AV;
  static_assert(pt_mode(MODE) && N * T <= 64 && 2 * PW * 64 <= NT && NF * N <= NT, "thread layout");
  extern __shared__ double lds[];
  const int tid = threadIdx.x;
  const int tile = tile_of_block(blockIdx.x, a.ntile, a.rev);
  const int wv = wave_uniform(tid >> 6), l = tid & 63;
  // flux point r of the lines of family fam: the end faces are the first four
  // wavefronts, one per SIMD
  const bool face = wv < 4;
  const int fam = wv & 1;
  const int r = face ? (wv >> 1) * N : 1 + ((wv - 4) >> 1);
  const int line = l / T, ci = l % T;
  int nb = 0, info = 0;
  if (face) face_words<N>(a, tile, ci, fam, line, r, nb, info);
  const int ti = a.tinfo[tile];
  {
    constexpr int NV2 = 9 * N2 * T / 2, NR = (NV2 + NT - 1) / NT;
    const double2 *src = reinterpret_cast<const double2 *>(a.qin + (size_t)tile * QT);
    double2 *dst = reinterpret_cast<double2 *>(lds);
    double2 st[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int i = tid + k * NT;
      st[k] = src[(k < NR - 1 || i < NV2) ? i : 0];
    }
#pragma unroll
    for (int k = 0; k < NR; ++k)
      if (k < NR - 1 || tid + k * NT < NV2) dst[tid + k * NT] = st[k];
  }
  if (tid < NF * N) lds[LD::OM + tid] = (&ops.M[0][0])[(tid / N) * NMAX + tid % N];
  const int mem = ti >> 6, nvt = ti & TI_VALID;
  const bool valid = line < N && ci < nvt;
  const MetLine<N, double> ml(a.met, a.mcomp, tile, ci, fam, line);
  const double *qs = lds;
  // ---- the neighbour's trace of an end face in another tile, the point's
  //      metric vector, and what the solution point will need from memory ---------
  double qn[9];
  int lci = -1;
  if (face && valid && ((info >> 3) & 7) == FT_INTERIOR) {
    const int nt = nb / QT;
    lci = nb - nt * QT;
    if (nt != tile) {
      int k, nfp, np0, nst;
      bool endN;
      end_face<N>(fam, line, r, k, nfp);
      neighbour_line<N>(info & 3, nfp, np0, nst, endN);
      double Lr[N];
#pragma unroll
      for (int s = 0; s < N; ++s) Lr[s] = endN ? ops.L[N][s] : ops.L[0][s];
      line_vals<N, double>(a.qin + (size_t)nt * QT, np0, nst, lci, [&](int v, const double *vals) {
        qn[v] = line_trace<N, double>(vals, Lr);
      });
      lci = -1;
    }
  }
  double sx = 0.0, sy = 0.0;
  if (valid) {
    sx = ml.x[r * T];
    sy = ml.y[r * T];
  }
  const int part = wv / PW, pi = (wv - part * PW) * 64 + l, p = pi / T, pci = pi % T;
  const bool pvalid = part < 2 && pi < N2 * T && pci < nvt;
  const int is = p % N, js = p / N;
  const size_t off = (size_t)tile * QT;
  double ji = 0.0, ax[9 - VS];
  if (pvalid) {
    ji = MetLine<N, double>(a.met, a.mcomp, tile, pci, 0, 0).ji[(js + N * is) * T];
    if (NAUX == 1 && EARLY) {
      if (part == 0) load_vars<N, 0, VS>(a.aux[0] + off, p, pci, ax);
      else load_vars<N, VS, 9>(a.aux[0] + off, p, pci, ax);
    }
  }
  double ge, gu, me, mu;
  lagged_maxima(a, ti, tid, ge, gu, me, mu);
  const double cr = a.dtm ? a.cr * a.dtm[mem] : a.cr;   // b * dt of the member
  const Phys &ph = a.phm[mem];
  const double c_h = sqrt(ge * (ge - gu));   // compflux.f90:6
  double eig = 0.0, um = 0.0, nres = 0.0, ndiv = 0.0;
  __syncthreads();

  // ---- the flux of the thread's flux point (compflux.f90:53-104) -----------------
  if (valid) {
    if (lci >= 0) face_trace_lds<N, double>(qs, ops, info, fam, line, r, lci, qn);
    double t[9], F[9], wb, wj, Lr[N];
#pragma unroll
    for (int s = 0; s < N; ++s) Lr[s] = ops.L[r][s];
    line_vals<N, double>(qs, fam ? line : N * line, fam ? N : 1, ci, [&](int v, const double *vals) {
      t[v] = line_trace<N, double>(vals, Lr);
    });
    if (face) {
      double Qv[9];
      face_flux<N, double>(info, fam, r, ph, c_h, t, qn, sx, sy, F, Qv, eig, um);
      wb = Qv[5] * sx + Qv[6] * sy;
      wj = Qv[6] * sx - Qv[5] * sy;
    } else {
      iflux_n<double>(t, c_h, sx, sy, F, um);
      wb = t[5] * sx + t[6] * sy;
      wj = t[6] * sx - t[5] * sy;
    }
    const int pt = ((fam * NF + r) * N + line) * T + ci;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      *reinterpret_cast<double2 *>(lds + LD::at(u, pt)) = double2{F[2 * u], F[2 * u + 1]};
    *reinterpret_cast<double2 *>(lds + LD::at(4, pt)) = double2{F[8], wb};
    if (AV) lds[LD::FJ + pt] = wj;
  }
  raise_maxima(a, mem, eig, um, me, mu);
  __syncthreads();

  // ---- solution points: variables V0..V1-1 of point (is, js) -----------------------
  auto points = [&](auto v0c, auto v1c) __attribute__((always_inline)) {
    constexpr int V0 = decltype(v0c)::value, V1 = decltype(v1c)::value;
    // d(flux)/d(line coordinate), the end points first, then the interior ones
    // (the line kernel's order); xi plus eta
    double D[9], db = 0.0, dj = 0.0;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      double d[9], e = 0.0, g = 0.0;
      const int s = f ? js : is, ln = f ? is : js;
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        const int rr = i == 0 ? 0 : (i == 1 ? N : i - 1);
        const double m = lds[LD::OM + rr * N + s];
        const int pt = ((f * NF + rr) * N + ln) * T + pci;
        #pragma unroll
        for (int u = V0 / 2; u < (V1 < 9 ? V1 / 2 : 4); ++u) {
          const double2 w = *reinterpret_cast<const double2 *>(lds + LD::at(u, pt));
          d[2 * u] = i == 0 ? w.x * m : fma(w.x, m, d[2 * u]);
          d[2 * u + 1] = i == 0 ? w.y * m : fma(w.y, m, d[2 * u + 1]);
        }
        if (V1 == 9) {
          const double2 w = *reinterpret_cast<const double2 *>(lds + LD::at(4, pt));
          d[8] = i == 0 ? w.x * m : fma(w.x, m, d[8]);
          e = i == 0 ? w.y * m : fma(w.y, m, e);
        } else {
          const double w = lds[LD::at(4, pt) + 1];
          e = i == 0 ? w * m : fma(w, m, e);
        }
        if (AV && V0 == 0) {
          const double w = lds[LD::FJ + pt];
          g = i == 0 ? w * m : fma(w, m, g);
        }
      }
#pragma unroll
      for (int v = V0; v < V1; ++v) D[v] = f ? D[v] + d[v] : d[v];
      db = f ? db + e : e;
      dj = f ? dj + g : g;
    }
    double R[9], q[9];
    load_vars<N, 0, 8>(qs, p, pci, q);
    if (V1 == 9) q[8] = qs[qo<N>(8, p, pci)];
    // resid = -(dF/dxi + dG/deta) / J (compresid.f90:41,56)
#pragma unroll
    for (int v = V0; v < V1; ++v) R[v] = -D[v] * ji;
    const double divB = db * ji;
    const double ri = rcp(q[0]);
    const double ux = q[1] * ri, uy = q[2] * ri, uz = q[3] * ri;
    // Powell source and GLM damping, compresid.f90:58-74
    if (V0 == 0) {
      R[1] -= divB * q[5];
      R[2] -= divB * q[6];
      R[3] -= divB * q[7];
    } else {
      R[4] -= divB * (ux * q[5] + uy * q[6] + uz * q[7]);
      R[5] -= divB * ux;
      R[6] -= divB * uy;
      R[7] -= divB * uz;
      R[8] -= ph.alpha * q[8];
    }
    if (AV && V0 == 0) {
      const double jz = dj * ji;
      lds[LD::XJ + p * T + pci] = jz * jz;
    }
    if (NORMS) {
#pragma unroll
      for (int v = V0; v < V1; ++v) nres = fma(R[v], R[v], nres);
      if (V0 == 0) ndiv = fma(divB, divB, ndiv);
    }
    double xs[9];
    if (NAUX > 1) {
#pragma unroll
      for (int v = V0; v < V1; ++v) xs[v] = 0.0;
#pragma unroll
      for (int i = 0; i < NAUX; ++i) {
        double xv[9];
        load_vars<N, V0, V1>(a.aux[i] + off, p, pci, xv);
#pragma unroll
        for (int v = V0; v < V1; ++v) xs[v] = fma(a.ca[i], xv[v - V0], xs[v]);
      }
    }
    if (NAUX == 1 && !EARLY) load_vars<N, V0, V1>(a.aux[0] + off, p, pci, ax);
    double out[9];
#pragma unroll
    for (int v = V0; v < V1; ++v) {
      double acc = a.cin * q[v];
      if (NAUX == 1) acc = fma(a.ca[0], ax[v - V0], acc);
      if (NAUX > 1) acc += xs[v];
      out[v - V0] = fma(cr, R[v], acc);
    }
    store_vars<N, V0, V1>(a.qout + off, p, pci, out);
    if (RSTORE) store_vars<N, V0, V1>(a.rstore + off, p, pci, R + V0);
  };
  if (pvalid) {
    if (part == 0) points(std::integral_constant<int, 0>{}, std::integral_constant<int, VS>{});
    else points(std::integral_constant<int, VS>{}, std::integral_constant<int, 9>{});
  }

  // ---- norms (iterations.f90:37-46) and the AV sensor (AV.f90:14-83) ---------------
  if constexpr (NORMS) {
    nres = wave_sum(nres);
    ndiv = wave_sum(ndiv);
    if (l == 0) {
      lds[LD::RED + wv] = nres;
      lds[LD::RED + LD::NW + wv] = ndiv;
    }
  }
  if constexpr (NORMS || AV) __syncthreads();
  if constexpr (AV) {
    if (wv == 0) {   // (its lines are xi-lines)
      double rs[N], js2[N];
#pragma unroll
      for (int s = 0; s < N; ++s) {
        rs[s] = valid ? qs[qo<N>(0, N * line + s, ci)] : 1.0;
        js2[s] = valid ? lds[LD::XJ + (N * line + s) * T + ci] : 0.0;
      }
      av_sensor_lines<N, T, true, 2>(a, lds + qo<N>(0, 0, 0), lds + LD::XJ, lds + LD::XJ, rs, js2,
                                     line, ci, tile * T + ci, valid);
    }
  }
  if constexpr (NORMS) {
    if (tid == 64) {
      double s1 = 0.0, s2 = 0.0;
#pragma unroll
      for (int w = 0; w < 2 * PW; ++w) {
        s1 += lds[LD::RED + w];
        s2 += lds[LD::RED + LD::NW + w];
      }
      a.normbuf[2 * tile] = s1;
      a.normbuf[2 * tile + 1] = s2;
    }
  }
}

}  // namespace sd2d
