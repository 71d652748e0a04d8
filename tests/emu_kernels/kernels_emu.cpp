// kernels_emu.cpp - the device kernels as the library launches them: the line and
// the point form of the stage kernel and the mixed one on the rotating maxima with
// either metric table, the viscous kernels, and a traced stage with its reverse
// sweep.  The headers are compiled unchanged with g++ against the CPU stand-ins of
// tests/emu/hip/hip_runtime.h, with AddressSanitizer and UBSan, and run on host
// threads (one per work-item, real barriers) on buffers of exactly the library's
// sizes.  Buffers and LDS start as NaN and a canary follows each launch's LDS, so
// an access out of bounds, a barrier that not every work-item reaches, LDS written
// past the launch's size or a read of what nothing wrote shows up.  Test
// infrastructure only (tests/test_emu_kernels.py).
//
//   kernels_emu IN OUT        (one order per program: EMU_N)
//
// IN as for tests/emu/stage_emu.cpp; job is a sum of
//   0 / 1 / 2  what: nsteps RK steps / one residual / one traced stage and its pullback
//   4          stages by the point kernel (else by the line kernel)
//   8          the full metric table (else the compact one where the mesh allows it)
// OUT: steps    Q(9,N,N,NCELL), the maxima set read next (4 bit patterns), SM_IND,
//               residual and divB sums of the last step
//      residual resid, the maxima set, SM_IND
//      traced   Q + R(Q), Qbar = (dR/dQ)^T Rbar with Rbar after Q in IN, c_hbar and
//               pbar(6); c_h of the maxima 2.3, 0.7
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "hip/hip_runtime.h"
// (named by kernels that are not run here: drag_kernel, adj_tail_kernel)
inline int __syncthreads_or(int) { return 0; }
static const emu_dim3 blockDim{0, 0, 0};

#include "sd2d_host.hpp"
#include "sd2d_rkseq.hpp"
#include "sd2d_stage_mx.hpp"
#include "sd2d_stage_pt.hpp"
#include "sd2d_visc.hpp"
#include "sd2d_adj.hpp"

// ---- the launch model ---------------------------------------------------------
namespace sd2d {
constexpr size_t LDS_BYTES = 163840, CANARY = 8192;
alignas(16) double lds[(LDS_BYTES + CANARY) / 8];
}  // namespace sd2d

namespace emu {
thread_local emu_dim3 tid3{0, 0, 0}, bid3{0, 0, 0};
constexpr int MAXT = 1024;
constexpr uint64_t POISON = 0x7FC07FC07FC07FC0ull;   // NaN as a double and as two floats

struct Group {
  int live = 0, arrived = 0;
  unsigned long gen = 0;
};
static std::mutex mtx, atomic_mtx;
static std::condition_variable cv[1 + MAXT / 64];
static Group grp[1 + MAXT / 64];   // the workgroup, then its wavefronts
static uint64_t xch[MAXT];
static bool gone[MAXT];

[[noreturn]] static void die(const std::string &msg) {
  std::fprintf(stderr, "emu: %s (workgroup %u, work-item %u)\n", msg.c_str(), bid3.x, tid3.x);
  std::fflush(stderr);
  std::abort();
}
static void release(int g) {
  grp[g].arrived = 0;
  ++grp[g].gen;
  cv[g].notify_all();
}
static void meet(int g, std::unique_lock<std::mutex> &lk) {
  const unsigned long my = grp[g].gen;
  if (++grp[g].arrived == grp[g].live) return release(g);
  if (!cv[g].wait_for(lk, std::chrono::seconds(120), [&] { return grp[g].gen != my; }))
    die("a barrier that not every live work-item reaches");
}
static int wave() { return 1 + (int)(tid3.x >> 6); }

void syncthreads() {
  std::unique_lock<std::mutex> lk(mtx);
  meet(0, lk);
}
void wave_sync() {
  std::unique_lock<std::mutex> lk(mtx);
  meet(wave(), lk);
}
uint64_t shfl_xor_bits(uint64_t b, int mask) {
  std::unique_lock<std::mutex> lk(mtx);
  const int t = (int)tid3.x, p = (t & ~63) | ((t & 63) ^ mask);
  if (mask < 0 || mask > 63) die("__shfl_xor lane mask outside the wavefront");
  xch[t] = b;
  meet(wave(), lk);
  if (gone[p]) die("__shfl_xor reads the lane of a work-item that has returned");
  const uint64_t r = xch[p];
  meet(wave(), lk);
  return r;
}
unsigned long long atomic_max(unsigned long long *p, unsigned long long v) {
  std::lock_guard<std::mutex> lk(atomic_mtx);
  const unsigned long long old = *p;
  if (v > old) *p = v;
  return old;
}

// nblocks workgroups of nthreads work-items with `bytes` of LDS, one after another
template <class F>
static void launch(int nblocks, int nthreads, size_t bytes, F &&body) {
  if (bytes > sd2d::LDS_BYTES) die("launch asks for more LDS than a CU has");
  for (int b = 0; b < nblocks; ++b) {
    for (int w = 0; w <= nthreads / 64; ++w) grp[w] = Group{w ? 64 : nthreads, 0, 0};
    for (int t = 0; t < nthreads; ++t) gone[t] = false;
    for (double &x : sd2d::lds) std::memcpy(&x, &POISON, 8);
    std::vector<std::thread> th;
    for (int t = 0; t < nthreads; ++t)
      th.emplace_back([&, t, b] {
        tid3 = emu_dim3{(unsigned)t, 0, 0};
        bid3 = emu_dim3{(unsigned)b, 0, 0};
        body();
        std::lock_guard<std::mutex> lk(mtx);
        gone[t] = true;
        for (int g : {0, wave()})
          if (--grp[g].live > 0 && grp[g].arrived == grp[g].live) release(g);
      });
    for (auto &x : th) x.join();
    const unsigned char *c = reinterpret_cast<const unsigned char *>(sd2d::lds);
    for (size_t i = bytes; i < sizeof(sd2d::lds); ++i)
      if (c[i] != reinterpret_cast<const unsigned char *>(&POISON)[i % 8])
        die("LDS written at byte " + std::to_string(i) + " beyond the launch's " + std::to_string(bytes));
  }
}
}  // namespace emu

// ---- the library's buffers and launches -----------------------------------------
namespace {
using namespace sd2d;
using u64 = unsigned long long;

template <class T>
std::vector<T> dev(size_t n) {   // uninitialised device memory
  std::vector<T> v(n);
  for (T &x : v) std::memcpy(&x, &emu::POISON, sizeof(T));
  return v;
}

struct Ctx {
  int N, nc, nt, cpw, mixed, pt, mset = 0, cur = 0, sfam = 1;
  long nlaunch = 0;
  HostTables tb;
  sd2d_params p{};
  std::vector<double> q[3], fsr[3], sm_ind, normbuf, resid, gq, visres, dei, divb, tmax, part;
  std::vector<int> tinfo, tloc;
  std::vector<u64> maxs, gm;
  std::vector<float> metf;
  std::vector<Phys> phm;
  OpsF opsf{};
};

u64 *max_set(Ctx &c, int k) { return c.maxs.data() + MSTRIDE * (k % 3); }

template <int N, int MODE>
void stage(Ctx &c, const StageArgs &a) {
  if constexpr ((MODE & (M_COMPAT | M_VIS | M_TRACE)) == 0) {
    if (c.mixed)
      return emu::launch(c.nt, STAGE_THREADS, stage_mx_lds_bytes<N, MODE>(), [&] {
        stage_kernel_mx<N, MODE>(a, c.opsf, c.metf.data());
      });
  }
  if constexpr (pt_mode(MODE)) {
    if (c.pt)
      return emu::launch(c.nt, PT_THREADS<N>, stage_pt_lds_bytes<N, MODE>(), [&] {
        stage_pt_kernel<N, MODE>(a, c.tb.ops);
      });
  }
  emu::launch(c.nt, STAGE_THREADS, stage_lds_bytes<N, MODE>(),
              [&] { stage_kernel<N, MODE>(a, c.tb.ops); });
}

template <int N>
int stage_n(Ctx &c, const StageArgs &a, int mode) {
  constexpr int R = M_RK, A1 = M_AUX1, A4 = M_AUX4, V = M_AV, NR = M_NORMS;
  switch (mode) {
#define MODE(m) case (m): stage<N, (m)>(c, a); return 0;
    MODE(M_COMPAT | V) MODE(M_COMPAT | M_VIS | V) MODE(M_TRACE | R)
    MODE(R) MODE(R | A1) MODE(R | A1 | V | NR)
    MODE(M_VIS | R) MODE(M_VIS | R | A1) MODE(M_VIS | R | A1 | V | NR)
#undef MODE
    case R | A1 | M_RSTORE: if (!c.mixed) { stage<N, R | A1 | M_RSTORE>(c, a); return 0; } break;
    case R | A4 | V | NR: if (!c.mixed) { stage<N, R | A4 | V | NR>(c, a); return 0; } break;
  }
  std::fprintf(stderr, "emu: stage mode %d is not built into the emulator\n", mode);
  return 1;
}

template <int N>
void viscous(Ctx &c, const double *q) {
  VisArgs va{};
  va.qin = q; va.ftab = c.tb.ft.data(); va.met = c.tb.met.data(); va.mcomp = c.tb.mcomp;
  va.metw = c.tb.metw.data(); va.gq = c.gq.data(); va.dei = c.dei.empty() ? nullptr : c.dei.data();
  va.visres = c.visres.data(); va.mu = c.p.mu; va.eta0 = c.p.eta0; va.ntile = c.nt;
  va.walls = !c.dei.empty(); va.tinfo = c.tinfo.data(); va.sfam = c.sfam;
  emu::launch(c.nt, STAGE_THREADS, vis_grad_lds_bytes<N>(),
              [&] { vis_grad_kernel<N>(va, c.tb.ops, c.tb.ph); });
  va.rev = 1;
  emu::launch(c.nt, VIS_FLUX_THREADS, vis_flux_lds_bytes<N>(),
              [&] { vis_flux_kernel<N>(va, c.tb.ops, c.tb.ph); });
}

// one evaluation: the viscous kernels, the stage kernel, the rotation of the maxima
int evaluate(Ctx &c, StageArgs &a, int mode) {
  a.rev = (int)(c.nlaunch++ & 1);
  a.mread = max_set(c, c.mset);
  a.mwrite = max_set(c, c.mset + 1);
  a.mclear = max_set(c, c.mset + 2);
  if (c.p.mu != 0.0 || c.p.eta0 != 0.0) {
    viscous<EMU_N>(c, a.qin);
    a.visres = c.visres.data();
    mode |= M_VIS;
  }
  const int r = stage_n<EMU_N>(c, a, mode);
  c.mset = (c.mset + 1) % 3;
  return r;
}

StageArgs base_args(Ctx &c) {
  StageArgs a{};
  a.met = c.tb.met.data(); a.mcomp = c.tb.mcomp; a.ftab = c.tb.ft.data();
  std::copy(c.tb.av.begin(), c.tb.av.end(), a.avf);
  a.ncell = c.nc; a.ntile = c.nt; a.sm_ind = c.sm_ind.data(); a.s2c = c.tb.s2c.data();
  a.tinfo = c.tinfo.data(); a.phm = c.phm.data(); a.sfam = c.sfam;
  return a;
}

// Fortran layout (9,N,N,NCELL) to and from tiles
void tiles(Ctx &c, double *f, double *t, bool to) {
  const int N2 = c.N * c.N, QT = 9 * N2 * c.cpw;
  for (int cell = 0; cell < c.nc; ++cell)
    for (int p = 0; p < N2; ++p)
      for (int v = 0; v < 9; ++v) {
        const int sl = c.tb.c2s[cell];
        double &x = f[v + 9 * (p + (size_t)N2 * cell)];
        double &y = t[(size_t)(sl / c.cpw) * QT + qo_rt(c.N, v, p, sl % c.cpw)];
        (to ? y : x) = to ? x : y;
      }
}

template <class T>
void rd(std::ifstream &f, std::vector<T> &v, size_t n) {
  v.resize(n);
  if (n) f.read(reinterpret_cast<char *>(v.data()), (std::streamsize)(n * sizeof(T)));
  if (!f) {
    std::fprintf(stderr, "emu: input file too short\n");
    std::exit(2);
  }
}
}  // namespace

int main(int argc, char **argv) {
  if (argc != 3) return 2;
  std::ifstream f(argv[1], std::ios::binary);
  std::vector<int32_t> h, if2c, list[6], cyc;
  std::vector<double> pr, lmat, mmat, xs, xsl, jac, s1, s2, Q, Rb;
  rd(f, h, 16);
  rd(f, pr, 16);
  const int N = h[0], nc = h[1], N2 = N * N, what = h[12] & 3;
  if (N != EMU_N) return 2;
  rd(f, if2c, (size_t)4 * h[2]);
  for (int i = 0; i < 6; ++i) rd(f, list[i], (size_t)h[3 + i]);
  rd(f, cyc, (size_t)2 * h[9]);
  rd(f, lmat, (size_t)(N + 1) * N);
  rd(f, mmat, (size_t)(N + 1) * N);
  rd(f, xs, N);
  rd(f, xsl, N - 1);
  rd(f, jac, (size_t)N2 * nc);
  rd(f, s1, (size_t)4 * (N + 1) * N * nc);
  rd(f, s2, (size_t)4 * N * (N + 1) * nc);
  rd(f, Q, (size_t)9 * N2 * nc);
  if (what == 2) rd(f, Rb, Q.size());

  sd2d_mesh m{};
  m.N = N; m.ncell = nc; m.nface = h[2]; m.if2c = if2c.data();
  m.ninter = h[3]; m.ibfinter = list[0].data();
  m.ninlet = h[4]; m.ibfinl = list[1].data();
  m.noutlet = h[5]; m.ibfout = list[2].data();
  m.nwall = h[6]; m.ibfwal = list[3].data();
  m.nsymp = h[7]; m.ibfsymp = list[4].data();
  m.nfree = h[8]; m.ibfree = list[5].data();
  m.npair = h[9]; m.cyc2fpair = cyc.data();
  m.lmat = lmat.data(); m.mmat = mmat.data(); m.xs = xs.data(); m.xs_low = xsl.data();
  m.jac = jac.data(); m.s1 = s1.data(); m.s2 = s2.data();
  Ctx c;
  sd2d_params &p = c.p;
  p.vismode = 1; p.artiv = h[11]; p.mu = pr[0]; p.eta0 = pr[1]; p.alpha = pr[2];
  p.rinf = pr[3]; p.pinf = pr[4]; p.uinf = pr[5]; p.vinf = pr[6]; p.bxinf = pr[7];
  p.byinf = pr[8]; p.dxcycl = pr[9]; p.dycycl = pr[10]; p.ncellglob = nc; p.k_stage = h[10];
  p.dt = pr[11]; p.precision = h[14]; p.tile_shape = h[15];
  std::string err;
  if (build_host_tables(&m, &p, c.tb, err, !(h[12] & 8) && lines_share_metrics(&m))) {
    std::fprintf(stderr, "emu: host tables: %s\n", err.c_str());
    return 3;
  }
  c.N = N; c.nc = nc; c.nt = c.tb.ntile; c.cpw = c.tb.cpw;
  c.mixed = p.precision == SD2D_MIXED;
  c.pt = (h[12] & 4) != 0;
  const size_t np = (size_t)c.nt * N2 * c.cpw, qn = 9 * np;
  for (auto &x : c.q) x = dev<double>(qn);
  if (p.k_stage == 5)
    for (auto &x : c.fsr) x = dev<double>(qn);
  c.tinfo = c.tb.tvalid;
  c.tinfo[0] |= TI_FIRST;
  c.maxs.assign(3 * MSTRIDE, 0);
  for (int k = 0; k < 3; ++k) c.maxs[MSTRIDE * k + 2] = c.maxs[MSTRIDE * k + 3] = MAX_NONE;
  c.sm_ind = dev<double>(2 * (size_t)nc);
  c.normbuf = dev<double>(2 * (size_t)c.nt);
  c.resid = dev<double>(Q.size());
  std::vector<double> nabla = dev<double>(2 * Q.size());
  c.phm.assign(1, c.tb.ph);
  c.metf.assign(c.tb.met.begin(), c.tb.met.end());
  for (int i = 0; i <= N; ++i)
    for (int j = 0; j < N; ++j) {
      c.opsf.L[i][j] = (float)c.tb.ops.L[i][j];
      c.opsf.M[i][j] = (float)c.tb.ops.M[i][j];
    }
  if (p.mu != 0.0 || p.eta0 != 0.0) {
    c.gq = dev<double>(2 * qn);
    c.visres = dev<double>(qn);
    if (m.nwall > 0) c.dei = dev<double>(2 * np);
  }
  {   // the staging family: the one with fewer end faces in other tiles
    long long cross[2] = {0, 0};
    const int QT = 9 * N2 * c.cpw;
    for (int t = 0; t < c.nt; ++t)
      for (int k = 0; k < 4; ++k)
        for (int ci = 0; ci < c.cpw; ++ci) {
          const int *ft = c.tb.ft.data() + ((size_t)t * 8 + 2 * k) * c.cpw + ci;
          if (((ft[c.cpw] >> 3) & 7) == FT_INTERIOR && ft[0] / QT != t) ++cross[k == 1 || k == 3 ? 0 : 1];
        }
    c.sfam = cross[0] < cross[1] ? 0 : 1;
  }
  tiles(c, Q.data(), c.q[0].data(), true);
  if (what == 2) {   // sd2d_set_state with maxima: c_h is formed from the pair
    u64 *s = max_set(c, 0);
    const double e = 2.3, u = 0.7;
    s[0] = s[2] = as_bits(e);
    s[1] = s[3] = as_bits(u);
  }

  std::ofstream o(argv[2], std::ios::binary);
  auto put = [&](const void *d, size_t n) { o.write(static_cast<const char *>(d), (std::streamsize)(8 * n)); };
  const int av = p.artiv == 1 ? M_AV : 0;
  if (what == 0) {
    for (int s = 0; s < h[13]; ++s) {
      RkBuffers rb{{c.q[0].data(), c.q[1].data(), c.q[2].data()},
                   {c.fsr[0].data(), c.fsr[1].data(), c.fsr[2].data()}, c.cur};
      auto launch = [&](StageArgs &a, int mode) {
        if (mode & M_NORMS) a.normbuf = c.normbuf.data();
        return evaluate(c, a, mode);
      };
      const int r = p.k_stage == 5 ? fsrk_sequence(rb, p.dt, true, av, base_args(c), launch)
                                   : s5p3_sequence(rb, p.dt, true, av, base_args(c), launch);
      if (r) return 4;
      c.cur = rb.cur;
    }
    tiles(c, Q.data(), c.q[c.cur].data(), false);
    put(Q.data(), Q.size());
    put(max_set(c, c.mset), MSTRIDE);
    put(c.sm_ind.data(), c.sm_ind.size());
    double s[2] = {0.0, 0.0};
    for (int t = 0; t < c.nt; ++t)
      for (int k = 0; k < 2; ++k) s[k] += c.normbuf[2 * (size_t)t + k];
    put(s, 2);
  } else if (what == 1) {
    StageArgs a = base_args(c);
    a.qin = c.q[0].data();
    a.resid_f = c.resid.data();
    a.nabla_f = nabla.data();
    if (evaluate(c, a, M_COMPAT | av)) return 4;
    put(c.resid.data(), c.resid.size());
    put(max_set(c, c.mset), MSTRIDE);
    put(c.sm_ind.data(), c.sm_ind.size());
  } else {
    // Qout = Q + R(Q), traced, then the reverse sweep of R
    c.divb = dev<double>(np);
    c.gm = dev<u64>(MSTRIDE);
    c.tmax = dev<double>(2 * (size_t)c.nt);
    c.tloc = dev<int>(2 * (size_t)c.nt);
    c.part = dev<double>((size_t)ADJ_NPART * c.nt);
    StageArgs a = base_args(c);
    a.qin = c.q[0].data();
    a.qout = c.q[1].data();
    a.cin = 1.0;
    a.cr = 1.0;
    a.divb = c.divb.data();
    a.gmrec = c.gm.data();
    a.tmax = c.tmax.data();
    a.tloc = c.tloc.data();
    if (evaluate(c, a, M_RK | M_TRACE)) return 4;
    // the recorded speeds are the largest of the evaluation, at points of the mesh
    double e = 0.0, u = 0.0;
    for (int t = 0; t < c.nt; ++t) {
      e = std::max(e, c.tmax[2 * (size_t)t]);
      u = std::max(u, c.tmax[2 * (size_t)t + 1]);
      for (int k = 0; k < 2; ++k) {
        const int slot = c.tloc[2 * (size_t)t + k] / ((N + 1) * N * 2);
        if (slot / c.cpw != t || c.tb.s2c[slot] < 0) emu::die("location code outside the tile's cells");
      }
    }
    const u64 *now = max_set(c, c.mset);
    if (now[0] != std::max(c.gm[0], as_bits(e)) || now[1] != std::max(c.gm[1], as_bits(u)))
      emu::die("traced speeds and running maxima differ");
    std::vector<double> rb = dev<double>(qn), qb = dev<double>(qn);
    tiles(c, Rb.data(), rb.data(), true);
    AdjArgs g{};
    g.q = c.q[0].data(); g.rbar = rb.data(); g.rscale = 1.0; g.divb = c.divb.data();
    g.met = c.tb.met.data(); g.mcomp = c.tb.mcomp; g.ftab = c.tb.ft.data(); g.tinfo = c.tinfo.data();
    g.phm = c.phm.data(); g.gm = c.gm.data(); g.qbar = qb.data(); g.part = c.part.data();
    g.alpha = c.tb.ph.alpha; g.ntile = c.nt;
    emu::launch(c.nt, STAGE_THREADS, adj_lds_bytes<EMU_N>(),
                [&] { adj_stage_kernel<EMU_N>(g, c.tb.ops); });
    tiles(c, Q.data(), c.q[1].data(), false);
    put(Q.data(), Q.size());
    tiles(c, Q.data(), qb.data(), false);
    put(Q.data(), Q.size());
    double s[ADJ_NPART] = {};
    for (int t = 0; t < c.nt; ++t)
      for (int k = 0; k < ADJ_NPART; ++k) s[k] += c.part[(size_t)ADJ_NPART * t + k];
    put(s, ADJ_NPART);
  }
  o.close();
  return o ? 0 : 5;
}
