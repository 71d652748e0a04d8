// visc_accuracy.cpp - the viscous flux (vflux_n) and the internal energy (enei_of)
// of sd2d_visc.hpp, compiled with g++ against the CPU stand-ins of tests/emu,
// against 113-bit arithmetic, beside the same formulas in double with IEEE
// divisions.  Test infrastructure only.  Prints one line per output: its number,
// the rms error of the header's form and that of the divisions (of the fluxes
// relative to the largest component).
#include <quadmath.h>

#include <algorithm>
#include <cstddef>
#include <cstdio>
#include <random>

#include "sd2d_visc.hpp"

namespace emu {   // (no kernel runs here)
thread_local emu_dim3 tid3, bid3;
void syncthreads() {}
void wave_sync() {}
uint64_t shfl_xor_bits(uint64_t b, int) { return b; }
unsigned long long atomic_max(unsigned long long *p, unsigned long long) { return *p; }
}  // namespace emu

using namespace sd2d;

// getVfluxvectors (getrusanov.f90:197-294) contracted with (sx, sy), variables 1-7,
// in the header's own expressions with a division for every quotient
template <typename T>
static void flux(const T *q, const T *g, T mu, T eta, T sx, T sy, T *Fn) {
  const T h = 0.5, two = 2.0, lam = LAMBDA_V, kp = T(GAM) / T(PRANDTL);
  const T u = q[1] / q[0], v = q[2] / q[0], w = q[3] / q[0];
  const T nu = u * u + v * v + w * w, nb = q[5] * q[5] + q[6] * q[6] + q[7] * q[7];
  const T e = (q[4] - h * nu * q[0] - h * nb - h * (q[8] * q[8])) / q[0];
  T du[2], dv[2], dw[2], de[2];
  for (int d = 0; d < 2; ++d) {
    const T dr = g[d];
    du[d] = (g[2 + d] - dr * u) / q[0];
    dv[d] = (g[4 + d] - dr * v) / q[0];
    dw[d] = (g[6 + d] - dr * w) / q[0];
    const T ke = h * nu * dr + q[0] * (u * du[d] + v * dv[d] + w * dw[d]);
    const T pb = q[5] * g[10 + d] + q[6] * g[12 + d] + q[7] * g[14 + d];
    de[d] = (g[8 + d] - ke - pb - dr * e - q[8] * g[16 + d]) / q[0];
  }
  const T ux = du[0], uy = du[1], vx = dv[0], vy = dv[1], wx = dw[0], wy = dw[1];
  const T xx = mu * (two * ux + lam * (ux + vy)), yy = mu * (two * vy + lam * (ux + vy));
  const T xy = mu * (vx + uy), xz = mu * wx, yz = mu * wy;
  const T jx = eta * g[15], jy = -eta * g[14], jz = eta * (g[12] - g[11]);
  const T f4 = u * xx + v * xy + w * xz + mu * kp * de[0] + jz * q[6] - jy * q[7];
  const T g4 = u * xy + v * yy + w * yz + mu * kp * de[1] - jz * q[5] + jx * q[7];
  Fn[0] = xx * sx + xy * sy;
  Fn[1] = xy * sx + yy * sy;
  Fn[2] = xz * sx + yz * sy;
  Fn[3] = f4 * sx + g4 * sy;
  Fn[4] = -jz * sy;
  Fn[5] = jz * sx;
  Fn[6] = jx * sy - jy * sx;
}

template <typename T>
static T energy(const T *q) {
  const T h = 0.5, u = q[1] / q[0], v = q[2] / q[0], w = q[3] / q[0];
  return (((q[4] / q[0] - h * (u * u)) - h * (v * v)) - h * (w * w)) -
         h * (((q[5] * q[5] + q[6] * q[6]) + q[7] * q[7]) + q[8] * q[8]) / q[0];
}

int main() {
  using Q = __float128;
  std::mt19937_64 rng(1);
  std::normal_distribution<double> n;
  std::uniform_real_distribution<double> u(0.0, 1.0);
  const int M = 200000;
  double ea[8] = {}, eb[8] = {};
  for (int i = 0; i < M; ++i) {
    double q[9], g[18], a[7], b[7];
    Q qq[9], gq[18], c[7];
    for (int v = 0; v < 9; ++v) q[v] = v == 0 ? 0.5 + u(rng) : v == 4 ? 4.0 + u(rng) : 0.5 * n(rng);
    for (double &x : g) x = n(rng);
    const double sx = n(rng), sy = n(rng);
    std::copy(q, q + 9, qq);
    std::copy(g, g + 18, gq);
    vflux_n(q, g, 0.01, 0.02, sx, sy, a);
    flux<double>(q, g, 0.01, 0.02, sx, sy, b);
    flux<Q>(qq, gq, 0.01, 0.02, sx, sy, c);
    double m = 0.0;
    for (Q x : c) m = std::max(m, (double)fabsq(x));
    for (int k = 0; k < 7; ++k) {
      const double x = (double)(a[k] - c[k]) / m, y = (double)(b[k] - c[k]) / m;
      ea[k] += x * x;
      eb[k] += y * y;
    }
    const Q e = energy<Q>(qq);
    const double x = (double)(enei_of(q) - e), y = (double)(energy<double>(q) - e);
    ea[7] += x * x;
    eb[7] += y * y;
  }
  for (int k = 0; k < 8; ++k) std::printf("%d %.6e %.6e\n", k, std::sqrt(ea[k] / M), std::sqrt(eb[k] / M));
  return 0;
}
