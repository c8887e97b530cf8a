// Kernels that build a simulation's constants on the device: the spectral
// operator tables and the single-precision medium maps, evaluated in double
// precision and rounded once, as the host evaluates them for small problems.
//
// A 256^3 absorbing problem has four tables of 8.5 million entries (a sine,
// a cosine or a power each) and seven maps of 16.8 million.  Built by sixteen
// host threads and copied one by one from pageable vectors its creation took
// 254 ms, bound by the page faults of the vectors and by pow; 43 ms with the
// tables written where they are read and the maps crossing the bus once, in
// double precision: the kernel reads them from two pinned chunks, of which one
// fills while it reads the other.
#pragma once

#include <cmath>

#include "kw_prob.h"

namespace kw {

enum SetupKind : int32_t {
  SETUP_SINC = 0,  // table of sinc(c_ref |k| dt / 2) (1 without the k-space method)
  SETUP_COS,       // table of cos(c_ref |k| dt / 2)
  SETUP_POW,       // table of |k|^expo, 0 where that is infinite
  SETUP_F32,       // map: out[0] = x
  SETUP_INV,       // map: out[0] = 1 / x
  SETUP_C0,        // sound speed: out[0] = x, out[1] = tau, out[2] = eta
};

struct SetupArgs {
  int32_t kind;
  int64_t n;          // elements of the launch
  // tables: half-spectrum geometry and the last-axis pass's tile order
  int32_t dim, Nx, Ny, Nz, Wm, nyq, Pn;
  double d[3];
  double c_ref, dt, expo, ntot;
  int32_t use_k;
  // maps: a chunk of doubles and the outputs it fills
  const double* src;
  float* out[3];
  double tau, tau_expo, eta, eta_expo;  // coefficient and power of the sound speed
};

KW_BODY double setup_k(int i, int N, double d) {
  const int n = (i < (N + 1) / 2) ? i : i - N;
  return (2.0 * 3.14159265358979323846264338327950288 / d) * ((double)n / (double)N);
}

constexpr int SETUP_T = 256;

template <class Ctx>
KW_BODY void body_setup(Ctx& c, const SetupArgs& A) {
  const int64_t e = (int64_t)c.bid() * SETUP_T + c.tid();
  if (e >= A.n) return;
  if (A.kind >= SETUP_F32) {
    const double x = KW_LD(A.src + e);
    KW_ST(A.out[0] + e, (float)(A.kind == SETUP_INV ? 1.0 / x : x));
    if (A.kind == SETUP_C0) {
      if (A.out[1]) KW_ST(A.out[1] + e, (float)(A.tau * pow(x, A.tau_expo)));
      if (A.out[2]) KW_ST(A.out[2] + e, (float)(A.eta * pow(x, A.eta_expo)));
    }
    return;
  }
  // element n of pencil p of tile t at (t N + n) Pn + p; the tiles of the
  // main block first, then those of the Nyquist plane; padding pencils zero
  const bool d3 = A.dim == 3;
  const int N = d3 ? A.Nz : A.Ny;
  const int64_t nH = d3 ? (int64_t)A.Wm * A.Ny : (int64_t)A.Wm;
  const int64_t nQ = A.nyq ? (d3 ? A.Ny : 1) : 0;
  const int64_t tH = (nH + A.Pn - 1) / A.Pn;
  const int p = (int)(e % A.Pn);
  const int64_t r = e / A.Pn;
  const int n = (int)(r % N);
  const int64_t tile = r / N;
  const bool main = tile < tH;
  const int64_t q = (main ? tile : tile - tH) * A.Pn + p;
  float v = 0.f;
  if (q < (main ? nH : nQ)) {
    const int ix = main ? (int)(q % A.Wm) : A.Nx / 2;
    const int iy = d3 ? (main ? (int)(q / A.Wm) : (int)q) : n;
    const double kx = setup_k(ix, A.Nx, A.d[0]), ky = setup_k(iy, A.Ny, A.d[1]);
    double k2 = kx * kx + ky * ky;
    if (d3) {
      const double kz = setup_k(n, A.Nz, A.d[2]);
      k2 = k2 + kz * kz;
    }
    const double k = sqrt(k2);
    double w = 1.0;
    if (A.kind == SETUP_POW) {
      w = pow(k, A.expo);
      if (!(w <= 1.7976931348623157e308)) w = 0.0;
    } else if (A.use_k) {
      const double x = A.c_ref * k * A.dt / 2;
      if (A.kind == SETUP_COS)
        w = cos(x);
      else
        w = x == 0.0 ? 1.0 : sin(x) / x;
    }
    v = (float)(w / A.ntot);
  }
  KW_ST(A.out[0] + e, v);
}

}  // namespace kw
