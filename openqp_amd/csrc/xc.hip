// xc.hip -- semilocal exchange-correlation build on the device: Vxc, E_xc and
// the grid electron count for the packed closed-shell or alpha/beta densities
// of OpenQP's Route-C Vxc seam (routec_vxc, source/modules/routec_bridge.F90:43-50;
// native path calc_dft_xc_density, source/scf_addons.F90:1857-1942 ->
// dmatd_density_blk, source/dftlib/dft_gridint_energy.F90:408-516).
//
// Grid: per atom a Treutler-Ahlrichs M4 radial grid (Chebyshev second kind,
// alpha = 0.6, per-element xi) times a Gauss-Legendre (cos theta) x uniform
// (phi) product angular grid, Stratmann-Scuseria-Frisch partition weights
// (a = 0.64) computed on the device, points with weight <= 1e-20 dropped.
// The kept points are sorted into cubic boxes (2 bohr) and cut into batches
// of at most 32768 points; a batch sees only the shells whose most diffuse
// primitive reaches its bounding box (|c| exp(-alpha r^2) >= 2.5e-13).
// Per-batch matrices are stored point-fastest (element (p, m) at m ld + p), so
// the kernels with one lane per point coalesce.
//
// Per group of batches, one launch each: phi (k_ao) -> X = phi D_b on the FP64
// matrix units and rho, grad rho from it (k_rho) -> the functional and its
// derivatives (forward-mode dual numbers, k_xc_point) -> Y = w (vrho/2 phi + v .
// grad phi) (k_y) -> V_b = phi^T Y (k_vmat) -> V += V_b (k_vsum); at the end V + V^T.
// Functionals: Slater, Becke 88, VWN (Ceperley-Alder "VWN5" and RPA fits),
// Lee-Yang-Parr, combined as libxc combines them for the names the reference
// accepts (source/dftlib/libxc.F90:300-460).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/oqph.h"
#include "ao_xform.h"
#include "session_view.h"

namespace oqph {
oqph_session* default_session();
void set_error_text(const char* msg);
}  // namespace oqph

namespace {

constexpr double PI = 3.14159265358979323846;
constexpr double RHO_CUT = 1e-10;    // points below this total density contribute nothing
constexpr double RHO_FLOOR = 1e-30;  // spin densities are floored here
constexpr double SSF_A = 0.64;
// bohr; the smaller, the fewer functions reach a batch and the more V_b there are.
// (H2O)32/6-31G(d): 4 bohr 23.2 ms per build (1.7e11 functions^2 points), 3 19.6, 2 15.9
// (0.94e11), 1.5 15.5 with twice the batches (13820) of 2, all at a cut-off of 1e-12
constexpr double BOX = 2.0;
constexpr int MAX_BATCH = 32768;
constexpr long long GROUP_ELEMS = 1ll << 28;  // basis-function values of a group of batches: 2 GB
// shells below it over a whole box are left out; with 1e-12 and 4-bohr boxes a build's
// error against exact functions was 7.9e-13 relative, on 2-bohr boxes 9.3e-13
constexpr double AO_EPS = 2.5e-13;

void err(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
void err(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  oqph::set_error_text(buf);
}

// ------------------------------------------------------------ functionals
enum Comp { C_LDAX = 0, C_B88, C_VWN5, C_VWNRPA, C_LYP };

struct XCFunc {
  int n;
  int comp[4];
  double w[4];
  double hfex;
  int gga;
};

bool lookup(const char* name, XCFunc* f) {
  std::string s(name ? name : "");
  for (auto& c : s) c = (char)tolower((unsigned char)c);
  if (s == "b3lypv5") s = "b3lyp5";
  if (s == "b3lypv1r") s = "b3lyp";
  if (s == "bhandhlyp") s = "bhhlyp";
  auto set = [&](std::initializer_list<std::pair<int, double>> cs, double hf) {
    f->n = 0;
    f->gga = 0;
    for (auto& c : cs) {
      f->comp[f->n] = c.first;
      f->w[f->n] = c.second;
      if (c.first == C_B88 || c.first == C_LYP) f->gga = 1;
      ++f->n;
    }
    f->hfex = hf;
  };
  if (s == "slater") set({{C_LDAX, 1.0}}, 0.0);
  else if (s == "svwn5") set({{C_LDAX, 1.0}, {C_VWN5, 1.0}}, 0.0);
  else if (s == "blyp") set({{C_B88, 1.0}, {C_LYP, 1.0}}, 0.0);
  else if (s == "b3lyp5") set({{C_LDAX, 0.08}, {C_B88, 0.72}, {C_VWN5, 0.19}, {C_LYP, 0.81}}, 0.20);
  else if (s == "b3lyp") set({{C_LDAX, 0.08}, {C_B88, 0.72}, {C_VWNRPA, 0.19}, {C_LYP, 0.81}}, 0.20);
  else if (s == "bhhlyp") set({{C_B88, 0.5}, {C_LYP, 1.0}}, 0.5);
  else return false;
  return true;
}

// forward-mode dual number over (rho_a, rho_b, sigma_aa, sigma_ab, sigma_bb)
struct Dual {
  double v, d[5];
};
__device__ inline Dual mk(double c) {
  Dual r;
  r.v = c;
  for (int k = 0; k < 5; ++k) r.d[k] = 0.0;
  return r;
}
__device__ inline Dual var(double x, int i) {
  Dual r = mk(x);
  r.d[i] = 1.0;
  return r;
}
__device__ inline Dual operator+(const Dual& a, const Dual& b) {
  Dual r;
  r.v = a.v + b.v;
  for (int k = 0; k < 5; ++k) r.d[k] = a.d[k] + b.d[k];
  return r;
}
__device__ inline Dual operator-(const Dual& a, const Dual& b) {
  Dual r;
  r.v = a.v - b.v;
  for (int k = 0; k < 5; ++k) r.d[k] = a.d[k] - b.d[k];
  return r;
}
__device__ inline Dual operator*(const Dual& a, const Dual& b) {
  Dual r;
  r.v = a.v * b.v;
  for (int k = 0; k < 5; ++k) r.d[k] = a.d[k] * b.v + a.v * b.d[k];
  return r;
}
__device__ inline Dual operator/(const Dual& a, const Dual& b) {
  Dual r;
  const double ib = 1.0 / b.v;
  r.v = a.v * ib;
  for (int k = 0; k < 5; ++k) r.d[k] = (a.d[k] - r.v * b.d[k]) * ib;
  return r;
}
__device__ inline Dual operator*(double c, const Dual& a) {
  Dual r;
  r.v = c * a.v;
  for (int k = 0; k < 5; ++k) r.d[k] = c * a.d[k];
  return r;
}
__device__ inline Dual operator+(double c, const Dual& a) {
  Dual r = a;
  r.v += c;
  return r;
}
__device__ inline Dual operator-(double c, const Dual& a) { return c + (-1.0) * a; }
__device__ inline Dual operator/(double c, const Dual& a) { return mk(c) / a; }
__device__ inline Dual chain(const Dual& a, double f, double fp) {
  Dual r;
  r.v = f;
  for (int k = 0; k < 5; ++k) r.d[k] = fp * a.d[k];
  return r;
}
__device__ inline Dual dpow(const Dual& a, double p) { return chain(a, pow(a.v, p), p * pow(a.v, p - 1.0)); }
__device__ inline Dual dexp(const Dual& a) {
  const double e = exp(a.v);
  return chain(a, e, e);
}
__device__ inline Dual dlog(const Dual& a) { return chain(a, log(a.v), 1.0 / a.v); }
__device__ inline Dual dsqrt(const Dual& a) {
  const double s = sqrt(a.v);
  return chain(a, s, 0.5 / s);
}
__device__ inline Dual datan(const Dual& a) { return chain(a, atan(a.v), 1.0 / (1.0 + a.v * a.v)); }
// g(y) = x asinh(x) with x = sqrt(y); g'(y) = asinh(x) / (2x) + 1 / (2 sqrt(1 + y)), -> 1 at y = 0
__device__ inline Dual dxasinhx(const Dual& y) {
  const double x = sqrt(y.v), as = asinh(x);
  const double g1 = (x > 1e-8 ? as / (2.0 * x) : 0.5) + 0.5 / sqrt(1.0 + y.v);
  return chain(y, x * as, g1);
}

// (3/4) (6/pi)^(1/3)
__device__ inline double cx() { return 0.75 * cbrt(6.0 / PI); }

__device__ Dual lda_x(const Dual& ra, const Dual& rb) { return (-cx()) * (dpow(ra, 4.0 / 3.0) + dpow(rb, 4.0 / 3.0)); }

__device__ Dual b88(const Dual& ra, const Dual& rb, const Dual& saa, const Dual& sbb) {
  const double beta = 0.0042;
  Dual out = mk(0.0);
  for (int s = 0; s < 2; ++s) {
    const Dual& r = s ? rb : ra;
    const Dual& sg = s ? sbb : saa;
    const Dual r43 = dpow(r, 4.0 / 3.0);
    const Dual y = sg / (r43 * r43);  // x^2
    out = out - cx() * r43 - beta * (r43 * y) / (1.0 + (6.0 * beta) * dxasinhx(y));
  }
  return out;
}

__device__ Dual vwn_aux(double A, double b, double c, double x0, const Dual& rs) {
  const Dual x = dsqrt(rs);
  const Dual X = x * x + b * x + mk(c);
  const double X0 = x0 * x0 + b * x0 + c, Q = sqrt(4.0 * c - b * b);
  const Dual at = datan(Q / (2.0 * x + mk(b)));
  const Dual xm = x + mk(-x0);
  return A * (dlog(x * x / X) + (2.0 * b / Q) * at -
              (b * x0 / X0) * (dlog(xm * xm / X) + (2.0 * (b + 2.0 * x0) / Q) * at));
}

__device__ Dual vwn(const Dual& ra, const Dual& rb, bool rpa) {
  const Dual r = ra + rb;
  const Dual rs = cbrt(3.0 / (4.0 * PI)) * dpow(r, -1.0 / 3.0);
  const Dual z = (ra - rb) / r;
  const double den = pow(2.0, 4.0 / 3.0) - 2.0;
  const Dual fz = (1.0 / den) * (dpow(1.0 + z, 4.0 / 3.0) + dpow(1.0 - z, 4.0 / 3.0) + mk(-2.0));
  if (rpa) {
    const Dual eP = vwn_aux(0.0310907, 13.0720, 42.7198, -0.409286, rs);
    const Dual eF = vwn_aux(0.01554535, 20.1231, 101.578, -0.743294, rs);
    return r * (eP * (1.0 - fz) + eF * fz);
  }
  const Dual eP = vwn_aux(0.0310907, 3.72744, 12.9352, -0.10498, rs);
  const Dual eF = vwn_aux(0.01554535, 7.06042, 18.0578, -0.32500, rs);
  const Dual ac = vwn_aux(-1.0 / (6.0 * PI * PI), 1.13107, 13.0045, -0.0047584, rs);
  const double fpp0 = 4.0 / (9.0 * (cbrt(2.0) - 1.0));
  const Dual z2 = z * z, z4 = z2 * z2;
  return r * (eP + (1.0 / fpp0) * (ac * fz * (1.0 - z4)) + (eF - eP) * fz * z4);
}

__device__ Dual lyp(const Dual& ra, const Dual& rb, const Dual& saa, const Dual& sab, const Dual& sbb) {
  const double a = 0.04918, b = 0.132, c = 0.2533, d = 0.349;
  const Dual r = ra + rb;
  const Dual rm = dpow(r, -1.0 / 3.0);
  const Dual den = 1.0 + d * rm;
  const Dual om = dexp((-c) * rm) / den * dpow(r, -11.0 / 3.0);
  const Dual dl = c * rm + d * rm / den;
  const double cf = 0.3 * pow(3.0 * PI * PI, 2.0 / 3.0);
  const Dual s = saa + 2.0 * sab + sbb;
  Dual t = ra * rb *
           ((pow(2.0, 11.0 / 3.0) * cf) * (dpow(ra, 8.0 / 3.0) + dpow(rb, 8.0 / 3.0)) +
            (47.0 / 18.0 - (7.0 / 18.0) * dl) * s - (2.5 - (1.0 / 18.0) * dl) * (saa + sbb) -
            (1.0 / 9.0) * (dl + mk(-11.0)) * (ra / r * saa + rb / r * sbb));
  const Dual r2 = r * r;
  t = t - (2.0 / 3.0) * r2 * s + ((2.0 / 3.0) * r2 - ra * ra) * sbb + ((2.0 / 3.0) * r2 - rb * rb) * saa;
  return (-4.0 * a) * (ra * rb / (r * den)) - (a * b) * om * t;
}

__device__ Dual energy_density(const XCFunc& f, const Dual& ra, const Dual& rb, const Dual& saa, const Dual& sab,
                               const Dual& sbb) {
  Dual e = mk(0.0);
  for (int i = 0; i < f.n; ++i) {
    Dual c;
    switch (f.comp[i]) {
      case C_LDAX: c = lda_x(ra, rb); break;
      case C_B88: c = b88(ra, rb, saa, sbb); break;
      case C_VWN5: c = vwn(ra, rb, false); break;
      case C_VWNRPA: c = vwn(ra, rb, true); break;
      default: c = lyp(ra, rb, saa, sab, sbb); break;
    }
    e = e + f.w[i] * c;
  }
  return e;
}

// ------------------------------------------------------------ grid kernel
struct GridArgs {
  const double* xyz;    // natm x 3
  const double* rinv;   // natm x natm inverse distances
  const double* rad;    // natm x nrad x 2 (r, w r^2 dr)
  const double* ang;    // nang x 4 (unit vector, weight)
  int natm, nrad, nang;
  long long n;          // natm nrad nang
  double* out;          // n x 4
};

__device__ inline double ssf_s(double mu) {
  if (mu <= -SSF_A) return 1.0;
  if (mu >= SSF_A) return 0.0;
  const double x = mu / SSF_A, x2 = x * x;
  const double g = x * (35.0 + x2 * (-35.0 + x2 * (21.0 - 5.0 * x2))) / 16.0;
  return 0.5 * (1.0 - g);
}

__device__ inline double dist(const double* xyz, int a, double x, double y, double z) {
  const double dx = x - xyz[3 * a], dy = y - xyz[3 * a + 1], dz = z - xyz[3 * a + 2];
  return sqrt(dx * dx + dy * dy + dz * dz);
}

// P_B = prod_{C != B} s(mu_BC) at (x, y, z), 0 as soon as a factor is 0
__device__ double cell(const GridArgs& g, int B, double dB, double x, double y, double z) {
  double P = 1.0;
  for (int C = 0; C < g.natm && P != 0.0; ++C) {
    if (C == B) continue;
    P *= ssf_s((dB - dist(g.xyz, C, x, y, z)) * g.rinv[(size_t)B * g.natm + C]);
  }
  return P;
}

__global__ void k_grid(GridArgs g) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= g.n) return;
  const int j = (int)(t % g.nang);
  const long long ar = t / g.nang;
  const int i = (int)(ar % g.nrad), A = (int)(ar / g.nrad);
  const double r = g.rad[((size_t)A * g.nrad + i) * 2], wr = g.rad[((size_t)A * g.nrad + i) * 2 + 1];
  const double* v = g.ang + 4 * j;
  const double x = g.xyz[3 * A] + r * v[0], y = g.xyz[3 * A + 1] + r * v[1], z = g.xyz[3 * A + 2] + r * v[2];
  double w = wr * v[3];
  if (g.natm > 1) {
    const double dA = dist(g.xyz, A, x, y, z);
    const double PA = cell(g, A, dA, x, y, z);
    double tot = 0.0;
    if (PA != 0.0) {
      for (int B = 0; B < g.natm; ++B) {
        if (B == A) {
          tot += PA;
          continue;
        }
        const double dB = dist(g.xyz, B, x, y, z);
        if (ssf_s((dB - dA) * g.rinv[(size_t)B * g.natm + A]) == 0.0) continue;  // factor C = A vanishes
        tot += cell(g, B, dB, x, y, z);
      }
    }
    w = PA != 0.0 ? w * (PA / tot) : 0.0;
  }
  double* o = g.out + 4 * t;
  o[0] = x;
  o[1] = y;
  o[2] = z;
  o[3] = w;
}

// ------------------------------------------------------------ batches and groups
// The batches are cut into groups of at most GROUP_ELEMS basis-function values (fewer
// where the device is short of memory); a build takes one launch of each kernel per
// group, over all its batches.  A launch per batch, three gathers of the density and three library products with
// phi, its gradient, X and Y in memory took 65 ms for (H2O)32/6-31G(d) with its
// 1045 batches of 4 bohr; this 15.9, and 17.0 with the present cut-off (groups of 2^25
// values: 28.1 against 23.8 for 2^28, both on boxes of 4 bohr).
struct DBatch {
  long long p0;   // first point of the grid
  long long off;  // first element of the batch's matrices in the group's arrays
  long long vb;   // first element of its partial V_b in the group's array
  int npts, ld;   // points, and rounded up to whole tiles of TILE
  int sh0, nsh, ao0, nb, nparts, pad;
};

struct AOTab {
  const int *am, *harm, *atom, *nprim, *poff;
  const double *ex, *cc, *xyz, *xf;
};

struct XArgs {
  AOTab ao;
  const double* pts;        // 4 per point (weight in [3])
  const DBatch* batch;      // all batches
  const int2* tile;         // the group's point tiles: batch, tile of the batch
  const int4* vt;           // the group's V_b tiles: batch, part, row tile, column tile (batch < 0: none)
  const int *shl, *col;     // significant shells and their first columns
  const int* idx;           // AO of every column
  double *phi, *Y;          // per batch and spin, point fastest: element (p, m) at off + m ld + p
  double *rho, *coef;       // [spin][4][npad]
  double* Vb;               // [spin][..]
  long long npad, ngrp, nvb;  // points of the group in whole tiles; elements of phi; of Vb per spin
};

constexpr int TILE = 64;

// Components of a shell at one point, in AO order: f(o, value, gradient)
template <int L, bool PURE, bool GRAD, typename F>
__device__ __forceinline__ void ao_shell_l(double dx, double dy, double dz, double R, double dR,
                                           const double* __restrict__ xf, F&& f) {
  constexpr int NC = (L + 1) * (L + 2) / 2;
  double px[L + 1], py[L + 1], pz[L + 1];
  px[0] = py[0] = pz[0] = 1.0;
#pragma unroll
  for (int k = 1; k <= L; ++k) {
    px[k] = px[k - 1] * dx;
    py[k] = py[k - 1] * dy;
    pz[k] = pz[k - 1] * dz;
  }
  double c[NC], g[3][GRAD ? NC : 1];
  int i = 0;  // canonical order: lx descending, then ly descending
#pragma unroll
  for (int lx = L; lx >= 0; --lx)
#pragma unroll
    for (int ly = L - lx; ly >= 0; --ly) {
      const int lz = L - lx - ly;
      const double m = px[lx] * py[ly] * pz[lz];
      c[i] = m * R;
      if constexpr (GRAD) {
        g[0][i] = (lx ? lx * px[lx > 0 ? lx - 1 : 0] * py[ly] * pz[lz] * R : 0.0) + m * dR * dx;
        g[1][i] = (ly ? ly * px[lx] * py[ly > 0 ? ly - 1 : 0] * pz[lz] * R : 0.0) + m * dR * dy;
        g[2][i] = (lz ? lz * px[lx] * py[ly] * pz[lz > 0 ? lz - 1 : 0] * R : 0.0) + m * dR * dz;
      }
      ++i;
    }
  if constexpr (L < 2) {
#pragma unroll
    for (int o = 0; o < NC; ++o) f(o, c[o], GRAD ? g[0][o] : 0.0, GRAD ? g[1][o] : 0.0, GRAD ? g[2][o] : 0.0);
  } else {
    constexpr int NO = PURE ? 2 * L + 1 : NC;
    const double* X = xf + ((L - 2) * 2 + (PURE ? 1 : 0)) * 100;
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      double v = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const double x = X[o * 10 + k];
        v += x * c[k];
        if constexpr (GRAD) {
          vx += x * g[0][k];
          vy += x * g[1][k];
          vz += x * g[2][k];
        }
      }
      f(o, v, vx, vy, vz);
    }
  }
}

// one shell (wavefront-uniform) at the lane's point
template <bool GRAD, typename F>
__device__ __forceinline__ void ao_shell(const AOTab& t, int sh, const double* r, F&& f) {
  const int l = t.am[sh], A = t.atom[sh], n = t.nprim[sh], k0 = t.poff[sh];
  const double dx = r[0] - t.xyz[3 * A], dy = r[1] - t.xyz[3 * A + 1], dz = r[2] - t.xyz[3 * A + 2];
  const double r2 = dx * dx + dy * dy + dz * dz;
  double R = 0.0, dR = 0.0;
  for (int k = 0; k < n; ++k) {
    const double al = t.ex[k0 + k], e = t.cc[k0 + k] * exp(-al * r2);
    R += e;
    if constexpr (GRAD) dR -= 2.0 * al * e;
  }
  if (l == 0) ao_shell_l<0, false, GRAD>(dx, dy, dz, R, dR, t.xf, f);
  else if (l == 1) ao_shell_l<1, false, GRAD>(dx, dy, dz, R, dR, t.xf, f);
  else if (l == 2 && t.harm[sh]) ao_shell_l<2, true, GRAD>(dx, dy, dz, R, dR, t.xf, f);
  else if (l == 2) ao_shell_l<2, false, GRAD>(dx, dy, dz, R, dR, t.xf, f);
  else if (t.harm[sh]) ao_shell_l<3, true, GRAD>(dx, dy, dz, R, dR, t.xf, f);
  else ao_shell_l<3, false, GRAD>(dx, dy, dz, R, dR, t.xf, f);
}

// the lane's point of tile t (the last one again past the end), its coordinates
__device__ __forceinline__ long long tile_point(const XArgs& a, const DBatch& b, int t, int lane, double* r) {
  const long long p = b.p0 + min(t * TILE + lane, b.npts - 1);
  for (int k = 0; k < 3; ++k) r[k] = a.pts[4 * p + k];
  return p;
}

// phi of one tile; a wavefront takes every fourth shell.  Bound by the 8 bytes it
// writes per value.  The gradients are evaluated again where they are used
// (k_rho, k_y): an exponential per primitive costs less than writing and reading
// three more arrays.
__global__ __launch_bounds__(256) void k_ao(XArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int2 tl = a.tile[blockIdx.x];
  const DBatch b = a.batch[tl.x];
  double r[3];
  tile_point(a, b, tl.y, lane, r);
  for (int q = wave; q < b.nsh; q += 4) {
    const int sh = a.shl[b.sh0 + q];
    double* out = a.phi + b.off + (size_t)a.col[b.sh0 + q] * b.ld + tl.y * TILE + lane;
    ao_shell<false>(a.ao, sh, r, [&](int o, double v, double, double, double) { out[(size_t)o * b.ld] = v; });
  }
}

// ------------------------------------------------------------ density on the grid
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

// rho and grad rho of one tile and spin: X = phi D_b on the FP64 matrix units,
// NV tiles of 16 columns per wavefront; phi through LDS (the four wavefronts share
// it), D through the column list (it stays in L2).  X meets phi and grad phi,
// evaluated per lane = point, through LDS and is never written.  Bound by the matrix
// units next to the exponentials: 7.0 ms for 9.4e10 columns^2 points ((H2O)32/
// 6-31G(d)), of which 5.1 the product (37 TFLOP/s) and 3.1 the functions alone.  Three
// wavefronts per SIMD (112 bytes of scratch in the f path) 7.0, two 7.6 ms; one pass
// over up to 192 columns with 12 tiles in registers 8.1.
template <int NV>
__device__ __forceinline__ void rho_pass(const double* __restrict__ ph, const double* __restrict__ Ds, int nbf, int nb,
                                         int ld, const int* s_idx, double* s_a, int n0, v4d (&acc)[4][2]) {
  constexpr int AS = 80;  // row length of the staged phi: rows 32 banks apart
  const int lane = threadIdx.x & 63, row = lane & 15, g = lane >> 4, sk = threadIdx.x >> 4, sp = (threadIdx.x & 15) * 4;
  const double* Dn[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) Dn[j] = Ds + s_idx[min(n0 + 16 * j + row, nb - 1)];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[t][j] = v4d{0.0, 0.0, 0.0, 0.0};
  v2d ra[2];
  double rb[4][NV];
  auto fetch = [&](int m0) {
    const bool ok = m0 + sk < nb;
    const double* pa = ph + (size_t)min(m0 + sk, nb - 1) * ld + sp;
#pragma unroll
    for (int h = 0; h < 2; ++h) ra[h] = ok ? *(const v2d*)(pa + 2 * h) : v2d{0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const size_t dr = (size_t)s_idx[min(m0 + 4 * k + g, nb - 1)] * nbf;
#pragma unroll
      for (int j = 0; j < NV; ++j) rb[k][j] = Dn[j][dr];
    }
  };
  fetch(0);
  for (int m0 = 0, cur = 0; m0 < nb; m0 += 16, cur ^= 1) {
    double* A = s_a + cur * 16 * AS;
#pragma unroll
    for (int h = 0; h < 2; ++h) *(v2d*)(A + sk * AS + sp + 2 * h) = ra[h];
    double y[4][NV];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < NV; ++j) y[k][j] = rb[k][j];
    __syncthreads();
    if (m0 + 16 < nb) fetch(m0 + 16);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      double x[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) x[t] = A[(4 * k + g) * AS + 16 * t + row];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t], y[k][j], acc[t][j], 0, 0, 0);
    }
  }
  __syncthreads();
}

template <bool GGA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_rho(XArgs a,
                                                                                   const double* __restrict__ D, int nbf) {
  extern __shared__ __align__(16) double s_dyn[];
  constexpr int XS = 16 * (TILE + 1);
  const int lane = threadIdx.x & 63, row = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double* s_x = s_dyn + wave * XS;
  int* s_idx = (int*)(s_dyn + 4 * XS);
  const int2 tl = a.tile[blockIdx.x];
  const DBatch b = a.batch[tl.x];
  const int nb = b.nb, ld = b.ld;
  for (int i = threadIdx.x; i < nb; i += 256) s_idx[i] = a.idx[b.ao0 + i];
  __syncthreads();
  const double* Ds = D + (size_t)blockIdx.y * nbf * nbf;
  double r[3];
  tile_point(a, b, tl.y, lane, r);
  const double* ph = a.phi + b.off + tl.y * TILE;
  double o0 = 0.0, o1 = 0.0, o2 = 0.0, o3 = 0.0;
  int q = 0;  // first shell that reaches the present columns
  for (int base = 0; base < nb;) {
    // 128 columns, or 64 where no more are left
    const int nv = nb - base <= 64 ? 1 : 2, n0 = base + 16 * nv * wave;
    v4d acc[4][2];
    if (nv == 1) rho_pass<1>(ph, Ds, nbf, nb, ld, s_idx, s_dyn, n0, acc);
    else rho_pass<2>(ph, Ds, nbf, nb, ld, s_idx, s_dyn, n0, acc);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c0 = n0 + 16 * j;
      if (j >= nv || c0 >= nb) break;
      // element i of a lane's result: point 16 t + 4 i + lane / 16, column lane % 16
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_x[row * (TILE + 1) + 16 * t + 4 * i + g] = acc[t][j][i];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      while (q + 1 < b.nsh && a.col[b.sh0 + q + 1] <= c0) ++q;
      for (int k = q; k < b.nsh && a.col[b.sh0 + k] < c0 + 16; ++k) {
        const int cs = a.col[b.sh0 + k] - c0;
        ao_shell<GGA>(a.ao, a.shl[b.sh0 + k], r, [&](int o, double v, double vx, double vy, double vz) {
          const int c = cs + o;
          if (c < 0 || c >= 16) return;
          const double x = s_x[c * (TILE + 1) + lane];
          o0 += x * v;
          if constexpr (GGA) {
            o1 += x * vx;
            o2 += x * vy;
            o3 += x * vz;
          }
        });
      }
    }
    base += 64 * nv;
    __syncthreads();
  }
  double* red = s_dyn + wave * 4 * TILE;
  red[lane] = o0;
  red[TILE + lane] = o1;
  red[2 * TILE + lane] = o2;
  red[3 * TILE + lane] = o3;
  __syncthreads();
  // thread = (quantity, point): the sum over the four wavefronts
  double v = 0.0;
  for (int w = 0; w < 4; ++w) v += s_dyn[w * 4 * TILE + threadIdx.x];
  a.rho[((size_t)blockIdx.y * 4 + wave) * a.npad + (size_t)blockIdx.x * TILE + lane] = v;
}

__device__ inline double wsum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The functional, lane = point: rho, grad rho -> the coefficients of phi and grad
// phi in Y; E_xc and the electron count into acc
__global__ __launch_bounds__(256) void k_xc_point(XArgs a, long long ntile, int ns, XCFunc f, double* acc) {
  const int lane = threadIdx.x & 63;
  double es = 0.0, nel = 0.0;
  for (long long tile = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); tile < ntile; tile += 4ll * gridDim.x) {
    const int2 tl = a.tile[tile];
    const DBatch& b = a.batch[tl.x];
    const int p = tl.y * TILE + lane;
    const size_t at = (size_t)tile * TILE + lane;
    const bool live = p < b.npts;
    double rho[2], g[2][3];
    for (int s = 0; s < ns; ++s) {
      rho[s] = a.rho[(size_t)s * 4 * a.npad + at];
      for (int k = 0; k < 3; ++k) g[s][k] = 2.0 * a.rho[((size_t)s * 4 + k + 1) * a.npad + at];
    }
    double ra, rb, ga[3], gb[3];
    if (ns == 1) {
      ra = rb = 0.5 * rho[0];
      for (int k = 0; k < 3; ++k) ga[k] = gb[k] = 0.5 * g[0][k];
    } else {
      ra = rho[0];
      rb = rho[1];
      for (int k = 0; k < 3; ++k) {
        ga[k] = g[0][k];
        gb[k] = g[1][k];
      }
    }
    const double w = live ? a.pts[4 * (b.p0 + p) + 3] : 0.0, rt = ra + rb;
    double c0[2] = {0.0, 0.0}, vec[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
    if (live && rt >= RHO_CUT) {
      const double saa = ga[0] * ga[0] + ga[1] * ga[1] + ga[2] * ga[2];
      const double sab = ga[0] * gb[0] + ga[1] * gb[1] + ga[2] * gb[2];
      const double sbb = gb[0] * gb[0] + gb[1] * gb[1] + gb[2] * gb[2];
      const Dual F = energy_density(f, var(fmax(ra, RHO_FLOOR), 0), var(fmax(rb, RHO_FLOOR), 1), var(saa, 2),
                                    var(sab, 3), var(sbb, 4));
      es += w * F.v;
      c0[0] = 0.5 * w * F.d[0];
      c0[1] = 0.5 * w * F.d[1];
      for (int k = 0; k < 3; ++k) {
        vec[0][k] = w * (2.0 * F.d[2] * ga[k] + F.d[3] * gb[k]);
        vec[1][k] = w * (2.0 * F.d[4] * gb[k] + F.d[3] * ga[k]);
      }
    }
    if (live) nel += w * rt;
    for (int s = 0; s < ns; ++s) {
      a.coef[(size_t)s * 4 * a.npad + at] = c0[s];
      for (int k = 0; k < 3; ++k) a.coef[((size_t)s * 4 + k + 1) * a.npad + at] = vec[s][k];
    }
  }
  es = wsum(es);
  nel = wsum(nel);
  if (lane == 0) {
    atomicAdd(acc, es);
    atomicAdd(acc + 1, nel);
  }
}

// Y = c phi + v . grad phi of one tile and spin, as k_ao; zero past the batch's points
template <bool GGA>
__global__ __launch_bounds__(256) void k_y(XArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int2 tl = a.tile[blockIdx.x];
  const DBatch b = a.batch[tl.x];
  double r[3];
  tile_point(a, b, tl.y, lane, r);
  const double* cf = a.coef + (size_t)blockIdx.y * 4 * a.npad + (size_t)blockIdx.x * TILE + lane;
  const double c = cf[0], c1 = cf[a.npad], c2 = cf[2 * a.npad], c3 = cf[3 * a.npad];
  for (int q = wave; q < b.nsh; q += 4) {
    const int sh = a.shl[b.sh0 + q];
    double* out = a.Y + (size_t)blockIdx.y * a.ngrp + b.off + (size_t)a.col[b.sh0 + q] * b.ld + tl.y * TILE + lane;
    ao_shell<GGA>(a.ao, sh, r, [&](int o, double v, double vx, double vy, double vz) {
      out[(size_t)o * b.ld] = GGA ? c * v + c1 * vx + c2 * vy + c3 * vz : c * v;
    });
  }
}

// One 64 x 64 tile of V_b = phi^T Y over PART points, 32 x 32 per wavefront on the
// FP64 matrix units, 16 points at a time through LDS (two buffers, the loads of the
// next PF steps in flight).  A lane takes 4 consecutive points of its rows; which
// point is the k-th of a matrix instruction does not matter as long as both sides
// agree.  Bound by the loads' latency next to the matrix units: 4.28 ms for 9.4e10
// columns^2 points (44 TFLOP/s); one step ahead 4.7, straight from memory without
// LDS 6.9, tiles of 128 x 128 on eight wavefronts 4.8, columns cut evenly 5.0.
constexpr int PART = 2048;
__global__ __launch_bounds__(256) void k_vmat(XArgs a) {
  constexpr int RS = 18, PF = 2;  // row length in LDS: 16 rows fall on distinct banks
  __shared__ __align__(16) double s_t[2][2][64 * RS];
  const int4 e = a.vt[blockIdx.x];
  if (e.x < 0) return;
  const DBatch b = a.batch[e.x];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), row = lane & 15, g = lane >> 4;
  const int nb = b.nb, ld = b.ld, mw = 32 * (wave & 1), nw = 32 * (wave >> 1);
  const int m0 = 64 * e.z + mw, n0 = 64 * e.w + nw;
  // staging: thread = (row, 4 points)
  const int sr = threadIdx.x >> 2, sp = (threadIdx.x & 3) * 4;
  const double* A = a.phi + b.off + (size_t)min(64 * e.z + sr, nb - 1) * ld + sp;
  const double* B = a.Y + (size_t)blockIdx.y * a.ngrp + b.off + (size_t)min(64 * e.w + sr, nb - 1) * ld + sp;
  v4d acc[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[t][j] = v4d{0.0, 0.0, 0.0, 0.0};
  const int p0 = e.y * PART, p1 = min(p0 + PART, ld);
  v2d ra[PF][2], rb[PF][2];
  auto fetch = [&](int f, int p) {
    p = min(p, p1 - 16);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ra[f][h] = *(const v2d*)(A + p + 2 * h);
      rb[f][h] = *(const v2d*)(B + p + 2 * h);
    }
  };
#pragma unroll
  for (int f = 0; f < PF; ++f) fetch(f, p0 + 16 * f);
  int cur = 0;
  for (int pp = p0; pp < p1; pp += 16 * PF)  // whole tiles of points: a multiple of 64
#pragma unroll
    for (int f = 0; f < PF; ++f, cur ^= 1) {
      double *sa = s_t[cur][0], *sb = s_t[cur][1];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        *(v2d*)(sa + sr * RS + sp + 2 * h) = ra[f][h];
        *(v2d*)(sb + sr * RS + sp + 2 * h) = rb[f][h];
      }
      __syncthreads();
      fetch(f, pp + 16 * (f + PF));
      v2d x[2][2], y[2][2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          x[t][h] = *(const v2d*)(sa + (mw + 16 * t + row) * RS + 4 * g + 2 * h);
          y[t][h] = *(const v2d*)(sb + (nw + 16 * t + row) * RS + 4 * g + 2 * h);
        }
      // 16 x 16 sub-tiles past the batch's columns are left out (wavefront-uniform)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (m0 + 16 * t < nb && n0 + 16 * j < nb)
#pragma unroll
            for (int k = 0; k < 4; ++k)
              acc[t][j] =
                  __builtin_amdgcn_mfma_f64_16x16x4f64(x[t][k / 2][k % 2], y[j][k / 2][k % 2], acc[t][j], 0, 0, 0);
    }
  double* V = a.Vb + (size_t)blockIdx.y * a.nvb + b.vb + (size_t)e.y * nb * nb;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + 16 * t + 4 * i + g, n = n0 + 16 * j + row;
        if (m < nb && n < nb) V[(size_t)m * nb + n] = acc[t][j][i];
      }
}

// V(i, .) += the rows of the group's V_b that belong to AO i: block = (i, VCOLS
// columns), a wavefront per batch that holds i, the row collected in LDS
constexpr int VCOLS = 4096;
__global__ __launch_bounds__(512) void k_vsum(XArgs a, const long long* __restrict__ ptr, const int2* __restrict__ ent,
                                              int nbf, double* V) {
  extern __shared__ double s_row[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = blockIdx.x, c0 = blockIdx.y * VCOLS, nc = min(VCOLS, nbf - c0);
  for (int j = threadIdx.x; j < nc; j += 512) s_row[j] = 0.0;
  __syncthreads();
  for (long long k = ptr[i] + wave; k < ptr[i + 1]; k += 8) {
    const int2 e = ent[k];  // batch, column of i
    const DBatch& b = a.batch[e.x];
    const int nb = b.nb;
    const double* x = a.Vb + (size_t)blockIdx.z * a.nvb + b.vb + (size_t)e.y * nb;
    for (int n = lane; n < nb; n += 64) {
      double v = 0.0;
      for (int s = 0; s < b.nparts; ++s) v += x[(size_t)s * nb * nb + n];
      const int c = a.idx[b.ao0 + n] - c0;
      if (c >= 0 && c < nc) unsafeAtomicAdd(&s_row[c], v);
    }
  }
  __syncthreads();
  double* row = V + ((size_t)blockIdx.z * nbf + i) * nbf + c0;
  for (int j = threadIdx.x; j < nc; j += 512) row[j] += s_row[j];
}

// ------------------------------------------------------------ packing
__global__ void k_unpack(const double* pk, int nbf, double* full) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nbf * nbf) return;
  const int i = (int)(t / nbf), j = (int)(t % nbf);
  const int hi = i > j ? i : j, lo = i > j ? j : i;
  full[t] = pk[(size_t)hi * (hi + 1) / 2 + lo];
}

// packed lower triangle of V + V^T
__global__ void k_pack(const double* V, int nbf, double* pk) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long ntri = (long long)nbf * (nbf + 1) / 2;
  if (t >= ntri) return;
  int i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) / 2.0);
  while ((long long)i * (i + 1) / 2 > t) --i;
  while ((long long)(i + 1) * (i + 2) / 2 <= t) ++i;
  const int j = (int)(t - (long long)i * (i + 1) / 2);
  pk[t] = V[(size_t)i * nbf + j] + V[(size_t)j * nbf + i];
}

inline unsigned nblk(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// ------------------------------------------------------------ device buffers
template <typename T>
struct Buf {
  T* p = nullptr;
  size_t n = 0;
  bool ensure(size_t m) {
    if (m <= n && p) return true;
    if (p) hipFree(p);
    p = nullptr;
    n = 0;
    if (hipMalloc((void**)&p, std::max<size_t>(m, 1) * sizeof(T)) != hipSuccess) {
      p = nullptr;
      err("XC: hipMalloc of %zu bytes failed", m * sizeof(T));
      return false;
    }
    n = std::max<size_t>(m, 1);
    return true;
  }
  void release() {
    if (p) hipFree(p);
    p = nullptr;
    n = 0;
  }
};

struct Batch {
  long long p0;
  int npts, sh0, nsh, ao0, nb;
};

// batches [b0, b1) built together
struct Group {
  int b0, b1;
  long long tile0, ntile, vt0, nvt, ngrp, nvb;
};

struct XCState {
  XCFunc f{};
  bool configured = false;
  int nrad = 96, ntheta = 15;
  // cache key of the grid
  std::vector<double> key_xyz, key_ex, key_cc;
  std::vector<int> key_am;
  int key_nbf = -1, key_nrad = 0, key_ntheta = 0;
  bool grid_ready = false;
  std::vector<double> grid;  // kept points (x, y, z, w), atom-major
  std::vector<Batch> batches;
  std::vector<Group> groups;
  int max_nb = 0;
  std::vector<int> idx;                             // AO of every column (d_idx)
  long long limit = 0;                              // elements of a group (build_groups)
  long long max_grp = 0, max_vb = 0, max_tile = 0;  // largest group: phi, V_b, point tiles
  Buf<double> d_pts, d_xf, d_D, d_pk, d_acc, d_phi, d_Y, d_rho, d_coef, d_Vb, d_V;
  Buf<DBatch> d_batch;
  Buf<int2> d_tile;
  Buf<int4> d_vt;
  Buf<long long> d_vptr;
  Buf<int2> d_vent;
  Buf<int> d_shl, d_col, d_idx, d_am, d_harm, d_atom, d_nprim, d_poff;
  Buf<double> d_ex, d_cc, d_xyz;
  void release() {
    for (auto* b : {&d_pts, &d_xf, &d_D, &d_pk, &d_acc, &d_phi, &d_Y, &d_rho, &d_coef, &d_Vb, &d_V, &d_ex, &d_cc, &d_xyz})
      b->release();
    d_batch.release();
    d_tile.release();
    d_vt.release();
    d_vptr.release();
    d_vent.release();
    for (auto* b : {&d_shl, &d_col, &d_idx, &d_am, &d_harm, &d_atom, &d_nprim, &d_poff}) b->release();
    grid_ready = false;
  }
};

std::mutex g_xmtx;
std::map<oqph_session*, XCState*> g_xc;

XCState* state(oqph_session* s, bool create) {
  std::lock_guard<std::mutex> lk(g_xmtx);
  auto it = g_xc.find(s);
  if (it != g_xc.end()) return it->second;
  if (!create) return nullptr;
  XCState* x = new XCState();
  g_xc[s] = x;
  return x;
}

// Treutler-Ahlrichs xi (J. Chem. Phys. 102, 346 (1995)); 1.0 beyond Kr
double ta_xi(int z) {
  static const double t[37] = {1.0, 0.8, 0.9, 1.8, 1.4, 1.3, 1.1, 0.9, 0.9, 0.9, 0.9, 1.4, 1.3,
                               1.3, 1.2, 1.1, 1.0, 1.0, 1.0, 1.5, 1.4, 1.3, 1.2, 1.2, 1.2, 1.2,
                               1.2, 1.2, 1.1, 1.1, 1.1, 1.1, 1.0, 0.9, 0.9, 0.9, 0.9};
  return (z >= 1 && z <= 36) ? t[z] : 1.0;
}

// Gauss-Legendre nodes and weights on [-1, 1] (Newton on P_n)
void gauss_legendre(int n, std::vector<double>& x, std::vector<double>& w) {
  x.assign(n, 0.0);
  w.assign(n, 0.0);
  for (int i = 0; i < n; ++i) {
    double z = cos(PI * (i + 0.75) / (n + 0.5)), dp = 0.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = z;
      for (int k = 2; k <= n; ++k) {
        const double p2 = ((2 * k - 1) * z * p1 - (k - 1) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      if (n == 1) p0 = 1.0;
      dp = n * (z * p1 - p0) / (z * z - 1.0);
      const double dz = p1 / dp;
      z -= dz;
      if (fabs(dz) < 1e-16) break;
    }
    double p0 = 1.0, p1 = z;
    for (int k = 2; k <= n; ++k) {
      const double p2 = ((2 * k - 1) * z * p1 - (k - 1) * p0) / k;
      p0 = p1;
      p1 = p2;
    }
    dp = n * (z * p1 - p0) / (z * z - 1.0);
    x[n - 1 - i] = z;
    w[n - 1 - i] = 2.0 / ((1.0 - z * z) * dp * dp);
  }
}

template <typename T>
bool upload(Buf<T>& b, const T* h, size_t n, hipStream_t st) {
  if (!b.ensure(n)) return false;
  if (n && hipMemcpyAsync(b.p, h, n * sizeof(T), hipMemcpyHostToDevice, st) != hipSuccess) {
    err("XC: host-to-device copy failed");
    return false;
  }
  return true;
}

// Cuts the batches into groups of at most `limit` basis-function values and V_b
// elements, with their point tiles and V_b tiles, and uploads them.
int build_groups(XCState* x, const oqph::SessionView& v, long long limit) {
  std::vector<DBatch> db;
  std::vector<int2> tile;
  std::vector<int4> vt;
  std::vector<long long> vptr;  // per group: nbf + 1 starts in vent
  std::vector<int2> vent;       // per AO: the batches that hold it and its column there
  x->groups.clear();
  long long max_grp = 0, max_vb = 0, max_tile = 0;
  for (int b0 = 0; b0 < (int)x->batches.size();) {
    Group g{b0, b0, (long long)tile.size(), 0, (long long)vt.size(), 0, 0, 0};
    std::vector<int4> list[8];  // tiles of a part stay on one XCD: blocks are dealt to the eight in turn
    while (g.b1 < (int)x->batches.size()) {
      const Batch& b = x->batches[g.b1];
      const int ld = (b.npts + TILE - 1) / TILE * TILE, nparts = (ld + PART - 1) / PART, nt = (b.nb + 63) / 64;
      const long long phi = (long long)ld * b.nb, vb = (long long)nparts * b.nb * b.nb;
      if (g.b1 > b0 && (g.ngrp + phi > limit || g.nvb + vb > limit)) break;
      db.push_back({b.p0, g.ngrp, g.nvb, b.npts, ld, b.sh0, b.nsh, b.ao0, b.nb, nparts, 0});
      for (int t = 0; t < ld / TILE; ++t) tile.push_back(int2{g.b1, t});
      for (int k = 0; k < nparts; ++k) {
        auto& l = *std::min_element(list, list + 8, [](const auto& p, const auto& q) { return p.size() < q.size(); });
        for (int m = 0; m < nt; ++m)
          for (int c = 0; c < nt; ++c) l.push_back(int4{g.b1, k, m, c});
      }
      g.ngrp += phi;
      g.nvb += vb;
      ++g.b1;
    }
    size_t len = 0;
    for (auto& l : list) len = std::max(len, l.size());
    for (size_t i = 0; i < len; ++i)
      for (auto& l : list) vt.push_back(i < l.size() ? l[i] : int4{-1, 0, 0, 0});
    const size_t p0 = vptr.size(), e0 = vent.size();
    vptr.resize(p0 + v.nbf + 1, 0);
    for (int k = b0; k < g.b1; ++k)
      for (int i = 0; i < x->batches[k].nb; ++i) ++vptr[p0 + 1 + x->idx[x->batches[k].ao0 + i]];
    vptr[p0] = (long long)e0;
    for (int i = 0; i < v.nbf; ++i) vptr[p0 + 1 + i] += vptr[p0 + i];
    vent.resize((size_t)vptr[p0 + v.nbf]);
    std::vector<long long> at(vptr.begin() + p0, vptr.end() - 1);
    for (int k = b0; k < g.b1; ++k)
      for (int i = 0; i < x->batches[k].nb; ++i) vent[at[x->idx[x->batches[k].ao0 + i]]++] = int2{k, i};
    g.ntile = (long long)tile.size() - g.tile0;
    g.nvt = (long long)vt.size() - g.vt0;
    max_grp = std::max(max_grp, g.ngrp);
    max_vb = std::max(max_vb, g.nvb);
    max_tile = std::max(max_tile, g.ntile);
    x->groups.push_back(g);
    b0 = g.b1;
  }
  x->limit = limit;
  x->max_grp = max_grp;
  x->max_vb = max_vb;
  x->max_tile = max_tile;
  hipStream_t st = v.stream;
  const bool ok = upload(x->d_batch, db.data(), db.size(), st) && upload(x->d_tile, tile.data(), tile.size(), st) &&
                  upload(x->d_vt, vt.data(), vt.size(), st) && upload(x->d_vptr, vptr.data(), vptr.size(), st) &&
                  upload(x->d_vent, vent.data(), vent.size(), st);
  return hipStreamSynchronize(st) == hipSuccess && ok ? 0 : 3;
}

// Device memory of a build: D, V and the packed matrices, and for the largest group phi,
// Y and V_b (up to 2 GB, and 4 GB each for two spins), rho and its coefficients.  Where
// the device has not that much left the groups get smaller, down to one batch each.
int workspace(XCState* x, const oqph::SessionView& v, size_t ns) {
  const size_t nbf = (size_t)v.nbf, ntri = nbf * (nbf + 1) / 2, nn = nbf * nbf;
  if (!x->d_pk.ensure(ntri * ns) || !x->d_D.ensure(nn * ns) || !x->d_V.ensure(nn * ns) || !x->d_acc.ensure(2)) return 3;
  const char* e = getenv("OQPH_XC_WORKSPACE");  // bytes of the group arrays counted as available (tests)
  const double most = e ? atof(e) : 1e300;
  for (;;) {
    const size_t npad = (size_t)x->max_tile * TILE;
    const double bytes = 8.0 * ((1.0 + ns) * x->max_grp + (double)ns * x->max_vb + 8.0 * ns * npad);
    if (bytes <= most && x->d_phi.ensure((size_t)x->max_grp) && x->d_Y.ensure(ns * x->max_grp) &&
        x->d_Vb.ensure(ns * x->max_vb) && x->d_rho.ensure(4 * ns * npad) && x->d_coef.ensure(4 * ns * npad))
      return 0;
    (void)hipGetLastError();  // out of memory
    if (x->groups.size() == x->batches.size()) {
      err("XC: no device memory for a group of one batch (%.0f bytes)", bytes);
      return 3;
    }
    for (auto* b : {&x->d_phi, &x->d_Y, &x->d_Vb, &x->d_rho, &x->d_coef}) b->release();
    const long long limit = std::max<long long>(std::min(x->limit, std::max(x->max_grp, x->max_vb)) / 4, 1);
    if (const int rc = build_groups(x, v, limit)) {
      x->grid_ready = false;
      return rc;
    }
  }
}

int build_grid(XCState* x, const oqph::SessionView& v) {
  const int natm = v.natm, nrad = x->nrad, nth = x->ntheta, nphi = 2 * nth, nang = nth * nphi;
  hipStream_t st = v.stream;
  // radial and angular tables
  std::vector<double> rad((size_t)natm * nrad * 2), ang((size_t)nang * 4);
  for (int A = 0; A < natm; ++A) {
    const double xi = ta_xi((int)lround(v.zn[A])), al = 0.6, c = xi / log(2.0);
    for (int i = 1; i <= nrad; ++i) {
      const double th = i * PI / (nrad + 1), xx = cos(th), lg = log(2.0 / (1.0 - xx));
      const double r = c * pow(1.0 + xx, al) * lg;
      const double drdx = c * (al * pow(1.0 + xx, al - 1.0) * lg + pow(1.0 + xx, al) / (1.0 - xx));
      rad[((size_t)A * nrad + i - 1) * 2] = r;
      rad[((size_t)A * nrad + i - 1) * 2 + 1] = PI / (nrad + 1) * sin(th) * drdx * r * r;
    }
  }
  std::vector<double> gt, gw;
  gauss_legendre(nth, gt, gw);
  for (int a = 0; a < nth; ++a)
    for (int b = 0; b < nphi; ++b) {
      const double ph = (b + 0.5) * (2.0 * PI / nphi), s = sqrt(1.0 - gt[a] * gt[a]);
      double* o = &ang[(size_t)(a * nphi + b) * 4];
      o[0] = s * cos(ph);
      o[1] = s * sin(ph);
      o[2] = gt[a];
      o[3] = gw[a] * (2.0 * PI / nphi);
    }
  std::vector<double> rinv((size_t)natm * natm, 0.0);
  for (int a = 0; a < natm; ++a)
    for (int b = 0; b < natm; ++b)
      if (a != b) {
        const double dx = v.xyz[3 * a] - v.xyz[3 * b], dy = v.xyz[3 * a + 1] - v.xyz[3 * b + 1],
                     dz = v.xyz[3 * a + 2] - v.xyz[3 * b + 2];
        rinv[(size_t)a * natm + b] = 1.0 / sqrt(dx * dx + dy * dy + dz * dz);
      }
  const long long nraw = (long long)natm * nrad * nang;
  Buf<double> d_rad, d_ang, d_rinv, d_raw;
  bool ok = upload(x->d_xyz, v.xyz, (size_t)3 * natm, st) && upload(d_rad, rad.data(), rad.size(), st) &&
            upload(d_ang, ang.data(), ang.size(), st) && upload(d_rinv, rinv.data(), rinv.size(), st) &&
            d_raw.ensure((size_t)nraw * 4);
  std::vector<double> raw;
  if (ok) {
    GridArgs g{x->d_xyz.p, d_rinv.p, d_rad.p, d_ang.p, natm, nrad, nang, nraw, d_raw.p};
    hipLaunchKernelGGL(k_grid, dim3(nblk(nraw, 256)), dim3(256), 0, st, g);
    raw.resize((size_t)nraw * 4);
    ok = hipMemcpyAsync(raw.data(), d_raw.p, raw.size() * sizeof(double), hipMemcpyDeviceToHost, st) == hipSuccess &&
         hipStreamSynchronize(st) == hipSuccess;
    if (!ok) err("XC: grid kernel failed: %s", hipGetErrorString(hipGetLastError()));
  }
  d_rad.release();
  d_ang.release();
  d_rinv.release();
  d_raw.release();
  if (!ok) return 2;
  // keep w > 1e-20 (atom-major order: the exported grid)
  x->grid.clear();
  for (long long t = 0; t < nraw; ++t)
    if (raw[4 * t + 3] > 1e-20) x->grid.insert(x->grid.end(), &raw[4 * t], &raw[4 * t] + 4);
  const long long n = (long long)x->grid.size() / 4;
  // boxes
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (long long t = 0; t < n; ++t)
    for (int k = 0; k < 3; ++k) {
      lo[k] = std::min(lo[k], x->grid[4 * t + k]);
      hi[k] = std::max(hi[k], x->grid[4 * t + k]);
    }
  long long nbx[3];
  for (int k = 0; k < 3; ++k) nbx[k] = std::max<long long>(1, (long long)((hi[k] - lo[k]) / BOX) + 1);
  std::vector<long long> key(n), order(n);
  auto box = [&](long long t, int k) { return std::min(nbx[k] - 1, (long long)((x->grid[4 * t + k] - lo[k]) / BOX)); };
  // Sorted by box, atom-major within a box: by counting while the boxes are not many more
  // than the points; a sparse system (far fragments) has empty boxes by the billion, and
  // its points are sorted by their box instead.
  const double most = 8.0 * (double)n + (1 << 20);
  if ((double)nbx[0] * nbx[1] * nbx[2] <= most) {
    const long long nkeys = nbx[0] * nbx[1] * nbx[2];
    std::vector<long long> start(nkeys + 1, 0);
    for (long long t = 0; t < n; ++t) {
      key[t] = (box(t, 0) * nbx[1] + box(t, 1)) * nbx[2] + box(t, 2);
      ++start[key[t] + 1];
    }
    for (long long k = 0; k < nkeys; ++k) start[k + 1] += start[k];
    for (long long t = 0; t < n; ++t) order[start[key[t]]++] = t;
  } else {
    std::vector<std::array<long long, 3>> at(n);
    for (long long t = 0; t < n; ++t) {
      at[t] = {box(t, 0), box(t, 1), box(t, 2)};
      order[t] = t;
    }
    std::stable_sort(order.begin(), order.end(), [&](long long i, long long j) { return at[i] < at[j]; });
    for (long long i = 0, k = 0; i < n; ++i) {
      if (i > 0 && at[order[i]] != at[order[i - 1]]) ++k;
      key[order[i]] = k;
    }
  }
  std::vector<double> sorted((size_t)n * 4);
  for (long long t = 0; t < n; ++t) memcpy(&sorted[4 * t], &x->grid[4 * order[t]], 4 * sizeof(double));
  // batches and their shells
  std::vector<double> rcut(v.nsh);
  for (int s = 0; s < v.nsh; ++s) {
    double rc = 0.0;
    for (int k = 0; k < v.nprim[s]; ++k) {
      const double c = fabs(v.cc[v.poff[s] + k]), al = v.ex[v.poff[s] + k];
      if (c > AO_EPS) rc = std::max(rc, sqrt(log(c / AO_EPS) / al));
    }
    rcut[s] = rc;
  }
  std::vector<int> shl, col, idx;
  x->batches.clear();
  x->max_nb = 0;
  for (long long t0 = 0; t0 < n;) {
    long long t1 = t0;
    while (t1 < n && key[order[t1]] == key[order[t0]] && t1 - t0 < MAX_BATCH) ++t1;
    // the batch's bounding box; a shell is kept when its centre lies within
    // its cutoff radius of the box
    double blo[3] = {1e300, 1e300, 1e300}, bhi[3] = {-1e300, -1e300, -1e300};
    for (long long t = t0; t < t1; ++t)
      for (int k = 0; k < 3; ++k) {
        blo[k] = std::min(blo[k], sorted[4 * t + k]);
        bhi[k] = std::max(bhi[k], sorted[4 * t + k]);
      }
    Batch b{t0, (int)(t1 - t0), (int)shl.size(), 0, (int)idx.size(), 0};
    for (int s = 0; s < v.nsh; ++s) {
      const int A = v.atom[s];
      double d2 = 0.0;
      for (int k = 0; k < 3; ++k) {
        const double a = v.xyz[3 * A + k], o = a < blo[k] ? blo[k] - a : (a > bhi[k] ? a - bhi[k] : 0.0);
        d2 += o * o;
      }
      if (sqrt(d2) > rcut[s]) continue;
      const int l = v.am[s], no = (v.harm[s] && l >= 2) ? 2 * l + 1 : (l + 1) * (l + 2) / 2;
      shl.push_back(s);
      col.push_back(b.nb);
      for (int o = 0; o < no; ++o) idx.push_back(v.aooff[s] + o);
      b.nb += no;
      ++b.nsh;
    }
    if (b.nsh > 0) {
      x->batches.push_back(b);
      x->max_nb = std::max(x->max_nb, b.nb);
    }
    t0 = t1;
  }
  // device copies
  std::vector<double> xf(400);
  oqph_host::build_xform(reinterpret_cast<double(*)[2][10][10]>(xf.data()));
  std::vector<int> harm(v.harm, v.harm + v.nsh);
  int nprim_tot = 0;
  for (int s = 0; s < v.nsh; ++s) nprim_tot = std::max(nprim_tot, v.poff[s] + v.nprim[s]);
  ok = upload(x->d_pts, sorted.data(), sorted.size(), st) && upload(x->d_xf, xf.data(), xf.size(), st) &&
       upload(x->d_shl, shl.data(), shl.size(), st) && upload(x->d_col, col.data(), col.size(), st) &&
       upload(x->d_idx, idx.data(), idx.size(), st) && upload(x->d_am, v.am, (size_t)v.nsh, st) &&
       upload(x->d_harm, harm.data(), harm.size(), st) && upload(x->d_atom, v.atom, (size_t)v.nsh, st) &&
       upload(x->d_nprim, v.nprim, (size_t)v.nsh, st) && upload(x->d_poff, v.poff, (size_t)v.nsh, st) &&
       upload(x->d_ex, v.ex, (size_t)nprim_tot, st) && upload(x->d_cc, v.cc, (size_t)nprim_tot, st);
  ok = hipStreamSynchronize(st) == hipSuccess && ok;
  if (!ok) return 3;
  x->idx.swap(idx);
  if (const int rc = build_groups(x, v, GROUP_ELEMS)) return rc;
  x->grid_ready = true;
  return 0;
}

bool grid_current(XCState* x, const oqph::SessionView& v) {
  if (!x->grid_ready || x->key_nbf != v.nbf || x->key_nrad != x->nrad || x->key_ntheta != x->ntheta) return false;
  if (x->key_xyz.size() != (size_t)3 * v.natm || !std::equal(x->key_xyz.begin(), x->key_xyz.end(), v.xyz))
    return false;
  int np = 0;
  for (int s = 0; s < v.nsh; ++s) np = std::max(np, v.poff[s] + v.nprim[s]);
  return x->key_ex.size() == (size_t)np && std::equal(x->key_ex.begin(), x->key_ex.end(), v.ex) &&
         std::equal(x->key_cc.begin(), x->key_cc.end(), v.cc) && x->key_am.size() == (size_t)v.nsh &&
         std::equal(x->key_am.begin(), x->key_am.end(), v.am);
}

int ensure_grid(XCState* x, const oqph::SessionView& v) {
  if (grid_current(x, v)) return 0;
  x->grid_ready = false;
  const int rc = build_grid(x, v);
  if (rc) return rc;
  x->key_nbf = v.nbf;
  x->key_nrad = x->nrad;
  x->key_ntheta = x->ntheta;
  x->key_xyz.assign(v.xyz, v.xyz + 3 * v.natm);
  int np = 0;
  for (int s = 0; s < v.nsh; ++s) np = std::max(np, v.poff[s] + v.nprim[s]);
  x->key_ex.assign(v.ex, v.ex + np);
  x->key_cc.assign(v.cc, v.cc + np);
  x->key_am.assign(v.am, v.am + v.nsh);
  return 0;
}

int vxc_run(oqph_session* s, const double* d, int nfocks, double* fxc, double* exc, double* nel) {
  oqph::SessionView v;
  if (!oqph::session_view(s, &v)) {
    err("oqph_vxc: the session has no basis or geometry");
    return 4;
  }
  XCState* x = state(s, false);
  if (!x || !x->configured) {
    err("oqph_vxc: no functional set (oqph_session_set_xc)");
    return 1;
  }
  if (nfocks != 1 && nfocks != 2) {
    err("oqph_vxc: nfocks %d (1 or 2)", nfocks);
    return 1;
  }
  if (!d || !fxc || !exc || !nel) {
    err("oqph_vxc: null argument");
    return 4;
  }
  hipSetDevice(v.device);
  hipStream_t st = v.stream;
  int rc = ensure_grid(x, v);
  if (rc) return rc;
  const int nbf = v.nbf;
  const size_t ntri = (size_t)nbf * (nbf + 1) / 2, nn = (size_t)nbf * nbf;
  const size_t ns = (size_t)nfocks;
  if ((rc = workspace(x, v, ns))) return rc;
  if (!upload(x->d_pk, d, ntri * ns, st)) {
    hipStreamSynchronize(st);  // the upload reads the caller's array
    return 3;
  }
  const size_t lds = (size_t)4 * 16 * (TILE + 1) * sizeof(double) + (size_t)x->max_nb * sizeof(int);
  for (int sp = 0; sp < nfocks; ++sp)
    hipLaunchKernelGGL(k_unpack, dim3(nblk((long long)nn, 256)), dim3(256), 0, st, x->d_pk.p + sp * ntri, nbf,
                       x->d_D.p + sp * nn);
  hipMemsetAsync(x->d_acc.p, 0, 2 * sizeof(double), st);
  hipMemsetAsync(x->d_V.p, 0, nn * ns * sizeof(double), st);
  XArgs a{};
  a.ao = {x->d_am.p, x->d_harm.p, x->d_atom.p, x->d_nprim.p, x->d_poff.p, x->d_ex.p, x->d_cc.p, x->d_xyz.p, x->d_xf.p};
  a.pts = x->d_pts.p;
  a.batch = x->d_batch.p;
  a.shl = x->d_shl.p;
  a.col = x->d_col.p;
  a.idx = x->d_idx.p;
  a.phi = x->d_phi.p;
  a.Y = x->d_Y.p;
  a.rho = x->d_rho.p;
  a.coef = x->d_coef.p;
  a.Vb = x->d_Vb.p;
  auto kr = x->f.gga ? k_rho<true> : k_rho<false>;
  auto ky = x->f.gga ? k_y<true> : k_y<false>;
  if (lds > 64 * 1024) hipFuncSetAttribute((const void*)kr, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  for (size_t gi = 0; gi < x->groups.size(); ++gi) {
    const Group& g = x->groups[gi];
    a.tile = x->d_tile.p + g.tile0;
    a.vt = x->d_vt.p + g.vt0;
    a.npad = g.ntile * TILE;
    a.ngrp = g.ngrp;
    a.nvb = g.nvb;
    const unsigned nt = (unsigned)g.ntile, sp = (unsigned)nfocks;
    hipLaunchKernelGGL(k_ao, dim3(nt), dim3(256), 0, st, a);
    hipLaunchKernelGGL(kr, dim3(nt, sp), dim3(256), lds, st, a, x->d_D.p, nbf);
    hipLaunchKernelGGL(k_xc_point, dim3(std::min(nblk(g.ntile, 4), 2048u)), dim3(256), 0, st, a, g.ntile, nfocks, x->f,
                       x->d_acc.p);
    hipLaunchKernelGGL(ky, dim3(nt, sp), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_vmat, dim3((unsigned)g.nvt, sp), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_vsum, dim3((unsigned)nbf, nblk(nbf, VCOLS), sp), dim3(512),
                       std::min(nbf, VCOLS) * sizeof(double), st, a, x->d_vptr.p + gi * (nbf + 1), x->d_vent.p, nbf,
                       x->d_V.p);
  }
  for (int sp = 0; sp < nfocks; ++sp)
    hipLaunchKernelGGL(k_pack, dim3(nblk((long long)ntri, 256)), dim3(256), 0, st, x->d_V.p + sp * nn, nbf,
                       x->d_pk.p + sp * ntri);
  hipError_t le = hipGetLastError();
  if (le != hipSuccess) {
    err("oqph_vxc: launch failed: %s", hipGetErrorString(le));
    hipStreamSynchronize(st);
    return 2;
  }
  double acc[2];
  if (hipMemcpyAsync(fxc, x->d_pk.p, ntri * nfocks * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(acc, x->d_acc.p, 2 * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess) {
    err("oqph_vxc: device error: %s", hipGetErrorString(hipGetLastError()));
    return 2;
  }
  *exc = acc[0];
  *nel = acc[1];
  return 0;
}

}  // namespace

void oqph::xc_release(oqph_session* s) {
  XCState* x = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_xmtx);
    auto it = g_xc.find(s);
    if (it == g_xc.end()) return;
    x = it->second;
    g_xc.erase(it);
  }
  x->release();
  delete x;
}

extern "C" int oqph_xc_functional_info(const char* name, double* hfex, int* gga) {
  XCFunc f;
  if (!lookup(name, &f)) return 1;
  if (hfex) *hfex = f.hfex;
  if (gga) *gga = f.gga;
  return 0;
}

extern "C" int oqph_session_set_xc(oqph_session* s, const char* name, int nrad, int ntheta) {
  if (!s) return 4;
  XCFunc f;
  if (!lookup(name, &f)) {
    err("oqph_session_set_xc: unknown functional '%s'", name ? name : "");
    return 1;
  }
  if (nrad < 2 || nrad > 1000 || ntheta < 2 || ntheta > 200) {
    err("oqph_session_set_xc: grid %d x %d out of range", nrad, ntheta);
    return 4;
  }
  XCState* x = state(s, true);
  x->f = f;
  x->configured = true;
  x->nrad = nrad;
  x->ntheta = ntheta;
  return 0;
}

extern "C" int oqph_vxc(oqph_session* s, const double* d, int nfocks, double* fxc, double* exc, double* nel) {
  if (!s) return 4;
  return vxc_run(s, d, nfocks, fxc, exc, nel);
}

extern "C" long long oqph_xc_grid(oqph_session* s, double* pts, long long cap) {
  oqph::SessionView v;
  if (!s || !oqph::session_view(s, &v)) return -4;
  XCState* x = state(s, false);
  if (!x || !x->configured) return -1;
  hipSetDevice(v.device);
  if (ensure_grid(x, v)) return -2;
  const long long n = (long long)x->grid.size() / 4;
  if (pts) memcpy(pts, x->grid.data(), (size_t)std::min(n, cap) * 4 * sizeof(double));
  return n;
}

extern "C" int oqph_xc_grid_stats(oqph_session* s, long long* out) {
  oqph::SessionView v;
  if (!s || !out || !oqph::session_view(s, &v)) return 4;
  XCState* x = state(s, false);
  if (!x || !x->configured) return 1;
  hipSetDevice(v.device);
  if (ensure_grid(x, v)) return 2;
  long long a = 0, b2 = 0;
  for (const Batch& b : x->batches) {
    a += (long long)b.npts * b.nb;
    b2 += (long long)b.npts * b.nb * b.nb;
  }
  out[0] = (long long)x->grid.size() / 4;
  out[1] = (long long)x->batches.size();
  out[2] = a;
  out[3] = b2;
  out[4] = x->max_nb;
  return 0;
}

extern "C" void routec_vxc(const double* d, double* fxc, const int* nbf, const int* nfocks, double* eexc,
                           double* totele, int* info) {
  int rc = 1;
  oqph_session* s = oqph::default_session();
  oqph::SessionView v;
  if (!info) return;
  if (!s || !nbf || !nfocks || !oqph::session_view(s, &v)) {
    err("routec_vxc: no default session");
  } else if (*nbf != v.nbf) {
    err("routec_vxc: nbf %d does not match the session basis (%d)", *nbf, v.nbf);
  } else {
    rc = vxc_run(s, d, *nfocks, fxc, eexc, totele);
    if (rc != 0) rc = 1;
  }
  *info = rc;
}
