// eri_device.h -- device-side building blocks of the J/K and gradient kernels.
//
// Electron-repulsion integrals are evaluated by Rys quadrature (Dupuis, Rys,
// King, J. Chem. Phys. 65, 111 (1976)): per primitive quartet and root, the
// 2D integrals G_d(i,k), i <= La+Lb, k <= Lc+Ld, come from the vertical
// recursion on centres A and C; the Cartesian (e0|f0) products are contracted
// over primitives and roots in registers; the horizontal transfer to (ab|cd)
// runs once per contracted quartet in its closed binomial form
//   (a b| = sum_j prod_d C(b_d, j_d) AB_d^(b_d - j_d) (a + j, 0| .
// Everything that depends on the angular momenta is a compile-time constant,
// so the loops unroll into straight-line register code for each class.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include <utility>
#include "oqph_common.h"

namespace oqph {

// ---------------------------------------------------------------- Cartesian
__host__ __device__ constexpr int ncart(int L) { return L < 0 ? 0 : (L + 1) * (L + 2) / 2; }
__host__ __device__ constexpr int ncum(int L) { return L < 0 ? 0 : (L + 1) * (L + 2) * (L + 3) / 6; }
// canonical order inside level L: lx descending, then ly descending
__host__ __device__ constexpr int c_k(int c) {  // k = L - lx
  int k = 0;
  while ((k + 1) * (k + 2) / 2 <= c) ++k;
  return k;
}
__host__ __device__ constexpr int c_lx(int L, int c) { return L - c_k(c); }
__host__ __device__ constexpr int c_lz(int L, int c) { return c - c_k(c) * (c_k(c) + 1) / 2; }
__host__ __device__ constexpr int c_ly(int L, int c) { return c_k(c) - c_lz(L, c); }
__host__ __device__ constexpr int c_idx(int lx, int ly, int lz) {  // local index in level lx+ly+lz
  return (ly + lz) * (ly + lz + 1) / 2 + lz;
}
// component of level L along axis d
__host__ __device__ constexpr int c_l(int L, int c, int d) {
  return d == 0 ? c_lx(L, c) : (d == 1 ? c_ly(L, c) : c_lz(L, c));
}
__host__ __device__ constexpr int binom(int n, int k) {
  int r = 1;
  for (int i = 1; i <= k; ++i) r = r * (n - i + 1) / i;
  return r;
}

// ------------------------------------------------------ compile-time loops
// sfor<N>(f) calls f(std::integral_constant<int, i>{}) for i = 0..N-1, so the
// body sees every index as a constant expression: Cartesian exponents, HRR
// binomials and register-array offsets are all resolved at compile time.
template <typename F, int... I>
__device__ __forceinline__ void sfor_impl(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void sfor(F&& f) {
  if constexpr (N > 0) sfor_impl(f, std::make_integer_sequence<int, N>{});
}
#define OQPH_CI(x) decltype(x)::value

// ------------------------------------------------------------------ FP64 rcp
// Hardware reciprocal / reciprocal square root seeds (relative error about
// 2^-22) refined to full precision: two Newton steps for the reciprocal, one
// third-order step (residual e^3, 2^-64) for the reciprocal square root, two
// operations shorter than two Newton steps; arguments are positive normal
// numbers (exponent sums, Boys arguments).
__device__ __forceinline__ double rcp64(double x) {
  double y = __builtin_amdgcn_rcp(x);
  double e = fma(-x, y, 1.0);
  y = fma(y, e, y);
  e = fma(-x, y, 1.0);
  return fma(y, e, y);
}
__device__ __forceinline__ double rsq64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);  // 1 - x y^2
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// Load a primitive pair whose index is uniform across the wavefront through
// the constant address space, so it is served by the scalar cache.
__device__ __forceinline__ PrimJK load_uniform(const PrimJK* p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
  const __attribute__((address_space(4))) double* q =
      (const __attribute__((address_space(4))) double*)(p + i);
  PrimJK r;
  r.g = q[0]; r.Kg = q[1]; r.X[0] = q[2]; r.X[1] = q[3]; r.X[2] = q[4]; r.h = q[5];
  return r;
#else
  return p[i];
#endif
}
__device__ __forceinline__ PrimF32 load_uniform(const PrimF32* p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
  const __attribute__((address_space(4))) float* q =
      (const __attribute__((address_space(4))) float*)(p + i);
  PrimF32 r;
  r.g = q[0]; r.Kg = q[1]; r.X[0] = q[2]; r.X[1] = q[3]; r.X[2] = q[4]; r.h = q[5];
  return r;
#else
  return p[i];
#endif
}
__device__ __forceinline__ PrimPair load_uniform(const PrimPair* p, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
  const __attribute__((address_space(4))) double* q =
      (const __attribute__((address_space(4))) double*)(p + i);
  PrimPair r;
  r.g = q[0]; r.Kg = q[1]; r.P[0] = q[2]; r.P[1] = q[3]; r.P[2] = q[4]; r.a = q[5]; r.b = q[6]; r.h = q[7];
  return r;
#else
  return p[i];
#endif
}

// ------------------------------------------------------------------ Rys roots
#include "rys_table.inc"
#include "rys_table_f32.inc"

// ------------------------------------------------------------ Boys functions
// The Boys tables follow the Rys tables in the device buffers.
#include "boys_table.inc"

// F[0..M], M <= 3, at T.  tab: the m0 = max(M - 1, 0) block of the table,
// rows of one polynomial in u = T_k - T around the nearest grid point T_k =
// k/2, whose value is F_m0 and whose derivative is F_m0+1; the lower orders
// follow from e^-T = (2 m0 + 1) F_m0 - 2 T F_m0+1 and the downward recursion.
// One row is 12 (FP64) or 8 (FP32) coefficients, against 26 (14) for a root
// and weight of the Rys fits and 52 (28) for two.  The step of 1/2 is a
// balance: 1/4 needs two coefficients less but 5 KB more LDS per block, which
// costs (ps|ss) its third block per CU.
template <int M, typename R>
__device__ __forceinline__ void boys(R T, const R* __restrict__ tab, R (&F)[M + 1]) {
  constexpr bool F32 = sizeof(R) == 4;
  constexpr int m0 = M > 0 ? M - 1 : 0, deg = F32 ? BOYS32_DEG : BOYS_DEG;
  if (T >= (R)BOYS_TMAX[m0]) {
    const R rs = F32 ? (R)__builtin_amdgcn_rsqf((float)T) : (R)rsq64((double)T);
    F[0] = (R)0.88622692545275801364 * rs;
    const R h = (R)0.5 * rs * rs;
#pragma unroll
    for (int m = 1; m <= M; ++m) F[m] = (R)(2 * m - 1) * h * F[m - 1];
    return;
  }
  // nearest multiple of 1/2: adding 1.5 2^51 (2^22) leaves an ulp of 1/2, and
  // the low bits of the sum count halves
  R Tk;
  int k;
  if constexpr (F32) {
    const float x = (float)T + 6291456.0f;
    k = __float_as_int(x) & 0x3ff;
    Tk = x - 6291456.0f;
  } else {
    const double x = (double)T + 3377699720527872.0;
    k = __double2loint(x) & 0x3ff;
    Tk = x - 3377699720527872.0;
  }
  const R u = Tk - T;
  R c[deg + 1];
  // rows are 16-byte aligned
  typedef typename std::conditional<F32, float4, double2>::type V;
  constexpr int nv = 16 / sizeof(R);
  const V* r = (const V*)(tab + k * (deg + 1));
#pragma unroll
  for (int j = 0; j <= deg; j += nv) {
    const V t = r[j / nv];
    c[j] = t.x;
    c[j + 1] = t.y;
    if constexpr (F32) {
      c[j + 2] = t.z;
      c[j + 3] = t.w;
    }
  }
  R v = c[deg], d = c[deg];
  v = v * u + c[deg - 1];
#pragma unroll
  for (int j = deg - 2; j >= 0; --j) {
    if (M > 0) d = d * u + v;
    v = v * u + c[j];
  }
  F[m0] = v;
  if constexpr (M > 0) {
    F[M] = d;
    if constexpr (M > 1) {
      const R T2 = T + T;
      const R e = (R)(2 * m0 + 1) * v - T2 * d;
#pragma unroll
      for (int m = m0; m > 0; --m) F[m - 1] = (T2 * F[m] + e) * (R)(1.0 / (2 * m - 1));
    }
  }
}

// length of the N-root block of each table (entries); the blocks start at
// RYS_OFF[N] / RYS32_OFF[N]
template <int N>
__host__ __device__ constexpr int rys_len() { return RYS_TASYM[N] * 2 * N * (RYS_DEG + 1); }
template <int N>
__host__ __device__ constexpr int rys32_len() { return RYS_TASYM[N] * 2 * N * (RYS32_DEG + 1); }

// Nodes t^2 and weights of the N-root Rys quadrature at argument T.  tabN is
// the N-root block of the FP64 table (global memory or a block-shared copy):
// per unit interval k = floor(T), 2N degree-12 polynomials in s = 2(T-k)-1.
// Beyond RYS_TASYM[N] the Hermite limit t^2 = r_i / T, w = h_i / sqrt(T).
template <int N>
__device__ __forceinline__ void rys_roots(double T, const double* __restrict__ tabN, double* x, double* w) {
  if (T >= (double)RYS_TASYM[N]) {
    const double rs = rsq64(T), it = rs * rs;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      x[i] = RYS_HERM[RYS_HOFF[N] + i] * it;
      w[i] = RYS_HERM[RYS_HOFF[N] + N + i] * rs;
    }
    return;
  }
  const int k = (int)T;
  const double s = 2.0 * (T - (double)k) - 1.0;
  const double* c = tabN + k * (2 * N * (RYS_DEG + 1));
#pragma unroll
  for (int f = 0; f < 2 * N; ++f) {
    double v = c[f * (RYS_DEG + 1) + RYS_DEG];
#pragma unroll
    for (int j = RYS_DEG - 1; j >= 0; --j) v = fma(v, s, c[f * (RYS_DEG + 1) + j]);
    if (f < N) x[f] = v; else w[f - N] = v;
  }
}

// FP32 roots: degree-6 fits on the same intervals, hardware rcp / rsqrt
template <int N>
__device__ __forceinline__ void rys_roots32(float T, const float* __restrict__ tabN, float* x, float* w) {
  if (T >= (float)RYS_TASYM[N]) {
    const float rs = __builtin_amdgcn_rsqf(T), it = rs * rs;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      x[i] = (float)RYS_HERM[RYS_HOFF[N] + i] * it;
      w[i] = (float)RYS_HERM[RYS_HOFF[N] + N + i] * rs;
    }
    return;
  }
  const int k = (int)T;
  const float s = 2.0f * (T - (float)k) - 1.0f;
  const float* c = tabN + k * (2 * N * (RYS32_DEG + 1));
#pragma unroll
  for (int f = 0; f < 2 * N; ++f) {
    float v = c[f * (RYS32_DEG + 1) + RYS32_DEG];
#pragma unroll
    for (int j = RYS32_DEG - 1; j >= 0; --j) v = fmaf(v, s, c[f * (RYS32_DEG + 1) + j]);
    if (f < N) x[f] = v; else w[f - N] = v;
  }
}

// One node/weight pair (root r, runtime index) of the N-root quadrature, for
// root loops kept rolled to bound register pressure.
template <int N, typename R>
__device__ __forceinline__ void rys_root_one(R T, const double* __restrict__ tabN, const float* __restrict__ tab32N,
                                             int r, R& x, R& w) {
  if constexpr (sizeof(R) == 4) {
    if (T >= (float)RYS_TASYM[N]) {
      const float rs = __builtin_amdgcn_rsqf(T);
      x = (float)RYS_HERM[RYS_HOFF[N] + r] * (rs * rs);
      w = (float)RYS_HERM[RYS_HOFF[N] + N + r] * rs;
      return;
    }
    const int k = (int)T;
    const float s = 2.0f * (T - (float)k) - 1.0f;
    const float* cx = tab32N + k * (2 * N * (RYS32_DEG + 1)) + r * (RYS32_DEG + 1);
    const float* cw = cx + N * (RYS32_DEG + 1);
    float vx = cx[RYS32_DEG], vw = cw[RYS32_DEG];
#pragma unroll
    for (int j = RYS32_DEG - 1; j >= 0; --j) {
      vx = fmaf(vx, s, cx[j]);
      vw = fmaf(vw, s, cw[j]);
    }
    x = vx;
    w = vw;
  } else {
    if (T >= (double)RYS_TASYM[N]) {
      const double rs = rsq64(T);
      x = RYS_HERM[RYS_HOFF[N] + r] * rs * rs;
      w = RYS_HERM[RYS_HOFF[N] + N + r] * rs;
      return;
    }
    const int k = (int)T;
    const double s = 2.0 * (T - (double)k) - 1.0;
    const double* cx = tabN + k * (2 * N * (RYS_DEG + 1)) + r * (RYS_DEG + 1);
    const double* cw = cx + N * (RYS_DEG + 1);
    double vx = cx[RYS_DEG], vw = cw[RYS_DEG];
#pragma unroll
    for (int j = RYS_DEG - 1; j >= 0; --j) {
      vx = fma(vx, s, cx[j]);
      vw = fma(vw, s, cw[j]);
    }
    x = vx;
    w = vw;
  }
}

// ------------------------------------------------- contracted (e0|f0) via Rys
// acc[e][f]: e over levels LA..LA+LB (local offset ncum(LA-1)), f over LC..LC+LD.
template <int LA, int LB, int LC, int LD>
struct Dims {
  static constexpr int LAB = LA + LB, LCD = LC + LD;
  static constexpr int NE = ncum(LAB) - ncum(LA - 1);
  static constexpr int NF = ncum(LCD) - ncum(LC - 1);
  static constexpr int NROOT = (LAB + LCD) / 2 + 1;
  static constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  static constexpr int NBLK = NA * NB * NC * ND;
};

// level and local index of the e-th entry of a level range starting at L0
template <int L0>
__host__ __device__ constexpr int range_level(int e) {
  int L = L0;
  while (e >= ncart(L)) { e -= ncart(L); ++L; }
  return L;
}
template <int L0>
__host__ __device__ constexpr int range_local(int e) {
  int L = L0;
  while (e >= ncart(L)) { e -= ncart(L); ++L; }
  return e;
}
template <int L0>
__host__ __device__ constexpr int range_index(int L, int c) { return ncum(L - 1) - ncum(L0 - 1) + c; }

// Algorithmic FLOP model of one surviving primitive quartet (Rys): roots,
// recursion coefficients, 2D VRR, (e0|f0) assembly -- shared with the
// benchmark's roofline accounting.
__host__ __device__ constexpr long long flops_prim_rt(int LA, int LB, int LC, int LD) {
  const int LAB = LA + LB, LCD = LC + LD, nr = (LAB + LCD) / 2 + 1;
  const int nc = ncart(LA) * ncart(LB) * ncart(LC) * ncart(LD);
  return (long long)nr * (56 + 12 * (LAB + 1) * (LCD + 1) + 6 * (LA + 1) * (LB + 1) * (LCD + 1) +
                          6 * (LA + 1) * (LB + 1) * (LC + 1) * (LD + 1) + 3 * nc);
}
template <int LA, int LB, int LC, int LD>
__host__ __device__ constexpr long long flops_prim() {
  return flops_prim_rt(LA, LB, LC, LD);
}
// The same model for the derivative integrals of the gradient: the
// differentiated centres raised by one, one more root level, and the
// assembly term four times (value and three derivative components).
__host__ __device__ constexpr long long flops_grad_prim_rt(int LA, int LB, int LC, int LD) {
  const int LAB = LA + LB + 1, LCD = LC + LD + 1, nr = (LAB + LCD - 1) / 2 + 1;
  const int nc = ncart(LA) * ncart(LB) * ncart(LC) * ncart(LD);
  return (long long)nr * (56 + 12 * (LAB + 1) * (LCD + 1) + 6 * (LA + 2) * (LB + 2) * (LCD + 1) +
                          6 * (LA + 2) * (LB + 2) * (LC + 2) * (LD + 1) + 3 * 4 * nc);
}

// Classes whose total angular momentum is at most 3: the (e0|f0) integrals
// come from F_0..F_3 by the Obara-Saika vertical recursion (J. Chem. Phys. 84,
// 3963 (1986)) instead of one or two Rys roots.  What bounds these classes is
// the instructions per primitive quartet (lane divergence apart) and the LDS
// reads of the fit; the recursion needs 2-6 Boys values from one table row and,
// for (ps|ps), 33 operations instead of the 90 of two roots.
template <int LA, int LB, int LC, int LD>
constexpr bool use_os() {
  return LA + LB + LC + LD <= 3;
}
// The class's table block: Boys functions or Rys roots (offset in the device
// buffers, length; in doubles / floats).
template <int LA, int LB, int LC, int LD>
struct QTab {
  static constexpr bool os = use_os<LA, LB, LC, LD>();
  static constexpr int NR = Dims<LA, LB, LC, LD>::NROOT;
  static constexpr int L = LA + LB + LC + LD, m0 = os ? (L > 0 ? L - 1 : 0) : 0;
  static constexpr int off64 = os ? RYS_TABLE_SIZE + BOYS_OFF[m0] : RYS_OFF[NR];
  static constexpr int len64 = os ? BOYS_OFF[m0 + 1] - BOYS_OFF[m0] : rys_len<NR>();
  static constexpr int off32 = os ? RYS32_TABLE_SIZE + BOYS32_OFF[m0] : RYS32_OFF[NR];
  static constexpr int len32 = os ? BOYS32_OFF[m0 + 1] - BOYS32_OFF[m0] : rys32_len<NR>();
};

// Recursion axis of component (x, y, z): an exponent of one where there is
// one (no (n - 1) term), else the first nonzero
__host__ __device__ constexpr int os_axis(int x, int y, int z) {
  return x == 1 ? 0 : y == 1 ? 1 : z == 1 ? 2 : x ? 0 : y ? 1 : 2;
}

// Adds pref (e0|f0) of one primitive quartet to acc from pF[m] = pref F_m.
// Ket classes of these classes have LCD <= 1 (the bra class is never the
// smaller one).  WP = W - P = -rz PQ, WQ = W - Q = re PQ.
template <int LA, int LB, int LC, int LD, typename R>
__device__ __forceinline__ void os_add(const R (&PA)[3], const R (&QC)[3], const R (&PQ)[3], R rz, R re, R h2z, R h2ze,
                                       const R (&pF)[LA + LB + LC + LD + 1],
                                       R (&acc)[Dims<LA, LB, LC, LD>::NE][Dims<LA, LB, LC, LD>::NF]) {
  constexpr int LAB = LA + LB, LCD = LC + LD, M = LAB + LCD, NC = ncum(LAB), E0 = ncum(LA - 1);
  static_assert(LCD <= 1 && M <= 3, "os_add: class out of range");
  R E[M + 1][NC], WP[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) WP[d] = -rz * PQ[d];
#pragma unroll
  for (int m = 0; m <= M; ++m) E[m][0] = pF[m];
  sfor<NC>([&](auto Ei) {
    constexpr int e = OQPH_CI(Ei);
    if constexpr (e > 0) {
      constexpr int L = range_level<0>(e), c = range_local<0>(e);
      constexpr int x = c_lx(L, c), y = c_ly(L, c), z = c_lz(L, c), ax = os_axis(x, y, z);
      constexpr int n = (ax == 0 ? x : ax == 1 ? y : z) - 1;  // exponent of the lower component
      constexpr int lo = range_index<0>(L - 1, c_idx(x - (ax == 0), y - (ax == 1), z - (ax == 2)));
      constexpr int lo2 = n > 0 ? range_index<0>(L - 2, c_idx(x - 2 * (ax == 0), y - 2 * (ax == 1), z - 2 * (ax == 2))) : 0;
      sfor<M - L + 1>([&](auto Mi) {
        constexpr int m = OQPH_CI(Mi);
        R v = PA[ax] * E[m][lo];
        v = WP[ax] * E[m + 1][lo] + v;
        if constexpr (n > 0) v = (R)n * h2z * (E[m][lo2] - rz * E[m + 1][lo2]) + v;
        E[m][e] = v;
      });
    }
  });
  if constexpr (LCD == 0) {
#pragma unroll
    for (int e = 0; e < Dims<LA, LB, LC, LD>::NE; ++e) acc[e][0] += E[0][E0 + e];
  } else {
    // |p_i): QC_i (e|^(0) + WQ_i (e|^(1) + e_i / (2 (zeta + eta)) (e - 1_i|^(1)
    R WQ[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) WQ[d] = re * PQ[d];
    sfor<Dims<LA, LB, LC, LD>::NE>([&](auto Ei) {
      constexpr int e = OQPH_CI(Ei) + E0;
      constexpr int L = range_level<0>(e), c = range_local<0>(e);
      sfor<3>([&](auto Di) {
        constexpr int d = OQPH_CI(Di), n = c_l(L, c, d);
        // component order of a p shell: x, y, z
        R v = acc[OQPH_CI(Ei)][d];
        v = QC[d] * E[0][e] + v;
        v = WQ[d] * E[1][e] + v;
        if constexpr (n > 0) {
          constexpr int lo = range_index<0>(L - 1, c_idx(c_lx(L, c) - (d == 0), c_ly(L, c) - (d == 1), c_lz(L, c) - (d == 2)));
          v = (R)n * h2ze * E[1][lo] + v;
        }
        acc[OQPH_CI(Ei)][d] = v;
      });
    });
  }
}

// The fields of a primitive pair that the quadrature reads, in one precision:
// X is the product centre relative to the pair's first centre.
template <typename R>
struct PrimV {
  R g, Kg, X[3], h;
};
// record k of a ket of two s shells from the piecewise copies (JKParams::kt64, kt32)
template <typename R>
__device__ __forceinline__ PrimV<R> ket_prim(const R* __restrict__ kt, unsigned at, int k) {
  typedef R R2 __attribute__((ext_vector_type(2)));
  const R2* t = (const R2*)kt + (at + 192ll * k);
  const R2 a = t[0], b = t[64], c = t[128];
  return {a.x, a.y, {b.x, b.y, c.x}, c.y};
}

template <typename R, typename PP>
__device__ __forceinline__ PrimV<R> prim_v(const PP& p) {
  return {(R)p.g, (R)p.Kg, {(R)p.X[0], (R)p.X[1], (R)p.X[2]}, (R)p.h};
}

template <int LA, int LB, int LC, int LD, typename R>
__device__ __forceinline__ void rys_add(const PrimV<R>& pp, const PrimV<R>& qq, const R (&AQ)[3], R ze, R sq, R ize,
                                        R pref, const double* __restrict__ tabN, const float* __restrict__ tab32N,
                                        R (&acc)[Dims<LA, LB, LC, LD>::NE][Dims<LA, LB, LC, LD>::NF]);

// The FP32 quadrature of the small classes folds the ket's product centre
// into the centre difference once per ket primitive pair: AQ = (A - C) - X_q,
// and PQ = AQ + X_p in the loop over bra primitives ((ps|ss) mixed 92 -> 89
// ms on (H2O)64/cc-pVDZ, with the ket prefetch).  Elsewhere AQ = A - C and
// PQ = AQ + X_p - X_q per quartet: FP64 needs all of the ket's 48-byte record
// before its bra loop then ((ps|ss) FP64 122 -> 139 ms), and the larger
// classes have no registers to spare.
template <int LA, int LB, int LC, int LD, typename R>
constexpr bool hoist_ket() {
  return use_os<LA, LB, LC, LD>() || (sizeof(R) == 4 && Dims<LA, LB, LC, LD>::NE * Dims<LA, LB, LC, LD>::NF <= 9);
}
template <int LA, int LB, int LC, int LD, typename R>
__device__ __forceinline__ void ket_offset(const R (&AC)[3], const PrimV<R>& qq, R (&AQ)[3]) {
#pragma unroll
  for (int d = 0; d < 3; ++d) AQ[d] = hoist_ket<LA, LB, LC, LD, R>() ? AC[d] - qq.X[d] : AC[d];
}

// Adds one primitive quartet's (e0|f0) to acc; returns false when the
// primitive prefactor screen |K_ab K_cd| / sqrt(zeta+eta) < qcut drops it.
// pp, qq: bra and ket primitive pairs (X = P - A and X = Q - C); AQ from
// ket_offset, so PA = X_p, QC = X_q and PQ = AQ + X_p (- X_q).
// imu2 = 1/mu^2 selects the erf(mu r)/r operator: zeta + eta becomes
// zeta + eta + zeta eta / mu^2 in every quantity of the quadrature
// (OpenQP's attenuated Rys setup, source/integrals/int_rys.F90:180-182, 227);
// imu2 = 0 is the plain Coulomb operator.
// tabN / tab32N: the NROOT-root blocks of the FP64 / FP32 root tables.
template <int LA, int LB, int LC, int LD, typename R>
__device__ __forceinline__ bool rys_accumulate(const PrimV<R>& pp, const PrimV<R>& qq, const R (&AQ)[3], R qcut2,
                                               R imu2, const double* __restrict__ tabN,
                                               const float* __restrict__ tab32N,
                                               R (&acc)[Dims<LA, LB, LC, LD>::NE][Dims<LA, LB, LC, LD>::NF]) {
  constexpr bool F32 = sizeof(R) == 4;
  const R zeta = pp.g, eta = qq.g;
  const R fqz = pp.Kg * qq.Kg;
  if constexpr (use_os<LA, LB, LC, LD>()) {
    // (1 + eta / mu^2) is constant over the bra primitives, and the survivors
    // need the prefactor anyway: it is screened itself
    const R ze = zeta * ((R)1 + eta * imu2) + eta;
    const R sq = F32 ? (R)__builtin_amdgcn_rsqf((float)ze) : (R)rsq64((double)ze);
    const R pref = fqz * sq;
    if (pref * pref < qcut2) return false;
    rys_add<LA, LB, LC, LD, R>(pp, qq, AQ, ze, sq, sq * sq, pref, tabN, tab32N, acc);
    return true;
  }
  const R ze = zeta + eta + zeta * eta * imu2;
  if (fqz * fqz < qcut2 * ze) return false;
  // 1/sqrt(ze) and its square: one transcendental (FP32: hardware rsq)
  const R sq = F32 ? (R)__builtin_amdgcn_rsqf((float)ze) : (R)rsq64((double)ze);
  const R ize = sq * sq;
  rys_add<LA, LB, LC, LD, R>(pp, qq, AQ, ze, sq, ize, fqz * sq, tabN, tab32N, acc);
  return true;
}

// The quadrature of one primitive quartet without the screen: adds the
// (e0|f0) products, scaled by pref, to acc.  ze = zeta + eta (+ zeta eta /
// mu^2 for the attenuated operator), sq = 1/sqrt(ze), ize = 1/ze.
template <int LA, int LB, int LC, int LD, typename R>
__device__ __forceinline__ void rys_add(const PrimV<R>& pp, const PrimV<R>& qq, const R (&AQ)[3], R ze, R sq, R ize,
                                        R pref, const double* __restrict__ tabN, const float* __restrict__ tab32N,
                                        R (&acc)[Dims<LA, LB, LC, LD>::NE][Dims<LA, LB, LC, LD>::NF]) {
  using Dm = Dims<LA, LB, LC, LD>;
  constexpr int LAB = Dm::LAB, LCD = Dm::LCD, NR = Dm::NROOT;
  constexpr bool F32 = sizeof(R) == 4;
  const R zeta = pp.g, eta = qq.g;
  const R rho = zeta * eta * ize;
  R PQ[3], PA[3], QC[3];
  R pq2 = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    PA[d] = pp.X[d];
    QC[d] = qq.X[d];
    PQ[d] = hoist_ket<LA, LB, LC, LD, R>() ? AQ[d] + pp.X[d] : AQ[d] + pp.X[d] - qq.X[d];
    pq2 += PQ[d] * PQ[d];
  }
  const R T = rho * pq2;
  // rho/zeta = eta/(zeta+eta), rho/eta = zeta/(zeta+eta): no further divisions
  const R rz = eta * ize, re = zeta * ize;
  if constexpr (use_os<LA, LB, LC, LD>()) {
    R F[LAB + LCD + 1];
    if constexpr (F32) boys<LAB + LCD, R>(T, tab32N, F);
    else boys<LAB + LCD, R>(T, tabN, F);
#pragma unroll
    for (int m = 0; m <= LAB + LCD; ++m) F[m] *= pref;
    os_add<LA, LB, LC, LD, R>(PA, QC, PQ, rz, re, pp.h, (R)0.5 * ize, F, acc);
    return;
  }
  const R h2z = pp.h, h2e = qq.h, h2ze = (R)0.5 * ize;
  // one root: 2D integrals G_d(i, k) by the vertical recursion, then the
  // (e0|f0) products
  auto root = [&](const R t2, const R wr) {
    const R B00 = h2ze * t2;
    const R B10 = h2z - h2z * rz * t2;
    const R B01 = h2e - h2e * re * t2;
    R G[3][LAB + 1][LCD + 1];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const R C00 = PA[d] - rz * t2 * PQ[d];
      const R D00 = QC[d] + re * t2 * PQ[d];
      G[d][0][0] = (d == 0) ? pref * wr : (R)1;
#pragma unroll
      for (int i = 1; i <= LAB; ++i) {
        R v = C00 * G[d][i - 1][0];
        if (i > 1) v += (R)(i - 1) * B10 * G[d][i - 2][0];
        G[d][i][0] = v;
      }
#pragma unroll
      for (int k = 1; k <= LCD; ++k) {
#pragma unroll
        for (int i = 0; i <= LAB; ++i) {
          R v = D00 * G[d][i][k - 1];
          if (k > 1) v += (R)(k - 1) * B01 * G[d][i][k - 2];
          if (i > 0) v += (R)i * B00 * G[d][i - 1][k - 1];
          G[d][i][k] = v;
        }
      }
    }
    sfor<Dm::NE>([&](auto E) {
      constexpr int e = OQPH_CI(E);
      constexpr int Le = range_level<LA>(e), ce = range_local<LA>(e);
      constexpr int ex = c_lx(Le, ce), ey = c_ly(Le, ce), ez = c_lz(Le, ce);
      sfor<Dm::NF>([&](auto F) {
        constexpr int f = OQPH_CI(F);
        constexpr int Lf = range_level<LC>(f), cf = range_local<LC>(f);
        constexpr int fx = c_lx(Lf, cf), fy = c_ly(Lf, cf), fz = c_lz(Lf, cf);
        acc[e][f] += G[0][ex][fx] * G[1][ey][fy] * G[2][ez][fz];
      });
    });
  };
  if constexpr (Dm::NE * Dm::NF <= 64) {
    // small classes: all roots at once, root loop unrolled
    R rx[NR], rw[NR];
    if constexpr (F32) rys_roots32<NR>(T, tab32N, rx, rw);
    else rys_roots<NR>(T, tabN, rx, rw);
#pragma unroll
    for (int r = 0; r < NR; ++r) root(rx[r], rw[r]);
  } else {
    // larger classes: one root per iteration of a rolled loop, so only one
    // root's 2D integrals are live next to the accumulators
#pragma unroll 1
    for (int r = 0; r < NR; ++r) {
      R t2, wr;
      rys_root_one<NR, R>(T, tabN, tab32N, r, t2, wr);
      root(t2, wr);
    }
  }
}

// ---------------------------------------------------------------- HRR
// Y[a][b][f] = sum_j prod_d C(b_d,j_d) AB_d^(b_d-j_d) acc[(a+j)][f]
// f runs outermost so each column of acc dies as its Y column is formed.
template <int LA, int LB, int NF, typename R>
__device__ __forceinline__ void hrr_bra(const R (&acc)[ncum(LA + LB) - ncum(LA - 1)][NF], const R* AB,
                                        R (&Y)[ncart(LA) * ncart(LB)][NF]) {
  R pw[3][LB + 1];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    pw[d][0] = (R)1;
#pragma unroll
    for (int k = 1; k <= LB; ++k) pw[d][k] = pw[d][k - 1] * AB[d];
  }
  sfor<NF>([&](auto Fi) {
    constexpr int f = OQPH_CI(Fi);
    sfor<ncart(LA)>([&](auto Ai) {
      constexpr int a = OQPH_CI(Ai);
      constexpr int ax = c_lx(LA, a), ay = c_ly(LA, a), az = c_lz(LA, a);
      sfor<ncart(LB)>([&](auto Bi) {
        constexpr int b = OQPH_CI(Bi);
        constexpr int bx = c_lx(LB, b), by = c_ly(LB, b), bz = c_lz(LB, b);
        R s = 0;
        sfor<bx + 1>([&](auto JX) {
          constexpr int jx = OQPH_CI(JX);
          sfor<by + 1>([&](auto JY) {
            constexpr int jy = OQPH_CI(JY);
            sfor<bz + 1>([&](auto JZ) {
              constexpr int jz = OQPH_CI(JZ);
              constexpr int e = range_index<LA>(LA + jx + jy + jz, c_idx(ax + jx, ay + jy, az + jz));
              constexpr int cb = binom(bx, jx) * binom(by, jy) * binom(bz, jz);
              s += (R)cb * pw[0][bx - jx] * pw[1][by - jy] * pw[2][bz - jz] * acc[e][f];
            });
          });
        });
        Y[a * ncart(LB) + b][f] = s;
      });
    });
  });
}

// V[ab][c][d] = sum_j prod_d C(d_d,j_d) CD_d^(d_d-j_d) Y[ab][(c+j)]
template <int LC, int LD, int NAB, typename R>
__device__ __forceinline__ void hrr_ket(const R (&Y)[NAB][ncum(LC + LD) - ncum(LC - 1)], const R* CD,
                                        R (&V)[NAB * ncart(LC) * ncart(LD)]) {
  R pw[3][LD + 1];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    pw[d][0] = (R)1;
#pragma unroll
    for (int k = 1; k <= LD; ++k) pw[d][k] = pw[d][k - 1] * CD[d];
  }
  sfor<NAB>([&](auto ABi) {
    constexpr int ab = OQPH_CI(ABi);
    sfor<ncart(LC)>([&](auto Ci) {
      constexpr int c = OQPH_CI(Ci);
      constexpr int cx = c_lx(LC, c), cy = c_ly(LC, c), cz = c_lz(LC, c);
      sfor<ncart(LD)>([&](auto Di) {
        constexpr int dd = OQPH_CI(Di);
        constexpr int dx = c_lx(LD, dd), dy = c_ly(LD, dd), dz = c_lz(LD, dd);
        R s = 0;
        sfor<dx + 1>([&](auto JX) {
          constexpr int jx = OQPH_CI(JX);
          sfor<dy + 1>([&](auto JY) {
            constexpr int jy = OQPH_CI(JY);
            sfor<dz + 1>([&](auto JZ) {
              constexpr int jz = OQPH_CI(JZ);
              constexpr int f = range_index<LC>(LC + jx + jy + jz, c_idx(cx + jx, cy + jy, cz + jz));
              constexpr int cb = binom(dx, jx) * binom(dy, jy) * binom(dz, jz);
              s += (R)cb * pw[0][dx - jx] * pw[1][dy - jy] * pw[2][dz - jz] * Y[ab][f];
            });
          });
        });
        V[(ab * ncart(LC) + c) * ncart(LD) + dd] = s;
      });
    });
  });
}

}  // namespace oqph
