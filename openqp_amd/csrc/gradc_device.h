// gradc_device.h -- cooperative 2e-gradient kernel of the larger quartet classes.
//
// One wavefront (one block) takes the kets of one bra segment and evaluates
// 64 / W quartets at a time, W lanes on each: one per (a, b), at least three per
// root, all 64 above 32; class known at compile time.  Per quartet:
//   0. lane = (a, b): its row Gamma[cd] of the two-particle density in
//      registers, and the fine screen;
// per batch of primitive quartets
//   1. lane = (primitive quartet, root, axis): the 2D integrals, one level
//      higher on each side, into LDS;
// and per primitive quartet and root
//   2. lane = (axis, ia, ib): the 2D integrals transferred to the exponents
//      (ia <= la + 1, ib <= lb + 1 | ic <= lc + 1, id <= ld) into LDS;
//   3. lane = (a, b): per axis the adjoint of the transferred integrals,
//      W_x[ic, id] = sum_cd Gamma I_y I_z, contracted with the rows of
//      ia + 1, ia - 1, ib + 1, ib - 1, ic + 1, ic - 1: 8 operations per component
//      and 18 per (ic, id) instead of 27 per component.
//
// What bounds it and why this split: the per-lane templates (k_grad) hold the
// Gamma block of a quartet and every transferred integral in one lane, take all
// 256 VGPRs and spill 0.6-3.2 KB; the run-time-class kernel (k_gradh) spends
// its time on index arithmetic and LDS round trips.  Here a lane holds one row
// of Gamma and two small tables, with constant indices; LDS reads and
// the serial chain of a quartet's primitives and roots remain.  A gradient of
// (H2O)16/cc-pVTZ 435 -> 247 ms, C20H42/6-31G(d) 18.7 -> 13.9 (224 and 12.1 with
// k_grad as it is now), one water in cc-pVTZ 25.3 -> 9.0; the figures per class are at gradc_class() in session.hip.
#pragma once
#include "eri_device.h"
#include "grad_params.h"

namespace oqph {

template <int LA, int LB, int LC, int LD>
struct GRC {
  static constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  static constexpr int NAB = NA * NB, NCD = NC * ND;
  static constexpr int NR = (LA + LB + LC + LD + 1) / 2 + 1;
  static constexpr int LAB = LA + LB + 1, LCD = LC + LD + 1, GA = (LAB + 1) * (LCD + 1);
  // lanes per quartet, quartets per wavefront
  // three quartets of up to 21 lanes where 16 do not suffice: (dp|ds) 16.6 -> 13.7 ms,
  // (dp|pp) 13.9 -> 11.7, (dp|dp) 7.9 -> 6.6 ((H2O)16/cc-pVTZ); groups of 9, 10 and 30
  // lanes gained nothing where more quartets of unequal length meet
  static constexpr int WMIN = NAB > 3 * NR ? NAB : 3 * NR;
  static constexpr int W = WMIN <= 16 ? 16 : WMIN <= 21 ? WMIN : WMIN <= 32 ? 32 : 64;
  static constexpr int NQ = 64 / W, AT = (NAB + W - 1) / W;
  // primitive quartets per batch of phase 1
  static constexpr int PB = W / (3 * NR) < 1 ? 1 : (W / (3 * NR) > 2 ? 2 : W / (3 * NR));
  static constexpr int TB = LB + 2, TR = (LC + 2) * (LD + 1);  // transferred rows: [axis][ia][ib][TR]
  static constexpr int NT = 3 * (LA + 2) * TB, TT = (NT + W - 1) / W;
  static constexpr int N2 = (LC + 1) * (LD + 1);
  static constexpr int SLOT = (PB * NR * 3 * GA + NT * TR) | 1;
  static constexpr int lds = 8 * NQ * SLOT;
  // Gamma rows and the two tables of a lane (doubles)
  static constexpr int live = AT * NCD + 6 * N2;
  static constexpr bool fits = lds <= 48 * 1024 && 3 * NR <= W && live <= 160;
  static constexpr int waves = live <= 80 ? 2 : 1;
};

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(GRC<LA, LB, LC, LD>::waves)))
void k_gradc(GradParams prm, WaveWork ww) {
  using J = GRC<LA, LB, LC, LD>;
  constexpr int NB = J::NB, NC = J::NC, ND = J::ND, NAB = J::NAB, NCD = J::NCD, NR = J::NR;
  constexpr int LAB = J::LAB, LCD = J::LCD, GA = J::GA, W = J::W, NQ = J::NQ, AT = J::AT, PB = J::PB, TB = J::TB,
                TR = J::TR, NT = J::NT, TT = J::TT, N2 = J::N2;
  __shared__ double s_slot[NQ][J::SLOT];
  extern __shared__ double s_de[];  // 3 natm
  // the lanes past the last quartet's take no part
  const int lane = (int)threadIdx.x, q = min(lane / W, NQ - 1), l = lane - q * W;
  const bool spare = l >= W;
  for (int i = lane; i < 3 * prm.natm; i += 64) s_de[i] = 0.0;
  // ---- the block's kets: [sub kpb, (sub + 1) kpb) of one 64-ket chunk of one segment
  const int kpb = ww.kpb > 0 ? ww.kpb : 64, per = 64 / kpb;
  const long long wave = (long long)blockIdx.x / per;
  const int sub = (int)((long long)blockIdx.x - wave * per);
  if (wave >= ww.nwaves) return;  // block-uniform
  int lo = 0, hi = ww.nseg;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (ww.choff[mid] <= wave) lo = mid; else hi = mid;
  }
  const int seg = __builtin_amdgcn_readfirstlane(lo);
  const int k0 = (int)(wave - ww.choff[seg]) * 64 + sub * kpb;
  const int nk = min(kpb, ww.seg_n[seg] - k0);  // kets of this block
  if (nk <= 0) return;                          // block-uniform
  const int ip = __builtin_amdgcn_readfirstlane(ww.seg_bra[seg]);
  const int ket0 = ww.seg_k0[seg] + k0;
  const ShellPair P = prm.pairs[ip];
  const int n = prm.ncf, oa = prm.coff[P.sa], ob = prm.coff[P.sb];
  const double* __restrict__ Dc = prm.Dc;
  double ABv[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) ABv[d] = P.A[d] - P.B[d];
  // this lane's transfers of phase 2: rows (x, ia, ib) and their coefficients
  // C(ib, j) AB_x^(ib - j) (0 for j > ib); row offsets of G
  int tx[TT], trow[TT];
  double cb[TT][LB + 2];
#pragma unroll
  for (int u = 0; u < TT; ++u) {
    const int t = l + W * u, x = t / ((LA + 2) * TB), r = t - x * (LA + 2) * TB, ia = r / TB, ib = r - ia * TB;
    const bool ok = !spare && t < NT && ia + ib <= LAB;
    tx[u] = ok ? x : -1;
    trow[u] = ia;
    const double ab = x == 0 ? ABv[0] : x == 1 ? ABv[1] : ABv[2];
#pragma unroll
    for (int j = 0; j < LB + 2; ++j) {
      double v = j <= ib ? 1.0 : 0.0;
      for (int i = j; i < ib; ++i) v *= ab;  // AB^(ib - j)
      double c = 1.0;
      for (int i = 1; i <= j; ++i) c = c * (double)(ib - i + 1) / (double)i;
      cb[u][j] = j <= ib ? v * c : 0.0;
    }
  }
  // this lane's components (a, b) of phases 0 and 3: exponents as rows of the transferred table
  int ra[AT], rb[AT], ea[AT][3], eb[AT][3];
#pragma unroll
  for (int t = 0; t < AT; ++t) {
    int ab = l + W * t;
    if (ab >= NAB) ab = 0;
    ra[t] = ab / NB;
    rb[t] = ab - ra[t] * NB;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      ea[t][x] = c_l(LA, ra[t], x);
      eb[t][x] = c_l(LB, rb[t], x);
    }
  }
  // phase 1: this lane's (primitive quartet of a batch, root, axis)
  const int pi = l / (3 * NR), r1 = (l - pi * 3 * NR) / 3, d1 = l - pi * 3 * NR - 3 * r1;
  const bool vrr_lane = !spare && l < PB * 3 * NR;
  double* G = s_slot[q];
  double* T = G + PB * NR * 3 * GA;
  const double* tabN = prm.rys + RYS_OFF[NR];
  const int at0 = prm.shell_atom[P.sa], at1 = prm.shell_atom[P.sb];
  double fA[3] = {0, 0, 0}, fB[3] = {0, 0, 0};  // the bra centres' sums over the block's kets
  unsigned n_comp = 0, n_skip = 0, n_prim = 0;
  for (int i0 = 0; i0 < nk; i0 += NQ) {
    const bool on = !spare && i0 + q < nk;
    const int jq = ww.ket[ket0 + (on ? i0 + q : 0)];
    const ShellPair Q = prm.pairs[jq];
    const int oc = prm.coff[Q.sa], od = prm.coff[Q.sb];
    // ---- phase 0: Gamma rows and the fine screen (grd2.F90:348)
    double Gam[AT][NCD], gm = 0.0;
#pragma unroll
    for (int t = 0; t < AT; ++t) {
      const int a = oa + ra[t], b = ob + rb[t];
      const bool in = !spare && l + W * t < NAB;
      const double dab = 4.0 * prm.cs * Dc[a * n + b];
      double Dac[NC], Dad[ND], Dbc[NC], Dbd[ND];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        Dac[c] = Dc[a * n + oc + c];
        Dbc[c] = Dc[b * n + oc + c];
      }
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        Dad[d] = Dc[a * n + od + d];
        Dbd[d] = Dc[b * n + od + d];
      }
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int d = 0; d < ND; ++d)
          Gam[t][c * ND + d] = dab * Dc[(oc + c) * n + od + d] - prm.hs * (Dac[c] * Dbd[d] + Dad[d] * Dbc[c]);
#pragma unroll
      for (int i = 0; i < NCD; ++i) {
        if (!in) Gam[t][i] = 0.0;
        gm = fmax(gm, fabs(Gam[t][i]));
      }
    }
    // largest of the quartet's lanes: cyclic shifts within the group
#pragma unroll
    for (int o = 1; o < W; o <<= 1) gm = fmax(gm, __shfl(gm, q * W + (l + o) % W));
    const bool skip = !on || gm * P.Q * Q.Q < 0.5 * prm.gcut;
    if (l == 0) {
      n_skip += (on && skip) ? 1 : 0;
      n_comp += skip ? 0 : 1;
    }
    if (__ballot(!skip) == 0ull) continue;  // block-uniform
    const double dab2 = gm * gm;
    double CDv[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) CDv[d] = Q.A[d] - Q.B[d];
    double f0[3] = {0, 0, 0}, f1[3] = {0, 0, 0}, f2[3] = {0, 0, 0};
    const int NP = P.nprim, NPQ = skip ? 0 : NP * Q.nprim;
    int Tmax = NPQ;
    if (NQ > 1)
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) Tmax = max(Tmax, __shfl_xor(Tmax, o));
    Tmax = __builtin_amdgcn_readfirstlane(Tmax);
    int pb = pi, pk = 0, np = 0;
    while (pb >= NP && pk < Q.nprim) { pb -= NP; ++pk; }
    for (int t0 = 0; t0 < Tmax; t0 += PB) {
      // ---- phase 1: 2D integrals G[(primitive, root, axis)][i][k]
      __syncthreads();  // the previous readers of G are done
      bool pass = false;
      if (vrr_lane) {
        const bool in = t0 + pi < NPQ;
        const PrimPair pp = prm.prims[P.prim0 + (in ? pb : 0)];
        const PrimPair qq = prm.prims[Q.prim0 + (in ? pk : 0)];
        const double zeta = pp.g, eta = qq.g, ze = zeta + eta, fqz = pp.Kg * qq.Kg;
        // primitive screens (grd2_rys.F90:375-376), prefactor cutoff (1e-20)^2
        pass = in && !(fqz * fqz < 1.0e-40 * ze) && !(fqz * fqz * dab2 < prm.dabcut2 * ze);
        np += (pass && r1 == 0 && d1 == 0) ? 1 : 0;
        const double sq = rsq64(ze), ize = sq * sq;
        const double PQ0 = pp.P[0] - qq.P[0], PQ1 = pp.P[1] - qq.P[1], PQ2 = pp.P[2] - qq.P[2];
        const double Tb = zeta * eta * ize * (PQ0 * PQ0 + PQ1 * PQ1 + PQ2 * PQ2);
        double t2, wr;
        rys_root_one<NR, double>(Tb, tabN, nullptr, r1, t2, wr);
        const double rz = eta * ize, re = zeta * ize;
        const double B00 = 0.5 * ize * t2, B10 = pp.h - pp.h * rz * t2, B01 = qq.h - qq.h * re * t2;
        const double PQ = d1 == 0 ? PQ0 : d1 == 1 ? PQ1 : PQ2;
        const double PA = d1 == 0 ? pp.P[0] - P.A[0] : d1 == 1 ? pp.P[1] - P.A[1] : pp.P[2] - P.A[2];
        const double QC = d1 == 0 ? qq.P[0] - Q.A[0] : d1 == 1 ? qq.P[1] - Q.A[1] : qq.P[2] - Q.A[2];
        const double C00 = PA - rz * t2 * PQ, D00 = QC + re * t2 * PQ;
        double* g = G + ((pi * NR + r1) * 3 + d1) * GA;
        double c1[LAB + 1], c2[LAB + 1];
        // a dropped primitive quartet contributes zeros through its x table
        c1[0] = d1 == 0 ? (pass ? fqz * sq * wr : 0.0) : 1.0;
#pragma unroll
        for (int i = 1; i <= LAB; ++i) {
          double v = C00 * c1[i - 1];
          if (i > 1) v += (double)(i - 1) * B10 * c1[i - 2];
          c1[i] = v;
        }
#pragma unroll
        for (int i = 0; i <= LAB; ++i) {
          g[i * (LCD + 1)] = c1[i];
          c2[i] = 0.0;
        }
#pragma unroll
        for (int kx = 1; kx <= LCD; ++kx) {
          double cn[LAB + 1];
#pragma unroll
          for (int i = 0; i <= LAB; ++i) {
            double v = D00 * c1[i];
            if (kx > 1) v += (double)(kx - 1) * B01 * c2[i];
            if (i > 0) v += (double)i * B00 * c1[i - 1];
            cn[i] = v;
            g[i * (LCD + 1) + kx] = v;
          }
#pragma unroll
          for (int i = 0; i <= LAB; ++i) {
            c2[i] = c1[i];
            c1[i] = cn[i];
          }
        }
      }
      const unsigned long long pmask = __ballot(pass);
#pragma unroll 1
      for (int b = 0; b < PB; ++b) {
        // exponents of batch primitive b, for this lane's quartet (its own pair index)
        const int tb = t0 + b;
        const bool in = tb < NPQ;
        const int ik = in ? tb / NP : 0, ib = in ? tb - ik * NP : 0;
        unsigned long long bmask = 0ull;  // lanes of phase 1 that hold primitive b
#pragma unroll
        for (int s = 0; s < NQ; ++s) bmask |= ((1ull << (3 * NR)) - 1ull) << (s * W + b * 3 * NR);
        if ((pmask & bmask) == 0ull) continue;  // wave-uniform: dropped in every quartet
        const double a2 = 2.0 * prm.prims[P.prim0 + ib].a, b2 = 2.0 * prm.prims[P.prim0 + ib].b,
                     c2x = 2.0 * prm.prims[Q.prim0 + ik].a;
#pragma unroll 1
        for (int r = 0; r < NR; ++r) {
          __syncthreads();  // G written, or the previous root's readers of T done
          // ---- phase 2: T[x][ia][ib][ic][id]
#pragma unroll
          for (int u = 0; u < TT; ++u) {
            const int x = tx[u];
            if (x >= 0) {
              const double* g = G + ((b * NR + r) * 3 + x) * GA;
              double h[LCD + 1];
#pragma unroll
              for (int kx = 0; kx <= LCD; ++kx) h[kx] = 0.0;
#pragma unroll
              for (int j = 0; j < LB + 2; ++j) {
                const double* gr = g + min(trow[u] + j, LAB) * (LCD + 1);
#pragma unroll
                for (int kx = 0; kx <= LCD; ++kx) h[kx] += cb[u][j] * gr[kx];
              }
              const double cd = x == 0 ? CDv[0] : x == 1 ? CDv[1] : CDv[2];
              double pw[LD + 1];
              pw[0] = 1.0;
#pragma unroll
              for (int i = 1; i <= LD; ++i) pw[i] = pw[i - 1] * cd;
              double* to = T + (l + W * u) * TR;
              sfor<LC + 2>([&](auto Ci) {
                constexpr int ic = OQPH_CI(Ci);
                sfor<LD + 1>([&](auto Di) {
                  constexpr int id = OQPH_CI(Di);
                  double v = 0.0;
                  sfor<id + 1>([&](auto Mi) {
                    constexpr int m = OQPH_CI(Mi);
                    if constexpr (ic + m <= LCD) v += (double)binom(id, m) * pw[id - m] * h[ic + m];
                  });
                  to[ic * (LD + 1) + id] = v;
                });
              });
            }
          }
          __syncthreads();
          // ---- phase 3
#pragma unroll
          for (int t = 0; t < AT; ++t) {
            double I[3][N2], Wx[3][N2];
            int row[3];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
              row[x] = ((x * (LA + 2) + ea[t][x]) * TB + eb[t][x]) * TR;
#pragma unroll
              for (int i = 0; i < N2; ++i) {
                I[x][i] = T[row[x] + i];
                Wx[x][i] = 0.0;
              }
            }
            sfor<NC>([&](auto Ci) {
              constexpr int c = OQPH_CI(Ci);
              sfor<ND>([&](auto Di) {
                constexpr int d = OQPH_CI(Di);
                constexpr int ix = c_lx(LC, c) * (LD + 1) + c_lx(LD, d), iy = c_ly(LC, c) * (LD + 1) + c_ly(LD, d),
                              iz = c_lz(LC, c) * (LD + 1) + c_lz(LD, d);
                const double g = Gam[t][c * ND + d];
                const double gz = g * I[2][iz], gy = g * I[1][iy];
                Wx[0][ix] += gz * I[1][iy];
                Wx[1][iy] += gz * I[0][ix];
                Wx[2][iz] += gy * I[0][ix];
              });
            });
#pragma unroll
            for (int x = 0; x < 3; ++x) {
              double ap = 0, am = 0, bp = 0, bm = 0, cp = 0, cm = 0;
              const double* Ta = T + row[x];
              // rows ia - 1 and ib - 1 exist only for positive exponents (their factor is 0 otherwise)
              const double* Tm = Ta - (ea[t][x] > 0 ? TB * TR : 0);
              const double* Bm = Ta - (eb[t][x] > 0 ? TR : 0);
#pragma unroll
              for (int i = 0; i < N2; ++i) {
                const double w = Wx[x][i];
                ap += w * Ta[TB * TR + i];
                am += w * Tm[i];
                bp += w * Ta[TR + i];
                bm += w * Bm[i];
                cp += w * Ta[i + LD + 1];
                if (i >= LD + 1) cm += (double)(i / (LD + 1)) * w * I[x][i - (LD + 1)];
              }
              f0[x] += a2 * ap - (double)ea[t][x] * am;
              f1[x] += b2 * bp - (double)eb[t][x] * bm;
              f2[x] += c2x * cp - cm;
            }
          }
        }
      }
      if (vrr_lane) {
        pb += PB;
        while (pb >= NP && pk < Q.nprim) { pb -= NP; ++pk; }
      }
    }
    n_prim += (unsigned)np;
    // ---- sums over the quartet's lanes; the bra centres stay in registers
    double deg = 1.0;
    if (P.sa == P.sb) deg *= 0.5;
    if (Q.sa == Q.sb) deg *= 0.5;
    if (ip == jq) deg *= 0.5;
    if (skip) deg = 0.0;
    const int at2 = prm.shell_atom[Q.sa], at3 = prm.shell_atom[Q.sb];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const double u0 = skip ? 0.0 : deg * f0[x], u1 = skip ? 0.0 : deg * f1[x];
      double u2 = skip ? 0.0 : deg * f2[x], ud = -(u0 + u1 + u2);
      fA[x] += u0;
      fB[x] += u1;
      // sums into the group's first lane
      if constexpr ((W & (W - 1)) == 0) {
#pragma unroll
        for (int o = 1; o < W; o <<= 1) {
          u2 += __shfl_xor(u2, o);
          ud += __shfl_xor(ud, o);
        }
      } else {
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) {
          const double v2 = __shfl_down(u2, o), vd = __shfl_down(ud, o);
          u2 += l + o < W ? v2 : 0.0;
          ud += l + o < W ? vd : 0.0;
        }
      }
      if (l == 0 && !skip) {
        atomicAdd(&s_de[3 * at2 + x], u2);
        atomicAdd(&s_de[3 * at3 + x], ud);
      }
    }
  }
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    double u = fA[x], v = fB[x];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      u += __shfl_xor(u, o);
      v += __shfl_xor(v, o);
    }
    if (lane == 0) {
      atomicAdd(&s_de[3 * at0 + x], u);
      atomicAdd(&s_de[3 * at1 + x], v);
    }
  }
  unsigned long long* ctr = prm.counters + 8 * (int)((long long)blockIdx.x & (OQPH_CTR_SLOTS - 1));
  {
    unsigned v[3] = {n_comp, n_skip, n_prim};
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) v[i] += __shfl_xor(v[i], o);
    if (lane == 0) {
      if (v[0]) atomicAdd(ctr + 0, (unsigned long long)v[0]);
      if (v[1]) atomicAdd(ctr + 1, (unsigned long long)v[1]);
      if (v[2]) {
        atomicAdd(ctr + 3, (unsigned long long)v[2] * (unsigned long long)flops_grad_prim_rt(LA, LB, LC, LD));
        atomicAdd(ctr + 4, (unsigned long long)v[2]);
      }
    }
  }
  __syncthreads();
  for (int i = lane; i < 3 * prm.natm; i += 64)
    if (s_de[i] != 0.0) unsafeAtomicAdd(prm.de + (size_t)(blockIdx.x & (OQPH_DE_SLOTS - 1)) * 3 * prm.natm + i, s_de[i]);
}

}  // namespace oqph
