// jkc_device.h -- cooperative J/K kernel of the larger quartet classes.
//
// One wavefront (one block) takes the kets of one bra segment and evaluates
// 64 / W quartets at a time, W = 16, 32 or 64 lanes on each, with the class
// known at compile time.  The lanes of a quartet change roles from phase to
// phase, and every phase keeps its working row in registers:
//   1. lane = (primitive quartet, root, axis): the 2D integrals into LDS;
//   2. lane = e: the row (e0|f0), f = 0.., contracted over primitives and roots;
//   3. lane = f: the bra transfer and AO transform of column f;
//   4. lane = (a, b): the ket transfer and AO transform of row ab, its J_ab
//      and its share of J_cd and of the four exchange blocks;
//   5. lane = an output element: sums of the shares, one atomic each.
//
// What bounds it and why this split.  The per-lane templates (k_jkb, k_jk:
// one lane = one quartet) need the whole (e0|f0) set and AO block in one
// lane's registers: above about 80 components they spill 0.4-2.4 KB per lane
// and issue VALU 5-10 % of the time, and their straight-line code (hundreds
// of KB) leaves a launch of few quartets waiting for instruction fetches.  The
// run-time-class kernel (k_jkh) has no spills, but 90 % of its instructions
// are index arithmetic, and a quartet of 81 outputs fills 64 lanes badly.
// Here a lane needs max(NF, NE + NA NB, NF + NC ND) doubles, all indices are
// constants, and the inner products read one LDS value per one to three FMAs.
// Measured ((H2O)64/cc-pVDZ, (H2O)16/cc-pVTZ): see jkc_class() in session.hip.
#pragma once
#include "jk_device.h"

namespace oqph {

template <int LA, int LB, int LC, int LD, bool PURE>
struct JKC {
  using Dm = Dims<LA, LB, LC, LD>;
  static constexpr int NE = Dm::NE, NF = Dm::NF, NR = Dm::NROOT;
  static constexpr int OA = AO<LA, PURE>::N, OB = AO<LB, PURE>::N, OC = AO<LC, PURE>::N, OD = AO<LD, PURE>::N;
  static constexpr int OAB = OA * OB, OCD = OC * OD;
  // lanes per quartet, quartets per wavefront
  static constexpr int W = NE <= 16 ? 16 : (NE <= 32 ? 32 : 64);
  static constexpr int NQ = 64 / W;
  // primitive quartets per batch of phase 1 (3 NR lanes each)
  static constexpr int PB = W / (3 * NR) > 0 ? W / (3 * NR) : 1;
  static constexpr int GA = (Dm::LAB + 1) * (Dm::LCD + 1);  // 2D integrals per root and axis
  static constexpr int NFp = NF | 1, CDp = OCD | 1;         // odd row strides: conflict-free column reads
  static constexpr int KS = 2 * (OC + OD), KSp = KS | 1;    // exchange shares per (a, b)
  static constexpr int mx(int a, int b) { return a > b ? a : b; }
  // LDS of one quartet (doubles): A = 2D integrals, then Y[ab][f], then the
  // exchange shares; B = (e0|f0), then the J_cd shares; D = density blocks
  static constexpr int SA = mx(mx(PB * NR * 3 * GA, OAB * NFp), OAB * KSp);
  static constexpr int SB = mx(NE * NFp, OAB * CDp);
  static constexpr int SD = OCD + OA * OC + OA * OD + OB * OC + OB * OD;
  static constexpr int SLOT = SA + SB + SD;
  static constexpr int ET = (NE + W - 1) / W, FT = (NF + W - 1) / W, AT = (OAB + W - 1) / W;
  // bra primitive pairs kept in LDS (the rest of a longer list is read from memory)
  static constexpr int MAXBRA = 32;
  static constexpr int lds = 8 * NQ * SLOT + (int)sizeof(PrimJK) * MAXBRA;
  // wavefronts per SIMD the register allocation aims at: what the LDS allows, at most 4
  static constexpr int waves = 160 * 1024 / lds / 4 < 1 ? 1 : (160 * 1024 / lds / 4 > 4 ? 4 : 160 * 1024 / lds / 4);
  static constexpr bool fits = lds <= 64 * 1024 && 3 * NR <= W;
};

// the same limit for both AO representations (the Cartesian one is larger)
template <int LA, int LB, int LC, int LD>
constexpr bool jkc_fits() {
  return JKC<LA, LB, LC, LD, true>::fits && JKC<LA, LB, LC, LD, false>::fits;
}

template <int LA, int LB, int LC, int LD, bool PURE, bool TWO>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(JKC<LA, LB, LC, LD, PURE>::waves)))
void k_jkc(JKParams prm, WaveWork ww) {
  using J = JKC<LA, LB, LC, LD, PURE>;
  using Dm = Dims<LA, LB, LC, LD>;
  constexpr int NE = J::NE, NF = J::NF, NR = J::NR, OA = J::OA, OB = J::OB, OC = J::OC, OD = J::OD;
  constexpr int OAB = J::OAB, OCD = J::OCD, W = J::W, NQ = J::NQ, PB = J::PB, GA = J::GA, NFp = J::NFp,
                CDp = J::CDp, KSp = J::KSp, ET = J::ET, FT = J::FT, AT = J::AT;
  constexpr int LAB = Dm::LAB, LCD = Dm::LCD;
  __shared__ double s_slot[NQ][J::SLOT];
  __shared__ PrimJK s_bra[J::MAXBRA];
  const int lane = (int)threadIdx.x, l = lane & (W - 1), q = lane / W;
  // ---- the block's kets: [sub kpb, (sub + 1) kpb) of one 64-ket chunk of one segment
  const int kpb = ww.kpb > 0 ? ww.kpb : 64, per = 64 / kpb;
  const long long block = (long long)blockIdx.y * gridDim.x + blockIdx.x, wave = block / per;
  const int sub = (int)(block - wave * per);
  if (wave >= ww.nwaves) return;  // block-uniform
  int lo = 0, hi = ww.nseg;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (ww.choff[mid] <= wave) lo = mid; else hi = mid;
  }
  const int seg = __builtin_amdgcn_readfirstlane(lo);
  const int k = (int)(wave - ww.choff[seg]) * 64 + sub * kpb + lane;
  const bool active = lane < kpb && k < ww.seg_n[seg];
  const int ip = __builtin_amdgcn_readfirstlane(ww.seg_bra[seg]);
  const ShellPair P = prm.pairs[ip];
  int iq = 0;
  bool skip = true, mine = true;
  if (active) {
    iq = ww.kofs + ww.seg_k0[seg] + k;  // the class lists are consecutive device pairs
    const ShellPair Q = prm.pairs[iq];
    // OpenQP screening (int2.F90:763-800)
    const bool p_first = (P.si > Q.si) || (P.si == Q.si && P.sj >= Q.sj);
    if (prm.own) mine = prm.own[p_first ? ip : iq] != 0;
    const double qbra = p_first ? P.Q : Q.Q;
    const int n = prm.nsh;
    const double* ds = prm.dsh;
    double dm = 4.0 * fmax(prm.dpm[ip], prm.dpm[iq]);
    dm = fmax(dm, fmax(ds[P.sj * n + Q.sj], ds[P.sj * n + Q.si]));
    dm = fmax(dm, fmax(ds[P.si * n + Q.sj], ds[P.si * n + Q.si]));
    skip = !mine || (qbra * prm.maxden < prm.cutoff) || (P.Q * Q.Q * dm < prm.cutoff);
  }
  unsigned long long* ctr = prm.counters + 8 * (int)(wave & (OQPH_CTR_SLOTS - 1));
  count_wave(ctr + 1, active && mine && skip);
  count_wave(ctr + 0, !skip);
  unsigned long long todo = __ballot(!skip);
  if (todo == 0ull) return;  // block-uniform
  const double cut = prm.cutoff, qcut = 1.0e-4 * cut, qcut2 = qcut * qcut, imu2 = prm.inv_mu2;
  // ---- bra primitive pairs that pass |K| >= qcut, compacted into LDS
  int nbra = 0;
  {
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int i0 = 0; i0 < P.nprim; i0 += 64) {
      const int i = i0 + lane;
      PrimJK r{};
      bool ok = false;
      if (i < P.nprim) {
        r = prm.prims[P.prim0 + i];
        ok = !(fabs(r.Kg) < qcut);
      }
      const unsigned long long m = __ballot(ok);
      const int at = nbra + __popcll(m & below);
      if (ok && at < J::MAXBRA) s_bra[at] = r;
      nbra += __popcll(m);
    }
  }
  // longer lists stay in memory (and keep the dropped records, which fail the quartet screen)
  const bool bra_lds = nbra <= J::MAXBRA;
  if (!bra_lds) nbra = P.nprim;
  const int oa = P.ao_a, ob = P.ao_b;
  double* F = prm.F;
  double Dab[AT], jab[AT];
#pragma unroll
  for (int t = 0; t < AT; ++t) {
    const int ab = l + W * t;
    jab[t] = 0.0;
    Dab[t] = ab < OAB ? prm.D[tri_idx(oa + ab / OB, ob + ab % OB)] : 0.0;
  }
  // this lane's (e0| component in phase 2
  int ox[ET], oy[ET], oz[ET];
#pragma unroll
  for (int t = 0; t < ET; ++t) {
    int c = l + W * t, L = LA;
    if (c >= NE) c = 0;
    while (c >= ncart(L)) { c -= ncart(L); ++L; }
    ox[t] = c_lx(L, c) * (LCD + 1);
    oy[t] = GA + c_ly(L, c) * (LCD + 1);
    oz[t] = 2 * GA + c_lz(L, c) * (LCD + 1);
  }
  // this lane's (primitive quartet of a batch, root, axis) in phase 1
  const int pi = l / (3 * NR), r1 = (l - pi * 3 * NR) / 3, d1 = l - pi * 3 * NR - 3 * r1;
  const bool vrr_lane = l < PB * 3 * NR;
  double* A = s_slot[q];
  double* Bf = A + J::SA;
  double* sD = Bf + J::SB;
  double *Dcd = sD, *Dac = sD + OCD, *Dad = Dac + OA * OC, *Dbc = Dad + OA * OD, *Dbd = Dbc + OB * OC;
  const double* tabN = prm.rys + RYS_OFF[NR];
  double ABv[3], ACl[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) ABv[d] = P.A[d] - P.B[d];
  unsigned n_prim = 0, n_valid = 0;

  while (todo) {
    // ---- the next NQ surviving kets, one per lane group
    int from = 0;
    bool on = false;
#pragma unroll
    for (int s = 0; s < NQ; ++s) {
      const bool have = todo != 0ull;
      const int b = have ? __ffsll((long long)todo) - 1 : 0;
      if (q == s) {
        from = b;
        on = have;
      }
      if (have) todo &= todo - 1ull;
    }
    const int jq = __shfl(iq, from);
    const ShellPair Q = prm.pairs[jq];
    const int oc = Q.ao_a, od = Q.ao_b;
    __syncthreads();  // the previous quartets' readers of LDS are done
    // density blocks of the quartet (phase 4 reads them)
    auto load_d = [&](const double* __restrict__ Dp) {
      for (int t = l; t < OA * OC; t += W) Dac[t] = Dp[tri_idx(oa + t / OC, oc + t % OC)];
      for (int t = l; t < OA * OD; t += W) Dad[t] = Dp[tri_idx(oa + t / OD, od + t % OD)];
      for (int t = l; t < OB * OC; t += W) Dbc[t] = Dp[tri_idx(ob + t / OC, oc + t % OC)];
      for (int t = l; t < OB * OD; t += W) Dbd[t] = Dp[tri_idx(ob + t / OD, od + t % OD)];
    };
    const double* Dk = prm.Dk + ww.jbase + (long long)(jq - ww.kofs) * OCD;
    for (int t = l; t < OCD; t += W) Dcd[t] = Dk[t];
    load_d(prm.D);
#pragma unroll
    for (int d = 0; d < 3; ++d) ACl[d] = P.A[d] - Q.A[d];
    double acc[ET][NF];
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
      for (int f = 0; f < NF; ++f) acc[t][f] = 0.0;
    // ---- phases 1 and 2 over batches of PB primitive quartets
    const int T = on ? nbra * Q.nprim : 0;
    int Tmax = T;
#pragma unroll
    for (int o = W; o < 64; o <<= 1) Tmax = max(Tmax, __shfl_xor(Tmax, o));
    Tmax = __builtin_amdgcn_readfirstlane(Tmax);
    int pb = 0, pk = 0, np = 0;  // this lane's bra / ket primitive pair
    pb = pi;
    while (pb >= nbra && pk < Q.nprim) { pb -= nbra; ++pk; }
    for (int t0 = 0; t0 < Tmax; t0 += PB) {
      bool pass = false;
      if (vrr_lane) {
        const bool in = t0 + pi < T;
        const int kb = in ? pb : 0, kk = in ? pk : 0;
        const PrimJK pp = bra_lds ? s_bra[kb] : prm.prims[P.prim0 + kb];
        const PrimJK qq = prm.prims[Q.prim0 + kk];
        const double zeta = pp.g, eta = qq.g, ze = zeta + eta + zeta * eta * imu2;
        const double fqz = pp.Kg * qq.Kg;
        pass = in && !(fabs(pp.Kg) < qcut) && !(fabs(qq.Kg) < qcut) && !(fqz * fqz < qcut2 * ze);
        np += (pass && r1 == 0 && d1 == 0) ? 1 : 0;
        const double sq = rsq64(ze), ize = sq * sq;
        const double PQ0 = ACl[0] + pp.X[0] - qq.X[0], PQ1 = ACl[1] + pp.X[1] - qq.X[1],
                     PQ2 = ACl[2] + pp.X[2] - qq.X[2];
        const double Tb = zeta * eta * ize * (PQ0 * PQ0 + PQ1 * PQ1 + PQ2 * PQ2);
        double t2, wr;
        rys_root_one<NR, double>(Tb, tabN, nullptr, r1, t2, wr);
        const double rz = eta * ize, re = zeta * ize;
        const double B00 = 0.5 * ize * t2, B10 = pp.h - pp.h * rz * t2, B01 = qq.h - qq.h * re * t2;
        const double PQ = d1 == 0 ? PQ0 : d1 == 1 ? PQ1 : PQ2;
        const double C00 = (d1 == 0 ? pp.X[0] : d1 == 1 ? pp.X[1] : pp.X[2]) - rz * t2 * PQ;
        const double D00 = (d1 == 0 ? qq.X[0] : d1 == 1 ? qq.X[1] : qq.X[2]) + re * t2 * PQ;
        double* g = A + ((pi * NR + r1) * 3 + d1) * GA;
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
        pb += PB;
        while (pb >= nbra && pk < Q.nprim) { pb -= nbra; ++pk; }
      }
      __syncthreads();
      if (__ballot(pass) != 0ull) {  // wave-uniform
#pragma unroll 1
        for (int pr = 0; pr < PB * NR; ++pr) {
          const double* g = A + pr * 3 * GA;
#pragma unroll
          for (int t = 0; t < ET; ++t) {
            double X[LCD + 1], Y[LCD + 1], Z[LCD + 1];
#pragma unroll
            for (int x = 0; x <= LCD; ++x) {
              X[x] = g[ox[t] + x];
              Y[x] = g[oy[t] + x];
              Z[x] = g[oz[t] + x];
            }
            double YZ[LCD + 1][LCD + 1];
#pragma unroll
            for (int y = 0; y <= LCD; ++y)
#pragma unroll
              for (int z = 0; z + y <= LCD; ++z) YZ[y][z] = Y[y] * Z[z];
            sfor<NF>([&](auto Fi) {
              constexpr int f = OQPH_CI(Fi);
              constexpr int Lf = range_level<LC>(f), cf = range_local<LC>(f);
              acc[t][f] += X[c_lx(Lf, cf)] * YZ[c_ly(Lf, cf)][c_lz(Lf, cf)];
            });
          }
        }
      }
      __syncthreads();
    }
    n_prim += (unsigned)np;
#pragma unroll
    for (int o = 1; o < W; o <<= 1) np += __shfl_xor(np, o);  // the quartet's surviving primitive quartets
    const bool valid = on && np > 0;
    n_valid += (valid && l == 0) ? 1 : 0;
    if (__ballot(valid) == 0ull) continue;  // block-uniform
    // ---- (e0|f0) to LDS; phase 3: bra transfer and AO transform per column f
#pragma unroll
    for (int t = 0; t < ET; ++t) {
      const int e = l + W * t;
      if (e < NE)
#pragma unroll
        for (int f = 0; f < NF; ++f) Bf[e * NFp + f] = acc[t][f];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < FT; ++t) {
      const int f = l + W * t;
      if (f < NF) {
        double ec[NE][1], Y[Dm::NA * Dm::NB][1];
#pragma unroll
        for (int e = 0; e < NE; ++e) ec[e][0] = Bf[e * NFp + f];
        hrr_bra<LA, LB, 1, double>(ec, ABv, Y);
        double* y = &Y[0][0];
        if constexpr (LA >= 2) xform_inplace<LA, PURE, 1, Dm::NB, double>(prm.xform, y);
        if constexpr (LB >= 2) xform_inplace<LB, PURE, OA, 1, double>(prm.xform, y);
#pragma unroll
        for (int ab = 0; ab < OAB; ++ab) A[ab * NFp + f] = y[ab];
      }
    }
    __syncthreads();
    // ---- phase 4: ket transfer and AO transform per row ab, element cutoff
    double deg = 1.0;
    if (P.sa == P.sb) deg *= 0.5;
    if (Q.sa == Q.sb) deg *= 0.5;
    if (ip == jq) deg *= 0.5;
    const double cj = 2.0 * deg * prm.sc, ck = -0.5 * deg * prm.se;
    double V[AT][Dm::NC * Dm::ND];
    {
      double CDv[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) CDv[d] = Q.A[d] - Q.B[d];
#pragma unroll
      for (int t = 0; t < AT; ++t) {
        const int ab = l + W * t;
        double Yr[1][NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) Yr[0][f] = ab < OAB ? A[ab * NFp + f] : 0.0;
        hrr_ket<LC, LD, 1, double>(Yr, CDv, V[t]);
        if constexpr (LC >= 2) xform_inplace<LC, PURE, 1, Dm::ND, double>(prm.xform, V[t]);
        if constexpr (LD >= 2) xform_inplace<LD, PURE, OC, 1, double>(prm.xform, V[t]);
        double jt = 0.0;
#pragma unroll
        for (int cd = 0; cd < OCD; ++cd) {
          double v = V[t][cd];
          if (!valid || ab >= OAB || fabs(v) < cut) v = 0.0;  // OpenQP element cutoff on the AO value
          V[t][cd] = v;
          jt += v * Dcd[cd];
          if (ab < OAB) Bf[ab * CDp + cd] = v * Dab[t];
        }
        jab[t] += cj * jt;
      }
    }
    if constexpr (!TWO)
      if (prm.T) {  // dense response pass: the integrals themselves
        const TSlots ts{P.sa == P.sb, Q.sa == Q.sb, ip == jq};
#pragma unroll
        for (int t = 0; t < AT; ++t) {
          const int ab = l + W * t;
          if (ab < OAB)
#pragma unroll
            for (int cd = 0; cd < OCD; ++cd) ts.put(prm, oa + ab / OB, ob + ab % OB, oc + cd / OD, od + cd % OD, V[t][cd]);
        }
        continue;
      }
    __syncthreads();
    // shares of the exchange blocks of row (a, b): K_ac from b, K_ad from b,
    // K_bc from a, K_bd from a; then their sums, one atomic per element
    auto exchange = [&](double* Fk) {
#pragma unroll
      for (int t = 0; t < AT; ++t) {
        const int ab = l + W * t, a = ab / OB, b = ab - a * OB;
        if (ab < OAB) {
          double* kp = A + ab * KSp;
#pragma unroll
          for (int c = 0; c < OC; ++c) {
            double s1 = 0.0, s2 = 0.0;
#pragma unroll
            for (int d = 0; d < OD; ++d) {
              s1 += V[t][c * OD + d] * Dbd[b * OD + d];
              s2 += V[t][c * OD + d] * Dad[a * OD + d];
            }
            kp[c] = s1;
            kp[OC + OD + c] = s2;
          }
#pragma unroll
          for (int d = 0; d < OD; ++d) {
            double s1 = 0.0, s2 = 0.0;
#pragma unroll
            for (int c = 0; c < OC; ++c) {
              s1 += V[t][c * OD + d] * Dbc[b * OC + c];
              s2 += V[t][c * OD + d] * Dac[a * OC + c];
            }
            kp[OC + d] = s1;
            kp[2 * OC + OD + d] = s2;
          }
        }
      }
      __syncthreads();
      if (!valid) return;
      auto put = [&](int x, int y, double v) {
        v *= ck * (x == y ? 2.0 : 1.0);
        if (v != 0.0) fatomic(Fk + tri_idx(x, y), v);
      };
      for (int t = l; t < OA * (OC + OD); t += W) {  // rows a: columns c, then d
        const int a = t / (OC + OD), c = t - a * (OC + OD);
        double s = 0.0;
#pragma unroll
        for (int b = 0; b < OB; ++b) s += A[(a * OB + b) * KSp + c];
        put(oa + a, c < OC ? oc + c : od + c - OC, s);
      }
      for (int t = l; t < OB * (OC + OD); t += W) {  // rows b
        const int b = t / (OC + OD), c = t - b * (OC + OD);
        double s = 0.0;
#pragma unroll
        for (int a = 0; a < OA; ++a) s += A[(a * OB + b) * KSp + OC + OD + c];
        put(ob + b, c < OC ? oc + c : od + c - OC, s);
      }
    };
    exchange(F);
    // ---- phase 5: J_cd into the ket's block of the ket-side Coulomb buffer
    if (valid) {
      double* Jd = prm.Jk + ww.jbase + (long long)(jq - ww.kofs) * OCD;
      for (int cd = l; cd < OCD; cd += W) {
        double s = 0.0;
#pragma unroll
        for (int ab = 0; ab < OAB; ++ab) s += Bf[ab * CDp + cd];
        s *= cj;
        if (s != 0.0) fatomic(Jd + cd, s);
      }
    }
    if constexpr (TWO) {  // the open-shell pass: D2's exchange blocks into F2
      __syncthreads();
      load_d(prm.D2);
      __syncthreads();
      exchange(prm.F2);
    }
  }
  // ---- J_ab over the wavefront's kets, statistics
#pragma unroll
  for (int t = 0; t < AT; ++t) {
    if (prm.T) break;
    double v = jab[t];
#pragma unroll
    for (int o = W; o < 64; o <<= 1) v += __shfl_xor(v, o);
    const int ab = l + W * t;
    if (q == 0 && ab < OAB && v != 0.0) {
      const int x = oa + ab / OB, y = ob + ab % OB;
      fatomic(F + tri_idx(x, y), v * (x == y ? 2.0 : 1.0));
    }
  }
  sum_wave(ctr + 3, (unsigned long long)n_prim * flops_prim<LA, LB, LC, LD>() +
                        (unsigned long long)n_valid * (TWO ? 24ull : prm.T ? 20ull * prm.gnd : 12ull) * (OAB * OCD));
  sum_wave(ctr + 4, (unsigned long long)n_prim);
}

}  // namespace oqph
