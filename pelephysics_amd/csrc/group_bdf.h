// Batched adaptive BDF with a group of G lanes per cell (64 / G cells per
// wavefront, G = 8, 16, 32 or 64).
//
// * lane g of a group holds equations i = e*G + g for slots e < EPL =
//   ceil(NEQ / G): its entries of the BDF difference array, the iterate, the
//   error weights and rows i of the inverted Newton matrix, in registers as far
//   as 256 go (four vectors in LDS; spilled with an FP32 inverse: drm19 74 at 32
//   lanes and 132 at 16, LiDryer 64 at 8, LuEthylene_qss 194, dodecane_lu 287,
//   heptane_lu_88sk 783, which has two rows of 89 in every lane);
// * the mechanism's packed tables (tab/<name>.h, struct Packed) are copied to
//   LDS once per block; the four waves of a block share them and never wait
//   for each other afterwards;
// * right-hand side: each lane evaluates the NASA7 polynomials and
//   exponentials of its species, concentrations and exponentials go to a small
//   per-group LDS area, reactions j = g, g + G, ... are spread over the lanes
//   and write their net rates of progress to LDS, the chunks of 8 terms that
//   the species' stoichiometric rows are cut into are spread over the lanes
//   again, and each lane adds up its species' chunks; mixture sums are group
//   reductions;
// * Jacobian (about one per cell and call): all 64 lanes of the wave work on one
//   group's cell at a time, or each group on its own (group_layout.h),
//   accumulating with FP64 atomics into an n x n area (LDS when it fits, else the
//   device workspace), then store the group's rows (molecular-weight scaling of
//   ReactorBDF.cpp:67-82) in LU_T in the workspace for the Newton-matrix
//   refreshes;
// * Newton matrix: inverted in LU_T by row-per-lane Gauss-Jordan exchange
//   steps with partial pivoting (the pivot row through LDS, rows never move,
//   the columns rotate through the registers so that the step loop is not
//   unrolled), so that each Newton iteration's solve is one dot product per
//   row: no sequential triangular sweeps.
//
// What bounds it: calls that fill the chip, the FP64 vector issue of two waves
// per SIMD (drm19 64^3 cells at 16 lanes: a vector instruction every 6.3 cycles of
// a SIMD, of which it takes 4; a wave waits 44% of its cycles, for LDS, spills and
// dependent results); others, the latency of the longest cells' trips (one
// right-hand side and one Newton iteration for every group of the wave).  Measured
// (one MI355X, box or 1-D call of 1e-5 s at rtol 1e-10, state restored before each
// call), against one cell per lane: drm19 64^3 cells 222 -> 70 ms, 2898 cells 95 ->
// 5.9 ms; dodecane_lu 10000 cells 1558 -> 13.6 ms; heptane_lu_88sk 2048 cells, 1e-6 s
// at rtol 1e-8, 1169 -> 11.0 ms; LuEthylene_qss 4096 cells 198 -> 4.2 ms.
//
// Every group reduction returns the bitwise-identical value in all lanes of
// the group (pairs are always added in commuted order on both partners), so
// the integrator's control flow is uniform within a group.  Different groups
// of a wave follow their own cells; every trip of the
// persistent loop evaluates one right-hand side for every group that is not
// waiting for a factorisation, and the groups' LU requests are served together
// once enough of them wait.  A cell's arithmetic does not depend on which
// groups share its wave, so results do not depend on the queue's order; it
// depends on the group's width, which a call's number of cells can choose.
//
// The step / order / Newton logic is that of adaptive_cell (reactors.h), the
// NDF family of SciPy's BDF integrator; every loop over a cell's work is
// bounded (queue length, RHS budget, the 200-iteration temperature inversion).
// The algorithm follows SciPy's scipy/integrate/_ivp/bdf.py (BSD-3-Clause,
// Copyright (c) 2001-2002 Enthought, Inc. 2003-2024, SciPy Developers; the
// notice and license are in THIRD_PARTY_NOTICES.md at the repository root).
#pragma once
#include "chem_table.h"
#include "reactors.h"
#include "wave.h"
#include "pack.h"
#include "group_layout.h"

namespace ppc {

// Cell input/output of the 1-D (YCOrder) form.
struct IO1D {
  double* y;
  const double* ysrc;
  double* rX;
  const double* rXsrc;
};

// phases of a cell's integration
enum : int { PH_F0 = 0, PH_F1 = 1, PH_NEWTON = 2 };

// ------------------------------------------------ group lane primitives --
template <int G>
struct Grp {
  static_assert(G == 8 || G == 16 || G == 32 || G == 64, "groups of 8, 16, 32 or 64 lanes");
  PPC_DI static int lane() { return (int)__lane_id() & (G - 1); }
  // v of the partner row(s): the two results hold, in every lane, the value of
  // this lane's 16-lane row (32-lane half) pair, the same pair on both sides
  template <bool HALF>
  PPC_DI static void pair32(unsigned v, unsigned& a, unsigned& b) {
    if constexpr (HALF) {
      const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
      a = r[0];
      b = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
      a = r[0];
      b = r[1];
    }
  }
  template <bool HALF>
  PPC_DI static void pair(double v, double& a, double& b) {
    unsigned al, bl, ah, bh;
    pair32<HALF>(wave::lo32(v), al, bl);
    pair32<HALF>(wave::hi32(v), ah, bh);
    a = wave::from32(ah, al);
    b = wave::from32(bh, bl);
  }
  template <bool HALF>
  PPC_DI static void pair(float v, float& a, float& b) {
    unsigned x, y;
    pair32<HALF>(__float_as_uint(v), x, y);
    a = __uint_as_float(x);
    b = __uint_as_float(y);
  }
  // all-reduce sum / max over the group, bitwise identical in every lane
  template <typename T>
  PPC_DI static T sum(T v) {
    v += wave::dpp<wave::DPP_XOR1>(v);
    v += wave::dpp<wave::DPP_XOR2>(v);
    v += wave::dpp<wave::DPP_HALF_MIRROR>(v);
    if (G >= 16) v += wave::dpp<wave::DPP_MIRROR>(v);
    T a, b;
    if (G >= 32) {
      pair<false>(v, a, b);
      v = a + b;
    }
    if (G >= 64) {
      pair<true>(v, a, b);
      v = a + b;
    }
    return v;
  }
  template <typename T>
  PPC_DI static T max(T v) {
    v = fmax(v, wave::dpp<wave::DPP_XOR1>(v));
    v = fmax(v, wave::dpp<wave::DPP_XOR2>(v));
    v = fmax(v, wave::dpp<wave::DPP_HALF_MIRROR>(v));
    if (G >= 16) v = fmax(v, wave::dpp<wave::DPP_MIRROR>(v));
    T a, b;
    if (G >= 32) {
      pair<false>(v, a, b);
      v = fmax(a, b);
    }
    if (G >= 64) {
      pair<true>(v, a, b);
      v = fmax(a, b);
    }
    return v;
  }
  // this group's bits of a ballot
  PPC_DI static unsigned long long bits(unsigned long long b) {
    if constexpr (G == 64) {
      return b;
    } else {
      return (b >> (__lane_id() & ~(unsigned)(G - 1))) & ((1ULL << G) - 1);
    }
  }
  PPC_DI static bool any(bool p) { return bits(__ballot(p)) != 0; }
  // value of lane src (0 <= src < G) of the group
  template <typename T>
  PPC_DI static T bcast(T v, int src) {
    return __shfl(v, src, G);
  }
};

// Orders this lane's LDS accesses around an exchange with other lanes of its
// wavefront: a wave's LDS operations execute in order, so only the compiler
// has to be held back.
PPC_DI void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Loads and stores of the Jacobian accumulator in the workspace, which the
// wave's lanes update with device-scope atomics.
PPC_DI double ws_load(const double* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
PPC_DI void ws_store(double* p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// The block's copy of a mechanism's packed tables.
template <class T>
PPC_DI typename T::Packed& lds_pack() {
  __shared__ typename T::Packed p;
  return p;
}

// Fills it, by every thread of the block.
template <class T>
PPC_DI const typename T::Packed& load_pack() {
  using PK = typename T::Packed;
  PK& pk = lds_pack<T>();
  const int4* from = reinterpret_cast<const int4*>(&T::pack());
  int4* to = reinterpret_cast<int4*>(&pk);
  static_assert(sizeof(PK) % 16 == 0, "packed tables in 16-byte words");
  for (int i = threadIdx.x; i < (int)(sizeof(PK) / 16); i += 64 * GROUP_WAVES) to[i] = from[i];
  __syncthreads();
  return pk;
}

// The table accessors TabMech::jac_reaction reads, in packed reaction order.
template <class T>
struct PackTab : T {
  PPC_DI static int sp(int k) { return k == T::NX ? -1 : k; }
  PPC_DI static double rxA_(int j) { return lds_pack<T>().rx[j].A; }
  PPC_DI static double rxB_(int j) { return lds_pack<T>().rx[j].b; }
  PPC_DI static double rxE_(int j) { return lds_pack<T>().rx[j].E; }
  PPC_DI static int rxR_(int i) { return sp(lds_pack<T>().rx[i / 3].r[i % 3]); }
  PPC_DI static int rxP_(int i) { return sp(lds_pack<T>().rx[i / 3].p[i % 3]); }
  PPC_DI static int rxDelta_(int j) { return lds_pack<T>().rx[j].delta; }
  PPC_DI static int rxRev_(int j) { return lds_pack<T>().rx[j].flags & 1; }
  PPC_DI static int rxFwdOff_(int j) { return lds_pack<T>().rx[j].flags & 2; }
  PPC_DI static int rxNet_(int i) {
    return T::rxNet_(T::MAXNET * (int)lds_pack<T>().perm[i / T::MAXNET] + i % T::MAXNET);
  }
  PPC_DI static double rxNu_(int i) {
    return T::rxNu_(T::MAXNET * (int)lds_pack<T>().perm[i / T::MAXNET] + i % T::MAXNET);
  }
  PPC_DI static int rxEff0_(int j) { return lds_pack<T>().eff[j - T::N_EL].e0; }
  PPC_DI static int rxEffN_(int j) { return lds_pack<T>().eff[j - T::N_EL].n; }
  PPC_DI static int effK_(int i) { return lds_pack<T>().effK[i]; }
  PPC_DI static double effV_(int i) { return lds_pack<T>().effV[i]; }
  PPC_DI static double foA_(int f) { return lds_pack<T>().fo[f].A; }
  PPC_DI static double foB_(int f) { return lds_pack<T>().fo[f].b; }
  PPC_DI static double foE_(int f) { return lds_pack<T>().fo[f].E; }
  PPC_DI static double troe_(int i) {
    const auto& f = lds_pack<T>().fo[i / 4];
    return i % 4 == 0 ? f.tA : (i % 4 == 1 ? f.t3 : (i % 4 == 2 ? f.t1 : f.t2));
  }
  PPC_DI static int troeT2_(int f) { return lds_pack<T>().fo[f].has2 != 0.0; }
};

// ------------------------------------------- the mechanism on a group --
typedef __attribute__((address_space(3))) double lds_double;
template <class T, int G, int WD>
__device__ void group_qss_jacobian(lds_double* area, double* Jws, const bool eform);

template <class T, int G>
struct GroupChem {
  using TM = TabMech<PackTab<T>>;
  using PK = typename T::Packed;
  using Gr = Grp<G>;
  using L = GroupLayout<T, G>;
  static constexpr int NS = L::NS, NR = L::NR, n = L::n, NX = L::NX, NCH = L::NCH, NQ = L::NQ, NROW = L::NROW;
  static constexpr int NG = L::NG, EPL = L::EPL, SPL = L::SPL, SPX = L::SPX, NP = L::NP, NRATE = L::NRATE;
  static constexpr int TL = NS % G, TS = NS / G;  // lane and slot of the temperature equation
  static constexpr int S_CA = L::S_CA, S_B = L::S_B, S_Q = L::S_Q, AREA = L::AREA, WAREA = L::WAREA;
  static constexpr bool JLDS = L::JLDS, JOWN = L::JOWN;
  static constexpr int J_AT = L::J_AT, JSQ = L::JSQ, JSTRIDE = L::JSTRIDE, JSPACE = L::JSPACE;
  static constexpr int cmax(int a, int b) { return L::cmax(a, b); }

  PPC_DI static void coefs(const PK& pk, const int k, const double Tv, double (&a)[7], double& imw) {
    const double* s = pk.sp[k].lo;
    const double* c = Tv < s[7] ? s : s + 8;
#pragma unroll
    for (int i = 0; i < 7; ++i) a[i] = c[i];
    imw = s[15];
  }

  // sum y h/RT imw and sum y cp/R imw (or e, cv) of the group's cell at Tv
  PPC_DI static void heat(const PK& pk, const int g, const bool eform, const double (&y)[EPL], const double Tv,
                          double& hs, double& cs, double (&hk)[SPL]) {
    const double invT = 1.0 / Tv;
    double h = 0.0, c = 0.0;
#pragma unroll
    for (int e = 0; e < SPL; ++e) {
      const int k = e * G + g;
      hk[e] = 0.0;
      if (k < NS) {
        double a[7], imw;
        coefs(pk, k, Tv, a, imw);
        double hp = TM::h_poly(a, Tv, invT), cp = TM::cp_poly(a, Tv);
        if (eform) {
          hp -= 1.0;
          cp -= 1.0;
        }
        const double yw = y[e] * imw;
        h += yw * hp;
        c += yw * cp;
        hk[e] = hp;
      }
    }
    hs = Gr::sum(h);
    cs = Gr::sum(c);
  }

  // GET_T_GIVEN_HY / GET_T_GIVEN_EY (Mechanisms/drm19/mechanism.H:2789-2890)
  // of the cell's energy per volume E: Newton on T, |dT| clamped to 100 K, stop
  // at |dT| < 1e-6, at most 200 iterations, linear extrapolation outside [90,
  // 4000] K.  The integrated temperature is nearly always within 1e-6 K, so
  // the energies at the bounds are formed only when the first iteration has
  // not ended there.  Also the heat sums and species energies at the result.
  PPC_DI static double T_from_energy(const PK& pk, const int g, const bool eform, const double E,
                                     const double (&y)[EPL], double Tv, double& cs, double (&hk)[SPL]) {
    const double tmin = 90.0, tmax = 4000.0;
    // 0: at the guess; 1, 2: at the bounds; 3: Newton; 4: at the final T
    int what = 0, it = 0;
    double Tq = Tv, dt = 0.0, rinv = 0.0, hmin = 0.0, cmin = 0.0;
#pragma unroll 1
    for (;;) {
      double hs;
      heat(pk, g, eform, y, Tq, hs, cs, hk);
      if (what == 4) break;
      if (what == 0 || what == 3) {
        dt = (E - hs * (RU * Tq)) / (cs * RU);
        if (fabs(dt) < 1.0e-6 && (what == 3 || (Tv >= tmin && Tv <= tmax))) break;
        if (what == 0) {
          double rs = 0.0;
#pragma unroll
          for (int e = 0; e < SPL; ++e)
            if (e * G + g < NS) rs += y[e];
          rinv = 1.0 / Gr::sum(rs);
          what = 1;
          Tq = tmin;
          continue;
        }
      } else if (what == 1) {
        hmin = hs * (RU * tmin * rinv);
        cmin = cs * (RU * rinv);
        what = 2;
        Tq = tmax;
        continue;
      } else {
        const double hv = E * rinv, hmax = hs * (RU * tmax * rinv), cmax = cs * (RU * rinv);
        if (hv < hmin || hv > hmax) {
          Tv = hv < hmin ? tmin - (hmin - hv) / cmin : tmax - (hmax - hv) / cmax;
          what = 4;
          Tq = Tv;
          continue;
        }
        what = 3;
        if (Tv < tmin || Tv > tmax) {
          Tv = tmin + (tmax - tmin) / (hmax - hmin) * (hv - hmin);
          Tq = Tv;
          continue;
        }
      }
      Tv += dt > 100.0 ? 100.0 : (dt < -100.0 ? -100.0 : dt);
      Tq = Tv;
      // 200 iterations, or NaN (as every further iterate would be)
      if (++it == 200 || !(dt == dt)) what = 4;
    }
    return Tv;
  }

  PPC_DI static double refc_pow(const int d, const double refC, const double refCinv) {
    double r = d > 0 ? refC : (d < 0 ? refCinv : 1.0);
    const double b = r;
    for (int i = d < 0 ? -d : d; i > 1; --i) r *= b;
    return r;
  }

  // rate of progress of reaction j (packed order) of KIND (0 elementary, 1
  // three-body, 2 Troe, 3 Lindemann falloff) from the group's LDS area: net
  // into q[j], or (QSS mechanisms) forward into q[j] and reverse into q[NR + j]
  template <int KIND>
  PPC_DI static void rate(const PK& pk, const double* ca, const double* b, double* q, const int j,
                          const double mixture, const double Tv, const double invT, const double logT,
                          const double refC, const double refCinv) {
    const tab::PackRx rx = pk.rx[j];
    const double kf0 = rx.A * exp(rx.b * logT - rx.E * invT);
    double kf = kf0;
    if constexpr (KIND >= 1) {
      double alpha = mixture;
      const tab::PackEff ef = pk.eff[j - T::N_EL];
#pragma unroll 4
      for (int i = 0; i < ef.n; ++i) alpha += pk.effV[ef.e0 + i] * ca[2 * pk.effK[ef.e0 + i]];
      if constexpr (KIND == 1) {
        kf *= alpha;
      } else {
        const tab::PackFo f = pk.fo[j - T::N_EL - T::N_TB];
        const double k0 = f.A * exp(f.b * logT - f.E * invT);
        const double redP = alpha / kf0 * k0;
        const double F = redP / (1.0 + redP);
        if constexpr (KIND == 2) {
          double Fcent = (1.0 - f.tA) * exp(-Tv / f.t3) + f.tA * exp(-Tv / f.t1);
          if (f.has2 != 0.0) Fcent += exp(-f.t2 * invT);
          const double logFcent = log10(Fcent);
          const double logPred = log10(redP);
          const double tc = -0.4 - 0.67 * logFcent;
          const double tn = 0.75 - 1.27 * logFcent;
          const double tr = (tc + logPred) / (tn - 0.14 * (tc + logPred));
          kf *= F * exp(LN10 * logFcent / (1.0 + tr * tr));
        } else {
          kf *= F;
        }
      }
    }
    const int r0 = rx.r[0], r1 = rx.r[1], r2 = rx.r[2];
    const double c0 = ca[2 * r0], a0 = ca[2 * r0 + 1], c1 = ca[2 * r1], a1 = ca[2 * r1 + 1];
    double qf = kf * c0 * c1;
    double a2 = 1.0;
    if (r2 != NX) {
      qf *= ca[2 * r2];
      a2 = ca[2 * r2 + 1];
    }
    double qr = 0.0;
    if (rx.flags & 1) {
      const int p2 = rx.p[2];
      qr = kf * refc_pow(rx.delta, refC, refCinv) * a0 * b[rx.p[0]] * a1 * a2 * b[rx.p[1]];
      if (p2 != NX) qr *= b[p2];
    }
    if constexpr (NQ > 0) {
      q[j] = rx.flags & 2 ? 0.0 : qf;
      q[NR + j] = qr;
    } else {
      q[j] = qf - qr;
    }
  }

  // sum of the terms of one chunk over the values in q
  PPC_DI static double chunk(const tab::PackCh& ch, const double* q) {
    double w = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) w += (double)((int)(ch.e[i] >> 12) - 8) * q[ch.e[i] & 0xfff];
    return w;
  }

  // QSS mechanisms: q holds the forward and reverse rates with the QSS
  // concentrations factored out.  Assembles the balances a row per lane (rows:
  // over the product exponentials, which are done with), solves them on
  // registers in every lane, puts the concentrations into ca, and makes q the
  // net rates.
  PPC_DI static void qss(const PK& pk, double* ca, double* q, double* rows, const int g) {
    if constexpr (NQ > 0) {
      wave_sync();
#pragma unroll 1
      for (int r = g; r < NROW; r += G) {
        double w = pk.qInit[r];
        const int v1 = pk.qRow[r + 1];
#pragma unroll 1
        for (int v = pk.qRow[r]; v < v1; ++v) w += chunk(pk.qch[v], q);
        rows[r] = w;
      }
      wave_sync();
      double A[T::NSLOT], x[NQ];
#pragma unroll
      for (int i = 0; i < T::NSLOT; ++i) A[i] = rows[i];
#pragma unroll
      for (int i = 0; i < NQ; ++i) x[i] = rows[T::NSLOT + i];
      T::qss_eliminate(A, x);
#pragma unroll
      for (int i = 0; i < NQ; ++i)
        if (g == i % G) ca[2 * (NS + i)] = x[i];
      wave_sync();
#pragma unroll 2
      for (int j = g; j < NR; j += G) {
        const tab::PackRx& rx = pk.rx[j];
        double f = q[j], r = q[NR + j];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
          const int kr = rx.r[l], kp = rx.p[l];
          if (kr >= NS && kr < NX) f *= ca[2 * kr];
          if (kp >= NS && kp < NX) r *= ca[2 * kp];
        }
        q[j] = f - r;
      }
      if (g == 0) q[NR] = 0.0;
    }
  }

  // w = production rates (mol/m^3/s) of this lane's species slots at Tv and the
  // densities y; hk[e] *= RT / molecular weight.  The group's LDS area is
  // overwritten; keep() runs when the rates are in q, the concentrations (the
  // QSS ones included) in ca and the QSS balances in b.
  template <class KEEP>
  PPC_DI static void production(const PK& pk, double* sh, const int g, const double Tv, const double invT,
                                const double (&y)[EPL], const double RT, double (&hk)[SPL], double (&w)[SPL],
                                const KEEP& keep) {
    const double logT = log(Tv);
    double* ca = sh + S_CA;
    double* b = sh + S_B;
    double* q = sh + S_Q;
    double msum = 0.0;
    if (g == 0) {
      ca[2 * NX] = 1.0;
      ca[2 * NX + 1] = 1.0;
      b[NX] = 1.0;
      q[NRATE - 1] = 0.0;
    }
#pragma unroll
    for (int e = 0; e < SPX; ++e) {
      const int k = e * G + g;
      if (k < NX) {
        double a[7], imw, sc = 1.0;  // QSS species: concentration factored out
        coefs(pk, k, Tv, a, imw);
        if (k < NS) {
          hk[e < SPL ? e : 0] *= RT * imw;  // CKUMS / CKHMS
          sc = (y[e < EPL ? e : 0] * imw) * 1.0e6;  // CKYTCR, SI
        }
        const double eg = exp(TM::g_poly(a, Tv, invT, logT));
        ca[2 * k] = sc;
        ca[2 * k + 1] = 1.0 / eg;
        b[k] = sc * eg;
        if (k < NS) msum += sc;
      }
    }
    const double mixture = Gr::sum(msum);
    const double refC = 101325.0 / 8.31446 * invT, refCinv = 1.0 / refC;
    wave_sync();
#pragma unroll 1
    for (int j = g; j < T::N_EL; j += G) rate<0>(pk, ca, b, q, j, mixture, Tv, invT, logT, refC, refCinv);
    if constexpr (T::N_TB > 0) {
#pragma unroll 1
      for (int j = T::N_EL + g; j < T::N_EL + T::N_TB; j += G)
        rate<1>(pk, ca, b, q, j, mixture, Tv, invT, logT, refC, refCinv);
    }
    if constexpr (T::N_TROE > 0) {
#pragma unroll 1
      for (int j = T::N_EL + T::N_TB + g; j < NR - T::N_LIND; j += G)
        rate<2>(pk, ca, b, q, j, mixture, Tv, invT, logT, refC, refCinv);
    }
    if constexpr (T::N_LIND > 0) {
#pragma unroll 1
      for (int j = NR - T::N_LIND + g; j < NR; j += G)
        rate<3>(pk, ca, b, q, j, mixture, Tv, invT, logT, refC, refCinv);
    }
    qss(pk, ca, q, b, g);
    wave_sync();
    keep();
    double* part = sh;
#pragma unroll 1
    for (int v = g; v < NCH; v += G) part[v] = chunk(pk.ch[v], q);
    wave_sync();
#pragma unroll
    for (int e = 0; e < SPL; ++e) {
      const int k = e * G + g;
      w[e] = 0.0;
      if (k < NS) {
        const int v1 = pk.spCh[k + 1];
#pragma unroll 2
        for (int v = pk.spCh[k]; v < v1; ++v) w[e] += part[v];
      }
    }
    wave_sync();
  }

  // fKernelSpec (Source/Reactions/ReactorUtils.H:358-415) for the group's
  // cell: y (this lane's equation slots), f = ydot of the same slots.
  PPC_DI static void rhs(const PK& pk, double* sh, const int g, const bool eform, const double dt_save,
                         const double (&y)[EPL], const double (&src)[SPL], const double rhoe_init,
                         const double rhoesrc_ext, double (&f)[EPL]) {
    double hk[SPL], cs, w[SPL];
    const double Tv = T_from_energy(pk, g, eform, rhoe_init + rhoesrc_ext * dt_save, y, Gr::bcast(y[TS], TL), cs, hk);
    production(pk, sh, g, Tv, 1.0 / Tv, y, RU * Tv, hk, w, [] {});
    double esum = 0.0;
#pragma unroll
    for (int e = 0; e < EPL; ++e) f[e] = 0.0;
#pragma unroll
    for (int e = 0; e < SPL; ++e) {
      const int k = e * G + g;
      if (k < NS) {
        const double s = w[e] * 1.0e-6 * pk.mw[k] + src[e];  // RTY2WDOT (CKWC units) + source
        f[e] = s;
        esum += s * hk[e];
      }
    }
    const double srcT = rhoesrc_ext - Gr::sum(esum);
    if (g == TL) f[TS] = srcT / (cs * RU);
  }

  // The BDF Jacobian d f_i / d y_j (bdf_jacobian in chem_cell.h with s = 1) of
  // one cell by WD lanes (the whole wave, or each group for its own cell): y in
  // wa[0..n) of their area, accumulated column-major (aJacobian / DWDOT layout)
  // in J, which is in LDS or, for the larger mechanisms, in the workspace;
  // jac_elem gives its elements.
  template <int CONSP, int WD>
  PPC_DI static void jacobian(const PK& pk, double* wa, double* J) {
    constexpr int W = (NS + WD - 1) / WD;
    const int l = Grp<WD>::lane();
    const double* y = wa;
    double *c = wa + NP, *gk = wa + 2 * NP, *hh = wa + 3 * NP, *wd = wa + 4 * NP;
    const auto ld = [&](int i) { return jload(J, i); };
    const auto st = [&](int i, double v) {
      if (JLDS)
        J[i] = v;
      else
        ws_store(J + i, v);
    };
    const auto jsync = [&]() {
      if (!JLDS) __threadfence();
      wave_sync();
    };
    const double Tv = y[NS];
    const double invT = 1.0 / Tv, invT2 = invT * invT, logT = log(Tv);
    const double refC = 101325.0 / 8.31446 * invT, refCinv = 1.0 / refC;
    double cR[W], dcR[W], eh[W], sc[W];
    double msum = 0.0;
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const int k = e * WD + l;
      cR[e] = dcR[e] = eh[e] = sc[e] = 0.0;
      if (k < NS) {
        double a[7], imw;
        coefs(pk, k, Tv, a, imw);
        const double hRT = TM::h_poly(a, Tv, invT), cpR = TM::cp_poly(a, Tv);
        sc[e] = y[k] * imw * 1.0e6;  // CKYTCR + DWDOT (x1e6)
        c[k] = sc[e];
        gk[k] = TM::g_poly(a, Tv, invT, logT);
        hh[k] = hRT;
        wd[k] = 0.0;
        cR[e] = (CONSP == 1) ? cpR : cpR - 1.0;
        eh[e] = (CONSP == 1) ? hRT : hRT - 1.0;
        dcR[e] = TM::dcp_poly(a, Tv);
        msum += sc[e];
      }
    }
#pragma unroll 1
    for (int i = l; i < n * n; i += WD) st(i, 0.0);
    const double mixture = Grp<WD>::sum(msum);
    jsync();
#pragma unroll 1
    for (int j = l; j < NR; j += WD)
      TM::template jac_reaction<CONSP>(
          j, c, gk, hh, mixture, Tv, invT, invT2, logT, refC, refCinv,
          [&](int idx, double v) {
            if (JLDS)
              __hip_atomic_fetch_add(J + idx, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            else
              unsafeAtomicAdd(J + idx, v);
          },
          [&](int m, double v) {
            __hip_atomic_fetch_add(wd + m, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          });
    jsync();
    // temperature row (aJacobian, Mechanisms/drm19/mechanism.H:15317-15352)
    double s_cm = 0.0, s_dcm = 0.0, s_eh = 0.0, s_deh = 0.0;
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const int k = e * WD + l;
      if (k < NS) {
        const double wdk = wd[k];
        s_cm += cR[e] * sc[e];
        s_dcm += dcR[e] * sc[e];
        s_eh += eh[e] * wdk;
        s_deh += invT * (cR[e] - eh[e]) * wdk + eh[e] * ld(NS * n + k);
      }
    }
    const double cmix = Grp<WD>::sum(s_cm), dcmixdT = Grp<WD>::sum(s_dcm);
    const double ehmix = Grp<WD>::sum(s_eh), dehmixdT = Grp<WD>::sum(s_deh);
    const double cmixinv = 1.0 / cmix;
    const double tmp1 = ehmix * cmixinv, tmp3 = cmixinv * Tv, tmp2 = tmp1 * tmp3;
    double trow[W];
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const int k = e * WD + l;
      trow[e] = 0.0;
      if (k < NS) {
        double d = 0.0;
#pragma unroll 8
        for (int mm = 0; mm < NS; ++mm) d += ((CONSP == 1) ? hh[mm] : hh[mm] - 1.0) * ld(k * n + mm);
        trow[e] = tmp2 * cR[e] - tmp3 * d;
      }
    }
    jsync();
#pragma unroll
    for (int e = 0; e < W; ++e)
      if (e * WD + l < NS) st((e * WD + l) * n + NS, trow[e]);
    if (l == 0) st(n * n - 1, -tmp1 + tmp2 * dcmixdT - tmp3 * dehmixdT);
    jsync();
  }
  PPC_DI static double jload(const double* J, const int i) { return JLDS ? J[i] : ws_load(J + i); }

  // The Jacobian of one cell by WD lanes, y in their area wa: in wa at J_AT or
  // (Jws) in the workspace.
  template <int WD>
  PPC_DI static void cell_jacobian(const PK& pk, double* wa, double* J, const bool eform) {
    if constexpr (NQ > 0) {
      group_qss_jacobian<T, G, WD>((lds_double*)wa, J, eform);
    } else if (eform) {
      jacobian<0, WD>(pk, wa, J);
    } else {
      jacobian<1, WD>(pk, wa, J);
    }
  }

  // d f_i / d y_j of jacobian()'s J: the DWDOT scaling (T column x1e-6, T row
  // x1e6) and the molecular-weight scaling
  PPC_DI static double jac_elem(const PK& pk, const double* J, const int i, const int j) {
    double v = jload(J, j * n + i);
    if (i == j) return v;  // no scaling, and no rounding, on the diagonal
    if (i == NS) v *= 1.0e6;
    if (j == NS) v *= 1.0e-6;
    v *= i < NS ? pk.mw[i] : 1.0;
    v *= j < NS ? pk.sp[j].imw : 1.0;
    return v;
  }
  // all of them by WD lanes, element (i, j) at out[(e*n + j)*G + g] for i = e*G + g
  // (unrolled four times it made the FP64 dodecane_lu_qss kernel spill 714 registers
  // in place of 463, ReactorCvode calls of 64 cells 3.1 -> 4.2 ms)
  template <int WD, typename JT>
  PPC_DI static void jac_rows(const PK& pk, const double* J, JT* out) {
    constexpr int U = NQ > 0 && !JLDS ? 2 : 4;
#pragma unroll U
    for (int t = WD == 64 ? (int)__lane_id() : Grp<WD>::lane(); t < n * n; t += WD) {
      const int j = t / n, i = t - j * n;
      out[((i / G) * n + j) * G + i % G] = (JT)jac_elem(pk, J, i, j);
    }
  }
};

// The QSS mechanisms' Jacobian (TabMech::jacobian_qss) of one cell by WD lanes
// (its group, or the wave): y in their LDS area, which is overwritten; J (n x n,
// column major) in that area at J_AT or in the workspace, followed by X, the
// derivatives of the balances by the concentrations (NQ x NS; then d x / d c), and
// W, d wdot / d x (NQ x NS).  Reactions are split over the lanes, with atomic sums;
// the QSS solves over the columns, and W X over its elements.
// Out of line: it is rare (about one per cell and call) and must not weigh on the
// registers of the steps.  What bounds it: the latency of the reactions' tables and
// of the rounds of unlike reaction kinds.  By one lane per cell it was 90% of a call
// (LuEthylene_qss, 4096 cells, 1e-5 s: 14 ms per Jacobian); with its sums in the
// workspace, and W X as a loop over all QSS reactions in every column, 65 to 90% of
// a call of up to 30 steps (figures at GroupLayout).
template <class T, int G, int WD>
__device__ __noinline__ void group_qss_jacobian(lds_double* area, double* Jws, const bool eform) {
  using C = GroupChem<T, WD>;
  using L = GroupLayout<T, G>;
  using Gr = Grp<WD>;
  using TM = TabMech<PackTab<T>>;
  constexpr int NS = T::NS, n = T::NEQ, NX = T::NX, NQ = T::NQ, SPL = C::SPL, SPX = C::SPX, NROW = C::NROW;
  constexpr int RPL = (NROW + WD - 1) / WD;
  const typename T::Packed& pk = lds_pack<T>();
  const int g = Gr::lane();
  double* const sh = (double*)area;
  double* const J = L::JLDS ? sh + L::J_AT : Jws;
  double *const X = J + L::JSQ, *const W = X + NQ * NS;
  const auto ld = [&](const double* p) { return L::JLDS ? *p : ws_load(p); };
  const auto st = [&](double* p, double v) {
    if (L::JLDS)
      *p = v;
    else
      ws_store(p, v);
  };
  const auto add = [&](double* p, double v) {
    if (L::JLDS)
      __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
      unsafeAtomicAdd(p, v);
  };
  const auto jsync = [&]() {
    if (!L::JLDS) __threadfence();
    wave_sync();
  };
  double y[C::EPL], w1[SPL], w0[SPL] = {}, hk[SPL], sce[SPX], rw[RPL];
  const double Tv = sh[NS];
#pragma unroll
  for (int e = 0; e < C::EPL; ++e) y[e] = e * WD + g < n ? sh[e * WD + g] : 0.0;
  wave_sync();
  // the rates at T + 1e-2 K (temperature column), then at T
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    const double Tq = pass == 0 ? Tv + 1.0e-2 : Tv;
#pragma unroll
    for (int e = 0; e < SPL; ++e) {
      w1[e] = w0[e];
      hk[e] = 0.0;
    }
    C::production(pk, sh, g, Tq, 1.0 / Tq, y, 1.0, hk, w0, [&] {
#pragma unroll
      for (int e = 0; e < SPX; ++e) sce[e] = e * WD + g < NX ? sh[C::S_CA + 2 * (e * WD + g)] : 0.0;
#pragma unroll
      for (int e = 0; e < RPL; ++e) rw[e] = e * WD + g < NROW ? sh[C::S_B + e * WD + g] : 0.0;
      wave_sync();
    });
  }
  double *c = sh, *gk = sh + NX, *hh = sh + 2 * NX, *c1 = sh + 3 * NX, *a = sh + 4 * NX, *b1 = sh + 5 * NX;
  double* const rows = sh + 6 * NX;
  const double invT = 1.0 / Tv, invT2 = invT * invT, logT = log(Tv);
  const double refC = 101325.0 / 8.31446 * invT, refCinv = 1.0 / refC;
  double cR[SPL], dcR[SPL], eh[SPL];
  double msum = 0.0;
#pragma unroll
  for (int e = 0; e < SPX; ++e) {
    const int k = e * WD + g;
    if (k < NX) {
      double p[7], imw;
      C::coefs(pk, k, Tv, p, imw);
      const double gr = TM::g_poly(p, Tv, invT, logT), hr = TM::h_poly(p, Tv, invT), eg = exp(gr);
      const double s1 = k < NS ? sce[e] : 1.0;
      c[k] = sce[e];
      gk[k] = gr;
      hh[k] = hr;
      c1[k] = s1;
      a[k] = 1.0 / eg;
      b1[k] = s1 * eg;
      if (e < SPL) {
        const double cp = TM::cp_poly(p, Tv);
        cR[e < SPL ? e : 0] = eform ? cp - 1.0 : cp;
        dcR[e < SPL ? e : 0] = TM::dcp_poly(p, Tv);
        eh[e < SPL ? e : 0] = eform ? hr - 1.0 : hr;
      }
      if (k < NS) msum += sce[e];
    }
  }
#pragma unroll
  for (int e = 0; e < RPL; ++e)
    if (e * WD + g < NROW) rows[e * WD + g] = rw[e];
#pragma unroll 1
  for (int i = g; i < L::JSTRIDE; i += WD) st(J + i, 0.0);
  const double mixture = Gr::sum(msum);
  jsync();
  const double* const x = c + NS;
  // (both from the last reaction down: the unlike kinds, which the tables have
  // last, share the first round)
#pragma unroll 1
  for (int i = T::NQR - 1 - g; i >= 0; i -= WD) {
    double qf, qr;
    TabMech<T>::qss_balance_terms(i, c1, a, b1, x, mixture, Tv, invT, logT, refC, refCinv, qf, qr,
                                  [&](int idx, double v) { add(X + idx, v); });
    const int j = T::qRx_(i);
    int qR = -1, qP = -1;
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const int r = T::rxR_(3 * j + l), p = T::rxP_(3 * j + l);
      if (r >= NS) qR = r - NS;
      if (p >= NS) qP = p - NS;
    }
    if (T::rxFwdOff_(j)) qR = -1;
    if (!T::rxRev_(j)) qP = -1;
#pragma unroll 1
    for (int l = 0; l < T::MAXNET; ++l) {
      const int m = T::rxNet_(T::MAXNET * j + l);
      if (m < 0) break;
      const double nu = T::rxNu_(T::MAXNET * j + l);
      if (qR >= 0) add(W + qR * NS + m, nu * qf);
      if (qP >= 0) add(W + qP * NS + m, -nu * qr);
    }
  }
#pragma unroll 1
  for (int j = T::NR - 1 - g; j >= 0; j -= WD)
    TM::template jac_reaction<0>(
        j, c, gk, hh, mixture, Tv, invT, invT2, logT, refC, refCinv,
        [&](int idx, double v) {
          if (idx < NS * n) add(J + idx, v);
        },
        [&](int, double) {});
  jsync();
  // d x / d c = -A^-1 d(balance)/d c, a column a lane
#pragma unroll 1
  for (int k = g; k < NS; k += WD) {
    double A[T::NSLOT], col[NQ];
#pragma unroll
    for (int i = 0; i < T::NSLOT; ++i) A[i] = rows[i];
#pragma unroll
    for (int i = 0; i < NQ; ++i) col[i] = -ld(X + i * NS + k);
    T::qss_eliminate(A, col);
#pragma unroll
    for (int i = 0; i < NQ; ++i) st(X + i * NS + k, col[i]);
  }
  jsync();
  // J += (d wdot / d x)(d x / d c); plain loads, which the fence has ordered after
  // the sums, and which the lanes of one round share in the cache
#pragma unroll 1
  for (int t = g; t < NS * NS; t += WD) {
    const int k = t / NS, m = t - k * NS;
    double d = J[k * n + m];
#pragma unroll
    for (int i = 0; i < NQ; ++i) d += W[i * NS + m] * X[i * NS + k];
    st(J + k * n + m, d);
  }
  jsync();
  // temperature column and row
  double s_cm = 0.0, s_dcm = 0.0, s_eh = 0.0, s_deh = 0.0;
#pragma unroll
  for (int e = 0; e < SPL; ++e) {
    const int k = e * WD + g;
    if (k < NS) {
      const double dT = (w1[e] - w0[e]) / 1.0e-2;
      st(J + NS * n + k, dT);
      s_cm += cR[e] * sce[e];
      s_dcm += dcR[e] * sce[e];
      s_eh += eh[e] * w0[e];
      s_deh += invT * (cR[e] - eh[e]) * w0[e] + eh[e] * dT;
    }
  }
  const double cmix = Gr::sum(s_cm), dcmixdT = Gr::sum(s_dcm);
  const double ehmix = Gr::sum(s_eh), dehmixdT = Gr::sum(s_deh);
  const double cmixinv = 1.0 / cmix;
  const double tmp1 = ehmix * cmixinv, tmp3 = cmixinv * Tv, tmp2 = tmp1 * tmp3;
#pragma unroll 1
  for (int k = g, e = 0; k < NS; k += WD, ++e) {
    double d = 0.0, ck = 0.0;
#pragma unroll 8
    for (int m = 0; m < NS; ++m) d += (eform ? hh[m] - 1.0 : hh[m]) * ld(J + k * n + m);
#pragma unroll
    for (int u = 0; u < SPL; ++u) ck = u == e ? cR[u] : ck;
    st(J + k * n + NS, tmp2 * ck - tmp3 * d);
  }
  if (g == 0) st(J + n * n - 1, -tmp1 + tmp2 * dcmixdT - tmp3 * dehmixdT);
  jsync();
}

// ------------------------------------------- group Newton-matrix inverse --
// Gauss-Jordan exchange steps on the row-distributed n x n matrix a (lane g
// holds rows i = e*G + g, e < EPL) with partial pivoting: step k pivots on the
// largest |a(i, k)| among the rows not yet used (the choice LU with partial
// pivoting makes); rows never move.  The pivot row goes through the group's
// LDS (prow).  Exchange on (r, k): a(r, k) <- 1 / a(r, k),
// a(r, j) <- -a(r, j) / a(r, k), a(i, k) <- a(i, k) / a(r, k) and
// a(i, j) <- a(i, j) - a(i, k) a(r, j) / a(r, k) for the other rows.  After the
// n steps (kstep[e] = the step at which row i was the pivot) A x = b is
// solved by x_{kstep(i)} = sum_j a(i, j) b_{p_j}, p_j the pivot row of step j.
//
// Every step's column is a[.][0]: the update of column j + 1 is written to
// place j and the exchanged column to place n - 1, so after n steps the
// columns are back in order, register indices are constants and the step loop
// is a loop: unrolled over n it is n^2 instructions per row slot (heptane,
// n = 89: ~0.4 MB of code) that miss the instruction cache at every step
// (heptane_lu_88sk, 2048 cells, one call of 1e-6 s at rtol 1e-8: 134 ms, 90%
// of it in this function, against 14.1 ms).
template <int n, int G, int EPL, typename LT>
PPC_DI void group_inv_factor(LT (&a)[EPL][n], int (&kstep)[EPL], LT* prow, const int g) {
  using Gr = Grp<G>;
#pragma unroll
  for (int e = 0; e < EPL; ++e) kstep[e] = (e * G + g < n) ? -1 : n;
#pragma unroll 1
  for (int k = 0; k < n; ++k) {
    LT best = LT(-1);
    int be = 0;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      LT m = fabs(a[e][0]);
      m = m == m ? m : LT(INFINITY);
      if (kstep[e] < 0 && m > best) {
        best = m;
        be = e;
      }
    }
    const LT mx = Gr::max(best);
    const int pl = __ffsll((long long)Gr::bits(__ballot(best == mx))) - 1;
    wave_sync();
    if (g == pl) {
#pragma unroll
      for (int j = 0; j < n; ++j) {
        LT v = a[0][j];
#pragma unroll
        for (int e = 1; e < EPL; ++e) v = (be == e) ? a[e][j] : v;
        prow[j] = v;
      }
    }
    wave_sync();
    const LT prs = LT(1) / prow[0];
    bool isp[EPL];
    LT f[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      isp[e] = g == pl && be == e;
      kstep[e] = isp[e] ? k : kstep[e];
      f[e] = isp[e] ? prs : a[e][0] * prs;
    }
#pragma unroll
    for (int j = 1; j < n; ++j) {
      if (j % 16 == 0) asm volatile("" ::: "memory");  // keeps few of the row's values in flight
      const LT r = prow[j];
#pragma unroll
      for (int e = 0; e < EPL; ++e) a[e][j - 1] = (isp[e] ? LT(0) : a[e][j]) - f[e] * r;
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) a[e][n - 1] = f[e];
  }
  wave_sync();
}

// x (this lane's equation slots) = A^-1 b (this lane's rows) from the
// exchanged matrix of group_inv_factor; v and w are n-vectors of the group's
// LDS.
template <int n, int G, int EPL, typename LT>
PPC_DI void group_inv_solve(const LT (&a)[EPL][n], const int (&kstep)[EPL], double* v, double* w, const int g,
                            const double (&b)[EPL], double (&x)[EPL]) {
#pragma unroll
  for (int e = 0; e < EPL; ++e)
    if (e * G + g < n) v[kstep[e]] = b[e];  // v_j = b_{p_j}
  wave_sync();
  double acc[EPL], acc2[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = acc2[e] = 0.0;
#pragma unroll
  for (int j = 0; j < n; ++j) {
    const double vj = v[j];
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      if (j % 2 == 0)
        acc[e] += (double)a[e][j] * vj;
      else
        acc2[e] += (double)a[e][j] * vj;
    }
  }
#pragma unroll
  for (int e = 0; e < EPL; ++e)
    if (e * G + g < n) w[kstep[e]] = acc[e] + acc2[e];  // x_{kstep(i)}
  wave_sync();
#pragma unroll
  for (int e = 0; e < EPL; ++e) x[e] = (e * G + g < n) ? w[e * G + g] : 0.0;
  wave_sync();
}

// D[0..order][e] <- (R U)^T D[0..order][e] for a step-size ratio `factor`
// (change_D in reactors.h) on this lane's equation slots, as U^T (R^T D):
// R[i][j] = prod_{m=1..i} (m - 1 - factor j) / m (R[i][0] = [i == 0]) and
// U = R at factor 1, both formed on the fly so that only the vector R^T D is
// held.
template <int EPL>
PPC_DI void group_change_D(double (&D)[AMAXORD + 3][EPL], const int order, const double factor) {
  constexpr double inv[AMAXORD + 1] = {0.0, 1.0, 0.5, 1.0 / 3.0, 0.25, 0.2};
  double w[AMAXORD + 1][EPL];
#pragma unroll
  for (int k = 0; k <= AMAXORD; ++k) {
    double r = 1.0;  // R[kp][k]
#pragma unroll
    for (int e = 0; e < EPL; ++e) w[k][e] = D[0][e];
#pragma unroll
    for (int kp = 1; kp <= AMAXORD; ++kp) {
      r *= (k == 0) ? 0.0 : (kp - 1 - factor * k) * inv[kp];
#pragma unroll
      for (int e = 0; e < EPL; ++e)
        if (kp <= order) w[k][e] += r * D[kp][e];
    }
  }
#pragma unroll
  for (int i = 0; i <= AMAXORD; ++i) {
    double u = 1.0;  // U[k][i]
    double s[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) s[e] = w[0][e];
#pragma unroll
    for (int k = 1; k <= AMAXORD; ++k) {
      u *= (i == 0) ? 0.0 : (k - 1 - i) * inv[k];  // zero for k > i: only terms k <= i <= order remain
#pragma unroll
      for (int e = 0; e < EPL; ++e)
        if (k <= i) s[e] += u * w[k][e];
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e)
      if (i <= order) D[i][e] = s[e];
  }
}

// A vector of the lane's equation slots kept in LDS: of the integrator's vectors
// the four that a trip reads and writes only a few times, so that the others
// and the inverse's rows stay in registers.
template <int EPL>
struct LaneVec {
  double* p;
  PPC_DI double& operator[](int e) const { return p[64 * e]; }
};

// 10 x the distance from t (>= 0) to the next double
PPC_DI double ten_ulps(const double t) {
  return 10.0 * (__longlong_as_double(__double_as_longlong(t) + 1) - t);
}

// Doubles of device workspace per wave: the Jacobian accumulator of the larger
// mechanisms (of every group's cell for the QSS ones) and the groups' Jacobian
// rows in JT.
template <class T, int G, typename JT>
constexpr long long group_ws_doubles() {
  constexpr int n = T::NEQ;
  constexpr long long epl = (n + G - 1) / G;
  return GroupChem<T, G>::JSPACE + (64 / G) * ((epl * n * G * (long long)sizeof(JT) + 15) / 16 * 2);
}

// Persistent kernel: each group of G lanes integrates cells from the queue
// until it is empty.  P.ws holds group_ws_doubles<T, G, LU_T>() doubles for
// each of P.ws_lanes / 64 waves; waves beyond that leave at once.
//
// CV: ReactorCvode's options (AdaptParamsDev), as adaptive_cell takes them: the
// order cap, the Newton iterations per attempt, the Jacobian's largest age and
// per-component absolute tolerances.
template <class T, typename LU_T, int G, int OCC, bool CV>
__global__ void __launch_bounds__(64 * GROUP_WAVES) __attribute__((amdgpu_waves_per_eu(OCC, 8)))
group_bdf_kernel(ReactParamsDev P, IO1D io, double dt, QueueArgs q, CellStats st) {
  using C = GroupChem<T, G>;
  using Gr = Grp<G>;
  using PK = typename T::Packed;
  constexpr int n = C::n, NS = C::NS, EPL = C::EPL, SPL = C::SPL, NP = C::NP;
  __shared__ __attribute__((aligned(16))) double lds[GROUP_WAVES * C::WAREA];
  __shared__ double lvec[GROUP_WAVES * C::L::LVEC];
  const PK& pk = load_pack<T>();
  const int wv = (int)(threadIdx.x >> 6);
  const long long wid = (long long)blockIdx.x * GROUP_WAVES + wv;
  if (wid >= P.ws_lanes / 64) return;  // the workspace holds no more waves
  const int g = Gr::lane();
  const int gi = (int)__lane_id() / G;
  double* const wa = lds + wv * C::WAREA;
  double* const lv = lvec + wv * C::L::LVEC + (threadIdx.x & 63);
  double* const sh = wa + gi * C::AREA;
  double* const sv = sh + C::S_Q;
  double* const sw = sv + NP;
  LU_T* const prow = reinterpret_cast<LU_T*>(sw + NP);
  constexpr long long GROWS = (long long)EPL * n * G;
  constexpr long long GSTRIDE = (GROWS * (long long)sizeof(LU_T) + 15) / 16 * 16 / (long long)sizeof(LU_T);
  double* const Jw = C::JLDS && !C::JOWN ? wa + C::J_AT : P.ws + wid * group_ws_doubles<T, G, LU_T>();
  // the groups' Jacobian rows: element (e, j) of lane g at [(e * n + j) * G + g]
  LU_T* const rows = reinterpret_cast<LU_T*>(P.ws + wid * group_ws_doubles<T, G, LU_T>() + C::JSPACE);
  const LU_T* const jrow = rows + gi * GSTRIDE + g;

  const AdaptParamsDev& ap = P.adapt;
  const bool eform = P.reactor_type == E_REACTOR;
  const double rtol = ap.rtol, atol = ap.atol;
  const double newton_tol = fmax(10 * 2.220446049250313e-16 / rtol, fmin(0.03, sqrt(rtol)));
  const double t_bound = dt;
  const long long rhs_cap = rhs_budget(ap.max_steps);
  const int maxord = CV && ap.max_order > 0 && ap.max_order < AMAXORD ? ap.max_order : AMAXORD;
  const int nmax = CV && ap.newton_maxiter > 0 ? ap.newton_maxiter : 4;
  // LU service: half of the wave's groups waiting, or as many trips.  A
  // factorisation for one group costs the whole wave the same, but a waiting
  // group idles (drm19, 262144 cells, 16 lanes per cell: 87 ms serving each
  // request at once, 79 ms at 2 groups or 2 trips, 83 ms at 4).
  constexpr int HALF = C::NG > 1 ? C::NG / 2 : 1;
  const int lu_batch = ap.lu_batch > 0 ? ap.lu_batch : HALF;
  const int lu_wait = ap.lu_wait > 0 ? ap.lu_wait : HALF;

  // this lane's equation slots (rows i = e*G + g); `valid` marks real equations
  bool valid[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) valid[e] = e * G + g < n;
  double atv[CV ? EPL : 1];
#pragma unroll
  for (int e = 0; e < (CV ? EPL : 1); ++e) atv[e] = CV && ap.atolv && valid[e] ? ap.atolv[e * G + g] : atol;
  // error weight of slot e at the value y
  auto weight = [&](int e, double y) { return atv[CV ? e : 0] + rtol * fabs(y); };
  int jac_step = 0;  // accepted steps at the last Jacobian
  double D[AMAXORD + 3][EPL];
  double yv[EPL];
  const LaneVec<EPL> d{lv}, ypred{lv + 64 * EPL}, psi{lv + 128 * EPL}, lus{lv + 192 * EPL};
  LU_T LU[EPL][n];  // the exchanged (inverted) Newton matrix, this lane's rows
  int kstep[EPL];
  double rhoe = 0, rhoesrc = 0;
  double t = 0, t_new = 0, h_abs = 0, c = 0, dy_norm_old = -1, h0 = 0;
  int order = 1, n_equal = 0, k_newton = 0, phase = PH_F0;
  int need_jac = 0;  // 1: at the initial state D[0], 2: at the predictor
  bool lu_valid = false, current_jac = false, need_lu = false;
  int nsteps = 0, nrhs = 0, njac = 0, nlu = 0, nnewton = 0, nrej = 0, status = 0, wait = 0;
  int cid = 0;
  bool active = false;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    kstep[e] = 0;
    yv[e] = 0.0;
    ypred[e] = 0.0;
#pragma unroll
    for (int j = 0; j < n; ++j) LU[e][j] = LU_T(0);
#pragma unroll
    for (int k = 0; k < AMAXORD + 3; ++k) D[k][e] = 0.0;
  }

  // sum over the cell's equations of (x / s)^2, root of its mean
  auto sq = [&](const double (&x)[EPL], const double (&s)[EPL]) {
    double acc = 0.0;
#pragma unroll
    for (int e = 0; e < EPL; ++e)
      if (valid[e]) {
        const double v = x[e] / s[e];
        acc += v * v;
      }
    return acc;
  };
  auto rms = [&](const double (&x)[EPL], const double (&s)[EPL]) { return sqrt(Gr::sum(sq(x, s)) / n); };

  auto next_cell = [&]() {
    int cl = 0;
    if (g == 0) cl = atomicAdd(q.counter, 1);
    const int cell = Gr::bcast(cl, 0);
    active = cell < q.ncells;
    if (!active) return;
    cid = q.order ? q.order[cell] : cell;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const int i = e * G + g;
      D[0][e] = valid[e] ? io.y[(long long)cid * n + i] : 0.0;
      yv[e] = D[0][e];
#pragma unroll
      for (int k = 1; k < AMAXORD + 3; ++k) D[k][e] = 0.0;
      d[e] = 0.0;
      ypred[e] = 0.0;
      psi[e] = 0.0;
      lus[e] = 1.0;
    }
    rhoe = io.rX[cid];
    rhoesrc = io.rXsrc[cid];
    t = 0.0;
    phase = PH_F0;
    order = 1;
    n_equal = 0;
    lu_valid = need_lu = false;
    need_jac = 0;
    jac_step = 0;
    wait = 0;
    nsteps = nrhs = njac = nlu = nnewton = nrej = status = 0;
  };

  auto finish_cell = [&]() {
#pragma unroll
    for (int e = 0; e < EPL; ++e)
      if (valid[e]) io.y[(long long)cid * n + e * G + g] = D[0][e];
    if (g == 0) {
      io.rX[cid] = rhoe + dt * rhoesrc;
      st.nsteps[cid] = status == 0 ? nsteps : status;
      if (st.nrhs) {
        st.nrhs[cid] = nrhs;
        st.njac[cid] = njac;
        st.nlu[cid] = nlu;
        st.nnewton[cid] = nnewton;
        st.nreject[cid] = nrej;
      }
    }
    next_cell();
  };

  next_cell();

  // S^-1 (I - c J) S in LU_T with S the error weights at the predictor, inverted
  auto factor = [&]() {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const double w = weight(e, ypred[e]);
      lus[e] = w;
      if (valid[e]) sv[e * G + g] = w;
    }
    wave_sync();
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      asm volatile("" ::: "memory");  // one slot's loads at a time
      const double si = 1.0 / lus[e];
      const int i = e * G + g;
#pragma unroll
      for (int j = 0; j < n; ++j) {
        const double jf = valid[e] ? (double)jrow[(e * n + j) * G] : 0.0;
        const double m = (i == j ? 1.0 : 0.0) - c * jf;
        LU[e][j] = valid[e] ? (LU_T)(si * m * sv[j]) : LU_T(0);
      }
    }
    group_inv_factor<n, G, EPL, LU_T>(LU, kstep, prow, g);
    nlu++;
    lu_valid = true;
  };

  // the loop runs until every group of the wave has drained the queue: all 64
  // lanes take part in the Jacobians
  while (__ballot(active)) {
    // ---- Jacobian requests: every group its own cell's, or the whole wave one
    // cell's after the other's (GroupLayout)
    unsigned long long jreq = __ballot(active && need_jac != 0 && g == 0);
    if constexpr (C::JOWN) {
      if (__builtin_expect(jreq != 0, 0)) {
        wave_sync();
        if (active && need_jac != 0) {
          double* const Jq = C::JLDS ? sh + C::J_AT : Jw + (long long)gi * C::JSTRIDE;
#pragma unroll
          for (int e = 0; e < EPL; ++e)
            if (valid[e]) sh[e * G + g] = need_jac == 1 ? D[0][e] : ypred[e];
          wave_sync();
          C::template cell_jacobian<G>(pk, sh, Jq, eform);
          C::template jac_rows<G>(pk, Jq, rows + gi * GSTRIDE);
          need_jac = 0;
          njac++;
        }
        __threadfence_block();
        wave_sync();
        jreq = 0;
      }
    }
    while (__builtin_expect(!C::JOWN && jreq != 0, 0)) {
      const int lead = __ffsll((long long)jreq) - 1, s = lead / G;
      jreq &= jreq - 1;
      wave_sync();
      if (gi == s) {
#pragma unroll
        for (int e = 0; e < EPL; ++e)
          if (valid[e]) wa[e * G + g] = need_jac == 1 ? D[0][e] : ypred[e];
      }
      wave_sync();
      // (without QSS species not through cell_jacobian, which made heptane_lu_88sk's
      // registers spill more: 783 -> 820, 10.5 -> 11.0 ms)
      if constexpr (T::NQ > 0)
        C::template cell_jacobian<64>(pk, wa, Jw, eform);
      else if (eform)
        C::template jacobian<0, 64>(pk, wa, Jw);
      else
        C::template jacobian<1, 64>(pk, wa, Jw);
      C::template jac_rows<64>(pk, Jw, rows + s * GSTRIDE);
      __threadfence_block();
      wave_sync();
      if (gi == s) {
        need_jac = 0;
        njac++;
      }
    }
    // ---- LU requests, served for the waiting groups together
    const unsigned long long lead = __ballot(active && g == 0);
    const unsigned long long waiting = __ballot(active && g == 0 && need_lu);
    if (waiting) {
      const bool stale = __ballot(active && need_lu && wait >= lu_wait) != 0;
      if ((__popcll(waiting) >= lu_batch || waiting == lead || stale) && active && need_lu) {
        factor();
        need_lu = false;
        wait = 0;
      }
    }
    if (!active) continue;
    if (need_lu) {  // not served yet: no RHS, no Newton iteration this trip
      ++wait;
      continue;
    }
    // what this trip leaves to do: a step attempt (of a new step or a repeated
    // one) after scaling D by a step-size ratio, or the end of the cell
    bool attempt = false, new_step = false, finish = false;
    double fac = 1.0;
    if (nrhs >= rhs_cap) {  // out of budget: the cell fails with the step-limit status
      status = -2;
      finish = true;
    } else {
      // ---- the one RHS evaluation of this trip
      const double t_eval = (phase == PH_F0) ? 0.0 : (phase == PH_F1 ? h0 : t_new);
      double f[EPL], src[SPL];
#pragma unroll
      for (int e = 0; e < SPL; ++e) {
        const int k = e * G + g;
        src[e] = k < NS ? io.ysrc[(long long)cid * NS + k] : 0.0;
      }
      C::rhs(pk, sh, g, eform, t_eval, yv, src, rhoe, rhoesrc, f);
      nrhs++;
      double scl[EPL];
      if (__builtin_expect(phase != PH_NEWTON, 0)) {
        // initial step size (Hairer, Norsett & Wanner I, II.4)
#pragma unroll
        for (int e = 0; e < EPL; ++e) scl[e] = weight(e, D[0][e]);
        if (phase == PH_F0) {
#pragma unroll
          for (int e = 0; e < EPL; ++e) D[1][e] = f[e];  // f0 kept in D[1] until h is known
          if (ap.first_step > 0) {
            h_abs = ap.first_step;
            attempt = true;
          } else {
            const double d0 = rms(D[0], scl), d1 = rms(f, scl);
            h0 = (d0 < 1e-5 || d1 < 1e-5) ? 1e-6 : 0.01 * d0 / d1;
            h0 = fmin(h0, t_bound);
#pragma unroll
            for (int e = 0; e < EPL; ++e) yv[e] = D[0][e] + h0 * f[e];
            phase = PH_F1;
          }
        } else {
#pragma unroll
          for (int e = 0; e < EPL; ++e) f[e] -= D[1][e];
          const double d1 = rms(D[1], scl);
          const double d2 = rms(f, scl) / h0;
          const double h1 = (d1 <= 1e-15 && d2 <= 1e-15) ? fmax(1e-6, h0 * 1e-3) : sqrt(0.01 / fmax(d1, d2));
          h_abs = fmin(fmin(100 * h0, h1), t_bound);
          attempt = true;
        }
        if (attempt) {
#pragma unroll
          for (int e = 0; e < EPL; ++e) D[1][e] *= h_abs;
          need_jac = 1;
          new_step = true;
          if (CV && !(t < t_bound)) {  // nothing to integrate (dt <= 0): no step, as adaptive_cell
            attempt = false;
            finish = true;
          }
        }
      } else {
        // one modified-Newton iteration with f = f(t_new, yv)
        nnewton++;
        bool bad = false;
#pragma unroll
        for (int e = 0; e < EPL; ++e) bad = bad || (valid[e] && !isfinite(f[e]));
        const bool finite = !Gr::any(bad);
        bool failed = !finite, converged = false;
        const int n_iter = k_newton + 1;
        if (finite) {
          double b[EPL], dy[EPL];
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            b[e] = valid[e] ? (c * f[e] - psi[e] - d[e]) / lus[e] : 0.0;
            scl[e] = weight(e, ypred[e]);
          }
          group_inv_solve<n, G, EPL, LU_T>(LU, kstep, sv, sw, g, b, dy);
#pragma unroll
          for (int e = 0; e < EPL; ++e) dy[e] *= lus[e];
          const double dy_norm = rms(dy, scl);
          const double rate = dy_norm_old < 0 ? -1.0 : dy_norm / dy_norm_old;
          double left = rate;  // rate^(nmax - k_newton)
          for (int i = k_newton; i < nmax - 1; ++i) left *= rate;
          if (rate >= 0 && (rate >= 1 || left / (1 - rate) * dy_norm > newton_tol)) {
            failed = true;
          } else {
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
              yv[e] += dy[e];
              d[e] += dy[e];
            }
            if (dy_norm == 0 || (rate >= 0 && rate / (1 - rate) * dy_norm < newton_tol)) {
              converged = true;
            } else {
              dy_norm_old = dy_norm;
              k_newton++;
              if (k_newton == nmax) failed = true;
            }
          }
        }
        if (failed) {
          if (!current_jac) {
            // refresh the Jacobian at the predictor and retry the same step
            need_jac = 2;
            current_jac = true;
            jac_step = nsteps;
            need_lu = true;
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
              yv[e] = ypred[e];
              d[e] = 0.0;
            }
            dy_norm_old = -1.0;
            k_newton = 0;
          } else {
            fac = 0.5;
            h_abs *= 0.5;
            n_equal = 0;
            lu_valid = false;
            nrej++;
            attempt = true;
          }
        } else if (converged) {
          const double safety = 0.9 * (2 * nmax + 1) / (double)(2 * nmax + n_iter);
          double err[EPL];
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            scl[e] = weight(e, yv[e]);
            err[e] = ndf_econst(order) * d[e];
          }
          const double error_norm = rms(err, scl);
          attempt = true;
          if (error_norm > 1) {
            fac = fmax(0.2, safety * exp(-log(error_norm) / (order + 1)));
            h_abs *= fac;
            n_equal = 0;
            nrej++;
          } else {
            // accept: D[order+2] = d - D[order+1]; D[order+1] = d; D[k] += D[k+1], k = order..0
            nsteps++;
            n_equal++;
            t = t_new;
            new_step = true;
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
#pragma unroll
              for (int kk = AMAXORD + 2; kk >= 1; --kk) {
                if (kk == order + 2) D[kk][e] = d[e] - D[kk - 1][e];
                if (kk == order + 1) D[kk][e] = d[e];
              }
#pragma unroll
              for (int kk = AMAXORD; kk >= 0; --kk)
                if (kk <= order) D[kk][e] += D[kk + 1][e];
            }
            if (n_equal >= order + 1) {
              double err2[EPL];
              const double cm = order > 1 ? ndf_econst(order - 1) : 0.0;
              const double cp = order < maxord ? ndf_econst(order + 1) : 0.0;
#pragma unroll
              for (int e = 0; e < EPL; ++e) {
                double vm = 0.0, vp = 0.0;
#pragma unroll
                for (int kk = 0; kk < AMAXORD + 3; ++kk) {
                  if (kk == order) vm = D[kk][e];
                  if (kk == order + 2) vp = D[kk][e];
                }
                err[e] = cm * vm;
                err2[e] = cp * vp;
              }
              const double sm = Gr::sum(sq(err, scl)), sp = Gr::sum(sq(err2, scl));
              const double norms[3] = {order > 1 ? sqrt(sm / n) : INFINITY, error_norm,
                                       order < maxord ? sqrt(sp / n) : INFINITY};
              double best = -1.0;
              int delta = 0;
#pragma unroll
              for (int i = 0; i < 3; ++i) {
                const double fct = (norms[i] == 0.0) ? INFINITY : exp(-log(norms[i]) / (order + i));
                if (fct > best) {
                  best = fct;
                  delta = i - 1;
                }
              }
              order += delta;
              fac = fmin(10.0, safety * best);
              h_abs *= fac;
              n_equal = 0;
              lu_valid = false;
            }
            if (!(t < t_bound)) {
              attempt = false;
              finish = true;
              // D[0] is the result whatever the next step size would be
              fac = 1.0;
            }
          }
        }
      }
    }
    if (attempt) {
      const double min_step = ten_ulps(t);
      if (new_step) {
        if (nsteps >= ap.max_steps) {
          status = -2;
          finish = true;
        } else if (h_abs < min_step) {
          fac *= min_step / h_abs;
          h_abs = min_step;
          n_equal = 0;
        }
        current_jac = false;
      }
      if (!finish && !(h_abs >= min_step)) {  // also ends a cell whose step size is NaN
        status = -3;
        finish = true;
      }
      if (!finish) {
        t_new = t + h_abs;
        if (t_new - t_bound > 0) {
          t_new = t_bound;
          fac *= fabs(t_new - t) / h_abs;
          n_equal = 0;
          lu_valid = false;
        }
        const double h = t_new - t;
        h_abs = fabs(h);
        if (fac != 1.0) group_change_D<EPL>(D, order, fac);
        const double inv_alpha = 1.0 / ndf_alpha(order);
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
          double sum = 0.0, ps = 0.0;
#pragma unroll
          for (int kk = 0; kk <= AMAXORD; ++kk)
            if (kk <= order) {
              sum += D[kk][e];
              if (kk > 0) ps += D[kk][e] * bdf_gamma(kk);
            }
          ypred[e] = sum;
          psi[e] = ps * inv_alpha;
          yv[e] = sum;
          d[e] = 0.0;
        }
        c = h * inv_alpha;
        // a Jacobian older than jac_age steps is re-evaluated at the prediction
        if (CV && ap.jac_age > 0 && !current_jac && nsteps - jac_step >= ap.jac_age) {
          need_jac = 2;
          current_jac = true;
          jac_step = nsteps;
          lu_valid = false;
        }
        if (!lu_valid) need_lu = true;
        dy_norm_old = -1.0;
        k_newton = 0;
        phase = PH_NEWTON;
      }
    }
    if (__builtin_expect(finish, 0)) finish_cell();
  }
}

}  // namespace ppc
