// ReactorRK64 and the fixed-step ReactorBDF with a group of G lanes per cell
// (the chemistry, lane layout and group primitives of group_bdf.h).
//
// One lane per cell (reactors.h) leaves most of the chip idle on boxes of up
// to a few ten thousand cells and keeps its matrices in private memory; here a
// cell's equations are spread over its group's lanes, its matrix rows sit in
// registers and the Krylov basis in LDS.  Box calls read and write the Array4
// views directly.  Arithmetic per cell is that of rk64_core and
// bdf_parity_cell / gmres up to the order of the sums.
#pragma once
#include "group_bdf.h"

namespace ppc {

// A call's cells: flat state (YCOrder) or a box, with the initial and final
// temperature inversions of ReactorBDF.cpp:376-389,461-478 for the box.
struct GroupIO {
  IO1D f;
  BoxArgs b;
};

template <class T, int G, bool BOX>
struct GroupCell {
  using C = GroupChem<T, G>;
  using PK = typename T::Packed;
  static constexpr int EPL = C::EPL, SPL = C::SPL, n = C::n, NS = C::NS;

  PPC_DI static void ijk(const BoxArgs& b, const int c, int& i, int& j, int& k) {
    i = b.lo[0] + c % b.len[0];
    j = b.lo[1] + (c / b.len[0]) % b.len[1];
    k = b.lo[2] + c / (b.len[0] * b.len[1]);
  }
  PPC_DI static void load(const GroupIO& io, const PK& pk, const int g, const bool eform, const int c,
                          double (&y)[EPL], double (&src)[SPL], double& rhoe, double& rhoesrc) {
    int i = 0, j = 0, k = 0;
    if (BOX) ijk(io.b, c, i, j, k);
#pragma unroll
    for (int e = 0; e < SPL; ++e) src[e] = 0.0;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const int s = e * G + g;
      y[e] = 0.0;
      if (s < NS) {
        y[e] = BOX ? io.b.rY(i, j, k, s) : io.f.y[(long long)c * n + s];
        src[e < SPL ? e : 0] = BOX ? io.b.rYsrc(i, j, k, s) : io.f.ysrc[(long long)c * NS + s];
      } else if (s == NS) {
        y[e] = BOX ? io.b.T(i, j, k, 0) : io.f.y[(long long)c * n + NS];
      }
    }
    rhoe = BOX ? io.b.rE(i, j, k, 0) : io.f.rX[c];
    rhoesrc = BOX ? io.b.rEsrc(i, j, k, 0) : io.f.rXsrc[c];
    if (BOX) {
      double cs, hk[SPL];
      const double Tv = C::T_from_energy(pk, g, eform, rhoe, y, Grp<G>::bcast(y[C::TS], C::TL), cs, hk);
      if (g == C::TL) y[C::TS] = Tv;
    }
  }
  PPC_DI static void store(const GroupIO& io, const PK& pk, const int g, const bool eform, const int c,
                           const double (&y)[EPL], const double rhoe, const double rhoesrc, const double dt,
                           const int steps, const CellStats& st) {
    int i = 0, j = 0, k = 0;
    const double E = rhoe + dt * rhoesrc;
    double Tv = 0.0;
    if (BOX) {
      ijk(io.b, c, i, j, k);
      double cs, hk[SPL];
      Tv = C::T_from_energy(pk, g, eform, E, y, Grp<G>::bcast(y[C::TS], C::TL), cs, hk);
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const int s = e * G + g;
      if (BOX) {
        if (s < NS) io.b.rY(i, j, k, s) = y[e];
      } else {
        if (s < n) io.f.y[(long long)c * n + s] = y[e];
      }
    }
    if (g == 0) {
      if (BOX) {
        io.b.rE(i, j, k, 0) = E;
        io.b.T(i, j, k, 0) = Tv;
        if (io.b.FC.p) io.b.FC(i, j, k, 0) = (double)steps;
      } else {
        io.f.rX[c] = E;
      }
      const int none[5] = {0, 0, 0, 0, 0};
      store_counters(st, c, steps, none);
    }
  }
};

// ------------------------------------------------------------- RK64 --------
// rk64_core (reactors.h) per group; every trip is one step of all six stages
// for every group of the wave, and a group that ends its cell takes the next.
// Bound by the latency of the right-hand sides at two waves per SIMD (170 to 209
// registers, nothing spilled).
template <class T, int G, bool BOX>
__global__ void __launch_bounds__(64 * GROUP_WAVES) __attribute__((amdgpu_waves_per_eu(2, 8)))
group_rk64_kernel(ReactParamsDev P, GroupIO io, double dt, int ncells, CellStats st) {
  using C = GroupChem<T, G>;
  using Gr = Grp<G>;
  using Cell = GroupCell<T, G, BOX>;
  constexpr int EPL = C::EPL, SPL = C::SPL, NG = 64 / G;
  __shared__ __attribute__((aligned(16))) double lds[GROUP_WAVES * NG * C::L::AREA_RHS];
  const auto& pk = load_pack<T>();
  const int g = Gr::lane();
  const int gb = (int)threadIdx.x / G;  // group of the block
  double* const sh = lds + gb * C::L::AREA_RHS;
  const bool eform = P.reactor_type == E_REACTOR;
  const RK64ParamsDev& p = P.rk64;
  const double dt_min = dt / (double)p.nsub_max, dt_max = dt / (double)p.nsub_min;
  const long long stride = (long long)gridDim.x * GROUP_WAVES * NG;
  long long c = (long long)blockIdx.x * GROUP_WAVES * NG + gb;
  double y[EPL], carry[EPL], src[SPL], rhoe = 0, rhoesrc = 0, now = 0, h = 0;
  int nsteps = 0;
  bool active = c < ncells;
  auto start = [&]() {
    Cell::load(io, pk, g, eform, (int)c, y, src, rhoe, rhoesrc);
#pragma unroll
    for (int e = 0; e < EPL; ++e) carry[e] = y[e];
    now = 0.0;
    h = dt / (double)p.nsub_guess;
    nsteps = 0;
  };
  if (active) start();
  while (active) {
    if (!(now < dt)) {
      Cell::store(io, pk, g, eform, (int)c, y, rhoe, rhoesrc, dt, nsteps, st);
      c += stride;
      active = c < ncells;
      if (active) start();
      continue;
    }
    double err[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) err[e] = 0.0;
#pragma unroll 1
    for (int s = 0; s < 6; ++s) {
      double f[EPL];
      C::rhs(pk, sh, g, eform, now, y, src, rhoe, rhoesrc, f);
      const double a = rk_alpha(s), b = rk_beta(s), er = rk_err(s);
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        err[e] += er * h * f[e];
        y[e] = carry[e] + a * h * f[e];
        carry[e] = y[e] + b * h * f[e];
      }
    }
    now += h;
    nsteps++;
    double me = 1e-50;
#pragma unroll
    for (int e = 0; e < EPL; ++e) me = fabs(err[e]) > me ? fabs(err[e]) : me;
    me = Gr::max(me);
    if (me < p.atol) {
      h = fmin(dt_max, h * pow(p.atol / me, 0.25));
    } else {
      h = fmax(dt_min, h * pow(p.atol / me, 0.2));
    }
    h = fmin(h, dt - now);
  }
}

// -------------------------------------------------- fixed-step BDF ----------
// bdf_parity_cell with gmres (reactors.h) on groups of 16 lanes, i.e. one DPP
// row per cell: the triangular sweeps of the preconditioner broadcast each
// unknown within the row by a DPP move (row_newbcast), without LDS.  A
// substep's first right-hand side is also the one at the old solution that the
// trapezoidal scheme asks for, since both states are the same there.
//
// GMRES stops at an absolute residual of 1e-10 in the equations' CGS units,
// below the rounding of hot cells' rates, so on such cells the result depends
// on how the sums round.  GMRES' own sums run over the same terms in the same
// order as in the one-lane form: rows of A and the sweeps by construction, the dot
// products one per lane (lane i takes basis vector i) over vectors in LDS, the
// norms in every lane.  The sums in the matrix and the right-hand side (Jacobian
// entries, heat and mixture sums, production rates) are the group's; the result on
// hot cells then lies within the spread of the one-lane form's own roundings
// (tests/test_gpu_fixed_group.py).
// One block per compute unit by its LDS (the Krylov bases of 16 cells), i.e. one
// wave per SIMD on dependent chains.
template <int J>
PPC_DI double row_bcast(const double v) {
  return wave::dpp<0x150 + J>(v);
}

template <int n, int EPL>
struct RowSolve {
  static constexpr int G = 16;
  using Gr = Grp<G>;

  // v / a with inv = 1 / a: the rounded product and one residual correction,
  // the quotient's own rounding without its ten-instruction chain
  PPC_DI static double div(const double v, const double a, const double inv) {
    const double q = v * inv;
    return fma(fma(-a, q, v), inv, q);
  }

  // x_j for j = J.. up: unknown J is lane J%16, slot J/16; s[e] sums A(i, j) x_j
  template <int J>
  PPC_DI static void forward(const double (&A)[EPL][n], const double (&dia)[EPL], const double (&inv)[EPL],
                             const double (&X)[EPL], double (&s)[EPL], double (&x)[EPL], const int g) {
    if constexpr (J < n) {
      constexpr int e0 = J / G;
      const double v = div(X[e0] - s[e0], dia[e0], inv[e0]);
      x[e0] = g == J % G ? v : x[e0];
      const double b = row_bcast<J % G>(v);
#pragma unroll
      for (int e = e0; e < EPL; ++e) s[e] += A[e][J] * b;
      forward<J + 1>(A, dia, inv, X, s, x, g);
    }
  }
  template <int J>
  PPC_DI static void backward(const double (&A)[EPL][n], const double (&dia)[EPL], const double (&inv)[EPL],
                              const double (&X)[EPL], double (&s)[EPL], double (&x)[EPL], const int g) {
    if constexpr (J >= 0) {
      constexpr int e0 = J / G;
      const double v = div(X[e0] - s[e0], dia[e0], inv[e0]);
      x[e0] = g == J % G ? v : x[e0];
      const double b = row_bcast<J % G>(v);
#pragma unroll
      for (int e = 0; e <= e0; ++e) s[e] += A[e][J] * b;
      backward<J - 1>(A, dia, inv, X, s, x, g);
    }
  }
  // M^-1 X (ReactorBDFsolver.H:12-91): 0 none, 1 Jacobi, 2 symmetric
  // Gauss-Seidel (D+L) D^-1 (D+U)
  PPC_DI static void precond(double (&out)[EPL], const double (&A)[EPL][n], const double (&dia)[EPL],
                             const double (&inv)[EPL], const double (&X)[EPL], const int type, const int g) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) out[e] = type == 0 ? X[e] : div(X[e], dia[e], inv[e]);
    if (type != 2) return;
    double s[EPL], yd[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) s[e] = yd[e] = 0.0;
    forward<0>(A, dia, inv, X, s, yd, g);
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      yd[e] *= dia[e];
      s[e] = 0.0;
    }
    backward<n - 1>(A, dia, inv, yd, s, out, g);
  }
  // A x with x (n doubles) in LDS
  PPC_DI static void mul(double (&out)[EPL], const double (&A)[EPL][n], const double* x) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) out[e] = 0.0;
#pragma unroll
    for (int j = 0; j < n; ++j) {
      const double v = x[j];
#pragma unroll
      for (int e = 0; e < EPL; ++e) out[e] += A[e][j] * v;
    }
  }
  // sum over l of a_l b_l in order, vectors in LDS
  PPC_DI static double dot(const double* a, const double* b) {
    double s = 0.0;
#pragma unroll
    for (int l = 0; l < n; ++l) s += a[l] * b[l];
    return s;
  }

  // The group's LDS of one solve (doubles): a vector, the basis, the rotated
  // Hessenberg columns (upper triangle, packed by column), rotations,
  // right-hand side and solution of the least-squares problem.
  static constexpr int NP = (n + 1) & ~1;
  static constexpr int S_V = NP, S_R = S_V + (n + 1) * n, S_CS = S_R + n * (n + 1) / 2, S_SN = S_CS + n,
                       S_BE = S_SN + n, S_Y = S_BE + n + 1, SIZE = S_Y + n + 1;

  // Restarted GMRES with warm start (gmres in reactors.h): x0 the initial
  // guess (overwritten), x the solution; false when a NaN/Inf appears in H.
  PPC_DI static bool gmres(double* sh, const double (&A)[EPL][n], const double (&dia)[EPL],
                           const double (&inv)[EPL], const double (&b)[EPL], double (&x0)[EPL], double (&x)[EPL],
                           const int ptype, const int restarts, const int kspiters, const double tol, const int g) {
    constexpr int K = n;
    double *V = sh + S_V, *R = sh + S_R, *cs = sh + S_CS, *sn = sh + S_SN, *be = sh + S_BE, *yv = sh + S_Y;
    auto put = [&](double* to, const double (&v)[EPL]) {
#pragma unroll
      for (int e = 0; e < EPL; ++e)
        if (e * G + g < n) to[e * G + g] = v[e];
    };
    auto get = [&](const double* from, double (&v)[EPL]) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) v[e] = e * G + g < n ? from[e * G + g] : 0.0;
    };
    for (int i = g; i < K * (K + 1) / 2; i += G) R[i] = 0.0;
    for (int i = g; i <= K; i += G) yv[i] = be[i] = 0.0;
    double r[EPL], t1[EPL], t2[EPL];
    put(sh, x0);
    wave_sync();
    mul(t1, A, sh);
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      t1[e] = b[e] - t1[e];
      x[e] = x0[e];
    }
    precond(r, A, dia, inv, t1, ptype, g);
    double residnorm = 0.0;
    bool lucky = false;
#pragma unroll 1
    for (int it = 0; it < restarts; ++it) {
      wave_sync();
      put(sh, r);
      wave_sync();
      const double beta = sqrt(dot(sh, sh));
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        x0[e] = x[e];
        t2[e] = r[e] / beta;
      }
      put(V, t2);
      double bk = beta;  // be[k]
      int opt = K;
#pragma unroll 1
      for (int k = 0; k < kspiters; ++k) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) x[e] = x0[e];
        wave_sync();
        mul(t1, A, V + k * n);
        precond(t2, A, dia, inv, t1, ptype, g);
        double* col = R + k * (k + 1) / 2;
        wave_sync();
        put(sh, t2);
        wave_sync();
#pragma unroll 1
        for (int i = g; i <= k; i += G) col[i] = dot(sh, V + i * n);
        wave_sync();
#pragma unroll 2
        for (int i = 0; i <= k; ++i) {
          double vi[EPL];
          get(V + i * n, vi);
          const double hi = col[i];
#pragma unroll
          for (int e = 0; e < EPL; ++e) t2[e] = t2[e] - hi * vi[e];
        }
        wave_sync();
        put(sh, t2);
        wave_sync();
        const double hn = sqrt(dot(sh, sh));
        lucky = false;
        if (hn > tol * 0.01) {
#pragma unroll
          for (int e = 0; e < EPL; ++e) t1[e] = t2[e] / hn;
          put(V + (k + 1) * n, t1);
        } else {
          if (!isfinite(hn)) return false;
          lucky = true;
        }
        double prev = col[0];
#pragma unroll 1
        for (int i = 0; i < k; ++i) {
          const double next = col[i + 1], c = cs[i], s = sn[i];
          const double tmp = c * prev + s * next;
          prev = -s * prev + c * next;
          if (g == 0) col[i] = tmp;
        }
        double c, sg;
        if (prev == 0) {
          c = 0.0;
          sg = 1.0;
        } else {
          const double d = sqrt(prev * prev + hn * hn);
          c = prev / d;
          sg = hn / d;
        }
        if (g == 0) {
          col[k] = c * prev + sg * hn;
          cs[k] = c;
          sn[k] = sg;
          be[k] = c * bk;
          be[k + 1] = -sg * bk;
        }
        bk = -sg * bk;
        residnorm = fabs(bk);
        if (lucky || residnorm <= tol) {
          opt = k + 1;
          break;
        }
      }
      wave_sync();
      // uppertrisolve (ReactorBDFsolver.H:368-382): the column index runs up to
      // opt inclusive; column K lies outside the Hessenberg matrix and is zero
#pragma unroll 1
      for (int i = opt - 1; i >= 0; --i) {
        double v = be[i];
#pragma unroll 1
        for (int j = i + 1; j <= opt && j < K; ++j) v -= R[j * (j + 1) / 2 + i] * yv[j];
        v /= R[i * (i + 1) / 2 + i];
        wave_sync();
        if (g == 0) yv[i] = v;
        wave_sync();
      }
#pragma unroll 1
      for (int i = 0; i < opt; ++i) {
        double vi[EPL];
        get(V + i * n, vi);
        const double s = yv[i];
#pragma unroll
        for (int e = 0; e < EPL; ++e) x[e] = x[e] + s * vi[e];
      }
      if (residnorm <= tol || lucky) break;
    }
    return true;
  }
};

// A group's Jacobian, right-hand side and Krylov space share one area (doubles).
template <class T>
constexpr int group_fixed_area() {
  using L = GroupLayout<T, 16>;
  return L::padded(L::cmax(L::cmax(RowSolve<L::n, L::EPL>::SIZE, L::S_RAW), L::JLEN));
}
template <class M>
constexpr bool group_fixed_fits() {
  if constexpr (group_fixed_ok<M>()) {
    using T = typename packed_tables<M>::type;
    return (long long)sizeof(typename T::Packed) + 8LL * GROUP_WAVES * 4 * group_fixed_area<T>() <= LDS_BYTES;
  }
  return false;
}

template <class T, bool BOX>
__global__ void __launch_bounds__(64 * GROUP_WAVES) __attribute__((amdgpu_waves_per_eu(1, 8)))
group_bdf_fixed_kernel(ReactParamsDev P, GroupIO io, double dt_react, int ncells, CellStats st) {
  constexpr int G = 16, NG = 4;
  using C = GroupChem<T, G>;
  using Gr = Grp<G>;
  using Cell = GroupCell<T, G, BOX>;
  constexpr int n = C::n, EPL = C::EPL, SPL = C::SPL;
  using RS = RowSolve<n, EPL>;
  constexpr int RSIZE = group_fixed_area<T>();
  static_assert(C::JLDS && C::NQ == 0, "the Jacobian of these mechanisms is in LDS");
  __shared__ __attribute__((aligned(16))) double lds[GROUP_WAVES * NG * RSIZE];
  const auto& pk = load_pack<T>();
  const int g = Gr::lane();
  double* const sh = lds + ((int)threadIdx.x / G) * RSIZE;
  const bool eform = P.reactor_type == E_REACTOR;
  const BDFParamsDev& p = P.bdf;
  const double dt = dt_react / (double)p.nsubsteps, dt_inv = 1.0 / dt;
  const int first = p.scheme >= 2 ? 1 : p.scheme, change = p.scheme - 2;
  const long long stride = (long long)gridDim.x * GROUP_WAVES * NG;
  long long c = (long long)blockIdx.x * GROUP_WAVES * NG + (int)threadIdx.x / G;
  for (; c < ncells; c += stride) {
    double y[EPL], soln[EPL], soln_n[EPL], nm1[EPL], nm2[EPL], ds[EPL], src[SPL], rhoe = 0, rhoesrc = 0;
#pragma unroll
    for (int e = 0; e < EPL; ++e) y[e] = 0.0;
    Cell::load(io, pk, g, eform, (int)c, y, src, rhoe, rhoesrc);
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      soln[e] = soln_n[e] = nm1[e] = nm2[e] = y[e];
      ds[e] = 0.0;
    }
    double now = 0.0;
    bool ok = true;  // no NaN so far
#pragma unroll 1
    for (int s = 0; s < p.nsubsteps; ++s) {
      const int ts = s > change ? p.scheme : first;
      const double t0 = tcoeff(ts, 0), t1 = tcoeff(ts, 1), t2 = tcoeff(ts, 2), t3 = tcoeff(ts, 3);
      const double f0 = fcoeff(ts, 0), f1 = fcoeff(ts, 1);
      double fn[EPL];
#pragma unroll
      for (int e = 0; e < EPL; ++e) fn[e] = 0.0;
      bool on = ok;  // this substep's Newton iterations go on
#pragma unroll 1
      for (int it = 0; it < p.nonlinear_iters && on; ++it) {
        // get_bdf_matrix_and_rhs (ReactorBDF.cpp:36-110)
        double A[EPL][n], dia[EPL], inv[EPL];
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
#pragma unroll
          for (int j = 0; j < n; ++j) A[e][j] = 0.0;
          dia[e] = 1.0;
        }
        // every group its own Jacobian: they all want one at the same time
        wave_sync();
#pragma unroll
        for (int e = 0; e < EPL; ++e)
          if (e * G + g < n) sh[e * G + g] = soln[e];
        wave_sync();
        if (eform)
          C::template jacobian<0, G>(pk, sh, sh + C::J_AT);
        else
          C::template jacobian<1, G>(pk, sh, sh + C::J_AT);
        wave_sync();
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
          const int i = e * G + g;
#pragma unroll
          for (int j = 0; j < n; ++j)
            if (i < n) {
              double v = -f0 * C::jac_elem(pk, sh + C::J_AT, i, j);
              if (i == j) {
                v += t0 * dt_inv;
                dia[e] = v;
              }
              A[e][j] = v;
            }
        }
        wave_sync();
        double f[EPL], rhs[EPL], ds0[EPL];
        C::rhs(pk, sh, g, eform, now, soln, src, rhoe, rhoesrc, f);
        double nrm = 0.0;
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
          if (ts == 1 && it == 0) fn[e] = f[e];  // the old solution is where the substep starts
          inv[e] = 1.0 / dia[e];
          ds0[e] = ds[e];
          double r = -t0 * soln[e] * dt_inv;
          r += -t1 * soln_n[e] * dt_inv;
          r += -t2 * nm1[e] * dt_inv;
          r += -t3 * nm2[e] * dt_inv;
          r += f0 * f[e];
          r += f1 * fn[e];
          rhs[e] = e * G + g < n ? r : 0.0;
          nrm += rhs[e] * rhs[e];
        }
        wave_sync();
        if (!RS::gmres(sh, A, dia, inv, rhs, ds0, ds, p.gmres_precond, p.gmres_restarts, p.gmres_kspiters,
                       p.gmres_tol, g)) {
          ok = on = false;
        } else {
#pragma unroll
          for (int e = 0; e < EPL; ++e) soln[e] += ds[e];
          if (sqrt(Gr::sum(nrm)) <= p.nonlin_tol) on = false;
        }
      }
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        nm2[e] = nm1[e];
        nm1[e] = soln_n[e];
        soln_n[e] = soln[e];
      }
      now += dt;
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) soln_n[e] = ok ? soln_n[e] : y[e];  // a failed cell keeps its state
    Cell::store(io, pk, g, eform, (int)c, soln_n, rhoe, rhoesrc, dt_react, ok ? p.nsubsteps : -1, st);
  }
}

}  // namespace ppc
