// Per-lane matrices of the larger mechanisms in an HBM workspace.
//
// A lane's private (scratch) frame is limited to 128 KiB on gfx950, and the
// compiler's frame handling breaks down well before that when the frame holds
// several n x n matrices (dodecane_lu: n = 54, heptane_lu_88sk: n = 89).  For
// mechanisms with NEQ > PPC_WS_MIN_NEQ the integrators keep their Jacobians,
// LU factors and Krylov bases in a workspace the host allocates instead, laid
// out element-major across lanes: element i of an array that starts at row o
// lives at ws[(o + i) * lanes + g] for lane g, so the 64 lanes of a wave touch
// 64 consecutive words (one coalesced 512-byte access for doubles), the same
// interleaving the hardware gives private memory.  A row is `lanes` doubles; an
// array of m floats takes ceil(m / 2) rows.
#pragma once
#include <type_traits>
#include "erk_tables.h"
#include "group_layout.h"
#include "ppc_common.h"
#include "reactors_fwd.h"

#ifndef PPC_WS_MIN_NEQ
#define PPC_WS_MIN_NEQ 32
#endif

namespace ppc {

template <class M>
constexpr bool uses_ws() {
  return M::NEQ > PPC_WS_MIN_NEQ;
}

// One lane's view of an array in the workspace: element i at p[i * s].
template <typename T>
struct LaneArr {
  T* p;
  long long s;
  PPC_DI T& operator[](long long i) const { return p[i * s]; }
};

struct LaneWS {
  double* base;     // workspace (lanes * rows doubles)
  long long lanes;  // lanes sharing it (a multiple of 64)
  long long g;      // this lane
  template <typename T>
  PPC_DI LaneArr<T> at(long long row) const {
    return {reinterpret_cast<T*>(base + row * lanes) + g, lanes};
  }
};

// Rows taken by m elements of T.
template <typename T>
constexpr long long ws_rows(long long m) {
  return sizeof(T) == 8 ? m : (m + 1) / 2;
}

// An array of T with m elements: private when WS is false (`priv` must hold
// m elements), else at `row` of the workspace.
template <bool WS, typename T>
PPC_DI auto lane_array(T* priv, const LaneWS& w, long long row) {
  if constexpr (WS)
    return w.template at<T>(row);
  else
    return priv;
}

// Workspace rows per lane of each integrator; 0 when the mechanism keeps its
// matrices in private memory.
template <class M>
constexpr long long integrator_ws_rows(int mode) {
  constexpr long long n = M::NEQ, nn = n * n;
  if (mode == MODE_ERK) return ERK_MAX_STAGES * n;  // the stages, every mechanism
  if (!uses_ws<M>()) return 0;
  switch (mode) {
    case MODE_BDF: return nn + 2 * (n + 1) * n;                   // A, Krylov basis V, Hessenberg H
    case MODE_ADAPTIVE: return 2 * nn;                            // J, LU (FP64)
    default: return 0;
  }
}

// ---- batched group kernel (group_bdf.h): G lanes per cell
template <class M, class = void>
struct has_table : std::false_type {};
template <class M>
struct has_table<M, std::void_t<decltype(M::kTable)>> : std::integral_constant<bool, M::kTable> {};

// Groups of G lanes per cell exist for the table-driven mechanisms with at most
// three equations per lane (NEQ <= 3 G) and at least half the lanes holding
// an equation (G <= 2 NEQ).
template <class M, class = void>
struct has_qss : std::false_type {};
template <class M>
struct has_qss<M, std::void_t<decltype(M::NQ)>> : std::integral_constant<bool, (M::NQ > 0)> {};

// The packed tables the group kernels read (the generator leaves them out for a
// mechanism that their records cannot hold).
template <class M, class = void>
struct packed_tables {
  using type = void;
};
template <class M>
struct packed_tables<M, std::void_t<typename M::Tables::Packed>> {
  using type = typename M::Tables;
};

// QSS mechanisms: at most one equation in four is in a second slot (NEQ <=
// 4 G / 3).  A group keeps its forward and reverse rates apart, twice the LDS,
// so a narrow group's waves do not share a SIMD (LuEthylene_qss, 65536 cells:
// 16 lanes 81 ms, 32 lanes 60 ms; 4096 cells 9.1 and 7.0 ms).  The tables and
// the areas of a block must fit the LDS: the narrower the groups, the more of
// them a wave has.
template <class M, int G>
constexpr bool group_ok() {
  using T = typename packed_tables<M>::type;
  if constexpr (std::is_void<T>::value) {
    return false;
  } else if constexpr (!(M::NEQ <= 3 * G && G <= 2 * M::NEQ && (!has_qss<M>::value || 3 * M::NEQ <= 4 * G))) {
    return false;
  } else {
    return has_table<M>::value && GroupLayout<T, G>::fits();
  }
}

// The fixed-step BDF's group kernel (16 lanes per cell) holds the Krylov bases
// of a wave's four cells in LDS: 24 equations at most; below 17 the one-lane
// kernel runs (fixed_cells_per_wave in capi.hip).
template <class M>
constexpr bool group_fixed_ok() {
  return group_ok<M, 16>() && !has_qss<M>::value && M::NEQ <= 24 && M::NEQ > 16;
}

// Device workspace of one wave of the group kernel (doubles, at most): an n x n
// FP64 Jacobian accumulator (QSS mechanisms: one per group, with the terms of
// the QSS balances) and the Jacobian rows of its 64 / G groups.
template <class M, int G>
constexpr long long group_wave_doubles() {
  constexpr long long n = M::NEQ, acc = n * n + 1, groups = 64 / G;
  constexpr long long rows = groups * ((n + G - 1) / G * n * G + 1);
  if constexpr (has_qss<M>::value)
    return groups * (acc + 2 * M::NQ * (n - 1) + 1) + rows;
  else
    return acc + rows;
}

// Workspace rows per lane (doubles, 64-lane blocks as lane_ws) of the group
// kernel with cells_per_wave cells per wave; 0 when there is no such kernel.
template <class M>
long long group_ws_rows(int cells_per_wave) {
  switch (cells_per_wave) {
    case 8: return group_ok<M, 8>() ? (group_wave_doubles<M, 8>() + 63) / 64 : 0;
    case 4: return group_ok<M, 16>() ? (group_wave_doubles<M, 16>() + 63) / 64 : 0;
    case 2: return group_ok<M, 32>() ? (group_wave_doubles<M, 32>() + 63) / 64 : 0;
    case 1: return group_ok<M, 64>() ? (group_wave_doubles<M, 64>() + 63) / 64 : 0;
    default: return 0;
  }
}

}  // namespace ppc
