// Kernel launch definitions, included by the per-(mechanism, integrator)
// instantiation units only.
#pragma once
#include <type_traits>
#include "launch.h"
#include "wave_bdf.h"
#include "wave_adjoint.h"
#include "group_bdf.h"
#include "group_fixed.h"
#include "flatten.h"

namespace ppc {

// Table-driven mechanism tables of a mechanism type (void for the generated
// straight-line mechanisms): the group and wave-per-cell kernels read them.
template <class M>
struct wave_tables {
  using type = void;
};
template <class T>
struct wave_tables<TabMech<T>> {
  using type = T;
};

// Blocks of the one-lane-per-cell kernels: one lane per cell, or, with a
// workspace, exactly the lanes it holds (the lanes then stride over the cells).
template <class M, int MODE>
int lane_grid(const ReactParamsDev& P, int ncells, int block) {
  if (integrator_ws_rows<M>(MODE) > 0) {
    if (!P.ws || P.ws_lanes < block || P.ws_lanes % block != 0) return -1;
    return (int)(P.ws_lanes / block);
  }
  return (ncells + block - 1) / block;
}

// The plain adaptive BDF is built at the compiler's occupancy and, for
// mechanisms without a workspace, also held to 2 and 4 waves per SIMD
// (P.adapt.lane_occ); the parity integrators at the compiler's choice only.
template <class M, int MODE>
hipError_t launch_1d_mode(const ReactParamsDev& P, double* y, const double* ysrc, double* rX,
                          const double* rXsrc, double dt, int ncells, CellStats st, int block, hipStream_t s) {
  const int grid = lane_grid<M, MODE>(P, ncells, block);
  if (grid < 0) return hipErrorInvalidValue;
  if constexpr (MODE == MODE_ADAPTIVE && !uses_ws<M>()) {
    auto k = P.adapt.lane_occ == 4 ? react_1d_kernel_held<M, MODE, 4>
                                   : (P.adapt.lane_occ == 2 ? react_1d_kernel_held<M, MODE, 2> : react_1d_kernel<M, MODE>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(block), 0, s, P, y, ysrc, rX, rXsrc, dt, ncells, st);
  } else {
    hipLaunchKernelGGL((react_1d_kernel<M, MODE>), dim3(grid), dim3(block), 0, s, P, y, ysrc, rX, rXsrc, dt,
                       ncells, st);
  }
  return hipGetLastError();
}

template <class M, int MODE>
hipError_t launch_box_mode(const ReactParamsDev& P, const BoxArgs& b, double dt, int ncells, CellStats st,
                           int block, hipStream_t s) {
  const int grid = lane_grid<M, MODE>(P, ncells, block);
  if (grid < 0) return hipErrorInvalidValue;
  if constexpr (MODE == MODE_ADAPTIVE && !uses_ws<M>()) {
    auto k = P.adapt.lane_occ == 4 ? react_box_kernel_held<M, MODE, 4>
                                   : (P.adapt.lane_occ == 2 ? react_box_kernel_held<M, MODE, 2> : react_box_kernel<M, MODE>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(block), 0, s, P, b, dt, ncells, st);
  } else {
    hipLaunchKernelGGL((react_box_kernel<M, MODE>), dim3(grid), dim3(block), 0, s, P, b, dt, ncells, st);
  }
  return hipGetLastError();
}

// Persistent launch: as many blocks as can be resident at once (never more than
// `lanes` needs); lanes or waves take cells from the queue.
template <class K>
int resident_blocks(K kernel, long long lanes, int block = 64) {
  int dev = 0, ncu = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess) return -1;
  if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return -1;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess) return -1;
  if (per_cu < 1) per_cu = 1;
  const long long need = (lanes + block - 1) / block;
  const long long blocks = (long long)ncu * per_cu;
  return (int)(blocks < need ? blocks : need);
}

// The group kernel (group_bdf.h) with G lanes per cell: a persistent grid of
// every resident block of GROUP_WAVES waves, at most q.max_blocks waves and the
// waves the workspace holds (group_ws_rows rows of 64 lanes per wave).
template <class T, typename LU_T, int G, bool CV>
hipError_t launch_group(const ReactParamsDev& P, double* y, const double* ysrc, double* rX, const double* rXsrc,
                        double dt, QueueArgs q, CellStats st, hipStream_t s) {
  static_assert(group_ws_doubles<T, G, LU_T>() <= group_wave_doubles<TabMech<T>, G>(), "workspace layout");
  // registers of the inverse's rows: above ~100 VGPRs hold the build to one wave per SIMD
  constexpr int lu_vgprs = (int)(((T::NEQ + G - 1) / G) * T::NEQ * sizeof(LU_T) / 4);
  auto k = group_bdf_kernel<T, LU_T, G, (lu_vgprs > 100 ? 1 : 2), CV>;
  int grid = resident_blocks(k, (long long)q.ncells * G, 64 * GROUP_WAVES);
  if (grid < 0) return hipErrorInvalidDevice;
  if (!P.ws || P.ws_lanes < 64 || P.ws_lanes % 64 != 0) return hipErrorInvalidValue;
  long long waves = P.ws_lanes / 64;
  if (q.max_blocks > 0 && q.max_blocks < waves) waves = q.max_blocks;
  const int most = (int)((waves + GROUP_WAVES - 1) / GROUP_WAVES);
  if (most < grid) grid = most;
  IO1D io{y, ysrc, rX, rXsrc};
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * GROUP_WAVES), 0, s, P, io, dt, q, st);
  return hipGetLastError();
}

template <class M, typename LU_T, bool CV>
hipError_t batched_group(const ReactParamsDev& P, double* y, const double* ysrc, double* rX, const double* rXsrc,
                         double dt, QueueArgs q, CellStats st, hipStream_t s) {
  using Tab = typename wave_tables<M>::type;
  if constexpr (!std::is_void<Tab>::value) {
    switch (P.adapt.group) {
      case 8:
        if constexpr (group_ok<M, 8>()) return launch_group<Tab, LU_T, 8, CV>(P, y, ysrc, rX, rXsrc, dt, q, st, s);
        break;
      case 4:
        if constexpr (group_ok<M, 16>()) return launch_group<Tab, LU_T, 16, CV>(P, y, ysrc, rX, rXsrc, dt, q, st, s);
        break;
      case 2:
        if constexpr (group_ok<M, 32>()) return launch_group<Tab, LU_T, 32, CV>(P, y, ysrc, rX, rXsrc, dt, q, st, s);
        break;
      case 1:
        if constexpr (group_ok<M, 64>()) return launch_group<Tab, LU_T, 64, CV>(P, y, ysrc, rX, rXsrc, dt, q, st, s);
        break;
      default:
        break;
    }
  }
  return hipErrorInvalidValue;
}

template <class M, int MODE>
hipError_t batched_1d_mode(const ReactParamsDev& P, double* y, const double* ysrc, double* rX, const double* rXsrc,
                           double dt, QueueArgs q, CellStats st, hipStream_t s) {
  using LU_T = typename std::conditional<MODE == MODE_BATCHED_MIXED, float, double>::type;
  constexpr bool CV = MODE == MODE_GROUP_CVODE;
  // a group of lanes per cell at every size (group_bdf.h): one cell per lane
  // measured 3.2 times as long on 64^3 drm19 cells and 16 to 115 times on
  // calls that do not fill the chip (figures there)
  return batched_group<M, LU_T, CV>(P, y, ysrc, rX, rXsrc, dt, q, st, s);
}

template <class T, int G, bool BOX>
hipError_t launch_group_rk64(const ReactParamsDev& P, const GroupIO& io, double dt, int ncells, CellStats st,
                             hipStream_t s) {
  auto k = group_rk64_kernel<T, G, BOX>;
  const int grid = resident_blocks(k, (long long)ncells * G, 64 * GROUP_WAVES);
  if (grid < 0) return hipErrorInvalidDevice;
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * GROUP_WAVES), 0, s, P, io, dt, ncells, st);
  return hipGetLastError();
}

template <class T, bool BOX>
hipError_t launch_group_bdf_fixed(const ReactParamsDev& P, const GroupIO& io, double dt, int ncells, CellStats st,
                                  hipStream_t s) {
  auto k = group_bdf_fixed_kernel<T, BOX>;
  const int grid = resident_blocks(k, (long long)ncells * 16, 64 * GROUP_WAVES);
  if (grid < 0) return hipErrorInvalidDevice;
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * GROUP_WAVES), 0, s, P, io, dt, ncells, st);
  return hipGetLastError();
}

template <class M>
hipError_t launch_group_fixed(int mode, const ReactParamsDev& P, double* y, const double* ysrc, double* rX,
                              const double* rXsrc, const BoxArgs* b, double dt, int ncells, int cells_per_wave,
                              CellStats st, hipStream_t s) {
  using Tab = typename wave_tables<M>::type;
  if constexpr (!std::is_void<Tab>::value) {
    GroupIO io{};
    io.f = IO1D{y, ysrc, rX, rXsrc};
    if (b) io.b = *b;
    if (mode == MODE_RK64) {
      if (ncells == 0) return hipSuccess;
      switch (cells_per_wave) {
        case 8:
          if constexpr (group_ok<M, 8>())
            return b ? launch_group_rk64<Tab, 8, true>(P, io, dt, ncells, st, s)
                     : launch_group_rk64<Tab, 8, false>(P, io, dt, ncells, st, s);
          break;
        case 4:
          if constexpr (group_ok<M, 16>())
            return b ? launch_group_rk64<Tab, 16, true>(P, io, dt, ncells, st, s)
                     : launch_group_rk64<Tab, 16, false>(P, io, dt, ncells, st, s);
          break;
        case 2:
          if constexpr (group_ok<M, 32>())
            return b ? launch_group_rk64<Tab, 32, true>(P, io, dt, ncells, st, s)
                     : launch_group_rk64<Tab, 32, false>(P, io, dt, ncells, st, s);
          break;
        case 1:
          if constexpr (group_ok<M, 64>())
            return b ? launch_group_rk64<Tab, 64, true>(P, io, dt, ncells, st, s)
                     : launch_group_rk64<Tab, 64, false>(P, io, dt, ncells, st, s);
          break;
        default:
          break;
      }
      return hipErrorInvalidValue;
    }
    if constexpr (group_fixed_fits<M>()) {
      if (mode == MODE_BDF) {
        if (ncells == 0) return hipSuccess;
        return b ? launch_group_bdf_fixed<Tab, true>(P, io, dt, ncells, st, s)
                 : launch_group_bdf_fixed<Tab, false>(P, io, dt, ncells, st, s);
      }
    }
  }
  return hipErrorNotSupported;
}

template <class M>
hipError_t launch_adjoint(const ReactParamsDev& P, const AdjointArgs& a, hipStream_t s) {
  using Tab = typename wave_tables<M>::type;
  // one equation per lane, at most two reactions per lane
  // (not QSS mechanisms: the adjoint differentiates plain mass-action rates)
  if constexpr (!std::is_void<Tab>::value && !has_qss<M>::value && M::NEQ <= 64 && M::NR <= 128) {
    auto k = wave_adjoint_kernel<Tab>;
    const int grid = resident_blocks(k, (long long)a.ncells * 64);
    if (grid < 0) return hipErrorInvalidDevice;
    hipLaunchKernelGGL(k, dim3(grid), dim3(64), 0, s, P, a);
    return hipGetLastError();
  } else {
    return hipErrorNotSupported;
  }
}

template <class M>
hipError_t launch_flatten(const FlatArgs& a, int unflatten, hipStream_t s) {
  const long long ncells = (long long)a.b.len[0] * a.b.len[1] * a.b.len[2];
  if (ncells <= 0) return hipSuccess;
  const int grid = (int)((ncells + 255) / 256 < 8192 ? (ncells + 255) / 256 : 8192);
  if (unflatten)
    hipLaunchKernelGGL(unflatten_kernel<M>, dim3(grid), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(flatten_kernel<M>, dim3(grid), dim3(256), 0, s, a);
  return hipGetLastError();
}

// productionRate (Mechanisms/drm19/mechanism.H:4421-5667), aJacobian
// (:10307-15357) or the net rates of progress q_f - q_r (comp_qfqr, :3600) of
// one cell per lane: sc[c*NS + k] (mol/m^3), T[c] (K); out[c*NS + k] = wdot_k
// (mol/m^3/s), out[c*n*n + ...] = the column-major Jacobian of cell c, or
// out[c*NR + j] = q_j (mol/m^3/s), written in place in the output array.
//
// One kernel per function: with the four in one, all took the Jacobian's 512
// registers, one wave per SIMD (drm19 rates: 203, two).  WHOLE: the rates' flat
// arrays pass through LDS in whole lines (a row is 65 cells: no bank conflicts
// either way), for calls that give every SIMD a wave, where a wave's cells take
// little LDS; below that a call waits for one wave's latency, and the way through
// LDS is part of it.  Bound by the FP64 vector issue: drm19 is 7800 vector
// instructions per wave, 57 us at the full rate for 262144 cells; a call of them
// 99.1 -> 86.6 us (65536 cells 43.7 -> 43.3; 8192 cells 36.7 -> 39.2 through LDS).
template <class M, int WHAT, bool WHOLE>
__global__ void __launch_bounds__(64) mech_eval_kernel(const double* __restrict__ sc, const double* __restrict__ T,
                                                       int ncells, double* out) {
  constexpr int NS = M::NS;
  const int l = threadIdx.x, c0 = blockIdx.x * 64, nc = min(64, ncells - c0);
  double s[NS];
  if constexpr (WHOLE) {
    __shared__ double row[NS * 65];
    const double* const from = sc + (long long)c0 * NS;
    for (int i = l; i < nc * NS; i += 64) row[i % NS * 65 + i / NS] = from[i];
    __syncthreads();
    const int m = min(l, nc - 1);  // lanes past the end repeat the last cell
    double w[NS];
    for (int k = 0; k < NS; ++k) s[k] = row[k * 65 + m];
    M::production_rate(w, s, T[c0 + m]);
    __syncthreads();
    for (int k = 0; k < NS; ++k) row[k * 65 + l] = w[k];
    __syncthreads();
    double* const to = out + (long long)c0 * NS;
    for (int i = l; i < nc * NS; i += 64) to[i] = row[i % NS * 65 + i / NS];
  } else {
    if (l >= nc) return;
    const long long c = c0 + l;
    for (int k = 0; k < NS; ++k) s[k] = sc[c * NS + k];
    const double Tv = T[c];
    if constexpr (WHAT == 0) {
      double w[NS];
      M::production_rate(w, s, Tv);
      for (int k = 0; k < NS; ++k) out[c * NS + k] = w[k];
    } else if constexpr (WHAT == 3) {
      M::progress_rates(out + c * M::NR, s, Tv);  // written in place: NR can be large
    } else {
      M::template jacobian<WHAT - 1>(out + c * M::NEQ * M::NEQ, s, Tv);
    }
  }
}

template <class M>
hipError_t launch_mech_eval(int what, const double* sc, const double* T, int ncells, double* out, hipStream_t s) {
  if (what < 0 || what > 3) return hipErrorInvalidValue;
  if (ncells <= 0) return hipSuccess;
  constexpr int fills = 64 * 4 * 256;  // a wave for each of the 4 SIMDs of 256 compute units
  auto k = what == 0   ? mech_eval_kernel<M, 0, false>
           : what == 1 ? mech_eval_kernel<M, 1, false>
           : what == 2 ? mech_eval_kernel<M, 2, false>
                       : mech_eval_kernel<M, 3, false>;
  if constexpr (M::NS <= 32)
    if (what == 0 && ncells >= fills) k = mech_eval_kernel<M, 0, true>;
  hipLaunchKernelGGL(k, dim3((ncells + 63) / 64), dim3(64), 0, s, sc, T, ncells, out);
  return hipGetLastError();
}

}  // namespace ppc

#define PPC_INSTANTIATE_FLATTEN(TYPE, MODE)                                                        \
  namespace ppc {                                                                                 \
  template hipError_t launch_flatten<TYPE>(const FlatArgs&, int, hipStream_t);                   \
  template hipError_t launch_mech_eval<TYPE>(int, const double*, const double*, int, double*,     \
                                             hipStream_t);                                        \
  }

#define PPC_INSTANTIATE_GFIXED(TYPE, MODE)                                                             \
  namespace ppc {                                                                                    \
  template hipError_t launch_group_fixed<TYPE>(int, const ReactParamsDev&, double*, const double*, double*, \
                                               const double*, const BoxArgs*, double, int, int, CellStats,  \
                                               hipStream_t);                                          \
  }

#define PPC_INSTANTIATE_ADJOINT(TYPE, MODE)                                                           \
  namespace ppc {                                                                                    \
  template hipError_t launch_adjoint<TYPE>(const ReactParamsDev&, const AdjointArgs&, hipStream_t);  \
  }

#define PPC_INSTANTIATE_MODE(TYPE, MODE)                                                              \
  namespace ppc {                                                                                    \
  template hipError_t launch_1d_mode<TYPE, MODE>(const ReactParamsDev&, double*, const double*, \
                                                       double*, const double*, double, int, CellStats, \
                                                       int, hipStream_t);                             \
  template hipError_t launch_box_mode<TYPE, MODE>(const ReactParamsDev&, const BoxArgs&, double, \
                                                        int, CellStats, int, hipStream_t);            \
  }

#define PPC_INSTANTIATE_BATCHED(TYPE, MODE)                                                             \
  namespace ppc {                                                                                      \
  template hipError_t batched_1d_mode<TYPE, MODE>(const ReactParamsDev&, double*, const double*,  \
                                                        double*, const double*, double, QueueArgs,      \
                                                        CellStats, hipStream_t);  \
  }
