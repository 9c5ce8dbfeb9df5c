// Layout of the group kernels' LDS areas (group_bdf.h, group_fixed.h), and the
// LDS that a block of them takes: mechanisms whose tables and areas do not fit
// a compute unit have no group kernels (group_ok in lane_ws.h).
#pragma once
#include <type_traits>

namespace ppc {

// Waves per block of the group kernels: they share one copy of the tables.
constexpr int GROUP_WAVES = 4;

constexpr long long LDS_BYTES = 160 * 1024;  // of a gfx950 compute unit

template <class T, int G>
struct GroupLayout {
  static constexpr int NS = T::NS, NR = T::NR, n = T::NEQ, NX = T::NX, NCH = T::NCH;
  static constexpr int NG = 64 / G;
  static constexpr int EPL = (n + G - 1) / G;    // equation slots per lane
  static constexpr int SPL = (NS + G - 1) / G;   // species slots per lane
  static constexpr int SPX = (NX + G - 1) / G;   // with the QSS species
  static constexpr int NP = (n + 1) & ~1;        // vectors of n, 16-byte aligned

  // A group's LDS area (doubles): concentrations with exp(-g/RT) and
  // c exp(g/RT) of every species, an unused place's ones after them (later
  // the chunk sums), then the rates of progress with a zero after them (later
  // the vectors of the Newton solve).  Its size is 4 modulo 8 doubles, so that
  // the groups' broadcasts fall into different banks.
  static constexpr int cmax(int a, int b) { return a > b ? a : b; }
  static constexpr int S_CA = 0, S_B = 2 * (NX + 1);
  static constexpr int NQ = T::NQ, NROW = NQ > 0 ? T::NSLOT + NQ : 0;  // QSS balances: entries and right-hand sides
  static constexpr int S_Q = (cmax(cmax(3 * (NX + 1), NCH), 2 * (NX + 1) + NROW) + 1) & ~1;
  static constexpr int NRATE = NQ > 0 ? 2 * NR + 1 : NR + 1;  // QSS: forward and reverse rates apart
  static constexpr int S_RAW = S_Q + cmax(NRATE, 3 * NP);
  static constexpr int padded(int a) { return ((a + 3) / 8) * 8 + 4; }
  static constexpr int AREA_RHS = padded(S_RAW);  // of a kernel without Jacobians

  // A Jacobian in LDS (doubles): its species vectors (QSS mechanisms: with the
  // balances), then the n x n accumulator (JSQ), for QSS mechanisms with the
  // derivatives of the balances and of the rates (NQ x NS each) after it.
  static constexpr int JVEC = NQ > 0 ? 6 * NX + NROW : 5 * NP;
  static constexpr int J_AT = (JVEC + 1) & ~1;
  static constexpr int JSQ = (n * n + 1) & ~1;
  static constexpr int JSTRIDE = (JSQ + 2 * NQ * NS + 1) & ~1;
  static constexpr int JLEN = J_AT + JSTRIDE;
  // vectors of the step that stay in LDS (group_bdf_kernel), per wave
  static constexpr int LVEC = 4 * 64 * EPL;
  static constexpr int own_area() { return padded(cmax(S_RAW, JLEN)); }
  static constexpr int wave_area() { return (cmax(NG * AREA_RHS, JLEN) + 3) & ~3; }
  static constexpr long long bytes(int area) {
    return (long long)sizeof(typename T::Packed) + 8LL * GROUP_WAVES * (area + LVEC);
  }
  // Who works on the Jacobians of a wave's cells, and where.  Every group on its
  // own cell's (JOWN), in its own area: the groups of a wave ask at the same time
  // when their cells start, which is most of a call of few steps per cell.  Or the
  // whole wave on one cell's after the other's, over all its groups' areas.  In LDS
  // (JLDS) where two blocks fit a compute unit, i.e. two waves per SIMD; else in
  // the workspace, by the groups for QSS mechanisms and by the wave for the others.
  // Without QSS species a group's own takes NR / G rounds of reactions, the wave NG
  // times NR / 64: its own where that is at most half.  Measured, calls of one step
  // per cell: LiDryer 262144 cells, 8 lanes, one cell after the other 5.7 ms, each
  // its own 1.3; CH4_lean_qss 262144 cells and LuEthylene_qss 65536, by the group in
  // the workspace 34.3 and 37.6 ms, in LDS by the group and by the wave 5.2 and 5.9.
  static constexpr bool two_blocks(int area) { return bytes(area) <= LDS_BYTES / 2; }
  static constexpr bool own_fits() { return n <= 32 && two_blocks(NG * own_area()); }
  static constexpr bool wave_fits() { return n <= 32 && (NQ == 0 || two_blocks(wave_area())); }
  static constexpr bool JOWN = NQ > 0 ? own_fits() || !wave_fits()
                                      : own_fits() && 2 * ((NR + G - 1) / G) <= NG * ((NR + 63) / 64);
  static constexpr bool JLDS = JOWN ? own_fits() : wave_fits();
  static constexpr int AREA = JOWN && JLDS ? own_area() : AREA_RHS;
  static constexpr int WAREA = JOWN || !JLDS ? (cmax(NG * AREA, JOWN ? 0 : J_AT) + 3) & ~3 : wave_area();
  // Jacobian accumulators in the workspace (doubles) of a wave
  static constexpr int JSPACE = NQ > 0 ? NG * JSTRIDE : JSTRIDE;

  // LDS of a block of the largest group kernel with G lanes per cell (the
  // adaptive BDF's; ReactorRK64's has the tables and the areas only)
  static constexpr bool fits() { return (!JOWN || JVEC <= AREA) && bytes(WAREA) <= LDS_BYTES; }
};

}  // namespace ppc
