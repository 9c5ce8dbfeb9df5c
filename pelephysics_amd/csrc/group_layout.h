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
  static constexpr int AREA = ((S_RAW + 3) / 8) * 8 + 4;
  // The wave's Jacobian area overlays its groups' areas: 5 species vectors and,
  // where n is small enough, the n x n accumulator.
  // (QSS mechanisms: each group works on its own cell's Jacobian, in the
  // workspace, with JVEC doubles of its area.)
  static constexpr bool JLDS = n <= 32 && NQ == 0;
  static constexpr int J_AT = (5 * NP + 1) & ~1;
  static constexpr int JVEC = NQ > 0 ? 6 * NX + NROW : 0;
  // Jacobian accumulators in the workspace (doubles): n x n (JSQ) of the wave,
  // or of each group with the QSS terms after it (JSTRIDE); of a wave
  static constexpr int JSQ = (n * n + 1) & ~1;
  static constexpr int JSTRIDE = NQ > 0 ? (JSQ + NQ * NS + 2 * T::NQR + 1) & ~1 : JSQ;
  static constexpr int JSPACE = NQ > 0 ? NG * JSTRIDE : JSTRIDE;
  static constexpr int WAREA = (cmax(NG * AREA, J_AT + (JLDS ? n * n : 0)) + 3) & ~3;
  // vectors of the step that stay in LDS (group_bdf_kernel), per wave
  static constexpr int LVEC = 4 * 64 * EPL;

  // LDS of a block of the largest group kernel with G lanes per cell (the
  // adaptive BDF's; ReactorRK64's has the tables and the areas only)
  static constexpr long long lds_bytes() {
    return (long long)sizeof(typename T::Packed) + 8LL * GROUP_WAVES * (WAREA + LVEC);
  }
  static constexpr bool fits() { return JVEC <= AREA && lds_bytes() <= LDS_BYTES; }
};

}  // namespace ppc
