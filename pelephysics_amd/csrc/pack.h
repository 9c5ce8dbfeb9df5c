// Records of the packed mechanism tables (tab/<name>.h, struct Packed), which
// the group kernels copy to LDS as they stand.
#pragma once
#include "ppc_common.h"

namespace ppc {

// regularisation of the QSS balances (comp_sc_qss epsilon of the reference's
// generated QSS mechanisms)
constexpr double QSS_EPS = 1e-12;

namespace tab {

// NASA7 coefficients below and above tmid, and the inverse molecular weight
struct alignas(16) PackSp {
  double lo[7], tmid, hi[7], imw;
};
// rate A T^b exp(-E/T), reactant and product species (NX: unused), power of
// refC in the reverse rate, flags (1: reversible, 2: forward direction removed)
struct alignas(16) PackRx {
  double A, b, E;
  unsigned char r[3], p[3];
  signed char delta;
  unsigned char flags;
};
// low-pressure rate, Troe a, T3, T1, T2, and 1 where T2 is given
struct alignas(16) PackFo {
  double A, b, E, tA, t3, t1, t2, has2;
};
// eight terms of a species' net stoichiometry: reaction | (coefficient + 8) << 12
struct alignas(16) PackCh {
  unsigned short e[8];
};
// first entry and count of a reaction's third-body enhancements
struct PackEff {
  unsigned short e0, n;
};

}  // namespace tab
}  // namespace ppc
