// Generated by pelephysics_amd/build.py: CH4_lean_qss x gfixed kernels.
#include "../tab/CH4_lean_qss.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::TabMech<ppc::tab::CH4_lean_qss>, ppc::MODE_BDF)
