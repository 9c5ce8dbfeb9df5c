// Generated by pelephysics_amd/build.py: heptane_lu_88sk x gfixed kernels.
#include "../tab/heptane_lu_88sk.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::TabMech<ppc::tab::heptane_lu_88sk>, ppc::MODE_BDF)
