// Generated by pelephysics_amd/build.py: dodecane_lu_qss x gfixed kernels.
#include "../tab/dodecane_lu_qss.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::TabMech<ppc::tab::dodecane_lu_qss>, ppc::MODE_BDF)
