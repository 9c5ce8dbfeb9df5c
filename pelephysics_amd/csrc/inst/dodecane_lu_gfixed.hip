// Generated by pelephysics_amd/build.py: dodecane_lu x gfixed kernels.
#include "../tab/dodecane_lu.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::TabMech<ppc::tab::dodecane_lu>, ppc::MODE_BDF)
