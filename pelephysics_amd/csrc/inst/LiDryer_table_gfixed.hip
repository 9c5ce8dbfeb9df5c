// Generated by pelephysics_amd/build.py: LiDryer_table x gfixed kernels.
#include "../tab/LiDryer.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::TabMech<ppc::tab::LiDryer>, ppc::MODE_BDF)
