// Generated by pelephysics_amd/build.py: drm19_table x gfixed kernels.
#include "../tab/drm19.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::TabMech<ppc::tab::drm19>, ppc::MODE_BDF)
