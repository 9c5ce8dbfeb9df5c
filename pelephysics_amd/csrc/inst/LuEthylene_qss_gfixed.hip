// Generated by pelephysics_amd/build.py: LuEthylene_qss x gfixed kernels.
#include "../tab/LuEthylene_qss.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::TabMech<ppc::tab::LuEthylene_qss>, ppc::MODE_BDF)
