// Generated by pelephysics_amd/build.py: LuEthylene_qss x cvode kernels.
#include "../tab/LuEthylene_qss.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_BATCHED(ppc::TabMech<ppc::tab::LuEthylene_qss>, ppc::MODE_GROUP_CVODE)
