// Generated by pelephysics_amd/build.py: CH4_lean_qss x cvode kernels.
#include "../tab/CH4_lean_qss.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_BATCHED(ppc::TabMech<ppc::tab::CH4_lean_qss>, ppc::MODE_GROUP_CVODE)
