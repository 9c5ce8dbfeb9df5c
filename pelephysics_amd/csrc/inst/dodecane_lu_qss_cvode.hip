// Generated by pelephysics_amd/build.py: dodecane_lu_qss x cvode kernels.
#include "../tab/dodecane_lu_qss.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_BATCHED(ppc::TabMech<ppc::tab::dodecane_lu_qss>, ppc::MODE_GROUP_CVODE)
