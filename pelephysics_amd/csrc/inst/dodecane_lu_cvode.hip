// Generated by pelephysics_amd/build.py: dodecane_lu x cvode kernels.
#include "../tab/dodecane_lu.h"
#include "../chem_table.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_BATCHED(ppc::TabMech<ppc::tab::dodecane_lu>, ppc::MODE_GROUP_CVODE)
