// Generated by pelephysics_amd/build.py: LiDryer x cvode kernels.
#include "../mech/LiDryer.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_BATCHED(ppc::mech::LiDryer, ppc::MODE_GROUP_CVODE)
