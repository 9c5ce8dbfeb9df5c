// Generated by pelephysics_amd/build.py: drm19 x cvode kernels.
#include "../mech/drm19.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_BATCHED(ppc::mech::drm19, ppc::MODE_GROUP_CVODE)
