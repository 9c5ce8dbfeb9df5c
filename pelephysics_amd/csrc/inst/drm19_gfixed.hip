// Generated by pelephysics_amd/build.py: drm19 x gfixed kernels.
#include "../mech/drm19.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::mech::drm19, ppc::MODE_BDF)
