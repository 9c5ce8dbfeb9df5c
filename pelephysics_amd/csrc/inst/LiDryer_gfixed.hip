// Generated by pelephysics_amd/build.py: LiDryer x gfixed kernels.
#include "../mech/LiDryer.h"
#include "../launch_impl.h"
PPC_INSTANTIATE_GFIXED(ppc::mech::LiDryer, ppc::MODE_BDF)
