// Launchers of the run-time sized transforms (agd_general.hip): classes with
// p0 == 0 and hb > 0.
#pragma once

#include "agd_gpu.h"

namespace agdgen {
// spatial transforms of the class's tasks: mode -1 the forward of X into U,
// else as agdg_adj_spatial
int spatial_general(AgdDev const *g, AgdClass const &c, float2 *X, float alpha, float lamb,
                    int mode, int fuse);
// time transforms of the class's blocks [first, first + n)
int fwd_time_general(AgdDev const *g, AgdClass const &c, int first, int n);
int adj_time_general(AgdDev const *g, AgdClass const &c, int first, int n, float const *Tin,
                     int plain);
}  // namespace agdgen
