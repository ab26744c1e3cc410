/* the per-bin likelihood kernels of IMRPhenomD, mixed-precision evaluation: every tiling class (gwh_tiles.h) */
#include "gwh_tiles.h"

template void gwh_launch_tiles<GWH_IMRPHENOMD, GWH_MIXED>(int, int, long long, hipStream_t, const WorkMap &, const EventDesc *,
                                      const InstCoef *, double *, const int *, const int *);
template void gwh_launch_worklist<GWH_IMRPHENOMD, GWH_MIXED>(int, long long, const int2 *, hipStream_t, const WorkMap &, const EventDesc *,
                                      const InstCoef *, double *, const int *);
template int gwh_tiles_load<GWH_IMRPHENOMD, GWH_MIXED>();
