// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "../qf_fuse.h"
#include "../qf_launch.h"
#include "coop_C1111.h"
#include "coop_C2011.h"
#include "coop_C2020.h"
#include "coop_C2111.h"
#include "coop_C2120.h"
#include "coop_C2121.h"
#include "coop_C2200.h"
#include "coop_C2210.h"
#include "coop_C2211.h"
#include "coop_C2220.h"
#include "coop_C3000.h"
#include "coop_C3010.h"
#include "coop_C3011.h"
#include "coop_C3020.h"
#include "coop_C3021.h"
#include "coop_C3030.h"
#include "coop_C3100.h"
#include "coop_C3110.h"
#include "coop_C3111.h"
#include "coop_C3120.h"
#include "coop_C3200.h"
#include "coop_C3210.h"
#include "coop_C3220.h"
#include "coop_C3300.h"
#include "coop_C3310.h"

namespace qf {

void launch_fuse_coop_small(const FusedBlock* list, int n, const TileGroup* g, const Task* t, const PairBlock* b,
    const MolDesc* m, int os, int waves, size_t lds, double* gscratch, LaunchTo& q)
{
    (void)g;
    (void)waves;
    const int grid = n;
    if (os)
        q((fused_coop_kernel<true, 1270,
        FuseMember<34, C1111Coop>,
        FuseMember<50, C2011Coop>,
        FuseMember<51, C2020Coop>,
        FuseMember<66, C2111Coop>,
        FuseMember<67, C2120Coop>,
        FuseMember<68, C2121Coop>,
        FuseMember<80, C2200Coop>,
        FuseMember<81, C2210Coop>,
        FuseMember<82, C2211Coop>,
        FuseMember<83, C2220Coop>,
        FuseMember<96, C3000Coop>,
        FuseMember<97, C3010Coop>,
        FuseMember<98, C3011Coop>,
        FuseMember<99, C3020Coop>,
        FuseMember<100, C3021Coop>,
        FuseMember<102, C3030Coop>,
        FuseMember<112, C3100Coop>,
        FuseMember<113, C3110Coop>,
        FuseMember<114, C3111Coop>,
        FuseMember<115, C3120Coop>,
        FuseMember<128, C3200Coop>,
        FuseMember<129, C3210Coop>,
        FuseMember<131, C3220Coop>,
        FuseMember<144, C3300Coop>,
        FuseMember<145, C3310Coop>>),
          dim3(grid), dim3(WAVE), lds, list, n, t, b, m, gscratch);
    else
        q((fused_coop_kernel<false, 1270,
        FuseMember<34, C1111Coop>,
        FuseMember<50, C2011Coop>,
        FuseMember<51, C2020Coop>,
        FuseMember<66, C2111Coop>,
        FuseMember<67, C2120Coop>,
        FuseMember<68, C2121Coop>,
        FuseMember<80, C2200Coop>,
        FuseMember<81, C2210Coop>,
        FuseMember<82, C2211Coop>,
        FuseMember<83, C2220Coop>,
        FuseMember<96, C3000Coop>,
        FuseMember<97, C3010Coop>,
        FuseMember<98, C3011Coop>,
        FuseMember<99, C3020Coop>,
        FuseMember<100, C3021Coop>,
        FuseMember<102, C3030Coop>,
        FuseMember<112, C3100Coop>,
        FuseMember<113, C3110Coop>,
        FuseMember<114, C3111Coop>,
        FuseMember<115, C3120Coop>,
        FuseMember<128, C3200Coop>,
        FuseMember<129, C3210Coop>,
        FuseMember<131, C3220Coop>,
        FuseMember<144, C3300Coop>,
        FuseMember<145, C3310Coop>>),
          dim3(grid), dim3(WAVE), lds, list, n, t, b, m, gscratch);
}

}  // namespace qf
