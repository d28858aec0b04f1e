// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "../qf_fuse.h"
#include "../qf_launch.h"
#include "coop_C2221.h"
#include "coop_C2222.h"
#include "coop_C3022.h"
#include "coop_C3121.h"
#include "coop_C3122.h"
#include "coop_C3130.h"
#include "coop_C3131.h"
#include "coop_C3211.h"
#include "coop_C3221.h"
#include "coop_C3222.h"
#include "coop_C3230.h"
#include "coop_C3231.h"
#include "coop_C3311.h"
#include "coop_C3320.h"
#include "coop_C3321.h"
#include "coop_C3330.h"

namespace qf {

void launch_fuse_coop_large(const FusedBlock* list, int n, const TileGroup* g, const Task* t, const PairBlock* b,
    const MolDesc* m, int os, int waves, size_t lds, double* gscratch, LaunchTo& q)
{
    (void)g;
    (void)waves;
    const int grid = n;
    if (os)
        q((fused_coop_kernel<true, 6650,
        FuseMember<84, C2221Coop>,
        FuseMember<85, C2222Coop>,
        FuseMember<101, C3022Coop>,
        FuseMember<116, C3121Coop>,
        FuseMember<117, C3122Coop>,
        FuseMember<118, C3130Coop>,
        FuseMember<119, C3131Coop>,
        FuseMember<130, C3211Coop>,
        FuseMember<132, C3221Coop>,
        FuseMember<133, C3222Coop>,
        FuseMember<134, C3230Coop>,
        FuseMember<135, C3231Coop>,
        FuseMember<146, C3311Coop>,
        FuseMember<147, C3320Coop>,
        FuseMember<148, C3321Coop>,
        FuseMember<150, C3330Coop>>),
          dim3(grid), dim3(WAVE), lds, list, n, t, b, m, gscratch);
    else
        q((fused_coop_kernel<false, 6650,
        FuseMember<84, C2221Coop>,
        FuseMember<85, C2222Coop>,
        FuseMember<101, C3022Coop>,
        FuseMember<116, C3121Coop>,
        FuseMember<117, C3122Coop>,
        FuseMember<118, C3130Coop>,
        FuseMember<119, C3131Coop>,
        FuseMember<130, C3211Coop>,
        FuseMember<132, C3221Coop>,
        FuseMember<133, C3222Coop>,
        FuseMember<134, C3230Coop>,
        FuseMember<135, C3231Coop>,
        FuseMember<146, C3311Coop>,
        FuseMember<147, C3320Coop>,
        FuseMember<148, C3321Coop>,
        FuseMember<150, C3330Coop>>),
          dim3(grid), dim3(WAVE), lds, list, n, t, b, m, gscratch);
}

}  // namespace qf
