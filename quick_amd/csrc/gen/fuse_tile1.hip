// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#include "../qf_fuse.h"
#include "../qf_launch.h"
#include "C1111.h"
#include "C2011.h"
#include "C2020.h"
#include "C2110.h"
#include "C2120.h"
#include "C2210.h"
#include "C3011.h"
#include "C3020.h"
#include "C3110.h"
#include "C3200.h"

namespace qf {

void launch_fuse_tile1(const FusedBlock* list, int n, const TileGroup* g, const Task* t, const PairBlock* b,
    const MolDesc* m, int os, int waves, size_t lds, double* gscratch, LaunchTo& q)
{
    (void)gscratch;
    if (os)
        q((fused_tile_kernel<1, true,
        FuseMember<34, C1111>,
        FuseMember<50, C2011>,
        FuseMember<51, C2020>,
        FuseMember<65, C2110>,
        FuseMember<67, C2120>,
        FuseMember<81, C2210>,
        FuseMember<98, C3011>,
        FuseMember<99, C3020>,
        FuseMember<113, C3110>,
        FuseMember<128, C3200>>),
          dim3(n), dim3(waves * WAVE), lds, list, g, t, b, m);
    else
        q((fused_tile_kernel<1, false,
        FuseMember<34, C1111>,
        FuseMember<50, C2011>,
        FuseMember<51, C2020>,
        FuseMember<65, C2110>,
        FuseMember<67, C2120>,
        FuseMember<81, C2210>,
        FuseMember<98, C3011>,
        FuseMember<99, C3020>,
        FuseMember<113, C3110>,
        FuseMember<128, C3200>>),
          dim3(n), dim3(waves * WAVE), lds, list, g, t, b, m);
}

}  // namespace qf
