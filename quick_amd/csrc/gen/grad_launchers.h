// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#pragma once
#include <hip/hip_runtime.h>
#include "../qf_launch.h"
#include "../qf_types.h"

namespace qf {

using GradLaunch = void (*)(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);

void launch_grad_C0000(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C0000(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C1000(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C1000(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C1010(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C1010(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C1100(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C1100(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C1110(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C1110(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C1111(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C1111(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2000(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2000(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2010(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2010(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2011(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2011(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2020(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2020(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2100(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2100(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2110(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2110(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2111(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2111(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2120(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2120(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2121(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2200(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2200(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2210(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_lane_C2210(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2211(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2220(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2221(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);
void launch_grad_C2222(const Task*, int, const PairBlock*, const MolDesc*, int, size_t, double*, int, LaunchTo&);

// nullptr: no gradient kernel for the class (f shells)
inline GradLaunch grad_launcher(int cb, int ck)
{
    if (cb == 0 && ck == 0) return launch_grad_C0000;
    if (cb == 1 && ck == 0) return launch_grad_C1000;
    if (cb == 1 && ck == 1) return launch_grad_C1010;
    if (cb == 2 && ck == 0) return launch_grad_C1100;
    if (cb == 2 && ck == 1) return launch_grad_C1110;
    if (cb == 2 && ck == 2) return launch_grad_C1111;
    if (cb == 3 && ck == 0) return launch_grad_C2000;
    if (cb == 3 && ck == 1) return launch_grad_C2010;
    if (cb == 3 && ck == 2) return launch_grad_C2011;
    if (cb == 3 && ck == 3) return launch_grad_C2020;
    if (cb == 4 && ck == 0) return launch_grad_C2100;
    if (cb == 4 && ck == 1) return launch_grad_C2110;
    if (cb == 4 && ck == 2) return launch_grad_C2111;
    if (cb == 4 && ck == 3) return launch_grad_C2120;
    if (cb == 4 && ck == 4) return launch_grad_C2121;
    if (cb == 5 && ck == 0) return launch_grad_C2200;
    if (cb == 5 && ck == 1) return launch_grad_C2210;
    if (cb == 5 && ck == 2) return launch_grad_C2211;
    if (cb == 5 && ck == 3) return launch_grad_C2220;
    if (cb == 5 && ck == 4) return launch_grad_C2221;
    if (cb == 5 && ck == 5) return launch_grad_C2222;
    return nullptr;
}

// per-lane gradient kernels (nullptr: the class has none)
inline GradLaunch grad_lane_launcher(int cb, int ck)
{
    if (cb == 0 && ck == 0) return launch_grad_lane_C0000;
    if (cb == 1 && ck == 0) return launch_grad_lane_C1000;
    if (cb == 1 && ck == 1) return launch_grad_lane_C1010;
    if (cb == 2 && ck == 0) return launch_grad_lane_C1100;
    if (cb == 2 && ck == 1) return launch_grad_lane_C1110;
    if (cb == 2 && ck == 2) return launch_grad_lane_C1111;
    if (cb == 3 && ck == 0) return launch_grad_lane_C2000;
    if (cb == 3 && ck == 1) return launch_grad_lane_C2010;
    if (cb == 3 && ck == 2) return launch_grad_lane_C2011;
    if (cb == 3 && ck == 3) return launch_grad_lane_C2020;
    if (cb == 4 && ck == 0) return launch_grad_lane_C2100;
    if (cb == 4 && ck == 1) return launch_grad_lane_C2110;
    if (cb == 4 && ck == 2) return launch_grad_lane_C2111;
    if (cb == 4 && ck == 3) return launch_grad_lane_C2120;
    if (cb == 5 && ck == 0) return launch_grad_lane_C2200;
    if (cb == 5 && ck == 1) return launch_grad_lane_C2210;
    return nullptr;
}

// doubles per workgroup slice of the global slot buffer (0: LDS slots)
inline int grad_global_doubles(int cb, int ck)
{
    if (cb == 5 && ck == 4) return 12720;
    if (cb == 5 && ck == 5) return 25290;
    return 0;
}

// LDS doubles of the node-program slots (0 when they are global)
inline int grad_lds_doubles(int cb, int ck)
{
    if (cb == 0 && ck == 0) return 75;
    if (cb == 1 && ck == 0) return 127;
    if (cb == 1 && ck == 1) return 280;
    if (cb == 2 && ck == 0) return 255;
    if (cb == 2 && ck == 1) return 623;
    if (cb == 2 && ck == 2) return 1725;
    if (cb == 3 && ck == 0) return 205;
    if (cb == 3 && ck == 1) return 495;
    if (cb == 3 && ck == 2) return 1232;
    if (cb == 3 && ck == 3) return 951;
    if (cb == 4 && ck == 0) return 425;
    if (cb == 4 && ck == 1) return 1077;
    if (cb == 4 && ck == 2) return 3038;
    if (cb == 4 && ck == 3) return 2083;
    if (cb == 4 && ck == 4) return 5661;
    if (cb == 5 && ck == 0) return 874;
    if (cb == 5 && ck == 1) return 2222;
    if (cb == 5 && ck == 2) return 6582;
    if (cb == 5 && ck == 3) return 4244;
    return 0;
}

// Algorithmic FLOPs of the gradient: per primitive quartet (Boys, VRR,
// accumulation) and per contracted quartet (HRR blocks, weights, nine derivatives).
inline double grad_class_flops(int cb, int ck, unsigned long long nq, unsigned long long np)
{
    if (cb == 0 && ck == 0) return double(np) * 100.0 + double(nq) * 52.0;
    if (cb == 1 && ck == 0) return double(np) * 194.0 + double(nq) * 156.0;
    if (cb == 1 && ck == 1) return double(np) * 535.0 + double(nq) * 468.0;
    if (cb == 2 && ck == 0) return double(np) * 433.0 + double(nq) * 592.0;
    if (cb == 2 && ck == 1) return double(np) * 1280.0 + double(nq) * 1740.0;
    if (cb == 2 && ck == 2) return double(np) * 3408.0 + double(nq) * 6354.0;
    if (cb == 3 && ck == 0) return double(np) * 362.0 + double(nq) * 312.0;
    if (cb == 3 && ck == 1) return double(np) * 1073.0 + double(nq) * 936.0;
    if (cb == 3 && ck == 2) return double(np) * 2904.0 + double(nq) * 3582.0;
    if (cb == 3 && ck == 3) return double(np) * 2646.0 + double(nq) * 1872.0;
    if (cb == 4 && ck == 0) return double(np) * 771.0 + double(nq) * 1172.0;
    if (cb == 4 && ck == 1) return double(np) * 2321.0 + double(nq) * 3444.0;
    if (cb == 4 && ck == 2) return double(np) * 6159.0 + double(nq) * 12282.0;
    if (cb == 4 && ck == 3) return double(np) * 5581.0 + double(nq) * 6852.0;
    if (cb == 4 && ck == 4) return double(np) * 12486.0 + double(nq) * 24360.0;
    if (cb == 5 && ck == 0) return double(np) * 1410.0 + double(nq) * 2942.0;
    if (cb == 5 && ck == 1) return double(np) * 4224.0 + double(nq) * 8510.0;
    if (cb == 5 && ck == 2) return double(np) * 11025.0 + double(nq) * 29226.0;
    if (cb == 5 && ck == 3) return double(np) * 9985.0 + double(nq) * 16862.0;
    if (cb == 5 && ck == 4) return double(np) * 22082.0 + double(nq) * 57792.0;
    if (cb == 5 && ck == 5) return double(np) * 41631.0 + double(nq) * 132726.0;
    return 0.0;
}

// (list, workgroups, tasks, blocks, mols, slot doubles in LDS, gradient doubles, global slots, target)
using GradFuseLaunch = void (*)(const FusedBlock*, int, const Task*, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fuse_grad_lane3(const FusedBlock*, int, const Task*, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fuse_grad_lane2(const FusedBlock*, int, const Task*, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fuse_grad_lane1(const FusedBlock*, int, const Task*, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fuse_grad_coop(const FusedBlock*, int, const Task*, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fuse_grad_coop_global(const FusedBlock*, int, const Task*, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);

struct GradFuseKernel {
    GradFuseLaunch launch;
    bool coop;          // wave-per-quartet classes
    int global;         // doubles of a workgroup's slice of the global slot buffer (0: slots in LDS)
};
constexpr int kGradFuseKernels = 5;
inline GradFuseKernel grad_fuse_kernel(int k)
{
    constexpr GradFuseKernel all[kGradFuseKernels] = {
        {launch_fuse_grad_lane3, false, 0},
        {launch_fuse_grad_lane2, false, 0},
        {launch_fuse_grad_lane1, false, 0},
        {launch_fuse_grad_coop, true, 0},
        {launch_fuse_grad_coop_global, true, 25290},
    };
    return all[k];
}

// the kernel that runs a class's gradient beside others (-1: none)
inline int grad_fuse_bucket(int cb, int ck)
{
    switch (cb * 16 + ck) {
    case 0: return 0;
    case 16: return 0;
    case 17: return 1;
    case 32: return 1;
    case 48: return 1;
    case 64: return 1;
    case 33: return 2;
    case 34: return 2;
    case 49: return 2;
    case 50: return 2;
    case 51: return 2;
    case 65: return 2;
    case 66: return 2;
    case 67: return 2;
    case 80: return 2;
    case 81: return 2;
    case 68: return 3;
    case 82: return 3;
    case 83: return 3;
    case 84: return 4;
    case 85: return 4;
    }
    return -1;
}

}  // namespace qf
