// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#pragma once
#include <hip/hip_runtime.h>
#include "../qf_launch.h"
#include "../qf_types.h"

namespace qf {

// returns nonzero when the launch is refused (FP32 on the direct kernel)
// (tasks, ntasks, blocks, mols, fp32, os, grid, target)
using FockLaunch = int (*)(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
// (groups, ngroups, tasks, blocks, mols, fp32, os, waves, lds bytes, grid, target)
using FockTileLaunch = void (*)(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
// (tasks, ntasks, blocks, mols, os, grid, global slots, target)
using FockCoopLaunch = void (*)(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
using SchwarzLaunch = void (*)(PairBlock, double*, double*, hipStream_t);

int launch_fock_C0000(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C0000(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_schwarz_C0000(PairBlock, double*, double*, hipStream_t);
int launch_fock_C1000(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C1000(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
int launch_fock_C1010(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C1010(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_schwarz_C1010(PairBlock, double*, double*, hipStream_t);
int launch_fock_C1100(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C1100(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
int launch_fock_C1110(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C1110(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
int launch_fock_C1111(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C1111(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C1111(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C1111(PairBlock, double*, double*, hipStream_t);
int launch_fock_C2000(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2000(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
int launch_fock_C2010(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2010(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
int launch_fock_C2011(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2011(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2011(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
int launch_fock_C2020(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2020(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2020(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C2020(PairBlock, double*, double*, hipStream_t);
int launch_fock_C2100(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2100(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
int launch_fock_C2110(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2110(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
int launch_fock_C2111(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2111(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2111(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
int launch_fock_C2120(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2120(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2120(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_tile_C2121(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2121(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C2121(PairBlock, double*, double*, hipStream_t);
int launch_fock_C2200(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2200(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2200(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
int launch_fock_C2210(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C2210(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2210(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_tile_C2211(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2211(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_tile_C2220(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C2220(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C2221(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C2222(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C2222(PairBlock, double*, double*, hipStream_t);
int launch_fock_C3000(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C3000(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C3000(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
int launch_fock_C3010(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C3010(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C3010(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
int launch_fock_C3011(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C3011(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C3011(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
int launch_fock_C3020(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C3020(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C3020(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3021(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3022(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3030(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C3030(PairBlock, double*, double*, hipStream_t);
int launch_fock_C3100(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C3100(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C3100(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
int launch_fock_C3110(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C3110(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C3110(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3111(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3120(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3121(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3122(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3130(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3131(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C3131(PairBlock, double*, double*, hipStream_t);
int launch_fock_C3200(const Task*, int, const PairBlock*, const MolDesc*, int, int, int, LaunchTo&);
void launch_fock_tile_C3200(const TileGroup*, int, const Task*, const PairBlock*, const MolDesc*, int, int, int, size_t, int, LaunchTo&);
void launch_fock_coop_C3200(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3210(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3211(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3220(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3221(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3222(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3230(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3231(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3232(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C3232(PairBlock, double*, double*, hipStream_t);
void launch_fock_coop_C3300(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3310(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3311(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3320(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3321(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3322(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3330(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3331(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3332(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_fock_coop_C3333(const Task*, int, const PairBlock*, const MolDesc*, int, int, double*, LaunchTo&);
void launch_schwarz_C3333(PairBlock, double*, double*, hipStream_t);

// Algorithmic FLOPs of nq quartets with np primitive quartets in class (cb|ck).
inline double class_flops(int cb, int ck, unsigned long long nq, unsigned long long np)
{
    if (cb == 0 && ck == 0) return double(np) * 59.0 + double(nq) * 12.0;
    if (cb == 1 && ck == 0) return double(np) * 74.0 + double(nq) * 36.0;
    if (cb == 1 && ck == 1) return double(np) * 126.0 + double(nq) * 108.0;
    if (cb == 2 && ck == 0) return double(np) * 120.0 + double(nq) * 126.0;
    if (cb == 2 && ck == 1) return double(np) * 286.0 + double(nq) * 378.0;
    if (cb == 2 && ck == 2) return double(np) * 773.0 + double(nq) * 1296.0;
    if (cb == 3 && ck == 0) return double(np) * 117.0 + double(nq) * 72.0;
    if (cb == 3 && ck == 1) return double(np) * 244.0 + double(nq) * 216.0;
    if (cb == 3 && ck == 2) return double(np) * 617.0 + double(nq) * 756.0;
    if (cb == 3 && ck == 3) return double(np) * 599.0 + double(nq) * 432.0;
    if (cb == 4 && ck == 0) return double(np) * 203.0 + double(nq) * 252.0;
    if (cb == 4 && ck == 1) return double(np) * 527.0 + double(nq) * 756.0;
    if (cb == 4 && ck == 2) return double(np) * 1473.0 + double(nq) * 2556.0;
    if (cb == 4 && ck == 3) return double(np) * 1425.0 + double(nq) * 1512.0;
    if (cb == 4 && ck == 4) return double(np) * 3360.0 + double(nq) * 5112.0;
    if (cb == 5 && ck == 0) return double(np) * 351.0 + double(nq) * 590.0;
    if (cb == 5 && ck == 1) return double(np) * 984.0 + double(nq) * 1770.0;
    if (cb == 5 && ck == 2) return double(np) * 2827.0 + double(nq) * 5868.0;
    if (cb == 5 && ck == 3) return double(np) * 2734.0 + double(nq) * 3540.0;
    if (cb == 5 && ck == 4) return double(np) * 6462.0 + double(nq) * 11736.0;
    if (cb == 5 && ck == 5) return double(np) * 13027.0 + double(nq) * 26138.0;
    if (cb == 6 && ck == 0) return double(np) * 191.0 + double(nq) * 120.0;
    if (cb == 6 && ck == 1) return double(np) * 428.0 + double(nq) * 360.0;
    if (cb == 6 && ck == 2) return double(np) * 1116.0 + double(nq) * 1260.0;
    if (cb == 6 && ck == 3) return double(np) * 1086.0 + double(nq) * 720.0;
    if (cb == 6 && ck == 4) return double(np) * 2525.0 + double(nq) * 2520.0;
    if (cb == 6 && ck == 5) return double(np) * 5099.0 + double(nq) * 5900.0;
    if (cb == 6 && ck == 6) return double(np) * 2446.0 + double(nq) * 1200.0;
    if (cb == 7 && ck == 0) return double(np) * 339.0 + double(nq) * 420.0;
    if (cb == 7 && ck == 1) return double(np) * 885.0 + double(nq) * 1260.0;
    if (cb == 7 && ck == 2) return double(np) * 2470.0 + double(nq) * 4230.0;
    if (cb == 7 && ck == 3) return double(np) * 2395.0 + double(nq) * 2520.0;
    if (cb == 7 && ck == 4) return double(np) * 5627.0 + double(nq) * 8460.0;
    if (cb == 7 && ck == 5) return double(np) * 11350.0 + double(nq) * 19070.0;
    if (cb == 7 && ck == 6) return double(np) * 5417.0 + double(nq) * 4200.0;
    if (cb == 7 && ck == 7) return double(np) * 11140.0 + double(nq) * 14100.0;
    if (cb == 8 && ck == 0) return double(np) * 571.0 + double(nq) * 978.0;
    if (cb == 8 && ck == 1) return double(np) * 1567.0 + double(nq) * 2934.0;
    if (cb == 8 && ck == 2) return double(np) * 4451.0 + double(nq) * 9630.0;
    if (cb == 8 && ck == 3) return double(np) * 4313.0 + double(nq) * 5868.0;
    if (cb == 8 && ck == 4) return double(np) * 10116.0 + double(nq) * 19260.0;
    if (cb == 8 && ck == 5) return double(np) * 20339.0 + double(nq) * 42476.0;
    if (cb == 8 && ck == 6) return double(np) * 9705.0 + double(nq) * 9780.0;
    if (cb == 8 && ck == 7) return double(np) * 19928.0 + double(nq) * 32100.0;
    if (cb == 8 && ck == 8) return double(np) * 36378.0 + double(nq) * 70548.0;
    if (cb == 9 && ck == 0) return double(np) * 924.0 + double(nq) * 1902.0;
    if (cb == 9 && ck == 1) return double(np) * 2534.0 + double(nq) * 5706.0;
    if (cb == 9 && ck == 2) return double(np) * 7191.0 + double(nq) * 18450.0;
    if (cb == 9 && ck == 3) return double(np) * 6969.0 + double(nq) * 11412.0;
    if (cb == 9 && ck == 4) return double(np) * 16257.0 + double(nq) * 36900.0;
    if (cb == 9 && ck == 5) return double(np) * 32565.0 + double(nq) * 80164.0;
    if (cb == 9 && ck == 6) return double(np) * 15557.0 + double(nq) * 19020.0;
    if (cb == 9 && ck == 7) return double(np) * 31865.0 + double(nq) * 61500.0;
    if (cb == 9 && ck == 8) return double(np) * 57995.0 + double(nq) * 133212.0;
    if (cb == 9 && ck == 9) return double(np) * 97635.0 + double(nq) * 242148.0;
    return 0.0;
}


// indexed [bra pair class][ket pair class], pair class = La*(La+1)/2 + Lb;
// nullptr: the class has no per-lane kernels (wave-per-quartet only)
inline FockLaunch fock_launcher(int cb, int ck)
{
    if (cb == 0 && ck == 0) return launch_fock_C0000;
    if (cb == 1 && ck == 0) return launch_fock_C1000;
    if (cb == 1 && ck == 1) return launch_fock_C1010;
    if (cb == 2 && ck == 0) return launch_fock_C1100;
    if (cb == 2 && ck == 1) return launch_fock_C1110;
    if (cb == 2 && ck == 2) return launch_fock_C1111;
    if (cb == 3 && ck == 0) return launch_fock_C2000;
    if (cb == 3 && ck == 1) return launch_fock_C2010;
    if (cb == 3 && ck == 2) return launch_fock_C2011;
    if (cb == 3 && ck == 3) return launch_fock_C2020;
    if (cb == 4 && ck == 0) return launch_fock_C2100;
    if (cb == 4 && ck == 1) return launch_fock_C2110;
    if (cb == 4 && ck == 2) return launch_fock_C2111;
    if (cb == 4 && ck == 3) return launch_fock_C2120;
    if (cb == 5 && ck == 0) return launch_fock_C2200;
    if (cb == 5 && ck == 1) return launch_fock_C2210;
    if (cb == 6 && ck == 0) return launch_fock_C3000;
    if (cb == 6 && ck == 1) return launch_fock_C3010;
    if (cb == 6 && ck == 2) return launch_fock_C3011;
    if (cb == 6 && ck == 3) return launch_fock_C3020;
    if (cb == 7 && ck == 0) return launch_fock_C3100;
    if (cb == 7 && ck == 1) return launch_fock_C3110;
    if (cb == 8 && ck == 0) return launch_fock_C3200;
    return nullptr;
}

inline FockTileLaunch fock_tile_launcher(int cb, int ck)
{
    if (cb == 0 && ck == 0) return launch_fock_tile_C0000;
    if (cb == 1 && ck == 0) return launch_fock_tile_C1000;
    if (cb == 1 && ck == 1) return launch_fock_tile_C1010;
    if (cb == 2 && ck == 0) return launch_fock_tile_C1100;
    if (cb == 2 && ck == 1) return launch_fock_tile_C1110;
    if (cb == 2 && ck == 2) return launch_fock_tile_C1111;
    if (cb == 3 && ck == 0) return launch_fock_tile_C2000;
    if (cb == 3 && ck == 1) return launch_fock_tile_C2010;
    if (cb == 3 && ck == 2) return launch_fock_tile_C2011;
    if (cb == 3 && ck == 3) return launch_fock_tile_C2020;
    if (cb == 4 && ck == 0) return launch_fock_tile_C2100;
    if (cb == 4 && ck == 1) return launch_fock_tile_C2110;
    if (cb == 4 && ck == 2) return launch_fock_tile_C2111;
    if (cb == 4 && ck == 3) return launch_fock_tile_C2120;
    if (cb == 4 && ck == 4) return launch_fock_tile_C2121;
    if (cb == 5 && ck == 0) return launch_fock_tile_C2200;
    if (cb == 5 && ck == 1) return launch_fock_tile_C2210;
    if (cb == 5 && ck == 2) return launch_fock_tile_C2211;
    if (cb == 5 && ck == 3) return launch_fock_tile_C2220;
    if (cb == 6 && ck == 0) return launch_fock_tile_C3000;
    if (cb == 6 && ck == 1) return launch_fock_tile_C3010;
    if (cb == 6 && ck == 2) return launch_fock_tile_C3011;
    if (cb == 6 && ck == 3) return launch_fock_tile_C3020;
    if (cb == 7 && ck == 0) return launch_fock_tile_C3100;
    if (cb == 7 && ck == 1) return launch_fock_tile_C3110;
    if (cb == 8 && ck == 0) return launch_fock_tile_C3200;
    return nullptr;
}

// the class's closed-shell FP64 tile kernel runs in Hermite Gaussians (fock_md_kernel)
inline bool fock_tile_is_md(int cb, int ck)
{
    return (cb == 4 && ck == 2) || (cb == 5 && ck == 3) || (cb == 4 && ck == 4) || (cb == 5 && ck == 2);
}

// wave-per-quartet kernels (nullptr: the class has none)
inline FockCoopLaunch fock_coop_launcher(int cb, int ck)
{
    if (cb == 2 && ck == 2) return launch_fock_coop_C1111;
    if (cb == 3 && ck == 2) return launch_fock_coop_C2011;
    if (cb == 3 && ck == 3) return launch_fock_coop_C2020;
    if (cb == 4 && ck == 2) return launch_fock_coop_C2111;
    if (cb == 4 && ck == 3) return launch_fock_coop_C2120;
    if (cb == 4 && ck == 4) return launch_fock_coop_C2121;
    if (cb == 5 && ck == 0) return launch_fock_coop_C2200;
    if (cb == 5 && ck == 1) return launch_fock_coop_C2210;
    if (cb == 5 && ck == 2) return launch_fock_coop_C2211;
    if (cb == 5 && ck == 3) return launch_fock_coop_C2220;
    if (cb == 5 && ck == 4) return launch_fock_coop_C2221;
    if (cb == 5 && ck == 5) return launch_fock_coop_C2222;
    if (cb == 6 && ck == 0) return launch_fock_coop_C3000;
    if (cb == 6 && ck == 1) return launch_fock_coop_C3010;
    if (cb == 6 && ck == 2) return launch_fock_coop_C3011;
    if (cb == 6 && ck == 3) return launch_fock_coop_C3020;
    if (cb == 6 && ck == 4) return launch_fock_coop_C3021;
    if (cb == 6 && ck == 5) return launch_fock_coop_C3022;
    if (cb == 6 && ck == 6) return launch_fock_coop_C3030;
    if (cb == 7 && ck == 0) return launch_fock_coop_C3100;
    if (cb == 7 && ck == 1) return launch_fock_coop_C3110;
    if (cb == 7 && ck == 2) return launch_fock_coop_C3111;
    if (cb == 7 && ck == 3) return launch_fock_coop_C3120;
    if (cb == 7 && ck == 4) return launch_fock_coop_C3121;
    if (cb == 7 && ck == 5) return launch_fock_coop_C3122;
    if (cb == 7 && ck == 6) return launch_fock_coop_C3130;
    if (cb == 7 && ck == 7) return launch_fock_coop_C3131;
    if (cb == 8 && ck == 0) return launch_fock_coop_C3200;
    if (cb == 8 && ck == 1) return launch_fock_coop_C3210;
    if (cb == 8 && ck == 2) return launch_fock_coop_C3211;
    if (cb == 8 && ck == 3) return launch_fock_coop_C3220;
    if (cb == 8 && ck == 4) return launch_fock_coop_C3221;
    if (cb == 8 && ck == 5) return launch_fock_coop_C3222;
    if (cb == 8 && ck == 6) return launch_fock_coop_C3230;
    if (cb == 8 && ck == 7) return launch_fock_coop_C3231;
    if (cb == 8 && ck == 8) return launch_fock_coop_C3232;
    if (cb == 9 && ck == 0) return launch_fock_coop_C3300;
    if (cb == 9 && ck == 1) return launch_fock_coop_C3310;
    if (cb == 9 && ck == 2) return launch_fock_coop_C3311;
    if (cb == 9 && ck == 3) return launch_fock_coop_C3320;
    if (cb == 9 && ck == 4) return launch_fock_coop_C3321;
    if (cb == 9 && ck == 5) return launch_fock_coop_C3322;
    if (cb == 9 && ck == 6) return launch_fock_coop_C3330;
    if (cb == 9 && ck == 7) return launch_fock_coop_C3331;
    if (cb == 9 && ck == 8) return launch_fock_coop_C3332;
    if (cb == 9 && ck == 9) return launch_fock_coop_C3333;
    return nullptr;
}

// doubles per workgroup slice of the global slot buffer (0: the class uses LDS)
inline int coop_global_doubles(int cb, int ck)
{
    if (cb == 8 && ck == 8) return 10910;
    if (cb == 9 && ck == 5) return 13046;
    if (cb == 9 && ck == 7) return 10954;
    if (cb == 9 && ck == 8) return 21574;
    if (cb == 9 && ck == 9) return 35734;
    return 0;
}

inline SchwarzLaunch schwarz_launcher(int c)
{
    if (c == 0) return launch_schwarz_C0000;
    if (c == 1) return launch_schwarz_C1010;
    if (c == 2) return launch_schwarz_C1111;
    if (c == 3) return launch_schwarz_C2020;
    if (c == 4) return launch_schwarz_C2121;
    if (c == 5) return launch_schwarz_C2222;
    if (c == 6) return launch_schwarz_C3030;
    if (c == 7) return launch_schwarz_C3131;
    if (c == 8) return launch_schwarz_C3232;
    if (c == 9) return launch_schwarz_C3333;
    return nullptr;
}

// (list, workgroups, groups, tasks, blocks, mols, os, waves, lds bytes, global slots, target)
using FuseLaunch = void (*)(const FusedBlock*, int, const TileGroup*, const Task*, const PairBlock*, const MolDesc*, int, int, size_t, double*, LaunchTo&);
void launch_fuse_tile3(const FusedBlock*, int, const TileGroup*, const Task*, const PairBlock*, const MolDesc*, int, int, size_t, double*, LaunchTo&);
void launch_fuse_tile2(const FusedBlock*, int, const TileGroup*, const Task*, const PairBlock*, const MolDesc*, int, int, size_t, double*, LaunchTo&);
void launch_fuse_tile1(const FusedBlock*, int, const TileGroup*, const Task*, const PairBlock*, const MolDesc*, int, int, size_t, double*, LaunchTo&);
void launch_fuse_coop_small(const FusedBlock*, int, const TileGroup*, const Task*, const PairBlock*, const MolDesc*, int, int, size_t, double*, LaunchTo&);
void launch_fuse_coop_large(const FusedBlock*, int, const TileGroup*, const Task*, const PairBlock*, const MolDesc*, int, int, size_t, double*, LaunchTo&);
void launch_fuse_coop_global(const FusedBlock*, int, const TileGroup*, const Task*, const PairBlock*, const MolDesc*, int, int, size_t, double*, LaunchTo&);

struct FuseKernel {
    FuseLaunch launch;
    bool coop;          // wave-per-quartet classes
    int global;         // doubles of a workgroup's slice of the global slot buffer (0: slots in LDS)
};
constexpr int kFuseKernels = 6;
inline FuseKernel fuse_kernel(int k)
{
    constexpr FuseKernel all[kFuseKernels] = {
        {launch_fuse_tile3, false, 0},
        {launch_fuse_tile2, false, 0},
        {launch_fuse_tile1, false, 0},
        {launch_fuse_coop_small, true, 0},
        {launch_fuse_coop_large, true, 0},
        {launch_fuse_coop_global, true, 35734},
    };
    return all[k];
}

// the kernel that runs a class beside others (-1: none), and the class's number in it
inline int fuse_bucket(int cb, int ck, bool coop)
{
    switch ((cb * 16 + ck) * 2 + (coop ? 1 : 0)) {
    case 0: return 0;
    case 32: return 0;
    case 34: return 0;
    case 64: return 0;
    case 96: return 0;
    case 128: return 0;
    case 192: return 0;
    case 66: return 1;
    case 98: return 1;
    case 160: return 1;
    case 194: return 1;
    case 224: return 1;
    case 68: return 2;
    case 100: return 2;
    case 102: return 2;
    case 130: return 2;
    case 134: return 2;
    case 162: return 2;
    case 196: return 2;
    case 198: return 2;
    case 226: return 2;
    case 256: return 2;
    case 69: return 3;
    case 101: return 3;
    case 103: return 3;
    case 133: return 3;
    case 135: return 3;
    case 137: return 3;
    case 161: return 3;
    case 163: return 3;
    case 165: return 3;
    case 167: return 3;
    case 193: return 3;
    case 195: return 3;
    case 197: return 3;
    case 199: return 3;
    case 201: return 3;
    case 205: return 3;
    case 225: return 3;
    case 227: return 3;
    case 229: return 3;
    case 231: return 3;
    case 257: return 3;
    case 259: return 3;
    case 263: return 3;
    case 289: return 3;
    case 291: return 3;
    case 169: return 4;
    case 171: return 4;
    case 203: return 4;
    case 233: return 4;
    case 235: return 4;
    case 237: return 4;
    case 239: return 4;
    case 261: return 4;
    case 265: return 4;
    case 267: return 4;
    case 269: return 4;
    case 271: return 4;
    case 293: return 4;
    case 295: return 4;
    case 297: return 4;
    case 301: return 4;
    case 273: return 5;
    case 299: return 5;
    case 303: return 5;
    case 305: return 5;
    case 307: return 5;
    }
    return -1;
}

// doubles of LDS a wave-per-quartet class needs (0: its slots are global)
inline int coop_lds_doubles(int cb, int ck)
{
    switch (cb * 16 + ck) {
    case 34: return 334;
    case 50: return 268;
    case 51: return 236;
    case 66: return 574;
    case 67: return 478;
    case 68: return 1090;
    case 80: return 205;
    case 81: return 451;
    case 82: return 1141;
    case 83: return 820;
    case 84: return 2176;
    case 85: return 4210;
    case 96: return 107;
    case 97: return 194;
    case 98: return 419;
    case 99: return 367;
    case 100: return 786;
    case 101: return 1386;
    case 102: return 660;
    case 112: return 182;
    case 113: return 354;
    case 114: return 889;
    case 115: return 734;
    case 116: return 1700;
    case 117: return 3311;
    case 118: return 1328;
    case 119: return 2802;
    case 128: return 302;
    case 129: return 686;
    case 130: return 1774;
    case 131: return 1262;
    case 132: return 3406;
    case 133: return 6622;
    case 134: return 2189;
    case 135: return 5582;
    case 144: return 526;
    case 145: return 1270;
    case 146: return 3422;
    case 147: return 2386;
    case 148: return 6650;
    case 150: return 3874;
    }
    return 0;
}

}  // namespace qf
