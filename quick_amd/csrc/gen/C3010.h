// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#pragma once
#include "../qf_device.h"
namespace qf {
// (fs|ps): 30 accumulators, 30 integrals, VRR 354 FLOP/prim, HRR 0 FLOP
struct C3010 {
  static constexpr int La = 3, Lb = 0, Lc = 1, Ld = 0, L = 4;
  static constexpr int NACC = 30, NI = 30;
  static constexpr int VRR_FLOP = 354, HRR_FLOP = 0;
  static constexpr int MIN_WAVES = 2;   // waves per SIMD the register budget targets
  static constexpr int MIN_WAVES_OS = 1;   // the same for the open-shell kernels
  static constexpr bool LEAN_K = false;   // FP64 tile kernels: first exchange re-read per quartet
  template <typename R>
  __host__ __device__ static __forceinline__ void vrr(const R (&F)[L + 1], const VrrPar<R>& p, R (&acc)[NACC]) {
    const R v000_000_4 = F[4];
    const R v000_000_3 = F[3];
    const R v000_000_2 = F[2];
    const R v000_000_1 = F[1];
    const R v000_000_0 = F[0];
    const R v001_000_3 = p.PA[2] * v000_000_3 + p.WP[2] * v000_000_4;
    const R v010_000_3 = p.PA[1] * v000_000_3 + p.WP[1] * v000_000_4;
    const R v100_000_3 = p.PA[0] * v000_000_3 + p.WP[0] * v000_000_4;
    const R v001_000_2 = p.PA[2] * v000_000_2 + p.WP[2] * v000_000_3;
    const R v010_000_2 = p.PA[1] * v000_000_2 + p.WP[1] * v000_000_3;
    const R v100_000_2 = p.PA[0] * v000_000_2 + p.WP[0] * v000_000_3;
    const R v001_000_1 = p.PA[2] * v000_000_1 + p.WP[2] * v000_000_2;
    const R v010_000_1 = p.PA[1] * v000_000_1 + p.WP[1] * v000_000_2;
    const R v100_000_1 = p.PA[0] * v000_000_1 + p.WP[0] * v000_000_2;
    const R v001_000_0 = p.PA[2] * v000_000_0 + p.WP[2] * v000_000_1;
    const R v010_000_0 = p.PA[1] * v000_000_0 + p.WP[1] * v000_000_1;
    const R v100_000_0 = p.PA[0] * v000_000_0 + p.WP[0] * v000_000_1;
    const R v002_000_2 = p.PA[2] * v001_000_2 + p.WP[2] * v001_000_3 + R(1) * p.oo2z * (v000_000_2 - p.rz * v000_000_3);
    const R v011_000_2 = p.PA[1] * v001_000_2 + p.WP[1] * v001_000_3;
    const R v020_000_2 = p.PA[1] * v010_000_2 + p.WP[1] * v010_000_3 + R(1) * p.oo2z * (v000_000_2 - p.rz * v000_000_3);
    const R v200_000_2 = p.PA[0] * v100_000_2 + p.WP[0] * v100_000_3 + R(1) * p.oo2z * (v000_000_2 - p.rz * v000_000_3);
    const R v002_000_1 = p.PA[2] * v001_000_1 + p.WP[2] * v001_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
    const R v011_000_1 = p.PA[1] * v001_000_1 + p.WP[1] * v001_000_2;
    const R v020_000_1 = p.PA[1] * v010_000_1 + p.WP[1] * v010_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
    const R v101_000_1 = p.PA[0] * v001_000_1 + p.WP[0] * v001_000_2;
    const R v110_000_1 = p.PA[0] * v010_000_1 + p.WP[0] * v010_000_2;
    const R v200_000_1 = p.PA[0] * v100_000_1 + p.WP[0] * v100_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
    const R v002_000_0 = p.PA[2] * v001_000_0 + p.WP[2] * v001_000_1 + R(1) * p.oo2z * (v000_000_0 - p.rz * v000_000_1);
    const R v011_000_0 = p.PA[1] * v001_000_0 + p.WP[1] * v001_000_1;
    const R v020_000_0 = p.PA[1] * v010_000_0 + p.WP[1] * v010_000_1 + R(1) * p.oo2z * (v000_000_0 - p.rz * v000_000_1);
    const R v200_000_0 = p.PA[0] * v100_000_0 + p.WP[0] * v100_000_1 + R(1) * p.oo2z * (v000_000_0 - p.rz * v000_000_1);
    const R v003_000_1 = p.PA[2] * v002_000_1 + p.WP[2] * v002_000_2 + R(2) * p.oo2z * (v001_000_1 - p.rz * v001_000_2);
    const R v012_000_1 = p.PA[1] * v002_000_1 + p.WP[1] * v002_000_2;
    const R v021_000_1 = p.PA[2] * v020_000_1 + p.WP[2] * v020_000_2;
    const R v030_000_1 = p.PA[1] * v020_000_1 + p.WP[1] * v020_000_2 + R(2) * p.oo2z * (v010_000_1 - p.rz * v010_000_2);
    const R v102_000_1 = p.PA[0] * v002_000_1 + p.WP[0] * v002_000_2;
    const R v111_000_1 = p.PA[0] * v011_000_1 + p.WP[0] * v011_000_2;
    const R v120_000_1 = p.PA[0] * v020_000_1 + p.WP[0] * v020_000_2;
    const R v201_000_1 = p.PA[2] * v200_000_1 + p.WP[2] * v200_000_2;
    const R v210_000_1 = p.PA[1] * v200_000_1 + p.WP[1] * v200_000_2;
    const R v300_000_1 = p.PA[0] * v200_000_1 + p.WP[0] * v200_000_2 + R(2) * p.oo2z * (v100_000_1 - p.rz * v100_000_2);
    const R v003_000_0 = p.PA[2] * v002_000_0 + p.WP[2] * v002_000_1 + R(2) * p.oo2z * (v001_000_0 - p.rz * v001_000_1);
    const R v012_000_0 = p.PA[1] * v002_000_0 + p.WP[1] * v002_000_1;
    const R v021_000_0 = p.PA[2] * v020_000_0 + p.WP[2] * v020_000_1;
    const R v030_000_0 = p.PA[1] * v020_000_0 + p.WP[1] * v020_000_1 + R(2) * p.oo2z * (v010_000_0 - p.rz * v010_000_1);
    const R v102_000_0 = p.PA[0] * v002_000_0 + p.WP[0] * v002_000_1;
    const R v111_000_0 = p.PA[0] * v011_000_0 + p.WP[0] * v011_000_1;
    const R v120_000_0 = p.PA[0] * v020_000_0 + p.WP[0] * v020_000_1;
    const R v201_000_0 = p.PA[2] * v200_000_0 + p.WP[2] * v200_000_1;
    const R v210_000_0 = p.PA[1] * v200_000_0 + p.WP[1] * v200_000_1;
    const R v300_000_0 = p.PA[0] * v200_000_0 + p.WP[0] * v200_000_1 + R(2) * p.oo2z * (v100_000_0 - p.rz * v100_000_1);
    const R v003_001_0 = p.QC[2] * v003_000_0 + p.WQ[2] * v003_000_1 + R(3) * p.oo2zn * v002_000_1;
    const R v003_010_0 = p.QC[1] * v003_000_0 + p.WQ[1] * v003_000_1;
    const R v003_100_0 = p.QC[0] * v003_000_0 + p.WQ[0] * v003_000_1;
    const R v012_001_0 = p.QC[2] * v012_000_0 + p.WQ[2] * v012_000_1 + R(2) * p.oo2zn * v011_000_1;
    const R v012_010_0 = p.QC[1] * v012_000_0 + p.WQ[1] * v012_000_1 + R(1) * p.oo2zn * v002_000_1;
    const R v012_100_0 = p.QC[0] * v012_000_0 + p.WQ[0] * v012_000_1;
    const R v021_001_0 = p.QC[2] * v021_000_0 + p.WQ[2] * v021_000_1 + R(1) * p.oo2zn * v020_000_1;
    const R v021_010_0 = p.QC[1] * v021_000_0 + p.WQ[1] * v021_000_1 + R(2) * p.oo2zn * v011_000_1;
    const R v021_100_0 = p.QC[0] * v021_000_0 + p.WQ[0] * v021_000_1;
    const R v030_001_0 = p.QC[2] * v030_000_0 + p.WQ[2] * v030_000_1;
    const R v030_010_0 = p.QC[1] * v030_000_0 + p.WQ[1] * v030_000_1 + R(3) * p.oo2zn * v020_000_1;
    const R v030_100_0 = p.QC[0] * v030_000_0 + p.WQ[0] * v030_000_1;
    const R v102_001_0 = p.QC[2] * v102_000_0 + p.WQ[2] * v102_000_1 + R(2) * p.oo2zn * v101_000_1;
    const R v102_010_0 = p.QC[1] * v102_000_0 + p.WQ[1] * v102_000_1;
    const R v102_100_0 = p.QC[0] * v102_000_0 + p.WQ[0] * v102_000_1 + R(1) * p.oo2zn * v002_000_1;
    const R v111_001_0 = p.QC[2] * v111_000_0 + p.WQ[2] * v111_000_1 + R(1) * p.oo2zn * v110_000_1;
    const R v111_010_0 = p.QC[1] * v111_000_0 + p.WQ[1] * v111_000_1 + R(1) * p.oo2zn * v101_000_1;
    const R v111_100_0 = p.QC[0] * v111_000_0 + p.WQ[0] * v111_000_1 + R(1) * p.oo2zn * v011_000_1;
    const R v120_001_0 = p.QC[2] * v120_000_0 + p.WQ[2] * v120_000_1;
    const R v120_010_0 = p.QC[1] * v120_000_0 + p.WQ[1] * v120_000_1 + R(2) * p.oo2zn * v110_000_1;
    const R v120_100_0 = p.QC[0] * v120_000_0 + p.WQ[0] * v120_000_1 + R(1) * p.oo2zn * v020_000_1;
    const R v201_001_0 = p.QC[2] * v201_000_0 + p.WQ[2] * v201_000_1 + R(1) * p.oo2zn * v200_000_1;
    const R v201_010_0 = p.QC[1] * v201_000_0 + p.WQ[1] * v201_000_1;
    const R v201_100_0 = p.QC[0] * v201_000_0 + p.WQ[0] * v201_000_1 + R(2) * p.oo2zn * v101_000_1;
    const R v210_001_0 = p.QC[2] * v210_000_0 + p.WQ[2] * v210_000_1;
    const R v210_010_0 = p.QC[1] * v210_000_0 + p.WQ[1] * v210_000_1 + R(1) * p.oo2zn * v200_000_1;
    const R v210_100_0 = p.QC[0] * v210_000_0 + p.WQ[0] * v210_000_1 + R(2) * p.oo2zn * v110_000_1;
    const R v300_001_0 = p.QC[2] * v300_000_0 + p.WQ[2] * v300_000_1;
    const R v300_010_0 = p.QC[1] * v300_000_0 + p.WQ[1] * v300_000_1;
    const R v300_100_0 = p.QC[0] * v300_000_0 + p.WQ[0] * v300_000_1 + R(3) * p.oo2zn * v200_000_1;
    acc[0] += v300_100_0;
    acc[1] += v300_010_0;
    acc[2] += v300_001_0;
    acc[3] += v210_100_0;
    acc[4] += v210_010_0;
    acc[5] += v210_001_0;
    acc[6] += v120_100_0;
    acc[7] += v120_010_0;
    acc[8] += v120_001_0;
    acc[9] += v030_100_0;
    acc[10] += v030_010_0;
    acc[11] += v030_001_0;
    acc[12] += v201_100_0;
    acc[13] += v201_010_0;
    acc[14] += v201_001_0;
    acc[15] += v111_100_0;
    acc[16] += v111_010_0;
    acc[17] += v111_001_0;
    acc[18] += v021_100_0;
    acc[19] += v021_010_0;
    acc[20] += v021_001_0;
    acc[21] += v102_100_0;
    acc[22] += v102_010_0;
    acc[23] += v102_001_0;
    acc[24] += v012_100_0;
    acc[25] += v012_010_0;
    acc[26] += v012_001_0;
    acc[27] += v003_100_0;
    acc[28] += v003_010_0;
    acc[29] += v003_001_0;
  }
  template <typename R>
  __host__ __device__ static __forceinline__ void hrr(const R (&acc)[NACC], const R (&AB)[3], const R (&CD)[3], R (&I)[NI]) {
    I[0] = acc[0];
    I[1] = acc[1];
    I[2] = acc[2];
    I[3] = acc[3];
    I[4] = acc[4];
    I[5] = acc[5];
    I[6] = acc[6];
    I[7] = acc[7];
    I[8] = acc[8];
    I[9] = acc[9];
    I[10] = acc[10];
    I[11] = acc[11];
    I[12] = acc[12];
    I[13] = acc[13];
    I[14] = acc[14];
    I[15] = acc[15];
    I[16] = acc[16];
    I[17] = acc[17];
    I[18] = acc[18];
    I[19] = acc[19];
    I[20] = acc[20];
    I[21] = acc[21];
    I[22] = acc[22];
    I[23] = acc[23];
    I[24] = acc[24];
    I[25] = acc[25];
    I[26] = acc[26];
    I[27] = acc[27];
    I[28] = acc[28];
    I[29] = acc[29];
  }
};
}  // namespace qf
