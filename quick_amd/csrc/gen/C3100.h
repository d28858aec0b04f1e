// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#pragma once
#include "../qf_device.h"
namespace qf {
// (fp|ss): 25 accumulators, 30 integrals, VRR 265 FLOP/prim, HRR 60 FLOP
struct C3100 {
  static constexpr int La = 3, Lb = 1, Lc = 0, Ld = 0, L = 4;
  static constexpr int NACC = 25, NI = 30;
  static constexpr int VRR_FLOP = 265, HRR_FLOP = 60;
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
    const R v020_000_2 = p.PA[1] * v010_000_2 + p.WP[1] * v010_000_3 + R(1) * p.oo2z * (v000_000_2 - p.rz * v000_000_3);
    const R v200_000_2 = p.PA[0] * v100_000_2 + p.WP[0] * v100_000_3 + R(1) * p.oo2z * (v000_000_2 - p.rz * v000_000_3);
    const R v002_000_1 = p.PA[2] * v001_000_1 + p.WP[2] * v001_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
    const R v011_000_1 = p.PA[1] * v001_000_1 + p.WP[1] * v001_000_2;
    const R v020_000_1 = p.PA[1] * v010_000_1 + p.WP[1] * v010_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
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
    const R v120_000_1 = p.PA[0] * v020_000_1 + p.WP[0] * v020_000_2;
    const R v201_000_1 = p.PA[2] * v200_000_1 + p.WP[2] * v200_000_2;
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
    const R v004_000_0 = p.PA[2] * v003_000_0 + p.WP[2] * v003_000_1 + R(3) * p.oo2z * (v002_000_0 - p.rz * v002_000_1);
    const R v013_000_0 = p.PA[1] * v003_000_0 + p.WP[1] * v003_000_1;
    const R v022_000_0 = p.PA[1] * v012_000_0 + p.WP[1] * v012_000_1 + R(1) * p.oo2z * (v002_000_0 - p.rz * v002_000_1);
    const R v031_000_0 = p.PA[2] * v030_000_0 + p.WP[2] * v030_000_1;
    const R v040_000_0 = p.PA[1] * v030_000_0 + p.WP[1] * v030_000_1 + R(3) * p.oo2z * (v020_000_0 - p.rz * v020_000_1);
    const R v103_000_0 = p.PA[0] * v003_000_0 + p.WP[0] * v003_000_1;
    const R v112_000_0 = p.PA[0] * v012_000_0 + p.WP[0] * v012_000_1;
    const R v121_000_0 = p.PA[0] * v021_000_0 + p.WP[0] * v021_000_1;
    const R v130_000_0 = p.PA[0] * v030_000_0 + p.WP[0] * v030_000_1;
    const R v202_000_0 = p.PA[0] * v102_000_0 + p.WP[0] * v102_000_1 + R(1) * p.oo2z * (v002_000_0 - p.rz * v002_000_1);
    const R v211_000_0 = p.PA[1] * v201_000_0 + p.WP[1] * v201_000_1;
    const R v220_000_0 = p.PA[0] * v120_000_0 + p.WP[0] * v120_000_1 + R(1) * p.oo2z * (v020_000_0 - p.rz * v020_000_1);
    const R v301_000_0 = p.PA[2] * v300_000_0 + p.WP[2] * v300_000_1;
    const R v310_000_0 = p.PA[1] * v300_000_0 + p.WP[1] * v300_000_1;
    const R v400_000_0 = p.PA[0] * v300_000_0 + p.WP[0] * v300_000_1 + R(3) * p.oo2z * (v200_000_0 - p.rz * v200_000_1);
    acc[0] += v300_000_0;
    acc[1] += v210_000_0;
    acc[2] += v120_000_0;
    acc[3] += v030_000_0;
    acc[4] += v201_000_0;
    acc[5] += v111_000_0;
    acc[6] += v021_000_0;
    acc[7] += v102_000_0;
    acc[8] += v012_000_0;
    acc[9] += v003_000_0;
    acc[10] += v400_000_0;
    acc[11] += v310_000_0;
    acc[12] += v301_000_0;
    acc[13] += v220_000_0;
    acc[14] += v211_000_0;
    acc[15] += v202_000_0;
    acc[16] += v130_000_0;
    acc[17] += v121_000_0;
    acc[18] += v112_000_0;
    acc[19] += v103_000_0;
    acc[20] += v040_000_0;
    acc[21] += v031_000_0;
    acc[22] += v022_000_0;
    acc[23] += v013_000_0;
    acc[24] += v004_000_0;
  }
  template <typename R>
  __host__ __device__ static __forceinline__ void hrr(const R (&acc)[NACC], const R (&AB)[3], const R (&CD)[3], R (&I)[NI]) {
    const R b300_100_000_000 = acc[10] + AB[0] * acc[0];
    const R b300_010_000_000 = acc[11] + AB[1] * acc[0];
    const R b300_001_000_000 = acc[12] + AB[2] * acc[0];
    const R b210_100_000_000 = acc[11] + AB[0] * acc[1];
    const R b210_010_000_000 = acc[13] + AB[1] * acc[1];
    const R b210_001_000_000 = acc[14] + AB[2] * acc[1];
    const R b120_100_000_000 = acc[13] + AB[0] * acc[2];
    const R b120_010_000_000 = acc[16] + AB[1] * acc[2];
    const R b120_001_000_000 = acc[17] + AB[2] * acc[2];
    const R b030_100_000_000 = acc[16] + AB[0] * acc[3];
    const R b030_010_000_000 = acc[20] + AB[1] * acc[3];
    const R b030_001_000_000 = acc[21] + AB[2] * acc[3];
    const R b201_100_000_000 = acc[12] + AB[0] * acc[4];
    const R b201_010_000_000 = acc[14] + AB[1] * acc[4];
    const R b201_001_000_000 = acc[15] + AB[2] * acc[4];
    const R b111_100_000_000 = acc[14] + AB[0] * acc[5];
    const R b111_010_000_000 = acc[17] + AB[1] * acc[5];
    const R b111_001_000_000 = acc[18] + AB[2] * acc[5];
    const R b021_100_000_000 = acc[17] + AB[0] * acc[6];
    const R b021_010_000_000 = acc[21] + AB[1] * acc[6];
    const R b021_001_000_000 = acc[22] + AB[2] * acc[6];
    const R b102_100_000_000 = acc[15] + AB[0] * acc[7];
    const R b102_010_000_000 = acc[18] + AB[1] * acc[7];
    const R b102_001_000_000 = acc[19] + AB[2] * acc[7];
    const R b012_100_000_000 = acc[18] + AB[0] * acc[8];
    const R b012_010_000_000 = acc[22] + AB[1] * acc[8];
    const R b012_001_000_000 = acc[23] + AB[2] * acc[8];
    const R b003_100_000_000 = acc[19] + AB[0] * acc[9];
    const R b003_010_000_000 = acc[23] + AB[1] * acc[9];
    const R b003_001_000_000 = acc[24] + AB[2] * acc[9];
    I[0] = b300_100_000_000;
    I[1] = b300_010_000_000;
    I[2] = b300_001_000_000;
    I[3] = b210_100_000_000;
    I[4] = b210_010_000_000;
    I[5] = b210_001_000_000;
    I[6] = b120_100_000_000;
    I[7] = b120_010_000_000;
    I[8] = b120_001_000_000;
    I[9] = b030_100_000_000;
    I[10] = b030_010_000_000;
    I[11] = b030_001_000_000;
    I[12] = b201_100_000_000;
    I[13] = b201_010_000_000;
    I[14] = b201_001_000_000;
    I[15] = b111_100_000_000;
    I[16] = b111_010_000_000;
    I[17] = b111_001_000_000;
    I[18] = b021_100_000_000;
    I[19] = b021_010_000_000;
    I[20] = b021_001_000_000;
    I[21] = b102_100_000_000;
    I[22] = b102_010_000_000;
    I[23] = b102_001_000_000;
    I[24] = b012_100_000_000;
    I[25] = b012_010_000_000;
    I[26] = b012_001_000_000;
    I[27] = b003_100_000_000;
    I[28] = b003_010_000_000;
    I[29] = b003_001_000_000;
  }
};
}  // namespace qf
