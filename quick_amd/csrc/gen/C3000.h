// Generated by quick_amd/codegen/gen_eri.py - do not edit.
#pragma once
#include "../qf_device.h"
namespace qf {
// (fs|ss): 10 accumulators, 10 integrals, VRR 121 FLOP/prim, HRR 0 FLOP
struct C3000 {
  static constexpr int La = 3, Lb = 0, Lc = 0, Ld = 0, L = 3;
  static constexpr int NACC = 10, NI = 10;
  static constexpr int VRR_FLOP = 121, HRR_FLOP = 0;
  static constexpr int MIN_WAVES = 3;   // waves per SIMD the register budget targets
  static constexpr int MIN_WAVES_OS = 2;   // the same for the open-shell kernels
  static constexpr bool LEAN_K = false;   // FP64 tile kernels: first exchange re-read per quartet
  template <typename R>
  __host__ __device__ static __forceinline__ void vrr(const R (&F)[L + 1], const VrrPar<R>& p, R (&acc)[NACC]) {
    const R v000_000_3 = F[3];
    const R v000_000_2 = F[2];
    const R v000_000_1 = F[1];
    const R v000_000_0 = F[0];
    const R v001_000_2 = p.PA[2] * v000_000_2 + p.WP[2] * v000_000_3;
    const R v010_000_2 = p.PA[1] * v000_000_2 + p.WP[1] * v000_000_3;
    const R v100_000_2 = p.PA[0] * v000_000_2 + p.WP[0] * v000_000_3;
    const R v001_000_1 = p.PA[2] * v000_000_1 + p.WP[2] * v000_000_2;
    const R v010_000_1 = p.PA[1] * v000_000_1 + p.WP[1] * v000_000_2;
    const R v100_000_1 = p.PA[0] * v000_000_1 + p.WP[0] * v000_000_2;
    const R v001_000_0 = p.PA[2] * v000_000_0 + p.WP[2] * v000_000_1;
    const R v010_000_0 = p.PA[1] * v000_000_0 + p.WP[1] * v000_000_1;
    const R v100_000_0 = p.PA[0] * v000_000_0 + p.WP[0] * v000_000_1;
    const R v002_000_1 = p.PA[2] * v001_000_1 + p.WP[2] * v001_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
    const R v011_000_1 = p.PA[1] * v001_000_1 + p.WP[1] * v001_000_2;
    const R v020_000_1 = p.PA[1] * v010_000_1 + p.WP[1] * v010_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
    const R v200_000_1 = p.PA[0] * v100_000_1 + p.WP[0] * v100_000_2 + R(1) * p.oo2z * (v000_000_1 - p.rz * v000_000_2);
    const R v002_000_0 = p.PA[2] * v001_000_0 + p.WP[2] * v001_000_1 + R(1) * p.oo2z * (v000_000_0 - p.rz * v000_000_1);
    const R v011_000_0 = p.PA[1] * v001_000_0 + p.WP[1] * v001_000_1;
    const R v020_000_0 = p.PA[1] * v010_000_0 + p.WP[1] * v010_000_1 + R(1) * p.oo2z * (v000_000_0 - p.rz * v000_000_1);
    const R v200_000_0 = p.PA[0] * v100_000_0 + p.WP[0] * v100_000_1 + R(1) * p.oo2z * (v000_000_0 - p.rz * v000_000_1);
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
  }
};
}  // namespace qf
