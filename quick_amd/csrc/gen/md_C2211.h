// Generated by quick_amd/codegen/gen_md.py - do not edit.
#pragma once
#include "../qf_md.h"
namespace qf {
// (dd|pp): 84 Hermite Coulomb integrals, 336 bra products
struct C2211Md {
  static constexpr int La = 2, Lb = 2, Lc = 1, Ld = 1, L = 6;
  static constexpr int N1 = 27, NE = 336;   // 1D entries per direction, product table
  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16
  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p
  template <class T>
  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, T out) {
    const double be010 = Y;
    const double be011 = h;
    const double be020 = fma(1.0, be011, be010 * Y);
    const double be021 = fma(be010, h, be011 * Y);
    const double be022 = be011 * h;
    const double be100 = X;
    const double be101 = h;
    const double be110 = fma(1.0, be101, be100 * Y);
    const double be111 = fma(be100, h, be101 * Y);
    const double be112 = be101 * h;
    const double be120 = fma(1.0, be111, be110 * Y);
    const double be121 = fma(2.0, be112, fma(be110, h, be111 * Y));
    const double be122 = fma(be111, h, be112 * Y);
    const double be123 = be112 * h;
    const double be200 = fma(1.0, be101, be100 * X);
    const double be201 = fma(be100, h, be101 * X);
    const double be202 = be101 * h;
    const double be210 = fma(1.0, be201, be200 * Y);
    const double be211 = fma(2.0, be202, fma(be200, h, be201 * Y));
    const double be212 = fma(be201, h, be202 * Y);
    const double be213 = be202 * h;
    const double be220 = fma(1.0, be211, be210 * Y);
    const double be221 = fma(2.0, be212, fma(be210, h, be211 * Y));
    const double be222 = fma(3.0, be213, fma(be211, h, be212 * Y));
    const double be223 = fma(be212, h, be213 * Y);
    const double be224 = be213 * h;
    out[0] = 1.0;
    out[1] = be010;
    out[2] = be011;
    out[3] = be020;
    out[4] = be021;
    out[5] = be022;
    out[6] = be100;
    out[7] = be101;
    out[8] = be110;
    out[9] = be111;
    out[10] = be112;
    out[11] = be120;
    out[12] = be121;
    out[13] = be122;
    out[14] = be123;
    out[15] = be200;
    out[16] = be201;
    out[17] = be202;
    out[18] = be210;
    out[19] = be211;
    out[20] = be212;
    out[21] = be213;
    out[22] = be220;
    out[23] = be221;
    out[24] = be222;
    out[25] = be223;
    out[26] = be224;
  }
  // Dbc and Dbd with the cons of b; oc, od: first elements of the a-c and a-d blocks of P
  template <class ET, class PT, class PU>
  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a, const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[9], const double (&Dbc)[18], const double (&Dbd)[18], double (&Jcd)[9], double (&Kbc)[18], double (&Kbd)[18], double (&Jab)[36], double (&Kac)[18], double (&Kad)[18]) {
    double am = pref;
    const double r000_0 = F[0] * am;
    am *= m2a;
    const double r000_1 = F[1] * am;
    am *= m2a;
    const double r000_2 = F[2] * am;
    am *= m2a;
    const double r000_3 = F[3] * am;
    am *= m2a;
    const double r000_4 = F[4] * am;
    am *= m2a;
    const double r000_5 = F[5] * am;
    am *= m2a;
    const double r000_6 = F[6] * am;
    const double r100_5 = PQ[0] * r000_6;
    const double r010_5 = PQ[1] * r000_6;
    const double r001_5 = PQ[2] * r000_6;
    const double r100_4 = PQ[0] * r000_5;
    const double r010_4 = PQ[1] * r000_5;
    const double r001_4 = PQ[2] * r000_5;
    const double r200_4 = fma(1.0, r000_5, PQ[0] * r100_5);
    const double r110_4 = PQ[0] * r010_5;
    const double r101_4 = PQ[0] * r001_5;
    const double r020_4 = fma(1.0, r000_5, PQ[1] * r010_5);
    const double r011_4 = PQ[1] * r001_5;
    const double r002_4 = fma(1.0, r000_5, PQ[2] * r001_5);
    const double r100_3 = PQ[0] * r000_4;
    const double r010_3 = PQ[1] * r000_4;
    const double r001_3 = PQ[2] * r000_4;
    const double r200_3 = fma(1.0, r000_4, PQ[0] * r100_4);
    const double r110_3 = PQ[0] * r010_4;
    const double r101_3 = PQ[0] * r001_4;
    const double r020_3 = fma(1.0, r000_4, PQ[1] * r010_4);
    const double r011_3 = PQ[1] * r001_4;
    const double r002_3 = fma(1.0, r000_4, PQ[2] * r001_4);
    const double r300_3 = fma(2.0, r100_4, PQ[0] * r200_4);
    const double r210_3 = PQ[1] * r200_4;
    const double r201_3 = PQ[2] * r200_4;
    const double r120_3 = PQ[0] * r020_4;
    const double r111_3 = PQ[0] * r011_4;
    const double r102_3 = PQ[0] * r002_4;
    const double r030_3 = fma(2.0, r010_4, PQ[1] * r020_4);
    const double r021_3 = PQ[2] * r020_4;
    const double r012_3 = PQ[1] * r002_4;
    const double r003_3 = fma(2.0, r001_4, PQ[2] * r002_4);
    const double r100_2 = PQ[0] * r000_3;
    const double r010_2 = PQ[1] * r000_3;
    const double r001_2 = PQ[2] * r000_3;
    const double r200_2 = fma(1.0, r000_3, PQ[0] * r100_3);
    const double r110_2 = PQ[0] * r010_3;
    const double r101_2 = PQ[0] * r001_3;
    const double r020_2 = fma(1.0, r000_3, PQ[1] * r010_3);
    const double r011_2 = PQ[1] * r001_3;
    const double r002_2 = fma(1.0, r000_3, PQ[2] * r001_3);
    const double r300_2 = fma(2.0, r100_3, PQ[0] * r200_3);
    const double r210_2 = PQ[1] * r200_3;
    const double r201_2 = PQ[2] * r200_3;
    const double r120_2 = PQ[0] * r020_3;
    const double r111_2 = PQ[0] * r011_3;
    const double r102_2 = PQ[0] * r002_3;
    const double r030_2 = fma(2.0, r010_3, PQ[1] * r020_3);
    const double r021_2 = PQ[2] * r020_3;
    const double r012_2 = PQ[1] * r002_3;
    const double r003_2 = fma(2.0, r001_3, PQ[2] * r002_3);
    const double r400_2 = fma(3.0, r200_3, PQ[0] * r300_3);
    const double r310_2 = PQ[1] * r300_3;
    const double r301_2 = PQ[2] * r300_3;
    const double r220_2 = fma(1.0, r020_3, PQ[0] * r120_3);
    const double r211_2 = PQ[1] * r201_3;
    const double r202_2 = fma(1.0, r002_3, PQ[0] * r102_3);
    const double r130_2 = PQ[0] * r030_3;
    const double r121_2 = PQ[0] * r021_3;
    const double r112_2 = PQ[0] * r012_3;
    const double r103_2 = PQ[0] * r003_3;
    const double r040_2 = fma(3.0, r020_3, PQ[1] * r030_3);
    const double r031_2 = PQ[2] * r030_3;
    const double r022_2 = fma(1.0, r002_3, PQ[1] * r012_3);
    const double r013_2 = PQ[1] * r003_3;
    const double r004_2 = fma(3.0, r002_3, PQ[2] * r003_3);
    const double r100_1 = PQ[0] * r000_2;
    const double r010_1 = PQ[1] * r000_2;
    const double r001_1 = PQ[2] * r000_2;
    const double r200_1 = fma(1.0, r000_2, PQ[0] * r100_2);
    const double r110_1 = PQ[0] * r010_2;
    const double r101_1 = PQ[0] * r001_2;
    const double r020_1 = fma(1.0, r000_2, PQ[1] * r010_2);
    const double r011_1 = PQ[1] * r001_2;
    const double r002_1 = fma(1.0, r000_2, PQ[2] * r001_2);
    const double r300_1 = fma(2.0, r100_2, PQ[0] * r200_2);
    const double r210_1 = PQ[1] * r200_2;
    const double r201_1 = PQ[2] * r200_2;
    const double r120_1 = PQ[0] * r020_2;
    const double r111_1 = PQ[0] * r011_2;
    const double r102_1 = PQ[0] * r002_2;
    const double r030_1 = fma(2.0, r010_2, PQ[1] * r020_2);
    const double r021_1 = PQ[2] * r020_2;
    const double r012_1 = PQ[1] * r002_2;
    const double r003_1 = fma(2.0, r001_2, PQ[2] * r002_2);
    const double r400_1 = fma(3.0, r200_2, PQ[0] * r300_2);
    const double r310_1 = PQ[1] * r300_2;
    const double r301_1 = PQ[2] * r300_2;
    const double r220_1 = fma(1.0, r020_2, PQ[0] * r120_2);
    const double r211_1 = PQ[1] * r201_2;
    const double r202_1 = fma(1.0, r002_2, PQ[0] * r102_2);
    const double r130_1 = PQ[0] * r030_2;
    const double r121_1 = PQ[0] * r021_2;
    const double r112_1 = PQ[0] * r012_2;
    const double r103_1 = PQ[0] * r003_2;
    const double r040_1 = fma(3.0, r020_2, PQ[1] * r030_2);
    const double r031_1 = PQ[2] * r030_2;
    const double r022_1 = fma(1.0, r002_2, PQ[1] * r012_2);
    const double r013_1 = PQ[1] * r003_2;
    const double r004_1 = fma(3.0, r002_2, PQ[2] * r003_2);
    const double r500_1 = fma(4.0, r300_2, PQ[0] * r400_2);
    const double r410_1 = PQ[1] * r400_2;
    const double r401_1 = PQ[2] * r400_2;
    const double r320_1 = fma(1.0, r300_2, PQ[1] * r310_2);
    const double r311_1 = PQ[1] * r301_2;
    const double r302_1 = fma(1.0, r300_2, PQ[2] * r301_2);
    const double r230_1 = fma(1.0, r030_2, PQ[0] * r130_2);
    const double r221_1 = PQ[2] * r220_2;
    const double r212_1 = PQ[1] * r202_2;
    const double r203_1 = fma(1.0, r003_2, PQ[0] * r103_2);
    const double r140_1 = PQ[0] * r040_2;
    const double r131_1 = PQ[0] * r031_2;
    const double r122_1 = PQ[0] * r022_2;
    const double r113_1 = PQ[0] * r013_2;
    const double r104_1 = PQ[0] * r004_2;
    const double r050_1 = fma(4.0, r030_2, PQ[1] * r040_2);
    const double r041_1 = PQ[2] * r040_2;
    const double r032_1 = fma(1.0, r030_2, PQ[2] * r031_2);
    const double r023_1 = fma(1.0, r003_2, PQ[1] * r013_2);
    const double r014_1 = PQ[1] * r004_2;
    const double r005_1 = fma(4.0, r003_2, PQ[2] * r004_2);
    const double r100_0 = PQ[0] * r000_1;
    const double r010_0 = PQ[1] * r000_1;
    const double r001_0 = PQ[2] * r000_1;
    const double r200_0 = fma(1.0, r000_1, PQ[0] * r100_1);
    const double r110_0 = PQ[0] * r010_1;
    const double r101_0 = PQ[0] * r001_1;
    const double r020_0 = fma(1.0, r000_1, PQ[1] * r010_1);
    const double r011_0 = PQ[1] * r001_1;
    const double r002_0 = fma(1.0, r000_1, PQ[2] * r001_1);
    const double r300_0 = fma(2.0, r100_1, PQ[0] * r200_1);
    const double r210_0 = PQ[1] * r200_1;
    const double r201_0 = PQ[2] * r200_1;
    const double r120_0 = PQ[0] * r020_1;
    const double r111_0 = PQ[0] * r011_1;
    const double r102_0 = PQ[0] * r002_1;
    const double r030_0 = fma(2.0, r010_1, PQ[1] * r020_1);
    const double r021_0 = PQ[2] * r020_1;
    const double r012_0 = PQ[1] * r002_1;
    const double r003_0 = fma(2.0, r001_1, PQ[2] * r002_1);
    const double r400_0 = fma(3.0, r200_1, PQ[0] * r300_1);
    const double r310_0 = PQ[1] * r300_1;
    const double r301_0 = PQ[2] * r300_1;
    const double r220_0 = fma(1.0, r020_1, PQ[0] * r120_1);
    const double r211_0 = PQ[1] * r201_1;
    const double r202_0 = fma(1.0, r002_1, PQ[0] * r102_1);
    const double r130_0 = PQ[0] * r030_1;
    const double r121_0 = PQ[0] * r021_1;
    const double r112_0 = PQ[0] * r012_1;
    const double r103_0 = PQ[0] * r003_1;
    const double r040_0 = fma(3.0, r020_1, PQ[1] * r030_1);
    const double r031_0 = PQ[2] * r030_1;
    const double r022_0 = fma(1.0, r002_1, PQ[1] * r012_1);
    const double r013_0 = PQ[1] * r003_1;
    const double r004_0 = fma(3.0, r002_1, PQ[2] * r003_1);
    const double r500_0 = fma(4.0, r300_1, PQ[0] * r400_1);
    const double r410_0 = PQ[1] * r400_1;
    const double r401_0 = PQ[2] * r400_1;
    const double r320_0 = fma(1.0, r300_1, PQ[1] * r310_1);
    const double r311_0 = PQ[1] * r301_1;
    const double r302_0 = fma(1.0, r300_1, PQ[2] * r301_1);
    const double r230_0 = fma(1.0, r030_1, PQ[0] * r130_1);
    const double r221_0 = PQ[2] * r220_1;
    const double r212_0 = PQ[1] * r202_1;
    const double r203_0 = fma(1.0, r003_1, PQ[0] * r103_1);
    const double r140_0 = PQ[0] * r040_1;
    const double r131_0 = PQ[0] * r031_1;
    const double r122_0 = PQ[0] * r022_1;
    const double r113_0 = PQ[0] * r013_1;
    const double r104_0 = PQ[0] * r004_1;
    const double r050_0 = fma(4.0, r030_1, PQ[1] * r040_1);
    const double r041_0 = PQ[2] * r040_1;
    const double r032_0 = fma(1.0, r030_1, PQ[2] * r031_1);
    const double r023_0 = fma(1.0, r003_1, PQ[1] * r013_1);
    const double r014_0 = PQ[1] * r004_1;
    const double r005_0 = fma(4.0, r003_1, PQ[2] * r004_1);
    const double r600_0 = fma(5.0, r400_1, PQ[0] * r500_1);
    const double r510_0 = PQ[1] * r500_1;
    const double r501_0 = PQ[2] * r500_1;
    const double r420_0 = fma(1.0, r400_1, PQ[1] * r410_1);
    const double r411_0 = PQ[1] * r401_1;
    const double r402_0 = fma(1.0, r400_1, PQ[2] * r401_1);
    const double r330_0 = fma(2.0, r130_1, PQ[0] * r230_1);
    const double r321_0 = PQ[2] * r320_1;
    const double r312_0 = PQ[1] * r302_1;
    const double r303_0 = fma(2.0, r103_1, PQ[0] * r203_1);
    const double r240_0 = fma(1.0, r040_1, PQ[0] * r140_1);
    const double r231_0 = PQ[2] * r230_1;
    const double r222_0 = fma(1.0, r022_1, PQ[0] * r122_1);
    const double r213_0 = PQ[1] * r203_1;
    const double r204_0 = fma(1.0, r004_1, PQ[0] * r104_1);
    const double r150_0 = PQ[0] * r050_1;
    const double r141_0 = PQ[0] * r041_1;
    const double r132_0 = PQ[0] * r032_1;
    const double r123_0 = PQ[0] * r023_1;
    const double r114_0 = PQ[0] * r014_1;
    const double r105_0 = PQ[0] * r005_1;
    const double r060_0 = fma(5.0, r040_1, PQ[1] * r050_1);
    const double r051_0 = PQ[2] * r050_1;
    const double r042_0 = fma(1.0, r040_1, PQ[2] * r041_1);
    const double r033_0 = fma(2.0, r013_1, PQ[1] * r023_1);
    const double r024_0 = fma(1.0, r004_1, PQ[1] * r014_1);
    const double r015_0 = PQ[1] * r005_1;
    const double r006_0 = fma(5.0, r004_1, PQ[2] * r005_1);
    const double kxe010 = QD[0];
    const double kxe011 = (-hk);
    const double kxe100 = QC[0];
    const double kxe101 = (-hk);
    const double kxe110 = fma(-1.0, kxe101, kxe100 * QD[0]);
    const double kxe111 = fma(kxe100, (-hk), kxe101 * QD[0]);
    const double kxe112 = kxe101 * (-hk);
    const double kye010 = QD[1];
    const double kye011 = (-hk);
    const double kye100 = QC[1];
    const double kye101 = (-hk);
    const double kye110 = fma(-1.0, kye101, kye100 * QD[1]);
    const double kye111 = fma(kye100, (-hk), kye101 * QD[1]);
    const double kye112 = kye101 * (-hk);
    const double kze010 = QD[2];
    const double kze011 = (-hk);
    const double kze100 = QC[2];
    const double kze101 = (-hk);
    const double kze110 = fma(-1.0, kze101, kze100 * QD[2]);
    const double kze111 = fma(kze100, (-hk), kze101 * QD[2]);
    const double kze112 = kze101 * (-hk);
    const double k0_0_000 = kxe110 * (kCons[1][0] * kCons[1][0]);
    const double k0_0_100 = kxe111 * (kCons[1][0] * kCons[1][0]);
    const double k0_0_200 = kxe112 * (kCons[1][0] * kCons[1][0]);
    const double k0_1_000 = kxe100 * kye010 * (kCons[1][0] * kCons[1][1]);
    const double k0_1_010 = kxe100 * kye011 * (kCons[1][0] * kCons[1][1]);
    const double k0_1_100 = kxe101 * kye010 * (kCons[1][0] * kCons[1][1]);
    const double k0_1_110 = kxe101 * kye011 * (kCons[1][0] * kCons[1][1]);
    const double k0_2_000 = kxe100 * kze010 * (kCons[1][0] * kCons[1][2]);
    const double k0_2_001 = kxe100 * kze011 * (kCons[1][0] * kCons[1][2]);
    const double k0_2_100 = kxe101 * kze010 * (kCons[1][0] * kCons[1][2]);
    const double k0_2_101 = kxe101 * kze011 * (kCons[1][0] * kCons[1][2]);
    const double k1_0_000 = kxe010 * kye100 * (kCons[1][1] * kCons[1][0]);
    const double k1_0_010 = kxe010 * kye101 * (kCons[1][1] * kCons[1][0]);
    const double k1_0_100 = kxe011 * kye100 * (kCons[1][1] * kCons[1][0]);
    const double k1_0_110 = kxe011 * kye101 * (kCons[1][1] * kCons[1][0]);
    const double k1_1_000 = kye110 * (kCons[1][1] * kCons[1][1]);
    const double k1_1_010 = kye111 * (kCons[1][1] * kCons[1][1]);
    const double k1_1_020 = kye112 * (kCons[1][1] * kCons[1][1]);
    const double k1_2_000 = kye100 * kze010 * (kCons[1][1] * kCons[1][2]);
    const double k1_2_001 = kye100 * kze011 * (kCons[1][1] * kCons[1][2]);
    const double k1_2_010 = kye101 * kze010 * (kCons[1][1] * kCons[1][2]);
    const double k1_2_011 = kye101 * kze011 * (kCons[1][1] * kCons[1][2]);
    const double k2_0_000 = kxe010 * kze100 * (kCons[1][2] * kCons[1][0]);
    const double k2_0_001 = kxe010 * kze101 * (kCons[1][2] * kCons[1][0]);
    const double k2_0_100 = kxe011 * kze100 * (kCons[1][2] * kCons[1][0]);
    const double k2_0_101 = kxe011 * kze101 * (kCons[1][2] * kCons[1][0]);
    const double k2_1_000 = kye010 * kze100 * (kCons[1][2] * kCons[1][1]);
    const double k2_1_001 = kye010 * kze101 * (kCons[1][2] * kCons[1][1]);
    const double k2_1_010 = kye011 * kze100 * (kCons[1][2] * kCons[1][1]);
    const double k2_1_011 = kye011 * kze101 * (kCons[1][2] * kCons[1][1]);
    const double k2_2_000 = kze110 * (kCons[1][2] * kCons[1][2]);
    const double k2_2_001 = kze111 * (kCons[1][2] * kCons[1][2]);
    const double k2_2_002 = kze112 * (kCons[1][2] * kCons[1][2]);
    QF_OPAQUE(oc);
    QF_OPAQUE(od);
    {
      const double ac0 = P[oc + 0 * n + 0] * kCons[2][0];
      const double ac1 = P[oc + 0 * n + 1] * kCons[2][0];
      const double ac2 = P[oc + 0 * n + 2] * kCons[2][0];
      const double ad0 = P[od + 0 * n + 0] * kCons[2][0];
      const double ad1 = P[od + 0 * n + 1] * kCons[2][0];
      const double ad2 = P[od + 0 * n + 2] * kCons[2][0];
      {
        const double ab = Pab[0 * n + 0] * (kCons[2][0] * kCons[2][0]);
        const double e0 = E[0];
        const double e1 = E[1];
        const double e2 = E[2];
        const double e3 = E[3];
        const double e4 = E[4];
        const double z000 = fma(e4, r400_0, fma(e3, r300_0, fma(e2, r200_0, fma(e1, r100_0, e0 * r000_0))));
        const double z001 = fma(e4, r401_0, fma(e3, r301_0, fma(e2, r201_0, fma(e1, r101_0, e0 * r001_0))));
        const double z010 = fma(e4, r410_0, fma(e3, r310_0, fma(e2, r210_0, fma(e1, r110_0, e0 * r010_0))));
        const double z100 = fma(e4, r500_0, fma(e3, r400_0, fma(e2, r300_0, fma(e1, r200_0, e0 * r100_0))));
        const double z002 = fma(e4, r402_0, fma(e3, r302_0, fma(e2, r202_0, fma(e1, r102_0, e0 * r002_0))));
        const double z011 = fma(e4, r411_0, fma(e3, r311_0, fma(e2, r211_0, fma(e1, r111_0, e0 * r011_0))));
        const double z020 = fma(e4, r420_0, fma(e3, r320_0, fma(e2, r220_0, fma(e1, r120_0, e0 * r020_0))));
        const double z101 = fma(e4, r501_0, fma(e3, r401_0, fma(e2, r301_0, fma(e1, r201_0, e0 * r101_0))));
        const double z110 = fma(e4, r510_0, fma(e3, r410_0, fma(e2, r310_0, fma(e1, r210_0, e0 * r110_0))));
        const double z200 = fma(e4, r600_0, fma(e3, r500_0, fma(e2, r400_0, fma(e1, r300_0, e0 * r200_0))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[0], v, Kac[0]);
          Kad[0] = fma(Dbc[0], v, Kad[0]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[1], v, Kac[0]);
          Kad[1] = fma(Dbc[0], v, Kad[1]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[2], v, Kac[0]);
          Kad[2] = fma(Dbc[0], v, Kad[2]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[0], v, Kac[1]);
          Kad[0] = fma(Dbc[1], v, Kad[0]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[1], v, Kac[1]);
          Kad[1] = fma(Dbc[1], v, Kad[1]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[2], v, Kac[1]);
          Kad[2] = fma(Dbc[1], v, Kad[2]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[0], v, Kac[2]);
          Kad[0] = fma(Dbc[2], v, Kad[0]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[1], v, Kac[2]);
          Kad[1] = fma(Dbc[2], v, Kad[1]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[2], v, Kac[2]);
          Kad[2] = fma(Dbc[2], v, Kad[2]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        Jab[0] += j;
      }
      {
        const double ab = Pab[0 * n + 1] * (kCons[2][0] * kCons[2][1]);
        const double e0 = E[5];
        const double e1 = E[6];
        const double e2 = E[7];
        const double e3 = E[8];
        const double e4 = E[9];
        const double e5 = E[10];
        const double e6 = E[11];
        const double e7 = E[12];
        const double z000 = fma(e7, r310_0, fma(e6, r300_0, fma(e5, r210_0, fma(e4, r200_0, fma(e3, r110_0, fma(e2, r100_0, fma(e1, r010_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r311_0, fma(e6, r301_0, fma(e5, r211_0, fma(e4, r201_0, fma(e3, r111_0, fma(e2, r101_0, fma(e1, r011_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r320_0, fma(e6, r310_0, fma(e5, r220_0, fma(e4, r210_0, fma(e3, r120_0, fma(e2, r110_0, fma(e1, r020_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r410_0, fma(e6, r400_0, fma(e5, r310_0, fma(e4, r300_0, fma(e3, r210_0, fma(e2, r200_0, fma(e1, r110_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r312_0, fma(e6, r302_0, fma(e5, r212_0, fma(e4, r202_0, fma(e3, r112_0, fma(e2, r102_0, fma(e1, r012_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r321_0, fma(e6, r311_0, fma(e5, r221_0, fma(e4, r211_0, fma(e3, r121_0, fma(e2, r111_0, fma(e1, r021_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r330_0, fma(e6, r320_0, fma(e5, r230_0, fma(e4, r220_0, fma(e3, r130_0, fma(e2, r120_0, fma(e1, r030_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r411_0, fma(e6, r401_0, fma(e5, r311_0, fma(e4, r301_0, fma(e3, r211_0, fma(e2, r201_0, fma(e1, r111_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r420_0, fma(e6, r410_0, fma(e5, r320_0, fma(e4, r310_0, fma(e3, r220_0, fma(e2, r210_0, fma(e1, r120_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r510_0, fma(e6, r500_0, fma(e5, r410_0, fma(e4, r400_0, fma(e3, r310_0, fma(e2, r300_0, fma(e1, r210_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[3], v, Kac[0]);
          Kad[0] = fma(Dbc[3], v, Kad[0]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[4], v, Kac[0]);
          Kad[1] = fma(Dbc[3], v, Kad[1]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[5], v, Kac[0]);
          Kad[2] = fma(Dbc[3], v, Kad[2]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[3], v, Kac[1]);
          Kad[0] = fma(Dbc[4], v, Kad[0]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[4], v, Kac[1]);
          Kad[1] = fma(Dbc[4], v, Kad[1]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[5], v, Kac[1]);
          Kad[2] = fma(Dbc[4], v, Kad[2]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[3], v, Kac[2]);
          Kad[0] = fma(Dbc[5], v, Kad[0]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[4], v, Kac[2]);
          Kad[1] = fma(Dbc[5], v, Kad[1]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[5], v, Kac[2]);
          Kad[2] = fma(Dbc[5], v, Kad[2]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        Jab[1] += j;
      }
      {
        const double ab = Pab[0 * n + 2] * (kCons[2][0] * kCons[2][2]);
        const double e0 = E[13];
        const double e1 = E[14];
        const double e2 = E[15];
        const double e3 = E[16];
        const double e4 = E[17];
        const double e5 = E[18];
        const double e6 = E[19];
        const double e7 = E[20];
        const double e8 = E[21];
        const double z000 = fma(e8, r220_0, fma(e7, r210_0, fma(e6, r200_0, fma(e5, r120_0, fma(e4, r110_0, fma(e3, r100_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r221_0, fma(e7, r211_0, fma(e6, r201_0, fma(e5, r121_0, fma(e4, r111_0, fma(e3, r101_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r230_0, fma(e7, r220_0, fma(e6, r210_0, fma(e5, r130_0, fma(e4, r120_0, fma(e3, r110_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r320_0, fma(e7, r310_0, fma(e6, r300_0, fma(e5, r220_0, fma(e4, r210_0, fma(e3, r200_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r222_0, fma(e7, r212_0, fma(e6, r202_0, fma(e5, r122_0, fma(e4, r112_0, fma(e3, r102_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r231_0, fma(e7, r221_0, fma(e6, r211_0, fma(e5, r131_0, fma(e4, r121_0, fma(e3, r111_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r240_0, fma(e7, r230_0, fma(e6, r220_0, fma(e5, r140_0, fma(e4, r130_0, fma(e3, r120_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r321_0, fma(e7, r311_0, fma(e6, r301_0, fma(e5, r221_0, fma(e4, r211_0, fma(e3, r201_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r330_0, fma(e7, r320_0, fma(e6, r310_0, fma(e5, r230_0, fma(e4, r220_0, fma(e3, r210_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r420_0, fma(e7, r410_0, fma(e6, r400_0, fma(e5, r320_0, fma(e4, r310_0, fma(e3, r300_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[6], v, Kac[0]);
          Kad[0] = fma(Dbc[6], v, Kad[0]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[7], v, Kac[0]);
          Kad[1] = fma(Dbc[6], v, Kad[1]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[8], v, Kac[0]);
          Kad[2] = fma(Dbc[6], v, Kad[2]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[6], v, Kac[1]);
          Kad[0] = fma(Dbc[7], v, Kad[0]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[7], v, Kac[1]);
          Kad[1] = fma(Dbc[7], v, Kad[1]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[8], v, Kac[1]);
          Kad[2] = fma(Dbc[7], v, Kad[2]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[6], v, Kac[2]);
          Kad[0] = fma(Dbc[8], v, Kad[0]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[7], v, Kac[2]);
          Kad[1] = fma(Dbc[8], v, Kad[1]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[8], v, Kac[2]);
          Kad[2] = fma(Dbc[8], v, Kad[2]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        Jab[2] += j;
      }
      {
        const double ab = Pab[0 * n + 3] * (kCons[2][0] * kCons[2][3]);
        const double e0 = E[22];
        const double e1 = E[23];
        const double e2 = E[24];
        const double e3 = E[25];
        const double e4 = E[26];
        const double e5 = E[27];
        const double e6 = E[28];
        const double e7 = E[29];
        const double z000 = fma(e7, r301_0, fma(e6, r300_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r101_0, fma(e2, r100_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r302_0, fma(e6, r301_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r102_0, fma(e2, r101_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r311_0, fma(e6, r310_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r401_0, fma(e6, r400_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r201_0, fma(e2, r200_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r303_0, fma(e6, r302_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r312_0, fma(e6, r311_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r321_0, fma(e6, r320_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r402_0, fma(e6, r401_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r202_0, fma(e2, r201_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r411_0, fma(e6, r410_0, fma(e5, r311_0, fma(e4, r310_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r501_0, fma(e6, r500_0, fma(e5, r401_0, fma(e4, r400_0, fma(e3, r301_0, fma(e2, r300_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[9], v, Kac[0]);
          Kad[0] = fma(Dbc[9], v, Kad[0]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[9] = fma(ac0, v, Kbd[9]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[10], v, Kac[0]);
          Kad[1] = fma(Dbc[9], v, Kad[1]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[10] = fma(ac0, v, Kbd[10]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[11], v, Kac[0]);
          Kad[2] = fma(Dbc[9], v, Kad[2]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[11] = fma(ac0, v, Kbd[11]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[9], v, Kac[1]);
          Kad[0] = fma(Dbc[10], v, Kad[0]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[9] = fma(ac1, v, Kbd[9]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[10], v, Kac[1]);
          Kad[1] = fma(Dbc[10], v, Kad[1]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[10] = fma(ac1, v, Kbd[10]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[11], v, Kac[1]);
          Kad[2] = fma(Dbc[10], v, Kad[2]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[11] = fma(ac1, v, Kbd[11]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[9], v, Kac[2]);
          Kad[0] = fma(Dbc[11], v, Kad[0]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[9] = fma(ac2, v, Kbd[9]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[10], v, Kac[2]);
          Kad[1] = fma(Dbc[11], v, Kad[1]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[10] = fma(ac2, v, Kbd[10]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[11], v, Kac[2]);
          Kad[2] = fma(Dbc[11], v, Kad[2]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[11] = fma(ac2, v, Kbd[11]);
        }
        Jab[3] += j;
      }
      {
        const double ab = Pab[0 * n + 4] * (kCons[2][0] * kCons[2][4]);
        const double e0 = E[30];
        const double e1 = E[31];
        const double e2 = E[32];
        const double e3 = E[33];
        const double e4 = E[34];
        const double e5 = E[35];
        const double e6 = E[36];
        const double e7 = E[37];
        const double e8 = E[38];
        const double e9 = E[39];
        const double e10 = E[40];
        const double e11 = E[41];
        const double z000 = fma(e11, r211_0, fma(e10, r210_0, fma(e9, r201_0, fma(e8, r200_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r202_0, fma(e8, r201_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r311_0, fma(e10, r310_0, fma(e9, r301_0, fma(e8, r300_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r203_0, fma(e8, r202_0, fma(e7, r113_0, fma(e6, r112_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r122_0, fma(e6, r121_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r302_0, fma(e8, r301_0, fma(e7, r212_0, fma(e6, r211_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r411_0, fma(e10, r410_0, fma(e9, r401_0, fma(e8, r400_0, fma(e7, r311_0, fma(e6, r310_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[12], v, Kac[0]);
          Kad[0] = fma(Dbc[12], v, Kad[0]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[12] = fma(ac0, v, Kbd[12]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[13], v, Kac[0]);
          Kad[1] = fma(Dbc[12], v, Kad[1]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[13] = fma(ac0, v, Kbd[13]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[14], v, Kac[0]);
          Kad[2] = fma(Dbc[12], v, Kad[2]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[14] = fma(ac0, v, Kbd[14]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[12], v, Kac[1]);
          Kad[0] = fma(Dbc[13], v, Kad[0]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[12] = fma(ac1, v, Kbd[12]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[13], v, Kac[1]);
          Kad[1] = fma(Dbc[13], v, Kad[1]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[13] = fma(ac1, v, Kbd[13]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[14], v, Kac[1]);
          Kad[2] = fma(Dbc[13], v, Kad[2]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[14] = fma(ac1, v, Kbd[14]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[12], v, Kac[2]);
          Kad[0] = fma(Dbc[14], v, Kad[0]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[12] = fma(ac2, v, Kbd[12]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[13], v, Kac[2]);
          Kad[1] = fma(Dbc[14], v, Kad[1]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[13] = fma(ac2, v, Kbd[13]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[14], v, Kac[2]);
          Kad[2] = fma(Dbc[14], v, Kad[2]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[14] = fma(ac2, v, Kbd[14]);
        }
        Jab[4] += j;
      }
      {
        const double ab = Pab[0 * n + 5] * (kCons[2][0] * kCons[2][5]);
        const double e0 = E[42];
        const double e1 = E[43];
        const double e2 = E[44];
        const double e3 = E[45];
        const double e4 = E[46];
        const double e5 = E[47];
        const double e6 = E[48];
        const double e7 = E[49];
        const double e8 = E[50];
        const double z000 = fma(e8, r202_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r100_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r203_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r101_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r212_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r302_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r200_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r204_0, fma(e7, r203_0, fma(e6, r202_0, fma(e5, r104_0, fma(e4, r103_0, fma(e3, r102_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r213_0, fma(e7, r212_0, fma(e6, r211_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r222_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r303_0, fma(e7, r302_0, fma(e6, r301_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r201_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r312_0, fma(e7, r311_0, fma(e6, r310_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r402_0, fma(e7, r401_0, fma(e6, r400_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r300_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[15], v, Kac[0]);
          Kad[0] = fma(Dbc[15], v, Kad[0]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[15] = fma(ac0, v, Kbd[15]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[16], v, Kac[0]);
          Kad[1] = fma(Dbc[15], v, Kad[1]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[16] = fma(ac0, v, Kbd[16]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[17], v, Kac[0]);
          Kad[2] = fma(Dbc[15], v, Kad[2]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[17] = fma(ac0, v, Kbd[17]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[15], v, Kac[1]);
          Kad[0] = fma(Dbc[16], v, Kad[0]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[15] = fma(ac1, v, Kbd[15]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[16], v, Kac[1]);
          Kad[1] = fma(Dbc[16], v, Kad[1]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[16] = fma(ac1, v, Kbd[16]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[17], v, Kac[1]);
          Kad[2] = fma(Dbc[16], v, Kad[2]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[17] = fma(ac1, v, Kbd[17]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[15], v, Kac[2]);
          Kad[0] = fma(Dbc[17], v, Kad[0]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[15] = fma(ac2, v, Kbd[15]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[16], v, Kac[2]);
          Kad[1] = fma(Dbc[17], v, Kad[1]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[16] = fma(ac2, v, Kbd[16]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[17], v, Kac[2]);
          Kad[2] = fma(Dbc[17], v, Kad[2]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[17] = fma(ac2, v, Kbd[17]);
        }
        Jab[5] += j;
      }
    }
    {
      const double ac0 = P[oc + 1 * n + 0] * kCons[2][1];
      const double ac1 = P[oc + 1 * n + 1] * kCons[2][1];
      const double ac2 = P[oc + 1 * n + 2] * kCons[2][1];
      const double ad0 = P[od + 1 * n + 0] * kCons[2][1];
      const double ad1 = P[od + 1 * n + 1] * kCons[2][1];
      const double ad2 = P[od + 1 * n + 2] * kCons[2][1];
      {
        const double ab = Pab[1 * n + 0] * (kCons[2][1] * kCons[2][0]);
        const double e0 = E[51];
        const double e1 = E[52];
        const double e2 = E[53];
        const double e3 = E[54];
        const double e4 = E[55];
        const double e5 = E[56];
        const double e6 = E[57];
        const double e7 = E[58];
        const double z000 = fma(e7, r310_0, fma(e6, r300_0, fma(e5, r210_0, fma(e4, r200_0, fma(e3, r110_0, fma(e2, r100_0, fma(e1, r010_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r311_0, fma(e6, r301_0, fma(e5, r211_0, fma(e4, r201_0, fma(e3, r111_0, fma(e2, r101_0, fma(e1, r011_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r320_0, fma(e6, r310_0, fma(e5, r220_0, fma(e4, r210_0, fma(e3, r120_0, fma(e2, r110_0, fma(e1, r020_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r410_0, fma(e6, r400_0, fma(e5, r310_0, fma(e4, r300_0, fma(e3, r210_0, fma(e2, r200_0, fma(e1, r110_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r312_0, fma(e6, r302_0, fma(e5, r212_0, fma(e4, r202_0, fma(e3, r112_0, fma(e2, r102_0, fma(e1, r012_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r321_0, fma(e6, r311_0, fma(e5, r221_0, fma(e4, r211_0, fma(e3, r121_0, fma(e2, r111_0, fma(e1, r021_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r330_0, fma(e6, r320_0, fma(e5, r230_0, fma(e4, r220_0, fma(e3, r130_0, fma(e2, r120_0, fma(e1, r030_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r411_0, fma(e6, r401_0, fma(e5, r311_0, fma(e4, r301_0, fma(e3, r211_0, fma(e2, r201_0, fma(e1, r111_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r420_0, fma(e6, r410_0, fma(e5, r320_0, fma(e4, r310_0, fma(e3, r220_0, fma(e2, r210_0, fma(e1, r120_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r510_0, fma(e6, r500_0, fma(e5, r410_0, fma(e4, r400_0, fma(e3, r310_0, fma(e2, r300_0, fma(e1, r210_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[3] = fma(Dbd[0], v, Kac[3]);
          Kad[3] = fma(Dbc[0], v, Kad[3]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[3] = fma(Dbd[1], v, Kac[3]);
          Kad[4] = fma(Dbc[0], v, Kad[4]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[3] = fma(Dbd[2], v, Kac[3]);
          Kad[5] = fma(Dbc[0], v, Kad[5]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[4] = fma(Dbd[0], v, Kac[4]);
          Kad[3] = fma(Dbc[1], v, Kad[3]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[4] = fma(Dbd[1], v, Kac[4]);
          Kad[4] = fma(Dbc[1], v, Kad[4]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[4] = fma(Dbd[2], v, Kac[4]);
          Kad[5] = fma(Dbc[1], v, Kad[5]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[5] = fma(Dbd[0], v, Kac[5]);
          Kad[3] = fma(Dbc[2], v, Kad[3]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[5] = fma(Dbd[1], v, Kac[5]);
          Kad[4] = fma(Dbc[2], v, Kad[4]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[5] = fma(Dbd[2], v, Kac[5]);
          Kad[5] = fma(Dbc[2], v, Kad[5]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        Jab[6] += j;
      }
      {
        const double ab = Pab[1 * n + 1] * (kCons[2][1] * kCons[2][1]);
        const double e0 = E[59];
        const double e1 = E[60];
        const double e2 = E[61];
        const double e3 = E[62];
        const double e4 = E[63];
        const double e5 = E[64];
        const double e6 = E[65];
        const double e7 = E[66];
        const double e8 = E[67];
        const double z000 = fma(e8, r220_0, fma(e7, r210_0, fma(e6, r200_0, fma(e5, r120_0, fma(e4, r110_0, fma(e3, r100_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r221_0, fma(e7, r211_0, fma(e6, r201_0, fma(e5, r121_0, fma(e4, r111_0, fma(e3, r101_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r230_0, fma(e7, r220_0, fma(e6, r210_0, fma(e5, r130_0, fma(e4, r120_0, fma(e3, r110_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r320_0, fma(e7, r310_0, fma(e6, r300_0, fma(e5, r220_0, fma(e4, r210_0, fma(e3, r200_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r222_0, fma(e7, r212_0, fma(e6, r202_0, fma(e5, r122_0, fma(e4, r112_0, fma(e3, r102_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r231_0, fma(e7, r221_0, fma(e6, r211_0, fma(e5, r131_0, fma(e4, r121_0, fma(e3, r111_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r240_0, fma(e7, r230_0, fma(e6, r220_0, fma(e5, r140_0, fma(e4, r130_0, fma(e3, r120_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r321_0, fma(e7, r311_0, fma(e6, r301_0, fma(e5, r221_0, fma(e4, r211_0, fma(e3, r201_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r330_0, fma(e7, r320_0, fma(e6, r310_0, fma(e5, r230_0, fma(e4, r220_0, fma(e3, r210_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r420_0, fma(e7, r410_0, fma(e6, r400_0, fma(e5, r320_0, fma(e4, r310_0, fma(e3, r300_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[3] = fma(Dbd[3], v, Kac[3]);
          Kad[3] = fma(Dbc[3], v, Kad[3]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[3] = fma(Dbd[4], v, Kac[3]);
          Kad[4] = fma(Dbc[3], v, Kad[4]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[3] = fma(Dbd[5], v, Kac[3]);
          Kad[5] = fma(Dbc[3], v, Kad[5]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[4] = fma(Dbd[3], v, Kac[4]);
          Kad[3] = fma(Dbc[4], v, Kad[3]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[4] = fma(Dbd[4], v, Kac[4]);
          Kad[4] = fma(Dbc[4], v, Kad[4]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[4] = fma(Dbd[5], v, Kac[4]);
          Kad[5] = fma(Dbc[4], v, Kad[5]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[5] = fma(Dbd[3], v, Kac[5]);
          Kad[3] = fma(Dbc[5], v, Kad[3]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[5] = fma(Dbd[4], v, Kac[5]);
          Kad[4] = fma(Dbc[5], v, Kad[4]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[5] = fma(Dbd[5], v, Kac[5]);
          Kad[5] = fma(Dbc[5], v, Kad[5]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        Jab[7] += j;
      }
      {
        const double ab = Pab[1 * n + 2] * (kCons[2][1] * kCons[2][2]);
        const double e0 = E[68];
        const double e1 = E[69];
        const double e2 = E[70];
        const double e3 = E[71];
        const double e4 = E[72];
        const double e5 = E[73];
        const double e6 = E[74];
        const double e7 = E[75];
        const double z000 = fma(e7, r130_0, fma(e6, r120_0, fma(e5, r110_0, fma(e4, r100_0, fma(e3, r030_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r131_0, fma(e6, r121_0, fma(e5, r111_0, fma(e4, r101_0, fma(e3, r031_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r140_0, fma(e6, r130_0, fma(e5, r120_0, fma(e4, r110_0, fma(e3, r040_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r230_0, fma(e6, r220_0, fma(e5, r210_0, fma(e4, r200_0, fma(e3, r130_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r132_0, fma(e6, r122_0, fma(e5, r112_0, fma(e4, r102_0, fma(e3, r032_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r141_0, fma(e6, r131_0, fma(e5, r121_0, fma(e4, r111_0, fma(e3, r041_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r150_0, fma(e6, r140_0, fma(e5, r130_0, fma(e4, r120_0, fma(e3, r050_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r231_0, fma(e6, r221_0, fma(e5, r211_0, fma(e4, r201_0, fma(e3, r131_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r240_0, fma(e6, r230_0, fma(e5, r220_0, fma(e4, r210_0, fma(e3, r140_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r330_0, fma(e6, r320_0, fma(e5, r310_0, fma(e4, r300_0, fma(e3, r230_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[3] = fma(Dbd[6], v, Kac[3]);
          Kad[3] = fma(Dbc[6], v, Kad[3]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[3] = fma(Dbd[7], v, Kac[3]);
          Kad[4] = fma(Dbc[6], v, Kad[4]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[3] = fma(Dbd[8], v, Kac[3]);
          Kad[5] = fma(Dbc[6], v, Kad[5]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[4] = fma(Dbd[6], v, Kac[4]);
          Kad[3] = fma(Dbc[7], v, Kad[3]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[4] = fma(Dbd[7], v, Kac[4]);
          Kad[4] = fma(Dbc[7], v, Kad[4]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[4] = fma(Dbd[8], v, Kac[4]);
          Kad[5] = fma(Dbc[7], v, Kad[5]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[5] = fma(Dbd[6], v, Kac[5]);
          Kad[3] = fma(Dbc[8], v, Kad[3]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[5] = fma(Dbd[7], v, Kac[5]);
          Kad[4] = fma(Dbc[8], v, Kad[4]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[5] = fma(Dbd[8], v, Kac[5]);
          Kad[5] = fma(Dbc[8], v, Kad[5]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        Jab[8] += j;
      }
      {
        const double ab = Pab[1 * n + 3] * (kCons[2][1] * kCons[2][3]);
        const double e0 = E[76];
        const double e1 = E[77];
        const double e2 = E[78];
        const double e3 = E[79];
        const double e4 = E[80];
        const double e5 = E[81];
        const double e6 = E[82];
        const double e7 = E[83];
        const double e8 = E[84];
        const double e9 = E[85];
        const double e10 = E[86];
        const double e11 = E[87];
        const double z000 = fma(e11, r211_0, fma(e10, r210_0, fma(e9, r201_0, fma(e8, r200_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r202_0, fma(e8, r201_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r311_0, fma(e10, r310_0, fma(e9, r301_0, fma(e8, r300_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r203_0, fma(e8, r202_0, fma(e7, r113_0, fma(e6, r112_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r122_0, fma(e6, r121_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r302_0, fma(e8, r301_0, fma(e7, r212_0, fma(e6, r211_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r411_0, fma(e10, r410_0, fma(e9, r401_0, fma(e8, r400_0, fma(e7, r311_0, fma(e6, r310_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[3] = fma(Dbd[9], v, Kac[3]);
          Kad[3] = fma(Dbc[9], v, Kad[3]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[9] = fma(ac0, v, Kbd[9]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[3] = fma(Dbd[10], v, Kac[3]);
          Kad[4] = fma(Dbc[9], v, Kad[4]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[10] = fma(ac0, v, Kbd[10]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[3] = fma(Dbd[11], v, Kac[3]);
          Kad[5] = fma(Dbc[9], v, Kad[5]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[11] = fma(ac0, v, Kbd[11]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[4] = fma(Dbd[9], v, Kac[4]);
          Kad[3] = fma(Dbc[10], v, Kad[3]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[9] = fma(ac1, v, Kbd[9]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[4] = fma(Dbd[10], v, Kac[4]);
          Kad[4] = fma(Dbc[10], v, Kad[4]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[10] = fma(ac1, v, Kbd[10]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[4] = fma(Dbd[11], v, Kac[4]);
          Kad[5] = fma(Dbc[10], v, Kad[5]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[11] = fma(ac1, v, Kbd[11]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[5] = fma(Dbd[9], v, Kac[5]);
          Kad[3] = fma(Dbc[11], v, Kad[3]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[9] = fma(ac2, v, Kbd[9]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[5] = fma(Dbd[10], v, Kac[5]);
          Kad[4] = fma(Dbc[11], v, Kad[4]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[10] = fma(ac2, v, Kbd[10]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[5] = fma(Dbd[11], v, Kac[5]);
          Kad[5] = fma(Dbc[11], v, Kad[5]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[11] = fma(ac2, v, Kbd[11]);
        }
        Jab[9] += j;
      }
      {
        const double ab = Pab[1 * n + 4] * (kCons[2][1] * kCons[2][4]);
        const double e0 = E[88];
        const double e1 = E[89];
        const double e2 = E[90];
        const double e3 = E[91];
        const double e4 = E[92];
        const double e5 = E[93];
        const double e6 = E[94];
        const double e7 = E[95];
        const double e8 = E[96];
        const double e9 = E[97];
        const double e10 = E[98];
        const double e11 = E[99];
        const double z000 = fma(e11, r121_0, fma(e10, r120_0, fma(e9, r111_0, fma(e8, r110_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r112_0, fma(e8, r111_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r131_0, fma(e10, r130_0, fma(e9, r121_0, fma(e8, r120_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r113_0, fma(e8, r112_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r122_0, fma(e8, r121_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r141_0, fma(e10, r140_0, fma(e9, r131_0, fma(e8, r130_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[3] = fma(Dbd[12], v, Kac[3]);
          Kad[3] = fma(Dbc[12], v, Kad[3]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[12] = fma(ac0, v, Kbd[12]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[3] = fma(Dbd[13], v, Kac[3]);
          Kad[4] = fma(Dbc[12], v, Kad[4]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[13] = fma(ac0, v, Kbd[13]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[3] = fma(Dbd[14], v, Kac[3]);
          Kad[5] = fma(Dbc[12], v, Kad[5]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[14] = fma(ac0, v, Kbd[14]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[4] = fma(Dbd[12], v, Kac[4]);
          Kad[3] = fma(Dbc[13], v, Kad[3]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[12] = fma(ac1, v, Kbd[12]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[4] = fma(Dbd[13], v, Kac[4]);
          Kad[4] = fma(Dbc[13], v, Kad[4]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[13] = fma(ac1, v, Kbd[13]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[4] = fma(Dbd[14], v, Kac[4]);
          Kad[5] = fma(Dbc[13], v, Kad[5]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[14] = fma(ac1, v, Kbd[14]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[5] = fma(Dbd[12], v, Kac[5]);
          Kad[3] = fma(Dbc[14], v, Kad[3]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[12] = fma(ac2, v, Kbd[12]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[5] = fma(Dbd[13], v, Kac[5]);
          Kad[4] = fma(Dbc[14], v, Kad[4]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[13] = fma(ac2, v, Kbd[13]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[5] = fma(Dbd[14], v, Kac[5]);
          Kad[5] = fma(Dbc[14], v, Kad[5]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[14] = fma(ac2, v, Kbd[14]);
        }
        Jab[10] += j;
      }
      {
        const double ab = Pab[1 * n + 5] * (kCons[2][1] * kCons[2][5]);
        const double e0 = E[100];
        const double e1 = E[101];
        const double e2 = E[102];
        const double e3 = E[103];
        const double e4 = E[104];
        const double e5 = E[105];
        const double e6 = E[106];
        const double e7 = E[107];
        const double e8 = E[108];
        const double e9 = E[109];
        const double e10 = E[110];
        const double e11 = E[111];
        const double z000 = fma(e11, r112_0, fma(e10, r111_0, fma(e9, r110_0, fma(e8, r102_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r113_0, fma(e10, r112_0, fma(e9, r111_0, fma(e8, r103_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r120_0, fma(e8, r112_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r210_0, fma(e8, r202_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r114_0, fma(e10, r113_0, fma(e9, r112_0, fma(e8, r104_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r121_0, fma(e8, r113_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r130_0, fma(e8, r122_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r211_0, fma(e8, r203_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r220_0, fma(e8, r212_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r310_0, fma(e8, r302_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[3] = fma(Dbd[15], v, Kac[3]);
          Kad[3] = fma(Dbc[15], v, Kad[3]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[15] = fma(ac0, v, Kbd[15]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[3] = fma(Dbd[16], v, Kac[3]);
          Kad[4] = fma(Dbc[15], v, Kad[4]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[16] = fma(ac0, v, Kbd[16]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[3] = fma(Dbd[17], v, Kac[3]);
          Kad[5] = fma(Dbc[15], v, Kad[5]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[17] = fma(ac0, v, Kbd[17]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[4] = fma(Dbd[15], v, Kac[4]);
          Kad[3] = fma(Dbc[16], v, Kad[3]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[15] = fma(ac1, v, Kbd[15]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[4] = fma(Dbd[16], v, Kac[4]);
          Kad[4] = fma(Dbc[16], v, Kad[4]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[16] = fma(ac1, v, Kbd[16]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[4] = fma(Dbd[17], v, Kac[4]);
          Kad[5] = fma(Dbc[16], v, Kad[5]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[17] = fma(ac1, v, Kbd[17]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[5] = fma(Dbd[15], v, Kac[5]);
          Kad[3] = fma(Dbc[17], v, Kad[3]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[15] = fma(ac2, v, Kbd[15]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[5] = fma(Dbd[16], v, Kac[5]);
          Kad[4] = fma(Dbc[17], v, Kad[4]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[16] = fma(ac2, v, Kbd[16]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[5] = fma(Dbd[17], v, Kac[5]);
          Kad[5] = fma(Dbc[17], v, Kad[5]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[17] = fma(ac2, v, Kbd[17]);
        }
        Jab[11] += j;
      }
    }
    {
      const double ac0 = P[oc + 2 * n + 0] * kCons[2][2];
      const double ac1 = P[oc + 2 * n + 1] * kCons[2][2];
      const double ac2 = P[oc + 2 * n + 2] * kCons[2][2];
      const double ad0 = P[od + 2 * n + 0] * kCons[2][2];
      const double ad1 = P[od + 2 * n + 1] * kCons[2][2];
      const double ad2 = P[od + 2 * n + 2] * kCons[2][2];
      {
        const double ab = Pab[2 * n + 0] * (kCons[2][2] * kCons[2][0]);
        const double e0 = E[112];
        const double e1 = E[113];
        const double e2 = E[114];
        const double e3 = E[115];
        const double e4 = E[116];
        const double e5 = E[117];
        const double e6 = E[118];
        const double e7 = E[119];
        const double e8 = E[120];
        const double z000 = fma(e8, r220_0, fma(e7, r210_0, fma(e6, r200_0, fma(e5, r120_0, fma(e4, r110_0, fma(e3, r100_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r221_0, fma(e7, r211_0, fma(e6, r201_0, fma(e5, r121_0, fma(e4, r111_0, fma(e3, r101_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r230_0, fma(e7, r220_0, fma(e6, r210_0, fma(e5, r130_0, fma(e4, r120_0, fma(e3, r110_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r320_0, fma(e7, r310_0, fma(e6, r300_0, fma(e5, r220_0, fma(e4, r210_0, fma(e3, r200_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r222_0, fma(e7, r212_0, fma(e6, r202_0, fma(e5, r122_0, fma(e4, r112_0, fma(e3, r102_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r231_0, fma(e7, r221_0, fma(e6, r211_0, fma(e5, r131_0, fma(e4, r121_0, fma(e3, r111_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r240_0, fma(e7, r230_0, fma(e6, r220_0, fma(e5, r140_0, fma(e4, r130_0, fma(e3, r120_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r321_0, fma(e7, r311_0, fma(e6, r301_0, fma(e5, r221_0, fma(e4, r211_0, fma(e3, r201_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r330_0, fma(e7, r320_0, fma(e6, r310_0, fma(e5, r230_0, fma(e4, r220_0, fma(e3, r210_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r420_0, fma(e7, r410_0, fma(e6, r400_0, fma(e5, r320_0, fma(e4, r310_0, fma(e3, r300_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[0], v, Kac[6]);
          Kad[6] = fma(Dbc[0], v, Kad[6]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[1], v, Kac[6]);
          Kad[7] = fma(Dbc[0], v, Kad[7]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[2], v, Kac[6]);
          Kad[8] = fma(Dbc[0], v, Kad[8]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[0], v, Kac[7]);
          Kad[6] = fma(Dbc[1], v, Kad[6]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[1], v, Kac[7]);
          Kad[7] = fma(Dbc[1], v, Kad[7]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[2], v, Kac[7]);
          Kad[8] = fma(Dbc[1], v, Kad[8]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[0], v, Kac[8]);
          Kad[6] = fma(Dbc[2], v, Kad[6]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[1], v, Kac[8]);
          Kad[7] = fma(Dbc[2], v, Kad[7]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[2], v, Kac[8]);
          Kad[8] = fma(Dbc[2], v, Kad[8]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        Jab[12] += j;
      }
      {
        const double ab = Pab[2 * n + 1] * (kCons[2][2] * kCons[2][1]);
        const double e0 = E[121];
        const double e1 = E[122];
        const double e2 = E[123];
        const double e3 = E[124];
        const double e4 = E[125];
        const double e5 = E[126];
        const double e6 = E[127];
        const double e7 = E[128];
        const double z000 = fma(e7, r130_0, fma(e6, r120_0, fma(e5, r110_0, fma(e4, r100_0, fma(e3, r030_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r131_0, fma(e6, r121_0, fma(e5, r111_0, fma(e4, r101_0, fma(e3, r031_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r140_0, fma(e6, r130_0, fma(e5, r120_0, fma(e4, r110_0, fma(e3, r040_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r230_0, fma(e6, r220_0, fma(e5, r210_0, fma(e4, r200_0, fma(e3, r130_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r132_0, fma(e6, r122_0, fma(e5, r112_0, fma(e4, r102_0, fma(e3, r032_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r141_0, fma(e6, r131_0, fma(e5, r121_0, fma(e4, r111_0, fma(e3, r041_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r150_0, fma(e6, r140_0, fma(e5, r130_0, fma(e4, r120_0, fma(e3, r050_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r231_0, fma(e6, r221_0, fma(e5, r211_0, fma(e4, r201_0, fma(e3, r131_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r240_0, fma(e6, r230_0, fma(e5, r220_0, fma(e4, r210_0, fma(e3, r140_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r330_0, fma(e6, r320_0, fma(e5, r310_0, fma(e4, r300_0, fma(e3, r230_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[3], v, Kac[6]);
          Kad[6] = fma(Dbc[3], v, Kad[6]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[4], v, Kac[6]);
          Kad[7] = fma(Dbc[3], v, Kad[7]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[5], v, Kac[6]);
          Kad[8] = fma(Dbc[3], v, Kad[8]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[3], v, Kac[7]);
          Kad[6] = fma(Dbc[4], v, Kad[6]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[4], v, Kac[7]);
          Kad[7] = fma(Dbc[4], v, Kad[7]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[5], v, Kac[7]);
          Kad[8] = fma(Dbc[4], v, Kad[8]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[3], v, Kac[8]);
          Kad[6] = fma(Dbc[5], v, Kad[6]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[4], v, Kac[8]);
          Kad[7] = fma(Dbc[5], v, Kad[7]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[5], v, Kac[8]);
          Kad[8] = fma(Dbc[5], v, Kad[8]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        Jab[13] += j;
      }
      {
        const double ab = Pab[2 * n + 2] * (kCons[2][2] * kCons[2][2]);
        const double e0 = E[129];
        const double e1 = E[130];
        const double e2 = E[131];
        const double e3 = E[132];
        const double e4 = E[133];
        const double z000 = fma(e4, r040_0, fma(e3, r030_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0))));
        const double z001 = fma(e4, r041_0, fma(e3, r031_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0))));
        const double z010 = fma(e4, r050_0, fma(e3, r040_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0))));
        const double z100 = fma(e4, r140_0, fma(e3, r130_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0))));
        const double z002 = fma(e4, r042_0, fma(e3, r032_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0))));
        const double z011 = fma(e4, r051_0, fma(e3, r041_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0))));
        const double z020 = fma(e4, r060_0, fma(e3, r050_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0))));
        const double z101 = fma(e4, r141_0, fma(e3, r131_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0))));
        const double z110 = fma(e4, r150_0, fma(e3, r140_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0))));
        const double z200 = fma(e4, r240_0, fma(e3, r230_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[6], v, Kac[6]);
          Kad[6] = fma(Dbc[6], v, Kad[6]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[7], v, Kac[6]);
          Kad[7] = fma(Dbc[6], v, Kad[7]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[8], v, Kac[6]);
          Kad[8] = fma(Dbc[6], v, Kad[8]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[6], v, Kac[7]);
          Kad[6] = fma(Dbc[7], v, Kad[6]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[7], v, Kac[7]);
          Kad[7] = fma(Dbc[7], v, Kad[7]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[8], v, Kac[7]);
          Kad[8] = fma(Dbc[7], v, Kad[8]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[6], v, Kac[8]);
          Kad[6] = fma(Dbc[8], v, Kad[6]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[7], v, Kac[8]);
          Kad[7] = fma(Dbc[8], v, Kad[7]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[8], v, Kac[8]);
          Kad[8] = fma(Dbc[8], v, Kad[8]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        Jab[14] += j;
      }
      {
        const double ab = Pab[2 * n + 3] * (kCons[2][2] * kCons[2][3]);
        const double e0 = E[134];
        const double e1 = E[135];
        const double e2 = E[136];
        const double e3 = E[137];
        const double e4 = E[138];
        const double e5 = E[139];
        const double e6 = E[140];
        const double e7 = E[141];
        const double e8 = E[142];
        const double e9 = E[143];
        const double e10 = E[144];
        const double e11 = E[145];
        const double z000 = fma(e11, r121_0, fma(e10, r120_0, fma(e9, r111_0, fma(e8, r110_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r112_0, fma(e8, r111_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r131_0, fma(e10, r130_0, fma(e9, r121_0, fma(e8, r120_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r113_0, fma(e8, r112_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r122_0, fma(e8, r121_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r141_0, fma(e10, r140_0, fma(e9, r131_0, fma(e8, r130_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[9], v, Kac[6]);
          Kad[6] = fma(Dbc[9], v, Kad[6]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[9] = fma(ac0, v, Kbd[9]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[10], v, Kac[6]);
          Kad[7] = fma(Dbc[9], v, Kad[7]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[10] = fma(ac0, v, Kbd[10]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[11], v, Kac[6]);
          Kad[8] = fma(Dbc[9], v, Kad[8]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[11] = fma(ac0, v, Kbd[11]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[9], v, Kac[7]);
          Kad[6] = fma(Dbc[10], v, Kad[6]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[9] = fma(ac1, v, Kbd[9]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[10], v, Kac[7]);
          Kad[7] = fma(Dbc[10], v, Kad[7]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[10] = fma(ac1, v, Kbd[10]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[11], v, Kac[7]);
          Kad[8] = fma(Dbc[10], v, Kad[8]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[11] = fma(ac1, v, Kbd[11]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[9], v, Kac[8]);
          Kad[6] = fma(Dbc[11], v, Kad[6]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[9] = fma(ac2, v, Kbd[9]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[10], v, Kac[8]);
          Kad[7] = fma(Dbc[11], v, Kad[7]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[10] = fma(ac2, v, Kbd[10]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[11], v, Kac[8]);
          Kad[8] = fma(Dbc[11], v, Kad[8]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[11] = fma(ac2, v, Kbd[11]);
        }
        Jab[15] += j;
      }
      {
        const double ab = Pab[2 * n + 4] * (kCons[2][2] * kCons[2][4]);
        const double e0 = E[146];
        const double e1 = E[147];
        const double e2 = E[148];
        const double e3 = E[149];
        const double e4 = E[150];
        const double e5 = E[151];
        const double e6 = E[152];
        const double e7 = E[153];
        const double z000 = fma(e7, r031_0, fma(e6, r030_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r032_0, fma(e6, r031_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r041_0, fma(e6, r040_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r033_0, fma(e6, r032_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r042_0, fma(e6, r041_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r051_0, fma(e6, r050_0, fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r132_0, fma(e6, r131_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r141_0, fma(e6, r140_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r231_0, fma(e6, r230_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[12], v, Kac[6]);
          Kad[6] = fma(Dbc[12], v, Kad[6]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[12] = fma(ac0, v, Kbd[12]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[13], v, Kac[6]);
          Kad[7] = fma(Dbc[12], v, Kad[7]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[13] = fma(ac0, v, Kbd[13]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[14], v, Kac[6]);
          Kad[8] = fma(Dbc[12], v, Kad[8]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[14] = fma(ac0, v, Kbd[14]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[12], v, Kac[7]);
          Kad[6] = fma(Dbc[13], v, Kad[6]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[12] = fma(ac1, v, Kbd[12]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[13], v, Kac[7]);
          Kad[7] = fma(Dbc[13], v, Kad[7]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[13] = fma(ac1, v, Kbd[13]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[14], v, Kac[7]);
          Kad[8] = fma(Dbc[13], v, Kad[8]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[14] = fma(ac1, v, Kbd[14]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[12], v, Kac[8]);
          Kad[6] = fma(Dbc[14], v, Kad[6]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[12] = fma(ac2, v, Kbd[12]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[13], v, Kac[8]);
          Kad[7] = fma(Dbc[14], v, Kad[7]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[13] = fma(ac2, v, Kbd[13]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[14], v, Kac[8]);
          Kad[8] = fma(Dbc[14], v, Kad[8]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[14] = fma(ac2, v, Kbd[14]);
        }
        Jab[16] += j;
      }
      {
        const double ab = Pab[2 * n + 5] * (kCons[2][2] * kCons[2][5]);
        const double e0 = E[154];
        const double e1 = E[155];
        const double e2 = E[156];
        const double e3 = E[157];
        const double e4 = E[158];
        const double e5 = E[159];
        const double e6 = E[160];
        const double e7 = E[161];
        const double e8 = E[162];
        const double z000 = fma(e8, r022_0, fma(e7, r021_0, fma(e6, r020_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r023_0, fma(e7, r022_0, fma(e6, r021_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r032_0, fma(e7, r031_0, fma(e6, r030_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r122_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r024_0, fma(e7, r023_0, fma(e6, r022_0, fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r033_0, fma(e7, r032_0, fma(e6, r031_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r042_0, fma(e7, r041_0, fma(e6, r040_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r123_0, fma(e7, r122_0, fma(e6, r121_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r132_0, fma(e7, r131_0, fma(e6, r130_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r222_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[15], v, Kac[6]);
          Kad[6] = fma(Dbc[15], v, Kad[6]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[15] = fma(ac0, v, Kbd[15]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[16], v, Kac[6]);
          Kad[7] = fma(Dbc[15], v, Kad[7]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[16] = fma(ac0, v, Kbd[16]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[17], v, Kac[6]);
          Kad[8] = fma(Dbc[15], v, Kad[8]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[17] = fma(ac0, v, Kbd[17]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[15], v, Kac[7]);
          Kad[6] = fma(Dbc[16], v, Kad[6]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[15] = fma(ac1, v, Kbd[15]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[16], v, Kac[7]);
          Kad[7] = fma(Dbc[16], v, Kad[7]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[16] = fma(ac1, v, Kbd[16]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[17], v, Kac[7]);
          Kad[8] = fma(Dbc[16], v, Kad[8]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[17] = fma(ac1, v, Kbd[17]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[15], v, Kac[8]);
          Kad[6] = fma(Dbc[17], v, Kad[6]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[15] = fma(ac2, v, Kbd[15]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[16], v, Kac[8]);
          Kad[7] = fma(Dbc[17], v, Kad[7]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[16] = fma(ac2, v, Kbd[16]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[17], v, Kac[8]);
          Kad[8] = fma(Dbc[17], v, Kad[8]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[17] = fma(ac2, v, Kbd[17]);
        }
        Jab[17] += j;
      }
    }
    {
      const double ac0 = P[oc + 3 * n + 0] * kCons[2][3];
      const double ac1 = P[oc + 3 * n + 1] * kCons[2][3];
      const double ac2 = P[oc + 3 * n + 2] * kCons[2][3];
      const double ad0 = P[od + 3 * n + 0] * kCons[2][3];
      const double ad1 = P[od + 3 * n + 1] * kCons[2][3];
      const double ad2 = P[od + 3 * n + 2] * kCons[2][3];
      {
        const double ab = Pab[3 * n + 0] * (kCons[2][3] * kCons[2][0]);
        const double e0 = E[163];
        const double e1 = E[164];
        const double e2 = E[165];
        const double e3 = E[166];
        const double e4 = E[167];
        const double e5 = E[168];
        const double e6 = E[169];
        const double e7 = E[170];
        const double z000 = fma(e7, r301_0, fma(e6, r300_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r101_0, fma(e2, r100_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r302_0, fma(e6, r301_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r102_0, fma(e2, r101_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r311_0, fma(e6, r310_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r401_0, fma(e6, r400_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r201_0, fma(e2, r200_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r303_0, fma(e6, r302_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r312_0, fma(e6, r311_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r321_0, fma(e6, r320_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r402_0, fma(e6, r401_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r202_0, fma(e2, r201_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r411_0, fma(e6, r410_0, fma(e5, r311_0, fma(e4, r310_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r501_0, fma(e6, r500_0, fma(e5, r401_0, fma(e4, r400_0, fma(e3, r301_0, fma(e2, r300_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[9] = fma(Dbd[0], v, Kac[9]);
          Kad[9] = fma(Dbc[0], v, Kad[9]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[9] = fma(Dbd[1], v, Kac[9]);
          Kad[10] = fma(Dbc[0], v, Kad[10]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[9] = fma(Dbd[2], v, Kac[9]);
          Kad[11] = fma(Dbc[0], v, Kad[11]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[10] = fma(Dbd[0], v, Kac[10]);
          Kad[9] = fma(Dbc[1], v, Kad[9]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[10] = fma(Dbd[1], v, Kac[10]);
          Kad[10] = fma(Dbc[1], v, Kad[10]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[10] = fma(Dbd[2], v, Kac[10]);
          Kad[11] = fma(Dbc[1], v, Kad[11]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[11] = fma(Dbd[0], v, Kac[11]);
          Kad[9] = fma(Dbc[2], v, Kad[9]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[11] = fma(Dbd[1], v, Kac[11]);
          Kad[10] = fma(Dbc[2], v, Kad[10]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[11] = fma(Dbd[2], v, Kac[11]);
          Kad[11] = fma(Dbc[2], v, Kad[11]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        Jab[18] += j;
      }
      {
        const double ab = Pab[3 * n + 1] * (kCons[2][3] * kCons[2][1]);
        const double e0 = E[171];
        const double e1 = E[172];
        const double e2 = E[173];
        const double e3 = E[174];
        const double e4 = E[175];
        const double e5 = E[176];
        const double e6 = E[177];
        const double e7 = E[178];
        const double e8 = E[179];
        const double e9 = E[180];
        const double e10 = E[181];
        const double e11 = E[182];
        const double z000 = fma(e11, r211_0, fma(e10, r210_0, fma(e9, r201_0, fma(e8, r200_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r202_0, fma(e8, r201_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r311_0, fma(e10, r310_0, fma(e9, r301_0, fma(e8, r300_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r203_0, fma(e8, r202_0, fma(e7, r113_0, fma(e6, r112_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r122_0, fma(e6, r121_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r302_0, fma(e8, r301_0, fma(e7, r212_0, fma(e6, r211_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r411_0, fma(e10, r410_0, fma(e9, r401_0, fma(e8, r400_0, fma(e7, r311_0, fma(e6, r310_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[9] = fma(Dbd[3], v, Kac[9]);
          Kad[9] = fma(Dbc[3], v, Kad[9]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[9] = fma(Dbd[4], v, Kac[9]);
          Kad[10] = fma(Dbc[3], v, Kad[10]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[9] = fma(Dbd[5], v, Kac[9]);
          Kad[11] = fma(Dbc[3], v, Kad[11]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[10] = fma(Dbd[3], v, Kac[10]);
          Kad[9] = fma(Dbc[4], v, Kad[9]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[10] = fma(Dbd[4], v, Kac[10]);
          Kad[10] = fma(Dbc[4], v, Kad[10]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[10] = fma(Dbd[5], v, Kac[10]);
          Kad[11] = fma(Dbc[4], v, Kad[11]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[11] = fma(Dbd[3], v, Kac[11]);
          Kad[9] = fma(Dbc[5], v, Kad[9]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[11] = fma(Dbd[4], v, Kac[11]);
          Kad[10] = fma(Dbc[5], v, Kad[10]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[11] = fma(Dbd[5], v, Kac[11]);
          Kad[11] = fma(Dbc[5], v, Kad[11]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        Jab[19] += j;
      }
      {
        const double ab = Pab[3 * n + 2] * (kCons[2][3] * kCons[2][2]);
        const double e0 = E[183];
        const double e1 = E[184];
        const double e2 = E[185];
        const double e3 = E[186];
        const double e4 = E[187];
        const double e5 = E[188];
        const double e6 = E[189];
        const double e7 = E[190];
        const double e8 = E[191];
        const double e9 = E[192];
        const double e10 = E[193];
        const double e11 = E[194];
        const double z000 = fma(e11, r121_0, fma(e10, r120_0, fma(e9, r111_0, fma(e8, r110_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r112_0, fma(e8, r111_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r131_0, fma(e10, r130_0, fma(e9, r121_0, fma(e8, r120_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r113_0, fma(e8, r112_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r122_0, fma(e8, r121_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r141_0, fma(e10, r140_0, fma(e9, r131_0, fma(e8, r130_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[9] = fma(Dbd[6], v, Kac[9]);
          Kad[9] = fma(Dbc[6], v, Kad[9]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[9] = fma(Dbd[7], v, Kac[9]);
          Kad[10] = fma(Dbc[6], v, Kad[10]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[9] = fma(Dbd[8], v, Kac[9]);
          Kad[11] = fma(Dbc[6], v, Kad[11]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[10] = fma(Dbd[6], v, Kac[10]);
          Kad[9] = fma(Dbc[7], v, Kad[9]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[10] = fma(Dbd[7], v, Kac[10]);
          Kad[10] = fma(Dbc[7], v, Kad[10]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[10] = fma(Dbd[8], v, Kac[10]);
          Kad[11] = fma(Dbc[7], v, Kad[11]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[11] = fma(Dbd[6], v, Kac[11]);
          Kad[9] = fma(Dbc[8], v, Kad[9]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[11] = fma(Dbd[7], v, Kac[11]);
          Kad[10] = fma(Dbc[8], v, Kad[10]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[11] = fma(Dbd[8], v, Kac[11]);
          Kad[11] = fma(Dbc[8], v, Kad[11]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        Jab[20] += j;
      }
      {
        const double ab = Pab[3 * n + 3] * (kCons[2][3] * kCons[2][3]);
        const double e0 = E[195];
        const double e1 = E[196];
        const double e2 = E[197];
        const double e3 = E[198];
        const double e4 = E[199];
        const double e5 = E[200];
        const double e6 = E[201];
        const double e7 = E[202];
        const double e8 = E[203];
        const double z000 = fma(e8, r202_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r100_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r203_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r101_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r212_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r302_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r200_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r204_0, fma(e7, r203_0, fma(e6, r202_0, fma(e5, r104_0, fma(e4, r103_0, fma(e3, r102_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r213_0, fma(e7, r212_0, fma(e6, r211_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r222_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r303_0, fma(e7, r302_0, fma(e6, r301_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r201_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r312_0, fma(e7, r311_0, fma(e6, r310_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r402_0, fma(e7, r401_0, fma(e6, r400_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r300_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[9] = fma(Dbd[9], v, Kac[9]);
          Kad[9] = fma(Dbc[9], v, Kad[9]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[9] = fma(ac0, v, Kbd[9]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[9] = fma(Dbd[10], v, Kac[9]);
          Kad[10] = fma(Dbc[9], v, Kad[10]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[10] = fma(ac0, v, Kbd[10]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[9] = fma(Dbd[11], v, Kac[9]);
          Kad[11] = fma(Dbc[9], v, Kad[11]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[11] = fma(ac0, v, Kbd[11]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[10] = fma(Dbd[9], v, Kac[10]);
          Kad[9] = fma(Dbc[10], v, Kad[9]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[9] = fma(ac1, v, Kbd[9]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[10] = fma(Dbd[10], v, Kac[10]);
          Kad[10] = fma(Dbc[10], v, Kad[10]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[10] = fma(ac1, v, Kbd[10]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[10] = fma(Dbd[11], v, Kac[10]);
          Kad[11] = fma(Dbc[10], v, Kad[11]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[11] = fma(ac1, v, Kbd[11]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[11] = fma(Dbd[9], v, Kac[11]);
          Kad[9] = fma(Dbc[11], v, Kad[9]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[9] = fma(ac2, v, Kbd[9]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[11] = fma(Dbd[10], v, Kac[11]);
          Kad[10] = fma(Dbc[11], v, Kad[10]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[10] = fma(ac2, v, Kbd[10]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[11] = fma(Dbd[11], v, Kac[11]);
          Kad[11] = fma(Dbc[11], v, Kad[11]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[11] = fma(ac2, v, Kbd[11]);
        }
        Jab[21] += j;
      }
      {
        const double ab = Pab[3 * n + 4] * (kCons[2][3] * kCons[2][4]);
        const double e0 = E[204];
        const double e1 = E[205];
        const double e2 = E[206];
        const double e3 = E[207];
        const double e4 = E[208];
        const double e5 = E[209];
        const double e6 = E[210];
        const double e7 = E[211];
        const double e8 = E[212];
        const double e9 = E[213];
        const double e10 = E[214];
        const double e11 = E[215];
        const double z000 = fma(e11, r112_0, fma(e10, r111_0, fma(e9, r110_0, fma(e8, r102_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r113_0, fma(e10, r112_0, fma(e9, r111_0, fma(e8, r103_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r120_0, fma(e8, r112_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r210_0, fma(e8, r202_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r114_0, fma(e10, r113_0, fma(e9, r112_0, fma(e8, r104_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r121_0, fma(e8, r113_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r130_0, fma(e8, r122_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r211_0, fma(e8, r203_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r220_0, fma(e8, r212_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r310_0, fma(e8, r302_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[9] = fma(Dbd[12], v, Kac[9]);
          Kad[9] = fma(Dbc[12], v, Kad[9]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[12] = fma(ac0, v, Kbd[12]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[9] = fma(Dbd[13], v, Kac[9]);
          Kad[10] = fma(Dbc[12], v, Kad[10]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[13] = fma(ac0, v, Kbd[13]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[9] = fma(Dbd[14], v, Kac[9]);
          Kad[11] = fma(Dbc[12], v, Kad[11]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[14] = fma(ac0, v, Kbd[14]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[10] = fma(Dbd[12], v, Kac[10]);
          Kad[9] = fma(Dbc[13], v, Kad[9]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[12] = fma(ac1, v, Kbd[12]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[10] = fma(Dbd[13], v, Kac[10]);
          Kad[10] = fma(Dbc[13], v, Kad[10]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[13] = fma(ac1, v, Kbd[13]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[10] = fma(Dbd[14], v, Kac[10]);
          Kad[11] = fma(Dbc[13], v, Kad[11]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[14] = fma(ac1, v, Kbd[14]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[11] = fma(Dbd[12], v, Kac[11]);
          Kad[9] = fma(Dbc[14], v, Kad[9]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[12] = fma(ac2, v, Kbd[12]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[11] = fma(Dbd[13], v, Kac[11]);
          Kad[10] = fma(Dbc[14], v, Kad[10]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[13] = fma(ac2, v, Kbd[13]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[11] = fma(Dbd[14], v, Kac[11]);
          Kad[11] = fma(Dbc[14], v, Kad[11]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[14] = fma(ac2, v, Kbd[14]);
        }
        Jab[22] += j;
      }
      {
        const double ab = Pab[3 * n + 5] * (kCons[2][3] * kCons[2][5]);
        const double e0 = E[216];
        const double e1 = E[217];
        const double e2 = E[218];
        const double e3 = E[219];
        const double e4 = E[220];
        const double e5 = E[221];
        const double e6 = E[222];
        const double e7 = E[223];
        const double z000 = fma(e7, r103_0, fma(e6, r102_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r003_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r104_0, fma(e6, r103_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r004_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r113_0, fma(e6, r112_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r203_0, fma(e6, r202_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r105_0, fma(e6, r104_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r005_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r114_0, fma(e6, r113_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r123_0, fma(e6, r122_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r204_0, fma(e6, r203_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r104_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r213_0, fma(e6, r212_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r303_0, fma(e6, r302_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r203_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[9] = fma(Dbd[15], v, Kac[9]);
          Kad[9] = fma(Dbc[15], v, Kad[9]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[15] = fma(ac0, v, Kbd[15]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[9] = fma(Dbd[16], v, Kac[9]);
          Kad[10] = fma(Dbc[15], v, Kad[10]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[16] = fma(ac0, v, Kbd[16]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[9] = fma(Dbd[17], v, Kac[9]);
          Kad[11] = fma(Dbc[15], v, Kad[11]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[17] = fma(ac0, v, Kbd[17]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[10] = fma(Dbd[15], v, Kac[10]);
          Kad[9] = fma(Dbc[16], v, Kad[9]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[15] = fma(ac1, v, Kbd[15]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[10] = fma(Dbd[16], v, Kac[10]);
          Kad[10] = fma(Dbc[16], v, Kad[10]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[16] = fma(ac1, v, Kbd[16]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[10] = fma(Dbd[17], v, Kac[10]);
          Kad[11] = fma(Dbc[16], v, Kad[11]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[17] = fma(ac1, v, Kbd[17]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[11] = fma(Dbd[15], v, Kac[11]);
          Kad[9] = fma(Dbc[17], v, Kad[9]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[15] = fma(ac2, v, Kbd[15]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[11] = fma(Dbd[16], v, Kac[11]);
          Kad[10] = fma(Dbc[17], v, Kad[10]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[16] = fma(ac2, v, Kbd[16]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[11] = fma(Dbd[17], v, Kac[11]);
          Kad[11] = fma(Dbc[17], v, Kad[11]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[17] = fma(ac2, v, Kbd[17]);
        }
        Jab[23] += j;
      }
    }
    {
      const double ac0 = P[oc + 4 * n + 0] * kCons[2][4];
      const double ac1 = P[oc + 4 * n + 1] * kCons[2][4];
      const double ac2 = P[oc + 4 * n + 2] * kCons[2][4];
      const double ad0 = P[od + 4 * n + 0] * kCons[2][4];
      const double ad1 = P[od + 4 * n + 1] * kCons[2][4];
      const double ad2 = P[od + 4 * n + 2] * kCons[2][4];
      {
        const double ab = Pab[4 * n + 0] * (kCons[2][4] * kCons[2][0]);
        const double e0 = E[224];
        const double e1 = E[225];
        const double e2 = E[226];
        const double e3 = E[227];
        const double e4 = E[228];
        const double e5 = E[229];
        const double e6 = E[230];
        const double e7 = E[231];
        const double e8 = E[232];
        const double e9 = E[233];
        const double e10 = E[234];
        const double e11 = E[235];
        const double z000 = fma(e11, r211_0, fma(e10, r210_0, fma(e9, r201_0, fma(e8, r200_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r202_0, fma(e8, r201_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r311_0, fma(e10, r310_0, fma(e9, r301_0, fma(e8, r300_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r203_0, fma(e8, r202_0, fma(e7, r113_0, fma(e6, r112_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r122_0, fma(e6, r121_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r302_0, fma(e8, r301_0, fma(e7, r212_0, fma(e6, r211_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r411_0, fma(e10, r410_0, fma(e9, r401_0, fma(e8, r400_0, fma(e7, r311_0, fma(e6, r310_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[0], v, Kac[12]);
          Kad[12] = fma(Dbc[0], v, Kad[12]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[1], v, Kac[12]);
          Kad[13] = fma(Dbc[0], v, Kad[13]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[2], v, Kac[12]);
          Kad[14] = fma(Dbc[0], v, Kad[14]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[0], v, Kac[13]);
          Kad[12] = fma(Dbc[1], v, Kad[12]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[1], v, Kac[13]);
          Kad[13] = fma(Dbc[1], v, Kad[13]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[2], v, Kac[13]);
          Kad[14] = fma(Dbc[1], v, Kad[14]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[0], v, Kac[14]);
          Kad[12] = fma(Dbc[2], v, Kad[12]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[1], v, Kac[14]);
          Kad[13] = fma(Dbc[2], v, Kad[13]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[2], v, Kac[14]);
          Kad[14] = fma(Dbc[2], v, Kad[14]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        Jab[24] += j;
      }
      {
        const double ab = Pab[4 * n + 1] * (kCons[2][4] * kCons[2][1]);
        const double e0 = E[236];
        const double e1 = E[237];
        const double e2 = E[238];
        const double e3 = E[239];
        const double e4 = E[240];
        const double e5 = E[241];
        const double e6 = E[242];
        const double e7 = E[243];
        const double e8 = E[244];
        const double e9 = E[245];
        const double e10 = E[246];
        const double e11 = E[247];
        const double z000 = fma(e11, r121_0, fma(e10, r120_0, fma(e9, r111_0, fma(e8, r110_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r112_0, fma(e8, r111_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r131_0, fma(e10, r130_0, fma(e9, r121_0, fma(e8, r120_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r221_0, fma(e10, r220_0, fma(e9, r211_0, fma(e8, r210_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r113_0, fma(e8, r112_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r122_0, fma(e8, r121_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r141_0, fma(e10, r140_0, fma(e9, r131_0, fma(e8, r130_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r212_0, fma(e8, r211_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r231_0, fma(e10, r230_0, fma(e9, r221_0, fma(e8, r220_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r321_0, fma(e10, r320_0, fma(e9, r311_0, fma(e8, r310_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[3], v, Kac[12]);
          Kad[12] = fma(Dbc[3], v, Kad[12]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[4], v, Kac[12]);
          Kad[13] = fma(Dbc[3], v, Kad[13]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[5], v, Kac[12]);
          Kad[14] = fma(Dbc[3], v, Kad[14]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[3], v, Kac[13]);
          Kad[12] = fma(Dbc[4], v, Kad[12]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[4], v, Kac[13]);
          Kad[13] = fma(Dbc[4], v, Kad[13]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[5], v, Kac[13]);
          Kad[14] = fma(Dbc[4], v, Kad[14]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[3], v, Kac[14]);
          Kad[12] = fma(Dbc[5], v, Kad[12]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[4], v, Kac[14]);
          Kad[13] = fma(Dbc[5], v, Kad[13]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[5], v, Kac[14]);
          Kad[14] = fma(Dbc[5], v, Kad[14]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        Jab[25] += j;
      }
      {
        const double ab = Pab[4 * n + 2] * (kCons[2][4] * kCons[2][2]);
        const double e0 = E[248];
        const double e1 = E[249];
        const double e2 = E[250];
        const double e3 = E[251];
        const double e4 = E[252];
        const double e5 = E[253];
        const double e6 = E[254];
        const double e7 = E[255];
        const double z000 = fma(e7, r031_0, fma(e6, r030_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r032_0, fma(e6, r031_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r041_0, fma(e6, r040_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r033_0, fma(e6, r032_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r042_0, fma(e6, r041_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r051_0, fma(e6, r050_0, fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r132_0, fma(e6, r131_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r141_0, fma(e6, r140_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r231_0, fma(e6, r230_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[6], v, Kac[12]);
          Kad[12] = fma(Dbc[6], v, Kad[12]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[7], v, Kac[12]);
          Kad[13] = fma(Dbc[6], v, Kad[13]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[8], v, Kac[12]);
          Kad[14] = fma(Dbc[6], v, Kad[14]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[6], v, Kac[13]);
          Kad[12] = fma(Dbc[7], v, Kad[12]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[7], v, Kac[13]);
          Kad[13] = fma(Dbc[7], v, Kad[13]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[8], v, Kac[13]);
          Kad[14] = fma(Dbc[7], v, Kad[14]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[6], v, Kac[14]);
          Kad[12] = fma(Dbc[8], v, Kad[12]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[7], v, Kac[14]);
          Kad[13] = fma(Dbc[8], v, Kad[13]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[8], v, Kac[14]);
          Kad[14] = fma(Dbc[8], v, Kad[14]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        Jab[26] += j;
      }
      {
        const double ab = Pab[4 * n + 3] * (kCons[2][4] * kCons[2][3]);
        const double e0 = E[256];
        const double e1 = E[257];
        const double e2 = E[258];
        const double e3 = E[259];
        const double e4 = E[260];
        const double e5 = E[261];
        const double e6 = E[262];
        const double e7 = E[263];
        const double e8 = E[264];
        const double e9 = E[265];
        const double e10 = E[266];
        const double e11 = E[267];
        const double z000 = fma(e11, r112_0, fma(e10, r111_0, fma(e9, r110_0, fma(e8, r102_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r113_0, fma(e10, r112_0, fma(e9, r111_0, fma(e8, r103_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r120_0, fma(e8, r112_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r210_0, fma(e8, r202_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r114_0, fma(e10, r113_0, fma(e9, r112_0, fma(e8, r104_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r121_0, fma(e8, r113_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r130_0, fma(e8, r122_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r211_0, fma(e8, r203_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r220_0, fma(e8, r212_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r310_0, fma(e8, r302_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[9], v, Kac[12]);
          Kad[12] = fma(Dbc[9], v, Kad[12]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[9] = fma(ac0, v, Kbd[9]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[10], v, Kac[12]);
          Kad[13] = fma(Dbc[9], v, Kad[13]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[10] = fma(ac0, v, Kbd[10]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[11], v, Kac[12]);
          Kad[14] = fma(Dbc[9], v, Kad[14]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[11] = fma(ac0, v, Kbd[11]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[9], v, Kac[13]);
          Kad[12] = fma(Dbc[10], v, Kad[12]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[9] = fma(ac1, v, Kbd[9]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[10], v, Kac[13]);
          Kad[13] = fma(Dbc[10], v, Kad[13]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[10] = fma(ac1, v, Kbd[10]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[11], v, Kac[13]);
          Kad[14] = fma(Dbc[10], v, Kad[14]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[11] = fma(ac1, v, Kbd[11]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[9], v, Kac[14]);
          Kad[12] = fma(Dbc[11], v, Kad[12]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[9] = fma(ac2, v, Kbd[9]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[10], v, Kac[14]);
          Kad[13] = fma(Dbc[11], v, Kad[13]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[10] = fma(ac2, v, Kbd[10]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[11], v, Kac[14]);
          Kad[14] = fma(Dbc[11], v, Kad[14]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[11] = fma(ac2, v, Kbd[11]);
        }
        Jab[27] += j;
      }
      {
        const double ab = Pab[4 * n + 4] * (kCons[2][4] * kCons[2][4]);
        const double e0 = E[268];
        const double e1 = E[269];
        const double e2 = E[270];
        const double e3 = E[271];
        const double e4 = E[272];
        const double e5 = E[273];
        const double e6 = E[274];
        const double e7 = E[275];
        const double e8 = E[276];
        const double z000 = fma(e8, r022_0, fma(e7, r021_0, fma(e6, r020_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r023_0, fma(e7, r022_0, fma(e6, r021_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r032_0, fma(e7, r031_0, fma(e6, r030_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r122_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r024_0, fma(e7, r023_0, fma(e6, r022_0, fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r033_0, fma(e7, r032_0, fma(e6, r031_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r042_0, fma(e7, r041_0, fma(e6, r040_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r123_0, fma(e7, r122_0, fma(e6, r121_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r132_0, fma(e7, r131_0, fma(e6, r130_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r222_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[12], v, Kac[12]);
          Kad[12] = fma(Dbc[12], v, Kad[12]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[12] = fma(ac0, v, Kbd[12]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[13], v, Kac[12]);
          Kad[13] = fma(Dbc[12], v, Kad[13]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[13] = fma(ac0, v, Kbd[13]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[14], v, Kac[12]);
          Kad[14] = fma(Dbc[12], v, Kad[14]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[14] = fma(ac0, v, Kbd[14]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[12], v, Kac[13]);
          Kad[12] = fma(Dbc[13], v, Kad[12]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[12] = fma(ac1, v, Kbd[12]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[13], v, Kac[13]);
          Kad[13] = fma(Dbc[13], v, Kad[13]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[13] = fma(ac1, v, Kbd[13]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[14], v, Kac[13]);
          Kad[14] = fma(Dbc[13], v, Kad[14]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[14] = fma(ac1, v, Kbd[14]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[12], v, Kac[14]);
          Kad[12] = fma(Dbc[14], v, Kad[12]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[12] = fma(ac2, v, Kbd[12]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[13], v, Kac[14]);
          Kad[13] = fma(Dbc[14], v, Kad[13]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[13] = fma(ac2, v, Kbd[13]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[14], v, Kac[14]);
          Kad[14] = fma(Dbc[14], v, Kad[14]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[14] = fma(ac2, v, Kbd[14]);
        }
        Jab[28] += j;
      }
      {
        const double ab = Pab[4 * n + 5] * (kCons[2][4] * kCons[2][5]);
        const double e0 = E[277];
        const double e1 = E[278];
        const double e2 = E[279];
        const double e3 = E[280];
        const double e4 = E[281];
        const double e5 = E[282];
        const double e6 = E[283];
        const double e7 = E[284];
        const double z000 = fma(e7, r013_0, fma(e6, r012_0, fma(e5, r011_0, fma(e4, r010_0, fma(e3, r003_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r014_0, fma(e6, r013_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r004_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r023_0, fma(e6, r022_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r113_0, fma(e6, r112_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r015_0, fma(e6, r014_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r005_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r024_0, fma(e6, r023_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r033_0, fma(e6, r032_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r114_0, fma(e6, r113_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r104_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r123_0, fma(e6, r122_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r213_0, fma(e6, r212_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r203_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[15], v, Kac[12]);
          Kad[12] = fma(Dbc[15], v, Kad[12]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[15] = fma(ac0, v, Kbd[15]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[16], v, Kac[12]);
          Kad[13] = fma(Dbc[15], v, Kad[13]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[16] = fma(ac0, v, Kbd[16]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[17], v, Kac[12]);
          Kad[14] = fma(Dbc[15], v, Kad[14]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[17] = fma(ac0, v, Kbd[17]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[15], v, Kac[13]);
          Kad[12] = fma(Dbc[16], v, Kad[12]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[15] = fma(ac1, v, Kbd[15]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[16], v, Kac[13]);
          Kad[13] = fma(Dbc[16], v, Kad[13]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[16] = fma(ac1, v, Kbd[16]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[17], v, Kac[13]);
          Kad[14] = fma(Dbc[16], v, Kad[14]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[17] = fma(ac1, v, Kbd[17]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[15], v, Kac[14]);
          Kad[12] = fma(Dbc[17], v, Kad[12]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[15] = fma(ac2, v, Kbd[15]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[16], v, Kac[14]);
          Kad[13] = fma(Dbc[17], v, Kad[13]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[16] = fma(ac2, v, Kbd[16]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[17], v, Kac[14]);
          Kad[14] = fma(Dbc[17], v, Kad[14]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[17] = fma(ac2, v, Kbd[17]);
        }
        Jab[29] += j;
      }
    }
    {
      const double ac0 = P[oc + 5 * n + 0] * kCons[2][5];
      const double ac1 = P[oc + 5 * n + 1] * kCons[2][5];
      const double ac2 = P[oc + 5 * n + 2] * kCons[2][5];
      const double ad0 = P[od + 5 * n + 0] * kCons[2][5];
      const double ad1 = P[od + 5 * n + 1] * kCons[2][5];
      const double ad2 = P[od + 5 * n + 2] * kCons[2][5];
      {
        const double ab = Pab[5 * n + 0] * (kCons[2][5] * kCons[2][0]);
        const double e0 = E[285];
        const double e1 = E[286];
        const double e2 = E[287];
        const double e3 = E[288];
        const double e4 = E[289];
        const double e5 = E[290];
        const double e6 = E[291];
        const double e7 = E[292];
        const double e8 = E[293];
        const double z000 = fma(e8, r202_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r100_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r203_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r101_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r212_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r302_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r200_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r204_0, fma(e7, r203_0, fma(e6, r202_0, fma(e5, r104_0, fma(e4, r103_0, fma(e3, r102_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r213_0, fma(e7, r212_0, fma(e6, r211_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r222_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r303_0, fma(e7, r302_0, fma(e6, r301_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r201_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r312_0, fma(e7, r311_0, fma(e6, r310_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r402_0, fma(e7, r401_0, fma(e6, r400_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r300_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[15] = fma(Dbd[0], v, Kac[15]);
          Kad[15] = fma(Dbc[0], v, Kad[15]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[15] = fma(Dbd[1], v, Kac[15]);
          Kad[16] = fma(Dbc[0], v, Kad[16]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[15] = fma(Dbd[2], v, Kac[15]);
          Kad[17] = fma(Dbc[0], v, Kad[17]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[16] = fma(Dbd[0], v, Kac[16]);
          Kad[15] = fma(Dbc[1], v, Kad[15]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[16] = fma(Dbd[1], v, Kac[16]);
          Kad[16] = fma(Dbc[1], v, Kad[16]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[16] = fma(Dbd[2], v, Kac[16]);
          Kad[17] = fma(Dbc[1], v, Kad[17]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[17] = fma(Dbd[0], v, Kac[17]);
          Kad[15] = fma(Dbc[2], v, Kad[15]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[17] = fma(Dbd[1], v, Kac[17]);
          Kad[16] = fma(Dbc[2], v, Kad[16]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[17] = fma(Dbd[2], v, Kac[17]);
          Kad[17] = fma(Dbc[2], v, Kad[17]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        Jab[30] += j;
      }
      {
        const double ab = Pab[5 * n + 1] * (kCons[2][5] * kCons[2][1]);
        const double e0 = E[294];
        const double e1 = E[295];
        const double e2 = E[296];
        const double e3 = E[297];
        const double e4 = E[298];
        const double e5 = E[299];
        const double e6 = E[300];
        const double e7 = E[301];
        const double e8 = E[302];
        const double e9 = E[303];
        const double e10 = E[304];
        const double e11 = E[305];
        const double z000 = fma(e11, r112_0, fma(e10, r111_0, fma(e9, r110_0, fma(e8, r102_0, fma(e7, r101_0, fma(e6, r100_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))))))));
        const double z001 = fma(e11, r113_0, fma(e10, r112_0, fma(e9, r111_0, fma(e8, r103_0, fma(e7, r102_0, fma(e6, r101_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))))))));
        const double z010 = fma(e11, r122_0, fma(e10, r121_0, fma(e9, r120_0, fma(e8, r112_0, fma(e7, r111_0, fma(e6, r110_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))))))));
        const double z100 = fma(e11, r212_0, fma(e10, r211_0, fma(e9, r210_0, fma(e8, r202_0, fma(e7, r201_0, fma(e6, r200_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))))))));
        const double z002 = fma(e11, r114_0, fma(e10, r113_0, fma(e9, r112_0, fma(e8, r104_0, fma(e7, r103_0, fma(e6, r102_0, fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))))))));
        const double z011 = fma(e11, r123_0, fma(e10, r122_0, fma(e9, r121_0, fma(e8, r113_0, fma(e7, r112_0, fma(e6, r111_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))))))));
        const double z020 = fma(e11, r132_0, fma(e10, r131_0, fma(e9, r130_0, fma(e8, r122_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))))))));
        const double z101 = fma(e11, r213_0, fma(e10, r212_0, fma(e9, r211_0, fma(e8, r203_0, fma(e7, r202_0, fma(e6, r201_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))))))));
        const double z110 = fma(e11, r222_0, fma(e10, r221_0, fma(e9, r220_0, fma(e8, r212_0, fma(e7, r211_0, fma(e6, r210_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))))))));
        const double z200 = fma(e11, r312_0, fma(e10, r311_0, fma(e9, r310_0, fma(e8, r302_0, fma(e7, r301_0, fma(e6, r300_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[15] = fma(Dbd[3], v, Kac[15]);
          Kad[15] = fma(Dbc[3], v, Kad[15]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[15] = fma(Dbd[4], v, Kac[15]);
          Kad[16] = fma(Dbc[3], v, Kad[16]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[15] = fma(Dbd[5], v, Kac[15]);
          Kad[17] = fma(Dbc[3], v, Kad[17]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[16] = fma(Dbd[3], v, Kac[16]);
          Kad[15] = fma(Dbc[4], v, Kad[15]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[16] = fma(Dbd[4], v, Kac[16]);
          Kad[16] = fma(Dbc[4], v, Kad[16]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[16] = fma(Dbd[5], v, Kac[16]);
          Kad[17] = fma(Dbc[4], v, Kad[17]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[17] = fma(Dbd[3], v, Kac[17]);
          Kad[15] = fma(Dbc[5], v, Kad[15]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[17] = fma(Dbd[4], v, Kac[17]);
          Kad[16] = fma(Dbc[5], v, Kad[16]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[17] = fma(Dbd[5], v, Kac[17]);
          Kad[17] = fma(Dbc[5], v, Kad[17]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        Jab[31] += j;
      }
      {
        const double ab = Pab[5 * n + 2] * (kCons[2][5] * kCons[2][2]);
        const double e0 = E[306];
        const double e1 = E[307];
        const double e2 = E[308];
        const double e3 = E[309];
        const double e4 = E[310];
        const double e5 = E[311];
        const double e6 = E[312];
        const double e7 = E[313];
        const double e8 = E[314];
        const double z000 = fma(e8, r022_0, fma(e7, r021_0, fma(e6, r020_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0))))))));
        const double z001 = fma(e8, r023_0, fma(e7, r022_0, fma(e6, r021_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0))))))));
        const double z010 = fma(e8, r032_0, fma(e7, r031_0, fma(e6, r030_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0))))))));
        const double z100 = fma(e8, r122_0, fma(e7, r121_0, fma(e6, r120_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0))))))));
        const double z002 = fma(e8, r024_0, fma(e7, r023_0, fma(e6, r022_0, fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0))))))));
        const double z011 = fma(e8, r033_0, fma(e7, r032_0, fma(e6, r031_0, fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0))))))));
        const double z020 = fma(e8, r042_0, fma(e7, r041_0, fma(e6, r040_0, fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0))))))));
        const double z101 = fma(e8, r123_0, fma(e7, r122_0, fma(e6, r121_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0))))))));
        const double z110 = fma(e8, r132_0, fma(e7, r131_0, fma(e6, r130_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0))))))));
        const double z200 = fma(e8, r222_0, fma(e7, r221_0, fma(e6, r220_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0))))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[15] = fma(Dbd[6], v, Kac[15]);
          Kad[15] = fma(Dbc[6], v, Kad[15]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[15] = fma(Dbd[7], v, Kac[15]);
          Kad[16] = fma(Dbc[6], v, Kad[16]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[15] = fma(Dbd[8], v, Kac[15]);
          Kad[17] = fma(Dbc[6], v, Kad[17]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[16] = fma(Dbd[6], v, Kac[16]);
          Kad[15] = fma(Dbc[7], v, Kad[15]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[16] = fma(Dbd[7], v, Kac[16]);
          Kad[16] = fma(Dbc[7], v, Kad[16]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[16] = fma(Dbd[8], v, Kac[16]);
          Kad[17] = fma(Dbc[7], v, Kad[17]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[17] = fma(Dbd[6], v, Kac[17]);
          Kad[15] = fma(Dbc[8], v, Kad[15]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[17] = fma(Dbd[7], v, Kac[17]);
          Kad[16] = fma(Dbc[8], v, Kad[16]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[17] = fma(Dbd[8], v, Kac[17]);
          Kad[17] = fma(Dbc[8], v, Kad[17]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        Jab[32] += j;
      }
      {
        const double ab = Pab[5 * n + 3] * (kCons[2][5] * kCons[2][3]);
        const double e0 = E[315];
        const double e1 = E[316];
        const double e2 = E[317];
        const double e3 = E[318];
        const double e4 = E[319];
        const double e5 = E[320];
        const double e6 = E[321];
        const double e7 = E[322];
        const double z000 = fma(e7, r103_0, fma(e6, r102_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r003_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r104_0, fma(e6, r103_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r004_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r113_0, fma(e6, r112_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r203_0, fma(e6, r202_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r105_0, fma(e6, r104_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r005_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r114_0, fma(e6, r113_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r123_0, fma(e6, r122_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r204_0, fma(e6, r203_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r104_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r213_0, fma(e6, r212_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r303_0, fma(e6, r302_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r203_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[15] = fma(Dbd[9], v, Kac[15]);
          Kad[15] = fma(Dbc[9], v, Kad[15]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[9] = fma(ac0, v, Kbd[9]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[15] = fma(Dbd[10], v, Kac[15]);
          Kad[16] = fma(Dbc[9], v, Kad[16]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[10] = fma(ac0, v, Kbd[10]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[15] = fma(Dbd[11], v, Kac[15]);
          Kad[17] = fma(Dbc[9], v, Kad[17]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[11] = fma(ac0, v, Kbd[11]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[16] = fma(Dbd[9], v, Kac[16]);
          Kad[15] = fma(Dbc[10], v, Kad[15]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[9] = fma(ac1, v, Kbd[9]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[16] = fma(Dbd[10], v, Kac[16]);
          Kad[16] = fma(Dbc[10], v, Kad[16]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[10] = fma(ac1, v, Kbd[10]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[16] = fma(Dbd[11], v, Kac[16]);
          Kad[17] = fma(Dbc[10], v, Kad[17]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[11] = fma(ac1, v, Kbd[11]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[17] = fma(Dbd[9], v, Kac[17]);
          Kad[15] = fma(Dbc[11], v, Kad[15]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[9] = fma(ac2, v, Kbd[9]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[17] = fma(Dbd[10], v, Kac[17]);
          Kad[16] = fma(Dbc[11], v, Kad[16]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[10] = fma(ac2, v, Kbd[10]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[17] = fma(Dbd[11], v, Kac[17]);
          Kad[17] = fma(Dbc[11], v, Kad[17]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[11] = fma(ac2, v, Kbd[11]);
        }
        Jab[33] += j;
      }
      {
        const double ab = Pab[5 * n + 4] * (kCons[2][5] * kCons[2][4]);
        const double e0 = E[323];
        const double e1 = E[324];
        const double e2 = E[325];
        const double e3 = E[326];
        const double e4 = E[327];
        const double e5 = E[328];
        const double e6 = E[329];
        const double e7 = E[330];
        const double z000 = fma(e7, r013_0, fma(e6, r012_0, fma(e5, r011_0, fma(e4, r010_0, fma(e3, r003_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r014_0, fma(e6, r013_0, fma(e5, r012_0, fma(e4, r011_0, fma(e3, r004_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r023_0, fma(e6, r022_0, fma(e5, r021_0, fma(e4, r020_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r113_0, fma(e6, r112_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r015_0, fma(e6, r014_0, fma(e5, r013_0, fma(e4, r012_0, fma(e3, r005_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r024_0, fma(e6, r023_0, fma(e5, r022_0, fma(e4, r021_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r033_0, fma(e6, r032_0, fma(e5, r031_0, fma(e4, r030_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r114_0, fma(e6, r113_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r104_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r123_0, fma(e6, r122_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r213_0, fma(e6, r212_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r203_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[15] = fma(Dbd[12], v, Kac[15]);
          Kad[15] = fma(Dbc[12], v, Kad[15]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[12] = fma(ac0, v, Kbd[12]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[15] = fma(Dbd[13], v, Kac[15]);
          Kad[16] = fma(Dbc[12], v, Kad[16]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[13] = fma(ac0, v, Kbd[13]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[15] = fma(Dbd[14], v, Kac[15]);
          Kad[17] = fma(Dbc[12], v, Kad[17]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[14] = fma(ac0, v, Kbd[14]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[16] = fma(Dbd[12], v, Kac[16]);
          Kad[15] = fma(Dbc[13], v, Kad[15]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[12] = fma(ac1, v, Kbd[12]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[16] = fma(Dbd[13], v, Kac[16]);
          Kad[16] = fma(Dbc[13], v, Kad[16]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[13] = fma(ac1, v, Kbd[13]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[16] = fma(Dbd[14], v, Kac[16]);
          Kad[17] = fma(Dbc[13], v, Kad[17]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[14] = fma(ac1, v, Kbd[14]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[17] = fma(Dbd[12], v, Kac[17]);
          Kad[15] = fma(Dbc[14], v, Kad[15]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[12] = fma(ac2, v, Kbd[12]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[17] = fma(Dbd[13], v, Kac[17]);
          Kad[16] = fma(Dbc[14], v, Kad[16]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[13] = fma(ac2, v, Kbd[13]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[17] = fma(Dbd[14], v, Kac[17]);
          Kad[17] = fma(Dbc[14], v, Kad[17]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[14] = fma(ac2, v, Kbd[14]);
        }
        Jab[34] += j;
      }
      {
        const double ab = Pab[5 * n + 5] * (kCons[2][5] * kCons[2][5]);
        const double e0 = E[331];
        const double e1 = E[332];
        const double e2 = E[333];
        const double e3 = E[334];
        const double e4 = E[335];
        const double z000 = fma(e4, r004_0, fma(e3, r003_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0))));
        const double z001 = fma(e4, r005_0, fma(e3, r004_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0))));
        const double z010 = fma(e4, r014_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0))));
        const double z100 = fma(e4, r104_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0))));
        const double z002 = fma(e4, r006_0, fma(e3, r005_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0))));
        const double z011 = fma(e4, r015_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0))));
        const double z020 = fma(e4, r024_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0))));
        const double z101 = fma(e4, r105_0, fma(e3, r104_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0))));
        const double z110 = fma(e4, r114_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0))));
        const double z200 = fma(e4, r204_0, fma(e3, r203_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0))));
        double j = 0.0;
        {
          const double v = fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[15] = fma(Dbd[15], v, Kac[15]);
          Kad[15] = fma(Dbc[15], v, Kad[15]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[15] = fma(ac0, v, Kbd[15]);
        }
        {
          const double v = fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[15] = fma(Dbd[16], v, Kac[15]);
          Kad[16] = fma(Dbc[15], v, Kad[16]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[16] = fma(ac0, v, Kbd[16]);
        }
        {
          const double v = fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[15] = fma(Dbd[17], v, Kac[15]);
          Kad[17] = fma(Dbc[15], v, Kad[17]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[17] = fma(ac0, v, Kbd[17]);
        }
        {
          const double v = fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[16] = fma(Dbd[15], v, Kac[16]);
          Kad[15] = fma(Dbc[16], v, Kad[15]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[15] = fma(ac1, v, Kbd[15]);
        }
        {
          const double v = fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[16] = fma(Dbd[16], v, Kac[16]);
          Kad[16] = fma(Dbc[16], v, Kad[16]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[16] = fma(ac1, v, Kbd[16]);
        }
        {
          const double v = fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[16] = fma(Dbd[17], v, Kac[16]);
          Kad[17] = fma(Dbc[16], v, Kad[17]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[17] = fma(ac1, v, Kbd[17]);
        }
        {
          const double v = fma(k2_0_101, z101, fma(k2_0_100, z100, fma(k2_0_001, z001, k2_0_000 * z000)));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[17] = fma(Dbd[15], v, Kac[17]);
          Kad[15] = fma(Dbc[17], v, Kad[15]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[15] = fma(ac2, v, Kbd[15]);
        }
        {
          const double v = fma(k2_1_011, z011, fma(k2_1_010, z010, fma(k2_1_001, z001, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[17] = fma(Dbd[16], v, Kac[17]);
          Kad[16] = fma(Dbc[17], v, Kad[16]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[16] = fma(ac2, v, Kbd[16]);
        }
        {
          const double v = fma(k2_2_002, z002, fma(k2_2_001, z001, k2_2_000 * z000));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[17] = fma(Dbd[17], v, Kac[17]);
          Kad[17] = fma(Dbc[17], v, Kad[17]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[17] = fma(ac2, v, Kbd[17]);
        }
        Jab[35] += j;
      }
    }
  }
};
__device__ const unsigned kC2211Md_index[336] = {22,23,24,25,26,274,530,275,531,276,532,277,533,783,1039,1295,784,1040,1296,785,1041,1297,65554,131090,65555,131091,65556,131092,65557,131093,65807,131343,66063,131599,65808,131344,66064,131600,65809,131345,66065,131601,196623,262159,327695,196624,262160,327696,196625,262161,327697,1547,1803,1548,1804,1549,1805,1550,1806,2056,2312,2568,2057,2313,2569,2058,2314,2570,2822,3078,3334,3590,2823,3079,3335,3591,67080,132616,67336,132872,67081,132617,67337,132873,67082,132618,67338,132874,67590,133126,67846,133382,68102,133638,67591,133127,67847,133383,68103,133639,198150,263686,329222,198406,263942,329478,198151,263687,329223,198407,263943,329479,3843,4099,4355,3844,4100,4356,3845,4101,4357,4609,4865,5121,5377,4610,4866,5122,5378,5632,5888,6144,6400,6656,69377,134913,69633,135169,69889,135425,69378,134914,69634,135170,69890,135426,70144,135680,70400,135936,70656,136192,70912,136448,200448,265984,331520,200704,266240,331776,200960,266496,332032,393227,458763,393228,458764,393229,458765,393230,458766,393480,459016,393736,459272,393481,459017,393737,459273,393482,459018,393738,459274,393990,459526,394246,459782,394502,460038,393991,459527,394247,459783,394503,460039,524296,589832,655368,524297,589833,655369,524298,589834,655370,524550,590086,655622,524806,590342,655878,524551,590087,655623,524807,590343,655879,720902,786438,851974,917510,720903,786439,851975,917511,394755,460291,395011,460547,394756,460292,395012,460548,394757,460293,395013,460549,395265,460801,395521,461057,395777,461313,395266,460802,395522,461058,395778,461314,396032,461568,396288,461824,396544,462080,396800,462336,525825,591361,656897,526081,591617,657153,525826,591362,656898,526082,591618,657154,526336,591872,657408,526592,592128,657664,526848,592384,657920,722432,787968,853504,919040,722688,788224,853760,919296,983043,1048579,1114115,983044,1048580,1114116,983045,1048581,1114117,983297,1048833,1114369,983553,1049089,1114625,983298,1048834,1114370,983554,1049090,1114626,983808,1049344,1114880,984064,1049600,1115136,984320,1049856,1115392,1179649,1245185,1310721,1376257,1179650,1245186,1310722,1376258,1179904,1245440,1310976,1376512,1180160,1245696,1311232,1376768,1441792,1507328,1572864,1638400,1703936};
__device__ inline const unsigned* C2211Md::index() { return kC2211Md_index; }
}  // namespace qf
