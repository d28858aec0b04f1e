// Generated by quick_amd/codegen/gen_md.py - do not edit.
#pragma once
#include "../qf_md.h"
namespace qf {
// (dp|dp): 84 Hermite Coulomb integrals, 108 bra products
struct C2121Md {
  static constexpr int La = 2, Lb = 1, Lc = 2, Ld = 1, L = 6;
  static constexpr int N1 = 15, NE = 108;   // 1D entries per direction, product table
  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16
  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p
  template <class T>
  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, T out) {
    const double be010 = Y;
    const double be011 = h;
    const double be100 = X;
    const double be101 = h;
    const double be110 = fma(1.0, be101, be100 * Y);
    const double be111 = fma(be100, h, be101 * Y);
    const double be112 = be101 * h;
    const double be200 = fma(1.0, be101, be100 * X);
    const double be201 = fma(be100, h, be101 * X);
    const double be202 = be101 * h;
    const double be210 = fma(1.0, be201, be200 * Y);
    const double be211 = fma(2.0, be202, fma(be200, h, be201 * Y));
    const double be212 = fma(be201, h, be202 * Y);
    const double be213 = be202 * h;
    out[0] = 1.0;
    out[1] = be010;
    out[2] = be011;
    out[3] = be100;
    out[4] = be101;
    out[5] = be110;
    out[6] = be111;
    out[7] = be112;
    out[8] = be200;
    out[9] = be201;
    out[10] = be202;
    out[11] = be210;
    out[12] = be211;
    out[13] = be212;
    out[14] = be213;
  }
  // Dbc and Dbd with the cons of b; oc, od: first elements of the a-c and a-d blocks of P
  template <class ET, class PT, class PU>
  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a, const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[18], const double (&Dbc)[18], const double (&Dbd)[9], double (&Jcd)[18], double (&Kbc)[18], double (&Kbd)[9], double (&Jab)[18], double (&Kac)[36], double (&Kad)[18]) {
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
    const double kxe200 = fma(-1.0, kxe101, kxe100 * QC[0]);
    const double kxe201 = fma(kxe100, (-hk), kxe101 * QC[0]);
    const double kxe202 = kxe101 * (-hk);
    const double kxe210 = fma(-1.0, kxe201, kxe200 * QD[0]);
    const double kxe211 = fma(-2.0, kxe202, fma(kxe200, (-hk), kxe201 * QD[0]));
    const double kxe212 = fma(kxe201, (-hk), kxe202 * QD[0]);
    const double kxe213 = kxe202 * (-hk);
    const double kye010 = QD[1];
    const double kye011 = (-hk);
    const double kye100 = QC[1];
    const double kye101 = (-hk);
    const double kye110 = fma(-1.0, kye101, kye100 * QD[1]);
    const double kye111 = fma(kye100, (-hk), kye101 * QD[1]);
    const double kye112 = kye101 * (-hk);
    const double kye200 = fma(-1.0, kye101, kye100 * QC[1]);
    const double kye201 = fma(kye100, (-hk), kye101 * QC[1]);
    const double kye202 = kye101 * (-hk);
    const double kye210 = fma(-1.0, kye201, kye200 * QD[1]);
    const double kye211 = fma(-2.0, kye202, fma(kye200, (-hk), kye201 * QD[1]));
    const double kye212 = fma(kye201, (-hk), kye202 * QD[1]);
    const double kye213 = kye202 * (-hk);
    const double kze010 = QD[2];
    const double kze011 = (-hk);
    const double kze100 = QC[2];
    const double kze101 = (-hk);
    const double kze110 = fma(-1.0, kze101, kze100 * QD[2]);
    const double kze111 = fma(kze100, (-hk), kze101 * QD[2]);
    const double kze112 = kze101 * (-hk);
    const double kze200 = fma(-1.0, kze101, kze100 * QC[2]);
    const double kze201 = fma(kze100, (-hk), kze101 * QC[2]);
    const double kze202 = kze101 * (-hk);
    const double kze210 = fma(-1.0, kze201, kze200 * QD[2]);
    const double kze211 = fma(-2.0, kze202, fma(kze200, (-hk), kze201 * QD[2]));
    const double kze212 = fma(kze201, (-hk), kze202 * QD[2]);
    const double kze213 = kze202 * (-hk);
    const double k0_0_000 = kxe210 * (kCons[2][0] * kCons[1][0]);
    const double k0_0_100 = kxe211 * (kCons[2][0] * kCons[1][0]);
    const double k0_0_200 = kxe212 * (kCons[2][0] * kCons[1][0]);
    const double k0_0_300 = kxe213 * (kCons[2][0] * kCons[1][0]);
    const double k0_1_000 = kxe200 * kye010 * (kCons[2][0] * kCons[1][1]);
    const double k0_1_010 = kxe200 * kye011 * (kCons[2][0] * kCons[1][1]);
    const double k0_1_100 = kxe201 * kye010 * (kCons[2][0] * kCons[1][1]);
    const double k0_1_110 = kxe201 * kye011 * (kCons[2][0] * kCons[1][1]);
    const double k0_1_200 = kxe202 * kye010 * (kCons[2][0] * kCons[1][1]);
    const double k0_1_210 = kxe202 * kye011 * (kCons[2][0] * kCons[1][1]);
    const double k0_2_000 = kxe200 * kze010 * (kCons[2][0] * kCons[1][2]);
    const double k0_2_001 = kxe200 * kze011 * (kCons[2][0] * kCons[1][2]);
    const double k0_2_100 = kxe201 * kze010 * (kCons[2][0] * kCons[1][2]);
    const double k0_2_101 = kxe201 * kze011 * (kCons[2][0] * kCons[1][2]);
    const double k0_2_200 = kxe202 * kze010 * (kCons[2][0] * kCons[1][2]);
    const double k0_2_201 = kxe202 * kze011 * (kCons[2][0] * kCons[1][2]);
    const double k1_0_000 = kxe110 * kye100 * (kCons[2][1] * kCons[1][0]);
    const double k1_0_010 = kxe110 * kye101 * (kCons[2][1] * kCons[1][0]);
    const double k1_0_100 = kxe111 * kye100 * (kCons[2][1] * kCons[1][0]);
    const double k1_0_110 = kxe111 * kye101 * (kCons[2][1] * kCons[1][0]);
    const double k1_0_200 = kxe112 * kye100 * (kCons[2][1] * kCons[1][0]);
    const double k1_0_210 = kxe112 * kye101 * (kCons[2][1] * kCons[1][0]);
    const double k1_1_000 = kxe100 * kye110 * (kCons[2][1] * kCons[1][1]);
    const double k1_1_010 = kxe100 * kye111 * (kCons[2][1] * kCons[1][1]);
    const double k1_1_020 = kxe100 * kye112 * (kCons[2][1] * kCons[1][1]);
    const double k1_1_100 = kxe101 * kye110 * (kCons[2][1] * kCons[1][1]);
    const double k1_1_110 = kxe101 * kye111 * (kCons[2][1] * kCons[1][1]);
    const double k1_1_120 = kxe101 * kye112 * (kCons[2][1] * kCons[1][1]);
    const double k1_2_000 = kxe100 * kye100 * kze010 * (kCons[2][1] * kCons[1][2]);
    const double k1_2_001 = kxe100 * kye100 * kze011 * (kCons[2][1] * kCons[1][2]);
    const double k1_2_010 = kxe100 * kye101 * kze010 * (kCons[2][1] * kCons[1][2]);
    const double k1_2_011 = kxe100 * kye101 * kze011 * (kCons[2][1] * kCons[1][2]);
    const double k1_2_100 = kxe101 * kye100 * kze010 * (kCons[2][1] * kCons[1][2]);
    const double k1_2_101 = kxe101 * kye100 * kze011 * (kCons[2][1] * kCons[1][2]);
    const double k1_2_110 = kxe101 * kye101 * kze010 * (kCons[2][1] * kCons[1][2]);
    const double k1_2_111 = kxe101 * kye101 * kze011 * (kCons[2][1] * kCons[1][2]);
    const double k2_0_000 = kxe010 * kye200 * (kCons[2][2] * kCons[1][0]);
    const double k2_0_010 = kxe010 * kye201 * (kCons[2][2] * kCons[1][0]);
    const double k2_0_020 = kxe010 * kye202 * (kCons[2][2] * kCons[1][0]);
    const double k2_0_100 = kxe011 * kye200 * (kCons[2][2] * kCons[1][0]);
    const double k2_0_110 = kxe011 * kye201 * (kCons[2][2] * kCons[1][0]);
    const double k2_0_120 = kxe011 * kye202 * (kCons[2][2] * kCons[1][0]);
    const double k2_1_000 = kye210 * (kCons[2][2] * kCons[1][1]);
    const double k2_1_010 = kye211 * (kCons[2][2] * kCons[1][1]);
    const double k2_1_020 = kye212 * (kCons[2][2] * kCons[1][1]);
    const double k2_1_030 = kye213 * (kCons[2][2] * kCons[1][1]);
    const double k2_2_000 = kye200 * kze010 * (kCons[2][2] * kCons[1][2]);
    const double k2_2_001 = kye200 * kze011 * (kCons[2][2] * kCons[1][2]);
    const double k2_2_010 = kye201 * kze010 * (kCons[2][2] * kCons[1][2]);
    const double k2_2_011 = kye201 * kze011 * (kCons[2][2] * kCons[1][2]);
    const double k2_2_020 = kye202 * kze010 * (kCons[2][2] * kCons[1][2]);
    const double k2_2_021 = kye202 * kze011 * (kCons[2][2] * kCons[1][2]);
    const double k3_0_000 = kxe110 * kze100 * (kCons[2][3] * kCons[1][0]);
    const double k3_0_001 = kxe110 * kze101 * (kCons[2][3] * kCons[1][0]);
    const double k3_0_100 = kxe111 * kze100 * (kCons[2][3] * kCons[1][0]);
    const double k3_0_101 = kxe111 * kze101 * (kCons[2][3] * kCons[1][0]);
    const double k3_0_200 = kxe112 * kze100 * (kCons[2][3] * kCons[1][0]);
    const double k3_0_201 = kxe112 * kze101 * (kCons[2][3] * kCons[1][0]);
    const double k3_1_000 = kxe100 * kye010 * kze100 * (kCons[2][3] * kCons[1][1]);
    const double k3_1_001 = kxe100 * kye010 * kze101 * (kCons[2][3] * kCons[1][1]);
    const double k3_1_010 = kxe100 * kye011 * kze100 * (kCons[2][3] * kCons[1][1]);
    const double k3_1_011 = kxe100 * kye011 * kze101 * (kCons[2][3] * kCons[1][1]);
    const double k3_1_100 = kxe101 * kye010 * kze100 * (kCons[2][3] * kCons[1][1]);
    const double k3_1_101 = kxe101 * kye010 * kze101 * (kCons[2][3] * kCons[1][1]);
    const double k3_1_110 = kxe101 * kye011 * kze100 * (kCons[2][3] * kCons[1][1]);
    const double k3_1_111 = kxe101 * kye011 * kze101 * (kCons[2][3] * kCons[1][1]);
    const double k3_2_000 = kxe100 * kze110 * (kCons[2][3] * kCons[1][2]);
    const double k3_2_001 = kxe100 * kze111 * (kCons[2][3] * kCons[1][2]);
    const double k3_2_002 = kxe100 * kze112 * (kCons[2][3] * kCons[1][2]);
    const double k3_2_100 = kxe101 * kze110 * (kCons[2][3] * kCons[1][2]);
    const double k3_2_101 = kxe101 * kze111 * (kCons[2][3] * kCons[1][2]);
    const double k3_2_102 = kxe101 * kze112 * (kCons[2][3] * kCons[1][2]);
    const double k4_0_000 = kxe010 * kye100 * kze100 * (kCons[2][4] * kCons[1][0]);
    const double k4_0_001 = kxe010 * kye100 * kze101 * (kCons[2][4] * kCons[1][0]);
    const double k4_0_010 = kxe010 * kye101 * kze100 * (kCons[2][4] * kCons[1][0]);
    const double k4_0_011 = kxe010 * kye101 * kze101 * (kCons[2][4] * kCons[1][0]);
    const double k4_0_100 = kxe011 * kye100 * kze100 * (kCons[2][4] * kCons[1][0]);
    const double k4_0_101 = kxe011 * kye100 * kze101 * (kCons[2][4] * kCons[1][0]);
    const double k4_0_110 = kxe011 * kye101 * kze100 * (kCons[2][4] * kCons[1][0]);
    const double k4_0_111 = kxe011 * kye101 * kze101 * (kCons[2][4] * kCons[1][0]);
    const double k4_1_000 = kye110 * kze100 * (kCons[2][4] * kCons[1][1]);
    const double k4_1_001 = kye110 * kze101 * (kCons[2][4] * kCons[1][1]);
    const double k4_1_010 = kye111 * kze100 * (kCons[2][4] * kCons[1][1]);
    const double k4_1_011 = kye111 * kze101 * (kCons[2][4] * kCons[1][1]);
    const double k4_1_020 = kye112 * kze100 * (kCons[2][4] * kCons[1][1]);
    const double k4_1_021 = kye112 * kze101 * (kCons[2][4] * kCons[1][1]);
    const double k4_2_000 = kye100 * kze110 * (kCons[2][4] * kCons[1][2]);
    const double k4_2_001 = kye100 * kze111 * (kCons[2][4] * kCons[1][2]);
    const double k4_2_002 = kye100 * kze112 * (kCons[2][4] * kCons[1][2]);
    const double k4_2_010 = kye101 * kze110 * (kCons[2][4] * kCons[1][2]);
    const double k4_2_011 = kye101 * kze111 * (kCons[2][4] * kCons[1][2]);
    const double k4_2_012 = kye101 * kze112 * (kCons[2][4] * kCons[1][2]);
    const double k5_0_000 = kxe010 * kze200 * (kCons[2][5] * kCons[1][0]);
    const double k5_0_001 = kxe010 * kze201 * (kCons[2][5] * kCons[1][0]);
    const double k5_0_002 = kxe010 * kze202 * (kCons[2][5] * kCons[1][0]);
    const double k5_0_100 = kxe011 * kze200 * (kCons[2][5] * kCons[1][0]);
    const double k5_0_101 = kxe011 * kze201 * (kCons[2][5] * kCons[1][0]);
    const double k5_0_102 = kxe011 * kze202 * (kCons[2][5] * kCons[1][0]);
    const double k5_1_000 = kye010 * kze200 * (kCons[2][5] * kCons[1][1]);
    const double k5_1_001 = kye010 * kze201 * (kCons[2][5] * kCons[1][1]);
    const double k5_1_002 = kye010 * kze202 * (kCons[2][5] * kCons[1][1]);
    const double k5_1_010 = kye011 * kze200 * (kCons[2][5] * kCons[1][1]);
    const double k5_1_011 = kye011 * kze201 * (kCons[2][5] * kCons[1][1]);
    const double k5_1_012 = kye011 * kze202 * (kCons[2][5] * kCons[1][1]);
    const double k5_2_000 = kze210 * (kCons[2][5] * kCons[1][2]);
    const double k5_2_001 = kze211 * (kCons[2][5] * kCons[1][2]);
    const double k5_2_002 = kze212 * (kCons[2][5] * kCons[1][2]);
    const double k5_2_003 = kze213 * (kCons[2][5] * kCons[1][2]);
    QF_OPAQUE(oc);
    QF_OPAQUE(od);
    {
      const double ac0 = P[oc + 0 * n + 0] * kCons[2][0];
      const double ac1 = P[oc + 0 * n + 1] * kCons[2][0];
      const double ac2 = P[oc + 0 * n + 2] * kCons[2][0];
      const double ac3 = P[oc + 0 * n + 3] * kCons[2][0];
      const double ac4 = P[oc + 0 * n + 4] * kCons[2][0];
      const double ac5 = P[oc + 0 * n + 5] * kCons[2][0];
      const double ad0 = P[od + 0 * n + 0] * kCons[2][0];
      const double ad1 = P[od + 0 * n + 1] * kCons[2][0];
      const double ad2 = P[od + 0 * n + 2] * kCons[2][0];
      {
        const double ab = Pab[0 * n + 0] * (kCons[2][0] * kCons[1][0]);
        const double e0 = E[0];
        const double e1 = E[1];
        const double e2 = E[2];
        const double e3 = E[3];
        const double z000 = fma(e3, r300_0, fma(e2, r200_0, fma(e1, r100_0, e0 * r000_0)));
        const double z001 = fma(e3, r301_0, fma(e2, r201_0, fma(e1, r101_0, e0 * r001_0)));
        const double z010 = fma(e3, r310_0, fma(e2, r210_0, fma(e1, r110_0, e0 * r010_0)));
        const double z100 = fma(e3, r400_0, fma(e2, r300_0, fma(e1, r200_0, e0 * r100_0)));
        const double z002 = fma(e3, r302_0, fma(e2, r202_0, fma(e1, r102_0, e0 * r002_0)));
        const double z011 = fma(e3, r311_0, fma(e2, r211_0, fma(e1, r111_0, e0 * r011_0)));
        const double z020 = fma(e3, r320_0, fma(e2, r220_0, fma(e1, r120_0, e0 * r020_0)));
        const double z101 = fma(e3, r401_0, fma(e2, r301_0, fma(e1, r201_0, e0 * r101_0)));
        const double z110 = fma(e3, r410_0, fma(e2, r310_0, fma(e1, r210_0, e0 * r110_0)));
        const double z200 = fma(e3, r500_0, fma(e2, r400_0, fma(e1, r300_0, e0 * r200_0)));
        const double z003 = fma(e3, r303_0, fma(e2, r203_0, fma(e1, r103_0, e0 * r003_0)));
        const double z012 = fma(e3, r312_0, fma(e2, r212_0, fma(e1, r112_0, e0 * r012_0)));
        const double z021 = fma(e3, r321_0, fma(e2, r221_0, fma(e1, r121_0, e0 * r021_0)));
        const double z030 = fma(e3, r330_0, fma(e2, r230_0, fma(e1, r130_0, e0 * r030_0)));
        const double z102 = fma(e3, r402_0, fma(e2, r302_0, fma(e1, r202_0, e0 * r102_0)));
        const double z111 = fma(e3, r411_0, fma(e2, r311_0, fma(e1, r211_0, e0 * r111_0)));
        const double z120 = fma(e3, r420_0, fma(e2, r320_0, fma(e1, r220_0, e0 * r120_0)));
        const double z201 = fma(e3, r501_0, fma(e2, r401_0, fma(e1, r301_0, e0 * r201_0)));
        const double z210 = fma(e3, r510_0, fma(e2, r410_0, fma(e1, r310_0, e0 * r210_0)));
        const double z300 = fma(e3, r600_0, fma(e2, r500_0, fma(e1, r400_0, e0 * r300_0)));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[0], v, Kac[0]);
          Kad[0] = fma(Dbc[0], v, Kad[0]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[1], v, Kac[0]);
          Kad[1] = fma(Dbc[0], v, Kad[1]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[2], v, Kac[0]);
          Kad[2] = fma(Dbc[0], v, Kad[2]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[0], v, Kac[1]);
          Kad[0] = fma(Dbc[1], v, Kad[0]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[1], v, Kac[1]);
          Kad[1] = fma(Dbc[1], v, Kad[1]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[2], v, Kac[1]);
          Kad[2] = fma(Dbc[1], v, Kad[2]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[0], v, Kac[2]);
          Kad[0] = fma(Dbc[2], v, Kad[0]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[1], v, Kac[2]);
          Kad[1] = fma(Dbc[2], v, Kad[1]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[2], v, Kac[2]);
          Kad[2] = fma(Dbc[2], v, Kad[2]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[3] = fma(Dbd[0], v, Kac[3]);
          Kad[0] = fma(Dbc[3], v, Kad[0]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[0] = fma(ac3, v, Kbd[0]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[3] = fma(Dbd[1], v, Kac[3]);
          Kad[1] = fma(Dbc[3], v, Kad[1]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[1] = fma(ac3, v, Kbd[1]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[3] = fma(Dbd[2], v, Kac[3]);
          Kad[2] = fma(Dbc[3], v, Kad[2]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[2] = fma(ac3, v, Kbd[2]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[4] = fma(Dbd[0], v, Kac[4]);
          Kad[0] = fma(Dbc[4], v, Kad[0]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[0] = fma(ac4, v, Kbd[0]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[4] = fma(Dbd[1], v, Kac[4]);
          Kad[1] = fma(Dbc[4], v, Kad[1]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[1] = fma(ac4, v, Kbd[1]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[4] = fma(Dbd[2], v, Kac[4]);
          Kad[2] = fma(Dbc[4], v, Kad[2]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[2] = fma(ac4, v, Kbd[2]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[5] = fma(Dbd[0], v, Kac[5]);
          Kad[0] = fma(Dbc[5], v, Kad[0]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[0] = fma(ac5, v, Kbd[0]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[5] = fma(Dbd[1], v, Kac[5]);
          Kad[1] = fma(Dbc[5], v, Kad[1]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[1] = fma(ac5, v, Kbd[1]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[5] = fma(Dbd[2], v, Kac[5]);
          Kad[2] = fma(Dbc[5], v, Kad[2]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[2] = fma(ac5, v, Kbd[2]);
        }
        Jab[0] += j;
      }
      {
        const double ab = Pab[0 * n + 1] * (kCons[2][0] * kCons[1][1]);
        const double e0 = E[4];
        const double e1 = E[5];
        const double e2 = E[6];
        const double e3 = E[7];
        const double e4 = E[8];
        const double e5 = E[9];
        const double z000 = fma(e5, r210_0, fma(e4, r200_0, fma(e3, r110_0, fma(e2, r100_0, fma(e1, r010_0, e0 * r000_0)))));
        const double z001 = fma(e5, r211_0, fma(e4, r201_0, fma(e3, r111_0, fma(e2, r101_0, fma(e1, r011_0, e0 * r001_0)))));
        const double z010 = fma(e5, r220_0, fma(e4, r210_0, fma(e3, r120_0, fma(e2, r110_0, fma(e1, r020_0, e0 * r010_0)))));
        const double z100 = fma(e5, r310_0, fma(e4, r300_0, fma(e3, r210_0, fma(e2, r200_0, fma(e1, r110_0, e0 * r100_0)))));
        const double z002 = fma(e5, r212_0, fma(e4, r202_0, fma(e3, r112_0, fma(e2, r102_0, fma(e1, r012_0, e0 * r002_0)))));
        const double z011 = fma(e5, r221_0, fma(e4, r211_0, fma(e3, r121_0, fma(e2, r111_0, fma(e1, r021_0, e0 * r011_0)))));
        const double z020 = fma(e5, r230_0, fma(e4, r220_0, fma(e3, r130_0, fma(e2, r120_0, fma(e1, r030_0, e0 * r020_0)))));
        const double z101 = fma(e5, r311_0, fma(e4, r301_0, fma(e3, r211_0, fma(e2, r201_0, fma(e1, r111_0, e0 * r101_0)))));
        const double z110 = fma(e5, r320_0, fma(e4, r310_0, fma(e3, r220_0, fma(e2, r210_0, fma(e1, r120_0, e0 * r110_0)))));
        const double z200 = fma(e5, r410_0, fma(e4, r400_0, fma(e3, r310_0, fma(e2, r300_0, fma(e1, r210_0, e0 * r200_0)))));
        const double z003 = fma(e5, r213_0, fma(e4, r203_0, fma(e3, r113_0, fma(e2, r103_0, fma(e1, r013_0, e0 * r003_0)))));
        const double z012 = fma(e5, r222_0, fma(e4, r212_0, fma(e3, r122_0, fma(e2, r112_0, fma(e1, r022_0, e0 * r012_0)))));
        const double z021 = fma(e5, r231_0, fma(e4, r221_0, fma(e3, r131_0, fma(e2, r121_0, fma(e1, r031_0, e0 * r021_0)))));
        const double z030 = fma(e5, r240_0, fma(e4, r230_0, fma(e3, r140_0, fma(e2, r130_0, fma(e1, r040_0, e0 * r030_0)))));
        const double z102 = fma(e5, r312_0, fma(e4, r302_0, fma(e3, r212_0, fma(e2, r202_0, fma(e1, r112_0, e0 * r102_0)))));
        const double z111 = fma(e5, r321_0, fma(e4, r311_0, fma(e3, r221_0, fma(e2, r211_0, fma(e1, r121_0, e0 * r111_0)))));
        const double z120 = fma(e5, r330_0, fma(e4, r320_0, fma(e3, r230_0, fma(e2, r220_0, fma(e1, r130_0, e0 * r120_0)))));
        const double z201 = fma(e5, r411_0, fma(e4, r401_0, fma(e3, r311_0, fma(e2, r301_0, fma(e1, r211_0, e0 * r201_0)))));
        const double z210 = fma(e5, r420_0, fma(e4, r410_0, fma(e3, r320_0, fma(e2, r310_0, fma(e1, r220_0, e0 * r210_0)))));
        const double z300 = fma(e5, r510_0, fma(e4, r500_0, fma(e3, r410_0, fma(e2, r400_0, fma(e1, r310_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[3], v, Kac[0]);
          Kad[0] = fma(Dbc[6], v, Kad[0]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[4], v, Kac[0]);
          Kad[1] = fma(Dbc[6], v, Kad[1]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[5], v, Kac[0]);
          Kad[2] = fma(Dbc[6], v, Kad[2]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[3], v, Kac[1]);
          Kad[0] = fma(Dbc[7], v, Kad[0]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[4], v, Kac[1]);
          Kad[1] = fma(Dbc[7], v, Kad[1]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[5], v, Kac[1]);
          Kad[2] = fma(Dbc[7], v, Kad[2]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[3], v, Kac[2]);
          Kad[0] = fma(Dbc[8], v, Kad[0]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[4], v, Kac[2]);
          Kad[1] = fma(Dbc[8], v, Kad[1]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[5], v, Kac[2]);
          Kad[2] = fma(Dbc[8], v, Kad[2]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[3] = fma(Dbd[3], v, Kac[3]);
          Kad[0] = fma(Dbc[9], v, Kad[0]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[3] = fma(ac3, v, Kbd[3]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[3] = fma(Dbd[4], v, Kac[3]);
          Kad[1] = fma(Dbc[9], v, Kad[1]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[4] = fma(ac3, v, Kbd[4]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[3] = fma(Dbd[5], v, Kac[3]);
          Kad[2] = fma(Dbc[9], v, Kad[2]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[5] = fma(ac3, v, Kbd[5]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[4] = fma(Dbd[3], v, Kac[4]);
          Kad[0] = fma(Dbc[10], v, Kad[0]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[3] = fma(ac4, v, Kbd[3]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[4] = fma(Dbd[4], v, Kac[4]);
          Kad[1] = fma(Dbc[10], v, Kad[1]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[4] = fma(ac4, v, Kbd[4]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[4] = fma(Dbd[5], v, Kac[4]);
          Kad[2] = fma(Dbc[10], v, Kad[2]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[5] = fma(ac4, v, Kbd[5]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[5] = fma(Dbd[3], v, Kac[5]);
          Kad[0] = fma(Dbc[11], v, Kad[0]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[3] = fma(ac5, v, Kbd[3]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[5] = fma(Dbd[4], v, Kac[5]);
          Kad[1] = fma(Dbc[11], v, Kad[1]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[4] = fma(ac5, v, Kbd[4]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[5] = fma(Dbd[5], v, Kac[5]);
          Kad[2] = fma(Dbc[11], v, Kad[2]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[5] = fma(ac5, v, Kbd[5]);
        }
        Jab[1] += j;
      }
      {
        const double ab = Pab[0 * n + 2] * (kCons[2][0] * kCons[1][2]);
        const double e0 = E[10];
        const double e1 = E[11];
        const double e2 = E[12];
        const double e3 = E[13];
        const double e4 = E[14];
        const double e5 = E[15];
        const double z000 = fma(e5, r201_0, fma(e4, r200_0, fma(e3, r101_0, fma(e2, r100_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r202_0, fma(e4, r201_0, fma(e3, r102_0, fma(e2, r101_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r211_0, fma(e4, r210_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r301_0, fma(e4, r300_0, fma(e3, r201_0, fma(e2, r200_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r203_0, fma(e4, r202_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r212_0, fma(e4, r211_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r221_0, fma(e4, r220_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r302_0, fma(e4, r301_0, fma(e3, r202_0, fma(e2, r201_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r311_0, fma(e4, r310_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r401_0, fma(e4, r400_0, fma(e3, r301_0, fma(e2, r300_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r204_0, fma(e4, r203_0, fma(e3, r104_0, fma(e2, r103_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r213_0, fma(e4, r212_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r122_0, fma(e2, r121_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r231_0, fma(e4, r230_0, fma(e3, r131_0, fma(e2, r130_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r303_0, fma(e4, r302_0, fma(e3, r203_0, fma(e2, r202_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r312_0, fma(e4, r311_0, fma(e3, r212_0, fma(e2, r211_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r321_0, fma(e4, r320_0, fma(e3, r221_0, fma(e2, r220_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r402_0, fma(e4, r401_0, fma(e3, r302_0, fma(e2, r301_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r411_0, fma(e4, r410_0, fma(e3, r311_0, fma(e2, r310_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r501_0, fma(e4, r500_0, fma(e3, r401_0, fma(e2, r400_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[0] = fma(Dbd[6], v, Kac[0]);
          Kad[0] = fma(Dbc[12], v, Kad[0]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[0] = fma(Dbd[7], v, Kac[0]);
          Kad[1] = fma(Dbc[12], v, Kad[1]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[0] = fma(Dbd[8], v, Kac[0]);
          Kad[2] = fma(Dbc[12], v, Kad[2]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[1] = fma(Dbd[6], v, Kac[1]);
          Kad[0] = fma(Dbc[13], v, Kad[0]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[1] = fma(Dbd[7], v, Kac[1]);
          Kad[1] = fma(Dbc[13], v, Kad[1]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[1] = fma(Dbd[8], v, Kac[1]);
          Kad[2] = fma(Dbc[13], v, Kad[2]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[2] = fma(Dbd[6], v, Kac[2]);
          Kad[0] = fma(Dbc[14], v, Kad[0]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[2] = fma(Dbd[7], v, Kac[2]);
          Kad[1] = fma(Dbc[14], v, Kad[1]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[2] = fma(Dbd[8], v, Kac[2]);
          Kad[2] = fma(Dbc[14], v, Kad[2]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[3] = fma(Dbd[6], v, Kac[3]);
          Kad[0] = fma(Dbc[15], v, Kad[0]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[6] = fma(ac3, v, Kbd[6]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[3] = fma(Dbd[7], v, Kac[3]);
          Kad[1] = fma(Dbc[15], v, Kad[1]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[7] = fma(ac3, v, Kbd[7]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[3] = fma(Dbd[8], v, Kac[3]);
          Kad[2] = fma(Dbc[15], v, Kad[2]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[8] = fma(ac3, v, Kbd[8]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[4] = fma(Dbd[6], v, Kac[4]);
          Kad[0] = fma(Dbc[16], v, Kad[0]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[6] = fma(ac4, v, Kbd[6]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[4] = fma(Dbd[7], v, Kac[4]);
          Kad[1] = fma(Dbc[16], v, Kad[1]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[7] = fma(ac4, v, Kbd[7]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[4] = fma(Dbd[8], v, Kac[4]);
          Kad[2] = fma(Dbc[16], v, Kad[2]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[8] = fma(ac4, v, Kbd[8]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[5] = fma(Dbd[6], v, Kac[5]);
          Kad[0] = fma(Dbc[17], v, Kad[0]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[6] = fma(ac5, v, Kbd[6]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[5] = fma(Dbd[7], v, Kac[5]);
          Kad[1] = fma(Dbc[17], v, Kad[1]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[7] = fma(ac5, v, Kbd[7]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[5] = fma(Dbd[8], v, Kac[5]);
          Kad[2] = fma(Dbc[17], v, Kad[2]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[8] = fma(ac5, v, Kbd[8]);
        }
        Jab[2] += j;
      }
    }
    {
      const double ac0 = P[oc + 1 * n + 0] * kCons[2][1];
      const double ac1 = P[oc + 1 * n + 1] * kCons[2][1];
      const double ac2 = P[oc + 1 * n + 2] * kCons[2][1];
      const double ac3 = P[oc + 1 * n + 3] * kCons[2][1];
      const double ac4 = P[oc + 1 * n + 4] * kCons[2][1];
      const double ac5 = P[oc + 1 * n + 5] * kCons[2][1];
      const double ad0 = P[od + 1 * n + 0] * kCons[2][1];
      const double ad1 = P[od + 1 * n + 1] * kCons[2][1];
      const double ad2 = P[od + 1 * n + 2] * kCons[2][1];
      {
        const double ab = Pab[1 * n + 0] * (kCons[2][1] * kCons[1][0]);
        const double e0 = E[16];
        const double e1 = E[17];
        const double e2 = E[18];
        const double e3 = E[19];
        const double e4 = E[20];
        const double e5 = E[21];
        const double z000 = fma(e5, r210_0, fma(e4, r200_0, fma(e3, r110_0, fma(e2, r100_0, fma(e1, r010_0, e0 * r000_0)))));
        const double z001 = fma(e5, r211_0, fma(e4, r201_0, fma(e3, r111_0, fma(e2, r101_0, fma(e1, r011_0, e0 * r001_0)))));
        const double z010 = fma(e5, r220_0, fma(e4, r210_0, fma(e3, r120_0, fma(e2, r110_0, fma(e1, r020_0, e0 * r010_0)))));
        const double z100 = fma(e5, r310_0, fma(e4, r300_0, fma(e3, r210_0, fma(e2, r200_0, fma(e1, r110_0, e0 * r100_0)))));
        const double z002 = fma(e5, r212_0, fma(e4, r202_0, fma(e3, r112_0, fma(e2, r102_0, fma(e1, r012_0, e0 * r002_0)))));
        const double z011 = fma(e5, r221_0, fma(e4, r211_0, fma(e3, r121_0, fma(e2, r111_0, fma(e1, r021_0, e0 * r011_0)))));
        const double z020 = fma(e5, r230_0, fma(e4, r220_0, fma(e3, r130_0, fma(e2, r120_0, fma(e1, r030_0, e0 * r020_0)))));
        const double z101 = fma(e5, r311_0, fma(e4, r301_0, fma(e3, r211_0, fma(e2, r201_0, fma(e1, r111_0, e0 * r101_0)))));
        const double z110 = fma(e5, r320_0, fma(e4, r310_0, fma(e3, r220_0, fma(e2, r210_0, fma(e1, r120_0, e0 * r110_0)))));
        const double z200 = fma(e5, r410_0, fma(e4, r400_0, fma(e3, r310_0, fma(e2, r300_0, fma(e1, r210_0, e0 * r200_0)))));
        const double z003 = fma(e5, r213_0, fma(e4, r203_0, fma(e3, r113_0, fma(e2, r103_0, fma(e1, r013_0, e0 * r003_0)))));
        const double z012 = fma(e5, r222_0, fma(e4, r212_0, fma(e3, r122_0, fma(e2, r112_0, fma(e1, r022_0, e0 * r012_0)))));
        const double z021 = fma(e5, r231_0, fma(e4, r221_0, fma(e3, r131_0, fma(e2, r121_0, fma(e1, r031_0, e0 * r021_0)))));
        const double z030 = fma(e5, r240_0, fma(e4, r230_0, fma(e3, r140_0, fma(e2, r130_0, fma(e1, r040_0, e0 * r030_0)))));
        const double z102 = fma(e5, r312_0, fma(e4, r302_0, fma(e3, r212_0, fma(e2, r202_0, fma(e1, r112_0, e0 * r102_0)))));
        const double z111 = fma(e5, r321_0, fma(e4, r311_0, fma(e3, r221_0, fma(e2, r211_0, fma(e1, r121_0, e0 * r111_0)))));
        const double z120 = fma(e5, r330_0, fma(e4, r320_0, fma(e3, r230_0, fma(e2, r220_0, fma(e1, r130_0, e0 * r120_0)))));
        const double z201 = fma(e5, r411_0, fma(e4, r401_0, fma(e3, r311_0, fma(e2, r301_0, fma(e1, r211_0, e0 * r201_0)))));
        const double z210 = fma(e5, r420_0, fma(e4, r410_0, fma(e3, r320_0, fma(e2, r310_0, fma(e1, r220_0, e0 * r210_0)))));
        const double z300 = fma(e5, r510_0, fma(e4, r500_0, fma(e3, r410_0, fma(e2, r400_0, fma(e1, r310_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[0], v, Kac[6]);
          Kad[3] = fma(Dbc[0], v, Kad[3]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[1], v, Kac[6]);
          Kad[4] = fma(Dbc[0], v, Kad[4]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[2], v, Kac[6]);
          Kad[5] = fma(Dbc[0], v, Kad[5]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[0], v, Kac[7]);
          Kad[3] = fma(Dbc[1], v, Kad[3]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[1], v, Kac[7]);
          Kad[4] = fma(Dbc[1], v, Kad[4]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[2], v, Kac[7]);
          Kad[5] = fma(Dbc[1], v, Kad[5]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[0], v, Kac[8]);
          Kad[3] = fma(Dbc[2], v, Kad[3]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[1], v, Kac[8]);
          Kad[4] = fma(Dbc[2], v, Kad[4]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[2], v, Kac[8]);
          Kad[5] = fma(Dbc[2], v, Kad[5]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[9] = fma(Dbd[0], v, Kac[9]);
          Kad[3] = fma(Dbc[3], v, Kad[3]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[0] = fma(ac3, v, Kbd[0]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[9] = fma(Dbd[1], v, Kac[9]);
          Kad[4] = fma(Dbc[3], v, Kad[4]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[1] = fma(ac3, v, Kbd[1]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[9] = fma(Dbd[2], v, Kac[9]);
          Kad[5] = fma(Dbc[3], v, Kad[5]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[2] = fma(ac3, v, Kbd[2]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[10] = fma(Dbd[0], v, Kac[10]);
          Kad[3] = fma(Dbc[4], v, Kad[3]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[0] = fma(ac4, v, Kbd[0]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[10] = fma(Dbd[1], v, Kac[10]);
          Kad[4] = fma(Dbc[4], v, Kad[4]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[1] = fma(ac4, v, Kbd[1]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[10] = fma(Dbd[2], v, Kac[10]);
          Kad[5] = fma(Dbc[4], v, Kad[5]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[2] = fma(ac4, v, Kbd[2]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[11] = fma(Dbd[0], v, Kac[11]);
          Kad[3] = fma(Dbc[5], v, Kad[3]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[0] = fma(ac5, v, Kbd[0]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[11] = fma(Dbd[1], v, Kac[11]);
          Kad[4] = fma(Dbc[5], v, Kad[4]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[1] = fma(ac5, v, Kbd[1]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[11] = fma(Dbd[2], v, Kac[11]);
          Kad[5] = fma(Dbc[5], v, Kad[5]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[2] = fma(ac5, v, Kbd[2]);
        }
        Jab[3] += j;
      }
      {
        const double ab = Pab[1 * n + 1] * (kCons[2][1] * kCons[1][1]);
        const double e0 = E[22];
        const double e1 = E[23];
        const double e2 = E[24];
        const double e3 = E[25];
        const double e4 = E[26];
        const double e5 = E[27];
        const double z000 = fma(e5, r120_0, fma(e4, r110_0, fma(e3, r100_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0)))));
        const double z001 = fma(e5, r121_0, fma(e4, r111_0, fma(e3, r101_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0)))));
        const double z010 = fma(e5, r130_0, fma(e4, r120_0, fma(e3, r110_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0)))));
        const double z100 = fma(e5, r220_0, fma(e4, r210_0, fma(e3, r200_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0)))));
        const double z002 = fma(e5, r122_0, fma(e4, r112_0, fma(e3, r102_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0)))));
        const double z011 = fma(e5, r131_0, fma(e4, r121_0, fma(e3, r111_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0)))));
        const double z020 = fma(e5, r140_0, fma(e4, r130_0, fma(e3, r120_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0)))));
        const double z101 = fma(e5, r221_0, fma(e4, r211_0, fma(e3, r201_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0)))));
        const double z110 = fma(e5, r230_0, fma(e4, r220_0, fma(e3, r210_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0)))));
        const double z200 = fma(e5, r320_0, fma(e4, r310_0, fma(e3, r300_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0)))));
        const double z003 = fma(e5, r123_0, fma(e4, r113_0, fma(e3, r103_0, fma(e2, r023_0, fma(e1, r013_0, e0 * r003_0)))));
        const double z012 = fma(e5, r132_0, fma(e4, r122_0, fma(e3, r112_0, fma(e2, r032_0, fma(e1, r022_0, e0 * r012_0)))));
        const double z021 = fma(e5, r141_0, fma(e4, r131_0, fma(e3, r121_0, fma(e2, r041_0, fma(e1, r031_0, e0 * r021_0)))));
        const double z030 = fma(e5, r150_0, fma(e4, r140_0, fma(e3, r130_0, fma(e2, r050_0, fma(e1, r040_0, e0 * r030_0)))));
        const double z102 = fma(e5, r222_0, fma(e4, r212_0, fma(e3, r202_0, fma(e2, r122_0, fma(e1, r112_0, e0 * r102_0)))));
        const double z111 = fma(e5, r231_0, fma(e4, r221_0, fma(e3, r211_0, fma(e2, r131_0, fma(e1, r121_0, e0 * r111_0)))));
        const double z120 = fma(e5, r240_0, fma(e4, r230_0, fma(e3, r220_0, fma(e2, r140_0, fma(e1, r130_0, e0 * r120_0)))));
        const double z201 = fma(e5, r321_0, fma(e4, r311_0, fma(e3, r301_0, fma(e2, r221_0, fma(e1, r211_0, e0 * r201_0)))));
        const double z210 = fma(e5, r330_0, fma(e4, r320_0, fma(e3, r310_0, fma(e2, r230_0, fma(e1, r220_0, e0 * r210_0)))));
        const double z300 = fma(e5, r420_0, fma(e4, r410_0, fma(e3, r400_0, fma(e2, r320_0, fma(e1, r310_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[3], v, Kac[6]);
          Kad[3] = fma(Dbc[6], v, Kad[3]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[4], v, Kac[6]);
          Kad[4] = fma(Dbc[6], v, Kad[4]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[5], v, Kac[6]);
          Kad[5] = fma(Dbc[6], v, Kad[5]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[3], v, Kac[7]);
          Kad[3] = fma(Dbc[7], v, Kad[3]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[4], v, Kac[7]);
          Kad[4] = fma(Dbc[7], v, Kad[4]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[5], v, Kac[7]);
          Kad[5] = fma(Dbc[7], v, Kad[5]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[3], v, Kac[8]);
          Kad[3] = fma(Dbc[8], v, Kad[3]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[4], v, Kac[8]);
          Kad[4] = fma(Dbc[8], v, Kad[4]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[5], v, Kac[8]);
          Kad[5] = fma(Dbc[8], v, Kad[5]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[9] = fma(Dbd[3], v, Kac[9]);
          Kad[3] = fma(Dbc[9], v, Kad[3]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[3] = fma(ac3, v, Kbd[3]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[9] = fma(Dbd[4], v, Kac[9]);
          Kad[4] = fma(Dbc[9], v, Kad[4]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[4] = fma(ac3, v, Kbd[4]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[9] = fma(Dbd[5], v, Kac[9]);
          Kad[5] = fma(Dbc[9], v, Kad[5]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[5] = fma(ac3, v, Kbd[5]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[10] = fma(Dbd[3], v, Kac[10]);
          Kad[3] = fma(Dbc[10], v, Kad[3]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[3] = fma(ac4, v, Kbd[3]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[10] = fma(Dbd[4], v, Kac[10]);
          Kad[4] = fma(Dbc[10], v, Kad[4]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[4] = fma(ac4, v, Kbd[4]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[10] = fma(Dbd[5], v, Kac[10]);
          Kad[5] = fma(Dbc[10], v, Kad[5]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[5] = fma(ac4, v, Kbd[5]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[11] = fma(Dbd[3], v, Kac[11]);
          Kad[3] = fma(Dbc[11], v, Kad[3]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[3] = fma(ac5, v, Kbd[3]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[11] = fma(Dbd[4], v, Kac[11]);
          Kad[4] = fma(Dbc[11], v, Kad[4]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[4] = fma(ac5, v, Kbd[4]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[11] = fma(Dbd[5], v, Kac[11]);
          Kad[5] = fma(Dbc[11], v, Kad[5]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[5] = fma(ac5, v, Kbd[5]);
        }
        Jab[4] += j;
      }
      {
        const double ab = Pab[1 * n + 2] * (kCons[2][1] * kCons[1][2]);
        const double e0 = E[28];
        const double e1 = E[29];
        const double e2 = E[30];
        const double e3 = E[31];
        const double e4 = E[32];
        const double e5 = E[33];
        const double e6 = E[34];
        const double e7 = E[35];
        const double z000 = fma(e7, r111_0, fma(e6, r110_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r112_0, fma(e6, r111_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r121_0, fma(e6, r120_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r211_0, fma(e6, r210_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r113_0, fma(e6, r112_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r122_0, fma(e6, r121_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r212_0, fma(e6, r211_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r221_0, fma(e6, r220_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r311_0, fma(e6, r310_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))));
        const double z003 = fma(e7, r114_0, fma(e6, r113_0, fma(e5, r104_0, fma(e4, r103_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r004_0, e0 * r003_0)))))));
        const double z012 = fma(e7, r123_0, fma(e6, r122_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r013_0, e0 * r012_0)))))));
        const double z021 = fma(e7, r132_0, fma(e6, r131_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r032_0, fma(e2, r031_0, fma(e1, r022_0, e0 * r021_0)))))));
        const double z030 = fma(e7, r141_0, fma(e6, r140_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r041_0, fma(e2, r040_0, fma(e1, r031_0, e0 * r030_0)))))));
        const double z102 = fma(e7, r213_0, fma(e6, r212_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r103_0, e0 * r102_0)))))));
        const double z111 = fma(e7, r222_0, fma(e6, r221_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r122_0, fma(e2, r121_0, fma(e1, r112_0, e0 * r111_0)))))));
        const double z120 = fma(e7, r231_0, fma(e6, r230_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r131_0, fma(e2, r130_0, fma(e1, r121_0, e0 * r120_0)))))));
        const double z201 = fma(e7, r312_0, fma(e6, r311_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r212_0, fma(e2, r211_0, fma(e1, r202_0, e0 * r201_0)))))));
        const double z210 = fma(e7, r321_0, fma(e6, r320_0, fma(e5, r311_0, fma(e4, r310_0, fma(e3, r221_0, fma(e2, r220_0, fma(e1, r211_0, e0 * r210_0)))))));
        const double z300 = fma(e7, r411_0, fma(e6, r410_0, fma(e5, r401_0, fma(e4, r400_0, fma(e3, r311_0, fma(e2, r310_0, fma(e1, r301_0, e0 * r300_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[6] = fma(Dbd[6], v, Kac[6]);
          Kad[3] = fma(Dbc[12], v, Kad[3]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[6] = fma(Dbd[7], v, Kac[6]);
          Kad[4] = fma(Dbc[12], v, Kad[4]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[6] = fma(Dbd[8], v, Kac[6]);
          Kad[5] = fma(Dbc[12], v, Kad[5]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[7] = fma(Dbd[6], v, Kac[7]);
          Kad[3] = fma(Dbc[13], v, Kad[3]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[7] = fma(Dbd[7], v, Kac[7]);
          Kad[4] = fma(Dbc[13], v, Kad[4]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[7] = fma(Dbd[8], v, Kac[7]);
          Kad[5] = fma(Dbc[13], v, Kad[5]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[8] = fma(Dbd[6], v, Kac[8]);
          Kad[3] = fma(Dbc[14], v, Kad[3]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[8] = fma(Dbd[7], v, Kac[8]);
          Kad[4] = fma(Dbc[14], v, Kad[4]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[8] = fma(Dbd[8], v, Kac[8]);
          Kad[5] = fma(Dbc[14], v, Kad[5]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[9] = fma(Dbd[6], v, Kac[9]);
          Kad[3] = fma(Dbc[15], v, Kad[3]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[6] = fma(ac3, v, Kbd[6]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[9] = fma(Dbd[7], v, Kac[9]);
          Kad[4] = fma(Dbc[15], v, Kad[4]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[7] = fma(ac3, v, Kbd[7]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[9] = fma(Dbd[8], v, Kac[9]);
          Kad[5] = fma(Dbc[15], v, Kad[5]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[8] = fma(ac3, v, Kbd[8]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[10] = fma(Dbd[6], v, Kac[10]);
          Kad[3] = fma(Dbc[16], v, Kad[3]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[6] = fma(ac4, v, Kbd[6]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[10] = fma(Dbd[7], v, Kac[10]);
          Kad[4] = fma(Dbc[16], v, Kad[4]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[7] = fma(ac4, v, Kbd[7]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[10] = fma(Dbd[8], v, Kac[10]);
          Kad[5] = fma(Dbc[16], v, Kad[5]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[8] = fma(ac4, v, Kbd[8]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[11] = fma(Dbd[6], v, Kac[11]);
          Kad[3] = fma(Dbc[17], v, Kad[3]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[6] = fma(ac5, v, Kbd[6]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[11] = fma(Dbd[7], v, Kac[11]);
          Kad[4] = fma(Dbc[17], v, Kad[4]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[7] = fma(ac5, v, Kbd[7]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[11] = fma(Dbd[8], v, Kac[11]);
          Kad[5] = fma(Dbc[17], v, Kad[5]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[8] = fma(ac5, v, Kbd[8]);
        }
        Jab[5] += j;
      }
    }
    {
      const double ac0 = P[oc + 2 * n + 0] * kCons[2][2];
      const double ac1 = P[oc + 2 * n + 1] * kCons[2][2];
      const double ac2 = P[oc + 2 * n + 2] * kCons[2][2];
      const double ac3 = P[oc + 2 * n + 3] * kCons[2][2];
      const double ac4 = P[oc + 2 * n + 4] * kCons[2][2];
      const double ac5 = P[oc + 2 * n + 5] * kCons[2][2];
      const double ad0 = P[od + 2 * n + 0] * kCons[2][2];
      const double ad1 = P[od + 2 * n + 1] * kCons[2][2];
      const double ad2 = P[od + 2 * n + 2] * kCons[2][2];
      {
        const double ab = Pab[2 * n + 0] * (kCons[2][2] * kCons[1][0]);
        const double e0 = E[36];
        const double e1 = E[37];
        const double e2 = E[38];
        const double e3 = E[39];
        const double e4 = E[40];
        const double e5 = E[41];
        const double z000 = fma(e5, r120_0, fma(e4, r110_0, fma(e3, r100_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0)))));
        const double z001 = fma(e5, r121_0, fma(e4, r111_0, fma(e3, r101_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0)))));
        const double z010 = fma(e5, r130_0, fma(e4, r120_0, fma(e3, r110_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0)))));
        const double z100 = fma(e5, r220_0, fma(e4, r210_0, fma(e3, r200_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0)))));
        const double z002 = fma(e5, r122_0, fma(e4, r112_0, fma(e3, r102_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0)))));
        const double z011 = fma(e5, r131_0, fma(e4, r121_0, fma(e3, r111_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0)))));
        const double z020 = fma(e5, r140_0, fma(e4, r130_0, fma(e3, r120_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0)))));
        const double z101 = fma(e5, r221_0, fma(e4, r211_0, fma(e3, r201_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0)))));
        const double z110 = fma(e5, r230_0, fma(e4, r220_0, fma(e3, r210_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0)))));
        const double z200 = fma(e5, r320_0, fma(e4, r310_0, fma(e3, r300_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0)))));
        const double z003 = fma(e5, r123_0, fma(e4, r113_0, fma(e3, r103_0, fma(e2, r023_0, fma(e1, r013_0, e0 * r003_0)))));
        const double z012 = fma(e5, r132_0, fma(e4, r122_0, fma(e3, r112_0, fma(e2, r032_0, fma(e1, r022_0, e0 * r012_0)))));
        const double z021 = fma(e5, r141_0, fma(e4, r131_0, fma(e3, r121_0, fma(e2, r041_0, fma(e1, r031_0, e0 * r021_0)))));
        const double z030 = fma(e5, r150_0, fma(e4, r140_0, fma(e3, r130_0, fma(e2, r050_0, fma(e1, r040_0, e0 * r030_0)))));
        const double z102 = fma(e5, r222_0, fma(e4, r212_0, fma(e3, r202_0, fma(e2, r122_0, fma(e1, r112_0, e0 * r102_0)))));
        const double z111 = fma(e5, r231_0, fma(e4, r221_0, fma(e3, r211_0, fma(e2, r131_0, fma(e1, r121_0, e0 * r111_0)))));
        const double z120 = fma(e5, r240_0, fma(e4, r230_0, fma(e3, r220_0, fma(e2, r140_0, fma(e1, r130_0, e0 * r120_0)))));
        const double z201 = fma(e5, r321_0, fma(e4, r311_0, fma(e3, r301_0, fma(e2, r221_0, fma(e1, r211_0, e0 * r201_0)))));
        const double z210 = fma(e5, r330_0, fma(e4, r320_0, fma(e3, r310_0, fma(e2, r230_0, fma(e1, r220_0, e0 * r210_0)))));
        const double z300 = fma(e5, r420_0, fma(e4, r410_0, fma(e3, r400_0, fma(e2, r320_0, fma(e1, r310_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[0], v, Kac[12]);
          Kad[6] = fma(Dbc[0], v, Kad[6]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[1], v, Kac[12]);
          Kad[7] = fma(Dbc[0], v, Kad[7]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[2], v, Kac[12]);
          Kad[8] = fma(Dbc[0], v, Kad[8]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[0], v, Kac[13]);
          Kad[6] = fma(Dbc[1], v, Kad[6]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[1], v, Kac[13]);
          Kad[7] = fma(Dbc[1], v, Kad[7]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[2], v, Kac[13]);
          Kad[8] = fma(Dbc[1], v, Kad[8]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[0], v, Kac[14]);
          Kad[6] = fma(Dbc[2], v, Kad[6]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[1], v, Kac[14]);
          Kad[7] = fma(Dbc[2], v, Kad[7]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[2], v, Kac[14]);
          Kad[8] = fma(Dbc[2], v, Kad[8]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[15] = fma(Dbd[0], v, Kac[15]);
          Kad[6] = fma(Dbc[3], v, Kad[6]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[0] = fma(ac3, v, Kbd[0]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[15] = fma(Dbd[1], v, Kac[15]);
          Kad[7] = fma(Dbc[3], v, Kad[7]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[1] = fma(ac3, v, Kbd[1]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[15] = fma(Dbd[2], v, Kac[15]);
          Kad[8] = fma(Dbc[3], v, Kad[8]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[2] = fma(ac3, v, Kbd[2]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[16] = fma(Dbd[0], v, Kac[16]);
          Kad[6] = fma(Dbc[4], v, Kad[6]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[0] = fma(ac4, v, Kbd[0]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[16] = fma(Dbd[1], v, Kac[16]);
          Kad[7] = fma(Dbc[4], v, Kad[7]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[1] = fma(ac4, v, Kbd[1]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[16] = fma(Dbd[2], v, Kac[16]);
          Kad[8] = fma(Dbc[4], v, Kad[8]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[2] = fma(ac4, v, Kbd[2]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[17] = fma(Dbd[0], v, Kac[17]);
          Kad[6] = fma(Dbc[5], v, Kad[6]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[0] = fma(ac5, v, Kbd[0]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[17] = fma(Dbd[1], v, Kac[17]);
          Kad[7] = fma(Dbc[5], v, Kad[7]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[1] = fma(ac5, v, Kbd[1]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[17] = fma(Dbd[2], v, Kac[17]);
          Kad[8] = fma(Dbc[5], v, Kad[8]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[2] = fma(ac5, v, Kbd[2]);
        }
        Jab[6] += j;
      }
      {
        const double ab = Pab[2 * n + 1] * (kCons[2][2] * kCons[1][1]);
        const double e0 = E[42];
        const double e1 = E[43];
        const double e2 = E[44];
        const double e3 = E[45];
        const double z000 = fma(e3, r030_0, fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0)));
        const double z001 = fma(e3, r031_0, fma(e2, r021_0, fma(e1, r011_0, e0 * r001_0)));
        const double z010 = fma(e3, r040_0, fma(e2, r030_0, fma(e1, r020_0, e0 * r010_0)));
        const double z100 = fma(e3, r130_0, fma(e2, r120_0, fma(e1, r110_0, e0 * r100_0)));
        const double z002 = fma(e3, r032_0, fma(e2, r022_0, fma(e1, r012_0, e0 * r002_0)));
        const double z011 = fma(e3, r041_0, fma(e2, r031_0, fma(e1, r021_0, e0 * r011_0)));
        const double z020 = fma(e3, r050_0, fma(e2, r040_0, fma(e1, r030_0, e0 * r020_0)));
        const double z101 = fma(e3, r131_0, fma(e2, r121_0, fma(e1, r111_0, e0 * r101_0)));
        const double z110 = fma(e3, r140_0, fma(e2, r130_0, fma(e1, r120_0, e0 * r110_0)));
        const double z200 = fma(e3, r230_0, fma(e2, r220_0, fma(e1, r210_0, e0 * r200_0)));
        const double z003 = fma(e3, r033_0, fma(e2, r023_0, fma(e1, r013_0, e0 * r003_0)));
        const double z012 = fma(e3, r042_0, fma(e2, r032_0, fma(e1, r022_0, e0 * r012_0)));
        const double z021 = fma(e3, r051_0, fma(e2, r041_0, fma(e1, r031_0, e0 * r021_0)));
        const double z030 = fma(e3, r060_0, fma(e2, r050_0, fma(e1, r040_0, e0 * r030_0)));
        const double z102 = fma(e3, r132_0, fma(e2, r122_0, fma(e1, r112_0, e0 * r102_0)));
        const double z111 = fma(e3, r141_0, fma(e2, r131_0, fma(e1, r121_0, e0 * r111_0)));
        const double z120 = fma(e3, r150_0, fma(e2, r140_0, fma(e1, r130_0, e0 * r120_0)));
        const double z201 = fma(e3, r231_0, fma(e2, r221_0, fma(e1, r211_0, e0 * r201_0)));
        const double z210 = fma(e3, r240_0, fma(e2, r230_0, fma(e1, r220_0, e0 * r210_0)));
        const double z300 = fma(e3, r330_0, fma(e2, r320_0, fma(e1, r310_0, e0 * r300_0)));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[3], v, Kac[12]);
          Kad[6] = fma(Dbc[6], v, Kad[6]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[4], v, Kac[12]);
          Kad[7] = fma(Dbc[6], v, Kad[7]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[5], v, Kac[12]);
          Kad[8] = fma(Dbc[6], v, Kad[8]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[3], v, Kac[13]);
          Kad[6] = fma(Dbc[7], v, Kad[6]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[4], v, Kac[13]);
          Kad[7] = fma(Dbc[7], v, Kad[7]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[5], v, Kac[13]);
          Kad[8] = fma(Dbc[7], v, Kad[8]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[3], v, Kac[14]);
          Kad[6] = fma(Dbc[8], v, Kad[6]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[4], v, Kac[14]);
          Kad[7] = fma(Dbc[8], v, Kad[7]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[5], v, Kac[14]);
          Kad[8] = fma(Dbc[8], v, Kad[8]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[15] = fma(Dbd[3], v, Kac[15]);
          Kad[6] = fma(Dbc[9], v, Kad[6]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[3] = fma(ac3, v, Kbd[3]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[15] = fma(Dbd[4], v, Kac[15]);
          Kad[7] = fma(Dbc[9], v, Kad[7]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[4] = fma(ac3, v, Kbd[4]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[15] = fma(Dbd[5], v, Kac[15]);
          Kad[8] = fma(Dbc[9], v, Kad[8]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[5] = fma(ac3, v, Kbd[5]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[16] = fma(Dbd[3], v, Kac[16]);
          Kad[6] = fma(Dbc[10], v, Kad[6]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[3] = fma(ac4, v, Kbd[3]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[16] = fma(Dbd[4], v, Kac[16]);
          Kad[7] = fma(Dbc[10], v, Kad[7]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[4] = fma(ac4, v, Kbd[4]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[16] = fma(Dbd[5], v, Kac[16]);
          Kad[8] = fma(Dbc[10], v, Kad[8]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[5] = fma(ac4, v, Kbd[5]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[17] = fma(Dbd[3], v, Kac[17]);
          Kad[6] = fma(Dbc[11], v, Kad[6]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[3] = fma(ac5, v, Kbd[3]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[17] = fma(Dbd[4], v, Kac[17]);
          Kad[7] = fma(Dbc[11], v, Kad[7]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[4] = fma(ac5, v, Kbd[4]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[17] = fma(Dbd[5], v, Kac[17]);
          Kad[8] = fma(Dbc[11], v, Kad[8]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[5] = fma(ac5, v, Kbd[5]);
        }
        Jab[7] += j;
      }
      {
        const double ab = Pab[2 * n + 2] * (kCons[2][2] * kCons[1][2]);
        const double e0 = E[46];
        const double e1 = E[47];
        const double e2 = E[48];
        const double e3 = E[49];
        const double e4 = E[50];
        const double e5 = E[51];
        const double z000 = fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r024_0, fma(e4, r023_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r033_0, fma(e4, r032_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r042_0, fma(e4, r041_0, fma(e3, r032_0, fma(e2, r031_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r051_0, fma(e4, r050_0, fma(e3, r041_0, fma(e2, r040_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r123_0, fma(e4, r122_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r132_0, fma(e4, r131_0, fma(e3, r122_0, fma(e2, r121_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r141_0, fma(e4, r140_0, fma(e3, r131_0, fma(e2, r130_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r212_0, fma(e2, r211_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r231_0, fma(e4, r230_0, fma(e3, r221_0, fma(e2, r220_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r321_0, fma(e4, r320_0, fma(e3, r311_0, fma(e2, r310_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[12] = fma(Dbd[6], v, Kac[12]);
          Kad[6] = fma(Dbc[12], v, Kad[6]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[12] = fma(Dbd[7], v, Kac[12]);
          Kad[7] = fma(Dbc[12], v, Kad[7]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[12] = fma(Dbd[8], v, Kac[12]);
          Kad[8] = fma(Dbc[12], v, Kad[8]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[13] = fma(Dbd[6], v, Kac[13]);
          Kad[6] = fma(Dbc[13], v, Kad[6]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[13] = fma(Dbd[7], v, Kac[13]);
          Kad[7] = fma(Dbc[13], v, Kad[7]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[13] = fma(Dbd[8], v, Kac[13]);
          Kad[8] = fma(Dbc[13], v, Kad[8]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[14] = fma(Dbd[6], v, Kac[14]);
          Kad[6] = fma(Dbc[14], v, Kad[6]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[14] = fma(Dbd[7], v, Kac[14]);
          Kad[7] = fma(Dbc[14], v, Kad[7]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[14] = fma(Dbd[8], v, Kac[14]);
          Kad[8] = fma(Dbc[14], v, Kad[8]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[15] = fma(Dbd[6], v, Kac[15]);
          Kad[6] = fma(Dbc[15], v, Kad[6]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[6] = fma(ac3, v, Kbd[6]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[15] = fma(Dbd[7], v, Kac[15]);
          Kad[7] = fma(Dbc[15], v, Kad[7]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[7] = fma(ac3, v, Kbd[7]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[15] = fma(Dbd[8], v, Kac[15]);
          Kad[8] = fma(Dbc[15], v, Kad[8]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[8] = fma(ac3, v, Kbd[8]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[16] = fma(Dbd[6], v, Kac[16]);
          Kad[6] = fma(Dbc[16], v, Kad[6]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[6] = fma(ac4, v, Kbd[6]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[16] = fma(Dbd[7], v, Kac[16]);
          Kad[7] = fma(Dbc[16], v, Kad[7]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[7] = fma(ac4, v, Kbd[7]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[16] = fma(Dbd[8], v, Kac[16]);
          Kad[8] = fma(Dbc[16], v, Kad[8]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[8] = fma(ac4, v, Kbd[8]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[17] = fma(Dbd[6], v, Kac[17]);
          Kad[6] = fma(Dbc[17], v, Kad[6]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[6] = fma(ac5, v, Kbd[6]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[17] = fma(Dbd[7], v, Kac[17]);
          Kad[7] = fma(Dbc[17], v, Kad[7]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[7] = fma(ac5, v, Kbd[7]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[17] = fma(Dbd[8], v, Kac[17]);
          Kad[8] = fma(Dbc[17], v, Kad[8]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[8] = fma(ac5, v, Kbd[8]);
        }
        Jab[8] += j;
      }
    }
    {
      const double ac0 = P[oc + 3 * n + 0] * kCons[2][3];
      const double ac1 = P[oc + 3 * n + 1] * kCons[2][3];
      const double ac2 = P[oc + 3 * n + 2] * kCons[2][3];
      const double ac3 = P[oc + 3 * n + 3] * kCons[2][3];
      const double ac4 = P[oc + 3 * n + 4] * kCons[2][3];
      const double ac5 = P[oc + 3 * n + 5] * kCons[2][3];
      const double ad0 = P[od + 3 * n + 0] * kCons[2][3];
      const double ad1 = P[od + 3 * n + 1] * kCons[2][3];
      const double ad2 = P[od + 3 * n + 2] * kCons[2][3];
      {
        const double ab = Pab[3 * n + 0] * (kCons[2][3] * kCons[1][0]);
        const double e0 = E[52];
        const double e1 = E[53];
        const double e2 = E[54];
        const double e3 = E[55];
        const double e4 = E[56];
        const double e5 = E[57];
        const double z000 = fma(e5, r201_0, fma(e4, r200_0, fma(e3, r101_0, fma(e2, r100_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r202_0, fma(e4, r201_0, fma(e3, r102_0, fma(e2, r101_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r211_0, fma(e4, r210_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r301_0, fma(e4, r300_0, fma(e3, r201_0, fma(e2, r200_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r203_0, fma(e4, r202_0, fma(e3, r103_0, fma(e2, r102_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r212_0, fma(e4, r211_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r221_0, fma(e4, r220_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r302_0, fma(e4, r301_0, fma(e3, r202_0, fma(e2, r201_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r311_0, fma(e4, r310_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r401_0, fma(e4, r400_0, fma(e3, r301_0, fma(e2, r300_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r204_0, fma(e4, r203_0, fma(e3, r104_0, fma(e2, r103_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r213_0, fma(e4, r212_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r122_0, fma(e2, r121_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r231_0, fma(e4, r230_0, fma(e3, r131_0, fma(e2, r130_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r303_0, fma(e4, r302_0, fma(e3, r203_0, fma(e2, r202_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r312_0, fma(e4, r311_0, fma(e3, r212_0, fma(e2, r211_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r321_0, fma(e4, r320_0, fma(e3, r221_0, fma(e2, r220_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r402_0, fma(e4, r401_0, fma(e3, r302_0, fma(e2, r301_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r411_0, fma(e4, r410_0, fma(e3, r311_0, fma(e2, r310_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r501_0, fma(e4, r500_0, fma(e3, r401_0, fma(e2, r400_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[18] = fma(Dbd[0], v, Kac[18]);
          Kad[9] = fma(Dbc[0], v, Kad[9]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[18] = fma(Dbd[1], v, Kac[18]);
          Kad[10] = fma(Dbc[0], v, Kad[10]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[18] = fma(Dbd[2], v, Kac[18]);
          Kad[11] = fma(Dbc[0], v, Kad[11]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[19] = fma(Dbd[0], v, Kac[19]);
          Kad[9] = fma(Dbc[1], v, Kad[9]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[19] = fma(Dbd[1], v, Kac[19]);
          Kad[10] = fma(Dbc[1], v, Kad[10]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[19] = fma(Dbd[2], v, Kac[19]);
          Kad[11] = fma(Dbc[1], v, Kad[11]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[20] = fma(Dbd[0], v, Kac[20]);
          Kad[9] = fma(Dbc[2], v, Kad[9]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[20] = fma(Dbd[1], v, Kac[20]);
          Kad[10] = fma(Dbc[2], v, Kad[10]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[20] = fma(Dbd[2], v, Kac[20]);
          Kad[11] = fma(Dbc[2], v, Kad[11]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[21] = fma(Dbd[0], v, Kac[21]);
          Kad[9] = fma(Dbc[3], v, Kad[9]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[0] = fma(ac3, v, Kbd[0]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[21] = fma(Dbd[1], v, Kac[21]);
          Kad[10] = fma(Dbc[3], v, Kad[10]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[1] = fma(ac3, v, Kbd[1]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[21] = fma(Dbd[2], v, Kac[21]);
          Kad[11] = fma(Dbc[3], v, Kad[11]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[2] = fma(ac3, v, Kbd[2]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[22] = fma(Dbd[0], v, Kac[22]);
          Kad[9] = fma(Dbc[4], v, Kad[9]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[0] = fma(ac4, v, Kbd[0]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[22] = fma(Dbd[1], v, Kac[22]);
          Kad[10] = fma(Dbc[4], v, Kad[10]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[1] = fma(ac4, v, Kbd[1]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[22] = fma(Dbd[2], v, Kac[22]);
          Kad[11] = fma(Dbc[4], v, Kad[11]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[2] = fma(ac4, v, Kbd[2]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[23] = fma(Dbd[0], v, Kac[23]);
          Kad[9] = fma(Dbc[5], v, Kad[9]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[0] = fma(ac5, v, Kbd[0]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[23] = fma(Dbd[1], v, Kac[23]);
          Kad[10] = fma(Dbc[5], v, Kad[10]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[1] = fma(ac5, v, Kbd[1]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[23] = fma(Dbd[2], v, Kac[23]);
          Kad[11] = fma(Dbc[5], v, Kad[11]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[2] = fma(ac5, v, Kbd[2]);
        }
        Jab[9] += j;
      }
      {
        const double ab = Pab[3 * n + 1] * (kCons[2][3] * kCons[1][1]);
        const double e0 = E[58];
        const double e1 = E[59];
        const double e2 = E[60];
        const double e3 = E[61];
        const double e4 = E[62];
        const double e5 = E[63];
        const double e6 = E[64];
        const double e7 = E[65];
        const double z000 = fma(e7, r111_0, fma(e6, r110_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r112_0, fma(e6, r111_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r121_0, fma(e6, r120_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r211_0, fma(e6, r210_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r113_0, fma(e6, r112_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r122_0, fma(e6, r121_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r212_0, fma(e6, r211_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r221_0, fma(e6, r220_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r311_0, fma(e6, r310_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))));
        const double z003 = fma(e7, r114_0, fma(e6, r113_0, fma(e5, r104_0, fma(e4, r103_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r004_0, e0 * r003_0)))))));
        const double z012 = fma(e7, r123_0, fma(e6, r122_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r013_0, e0 * r012_0)))))));
        const double z021 = fma(e7, r132_0, fma(e6, r131_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r032_0, fma(e2, r031_0, fma(e1, r022_0, e0 * r021_0)))))));
        const double z030 = fma(e7, r141_0, fma(e6, r140_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r041_0, fma(e2, r040_0, fma(e1, r031_0, e0 * r030_0)))))));
        const double z102 = fma(e7, r213_0, fma(e6, r212_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r103_0, e0 * r102_0)))))));
        const double z111 = fma(e7, r222_0, fma(e6, r221_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r122_0, fma(e2, r121_0, fma(e1, r112_0, e0 * r111_0)))))));
        const double z120 = fma(e7, r231_0, fma(e6, r230_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r131_0, fma(e2, r130_0, fma(e1, r121_0, e0 * r120_0)))))));
        const double z201 = fma(e7, r312_0, fma(e6, r311_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r212_0, fma(e2, r211_0, fma(e1, r202_0, e0 * r201_0)))))));
        const double z210 = fma(e7, r321_0, fma(e6, r320_0, fma(e5, r311_0, fma(e4, r310_0, fma(e3, r221_0, fma(e2, r220_0, fma(e1, r211_0, e0 * r210_0)))))));
        const double z300 = fma(e7, r411_0, fma(e6, r410_0, fma(e5, r401_0, fma(e4, r400_0, fma(e3, r311_0, fma(e2, r310_0, fma(e1, r301_0, e0 * r300_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[18] = fma(Dbd[3], v, Kac[18]);
          Kad[9] = fma(Dbc[6], v, Kad[9]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[18] = fma(Dbd[4], v, Kac[18]);
          Kad[10] = fma(Dbc[6], v, Kad[10]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[18] = fma(Dbd[5], v, Kac[18]);
          Kad[11] = fma(Dbc[6], v, Kad[11]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[19] = fma(Dbd[3], v, Kac[19]);
          Kad[9] = fma(Dbc[7], v, Kad[9]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[19] = fma(Dbd[4], v, Kac[19]);
          Kad[10] = fma(Dbc[7], v, Kad[10]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[19] = fma(Dbd[5], v, Kac[19]);
          Kad[11] = fma(Dbc[7], v, Kad[11]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[20] = fma(Dbd[3], v, Kac[20]);
          Kad[9] = fma(Dbc[8], v, Kad[9]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[20] = fma(Dbd[4], v, Kac[20]);
          Kad[10] = fma(Dbc[8], v, Kad[10]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[20] = fma(Dbd[5], v, Kac[20]);
          Kad[11] = fma(Dbc[8], v, Kad[11]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[21] = fma(Dbd[3], v, Kac[21]);
          Kad[9] = fma(Dbc[9], v, Kad[9]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[3] = fma(ac3, v, Kbd[3]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[21] = fma(Dbd[4], v, Kac[21]);
          Kad[10] = fma(Dbc[9], v, Kad[10]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[4] = fma(ac3, v, Kbd[4]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[21] = fma(Dbd[5], v, Kac[21]);
          Kad[11] = fma(Dbc[9], v, Kad[11]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[5] = fma(ac3, v, Kbd[5]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[22] = fma(Dbd[3], v, Kac[22]);
          Kad[9] = fma(Dbc[10], v, Kad[9]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[3] = fma(ac4, v, Kbd[3]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[22] = fma(Dbd[4], v, Kac[22]);
          Kad[10] = fma(Dbc[10], v, Kad[10]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[4] = fma(ac4, v, Kbd[4]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[22] = fma(Dbd[5], v, Kac[22]);
          Kad[11] = fma(Dbc[10], v, Kad[11]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[5] = fma(ac4, v, Kbd[5]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[23] = fma(Dbd[3], v, Kac[23]);
          Kad[9] = fma(Dbc[11], v, Kad[9]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[3] = fma(ac5, v, Kbd[3]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[23] = fma(Dbd[4], v, Kac[23]);
          Kad[10] = fma(Dbc[11], v, Kad[10]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[4] = fma(ac5, v, Kbd[4]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[23] = fma(Dbd[5], v, Kac[23]);
          Kad[11] = fma(Dbc[11], v, Kad[11]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[5] = fma(ac5, v, Kbd[5]);
        }
        Jab[10] += j;
      }
      {
        const double ab = Pab[3 * n + 2] * (kCons[2][3] * kCons[1][2]);
        const double e0 = E[66];
        const double e1 = E[67];
        const double e2 = E[68];
        const double e3 = E[69];
        const double e4 = E[70];
        const double e5 = E[71];
        const double z000 = fma(e5, r102_0, fma(e4, r101_0, fma(e3, r100_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r103_0, fma(e4, r102_0, fma(e3, r101_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r202_0, fma(e4, r201_0, fma(e3, r200_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r104_0, fma(e4, r103_0, fma(e3, r102_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r203_0, fma(e4, r202_0, fma(e3, r201_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r302_0, fma(e4, r301_0, fma(e3, r300_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r105_0, fma(e4, r104_0, fma(e3, r103_0, fma(e2, r005_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r114_0, fma(e4, r113_0, fma(e3, r112_0, fma(e2, r014_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r123_0, fma(e4, r122_0, fma(e3, r121_0, fma(e2, r023_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r132_0, fma(e4, r131_0, fma(e3, r130_0, fma(e2, r032_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r204_0, fma(e4, r203_0, fma(e3, r202_0, fma(e2, r104_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r213_0, fma(e4, r212_0, fma(e3, r211_0, fma(e2, r113_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r220_0, fma(e2, r122_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r303_0, fma(e4, r302_0, fma(e3, r301_0, fma(e2, r203_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r312_0, fma(e4, r311_0, fma(e3, r310_0, fma(e2, r212_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r402_0, fma(e4, r401_0, fma(e3, r400_0, fma(e2, r302_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[18] = fma(Dbd[6], v, Kac[18]);
          Kad[9] = fma(Dbc[12], v, Kad[9]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[18] = fma(Dbd[7], v, Kac[18]);
          Kad[10] = fma(Dbc[12], v, Kad[10]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[18] = fma(Dbd[8], v, Kac[18]);
          Kad[11] = fma(Dbc[12], v, Kad[11]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[19] = fma(Dbd[6], v, Kac[19]);
          Kad[9] = fma(Dbc[13], v, Kad[9]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[19] = fma(Dbd[7], v, Kac[19]);
          Kad[10] = fma(Dbc[13], v, Kad[10]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[19] = fma(Dbd[8], v, Kac[19]);
          Kad[11] = fma(Dbc[13], v, Kad[11]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[20] = fma(Dbd[6], v, Kac[20]);
          Kad[9] = fma(Dbc[14], v, Kad[9]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[20] = fma(Dbd[7], v, Kac[20]);
          Kad[10] = fma(Dbc[14], v, Kad[10]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[20] = fma(Dbd[8], v, Kac[20]);
          Kad[11] = fma(Dbc[14], v, Kad[11]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[21] = fma(Dbd[6], v, Kac[21]);
          Kad[9] = fma(Dbc[15], v, Kad[9]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[6] = fma(ac3, v, Kbd[6]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[21] = fma(Dbd[7], v, Kac[21]);
          Kad[10] = fma(Dbc[15], v, Kad[10]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[7] = fma(ac3, v, Kbd[7]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[21] = fma(Dbd[8], v, Kac[21]);
          Kad[11] = fma(Dbc[15], v, Kad[11]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[8] = fma(ac3, v, Kbd[8]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[22] = fma(Dbd[6], v, Kac[22]);
          Kad[9] = fma(Dbc[16], v, Kad[9]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[6] = fma(ac4, v, Kbd[6]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[22] = fma(Dbd[7], v, Kac[22]);
          Kad[10] = fma(Dbc[16], v, Kad[10]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[7] = fma(ac4, v, Kbd[7]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[22] = fma(Dbd[8], v, Kac[22]);
          Kad[11] = fma(Dbc[16], v, Kad[11]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[8] = fma(ac4, v, Kbd[8]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[23] = fma(Dbd[6], v, Kac[23]);
          Kad[9] = fma(Dbc[17], v, Kad[9]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[6] = fma(ac5, v, Kbd[6]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[23] = fma(Dbd[7], v, Kac[23]);
          Kad[10] = fma(Dbc[17], v, Kad[10]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[7] = fma(ac5, v, Kbd[7]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[23] = fma(Dbd[8], v, Kac[23]);
          Kad[11] = fma(Dbc[17], v, Kad[11]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[8] = fma(ac5, v, Kbd[8]);
        }
        Jab[11] += j;
      }
    }
    {
      const double ac0 = P[oc + 4 * n + 0] * kCons[2][4];
      const double ac1 = P[oc + 4 * n + 1] * kCons[2][4];
      const double ac2 = P[oc + 4 * n + 2] * kCons[2][4];
      const double ac3 = P[oc + 4 * n + 3] * kCons[2][4];
      const double ac4 = P[oc + 4 * n + 4] * kCons[2][4];
      const double ac5 = P[oc + 4 * n + 5] * kCons[2][4];
      const double ad0 = P[od + 4 * n + 0] * kCons[2][4];
      const double ad1 = P[od + 4 * n + 1] * kCons[2][4];
      const double ad2 = P[od + 4 * n + 2] * kCons[2][4];
      {
        const double ab = Pab[4 * n + 0] * (kCons[2][4] * kCons[1][0]);
        const double e0 = E[72];
        const double e1 = E[73];
        const double e2 = E[74];
        const double e3 = E[75];
        const double e4 = E[76];
        const double e5 = E[77];
        const double e6 = E[78];
        const double e7 = E[79];
        const double z000 = fma(e7, r111_0, fma(e6, r110_0, fma(e5, r101_0, fma(e4, r100_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))))));
        const double z001 = fma(e7, r112_0, fma(e6, r111_0, fma(e5, r102_0, fma(e4, r101_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))))));
        const double z010 = fma(e7, r121_0, fma(e6, r120_0, fma(e5, r111_0, fma(e4, r110_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))))));
        const double z100 = fma(e7, r211_0, fma(e6, r210_0, fma(e5, r201_0, fma(e4, r200_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))))));
        const double z002 = fma(e7, r113_0, fma(e6, r112_0, fma(e5, r103_0, fma(e4, r102_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))))));
        const double z011 = fma(e7, r122_0, fma(e6, r121_0, fma(e5, r112_0, fma(e4, r111_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))))));
        const double z020 = fma(e7, r131_0, fma(e6, r130_0, fma(e5, r121_0, fma(e4, r120_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))))));
        const double z101 = fma(e7, r212_0, fma(e6, r211_0, fma(e5, r202_0, fma(e4, r201_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))))));
        const double z110 = fma(e7, r221_0, fma(e6, r220_0, fma(e5, r211_0, fma(e4, r210_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))))));
        const double z200 = fma(e7, r311_0, fma(e6, r310_0, fma(e5, r301_0, fma(e4, r300_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))))));
        const double z003 = fma(e7, r114_0, fma(e6, r113_0, fma(e5, r104_0, fma(e4, r103_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r004_0, e0 * r003_0)))))));
        const double z012 = fma(e7, r123_0, fma(e6, r122_0, fma(e5, r113_0, fma(e4, r112_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r013_0, e0 * r012_0)))))));
        const double z021 = fma(e7, r132_0, fma(e6, r131_0, fma(e5, r122_0, fma(e4, r121_0, fma(e3, r032_0, fma(e2, r031_0, fma(e1, r022_0, e0 * r021_0)))))));
        const double z030 = fma(e7, r141_0, fma(e6, r140_0, fma(e5, r131_0, fma(e4, r130_0, fma(e3, r041_0, fma(e2, r040_0, fma(e1, r031_0, e0 * r030_0)))))));
        const double z102 = fma(e7, r213_0, fma(e6, r212_0, fma(e5, r203_0, fma(e4, r202_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r103_0, e0 * r102_0)))))));
        const double z111 = fma(e7, r222_0, fma(e6, r221_0, fma(e5, r212_0, fma(e4, r211_0, fma(e3, r122_0, fma(e2, r121_0, fma(e1, r112_0, e0 * r111_0)))))));
        const double z120 = fma(e7, r231_0, fma(e6, r230_0, fma(e5, r221_0, fma(e4, r220_0, fma(e3, r131_0, fma(e2, r130_0, fma(e1, r121_0, e0 * r120_0)))))));
        const double z201 = fma(e7, r312_0, fma(e6, r311_0, fma(e5, r302_0, fma(e4, r301_0, fma(e3, r212_0, fma(e2, r211_0, fma(e1, r202_0, e0 * r201_0)))))));
        const double z210 = fma(e7, r321_0, fma(e6, r320_0, fma(e5, r311_0, fma(e4, r310_0, fma(e3, r221_0, fma(e2, r220_0, fma(e1, r211_0, e0 * r210_0)))))));
        const double z300 = fma(e7, r411_0, fma(e6, r410_0, fma(e5, r401_0, fma(e4, r400_0, fma(e3, r311_0, fma(e2, r310_0, fma(e1, r301_0, e0 * r300_0)))))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[24] = fma(Dbd[0], v, Kac[24]);
          Kad[12] = fma(Dbc[0], v, Kad[12]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[24] = fma(Dbd[1], v, Kac[24]);
          Kad[13] = fma(Dbc[0], v, Kad[13]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[24] = fma(Dbd[2], v, Kac[24]);
          Kad[14] = fma(Dbc[0], v, Kad[14]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[25] = fma(Dbd[0], v, Kac[25]);
          Kad[12] = fma(Dbc[1], v, Kad[12]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[25] = fma(Dbd[1], v, Kac[25]);
          Kad[13] = fma(Dbc[1], v, Kad[13]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[25] = fma(Dbd[2], v, Kac[25]);
          Kad[14] = fma(Dbc[1], v, Kad[14]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[26] = fma(Dbd[0], v, Kac[26]);
          Kad[12] = fma(Dbc[2], v, Kad[12]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[26] = fma(Dbd[1], v, Kac[26]);
          Kad[13] = fma(Dbc[2], v, Kad[13]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[26] = fma(Dbd[2], v, Kac[26]);
          Kad[14] = fma(Dbc[2], v, Kad[14]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[27] = fma(Dbd[0], v, Kac[27]);
          Kad[12] = fma(Dbc[3], v, Kad[12]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[0] = fma(ac3, v, Kbd[0]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[27] = fma(Dbd[1], v, Kac[27]);
          Kad[13] = fma(Dbc[3], v, Kad[13]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[1] = fma(ac3, v, Kbd[1]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[27] = fma(Dbd[2], v, Kac[27]);
          Kad[14] = fma(Dbc[3], v, Kad[14]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[2] = fma(ac3, v, Kbd[2]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[28] = fma(Dbd[0], v, Kac[28]);
          Kad[12] = fma(Dbc[4], v, Kad[12]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[0] = fma(ac4, v, Kbd[0]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[28] = fma(Dbd[1], v, Kac[28]);
          Kad[13] = fma(Dbc[4], v, Kad[13]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[1] = fma(ac4, v, Kbd[1]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[28] = fma(Dbd[2], v, Kac[28]);
          Kad[14] = fma(Dbc[4], v, Kad[14]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[2] = fma(ac4, v, Kbd[2]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[29] = fma(Dbd[0], v, Kac[29]);
          Kad[12] = fma(Dbc[5], v, Kad[12]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[0] = fma(ac5, v, Kbd[0]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[29] = fma(Dbd[1], v, Kac[29]);
          Kad[13] = fma(Dbc[5], v, Kad[13]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[1] = fma(ac5, v, Kbd[1]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[29] = fma(Dbd[2], v, Kac[29]);
          Kad[14] = fma(Dbc[5], v, Kad[14]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[2] = fma(ac5, v, Kbd[2]);
        }
        Jab[12] += j;
      }
      {
        const double ab = Pab[4 * n + 1] * (kCons[2][4] * kCons[1][1]);
        const double e0 = E[80];
        const double e1 = E[81];
        const double e2 = E[82];
        const double e3 = E[83];
        const double e4 = E[84];
        const double e5 = E[85];
        const double z000 = fma(e5, r021_0, fma(e4, r020_0, fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r022_0, fma(e4, r021_0, fma(e3, r012_0, fma(e2, r011_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r031_0, fma(e4, r030_0, fma(e3, r021_0, fma(e2, r020_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r121_0, fma(e4, r120_0, fma(e3, r111_0, fma(e2, r110_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r023_0, fma(e4, r022_0, fma(e3, r013_0, fma(e2, r012_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r032_0, fma(e4, r031_0, fma(e3, r022_0, fma(e2, r021_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r041_0, fma(e4, r040_0, fma(e3, r031_0, fma(e2, r030_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r122_0, fma(e4, r121_0, fma(e3, r112_0, fma(e2, r111_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r131_0, fma(e4, r130_0, fma(e3, r121_0, fma(e2, r120_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r221_0, fma(e4, r220_0, fma(e3, r211_0, fma(e2, r210_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r024_0, fma(e4, r023_0, fma(e3, r014_0, fma(e2, r013_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r033_0, fma(e4, r032_0, fma(e3, r023_0, fma(e2, r022_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r042_0, fma(e4, r041_0, fma(e3, r032_0, fma(e2, r031_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r051_0, fma(e4, r050_0, fma(e3, r041_0, fma(e2, r040_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r123_0, fma(e4, r122_0, fma(e3, r113_0, fma(e2, r112_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r132_0, fma(e4, r131_0, fma(e3, r122_0, fma(e2, r121_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r141_0, fma(e4, r140_0, fma(e3, r131_0, fma(e2, r130_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r212_0, fma(e2, r211_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r231_0, fma(e4, r230_0, fma(e3, r221_0, fma(e2, r220_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r321_0, fma(e4, r320_0, fma(e3, r311_0, fma(e2, r310_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[24] = fma(Dbd[3], v, Kac[24]);
          Kad[12] = fma(Dbc[6], v, Kad[12]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[24] = fma(Dbd[4], v, Kac[24]);
          Kad[13] = fma(Dbc[6], v, Kad[13]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[24] = fma(Dbd[5], v, Kac[24]);
          Kad[14] = fma(Dbc[6], v, Kad[14]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[25] = fma(Dbd[3], v, Kac[25]);
          Kad[12] = fma(Dbc[7], v, Kad[12]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[25] = fma(Dbd[4], v, Kac[25]);
          Kad[13] = fma(Dbc[7], v, Kad[13]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[25] = fma(Dbd[5], v, Kac[25]);
          Kad[14] = fma(Dbc[7], v, Kad[14]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[26] = fma(Dbd[3], v, Kac[26]);
          Kad[12] = fma(Dbc[8], v, Kad[12]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[26] = fma(Dbd[4], v, Kac[26]);
          Kad[13] = fma(Dbc[8], v, Kad[13]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[26] = fma(Dbd[5], v, Kac[26]);
          Kad[14] = fma(Dbc[8], v, Kad[14]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[27] = fma(Dbd[3], v, Kac[27]);
          Kad[12] = fma(Dbc[9], v, Kad[12]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[3] = fma(ac3, v, Kbd[3]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[27] = fma(Dbd[4], v, Kac[27]);
          Kad[13] = fma(Dbc[9], v, Kad[13]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[4] = fma(ac3, v, Kbd[4]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[27] = fma(Dbd[5], v, Kac[27]);
          Kad[14] = fma(Dbc[9], v, Kad[14]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[5] = fma(ac3, v, Kbd[5]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[28] = fma(Dbd[3], v, Kac[28]);
          Kad[12] = fma(Dbc[10], v, Kad[12]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[3] = fma(ac4, v, Kbd[3]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[28] = fma(Dbd[4], v, Kac[28]);
          Kad[13] = fma(Dbc[10], v, Kad[13]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[4] = fma(ac4, v, Kbd[4]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[28] = fma(Dbd[5], v, Kac[28]);
          Kad[14] = fma(Dbc[10], v, Kad[14]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[5] = fma(ac4, v, Kbd[5]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[29] = fma(Dbd[3], v, Kac[29]);
          Kad[12] = fma(Dbc[11], v, Kad[12]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[3] = fma(ac5, v, Kbd[3]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[29] = fma(Dbd[4], v, Kac[29]);
          Kad[13] = fma(Dbc[11], v, Kad[13]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[4] = fma(ac5, v, Kbd[4]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[29] = fma(Dbd[5], v, Kac[29]);
          Kad[14] = fma(Dbc[11], v, Kad[14]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[5] = fma(ac5, v, Kbd[5]);
        }
        Jab[13] += j;
      }
      {
        const double ab = Pab[4 * n + 2] * (kCons[2][4] * kCons[1][2]);
        const double e0 = E[86];
        const double e1 = E[87];
        const double e2 = E[88];
        const double e3 = E[89];
        const double e4 = E[90];
        const double e5 = E[91];
        const double z000 = fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r015_0, fma(e4, r014_0, fma(e3, r013_0, fma(e2, r005_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r024_0, fma(e4, r023_0, fma(e3, r022_0, fma(e2, r014_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r033_0, fma(e4, r032_0, fma(e3, r031_0, fma(e2, r023_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r042_0, fma(e4, r041_0, fma(e3, r040_0, fma(e2, r032_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r114_0, fma(e4, r113_0, fma(e3, r112_0, fma(e2, r104_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r123_0, fma(e4, r122_0, fma(e3, r121_0, fma(e2, r113_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r132_0, fma(e4, r131_0, fma(e3, r130_0, fma(e2, r122_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r213_0, fma(e4, r212_0, fma(e3, r211_0, fma(e2, r203_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r220_0, fma(e2, r212_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r312_0, fma(e4, r311_0, fma(e3, r310_0, fma(e2, r302_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[24] = fma(Dbd[6], v, Kac[24]);
          Kad[12] = fma(Dbc[12], v, Kad[12]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[24] = fma(Dbd[7], v, Kac[24]);
          Kad[13] = fma(Dbc[12], v, Kad[13]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[24] = fma(Dbd[8], v, Kac[24]);
          Kad[14] = fma(Dbc[12], v, Kad[14]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[25] = fma(Dbd[6], v, Kac[25]);
          Kad[12] = fma(Dbc[13], v, Kad[12]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[25] = fma(Dbd[7], v, Kac[25]);
          Kad[13] = fma(Dbc[13], v, Kad[13]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[25] = fma(Dbd[8], v, Kac[25]);
          Kad[14] = fma(Dbc[13], v, Kad[14]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[26] = fma(Dbd[6], v, Kac[26]);
          Kad[12] = fma(Dbc[14], v, Kad[12]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[26] = fma(Dbd[7], v, Kac[26]);
          Kad[13] = fma(Dbc[14], v, Kad[13]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[26] = fma(Dbd[8], v, Kac[26]);
          Kad[14] = fma(Dbc[14], v, Kad[14]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[27] = fma(Dbd[6], v, Kac[27]);
          Kad[12] = fma(Dbc[15], v, Kad[12]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[6] = fma(ac3, v, Kbd[6]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[27] = fma(Dbd[7], v, Kac[27]);
          Kad[13] = fma(Dbc[15], v, Kad[13]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[7] = fma(ac3, v, Kbd[7]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[27] = fma(Dbd[8], v, Kac[27]);
          Kad[14] = fma(Dbc[15], v, Kad[14]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[8] = fma(ac3, v, Kbd[8]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[28] = fma(Dbd[6], v, Kac[28]);
          Kad[12] = fma(Dbc[16], v, Kad[12]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[6] = fma(ac4, v, Kbd[6]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[28] = fma(Dbd[7], v, Kac[28]);
          Kad[13] = fma(Dbc[16], v, Kad[13]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[7] = fma(ac4, v, Kbd[7]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[28] = fma(Dbd[8], v, Kac[28]);
          Kad[14] = fma(Dbc[16], v, Kad[14]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[8] = fma(ac4, v, Kbd[8]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[29] = fma(Dbd[6], v, Kac[29]);
          Kad[12] = fma(Dbc[17], v, Kad[12]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[6] = fma(ac5, v, Kbd[6]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[29] = fma(Dbd[7], v, Kac[29]);
          Kad[13] = fma(Dbc[17], v, Kad[13]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[7] = fma(ac5, v, Kbd[7]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[29] = fma(Dbd[8], v, Kac[29]);
          Kad[14] = fma(Dbc[17], v, Kad[14]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[8] = fma(ac5, v, Kbd[8]);
        }
        Jab[14] += j;
      }
    }
    {
      const double ac0 = P[oc + 5 * n + 0] * kCons[2][5];
      const double ac1 = P[oc + 5 * n + 1] * kCons[2][5];
      const double ac2 = P[oc + 5 * n + 2] * kCons[2][5];
      const double ac3 = P[oc + 5 * n + 3] * kCons[2][5];
      const double ac4 = P[oc + 5 * n + 4] * kCons[2][5];
      const double ac5 = P[oc + 5 * n + 5] * kCons[2][5];
      const double ad0 = P[od + 5 * n + 0] * kCons[2][5];
      const double ad1 = P[od + 5 * n + 1] * kCons[2][5];
      const double ad2 = P[od + 5 * n + 2] * kCons[2][5];
      {
        const double ab = Pab[5 * n + 0] * (kCons[2][5] * kCons[1][0]);
        const double e0 = E[92];
        const double e1 = E[93];
        const double e2 = E[94];
        const double e3 = E[95];
        const double e4 = E[96];
        const double e5 = E[97];
        const double z000 = fma(e5, r102_0, fma(e4, r101_0, fma(e3, r100_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r103_0, fma(e4, r102_0, fma(e3, r101_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r202_0, fma(e4, r201_0, fma(e3, r200_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r104_0, fma(e4, r103_0, fma(e3, r102_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r203_0, fma(e4, r202_0, fma(e3, r201_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r302_0, fma(e4, r301_0, fma(e3, r300_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r105_0, fma(e4, r104_0, fma(e3, r103_0, fma(e2, r005_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r114_0, fma(e4, r113_0, fma(e3, r112_0, fma(e2, r014_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r123_0, fma(e4, r122_0, fma(e3, r121_0, fma(e2, r023_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r132_0, fma(e4, r131_0, fma(e3, r130_0, fma(e2, r032_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r204_0, fma(e4, r203_0, fma(e3, r202_0, fma(e2, r104_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r213_0, fma(e4, r212_0, fma(e3, r211_0, fma(e2, r113_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r220_0, fma(e2, r122_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r303_0, fma(e4, r302_0, fma(e3, r301_0, fma(e2, r203_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r312_0, fma(e4, r311_0, fma(e3, r310_0, fma(e2, r212_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r402_0, fma(e4, r401_0, fma(e3, r400_0, fma(e2, r302_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[30] = fma(Dbd[0], v, Kac[30]);
          Kad[15] = fma(Dbc[0], v, Kad[15]);
          Kbc[0] = fma(ad0, v, Kbc[0]);
          Kbd[0] = fma(ac0, v, Kbd[0]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[30] = fma(Dbd[1], v, Kac[30]);
          Kad[16] = fma(Dbc[0], v, Kad[16]);
          Kbc[0] = fma(ad1, v, Kbc[0]);
          Kbd[1] = fma(ac0, v, Kbd[1]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[30] = fma(Dbd[2], v, Kac[30]);
          Kad[17] = fma(Dbc[0], v, Kad[17]);
          Kbc[0] = fma(ad2, v, Kbc[0]);
          Kbd[2] = fma(ac0, v, Kbd[2]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[31] = fma(Dbd[0], v, Kac[31]);
          Kad[15] = fma(Dbc[1], v, Kad[15]);
          Kbc[1] = fma(ad0, v, Kbc[1]);
          Kbd[0] = fma(ac1, v, Kbd[0]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[31] = fma(Dbd[1], v, Kac[31]);
          Kad[16] = fma(Dbc[1], v, Kad[16]);
          Kbc[1] = fma(ad1, v, Kbc[1]);
          Kbd[1] = fma(ac1, v, Kbd[1]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[31] = fma(Dbd[2], v, Kac[31]);
          Kad[17] = fma(Dbc[1], v, Kad[17]);
          Kbc[1] = fma(ad2, v, Kbc[1]);
          Kbd[2] = fma(ac1, v, Kbd[2]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[32] = fma(Dbd[0], v, Kac[32]);
          Kad[15] = fma(Dbc[2], v, Kad[15]);
          Kbc[2] = fma(ad0, v, Kbc[2]);
          Kbd[0] = fma(ac2, v, Kbd[0]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[32] = fma(Dbd[1], v, Kac[32]);
          Kad[16] = fma(Dbc[2], v, Kad[16]);
          Kbc[2] = fma(ad1, v, Kbc[2]);
          Kbd[1] = fma(ac2, v, Kbd[1]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[32] = fma(Dbd[2], v, Kac[32]);
          Kad[17] = fma(Dbc[2], v, Kad[17]);
          Kbc[2] = fma(ad2, v, Kbc[2]);
          Kbd[2] = fma(ac2, v, Kbd[2]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[33] = fma(Dbd[0], v, Kac[33]);
          Kad[15] = fma(Dbc[3], v, Kad[15]);
          Kbc[3] = fma(ad0, v, Kbc[3]);
          Kbd[0] = fma(ac3, v, Kbd[0]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[33] = fma(Dbd[1], v, Kac[33]);
          Kad[16] = fma(Dbc[3], v, Kad[16]);
          Kbc[3] = fma(ad1, v, Kbc[3]);
          Kbd[1] = fma(ac3, v, Kbd[1]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[33] = fma(Dbd[2], v, Kac[33]);
          Kad[17] = fma(Dbc[3], v, Kad[17]);
          Kbc[3] = fma(ad2, v, Kbc[3]);
          Kbd[2] = fma(ac3, v, Kbd[2]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[34] = fma(Dbd[0], v, Kac[34]);
          Kad[15] = fma(Dbc[4], v, Kad[15]);
          Kbc[4] = fma(ad0, v, Kbc[4]);
          Kbd[0] = fma(ac4, v, Kbd[0]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[34] = fma(Dbd[1], v, Kac[34]);
          Kad[16] = fma(Dbc[4], v, Kad[16]);
          Kbc[4] = fma(ad1, v, Kbc[4]);
          Kbd[1] = fma(ac4, v, Kbd[1]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[34] = fma(Dbd[2], v, Kac[34]);
          Kad[17] = fma(Dbc[4], v, Kad[17]);
          Kbc[4] = fma(ad2, v, Kbc[4]);
          Kbd[2] = fma(ac4, v, Kbd[2]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[35] = fma(Dbd[0], v, Kac[35]);
          Kad[15] = fma(Dbc[5], v, Kad[15]);
          Kbc[5] = fma(ad0, v, Kbc[5]);
          Kbd[0] = fma(ac5, v, Kbd[0]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[35] = fma(Dbd[1], v, Kac[35]);
          Kad[16] = fma(Dbc[5], v, Kad[16]);
          Kbc[5] = fma(ad1, v, Kbc[5]);
          Kbd[1] = fma(ac5, v, Kbd[1]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[35] = fma(Dbd[2], v, Kac[35]);
          Kad[17] = fma(Dbc[5], v, Kad[17]);
          Kbc[5] = fma(ad2, v, Kbc[5]);
          Kbd[2] = fma(ac5, v, Kbd[2]);
        }
        Jab[15] += j;
      }
      {
        const double ab = Pab[5 * n + 1] * (kCons[2][5] * kCons[1][1]);
        const double e0 = E[98];
        const double e1 = E[99];
        const double e2 = E[100];
        const double e3 = E[101];
        const double e4 = E[102];
        const double e5 = E[103];
        const double z000 = fma(e5, r012_0, fma(e4, r011_0, fma(e3, r010_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)))));
        const double z001 = fma(e5, r013_0, fma(e4, r012_0, fma(e3, r011_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)))));
        const double z010 = fma(e5, r022_0, fma(e4, r021_0, fma(e3, r020_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)))));
        const double z100 = fma(e5, r112_0, fma(e4, r111_0, fma(e3, r110_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)))));
        const double z002 = fma(e5, r014_0, fma(e4, r013_0, fma(e3, r012_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)))));
        const double z011 = fma(e5, r023_0, fma(e4, r022_0, fma(e3, r021_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)))));
        const double z020 = fma(e5, r032_0, fma(e4, r031_0, fma(e3, r030_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)))));
        const double z101 = fma(e5, r113_0, fma(e4, r112_0, fma(e3, r111_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)))));
        const double z110 = fma(e5, r122_0, fma(e4, r121_0, fma(e3, r120_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)))));
        const double z200 = fma(e5, r212_0, fma(e4, r211_0, fma(e3, r210_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)))));
        const double z003 = fma(e5, r015_0, fma(e4, r014_0, fma(e3, r013_0, fma(e2, r005_0, fma(e1, r004_0, e0 * r003_0)))));
        const double z012 = fma(e5, r024_0, fma(e4, r023_0, fma(e3, r022_0, fma(e2, r014_0, fma(e1, r013_0, e0 * r012_0)))));
        const double z021 = fma(e5, r033_0, fma(e4, r032_0, fma(e3, r031_0, fma(e2, r023_0, fma(e1, r022_0, e0 * r021_0)))));
        const double z030 = fma(e5, r042_0, fma(e4, r041_0, fma(e3, r040_0, fma(e2, r032_0, fma(e1, r031_0, e0 * r030_0)))));
        const double z102 = fma(e5, r114_0, fma(e4, r113_0, fma(e3, r112_0, fma(e2, r104_0, fma(e1, r103_0, e0 * r102_0)))));
        const double z111 = fma(e5, r123_0, fma(e4, r122_0, fma(e3, r121_0, fma(e2, r113_0, fma(e1, r112_0, e0 * r111_0)))));
        const double z120 = fma(e5, r132_0, fma(e4, r131_0, fma(e3, r130_0, fma(e2, r122_0, fma(e1, r121_0, e0 * r120_0)))));
        const double z201 = fma(e5, r213_0, fma(e4, r212_0, fma(e3, r211_0, fma(e2, r203_0, fma(e1, r202_0, e0 * r201_0)))));
        const double z210 = fma(e5, r222_0, fma(e4, r221_0, fma(e3, r220_0, fma(e2, r212_0, fma(e1, r211_0, e0 * r210_0)))));
        const double z300 = fma(e5, r312_0, fma(e4, r311_0, fma(e3, r310_0, fma(e2, r302_0, fma(e1, r301_0, e0 * r300_0)))));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[30] = fma(Dbd[3], v, Kac[30]);
          Kad[15] = fma(Dbc[6], v, Kad[15]);
          Kbc[6] = fma(ad0, v, Kbc[6]);
          Kbd[3] = fma(ac0, v, Kbd[3]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[30] = fma(Dbd[4], v, Kac[30]);
          Kad[16] = fma(Dbc[6], v, Kad[16]);
          Kbc[6] = fma(ad1, v, Kbc[6]);
          Kbd[4] = fma(ac0, v, Kbd[4]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[30] = fma(Dbd[5], v, Kac[30]);
          Kad[17] = fma(Dbc[6], v, Kad[17]);
          Kbc[6] = fma(ad2, v, Kbc[6]);
          Kbd[5] = fma(ac0, v, Kbd[5]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[31] = fma(Dbd[3], v, Kac[31]);
          Kad[15] = fma(Dbc[7], v, Kad[15]);
          Kbc[7] = fma(ad0, v, Kbc[7]);
          Kbd[3] = fma(ac1, v, Kbd[3]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[31] = fma(Dbd[4], v, Kac[31]);
          Kad[16] = fma(Dbc[7], v, Kad[16]);
          Kbc[7] = fma(ad1, v, Kbc[7]);
          Kbd[4] = fma(ac1, v, Kbd[4]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[31] = fma(Dbd[5], v, Kac[31]);
          Kad[17] = fma(Dbc[7], v, Kad[17]);
          Kbc[7] = fma(ad2, v, Kbc[7]);
          Kbd[5] = fma(ac1, v, Kbd[5]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[32] = fma(Dbd[3], v, Kac[32]);
          Kad[15] = fma(Dbc[8], v, Kad[15]);
          Kbc[8] = fma(ad0, v, Kbc[8]);
          Kbd[3] = fma(ac2, v, Kbd[3]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[32] = fma(Dbd[4], v, Kac[32]);
          Kad[16] = fma(Dbc[8], v, Kad[16]);
          Kbc[8] = fma(ad1, v, Kbc[8]);
          Kbd[4] = fma(ac2, v, Kbd[4]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[32] = fma(Dbd[5], v, Kac[32]);
          Kad[17] = fma(Dbc[8], v, Kad[17]);
          Kbc[8] = fma(ad2, v, Kbc[8]);
          Kbd[5] = fma(ac2, v, Kbd[5]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[33] = fma(Dbd[3], v, Kac[33]);
          Kad[15] = fma(Dbc[9], v, Kad[15]);
          Kbc[9] = fma(ad0, v, Kbc[9]);
          Kbd[3] = fma(ac3, v, Kbd[3]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[33] = fma(Dbd[4], v, Kac[33]);
          Kad[16] = fma(Dbc[9], v, Kad[16]);
          Kbc[9] = fma(ad1, v, Kbc[9]);
          Kbd[4] = fma(ac3, v, Kbd[4]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[33] = fma(Dbd[5], v, Kac[33]);
          Kad[17] = fma(Dbc[9], v, Kad[17]);
          Kbc[9] = fma(ad2, v, Kbc[9]);
          Kbd[5] = fma(ac3, v, Kbd[5]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[34] = fma(Dbd[3], v, Kac[34]);
          Kad[15] = fma(Dbc[10], v, Kad[15]);
          Kbc[10] = fma(ad0, v, Kbc[10]);
          Kbd[3] = fma(ac4, v, Kbd[3]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[34] = fma(Dbd[4], v, Kac[34]);
          Kad[16] = fma(Dbc[10], v, Kad[16]);
          Kbc[10] = fma(ad1, v, Kbc[10]);
          Kbd[4] = fma(ac4, v, Kbd[4]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[34] = fma(Dbd[5], v, Kac[34]);
          Kad[17] = fma(Dbc[10], v, Kad[17]);
          Kbc[10] = fma(ad2, v, Kbc[10]);
          Kbd[5] = fma(ac4, v, Kbd[5]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[35] = fma(Dbd[3], v, Kac[35]);
          Kad[15] = fma(Dbc[11], v, Kad[15]);
          Kbc[11] = fma(ad0, v, Kbc[11]);
          Kbd[3] = fma(ac5, v, Kbd[3]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[35] = fma(Dbd[4], v, Kac[35]);
          Kad[16] = fma(Dbc[11], v, Kad[16]);
          Kbc[11] = fma(ad1, v, Kbc[11]);
          Kbd[4] = fma(ac5, v, Kbd[4]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[35] = fma(Dbd[5], v, Kac[35]);
          Kad[17] = fma(Dbc[11], v, Kad[17]);
          Kbc[11] = fma(ad2, v, Kbc[11]);
          Kbd[5] = fma(ac5, v, Kbd[5]);
        }
        Jab[16] += j;
      }
      {
        const double ab = Pab[5 * n + 2] * (kCons[2][5] * kCons[1][2]);
        const double e0 = E[104];
        const double e1 = E[105];
        const double e2 = E[106];
        const double e3 = E[107];
        const double z000 = fma(e3, r003_0, fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0)));
        const double z001 = fma(e3, r004_0, fma(e2, r003_0, fma(e1, r002_0, e0 * r001_0)));
        const double z010 = fma(e3, r013_0, fma(e2, r012_0, fma(e1, r011_0, e0 * r010_0)));
        const double z100 = fma(e3, r103_0, fma(e2, r102_0, fma(e1, r101_0, e0 * r100_0)));
        const double z002 = fma(e3, r005_0, fma(e2, r004_0, fma(e1, r003_0, e0 * r002_0)));
        const double z011 = fma(e3, r014_0, fma(e2, r013_0, fma(e1, r012_0, e0 * r011_0)));
        const double z020 = fma(e3, r023_0, fma(e2, r022_0, fma(e1, r021_0, e0 * r020_0)));
        const double z101 = fma(e3, r104_0, fma(e2, r103_0, fma(e1, r102_0, e0 * r101_0)));
        const double z110 = fma(e3, r113_0, fma(e2, r112_0, fma(e1, r111_0, e0 * r110_0)));
        const double z200 = fma(e3, r203_0, fma(e2, r202_0, fma(e1, r201_0, e0 * r200_0)));
        const double z003 = fma(e3, r006_0, fma(e2, r005_0, fma(e1, r004_0, e0 * r003_0)));
        const double z012 = fma(e3, r015_0, fma(e2, r014_0, fma(e1, r013_0, e0 * r012_0)));
        const double z021 = fma(e3, r024_0, fma(e2, r023_0, fma(e1, r022_0, e0 * r021_0)));
        const double z030 = fma(e3, r033_0, fma(e2, r032_0, fma(e1, r031_0, e0 * r030_0)));
        const double z102 = fma(e3, r105_0, fma(e2, r104_0, fma(e1, r103_0, e0 * r102_0)));
        const double z111 = fma(e3, r114_0, fma(e2, r113_0, fma(e1, r112_0, e0 * r111_0)));
        const double z120 = fma(e3, r123_0, fma(e2, r122_0, fma(e1, r121_0, e0 * r120_0)));
        const double z201 = fma(e3, r204_0, fma(e2, r203_0, fma(e1, r202_0, e0 * r201_0)));
        const double z210 = fma(e3, r213_0, fma(e2, r212_0, fma(e1, r211_0, e0 * r210_0)));
        const double z300 = fma(e3, r303_0, fma(e2, r302_0, fma(e1, r301_0, e0 * r300_0)));
        double j = 0.0;
        {
          const double v = fma(k0_0_300, z300, fma(k0_0_200, z200, fma(k0_0_100, z100, k0_0_000 * z000)));
          j = fma(Dcd[0], v, j);
          Jcd[0] = fma(ab, v, Jcd[0]);
          Kac[30] = fma(Dbd[6], v, Kac[30]);
          Kad[15] = fma(Dbc[12], v, Kad[15]);
          Kbc[12] = fma(ad0, v, Kbc[12]);
          Kbd[6] = fma(ac0, v, Kbd[6]);
        }
        {
          const double v = fma(k0_1_210, z210, fma(k0_1_200, z200, fma(k0_1_110, z110, fma(k0_1_100, z100, fma(k0_1_010, z010, k0_1_000 * z000)))));
          j = fma(Dcd[1], v, j);
          Jcd[1] = fma(ab, v, Jcd[1]);
          Kac[30] = fma(Dbd[7], v, Kac[30]);
          Kad[16] = fma(Dbc[12], v, Kad[16]);
          Kbc[12] = fma(ad1, v, Kbc[12]);
          Kbd[7] = fma(ac0, v, Kbd[7]);
        }
        {
          const double v = fma(k0_2_201, z201, fma(k0_2_200, z200, fma(k0_2_101, z101, fma(k0_2_100, z100, fma(k0_2_001, z001, k0_2_000 * z000)))));
          j = fma(Dcd[2], v, j);
          Jcd[2] = fma(ab, v, Jcd[2]);
          Kac[30] = fma(Dbd[8], v, Kac[30]);
          Kad[17] = fma(Dbc[12], v, Kad[17]);
          Kbc[12] = fma(ad2, v, Kbc[12]);
          Kbd[8] = fma(ac0, v, Kbd[8]);
        }
        {
          const double v = fma(k1_0_210, z210, fma(k1_0_200, z200, fma(k1_0_110, z110, fma(k1_0_100, z100, fma(k1_0_010, z010, k1_0_000 * z000)))));
          j = fma(Dcd[3], v, j);
          Jcd[3] = fma(ab, v, Jcd[3]);
          Kac[31] = fma(Dbd[6], v, Kac[31]);
          Kad[15] = fma(Dbc[13], v, Kad[15]);
          Kbc[13] = fma(ad0, v, Kbc[13]);
          Kbd[6] = fma(ac1, v, Kbd[6]);
        }
        {
          const double v = fma(k1_1_120, z120, fma(k1_1_110, z110, fma(k1_1_100, z100, fma(k1_1_020, z020, fma(k1_1_010, z010, k1_1_000 * z000)))));
          j = fma(Dcd[4], v, j);
          Jcd[4] = fma(ab, v, Jcd[4]);
          Kac[31] = fma(Dbd[7], v, Kac[31]);
          Kad[16] = fma(Dbc[13], v, Kad[16]);
          Kbc[13] = fma(ad1, v, Kbc[13]);
          Kbd[7] = fma(ac1, v, Kbd[7]);
        }
        {
          const double v = fma(k1_2_111, z111, fma(k1_2_110, z110, fma(k1_2_101, z101, fma(k1_2_100, z100, fma(k1_2_011, z011, fma(k1_2_010, z010, fma(k1_2_001, z001, k1_2_000 * z000)))))));
          j = fma(Dcd[5], v, j);
          Jcd[5] = fma(ab, v, Jcd[5]);
          Kac[31] = fma(Dbd[8], v, Kac[31]);
          Kad[17] = fma(Dbc[13], v, Kad[17]);
          Kbc[13] = fma(ad2, v, Kbc[13]);
          Kbd[8] = fma(ac1, v, Kbd[8]);
        }
        {
          const double v = fma(k2_0_120, z120, fma(k2_0_110, z110, fma(k2_0_100, z100, fma(k2_0_020, z020, fma(k2_0_010, z010, k2_0_000 * z000)))));
          j = fma(Dcd[6], v, j);
          Jcd[6] = fma(ab, v, Jcd[6]);
          Kac[32] = fma(Dbd[6], v, Kac[32]);
          Kad[15] = fma(Dbc[14], v, Kad[15]);
          Kbc[14] = fma(ad0, v, Kbc[14]);
          Kbd[6] = fma(ac2, v, Kbd[6]);
        }
        {
          const double v = fma(k2_1_030, z030, fma(k2_1_020, z020, fma(k2_1_010, z010, k2_1_000 * z000)));
          j = fma(Dcd[7], v, j);
          Jcd[7] = fma(ab, v, Jcd[7]);
          Kac[32] = fma(Dbd[7], v, Kac[32]);
          Kad[16] = fma(Dbc[14], v, Kad[16]);
          Kbc[14] = fma(ad1, v, Kbc[14]);
          Kbd[7] = fma(ac2, v, Kbd[7]);
        }
        {
          const double v = fma(k2_2_021, z021, fma(k2_2_020, z020, fma(k2_2_011, z011, fma(k2_2_010, z010, fma(k2_2_001, z001, k2_2_000 * z000)))));
          j = fma(Dcd[8], v, j);
          Jcd[8] = fma(ab, v, Jcd[8]);
          Kac[32] = fma(Dbd[8], v, Kac[32]);
          Kad[17] = fma(Dbc[14], v, Kad[17]);
          Kbc[14] = fma(ad2, v, Kbc[14]);
          Kbd[8] = fma(ac2, v, Kbd[8]);
        }
        {
          const double v = fma(k3_0_201, z201, fma(k3_0_200, z200, fma(k3_0_101, z101, fma(k3_0_100, z100, fma(k3_0_001, z001, k3_0_000 * z000)))));
          j = fma(Dcd[9], v, j);
          Jcd[9] = fma(ab, v, Jcd[9]);
          Kac[33] = fma(Dbd[6], v, Kac[33]);
          Kad[15] = fma(Dbc[15], v, Kad[15]);
          Kbc[15] = fma(ad0, v, Kbc[15]);
          Kbd[6] = fma(ac3, v, Kbd[6]);
        }
        {
          const double v = fma(k3_1_111, z111, fma(k3_1_110, z110, fma(k3_1_101, z101, fma(k3_1_100, z100, fma(k3_1_011, z011, fma(k3_1_010, z010, fma(k3_1_001, z001, k3_1_000 * z000)))))));
          j = fma(Dcd[10], v, j);
          Jcd[10] = fma(ab, v, Jcd[10]);
          Kac[33] = fma(Dbd[7], v, Kac[33]);
          Kad[16] = fma(Dbc[15], v, Kad[16]);
          Kbc[15] = fma(ad1, v, Kbc[15]);
          Kbd[7] = fma(ac3, v, Kbd[7]);
        }
        {
          const double v = fma(k3_2_102, z102, fma(k3_2_101, z101, fma(k3_2_100, z100, fma(k3_2_002, z002, fma(k3_2_001, z001, k3_2_000 * z000)))));
          j = fma(Dcd[11], v, j);
          Jcd[11] = fma(ab, v, Jcd[11]);
          Kac[33] = fma(Dbd[8], v, Kac[33]);
          Kad[17] = fma(Dbc[15], v, Kad[17]);
          Kbc[15] = fma(ad2, v, Kbc[15]);
          Kbd[8] = fma(ac3, v, Kbd[8]);
        }
        {
          const double v = fma(k4_0_111, z111, fma(k4_0_110, z110, fma(k4_0_101, z101, fma(k4_0_100, z100, fma(k4_0_011, z011, fma(k4_0_010, z010, fma(k4_0_001, z001, k4_0_000 * z000)))))));
          j = fma(Dcd[12], v, j);
          Jcd[12] = fma(ab, v, Jcd[12]);
          Kac[34] = fma(Dbd[6], v, Kac[34]);
          Kad[15] = fma(Dbc[16], v, Kad[15]);
          Kbc[16] = fma(ad0, v, Kbc[16]);
          Kbd[6] = fma(ac4, v, Kbd[6]);
        }
        {
          const double v = fma(k4_1_021, z021, fma(k4_1_020, z020, fma(k4_1_011, z011, fma(k4_1_010, z010, fma(k4_1_001, z001, k4_1_000 * z000)))));
          j = fma(Dcd[13], v, j);
          Jcd[13] = fma(ab, v, Jcd[13]);
          Kac[34] = fma(Dbd[7], v, Kac[34]);
          Kad[16] = fma(Dbc[16], v, Kad[16]);
          Kbc[16] = fma(ad1, v, Kbc[16]);
          Kbd[7] = fma(ac4, v, Kbd[7]);
        }
        {
          const double v = fma(k4_2_012, z012, fma(k4_2_011, z011, fma(k4_2_010, z010, fma(k4_2_002, z002, fma(k4_2_001, z001, k4_2_000 * z000)))));
          j = fma(Dcd[14], v, j);
          Jcd[14] = fma(ab, v, Jcd[14]);
          Kac[34] = fma(Dbd[8], v, Kac[34]);
          Kad[17] = fma(Dbc[16], v, Kad[17]);
          Kbc[16] = fma(ad2, v, Kbc[16]);
          Kbd[8] = fma(ac4, v, Kbd[8]);
        }
        {
          const double v = fma(k5_0_102, z102, fma(k5_0_101, z101, fma(k5_0_100, z100, fma(k5_0_002, z002, fma(k5_0_001, z001, k5_0_000 * z000)))));
          j = fma(Dcd[15], v, j);
          Jcd[15] = fma(ab, v, Jcd[15]);
          Kac[35] = fma(Dbd[6], v, Kac[35]);
          Kad[15] = fma(Dbc[17], v, Kad[15]);
          Kbc[17] = fma(ad0, v, Kbc[17]);
          Kbd[6] = fma(ac5, v, Kbd[6]);
        }
        {
          const double v = fma(k5_1_012, z012, fma(k5_1_011, z011, fma(k5_1_010, z010, fma(k5_1_002, z002, fma(k5_1_001, z001, k5_1_000 * z000)))));
          j = fma(Dcd[16], v, j);
          Jcd[16] = fma(ab, v, Jcd[16]);
          Kac[35] = fma(Dbd[7], v, Kac[35]);
          Kad[16] = fma(Dbc[17], v, Kad[16]);
          Kbc[17] = fma(ad1, v, Kbc[17]);
          Kbd[7] = fma(ac5, v, Kbd[7]);
        }
        {
          const double v = fma(k5_2_003, z003, fma(k5_2_002, z002, fma(k5_2_001, z001, k5_2_000 * z000)));
          j = fma(Dcd[17], v, j);
          Jcd[17] = fma(ab, v, Jcd[17]);
          Kac[35] = fma(Dbd[8], v, Kac[35]);
          Kad[17] = fma(Dbc[17], v, Kad[17]);
          Kbc[17] = fma(ad2, v, Kbc[17]);
          Kbd[8] = fma(ac5, v, Kbd[8]);
        }
        Jab[17] += j;
      }
    }
  }
};
__device__ const unsigned kC2121Md_index[108] = {11,12,13,14,264,520,265,521,266,522,65544,131080,65545,131081,65546,131082,773,1029,774,1030,775,1031,1283,1539,1795,1284,1540,1796,66307,131843,66563,132099,66308,131844,66564,132100,2049,2305,2561,2050,2306,2562,2816,3072,3328,3584,67584,133120,67840,133376,68096,133632,196613,262149,196614,262150,196615,262151,196867,262403,197123,262659,196868,262404,197124,262660,327683,393219,458755,327684,393220,458756,197377,262913,197633,263169,197378,262914,197634,263170,197888,263424,198144,263680,198400,263936,328448,393984,459520,328704,394240,459776,524289,589825,655361,524290,589826,655362,524544,590080,655616,524800,590336,655872,720896,786432,851968,917504};
__device__ inline const unsigned* C2121Md::index() { return kC2121Md_index; }
}  // namespace qf
