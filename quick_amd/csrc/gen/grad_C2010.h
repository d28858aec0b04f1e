// Generated by quick_amd/codegen/gen_grad.py - do not edit.
#pragma once
#include "../qf_grad.h"
namespace qf {
struct C2010Grad {
  static constexpr int La = 2, Lb = 0, Lc = 1, Ld = 0, L = 4;
  static constexpr int NACC = 129, NV = 170, NLV = 4, NX = 129, NH = 135, NLH = 1, NI = 18;
  static constexpr int ZS = 129, SINK = 130, CF = 418, DM = 458, LDS = 495;
  // output blocks (a+1 b|cd), (a-1 b|cd), (a b+1|cd), (a b-1|cd), (ab|c+1 d), (ab|c-1 d); -1: absent
  static constexpr int OAP = 131, OAM = 161, OBP = 170, OBM = -1, OCP = 224, OCM = 260;
  static constexpr bool GLOBAL_SLOTS = false;   // slots in a global scratch buffer (over 64 KiB)
  static constexpr int NT = 64;   // threads per workgroup: one wave
  static constexpr int PRIM_FLOP = 1073, QUARTET_FLOP = 936;
  static constexpr unsigned short FSLOT[5] = {266,267,268,269,270};   // slots of [00|00]^(m)
  __device__ static const CoopVNode* vrr();
  __device__ static const int* vlev();
  __device__ static const GradAcc* acc();
  __device__ static const CoopHNode* hrr();
  __device__ static const int* hlev();
};
__device__ const CoopVNode kC2010Grad_vrr[170] = {{269,270,129,129,129,271,65535,2},{269,270,129,129,129,272,65535,1},{269,270,129,129,129,273,65535,0},{268,269,129,129,129,274,65535,2},{268,269,129,129,129,275,65535,1},{268,269,129,129,129,276,65535,0},{267,268,129,129,129,277,65535,2},{267,268,129,129,129,278,65535,1},{267,268,129,129,129,279,65535,0},{266,267,129,129,129,280,65535,2},{266,267,129,129,129,281,65535,1},{266,267,129,129,129,282,65535,0},{274,271,268,269,129,270,65535,18},{274,271,129,129,129,283,65535,1},{275,272,268,269,129,284,65535,17},{274,271,129,129,129,285,65535,0},{275,272,129,129,129,286,65535,0},{276,273,268,269,129,287,65535,16},{277,274,267,268,129,288,65535,18},{277,274,129,129,129,289,65535,1},{278,275,267,268,129,290,65535,17},{277,274,129,129,129,291,65535,0},{278,275,129,129,129,292,65535,0},{279,276,267,268,129,293,65535,16},{280,277,266,267,129,294,65535,18},{280,277,129,129,129,295,65535,1},{281,278,266,267,129,296,65535,17},{280,277,129,129,129,297,65535,0},{281,278,129,129,129,298,65535,0},{282,279,266,267,129,299,65535,16},{277,274,129,129,268,300,65535,261},{277,274,129,129,129,301,65535,4},{277,274,129,129,129,302,65535,3},{278,275,129,129,129,303,65535,5},{278,275,129,129,268,304,65535,260},{278,275,129,129,129,305,65535,3},{279,276,129,129,129,306,65535,5},{279,276,129,129,129,307,65535,4},{279,276,129,129,268,308,65535,259},{280,277,129,129,267,309,65535,261},{280,277,129,129,129,310,65535,4},{280,277,129,129,129,311,65535,3},{281,278,129,129,129,312,65535,5},{281,278,129,129,267,313,65535,260},{281,278,129,129,129,314,65535,3},{282,279,129,129,129,315,65535,5},{282,279,129,129,129,316,65535,4},{282,279,129,129,267,317,65535,259},{288,270,277,274,129,266,65535,34},{288,270,129,129,129,267,65535,1},{290,284,129,129,129,268,65535,2},{290,284,278,275,129,269,65535,33},{288,270,129,129,129,271,65535,0},{289,283,129,129,129,272,65535,0},{290,284,129,129,129,273,65535,0},{293,287,129,129,129,318,65535,2},{293,287,129,129,129,319,65535,1},{293,287,279,276,129,320,65535,32},{294,288,280,277,129,321,65535,34},{294,288,129,129,129,322,65535,1},{296,290,129,129,129,323,65535,2},{296,290,281,278,129,324,65535,33},{294,288,129,129,129,325,65535,0},{295,289,129,129,129,326,65535,0},{296,290,129,129,129,327,65535,0},{299,293,129,129,129,328,65535,2},{299,293,129,129,129,329,65535,1},{299,293,282,279,129,330,65535,32},{288,270,129,129,274,331,65535,517},{288,270,129,129,129,332,65535,4},{288,270,129,129,129,333,65535,3},{289,283,129,129,275,334,65535,261},{289,283,129,129,274,335,65535,260},{289,283,129,129,129,336,65535,3},{290,284,129,129,129,337,65535,5},{290,284,129,129,275,338,65535,516},{290,284,129,129,129,339,65535,3},{291,285,129,129,276,340,65535,261},{291,285,129,129,129,341,65535,4},{291,285,129,129,274,342,65535,259},{292,286,129,129,129,343,65535,5},{292,286,129,129,276,344,65535,260},{292,286,129,129,275,345,65535,259},{293,287,129,129,129,346,65535,5},{293,287,129,129,129,347,65535,4},{293,287,129,129,276,348,65535,515},{294,288,129,129,277,349,65535,517},{294,288,129,129,129,350,65535,4},{294,288,129,129,129,351,65535,3},{295,289,129,129,278,352,65535,261},{295,289,129,129,277,353,65535,260},{295,289,129,129,129,354,65535,3},{296,290,129,129,129,355,65535,5},{296,290,129,129,278,356,65535,516},{296,290,129,129,129,357,65535,3},{297,291,129,129,279,358,65535,261},{297,291,129,129,129,359,65535,4},{297,291,129,129,277,360,65535,259},{298,292,129,129,129,361,65535,5},{298,292,129,129,279,362,65535,260},{298,292,129,129,278,363,65535,259},{299,293,129,129,129,364,65535,5},{299,293,129,129,129,365,65535,4},{299,293,129,129,279,366,65535,515},{321,266,129,129,288,270,65535,773},{321,266,129,129,129,274,65535,4},{321,266,129,129,129,275,65535,3},{322,267,129,129,289,276,65535,517},{322,267,129,129,288,277,65535,260},{322,267,129,129,129,278,65535,3},{323,268,129,129,290,279,65535,261},{323,268,129,129,289,280,65535,516},{323,268,129,129,129,281,65535,3},{324,269,129,129,129,282,65535,5},{324,269,129,129,290,283,65535,772},{324,269,129,129,129,284,65535,3},{325,271,129,129,291,285,65535,517},{325,271,129,129,129,286,65535,4},{325,271,129,129,288,287,65535,259},{326,272,129,129,292,367,65535,261},{326,272,129,129,291,368,65535,260},{326,272,129,129,289,369,65535,259},{327,273,129,129,129,370,65535,5},{327,273,129,129,292,371,65535,516},{327,273,129,129,290,372,65535,259},{328,318,129,129,293,373,65535,261},{328,318,129,129,129,374,65535,4},{328,318,129,129,291,375,65535,515},{329,319,129,129,129,376,65535,5},{329,319,129,129,293,377,65535,260},{329,319,129,129,292,378,65535,515},{330,320,129,129,129,379,65535,5},{330,320,129,129,129,380,65535,4},{330,320,129,129,293,381,65535,771},{349,331,294,288,300,382,65535,533},{349,331,129,129,129,383,65535,4},{350,332,294,288,129,384,65535,20},{349,331,129,129,129,385,65535,3},{350,332,129,129,129,386,65535,3},{351,333,294,288,129,387,65535,19},{352,334,295,289,303,388,65535,277},{352,334,129,129,300,389,65535,260},{353,335,295,289,301,390,65535,276},{352,334,129,129,129,391,65535,3},{353,335,129,129,129,392,65535,3},{354,336,295,289,129,393,65535,19},{355,337,296,290,129,394,65535,21},{356,338,129,129,129,395,65535,5},{356,338,296,290,304,396,65535,532},{355,337,129,129,129,397,65535,3},{356,338,129,129,129,398,65535,3},{357,339,296,290,129,399,65535,19},{358,340,297,291,306,400,65535,277},{358,340,129,129,129,401,65535,4},{359,341,297,291,129,402,65535,20},{358,340,129,129,300,403,65535,259},{360,342,129,129,129,404,65535,4},{360,342,297,291,302,405,65535,275},{361,343,298,292,129,406,65535,21},{362,344,129,129,129,407,65535,5},{362,344,298,292,307,408,65535,276},{363,345,129,129,129,409,65535,5},{362,344,129,129,304,410,65535,259},{363,345,298,292,305,411,65535,275},{364,346,299,293,129,412,65535,21},{364,346,129,129,129,413,65535,4},{365,347,299,293,129,414,65535,20},{366,348,129,129,129,415,65535,5},{366,348,129,129,129,416,65535,4},{366,348,299,293,308,417,65535,531}};
__device__ const int kC2010Grad_vlev[5] = {0,12,48,104,170};
__device__ const GradAcc kC2010Grad_acc[129] = {{317,0,0},{316,1,0},{315,2,0},{314,3,0},{313,4,0},{312,5,0},{311,6,0},{310,7,0},{309,8,0},{299,9,0},{298,10,0},{296,11,0},{297,12,0},{295,13,0},{294,14,0},{381,15,1},{380,16,1},{379,17,1},{378,18,1},{377,19,1},{376,20,1},{372,21,1},{371,22,1},{370,23,1},{284,24,1},{283,25,1},{282,26,1},{375,27,1},{374,28,1},{373,29,1},{369,30,1},{368,31,1},{367,32,1},{281,33,1},{280,34,1},{279,35,1},{287,36,1},{286,37,1},{285,38,1},{278,39,1},{277,40,1},{276,41,1},{275,42,1},{274,43,1},{270,44,1},{366,45,2},{365,46,2},{364,47,2},{363,48,2},{362,49,2},{361,50,2},{357,51,2},{356,52,2},{355,53,2},{360,54,2},{359,55,2},{358,56,2},{354,57,2},{353,58,2},{352,59,2},{351,60,2},{350,61,2},{349,62,2},{381,63,2},{380,64,2},{379,65,2},{378,66,2},{377,67,2},{376,68,2},{372,69,2},{371,70,2},{370,71,2},{284,72,2},{283,73,2},{282,74,2},{375,75,2},{374,76,2},{373,77,2},{369,78,2},{368,79,2},{367,80,2},{281,81,2},{280,82,2},{279,83,2},{287,84,2},{286,85,2},{285,86,2},{278,87,2},{277,88,2},{276,89,2},{275,90,2},{274,91,2},{270,92,2},{417,93,3},{416,94,3},{414,95,3},{415,96,3},{413,97,3},{412,98,3},{411,99,3},{410,100,3},{408,101,3},{409,102,3},{407,103,3},{406,104,3},{399,105,3},{398,106,3},{396,107,3},{397,108,3},{395,109,3},{394,110,3},{405,111,3},{404,112,3},{402,113,3},{403,114,3},{401,115,3},{400,116,3},{393,117,3},{392,118,3},{390,119,3},{391,120,3},{389,121,3},{388,122,3},{387,123,3},{386,124,3},{384,125,3},{385,126,3},{383,127,3},{382,128,3}};
__device__ const CoopHNode kC2010Grad_hrr[135] = {{223,92,62,5},{222,91,61,5},{221,90,60,5},{220,89,62,4},{219,88,61,4},{218,87,60,4},{217,86,62,3},{216,85,61,3},{215,84,60,3},{214,89,59,5},{213,88,58,5},{212,87,57,5},{211,83,59,4},{210,82,58,4},{209,81,57,4},{208,80,59,3},{207,79,58,3},{206,78,57,3},{196,83,53,5},{195,82,52,5},{194,81,51,5},{193,74,53,4},{192,73,52,4},{191,72,51,4},{190,71,53,3},{189,70,52,3},{188,69,51,3},{205,86,56,5},{204,85,55,5},{203,84,54,5},{202,80,56,4},{201,79,55,4},{200,78,54,4},{199,77,56,3},{198,76,55,3},{197,75,54,3},{187,80,50,5},{186,79,49,5},{185,78,48,5},{184,71,50,4},{183,70,49,4},{182,69,48,4},{181,68,50,3},{180,67,49,3},{179,66,48,3},{178,77,47,5},{177,76,46,5},{176,75,45,5},{175,68,47,4},{174,67,46,4},{173,66,45,4},{172,65,47,3},{171,64,46,3},{170,63,45,3},{161,0,129,0},{162,1,129,0},{163,2,129,0},{164,3,129,0},{165,4,129,0},{166,5,129,0},{167,6,129,0},{168,7,129,0},{169,8,129,0},{131,15,129,0},{132,16,129,0},{141,25,129,0},{142,26,129,0},{143,27,129,0},{144,28,129,0},{145,29,129,0},{146,30,129,0},{147,31,129,0},{148,32,129,0},{149,33,129,0},{150,34,129,0},{133,17,129,0},{151,35,129,0},{152,36,129,0},{153,37,129,0},{154,38,129,0},{155,39,129,0},{156,40,129,0},{157,41,129,0},{158,42,129,0},{159,43,129,0},{160,44,129,0},{134,18,129,0},{135,19,129,0},{136,20,129,0},{137,21,129,0},{138,22,129,0},{139,23,129,0},{140,24,129,0},{260,9,129,0},{261,10,129,0},{262,11,129,0},{263,12,129,0},{264,13,129,0},{265,14,129,0},{224,93,129,0},{225,94,129,0},{234,103,129,0},{235,104,129,0},{236,105,129,0},{237,106,129,0},{238,107,129,0},{239,108,129,0},{240,109,129,0},{241,110,129,0},{242,111,129,0},{243,112,129,0},{226,95,129,0},{244,113,129,0},{245,114,129,0},{246,115,129,0},{247,116,129,0},{248,117,129,0},{249,118,129,0},{250,119,129,0},{251,120,129,0},{252,121,129,0},{253,122,129,0},{227,96,129,0},{254,123,129,0},{255,124,129,0},{256,125,129,0},{257,126,129,0},{258,127,129,0},{259,128,129,0},{228,97,129,0},{229,98,129,0},{230,99,129,0},{231,100,129,0},{232,101,129,0},{233,102,129,0}};
__device__ const int kC2010Grad_hlev[2] = {0,135};
__device__ inline const CoopVNode* C2010Grad::vrr() { return kC2010Grad_vrr; }
__device__ inline const int* C2010Grad::vlev() { return kC2010Grad_vlev; }
__device__ inline const GradAcc* C2010Grad::acc() { return kC2010Grad_acc; }
__device__ inline const CoopHNode* C2010Grad::hrr() { return kC2010Grad_hrr; }
__device__ inline const int* C2010Grad::hlev() { return kC2010Grad_hlev; }
// (ds|ps): 35 Hermite Coulomb integrals, 39 bra products
struct C2010GradMd {
  static constexpr int La = 2, Lb = 0, Lc = 1, Ld = 0, L = 4;
  static constexpr int N1 = 9, NE = 39;   // 1D entries per direction, product table
  static constexpr int MIN_WAVES = 1;      // waves per SIMD the register budget targets
  __device__ static const unsigned* index();   // 1D entries of a product, x | y << 8 | z << 16
  // 1D coefficients of one direction: X = P - A, Y = P - B, h = 1/2p, rx = -beta/p, ry = alpha/p
  template <class T>
  __host__ __device__ static __forceinline__ void bra1d(double X, double Y, double h, double rx, double ry, T out) {
    const double be100 = X;
    const double be101 = h;
    const double bd100 = rx;
    const double be200 = fma(1.0, be101, be100 * X);
    const double be201 = fma(be100, h, be101 * X);
    const double be202 = be101 * h;
    const double bd200 = fma(be100, rx, bd100 * X);
    const double bd201 = fma(be101, rx, bd100 * h);
    out[0] = 1.0;
    out[1] = be100;
    out[2] = be101;
    out[3] = bd100;
    out[4] = be200;
    out[5] = be201;
    out[6] = be202;
    out[7] = bd200;
    out[8] = bd201;
  }
  // Dcd with 2 cons, Dbc and Dbd with hyb/2 cons; oc, od: first elements of the a-c and a-d blocks of P
  template <class ET, class PT, class PU>
  __host__ __device__ static __forceinline__ void prim(const double (&F)[L + 1], double pref, double m2a, const double (&PQ)[3], const double (&QC)[3], const double (&QD)[3], double hk, double rc, double rd, const ET E, const PU Pab, const PT P, int n, int oc, int od, const double (&Dcd)[3], const double (&Dbc)[3], const double (&Dbd)[1], double& W, double (&gP)[3], double (&gR)[3], double (&gS)[3]) {
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
    const double r100_3 = PQ[0] * r000_4;
    const double r010_3 = PQ[1] * r000_4;
    const double r001_3 = PQ[2] * r000_4;
    const double r100_2 = PQ[0] * r000_3;
    const double r010_2 = PQ[1] * r000_3;
    const double r001_2 = PQ[2] * r000_3;
    const double r200_2 = fma(1.0, r000_3, PQ[0] * r100_3);
    const double r110_2 = PQ[0] * r010_3;
    const double r101_2 = PQ[0] * r001_3;
    const double r020_2 = fma(1.0, r000_3, PQ[1] * r010_3);
    const double r011_2 = PQ[1] * r001_3;
    const double r002_2 = fma(1.0, r000_3, PQ[2] * r001_3);
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
    const double kxe100 = QC[0];
    const double kxe101 = (-hk);
    const double kxd100 = rc;
    const double kye100 = QC[1];
    const double kye101 = (-hk);
    const double kyd100 = rc;
    const double kze100 = QC[2];
    const double kze101 = (-hk);
    const double kzd100 = rc;
    const double k0_0_000 = kxe100;
    const double k0_0_100 = kxe101;
    const double k1_0_000 = kye100;
    const double k1_0_010 = kye101;
    const double k2_0_000 = kze100;
    const double k2_0_001 = kze101;
    double K0_0_000 = 0.0;
    double K1_0_000 = 0.0;
    double K2_0_000 = 0.0;
    double w = 0.0, px = 0.0, py = 0.0, pz = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
    QF_OPAQUE(oc);
    QF_OPAQUE(od);
    {
      const double ac0 = P[oc + 0 * n + 0] * (kCons[2][0] * kCons[1][0]);
      const double ac1 = P[oc + 0 * n + 1] * (kCons[2][0] * kCons[1][1]);
      const double ac2 = P[oc + 0 * n + 2] * (kCons[2][0] * kCons[1][2]);
      const double ad0 = P[od + 0 * n + 0] * (kCons[2][0] * kCons[0][0]);
      {
        const double ab = Pab[0 * n + 0] * (kCons[2][0] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t101 = fma(y100, r201_0, fma(y010, r111_0, fma(y001, r102_0, y000 * r101_0)));
        const double t110 = fma(y100, r210_0, fma(y010, r120_0, fma(y001, r111_0, y000 * r110_0)));
        const double t200 = fma(y100, r300_0, fma(y010, r210_0, fma(y001, r201_0, y000 * r200_0)));
        const double t201 = fma(y100, r301_0, fma(y010, r211_0, fma(y001, r202_0, y000 * r201_0)));
        const double t210 = fma(y100, r310_0, fma(y010, r220_0, fma(y001, r211_0, y000 * r210_0)));
        const double t300 = fma(y100, r400_0, fma(y010, r310_0, fma(y001, r301_0, y000 * r300_0)));
        const double e0 = E[0];
        const double e1 = E[1];
        const double e2 = E[2];
        w = fma(e2, t200, fma(e1, t100, fma(e0, t000, w)));
        px = fma(e2, t300, fma(e1, t200, fma(e0, t100, px)));
        py = fma(e2, t210, fma(e1, t110, fma(e0, t010, py)));
        pz = fma(e2, t201, fma(e1, t101, fma(e0, t001, pz)));
        sx = fma(E[4], t100, fma(E[3], t000, sx));
        const double z000 = fma(e2, r200_0, fma(e1, r100_0, e0 * r000_0));
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    {
      const double ac0 = P[oc + 1 * n + 0] * (kCons[2][1] * kCons[1][0]);
      const double ac1 = P[oc + 1 * n + 1] * (kCons[2][1] * kCons[1][1]);
      const double ac2 = P[oc + 1 * n + 2] * (kCons[2][1] * kCons[1][2]);
      const double ad0 = P[od + 1 * n + 0] * (kCons[2][1] * kCons[0][0]);
      {
        const double ab = Pab[1 * n + 0] * (kCons[2][1] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t011 = fma(y100, r111_0, fma(y010, r021_0, fma(y001, r012_0, y000 * r011_0)));
        const double t020 = fma(y100, r120_0, fma(y010, r030_0, fma(y001, r021_0, y000 * r020_0)));
        const double t101 = fma(y100, r201_0, fma(y010, r111_0, fma(y001, r102_0, y000 * r101_0)));
        const double t110 = fma(y100, r210_0, fma(y010, r120_0, fma(y001, r111_0, y000 * r110_0)));
        const double t200 = fma(y100, r300_0, fma(y010, r210_0, fma(y001, r201_0, y000 * r200_0)));
        const double t111 = fma(y100, r211_0, fma(y010, r121_0, fma(y001, r112_0, y000 * r111_0)));
        const double t120 = fma(y100, r220_0, fma(y010, r130_0, fma(y001, r121_0, y000 * r120_0)));
        const double t210 = fma(y100, r310_0, fma(y010, r220_0, fma(y001, r211_0, y000 * r210_0)));
        const double e0 = E[5];
        const double e1 = E[6];
        const double e2 = E[7];
        const double e3 = E[8];
        w = fma(e3, t110, fma(e2, t100, fma(e1, t010, fma(e0, t000, w))));
        px = fma(e3, t210, fma(e2, t200, fma(e1, t110, fma(e0, t100, px))));
        py = fma(e3, t120, fma(e2, t110, fma(e1, t020, fma(e0, t010, py))));
        pz = fma(e3, t111, fma(e2, t101, fma(e1, t011, fma(e0, t001, pz))));
        sx = fma(E[10], t010, fma(E[9], t000, sx));
        sy = fma(E[12], t100, fma(E[11], t000, sy));
        const double z000 = fma(e3, r110_0, fma(e2, r100_0, fma(e1, r010_0, e0 * r000_0)));
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    {
      const double ac0 = P[oc + 2 * n + 0] * (kCons[2][2] * kCons[1][0]);
      const double ac1 = P[oc + 2 * n + 1] * (kCons[2][2] * kCons[1][1]);
      const double ac2 = P[oc + 2 * n + 2] * (kCons[2][2] * kCons[1][2]);
      const double ad0 = P[od + 2 * n + 0] * (kCons[2][2] * kCons[0][0]);
      {
        const double ab = Pab[2 * n + 0] * (kCons[2][2] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t011 = fma(y100, r111_0, fma(y010, r021_0, fma(y001, r012_0, y000 * r011_0)));
        const double t020 = fma(y100, r120_0, fma(y010, r030_0, fma(y001, r021_0, y000 * r020_0)));
        const double t110 = fma(y100, r210_0, fma(y010, r120_0, fma(y001, r111_0, y000 * r110_0)));
        const double t021 = fma(y100, r121_0, fma(y010, r031_0, fma(y001, r022_0, y000 * r021_0)));
        const double t030 = fma(y100, r130_0, fma(y010, r040_0, fma(y001, r031_0, y000 * r030_0)));
        const double t120 = fma(y100, r220_0, fma(y010, r130_0, fma(y001, r121_0, y000 * r120_0)));
        const double e0 = E[13];
        const double e1 = E[14];
        const double e2 = E[15];
        w = fma(e2, t020, fma(e1, t010, fma(e0, t000, w)));
        px = fma(e2, t120, fma(e1, t110, fma(e0, t100, px)));
        py = fma(e2, t030, fma(e1, t020, fma(e0, t010, py)));
        pz = fma(e2, t021, fma(e1, t011, fma(e0, t001, pz)));
        sy = fma(E[17], t010, fma(E[16], t000, sy));
        const double z000 = fma(e2, r020_0, fma(e1, r010_0, e0 * r000_0));
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    {
      const double ac0 = P[oc + 3 * n + 0] * (kCons[2][3] * kCons[1][0]);
      const double ac1 = P[oc + 3 * n + 1] * (kCons[2][3] * kCons[1][1]);
      const double ac2 = P[oc + 3 * n + 2] * (kCons[2][3] * kCons[1][2]);
      const double ad0 = P[od + 3 * n + 0] * (kCons[2][3] * kCons[0][0]);
      {
        const double ab = Pab[3 * n + 0] * (kCons[2][3] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t002 = fma(y100, r102_0, fma(y010, r012_0, fma(y001, r003_0, y000 * r002_0)));
        const double t011 = fma(y100, r111_0, fma(y010, r021_0, fma(y001, r012_0, y000 * r011_0)));
        const double t101 = fma(y100, r201_0, fma(y010, r111_0, fma(y001, r102_0, y000 * r101_0)));
        const double t110 = fma(y100, r210_0, fma(y010, r120_0, fma(y001, r111_0, y000 * r110_0)));
        const double t200 = fma(y100, r300_0, fma(y010, r210_0, fma(y001, r201_0, y000 * r200_0)));
        const double t102 = fma(y100, r202_0, fma(y010, r112_0, fma(y001, r103_0, y000 * r102_0)));
        const double t111 = fma(y100, r211_0, fma(y010, r121_0, fma(y001, r112_0, y000 * r111_0)));
        const double t201 = fma(y100, r301_0, fma(y010, r211_0, fma(y001, r202_0, y000 * r201_0)));
        const double e0 = E[18];
        const double e1 = E[19];
        const double e2 = E[20];
        const double e3 = E[21];
        w = fma(e3, t101, fma(e2, t100, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t201, fma(e2, t200, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t111, fma(e2, t110, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t102, fma(e2, t101, fma(e1, t002, fma(e0, t001, pz))));
        sx = fma(E[23], t001, fma(E[22], t000, sx));
        sz = fma(E[25], t100, fma(E[24], t000, sz));
        const double z000 = fma(e3, r101_0, fma(e2, r100_0, fma(e1, r001_0, e0 * r000_0)));
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    {
      const double ac0 = P[oc + 4 * n + 0] * (kCons[2][4] * kCons[1][0]);
      const double ac1 = P[oc + 4 * n + 1] * (kCons[2][4] * kCons[1][1]);
      const double ac2 = P[oc + 4 * n + 2] * (kCons[2][4] * kCons[1][2]);
      const double ad0 = P[od + 4 * n + 0] * (kCons[2][4] * kCons[0][0]);
      {
        const double ab = Pab[4 * n + 0] * (kCons[2][4] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t002 = fma(y100, r102_0, fma(y010, r012_0, fma(y001, r003_0, y000 * r002_0)));
        const double t011 = fma(y100, r111_0, fma(y010, r021_0, fma(y001, r012_0, y000 * r011_0)));
        const double t020 = fma(y100, r120_0, fma(y010, r030_0, fma(y001, r021_0, y000 * r020_0)));
        const double t101 = fma(y100, r201_0, fma(y010, r111_0, fma(y001, r102_0, y000 * r101_0)));
        const double t110 = fma(y100, r210_0, fma(y010, r120_0, fma(y001, r111_0, y000 * r110_0)));
        const double t012 = fma(y100, r112_0, fma(y010, r022_0, fma(y001, r013_0, y000 * r012_0)));
        const double t021 = fma(y100, r121_0, fma(y010, r031_0, fma(y001, r022_0, y000 * r021_0)));
        const double t111 = fma(y100, r211_0, fma(y010, r121_0, fma(y001, r112_0, y000 * r111_0)));
        const double e0 = E[26];
        const double e1 = E[27];
        const double e2 = E[28];
        const double e3 = E[29];
        w = fma(e3, t011, fma(e2, t010, fma(e1, t001, fma(e0, t000, w))));
        px = fma(e3, t111, fma(e2, t110, fma(e1, t101, fma(e0, t100, px))));
        py = fma(e3, t021, fma(e2, t020, fma(e1, t011, fma(e0, t010, py))));
        pz = fma(e3, t012, fma(e2, t011, fma(e1, t002, fma(e0, t001, pz))));
        sy = fma(E[31], t001, fma(E[30], t000, sy));
        sz = fma(E[33], t010, fma(E[32], t000, sz));
        const double z000 = fma(e3, r011_0, fma(e2, r010_0, fma(e1, r001_0, e0 * r000_0)));
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    {
      const double ac0 = P[oc + 5 * n + 0] * (kCons[2][5] * kCons[1][0]);
      const double ac1 = P[oc + 5 * n + 1] * (kCons[2][5] * kCons[1][1]);
      const double ac2 = P[oc + 5 * n + 2] * (kCons[2][5] * kCons[1][2]);
      const double ad0 = P[od + 5 * n + 0] * (kCons[2][5] * kCons[0][0]);
      {
        const double ab = Pab[5 * n + 0] * (kCons[2][5] * kCons[0][0]);
        const double g0_0 = fma(-ad0, Dbc[0], fma(-ac0, Dbd[0], ab * Dcd[0]));
        const double g1_0 = fma(-ad0, Dbc[1], fma(-ac1, Dbd[0], ab * Dcd[1]));
        const double g2_0 = fma(-ad0, Dbc[2], fma(-ac2, Dbd[0], ab * Dcd[2]));
        const double y000 = fma(k2_0_000, g2_0, fma(k1_0_000, g1_0, k0_0_000 * g0_0));
        const double y001 = k2_0_001 * g2_0;
        const double y010 = k1_0_010 * g1_0;
        const double y100 = k0_0_100 * g0_0;
        const double t000 = fma(y100, r100_0, fma(y010, r010_0, fma(y001, r001_0, y000 * r000_0)));
        const double t001 = fma(y100, r101_0, fma(y010, r011_0, fma(y001, r002_0, y000 * r001_0)));
        const double t010 = fma(y100, r110_0, fma(y010, r020_0, fma(y001, r011_0, y000 * r010_0)));
        const double t100 = fma(y100, r200_0, fma(y010, r110_0, fma(y001, r101_0, y000 * r100_0)));
        const double t002 = fma(y100, r102_0, fma(y010, r012_0, fma(y001, r003_0, y000 * r002_0)));
        const double t011 = fma(y100, r111_0, fma(y010, r021_0, fma(y001, r012_0, y000 * r011_0)));
        const double t101 = fma(y100, r201_0, fma(y010, r111_0, fma(y001, r102_0, y000 * r101_0)));
        const double t003 = fma(y100, r103_0, fma(y010, r013_0, fma(y001, r004_0, y000 * r003_0)));
        const double t012 = fma(y100, r112_0, fma(y010, r022_0, fma(y001, r013_0, y000 * r012_0)));
        const double t102 = fma(y100, r202_0, fma(y010, r112_0, fma(y001, r103_0, y000 * r102_0)));
        const double e0 = E[34];
        const double e1 = E[35];
        const double e2 = E[36];
        w = fma(e2, t002, fma(e1, t001, fma(e0, t000, w)));
        px = fma(e2, t102, fma(e1, t101, fma(e0, t100, px)));
        py = fma(e2, t012, fma(e1, t011, fma(e0, t010, py)));
        pz = fma(e2, t003, fma(e1, t002, fma(e0, t001, pz)));
        sz = fma(E[38], t001, fma(E[37], t000, sz));
        const double z000 = fma(e2, r002_0, fma(e1, r001_0, e0 * r000_0));
        K0_0_000 = fma(g0_0, z000, K0_0_000);
        K1_0_000 = fma(g1_0, z000, K1_0_000);
        K2_0_000 = fma(g2_0, z000, K2_0_000);
      }
    }
    W = w;
    gP[0] = px; gP[1] = py; gP[2] = pz;
    gR[0] = sx; gR[1] = sy; gR[2] = sz;
    gS[0] = kxd100 * K0_0_000;
    gS[1] = kyd100 * K1_0_000;
    gS[2] = kzd100 * K2_0_000;
  }
};
__device__ const unsigned kC2010GradMd_index[39] = {4,5,6,7,8,257,513,258,514,259,515,769,770,1024,1280,1536,1792,2048,65537,131073,65538,131074,65539,131075,196609,196610,65792,131328,66048,131584,66304,131840,196864,197120,262144,327680,393216,458752,524288};
__device__ inline const unsigned* C2010GradMd::index() { return kC2010GradMd_index; }
}  // namespace qf
