// Generated by nrpy_amd/codegen/hip_gen.py -- do not edit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "../bhah_device_types.h"
// ---- adjoint of the BSSN step: Spherical, symmetry axes '2', fd_order=4; 210 adjoint slots
#define Rational_1_2 (1.0 / 2.0)
#define Rational_1_3 (1.0 / 3.0)
#define Rational_1_4 (1.0 / 4.0)
#define Rational_2_3 (2.0 / 3.0)
#define Rational_3_2 (3.0 / 2.0)
#define Rational_3_4 (3.0 / 4.0)
#define Rational_4_3 (4.0 / 3.0)
#define Rational_8_3 (8.0 / 3.0)
#define Rational_m1_2 (-1.0 / 2.0)
#define Rational_m1_3 (-1.0 / 3.0)
#define Rational_m2_3 (-2.0 / 3.0)
#define Rational_m8_3 (-8.0 / 3.0)

// 3 output groups, one wave each over the same 64 points; 261 LDS rows of partial sums
extern "C" __global__ void __launch_bounds__(192)
adj_rhs_Spherical_sym2_KO0_fd4(const double *__restrict__ in, const double *__restrict__ aux, const double *__restrict__ lam,
    double *__restrict__ S, const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  __shared__ double red[261 * 64];
  const int lane = (int)threadIdx.x, group = (int)threadIdx.y;
  const int i0r = p.NG + (int)blockIdx.x * 64 + lane;
  const bool active = i0r < p.Nx0 - p.NG;
  const int i0 = active ? i0r : p.Nx0 - p.NG - 1;  // idle lanes repeat the row's last point
  const int i1 = p.NG + (int)blockIdx.y;
  const int i2 = p.NG + (int)blockIdx.z;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;
  const double up_f0_of_xx0 = rfm0[i0];
  const double up_f1_of_xx1 = rfm1[i1];
  const double up_vetU0 = in[21 * Ntot + idx];
  const double up_vetU1 = in[22 * Ntot + idx];
  const double up_vetU2 = in[23 * Ntot + idx];
  const double betaU0 = up_vetU0;
  const double betaU1 = up_vetU1/up_f0_of_xx0;
  const double betaU2 = up_vetU2/(up_f0_of_xx0*up_f1_of_xx1);
  double uw0[7];
  uw0[0] = (betaU0 > 0.0) ? 0.0 : (-1.0 / 12.0);
  uw0[1] = (betaU0 > 0.0) ? 0.0 : (1.0 / 2.0);
  uw0[2] = (betaU0 > 0.0) ? (-1.0 / 4.0) : (-3.0 / 2.0);
  uw0[3] = (betaU0 > 0.0) ? (-5.0 / 6.0) : (5.0 / 6.0);
  uw0[4] = (betaU0 > 0.0) ? (3.0 / 2.0) : (1.0 / 4.0);
  uw0[5] = (betaU0 > 0.0) ? (-1.0 / 2.0) : 0.0;
  uw0[6] = (betaU0 > 0.0) ? (1.0 / 12.0) : 0.0;
  double uw1[7];
  uw1[0] = (betaU1 > 0.0) ? 0.0 : (-1.0 / 12.0);
  uw1[1] = (betaU1 > 0.0) ? 0.0 : (1.0 / 2.0);
  uw1[2] = (betaU1 > 0.0) ? (-1.0 / 4.0) : (-3.0 / 2.0);
  uw1[3] = (betaU1 > 0.0) ? (-5.0 / 6.0) : (5.0 / 6.0);
  uw1[4] = (betaU1 > 0.0) ? (3.0 / 2.0) : (1.0 / 4.0);
  uw1[5] = (betaU1 > 0.0) ? (-1.0 / 2.0) : 0.0;
  uw1[6] = (betaU1 > 0.0) ? (1.0 / 12.0) : 0.0;
  double uw2[7];
  uw2[0] = (betaU2 > 0.0) ? 0.0 : (-1.0 / 12.0);
  uw2[1] = (betaU2 > 0.0) ? 0.0 : (1.0 / 2.0);
  uw2[2] = (betaU2 > 0.0) ? (-1.0 / 4.0) : (-3.0 / 2.0);
  uw2[3] = (betaU2 > 0.0) ? (-5.0 / 6.0) : (5.0 / 6.0);
  uw2[4] = (betaU2 > 0.0) ? (3.0 / 2.0) : (1.0 / 4.0);
  uw2[5] = (betaU2 > 0.0) ? (-1.0 / 2.0) : 0.0;
  uw2[6] = (betaU2 > 0.0) ? (1.0 / 12.0) : 0.0;
  switch (group) {
  case 0: { // betU0, betU1, betU2
  const double aDD00 = in[idx];
  const double aDD01 = in[1 * Ntot + idx];
  const double aDD02 = in[2 * Ntot + idx];
  const double aDD11 = in[3 * Ntot + idx];
  const double aDD12 = in[4 * Ntot + idx];
  const double aDD22 = in[5 * Ntot + idx];
  const double alpha = in[6 * Ntot + idx];
  const double alpha_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[6 * Ntot + idx + (1)] - in[6 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2)] - in[6 * Ntot + idx + (-2)]));
  const double alpha_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[6 * Ntot + idx + (1 * s1)] - in[6 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2 * s1)] - in[6 * Ntot + idx + (-2 * s1)]));
  const double betU0 = in[7 * Ntot + idx];
  const double betU1 = in[8 * Ntot + idx];
  const double betU2 = in[9 * Ntot + idx];
  const double betU_dupD00 = p.invdxx0 * (uw0[0] * in[7 * Ntot + idx + (-3)] + uw0[1] * in[7 * Ntot + idx + (-2)] + uw0[2] * in[7 * Ntot + idx + (-1)] + uw0[3] * in[7 * Ntot + idx] + uw0[4] * in[7 * Ntot + idx + (1)] + uw0[5] * in[7 * Ntot + idx + (2)] + uw0[6] * in[7 * Ntot + idx + (3)]);
  const double betU_dupD01 = p.invdxx1 * (uw1[0] * in[7 * Ntot + idx + (-3 * s1)] + uw1[1] * in[7 * Ntot + idx + (-2 * s1)] + uw1[2] * in[7 * Ntot + idx + (-1 * s1)] + uw1[3] * in[7 * Ntot + idx] + uw1[4] * in[7 * Ntot + idx + (1 * s1)] + uw1[5] * in[7 * Ntot + idx + (2 * s1)] + uw1[6] * in[7 * Ntot + idx + (3 * s1)]);
  const double betU_dupD10 = p.invdxx0 * (uw0[0] * in[8 * Ntot + idx + (-3)] + uw0[1] * in[8 * Ntot + idx + (-2)] + uw0[2] * in[8 * Ntot + idx + (-1)] + uw0[3] * in[8 * Ntot + idx] + uw0[4] * in[8 * Ntot + idx + (1)] + uw0[5] * in[8 * Ntot + idx + (2)] + uw0[6] * in[8 * Ntot + idx + (3)]);
  const double betU_dupD11 = p.invdxx1 * (uw1[0] * in[8 * Ntot + idx + (-3 * s1)] + uw1[1] * in[8 * Ntot + idx + (-2 * s1)] + uw1[2] * in[8 * Ntot + idx + (-1 * s1)] + uw1[3] * in[8 * Ntot + idx] + uw1[4] * in[8 * Ntot + idx + (1 * s1)] + uw1[5] * in[8 * Ntot + idx + (2 * s1)] + uw1[6] * in[8 * Ntot + idx + (3 * s1)]);
  const double betU_dupD20 = p.invdxx0 * (uw0[0] * in[9 * Ntot + idx + (-3)] + uw0[1] * in[9 * Ntot + idx + (-2)] + uw0[2] * in[9 * Ntot + idx + (-1)] + uw0[3] * in[9 * Ntot + idx] + uw0[4] * in[9 * Ntot + idx + (1)] + uw0[5] * in[9 * Ntot + idx + (2)] + uw0[6] * in[9 * Ntot + idx + (3)]);
  const double betU_dupD21 = p.invdxx1 * (uw1[0] * in[9 * Ntot + idx + (-3 * s1)] + uw1[1] * in[9 * Ntot + idx + (-2 * s1)] + uw1[2] * in[9 * Ntot + idx + (-1 * s1)] + uw1[3] * in[9 * Ntot + idx] + uw1[4] * in[9 * Ntot + idx + (1 * s1)] + uw1[5] * in[9 * Ntot + idx + (2 * s1)] + uw1[6] * in[9 * Ntot + idx + (3 * s1)]);
  const double cf = in[10 * Ntot + idx];
  const double cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1)] - in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] - in[10 * Ntot + idx + (-2)]));
  const double cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] - in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] - in[10 * Ntot + idx + (-2 * s1)]));
  const double eta = p.eta;
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double hDD00 = in[11 * Ntot + idx];
  const double hDD01 = in[12 * Ntot + idx];
  const double hDD02 = in[13 * Ntot + idx];
  const double hDD11 = in[14 * Ntot + idx];
  const double hDD12 = in[15 * Ntot + idx];
  const double hDD22 = in[16 * Ntot + idx];
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  const double lambdaU0 = in[17 * Ntot + idx];
  const double lambdaU1 = in[18 * Ntot + idx];
  const double lambdaU2 = in[19 * Ntot + idx];
  const double trK_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1)] - in[20 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2)] - in[20 * Ntot + idx + (-2)]));
  const double trK_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1 * s1)] - in[20 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2 * s1)] - in[20 * Ntot + idx + (-2 * s1)]));
  const double vetU0 = in[21 * Ntot + idx];
  const double vetU1 = in[22 * Ntot + idx];
  const double vetU2 = in[23 * Ntot + idx];
  const double vetU_dD00 = p.invdxx0 * ((2.0 / 3.0) * (in[21 * Ntot + idx + (1)] - in[21 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2)] - in[21 * Ntot + idx + (-2)]));
  const double vetU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (in[21 * Ntot + idx + (1 * s1)] - in[21 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2 * s1)] - in[21 * Ntot + idx + (-2 * s1)]));
  const double vetU_dD10 = p.invdxx0 * ((2.0 / 3.0) * (in[22 * Ntot + idx + (1)] - in[22 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2)] - in[22 * Ntot + idx + (-2)]));
  const double vetU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (in[22 * Ntot + idx + (1 * s1)] - in[22 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2 * s1)] - in[22 * Ntot + idx + (-2 * s1)]));
  const double vetU_dD20 = p.invdxx0 * ((2.0 / 3.0) * (in[23 * Ntot + idx + (1)] - in[23 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2)] - in[23 * Ntot + idx + (-2)]));
  const double vetU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (in[23 * Ntot + idx + (1 * s1)] - in[23 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2 * s1)] - in[23 * Ntot + idx + (-2 * s1)]));
  const double vetU_dDD000 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[21 * Ntot + idx] + (4.0 / 3.0) * (in[21 * Ntot + idx + (1)] + in[21 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2)] + in[21 * Ntot + idx + (-2)]));
  const double vetU_dDD001 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[21 * Ntot + idx + (1 + 1 * s1)] - in[21 * Ntot + idx + (1 + -1 * s1)]) - (in[21 * Ntot + idx + (-1 + 1 * s1)] - in[21 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[21 * Ntot + idx + (1 + 2 * s1)] - in[21 * Ntot + idx + (1 + -2 * s1)]) - (in[21 * Ntot + idx + (-1 + 2 * s1)] - in[21 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[21 * Ntot + idx + (2 + 1 * s1)] - in[21 * Ntot + idx + (2 + -1 * s1)]) - (in[21 * Ntot + idx + (-2 + 1 * s1)] - in[21 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[21 * Ntot + idx + (2 + 2 * s1)] - in[21 * Ntot + idx + (2 + -2 * s1)]) - (in[21 * Ntot + idx + (-2 + 2 * s1)] - in[21 * Ntot + idx + (-2 + -2 * s1)])));
  const double vetU_dDD011 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[21 * Ntot + idx] + (4.0 / 3.0) * (in[21 * Ntot + idx + (1 * s1)] + in[21 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2 * s1)] + in[21 * Ntot + idx + (-2 * s1)]));
  const double vetU_dDD100 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[22 * Ntot + idx] + (4.0 / 3.0) * (in[22 * Ntot + idx + (1)] + in[22 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2)] + in[22 * Ntot + idx + (-2)]));
  const double vetU_dDD101 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[22 * Ntot + idx + (1 + 1 * s1)] - in[22 * Ntot + idx + (1 + -1 * s1)]) - (in[22 * Ntot + idx + (-1 + 1 * s1)] - in[22 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[22 * Ntot + idx + (1 + 2 * s1)] - in[22 * Ntot + idx + (1 + -2 * s1)]) - (in[22 * Ntot + idx + (-1 + 2 * s1)] - in[22 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[22 * Ntot + idx + (2 + 1 * s1)] - in[22 * Ntot + idx + (2 + -1 * s1)]) - (in[22 * Ntot + idx + (-2 + 1 * s1)] - in[22 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[22 * Ntot + idx + (2 + 2 * s1)] - in[22 * Ntot + idx + (2 + -2 * s1)]) - (in[22 * Ntot + idx + (-2 + 2 * s1)] - in[22 * Ntot + idx + (-2 + -2 * s1)])));
  const double vetU_dDD111 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[22 * Ntot + idx] + (4.0 / 3.0) * (in[22 * Ntot + idx + (1 * s1)] + in[22 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2 * s1)] + in[22 * Ntot + idx + (-2 * s1)]));
  const double vetU_dDD200 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[23 * Ntot + idx] + (4.0 / 3.0) * (in[23 * Ntot + idx + (1)] + in[23 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2)] + in[23 * Ntot + idx + (-2)]));
  const double vetU_dDD201 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[23 * Ntot + idx + (1 + 1 * s1)] - in[23 * Ntot + idx + (1 + -1 * s1)]) - (in[23 * Ntot + idx + (-1 + 1 * s1)] - in[23 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[23 * Ntot + idx + (1 + 2 * s1)] - in[23 * Ntot + idx + (1 + -2 * s1)]) - (in[23 * Ntot + idx + (-1 + 2 * s1)] - in[23 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[23 * Ntot + idx + (2 + 1 * s1)] - in[23 * Ntot + idx + (2 + -1 * s1)]) - (in[23 * Ntot + idx + (-2 + 1 * s1)] - in[23 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[23 * Ntot + idx + (2 + 2 * s1)] - in[23 * Ntot + idx + (2 + -2 * s1)]) - (in[23 * Ntot + idx + (-2 + 2 * s1)] - in[23 * Ntot + idx + (-2 + -2 * s1)])));
  const double vetU_dDD211 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[23 * Ntot + idx] + (4.0 / 3.0) * (in[23 * Ntot + idx + (1 * s1)] + in[23 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2 * s1)] + in[23 * Ntot + idx + (-2 * s1)]));
  const double g0t0 = (Rational_3_4)*lambdaU0;
  const double g0t1 = (f0_of_xx0*f0_of_xx0);
  const double g0t2 = g0t1*hDD11 + g0t1;
  const double g0t3 = (f1_of_xx1*f1_of_xx1);
  const double g0t4 = g0t1*g0t3;
  const double g0t5 = g0t4*hDD22 + g0t4;
  const double g0t6 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g0t7 = g0t3*g0t6*(hDD12*hDD12);
  const double g0t8 = g0t2*g0t5 - g0t7;
  const double g0t9 = g0t1*(hDD01*hDD01);
  const double g0t10 = hDD00 + 1.0;
  const double g0t11 = g0t4*(hDD02*hDD02);
  const double g0t12 = g0t10*g0t2*g0t5 - g0t10*g0t7 - g0t11*g0t2 + 2.0*g0t3*g0t6*hDD01*hDD02*hDD12 - g0t5*g0t9;
  const double g0t13 = (1.0 / (g0t12*g0t12));
  const double g0t14 = aDD00*g0t13;
  const double g0t15 = g0t14*(g0t8*g0t8);
  const double g0t16 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g0t17 = g0t16*hDD12;
  const double g0t18 = -f0_of_xx0*g0t5*hDD01 + g0t17*g0t3*hDD02;
  const double g0t19 = (g0t18*g0t18);
  const double g0t20 = g0t13*g0t19;
  const double g0t21 = 2.0*g0t1;
  const double g0t22 = aDD11*g0t21;
  const double g0t23 = f1_of_xx1*hDD02;
  const double g0t24 = -f0_of_xx0*g0t2*g0t23 + f1_of_xx1*g0t17*hDD01;
  const double g0t25 = (g0t24*g0t24);
  const double g0t26 = g0t13*g0t25;
  const double g0t27 = aDD22*g0t4;
  const double g0t28 = g0t26*g0t27;
  const double g0t29 = g0t18*g0t8;
  const double g0t30 = aDD01*f0_of_xx0;
  const double g0t31 = g0t13*g0t30;
  const double g0t32 = g0t24*g0t8;
  const double g0t33 = f0_of_xx0*f1_of_xx1;
  const double g0t34 = aDD02*g0t33;
  const double g0t35 = g0t13*g0t34;
  const double g0t36 = 4.0*g0t35;
  const double g0t37 = g0t18*g0t24;
  const double g0t38 = f1_of_xx1*g0t1;
  const double g0t39 = aDD12*g0t38;
  const double g0t40 = g0t13*g0t39;
  const double g0t41 = 3.0*alpha;
  const double g0t42 = g0t41/cf;
  const double g0t43 = (Rational_3_4)*alpha_dD0 + (Rational_3_4)*cf_dD0*g0t42;
  const double g0t44 = g0t14*g0t29;
  const double g0t45 = 2.0*f0_of_xx0;
  const double g0t46 = aDD01*g0t20;
  const double g0t47 = g0t10*g0t5 - g0t11;
  const double g0t48 = g0t13*g0t47;
  const double g0t49 = g0t48*g0t8;
  const double g0t50 = aDD01*g0t45;
  const double g0t51 = g0t18*g0t48;
  const double g0t52 = g0t1*g0t23*hDD01 - g0t10*g0t38*hDD12;
  const double g0t53 = g0t52*g0t8;
  const double g0t54 = f1_of_xx1*g0t45;
  const double g0t55 = aDD02*g0t54;
  const double g0t56 = g0t13*g0t55;
  const double g0t57 = g0t24*g0t48;
  const double g0t58 = 2.0*g0t38;
  const double g0t59 = aDD12*g0t58;
  const double g0t60 = g0t18*g0t52;
  const double g0t61 = g0t13*g0t59;
  const double g0t62 = g0t13*g0t27;
  const double g0t63 = g0t24*g0t52;
  const double g0t64 = g0t62*g0t63;
  const double g0t65 = -g0t22*g0t51 - g0t37*g0t56 - 2.0*g0t44 - g0t45*g0t46 - g0t49*g0t50 - g0t53*g0t56 - g0t57*g0t59 - g0t60*g0t61 - 2.0*g0t64;
  const double g0t66 = (Rational_3_4)*alpha_dD1 + (Rational_3_4)*cf_dD1*g0t42;
  const double g0t67 = f0_of_xx0*g0t3;
  const double g0t68 = 2.0*g0t67;
  const double g0t69 = g0t4*hDD_dD220 + g0t68*hDD22 + g0t68;
  const double g0t70 = -g0t69;
  const double g0t71 = (1.0 / g0t12);
  const double g0t72 = (Rational_1_2)*g0t71;
  const double g0t73 = g0t72*g0t8;
  const double g0t74 = f1_of_xx1*f1_of_xx1__D1;
  const double g0t75 = g0t21*g0t74;
  const double g0t76 = g0t4*hDD_dD221 + g0t75*hDD22 + g0t75;
  const double g0t77 = -g0t76;
  const double g0t78 = g0t18*g0t72;
  const double g0t79 = g0t70*g0t73 + g0t77*g0t78;
  const double g0t80 = g0t67 + g0t79;
  const double g0t81 = g0t10*g0t2 - g0t9;
  const double g0t82 = (Rational_2_3)*g0t71;
  const double g0t83 = g0t81*g0t82;
  const double g0t84 = g0t1*hDD_dD110 + g0t45*hDD11 + g0t45;
  const double g0t85 = 2.0*f0_of_xx0*hDD_dD011 - g0t84;
  const double g0t86 = f1_of_xx1__D1*g0t21*hDD12 + g0t58*hDD_dD121;
  const double g0t87 = g0t24*g0t72;
  const double g0t88 = g0t1*hDD_dD111;
  const double g0t89 = g0t73*g0t85 + g0t78*g0t88 + g0t86*g0t87;
  const double g0t90 = f0_of_xx0 + g0t89;
  const double g0t91 = g0t47*g0t82;
  const double g0t92 = 2.0*g0t23 + g0t54*hDD_dD020;
  const double g0t93 = g0t45*hDD_dD010 + 2.0*hDD01 - hDD_dD001;
  const double g0t94 = g0t73*hDD_dD000 + g0t78*g0t93 + g0t87*g0t92;
  const double g0t95 = g0t8*g0t82;
  const double g0t96 = g0t38*hDD_dD120 + g0t54*hDD12;
  const double g0t97 = -f0_of_xx0*f1_of_xx1*hDD_dD021 - f0_of_xx0*f1_of_xx1__D1*hDD02 + g0t96;
  const double g0t98 = -g0t97;
  const double g0t99 = g0t73*g0t98 + g0t76*g0t87;
  const double g0t100 = (Rational_4_3)*g0t71;
  const double g0t101 = g0t100*g0t52;
  const double g0t102 = g0t69*g0t87 + g0t78*g0t97;
  const double g0t103 = g0t100*g0t24;
  const double g0t104 = f0_of_xx0*f1_of_xx1__D1*hDD02 + g0t33*hDD_dD021 + g0t96;
  const double g0t105 = g0t104*g0t87 + g0t73*hDD_dD001 + g0t78*g0t84;
  const double g0t106 = g0t100*g0t18;
  const double g0t107 = (1.0 / f0_of_xx0);
  const double g0t108 = g0t107*vetU_dD11;
  const double g0t109 = 2.0*g0t107;
  const double g0t110 = (1.0 / f1_of_xx1);
  const double g0t111 = f1_of_xx1__D1*g0t110;
  const double g0t112 = g0t107*vetU1;
  const double g0t113 = (Rational_3_4)*g0t108 + (Rational_3_4)*g0t109*vetU0 + (Rational_3_4)*g0t111*g0t112 + (Rational_3_4)*vetU_dD00;
  const double g0t114 = betU0*vetU0;
  const double g0t115 = g0t14*g0t24;
  const double g0t116 = g0t115*g0t18;
  const double g0t117 = aDD11*g0t1;
  const double g0t118 = g0t117*g0t13;
  const double g0t119 = g0t118*g0t47;
  const double g0t120 = g0t13*(g0t52*g0t52);
  const double g0t121 = g0t35*g0t81;
  const double g0t122 = g0t39*g0t81;
  const double g0t123 = g0t62*g0t81;
  const double g0t124 = g0t123*g0t52;
  const double g0t125 = g0t41*(g0t116 + g0t119*g0t52 + g0t120*g0t39 + g0t121*g0t18 + g0t122*g0t48 + g0t124 + g0t30*g0t57 + g0t31*g0t60 + g0t35*g0t63);
  const double g0t126 = g0t115*g0t8;
  const double g0t127 = g0t13*g0t18;
  const double g0t128 = g0t123*g0t24;
  const double g0t129 = g0t41*(g0t118*g0t60 + g0t121*g0t8 + g0t122*g0t127 + g0t126 + g0t128 + g0t26*g0t34 + g0t31*g0t37 + g0t31*g0t53 + g0t40*g0t63);
  const double g0t130 = g0t41*(f0_of_xx0*g0t46 + g0t119*g0t18 + g0t30*g0t49 + g0t35*g0t37 + g0t35*g0t53 + g0t39*g0t57 + g0t40*g0t60 + g0t44 + g0t64);
  const double g0t131 = g0t0*vetU0;
  const double g0t132 = g0t107*vetU_dD01;
  const double g0t133 = (Rational_3_4)*lambdaU1;
  const double g0t134 = (1.0 / g0t1);
  const double g0t135 = g0t134*vetU0;
  const double g0t136 = 4.0*g0t16*g0t3;
  const double g0t137 = (1.0 / g0t3);
  const double g0t138 = (Rational_1_2)*g0t137/g0t6;
  const double g0t139 = g0t134*vetU1;
  const double g0t140 = g0t107*vetU_dD10 - g0t139;
  const double g0t141 = 2.0*g0t6;
  const double g0t142 = 8.0*g0t74;
  const double g0t143 = 4.0*g0t111;
  const double g0t144 = g0t134*vetU_dD11;
  const double g0t145 = g0t107*vetU_dDD101 - g0t144;
  const double g0t146 = (Rational_1_4)*g0t71;
  const double g0t147 = g0t146*(-8.0*g0t135 + g0t138*(g0t136*vetU_dD00 + 12.0*g0t4*vetU0) + g0t138*(g0t1*g0t142*vetU1 + g0t140*g0t141*g0t74) - g0t139*g0t143 + g0t145 + vetU_dDD000);
  const double g0t148 = g0t107*vetU_dDD111;
  const double g0t149 = (f1_of_xx1__D1*f1_of_xx1__D1);
  const double g0t150 = f1_of_xx1*f1_of_xx1__DD11;
  const double g0t151 = 2.0*vetU_dD11;
  const double g0t152 = g0t137*g0t149;
  const double g0t153 = g0t112*g0t152;
  const double g0t154 = g0t146*(-g0t107*g0t143*vetU0 + g0t138*(g0t112*(g0t141*g0t149 + g0t141*g0t150) + g0t151*g0t16*g0t74) + g0t138*(g0t136*vetU_dD01 + g0t142*g0t16*vetU0) + g0t148 - 2.0*g0t153 + vetU_dDD001);
  const double g0t155 = g0t13*g0t50;
  const double g0t156 = g0t56*g0t81;
  const double g0t157 = (Rational_3_2)*alpha;
  const double g0t158 = g0t157*(g0t117*g0t120 + g0t14*g0t25 + g0t155*g0t63 + g0t156*g0t24 + g0t52*g0t61*g0t81 + g0t62*(g0t81*g0t81));
  const double g0t159 = g0t157*(g0t117*g0t20 + g0t15 + g0t155*g0t29 + g0t28 + g0t32*g0t56 + g0t37*g0t61);
  const double g0t160 = g0t14*g0t19;
  const double g0t161 = (g0t47*g0t47);
  const double g0t162 = g0t120*g0t27;
  const double g0t163 = g0t48*g0t52;
  const double g0t164 = g0t157*(g0t118*g0t161 + g0t160 + g0t162 + g0t163*g0t59 + g0t50*g0t51 + g0t56*g0t60);
  const double g0t165 = f0_of_xx0*g0t140;
  const double g0t166 = g0t18*g0t71;
  const double g0t167 = (Rational_3_2)*g0t166;
  const double g0t168 = (Rational_3_4)*g0t71;
  const double g0t169 = g0t168*g0t8;
  const double g0t170 = 2.0*vetU1;
  const double g0t171 = g0t168*g0t81;
  const double g0t172 = g0t168*g0t47;
  const double g0t173 = betU0*g0t112;
  const double g0t174 = betU1*g0t107;
  const double g0t175 = g0t174*vetU0;
  const double g0t176 = betU1*g0t139;
  const double g0t177 = alpha*trK_dD0;
  const double g0t178 = g0t177*g0t71;
  const double g0t179 = alpha*trK_dD1;
  const double g0t180 = g0t0*g0t112;
  const double g0t181 = g0t107*g0t133;
  const double g0t182 = g0t181*vetU0;
  const double g0t183 = g0t133*g0t139;
  const double g0t184 = g0t107*g0t110;
  const double g0t185 = g0t184*vetU2;
  const double g0t186 = betU0*g0t185;
  const double g0t187 = betU1*g0t134;
  const double g0t188 = g0t110*vetU2;
  const double g0t189 = g0t187*g0t188;
  const double g0t190 = betU2*g0t184;
  const double g0t191 = g0t190*vetU0;
  const double g0t192 = g0t110*g0t139;
  const double g0t193 = betU2*g0t192;
  const double g0t194 = g0t134*vetU2;
  const double g0t195 = g0t137*g0t194;
  const double g0t196 = betU2*g0t195;
  const double g0t197 = g0t110*g0t134;
  const double g0t198 = g0t197*vetU2;
  const double g0t199 = g0t184*vetU_dD20 - g0t198;
  const double g0t200 = g0t199*g0t67;
  const double g0t201 = (Rational_3_2)*g0t71;
  const double g0t202 = g0t201*g0t24;
  const double g0t203 = g0t107*vetU2;
  const double g0t204 = f1_of_xx1__D1*g0t137;
  const double g0t205 = g0t184*vetU_dD21 - g0t203*g0t204;
  const double g0t206 = g0t0*g0t185;
  const double g0t207 = g0t133*g0t198;
  const double g0t208 = (Rational_3_4)*lambdaU2;
  const double g0t209 = g0t184*g0t208*vetU0;
  const double g0t210 = g0t192*g0t208;
  const double g0t211 = g0t195*g0t208;
  const double g0t212 = g0t13*g0t22;
  const double g0t213 = g0t47*g0t72;
  const double g0t214 = g0t213*g0t77 + g0t70*g0t78;
  const double g0t215 = g0t214 + g0t74;
  const double g0t216 = g0t52*g0t72;
  const double g0t217 = g0t213*g0t88 + g0t216*g0t86 + g0t78*g0t85;
  const double g0t218 = g0t213*g0t93 + g0t216*g0t92 + g0t78*hDD_dD000;
  const double g0t219 = g0t213*g0t97 + g0t216*g0t69;
  const double g0t220 = g0t216*g0t76 + g0t78*g0t98;
  const double g0t221 = -g0t107;
  const double g0t222 = g0t104*g0t216 + g0t213*g0t84 + g0t78*hDD_dD001;
  const double g0t223 = g0t221 + g0t222;
  const double g0t224 = g0t107*vetU_dD00 - g0t135;
  const double g0t225 = (1.0 / g0t16);
  const double g0t226 = g0t205*g0t74;
  const double g0t227 = g0t168*g0t52;
  const double g0t228 = g0t179*g0t71;
  const double g0t229 = g0t127*g0t81;
  const double g0t230 = g0t216*g0t77 + g0t70*g0t87;
  const double g0t231 = g0t72*g0t81;
  const double g0t232 = g0t216*g0t88 + g0t231*g0t86 + g0t85*g0t87;
  const double g0t233 = g0t216*g0t93 + g0t231*g0t92 + g0t87*hDD_dD000;
  const double g0t234 = g0t104*g0t231 + g0t216*g0t84 + g0t87*hDD_dD001;
  const double g0t235 = g0t231*g0t76 + g0t87*g0t98;
  const double g0t236 = -g0t111 + g0t235;
  const double g0t237 = g0t216*g0t97 + g0t231*g0t69;
  const double g0t238 = g0t221 + g0t237;
  const double g0t239 = g0t107*g0t137;
  const double g0t240 = f1_of_xx1__D1*g0t239;
  const double g0t241 = (1.0 / (f1_of_xx1*f1_of_xx1*f1_of_xx1));
  const double g0t242 = f1_of_xx1__DD11*g0t110 - g0t152;
  double a_betU0 = lam[7 * Ntot + idx] * (-eta);
  double a_betU_dupD00 = lam[7 * Ntot + idx] * (vetU0);
  double a_betU_dupD01 = lam[7 * Ntot + idx] * (g0t112);
  double a_eta = lam[7 * Ntot + idx] * (-betU0);
  double a_f0_of_xx0 = lam[7 * Ntot + idx] * (g0t172*vetU_dD00);
  double a_g0t0 = lam[7 * Ntot + idx] * (-vetU_dD00);
  double a_g0t101 = lam[7 * Ntot + idx] * (g0t113*g0t99);
  double a_g0t102 = lam[7 * Ntot + idx] * (g0t103*g0t113 + g0t129 + g0t186 + g0t191 - g0t206 - g0t209);
  double a_g0t103 = lam[7 * Ntot + idx] * (g0t102*g0t113);
  double a_g0t105 = lam[7 * Ntot + idx] * (g0t106*g0t113 + g0t130 + g0t173 + g0t175 - g0t180 - g0t182);
  double a_g0t106 = lam[7 * Ntot + idx] * (g0t105*g0t113);
  double a_g0t112 = lam[7 * Ntot + idx] * (betU_dupD01);
  double a_g0t113 = lam[7 * Ntot + idx] * (g0t101*g0t99 + g0t102*g0t103 + g0t105*g0t106 + g0t80*g0t83 + g0t90*g0t91 + g0t94*g0t95);
  double a_g0t114 = lam[7 * Ntot + idx] * (g0t94);
  double a_g0t125 = lam[7 * Ntot + idx] * (g0t99);
  double a_g0t129 = lam[7 * Ntot + idx] * (g0t102);
  double a_g0t130 = lam[7 * Ntot + idx] * (g0t105);
  double a_g0t131 = lam[7 * Ntot + idx] * (-g0t94);
  double a_g0t132 = lam[7 * Ntot + idx] * (-g0t133 - g0t167);
  double a_g0t133 = lam[7 * Ntot + idx] * (-g0t132);
  double a_g0t147 = lam[7 * Ntot + idx] * (g0t8);
  double a_g0t15 = lam[7 * Ntot + idx] * (-2.0*g0t43);
  double a_g0t151 = lam[7 * Ntot + idx] * (-g0t172);
  double a_g0t154 = lam[7 * Ntot + idx] * (g0t18);
  double a_g0t158 = lam[7 * Ntot + idx] * (g0t80);
  double a_g0t159 = lam[7 * Ntot + idx] * (g0t94);
  double a_g0t164 = lam[7 * Ntot + idx] * (g0t90);
  double a_g0t165 = lam[7 * Ntot + idx] * (-g0t167);
  double a_g0t166 = lam[7 * Ntot + idx] * (-g0t179);
  double a_g0t167 = lam[7 * Ntot + idx] * (-g0t132 - g0t165 + vetU_dDD001);
  double a_g0t169 = lam[7 * Ntot + idx] * (vetU_dDD000);
  double a_g0t170 = lam[7 * Ntot + idx] * (-g0t171*g0t74);
  double a_g0t171 = lam[7 * Ntot + idx] * (-g0t170*g0t74 - g0t3*vetU0 + g0t67*vetU_dD00 + g0t74*vetU_dD01);
  double a_g0t172 = lam[7 * Ntot + idx] * (f0_of_xx0*vetU_dD00 - g0t151 - vetU0 + vetU_dDD011);
  double a_g0t173 = lam[7 * Ntot + idx] * (g0t105);
  double a_g0t175 = lam[7 * Ntot + idx] * (g0t105);
  double a_g0t176 = lam[7 * Ntot + idx] * (g0t89);
  double a_g0t178 = lam[7 * Ntot + idx] * (-g0t8);
  double a_g0t179 = lam[7 * Ntot + idx] * (-g0t166);
  double a_g0t18 = lam[7 * Ntot + idx] * (g0t154);
  double a_g0t180 = lam[7 * Ntot + idx] * (-g0t105);
  double a_g0t182 = lam[7 * Ntot + idx] * (-g0t105);
  double a_g0t183 = lam[7 * Ntot + idx] * (-g0t89);
  double a_g0t186 = lam[7 * Ntot + idx] * (g0t102);
  double a_g0t189 = lam[7 * Ntot + idx] * (g0t99);
  double a_g0t191 = lam[7 * Ntot + idx] * (g0t102);
  double a_g0t193 = lam[7 * Ntot + idx] * (g0t99);
  double a_g0t196 = lam[7 * Ntot + idx] * (g0t79);
  double a_g0t20 = lam[7 * Ntot + idx] * (-g0t22*g0t43);
  double a_g0t200 = lam[7 * Ntot + idx] * (-g0t202);
  double a_g0t201 = lam[7 * Ntot + idx] * (-g0t205*g0t52*g0t67);
  double a_g0t202 = lam[7 * Ntot + idx] * (-g0t200);
  double a_g0t205 = lam[7 * Ntot + idx] * (-g0t201*g0t52*g0t67);
  double a_g0t206 = lam[7 * Ntot + idx] * (-g0t102);
  double a_g0t207 = lam[7 * Ntot + idx] * (-g0t99);
  double a_g0t209 = lam[7 * Ntot + idx] * (-g0t102);
  double a_g0t210 = lam[7 * Ntot + idx] * (-g0t99);
  double a_g0t211 = lam[7 * Ntot + idx] * (-g0t79);
  double a_g0t22 = lam[7 * Ntot + idx] * (-g0t20*g0t43);
  double a_g0t28 = lam[7 * Ntot + idx] * (-2.0*g0t43);
  double a_g0t29 = lam[7 * Ntot + idx] * (-4.0*g0t31*g0t43);
  double a_g0t3 = lam[7 * Ntot + idx] * (-g0t171*vetU0);
  double a_g0t31 = lam[7 * Ntot + idx] * (-4.0*g0t29*g0t43);
  double a_g0t32 = lam[7 * Ntot + idx] * (-g0t36*g0t43);
  double a_g0t36 = lam[7 * Ntot + idx] * (-g0t32*g0t43);
  double a_g0t37 = lam[7 * Ntot + idx] * (-4.0*g0t40*g0t43);
  double a_g0t40 = lam[7 * Ntot + idx] * (-4.0*g0t37*g0t43);
  double a_g0t43 = lam[7 * Ntot + idx] * (-2.0*g0t15 - g0t20*g0t22 - 2.0*g0t28 - 4.0*g0t29*g0t31 - g0t32*g0t36 - 4.0*g0t37*g0t40);
  double a_g0t52 = lam[7 * Ntot + idx] * (-g0t201*g0t205*g0t67);
  double a_g0t65 = lam[7 * Ntot + idx] * (g0t66);
  double a_g0t66 = lam[7 * Ntot + idx] * (g0t65);
  double a_g0t67 = lam[7 * Ntot + idx] * (g0t171*vetU_dD00 - g0t201*g0t205*g0t52);
  double a_g0t74 = lam[7 * Ntot + idx] * (g0t171*(-g0t170 + vetU_dD01));
  double a_g0t79 = lam[7 * Ntot + idx] * (g0t196 - g0t211);
  double a_g0t8 = lam[7 * Ntot + idx] * (g0t147 - g0t178);
  double a_g0t80 = lam[7 * Ntot + idx] * (g0t113*g0t83 + g0t158);
  double a_g0t83 = lam[7 * Ntot + idx] * (g0t113*g0t80);
  double a_g0t89 = lam[7 * Ntot + idx] * (g0t176 - g0t183);
  double a_g0t90 = lam[7 * Ntot + idx] * (g0t113*g0t91 + g0t164);
  double a_g0t91 = lam[7 * Ntot + idx] * (g0t113*g0t90);
  double a_g0t94 = lam[7 * Ntot + idx] * (g0t113*g0t95 + g0t114 - g0t131 + g0t159);
  double a_g0t95 = lam[7 * Ntot + idx] * (g0t113*g0t94);
  double a_g0t99 = lam[7 * Ntot + idx] * (g0t101*g0t113 + g0t125 + g0t189 + g0t193 - g0t207 - g0t210);
  double a_vetU0 = lam[7 * Ntot + idx] * (betU_dupD00 - g0t171*g0t3 - g0t172);
  double a_vetU_dD00 = lam[7 * Ntot + idx] * (f0_of_xx0*g0t172 - g0t0 + g0t171*g0t67);
  double a_vetU_dD01 = lam[7 * Ntot + idx] * (g0t171*g0t74);
  double a_vetU_dDD000 = lam[7 * Ntot + idx] * (g0t169);
  double a_vetU_dDD001 = lam[7 * Ntot + idx] * (g0t167);
  double a_vetU_dDD011 = lam[7 * Ntot + idx] * (g0t172);
  double a_betU_dupD10 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t107*vetU0);
  double a_betU_dupD11 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t139);
  a_eta += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t174);
  a_f0_of_xx0 += lam[8 * Ntot + idx] * (betU_dupD11*g0t139 - eta*g0t174 - g0t0*g0t140 + g0t113*(g0t101*g0t220 + g0t103*g0t219 + g0t106*g0t223 + g0t215*g0t83 + g0t217*g0t91 + g0t218*g0t95) + g0t114*g0t218 + g0t125*g0t220 + g0t129*g0t219 + g0t130*g0t223 - g0t131*g0t218 - g0t133*g0t144 + g0t147*g0t18 + g0t154*g0t47 + g0t158*g0t215 + g0t159*g0t218 + g0t164*g0t217 - g0t166*g0t177 + g0t167*(g0t145 + g0t224) + g0t169*(g0t107*vetU_dDD100 + g0t109*g0t140 - 2.0*g0t134*vetU_dD10 + g0t170*g0t225) + g0t171*(g0t108*g0t74 - g0t112*g0t149 + g0t112*g0t3 + g0t140*g0t67) + g0t172*(2.0*g0t132 + g0t148 + g0t165) + g0t173*g0t222 + g0t175*g0t222 + g0t176*g0t217 - g0t180*g0t222 - g0t182*g0t222 - g0t183*g0t217 + g0t186*g0t219 + g0t189*g0t220 + g0t191*g0t219 + g0t193*g0t220 + g0t196*g0t214 - g0t199*g0t202*g0t74 - g0t206*g0t219 - g0t207*g0t220 - g0t209*g0t219 - g0t210*g0t220 - g0t211*g0t214 - g0t226*g0t227 + g0t227*(-f1_of_xx1*g0t203 + g0t107*g0t110*g0t149*vetU2 + g0t107*g0t110*vetU2*(-g0t149 - g0t150) - g0t226) - g0t228*g0t47 + g0t43*g0t65 + g0t66*(-2.0*g0t160 - g0t161*g0t212 - 2.0*g0t162 - 4.0*g0t163*g0t39 - 4.0*g0t30*g0t51 - g0t36*g0t60) + vetU0*(betU_dupD10*g0t107 - g0t187));
  double a_f1_of_xx1 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t203*g0t227);
  a_g0t0 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t140);
  a_g0t101 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t113*g0t220);
  a_g0t103 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t113*g0t219);
  a_g0t106 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t113*g0t223);
  double a_g0t107 = lam[8 * Ntot + idx] * (f0_of_xx0*(betU_dupD10*vetU0 + g0t169*vetU_dDD100 + g0t227*(g0t110*g0t149*vetU2 + g0t110*vetU2*(-g0t149 - g0t150))));
  double a_g0t108 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t171*g0t74);
  double a_g0t109 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t140*g0t169);
  double a_g0t110 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t227*(g0t107*g0t149*vetU2 + g0t107*vetU2*(-g0t149 - g0t150)));
  a_g0t112 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t171*(-g0t149 + g0t3));
  a_g0t113 += lam[8 * Ntot + idx] * (f0_of_xx0*(g0t101*g0t220 + g0t103*g0t219 + g0t106*g0t223 + g0t215*g0t83 + g0t217*g0t91 + g0t218*g0t95));
  a_g0t114 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t218);
  a_g0t125 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t220);
  a_g0t129 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t219);
  a_g0t130 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t223);
  a_g0t131 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t218);
  a_g0t132 += lam[8 * Ntot + idx] * (2.0*f0_of_xx0*g0t172);
  a_g0t133 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t144);
  double a_g0t134 = lam[8 * Ntot + idx] * (-2.0*f0_of_xx0*g0t169*vetU_dD10);
  double a_g0t139 = lam[8 * Ntot + idx] * (betU_dupD11*f0_of_xx0);
  double a_g0t140 = lam[8 * Ntot + idx] * (f0_of_xx0*(-g0t0 + g0t109*g0t169 + g0t171*g0t67));
  double a_g0t144 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t133);
  double a_g0t145 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t167);
  a_g0t147 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t18);
  double a_g0t148 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t172);
  double a_g0t149 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t112*g0t171);
  double a_g0t150 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t107*g0t110*g0t227*vetU2);
  a_g0t154 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t47);
  a_g0t158 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t215);
  a_g0t159 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t218);
  double a_g0t160 = lam[8 * Ntot + idx] * (-2.0*f0_of_xx0*g0t66);
  double a_g0t161 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t212*g0t66);
  double a_g0t162 = lam[8 * Ntot + idx] * (-2.0*f0_of_xx0*g0t66);
  double a_g0t163 = lam[8 * Ntot + idx] * (-4.0*f0_of_xx0*g0t39*g0t66);
  a_g0t164 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t217);
  a_g0t165 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t172);
  a_g0t166 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t177);
  a_g0t167 += lam[8 * Ntot + idx] * (f0_of_xx0*(g0t145 + g0t224));
  a_g0t169 += lam[8 * Ntot + idx] * (f0_of_xx0*(g0t107*vetU_dDD100 + g0t109*g0t140 - 2.0*g0t134*vetU_dD10 + g0t170*g0t225));
  a_g0t170 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t169*g0t225);
  a_g0t171 += lam[8 * Ntot + idx] * (f0_of_xx0*(g0t108*g0t74 - g0t112*g0t149 + g0t112*g0t3 + g0t140*g0t67));
  a_g0t172 += lam[8 * Ntot + idx] * (f0_of_xx0*(2.0*g0t132 + g0t148 + g0t165));
  a_g0t173 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t222);
  double a_g0t174 = lam[8 * Ntot + idx] * (-eta*f0_of_xx0);
  a_g0t175 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t222);
  a_g0t176 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t217);
  double a_g0t177 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t166);
  a_g0t18 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t147);
  a_g0t180 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t222);
  a_g0t182 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t222);
  a_g0t183 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t217);
  a_g0t186 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t219);
  double a_g0t187 = lam[8 * Ntot + idx] * (-f0_of_xx0*vetU0);
  a_g0t189 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t220);
  a_g0t191 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t219);
  a_g0t193 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t220);
  a_g0t196 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t214);
  double a_g0t199 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t202*g0t74);
  a_g0t202 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t199*g0t74);
  double a_g0t203 = lam[8 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1*g0t227);
  a_g0t206 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t219);
  a_g0t207 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t220);
  a_g0t209 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t219);
  a_g0t210 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t220);
  a_g0t211 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t214);
  double a_g0t212 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t161*g0t66);
  double a_g0t214 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t196 - g0t211));
  double a_g0t215 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t113*g0t83 + g0t158));
  double a_g0t217 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t113*g0t91 + g0t164 + g0t176 - g0t183));
  double a_g0t218 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t113*g0t95 + g0t114 - g0t131 + g0t159));
  double a_g0t219 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t103*g0t113 + g0t129 + g0t186 + g0t191 - g0t206 - g0t209));
  double a_g0t220 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t101*g0t113 + g0t125 + g0t189 + g0t193 - g0t207 - g0t210));
  double a_g0t222 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t173 + g0t175 - g0t180 - g0t182));
  double a_g0t223 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t106*g0t113 + g0t130));
  double a_g0t224 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t167);
  double a_g0t225 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t169*g0t170);
  double a_g0t226 = lam[8 * Ntot + idx] * (-2.0*f0_of_xx0*g0t227);
  double a_g0t227 = lam[8 * Ntot + idx] * (f0_of_xx0*(-f1_of_xx1*g0t203 + g0t107*g0t110*g0t149*vetU2 + g0t107*g0t110*vetU2*(-g0t149 - g0t150) - 2.0*g0t226));
  double a_g0t228 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t47);
  a_g0t3 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t112*g0t171);
  double a_g0t30 = lam[8 * Ntot + idx] * (-4.0*f0_of_xx0*g0t51*g0t66);
  a_g0t36 += lam[8 * Ntot + idx] * (-f0_of_xx0*g0t60*g0t66);
  double a_g0t39 = lam[8 * Ntot + idx] * (-4.0*f0_of_xx0*g0t163*g0t66);
  a_g0t43 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t65);
  double a_g0t47 = lam[8 * Ntot + idx] * (f0_of_xx0*(g0t154 - g0t228));
  double a_g0t51 = lam[8 * Ntot + idx] * (-4.0*f0_of_xx0*g0t30*g0t66);
  double a_g0t60 = lam[8 * Ntot + idx] * (-f0_of_xx0*g0t36*g0t66);
  a_g0t65 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t43);
  a_g0t66 += lam[8 * Ntot + idx] * (f0_of_xx0*(-2.0*g0t160 - g0t161*g0t212 - 2.0*g0t162 - 4.0*g0t163*g0t39 - 4.0*g0t30*g0t51 - g0t36*g0t60));
  a_g0t67 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t140*g0t171);
  a_g0t74 += lam[8 * Ntot + idx] * (f0_of_xx0*(g0t108*g0t171 - g0t199*g0t202));
  a_g0t83 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t113*g0t215);
  a_g0t91 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t113*g0t217);
  a_g0t95 += lam[8 * Ntot + idx] * (f0_of_xx0*g0t113*g0t218);
  a_vetU0 += lam[8 * Ntot + idx] * (f0_of_xx0*(betU_dupD10*g0t107 - g0t187));
  double a_vetU2 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t227*(g0t107*g0t110*g0t149 + g0t107*g0t110*(-g0t149 - g0t150)));
  double a_vetU_dD10 = lam[8 * Ntot + idx] * (-2.0*f0_of_xx0*g0t134*g0t169);
  double a_vetU_dDD100 = lam[8 * Ntot + idx] * (f0_of_xx0*g0t107*g0t169);
  double a_betU2 = lam[9 * Ntot + idx] * (g0t33*(-g0t112*g0t240 - g0t197*vetU0));
  double a_betU_dupD20 = lam[9 * Ntot + idx] * (g0t107*g0t110*g0t33*vetU0);
  double a_betU_dupD21 = lam[9 * Ntot + idx] * (g0t107*g0t110*g0t112*g0t33);
  a_eta += lam[9 * Ntot + idx] * (-g0t190*g0t33);
  a_f0_of_xx0 += lam[9 * Ntot + idx] * (g0t172*g0t199*g0t33);
  double a_f1_of_xx1__D1 = lam[9 * Ntot + idx] * (g0t107*g0t110*g0t227*g0t33*vetU_dD11);
  double a_f1_of_xx1__DD11 = lam[9 * Ntot + idx] * (-g0t172*g0t239*g0t33*vetU2);
  a_g0t0 += lam[9 * Ntot + idx] * (-g0t199*g0t33);
  a_g0t101 += lam[9 * Ntot + idx] * (g0t113*g0t236*g0t33);
  a_g0t103 += lam[9 * Ntot + idx] * (g0t113*g0t238*g0t33);
  a_g0t106 += lam[9 * Ntot + idx] * (g0t113*g0t234*g0t33);
  a_g0t107 += lam[9 * Ntot + idx] * (g0t33*(betU_dupD20*g0t110*vetU0 + betU_dupD21*g0t110*g0t112 + f1_of_xx1__D1*g0t110*g0t227*vetU_dD11 + 2.0*g0t149*g0t172*g0t241*vetU2));
  a_g0t108 += lam[9 * Ntot + idx] * (g0t111*g0t227*g0t33);
  a_g0t109 += lam[9 * Ntot + idx] * (g0t33*(g0t169*g0t199 - g0t172*g0t204*vetU_dD21));
  a_g0t110 += lam[9 * Ntot + idx] * (g0t33*(betU_dupD20*g0t107*vetU0 + betU_dupD21*g0t107*g0t112 + f1_of_xx1__D1*g0t107*g0t227*vetU_dD11));
  double a_g0t111 = lam[9 * Ntot + idx] * (g0t33*(g0t108*g0t227 + g0t140*g0t202 + g0t167*g0t199 + 2.0*g0t172*g0t205));
  a_g0t112 += lam[9 * Ntot + idx] * (g0t33*(-betU2*g0t240 + betU_dupD21*g0t107*g0t110 + g0t227*g0t242 - g0t227));
  a_g0t113 += lam[9 * Ntot + idx] * (g0t33*(g0t101*g0t236 + g0t103*g0t238 + g0t106*g0t234 + g0t230*g0t83 + g0t232*g0t91 + g0t233*g0t95));
  a_g0t114 += lam[9 * Ntot + idx] * (g0t233*g0t33);
  double a_g0t116 = lam[9 * Ntot + idx] * (-2.0*g0t33*g0t66);
  double a_g0t120 = lam[9 * Ntot + idx] * (-g0t33*g0t59*g0t66);
  double a_g0t124 = lam[9 * Ntot + idx] * (-2.0*g0t33*g0t66);
  a_g0t125 += lam[9 * Ntot + idx] * (g0t236*g0t33);
  double a_g0t126 = lam[9 * Ntot + idx] * (-2.0*g0t33*g0t43);
  double a_g0t128 = lam[9 * Ntot + idx] * (-2.0*g0t33*g0t43);
  a_g0t129 += lam[9 * Ntot + idx] * (g0t238*g0t33);
  a_g0t130 += lam[9 * Ntot + idx] * (g0t234*g0t33);
  a_g0t131 += lam[9 * Ntot + idx] * (-g0t233*g0t33);
  a_g0t132 += lam[9 * Ntot + idx] * (2.0*g0t227*g0t33);
  a_g0t140 += lam[9 * Ntot + idx] * (g0t111*g0t202*g0t33);
  a_g0t147 += lam[9 * Ntot + idx] * (g0t24*g0t33);
  a_g0t149 += lam[9 * Ntot + idx] * (g0t172*g0t33*(2.0*g0t107*g0t241*vetU2 + g0t203*g0t241));
  double a_g0t153 = lam[9 * Ntot + idx] * (-g0t227*g0t33);
  a_g0t154 += lam[9 * Ntot + idx] * (g0t33*g0t52);
  double a_g0t155 = lam[9 * Ntot + idx] * (g0t33*(g0t43*(-g0t37 - g0t53) - g0t60*g0t66));
  double a_g0t156 = lam[9 * Ntot + idx] * (-g0t33*g0t43*g0t8);
  a_g0t158 += lam[9 * Ntot + idx] * (g0t230*g0t33);
  a_g0t159 += lam[9 * Ntot + idx] * (g0t233*g0t33);
  a_g0t163 += lam[9 * Ntot + idx] * (-g0t22*g0t33*g0t66);
  a_g0t164 += lam[9 * Ntot + idx] * (g0t232*g0t33);
  a_g0t167 += lam[9 * Ntot + idx] * (g0t33*(g0t111*g0t199 + g0t184*vetU_dDD201 + g0t194*g0t204 - g0t197*vetU_dD21 - g0t240*vetU_dD20));
  a_g0t169 += lam[9 * Ntot + idx] * (g0t33*(g0t109*g0t199 + g0t184*vetU_dDD200 + 2.0*g0t188*g0t225 - 2.0*g0t197*vetU_dD20));
  a_g0t171 += lam[9 * Ntot + idx] * (g0t33*(g0t200 + g0t226));
  a_g0t172 += lam[9 * Ntot + idx] * (g0t33*(f0_of_xx0*g0t199 - g0t109*g0t204*vetU_dD21 + 2.0*g0t111*g0t205 + g0t149*g0t203*g0t241 + g0t184*vetU_dDD211 + g0t185*g0t242 + g0t185 + vetU2*(-f1_of_xx1__DD11*g0t239 + 2.0*g0t107*g0t149*g0t241)));
  a_g0t173 += lam[9 * Ntot + idx] * (g0t234*g0t33);
  a_g0t175 += lam[9 * Ntot + idx] * (g0t234*g0t33);
  a_g0t176 += lam[9 * Ntot + idx] * (g0t232*g0t33);
  a_g0t178 += lam[9 * Ntot + idx] * (-g0t24*g0t33);
  a_g0t180 += lam[9 * Ntot + idx] * (-g0t234*g0t33);
  double a_g0t181 = lam[9 * Ntot + idx] * (-g0t205*g0t33);
  a_g0t182 += lam[9 * Ntot + idx] * (-g0t234*g0t33);
  a_g0t183 += lam[9 * Ntot + idx] * (-g0t232*g0t33);
  double a_g0t184 = lam[9 * Ntot + idx] * (g0t33*(g0t167*vetU_dDD201 + g0t169*vetU_dDD200 + g0t172*vetU_dDD211));
  double a_g0t185 = lam[9 * Ntot + idx] * (g0t172*g0t33*(g0t242 + 1.0));
  a_g0t186 += lam[9 * Ntot + idx] * (g0t237*g0t33);
  double a_g0t188 = lam[9 * Ntot + idx] * (2.0*g0t169*g0t225*g0t33);
  a_g0t189 += lam[9 * Ntot + idx] * (g0t235*g0t33);
  double a_g0t190 = lam[9 * Ntot + idx] * (-eta*g0t33);
  a_g0t191 += lam[9 * Ntot + idx] * (g0t237*g0t33);
  a_g0t193 += lam[9 * Ntot + idx] * (g0t235*g0t33);
  double a_g0t194 = lam[9 * Ntot + idx] * (g0t167*g0t204*g0t33);
  a_g0t196 += lam[9 * Ntot + idx] * (g0t230*g0t33);
  double a_g0t197 = lam[9 * Ntot + idx] * (g0t33*(-betU2*vetU0 - g0t167*vetU_dD21 - 2.0*g0t169*vetU_dD20));
  a_g0t199 += lam[9 * Ntot + idx] * (g0t33*(f0_of_xx0*g0t172 - g0t0 + g0t109*g0t169 + g0t111*g0t167));
  a_g0t200 += lam[9 * Ntot + idx] * (g0t171*g0t33);
  a_g0t202 += lam[9 * Ntot + idx] * (g0t33*(g0t111*g0t140 + g0t224));
  a_g0t203 += lam[9 * Ntot + idx] * (g0t149*g0t172*g0t241*g0t33);
  double a_g0t204 = lam[9 * Ntot + idx] * (g0t33*(-g0t109*g0t172*vetU_dD21 + g0t167*g0t194));
  a_g0t205 += lam[9 * Ntot + idx] * (g0t33*(2.0*g0t111*g0t172 - g0t181));
  a_g0t206 += lam[9 * Ntot + idx] * (-g0t237*g0t33);
  a_g0t207 += lam[9 * Ntot + idx] * (-g0t235*g0t33);
  a_g0t209 += lam[9 * Ntot + idx] * (-g0t237*g0t33);
  a_g0t210 += lam[9 * Ntot + idx] * (-g0t235*g0t33);
  a_g0t211 += lam[9 * Ntot + idx] * (-g0t230*g0t33);
  a_g0t212 += lam[9 * Ntot + idx] * (-g0t33*g0t43*g0t60);
  a_g0t22 += lam[9 * Ntot + idx] * (-g0t163*g0t33*g0t66);
  a_g0t224 += lam[9 * Ntot + idx] * (g0t202*g0t33);
  a_g0t225 += lam[9 * Ntot + idx] * (2.0*g0t169*g0t188*g0t33);
  a_g0t226 += lam[9 * Ntot + idx] * (g0t171*g0t33);
  a_g0t227 += lam[9 * Ntot + idx] * (g0t33*(f1_of_xx1__D1*g0t107*g0t110*vetU_dD11 + g0t108*g0t111 + g0t112*g0t242 - g0t112 + 2.0*g0t132 - g0t153));
  a_g0t228 += lam[9 * Ntot + idx] * (-g0t33*g0t52);
  double a_g0t229 = lam[9 * Ntot + idx] * (g0t33*(-g0t43*g0t59 - g0t55*g0t66));
  double a_g0t230 = lam[9 * Ntot + idx] * (g0t33*(g0t113*g0t83 + g0t158 + g0t196 - g0t211));
  double a_g0t232 = lam[9 * Ntot + idx] * (g0t33*(g0t113*g0t91 + g0t164 + g0t176 - g0t183));
  double a_g0t233 = lam[9 * Ntot + idx] * (g0t33*(g0t113*g0t95 + g0t114 - g0t131 + g0t159));
  double a_g0t234 = lam[9 * Ntot + idx] * (g0t33*(g0t106*g0t113 + g0t130 + g0t173 + g0t175 - g0t180 - g0t182));
  double a_g0t235 = lam[9 * Ntot + idx] * (g0t33*(g0t189 + g0t193 - g0t207 - g0t210));
  double a_g0t236 = lam[9 * Ntot + idx] * (g0t33*(g0t101*g0t113 + g0t125));
  double a_g0t237 = lam[9 * Ntot + idx] * (g0t33*(g0t186 + g0t191 - g0t206 - g0t209));
  double a_g0t238 = lam[9 * Ntot + idx] * (g0t33*(g0t103*g0t113 + g0t129));
  double a_g0t239 = lam[9 * Ntot + idx] * (-f1_of_xx1__DD11*g0t172*g0t33*vetU2);
  double a_g0t24 = lam[9 * Ntot + idx] * (g0t33*(g0t147 - g0t178));
  double a_g0t240 = lam[9 * Ntot + idx] * (g0t33*(-betU2*g0t112 - g0t167*vetU_dD20));
  double a_g0t241 = lam[9 * Ntot + idx] * (g0t172*g0t33*(2.0*g0t107*g0t149*vetU2 + g0t149*g0t203));
  double a_g0t242 = lam[9 * Ntot + idx] * (g0t33*(g0t112*g0t227 + g0t172*g0t185));
  double a_g0t26 = lam[9 * Ntot + idx] * (-g0t33*g0t43*g0t55);
  double a_g0t33 = lam[9 * Ntot + idx] * (-eta*g0t190 - g0t0*g0t199 + g0t112*(-betU2*g0t240 + betU_dupD21*g0t107*g0t110) + g0t113*(g0t101*g0t236 + g0t103*g0t238 + g0t106*g0t234 + g0t230*g0t83 + g0t232*g0t91 + g0t233*g0t95) + g0t114*g0t233 + g0t125*g0t236 + g0t129*g0t238 + g0t130*g0t234 - g0t131*g0t233 + g0t147*g0t24 + g0t154*g0t52 + g0t158*g0t230 + g0t159*g0t233 + g0t164*g0t232 + g0t167*(g0t111*g0t199 + g0t184*vetU_dDD201 + g0t194*g0t204 - g0t197*vetU_dD21 - g0t240*vetU_dD20) + g0t169*(g0t109*g0t199 + g0t184*vetU_dDD200 + 2.0*g0t188*g0t225 - 2.0*g0t197*vetU_dD20) + g0t171*(g0t200 + g0t226) + g0t172*(f0_of_xx0*g0t199 - g0t109*g0t204*vetU_dD21 + 2.0*g0t111*g0t205 + g0t149*g0t203*g0t241 + g0t184*vetU_dDD211 + g0t185*g0t242 + g0t185 + vetU2*(-f1_of_xx1__DD11*g0t239 + 2.0*g0t107*g0t149*g0t241)) + g0t173*g0t234 + g0t175*g0t234 + g0t176*g0t232 - g0t178*g0t24 - g0t180*g0t234 - g0t181*g0t205 - g0t182*g0t234 - g0t183*g0t232 + g0t186*g0t237 + g0t189*g0t235 + g0t191*g0t237 + g0t193*g0t235 + g0t196*g0t230 + g0t202*(g0t111*g0t140 + g0t224) - g0t206*g0t237 - g0t207*g0t235 - g0t209*g0t237 - g0t210*g0t235 - g0t211*g0t230 + g0t227*(g0t108*g0t111 + g0t112*g0t242 + g0t132) + g0t227*(f1_of_xx1__D1*g0t107*g0t110*vetU_dD11 - g0t112 + g0t132 - g0t153) - g0t228*g0t52 + g0t43*(-2.0*g0t126 - 2.0*g0t128 - g0t155*g0t37 - g0t155*g0t53 - g0t156*g0t8 - g0t212*g0t60 - g0t229*g0t59 - g0t26*g0t55 - g0t61*g0t63) + g0t66*(-2.0*g0t116 - g0t120*g0t59 - 2.0*g0t124 - g0t155*g0t60 - g0t163*g0t22 - g0t229*g0t55 - g0t48*g0t59*g0t81 - g0t50*g0t57 - g0t56*g0t63) + vetU0*(-betU2*g0t197 + betU_dupD20*g0t107*g0t110));
  a_g0t37 += lam[9 * Ntot + idx] * (-g0t155*g0t33*g0t43);
  a_g0t43 += lam[9 * Ntot + idx] * (g0t33*(-2.0*g0t126 - 2.0*g0t128 - g0t155*g0t37 - g0t155*g0t53 - g0t156*g0t8 - g0t212*g0t60 - g0t229*g0t59 - g0t26*g0t55 - g0t61*g0t63));
  double a_g0t48 = lam[9 * Ntot + idx] * (-g0t33*g0t59*g0t66*g0t81);
  double a_g0t50 = lam[9 * Ntot + idx] * (-g0t33*g0t57*g0t66);
  a_g0t52 += lam[9 * Ntot + idx] * (g0t33*(g0t154 - g0t228));
  double a_g0t53 = lam[9 * Ntot + idx] * (-g0t155*g0t33*g0t43);
  double a_g0t55 = lam[9 * Ntot + idx] * (g0t33*(-g0t229*g0t66 - g0t26*g0t43));
  double a_g0t56 = lam[9 * Ntot + idx] * (-g0t33*g0t63*g0t66);
  double a_g0t57 = lam[9 * Ntot + idx] * (-g0t33*g0t50*g0t66);
  double a_g0t59 = lam[9 * Ntot + idx] * (g0t33*(-g0t229*g0t43 + g0t66*(-g0t120 - g0t48*g0t81)));
  a_g0t60 += lam[9 * Ntot + idx] * (g0t33*(-g0t155*g0t66 - g0t212*g0t43));
  double a_g0t61 = lam[9 * Ntot + idx] * (-g0t33*g0t43*g0t63);
  double a_g0t63 = lam[9 * Ntot + idx] * (g0t33*(-g0t43*g0t61 - g0t56*g0t66));
  a_g0t66 += lam[9 * Ntot + idx] * (g0t33*(-2.0*g0t116 - g0t120*g0t59 - 2.0*g0t124 - g0t155*g0t60 - g0t163*g0t22 - g0t229*g0t55 - g0t48*g0t59*g0t81 - g0t50*g0t57 - g0t56*g0t63));
  a_g0t8 += lam[9 * Ntot + idx] * (-g0t156*g0t33*g0t43);
  double a_g0t81 = lam[9 * Ntot + idx] * (-g0t33*g0t48*g0t59*g0t66);
  a_g0t83 += lam[9 * Ntot + idx] * (g0t113*g0t230*g0t33);
  a_g0t91 += lam[9 * Ntot + idx] * (g0t113*g0t232*g0t33);
  a_g0t95 += lam[9 * Ntot + idx] * (g0t113*g0t233*g0t33);
  a_vetU0 += lam[9 * Ntot + idx] * (g0t33*(-betU2*g0t197 + betU_dupD20*g0t107*g0t110));
  a_vetU2 += lam[9 * Ntot + idx] * (g0t172*g0t33*(-f1_of_xx1__DD11*g0t239 + 2.0*g0t107*g0t149*g0t241));
  double a_vetU_dD11 = lam[9 * Ntot + idx] * (f1_of_xx1__D1*g0t107*g0t110*g0t227*g0t33);
  double a_vetU_dD20 = lam[9 * Ntot + idx] * (g0t33*(-g0t167*g0t240 - 2.0*g0t169*g0t197));
  double a_vetU_dD21 = lam[9 * Ntot + idx] * (g0t33*(-g0t109*g0t172*g0t204 - g0t167*g0t197));
  double a_vetU_dDD200 = lam[9 * Ntot + idx] * (g0t169*g0t184*g0t33);
  double a_vetU_dDD201 = lam[9 * Ntot + idx] * (g0t167*g0t184*g0t33);
  double a_vetU_dDD211 = lam[9 * Ntot + idx] * (g0t172*g0t184*g0t33);
  a_f1_of_xx1__DD11 += a_g0t242 * (g0t110);
  a_g0t110 += a_g0t242 * (f1_of_xx1__DD11);
  double a_g0t152 = a_g0t242 * (-1.0);
  a_f1_of_xx1 += a_g0t241 * (-3.0/(f1_of_xx1*f1_of_xx1*f1_of_xx1*f1_of_xx1));
  a_f1_of_xx1__D1 += a_g0t240 * (g0t239);
  a_g0t239 += a_g0t240 * (f1_of_xx1__D1);
  a_g0t107 += a_g0t239 * (g0t137);
  double a_g0t137 = a_g0t239 * (g0t107);
  double a_g0t221 = a_g0t238 * (1.0);
  a_g0t237 += a_g0t238 * (1.0);
  double a_g0t216 = a_g0t237 * (g0t97);
  double a_g0t231 = a_g0t237 * (g0t69);
  double a_g0t69 = a_g0t237 * (g0t231);
  double a_g0t97 = a_g0t237 * (g0t216);
  a_g0t111 += a_g0t236 * (-1.0);
  a_g0t235 += a_g0t236 * (1.0);
  a_g0t231 += a_g0t235 * (g0t76);
  double a_g0t76 = a_g0t235 * (g0t231);
  double a_g0t87 = a_g0t235 * (g0t98);
  double a_g0t98 = a_g0t235 * (g0t87);
  double a_g0t104 = a_g0t234 * (g0t231);
  a_g0t216 += a_g0t234 * (g0t84);
  a_g0t231 += a_g0t234 * (g0t104);
  double a_g0t84 = a_g0t234 * (g0t216);
  a_g0t87 += a_g0t234 * (hDD_dD001);
  double a_hDD_dD001 = a_g0t234 * (g0t87);
  a_g0t216 += a_g0t233 * (g0t93);
  a_g0t231 += a_g0t233 * (g0t92);
  a_g0t87 += a_g0t233 * (hDD_dD000);
  double a_g0t92 = a_g0t233 * (g0t231);
  double a_g0t93 = a_g0t233 * (g0t216);
  double a_hDD_dD000 = a_g0t233 * (g0t87);
  a_g0t216 += a_g0t232 * (g0t88);
  a_g0t231 += a_g0t232 * (g0t86);
  double a_g0t85 = a_g0t232 * (g0t87);
  double a_g0t86 = a_g0t232 * (g0t231);
  a_g0t87 += a_g0t232 * (g0t85);
  double a_g0t88 = a_g0t232 * (g0t216);
  double a_g0t72 = a_g0t231 * (g0t81);
  a_g0t81 += a_g0t231 * (g0t72);
  a_g0t216 += a_g0t230 * (g0t77);
  double a_g0t70 = a_g0t230 * (g0t87);
  double a_g0t77 = a_g0t230 * (g0t216);
  a_g0t87 += a_g0t230 * (g0t70);
  double a_g0t127 = a_g0t229 * (g0t81);
  a_g0t81 += a_g0t229 * (g0t127);
  a_g0t179 += a_g0t228 * (g0t71);
  double a_g0t71 = a_g0t228 * (g0t179);
  double a_g0t168 = a_g0t227 * (g0t52);
  a_g0t52 += a_g0t227 * (g0t168);
  a_g0t205 += a_g0t226 * (g0t74);
  a_g0t74 += a_g0t226 * (g0t205);
  double a_g0t16 = a_g0t225 * (-1.0/(g0t16*g0t16));
  a_g0t107 += a_g0t224 * (vetU_dD00);
  double a_g0t135 = a_g0t224 * (-1.0);
  a_vetU_dD00 += a_g0t224 * (g0t107);
  a_g0t221 += a_g0t223 * (1.0);
  a_g0t222 += a_g0t223 * (1.0);
  a_g0t104 += a_g0t222 * (g0t216);
  double a_g0t213 = a_g0t222 * (g0t84);
  a_g0t216 += a_g0t222 * (g0t104);
  double a_g0t78 = a_g0t222 * (hDD_dD001);
  a_g0t84 += a_g0t222 * (g0t213);
  a_hDD_dD001 += a_g0t222 * (g0t78);
  a_g0t107 += a_g0t221 * (-1.0);
  a_g0t216 += a_g0t220 * (g0t76);
  a_g0t76 += a_g0t220 * (g0t216);
  a_g0t78 += a_g0t220 * (g0t98);
  a_g0t98 += a_g0t220 * (g0t78);
  a_g0t213 += a_g0t219 * (g0t97);
  a_g0t216 += a_g0t219 * (g0t69);
  a_g0t69 += a_g0t219 * (g0t216);
  a_g0t97 += a_g0t219 * (g0t213);
  a_g0t213 += a_g0t218 * (g0t93);
  a_g0t216 += a_g0t218 * (g0t92);
  a_g0t78 += a_g0t218 * (hDD_dD000);
  a_g0t92 += a_g0t218 * (g0t216);
  a_g0t93 += a_g0t218 * (g0t213);
  a_hDD_dD000 += a_g0t218 * (g0t78);
  a_g0t213 += a_g0t217 * (g0t88);
  a_g0t216 += a_g0t217 * (g0t86);
  a_g0t78 += a_g0t217 * (g0t85);
  a_g0t85 += a_g0t217 * (g0t78);
  a_g0t86 += a_g0t217 * (g0t216);
  a_g0t88 += a_g0t217 * (g0t213);
  a_g0t52 += a_g0t216 * (g0t72);
  a_g0t72 += a_g0t216 * (g0t52);
  a_g0t214 += a_g0t215 * (1.0);
  a_g0t74 += a_g0t215 * (1.0);
  a_g0t213 += a_g0t214 * (g0t77);
  a_g0t70 += a_g0t214 * (g0t78);
  a_g0t77 += a_g0t214 * (g0t213);
  a_g0t78 += a_g0t214 * (g0t70);
  a_g0t47 += a_g0t213 * (g0t72);
  a_g0t72 += a_g0t213 * (g0t47);
  double a_g0t13 = a_g0t212 * (g0t22);
  a_g0t22 += a_g0t212 * (g0t13);
  double a_g0t195 = a_g0t211 * (g0t208);
  double a_g0t208 = a_g0t211 * (g0t195);
  double a_g0t192 = a_g0t210 * (g0t208);
  a_g0t208 += a_g0t210 * (g0t192);
  a_g0t184 += a_g0t209 * (g0t208*vetU0);
  a_g0t208 += a_g0t209 * (g0t184*vetU0);
  a_vetU0 += a_g0t209 * (g0t184*g0t208);
  double a_lambdaU2 = a_g0t208 * (Rational_3_4);
  a_g0t133 += a_g0t207 * (g0t198);
  double a_g0t198 = a_g0t207 * (g0t133);
  a_g0t0 += a_g0t206 * (g0t185);
  a_g0t185 += a_g0t206 * (g0t0);
  a_g0t184 += a_g0t205 * (vetU_dD21);
  a_g0t203 += a_g0t205 * (-g0t204);
  a_g0t204 += a_g0t205 * (-g0t203);
  a_vetU_dD21 += a_g0t205 * (g0t184);
  a_f1_of_xx1__D1 += a_g0t204 * (g0t137);
  a_g0t137 += a_g0t204 * (f1_of_xx1__D1);
  a_g0t107 += a_g0t203 * (vetU2);
  a_vetU2 += a_g0t203 * (g0t107);
  a_g0t201 += a_g0t202 * (g0t24);
  a_g0t24 += a_g0t202 * (g0t201);
  a_g0t71 += a_g0t201 * (Rational_3_2);
  a_g0t199 += a_g0t200 * (g0t67);
  a_g0t67 += a_g0t200 * (g0t199);
  a_g0t184 += a_g0t199 * (vetU_dD20);
  a_g0t198 += a_g0t199 * (-1.0);
  a_vetU_dD20 += a_g0t199 * (g0t184);
  a_g0t197 += a_g0t198 * (vetU2);
  a_vetU2 += a_g0t198 * (g0t197);
  a_g0t110 += a_g0t197 * (g0t134);
  a_g0t134 += a_g0t197 * (g0t110);
  a_betU2 += a_g0t196 * (g0t195);
  a_g0t195 += a_g0t196 * (betU2);
  a_g0t137 += a_g0t195 * (g0t194);
  a_g0t194 += a_g0t195 * (g0t137);
  a_g0t134 += a_g0t194 * (vetU2);
  a_vetU2 += a_g0t194 * (g0t134);
  a_betU2 += a_g0t193 * (g0t192);
  a_g0t192 += a_g0t193 * (betU2);
  a_g0t110 += a_g0t192 * (g0t139);
  a_g0t139 += a_g0t192 * (g0t110);
  a_g0t190 += a_g0t191 * (vetU0);
  a_vetU0 += a_g0t191 * (g0t190);
  a_betU2 += a_g0t190 * (g0t184);
  a_g0t184 += a_g0t190 * (betU2);
  a_g0t187 += a_g0t189 * (g0t188);
  a_g0t188 += a_g0t189 * (g0t187);
  a_g0t110 += a_g0t188 * (vetU2);
  a_vetU2 += a_g0t188 * (g0t110);
  double a_betU1 = a_g0t187 * (g0t134);
  a_g0t134 += a_g0t187 * (betU1);
  a_betU0 += a_g0t186 * (g0t185);
  a_g0t185 += a_g0t186 * (betU0);
  a_g0t184 += a_g0t185 * (vetU2);
  a_vetU2 += a_g0t185 * (g0t184);
  a_g0t107 += a_g0t184 * (g0t110);
  a_g0t110 += a_g0t184 * (g0t107);
  a_g0t133 += a_g0t183 * (g0t139);
  a_g0t139 += a_g0t183 * (g0t133);
  a_g0t181 += a_g0t182 * (vetU0);
  a_vetU0 += a_g0t182 * (g0t181);
  a_g0t107 += a_g0t181 * (g0t133);
  a_g0t133 += a_g0t181 * (g0t107);
  a_g0t0 += a_g0t180 * (g0t112);
  a_g0t112 += a_g0t180 * (g0t0);
  double a_alpha = a_g0t179 * (trK_dD1);
  double a_trK_dD1 = a_g0t179 * (alpha);
  a_g0t177 += a_g0t178 * (g0t71);
  a_g0t71 += a_g0t178 * (g0t177);
  a_alpha += a_g0t177 * (trK_dD0);
  double a_trK_dD0 = a_g0t177 * (alpha);
  a_betU1 += a_g0t176 * (g0t139);
  a_g0t139 += a_g0t176 * (betU1);
  a_g0t174 += a_g0t175 * (vetU0);
  a_vetU0 += a_g0t175 * (g0t174);
  a_betU1 += a_g0t174 * (g0t107);
  a_g0t107 += a_g0t174 * (betU1);
  a_betU0 += a_g0t173 * (g0t112);
  a_g0t112 += a_g0t173 * (betU0);
  a_g0t168 += a_g0t172 * (g0t47);
  a_g0t47 += a_g0t172 * (g0t168);
  a_g0t168 += a_g0t171 * (g0t81);
  a_g0t81 += a_g0t171 * (g0t168);
  double a_vetU1 = a_g0t170 * (2.0);
  a_g0t168 += a_g0t169 * (g0t8);
  a_g0t8 += a_g0t169 * (g0t168);
  a_g0t71 += a_g0t168 * (Rational_3_4);
  a_g0t166 += a_g0t167 * (Rational_3_2);
  a_g0t18 += a_g0t166 * (g0t71);
  a_g0t71 += a_g0t166 * (g0t18);
  a_f0_of_xx0 += a_g0t165 * (g0t140);
  a_g0t140 += a_g0t165 * (f0_of_xx0);
  double a_g0t118 = a_g0t164 * (g0t157*g0t161);
  double a_g0t157 = a_g0t164 * (g0t118*g0t161 + g0t160 + g0t162 + g0t163*g0t59 + g0t50*g0t51 + g0t56*g0t60);
  a_g0t160 += a_g0t164 * (g0t157);
  a_g0t161 += a_g0t164 * (g0t118*g0t157);
  a_g0t162 += a_g0t164 * (g0t157);
  a_g0t163 += a_g0t164 * (g0t157*g0t59);
  a_g0t50 += a_g0t164 * (g0t157*g0t51);
  a_g0t51 += a_g0t164 * (g0t157*g0t50);
  a_g0t56 += a_g0t164 * (g0t157*g0t60);
  a_g0t59 += a_g0t164 * (g0t157*g0t163);
  a_g0t60 += a_g0t164 * (g0t157*g0t56);
  a_g0t48 += a_g0t163 * (g0t52);
  a_g0t52 += a_g0t163 * (g0t48);
  a_g0t120 += a_g0t162 * (g0t27);
  double a_g0t27 = a_g0t162 * (g0t120);
  a_g0t47 += a_g0t161 * (2.0*g0t47);
  double a_g0t14 = a_g0t160 * (g0t19);
  double a_g0t19 = a_g0t160 * (g0t14);
  double a_g0t117 = a_g0t159 * (g0t157*g0t20);
  a_g0t15 += a_g0t159 * (g0t157);
  a_g0t155 += a_g0t159 * (g0t157*g0t29);
  a_g0t157 += a_g0t159 * (g0t117*g0t20 + g0t15 + g0t155*g0t29 + g0t28 + g0t32*g0t56 + g0t37*g0t61);
  a_g0t20 += a_g0t159 * (g0t117*g0t157);
  a_g0t28 += a_g0t159 * (g0t157);
  a_g0t29 += a_g0t159 * (g0t155*g0t157);
  a_g0t32 += a_g0t159 * (g0t157*g0t56);
  a_g0t37 += a_g0t159 * (g0t157*g0t61);
  a_g0t56 += a_g0t159 * (g0t157*g0t32);
  a_g0t61 += a_g0t159 * (g0t157*g0t37);
  a_g0t117 += a_g0t158 * (g0t120*g0t157);
  a_g0t120 += a_g0t158 * (g0t117*g0t157);
  a_g0t14 += a_g0t158 * (g0t157*g0t25);
  a_g0t155 += a_g0t158 * (g0t157*g0t63);
  a_g0t156 += a_g0t158 * (g0t157*g0t24);
  a_g0t157 += a_g0t158 * (g0t117*g0t120 + g0t14*g0t25 + g0t155*g0t63 + g0t156*g0t24 + g0t52*g0t61*g0t81 + g0t62*(g0t81*g0t81));
  a_g0t24 += a_g0t158 * (g0t156*g0t157);
  double a_g0t25 = a_g0t158 * (g0t14*g0t157);
  a_g0t52 += a_g0t158 * (g0t157*g0t61*g0t81);
  a_g0t61 += a_g0t158 * (g0t157*g0t52*g0t81);
  double a_g0t62 = a_g0t158 * (g0t157*(g0t81*g0t81));
  a_g0t63 += a_g0t158 * (g0t155*g0t157);
  a_g0t81 += a_g0t158 * (g0t157*(g0t52*g0t61 + 2.0*g0t62*g0t81));
  a_alpha += a_g0t157 * (Rational_3_2);
  a_g0t56 += a_g0t156 * (g0t81);
  a_g0t81 += a_g0t156 * (g0t56);
  a_g0t13 += a_g0t155 * (g0t50);
  a_g0t50 += a_g0t155 * (g0t13);
  a_g0t107 += a_g0t154 * (-g0t143*g0t146*vetU0);
  a_g0t112 += a_g0t154 * (g0t138*g0t146*(g0t141*g0t149 + g0t141*g0t150));
  double a_g0t136 = a_g0t154 * (g0t138*g0t146*vetU_dD01);
  double a_g0t138 = a_g0t154 * (g0t146*(g0t112*(g0t141*g0t149 + g0t141*g0t150) + g0t136*vetU_dD01 + g0t142*g0t16*vetU0 + g0t151*g0t16*g0t74));
  double a_g0t141 = a_g0t154 * (g0t112*g0t138*g0t146*(g0t149 + g0t150));
  double a_g0t142 = a_g0t154 * (g0t138*g0t146*g0t16*vetU0);
  double a_g0t143 = a_g0t154 * (-g0t107*g0t146*vetU0);
  double a_g0t146 = a_g0t154 * (-g0t107*g0t143*vetU0 + g0t138*(g0t112*(g0t141*g0t149 + g0t141*g0t150) + g0t151*g0t16*g0t74) + g0t138*(g0t136*vetU_dD01 + g0t142*g0t16*vetU0) + g0t148 - 2.0*g0t153 + vetU_dDD001);
  a_g0t148 += a_g0t154 * (g0t146);
  a_g0t149 += a_g0t154 * (g0t112*g0t138*g0t141*g0t146);
  a_g0t150 += a_g0t154 * (g0t112*g0t138*g0t141*g0t146);
  a_g0t151 += a_g0t154 * (g0t138*g0t146*g0t16*g0t74);
  a_g0t153 += a_g0t154 * (-2.0*g0t146);
  a_g0t16 += a_g0t154 * (g0t146*(g0t138*g0t142*vetU0 + g0t138*g0t151*g0t74));
  a_g0t74 += a_g0t154 * (g0t138*g0t146*g0t151*g0t16);
  a_vetU0 += a_g0t154 * (g0t146*(-g0t107*g0t143 + g0t138*g0t142*g0t16));
  a_vetU_dD01 += a_g0t154 * (g0t136*g0t138*g0t146);
  a_vetU_dDD001 += a_g0t154 * (g0t146);
  a_g0t112 += a_g0t153 * (g0t152);
  a_g0t152 += a_g0t153 * (g0t112);
  a_g0t137 += a_g0t152 * (g0t149);
  a_g0t149 += a_g0t152 * (g0t137);
  a_vetU_dD11 += a_g0t151 * (2.0);
  a_f1_of_xx1 += a_g0t150 * (f1_of_xx1__DD11);
  a_f1_of_xx1__DD11 += a_g0t150 * (f1_of_xx1);
  a_f1_of_xx1__D1 += a_g0t149 * (2.0*f1_of_xx1__D1);
  a_g0t107 += a_g0t148 * (vetU_dDD111);
  double a_vetU_dDD111 = a_g0t148 * (g0t107);
  double a_g0t1 = a_g0t147 * (g0t138*g0t142*g0t146*vetU1);
  a_g0t135 += a_g0t147 * (-8.0*g0t146);
  a_g0t136 += a_g0t147 * (g0t138*g0t146*vetU_dD00);
  a_g0t138 += a_g0t147 * (g0t146*(g0t1*g0t142*vetU1 + g0t136*vetU_dD00 + g0t140*g0t141*g0t74 + 12.0*g0t4*vetU0));
  a_g0t139 += a_g0t147 * (-g0t143*g0t146);
  a_g0t140 += a_g0t147 * (g0t138*g0t141*g0t146*g0t74);
  a_g0t141 += a_g0t147 * (g0t138*g0t140*g0t146*g0t74);
  a_g0t142 += a_g0t147 * (g0t1*g0t138*g0t146*vetU1);
  a_g0t143 += a_g0t147 * (-g0t139*g0t146);
  a_g0t145 += a_g0t147 * (g0t146);
  a_g0t146 += a_g0t147 * (-8.0*g0t135 + g0t138*(g0t136*vetU_dD00 + 12.0*g0t4*vetU0) + g0t138*(g0t1*g0t142*vetU1 + g0t140*g0t141*g0t74) - g0t139*g0t143 + g0t145 + vetU_dDD000);
  double a_g0t4 = a_g0t147 * (12.0*g0t138*g0t146*vetU0);
  a_g0t74 += a_g0t147 * (g0t138*g0t140*g0t141*g0t146);
  a_vetU0 += a_g0t147 * (12.0*g0t138*g0t146*g0t4);
  a_vetU1 += a_g0t147 * (g0t1*g0t138*g0t142*g0t146);
  a_vetU_dD00 += a_g0t147 * (g0t136*g0t138*g0t146);
  a_vetU_dDD000 += a_g0t147 * (g0t146);
  a_g0t71 += a_g0t146 * (Rational_1_4);
  a_g0t107 += a_g0t145 * (vetU_dDD101);
  a_g0t144 += a_g0t145 * (-1.0);
  double a_vetU_dDD101 = a_g0t145 * (g0t107);
  a_g0t134 += a_g0t144 * (vetU_dD11);
  a_vetU_dD11 += a_g0t144 * (g0t134);
  a_g0t111 += a_g0t143 * (4.0);
  a_g0t74 += a_g0t142 * (8.0);
  double a_g0t6 = a_g0t141 * (2.0);
  a_g0t107 += a_g0t140 * (vetU_dD10);
  a_g0t139 += a_g0t140 * (-1.0);
  a_vetU_dD10 += a_g0t140 * (g0t107);
  a_g0t134 += a_g0t139 * (vetU1);
  a_vetU1 += a_g0t139 * (g0t134);
  a_g0t137 += a_g0t138 * ((Rational_1_2)/g0t6);
  a_g0t6 += a_g0t138 * (-Rational_1_2*g0t137/(g0t6*g0t6));
  a_g0t3 += a_g0t137 * (-1.0/(g0t3*g0t3));
  a_g0t16 += a_g0t136 * (4.0*g0t3);
  a_g0t3 += a_g0t136 * (4.0*g0t16);
  a_g0t134 += a_g0t135 * (vetU0);
  a_vetU0 += a_g0t135 * (g0t134);
  a_g0t1 += a_g0t134 * (-1.0/(g0t1*g0t1));
  double a_lambdaU1 = a_g0t133 * (Rational_3_4);
  a_g0t107 += a_g0t132 * (vetU_dD01);
  a_vetU_dD01 += a_g0t132 * (g0t107);
  a_g0t0 += a_g0t131 * (vetU0);
  a_vetU0 += a_g0t131 * (g0t0);
  a_f0_of_xx0 += a_g0t130 * (g0t41*g0t46);
  double a_g0t119 = a_g0t130 * (g0t18*g0t41);
  a_g0t18 += a_g0t130 * (g0t119*g0t41);
  a_g0t30 += a_g0t130 * (g0t41*g0t49);
  double a_g0t35 = a_g0t130 * (g0t41*(g0t37 + g0t53));
  a_g0t37 += a_g0t130 * (g0t35*g0t41);
  a_g0t39 += a_g0t130 * (g0t41*g0t57);
  a_g0t40 += a_g0t130 * (g0t41*g0t60);
  double a_g0t41 = a_g0t130 * (f0_of_xx0*g0t46 + g0t119*g0t18 + g0t30*g0t49 + g0t35*g0t37 + g0t35*g0t53 + g0t39*g0t57 + g0t40*g0t60 + g0t44 + g0t64);
  double a_g0t44 = a_g0t130 * (g0t41);
  double a_g0t46 = a_g0t130 * (f0_of_xx0*g0t41);
  double a_g0t49 = a_g0t130 * (g0t30*g0t41);
  a_g0t53 += a_g0t130 * (g0t35*g0t41);
  a_g0t57 += a_g0t130 * (g0t39*g0t41);
  a_g0t60 += a_g0t130 * (g0t40*g0t41);
  double a_g0t64 = a_g0t130 * (g0t41);
  a_g0t118 += a_g0t129 * (g0t41*g0t60);
  double a_g0t121 = a_g0t129 * (g0t41*g0t8);
  double a_g0t122 = a_g0t129 * (g0t127*g0t41);
  a_g0t126 += a_g0t129 * (g0t41);
  a_g0t127 += a_g0t129 * (g0t122*g0t41);
  a_g0t128 += a_g0t129 * (g0t41);
  a_g0t26 += a_g0t129 * (g0t34*g0t41);
  a_g0t31 += a_g0t129 * (g0t41*(g0t37 + g0t53));
  double a_g0t34 = a_g0t129 * (g0t26*g0t41);
  a_g0t37 += a_g0t129 * (g0t31*g0t41);
  a_g0t40 += a_g0t129 * (g0t41*g0t63);
  a_g0t41 += a_g0t129 * (g0t118*g0t60 + g0t121*g0t8 + g0t122*g0t127 + g0t126 + g0t128 + g0t26*g0t34 + g0t31*g0t37 + g0t31*g0t53 + g0t40*g0t63);
  a_g0t53 += a_g0t129 * (g0t31*g0t41);
  a_g0t60 += a_g0t129 * (g0t118*g0t41);
  a_g0t63 += a_g0t129 * (g0t40*g0t41);
  a_g0t8 += a_g0t129 * (g0t121*g0t41);
  double a_g0t123 = a_g0t128 * (g0t24);
  a_g0t24 += a_g0t128 * (g0t123);
  a_g0t13 += a_g0t127 * (g0t18);
  a_g0t18 += a_g0t127 * (g0t13);
  double a_g0t115 = a_g0t126 * (g0t8);
  a_g0t8 += a_g0t126 * (g0t115);
  a_g0t116 += a_g0t125 * (g0t41);
  a_g0t119 += a_g0t125 * (g0t41*g0t52);
  a_g0t120 += a_g0t125 * (g0t39*g0t41);
  a_g0t121 += a_g0t125 * (g0t18*g0t41);
  a_g0t122 += a_g0t125 * (g0t41*g0t48);
  a_g0t124 += a_g0t125 * (g0t41);
  a_g0t18 += a_g0t125 * (g0t121*g0t41);
  a_g0t30 += a_g0t125 * (g0t41*g0t57);
  a_g0t31 += a_g0t125 * (g0t41*g0t60);
  a_g0t35 += a_g0t125 * (g0t41*g0t63);
  a_g0t39 += a_g0t125 * (g0t120*g0t41);
  a_g0t41 += a_g0t125 * (g0t116 + g0t119*g0t52 + g0t120*g0t39 + g0t121*g0t18 + g0t122*g0t48 + g0t124 + g0t30*g0t57 + g0t31*g0t60 + g0t35*g0t63);
  a_g0t48 += a_g0t125 * (g0t122*g0t41);
  a_g0t52 += a_g0t125 * (g0t119*g0t41);
  a_g0t57 += a_g0t125 * (g0t30*g0t41);
  a_g0t60 += a_g0t125 * (g0t31*g0t41);
  a_g0t63 += a_g0t125 * (g0t35*g0t41);
  a_g0t123 += a_g0t124 * (g0t52);
  a_g0t52 += a_g0t124 * (g0t123);
  a_g0t62 += a_g0t123 * (g0t81);
  a_g0t81 += a_g0t123 * (g0t62);
  a_g0t39 += a_g0t122 * (g0t81);
  a_g0t81 += a_g0t122 * (g0t39);
  a_g0t35 += a_g0t121 * (g0t81);
  a_g0t81 += a_g0t121 * (g0t35);
  a_g0t13 += a_g0t120 * ((g0t52*g0t52));
  a_g0t52 += a_g0t120 * (2.0*g0t13*g0t52);
  a_g0t118 += a_g0t119 * (g0t47);
  a_g0t47 += a_g0t119 * (g0t118);
  a_g0t117 += a_g0t118 * (g0t13);
  a_g0t13 += a_g0t118 * (g0t117);
  double a_aDD11 = a_g0t117 * (g0t1);
  a_g0t1 += a_g0t117 * (aDD11);
  a_g0t115 += a_g0t116 * (g0t18);
  a_g0t18 += a_g0t116 * (g0t115);
  a_g0t14 += a_g0t115 * (g0t24);
  a_g0t24 += a_g0t115 * (g0t14);
  a_betU0 += a_g0t114 * (vetU0);
  a_vetU0 += a_g0t114 * (betU0);
  a_g0t108 += a_g0t113 * (Rational_3_4);
  a_g0t109 += a_g0t113 * ((Rational_3_4)*vetU0);
  a_g0t111 += a_g0t113 * ((Rational_3_4)*g0t112);
  a_g0t112 += a_g0t113 * ((Rational_3_4)*g0t111);
  a_vetU0 += a_g0t113 * ((Rational_3_4)*g0t109);
  a_vetU_dD00 += a_g0t113 * (Rational_3_4);
  a_g0t107 += a_g0t112 * (vetU1);
  a_vetU1 += a_g0t112 * (g0t107);
  a_f1_of_xx1__D1 += a_g0t111 * (g0t110);
  a_g0t110 += a_g0t111 * (f1_of_xx1__D1);
  a_f1_of_xx1 += a_g0t110 * (-1.0/(f1_of_xx1*f1_of_xx1));
  a_g0t107 += a_g0t109 * (2.0);
  a_g0t107 += a_g0t108 * (vetU_dD11);
  a_vetU_dD11 += a_g0t108 * (g0t107);
  a_f0_of_xx0 += a_g0t107 * (-1.0/(f0_of_xx0*f0_of_xx0));
  double a_g0t100 = a_g0t106 * (g0t18);
  a_g0t18 += a_g0t106 * (g0t100);
  a_g0t104 += a_g0t105 * (g0t87);
  double a_g0t73 = a_g0t105 * (hDD_dD001);
  a_g0t78 += a_g0t105 * (g0t84);
  a_g0t84 += a_g0t105 * (g0t78);
  a_g0t87 += a_g0t105 * (g0t104);
  a_hDD_dD001 += a_g0t105 * (g0t73);
  a_f0_of_xx0 += a_g0t104 * (f1_of_xx1__D1*hDD02);
  a_f1_of_xx1__D1 += a_g0t104 * (f0_of_xx0*hDD02);
  a_g0t33 += a_g0t104 * (hDD_dD021);
  double a_g0t96 = a_g0t104 * (1.0);
  double a_hDD02 = a_g0t104 * (f0_of_xx0*f1_of_xx1__D1);
  double a_hDD_dD021 = a_g0t104 * (g0t33);
  a_g0t100 += a_g0t103 * (g0t24);
  a_g0t24 += a_g0t103 * (g0t100);
  a_g0t69 += a_g0t102 * (g0t87);
  a_g0t78 += a_g0t102 * (g0t97);
  a_g0t87 += a_g0t102 * (g0t69);
  a_g0t97 += a_g0t102 * (g0t78);
  a_g0t100 += a_g0t101 * (g0t52);
  a_g0t52 += a_g0t101 * (g0t100);
  a_g0t71 += a_g0t100 * (Rational_4_3);
  a_g0t73 += a_g0t99 * (g0t98);
  a_g0t76 += a_g0t99 * (g0t87);
  a_g0t87 += a_g0t99 * (g0t76);
  a_g0t98 += a_g0t99 * (g0t73);
  a_g0t97 += a_g0t98 * (-1.0);
  a_f0_of_xx0 += a_g0t97 * (-f1_of_xx1*hDD_dD021 - f1_of_xx1__D1*hDD02);
  a_f1_of_xx1 += a_g0t97 * (-f0_of_xx0*hDD_dD021);
  a_f1_of_xx1__D1 += a_g0t97 * (-f0_of_xx0*hDD02);
  a_g0t96 += a_g0t97 * (1.0);
  a_hDD02 += a_g0t97 * (-f0_of_xx0*f1_of_xx1__D1);
  a_hDD_dD021 += a_g0t97 * (-f0_of_xx0*f1_of_xx1);
  double a_g0t38 = a_g0t96 * (hDD_dD120);
  double a_g0t54 = a_g0t96 * (hDD12);
  double a_hDD12 = a_g0t96 * (g0t54);
  double a_hDD_dD120 = a_g0t96 * (g0t38);
  a_g0t8 += a_g0t95 * (g0t82);
  double a_g0t82 = a_g0t95 * (g0t8);
  a_g0t73 += a_g0t94 * (hDD_dD000);
  a_g0t78 += a_g0t94 * (g0t93);
  a_g0t87 += a_g0t94 * (g0t92);
  a_g0t92 += a_g0t94 * (g0t87);
  a_g0t93 += a_g0t94 * (g0t78);
  a_hDD_dD000 += a_g0t94 * (g0t73);
  double a_g0t45 = a_g0t93 * (hDD_dD010);
  double a_hDD01 = a_g0t93 * (2.0);
  a_hDD_dD001 += a_g0t93 * (-1.0);
  double a_hDD_dD010 = a_g0t93 * (g0t45);
  double a_g0t23 = a_g0t92 * (2.0);
  a_g0t54 += a_g0t92 * (hDD_dD020);
  double a_hDD_dD020 = a_g0t92 * (g0t54);
  a_g0t47 += a_g0t91 * (g0t82);
  a_g0t82 += a_g0t91 * (g0t47);
  a_f0_of_xx0 += a_g0t90 * (1.0);
  a_g0t89 += a_g0t90 * (1.0);
  a_g0t73 += a_g0t89 * (g0t85);
  a_g0t78 += a_g0t89 * (g0t88);
  a_g0t85 += a_g0t89 * (g0t73);
  a_g0t86 += a_g0t89 * (g0t87);
  a_g0t87 += a_g0t89 * (g0t86);
  a_g0t88 += a_g0t89 * (g0t78);
  a_g0t1 += a_g0t88 * (hDD_dD111);
  double a_hDD_dD111 = a_g0t88 * (g0t1);
  a_g0t24 += a_g0t87 * (g0t72);
  a_g0t72 += a_g0t87 * (g0t24);
  a_f1_of_xx1__D1 += a_g0t86 * (g0t21*hDD12);
  double a_g0t21 = a_g0t86 * (f1_of_xx1__D1*hDD12);
  double a_g0t58 = a_g0t86 * (hDD_dD121);
  a_hDD12 += a_g0t86 * (f1_of_xx1__D1*g0t21);
  double a_hDD_dD121 = a_g0t86 * (g0t58);
  a_f0_of_xx0 += a_g0t85 * (2.0*hDD_dD011);
  a_g0t84 += a_g0t85 * (-1.0);
  double a_hDD_dD011 = a_g0t85 * (2.0*f0_of_xx0);
  a_g0t1 += a_g0t84 * (hDD_dD110);
  a_g0t45 += a_g0t84 * (hDD11 + 1.0);
  double a_hDD11 = a_g0t84 * (g0t45);
  double a_hDD_dD110 = a_g0t84 * (g0t1);
  a_g0t81 += a_g0t83 * (g0t82);
  a_g0t82 += a_g0t83 * (g0t81);
  a_g0t71 += a_g0t82 * (Rational_2_3);
  double a_g0t10 = a_g0t81 * (g0t2);
  double a_g0t2 = a_g0t81 * (g0t10);
  double a_g0t9 = a_g0t81 * (-1.0);
  a_g0t67 += a_g0t80 * (1.0);
  a_g0t79 += a_g0t80 * (1.0);
  a_g0t70 += a_g0t79 * (g0t73);
  a_g0t73 += a_g0t79 * (g0t70);
  a_g0t77 += a_g0t79 * (g0t78);
  a_g0t78 += a_g0t79 * (g0t77);
  a_g0t18 += a_g0t78 * (g0t72);
  a_g0t72 += a_g0t78 * (g0t18);
  a_g0t76 += a_g0t77 * (-1.0);
  a_g0t4 += a_g0t76 * (hDD_dD221);
  double a_g0t75 = a_g0t76 * (hDD22 + 1.0);
  double a_hDD22 = a_g0t76 * (g0t75);
  double a_hDD_dD221 = a_g0t76 * (g0t4);
  a_g0t21 += a_g0t75 * (g0t74);
  a_g0t74 += a_g0t75 * (g0t21);
  a_f1_of_xx1 += a_g0t74 * (f1_of_xx1__D1);
  a_f1_of_xx1__D1 += a_g0t74 * (f1_of_xx1);
  a_g0t72 += a_g0t73 * (g0t8);
  a_g0t8 += a_g0t73 * (g0t72);
  a_g0t71 += a_g0t72 * (Rational_1_2);
  double a_g0t12 = a_g0t71 * (-1.0/(g0t12*g0t12));
  a_g0t69 += a_g0t70 * (-1.0);
  a_g0t4 += a_g0t69 * (hDD_dD220);
  double a_g0t68 = a_g0t69 * (hDD22 + 1.0);
  a_hDD22 += a_g0t69 * (g0t68);
  double a_hDD_dD220 = a_g0t69 * (g0t4);
  a_g0t67 += a_g0t68 * (2.0);
  a_f0_of_xx0 += a_g0t67 * (g0t3);
  a_g0t3 += a_g0t67 * (f0_of_xx0);
  double a_alpha_dD1 = a_g0t66 * (Rational_3_4);
  double a_cf_dD1 = a_g0t66 * ((Rational_3_4)*g0t42);
  double a_g0t42 = a_g0t66 * ((Rational_3_4)*cf_dD1);
  a_g0t22 += a_g0t65 * (-g0t51);
  a_g0t37 += a_g0t65 * (-g0t56);
  a_g0t44 += a_g0t65 * (-2.0);
  a_g0t45 += a_g0t65 * (-g0t46);
  a_g0t46 += a_g0t65 * (-g0t45);
  a_g0t49 += a_g0t65 * (-g0t50);
  a_g0t50 += a_g0t65 * (-g0t49);
  a_g0t51 += a_g0t65 * (-g0t22);
  a_g0t53 += a_g0t65 * (-g0t56);
  a_g0t56 += a_g0t65 * (-g0t37 - g0t53);
  a_g0t57 += a_g0t65 * (-g0t59);
  a_g0t59 += a_g0t65 * (-g0t57);
  a_g0t60 += a_g0t65 * (-g0t61);
  a_g0t61 += a_g0t65 * (-g0t60);
  a_g0t64 += a_g0t65 * (-2.0);
  a_g0t62 += a_g0t64 * (g0t63);
  a_g0t63 += a_g0t64 * (g0t62);
  a_g0t24 += a_g0t63 * (g0t52);
  a_g0t52 += a_g0t63 * (g0t24);
  a_g0t13 += a_g0t62 * (g0t27);
  a_g0t27 += a_g0t62 * (g0t13);
  a_g0t13 += a_g0t61 * (g0t59);
  a_g0t59 += a_g0t61 * (g0t13);
  a_g0t18 += a_g0t60 * (g0t52);
  a_g0t52 += a_g0t60 * (g0t18);
  double a_aDD12 = a_g0t59 * (g0t58);
  a_g0t58 += a_g0t59 * (aDD12);
  a_g0t38 += a_g0t58 * (2.0);
  a_g0t24 += a_g0t57 * (g0t48);
  a_g0t48 += a_g0t57 * (g0t24);
  a_g0t13 += a_g0t56 * (g0t55);
  a_g0t55 += a_g0t56 * (g0t13);
  double a_aDD02 = a_g0t55 * (g0t54);
  a_g0t54 += a_g0t55 * (aDD02);
  a_f1_of_xx1 += a_g0t54 * (g0t45);
  a_g0t45 += a_g0t54 * (f1_of_xx1);
  a_g0t52 += a_g0t53 * (g0t8);
  a_g0t8 += a_g0t53 * (g0t52);
  a_g0t1 += a_g0t52 * (g0t23*hDD01);
  a_g0t10 += a_g0t52 * (-g0t38*hDD12);
  a_g0t23 += a_g0t52 * (g0t1*hDD01);
  a_g0t38 += a_g0t52 * (-g0t10*hDD12);
  a_hDD01 += a_g0t52 * (g0t1*g0t23);
  a_hDD12 += a_g0t52 * (-g0t10*g0t38);
  a_g0t18 += a_g0t51 * (g0t48);
  a_g0t48 += a_g0t51 * (g0t18);
  double a_aDD01 = a_g0t50 * (g0t45);
  a_g0t45 += a_g0t50 * (aDD01);
  a_g0t48 += a_g0t49 * (g0t8);
  a_g0t8 += a_g0t49 * (g0t48);
  a_g0t13 += a_g0t48 * (g0t47);
  a_g0t47 += a_g0t48 * (g0t13);
  a_g0t10 += a_g0t47 * (g0t5);
  double a_g0t11 = a_g0t47 * (-1.0);
  double a_g0t5 = a_g0t47 * (g0t10);
  a_aDD01 += a_g0t46 * (g0t20);
  a_g0t20 += a_g0t46 * (aDD01);
  a_f0_of_xx0 += a_g0t45 * (2.0);
  a_g0t14 += a_g0t44 * (g0t29);
  a_g0t29 += a_g0t44 * (g0t14);
  double a_alpha_dD0 = a_g0t43 * (Rational_3_4);
  double a_cf_dD0 = a_g0t43 * ((Rational_3_4)*g0t42);
  a_g0t42 += a_g0t43 * ((Rational_3_4)*cf_dD0);
  double a_cf = a_g0t42 * (-g0t41/(cf*cf));
  a_g0t41 += a_g0t42 * ((1.0 / cf));
  a_alpha += a_g0t41 * (3.0);
  a_g0t13 += a_g0t40 * (g0t39);
  a_g0t39 += a_g0t40 * (g0t13);
  a_aDD12 += a_g0t39 * (g0t38);
  a_g0t38 += a_g0t39 * (aDD12);
  a_f1_of_xx1 += a_g0t38 * (g0t1);
  a_g0t1 += a_g0t38 * (f1_of_xx1);
  a_g0t18 += a_g0t37 * (g0t24);
  a_g0t24 += a_g0t37 * (g0t18);
  a_g0t35 += a_g0t36 * (4.0);
  a_g0t13 += a_g0t35 * (g0t34);
  a_g0t34 += a_g0t35 * (g0t13);
  a_aDD02 += a_g0t34 * (g0t33);
  a_g0t33 += a_g0t34 * (aDD02);
  a_f0_of_xx0 += a_g0t33 * (f1_of_xx1);
  a_f1_of_xx1 += a_g0t33 * (f0_of_xx0);
  a_g0t24 += a_g0t32 * (g0t8);
  a_g0t8 += a_g0t32 * (g0t24);
  a_g0t13 += a_g0t31 * (g0t30);
  a_g0t30 += a_g0t31 * (g0t13);
  a_aDD01 += a_g0t30 * (f0_of_xx0);
  a_f0_of_xx0 += a_g0t30 * (aDD01);
  a_g0t18 += a_g0t29 * (g0t8);
  a_g0t8 += a_g0t29 * (g0t18);
  a_g0t26 += a_g0t28 * (g0t27);
  a_g0t27 += a_g0t28 * (g0t26);
  double a_aDD22 = a_g0t27 * (g0t4);
  a_g0t4 += a_g0t27 * (aDD22);
  a_g0t13 += a_g0t26 * (g0t25);
  a_g0t25 += a_g0t26 * (g0t13);
  a_g0t24 += a_g0t25 * (2.0*g0t24);
  a_f0_of_xx0 += a_g0t24 * (-g0t2*g0t23);
  a_f1_of_xx1 += a_g0t24 * (g0t17*hDD01);
  double a_g0t17 = a_g0t24 * (f1_of_xx1*hDD01);
  a_g0t2 += a_g0t24 * (-f0_of_xx0*g0t23);
  a_g0t23 += a_g0t24 * (-f0_of_xx0*g0t2);
  a_hDD01 += a_g0t24 * (f1_of_xx1*g0t17);
  a_f1_of_xx1 += a_g0t23 * (hDD02);
  a_hDD02 += a_g0t23 * (f1_of_xx1);
  a_aDD11 += a_g0t22 * (g0t21);
  a_g0t21 += a_g0t22 * (aDD11);
  a_g0t1 += a_g0t21 * (2.0);
  a_g0t13 += a_g0t20 * (g0t19);
  a_g0t19 += a_g0t20 * (g0t13);
  a_g0t18 += a_g0t19 * (2.0*g0t18);
  a_f0_of_xx0 += a_g0t18 * (-g0t5*hDD01);
  a_g0t17 += a_g0t18 * (g0t3*hDD02);
  a_g0t3 += a_g0t18 * (g0t17*hDD02);
  a_g0t5 += a_g0t18 * (-f0_of_xx0*hDD01);
  a_hDD01 += a_g0t18 * (-f0_of_xx0*g0t5);
  a_hDD02 += a_g0t18 * (g0t17*g0t3);
  a_g0t16 += a_g0t17 * (hDD12);
  a_hDD12 += a_g0t17 * (g0t16);
  a_f0_of_xx0 += a_g0t16 * (3.0*(f0_of_xx0*f0_of_xx0));
  a_g0t14 += a_g0t15 * ((g0t8*g0t8));
  a_g0t8 += a_g0t15 * (2.0*g0t14*g0t8);
  double a_aDD00 = a_g0t14 * (g0t13);
  a_g0t13 += a_g0t14 * (aDD00);
  a_g0t12 += a_g0t13 * (-2.0/(g0t12*g0t12*g0t12));
  a_g0t10 += a_g0t12 * (g0t2*g0t5 - g0t7);
  a_g0t11 += a_g0t12 * (-g0t2);
  a_g0t2 += a_g0t12 * (g0t10*g0t5 - g0t11);
  a_g0t3 += a_g0t12 * (2.0*g0t6*hDD01*hDD02*hDD12);
  a_g0t5 += a_g0t12 * (g0t10*g0t2 - g0t9);
  a_g0t6 += a_g0t12 * (2.0*g0t3*hDD01*hDD02*hDD12);
  double a_g0t7 = a_g0t12 * (-g0t10);
  a_g0t9 += a_g0t12 * (-g0t5);
  a_hDD01 += a_g0t12 * (2.0*g0t3*g0t6*hDD02*hDD12);
  a_hDD02 += a_g0t12 * (2.0*g0t3*g0t6*hDD01*hDD12);
  a_hDD12 += a_g0t12 * (2.0*g0t3*g0t6*hDD01*hDD02);
  a_g0t4 += a_g0t11 * ((hDD02*hDD02));
  a_hDD02 += a_g0t11 * (2.0*g0t4*hDD02);
  double a_hDD00 = a_g0t10 * (1.0);
  a_g0t1 += a_g0t9 * ((hDD01*hDD01));
  a_hDD01 += a_g0t9 * (2.0*g0t1*hDD01);
  a_g0t2 += a_g0t8 * (g0t5);
  a_g0t5 += a_g0t8 * (g0t2);
  a_g0t7 += a_g0t8 * (-1.0);
  a_g0t3 += a_g0t7 * (g0t6*(hDD12*hDD12));
  a_g0t6 += a_g0t7 * (g0t3*(hDD12*hDD12));
  a_hDD12 += a_g0t7 * (2.0*g0t3*g0t6*hDD12);
  a_f0_of_xx0 += a_g0t6 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_g0t4 += a_g0t5 * (hDD22 + 1.0);
  a_hDD22 += a_g0t5 * (g0t4);
  a_g0t1 += a_g0t4 * (g0t3);
  a_g0t3 += a_g0t4 * (g0t1);
  a_f1_of_xx1 += a_g0t3 * (2.0*f1_of_xx1);
  a_g0t1 += a_g0t2 * (hDD11 + 1.0);
  a_hDD11 += a_g0t2 * (g0t1);
  a_f0_of_xx0 += a_g0t1 * (2.0*f0_of_xx0);
  double a_lambdaU0 = a_g0t0 * (Rational_3_4);
  red[0 * 64 + lane] = a_aDD00;
  red[1 * 64 + lane] = a_aDD01;
  red[2 * 64 + lane] = a_aDD02;
  red[3 * 64 + lane] = a_aDD11;
  red[4 * 64 + lane] = a_aDD12;
  red[5 * 64 + lane] = a_aDD22;
  red[6 * 64 + lane] = a_alpha;
  red[7 * 64 + lane] = a_alpha_dD0;
  red[8 * 64 + lane] = a_alpha_dD1;
  red[9 * 64 + lane] = a_betU0;
  red[10 * 64 + lane] = a_betU1;
  red[11 * 64 + lane] = a_betU2;
  red[12 * 64 + lane] = (betaU0 > 0.0) ? a_betU_dupD00 : 0.0;
  red[13 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_betU_dupD00;
  red[14 * 64 + lane] = (betaU1 > 0.0) ? a_betU_dupD01 : 0.0;
  red[15 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_betU_dupD01;
  red[16 * 64 + lane] = (betaU0 > 0.0) ? a_betU_dupD10 : 0.0;
  red[17 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_betU_dupD10;
  red[18 * 64 + lane] = (betaU1 > 0.0) ? a_betU_dupD11 : 0.0;
  red[19 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_betU_dupD11;
  red[20 * 64 + lane] = (betaU0 > 0.0) ? a_betU_dupD20 : 0.0;
  red[21 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_betU_dupD20;
  red[22 * 64 + lane] = (betaU1 > 0.0) ? a_betU_dupD21 : 0.0;
  red[23 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_betU_dupD21;
  red[24 * 64 + lane] = a_cf;
  red[25 * 64 + lane] = a_cf_dD0;
  red[26 * 64 + lane] = a_cf_dD1;
  red[27 * 64 + lane] = a_hDD00;
  red[28 * 64 + lane] = a_hDD01;
  red[29 * 64 + lane] = a_hDD02;
  red[30 * 64 + lane] = a_hDD11;
  red[31 * 64 + lane] = a_hDD12;
  red[32 * 64 + lane] = a_hDD22;
  red[33 * 64 + lane] = a_hDD_dD000;
  red[34 * 64 + lane] = a_hDD_dD001;
  red[35 * 64 + lane] = a_hDD_dD010;
  red[36 * 64 + lane] = a_hDD_dD011;
  red[37 * 64 + lane] = a_hDD_dD020;
  red[38 * 64 + lane] = a_hDD_dD021;
  red[39 * 64 + lane] = a_hDD_dD110;
  red[40 * 64 + lane] = a_hDD_dD111;
  red[41 * 64 + lane] = a_hDD_dD120;
  red[42 * 64 + lane] = a_hDD_dD121;
  red[43 * 64 + lane] = a_hDD_dD220;
  red[44 * 64 + lane] = a_hDD_dD221;
  red[45 * 64 + lane] = a_lambdaU0;
  red[46 * 64 + lane] = a_lambdaU1;
  red[47 * 64 + lane] = a_lambdaU2;
  red[48 * 64 + lane] = a_trK_dD0;
  red[49 * 64 + lane] = a_trK_dD1;
  red[50 * 64 + lane] = a_vetU0;
  red[51 * 64 + lane] = a_vetU1;
  red[52 * 64 + lane] = a_vetU2;
  red[53 * 64 + lane] = a_vetU_dD00;
  red[54 * 64 + lane] = a_vetU_dD01;
  red[55 * 64 + lane] = a_vetU_dD10;
  red[56 * 64 + lane] = a_vetU_dD11;
  red[57 * 64 + lane] = a_vetU_dD20;
  red[58 * 64 + lane] = a_vetU_dD21;
  red[59 * 64 + lane] = a_vetU_dDD000;
  red[60 * 64 + lane] = a_vetU_dDD001;
  red[61 * 64 + lane] = a_vetU_dDD011;
  red[62 * 64 + lane] = a_vetU_dDD100;
  red[63 * 64 + lane] = a_vetU_dDD101;
  red[64 * 64 + lane] = a_vetU_dDD111;
  red[65 * 64 + lane] = a_vetU_dDD200;
  red[66 * 64 + lane] = a_vetU_dDD201;
  red[67 * 64 + lane] = a_vetU_dDD211;
  break;
  }
  case 1: { // alpha, lambdaU0, lambdaU1, lambdaU2, vetU0, vetU1, vetU2
  const double aDD00 = in[idx];
  const double aDD01 = in[1 * Ntot + idx];
  const double aDD02 = in[2 * Ntot + idx];
  const double aDD11 = in[3 * Ntot + idx];
  const double aDD12 = in[4 * Ntot + idx];
  const double aDD22 = in[5 * Ntot + idx];
  const double alpha = in[6 * Ntot + idx];
  const double alpha_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[6 * Ntot + idx + (1)] - in[6 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2)] - in[6 * Ntot + idx + (-2)]));
  const double alpha_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[6 * Ntot + idx + (1 * s1)] - in[6 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2 * s1)] - in[6 * Ntot + idx + (-2 * s1)]));
  const double alpha_dupD0 = p.invdxx0 * (uw0[0] * in[6 * Ntot + idx + (-3)] + uw0[1] * in[6 * Ntot + idx + (-2)] + uw0[2] * in[6 * Ntot + idx + (-1)] + uw0[3] * in[6 * Ntot + idx] + uw0[4] * in[6 * Ntot + idx + (1)] + uw0[5] * in[6 * Ntot + idx + (2)] + uw0[6] * in[6 * Ntot + idx + (3)]);
  const double alpha_dupD1 = p.invdxx1 * (uw1[0] * in[6 * Ntot + idx + (-3 * s1)] + uw1[1] * in[6 * Ntot + idx + (-2 * s1)] + uw1[2] * in[6 * Ntot + idx + (-1 * s1)] + uw1[3] * in[6 * Ntot + idx] + uw1[4] * in[6 * Ntot + idx + (1 * s1)] + uw1[5] * in[6 * Ntot + idx + (2 * s1)] + uw1[6] * in[6 * Ntot + idx + (3 * s1)]);
  const double betU0 = in[7 * Ntot + idx];
  const double betU1 = in[8 * Ntot + idx];
  const double betU2 = in[9 * Ntot + idx];
  const double cf = in[10 * Ntot + idx];
  const double cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1)] - in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] - in[10 * Ntot + idx + (-2)]));
  const double cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] - in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] - in[10 * Ntot + idx + (-2 * s1)]));
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double hDD00 = in[11 * Ntot + idx];
  const double hDD01 = in[12 * Ntot + idx];
  const double hDD02 = in[13 * Ntot + idx];
  const double hDD11 = in[14 * Ntot + idx];
  const double hDD12 = in[15 * Ntot + idx];
  const double hDD22 = in[16 * Ntot + idx];
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  const double lambdaU0 = in[17 * Ntot + idx];
  const double lambdaU1 = in[18 * Ntot + idx];
  const double lambdaU2 = in[19 * Ntot + idx];
  const double lambdaU_dupD00 = p.invdxx0 * (uw0[0] * in[17 * Ntot + idx + (-3)] + uw0[1] * in[17 * Ntot + idx + (-2)] + uw0[2] * in[17 * Ntot + idx + (-1)] + uw0[3] * in[17 * Ntot + idx] + uw0[4] * in[17 * Ntot + idx + (1)] + uw0[5] * in[17 * Ntot + idx + (2)] + uw0[6] * in[17 * Ntot + idx + (3)]);
  const double lambdaU_dupD01 = p.invdxx1 * (uw1[0] * in[17 * Ntot + idx + (-3 * s1)] + uw1[1] * in[17 * Ntot + idx + (-2 * s1)] + uw1[2] * in[17 * Ntot + idx + (-1 * s1)] + uw1[3] * in[17 * Ntot + idx] + uw1[4] * in[17 * Ntot + idx + (1 * s1)] + uw1[5] * in[17 * Ntot + idx + (2 * s1)] + uw1[6] * in[17 * Ntot + idx + (3 * s1)]);
  const double lambdaU_dupD10 = p.invdxx0 * (uw0[0] * in[18 * Ntot + idx + (-3)] + uw0[1] * in[18 * Ntot + idx + (-2)] + uw0[2] * in[18 * Ntot + idx + (-1)] + uw0[3] * in[18 * Ntot + idx] + uw0[4] * in[18 * Ntot + idx + (1)] + uw0[5] * in[18 * Ntot + idx + (2)] + uw0[6] * in[18 * Ntot + idx + (3)]);
  const double lambdaU_dupD11 = p.invdxx1 * (uw1[0] * in[18 * Ntot + idx + (-3 * s1)] + uw1[1] * in[18 * Ntot + idx + (-2 * s1)] + uw1[2] * in[18 * Ntot + idx + (-1 * s1)] + uw1[3] * in[18 * Ntot + idx] + uw1[4] * in[18 * Ntot + idx + (1 * s1)] + uw1[5] * in[18 * Ntot + idx + (2 * s1)] + uw1[6] * in[18 * Ntot + idx + (3 * s1)]);
  const double lambdaU_dupD20 = p.invdxx0 * (uw0[0] * in[19 * Ntot + idx + (-3)] + uw0[1] * in[19 * Ntot + idx + (-2)] + uw0[2] * in[19 * Ntot + idx + (-1)] + uw0[3] * in[19 * Ntot + idx] + uw0[4] * in[19 * Ntot + idx + (1)] + uw0[5] * in[19 * Ntot + idx + (2)] + uw0[6] * in[19 * Ntot + idx + (3)]);
  const double lambdaU_dupD21 = p.invdxx1 * (uw1[0] * in[19 * Ntot + idx + (-3 * s1)] + uw1[1] * in[19 * Ntot + idx + (-2 * s1)] + uw1[2] * in[19 * Ntot + idx + (-1 * s1)] + uw1[3] * in[19 * Ntot + idx] + uw1[4] * in[19 * Ntot + idx + (1 * s1)] + uw1[5] * in[19 * Ntot + idx + (2 * s1)] + uw1[6] * in[19 * Ntot + idx + (3 * s1)]);
  const double trK = in[20 * Ntot + idx];
  const double trK_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1)] - in[20 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2)] - in[20 * Ntot + idx + (-2)]));
  const double trK_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1 * s1)] - in[20 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2 * s1)] - in[20 * Ntot + idx + (-2 * s1)]));
  const double vetU0 = in[21 * Ntot + idx];
  const double vetU1 = in[22 * Ntot + idx];
  const double vetU2 = in[23 * Ntot + idx];
  const double vetU_dD00 = p.invdxx0 * ((2.0 / 3.0) * (in[21 * Ntot + idx + (1)] - in[21 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2)] - in[21 * Ntot + idx + (-2)]));
  const double vetU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (in[21 * Ntot + idx + (1 * s1)] - in[21 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2 * s1)] - in[21 * Ntot + idx + (-2 * s1)]));
  const double vetU_dD10 = p.invdxx0 * ((2.0 / 3.0) * (in[22 * Ntot + idx + (1)] - in[22 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2)] - in[22 * Ntot + idx + (-2)]));
  const double vetU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (in[22 * Ntot + idx + (1 * s1)] - in[22 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2 * s1)] - in[22 * Ntot + idx + (-2 * s1)]));
  const double vetU_dD20 = p.invdxx0 * ((2.0 / 3.0) * (in[23 * Ntot + idx + (1)] - in[23 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2)] - in[23 * Ntot + idx + (-2)]));
  const double vetU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (in[23 * Ntot + idx + (1 * s1)] - in[23 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2 * s1)] - in[23 * Ntot + idx + (-2 * s1)]));
  const double vetU_dDD000 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[21 * Ntot + idx] + (4.0 / 3.0) * (in[21 * Ntot + idx + (1)] + in[21 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2)] + in[21 * Ntot + idx + (-2)]));
  const double vetU_dDD001 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[21 * Ntot + idx + (1 + 1 * s1)] - in[21 * Ntot + idx + (1 + -1 * s1)]) - (in[21 * Ntot + idx + (-1 + 1 * s1)] - in[21 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[21 * Ntot + idx + (1 + 2 * s1)] - in[21 * Ntot + idx + (1 + -2 * s1)]) - (in[21 * Ntot + idx + (-1 + 2 * s1)] - in[21 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[21 * Ntot + idx + (2 + 1 * s1)] - in[21 * Ntot + idx + (2 + -1 * s1)]) - (in[21 * Ntot + idx + (-2 + 1 * s1)] - in[21 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[21 * Ntot + idx + (2 + 2 * s1)] - in[21 * Ntot + idx + (2 + -2 * s1)]) - (in[21 * Ntot + idx + (-2 + 2 * s1)] - in[21 * Ntot + idx + (-2 + -2 * s1)])));
  const double vetU_dDD011 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[21 * Ntot + idx] + (4.0 / 3.0) * (in[21 * Ntot + idx + (1 * s1)] + in[21 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2 * s1)] + in[21 * Ntot + idx + (-2 * s1)]));
  const double vetU_dDD100 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[22 * Ntot + idx] + (4.0 / 3.0) * (in[22 * Ntot + idx + (1)] + in[22 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2)] + in[22 * Ntot + idx + (-2)]));
  const double vetU_dDD101 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[22 * Ntot + idx + (1 + 1 * s1)] - in[22 * Ntot + idx + (1 + -1 * s1)]) - (in[22 * Ntot + idx + (-1 + 1 * s1)] - in[22 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[22 * Ntot + idx + (1 + 2 * s1)] - in[22 * Ntot + idx + (1 + -2 * s1)]) - (in[22 * Ntot + idx + (-1 + 2 * s1)] - in[22 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[22 * Ntot + idx + (2 + 1 * s1)] - in[22 * Ntot + idx + (2 + -1 * s1)]) - (in[22 * Ntot + idx + (-2 + 1 * s1)] - in[22 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[22 * Ntot + idx + (2 + 2 * s1)] - in[22 * Ntot + idx + (2 + -2 * s1)]) - (in[22 * Ntot + idx + (-2 + 2 * s1)] - in[22 * Ntot + idx + (-2 + -2 * s1)])));
  const double vetU_dDD111 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[22 * Ntot + idx] + (4.0 / 3.0) * (in[22 * Ntot + idx + (1 * s1)] + in[22 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2 * s1)] + in[22 * Ntot + idx + (-2 * s1)]));
  const double vetU_dDD200 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[23 * Ntot + idx] + (4.0 / 3.0) * (in[23 * Ntot + idx + (1)] + in[23 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2)] + in[23 * Ntot + idx + (-2)]));
  const double vetU_dDD201 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[23 * Ntot + idx + (1 + 1 * s1)] - in[23 * Ntot + idx + (1 + -1 * s1)]) - (in[23 * Ntot + idx + (-1 + 1 * s1)] - in[23 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[23 * Ntot + idx + (1 + 2 * s1)] - in[23 * Ntot + idx + (1 + -2 * s1)]) - (in[23 * Ntot + idx + (-1 + 2 * s1)] - in[23 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[23 * Ntot + idx + (2 + 1 * s1)] - in[23 * Ntot + idx + (2 + -1 * s1)]) - (in[23 * Ntot + idx + (-2 + 1 * s1)] - in[23 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[23 * Ntot + idx + (2 + 2 * s1)] - in[23 * Ntot + idx + (2 + -2 * s1)]) - (in[23 * Ntot + idx + (-2 + 2 * s1)] - in[23 * Ntot + idx + (-2 + -2 * s1)])));
  const double vetU_dDD211 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[23 * Ntot + idx] + (4.0 / 3.0) * (in[23 * Ntot + idx + (1 * s1)] + in[23 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2 * s1)] + in[23 * Ntot + idx + (-2 * s1)]));
  const double vetU_dupD00 = p.invdxx0 * (uw0[0] * in[21 * Ntot + idx + (-3)] + uw0[1] * in[21 * Ntot + idx + (-2)] + uw0[2] * in[21 * Ntot + idx + (-1)] + uw0[3] * in[21 * Ntot + idx] + uw0[4] * in[21 * Ntot + idx + (1)] + uw0[5] * in[21 * Ntot + idx + (2)] + uw0[6] * in[21 * Ntot + idx + (3)]);
  const double vetU_dupD01 = p.invdxx1 * (uw1[0] * in[21 * Ntot + idx + (-3 * s1)] + uw1[1] * in[21 * Ntot + idx + (-2 * s1)] + uw1[2] * in[21 * Ntot + idx + (-1 * s1)] + uw1[3] * in[21 * Ntot + idx] + uw1[4] * in[21 * Ntot + idx + (1 * s1)] + uw1[5] * in[21 * Ntot + idx + (2 * s1)] + uw1[6] * in[21 * Ntot + idx + (3 * s1)]);
  const double vetU_dupD10 = p.invdxx0 * (uw0[0] * in[22 * Ntot + idx + (-3)] + uw0[1] * in[22 * Ntot + idx + (-2)] + uw0[2] * in[22 * Ntot + idx + (-1)] + uw0[3] * in[22 * Ntot + idx] + uw0[4] * in[22 * Ntot + idx + (1)] + uw0[5] * in[22 * Ntot + idx + (2)] + uw0[6] * in[22 * Ntot + idx + (3)]);
  const double vetU_dupD11 = p.invdxx1 * (uw1[0] * in[22 * Ntot + idx + (-3 * s1)] + uw1[1] * in[22 * Ntot + idx + (-2 * s1)] + uw1[2] * in[22 * Ntot + idx + (-1 * s1)] + uw1[3] * in[22 * Ntot + idx] + uw1[4] * in[22 * Ntot + idx + (1 * s1)] + uw1[5] * in[22 * Ntot + idx + (2 * s1)] + uw1[6] * in[22 * Ntot + idx + (3 * s1)]);
  const double vetU_dupD20 = p.invdxx0 * (uw0[0] * in[23 * Ntot + idx + (-3)] + uw0[1] * in[23 * Ntot + idx + (-2)] + uw0[2] * in[23 * Ntot + idx + (-1)] + uw0[3] * in[23 * Ntot + idx] + uw0[4] * in[23 * Ntot + idx + (1)] + uw0[5] * in[23 * Ntot + idx + (2)] + uw0[6] * in[23 * Ntot + idx + (3)]);
  const double vetU_dupD21 = p.invdxx1 * (uw1[0] * in[23 * Ntot + idx + (-3 * s1)] + uw1[1] * in[23 * Ntot + idx + (-2 * s1)] + uw1[2] * in[23 * Ntot + idx + (-1 * s1)] + uw1[3] * in[23 * Ntot + idx] + uw1[4] * in[23 * Ntot + idx + (1 * s1)] + uw1[5] * in[23 * Ntot + idx + (2 * s1)] + uw1[6] * in[23 * Ntot + idx + (3 * s1)]);
  const double g1t0 = 2.0*alpha;
  const double g1t1 = (1.0 / f0_of_xx0);
  const double g1t2 = g1t1*vetU1;
  const double g1t3 = 3.0*alpha/cf;
  const double g1t4 = alpha_dD0 + cf_dD0*g1t3;
  const double g1t5 = (f0_of_xx0*f0_of_xx0);
  const double g1t6 = g1t5*hDD11 + g1t5;
  const double g1t7 = (f1_of_xx1*f1_of_xx1);
  const double g1t8 = g1t5*g1t7;
  const double g1t9 = g1t8*hDD22 + g1t8;
  const double g1t10 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g1t11 = g1t10*g1t7*(hDD12*hDD12);
  const double g1t12 = -g1t11 + g1t6*g1t9;
  const double g1t13 = g1t5*(hDD01*hDD01);
  const double g1t14 = hDD00 + 1.0;
  const double g1t15 = g1t8*(hDD02*hDD02);
  const double g1t16 = 2.0*g1t10*g1t7*hDD01*hDD02*hDD12 - g1t11*g1t14 - g1t13*g1t9 + g1t14*g1t6*g1t9 - g1t15*g1t6;
  const double g1t17 = (1.0 / (g1t16*g1t16));
  const double g1t18 = aDD00*g1t17;
  const double g1t19 = (g1t12*g1t12)*g1t18;
  const double g1t20 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g1t21 = g1t20*hDD12;
  const double g1t22 = -f0_of_xx0*g1t9*hDD01 + g1t21*g1t7*hDD02;
  const double g1t23 = (g1t22*g1t22);
  const double g1t24 = 2.0*g1t5;
  const double g1t25 = aDD11*g1t17;
  const double g1t26 = g1t24*g1t25;
  const double g1t27 = f1_of_xx1*hDD02;
  const double g1t28 = -f0_of_xx0*g1t27*g1t6 + f1_of_xx1*g1t21*hDD01;
  const double g1t29 = (g1t28*g1t28);
  const double g1t30 = aDD22*g1t17*g1t8;
  const double g1t31 = g1t29*g1t30;
  const double g1t32 = g1t12*g1t22;
  const double g1t33 = aDD01*g1t17;
  const double g1t34 = f0_of_xx0*g1t33;
  const double g1t35 = 4.0*g1t34;
  const double g1t36 = g1t12*g1t28;
  const double g1t37 = f0_of_xx0*f1_of_xx1;
  const double g1t38 = aDD02*g1t17;
  const double g1t39 = g1t37*g1t38;
  const double g1t40 = 4.0*g1t39;
  const double g1t41 = g1t22*g1t28;
  const double g1t42 = f1_of_xx1*g1t5;
  const double g1t43 = aDD12*g1t17;
  const double g1t44 = g1t42*g1t43;
  const double g1t45 = 4.0*g1t44;
  const double g1t46 = alpha_dD1 + cf_dD1*g1t3;
  const double g1t47 = g1t18*g1t32;
  const double g1t48 = 2.0*f0_of_xx0;
  const double g1t49 = g1t23*g1t33;
  const double g1t50 = g1t14*g1t9 - g1t15;
  const double g1t51 = g1t12*g1t50;
  const double g1t52 = g1t33*g1t48;
  const double g1t53 = g1t22*g1t50;
  const double g1t54 = -g1t14*g1t42*hDD12 + g1t27*g1t5*hDD01;
  const double g1t55 = g1t12*g1t54;
  const double g1t56 = f1_of_xx1*g1t48;
  const double g1t57 = g1t38*g1t56;
  const double g1t58 = g1t28*g1t50;
  const double g1t59 = 2.0*g1t42;
  const double g1t60 = g1t43*g1t59;
  const double g1t61 = g1t22*g1t54;
  const double g1t62 = g1t28*g1t54;
  const double g1t63 = g1t30*g1t62;
  const double g1t64 = -g1t26*g1t53 - g1t41*g1t57 - 2.0*g1t47 - g1t48*g1t49 - g1t51*g1t52 - g1t55*g1t57 - g1t58*g1t60 - g1t60*g1t61 - 2.0*g1t63;
  const double g1t65 = g1t1*vetU_dD11;
  const double g1t66 = 2.0*g1t1;
  const double g1t67 = g1t66*vetU0;
  const double g1t68 = (1.0 / f1_of_xx1);
  const double g1t69 = f1_of_xx1__D1*g1t68;
  const double g1t70 = g1t2*g1t69 + g1t65 + g1t67 + vetU_dD00;
  const double g1t71 = f0_of_xx0*g1t7;
  const double g1t72 = 2.0*g1t71;
  const double g1t73 = g1t72*hDD22 + g1t72 + g1t8*hDD_dD220;
  const double g1t74 = -g1t73;
  const double g1t75 = (1.0 / g1t16);
  const double g1t76 = g1t12*g1t75;
  const double g1t77 = (Rational_1_2)*g1t76;
  const double g1t78 = f1_of_xx1*f1_of_xx1__D1;
  const double g1t79 = g1t24*g1t78;
  const double g1t80 = g1t79*hDD22 + g1t79 + g1t8*hDD_dD221;
  const double g1t81 = -g1t80;
  const double g1t82 = (Rational_1_2)*g1t75;
  const double g1t83 = g1t22*g1t82;
  const double g1t84 = g1t74*g1t77 + g1t81*g1t83;
  const double g1t85 = g1t71 + g1t84;
  const double g1t86 = -g1t13 + g1t14*g1t6;
  const double g1t87 = g1t75*g1t86;
  const double g1t88 = (Rational_2_3)*g1t87;
  const double g1t89 = g1t48*hDD11 + g1t48 + g1t5*hDD_dD110;
  const double g1t90 = 2.0*f0_of_xx0*hDD_dD011 - g1t89;
  const double g1t91 = f1_of_xx1__D1*g1t24*hDD12 + g1t59*hDD_dD121;
  const double g1t92 = g1t28*g1t82;
  const double g1t93 = g1t5*hDD_dD111;
  const double g1t94 = g1t77*g1t90 + g1t83*g1t93 + g1t91*g1t92;
  const double g1t95 = f0_of_xx0 + g1t94;
  const double g1t96 = g1t50*g1t75;
  const double g1t97 = (Rational_2_3)*g1t96;
  const double g1t98 = 2.0*g1t27 + g1t56*hDD_dD020;
  const double g1t99 = g1t48*hDD_dD010 + 2.0*hDD01 - hDD_dD001;
  const double g1t100 = g1t77*hDD_dD000 + g1t83*g1t99 + g1t92*g1t98;
  const double g1t101 = (Rational_2_3)*g1t76;
  const double g1t102 = g1t42*hDD_dD120 + g1t56*hDD12;
  const double g1t103 = -f0_of_xx0*f1_of_xx1*hDD_dD021 - f0_of_xx0*f1_of_xx1__D1*hDD02 + g1t102;
  const double g1t104 = -g1t103;
  const double g1t105 = g1t104*g1t77 + g1t80*g1t92;
  const double g1t106 = g1t54*g1t75;
  const double g1t107 = (Rational_4_3)*g1t106;
  const double g1t108 = g1t103*g1t83 + g1t73*g1t92;
  const double g1t109 = (Rational_4_3)*g1t75;
  const double g1t110 = g1t109*g1t28;
  const double g1t111 = f0_of_xx0*f1_of_xx1__D1*hDD02 + g1t102 + g1t37*hDD_dD021;
  const double g1t112 = g1t111*g1t92 + g1t77*hDD_dD001 + g1t83*g1t89;
  const double g1t113 = g1t109*g1t22;
  const double g1t114 = 2.0*vetU1;
  const double g1t115 = 2.0*vetU_dD11;
  const double g1t116 = g1t1*vetU_dD01;
  const double g1t117 = (g1t54*g1t54);
  const double g1t118 = g1t25*g1t5;
  const double g1t119 = g1t57*g1t86;
  const double g1t120 = g1t60*g1t86;
  const double g1t121 = g1t0*(g1t117*g1t118 + g1t119*g1t28 + g1t120*g1t54 + g1t18*g1t29 + g1t30*(g1t86*g1t86) + g1t52*g1t62);
  const double g1t122 = g1t0*(g1t118*g1t23 + g1t19 + g1t31 + g1t32*g1t52 + g1t36*g1t57 + g1t41*g1t60);
  const double g1t123 = g1t18*g1t23;
  const double g1t124 = (g1t50*g1t50);
  const double g1t125 = g1t117*g1t30;
  const double g1t126 = g1t50*g1t54;
  const double g1t127 = g1t0*(g1t118*g1t124 + g1t123 + g1t125 + g1t126*g1t60 + g1t52*g1t53 + g1t57*g1t61);
  const double g1t128 = (1.0 / g1t5);
  const double g1t129 = g1t128*vetU1;
  const double g1t130 = -g1t129;
  const double g1t131 = g1t1*vetU_dD10 + g1t130;
  const double g1t132 = f0_of_xx0*g1t131;
  const double g1t133 = g1t22*g1t75;
  const double g1t134 = 2.0*g1t133;
  const double g1t135 = g1t18*g1t28;
  const double g1t136 = g1t135*g1t22;
  const double g1t137 = g1t34*g1t54;
  const double g1t138 = g1t118*g1t54;
  const double g1t139 = g1t39*g1t86;
  const double g1t140 = g1t44*g1t86;
  const double g1t141 = g1t30*g1t86;
  const double g1t142 = g1t141*g1t54;
  const double g1t143 = 4.0*alpha;
  const double g1t144 = g1t143*(g1t117*g1t44 + g1t136 + g1t137*g1t22 + g1t138*g1t50 + g1t139*g1t22 + g1t140*g1t50 + g1t142 + g1t34*g1t58 + g1t39*g1t62);
  const double g1t145 = g1t12*g1t135;
  const double g1t146 = g1t141*g1t28;
  const double g1t147 = g1t143*(g1t12*g1t137 + g1t12*g1t139 + g1t138*g1t22 + g1t140*g1t22 + g1t145 + g1t146 + g1t29*g1t39 + g1t34*g1t41 + g1t44*g1t62);
  const double g1t148 = g1t143*(f0_of_xx0*g1t49 + g1t118*g1t53 + g1t34*g1t51 + g1t39*g1t41 + g1t39*g1t55 + g1t44*g1t58 + g1t44*g1t61 + g1t47 + g1t63);
  const double g1t149 = g1t128*vetU0;
  const double g1t150 = 4.0*g1t20*g1t7;
  const double g1t151 = (1.0 / g1t7);
  const double g1t152 = (Rational_1_2)*g1t151/g1t10;
  const double g1t153 = 2.0*g1t10;
  const double g1t154 = 8.0*g1t78;
  const double g1t155 = 4.0*g1t69;
  const double g1t156 = g1t128*vetU_dD11;
  const double g1t157 = g1t1*vetU_dDD101 - g1t156;
  const double g1t158 = -Rational_1_3*g1t129*g1t155 - Rational_8_3*g1t149 + (Rational_1_3)*g1t152*(g1t150*vetU_dD00 + 12.0*g1t8*vetU0) + (Rational_1_3)*g1t152*(g1t131*g1t153*g1t78 + g1t154*g1t5*vetU1) + (Rational_1_3)*g1t157 + (Rational_1_3)*vetU_dDD000;
  const double g1t159 = g1t1*vetU_dDD111;
  const double g1t160 = (f1_of_xx1__D1*f1_of_xx1__D1);
  const double g1t161 = f1_of_xx1*f1_of_xx1__DD11;
  const double g1t162 = g1t151*g1t160;
  const double g1t163 = g1t162*g1t2;
  const double g1t164 = -Rational_1_3*g1t1*g1t155*vetU0 + (Rational_1_3)*g1t152*(g1t150*vetU_dD01 + g1t154*g1t20*vetU0) + (Rational_1_3)*g1t152*(g1t115*g1t20*g1t78 + g1t2*(g1t153*g1t160 + g1t153*g1t161)) + (Rational_1_3)*g1t159 - Rational_2_3*g1t163 + (Rational_1_3)*vetU_dDD001;
  const double g1t165 = alpha*trK_dD0;
  const double g1t166 = alpha*trK_dD1;
  const double g1t167 = g1t1*g1t68;
  const double g1t168 = g1t128*g1t68;
  const double g1t169 = -g1t168*vetU2;
  const double g1t170 = g1t167*vetU_dD20 + g1t169;
  const double g1t171 = g1t28*g1t75;
  const double g1t172 = g1t1*vetU2;
  const double g1t173 = f1_of_xx1__D1*g1t151;
  const double g1t174 = -g1t172*g1t173;
  const double g1t175 = g1t167*vetU_dD21 + g1t174;
  const double g1t176 = (Rational_1_2)*g1t96;
  const double g1t177 = g1t176*g1t81 + g1t74*g1t83;
  const double g1t178 = g1t177 + g1t78;
  const double g1t179 = (Rational_1_2)*g1t106;
  const double g1t180 = g1t176*g1t93 + g1t179*g1t91 + g1t83*g1t90;
  const double g1t181 = g1t176*g1t99 + g1t179*g1t98 + g1t83*hDD_dD000;
  const double g1t182 = g1t103*g1t176 + g1t179*g1t73;
  const double g1t183 = g1t104*g1t83 + g1t179*g1t80;
  const double g1t184 = -g1t1;
  const double g1t185 = g1t111*g1t179 + g1t176*g1t89 + g1t83*hDD_dD001;
  const double g1t186 = g1t184 + g1t185;
  const double g1t187 = (1.0 / g1t20);
  const double g1t188 = g1t175*g1t78;
  const double g1t189 = g1t1*vetU_dD00 - g1t149;
  const double g1t190 = 2.0*g1t171;
  const double g1t191 = g1t179*g1t81 + g1t74*g1t92;
  const double g1t192 = (Rational_1_2)*g1t87;
  const double g1t193 = g1t179*g1t93 + g1t192*g1t91 + g1t90*g1t92;
  const double g1t194 = g1t179*g1t99 + g1t192*g1t98 + g1t92*hDD_dD000;
  const double g1t195 = g1t111*g1t192 + g1t179*g1t89 + g1t92*hDD_dD001;
  const double g1t196 = g1t104*g1t92 + g1t192*g1t80;
  const double g1t197 = g1t196 - g1t69;
  const double g1t198 = g1t103*g1t179 + g1t192*g1t73;
  const double g1t199 = g1t184 + g1t198;
  const double g1t200 = g1t1*g1t151;
  const double g1t201 = f1_of_xx1__D1*g1t200;
  const double g1t202 = (1.0 / (f1_of_xx1*f1_of_xx1*f1_of_xx1));
  const double g1t203 = g1t167*vetU2;
  const double g1t204 = f1_of_xx1__DD11*g1t68 - g1t162;
  const double g1t205 = g1t68*vetU2;
  const double g1t206 = 2.0*g1t205;
  const double g1t207 = (vetU0*vetU0);
  const double g1t208 = g1t128*(vetU1*vetU1);
  const double g1t209 = g1t128*g1t151*(vetU2*vetU2);
  const double g1t210 = 2.0*g1t2*vetU0;
  const double g1t211 = g1t205*g1t67;
  const double g1t212 = g1t129*g1t206;
  double a_alpha_dupD0 = lam[6 * Ntot + idx] * (vetU0);
  double a_alpha_dupD1 = lam[6 * Ntot + idx] * (g1t2);
  double a_g1t0 = lam[6 * Ntot + idx] * (-trK);
  double a_g1t2 = lam[6 * Ntot + idx] * (alpha_dupD1);
  double a_trK = lam[6 * Ntot + idx] * (-g1t0);
  double a_vetU0 = lam[6 * Ntot + idx] * (alpha_dupD0);
  double a_f0_of_xx0 = lam[17 * Ntot + idx] * (g1t96*vetU_dD00);
  double a_g1t100 = lam[17 * Ntot + idx] * (g1t101*g1t70 + g1t122);
  double a_g1t101 = lam[17 * Ntot + idx] * (g1t100*g1t70);
  double a_g1t105 = lam[17 * Ntot + idx] * (g1t107*g1t70 + g1t144);
  double a_g1t106 = lam[17 * Ntot + idx] * (-g1t175*g1t72);
  double a_g1t107 = lam[17 * Ntot + idx] * (g1t105*g1t70);
  double a_g1t108 = lam[17 * Ntot + idx] * (g1t110*g1t70 + g1t147);
  double a_g1t110 = lam[17 * Ntot + idx] * (g1t108*g1t70);
  double a_g1t112 = lam[17 * Ntot + idx] * (g1t113*g1t70 + g1t148);
  double a_g1t113 = lam[17 * Ntot + idx] * (g1t112*g1t70 - g1t166);
  double a_g1t114 = lam[17 * Ntot + idx] * (-g1t78*g1t87);
  double a_g1t115 = lam[17 * Ntot + idx] * (-g1t96);
  double a_g1t116 = lam[17 * Ntot + idx] * (-g1t134 - lambdaU1);
  double a_g1t121 = lam[17 * Ntot + idx] * (g1t85);
  double a_g1t122 = lam[17 * Ntot + idx] * (g1t100);
  double a_g1t127 = lam[17 * Ntot + idx] * (g1t95);
  double a_g1t132 = lam[17 * Ntot + idx] * (-g1t134);
  double a_g1t133 = lam[17 * Ntot + idx] * (g1t164);
  double a_g1t134 = lam[17 * Ntot + idx] * (-g1t116 - g1t132 + vetU_dDD001);
  double a_g1t144 = lam[17 * Ntot + idx] * (g1t105);
  double a_g1t147 = lam[17 * Ntot + idx] * (g1t108);
  double a_g1t148 = lam[17 * Ntot + idx] * (g1t112);
  double a_g1t158 = lam[17 * Ntot + idx] * (g1t76);
  double a_g1t164 = lam[17 * Ntot + idx] * (g1t133);
  double a_g1t165 = lam[17 * Ntot + idx] * (-Rational_4_3*g1t76);
  double a_g1t166 = lam[17 * Ntot + idx] * (-g1t113);
  double a_g1t170 = lam[17 * Ntot + idx] * (-g1t171*g1t72);
  double a_g1t171 = lam[17 * Ntot + idx] * (-g1t170*g1t72);
  double a_g1t175 = lam[17 * Ntot + idx] * (-g1t106*g1t72);
  double a_g1t19 = lam[17 * Ntot + idx] * (-2.0*g1t4);
  a_g1t2 += lam[17 * Ntot + idx] * (lambdaU_dupD01);
  double a_g1t23 = lam[17 * Ntot + idx] * (-g1t26*g1t4);
  double a_g1t26 = lam[17 * Ntot + idx] * (-g1t23*g1t4);
  double a_g1t31 = lam[17 * Ntot + idx] * (-2.0*g1t4);
  double a_g1t32 = lam[17 * Ntot + idx] * (-g1t35*g1t4);
  double a_g1t35 = lam[17 * Ntot + idx] * (-g1t32*g1t4);
  double a_g1t36 = lam[17 * Ntot + idx] * (-g1t4*g1t40);
  double a_g1t4 = lam[17 * Ntot + idx] * (-2.0*g1t19 - g1t23*g1t26 - 2.0*g1t31 - g1t32*g1t35 - g1t36*g1t40 - g1t41*g1t45);
  double a_g1t40 = lam[17 * Ntot + idx] * (-g1t36*g1t4);
  double a_g1t41 = lam[17 * Ntot + idx] * (-g1t4*g1t45);
  double a_g1t45 = lam[17 * Ntot + idx] * (-g1t4*g1t41);
  double a_g1t46 = lam[17 * Ntot + idx] * (g1t64);
  double a_g1t64 = lam[17 * Ntot + idx] * (g1t46);
  double a_g1t7 = lam[17 * Ntot + idx] * (-g1t87*vetU0);
  double a_g1t70 = lam[17 * Ntot + idx] * (g1t100*g1t101 + g1t105*g1t107 + g1t108*g1t110 + g1t112*g1t113 + g1t85*g1t88 + g1t95*g1t97);
  double a_g1t71 = lam[17 * Ntot + idx] * (g1t87*vetU_dD00);
  double a_g1t72 = lam[17 * Ntot + idx] * (-g1t106*g1t175 - g1t170*g1t171);
  double a_g1t76 = lam[17 * Ntot + idx] * (g1t158 - Rational_4_3*g1t165 + vetU_dDD000);
  double a_g1t78 = lam[17 * Ntot + idx] * (g1t87*(-g1t114 + vetU_dD01));
  double a_g1t85 = lam[17 * Ntot + idx] * (g1t121 + g1t70*g1t88);
  double a_g1t87 = lam[17 * Ntot + idx] * (-g1t114*g1t78 - g1t7*vetU0 + g1t71*vetU_dD00 + g1t78*vetU_dD01);
  double a_g1t88 = lam[17 * Ntot + idx] * (g1t70*g1t85);
  double a_g1t95 = lam[17 * Ntot + idx] * (g1t127 + g1t70*g1t97);
  double a_g1t96 = lam[17 * Ntot + idx] * (f0_of_xx0*vetU_dD00 - g1t115 - vetU0 + vetU_dDD011);
  double a_g1t97 = lam[17 * Ntot + idx] * (g1t70*g1t95);
  double a_lambdaU0 = lam[17 * Ntot + idx] * (-vetU_dD00);
  double a_lambdaU1 = lam[17 * Ntot + idx] * (-g1t116);
  double a_lambdaU_dupD00 = lam[17 * Ntot + idx] * (vetU0);
  double a_lambdaU_dupD01 = lam[17 * Ntot + idx] * (g1t2);
  a_vetU0 += lam[17 * Ntot + idx] * (-g1t7*g1t87 - g1t96 + lambdaU_dupD00);
  double a_vetU_dD00 = lam[17 * Ntot + idx] * (f0_of_xx0*g1t96 + g1t71*g1t87 - lambdaU0);
  double a_vetU_dD01 = lam[17 * Ntot + idx] * (g1t78*g1t87);
  double a_vetU_dDD000 = lam[17 * Ntot + idx] * (g1t76);
  double a_vetU_dDD001 = lam[17 * Ntot + idx] * (g1t134);
  double a_vetU_dDD011 = lam[17 * Ntot + idx] * (g1t96);
  a_f0_of_xx0 += lam[18 * Ntot + idx] * (-g1t106*g1t188 + g1t106*(-f1_of_xx1*g1t172 + g1t1*g1t160*g1t68*vetU2 + g1t1*g1t68*vetU2*(-g1t160 - g1t161) - g1t188) - g1t113*g1t165 + g1t121*g1t178 + g1t122*g1t181 + g1t127*g1t180 + g1t129*lambdaU_dupD11 - g1t131*lambdaU0 + g1t133*g1t158 + g1t134*(g1t157 + g1t189) + g1t144*g1t183 + g1t147*g1t182 + g1t148*g1t186 - g1t156*lambdaU1 + g1t164*g1t96 - Rational_4_3*g1t166*g1t96 - g1t170*g1t190*g1t78 + g1t4*g1t64 + g1t46*(-2.0*g1t123 - g1t124*g1t26 - 2.0*g1t125 - g1t126*g1t45 - g1t35*g1t53 - g1t40*g1t61) + g1t70*(g1t101*g1t181 + g1t107*g1t183 + g1t110*g1t182 + g1t113*g1t186 + g1t178*g1t88 + g1t180*g1t97) + g1t76*(g1t1*vetU_dDD100 + g1t114*g1t187 - 2.0*g1t128*vetU_dD10 + g1t131*g1t66) + g1t87*(g1t131*g1t71 - g1t160*g1t2 + g1t2*g1t7 + g1t65*g1t78) + g1t96*(2.0*g1t116 + g1t132 + g1t159) + vetU0*(g1t1*lambdaU_dupD10 - g1t128*lambdaU1));
  double a_f1_of_xx1 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t106*g1t172);
  double a_g1t1 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t106*(g1t160*g1t68*vetU2 + g1t68*vetU2*(-g1t160 - g1t161)) + g1t76*vetU_dDD100 + lambdaU_dupD10*vetU0));
  a_g1t101 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t181*g1t70);
  a_g1t106 += lam[18 * Ntot + idx] * (f0_of_xx0*(-f1_of_xx1*g1t172 + g1t1*g1t160*g1t68*vetU2 + g1t1*g1t68*vetU2*(-g1t160 - g1t161) - 2.0*g1t188));
  a_g1t107 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t183*g1t70);
  a_g1t110 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t182*g1t70);
  a_g1t113 += lam[18 * Ntot + idx] * (f0_of_xx0*(-g1t165 + g1t186*g1t70));
  a_g1t114 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t187*g1t76);
  a_g1t116 += lam[18 * Ntot + idx] * (2.0*f0_of_xx0*g1t96);
  a_g1t121 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t178);
  a_g1t122 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t181);
  double a_g1t123 = lam[18 * Ntot + idx] * (-2.0*f0_of_xx0*g1t46);
  double a_g1t124 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t26*g1t46);
  double a_g1t125 = lam[18 * Ntot + idx] * (-2.0*f0_of_xx0*g1t46);
  double a_g1t126 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t45*g1t46);
  a_g1t127 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t180);
  double a_g1t128 = lam[18 * Ntot + idx] * (f0_of_xx0*(-2.0*g1t76*vetU_dD10 - lambdaU1*vetU0));
  double a_g1t129 = lam[18 * Ntot + idx] * (f0_of_xx0*lambdaU_dupD11);
  double a_g1t131 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t66*g1t76 + g1t71*g1t87 - lambdaU0));
  a_g1t132 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t96);
  a_g1t133 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t158);
  a_g1t134 += lam[18 * Ntot + idx] * (f0_of_xx0*(g1t157 + g1t189));
  a_g1t144 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t183);
  a_g1t147 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t182);
  a_g1t148 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t186);
  double a_g1t156 = lam[18 * Ntot + idx] * (-f0_of_xx0*lambdaU1);
  double a_g1t157 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t134);
  a_g1t158 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t133);
  double a_g1t159 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t96);
  double a_g1t160 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t2*g1t87);
  double a_g1t161 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t1*g1t106*g1t68*vetU2);
  a_g1t164 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t96);
  a_g1t165 += lam[18 * Ntot + idx] * (-f0_of_xx0*g1t113);
  a_g1t166 += lam[18 * Ntot + idx] * (-Rational_4_3*f0_of_xx0*g1t96);
  a_g1t170 += lam[18 * Ntot + idx] * (-f0_of_xx0*g1t190*g1t78);
  double a_g1t172 = lam[18 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1*g1t106);
  double a_g1t178 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t121 + g1t70*g1t88));
  double a_g1t180 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t127 + g1t70*g1t97));
  double a_g1t181 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t101*g1t70 + g1t122));
  double a_g1t182 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t110*g1t70 + g1t147));
  double a_g1t183 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t107*g1t70 + g1t144));
  double a_g1t186 = lam[18 * Ntot + idx] * (f0_of_xx0*(g1t113*g1t70 + g1t148));
  double a_g1t187 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t114*g1t76);
  double a_g1t188 = lam[18 * Ntot + idx] * (-2.0*f0_of_xx0*g1t106);
  double a_g1t189 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t134);
  double a_g1t190 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t170*g1t78);
  a_g1t2 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t87*(-g1t160 + g1t7));
  a_g1t26 += lam[18 * Ntot + idx] * (-f0_of_xx0*g1t124*g1t46);
  a_g1t35 += lam[18 * Ntot + idx] * (-f0_of_xx0*g1t46*g1t53);
  a_g1t4 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t64);
  a_g1t40 += lam[18 * Ntot + idx] * (-f0_of_xx0*g1t46*g1t61);
  a_g1t45 += lam[18 * Ntot + idx] * (-f0_of_xx0*g1t126*g1t46);
  a_g1t46 += lam[18 * Ntot + idx] * (f0_of_xx0*(-2.0*g1t123 - g1t124*g1t26 - 2.0*g1t125 - g1t126*g1t45 - g1t35*g1t53 - g1t40*g1t61));
  double a_g1t53 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t35*g1t46);
  double a_g1t61 = lam[18 * Ntot + idx] * (-f0_of_xx0*g1t40*g1t46);
  a_g1t64 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t4);
  double a_g1t65 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t78*g1t87);
  double a_g1t66 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t131*g1t76);
  double a_g1t68 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t106*(g1t1*g1t160*vetU2 + g1t1*vetU2*(-g1t160 - g1t161)));
  a_g1t7 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t2*g1t87);
  a_g1t70 += lam[18 * Ntot + idx] * (f0_of_xx0*(g1t101*g1t181 + g1t107*g1t183 + g1t110*g1t182 + g1t113*g1t186 + g1t178*g1t88 + g1t180*g1t97));
  a_g1t71 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t131*g1t87);
  a_g1t76 += lam[18 * Ntot + idx] * (f0_of_xx0*(g1t1*vetU_dDD100 + g1t114*g1t187 - 2.0*g1t128*vetU_dD10 + g1t131*g1t66));
  a_g1t78 += lam[18 * Ntot + idx] * (f0_of_xx0*(-g1t170*g1t190 + g1t65*g1t87));
  a_g1t87 += lam[18 * Ntot + idx] * (f0_of_xx0*(g1t131*g1t71 - g1t160*g1t2 + g1t2*g1t7 + g1t65*g1t78));
  a_g1t88 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t178*g1t70);
  a_g1t96 += lam[18 * Ntot + idx] * (f0_of_xx0*(2.0*g1t116 + g1t132 + g1t159 + g1t164 - Rational_4_3*g1t166));
  a_g1t97 += lam[18 * Ntot + idx] * (f0_of_xx0*g1t180*g1t70);
  a_lambdaU0 += lam[18 * Ntot + idx] * (-f0_of_xx0*g1t131);
  a_lambdaU1 += lam[18 * Ntot + idx] * (f0_of_xx0*(-g1t128*vetU0 - g1t156));
  double a_lambdaU_dupD10 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t1*vetU0);
  double a_lambdaU_dupD11 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t129);
  a_vetU0 += lam[18 * Ntot + idx] * (f0_of_xx0*(g1t1*lambdaU_dupD10 - g1t128*lambdaU1));
  double a_vetU2 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t106*(g1t1*g1t160*g1t68 + g1t1*g1t68*(-g1t160 - g1t161)));
  double a_vetU_dD10 = lam[18 * Ntot + idx] * (-2.0*f0_of_xx0*g1t128*g1t76);
  double a_vetU_dDD100 = lam[18 * Ntot + idx] * (f0_of_xx0*g1t1*g1t76);
  a_f0_of_xx0 += lam[19 * Ntot + idx] * (g1t170*g1t37*g1t96);
  double a_f1_of_xx1__D1 = lam[19 * Ntot + idx] * (g1t1*g1t106*g1t37*g1t68*vetU_dD11);
  double a_f1_of_xx1__DD11 = lam[19 * Ntot + idx] * (-g1t200*g1t37*g1t96*vetU2);
  a_g1t1 += lam[19 * Ntot + idx] * (g1t37*(f1_of_xx1__D1*g1t106*g1t68*vetU_dD11 + 2.0*g1t160*g1t202*g1t96*vetU2 - g1t175*lambdaU1));
  a_g1t101 += lam[19 * Ntot + idx] * (g1t194*g1t37*g1t70);
  a_g1t106 += lam[19 * Ntot + idx] * (g1t37*(f1_of_xx1__D1*g1t1*g1t68*vetU_dD11 + 2.0*g1t116 - g1t163 + g1t164 + g1t2*g1t204 - g1t2 + g1t65*g1t69));
  a_g1t107 += lam[19 * Ntot + idx] * (g1t37*(-g1t166 + g1t197*g1t70));
  a_g1t110 += lam[19 * Ntot + idx] * (g1t37*(-g1t165 + g1t199*g1t70));
  a_g1t113 += lam[19 * Ntot + idx] * (g1t195*g1t37*g1t70);
  a_g1t116 += lam[19 * Ntot + idx] * (2.0*g1t106*g1t37);
  double a_g1t117 = lam[19 * Ntot + idx] * (-g1t37*g1t46*g1t60);
  double a_g1t119 = lam[19 * Ntot + idx] * (g1t37*(-g1t12*g1t4 - g1t22*g1t46));
  double a_g1t12 = lam[19 * Ntot + idx] * (-g1t119*g1t37*g1t4);
  double a_g1t120 = lam[19 * Ntot + idx] * (g1t37*(-g1t22*g1t4 - g1t46*g1t50));
  a_g1t121 += lam[19 * Ntot + idx] * (g1t191*g1t37);
  a_g1t122 += lam[19 * Ntot + idx] * (g1t194*g1t37);
  a_g1t126 += lam[19 * Ntot + idx] * (-g1t26*g1t37*g1t46);
  a_g1t127 += lam[19 * Ntot + idx] * (g1t193*g1t37);
  a_g1t128 += lam[19 * Ntot + idx] * (g1t134*g1t173*g1t37*vetU2);
  a_g1t131 += lam[19 * Ntot + idx] * (g1t190*g1t37*g1t69);
  a_g1t134 += lam[19 * Ntot + idx] * (g1t37*(g1t128*g1t173*vetU2 + g1t167*vetU_dDD201 - g1t168*vetU_dD21 + g1t170*g1t69 - g1t201*vetU_dD20));
  double a_g1t136 = lam[19 * Ntot + idx] * (-2.0*g1t37*g1t46);
  double a_g1t142 = lam[19 * Ntot + idx] * (-2.0*g1t37*g1t46);
  a_g1t144 += lam[19 * Ntot + idx] * (g1t197*g1t37);
  double a_g1t145 = lam[19 * Ntot + idx] * (-2.0*g1t37*g1t4);
  double a_g1t146 = lam[19 * Ntot + idx] * (-2.0*g1t37*g1t4);
  a_g1t147 += lam[19 * Ntot + idx] * (g1t199*g1t37);
  a_g1t148 += lam[19 * Ntot + idx] * (g1t195*g1t37);
  a_g1t158 += lam[19 * Ntot + idx] * (g1t171*g1t37);
  a_g1t160 += lam[19 * Ntot + idx] * (g1t37*g1t96*(2.0*g1t1*g1t202*vetU2 + g1t172*g1t202));
  double a_g1t163 = lam[19 * Ntot + idx] * (-g1t106*g1t37);
  a_g1t164 += lam[19 * Ntot + idx] * (g1t106*g1t37);
  a_g1t165 += lam[19 * Ntot + idx] * (-g1t110*g1t37);
  a_g1t166 += lam[19 * Ntot + idx] * (-g1t107*g1t37);
  double a_g1t167 = lam[19 * Ntot + idx] * (g1t37*(g1t134*vetU_dDD201 + g1t2*lambdaU_dupD21 + g1t76*vetU_dDD200 + g1t96*vetU_dDD211 + lambdaU_dupD20*vetU0));
  double a_g1t168 = lam[19 * Ntot + idx] * (g1t37*(-g1t134*vetU_dD21 - 2.0*g1t76*vetU_dD20 - lambdaU2*vetU0));
  a_g1t170 += lam[19 * Ntot + idx] * (g1t37*(f0_of_xx0*g1t96 + g1t134*g1t69 + g1t66*g1t76 + g1t71*g1t87 - lambdaU0));
  a_g1t171 += lam[19 * Ntot + idx] * (g1t158*g1t37);
  a_g1t172 += lam[19 * Ntot + idx] * (g1t160*g1t202*g1t37*g1t96);
  double a_g1t173 = lam[19 * Ntot + idx] * (g1t37*(g1t128*g1t134*vetU2 - g1t66*g1t96*vetU_dD21));
  a_g1t175 += lam[19 * Ntot + idx] * (g1t37*(-g1t1*lambdaU1 + 2.0*g1t69*g1t96));
  a_g1t187 += lam[19 * Ntot + idx] * (g1t206*g1t37*g1t76);
  a_g1t188 += lam[19 * Ntot + idx] * (g1t37*g1t87);
  a_g1t189 += lam[19 * Ntot + idx] * (g1t190*g1t37);
  a_g1t190 += lam[19 * Ntot + idx] * (g1t37*(g1t131*g1t69 + g1t189));
  double a_g1t191 = lam[19 * Ntot + idx] * (g1t37*(g1t121 + g1t70*g1t88));
  double a_g1t193 = lam[19 * Ntot + idx] * (g1t37*(g1t127 + g1t70*g1t97));
  double a_g1t194 = lam[19 * Ntot + idx] * (g1t37*(g1t101*g1t70 + g1t122));
  double a_g1t195 = lam[19 * Ntot + idx] * (g1t37*(g1t113*g1t70 + g1t148));
  double a_g1t197 = lam[19 * Ntot + idx] * (g1t37*(g1t107*g1t70 + g1t144));
  double a_g1t199 = lam[19 * Ntot + idx] * (g1t37*(g1t110*g1t70 + g1t147));
  a_g1t2 += lam[19 * Ntot + idx] * (g1t37*(g1t106*g1t204 - g1t106 + g1t167*lambdaU_dupD21 - g1t201*lambdaU2));
  double a_g1t200 = lam[19 * Ntot + idx] * (-f1_of_xx1__DD11*g1t37*g1t96*vetU2);
  double a_g1t201 = lam[19 * Ntot + idx] * (g1t37*(-g1t134*vetU_dD20 - g1t2*lambdaU2));
  double a_g1t202 = lam[19 * Ntot + idx] * (g1t37*g1t96*(2.0*g1t1*g1t160*vetU2 + g1t160*g1t172));
  double a_g1t203 = lam[19 * Ntot + idx] * (g1t37*g1t96*(g1t204 + 1.0));
  double a_g1t204 = lam[19 * Ntot + idx] * (g1t37*(g1t106*g1t2 + g1t203*g1t96));
  double a_g1t206 = lam[19 * Ntot + idx] * (g1t187*g1t37*g1t76);
  double a_g1t22 = lam[19 * Ntot + idx] * (g1t37*(-g1t119*g1t46 - g1t120*g1t4));
  a_g1t26 += lam[19 * Ntot + idx] * (g1t37*(-g1t126*g1t46 - g1t4*g1t61));
  double a_g1t29 = lam[19 * Ntot + idx] * (-g1t37*g1t4*g1t57);
  double a_g1t37 = lam[19 * Ntot + idx] * (-g1t1*g1t175*lambdaU1 + g1t106*g1t164 + g1t106*(g1t116 + g1t2*g1t204 + g1t65*g1t69) + g1t106*(f1_of_xx1__D1*g1t1*g1t68*vetU_dD11 + g1t116 - g1t163 - g1t2) - g1t107*g1t166 - g1t110*g1t165 + g1t121*g1t191 + g1t122*g1t194 + g1t127*g1t193 + g1t134*(g1t128*g1t173*vetU2 + g1t167*vetU_dDD201 - g1t168*vetU_dD21 + g1t170*g1t69 - g1t201*vetU_dD20) + g1t144*g1t197 + g1t147*g1t199 + g1t148*g1t195 + g1t158*g1t171 - g1t170*lambdaU0 + g1t190*(g1t131*g1t69 + g1t189) + g1t2*(g1t167*lambdaU_dupD21 - g1t201*lambdaU2) + g1t4*(-g1t119*g1t12 - g1t120*g1t22 - 2.0*g1t145 - 2.0*g1t146 - g1t26*g1t61 - g1t29*g1t57 - g1t41*g1t52 - g1t52*g1t55 - g1t60*g1t62) + g1t46*(-g1t117*g1t60 - g1t119*g1t22 - g1t120*g1t50 - g1t126*g1t26 - 2.0*g1t136 - 2.0*g1t142 - g1t52*g1t58 - g1t52*g1t61 - g1t57*g1t62) + g1t70*(g1t101*g1t194 + g1t107*g1t197 + g1t110*g1t199 + g1t113*g1t195 + g1t191*g1t88 + g1t193*g1t97) + g1t76*(g1t167*vetU_dDD200 - 2.0*g1t168*vetU_dD20 + g1t170*g1t66 + g1t187*g1t206) + g1t87*(g1t170*g1t71 + g1t188) + g1t96*(f0_of_xx0*g1t170 + g1t160*g1t172*g1t202 + g1t167*vetU_dDD211 - g1t173*g1t66*vetU_dD21 + 2.0*g1t175*g1t69 + g1t203*g1t204 + g1t203 + vetU2*(-f1_of_xx1__DD11*g1t200 + 2.0*g1t1*g1t160*g1t202)) + vetU0*(g1t167*lambdaU_dupD20 - g1t168*lambdaU2));
  a_g1t4 += lam[19 * Ntot + idx] * (g1t37*(-g1t119*g1t12 - g1t120*g1t22 - 2.0*g1t145 - 2.0*g1t146 - g1t26*g1t61 - g1t29*g1t57 - g1t41*g1t52 - g1t52*g1t55 - g1t60*g1t62));
  a_g1t41 += lam[19 * Ntot + idx] * (-g1t37*g1t4*g1t52);
  a_g1t46 += lam[19 * Ntot + idx] * (g1t37*(-g1t117*g1t60 - g1t119*g1t22 - g1t120*g1t50 - g1t126*g1t26 - 2.0*g1t136 - 2.0*g1t142 - g1t52*g1t58 - g1t52*g1t61 - g1t57*g1t62));
  double a_g1t50 = lam[19 * Ntot + idx] * (-g1t120*g1t37*g1t46);
  double a_g1t52 = lam[19 * Ntot + idx] * (g1t37*(g1t4*(-g1t41 - g1t55) + g1t46*(-g1t58 - g1t61)));
  double a_g1t55 = lam[19 * Ntot + idx] * (-g1t37*g1t4*g1t52);
  double a_g1t57 = lam[19 * Ntot + idx] * (g1t37*(-g1t29*g1t4 - g1t46*g1t62));
  double a_g1t58 = lam[19 * Ntot + idx] * (-g1t37*g1t46*g1t52);
  double a_g1t60 = lam[19 * Ntot + idx] * (g1t37*(-g1t117*g1t46 - g1t4*g1t62));
  a_g1t61 += lam[19 * Ntot + idx] * (g1t37*(-g1t26*g1t4 - g1t46*g1t52));
  double a_g1t62 = lam[19 * Ntot + idx] * (g1t37*(-g1t4*g1t60 - g1t46*g1t57));
  a_g1t65 += lam[19 * Ntot + idx] * (g1t106*g1t37*g1t69);
  a_g1t66 += lam[19 * Ntot + idx] * (g1t37*(g1t170*g1t76 - g1t173*g1t96*vetU_dD21));
  a_g1t68 += lam[19 * Ntot + idx] * (f1_of_xx1__D1*g1t1*g1t106*g1t37*vetU_dD11);
  double a_g1t69 = lam[19 * Ntot + idx] * (g1t37*(g1t106*g1t65 + g1t131*g1t190 + g1t134*g1t170 + 2.0*g1t175*g1t96));
  a_g1t70 += lam[19 * Ntot + idx] * (g1t37*(g1t101*g1t194 + g1t107*g1t197 + g1t110*g1t199 + g1t113*g1t195 + g1t191*g1t88 + g1t193*g1t97));
  a_g1t71 += lam[19 * Ntot + idx] * (g1t170*g1t37*g1t87);
  a_g1t76 += lam[19 * Ntot + idx] * (g1t37*(g1t167*vetU_dDD200 - 2.0*g1t168*vetU_dD20 + g1t170*g1t66 + g1t187*g1t206));
  a_g1t87 += lam[19 * Ntot + idx] * (g1t37*(g1t170*g1t71 + g1t188));
  a_g1t88 += lam[19 * Ntot + idx] * (g1t191*g1t37*g1t70);
  a_g1t96 += lam[19 * Ntot + idx] * (g1t37*(f0_of_xx0*g1t170 + g1t160*g1t172*g1t202 + g1t167*vetU_dDD211 - g1t173*g1t66*vetU_dD21 + 2.0*g1t175*g1t69 + g1t203*g1t204 + g1t203 + vetU2*(-f1_of_xx1__DD11*g1t200 + 2.0*g1t1*g1t160*g1t202)));
  a_g1t97 += lam[19 * Ntot + idx] * (g1t193*g1t37*g1t70);
  a_lambdaU0 += lam[19 * Ntot + idx] * (-g1t170*g1t37);
  a_lambdaU1 += lam[19 * Ntot + idx] * (-g1t1*g1t175*g1t37);
  double a_lambdaU2 = lam[19 * Ntot + idx] * (g1t37*(-g1t168*vetU0 - g1t2*g1t201));
  double a_lambdaU_dupD20 = lam[19 * Ntot + idx] * (g1t167*g1t37*vetU0);
  double a_lambdaU_dupD21 = lam[19 * Ntot + idx] * (g1t167*g1t2*g1t37);
  a_vetU0 += lam[19 * Ntot + idx] * (g1t37*(g1t167*lambdaU_dupD20 - g1t168*lambdaU2));
  a_vetU2 += lam[19 * Ntot + idx] * (g1t37*(g1t128*g1t134*g1t173 + g1t96*(-f1_of_xx1__DD11*g1t200 + 2.0*g1t1*g1t160*g1t202)));
  double a_vetU_dD11 = lam[19 * Ntot + idx] * (f1_of_xx1__D1*g1t1*g1t106*g1t37*g1t68);
  double a_vetU_dD20 = lam[19 * Ntot + idx] * (g1t37*(-g1t134*g1t201 - 2.0*g1t168*g1t76));
  double a_vetU_dD21 = lam[19 * Ntot + idx] * (g1t37*(-g1t134*g1t168 - g1t173*g1t66*g1t96));
  double a_vetU_dDD200 = lam[19 * Ntot + idx] * (g1t167*g1t37*g1t76);
  double a_vetU_dDD201 = lam[19 * Ntot + idx] * (g1t134*g1t167*g1t37);
  double a_vetU_dDD211 = lam[19 * Ntot + idx] * (g1t167*g1t37*g1t96);
  double a_betU0 = lam[21 * Ntot + idx] * (1.0);
  a_g1t100 += lam[21 * Ntot + idx] * (g1t207);
  a_g1t105 += lam[21 * Ntot + idx] * (g1t212);
  a_g1t108 += lam[21 * Ntot + idx] * (g1t211);
  a_g1t112 += lam[21 * Ntot + idx] * (g1t210);
  a_g1t2 += lam[21 * Ntot + idx] * (vetU_dupD01);
  double a_g1t207 = lam[21 * Ntot + idx] * (g1t100);
  double a_g1t208 = lam[21 * Ntot + idx] * (g1t94);
  double a_g1t209 = lam[21 * Ntot + idx] * (g1t84);
  double a_g1t210 = lam[21 * Ntot + idx] * (g1t112);
  double a_g1t211 = lam[21 * Ntot + idx] * (g1t108);
  double a_g1t212 = lam[21 * Ntot + idx] * (g1t105);
  double a_g1t84 = lam[21 * Ntot + idx] * (g1t209);
  double a_g1t94 = lam[21 * Ntot + idx] * (g1t208);
  a_vetU0 += lam[21 * Ntot + idx] * (vetU_dupD00);
  double a_vetU_dupD00 = lam[21 * Ntot + idx] * (vetU0);
  double a_vetU_dupD01 = lam[21 * Ntot + idx] * (g1t2);
  double a_betU1 = lam[22 * Ntot + idx] * (f0_of_xx0*g1t1);
  a_f0_of_xx0 += lam[22 * Ntot + idx] * (betU1*g1t1 + g1t129*vetU_dupD11 + g1t177*g1t209 + g1t180*g1t208 + g1t181*g1t207 + g1t182*g1t211 + g1t183*g1t212 + g1t185*g1t210 + vetU0*(g1t1*vetU_dupD10 + g1t130));
  a_g1t1 += lam[22 * Ntot + idx] * (f0_of_xx0*(betU1 + vetU0*vetU_dupD10));
  a_g1t129 += lam[22 * Ntot + idx] * (f0_of_xx0*vetU_dupD11);
  double a_g1t130 = lam[22 * Ntot + idx] * (f0_of_xx0*vetU0);
  double a_g1t177 = lam[22 * Ntot + idx] * (f0_of_xx0*g1t209);
  a_g1t180 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t208);
  a_g1t181 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t207);
  a_g1t182 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t211);
  a_g1t183 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t212);
  double a_g1t185 = lam[22 * Ntot + idx] * (f0_of_xx0*g1t210);
  a_g1t207 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t181);
  a_g1t208 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t180);
  a_g1t209 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t177);
  a_g1t210 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t185);
  a_g1t211 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t182);
  a_g1t212 += lam[22 * Ntot + idx] * (f0_of_xx0*g1t183);
  a_vetU0 += lam[22 * Ntot + idx] * (f0_of_xx0*(g1t1*vetU_dupD10 + g1t130));
  double a_vetU_dupD10 = lam[22 * Ntot + idx] * (f0_of_xx0*g1t1*vetU0);
  double a_vetU_dupD11 = lam[22 * Ntot + idx] * (f0_of_xx0*g1t129);
  double a_betU2 = lam[23 * Ntot + idx] * (g1t167*g1t37);
  a_g1t167 += lam[23 * Ntot + idx] * (g1t37*(betU2 + g1t2*vetU_dupD21 + vetU0*vetU_dupD20));
  double a_g1t169 = lam[23 * Ntot + idx] * (g1t37*vetU0);
  double a_g1t174 = lam[23 * Ntot + idx] * (g1t2*g1t37);
  a_g1t191 += lam[23 * Ntot + idx] * (g1t209*g1t37);
  a_g1t193 += lam[23 * Ntot + idx] * (g1t208*g1t37);
  a_g1t194 += lam[23 * Ntot + idx] * (g1t207*g1t37);
  a_g1t195 += lam[23 * Ntot + idx] * (g1t210*g1t37);
  double a_g1t196 = lam[23 * Ntot + idx] * (g1t212*g1t37);
  double a_g1t198 = lam[23 * Ntot + idx] * (g1t211*g1t37);
  a_g1t2 += lam[23 * Ntot + idx] * (g1t37*(g1t167*vetU_dupD21 + g1t174));
  a_g1t207 += lam[23 * Ntot + idx] * (g1t194*g1t37);
  a_g1t208 += lam[23 * Ntot + idx] * (g1t193*g1t37);
  a_g1t209 += lam[23 * Ntot + idx] * (g1t191*g1t37);
  a_g1t210 += lam[23 * Ntot + idx] * (g1t195*g1t37);
  a_g1t211 += lam[23 * Ntot + idx] * (g1t198*g1t37);
  a_g1t212 += lam[23 * Ntot + idx] * (g1t196*g1t37);
  a_g1t37 += lam[23 * Ntot + idx] * (betU2*g1t167 + g1t191*g1t209 + g1t193*g1t208 + g1t194*g1t207 + g1t195*g1t210 + g1t196*g1t212 + g1t198*g1t211 + g1t2*(g1t167*vetU_dupD21 + g1t174) + vetU0*(g1t167*vetU_dupD20 + g1t169));
  a_vetU0 += lam[23 * Ntot + idx] * (g1t37*(g1t167*vetU_dupD20 + g1t169));
  double a_vetU_dupD20 = lam[23 * Ntot + idx] * (g1t167*g1t37*vetU0);
  double a_vetU_dupD21 = lam[23 * Ntot + idx] * (g1t167*g1t2*g1t37);
  a_g1t129 += a_g1t212 * (g1t206);
  a_g1t206 += a_g1t212 * (g1t129);
  double a_g1t205 = a_g1t211 * (g1t67);
  double a_g1t67 = a_g1t211 * (g1t205);
  a_g1t2 += a_g1t210 * (2.0*vetU0);
  a_vetU0 += a_g1t210 * (2.0*g1t2);
  a_g1t128 += a_g1t209 * (g1t151*(vetU2*vetU2));
  double a_g1t151 = a_g1t209 * (g1t128*(vetU2*vetU2));
  a_vetU2 += a_g1t209 * (2.0*g1t128*g1t151*vetU2);
  a_g1t128 += a_g1t208 * ((vetU1*vetU1));
  double a_vetU1 = a_g1t208 * (2.0*g1t128*vetU1);
  a_vetU0 += a_g1t207 * (2.0*vetU0);
  a_g1t205 += a_g1t206 * (2.0);
  a_g1t68 += a_g1t205 * (vetU2);
  a_vetU2 += a_g1t205 * (g1t68);
  a_f1_of_xx1__DD11 += a_g1t204 * (g1t68);
  double a_g1t162 = a_g1t204 * (-1.0);
  a_g1t68 += a_g1t204 * (f1_of_xx1__DD11);
  a_g1t167 += a_g1t203 * (vetU2);
  a_vetU2 += a_g1t203 * (g1t167);
  a_f1_of_xx1 += a_g1t202 * (-3.0/(f1_of_xx1*f1_of_xx1*f1_of_xx1*f1_of_xx1));
  a_f1_of_xx1__D1 += a_g1t201 * (g1t200);
  a_g1t200 += a_g1t201 * (f1_of_xx1__D1);
  a_g1t1 += a_g1t200 * (g1t151);
  a_g1t151 += a_g1t200 * (g1t1);
  double a_g1t184 = a_g1t199 * (1.0);
  a_g1t198 += a_g1t199 * (1.0);
  double a_g1t103 = a_g1t198 * (g1t179);
  double a_g1t179 = a_g1t198 * (g1t103);
  double a_g1t192 = a_g1t198 * (g1t73);
  double a_g1t73 = a_g1t198 * (g1t192);
  a_g1t196 += a_g1t197 * (1.0);
  a_g1t69 += a_g1t197 * (-1.0);
  double a_g1t104 = a_g1t196 * (g1t92);
  a_g1t192 += a_g1t196 * (g1t80);
  double a_g1t80 = a_g1t196 * (g1t192);
  double a_g1t92 = a_g1t196 * (g1t104);
  double a_g1t111 = a_g1t195 * (g1t192);
  a_g1t179 += a_g1t195 * (g1t89);
  a_g1t192 += a_g1t195 * (g1t111);
  double a_g1t89 = a_g1t195 * (g1t179);
  a_g1t92 += a_g1t195 * (hDD_dD001);
  double a_hDD_dD001 = a_g1t195 * (g1t92);
  a_g1t179 += a_g1t194 * (g1t99);
  a_g1t192 += a_g1t194 * (g1t98);
  a_g1t92 += a_g1t194 * (hDD_dD000);
  double a_g1t98 = a_g1t194 * (g1t192);
  double a_g1t99 = a_g1t194 * (g1t179);
  double a_hDD_dD000 = a_g1t194 * (g1t92);
  a_g1t179 += a_g1t193 * (g1t93);
  a_g1t192 += a_g1t193 * (g1t91);
  double a_g1t90 = a_g1t193 * (g1t92);
  double a_g1t91 = a_g1t193 * (g1t192);
  a_g1t92 += a_g1t193 * (g1t90);
  double a_g1t93 = a_g1t193 * (g1t179);
  a_g1t87 += a_g1t192 * (Rational_1_2);
  a_g1t179 += a_g1t191 * (g1t81);
  double a_g1t74 = a_g1t191 * (g1t92);
  double a_g1t81 = a_g1t191 * (g1t179);
  a_g1t92 += a_g1t191 * (g1t74);
  a_g1t171 += a_g1t190 * (2.0);
  a_g1t1 += a_g1t189 * (vetU_dD00);
  double a_g1t149 = a_g1t189 * (-1.0);
  a_vetU_dD00 += a_g1t189 * (g1t1);
  a_g1t175 += a_g1t188 * (g1t78);
  a_g1t78 += a_g1t188 * (g1t175);
  double a_g1t20 = a_g1t187 * (-1.0/(g1t20*g1t20));
  a_g1t184 += a_g1t186 * (1.0);
  a_g1t185 += a_g1t186 * (1.0);
  a_g1t111 += a_g1t185 * (g1t179);
  double a_g1t176 = a_g1t185 * (g1t89);
  a_g1t179 += a_g1t185 * (g1t111);
  double a_g1t83 = a_g1t185 * (hDD_dD001);
  a_g1t89 += a_g1t185 * (g1t176);
  a_hDD_dD001 += a_g1t185 * (g1t83);
  a_g1t1 += a_g1t184 * (-1.0);
  a_g1t104 += a_g1t183 * (g1t83);
  a_g1t179 += a_g1t183 * (g1t80);
  a_g1t80 += a_g1t183 * (g1t179);
  a_g1t83 += a_g1t183 * (g1t104);
  a_g1t103 += a_g1t182 * (g1t176);
  a_g1t176 += a_g1t182 * (g1t103);
  a_g1t179 += a_g1t182 * (g1t73);
  a_g1t73 += a_g1t182 * (g1t179);
  a_g1t176 += a_g1t181 * (g1t99);
  a_g1t179 += a_g1t181 * (g1t98);
  a_g1t83 += a_g1t181 * (hDD_dD000);
  a_g1t98 += a_g1t181 * (g1t179);
  a_g1t99 += a_g1t181 * (g1t176);
  a_hDD_dD000 += a_g1t181 * (g1t83);
  a_g1t176 += a_g1t180 * (g1t93);
  a_g1t179 += a_g1t180 * (g1t91);
  a_g1t83 += a_g1t180 * (g1t90);
  a_g1t90 += a_g1t180 * (g1t83);
  a_g1t91 += a_g1t180 * (g1t179);
  a_g1t93 += a_g1t180 * (g1t176);
  a_g1t106 += a_g1t179 * (Rational_1_2);
  a_g1t177 += a_g1t178 * (1.0);
  a_g1t78 += a_g1t178 * (1.0);
  a_g1t176 += a_g1t177 * (g1t81);
  a_g1t74 += a_g1t177 * (g1t83);
  a_g1t81 += a_g1t177 * (g1t176);
  a_g1t83 += a_g1t177 * (g1t74);
  a_g1t96 += a_g1t176 * (Rational_1_2);
  a_g1t167 += a_g1t175 * (vetU_dD21);
  a_g1t174 += a_g1t175 * (1.0);
  a_vetU_dD21 += a_g1t175 * (g1t167);
  a_g1t172 += a_g1t174 * (-g1t173);
  a_g1t173 += a_g1t174 * (-g1t172);
  a_f1_of_xx1__D1 += a_g1t173 * (g1t151);
  a_g1t151 += a_g1t173 * (f1_of_xx1__D1);
  a_g1t1 += a_g1t172 * (vetU2);
  a_vetU2 += a_g1t172 * (g1t1);
  double a_g1t28 = a_g1t171 * (g1t75);
  double a_g1t75 = a_g1t171 * (g1t28);
  a_g1t167 += a_g1t170 * (vetU_dD20);
  a_g1t169 += a_g1t170 * (1.0);
  a_vetU_dD20 += a_g1t170 * (g1t167);
  a_g1t168 += a_g1t169 * (-vetU2);
  a_vetU2 += a_g1t169 * (-g1t168);
  a_g1t128 += a_g1t168 * (g1t68);
  a_g1t68 += a_g1t168 * (g1t128);
  a_g1t1 += a_g1t167 * (g1t68);
  a_g1t68 += a_g1t167 * (g1t1);
  double a_alpha = a_g1t166 * (trK_dD1);
  double a_trK_dD1 = a_g1t166 * (alpha);
  a_alpha += a_g1t165 * (trK_dD0);
  double a_trK_dD0 = a_g1t165 * (alpha);
  a_g1t1 += a_g1t164 * (-Rational_1_3*g1t155*vetU0);
  a_g1t115 += a_g1t164 * ((Rational_1_3)*g1t152*g1t20*g1t78);
  double a_g1t150 = a_g1t164 * ((Rational_1_3)*g1t152*vetU_dD01);
  double a_g1t152 = a_g1t164 * ((Rational_1_3)*g1t115*g1t20*g1t78 + (Rational_1_3)*g1t150*vetU_dD01 + (Rational_1_3)*g1t154*g1t20*vetU0 + (Rational_1_3)*g1t2*(g1t153*g1t160 + g1t153*g1t161));
  double a_g1t153 = a_g1t164 * ((Rational_1_3)*g1t152*g1t2*(g1t160 + g1t161));
  double a_g1t154 = a_g1t164 * ((Rational_1_3)*g1t152*g1t20*vetU0);
  double a_g1t155 = a_g1t164 * (-Rational_1_3*g1t1*vetU0);
  a_g1t159 += a_g1t164 * (Rational_1_3);
  a_g1t160 += a_g1t164 * ((Rational_1_3)*g1t152*g1t153*g1t2);
  a_g1t161 += a_g1t164 * ((Rational_1_3)*g1t152*g1t153*g1t2);
  a_g1t163 += a_g1t164 * (Rational_m2_3);
  a_g1t2 += a_g1t164 * ((Rational_1_3)*g1t152*(g1t153*g1t160 + g1t153*g1t161));
  a_g1t20 += a_g1t164 * ((Rational_1_3)*g1t115*g1t152*g1t78 + (Rational_1_3)*g1t152*g1t154*vetU0);
  a_g1t78 += a_g1t164 * ((Rational_1_3)*g1t115*g1t152*g1t20);
  a_vetU0 += a_g1t164 * (-Rational_1_3*g1t1*g1t155 + (Rational_1_3)*g1t152*g1t154*g1t20);
  a_vetU_dD01 += a_g1t164 * ((Rational_1_3)*g1t150*g1t152);
  a_vetU_dDD001 += a_g1t164 * (Rational_1_3);
  a_g1t162 += a_g1t163 * (g1t2);
  a_g1t2 += a_g1t163 * (g1t162);
  a_g1t151 += a_g1t162 * (g1t160);
  a_g1t160 += a_g1t162 * (g1t151);
  a_f1_of_xx1 += a_g1t161 * (f1_of_xx1__DD11);
  a_f1_of_xx1__DD11 += a_g1t161 * (f1_of_xx1);
  a_f1_of_xx1__D1 += a_g1t160 * (2.0*f1_of_xx1__D1);
  a_g1t1 += a_g1t159 * (vetU_dDD111);
  double a_vetU_dDD111 = a_g1t159 * (g1t1);
  a_g1t129 += a_g1t158 * (-Rational_1_3*g1t155);
  a_g1t131 += a_g1t158 * ((Rational_1_3)*g1t152*g1t153*g1t78);
  a_g1t149 += a_g1t158 * (Rational_m8_3);
  a_g1t150 += a_g1t158 * ((Rational_1_3)*g1t152*vetU_dD00);
  a_g1t152 += a_g1t158 * ((Rational_1_3)*g1t131*g1t153*g1t78 + (Rational_1_3)*g1t150*vetU_dD00 + (Rational_1_3)*g1t154*g1t5*vetU1 + 4.0*g1t8*vetU0);
  a_g1t153 += a_g1t158 * ((Rational_1_3)*g1t131*g1t152*g1t78);
  a_g1t154 += a_g1t158 * ((Rational_1_3)*g1t152*g1t5*vetU1);
  a_g1t155 += a_g1t158 * (-Rational_1_3*g1t129);
  a_g1t157 += a_g1t158 * (Rational_1_3);
  double a_g1t5 = a_g1t158 * ((Rational_1_3)*g1t152*g1t154*vetU1);
  a_g1t78 += a_g1t158 * ((Rational_1_3)*g1t131*g1t152*g1t153);
  double a_g1t8 = a_g1t158 * (4.0*g1t152*vetU0);
  a_vetU0 += a_g1t158 * (4.0*g1t152*g1t8);
  a_vetU1 += a_g1t158 * ((Rational_1_3)*g1t152*g1t154*g1t5);
  a_vetU_dD00 += a_g1t158 * ((Rational_1_3)*g1t150*g1t152);
  a_vetU_dDD000 += a_g1t158 * (Rational_1_3);
  a_g1t1 += a_g1t157 * (vetU_dDD101);
  a_g1t156 += a_g1t157 * (-1.0);
  double a_vetU_dDD101 = a_g1t157 * (g1t1);
  a_g1t128 += a_g1t156 * (vetU_dD11);
  a_vetU_dD11 += a_g1t156 * (g1t128);
  a_g1t69 += a_g1t155 * (4.0);
  a_g1t78 += a_g1t154 * (8.0);
  double a_g1t10 = a_g1t153 * (2.0);
  a_g1t10 += a_g1t152 * (-Rational_1_2*g1t151/(g1t10*g1t10));
  a_g1t151 += a_g1t152 * ((Rational_1_2)/g1t10);
  a_g1t7 += a_g1t151 * (-1.0/(g1t7*g1t7));
  a_g1t20 += a_g1t150 * (4.0*g1t7);
  a_g1t7 += a_g1t150 * (4.0*g1t20);
  a_g1t128 += a_g1t149 * (vetU0);
  a_vetU0 += a_g1t149 * (g1t128);
  a_f0_of_xx0 += a_g1t148 * (g1t143*g1t49);
  double a_g1t118 = a_g1t148 * (g1t143*g1t53);
  double a_g1t143 = a_g1t148 * (f0_of_xx0*g1t49 + g1t118*g1t53 + g1t34*g1t51 + g1t39*g1t41 + g1t39*g1t55 + g1t44*g1t58 + g1t44*g1t61 + g1t47 + g1t63);
  double a_g1t34 = a_g1t148 * (g1t143*g1t51);
  double a_g1t39 = a_g1t148 * (g1t143*(g1t41 + g1t55));
  a_g1t41 += a_g1t148 * (g1t143*g1t39);
  double a_g1t44 = a_g1t148 * (g1t143*(g1t58 + g1t61));
  double a_g1t47 = a_g1t148 * (g1t143);
  double a_g1t49 = a_g1t148 * (f0_of_xx0*g1t143);
  double a_g1t51 = a_g1t148 * (g1t143*g1t34);
  a_g1t53 += a_g1t148 * (g1t118*g1t143);
  a_g1t55 += a_g1t148 * (g1t143*g1t39);
  a_g1t58 += a_g1t148 * (g1t143*g1t44);
  a_g1t61 += a_g1t148 * (g1t143*g1t44);
  double a_g1t63 = a_g1t148 * (g1t143);
  a_g1t12 += a_g1t147 * (g1t143*(g1t137 + g1t139));
  double a_g1t137 = a_g1t147 * (g1t12*g1t143);
  double a_g1t138 = a_g1t147 * (g1t143*g1t22);
  double a_g1t139 = a_g1t147 * (g1t12*g1t143);
  double a_g1t140 = a_g1t147 * (g1t143*g1t22);
  a_g1t143 += a_g1t147 * (g1t12*g1t137 + g1t12*g1t139 + g1t138*g1t22 + g1t140*g1t22 + g1t145 + g1t146 + g1t29*g1t39 + g1t34*g1t41 + g1t44*g1t62);
  a_g1t145 += a_g1t147 * (g1t143);
  a_g1t146 += a_g1t147 * (g1t143);
  a_g1t22 += a_g1t147 * (g1t143*(g1t138 + g1t140));
  a_g1t29 += a_g1t147 * (g1t143*g1t39);
  a_g1t34 += a_g1t147 * (g1t143*g1t41);
  a_g1t39 += a_g1t147 * (g1t143*g1t29);
  a_g1t41 += a_g1t147 * (g1t143*g1t34);
  a_g1t44 += a_g1t147 * (g1t143*g1t62);
  a_g1t62 += a_g1t147 * (g1t143*g1t44);
  double a_g1t141 = a_g1t146 * (g1t28);
  a_g1t28 += a_g1t146 * (g1t141);
  a_g1t12 += a_g1t145 * (g1t135);
  double a_g1t135 = a_g1t145 * (g1t12);
  a_g1t117 += a_g1t144 * (g1t143*g1t44);
  a_g1t136 += a_g1t144 * (g1t143);
  a_g1t137 += a_g1t144 * (g1t143*g1t22);
  a_g1t138 += a_g1t144 * (g1t143*g1t50);
  a_g1t139 += a_g1t144 * (g1t143*g1t22);
  a_g1t140 += a_g1t144 * (g1t143*g1t50);
  a_g1t142 += a_g1t144 * (g1t143);
  a_g1t143 += a_g1t144 * (g1t117*g1t44 + g1t136 + g1t137*g1t22 + g1t138*g1t50 + g1t139*g1t22 + g1t140*g1t50 + g1t142 + g1t34*g1t58 + g1t39*g1t62);
  a_g1t22 += a_g1t144 * (g1t143*(g1t137 + g1t139));
  a_g1t34 += a_g1t144 * (g1t143*g1t58);
  a_g1t39 += a_g1t144 * (g1t143*g1t62);
  a_g1t44 += a_g1t144 * (g1t117*g1t143);
  a_g1t50 += a_g1t144 * (g1t143*(g1t138 + g1t140));
  a_g1t58 += a_g1t144 * (g1t143*g1t34);
  a_g1t62 += a_g1t144 * (g1t143*g1t39);
  a_alpha += a_g1t143 * (4.0);
  a_g1t141 += a_g1t142 * (g1t54);
  double a_g1t54 = a_g1t142 * (g1t141);
  double a_g1t30 = a_g1t141 * (g1t86);
  double a_g1t86 = a_g1t141 * (g1t30);
  a_g1t44 += a_g1t140 * (g1t86);
  a_g1t86 += a_g1t140 * (g1t44);
  a_g1t39 += a_g1t139 * (g1t86);
  a_g1t86 += a_g1t139 * (g1t39);
  a_g1t118 += a_g1t138 * (g1t54);
  a_g1t54 += a_g1t138 * (g1t118);
  a_g1t34 += a_g1t137 * (g1t54);
  a_g1t54 += a_g1t137 * (g1t34);
  a_g1t135 += a_g1t136 * (g1t22);
  a_g1t22 += a_g1t136 * (g1t135);
  double a_g1t18 = a_g1t135 * (g1t28);
  a_g1t28 += a_g1t135 * (g1t18);
  a_g1t133 += a_g1t134 * (2.0);
  a_g1t22 += a_g1t133 * (g1t75);
  a_g1t75 += a_g1t133 * (g1t22);
  a_f0_of_xx0 += a_g1t132 * (g1t131);
  a_g1t131 += a_g1t132 * (f0_of_xx0);
  a_g1t1 += a_g1t131 * (vetU_dD10);
  a_g1t130 += a_g1t131 * (1.0);
  a_vetU_dD10 += a_g1t131 * (g1t1);
  a_g1t129 += a_g1t130 * (-1.0);
  a_g1t128 += a_g1t129 * (vetU1);
  a_vetU1 += a_g1t129 * (g1t128);
  a_g1t5 += a_g1t128 * (-1.0/(g1t5*g1t5));
  a_g1t0 += a_g1t127 * (g1t118*g1t124 + g1t123 + g1t125 + g1t126*g1t60 + g1t52*g1t53 + g1t57*g1t61);
  a_g1t118 += a_g1t127 * (g1t0*g1t124);
  a_g1t123 += a_g1t127 * (g1t0);
  a_g1t124 += a_g1t127 * (g1t0*g1t118);
  a_g1t125 += a_g1t127 * (g1t0);
  a_g1t126 += a_g1t127 * (g1t0*g1t60);
  a_g1t52 += a_g1t127 * (g1t0*g1t53);
  a_g1t53 += a_g1t127 * (g1t0*g1t52);
  a_g1t57 += a_g1t127 * (g1t0*g1t61);
  a_g1t60 += a_g1t127 * (g1t0*g1t126);
  a_g1t61 += a_g1t127 * (g1t0*g1t57);
  a_g1t50 += a_g1t126 * (g1t54);
  a_g1t54 += a_g1t126 * (g1t50);
  a_g1t117 += a_g1t125 * (g1t30);
  a_g1t30 += a_g1t125 * (g1t117);
  a_g1t50 += a_g1t124 * (2.0*g1t50);
  a_g1t18 += a_g1t123 * (g1t23);
  a_g1t23 += a_g1t123 * (g1t18);
  a_g1t0 += a_g1t122 * (g1t118*g1t23 + g1t19 + g1t31 + g1t32*g1t52 + g1t36*g1t57 + g1t41*g1t60);
  a_g1t118 += a_g1t122 * (g1t0*g1t23);
  a_g1t19 += a_g1t122 * (g1t0);
  a_g1t23 += a_g1t122 * (g1t0*g1t118);
  a_g1t31 += a_g1t122 * (g1t0);
  a_g1t32 += a_g1t122 * (g1t0*g1t52);
  a_g1t36 += a_g1t122 * (g1t0*g1t57);
  a_g1t41 += a_g1t122 * (g1t0*g1t60);
  a_g1t52 += a_g1t122 * (g1t0*g1t32);
  a_g1t57 += a_g1t122 * (g1t0*g1t36);
  a_g1t60 += a_g1t122 * (g1t0*g1t41);
  a_g1t0 += a_g1t121 * (g1t117*g1t118 + g1t119*g1t28 + g1t120*g1t54 + g1t18*g1t29 + g1t30*(g1t86*g1t86) + g1t52*g1t62);
  a_g1t117 += a_g1t121 * (g1t0*g1t118);
  a_g1t118 += a_g1t121 * (g1t0*g1t117);
  a_g1t119 += a_g1t121 * (g1t0*g1t28);
  a_g1t120 += a_g1t121 * (g1t0*g1t54);
  a_g1t18 += a_g1t121 * (g1t0*g1t29);
  a_g1t28 += a_g1t121 * (g1t0*g1t119);
  a_g1t29 += a_g1t121 * (g1t0*g1t18);
  a_g1t30 += a_g1t121 * (g1t0*(g1t86*g1t86));
  a_g1t52 += a_g1t121 * (g1t0*g1t62);
  a_g1t54 += a_g1t121 * (g1t0*g1t120);
  a_g1t62 += a_g1t121 * (g1t0*g1t52);
  a_g1t86 += a_g1t121 * (2.0*g1t0*g1t30*g1t86);
  a_g1t60 += a_g1t120 * (g1t86);
  a_g1t86 += a_g1t120 * (g1t60);
  a_g1t57 += a_g1t119 * (g1t86);
  a_g1t86 += a_g1t119 * (g1t57);
  double a_g1t25 = a_g1t118 * (g1t5);
  a_g1t5 += a_g1t118 * (g1t25);
  a_g1t54 += a_g1t117 * (2.0*g1t54);
  a_g1t1 += a_g1t116 * (vetU_dD01);
  a_vetU_dD01 += a_g1t116 * (g1t1);
  a_vetU_dD11 += a_g1t115 * (2.0);
  a_vetU1 += a_g1t114 * (2.0);
  double a_g1t109 = a_g1t113 * (g1t22);
  a_g1t22 += a_g1t113 * (g1t109);
  a_g1t111 += a_g1t112 * (g1t92);
  double a_g1t77 = a_g1t112 * (hDD_dD001);
  a_g1t83 += a_g1t112 * (g1t89);
  a_g1t89 += a_g1t112 * (g1t83);
  a_g1t92 += a_g1t112 * (g1t111);
  a_hDD_dD001 += a_g1t112 * (g1t77);
  a_f0_of_xx0 += a_g1t111 * (f1_of_xx1__D1*hDD02);
  a_f1_of_xx1__D1 += a_g1t111 * (f0_of_xx0*hDD02);
  double a_g1t102 = a_g1t111 * (1.0);
  a_g1t37 += a_g1t111 * (hDD_dD021);
  double a_hDD02 = a_g1t111 * (f0_of_xx0*f1_of_xx1__D1);
  double a_hDD_dD021 = a_g1t111 * (g1t37);
  a_g1t109 += a_g1t110 * (g1t28);
  a_g1t28 += a_g1t110 * (g1t109);
  a_g1t75 += a_g1t109 * (Rational_4_3);
  a_g1t103 += a_g1t108 * (g1t83);
  a_g1t73 += a_g1t108 * (g1t92);
  a_g1t83 += a_g1t108 * (g1t103);
  a_g1t92 += a_g1t108 * (g1t73);
  a_g1t106 += a_g1t107 * (Rational_4_3);
  a_g1t54 += a_g1t106 * (g1t75);
  a_g1t75 += a_g1t106 * (g1t54);
  a_g1t104 += a_g1t105 * (g1t77);
  a_g1t77 += a_g1t105 * (g1t104);
  a_g1t80 += a_g1t105 * (g1t92);
  a_g1t92 += a_g1t105 * (g1t80);
  a_g1t103 += a_g1t104 * (-1.0);
  a_f0_of_xx0 += a_g1t103 * (-f1_of_xx1*hDD_dD021 - f1_of_xx1__D1*hDD02);
  a_f1_of_xx1 += a_g1t103 * (-f0_of_xx0*hDD_dD021);
  a_f1_of_xx1__D1 += a_g1t103 * (-f0_of_xx0*hDD02);
  a_g1t102 += a_g1t103 * (1.0);
  a_hDD02 += a_g1t103 * (-f0_of_xx0*f1_of_xx1__D1);
  a_hDD_dD021 += a_g1t103 * (-f0_of_xx0*f1_of_xx1);
  double a_g1t42 = a_g1t102 * (hDD_dD120);
  double a_g1t56 = a_g1t102 * (hDD12);
  double a_hDD12 = a_g1t102 * (g1t56);
  double a_hDD_dD120 = a_g1t102 * (g1t42);
  a_g1t76 += a_g1t101 * (Rational_2_3);
  a_g1t77 += a_g1t100 * (hDD_dD000);
  a_g1t83 += a_g1t100 * (g1t99);
  a_g1t92 += a_g1t100 * (g1t98);
  a_g1t98 += a_g1t100 * (g1t92);
  a_g1t99 += a_g1t100 * (g1t83);
  a_hDD_dD000 += a_g1t100 * (g1t77);
  double a_g1t48 = a_g1t99 * (hDD_dD010);
  double a_hDD01 = a_g1t99 * (2.0);
  a_hDD_dD001 += a_g1t99 * (-1.0);
  double a_hDD_dD010 = a_g1t99 * (g1t48);
  double a_g1t27 = a_g1t98 * (2.0);
  a_g1t56 += a_g1t98 * (hDD_dD020);
  double a_hDD_dD020 = a_g1t98 * (g1t56);
  a_g1t96 += a_g1t97 * (Rational_2_3);
  a_g1t50 += a_g1t96 * (g1t75);
  a_g1t75 += a_g1t96 * (g1t50);
  a_f0_of_xx0 += a_g1t95 * (1.0);
  a_g1t94 += a_g1t95 * (1.0);
  a_g1t77 += a_g1t94 * (g1t90);
  a_g1t83 += a_g1t94 * (g1t93);
  a_g1t90 += a_g1t94 * (g1t77);
  a_g1t91 += a_g1t94 * (g1t92);
  a_g1t92 += a_g1t94 * (g1t91);
  a_g1t93 += a_g1t94 * (g1t83);
  a_g1t5 += a_g1t93 * (hDD_dD111);
  double a_hDD_dD111 = a_g1t93 * (g1t5);
  a_g1t28 += a_g1t92 * (g1t82);
  double a_g1t82 = a_g1t92 * (g1t28);
  a_f1_of_xx1__D1 += a_g1t91 * (g1t24*hDD12);
  double a_g1t24 = a_g1t91 * (f1_of_xx1__D1*hDD12);
  double a_g1t59 = a_g1t91 * (hDD_dD121);
  a_hDD12 += a_g1t91 * (f1_of_xx1__D1*g1t24);
  double a_hDD_dD121 = a_g1t91 * (g1t59);
  a_f0_of_xx0 += a_g1t90 * (2.0*hDD_dD011);
  a_g1t89 += a_g1t90 * (-1.0);
  double a_hDD_dD011 = a_g1t90 * (2.0*f0_of_xx0);
  a_g1t48 += a_g1t89 * (hDD11 + 1.0);
  a_g1t5 += a_g1t89 * (hDD_dD110);
  double a_hDD11 = a_g1t89 * (g1t48);
  double a_hDD_dD110 = a_g1t89 * (g1t5);
  a_g1t87 += a_g1t88 * (Rational_2_3);
  a_g1t75 += a_g1t87 * (g1t86);
  a_g1t86 += a_g1t87 * (g1t75);
  double a_g1t13 = a_g1t86 * (-1.0);
  double a_g1t14 = a_g1t86 * (g1t6);
  double a_g1t6 = a_g1t86 * (g1t14);
  a_g1t71 += a_g1t85 * (1.0);
  a_g1t84 += a_g1t85 * (1.0);
  a_g1t74 += a_g1t84 * (g1t77);
  a_g1t77 += a_g1t84 * (g1t74);
  a_g1t81 += a_g1t84 * (g1t83);
  a_g1t83 += a_g1t84 * (g1t81);
  a_g1t22 += a_g1t83 * (g1t82);
  a_g1t82 += a_g1t83 * (g1t22);
  a_g1t75 += a_g1t82 * (Rational_1_2);
  a_g1t80 += a_g1t81 * (-1.0);
  double a_g1t79 = a_g1t80 * (hDD22 + 1.0);
  a_g1t8 += a_g1t80 * (hDD_dD221);
  double a_hDD22 = a_g1t80 * (g1t79);
  double a_hDD_dD221 = a_g1t80 * (g1t8);
  a_g1t24 += a_g1t79 * (g1t78);
  a_g1t78 += a_g1t79 * (g1t24);
  a_f1_of_xx1 += a_g1t78 * (f1_of_xx1__D1);
  a_f1_of_xx1__D1 += a_g1t78 * (f1_of_xx1);
  a_g1t76 += a_g1t77 * (Rational_1_2);
  a_g1t12 += a_g1t76 * (g1t75);
  a_g1t75 += a_g1t76 * (g1t12);
  double a_g1t16 = a_g1t75 * (-1.0/(g1t16*g1t16));
  a_g1t73 += a_g1t74 * (-1.0);
  a_g1t72 += a_g1t73 * (hDD22 + 1.0);
  a_g1t8 += a_g1t73 * (hDD_dD220);
  a_hDD22 += a_g1t73 * (g1t72);
  double a_hDD_dD220 = a_g1t73 * (g1t8);
  a_g1t71 += a_g1t72 * (2.0);
  a_f0_of_xx0 += a_g1t71 * (g1t7);
  a_g1t7 += a_g1t71 * (f0_of_xx0);
  a_g1t2 += a_g1t70 * (g1t69);
  a_g1t65 += a_g1t70 * (1.0);
  a_g1t67 += a_g1t70 * (1.0);
  a_g1t69 += a_g1t70 * (g1t2);
  a_vetU_dD00 += a_g1t70 * (1.0);
  a_f1_of_xx1__D1 += a_g1t69 * (g1t68);
  a_g1t68 += a_g1t69 * (f1_of_xx1__D1);
  a_f1_of_xx1 += a_g1t68 * (-1.0/(f1_of_xx1*f1_of_xx1));
  a_g1t66 += a_g1t67 * (vetU0);
  a_vetU0 += a_g1t67 * (g1t66);
  a_g1t1 += a_g1t66 * (2.0);
  a_g1t1 += a_g1t65 * (vetU_dD11);
  a_vetU_dD11 += a_g1t65 * (g1t1);
  a_g1t26 += a_g1t64 * (-g1t53);
  a_g1t41 += a_g1t64 * (-g1t57);
  a_g1t47 += a_g1t64 * (-2.0);
  a_g1t48 += a_g1t64 * (-g1t49);
  a_g1t49 += a_g1t64 * (-g1t48);
  a_g1t51 += a_g1t64 * (-g1t52);
  a_g1t52 += a_g1t64 * (-g1t51);
  a_g1t53 += a_g1t64 * (-g1t26);
  a_g1t55 += a_g1t64 * (-g1t57);
  a_g1t57 += a_g1t64 * (-g1t41 - g1t55);
  a_g1t58 += a_g1t64 * (-g1t60);
  a_g1t60 += a_g1t64 * (-g1t58 - g1t61);
  a_g1t61 += a_g1t64 * (-g1t60);
  a_g1t63 += a_g1t64 * (-2.0);
  a_g1t30 += a_g1t63 * (g1t62);
  a_g1t62 += a_g1t63 * (g1t30);
  a_g1t28 += a_g1t62 * (g1t54);
  a_g1t54 += a_g1t62 * (g1t28);
  a_g1t22 += a_g1t61 * (g1t54);
  a_g1t54 += a_g1t61 * (g1t22);
  double a_g1t43 = a_g1t60 * (g1t59);
  a_g1t59 += a_g1t60 * (g1t43);
  a_g1t42 += a_g1t59 * (2.0);
  a_g1t28 += a_g1t58 * (g1t50);
  a_g1t50 += a_g1t58 * (g1t28);
  double a_g1t38 = a_g1t57 * (g1t56);
  a_g1t56 += a_g1t57 * (g1t38);
  a_f1_of_xx1 += a_g1t56 * (g1t48);
  a_g1t48 += a_g1t56 * (f1_of_xx1);
  a_g1t12 += a_g1t55 * (g1t54);
  a_g1t54 += a_g1t55 * (g1t12);
  a_g1t14 += a_g1t54 * (-g1t42*hDD12);
  a_g1t27 += a_g1t54 * (g1t5*hDD01);
  a_g1t42 += a_g1t54 * (-g1t14*hDD12);
  a_g1t5 += a_g1t54 * (g1t27*hDD01);
  a_hDD01 += a_g1t54 * (g1t27*g1t5);
  a_hDD12 += a_g1t54 * (-g1t14*g1t42);
  a_g1t22 += a_g1t53 * (g1t50);
  a_g1t50 += a_g1t53 * (g1t22);
  double a_g1t33 = a_g1t52 * (g1t48);
  a_g1t48 += a_g1t52 * (g1t33);
  a_g1t12 += a_g1t51 * (g1t50);
  a_g1t50 += a_g1t51 * (g1t12);
  a_g1t14 += a_g1t50 * (g1t9);
  double a_g1t15 = a_g1t50 * (-1.0);
  double a_g1t9 = a_g1t50 * (g1t14);
  a_g1t23 += a_g1t49 * (g1t33);
  a_g1t33 += a_g1t49 * (g1t23);
  a_f0_of_xx0 += a_g1t48 * (2.0);
  a_g1t18 += a_g1t47 * (g1t32);
  a_g1t32 += a_g1t47 * (g1t18);
  double a_alpha_dD1 = a_g1t46 * (1.0);
  double a_cf_dD1 = a_g1t46 * (g1t3);
  double a_g1t3 = a_g1t46 * (cf_dD1);
  a_g1t44 += a_g1t45 * (4.0);
  a_g1t42 += a_g1t44 * (g1t43);
  a_g1t43 += a_g1t44 * (g1t42);
  double a_aDD12 = a_g1t43 * (g1t17);
  double a_g1t17 = a_g1t43 * (aDD12);
  a_f1_of_xx1 += a_g1t42 * (g1t5);
  a_g1t5 += a_g1t42 * (f1_of_xx1);
  a_g1t22 += a_g1t41 * (g1t28);
  a_g1t28 += a_g1t41 * (g1t22);
  a_g1t39 += a_g1t40 * (4.0);
  a_g1t37 += a_g1t39 * (g1t38);
  a_g1t38 += a_g1t39 * (g1t37);
  double a_aDD02 = a_g1t38 * (g1t17);
  a_g1t17 += a_g1t38 * (aDD02);
  a_f0_of_xx0 += a_g1t37 * (f1_of_xx1);
  a_f1_of_xx1 += a_g1t37 * (f0_of_xx0);
  a_g1t12 += a_g1t36 * (g1t28);
  a_g1t28 += a_g1t36 * (g1t12);
  a_g1t34 += a_g1t35 * (4.0);
  a_f0_of_xx0 += a_g1t34 * (g1t33);
  a_g1t33 += a_g1t34 * (f0_of_xx0);
  double a_aDD01 = a_g1t33 * (g1t17);
  a_g1t17 += a_g1t33 * (aDD01);
  a_g1t12 += a_g1t32 * (g1t22);
  a_g1t22 += a_g1t32 * (g1t12);
  a_g1t29 += a_g1t31 * (g1t30);
  a_g1t30 += a_g1t31 * (g1t29);
  double a_aDD22 = a_g1t30 * (g1t17*g1t8);
  a_g1t17 += a_g1t30 * (aDD22*g1t8);
  a_g1t8 += a_g1t30 * (aDD22*g1t17);
  a_g1t28 += a_g1t29 * (2.0*g1t28);
  a_f0_of_xx0 += a_g1t28 * (-g1t27*g1t6);
  a_f1_of_xx1 += a_g1t28 * (g1t21*hDD01);
  double a_g1t21 = a_g1t28 * (f1_of_xx1*hDD01);
  a_g1t27 += a_g1t28 * (-f0_of_xx0*g1t6);
  a_g1t6 += a_g1t28 * (-f0_of_xx0*g1t27);
  a_hDD01 += a_g1t28 * (f1_of_xx1*g1t21);
  a_f1_of_xx1 += a_g1t27 * (hDD02);
  a_hDD02 += a_g1t27 * (f1_of_xx1);
  a_g1t24 += a_g1t26 * (g1t25);
  a_g1t25 += a_g1t26 * (g1t24);
  double a_aDD11 = a_g1t25 * (g1t17);
  a_g1t17 += a_g1t25 * (aDD11);
  a_g1t5 += a_g1t24 * (2.0);
  a_g1t22 += a_g1t23 * (2.0*g1t22);
  a_f0_of_xx0 += a_g1t22 * (-g1t9*hDD01);
  a_g1t21 += a_g1t22 * (g1t7*hDD02);
  a_g1t7 += a_g1t22 * (g1t21*hDD02);
  a_g1t9 += a_g1t22 * (-f0_of_xx0*hDD01);
  a_hDD01 += a_g1t22 * (-f0_of_xx0*g1t9);
  a_hDD02 += a_g1t22 * (g1t21*g1t7);
  a_g1t20 += a_g1t21 * (hDD12);
  a_hDD12 += a_g1t21 * (g1t20);
  a_f0_of_xx0 += a_g1t20 * (3.0*(f0_of_xx0*f0_of_xx0));
  a_g1t12 += a_g1t19 * (2.0*g1t12*g1t18);
  a_g1t18 += a_g1t19 * ((g1t12*g1t12));
  double a_aDD00 = a_g1t18 * (g1t17);
  a_g1t17 += a_g1t18 * (aDD00);
  a_g1t16 += a_g1t17 * (-2.0/(g1t16*g1t16*g1t16));
  a_g1t10 += a_g1t16 * (2.0*g1t7*hDD01*hDD02*hDD12);
  double a_g1t11 = a_g1t16 * (-g1t14);
  a_g1t13 += a_g1t16 * (-g1t9);
  a_g1t14 += a_g1t16 * (-g1t11 + g1t6*g1t9);
  a_g1t15 += a_g1t16 * (-g1t6);
  a_g1t6 += a_g1t16 * (g1t14*g1t9 - g1t15);
  a_g1t7 += a_g1t16 * (2.0*g1t10*hDD01*hDD02*hDD12);
  a_g1t9 += a_g1t16 * (-g1t13 + g1t14*g1t6);
  a_hDD01 += a_g1t16 * (2.0*g1t10*g1t7*hDD02*hDD12);
  a_hDD02 += a_g1t16 * (2.0*g1t10*g1t7*hDD01*hDD12);
  a_hDD12 += a_g1t16 * (2.0*g1t10*g1t7*hDD01*hDD02);
  a_g1t8 += a_g1t15 * ((hDD02*hDD02));
  a_hDD02 += a_g1t15 * (2.0*g1t8*hDD02);
  double a_hDD00 = a_g1t14 * (1.0);
  a_g1t5 += a_g1t13 * ((hDD01*hDD01));
  a_hDD01 += a_g1t13 * (2.0*g1t5*hDD01);
  a_g1t11 += a_g1t12 * (-1.0);
  a_g1t6 += a_g1t12 * (g1t9);
  a_g1t9 += a_g1t12 * (g1t6);
  a_g1t10 += a_g1t11 * (g1t7*(hDD12*hDD12));
  a_g1t7 += a_g1t11 * (g1t10*(hDD12*hDD12));
  a_hDD12 += a_g1t11 * (2.0*g1t10*g1t7*hDD12);
  a_f0_of_xx0 += a_g1t10 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_g1t8 += a_g1t9 * (hDD22 + 1.0);
  a_hDD22 += a_g1t9 * (g1t8);
  a_g1t5 += a_g1t8 * (g1t7);
  a_g1t7 += a_g1t8 * (g1t5);
  a_f1_of_xx1 += a_g1t7 * (2.0*f1_of_xx1);
  a_g1t5 += a_g1t6 * (hDD11 + 1.0);
  a_hDD11 += a_g1t6 * (g1t5);
  a_f0_of_xx0 += a_g1t5 * (2.0*f0_of_xx0);
  double a_alpha_dD0 = a_g1t4 * (1.0);
  double a_cf_dD0 = a_g1t4 * (g1t3);
  a_g1t3 += a_g1t4 * (cf_dD0);
  a_alpha += a_g1t3 * (3.0/cf);
  double a_cf = a_g1t3 * (-3.0*alpha/(cf*cf));
  a_g1t1 += a_g1t2 * (vetU1);
  a_vetU1 += a_g1t2 * (g1t1);
  a_f0_of_xx0 += a_g1t1 * (-1.0/(f0_of_xx0*f0_of_xx0));
  a_alpha += a_g1t0 * (2.0);
  red[68 * 64 + lane] = a_aDD00;
  red[69 * 64 + lane] = a_aDD01;
  red[70 * 64 + lane] = a_aDD02;
  red[71 * 64 + lane] = a_aDD11;
  red[72 * 64 + lane] = a_aDD12;
  red[73 * 64 + lane] = a_aDD22;
  red[74 * 64 + lane] = a_alpha;
  red[75 * 64 + lane] = a_alpha_dD0;
  red[76 * 64 + lane] = a_alpha_dD1;
  red[77 * 64 + lane] = (betaU0 > 0.0) ? a_alpha_dupD0 : 0.0;
  red[78 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_alpha_dupD0;
  red[79 * 64 + lane] = (betaU1 > 0.0) ? a_alpha_dupD1 : 0.0;
  red[80 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_alpha_dupD1;
  red[81 * 64 + lane] = a_betU0;
  red[82 * 64 + lane] = a_betU1;
  red[83 * 64 + lane] = a_betU2;
  red[84 * 64 + lane] = a_cf;
  red[85 * 64 + lane] = a_cf_dD0;
  red[86 * 64 + lane] = a_cf_dD1;
  red[87 * 64 + lane] = a_hDD00;
  red[88 * 64 + lane] = a_hDD01;
  red[89 * 64 + lane] = a_hDD02;
  red[90 * 64 + lane] = a_hDD11;
  red[91 * 64 + lane] = a_hDD12;
  red[92 * 64 + lane] = a_hDD22;
  red[93 * 64 + lane] = a_hDD_dD000;
  red[94 * 64 + lane] = a_hDD_dD001;
  red[95 * 64 + lane] = a_hDD_dD010;
  red[96 * 64 + lane] = a_hDD_dD011;
  red[97 * 64 + lane] = a_hDD_dD020;
  red[98 * 64 + lane] = a_hDD_dD021;
  red[99 * 64 + lane] = a_hDD_dD110;
  red[100 * 64 + lane] = a_hDD_dD111;
  red[101 * 64 + lane] = a_hDD_dD120;
  red[102 * 64 + lane] = a_hDD_dD121;
  red[103 * 64 + lane] = a_hDD_dD220;
  red[104 * 64 + lane] = a_hDD_dD221;
  red[105 * 64 + lane] = a_lambdaU0;
  red[106 * 64 + lane] = a_lambdaU1;
  red[107 * 64 + lane] = a_lambdaU2;
  red[108 * 64 + lane] = (betaU0 > 0.0) ? a_lambdaU_dupD00 : 0.0;
  red[109 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_lambdaU_dupD00;
  red[110 * 64 + lane] = (betaU1 > 0.0) ? a_lambdaU_dupD01 : 0.0;
  red[111 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_lambdaU_dupD01;
  red[112 * 64 + lane] = (betaU0 > 0.0) ? a_lambdaU_dupD10 : 0.0;
  red[113 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_lambdaU_dupD10;
  red[114 * 64 + lane] = (betaU1 > 0.0) ? a_lambdaU_dupD11 : 0.0;
  red[115 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_lambdaU_dupD11;
  red[116 * 64 + lane] = (betaU0 > 0.0) ? a_lambdaU_dupD20 : 0.0;
  red[117 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_lambdaU_dupD20;
  red[118 * 64 + lane] = (betaU1 > 0.0) ? a_lambdaU_dupD21 : 0.0;
  red[119 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_lambdaU_dupD21;
  red[120 * 64 + lane] = a_trK;
  red[121 * 64 + lane] = a_trK_dD0;
  red[122 * 64 + lane] = a_trK_dD1;
  red[123 * 64 + lane] = a_vetU0;
  red[124 * 64 + lane] = a_vetU1;
  red[125 * 64 + lane] = a_vetU2;
  red[126 * 64 + lane] = a_vetU_dD00;
  red[127 * 64 + lane] = a_vetU_dD01;
  red[128 * 64 + lane] = a_vetU_dD10;
  red[129 * 64 + lane] = a_vetU_dD11;
  red[130 * 64 + lane] = a_vetU_dD20;
  red[131 * 64 + lane] = a_vetU_dD21;
  red[132 * 64 + lane] = a_vetU_dDD000;
  red[133 * 64 + lane] = a_vetU_dDD001;
  red[134 * 64 + lane] = a_vetU_dDD011;
  red[135 * 64 + lane] = a_vetU_dDD100;
  red[136 * 64 + lane] = a_vetU_dDD101;
  red[137 * 64 + lane] = a_vetU_dDD111;
  red[138 * 64 + lane] = a_vetU_dDD200;
  red[139 * 64 + lane] = a_vetU_dDD201;
  red[140 * 64 + lane] = a_vetU_dDD211;
  red[141 * 64 + lane] = (betaU0 > 0.0) ? a_vetU_dupD00 : 0.0;
  red[142 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_vetU_dupD00;
  red[143 * 64 + lane] = (betaU1 > 0.0) ? a_vetU_dupD01 : 0.0;
  red[144 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_vetU_dupD01;
  red[145 * 64 + lane] = (betaU0 > 0.0) ? a_vetU_dupD10 : 0.0;
  red[146 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_vetU_dupD10;
  red[147 * 64 + lane] = (betaU1 > 0.0) ? a_vetU_dupD11 : 0.0;
  red[148 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_vetU_dupD11;
  red[149 * 64 + lane] = (betaU0 > 0.0) ? a_vetU_dupD20 : 0.0;
  red[150 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_vetU_dupD20;
  red[151 * 64 + lane] = (betaU1 > 0.0) ? a_vetU_dupD21 : 0.0;
  red[152 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_vetU_dupD21;
  break;
  }
  case 2: { // aDD00, aDD01, aDD02, aDD11, aDD12, aDD22, cf, hDD00, hDD01, hDD02, hDD11, hDD12, hDD22, trK
  const double RbarDD00 = aux[0 * Ntot + idx];
  const double RbarDD01 = aux[1 * Ntot + idx];
  const double RbarDD02 = aux[2 * Ntot + idx];
  const double RbarDD11 = aux[3 * Ntot + idx];
  const double RbarDD12 = aux[4 * Ntot + idx];
  const double RbarDD22 = aux[5 * Ntot + idx];
  const double aDD00 = in[idx];
  const double aDD01 = in[1 * Ntot + idx];
  const double aDD02 = in[2 * Ntot + idx];
  const double aDD11 = in[3 * Ntot + idx];
  const double aDD12 = in[4 * Ntot + idx];
  const double aDD22 = in[5 * Ntot + idx];
  const double aDD_dupD000 = p.invdxx0 * (uw0[0] * in[idx + (-3)] + uw0[1] * in[idx + (-2)] + uw0[2] * in[idx + (-1)] + uw0[3] * in[idx] + uw0[4] * in[idx + (1)] + uw0[5] * in[idx + (2)] + uw0[6] * in[idx + (3)]);
  const double aDD_dupD001 = p.invdxx1 * (uw1[0] * in[idx + (-3 * s1)] + uw1[1] * in[idx + (-2 * s1)] + uw1[2] * in[idx + (-1 * s1)] + uw1[3] * in[idx] + uw1[4] * in[idx + (1 * s1)] + uw1[5] * in[idx + (2 * s1)] + uw1[6] * in[idx + (3 * s1)]);
  const double aDD_dupD010 = p.invdxx0 * (uw0[0] * in[1 * Ntot + idx + (-3)] + uw0[1] * in[1 * Ntot + idx + (-2)] + uw0[2] * in[1 * Ntot + idx + (-1)] + uw0[3] * in[1 * Ntot + idx] + uw0[4] * in[1 * Ntot + idx + (1)] + uw0[5] * in[1 * Ntot + idx + (2)] + uw0[6] * in[1 * Ntot + idx + (3)]);
  const double aDD_dupD011 = p.invdxx1 * (uw1[0] * in[1 * Ntot + idx + (-3 * s1)] + uw1[1] * in[1 * Ntot + idx + (-2 * s1)] + uw1[2] * in[1 * Ntot + idx + (-1 * s1)] + uw1[3] * in[1 * Ntot + idx] + uw1[4] * in[1 * Ntot + idx + (1 * s1)] + uw1[5] * in[1 * Ntot + idx + (2 * s1)] + uw1[6] * in[1 * Ntot + idx + (3 * s1)]);
  const double aDD_dupD020 = p.invdxx0 * (uw0[0] * in[2 * Ntot + idx + (-3)] + uw0[1] * in[2 * Ntot + idx + (-2)] + uw0[2] * in[2 * Ntot + idx + (-1)] + uw0[3] * in[2 * Ntot + idx] + uw0[4] * in[2 * Ntot + idx + (1)] + uw0[5] * in[2 * Ntot + idx + (2)] + uw0[6] * in[2 * Ntot + idx + (3)]);
  const double aDD_dupD021 = p.invdxx1 * (uw1[0] * in[2 * Ntot + idx + (-3 * s1)] + uw1[1] * in[2 * Ntot + idx + (-2 * s1)] + uw1[2] * in[2 * Ntot + idx + (-1 * s1)] + uw1[3] * in[2 * Ntot + idx] + uw1[4] * in[2 * Ntot + idx + (1 * s1)] + uw1[5] * in[2 * Ntot + idx + (2 * s1)] + uw1[6] * in[2 * Ntot + idx + (3 * s1)]);
  const double aDD_dupD110 = p.invdxx0 * (uw0[0] * in[3 * Ntot + idx + (-3)] + uw0[1] * in[3 * Ntot + idx + (-2)] + uw0[2] * in[3 * Ntot + idx + (-1)] + uw0[3] * in[3 * Ntot + idx] + uw0[4] * in[3 * Ntot + idx + (1)] + uw0[5] * in[3 * Ntot + idx + (2)] + uw0[6] * in[3 * Ntot + idx + (3)]);
  const double aDD_dupD111 = p.invdxx1 * (uw1[0] * in[3 * Ntot + idx + (-3 * s1)] + uw1[1] * in[3 * Ntot + idx + (-2 * s1)] + uw1[2] * in[3 * Ntot + idx + (-1 * s1)] + uw1[3] * in[3 * Ntot + idx] + uw1[4] * in[3 * Ntot + idx + (1 * s1)] + uw1[5] * in[3 * Ntot + idx + (2 * s1)] + uw1[6] * in[3 * Ntot + idx + (3 * s1)]);
  const double aDD_dupD120 = p.invdxx0 * (uw0[0] * in[4 * Ntot + idx + (-3)] + uw0[1] * in[4 * Ntot + idx + (-2)] + uw0[2] * in[4 * Ntot + idx + (-1)] + uw0[3] * in[4 * Ntot + idx] + uw0[4] * in[4 * Ntot + idx + (1)] + uw0[5] * in[4 * Ntot + idx + (2)] + uw0[6] * in[4 * Ntot + idx + (3)]);
  const double aDD_dupD121 = p.invdxx1 * (uw1[0] * in[4 * Ntot + idx + (-3 * s1)] + uw1[1] * in[4 * Ntot + idx + (-2 * s1)] + uw1[2] * in[4 * Ntot + idx + (-1 * s1)] + uw1[3] * in[4 * Ntot + idx] + uw1[4] * in[4 * Ntot + idx + (1 * s1)] + uw1[5] * in[4 * Ntot + idx + (2 * s1)] + uw1[6] * in[4 * Ntot + idx + (3 * s1)]);
  const double aDD_dupD220 = p.invdxx0 * (uw0[0] * in[5 * Ntot + idx + (-3)] + uw0[1] * in[5 * Ntot + idx + (-2)] + uw0[2] * in[5 * Ntot + idx + (-1)] + uw0[3] * in[5 * Ntot + idx] + uw0[4] * in[5 * Ntot + idx + (1)] + uw0[5] * in[5 * Ntot + idx + (2)] + uw0[6] * in[5 * Ntot + idx + (3)]);
  const double aDD_dupD221 = p.invdxx1 * (uw1[0] * in[5 * Ntot + idx + (-3 * s1)] + uw1[1] * in[5 * Ntot + idx + (-2 * s1)] + uw1[2] * in[5 * Ntot + idx + (-1 * s1)] + uw1[3] * in[5 * Ntot + idx] + uw1[4] * in[5 * Ntot + idx + (1 * s1)] + uw1[5] * in[5 * Ntot + idx + (2 * s1)] + uw1[6] * in[5 * Ntot + idx + (3 * s1)]);
  const double alpha = in[6 * Ntot + idx];
  const double alpha_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[6 * Ntot + idx + (1)] - in[6 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2)] - in[6 * Ntot + idx + (-2)]));
  const double alpha_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[6 * Ntot + idx + (1 * s1)] - in[6 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2 * s1)] - in[6 * Ntot + idx + (-2 * s1)]));
  const double alpha_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[6 * Ntot + idx] + (4.0 / 3.0) * (in[6 * Ntot + idx + (1)] + in[6 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2)] + in[6 * Ntot + idx + (-2)]));
  const double alpha_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[6 * Ntot + idx + (1 + 1 * s1)] - in[6 * Ntot + idx + (1 + -1 * s1)]) - (in[6 * Ntot + idx + (-1 + 1 * s1)] - in[6 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[6 * Ntot + idx + (1 + 2 * s1)] - in[6 * Ntot + idx + (1 + -2 * s1)]) - (in[6 * Ntot + idx + (-1 + 2 * s1)] - in[6 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[6 * Ntot + idx + (2 + 1 * s1)] - in[6 * Ntot + idx + (2 + -1 * s1)]) - (in[6 * Ntot + idx + (-2 + 1 * s1)] - in[6 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[6 * Ntot + idx + (2 + 2 * s1)] - in[6 * Ntot + idx + (2 + -2 * s1)]) - (in[6 * Ntot + idx + (-2 + 2 * s1)] - in[6 * Ntot + idx + (-2 + -2 * s1)])));
  const double alpha_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[6 * Ntot + idx] + (4.0 / 3.0) * (in[6 * Ntot + idx + (1 * s1)] + in[6 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[6 * Ntot + idx + (2 * s1)] + in[6 * Ntot + idx + (-2 * s1)]));
  const double cf = in[10 * Ntot + idx];
  const double cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1)] - in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] - in[10 * Ntot + idx + (-2)]));
  const double cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] - in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] - in[10 * Ntot + idx + (-2 * s1)]));
  const double cf_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[10 * Ntot + idx] + (4.0 / 3.0) * (in[10 * Ntot + idx + (1)] + in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] + in[10 * Ntot + idx + (-2)]));
  const double cf_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[10 * Ntot + idx + (1 + 1 * s1)] - in[10 * Ntot + idx + (1 + -1 * s1)]) - (in[10 * Ntot + idx + (-1 + 1 * s1)] - in[10 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (1 + 2 * s1)] - in[10 * Ntot + idx + (1 + -2 * s1)]) - (in[10 * Ntot + idx + (-1 + 2 * s1)] - in[10 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (2 + 1 * s1)] - in[10 * Ntot + idx + (2 + -1 * s1)]) - (in[10 * Ntot + idx + (-2 + 1 * s1)] - in[10 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[10 * Ntot + idx + (2 + 2 * s1)] - in[10 * Ntot + idx + (2 + -2 * s1)]) - (in[10 * Ntot + idx + (-2 + 2 * s1)] - in[10 * Ntot + idx + (-2 + -2 * s1)])));
  const double cf_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[10 * Ntot + idx] + (4.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] + in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] + in[10 * Ntot + idx + (-2 * s1)]));
  const double cf_dupD0 = p.invdxx0 * (uw0[0] * in[10 * Ntot + idx + (-3)] + uw0[1] * in[10 * Ntot + idx + (-2)] + uw0[2] * in[10 * Ntot + idx + (-1)] + uw0[3] * in[10 * Ntot + idx] + uw0[4] * in[10 * Ntot + idx + (1)] + uw0[5] * in[10 * Ntot + idx + (2)] + uw0[6] * in[10 * Ntot + idx + (3)]);
  const double cf_dupD1 = p.invdxx1 * (uw1[0] * in[10 * Ntot + idx + (-3 * s1)] + uw1[1] * in[10 * Ntot + idx + (-2 * s1)] + uw1[2] * in[10 * Ntot + idx + (-1 * s1)] + uw1[3] * in[10 * Ntot + idx] + uw1[4] * in[10 * Ntot + idx + (1 * s1)] + uw1[5] * in[10 * Ntot + idx + (2 * s1)] + uw1[6] * in[10 * Ntot + idx + (3 * s1)]);
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double hDD00 = in[11 * Ntot + idx];
  const double hDD01 = in[12 * Ntot + idx];
  const double hDD02 = in[13 * Ntot + idx];
  const double hDD11 = in[14 * Ntot + idx];
  const double hDD12 = in[15 * Ntot + idx];
  const double hDD22 = in[16 * Ntot + idx];
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  const double hDD_dupD000 = p.invdxx0 * (uw0[0] * in[11 * Ntot + idx + (-3)] + uw0[1] * in[11 * Ntot + idx + (-2)] + uw0[2] * in[11 * Ntot + idx + (-1)] + uw0[3] * in[11 * Ntot + idx] + uw0[4] * in[11 * Ntot + idx + (1)] + uw0[5] * in[11 * Ntot + idx + (2)] + uw0[6] * in[11 * Ntot + idx + (3)]);
  const double hDD_dupD001 = p.invdxx1 * (uw1[0] * in[11 * Ntot + idx + (-3 * s1)] + uw1[1] * in[11 * Ntot + idx + (-2 * s1)] + uw1[2] * in[11 * Ntot + idx + (-1 * s1)] + uw1[3] * in[11 * Ntot + idx] + uw1[4] * in[11 * Ntot + idx + (1 * s1)] + uw1[5] * in[11 * Ntot + idx + (2 * s1)] + uw1[6] * in[11 * Ntot + idx + (3 * s1)]);
  const double hDD_dupD010 = p.invdxx0 * (uw0[0] * in[12 * Ntot + idx + (-3)] + uw0[1] * in[12 * Ntot + idx + (-2)] + uw0[2] * in[12 * Ntot + idx + (-1)] + uw0[3] * in[12 * Ntot + idx] + uw0[4] * in[12 * Ntot + idx + (1)] + uw0[5] * in[12 * Ntot + idx + (2)] + uw0[6] * in[12 * Ntot + idx + (3)]);
  const double hDD_dupD011 = p.invdxx1 * (uw1[0] * in[12 * Ntot + idx + (-3 * s1)] + uw1[1] * in[12 * Ntot + idx + (-2 * s1)] + uw1[2] * in[12 * Ntot + idx + (-1 * s1)] + uw1[3] * in[12 * Ntot + idx] + uw1[4] * in[12 * Ntot + idx + (1 * s1)] + uw1[5] * in[12 * Ntot + idx + (2 * s1)] + uw1[6] * in[12 * Ntot + idx + (3 * s1)]);
  const double hDD_dupD020 = p.invdxx0 * (uw0[0] * in[13 * Ntot + idx + (-3)] + uw0[1] * in[13 * Ntot + idx + (-2)] + uw0[2] * in[13 * Ntot + idx + (-1)] + uw0[3] * in[13 * Ntot + idx] + uw0[4] * in[13 * Ntot + idx + (1)] + uw0[5] * in[13 * Ntot + idx + (2)] + uw0[6] * in[13 * Ntot + idx + (3)]);
  const double hDD_dupD021 = p.invdxx1 * (uw1[0] * in[13 * Ntot + idx + (-3 * s1)] + uw1[1] * in[13 * Ntot + idx + (-2 * s1)] + uw1[2] * in[13 * Ntot + idx + (-1 * s1)] + uw1[3] * in[13 * Ntot + idx] + uw1[4] * in[13 * Ntot + idx + (1 * s1)] + uw1[5] * in[13 * Ntot + idx + (2 * s1)] + uw1[6] * in[13 * Ntot + idx + (3 * s1)]);
  const double hDD_dupD110 = p.invdxx0 * (uw0[0] * in[14 * Ntot + idx + (-3)] + uw0[1] * in[14 * Ntot + idx + (-2)] + uw0[2] * in[14 * Ntot + idx + (-1)] + uw0[3] * in[14 * Ntot + idx] + uw0[4] * in[14 * Ntot + idx + (1)] + uw0[5] * in[14 * Ntot + idx + (2)] + uw0[6] * in[14 * Ntot + idx + (3)]);
  const double hDD_dupD111 = p.invdxx1 * (uw1[0] * in[14 * Ntot + idx + (-3 * s1)] + uw1[1] * in[14 * Ntot + idx + (-2 * s1)] + uw1[2] * in[14 * Ntot + idx + (-1 * s1)] + uw1[3] * in[14 * Ntot + idx] + uw1[4] * in[14 * Ntot + idx + (1 * s1)] + uw1[5] * in[14 * Ntot + idx + (2 * s1)] + uw1[6] * in[14 * Ntot + idx + (3 * s1)]);
  const double hDD_dupD120 = p.invdxx0 * (uw0[0] * in[15 * Ntot + idx + (-3)] + uw0[1] * in[15 * Ntot + idx + (-2)] + uw0[2] * in[15 * Ntot + idx + (-1)] + uw0[3] * in[15 * Ntot + idx] + uw0[4] * in[15 * Ntot + idx + (1)] + uw0[5] * in[15 * Ntot + idx + (2)] + uw0[6] * in[15 * Ntot + idx + (3)]);
  const double hDD_dupD121 = p.invdxx1 * (uw1[0] * in[15 * Ntot + idx + (-3 * s1)] + uw1[1] * in[15 * Ntot + idx + (-2 * s1)] + uw1[2] * in[15 * Ntot + idx + (-1 * s1)] + uw1[3] * in[15 * Ntot + idx] + uw1[4] * in[15 * Ntot + idx + (1 * s1)] + uw1[5] * in[15 * Ntot + idx + (2 * s1)] + uw1[6] * in[15 * Ntot + idx + (3 * s1)]);
  const double hDD_dupD220 = p.invdxx0 * (uw0[0] * in[16 * Ntot + idx + (-3)] + uw0[1] * in[16 * Ntot + idx + (-2)] + uw0[2] * in[16 * Ntot + idx + (-1)] + uw0[3] * in[16 * Ntot + idx] + uw0[4] * in[16 * Ntot + idx + (1)] + uw0[5] * in[16 * Ntot + idx + (2)] + uw0[6] * in[16 * Ntot + idx + (3)]);
  const double hDD_dupD221 = p.invdxx1 * (uw1[0] * in[16 * Ntot + idx + (-3 * s1)] + uw1[1] * in[16 * Ntot + idx + (-2 * s1)] + uw1[2] * in[16 * Ntot + idx + (-1 * s1)] + uw1[3] * in[16 * Ntot + idx] + uw1[4] * in[16 * Ntot + idx + (1 * s1)] + uw1[5] * in[16 * Ntot + idx + (2 * s1)] + uw1[6] * in[16 * Ntot + idx + (3 * s1)]);
  const double trK = in[20 * Ntot + idx];
  const double trK_dupD0 = p.invdxx0 * (uw0[0] * in[20 * Ntot + idx + (-3)] + uw0[1] * in[20 * Ntot + idx + (-2)] + uw0[2] * in[20 * Ntot + idx + (-1)] + uw0[3] * in[20 * Ntot + idx] + uw0[4] * in[20 * Ntot + idx + (1)] + uw0[5] * in[20 * Ntot + idx + (2)] + uw0[6] * in[20 * Ntot + idx + (3)]);
  const double trK_dupD1 = p.invdxx1 * (uw1[0] * in[20 * Ntot + idx + (-3 * s1)] + uw1[1] * in[20 * Ntot + idx + (-2 * s1)] + uw1[2] * in[20 * Ntot + idx + (-1 * s1)] + uw1[3] * in[20 * Ntot + idx] + uw1[4] * in[20 * Ntot + idx + (1 * s1)] + uw1[5] * in[20 * Ntot + idx + (2 * s1)] + uw1[6] * in[20 * Ntot + idx + (3 * s1)]);
  const double vetU0 = in[21 * Ntot + idx];
  const double vetU1 = in[22 * Ntot + idx];
  const double vetU2 = in[23 * Ntot + idx];
  const double vetU_dD00 = p.invdxx0 * ((2.0 / 3.0) * (in[21 * Ntot + idx + (1)] - in[21 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2)] - in[21 * Ntot + idx + (-2)]));
  const double vetU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (in[21 * Ntot + idx + (1 * s1)] - in[21 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[21 * Ntot + idx + (2 * s1)] - in[21 * Ntot + idx + (-2 * s1)]));
  const double vetU_dD10 = p.invdxx0 * ((2.0 / 3.0) * (in[22 * Ntot + idx + (1)] - in[22 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2)] - in[22 * Ntot + idx + (-2)]));
  const double vetU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (in[22 * Ntot + idx + (1 * s1)] - in[22 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[22 * Ntot + idx + (2 * s1)] - in[22 * Ntot + idx + (-2 * s1)]));
  const double vetU_dD20 = p.invdxx0 * ((2.0 / 3.0) * (in[23 * Ntot + idx + (1)] - in[23 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2)] - in[23 * Ntot + idx + (-2)]));
  const double vetU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (in[23 * Ntot + idx + (1 * s1)] - in[23 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[23 * Ntot + idx + (2 * s1)] - in[23 * Ntot + idx + (-2 * s1)]));
  const double g2t0 = (cf*cf);
  const double g2t1 = (f0_of_xx0*f0_of_xx0);
  const double g2t2 = (f1_of_xx1*f1_of_xx1);
  const double g2t3 = g2t1*g2t2;
  const double g2t4 = 2.0*f0_of_xx0;
  const double g2t5 = g2t2*g2t4;
  const double g2t6 = g2t5*hDD22 + g2t5;
  const double g2t7 = g2t3*hDD_dD220 + g2t6;
  const double g2t8 = -g2t7;
  const double g2t9 = g2t3*hDD22;
  const double g2t10 = g2t3 + g2t9;
  const double g2t11 = g2t1*(hDD01*hDD01);
  const double g2t12 = hDD00 + 1.0;
  const double g2t13 = g2t1*hDD11;
  const double g2t14 = g2t1 + g2t13;
  const double g2t15 = g2t3*(hDD02*hDD02);
  const double g2t16 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g2t17 = g2t16*g2t2*(hDD12*hDD12);
  const double g2t18 = -g2t10*g2t11 + g2t10*g2t12*g2t14 - g2t12*g2t17 - g2t14*g2t15 + 2.0*g2t16*g2t2*hDD01*hDD02*hDD12;
  const double g2t19 = (1.0 / g2t18);
  const double g2t20 = g2t10*g2t14 - g2t17;
  const double g2t21 = g2t19*g2t20;
  const double g2t22 = (Rational_1_2)*g2t21;
  const double g2t23 = f1_of_xx1*g2t1;
  const double g2t24 = 2.0*g2t23;
  const double g2t25 = f1_of_xx1__D1*g2t24;
  const double g2t26 = g2t25*hDD22 + g2t25;
  const double g2t27 = g2t26 + g2t3*hDD_dD221;
  const double g2t28 = -g2t27;
  const double g2t29 = f0_of_xx0*hDD01;
  const double g2t30 = (f0_of_xx0*f0_of_xx0*f0_of_xx0)*hDD12;
  const double g2t31 = -g2t10*g2t29 + g2t2*g2t30*hDD02;
  const double g2t32 = (Rational_1_2)*g2t19;
  const double g2t33 = g2t31*g2t32;
  const double g2t34 = g2t22*g2t8 + g2t28*g2t33;
  const double g2t35 = (1.0 / cf);
  const double g2t36 = (Rational_1_2)*g2t35;
  const double g2t37 = cf_dD0*g2t36;
  const double g2t38 = g2t10*g2t12 - g2t15;
  const double g2t39 = g2t19*g2t38;
  const double g2t40 = (Rational_1_2)*g2t39;
  const double g2t41 = g2t28*g2t40 + g2t33*g2t8;
  const double g2t42 = cf_dD1*g2t36;
  const double g2t43 = 2.0*alpha;
  const double g2t44 = alpha_dD0*g2t34 + alpha_dD1*g2t41;
  const double g2t45 = RbarDD22*alpha - g2t43*(g2t34*g2t37 + g2t41*g2t42) + g2t44;
  const double g2t46 = -g2t11 + g2t12*g2t14;
  const double g2t47 = g2t19*g2t46;
  const double g2t48 = (cf_dD1*cf_dD1);
  const double g2t49 = g2t4*hDD11 + g2t4;
  const double g2t50 = g2t1*hDD_dD110 + g2t49;
  const double g2t51 = 2.0*f0_of_xx0*hDD_dD011 - g2t50;
  const double g2t52 = f1_of_xx1*hDD02;
  const double g2t53 = f0_of_xx0*g2t52;
  const double g2t54 = f1_of_xx1*g2t30*hDD01 - g2t14*g2t53;
  const double g2t55 = f1_of_xx1__D1*g2t1;
  const double g2t56 = g2t55*hDD12;
  const double g2t57 = g2t32*(g2t24*hDD_dD121 + 2.0*g2t56);
  const double g2t58 = g2t1*hDD_dD111;
  const double g2t59 = g2t22*g2t51 + g2t33*g2t58 + g2t54*g2t57;
  const double g2t60 = g2t23*hDD12;
  const double g2t61 = g2t1*g2t52*hDD01 - g2t12*g2t60;
  const double g2t62 = g2t33*g2t51 + g2t40*g2t58 + g2t57*g2t61;
  const double g2t63 = (1.0 / g2t0);
  const double g2t64 = alpha*g2t63;
  const double g2t65 = cf_dD1*g2t35;
  const double g2t66 = alpha_dD1*g2t65;
  const double g2t67 = alpha_dD0*g2t59 + alpha_dD1*g2t62 - alpha_dDD11;
  const double g2t68 = RbarDD11*alpha - g2t43*(g2t36*(-cf_dDD11 + g2t35*g2t48) + g2t37*g2t59 + g2t42*g2t62) + g2t48*g2t64 - 2.0*g2t66 + g2t67;
  const double g2t69 = (cf_dD0*cf_dD0);
  const double g2t70 = (Rational_1_2)*hDD_dD000;
  const double g2t71 = f1_of_xx1*g2t4;
  const double g2t72 = g2t32*(2.0*g2t52 + g2t71*hDD_dD020);
  const double g2t73 = 2.0*hDD01;
  const double g2t74 = g2t4*hDD_dD010 + g2t73 - hDD_dD001;
  const double g2t75 = g2t21*g2t70 + g2t33*g2t74 + g2t54*g2t72;
  const double g2t76 = g2t19*g2t31;
  const double g2t77 = g2t40*g2t74 + g2t61*g2t72 + g2t70*g2t76;
  const double g2t78 = cf_dD0*g2t35;
  const double g2t79 = alpha_dD0*g2t78;
  const double g2t80 = alpha_dD0*g2t75 + alpha_dD1*g2t77 - alpha_dDD00;
  const double g2t81 = RbarDD00*alpha - g2t43*(g2t36*(-cf_dDD00 + g2t35*g2t69) + g2t37*g2t75 + g2t42*g2t77) + g2t64*g2t69 - 2.0*g2t79 + g2t80;
  const double g2t82 = f0_of_xx0*f1_of_xx1__D1;
  const double g2t83 = g2t82*hDD02;
  const double g2t84 = f0_of_xx0*f1_of_xx1;
  const double g2t85 = g2t71*hDD12;
  const double g2t86 = g2t23*hDD_dD120 + g2t85;
  const double g2t87 = g2t32*(g2t83 + g2t84*hDD_dD021 + g2t86);
  const double g2t88 = g2t22*hDD_dD001 + g2t33*g2t50 + g2t54*g2t87;
  const double g2t89 = g2t33*hDD_dD001 + g2t40*g2t50 + g2t61*g2t87;
  const double g2t90 = g2t43*(g2t36*(cf_dD0*cf_dD1*g2t35 - cf_dDD01) + g2t37*g2t88 + g2t42*g2t89);
  const double g2t91 = alpha_dD0*g2t65;
  const double g2t92 = alpha_dD1*g2t78;
  const double g2t93 = alpha_dD0*g2t88;
  const double g2t94 = alpha_dD1*g2t89;
  const double g2t95 = -alpha_dDD01 + g2t93 + g2t94;
  const double g2t96 = -f0_of_xx0*f1_of_xx1*hDD_dD021 - f0_of_xx0*f1_of_xx1__D1*hDD02 + g2t86;
  const double g2t97 = -g2t96;
  const double g2t98 = g2t27*g2t32;
  const double g2t99 = g2t22*g2t97 + g2t54*g2t98;
  const double g2t100 = g2t33*g2t97 + g2t61*g2t98;
  const double g2t101 = alpha_dD0*g2t99 + alpha_dD1*g2t100;
  const double g2t102 = RbarDD12*alpha + g2t101 - g2t43*(g2t100*g2t42 + g2t37*g2t99);
  const double g2t103 = 2.0*g2t19;
  const double g2t104 = g2t103*g2t61;
  const double g2t105 = g2t32*g2t7;
  const double g2t106 = g2t105*g2t54 + g2t33*g2t96;
  const double g2t107 = g2t105*g2t61 + g2t40*g2t96;
  const double g2t108 = alpha_dD0*g2t106 + alpha_dD1*g2t107;
  const double g2t109 = RbarDD02*alpha + g2t108 - g2t43*(g2t106*g2t37 + g2t107*g2t42);
  const double g2t110 = g2t103*g2t54;
  const double g2t111 = g2t102*g2t104 + g2t109*g2t110 + g2t21*g2t81 + g2t39*g2t68 + g2t45*g2t47 + 2.0*g2t76*(RbarDD01*alpha + cf_dD0*cf_dD1*g2t64 - g2t90 - g2t91 - g2t92 + g2t95);
  const double g2t112 = 2.0*vetU_dD00;
  const double g2t113 = (1.0 / f0_of_xx0);
  const double g2t114 = g2t113*vetU_dD11;
  const double g2t115 = g2t113*vetU0;
  const double g2t116 = (1.0 / f1_of_xx1);
  const double g2t117 = g2t113*vetU1;
  const double g2t118 = f1_of_xx1__D1*g2t116*g2t117;
  const double g2t119 = g2t114 + 2.0*g2t115 + g2t118 + vetU_dD00;
  const double g2t120 = (Rational_2_3)*g2t119;
  const double g2t121 = alpha*trK;
  const double g2t122 = aDD00*g2t21;
  const double g2t123 = aDD01*f0_of_xx0;
  const double g2t124 = g2t123*g2t76;
  const double g2t125 = aDD02*f1_of_xx1;
  const double g2t126 = f0_of_xx0*g2t125;
  const double g2t127 = g2t19*g2t54;
  const double g2t128 = g2t126*g2t127;
  const double g2t129 = aDD00*g2t43;
  const double g2t130 = (1.0 / g2t1);
  const double g2t131 = g2t113*vetU_dD10 - g2t130*vetU1;
  const double g2t132 = aDD01*g2t4;
  const double g2t133 = aDD00*g2t19;
  const double g2t134 = g2t19*g2t61;
  const double g2t135 = alpha*g2t132;
  const double g2t136 = g2t113*g2t116;
  const double g2t137 = g2t116*g2t130;
  const double g2t138 = g2t136*vetU_dD20 - g2t137*vetU2;
  const double g2t139 = g2t138*g2t4;
  const double g2t140 = g2t123*g2t19;
  const double g2t141 = g2t125*g2t4;
  const double g2t142 = alpha*g2t141;
  const double g2t143 = (Rational_1_3)*g2t111;
  const double g2t144 = aDD11*g2t1;
  const double g2t145 = aDD12*g2t23;
  const double g2t146 = g2t123*g2t21 + g2t127*g2t145 + g2t144*g2t76;
  const double g2t147 = (1.0 / g2t2);
  const double g2t148 = -f1_of_xx1__D1*g2t113*g2t147*vetU2 + g2t136*vetU_dD21;
  const double g2t149 = g2t144*g2t39;
  const double g2t150 = g2t134*g2t145;
  const double g2t151 = g2t124 + g2t149 + g2t150;
  const double g2t152 = g2t134*g2t144 + g2t140*g2t54 + g2t145*g2t47;
  const double g2t153 = aDD22*g2t3;
  const double g2t154 = g2t126*g2t21 + g2t127*g2t153 + g2t145*g2t76;
  const double g2t155 = g2t126*g2t76 + g2t134*g2t153 + g2t145*g2t39;
  const double g2t156 = g2t153*g2t47;
  const double g2t157 = g2t128 + g2t150 + g2t156;
  const double g2t158 = aDD11*g2t4;
  const double g2t159 = (Rational_1_3)*g2t1;
  const double g2t160 = f0_of_xx0*vetU1;
  const double g2t161 = (Rational_2_3)*g2t1;
  const double g2t162 = g2t119*g2t161;
  const double g2t163 = g2t144*g2t43;
  const double g2t164 = aDD12*g2t24;
  const double g2t165 = g2t145*g2t43;
  const double g2t166 = f1_of_xx1*hDD12;
  const double g2t167 = g2t84*vetU_dD11;
  const double g2t168 = g2t153*g2t43;
  const double g2t169 = g2t130*g2t147;
  const double g2t170 = alpha*(g2t122 + g2t127*g2t141 + g2t132*g2t76 + g2t134*g2t164 + g2t149 + g2t156) - g2t119;
  const double g2t171 = f0_of_xx0*g2t73;
  const double g2t172 = (Rational_2_3)*g2t170;
  const double g2t173 = (1.0 / (g2t18*g2t18));
  const double g2t174 = aDD00*g2t173;
  const double g2t175 = (g2t31*g2t31);
  const double g2t176 = g2t144*g2t173;
  const double g2t177 = (g2t54*g2t54);
  const double g2t178 = g2t153*g2t173;
  const double g2t179 = g2t132*g2t173;
  const double g2t180 = g2t179*g2t31;
  const double g2t181 = g2t141*g2t173;
  const double g2t182 = g2t181*g2t54;
  const double g2t183 = g2t31*g2t54;
  const double g2t184 = g2t164*g2t173;
  const double g2t185 = (g2t61*g2t61);
  const double g2t186 = g2t31*g2t61;
  const double g2t187 = g2t38*g2t61;
  const double g2t188 = g2t0*g2t76;
  const double g2t189 = g2t174*g2t20;
  const double g2t190 = g2t123*g2t173;
  const double g2t191 = g2t190*g2t20;
  const double g2t192 = g2t176*g2t31;
  const double g2t193 = g2t126*g2t173;
  const double g2t194 = g2t193*g2t20;
  const double g2t195 = g2t38*g2t54;
  const double g2t196 = g2t145*g2t173;
  const double g2t197 = g2t54*g2t61;
  const double g2t198 = g2t31*g2t46;
  const double g2t199 = g2t178*g2t46;
  double a_aDD00 = lam[0 * Ntot + idx] * (g2t112 - g2t120 + g2t121);
  double a_aDD_dupD000 = lam[0 * Ntot + idx] * (vetU0);
  double a_aDD_dupD001 = lam[0 * Ntot + idx] * (g2t117);
  double a_g2t0 = lam[0 * Ntot + idx] * (-g2t111*((Rational_1_3)*hDD00 + Rational_1_3) + g2t81);
  double a_g2t111 = lam[0 * Ntot + idx] * (g2t0*(-Rational_1_3*hDD00 + Rational_m1_3));
  double a_g2t112 = lam[0 * Ntot + idx] * (aDD00);
  double a_g2t117 = lam[0 * Ntot + idx] * (aDD_dupD001);
  double a_g2t120 = lam[0 * Ntot + idx] * (-aDD00);
  double a_g2t121 = lam[0 * Ntot + idx] * (aDD00);
  double a_g2t122 = lam[0 * Ntot + idx] * (-g2t129);
  double a_g2t123 = lam[0 * Ntot + idx] * (-g2t135*g2t39);
  double a_g2t124 = lam[0 * Ntot + idx] * (-g2t129);
  double a_g2t125 = lam[0 * Ntot + idx] * (g2t139);
  double a_g2t126 = lam[0 * Ntot + idx] * (-g2t134*g2t135 - g2t142*g2t47);
  double a_g2t128 = lam[0 * Ntot + idx] * (-g2t129);
  double a_g2t129 = lam[0 * Ntot + idx] * (-g2t122 - g2t124 - g2t128);
  double a_g2t131 = lam[0 * Ntot + idx] * (g2t132);
  double a_g2t132 = lam[0 * Ntot + idx] * (g2t131);
  double a_g2t133 = lam[0 * Ntot + idx] * (-g2t135*g2t31 - g2t142*g2t54);
  double a_g2t134 = lam[0 * Ntot + idx] * (-g2t126*g2t135);
  double a_g2t135 = lam[0 * Ntot + idx] * (-g2t123*g2t39 - g2t126*g2t134 - g2t133*g2t31);
  double a_g2t139 = lam[0 * Ntot + idx] * (g2t125);
  double a_g2t140 = lam[0 * Ntot + idx] * (-g2t142*g2t61);
  double a_g2t142 = lam[0 * Ntot + idx] * (-g2t126*g2t47 - g2t133*g2t54 - g2t140*g2t61);
  double a_g2t31 = lam[0 * Ntot + idx] * (-g2t133*g2t135);
  double a_g2t39 = lam[0 * Ntot + idx] * (-g2t123*g2t135);
  double a_g2t47 = lam[0 * Ntot + idx] * (-g2t126*g2t142);
  double a_g2t54 = lam[0 * Ntot + idx] * (-g2t133*g2t142);
  double a_g2t61 = lam[0 * Ntot + idx] * (-g2t140*g2t142);
  double a_g2t81 = lam[0 * Ntot + idx] * (g2t0);
  double a_hDD00 = lam[0 * Ntot + idx] * (-Rational_1_3*g2t0*g2t111);
  double a_vetU0 = lam[0 * Ntot + idx] * (aDD_dupD000);
  double a_RbarDD01 = lam[1 * Ntot + idx] * (alpha*g2t0*g2t113);
  a_aDD00 += lam[1 * Ntot + idx] * (g2t113*vetU_dD01);
  double a_aDD01 = lam[1 * Ntot + idx] * (g2t113*(vetU0 + vetU_dD11));
  double a_aDD_dupD010 = lam[1 * Ntot + idx] * (f0_of_xx0*g2t113*vetU0);
  double a_aDD_dupD011 = lam[1 * Ntot + idx] * (g2t113*vetU1);
  double a_alpha = lam[1 * Ntot + idx] * (g2t0*g2t113*(RbarDD01 + cf_dD0*cf_dD1*g2t63));
  double a_alpha_dDD01 = lam[1 * Ntot + idx] * (-g2t0*g2t113);
  double a_cf_dD0 = lam[1 * Ntot + idx] * (alpha*cf_dD1*g2t0*g2t113*g2t63);
  double a_cf_dD1 = lam[1 * Ntot + idx] * (alpha*cf_dD0*g2t0*g2t113*g2t63);
  double a_f0_of_xx0 = lam[1 * Ntot + idx] * (aDD_dupD010*g2t113*vetU0);
  a_g2t0 += lam[1 * Ntot + idx] * (g2t113*(RbarDD01*alpha + alpha*cf_dD0*cf_dD1*g2t63 - alpha_dDD01 - g2t143*g2t29 - g2t90 - g2t91 - g2t92 + g2t93 + g2t94));
  double a_g2t113 = lam[1 * Ntot + idx] * (aDD00*vetU_dD01 + aDD01*vetU_dD11 + aDD_dupD011*vetU1 + g2t0*(RbarDD01*alpha + alpha*cf_dD0*cf_dD1*g2t63 - alpha_dDD01 - g2t143*g2t29 - g2t90 - g2t91 - g2t92 + g2t93 + g2t94) - g2t120*g2t123 + g2t121*g2t123 + g2t123*vetU_dD00 + g2t126*g2t148 - g2t129*g2t146 + g2t131*g2t144 - g2t135*g2t151 + g2t138*g2t145 - g2t142*g2t152 + vetU0*(aDD01 + aDD_dupD010*f0_of_xx0));
  a_g2t120 += lam[1 * Ntot + idx] * (-g2t113*g2t123);
  a_g2t121 += lam[1 * Ntot + idx] * (g2t113*g2t123);
  a_g2t123 += lam[1 * Ntot + idx] * (g2t113*(-g2t120 + g2t121 + vetU_dD00));
  a_g2t126 += lam[1 * Ntot + idx] * (g2t113*g2t148);
  a_g2t129 += lam[1 * Ntot + idx] * (-g2t113*g2t146);
  a_g2t131 += lam[1 * Ntot + idx] * (g2t113*g2t144);
  a_g2t135 += lam[1 * Ntot + idx] * (-g2t113*g2t151);
  double a_g2t138 = lam[1 * Ntot + idx] * (g2t113*g2t145);
  a_g2t142 += lam[1 * Ntot + idx] * (-g2t113*g2t152);
  double a_g2t143 = lam[1 * Ntot + idx] * (-g2t0*g2t113*g2t29);
  double a_g2t144 = lam[1 * Ntot + idx] * (g2t113*g2t131);
  double a_g2t145 = lam[1 * Ntot + idx] * (g2t113*g2t138);
  double a_g2t146 = lam[1 * Ntot + idx] * (-g2t113*g2t129);
  double a_g2t148 = lam[1 * Ntot + idx] * (g2t113*g2t126);
  double a_g2t151 = lam[1 * Ntot + idx] * (-g2t113*g2t135);
  double a_g2t152 = lam[1 * Ntot + idx] * (-g2t113*g2t142);
  double a_g2t29 = lam[1 * Ntot + idx] * (-g2t0*g2t113*g2t143);
  double a_g2t63 = lam[1 * Ntot + idx] * (alpha*cf_dD0*cf_dD1*g2t0*g2t113);
  double a_g2t90 = lam[1 * Ntot + idx] * (-g2t0*g2t113);
  double a_g2t91 = lam[1 * Ntot + idx] * (-g2t0*g2t113);
  double a_g2t92 = lam[1 * Ntot + idx] * (-g2t0*g2t113);
  double a_g2t93 = lam[1 * Ntot + idx] * (g2t0*g2t113);
  double a_g2t94 = lam[1 * Ntot + idx] * (g2t0*g2t113);
  a_vetU0 += lam[1 * Ntot + idx] * (g2t113*(aDD01 + aDD_dupD010*f0_of_xx0));
  double a_vetU1 = lam[1 * Ntot + idx] * (aDD_dupD011*g2t113);
  double a_vetU_dD00 = lam[1 * Ntot + idx] * (g2t113*g2t123);
  double a_vetU_dD01 = lam[1 * Ntot + idx] * (aDD00*g2t113);
  double a_vetU_dD11 = lam[1 * Ntot + idx] * (aDD01*g2t113);
  double a_aDD02 = lam[2 * Ntot + idx] * (g2t117*g2t136*g2t82);
  double a_aDD_dupD020 = lam[2 * Ntot + idx] * (g2t136*g2t84*vetU0);
  double a_aDD_dupD021 = lam[2 * Ntot + idx] * (g2t117*g2t136*g2t84);
  a_g2t0 += lam[2 * Ntot + idx] * (g2t136*(g2t109 - g2t143*g2t53));
  double a_g2t109 = lam[2 * Ntot + idx] * (g2t0*g2t136);
  a_g2t117 += lam[2 * Ntot + idx] * (g2t136*(aDD02*g2t82 + aDD_dupD021*g2t84));
  a_g2t120 += lam[2 * Ntot + idx] * (-g2t126*g2t136);
  a_g2t121 += lam[2 * Ntot + idx] * (g2t126*g2t136);
  a_g2t125 += lam[2 * Ntot + idx] * (g2t136*vetU0);
  a_g2t126 += lam[2 * Ntot + idx] * (g2t136*(-g2t120 + g2t121 + vetU_dD00));
  a_g2t129 += lam[2 * Ntot + idx] * (-g2t136*g2t154);
  a_g2t131 += lam[2 * Ntot + idx] * (g2t136*g2t145);
  a_g2t135 += lam[2 * Ntot + idx] * (-g2t136*g2t155);
  double a_g2t136 = lam[2 * Ntot + idx] * (g2t0*(g2t109 - g2t143*g2t53) + g2t117*(aDD02*g2t82 + aDD_dupD021*g2t84) - g2t120*g2t126 + g2t121*g2t126 + g2t126*vetU_dD00 - g2t129*g2t154 + g2t131*g2t145 - g2t135*g2t155 + g2t138*g2t153 - g2t142*g2t157 + vetU0*(aDD_dupD020*g2t84 + g2t125));
  a_g2t138 += lam[2 * Ntot + idx] * (g2t136*g2t153);
  a_g2t142 += lam[2 * Ntot + idx] * (-g2t136*g2t157);
  a_g2t143 += lam[2 * Ntot + idx] * (-g2t0*g2t136*g2t53);
  a_g2t145 += lam[2 * Ntot + idx] * (g2t131*g2t136);
  double a_g2t153 = lam[2 * Ntot + idx] * (g2t136*g2t138);
  double a_g2t154 = lam[2 * Ntot + idx] * (-g2t129*g2t136);
  double a_g2t155 = lam[2 * Ntot + idx] * (-g2t135*g2t136);
  double a_g2t157 = lam[2 * Ntot + idx] * (-g2t136*g2t142);
  double a_g2t53 = lam[2 * Ntot + idx] * (-g2t0*g2t136*g2t143);
  double a_g2t82 = lam[2 * Ntot + idx] * (aDD02*g2t117*g2t136);
  double a_g2t84 = lam[2 * Ntot + idx] * (g2t136*(aDD_dupD020*vetU0 + aDD_dupD021*g2t117));
  a_vetU0 += lam[2 * Ntot + idx] * (g2t136*(aDD_dupD020*g2t84 + g2t125));
  a_vetU_dD00 += lam[2 * Ntot + idx] * (g2t126*g2t136);
  double a_aDD11 = lam[3 * Ntot + idx] * (-g2t130*g2t162);
  double a_aDD_dupD110 = lam[3 * Ntot + idx] * (g2t1*g2t130*vetU0);
  double a_aDD_dupD111 = lam[3 * Ntot + idx] * (g2t130*g2t160);
  a_g2t0 += lam[3 * Ntot + idx] * (g2t130*(-g2t111*((Rational_1_3)*g2t13 + g2t159) + g2t68));
  double a_g2t1 = lam[3 * Ntot + idx] * (aDD_dupD110*g2t130*vetU0);
  a_g2t111 += lam[3 * Ntot + idx] * (g2t0*g2t130*(-Rational_1_3*g2t13 - g2t159));
  a_g2t121 += lam[3 * Ntot + idx] * (g2t130*g2t144);
  double a_g2t13 = lam[3 * Ntot + idx] * (-Rational_1_3*g2t0*g2t111*g2t130);
  double a_g2t130 = lam[3 * Ntot + idx] * (-aDD11*g2t162 + aDD_dupD111*g2t160 + g2t0*(-g2t111*((Rational_1_3)*g2t13 + g2t159) + g2t68) + g2t121*g2t144 + g2t132*vetU_dD01 - g2t135*g2t146 + g2t148*g2t164 - g2t151*g2t163 - g2t152*g2t165 + g2t158*vetU_dD11 + vetU0*(aDD_dupD110*g2t1 + g2t158));
  a_g2t132 += lam[3 * Ntot + idx] * (g2t130*vetU_dD01);
  a_g2t135 += lam[3 * Ntot + idx] * (-g2t130*g2t146);
  a_g2t144 += lam[3 * Ntot + idx] * (g2t121*g2t130);
  a_g2t146 += lam[3 * Ntot + idx] * (-g2t130*g2t135);
  a_g2t148 += lam[3 * Ntot + idx] * (g2t130*g2t164);
  a_g2t151 += lam[3 * Ntot + idx] * (-g2t130*g2t163);
  a_g2t152 += lam[3 * Ntot + idx] * (-g2t130*g2t165);
  double a_g2t158 = lam[3 * Ntot + idx] * (g2t130*(vetU0 + vetU_dD11));
  double a_g2t159 = lam[3 * Ntot + idx] * (-g2t0*g2t111*g2t130);
  double a_g2t160 = lam[3 * Ntot + idx] * (aDD_dupD111*g2t130);
  double a_g2t162 = lam[3 * Ntot + idx] * (-aDD11*g2t130);
  double a_g2t163 = lam[3 * Ntot + idx] * (-g2t130*g2t151);
  double a_g2t164 = lam[3 * Ntot + idx] * (g2t130*g2t148);
  double a_g2t165 = lam[3 * Ntot + idx] * (-g2t130*g2t152);
  double a_g2t68 = lam[3 * Ntot + idx] * (g2t0*g2t130);
  a_vetU0 += lam[3 * Ntot + idx] * (g2t130*(aDD_dupD110*g2t1 + g2t158));
  a_vetU_dD01 += lam[3 * Ntot + idx] * (g2t130*g2t132);
  a_vetU_dD11 += lam[3 * Ntot + idx] * (g2t130*g2t158);
  double a_aDD12 = lam[4 * Ntot + idx] * (g2t137*(-f1_of_xx1*g2t162 + g2t117*g2t55 + g2t167 + g2t71*vetU0));
  double a_aDD_dupD120 = lam[4 * Ntot + idx] * (g2t137*g2t23*vetU0);
  double a_aDD_dupD121 = lam[4 * Ntot + idx] * (g2t117*g2t137*g2t23);
  double a_f1_of_xx1 = lam[4 * Ntot + idx] * (-aDD12*g2t137*g2t162);
  a_g2t0 += lam[4 * Ntot + idx] * (g2t137*(g2t102 - g2t111*g2t159*g2t166));
  double a_g2t102 = lam[4 * Ntot + idx] * (g2t0*g2t137);
  a_g2t111 += lam[4 * Ntot + idx] * (-g2t0*g2t137*g2t159*g2t166);
  a_g2t117 += lam[4 * Ntot + idx] * (g2t137*(aDD12*g2t55 + aDD_dupD121*g2t23));
  a_g2t121 += lam[4 * Ntot + idx] * (g2t137*g2t145);
  a_g2t126 += lam[4 * Ntot + idx] * (g2t137*vetU_dD01);
  a_g2t135 += lam[4 * Ntot + idx] * (-g2t137*g2t154);
  double a_g2t137 = lam[4 * Ntot + idx] * (-aDD12*f1_of_xx1*g2t162 + aDD12*g2t167 + g2t0*(g2t102 - g2t111*g2t159*g2t166) + g2t117*(aDD12*g2t55 + aDD_dupD121*g2t23) + g2t121*g2t145 + g2t126*vetU_dD01 - g2t135*g2t154 + g2t148*g2t153 - g2t155*g2t163 - g2t157*g2t165 + vetU0*(aDD12*g2t71 + aDD_dupD120*g2t23));
  a_g2t145 += lam[4 * Ntot + idx] * (g2t121*g2t137);
  a_g2t148 += lam[4 * Ntot + idx] * (g2t137*g2t153);
  a_g2t153 += lam[4 * Ntot + idx] * (g2t137*g2t148);
  a_g2t154 += lam[4 * Ntot + idx] * (-g2t135*g2t137);
  a_g2t155 += lam[4 * Ntot + idx] * (-g2t137*g2t163);
  a_g2t157 += lam[4 * Ntot + idx] * (-g2t137*g2t165);
  a_g2t159 += lam[4 * Ntot + idx] * (-g2t0*g2t111*g2t137*g2t166);
  a_g2t162 += lam[4 * Ntot + idx] * (-aDD12*f1_of_xx1*g2t137);
  a_g2t163 += lam[4 * Ntot + idx] * (-g2t137*g2t155);
  a_g2t165 += lam[4 * Ntot + idx] * (-g2t137*g2t157);
  double a_g2t166 = lam[4 * Ntot + idx] * (-g2t0*g2t111*g2t137*g2t159);
  double a_g2t167 = lam[4 * Ntot + idx] * (aDD12*g2t137);
  double a_g2t23 = lam[4 * Ntot + idx] * (g2t137*(aDD_dupD120*vetU0 + aDD_dupD121*g2t117));
  double a_g2t55 = lam[4 * Ntot + idx] * (aDD12*g2t117*g2t137);
  double a_g2t71 = lam[4 * Ntot + idx] * (aDD12*g2t137*vetU0);
  a_vetU0 += lam[4 * Ntot + idx] * (g2t137*(aDD12*g2t71 + aDD_dupD120*g2t23));
  a_vetU_dD01 += lam[4 * Ntot + idx] * (g2t126*g2t137);
  double a_aDD22 = lam[5 * Ntot + idx] * (g2t169*(alpha*g2t1*g2t2*trK + g2t113*g2t25*vetU1 + g2t5*vetU0));
  double a_aDD_dupD220 = lam[5 * Ntot + idx] * (g2t169*g2t3*vetU0);
  double a_aDD_dupD221 = lam[5 * Ntot + idx] * (g2t113*g2t169*g2t3*vetU1);
  a_alpha += lam[5 * Ntot + idx] * (aDD22*g2t1*g2t169*g2t2*trK);
  a_g2t0 += lam[5 * Ntot + idx] * (g2t169*(-g2t111*((Rational_1_3)*g2t3 + (Rational_1_3)*g2t9) + g2t45));
  a_g2t1 += lam[5 * Ntot + idx] * (aDD22*alpha*g2t169*g2t2*trK);
  a_g2t111 += lam[5 * Ntot + idx] * (g2t0*g2t169*(-Rational_1_3*g2t3 - Rational_1_3*g2t9));
  a_g2t113 += lam[5 * Ntot + idx] * (g2t169*vetU1*(aDD22*g2t25 + aDD_dupD221*g2t3));
  a_g2t120 += lam[5 * Ntot + idx] * (-g2t153*g2t169);
  a_g2t142 += lam[5 * Ntot + idx] * (-g2t154*g2t169);
  a_g2t153 += lam[5 * Ntot + idx] * (-g2t120*g2t169);
  a_g2t154 += lam[5 * Ntot + idx] * (-g2t142*g2t169);
  a_g2t155 += lam[5 * Ntot + idx] * (-g2t165*g2t169);
  a_g2t157 += lam[5 * Ntot + idx] * (-g2t168*g2t169);
  a_g2t165 += lam[5 * Ntot + idx] * (-g2t155*g2t169);
  double a_g2t168 = lam[5 * Ntot + idx] * (-g2t157*g2t169);
  double a_g2t169 = lam[5 * Ntot + idx] * (aDD22*alpha*g2t1*g2t2*trK + g2t0*(-g2t111*((Rational_1_3)*g2t3 + (Rational_1_3)*g2t9) + g2t45) + g2t113*vetU1*(aDD22*g2t25 + aDD_dupD221*g2t3) - g2t120*g2t153 - g2t142*g2t154 - g2t155*g2t165 - g2t157*g2t168 + vetU0*(aDD22*g2t5 + aDD_dupD220*g2t3));
  double a_g2t2 = lam[5 * Ntot + idx] * (aDD22*alpha*g2t1*g2t169*trK);
  double a_g2t25 = lam[5 * Ntot + idx] * (aDD22*g2t113*g2t169*vetU1);
  double a_g2t3 = lam[5 * Ntot + idx] * (g2t169*(aDD_dupD220*vetU0 + aDD_dupD221*g2t113*vetU1 - Rational_1_3*g2t0*g2t111));
  double a_g2t45 = lam[5 * Ntot + idx] * (g2t0*g2t169);
  double a_g2t5 = lam[5 * Ntot + idx] * (aDD22*g2t169*vetU0);
  double a_g2t9 = lam[5 * Ntot + idx] * (-Rational_1_3*g2t0*g2t111*g2t169);
  double a_trK = lam[5 * Ntot + idx] * (aDD22*alpha*g2t1*g2t169*g2t2);
  a_vetU0 += lam[5 * Ntot + idx] * (g2t169*(aDD22*g2t5 + aDD_dupD220*g2t3));
  a_vetU1 += lam[5 * Ntot + idx] * (g2t113*g2t169*(aDD22*g2t25 + aDD_dupD221*g2t3));
  double a_cf = lam[10 * Ntot + idx] * (2.0*cf_dupD0*g2t36*vetU0 + 2.0*cf_dupD1*g2t117*g2t36 - Rational_1_3*g2t114 - Rational_2_3*g2t115 - Rational_1_3*g2t118 + (Rational_1_3)*g2t121 - Rational_1_3*vetU_dD00);
  double a_cf_dupD0 = lam[10 * Ntot + idx] * (2.0*cf*g2t36*vetU0);
  double a_cf_dupD1 = lam[10 * Ntot + idx] * (2.0*cf*g2t117*g2t36);
  double a_g2t114 = lam[10 * Ntot + idx] * (-Rational_1_3*cf);
  double a_g2t115 = lam[10 * Ntot + idx] * (-Rational_2_3*cf);
  a_g2t117 += lam[10 * Ntot + idx] * (2.0*cf*cf_dupD1*g2t36);
  double a_g2t118 = lam[10 * Ntot + idx] * (-Rational_1_3*cf);
  a_g2t121 += lam[10 * Ntot + idx] * ((Rational_1_3)*cf);
  double a_g2t36 = lam[10 * Ntot + idx] * (-2.0*cf*(-cf_dupD0*vetU0 - cf_dupD1*g2t117));
  a_vetU0 += lam[10 * Ntot + idx] * (2.0*cf*cf_dupD0*g2t36);
  a_vetU_dD00 += lam[10 * Ntot + idx] * (-Rational_1_3*cf);
  a_g2t112 += lam[11 * Ntot + idx] * (g2t12);
  a_g2t117 += lam[11 * Ntot + idx] * (hDD_dupD001);
  double a_g2t12 = lam[11 * Ntot + idx] * (g2t112);
  a_g2t129 += lam[11 * Ntot + idx] * (-1.0);
  a_g2t131 += lam[11 * Ntot + idx] * (g2t171);
  a_g2t139 += lam[11 * Ntot + idx] * (g2t52);
  double a_g2t170 = lam[11 * Ntot + idx] * ((Rational_2_3)*hDD00 + Rational_2_3);
  double a_g2t171 = lam[11 * Ntot + idx] * (g2t131);
  double a_g2t52 = lam[11 * Ntot + idx] * (g2t139);
  a_hDD00 += lam[11 * Ntot + idx] * ((Rational_2_3)*g2t170);
  double a_hDD_dupD000 = lam[11 * Ntot + idx] * (vetU0);
  double a_hDD_dupD001 = lam[11 * Ntot + idx] * (g2t117);
  a_vetU0 += lam[11 * Ntot + idx] * (hDD_dupD000);
  a_f0_of_xx0 += lam[12 * Ntot + idx] * (g2t113*hDD_dupD010*vetU0);
  a_g2t113 += lam[12 * Ntot + idx] * (g2t12*vetU_dD01 + g2t131*g2t14 - g2t135 + g2t138*g2t60 + g2t148*g2t53 + g2t172*g2t29 + g2t29*vetU_dD00 + hDD01*vetU_dD11 + hDD_dupD011*vetU1 + vetU0*(f0_of_xx0*hDD_dupD010 + hDD01));
  a_g2t12 += lam[12 * Ntot + idx] * (g2t113*vetU_dD01);
  a_g2t131 += lam[12 * Ntot + idx] * (g2t113*g2t14);
  a_g2t135 += lam[12 * Ntot + idx] * (-g2t113);
  a_g2t138 += lam[12 * Ntot + idx] * (g2t113*g2t60);
  double a_g2t14 = lam[12 * Ntot + idx] * (g2t113*g2t131);
  a_g2t148 += lam[12 * Ntot + idx] * (g2t113*g2t53);
  double a_g2t172 = lam[12 * Ntot + idx] * (g2t113*g2t29);
  a_g2t29 += lam[12 * Ntot + idx] * (g2t113*(g2t172 + vetU_dD00));
  a_g2t53 += lam[12 * Ntot + idx] * (g2t113*g2t148);
  double a_g2t60 = lam[12 * Ntot + idx] * (g2t113*g2t138);
  double a_hDD01 = lam[12 * Ntot + idx] * (g2t113*(vetU0 + vetU_dD11));
  double a_hDD_dupD010 = lam[12 * Ntot + idx] * (f0_of_xx0*g2t113*vetU0);
  double a_hDD_dupD011 = lam[12 * Ntot + idx] * (g2t113*vetU1);
  a_vetU0 += lam[12 * Ntot + idx] * (g2t113*(f0_of_xx0*hDD_dupD010 + hDD01));
  a_vetU1 += lam[12 * Ntot + idx] * (g2t113*hDD_dupD011);
  a_vetU_dD00 += lam[12 * Ntot + idx] * (g2t113*g2t29);
  a_vetU_dD01 += lam[12 * Ntot + idx] * (g2t113*g2t12);
  a_vetU_dD11 += lam[12 * Ntot + idx] * (g2t113*hDD01);
  double a_g2t10 = lam[13 * Ntot + idx] * (g2t136*g2t138);
  a_g2t117 += lam[13 * Ntot + idx] * (g2t136*(g2t83 + g2t84*hDD_dupD021));
  a_g2t131 += lam[13 * Ntot + idx] * (g2t136*g2t60);
  a_g2t136 += lam[13 * Ntot + idx] * (g2t10*g2t138 + g2t117*(g2t83 + g2t84*hDD_dupD021) + g2t131*g2t60 - g2t142 + g2t172*g2t53 + g2t53*vetU_dD00 + vetU0*(g2t52 + g2t84*hDD_dupD020));
  a_g2t138 += lam[13 * Ntot + idx] * (g2t10*g2t136);
  a_g2t142 += lam[13 * Ntot + idx] * (-g2t136);
  a_g2t172 += lam[13 * Ntot + idx] * (g2t136*g2t53);
  a_g2t52 += lam[13 * Ntot + idx] * (g2t136*vetU0);
  a_g2t53 += lam[13 * Ntot + idx] * (g2t136*(g2t172 + vetU_dD00));
  a_g2t60 += lam[13 * Ntot + idx] * (g2t131*g2t136);
  double a_g2t83 = lam[13 * Ntot + idx] * (g2t117*g2t136);
  a_g2t84 += lam[13 * Ntot + idx] * (g2t136*(g2t117*hDD_dupD021 + hDD_dupD020*vetU0));
  double a_hDD_dupD020 = lam[13 * Ntot + idx] * (g2t136*g2t84*vetU0);
  double a_hDD_dupD021 = lam[13 * Ntot + idx] * (g2t117*g2t136*g2t84);
  a_vetU0 += lam[13 * Ntot + idx] * (g2t136*(g2t52 + g2t84*hDD_dupD020));
  a_vetU_dD00 += lam[13 * Ntot + idx] * (g2t136*g2t53);
  a_g2t1 += lam[14 * Ntot + idx] * (g2t130*hDD_dupD110*vetU0);
  a_g2t114 += lam[14 * Ntot + idx] * (2.0*g2t130*g2t14);
  a_g2t13 += lam[14 * Ntot + idx] * ((Rational_2_3)*g2t130*g2t170);
  a_g2t130 += lam[14 * Ntot + idx] * (2.0*g2t114*g2t14 + 2.0*g2t148*g2t60 + g2t160*hDD_dupD111 - g2t163 + g2t170*((Rational_2_3)*g2t13 + g2t161) + g2t171*vetU_dD01 + vetU0*(g2t1*hDD_dupD110 + g2t49));
  a_g2t14 += lam[14 * Ntot + idx] * (2.0*g2t114*g2t130);
  a_g2t148 += lam[14 * Ntot + idx] * (2.0*g2t130*g2t60);
  a_g2t160 += lam[14 * Ntot + idx] * (g2t130*hDD_dupD111);
  double a_g2t161 = lam[14 * Ntot + idx] * (g2t130*g2t170);
  a_g2t163 += lam[14 * Ntot + idx] * (-g2t130);
  a_g2t170 += lam[14 * Ntot + idx] * (g2t130*((Rational_2_3)*g2t13 + g2t161));
  a_g2t171 += lam[14 * Ntot + idx] * (g2t130*vetU_dD01);
  double a_g2t49 = lam[14 * Ntot + idx] * (g2t130*vetU0);
  a_g2t60 += lam[14 * Ntot + idx] * (2.0*g2t130*g2t148);
  double a_hDD_dupD110 = lam[14 * Ntot + idx] * (g2t1*g2t130*vetU0);
  double a_hDD_dupD111 = lam[14 * Ntot + idx] * (g2t130*g2t160);
  a_vetU0 += lam[14 * Ntot + idx] * (g2t130*(g2t1*hDD_dupD110 + g2t49));
  a_vetU_dD01 += lam[14 * Ntot + idx] * (g2t130*g2t171);
  a_g2t10 += lam[15 * Ntot + idx] * (g2t137*g2t148);
  a_g2t117 += lam[15 * Ntot + idx] * (g2t137*(g2t23*hDD_dupD121 + g2t56));
  a_g2t137 += lam[15 * Ntot + idx] * (g2t10*g2t148 + g2t117*(g2t23*hDD_dupD121 + g2t56) + g2t161*g2t166*g2t170 - g2t165 + g2t167*hDD12 + g2t53*vetU_dD01 + vetU0*(g2t23*hDD_dupD120 + g2t85));
  a_g2t148 += lam[15 * Ntot + idx] * (g2t10*g2t137);
  a_g2t161 += lam[15 * Ntot + idx] * (g2t137*g2t166*g2t170);
  a_g2t165 += lam[15 * Ntot + idx] * (-g2t137);
  a_g2t166 += lam[15 * Ntot + idx] * (g2t137*g2t161*g2t170);
  a_g2t167 += lam[15 * Ntot + idx] * (g2t137*hDD12);
  a_g2t170 += lam[15 * Ntot + idx] * (g2t137*g2t161*g2t166);
  a_g2t23 += lam[15 * Ntot + idx] * (g2t137*(g2t117*hDD_dupD121 + hDD_dupD120*vetU0));
  a_g2t53 += lam[15 * Ntot + idx] * (g2t137*vetU_dD01);
  double a_g2t56 = lam[15 * Ntot + idx] * (g2t117*g2t137);
  double a_g2t85 = lam[15 * Ntot + idx] * (g2t137*vetU0);
  double a_hDD12 = lam[15 * Ntot + idx] * (g2t137*g2t167);
  double a_hDD_dupD120 = lam[15 * Ntot + idx] * (g2t137*g2t23*vetU0);
  double a_hDD_dupD121 = lam[15 * Ntot + idx] * (g2t117*g2t137*g2t23);
  a_vetU0 += lam[15 * Ntot + idx] * (g2t137*(g2t23*hDD_dupD120 + g2t85));
  a_vetU_dD01 += lam[15 * Ntot + idx] * (g2t137*g2t53);
  a_g2t117 += lam[16 * Ntot + idx] * (g2t169*(g2t26 + g2t3*hDD_dupD221));
  a_g2t168 += lam[16 * Ntot + idx] * (-g2t169);
  a_g2t169 += lam[16 * Ntot + idx] * (g2t117*(g2t26 + g2t3*hDD_dupD221) - g2t168 + g2t170*((Rational_2_3)*g2t3 + (Rational_2_3)*g2t9) + vetU0*(g2t3*hDD_dupD220 + g2t6));
  a_g2t170 += lam[16 * Ntot + idx] * (g2t169*((Rational_2_3)*g2t3 + (Rational_2_3)*g2t9));
  double a_g2t26 = lam[16 * Ntot + idx] * (g2t117*g2t169);
  a_g2t3 += lam[16 * Ntot + idx] * (g2t169*(g2t117*hDD_dupD221 + (Rational_2_3)*g2t170 + hDD_dupD220*vetU0));
  double a_g2t6 = lam[16 * Ntot + idx] * (g2t169*vetU0);
  a_g2t9 += lam[16 * Ntot + idx] * ((Rational_2_3)*g2t169*g2t170);
  double a_hDD_dupD220 = lam[16 * Ntot + idx] * (g2t169*g2t3*vetU0);
  double a_hDD_dupD221 = lam[16 * Ntot + idx] * (g2t117*g2t169*g2t3);
  a_vetU0 += lam[16 * Ntot + idx] * (g2t169*(g2t3*hDD_dupD220 + g2t6));
  a_aDD00 += lam[20 * Ntot + idx] * (alpha*(g2t174*(g2t20*g2t20) + g2t175*g2t176 + g2t177*g2t178 + g2t180*g2t20 + g2t182*g2t20 + g2t183*g2t184));
  a_alpha += lam[20 * Ntot + idx] * (aDD00*(g2t174*(g2t20*g2t20) + g2t175*g2t176 + g2t177*g2t178 + g2t180*g2t20 + g2t182*g2t20 + g2t183*g2t184) + g2t144*(g2t174*g2t175 + g2t176*(g2t38*g2t38) + g2t178*g2t185 + g2t180*g2t38 + g2t181*g2t186 + g2t184*g2t187) + g2t153*(g2t174*g2t177 + g2t176*g2t185 + g2t178*(g2t46*g2t46) + g2t179*g2t197 + g2t182*g2t46 + g2t184*g2t46*g2t61) + (Rational_1_3)*(trK*trK));
  a_g2t0 += lam[20 * Ntot + idx] * (g2t101*g2t104 + g2t108*g2t110 - g2t21*(-g2t79 - g2t80) - g2t39*(-g2t66 - g2t67) + g2t44*g2t47);
  double a_g2t101 = lam[20 * Ntot + idx] * (g2t0*g2t104);
  double a_g2t104 = lam[20 * Ntot + idx] * (g2t0*g2t101);
  double a_g2t108 = lam[20 * Ntot + idx] * (g2t0*g2t110);
  double a_g2t110 = lam[20 * Ntot + idx] * (g2t0*g2t108);
  a_g2t117 += lam[20 * Ntot + idx] * (trK_dupD1);
  a_g2t135 += lam[20 * Ntot + idx] * (g2t175*g2t190 + g2t178*g2t197 + g2t183*g2t193 + g2t186*g2t196 + g2t189*g2t31 + g2t191*g2t38 + g2t192*g2t38 + g2t194*g2t61 + g2t195*g2t196);
  a_g2t142 += lam[20 * Ntot + idx] * (g2t177*g2t193 + g2t183*g2t190 + g2t189*g2t54 + g2t191*g2t61 + g2t192*g2t61 + g2t194*g2t46 + g2t196*g2t197 + g2t196*g2t198 + g2t199*g2t54);
  a_g2t144 += lam[20 * Ntot + idx] * (alpha*(g2t174*g2t175 + g2t176*(g2t38*g2t38) + g2t178*g2t185 + g2t180*g2t38 + g2t181*g2t186 + g2t184*g2t187));
  a_g2t153 += lam[20 * Ntot + idx] * (alpha*(g2t174*g2t177 + g2t176*g2t185 + g2t178*(g2t46*g2t46) + g2t179*g2t197 + g2t182*g2t46 + g2t184*g2t46*g2t61));
  a_g2t165 += lam[20 * Ntot + idx] * (g2t174*g2t183 + g2t176*g2t187 + g2t185*g2t196 + g2t186*g2t190 + g2t190*g2t195 + g2t193*g2t197 + g2t193*g2t198 + g2t196*g2t38*g2t46 + g2t199*g2t61);
  double a_g2t174 = lam[20 * Ntot + idx] * (aDD00*alpha*(g2t20*g2t20) + alpha*g2t144*g2t175 + alpha*g2t153*g2t177 + g2t165*g2t183);
  double a_g2t175 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t176 + alpha*g2t144*g2t174 + g2t135*g2t190);
  double a_g2t176 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t175 + alpha*g2t144*(g2t38*g2t38) + alpha*g2t153*g2t185 + g2t165*g2t187);
  double a_g2t177 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t178 + alpha*g2t153*g2t174 + g2t142*g2t193);
  double a_g2t178 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t177 + alpha*g2t144*g2t185 + alpha*g2t153*(g2t46*g2t46) + g2t135*g2t197);
  double a_g2t179 = lam[20 * Ntot + idx] * (alpha*g2t153*g2t197);
  double a_g2t180 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t20 + alpha*g2t144*g2t38);
  double a_g2t181 = lam[20 * Ntot + idx] * (alpha*g2t144*g2t186);
  double a_g2t182 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t20 + alpha*g2t153*g2t46);
  double a_g2t183 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t184 + g2t135*g2t193 + g2t142*g2t190 + g2t165*g2t174);
  double a_g2t184 = lam[20 * Ntot + idx] * (aDD00*alpha*g2t183 + alpha*g2t144*g2t187 + alpha*g2t153*g2t46*g2t61);
  double a_g2t185 = lam[20 * Ntot + idx] * (alpha*g2t144*g2t178 + alpha*g2t153*g2t176 + g2t165*g2t196);
  double a_g2t186 = lam[20 * Ntot + idx] * (alpha*g2t144*g2t181 + g2t135*g2t196 + g2t165*g2t190);
  double a_g2t187 = lam[20 * Ntot + idx] * (alpha*g2t144*g2t184 + g2t165*g2t176);
  double a_g2t188 = lam[20 * Ntot + idx] * (g2t91 + g2t92 + 2.0*g2t95);
  double a_g2t189 = lam[20 * Ntot + idx] * (g2t135*g2t31 + g2t142*g2t54);
  double a_g2t190 = lam[20 * Ntot + idx] * (g2t135*g2t175 + g2t142*g2t183 + g2t165*(g2t186 + g2t195));
  double a_g2t191 = lam[20 * Ntot + idx] * (g2t135*g2t38 + g2t142*g2t61);
  double a_g2t192 = lam[20 * Ntot + idx] * (g2t135*g2t38 + g2t142*g2t61);
  double a_g2t193 = lam[20 * Ntot + idx] * (g2t135*g2t183 + g2t142*g2t177 + g2t165*(g2t197 + g2t198));
  double a_g2t194 = lam[20 * Ntot + idx] * (g2t135*g2t61 + g2t142*g2t46);
  double a_g2t195 = lam[20 * Ntot + idx] * (g2t135*g2t196 + g2t165*g2t190);
  double a_g2t196 = lam[20 * Ntot + idx] * (g2t135*(g2t186 + g2t195) + g2t142*(g2t197 + g2t198) + g2t165*(g2t185 + g2t38*g2t46));
  double a_g2t197 = lam[20 * Ntot + idx] * (alpha*g2t153*g2t179 + g2t135*g2t178 + g2t142*g2t196 + g2t165*g2t193);
  double a_g2t198 = lam[20 * Ntot + idx] * (g2t142*g2t196 + g2t165*g2t193);
  double a_g2t199 = lam[20 * Ntot + idx] * (g2t142*g2t54 + g2t165*g2t61);
  double a_g2t20 = lam[20 * Ntot + idx] * (aDD00*alpha*(2.0*g2t174*g2t20 + g2t180 + g2t182));
  double a_g2t21 = lam[20 * Ntot + idx] * (-g2t0*(-g2t79 - g2t80));
  a_g2t31 += lam[20 * Ntot + idx] * (g2t135*g2t189);
  double a_g2t38 = lam[20 * Ntot + idx] * (alpha*g2t144*(2.0*g2t176*g2t38 + g2t180) + g2t135*(g2t191 + g2t192) + g2t165*g2t196*g2t46);
  a_g2t39 += lam[20 * Ntot + idx] * (-g2t0*(-g2t66 - g2t67));
  double a_g2t44 = lam[20 * Ntot + idx] * (g2t0*g2t47);
  double a_g2t46 = lam[20 * Ntot + idx] * (alpha*g2t153*(2.0*g2t178*g2t46 + g2t182 + g2t184*g2t61) + g2t142*g2t194 + g2t165*g2t196*g2t38);
  a_g2t47 += lam[20 * Ntot + idx] * (g2t0*g2t44);
  a_g2t54 += lam[20 * Ntot + idx] * (g2t142*(g2t189 + g2t199));
  a_g2t61 += lam[20 * Ntot + idx] * (alpha*g2t153*g2t184*g2t46 + g2t135*g2t194 + g2t142*(g2t191 + g2t192) + g2t165*g2t199);
  double a_g2t66 = lam[20 * Ntot + idx] * (g2t0*g2t39);
  double a_g2t67 = lam[20 * Ntot + idx] * (g2t0*g2t39);
  double a_g2t79 = lam[20 * Ntot + idx] * (g2t0*g2t21);
  double a_g2t80 = lam[20 * Ntot + idx] * (g2t0*g2t21);
  a_g2t91 += lam[20 * Ntot + idx] * (g2t188);
  a_g2t92 += lam[20 * Ntot + idx] * (g2t188);
  double a_g2t95 = lam[20 * Ntot + idx] * (2.0*g2t188);
  a_trK += lam[20 * Ntot + idx] * ((Rational_2_3)*alpha*trK);
  double a_trK_dupD0 = lam[20 * Ntot + idx] * (vetU0);
  double a_trK_dupD1 = lam[20 * Ntot + idx] * (g2t117);
  a_vetU0 += lam[20 * Ntot + idx] * (trK_dupD0);
  a_g2t178 += a_g2t199 * (g2t46);
  a_g2t46 += a_g2t199 * (g2t178);
  a_g2t31 += a_g2t198 * (g2t46);
  a_g2t46 += a_g2t198 * (g2t31);
  a_g2t54 += a_g2t197 * (g2t61);
  a_g2t61 += a_g2t197 * (g2t54);
  a_g2t145 += a_g2t196 * (g2t173);
  double a_g2t173 = a_g2t196 * (g2t145);
  a_g2t38 += a_g2t195 * (g2t54);
  a_g2t54 += a_g2t195 * (g2t38);
  a_g2t193 += a_g2t194 * (g2t20);
  a_g2t20 += a_g2t194 * (g2t193);
  a_g2t126 += a_g2t193 * (g2t173);
  a_g2t173 += a_g2t193 * (g2t126);
  a_g2t176 += a_g2t192 * (g2t31);
  a_g2t31 += a_g2t192 * (g2t176);
  a_g2t190 += a_g2t191 * (g2t20);
  a_g2t20 += a_g2t191 * (g2t190);
  a_g2t123 += a_g2t190 * (g2t173);
  a_g2t173 += a_g2t190 * (g2t123);
  a_g2t174 += a_g2t189 * (g2t20);
  a_g2t20 += a_g2t189 * (g2t174);
  a_g2t0 += a_g2t188 * (g2t76);
  double a_g2t76 = a_g2t188 * (g2t0);
  a_g2t38 += a_g2t187 * (g2t61);
  a_g2t61 += a_g2t187 * (g2t38);
  a_g2t31 += a_g2t186 * (g2t61);
  a_g2t61 += a_g2t186 * (g2t31);
  a_g2t61 += a_g2t185 * (2.0*g2t61);
  a_g2t164 += a_g2t184 * (g2t173);
  a_g2t173 += a_g2t184 * (g2t164);
  a_g2t31 += a_g2t183 * (g2t54);
  a_g2t54 += a_g2t183 * (g2t31);
  a_g2t181 += a_g2t182 * (g2t54);
  a_g2t54 += a_g2t182 * (g2t181);
  double a_g2t141 = a_g2t181 * (g2t173);
  a_g2t173 += a_g2t181 * (g2t141);
  a_g2t179 += a_g2t180 * (g2t31);
  a_g2t31 += a_g2t180 * (g2t179);
  a_g2t132 += a_g2t179 * (g2t173);
  a_g2t173 += a_g2t179 * (g2t132);
  a_g2t153 += a_g2t178 * (g2t173);
  a_g2t173 += a_g2t178 * (g2t153);
  a_g2t54 += a_g2t177 * (2.0*g2t54);
  a_g2t144 += a_g2t176 * (g2t173);
  a_g2t173 += a_g2t176 * (g2t144);
  a_g2t31 += a_g2t175 * (2.0*g2t31);
  a_aDD00 += a_g2t174 * (g2t173);
  a_g2t173 += a_g2t174 * (aDD00);
  double a_g2t18 = a_g2t173 * (-2.0/(g2t18*g2t18*g2t18));
  a_g2t170 += a_g2t172 * (Rational_2_3);
  a_f0_of_xx0 += a_g2t171 * (g2t73);
  double a_g2t73 = a_g2t171 * (f0_of_xx0);
  a_alpha += a_g2t170 * (g2t122 + g2t127*g2t141 + g2t132*g2t76 + g2t134*g2t164 + g2t149 + g2t156);
  double a_g2t119 = a_g2t170 * (-1.0);
  a_g2t122 += a_g2t170 * (alpha);
  double a_g2t127 = a_g2t170 * (alpha*g2t141);
  a_g2t132 += a_g2t170 * (alpha*g2t76);
  a_g2t134 += a_g2t170 * (alpha*g2t164);
  a_g2t141 += a_g2t170 * (alpha*g2t127);
  double a_g2t149 = a_g2t170 * (alpha);
  double a_g2t156 = a_g2t170 * (alpha);
  a_g2t164 += a_g2t170 * (alpha*g2t134);
  a_g2t76 += a_g2t170 * (alpha*g2t132);
  a_g2t130 += a_g2t169 * (g2t147);
  double a_g2t147 = a_g2t169 * (g2t130);
  a_g2t153 += a_g2t168 * (g2t43);
  double a_g2t43 = a_g2t168 * (g2t153);
  a_g2t84 += a_g2t167 * (vetU_dD11);
  a_vetU_dD11 += a_g2t167 * (g2t84);
  a_f1_of_xx1 += a_g2t166 * (hDD12);
  a_hDD12 += a_g2t166 * (f1_of_xx1);
  a_g2t145 += a_g2t165 * (g2t43);
  a_g2t43 += a_g2t165 * (g2t145);
  a_aDD12 += a_g2t164 * (g2t24);
  double a_g2t24 = a_g2t164 * (aDD12);
  a_g2t144 += a_g2t163 * (g2t43);
  a_g2t43 += a_g2t163 * (g2t144);
  a_g2t119 += a_g2t162 * (g2t161);
  a_g2t161 += a_g2t162 * (g2t119);
  a_g2t1 += a_g2t161 * (Rational_2_3);
  a_f0_of_xx0 += a_g2t160 * (vetU1);
  a_vetU1 += a_g2t160 * (f0_of_xx0);
  a_g2t1 += a_g2t159 * (Rational_1_3);
  a_aDD11 += a_g2t158 * (g2t4);
  double a_g2t4 = a_g2t158 * (aDD11);
  a_g2t128 += a_g2t157 * (1.0);
  double a_g2t150 = a_g2t157 * (1.0);
  a_g2t156 += a_g2t157 * (1.0);
  a_g2t153 += a_g2t156 * (g2t47);
  a_g2t47 += a_g2t156 * (g2t153);
  a_g2t126 += a_g2t155 * (g2t76);
  a_g2t134 += a_g2t155 * (g2t153);
  a_g2t145 += a_g2t155 * (g2t39);
  a_g2t153 += a_g2t155 * (g2t134);
  a_g2t39 += a_g2t155 * (g2t145);
  a_g2t76 += a_g2t155 * (g2t126);
  a_g2t126 += a_g2t154 * (g2t21);
  a_g2t127 += a_g2t154 * (g2t153);
  a_g2t145 += a_g2t154 * (g2t76);
  a_g2t153 += a_g2t154 * (g2t127);
  a_g2t21 += a_g2t154 * (g2t126);
  a_g2t76 += a_g2t154 * (g2t145);
  a_aDD22 += a_g2t153 * (g2t3);
  a_g2t3 += a_g2t153 * (aDD22);
  a_g2t134 += a_g2t152 * (g2t144);
  a_g2t140 += a_g2t152 * (g2t54);
  a_g2t144 += a_g2t152 * (g2t134);
  a_g2t145 += a_g2t152 * (g2t47);
  a_g2t47 += a_g2t152 * (g2t145);
  a_g2t54 += a_g2t152 * (g2t140);
  a_g2t124 += a_g2t151 * (1.0);
  a_g2t149 += a_g2t151 * (1.0);
  a_g2t150 += a_g2t151 * (1.0);
  a_g2t134 += a_g2t150 * (g2t145);
  a_g2t145 += a_g2t150 * (g2t134);
  a_g2t144 += a_g2t149 * (g2t39);
  a_g2t39 += a_g2t149 * (g2t144);
  double a_f1_of_xx1__D1 = a_g2t148 * (-g2t113*g2t147*vetU2);
  a_g2t113 += a_g2t148 * (-f1_of_xx1__D1*g2t147*vetU2);
  a_g2t136 += a_g2t148 * (vetU_dD21);
  a_g2t147 += a_g2t148 * (-f1_of_xx1__D1*g2t113*vetU2);
  double a_vetU2 = a_g2t148 * (-f1_of_xx1__D1*g2t113*g2t147);
  double a_vetU_dD21 = a_g2t148 * (g2t136);
  a_g2t2 += a_g2t147 * (-1.0/(g2t2*g2t2));
  a_g2t123 += a_g2t146 * (g2t21);
  a_g2t127 += a_g2t146 * (g2t145);
  a_g2t144 += a_g2t146 * (g2t76);
  a_g2t145 += a_g2t146 * (g2t127);
  a_g2t21 += a_g2t146 * (g2t123);
  a_g2t76 += a_g2t146 * (g2t144);
  a_aDD12 += a_g2t145 * (g2t23);
  a_g2t23 += a_g2t145 * (aDD12);
  a_aDD11 += a_g2t144 * (g2t1);
  a_g2t1 += a_g2t144 * (aDD11);
  a_g2t111 += a_g2t143 * (Rational_1_3);
  a_alpha += a_g2t142 * (g2t141);
  a_g2t141 += a_g2t142 * (alpha);
  a_g2t125 += a_g2t141 * (g2t4);
  a_g2t4 += a_g2t141 * (g2t125);
  a_g2t123 += a_g2t140 * (g2t19);
  double a_g2t19 = a_g2t140 * (g2t123);
  a_g2t138 += a_g2t139 * (g2t4);
  a_g2t4 += a_g2t139 * (g2t138);
  a_g2t136 += a_g2t138 * (vetU_dD20);
  a_g2t137 += a_g2t138 * (-vetU2);
  a_vetU2 += a_g2t138 * (-g2t137);
  double a_vetU_dD20 = a_g2t138 * (g2t136);
  double a_g2t116 = a_g2t137 * (g2t130);
  a_g2t130 += a_g2t137 * (g2t116);
  a_g2t113 += a_g2t136 * (g2t116);
  a_g2t116 += a_g2t136 * (g2t113);
  a_alpha += a_g2t135 * (g2t132);
  a_g2t132 += a_g2t135 * (alpha);
  a_g2t19 += a_g2t134 * (g2t61);
  a_g2t61 += a_g2t134 * (g2t19);
  a_aDD00 += a_g2t133 * (g2t19);
  a_g2t19 += a_g2t133 * (aDD00);
  a_aDD01 += a_g2t132 * (g2t4);
  a_g2t4 += a_g2t132 * (aDD01);
  a_g2t113 += a_g2t131 * (vetU_dD10);
  a_g2t130 += a_g2t131 * (-vetU1);
  a_vetU1 += a_g2t131 * (-g2t130);
  double a_vetU_dD10 = a_g2t131 * (g2t113);
  a_g2t1 += a_g2t130 * (-1.0/(g2t1*g2t1));
  a_aDD00 += a_g2t129 * (g2t43);
  a_g2t43 += a_g2t129 * (aDD00);
  a_g2t126 += a_g2t128 * (g2t127);
  a_g2t127 += a_g2t128 * (g2t126);
  a_g2t19 += a_g2t127 * (g2t54);
  a_g2t54 += a_g2t127 * (g2t19);
  a_f0_of_xx0 += a_g2t126 * (g2t125);
  a_g2t125 += a_g2t126 * (f0_of_xx0);
  a_aDD02 += a_g2t125 * (f1_of_xx1);
  a_f1_of_xx1 += a_g2t125 * (aDD02);
  a_g2t123 += a_g2t124 * (g2t76);
  a_g2t76 += a_g2t124 * (g2t123);
  a_aDD01 += a_g2t123 * (f0_of_xx0);
  a_f0_of_xx0 += a_g2t123 * (aDD01);
  a_aDD00 += a_g2t122 * (g2t21);
  a_g2t21 += a_g2t122 * (aDD00);
  a_alpha += a_g2t121 * (trK);
  a_trK += a_g2t121 * (alpha);
  a_g2t119 += a_g2t120 * (Rational_2_3);
  a_g2t114 += a_g2t119 * (1.0);
  a_g2t115 += a_g2t119 * (2.0);
  a_g2t118 += a_g2t119 * (1.0);
  a_vetU_dD00 += a_g2t119 * (1.0);
  a_f1_of_xx1__D1 += a_g2t118 * (g2t116*g2t117);
  a_g2t116 += a_g2t118 * (f1_of_xx1__D1*g2t117);
  a_g2t117 += a_g2t118 * (f1_of_xx1__D1*g2t116);
  a_g2t113 += a_g2t117 * (vetU1);
  a_vetU1 += a_g2t117 * (g2t113);
  a_f1_of_xx1 += a_g2t116 * (-1.0/(f1_of_xx1*f1_of_xx1));
  a_g2t113 += a_g2t115 * (vetU0);
  a_vetU0 += a_g2t115 * (g2t113);
  a_g2t113 += a_g2t114 * (vetU_dD11);
  a_vetU_dD11 += a_g2t114 * (g2t113);
  a_f0_of_xx0 += a_g2t113 * (-1.0/(f0_of_xx0*f0_of_xx0));
  a_vetU_dD00 += a_g2t112 * (2.0);
  a_RbarDD01 += a_g2t111 * (2.0*alpha*g2t76);
  a_alpha += a_g2t111 * (2.0*RbarDD01*g2t76);
  a_cf_dD0 += a_g2t111 * (2.0*cf_dD1*g2t64*g2t76);
  a_cf_dD1 += a_g2t111 * (2.0*cf_dD0*g2t64*g2t76);
  a_g2t102 += a_g2t111 * (g2t104);
  a_g2t104 += a_g2t111 * (g2t102);
  a_g2t109 += a_g2t111 * (g2t110);
  a_g2t110 += a_g2t111 * (g2t109);
  a_g2t21 += a_g2t111 * (g2t81);
  a_g2t39 += a_g2t111 * (g2t68);
  a_g2t45 += a_g2t111 * (g2t47);
  a_g2t47 += a_g2t111 * (g2t45);
  double a_g2t64 = a_g2t111 * (2.0*cf_dD0*cf_dD1*g2t76);
  a_g2t68 += a_g2t111 * (g2t39);
  a_g2t76 += a_g2t111 * (2.0*RbarDD01*alpha + 2.0*cf_dD0*cf_dD1*g2t64 - 2.0*g2t90 - 2.0*g2t91 - 2.0*g2t92 + 2.0*g2t95);
  a_g2t81 += a_g2t111 * (g2t21);
  a_g2t90 += a_g2t111 * (-2.0*g2t76);
  a_g2t91 += a_g2t111 * (-2.0*g2t76);
  a_g2t92 += a_g2t111 * (-2.0*g2t76);
  a_g2t95 += a_g2t111 * (2.0*g2t76);
  double a_g2t103 = a_g2t110 * (g2t54);
  a_g2t54 += a_g2t110 * (g2t103);
  double a_RbarDD02 = a_g2t109 * (alpha);
  a_alpha += a_g2t109 * (RbarDD02);
  double a_g2t106 = a_g2t109 * (-g2t37*g2t43);
  double a_g2t107 = a_g2t109 * (-g2t42*g2t43);
  a_g2t108 += a_g2t109 * (1.0);
  double a_g2t37 = a_g2t109 * (-g2t106*g2t43);
  double a_g2t42 = a_g2t109 * (-g2t107*g2t43);
  a_g2t43 += a_g2t109 * (-g2t106*g2t37 - g2t107*g2t42);
  double a_alpha_dD0 = a_g2t108 * (g2t106);
  double a_alpha_dD1 = a_g2t108 * (g2t107);
  a_g2t106 += a_g2t108 * (alpha_dD0);
  a_g2t107 += a_g2t108 * (alpha_dD1);
  double a_g2t105 = a_g2t107 * (g2t61);
  double a_g2t40 = a_g2t107 * (g2t96);
  a_g2t61 += a_g2t107 * (g2t105);
  double a_g2t96 = a_g2t107 * (g2t40);
  a_g2t105 += a_g2t106 * (g2t54);
  double a_g2t33 = a_g2t106 * (g2t96);
  a_g2t54 += a_g2t106 * (g2t105);
  a_g2t96 += a_g2t106 * (g2t33);
  double a_g2t32 = a_g2t105 * (g2t7);
  double a_g2t7 = a_g2t105 * (g2t32);
  a_g2t103 += a_g2t104 * (g2t61);
  a_g2t61 += a_g2t104 * (g2t103);
  a_g2t19 += a_g2t103 * (2.0);
  double a_RbarDD12 = a_g2t102 * (alpha);
  a_alpha += a_g2t102 * (RbarDD12);
  double a_g2t100 = a_g2t102 * (-g2t42*g2t43);
  a_g2t101 += a_g2t102 * (1.0);
  a_g2t37 += a_g2t102 * (-g2t43*g2t99);
  a_g2t42 += a_g2t102 * (-g2t100*g2t43);
  a_g2t43 += a_g2t102 * (-g2t100*g2t42 - g2t37*g2t99);
  double a_g2t99 = a_g2t102 * (-g2t37*g2t43);
  a_alpha_dD0 += a_g2t101 * (g2t99);
  a_alpha_dD1 += a_g2t101 * (g2t100);
  a_g2t100 += a_g2t101 * (alpha_dD1);
  a_g2t99 += a_g2t101 * (alpha_dD0);
  a_g2t33 += a_g2t100 * (g2t97);
  a_g2t61 += a_g2t100 * (g2t98);
  double a_g2t97 = a_g2t100 * (g2t33);
  double a_g2t98 = a_g2t100 * (g2t61);
  double a_g2t22 = a_g2t99 * (g2t97);
  a_g2t54 += a_g2t99 * (g2t98);
  a_g2t97 += a_g2t99 * (g2t22);
  a_g2t98 += a_g2t99 * (g2t54);
  double a_g2t27 = a_g2t98 * (g2t32);
  a_g2t32 += a_g2t98 * (g2t27);
  a_g2t96 += a_g2t97 * (-1.0);
  a_f0_of_xx0 += a_g2t96 * (-f1_of_xx1*hDD_dD021 - f1_of_xx1__D1*hDD02);
  a_f1_of_xx1 += a_g2t96 * (-f0_of_xx0*hDD_dD021);
  a_f1_of_xx1__D1 += a_g2t96 * (-f0_of_xx0*hDD02);
  double a_g2t86 = a_g2t96 * (1.0);
  double a_hDD02 = a_g2t96 * (-f0_of_xx0*f1_of_xx1__D1);
  double a_hDD_dD021 = a_g2t96 * (-f0_of_xx0*f1_of_xx1);
  a_alpha_dDD01 += a_g2t95 * (-1.0);
  a_g2t93 += a_g2t95 * (1.0);
  a_g2t94 += a_g2t95 * (1.0);
  a_alpha_dD1 += a_g2t94 * (g2t89);
  double a_g2t89 = a_g2t94 * (alpha_dD1);
  a_alpha_dD0 += a_g2t93 * (g2t88);
  double a_g2t88 = a_g2t93 * (alpha_dD0);
  a_alpha_dD1 += a_g2t92 * (g2t78);
  double a_g2t78 = a_g2t92 * (alpha_dD1);
  a_alpha_dD0 += a_g2t91 * (g2t65);
  double a_g2t65 = a_g2t91 * (alpha_dD0);
  a_cf_dD0 += a_g2t90 * (cf_dD1*g2t35*g2t36*g2t43);
  a_cf_dD1 += a_g2t90 * (cf_dD0*g2t35*g2t36*g2t43);
  double a_cf_dDD01 = a_g2t90 * (-g2t36*g2t43);
  double a_g2t35 = a_g2t90 * (cf_dD0*cf_dD1*g2t36*g2t43);
  a_g2t36 += a_g2t90 * (g2t43*(cf_dD0*cf_dD1*g2t35 - cf_dDD01));
  a_g2t37 += a_g2t90 * (g2t43*g2t88);
  a_g2t42 += a_g2t90 * (g2t43*g2t89);
  a_g2t43 += a_g2t90 * (g2t36*(cf_dD0*cf_dD1*g2t35 - cf_dDD01) + g2t37*g2t88 + g2t42*g2t89);
  a_g2t88 += a_g2t90 * (g2t37*g2t43);
  a_g2t89 += a_g2t90 * (g2t42*g2t43);
  a_g2t33 += a_g2t89 * (hDD_dD001);
  a_g2t40 += a_g2t89 * (g2t50);
  double a_g2t50 = a_g2t89 * (g2t40);
  a_g2t61 += a_g2t89 * (g2t87);
  double a_g2t87 = a_g2t89 * (g2t61);
  double a_hDD_dD001 = a_g2t89 * (g2t33);
  a_g2t22 += a_g2t88 * (hDD_dD001);
  a_g2t33 += a_g2t88 * (g2t50);
  a_g2t50 += a_g2t88 * (g2t33);
  a_g2t54 += a_g2t88 * (g2t87);
  a_g2t87 += a_g2t88 * (g2t54);
  a_hDD_dD001 += a_g2t88 * (g2t22);
  a_g2t32 += a_g2t87 * (g2t83 + g2t84*hDD_dD021 + g2t86);
  a_g2t83 += a_g2t87 * (g2t32);
  a_g2t84 += a_g2t87 * (g2t32*hDD_dD021);
  a_g2t86 += a_g2t87 * (g2t32);
  a_hDD_dD021 += a_g2t87 * (g2t32*g2t84);
  a_g2t23 += a_g2t86 * (hDD_dD120);
  a_g2t85 += a_g2t86 * (1.0);
  double a_hDD_dD120 = a_g2t86 * (g2t23);
  a_g2t71 += a_g2t85 * (hDD12);
  a_hDD12 += a_g2t85 * (g2t71);
  a_f0_of_xx0 += a_g2t84 * (f1_of_xx1);
  a_f1_of_xx1 += a_g2t84 * (f0_of_xx0);
  a_g2t82 += a_g2t83 * (hDD02);
  a_hDD02 += a_g2t83 * (g2t82);
  a_f0_of_xx0 += a_g2t82 * (f1_of_xx1__D1);
  a_f1_of_xx1__D1 += a_g2t82 * (f0_of_xx0);
  double a_RbarDD00 = a_g2t81 * (alpha);
  a_alpha += a_g2t81 * (RbarDD00);
  double a_cf_dDD00 = a_g2t81 * (g2t36*g2t43);
  a_g2t35 += a_g2t81 * (-g2t36*g2t43*g2t69);
  a_g2t36 += a_g2t81 * (-g2t43*(-cf_dDD00 + g2t35*g2t69));
  a_g2t37 += a_g2t81 * (-g2t43*g2t75);
  a_g2t42 += a_g2t81 * (-g2t43*g2t77);
  a_g2t43 += a_g2t81 * (-g2t36*(-cf_dDD00 + g2t35*g2t69) - g2t37*g2t75 - g2t42*g2t77);
  a_g2t64 += a_g2t81 * (g2t69);
  double a_g2t69 = a_g2t81 * (-g2t35*g2t36*g2t43 + g2t64);
  double a_g2t75 = a_g2t81 * (-g2t37*g2t43);
  double a_g2t77 = a_g2t81 * (-g2t42*g2t43);
  a_g2t79 += a_g2t81 * (-2.0);
  a_g2t80 += a_g2t81 * (1.0);
  a_alpha_dD0 += a_g2t80 * (g2t75);
  a_alpha_dD1 += a_g2t80 * (g2t77);
  double a_alpha_dDD00 = a_g2t80 * (-1.0);
  a_g2t75 += a_g2t80 * (alpha_dD0);
  a_g2t77 += a_g2t80 * (alpha_dD1);
  a_alpha_dD0 += a_g2t79 * (g2t78);
  a_g2t78 += a_g2t79 * (alpha_dD0);
  a_cf_dD0 += a_g2t78 * (g2t35);
  a_g2t35 += a_g2t78 * (cf_dD0);
  a_g2t40 += a_g2t77 * (g2t74);
  a_g2t61 += a_g2t77 * (g2t72);
  double a_g2t70 = a_g2t77 * (g2t76);
  double a_g2t72 = a_g2t77 * (g2t61);
  double a_g2t74 = a_g2t77 * (g2t40);
  a_g2t76 += a_g2t77 * (g2t70);
  a_g2t19 += a_g2t76 * (g2t31);
  a_g2t31 += a_g2t76 * (g2t19);
  a_g2t21 += a_g2t75 * (g2t70);
  a_g2t33 += a_g2t75 * (g2t74);
  a_g2t54 += a_g2t75 * (g2t72);
  a_g2t70 += a_g2t75 * (g2t21);
  a_g2t72 += a_g2t75 * (g2t54);
  a_g2t74 += a_g2t75 * (g2t33);
  a_g2t4 += a_g2t74 * (hDD_dD010);
  a_g2t73 += a_g2t74 * (1.0);
  a_hDD_dD001 += a_g2t74 * (-1.0);
  double a_hDD_dD010 = a_g2t74 * (g2t4);
  a_hDD01 += a_g2t73 * (2.0);
  a_g2t32 += a_g2t72 * (2.0*g2t52 + g2t71*hDD_dD020);
  a_g2t52 += a_g2t72 * (2.0*g2t32);
  a_g2t71 += a_g2t72 * (g2t32*hDD_dD020);
  double a_hDD_dD020 = a_g2t72 * (g2t32*g2t71);
  a_f1_of_xx1 += a_g2t71 * (g2t4);
  a_g2t4 += a_g2t71 * (f1_of_xx1);
  double a_hDD_dD000 = a_g2t70 * (Rational_1_2);
  a_cf_dD0 += a_g2t69 * (2.0*cf_dD0);
  double a_RbarDD11 = a_g2t68 * (alpha);
  a_alpha += a_g2t68 * (RbarDD11);
  double a_cf_dDD11 = a_g2t68 * (g2t36*g2t43);
  a_g2t35 += a_g2t68 * (-g2t36*g2t43*g2t48);
  a_g2t36 += a_g2t68 * (-g2t43*(-cf_dDD11 + g2t35*g2t48));
  a_g2t37 += a_g2t68 * (-g2t43*g2t59);
  a_g2t42 += a_g2t68 * (-g2t43*g2t62);
  a_g2t43 += a_g2t68 * (-g2t36*(-cf_dDD11 + g2t35*g2t48) - g2t37*g2t59 - g2t42*g2t62);
  double a_g2t48 = a_g2t68 * (-g2t35*g2t36*g2t43 + g2t64);
  double a_g2t59 = a_g2t68 * (-g2t37*g2t43);
  double a_g2t62 = a_g2t68 * (-g2t42*g2t43);
  a_g2t64 += a_g2t68 * (g2t48);
  a_g2t66 += a_g2t68 * (-2.0);
  a_g2t67 += a_g2t68 * (1.0);
  a_alpha_dD0 += a_g2t67 * (g2t59);
  a_alpha_dD1 += a_g2t67 * (g2t62);
  double a_alpha_dDD11 = a_g2t67 * (-1.0);
  a_g2t59 += a_g2t67 * (alpha_dD0);
  a_g2t62 += a_g2t67 * (alpha_dD1);
  a_alpha_dD1 += a_g2t66 * (g2t65);
  a_g2t65 += a_g2t66 * (alpha_dD1);
  a_cf_dD1 += a_g2t65 * (g2t35);
  a_g2t35 += a_g2t65 * (cf_dD1);
  a_alpha += a_g2t64 * (g2t63);
  a_g2t63 += a_g2t64 * (alpha);
  a_g2t0 += a_g2t63 * (-1.0/(g2t0*g2t0));
  a_g2t33 += a_g2t62 * (g2t51);
  a_g2t40 += a_g2t62 * (g2t58);
  double a_g2t51 = a_g2t62 * (g2t33);
  double a_g2t57 = a_g2t62 * (g2t61);
  double a_g2t58 = a_g2t62 * (g2t40);
  a_g2t61 += a_g2t62 * (g2t57);
  a_g2t1 += a_g2t61 * (g2t52*hDD01);
  a_g2t12 += a_g2t61 * (-g2t60);
  a_g2t52 += a_g2t61 * (g2t1*hDD01);
  a_g2t60 += a_g2t61 * (-g2t12);
  a_hDD01 += a_g2t61 * (g2t1*g2t52);
  a_g2t23 += a_g2t60 * (hDD12);
  a_hDD12 += a_g2t60 * (g2t23);
  a_g2t22 += a_g2t59 * (g2t51);
  a_g2t33 += a_g2t59 * (g2t58);
  a_g2t51 += a_g2t59 * (g2t22);
  a_g2t54 += a_g2t59 * (g2t57);
  a_g2t57 += a_g2t59 * (g2t54);
  a_g2t58 += a_g2t59 * (g2t33);
  a_g2t1 += a_g2t58 * (hDD_dD111);
  double a_hDD_dD111 = a_g2t58 * (g2t1);
  a_g2t24 += a_g2t57 * (g2t32*hDD_dD121);
  a_g2t32 += a_g2t57 * (g2t24*hDD_dD121 + 2.0*g2t56);
  a_g2t56 += a_g2t57 * (2.0*g2t32);
  double a_hDD_dD121 = a_g2t57 * (g2t24*g2t32);
  a_g2t55 += a_g2t56 * (hDD12);
  a_hDD12 += a_g2t56 * (g2t55);
  a_f1_of_xx1__D1 += a_g2t55 * (g2t1);
  a_g2t1 += a_g2t55 * (f1_of_xx1__D1);
  a_f1_of_xx1 += a_g2t54 * (g2t30*hDD01);
  a_g2t14 += a_g2t54 * (-g2t53);
  double a_g2t30 = a_g2t54 * (f1_of_xx1*hDD01);
  a_g2t53 += a_g2t54 * (-g2t14);
  a_hDD01 += a_g2t54 * (f1_of_xx1*g2t30);
  a_f0_of_xx0 += a_g2t53 * (g2t52);
  a_g2t52 += a_g2t53 * (f0_of_xx0);
  a_f1_of_xx1 += a_g2t52 * (hDD02);
  a_hDD02 += a_g2t52 * (f1_of_xx1);
  a_f0_of_xx0 += a_g2t51 * (2.0*hDD_dD011);
  a_g2t50 += a_g2t51 * (-1.0);
  double a_hDD_dD011 = a_g2t51 * (2.0*f0_of_xx0);
  a_g2t1 += a_g2t50 * (hDD_dD110);
  a_g2t49 += a_g2t50 * (1.0);
  double a_hDD_dD110 = a_g2t50 * (g2t1);
  a_g2t4 += a_g2t49 * (hDD11 + 1.0);
  double a_hDD11 = a_g2t49 * (g2t4);
  a_cf_dD1 += a_g2t48 * (2.0*cf_dD1);
  a_g2t19 += a_g2t47 * (g2t46);
  a_g2t46 += a_g2t47 * (g2t19);
  double a_g2t11 = a_g2t46 * (-1.0);
  a_g2t12 += a_g2t46 * (g2t14);
  a_g2t14 += a_g2t46 * (g2t12);
  double a_RbarDD22 = a_g2t45 * (alpha);
  a_alpha += a_g2t45 * (RbarDD22);
  double a_g2t34 = a_g2t45 * (-g2t37*g2t43);
  a_g2t37 += a_g2t45 * (-g2t34*g2t43);
  double a_g2t41 = a_g2t45 * (-g2t42*g2t43);
  a_g2t42 += a_g2t45 * (-g2t41*g2t43);
  a_g2t43 += a_g2t45 * (-g2t34*g2t37 - g2t41*g2t42);
  a_g2t44 += a_g2t45 * (1.0);
  a_alpha_dD0 += a_g2t44 * (g2t34);
  a_alpha_dD1 += a_g2t44 * (g2t41);
  a_g2t34 += a_g2t44 * (alpha_dD0);
  a_g2t41 += a_g2t44 * (alpha_dD1);
  a_alpha += a_g2t43 * (2.0);
  a_cf_dD1 += a_g2t42 * (g2t36);
  a_g2t36 += a_g2t42 * (cf_dD1);
  double a_g2t28 = a_g2t41 * (g2t40);
  a_g2t33 += a_g2t41 * (g2t8);
  a_g2t40 += a_g2t41 * (g2t28);
  double a_g2t8 = a_g2t41 * (g2t33);
  a_g2t39 += a_g2t40 * (Rational_1_2);
  a_g2t19 += a_g2t39 * (g2t38);
  a_g2t38 += a_g2t39 * (g2t19);
  a_g2t10 += a_g2t38 * (g2t12);
  a_g2t12 += a_g2t38 * (g2t10);
  double a_g2t15 = a_g2t38 * (-1.0);
  a_cf_dD0 += a_g2t37 * (g2t36);
  a_g2t36 += a_g2t37 * (cf_dD0);
  a_g2t35 += a_g2t36 * (Rational_1_2);
  a_cf += a_g2t35 * (-1.0/(cf*cf));
  a_g2t22 += a_g2t34 * (g2t8);
  a_g2t28 += a_g2t34 * (g2t33);
  a_g2t33 += a_g2t34 * (g2t28);
  a_g2t8 += a_g2t34 * (g2t22);
  a_g2t31 += a_g2t33 * (g2t32);
  a_g2t32 += a_g2t33 * (g2t31);
  a_g2t19 += a_g2t32 * (Rational_1_2);
  a_g2t10 += a_g2t31 * (-g2t29);
  a_g2t2 += a_g2t31 * (g2t30*hDD02);
  a_g2t29 += a_g2t31 * (-g2t10);
  a_g2t30 += a_g2t31 * (g2t2*hDD02);
  a_hDD02 += a_g2t31 * (g2t2*g2t30);
  a_f0_of_xx0 += a_g2t30 * (3.0*(f0_of_xx0*f0_of_xx0)*hDD12);
  a_hDD12 += a_g2t30 * ((f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_f0_of_xx0 += a_g2t29 * (hDD01);
  a_hDD01 += a_g2t29 * (f0_of_xx0);
  a_g2t27 += a_g2t28 * (-1.0);
  a_g2t26 += a_g2t27 * (1.0);
  a_g2t3 += a_g2t27 * (hDD_dD221);
  double a_hDD_dD221 = a_g2t27 * (g2t3);
  a_g2t25 += a_g2t26 * (hDD22 + 1.0);
  double a_hDD22 = a_g2t26 * (g2t25);
  a_f1_of_xx1__D1 += a_g2t25 * (g2t24);
  a_g2t24 += a_g2t25 * (f1_of_xx1__D1);
  a_g2t23 += a_g2t24 * (2.0);
  a_f1_of_xx1 += a_g2t23 * (g2t1);
  a_g2t1 += a_g2t23 * (f1_of_xx1);
  a_g2t21 += a_g2t22 * (Rational_1_2);
  a_g2t19 += a_g2t21 * (g2t20);
  a_g2t20 += a_g2t21 * (g2t19);
  a_g2t10 += a_g2t20 * (g2t14);
  a_g2t14 += a_g2t20 * (g2t10);
  double a_g2t17 = a_g2t20 * (-1.0);
  a_g2t18 += a_g2t19 * (-1.0/(g2t18*g2t18));
  a_g2t10 += a_g2t18 * (-g2t11 + g2t12*g2t14);
  a_g2t11 += a_g2t18 * (-g2t10);
  a_g2t12 += a_g2t18 * (g2t10*g2t14 - g2t17);
  a_g2t14 += a_g2t18 * (g2t10*g2t12 - g2t15);
  a_g2t15 += a_g2t18 * (-g2t14);
  double a_g2t16 = a_g2t18 * (2.0*g2t2*hDD01*hDD02*hDD12);
  a_g2t17 += a_g2t18 * (-g2t12);
  a_g2t2 += a_g2t18 * (2.0*g2t16*hDD01*hDD02*hDD12);
  a_hDD01 += a_g2t18 * (2.0*g2t16*g2t2*hDD02*hDD12);
  a_hDD02 += a_g2t18 * (2.0*g2t16*g2t2*hDD01*hDD12);
  a_hDD12 += a_g2t18 * (2.0*g2t16*g2t2*hDD01*hDD02);
  a_g2t16 += a_g2t17 * (g2t2*(hDD12*hDD12));
  a_g2t2 += a_g2t17 * (g2t16*(hDD12*hDD12));
  a_hDD12 += a_g2t17 * (2.0*g2t16*g2t2*hDD12);
  a_f0_of_xx0 += a_g2t16 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_g2t3 += a_g2t15 * ((hDD02*hDD02));
  a_hDD02 += a_g2t15 * (2.0*g2t3*hDD02);
  a_g2t1 += a_g2t14 * (1.0);
  a_g2t13 += a_g2t14 * (1.0);
  a_g2t1 += a_g2t13 * (hDD11);
  a_hDD11 += a_g2t13 * (g2t1);
  a_hDD00 += a_g2t12 * (1.0);
  a_g2t1 += a_g2t11 * ((hDD01*hDD01));
  a_hDD01 += a_g2t11 * (2.0*g2t1*hDD01);
  a_g2t3 += a_g2t10 * (1.0);
  a_g2t9 += a_g2t10 * (1.0);
  a_g2t3 += a_g2t9 * (hDD22);
  a_hDD22 += a_g2t9 * (g2t3);
  a_g2t7 += a_g2t8 * (-1.0);
  a_g2t3 += a_g2t7 * (hDD_dD220);
  a_g2t6 += a_g2t7 * (1.0);
  double a_hDD_dD220 = a_g2t7 * (g2t3);
  a_g2t5 += a_g2t6 * (hDD22 + 1.0);
  a_hDD22 += a_g2t6 * (g2t5);
  a_g2t2 += a_g2t5 * (g2t4);
  a_g2t4 += a_g2t5 * (g2t2);
  a_f0_of_xx0 += a_g2t4 * (2.0);
  a_g2t1 += a_g2t3 * (g2t2);
  a_g2t2 += a_g2t3 * (g2t1);
  a_f1_of_xx1 += a_g2t2 * (2.0*f1_of_xx1);
  a_f0_of_xx0 += a_g2t1 * (2.0*f0_of_xx0);
  a_cf += a_g2t0 * (2.0*cf);
  red[153 * 64 + lane] = a_RbarDD00;
  red[154 * 64 + lane] = a_RbarDD01;
  red[155 * 64 + lane] = a_RbarDD02;
  red[156 * 64 + lane] = a_RbarDD11;
  red[157 * 64 + lane] = a_RbarDD12;
  red[158 * 64 + lane] = a_RbarDD22;
  red[159 * 64 + lane] = a_aDD00;
  red[160 * 64 + lane] = a_aDD01;
  red[161 * 64 + lane] = a_aDD02;
  red[162 * 64 + lane] = a_aDD11;
  red[163 * 64 + lane] = a_aDD12;
  red[164 * 64 + lane] = a_aDD22;
  red[165 * 64 + lane] = (betaU0 > 0.0) ? a_aDD_dupD000 : 0.0;
  red[166 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_aDD_dupD000;
  red[167 * 64 + lane] = (betaU1 > 0.0) ? a_aDD_dupD001 : 0.0;
  red[168 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_aDD_dupD001;
  red[169 * 64 + lane] = (betaU0 > 0.0) ? a_aDD_dupD010 : 0.0;
  red[170 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_aDD_dupD010;
  red[171 * 64 + lane] = (betaU1 > 0.0) ? a_aDD_dupD011 : 0.0;
  red[172 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_aDD_dupD011;
  red[173 * 64 + lane] = (betaU0 > 0.0) ? a_aDD_dupD020 : 0.0;
  red[174 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_aDD_dupD020;
  red[175 * 64 + lane] = (betaU1 > 0.0) ? a_aDD_dupD021 : 0.0;
  red[176 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_aDD_dupD021;
  red[177 * 64 + lane] = (betaU0 > 0.0) ? a_aDD_dupD110 : 0.0;
  red[178 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_aDD_dupD110;
  red[179 * 64 + lane] = (betaU1 > 0.0) ? a_aDD_dupD111 : 0.0;
  red[180 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_aDD_dupD111;
  red[181 * 64 + lane] = (betaU0 > 0.0) ? a_aDD_dupD120 : 0.0;
  red[182 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_aDD_dupD120;
  red[183 * 64 + lane] = (betaU1 > 0.0) ? a_aDD_dupD121 : 0.0;
  red[184 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_aDD_dupD121;
  red[185 * 64 + lane] = (betaU0 > 0.0) ? a_aDD_dupD220 : 0.0;
  red[186 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_aDD_dupD220;
  red[187 * 64 + lane] = (betaU1 > 0.0) ? a_aDD_dupD221 : 0.0;
  red[188 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_aDD_dupD221;
  red[189 * 64 + lane] = a_alpha;
  red[190 * 64 + lane] = a_alpha_dD0;
  red[191 * 64 + lane] = a_alpha_dD1;
  red[192 * 64 + lane] = a_alpha_dDD00;
  red[193 * 64 + lane] = a_alpha_dDD01;
  red[194 * 64 + lane] = a_alpha_dDD11;
  red[195 * 64 + lane] = a_cf;
  red[196 * 64 + lane] = a_cf_dD0;
  red[197 * 64 + lane] = a_cf_dD1;
  red[198 * 64 + lane] = a_cf_dDD00;
  red[199 * 64 + lane] = a_cf_dDD01;
  red[200 * 64 + lane] = a_cf_dDD11;
  red[201 * 64 + lane] = (betaU0 > 0.0) ? a_cf_dupD0 : 0.0;
  red[202 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_cf_dupD0;
  red[203 * 64 + lane] = (betaU1 > 0.0) ? a_cf_dupD1 : 0.0;
  red[204 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_cf_dupD1;
  red[205 * 64 + lane] = a_hDD00;
  red[206 * 64 + lane] = a_hDD01;
  red[207 * 64 + lane] = a_hDD02;
  red[208 * 64 + lane] = a_hDD11;
  red[209 * 64 + lane] = a_hDD12;
  red[210 * 64 + lane] = a_hDD22;
  red[211 * 64 + lane] = a_hDD_dD000;
  red[212 * 64 + lane] = a_hDD_dD001;
  red[213 * 64 + lane] = a_hDD_dD010;
  red[214 * 64 + lane] = a_hDD_dD011;
  red[215 * 64 + lane] = a_hDD_dD020;
  red[216 * 64 + lane] = a_hDD_dD021;
  red[217 * 64 + lane] = a_hDD_dD110;
  red[218 * 64 + lane] = a_hDD_dD111;
  red[219 * 64 + lane] = a_hDD_dD120;
  red[220 * 64 + lane] = a_hDD_dD121;
  red[221 * 64 + lane] = a_hDD_dD220;
  red[222 * 64 + lane] = a_hDD_dD221;
  red[223 * 64 + lane] = (betaU0 > 0.0) ? a_hDD_dupD000 : 0.0;
  red[224 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_hDD_dupD000;
  red[225 * 64 + lane] = (betaU1 > 0.0) ? a_hDD_dupD001 : 0.0;
  red[226 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_hDD_dupD001;
  red[227 * 64 + lane] = (betaU0 > 0.0) ? a_hDD_dupD010 : 0.0;
  red[228 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_hDD_dupD010;
  red[229 * 64 + lane] = (betaU1 > 0.0) ? a_hDD_dupD011 : 0.0;
  red[230 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_hDD_dupD011;
  red[231 * 64 + lane] = (betaU0 > 0.0) ? a_hDD_dupD020 : 0.0;
  red[232 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_hDD_dupD020;
  red[233 * 64 + lane] = (betaU1 > 0.0) ? a_hDD_dupD021 : 0.0;
  red[234 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_hDD_dupD021;
  red[235 * 64 + lane] = (betaU0 > 0.0) ? a_hDD_dupD110 : 0.0;
  red[236 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_hDD_dupD110;
  red[237 * 64 + lane] = (betaU1 > 0.0) ? a_hDD_dupD111 : 0.0;
  red[238 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_hDD_dupD111;
  red[239 * 64 + lane] = (betaU0 > 0.0) ? a_hDD_dupD120 : 0.0;
  red[240 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_hDD_dupD120;
  red[241 * 64 + lane] = (betaU1 > 0.0) ? a_hDD_dupD121 : 0.0;
  red[242 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_hDD_dupD121;
  red[243 * 64 + lane] = (betaU0 > 0.0) ? a_hDD_dupD220 : 0.0;
  red[244 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_hDD_dupD220;
  red[245 * 64 + lane] = (betaU1 > 0.0) ? a_hDD_dupD221 : 0.0;
  red[246 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_hDD_dupD221;
  red[247 * 64 + lane] = a_trK;
  red[248 * 64 + lane] = (betaU0 > 0.0) ? a_trK_dupD0 : 0.0;
  red[249 * 64 + lane] = (betaU0 > 0.0) ? 0.0 : a_trK_dupD0;
  red[250 * 64 + lane] = (betaU1 > 0.0) ? a_trK_dupD1 : 0.0;
  red[251 * 64 + lane] = (betaU1 > 0.0) ? 0.0 : a_trK_dupD1;
  red[252 * 64 + lane] = a_vetU0;
  red[253 * 64 + lane] = a_vetU1;
  red[254 * 64 + lane] = a_vetU2;
  red[255 * 64 + lane] = a_vetU_dD00;
  red[256 * 64 + lane] = a_vetU_dD01;
  red[257 * 64 + lane] = a_vetU_dD10;
  red[258 * 64 + lane] = a_vetU_dD11;
  red[259 * 64 + lane] = a_vetU_dD20;
  red[260 * 64 + lane] = a_vetU_dD21;
  break;
  }
  default:
    break;
  }
  __syncthreads();
  if (!active) return;
  switch (group) {
  case 0:
    S[0 * Ntot + idx] = red[153 * 64 + lane];
    S[3 * Ntot + idx] = red[156 * 64 + lane];
    S[6 * Ntot + idx] = red[0 * 64 + lane] + red[68 * 64 + lane] + red[159 * 64 + lane];
    S[9 * Ntot + idx] = red[3 * 64 + lane] + red[71 * 64 + lane] + red[162 * 64 + lane];
    S[12 * Ntot + idx] = red[165 * 64 + lane];
    S[15 * Ntot + idx] = red[168 * 64 + lane];
    S[18 * Ntot + idx] = red[171 * 64 + lane];
    S[21 * Ntot + idx] = red[174 * 64 + lane];
    S[24 * Ntot + idx] = red[177 * 64 + lane];
    S[27 * Ntot + idx] = red[180 * 64 + lane];
    S[30 * Ntot + idx] = red[183 * 64 + lane];
    S[33 * Ntot + idx] = red[186 * 64 + lane];
    S[36 * Ntot + idx] = red[6 * 64 + lane] + red[74 * 64 + lane] + red[189 * 64 + lane];
    S[39 * Ntot + idx] = red[192 * 64 + lane];
    S[42 * Ntot + idx] = red[77 * 64 + lane];
    S[45 * Ntot + idx] = red[80 * 64 + lane];
    S[48 * Ntot + idx] = red[11 * 64 + lane] + red[83 * 64 + lane];
    S[51 * Ntot + idx] = red[14 * 64 + lane];
    S[54 * Ntot + idx] = red[17 * 64 + lane];
    S[57 * Ntot + idx] = red[20 * 64 + lane];
    S[60 * Ntot + idx] = red[23 * 64 + lane];
    S[63 * Ntot + idx] = red[26 * 64 + lane] + red[86 * 64 + lane] + red[197 * 64 + lane];
    S[66 * Ntot + idx] = red[200 * 64 + lane];
    S[69 * Ntot + idx] = red[203 * 64 + lane];
    S[72 * Ntot + idx] = red[28 * 64 + lane] + red[88 * 64 + lane] + red[206 * 64 + lane];
    S[75 * Ntot + idx] = red[31 * 64 + lane] + red[91 * 64 + lane] + red[209 * 64 + lane];
    S[78 * Ntot + idx] = red[34 * 64 + lane] + red[94 * 64 + lane] + red[212 * 64 + lane];
    S[81 * Ntot + idx] = red[37 * 64 + lane] + red[97 * 64 + lane] + red[215 * 64 + lane];
    S[84 * Ntot + idx] = red[40 * 64 + lane] + red[100 * 64 + lane] + red[218 * 64 + lane];
    S[87 * Ntot + idx] = red[43 * 64 + lane] + red[103 * 64 + lane] + red[221 * 64 + lane];
    S[90 * Ntot + idx] = red[224 * 64 + lane];
    S[93 * Ntot + idx] = red[227 * 64 + lane];
    S[96 * Ntot + idx] = red[230 * 64 + lane];
    S[99 * Ntot + idx] = red[233 * 64 + lane];
    S[102 * Ntot + idx] = red[236 * 64 + lane];
    S[105 * Ntot + idx] = red[239 * 64 + lane];
    S[108 * Ntot + idx] = red[242 * 64 + lane];
    S[111 * Ntot + idx] = red[245 * 64 + lane];
    S[114 * Ntot + idx] = red[46 * 64 + lane] + red[106 * 64 + lane];
    S[117 * Ntot + idx] = red[109 * 64 + lane];
    S[120 * Ntot + idx] = red[112 * 64 + lane];
    S[123 * Ntot + idx] = red[115 * 64 + lane];
    S[126 * Ntot + idx] = red[118 * 64 + lane];
    S[129 * Ntot + idx] = red[48 * 64 + lane] + red[121 * 64 + lane];
    S[132 * Ntot + idx] = red[249 * 64 + lane];
    S[135 * Ntot + idx] = red[50 * 64 + lane] + red[123 * 64 + lane] + red[252 * 64 + lane];
    S[138 * Ntot + idx] = red[53 * 64 + lane] + red[126 * 64 + lane] + red[255 * 64 + lane];
    S[141 * Ntot + idx] = red[56 * 64 + lane] + red[129 * 64 + lane] + red[258 * 64 + lane];
    S[144 * Ntot + idx] = red[59 * 64 + lane] + red[132 * 64 + lane];
    S[147 * Ntot + idx] = red[62 * 64 + lane] + red[135 * 64 + lane];
    S[150 * Ntot + idx] = red[65 * 64 + lane] + red[138 * 64 + lane];
    S[153 * Ntot + idx] = red[141 * 64 + lane];
    S[156 * Ntot + idx] = red[144 * 64 + lane];
    S[159 * Ntot + idx] = red[147 * 64 + lane];
    S[162 * Ntot + idx] = red[150 * 64 + lane];
    break;
  case 1:
    S[1 * Ntot + idx] = red[154 * 64 + lane];
    S[4 * Ntot + idx] = red[157 * 64 + lane];
    S[7 * Ntot + idx] = red[1 * 64 + lane] + red[69 * 64 + lane] + red[160 * 64 + lane];
    S[10 * Ntot + idx] = red[4 * 64 + lane] + red[72 * 64 + lane] + red[163 * 64 + lane];
    S[13 * Ntot + idx] = red[166 * 64 + lane];
    S[16 * Ntot + idx] = red[169 * 64 + lane];
    S[19 * Ntot + idx] = red[172 * 64 + lane];
    S[22 * Ntot + idx] = red[175 * 64 + lane];
    S[25 * Ntot + idx] = red[178 * 64 + lane];
    S[28 * Ntot + idx] = red[181 * 64 + lane];
    S[31 * Ntot + idx] = red[184 * 64 + lane];
    S[34 * Ntot + idx] = red[187 * 64 + lane];
    S[37 * Ntot + idx] = red[7 * 64 + lane] + red[75 * 64 + lane] + red[190 * 64 + lane];
    S[40 * Ntot + idx] = red[193 * 64 + lane];
    S[43 * Ntot + idx] = red[78 * 64 + lane];
    S[46 * Ntot + idx] = red[9 * 64 + lane] + red[81 * 64 + lane];
    S[49 * Ntot + idx] = red[12 * 64 + lane];
    S[52 * Ntot + idx] = red[15 * 64 + lane];
    S[55 * Ntot + idx] = red[18 * 64 + lane];
    S[58 * Ntot + idx] = red[21 * 64 + lane];
    S[61 * Ntot + idx] = red[24 * 64 + lane] + red[84 * 64 + lane] + red[195 * 64 + lane];
    S[64 * Ntot + idx] = red[198 * 64 + lane];
    S[67 * Ntot + idx] = red[201 * 64 + lane];
    S[70 * Ntot + idx] = red[204 * 64 + lane];
    S[73 * Ntot + idx] = red[29 * 64 + lane] + red[89 * 64 + lane] + red[207 * 64 + lane];
    S[76 * Ntot + idx] = red[32 * 64 + lane] + red[92 * 64 + lane] + red[210 * 64 + lane];
    S[79 * Ntot + idx] = red[35 * 64 + lane] + red[95 * 64 + lane] + red[213 * 64 + lane];
    S[82 * Ntot + idx] = red[38 * 64 + lane] + red[98 * 64 + lane] + red[216 * 64 + lane];
    S[85 * Ntot + idx] = red[41 * 64 + lane] + red[101 * 64 + lane] + red[219 * 64 + lane];
    S[88 * Ntot + idx] = red[44 * 64 + lane] + red[104 * 64 + lane] + red[222 * 64 + lane];
    S[91 * Ntot + idx] = red[225 * 64 + lane];
    S[94 * Ntot + idx] = red[228 * 64 + lane];
    S[97 * Ntot + idx] = red[231 * 64 + lane];
    S[100 * Ntot + idx] = red[234 * 64 + lane];
    S[103 * Ntot + idx] = red[237 * 64 + lane];
    S[106 * Ntot + idx] = red[240 * 64 + lane];
    S[109 * Ntot + idx] = red[243 * 64 + lane];
    S[112 * Ntot + idx] = red[246 * 64 + lane];
    S[115 * Ntot + idx] = red[47 * 64 + lane] + red[107 * 64 + lane];
    S[118 * Ntot + idx] = red[110 * 64 + lane];
    S[121 * Ntot + idx] = red[113 * 64 + lane];
    S[124 * Ntot + idx] = red[116 * 64 + lane];
    S[127 * Ntot + idx] = red[119 * 64 + lane];
    S[130 * Ntot + idx] = red[49 * 64 + lane] + red[122 * 64 + lane];
    S[133 * Ntot + idx] = red[250 * 64 + lane];
    S[136 * Ntot + idx] = red[51 * 64 + lane] + red[124 * 64 + lane] + red[253 * 64 + lane];
    S[139 * Ntot + idx] = red[54 * 64 + lane] + red[127 * 64 + lane] + red[256 * 64 + lane];
    S[142 * Ntot + idx] = red[57 * 64 + lane] + red[130 * 64 + lane] + red[259 * 64 + lane];
    S[145 * Ntot + idx] = red[60 * 64 + lane] + red[133 * 64 + lane];
    S[148 * Ntot + idx] = red[63 * 64 + lane] + red[136 * 64 + lane];
    S[151 * Ntot + idx] = red[66 * 64 + lane] + red[139 * 64 + lane];
    S[154 * Ntot + idx] = red[142 * 64 + lane];
    S[157 * Ntot + idx] = red[145 * 64 + lane];
    S[160 * Ntot + idx] = red[148 * 64 + lane];
    S[163 * Ntot + idx] = red[151 * 64 + lane];
    break;
  case 2:
    S[2 * Ntot + idx] = red[155 * 64 + lane];
    S[5 * Ntot + idx] = red[158 * 64 + lane];
    S[8 * Ntot + idx] = red[2 * 64 + lane] + red[70 * 64 + lane] + red[161 * 64 + lane];
    S[11 * Ntot + idx] = red[5 * 64 + lane] + red[73 * 64 + lane] + red[164 * 64 + lane];
    S[14 * Ntot + idx] = red[167 * 64 + lane];
    S[17 * Ntot + idx] = red[170 * 64 + lane];
    S[20 * Ntot + idx] = red[173 * 64 + lane];
    S[23 * Ntot + idx] = red[176 * 64 + lane];
    S[26 * Ntot + idx] = red[179 * 64 + lane];
    S[29 * Ntot + idx] = red[182 * 64 + lane];
    S[32 * Ntot + idx] = red[185 * 64 + lane];
    S[35 * Ntot + idx] = red[188 * 64 + lane];
    S[38 * Ntot + idx] = red[8 * 64 + lane] + red[76 * 64 + lane] + red[191 * 64 + lane];
    S[41 * Ntot + idx] = red[194 * 64 + lane];
    S[44 * Ntot + idx] = red[79 * 64 + lane];
    S[47 * Ntot + idx] = red[10 * 64 + lane] + red[82 * 64 + lane];
    S[50 * Ntot + idx] = red[13 * 64 + lane];
    S[53 * Ntot + idx] = red[16 * 64 + lane];
    S[56 * Ntot + idx] = red[19 * 64 + lane];
    S[59 * Ntot + idx] = red[22 * 64 + lane];
    S[62 * Ntot + idx] = red[25 * 64 + lane] + red[85 * 64 + lane] + red[196 * 64 + lane];
    S[65 * Ntot + idx] = red[199 * 64 + lane];
    S[68 * Ntot + idx] = red[202 * 64 + lane];
    S[71 * Ntot + idx] = red[27 * 64 + lane] + red[87 * 64 + lane] + red[205 * 64 + lane];
    S[74 * Ntot + idx] = red[30 * 64 + lane] + red[90 * 64 + lane] + red[208 * 64 + lane];
    S[77 * Ntot + idx] = red[33 * 64 + lane] + red[93 * 64 + lane] + red[211 * 64 + lane];
    S[80 * Ntot + idx] = red[36 * 64 + lane] + red[96 * 64 + lane] + red[214 * 64 + lane];
    S[83 * Ntot + idx] = red[39 * 64 + lane] + red[99 * 64 + lane] + red[217 * 64 + lane];
    S[86 * Ntot + idx] = red[42 * 64 + lane] + red[102 * 64 + lane] + red[220 * 64 + lane];
    S[89 * Ntot + idx] = red[223 * 64 + lane];
    S[92 * Ntot + idx] = red[226 * 64 + lane];
    S[95 * Ntot + idx] = red[229 * 64 + lane];
    S[98 * Ntot + idx] = red[232 * 64 + lane];
    S[101 * Ntot + idx] = red[235 * 64 + lane];
    S[104 * Ntot + idx] = red[238 * 64 + lane];
    S[107 * Ntot + idx] = red[241 * 64 + lane];
    S[110 * Ntot + idx] = red[244 * 64 + lane];
    S[113 * Ntot + idx] = red[45 * 64 + lane] + red[105 * 64 + lane];
    S[116 * Ntot + idx] = red[108 * 64 + lane];
    S[119 * Ntot + idx] = red[111 * 64 + lane];
    S[122 * Ntot + idx] = red[114 * 64 + lane];
    S[125 * Ntot + idx] = red[117 * 64 + lane];
    S[128 * Ntot + idx] = red[120 * 64 + lane] + red[247 * 64 + lane];
    S[131 * Ntot + idx] = red[248 * 64 + lane];
    S[134 * Ntot + idx] = red[251 * 64 + lane];
    S[137 * Ntot + idx] = red[52 * 64 + lane] + red[125 * 64 + lane] + red[254 * 64 + lane];
    S[140 * Ntot + idx] = red[55 * 64 + lane] + red[128 * 64 + lane] + red[257 * 64 + lane];
    S[143 * Ntot + idx] = red[58 * 64 + lane] + red[131 * 64 + lane] + red[260 * 64 + lane];
    S[146 * Ntot + idx] = red[61 * 64 + lane] + red[134 * 64 + lane];
    S[149 * Ntot + idx] = red[64 * 64 + lane] + red[137 * 64 + lane];
    S[152 * Ntot + idx] = red[67 * 64 + lane] + red[140 * 64 + lane];
    S[155 * Ntot + idx] = red[143 * 64 + lane];
    S[158 * Ntot + idx] = red[146 * 64 + lane];
    S[161 * Ntot + idx] = red[149 * 64 + lane];
    S[164 * Ntot + idx] = red[152 * 64 + lane];
    break;
  default:
    break;
  }
}
// workgroups of 64 points of one xx0 row x 3 output groups
static void adj_rhs_Spherical_sym2_KO0_fd4_dims(const bhah_kparams &p, dim3 &g, dim3 &b) {
  g = dim3((unsigned)((p.Nx0 - 2 * p.NG + 63) / 64), (unsigned)(p.Nx1 - 2 * p.NG), (unsigned)(p.Nx2 - 2 * p.NG));
  b = dim3(64, 3);
}

// 3 output groups, one wave each over the same 64 points; 95 LDS rows of partial sums
extern "C" __global__ void __launch_bounds__(192)
adj_ricci_Spherical_sym2_KO0_fd4(const double *__restrict__ in, double *__restrict__ S, const double *__restrict__ rfm0,
    const double *__restrict__ rfm1, const bhah_kparams p) {
  __shared__ double red[95 * 64];
  const int lane = (int)threadIdx.x, group = (int)threadIdx.y;
  const int i0r = p.NG + (int)blockIdx.x * 64 + lane;
  const bool active = i0r < p.Nx0 - p.NG;
  const int i0 = active ? i0r : p.Nx0 - p.NG - 1;  // idle lanes repeat the row's last point
  const int i1 = p.NG + (int)blockIdx.y;
  const int i2 = p.NG + (int)blockIdx.z;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;

  switch (group) {
  case 0: { // RbarDD00, RbarDD01
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double hDD00 = in[11 * Ntot + idx];
  const double hDD01 = in[12 * Ntot + idx];
  const double hDD02 = in[13 * Ntot + idx];
  const double hDD11 = in[14 * Ntot + idx];
  const double hDD12 = in[15 * Ntot + idx];
  const double hDD22 = in[16 * Ntot + idx];
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  const double hDD_dDD0000 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[11 * Ntot + idx] + (4.0 / 3.0) * (in[11 * Ntot + idx + (1)] + in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] + in[11 * Ntot + idx + (-2)]));
  const double hDD_dDD0001 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[11 * Ntot + idx + (1 + 1 * s1)] - in[11 * Ntot + idx + (1 + -1 * s1)]) - (in[11 * Ntot + idx + (-1 + 1 * s1)] - in[11 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[11 * Ntot + idx + (1 + 2 * s1)] - in[11 * Ntot + idx + (1 + -2 * s1)]) - (in[11 * Ntot + idx + (-1 + 2 * s1)] - in[11 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[11 * Ntot + idx + (2 + 1 * s1)] - in[11 * Ntot + idx + (2 + -1 * s1)]) - (in[11 * Ntot + idx + (-2 + 1 * s1)] - in[11 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[11 * Ntot + idx + (2 + 2 * s1)] - in[11 * Ntot + idx + (2 + -2 * s1)]) - (in[11 * Ntot + idx + (-2 + 2 * s1)] - in[11 * Ntot + idx + (-2 + -2 * s1)])));
  const double hDD_dDD0011 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[11 * Ntot + idx] + (4.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] + in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] + in[11 * Ntot + idx + (-2 * s1)]));
  const double hDD_dDD0100 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[12 * Ntot + idx] + (4.0 / 3.0) * (in[12 * Ntot + idx + (1)] + in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] + in[12 * Ntot + idx + (-2)]));
  const double hDD_dDD0101 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[12 * Ntot + idx + (1 + 1 * s1)] - in[12 * Ntot + idx + (1 + -1 * s1)]) - (in[12 * Ntot + idx + (-1 + 1 * s1)] - in[12 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[12 * Ntot + idx + (1 + 2 * s1)] - in[12 * Ntot + idx + (1 + -2 * s1)]) - (in[12 * Ntot + idx + (-1 + 2 * s1)] - in[12 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[12 * Ntot + idx + (2 + 1 * s1)] - in[12 * Ntot + idx + (2 + -1 * s1)]) - (in[12 * Ntot + idx + (-2 + 1 * s1)] - in[12 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[12 * Ntot + idx + (2 + 2 * s1)] - in[12 * Ntot + idx + (2 + -2 * s1)]) - (in[12 * Ntot + idx + (-2 + 2 * s1)] - in[12 * Ntot + idx + (-2 + -2 * s1)])));
  const double hDD_dDD0111 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[12 * Ntot + idx] + (4.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] + in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] + in[12 * Ntot + idx + (-2 * s1)]));
  const double lambdaU0 = in[17 * Ntot + idx];
  const double lambdaU1 = in[18 * Ntot + idx];
  const double lambdaU_dD00 = p.invdxx0 * ((2.0 / 3.0) * (in[17 * Ntot + idx + (1)] - in[17 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[17 * Ntot + idx + (2)] - in[17 * Ntot + idx + (-2)]));
  const double lambdaU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (in[17 * Ntot + idx + (1 * s1)] - in[17 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[17 * Ntot + idx + (2 * s1)] - in[17 * Ntot + idx + (-2 * s1)]));
  const double lambdaU_dD10 = p.invdxx0 * ((2.0 / 3.0) * (in[18 * Ntot + idx + (1)] - in[18 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[18 * Ntot + idx + (2)] - in[18 * Ntot + idx + (-2)]));
  const double lambdaU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (in[18 * Ntot + idx + (1 * s1)] - in[18 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[18 * Ntot + idx + (2 * s1)] - in[18 * Ntot + idx + (-2 * s1)]));
  const double lambdaU_dD20 = p.invdxx0 * ((2.0 / 3.0) * (in[19 * Ntot + idx + (1)] - in[19 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[19 * Ntot + idx + (2)] - in[19 * Ntot + idx + (-2)]));
  const double lambdaU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (in[19 * Ntot + idx + (1 * s1)] - in[19 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[19 * Ntot + idx + (2 * s1)] - in[19 * Ntot + idx + (-2 * s1)]));
  const double g0t0 = hDD00 + 1.0;
  const double g0t1 = (f0_of_xx0*f0_of_xx0);
  const double g0t2 = (f1_of_xx1*f1_of_xx1);
  const double g0t3 = g0t1*g0t2;
  const double g0t4 = g0t3*hDD22 + g0t3;
  const double g0t5 = g0t1*(hDD01*hDD01);
  const double g0t6 = g0t1*hDD11;
  const double g0t7 = g0t1 + g0t6;
  const double g0t8 = g0t3*(hDD02*hDD02);
  const double g0t9 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g0t10 = g0t2*g0t9*(hDD12*hDD12);
  const double g0t11 = (1.0 / (-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8));
  const double g0t12 = f0_of_xx0*hDD01;
  const double g0t13 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g0t14 = g0t11*(-g0t12*g0t4 + g0t13*g0t2*hDD02*hDD12);
  const double g0t15 = f0_of_xx0*f1_of_xx1;
  const double g0t16 = g0t15*hDD_dD021;
  const double g0t17 = -g0t16;
  const double g0t18 = f1_of_xx1__D1*hDD02;
  const double g0t19 = f0_of_xx0*g0t18;
  const double g0t20 = f1_of_xx1*g0t1;
  const double g0t21 = 2.0*f0_of_xx0;
  const double g0t22 = f1_of_xx1*hDD12;
  const double g0t23 = g0t20*hDD_dD120 + g0t21*g0t22;
  const double g0t24 = g0t17 - g0t19 + g0t23;
  const double g0t25 = (Rational_1_2)*g0t24;
  const double g0t26 = f1_of_xx1*hDD02;
  const double g0t27 = f0_of_xx0*g0t26;
  const double g0t28 = g0t11*(g0t13*g0t22*hDD01 - g0t27*g0t7);
  const double g0t29 = g0t2*g0t21;
  const double g0t30 = g0t29*hDD22 + g0t29 + g0t3*hDD_dD220;
  const double g0t31 = (Rational_1_2)*g0t30;
  const double g0t32 = g0t14*g0t25 + g0t28*g0t31;
  const double g0t33 = g0t0*g0t32;
  const double g0t34 = g0t11*(g0t0*g0t4 - g0t8);
  const double g0t35 = g0t1*g0t26;
  const double g0t36 = g0t1*g0t22;
  const double g0t37 = g0t11*(-g0t0*g0t36 + g0t35*hDD01);
  const double g0t38 = g0t25*g0t34 + g0t31*g0t37;
  const double g0t39 = g0t21*hDD01;
  const double g0t40 = (1.0 / f0_of_xx0);
  const double g0t41 = -g0t40;
  const double g0t42 = g0t11*(g0t0*g0t7 - g0t5);
  const double g0t43 = g0t25*g0t37 + g0t31*g0t42 + g0t41;
  const double g0t44 = g0t21*g0t26;
  const double g0t45 = (Rational_1_2)*g0t28;
  const double g0t46 = g0t16 + g0t19;
  const double g0t47 = g0t23 + g0t46;
  const double g0t48 = (Rational_1_2)*g0t42;
  const double g0t49 = g0t1*hDD_dD110 + g0t21*hDD11;
  const double g0t50 = g0t21 + g0t49;
  const double g0t51 = (Rational_1_2)*g0t37;
  const double g0t52 = g0t45*hDD_dD001 + g0t47*g0t48 + g0t50*g0t51;
  const double g0t53 = (1.0 / f1_of_xx1);
  const double g0t54 = f1_of_xx1__D1*g0t53;
  const double g0t55 = f1_of_xx1*f1_of_xx1__D1;
  const double g0t56 = g0t1*g0t55;
  const double g0t57 = 2.0*g0t56;
  const double g0t58 = g0t3*hDD_dD221 + g0t57*hDD22 + g0t57;
  const double g0t59 = -g0t24;
  const double g0t60 = g0t45*g0t59 + g0t48*g0t58 - g0t54;
  const double g0t61 = -g0t58;
  const double g0t62 = -g0t30;
  const double g0t63 = g0t45*g0t62 + g0t51*g0t61;
  const double g0t64 = g0t20*hDD_dD121;
  const double g0t65 = f1_of_xx1__D1*g0t1*hDD12;
  const double g0t66 = 2.0*g0t64 + 2.0*g0t65;
  const double g0t67 = 2.0*f0_of_xx0*hDD_dD011 - g0t50;
  const double g0t68 = g0t1*hDD_dD111;
  const double g0t69 = g0t45*g0t67 + g0t48*g0t66 + g0t51*g0t68;
  const double g0t70 = (Rational_1_2)*g0t34;
  const double g0t71 = f1_of_xx1*hDD_dD020;
  const double g0t72 = g0t21*g0t71 + 2.0*g0t26;
  const double g0t73 = 2.0*hDD01;
  const double g0t74 = g0t73 - hDD_dD001;
  const double g0t75 = g0t21*hDD_dD010 + g0t74;
  const double g0t76 = g0t45*hDD_dD000 + g0t48*g0t72 + g0t51*g0t75;
  const double g0t77 = g0t11*(-g0t10 + g0t4*g0t7);
  const double g0t78 = (Rational_1_2)*g0t77;
  const double g0t79 = g0t14*g0t52 + g0t28*g0t43 + g0t37*g0t60 + g0t48*g0t63 + g0t69*g0t70 + g0t76*g0t78;
  const double g0t80 = (Rational_1_2)*g0t14;
  const double g0t81 = g0t45*g0t72 + g0t75*g0t80 + g0t78*hDD_dD000;
  const double g0t82 = g0t0*g0t81;
  const double g0t83 = g0t51*g0t72 + g0t70*g0t75 + g0t80*hDD_dD000;
  const double g0t84 = g0t45*g0t58 + g0t59*g0t78;
  const double g0t85 = g0t28*g0t32;
  const double g0t86 = g0t45*g0t47 + g0t50*g0t80 + g0t78*hDD_dD001;
  const double g0t87 = f0_of_xx0*g0t2;
  const double g0t88 = g0t61*g0t80 + g0t62*g0t78 + g0t87;
  const double g0t89 = f0_of_xx0 + g0t45*g0t66 + g0t67*g0t78 + g0t68*g0t80;
  const double g0t90 = g0t14*g0t86 + g0t37*g0t84 + g0t48*g0t88 + g0t70*g0t89 + g0t78*g0t81 + g0t85;
  const double g0t91 = g0t0*g0t86;
  const double g0t92 = g0t41 + g0t47*g0t51 + g0t50*g0t70 + g0t80*hDD_dD001;
  const double g0t93 = g0t51*g0t58 + g0t59*g0t80;
  const double g0t94 = g0t55 + g0t61*g0t70 + g0t62*g0t80;
  const double g0t95 = g0t51*g0t66 + g0t67*g0t80 + g0t68*g0t70;
  const double g0t96 = g0t14*g0t92 + g0t28*g0t38 + g0t37*g0t93 + g0t48*g0t94 + g0t70*g0t95 + g0t78*g0t83;
  const double g0t97 = g0t12*g0t32 + g0t36*g0t43 + g0t38*g0t7;
  const double g0t98 = g0t0*g0t84 + g0t12*g0t93 + g0t27*g0t60;
  const double g0t99 = 2.0*g0t38;
  const double g0t100 = g0t27*g0t32 + g0t36*g0t38 + g0t4*g0t43;
  const double g0t101 = g0t0*g0t88 + g0t12*g0t94 + g0t27*g0t63;
  const double g0t102 = 2.0*g0t43;
  const double g0t103 = g0t12*g0t86 + g0t36*g0t52 + g0t7*g0t92;
  const double g0t104 = g0t103*g0t92;
  const double g0t105 = g0t0*g0t89 + g0t12*g0t95 + g0t27*g0t69;
  const double g0t106 = g0t105*g0t92;
  const double g0t107 = g0t27*g0t86 + g0t36*g0t92 + g0t4*g0t52;
  const double g0t108 = g0t107*g0t52;
  const double g0t109 = g0t52*g0t98;
  const double g0t110 = g0t12*g0t81 + g0t36*g0t76 + g0t7*g0t83;
  const double g0t111 = g0t12*g0t92 + g0t27*g0t52 + g0t91;
  const double g0t112 = 2.0*g0t83;
  const double g0t113 = g0t27*g0t81 + g0t36*g0t83 + g0t4*g0t76;
  const double g0t114 = g0t12*g0t38 + g0t27*g0t43 + g0t33;
  const double g0t115 = 2.0*g0t76;
  const double g0t116 = g0t103*g0t38;
  const double g0t117 = g0t107*g0t43;
  const double g0t118 = g0t92*g0t98;
  const double g0t119 = g0t111*g0t92;
  const double g0t120 = g0t103*g0t83;
  const double g0t121 = g0t101*g0t52;
  const double g0t122 = g0t114*g0t52;
  const double g0t123 = g0t107*g0t76;
  const double g0t124 = g0t12*g0t55 + g0t87*hDD00 - g0t87*hDD22;
  const double g0t125 = 2.0*g0t40;
  const double g0t126 = -g0t74;
  const double g0t127 = f0_of_xx0*hDD_dD000;
  const double g0t128 = f0_of_xx0*hDD00 - f0_of_xx0*hDD11 + f0_of_xx0*hDD_dD011;
  const double g0t129 = g0t128*g0t40;
  const double g0t130 = g0t127 - 2.0*g0t129;
  const double g0t131 = g0t15*hDD_dD020 + g0t26;
  const double g0t132 = f0_of_xx0*g0t22;
  const double g0t133 = -g0t132 - g0t17;
  const double g0t134 = g0t126*g0t40;
  const double g0t135 = g0t40*(f0_of_xx0*hDD_dD010 + hDD01);
  const double g0t136 = -g0t132 - g0t19;
  const double g0t137 = g0t136*g0t40;
  const double g0t138 = 2.0*g0t137;
  const double g0t139 = 3.0*g0t114;
  const double g0t140 = g0t111*g0t86;
  const double g0t141 = g0t12*g0t83 + g0t27*g0t76 + g0t82;
  const double g0t142 = 3.0*g0t141;
  const double g0t143 = g0t111*g0t32;
  const double g0t144 = 3.0*g0t37;
  const double g0t145 = g0t141*g0t86;
  const double g0t146 = 3.0*g0t14;
  const double g0t147 = g0t111*g0t81;
  const double g0t148 = g0t114*g0t86;
  const double g0t149 = g0t12*g0t84 + g0t36*g0t60 + g0t7*g0t93;
  const double g0t150 = g0t12*g0t88 + g0t36*g0t63 + g0t7*g0t94;
  const double g0t151 = g0t27*g0t84 + g0t36*g0t93 + g0t4*g0t60;
  const double g0t152 = g0t12*g0t89 + g0t36*g0t69 + g0t7*g0t95;
  const double g0t153 = 2.0*g0t92;
  const double g0t154 = g0t27*g0t89 + g0t36*g0t95 + g0t4*g0t69;
  const double g0t155 = (Rational_1_2)*g0t12;
  const double g0t156 = f0_of_xx0*hDD_dDD0101;
  const double g0t157 = g0t136*g0t54;
  double a_f1_of_xx1 = S[0 * Ntot + idx] * (-2.0*g0t40*g0t45*hDD02);
  double a_f1_of_xx1__D1 = S[0 * Ntot + idx] * (-2.0*g0t51*hDD02);
  double a_g0t0 = S[0 * Ntot + idx] * (lambdaU_dD00);
  double a_g0t100 = S[0 * Ntot + idx] * (g0t28*g0t76 + g0t37*g0t52 + g0t42*g0t43);
  double a_g0t101 = S[0 * Ntot + idx] * (g0t102*g0t42 + g0t115*g0t28);
  double a_g0t102 = S[0 * Ntot + idx] * (g0t101*g0t42 + g0t114*g0t28 + g0t37*g0t98);
  double a_g0t104 = S[0 * Ntot + idx] * (g0t34);
  double a_g0t105 = S[0 * Ntot + idx] * (g0t112*g0t14 + g0t37*g0t99);
  double a_g0t106 = S[0 * Ntot + idx] * (2.0*g0t34);
  double a_g0t108 = S[0 * Ntot + idx] * (g0t34);
  double a_g0t109 = S[0 * Ntot + idx] * (2.0*g0t34);
  double a_g0t110 = S[0 * Ntot + idx] * (g0t14*g0t92 + g0t28*g0t38 + g0t77*g0t83);
  double a_g0t111 = S[0 * Ntot + idx] * (g0t112*g0t77 + g0t28*g0t99);
  double a_g0t112 = S[0 * Ntot + idx] * (g0t105*g0t14 + g0t111*g0t77 + g0t28*g0t98);
  double a_g0t113 = S[0 * Ntot + idx] * (g0t14*g0t52 + g0t28*g0t43 + g0t76*g0t77);
  double a_g0t114 = S[0 * Ntot + idx] * (g0t102*g0t28 + g0t115*g0t77);
  double a_g0t115 = S[0 * Ntot + idx] * (g0t101*g0t28 + g0t114*g0t77 + g0t14*g0t98);
  double a_g0t116 = S[0 * Ntot + idx] * (g0t37);
  double a_g0t117 = S[0 * Ntot + idx] * (g0t37);
  double a_g0t118 = S[0 * Ntot + idx] * (2.0*g0t37);
  double a_g0t119 = S[0 * Ntot + idx] * (2.0*g0t14);
  double a_g0t120 = S[0 * Ntot + idx] * (g0t14);
  double a_g0t121 = S[0 * Ntot + idx] * (2.0*g0t37);
  double a_g0t122 = S[0 * Ntot + idx] * (2.0*g0t14);
  double a_g0t123 = S[0 * Ntot + idx] * (g0t14);
  double a_g0t124 = S[0 * Ntot + idx] * (g0t125*g0t48);
  double a_g0t125 = S[0 * Ntot + idx] * (g0t124*g0t48 + g0t131*g0t45 + g0t133*g0t51 + g0t46*g0t51);
  double a_g0t126 = S[0 * Ntot + idx] * (-g0t48*g0t55);
  double a_g0t130 = S[0 * Ntot + idx] * (-g0t70);
  double a_g0t131 = S[0 * Ntot + idx] * (g0t125*g0t45);
  double a_g0t133 = S[0 * Ntot + idx] * (g0t125*g0t51);
  double a_g0t134 = S[0 * Ntot + idx] * (2.0*g0t80);
  double a_g0t135 = S[0 * Ntot + idx] * (2.0*g0t80);
  double a_g0t138 = S[0 * Ntot + idx] * (g0t51);
  double a_g0t139 = S[0 * Ntot + idx] * (g0t28*g0t81 + g0t32*g0t42);
  double a_g0t14 = S[0 * Ntot + idx] * (g0t105*g0t112 + g0t110*g0t92 + g0t113*g0t52 + g0t115*g0t98 + 2.0*g0t119 + g0t120 + 2.0*g0t122 + g0t123);
  double a_g0t140 = S[0 * Ntot + idx] * (3.0*g0t34);
  double a_g0t142 = S[0 * Ntot + idx] * (g0t77*g0t81 + g0t85);
  double a_g0t143 = S[0 * Ntot + idx] * (g0t144);
  double a_g0t144 = S[0 * Ntot + idx] * (g0t143 + g0t148);
  double a_g0t145 = S[0 * Ntot + idx] * (g0t146);
  double a_g0t146 = S[0 * Ntot + idx] * (g0t145 + g0t147);
  double a_g0t147 = S[0 * Ntot + idx] * (g0t146);
  double a_g0t148 = S[0 * Ntot + idx] * (g0t144);
  double a_g0t18 = S[0 * Ntot + idx] * (-2.0*g0t51);
  double a_g0t26 = S[0 * Ntot + idx] * (-4.0*g0t40*g0t45);
  double a_g0t28 = S[0 * Ntot + idx] * (g0t100*g0t76 + g0t101*g0t115 + g0t102*g0t114 + g0t110*g0t38 + g0t111*g0t99 + g0t112*g0t98 + g0t113*g0t43 + g0t139*g0t81 + g0t83*g0t97);
  double a_g0t32 = S[0 * Ntot + idx] * (g0t139*g0t42);
  double a_g0t33 = S[0 * Ntot + idx] * (2.0*g0t79);
  double a_g0t34 = S[0 * Ntot + idx] * (g0t104 + 2.0*g0t106 + g0t108 + 2.0*g0t109 + 3.0*g0t140);
  double a_g0t37 = S[0 * Ntot + idx] * (g0t100*g0t52 + g0t102*g0t98 + g0t105*g0t99 + g0t116 + g0t117 + 2.0*g0t118 + 2.0*g0t121 + g0t92*g0t97);
  double a_g0t38 = S[0 * Ntot + idx] * (g0t110*g0t28 + g0t39*g0t79 + g0t42*g0t97);
  double a_g0t39 = S[0 * Ntot + idx] * (g0t38*g0t79 + g0t83*g0t90 + g0t92*g0t96);
  double a_g0t40 = S[0 * Ntot + idx] * (-2.0*f1_of_xx1*g0t45*hDD02 - 4.0*g0t26*g0t45 - g0t73*g0t80);
  double a_g0t42 = S[0 * Ntot + idx] * (g0t100*g0t43 + g0t101*g0t102 + g0t139*g0t32 + g0t38*g0t97 + g0t98*g0t99);
  double a_g0t43 = S[0 * Ntot + idx] * (g0t100*g0t42 + g0t113*g0t28 + g0t44*g0t79);
  double a_g0t44 = S[0 * Ntot + idx] * (g0t43*g0t79 + g0t52*g0t96 + g0t76*g0t90);
  double a_g0t45 = S[0 * Ntot + idx] * (-2.0*f1_of_xx1*g0t40*hDD02 + g0t125*g0t131 - 4.0*g0t26*g0t40 + 2.0*g0t71);
  double a_g0t46 = S[0 * Ntot + idx] * (g0t125*g0t51);
  double a_g0t48 = S[0 * Ntot + idx] * (g0t124*g0t125 - g0t126*g0t55 - g0t87*hDD_dD000);
  double a_g0t51 = S[0 * Ntot + idx] * (-2.0*f1_of_xx1__D1*hDD02 + g0t125*g0t133 + g0t125*g0t46 + g0t138 - 2.0*g0t18);
  double a_g0t52 = S[0 * Ntot + idx] * (g0t100*g0t37 + g0t113*g0t14 + g0t44*g0t96);
  double a_g0t55 = S[0 * Ntot + idx] * (-g0t126*g0t48);
  double a_g0t70 = S[0 * Ntot + idx] * (-g0t130 + 2.0*hDD_dD011 - hDD_dDD0011);
  double a_g0t71 = S[0 * Ntot + idx] * (2.0*g0t45);
  double a_g0t73 = S[0 * Ntot + idx] * (-g0t40*g0t80);
  double a_g0t76 = S[0 * Ntot + idx] * (g0t100*g0t28 + g0t113*g0t77 + g0t44*g0t90);
  double a_g0t77 = S[0 * Ntot + idx] * (g0t110*g0t83 + g0t111*g0t112 + g0t113*g0t76 + g0t114*g0t115 + g0t142*g0t81);
  double a_g0t78 = S[0 * Ntot + idx] * (-hDD_dDD0000);
  double a_g0t79 = S[0 * Ntot + idx] * (2.0*g0t33 + g0t38*g0t39 + g0t43*g0t44);
  double a_g0t80 = S[0 * Ntot + idx] * (2.0*g0t134 + 2.0*g0t135 - g0t40*g0t73 + 2.0*hDD_dD010 - 2.0*hDD_dDD0001);
  double a_g0t81 = S[0 * Ntot + idx] * (g0t139*g0t28 + g0t142*g0t77);
  double a_g0t82 = S[0 * Ntot + idx] * (2.0*g0t90);
  double a_g0t83 = S[0 * Ntot + idx] * (g0t110*g0t77 + g0t28*g0t97 + g0t39*g0t90);
  double a_g0t85 = S[0 * Ntot + idx] * (g0t142);
  double a_g0t87 = S[0 * Ntot + idx] * (-g0t48*hDD_dD000);
  double a_g0t90 = S[0 * Ntot + idx] * (g0t39*g0t83 + g0t44*g0t76 + 2.0*g0t82);
  double a_g0t91 = S[0 * Ntot + idx] * (2.0*g0t96);
  double a_g0t92 = S[0 * Ntot + idx] * (g0t110*g0t14 + g0t37*g0t97 + g0t39*g0t96);
  double a_g0t96 = S[0 * Ntot + idx] * (g0t39*g0t92 + g0t44*g0t52 + 2.0*g0t91);
  double a_g0t97 = S[0 * Ntot + idx] * (g0t28*g0t83 + g0t37*g0t92 + g0t38*g0t42);
  double a_g0t98 = S[0 * Ntot + idx] * (g0t102*g0t37 + g0t112*g0t28 + g0t115*g0t14 + g0t42*g0t99);
  double a_g0t99 = S[0 * Ntot + idx] * (g0t105*g0t37 + g0t111*g0t28 + g0t42*g0t98);
  double a_hDD01 = S[0 * Ntot + idx] * (lambdaU_dD10);
  double a_hDD02 = S[0 * Ntot + idx] * (-2.0*f1_of_xx1*g0t40*g0t45 - 2.0*f1_of_xx1__D1*g0t51 + lambdaU_dD20);
  double a_hDD_dD000 = S[0 * Ntot + idx] * (-g0t48*g0t87);
  double a_hDD_dD010 = S[0 * Ntot + idx] * (2.0*g0t80);
  double a_hDD_dD011 = S[0 * Ntot + idx] * (2.0*g0t70);
  double a_hDD_dDD0000 = S[0 * Ntot + idx] * (-g0t78);
  double a_hDD_dDD0001 = S[0 * Ntot + idx] * (-2.0*g0t80);
  double a_hDD_dDD0011 = S[0 * Ntot + idx] * (-g0t70);
  double a_lambdaU_dD00 = S[0 * Ntot + idx] * (g0t0);
  double a_lambdaU_dD10 = S[0 * Ntot + idx] * (hDD01);
  double a_lambdaU_dD20 = S[0 * Ntot + idx] * (hDD02);
  double a_f0_of_xx0 = S[1 * Ntot + idx] * (f1_of_xx1__D1*g0t45*hDD_dD020 - 2.0*f1_of_xx1__D1*g0t51*hDD12 - g0t70*(g0t126 + hDD_dD001 - hDD_dD111 + hDD_dDD0111) - g0t78*hDD_dDD0100 + g0t80*hDD_dD110 + (Rational_1_2)*hDD12*lambdaU_dD20);
  a_f1_of_xx1 += S[1 * Ntot + idx] * (-g0t45*hDD12);
  a_f1_of_xx1__D1 += S[1 * Ntot + idx] * (f0_of_xx0*g0t45*hDD_dD020 - g0t51*(2.0*f0_of_xx0*hDD12 + 2.0*f1_of_xx1__D1*g0t27/g0t2));
  double a_f1_of_xx1__DD11 = S[1 * Ntot + idx] * (g0t27*g0t51*g0t53);
  a_g0t0 += S[1 * Ntot + idx] * (-Rational_1_2*lambdaU1 + (Rational_1_2)*lambdaU_dD01);
  double a_g0t1 = S[1 * Ntot + idx] * (-g0t70*(-g0t40*g0t73 + hDD_dD010));
  a_g0t101 += S[1 * Ntot + idx] * (g0t37*g0t69 + g0t42*g0t60);
  double a_g0t103 = S[1 * Ntot + idx] * (g0t14*g0t81 + g0t32*g0t37 + g0t34*g0t86 + g0t96);
  a_g0t104 += S[1 * Ntot + idx] * (2.0*g0t14);
  a_g0t105 += S[1 * Ntot + idx] * (g0t14*g0t81 + g0t32*g0t37 + g0t34*g0t86 + g0t34*g0t95 + g0t37*g0t93 + g0t96);
  a_g0t106 += S[1 * Ntot + idx] * (g0t14);
  a_g0t108 += S[1 * Ntot + idx] * (g0t14);
  a_g0t109 += S[1 * Ntot + idx] * (g0t14);
  a_g0t110 += S[1 * Ntot + idx] * (g0t14*g0t86 + g0t28*g0t32 + g0t77*g0t81 + g0t90);
  a_g0t111 += S[1 * Ntot + idx] * (g0t14*g0t95 + g0t28*g0t93 + g0t34*g0t89 + g0t37*g0t84 + g0t90);
  a_g0t112 += S[1 * Ntot + idx] * (g0t14*g0t152 + g0t149*g0t28);
  a_g0t114 += S[1 * Ntot + idx] * (g0t14*g0t69 + g0t28*g0t60 + g0t37*g0t89 + g0t42*g0t84);
  a_g0t116 += S[1 * Ntot + idx] * (2.0*g0t28);
  a_g0t117 += S[1 * Ntot + idx] * (g0t28);
  a_g0t118 += S[1 * Ntot + idx] * (g0t28);
  a_g0t119 += S[1 * Ntot + idx] * (g0t77);
  a_g0t120 += S[1 * Ntot + idx] * (2.0*g0t77);
  a_g0t121 += S[1 * Ntot + idx] * (g0t28);
  a_g0t122 += S[1 * Ntot + idx] * (g0t77);
  a_g0t123 += S[1 * Ntot + idx] * (g0t77);
  a_g0t124 += S[1 * Ntot + idx] * (g0t48*g0t54);
  a_g0t126 += S[1 * Ntot + idx] * (-f0_of_xx0*g0t70);
  double a_g0t127 = S[1 * Ntot + idx] * (-g0t80);
  double a_g0t128 = S[1 * Ntot + idx] * (-g0t48*g0t55);
  double a_g0t129 = S[1 * Ntot + idx] * (g0t80);
  a_g0t130 += S[1 * Ntot + idx] * (-g0t80);
  a_g0t131 += S[1 * Ntot + idx] * (g0t45*g0t54);
  a_g0t133 += S[1 * Ntot + idx] * (g0t51*g0t54);
  a_g0t135 += S[1 * Ntot + idx] * (g0t78);
  double a_g0t137 = S[1 * Ntot + idx] * (g0t45);
  a_g0t138 += S[1 * Ntot + idx] * (g0t45);
  a_g0t14 += S[1 * Ntot + idx] * (g0t103*g0t81 + 2.0*g0t104 + g0t105*g0t81 + g0t106 + g0t108 + g0t109 + g0t110*g0t86 + g0t111*g0t95 + g0t112*g0t152 + g0t114*g0t69 + 2.0*g0t140 + g0t141*g0t89 + g0t149*g0t76 + g0t154*g0t76 + g0t52*g0t97);
  a_g0t140 += S[1 * Ntot + idx] * (2.0*g0t14);
  double a_g0t141 = S[1 * Ntot + idx] * (g0t14*g0t89 + g0t28*g0t84);
  a_g0t143 += S[1 * Ntot + idx] * (g0t28);
  a_g0t145 += S[1 * Ntot + idx] * (g0t77);
  a_g0t147 += S[1 * Ntot + idx] * (g0t77);
  a_g0t148 += S[1 * Ntot + idx] * (g0t28);
  double a_g0t149 = S[1 * Ntot + idx] * (g0t112*g0t28 + g0t14*g0t76 + g0t153*g0t37 + g0t34*g0t52 + g0t37*g0t43 + g0t42*g0t99);
  double a_g0t15 = S[1 * Ntot + idx] * (g0t45*hDD_dD120);
  double a_g0t150 = S[1 * Ntot + idx] * (g0t28*g0t76 + g0t37*g0t52 + g0t42*g0t43);
  double a_g0t151 = S[1 * Ntot + idx] * (g0t28*g0t76 + g0t37*g0t52 + g0t42*g0t43);
  double a_g0t152 = S[1 * Ntot + idx] * (g0t112*g0t14 + g0t153*g0t34 + g0t37*g0t99);
  double a_g0t153 = S[1 * Ntot + idx] * (g0t149*g0t37 + g0t152*g0t34);
  double a_g0t154 = S[1 * Ntot + idx] * (g0t14*g0t76 + g0t34*g0t52 + g0t37*g0t43);
  double a_g0t155 = S[1 * Ntot + idx] * (g0t40*lambdaU0 + g0t40*lambdaU_dD11 + lambdaU_dD00);
  double a_g0t156 = S[1 * Ntot + idx] * (-2.0*g0t80);
  double a_g0t157 = S[1 * Ntot + idx] * (2.0*g0t51);
  double a_g0t2 = S[1 * Ntot + idx] * ((f1_of_xx1__D1*f1_of_xx1__D1)*g0t27*g0t51/(g0t2*g0t2));
  double a_g0t23 = S[1 * Ntot + idx] * (g0t40*g0t45);
  double a_g0t27 = S[1 * Ntot + idx] * (-g0t51*((f1_of_xx1__D1*f1_of_xx1__D1)/g0t2 - f1_of_xx1__DD11*g0t53));
  a_g0t28 += S[1 * Ntot + idx] * (g0t110*g0t32 + g0t111*g0t93 + g0t112*g0t149 + g0t114*g0t60 + 2.0*g0t116 + g0t117 + g0t118 + g0t121 + g0t141*g0t84 + g0t143 + g0t148 + g0t150*g0t76 + g0t151*g0t76 + g0t43*g0t97 + g0t81*g0t97 + g0t81*g0t98);
  double a_g0t3 = S[1 * Ntot + idx] * (-g0t48*(-g0t40*hDD01 + hDD_dD010));
  a_g0t32 += S[1 * Ntot + idx] * (g0t110*g0t28 + g0t37*(g0t103 + g0t105) + g0t42*(g0t97 + g0t98));
  a_g0t34 += S[1 * Ntot + idx] * (g0t103*g0t86 + g0t105*g0t86 + g0t105*g0t95 + g0t111*g0t89 + g0t149*g0t52 + g0t152*g0t153 + g0t154*g0t52 + g0t69*g0t98);
  double a_g0t35 = S[1 * Ntot + idx] * (g0t40*g0t51);
  a_g0t37 += S[1 * Ntot + idx] * (g0t101*g0t69 + g0t103*g0t32 + g0t105*g0t32 + g0t105*g0t93 + g0t111*g0t84 + g0t114*g0t89 + g0t149*g0t153 + g0t149*g0t43 + g0t150*g0t52 + g0t151*g0t52 + g0t152*g0t99 + g0t154*g0t43 + g0t60*g0t98 + g0t86*g0t97 + g0t86*g0t98 + g0t95*g0t98);
  a_g0t40 += S[1 * Ntot + idx] * (g0t155*(lambdaU0 + lambdaU_dD11) + g0t23*g0t45 - g0t48*(-g0t3*hDD01 - g0t55*g0t6 + g0t56*hDD22) + g0t49*g0t80 - g0t51*(-g0t35 - g0t64) - g0t51*(-g0t64 - g0t65) + (Rational_1_2)*g0t7*lambdaU_dD10 - g0t70*(-g0t1*g0t73 - g0t68) - g0t78*hDD01);
  a_g0t42 += S[1 * Ntot + idx] * (g0t101*g0t60 + g0t114*g0t84 + g0t149*g0t99 + g0t150*g0t43 + g0t151*g0t43 + g0t32*g0t97 + g0t32*g0t98 + g0t93*g0t98);
  a_g0t43 += S[1 * Ntot + idx] * (g0t28*g0t97 + g0t37*(g0t149 + g0t154) + g0t42*(g0t150 + g0t151));
  a_g0t44 += S[1 * Ntot + idx] * (g0t51);
  a_g0t45 += S[1 * Ntot + idx] * (f0_of_xx0*f1_of_xx1__D1*hDD_dD020 - f1_of_xx1*hDD12 + g0t131*g0t54 + g0t137 + g0t138 + g0t15*hDD_dD120 + g0t23*g0t40);
  a_g0t46 += S[1 * Ntot + idx] * (g0t51*g0t54);
  a_g0t48 += S[1 * Ntot + idx] * (g0t124*g0t54 - g0t128*g0t55 - g0t3*hDD_dD010 + g0t40*(g0t3*hDD01 + g0t55*g0t6 - g0t56*hDD22));
  double a_g0t49 = S[1 * Ntot + idx] * (g0t40*g0t80);
  a_g0t51 += S[1 * Ntot + idx] * (-2.0*f0_of_xx0*f1_of_xx1__D1*hDD12 + g0t133*g0t54 + 2.0*g0t157 + g0t27*(-(f1_of_xx1__D1*f1_of_xx1__D1)/g0t2 + f1_of_xx1__DD11*g0t53) + g0t40*(g0t35 + g0t64) + g0t40*(g0t64 + g0t65) + g0t44 + g0t46*g0t54);
  a_g0t52 += S[1 * Ntot + idx] * (g0t14*g0t97 + g0t34*(g0t149 + g0t154) + g0t37*(g0t150 + g0t151));
  double a_g0t53 = S[1 * Ntot + idx] * (f1_of_xx1__DD11*g0t27*g0t51);
  double a_g0t54 = S[1 * Ntot + idx] * (g0t124*g0t48 + g0t131*g0t45 + g0t133*g0t51 + g0t46*g0t51);
  a_g0t55 += S[1 * Ntot + idx] * (-g0t48*(g0t128 - g0t40*g0t6));
  double a_g0t56 = S[1 * Ntot + idx] * (-g0t40*g0t48*hDD22);
  double a_g0t6 = S[1 * Ntot + idx] * (g0t40*g0t48*g0t55);
  double a_g0t60 = S[1 * Ntot + idx] * (g0t101*g0t42 + g0t114*g0t28 + g0t37*g0t98);
  double a_g0t64 = S[1 * Ntot + idx] * (2.0*g0t40*g0t51);
  double a_g0t65 = S[1 * Ntot + idx] * (g0t40*g0t51);
  double a_g0t68 = S[1 * Ntot + idx] * (g0t40*g0t70);
  double a_g0t69 = S[1 * Ntot + idx] * (g0t101*g0t37 + g0t114*g0t14 + g0t34*g0t98);
  double a_g0t7 = S[1 * Ntot + idx] * ((Rational_1_2)*g0t40*lambdaU_dD10);
  a_g0t70 += S[1 * Ntot + idx] * (-f0_of_xx0*g0t126 - f0_of_xx0*hDD_dD001 + f0_of_xx0*hDD_dD111 - f0_of_xx0*hDD_dDD0111 - g0t1*hDD_dD010 + g0t40*(g0t1*g0t73 + g0t68));
  a_g0t73 += S[1 * Ntot + idx] * (g0t1*g0t40*g0t70);
  a_g0t76 += S[1 * Ntot + idx] * (g0t14*(g0t149 + g0t154) + g0t28*(g0t150 + g0t151) + g0t77*g0t97);
  a_g0t77 += S[1 * Ntot + idx] * (g0t110*g0t81 + g0t119 + 2.0*g0t120 + g0t122 + g0t123 + g0t145 + g0t147 + g0t76*g0t97);
  a_g0t78 += S[1 * Ntot + idx] * (-f0_of_xx0*hDD_dDD0100 + g0t135 - g0t40*hDD01 - hDD_dD010);
  a_g0t79 += S[1 * Ntot + idx] * (g0t97 + g0t98);
  a_g0t80 += S[1 * Ntot + idx] * (f0_of_xx0*hDD_dD110 - g0t127 + g0t129 - g0t130 - 2.0*g0t156 + g0t40*g0t49 - hDD00 - hDD11 - hDD_dD011);
  a_g0t81 += S[1 * Ntot + idx] * (g0t110*g0t77 + g0t14*(g0t103 + g0t105) + g0t28*(g0t97 + g0t98));
  double a_g0t84 = S[1 * Ntot + idx] * (g0t111*g0t37 + g0t114*g0t42 + g0t141*g0t28);
  double a_g0t86 = S[1 * Ntot + idx] * (g0t110*g0t14 + g0t34*(g0t103 + g0t105) + g0t37*(g0t97 + g0t98));
  double a_g0t89 = S[1 * Ntot + idx] * (g0t111*g0t34 + g0t114*g0t37 + g0t14*g0t141);
  a_g0t90 += S[1 * Ntot + idx] * (g0t110 + g0t111);
  double a_g0t93 = S[1 * Ntot + idx] * (g0t105*g0t37 + g0t111*g0t28 + g0t42*g0t98);
  double a_g0t95 = S[1 * Ntot + idx] * (g0t105*g0t34 + g0t111*g0t14 + g0t37*g0t98);
  a_g0t96 += S[1 * Ntot + idx] * (g0t103 + g0t105);
  a_g0t97 += S[1 * Ntot + idx] * (g0t14*g0t52 + g0t28*g0t43 + g0t28*g0t81 + g0t32*g0t42 + g0t37*g0t86 + g0t76*g0t77 + g0t79);
  a_g0t98 += S[1 * Ntot + idx] * (g0t28*g0t81 + g0t32*g0t42 + g0t34*g0t69 + g0t37*g0t60 + g0t37*g0t86 + g0t37*g0t95 + g0t42*g0t93 + g0t79);
  a_g0t99 += S[1 * Ntot + idx] * (g0t149*g0t42 + g0t152*g0t37);
  double a_hDD00 = S[1 * Ntot + idx] * (-g0t80);
  a_hDD01 += S[1 * Ntot + idx] * (g0t3*g0t40*g0t48 - g0t40*g0t78);
  a_hDD02 += S[1 * Ntot + idx] * ((Rational_1_2)*lambdaU_dD21);
  double a_hDD11 = S[1 * Ntot + idx] * (-g0t80);
  double a_hDD12 = S[1 * Ntot + idx] * (-2.0*f0_of_xx0*f1_of_xx1__D1*g0t51 + (Rational_1_2)*f0_of_xx0*lambdaU_dD20 - f1_of_xx1*g0t45);
  double a_hDD22 = S[1 * Ntot + idx] * (-g0t40*g0t48*g0t56);
  double a_hDD_dD001 = S[1 * Ntot + idx] * (-f0_of_xx0*g0t70);
  a_hDD_dD010 += S[1 * Ntot + idx] * (-g0t1*g0t70 - g0t3*g0t48 - g0t78);
  a_hDD_dD011 += S[1 * Ntot + idx] * (-g0t80);
  double a_hDD_dD020 = S[1 * Ntot + idx] * (f0_of_xx0*f1_of_xx1__D1*g0t45);
  double a_hDD_dD110 = S[1 * Ntot + idx] * (f0_of_xx0*g0t80);
  double a_hDD_dD111 = S[1 * Ntot + idx] * (f0_of_xx0*g0t70);
  double a_hDD_dD120 = S[1 * Ntot + idx] * (g0t15*g0t45);
  double a_hDD_dDD0100 = S[1 * Ntot + idx] * (-f0_of_xx0*g0t78);
  double a_hDD_dDD0111 = S[1 * Ntot + idx] * (-f0_of_xx0*g0t70);
  double a_lambdaU0 = S[1 * Ntot + idx] * (g0t155*g0t40);
  double a_lambdaU1 = S[1 * Ntot + idx] * (-Rational_1_2*g0t0);
  a_lambdaU_dD00 += S[1 * Ntot + idx] * (g0t155);
  double a_lambdaU_dD01 = S[1 * Ntot + idx] * ((Rational_1_2)*g0t0);
  a_lambdaU_dD10 += S[1 * Ntot + idx] * ((Rational_1_2)*g0t40*g0t7);
  double a_lambdaU_dD11 = S[1 * Ntot + idx] * (g0t155*g0t40);
  a_lambdaU_dD20 += S[1 * Ntot + idx] * ((Rational_1_2)*f0_of_xx0*hDD12);
  double a_lambdaU_dD21 = S[1 * Ntot + idx] * ((Rational_1_2)*hDD02);
  double a_g0t136 = a_g0t157 * (g0t54);
  a_g0t54 += a_g0t157 * (g0t136);
  a_f0_of_xx0 += a_g0t156 * (hDD_dDD0101);
  double a_hDD_dDD0101 = a_g0t156 * (f0_of_xx0);
  double a_g0t12 = a_g0t155 * (Rational_1_2);
  a_g0t27 += a_g0t154 * (g0t89);
  double a_g0t36 = a_g0t154 * (g0t95);
  double a_g0t4 = a_g0t154 * (g0t69);
  a_g0t69 += a_g0t154 * (g0t4);
  a_g0t89 += a_g0t154 * (g0t27);
  a_g0t95 += a_g0t154 * (g0t36);
  a_g0t92 += a_g0t153 * (2.0);
  a_g0t12 += a_g0t152 * (g0t89);
  a_g0t36 += a_g0t152 * (g0t69);
  a_g0t69 += a_g0t152 * (g0t36);
  a_g0t7 += a_g0t152 * (g0t95);
  a_g0t89 += a_g0t152 * (g0t12);
  a_g0t95 += a_g0t152 * (g0t7);
  a_g0t27 += a_g0t151 * (g0t84);
  a_g0t36 += a_g0t151 * (g0t93);
  a_g0t4 += a_g0t151 * (g0t60);
  a_g0t60 += a_g0t151 * (g0t4);
  a_g0t84 += a_g0t151 * (g0t27);
  a_g0t93 += a_g0t151 * (g0t36);
  a_g0t12 += a_g0t150 * (g0t88);
  a_g0t36 += a_g0t150 * (g0t63);
  double a_g0t63 = a_g0t150 * (g0t36);
  a_g0t7 += a_g0t150 * (g0t94);
  double a_g0t88 = a_g0t150 * (g0t12);
  double a_g0t94 = a_g0t150 * (g0t7);
  a_g0t12 += a_g0t149 * (g0t84);
  a_g0t36 += a_g0t149 * (g0t60);
  a_g0t60 += a_g0t149 * (g0t36);
  a_g0t7 += a_g0t149 * (g0t93);
  a_g0t84 += a_g0t149 * (g0t12);
  a_g0t93 += a_g0t149 * (g0t7);
  a_g0t114 += a_g0t148 * (g0t86);
  a_g0t86 += a_g0t148 * (g0t114);
  a_g0t111 += a_g0t147 * (g0t81);
  a_g0t81 += a_g0t147 * (g0t111);
  a_g0t14 += a_g0t146 * (3.0);
  a_g0t141 += a_g0t145 * (g0t86);
  a_g0t86 += a_g0t145 * (g0t141);
  a_g0t37 += a_g0t144 * (3.0);
  a_g0t111 += a_g0t143 * (g0t32);
  a_g0t32 += a_g0t143 * (g0t111);
  a_g0t141 += a_g0t142 * (3.0);
  a_g0t12 += a_g0t141 * (g0t83);
  a_g0t27 += a_g0t141 * (g0t76);
  a_g0t76 += a_g0t141 * (g0t27);
  a_g0t82 += a_g0t141 * (1.0);
  a_g0t83 += a_g0t141 * (g0t12);
  a_g0t111 += a_g0t140 * (g0t86);
  a_g0t86 += a_g0t140 * (g0t111);
  a_g0t114 += a_g0t139 * (3.0);
  a_g0t137 += a_g0t138 * (2.0);
  a_g0t136 += a_g0t137 * (g0t40);
  a_g0t40 += a_g0t137 * (g0t136);
  double a_g0t132 = a_g0t136 * (-1.0);
  double a_g0t19 = a_g0t136 * (-1.0);
  a_f0_of_xx0 += a_g0t135 * (g0t40*hDD_dD010);
  a_g0t40 += a_g0t135 * (f0_of_xx0*hDD_dD010 + hDD01);
  a_hDD01 += a_g0t135 * (g0t40);
  a_hDD_dD010 += a_g0t135 * (f0_of_xx0*g0t40);
  a_g0t126 += a_g0t134 * (g0t40);
  a_g0t40 += a_g0t134 * (g0t126);
  a_g0t132 += a_g0t133 * (-1.0);
  double a_g0t17 = a_g0t133 * (-1.0);
  a_f0_of_xx0 += a_g0t132 * (g0t22);
  double a_g0t22 = a_g0t132 * (f0_of_xx0);
  a_g0t15 += a_g0t131 * (hDD_dD020);
  a_g0t26 += a_g0t131 * (1.0);
  a_hDD_dD020 += a_g0t131 * (g0t15);
  a_g0t127 += a_g0t130 * (1.0);
  a_g0t129 += a_g0t130 * (-2.0);
  a_g0t128 += a_g0t129 * (g0t40);
  a_g0t40 += a_g0t129 * (g0t128);
  a_f0_of_xx0 += a_g0t128 * (hDD00 - hDD11 + hDD_dD011);
  a_hDD00 += a_g0t128 * (f0_of_xx0);
  a_hDD11 += a_g0t128 * (-f0_of_xx0);
  a_hDD_dD011 += a_g0t128 * (f0_of_xx0);
  a_f0_of_xx0 += a_g0t127 * (hDD_dD000);
  a_hDD_dD000 += a_g0t127 * (f0_of_xx0);
  double a_g0t74 = a_g0t126 * (-1.0);
  a_g0t40 += a_g0t125 * (2.0);
  a_g0t12 += a_g0t124 * (g0t55);
  a_g0t55 += a_g0t124 * (g0t12);
  a_g0t87 += a_g0t124 * (hDD00 - hDD22);
  a_hDD00 += a_g0t124 * (g0t87);
  a_hDD22 += a_g0t124 * (-g0t87);
  double a_g0t107 = a_g0t123 * (g0t76);
  a_g0t76 += a_g0t123 * (g0t107);
  a_g0t114 += a_g0t122 * (g0t52);
  a_g0t52 += a_g0t122 * (g0t114);
  a_g0t101 += a_g0t121 * (g0t52);
  a_g0t52 += a_g0t121 * (g0t101);
  a_g0t103 += a_g0t120 * (g0t83);
  a_g0t83 += a_g0t120 * (g0t103);
  a_g0t111 += a_g0t119 * (g0t92);
  a_g0t92 += a_g0t119 * (g0t111);
  a_g0t92 += a_g0t118 * (g0t98);
  a_g0t98 += a_g0t118 * (g0t92);
  a_g0t107 += a_g0t117 * (g0t43);
  a_g0t43 += a_g0t117 * (g0t107);
  a_g0t103 += a_g0t116 * (g0t38);
  a_g0t38 += a_g0t116 * (g0t103);
  a_g0t76 += a_g0t115 * (2.0);
  a_g0t12 += a_g0t114 * (g0t38);
  a_g0t27 += a_g0t114 * (g0t43);
  a_g0t33 += a_g0t114 * (1.0);
  a_g0t38 += a_g0t114 * (g0t12);
  a_g0t43 += a_g0t114 * (g0t27);
  a_g0t27 += a_g0t113 * (g0t81);
  a_g0t36 += a_g0t113 * (g0t83);
  a_g0t4 += a_g0t113 * (g0t76);
  a_g0t76 += a_g0t113 * (g0t4);
  a_g0t81 += a_g0t113 * (g0t27);
  a_g0t83 += a_g0t113 * (g0t36);
  a_g0t83 += a_g0t112 * (2.0);
  a_g0t12 += a_g0t111 * (g0t92);
  a_g0t27 += a_g0t111 * (g0t52);
  a_g0t52 += a_g0t111 * (g0t27);
  a_g0t91 += a_g0t111 * (1.0);
  a_g0t92 += a_g0t111 * (g0t12);
  a_g0t12 += a_g0t110 * (g0t81);
  a_g0t36 += a_g0t110 * (g0t76);
  a_g0t7 += a_g0t110 * (g0t83);
  a_g0t76 += a_g0t110 * (g0t36);
  a_g0t81 += a_g0t110 * (g0t12);
  a_g0t83 += a_g0t110 * (g0t7);
  a_g0t52 += a_g0t109 * (g0t98);
  a_g0t98 += a_g0t109 * (g0t52);
  a_g0t107 += a_g0t108 * (g0t52);
  a_g0t52 += a_g0t108 * (g0t107);
  a_g0t27 += a_g0t107 * (g0t86);
  a_g0t36 += a_g0t107 * (g0t92);
  a_g0t4 += a_g0t107 * (g0t52);
  a_g0t52 += a_g0t107 * (g0t4);
  a_g0t86 += a_g0t107 * (g0t27);
  a_g0t92 += a_g0t107 * (g0t36);
  a_g0t105 += a_g0t106 * (g0t92);
  a_g0t92 += a_g0t106 * (g0t105);
  a_g0t0 += a_g0t105 * (g0t89);
  a_g0t12 += a_g0t105 * (g0t95);
  a_g0t27 += a_g0t105 * (g0t69);
  a_g0t69 += a_g0t105 * (g0t27);
  a_g0t89 += a_g0t105 * (g0t0);
  a_g0t95 += a_g0t105 * (g0t12);
  a_g0t103 += a_g0t104 * (g0t92);
  a_g0t92 += a_g0t104 * (g0t103);
  a_g0t12 += a_g0t103 * (g0t86);
  a_g0t36 += a_g0t103 * (g0t52);
  a_g0t52 += a_g0t103 * (g0t36);
  a_g0t7 += a_g0t103 * (g0t92);
  a_g0t86 += a_g0t103 * (g0t12);
  a_g0t92 += a_g0t103 * (g0t7);
  a_g0t43 += a_g0t102 * (2.0);
  a_g0t0 += a_g0t101 * (g0t88);
  a_g0t12 += a_g0t101 * (g0t94);
  a_g0t27 += a_g0t101 * (g0t63);
  a_g0t63 += a_g0t101 * (g0t27);
  a_g0t88 += a_g0t101 * (g0t0);
  a_g0t94 += a_g0t101 * (g0t12);
  a_g0t27 += a_g0t100 * (g0t32);
  a_g0t32 += a_g0t100 * (g0t27);
  a_g0t36 += a_g0t100 * (g0t38);
  a_g0t38 += a_g0t100 * (g0t36);
  a_g0t4 += a_g0t100 * (g0t43);
  a_g0t43 += a_g0t100 * (g0t4);
  a_g0t38 += a_g0t99 * (2.0);
  a_g0t0 += a_g0t98 * (g0t84);
  a_g0t12 += a_g0t98 * (g0t93);
  a_g0t27 += a_g0t98 * (g0t60);
  a_g0t60 += a_g0t98 * (g0t27);
  a_g0t84 += a_g0t98 * (g0t0);
  a_g0t93 += a_g0t98 * (g0t12);
  a_g0t12 += a_g0t97 * (g0t32);
  a_g0t32 += a_g0t97 * (g0t12);
  a_g0t36 += a_g0t97 * (g0t43);
  a_g0t38 += a_g0t97 * (g0t7);
  a_g0t43 += a_g0t97 * (g0t36);
  a_g0t7 += a_g0t97 * (g0t38);
  a_g0t14 += a_g0t96 * (g0t92);
  a_g0t28 += a_g0t96 * (g0t38);
  a_g0t37 += a_g0t96 * (g0t93);
  a_g0t38 += a_g0t96 * (g0t28);
  a_g0t48 += a_g0t96 * (g0t94);
  a_g0t70 += a_g0t96 * (g0t95);
  a_g0t78 += a_g0t96 * (g0t83);
  a_g0t83 += a_g0t96 * (g0t78);
  a_g0t92 += a_g0t96 * (g0t14);
  a_g0t93 += a_g0t96 * (g0t37);
  a_g0t94 += a_g0t96 * (g0t48);
  a_g0t95 += a_g0t96 * (g0t70);
  a_g0t51 += a_g0t95 * (g0t66);
  double a_g0t66 = a_g0t95 * (g0t51);
  double a_g0t67 = a_g0t95 * (g0t80);
  a_g0t68 += a_g0t95 * (g0t70);
  a_g0t70 += a_g0t95 * (g0t68);
  a_g0t80 += a_g0t95 * (g0t67);
  a_g0t55 += a_g0t94 * (1.0);
  double a_g0t61 = a_g0t94 * (g0t70);
  double a_g0t62 = a_g0t94 * (g0t80);
  a_g0t70 += a_g0t94 * (g0t61);
  a_g0t80 += a_g0t94 * (g0t62);
  a_g0t51 += a_g0t93 * (g0t58);
  double a_g0t58 = a_g0t93 * (g0t51);
  double a_g0t59 = a_g0t93 * (g0t80);
  a_g0t80 += a_g0t93 * (g0t59);
  double a_g0t41 = a_g0t92 * (1.0);
  double a_g0t47 = a_g0t92 * (g0t51);
  double a_g0t50 = a_g0t92 * (g0t70);
  a_g0t51 += a_g0t92 * (g0t47);
  a_g0t70 += a_g0t92 * (g0t50);
  a_g0t80 += a_g0t92 * (hDD_dD001);
  a_hDD_dD001 += a_g0t92 * (g0t80);
  a_g0t0 += a_g0t91 * (g0t86);
  a_g0t86 += a_g0t91 * (g0t0);
  a_g0t14 += a_g0t90 * (g0t86);
  a_g0t37 += a_g0t90 * (g0t84);
  a_g0t48 += a_g0t90 * (g0t88);
  a_g0t70 += a_g0t90 * (g0t89);
  a_g0t78 += a_g0t90 * (g0t81);
  a_g0t81 += a_g0t90 * (g0t78);
  a_g0t84 += a_g0t90 * (g0t37);
  a_g0t85 += a_g0t90 * (1.0);
  a_g0t86 += a_g0t90 * (g0t14);
  a_g0t88 += a_g0t90 * (g0t48);
  a_g0t89 += a_g0t90 * (g0t70);
  a_f0_of_xx0 += a_g0t89 * (1.0);
  a_g0t45 += a_g0t89 * (g0t66);
  a_g0t66 += a_g0t89 * (g0t45);
  a_g0t67 += a_g0t89 * (g0t78);
  a_g0t68 += a_g0t89 * (g0t80);
  a_g0t78 += a_g0t89 * (g0t67);
  a_g0t80 += a_g0t89 * (g0t68);
  a_g0t61 += a_g0t88 * (g0t80);
  a_g0t62 += a_g0t88 * (g0t78);
  a_g0t78 += a_g0t88 * (g0t62);
  a_g0t80 += a_g0t88 * (g0t61);
  a_g0t87 += a_g0t88 * (1.0);
  a_f0_of_xx0 += a_g0t87 * (g0t2);
  a_g0t2 += a_g0t87 * (f0_of_xx0);
  a_g0t45 += a_g0t86 * (g0t47);
  a_g0t47 += a_g0t86 * (g0t45);
  a_g0t50 += a_g0t86 * (g0t80);
  a_g0t78 += a_g0t86 * (hDD_dD001);
  a_g0t80 += a_g0t86 * (g0t50);
  a_hDD_dD001 += a_g0t86 * (g0t78);
  a_g0t28 += a_g0t85 * (g0t32);
  a_g0t32 += a_g0t85 * (g0t28);
  a_g0t45 += a_g0t84 * (g0t58);
  a_g0t58 += a_g0t84 * (g0t45);
  a_g0t59 += a_g0t84 * (g0t78);
  a_g0t78 += a_g0t84 * (g0t59);
  a_g0t51 += a_g0t83 * (g0t72);
  a_g0t70 += a_g0t83 * (g0t75);
  double a_g0t72 = a_g0t83 * (g0t51);
  double a_g0t75 = a_g0t83 * (g0t70);
  a_g0t80 += a_g0t83 * (hDD_dD000);
  a_hDD_dD000 += a_g0t83 * (g0t80);
  a_g0t0 += a_g0t82 * (g0t81);
  a_g0t81 += a_g0t82 * (g0t0);
  a_g0t45 += a_g0t81 * (g0t72);
  a_g0t72 += a_g0t81 * (g0t45);
  a_g0t75 += a_g0t81 * (g0t80);
  a_g0t78 += a_g0t81 * (hDD_dD000);
  a_g0t80 += a_g0t81 * (g0t75);
  a_hDD_dD000 += a_g0t81 * (g0t78);
  a_g0t14 += a_g0t80 * (Rational_1_2);
  a_g0t14 += a_g0t79 * (g0t52);
  a_g0t28 += a_g0t79 * (g0t43);
  a_g0t37 += a_g0t79 * (g0t60);
  a_g0t43 += a_g0t79 * (g0t28);
  a_g0t48 += a_g0t79 * (g0t63);
  a_g0t52 += a_g0t79 * (g0t14);
  a_g0t60 += a_g0t79 * (g0t37);
  a_g0t63 += a_g0t79 * (g0t48);
  a_g0t69 += a_g0t79 * (g0t70);
  a_g0t70 += a_g0t79 * (g0t69);
  a_g0t76 += a_g0t79 * (g0t78);
  a_g0t78 += a_g0t79 * (g0t76);
  a_g0t77 += a_g0t78 * (Rational_1_2);
  double a_g0t10 = a_g0t77 * (-g0t11);
  double a_g0t11 = a_g0t77 * (-g0t10 + g0t4*g0t7);
  a_g0t4 += a_g0t77 * (g0t11*g0t7);
  a_g0t7 += a_g0t77 * (g0t11*g0t4);
  a_g0t45 += a_g0t76 * (hDD_dD000);
  a_g0t48 += a_g0t76 * (g0t72);
  a_g0t51 += a_g0t76 * (g0t75);
  a_g0t72 += a_g0t76 * (g0t48);
  a_g0t75 += a_g0t76 * (g0t51);
  a_hDD_dD000 += a_g0t76 * (g0t45);
  double a_g0t21 = a_g0t75 * (hDD_dD010);
  a_g0t74 += a_g0t75 * (1.0);
  a_hDD_dD010 += a_g0t75 * (g0t21);
  a_g0t73 += a_g0t74 * (1.0);
  a_hDD_dD001 += a_g0t74 * (-1.0);
  a_hDD01 += a_g0t73 * (2.0);
  a_g0t21 += a_g0t72 * (g0t71);
  a_g0t26 += a_g0t72 * (2.0);
  a_g0t71 += a_g0t72 * (g0t21);
  a_f1_of_xx1 += a_g0t71 * (hDD_dD020);
  a_hDD_dD020 += a_g0t71 * (f1_of_xx1);
  a_g0t34 += a_g0t70 * (Rational_1_2);
  a_g0t45 += a_g0t69 * (g0t67);
  a_g0t48 += a_g0t69 * (g0t66);
  a_g0t51 += a_g0t69 * (g0t68);
  a_g0t66 += a_g0t69 * (g0t48);
  a_g0t67 += a_g0t69 * (g0t45);
  a_g0t68 += a_g0t69 * (g0t51);
  a_g0t1 += a_g0t68 * (hDD_dD111);
  a_hDD_dD111 += a_g0t68 * (g0t1);
  a_f0_of_xx0 += a_g0t67 * (2.0*hDD_dD011);
  a_g0t50 += a_g0t67 * (-1.0);
  a_hDD_dD011 += a_g0t67 * (2.0*f0_of_xx0);
  a_g0t64 += a_g0t66 * (2.0);
  a_g0t65 += a_g0t66 * (2.0);
  a_f1_of_xx1__D1 += a_g0t65 * (g0t1*hDD12);
  a_g0t1 += a_g0t65 * (f1_of_xx1__D1*hDD12);
  a_hDD12 += a_g0t65 * (f1_of_xx1__D1*g0t1);
  double a_g0t20 = a_g0t64 * (hDD_dD121);
  double a_hDD_dD121 = a_g0t64 * (g0t20);
  a_g0t45 += a_g0t63 * (g0t62);
  a_g0t51 += a_g0t63 * (g0t61);
  a_g0t61 += a_g0t63 * (g0t51);
  a_g0t62 += a_g0t63 * (g0t45);
  double a_g0t30 = a_g0t62 * (-1.0);
  a_g0t58 += a_g0t61 * (-1.0);
  a_g0t45 += a_g0t60 * (g0t59);
  a_g0t48 += a_g0t60 * (g0t58);
  a_g0t54 += a_g0t60 * (-1.0);
  a_g0t58 += a_g0t60 * (g0t48);
  a_g0t59 += a_g0t60 * (g0t45);
  double a_g0t24 = a_g0t59 * (-1.0);
  a_g0t3 += a_g0t58 * (hDD_dD221);
  double a_g0t57 = a_g0t58 * (hDD22 + 1.0);
  a_hDD22 += a_g0t58 * (g0t57);
  double a_hDD_dD221 = a_g0t58 * (g0t3);
  a_g0t56 += a_g0t57 * (2.0);
  a_g0t1 += a_g0t56 * (g0t55);
  a_g0t55 += a_g0t56 * (g0t1);
  a_f1_of_xx1 += a_g0t55 * (f1_of_xx1__D1);
  a_f1_of_xx1__D1 += a_g0t55 * (f1_of_xx1);
  a_f1_of_xx1__D1 += a_g0t54 * (g0t53);
  a_g0t53 += a_g0t54 * (f1_of_xx1__D1);
  a_f1_of_xx1 += a_g0t53 * (-1.0/(f1_of_xx1*f1_of_xx1));
  a_g0t45 += a_g0t52 * (hDD_dD001);
  a_g0t47 += a_g0t52 * (g0t48);
  a_g0t48 += a_g0t52 * (g0t47);
  a_g0t50 += a_g0t52 * (g0t51);
  a_g0t51 += a_g0t52 * (g0t50);
  a_hDD_dD001 += a_g0t52 * (g0t45);
  a_g0t37 += a_g0t51 * (Rational_1_2);
  a_g0t21 += a_g0t50 * (1.0);
  a_g0t49 += a_g0t50 * (1.0);
  a_g0t1 += a_g0t49 * (hDD_dD110);
  a_g0t21 += a_g0t49 * (hDD11);
  a_hDD11 += a_g0t49 * (g0t21);
  a_hDD_dD110 += a_g0t49 * (g0t1);
  a_g0t42 += a_g0t48 * (Rational_1_2);
  a_g0t23 += a_g0t47 * (1.0);
  a_g0t46 += a_g0t47 * (1.0);
  double a_g0t16 = a_g0t46 * (1.0);
  a_g0t19 += a_g0t46 * (1.0);
  a_g0t28 += a_g0t45 * (Rational_1_2);
  a_g0t21 += a_g0t44 * (g0t26);
  a_g0t26 += a_g0t44 * (g0t21);
  double a_g0t25 = a_g0t43 * (g0t37);
  double a_g0t31 = a_g0t43 * (g0t42);
  a_g0t37 += a_g0t43 * (g0t25);
  a_g0t41 += a_g0t43 * (1.0);
  a_g0t42 += a_g0t43 * (g0t31);
  a_g0t0 += a_g0t42 * (g0t11*g0t7);
  a_g0t11 += a_g0t42 * (g0t0*g0t7 - g0t5);
  double a_g0t5 = a_g0t42 * (-g0t11);
  a_g0t7 += a_g0t42 * (g0t0*g0t11);
  a_g0t40 += a_g0t41 * (-1.0);
  a_f0_of_xx0 += a_g0t40 * (-1.0/(f0_of_xx0*f0_of_xx0));
  a_g0t21 += a_g0t39 * (hDD01);
  a_hDD01 += a_g0t39 * (g0t21);
  a_g0t25 += a_g0t38 * (g0t34);
  a_g0t31 += a_g0t38 * (g0t37);
  a_g0t34 += a_g0t38 * (g0t25);
  a_g0t37 += a_g0t38 * (g0t31);
  a_g0t0 += a_g0t37 * (-g0t11*g0t36);
  a_g0t11 += a_g0t37 * (-g0t0*g0t36 + g0t35*hDD01);
  a_g0t35 += a_g0t37 * (g0t11*hDD01);
  a_g0t36 += a_g0t37 * (-g0t0*g0t11);
  a_hDD01 += a_g0t37 * (g0t11*g0t35);
  a_g0t1 += a_g0t36 * (g0t22);
  a_g0t22 += a_g0t36 * (g0t1);
  a_g0t1 += a_g0t35 * (g0t26);
  a_g0t26 += a_g0t35 * (g0t1);
  a_g0t0 += a_g0t34 * (g0t11*g0t4);
  a_g0t11 += a_g0t34 * (g0t0*g0t4 - g0t8);
  a_g0t4 += a_g0t34 * (g0t0*g0t11);
  double a_g0t8 = a_g0t34 * (-g0t11);
  a_g0t0 += a_g0t33 * (g0t32);
  a_g0t32 += a_g0t33 * (g0t0);
  a_g0t14 += a_g0t32 * (g0t25);
  a_g0t25 += a_g0t32 * (g0t14);
  a_g0t28 += a_g0t32 * (g0t31);
  a_g0t31 += a_g0t32 * (g0t28);
  a_g0t30 += a_g0t31 * (Rational_1_2);
  double a_g0t29 = a_g0t30 * (hDD22 + 1.0);
  a_g0t3 += a_g0t30 * (hDD_dD220);
  a_hDD22 += a_g0t30 * (g0t29);
  double a_hDD_dD220 = a_g0t30 * (g0t3);
  a_g0t2 += a_g0t29 * (g0t21);
  a_g0t21 += a_g0t29 * (g0t2);
  a_g0t11 += a_g0t28 * (g0t13*g0t22*hDD01 - g0t27*g0t7);
  double a_g0t13 = a_g0t28 * (g0t11*g0t22*hDD01);
  a_g0t22 += a_g0t28 * (g0t11*g0t13*hDD01);
  a_g0t27 += a_g0t28 * (-g0t11*g0t7);
  a_g0t7 += a_g0t28 * (-g0t11*g0t27);
  a_hDD01 += a_g0t28 * (g0t11*g0t13*g0t22);
  a_f0_of_xx0 += a_g0t27 * (g0t26);
  a_g0t26 += a_g0t27 * (f0_of_xx0);
  a_f1_of_xx1 += a_g0t26 * (hDD02);
  a_hDD02 += a_g0t26 * (f1_of_xx1);
  a_g0t24 += a_g0t25 * (Rational_1_2);
  a_g0t17 += a_g0t24 * (1.0);
  a_g0t19 += a_g0t24 * (-1.0);
  a_g0t23 += a_g0t24 * (1.0);
  a_g0t20 += a_g0t23 * (hDD_dD120);
  a_g0t21 += a_g0t23 * (g0t22);
  a_g0t22 += a_g0t23 * (g0t21);
  a_hDD_dD120 += a_g0t23 * (g0t20);
  a_f1_of_xx1 += a_g0t22 * (hDD12);
  a_hDD12 += a_g0t22 * (f1_of_xx1);
  a_f0_of_xx0 += a_g0t21 * (2.0);
  a_f1_of_xx1 += a_g0t20 * (g0t1);
  a_g0t1 += a_g0t20 * (f1_of_xx1);
  a_f0_of_xx0 += a_g0t19 * (g0t18);
  a_g0t18 += a_g0t19 * (f0_of_xx0);
  a_f1_of_xx1__D1 += a_g0t18 * (hDD02);
  a_hDD02 += a_g0t18 * (f1_of_xx1__D1);
  a_g0t16 += a_g0t17 * (-1.0);
  a_g0t15 += a_g0t16 * (hDD_dD021);
  double a_hDD_dD021 = a_g0t16 * (g0t15);
  a_f0_of_xx0 += a_g0t15 * (f1_of_xx1);
  a_f1_of_xx1 += a_g0t15 * (f0_of_xx0);
  a_g0t11 += a_g0t14 * (-g0t12*g0t4 + g0t13*g0t2*hDD02*hDD12);
  a_g0t12 += a_g0t14 * (-g0t11*g0t4);
  a_g0t13 += a_g0t14 * (g0t11*g0t2*hDD02*hDD12);
  a_g0t2 += a_g0t14 * (g0t11*g0t13*hDD02*hDD12);
  a_g0t4 += a_g0t14 * (-g0t11*g0t12);
  a_hDD02 += a_g0t14 * (g0t11*g0t13*g0t2*hDD12);
  a_hDD12 += a_g0t14 * (g0t11*g0t13*g0t2*hDD02);
  a_f0_of_xx0 += a_g0t13 * (3.0*(f0_of_xx0*f0_of_xx0));
  a_f0_of_xx0 += a_g0t12 * (hDD01);
  a_hDD01 += a_g0t12 * (f0_of_xx0);
  a_g0t0 += a_g0t11 * ((g0t10 - g0t4*g0t7)/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_g0t10 += a_g0t11 * (g0t0/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_g0t2 += a_g0t11 * (-2.0*g0t9*hDD01*hDD02*hDD12/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_g0t4 += a_g0t11 * ((-g0t0*g0t7 + g0t5)/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_g0t5 += a_g0t11 * (g0t4/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_g0t7 += a_g0t11 * ((-g0t0*g0t4 + g0t8)/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_g0t8 += a_g0t11 * (g0t7/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  double a_g0t9 = a_g0t11 * (-2.0*g0t2*hDD01*hDD02*hDD12/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_hDD01 += a_g0t11 * (-2.0*g0t2*g0t9*hDD02*hDD12/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_hDD02 += a_g0t11 * (-2.0*g0t2*g0t9*hDD01*hDD12/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_hDD12 += a_g0t11 * (-2.0*g0t2*g0t9*hDD01*hDD02/((-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)*(-g0t0*g0t10 + g0t0*g0t4*g0t7 + 2.0*g0t2*g0t9*hDD01*hDD02*hDD12 - g0t4*g0t5 - g0t7*g0t8)));
  a_g0t2 += a_g0t10 * (g0t9*(hDD12*hDD12));
  a_g0t9 += a_g0t10 * (g0t2*(hDD12*hDD12));
  a_hDD12 += a_g0t10 * (2.0*g0t2*g0t9*hDD12);
  a_f0_of_xx0 += a_g0t9 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_g0t3 += a_g0t8 * ((hDD02*hDD02));
  a_hDD02 += a_g0t8 * (2.0*g0t3*hDD02);
  a_g0t1 += a_g0t7 * (1.0);
  a_g0t6 += a_g0t7 * (1.0);
  a_g0t1 += a_g0t6 * (hDD11);
  a_hDD11 += a_g0t6 * (g0t1);
  a_g0t1 += a_g0t5 * ((hDD01*hDD01));
  a_hDD01 += a_g0t5 * (2.0*g0t1*hDD01);
  a_g0t3 += a_g0t4 * (hDD22 + 1.0);
  a_hDD22 += a_g0t4 * (g0t3);
  a_g0t1 += a_g0t3 * (g0t2);
  a_g0t2 += a_g0t3 * (g0t1);
  a_f1_of_xx1 += a_g0t2 * (2.0*f1_of_xx1);
  a_f0_of_xx0 += a_g0t1 * (2.0*f0_of_xx0);
  a_hDD00 += a_g0t0 * (1.0);
  red[0 * 64 + lane] = a_hDD00;
  red[1 * 64 + lane] = a_hDD01;
  red[2 * 64 + lane] = a_hDD02;
  red[3 * 64 + lane] = a_hDD11;
  red[4 * 64 + lane] = a_hDD12;
  red[5 * 64 + lane] = a_hDD22;
  red[6 * 64 + lane] = a_hDD_dD000;
  red[7 * 64 + lane] = a_hDD_dD001;
  red[8 * 64 + lane] = a_hDD_dD010;
  red[9 * 64 + lane] = a_hDD_dD011;
  red[10 * 64 + lane] = a_hDD_dD020;
  red[11 * 64 + lane] = a_hDD_dD021;
  red[12 * 64 + lane] = a_hDD_dD110;
  red[13 * 64 + lane] = a_hDD_dD111;
  red[14 * 64 + lane] = a_hDD_dD120;
  red[15 * 64 + lane] = a_hDD_dD121;
  red[16 * 64 + lane] = a_hDD_dD220;
  red[17 * 64 + lane] = a_hDD_dD221;
  red[18 * 64 + lane] = a_hDD_dDD0000;
  red[19 * 64 + lane] = a_hDD_dDD0001;
  red[20 * 64 + lane] = a_hDD_dDD0011;
  red[21 * 64 + lane] = a_hDD_dDD0100;
  red[22 * 64 + lane] = a_hDD_dDD0101;
  red[23 * 64 + lane] = a_hDD_dDD0111;
  red[24 * 64 + lane] = a_lambdaU0;
  red[25 * 64 + lane] = a_lambdaU1;
  red[26 * 64 + lane] = a_lambdaU_dD00;
  red[27 * 64 + lane] = a_lambdaU_dD01;
  red[28 * 64 + lane] = a_lambdaU_dD10;
  red[29 * 64 + lane] = a_lambdaU_dD11;
  red[30 * 64 + lane] = a_lambdaU_dD20;
  red[31 * 64 + lane] = a_lambdaU_dD21;
  break;
  }
  case 1: { // RbarDD02, RbarDD11
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double hDD00 = in[11 * Ntot + idx];
  const double hDD01 = in[12 * Ntot + idx];
  const double hDD02 = in[13 * Ntot + idx];
  const double hDD11 = in[14 * Ntot + idx];
  const double hDD12 = in[15 * Ntot + idx];
  const double hDD22 = in[16 * Ntot + idx];
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  const double hDD_dDD0200 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[13 * Ntot + idx] + (4.0 / 3.0) * (in[13 * Ntot + idx + (1)] + in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] + in[13 * Ntot + idx + (-2)]));
  const double hDD_dDD0201 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[13 * Ntot + idx + (1 + 1 * s1)] - in[13 * Ntot + idx + (1 + -1 * s1)]) - (in[13 * Ntot + idx + (-1 + 1 * s1)] - in[13 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[13 * Ntot + idx + (1 + 2 * s1)] - in[13 * Ntot + idx + (1 + -2 * s1)]) - (in[13 * Ntot + idx + (-1 + 2 * s1)] - in[13 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[13 * Ntot + idx + (2 + 1 * s1)] - in[13 * Ntot + idx + (2 + -1 * s1)]) - (in[13 * Ntot + idx + (-2 + 1 * s1)] - in[13 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[13 * Ntot + idx + (2 + 2 * s1)] - in[13 * Ntot + idx + (2 + -2 * s1)]) - (in[13 * Ntot + idx + (-2 + 2 * s1)] - in[13 * Ntot + idx + (-2 + -2 * s1)])));
  const double hDD_dDD0211 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[13 * Ntot + idx] + (4.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] + in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] + in[13 * Ntot + idx + (-2 * s1)]));
  const double hDD_dDD1100 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[14 * Ntot + idx] + (4.0 / 3.0) * (in[14 * Ntot + idx + (1)] + in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] + in[14 * Ntot + idx + (-2)]));
  const double hDD_dDD1101 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[14 * Ntot + idx + (1 + 1 * s1)] - in[14 * Ntot + idx + (1 + -1 * s1)]) - (in[14 * Ntot + idx + (-1 + 1 * s1)] - in[14 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[14 * Ntot + idx + (1 + 2 * s1)] - in[14 * Ntot + idx + (1 + -2 * s1)]) - (in[14 * Ntot + idx + (-1 + 2 * s1)] - in[14 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[14 * Ntot + idx + (2 + 1 * s1)] - in[14 * Ntot + idx + (2 + -1 * s1)]) - (in[14 * Ntot + idx + (-2 + 1 * s1)] - in[14 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[14 * Ntot + idx + (2 + 2 * s1)] - in[14 * Ntot + idx + (2 + -2 * s1)]) - (in[14 * Ntot + idx + (-2 + 2 * s1)] - in[14 * Ntot + idx + (-2 + -2 * s1)])));
  const double hDD_dDD1111 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[14 * Ntot + idx] + (4.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] + in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] + in[14 * Ntot + idx + (-2 * s1)]));
  const double lambdaU0 = in[17 * Ntot + idx];
  const double lambdaU1 = in[18 * Ntot + idx];
  const double lambdaU2 = in[19 * Ntot + idx];
  const double lambdaU_dD00 = p.invdxx0 * ((2.0 / 3.0) * (in[17 * Ntot + idx + (1)] - in[17 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[17 * Ntot + idx + (2)] - in[17 * Ntot + idx + (-2)]));
  const double lambdaU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (in[17 * Ntot + idx + (1 * s1)] - in[17 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[17 * Ntot + idx + (2 * s1)] - in[17 * Ntot + idx + (-2 * s1)]));
  const double lambdaU_dD10 = p.invdxx0 * ((2.0 / 3.0) * (in[18 * Ntot + idx + (1)] - in[18 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[18 * Ntot + idx + (2)] - in[18 * Ntot + idx + (-2)]));
  const double lambdaU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (in[18 * Ntot + idx + (1 * s1)] - in[18 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[18 * Ntot + idx + (2 * s1)] - in[18 * Ntot + idx + (-2 * s1)]));
  const double lambdaU_dD20 = p.invdxx0 * ((2.0 / 3.0) * (in[19 * Ntot + idx + (1)] - in[19 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[19 * Ntot + idx + (2)] - in[19 * Ntot + idx + (-2)]));
  const double lambdaU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (in[19 * Ntot + idx + (1 * s1)] - in[19 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[19 * Ntot + idx + (2 * s1)] - in[19 * Ntot + idx + (-2 * s1)]));
  const double g1t0 = hDD00 + 1.0;
  const double g1t1 = (f0_of_xx0*f0_of_xx0);
  const double g1t2 = (f1_of_xx1*f1_of_xx1);
  const double g1t3 = g1t1*g1t2;
  const double g1t4 = g1t3*hDD22 + g1t3;
  const double g1t5 = g1t1*(hDD01*hDD01);
  const double g1t6 = g1t1*hDD11;
  const double g1t7 = g1t1 + g1t6;
  const double g1t8 = g1t3*(hDD02*hDD02);
  const double g1t9 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g1t10 = g1t2*g1t9*(hDD12*hDD12);
  const double g1t11 = (1.0 / (-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8));
  const double g1t12 = g1t11*(-g1t10 + g1t4*g1t7);
  const double g1t13 = -f0_of_xx0*f1_of_xx1*hDD_dD021;
  const double g1t14 = f1_of_xx1__D1*hDD02;
  const double g1t15 = f0_of_xx0*g1t14;
  const double g1t16 = f1_of_xx1*g1t1;
  const double g1t17 = 2.0*f0_of_xx0;
  const double g1t18 = f1_of_xx1*hDD12;
  const double g1t19 = g1t16*hDD_dD120 + g1t17*g1t18;
  const double g1t20 = g1t13 - g1t15 + g1t19;
  const double g1t21 = -Rational_1_2*g1t20;
  const double g1t22 = f1_of_xx1*f1_of_xx1__D1;
  const double g1t23 = 2.0*g1t1;
  const double g1t24 = g1t22*g1t23;
  const double g1t25 = g1t24*hDD22 + g1t3*hDD_dD221;
  const double g1t26 = g1t24 + g1t25;
  const double g1t27 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g1t28 = f1_of_xx1*hDD02;
  const double g1t29 = f0_of_xx0*g1t28;
  const double g1t30 = g1t11*(g1t18*g1t27*hDD01 - g1t29*g1t7);
  const double g1t31 = (Rational_1_2)*g1t30;
  const double g1t32 = g1t12*g1t21 + g1t26*g1t31;
  const double g1t33 = f0_of_xx0*hDD01;
  const double g1t34 = g1t11*(g1t2*g1t27*hDD02*hDD12 - g1t33*g1t4);
  const double g1t35 = g1t1*g1t28;
  const double g1t36 = g1t1*g1t18;
  const double g1t37 = g1t11*(-g1t0*g1t36 + g1t35*hDD01);
  const double g1t38 = (Rational_1_2)*g1t37;
  const double g1t39 = g1t21*g1t34 + g1t26*g1t38;
  const double g1t40 = (1.0 / f1_of_xx1);
  const double g1t41 = f1_of_xx1__D1*g1t40;
  const double g1t42 = g1t11*(g1t0*g1t7 - g1t5);
  const double g1t43 = (Rational_1_2)*g1t42;
  const double g1t44 = g1t21*g1t30 + g1t26*g1t43 - g1t41;
  const double g1t45 = g1t0*g1t32 + g1t29*g1t44 + g1t33*g1t39;
  const double g1t46 = f1_of_xx1*hDD_dD021;
  const double g1t47 = f0_of_xx0*g1t46 + g1t15;
  const double g1t48 = g1t19 + g1t47;
  const double g1t49 = g1t1*hDD_dD110 + g1t17*hDD11;
  const double g1t50 = g1t17 + g1t49;
  const double g1t51 = g1t31*hDD_dD001 + g1t38*g1t50 + g1t43*g1t48;
  const double g1t52 = (Rational_1_2)*hDD_dD001;
  const double g1t53 = (Rational_1_2)*g1t50;
  const double g1t54 = g1t12*g1t52 + g1t31*g1t48 + g1t34*g1t53;
  const double g1t55 = (1.0 / f0_of_xx0);
  const double g1t56 = -g1t55;
  const double g1t57 = g1t11*(g1t0*g1t4 - g1t8);
  const double g1t58 = g1t34*g1t52 + g1t38*g1t48 + g1t53*g1t57 + g1t56;
  const double g1t59 = g1t29*g1t54 + g1t36*g1t58 + g1t4*g1t51;
  const double g1t60 = (Rational_1_2)*g1t57;
  const double g1t61 = g1t2*hDD22;
  const double g1t62 = g1t17*g1t61 + g1t3*hDD_dD220;
  const double g1t63 = g1t17*g1t2 + g1t62;
  const double g1t64 = g1t20*g1t60 + g1t38*g1t63;
  const double g1t65 = g1t37*g1t39;
  const double g1t66 = g1t34*g1t58;
  const double g1t67 = -g1t26;
  const double g1t68 = -g1t63;
  const double g1t69 = (Rational_1_2)*g1t34;
  const double g1t70 = g1t22 + g1t60*g1t67 + g1t68*g1t69;
  const double g1t71 = 2.0*f0_of_xx0*hDD_dD011 - g1t50;
  const double g1t72 = g1t16*hDD_dD121;
  const double g1t73 = f1_of_xx1__D1*g1t1;
  const double g1t74 = g1t73*hDD12;
  const double g1t75 = 2.0*g1t72 + 2.0*g1t74;
  const double g1t76 = g1t1*hDD_dD111;
  const double g1t77 = g1t38*g1t75 + g1t60*g1t76 + g1t69*g1t71;
  const double g1t78 = 2.0*hDD01;
  const double g1t79 = g1t78 - hDD_dD001;
  const double g1t80 = g1t17*hDD_dD010 + g1t79;
  const double g1t81 = f1_of_xx1*hDD_dD020;
  const double g1t82 = g1t17*g1t81 + 2.0*g1t28;
  const double g1t83 = g1t38*g1t82 + g1t60*g1t80 + g1t69*hDD_dD000;
  const double g1t84 = (Rational_1_2)*g1t12;
  const double g1t85 = g1t30*g1t64 + g1t43*g1t70 + g1t60*g1t77 + g1t65 + g1t66 + g1t83*g1t84;
  const double g1t86 = g1t20*g1t69 + g1t31*g1t63;
  const double g1t87 = g1t20*g1t38 + g1t43*g1t63 + g1t56;
  const double g1t88 = g1t0*g1t86 + g1t29*g1t87 + g1t33*g1t64;
  const double g1t89 = g1t31*hDD_dD000 + g1t38*g1t80 + g1t43*g1t82;
  const double g1t90 = g1t31*g1t82 + g1t69*g1t80 + g1t84*hDD_dD000;
  const double g1t91 = g1t29*g1t90 + g1t36*g1t83 + g1t4*g1t89;
  const double g1t92 = f0_of_xx0*g1t2;
  const double g1t93 = g1t67*g1t69 + g1t68*g1t84 + g1t92;
  const double g1t94 = f0_of_xx0 + g1t31*g1t75 + g1t69*g1t76 + g1t71*g1t84;
  const double g1t95 = g1t30*g1t86 + g1t32*g1t37 + g1t34*g1t54 + g1t43*g1t93 + g1t60*g1t94 + g1t84*g1t90;
  const double g1t96 = g1t31*g1t68 + g1t38*g1t67;
  const double g1t97 = g1t0*g1t93 + g1t29*g1t96 + g1t33*g1t70;
  const double g1t98 = g1t29*g1t86 + g1t36*g1t64 + g1t4*g1t87;
  const double g1t99 = g1t31*g1t71 + g1t38*g1t76 + g1t43*g1t75;
  const double g1t100 = g1t30*g1t87 + g1t34*g1t51 + g1t37*g1t44 + g1t43*g1t96 + g1t60*g1t99 + g1t84*g1t89;
  const double g1t101 = g1t29*g1t93 + g1t36*g1t70 + g1t4*g1t96;
  const double g1t102 = 2.0*g1t87;
  const double g1t103 = g1t33*g1t93 + g1t36*g1t96 + g1t7*g1t70;
  const double g1t104 = g1t29*g1t32 + g1t36*g1t39 + g1t4*g1t44;
  const double g1t105 = g1t104*g1t51;
  const double g1t106 = g1t0*g1t54 + g1t29*g1t51 + g1t33*g1t58;
  const double g1t107 = g1t106*g1t32;
  const double g1t108 = g1t45*g1t54;
  const double g1t109 = g1t0*g1t94 + g1t29*g1t99 + g1t33*g1t77;
  const double g1t110 = g1t39*g1t7;
  const double g1t111 = g1t110 + g1t32*g1t33 + g1t36*g1t44;
  const double g1t112 = g1t111*g1t58;
  const double g1t113 = g1t29*g1t94 + g1t36*g1t77 + g1t4*g1t99;
  const double g1t114 = 2.0*g1t89;
  const double g1t115 = g1t33*g1t86 + g1t36*g1t87 + g1t64*g1t7;
  const double g1t116 = g1t0*g1t90 + g1t29*g1t89 + g1t33*g1t83;
  const double g1t117 = 2.0*g1t51;
  const double g1t118 = g1t86*g1t88;
  const double g1t119 = (Rational_1_2)*lambdaU2;
  const double g1t120 = (f1_of_xx1*f1_of_xx1*f1_of_xx1);
  const double g1t121 = g1t1*g1t120;
  const double g1t122 = f0_of_xx0*g1t18;
  const double g1t123 = -g1t122 - g1t13;
  const double g1t124 = -g1t122 - g1t15;
  const double g1t125 = g1t35 + g1t72;
  const double g1t126 = g1t72 + g1t74;
  const double g1t127 = (f1_of_xx1__D1*f1_of_xx1__D1);
  const double g1t128 = f1_of_xx1__DD11*g1t40 - g1t127/g1t2;
  const double g1t129 = f0_of_xx0*g1t81 + g1t28;
  const double g1t130 = f0_of_xx0*f1_of_xx1;
  const double g1t131 = g1t123*g1t55;
  const double g1t132 = f0_of_xx0*f1_of_xx1__D1;
  const double g1t133 = g1t22*g1t33 + g1t92*hDD00 - g1t92*hDD22;
  const double g1t134 = g1t133*g1t41;
  const double g1t135 = f0_of_xx0*hDD00 - f0_of_xx0*hDD11 + f0_of_xx0*hDD_dD011;
  const double g1t136 = -g1t1*g1t22*hDD22 + g1t22*g1t6 + g1t3*hDD01;
  const double g1t137 = g1t133*g1t55;
  const double g1t138 = g1t92*hDD_dD000;
  const double g1t139 = f0_of_xx0*hDD_dD010;
  const double g1t140 = g1t139 + hDD01;
  const double g1t141 = (Rational_1_2)*g1t29;
  const double g1t142 = g1t55*lambdaU0;
  const double g1t143 = g1t17*hDD01;
  const double g1t144 = 2.0*g1t44;
  const double g1t145 = g1t7*g1t77;
  const double g1t146 = 2.0*g1t99;
  const double g1t147 = g1t58*g1t7;
  const double g1t148 = 2.0*g1t32;
  const double g1t149 = 2.0*g1t103;
  const double g1t150 = g1t147 + g1t33*g1t54 + g1t36*g1t51;
  const double g1t151 = 2.0*g1t94;
  const double g1t152 = g1t33*g1t90 + g1t36*g1t89 + g1t7*g1t83;
  const double g1t153 = 2.0*g1t54;
  const double g1t154 = g1t1*g1t78 + g1t76;
  const double g1t155 = g1t27*hDD_dD110;
  const double g1t156 = 2.0*g1t41;
  const double g1t157 = g1t1*hDD_dDD1101;
  const double g1t158 = g1t154*g1t55;
  const double g1t159 = g1t127*g1t23*g1t40*hDD12;
  const double g1t160 = 3.0*g1t39;
  const double g1t161 = 3.0*g1t145 + 3.0*g1t33*g1t94 + 3.0*g1t36*g1t99;
  const double g1t162 = 3.0*g1t150;
  double a_f0_of_xx0 = S[2 * Ntot + idx] * (-f1_of_xx1*g1t69*hDD_dDD0201 + g1t2*g1t38*g1t79 - g1t38*(2.0*f1_of_xx1*f1_of_xx1__D1*hDD00 + f1_of_xx1*f1_of_xx1__D1*hDD_dD011 + g1t2*hDD_dD001) - g1t60*(f1_of_xx1*hDD_dDD0211 + 2.0*f1_of_xx1__D1*hDD_dD021 + f1_of_xx1__DD11*hDD02));
  double a_f1_of_xx1 = S[2 * Ntot + idx] * (-f1_of_xx1__D1*g1t135*g1t38 - g1t0*g1t119 - g1t38*(2.0*f0_of_xx0*f1_of_xx1__D1*hDD00 + f0_of_xx0*f1_of_xx1__D1*hDD_dD011 + f1_of_xx1__DD11*g1t33) - g1t60*(f0_of_xx0*hDD_dDD0211 + g1t1*hDD_dD020) - g1t69*(f0_of_xx0*hDD_dDD0201 + hDD_dD021));
  double a_f1_of_xx1__D1 = S[2 * Ntot + idx] * (-2.0*f0_of_xx0*g1t60*hDD_dD021 - f1_of_xx1*g1t135*g1t38 - g1t119*hDD01 + 2.0*g1t3*g1t43*g1t55*hDD12 - g1t38*(2.0*f0_of_xx0*f1_of_xx1*hDD00 + f0_of_xx0*f1_of_xx1*hDD_dD011) - g1t69*hDD02);
  double a_f1_of_xx1__DD11 = S[2 * Ntot + idx] * (-f0_of_xx0*g1t60*hDD02 - f1_of_xx1*g1t33*g1t38);
  double a_g1t0 = S[2 * Ntot + idx] * (-f1_of_xx1*g1t119);
  double a_g1t1 = S[2 * Ntot + idx] * (-f1_of_xx1*g1t60*hDD_dD020);
  double a_g1t100 = S[2 * Ntot + idx] * (g1t97 + g1t98);
  double a_g1t101 = S[2 * Ntot + idx] * (g1t102*g1t42 + g1t114*g1t30 + g1t117*g1t37);
  double a_g1t102 = S[2 * Ntot + idx] * (g1t101*g1t42 + g1t104*g1t37 + g1t30*g1t98);
  double a_g1t103 = S[2 * Ntot + idx] * (g1t30*g1t83 + g1t37*g1t58 + g1t42*g1t64);
  double a_g1t104 = S[2 * Ntot + idx] * (g1t102*g1t37 + g1t114*g1t34 + g1t30*g1t83 + g1t37*g1t58 + g1t42*g1t64);
  double a_g1t105 = S[2 * Ntot + idx] * (2.0*g1t57);
  double a_g1t106 = S[2 * Ntot + idx] * (g1t12*g1t64 + g1t30*g1t70 + g1t34*g1t39 + g1t34*g1t86 + g1t37*g1t93);
  double a_g1t107 = S[2 * Ntot + idx] * (g1t57);
  double a_g1t108 = S[2 * Ntot + idx] * (g1t57);
  double a_g1t109 = S[2 * Ntot + idx] * (g1t34*g1t64 + g1t37*g1t70 + g1t39*g1t57);
  double a_g1t111 = S[2 * Ntot + idx] * (g1t34*g1t83 + g1t37*g1t64);
  double a_g1t112 = S[2 * Ntot + idx] * (g1t57);
  double a_g1t113 = S[2 * Ntot + idx] * (g1t34*g1t83 + g1t37*g1t64 + g1t57*g1t58);
  double a_g1t114 = S[2 * Ntot + idx] * (g1t101*g1t30 + g1t104*g1t34 + g1t12*g1t98);
  double a_g1t115 = S[2 * Ntot + idx] * (g1t12*g1t83 + g1t30*g1t64 + g1t34*g1t58);
  double a_g1t116 = S[2 * Ntot + idx] * (g1t12*g1t86 + g1t30*g1t93 + g1t32*g1t34);
  double a_g1t117 = S[2 * Ntot + idx] * (g1t101*g1t37 + g1t34*g1t98);
  double a_g1t118 = S[2 * Ntot + idx] * (2.0*g1t30);
  double a_g1t119 = S[2 * Ntot + idx] * (-f1_of_xx1*g1t0 - f1_of_xx1__D1*hDD01);
  double a_g1t12 = S[2 * Ntot + idx] * (g1t106*g1t64 + g1t114*g1t98 + g1t115*g1t83 + g1t116*g1t86 + g1t59*g1t83 + g1t87*g1t88 + g1t88*g1t90 + g1t90*g1t91);
  double a_g1t120 = S[2 * Ntot + idx] * (g1t17*g1t43*hDD02);
  double a_g1t121 = S[2 * Ntot + idx] * (-g1t43*(-2.0*g1t55*hDD02 + hDD_dD020));
  double a_g1t122 = S[2 * Ntot + idx] * ((Rational_1_2)*lambdaU_dD10);
  double a_g1t123 = S[2 * Ntot + idx] * (-g1t22*g1t43 + g1t41*g1t60);
  double a_g1t124 = S[2 * Ntot + idx] * (-g1t22*g1t43);
  double a_g1t125 = S[2 * Ntot + idx] * (g1t55*g1t60);
  double a_g1t126 = S[2 * Ntot + idx] * (g1t55*g1t60);
  double a_g1t127 = S[2 * Ntot + idx] * (-g1t33*g1t38);
  double a_g1t128 = S[2 * Ntot + idx] * (g1t29*g1t60);
  double a_g1t129 = S[2 * Ntot + idx] * (g1t41*g1t69 + g1t55*g1t84);
  double a_g1t130 = S[2 * Ntot + idx] * (g1t69*hDD_dD120 - g1t69*hDD_dDD0201 - g1t84*hDD_dDD0200);
  double a_g1t131 = S[2 * Ntot + idx] * (3.0*g1t69);
  double a_g1t132 = S[2 * Ntot + idx] * (-g1t69*hDD_dD020);
  double a_g1t134 = S[2 * Ntot + idx] * (3.0*g1t38);
  double a_g1t135 = S[2 * Ntot + idx] * (-f1_of_xx1*f1_of_xx1__D1*g1t38);
  double a_g1t136 = S[2 * Ntot + idx] * (g1t38*g1t55);
  double a_g1t137 = S[2 * Ntot + idx] * (3.0*g1t31);
  double a_g1t138 = S[2 * Ntot + idx] * (-2.0*g1t31);
  double a_g1t139 = S[2 * Ntot + idx] * (-g1t22*g1t31);
  double a_g1t14 = S[2 * Ntot + idx] * (-g1t69);
  double a_g1t140 = S[2 * Ntot + idx] * (-g1t22*g1t31);
  double a_g1t141 = S[2 * Ntot + idx] * (g1t142 + g1t41*g1t55*lambdaU1 + lambdaU_dD00);
  double a_g1t142 = S[2 * Ntot + idx] * (g1t141);
  double a_g1t17 = S[2 * Ntot + idx] * (g1t120*g1t43*hDD02);
  double a_g1t18 = S[2 * Ntot + idx] * (-g1t69);
  double a_g1t19 = S[2 * Ntot + idx] * (g1t55*g1t69);
  double a_g1t2 = S[2 * Ntot + idx] * (f0_of_xx0*g1t38*g1t79 - f0_of_xx0*g1t38*hDD_dD001 - g1t31*hDD00);
  double a_g1t22 = S[2 * Ntot + idx] * (-g1t139*g1t31 - g1t140*g1t31 - g1t43*(g1t123 + g1t124));
  double a_g1t25 = S[2 * Ntot + idx] * (g1t38*g1t55);
  double a_g1t28 = S[2 * Ntot + idx] * (-g1t55*g1t84);
  double a_g1t29 = S[2 * Ntot + idx] * (g1t128*g1t60);
  double a_g1t3 = S[2 * Ntot + idx] * (2.0*f1_of_xx1__D1*g1t43*g1t55*hDD12);
  double a_g1t30 = S[2 * Ntot + idx] * (g1t101*g1t114 + g1t102*g1t98 + g1t103*g1t83 + g1t104*g1t83 + g1t106*g1t70 + g1t115*g1t64 + g1t116*g1t93 + 2.0*g1t118 + g1t45*g1t64 + g1t59*g1t64 + g1t86*g1t91 + g1t87*g1t97 + g1t88*g1t96 + g1t90*g1t97 + g1t90*g1t98);
  double a_g1t31 = S[2 * Ntot + idx] * (3.0*g1t137 - 2.0*g1t138 - g1t139*g1t22 - g1t140*g1t22 - g1t2*hDD00 + g1t55*g1t62 - g1t61 + g1t92*hDD_dD220);
  double a_g1t32 = S[2 * Ntot + idx] * (g1t116*g1t34 + g1t37*g1t88);
  double a_g1t33 = S[2 * Ntot + idx] * (-g1t38*(f1_of_xx1*f1_of_xx1__DD11 + g1t127));
  double a_g1t34 = S[2 * Ntot + idx] * (g1t104*g1t114 + g1t106*g1t39 + g1t106*g1t86 + g1t109*g1t64 + g1t111*g1t83 + g1t113*g1t83 + g1t115*g1t58 + g1t116*g1t32 + g1t117*g1t98 + g1t44*g1t88 + g1t45*g1t87 + g1t45*g1t90 + g1t54*g1t88 + g1t54*g1t91 + g1t58*g1t59 + g1t59*g1t90);
  double a_g1t37 = S[2 * Ntot + idx] * (g1t101*g1t117 + g1t102*g1t104 + g1t103*g1t58 + g1t104*g1t58 + g1t106*g1t93 + g1t109*g1t70 + g1t111*g1t64 + g1t113*g1t64 + g1t32*g1t88 + g1t39*g1t45 + g1t44*g1t97 + g1t45*g1t86 + g1t45*g1t96 + g1t54*g1t97 + g1t54*g1t98 + g1t59*g1t86);
  double a_g1t38 = S[2 * Ntot + idx] * (-2.0*f0_of_xx0*f1_of_xx1*f1_of_xx1__D1*hDD00 - f0_of_xx0*f1_of_xx1*f1_of_xx1__D1*hDD_dD011 + f0_of_xx0*g1t2*g1t79 - f0_of_xx0*g1t2*hDD_dD001 - f1_of_xx1*f1_of_xx1__D1*g1t135 + 3.0*g1t134 + g1t136*g1t55 + g1t25*g1t55 + g1t33*(-f1_of_xx1*f1_of_xx1__DD11 - g1t127) + g1t92*hDD_dD221);
  double a_g1t39 = S[2 * Ntot + idx] * (g1t106*g1t34 + g1t109*g1t57 + g1t37*g1t45);
  double a_g1t4 = S[2 * Ntot + idx] * ((Rational_1_2)*g1t40*g1t55*lambdaU_dD20);
  double a_g1t40 = S[2 * Ntot + idx] * ((Rational_1_2)*g1t4*g1t55*lambdaU_dD20);
  double a_g1t41 = S[2 * Ntot + idx] * (g1t129*g1t69 + g1t141*g1t55*lambdaU1 - g1t60*(-g1t123 - g1t47));
  double a_g1t42 = S[2 * Ntot + idx] * (g1t101*g1t102 + g1t103*g1t64 + g1t104*g1t64 + g1t45*g1t70 + g1t86*g1t97 + g1t86*g1t98 + g1t88*g1t93 + g1t96*g1t97);
  double a_g1t43 = S[2 * Ntot + idx] * (g1t120*g1t17*hDD02 - g1t121*hDD_dD020 - g1t123*g1t22 - g1t124*g1t22 + g1t55*(2.0*f1_of_xx1__D1*g1t3*hDD12 + 2.0*g1t121*hDD02));
  double a_g1t44 = S[2 * Ntot + idx] * (g1t34*g1t88 + g1t37*g1t97 + g1t45*g1t57);
  double a_g1t45 = S[2 * Ntot + idx] * (g1t30*g1t64 + g1t34*g1t87 + g1t34*g1t90 + g1t37*g1t39 + g1t37*g1t86 + g1t37*g1t96 + g1t42*g1t70 + g1t44*g1t57 + g1t85);
  double a_g1t46 = S[2 * Ntot + idx] * (-g1t69);
  double a_g1t47 = S[2 * Ntot + idx] * (g1t41*g1t60 + g1t55*g1t69);
  double a_g1t54 = S[2 * Ntot + idx] * (g1t34*(g1t88 + g1t91) + g1t37*(g1t97 + g1t98) + g1t57*g1t59);
  double a_g1t55 = S[2 * Ntot + idx] * (g1t141*g1t41*lambdaU1 + g1t19*g1t69 + g1t31*g1t62 - g1t38*(-g1t136 - g1t25) + (Rational_1_2)*g1t4*g1t40*lambdaU_dD20 - g1t43*(-2.0*f1_of_xx1__D1*g1t3*hDD12 - 2.0*g1t121*hDD02) + g1t47*g1t69 - g1t60*(-g1t125 - g1t126) - g1t84*(-g1t129 + g1t28));
  double a_g1t57 = S[2 * Ntot + idx] * (2.0*g1t105 + g1t107 + g1t108 + g1t109*g1t39 + g1t112 + g1t113*g1t58 + g1t44*g1t45 + g1t54*g1t59);
  double a_g1t58 = S[2 * Ntot + idx] * (g1t113*g1t57 + g1t34*(g1t115 + g1t59) + g1t37*(g1t103 + g1t104));
  double a_g1t59 = S[2 * Ntot + idx] * (g1t12*g1t83 + g1t30*g1t64 + g1t34*g1t58 + g1t34*g1t90 + g1t37*g1t86 + g1t54*g1t57 + g1t85);
  double a_g1t60 = S[2 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1*hDD_dDD0211 - 2.0*f0_of_xx0*f1_of_xx1__D1*hDD_dD021 - f0_of_xx0*f1_of_xx1__DD11*hDD02 - f1_of_xx1*g1t1*hDD_dD020 + g1t123*g1t41 + g1t125*g1t55 + g1t126*g1t55 + g1t128*g1t29 + g1t41*g1t47);
  double a_g1t61 = S[2 * Ntot + idx] * (-g1t31);
  double a_g1t62 = S[2 * Ntot + idx] * (g1t31*g1t55);
  double a_g1t64 = S[2 * Ntot + idx] * (g1t106*g1t12 + g1t109*g1t34 + g1t30*g1t45 + g1t30*(g1t115 + g1t59) + g1t37*(g1t111 + g1t113) + g1t42*(g1t103 + g1t104));
  double a_g1t69 = S[2 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1*hDD_dDD0201 - f1_of_xx1*hDD_dD021 - f1_of_xx1__D1*hDD02 + g1t129*g1t41 + g1t130*hDD_dD120 - g1t130*hDD_dDD0201 + 3.0*g1t131 - g1t132*hDD_dD020 - g1t14 - g1t18 + g1t19*g1t55 - g1t46 + g1t47*g1t55);
  double a_g1t70 = S[2 * Ntot + idx] * (g1t106*g1t30 + g1t109*g1t37 + g1t42*g1t45);
  double a_g1t79 = S[2 * Ntot + idx] * (f0_of_xx0*g1t2*g1t38);
  double a_g1t81 = S[2 * Ntot + idx] * (-g1t84);
  double a_g1t83 = S[2 * Ntot + idx] * (g1t12*(g1t115 + g1t59) + g1t30*(g1t103 + g1t104) + g1t34*(g1t111 + g1t113));
  double a_g1t84 = S[2 * Ntot + idx] * (g1t129*g1t55 - g1t130*hDD_dDD0200 - g1t28*g1t55 - g1t81);
  double a_g1t85 = S[2 * Ntot + idx] * (g1t45 + g1t59);
  double a_g1t86 = S[2 * Ntot + idx] * (g1t106*g1t34 + g1t116*g1t12 + g1t30*g1t91 + g1t37*(g1t45 + g1t59) + g1t42*(g1t97 + g1t98));
  double a_g1t87 = S[2 * Ntot + idx] * (g1t12*g1t88 + g1t30*g1t97 + g1t34*g1t45);
  double a_g1t88 = S[2 * Ntot + idx] * (g1t12*g1t87 + g1t12*g1t90 + g1t30*g1t96 + g1t32*g1t37 + g1t34*g1t44 + g1t34*g1t54 + g1t42*g1t93 + g1t95);
  double a_g1t90 = S[2 * Ntot + idx] * (g1t12*(g1t88 + g1t91) + g1t30*(g1t97 + g1t98) + g1t34*(g1t45 + g1t59));
  double a_g1t91 = S[2 * Ntot + idx] * (g1t12*g1t90 + g1t30*g1t86 + g1t34*g1t54 + g1t95);
  double a_g1t92 = S[2 * Ntot + idx] * (g1t31*hDD_dD220 + g1t38*hDD_dD221);
  double a_g1t93 = S[2 * Ntot + idx] * (g1t106*g1t37 + g1t116*g1t30 + g1t42*g1t88);
  double a_g1t95 = S[2 * Ntot + idx] * (g1t88 + g1t91);
  double a_g1t96 = S[2 * Ntot + idx] * (g1t30*g1t88 + g1t37*g1t45 + g1t42*g1t97);
  double a_g1t97 = S[2 * Ntot + idx] * (g1t100 + g1t30*g1t87 + g1t30*g1t90 + g1t37*g1t44 + g1t37*g1t54 + g1t42*g1t86 + g1t42*g1t96);
  double a_g1t98 = S[2 * Ntot + idx] * (g1t100 + g1t102*g1t30 + g1t114*g1t12 + g1t117*g1t34 + g1t30*g1t90 + g1t37*g1t54 + g1t42*g1t86);
  double a_hDD00 = S[2 * Ntot + idx] * (-2.0*f0_of_xx0*f1_of_xx1*f1_of_xx1__D1*g1t38 - g1t2*g1t31);
  double a_hDD01 = S[2 * Ntot + idx] * (-f1_of_xx1__D1*g1t119);
  double a_hDD02 = S[2 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1__DD11*g1t60 - f1_of_xx1__D1*g1t69 - g1t43*(-g1t120*g1t17 - 2.0*g1t121*g1t55));
  double a_hDD12 = S[2 * Ntot + idx] * (2.0*f1_of_xx1__D1*g1t3*g1t43*g1t55);
  double a_hDD_dD001 = S[2 * Ntot + idx] * (-f0_of_xx0*g1t2*g1t38);
  double a_hDD_dD011 = S[2 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1*f1_of_xx1__D1*g1t38);
  double a_hDD_dD020 = S[2 * Ntot + idx] * (-f1_of_xx1*g1t1*g1t60 - g1t121*g1t43 - g1t132*g1t69);
  double a_hDD_dD021 = S[2 * Ntot + idx] * (-2.0*f0_of_xx0*f1_of_xx1__D1*g1t60 - f1_of_xx1*g1t69);
  double a_hDD_dD120 = S[2 * Ntot + idx] * (g1t130*g1t69);
  double a_hDD_dD220 = S[2 * Ntot + idx] * (g1t31*g1t92);
  double a_hDD_dD221 = S[2 * Ntot + idx] * (g1t38*g1t92);
  double a_hDD_dDD0200 = S[2 * Ntot + idx] * (-g1t130*g1t84);
  double a_hDD_dDD0201 = S[2 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1*g1t69 - g1t130*g1t69);
  double a_hDD_dDD0211 = S[2 * Ntot + idx] * (-f0_of_xx0*f1_of_xx1*g1t60);
  double a_lambdaU1 = S[2 * Ntot + idx] * (g1t141*g1t41*g1t55);
  double a_lambdaU_dD00 = S[2 * Ntot + idx] * (g1t141);
  double a_lambdaU_dD10 = S[2 * Ntot + idx] * ((Rational_1_2)*g1t122);
  double a_lambdaU_dD20 = S[2 * Ntot + idx] * ((Rational_1_2)*g1t4*g1t40*g1t55);
  a_f0_of_xx0 += S[3 * Ntot + idx] * (-2.0*f1_of_xx1__D1*g1t31*hDD12 + hDD12*lambdaU_dD21);
  a_f1_of_xx1__D1 += S[3 * Ntot + idx] * (-2.0*f0_of_xx0*g1t31*hDD12);
  a_g1t1 += S[3 * Ntot + idx] * (-g1t60*hDD_dDD1111 - g1t84*hDD_dDD1100);
  a_g1t100 += S[3 * Ntot + idx] * (2.0*g1t110 + g1t143*g1t32 + g1t144*g1t36);
  a_g1t103 += S[3 * Ntot + idx] * (g1t117*g1t30);
  a_g1t104 += S[3 * Ntot + idx] * (g1t37*g1t99 + g1t42*g1t44);
  a_g1t105 += S[3 * Ntot + idx] * (g1t30);
  a_g1t106 += S[3 * Ntot + idx] * (g1t12*g1t54 + g1t34*g1t94);
  a_g1t107 += S[3 * Ntot + idx] * (g1t30);
  a_g1t108 += S[3 * Ntot + idx] * (g1t30);
  a_g1t109 += S[3 * Ntot + idx] * (g1t32*g1t37 + g1t34*g1t54 + g1t57*g1t94);
  double a_g1t110 = S[3 * Ntot + idx] * (2.0*g1t100);
  a_g1t111 += S[3 * Ntot + idx] * (g1t117*g1t34 + g1t144*g1t37 + g1t146*g1t57 + g1t160*g1t42 + 3.0*g1t37*g1t77);
  a_g1t112 += S[3 * Ntot + idx] * (3.0*g1t30);
  a_g1t113 += S[3 * Ntot + idx] * (g1t34*g1t51 + g1t37*g1t44 + g1t57*g1t99);
  a_g1t115 += S[3 * Ntot + idx] * (g1t117*g1t12 + g1t144*g1t30 + g1t146*g1t34 + g1t148*g1t42 + g1t151*g1t37 + g1t153*g1t30);
  a_g1t117 += S[3 * Ntot + idx] * (g1t103*g1t30 + g1t111*g1t34 + g1t115*g1t12 + g1t36*g1t95);
  a_g1t12 += S[3 * Ntot + idx] * (g1t106*g1t54 + g1t115*g1t117 + g1t152*g1t153 + g1t162*g1t58 + g1t51*g1t59);
  a_g1t124 += S[3 * Ntot + idx] * (-g1t17*g1t38);
  a_g1t125 += S[3 * Ntot + idx] * (g1t156*g1t38);
  a_g1t126 += S[3 * Ntot + idx] * (g1t156*g1t38);
  a_g1t128 += S[3 * Ntot + idx] * (2.0*g1t36*g1t38);
  a_g1t132 += S[3 * Ntot + idx] * (-6.0*g1t31*hDD12);
  a_g1t135 += S[3 * Ntot + idx] * (-g1t17*g1t60);
  a_g1t136 += S[3 * Ntot + idx] * (g1t156*g1t43);
  a_g1t140 += S[3 * Ntot + idx] * (-g1t17*g1t69);
  a_g1t142 += S[3 * Ntot + idx] * (g1t7);
  double a_g1t143 = S[3 * Ntot + idx] * (g1t100*g1t32 + g1t54*g1t95 - g1t69 + g1t85*g1t94);
  double a_g1t144 = S[3 * Ntot + idx] * (g1t100*g1t36 + g1t111*g1t37 + g1t115*g1t30);
  double a_g1t145 = S[3 * Ntot + idx] * (2.0*g1t85);
  double a_g1t146 = S[3 * Ntot + idx] * (g1t111*g1t57 + g1t115*g1t34 + g1t36*g1t85);
  double a_g1t147 = S[3 * Ntot + idx] * (2.0*g1t95);
  double a_g1t148 = S[3 * Ntot + idx] * (g1t115*g1t42 + g1t150*g1t37 + g1t152*g1t30);
  double a_g1t149 = S[3 * Ntot + idx] * (g1t37*g1t99 + g1t42*g1t44);
  double a_g1t150 = S[3 * Ntot + idx] * (g1t148*g1t37 + g1t151*g1t57 + g1t153*g1t34 + g1t160*g1t30);
  double a_g1t151 = S[3 * Ntot + idx] * (g1t115*g1t37 + g1t150*g1t57 + g1t152*g1t34);
  double a_g1t152 = S[3 * Ntot + idx] * (g1t12*g1t153 + g1t148*g1t30 + g1t151*g1t34);
  double a_g1t153 = S[3 * Ntot + idx] * (g1t115*g1t30 + g1t12*g1t152 + g1t150*g1t34);
  double a_g1t154 = S[3 * Ntot + idx] * (-g1t22*g1t43);
  double a_g1t155 = S[3 * Ntot + idx] * (-g1t2*g1t43 - g1t60);
  double a_g1t156 = S[3 * Ntot + idx] * (g1t125*g1t38 + g1t126*g1t38 + g1t136*g1t43 + g1t19*g1t31);
  double a_g1t157 = S[3 * Ntot + idx] * (-2.0*g1t69);
  double a_g1t158 = S[3 * Ntot + idx] * (4.0*g1t69);
  double a_g1t159 = S[3 * Ntot + idx] * (-2.0*g1t38);
  double a_g1t160 = S[3 * Ntot + idx] * (g1t111*g1t42 + g1t150*g1t30);
  double a_g1t161 = S[3 * Ntot + idx] * (g1t57*g1t77 + g1t65 + g1t66);
  double a_g1t162 = S[3 * Ntot + idx] * (g1t12*g1t58 + g1t34*g1t77);
  a_g1t17 += S[3 * Ntot + idx] * (-g1t124*g1t38 - g1t135*g1t60 - g1t69*(g1t140 + hDD_dD111) - g1t84*hDD_dD110);
  a_g1t19 += S[3 * Ntot + idx] * (g1t156*g1t31);
  a_g1t2 += S[3 * Ntot + idx] * (-g1t155*g1t43);
  a_g1t22 += S[3 * Ntot + idx] * (-g1t154*g1t43);
  double a_g1t23 = S[3 * Ntot + idx] * (-g1t60*hDD_dD011 - g1t69*hDD_dD010);
  a_g1t30 += S[3 * Ntot + idx] * (g1t103*g1t117 + g1t105 + g1t107 + g1t108 + 3.0*g1t112 + g1t115*g1t144 + g1t115*g1t153 + g1t148*g1t152 + g1t150*g1t160 + g1t44*g1t59);
  a_g1t31 += S[3 * Ntot + idx] * (-2.0*f0_of_xx0*f1_of_xx1__D1*hDD12 - 6.0*g1t132*hDD12 + g1t156*g1t19 + 2.0*g1t73*hDD_dD120);
  a_g1t32 += S[3 * Ntot + idx] * (g1t100*g1t143 + g1t109*g1t37 + g1t42*g1t45);
  a_g1t33 += S[3 * Ntot + idx] * (-lambdaU1 + lambdaU_dD01);
  a_g1t34 += S[3 * Ntot + idx] * (g1t106*g1t94 + g1t109*g1t54 + g1t111*g1t117 + g1t113*g1t51 + g1t115*g1t146 + g1t150*g1t153 + g1t151*g1t152 + g1t162*g1t77 + g1t59*g1t99);
  double a_g1t36 = S[3 * Ntot + idx] * (g1t100*g1t144 + g1t117*g1t95 + 2.0*g1t128*g1t38 + g1t146*g1t85);
  a_g1t37 += S[3 * Ntot + idx] * (g1t104*g1t99 + g1t109*g1t32 + g1t111*g1t144 + 3.0*g1t111*g1t77 + g1t113*g1t44 + g1t115*g1t151 + g1t148*g1t150 + g1t149*g1t99 + g1t45*g1t94);
  a_g1t38 += S[3 * Ntot + idx] * (-g1t124*g1t17 + g1t125*g1t156 + g1t126*g1t156 + 2.0*g1t128*g1t36 - 2.0*g1t159);
  a_g1t42 += S[3 * Ntot + idx] * (g1t104*g1t44 + g1t111*g1t160 + g1t115*g1t148 + g1t149*g1t44 + g1t32*g1t45);
  a_g1t43 += S[3 * Ntot + idx] * (g1t136*g1t156 - g1t154*g1t22 - g1t155*g1t2);
  a_g1t44 += S[3 * Ntot + idx] * (g1t113*g1t37 + g1t30*g1t59 + g1t42*(g1t104 + g1t149));
  a_g1t45 += S[3 * Ntot + idx] * (g1t32*g1t42 + g1t37*g1t94);
  double a_g1t49 = S[3 * Ntot + idx] * (2.0*g1t55*g1t84);
  double a_g1t51 = S[3 * Ntot + idx] * (g1t113*g1t34 + g1t12*g1t59);
  a_g1t54 += S[3 * Ntot + idx] * (g1t106*g1t12 + g1t109*g1t34 + g1t143*g1t95);
  a_g1t55 += S[3 * Ntot + idx] * (2.0*g1t49*g1t84 + g1t7*lambdaU_dD11);
  a_g1t57 += S[3 * Ntot + idx] * (g1t109*g1t94 + g1t111*g1t146 + g1t113*g1t99 + g1t150*g1t151 + g1t161*g1t77);
  a_g1t58 += S[3 * Ntot + idx] * (g1t12*g1t162);
  a_g1t59 += S[3 * Ntot + idx] * (g1t12*g1t51 + g1t30*g1t44 + g1t34*g1t99);
  a_g1t60 += S[3 * Ntot + idx] * (-g1t1*hDD_dDD1111 - g1t135*g1t17 - g1t155 - g1t23*hDD_dD011);
  double a_g1t65 = S[3 * Ntot + idx] * (g1t161);
  double a_g1t66 = S[3 * Ntot + idx] * (g1t161);
  a_g1t69 += S[3 * Ntot + idx] * (-g1t140*g1t17 - g1t143 - 2.0*g1t157 + 4.0*g1t158 - g1t17*hDD_dD111 - g1t23*hDD_dD010);
  double a_g1t7 = S[3 * Ntot + idx] * (g1t142 + g1t55*lambdaU_dD11);
  double a_g1t73 = S[3 * Ntot + idx] * (2.0*g1t31*hDD_dD120);
  double a_g1t77 = S[3 * Ntot + idx] * (3.0*g1t111*g1t37 + g1t161*g1t57 + g1t162*g1t34);
  a_g1t84 += S[3 * Ntot + idx] * (-g1t1*hDD_dDD1100 - g1t17*hDD_dD110 + 2.0*g1t49*g1t55 - 4.0*hDD11);
  a_g1t85 += S[3 * Ntot + idx] * (g1t143*g1t94 + 2.0*g1t145 + g1t146*g1t36);
  double a_g1t94 = S[3 * Ntot + idx] * (g1t106*g1t34 + g1t109*g1t57 + g1t143*g1t85 + g1t37*g1t45);
  a_g1t95 += S[3 * Ntot + idx] * (g1t117*g1t36 + g1t143*g1t54 + 2.0*g1t147);
  double a_g1t99 = S[3 * Ntot + idx] * (g1t113*g1t57 + g1t34*g1t59 + g1t37*(g1t104 + g1t149));
  double a_hDD11 = S[3 * Ntot + idx] * (-4.0*g1t84);
  a_hDD12 += S[3 * Ntot + idx] * (-2.0*f0_of_xx0*f1_of_xx1__D1*g1t31 + f0_of_xx0*lambdaU_dD21 - 6.0*g1t132*g1t31);
  double a_hDD_dD010 = S[3 * Ntot + idx] * (-g1t23*g1t69);
  a_hDD_dD011 += S[3 * Ntot + idx] * (-g1t23*g1t60);
  double a_hDD_dD110 = S[3 * Ntot + idx] * (-g1t17*g1t84);
  double a_hDD_dD111 = S[3 * Ntot + idx] * (-g1t17*g1t69);
  a_hDD_dD120 += S[3 * Ntot + idx] * (2.0*g1t31*g1t73);
  double a_hDD_dDD1100 = S[3 * Ntot + idx] * (-g1t1*g1t84);
  double a_hDD_dDD1111 = S[3 * Ntot + idx] * (-g1t1*g1t60);
  a_lambdaU1 += S[3 * Ntot + idx] * (-g1t33);
  double a_lambdaU_dD01 = S[3 * Ntot + idx] * (g1t33);
  double a_lambdaU_dD11 = S[3 * Ntot + idx] * (g1t55*g1t7);
  double a_lambdaU_dD21 = S[3 * Ntot + idx] * (f0_of_xx0*hDD12);
  a_g1t150 += a_g1t162 * (3.0);
  a_g1t145 += a_g1t161 * (3.0);
  a_g1t33 += a_g1t161 * (3.0*g1t94);
  a_g1t36 += a_g1t161 * (3.0*g1t99);
  a_g1t94 += a_g1t161 * (3.0*g1t33);
  a_g1t99 += a_g1t161 * (3.0*g1t36);
  a_g1t39 += a_g1t160 * (3.0);
  a_g1t127 += a_g1t159 * (g1t23*g1t40*hDD12);
  a_g1t23 += a_g1t159 * (g1t127*g1t40*hDD12);
  a_g1t40 += a_g1t159 * (g1t127*g1t23*hDD12);
  a_hDD12 += a_g1t159 * (g1t127*g1t23*g1t40);
  a_g1t154 += a_g1t158 * (g1t55);
  a_g1t55 += a_g1t158 * (g1t154);
  a_g1t1 += a_g1t157 * (hDD_dDD1101);
  double a_hDD_dDD1101 = a_g1t157 * (g1t1);
  a_g1t41 += a_g1t156 * (2.0);
  double a_g1t27 = a_g1t155 * (hDD_dD110);
  a_hDD_dD110 += a_g1t155 * (g1t27);
  a_g1t1 += a_g1t154 * (g1t78);
  double a_g1t76 = a_g1t154 * (1.0);
  double a_g1t78 = a_g1t154 * (g1t1);
  a_g1t54 += a_g1t153 * (2.0);
  a_g1t33 += a_g1t152 * (g1t90);
  a_g1t36 += a_g1t152 * (g1t89);
  a_g1t7 += a_g1t152 * (g1t83);
  a_g1t83 += a_g1t152 * (g1t7);
  double a_g1t89 = a_g1t152 * (g1t36);
  a_g1t90 += a_g1t152 * (g1t33);
  a_g1t94 += a_g1t151 * (2.0);
  a_g1t147 += a_g1t150 * (1.0);
  a_g1t33 += a_g1t150 * (g1t54);
  a_g1t36 += a_g1t150 * (g1t51);
  a_g1t51 += a_g1t150 * (g1t36);
  a_g1t54 += a_g1t150 * (g1t33);
  a_g1t103 += a_g1t149 * (2.0);
  a_g1t32 += a_g1t148 * (2.0);
  a_g1t58 += a_g1t147 * (g1t7);
  a_g1t7 += a_g1t147 * (g1t58);
  a_g1t99 += a_g1t146 * (2.0);
  a_g1t7 += a_g1t145 * (g1t77);
  a_g1t77 += a_g1t145 * (g1t7);
  a_g1t44 += a_g1t144 * (2.0);
  a_g1t17 += a_g1t143 * (hDD01);
  a_hDD01 += a_g1t143 * (g1t17);
  a_g1t55 += a_g1t142 * (lambdaU0);
  double a_lambdaU0 = a_g1t142 * (g1t55);
  a_g1t29 += a_g1t141 * (Rational_1_2);
  a_g1t139 += a_g1t140 * (1.0);
  a_hDD01 += a_g1t140 * (1.0);
  a_f0_of_xx0 += a_g1t139 * (hDD_dD010);
  a_hDD_dD010 += a_g1t139 * (f0_of_xx0);
  a_g1t92 += a_g1t138 * (hDD_dD000);
  double a_hDD_dD000 = a_g1t138 * (g1t92);
  double a_g1t133 = a_g1t137 * (g1t55);
  a_g1t55 += a_g1t137 * (g1t133);
  a_g1t1 += a_g1t136 * (-g1t22*hDD22);
  a_g1t22 += a_g1t136 * (-g1t1*hDD22 + g1t6);
  a_g1t3 += a_g1t136 * (hDD01);
  double a_g1t6 = a_g1t136 * (g1t22);
  a_hDD01 += a_g1t136 * (g1t3);
  double a_hDD22 = a_g1t136 * (-g1t1*g1t22);
  a_f0_of_xx0 += a_g1t135 * (hDD00 - hDD11 + hDD_dD011);
  a_hDD00 += a_g1t135 * (f0_of_xx0);
  a_hDD11 += a_g1t135 * (-f0_of_xx0);
  a_hDD_dD011 += a_g1t135 * (f0_of_xx0);
  a_g1t133 += a_g1t134 * (g1t41);
  a_g1t41 += a_g1t134 * (g1t133);
  a_g1t22 += a_g1t133 * (g1t33);
  a_g1t33 += a_g1t133 * (g1t22);
  a_g1t92 += a_g1t133 * (hDD00 - hDD22);
  a_hDD00 += a_g1t133 * (g1t92);
  a_hDD22 += a_g1t133 * (-g1t92);
  a_f0_of_xx0 += a_g1t132 * (f1_of_xx1__D1);
  a_f1_of_xx1__D1 += a_g1t132 * (f0_of_xx0);
  a_g1t123 += a_g1t131 * (g1t55);
  a_g1t55 += a_g1t131 * (g1t123);
  a_f0_of_xx0 += a_g1t130 * (f1_of_xx1);
  a_f1_of_xx1 += a_g1t130 * (f0_of_xx0);
  a_f0_of_xx0 += a_g1t129 * (g1t81);
  a_g1t28 += a_g1t129 * (1.0);
  a_g1t81 += a_g1t129 * (f0_of_xx0);
  a_f1_of_xx1__DD11 += a_g1t128 * (g1t40);
  a_g1t127 += a_g1t128 * (-1.0/g1t2);
  a_g1t2 += a_g1t128 * (g1t127/(g1t2*g1t2));
  a_g1t40 += a_g1t128 * (f1_of_xx1__DD11);
  a_f1_of_xx1__D1 += a_g1t127 * (2.0*f1_of_xx1__D1);
  double a_g1t72 = a_g1t126 * (1.0);
  double a_g1t74 = a_g1t126 * (1.0);
  double a_g1t35 = a_g1t125 * (1.0);
  a_g1t72 += a_g1t125 * (1.0);
  a_g1t122 += a_g1t124 * (-1.0);
  double a_g1t15 = a_g1t124 * (-1.0);
  a_g1t122 += a_g1t123 * (-1.0);
  double a_g1t13 = a_g1t123 * (-1.0);
  a_f0_of_xx0 += a_g1t122 * (g1t18);
  a_g1t18 += a_g1t122 * (f0_of_xx0);
  a_g1t1 += a_g1t121 * (g1t120);
  a_g1t120 += a_g1t121 * (g1t1);
  a_f1_of_xx1 += a_g1t120 * (3.0*(f1_of_xx1*f1_of_xx1));
  double a_lambdaU2 = a_g1t119 * (Rational_1_2);
  a_g1t86 += a_g1t118 * (g1t88);
  a_g1t88 += a_g1t118 * (g1t86);
  a_g1t51 += a_g1t117 * (2.0);
  a_g1t0 += a_g1t116 * (g1t90);
  a_g1t29 += a_g1t116 * (g1t89);
  a_g1t33 += a_g1t116 * (g1t83);
  a_g1t83 += a_g1t116 * (g1t33);
  a_g1t89 += a_g1t116 * (g1t29);
  a_g1t90 += a_g1t116 * (g1t0);
  a_g1t33 += a_g1t115 * (g1t86);
  a_g1t36 += a_g1t115 * (g1t87);
  a_g1t64 += a_g1t115 * (g1t7);
  a_g1t7 += a_g1t115 * (g1t64);
  a_g1t86 += a_g1t115 * (g1t33);
  a_g1t87 += a_g1t115 * (g1t36);
  a_g1t89 += a_g1t114 * (2.0);
  a_g1t29 += a_g1t113 * (g1t94);
  a_g1t36 += a_g1t113 * (g1t77);
  a_g1t4 += a_g1t113 * (g1t99);
  a_g1t77 += a_g1t113 * (g1t36);
  a_g1t94 += a_g1t113 * (g1t29);
  a_g1t99 += a_g1t113 * (g1t4);
  a_g1t111 += a_g1t112 * (g1t58);
  a_g1t58 += a_g1t112 * (g1t111);
  a_g1t110 += a_g1t111 * (1.0);
  a_g1t32 += a_g1t111 * (g1t33);
  a_g1t33 += a_g1t111 * (g1t32);
  a_g1t36 += a_g1t111 * (g1t44);
  a_g1t44 += a_g1t111 * (g1t36);
  a_g1t39 += a_g1t110 * (g1t7);
  a_g1t7 += a_g1t110 * (g1t39);
  a_g1t0 += a_g1t109 * (g1t94);
  a_g1t29 += a_g1t109 * (g1t99);
  a_g1t33 += a_g1t109 * (g1t77);
  a_g1t77 += a_g1t109 * (g1t33);
  a_g1t94 += a_g1t109 * (g1t0);
  a_g1t99 += a_g1t109 * (g1t29);
  a_g1t45 += a_g1t108 * (g1t54);
  a_g1t54 += a_g1t108 * (g1t45);
  a_g1t106 += a_g1t107 * (g1t32);
  a_g1t32 += a_g1t107 * (g1t106);
  a_g1t0 += a_g1t106 * (g1t54);
  a_g1t29 += a_g1t106 * (g1t51);
  a_g1t33 += a_g1t106 * (g1t58);
  a_g1t51 += a_g1t106 * (g1t29);
  a_g1t54 += a_g1t106 * (g1t0);
  a_g1t58 += a_g1t106 * (g1t33);
  a_g1t104 += a_g1t105 * (g1t51);
  a_g1t51 += a_g1t105 * (g1t104);
  a_g1t29 += a_g1t104 * (g1t32);
  a_g1t32 += a_g1t104 * (g1t29);
  a_g1t36 += a_g1t104 * (g1t39);
  a_g1t39 += a_g1t104 * (g1t36);
  a_g1t4 += a_g1t104 * (g1t44);
  a_g1t44 += a_g1t104 * (g1t4);
  a_g1t33 += a_g1t103 * (g1t93);
  a_g1t36 += a_g1t103 * (g1t96);
  a_g1t7 += a_g1t103 * (g1t70);
  a_g1t70 += a_g1t103 * (g1t7);
  a_g1t93 += a_g1t103 * (g1t33);
  a_g1t96 += a_g1t103 * (g1t36);
  a_g1t87 += a_g1t102 * (2.0);
  a_g1t29 += a_g1t101 * (g1t93);
  a_g1t36 += a_g1t101 * (g1t70);
  a_g1t4 += a_g1t101 * (g1t96);
  a_g1t70 += a_g1t101 * (g1t36);
  a_g1t93 += a_g1t101 * (g1t29);
  a_g1t96 += a_g1t101 * (g1t4);
  a_g1t30 += a_g1t100 * (g1t87);
  a_g1t34 += a_g1t100 * (g1t51);
  a_g1t37 += a_g1t100 * (g1t44);
  a_g1t43 += a_g1t100 * (g1t96);
  a_g1t44 += a_g1t100 * (g1t37);
  a_g1t51 += a_g1t100 * (g1t34);
  a_g1t60 += a_g1t100 * (g1t99);
  a_g1t84 += a_g1t100 * (g1t89);
  a_g1t87 += a_g1t100 * (g1t30);
  a_g1t89 += a_g1t100 * (g1t84);
  a_g1t96 += a_g1t100 * (g1t43);
  a_g1t99 += a_g1t100 * (g1t60);
  a_g1t31 += a_g1t99 * (g1t71);
  a_g1t38 += a_g1t99 * (g1t76);
  a_g1t43 += a_g1t99 * (g1t75);
  double a_g1t71 = a_g1t99 * (g1t31);
  double a_g1t75 = a_g1t99 * (g1t43);
  a_g1t76 += a_g1t99 * (g1t38);
  a_g1t29 += a_g1t98 * (g1t86);
  a_g1t36 += a_g1t98 * (g1t64);
  a_g1t4 += a_g1t98 * (g1t87);
  a_g1t64 += a_g1t98 * (g1t36);
  a_g1t86 += a_g1t98 * (g1t29);
  a_g1t87 += a_g1t98 * (g1t4);
  a_g1t0 += a_g1t97 * (g1t93);
  a_g1t29 += a_g1t97 * (g1t96);
  a_g1t33 += a_g1t97 * (g1t70);
  a_g1t70 += a_g1t97 * (g1t33);
  a_g1t93 += a_g1t97 * (g1t0);
  a_g1t96 += a_g1t97 * (g1t29);
  a_g1t31 += a_g1t96 * (g1t68);
  a_g1t38 += a_g1t96 * (g1t67);
  double a_g1t67 = a_g1t96 * (g1t38);
  double a_g1t68 = a_g1t96 * (g1t31);
  a_g1t30 += a_g1t95 * (g1t86);
  a_g1t32 += a_g1t95 * (g1t37);
  a_g1t34 += a_g1t95 * (g1t54);
  a_g1t37 += a_g1t95 * (g1t32);
  a_g1t43 += a_g1t95 * (g1t93);
  a_g1t54 += a_g1t95 * (g1t34);
  a_g1t60 += a_g1t95 * (g1t94);
  a_g1t84 += a_g1t95 * (g1t90);
  a_g1t86 += a_g1t95 * (g1t30);
  a_g1t90 += a_g1t95 * (g1t84);
  a_g1t93 += a_g1t95 * (g1t43);
  a_g1t94 += a_g1t95 * (g1t60);
  a_f0_of_xx0 += a_g1t94 * (1.0);
  a_g1t31 += a_g1t94 * (g1t75);
  a_g1t69 += a_g1t94 * (g1t76);
  a_g1t71 += a_g1t94 * (g1t84);
  a_g1t75 += a_g1t94 * (g1t31);
  a_g1t76 += a_g1t94 * (g1t69);
  a_g1t84 += a_g1t94 * (g1t71);
  a_g1t67 += a_g1t93 * (g1t69);
  a_g1t68 += a_g1t93 * (g1t84);
  a_g1t69 += a_g1t93 * (g1t67);
  a_g1t84 += a_g1t93 * (g1t68);
  a_g1t92 += a_g1t93 * (1.0);
  a_f0_of_xx0 += a_g1t92 * (g1t2);
  a_g1t2 += a_g1t92 * (f0_of_xx0);
  a_g1t29 += a_g1t91 * (g1t90);
  a_g1t36 += a_g1t91 * (g1t83);
  a_g1t4 += a_g1t91 * (g1t89);
  a_g1t83 += a_g1t91 * (g1t36);
  a_g1t89 += a_g1t91 * (g1t4);
  a_g1t90 += a_g1t91 * (g1t29);
  a_g1t31 += a_g1t90 * (g1t82);
  a_g1t69 += a_g1t90 * (g1t80);
  double a_g1t80 = a_g1t90 * (g1t69);
  double a_g1t82 = a_g1t90 * (g1t31);
  a_g1t84 += a_g1t90 * (hDD_dD000);
  a_hDD_dD000 += a_g1t90 * (g1t84);
  a_g1t31 += a_g1t89 * (hDD_dD000);
  a_g1t38 += a_g1t89 * (g1t80);
  a_g1t43 += a_g1t89 * (g1t82);
  a_g1t80 += a_g1t89 * (g1t38);
  a_g1t82 += a_g1t89 * (g1t43);
  a_hDD_dD000 += a_g1t89 * (g1t31);
  a_g1t0 += a_g1t88 * (g1t86);
  a_g1t29 += a_g1t88 * (g1t87);
  a_g1t33 += a_g1t88 * (g1t64);
  a_g1t64 += a_g1t88 * (g1t33);
  a_g1t86 += a_g1t88 * (g1t0);
  a_g1t87 += a_g1t88 * (g1t29);
  double a_g1t20 = a_g1t87 * (g1t38);
  a_g1t38 += a_g1t87 * (g1t20);
  a_g1t43 += a_g1t87 * (g1t63);
  double a_g1t56 = a_g1t87 * (1.0);
  double a_g1t63 = a_g1t87 * (g1t43);
  a_g1t20 += a_g1t86 * (g1t69);
  a_g1t31 += a_g1t86 * (g1t63);
  a_g1t63 += a_g1t86 * (g1t31);
  a_g1t69 += a_g1t86 * (g1t20);
  a_g1t30 += a_g1t85 * (g1t64);
  a_g1t43 += a_g1t85 * (g1t70);
  a_g1t60 += a_g1t85 * (g1t77);
  a_g1t64 += a_g1t85 * (g1t30);
  a_g1t65 += a_g1t85 * (1.0);
  a_g1t66 += a_g1t85 * (1.0);
  a_g1t70 += a_g1t85 * (g1t43);
  a_g1t77 += a_g1t85 * (g1t60);
  a_g1t83 += a_g1t85 * (g1t84);
  a_g1t84 += a_g1t85 * (g1t83);
  a_g1t12 += a_g1t84 * (Rational_1_2);
  a_g1t38 += a_g1t83 * (g1t82);
  a_g1t60 += a_g1t83 * (g1t80);
  a_g1t69 += a_g1t83 * (hDD_dD000);
  a_g1t80 += a_g1t83 * (g1t60);
  a_g1t82 += a_g1t83 * (g1t38);
  a_hDD_dD000 += a_g1t83 * (g1t69);
  a_g1t17 += a_g1t82 * (g1t81);
  a_g1t28 += a_g1t82 * (2.0);
  a_g1t81 += a_g1t82 * (g1t17);
  a_f1_of_xx1 += a_g1t81 * (hDD_dD020);
  a_hDD_dD020 += a_g1t81 * (f1_of_xx1);
  a_g1t17 += a_g1t80 * (hDD_dD010);
  a_g1t79 += a_g1t80 * (1.0);
  a_hDD_dD010 += a_g1t80 * (g1t17);
  a_g1t78 += a_g1t79 * (1.0);
  a_hDD_dD001 += a_g1t79 * (-1.0);
  a_hDD01 += a_g1t78 * (2.0);
  a_g1t38 += a_g1t77 * (g1t75);
  a_g1t60 += a_g1t77 * (g1t76);
  a_g1t69 += a_g1t77 * (g1t71);
  a_g1t71 += a_g1t77 * (g1t69);
  a_g1t75 += a_g1t77 * (g1t38);
  a_g1t76 += a_g1t77 * (g1t60);
  a_g1t1 += a_g1t76 * (hDD_dD111);
  a_hDD_dD111 += a_g1t76 * (g1t1);
  a_g1t72 += a_g1t75 * (2.0);
  a_g1t74 += a_g1t75 * (2.0);
  a_g1t73 += a_g1t74 * (hDD12);
  a_hDD12 += a_g1t74 * (g1t73);
  a_f1_of_xx1__D1 += a_g1t73 * (g1t1);
  a_g1t1 += a_g1t73 * (f1_of_xx1__D1);
  double a_g1t16 = a_g1t72 * (hDD_dD121);
  double a_hDD_dD121 = a_g1t72 * (g1t16);
  a_f0_of_xx0 += a_g1t71 * (2.0*hDD_dD011);
  double a_g1t50 = a_g1t71 * (-1.0);
  a_hDD_dD011 += a_g1t71 * (2.0*f0_of_xx0);
  a_g1t22 += a_g1t70 * (1.0);
  a_g1t60 += a_g1t70 * (g1t67);
  a_g1t67 += a_g1t70 * (g1t60);
  a_g1t68 += a_g1t70 * (g1t69);
  a_g1t69 += a_g1t70 * (g1t68);
  a_g1t34 += a_g1t69 * (Rational_1_2);
  a_g1t63 += a_g1t68 * (-1.0);
  double a_g1t26 = a_g1t67 * (-1.0);
  a_g1t34 += a_g1t66 * (g1t58);
  a_g1t58 += a_g1t66 * (g1t34);
  a_g1t37 += a_g1t65 * (g1t39);
  a_g1t39 += a_g1t65 * (g1t37);
  a_g1t20 += a_g1t64 * (g1t60);
  a_g1t38 += a_g1t64 * (g1t63);
  a_g1t60 += a_g1t64 * (g1t20);
  a_g1t63 += a_g1t64 * (g1t38);
  a_g1t17 += a_g1t63 * (g1t2);
  a_g1t2 += a_g1t63 * (g1t17);
  a_g1t62 += a_g1t63 * (1.0);
  a_g1t17 += a_g1t62 * (g1t61);
  a_g1t3 += a_g1t62 * (hDD_dD220);
  a_g1t61 += a_g1t62 * (g1t17);
  a_hDD_dD220 += a_g1t62 * (g1t3);
  a_g1t2 += a_g1t61 * (hDD22);
  a_hDD22 += a_g1t61 * (g1t2);
  a_g1t57 += a_g1t60 * (Rational_1_2);
  a_g1t29 += a_g1t59 * (g1t54);
  a_g1t36 += a_g1t59 * (g1t58);
  a_g1t4 += a_g1t59 * (g1t51);
  a_g1t51 += a_g1t59 * (g1t4);
  a_g1t54 += a_g1t59 * (g1t29);
  a_g1t58 += a_g1t59 * (g1t36);
  a_g1t34 += a_g1t58 * (g1t52);
  a_g1t38 += a_g1t58 * (g1t48);
  double a_g1t48 = a_g1t58 * (g1t38);
  double a_g1t52 = a_g1t58 * (g1t34);
  double a_g1t53 = a_g1t58 * (g1t57);
  a_g1t56 += a_g1t58 * (1.0);
  a_g1t57 += a_g1t58 * (g1t53);
  a_g1t0 += a_g1t57 * (g1t11*g1t4);
  double a_g1t11 = a_g1t57 * (g1t0*g1t4 - g1t8);
  a_g1t4 += a_g1t57 * (g1t0*g1t11);
  double a_g1t8 = a_g1t57 * (-g1t11);
  a_g1t55 += a_g1t56 * (-1.0);
  a_f0_of_xx0 += a_g1t55 * (-1.0/(f0_of_xx0*f0_of_xx0));
  a_g1t12 += a_g1t54 * (g1t52);
  a_g1t31 += a_g1t54 * (g1t48);
  a_g1t34 += a_g1t54 * (g1t53);
  a_g1t48 += a_g1t54 * (g1t31);
  a_g1t52 += a_g1t54 * (g1t12);
  a_g1t53 += a_g1t54 * (g1t34);
  a_g1t50 += a_g1t53 * (Rational_1_2);
  a_hDD_dD001 += a_g1t52 * (Rational_1_2);
  a_g1t31 += a_g1t51 * (hDD_dD001);
  a_g1t38 += a_g1t51 * (g1t50);
  a_g1t43 += a_g1t51 * (g1t48);
  a_g1t48 += a_g1t51 * (g1t43);
  a_g1t50 += a_g1t51 * (g1t38);
  a_hDD_dD001 += a_g1t51 * (g1t31);
  a_g1t17 += a_g1t50 * (1.0);
  a_g1t49 += a_g1t50 * (1.0);
  a_g1t1 += a_g1t49 * (hDD_dD110);
  a_g1t17 += a_g1t49 * (hDD11);
  a_hDD11 += a_g1t49 * (g1t17);
  a_hDD_dD110 += a_g1t49 * (g1t1);
  a_g1t19 += a_g1t48 * (1.0);
  a_g1t47 += a_g1t48 * (1.0);
  a_f0_of_xx0 += a_g1t47 * (g1t46);
  a_g1t15 += a_g1t47 * (1.0);
  a_g1t46 += a_g1t47 * (f0_of_xx0);
  a_f1_of_xx1 += a_g1t46 * (hDD_dD021);
  a_hDD_dD021 += a_g1t46 * (f1_of_xx1);
  a_g1t0 += a_g1t45 * (g1t32);
  a_g1t29 += a_g1t45 * (g1t44);
  a_g1t32 += a_g1t45 * (g1t0);
  a_g1t33 += a_g1t45 * (g1t39);
  a_g1t39 += a_g1t45 * (g1t33);
  a_g1t44 += a_g1t45 * (g1t29);
  double a_g1t21 = a_g1t44 * (g1t30);
  a_g1t26 += a_g1t44 * (g1t43);
  a_g1t30 += a_g1t44 * (g1t21);
  a_g1t41 += a_g1t44 * (-1.0);
  a_g1t43 += a_g1t44 * (g1t26);
  a_g1t42 += a_g1t43 * (Rational_1_2);
  a_g1t0 += a_g1t42 * (g1t11*g1t7);
  a_g1t11 += a_g1t42 * (g1t0*g1t7 - g1t5);
  double a_g1t5 = a_g1t42 * (-g1t11);
  a_g1t7 += a_g1t42 * (g1t0*g1t11);
  a_f1_of_xx1__D1 += a_g1t41 * (g1t40);
  a_g1t40 += a_g1t41 * (f1_of_xx1__D1);
  a_f1_of_xx1 += a_g1t40 * (-1.0/(f1_of_xx1*f1_of_xx1));
  a_g1t21 += a_g1t39 * (g1t34);
  a_g1t26 += a_g1t39 * (g1t38);
  a_g1t34 += a_g1t39 * (g1t21);
  a_g1t38 += a_g1t39 * (g1t26);
  a_g1t37 += a_g1t38 * (Rational_1_2);
  a_g1t0 += a_g1t37 * (-g1t11*g1t36);
  a_g1t11 += a_g1t37 * (-g1t0*g1t36 + g1t35*hDD01);
  a_g1t35 += a_g1t37 * (g1t11*hDD01);
  a_g1t36 += a_g1t37 * (-g1t0*g1t11);
  a_hDD01 += a_g1t37 * (g1t11*g1t35);
  a_g1t1 += a_g1t36 * (g1t18);
  a_g1t18 += a_g1t36 * (g1t1);
  a_g1t1 += a_g1t35 * (g1t28);
  a_g1t28 += a_g1t35 * (g1t1);
  a_g1t11 += a_g1t34 * (g1t2*g1t27*hDD02*hDD12 - g1t33*g1t4);
  a_g1t2 += a_g1t34 * (g1t11*g1t27*hDD02*hDD12);
  a_g1t27 += a_g1t34 * (g1t11*g1t2*hDD02*hDD12);
  a_g1t33 += a_g1t34 * (-g1t11*g1t4);
  a_g1t4 += a_g1t34 * (-g1t11*g1t33);
  a_hDD02 += a_g1t34 * (g1t11*g1t2*g1t27*hDD12);
  a_hDD12 += a_g1t34 * (g1t11*g1t2*g1t27*hDD02);
  a_f0_of_xx0 += a_g1t33 * (hDD01);
  a_hDD01 += a_g1t33 * (f0_of_xx0);
  a_g1t12 += a_g1t32 * (g1t21);
  a_g1t21 += a_g1t32 * (g1t12);
  a_g1t26 += a_g1t32 * (g1t31);
  a_g1t31 += a_g1t32 * (g1t26);
  a_g1t30 += a_g1t31 * (Rational_1_2);
  a_g1t11 += a_g1t30 * (g1t18*g1t27*hDD01 - g1t29*g1t7);
  a_g1t18 += a_g1t30 * (g1t11*g1t27*hDD01);
  a_g1t27 += a_g1t30 * (g1t11*g1t18*hDD01);
  a_g1t29 += a_g1t30 * (-g1t11*g1t7);
  a_g1t7 += a_g1t30 * (-g1t11*g1t29);
  a_hDD01 += a_g1t30 * (g1t11*g1t18*g1t27);
  a_f0_of_xx0 += a_g1t29 * (g1t28);
  a_g1t28 += a_g1t29 * (f0_of_xx0);
  a_f1_of_xx1 += a_g1t28 * (hDD02);
  a_hDD02 += a_g1t28 * (f1_of_xx1);
  a_f0_of_xx0 += a_g1t27 * (3.0*(f0_of_xx0*f0_of_xx0));
  double a_g1t24 = a_g1t26 * (1.0);
  a_g1t25 += a_g1t26 * (1.0);
  a_g1t24 += a_g1t25 * (hDD22);
  a_g1t3 += a_g1t25 * (hDD_dD221);
  a_hDD22 += a_g1t25 * (g1t24);
  a_hDD_dD221 += a_g1t25 * (g1t3);
  a_g1t22 += a_g1t24 * (g1t23);
  a_g1t23 += a_g1t24 * (g1t22);
  a_g1t1 += a_g1t23 * (2.0);
  a_f1_of_xx1 += a_g1t22 * (f1_of_xx1__D1);
  a_f1_of_xx1__D1 += a_g1t22 * (f1_of_xx1);
  a_g1t20 += a_g1t21 * (Rational_m1_2);
  a_g1t13 += a_g1t20 * (1.0);
  a_g1t15 += a_g1t20 * (-1.0);
  a_g1t19 += a_g1t20 * (1.0);
  a_g1t16 += a_g1t19 * (hDD_dD120);
  a_g1t17 += a_g1t19 * (g1t18);
  a_g1t18 += a_g1t19 * (g1t17);
  a_hDD_dD120 += a_g1t19 * (g1t16);
  a_f1_of_xx1 += a_g1t18 * (hDD12);
  a_hDD12 += a_g1t18 * (f1_of_xx1);
  a_f0_of_xx0 += a_g1t17 * (2.0);
  a_f1_of_xx1 += a_g1t16 * (g1t1);
  a_g1t1 += a_g1t16 * (f1_of_xx1);
  a_f0_of_xx0 += a_g1t15 * (g1t14);
  a_g1t14 += a_g1t15 * (f0_of_xx0);
  a_f1_of_xx1__D1 += a_g1t14 * (hDD02);
  a_hDD02 += a_g1t14 * (f1_of_xx1__D1);
  a_f0_of_xx0 += a_g1t13 * (-f1_of_xx1*hDD_dD021);
  a_f1_of_xx1 += a_g1t13 * (-f0_of_xx0*hDD_dD021);
  a_hDD_dD021 += a_g1t13 * (-f0_of_xx0*f1_of_xx1);
  double a_g1t10 = a_g1t12 * (-g1t11);
  a_g1t11 += a_g1t12 * (-g1t10 + g1t4*g1t7);
  a_g1t4 += a_g1t12 * (g1t11*g1t7);
  a_g1t7 += a_g1t12 * (g1t11*g1t4);
  a_g1t0 += a_g1t11 * ((g1t10 - g1t4*g1t7)/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_g1t10 += a_g1t11 * (g1t0/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_g1t2 += a_g1t11 * (-2.0*g1t9*hDD01*hDD02*hDD12/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_g1t4 += a_g1t11 * ((-g1t0*g1t7 + g1t5)/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_g1t5 += a_g1t11 * (g1t4/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_g1t7 += a_g1t11 * ((-g1t0*g1t4 + g1t8)/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_g1t8 += a_g1t11 * (g1t7/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  double a_g1t9 = a_g1t11 * (-2.0*g1t2*hDD01*hDD02*hDD12/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_hDD01 += a_g1t11 * (-2.0*g1t2*g1t9*hDD02*hDD12/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_hDD02 += a_g1t11 * (-2.0*g1t2*g1t9*hDD01*hDD12/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_hDD12 += a_g1t11 * (-2.0*g1t2*g1t9*hDD01*hDD02/((-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)*(-g1t0*g1t10 + g1t0*g1t4*g1t7 + 2.0*g1t2*g1t9*hDD01*hDD02*hDD12 - g1t4*g1t5 - g1t7*g1t8)));
  a_g1t2 += a_g1t10 * (g1t9*(hDD12*hDD12));
  a_g1t9 += a_g1t10 * (g1t2*(hDD12*hDD12));
  a_hDD12 += a_g1t10 * (2.0*g1t2*g1t9*hDD12);
  a_f0_of_xx0 += a_g1t9 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_g1t3 += a_g1t8 * ((hDD02*hDD02));
  a_hDD02 += a_g1t8 * (2.0*g1t3*hDD02);
  a_g1t1 += a_g1t7 * (1.0);
  a_g1t6 += a_g1t7 * (1.0);
  a_g1t1 += a_g1t6 * (hDD11);
  a_hDD11 += a_g1t6 * (g1t1);
  a_g1t1 += a_g1t5 * ((hDD01*hDD01));
  a_hDD01 += a_g1t5 * (2.0*g1t1*hDD01);
  a_g1t3 += a_g1t4 * (hDD22 + 1.0);
  a_hDD22 += a_g1t4 * (g1t3);
  a_g1t1 += a_g1t3 * (g1t2);
  a_g1t2 += a_g1t3 * (g1t1);
  a_f1_of_xx1 += a_g1t2 * (2.0*f1_of_xx1);
  a_f0_of_xx0 += a_g1t1 * (2.0*f0_of_xx0);
  a_hDD00 += a_g1t0 * (1.0);
  red[32 * 64 + lane] = a_hDD00;
  red[33 * 64 + lane] = a_hDD01;
  red[34 * 64 + lane] = a_hDD02;
  red[35 * 64 + lane] = a_hDD11;
  red[36 * 64 + lane] = a_hDD12;
  red[37 * 64 + lane] = a_hDD22;
  red[38 * 64 + lane] = a_hDD_dD000;
  red[39 * 64 + lane] = a_hDD_dD001;
  red[40 * 64 + lane] = a_hDD_dD010;
  red[41 * 64 + lane] = a_hDD_dD011;
  red[42 * 64 + lane] = a_hDD_dD020;
  red[43 * 64 + lane] = a_hDD_dD021;
  red[44 * 64 + lane] = a_hDD_dD110;
  red[45 * 64 + lane] = a_hDD_dD111;
  red[46 * 64 + lane] = a_hDD_dD120;
  red[47 * 64 + lane] = a_hDD_dD121;
  red[48 * 64 + lane] = a_hDD_dD220;
  red[49 * 64 + lane] = a_hDD_dD221;
  red[50 * 64 + lane] = a_hDD_dDD0200;
  red[51 * 64 + lane] = a_hDD_dDD0201;
  red[52 * 64 + lane] = a_hDD_dDD0211;
  red[53 * 64 + lane] = a_hDD_dDD1100;
  red[54 * 64 + lane] = a_hDD_dDD1101;
  red[55 * 64 + lane] = a_hDD_dDD1111;
  red[56 * 64 + lane] = a_lambdaU0;
  red[57 * 64 + lane] = a_lambdaU1;
  red[58 * 64 + lane] = a_lambdaU2;
  red[59 * 64 + lane] = a_lambdaU_dD00;
  red[60 * 64 + lane] = a_lambdaU_dD01;
  red[61 * 64 + lane] = a_lambdaU_dD10;
  red[62 * 64 + lane] = a_lambdaU_dD11;
  red[63 * 64 + lane] = a_lambdaU_dD20;
  red[64 * 64 + lane] = a_lambdaU_dD21;
  break;
  }
  case 2: { // RbarDD12, RbarDD22
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double hDD00 = in[11 * Ntot + idx];
  const double hDD01 = in[12 * Ntot + idx];
  const double hDD02 = in[13 * Ntot + idx];
  const double hDD11 = in[14 * Ntot + idx];
  const double hDD12 = in[15 * Ntot + idx];
  const double hDD22 = in[16 * Ntot + idx];
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  const double hDD_dDD1200 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[15 * Ntot + idx] + (4.0 / 3.0) * (in[15 * Ntot + idx + (1)] + in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] + in[15 * Ntot + idx + (-2)]));
  const double hDD_dDD1201 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[15 * Ntot + idx + (1 + 1 * s1)] - in[15 * Ntot + idx + (1 + -1 * s1)]) - (in[15 * Ntot + idx + (-1 + 1 * s1)] - in[15 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[15 * Ntot + idx + (1 + 2 * s1)] - in[15 * Ntot + idx + (1 + -2 * s1)]) - (in[15 * Ntot + idx + (-1 + 2 * s1)] - in[15 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[15 * Ntot + idx + (2 + 1 * s1)] - in[15 * Ntot + idx + (2 + -1 * s1)]) - (in[15 * Ntot + idx + (-2 + 1 * s1)] - in[15 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[15 * Ntot + idx + (2 + 2 * s1)] - in[15 * Ntot + idx + (2 + -2 * s1)]) - (in[15 * Ntot + idx + (-2 + 2 * s1)] - in[15 * Ntot + idx + (-2 + -2 * s1)])));
  const double hDD_dDD1211 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[15 * Ntot + idx] + (4.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] + in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] + in[15 * Ntot + idx + (-2 * s1)]));
  const double hDD_dDD2200 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[16 * Ntot + idx] + (4.0 / 3.0) * (in[16 * Ntot + idx + (1)] + in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] + in[16 * Ntot + idx + (-2)]));
  const double hDD_dDD2201 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[16 * Ntot + idx + (1 + 1 * s1)] - in[16 * Ntot + idx + (1 + -1 * s1)]) - (in[16 * Ntot + idx + (-1 + 1 * s1)] - in[16 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[16 * Ntot + idx + (1 + 2 * s1)] - in[16 * Ntot + idx + (1 + -2 * s1)]) - (in[16 * Ntot + idx + (-1 + 2 * s1)] - in[16 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[16 * Ntot + idx + (2 + 1 * s1)] - in[16 * Ntot + idx + (2 + -1 * s1)]) - (in[16 * Ntot + idx + (-2 + 1 * s1)] - in[16 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[16 * Ntot + idx + (2 + 2 * s1)] - in[16 * Ntot + idx + (2 + -2 * s1)]) - (in[16 * Ntot + idx + (-2 + 2 * s1)] - in[16 * Ntot + idx + (-2 + -2 * s1)])));
  const double hDD_dDD2211 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[16 * Ntot + idx] + (4.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] + in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] + in[16 * Ntot + idx + (-2 * s1)]));
  const double lambdaU0 = in[17 * Ntot + idx];
  const double lambdaU1 = in[18 * Ntot + idx];
  const double lambdaU2 = in[19 * Ntot + idx];
  const double lambdaU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (in[17 * Ntot + idx + (1 * s1)] - in[17 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[17 * Ntot + idx + (2 * s1)] - in[17 * Ntot + idx + (-2 * s1)]));
  const double lambdaU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (in[18 * Ntot + idx + (1 * s1)] - in[18 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[18 * Ntot + idx + (2 * s1)] - in[18 * Ntot + idx + (-2 * s1)]));
  const double lambdaU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (in[19 * Ntot + idx + (1 * s1)] - in[19 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[19 * Ntot + idx + (2 * s1)] - in[19 * Ntot + idx + (-2 * s1)]));
  const double g2t0 = (f0_of_xx0*f0_of_xx0);
  const double g2t1 = g2t0*hDD11;
  const double g2t2 = g2t0 + g2t1;
  const double g2t3 = (f1_of_xx1*f1_of_xx1);
  const double g2t4 = g2t0*g2t3;
  const double g2t5 = g2t4*hDD22;
  const double g2t6 = g2t4 + g2t5;
  const double g2t7 = g2t0*(hDD01*hDD01);
  const double g2t8 = hDD00 + 1.0;
  const double g2t9 = g2t4*(hDD02*hDD02);
  const double g2t10 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g2t11 = g2t10*g2t3*(hDD12*hDD12);
  const double g2t12 = (1.0 / (2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7));
  const double g2t13 = g2t12*(g2t6*g2t8 - g2t9);
  const double g2t14 = f0_of_xx0*f1_of_xx1;
  const double g2t15 = g2t14*hDD_dD021;
  const double g2t16 = -g2t15;
  const double g2t17 = f1_of_xx1__D1*hDD02;
  const double g2t18 = f0_of_xx0*g2t17;
  const double g2t19 = f1_of_xx1*g2t0;
  const double g2t20 = 2.0*f0_of_xx0;
  const double g2t21 = f1_of_xx1*hDD12;
  const double g2t22 = g2t19*hDD_dD120 + g2t20*g2t21;
  const double g2t23 = g2t16 - g2t18 + g2t22;
  const double g2t24 = (Rational_1_2)*g2t23;
  const double g2t25 = g2t20*g2t3;
  const double g2t26 = g2t25*hDD22 + g2t4*hDD_dD220;
  const double g2t27 = g2t25 + g2t26;
  const double g2t28 = f1_of_xx1*hDD02;
  const double g2t29 = g2t0*g2t28;
  const double g2t30 = g2t19*hDD12;
  const double g2t31 = g2t12*(g2t29*hDD01 - g2t30*g2t8);
  const double g2t32 = (Rational_1_2)*g2t31;
  const double g2t33 = g2t13*g2t24 + g2t27*g2t32;
  const double g2t34 = f0_of_xx0*hDD01;
  const double g2t35 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double g2t36 = g2t12*(g2t3*g2t35*hDD02*hDD12 - g2t34*g2t6);
  const double g2t37 = f0_of_xx0*g2t28;
  const double g2t38 = g2t12*(-g2t2*g2t37 + g2t21*g2t35*hDD01);
  const double g2t39 = (Rational_1_2)*g2t38;
  const double g2t40 = g2t24*g2t36 + g2t27*g2t39;
  const double g2t41 = (1.0 / f0_of_xx0);
  const double g2t42 = -g2t41;
  const double g2t43 = g2t12*(g2t2*g2t8 - g2t7);
  const double g2t44 = (Rational_1_2)*g2t43;
  const double g2t45 = g2t24*g2t31 + g2t27*g2t44 + g2t42;
  const double g2t46 = g2t2*g2t33 + g2t30*g2t45 + g2t34*g2t40;
  const double g2t47 = g2t15 + g2t18;
  const double g2t48 = g2t22 + g2t47;
  const double g2t49 = g2t0*hDD_dD110;
  const double g2t50 = g2t20*hDD11 + g2t49;
  const double g2t51 = g2t20 + g2t50;
  const double g2t52 = g2t32*g2t51 + g2t39*hDD_dD001 + g2t44*g2t48;
  const double g2t53 = g2t12*(-g2t11 + g2t2*g2t6);
  const double g2t54 = (Rational_1_2)*hDD_dD001;
  const double g2t55 = (Rational_1_2)*g2t51;
  const double g2t56 = g2t36*g2t55 + g2t39*g2t48 + g2t53*g2t54;
  const double g2t57 = g2t13*g2t55 + g2t32*g2t48 + g2t36*g2t54 + g2t42;
  const double g2t58 = g2t30*g2t57 + g2t37*g2t56 + g2t52*g2t6;
  const double g2t59 = -g2t23;
  const double g2t60 = (Rational_1_2)*g2t53;
  const double g2t61 = f1_of_xx1*f1_of_xx1__D1;
  const double g2t62 = 2.0*g2t0;
  const double g2t63 = g2t61*g2t62;
  const double g2t64 = g2t4*hDD_dD221 + g2t63*hDD22;
  const double g2t65 = g2t63 + g2t64;
  const double g2t66 = g2t39*g2t65 + g2t59*g2t60;
  const double g2t67 = f0_of_xx0*g2t3;
  const double g2t68 = -g2t27;
  const double g2t69 = -g2t65;
  const double g2t70 = (Rational_1_2)*g2t36;
  const double g2t71 = g2t60*g2t68 + g2t67 + g2t69*g2t70;
  const double g2t72 = 2.0*f0_of_xx0*hDD_dD011 - g2t51;
  const double g2t73 = g2t19*hDD_dD121;
  const double g2t74 = g2t0*hDD12;
  const double g2t75 = f1_of_xx1__D1*g2t74;
  const double g2t76 = 2.0*g2t73 + 2.0*g2t75;
  const double g2t77 = g2t0*hDD_dD111;
  const double g2t78 = f0_of_xx0 + g2t39*g2t76 + g2t60*g2t72 + g2t70*g2t77;
  const double g2t79 = (Rational_1_2)*g2t13;
  const double g2t80 = f1_of_xx1*g2t20;
  const double g2t81 = 2.0*g2t28 + g2t80*hDD_dD020;
  const double g2t82 = 2.0*hDD01;
  const double g2t83 = g2t20*hDD_dD010 + g2t82 - hDD_dD001;
  const double g2t84 = g2t39*g2t81 + g2t60*hDD_dD000 + g2t70*g2t83;
  const double g2t85 = g2t31*g2t66 + g2t36*g2t56 + g2t38*g2t40 + g2t44*g2t71 + g2t60*g2t84 + g2t78*g2t79;
  const double g2t86 = g2t32*g2t65 + g2t59*g2t70;
  const double g2t87 = (1.0 / f1_of_xx1);
  const double g2t88 = f1_of_xx1__D1*g2t87;
  const double g2t89 = g2t39*g2t59 + g2t44*g2t65 - g2t88;
  const double g2t90 = g2t2*g2t86 + g2t30*g2t89 + g2t34*g2t66;
  const double g2t91 = g2t32*g2t77 + g2t39*g2t72 + g2t44*g2t76;
  const double g2t92 = g2t32*g2t76 + g2t70*g2t72 + g2t77*g2t79;
  const double g2t93 = g2t30*g2t92 + g2t37*g2t78 + g2t6*g2t91;
  const double g2t94 = g2t61 + g2t68*g2t70 + g2t69*g2t79;
  const double g2t95 = g2t32*g2t81 + g2t70*hDD_dD000 + g2t79*g2t83;
  const double g2t96 = g2t31*g2t86 + g2t33*g2t38 + g2t36*g2t57 + g2t44*g2t94 + g2t60*g2t95 + g2t79*g2t92;
  const double g2t97 = g2t32*g2t69 + g2t39*g2t68;
  const double g2t98 = g2t2*g2t94 + g2t30*g2t97 + g2t34*g2t71;
  const double g2t99 = g2t6*g2t89;
  const double g2t100 = g2t30*g2t86;
  const double g2t101 = g2t100 + g2t37*g2t66 + g2t99;
  const double g2t102 = g2t31*g2t89;
  const double g2t103 = g2t38*g2t45;
  const double g2t104 = g2t32*g2t83 + g2t39*hDD_dD000 + g2t44*g2t81;
  const double g2t105 = g2t102 + g2t103 + g2t104*g2t60 + g2t36*g2t52 + g2t44*g2t97 + g2t79*g2t91;
  const double g2t106 = g2t6*g2t97;
  const double g2t107 = g2t106 + g2t30*g2t94 + g2t37*g2t71;
  const double g2t108 = 2.0*g2t89;
  const double g2t109 = g2t34*g2t94 + g2t37*g2t97 + g2t71*g2t8;
  const double g2t110 = g2t109*g2t66;
  const double g2t111 = g2t45*g2t6;
  const double g2t112 = g2t111 + g2t30*g2t33 + g2t37*g2t40;
  const double g2t113 = g2t112*g2t66;
  const double g2t114 = g2t86*g2t98;
  const double g2t115 = g2t101*g2t86;
  const double g2t116 = g2t90*g2t94;
  const double g2t117 = 2.0*g2t101;
  const double g2t118 = g2t2*g2t57 + g2t30*g2t52 + g2t34*g2t56;
  const double g2t119 = g2t34*g2t86 + g2t37*g2t89 + g2t66*g2t8;
  const double g2t120 = g2t2*g2t92 + g2t30*g2t91 + g2t34*g2t78;
  const double g2t121 = 2.0*g2t52;
  const double g2t122 = g2t104*g2t30 + g2t2*g2t95 + g2t34*g2t84;
  const double g2t123 = g2t33*g2t34 + g2t37*g2t45 + g2t40*g2t8;
  const double g2t124 = g2t104*g2t6 + g2t30*g2t95 + g2t37*g2t84;
  const double g2t125 = 2.0*g2t91;
  const double g2t126 = g2t119*g2t66;
  const double g2t127 = g2t58*g2t66;
  const double g2t128 = g2t86*g2t90;
  const double g2t129 = g2t86*g2t93;
  const double g2t130 = g2t33*g2t90;
  const double g2t131 = g2t123*g2t66;
  const double g2t132 = g2t124*g2t66;
  const double g2t133 = g2t46*g2t86;
  const double g2t134 = g2t58*g2t86;
  const double g2t135 = g2t14*hDD12;
  const double g2t136 = g2t29 + g2t73;
  const double g2t137 = g2t136*g2t61;
  const double g2t138 = (f1_of_xx1*f1_of_xx1*f1_of_xx1);
  const double g2t139 = g2t35*hDD_dD120;
  const double g2t140 = g2t138*g2t62;
  const double g2t141 = f1_of_xx1__D1*hDD12;
  const double g2t142 = 2.0*g2t4;
  const double g2t143 = g2t140*hDD02 + g2t141*g2t142;
  const double g2t144 = g2t143*g2t88;
  const double g2t145 = -g2t144;
  const double g2t146 = (f1_of_xx1__D1*f1_of_xx1__D1);
  const double g2t147 = -g2t135 - g2t16;
  const double g2t148 = g2t73 + g2t75;
  const double g2t149 = f1_of_xx1__D1*g2t0;
  const double g2t150 = f1_of_xx1__DD11*g2t87 - g2t146/g2t3;
  const double g2t151 = 2.0*g2t41;
  const double g2t152 = g2t136*g2t41;
  const double g2t153 = g2t141*g2t20 + g2t19*hDD_dDD1201 + g2t80*hDD_dD121;
  const double g2t154 = g2t14*hDD_dD020 + g2t28;
  const double g2t155 = g2t0*g2t61;
  const double g2t156 = g2t1*g2t61 - g2t155*hDD22 + g2t4*hDD01;
  const double g2t157 = g2t156*g2t88;
  const double g2t158 = g2t0*g2t82;
  const double g2t159 = g2t34*g2t61 + g2t67*hDD00 - g2t67*hDD22;
  const double g2t160 = g2t64*g2t88;
  const double g2t161 = f1_of_xx1*f1_of_xx1__DD11;
  const double g2t162 = g2t146 + g2t161;
  const double g2t163 = -g2t162;
  const double g2t164 = -g2t150*g2t5;
  const double g2t165 = g2t156*g2t41;
  const double g2t166 = g2t26*g2t88;
  const double g2t167 = g2t41*lambdaU0;
  const double g2t168 = (Rational_1_2)*g2t30;
  const double g2t169 = g2t167 + g2t41*g2t88*lambdaU1;
  const double g2t170 = (Rational_1_2)*g2t41;
  const double g2t171 = g2t20*g2t28;
  const double g2t172 = 2.0*g2t94;
  const double g2t173 = 2.0*g2t33;
  const double g2t174 = 2.0*g2t112;
  const double g2t175 = 2.0*g2t40;
  const double g2t176 = 2.0*g2t71;
  const double g2t177 = g2t35*hDD_dD220;
  const double g2t178 = 2.0*g2t61;
  const double g2t179 = 4.0*hDD22;
  const double g2t180 = g2t67*hDD_dD221;
  const double g2t181 = f0_of_xx0*g2t61;
  const double g2t182 = g2t179*g2t181 + g2t4*hDD_dDD2201;
  const double g2t183 = g2t143*g2t41;
  const double g2t184 = 3.0*g2t97;
  const double g2t185 = 3.0*g2t101;
  const double g2t186 = 3.0*g2t112;
  const double g2t187 = 3.0*g2t107;
  double a_f0_of_xx0 = S[4 * Ntot + idx] * (-g2t154*g2t70 - g2t159*g2t32 - g2t32*(f0_of_xx0*g2t3*(hDD00 - hDD11 + hDD_dD011) + g2t3*(f0_of_xx0*hDD00 - f0_of_xx0*hDD11 + f0_of_xx0*hDD_dD011)) - g2t39*g2t67*hDD_dD010 - g2t79*(g2t147 + g2t47));
  double a_f1_of_xx1 = S[4 * Ntot + idx] * (-f1_of_xx1__D1*g2t32*(g2t158 + g2t77) - g2t139*g2t79);
  double a_f1_of_xx1__D1 = S[4 * Ntot + idx] * (-f1_of_xx1*g2t32*(g2t158 + g2t77) - g2t170*g2t2*lambdaU2);
  double a_f1_of_xx1__DD11 = S[4 * Ntot + idx] * (-g2t74*g2t79);
  double a_g2t1 = S[4 * Ntot + idx] * (g2t163*g2t32);
  double a_g2t101 = S[4 * Ntot + idx] * (g2t105 + g2t108*g2t31 + g2t31*g2t92 + g2t38*g2t57);
  double a_g2t105 = S[4 * Ntot + idx] * (g2t101 + g2t98);
  double a_g2t107 = S[4 * Ntot + idx] * (g2t108*g2t43 + g2t121*g2t38 + g2t125*g2t31);
  double a_g2t108 = S[4 * Ntot + idx] * (g2t101*g2t31 + g2t107*g2t43 + g2t112*g2t38);
  double a_g2t109 = S[4 * Ntot + idx] * (g2t31*g2t78 + g2t38*g2t56);
  double a_g2t110 = S[4 * Ntot + idx] * (g2t43);
  double a_g2t112 = S[4 * Ntot + idx] * (g2t108*g2t38 + g2t121*g2t53 + g2t125*g2t36 + g2t31*g2t78 + g2t38*g2t56);
  double a_g2t113 = S[4 * Ntot + idx] * (g2t43);
  double a_g2t114 = S[4 * Ntot + idx] * (g2t43);
  double a_g2t115 = S[4 * Ntot + idx] * (g2t43);
  double a_g2t116 = S[4 * Ntot + idx] * (g2t43);
  double a_g2t117 = S[4 * Ntot + idx] * (g2t13*g2t91 + g2t36*g2t52);
  double a_g2t118 = S[4 * Ntot + idx] * (g2t13*g2t66 + g2t31*g2t71 + g2t33*g2t53 + g2t36*g2t40 + g2t36*g2t86 + g2t38*g2t94);
  double a_g2t119 = S[4 * Ntot + idx] * (g2t13*g2t78 + g2t36*g2t56);
  double a_g2t120 = S[4 * Ntot + idx] * (g2t13*g2t86 + g2t31*g2t94 + g2t33*g2t36);
  double a_g2t121 = S[4 * Ntot + idx] * (g2t107*g2t38 + g2t112*g2t53);
  double a_g2t122 = S[4 * Ntot + idx] * (g2t36*g2t66 + g2t38*g2t71 + g2t40*g2t53);
  double a_g2t123 = S[4 * Ntot + idx] * (g2t36*g2t78 + g2t53*g2t56);
  double a_g2t124 = S[4 * Ntot + idx] * (g2t36*g2t78 + g2t53*g2t56);
  double a_g2t125 = S[4 * Ntot + idx] * (g2t107*g2t31 + g2t112*g2t36);
  double a_g2t126 = S[4 * Ntot + idx] * (g2t31);
  double a_g2t127 = S[4 * Ntot + idx] * (g2t31);
  double a_g2t128 = S[4 * Ntot + idx] * (2.0*g2t31);
  double a_g2t129 = S[4 * Ntot + idx] * (g2t31);
  double a_g2t13 = S[4 * Ntot + idx] * (g2t117*g2t91 + g2t118*g2t66 + g2t119*g2t78 + g2t120*g2t86 + g2t58*g2t78 + g2t89*g2t90 + g2t90*g2t92 + g2t92*g2t93);
  double a_g2t130 = S[4 * Ntot + idx] * (g2t38);
  double a_g2t131 = S[4 * Ntot + idx] * (g2t38);
  double a_g2t132 = S[4 * Ntot + idx] * (g2t38);
  double a_g2t133 = S[4 * Ntot + idx] * (g2t38);
  double a_g2t134 = S[4 * Ntot + idx] * (g2t38);
  double a_g2t135 = S[4 * Ntot + idx] * (g2t44*g2t67);
  double a_g2t136 = S[4 * Ntot + idx] * (g2t79*g2t88);
  double a_g2t137 = S[4 * Ntot + idx] * (-g2t44);
  double a_g2t138 = S[4 * Ntot + idx] * (-g2t139*g2t44);
  double a_g2t139 = S[4 * Ntot + idx] * (-f1_of_xx1*g2t79 - g2t138*g2t44);
  double a_g2t14 = S[4 * Ntot + idx] * (-Rational_1_2*hDD01*lambdaU2);
  double a_g2t145 = S[4 * Ntot + idx] * (-g2t44);
  double a_g2t146 = S[4 * Ntot + idx] * (2.0*g2t30*g2t44);
  double a_g2t147 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t79);
  double a_g2t148 = S[4 * Ntot + idx] * (g2t151*g2t70 + g2t79*g2t88);
  double a_g2t149 = S[4 * Ntot + idx] * (-g2t70*hDD_dD120 - 2.0*g2t79*hDD_dD121);
  double a_g2t150 = S[4 * Ntot + idx] * (g2t30*g2t79);
  double a_g2t151 = S[4 * Ntot + idx] * (g2t148*g2t70 + g2t22*g2t60);
  double a_g2t152 = S[4 * Ntot + idx] * (4.0*g2t70);
  double a_g2t153 = S[4 * Ntot + idx] * (-2.0*g2t70);
  double a_g2t154 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t70);
  double a_g2t155 = S[4 * Ntot + idx] * (g2t32*hDD_dD221 + g2t39*hDD_dD220);
  double a_g2t157 = S[4 * Ntot + idx] * (3.0*g2t32);
  double a_g2t158 = S[4 * Ntot + idx] * (-f1_of_xx1*f1_of_xx1__D1*g2t32 - g2t32*g2t61);
  double a_g2t159 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t32);
  double a_g2t160 = S[4 * Ntot + idx] * (g2t32);
  double a_g2t163 = S[4 * Ntot + idx] * (g2t1*g2t32);
  double a_g2t164 = S[4 * Ntot + idx] * (-g2t32);
  double a_g2t165 = S[4 * Ntot + idx] * (4.0*g2t39);
  double a_g2t166 = S[4 * Ntot + idx] * (g2t39);
  double a_g2t167 = S[4 * Ntot + idx] * (g2t168);
  double a_g2t168 = S[4 * Ntot + idx] * (g2t167 + g2t169 + g2t41*lambdaU_dD11);
  double a_g2t169 = S[4 * Ntot + idx] * (g2t168);
  double a_g2t170 = S[4 * Ntot + idx] * (-f1_of_xx1__D1*g2t2*lambdaU2 + g2t6*g2t87*lambdaU_dD21);
  double a_g2t18 = S[4 * Ntot + idx] * (g2t44*g2t67);
  double a_g2t19 = S[4 * Ntot + idx] * (-g2t60*hDD_dDD1200 - g2t70*hDD_dD020 - g2t79*hDD_dDD1211);
  double a_g2t2 = S[4 * Ntot + idx] * (-f1_of_xx1__D1*g2t170*lambdaU2);
  double a_g2t21 = S[4 * Ntot + idx] * (-4.0*g2t60);
  double a_g2t22 = S[4 * Ntot + idx] * (g2t151*g2t60 + g2t70*g2t88);
  double a_g2t3 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t32*(f0_of_xx0*hDD00 - f0_of_xx0*hDD11 + f0_of_xx0*hDD_dD011));
  double a_g2t30 = S[4 * Ntot + idx] * (2.0*g2t146*g2t44 + g2t150*g2t79);
  double a_g2t31 = S[4 * Ntot + idx] * (g2t101*g2t108 + g2t101*g2t92 + g2t107*g2t125 + g2t109*g2t78 + g2t112*g2t78 + g2t118*g2t71 + g2t120*g2t94 + g2t126 + g2t127 + 2.0*g2t128 + g2t129 + g2t46*g2t66 + g2t89*g2t98 + g2t90*g2t97 + g2t92*g2t98);
  double a_g2t32 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t159 - f0_of_xx0*g2t3*(f0_of_xx0*hDD00 - f0_of_xx0*hDD11 + f0_of_xx0*hDD_dD011) - f1_of_xx1*f1_of_xx1__D1*(g2t158 + g2t77) + g2t1*g2t163 + g2t155*hDD_dD221 + 3.0*g2t157 - g2t158*g2t61 + g2t160 - g2t164 - g2t4*hDD_dD011 - g2t61*g2t77);
  double a_g2t33 = S[4 * Ntot + idx] * (g2t118*g2t53 + g2t120*g2t36);
  double a_g2t36 = S[4 * Ntot + idx] * (g2t112*g2t125 + g2t117*g2t52 + g2t118*g2t40 + g2t118*g2t86 + g2t119*g2t56 + g2t120*g2t33 + g2t122*g2t66 + g2t123*g2t78 + g2t124*g2t78 + g2t45*g2t90 + g2t46*g2t89 + g2t46*g2t92 + g2t56*g2t58 + g2t57*g2t90 + g2t57*g2t93 + g2t58*g2t92);
  double a_g2t37 = S[4 * Ntot + idx] * (-g2t70 - Rational_1_2*lambdaU1 + (Rational_1_2)*lambdaU_dD01);
  double a_g2t38 = S[4 * Ntot + idx] * (g2t101*g2t57 + g2t107*g2t121 + g2t108*g2t112 + g2t109*g2t56 + g2t112*g2t56 + g2t118*g2t94 + g2t122*g2t71 + g2t130 + g2t131 + g2t132 + g2t133 + g2t134 + g2t40*g2t46 + g2t45*g2t98 + g2t46*g2t97 + g2t57*g2t98);
  double a_g2t39 = S[4 * Ntot + idx] * (g2t155*hDD_dD220 + 4.0*g2t165 + g2t166 - g2t4*hDD_dD010 - g2t49*g2t61 - g2t50*g2t61 - g2t67*hDD01 - g2t67*(f0_of_xx0*hDD_dD010 + hDD01));
  double a_g2t4 = S[4 * Ntot + idx] * (-g2t32*hDD_dD011 - g2t39*hDD_dD010);
  double a_g2t40 = S[4 * Ntot + idx] * (g2t118*g2t36 + g2t122*g2t53 + g2t38*g2t46);
  double a_g2t41 = S[4 * Ntot + idx] * (g2t168*lambdaU_dD11);
  double a_g2t43 = S[4 * Ntot + idx] * (g2t107*g2t108 + g2t110 + g2t113 + g2t114 + g2t115 + g2t116 + g2t46*g2t71 + g2t97*g2t98);
  double a_g2t44 = S[4 * Ntot + idx] * (-g2t137 - g2t138*g2t139 - g2t145 + 2.0*g2t146*g2t30 - g2t67*(-g2t135 - g2t18));
  double a_g2t45 = S[4 * Ntot + idx] * (g2t36*g2t90 + g2t38*g2t98 + g2t46*g2t53);
  double a_g2t46 = S[4 * Ntot + idx] * (g2t31*g2t66 + g2t36*g2t89 + g2t36*g2t92 + g2t38*g2t40 + g2t38*g2t97 + g2t43*g2t71 + g2t45*g2t53 + g2t53*g2t57 + g2t85);
  double a_g2t47 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t79);
  double a_g2t49 = S[4 * Ntot + idx] * (-g2t39*g2t61);
  double a_g2t50 = S[4 * Ntot + idx] * (-g2t39*g2t61);
  double a_g2t52 = S[4 * Ntot + idx] * (g2t117*g2t36);
  double a_g2t53 = S[4 * Ntot + idx] * (g2t112*g2t121 + g2t118*g2t33 + g2t122*g2t40 + g2t123*g2t56 + g2t124*g2t56 + g2t45*g2t46 + g2t46*g2t57 + g2t57*g2t58);
  double a_g2t56 = S[4 * Ntot + idx] * (g2t36*(g2t119 + g2t58) + g2t38*(g2t109 + g2t112) + g2t53*(g2t123 + g2t124));
  double a_g2t57 = S[4 * Ntot + idx] * (g2t36*(g2t90 + g2t93) + g2t38*(g2t101 + g2t98) + g2t53*(g2t46 + g2t58));
  double a_g2t58 = S[4 * Ntot + idx] * (g2t13*g2t78 + g2t36*g2t56 + g2t36*g2t92 + g2t53*g2t57 + g2t85);
  double a_g2t6 = S[4 * Ntot + idx] * (g2t170*g2t87*lambdaU_dD21);
  double a_g2t60 = S[4 * Ntot + idx] * (g2t151*g2t22 - g2t19*hDD_dDD1200 - 4.0*g2t21 - g2t80*hDD_dD120);
  double a_g2t61 = S[4 * Ntot + idx] * (-g2t32*(g2t158 + g2t77) - g2t39*g2t49 - g2t39*g2t50);
  double a_g2t66 = S[4 * Ntot + idx] * (g2t118*g2t13 + g2t122*g2t36 + g2t31*g2t46);
  double a_g2t67 = S[4 * Ntot + idx] * (-g2t39*(f0_of_xx0*hDD_dD010 + 2.0*hDD01) - g2t44*(-g2t135 - g2t18));
  double a_g2t70 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t154 + g2t148*g2t151 - g2t149*hDD_dD120 + 4.0*g2t152 - 2.0*g2t153 - g2t19*hDD_dD020 + g2t22*g2t88 - g2t37);
  double a_g2t71 = S[4 * Ntot + idx] * (g2t118*g2t31 + g2t122*g2t38 + g2t43*g2t46);
  double a_g2t74 = S[4 * Ntot + idx] * (-f1_of_xx1__DD11*g2t79);
  double a_g2t77 = S[4 * Ntot + idx] * (-f1_of_xx1*f1_of_xx1__D1*g2t32 - g2t32*g2t61);
  double a_g2t78 = S[4 * Ntot + idx] * (g2t13*(g2t119 + g2t58) + g2t31*(g2t109 + g2t112) + g2t36*(g2t123 + g2t124));
  double a_g2t79 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t147 - f0_of_xx0*g2t47 - f1_of_xx1*g2t139 - f1_of_xx1__DD11*g2t74 + g2t136*g2t88 + g2t148*g2t88 - 2.0*g2t149*hDD_dD121 + g2t150*g2t30 - g2t19*hDD_dDD1211);
  double a_g2t80 = S[4 * Ntot + idx] * (-g2t60*hDD_dD120);
  double a_g2t85 = S[4 * Ntot + idx] * (g2t46 + g2t58);
  double a_g2t86 = S[4 * Ntot + idx] * (g2t118*g2t36 + g2t120*g2t13);
  double a_g2t87 = S[4 * Ntot + idx] * (g2t170*g2t6*lambdaU_dD21);
  double a_g2t88 = S[4 * Ntot + idx] * (g2t22*g2t70 - g2t79*(-g2t136 - g2t148));
  double a_g2t89 = S[4 * Ntot + idx] * (g2t13*g2t90 + g2t31*g2t98 + g2t36*g2t46);
  double a_g2t90 = S[4 * Ntot + idx] * (g2t13*g2t89 + g2t13*g2t92 + g2t31*g2t97 + g2t36*g2t45 + g2t36*g2t57 + g2t96);
  double a_g2t91 = S[4 * Ntot + idx] * (g2t117*g2t13);
  double a_g2t92 = S[4 * Ntot + idx] * (g2t13*(g2t90 + g2t93) + g2t31*(g2t101 + g2t98) + g2t36*(g2t46 + g2t58));
  double a_g2t93 = S[4 * Ntot + idx] * (g2t13*g2t92 + g2t36*g2t57 + g2t96);
  double a_g2t94 = S[4 * Ntot + idx] * (g2t118*g2t38 + g2t120*g2t31);
  double a_g2t96 = S[4 * Ntot + idx] * (g2t90 + g2t93);
  double a_g2t97 = S[4 * Ntot + idx] * (g2t31*g2t90 + g2t38*g2t46 + g2t43*g2t98);
  double a_g2t98 = S[4 * Ntot + idx] * (g2t105 + g2t31*g2t89 + g2t31*g2t92 + g2t38*g2t45 + g2t38*g2t57 + g2t43*g2t97);
  double a_hDD00 = S[4 * Ntot + idx] * (-(f0_of_xx0*f0_of_xx0)*g2t3*g2t32);
  double a_hDD01 = S[4 * Ntot + idx] * (-Rational_1_2*g2t14*lambdaU2 - 2.0*g2t39*g2t67);
  double a_hDD11 = S[4 * Ntot + idx] * ((f0_of_xx0*f0_of_xx0)*g2t3*g2t32);
  double a_hDD_dD010 = S[4 * Ntot + idx] * (-f0_of_xx0*g2t39*g2t67 - g2t39*g2t4);
  double a_hDD_dD011 = S[4 * Ntot + idx] * (-(f0_of_xx0*f0_of_xx0)*g2t3*g2t32 - g2t32*g2t4);
  double a_hDD_dD020 = S[4 * Ntot + idx] * (-g2t19*g2t70);
  double a_hDD_dD120 = S[4 * Ntot + idx] * (-g2t149*g2t70 - g2t60*g2t80);
  double a_hDD_dD121 = S[4 * Ntot + idx] * (-2.0*g2t149*g2t79);
  double a_hDD_dD220 = S[4 * Ntot + idx] * (g2t155*g2t39);
  double a_hDD_dD221 = S[4 * Ntot + idx] * (g2t155*g2t32);
  double a_hDD_dDD1200 = S[4 * Ntot + idx] * (-g2t19*g2t60);
  double a_hDD_dDD1211 = S[4 * Ntot + idx] * (-g2t19*g2t79);
  double a_lambdaU1 = S[4 * Ntot + idx] * (-Rational_1_2*g2t37);
  double a_lambdaU2 = S[4 * Ntot + idx] * (-f1_of_xx1__D1*g2t170*g2t2 - Rational_1_2*g2t14*hDD01);
  double a_lambdaU_dD01 = S[4 * Ntot + idx] * ((Rational_1_2)*g2t37);
  double a_lambdaU_dD11 = S[4 * Ntot + idx] * (g2t168*g2t41);
  double a_lambdaU_dD21 = S[4 * Ntot + idx] * (g2t170*g2t6*g2t87);
  a_f1_of_xx1 += S[5 * Ntot + idx] * (-4.0*(f1_of_xx1*f1_of_xx1*f1_of_xx1)*g2t177*g2t44);
  a_f1_of_xx1__D1 += S[5 * Ntot + idx] * (-g2t142*g2t39*hDD_dD120);
  double a_g2t100 = S[5 * Ntot + idx] * (2.0*g2t96);
  a_g2t101 += S[5 * Ntot + idx] * (g2t184*g2t31);
  double a_g2t102 = S[5 * Ntot + idx] * (g2t187);
  double a_g2t103 = S[5 * Ntot + idx] * (g2t187);
  a_g2t105 += S[5 * Ntot + idx] * (2.0*g2t106 + g2t171*g2t71 + g2t172*g2t30);
  double a_g2t106 = S[5 * Ntot + idx] * (2.0*g2t105);
  a_g2t107 += S[5 * Ntot + idx] * (g2t184*g2t43);
  a_g2t109 += S[5 * Ntot + idx] * (g2t38*g2t40 + g2t43*g2t71);
  a_g2t110 += S[5 * Ntot + idx] * (g2t31);
  double a_g2t111 = S[5 * Ntot + idx] * (2.0*g2t85);
  a_g2t112 += S[5 * Ntot + idx] * (g2t184*g2t38);
  a_g2t113 += S[5 * Ntot + idx] * (2.0*g2t31);
  a_g2t114 += S[5 * Ntot + idx] * (g2t31);
  a_g2t115 += S[5 * Ntot + idx] * (2.0*g2t31);
  a_g2t116 += S[5 * Ntot + idx] * (g2t31);
  a_g2t117 += S[5 * Ntot + idx] * (g2t33*g2t38 + g2t43*g2t94);
  a_g2t119 += S[5 * Ntot + idx] * (g2t31*g2t71 + g2t36*g2t40);
  a_g2t123 += S[5 * Ntot + idx] * (g2t38*g2t71 + g2t40*g2t53);
  a_g2t124 += S[5 * Ntot + idx] * (g2t175*g2t53 + g2t176*g2t38);
  a_g2t126 += S[5 * Ntot + idx] * (g2t13);
  a_g2t127 += S[5 * Ntot + idx] * (2.0*g2t13);
  a_g2t128 += S[5 * Ntot + idx] * (g2t13);
  a_g2t129 += S[5 * Ntot + idx] * (2.0*g2t13);
  a_g2t13 += S[5 * Ntot + idx] * (g2t126 + 2.0*g2t127 + g2t128 + 2.0*g2t129 + g2t185*g2t89);
  a_g2t130 += S[5 * Ntot + idx] * (g2t36);
  a_g2t131 += S[5 * Ntot + idx] * (g2t36);
  a_g2t132 += S[5 * Ntot + idx] * (2.0*g2t36);
  a_g2t133 += S[5 * Ntot + idx] * (g2t36);
  a_g2t134 += S[5 * Ntot + idx] * (2.0*g2t36);
  a_g2t137 += S[5 * Ntot + idx] * (-2.0*g2t32);
  a_g2t138 += S[5 * Ntot + idx] * (-g2t149*g2t44*hDD_dD221 - g2t20*g2t39*hDD02);
  double a_g2t140 = S[5 * Ntot + idx] * (-g2t39*hDD_dD020);
  double a_g2t142 = S[5 * Ntot + idx] * (-f1_of_xx1__D1*g2t39*hDD_dD120);
  double a_g2t144 = S[5 * Ntot + idx] * (3.0*g2t32);
  a_g2t145 += S[5 * Ntot + idx] * (-g2t32);
  a_g2t146 += S[5 * Ntot + idx] * (-g2t62*g2t79*hDD22);
  a_g2t147 += S[5 * Ntot + idx] * (-g2t25*g2t32);
  a_g2t148 += S[5 * Ntot + idx] * (-g2t178*g2t32);
  a_g2t149 += S[5 * Ntot + idx] * (-g2t138*g2t44*hDD_dD221);
  a_g2t150 += S[5 * Ntot + idx] * (g2t5*g2t79);
  a_g2t151 += S[5 * Ntot + idx] * (g2t26*g2t60 + g2t64*g2t70);
  a_g2t154 += S[5 * Ntot + idx] * (-g2t25*g2t39);
  double a_g2t156 = S[5 * Ntot + idx] * (-g2t178*g2t44);
  a_g2t159 += S[5 * Ntot + idx] * (-g2t25*g2t44);
  a_g2t160 += S[5 * Ntot + idx] * (2.0*g2t79);
  double a_g2t161 = S[5 * Ntot + idx] * (-g2t62*g2t79*hDD22);
  double a_g2t162 = S[5 * Ntot + idx] * (-g2t30*g2t32);
  a_g2t163 += S[5 * Ntot + idx] * (g2t30*g2t32);
  a_g2t164 += S[5 * Ntot + idx] * (-g2t79);
  a_g2t166 += S[5 * Ntot + idx] * (2.0*g2t70);
  a_g2t169 += S[5 * Ntot + idx] * (g2t6);
  double a_g2t17 = S[5 * Ntot + idx] * (-4.0*g2t32*g2t4);
  double a_g2t171 = S[5 * Ntot + idx] * (g2t105*g2t71 + g2t40*g2t85 + g2t66*g2t96);
  double a_g2t172 = S[5 * Ntot + idx] * (g2t105*g2t30 + g2t31*g2t93 + g2t38*g2t58);
  double a_g2t173 = S[5 * Ntot + idx] * (g2t30*g2t85 + g2t36*g2t93 + g2t53*g2t58);
  double a_g2t174 = S[5 * Ntot + idx] * (g2t38*g2t40 + g2t43*g2t71);
  double a_g2t175 = S[5 * Ntot + idx] * (g2t124*g2t53 + g2t36*g2t58);
  double a_g2t176 = S[5 * Ntot + idx] * (g2t124*g2t38 + g2t31*g2t58);
  double a_g2t177 = S[5 * Ntot + idx] * (-(f1_of_xx1*f1_of_xx1*f1_of_xx1*f1_of_xx1)*g2t44 - g2t3*g2t79);
  double a_g2t178 = S[5 * Ntot + idx] * (-g2t148*g2t32 - g2t156*g2t44 - g2t22*g2t39);
  double a_g2t179 = S[5 * Ntot + idx] * (-g2t3*g2t60);
  double a_g2t181 = S[5 * Ntot + idx] * (-hDD12*lambdaU2);
  double a_g2t182 = S[5 * Ntot + idx] * (-2.0*g2t70);
  double a_g2t183 = S[5 * Ntot + idx] * (4.0*g2t39);
  double a_g2t184 = S[5 * Ntot + idx] * (g2t101*g2t31 + g2t107*g2t43 + g2t112*g2t38);
  double a_g2t185 = S[5 * Ntot + idx] * (g2t13*g2t89 + g2t36*g2t45);
  double a_g2t186 = S[5 * Ntot + idx] * (g2t36*g2t89 + g2t45*g2t53);
  double a_g2t187 = S[5 * Ntot + idx] * (g2t102 + g2t103);
  double a_g2t20 = S[5 * Ntot + idx] * (-g2t138*g2t39*hDD02);
  a_g2t22 += S[5 * Ntot + idx] * (-g2t178*g2t39);
  double a_g2t25 = S[5 * Ntot + idx] * (-g2t147*g2t32 - g2t154*g2t39 - g2t159*g2t44 - g2t32*g2t47 - g2t60*hDD_dD220);
  double a_g2t26 = S[5 * Ntot + idx] * (g2t151*g2t60);
  a_g2t3 += S[5 * Ntot + idx] * (-g2t177*g2t79 - g2t179*g2t60);
  a_g2t30 += S[5 * Ntot + idx] * (g2t105*g2t172 + g2t173*g2t85 - g2t32*(g2t162 - g2t163));
  a_g2t31 += S[5 * Ntot + idx] * (g2t101*g2t184 + g2t110 + 2.0*g2t113 + g2t114 + 2.0*g2t115 + g2t116 + g2t119*g2t71 + g2t172*g2t93 + g2t176*g2t58);
  a_g2t32 += S[5 * Ntot + idx] * (-2.0*g2t137 + 3.0*g2t144 - g2t145 - g2t147*g2t25 - g2t148*g2t178 - g2t162*g2t30 + g2t163*g2t30 - 4.0*g2t17*g2t4 - g2t25*g2t47);
  a_g2t33 += S[5 * Ntot + idx] * (g2t38*(g2t117 + g2t98) + g2t46*g2t53);
  a_g2t36 += S[5 * Ntot + idx] * (g2t119*g2t40 + g2t130 + g2t131 + 2.0*g2t132 + g2t133 + 2.0*g2t134 + g2t173*g2t93 + g2t175*g2t58 + g2t185*g2t45 + g2t186*g2t89);
  a_g2t38 += S[5 * Ntot + idx] * (g2t109*g2t40 + g2t112*g2t184 + g2t117*g2t33 + g2t123*g2t71 + g2t124*g2t176 + g2t172*g2t58 + g2t174*g2t40 + g2t33*g2t98 + g2t46*g2t94);
  a_g2t39 += S[5 * Ntot + idx] * (-f1_of_xx1__D1*g2t142*hDD_dD120 - g2t138*g2t20*hDD02 - g2t140*hDD_dD020 - g2t154*g2t25 - g2t178*g2t22 + 4.0*g2t183);
  a_g2t4 += S[5 * Ntot + idx] * (-4.0*g2t17*g2t32 - g2t60*hDD_dDD2200 - g2t79*hDD_dDD2211);
  a_g2t40 += S[5 * Ntot + idx] * (g2t119*g2t36 + g2t123*g2t53 + g2t171*g2t85 + g2t38*(g2t109 + g2t174));
  a_g2t43 += S[5 * Ntot + idx] * (g2t107*g2t184 + g2t109*g2t71 + g2t117*g2t94 + g2t174*g2t71 + g2t94*g2t98);
  a_g2t44 += S[5 * Ntot + idx] * (-(f1_of_xx1*f1_of_xx1*f1_of_xx1*f1_of_xx1)*g2t177 - g2t138*g2t149*hDD_dD221 - g2t156*g2t178 - g2t159*g2t25);
  a_g2t45 += S[5 * Ntot + idx] * (g2t185*g2t36 + g2t186*g2t53);
  a_g2t46 += S[5 * Ntot + idx] * (g2t33*g2t53 + g2t38*g2t94);
  a_g2t47 += S[5 * Ntot + idx] * (-g2t25*g2t32);
  double a_g2t5 = S[5 * Ntot + idx] * (g2t150*g2t79);
  a_g2t53 += S[5 * Ntot + idx] * (g2t123*g2t40 + g2t124*g2t175 + g2t173*g2t58 + g2t186*g2t45 + g2t33*g2t46);
  a_g2t58 += S[5 * Ntot + idx] * (g2t172*g2t38 + g2t173*g2t53 + g2t175*g2t36 + g2t176*g2t31);
  a_g2t6 += S[5 * Ntot + idx] * (g2t169);
  a_g2t60 += S[5 * Ntot + idx] * (g2t151*g2t26 - g2t179*g2t3 - g2t25*hDD_dD220 - g2t4*hDD_dDD2200);
  double a_g2t62 = S[5 * Ntot + idx] * (-g2t79*hDD22*(g2t146 + g2t161));
  double a_g2t63 = S[5 * Ntot + idx] * (-g2t70*hDD_dD220 - g2t79*hDD_dD221);
  double a_g2t64 = S[5 * Ntot + idx] * (g2t151*g2t70);
  a_g2t66 += S[5 * Ntot + idx] * (g2t171*g2t96);
  a_g2t67 += S[5 * Ntot + idx] * (-hDD02*lambdaU2);
  a_g2t70 += S[5 * Ntot + idx] * (g2t151*g2t64 + 2.0*g2t166 - 2.0*g2t182 - g2t63*hDD_dD220);
  a_g2t71 += S[5 * Ntot + idx] * (g2t105*g2t171 + g2t119*g2t31 + g2t123*g2t38 + g2t43*(g2t109 + g2t174));
  a_g2t79 += S[5 * Ntot + idx] * (g2t150*g2t5 + 2.0*g2t160 - g2t164 - g2t177*g2t3 - g2t4*hDD_dDD2211 - g2t63*hDD_dD221 - hDD22*(g2t146*g2t62 + g2t161*g2t62));
  a_g2t85 += S[5 * Ntot + idx] * (2.0*g2t111 + g2t171*g2t40 + g2t173*g2t30);
  a_g2t89 += S[5 * Ntot + idx] * (g2t13*g2t185 + g2t186*g2t36);
  a_g2t93 += S[5 * Ntot + idx] * (g2t172*g2t31 + g2t173*g2t36);
  a_g2t94 += S[5 * Ntot + idx] * (g2t38*g2t46 + g2t43*(g2t117 + g2t98));
  a_g2t96 += S[5 * Ntot + idx] * (2.0*g2t100 + g2t171*g2t66 + 2.0*g2t99);
  a_g2t98 += S[5 * Ntot + idx] * (g2t33*g2t38 + g2t43*g2t94);
  double a_g2t99 = S[5 * Ntot + idx] * (2.0*g2t96);
  double a_hDD02 = S[5 * Ntot + idx] * (-g2t138*g2t20*g2t39 - g2t67*lambdaU2);
  double a_hDD12 = S[5 * Ntot + idx] * (-g2t181*lambdaU2);
  double a_hDD22 = S[5 * Ntot + idx] * (-g2t79*(g2t146*g2t62 + g2t161*g2t62));
  a_hDD_dD020 += S[5 * Ntot + idx] * (-g2t140*g2t39);
  a_hDD_dD120 += S[5 * Ntot + idx] * (-f1_of_xx1__D1*g2t142*g2t39);
  a_hDD_dD220 += S[5 * Ntot + idx] * (-g2t25*g2t60 - g2t63*g2t70);
  a_hDD_dD221 += S[5 * Ntot + idx] * (-g2t138*g2t149*g2t44 - g2t63*g2t79);
  double a_hDD_dDD2200 = S[5 * Ntot + idx] * (-g2t4*g2t60);
  double a_hDD_dDD2211 = S[5 * Ntot + idx] * (-g2t4*g2t79);
  a_lambdaU2 += S[5 * Ntot + idx] * (-g2t181*hDD12 - g2t67*hDD02);
  a_g2t107 += a_g2t187 * (3.0);
  a_g2t112 += a_g2t186 * (3.0);
  a_g2t101 += a_g2t185 * (3.0);
  a_g2t97 += a_g2t184 * (3.0);
  double a_g2t143 = a_g2t183 * (g2t41);
  a_g2t41 += a_g2t183 * (g2t143);
  a_g2t179 += a_g2t182 * (g2t181);
  a_g2t181 += a_g2t182 * (g2t179);
  a_g2t4 += a_g2t182 * (hDD_dDD2201);
  double a_hDD_dDD2201 = a_g2t182 * (g2t4);
  a_f0_of_xx0 += a_g2t181 * (g2t61);
  a_g2t61 += a_g2t181 * (f0_of_xx0);
  a_hDD22 += a_g2t179 * (4.0);
  a_g2t61 += a_g2t178 * (2.0);
  double a_g2t35 = a_g2t177 * (hDD_dD220);
  a_hDD_dD220 += a_g2t177 * (g2t35);
  a_g2t71 += a_g2t176 * (2.0);
  a_g2t40 += a_g2t175 * (2.0);
  a_g2t112 += a_g2t174 * (2.0);
  a_g2t33 += a_g2t173 * (2.0);
  a_g2t94 += a_g2t172 * (2.0);
  a_g2t20 += a_g2t171 * (g2t28);
  double a_g2t28 = a_g2t171 * (g2t20);
  a_g2t41 += a_g2t170 * (Rational_1_2);
  a_g2t167 += a_g2t169 * (1.0);
  a_g2t41 += a_g2t169 * (g2t88*lambdaU1);
  a_g2t88 += a_g2t169 * (g2t41*lambdaU1);
  a_lambdaU1 += a_g2t169 * (g2t41*g2t88);
  a_g2t30 += a_g2t168 * (Rational_1_2);
  a_g2t41 += a_g2t167 * (lambdaU0);
  double a_lambdaU0 = a_g2t167 * (g2t41);
  a_g2t26 += a_g2t166 * (g2t88);
  a_g2t88 += a_g2t166 * (g2t26);
  a_g2t156 += a_g2t165 * (g2t41);
  a_g2t41 += a_g2t165 * (g2t156);
  a_g2t150 += a_g2t164 * (-g2t5);
  a_g2t5 += a_g2t164 * (-g2t150);
  a_g2t162 += a_g2t163 * (-1.0);
  a_g2t146 += a_g2t162 * (1.0);
  a_g2t161 += a_g2t162 * (1.0);
  a_f1_of_xx1 += a_g2t161 * (f1_of_xx1__DD11);
  a_f1_of_xx1__DD11 += a_g2t161 * (f1_of_xx1);
  a_g2t64 += a_g2t160 * (g2t88);
  a_g2t88 += a_g2t160 * (g2t64);
  double a_g2t34 = a_g2t159 * (g2t61);
  a_g2t61 += a_g2t159 * (g2t34);
  a_g2t67 += a_g2t159 * (hDD00 - hDD22);
  a_hDD00 += a_g2t159 * (g2t67);
  a_hDD22 += a_g2t159 * (-g2t67);
  double a_g2t0 = a_g2t158 * (g2t82);
  double a_g2t82 = a_g2t158 * (g2t0);
  a_g2t156 += a_g2t157 * (g2t88);
  a_g2t88 += a_g2t157 * (g2t156);
  a_g2t1 += a_g2t156 * (g2t61);
  a_g2t155 += a_g2t156 * (-hDD22);
  a_g2t4 += a_g2t156 * (hDD01);
  a_g2t61 += a_g2t156 * (g2t1);
  a_hDD01 += a_g2t156 * (g2t4);
  a_hDD22 += a_g2t156 * (-g2t155);
  a_g2t0 += a_g2t155 * (g2t61);
  a_g2t61 += a_g2t155 * (g2t0);
  a_g2t14 += a_g2t154 * (hDD_dD020);
  a_g2t28 += a_g2t154 * (1.0);
  a_hDD_dD020 += a_g2t154 * (g2t14);
  double a_g2t141 = a_g2t153 * (g2t20);
  a_g2t19 += a_g2t153 * (hDD_dDD1201);
  a_g2t20 += a_g2t153 * (g2t141);
  a_g2t80 += a_g2t153 * (hDD_dD121);
  a_hDD_dD121 += a_g2t153 * (g2t80);
  double a_hDD_dDD1201 = a_g2t153 * (g2t19);
  a_g2t136 += a_g2t152 * (g2t41);
  a_g2t41 += a_g2t152 * (g2t136);
  a_g2t41 += a_g2t151 * (2.0);
  a_f1_of_xx1__DD11 += a_g2t150 * (g2t87);
  a_g2t146 += a_g2t150 * (-1.0/g2t3);
  a_g2t3 += a_g2t150 * (g2t146/(g2t3*g2t3));
  a_g2t87 += a_g2t150 * (f1_of_xx1__DD11);
  a_f1_of_xx1__D1 += a_g2t149 * (g2t0);
  a_g2t0 += a_g2t149 * (f1_of_xx1__D1);
  double a_g2t73 = a_g2t148 * (1.0);
  double a_g2t75 = a_g2t148 * (1.0);
  a_g2t135 += a_g2t147 * (-1.0);
  double a_g2t16 = a_g2t147 * (-1.0);
  a_f1_of_xx1__D1 += a_g2t146 * (2.0*f1_of_xx1__D1);
  a_g2t144 += a_g2t145 * (-1.0);
  a_g2t143 += a_g2t144 * (g2t88);
  a_g2t88 += a_g2t144 * (g2t143);
  a_g2t140 += a_g2t143 * (hDD02);
  a_g2t141 += a_g2t143 * (g2t142);
  a_g2t142 += a_g2t143 * (g2t141);
  a_hDD02 += a_g2t143 * (g2t140);
  a_g2t4 += a_g2t142 * (2.0);
  a_f1_of_xx1__D1 += a_g2t141 * (hDD12);
  a_hDD12 += a_g2t141 * (f1_of_xx1__D1);
  a_g2t138 += a_g2t140 * (g2t62);
  a_g2t62 += a_g2t140 * (g2t138);
  a_g2t35 += a_g2t139 * (hDD_dD120);
  a_hDD_dD120 += a_g2t139 * (g2t35);
  a_f1_of_xx1 += a_g2t138 * (3.0*(f1_of_xx1*f1_of_xx1));
  a_g2t136 += a_g2t137 * (g2t61);
  a_g2t61 += a_g2t137 * (g2t136);
  double a_g2t29 = a_g2t136 * (1.0);
  a_g2t73 += a_g2t136 * (1.0);
  a_g2t14 += a_g2t135 * (hDD12);
  a_hDD12 += a_g2t135 * (g2t14);
  a_g2t58 += a_g2t134 * (g2t86);
  a_g2t86 += a_g2t134 * (g2t58);
  a_g2t46 += a_g2t133 * (g2t86);
  a_g2t86 += a_g2t133 * (g2t46);
  a_g2t124 += a_g2t132 * (g2t66);
  a_g2t66 += a_g2t132 * (g2t124);
  a_g2t123 += a_g2t131 * (g2t66);
  a_g2t66 += a_g2t131 * (g2t123);
  a_g2t33 += a_g2t130 * (g2t90);
  a_g2t90 += a_g2t130 * (g2t33);
  a_g2t86 += a_g2t129 * (g2t93);
  a_g2t93 += a_g2t129 * (g2t86);
  a_g2t86 += a_g2t128 * (g2t90);
  a_g2t90 += a_g2t128 * (g2t86);
  a_g2t58 += a_g2t127 * (g2t66);
  a_g2t66 += a_g2t127 * (g2t58);
  a_g2t119 += a_g2t126 * (g2t66);
  a_g2t66 += a_g2t126 * (g2t119);
  a_g2t91 += a_g2t125 * (2.0);
  double a_g2t104 = a_g2t124 * (g2t6);
  a_g2t30 += a_g2t124 * (g2t95);
  a_g2t37 += a_g2t124 * (g2t84);
  a_g2t6 += a_g2t124 * (g2t104);
  double a_g2t84 = a_g2t124 * (g2t37);
  double a_g2t95 = a_g2t124 * (g2t30);
  a_g2t33 += a_g2t123 * (g2t34);
  a_g2t34 += a_g2t123 * (g2t33);
  a_g2t37 += a_g2t123 * (g2t45);
  a_g2t40 += a_g2t123 * (g2t8);
  a_g2t45 += a_g2t123 * (g2t37);
  double a_g2t8 = a_g2t123 * (g2t40);
  a_g2t104 += a_g2t122 * (g2t30);
  a_g2t2 += a_g2t122 * (g2t95);
  a_g2t30 += a_g2t122 * (g2t104);
  a_g2t34 += a_g2t122 * (g2t84);
  a_g2t84 += a_g2t122 * (g2t34);
  a_g2t95 += a_g2t122 * (g2t2);
  a_g2t52 += a_g2t121 * (2.0);
  a_g2t2 += a_g2t120 * (g2t92);
  a_g2t30 += a_g2t120 * (g2t91);
  a_g2t34 += a_g2t120 * (g2t78);
  a_g2t78 += a_g2t120 * (g2t34);
  a_g2t91 += a_g2t120 * (g2t30);
  a_g2t92 += a_g2t120 * (g2t2);
  a_g2t34 += a_g2t119 * (g2t86);
  a_g2t37 += a_g2t119 * (g2t89);
  a_g2t66 += a_g2t119 * (g2t8);
  a_g2t8 += a_g2t119 * (g2t66);
  a_g2t86 += a_g2t119 * (g2t34);
  a_g2t89 += a_g2t119 * (g2t37);
  a_g2t2 += a_g2t118 * (g2t57);
  a_g2t30 += a_g2t118 * (g2t52);
  a_g2t34 += a_g2t118 * (g2t56);
  a_g2t52 += a_g2t118 * (g2t30);
  a_g2t56 += a_g2t118 * (g2t34);
  a_g2t57 += a_g2t118 * (g2t2);
  a_g2t101 += a_g2t117 * (2.0);
  a_g2t90 += a_g2t116 * (g2t94);
  a_g2t94 += a_g2t116 * (g2t90);
  a_g2t101 += a_g2t115 * (g2t86);
  a_g2t86 += a_g2t115 * (g2t101);
  a_g2t86 += a_g2t114 * (g2t98);
  a_g2t98 += a_g2t114 * (g2t86);
  a_g2t112 += a_g2t113 * (g2t66);
  a_g2t66 += a_g2t113 * (g2t112);
  a_g2t111 += a_g2t112 * (1.0);
  a_g2t30 += a_g2t112 * (g2t33);
  a_g2t33 += a_g2t112 * (g2t30);
  a_g2t37 += a_g2t112 * (g2t40);
  a_g2t40 += a_g2t112 * (g2t37);
  a_g2t45 += a_g2t111 * (g2t6);
  a_g2t6 += a_g2t111 * (g2t45);
  a_g2t109 += a_g2t110 * (g2t66);
  a_g2t66 += a_g2t110 * (g2t109);
  a_g2t34 += a_g2t109 * (g2t94);
  a_g2t37 += a_g2t109 * (g2t97);
  a_g2t71 += a_g2t109 * (g2t8);
  a_g2t8 += a_g2t109 * (g2t71);
  a_g2t94 += a_g2t109 * (g2t34);
  a_g2t97 += a_g2t109 * (g2t37);
  a_g2t89 += a_g2t108 * (2.0);
  a_g2t106 += a_g2t107 * (1.0);
  a_g2t30 += a_g2t107 * (g2t94);
  a_g2t37 += a_g2t107 * (g2t71);
  a_g2t71 += a_g2t107 * (g2t37);
  a_g2t94 += a_g2t107 * (g2t30);
  a_g2t6 += a_g2t106 * (g2t97);
  a_g2t97 += a_g2t106 * (g2t6);
  a_g2t102 += a_g2t105 * (1.0);
  a_g2t103 += a_g2t105 * (1.0);
  a_g2t104 += a_g2t105 * (g2t60);
  a_g2t36 += a_g2t105 * (g2t52);
  a_g2t44 += a_g2t105 * (g2t97);
  a_g2t52 += a_g2t105 * (g2t36);
  a_g2t60 += a_g2t105 * (g2t104);
  a_g2t79 += a_g2t105 * (g2t91);
  a_g2t91 += a_g2t105 * (g2t79);
  a_g2t97 += a_g2t105 * (g2t44);
  a_g2t32 += a_g2t104 * (g2t83);
  a_g2t39 += a_g2t104 * (hDD_dD000);
  a_g2t44 += a_g2t104 * (g2t81);
  double a_g2t81 = a_g2t104 * (g2t44);
  double a_g2t83 = a_g2t104 * (g2t32);
  double a_hDD_dD000 = a_g2t104 * (g2t39);
  a_g2t38 += a_g2t103 * (g2t45);
  a_g2t45 += a_g2t103 * (g2t38);
  a_g2t31 += a_g2t102 * (g2t89);
  a_g2t89 += a_g2t102 * (g2t31);
  a_g2t100 += a_g2t101 * (1.0);
  a_g2t37 += a_g2t101 * (g2t66);
  a_g2t66 += a_g2t101 * (g2t37);
  a_g2t99 += a_g2t101 * (1.0);
  a_g2t30 += a_g2t100 * (g2t86);
  a_g2t86 += a_g2t100 * (g2t30);
  a_g2t6 += a_g2t99 * (g2t89);
  a_g2t89 += a_g2t99 * (g2t6);
  a_g2t2 += a_g2t98 * (g2t94);
  a_g2t30 += a_g2t98 * (g2t97);
  a_g2t34 += a_g2t98 * (g2t71);
  a_g2t71 += a_g2t98 * (g2t34);
  a_g2t94 += a_g2t98 * (g2t2);
  a_g2t97 += a_g2t98 * (g2t30);
  a_g2t32 += a_g2t97 * (g2t69);
  a_g2t39 += a_g2t97 * (g2t68);
  double a_g2t68 = a_g2t97 * (g2t39);
  double a_g2t69 = a_g2t97 * (g2t32);
  a_g2t31 += a_g2t96 * (g2t86);
  a_g2t33 += a_g2t96 * (g2t38);
  a_g2t36 += a_g2t96 * (g2t57);
  a_g2t38 += a_g2t96 * (g2t33);
  a_g2t44 += a_g2t96 * (g2t94);
  a_g2t57 += a_g2t96 * (g2t36);
  a_g2t60 += a_g2t96 * (g2t95);
  a_g2t79 += a_g2t96 * (g2t92);
  a_g2t86 += a_g2t96 * (g2t31);
  a_g2t92 += a_g2t96 * (g2t79);
  a_g2t94 += a_g2t96 * (g2t44);
  a_g2t95 += a_g2t96 * (g2t60);
  a_g2t32 += a_g2t95 * (g2t81);
  a_g2t70 += a_g2t95 * (hDD_dD000);
  a_g2t79 += a_g2t95 * (g2t83);
  a_g2t81 += a_g2t95 * (g2t32);
  a_g2t83 += a_g2t95 * (g2t79);
  a_hDD_dD000 += a_g2t95 * (g2t70);
  a_g2t61 += a_g2t94 * (1.0);
  a_g2t68 += a_g2t94 * (g2t70);
  a_g2t69 += a_g2t94 * (g2t79);
  a_g2t70 += a_g2t94 * (g2t68);
  a_g2t79 += a_g2t94 * (g2t69);
  a_g2t30 += a_g2t93 * (g2t92);
  a_g2t37 += a_g2t93 * (g2t78);
  a_g2t6 += a_g2t93 * (g2t91);
  a_g2t78 += a_g2t93 * (g2t37);
  a_g2t91 += a_g2t93 * (g2t6);
  a_g2t92 += a_g2t93 * (g2t30);
  a_g2t32 += a_g2t92 * (g2t76);
  a_g2t70 += a_g2t92 * (g2t72);
  double a_g2t72 = a_g2t92 * (g2t70);
  double a_g2t76 = a_g2t92 * (g2t32);
  a_g2t77 += a_g2t92 * (g2t79);
  a_g2t79 += a_g2t92 * (g2t77);
  a_g2t32 += a_g2t91 * (g2t77);
  a_g2t39 += a_g2t91 * (g2t72);
  a_g2t44 += a_g2t91 * (g2t76);
  a_g2t72 += a_g2t91 * (g2t39);
  a_g2t76 += a_g2t91 * (g2t44);
  a_g2t77 += a_g2t91 * (g2t32);
  a_g2t2 += a_g2t90 * (g2t86);
  a_g2t30 += a_g2t90 * (g2t89);
  a_g2t34 += a_g2t90 * (g2t66);
  a_g2t66 += a_g2t90 * (g2t34);
  a_g2t86 += a_g2t90 * (g2t2);
  a_g2t89 += a_g2t90 * (g2t30);
  a_g2t39 += a_g2t89 * (g2t59);
  a_g2t44 += a_g2t89 * (g2t65);
  double a_g2t59 = a_g2t89 * (g2t39);
  double a_g2t65 = a_g2t89 * (g2t44);
  a_g2t88 += a_g2t89 * (-1.0);
  a_f1_of_xx1__D1 += a_g2t88 * (g2t87);
  a_g2t87 += a_g2t88 * (f1_of_xx1__D1);
  a_f1_of_xx1 += a_g2t87 * (-1.0/(f1_of_xx1*f1_of_xx1));
  a_g2t32 += a_g2t86 * (g2t65);
  a_g2t59 += a_g2t86 * (g2t70);
  a_g2t65 += a_g2t86 * (g2t32);
  a_g2t70 += a_g2t86 * (g2t59);
  a_g2t31 += a_g2t85 * (g2t66);
  a_g2t36 += a_g2t85 * (g2t56);
  a_g2t38 += a_g2t85 * (g2t40);
  a_g2t40 += a_g2t85 * (g2t38);
  a_g2t44 += a_g2t85 * (g2t71);
  a_g2t56 += a_g2t85 * (g2t36);
  a_g2t60 += a_g2t85 * (g2t84);
  a_g2t66 += a_g2t85 * (g2t31);
  a_g2t71 += a_g2t85 * (g2t44);
  a_g2t78 += a_g2t85 * (g2t79);
  a_g2t79 += a_g2t85 * (g2t78);
  a_g2t84 += a_g2t85 * (g2t60);
  a_g2t39 += a_g2t84 * (g2t81);
  a_g2t60 += a_g2t84 * (hDD_dD000);
  a_g2t70 += a_g2t84 * (g2t83);
  a_g2t81 += a_g2t84 * (g2t39);
  a_g2t83 += a_g2t84 * (g2t70);
  a_hDD_dD000 += a_g2t84 * (g2t60);
  a_g2t20 += a_g2t83 * (hDD_dD010);
  a_g2t82 += a_g2t83 * (1.0);
  double a_hDD_dD001 = a_g2t83 * (-1.0);
  a_hDD_dD010 += a_g2t83 * (g2t20);
  a_hDD01 += a_g2t82 * (2.0);
  a_g2t28 += a_g2t81 * (2.0);
  a_g2t80 += a_g2t81 * (hDD_dD020);
  a_hDD_dD020 += a_g2t81 * (g2t80);
  a_f1_of_xx1 += a_g2t80 * (g2t20);
  a_g2t20 += a_g2t80 * (f1_of_xx1);
  a_g2t13 += a_g2t79 * (Rational_1_2);
  a_f0_of_xx0 += a_g2t78 * (1.0);
  a_g2t39 += a_g2t78 * (g2t76);
  a_g2t60 += a_g2t78 * (g2t72);
  a_g2t70 += a_g2t78 * (g2t77);
  a_g2t72 += a_g2t78 * (g2t60);
  a_g2t76 += a_g2t78 * (g2t39);
  a_g2t77 += a_g2t78 * (g2t70);
  a_g2t0 += a_g2t77 * (hDD_dD111);
  double a_hDD_dD111 = a_g2t77 * (g2t0);
  a_g2t73 += a_g2t76 * (2.0);
  a_g2t75 += a_g2t76 * (2.0);
  a_f1_of_xx1__D1 += a_g2t75 * (g2t74);
  a_g2t74 += a_g2t75 * (f1_of_xx1__D1);
  a_g2t0 += a_g2t74 * (hDD12);
  a_hDD12 += a_g2t74 * (g2t0);
  a_g2t19 += a_g2t73 * (hDD_dD121);
  a_hDD_dD121 += a_g2t73 * (g2t19);
  a_f0_of_xx0 += a_g2t72 * (2.0*hDD_dD011);
  double a_g2t51 = a_g2t72 * (-1.0);
  a_hDD_dD011 += a_g2t72 * (2.0*f0_of_xx0);
  a_g2t60 += a_g2t71 * (g2t68);
  a_g2t67 += a_g2t71 * (1.0);
  a_g2t68 += a_g2t71 * (g2t60);
  a_g2t69 += a_g2t71 * (g2t70);
  a_g2t70 += a_g2t71 * (g2t69);
  a_g2t36 += a_g2t70 * (Rational_1_2);
  a_g2t65 += a_g2t69 * (-1.0);
  double a_g2t27 = a_g2t68 * (-1.0);
  a_f0_of_xx0 += a_g2t67 * (g2t3);
  a_g2t3 += a_g2t67 * (f0_of_xx0);
  a_g2t39 += a_g2t66 * (g2t65);
  a_g2t59 += a_g2t66 * (g2t60);
  a_g2t60 += a_g2t66 * (g2t59);
  a_g2t65 += a_g2t66 * (g2t39);
  a_g2t63 += a_g2t65 * (1.0);
  a_g2t64 += a_g2t65 * (1.0);
  a_g2t4 += a_g2t64 * (hDD_dD221);
  a_g2t63 += a_g2t64 * (hDD22);
  a_hDD22 += a_g2t64 * (g2t63);
  a_hDD_dD221 += a_g2t64 * (g2t4);
  a_g2t61 += a_g2t63 * (g2t62);
  a_g2t62 += a_g2t63 * (g2t61);
  a_g2t0 += a_g2t62 * (2.0);
  a_f1_of_xx1 += a_g2t61 * (f1_of_xx1__D1);
  a_f1_of_xx1__D1 += a_g2t61 * (f1_of_xx1);
  a_g2t53 += a_g2t60 * (Rational_1_2);
  double a_g2t23 = a_g2t59 * (-1.0);
  a_g2t30 += a_g2t58 * (g2t57);
  a_g2t37 += a_g2t58 * (g2t56);
  a_g2t52 += a_g2t58 * (g2t6);
  a_g2t56 += a_g2t58 * (g2t37);
  a_g2t57 += a_g2t58 * (g2t30);
  a_g2t6 += a_g2t58 * (g2t52);
  a_g2t13 += a_g2t57 * (g2t55);
  a_g2t32 += a_g2t57 * (g2t48);
  a_g2t36 += a_g2t57 * (g2t54);
  double a_g2t42 = a_g2t57 * (1.0);
  double a_g2t48 = a_g2t57 * (g2t32);
  double a_g2t54 = a_g2t57 * (g2t36);
  double a_g2t55 = a_g2t57 * (g2t13);
  a_g2t36 += a_g2t56 * (g2t55);
  a_g2t39 += a_g2t56 * (g2t48);
  a_g2t48 += a_g2t56 * (g2t39);
  a_g2t53 += a_g2t56 * (g2t54);
  a_g2t54 += a_g2t56 * (g2t53);
  a_g2t55 += a_g2t56 * (g2t36);
  a_g2t51 += a_g2t55 * (Rational_1_2);
  a_hDD_dD001 += a_g2t54 * (Rational_1_2);
  double a_g2t11 = a_g2t53 * (-g2t12);
  double a_g2t12 = a_g2t53 * (-g2t11 + g2t2*g2t6);
  a_g2t2 += a_g2t53 * (g2t12*g2t6);
  a_g2t6 += a_g2t53 * (g2t12*g2t2);
  a_g2t32 += a_g2t52 * (g2t51);
  a_g2t39 += a_g2t52 * (hDD_dD001);
  a_g2t44 += a_g2t52 * (g2t48);
  a_g2t48 += a_g2t52 * (g2t44);
  a_g2t51 += a_g2t52 * (g2t32);
  a_hDD_dD001 += a_g2t52 * (g2t39);
  a_g2t20 += a_g2t51 * (1.0);
  a_g2t50 += a_g2t51 * (1.0);
  a_g2t20 += a_g2t50 * (hDD11);
  a_g2t49 += a_g2t50 * (1.0);
  a_hDD11 += a_g2t50 * (g2t20);
  a_g2t0 += a_g2t49 * (hDD_dD110);
  double a_hDD_dD110 = a_g2t49 * (g2t0);
  a_g2t22 += a_g2t48 * (1.0);
  a_g2t47 += a_g2t48 * (1.0);
  double a_g2t15 = a_g2t47 * (1.0);
  a_g2t18 += a_g2t47 * (1.0);
  a_g2t2 += a_g2t46 * (g2t33);
  a_g2t30 += a_g2t46 * (g2t45);
  a_g2t33 += a_g2t46 * (g2t2);
  a_g2t34 += a_g2t46 * (g2t40);
  a_g2t40 += a_g2t46 * (g2t34);
  a_g2t45 += a_g2t46 * (g2t30);
  double a_g2t24 = a_g2t45 * (g2t31);
  a_g2t27 += a_g2t45 * (g2t44);
  a_g2t31 += a_g2t45 * (g2t24);
  a_g2t42 += a_g2t45 * (1.0);
  a_g2t44 += a_g2t45 * (g2t27);
  a_g2t43 += a_g2t44 * (Rational_1_2);
  a_g2t12 += a_g2t43 * (g2t2*g2t8 - g2t7);
  a_g2t2 += a_g2t43 * (g2t12*g2t8);
  double a_g2t7 = a_g2t43 * (-g2t12);
  a_g2t8 += a_g2t43 * (g2t12*g2t2);
  a_g2t41 += a_g2t42 * (-1.0);
  a_f0_of_xx0 += a_g2t41 * (-1.0/(f0_of_xx0*f0_of_xx0));
  a_g2t24 += a_g2t40 * (g2t36);
  a_g2t27 += a_g2t40 * (g2t39);
  a_g2t36 += a_g2t40 * (g2t24);
  a_g2t39 += a_g2t40 * (g2t27);
  a_g2t38 += a_g2t39 * (Rational_1_2);
  a_g2t12 += a_g2t38 * (-g2t2*g2t37 + g2t21*g2t35*hDD01);
  a_g2t2 += a_g2t38 * (-g2t12*g2t37);
  a_g2t21 += a_g2t38 * (g2t12*g2t35*hDD01);
  a_g2t35 += a_g2t38 * (g2t12*g2t21*hDD01);
  a_g2t37 += a_g2t38 * (-g2t12*g2t2);
  a_hDD01 += a_g2t38 * (g2t12*g2t21*g2t35);
  a_f0_of_xx0 += a_g2t37 * (g2t28);
  a_g2t28 += a_g2t37 * (f0_of_xx0);
  a_g2t12 += a_g2t36 * (g2t3*g2t35*hDD02*hDD12 - g2t34*g2t6);
  a_g2t3 += a_g2t36 * (g2t12*g2t35*hDD02*hDD12);
  a_g2t34 += a_g2t36 * (-g2t12*g2t6);
  a_g2t35 += a_g2t36 * (g2t12*g2t3*hDD02*hDD12);
  a_g2t6 += a_g2t36 * (-g2t12*g2t34);
  a_hDD02 += a_g2t36 * (g2t12*g2t3*g2t35*hDD12);
  a_hDD12 += a_g2t36 * (g2t12*g2t3*g2t35*hDD02);
  a_f0_of_xx0 += a_g2t35 * (3.0*(f0_of_xx0*f0_of_xx0));
  a_f0_of_xx0 += a_g2t34 * (hDD01);
  a_hDD01 += a_g2t34 * (f0_of_xx0);
  a_g2t13 += a_g2t33 * (g2t24);
  a_g2t24 += a_g2t33 * (g2t13);
  a_g2t27 += a_g2t33 * (g2t32);
  a_g2t32 += a_g2t33 * (g2t27);
  a_g2t31 += a_g2t32 * (Rational_1_2);
  a_g2t12 += a_g2t31 * (g2t29*hDD01 - g2t30*g2t8);
  a_g2t29 += a_g2t31 * (g2t12*hDD01);
  a_g2t30 += a_g2t31 * (-g2t12*g2t8);
  a_g2t8 += a_g2t31 * (-g2t12*g2t30);
  a_hDD01 += a_g2t31 * (g2t12*g2t29);
  a_g2t19 += a_g2t30 * (hDD12);
  a_hDD12 += a_g2t30 * (g2t19);
  a_g2t0 += a_g2t29 * (g2t28);
  a_g2t28 += a_g2t29 * (g2t0);
  a_f1_of_xx1 += a_g2t28 * (hDD02);
  a_hDD02 += a_g2t28 * (f1_of_xx1);
  a_g2t25 += a_g2t27 * (1.0);
  a_g2t26 += a_g2t27 * (1.0);
  a_g2t25 += a_g2t26 * (hDD22);
  a_g2t4 += a_g2t26 * (hDD_dD220);
  a_hDD22 += a_g2t26 * (g2t25);
  a_hDD_dD220 += a_g2t26 * (g2t4);
  a_g2t20 += a_g2t25 * (g2t3);
  a_g2t3 += a_g2t25 * (g2t20);
  a_g2t23 += a_g2t24 * (Rational_1_2);
  a_g2t16 += a_g2t23 * (1.0);
  a_g2t18 += a_g2t23 * (-1.0);
  a_g2t22 += a_g2t23 * (1.0);
  a_g2t19 += a_g2t22 * (hDD_dD120);
  a_g2t20 += a_g2t22 * (g2t21);
  a_g2t21 += a_g2t22 * (g2t20);
  a_hDD_dD120 += a_g2t22 * (g2t19);
  a_f1_of_xx1 += a_g2t21 * (hDD12);
  a_hDD12 += a_g2t21 * (f1_of_xx1);
  a_f0_of_xx0 += a_g2t20 * (2.0);
  a_f1_of_xx1 += a_g2t19 * (g2t0);
  a_g2t0 += a_g2t19 * (f1_of_xx1);
  a_f0_of_xx0 += a_g2t18 * (g2t17);
  a_g2t17 += a_g2t18 * (f0_of_xx0);
  a_f1_of_xx1__D1 += a_g2t17 * (hDD02);
  a_hDD02 += a_g2t17 * (f1_of_xx1__D1);
  a_g2t15 += a_g2t16 * (-1.0);
  a_g2t14 += a_g2t15 * (hDD_dD021);
  double a_hDD_dD021 = a_g2t15 * (g2t14);
  a_f0_of_xx0 += a_g2t14 * (f1_of_xx1);
  a_f1_of_xx1 += a_g2t14 * (f0_of_xx0);
  a_g2t12 += a_g2t13 * (g2t6*g2t8 - g2t9);
  a_g2t6 += a_g2t13 * (g2t12*g2t8);
  a_g2t8 += a_g2t13 * (g2t12*g2t6);
  double a_g2t9 = a_g2t13 * (-g2t12);
  double a_g2t10 = a_g2t12 * (-2.0*g2t3*hDD01*hDD02*hDD12/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t11 += a_g2t12 * (g2t8/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t2 += a_g2t12 * ((-g2t6*g2t8 + g2t9)/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t3 += a_g2t12 * (-2.0*g2t10*hDD01*hDD02*hDD12/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t6 += a_g2t12 * ((-g2t2*g2t8 + g2t7)/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t7 += a_g2t12 * (g2t6/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t8 += a_g2t12 * ((g2t11 - g2t2*g2t6)/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t9 += a_g2t12 * (g2t2/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_hDD01 += a_g2t12 * (-2.0*g2t10*g2t3*hDD02*hDD12/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_hDD02 += a_g2t12 * (-2.0*g2t10*g2t3*hDD01*hDD12/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_hDD12 += a_g2t12 * (-2.0*g2t10*g2t3*hDD01*hDD02/((2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)*(2.0*g2t10*g2t3*hDD01*hDD02*hDD12 - g2t11*g2t8 + g2t2*g2t6*g2t8 - g2t2*g2t9 - g2t6*g2t7)));
  a_g2t10 += a_g2t11 * (g2t3*(hDD12*hDD12));
  a_g2t3 += a_g2t11 * (g2t10*(hDD12*hDD12));
  a_hDD12 += a_g2t11 * (2.0*g2t10*g2t3*hDD12);
  a_f0_of_xx0 += a_g2t10 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_g2t4 += a_g2t9 * ((hDD02*hDD02));
  a_hDD02 += a_g2t9 * (2.0*g2t4*hDD02);
  a_hDD00 += a_g2t8 * (1.0);
  a_g2t0 += a_g2t7 * ((hDD01*hDD01));
  a_hDD01 += a_g2t7 * (2.0*g2t0*hDD01);
  a_g2t4 += a_g2t6 * (1.0);
  a_g2t5 += a_g2t6 * (1.0);
  a_g2t4 += a_g2t5 * (hDD22);
  a_hDD22 += a_g2t5 * (g2t4);
  a_g2t0 += a_g2t4 * (g2t3);
  a_g2t3 += a_g2t4 * (g2t0);
  a_f1_of_xx1 += a_g2t3 * (2.0*f1_of_xx1);
  a_g2t0 += a_g2t2 * (1.0);
  a_g2t1 += a_g2t2 * (1.0);
  a_g2t0 += a_g2t1 * (hDD11);
  a_hDD11 += a_g2t1 * (g2t0);
  a_f0_of_xx0 += a_g2t0 * (2.0*f0_of_xx0);
  red[65 * 64 + lane] = a_hDD00;
  red[66 * 64 + lane] = a_hDD01;
  red[67 * 64 + lane] = a_hDD02;
  red[68 * 64 + lane] = a_hDD11;
  red[69 * 64 + lane] = a_hDD12;
  red[70 * 64 + lane] = a_hDD22;
  red[71 * 64 + lane] = a_hDD_dD000;
  red[72 * 64 + lane] = a_hDD_dD001;
  red[73 * 64 + lane] = a_hDD_dD010;
  red[74 * 64 + lane] = a_hDD_dD011;
  red[75 * 64 + lane] = a_hDD_dD020;
  red[76 * 64 + lane] = a_hDD_dD021;
  red[77 * 64 + lane] = a_hDD_dD110;
  red[78 * 64 + lane] = a_hDD_dD111;
  red[79 * 64 + lane] = a_hDD_dD120;
  red[80 * 64 + lane] = a_hDD_dD121;
  red[81 * 64 + lane] = a_hDD_dD220;
  red[82 * 64 + lane] = a_hDD_dD221;
  red[83 * 64 + lane] = a_hDD_dDD1200;
  red[84 * 64 + lane] = a_hDD_dDD1201;
  red[85 * 64 + lane] = a_hDD_dDD1211;
  red[86 * 64 + lane] = a_hDD_dDD2200;
  red[87 * 64 + lane] = a_hDD_dDD2201;
  red[88 * 64 + lane] = a_hDD_dDD2211;
  red[89 * 64 + lane] = a_lambdaU0;
  red[90 * 64 + lane] = a_lambdaU1;
  red[91 * 64 + lane] = a_lambdaU2;
  red[92 * 64 + lane] = a_lambdaU_dD01;
  red[93 * 64 + lane] = a_lambdaU_dD11;
  red[94 * 64 + lane] = a_lambdaU_dD21;
  break;
  }
  default:
    break;
  }
  __syncthreads();
  if (!active) return;
  switch (group) {
  case 0:
    S[165 * Ntot + idx] = red[0 * 64 + lane] + red[32 * 64 + lane] + red[65 * 64 + lane];
    S[168 * Ntot + idx] = red[3 * 64 + lane] + red[35 * 64 + lane] + red[68 * 64 + lane];
    S[171 * Ntot + idx] = red[6 * 64 + lane] + red[38 * 64 + lane] + red[71 * 64 + lane];
    S[174 * Ntot + idx] = red[9 * 64 + lane] + red[41 * 64 + lane] + red[74 * 64 + lane];
    S[177 * Ntot + idx] = red[12 * 64 + lane] + red[44 * 64 + lane] + red[77 * 64 + lane];
    S[180 * Ntot + idx] = red[15 * 64 + lane] + red[47 * 64 + lane] + red[80 * 64 + lane];
    S[183 * Ntot + idx] = red[18 * 64 + lane];
    S[186 * Ntot + idx] = red[21 * 64 + lane];
    S[189 * Ntot + idx] = red[50 * 64 + lane];
    S[192 * Ntot + idx] = red[53 * 64 + lane];
    S[195 * Ntot + idx] = red[83 * 64 + lane];
    S[198 * Ntot + idx] = red[86 * 64 + lane];
    S[201 * Ntot + idx] = red[24 * 64 + lane] + red[56 * 64 + lane] + red[89 * 64 + lane];
    S[204 * Ntot + idx] = red[26 * 64 + lane] + red[59 * 64 + lane];
    S[207 * Ntot + idx] = red[29 * 64 + lane] + red[62 * 64 + lane] + red[93 * 64 + lane];
    break;
  case 1:
    S[166 * Ntot + idx] = red[1 * 64 + lane] + red[33 * 64 + lane] + red[66 * 64 + lane];
    S[169 * Ntot + idx] = red[4 * 64 + lane] + red[36 * 64 + lane] + red[69 * 64 + lane];
    S[172 * Ntot + idx] = red[7 * 64 + lane] + red[39 * 64 + lane] + red[72 * 64 + lane];
    S[175 * Ntot + idx] = red[10 * 64 + lane] + red[42 * 64 + lane] + red[75 * 64 + lane];
    S[178 * Ntot + idx] = red[13 * 64 + lane] + red[45 * 64 + lane] + red[78 * 64 + lane];
    S[181 * Ntot + idx] = red[16 * 64 + lane] + red[48 * 64 + lane] + red[81 * 64 + lane];
    S[184 * Ntot + idx] = red[19 * 64 + lane];
    S[187 * Ntot + idx] = red[22 * 64 + lane];
    S[190 * Ntot + idx] = red[51 * 64 + lane];
    S[193 * Ntot + idx] = red[54 * 64 + lane];
    S[196 * Ntot + idx] = red[84 * 64 + lane];
    S[199 * Ntot + idx] = red[87 * 64 + lane];
    S[202 * Ntot + idx] = red[25 * 64 + lane] + red[57 * 64 + lane] + red[90 * 64 + lane];
    S[205 * Ntot + idx] = red[27 * 64 + lane] + red[60 * 64 + lane] + red[92 * 64 + lane];
    S[208 * Ntot + idx] = red[30 * 64 + lane] + red[63 * 64 + lane];
    break;
  case 2:
    S[167 * Ntot + idx] = red[2 * 64 + lane] + red[34 * 64 + lane] + red[67 * 64 + lane];
    S[170 * Ntot + idx] = red[5 * 64 + lane] + red[37 * 64 + lane] + red[70 * 64 + lane];
    S[173 * Ntot + idx] = red[8 * 64 + lane] + red[40 * 64 + lane] + red[73 * 64 + lane];
    S[176 * Ntot + idx] = red[11 * 64 + lane] + red[43 * 64 + lane] + red[76 * 64 + lane];
    S[179 * Ntot + idx] = red[14 * 64 + lane] + red[46 * 64 + lane] + red[79 * 64 + lane];
    S[182 * Ntot + idx] = red[17 * 64 + lane] + red[49 * 64 + lane] + red[82 * 64 + lane];
    S[185 * Ntot + idx] = red[20 * 64 + lane];
    S[188 * Ntot + idx] = red[23 * 64 + lane];
    S[191 * Ntot + idx] = red[52 * 64 + lane];
    S[194 * Ntot + idx] = red[55 * 64 + lane];
    S[197 * Ntot + idx] = red[85 * 64 + lane];
    S[200 * Ntot + idx] = red[88 * 64 + lane];
    S[203 * Ntot + idx] = red[58 * 64 + lane] + red[91 * 64 + lane];
    S[206 * Ntot + idx] = red[28 * 64 + lane] + red[61 * 64 + lane];
    S[209 * Ntot + idx] = red[31 * 64 + lane] + red[64 * 64 + lane] + red[94 * 64 + lane];
    break;
  default:
    break;
  }
}
// workgroups of 64 points of one xx0 row x 3 output groups
static void adj_ricci_Spherical_sym2_KO0_fd4_dims(const bhah_kparams &p, dim3 &g, dim3 &b) {
  g = dim3((unsigned)((p.Nx0 - 2 * p.NG + 63) / 64), (unsigned)(p.Nx1 - 2 * p.NG), (unsigned)(p.Nx2 - 2 * p.NG));
  b = dim3(64, 3);
}

extern "C" __global__ void __launch_bounds__(256)
adj_final_Spherical_sym2_KO0_fd4(const double *__restrict__ y, const double *__restrict__ K, double b0, double b1, double b2,
                double b3, const double *__restrict__ lam, double *__restrict__ lamYN, double *__restrict__ lamK,
                const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  const int grp = (int)(blockIdx.x & 3u);
  const int i0 = (int)((blockIdx.x >> 2) * blockDim.x + threadIdx.x);
  const int i1 = (int)(blockIdx.y * blockDim.y + threadIdx.y);
  const int i2 = (int)blockIdx.z;
  if (i0 >= p.Nx0 || i1 >= p.Nx1) return;
  const long Ntot = p.Ntot, nv = 24 * Ntot;
  const long idx = i0 + p.s1 * i1 + p.s2 * i2;
  if (grp == 0) {
  const double hDD00 = y[11 * Ntot + idx] + b0 * K[11 * Ntot + idx] + b1 * K[nv + 11 * Ntot + idx] + b2 * K[2 * nv + 11 * Ntot + idx] + b3 * K[3 * nv + 11 * Ntot + idx];
  const double hDD01 = y[12 * Ntot + idx] + b0 * K[12 * Ntot + idx] + b1 * K[nv + 12 * Ntot + idx] + b2 * K[2 * nv + 12 * Ntot + idx] + b3 * K[3 * nv + 12 * Ntot + idx];
  const double hDD02 = y[13 * Ntot + idx] + b0 * K[13 * Ntot + idx] + b1 * K[nv + 13 * Ntot + idx] + b2 * K[2 * nv + 13 * Ntot + idx] + b3 * K[3 * nv + 13 * Ntot + idx];
  const double hDD11 = y[14 * Ntot + idx] + b0 * K[14 * Ntot + idx] + b1 * K[nv + 14 * Ntot + idx] + b2 * K[2 * nv + 14 * Ntot + idx] + b3 * K[3 * nv + 14 * Ntot + idx];
  const double hDD12 = y[15 * Ntot + idx] + b0 * K[15 * Ntot + idx] + b1 * K[nv + 15 * Ntot + idx] + b2 * K[2 * nv + 15 * Ntot + idx] + b3 * K[3 * nv + 15 * Ntot + idx];
  const double hDD22 = y[16 * Ntot + idx] + b0 * K[16 * Ntot + idx] + b1 * K[nv + 16 * Ntot + idx] + b2 * K[2 * nv + 16 * Ntot + idx] + b3 * K[3 * nv + 16 * Ntot + idx];
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double l_hDD00 = lam[11 * Ntot + idx];
  const double l_hDD01 = lam[12 * Ntot + idx];
  const double l_hDD02 = lam[13 * Ntot + idx];
  const double l_hDD11 = lam[14 * Ntot + idx];
  const double l_hDD12 = lam[15 * Ntot + idx];
  const double l_hDD22 = lam[16 * Ntot + idx];
  const double w0 = hDD00 + 1.0;
  const double w1 = (f0_of_xx0*f0_of_xx0);
  const double w2 = (f1_of_xx1*f1_of_xx1);
  const double w3 = w1*w2;
  const double w4 = hDD22*w3 + w3;
  const double w5 = hDD11*w1 + w1;
  const double w6 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double w7 = cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3);
  double a_w0 = l_hDD00 * (w7);
  double a_w7 = l_hDD00 * (w0);
  double a_hDD01 = l_hDD01 * (w7);
  a_w7 += l_hDD01 * (hDD01);
  double a_hDD02 = l_hDD02 * (w7);
  a_w7 += l_hDD02 * (hDD02);
  double a_hDD11 = l_hDD11 * (w7);
  a_w7 += l_hDD11 * (hDD11 + 1.0);
  double a_hDD12 = l_hDD12 * (w7);
  a_w7 += l_hDD12 * (hDD12);
  double a_hDD22 = l_hDD22 * (w7);
  a_w7 += l_hDD22 * (hDD22 + 1.0);
  double a_f0_of_xx0 = a_w7 * ((Rational_4_3)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*cbrt(fabs(f0_of_xx0))*pow(fabs(f1_of_xx1), Rational_2_3)*(((f0_of_xx0) > 0) - ((f0_of_xx0) < 0)));
  double a_f1_of_xx1 = a_w7 * ((Rational_2_3)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*(((f1_of_xx1) > 0) - ((f1_of_xx1) < 0))/cbrt(fabs(f1_of_xx1)));
  a_hDD01 += a_w7 * ((Rational_1_3)*(2.0*hDD01*w1*w4 - 2.0*hDD02*hDD12*w2*w6)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_hDD02 += a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD12*w2*w6 + 2.0*hDD02*w3*w5)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_hDD12 += a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD02*w2*w6 + 2.0*hDD12*w0*w2*w6)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_w0 += a_w7 * ((Rational_1_3)*((hDD12*hDD12)*w2*w6 - w4*w5)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w1 = a_w7 * ((Rational_1_3)*(hDD01*hDD01)*w4*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w2 = a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD02*hDD12*w6 + (hDD12*hDD12)*w0*w6)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w3 = a_w7 * ((Rational_1_3)*(hDD02*hDD02)*w5*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w4 = a_w7 * ((Rational_1_3)*((hDD01*hDD01)*w1 - w0*w5)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w5 = a_w7 * ((Rational_1_3)*((hDD02*hDD02)*w3 - w0*w4)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w6 = a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD02*hDD12*w2 + (hDD12*hDD12)*w0*w2)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_f0_of_xx0 += a_w6 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_hDD11 += a_w5 * (w1);
  a_w1 += a_w5 * (hDD11 + 1.0);
  a_hDD22 += a_w4 * (w3);
  a_w3 += a_w4 * (hDD22 + 1.0);
  a_w1 += a_w3 * (w2);
  a_w2 += a_w3 * (w1);
  a_f1_of_xx1 += a_w2 * (2.0*f1_of_xx1);
  a_f0_of_xx0 += a_w1 * (2.0*f0_of_xx0);
  double a_hDD00 = a_w0 * (1.0);
  const double v11 = a_hDD00;
  const double v12 = a_hDD01;
  const double v13 = a_hDD02;
  const double v14 = a_hDD11;
  const double v15 = a_hDD12;
  const double v16 = a_hDD22;
  lamYN[11 * Ntot + idx] = v11;
  lamYN[12 * Ntot + idx] = v12;
  lamYN[13 * Ntot + idx] = v13;
  lamYN[14 * Ntot + idx] = v14;
  lamYN[15 * Ntot + idx] = v15;
  lamYN[16 * Ntot + idx] = v16;
  lamK[0 * nv + 11 * Ntot + idx] = b0 * v11;
  lamK[0 * nv + 12 * Ntot + idx] = b0 * v12;
  lamK[0 * nv + 13 * Ntot + idx] = b0 * v13;
  lamK[0 * nv + 14 * Ntot + idx] = b0 * v14;
  lamK[0 * nv + 15 * Ntot + idx] = b0 * v15;
  lamK[0 * nv + 16 * Ntot + idx] = b0 * v16;
  lamK[1 * nv + 11 * Ntot + idx] = b1 * v11;
  lamK[1 * nv + 12 * Ntot + idx] = b1 * v12;
  lamK[1 * nv + 13 * Ntot + idx] = b1 * v13;
  lamK[1 * nv + 14 * Ntot + idx] = b1 * v14;
  lamK[1 * nv + 15 * Ntot + idx] = b1 * v15;
  lamK[1 * nv + 16 * Ntot + idx] = b1 * v16;
  lamK[2 * nv + 11 * Ntot + idx] = b2 * v11;
  lamK[2 * nv + 12 * Ntot + idx] = b2 * v12;
  lamK[2 * nv + 13 * Ntot + idx] = b2 * v13;
  lamK[2 * nv + 14 * Ntot + idx] = b2 * v14;
  lamK[2 * nv + 15 * Ntot + idx] = b2 * v15;
  lamK[2 * nv + 16 * Ntot + idx] = b2 * v16;
  lamK[3 * nv + 11 * Ntot + idx] = b3 * v11;
  lamK[3 * nv + 12 * Ntot + idx] = b3 * v12;
  lamK[3 * nv + 13 * Ntot + idx] = b3 * v13;
  lamK[3 * nv + 14 * Ntot + idx] = b3 * v14;
  lamK[3 * nv + 15 * Ntot + idx] = b3 * v15;
  lamK[3 * nv + 16 * Ntot + idx] = b3 * v16;
  } else if (grp == 1) {
  const double v0 = lam[0 * Ntot + idx];
  const double v1 = lam[1 * Ntot + idx];
  const double v2 = lam[2 * Ntot + idx];
  const double v3 = lam[3 * Ntot + idx];
  const double v4 = lam[4 * Ntot + idx];
  const double v5 = lam[5 * Ntot + idx];
  lamYN[0 * Ntot + idx] = v0;
  lamYN[1 * Ntot + idx] = v1;
  lamYN[2 * Ntot + idx] = v2;
  lamYN[3 * Ntot + idx] = v3;
  lamYN[4 * Ntot + idx] = v4;
  lamYN[5 * Ntot + idx] = v5;
  lamK[0 * nv + 0 * Ntot + idx] = b0 * v0;
  lamK[0 * nv + 1 * Ntot + idx] = b0 * v1;
  lamK[0 * nv + 2 * Ntot + idx] = b0 * v2;
  lamK[0 * nv + 3 * Ntot + idx] = b0 * v3;
  lamK[0 * nv + 4 * Ntot + idx] = b0 * v4;
  lamK[0 * nv + 5 * Ntot + idx] = b0 * v5;
  lamK[1 * nv + 0 * Ntot + idx] = b1 * v0;
  lamK[1 * nv + 1 * Ntot + idx] = b1 * v1;
  lamK[1 * nv + 2 * Ntot + idx] = b1 * v2;
  lamK[1 * nv + 3 * Ntot + idx] = b1 * v3;
  lamK[1 * nv + 4 * Ntot + idx] = b1 * v4;
  lamK[1 * nv + 5 * Ntot + idx] = b1 * v5;
  lamK[2 * nv + 0 * Ntot + idx] = b2 * v0;
  lamK[2 * nv + 1 * Ntot + idx] = b2 * v1;
  lamK[2 * nv + 2 * Ntot + idx] = b2 * v2;
  lamK[2 * nv + 3 * Ntot + idx] = b2 * v3;
  lamK[2 * nv + 4 * Ntot + idx] = b2 * v4;
  lamK[2 * nv + 5 * Ntot + idx] = b2 * v5;
  lamK[3 * nv + 0 * Ntot + idx] = b3 * v0;
  lamK[3 * nv + 1 * Ntot + idx] = b3 * v1;
  lamK[3 * nv + 2 * Ntot + idx] = b3 * v2;
  lamK[3 * nv + 3 * Ntot + idx] = b3 * v3;
  lamK[3 * nv + 4 * Ntot + idx] = b3 * v4;
  lamK[3 * nv + 5 * Ntot + idx] = b3 * v5;
  } else if (grp == 2) {
  const double v6 = lam[6 * Ntot + idx];
  const double v7 = lam[7 * Ntot + idx];
  const double v8 = lam[8 * Ntot + idx];
  const double v9 = lam[9 * Ntot + idx];
  const double v10 = lam[10 * Ntot + idx];
  const double v17 = lam[17 * Ntot + idx];
  lamYN[6 * Ntot + idx] = v6;
  lamYN[7 * Ntot + idx] = v7;
  lamYN[8 * Ntot + idx] = v8;
  lamYN[9 * Ntot + idx] = v9;
  lamYN[10 * Ntot + idx] = v10;
  lamYN[17 * Ntot + idx] = v17;
  lamK[0 * nv + 6 * Ntot + idx] = b0 * v6;
  lamK[0 * nv + 7 * Ntot + idx] = b0 * v7;
  lamK[0 * nv + 8 * Ntot + idx] = b0 * v8;
  lamK[0 * nv + 9 * Ntot + idx] = b0 * v9;
  lamK[0 * nv + 10 * Ntot + idx] = b0 * v10;
  lamK[0 * nv + 17 * Ntot + idx] = b0 * v17;
  lamK[1 * nv + 6 * Ntot + idx] = b1 * v6;
  lamK[1 * nv + 7 * Ntot + idx] = b1 * v7;
  lamK[1 * nv + 8 * Ntot + idx] = b1 * v8;
  lamK[1 * nv + 9 * Ntot + idx] = b1 * v9;
  lamK[1 * nv + 10 * Ntot + idx] = b1 * v10;
  lamK[1 * nv + 17 * Ntot + idx] = b1 * v17;
  lamK[2 * nv + 6 * Ntot + idx] = b2 * v6;
  lamK[2 * nv + 7 * Ntot + idx] = b2 * v7;
  lamK[2 * nv + 8 * Ntot + idx] = b2 * v8;
  lamK[2 * nv + 9 * Ntot + idx] = b2 * v9;
  lamK[2 * nv + 10 * Ntot + idx] = b2 * v10;
  lamK[2 * nv + 17 * Ntot + idx] = b2 * v17;
  lamK[3 * nv + 6 * Ntot + idx] = b3 * v6;
  lamK[3 * nv + 7 * Ntot + idx] = b3 * v7;
  lamK[3 * nv + 8 * Ntot + idx] = b3 * v8;
  lamK[3 * nv + 9 * Ntot + idx] = b3 * v9;
  lamK[3 * nv + 10 * Ntot + idx] = b3 * v10;
  lamK[3 * nv + 17 * Ntot + idx] = b3 * v17;
  } else {
  const double v18 = lam[18 * Ntot + idx];
  const double v19 = lam[19 * Ntot + idx];
  const double v20 = lam[20 * Ntot + idx];
  const double v21 = lam[21 * Ntot + idx];
  const double v22 = lam[22 * Ntot + idx];
  const double v23 = lam[23 * Ntot + idx];
  lamYN[18 * Ntot + idx] = v18;
  lamYN[19 * Ntot + idx] = v19;
  lamYN[20 * Ntot + idx] = v20;
  lamYN[21 * Ntot + idx] = v21;
  lamYN[22 * Ntot + idx] = v22;
  lamYN[23 * Ntot + idx] = v23;
  lamK[0 * nv + 18 * Ntot + idx] = b0 * v18;
  lamK[0 * nv + 19 * Ntot + idx] = b0 * v19;
  lamK[0 * nv + 20 * Ntot + idx] = b0 * v20;
  lamK[0 * nv + 21 * Ntot + idx] = b0 * v21;
  lamK[0 * nv + 22 * Ntot + idx] = b0 * v22;
  lamK[0 * nv + 23 * Ntot + idx] = b0 * v23;
  lamK[1 * nv + 18 * Ntot + idx] = b1 * v18;
  lamK[1 * nv + 19 * Ntot + idx] = b1 * v19;
  lamK[1 * nv + 20 * Ntot + idx] = b1 * v20;
  lamK[1 * nv + 21 * Ntot + idx] = b1 * v21;
  lamK[1 * nv + 22 * Ntot + idx] = b1 * v22;
  lamK[1 * nv + 23 * Ntot + idx] = b1 * v23;
  lamK[2 * nv + 18 * Ntot + idx] = b2 * v18;
  lamK[2 * nv + 19 * Ntot + idx] = b2 * v19;
  lamK[2 * nv + 20 * Ntot + idx] = b2 * v20;
  lamK[2 * nv + 21 * Ntot + idx] = b2 * v21;
  lamK[2 * nv + 22 * Ntot + idx] = b2 * v22;
  lamK[2 * nv + 23 * Ntot + idx] = b2 * v23;
  lamK[3 * nv + 18 * Ntot + idx] = b3 * v18;
  lamK[3 * nv + 19 * Ntot + idx] = b3 * v19;
  lamK[3 * nv + 20 * Ntot + idx] = b3 * v20;
  lamK[3 * nv + 21 * Ntot + idx] = b3 * v21;
  lamK[3 * nv + 22 * Ntot + idx] = b3 * v22;
  lamK[3 * nv + 23 * Ntot + idx] = b3 * v23;
  }
}

extern "C" __global__ void __launch_bounds__(256)
adj_stage_Spherical_sym2_KO0_fd4(const double *__restrict__ y, const double *__restrict__ K, double a,
                double *__restrict__ lamY, double *__restrict__ lamYN, double *__restrict__ lamK,
                const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  const int grp = (int)(blockIdx.x & 3u);
  const int i0 = (int)((blockIdx.x >> 2) * blockDim.x + threadIdx.x);
  const int i1 = (int)(blockIdx.y * blockDim.y + threadIdx.y);
  const int i2 = (int)blockIdx.z;
  if (i0 >= p.Nx0 || i1 >= p.Nx1) return;
  const long Ntot = p.Ntot, nv = 24 * Ntot;
  const long idx = i0 + p.s1 * i1 + p.s2 * i2;
  if (grp == 0) {
  const double hDD00 = y[11 * Ntot + idx] + a * K[11 * Ntot + idx];
  const double hDD01 = y[12 * Ntot + idx] + a * K[12 * Ntot + idx];
  const double hDD02 = y[13 * Ntot + idx] + a * K[13 * Ntot + idx];
  const double hDD11 = y[14 * Ntot + idx] + a * K[14 * Ntot + idx];
  const double hDD12 = y[15 * Ntot + idx] + a * K[15 * Ntot + idx];
  const double hDD22 = y[16 * Ntot + idx] + a * K[16 * Ntot + idx];
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double l_hDD00 = lamY[11 * Ntot + idx];
  const double l_hDD01 = lamY[12 * Ntot + idx];
  const double l_hDD02 = lamY[13 * Ntot + idx];
  const double l_hDD11 = lamY[14 * Ntot + idx];
  const double l_hDD12 = lamY[15 * Ntot + idx];
  const double l_hDD22 = lamY[16 * Ntot + idx];
  const double w0 = hDD00 + 1.0;
  const double w1 = (f0_of_xx0*f0_of_xx0);
  const double w2 = (f1_of_xx1*f1_of_xx1);
  const double w3 = w1*w2;
  const double w4 = hDD22*w3 + w3;
  const double w5 = hDD11*w1 + w1;
  const double w6 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double w7 = cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3);
  double a_w0 = l_hDD00 * (w7);
  double a_w7 = l_hDD00 * (w0);
  double a_hDD01 = l_hDD01 * (w7);
  a_w7 += l_hDD01 * (hDD01);
  double a_hDD02 = l_hDD02 * (w7);
  a_w7 += l_hDD02 * (hDD02);
  double a_hDD11 = l_hDD11 * (w7);
  a_w7 += l_hDD11 * (hDD11 + 1.0);
  double a_hDD12 = l_hDD12 * (w7);
  a_w7 += l_hDD12 * (hDD12);
  double a_hDD22 = l_hDD22 * (w7);
  a_w7 += l_hDD22 * (hDD22 + 1.0);
  double a_f0_of_xx0 = a_w7 * ((Rational_4_3)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*cbrt(fabs(f0_of_xx0))*pow(fabs(f1_of_xx1), Rational_2_3)*(((f0_of_xx0) > 0) - ((f0_of_xx0) < 0)));
  double a_f1_of_xx1 = a_w7 * ((Rational_2_3)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*(((f1_of_xx1) > 0) - ((f1_of_xx1) < 0))/cbrt(fabs(f1_of_xx1)));
  a_hDD01 += a_w7 * ((Rational_1_3)*(2.0*hDD01*w1*w4 - 2.0*hDD02*hDD12*w2*w6)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_hDD02 += a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD12*w2*w6 + 2.0*hDD02*w3*w5)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_hDD12 += a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD02*w2*w6 + 2.0*hDD12*w0*w2*w6)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_w0 += a_w7 * ((Rational_1_3)*((hDD12*hDD12)*w2*w6 - w4*w5)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w1 = a_w7 * ((Rational_1_3)*(hDD01*hDD01)*w4*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w2 = a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD02*hDD12*w6 + (hDD12*hDD12)*w0*w6)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w3 = a_w7 * ((Rational_1_3)*(hDD02*hDD02)*w5*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w4 = a_w7 * ((Rational_1_3)*((hDD01*hDD01)*w1 - w0*w5)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w5 = a_w7 * ((Rational_1_3)*((hDD02*hDD02)*w3 - w0*w4)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  double a_w6 = a_w7 * ((Rational_1_3)*(-2.0*hDD01*hDD02*hDD12*w2 + (hDD12*hDD12)*w0*w2)*cbrt((1.0 / (-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5)))*pow(fabs(f0_of_xx0), Rational_4_3)*pow(fabs(f1_of_xx1), Rational_2_3)/(-(hDD01*hDD01)*w1*w4 + 2.0*hDD01*hDD02*hDD12*w2*w6 - (hDD02*hDD02)*w3*w5 - (hDD12*hDD12)*w0*w2*w6 + w0*w4*w5));
  a_f0_of_xx0 += a_w6 * (4.0*(f0_of_xx0*f0_of_xx0*f0_of_xx0));
  a_hDD11 += a_w5 * (w1);
  a_w1 += a_w5 * (hDD11 + 1.0);
  a_hDD22 += a_w4 * (w3);
  a_w3 += a_w4 * (hDD22 + 1.0);
  a_w1 += a_w3 * (w2);
  a_w2 += a_w3 * (w1);
  a_f1_of_xx1 += a_w2 * (2.0*f1_of_xx1);
  a_f0_of_xx0 += a_w1 * (2.0*f0_of_xx0);
  double a_hDD00 = a_w0 * (1.0);
  const double v11 = a_hDD00;
  const double v12 = a_hDD01;
  const double v13 = a_hDD02;
  const double v14 = a_hDD11;
  const double v15 = a_hDD12;
  const double v16 = a_hDD22;
  const double w11 = lamYN[11 * Ntot + idx], x11 = lamK[11 * Ntot + idx];
  const double w12 = lamYN[12 * Ntot + idx], x12 = lamK[12 * Ntot + idx];
  const double w13 = lamYN[13 * Ntot + idx], x13 = lamK[13 * Ntot + idx];
  const double w14 = lamYN[14 * Ntot + idx], x14 = lamK[14 * Ntot + idx];
  const double w15 = lamYN[15 * Ntot + idx], x15 = lamK[15 * Ntot + idx];
  const double w16 = lamYN[16 * Ntot + idx], x16 = lamK[16 * Ntot + idx];
  lamYN[11 * Ntot + idx] = w11 + v11;
  lamK[11 * Ntot + idx] = x11 + a * v11;
  lamY[11 * Ntot + idx] = 0.0;
  lamYN[12 * Ntot + idx] = w12 + v12;
  lamK[12 * Ntot + idx] = x12 + a * v12;
  lamY[12 * Ntot + idx] = 0.0;
  lamYN[13 * Ntot + idx] = w13 + v13;
  lamK[13 * Ntot + idx] = x13 + a * v13;
  lamY[13 * Ntot + idx] = 0.0;
  lamYN[14 * Ntot + idx] = w14 + v14;
  lamK[14 * Ntot + idx] = x14 + a * v14;
  lamY[14 * Ntot + idx] = 0.0;
  lamYN[15 * Ntot + idx] = w15 + v15;
  lamK[15 * Ntot + idx] = x15 + a * v15;
  lamY[15 * Ntot + idx] = 0.0;
  lamYN[16 * Ntot + idx] = w16 + v16;
  lamK[16 * Ntot + idx] = x16 + a * v16;
  lamY[16 * Ntot + idx] = 0.0;
  } else if (grp == 1) {
  const double v0 = lamY[0 * Ntot + idx];
  const double v1 = lamY[1 * Ntot + idx];
  const double v2 = lamY[2 * Ntot + idx];
  const double v3 = lamY[3 * Ntot + idx];
  const double v4 = lamY[4 * Ntot + idx];
  const double v5 = lamY[5 * Ntot + idx];
  const double w0 = lamYN[0 * Ntot + idx], x0 = lamK[0 * Ntot + idx];
  const double w1 = lamYN[1 * Ntot + idx], x1 = lamK[1 * Ntot + idx];
  const double w2 = lamYN[2 * Ntot + idx], x2 = lamK[2 * Ntot + idx];
  const double w3 = lamYN[3 * Ntot + idx], x3 = lamK[3 * Ntot + idx];
  const double w4 = lamYN[4 * Ntot + idx], x4 = lamK[4 * Ntot + idx];
  const double w5 = lamYN[5 * Ntot + idx], x5 = lamK[5 * Ntot + idx];
  lamYN[0 * Ntot + idx] = w0 + v0;
  lamK[0 * Ntot + idx] = x0 + a * v0;
  lamY[0 * Ntot + idx] = 0.0;
  lamYN[1 * Ntot + idx] = w1 + v1;
  lamK[1 * Ntot + idx] = x1 + a * v1;
  lamY[1 * Ntot + idx] = 0.0;
  lamYN[2 * Ntot + idx] = w2 + v2;
  lamK[2 * Ntot + idx] = x2 + a * v2;
  lamY[2 * Ntot + idx] = 0.0;
  lamYN[3 * Ntot + idx] = w3 + v3;
  lamK[3 * Ntot + idx] = x3 + a * v3;
  lamY[3 * Ntot + idx] = 0.0;
  lamYN[4 * Ntot + idx] = w4 + v4;
  lamK[4 * Ntot + idx] = x4 + a * v4;
  lamY[4 * Ntot + idx] = 0.0;
  lamYN[5 * Ntot + idx] = w5 + v5;
  lamK[5 * Ntot + idx] = x5 + a * v5;
  lamY[5 * Ntot + idx] = 0.0;
  } else if (grp == 2) {
  const double v6 = lamY[6 * Ntot + idx];
  const double v7 = lamY[7 * Ntot + idx];
  const double v8 = lamY[8 * Ntot + idx];
  const double v9 = lamY[9 * Ntot + idx];
  const double v10 = lamY[10 * Ntot + idx];
  const double v17 = lamY[17 * Ntot + idx];
  const double w6 = lamYN[6 * Ntot + idx], x6 = lamK[6 * Ntot + idx];
  const double w7 = lamYN[7 * Ntot + idx], x7 = lamK[7 * Ntot + idx];
  const double w8 = lamYN[8 * Ntot + idx], x8 = lamK[8 * Ntot + idx];
  const double w9 = lamYN[9 * Ntot + idx], x9 = lamK[9 * Ntot + idx];
  const double w10 = lamYN[10 * Ntot + idx], x10 = lamK[10 * Ntot + idx];
  const double w17 = lamYN[17 * Ntot + idx], x17 = lamK[17 * Ntot + idx];
  lamYN[6 * Ntot + idx] = w6 + v6;
  lamK[6 * Ntot + idx] = x6 + a * v6;
  lamY[6 * Ntot + idx] = 0.0;
  lamYN[7 * Ntot + idx] = w7 + v7;
  lamK[7 * Ntot + idx] = x7 + a * v7;
  lamY[7 * Ntot + idx] = 0.0;
  lamYN[8 * Ntot + idx] = w8 + v8;
  lamK[8 * Ntot + idx] = x8 + a * v8;
  lamY[8 * Ntot + idx] = 0.0;
  lamYN[9 * Ntot + idx] = w9 + v9;
  lamK[9 * Ntot + idx] = x9 + a * v9;
  lamY[9 * Ntot + idx] = 0.0;
  lamYN[10 * Ntot + idx] = w10 + v10;
  lamK[10 * Ntot + idx] = x10 + a * v10;
  lamY[10 * Ntot + idx] = 0.0;
  lamYN[17 * Ntot + idx] = w17 + v17;
  lamK[17 * Ntot + idx] = x17 + a * v17;
  lamY[17 * Ntot + idx] = 0.0;
  } else {
  const double v18 = lamY[18 * Ntot + idx];
  const double v19 = lamY[19 * Ntot + idx];
  const double v20 = lamY[20 * Ntot + idx];
  const double v21 = lamY[21 * Ntot + idx];
  const double v22 = lamY[22 * Ntot + idx];
  const double v23 = lamY[23 * Ntot + idx];
  const double w18 = lamYN[18 * Ntot + idx], x18 = lamK[18 * Ntot + idx];
  const double w19 = lamYN[19 * Ntot + idx], x19 = lamK[19 * Ntot + idx];
  const double w20 = lamYN[20 * Ntot + idx], x20 = lamK[20 * Ntot + idx];
  const double w21 = lamYN[21 * Ntot + idx], x21 = lamK[21 * Ntot + idx];
  const double w22 = lamYN[22 * Ntot + idx], x22 = lamK[22 * Ntot + idx];
  const double w23 = lamYN[23 * Ntot + idx], x23 = lamK[23 * Ntot + idx];
  lamYN[18 * Ntot + idx] = w18 + v18;
  lamK[18 * Ntot + idx] = x18 + a * v18;
  lamY[18 * Ntot + idx] = 0.0;
  lamYN[19 * Ntot + idx] = w19 + v19;
  lamK[19 * Ntot + idx] = x19 + a * v19;
  lamY[19 * Ntot + idx] = 0.0;
  lamYN[20 * Ntot + idx] = w20 + v20;
  lamK[20 * Ntot + idx] = x20 + a * v20;
  lamY[20 * Ntot + idx] = 0.0;
  lamYN[21 * Ntot + idx] = w21 + v21;
  lamK[21 * Ntot + idx] = x21 + a * v21;
  lamY[21 * Ntot + idx] = 0.0;
  lamYN[22 * Ntot + idx] = w22 + v22;
  lamK[22 * Ntot + idx] = x22 + a * v22;
  lamY[22 * Ntot + idx] = 0.0;
  lamYN[23 * Ntot + idx] = w23 + v23;
  lamK[23 * Ntot + idx] = x23 + a * v23;
  lamY[23 * Ntot + idx] = 0.0;
  }
}

__device__ __forceinline__ double adjg_tap(const double *__restrict__ Sk, long j, long Ntot, unsigned ok) {
  j = j < 0 ? 0 : (j >= Ntot ? Ntot - 1 : j);
  const double v = Sk[j];
  return ok ? v : 0.0;
}

// One thread per (point, gridfunction); all points.  Bit o + 3 of m<d> says that the point
// o steps below along direction d lies inside the array.
extern "C" __global__ void __launch_bounds__(256)
adj_gather_Spherical_sym2_KO0_fd4(const double *__restrict__ S, double *__restrict__ lam_y, const bhah_kparams p) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int g = (int)(t / p.Ntot);
  if (g >= 24) return;
  const long Ntot = p.Ntot, s1 = p.s1, s2 = p.s2;
  const long q = t - (long)g * Ntot;
  const int i[3] = {(int)(q % p.Nx0), (int)((q / p.Nx0) % p.Nx1), (int)(q / s2)};
  const int Nx[3] = {p.Nx0, p.Nx1, p.Nx2};
  unsigned m[3];
  for (int d = 0; d < 3; d++) {
    m[d] = 0u;
    for (int o = -3; o <= 3; o++) m[d] |= ((unsigned)(i[d] - o) < (unsigned)Nx[d] ? 1u : 0u) << (o + 3);
  }
  const unsigned m0 = m[0], m1 = m[1], m2 = m[2];
  const double inv0 = p.invdxx0, inv1 = p.invdxx1, inv2 = p.invdxx2;
  double acc = 0.0;
  switch (g) {
    case 0: {
      acc += 1.0 * (1.0 * adjg_tap(S + 6 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 12 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 12 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 12 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 12 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 12 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 13 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 13 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 13 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 13 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 13 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 14 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 14 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 14 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 14 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 14 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 15 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 15 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 15 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 15 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 15 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 1: {
      acc += 1.0 * (1.0 * adjg_tap(S + 7 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 16 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 16 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 16 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 16 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 16 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 17 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 17 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 17 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 17 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 17 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 18 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 18 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 18 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 18 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 18 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 19 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 19 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 19 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 19 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 19 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 2: {
      acc += 1.0 * (1.0 * adjg_tap(S + 8 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 20 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 20 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 20 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 20 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 20 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 21 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 21 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 21 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 21 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 21 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 22 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 22 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 22 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 22 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 22 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 23 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 23 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 23 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 23 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 23 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 3: {
      acc += 1.0 * (1.0 * adjg_tap(S + 9 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 24 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 24 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 24 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 24 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 24 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 25 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 25 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 25 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 25 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 25 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 26 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 26 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 26 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 26 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 26 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 27 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 27 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 27 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 27 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 27 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 4: {
      acc += 1.0 * (1.0 * adjg_tap(S + 10 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 28 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 28 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 28 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 28 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 28 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 29 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 29 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 29 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 29 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 29 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 30 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 30 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 30 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 30 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 30 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 31 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 31 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 31 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 31 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 31 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 5: {
      acc += 1.0 * (1.0 * adjg_tap(S + 11 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 32 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 32 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 32 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 32 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 32 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 33 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 33 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 33 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 33 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 33 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 34 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 34 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 34 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 34 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 34 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 35 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 35 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 35 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 35 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 35 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 6: {
      acc += 1.0 * (1.0 * adjg_tap(S + 36 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 37 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 37 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 37 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 37 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 38 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 38 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 38 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 38 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 39 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 39 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 39 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 39 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 39 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 40 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 40 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 40 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 40 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 40 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 40 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 40 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 40 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 40 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 41 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 41 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 41 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 41 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 41 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 42 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 42 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 42 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 42 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 42 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 43 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 43 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 43 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 43 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 43 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 44 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 44 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 44 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 44 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 44 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 45 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 45 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 45 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 45 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 45 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 7: {
      acc += 1.0 * (1.0 * adjg_tap(S + 46 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 49 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 49 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 49 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 49 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 49 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 50 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 50 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 50 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 50 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 50 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 51 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 51 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 51 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 51 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 51 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 52 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 52 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 52 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 52 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 52 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 8: {
      acc += 1.0 * (1.0 * adjg_tap(S + 47 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 53 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 53 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 53 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 53 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 53 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 54 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 54 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 54 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 54 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 54 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 55 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 55 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 55 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 55 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 55 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 56 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 56 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 56 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 56 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 56 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 9: {
      acc += 1.0 * (1.0 * adjg_tap(S + 48 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 57 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 57 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 57 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 57 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 57 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 58 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 58 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 58 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 58 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 58 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 59 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 59 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 59 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 59 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 59 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 60 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 60 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 60 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 60 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 60 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 10: {
      acc += 1.0 * (1.0 * adjg_tap(S + 61 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 62 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 62 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 62 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 62 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 63 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 63 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 63 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 63 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 64 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 64 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 64 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 64 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 64 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 65 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 65 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 65 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 65 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 65 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 65 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 65 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 65 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 65 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 66 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 66 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 66 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 66 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 66 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 67 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 67 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 67 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 67 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 67 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 68 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 68 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 68 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 68 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 68 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 69 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 69 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 69 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 69 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 69 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 70 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 70 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 70 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 70 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 70 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 11: {
      acc += 1.0 * (1.0 * adjg_tap(S + 71 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 77 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 77 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 77 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 77 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 78 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 78 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 78 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 78 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 89 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 89 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 89 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 89 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 89 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 90 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 90 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 90 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 90 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 90 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 91 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 91 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 91 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 91 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 91 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 92 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 92 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 92 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 92 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 92 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 165 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 171 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 171 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 171 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 171 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 172 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 172 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 172 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 172 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 183 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 183 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 183 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 183 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 183 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 184 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 184 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 184 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 184 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 184 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 184 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 184 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 184 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 184 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 185 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 185 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 185 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 185 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 185 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 12: {
      acc += 1.0 * (1.0 * adjg_tap(S + 72 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 79 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 79 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 79 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 79 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 80 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 80 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 80 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 80 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 93 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 93 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 93 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 93 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 93 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 94 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 94 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 94 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 94 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 94 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 95 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 95 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 95 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 95 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 95 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 96 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 96 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 96 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 96 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 96 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 166 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 173 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 173 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 173 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 173 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 174 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 174 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 174 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 174 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 186 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 186 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 186 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 186 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 186 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 187 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 187 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 187 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 187 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 187 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 187 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 187 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 187 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 187 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 188 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 188 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 188 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 188 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 188 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 13: {
      acc += 1.0 * (1.0 * adjg_tap(S + 73 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 81 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 81 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 81 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 81 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 82 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 82 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 82 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 82 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 97 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 97 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 97 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 97 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 97 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 98 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 98 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 98 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 98 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 98 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 99 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 99 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 99 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 99 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 99 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 100 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 100 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 100 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 100 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 100 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 167 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 175 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 175 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 175 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 175 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 176 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 176 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 176 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 176 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 189 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 189 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 189 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 189 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 189 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 190 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 190 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 190 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 190 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 190 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 190 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 190 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 190 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 190 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 191 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 191 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 191 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 191 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 191 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 14: {
      acc += 1.0 * (1.0 * adjg_tap(S + 74 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 83 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 83 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 83 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 83 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 84 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 84 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 84 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 84 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 101 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 101 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 101 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 101 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 101 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 102 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 102 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 102 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 102 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 102 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 103 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 103 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 103 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 103 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 103 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 104 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 104 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 104 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 104 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 104 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 168 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 177 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 177 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 177 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 177 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 178 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 178 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 178 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 178 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 192 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 192 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 192 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 192 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 192 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 193 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 193 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 193 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 193 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 193 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 193 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 193 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 193 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 193 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 194 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 194 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 194 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 194 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 194 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 15: {
      acc += 1.0 * (1.0 * adjg_tap(S + 75 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 85 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 85 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 85 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 85 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 86 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 86 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 86 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 86 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 105 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 105 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 105 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 105 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 105 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 106 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 106 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 106 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 106 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 106 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 107 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 107 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 107 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 107 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 107 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 108 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 108 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 108 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 108 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 108 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 169 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 179 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 179 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 179 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 179 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 180 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 180 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 180 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 180 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 195 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 195 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 195 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 195 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 195 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 196 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 196 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 196 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 196 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 196 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 196 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 196 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 196 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 196 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 197 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 197 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 197 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 197 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 197 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 16: {
      acc += 1.0 * (1.0 * adjg_tap(S + 76 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 87 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 87 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 87 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 87 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 88 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 88 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 88 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 88 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 109 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 109 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 109 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 109 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 109 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 110 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 110 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 110 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 110 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 110 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 111 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 111 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 111 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 111 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 111 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 112 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 112 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 112 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 112 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 112 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 170 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 181 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 181 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 181 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 181 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 182 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 182 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 182 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 182 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 198 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 198 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 198 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 198 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 198 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 199 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 199 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 199 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 199 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 199 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 199 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 199 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 199 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 199 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 200 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 200 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 200 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 200 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 200 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 17: {
      acc += 1.0 * (1.0 * adjg_tap(S + 113 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 116 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 116 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 116 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 116 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 116 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 117 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 117 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 117 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 117 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 117 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 118 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 118 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 118 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 118 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 118 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 119 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 119 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 119 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 119 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 119 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 201 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 204 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 204 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 204 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 204 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 205 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 205 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 205 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 205 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 18: {
      acc += 1.0 * (1.0 * adjg_tap(S + 114 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 120 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 120 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 120 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 120 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 120 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 121 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 121 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 121 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 121 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 121 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 122 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 122 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 122 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 122 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 122 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 123 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 123 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 123 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 123 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 123 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 202 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 206 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 206 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 206 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 206 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 207 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 207 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 207 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 207 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 19: {
      acc += 1.0 * (1.0 * adjg_tap(S + 115 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 124 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 124 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 124 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 124 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 124 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 125 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 125 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 125 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 125 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 125 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 126 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 126 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 126 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 126 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 126 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 127 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 127 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 127 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 127 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 127 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      acc += 1.0 * (1.0 * adjg_tap(S + 203 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 208 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 208 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 208 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 208 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 209 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 209 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 209 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 209 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      break;
    }
    case 20: {
      acc += 1.0 * (1.0 * adjg_tap(S + 128 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 129 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 129 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 129 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 129 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 130 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 130 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 130 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 130 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 131 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 131 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 131 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 131 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 131 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 132 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 132 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 132 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 132 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 132 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 133 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 133 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 133 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 133 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 133 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 134 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 134 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 134 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 134 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 134 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 21: {
      acc += 1.0 * (1.0 * adjg_tap(S + 135 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 138 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 138 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 138 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 138 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 139 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 139 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 139 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 139 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 144 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 144 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 144 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 144 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 144 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 145 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 145 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 145 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 145 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 145 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 145 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 145 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 145 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 145 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 146 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 146 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 146 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 146 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 146 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 153 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 153 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 153 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 153 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 153 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 154 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 154 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 154 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 154 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 154 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 155 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 155 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 155 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 155 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 155 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 156 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 156 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 156 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 156 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 156 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 22: {
      acc += 1.0 * (1.0 * adjg_tap(S + 136 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 140 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 140 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 140 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 140 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 141 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 141 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 141 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 141 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 147 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 147 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 147 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 147 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 147 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 148 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 148 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 148 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 148 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 148 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 148 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 148 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 148 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 148 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 149 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 149 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 149 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 149 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 149 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 157 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 157 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 157 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 157 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 157 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 158 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 158 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 158 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 158 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 158 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 159 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 159 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 159 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 159 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 159 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 160 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 160 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 160 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 160 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 160 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    case 23: {
      acc += 1.0 * (1.0 * adjg_tap(S + 137 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((1.0 / 12.0) * adjg_tap(S + 142 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 142 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 142 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 142 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((1.0 / 12.0) * adjg_tap(S + 143 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-2.0 / 3.0) * adjg_tap(S + 143 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (2.0 / 3.0) * adjg_tap(S + 143 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 143 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * inv0 * ((-1.0 / 12.0) * adjg_tap(S + 150 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 150 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 150 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 150 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 150 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * inv1 * ((1.0 / 144.0) * adjg_tap(S + 151 * Ntot, q - (-2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (-2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (-2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 151 * Ntot, q - (-2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (-1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 151 * Ntot, q - (-1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 151 * Ntot, q - (-1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (-1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (1 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-4.0 / 9.0) * adjg_tap(S + 151 * Ntot, q - (1 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (4.0 / 9.0) * adjg_tap(S + 151 * Ntot, q - (1 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (1 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (-1.0 / 144.0) * adjg_tap(S + 151 * Ntot, q - (2 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (2 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-1.0 / 18.0) * adjg_tap(S + 151 * Ntot, q - (2 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (1.0 / 144.0) * adjg_tap(S + 151 * Ntot, q - (2 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv1 * inv1 * ((-1.0 / 12.0) * adjg_tap(S + 152 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 152 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 2.0) * adjg_tap(S + 152 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (4.0 / 3.0) * adjg_tap(S + 152 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 12.0) * adjg_tap(S + 152 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 4.0) * adjg_tap(S + 161 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 161 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 161 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 161 * Ntot, q - (2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 5) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 161 * Ntot, q - (3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 6) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv0 * ((-1.0 / 12.0) * adjg_tap(S + 162 * Ntot, q - (-3 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 0) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 162 * Ntot, q - (-2 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 1) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 162 * Ntot, q - (-1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 2) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 162 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 162 * Ntot, q - (1 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 4) & (m1 >> 3) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 4.0) * adjg_tap(S + 163 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (-5.0 / 6.0) * adjg_tap(S + 163 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (3.0 / 2.0) * adjg_tap(S + 163 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u)
          + (-1.0 / 2.0) * adjg_tap(S + 163 * Ntot, q - (0 + 2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 5) & (m2 >> 3)) & 1u)
          + (1.0 / 12.0) * adjg_tap(S + 163 * Ntot, q - (0 + 3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 6) & (m2 >> 3)) & 1u));
      acc += inv1 * ((-1.0 / 12.0) * adjg_tap(S + 164 * Ntot, q - (0 + -3 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 0) & (m2 >> 3)) & 1u)
          + (1.0 / 2.0) * adjg_tap(S + 164 * Ntot, q - (0 + -2 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 1) & (m2 >> 3)) & 1u)
          + (-3.0 / 2.0) * adjg_tap(S + 164 * Ntot, q - (0 + -1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 2) & (m2 >> 3)) & 1u)
          + (5.0 / 6.0) * adjg_tap(S + 164 * Ntot, q - (0 + 0 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 3) & (m2 >> 3)) & 1u)
          + (1.0 / 4.0) * adjg_tap(S + 164 * Ntot, q - (0 + 1 * s1 + 0 * s2), Ntot, ((m0 >> 3) & (m1 >> 4) & (m2 >> 3)) & 1u));
      break;
    }
    default:
      break;
  }
  lam_y[t] += acc;
}
#undef Rational_1_2
#undef Rational_1_3
#undef Rational_1_4
#undef Rational_2_3
#undef Rational_3_2
#undef Rational_3_4
#undef Rational_4_3
#undef Rational_8_3
#undef Rational_m1_2
#undef Rational_m1_3
#undef Rational_m2_3
#undef Rational_m8_3

extern "C" int adj_nslots_Spherical_sym2_KO0_fd4(void) { return 210; }
extern "C" hipError_t launch_adj_rhs_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, const double *in, const double *aux,
    const double *lam, double *S, const double *rfm0, const double *rfm1, bhah_kparams p) {
  adj_rhs_Spherical_sym2_KO0_fd4_dims(p, g, b);
  hipLaunchKernelGGL(adj_rhs_Spherical_sym2_KO0_fd4, g, b, 0, s, in, aux, lam, S, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_adj_ricci_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, const double *in, double *S,
    const double *rfm0, const double *rfm1, bhah_kparams p) {
  adj_ricci_Spherical_sym2_KO0_fd4_dims(p, g, b);
  hipLaunchKernelGGL(adj_ricci_Spherical_sym2_KO0_fd4, g, b, 0, s, in, S, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_adj_final_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, const double *y, const double *K,
    double b0, double b1, double b2, double b3, const double *lam, double *lamYN, double *lamK, const double *rfm0,
    const double *rfm1, bhah_kparams p) {
  g.x *= 4;
  hipLaunchKernelGGL(adj_final_Spherical_sym2_KO0_fd4, g, b, 0, s, y, K, b0, b1, b2, b3, lam, lamYN, lamK, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_adj_stage_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, const double *y, const double *K, double a,
    double *lamY, double *lamYN, double *lamK, const double *rfm0, const double *rfm1, bhah_kparams p) {
  g.x *= 4;
  hipLaunchKernelGGL(adj_stage_Spherical_sym2_KO0_fd4, g, b, 0, s, y, K, a, lamY, lamYN, lamK, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_adj_gather_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, const double *S, double *lam_y,
    bhah_kparams p) {
  hipLaunchKernelGGL(adj_gather_Spherical_sym2_KO0_fd4, g, b, 0, s, S, lam_y, p);
  return hipGetLastError();
}
