// Generated by nrpy_amd/codegen/hip_gen.py -- do not edit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "../bhah_device_types.h"
// ---- rhs candidate p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub: 1 kernel(s); Spherical, fd_order=4
#ifndef BHAH_PIN
#define BHAH_PIN(x) asm volatile("" : "+v"(x))
// several values at once: BHAH_PINS("+v"(a), "+v"(b), ...)
#define BHAH_PINS(...) asm volatile("" : __VA_ARGS__)
#endif
#ifndef BHAH_DMA16
// 16 bytes per lane straight from global memory into LDS at dst + 16 * lane (dst uniform per wave)
#define BHAH_DMA16(src, dst) __builtin_amdgcn_global_load_lds((const void *)(src), (__attribute__((address_space(3))) void *)(dst), 16, 0, 0)
// the same from a uniform byte base plus a 32-bit per-lane byte offset, widened at the load
// itself so it is addressed as scalar base + vector offset
#define BHAH_DMA16O(base, off, dst) do { unsigned o_ = (off); asm volatile("" : "+v"(o_)); BHAH_DMA16((base) + o_, dst); } while (0)
// wait until at most n vector-memory operations of this wave are outstanding (gfx9 encoding)
#define BHAH_VMWAIT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | 0x0F70)
// workgroup barrier without a memory fence (LDS reads of this wave retired first)
#define BHAH_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")
// the same before the LDS reads of DMA phase n; the comment marks it in the assembly listing
// for the build's wait check (nrpy_amd/isa_check.py)
#define BHAH_BARRIER_PHASE(n) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier ; bhah_read_phase " #n ::: "memory")
#endif
#ifndef BHAH_WAVE_SYNC
// order of LDS accesses of one wave: the hardware runs them in program order, and the clobber keeps
// the compiler from moving a lane's load above the stores other lanes make for it
#define BHAH_WAVE_SYNC() asm volatile("" ::: "memory")
#endif
#define Rational_1_2 (1.0 / 2.0)
#define Rational_1_3 (1.0 / 3.0)
#define Rational_1_4 (1.0 / 4.0)
#define Rational_1_6 (1.0 / 6.0)
#define Rational_2_3 (2.0 / 3.0)
#define Rational_3_2 (3.0 / 2.0)
#define Rational_3_4 (3.0 / 4.0)
#define Rational_4_3 (4.0 / 3.0)

// bhah-dma-issue bssn_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0: 0:2 1:2 2:2 3:2 4:2 5:2 6:2 7:2 8:2 9:2 10:2 11:2 12:2 13:2 14:2 15:2 16:2 17:2 18:2 19:2 20:2 21:2 22:2 23:2
// bhah-dma-issue bssn_ens_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0: 0:2 1:2 2:2 3:2 4:2 5:2 6:2 7:2 8:2 9:2 10:2 11:2 12:2 13:2 14:2 15:2 16:2 17:2 18:2 19:2 20:2 21:2 22:2 23:2
extern "C" __global__ void __launch_bounds__(256)
bssn_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0(const double *__restrict__ in, const double *__restrict__ aux, double *__restrict__ out,
        const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  __shared__ double sh[3072];
  const unsigned bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  // Tile of 16x8x2 interior points; halo box 22x14x2 = 616 values per gridfunction.
  constexpr int BX = 22, BY = 14, NB = 616, NT = 256, NL = 3;
  const int tid = (int)threadIdx.x;
  const int lx = tid % 16, ly = (tid / 16) % 8, lz = tid / 128;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const int o0 = p.NG + (int)bx * 16, o1 = p.NG + (int)by * 8, o2 = p.NG + (int)bz * 2;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned pofs[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int e = 2 * (tid + NT * j);
    const int ex = e % BX, ey = (e / BX) % BY, ez = e / (BX * BY);
    const int g0 = min(o0 - 3 + ex, p.Nx0 - 2), g1 = min(o1 - 3 + ey, p.Nx1 - 1), g2 = min(o2 - 0 + ez, p.Nx2 - 1);
    pofs[j] = 8u * (unsigned)(g0 + (int)s1 * g1 + (int)s2 * g2);
  }
  const int c0 = (lx + 3) + BX * (ly + 3) + BX * BY * (lz + 0);
  const double ius0 = p.invdxx0 * (1.0 / 12.0), nius0 = -ius0, ikos0 = p.invdxx0 * (1.0 / 64.0);
  const double ius1 = p.invdxx1 * (1.0 / 12.0), nius1 = -ius1, ikos1 = p.invdxx1 * (1.0 / 64.0);
  const double ius2 = p.invdxx2 * (1.0 / 12.0), nius2 = -ius2, ikos2 = p.invdxx2 * (1.0 / 64.0);
  double L0_coef[2], L0_beta[3];
  {
    const int i0 = min(o0 + lx, p.Nx0 - p.NG - 1), i1 = min(o1 + ly, p.Nx1 - p.NG - 1);
    const long idx = i0 + s1 * i1 + s2 * min(o2 + lz + 0, p.Nx2 - p.NG - 1);
    const double f0_of_xx0 = rfm0[i0];
    const double f1_of_xx1 = rfm1[i1];
    const double vetU0 = in[21 * Ntot + idx];
    const double vetU1 = in[22 * Ntot + idx];
    const double vetU2 = in[23 * Ntot + idx];
    L0_coef[0] = vetU0;
    L0_coef[1] = vetU1/f0_of_xx0;
    L0_beta[0] = vetU0;
    L0_beta[1] = vetU1/f0_of_xx0;
    L0_beta[2] = vetU2/(f0_of_xx0*f1_of_xx1);
  }
  double V0_lin_aDD00 = 0.0;
  double V0_lin_aDD01 = 0.0;
  double V0_lin_aDD02 = 0.0;
  double V0_lin_aDD11 = 0.0;
  double V0_lin_aDD12 = 0.0;
  double V0_lin_aDD22 = 0.0;
  double V0_lin_alpha = 0.0;
  double V0_lin_betU0 = 0.0;
  double V0_lin_betU1 = 0.0;
  double V0_lin_betU2 = 0.0;
  double V0_lin_cf = 0.0;
  double V0_lin_hDD00 = 0.0;
  double V0_lin_hDD01 = 0.0;
  double V0_lin_hDD02 = 0.0;
  double V0_lin_hDD11 = 0.0;
  double V0_lin_hDD12 = 0.0;
  double V0_lin_hDD22 = 0.0;
  double V0_lin_lambdaU0 = 0.0;
  double V0_lin_lambdaU1 = 0.0;
  double V0_lin_lambdaU2 = 0.0;
  double V0_lin_trK = 0.0;
  double V0_lin_vetU0 = 0.0;
  double V0_lin_vetU1 = 0.0;
  double V0_lin_vetU2 = 0.0;
  {
    const char *src = (const char *)(in + 0 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  {
    const char *src = (const char *)(in + 1 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  // ---- aDD00
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(0);
  {
    const char *src = (const char *)(in + 2 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD00 = sh[c0];
  const double U0_aDD00_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_aDD00_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_aDD00 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD00_0 : D0_aDD00_0);
  const double U0_aDD00_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_aDD00_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_aDD00 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD00_1 : D0_aDD00_1);
  BHAH_PINS("+v"(V0_aDD00), "+v"(V0_lin_aDD00));
  // ---- aDD01
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(1);
  {
    const char *src = (const char *)(in + 3 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD01 = sh[c0 + 1024];
  const double U0_aDD01_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_aDD01_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD01 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD01_0 : D0_aDD01_0);
  const double U0_aDD01_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_aDD01_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD01 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD01_1 : D0_aDD01_1);
  BHAH_PINS("+v"(V0_aDD01), "+v"(V0_lin_aDD01));
  // ---- aDD02
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(2);
  {
    const char *src = (const char *)(in + 4 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD02 = sh[c0 + 2048];
  const double U0_aDD02_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_aDD02_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD02 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD02_0 : D0_aDD02_0);
  const double U0_aDD02_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_aDD02_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD02 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD02_1 : D0_aDD02_1);
  BHAH_PINS("+v"(V0_aDD02), "+v"(V0_lin_aDD02));
  // ---- aDD11
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(3);
  {
    const char *src = (const char *)(in + 5 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD11 = sh[c0];
  const double U0_aDD11_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_aDD11_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_aDD11 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD11_0 : D0_aDD11_0);
  const double U0_aDD11_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_aDD11_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_aDD11 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD11_1 : D0_aDD11_1);
  BHAH_PINS("+v"(V0_aDD11), "+v"(V0_lin_aDD11));
  // ---- aDD12
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(4);
  {
    const char *src = (const char *)(in + 6 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD12 = sh[c0 + 1024];
  const double U0_aDD12_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_aDD12_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD12 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD12_0 : D0_aDD12_0);
  const double U0_aDD12_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_aDD12_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD12 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD12_1 : D0_aDD12_1);
  BHAH_PINS("+v"(V0_aDD12), "+v"(V0_lin_aDD12));
  // ---- aDD22
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(5);
  {
    const char *src = (const char *)(in + 7 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD22 = sh[c0 + 2048];
  const double U0_aDD22_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_aDD22_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD22 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD22_0 : D0_aDD22_0);
  const double U0_aDD22_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_aDD22_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD22 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD22_1 : D0_aDD22_1);
  BHAH_PINS("+v"(V0_aDD22), "+v"(V0_lin_aDD22));
  // ---- alpha
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(6);
  {
    const char *src = (const char *)(in + 8 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_alpha = sh[c0];
  double V0_alpha_dD0 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_alpha_dD1 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  double V0_alpha_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 1] + sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] + sh[c0 - 2]));
  double V0_alpha_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 23] - sh[c0 - 21]) - (sh[c0 + 21] - sh[c0 - 23])) + (-1.0 / 18.0) * ((sh[c0 + 45] - sh[c0 - 43]) - (sh[c0 + 43] - sh[c0 - 45])) + (-1.0 / 18.0) * ((sh[c0 + 24] - sh[c0 - 20]) - (sh[c0 + 20] - sh[c0 - 24])) + (1.0 / 144.0) * ((sh[c0 + 46] - sh[c0 - 42]) - (sh[c0 + 42] - sh[c0 - 46])));
  double V0_alpha_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 22] + sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] + sh[c0 - 44]));
  const double U0_alpha_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_alpha_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_alpha += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_alpha_0 : D0_alpha_0);
  const double U0_alpha_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_alpha_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_alpha += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_alpha_1 : D0_alpha_1);
  BHAH_PINS("+v"(V0_alpha), "+v"(V0_alpha_dD0), "+v"(V0_alpha_dD1), "+v"(V0_alpha_dDD00), "+v"(V0_alpha_dDD01), "+v"(V0_alpha_dDD11), "+v"(V0_lin_alpha));
  // ---- betU0
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(7);
  {
    const char *src = (const char *)(in + 9 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU0 = sh[c0 + 1024];
  const double U0_betU0_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_betU0_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_betU0 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_betU0_0 : D0_betU0_0);
  const double U0_betU0_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_betU0_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_betU0 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_betU0_1 : D0_betU0_1);
  BHAH_PINS("+v"(V0_betU0), "+v"(V0_lin_betU0));
  // ---- betU1
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(8);
  {
    const char *src = (const char *)(in + 10 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU1 = sh[c0 + 2048];
  const double U0_betU1_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_betU1_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_betU1 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_betU1_0 : D0_betU1_0);
  const double U0_betU1_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_betU1_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_betU1 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_betU1_1 : D0_betU1_1);
  BHAH_PINS("+v"(V0_betU1), "+v"(V0_lin_betU1));
  // ---- betU2
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(9);
  {
    const char *src = (const char *)(in + 11 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU2 = sh[c0];
  const double U0_betU2_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_betU2_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_betU2 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_betU2_0 : D0_betU2_0);
  const double U0_betU2_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_betU2_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_betU2 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_betU2_1 : D0_betU2_1);
  BHAH_PINS("+v"(V0_betU2), "+v"(V0_lin_betU2));
  // ---- cf
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(10);
  {
    const char *src = (const char *)(in + 12 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_cf = sh[c0 + 1024];
  double V0_cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  double V0_cf_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1025] + sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] + sh[c0 + 1022]));
  double V0_cf_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 1047] - sh[c0 + 1003]) - (sh[c0 + 1045] - sh[c0 + 1001])) + (-1.0 / 18.0) * ((sh[c0 + 1069] - sh[c0 + 981]) - (sh[c0 + 1067] - sh[c0 + 979])) + (-1.0 / 18.0) * ((sh[c0 + 1048] - sh[c0 + 1004]) - (sh[c0 + 1044] - sh[c0 + 1000])) + (1.0 / 144.0) * ((sh[c0 + 1070] - sh[c0 + 982]) - (sh[c0 + 1066] - sh[c0 + 978])));
  double V0_cf_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1046] + sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] + sh[c0 + 980]));
  const double U0_cf_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_cf_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_cf += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_cf_0 : D0_cf_0);
  const double U0_cf_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_cf_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_cf += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_cf_1 : D0_cf_1);
  BHAH_PINS("+v"(V0_cf), "+v"(V0_cf_dD0), "+v"(V0_cf_dD1), "+v"(V0_cf_dDD00), "+v"(V0_cf_dDD01), "+v"(V0_cf_dDD11), "+v"(V0_lin_cf));
  // ---- hDD00
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(11);
  {
    const char *src = (const char *)(in + 13 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD00 = sh[c0 + 2048];
  double V0_hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  const double U0_hDD00_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_hDD00_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD00 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD00_0 : D0_hDD00_0);
  const double U0_hDD00_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_hDD00_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD00 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD00_1 : D0_hDD00_1);
  BHAH_PINS("+v"(V0_hDD00), "+v"(V0_hDD_dD000), "+v"(V0_hDD_dD001), "+v"(V0_lin_hDD00));
  // ---- hDD01
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(12);
  {
    const char *src = (const char *)(in + 14 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD01 = sh[c0];
  double V0_hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  const double U0_hDD01_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_hDD01_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_hDD01 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD01_0 : D0_hDD01_0);
  const double U0_hDD01_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_hDD01_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_hDD01 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD01_1 : D0_hDD01_1);
  BHAH_PINS("+v"(V0_hDD01), "+v"(V0_hDD_dD010), "+v"(V0_hDD_dD011), "+v"(V0_lin_hDD01));
  // ---- hDD02
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(13);
  {
    const char *src = (const char *)(in + 15 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD02 = sh[c0 + 1024];
  double V0_hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  const double U0_hDD02_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_hDD02_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD02 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD02_0 : D0_hDD02_0);
  const double U0_hDD02_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_hDD02_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD02 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD02_1 : D0_hDD02_1);
  BHAH_PINS("+v"(V0_hDD02), "+v"(V0_hDD_dD020), "+v"(V0_hDD_dD021), "+v"(V0_lin_hDD02));
  // ---- hDD11
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(14);
  {
    const char *src = (const char *)(in + 16 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD11 = sh[c0 + 2048];
  double V0_hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  const double U0_hDD11_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_hDD11_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD11 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD11_0 : D0_hDD11_0);
  const double U0_hDD11_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_hDD11_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD11 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD11_1 : D0_hDD11_1);
  BHAH_PINS("+v"(V0_hDD11), "+v"(V0_hDD_dD110), "+v"(V0_hDD_dD111), "+v"(V0_lin_hDD11));
  // ---- hDD12
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(15);
  {
    const char *src = (const char *)(in + 17 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD12 = sh[c0];
  double V0_hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  const double U0_hDD12_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_hDD12_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_hDD12 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD12_0 : D0_hDD12_0);
  const double U0_hDD12_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_hDD12_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_hDD12 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD12_1 : D0_hDD12_1);
  BHAH_PINS("+v"(V0_hDD12), "+v"(V0_hDD_dD120), "+v"(V0_hDD_dD121), "+v"(V0_lin_hDD12));
  // ---- hDD22
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(16);
  {
    const char *src = (const char *)(in + 18 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD22 = sh[c0 + 1024];
  double V0_hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  const double U0_hDD22_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_hDD22_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD22 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD22_0 : D0_hDD22_0);
  const double U0_hDD22_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_hDD22_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD22 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD22_1 : D0_hDD22_1);
  BHAH_PINS("+v"(V0_hDD22), "+v"(V0_hDD_dD220), "+v"(V0_hDD_dD221), "+v"(V0_lin_hDD22));
  // ---- lambdaU0
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(17);
  {
    const char *src = (const char *)(in + 19 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU0 = sh[c0 + 2048];
  const double U0_lambdaU0_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_lambdaU0_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_lambdaU0 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_lambdaU0_0 : D0_lambdaU0_0);
  const double U0_lambdaU0_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_lambdaU0_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_lambdaU0 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_lambdaU0_1 : D0_lambdaU0_1);
  BHAH_PINS("+v"(V0_lambdaU0), "+v"(V0_lin_lambdaU0));
  // ---- lambdaU1
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(18);
  {
    const char *src = (const char *)(in + 20 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU1 = sh[c0];
  const double U0_lambdaU1_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_lambdaU1_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_lambdaU1 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_lambdaU1_0 : D0_lambdaU1_0);
  const double U0_lambdaU1_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_lambdaU1_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_lambdaU1 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_lambdaU1_1 : D0_lambdaU1_1);
  BHAH_PINS("+v"(V0_lambdaU1), "+v"(V0_lin_lambdaU1));
  // ---- lambdaU2
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(19);
  {
    const char *src = (const char *)(in + 21 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU2 = sh[c0 + 1024];
  const double U0_lambdaU2_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_lambdaU2_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_lambdaU2 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_lambdaU2_0 : D0_lambdaU2_0);
  const double U0_lambdaU2_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_lambdaU2_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_lambdaU2 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_lambdaU2_1 : D0_lambdaU2_1);
  BHAH_PINS("+v"(V0_lambdaU2), "+v"(V0_lin_lambdaU2));
  // ---- trK
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(20);
  {
    const char *src = (const char *)(in + 22 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_trK = sh[c0 + 2048];
  double V0_trK_dD0 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_trK_dD1 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  const double U0_trK_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_trK_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_trK += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_trK_0 : D0_trK_0);
  const double U0_trK_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_trK_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_trK += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_trK_1 : D0_trK_1);
  BHAH_PINS("+v"(V0_trK), "+v"(V0_trK_dD0), "+v"(V0_trK_dD1), "+v"(V0_lin_trK));
  // ---- vetU0
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(21);
  {
    const char *src = (const char *)(in + 23 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_vetU0 = sh[c0];
  double V0_vetU_dD00 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_vetU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  double V0_vetU_dDD000 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 1] + sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] + sh[c0 - 2]));
  double V0_vetU_dDD001 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 23] - sh[c0 - 21]) - (sh[c0 + 21] - sh[c0 - 23])) + (-1.0 / 18.0) * ((sh[c0 + 45] - sh[c0 - 43]) - (sh[c0 + 43] - sh[c0 - 45])) + (-1.0 / 18.0) * ((sh[c0 + 24] - sh[c0 - 20]) - (sh[c0 + 20] - sh[c0 - 24])) + (1.0 / 144.0) * ((sh[c0 + 46] - sh[c0 - 42]) - (sh[c0 + 42] - sh[c0 - 46])));
  double V0_vetU_dDD011 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 22] + sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] + sh[c0 - 44]));
  const double U0_vetU0_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_vetU0_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_vetU0 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_vetU0_0 : D0_vetU0_0);
  const double U0_vetU0_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_vetU0_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_vetU0 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_vetU0_1 : D0_vetU0_1);
  BHAH_PINS("+v"(V0_vetU0), "+v"(V0_vetU_dD00), "+v"(V0_vetU_dD01), "+v"(V0_vetU_dDD000), "+v"(V0_vetU_dDD001), "+v"(V0_vetU_dDD011), "+v"(V0_lin_vetU0));
  // ---- vetU1
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(22);
  double V0_vetU1 = sh[c0 + 1024];
  double V0_vetU_dD10 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_vetU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  double V0_vetU_dDD100 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1025] + sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] + sh[c0 + 1022]));
  double V0_vetU_dDD101 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 1047] - sh[c0 + 1003]) - (sh[c0 + 1045] - sh[c0 + 1001])) + (-1.0 / 18.0) * ((sh[c0 + 1069] - sh[c0 + 981]) - (sh[c0 + 1067] - sh[c0 + 979])) + (-1.0 / 18.0) * ((sh[c0 + 1048] - sh[c0 + 1004]) - (sh[c0 + 1044] - sh[c0 + 1000])) + (1.0 / 144.0) * ((sh[c0 + 1070] - sh[c0 + 982]) - (sh[c0 + 1066] - sh[c0 + 978])));
  double V0_vetU_dDD111 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1046] + sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] + sh[c0 + 980]));
  const double U0_vetU1_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_vetU1_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_vetU1 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_vetU1_0 : D0_vetU1_0);
  const double U0_vetU1_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_vetU1_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_vetU1 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_vetU1_1 : D0_vetU1_1);
  BHAH_PINS("+v"(V0_vetU1), "+v"(V0_vetU_dD10), "+v"(V0_vetU_dD11), "+v"(V0_vetU_dDD100), "+v"(V0_vetU_dDD101), "+v"(V0_vetU_dDD111), "+v"(V0_lin_vetU1));
  // ---- vetU2
  BHAH_VMWAIT(0);
  BHAH_BARRIER_PHASE(23);
  double V0_vetU2 = sh[c0 + 2048];
  double V0_vetU_dD20 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_vetU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  double V0_vetU_dDD200 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0 + 2048] + (4.0 / 3.0) * (sh[c0 + 2049] + sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] + sh[c0 + 2046]));
  double V0_vetU_dDD201 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 2071] - sh[c0 + 2027]) - (sh[c0 + 2069] - sh[c0 + 2025])) + (-1.0 / 18.0) * ((sh[c0 + 2093] - sh[c0 + 2005]) - (sh[c0 + 2091] - sh[c0 + 2003])) + (-1.0 / 18.0) * ((sh[c0 + 2072] - sh[c0 + 2028]) - (sh[c0 + 2068] - sh[c0 + 2024])) + (1.0 / 144.0) * ((sh[c0 + 2094] - sh[c0 + 2006]) - (sh[c0 + 2090] - sh[c0 + 2002])));
  double V0_vetU_dDD211 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0 + 2048] + (4.0 / 3.0) * (sh[c0 + 2070] + sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] + sh[c0 + 2004]));
  const double U0_vetU2_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_vetU2_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_vetU2 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_vetU2_0 : D0_vetU2_0);
  const double U0_vetU2_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_vetU2_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_vetU2 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_vetU2_1 : D0_vetU2_1);
  BHAH_PINS("+v"(V0_vetU2), "+v"(V0_vetU_dD20), "+v"(V0_vetU_dD21), "+v"(V0_vetU_dDD200), "+v"(V0_vetU_dDD201), "+v"(V0_vetU_dDD211), "+v"(V0_lin_vetU2));
  {
    const int i0 = o0 + lx, i1 = o1 + ly, i2 = o2 + lz + 0;
    if (i0 < p.Nx0 - p.NG && i1 < p.Nx1 - p.NG && i2 < p.Nx2 - p.NG) {
      const long idx = i0 + s1 * i1 + s2 * i2;
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double t5 = f0_of_xx0*f1_of_xx1;
  const double aDD02 = V0_aDD02;
  const double _AbDD02 = aDD02*t5;
  const double aDD01 = V0_aDD01;
  const double _AbDD01 = aDD01*f0_of_xx0;
  const double hDD01 = V0_hDD01;
  const double _gbDD01 = f0_of_xx0*hDD01;
  const double hDD02 = V0_hDD02;
  const double t0 = f1_of_xx1*hDD02;
  const double _gbDD02 = f0_of_xx0*t0;
  const double t1 = (f0_of_xx0*f0_of_xx0);
  const double t2 = f1_of_xx1*t1;
  const double hDD12 = V0_hDD12;
  const double _gbDD12 = hDD12*t2;
  const double t3 = (f1_of_xx1*f1_of_xx1);
  const double t4 = t1*t3;
  const double hDD22 = V0_hDD22;
  const double _gbDD22 = hDD22*t4 + t4;
  const double hDD00 = V0_hDD00;
  const double _gbDD00 = hDD00 + 1.0;
  const double hDD11 = V0_hDD11;
  const double _gbDD11 = hDD11*t1 + t1;
  const double t6 = (_gbDD12*_gbDD12);
  const double t7 = (_gbDD02*_gbDD02);
  const double t8 = (_gbDD01*_gbDD01);
  const double t9 = (1.0 / (_gbDD00*_gbDD11*_gbDD22 - _gbDD00*t6 + 2.0*_gbDD01*_gbDD02*_gbDD12 - _gbDD11*t7 - _gbDD22*t8));
  const double _gbUU01 = t9*(-_gbDD01*_gbDD22 + _gbDD02*_gbDD12);
  const double t34 = _AbDD01*_gbUU01;
  const double _gbUU02 = t9*(_gbDD01*_gbDD12 - _gbDD02*_gbDD11);
  const double t35 = _AbDD02*_gbUU02;
  const double _gbUU00 = t9*(_gbDD11*_gbDD22 - t6);
  const double aDD00 = V0_aDD00;
  const double t36 = _gbUU00*aDD00;
  const double _AbUD00 = t34 + t35 + t36;
  const double _gbUU11 = t9*(_gbDD00*_gbDD22 - t7);
  const double _gbUU12 = t9*(-_gbDD00*_gbDD12 + _gbDD01*_gbDD02);
  const double _AbUD10 = _AbDD01*_gbUU11 + _AbDD02*_gbUU12 + _gbUU01*aDD00;
  const double _gbUU22 = t9*(_gbDD00*_gbDD11 - t8);
  const double _AbUD20 = _AbDD01*_gbUU12 + _AbDD02*_gbUU22 + _gbUU02*aDD00;
  const double t41 = (1.0 / f0_of_xx0);
  const double t48 = (1.0 / t1);
  const double vetU1 = V0_vetU1;
  const double t49 = t48*vetU1;
  const double vetU_dD10 = V0_vetU_dD10;
  const double _bUdD10 = t41*vetU_dD10 - t49;
  const double hDD_dD020 = V0_hDD_dD020;
  const double _gbDDdD020 = hDD_dD020*t5 + t0;
  const double t21 = (Rational_1_2)*_gbUU00;
  const double hDD_dD010 = V0_hDD_dD010;
  const double _gbDDdD010 = f0_of_xx0*hDD_dD010 + hDD01;
  const double hDD_dD001 = V0_hDD_dD001;
  const double t22 = 2.0*_gbDDdD010 - hDD_dD001;
  const double t23 = (Rational_1_2)*_gbUU01;
  const double hDD_dD000 = V0_hDD_dD000;
  const double _GbUDD000 = _gbDDdD020*_gbUU02 + hDD_dD000*t21 + t22*t23;
  const double t30 = (Rational_1_2)*_gbUU11;
  const double _GbUDD100 = _gbDDdD020*_gbUU12 + hDD_dD000*t23 + t22*t30;
  const double alpha_dD0 = V0_alpha_dD0;
  const double alpha_dD1 = V0_alpha_dD1;
  const double alpha_dDD00 = V0_alpha_dDD00;
  const double _adBDD00 = -_GbUDD000*alpha_dD0 - _GbUDD100*alpha_dD1 + alpha_dDD00;
  const double cf = V0_cf;
  const double t63 = (1.0 / cf);
  const double t64 = (Rational_1_2)*t63;
  const double cf_dD0 = V0_cf_dD0;
  const double _phidD0 = -cf_dD0*t64;
  const double cf_dD1 = V0_cf_dD1;
  const double _phidD1 = -cf_dD1*t64;
  const double cf_dDD00 = V0_cf_dDD00;
  const double _phidBDD00 = -_GbUDD000*_phidD0 - _GbUDD100*_phidD1 + (Rational_1_2)*t63*((cf_dD0*cf_dD0)*t63 - cf_dDD00);
  const double alpha = V0_alpha;
  const double t67 = 2.0*alpha;
  const double t68 = _phidD0*alpha_dD0;
  const double t69 = 4.0*alpha;
  const double RbarDD00 = aux[0 * Ntot + idx];
  const double _curly00 = RbarDD00*alpha - _adBDD00 - _phidBDD00*t67 + (_phidD0*_phidD0)*t69 + 4.0*t68;
  const double t73 = (cf*cf);
  const double t11 = 2.0*f0_of_xx0;
  const double t12 = hDD11*t11 + t11;
  const double hDD_dD110 = V0_hDD_dD110;
  const double _gbDDdD110 = hDD_dD110*t1 + t12;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t10 = f1_of_xx1__D1*hDD02;
  const double hDD_dD021 = V0_hDD_dD021;
  const double _gbDDdD021 = f0_of_xx0*t10 + hDD_dD021*t5;
  const double t13 = hDD12*t11;
  const double hDD_dD120 = V0_hDD_dD120;
  const double _gbDDdD120 = f1_of_xx1*t13 + hDD_dD120*t2;
  const double t24 = _gbDDdD021 + _gbDDdD120;
  const double t25 = (Rational_1_2)*_gbUU02;
  const double _GbUDD001 = _gbDDdD110*t23 + hDD_dD001*t21 + t24*t25;
  const double t31 = (Rational_1_2)*_gbUU12;
  const double _GbUDD101 = _gbDDdD110*t30 + hDD_dD001*t23 + t24*t31;
  const double alpha_dDD01 = V0_alpha_dDD01;
  const double _adBDD01 = -_GbUDD001*alpha_dD0 - _GbUDD101*alpha_dD1 + alpha_dDD01;
  const double cf_dDD01 = V0_cf_dDD01;
  const double _phidBDD01 = -_GbUDD001*_phidD0 - _GbUDD101*_phidD1 + (Rational_1_2)*t63*(cf_dD0*cf_dD1*t63 - cf_dDD01);
  const double t70 = 2.0*alpha_dD1;
  const double t71 = _phidD0*t70;
  const double t72 = 2.0*_phidD1*alpha_dD0;
  const double RbarDD01 = aux[1 * Ntot + idx];
  const double _curly01 = RbarDD01*alpha - _adBDD01 - _phidBDD01*t67 + _phidD0*_phidD1*t69 + t71 + t72;
  const double t15 = t11*t3;
  const double t16 = hDD22*t15 + t15;
  const double hDD_dD220 = V0_hDD_dD220;
  const double _gbDDdD220 = hDD_dD220*t4 + t16;
  const double t26 = _gbDDdD220*t25;
  const double t27 = _gbDDdD021 - _gbDDdD120;
  const double t28 = -t27;
  const double _GbUDD002 = t23*t28 + t26;
  const double _GbUDD102 = _gbDDdD220*t31 + t28*t30;
  const double _adBDD02 = -_GbUDD002*alpha_dD0 - _GbUDD102*alpha_dD1;
  const double _phidBDD02 = -_GbUDD002*_phidD0 - _GbUDD102*_phidD1;
  const double RbarDD02 = aux[2 * Ntot + idx];
  const double _curly02 = RbarDD02*alpha - _adBDD02 - _phidBDD02*t67;
  const double hDD_dD111 = V0_hDD_dD111;
  const double _gbDDdD111 = hDD_dD111*t1;
  const double t14 = f1_of_xx1__D1*hDD12;
  const double hDD_dD121 = V0_hDD_dD121;
  const double _gbDDdD121 = hDD_dD121*t2 + t1*t14;
  const double hDD_dD011 = V0_hDD_dD011;
  const double _gbDDdD011 = f0_of_xx0*hDD_dD011;
  const double t29 = 2.0*_gbDDdD011 - _gbDDdD110;
  const double _GbUDD011 = _gbDDdD111*t23 + _gbDDdD121*_gbUU02 + t21*t29;
  const double _GbUDD111 = _gbDDdD111*t30 + _gbDDdD121*_gbUU12 + t23*t29;
  const double alpha_dDD11 = V0_alpha_dDD11;
  const double _adBDD11 = -_GbUDD011*alpha_dD0 - _GbUDD111*alpha_dD1 + alpha_dDD11;
  const double cf_dDD11 = V0_cf_dDD11;
  const double _phidBDD11 = -_GbUDD011*_phidD0 - _GbUDD111*_phidD1 + (Rational_1_2)*t63*((cf_dD1*cf_dD1)*t63 - cf_dDD11);
  const double RbarDD11 = aux[3 * Ntot + idx];
  const double _curly11 = RbarDD11*alpha - _adBDD11 - _phidBDD11*t67 + (_phidD1*_phidD1)*t69 + 4.0*_phidD1*alpha_dD1;
  const double t17 = f1_of_xx1*f1_of_xx1__D1;
  const double t18 = 2.0*t17;
  const double t19 = t1*t18;
  const double t20 = hDD22*t19 + t19;
  const double hDD_dD221 = V0_hDD_dD221;
  const double _gbDDdD221 = hDD_dD221*t4 + t20;
  const double _GbUDD012 = _gbDDdD221*t25 + t21*t27;
  const double t32 = _gbDDdD221*t31;
  const double _GbUDD112 = t23*t27 + t32;
  const double _adBDD12 = -_GbUDD012*alpha_dD0 - _GbUDD112*alpha_dD1;
  const double _phidBDD12 = -_GbUDD012*_phidD0 - _GbUDD112*_phidD1;
  const double RbarDD12 = aux[4 * Ntot + idx];
  const double _curly12 = RbarDD12*alpha - _adBDD12 - _phidBDD12*t67;
  const double _GbUDD022 = -_gbDDdD220*t21 - _gbDDdD221*t23;
  const double _GbUDD122 = -_gbDDdD220*t23 - _gbDDdD221*t30;
  const double _adBDD22 = -_GbUDD022*alpha_dD0 - _GbUDD122*alpha_dD1;
  const double _phidBDD22 = -_GbUDD022*_phidD0 - _GbUDD122*_phidD1;
  const double RbarDD22 = aux[5 * Ntot + idx];
  const double _curly22 = RbarDD22*alpha - _adBDD22 - _phidBDD22*t67;
  const double t45 = 2.0*_gbUU01;
  const double t46 = 2.0*_gbUU02;
  const double t47 = 2.0*_gbUU12;
  const double _curlytr = _curly00*_gbUU00 + _curly01*t45 + _curly02*t46 + _curly11*_gbUU11 + _curly12*t47 + _curly22*_gbUU22;
  const double t74 = (Rational_1_3)*_curlytr;
  const double t75 = 2.0*_AbDD01;
  const double t43 = (1.0 / f1_of_xx1);
  const double t50 = t41*t43;
  const double t51 = t43*t48;
  const double vetU2 = V0_vetU2;
  const double t52 = t51*vetU2;
  const double vetU_dD20 = V0_vetU_dD20;
  const double _bUdD20 = t50*vetU_dD20 - t52;
  const double t76 = 2.0*_bUdD20;
  const double vetU_dD00 = V0_vetU_dD00;
  const double t77 = 2.0*vetU_dD00;
  const double vetU_dD11 = V0_vetU_dD11;
  const double _bUdD11 = t41*vetU_dD11;
  const double t44 = f1_of_xx1__D1*t43;
  const double t65 = 2.0*t41;
  const double t66 = t41*vetU1;
  const double vetU0 = V0_vetU0;
  const double _Dbb = _bUdD11 + t44*t66 + t65*vetU0 + vetU_dD00;
  const double t78 = (Rational_2_3)*_Dbb;
  const double trK = V0_trK;
  const double t79 = alpha*trK;
  const double t80 = _AbDD01*t67;
  const double t81 = _AbDD02*t67;
  const double t82 = aDD00*t67;
  out[0 * Ntot + idx] = _AbDD02*t76 - _AbUD00*t82 - _AbUD10*t80 - _AbUD20*t81 + _bUdD10*t75 + aDD00*t77 - aDD00*t78 + aDD00*t79 + t73*(_curly00 - _gbDD00*t74) + V0_lin_aDD00;
  const double aDD11 = V0_aDD11;
  const double _AbDD11 = aDD11*t1;
  const double aDD12 = V0_aDD12;
  const double _AbDD12 = aDD12*t2;
  const double _AbUD01 = _AbDD01*_gbUU00 + _AbDD11*_gbUU01 + _AbDD12*_gbUU02;
  const double t37 = _AbDD11*_gbUU11;
  const double t38 = _AbDD12*_gbUU12;
  const double _AbUD11 = t34 + t37 + t38;
  const double _AbUD21 = _AbDD01*_gbUU02 + _AbDD11*_gbUU12 + _AbDD12*_gbUU22;
  const double t53 = (1.0 / t3);
  const double t54 = t41*t53;
  const double t55 = f1_of_xx1__D1*vetU2;
  const double vetU_dD21 = V0_vetU_dD21;
  const double _bUdD21 = t50*vetU_dD21 - t54*t55;
  const double vetU_dD01 = V0_vetU_dD01;
  out[1 * Ntot + idx] = t41*(_AbDD01*_bUdD11 - _AbDD01*t78 + _AbDD01*t79 + _AbDD01*vetU_dD00 + _AbDD02*_bUdD21 + _AbDD11*_bUdD10 + _AbDD12*_bUdD20 - _AbUD01*t82 - _AbUD11*t80 - _AbUD21*t81 + aDD00*vetU_dD01 + aDD01*vetU0 + t73*(_curly01 - _gbDD01*t74)) + V0_lin_aDD01;
  const double aDD22 = V0_aDD22;
  const double _AbDD22 = aDD22*t4;
  const double _AbUD02 = _AbDD02*_gbUU00 + _AbDD12*_gbUU01 + _AbDD22*_gbUU02;
  const double _AbUD12 = _AbDD02*_gbUU01 + _AbDD12*_gbUU11 + _AbDD22*_gbUU12;
  const double t39 = _AbDD22*_gbUU22;
  const double _AbUD22 = t35 + t38 + t39;
  const double t83 = f1_of_xx1*vetU0;
  const double t84 = f1_of_xx1__D1*vetU1;
  out[2 * Ntot + idx] = t50*(-_AbDD02*t78 + _AbDD02*t79 + _AbDD02*vetU_dD00 + _AbDD12*_bUdD10 + _AbDD22*_bUdD20 - _AbUD02*t82 - _AbUD12*t80 - _AbUD22*t81 + aDD02*t83 + aDD02*t84 + t73*(_curly02 - _gbDD02*t74)) + V0_lin_aDD02;
  const double t85 = 2.0*_bUdD11;
  const double t86 = 2.0*_bUdD21;
  const double t87 = _AbDD11*t67;
  const double t88 = _AbDD12*t67;
  out[3 * Ntot + idx] = t48*(-_AbDD11*t78 + _AbDD11*t79 + _AbDD11*t85 + _AbDD12*t86 - _AbUD01*t80 - _AbUD11*t87 - _AbUD21*t88 + aDD11*t11*vetU0 + t73*(_curly11 - _gbDD11*t74) + t75*vetU_dD01) + V0_lin_aDD11;
  out[4 * Ntot + idx] = t51*(_AbDD02*vetU_dD01 + _AbDD12*_bUdD11 - _AbDD12*t78 + _AbDD12*t79 + _AbDD22*_bUdD21 - _AbUD02*t80 - _AbUD12*t87 - _AbUD22*t88 + aDD12*f0_of_xx0*t84 + aDD12*t11*t83 + t73*(_curly12 - _gbDD12*t74)) + V0_lin_aDD12;
  const double t59 = t48*t53;
  const double t89 = _AbDD22*t67;
  out[5 * Ntot + idx] = t59*(_AbDD22*alpha*trK - _AbDD22*t78 - _AbUD02*t81 - _AbUD12*t88 - _AbUD22*t89 + 2.0*aDD22*f0_of_xx0*f1_of_xx1*f1_of_xx1__D1*vetU1 + 2.0*aDD22*f0_of_xx0*t3*vetU0 + t73*(_curly22 - _gbDD22*t74)) + V0_lin_aDD22;
  out[6 * Ntot + idx] = -t67*trK + V0_lin_alpha;
  const double _AbUU00 = _AbUD00*_gbUU00 + _AbUD01*_gbUU01 + _AbUD02*_gbUU02;
  const double _AbUU01 = _AbUD00*_gbUU01 + _AbUD01*_gbUU11 + _AbUD02*_gbUU12;
  const double _AbUU02 = _AbUD00*_gbUU02 + _AbUD01*_gbUU12 + _AbUD02*_gbUU22;
  const double _AbUU12 = _AbUD10*_gbUU02 + _AbUD11*_gbUU12 + _AbUD12*_gbUU22;
  const double _AbUU20 = _AbUD20*_gbUU00 + _AbUD21*_gbUU01 + _AbUD22*_gbUU02;
  const double _AbUU21 = _AbUD20*_gbUU01 + _AbUD21*_gbUU11 + _AbUD22*_gbUU12;
  const double _DGUDD011 = _GbUDD011 + f0_of_xx0;
  const double t40 = f0_of_xx0*t3;
  const double _DGUDD022 = _GbUDD022 + t40;
  const double _DGU0 = _DGUDD011*_gbUU11 + _DGUDD022*_gbUU22 + _GbUDD000*_gbUU00 + _GbUDD001*t45 + _GbUDD002*t46 + _GbUDD012*t47;
  const double vetU_dDD101 = V0_vetU_dDD101;
  const double _bUdDD101 = t41*vetU_dDD101 - t48*vetU_dD11;
  const double t99 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t100 = (Rational_1_2)*t53/t99;
  const double t101 = 2.0*t99;
  const double t102 = 8.0*t17;
  const double t103 = 4.0*t44;
  const double t97 = t48*vetU0;
  const double t56 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t98 = 4.0*t3*t56;
  const double vetU_dDD000 = V0_vetU_dDD000;
  const double t104 = _bUdDD101 + t100*(12.0*t4*vetU0 + t98*vetU_dD00) + t100*(_bUdD10*t101*t17 + t1*t102*vetU1) - t103*t49 - 8.0*t97 + vetU_dDD000;
  const double t105 = (Rational_1_4)*t104;
  const double vetU_dDD111 = V0_vetU_dDD111;
  const double _bUdDD111 = t41*vetU_dDD111;
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double t106 = f1_of_xx1*f1_of_xx1__DD11;
  const double t62 = (f1_of_xx1__D1*f1_of_xx1__D1);
  const double t107 = t53*t62;
  const double t108 = t107*t66;
  const double vetU_dDD001 = V0_vetU_dDD001;
  const double t109 = _bUdDD111 + t100*(t102*t56*vetU0 + t98*vetU_dD01) + t100*(t17*t85*t99 + t66*(t101*t106 + t101*t62)) - t103*t41*vetU0 - 2.0*t108 + vetU_dDD001;
  const double t110 = (Rational_1_4)*t109;
  const double t111 = _bUdD10*f0_of_xx0;
  const double t112 = t41*vetU_dD01;
  const double t113 = -t111 - t112 + vetU_dDD001;
  const double t114 = (Rational_3_2)*_gbUU01;
  const double t115 = _gbUU00*vetU_dDD000;
  const double vetU_dDD011 = V0_vetU_dDD011;
  const double t116 = _gbUU11*(-_bUdD11*t11 + f0_of_xx0*vetU_dD00 - vetU0 + vetU_dDD011);
  const double t117 = _gbUU22*(t17*vetU_dD01 - t18*vetU1 - t3*vetU0 + t40*vetU_dD00);
  const double betU0 = V0_betU0;
  const double t118 = betU0*vetU0;
  const double trK_dD0 = V0_trK_dD0;
  const double t119 = alpha*trK_dD0;
  const double t120 = _gbUU00*t119;
  const double trK_dD1 = V0_trK_dD1;
  const double t121 = alpha*trK_dD1;
  const double t122 = _gbUU01*t121;
  const double lambdaU0 = V0_lambdaU0;
  const double t123 = (Rational_3_4)*lambdaU0;
  const double t124 = t123*vetU0;
  const double lambdaU1 = V0_lambdaU1;
  const double t125 = lambdaU1*t112;
  const double t126 = _AbUU00*alpha;
  const double t127 = (Rational_3_2)*t126;
  const double t128 = (Rational_3_2)*alpha;
  const double t129 = _AbUU01*_GbUDD001;
  const double t130 = _GbUDD002*t128;
  const double _AbUU10 = _AbUD10*_gbUU00 + _AbUD11*_gbUU01 + _AbUD12*_gbUU02;
  const double t131 = _AbUU10*t128;
  const double _AbUU11 = _AbUD10*_gbUU01 + _AbUD11*_gbUU11 + _AbUD12*_gbUU12;
  const double t132 = _AbUU11*alpha;
  const double t133 = (Rational_3_2)*t132;
  const double t134 = _GbUDD012*t128;
  const double _AbUU22 = _AbUD20*_gbUU02 + _AbUD21*_gbUU12 + _AbUD22*_gbUU22;
  const double t135 = _AbUU22*alpha;
  const double t136 = (Rational_3_2)*t135;
  const double t137 = betU0*t66;
  const double betU1 = V0_betU1;
  const double t138 = betU1*t41;
  const double t139 = t138*vetU0;
  const double t140 = betU1*t49;
  const double t141 = (Rational_3_2)*_gbUU02;
  const double t142 = _bUdD20*t40;
  const double t143 = _bUdD21*_gbUU12;
  const double t144 = t123*t66;
  const double t145 = _GbUDD001*vetU0;
  const double t146 = lambdaU1*t41;
  const double t147 = (Rational_3_4)*t146;
  const double t148 = (Rational_3_4)*lambdaU1;
  const double t149 = t148*t49;
  const double t150 = t50*vetU2;
  const double t151 = betU0*t150;
  const double betU2 = V0_betU2;
  const double t152 = betU2*t50;
  const double t153 = t152*vetU0;
  const double t154 = betU1*t52;
  const double t155 = betU2*t49;
  const double t156 = t155*t43;
  const double t157 = t59*vetU2;
  const double t158 = betU2*t157;
  const double t159 = t123*t150;
  const double t160 = _GbUDD002*vetU0;
  const double lambdaU2 = V0_lambdaU2;
  const double t161 = (Rational_3_4)*lambdaU2;
  const double t162 = t161*t50;
  const double t163 = t148*t52;
  const double t164 = lambdaU2*t49;
  const double t165 = (Rational_3_4)*t164*t43;
  const double t166 = t157*t161;
  const double t90 = (Rational_1_2)*_Dbb;
  const double t91 = 6.0*alpha;
  const double t92 = -_phidD0*t91 + alpha_dD0;
  const double t93 = (Rational_3_2)*t92;
  const double t94 = -_phidD1*t91 + alpha_dD1;
  const double t95 = (Rational_3_2)*t94;
  const double t96 = lambdaU0*vetU_dD00;
  const double eta = p.eta;
  out[7 * Ntot + idx] = -_AbUU00*t93 - _AbUU01*t95 + _AbUU02*t130 + _AbUU12*t134 + _AbUU20*t130 + _AbUU21*t134 + _DGU0*t90 + _DGUDD011*t133 + _DGUDD022*t136 + _GbUDD000*t118 - _GbUDD000*t124 + _GbUDD000*t127 + _GbUDD001*t131 + _GbUDD001*t137 + _GbUDD001*t139 - _GbUDD001*t144 + _GbUDD002*t151 + _GbUDD002*t153 - _GbUDD002*t159 + _GbUDD011*t140 - _GbUDD011*t149 + _GbUDD012*t154 + _GbUDD012*t156 - _GbUDD012*t163 - _GbUDD012*t165 + _GbUDD022*t158 - _GbUDD022*t166 + _gbUU00*t105 + _gbUU01*t110 - betU0*eta + t113*t114 + (Rational_3_4)*t115 + (Rational_3_4)*t116 + (Rational_3_4)*t117 - t120 - t122 - Rational_3_4*t125 + t128*t129 - t141*t142 - Rational_3_2*t143*t40 - t145*t147 - t160*t162 - Rational_3_4*t96 + V0_lin_betU0;
  const double t42 = -t41;
  const double _DGUDD101 = _GbUDD101 + t42;
  const double _DGUDD122 = _GbUDD122 + t17;
  const double _DGU1 = _DGUDD101*t45 + _DGUDD122*_gbUU22 + _GbUDD100*_gbUU00 + _GbUDD102*t46 + _GbUDD111*_gbUU11 + _GbUDD112*t47;
  const double t167 = _bUdD10*lambdaU0;
  const double t168 = t41*vetU_dD00 - t97;
  const double t169 = _bUdDD101 + t168;
  const double t57 = 2.0/t56;
  const double vetU_dDD100 = V0_vetU_dDD100;
  const double _bUdDD100 = t41*vetU_dDD100 - 2.0*t48*vetU_dD10 + t57*vetU1;
  const double t170 = _gbUU00*(_bUdD10*t65 + _bUdDD100);
  const double t171 = _gbUU11*(_bUdDD111 + t111 + 2.0*t112);
  const double t172 = _bUdD21*t17;
  const double t173 = t41*vetU2;
  const double t174 = _gbUU12*(-f1_of_xx1*t173 - t172 + t41*t43*t62*vetU2 + t41*t43*vetU2*(-t106 - t62));
  const double t175 = _gbUU22*(_bUdD10*t40 + _bUdD11*t17 + t3*t66 - t62*t66);
  const double t176 = _gbUU01*t119;
  const double t177 = _gbUU11*t121;
  const double t178 = _bUdD11*t146;
  const double t179 = _AbUU01*t128;
  const double t180 = _GbUDD102*t128;
  const double t181 = _GbUDD112*t128;
  const double t182 = _bUdD20*t17;
  const double t183 = t147*vetU0;
  const double t184 = _gbUU12*t172;
  const double t185 = t162*vetU0;
  out[8 * Ntot + idx] = f0_of_xx0*(_AbUU02*t180 - _AbUU10*t93 - _AbUU11*t95 + _AbUU12*t181 + _AbUU20*t180 + _AbUU21*t181 + _DGU1*t90 + _DGUDD101*t131 + _DGUDD101*t179 + _DGUDD122*t136 + _GbUDD100*t118 - _GbUDD100*t124 + _GbUDD100*t127 + _GbUDD101*t137 + _GbUDD101*t139 - _GbUDD101*t144 - _GbUDD101*t183 + _GbUDD102*t151 + _GbUDD102*t153 - _GbUDD102*t159 - _GbUDD102*t185 + _GbUDD111*t133 + _GbUDD111*t140 - _GbUDD111*t149 + _GbUDD112*t154 + _GbUDD112*t156 - _GbUDD112*t163 - _GbUDD112*t165 + _GbUDD122*t158 - _GbUDD122*t166 + _gbUU01*t105 + _gbUU11*t110 - betU1*t97 - eta*t138 + t114*t169 - t141*t182 - Rational_3_4*t167 + (Rational_3_4)*t170 + (Rational_3_4)*t171 + (Rational_3_4)*t174 + (Rational_3_4)*t175 - t176 - t177 - Rational_3_4*t178 - Rational_3_4*t184) + V0_lin_betU1;
  const double t33 = (Rational_1_2)*_gbUU22;
  const double _GbUDD202 = _gbDDdD220*t33 + t28*t31;
  const double _DGUDD202 = _GbUDD202 + t42;
  const double _GbUDD212 = _gbDDdD221*t33 + t25*t27;
  const double _DGUDD212 = _GbUDD212 - t44;
  const double _GbUDD200 = _gbDDdD020*_gbUU22 + hDD_dD000*t25 + t22*t31;
  const double _GbUDD201 = _gbDDdD110*t31 + hDD_dD001*t25 + t24*t33;
  const double _GbUDD211 = _gbDDdD111*t31 + _gbDDdD121*_gbUU22 + t25*t29;
  const double _GbUDD222 = -t26 - t32;
  const double _DGU2 = _DGUDD202*t46 + _DGUDD212*t47 + _GbUDD200*_gbUU00 + _GbUDD201*t45 + _GbUDD211*_gbUU11 + _GbUDD222*_gbUU22;
  const double t186 = _bUdD20*lambdaU0;
  const double t60 = f1_of_xx1__D1*t54;
  const double vetU_dDD201 = V0_vetU_dDD201;
  const double _bUdDD201 = t50*vetU_dDD201 - t51*vetU_dD21 + t55*t59 - t60*vetU_dD20;
  const double t187 = _bUdD20*t44 + _bUdDD201;
  const double t188 = _bUdD10*t44 + t168;
  const double t58 = t43*vetU2;
  const double vetU_dDD200 = V0_vetU_dDD200;
  const double _bUdDD200 = t50*vetU_dDD200 - 2.0*t51*vetU_dD20 + t57*t58;
  const double t189 = _gbUU00*(_bUdD20*t65 + _bUdDD200);
  const double t61 = (1.0 / (f1_of_xx1*f1_of_xx1*f1_of_xx1));
  const double vetU_dDD211 = V0_vetU_dDD211;
  const double _bUdDD211 = t50*vetU_dDD211 - 2.0*t60*vetU_dD21 + vetU2*(-f1_of_xx1__DD11*t54 + 2.0*t41*t61*t62);
  const double t190 = f1_of_xx1__DD11*t43 - t107;
  const double t191 = _gbUU11*(_bUdD20*f0_of_xx0 + _bUdDD211 + t150*t190 + t150 + t173*t61*t62 + t44*t86);
  const double t192 = _bUdD11*t44 + t112;
  const double t193 = _gbUU12*(t190*t66 + t192);
  const double t194 = _gbUU12*(-t108 + t192 - t66);
  const double t195 = _gbUU22*(t142 + t172);
  const double t196 = _gbUU02*t119;
  const double t197 = _gbUU12*t121;
  const double t198 = _bUdD21*t146;
  const double t199 = _DGUDD202*t128;
  const double t200 = _DGUDD212*t128;
  const double t201 = t43*t97;
  const double t202 = f1_of_xx1__D1*t53;
  out[9 * Ntot + idx] = t5*(_AbUU02*t199 + _AbUU12*t200 + _AbUU20*t199 - _AbUU20*t93 + _AbUU21*t200 - _AbUU21*t95 + _DGU2*t90 + _GbUDD200*t118 - _GbUDD200*t124 + _GbUDD200*t127 + _GbUDD201*t131 + _GbUDD201*t137 + _GbUDD201*t139 - _GbUDD201*t144 + _GbUDD201*t179 - _GbUDD201*t183 + _GbUDD202*t151 + _GbUDD202*t153 - _GbUDD202*t159 - _GbUDD202*t185 + _GbUDD211*t133 + _GbUDD211*t140 - _GbUDD211*t149 + _GbUDD212*t154 + _GbUDD212*t156 - _GbUDD212*t163 - _GbUDD212*t165 + _GbUDD222*t136 + _GbUDD222*t158 - _GbUDD222*t166 + _gbUU02*t105 + _gbUU12*t110 - betU2*t201 - eta*t152 + t114*t187 + t141*t188 - t155*t202 - Rational_3_4*t186 + (Rational_3_4)*t189 + (Rational_3_4)*t191 + (Rational_3_4)*t193 + (Rational_3_4)*t194 + (Rational_3_4)*t195 - t196 - t197 - Rational_3_4*t198) + V0_lin_betU2;
  out[10 * Ntot + idx] = -2.0*cf*((Rational_1_6)*_Dbb - Rational_1_6*t79) + V0_lin_cf;
  const double t203 = 2.0*_gbDD01;
  const double _trAb = 2.0*t34 + 2.0*t35 + t36 + t37 + 2.0*t38 + t39;
  const double t204 = -Rational_2_3*_Dbb + (Rational_2_3)*_trAb*alpha;
  out[11 * Ntot + idx] = _bUdD10*t203 + _gbDD00*t204 + _gbDD00*t77 + _gbDD02*t76 - t82 + V0_lin_hDD00;
  out[12 * Ntot + idx] = t41*(_bUdD10*_gbDD11 + _bUdD11*_gbDD01 + _bUdD20*_gbDD12 + _bUdD21*_gbDD02 + _gbDD00*vetU_dD01 + _gbDD01*t204 + _gbDD01*vetU_dD00 + hDD01*vetU0 - t80) + V0_lin_hDD01;
  out[13 * Ntot + idx] = t50*(_bUdD10*_gbDD12 + _bUdD20*_gbDD22 + _gbDD02*t204 + _gbDD02*vetU_dD00 + t0*vetU0 + t10*vetU1 - t81) + V0_lin_hDD02;
  out[14 * Ntot + idx] = t48*(_gbDD11*t204 + _gbDD11*t85 + _gbDD12*t86 + t12*vetU0 + t203*vetU_dD01 - t87) + V0_lin_hDD11;
  out[15 * Ntot + idx] = t51*(_bUdD11*_gbDD12 + _bUdD21*_gbDD22 + _gbDD02*vetU_dD01 + _gbDD12*t204 + f0_of_xx0*t14*vetU1 + t13*t83 - t88) + V0_lin_hDD12;
  out[16 * Ntot + idx] = t59*(_gbDD22*t204 + t16*vetU0 + t20*t66 - t89) + V0_lin_hDD22;
  const double t205 = 2.0*t92;
  const double t206 = 2.0*t94;
  const double t207 = (Rational_1_3)*t104;
  const double t208 = (Rational_1_3)*t109;
  const double t209 = _AbUU00*t67;
  const double t210 = _GbUDD002*t67;
  const double t211 = _AbUU10*t67;
  const double t212 = _AbUU11*t67;
  const double t213 = _GbUDD012*t67;
  const double t214 = _AbUU22*t67;
  out[17 * Ntot + idx] = -_AbUU00*t205 - _AbUU01*t206 + _AbUU02*t210 + _AbUU12*t213 + _AbUU20*t210 + _AbUU21*t213 + _DGU0*t78 + _DGUDD011*t212 + _DGUDD022*t214 + _GbUDD000*t209 + _GbUDD001*t211 - _bUdD20*_gbUU02*t15 + _gbUU00*t207 + _gbUU01*t208 + t113*t45 + t115 + t116 + t117 - Rational_4_3*t120 - Rational_4_3*t122 - t125 + t129*t67 - t143*t15 - t96 + V0_lin_lambdaU0;
  const double t215 = _AbUU01*t67;
  const double t216 = _GbUDD102*t67;
  const double t217 = _GbUDD112*t67;
  out[18 * Ntot + idx] = f0_of_xx0*(_AbUU02*t216 - _AbUU10*t205 - _AbUU11*t206 + _AbUU12*t217 + _AbUU20*t216 + _AbUU21*t217 + _DGU1*t78 + _DGUDD101*t211 + _DGUDD101*t215 + _DGUDD122*t214 + _GbUDD100*t209 + _GbUDD111*t212 + _gbUU01*t207 + _gbUU11*t208 - lambdaU1*t97 - t167 + t169*t45 + t170 + t171 + t174 + t175 - Rational_4_3*t176 - Rational_4_3*t177 - t178 - t182*t46 - t184) + V0_lin_lambdaU1;
  const double t218 = _DGUDD202*t67;
  const double t219 = _DGUDD212*t67;
  out[19 * Ntot + idx] = t5*(_AbUU02*t218 + _AbUU12*t219 - _AbUU20*t205 + _AbUU20*t218 - _AbUU21*t206 + _AbUU21*t219 + _DGU2*t78 + _GbUDD200*t209 + _GbUDD201*t211 + _GbUDD201*t215 + _GbUDD211*t212 + _GbUDD222*t214 + _gbUU02*t207 + _gbUU12*t208 - lambdaU2*t201 - t164*t202 - t186 + t187*t45 + t188*t46 + t189 + t191 + t193 + t194 + t195 - Rational_4_3*t196 - Rational_4_3*t197 - t198) + V0_lin_lambdaU2;
  const double t220 = _AbDD01*alpha;
  const double t221 = _AbDD02*alpha;
  const double t222 = _AbDD12*alpha;
  const double t223 = _gbUU01*t73;
  out[20 * Ntot + idx] = _AbDD11*t132 + _AbDD22*t135 + _AbUU01*t220 + _AbUU02*t221 + _AbUU10*t220 + _AbUU12*t222 + _AbUU20*t221 + _AbUU21*t222 - _adBDD02*t46*t73 - _adBDD12*t47*t73 - _adBDD22*_gbUU22*t73 - _gbUU00*t73*(_adBDD00 + 2.0*t68) - _gbUU11*t73*(_adBDD11 + _phidD1*t70) + aDD00*t126 + (Rational_1_3)*alpha*(trK*trK) - t223*(_adBDD01 + t71) - t223*(_adBDD01 + t72) + V0_lin_trK;
  const double t224 = (vetU0*vetU0);
  const double t225 = t48*(vetU1*vetU1);
  const double t226 = t59*(vetU2*vetU2);
  const double t227 = 2.0*t66;
  const double t228 = 2.0*t150;
  const double t229 = 2.0*t49*t58;
  out[21 * Ntot + idx] = _GbUDD000*t224 + _GbUDD011*t225 + _GbUDD012*t229 + _GbUDD022*t226 + betU0 + t145*t227 + t160*t228 + V0_lin_vetU0;
  const double t230 = t227*vetU0;
  const double t231 = t228*vetU0;
  out[22 * Ntot + idx] = f0_of_xx0*(_GbUDD100*t224 + _GbUDD101*t230 + _GbUDD102*t231 + _GbUDD111*t225 + _GbUDD112*t229 + _GbUDD122*t226 + t138 - t49*vetU0) + V0_lin_vetU1;
  out[23 * Ntot + idx] = t5*(_GbUDD200*t224 + _GbUDD201*t230 + _GbUDD202*t231 + _GbUDD211*t225 + _GbUDD212*t229 + _GbUDD222*t226 + t152 - t49*t53*t55 - t58*t97) + V0_lin_vetU2;
    }
  }
}

static __device__ __forceinline__ void bssn_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0_tile(const double *__restrict__ in, const double *__restrict__ aux,
        double *__restrict__ out, const double *__restrict__ rfm0, const double *__restrict__ rfm1,
        const bhah_kparams p, const unsigned bx, const unsigned by, const unsigned bz, double *sh) {
  // Tile of 16x8x2 interior points; halo box 22x14x2 = 616 values per gridfunction.
  constexpr int BX = 22, BY = 14, NB = 616, NT = 256, NL = 3;
  const int tid = (int)threadIdx.x;
  const int lx = tid % 16, ly = (tid / 16) % 8, lz = tid / 128;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const int o0 = p.NG + (int)bx * 16, o1 = p.NG + (int)by * 8, o2 = p.NG + (int)bz * 2;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned pofs[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int e = 2 * (tid + NT * j);
    const int ex = e % BX, ey = (e / BX) % BY, ez = e / (BX * BY);
    const int g0 = min(o0 - 3 + ex, p.Nx0 - 2), g1 = min(o1 - 3 + ey, p.Nx1 - 1), g2 = min(o2 - 0 + ez, p.Nx2 - 1);
    pofs[j] = 8u * (unsigned)(g0 + (int)s1 * g1 + (int)s2 * g2);
  }
  const int c0 = (lx + 3) + BX * (ly + 3) + BX * BY * (lz + 0);
  const double ius0 = p.invdxx0 * (1.0 / 12.0), nius0 = -ius0, ikos0 = p.invdxx0 * (1.0 / 64.0);
  const double ius1 = p.invdxx1 * (1.0 / 12.0), nius1 = -ius1, ikos1 = p.invdxx1 * (1.0 / 64.0);
  const double ius2 = p.invdxx2 * (1.0 / 12.0), nius2 = -ius2, ikos2 = p.invdxx2 * (1.0 / 64.0);
  double L0_coef[2], L0_beta[3];
  {
    const int i0 = min(o0 + lx, p.Nx0 - p.NG - 1), i1 = min(o1 + ly, p.Nx1 - p.NG - 1);
    const long idx = i0 + s1 * i1 + s2 * min(o2 + lz + 0, p.Nx2 - p.NG - 1);
    const double f0_of_xx0 = rfm0[i0];
    const double f1_of_xx1 = rfm1[i1];
    const double vetU0 = in[21 * Ntot + idx];
    const double vetU1 = in[22 * Ntot + idx];
    const double vetU2 = in[23 * Ntot + idx];
    L0_coef[0] = vetU0;
    L0_coef[1] = vetU1/f0_of_xx0;
    L0_beta[0] = vetU0;
    L0_beta[1] = vetU1/f0_of_xx0;
    L0_beta[2] = vetU2/(f0_of_xx0*f1_of_xx1);
  }
  double V0_lin_aDD00 = 0.0;
  double V0_lin_aDD01 = 0.0;
  double V0_lin_aDD02 = 0.0;
  double V0_lin_aDD11 = 0.0;
  double V0_lin_aDD12 = 0.0;
  double V0_lin_aDD22 = 0.0;
  double V0_lin_alpha = 0.0;
  double V0_lin_betU0 = 0.0;
  double V0_lin_betU1 = 0.0;
  double V0_lin_betU2 = 0.0;
  double V0_lin_cf = 0.0;
  double V0_lin_hDD00 = 0.0;
  double V0_lin_hDD01 = 0.0;
  double V0_lin_hDD02 = 0.0;
  double V0_lin_hDD11 = 0.0;
  double V0_lin_hDD12 = 0.0;
  double V0_lin_hDD22 = 0.0;
  double V0_lin_lambdaU0 = 0.0;
  double V0_lin_lambdaU1 = 0.0;
  double V0_lin_lambdaU2 = 0.0;
  double V0_lin_trK = 0.0;
  double V0_lin_vetU0 = 0.0;
  double V0_lin_vetU1 = 0.0;
  double V0_lin_vetU2 = 0.0;
  {
    const char *src = (const char *)(in + 0 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  {
    const char *src = (const char *)(in + 1 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  // ---- aDD00
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(0);
  {
    const char *src = (const char *)(in + 2 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD00 = sh[c0];
  const double U0_aDD00_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_aDD00_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_aDD00 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD00_0 : D0_aDD00_0);
  const double U0_aDD00_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_aDD00_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_aDD00 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD00_1 : D0_aDD00_1);
  BHAH_PINS("+v"(V0_aDD00), "+v"(V0_lin_aDD00));
  // ---- aDD01
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(1);
  {
    const char *src = (const char *)(in + 3 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD01 = sh[c0 + 1024];
  const double U0_aDD01_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_aDD01_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD01 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD01_0 : D0_aDD01_0);
  const double U0_aDD01_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_aDD01_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD01 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD01_1 : D0_aDD01_1);
  BHAH_PINS("+v"(V0_aDD01), "+v"(V0_lin_aDD01));
  // ---- aDD02
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(2);
  {
    const char *src = (const char *)(in + 4 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD02 = sh[c0 + 2048];
  const double U0_aDD02_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_aDD02_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD02 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD02_0 : D0_aDD02_0);
  const double U0_aDD02_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_aDD02_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD02 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD02_1 : D0_aDD02_1);
  BHAH_PINS("+v"(V0_aDD02), "+v"(V0_lin_aDD02));
  // ---- aDD11
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(3);
  {
    const char *src = (const char *)(in + 5 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD11 = sh[c0];
  const double U0_aDD11_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_aDD11_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_aDD11 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD11_0 : D0_aDD11_0);
  const double U0_aDD11_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_aDD11_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_aDD11 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD11_1 : D0_aDD11_1);
  BHAH_PINS("+v"(V0_aDD11), "+v"(V0_lin_aDD11));
  // ---- aDD12
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(4);
  {
    const char *src = (const char *)(in + 6 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD12 = sh[c0 + 1024];
  const double U0_aDD12_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_aDD12_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD12 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD12_0 : D0_aDD12_0);
  const double U0_aDD12_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_aDD12_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_aDD12 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD12_1 : D0_aDD12_1);
  BHAH_PINS("+v"(V0_aDD12), "+v"(V0_lin_aDD12));
  // ---- aDD22
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(5);
  {
    const char *src = (const char *)(in + 7 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD22 = sh[c0 + 2048];
  const double U0_aDD22_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_aDD22_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD22 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_aDD22_0 : D0_aDD22_0);
  const double U0_aDD22_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_aDD22_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_aDD22 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_aDD22_1 : D0_aDD22_1);
  BHAH_PINS("+v"(V0_aDD22), "+v"(V0_lin_aDD22));
  // ---- alpha
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(6);
  {
    const char *src = (const char *)(in + 8 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_alpha = sh[c0];
  double V0_alpha_dD0 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_alpha_dD1 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  double V0_alpha_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 1] + sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] + sh[c0 - 2]));
  double V0_alpha_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 23] - sh[c0 - 21]) - (sh[c0 + 21] - sh[c0 - 23])) + (-1.0 / 18.0) * ((sh[c0 + 45] - sh[c0 - 43]) - (sh[c0 + 43] - sh[c0 - 45])) + (-1.0 / 18.0) * ((sh[c0 + 24] - sh[c0 - 20]) - (sh[c0 + 20] - sh[c0 - 24])) + (1.0 / 144.0) * ((sh[c0 + 46] - sh[c0 - 42]) - (sh[c0 + 42] - sh[c0 - 46])));
  double V0_alpha_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 22] + sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] + sh[c0 - 44]));
  const double U0_alpha_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_alpha_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_alpha += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_alpha_0 : D0_alpha_0);
  const double U0_alpha_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_alpha_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_alpha += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_alpha_1 : D0_alpha_1);
  BHAH_PINS("+v"(V0_alpha), "+v"(V0_alpha_dD0), "+v"(V0_alpha_dD1), "+v"(V0_alpha_dDD00), "+v"(V0_alpha_dDD01), "+v"(V0_alpha_dDD11), "+v"(V0_lin_alpha));
  // ---- betU0
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(7);
  {
    const char *src = (const char *)(in + 9 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU0 = sh[c0 + 1024];
  const double U0_betU0_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_betU0_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_betU0 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_betU0_0 : D0_betU0_0);
  const double U0_betU0_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_betU0_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_betU0 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_betU0_1 : D0_betU0_1);
  BHAH_PINS("+v"(V0_betU0), "+v"(V0_lin_betU0));
  // ---- betU1
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(8);
  {
    const char *src = (const char *)(in + 10 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU1 = sh[c0 + 2048];
  const double U0_betU1_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_betU1_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_betU1 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_betU1_0 : D0_betU1_0);
  const double U0_betU1_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_betU1_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_betU1 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_betU1_1 : D0_betU1_1);
  BHAH_PINS("+v"(V0_betU1), "+v"(V0_lin_betU1));
  // ---- betU2
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(9);
  {
    const char *src = (const char *)(in + 11 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU2 = sh[c0];
  const double U0_betU2_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_betU2_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_betU2 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_betU2_0 : D0_betU2_0);
  const double U0_betU2_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_betU2_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_betU2 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_betU2_1 : D0_betU2_1);
  BHAH_PINS("+v"(V0_betU2), "+v"(V0_lin_betU2));
  // ---- cf
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(10);
  {
    const char *src = (const char *)(in + 12 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_cf = sh[c0 + 1024];
  double V0_cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  double V0_cf_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1025] + sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] + sh[c0 + 1022]));
  double V0_cf_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 1047] - sh[c0 + 1003]) - (sh[c0 + 1045] - sh[c0 + 1001])) + (-1.0 / 18.0) * ((sh[c0 + 1069] - sh[c0 + 981]) - (sh[c0 + 1067] - sh[c0 + 979])) + (-1.0 / 18.0) * ((sh[c0 + 1048] - sh[c0 + 1004]) - (sh[c0 + 1044] - sh[c0 + 1000])) + (1.0 / 144.0) * ((sh[c0 + 1070] - sh[c0 + 982]) - (sh[c0 + 1066] - sh[c0 + 978])));
  double V0_cf_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1046] + sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] + sh[c0 + 980]));
  const double U0_cf_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_cf_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_cf += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_cf_0 : D0_cf_0);
  const double U0_cf_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_cf_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_cf += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_cf_1 : D0_cf_1);
  BHAH_PINS("+v"(V0_cf), "+v"(V0_cf_dD0), "+v"(V0_cf_dD1), "+v"(V0_cf_dDD00), "+v"(V0_cf_dDD01), "+v"(V0_cf_dDD11), "+v"(V0_lin_cf));
  // ---- hDD00
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(11);
  {
    const char *src = (const char *)(in + 13 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD00 = sh[c0 + 2048];
  double V0_hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  const double U0_hDD00_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_hDD00_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD00 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD00_0 : D0_hDD00_0);
  const double U0_hDD00_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_hDD00_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD00 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD00_1 : D0_hDD00_1);
  BHAH_PINS("+v"(V0_hDD00), "+v"(V0_hDD_dD000), "+v"(V0_hDD_dD001), "+v"(V0_lin_hDD00));
  // ---- hDD01
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(12);
  {
    const char *src = (const char *)(in + 14 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD01 = sh[c0];
  double V0_hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  const double U0_hDD01_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_hDD01_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_hDD01 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD01_0 : D0_hDD01_0);
  const double U0_hDD01_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_hDD01_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_hDD01 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD01_1 : D0_hDD01_1);
  BHAH_PINS("+v"(V0_hDD01), "+v"(V0_hDD_dD010), "+v"(V0_hDD_dD011), "+v"(V0_lin_hDD01));
  // ---- hDD02
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(13);
  {
    const char *src = (const char *)(in + 15 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD02 = sh[c0 + 1024];
  double V0_hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  const double U0_hDD02_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_hDD02_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD02 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD02_0 : D0_hDD02_0);
  const double U0_hDD02_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_hDD02_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD02 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD02_1 : D0_hDD02_1);
  BHAH_PINS("+v"(V0_hDD02), "+v"(V0_hDD_dD020), "+v"(V0_hDD_dD021), "+v"(V0_lin_hDD02));
  // ---- hDD11
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(14);
  {
    const char *src = (const char *)(in + 16 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD11 = sh[c0 + 2048];
  double V0_hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  const double U0_hDD11_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_hDD11_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD11 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD11_0 : D0_hDD11_0);
  const double U0_hDD11_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_hDD11_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_hDD11 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD11_1 : D0_hDD11_1);
  BHAH_PINS("+v"(V0_hDD11), "+v"(V0_hDD_dD110), "+v"(V0_hDD_dD111), "+v"(V0_lin_hDD11));
  // ---- hDD12
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(15);
  {
    const char *src = (const char *)(in + 17 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD12 = sh[c0];
  double V0_hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  const double U0_hDD12_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_hDD12_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_hDD12 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD12_0 : D0_hDD12_0);
  const double U0_hDD12_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_hDD12_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_hDD12 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD12_1 : D0_hDD12_1);
  BHAH_PINS("+v"(V0_hDD12), "+v"(V0_hDD_dD120), "+v"(V0_hDD_dD121), "+v"(V0_lin_hDD12));
  // ---- hDD22
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(16);
  {
    const char *src = (const char *)(in + 18 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD22 = sh[c0 + 1024];
  double V0_hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  const double U0_hDD22_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_hDD22_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD22 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_hDD22_0 : D0_hDD22_0);
  const double U0_hDD22_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_hDD22_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_hDD22 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_hDD22_1 : D0_hDD22_1);
  BHAH_PINS("+v"(V0_hDD22), "+v"(V0_hDD_dD220), "+v"(V0_hDD_dD221), "+v"(V0_lin_hDD22));
  // ---- lambdaU0
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(17);
  {
    const char *src = (const char *)(in + 19 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU0 = sh[c0 + 2048];
  const double U0_lambdaU0_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_lambdaU0_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_lambdaU0 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_lambdaU0_0 : D0_lambdaU0_0);
  const double U0_lambdaU0_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_lambdaU0_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_lambdaU0 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_lambdaU0_1 : D0_lambdaU0_1);
  BHAH_PINS("+v"(V0_lambdaU0), "+v"(V0_lin_lambdaU0));
  // ---- lambdaU1
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(18);
  {
    const char *src = (const char *)(in + 20 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU1 = sh[c0];
  const double U0_lambdaU1_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_lambdaU1_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_lambdaU1 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_lambdaU1_0 : D0_lambdaU1_0);
  const double U0_lambdaU1_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_lambdaU1_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_lambdaU1 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_lambdaU1_1 : D0_lambdaU1_1);
  BHAH_PINS("+v"(V0_lambdaU1), "+v"(V0_lin_lambdaU1));
  // ---- lambdaU2
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(19);
  {
    const char *src = (const char *)(in + 21 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU2 = sh[c0 + 1024];
  const double U0_lambdaU2_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_lambdaU2_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_lambdaU2 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_lambdaU2_0 : D0_lambdaU2_0);
  const double U0_lambdaU2_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_lambdaU2_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_lambdaU2 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_lambdaU2_1 : D0_lambdaU2_1);
  BHAH_PINS("+v"(V0_lambdaU2), "+v"(V0_lin_lambdaU2));
  // ---- trK
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(20);
  {
    const char *src = (const char *)(in + 22 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 1024 + 2 * (NT * j + 64 * wv));
  }
  double V0_trK = sh[c0 + 2048];
  double V0_trK_dD0 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_trK_dD1 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  const double U0_trK_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_trK_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_trK += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_trK_0 : D0_trK_0);
  const double U0_trK_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_trK_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_trK += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_trK_1 : D0_trK_1);
  BHAH_PINS("+v"(V0_trK), "+v"(V0_trK_dD0), "+v"(V0_trK_dD1), "+v"(V0_lin_trK));
  // ---- vetU0
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(21);
  {
    const char *src = (const char *)(in + 23 * Ntot);
#pragma unroll
    for (int j = 0; j < 2; j++) BHAH_DMA16O(src, pofs[j], sh + 2048 + 2 * (NT * j + 64 * wv));
  }
  double V0_vetU0 = sh[c0];
  double V0_vetU_dD00 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] - sh[c0 - 2]));
  double V0_vetU_dD01 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 22] - sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] - sh[c0 - 44]));
  double V0_vetU_dDD000 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 1] + sh[c0 - 1]) + (-1.0 / 12.0) * (sh[c0 + 2] + sh[c0 - 2]));
  double V0_vetU_dDD001 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 23] - sh[c0 - 21]) - (sh[c0 + 21] - sh[c0 - 23])) + (-1.0 / 18.0) * ((sh[c0 + 45] - sh[c0 - 43]) - (sh[c0 + 43] - sh[c0 - 45])) + (-1.0 / 18.0) * ((sh[c0 + 24] - sh[c0 - 20]) - (sh[c0 + 20] - sh[c0 - 24])) + (1.0 / 144.0) * ((sh[c0 + 46] - sh[c0 - 42]) - (sh[c0 + 42] - sh[c0 - 46])));
  double V0_vetU_dDD011 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0] + (4.0 / 3.0) * (sh[c0 + 22] + sh[c0 - 22]) + (-1.0 / 12.0) * (sh[c0 + 44] + sh[c0 - 44]));
  const double U0_vetU0_0 = ius0 * (sh[c0 + 3] + -6.0 * sh[c0 + 2] + -3.0 * sh[c0 - 1] + 18.0 * sh[c0 + 1] + -10.0 * sh[c0]), D0_vetU0_0 = nius0 * (sh[c0 - 3] + -6.0 * sh[c0 - 2] + 18.0 * sh[c0 - 1] + -3.0 * sh[c0 + 1] + -10.0 * sh[c0]);
  V0_lin_vetU0 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_vetU0_0 : D0_vetU0_0);
  const double U0_vetU0_1 = ius1 * (sh[c0 + 66] + -6.0 * sh[c0 + 44] + -3.0 * sh[c0 - 22] + 18.0 * sh[c0 + 22] + -10.0 * sh[c0]), D0_vetU0_1 = nius1 * (sh[c0 - 66] + -6.0 * sh[c0 - 44] + 18.0 * sh[c0 - 22] + -3.0 * sh[c0 + 22] + -10.0 * sh[c0]);
  V0_lin_vetU0 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_vetU0_1 : D0_vetU0_1);
  BHAH_PINS("+v"(V0_vetU0), "+v"(V0_vetU_dD00), "+v"(V0_vetU_dD01), "+v"(V0_vetU_dDD000), "+v"(V0_vetU_dDD001), "+v"(V0_vetU_dDD011), "+v"(V0_lin_vetU0));
  // ---- vetU1
  BHAH_VMWAIT(2);
  BHAH_BARRIER_PHASE(22);
  double V0_vetU1 = sh[c0 + 1024];
  double V0_vetU_dD10 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 1025] - sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] - sh[c0 + 1022]));
  double V0_vetU_dD11 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 1046] - sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] - sh[c0 + 980]));
  double V0_vetU_dDD100 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1025] + sh[c0 + 1023]) + (-1.0 / 12.0) * (sh[c0 + 1026] + sh[c0 + 1022]));
  double V0_vetU_dDD101 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 1047] - sh[c0 + 1003]) - (sh[c0 + 1045] - sh[c0 + 1001])) + (-1.0 / 18.0) * ((sh[c0 + 1069] - sh[c0 + 981]) - (sh[c0 + 1067] - sh[c0 + 979])) + (-1.0 / 18.0) * ((sh[c0 + 1048] - sh[c0 + 1004]) - (sh[c0 + 1044] - sh[c0 + 1000])) + (1.0 / 144.0) * ((sh[c0 + 1070] - sh[c0 + 982]) - (sh[c0 + 1066] - sh[c0 + 978])));
  double V0_vetU_dDD111 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0 + 1024] + (4.0 / 3.0) * (sh[c0 + 1046] + sh[c0 + 1002]) + (-1.0 / 12.0) * (sh[c0 + 1068] + sh[c0 + 980]));
  const double U0_vetU1_0 = ius0 * (sh[c0 + 1027] + -6.0 * sh[c0 + 1026] + -3.0 * sh[c0 + 1023] + 18.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]), D0_vetU1_0 = nius0 * (sh[c0 + 1021] + -6.0 * sh[c0 + 1022] + 18.0 * sh[c0 + 1023] + -3.0 * sh[c0 + 1025] + -10.0 * sh[c0 + 1024]);
  V0_lin_vetU1 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_vetU1_0 : D0_vetU1_0);
  const double U0_vetU1_1 = ius1 * (sh[c0 + 1090] + -6.0 * sh[c0 + 1068] + -3.0 * sh[c0 + 1002] + 18.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]), D0_vetU1_1 = nius1 * (sh[c0 + 958] + -6.0 * sh[c0 + 980] + 18.0 * sh[c0 + 1002] + -3.0 * sh[c0 + 1046] + -10.0 * sh[c0 + 1024]);
  V0_lin_vetU1 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_vetU1_1 : D0_vetU1_1);
  BHAH_PINS("+v"(V0_vetU1), "+v"(V0_vetU_dD10), "+v"(V0_vetU_dD11), "+v"(V0_vetU_dDD100), "+v"(V0_vetU_dDD101), "+v"(V0_vetU_dDD111), "+v"(V0_lin_vetU1));
  // ---- vetU2
  BHAH_VMWAIT(0);
  BHAH_BARRIER_PHASE(23);
  double V0_vetU2 = sh[c0 + 2048];
  double V0_vetU_dD20 = p.invdxx0 * ((2.0 / 3.0) * (sh[c0 + 2049] - sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] - sh[c0 + 2046]));
  double V0_vetU_dD21 = p.invdxx1 * ((2.0 / 3.0) * (sh[c0 + 2070] - sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] - sh[c0 + 2004]));
  double V0_vetU_dDD200 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * sh[c0 + 2048] + (4.0 / 3.0) * (sh[c0 + 2049] + sh[c0 + 2047]) + (-1.0 / 12.0) * (sh[c0 + 2050] + sh[c0 + 2046]));
  double V0_vetU_dDD201 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((sh[c0 + 2071] - sh[c0 + 2027]) - (sh[c0 + 2069] - sh[c0 + 2025])) + (-1.0 / 18.0) * ((sh[c0 + 2093] - sh[c0 + 2005]) - (sh[c0 + 2091] - sh[c0 + 2003])) + (-1.0 / 18.0) * ((sh[c0 + 2072] - sh[c0 + 2028]) - (sh[c0 + 2068] - sh[c0 + 2024])) + (1.0 / 144.0) * ((sh[c0 + 2094] - sh[c0 + 2006]) - (sh[c0 + 2090] - sh[c0 + 2002])));
  double V0_vetU_dDD211 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * sh[c0 + 2048] + (4.0 / 3.0) * (sh[c0 + 2070] + sh[c0 + 2026]) + (-1.0 / 12.0) * (sh[c0 + 2092] + sh[c0 + 2004]));
  const double U0_vetU2_0 = ius0 * (sh[c0 + 2051] + -6.0 * sh[c0 + 2050] + -3.0 * sh[c0 + 2047] + 18.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]), D0_vetU2_0 = nius0 * (sh[c0 + 2045] + -6.0 * sh[c0 + 2046] + 18.0 * sh[c0 + 2047] + -3.0 * sh[c0 + 2049] + -10.0 * sh[c0 + 2048]);
  V0_lin_vetU2 += L0_coef[0] * ((L0_beta[0] > 0.0) ? U0_vetU2_0 : D0_vetU2_0);
  const double U0_vetU2_1 = ius1 * (sh[c0 + 2114] + -6.0 * sh[c0 + 2092] + -3.0 * sh[c0 + 2026] + 18.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]), D0_vetU2_1 = nius1 * (sh[c0 + 1982] + -6.0 * sh[c0 + 2004] + 18.0 * sh[c0 + 2026] + -3.0 * sh[c0 + 2070] + -10.0 * sh[c0 + 2048]);
  V0_lin_vetU2 += L0_coef[1] * ((L0_beta[1] > 0.0) ? U0_vetU2_1 : D0_vetU2_1);
  BHAH_PINS("+v"(V0_vetU2), "+v"(V0_vetU_dD20), "+v"(V0_vetU_dD21), "+v"(V0_vetU_dDD200), "+v"(V0_vetU_dDD201), "+v"(V0_vetU_dDD211), "+v"(V0_lin_vetU2));
  {
    const int i0 = o0 + lx, i1 = o1 + ly, i2 = o2 + lz + 0;
    if (i0 < p.Nx0 - p.NG && i1 < p.Nx1 - p.NG && i2 < p.Nx2 - p.NG) {
      const long idx = i0 + s1 * i1 + s2 * i2;
  const double f0_of_xx0 = rfm0[i0];
  const double f1_of_xx1 = rfm1[i1];
  const double t5 = f0_of_xx0*f1_of_xx1;
  const double aDD02 = V0_aDD02;
  const double _AbDD02 = aDD02*t5;
  const double aDD01 = V0_aDD01;
  const double _AbDD01 = aDD01*f0_of_xx0;
  const double hDD01 = V0_hDD01;
  const double _gbDD01 = f0_of_xx0*hDD01;
  const double hDD02 = V0_hDD02;
  const double t0 = f1_of_xx1*hDD02;
  const double _gbDD02 = f0_of_xx0*t0;
  const double t1 = (f0_of_xx0*f0_of_xx0);
  const double t2 = f1_of_xx1*t1;
  const double hDD12 = V0_hDD12;
  const double _gbDD12 = hDD12*t2;
  const double t3 = (f1_of_xx1*f1_of_xx1);
  const double t4 = t1*t3;
  const double hDD22 = V0_hDD22;
  const double _gbDD22 = hDD22*t4 + t4;
  const double hDD00 = V0_hDD00;
  const double _gbDD00 = hDD00 + 1.0;
  const double hDD11 = V0_hDD11;
  const double _gbDD11 = hDD11*t1 + t1;
  const double t6 = (_gbDD12*_gbDD12);
  const double t7 = (_gbDD02*_gbDD02);
  const double t8 = (_gbDD01*_gbDD01);
  const double t9 = (1.0 / (_gbDD00*_gbDD11*_gbDD22 - _gbDD00*t6 + 2.0*_gbDD01*_gbDD02*_gbDD12 - _gbDD11*t7 - _gbDD22*t8));
  const double _gbUU01 = t9*(-_gbDD01*_gbDD22 + _gbDD02*_gbDD12);
  const double t34 = _AbDD01*_gbUU01;
  const double _gbUU02 = t9*(_gbDD01*_gbDD12 - _gbDD02*_gbDD11);
  const double t35 = _AbDD02*_gbUU02;
  const double _gbUU00 = t9*(_gbDD11*_gbDD22 - t6);
  const double aDD00 = V0_aDD00;
  const double t36 = _gbUU00*aDD00;
  const double _AbUD00 = t34 + t35 + t36;
  const double _gbUU11 = t9*(_gbDD00*_gbDD22 - t7);
  const double _gbUU12 = t9*(-_gbDD00*_gbDD12 + _gbDD01*_gbDD02);
  const double _AbUD10 = _AbDD01*_gbUU11 + _AbDD02*_gbUU12 + _gbUU01*aDD00;
  const double _gbUU22 = t9*(_gbDD00*_gbDD11 - t8);
  const double _AbUD20 = _AbDD01*_gbUU12 + _AbDD02*_gbUU22 + _gbUU02*aDD00;
  const double t41 = (1.0 / f0_of_xx0);
  const double t48 = (1.0 / t1);
  const double vetU1 = V0_vetU1;
  const double t49 = t48*vetU1;
  const double vetU_dD10 = V0_vetU_dD10;
  const double _bUdD10 = t41*vetU_dD10 - t49;
  const double hDD_dD020 = V0_hDD_dD020;
  const double _gbDDdD020 = hDD_dD020*t5 + t0;
  const double t21 = (Rational_1_2)*_gbUU00;
  const double hDD_dD010 = V0_hDD_dD010;
  const double _gbDDdD010 = f0_of_xx0*hDD_dD010 + hDD01;
  const double hDD_dD001 = V0_hDD_dD001;
  const double t22 = 2.0*_gbDDdD010 - hDD_dD001;
  const double t23 = (Rational_1_2)*_gbUU01;
  const double hDD_dD000 = V0_hDD_dD000;
  const double _GbUDD000 = _gbDDdD020*_gbUU02 + hDD_dD000*t21 + t22*t23;
  const double t30 = (Rational_1_2)*_gbUU11;
  const double _GbUDD100 = _gbDDdD020*_gbUU12 + hDD_dD000*t23 + t22*t30;
  const double alpha_dD0 = V0_alpha_dD0;
  const double alpha_dD1 = V0_alpha_dD1;
  const double alpha_dDD00 = V0_alpha_dDD00;
  const double _adBDD00 = -_GbUDD000*alpha_dD0 - _GbUDD100*alpha_dD1 + alpha_dDD00;
  const double cf = V0_cf;
  const double t63 = (1.0 / cf);
  const double t64 = (Rational_1_2)*t63;
  const double cf_dD0 = V0_cf_dD0;
  const double _phidD0 = -cf_dD0*t64;
  const double cf_dD1 = V0_cf_dD1;
  const double _phidD1 = -cf_dD1*t64;
  const double cf_dDD00 = V0_cf_dDD00;
  const double _phidBDD00 = -_GbUDD000*_phidD0 - _GbUDD100*_phidD1 + (Rational_1_2)*t63*((cf_dD0*cf_dD0)*t63 - cf_dDD00);
  const double alpha = V0_alpha;
  const double t67 = 2.0*alpha;
  const double t68 = _phidD0*alpha_dD0;
  const double t69 = 4.0*alpha;
  const double RbarDD00 = aux[0 * Ntot + idx];
  const double _curly00 = RbarDD00*alpha - _adBDD00 - _phidBDD00*t67 + (_phidD0*_phidD0)*t69 + 4.0*t68;
  const double t73 = (cf*cf);
  const double t11 = 2.0*f0_of_xx0;
  const double t12 = hDD11*t11 + t11;
  const double hDD_dD110 = V0_hDD_dD110;
  const double _gbDDdD110 = hDD_dD110*t1 + t12;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t10 = f1_of_xx1__D1*hDD02;
  const double hDD_dD021 = V0_hDD_dD021;
  const double _gbDDdD021 = f0_of_xx0*t10 + hDD_dD021*t5;
  const double t13 = hDD12*t11;
  const double hDD_dD120 = V0_hDD_dD120;
  const double _gbDDdD120 = f1_of_xx1*t13 + hDD_dD120*t2;
  const double t24 = _gbDDdD021 + _gbDDdD120;
  const double t25 = (Rational_1_2)*_gbUU02;
  const double _GbUDD001 = _gbDDdD110*t23 + hDD_dD001*t21 + t24*t25;
  const double t31 = (Rational_1_2)*_gbUU12;
  const double _GbUDD101 = _gbDDdD110*t30 + hDD_dD001*t23 + t24*t31;
  const double alpha_dDD01 = V0_alpha_dDD01;
  const double _adBDD01 = -_GbUDD001*alpha_dD0 - _GbUDD101*alpha_dD1 + alpha_dDD01;
  const double cf_dDD01 = V0_cf_dDD01;
  const double _phidBDD01 = -_GbUDD001*_phidD0 - _GbUDD101*_phidD1 + (Rational_1_2)*t63*(cf_dD0*cf_dD1*t63 - cf_dDD01);
  const double t70 = 2.0*alpha_dD1;
  const double t71 = _phidD0*t70;
  const double t72 = 2.0*_phidD1*alpha_dD0;
  const double RbarDD01 = aux[1 * Ntot + idx];
  const double _curly01 = RbarDD01*alpha - _adBDD01 - _phidBDD01*t67 + _phidD0*_phidD1*t69 + t71 + t72;
  const double t15 = t11*t3;
  const double t16 = hDD22*t15 + t15;
  const double hDD_dD220 = V0_hDD_dD220;
  const double _gbDDdD220 = hDD_dD220*t4 + t16;
  const double t26 = _gbDDdD220*t25;
  const double t27 = _gbDDdD021 - _gbDDdD120;
  const double t28 = -t27;
  const double _GbUDD002 = t23*t28 + t26;
  const double _GbUDD102 = _gbDDdD220*t31 + t28*t30;
  const double _adBDD02 = -_GbUDD002*alpha_dD0 - _GbUDD102*alpha_dD1;
  const double _phidBDD02 = -_GbUDD002*_phidD0 - _GbUDD102*_phidD1;
  const double RbarDD02 = aux[2 * Ntot + idx];
  const double _curly02 = RbarDD02*alpha - _adBDD02 - _phidBDD02*t67;
  const double hDD_dD111 = V0_hDD_dD111;
  const double _gbDDdD111 = hDD_dD111*t1;
  const double t14 = f1_of_xx1__D1*hDD12;
  const double hDD_dD121 = V0_hDD_dD121;
  const double _gbDDdD121 = hDD_dD121*t2 + t1*t14;
  const double hDD_dD011 = V0_hDD_dD011;
  const double _gbDDdD011 = f0_of_xx0*hDD_dD011;
  const double t29 = 2.0*_gbDDdD011 - _gbDDdD110;
  const double _GbUDD011 = _gbDDdD111*t23 + _gbDDdD121*_gbUU02 + t21*t29;
  const double _GbUDD111 = _gbDDdD111*t30 + _gbDDdD121*_gbUU12 + t23*t29;
  const double alpha_dDD11 = V0_alpha_dDD11;
  const double _adBDD11 = -_GbUDD011*alpha_dD0 - _GbUDD111*alpha_dD1 + alpha_dDD11;
  const double cf_dDD11 = V0_cf_dDD11;
  const double _phidBDD11 = -_GbUDD011*_phidD0 - _GbUDD111*_phidD1 + (Rational_1_2)*t63*((cf_dD1*cf_dD1)*t63 - cf_dDD11);
  const double RbarDD11 = aux[3 * Ntot + idx];
  const double _curly11 = RbarDD11*alpha - _adBDD11 - _phidBDD11*t67 + (_phidD1*_phidD1)*t69 + 4.0*_phidD1*alpha_dD1;
  const double t17 = f1_of_xx1*f1_of_xx1__D1;
  const double t18 = 2.0*t17;
  const double t19 = t1*t18;
  const double t20 = hDD22*t19 + t19;
  const double hDD_dD221 = V0_hDD_dD221;
  const double _gbDDdD221 = hDD_dD221*t4 + t20;
  const double _GbUDD012 = _gbDDdD221*t25 + t21*t27;
  const double t32 = _gbDDdD221*t31;
  const double _GbUDD112 = t23*t27 + t32;
  const double _adBDD12 = -_GbUDD012*alpha_dD0 - _GbUDD112*alpha_dD1;
  const double _phidBDD12 = -_GbUDD012*_phidD0 - _GbUDD112*_phidD1;
  const double RbarDD12 = aux[4 * Ntot + idx];
  const double _curly12 = RbarDD12*alpha - _adBDD12 - _phidBDD12*t67;
  const double _GbUDD022 = -_gbDDdD220*t21 - _gbDDdD221*t23;
  const double _GbUDD122 = -_gbDDdD220*t23 - _gbDDdD221*t30;
  const double _adBDD22 = -_GbUDD022*alpha_dD0 - _GbUDD122*alpha_dD1;
  const double _phidBDD22 = -_GbUDD022*_phidD0 - _GbUDD122*_phidD1;
  const double RbarDD22 = aux[5 * Ntot + idx];
  const double _curly22 = RbarDD22*alpha - _adBDD22 - _phidBDD22*t67;
  const double t45 = 2.0*_gbUU01;
  const double t46 = 2.0*_gbUU02;
  const double t47 = 2.0*_gbUU12;
  const double _curlytr = _curly00*_gbUU00 + _curly01*t45 + _curly02*t46 + _curly11*_gbUU11 + _curly12*t47 + _curly22*_gbUU22;
  const double t74 = (Rational_1_3)*_curlytr;
  const double t75 = 2.0*_AbDD01;
  const double t43 = (1.0 / f1_of_xx1);
  const double t50 = t41*t43;
  const double t51 = t43*t48;
  const double vetU2 = V0_vetU2;
  const double t52 = t51*vetU2;
  const double vetU_dD20 = V0_vetU_dD20;
  const double _bUdD20 = t50*vetU_dD20 - t52;
  const double t76 = 2.0*_bUdD20;
  const double vetU_dD00 = V0_vetU_dD00;
  const double t77 = 2.0*vetU_dD00;
  const double vetU_dD11 = V0_vetU_dD11;
  const double _bUdD11 = t41*vetU_dD11;
  const double t44 = f1_of_xx1__D1*t43;
  const double t65 = 2.0*t41;
  const double t66 = t41*vetU1;
  const double vetU0 = V0_vetU0;
  const double _Dbb = _bUdD11 + t44*t66 + t65*vetU0 + vetU_dD00;
  const double t78 = (Rational_2_3)*_Dbb;
  const double trK = V0_trK;
  const double t79 = alpha*trK;
  const double t80 = _AbDD01*t67;
  const double t81 = _AbDD02*t67;
  const double t82 = aDD00*t67;
  out[0 * Ntot + idx] = _AbDD02*t76 - _AbUD00*t82 - _AbUD10*t80 - _AbUD20*t81 + _bUdD10*t75 + aDD00*t77 - aDD00*t78 + aDD00*t79 + t73*(_curly00 - _gbDD00*t74) + V0_lin_aDD00;
  const double aDD11 = V0_aDD11;
  const double _AbDD11 = aDD11*t1;
  const double aDD12 = V0_aDD12;
  const double _AbDD12 = aDD12*t2;
  const double _AbUD01 = _AbDD01*_gbUU00 + _AbDD11*_gbUU01 + _AbDD12*_gbUU02;
  const double t37 = _AbDD11*_gbUU11;
  const double t38 = _AbDD12*_gbUU12;
  const double _AbUD11 = t34 + t37 + t38;
  const double _AbUD21 = _AbDD01*_gbUU02 + _AbDD11*_gbUU12 + _AbDD12*_gbUU22;
  const double t53 = (1.0 / t3);
  const double t54 = t41*t53;
  const double t55 = f1_of_xx1__D1*vetU2;
  const double vetU_dD21 = V0_vetU_dD21;
  const double _bUdD21 = t50*vetU_dD21 - t54*t55;
  const double vetU_dD01 = V0_vetU_dD01;
  out[1 * Ntot + idx] = t41*(_AbDD01*_bUdD11 - _AbDD01*t78 + _AbDD01*t79 + _AbDD01*vetU_dD00 + _AbDD02*_bUdD21 + _AbDD11*_bUdD10 + _AbDD12*_bUdD20 - _AbUD01*t82 - _AbUD11*t80 - _AbUD21*t81 + aDD00*vetU_dD01 + aDD01*vetU0 + t73*(_curly01 - _gbDD01*t74)) + V0_lin_aDD01;
  const double aDD22 = V0_aDD22;
  const double _AbDD22 = aDD22*t4;
  const double _AbUD02 = _AbDD02*_gbUU00 + _AbDD12*_gbUU01 + _AbDD22*_gbUU02;
  const double _AbUD12 = _AbDD02*_gbUU01 + _AbDD12*_gbUU11 + _AbDD22*_gbUU12;
  const double t39 = _AbDD22*_gbUU22;
  const double _AbUD22 = t35 + t38 + t39;
  const double t83 = f1_of_xx1*vetU0;
  const double t84 = f1_of_xx1__D1*vetU1;
  out[2 * Ntot + idx] = t50*(-_AbDD02*t78 + _AbDD02*t79 + _AbDD02*vetU_dD00 + _AbDD12*_bUdD10 + _AbDD22*_bUdD20 - _AbUD02*t82 - _AbUD12*t80 - _AbUD22*t81 + aDD02*t83 + aDD02*t84 + t73*(_curly02 - _gbDD02*t74)) + V0_lin_aDD02;
  const double t85 = 2.0*_bUdD11;
  const double t86 = 2.0*_bUdD21;
  const double t87 = _AbDD11*t67;
  const double t88 = _AbDD12*t67;
  out[3 * Ntot + idx] = t48*(-_AbDD11*t78 + _AbDD11*t79 + _AbDD11*t85 + _AbDD12*t86 - _AbUD01*t80 - _AbUD11*t87 - _AbUD21*t88 + aDD11*t11*vetU0 + t73*(_curly11 - _gbDD11*t74) + t75*vetU_dD01) + V0_lin_aDD11;
  out[4 * Ntot + idx] = t51*(_AbDD02*vetU_dD01 + _AbDD12*_bUdD11 - _AbDD12*t78 + _AbDD12*t79 + _AbDD22*_bUdD21 - _AbUD02*t80 - _AbUD12*t87 - _AbUD22*t88 + aDD12*f0_of_xx0*t84 + aDD12*t11*t83 + t73*(_curly12 - _gbDD12*t74)) + V0_lin_aDD12;
  const double t59 = t48*t53;
  const double t89 = _AbDD22*t67;
  out[5 * Ntot + idx] = t59*(_AbDD22*alpha*trK - _AbDD22*t78 - _AbUD02*t81 - _AbUD12*t88 - _AbUD22*t89 + 2.0*aDD22*f0_of_xx0*f1_of_xx1*f1_of_xx1__D1*vetU1 + 2.0*aDD22*f0_of_xx0*t3*vetU0 + t73*(_curly22 - _gbDD22*t74)) + V0_lin_aDD22;
  out[6 * Ntot + idx] = -t67*trK + V0_lin_alpha;
  const double _AbUU00 = _AbUD00*_gbUU00 + _AbUD01*_gbUU01 + _AbUD02*_gbUU02;
  const double _AbUU01 = _AbUD00*_gbUU01 + _AbUD01*_gbUU11 + _AbUD02*_gbUU12;
  const double _AbUU02 = _AbUD00*_gbUU02 + _AbUD01*_gbUU12 + _AbUD02*_gbUU22;
  const double _AbUU12 = _AbUD10*_gbUU02 + _AbUD11*_gbUU12 + _AbUD12*_gbUU22;
  const double _AbUU20 = _AbUD20*_gbUU00 + _AbUD21*_gbUU01 + _AbUD22*_gbUU02;
  const double _AbUU21 = _AbUD20*_gbUU01 + _AbUD21*_gbUU11 + _AbUD22*_gbUU12;
  const double _DGUDD011 = _GbUDD011 + f0_of_xx0;
  const double t40 = f0_of_xx0*t3;
  const double _DGUDD022 = _GbUDD022 + t40;
  const double _DGU0 = _DGUDD011*_gbUU11 + _DGUDD022*_gbUU22 + _GbUDD000*_gbUU00 + _GbUDD001*t45 + _GbUDD002*t46 + _GbUDD012*t47;
  const double vetU_dDD101 = V0_vetU_dDD101;
  const double _bUdDD101 = t41*vetU_dDD101 - t48*vetU_dD11;
  const double t99 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t100 = (Rational_1_2)*t53/t99;
  const double t101 = 2.0*t99;
  const double t102 = 8.0*t17;
  const double t103 = 4.0*t44;
  const double t97 = t48*vetU0;
  const double t56 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t98 = 4.0*t3*t56;
  const double vetU_dDD000 = V0_vetU_dDD000;
  const double t104 = _bUdDD101 + t100*(12.0*t4*vetU0 + t98*vetU_dD00) + t100*(_bUdD10*t101*t17 + t1*t102*vetU1) - t103*t49 - 8.0*t97 + vetU_dDD000;
  const double t105 = (Rational_1_4)*t104;
  const double vetU_dDD111 = V0_vetU_dDD111;
  const double _bUdDD111 = t41*vetU_dDD111;
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double t106 = f1_of_xx1*f1_of_xx1__DD11;
  const double t62 = (f1_of_xx1__D1*f1_of_xx1__D1);
  const double t107 = t53*t62;
  const double t108 = t107*t66;
  const double vetU_dDD001 = V0_vetU_dDD001;
  const double t109 = _bUdDD111 + t100*(t102*t56*vetU0 + t98*vetU_dD01) + t100*(t17*t85*t99 + t66*(t101*t106 + t101*t62)) - t103*t41*vetU0 - 2.0*t108 + vetU_dDD001;
  const double t110 = (Rational_1_4)*t109;
  const double t111 = _bUdD10*f0_of_xx0;
  const double t112 = t41*vetU_dD01;
  const double t113 = -t111 - t112 + vetU_dDD001;
  const double t114 = (Rational_3_2)*_gbUU01;
  const double t115 = _gbUU00*vetU_dDD000;
  const double vetU_dDD011 = V0_vetU_dDD011;
  const double t116 = _gbUU11*(-_bUdD11*t11 + f0_of_xx0*vetU_dD00 - vetU0 + vetU_dDD011);
  const double t117 = _gbUU22*(t17*vetU_dD01 - t18*vetU1 - t3*vetU0 + t40*vetU_dD00);
  const double betU0 = V0_betU0;
  const double t118 = betU0*vetU0;
  const double trK_dD0 = V0_trK_dD0;
  const double t119 = alpha*trK_dD0;
  const double t120 = _gbUU00*t119;
  const double trK_dD1 = V0_trK_dD1;
  const double t121 = alpha*trK_dD1;
  const double t122 = _gbUU01*t121;
  const double lambdaU0 = V0_lambdaU0;
  const double t123 = (Rational_3_4)*lambdaU0;
  const double t124 = t123*vetU0;
  const double lambdaU1 = V0_lambdaU1;
  const double t125 = lambdaU1*t112;
  const double t126 = _AbUU00*alpha;
  const double t127 = (Rational_3_2)*t126;
  const double t128 = (Rational_3_2)*alpha;
  const double t129 = _AbUU01*_GbUDD001;
  const double t130 = _GbUDD002*t128;
  const double _AbUU10 = _AbUD10*_gbUU00 + _AbUD11*_gbUU01 + _AbUD12*_gbUU02;
  const double t131 = _AbUU10*t128;
  const double _AbUU11 = _AbUD10*_gbUU01 + _AbUD11*_gbUU11 + _AbUD12*_gbUU12;
  const double t132 = _AbUU11*alpha;
  const double t133 = (Rational_3_2)*t132;
  const double t134 = _GbUDD012*t128;
  const double _AbUU22 = _AbUD20*_gbUU02 + _AbUD21*_gbUU12 + _AbUD22*_gbUU22;
  const double t135 = _AbUU22*alpha;
  const double t136 = (Rational_3_2)*t135;
  const double t137 = betU0*t66;
  const double betU1 = V0_betU1;
  const double t138 = betU1*t41;
  const double t139 = t138*vetU0;
  const double t140 = betU1*t49;
  const double t141 = (Rational_3_2)*_gbUU02;
  const double t142 = _bUdD20*t40;
  const double t143 = _bUdD21*_gbUU12;
  const double t144 = t123*t66;
  const double t145 = _GbUDD001*vetU0;
  const double t146 = lambdaU1*t41;
  const double t147 = (Rational_3_4)*t146;
  const double t148 = (Rational_3_4)*lambdaU1;
  const double t149 = t148*t49;
  const double t150 = t50*vetU2;
  const double t151 = betU0*t150;
  const double betU2 = V0_betU2;
  const double t152 = betU2*t50;
  const double t153 = t152*vetU0;
  const double t154 = betU1*t52;
  const double t155 = betU2*t49;
  const double t156 = t155*t43;
  const double t157 = t59*vetU2;
  const double t158 = betU2*t157;
  const double t159 = t123*t150;
  const double t160 = _GbUDD002*vetU0;
  const double lambdaU2 = V0_lambdaU2;
  const double t161 = (Rational_3_4)*lambdaU2;
  const double t162 = t161*t50;
  const double t163 = t148*t52;
  const double t164 = lambdaU2*t49;
  const double t165 = (Rational_3_4)*t164*t43;
  const double t166 = t157*t161;
  const double t90 = (Rational_1_2)*_Dbb;
  const double t91 = 6.0*alpha;
  const double t92 = -_phidD0*t91 + alpha_dD0;
  const double t93 = (Rational_3_2)*t92;
  const double t94 = -_phidD1*t91 + alpha_dD1;
  const double t95 = (Rational_3_2)*t94;
  const double t96 = lambdaU0*vetU_dD00;
  const double eta = p.eta;
  out[7 * Ntot + idx] = -_AbUU00*t93 - _AbUU01*t95 + _AbUU02*t130 + _AbUU12*t134 + _AbUU20*t130 + _AbUU21*t134 + _DGU0*t90 + _DGUDD011*t133 + _DGUDD022*t136 + _GbUDD000*t118 - _GbUDD000*t124 + _GbUDD000*t127 + _GbUDD001*t131 + _GbUDD001*t137 + _GbUDD001*t139 - _GbUDD001*t144 + _GbUDD002*t151 + _GbUDD002*t153 - _GbUDD002*t159 + _GbUDD011*t140 - _GbUDD011*t149 + _GbUDD012*t154 + _GbUDD012*t156 - _GbUDD012*t163 - _GbUDD012*t165 + _GbUDD022*t158 - _GbUDD022*t166 + _gbUU00*t105 + _gbUU01*t110 - betU0*eta + t113*t114 + (Rational_3_4)*t115 + (Rational_3_4)*t116 + (Rational_3_4)*t117 - t120 - t122 - Rational_3_4*t125 + t128*t129 - t141*t142 - Rational_3_2*t143*t40 - t145*t147 - t160*t162 - Rational_3_4*t96 + V0_lin_betU0;
  const double t42 = -t41;
  const double _DGUDD101 = _GbUDD101 + t42;
  const double _DGUDD122 = _GbUDD122 + t17;
  const double _DGU1 = _DGUDD101*t45 + _DGUDD122*_gbUU22 + _GbUDD100*_gbUU00 + _GbUDD102*t46 + _GbUDD111*_gbUU11 + _GbUDD112*t47;
  const double t167 = _bUdD10*lambdaU0;
  const double t168 = t41*vetU_dD00 - t97;
  const double t169 = _bUdDD101 + t168;
  const double t57 = 2.0/t56;
  const double vetU_dDD100 = V0_vetU_dDD100;
  const double _bUdDD100 = t41*vetU_dDD100 - 2.0*t48*vetU_dD10 + t57*vetU1;
  const double t170 = _gbUU00*(_bUdD10*t65 + _bUdDD100);
  const double t171 = _gbUU11*(_bUdDD111 + t111 + 2.0*t112);
  const double t172 = _bUdD21*t17;
  const double t173 = t41*vetU2;
  const double t174 = _gbUU12*(-f1_of_xx1*t173 - t172 + t41*t43*t62*vetU2 + t41*t43*vetU2*(-t106 - t62));
  const double t175 = _gbUU22*(_bUdD10*t40 + _bUdD11*t17 + t3*t66 - t62*t66);
  const double t176 = _gbUU01*t119;
  const double t177 = _gbUU11*t121;
  const double t178 = _bUdD11*t146;
  const double t179 = _AbUU01*t128;
  const double t180 = _GbUDD102*t128;
  const double t181 = _GbUDD112*t128;
  const double t182 = _bUdD20*t17;
  const double t183 = t147*vetU0;
  const double t184 = _gbUU12*t172;
  const double t185 = t162*vetU0;
  out[8 * Ntot + idx] = f0_of_xx0*(_AbUU02*t180 - _AbUU10*t93 - _AbUU11*t95 + _AbUU12*t181 + _AbUU20*t180 + _AbUU21*t181 + _DGU1*t90 + _DGUDD101*t131 + _DGUDD101*t179 + _DGUDD122*t136 + _GbUDD100*t118 - _GbUDD100*t124 + _GbUDD100*t127 + _GbUDD101*t137 + _GbUDD101*t139 - _GbUDD101*t144 - _GbUDD101*t183 + _GbUDD102*t151 + _GbUDD102*t153 - _GbUDD102*t159 - _GbUDD102*t185 + _GbUDD111*t133 + _GbUDD111*t140 - _GbUDD111*t149 + _GbUDD112*t154 + _GbUDD112*t156 - _GbUDD112*t163 - _GbUDD112*t165 + _GbUDD122*t158 - _GbUDD122*t166 + _gbUU01*t105 + _gbUU11*t110 - betU1*t97 - eta*t138 + t114*t169 - t141*t182 - Rational_3_4*t167 + (Rational_3_4)*t170 + (Rational_3_4)*t171 + (Rational_3_4)*t174 + (Rational_3_4)*t175 - t176 - t177 - Rational_3_4*t178 - Rational_3_4*t184) + V0_lin_betU1;
  const double t33 = (Rational_1_2)*_gbUU22;
  const double _GbUDD202 = _gbDDdD220*t33 + t28*t31;
  const double _DGUDD202 = _GbUDD202 + t42;
  const double _GbUDD212 = _gbDDdD221*t33 + t25*t27;
  const double _DGUDD212 = _GbUDD212 - t44;
  const double _GbUDD200 = _gbDDdD020*_gbUU22 + hDD_dD000*t25 + t22*t31;
  const double _GbUDD201 = _gbDDdD110*t31 + hDD_dD001*t25 + t24*t33;
  const double _GbUDD211 = _gbDDdD111*t31 + _gbDDdD121*_gbUU22 + t25*t29;
  const double _GbUDD222 = -t26 - t32;
  const double _DGU2 = _DGUDD202*t46 + _DGUDD212*t47 + _GbUDD200*_gbUU00 + _GbUDD201*t45 + _GbUDD211*_gbUU11 + _GbUDD222*_gbUU22;
  const double t186 = _bUdD20*lambdaU0;
  const double t60 = f1_of_xx1__D1*t54;
  const double vetU_dDD201 = V0_vetU_dDD201;
  const double _bUdDD201 = t50*vetU_dDD201 - t51*vetU_dD21 + t55*t59 - t60*vetU_dD20;
  const double t187 = _bUdD20*t44 + _bUdDD201;
  const double t188 = _bUdD10*t44 + t168;
  const double t58 = t43*vetU2;
  const double vetU_dDD200 = V0_vetU_dDD200;
  const double _bUdDD200 = t50*vetU_dDD200 - 2.0*t51*vetU_dD20 + t57*t58;
  const double t189 = _gbUU00*(_bUdD20*t65 + _bUdDD200);
  const double t61 = (1.0 / (f1_of_xx1*f1_of_xx1*f1_of_xx1));
  const double vetU_dDD211 = V0_vetU_dDD211;
  const double _bUdDD211 = t50*vetU_dDD211 - 2.0*t60*vetU_dD21 + vetU2*(-f1_of_xx1__DD11*t54 + 2.0*t41*t61*t62);
  const double t190 = f1_of_xx1__DD11*t43 - t107;
  const double t191 = _gbUU11*(_bUdD20*f0_of_xx0 + _bUdDD211 + t150*t190 + t150 + t173*t61*t62 + t44*t86);
  const double t192 = _bUdD11*t44 + t112;
  const double t193 = _gbUU12*(t190*t66 + t192);
  const double t194 = _gbUU12*(-t108 + t192 - t66);
  const double t195 = _gbUU22*(t142 + t172);
  const double t196 = _gbUU02*t119;
  const double t197 = _gbUU12*t121;
  const double t198 = _bUdD21*t146;
  const double t199 = _DGUDD202*t128;
  const double t200 = _DGUDD212*t128;
  const double t201 = t43*t97;
  const double t202 = f1_of_xx1__D1*t53;
  out[9 * Ntot + idx] = t5*(_AbUU02*t199 + _AbUU12*t200 + _AbUU20*t199 - _AbUU20*t93 + _AbUU21*t200 - _AbUU21*t95 + _DGU2*t90 + _GbUDD200*t118 - _GbUDD200*t124 + _GbUDD200*t127 + _GbUDD201*t131 + _GbUDD201*t137 + _GbUDD201*t139 - _GbUDD201*t144 + _GbUDD201*t179 - _GbUDD201*t183 + _GbUDD202*t151 + _GbUDD202*t153 - _GbUDD202*t159 - _GbUDD202*t185 + _GbUDD211*t133 + _GbUDD211*t140 - _GbUDD211*t149 + _GbUDD212*t154 + _GbUDD212*t156 - _GbUDD212*t163 - _GbUDD212*t165 + _GbUDD222*t136 + _GbUDD222*t158 - _GbUDD222*t166 + _gbUU02*t105 + _gbUU12*t110 - betU2*t201 - eta*t152 + t114*t187 + t141*t188 - t155*t202 - Rational_3_4*t186 + (Rational_3_4)*t189 + (Rational_3_4)*t191 + (Rational_3_4)*t193 + (Rational_3_4)*t194 + (Rational_3_4)*t195 - t196 - t197 - Rational_3_4*t198) + V0_lin_betU2;
  out[10 * Ntot + idx] = -2.0*cf*((Rational_1_6)*_Dbb - Rational_1_6*t79) + V0_lin_cf;
  const double t203 = 2.0*_gbDD01;
  const double _trAb = 2.0*t34 + 2.0*t35 + t36 + t37 + 2.0*t38 + t39;
  const double t204 = -Rational_2_3*_Dbb + (Rational_2_3)*_trAb*alpha;
  out[11 * Ntot + idx] = _bUdD10*t203 + _gbDD00*t204 + _gbDD00*t77 + _gbDD02*t76 - t82 + V0_lin_hDD00;
  out[12 * Ntot + idx] = t41*(_bUdD10*_gbDD11 + _bUdD11*_gbDD01 + _bUdD20*_gbDD12 + _bUdD21*_gbDD02 + _gbDD00*vetU_dD01 + _gbDD01*t204 + _gbDD01*vetU_dD00 + hDD01*vetU0 - t80) + V0_lin_hDD01;
  out[13 * Ntot + idx] = t50*(_bUdD10*_gbDD12 + _bUdD20*_gbDD22 + _gbDD02*t204 + _gbDD02*vetU_dD00 + t0*vetU0 + t10*vetU1 - t81) + V0_lin_hDD02;
  out[14 * Ntot + idx] = t48*(_gbDD11*t204 + _gbDD11*t85 + _gbDD12*t86 + t12*vetU0 + t203*vetU_dD01 - t87) + V0_lin_hDD11;
  out[15 * Ntot + idx] = t51*(_bUdD11*_gbDD12 + _bUdD21*_gbDD22 + _gbDD02*vetU_dD01 + _gbDD12*t204 + f0_of_xx0*t14*vetU1 + t13*t83 - t88) + V0_lin_hDD12;
  out[16 * Ntot + idx] = t59*(_gbDD22*t204 + t16*vetU0 + t20*t66 - t89) + V0_lin_hDD22;
  const double t205 = 2.0*t92;
  const double t206 = 2.0*t94;
  const double t207 = (Rational_1_3)*t104;
  const double t208 = (Rational_1_3)*t109;
  const double t209 = _AbUU00*t67;
  const double t210 = _GbUDD002*t67;
  const double t211 = _AbUU10*t67;
  const double t212 = _AbUU11*t67;
  const double t213 = _GbUDD012*t67;
  const double t214 = _AbUU22*t67;
  out[17 * Ntot + idx] = -_AbUU00*t205 - _AbUU01*t206 + _AbUU02*t210 + _AbUU12*t213 + _AbUU20*t210 + _AbUU21*t213 + _DGU0*t78 + _DGUDD011*t212 + _DGUDD022*t214 + _GbUDD000*t209 + _GbUDD001*t211 - _bUdD20*_gbUU02*t15 + _gbUU00*t207 + _gbUU01*t208 + t113*t45 + t115 + t116 + t117 - Rational_4_3*t120 - Rational_4_3*t122 - t125 + t129*t67 - t143*t15 - t96 + V0_lin_lambdaU0;
  const double t215 = _AbUU01*t67;
  const double t216 = _GbUDD102*t67;
  const double t217 = _GbUDD112*t67;
  out[18 * Ntot + idx] = f0_of_xx0*(_AbUU02*t216 - _AbUU10*t205 - _AbUU11*t206 + _AbUU12*t217 + _AbUU20*t216 + _AbUU21*t217 + _DGU1*t78 + _DGUDD101*t211 + _DGUDD101*t215 + _DGUDD122*t214 + _GbUDD100*t209 + _GbUDD111*t212 + _gbUU01*t207 + _gbUU11*t208 - lambdaU1*t97 - t167 + t169*t45 + t170 + t171 + t174 + t175 - Rational_4_3*t176 - Rational_4_3*t177 - t178 - t182*t46 - t184) + V0_lin_lambdaU1;
  const double t218 = _DGUDD202*t67;
  const double t219 = _DGUDD212*t67;
  out[19 * Ntot + idx] = t5*(_AbUU02*t218 + _AbUU12*t219 - _AbUU20*t205 + _AbUU20*t218 - _AbUU21*t206 + _AbUU21*t219 + _DGU2*t78 + _GbUDD200*t209 + _GbUDD201*t211 + _GbUDD201*t215 + _GbUDD211*t212 + _GbUDD222*t214 + _gbUU02*t207 + _gbUU12*t208 - lambdaU2*t201 - t164*t202 - t186 + t187*t45 + t188*t46 + t189 + t191 + t193 + t194 + t195 - Rational_4_3*t196 - Rational_4_3*t197 - t198) + V0_lin_lambdaU2;
  const double t220 = _AbDD01*alpha;
  const double t221 = _AbDD02*alpha;
  const double t222 = _AbDD12*alpha;
  const double t223 = _gbUU01*t73;
  out[20 * Ntot + idx] = _AbDD11*t132 + _AbDD22*t135 + _AbUU01*t220 + _AbUU02*t221 + _AbUU10*t220 + _AbUU12*t222 + _AbUU20*t221 + _AbUU21*t222 - _adBDD02*t46*t73 - _adBDD12*t47*t73 - _adBDD22*_gbUU22*t73 - _gbUU00*t73*(_adBDD00 + 2.0*t68) - _gbUU11*t73*(_adBDD11 + _phidD1*t70) + aDD00*t126 + (Rational_1_3)*alpha*(trK*trK) - t223*(_adBDD01 + t71) - t223*(_adBDD01 + t72) + V0_lin_trK;
  const double t224 = (vetU0*vetU0);
  const double t225 = t48*(vetU1*vetU1);
  const double t226 = t59*(vetU2*vetU2);
  const double t227 = 2.0*t66;
  const double t228 = 2.0*t150;
  const double t229 = 2.0*t49*t58;
  out[21 * Ntot + idx] = _GbUDD000*t224 + _GbUDD011*t225 + _GbUDD012*t229 + _GbUDD022*t226 + betU0 + t145*t227 + t160*t228 + V0_lin_vetU0;
  const double t230 = t227*vetU0;
  const double t231 = t228*vetU0;
  out[22 * Ntot + idx] = f0_of_xx0*(_GbUDD100*t224 + _GbUDD101*t230 + _GbUDD102*t231 + _GbUDD111*t225 + _GbUDD112*t229 + _GbUDD122*t226 + t138 - t49*vetU0) + V0_lin_vetU1;
  out[23 * Ntot + idx] = t5*(_GbUDD200*t224 + _GbUDD201*t230 + _GbUDD202*t231 + _GbUDD211*t225 + _GbUDD212*t229 + _GbUDD222*t226 + t152 - t49*t53*t55 - t58*t97) + V0_lin_vetU2;
    }
  }
}
extern "C" __global__ void __launch_bounds__(256)
bssn_ens_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0(const bhah_member *__restrict__ mem, const bhah_item *__restrict__ items, const int nitems,
        const int in_sel, const int aux_sel, const int out_sel) {
  __shared__ double sh[3072];
  for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
    const bhah_item w = items[it];
    const bhah_member *M = &mem[w.m];
    BHAH_BARRIER();
    bssn_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0_tile(M->arr[in_sel], M->arr[aux_sel], M->arr[out_sel], M->rfm0, M->rfm1, M->kp, (unsigned)w.bx,
                 (unsigned)w.by, (unsigned)w.bz, sh);
  }
}
#undef Rational_1_2
#undef Rational_1_3
#undef Rational_1_4
#undef Rational_1_6
#undef Rational_2_3
#undef Rational_3_2
#undef Rational_3_4
#undef Rational_4_3

extern "C" hipError_t launch_bssn_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub(dim3 g, dim3 b, hipStream_t s, const double *in, const double *aux, double *out, const double *rfm0, const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0, dim3((p.Nx0 - 2 * p.NG + 15) / 16, (p.Nx1 - 2 * p.NG + 7) / 8, (p.Nx2 - 2 * p.NG + 1) / 2), dim3(256), 0, s, in, aux, out, rfm0, rfm1, p);
  return hipGetLastError();
}

extern "C" hipError_t launch_bssn_ens_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub(dim3 g, dim3 b, hipStream_t s, const bhah_member *mem, const bhah_item *items, int nitems, int in_sel, int aux_sel, int out_sel) {
  hipLaunchKernelGGL(bssn_ens_rhs_Spherical_sym2_KO0_fd4_p1_lb1_sj_L16x8x2x1_d3_dma_rb1_pg8_ub_g0, g, dim3(256), 0, s, mem, items, nitems, in_sel, aux_sel, out_sel);
  return hipGetLastError();
}
