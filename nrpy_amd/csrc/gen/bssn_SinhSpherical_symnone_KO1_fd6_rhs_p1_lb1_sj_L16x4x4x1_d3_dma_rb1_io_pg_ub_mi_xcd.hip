// Generated by nrpy_amd/codegen/hip_gen.py -- do not edit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "../bhah_device_types.h"
// ---- rhs candidate p1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg_ub_mi_xcd: 1 kernel(s); SinhSpherical, fd_order=6
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

// bhah-dma-issue bssn_rhs_SinhSpherical_symnone_KO1_fd6_p1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg_ub_mi_xcd_g0: 0:7 1:7 2:7 3:7 4:7 5:7 6:7 7:7 8:7 9:7 10:7 11:7 12:7 13:7 14:7 15:7 16:7 17:7 18:7 19:7 20:7 21:7 22:7 23:7
extern "C" __global__ void __launch_bounds__(256)
bssn_rhs_SinhSpherical_symnone_KO1_fd6_p1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg_ub_mi_xcd_g0(const double *__restrict__ in, const double *__restrict__ aux, double *__restrict__ out,
        const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  __shared__ double sh[10752];
  unsigned bx, by, bz;
  {
    const unsigned gx = gridDim.x, gy = gridDim.y, gz = gridDim.z, n = gx * gy * gz;
    const unsigned h = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const unsigned l = (h & 7u) * (n >> 3) + min((int)(h & 7u), (int)(n & 7u)) + (h >> 3);
    bx = l % gx;
    by = (l / gx) % gy;
    bz = l / (gx * gy);
  }
  // Tile of 16x4x4 interior points; halo box 24x12x12 = 3456 values per gridfunction.
  constexpr int BX = 24, BY = 12, NB = 3456, NT = 256, NL = 14;
  const int tid = (int)threadIdx.x;
  const int lx = tid % 16, ly = (tid / 16) % 4, lz = tid / 64;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const int o0 = p.NG + (int)bx * 16, o1 = p.NG + (int)by * 4, o2 = p.NG + (int)bz * 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned pofs[7];
#pragma unroll
  for (int j = 0; j < 7; j++) {
    const int e = 2 * (tid + NT * j);
    const int ex = e % BX, ey = (e / BX) % BY, ez = e / (BX * BY);
    const int g0 = min(o0 - 4 + ex, p.Nx0 - 2), g1 = min(o1 - 4 + ey, p.Nx1 - 1), g2 = min(o2 - 4 + ez, p.Nx2 - 1);
    pofs[j] = 8u * (unsigned)(g0 + (int)s1 * g1 + (int)s2 * g2);
  }
  const int c0 = (lx + 4) + BX * (ly + 4) + BX * BY * (lz + 4);
  const double ius0 = p.invdxx0 * (1.0 / 60.0), nius0 = -ius0, ikos0 = p.invdxx0 * (1.0 / 256.0);
  const double ius1 = p.invdxx1 * (1.0 / 60.0), nius1 = -ius1, ikos1 = p.invdxx1 * (1.0 / 256.0);
  const double ius2 = p.invdxx2 * (1.0 / 60.0), nius2 = -ius2, ikos2 = p.invdxx2 * (1.0 / 256.0);
  double L0_coef[9], L0_beta[3];
  {
    const int i0 = min(o0 + lx, p.Nx0 - p.NG - 1), i1 = min(o1 + ly, p.Nx1 - p.NG - 1);
    const long idx = i0 + s1 * i1 + s2 * min(o2 + lz + 0, p.Nx2 - p.NG - 1);
    const double KreissOliger_strength_gauge = p.KO_gauge;
    const double KreissOliger_strength_nongauge = p.KO_nongauge;
    const double f0_of_xx0 = rfm0[i0];
    const double f0_of_xx0__D0 = rfm0[p.Nx0 + i0];
    const double f1_of_xx1 = rfm1[i1];
    const double vetU0 = in[21 * Ntot + idx];
    const double vetU1 = in[22 * Ntot + idx];
    const double vetU2 = in[23 * Ntot + idx];
    const double lc0 = (1.0 / f0_of_xx0);
    const double lc1 = KreissOliger_strength_gauge*lc0;
    const double lc2 = (1.0 / f0_of_xx0__D0);
    const double lc3 = KreissOliger_strength_nongauge*lc0;
    const double lc4 = (1.0 / f1_of_xx1);
    L0_coef[0] = lc1;
    L0_coef[1] = KreissOliger_strength_gauge*lc2;
    L0_coef[2] = lc3;
    L0_coef[3] = KreissOliger_strength_nongauge*lc2;
    L0_coef[4] = lc0*vetU1;
    L0_coef[5] = lc2*vetU0;
    L0_coef[6] = lc1*lc4;
    L0_coef[7] = lc3*lc4;
    L0_coef[8] = lc0*lc4*vetU2;
    L0_beta[0] = vetU0/f0_of_xx0__D0;
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
    const char *src = (const char *)(in + 6 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  {
    const char *src = (const char *)(in + 0 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  // ---- alpha
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(0);
  {
    const char *src = (const char *)(in + 1 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_alpha = sh[c0];
  double V0_alpha_dD0 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-3.0 / 20.0) * (sh[c0 + 2] - sh[c0 - 2]) + (1.0 / 60.0) * (sh[c0 + 3] - sh[c0 - 3]));
  double V0_alpha_dD1 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 24] - sh[c0 - 24]) + (-3.0 / 20.0) * (sh[c0 + 48] - sh[c0 - 48]) + (1.0 / 60.0) * (sh[c0 + 72] - sh[c0 - 72]));
  double V0_alpha_dD2 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 288] - sh[c0 - 288]) + (-3.0 / 20.0) * (sh[c0 + 576] - sh[c0 - 576]) + (1.0 / 60.0) * (sh[c0 + 864] - sh[c0 - 864]));
  double V0_alpha_dDD00 = p.invdxx0 * p.invdxx0 * ((-49.0 / 18.0) * sh[c0] + (3.0 / 2.0) * (sh[c0 + 1] + sh[c0 - 1]) + (-3.0 / 20.0) * (sh[c0 + 2] + sh[c0 - 2]) + (1.0 / 90.0) * (sh[c0 + 3] + sh[c0 - 3]));
  double V0_alpha_dDD01 = p.invdxx0 * p.invdxx1 * ((9.0 / 16.0) * ((sh[c0 + 25] - sh[c0 - 23]) - (sh[c0 + 23] - sh[c0 - 25])) + (-9.0 / 80.0) * ((sh[c0 + 49] - sh[c0 - 47]) - (sh[c0 + 47] - sh[c0 - 49])) + (1.0 / 80.0) * ((sh[c0 + 73] - sh[c0 - 71]) - (sh[c0 + 71] - sh[c0 - 73])) + (-9.0 / 80.0) * ((sh[c0 + 26] - sh[c0 - 22]) - (sh[c0 + 22] - sh[c0 - 26])) + (9.0 / 400.0) * ((sh[c0 + 50] - sh[c0 - 46]) - (sh[c0 + 46] - sh[c0 - 50])) + (-1.0 / 400.0) * ((sh[c0 + 74] - sh[c0 - 70]) - (sh[c0 + 70] - sh[c0 - 74])) + (1.0 / 80.0) * ((sh[c0 + 27] - sh[c0 - 21]) - (sh[c0 + 21] - sh[c0 - 27])) + (-1.0 / 400.0) * ((sh[c0 + 51] - sh[c0 - 45]) - (sh[c0 + 45] - sh[c0 - 51])) + (1.0 / 3600.0) * ((sh[c0 + 75] - sh[c0 - 69]) - (sh[c0 + 69] - sh[c0 - 75])));
  double V0_alpha_dDD02 = p.invdxx0 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 289] - sh[c0 - 287]) - (sh[c0 + 287] - sh[c0 - 289])) + (-9.0 / 80.0) * ((sh[c0 + 577] - sh[c0 - 575]) - (sh[c0 + 575] - sh[c0 - 577])) + (1.0 / 80.0) * ((sh[c0 + 865] - sh[c0 - 863]) - (sh[c0 + 863] - sh[c0 - 865])) + (-9.0 / 80.0) * ((sh[c0 + 290] - sh[c0 - 286]) - (sh[c0 + 286] - sh[c0 - 290])) + (9.0 / 400.0) * ((sh[c0 + 578] - sh[c0 - 574]) - (sh[c0 + 574] - sh[c0 - 578])) + (-1.0 / 400.0) * ((sh[c0 + 866] - sh[c0 - 862]) - (sh[c0 + 862] - sh[c0 - 866])) + (1.0 / 80.0) * ((sh[c0 + 291] - sh[c0 - 285]) - (sh[c0 + 285] - sh[c0 - 291])) + (-1.0 / 400.0) * ((sh[c0 + 579] - sh[c0 - 573]) - (sh[c0 + 573] - sh[c0 - 579])) + (1.0 / 3600.0) * ((sh[c0 + 867] - sh[c0 - 861]) - (sh[c0 + 861] - sh[c0 - 867])));
  double V0_alpha_dDD11 = p.invdxx1 * p.invdxx1 * ((-49.0 / 18.0) * sh[c0] + (3.0 / 2.0) * (sh[c0 + 24] + sh[c0 - 24]) + (-3.0 / 20.0) * (sh[c0 + 48] + sh[c0 - 48]) + (1.0 / 90.0) * (sh[c0 + 72] + sh[c0 - 72]));
  double V0_alpha_dDD12 = p.invdxx1 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 312] - sh[c0 - 264]) - (sh[c0 + 264] - sh[c0 - 312])) + (-9.0 / 80.0) * ((sh[c0 + 600] - sh[c0 - 552]) - (sh[c0 + 552] - sh[c0 - 600])) + (1.0 / 80.0) * ((sh[c0 + 888] - sh[c0 - 840]) - (sh[c0 + 840] - sh[c0 - 888])) + (-9.0 / 80.0) * ((sh[c0 + 336] - sh[c0 - 240]) - (sh[c0 + 240] - sh[c0 - 336])) + (9.0 / 400.0) * ((sh[c0 + 624] - sh[c0 - 528]) - (sh[c0 + 528] - sh[c0 - 624])) + (-1.0 / 400.0) * ((sh[c0 + 912] - sh[c0 - 816]) - (sh[c0 + 816] - sh[c0 - 912])) + (1.0 / 80.0) * ((sh[c0 + 360] - sh[c0 - 216]) - (sh[c0 + 216] - sh[c0 - 360])) + (-1.0 / 400.0) * ((sh[c0 + 648] - sh[c0 - 504]) - (sh[c0 + 504] - sh[c0 - 648])) + (1.0 / 3600.0) * ((sh[c0 + 936] - sh[c0 - 792]) - (sh[c0 + 792] - sh[c0 - 936])));
  double V0_alpha_dDD22 = p.invdxx2 * p.invdxx2 * ((-49.0 / 18.0) * sh[c0] + (3.0 / 2.0) * (sh[c0 + 288] + sh[c0 - 288]) + (-3.0 / 20.0) * (sh[c0 + 576] + sh[c0 - 576]) + (1.0 / 90.0) * (sh[c0 + 864] + sh[c0 - 864]));
  const double U0_alpha_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_alpha_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_alpha += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_alpha_0 : D0_alpha_0) + L0_coef[1] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_alpha_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_alpha_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_alpha += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_alpha_1 : D0_alpha_1) + L0_coef[0] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_alpha_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_alpha_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_alpha += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_alpha_2 : D0_alpha_2) + L0_coef[6] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_alpha), "+v"(V0_alpha_dD0), "+v"(V0_alpha_dD1), "+v"(V0_alpha_dD2), "+v"(V0_alpha_dDD00), "+v"(V0_alpha_dDD01), "+v"(V0_alpha_dDD02), "+v"(V0_alpha_dDD11), "+v"(V0_alpha_dDD12), "+v"(V0_alpha_dDD22), "+v"(V0_lin_alpha));
  // ---- aDD00
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(1);
  {
    const char *src = (const char *)(in + 2 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD00 = sh[c0 + 3584];
  const double U0_aDD00_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_aDD00_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_aDD00 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_aDD00_0 : D0_aDD00_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_aDD00_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_aDD00_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_aDD00 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_aDD00_1 : D0_aDD00_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_aDD00_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_aDD00_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_aDD00 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_aDD00_2 : D0_aDD00_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_aDD00), "+v"(V0_lin_aDD00));
  // ---- aDD01
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(2);
  {
    const char *src = (const char *)(in + 10 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD01 = sh[c0 + 7168];
  const double U0_aDD01_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_aDD01_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_aDD01 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_aDD01_0 : D0_aDD01_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_aDD01_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_aDD01_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_aDD01 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_aDD01_1 : D0_aDD01_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_aDD01_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_aDD01_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_aDD01 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_aDD01_2 : D0_aDD01_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_aDD01), "+v"(V0_lin_aDD01));
  // ---- aDD02
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(3);
  {
    const char *src = (const char *)(in + 3 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD02 = sh[c0];
  const double U0_aDD02_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_aDD02_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_aDD02 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_aDD02_0 : D0_aDD02_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_aDD02_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_aDD02_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_aDD02 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_aDD02_1 : D0_aDD02_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_aDD02_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_aDD02_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_aDD02 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_aDD02_2 : D0_aDD02_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_aDD02), "+v"(V0_lin_aDD02));
  // ---- cf
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(4);
  {
    const char *src = (const char *)(in + 4 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_cf = sh[c0 + 3584];
  double V0_cf_dD0 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 3585] - sh[c0 + 3583]) + (-3.0 / 20.0) * (sh[c0 + 3586] - sh[c0 + 3582]) + (1.0 / 60.0) * (sh[c0 + 3587] - sh[c0 + 3581]));
  double V0_cf_dD1 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 3608] - sh[c0 + 3560]) + (-3.0 / 20.0) * (sh[c0 + 3632] - sh[c0 + 3536]) + (1.0 / 60.0) * (sh[c0 + 3656] - sh[c0 + 3512]));
  double V0_cf_dD2 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 3872] - sh[c0 + 3296]) + (-3.0 / 20.0) * (sh[c0 + 4160] - sh[c0 + 3008]) + (1.0 / 60.0) * (sh[c0 + 4448] - sh[c0 + 2720]));
  double V0_cf_dDD00 = p.invdxx0 * p.invdxx0 * ((-49.0 / 18.0) * sh[c0 + 3584] + (3.0 / 2.0) * (sh[c0 + 3585] + sh[c0 + 3583]) + (-3.0 / 20.0) * (sh[c0 + 3586] + sh[c0 + 3582]) + (1.0 / 90.0) * (sh[c0 + 3587] + sh[c0 + 3581]));
  double V0_cf_dDD01 = p.invdxx0 * p.invdxx1 * ((9.0 / 16.0) * ((sh[c0 + 3609] - sh[c0 + 3561]) - (sh[c0 + 3607] - sh[c0 + 3559])) + (-9.0 / 80.0) * ((sh[c0 + 3633] - sh[c0 + 3537]) - (sh[c0 + 3631] - sh[c0 + 3535])) + (1.0 / 80.0) * ((sh[c0 + 3657] - sh[c0 + 3513]) - (sh[c0 + 3655] - sh[c0 + 3511])) + (-9.0 / 80.0) * ((sh[c0 + 3610] - sh[c0 + 3562]) - (sh[c0 + 3606] - sh[c0 + 3558])) + (9.0 / 400.0) * ((sh[c0 + 3634] - sh[c0 + 3538]) - (sh[c0 + 3630] - sh[c0 + 3534])) + (-1.0 / 400.0) * ((sh[c0 + 3658] - sh[c0 + 3514]) - (sh[c0 + 3654] - sh[c0 + 3510])) + (1.0 / 80.0) * ((sh[c0 + 3611] - sh[c0 + 3563]) - (sh[c0 + 3605] - sh[c0 + 3557])) + (-1.0 / 400.0) * ((sh[c0 + 3635] - sh[c0 + 3539]) - (sh[c0 + 3629] - sh[c0 + 3533])) + (1.0 / 3600.0) * ((sh[c0 + 3659] - sh[c0 + 3515]) - (sh[c0 + 3653] - sh[c0 + 3509])));
  double V0_cf_dDD02 = p.invdxx0 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 3873] - sh[c0 + 3297]) - (sh[c0 + 3871] - sh[c0 + 3295])) + (-9.0 / 80.0) * ((sh[c0 + 4161] - sh[c0 + 3009]) - (sh[c0 + 4159] - sh[c0 + 3007])) + (1.0 / 80.0) * ((sh[c0 + 4449] - sh[c0 + 2721]) - (sh[c0 + 4447] - sh[c0 + 2719])) + (-9.0 / 80.0) * ((sh[c0 + 3874] - sh[c0 + 3298]) - (sh[c0 + 3870] - sh[c0 + 3294])) + (9.0 / 400.0) * ((sh[c0 + 4162] - sh[c0 + 3010]) - (sh[c0 + 4158] - sh[c0 + 3006])) + (-1.0 / 400.0) * ((sh[c0 + 4450] - sh[c0 + 2722]) - (sh[c0 + 4446] - sh[c0 + 2718])) + (1.0 / 80.0) * ((sh[c0 + 3875] - sh[c0 + 3299]) - (sh[c0 + 3869] - sh[c0 + 3293])) + (-1.0 / 400.0) * ((sh[c0 + 4163] - sh[c0 + 3011]) - (sh[c0 + 4157] - sh[c0 + 3005])) + (1.0 / 3600.0) * ((sh[c0 + 4451] - sh[c0 + 2723]) - (sh[c0 + 4445] - sh[c0 + 2717])));
  double V0_cf_dDD11 = p.invdxx1 * p.invdxx1 * ((-49.0 / 18.0) * sh[c0 + 3584] + (3.0 / 2.0) * (sh[c0 + 3608] + sh[c0 + 3560]) + (-3.0 / 20.0) * (sh[c0 + 3632] + sh[c0 + 3536]) + (1.0 / 90.0) * (sh[c0 + 3656] + sh[c0 + 3512]));
  double V0_cf_dDD12 = p.invdxx1 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 3896] - sh[c0 + 3320]) - (sh[c0 + 3848] - sh[c0 + 3272])) + (-9.0 / 80.0) * ((sh[c0 + 4184] - sh[c0 + 3032]) - (sh[c0 + 4136] - sh[c0 + 2984])) + (1.0 / 80.0) * ((sh[c0 + 4472] - sh[c0 + 2744]) - (sh[c0 + 4424] - sh[c0 + 2696])) + (-9.0 / 80.0) * ((sh[c0 + 3920] - sh[c0 + 3344]) - (sh[c0 + 3824] - sh[c0 + 3248])) + (9.0 / 400.0) * ((sh[c0 + 4208] - sh[c0 + 3056]) - (sh[c0 + 4112] - sh[c0 + 2960])) + (-1.0 / 400.0) * ((sh[c0 + 4496] - sh[c0 + 2768]) - (sh[c0 + 4400] - sh[c0 + 2672])) + (1.0 / 80.0) * ((sh[c0 + 3944] - sh[c0 + 3368]) - (sh[c0 + 3800] - sh[c0 + 3224])) + (-1.0 / 400.0) * ((sh[c0 + 4232] - sh[c0 + 3080]) - (sh[c0 + 4088] - sh[c0 + 2936])) + (1.0 / 3600.0) * ((sh[c0 + 4520] - sh[c0 + 2792]) - (sh[c0 + 4376] - sh[c0 + 2648])));
  double V0_cf_dDD22 = p.invdxx2 * p.invdxx2 * ((-49.0 / 18.0) * sh[c0 + 3584] + (3.0 / 2.0) * (sh[c0 + 3872] + sh[c0 + 3296]) + (-3.0 / 20.0) * (sh[c0 + 4160] + sh[c0 + 3008]) + (1.0 / 90.0) * (sh[c0 + 4448] + sh[c0 + 2720]));
  const double U0_cf_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_cf_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_cf += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_cf_0 : D0_cf_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_cf_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_cf_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_cf += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_cf_1 : D0_cf_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_cf_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_cf_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_cf += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_cf_2 : D0_cf_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_cf), "+v"(V0_cf_dD0), "+v"(V0_cf_dD1), "+v"(V0_cf_dD2), "+v"(V0_cf_dDD00), "+v"(V0_cf_dDD01), "+v"(V0_cf_dDD02), "+v"(V0_cf_dDD11), "+v"(V0_cf_dDD12), "+v"(V0_cf_dDD22), "+v"(V0_lin_cf));
  // ---- aDD11
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(5);
  {
    const char *src = (const char *)(in + 5 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD11 = sh[c0 + 7168];
  const double U0_aDD11_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_aDD11_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_aDD11 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_aDD11_0 : D0_aDD11_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_aDD11_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_aDD11_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_aDD11 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_aDD11_1 : D0_aDD11_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_aDD11_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_aDD11_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_aDD11 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_aDD11_2 : D0_aDD11_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_aDD11), "+v"(V0_lin_aDD11));
  // ---- aDD12
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(6);
  {
    const char *src = (const char *)(in + 7 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD12 = sh[c0];
  const double U0_aDD12_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_aDD12_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_aDD12 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_aDD12_0 : D0_aDD12_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_aDD12_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_aDD12_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_aDD12 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_aDD12_1 : D0_aDD12_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_aDD12_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_aDD12_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_aDD12 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_aDD12_2 : D0_aDD12_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_aDD12), "+v"(V0_lin_aDD12));
  // ---- aDD22
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(7);
  {
    const char *src = (const char *)(in + 21 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_aDD22 = sh[c0 + 3584];
  const double U0_aDD22_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_aDD22_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_aDD22 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_aDD22_0 : D0_aDD22_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_aDD22_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_aDD22_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_aDD22 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_aDD22_1 : D0_aDD22_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_aDD22_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_aDD22_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_aDD22 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_aDD22_2 : D0_aDD22_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_aDD22), "+v"(V0_lin_aDD22));
  // ---- betU0
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(8);
  {
    const char *src = (const char *)(in + 8 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU0 = sh[c0 + 7168];
  const double U0_betU0_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_betU0_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_betU0 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_betU0_0 : D0_betU0_0) + L0_coef[1] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_betU0_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_betU0_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_betU0 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_betU0_1 : D0_betU0_1) + L0_coef[0] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_betU0_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_betU0_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_betU0 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_betU0_2 : D0_betU0_2) + L0_coef[6] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_betU0), "+v"(V0_lin_betU0));
  // ---- vetU0
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(9);
  {
    const char *src = (const char *)(in + 9 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_vetU0 = sh[c0];
  double V0_vetU_dD00 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-3.0 / 20.0) * (sh[c0 + 2] - sh[c0 - 2]) + (1.0 / 60.0) * (sh[c0 + 3] - sh[c0 - 3]));
  double V0_vetU_dD01 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 24] - sh[c0 - 24]) + (-3.0 / 20.0) * (sh[c0 + 48] - sh[c0 - 48]) + (1.0 / 60.0) * (sh[c0 + 72] - sh[c0 - 72]));
  double V0_vetU_dD02 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 288] - sh[c0 - 288]) + (-3.0 / 20.0) * (sh[c0 + 576] - sh[c0 - 576]) + (1.0 / 60.0) * (sh[c0 + 864] - sh[c0 - 864]));
  double V0_vetU_dDD000 = p.invdxx0 * p.invdxx0 * ((-49.0 / 18.0) * sh[c0] + (3.0 / 2.0) * (sh[c0 + 1] + sh[c0 - 1]) + (-3.0 / 20.0) * (sh[c0 + 2] + sh[c0 - 2]) + (1.0 / 90.0) * (sh[c0 + 3] + sh[c0 - 3]));
  double V0_vetU_dDD001 = p.invdxx0 * p.invdxx1 * ((9.0 / 16.0) * ((sh[c0 + 25] - sh[c0 - 23]) - (sh[c0 + 23] - sh[c0 - 25])) + (-9.0 / 80.0) * ((sh[c0 + 49] - sh[c0 - 47]) - (sh[c0 + 47] - sh[c0 - 49])) + (1.0 / 80.0) * ((sh[c0 + 73] - sh[c0 - 71]) - (sh[c0 + 71] - sh[c0 - 73])) + (-9.0 / 80.0) * ((sh[c0 + 26] - sh[c0 - 22]) - (sh[c0 + 22] - sh[c0 - 26])) + (9.0 / 400.0) * ((sh[c0 + 50] - sh[c0 - 46]) - (sh[c0 + 46] - sh[c0 - 50])) + (-1.0 / 400.0) * ((sh[c0 + 74] - sh[c0 - 70]) - (sh[c0 + 70] - sh[c0 - 74])) + (1.0 / 80.0) * ((sh[c0 + 27] - sh[c0 - 21]) - (sh[c0 + 21] - sh[c0 - 27])) + (-1.0 / 400.0) * ((sh[c0 + 51] - sh[c0 - 45]) - (sh[c0 + 45] - sh[c0 - 51])) + (1.0 / 3600.0) * ((sh[c0 + 75] - sh[c0 - 69]) - (sh[c0 + 69] - sh[c0 - 75])));
  double V0_vetU_dDD002 = p.invdxx0 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 289] - sh[c0 - 287]) - (sh[c0 + 287] - sh[c0 - 289])) + (-9.0 / 80.0) * ((sh[c0 + 577] - sh[c0 - 575]) - (sh[c0 + 575] - sh[c0 - 577])) + (1.0 / 80.0) * ((sh[c0 + 865] - sh[c0 - 863]) - (sh[c0 + 863] - sh[c0 - 865])) + (-9.0 / 80.0) * ((sh[c0 + 290] - sh[c0 - 286]) - (sh[c0 + 286] - sh[c0 - 290])) + (9.0 / 400.0) * ((sh[c0 + 578] - sh[c0 - 574]) - (sh[c0 + 574] - sh[c0 - 578])) + (-1.0 / 400.0) * ((sh[c0 + 866] - sh[c0 - 862]) - (sh[c0 + 862] - sh[c0 - 866])) + (1.0 / 80.0) * ((sh[c0 + 291] - sh[c0 - 285]) - (sh[c0 + 285] - sh[c0 - 291])) + (-1.0 / 400.0) * ((sh[c0 + 579] - sh[c0 - 573]) - (sh[c0 + 573] - sh[c0 - 579])) + (1.0 / 3600.0) * ((sh[c0 + 867] - sh[c0 - 861]) - (sh[c0 + 861] - sh[c0 - 867])));
  double V0_vetU_dDD011 = p.invdxx1 * p.invdxx1 * ((-49.0 / 18.0) * sh[c0] + (3.0 / 2.0) * (sh[c0 + 24] + sh[c0 - 24]) + (-3.0 / 20.0) * (sh[c0 + 48] + sh[c0 - 48]) + (1.0 / 90.0) * (sh[c0 + 72] + sh[c0 - 72]));
  double V0_vetU_dDD012 = p.invdxx1 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 312] - sh[c0 - 264]) - (sh[c0 + 264] - sh[c0 - 312])) + (-9.0 / 80.0) * ((sh[c0 + 600] - sh[c0 - 552]) - (sh[c0 + 552] - sh[c0 - 600])) + (1.0 / 80.0) * ((sh[c0 + 888] - sh[c0 - 840]) - (sh[c0 + 840] - sh[c0 - 888])) + (-9.0 / 80.0) * ((sh[c0 + 336] - sh[c0 - 240]) - (sh[c0 + 240] - sh[c0 - 336])) + (9.0 / 400.0) * ((sh[c0 + 624] - sh[c0 - 528]) - (sh[c0 + 528] - sh[c0 - 624])) + (-1.0 / 400.0) * ((sh[c0 + 912] - sh[c0 - 816]) - (sh[c0 + 816] - sh[c0 - 912])) + (1.0 / 80.0) * ((sh[c0 + 360] - sh[c0 - 216]) - (sh[c0 + 216] - sh[c0 - 360])) + (-1.0 / 400.0) * ((sh[c0 + 648] - sh[c0 - 504]) - (sh[c0 + 504] - sh[c0 - 648])) + (1.0 / 3600.0) * ((sh[c0 + 936] - sh[c0 - 792]) - (sh[c0 + 792] - sh[c0 - 936])));
  double V0_vetU_dDD022 = p.invdxx2 * p.invdxx2 * ((-49.0 / 18.0) * sh[c0] + (3.0 / 2.0) * (sh[c0 + 288] + sh[c0 - 288]) + (-3.0 / 20.0) * (sh[c0 + 576] + sh[c0 - 576]) + (1.0 / 90.0) * (sh[c0 + 864] + sh[c0 - 864]));
  const double U0_vetU0_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_vetU0_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_vetU0 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_vetU0_0 : D0_vetU0_0) + L0_coef[1] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_vetU0_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_vetU0_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_vetU0 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_vetU0_1 : D0_vetU0_1) + L0_coef[0] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_vetU0_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_vetU0_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_vetU0 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_vetU0_2 : D0_vetU0_2) + L0_coef[6] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_vetU0), "+v"(V0_vetU_dD00), "+v"(V0_vetU_dD01), "+v"(V0_vetU_dD02), "+v"(V0_vetU_dDD000), "+v"(V0_vetU_dDD001), "+v"(V0_vetU_dDD002), "+v"(V0_vetU_dDD011), "+v"(V0_vetU_dDD012), "+v"(V0_vetU_dDD022), "+v"(V0_lin_vetU0));
  // ---- betU1
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(10);
  {
    const char *src = (const char *)(in + 11 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU1 = sh[c0 + 3584];
  const double U0_betU1_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_betU1_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_betU1 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_betU1_0 : D0_betU1_0) + L0_coef[1] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_betU1_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_betU1_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_betU1 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_betU1_1 : D0_betU1_1) + L0_coef[0] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_betU1_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_betU1_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_betU1 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_betU1_2 : D0_betU1_2) + L0_coef[6] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_betU1), "+v"(V0_lin_betU1));
  // ---- betU2
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(11);
  {
    const char *src = (const char *)(in + 12 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  double V0_betU2 = sh[c0 + 7168];
  const double U0_betU2_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_betU2_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_betU2 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_betU2_0 : D0_betU2_0) + L0_coef[1] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_betU2_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_betU2_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_betU2 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_betU2_1 : D0_betU2_1) + L0_coef[0] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_betU2_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_betU2_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_betU2 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_betU2_2 : D0_betU2_2) + L0_coef[6] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_betU2), "+v"(V0_lin_betU2));
  // ---- hDD00
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(12);
  {
    const char *src = (const char *)(in + 22 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD00 = sh[c0];
  double V0_hDD_dD000 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-3.0 / 20.0) * (sh[c0 + 2] - sh[c0 - 2]) + (1.0 / 60.0) * (sh[c0 + 3] - sh[c0 - 3]));
  double V0_hDD_dD001 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 24] - sh[c0 - 24]) + (-3.0 / 20.0) * (sh[c0 + 48] - sh[c0 - 48]) + (1.0 / 60.0) * (sh[c0 + 72] - sh[c0 - 72]));
  double V0_hDD_dD002 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 288] - sh[c0 - 288]) + (-3.0 / 20.0) * (sh[c0 + 576] - sh[c0 - 576]) + (1.0 / 60.0) * (sh[c0 + 864] - sh[c0 - 864]));
  const double U0_hDD00_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_hDD00_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_hDD00 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_hDD00_0 : D0_hDD00_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_hDD00_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_hDD00_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_hDD00 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_hDD00_1 : D0_hDD00_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_hDD00_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_hDD00_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_hDD00 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_hDD00_2 : D0_hDD00_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_hDD00), "+v"(V0_hDD_dD000), "+v"(V0_hDD_dD001), "+v"(V0_hDD_dD002), "+v"(V0_lin_hDD00));
  // ---- hDD01
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(13);
  {
    const char *src = (const char *)(in + 13 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD01 = sh[c0 + 3584];
  double V0_hDD_dD010 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 3585] - sh[c0 + 3583]) + (-3.0 / 20.0) * (sh[c0 + 3586] - sh[c0 + 3582]) + (1.0 / 60.0) * (sh[c0 + 3587] - sh[c0 + 3581]));
  double V0_hDD_dD011 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 3608] - sh[c0 + 3560]) + (-3.0 / 20.0) * (sh[c0 + 3632] - sh[c0 + 3536]) + (1.0 / 60.0) * (sh[c0 + 3656] - sh[c0 + 3512]));
  double V0_hDD_dD012 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 3872] - sh[c0 + 3296]) + (-3.0 / 20.0) * (sh[c0 + 4160] - sh[c0 + 3008]) + (1.0 / 60.0) * (sh[c0 + 4448] - sh[c0 + 2720]));
  const double U0_hDD01_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_hDD01_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_hDD01 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_hDD01_0 : D0_hDD01_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_hDD01_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_hDD01_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_hDD01 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_hDD01_1 : D0_hDD01_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_hDD01_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_hDD01_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_hDD01 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_hDD01_2 : D0_hDD01_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_hDD01), "+v"(V0_hDD_dD010), "+v"(V0_hDD_dD011), "+v"(V0_hDD_dD012), "+v"(V0_lin_hDD01));
  // ---- vetU1
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(14);
  {
    const char *src = (const char *)(in + 14 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  double V0_vetU1 = sh[c0 + 7168];
  double V0_vetU_dD10 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 7169] - sh[c0 + 7167]) + (-3.0 / 20.0) * (sh[c0 + 7170] - sh[c0 + 7166]) + (1.0 / 60.0) * (sh[c0 + 7171] - sh[c0 + 7165]));
  double V0_vetU_dD11 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 7192] - sh[c0 + 7144]) + (-3.0 / 20.0) * (sh[c0 + 7216] - sh[c0 + 7120]) + (1.0 / 60.0) * (sh[c0 + 7240] - sh[c0 + 7096]));
  double V0_vetU_dD12 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 7456] - sh[c0 + 6880]) + (-3.0 / 20.0) * (sh[c0 + 7744] - sh[c0 + 6592]) + (1.0 / 60.0) * (sh[c0 + 8032] - sh[c0 + 6304]));
  double V0_vetU_dDD100 = p.invdxx0 * p.invdxx0 * ((-49.0 / 18.0) * sh[c0 + 7168] + (3.0 / 2.0) * (sh[c0 + 7169] + sh[c0 + 7167]) + (-3.0 / 20.0) * (sh[c0 + 7170] + sh[c0 + 7166]) + (1.0 / 90.0) * (sh[c0 + 7171] + sh[c0 + 7165]));
  double V0_vetU_dDD101 = p.invdxx0 * p.invdxx1 * ((9.0 / 16.0) * ((sh[c0 + 7193] - sh[c0 + 7145]) - (sh[c0 + 7191] - sh[c0 + 7143])) + (-9.0 / 80.0) * ((sh[c0 + 7217] - sh[c0 + 7121]) - (sh[c0 + 7215] - sh[c0 + 7119])) + (1.0 / 80.0) * ((sh[c0 + 7241] - sh[c0 + 7097]) - (sh[c0 + 7239] - sh[c0 + 7095])) + (-9.0 / 80.0) * ((sh[c0 + 7194] - sh[c0 + 7146]) - (sh[c0 + 7190] - sh[c0 + 7142])) + (9.0 / 400.0) * ((sh[c0 + 7218] - sh[c0 + 7122]) - (sh[c0 + 7214] - sh[c0 + 7118])) + (-1.0 / 400.0) * ((sh[c0 + 7242] - sh[c0 + 7098]) - (sh[c0 + 7238] - sh[c0 + 7094])) + (1.0 / 80.0) * ((sh[c0 + 7195] - sh[c0 + 7147]) - (sh[c0 + 7189] - sh[c0 + 7141])) + (-1.0 / 400.0) * ((sh[c0 + 7219] - sh[c0 + 7123]) - (sh[c0 + 7213] - sh[c0 + 7117])) + (1.0 / 3600.0) * ((sh[c0 + 7243] - sh[c0 + 7099]) - (sh[c0 + 7237] - sh[c0 + 7093])));
  double V0_vetU_dDD102 = p.invdxx0 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 7457] - sh[c0 + 6881]) - (sh[c0 + 7455] - sh[c0 + 6879])) + (-9.0 / 80.0) * ((sh[c0 + 7745] - sh[c0 + 6593]) - (sh[c0 + 7743] - sh[c0 + 6591])) + (1.0 / 80.0) * ((sh[c0 + 8033] - sh[c0 + 6305]) - (sh[c0 + 8031] - sh[c0 + 6303])) + (-9.0 / 80.0) * ((sh[c0 + 7458] - sh[c0 + 6882]) - (sh[c0 + 7454] - sh[c0 + 6878])) + (9.0 / 400.0) * ((sh[c0 + 7746] - sh[c0 + 6594]) - (sh[c0 + 7742] - sh[c0 + 6590])) + (-1.0 / 400.0) * ((sh[c0 + 8034] - sh[c0 + 6306]) - (sh[c0 + 8030] - sh[c0 + 6302])) + (1.0 / 80.0) * ((sh[c0 + 7459] - sh[c0 + 6883]) - (sh[c0 + 7453] - sh[c0 + 6877])) + (-1.0 / 400.0) * ((sh[c0 + 7747] - sh[c0 + 6595]) - (sh[c0 + 7741] - sh[c0 + 6589])) + (1.0 / 3600.0) * ((sh[c0 + 8035] - sh[c0 + 6307]) - (sh[c0 + 8029] - sh[c0 + 6301])));
  double V0_vetU_dDD111 = p.invdxx1 * p.invdxx1 * ((-49.0 / 18.0) * sh[c0 + 7168] + (3.0 / 2.0) * (sh[c0 + 7192] + sh[c0 + 7144]) + (-3.0 / 20.0) * (sh[c0 + 7216] + sh[c0 + 7120]) + (1.0 / 90.0) * (sh[c0 + 7240] + sh[c0 + 7096]));
  double V0_vetU_dDD112 = p.invdxx1 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 7480] - sh[c0 + 6904]) - (sh[c0 + 7432] - sh[c0 + 6856])) + (-9.0 / 80.0) * ((sh[c0 + 7768] - sh[c0 + 6616]) - (sh[c0 + 7720] - sh[c0 + 6568])) + (1.0 / 80.0) * ((sh[c0 + 8056] - sh[c0 + 6328]) - (sh[c0 + 8008] - sh[c0 + 6280])) + (-9.0 / 80.0) * ((sh[c0 + 7504] - sh[c0 + 6928]) - (sh[c0 + 7408] - sh[c0 + 6832])) + (9.0 / 400.0) * ((sh[c0 + 7792] - sh[c0 + 6640]) - (sh[c0 + 7696] - sh[c0 + 6544])) + (-1.0 / 400.0) * ((sh[c0 + 8080] - sh[c0 + 6352]) - (sh[c0 + 7984] - sh[c0 + 6256])) + (1.0 / 80.0) * ((sh[c0 + 7528] - sh[c0 + 6952]) - (sh[c0 + 7384] - sh[c0 + 6808])) + (-1.0 / 400.0) * ((sh[c0 + 7816] - sh[c0 + 6664]) - (sh[c0 + 7672] - sh[c0 + 6520])) + (1.0 / 3600.0) * ((sh[c0 + 8104] - sh[c0 + 6376]) - (sh[c0 + 7960] - sh[c0 + 6232])));
  double V0_vetU_dDD122 = p.invdxx2 * p.invdxx2 * ((-49.0 / 18.0) * sh[c0 + 7168] + (3.0 / 2.0) * (sh[c0 + 7456] + sh[c0 + 6880]) + (-3.0 / 20.0) * (sh[c0 + 7744] + sh[c0 + 6592]) + (1.0 / 90.0) * (sh[c0 + 8032] + sh[c0 + 6304]));
  const double U0_vetU1_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_vetU1_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_vetU1 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_vetU1_0 : D0_vetU1_0) + L0_coef[1] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_vetU1_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_vetU1_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_vetU1 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_vetU1_1 : D0_vetU1_1) + L0_coef[0] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_vetU1_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_vetU1_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_vetU1 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_vetU1_2 : D0_vetU1_2) + L0_coef[6] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_vetU1), "+v"(V0_vetU_dD10), "+v"(V0_vetU_dD11), "+v"(V0_vetU_dD12), "+v"(V0_vetU_dDD100), "+v"(V0_vetU_dDD101), "+v"(V0_vetU_dDD102), "+v"(V0_vetU_dDD111), "+v"(V0_vetU_dDD112), "+v"(V0_vetU_dDD122), "+v"(V0_lin_vetU1));
  // ---- hDD02
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(15);
  {
    const char *src = (const char *)(in + 15 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD02 = sh[c0];
  double V0_hDD_dD020 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-3.0 / 20.0) * (sh[c0 + 2] - sh[c0 - 2]) + (1.0 / 60.0) * (sh[c0 + 3] - sh[c0 - 3]));
  double V0_hDD_dD021 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 24] - sh[c0 - 24]) + (-3.0 / 20.0) * (sh[c0 + 48] - sh[c0 - 48]) + (1.0 / 60.0) * (sh[c0 + 72] - sh[c0 - 72]));
  double V0_hDD_dD022 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 288] - sh[c0 - 288]) + (-3.0 / 20.0) * (sh[c0 + 576] - sh[c0 - 576]) + (1.0 / 60.0) * (sh[c0 + 864] - sh[c0 - 864]));
  const double U0_hDD02_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_hDD02_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_hDD02 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_hDD02_0 : D0_hDD02_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_hDD02_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_hDD02_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_hDD02 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_hDD02_1 : D0_hDD02_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_hDD02_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_hDD02_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_hDD02 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_hDD02_2 : D0_hDD02_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_hDD02), "+v"(V0_hDD_dD020), "+v"(V0_hDD_dD021), "+v"(V0_hDD_dD022), "+v"(V0_lin_hDD02));
  // ---- hDD11
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(16);
  {
    const char *src = (const char *)(in + 16 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD11 = sh[c0 + 3584];
  double V0_hDD_dD110 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 3585] - sh[c0 + 3583]) + (-3.0 / 20.0) * (sh[c0 + 3586] - sh[c0 + 3582]) + (1.0 / 60.0) * (sh[c0 + 3587] - sh[c0 + 3581]));
  double V0_hDD_dD111 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 3608] - sh[c0 + 3560]) + (-3.0 / 20.0) * (sh[c0 + 3632] - sh[c0 + 3536]) + (1.0 / 60.0) * (sh[c0 + 3656] - sh[c0 + 3512]));
  double V0_hDD_dD112 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 3872] - sh[c0 + 3296]) + (-3.0 / 20.0) * (sh[c0 + 4160] - sh[c0 + 3008]) + (1.0 / 60.0) * (sh[c0 + 4448] - sh[c0 + 2720]));
  const double U0_hDD11_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_hDD11_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_hDD11 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_hDD11_0 : D0_hDD11_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_hDD11_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_hDD11_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_hDD11 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_hDD11_1 : D0_hDD11_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_hDD11_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_hDD11_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_hDD11 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_hDD11_2 : D0_hDD11_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_hDD11), "+v"(V0_hDD_dD110), "+v"(V0_hDD_dD111), "+v"(V0_hDD_dD112), "+v"(V0_lin_hDD11));
  // ---- hDD12
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(17);
  {
    const char *src = (const char *)(in + 23 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD12 = sh[c0 + 7168];
  double V0_hDD_dD120 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 7169] - sh[c0 + 7167]) + (-3.0 / 20.0) * (sh[c0 + 7170] - sh[c0 + 7166]) + (1.0 / 60.0) * (sh[c0 + 7171] - sh[c0 + 7165]));
  double V0_hDD_dD121 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 7192] - sh[c0 + 7144]) + (-3.0 / 20.0) * (sh[c0 + 7216] - sh[c0 + 7120]) + (1.0 / 60.0) * (sh[c0 + 7240] - sh[c0 + 7096]));
  double V0_hDD_dD122 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 7456] - sh[c0 + 6880]) + (-3.0 / 20.0) * (sh[c0 + 7744] - sh[c0 + 6592]) + (1.0 / 60.0) * (sh[c0 + 8032] - sh[c0 + 6304]));
  const double U0_hDD12_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_hDD12_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_hDD12 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_hDD12_0 : D0_hDD12_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_hDD12_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_hDD12_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_hDD12 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_hDD12_1 : D0_hDD12_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_hDD12_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_hDD12_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_hDD12 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_hDD12_2 : D0_hDD12_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_hDD12), "+v"(V0_hDD_dD120), "+v"(V0_hDD_dD121), "+v"(V0_hDD_dD122), "+v"(V0_lin_hDD12));
  // ---- hDD22
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(18);
  {
    const char *src = (const char *)(in + 17 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_hDD22 = sh[c0];
  double V0_hDD_dD220 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 1] - sh[c0 - 1]) + (-3.0 / 20.0) * (sh[c0 + 2] - sh[c0 - 2]) + (1.0 / 60.0) * (sh[c0 + 3] - sh[c0 - 3]));
  double V0_hDD_dD221 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 24] - sh[c0 - 24]) + (-3.0 / 20.0) * (sh[c0 + 48] - sh[c0 - 48]) + (1.0 / 60.0) * (sh[c0 + 72] - sh[c0 - 72]));
  double V0_hDD_dD222 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 288] - sh[c0 - 288]) + (-3.0 / 20.0) * (sh[c0 + 576] - sh[c0 - 576]) + (1.0 / 60.0) * (sh[c0 + 864] - sh[c0 - 864]));
  const double U0_hDD22_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_hDD22_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_hDD22 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_hDD22_0 : D0_hDD22_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_hDD22_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_hDD22_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_hDD22 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_hDD22_1 : D0_hDD22_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_hDD22_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_hDD22_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_hDD22 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_hDD22_2 : D0_hDD22_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_hDD22), "+v"(V0_hDD_dD220), "+v"(V0_hDD_dD221), "+v"(V0_hDD_dD222), "+v"(V0_lin_hDD22));
  // ---- vetU2
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(19);
  {
    const char *src = (const char *)(in + 18 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  double V0_vetU2 = sh[c0 + 3584];
  double V0_vetU_dD20 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 3585] - sh[c0 + 3583]) + (-3.0 / 20.0) * (sh[c0 + 3586] - sh[c0 + 3582]) + (1.0 / 60.0) * (sh[c0 + 3587] - sh[c0 + 3581]));
  double V0_vetU_dD21 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 3608] - sh[c0 + 3560]) + (-3.0 / 20.0) * (sh[c0 + 3632] - sh[c0 + 3536]) + (1.0 / 60.0) * (sh[c0 + 3656] - sh[c0 + 3512]));
  double V0_vetU_dD22 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 3872] - sh[c0 + 3296]) + (-3.0 / 20.0) * (sh[c0 + 4160] - sh[c0 + 3008]) + (1.0 / 60.0) * (sh[c0 + 4448] - sh[c0 + 2720]));
  double V0_vetU_dDD200 = p.invdxx0 * p.invdxx0 * ((-49.0 / 18.0) * sh[c0 + 3584] + (3.0 / 2.0) * (sh[c0 + 3585] + sh[c0 + 3583]) + (-3.0 / 20.0) * (sh[c0 + 3586] + sh[c0 + 3582]) + (1.0 / 90.0) * (sh[c0 + 3587] + sh[c0 + 3581]));
  double V0_vetU_dDD201 = p.invdxx0 * p.invdxx1 * ((9.0 / 16.0) * ((sh[c0 + 3609] - sh[c0 + 3561]) - (sh[c0 + 3607] - sh[c0 + 3559])) + (-9.0 / 80.0) * ((sh[c0 + 3633] - sh[c0 + 3537]) - (sh[c0 + 3631] - sh[c0 + 3535])) + (1.0 / 80.0) * ((sh[c0 + 3657] - sh[c0 + 3513]) - (sh[c0 + 3655] - sh[c0 + 3511])) + (-9.0 / 80.0) * ((sh[c0 + 3610] - sh[c0 + 3562]) - (sh[c0 + 3606] - sh[c0 + 3558])) + (9.0 / 400.0) * ((sh[c0 + 3634] - sh[c0 + 3538]) - (sh[c0 + 3630] - sh[c0 + 3534])) + (-1.0 / 400.0) * ((sh[c0 + 3658] - sh[c0 + 3514]) - (sh[c0 + 3654] - sh[c0 + 3510])) + (1.0 / 80.0) * ((sh[c0 + 3611] - sh[c0 + 3563]) - (sh[c0 + 3605] - sh[c0 + 3557])) + (-1.0 / 400.0) * ((sh[c0 + 3635] - sh[c0 + 3539]) - (sh[c0 + 3629] - sh[c0 + 3533])) + (1.0 / 3600.0) * ((sh[c0 + 3659] - sh[c0 + 3515]) - (sh[c0 + 3653] - sh[c0 + 3509])));
  double V0_vetU_dDD202 = p.invdxx0 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 3873] - sh[c0 + 3297]) - (sh[c0 + 3871] - sh[c0 + 3295])) + (-9.0 / 80.0) * ((sh[c0 + 4161] - sh[c0 + 3009]) - (sh[c0 + 4159] - sh[c0 + 3007])) + (1.0 / 80.0) * ((sh[c0 + 4449] - sh[c0 + 2721]) - (sh[c0 + 4447] - sh[c0 + 2719])) + (-9.0 / 80.0) * ((sh[c0 + 3874] - sh[c0 + 3298]) - (sh[c0 + 3870] - sh[c0 + 3294])) + (9.0 / 400.0) * ((sh[c0 + 4162] - sh[c0 + 3010]) - (sh[c0 + 4158] - sh[c0 + 3006])) + (-1.0 / 400.0) * ((sh[c0 + 4450] - sh[c0 + 2722]) - (sh[c0 + 4446] - sh[c0 + 2718])) + (1.0 / 80.0) * ((sh[c0 + 3875] - sh[c0 + 3299]) - (sh[c0 + 3869] - sh[c0 + 3293])) + (-1.0 / 400.0) * ((sh[c0 + 4163] - sh[c0 + 3011]) - (sh[c0 + 4157] - sh[c0 + 3005])) + (1.0 / 3600.0) * ((sh[c0 + 4451] - sh[c0 + 2723]) - (sh[c0 + 4445] - sh[c0 + 2717])));
  double V0_vetU_dDD211 = p.invdxx1 * p.invdxx1 * ((-49.0 / 18.0) * sh[c0 + 3584] + (3.0 / 2.0) * (sh[c0 + 3608] + sh[c0 + 3560]) + (-3.0 / 20.0) * (sh[c0 + 3632] + sh[c0 + 3536]) + (1.0 / 90.0) * (sh[c0 + 3656] + sh[c0 + 3512]));
  double V0_vetU_dDD212 = p.invdxx1 * p.invdxx2 * ((9.0 / 16.0) * ((sh[c0 + 3896] - sh[c0 + 3320]) - (sh[c0 + 3848] - sh[c0 + 3272])) + (-9.0 / 80.0) * ((sh[c0 + 4184] - sh[c0 + 3032]) - (sh[c0 + 4136] - sh[c0 + 2984])) + (1.0 / 80.0) * ((sh[c0 + 4472] - sh[c0 + 2744]) - (sh[c0 + 4424] - sh[c0 + 2696])) + (-9.0 / 80.0) * ((sh[c0 + 3920] - sh[c0 + 3344]) - (sh[c0 + 3824] - sh[c0 + 3248])) + (9.0 / 400.0) * ((sh[c0 + 4208] - sh[c0 + 3056]) - (sh[c0 + 4112] - sh[c0 + 2960])) + (-1.0 / 400.0) * ((sh[c0 + 4496] - sh[c0 + 2768]) - (sh[c0 + 4400] - sh[c0 + 2672])) + (1.0 / 80.0) * ((sh[c0 + 3944] - sh[c0 + 3368]) - (sh[c0 + 3800] - sh[c0 + 3224])) + (-1.0 / 400.0) * ((sh[c0 + 4232] - sh[c0 + 3080]) - (sh[c0 + 4088] - sh[c0 + 2936])) + (1.0 / 3600.0) * ((sh[c0 + 4520] - sh[c0 + 2792]) - (sh[c0 + 4376] - sh[c0 + 2648])));
  double V0_vetU_dDD222 = p.invdxx2 * p.invdxx2 * ((-49.0 / 18.0) * sh[c0 + 3584] + (3.0 / 2.0) * (sh[c0 + 3872] + sh[c0 + 3296]) + (-3.0 / 20.0) * (sh[c0 + 4160] + sh[c0 + 3008]) + (1.0 / 90.0) * (sh[c0 + 4448] + sh[c0 + 2720]));
  const double U0_vetU2_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_vetU2_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_vetU2 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_vetU2_0 : D0_vetU2_0) + L0_coef[1] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_vetU2_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_vetU2_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_vetU2 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_vetU2_1 : D0_vetU2_1) + L0_coef[0] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_vetU2_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_vetU2_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_vetU2 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_vetU2_2 : D0_vetU2_2) + L0_coef[6] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_vetU2), "+v"(V0_vetU_dD20), "+v"(V0_vetU_dD21), "+v"(V0_vetU_dD22), "+v"(V0_vetU_dDD200), "+v"(V0_vetU_dDD201), "+v"(V0_vetU_dDD202), "+v"(V0_vetU_dDD211), "+v"(V0_vetU_dDD212), "+v"(V0_vetU_dDD222), "+v"(V0_lin_vetU2));
  // ---- lambdaU0
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(20);
  {
    const char *src = (const char *)(in + 19 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 3584 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU0 = sh[c0 + 7168];
  const double U0_lambdaU0_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_lambdaU0_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_lambdaU0 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_lambdaU0_0 : D0_lambdaU0_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_lambdaU0_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_lambdaU0_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_lambdaU0 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_lambdaU0_1 : D0_lambdaU0_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_lambdaU0_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_lambdaU0_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_lambdaU0 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_lambdaU0_2 : D0_lambdaU0_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_lambdaU0), "+v"(V0_lin_lambdaU0));
  // ---- lambdaU1
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(21);
  {
    const char *src = (const char *)(in + 20 * Ntot);
#pragma unroll
    for (int j = 0; j < 7; j++) BHAH_DMA16O(src, pofs[j], sh + 7168 + 2 * (NT * j + 64 * wv));
  }
  double V0_lambdaU1 = sh[c0];
  const double U0_lambdaU1_0 = nius0 * (sh[c0 + 4] + -8.0 * sh[c0 + 3] + -2.0 * sh[c0 - 2] + 30.0 * sh[c0 + 2] + 24.0 * sh[c0 - 1] + -80.0 * sh[c0 + 1] + 35.0 * sh[c0]), D0_lambdaU1_0 = ius0 * (sh[c0 - 4] + -8.0 * sh[c0 - 3] + 30.0 * sh[c0 - 2] + -2.0 * sh[c0 + 2] + -80.0 * sh[c0 - 1] + 24.0 * sh[c0 + 1] + 35.0 * sh[c0]);
  V0_lin_lambdaU1 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_lambdaU1_0 : D0_lambdaU1_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 4] + sh[c0 - 4]) + -8.0 * (sh[c0 + 3] + sh[c0 - 3]) + 28.0 * (sh[c0 + 2] + sh[c0 - 2]) + -56.0 * (sh[c0 + 1] + sh[c0 - 1]) + 70.0 * sh[c0]));
  const double U0_lambdaU1_1 = nius1 * (sh[c0 + 96] + -8.0 * sh[c0 + 72] + -2.0 * sh[c0 - 48] + 30.0 * sh[c0 + 48] + 24.0 * sh[c0 - 24] + -80.0 * sh[c0 + 24] + 35.0 * sh[c0]), D0_lambdaU1_1 = ius1 * (sh[c0 - 96] + -8.0 * sh[c0 - 72] + 30.0 * sh[c0 - 48] + -2.0 * sh[c0 + 48] + -80.0 * sh[c0 - 24] + 24.0 * sh[c0 + 24] + 35.0 * sh[c0]);
  V0_lin_lambdaU1 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_lambdaU1_1 : D0_lambdaU1_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 96] + sh[c0 - 96]) + -8.0 * (sh[c0 + 72] + sh[c0 - 72]) + 28.0 * (sh[c0 + 48] + sh[c0 - 48]) + -56.0 * (sh[c0 + 24] + sh[c0 - 24]) + 70.0 * sh[c0]));
  const double U0_lambdaU1_2 = nius2 * (sh[c0 + 1152] + -8.0 * sh[c0 + 864] + -2.0 * sh[c0 - 576] + 30.0 * sh[c0 + 576] + 24.0 * sh[c0 - 288] + -80.0 * sh[c0 + 288] + 35.0 * sh[c0]), D0_lambdaU1_2 = ius2 * (sh[c0 - 1152] + -8.0 * sh[c0 - 864] + 30.0 * sh[c0 - 576] + -2.0 * sh[c0 + 576] + -80.0 * sh[c0 - 288] + 24.0 * sh[c0 + 288] + 35.0 * sh[c0]);
  V0_lin_lambdaU1 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_lambdaU1_2 : D0_lambdaU1_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 1152] + sh[c0 - 1152]) + -8.0 * (sh[c0 + 864] + sh[c0 - 864]) + 28.0 * (sh[c0 + 576] + sh[c0 - 576]) + -56.0 * (sh[c0 + 288] + sh[c0 - 288]) + 70.0 * sh[c0]));
  BHAH_PINS("+v"(V0_lambdaU1), "+v"(V0_lin_lambdaU1));
  // ---- lambdaU2
  BHAH_VMWAIT(7);
  BHAH_BARRIER_PHASE(22);
  double V0_lambdaU2 = sh[c0 + 3584];
  const double U0_lambdaU2_0 = nius0 * (sh[c0 + 3588] + -8.0 * sh[c0 + 3587] + -2.0 * sh[c0 + 3582] + 30.0 * sh[c0 + 3586] + 24.0 * sh[c0 + 3583] + -80.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]), D0_lambdaU2_0 = ius0 * (sh[c0 + 3580] + -8.0 * sh[c0 + 3581] + 30.0 * sh[c0 + 3582] + -2.0 * sh[c0 + 3586] + -80.0 * sh[c0 + 3583] + 24.0 * sh[c0 + 3585] + 35.0 * sh[c0 + 3584]);
  V0_lin_lambdaU2 += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_lambdaU2_0 : D0_lambdaU2_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 3588] + sh[c0 + 3580]) + -8.0 * (sh[c0 + 3587] + sh[c0 + 3581]) + 28.0 * (sh[c0 + 3586] + sh[c0 + 3582]) + -56.0 * (sh[c0 + 3585] + sh[c0 + 3583]) + 70.0 * sh[c0 + 3584]));
  const double U0_lambdaU2_1 = nius1 * (sh[c0 + 3680] + -8.0 * sh[c0 + 3656] + -2.0 * sh[c0 + 3536] + 30.0 * sh[c0 + 3632] + 24.0 * sh[c0 + 3560] + -80.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]), D0_lambdaU2_1 = ius1 * (sh[c0 + 3488] + -8.0 * sh[c0 + 3512] + 30.0 * sh[c0 + 3536] + -2.0 * sh[c0 + 3632] + -80.0 * sh[c0 + 3560] + 24.0 * sh[c0 + 3608] + 35.0 * sh[c0 + 3584]);
  V0_lin_lambdaU2 += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_lambdaU2_1 : D0_lambdaU2_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 3680] + sh[c0 + 3488]) + -8.0 * (sh[c0 + 3656] + sh[c0 + 3512]) + 28.0 * (sh[c0 + 3632] + sh[c0 + 3536]) + -56.0 * (sh[c0 + 3608] + sh[c0 + 3560]) + 70.0 * sh[c0 + 3584]));
  const double U0_lambdaU2_2 = nius2 * (sh[c0 + 4736] + -8.0 * sh[c0 + 4448] + -2.0 * sh[c0 + 3008] + 30.0 * sh[c0 + 4160] + 24.0 * sh[c0 + 3296] + -80.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]), D0_lambdaU2_2 = ius2 * (sh[c0 + 2432] + -8.0 * sh[c0 + 2720] + 30.0 * sh[c0 + 3008] + -2.0 * sh[c0 + 4160] + -80.0 * sh[c0 + 3296] + 24.0 * sh[c0 + 3872] + 35.0 * sh[c0 + 3584]);
  V0_lin_lambdaU2 += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_lambdaU2_2 : D0_lambdaU2_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 4736] + sh[c0 + 2432]) + -8.0 * (sh[c0 + 4448] + sh[c0 + 2720]) + 28.0 * (sh[c0 + 4160] + sh[c0 + 3008]) + -56.0 * (sh[c0 + 3872] + sh[c0 + 3296]) + 70.0 * sh[c0 + 3584]));
  BHAH_PINS("+v"(V0_lambdaU2), "+v"(V0_lin_lambdaU2));
  // ---- trK
  BHAH_VMWAIT(0);
  BHAH_BARRIER_PHASE(23);
  double V0_trK = sh[c0 + 7168];
  double V0_trK_dD0 = p.invdxx0 * ((3.0 / 4.0) * (sh[c0 + 7169] - sh[c0 + 7167]) + (-3.0 / 20.0) * (sh[c0 + 7170] - sh[c0 + 7166]) + (1.0 / 60.0) * (sh[c0 + 7171] - sh[c0 + 7165]));
  double V0_trK_dD1 = p.invdxx1 * ((3.0 / 4.0) * (sh[c0 + 7192] - sh[c0 + 7144]) + (-3.0 / 20.0) * (sh[c0 + 7216] - sh[c0 + 7120]) + (1.0 / 60.0) * (sh[c0 + 7240] - sh[c0 + 7096]));
  double V0_trK_dD2 = p.invdxx2 * ((3.0 / 4.0) * (sh[c0 + 7456] - sh[c0 + 6880]) + (-3.0 / 20.0) * (sh[c0 + 7744] - sh[c0 + 6592]) + (1.0 / 60.0) * (sh[c0 + 8032] - sh[c0 + 6304]));
  const double U0_trK_0 = nius0 * (sh[c0 + 7172] + -8.0 * sh[c0 + 7171] + -2.0 * sh[c0 + 7166] + 30.0 * sh[c0 + 7170] + 24.0 * sh[c0 + 7167] + -80.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]), D0_trK_0 = ius0 * (sh[c0 + 7164] + -8.0 * sh[c0 + 7165] + 30.0 * sh[c0 + 7166] + -2.0 * sh[c0 + 7170] + -80.0 * sh[c0 + 7167] + 24.0 * sh[c0 + 7169] + 35.0 * sh[c0 + 7168]);
  V0_lin_trK += L0_coef[5] * ((L0_beta[0] > 0.0) ? U0_trK_0 : D0_trK_0) + L0_coef[3] * (ikos0 * -((sh[c0 + 7172] + sh[c0 + 7164]) + -8.0 * (sh[c0 + 7171] + sh[c0 + 7165]) + 28.0 * (sh[c0 + 7170] + sh[c0 + 7166]) + -56.0 * (sh[c0 + 7169] + sh[c0 + 7167]) + 70.0 * sh[c0 + 7168]));
  const double U0_trK_1 = nius1 * (sh[c0 + 7264] + -8.0 * sh[c0 + 7240] + -2.0 * sh[c0 + 7120] + 30.0 * sh[c0 + 7216] + 24.0 * sh[c0 + 7144] + -80.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]), D0_trK_1 = ius1 * (sh[c0 + 7072] + -8.0 * sh[c0 + 7096] + 30.0 * sh[c0 + 7120] + -2.0 * sh[c0 + 7216] + -80.0 * sh[c0 + 7144] + 24.0 * sh[c0 + 7192] + 35.0 * sh[c0 + 7168]);
  V0_lin_trK += L0_coef[4] * ((L0_beta[1] > 0.0) ? U0_trK_1 : D0_trK_1) + L0_coef[2] * (ikos1 * -((sh[c0 + 7264] + sh[c0 + 7072]) + -8.0 * (sh[c0 + 7240] + sh[c0 + 7096]) + 28.0 * (sh[c0 + 7216] + sh[c0 + 7120]) + -56.0 * (sh[c0 + 7192] + sh[c0 + 7144]) + 70.0 * sh[c0 + 7168]));
  const double U0_trK_2 = nius2 * (sh[c0 + 8320] + -8.0 * sh[c0 + 8032] + -2.0 * sh[c0 + 6592] + 30.0 * sh[c0 + 7744] + 24.0 * sh[c0 + 6880] + -80.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]), D0_trK_2 = ius2 * (sh[c0 + 6016] + -8.0 * sh[c0 + 6304] + 30.0 * sh[c0 + 6592] + -2.0 * sh[c0 + 7744] + -80.0 * sh[c0 + 6880] + 24.0 * sh[c0 + 7456] + 35.0 * sh[c0 + 7168]);
  V0_lin_trK += L0_coef[8] * ((L0_beta[2] > 0.0) ? U0_trK_2 : D0_trK_2) + L0_coef[7] * (ikos2 * -((sh[c0 + 8320] + sh[c0 + 6016]) + -8.0 * (sh[c0 + 8032] + sh[c0 + 6304]) + 28.0 * (sh[c0 + 7744] + sh[c0 + 6592]) + -56.0 * (sh[c0 + 7456] + sh[c0 + 6880]) + 70.0 * sh[c0 + 7168]));
  BHAH_PINS("+v"(V0_trK), "+v"(V0_trK_dD0), "+v"(V0_trK_dD1), "+v"(V0_trK_dD2), "+v"(V0_lin_trK));
  {
    const int i0 = o0 + lx, i1 = o1 + ly, i2 = o2 + lz + 0;
    if (i0 < p.Nx0 - p.NG && i1 < p.Nx1 - p.NG && i2 < p.Nx2 - p.NG) {
      const long idx = i0 + s1 * i1 + s2 * i2;
  const double f0_of_xx0__D0 = rfm0[p.Nx0 + i0];
  const double t0 = (f0_of_xx0__D0*f0_of_xx0__D0);
  const double aDD00 = V0_aDD00;
  const double _AbDD00 = aDD00*t0;
  const double f0_of_xx0 = rfm0[i0];
  const double t3 = (f0_of_xx0*f0_of_xx0);
  const double hDD11 = V0_hDD11;
  const double _gbDD11 = hDD11*t3 + t3;
  const double f1_of_xx1 = rfm1[i1];
  const double t5 = (f1_of_xx1*f1_of_xx1);
  const double t6 = t3*t5;
  const double hDD22 = V0_hDD22;
  const double _gbDD22 = hDD22*t6 + t6;
  const double hDD00 = V0_hDD00;
  const double _gbDD00 = hDD00*t0 + t0;
  const double t1 = f0_of_xx0*f0_of_xx0__D0;
  const double hDD01 = V0_hDD01;
  const double _gbDD01 = hDD01*t1;
  const double t2 = f1_of_xx1*t1;
  const double hDD02 = V0_hDD02;
  const double _gbDD02 = hDD02*t2;
  const double t4 = f1_of_xx1*t3;
  const double hDD12 = V0_hDD12;
  const double _gbDD12 = hDD12*t4;
  const double t7 = (_gbDD12*_gbDD12);
  const double t8 = (_gbDD02*_gbDD02);
  const double t9 = (_gbDD01*_gbDD01);
  const double t10 = (1.0 / (_gbDD00*_gbDD11*_gbDD22 - _gbDD00*t7 + 2.0*_gbDD01*_gbDD02*_gbDD12 - _gbDD11*t8 - _gbDD22*t9));
  const double _gbUU00 = t10*(_gbDD11*_gbDD22 - t7);
  const double t45 = _AbDD00*_gbUU00;
  const double aDD01 = V0_aDD01;
  const double _AbDD01 = aDD01*t1;
  const double _gbUU01 = t10*(-_gbDD01*_gbDD22 + _gbDD02*_gbDD12);
  const double t46 = _AbDD01*_gbUU01;
  const double aDD02 = V0_aDD02;
  const double _AbDD02 = aDD02*t2;
  const double _gbUU02 = t10*(_gbDD01*_gbDD12 - _gbDD02*_gbDD11);
  const double t47 = _AbDD02*_gbUU02;
  const double _AbUD00 = t45 + t46 + t47;
  const double _gbUU11 = t10*(_gbDD00*_gbDD22 - t8);
  const double _gbUU12 = t10*(-_gbDD00*_gbDD12 + _gbDD01*_gbDD02);
  const double _AbUD10 = _AbDD00*_gbUU01 + _AbDD01*_gbUU11 + _AbDD02*_gbUU12;
  const double _gbUU22 = t10*(_gbDD00*_gbDD11 - t9);
  const double _AbUD20 = _AbDD00*_gbUU02 + _AbDD01*_gbUU12 + _AbDD02*_gbUU22;
  const double t55 = (1.0 / f0_of_xx0);
  const double t65 = (1.0 / t3);
  const double t66 = f0_of_xx0__D0*t65;
  const double vetU1 = V0_vetU1;
  const double vetU_dD10 = V0_vetU_dD10;
  const double _bUdD10 = t55*vetU_dD10 - t66*vetU1;
  const double t58 = (1.0 / f1_of_xx1);
  const double t67 = t55*t58;
  const double t68 = t58*t66;
  const double vetU2 = V0_vetU2;
  const double vetU_dD20 = V0_vetU_dD20;
  const double _bUdD20 = t67*vetU_dD20 - t68*vetU2;
  const double f0_of_xx0__DD00 = rfm0[2 * p.Nx0 + i0];
  const double t11 = 2.0*f0_of_xx0__DD00;
  const double t12 = f0_of_xx0__D0*t11;
  const double t13 = hDD00*t12 + t12;
  const double hDD_dD000 = V0_hDD_dD000;
  const double _gbDDdD000 = hDD_dD000*t0 + t13;
  const double t30 = (Rational_1_2)*_gbUU00;
  const double hDD_dD001 = V0_hDD_dD001;
  const double _gbDDdD001 = hDD_dD001*t0;
  const double t14 = f0_of_xx0*f0_of_xx0__DD00;
  const double t15 = t0 + t14;
  const double t16 = hDD01*t15;
  const double hDD_dD010 = V0_hDD_dD010;
  const double _gbDDdD010 = hDD_dD010*t1 + t16;
  const double t31 = -_gbDDdD001 + 2.0*_gbDDdD010;
  const double t32 = (Rational_1_2)*_gbUU01;
  const double hDD_dD002 = V0_hDD_dD002;
  const double _gbDDdD002 = hDD_dD002*t0;
  const double t17 = f1_of_xx1*t0;
  const double t18 = f1_of_xx1*t14 + t17;
  const double t19 = hDD02*t18;
  const double hDD_dD020 = V0_hDD_dD020;
  const double _gbDDdD020 = hDD_dD020*t2 + t19;
  const double t33 = -_gbDDdD002 + 2.0*_gbDDdD020;
  const double t34 = (Rational_1_2)*_gbUU02;
  const double _GbUDD000 = _gbDDdD000*t30 + t31*t32 + t33*t34;
  const double t42 = (Rational_1_2)*_gbUU11;
  const double t43 = (Rational_1_2)*_gbUU12;
  const double _GbUDD100 = _gbDDdD000*t32 + t31*t42 + t33*t43;
  const double t44 = (Rational_1_2)*_gbUU22;
  const double _GbUDD200 = _gbDDdD000*t34 + t31*t43 + t33*t44;
  const double alpha_dD0 = V0_alpha_dD0;
  const double alpha_dD1 = V0_alpha_dD1;
  const double alpha_dD2 = V0_alpha_dD2;
  const double alpha_dDD00 = V0_alpha_dDD00;
  const double _adBDD00 = -_GbUDD000*alpha_dD0 - _GbUDD100*alpha_dD1 - _GbUDD200*alpha_dD2 + alpha_dDD00;
  const double cf = V0_cf;
  const double t81 = (1.0 / cf);
  const double t82 = (Rational_1_2)*t81;
  const double cf_dD0 = V0_cf_dD0;
  const double _phidD0 = -cf_dD0*t82;
  const double cf_dD1 = V0_cf_dD1;
  const double _phidD1 = -cf_dD1*t82;
  const double cf_dD2 = V0_cf_dD2;
  const double _phidD2 = -cf_dD2*t82;
  const double cf_dDD00 = V0_cf_dDD00;
  const double _phidBDD00 = -_GbUDD000*_phidD0 - _GbUDD100*_phidD1 - _GbUDD200*_phidD2 + (Rational_1_2)*t81*((cf_dD0*cf_dD0)*t81 - cf_dDD00);
  const double alpha = V0_alpha;
  const double t92 = 2.0*alpha;
  const double t93 = _phidD0*alpha_dD0;
  const double t94 = 4.0*alpha;
  const double RbarDD00 = aux[0 * Ntot + idx];
  const double _curly00 = RbarDD00*alpha - _adBDD00 - _phidBDD00*t92 + (_phidD0*_phidD0)*t94 + 4.0*t93;
  const double t106 = (cf*cf);
  const double t21 = 2.0*t1;
  const double t22 = hDD11*t21 + t21;
  const double hDD_dD110 = V0_hDD_dD110;
  const double _gbDDdD110 = hDD_dD110*t3 + t22;
  const double hDD_dD012 = V0_hDD_dD012;
  const double _gbDDdD012 = hDD_dD012*t1;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t20 = f1_of_xx1__D1*hDD02;
  const double hDD_dD021 = V0_hDD_dD021;
  const double _gbDDdD021 = hDD_dD021*t2 + t1*t20;
  const double hDD_dD120 = V0_hDD_dD120;
  const double _gbDDdD120 = f1_of_xx1*hDD12*t21 + hDD_dD120*t4;
  const double t35 = -_gbDDdD012 + _gbDDdD021 + _gbDDdD120;
  const double _GbUDD001 = _gbDDdD001*t30 + _gbDDdD110*t32 + t34*t35;
  const double _GbUDD101 = _gbDDdD001*t32 + _gbDDdD110*t42 + t35*t43;
  const double _GbUDD201 = _gbDDdD001*t34 + _gbDDdD110*t43 + t35*t44;
  const double alpha_dDD01 = V0_alpha_dDD01;
  const double _adBDD01 = -_GbUDD001*alpha_dD0 - _GbUDD101*alpha_dD1 - _GbUDD201*alpha_dD2 + alpha_dDD01;
  const double cf_dDD01 = V0_cf_dDD01;
  const double _phidBDD01 = -_GbUDD001*_phidD0 - _GbUDD101*_phidD1 - _GbUDD201*_phidD2 + (Rational_1_2)*t81*(cf_dD0*cf_dD1*t81 - cf_dDD01);
  const double t95 = 2.0*_phidD0;
  const double t96 = alpha_dD1*t95;
  const double t97 = 2.0*alpha_dD0;
  const double t98 = _phidD1*t97;
  const double t99 = _phidD0*t94;
  const double RbarDD01 = aux[1 * Ntot + idx];
  const double _curly01 = RbarDD01*alpha - _adBDD01 - _phidBDD01*t92 + _phidD1*t99 + t96 + t98;
  const double t24 = t21*t5;
  const double t25 = hDD22*t24 + t24;
  const double hDD_dD220 = V0_hDD_dD220;
  const double _gbDDdD220 = hDD_dD220*t6 + t25;
  const double t36 = _gbDDdD012 - _gbDDdD021 + _gbDDdD120;
  const double _GbUDD002 = _gbDDdD002*t30 + _gbDDdD220*t34 + t32*t36;
  const double _GbUDD102 = _gbDDdD002*t32 + _gbDDdD220*t43 + t36*t42;
  const double _GbUDD202 = _gbDDdD002*t34 + _gbDDdD220*t44 + t36*t43;
  const double alpha_dDD02 = V0_alpha_dDD02;
  const double _adBDD02 = -_GbUDD002*alpha_dD0 - _GbUDD102*alpha_dD1 - _GbUDD202*alpha_dD2 + alpha_dDD02;
  const double cf_dDD02 = V0_cf_dDD02;
  const double _phidBDD02 = -_GbUDD002*_phidD0 - _GbUDD102*_phidD1 - _GbUDD202*_phidD2 + (Rational_1_2)*t81*(cf_dD0*cf_dD2*t81 - cf_dDD02);
  const double t100 = alpha_dD2*t95;
  const double t101 = _phidD2*t97;
  const double RbarDD02 = aux[2 * Ntot + idx];
  const double _curly02 = RbarDD02*alpha - _adBDD02 - _phidBDD02*t92 + _phidD2*t99 + t100 + t101;
  const double hDD_dD111 = V0_hDD_dD111;
  const double _gbDDdD111 = hDD_dD111*t3;
  const double hDD_dD011 = V0_hDD_dD011;
  const double _gbDDdD011 = hDD_dD011*t1;
  const double t37 = 2.0*_gbDDdD011 - _gbDDdD110;
  const double hDD_dD112 = V0_hDD_dD112;
  const double _gbDDdD112 = hDD_dD112*t3;
  const double t23 = f1_of_xx1__D1*hDD12;
  const double hDD_dD121 = V0_hDD_dD121;
  const double _gbDDdD121 = hDD_dD121*t4 + t23*t3;
  const double t38 = -_gbDDdD112 + 2.0*_gbDDdD121;
  const double _GbUDD011 = _gbDDdD111*t32 + t30*t37 + t34*t38;
  const double _GbUDD111 = _gbDDdD111*t42 + t32*t37 + t38*t43;
  const double _GbUDD211 = _gbDDdD111*t43 + t34*t37 + t38*t44;
  const double alpha_dDD11 = V0_alpha_dDD11;
  const double _adBDD11 = -_GbUDD011*alpha_dD0 - _GbUDD111*alpha_dD1 - _GbUDD211*alpha_dD2 + alpha_dDD11;
  const double cf_dDD11 = V0_cf_dDD11;
  const double _phidBDD11 = -_GbUDD011*_phidD0 - _GbUDD111*_phidD1 - _GbUDD211*_phidD2 + (Rational_1_2)*t81*((cf_dD1*cf_dD1)*t81 - cf_dDD11);
  const double t102 = _phidD1*alpha_dD1;
  const double RbarDD11 = aux[3 * Ntot + idx];
  const double _curly11 = RbarDD11*alpha - _adBDD11 - _phidBDD11*t92 + (_phidD1*_phidD1)*t94 + 4.0*t102;
  const double t26 = f1_of_xx1*f1_of_xx1__D1;
  const double t27 = 2.0*t26;
  const double t28 = t27*t3;
  const double t29 = hDD22*t28 + t28;
  const double hDD_dD221 = V0_hDD_dD221;
  const double _gbDDdD221 = hDD_dD221*t6 + t29;
  const double t39 = _gbDDdD012 + _gbDDdD021 - _gbDDdD120;
  const double _GbUDD012 = _gbDDdD112*t32 + _gbDDdD221*t34 + t30*t39;
  const double _GbUDD112 = _gbDDdD112*t42 + _gbDDdD221*t43 + t32*t39;
  const double _GbUDD212 = _gbDDdD112*t43 + _gbDDdD221*t44 + t34*t39;
  const double alpha_dDD12 = V0_alpha_dDD12;
  const double _adBDD12 = -_GbUDD012*alpha_dD0 - _GbUDD112*alpha_dD1 - _GbUDD212*alpha_dD2 + alpha_dDD12;
  const double cf_dDD12 = V0_cf_dDD12;
  const double _phidBDD12 = -_GbUDD012*_phidD0 - _GbUDD112*_phidD1 - _GbUDD212*_phidD2 + (Rational_1_2)*t81*(cf_dD1*cf_dD2*t81 - cf_dDD12);
  const double t103 = 2.0*alpha_dD2;
  const double t104 = _phidD1*t103;
  const double t105 = 2.0*_phidD2*alpha_dD1;
  const double RbarDD12 = aux[4 * Ntot + idx];
  const double _curly12 = RbarDD12*alpha - _adBDD12 - _phidBDD12*t92 + _phidD1*_phidD2*t94 + t104 + t105;
  const double hDD_dD222 = V0_hDD_dD222;
  const double _gbDDdD222 = hDD_dD222*t6;
  const double hDD_dD022 = V0_hDD_dD022;
  const double _gbDDdD022 = hDD_dD022*t2;
  const double t40 = 2.0*_gbDDdD022 - _gbDDdD220;
  const double hDD_dD122 = V0_hDD_dD122;
  const double _gbDDdD122 = hDD_dD122*t4;
  const double t41 = 2.0*_gbDDdD122 - _gbDDdD221;
  const double _GbUDD022 = _gbDDdD222*t34 + t30*t40 + t32*t41;
  const double _GbUDD122 = _gbDDdD222*t43 + t32*t40 + t41*t42;
  const double _GbUDD222 = _gbDDdD222*t44 + t34*t40 + t41*t43;
  const double alpha_dDD22 = V0_alpha_dDD22;
  const double _adBDD22 = -_GbUDD022*alpha_dD0 - _GbUDD122*alpha_dD1 - _GbUDD222*alpha_dD2 + alpha_dDD22;
  const double cf_dDD22 = V0_cf_dDD22;
  const double _phidBDD22 = -_GbUDD022*_phidD0 - _GbUDD122*_phidD1 - _GbUDD222*_phidD2 + (Rational_1_2)*t81*((cf_dD2*cf_dD2)*t81 - cf_dDD22);
  const double RbarDD22 = aux[5 * Ntot + idx];
  const double _curly22 = RbarDD22*alpha - _adBDD22 - _phidBDD22*t92 + (_phidD2*_phidD2)*t94 + 4.0*_phidD2*alpha_dD2;
  const double t60 = 2.0*_gbUU01;
  const double t61 = 2.0*_gbUU02;
  const double t62 = 2.0*_gbUU12;
  const double _curlytr = _curly00*_gbUU00 + _curly01*t60 + _curly02*t61 + _curly11*_gbUU11 + _curly12*t62 + _curly22*_gbUU22;
  const double t107 = (Rational_1_3)*_curlytr;
  const double t51 = (1.0 / f0_of_xx0__D0);
  const double t63 = (1.0 / t0);
  const double t64 = f0_of_xx0__DD00*t63;
  const double vetU0 = V0_vetU0;
  const double vetU_dD00 = V0_vetU_dD00;
  const double _bUdD00 = t51*vetU_dD00 - t64*vetU0;
  const double t108 = 2.0*_bUdD00;
  const double t109 = 2.0*_AbDD01;
  const double t110 = 2.0*_AbDD02;
  const double vetU_dD11 = V0_vetU_dD11;
  const double _bUdD11 = t55*vetU_dD11;
  const double vetU_dD22 = V0_vetU_dD22;
  const double _bUdD22 = t67*vetU_dD22;
  const double t59 = f1_of_xx1__D1*t58;
  const double t83 = t55*vetU1;
  const double t69 = (1.0 / t5);
  const double t84 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t85 = (1.0 / t84);
  const double t86 = (Rational_1_2)*t69*t85;
  const double t72 = (f0_of_xx0__D0*f0_of_xx0__D0*f0_of_xx0__D0);
  const double t76 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t87 = t5*t76;
  const double t88 = t5*t84;
  const double t89 = t12*t88 + 4.0*t72*t87;
  const double t73 = (1.0 / t72);
  const double t90 = t73*vetU0;
  const double t91 = t89*t90;
  const double _Dbb = _bUdD00 + _bUdD11 + _bUdD22 + t59*t83 + t86*t91;
  const double t111 = (Rational_2_3)*_Dbb;
  const double trK = V0_trK;
  const double t112 = alpha*trK;
  const double t113 = _AbDD00*t92;
  const double t114 = _AbDD01*t92;
  const double t115 = _AbDD02*t92;
  out[0 * Ntot + idx] = t63*(_AbDD00*t108 - _AbDD00*t111 + _AbDD00*t112 - _AbUD00*t113 - _AbUD10*t114 - _AbUD20*t115 + _bUdD10*t109 + _bUdD20*t110 + aDD00*t11*vetU0 + t106*(_curly00 - _gbDD00*t107)) + V0_lin_aDD00;
  const double aDD11 = V0_aDD11;
  const double _AbDD11 = aDD11*t3;
  const double aDD12 = V0_aDD12;
  const double _AbDD12 = aDD12*t4;
  const double _AbUD01 = _AbDD01*_gbUU00 + _AbDD11*_gbUU01 + _AbDD12*_gbUU02;
  const double t48 = _AbDD11*_gbUU11;
  const double t49 = _AbDD12*_gbUU12;
  const double _AbUD11 = t46 + t48 + t49;
  const double _AbUD21 = _AbDD01*_gbUU02 + _AbDD11*_gbUU12 + _AbDD12*_gbUU22;
  const double vetU_dD01 = V0_vetU_dD01;
  const double _bUdD01 = t51*vetU_dD01;
  const double t70 = t55*t69;
  const double t71 = f1_of_xx1__D1*t70;
  const double vetU_dD21 = V0_vetU_dD21;
  const double _bUdD21 = t67*vetU_dD21 - t71*vetU2;
  const double t116 = t51*vetU0;
  const double t117 = t51*t55;
  out[1 * Ntot + idx] = t117*(_AbDD00*_bUdD01 + _AbDD01*_bUdD00 + _AbDD01*_bUdD11 - _AbDD01*t111 + _AbDD01*t112 + _AbDD02*_bUdD21 + _AbDD11*_bUdD10 + _AbDD12*_bUdD20 - _AbUD01*t113 - _AbUD11*t114 - _AbUD21*t115 + aDD01*t116*t15 + t106*(_curly01 - _gbDD01*t107)) + V0_lin_aDD01;
  const double aDD22 = V0_aDD22;
  const double _AbDD22 = aDD22*t6;
  const double _AbUD02 = _AbDD02*_gbUU00 + _AbDD12*_gbUU01 + _AbDD22*_gbUU02;
  const double _AbUD12 = _AbDD02*_gbUU01 + _AbDD12*_gbUU11 + _AbDD22*_gbUU12;
  const double t50 = _AbDD22*_gbUU22;
  const double _AbUD22 = t47 + t49 + t50;
  const double vetU_dD02 = V0_vetU_dD02;
  const double _bUdD02 = t51*vetU_dD02;
  const double vetU_dD12 = V0_vetU_dD12;
  const double _bUdD12 = t55*vetU_dD12;
  const double t118 = f1_of_xx1__D1*vetU1;
  const double t119 = t51*t67;
  out[2 * Ntot + idx] = t119*(_AbDD00*_bUdD02 + _AbDD01*_bUdD12 + _AbDD02*_bUdD00 + _AbDD02*_bUdD22 - _AbDD02*t111 + _AbDD02*t112 + _AbDD12*_bUdD10 + _AbDD22*_bUdD20 - _AbUD02*t113 - _AbUD12*t114 - _AbUD22*t115 + aDD02*f0_of_xx0__D0*t118 + aDD02*t116*t18 + t106*(_curly02 - _gbDD02*t107)) + V0_lin_aDD02;
  const double t120 = 2.0*_bUdD11;
  const double t121 = 2.0*_AbDD12;
  const double t122 = _AbDD11*t92;
  const double t123 = _AbDD12*t92;
  const double t124 = 2.0*vetU0;
  const double t125 = f0_of_xx0*t124;
  out[3 * Ntot + idx] = t65*(-_AbDD11*t111 + _AbDD11*t112 + _AbDD11*t120 - _AbUD01*t114 - _AbUD11*t122 - _AbUD21*t123 + _bUdD01*t109 + _bUdD21*t121 + aDD11*t125 + t106*(_curly11 - _gbDD11*t107)) + V0_lin_aDD11;
  const double t126 = f0_of_xx0*f1_of_xx1;
  const double t127 = t124*t126;
  const double t128 = t58*t65;
  out[4 * Ntot + idx] = t128*(_AbDD01*_bUdD02 + _AbDD02*_bUdD01 + _AbDD11*_bUdD12 + _AbDD12*_bUdD11 + _AbDD12*_bUdD22 - _AbDD12*t111 + _AbDD12*t112 + _AbDD22*_bUdD21 - _AbUD02*t114 - _AbUD12*t122 - _AbUD22*t123 + aDD12*f0_of_xx0*t118 + aDD12*t127 + t106*(_curly12 - _gbDD12*t107)) + V0_lin_aDD12;
  const double t129 = 2.0*_bUdD22;
  const double t130 = _AbDD22*t92;
  const double t131 = f0_of_xx0*vetU1;
  const double t132 = t65*t69;
  out[5 * Ntot + idx] = t132*(-_AbDD22*t111 + _AbDD22*t112 + _AbDD22*t129 - _AbUD02*t115 - _AbUD12*t123 - _AbUD22*t130 + _bUdD02*t110 + _bUdD12*t121 + aDD22*t125*t5 + aDD22*t131*t27 + t106*(_curly22 - _gbDD22*t107)) + V0_lin_aDD22;
  out[6 * Ntot + idx] = -t92*trK + V0_lin_alpha;
  const double _AbUU00 = _AbUD00*_gbUU00 + _AbUD01*_gbUU01 + _AbUD02*_gbUU02;
  const double _AbUU01 = _AbUD00*_gbUU01 + _AbUD01*_gbUU11 + _AbUD02*_gbUU12;
  const double _AbUU02 = _AbUD00*_gbUU02 + _AbUD01*_gbUU12 + _AbUD02*_gbUU22;
  const double _AbUU12 = _AbUD10*_gbUU02 + _AbUD11*_gbUU12 + _AbUD12*_gbUU22;
  const double _AbUU20 = _AbUD20*_gbUU00 + _AbUD21*_gbUU01 + _AbUD22*_gbUU02;
  const double _AbUU21 = _AbUD20*_gbUU01 + _AbUD21*_gbUU11 + _AbUD22*_gbUU12;
  const double t52 = f0_of_xx0__DD00*t51;
  const double _DGUDD000 = _GbUDD000 - t52;
  const double t53 = f0_of_xx0*t51;
  const double _DGUDD011 = _GbUDD011 + t53;
  const double t54 = t5*t53;
  const double _DGUDD022 = _GbUDD022 + t54;
  const double _DGU0 = _DGUDD000*_gbUU00 + _DGUDD011*_gbUU11 + _DGUDD022*_gbUU22 + _GbUDD001*t60 + _GbUDD002*t61 + _GbUDD012*t62;
  const double t133 = (Rational_1_2)*_Dbb;
  const double t134 = 6.0*alpha;
  const double t135 = -_phidD0*t134 + alpha_dD0;
  const double t136 = (Rational_3_2)*t135;
  const double t137 = -_phidD1*t134 + alpha_dD1;
  const double t138 = (Rational_3_2)*t137;
  const double t139 = -_phidD2*t134 + alpha_dD2;
  const double t140 = (Rational_3_2)*t139;
  const double t74 = (f0_of_xx0__DD00*f0_of_xx0__DD00);
  const double f0_of_xx0__DDD000 = rfm0[3 * p.Nx0 + i0];
  const double vetU_dDD000 = V0_vetU_dDD000;
  const double _bUdDD000 = -t11*t63*vetU_dD00 + t51*vetU_dDD000 + vetU0*(-f0_of_xx0__DDD000*t63 + 2.0*t73*t74);
  const double vetU_dDD101 = V0_vetU_dDD101;
  const double _bUdDD101 = t55*vetU_dDD101 - t66*vetU_dD11;
  const double vetU_dDD202 = V0_vetU_dDD202;
  const double _bUdDD202 = t67*vetU_dDD202 - t68*vetU_dD22;
  const double t141 = t63*t86;
  const double t142 = 4.0*f0_of_xx0__D0*f0_of_xx0__DD00*t26*t84 + 8.0*t26*t72*t76;
  const double t143 = t17*t84;
  const double t144 = 2.0*t143;
  const double t79 = (1.0 / (f1_of_xx1*f1_of_xx1*f1_of_xx1));
  const double t145 = _bUdDD000 + _bUdDD101 + _bUdDD202 + t141*(_bUdD00*t89 + t116*(12.0*(f0_of_xx0__D0*f0_of_xx0__D0*f0_of_xx0__D0*f0_of_xx0__D0)*t6 + 2.0*f0_of_xx0__D0*f0_of_xx0__DDD000*t88 + 20.0*f0_of_xx0__DD00*t0*t87 + 2.0*t74*t88)) + t141*(_bUdD10*f1_of_xx1__D1*t144 + t142*t83) - t118*t63*t79*t89/(f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0) - Rational_1_2*(t89*t89)*vetU0/((f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0)*(f0_of_xx0__D0*f0_of_xx0__D0*f0_of_xx0__D0*f0_of_xx0__D0*f0_of_xx0__D0)*(f1_of_xx1*f1_of_xx1*f1_of_xx1*f1_of_xx1));
  const double t146 = (Rational_1_4)*t145;
  const double vetU_dDD001 = V0_vetU_dDD001;
  const double _bUdDD001 = t51*vetU_dDD001 - t64*vetU_dD01;
  const double vetU_dDD111 = V0_vetU_dDD111;
  const double _bUdDD111 = t55*vetU_dDD111;
  const double vetU_dDD212 = V0_vetU_dDD212;
  const double _bUdDD212 = t67*vetU_dDD212 - t71*vetU_dD22;
  const double t80 = (f1_of_xx1__D1*f1_of_xx1__D1);
  const double t147 = t69*t80;
  const double t148 = t147*t83;
  const double f1_of_xx1__DD11 = rfm1[2 * p.Nx1 + i1];
  const double t149 = _bUdDD001 + _bUdDD111 + _bUdDD212 - f1_of_xx1__D1*t79*t85*t91 + t141*(_bUdD01*t89 + t116*t142) + t141*(f1_of_xx1__D1*t120*t143 + t83*(f1_of_xx1__DD11*t144 + 2.0*t0*t80*t84)) - 2.0*t148;
  const double t150 = (Rational_1_4)*t149;
  const double vetU_dDD002 = V0_vetU_dDD002;
  const double _bUdDD002 = t51*vetU_dDD002 - t64*vetU_dD02;
  const double vetU_dDD112 = V0_vetU_dDD112;
  const double _bUdDD112 = t55*vetU_dDD112;
  const double vetU_dDD222 = V0_vetU_dDD222;
  const double _bUdDD222 = t67*vetU_dDD222;
  const double t151 = _bUdD12*t59;
  const double t152 = _bUdD02*t141*t89 + _bUdDD002 + _bUdDD112 + _bUdDD222 + t151;
  const double t153 = (Rational_1_4)*t152;
  const double vetU_dDD012 = V0_vetU_dDD012;
  const double _bUdDD012 = t51*vetU_dDD012;
  const double t154 = -_bUdD02*t59 - _bUdD12*t53 - _bUdD21*t54 + _bUdDD012;
  const double t155 = _gbUU00*(_bUdD00*t52 + _bUdDD000 + t116*(f0_of_xx0__DDD000*t51 - t63*t74));
  const double t56 = f0_of_xx0__D0*t55;
  const double t156 = _bUdD01*t56;
  const double t157 = _bUdD10*t53;
  const double t158 = _bUdD01*t52 + _bUdDD001 - t156 - t157;
  const double t159 = _gbUU01*t158;
  const double t160 = t14*t63;
  const double t161 = _gbUU01*(t158 - t64*vetU1 + t83*(t160 - 1.0) + t83);
  const double t162 = _bUdD02*t56;
  const double t163 = _bUdD20*t54;
  const double t164 = _bUdD02*t52 + _bUdDD002 - t162 - t163;
  const double t165 = _gbUU02*t164;
  const double t166 = f1_of_xx1*vetU2;
  const double t167 = t166*t55;
  const double t168 = t67*vetU2;
  const double t169 = _gbUU02*(t164 - t166*t64 + t167 + t168*(t160*t5 - t5));
  const double vetU_dDD011 = V0_vetU_dDD011;
  const double _bUdDD011 = t51*vetU_dDD011;
  const double t170 = t14*t90;
  const double t171 = _gbUU11*(_bUdD00*t53 + _bUdDD011 - t116 - t120*t53 + t170);
  const double vetU_dDD022 = V0_vetU_dDD022;
  const double _bUdDD022 = t51*vetU_dDD022;
  const double t172 = _gbUU22*(_bUdD00*t54 + _bUdD01*t26 + _bUdDD022 - t116*t5 - t129*t54 + t170*t5 - t27*t51*vetU1);
  const double trK_dD0 = V0_trK_dD0;
  const double t173 = alpha*trK_dD0;
  const double t174 = _gbUU00*t173;
  const double trK_dD1 = V0_trK_dD1;
  const double t175 = alpha*trK_dD1;
  const double t176 = _gbUU01*t175;
  const double trK_dD2 = V0_trK_dD2;
  const double t177 = alpha*trK_dD2;
  const double t178 = _gbUU02*t177;
  const double betU0 = V0_betU0;
  const double t179 = betU0*t51;
  const double lambdaU0 = V0_lambdaU0;
  const double t180 = lambdaU0*t51;
  const double t181 = _bUdD00*t180;
  const double lambdaU1 = V0_lambdaU1;
  const double t182 = lambdaU1*t55;
  const double t183 = _bUdD01*t182;
  const double t184 = _AbUU00*alpha;
  const double t185 = (Rational_3_2)*t184;
  const double t186 = (Rational_3_2)*alpha;
  const double t187 = _AbUU01*_GbUDD001;
  const double t188 = _GbUDD002*t186;
  const double _AbUU10 = _AbUD10*_gbUU00 + _AbUD11*_gbUU01 + _AbUD12*_gbUU02;
  const double t189 = _AbUU10*t186;
  const double _AbUU11 = _AbUD10*_gbUU01 + _AbUD11*_gbUU11 + _AbUD12*_gbUU12;
  const double t190 = _AbUU11*alpha;
  const double t191 = (Rational_3_2)*t190;
  const double t192 = _GbUDD012*t186;
  const double _AbUU22 = _AbUD20*_gbUU02 + _AbUD21*_gbUU12 + _AbUD22*_gbUU22;
  const double t193 = _AbUU22*alpha;
  const double t194 = (Rational_3_2)*t193;
  const double t195 = betU0*vetU0;
  const double t196 = t195*t63;
  const double t197 = t65*vetU1;
  const double betU1 = V0_betU1;
  const double t198 = betU1*t197;
  const double t199 = f0_of_xx0__DD00*t73;
  const double t200 = lambdaU0*vetU0;
  const double t201 = (Rational_3_4)*t200*t63;
  const double t202 = (Rational_3_4)*lambdaU1;
  const double t203 = t197*t202;
  const double lambdaU2 = V0_lambdaU2;
  const double t204 = lambdaU2*t67;
  const double t205 = _bUdD02*t204;
  const double t206 = t179*t83;
  const double t207 = betU1*t55;
  const double t208 = t116*t207;
  const double t209 = _GbUDD012*t128;
  const double t210 = betU1*vetU2;
  const double betU2 = V0_betU2;
  const double t211 = betU2*vetU1;
  const double t212 = betU2*t132;
  const double t213 = t212*vetU2;
  const double t214 = (Rational_3_4)*_GbUDD001;
  const double t215 = t180*t83;
  const double t216 = t116*t182;
  const double t217 = t202*vetU2;
  const double t218 = (Rational_3_4)*lambdaU2;
  const double t219 = t209*vetU1;
  const double t220 = t132*t218*vetU2;
  const double t221 = t168*t179;
  const double t222 = betU2*t67;
  const double t223 = t116*t222;
  const double t224 = (Rational_3_4)*_GbUDD002;
  const double t225 = t168*t180;
  const double t226 = t116*t204;
  const double eta = p.eta;
  out[7 * Ntot + idx] = f0_of_xx0__D0*(-_AbUU00*t136 - _AbUU01*t138 - _AbUU02*t140 + _AbUU02*t188 + _AbUU12*t192 + _AbUU20*t188 + _AbUU21*t192 + _DGU0*t133 + _DGUDD000*t185 + _DGUDD011*t191 + _DGUDD022*t194 + _GbUDD000*t196 - _GbUDD000*t201 + _GbUDD001*t189 + _GbUDD001*t206 + _GbUDD001*t208 + _GbUDD002*t221 + _GbUDD002*t223 + _GbUDD011*t198 - _GbUDD011*t203 + _GbUDD022*t213 - _GbUDD022*t220 + _gbUU00*t146 + _gbUU01*t150 + _gbUU02*t153 + (Rational_3_2)*_gbUU12*t154 - eta*t179 + (Rational_3_4)*t155 + (Rational_3_4)*t159 + (Rational_3_4)*t161 + (Rational_3_4)*t165 + (Rational_3_4)*t169 + (Rational_3_4)*t171 + (Rational_3_4)*t172 - t174 - t176 - t178 - Rational_3_4*t181 - Rational_3_4*t183 + t186*t187 - t195*t199 - Rational_3_4*t205 + t209*t210 + t209*t211 - t209*t217 - t214*t215 - t214*t216 - t218*t219 - t224*t225 - t224*t226) + V0_lin_betU0;
  const double t57 = -t56;
  const double _DGUDD101 = _GbUDD101 + t57;
  const double _DGUDD122 = _GbUDD122 + t26;
  const double _DGU1 = _DGUDD101*t60 + _DGUDD122*_gbUU22 + _GbUDD100*_gbUU00 + _GbUDD102*t61 + _GbUDD111*_gbUU11 + _GbUDD112*t62;
  const double vetU_dDD102 = V0_vetU_dDD102;
  const double _bUdDD102 = t55*vetU_dDD102 - t66*vetU_dD12;
  const double t227 = -_bUdD20*t26 + _bUdDD102;
  const double t75 = f0_of_xx0__DD00*t65;
  const double t77 = (1.0 / t76);
  const double vetU_dDD100 = V0_vetU_dDD100;
  const double _bUdDD100 = t55*vetU_dDD100 - 2.0*t66*vetU_dD10 + vetU1*(2.0*t0*t77 - t75);
  const double t228 = f0_of_xx0__DD00*t55 - t0*t65;
  const double t229 = t0*t77;
  const double t230 = 2.0*t56;
  const double t231 = _gbUU00*(_bUdD10*t230 - _bUdD10*t52 + _bUdDD100 + t228*t83 + t229*vetU1 - t75*vetU1);
  const double t232 = t116*t228;
  const double t233 = _bUdD00*t56;
  const double t234 = _bUdDD101 + t233;
  const double t235 = _gbUU01*(t232 + t234);
  const double t236 = t52*t55*vetU0 - t66*vetU0;
  const double t237 = _gbUU01*(t234 + t236);
  const double t238 = _gbUU11*(_bUdDD111 + 2.0*t156 + t157);
  const double t239 = _bUdD21*t26;
  const double t240 = _bUdDD112 - t151 + t162 - t239;
  const double t241 = _gbUU12*t240;
  const double t242 = _gbUU12*(-t167 + t168*t80 + t168*(-f1_of_xx1*f1_of_xx1__DD11 - t80) + t240);
  const double vetU_dDD122 = V0_vetU_dDD122;
  const double _bUdDD122 = t55*vetU_dDD122;
  const double t243 = _gbUU22*(_bUdD10*t54 + _bUdD11*t26 + _bUdDD122 - t129*t26 + t5*t83 - t80*t83);
  const double t244 = _gbUU01*t173;
  const double t245 = _gbUU11*t175;
  const double t246 = _gbUU12*t177;
  const double t247 = t65*vetU0;
  const double t248 = _bUdD10*t180;
  const double t249 = _bUdD11*t182;
  const double t250 = _AbUU01*t186;
  const double t251 = _GbUDD102*t186;
  const double t252 = _GbUDD112*t186;
  const double t253 = _bUdD12*t204;
  const double t254 = _GbUDD112*t128;
  const double t255 = (Rational_3_4)*_GbUDD101;
  const double t256 = t218*vetU1;
  const double t257 = (Rational_3_4)*_GbUDD102;
  out[8 * Ntot + idx] = f0_of_xx0*(_AbUU02*t251 - _AbUU10*t136 - _AbUU11*t138 - _AbUU12*t140 + _AbUU12*t252 + _AbUU20*t251 + _AbUU21*t252 + _DGU1*t133 + _DGUDD101*t189 + _DGUDD101*t250 + _DGUDD122*t194 + _GbUDD100*t185 + _GbUDD100*t196 - _GbUDD100*t201 + _GbUDD101*t206 + _GbUDD101*t208 + _GbUDD102*t221 + _GbUDD102*t223 + _GbUDD111*t191 + _GbUDD111*t198 - _GbUDD111*t203 + _GbUDD122*t213 - _GbUDD122*t220 + _gbUU01*t146 + (Rational_3_2)*_gbUU02*t227 + _gbUU11*t150 + _gbUU12*t153 - betU1*t247 - eta*t207 + t210*t254 + t211*t254 - t215*t255 - t216*t255 - t217*t254 - t225*t257 - t226*t257 + (Rational_3_4)*t231 + (Rational_3_4)*t235 + (Rational_3_4)*t237 + (Rational_3_4)*t238 + (Rational_3_4)*t241 + (Rational_3_4)*t242 + (Rational_3_4)*t243 - t244 - t245 - t246 - Rational_3_4*t248 - Rational_3_4*t249 - Rational_3_4*t253 - t254*t256) + V0_lin_betU1;
  const double _DGUDD202 = _GbUDD202 + t57;
  const double _DGUDD212 = _GbUDD212 - t59;
  const double _DGU2 = _DGUDD202*t61 + _DGUDD212*t62 + _GbUDD200*_gbUU00 + _GbUDD201*t60 + _GbUDD211*_gbUU11 + _GbUDD222*_gbUU22;
  const double vetU_dDD201 = V0_vetU_dDD201;
  const double _bUdDD201 = f1_of_xx1__D1*t66*t69*vetU2 + t67*vetU_dDD201 - t68*vetU_dD21 - t71*vetU_dD20;
  const double t258 = _bUdD20*t59 + _bUdDD201;
  const double t78 = t58*t75;
  const double vetU_dDD200 = V0_vetU_dDD200;
  const double _bUdDD200 = t67*vetU_dDD200 - 2.0*t68*vetU_dD20 + vetU2*(2.0*t0*t58*t77 - t78);
  const double t259 = _gbUU00*(_bUdD20*t230 - _bUdD20*t52 + _bUdDD200 + t168*t228 + t229*t58*vetU2 - t78*vetU2);
  const double t260 = _bUdD10*t59 + _bUdDD202 + t233;
  const double t261 = _gbUU02*(t232 + t260);
  const double t262 = _gbUU02*(t236 + t260);
  const double vetU_dDD211 = V0_vetU_dDD211;
  const double _bUdDD211 = t67*vetU_dDD211 - 2.0*t71*vetU_dD21 + vetU2*(-f1_of_xx1__DD11*t70 + 2.0*t55*t79*t80);
  const double t263 = f1_of_xx1__DD11*t58 - t147;
  const double t264 = _gbUU11*(_bUdD20*t53 + 2.0*_bUdD21*t59 + _bUdDD211 + t168*t263 + t168 + t55*t79*t80*vetU2);
  const double t265 = _bUdD11*t59 + _bUdDD212 + t156;
  const double t266 = _gbUU12*(t263*t83 + t265);
  const double t267 = _gbUU12*(-t148 + t265 - t83);
  const double t268 = _gbUU22*(_bUdDD222 + 2.0*t151 + 2.0*t162 + t163 + t239);
  const double t269 = _gbUU02*t173;
  const double t270 = _gbUU12*t175;
  const double t271 = _gbUU22*t177;
  const double t272 = _bUdD20*t180;
  const double t273 = _bUdD21*t182;
  const double t274 = _DGUDD202*t186;
  const double t275 = _DGUDD212*t186;
  const double t276 = t128*vetU0;
  const double t277 = _bUdD22*t204;
  const double t278 = _GbUDD212*t128;
  const double t279 = (Rational_3_4)*_GbUDD201;
  const double t280 = (Rational_3_4)*_GbUDD202;
  out[9 * Ntot + idx] = t126*(_AbUU02*t274 + _AbUU12*t275 - _AbUU20*t136 + _AbUU20*t274 - _AbUU21*t138 + _AbUU21*t275 - _AbUU22*t140 + _DGU2*t133 + _GbUDD200*t185 + _GbUDD200*t196 - _GbUDD200*t201 + _GbUDD201*t189 + _GbUDD201*t206 + _GbUDD201*t208 + _GbUDD201*t250 + _GbUDD202*t221 + _GbUDD202*t223 + _GbUDD211*t191 + _GbUDD211*t198 - _GbUDD211*t203 + _GbUDD222*t194 + _GbUDD222*t213 - _GbUDD222*t220 + (Rational_3_2)*_gbUU01*t258 + _gbUU02*t146 + _gbUU12*t150 + _gbUU22*t153 - betU2*t276 - eta*t222 - t118*t212 + t210*t278 + t211*t278 - t215*t279 - t216*t279 - t217*t278 - t225*t280 - t226*t280 - t256*t278 + (Rational_3_4)*t259 + (Rational_3_4)*t261 + (Rational_3_4)*t262 + (Rational_3_4)*t264 + (Rational_3_4)*t266 + (Rational_3_4)*t267 + (Rational_3_4)*t268 - t269 - t270 - t271 - Rational_3_4*t272 - Rational_3_4*t273 - Rational_3_4*t277) + V0_lin_betU2;
  out[10 * Ntot + idx] = -2.0*cf*((Rational_1_6)*_Dbb - Rational_1_6*t112) + V0_lin_cf;
  const double t281 = 2.0*_gbDD01;
  const double t282 = 2.0*_gbDD02;
  const double _trAb = t45 + 2.0*t46 + 2.0*t47 + t48 + 2.0*t49 + t50;
  const double t283 = -Rational_2_3*_Dbb + (Rational_2_3)*_trAb*alpha;
  out[11 * Ntot + idx] = t63*(_bUdD10*t281 + _bUdD20*t282 + _gbDD00*t108 + _gbDD00*t283 - t113 + t116*t13) + V0_lin_hDD00;
  out[12 * Ntot + idx] = t117*(_bUdD00*_gbDD01 + _bUdD01*_gbDD00 + _bUdD10*_gbDD11 + _bUdD11*_gbDD01 + _bUdD20*_gbDD12 + _bUdD21*_gbDD02 + _gbDD01*t283 - t114 + t116*t16) + V0_lin_hDD01;
  out[13 * Ntot + idx] = t119*(_bUdD00*_gbDD02 + _bUdD02*_gbDD00 + _bUdD10*_gbDD12 + _bUdD12*_gbDD01 + _bUdD20*_gbDD22 + _bUdD22*_gbDD02 + _gbDD02*t283 + f0_of_xx0__D0*t20*vetU1 - t115 + t116*t19) + V0_lin_hDD02;
  const double t284 = 2.0*_gbDD12;
  out[14 * Ntot + idx] = t65*(_bUdD01*t281 + _bUdD21*t284 + _gbDD11*t120 + _gbDD11*t283 + t116*t22 - t122) + V0_lin_hDD11;
  out[15 * Ntot + idx] = t128*(_bUdD01*_gbDD02 + _bUdD02*_gbDD01 + _bUdD11*_gbDD12 + _bUdD12*_gbDD11 + _bUdD21*_gbDD22 + _bUdD22*_gbDD12 + _gbDD12*t283 + hDD12*t127 - t123 + t131*t23) + V0_lin_hDD12;
  out[16 * Ntot + idx] = t132*(_bUdD02*t282 + _bUdD12*t284 + _gbDD22*t129 + _gbDD22*t283 + t116*t25 - t130 + t29*t83) + V0_lin_hDD22;
  const double t285 = 2.0*t135;
  const double t286 = 2.0*t137;
  const double t287 = 2.0*t139;
  const double t288 = (Rational_1_3)*t145;
  const double t289 = (Rational_1_3)*t149;
  const double t290 = (Rational_1_3)*t152;
  const double t291 = _AbUU00*t92;
  const double t292 = _GbUDD002*t92;
  const double t293 = _AbUU10*t92;
  const double t294 = _AbUU11*t92;
  const double t295 = _GbUDD012*t92;
  const double t296 = _AbUU22*t92;
  out[17 * Ntot + idx] = f0_of_xx0__D0*(-_AbUU00*t285 - _AbUU01*t286 - _AbUU02*t287 + _AbUU02*t292 + _AbUU12*t295 + _AbUU20*t292 + _AbUU21*t295 + _DGU0*t111 + _DGUDD000*t291 + _DGUDD011*t294 + _DGUDD022*t296 + _GbUDD001*t293 + _gbUU00*t288 + _gbUU01*t289 + _gbUU02*t290 + t154*t62 + t155 + t159 + t161 + t165 + t169 + t171 + t172 - Rational_4_3*t174 - Rational_4_3*t176 - Rational_4_3*t178 - t181 - t183 + t187*t92 - t199*t200 - t205) + V0_lin_lambdaU0;
  const double t297 = _AbUU01*t92;
  const double t298 = _GbUDD102*t92;
  const double t299 = _GbUDD112*t92;
  out[18 * Ntot + idx] = f0_of_xx0*(_AbUU02*t298 - _AbUU10*t285 - _AbUU11*t286 - _AbUU12*t287 + _AbUU12*t299 + _AbUU20*t298 + _AbUU21*t299 + _DGU1*t111 + _DGUDD101*t293 + _DGUDD101*t297 + _DGUDD122*t296 + _GbUDD100*t291 + _GbUDD111*t294 + _gbUU01*t288 + _gbUU11*t289 + _gbUU12*t290 - lambdaU1*t247 + t227*t61 + t231 + t235 + t237 + t238 + t241 + t242 + t243 - Rational_4_3*t244 - Rational_4_3*t245 - Rational_4_3*t246 - t248 - t249 - t253) + V0_lin_lambdaU1;
  const double t300 = _DGUDD202*t92;
  const double t301 = _DGUDD212*t92;
  const double t302 = t118*t132;
  out[19 * Ntot + idx] = t126*(_AbUU02*t300 + _AbUU12*t301 - _AbUU20*t285 + _AbUU20*t300 - _AbUU21*t286 + _AbUU21*t301 - _AbUU22*t287 + _DGU2*t111 + _GbUDD200*t291 + _GbUDD201*t293 + _GbUDD201*t297 + _GbUDD211*t294 + _GbUDD222*t296 + _gbUU02*t288 + _gbUU12*t289 + _gbUU22*t290 - lambdaU2*t276 - lambdaU2*t302 + t258*t60 + t259 + t261 + t262 + t264 + t266 + t267 + t268 - Rational_4_3*t269 - Rational_4_3*t270 - Rational_4_3*t271 - t272 - t273 - t277) + V0_lin_lambdaU2;
  const double t303 = _AbDD01*alpha;
  const double t304 = _AbDD02*alpha;
  const double t305 = _AbDD12*alpha;
  const double t306 = _gbUU01*t106;
  const double t307 = _gbUU02*t106;
  const double t308 = _gbUU12*t106;
  out[20 * Ntot + idx] = _AbDD00*t184 + _AbDD11*t190 + _AbDD22*t193 + _AbUU01*t303 + _AbUU02*t304 + _AbUU10*t303 + _AbUU12*t305 + _AbUU20*t304 + _AbUU21*t305 - _gbUU00*t106*(_adBDD00 + 2.0*t93) - _gbUU11*t106*(_adBDD11 + 2.0*t102) - _gbUU22*t106*(_adBDD22 + _phidD2*t103) + (Rational_1_3)*alpha*(trK*trK) - t306*(_adBDD01 + t96) - t306*(_adBDD01 + t98) - t307*(_adBDD02 + t100) - t307*(_adBDD02 + t101) - t308*(_adBDD12 + t104) - t308*(_adBDD12 + t105) + V0_lin_trK;
  const double t309 = (vetU0*vetU0);
  const double t310 = t309*t63;
  const double t311 = t65*(vetU1*vetU1);
  const double t312 = t132*(vetU2*vetU2);
  const double t313 = 2.0*t116;
  const double t314 = t313*t83;
  const double t315 = 2.0*vetU2;
  const double t316 = t168*t313;
  out[21 * Ntot + idx] = f0_of_xx0__D0*(_GbUDD000*t310 + _GbUDD001*t314 + _GbUDD002*t316 + _GbUDD011*t311 + _GbUDD022*t312 + t179 - t199*t309 + t219*t315) + V0_lin_vetU0;
  const double t317 = t315*vetU1;
  out[22 * Ntot + idx] = f0_of_xx0*(_GbUDD100*t310 + _GbUDD101*t314 + _GbUDD102*t316 + _GbUDD111*t311 + _GbUDD122*t312 + t207 - t247*vetU1 + t254*t317) + V0_lin_vetU1;
  out[23 * Ntot + idx] = t126*(_GbUDD200*t310 + _GbUDD201*t314 + _GbUDD202*t316 + _GbUDD211*t311 + _GbUDD222*t312 + t222 - t276*vetU2 + t278*t317 - t302*vetU2) + V0_lin_vetU2;
    }
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

extern "C" hipError_t launch_bssn_rhs_SinhSpherical_symnone_KO1_fd6_p1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg_ub_mi_xcd(dim3 g, dim3 b, hipStream_t s, const double *in, const double *aux, double *out, const double *rfm0, const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_rhs_SinhSpherical_symnone_KO1_fd6_p1_lb1_sj_L16x4x4x1_d3_dma_rb1_io_pg_ub_mi_xcd_g0, dim3((p.Nx0 - 2 * p.NG + 15) / 16, (p.Nx1 - 2 * p.NG + 3) / 4, (p.Nx2 - 2 * p.NG + 3) / 4), dim3(256), 0, s, in, aux, out, rfm0, rfm1, p);
  return hipGetLastError();
}
