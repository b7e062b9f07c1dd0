// Generated by nrpy_amd/codegen/hip_gen.py -- do not edit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "../bhah_device_types.h"
// ---- constraints candidate k1_lb1_L16x2x2x1_d3_dmo_rb1_io_pg_lr40_di_mi_xcd: 1 kernel(s); Spherical, fd_order=4
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
#define Rational_2_3 (2.0 / 3.0)

// bhah-dma-issue bssn_constraints_Spherical_sym2_KO0_fd4_k1_lb1_L16x2x2x1_d3_dmo_rb1_io_pg_lr40_di_mi_xcd_g0: 0:3 1:3 2:3 3:3 4:3 5:3 6:3 7:3 8:3 9:3 10:3 11:3 12:3 13:3
extern "C" __global__ void __launch_bounds__(64)
bssn_constraints_Spherical_sym2_KO0_fd4_k1_lb1_L16x2x2x1_d3_dmo_rb1_io_pg_lr40_di_mi_xcd_g0(const double *__restrict__ in, const double *__restrict__ aux, double *__restrict__ out,
        const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  __shared__ double sh[1152];
  unsigned bx, by, bz;
  {
    const unsigned gx = gridDim.x, gy = gridDim.y, gz = gridDim.z, n = gx * gy * gz;
    const unsigned h = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const unsigned l = (h & 7u) * (n >> 3) + min((int)(h & 7u), (int)(n & 7u)) + (h >> 3);
    bx = l % gx;
    by = (l / gx) % gy;
    bz = l / (gx * gy);
  }
  // Tile of 16x2x2 interior points; halo box 22x6x2 = 264 values per gridfunction.
  constexpr int BX = 22, BY = 6, NB = 264, NT = 64, NL = 5;
  const int tid = (int)threadIdx.x;
  const int lx = tid % 16, ly = (tid / 16) % 2, lz = tid / 32;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const int o0 = p.NG + (int)bx * 16, o1 = p.NG + (int)by * 2, o2 = p.NG + (int)bz * 2;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned pofs[3];
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const int e = 2 * (tid + NT * j);
    const int ex = e % BX, ey = (e / BX) % BY, ez = e / (BX * BY);
    const int g1 = min(o1 - 2 + ey, p.Nx1 - 1), g2 = min(o2 - 0 + ez, p.Nx2 - 1);
    const int row = (o0 - 2 + (int)s1 * g1 + (int)s2 * g2) & ~1;
    pofs[j] = 8u * (unsigned)min(row + ex, (int)Ntot - 2);
  }
  const int c0b = (lx + 2) + BX * (ly + 2) + BX * BY * (lz + 0);
  const int q0 = (o0 - 2 + (int)s1 * (o1 + ly) + (int)s2 * (o2 + lz + 0)) & 1;
  const int c0 = c0b + q0, c0y = c0b + (q0 ^ ((int)s1 & 1)), c0z = c0b + (q0 ^ ((int)s2 & 1)),
            c0w = c0b + (q0 ^ ((int)(s1 + s2) & 1));
  const double ius0 = p.invdxx0 * (1.0 / 12.0), nius0 = -ius0, ikos0 = p.invdxx0 * (1.0 / 64.0);
  const double ius1 = p.invdxx1 * (1.0 / 12.0), nius1 = -ius1, ikos1 = p.invdxx1 * (1.0 / 64.0);
  const double ius2 = p.invdxx2 * (1.0 / 12.0), nius2 = -ius2, ikos2 = p.invdxx2 * (1.0 / 64.0);
  {
    const char *src = (const char *)(in + 10 * Ntot);
#pragma unroll
    for (int j = 0; j < 3; j++) BHAH_DMA16O(src, pofs[j], sh + 0 + 2 * (NT * j + 64 * wv));
  }
  {
    const char *src = (const char *)(in + 0 * Ntot);
#pragma unroll
    for (int j = 0; j < 3; j++) BHAH_DMA16O(src, pofs[j], sh + 384 + 2 * (NT * j + 64 * wv));
  }
  // ---- cf
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(0);
  double R0_cf_0_0 = sh[c0];
  double R0_cf_0_1 = sh[c0 + 1];
  double R0_cf_0_2 = sh[c0 - 1];
  double R0_cf_0_3 = sh[c0 + 2];
  double R0_cf_0_4 = sh[c0 - 2];
  double R0_cf_0_5 = sh[c0y + 22];
  double R0_cf_0_6 = sh[c0y - 22];
  double R0_cf_0_7 = sh[c0 + 44];
  double R0_cf_0_8 = sh[c0 - 44];
  double R0_cf_0_9 = sh[c0y + 23];
  double R0_cf_0_10 = sh[c0y - 21];
  double R0_cf_0_11 = sh[c0y + 21];
  double R0_cf_0_12 = sh[c0y - 23];
  double R0_cf_0_13 = sh[c0 + 45];
  double R0_cf_0_14 = sh[c0 - 43];
  double R0_cf_0_15 = sh[c0 + 43];
  double R0_cf_0_16 = sh[c0 - 45];
  double R0_cf_0_17 = sh[c0y + 24];
  double R0_cf_0_18 = sh[c0y - 20];
  double R0_cf_0_19 = sh[c0y + 20];
  double R0_cf_0_20 = sh[c0y - 24];
  double R0_cf_0_21 = sh[c0 + 46];
  double R0_cf_0_22 = sh[c0 - 42];
  double R0_cf_0_23 = sh[c0 + 42];
  double R0_cf_0_24 = sh[c0 - 46];
  BHAH_DMA16O((const char *)(in + 1 * Ntot), pofs[0], sh + 768 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_cf_0_0), "+v"(R0_cf_0_1), "+v"(R0_cf_0_2), "+v"(R0_cf_0_3), "+v"(R0_cf_0_4), "+v"(R0_cf_0_5), "+v"(R0_cf_0_6), "+v"(R0_cf_0_7), "+v"(R0_cf_0_8), "+v"(R0_cf_0_9), "+v"(R0_cf_0_10), "+v"(R0_cf_0_11), "+v"(R0_cf_0_12), "+v"(R0_cf_0_13), "+v"(R0_cf_0_14), "+v"(R0_cf_0_15), "+v"(R0_cf_0_16), "+v"(R0_cf_0_17), "+v"(R0_cf_0_18), "+v"(R0_cf_0_19), "+v"(R0_cf_0_20), "+v"(R0_cf_0_21), "+v"(R0_cf_0_22), "+v"(R0_cf_0_23));
  BHAH_DMA16O((const char *)(in + 1 * Ntot), pofs[1], sh + 768 + 2 * (NT * 1 + 64 * wv));
  BHAH_PINS("+v"(R0_cf_0_24));
  double V0_cf = R0_cf_0_0;
  double V0_cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (R0_cf_0_1 - R0_cf_0_2) + (-1.0 / 12.0) * (R0_cf_0_3 - R0_cf_0_4));
  double V0_cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (R0_cf_0_5 - R0_cf_0_6) + (-1.0 / 12.0) * (R0_cf_0_7 - R0_cf_0_8));
  double V0_cf_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * R0_cf_0_0 + (4.0 / 3.0) * (R0_cf_0_1 + R0_cf_0_2) + (-1.0 / 12.0) * (R0_cf_0_3 + R0_cf_0_4));
  double V0_cf_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * R0_cf_0_0 + (4.0 / 3.0) * (R0_cf_0_5 + R0_cf_0_6) + (-1.0 / 12.0) * (R0_cf_0_7 + R0_cf_0_8));
  BHAH_DMA16O((const char *)(in + 1 * Ntot), pofs[2], sh + 768 + 2 * (NT * 2 + 64 * wv));
  double V0_cf_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((R0_cf_0_9 - R0_cf_0_10) - (R0_cf_0_11 - R0_cf_0_12)) + (-1.0 / 18.0) * ((R0_cf_0_13 - R0_cf_0_14) - (R0_cf_0_15 - R0_cf_0_16)) + (-1.0 / 18.0) * ((R0_cf_0_17 - R0_cf_0_18) - (R0_cf_0_19 - R0_cf_0_20)) + (1.0 / 144.0) * ((R0_cf_0_21 - R0_cf_0_22) - (R0_cf_0_23 - R0_cf_0_24)));
  BHAH_PINS("+v"(V0_cf), "+v"(V0_cf_dD0), "+v"(V0_cf_dD1), "+v"(V0_cf_dDD00), "+v"(V0_cf_dDD11), "+v"(V0_cf_dDD01));
  // ---- aDD00
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(1);
  double R0_aDD00_0_0 = sh[c0 + 384];
  double R0_aDD00_0_1 = sh[c0 + 385];
  double R0_aDD00_0_2 = sh[c0 + 383];
  double R0_aDD00_0_3 = sh[c0 + 386];
  double R0_aDD00_0_4 = sh[c0 + 382];
  double R0_aDD00_0_5 = sh[c0y + 406];
  double R0_aDD00_0_6 = sh[c0y + 362];
  double R0_aDD00_0_7 = sh[c0 + 428];
  double R0_aDD00_0_8 = sh[c0 + 340];
  BHAH_DMA16O((const char *)(in + 2 * Ntot), pofs[0], sh + 0 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_aDD00_0_0), "+v"(R0_aDD00_0_1), "+v"(R0_aDD00_0_2), "+v"(R0_aDD00_0_3), "+v"(R0_aDD00_0_4), "+v"(R0_aDD00_0_5), "+v"(R0_aDD00_0_6), "+v"(R0_aDD00_0_7), "+v"(R0_aDD00_0_8));
  BHAH_DMA16O((const char *)(in + 2 * Ntot), pofs[1], sh + 0 + 2 * (NT * 1 + 64 * wv));
  double V0_aDD00 = R0_aDD00_0_0;
  double V0_aDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (R0_aDD00_0_1 - R0_aDD00_0_2) + (-1.0 / 12.0) * (R0_aDD00_0_3 - R0_aDD00_0_4));
  BHAH_DMA16O((const char *)(in + 2 * Ntot), pofs[2], sh + 0 + 2 * (NT * 2 + 64 * wv));
  double V0_aDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (R0_aDD00_0_5 - R0_aDD00_0_6) + (-1.0 / 12.0) * (R0_aDD00_0_7 - R0_aDD00_0_8));
  BHAH_PINS("+v"(V0_aDD00), "+v"(V0_aDD_dD000), "+v"(V0_aDD_dD001));
  // ---- aDD01
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(2);
  double R0_aDD01_0_0 = sh[c0 + 768];
  double R0_aDD01_0_1 = sh[c0 + 769];
  double R0_aDD01_0_2 = sh[c0 + 767];
  double R0_aDD01_0_3 = sh[c0 + 770];
  double R0_aDD01_0_4 = sh[c0 + 766];
  double R0_aDD01_0_5 = sh[c0y + 790];
  double R0_aDD01_0_6 = sh[c0y + 746];
  double R0_aDD01_0_7 = sh[c0 + 812];
  double R0_aDD01_0_8 = sh[c0 + 724];
  BHAH_DMA16O((const char *)(in + 3 * Ntot), pofs[0], sh + 384 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_aDD01_0_0), "+v"(R0_aDD01_0_1), "+v"(R0_aDD01_0_2), "+v"(R0_aDD01_0_3), "+v"(R0_aDD01_0_4), "+v"(R0_aDD01_0_5), "+v"(R0_aDD01_0_6), "+v"(R0_aDD01_0_7), "+v"(R0_aDD01_0_8));
  BHAH_DMA16O((const char *)(in + 3 * Ntot), pofs[1], sh + 384 + 2 * (NT * 1 + 64 * wv));
  double V0_aDD01 = R0_aDD01_0_0;
  double V0_aDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (R0_aDD01_0_1 - R0_aDD01_0_2) + (-1.0 / 12.0) * (R0_aDD01_0_3 - R0_aDD01_0_4));
  BHAH_DMA16O((const char *)(in + 3 * Ntot), pofs[2], sh + 384 + 2 * (NT * 2 + 64 * wv));
  double V0_aDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (R0_aDD01_0_5 - R0_aDD01_0_6) + (-1.0 / 12.0) * (R0_aDD01_0_7 - R0_aDD01_0_8));
  BHAH_PINS("+v"(V0_aDD01), "+v"(V0_aDD_dD010), "+v"(V0_aDD_dD011));
  // ---- aDD02
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(3);
  double R0_aDD02_0_0 = sh[c0];
  double R0_aDD02_0_1 = sh[c0 + 1];
  double R0_aDD02_0_2 = sh[c0 - 1];
  double R0_aDD02_0_3 = sh[c0 + 2];
  double R0_aDD02_0_4 = sh[c0 - 2];
  double R0_aDD02_0_5 = sh[c0y + 22];
  double R0_aDD02_0_6 = sh[c0y - 22];
  double R0_aDD02_0_7 = sh[c0 + 44];
  double R0_aDD02_0_8 = sh[c0 - 44];
  BHAH_DMA16O((const char *)(in + 4 * Ntot), pofs[0], sh + 768 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_aDD02_0_0), "+v"(R0_aDD02_0_1), "+v"(R0_aDD02_0_2), "+v"(R0_aDD02_0_3), "+v"(R0_aDD02_0_4), "+v"(R0_aDD02_0_5), "+v"(R0_aDD02_0_6), "+v"(R0_aDD02_0_7), "+v"(R0_aDD02_0_8));
  BHAH_DMA16O((const char *)(in + 4 * Ntot), pofs[1], sh + 768 + 2 * (NT * 1 + 64 * wv));
  double V0_aDD02 = R0_aDD02_0_0;
  double V0_aDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (R0_aDD02_0_1 - R0_aDD02_0_2) + (-1.0 / 12.0) * (R0_aDD02_0_3 - R0_aDD02_0_4));
  BHAH_DMA16O((const char *)(in + 4 * Ntot), pofs[2], sh + 768 + 2 * (NT * 2 + 64 * wv));
  double V0_aDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (R0_aDD02_0_5 - R0_aDD02_0_6) + (-1.0 / 12.0) * (R0_aDD02_0_7 - R0_aDD02_0_8));
  BHAH_PINS("+v"(V0_aDD02), "+v"(V0_aDD_dD020), "+v"(V0_aDD_dD021));
  // ---- aDD11
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(4);
  double R0_aDD11_0_0 = sh[c0 + 384];
  double R0_aDD11_0_1 = sh[c0 + 385];
  double R0_aDD11_0_2 = sh[c0 + 383];
  double R0_aDD11_0_3 = sh[c0 + 386];
  double R0_aDD11_0_4 = sh[c0 + 382];
  double R0_aDD11_0_5 = sh[c0y + 406];
  double R0_aDD11_0_6 = sh[c0y + 362];
  double R0_aDD11_0_7 = sh[c0 + 428];
  double R0_aDD11_0_8 = sh[c0 + 340];
  BHAH_DMA16O((const char *)(in + 5 * Ntot), pofs[0], sh + 0 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_aDD11_0_0), "+v"(R0_aDD11_0_1), "+v"(R0_aDD11_0_2), "+v"(R0_aDD11_0_3), "+v"(R0_aDD11_0_4), "+v"(R0_aDD11_0_5), "+v"(R0_aDD11_0_6), "+v"(R0_aDD11_0_7), "+v"(R0_aDD11_0_8));
  BHAH_DMA16O((const char *)(in + 5 * Ntot), pofs[1], sh + 0 + 2 * (NT * 1 + 64 * wv));
  double V0_aDD11 = R0_aDD11_0_0;
  double V0_aDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (R0_aDD11_0_1 - R0_aDD11_0_2) + (-1.0 / 12.0) * (R0_aDD11_0_3 - R0_aDD11_0_4));
  BHAH_DMA16O((const char *)(in + 5 * Ntot), pofs[2], sh + 0 + 2 * (NT * 2 + 64 * wv));
  double V0_aDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (R0_aDD11_0_5 - R0_aDD11_0_6) + (-1.0 / 12.0) * (R0_aDD11_0_7 - R0_aDD11_0_8));
  BHAH_PINS("+v"(V0_aDD11), "+v"(V0_aDD_dD110), "+v"(V0_aDD_dD111));
  // ---- aDD12
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(5);
  double R0_aDD12_0_0 = sh[c0 + 768];
  double R0_aDD12_0_1 = sh[c0 + 769];
  double R0_aDD12_0_2 = sh[c0 + 767];
  double R0_aDD12_0_3 = sh[c0 + 770];
  double R0_aDD12_0_4 = sh[c0 + 766];
  double R0_aDD12_0_5 = sh[c0y + 790];
  double R0_aDD12_0_6 = sh[c0y + 746];
  double R0_aDD12_0_7 = sh[c0 + 812];
  double R0_aDD12_0_8 = sh[c0 + 724];
  BHAH_DMA16O((const char *)(in + 11 * Ntot), pofs[0], sh + 384 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_aDD12_0_0), "+v"(R0_aDD12_0_1), "+v"(R0_aDD12_0_2), "+v"(R0_aDD12_0_3), "+v"(R0_aDD12_0_4), "+v"(R0_aDD12_0_5), "+v"(R0_aDD12_0_6), "+v"(R0_aDD12_0_7), "+v"(R0_aDD12_0_8));
  BHAH_DMA16O((const char *)(in + 11 * Ntot), pofs[1], sh + 384 + 2 * (NT * 1 + 64 * wv));
  double V0_aDD12 = R0_aDD12_0_0;
  double V0_aDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (R0_aDD12_0_1 - R0_aDD12_0_2) + (-1.0 / 12.0) * (R0_aDD12_0_3 - R0_aDD12_0_4));
  BHAH_DMA16O((const char *)(in + 11 * Ntot), pofs[2], sh + 384 + 2 * (NT * 2 + 64 * wv));
  double V0_aDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (R0_aDD12_0_5 - R0_aDD12_0_6) + (-1.0 / 12.0) * (R0_aDD12_0_7 - R0_aDD12_0_8));
  BHAH_PINS("+v"(V0_aDD12), "+v"(V0_aDD_dD120), "+v"(V0_aDD_dD121));
  // ---- aDD22
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(6);
  double R0_aDD22_0_0 = sh[c0];
  double R0_aDD22_0_1 = sh[c0 + 1];
  double R0_aDD22_0_2 = sh[c0 - 1];
  double R0_aDD22_0_3 = sh[c0 + 2];
  double R0_aDD22_0_4 = sh[c0 - 2];
  double R0_aDD22_0_5 = sh[c0y + 22];
  double R0_aDD22_0_6 = sh[c0y - 22];
  double R0_aDD22_0_7 = sh[c0 + 44];
  double R0_aDD22_0_8 = sh[c0 - 44];
  BHAH_DMA16O((const char *)(in + 12 * Ntot), pofs[0], sh + 768 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_aDD22_0_0), "+v"(R0_aDD22_0_1), "+v"(R0_aDD22_0_2), "+v"(R0_aDD22_0_3), "+v"(R0_aDD22_0_4), "+v"(R0_aDD22_0_5), "+v"(R0_aDD22_0_6), "+v"(R0_aDD22_0_7), "+v"(R0_aDD22_0_8));
  BHAH_DMA16O((const char *)(in + 12 * Ntot), pofs[1], sh + 768 + 2 * (NT * 1 + 64 * wv));
  double V0_aDD22 = R0_aDD22_0_0;
  double V0_aDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (R0_aDD22_0_1 - R0_aDD22_0_2) + (-1.0 / 12.0) * (R0_aDD22_0_3 - R0_aDD22_0_4));
  BHAH_DMA16O((const char *)(in + 12 * Ntot), pofs[2], sh + 768 + 2 * (NT * 2 + 64 * wv));
  double V0_aDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (R0_aDD22_0_5 - R0_aDD22_0_6) + (-1.0 / 12.0) * (R0_aDD22_0_7 - R0_aDD22_0_8));
  BHAH_PINS("+v"(V0_aDD22), "+v"(V0_aDD_dD220), "+v"(V0_aDD_dD221));
  // ---- hDD00
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(7);
  double R0_hDD00_0_0 = sh[c0 + 384];
  double R0_hDD00_0_1 = sh[c0 + 385];
  double R0_hDD00_0_2 = sh[c0 + 383];
  double R0_hDD00_0_3 = sh[c0 + 386];
  double R0_hDD00_0_4 = sh[c0 + 382];
  double R0_hDD00_0_5 = sh[c0y + 406];
  double R0_hDD00_0_6 = sh[c0y + 362];
  double R0_hDD00_0_7 = sh[c0 + 428];
  double R0_hDD00_0_8 = sh[c0 + 340];
  BHAH_DMA16O((const char *)(in + 13 * Ntot), pofs[0], sh + 0 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_hDD00_0_0), "+v"(R0_hDD00_0_1), "+v"(R0_hDD00_0_2), "+v"(R0_hDD00_0_3), "+v"(R0_hDD00_0_4), "+v"(R0_hDD00_0_5), "+v"(R0_hDD00_0_6), "+v"(R0_hDD00_0_7), "+v"(R0_hDD00_0_8));
  BHAH_DMA16O((const char *)(in + 13 * Ntot), pofs[1], sh + 0 + 2 * (NT * 1 + 64 * wv));
  double V0_hDD00 = R0_hDD00_0_0;
  double V0_hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (R0_hDD00_0_1 - R0_hDD00_0_2) + (-1.0 / 12.0) * (R0_hDD00_0_3 - R0_hDD00_0_4));
  BHAH_DMA16O((const char *)(in + 13 * Ntot), pofs[2], sh + 0 + 2 * (NT * 2 + 64 * wv));
  double V0_hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (R0_hDD00_0_5 - R0_hDD00_0_6) + (-1.0 / 12.0) * (R0_hDD00_0_7 - R0_hDD00_0_8));
  BHAH_PINS("+v"(V0_hDD00), "+v"(V0_hDD_dD000), "+v"(V0_hDD_dD001));
  // ---- hDD01
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(8);
  double R0_hDD01_0_0 = sh[c0 + 768];
  double R0_hDD01_0_1 = sh[c0 + 769];
  double R0_hDD01_0_2 = sh[c0 + 767];
  double R0_hDD01_0_3 = sh[c0 + 770];
  double R0_hDD01_0_4 = sh[c0 + 766];
  double R0_hDD01_0_5 = sh[c0y + 790];
  double R0_hDD01_0_6 = sh[c0y + 746];
  double R0_hDD01_0_7 = sh[c0 + 812];
  double R0_hDD01_0_8 = sh[c0 + 724];
  BHAH_DMA16O((const char *)(in + 14 * Ntot), pofs[0], sh + 384 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_hDD01_0_0), "+v"(R0_hDD01_0_1), "+v"(R0_hDD01_0_2), "+v"(R0_hDD01_0_3), "+v"(R0_hDD01_0_4), "+v"(R0_hDD01_0_5), "+v"(R0_hDD01_0_6), "+v"(R0_hDD01_0_7), "+v"(R0_hDD01_0_8));
  BHAH_DMA16O((const char *)(in + 14 * Ntot), pofs[1], sh + 384 + 2 * (NT * 1 + 64 * wv));
  double V0_hDD01 = R0_hDD01_0_0;
  double V0_hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (R0_hDD01_0_1 - R0_hDD01_0_2) + (-1.0 / 12.0) * (R0_hDD01_0_3 - R0_hDD01_0_4));
  BHAH_DMA16O((const char *)(in + 14 * Ntot), pofs[2], sh + 384 + 2 * (NT * 2 + 64 * wv));
  double V0_hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (R0_hDD01_0_5 - R0_hDD01_0_6) + (-1.0 / 12.0) * (R0_hDD01_0_7 - R0_hDD01_0_8));
  BHAH_PINS("+v"(V0_hDD01), "+v"(V0_hDD_dD010), "+v"(V0_hDD_dD011));
  // ---- hDD02
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(9);
  double R0_hDD02_0_0 = sh[c0];
  double R0_hDD02_0_1 = sh[c0 + 1];
  double R0_hDD02_0_2 = sh[c0 - 1];
  double R0_hDD02_0_3 = sh[c0 + 2];
  double R0_hDD02_0_4 = sh[c0 - 2];
  double R0_hDD02_0_5 = sh[c0y + 22];
  double R0_hDD02_0_6 = sh[c0y - 22];
  double R0_hDD02_0_7 = sh[c0 + 44];
  double R0_hDD02_0_8 = sh[c0 - 44];
  BHAH_DMA16O((const char *)(in + 15 * Ntot), pofs[0], sh + 768 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_hDD02_0_0), "+v"(R0_hDD02_0_1), "+v"(R0_hDD02_0_2), "+v"(R0_hDD02_0_3), "+v"(R0_hDD02_0_4), "+v"(R0_hDD02_0_5), "+v"(R0_hDD02_0_6), "+v"(R0_hDD02_0_7), "+v"(R0_hDD02_0_8));
  BHAH_DMA16O((const char *)(in + 15 * Ntot), pofs[1], sh + 768 + 2 * (NT * 1 + 64 * wv));
  double V0_hDD02 = R0_hDD02_0_0;
  double V0_hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (R0_hDD02_0_1 - R0_hDD02_0_2) + (-1.0 / 12.0) * (R0_hDD02_0_3 - R0_hDD02_0_4));
  BHAH_DMA16O((const char *)(in + 15 * Ntot), pofs[2], sh + 768 + 2 * (NT * 2 + 64 * wv));
  double V0_hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (R0_hDD02_0_5 - R0_hDD02_0_6) + (-1.0 / 12.0) * (R0_hDD02_0_7 - R0_hDD02_0_8));
  BHAH_PINS("+v"(V0_hDD02), "+v"(V0_hDD_dD020), "+v"(V0_hDD_dD021));
  // ---- hDD11
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(10);
  double R0_hDD11_0_0 = sh[c0 + 384];
  double R0_hDD11_0_1 = sh[c0 + 385];
  double R0_hDD11_0_2 = sh[c0 + 383];
  double R0_hDD11_0_3 = sh[c0 + 386];
  double R0_hDD11_0_4 = sh[c0 + 382];
  double R0_hDD11_0_5 = sh[c0y + 406];
  double R0_hDD11_0_6 = sh[c0y + 362];
  double R0_hDD11_0_7 = sh[c0 + 428];
  double R0_hDD11_0_8 = sh[c0 + 340];
  BHAH_DMA16O((const char *)(in + 16 * Ntot), pofs[0], sh + 0 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_hDD11_0_0), "+v"(R0_hDD11_0_1), "+v"(R0_hDD11_0_2), "+v"(R0_hDD11_0_3), "+v"(R0_hDD11_0_4), "+v"(R0_hDD11_0_5), "+v"(R0_hDD11_0_6), "+v"(R0_hDD11_0_7), "+v"(R0_hDD11_0_8));
  BHAH_DMA16O((const char *)(in + 16 * Ntot), pofs[1], sh + 0 + 2 * (NT * 1 + 64 * wv));
  double V0_hDD11 = R0_hDD11_0_0;
  double V0_hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (R0_hDD11_0_1 - R0_hDD11_0_2) + (-1.0 / 12.0) * (R0_hDD11_0_3 - R0_hDD11_0_4));
  BHAH_DMA16O((const char *)(in + 16 * Ntot), pofs[2], sh + 0 + 2 * (NT * 2 + 64 * wv));
  double V0_hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (R0_hDD11_0_5 - R0_hDD11_0_6) + (-1.0 / 12.0) * (R0_hDD11_0_7 - R0_hDD11_0_8));
  BHAH_PINS("+v"(V0_hDD11), "+v"(V0_hDD_dD110), "+v"(V0_hDD_dD111));
  // ---- hDD12
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(11);
  double R0_hDD12_0_0 = sh[c0 + 768];
  double R0_hDD12_0_1 = sh[c0 + 769];
  double R0_hDD12_0_2 = sh[c0 + 767];
  double R0_hDD12_0_3 = sh[c0 + 770];
  double R0_hDD12_0_4 = sh[c0 + 766];
  double R0_hDD12_0_5 = sh[c0y + 790];
  double R0_hDD12_0_6 = sh[c0y + 746];
  double R0_hDD12_0_7 = sh[c0 + 812];
  double R0_hDD12_0_8 = sh[c0 + 724];
  BHAH_DMA16O((const char *)(in + 20 * Ntot), pofs[0], sh + 384 + 2 * (NT * 0 + 64 * wv));
  BHAH_PINS("+v"(R0_hDD12_0_0), "+v"(R0_hDD12_0_1), "+v"(R0_hDD12_0_2), "+v"(R0_hDD12_0_3), "+v"(R0_hDD12_0_4), "+v"(R0_hDD12_0_5), "+v"(R0_hDD12_0_6), "+v"(R0_hDD12_0_7), "+v"(R0_hDD12_0_8));
  BHAH_DMA16O((const char *)(in + 20 * Ntot), pofs[1], sh + 384 + 2 * (NT * 1 + 64 * wv));
  double V0_hDD12 = R0_hDD12_0_0;
  double V0_hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (R0_hDD12_0_1 - R0_hDD12_0_2) + (-1.0 / 12.0) * (R0_hDD12_0_3 - R0_hDD12_0_4));
  BHAH_DMA16O((const char *)(in + 20 * Ntot), pofs[2], sh + 384 + 2 * (NT * 2 + 64 * wv));
  double V0_hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (R0_hDD12_0_5 - R0_hDD12_0_6) + (-1.0 / 12.0) * (R0_hDD12_0_7 - R0_hDD12_0_8));
  BHAH_PINS("+v"(V0_hDD12), "+v"(V0_hDD_dD120), "+v"(V0_hDD_dD121));
  // ---- hDD22
  BHAH_VMWAIT(3);
  BHAH_BARRIER_PHASE(12);
  double R0_hDD22_0_0 = sh[c0];
  double R0_hDD22_0_1 = sh[c0 + 1];
  double R0_hDD22_0_2 = sh[c0 - 1];
  double R0_hDD22_0_3 = sh[c0 + 2];
  double R0_hDD22_0_4 = sh[c0 - 2];
  double R0_hDD22_0_5 = sh[c0y + 22];
  double R0_hDD22_0_6 = sh[c0y - 22];
  double R0_hDD22_0_7 = sh[c0 + 44];
  double R0_hDD22_0_8 = sh[c0 - 44];
  BHAH_PINS("+v"(R0_hDD22_0_0), "+v"(R0_hDD22_0_1), "+v"(R0_hDD22_0_2), "+v"(R0_hDD22_0_3), "+v"(R0_hDD22_0_4), "+v"(R0_hDD22_0_5), "+v"(R0_hDD22_0_6), "+v"(R0_hDD22_0_7), "+v"(R0_hDD22_0_8));
  double V0_hDD22 = R0_hDD22_0_0;
  double V0_hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (R0_hDD22_0_1 - R0_hDD22_0_2) + (-1.0 / 12.0) * (R0_hDD22_0_3 - R0_hDD22_0_4));
  double V0_hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (R0_hDD22_0_5 - R0_hDD22_0_6) + (-1.0 / 12.0) * (R0_hDD22_0_7 - R0_hDD22_0_8));
  BHAH_PINS("+v"(V0_hDD22), "+v"(V0_hDD_dD220), "+v"(V0_hDD_dD221));
  // ---- trK
  BHAH_VMWAIT(0);
  BHAH_BARRIER_PHASE(13);
  double R0_trK_0_0 = sh[c0 + 384];
  double R0_trK_0_1 = sh[c0 + 385];
  double R0_trK_0_2 = sh[c0 + 383];
  double R0_trK_0_3 = sh[c0 + 386];
  double R0_trK_0_4 = sh[c0 + 382];
  double R0_trK_0_5 = sh[c0y + 406];
  double R0_trK_0_6 = sh[c0y + 362];
  double R0_trK_0_7 = sh[c0 + 428];
  double R0_trK_0_8 = sh[c0 + 340];
  BHAH_PINS("+v"(R0_trK_0_0), "+v"(R0_trK_0_1), "+v"(R0_trK_0_2), "+v"(R0_trK_0_3), "+v"(R0_trK_0_4), "+v"(R0_trK_0_5), "+v"(R0_trK_0_6), "+v"(R0_trK_0_7), "+v"(R0_trK_0_8));
  double V0_trK = R0_trK_0_0;
  double V0_trK_dD0 = p.invdxx0 * ((2.0 / 3.0) * (R0_trK_0_1 - R0_trK_0_2) + (-1.0 / 12.0) * (R0_trK_0_3 - R0_trK_0_4));
  double V0_trK_dD1 = p.invdxx1 * ((2.0 / 3.0) * (R0_trK_0_5 - R0_trK_0_6) + (-1.0 / 12.0) * (R0_trK_0_7 - R0_trK_0_8));
  BHAH_PINS("+v"(V0_trK), "+v"(V0_trK_dD0), "+v"(V0_trK_dD1));
  {
    const int i0 = o0 + lx, i1 = o1 + ly, i2 = o2 + lz + 0;
    if (i0 < p.Nx0 - p.NG && i1 < p.Nx1 - p.NG && i2 < p.Nx2 - p.NG) {
      const long idx = i0 + s1 * i1 + s2 * i2;
  const double cf = V0_cf;
  const double t41 = (cf*cf);
  const double t100 = (1.0 / t41);
  const double t101 = 2.0*t100;
  const double f0_of_xx0 = rfm0[i0];
  const double t0 = (f0_of_xx0*f0_of_xx0);
  const double hDD11 = V0_hDD11;
  const double t1 = hDD11*t0 + t0;
  const double hDD00 = V0_hDD00;
  const double t10 = hDD00 + 1.0;
  const double f1_of_xx1 = rfm1[i1];
  const double t2 = (f1_of_xx1*f1_of_xx1);
  const double t3 = t0*t2;
  const double hDD02 = V0_hDD02;
  const double t11 = (hDD02*hDD02)*t3;
  const double hDD22 = V0_hDD22;
  const double t4 = hDD22*t3 + t3;
  const double t5 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double hDD12 = V0_hDD12;
  const double t6 = (hDD12*hDD12)*t2*t5;
  const double hDD01 = V0_hDD01;
  const double t9 = (hDD01*hDD01)*t0;
  const double t12 = 2.0*hDD01*hDD02*hDD12*t2*t5 + t1*t10*t4 - t1*t11 - t10*t6 - t4*t9;
  const double t13 = (1.0 / (t12*t12));
  const double aDD00 = V0_aDD00;
  const double t14 = aDD00*t13;
  const double t17 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t18 = -f0_of_xx0*hDD01*t4 + hDD02*hDD12*t17*t2;
  const double t19 = (t18*t18);
  const double t102 = t14*t19;
  const double t43 = t10*t4 - t11;
  const double t103 = t13*(t43*t43);
  const double aDD11 = V0_aDD11;
  const double t16 = aDD11*t0;
  const double t104 = t103*t16;
  const double t38 = f1_of_xx1*t0;
  const double t45 = hDD12*t38;
  const double t46 = hDD01*hDD02*t38 - t10*t45;
  const double t105 = t13*(t46*t46);
  const double aDD22 = V0_aDD22;
  const double t27 = aDD22*t3;
  const double t106 = t105*t27;
  const double t107 = t13*t43;
  const double t108 = t107*t18;
  const double t109 = t13*t46;
  const double t110 = t109*t18;
  const double t111 = t107*t46;
  const double t7 = t1*t4 - t6;
  const double t112 = t14*t7;
  const double t113 = t112*t18;
  const double aDD01 = V0_aDD01;
  const double t114 = aDD01*f0_of_xx0;
  const double t20 = t13*t19;
  const double t115 = t114*t20;
  const double t116 = t107*t7;
  const double t117 = t114*t116;
  const double t118 = t108*t16;
  const double aDD02 = V0_aDD02;
  const double t34 = aDD02*f1_of_xx1;
  const double t119 = f0_of_xx0*t34;
  const double t31 = t13*t7;
  const double t120 = t31*t46;
  const double t121 = t119*t120;
  const double t22 = f1_of_xx1*hDD12;
  const double t23 = f0_of_xx0*f1_of_xx1;
  const double t24 = hDD01*t17*t22 - hDD02*t1*t23;
  const double t36 = t18*t24;
  const double t37 = t13*t36;
  const double t122 = t119*t37;
  const double aDD12 = V0_aDD12;
  const double t123 = aDD12*t38;
  const double t124 = t107*t24;
  const double t125 = t123*t124;
  const double t126 = t110*t123;
  const double t127 = t109*t24;
  const double t128 = t127*t27;
  const double t44 = t1*t10 - t9;
  const double t129 = (t44*t44);
  const double t130 = t13*t44;
  const double t131 = t130*t24;
  const double t132 = t130*t46;
  const double t133 = t112*t24;
  const double t134 = t114*t120;
  const double t135 = t114*t37;
  const double t25 = (t24*t24);
  const double t26 = t13*t25;
  const double t136 = t119*t26;
  const double t137 = t110*t16;
  const double t138 = t130*t7;
  const double t139 = t119*t138;
  const double t140 = t130*t18;
  const double t141 = t123*t140;
  const double t142 = t123*t127;
  const double t143 = t131*t27;
  const double t144 = t14*t36;
  const double t145 = t114*t124;
  const double t146 = t110*t114;
  const double t147 = t111*t16;
  const double t148 = t105*t123;
  const double t149 = t119*t140;
  const double t8 = (t7*t7);
  const double t15 = t14*t8;
  const double t150 = t119*t127;
  const double t151 = t130*t43;
  const double t152 = t123*t151;
  const double t153 = t132*t27;
  const double t21 = t16*t20;
  const double t28 = t26*t27;
  const double t29 = 2.0*f0_of_xx0;
  const double t30 = aDD01*t29;
  const double t32 = t18*t31;
  const double t33 = t24*t31;
  const double t35 = t29*t34;
  const double t39 = 2.0*t38;
  const double t40 = aDD12*t39;
  const double t42 = (1.0 / t12);
  const double t50 = t42*t7;
  const double t47 = t2*t29;
  const double hDD_dD220 = V0_hDD_dD220;
  const double t48 = hDD22*t47 + hDD_dD220*t3 + t47;
  const double t49 = -t48;
  const double t51 = (Rational_1_2)*t50;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t52 = f1_of_xx1*f1_of_xx1__D1;
  const double t53 = 2.0*t0*t52;
  const double hDD_dD221 = V0_hDD_dD221;
  const double t54 = hDD22*t53 + hDD_dD221*t3 + t53;
  const double t55 = -t54;
  const double t56 = (Rational_1_2)*t42;
  const double t57 = t18*t56;
  const double t58 = t49*t51 + t55*t57;
  const double t59 = (1.0 / cf);
  const double cf_dD0 = V0_cf_dD0;
  const double t60 = (Rational_1_2)*cf_dD0*t59;
  const double t61 = t42*t43;
  const double t62 = (Rational_1_2)*t61;
  const double t63 = t49*t57 + t55*t62;
  const double t64 = (Rational_1_2)*t59;
  const double cf_dD1 = V0_cf_dD1;
  const double t65 = cf_dD1*t64;
  const double t66 = t42*t44;
  const double t67 = (cf_dD1*cf_dD1);
  const double hDD_dD110 = V0_hDD_dD110;
  const double t68 = hDD11*t29 + hDD_dD110*t0 + t29;
  const double hDD_dD011 = V0_hDD_dD011;
  const double t69 = 2.0*f0_of_xx0*hDD_dD011 - t68;
  const double t70 = f1_of_xx1__D1*t0;
  const double hDD_dD121 = V0_hDD_dD121;
  const double t71 = 2.0*hDD12*t70 + hDD_dD121*t39;
  const double t72 = t56*t71;
  const double hDD_dD111 = V0_hDD_dD111;
  const double t73 = hDD_dD111*t0;
  const double t74 = t24*t72 + t51*t69 + t57*t73;
  const double t75 = t46*t72 + t57*t69 + t62*t73;
  const double t76 = (cf_dD0*cf_dD0);
  const double t77 = f1_of_xx1*hDD02;
  const double t78 = f1_of_xx1*t29;
  const double hDD_dD020 = V0_hDD_dD020;
  const double t79 = hDD_dD020*t78 + 2.0*t77;
  const double t80 = t56*t79;
  const double hDD_dD001 = V0_hDD_dD001;
  const double hDD_dD010 = V0_hDD_dD010;
  const double t81 = 2.0*hDD01 - hDD_dD001 + hDD_dD010*t29;
  const double hDD_dD000 = V0_hDD_dD000;
  const double t82 = hDD_dD000*t51 + t24*t80 + t57*t81;
  const double t83 = hDD_dD000*t57 + t46*t80 + t62*t81;
  const double hDD_dD120 = V0_hDD_dD120;
  const double t84 = hDD_dD120*t38 + t22*t29;
  const double hDD_dD021 = V0_hDD_dD021;
  const double t85 = -f0_of_xx0*f1_of_xx1*hDD_dD021 - f0_of_xx0*f1_of_xx1__D1*hDD02 + t84;
  const double t86 = -Rational_1_2*t85;
  const double t87 = t54*t56;
  const double t88 = t24*t87 + t50*t86;
  const double t89 = t18*t42;
  const double t90 = t46*t87 + t86*t89;
  const double t91 = 16.0*t42;
  const double t92 = t48*t56;
  const double t93 = t24*t92 + t57*t85;
  const double t94 = t46*t92 + t62*t85;
  const double t95 = f0_of_xx0*f1_of_xx1__D1;
  const double t96 = hDD02*t95 + hDD_dD021*t23 + t84;
  const double t97 = t56*t96;
  const double t98 = hDD_dD001*t51 + t24*t97 + t57*t68;
  const double t99 = hDD_dD001*t57 + t46*t97 + t62*t68;
  const double RbarDD00 = aux[0 * Ntot + idx];
  const double RbarDD01 = aux[1 * Ntot + idx];
  const double RbarDD02 = aux[2 * Ntot + idx];
  const double RbarDD11 = aux[3 * Ntot + idx];
  const double RbarDD12 = aux[4 * Ntot + idx];
  const double RbarDD22 = aux[5 * Ntot + idx];
  const double cf_dDD00 = V0_cf_dDD00;
  const double cf_dDD01 = V0_cf_dDD01;
  const double cf_dDD11 = V0_cf_dDD11;
  const double trK = V0_trK;
  out[0 * Ntot + idx] = -aDD00*(t15 + t21 + t28 + t30*t32 + t33*t35 + t37*t40) - t16*(t102 + t104 + t106 + t108*t30 + t110*t35 + t111*t40) - t27*(t105*t16 + t127*t30 + t129*t13*t27 + t131*t35 + t132*t40 + t14*t25) - t30*(t113 + t115 + t117 + t118 + t121 + t122 + t125 + t126 + t128) - t35*(t133 + t134 + t135 + t136 + t137 + t139 + t141 + t142 + t143) - t40*(t144 + t145 + t146 + t147 + t148 + t149 + t150 + t152 + t153) + t41*(RbarDD00*t42*t7 + 2.0*RbarDD01*t18*t42 + 2.0*RbarDD02*t24*t42 + RbarDD11*t42*t43 + 2.0*RbarDD12*t42*t46 + RbarDD22*t42*t44 - 4.0*cf_dD0*cf_dD1*t100*t89 - t101*t50*t76 - t101*t61*t67 - t24*t91*(t60*t93 + t65*t94) - t46*t91*(t60*t88 + t65*t90) - 8.0*t50*(t60*t82 + t64*(-cf_dDD00 + t59*t76) + t65*t83) - 8.0*t61*(t60*t74 + t64*(-cf_dDD11 + t59*t67) + t65*t75) - 8.0*t66*(t58*t60 + t63*t65) - 16.0*t89*(t60*t98 + t64*(cf_dD0*cf_dD1*t59 - cf_dDD01) + t65*t99)) + (Rational_2_3)*(trK*trK);
  const double t154 = -t82;
  const double t155 = -t83;
  const double t156 = t24*t56;
  const double t157 = (Rational_1_2)*t66;
  const double t158 = t46*t56;
  const double t159 = hDD_dD000*t156 + t157*t79 + t158*t81;
  const double t160 = -t159;
  const double aDD_dD000 = V0_aDD_dD000;
  const double t161 = t13*(aDD00*t154 - aDD00*t82 + aDD_dD000 + t114*t155 - t114*t83 - t119*t159 + t119*t160);
  const double t162 = -t74;
  const double aDD_dD011 = V0_aDD_dD011;
  const double t163 = aDD_dD011*f0_of_xx0;
  const double t164 = -t75;
  const double t165 = t156*t69 + t157*t71 + t158*t73;
  const double t166 = -t165;
  const double t167 = hDD_dD001*t156 + t157*t96 + t158*t68;
  const double t168 = -t114*t98 - t123*t167 - t16*t99;
  const double t169 = aDD00*t162 + t114*t164 + t119*t166 + t163 + t168;
  const double t170 = -t98;
  const double t171 = -t99;
  const double t172 = -t167;
  const double t173 = t114*t170 + t123*t172 + t16*t171;
  const double aDD_dD110 = V0_aDD_dD110;
  const double t174 = aDD11*t29 + aDD_dD110*t0 + t168 + t173;
  const double t175 = -t58;
  const double t176 = -t63;
  const double t177 = t156*t49 + t158*t55;
  const double t178 = -t177;
  const double t179 = t157*t48 + t158*t85;
  const double t180 = -t119*t93 - t123*t94 - t179*t27;
  const double t181 = aDD00*t175 + t114*t176 + t119*t178 + t180;
  const double t182 = -t93;
  const double t183 = -t94;
  const double t184 = -t179;
  const double aDD_dD220 = V0_aDD_dD220;
  const double t185 = aDD22*t47 + aDD_dD220*t3 + t119*t182 + t123*t183 + t180 + t184*t27;
  const double trK_dD0 = V0_trK_dD0;
  const double t186 = (Rational_2_3)*trK_dD0;
  const double trK_dD1 = V0_trK_dD1;
  const double t187 = (Rational_2_3)*trK_dD1;
  const double t188 = 12.0*t114;
  const double t189 = 12.0*t119;
  const double t190 = 12.0*t123;
  const double t191 = 6.0*t113 + 6.0*t115 + 6.0*t117 + 6.0*t118 + 6.0*t121 + 6.0*t122 + 6.0*t125 + 6.0*t126 + 6.0*t128;
  const double t192 = t130*(-aDD00*t58 + aDD02*f0_of_xx0*f1_of_xx1*t182 + aDD12*f1_of_xx1*t0*t183 + aDD22*t0*t184*t2 - t114*t63 - t119*t177);
  const double t193 = -t88;
  const double t194 = -t90;
  const double t195 = t24*t42;
  const double t196 = t157*t54 + t195*t86;
  const double t197 = -t196;
  const double t198 = t130*(aDD02*f0_of_xx0*f1_of_xx1*t193 + aDD12*f1_of_xx1*t0*t194 + aDD22*t0*t197*t2 - t114*t58 - t123*t177 - t16*t63);
  const double t199 = t13*(t119*t175 - t119*t58 + t123*t176 - t123*t63 - t177*t27 + t178*t27);
  const double t200 = t199*t44;
  const double t201 = -aDD00*t74 - t114*t75 - t119*t165 + t163 + t173;
  const double aDD_dD111 = V0_aDD_dD111;
  const double t202 = aDD_dD111*t0 + t114*t162 - t114*t74 - t123*t165 + t123*t166 + t16*t164 - t16*t75;
  const double t203 = t114*t193 + t123*t197 + t16*t194;
  const double aDD_dD121 = V0_aDD_dD121;
  const double t204 = aDD12*t70 + aDD_dD121*t38;
  const double t205 = -t119*t74 - t123*t75 - t165*t27 + t203 + t204;
  const double t206 = t107*t205;
  const double t207 = aDD00*t170 + t114*t171 + t119*t172;
  const double t208 = -aDD00*t98 - t114*t99 - t119*t167;
  const double aDD_dD001 = V0_aDD_dD001;
  const double t209 = aDD_dD001 + t207 + t208;
  const double aDD_dD010 = V0_aDD_dD010;
  const double t210 = aDD01 + aDD_dD010*f0_of_xx0;
  const double t211 = -t114*t82 - t123*t159 - t16*t83 + t207 + t210;
  const double t212 = t114*t154 + t123*t160 + t155*t16 + t208 + t210;
  const double t213 = aDD00*t88;
  const double t214 = t114*t90;
  const double t215 = t119*t196;
  const double t216 = aDD01*f0_of_xx0*t182 + aDD11*t0*t183 + aDD12*f1_of_xx1*t0*t184 - t213 - t214 - t215;
  const double aDD_dD021 = V0_aDD_dD021;
  const double t217 = aDD02*t95 + aDD_dD021*t23;
  const double t218 = t119*t170 + t123*t171 + t172*t27;
  const double t219 = -t213 - t214 - t215 + t217 + t218;
  const double t220 = aDD00*t182 + t114*t183 + t119*t184;
  const double t221 = -aDD00*t93 - t114*t94 - t119*t179;
  const double t222 = t220 + t221;
  const double aDD_dD020 = V0_aDD_dD020;
  const double t223 = aDD_dD020*t23 + t34;
  const double t224 = -t119*t82 - t123*t83 - t159*t27 + t220 + t223;
  const double t225 = t119*t154 + t123*t155 + t160*t27 + t221 + t223;
  const double t226 = -t114*t88 - t123*t196 - t16*t90;
  const double t227 = t203 + t226;
  const double t228 = t119*t162 + t123*t164 + t166*t27 + t204 + t226;
  const double t229 = aDD00*t193 + t114*t194 + t119*t197;
  const double t230 = -t114*t93 - t123*t179 - t16*t94;
  const double t231 = t229 + t230;
  const double t232 = -t119*t98 - t123*t99 - t167*t27;
  const double t233 = t217 + t229 + t232;
  const double aDD_dD120 = V0_aDD_dD120;
  const double t234 = aDD12*t78 + aDD_dD120*t38;
  const double t235 = t114*t182 + t123*t184 + t16*t183 + t232 + t234;
  const double t236 = t218 + t230 + t234;
  const double t237 = -t119*t88 - t123*t90 - t196*t27;
  const double t238 = t114*t175 + t123*t178 + t16*t176 + t237;
  const double aDD_dD221 = V0_aDD_dD221;
  const double t239 = aDD22*t53 + aDD_dD221*t3 + t119*t193 + t123*t194 + t197*t27 + t237;
  const double t240 = t108*t202 + t110*t227 + t110*t228 + t116*t201 + t120*t216 + t120*t219 + t127*t238 + t127*t239 + t161*t8 + t169*t20 + t174*t20 + t18*t198 + t181*t26 + t185*t26 - t186*t50 - t187*t89 - t191*t65 + t192*t7 + t200*t24 + t206*t24 + t209*t32 + t211*t32 + t212*t32 + t222*t33 + t224*t33 + t225*t33 + t231*t37 + t233*t37 + t235*t37 + t236*t37 - t60*(6.0*t15 + t188*t32 + t189*t33 + t190*t37 + 6.0*t21 + 6.0*t28);
  out[1 * Ntot + idx] = t240*t41;
  const double t241 = t161*t7;
  const double t242 = t103*t202 + t105*t238 + t105*t239 + t108*t169 + t108*t174 + t108*t201 + t110*t216 + t110*t219 + t110*t233 + t110*t235 + t111*t227 + t111*t228 + t116*t211 + t120*t224 + t124*t231 + t124*t236 + t127*t181 + t127*t185 + t18*t192 + t18*t241 - t186*t89 - t187*t61 - t191*t60 + t198*t43 + t20*t209 + t20*t212 + t200*t46 + t206*t46 + t222*t37 + t225*t37 - t65*(6.0*t102 + 6.0*t104 + 6.0*t106 + t108*t188 + t110*t189 + t111*t190);
  out[2 * Ntot + idx] = t242*t41;
  const double t243 = t105*t227 + t105*t228 + t110*t169 + t110*t174 + t111*t202 + t120*t211 + t124*t201 + t127*t216 + t127*t219 + t127*t231 + t127*t236 + t129*t199 + t131*t181 + t131*t185 + t132*t238 + t132*t239 + t138*t224 + t140*t233 + t140*t235 + t151*t205 - t186*t195 - t187*t42*t46 + t192*t24 + t198*t46 + t209*t37 + t212*t37 + t222*t26 + t225*t26 + t24*t241 - t60*(6.0*t133 + 6.0*t134 + 6.0*t135 + 6.0*t136 + 6.0*t137 + 6.0*t139 + 6.0*t141 + 6.0*t142 + 6.0*t143) - t65*(6.0*t144 + 6.0*t145 + 6.0*t146 + 6.0*t147 + 6.0*t148 + 6.0*t149 + 6.0*t150 + 6.0*t152 + 6.0*t153);
  out[3 * Ntot + idx] = t243*t41;
  const double t244 = (cf*cf*cf*cf);
  const double t245 = hDD01*t29;
  const double t246 = t240*t244;
  const double t247 = t29*t77;
  const double t248 = 2.0*t45;
  out[4 * Ntot + idx] = t100*(t1*(t242*t242)*t244 + t10*(t240*t240)*t244 + t242*t243*t244*t248 + t242*t245*t246 + (t243*t243)*t244*t4 + t243*t246*t247);
  const double t249 = 2.0*t42;
  const double t250 = t249*t46;
  const double t251 = t24*t249;
  const double t252 = 2.0*t89;
  const double lambdaU0 = in[17 * Ntot + idx];
  const double t253 = lambdaU0 - t250*t88 - t251*t93 - t252*t98 - t50*t82 - t61*(f0_of_xx0 + t74) - t66*(f0_of_xx0*t2 + t58);
  const double t254 = (1.0 / f0_of_xx0);
  const double t255 = -t254;
  const double lambdaU1 = in[18 * Ntot + idx];
  const double t256 = lambdaU1*t254 - t250*t90 - t251*t94 - t252*(t255 + t99) - t50*t83 - t61*t75 - t66*(t52 + t63);
  const double t257 = (1.0 / f1_of_xx1);
  const double lambdaU2 = in[19 * Ntot + idx];
  const double t258 = lambdaU2*t254*t257 - t159*t50 - t165*t61 - t167*t252 - t177*t66 - t250*(-f1_of_xx1__D1*t257 + t196) - t251*(t179 + t255);
  out[5 * Ntot + idx] = sqrt(t1*(t256*t256) + t10*(t253*t253) + t245*t253*t256 + t247*t253*t258 + t248*t256*t258 + (t258*t258)*t4);
    }
  }
}
#undef Rational_1_2
#undef Rational_2_3

extern "C" hipError_t launch_bssn_constraints_Spherical_sym2_KO0_fd4_k1_lb1_L16x2x2x1_d3_dmo_rb1_io_pg_lr40_di_mi_xcd(dim3 g, dim3 b, hipStream_t s, const double *in, const double *aux, double *out, const double *rfm0, const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_constraints_Spherical_sym2_KO0_fd4_k1_lb1_L16x2x2x1_d3_dmo_rb1_io_pg_lr40_di_mi_xcd_g0, dim3((p.Nx0 - 2 * p.NG + 15) / 16, (p.Nx1 - 2 * p.NG + 1) / 2, (p.Nx2 - 2 * p.NG + 1) / 2), dim3(64), 0, s, in, aux, out, rfm0, rfm1, p);
  return hipGetLastError();
}
