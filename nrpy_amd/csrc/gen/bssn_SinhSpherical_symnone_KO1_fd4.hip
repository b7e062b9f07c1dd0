// Generated by nrpy_amd/codegen/hip_gen.py -- do not edit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "../bhah_device_types.h"
// ---- BSSN kernels: SinhSpherical, symmetry axes '', KO=True, fd_order=4
#define Rational_1_2 (1.0 / 2.0)
#define Rational_2_3 (2.0 / 3.0)

typedef double bhah_d2 __attribute__((ext_vector_type(2)));
namespace rk_SinhSpherical_symnone_KO1_fd4 {
constexpr int PAR[24] = {4, 5, 6, 7, 8, 9, 0, 1, 2, 3, 0, 4, 5, 6, 7, 8, 9, 1, 2, 3, 0, 1, 2, 3};
// gridfunction j of group G
constexpr __host__ __device__ int gf(int G, int j) {
  return G == 0 ? 11 + j : G == 1 ? j : G == 2 ? (j < 5 ? 6 + j : 17) : 18 + j;
}
// NP consecutive values; NT: with the non-temporal hint
constexpr __host__ __device__ bool ricci_reads(int g) { return (g >= 11 && g <= 16) || (g >= 17 && g <= 19); }
template <int NP>
struct Vec;
template <>
struct Vec<1> {
  double v[1];
  template <bool NT>
  static __device__ __forceinline__ Vec ld(const double *q) {
    return {{NT ? __builtin_nontemporal_load(q) : *q}};
  }
  template <bool NT>
  __device__ __forceinline__ void st(double *q) const {
    if (NT) __builtin_nontemporal_store(v[0], q);
    else *q = v[0];
  }
};
template <>
struct Vec<2> {
  double v[2];
  template <bool NT>
  static __device__ __forceinline__ Vec ld(const double *q) {
    const bhah_d2 t = NT ? __builtin_nontemporal_load((const bhah_d2 *)q) : *(const bhah_d2 *)q;
    return {{t.x, t.y}};
  }
  template <bool NT>
  __device__ __forceinline__ void st(double *q) const {
    bhah_d2 t;
    t.x = v[0];
    t.y = v[1];
    if (NT) __builtin_nontemporal_store(t, (bhah_d2 *)q);
    else *(bhah_d2 *)q = t;
  }
};
// Where this thread's points find the right-hand side: a point or an aligned pair (from, code), or,
// for a pair whose sources are apart, two points with their parity masks.
struct Source {
  long from, s0, s1;
  unsigned code, m0, m1;
  bool split, ghost;  // ghost: every point of this thread is an inner ghost point
};
template <int NP>
__device__ __forceinline__ Source find_source(const int2 *map, const int2 *pairs, long q) {
  Source S;
  const int2 m = (NP == 2) ? pairs[q] : map[q];
  S.split = NP == 2 && m.y < 0;
  S.code = (unsigned)m.y;
  S.from = (long)m.x * NP;
  S.s0 = S.s1 = 0;
  S.m0 = S.m1 = 0;
  S.ghost = S.from != q * NP;
  if (S.split) {
    const int4 t = ((const int4 *)map)[q];
    S.s0 = t.x;
    S.m0 = (unsigned)t.y;
    S.s1 = t.z;
    S.m1 = (unsigned)t.w;
    S.ghost = S.s0 != 2 * q && S.s1 != 2 * q + 1;
  }
  return S;
}
// The six gridfunctions of group G of f at this thread's sources, with their parity signs.
template <int G, int NP, bool NT>
__device__ __forceinline__ void at_source(Vec<NP> (&r)[6], const double *f, const long Ntot, const Source &S) {
  if (NP == 2 && S.split) {
#pragma unroll
    for (int j = 0; j < 6; j++) {
      r[j].v[0] = f[gf(G, j) * Ntot + S.s0];
      r[j].v[NP - 1] = f[gf(G, j) * Ntot + S.s1];
    }
#pragma unroll
    for (int j = 0; j < 6; j++) {
      r[j].v[0] = ((S.m0 >> PAR[gf(G, j)]) & 1u) ? -r[j].v[0] : r[j].v[0];
      r[j].v[NP - 1] = ((S.m1 >> PAR[gf(G, j)]) & 1u) ? -r[j].v[NP - 1] : r[j].v[NP - 1];
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < 6; j++) r[j] = Vec<NP>::template ld<NT>(f + gf(G, j) * Ntot + S.from);
#pragma unroll
  for (int j = 0; j < 6; j++) {
    const int t = PAR[gf(G, j)];
    if (NP == 1) {
      r[j].v[0] = ((S.code >> t) & 1u) ? -r[j].v[0] : r[j].v[0];
    } else {
      const double a = (S.code & 1u) ? r[j].v[NP - 1] : r[j].v[0], b = (S.code & 2u) ? r[j].v[NP - 1] : r[j].v[0];
      r[j].v[0] = ((S.code >> (4 + t)) & 1u) ? -a : a;
      r[j].v[NP - 1] = ((S.code >> (16 + t)) & 1u) ? -b : b;
    }
  }
}
// KEEP: the pass also writes k at inner ghost points, which a taped step keeps.  Only the pass that
// folds the inner condition and leaves k alone has k in an array of its own: without the fold the
// stage is written over k.
template <bool INNER, bool KEEP>
struct KPtr {
  typedef const double *type;
};
template <>
struct KPtr<true, false> {
  typedef const double *__restrict__ type;
};
template <>
struct KPtr<true, true> {
  typedef double *type;
};
template <bool INNER, bool KEEP>
using k_ptr = typename KPtr<INNER, KEEP>::type;
// Write the inner ghost points' k among this thread's points: each point's own thread writes it, and
// no thread takes a value from it (sources are never inner ghost points).
template <int G, int NP>
__device__ __forceinline__ void keep_ghosts(double *f, const Vec<NP> (&k)[6], const long Ntot, const Source &S,
                                            const long idx) {
  const bool g0 = (NP == 2 && S.split) ? S.s0 != idx : S.from != idx || (NP == 2 && (S.code & 1u));
  const bool g1 = NP == 2 && (S.split ? S.s1 != idx + 1 : S.from != idx || !(S.code & 2u));
#pragma unroll
  for (int j = 0; j < 6; j++) {
    double *o = f + gf(G, j) * Ntot + idx;
    if (NP == 2 && g0 && g1) {
      k[j].template st<false>(o);
    } else {
      if (g0) o[0] = k[j].v[0];
      if (g1) o[1] = k[j].v[NP - 1];
    }
  }
}
template <int G, int NP, bool INNER, bool NT, bool KEEP>
__device__ __forceinline__ void group(k_ptr<INNER, KEEP> kin, const double *y_n, double *y_run, double *out,
                                      const double *__restrict__ rfm0, const double *__restrict__ rfm1,
                                      const bhah_kparams &p, const int2 *__restrict__ map,
                                      const int2 *__restrict__ pairs, const long q) {
  const long Ntot = p.Ntot, idx = q * NP;
  constexpr int N = 6;
  const double dt = p.dt;
  Vec<NP> k[N], y[N], r[N];
  Source S;
  S.ghost = false;
  if (INNER) {
    S = find_source<NP>(map, pairs, q);
    at_source<G, NP, NT>(k, kin, Ntot, S);
  } else {
#pragma unroll
    for (int j = 0; j < N; j++) k[j] = Vec<NP>::template ld<NT>(kin + gf(G, j) * Ntot + idx);
  }
  const bool ghost = S.ghost;
#pragma unroll
  for (int j = 0; j < N; j++) y[j] = Vec<NP>::template ld<NT>(y_n + gf(G, j) * Ntot + idx);
  // RK4 substep update (register_all_MoL_step_forward_in_time.c:4-103), in registers.
  if (p.substep == 4) {
    if (INNER && ghost) {
      at_source<G, NP, true>(r, y_run, Ntot, S);
    } else {
#pragma unroll
      for (int j = 0; j < N; j++) r[j] = Vec<NP>::template ld<true>(y_run + gf(G, j) * Ntot + idx);
    }
#pragma unroll
    for (int j = 0; j < N; j++)
#pragma unroll
      for (int e = 0; e < NP; e++) y[j].v[e] = (1.0 / 6.0) * dt * k[j].v[e] + y[j].v[e] + r[j].v[e];
  } else {
    if (!ghost) {
      if (p.substep == 1) {
#pragma unroll
        for (int j = 0; j < N; j++)
#pragma unroll
          for (int e = 0; e < NP; e++) r[j].v[e] = (1.0 / 6.0) * dt * k[j].v[e];
      } else {
#pragma unroll
        for (int j = 0; j < N; j++) r[j] = Vec<NP>::template ld<true>(y_run + gf(G, j) * Ntot + idx);
#pragma unroll
        for (int j = 0; j < N; j++)
#pragma unroll
          for (int e = 0; e < NP; e++) r[j].v[e] = (1.0 / 3.0) * dt * k[j].v[e] + r[j].v[e];
      }
#pragma unroll
      for (int j = 0; j < N; j++) r[j].template st<true>(y_run + gf(G, j) * Ntot + idx);
    }
    const double a = (p.substep == 3) ? 1.0 : (1.0 / 2.0);
#pragma unroll
    for (int j = 0; j < N; j++)
#pragma unroll
      for (int e = 0; e < NP; e++) y[j].v[e] = a * dt * k[j].v[e] + y[j].v[e];
  }
  if (G == 0) {
#pragma unroll
    for (int e = 0; e < NP; e++) {
      const unsigned long u = (unsigned long)(idx + e), row = u / (unsigned)p.Nx0;
      const int i0 = (int)(u - row * (unsigned)p.Nx0), i1 = (int)(row % (unsigned)p.Nx1);
      double nxt[N];
#pragma unroll
      for (int j = 0; j < N; j++) nxt[j] = y[j].v[e];
  {
    const double hDD00 = nxt[0];
    const double hDD01 = nxt[1];
    const double hDD02 = nxt[2];
    const double hDD11 = nxt[3];
    const double hDD12 = nxt[4];
    const double hDD22 = nxt[5];
    const double f0_of_xx0 = rfm0[i0];
    const double f0_of_xx0__D0 = rfm0[p.Nx0 + i0];
    const double f1_of_xx1 = rfm1[i1];
    const double dg0 = (f0_of_xx0*f0_of_xx0);
    const double dg1 = dg0*hDD11 + dg0;
    const double dg2 = (f0_of_xx0__D0*f0_of_xx0__D0);
    const double dg3 = dg2*hDD00 + dg2;
    const double dg4 = (f1_of_xx1*f1_of_xx1);
    const double dg5 = dg0*dg4;
    const double dg6 = dg5*hDD22 + dg5;
    const double dg7 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
    const double dg8 = dg4*dg7;
    const double dg9 = cbrt(fabs(dg2*dg8)/(-dg0*dg2*dg6*(hDD01*hDD01) - dg1*dg2*dg5*(hDD02*hDD02) + dg1*dg3*dg6 + 2.0*dg2*dg4*dg7*hDD01*hDD02*hDD12 - dg3*dg8*(hDD12*hDD12)));
    const double new_hDD00 = dg9*(hDD00 + 1.0) - 1.0;
    const double new_hDD01 = dg9*hDD01;
    const double new_hDD02 = dg9*hDD02;
    const double new_hDD11 = dg9*(hDD11 + 1.0) - 1.0;
    const double new_hDD12 = dg9*hDD12;
    const double new_hDD22 = dg9*(hDD22 + 1.0) - 1.0;
    nxt[0] = new_hDD00;
    nxt[1] = new_hDD01;
    nxt[2] = new_hDD02;
    nxt[3] = new_hDD11;
    nxt[4] = new_hDD12;
    nxt[5] = new_hDD22;
  }
#pragma unroll
      for (int j = 0; j < N; j++) y[j].v[e] = nxt[j];
    }
  }
#pragma unroll
  for (int j = 0; j < N; j++) {
    double *o = out + gf(G, j) * Ntot + idx;
    if (NT && !ricci_reads(gf(G, j))) y[j].template st<true>(o);
    else y[j].template st<false>(o);
  }
  if constexpr (KEEP) keep_ghosts<G, NP>(kin, k, Ntot, S, idx);
}
template <int NP, bool INNER, bool NT, bool KEEP>
__device__ __forceinline__ void any_group(int G, k_ptr<INNER, KEEP> kin, const double *y_n, double *y_run,
                                          double *out, const double *__restrict__ rfm0,
                                          const double *__restrict__ rfm1, const bhah_kparams &p,
                                          const int2 *__restrict__ map, const int2 *__restrict__ pairs,
                                          const long q) {
  if (q * NP >= p.Ntot) return;
  if (G == 0) group<0, NP, INNER, NT, KEEP>(kin, y_n, y_run, out, rfm0, rfm1, p, map, pairs, q);
  else if (G == 1) group<1, NP, INNER, NT, KEEP>(kin, y_n, y_run, out, rfm0, rfm1, p, map, pairs, q);
  else if (G == 2) group<2, NP, INNER, NT, KEEP>(kin, y_n, y_run, out, rfm0, rfm1, p, map, pairs, q);
  else group<3, NP, INNER, NT, KEEP>(kin, y_n, y_run, out, rfm0, rfm1, p, map, pairs, q);
}
}  // namespace rk_SinhSpherical_symnone_KO1_fd4
template <int NP, bool INNER, bool NT, bool KEEP>
__global__ void __launch_bounds__(256)
bssn_rk_det_SinhSpherical_symnone_KO1_fd4(rk_SinhSpherical_symnone_KO1_fd4::k_ptr<INNER, KEEP> kin, const double *y_n, double *y_run, double *out,
                  const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p,
                  const int2 *__restrict__ map, const int2 *__restrict__ pairs) {
  rk_SinhSpherical_symnone_KO1_fd4::any_group<NP, INNER, NT, KEEP>((int)(blockIdx.x & 3u), kin, y_n, y_run, out, rfm0, rfm1, p, map, pairs,
                                 (long)(blockIdx.x >> 2) * blockDim.x + threadIdx.x);
}

extern "C" __global__ void __launch_bounds__(256)
bssn_detgamma_SinhSpherical_symnone_KO1_fd4(double *__restrict__ gfs, const double *__restrict__ rfm0, const double *__restrict__ rfm1,
                    const bhah_kparams p) {
  const int i0 = 0 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int i1 = 0 + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  const int i2 = 0 + (int)blockIdx.z;
  if (i0 >= p.Nx0 - 0 || i1 >= p.Nx1 - 0) return;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;

  double nxt[24];
#pragma unroll
  for (int g = 0; g < 24; g++) nxt[g] = 0.0;
  nxt[11] = gfs[11 * Ntot + idx];
  nxt[12] = gfs[12 * Ntot + idx];
  nxt[13] = gfs[13 * Ntot + idx];
  nxt[14] = gfs[14 * Ntot + idx];
  nxt[15] = gfs[15 * Ntot + idx];
  nxt[16] = gfs[16 * Ntot + idx];

  {
    const double hDD00 = nxt[11];
    const double hDD01 = nxt[12];
    const double hDD02 = nxt[13];
    const double hDD11 = nxt[14];
    const double hDD12 = nxt[15];
    const double hDD22 = nxt[16];
    const double f0_of_xx0 = rfm0[i0];
    const double f0_of_xx0__D0 = rfm0[p.Nx0 + i0];
    const double f1_of_xx1 = rfm1[i1];
    const double dg0 = (f0_of_xx0*f0_of_xx0);
    const double dg1 = dg0*hDD11 + dg0;
    const double dg2 = (f0_of_xx0__D0*f0_of_xx0__D0);
    const double dg3 = dg2*hDD00 + dg2;
    const double dg4 = (f1_of_xx1*f1_of_xx1);
    const double dg5 = dg0*dg4;
    const double dg6 = dg5*hDD22 + dg5;
    const double dg7 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
    const double dg8 = dg4*dg7;
    const double dg9 = cbrt(fabs(dg2*dg8)/(-dg0*dg2*dg6*(hDD01*hDD01) - dg1*dg2*dg5*(hDD02*hDD02) + dg1*dg3*dg6 + 2.0*dg2*dg4*dg7*hDD01*hDD02*hDD12 - dg3*dg8*(hDD12*hDD12)));
    const double new_hDD00 = dg9*(hDD00 + 1.0) - 1.0;
    const double new_hDD01 = dg9*hDD01;
    const double new_hDD02 = dg9*hDD02;
    const double new_hDD11 = dg9*(hDD11 + 1.0) - 1.0;
    const double new_hDD12 = dg9*hDD12;
    const double new_hDD22 = dg9*(hDD22 + 1.0) - 1.0;
    nxt[11] = new_hDD00;
    nxt[12] = new_hDD01;
    nxt[13] = new_hDD02;
    nxt[14] = new_hDD11;
    nxt[15] = new_hDD12;
    nxt[16] = new_hDD22;
  }
  gfs[11 * Ntot + idx] = nxt[11];
  gfs[12 * Ntot + idx] = nxt[12];
  gfs[13 * Ntot + idx] = nxt[13];
  gfs[14 * Ntot + idx] = nxt[14];
  gfs[15 * Ntot + idx] = nxt[15];
  gfs[16 * Ntot + idx] = nxt[16];

}

extern "C" __global__ void __launch_bounds__(256)
bssn_constraints_SinhSpherical_symnone_KO1_fd4(const double *__restrict__ in, const double *__restrict__ aux, double *__restrict__ diag,
                       const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  const int i0 = p.NG + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int i1 = p.NG + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  const int i2 = p.NG + (int)blockIdx.z;
  if (i0 >= p.Nx0 - p.NG || i1 >= p.Nx1 - p.NG) return;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;

  const double cf = in[10 * Ntot + idx];
  const double t0 = (cf*cf);
  const double f0_of_xx0 = rfm0[i0];
  const double f0_of_xx0__D0 = rfm0[p.Nx0 + i0];
  const double t18 = (f0_of_xx0*f0_of_xx0*f0_of_xx0)*f0_of_xx0__D0;
  const double t1 = (f0_of_xx0*f0_of_xx0);
  const double hDD11 = in[14 * Ntot + idx];
  const double t2 = hDD11*t1 + t1;
  const double f1_of_xx1 = rfm1[i1];
  const double hDD12 = in[15 * Ntot + idx];
  const double t20 = f1_of_xx1*hDD12;
  const double t17 = f0_of_xx0*f0_of_xx0__D0;
  const double t21 = f1_of_xx1*t17;
  const double hDD01 = in[12 * Ntot + idx];
  const double hDD02 = in[13 * Ntot + idx];
  const double t22 = hDD01*t18*t20 - hDD02*t2*t21;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t36 = f1_of_xx1*f1_of_xx1__D1;
  const double t37 = 2.0*t1*t36;
  const double t5 = (f1_of_xx1*f1_of_xx1);
  const double t6 = t1*t5;
  const double hDD22 = in[16 * Ntot + idx];
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t38 = hDD22*t37 + hDD_dD221*t6 + t37;
  const double t23 = f1_of_xx1*t1;
  const double t24 = hDD12*t23;
  const double t3 = (f0_of_xx0__D0*f0_of_xx0__D0);
  const double t25 = f1_of_xx1*t3;
  const double hDD00 = in[11 * Ntot + idx];
  const double t4 = hDD00*t3 + t3;
  const double t26 = hDD01*hDD02*t1*t25 - t24*t4;
  const double t9 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t10 = (hDD12*hDD12)*t5*t9;
  const double t11 = (hDD02*hDD02)*t3*t6;
  const double t7 = hDD22*t6 + t6;
  const double t8 = (hDD01*hDD01)*t1*t3;
  const double t12 = 2.0*hDD01*hDD02*hDD12*t3*t5*t9 - t10*t4 - t11*t2 + t2*t4*t7 - t7*t8;
  const double t13 = (1.0 / t12);
  const double t40 = (Rational_1_2)*t13;
  const double t48 = t26*t40;
  const double t16 = t2*t4 - t8;
  const double t51 = t13*t16;
  const double t52 = (Rational_1_2)*t51;
  const double hDD_dD112 = p.invdxx2 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s2)] - in[14 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s2)] - in[14 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t72 = hDD_dD112*t1;
  const double hDD_dD012 = p.invdxx2 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s2)] - in[12 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s2)] - in[12 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t81 = hDD_dD012*t17;
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t82 = hDD_dD021*t21;
  const double t83 = f1_of_xx1__D1*t17;
  const double t84 = hDD02*t83;
  const double t85 = t82 + t84;
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t86 = hDD_dD120*t23;
  const double t30 = 2.0*t17;
  const double t87 = t20*t30;
  const double t95 = t81 + t85 - t86 - t87;
  const double t98 = t40*t95;
  const double t100 = t22*t98 + t38*t52 + t48*t72;
  const double t88 = t86 + t87;
  const double t101 = t81 - t82 - t84 + t88;
  const double t102 = t101*t40;
  const double t31 = t30*t5;
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t32 = hDD22*t31 + hDD_dD220*t6 + t31;
  const double t103 = t32*t40;
  const double t19 = -hDD01*t17*t7 + hDD02*hDD12*t18*t5;
  const double t14 = -t10 + t2*t7;
  const double t34 = t13*t14;
  const double t35 = (Rational_1_2)*t34;
  const double hDD_dD002 = p.invdxx2 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s2)] - in[11 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s2)] - in[11 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t62 = hDD_dD002*t3;
  const double t104 = t102*t19 + t103*t22 + t35*t62;
  const double t41 = t19*t40;
  const double t15 = -t11 + t4*t7;
  const double t46 = t13*t15;
  const double t47 = (Rational_1_2)*t46;
  const double t105 = t101*t47 + t103*t26 + t41*t62;
  const double t42 = t22*t40;
  const double t106 = t102*t26 + t32*t52 + t42*t62;
  const double t107 = (1.0 / t0);
  const double t108 = 2.0*t107;
  const double t109 = 4.0*t107*t13;
  const double cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] - in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] - in[10 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t110 = cf_dD1*t109;
  const double aDD00 = in[idx];
  const double t111 = aDD00*t3;
  const double t112 = (1.0 / (t12*t12));
  const double t113 = t112*(t14*t14);
  const double t114 = t111*t113;
  const double aDD11 = in[3 * Ntot + idx];
  const double t115 = aDD11*t1;
  const double t116 = t112*(t19*t19);
  const double t117 = t115*t116;
  const double aDD22 = in[5 * Ntot + idx];
  const double t119 = aDD22*t6;
  const double t118 = t112*(t22*t22);
  const double t120 = t118*t119;
  const double t121 = t112*t14;
  const double t122 = t121*t19;
  const double aDD01 = in[1 * Ntot + idx];
  const double t123 = aDD01*t30;
  const double t124 = t112*t19;
  const double t125 = t124*t22;
  const double t73 = 2.0*t23;
  const double aDD12 = in[4 * Ntot + idx];
  const double t126 = aDD12*t73;
  const double t127 = t121*t22;
  const double t64 = f1_of_xx1*t30;
  const double aDD02 = in[2 * Ntot + idx];
  const double t128 = aDD02*t64;
  const double t129 = t111*t116;
  const double t130 = t112*(t15*t15);
  const double t131 = t115*t130;
  const double t132 = t112*(t26*t26);
  const double t133 = t119*t132;
  const double t134 = t112*t15;
  const double t135 = t134*t19;
  const double t136 = t134*t26;
  const double t137 = t124*t26;
  const double t138 = t111*t118;
  const double t139 = t115*t132;
  const double t140 = (t16*t16);
  const double t141 = t112*t119*t140;
  const double t142 = t112*t22;
  const double t143 = t142*t26;
  const double t144 = t112*t16;
  const double t145 = t144*t26;
  const double t146 = t144*t22;
  const double t147 = t111*t122;
  const double t148 = aDD01*t17;
  const double t149 = t116*t148;
  const double t150 = t115*t135;
  const double t151 = t121*t15;
  const double t152 = t148*t151;
  const double t153 = aDD12*t23;
  const double t154 = t134*t22;
  const double t155 = t153*t154;
  const double t156 = t137*t153;
  const double t157 = t119*t143;
  const double t158 = t121*t26;
  const double t159 = aDD02*t21;
  const double t160 = t158*t159;
  const double t161 = t125*t159;
  const double t162 = t111*t125;
  const double t163 = t115*t136;
  const double t164 = t132*t153;
  const double t165 = t148*t154;
  const double t166 = t137*t148;
  const double t167 = t144*t15;
  const double t168 = t153*t167;
  const double t169 = t119*t145;
  const double t170 = t144*t19;
  const double t171 = t159*t170;
  const double t172 = t143*t159;
  const double t173 = t111*t127;
  const double t174 = t115*t137;
  const double t175 = t148*t158;
  const double t176 = t125*t148;
  const double t177 = t118*t159;
  const double t178 = t153*t170;
  const double t179 = t143*t153;
  const double t180 = t119*t146;
  const double t181 = t14*t144;
  const double t182 = t159*t181;
  const double t27 = (1.0 / cf);
  const double cf_dD2 = p.invdxx2 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1 * s2)] - in[10 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s2)] - in[10 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t28 = (cf_dD2*cf_dD2);
  const double t29 = (Rational_1_2)*t27;
  const double hDD_dD022 = p.invdxx2 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s2)] - in[13 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s2)] - in[13 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t33 = 2.0*f0_of_xx0*f0_of_xx0__D0*f1_of_xx1*hDD_dD022 - t32;
  const double hDD_dD122 = p.invdxx2 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s2)] - in[15 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s2)] - in[15 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t39 = 2.0*f1_of_xx1*hDD_dD122*t1 - t38;
  const double hDD_dD222 = p.invdxx2 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s2)] - in[16 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s2)] - in[16 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t43 = hDD_dD222*t6;
  const double t44 = t33*t35 + t39*t41 + t42*t43;
  const double cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1)] - in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] - in[10 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t45 = cf_dD0*t29;
  const double t49 = t33*t41 + t39*t47 + t43*t48;
  const double t50 = (Rational_1_2)*cf_dD1*t27;
  const double t53 = t33*t42 + t39*t48 + t43*t52;
  const double t54 = cf_dD2*t29;
  const double t55 = (cf_dD0*cf_dD0);
  const double f0_of_xx0__DD00 = rfm0[2 * p.Nx0 + i0];
  const double t56 = 2.0*f0_of_xx0__D0*f0_of_xx0__DD00;
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t57 = hDD00*t56 + hDD_dD000*t3 + t56;
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t58 = hDD_dD001*t3;
  const double t59 = f0_of_xx0*f0_of_xx0__DD00;
  const double t60 = t3 + t59;
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t61 = 2.0*hDD01*t60 + hDD_dD010*t30 - t58;
  const double t63 = f1_of_xx1*t59 + t25;
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t65 = 2.0*hDD02*t63 + hDD_dD020*t64 - t62;
  const double t66 = t35*t57 + t41*t61 + t42*t65;
  const double t67 = t41*t57 + t47*t61 + t48*t65;
  const double t68 = t42*t57 + t48*t61 + t52*t65;
  const double t69 = (cf_dD1*cf_dD1);
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t70 = hDD11*t30 + hDD_dD110*t1 + t30;
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t71 = 2.0*f0_of_xx0*f0_of_xx0__D0*hDD_dD011 - t70;
  const double t74 = f1_of_xx1__D1*t1;
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t75 = 2.0*hDD12*t74 + hDD_dD121*t73 - t72;
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t76 = hDD_dD111*t1;
  const double t77 = t35*t71 + t41*t76 + t42*t75;
  const double t78 = t41*t71 + t47*t76 + t48*t75;
  const double t79 = t42*t71 + t48*t76 + t52*t75;
  const double t80 = t40*t70;
  const double t89 = -t81 + t85 + t88;
  const double t90 = t40*t89;
  const double t91 = t19*t80 + t22*t90 + t35*t58;
  const double t92 = t26*t90 + t41*t58 + t47*t70;
  const double t93 = t26*t80 + t42*t58 + t52*t89;
  const double t94 = 16.0*t13;
  const double t96 = t38*t40;
  const double t97 = t22*t96 + t35*t95 + t41*t72;
  const double t99 = t19*t98 + t26*t96 + t47*t72;
  const double RbarDD00 = aux[0 * Ntot + idx];
  const double RbarDD01 = aux[1 * Ntot + idx];
  const double RbarDD02 = aux[2 * Ntot + idx];
  const double RbarDD11 = aux[3 * Ntot + idx];
  const double RbarDD12 = aux[4 * Ntot + idx];
  const double RbarDD22 = aux[5 * Ntot + idx];
  const double cf_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[10 * Ntot + idx] + (4.0 / 3.0) * (in[10 * Ntot + idx + (1)] + in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] + in[10 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double cf_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[10 * Ntot + idx + (1 + 1 * s1)] - in[10 * Ntot + idx + (1 + -1 * s1)]) - (in[10 * Ntot + idx + (-1 + 1 * s1)] - in[10 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (1 + 2 * s1)] - in[10 * Ntot + idx + (1 + -2 * s1)]) - (in[10 * Ntot + idx + (-1 + 2 * s1)] - in[10 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (2 + 1 * s1)] - in[10 * Ntot + idx + (2 + -1 * s1)]) - (in[10 * Ntot + idx + (-2 + 1 * s1)] - in[10 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[10 * Ntot + idx + (2 + 2 * s1)] - in[10 * Ntot + idx + (2 + -2 * s1)]) - (in[10 * Ntot + idx + (-2 + 2 * s1)] - in[10 * Ntot + idx + (-2 + -2 * s1)])));
  __builtin_amdgcn_sched_barrier(0);
  const double cf_dDD02 = p.invdxx0 * p.invdxx2 * ((4.0 / 9.0) * ((in[10 * Ntot + idx + (1 + 1 * s2)] - in[10 * Ntot + idx + (1 + -1 * s2)]) - (in[10 * Ntot + idx + (-1 + 1 * s2)] - in[10 * Ntot + idx + (-1 + -1 * s2)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (1 + 2 * s2)] - in[10 * Ntot + idx + (1 + -2 * s2)]) - (in[10 * Ntot + idx + (-1 + 2 * s2)] - in[10 * Ntot + idx + (-1 + -2 * s2)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (2 + 1 * s2)] - in[10 * Ntot + idx + (2 + -1 * s2)]) - (in[10 * Ntot + idx + (-2 + 1 * s2)] - in[10 * Ntot + idx + (-2 + -1 * s2)])) + (1.0 / 144.0) * ((in[10 * Ntot + idx + (2 + 2 * s2)] - in[10 * Ntot + idx + (2 + -2 * s2)]) - (in[10 * Ntot + idx + (-2 + 2 * s2)] - in[10 * Ntot + idx + (-2 + -2 * s2)])));
  __builtin_amdgcn_sched_barrier(0);
  const double cf_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[10 * Ntot + idx] + (4.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] + in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] + in[10 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double cf_dDD12 = p.invdxx1 * p.invdxx2 * ((4.0 / 9.0) * ((in[10 * Ntot + idx + (1 * s1 + 1 * s2)] - in[10 * Ntot + idx + (1 * s1 + -1 * s2)]) - (in[10 * Ntot + idx + (-1 * s1 + 1 * s2)] - in[10 * Ntot + idx + (-1 * s1 + -1 * s2)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (1 * s1 + 2 * s2)] - in[10 * Ntot + idx + (1 * s1 + -2 * s2)]) - (in[10 * Ntot + idx + (-1 * s1 + 2 * s2)] - in[10 * Ntot + idx + (-1 * s1 + -2 * s2)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (2 * s1 + 1 * s2)] - in[10 * Ntot + idx + (2 * s1 + -1 * s2)]) - (in[10 * Ntot + idx + (-2 * s1 + 1 * s2)] - in[10 * Ntot + idx + (-2 * s1 + -1 * s2)])) + (1.0 / 144.0) * ((in[10 * Ntot + idx + (2 * s1 + 2 * s2)] - in[10 * Ntot + idx + (2 * s1 + -2 * s2)]) - (in[10 * Ntot + idx + (-2 * s1 + 2 * s2)] - in[10 * Ntot + idx + (-2 * s1 + -2 * s2)])));
  __builtin_amdgcn_sched_barrier(0);
  const double cf_dDD22 = p.invdxx2 * p.invdxx2 * ((-5.0 / 2.0) * in[10 * Ntot + idx] + (4.0 / 3.0) * (in[10 * Ntot + idx + (1 * s2)] + in[10 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s2)] + in[10 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double trK = in[20 * Ntot + idx];
  diag[0 * Ntot + idx] = t0*(RbarDD00*t13*t14 + 2.0*RbarDD01*t13*t19 + 2.0*RbarDD02*t13*t22 + RbarDD11*t13*t15 + 2.0*RbarDD12*t13*t26 + RbarDD22*t13*t16 - cf_dD0*cf_dD2*t109*t22 - cf_dD0*t110*t19 - cf_dD2*t110*t26 - t108*t28*t51 - t108*t34*t55 - t108*t46*t69 - t19*t94*(t29*(cf_dD0*cf_dD1*t27 - cf_dDD01) + t45*t91 + t50*t92 + t54*t93) - t22*t94*(t104*t45 + t105*t50 + t106*t54 + t29*(cf_dD0*cf_dD2*t27 - cf_dDD02)) - t26*t94*(t100*t54 + t29*(cf_dD1*cf_dD2*t27 - cf_dDD12) + t45*t97 + t50*t99) - 8.0*t34*(t29*(-cf_dDD00 + t27*t55) + t45*t66 + t50*t67 + t54*t68) - 8.0*t46*(t29*(-cf_dDD11 + t27*t69) + t45*t77 + t50*t78 + t54*t79) - 8.0*t51*(t29*(-cf_dDD22 + t27*t28) + t44*t45 + t49*t50 + t53*t54)) - t111*(t114 + t117 + t120 + t122*t123 + t125*t126 + t127*t128) - t115*(t123*t135 + t126*t136 + t128*t137 + t129 + t131 + t133) - t119*(t123*t143 + t126*t145 + t128*t146 + t138 + t139 + t141) - t123*(t147 + t149 + t150 + t152 + t155 + t156 + t157 + t160 + t161) - t126*(t162 + t163 + t164 + t165 + t166 + t168 + t169 + t171 + t172) - t128*(t173 + t174 + t175 + t176 + t177 + t178 + t179 + t180 + t182) + (Rational_2_3)*(trK*trK);
  const double t183 = -t66;
  const double t184 = -t67;
  const double t185 = -t68;
  const double aDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[idx + (1)] - in[idx + (-1)]) + (-1.0 / 12.0) * (in[idx + (2)] - in[idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t186 = aDD00*t56 + aDD_dD000*t3 + t111*t183 - t111*t66 + t148*t184 - t148*t67 + t159*t185 - t159*t68;
  const double t187 = -t77;
  const double aDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[1 * Ntot + idx + (1 * s1)] - in[1 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[1 * Ntot + idx + (2 * s1)] - in[1 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t188 = aDD_dD011*t17;
  const double t189 = -t78;
  const double t190 = -t79;
  const double t191 = -t115*t92 - t148*t91 - t153*t93;
  const double t192 = t111*t187 + t148*t189 + t159*t190 + t188 + t191;
  const double t193 = -t92;
  const double t194 = -t91;
  const double t195 = -t93;
  const double t196 = t115*t193 + t148*t194 + t153*t195;
  const double aDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[3 * Ntot + idx + (1)] - in[3 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[3 * Ntot + idx + (2)] - in[3 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t197 = aDD11*t30 + aDD_dD110*t1 + t191 + t196;
  const double t198 = -t44;
  const double t199 = -t49;
  const double aDD_dD022 = p.invdxx2 * ((2.0 / 3.0) * (in[2 * Ntot + idx + (1 * s2)] - in[2 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[2 * Ntot + idx + (2 * s2)] - in[2 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t200 = aDD_dD022*t21;
  const double t201 = -t53;
  const double t202 = -t104*t159 - t105*t153 - t106*t119;
  const double t203 = t111*t198 + t148*t199 + t159*t201 + t200 + t202;
  const double t204 = -t105;
  const double t205 = -t106;
  const double t206 = -t104;
  const double t207 = t119*t205 + t153*t204 + t159*t206;
  const double aDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[5 * Ntot + idx + (1)] - in[5 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[5 * Ntot + idx + (2)] - in[5 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t208 = aDD22*t31 + aDD_dD220*t6 + t202 + t207;
  const double trK_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1)] - in[20 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2)] - in[20 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t209 = (Rational_2_3)*trK_dD0;
  const double t210 = (Rational_2_3)*t13;
  const double trK_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1 * s1)] - in[20 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2 * s1)] - in[20 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t211 = t210*trK_dD1;
  const double trK_dD2 = p.invdxx2 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1 * s2)] - in[20 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2 * s2)] - in[20 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t212 = t210*trK_dD2;
  const double t213 = 12.0*t148;
  const double t214 = 12.0*t153;
  const double t215 = 12.0*t159;
  const double t216 = 6.0*t147 + 6.0*t149 + 6.0*t150 + 6.0*t152 + 6.0*t155 + 6.0*t156 + 6.0*t157 + 6.0*t160 + 6.0*t161;
  const double t217 = 6.0*t173 + 6.0*t174 + 6.0*t175 + 6.0*t176 + 6.0*t177 + 6.0*t178 + 6.0*t179 + 6.0*t180 + 6.0*t182;
  const double t218 = t144*(-t111*t44 - t148*t49 - t159*t53 + t200 + t207);
  const double aDD_dD122 = p.invdxx2 * ((2.0 / 3.0) * (in[4 * Ntot + idx + (1 * s2)] - in[4 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[4 * Ntot + idx + (2 * s2)] - in[4 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t219 = aDD_dD122*t23;
  const double t220 = -t99;
  const double t221 = -t100;
  const double t222 = -t97;
  const double t223 = t119*t221 + t153*t220 + t159*t222;
  const double t224 = t144*(-t115*t49 - t148*t44 - t153*t53 + t219 + t223);
  const double aDD_dD222 = p.invdxx2 * ((2.0 / 3.0) * (in[5 * Ntot + idx + (1 * s2)] - in[5 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[5 * Ntot + idx + (2 * s2)] - in[5 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t225 = t112*(aDD_dD222*t6 + t119*t201 - t119*t53 + t153*t199 - t153*t49 + t159*t198 - t159*t44);
  const double t226 = t16*t225;
  const double t227 = -t111*t77 - t148*t78 - t159*t79 + t188 + t196;
  const double t228 = t111*t194 + t148*t193 + t159*t195;
  const double t229 = -t111*t91 - t148*t92 - t159*t93;
  const double aDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[idx + (1 * s1)] - in[idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[idx + (2 * s1)] - in[idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t230 = aDD_dD001*t3 + t228 + t229;
  const double aDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[1 * Ntot + idx + (1)] - in[1 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[1 * Ntot + idx + (2)] - in[1 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t231 = aDD01*t60 + aDD_dD010*t17;
  const double t232 = -t115*t67 - t148*t66 - t153*t68 + t228 + t231;
  const double t233 = t115*t184 + t148*t183 + t153*t185 + t229 + t231;
  const double aDD_dD012 = p.invdxx2 * ((2.0 / 3.0) * (in[1 * Ntot + idx + (1 * s2)] - in[1 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[1 * Ntot + idx + (2 * s2)] - in[1 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t234 = aDD_dD012*t17;
  const double t235 = -t100*t159 - t111*t97 - t148*t99;
  const double t236 = t115*t204 + t148*t206 + t153*t205;
  const double t237 = t234 + t235 + t236;
  const double aDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[2 * Ntot + idx + (1 * s1)] - in[2 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[2 * Ntot + idx + (2 * s1)] - in[2 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t238 = aDD02*t83 + aDD_dD021*t21;
  const double t239 = t119*t195 + t153*t193 + t159*t194;
  const double t240 = t235 + t238 + t239;
  const double t241 = t111*t206 + t148*t204 + t159*t205;
  const double t242 = -t104*t111 - t105*t148 - t106*t159;
  const double aDD_dD002 = p.invdxx2 * ((2.0 / 3.0) * (in[idx + (1 * s2)] - in[idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[idx + (2 * s2)] - in[idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t243 = aDD_dD002*t3 + t241 + t242;
  const double aDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[2 * Ntot + idx + (1)] - in[2 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[2 * Ntot + idx + (2)] - in[2 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t244 = aDD02*t63 + aDD_dD020*t21;
  const double t245 = -t119*t68 - t153*t67 - t159*t66 + t241 + t244;
  const double t246 = t119*t185 + t153*t184 + t159*t183 + t242 + t244;
  const double aDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[3 * Ntot + idx + (1 * s1)] - in[3 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[3 * Ntot + idx + (2 * s1)] - in[3 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t247 = aDD_dD111*t1 + t115*t189 - t115*t78 + t148*t187 - t148*t77 + t153*t190 - t153*t79;
  const double t248 = t115*t220 + t148*t222 + t153*t221;
  const double aDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[4 * Ntot + idx + (1 * s1)] - in[4 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[4 * Ntot + idx + (2 * s1)] - in[4 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t249 = aDD12*t74 + aDD_dD121*t23;
  const double t250 = -t119*t79 - t153*t78 - t159*t77 + t248 + t249;
  const double t251 = t134*t250;
  const double t252 = -t100*t153 - t115*t99 - t148*t97;
  const double aDD_dD112 = p.invdxx2 * ((2.0 / 3.0) * (in[3 * Ntot + idx + (1 * s2)] - in[3 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[3 * Ntot + idx + (2 * s2)] - in[3 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t253 = aDD_dD112*t1 + t248 + t252;
  const double t254 = t253*t26;
  const double t255 = t119*t190 + t153*t189 + t159*t187 + t249 + t252;
  const double t256 = t255*t26;
  const double t257 = t111*t222 + t148*t220 + t159*t221;
  const double t258 = -t104*t148 - t105*t115 - t106*t153;
  const double t259 = t234 + t257 + t258;
  const double t260 = -t119*t93 - t153*t92 - t159*t91;
  const double t261 = t238 + t257 + t260;
  const double aDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[4 * Ntot + idx + (1)] - in[4 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[4 * Ntot + idx + (2)] - in[4 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t262 = aDD12*t64 + aDD_dD120*t23;
  const double t263 = t236 + t260 + t262;
  const double t264 = t239 + t258 + t262;
  const double t265 = -t100*t119 - t153*t99 - t159*t97;
  const double t266 = t115*t199 + t148*t198 + t153*t201 + t219 + t265;
  const double t267 = t26*t266;
  const double aDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[5 * Ntot + idx + (1 * s1)] - in[5 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[5 * Ntot + idx + (2 * s1)] - in[5 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t268 = aDD22*t37 + aDD_dD221*t6 + t223 + t265;
  const double t269 = t113*t186 + t116*t192 + t116*t197 + t118*t203 + t118*t208 + t122*t230 + t122*t232 + t122*t233 + t124*t254 + t124*t256 + t125*t259 + t125*t261 + t125*t263 + t125*t264 + t127*t243 + t127*t245 + t127*t246 + t135*t247 + t14*t218 + t142*t267 + t143*t268 + t151*t227 + t158*t237 + t158*t240 - t19*t211 + t19*t224 - t209*t34 - t212*t22 - t216*t50 - t217*t54 + t22*t226 + t22*t251 - t45*(6.0*t114 + 6.0*t117 + 6.0*t120 + t122*t213 + t125*t214 + t127*t215);
  diag[1 * Ntot + idx] = t0*t269;
  const double t270 = t13*t209;
  const double t271 = 6.0*t162 + 6.0*t163 + 6.0*t164 + 6.0*t165 + 6.0*t166 + 6.0*t168 + 6.0*t169 + 6.0*t171 + 6.0*t172;
  const double t272 = t116*t230 + t116*t233 + t122*t186 + t125*t243 + t125*t246 + t130*t247 + t132*t266 + t132*t268 + t134*t254 + t134*t256 + t135*t192 + t135*t197 + t135*t227 + t137*t237 + t137*t240 + t137*t261 + t137*t263 + t143*t203 + t143*t208 + t15*t224 + t151*t232 + t154*t259 + t154*t264 + t158*t245 + t19*t218 - t19*t270 - t212*t26 - t216*t45 + t226*t26 + t251*t26 - t271*t54 - Rational_2_3*t46*trK_dD1 - t50*(6.0*t129 + 6.0*t131 + 6.0*t133 + t135*t213 + t136*t214 + t137*t215);
  diag[2 * Ntot + idx] = t0*t272;
  const double t273 = t118*t243 + t118*t246 + t125*t230 + t125*t233 + t127*t186 + t132*t253 + t132*t255 + t136*t247 + t137*t192 + t137*t197 + t140*t225 + t143*t237 + t143*t240 + t143*t259 + t143*t264 + t144*t267 + t145*t268 + t146*t203 + t146*t208 + t154*t227 + t158*t232 + t167*t250 + t170*t261 + t170*t263 + t181*t245 - t211*t26 - t217*t45 + t218*t22 - t22*t270 + t224*t26 - t271*t50 - Rational_2_3*t51*trK_dD2 - t54*(6.0*t138 + 6.0*t139 + 6.0*t141 + t143*t213 + t145*t214 + t146*t215);
  diag[3 * Ntot + idx] = t0*t273;
  const double t274 = (cf*cf*cf*cf);
  const double t275 = hDD01*t30;
  const double t276 = t272*t274;
  const double t277 = 2.0*t24;
  const double t278 = hDD02*t64;
  diag[4 * Ntot + idx] = t107*(t2*(t272*t272)*t274 + (t269*t269)*t274*t4 + t269*t273*t274*t278 + t269*t275*t276 + (t273*t273)*t274*t7 + t273*t276*t277);
  const double t279 = (1.0 / f0_of_xx0__D0);
  const double t280 = f0_of_xx0*t279;
  const double t281 = 2.0*t13;
  const double t282 = t19*t281;
  const double t283 = t26*t281;
  const double t284 = t22*t281;
  const double lambdaU0 = in[17 * Ntot + idx];
  const double t285 = lambdaU0*t279 - t104*t284 - t282*t91 - t283*t97 - t34*(-f0_of_xx0__DD00*t279 + t66) - t46*(t280 + t77) - t51*(t280*t5 + t44);
  const double t286 = (1.0 / f0_of_xx0);
  const double t287 = -f0_of_xx0__D0*t286;
  const double lambdaU1 = in[18 * Ntot + idx];
  const double t288 = lambdaU1*t286 - t105*t284 - t282*(t287 + t92) - t283*t99 - t34*t67 - t46*t78 - t51*(t36 + t49);
  const double t289 = (1.0 / f1_of_xx1);
  const double lambdaU2 = in[19 * Ntot + idx];
  const double t290 = lambdaU2*t286*t289 - t282*t93 - t283*(-f1_of_xx1__D1*t289 + t100) - t284*(t106 + t287) - t34*t68 - t46*t79 - t51*t53;
  diag[5 * Ntot + idx] = sqrt(t2*(t288*t288) + t275*t285*t288 + t277*t288*t290 + t278*t285*t290 + (t285*t285)*t4 + (t290*t290)*t7);
}

extern "C" __global__ void __launch_bounds__(256)
bssn_initial_lambda_SinhSpherical_symnone_KO1_fd4(double *gfs, const double *__restrict__ rfm0, const double *__restrict__ rfm1,
                          const bhah_kparams p) {
  const double *in = gfs;
  const int i0 = p.NG + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int i1 = p.NG + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  const int i2 = p.NG + (int)blockIdx.z;
  if (i0 >= p.Nx0 - p.NG || i1 >= p.Nx1 - p.NG) return;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;

  const double f1_of_xx1 = rfm1[i1];
  const double t0 = (f1_of_xx1*f1_of_xx1);
  const double f0_of_xx0__D0 = rfm0[p.Nx0 + i0];
  const double t1 = (1.0 / f0_of_xx0__D0);
  const double f0_of_xx0 = rfm0[i0];
  const double t3 = (f0_of_xx0*f0_of_xx0);
  const double hDD11 = in[14 * Ntot + idx];
  const double t10 = hDD11*t3 + t3;
  const double t4 = t0*t3;
  const double hDD22 = in[16 * Ntot + idx];
  const double t13 = hDD22*t4 + t4;
  const double t15 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double hDD12 = in[15 * Ntot + idx];
  const double t16 = (hDD12*hDD12)*t0*t15;
  const double t11 = (f0_of_xx0__D0*f0_of_xx0__D0);
  const double hDD00 = in[11 * Ntot + idx];
  const double t12 = hDD00*t11 + t11;
  const double hDD01 = in[12 * Ntot + idx];
  const double t14 = (hDD01*hDD01)*t11*t3;
  const double hDD02 = in[13 * Ntot + idx];
  const double t17 = (hDD02*hDD02)*t11*t4;
  const double t18 = (1.0 / (2.0*hDD01*hDD02*hDD12*t0*t11*t15 + t10*t12*t13 - t10*t17 - t12*t16 - t13*t14));
  const double t19 = t18*(t10*t13 - t16);
  const double t2 = f0_of_xx0*t1;
  const double t20 = (Rational_1_2)*t19;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t21 = f1_of_xx1*f1_of_xx1__D1;
  const double t22 = 2.0*t3;
  const double t23 = t21*t22;
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t24 = hDD22*t23 + hDD_dD221*t4 + t23;
  const double hDD_dD122 = p.invdxx2 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s2)] - in[15 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s2)] - in[15 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t25 = 2.0*f1_of_xx1*hDD_dD122*t3 - t24;
  const double t26 = f0_of_xx0*f0_of_xx0__D0;
  const double t27 = (f0_of_xx0*f0_of_xx0*f0_of_xx0)*f0_of_xx0__D0;
  const double t28 = -hDD01*t13*t26 + hDD02*hDD12*t0*t27;
  const double t29 = (Rational_1_2)*t18;
  const double t30 = t28*t29;
  const double t31 = f1_of_xx1*t26;
  const double t32 = f1_of_xx1*hDD01*hDD12*t27 - hDD02*t10*t31;
  const double t33 = t29*t32;
  const double hDD_dD222 = p.invdxx2 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s2)] - in[16 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s2)] - in[16 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t34 = hDD_dD222*t4;
  const double t35 = t18*(t10*t12 - t14);
  const double t5 = 2.0*f0_of_xx0__D0;
  const double f0_of_xx0__DD00 = rfm0[2 * p.Nx0 + i0];
  const double t36 = f0_of_xx0__DD00*t5;
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t37 = hDD00*t36 + hDD_dD000*t11 + t36;
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t38 = hDD_dD001*t11;
  const double t39 = f0_of_xx0*f0_of_xx0__DD00;
  const double t6 = f0_of_xx0*t5;
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t40 = 2.0*hDD01*(t11 + t39) + hDD_dD010*t6 - t38;
  const double hDD_dD002 = p.invdxx2 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s2)] - in[11 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s2)] - in[11 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t41 = hDD_dD002*t11;
  const double t42 = f1_of_xx1*t11;
  const double t43 = f1_of_xx1*t6;
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t44 = 2.0*hDD02*(f1_of_xx1*t39 + t42) + hDD_dD020*t43 - t41;
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t45 = hDD11*t6 + hDD_dD110*t3 + t6;
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t46 = 2.0*f0_of_xx0*f0_of_xx0__D0*hDD_dD011 - t45;
  const double hDD_dD112 = p.invdxx2 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s2)] - in[14 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s2)] - in[14 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t47 = hDD_dD112*t3;
  const double t48 = f1_of_xx1*t3;
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t49 = f1_of_xx1__D1*hDD12*t22 + 2.0*hDD_dD121*t48 - t47;
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t50 = hDD_dD111*t3;
  const double t51 = t18*(t12*t13 - t17);
  const double hDD_dD012 = p.invdxx2 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s2)] - in[12 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s2)] - in[12 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t52 = hDD_dD012*t26;
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t53 = hDD_dD021*t31;
  const double t54 = f1_of_xx1__D1*hDD02*t26;
  const double t55 = t53 + t54;
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t56 = hDD_dD120*t48;
  const double t57 = hDD12*t43;
  const double t58 = t56 + t57;
  const double t59 = -t52 + t55 + t58;
  const double t60 = 2.0*t18;
  const double t61 = t28*t60;
  const double t62 = t52 + t55 - t56 - t57;
  const double t63 = hDD01*hDD02*t3*t42 - hDD12*t12*t48;
  const double t64 = t60*t63;
  const double t65 = t52 - t53 - t54 + t58;
  const double t66 = t32*t60;
  const double t7 = t0*t6;
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t8 = hDD22*t7 + hDD_dD220*t4 + t7;
  const double hDD_dD022 = p.invdxx2 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s2)] - in[13 * Ntot + idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s2)] - in[13 * Ntot + idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t9 = 2.0*f0_of_xx0*f0_of_xx0__D0*f1_of_xx1*hDD_dD022 - t8;
  gfs[17 * Ntot + idx] = f0_of_xx0__D0*(t19*(-f0_of_xx0__DD00*t1 + t20*t37 + t30*t40 + t33*t44) + t35*(t0*t2 + t20*t9 + t25*t30 + t33*t34) + t51*(t2 + t20*t46 + t30*t50 + t33*t49) + t61*(t20*t38 + t30*t45 + t33*t59) + t64*(t20*t62 + t24*t33 + t30*t47) + t66*(t20*t41 + t30*t65 + t33*t8));
  const double t67 = (Rational_1_2)*t51;
  const double t68 = t29*t63;
  const double t69 = -f0_of_xx0__D0/f0_of_xx0;
  gfs[18 * Ntot + idx] = f0_of_xx0*(t19*(t30*t37 + t40*t67 + t44*t68) + t35*(t21 + t25*t67 + t30*t9 + t34*t68) + t51*(t30*t46 + t49*t68 + t50*t67) + t61*(t30*t38 + t45*t67 + t59*t68 + t69) + t64*(t24*t68 + t30*t62 + t47*t67) + t66*(t30*t41 + t65*t67 + t68*t8));
  const double t70 = (Rational_1_2)*t35;
  gfs[19 * Ntot + idx] = f0_of_xx0*f1_of_xx1*(t19*(t33*t37 + t40*t68 + t44*t70) + t35*(t25*t68 + t33*t9 + t34*t70) + t51*(t33*t46 + t49*t70 + t50*t68) + t61*(t33*t38 + t45*t68 + t59*t70) + t64*(t24*t70 + t33*t62 + t47*t68 - f1_of_xx1__D1/f1_of_xx1) + t66*(t33*t41 + t65*t68 + t69 + t70*t8));
}
#undef Rational_1_2
#undef Rational_2_3

template <bool KEEP, typename K>
static hipError_t rk_det_launch_SinhSpherical_symnone_KO1_fd4(hipStream_t s, K *kin, const double *y_n, double *y_run, double *out,
    const double *rfm0, const double *rfm1, const bhah_kparams &p, const int2 *map, const int2 *pairs) {
  const int np = (!(p.Ntot & 1) && !((reinterpret_cast<uintptr_t>(kin) | reinterpret_cast<uintptr_t>(y_n) |
                                      reinterpret_cast<uintptr_t>(y_run) | reinterpret_cast<uintptr_t>(out)) & 15))
                     ? 2
                     : 1;
  const long units = p.Ntot / np;
  // 256 threads a workgroup where that gives every CU several; 64 on small grids
  const unsigned nt = units >= (1L << 17) ? 256 : 64;
  const dim3 g(4u * (unsigned)((units + nt - 1) / nt));
  // The running sum is not read again before the next substep, so it always streams past the
  // caches.  The other arrays are read by the next kernels: caching them gains while a good part
  // of them stays in the 256 MB last-level cache.  What counts is the interior (an inner ghost
  // point takes the k of an interior one): streaming against caching, per step, takes 1.12 / 1.09 /
  // 1.04 / 0.99 / 0.96 at 256 x 64 x 16 / 20 / 24 and 256 x 96 x 20 / 24 points phi-symmetric (262,000 to
  // 590,000 interior points), 1.04 / 0.95 at 800x96x4 / 1200x128x4, 1.04 / 0.98 at 1600x128x2 /
  // 2400x192x2; 1.06 / 1.01 / 0.997 / 0.98 / 0.96 at 112, 120, 128, 136 x half x half and 160x80x80 fd4;
  // 1.024 / 1.005 / 0.990 / 0.96 / 0.98 / 0.99 at 112x56x56, 120x60x60, 127x63x62, 160x80x80,
  // 192x96x96, 224x112x112 fd6.  Above 2.6 million phi-symmetric or fd4 points it is within 1.2%
  // either way.
  const long interior = (long)(p.Nx0 - 2 * p.NG) * (p.Nx1 - 2 * p.NG) * (p.Nx2 - 2 * p.NG);
  const bool nt_all = interior > 470000;
#define RK_LAUNCH(NP_, IN_, NT_)                                                                                     \
  if (np == NP_ && (map != nullptr) == IN_ && nt_all == NT_)                                                         \
    hipLaunchKernelGGL((bssn_rk_det_SinhSpherical_symnone_KO1_fd4<NP_, IN_, NT_, KEEP>), g, dim3(nt), 0, s, kin, y_n, y_run, out, rfm0, rfm1, p,   \
                       map, pairs)
  if constexpr (!KEEP) {
    RK_LAUNCH(1, false, false);
    RK_LAUNCH(1, false, true);
    RK_LAUNCH(2, false, false);
    RK_LAUNCH(2, false, true);
  }
  RK_LAUNCH(1, true, false);
  RK_LAUNCH(1, true, true);
  RK_LAUNCH(2, true, false);
  RK_LAUNCH(2, true, true);
#undef RK_LAUNCH
  return hipGetLastError();
}
extern "C" hipError_t launch_bssn_rk_det_SinhSpherical_symnone_KO1_fd4(hipStream_t s, const double *kin, const double *y_n, double *y_run,
    double *out, const double *rfm0, const double *rfm1, bhah_kparams p) {
  return rk_det_launch_SinhSpherical_symnone_KO1_fd4<false>(s, kin, y_n, y_run, out, rfm0, rfm1, p, nullptr, nullptr);
}
// The RK pass with the inner boundary condition folded in.
extern "C" hipError_t launch_bssn_rk_det_inner_SinhSpherical_symnone_KO1_fd4(hipStream_t s, const double *kin, const double *y_n,
    double *y_run, double *out, const double *rfm0, const double *rfm1, bhah_kparams p, const int *map,
    const int *pairs) {
  return rk_det_launch_SinhSpherical_symnone_KO1_fd4<false>(s, kin, y_n, y_run, out, rfm0, rfm1, p, reinterpret_cast<const int2 *>(map),
                                    reinterpret_cast<const int2 *>(pairs));
}

// Host-side launchers (one translation unit per variant; no relocatable device code needed).
extern "C" hipError_t launch_bssn_constraints_SinhSpherical_symnone_KO1_fd4(dim3 g, dim3 b, hipStream_t s, const double *in,
    const double *aux, double *diag, const double *rfm0, const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_constraints_SinhSpherical_symnone_KO1_fd4, g, b, 0, s, in, aux, diag, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_bssn_detgamma_SinhSpherical_symnone_KO1_fd4(dim3 g, dim3 b, hipStream_t s, double *gfs, const double *rfm0,
    const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_detgamma_SinhSpherical_symnone_KO1_fd4, g, b, 0, s, gfs, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_bssn_initial_lambda_SinhSpherical_symnone_KO1_fd4(dim3 g, dim3 b, hipStream_t s, double *gfs, const double *rfm0,
    const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_initial_lambda_SinhSpherical_symnone_KO1_fd4, g, b, 0, s, gfs, rfm0, rfm1, p);
  return hipGetLastError();
}
