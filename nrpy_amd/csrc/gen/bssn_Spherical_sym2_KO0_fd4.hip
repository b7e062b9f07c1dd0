// Generated by nrpy_amd/codegen/hip_gen.py -- do not edit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "../bhah_device_types.h"
// ---- BSSN kernels: Spherical, symmetry axes '2', KO=False, fd_order=4
#define Rational_1_2 (1.0 / 2.0)
#define Rational_2_3 (2.0 / 3.0)

typedef double bhah_d2 __attribute__((ext_vector_type(2)));
namespace rk_Spherical_sym2_KO0_fd4 {
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
    const double f1_of_xx1 = rfm1[i1];
    const double dg0 = (f0_of_xx0*f0_of_xx0);
    const double dg1 = (f1_of_xx1*f1_of_xx1);
    const double dg2 = dg0*dg1;
    const double dg3 = dg2*hDD22 + dg2;
    const double dg4 = hDD00 + 1.0;
    const double dg5 = dg0*hDD11 + dg0;
    const double dg6 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
    const double dg7 = dg1*dg6;
    const double dg8 = cbrt(fabs(dg7)/(-dg0*dg3*(hDD01*hDD01) + 2.0*dg1*dg6*hDD01*hDD02*hDD12 - dg2*dg5*(hDD02*hDD02) + dg3*dg4*dg5 - dg4*dg7*(hDD12*hDD12)));
    const double new_hDD00 = dg4*dg8 - 1.0;
    const double new_hDD01 = dg8*hDD01;
    const double new_hDD02 = dg8*hDD02;
    const double new_hDD11 = dg8*(hDD11 + 1.0) - 1.0;
    const double new_hDD12 = dg8*hDD12;
    const double new_hDD22 = dg8*(hDD22 + 1.0) - 1.0;
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
}  // namespace rk_Spherical_sym2_KO0_fd4
template <int NP, bool INNER, bool NT, bool KEEP>
__global__ void __launch_bounds__(256)
bssn_rk_det_Spherical_sym2_KO0_fd4(rk_Spherical_sym2_KO0_fd4::k_ptr<INNER, KEEP> kin, const double *y_n, double *y_run, double *out,
                  const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p,
                  const int2 *__restrict__ map, const int2 *__restrict__ pairs) {
  rk_Spherical_sym2_KO0_fd4::any_group<NP, INNER, NT, KEEP>((int)(blockIdx.x & 3u), kin, y_n, y_run, out, rfm0, rfm1, p, map, pairs,
                                 (long)(blockIdx.x >> 2) * blockDim.x + threadIdx.x);
}

// Records are (member, chunk): 256 consecutive units of NP points of the member's arrays, in array
// order; each is walked by four consecutive workgroups, one per group of gridfunctions.
// No form that streams the stage arrays: it loses at every total (per step, streamed against cached, 1.01 /
// 1.006 / 1.03 / 1.04 / 1.06 / 1.07 for 32, 64, 80, 96, 128 and 256 members of 0.7 to 6.2 GB).
template <int NP>
__global__ void __launch_bounds__(256)
bssn_ens_rk_det_Spherical_sym2_KO0_fd4(const bhah_member *__restrict__ mem, const bhah_item *__restrict__ items, const int nitems,
                      const int k_sel, const int out_sel, const int substep) {
  for (int it = blockIdx.x; it < 4 * nitems; it += gridDim.x) {
    const bhah_item w = items[it >> 2];
    const bhah_member *M = &mem[w.m];
    bhah_kparams p = M->kp;
    p.substep = substep;
    rk_Spherical_sym2_KO0_fd4::any_group<NP, true, false, false>(it & 3, M->arr[k_sel], M->arr[0], M->arr[1], M->arr[out_sel], M->rfm0, M->rfm1, p,
                                  reinterpret_cast<const int2 *>(M->inner_map),
                                  reinterpret_cast<const int2 *>(M->inner_pairs), (long)w.bx * 256 + threadIdx.x);
  }
}

extern "C" __global__ void __launch_bounds__(256)
bssn_detgamma_Spherical_sym2_KO0_fd4(double *__restrict__ gfs, const double *__restrict__ rfm0, const double *__restrict__ rfm1,
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
    const double f1_of_xx1 = rfm1[i1];
    const double dg0 = (f0_of_xx0*f0_of_xx0);
    const double dg1 = (f1_of_xx1*f1_of_xx1);
    const double dg2 = dg0*dg1;
    const double dg3 = dg2*hDD22 + dg2;
    const double dg4 = hDD00 + 1.0;
    const double dg5 = dg0*hDD11 + dg0;
    const double dg6 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
    const double dg7 = dg1*dg6;
    const double dg8 = cbrt(fabs(dg7)/(-dg0*dg3*(hDD01*hDD01) + 2.0*dg1*dg6*hDD01*hDD02*hDD12 - dg2*dg5*(hDD02*hDD02) + dg3*dg4*dg5 - dg4*dg7*(hDD12*hDD12)));
    const double new_hDD00 = dg4*dg8 - 1.0;
    const double new_hDD01 = dg8*hDD01;
    const double new_hDD02 = dg8*hDD02;
    const double new_hDD11 = dg8*(hDD11 + 1.0) - 1.0;
    const double new_hDD12 = dg8*hDD12;
    const double new_hDD22 = dg8*(hDD22 + 1.0) - 1.0;
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
bssn_constraints_Spherical_sym2_KO0_fd4(const double *__restrict__ in, const double *__restrict__ aux, double *__restrict__ diag,
                       const double *__restrict__ rfm0, const double *__restrict__ rfm1, const bhah_kparams p) {
  const int i0 = p.NG + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int i1 = p.NG + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  const int i2 = p.NG + (int)blockIdx.z;
  if (i0 >= p.Nx0 - p.NG || i1 >= p.Nx1 - p.NG) return;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;

  const double cf = in[10 * Ntot + idx];
  const double t41 = (cf*cf);
  const double t100 = (1.0 / t41);
  const double t101 = 2.0*t100;
  const double f0_of_xx0 = rfm0[i0];
  const double t0 = (f0_of_xx0*f0_of_xx0);
  const double hDD11 = in[14 * Ntot + idx];
  const double t1 = hDD11*t0 + t0;
  const double hDD00 = in[11 * Ntot + idx];
  const double t10 = hDD00 + 1.0;
  const double f1_of_xx1 = rfm1[i1];
  const double t2 = (f1_of_xx1*f1_of_xx1);
  const double t3 = t0*t2;
  const double hDD02 = in[13 * Ntot + idx];
  const double t11 = (hDD02*hDD02)*t3;
  const double hDD22 = in[16 * Ntot + idx];
  const double t4 = hDD22*t3 + t3;
  const double t5 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double hDD12 = in[15 * Ntot + idx];
  const double t6 = (hDD12*hDD12)*t2*t5;
  const double hDD01 = in[12 * Ntot + idx];
  const double t9 = (hDD01*hDD01)*t0;
  const double t12 = 2.0*hDD01*hDD02*hDD12*t2*t5 + t1*t10*t4 - t1*t11 - t10*t6 - t4*t9;
  const double t13 = (1.0 / (t12*t12));
  const double aDD00 = in[idx];
  const double t14 = aDD00*t13;
  const double t17 = (f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double t18 = -f0_of_xx0*hDD01*t4 + hDD02*hDD12*t17*t2;
  const double t19 = (t18*t18);
  const double t102 = t14*t19;
  const double t43 = t10*t4 - t11;
  const double t103 = t13*(t43*t43);
  const double aDD11 = in[3 * Ntot + idx];
  const double t16 = aDD11*t0;
  const double t104 = t103*t16;
  const double t38 = f1_of_xx1*t0;
  const double t45 = hDD12*t38;
  const double t46 = hDD01*hDD02*t38 - t10*t45;
  const double t105 = t13*(t46*t46);
  const double aDD22 = in[5 * Ntot + idx];
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
  const double aDD01 = in[1 * Ntot + idx];
  const double t114 = aDD01*f0_of_xx0;
  const double t20 = t13*t19;
  const double t115 = t114*t20;
  const double t116 = t107*t7;
  const double t117 = t114*t116;
  const double t118 = t108*t16;
  const double aDD02 = in[2 * Ntot + idx];
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
  const double aDD12 = in[4 * Ntot + idx];
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
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t48 = hDD22*t47 + hDD_dD220*t3 + t47;
  const double t49 = -t48;
  const double t51 = (Rational_1_2)*t50;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t52 = f1_of_xx1*f1_of_xx1__D1;
  const double t53 = 2.0*t0*t52;
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t54 = hDD22*t53 + hDD_dD221*t3 + t53;
  const double t55 = -t54;
  const double t56 = (Rational_1_2)*t42;
  const double t57 = t18*t56;
  const double t58 = t49*t51 + t55*t57;
  const double t59 = (1.0 / cf);
  const double cf_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1)] - in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] - in[10 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t60 = (Rational_1_2)*cf_dD0*t59;
  const double t61 = t42*t43;
  const double t62 = (Rational_1_2)*t61;
  const double t63 = t49*t57 + t55*t62;
  const double t64 = (Rational_1_2)*t59;
  const double cf_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] - in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] - in[10 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t65 = cf_dD1*t64;
  const double t66 = t42*t44;
  const double t67 = (cf_dD1*cf_dD1);
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t68 = hDD11*t29 + hDD_dD110*t0 + t29;
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t69 = 2.0*f0_of_xx0*hDD_dD011 - t68;
  const double t70 = f1_of_xx1__D1*t0;
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t71 = 2.0*hDD12*t70 + hDD_dD121*t39;
  const double t72 = t56*t71;
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t73 = hDD_dD111*t0;
  const double t74 = t24*t72 + t51*t69 + t57*t73;
  const double t75 = t46*t72 + t57*t69 + t62*t73;
  const double t76 = (cf_dD0*cf_dD0);
  const double t77 = f1_of_xx1*hDD02;
  const double t78 = f1_of_xx1*t29;
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t79 = hDD_dD020*t78 + 2.0*t77;
  const double t80 = t56*t79;
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t81 = 2.0*hDD01 - hDD_dD001 + hDD_dD010*t29;
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t82 = hDD_dD000*t51 + t24*t80 + t57*t81;
  const double t83 = hDD_dD000*t57 + t46*t80 + t62*t81;
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t84 = hDD_dD120*t38 + t22*t29;
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
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
  const double cf_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[10 * Ntot + idx] + (4.0 / 3.0) * (in[10 * Ntot + idx + (1)] + in[10 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2)] + in[10 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double cf_dDD01 = p.invdxx0 * p.invdxx1 * ((4.0 / 9.0) * ((in[10 * Ntot + idx + (1 + 1 * s1)] - in[10 * Ntot + idx + (1 + -1 * s1)]) - (in[10 * Ntot + idx + (-1 + 1 * s1)] - in[10 * Ntot + idx + (-1 + -1 * s1)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (1 + 2 * s1)] - in[10 * Ntot + idx + (1 + -2 * s1)]) - (in[10 * Ntot + idx + (-1 + 2 * s1)] - in[10 * Ntot + idx + (-1 + -2 * s1)])) + (-1.0 / 18.0) * ((in[10 * Ntot + idx + (2 + 1 * s1)] - in[10 * Ntot + idx + (2 + -1 * s1)]) - (in[10 * Ntot + idx + (-2 + 1 * s1)] - in[10 * Ntot + idx + (-2 + -1 * s1)])) + (1.0 / 144.0) * ((in[10 * Ntot + idx + (2 + 2 * s1)] - in[10 * Ntot + idx + (2 + -2 * s1)]) - (in[10 * Ntot + idx + (-2 + 2 * s1)] - in[10 * Ntot + idx + (-2 + -2 * s1)])));
  __builtin_amdgcn_sched_barrier(0);
  const double cf_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[10 * Ntot + idx] + (4.0 / 3.0) * (in[10 * Ntot + idx + (1 * s1)] + in[10 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[10 * Ntot + idx + (2 * s1)] + in[10 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double trK = in[20 * Ntot + idx];
  diag[0 * Ntot + idx] = -aDD00*(t15 + t21 + t28 + t30*t32 + t33*t35 + t37*t40) - t16*(t102 + t104 + t106 + t108*t30 + t110*t35 + t111*t40) - t27*(t105*t16 + t127*t30 + t129*t13*t27 + t131*t35 + t132*t40 + t14*t25) - t30*(t113 + t115 + t117 + t118 + t121 + t122 + t125 + t126 + t128) - t35*(t133 + t134 + t135 + t136 + t137 + t139 + t141 + t142 + t143) - t40*(t144 + t145 + t146 + t147 + t148 + t149 + t150 + t152 + t153) + t41*(RbarDD00*t42*t7 + 2.0*RbarDD01*t18*t42 + 2.0*RbarDD02*t24*t42 + RbarDD11*t42*t43 + 2.0*RbarDD12*t42*t46 + RbarDD22*t42*t44 - 4.0*cf_dD0*cf_dD1*t100*t89 - t101*t50*t76 - t101*t61*t67 - t24*t91*(t60*t93 + t65*t94) - t46*t91*(t60*t88 + t65*t90) - 8.0*t50*(t60*t82 + t64*(-cf_dDD00 + t59*t76) + t65*t83) - 8.0*t61*(t60*t74 + t64*(-cf_dDD11 + t59*t67) + t65*t75) - 8.0*t66*(t58*t60 + t63*t65) - 16.0*t89*(t60*t98 + t64*(cf_dD0*cf_dD1*t59 - cf_dDD01) + t65*t99)) + (Rational_2_3)*(trK*trK);
  const double t154 = -t82;
  const double t155 = -t83;
  const double t156 = t24*t56;
  const double t157 = (Rational_1_2)*t66;
  const double t158 = t46*t56;
  const double t159 = hDD_dD000*t156 + t157*t79 + t158*t81;
  const double t160 = -t159;
  const double aDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[idx + (1)] - in[idx + (-1)]) + (-1.0 / 12.0) * (in[idx + (2)] - in[idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t161 = t13*(aDD00*t154 - aDD00*t82 + aDD_dD000 + t114*t155 - t114*t83 - t119*t159 + t119*t160);
  const double t162 = -t74;
  const double aDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[1 * Ntot + idx + (1 * s1)] - in[1 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[1 * Ntot + idx + (2 * s1)] - in[1 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
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
  const double aDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[3 * Ntot + idx + (1)] - in[3 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[3 * Ntot + idx + (2)] - in[3 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
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
  const double aDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[5 * Ntot + idx + (1)] - in[5 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[5 * Ntot + idx + (2)] - in[5 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t185 = aDD22*t47 + aDD_dD220*t3 + t119*t182 + t123*t183 + t180 + t184*t27;
  const double trK_dD0 = p.invdxx0 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1)] - in[20 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2)] - in[20 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t186 = (Rational_2_3)*trK_dD0;
  const double trK_dD1 = p.invdxx1 * ((2.0 / 3.0) * (in[20 * Ntot + idx + (1 * s1)] - in[20 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[20 * Ntot + idx + (2 * s1)] - in[20 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
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
  const double aDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[3 * Ntot + idx + (1 * s1)] - in[3 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[3 * Ntot + idx + (2 * s1)] - in[3 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t202 = aDD_dD111*t0 + t114*t162 - t114*t74 - t123*t165 + t123*t166 + t16*t164 - t16*t75;
  const double t203 = t114*t193 + t123*t197 + t16*t194;
  const double aDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[4 * Ntot + idx + (1 * s1)] - in[4 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[4 * Ntot + idx + (2 * s1)] - in[4 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t204 = aDD12*t70 + aDD_dD121*t38;
  const double t205 = -t119*t74 - t123*t75 - t165*t27 + t203 + t204;
  const double t206 = t107*t205;
  const double t207 = aDD00*t170 + t114*t171 + t119*t172;
  const double t208 = -aDD00*t98 - t114*t99 - t119*t167;
  const double aDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[idx + (1 * s1)] - in[idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[idx + (2 * s1)] - in[idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t209 = aDD_dD001 + t207 + t208;
  const double aDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[1 * Ntot + idx + (1)] - in[1 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[1 * Ntot + idx + (2)] - in[1 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t210 = aDD01 + aDD_dD010*f0_of_xx0;
  const double t211 = -t114*t82 - t123*t159 - t16*t83 + t207 + t210;
  const double t212 = t114*t154 + t123*t160 + t155*t16 + t208 + t210;
  const double t213 = aDD00*t88;
  const double t214 = t114*t90;
  const double t215 = t119*t196;
  const double t216 = aDD01*f0_of_xx0*t182 + aDD11*t0*t183 + aDD12*f1_of_xx1*t0*t184 - t213 - t214 - t215;
  const double aDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[2 * Ntot + idx + (1 * s1)] - in[2 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[2 * Ntot + idx + (2 * s1)] - in[2 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t217 = aDD02*t95 + aDD_dD021*t23;
  const double t218 = t119*t170 + t123*t171 + t172*t27;
  const double t219 = -t213 - t214 - t215 + t217 + t218;
  const double t220 = aDD00*t182 + t114*t183 + t119*t184;
  const double t221 = -aDD00*t93 - t114*t94 - t119*t179;
  const double t222 = t220 + t221;
  const double aDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[2 * Ntot + idx + (1)] - in[2 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[2 * Ntot + idx + (2)] - in[2 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
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
  const double aDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[4 * Ntot + idx + (1)] - in[4 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[4 * Ntot + idx + (2)] - in[4 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t234 = aDD12*t78 + aDD_dD120*t38;
  const double t235 = t114*t182 + t123*t184 + t16*t183 + t232 + t234;
  const double t236 = t218 + t230 + t234;
  const double t237 = -t119*t88 - t123*t90 - t196*t27;
  const double t238 = t114*t175 + t123*t178 + t16*t176 + t237;
  const double aDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[5 * Ntot + idx + (1 * s1)] - in[5 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[5 * Ntot + idx + (2 * s1)] - in[5 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t239 = aDD22*t53 + aDD_dD221*t3 + t119*t193 + t123*t194 + t197*t27 + t237;
  const double t240 = t108*t202 + t110*t227 + t110*t228 + t116*t201 + t120*t216 + t120*t219 + t127*t238 + t127*t239 + t161*t8 + t169*t20 + t174*t20 + t18*t198 + t181*t26 + t185*t26 - t186*t50 - t187*t89 - t191*t65 + t192*t7 + t200*t24 + t206*t24 + t209*t32 + t211*t32 + t212*t32 + t222*t33 + t224*t33 + t225*t33 + t231*t37 + t233*t37 + t235*t37 + t236*t37 - t60*(6.0*t15 + t188*t32 + t189*t33 + t190*t37 + 6.0*t21 + 6.0*t28);
  diag[1 * Ntot + idx] = t240*t41;
  const double t241 = t161*t7;
  const double t242 = t103*t202 + t105*t238 + t105*t239 + t108*t169 + t108*t174 + t108*t201 + t110*t216 + t110*t219 + t110*t233 + t110*t235 + t111*t227 + t111*t228 + t116*t211 + t120*t224 + t124*t231 + t124*t236 + t127*t181 + t127*t185 + t18*t192 + t18*t241 - t186*t89 - t187*t61 - t191*t60 + t198*t43 + t20*t209 + t20*t212 + t200*t46 + t206*t46 + t222*t37 + t225*t37 - t65*(6.0*t102 + 6.0*t104 + 6.0*t106 + t108*t188 + t110*t189 + t111*t190);
  diag[2 * Ntot + idx] = t242*t41;
  const double t243 = t105*t227 + t105*t228 + t110*t169 + t110*t174 + t111*t202 + t120*t211 + t124*t201 + t127*t216 + t127*t219 + t127*t231 + t127*t236 + t129*t199 + t131*t181 + t131*t185 + t132*t238 + t132*t239 + t138*t224 + t140*t233 + t140*t235 + t151*t205 - t186*t195 - t187*t42*t46 + t192*t24 + t198*t46 + t209*t37 + t212*t37 + t222*t26 + t225*t26 + t24*t241 - t60*(6.0*t133 + 6.0*t134 + 6.0*t135 + 6.0*t136 + 6.0*t137 + 6.0*t139 + 6.0*t141 + 6.0*t142 + 6.0*t143) - t65*(6.0*t144 + 6.0*t145 + 6.0*t146 + 6.0*t147 + 6.0*t148 + 6.0*t149 + 6.0*t150 + 6.0*t152 + 6.0*t153);
  diag[3 * Ntot + idx] = t243*t41;
  const double t244 = (cf*cf*cf*cf);
  const double t245 = hDD01*t29;
  const double t246 = t240*t244;
  const double t247 = t29*t77;
  const double t248 = 2.0*t45;
  diag[4 * Ntot + idx] = t100*(t1*(t242*t242)*t244 + t10*(t240*t240)*t244 + t242*t243*t244*t248 + t242*t245*t246 + (t243*t243)*t244*t4 + t243*t246*t247);
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
  diag[5 * Ntot + idx] = sqrt(t1*(t256*t256) + t10*(t253*t253) + t245*t253*t256 + t247*t253*t258 + t248*t256*t258 + (t258*t258)*t4);
}

extern "C" __global__ void __launch_bounds__(256)
bssn_initial_lambda_Spherical_sym2_KO0_fd4(double *gfs, const double *__restrict__ rfm0, const double *__restrict__ rfm1,
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
  const double f0_of_xx0 = rfm0[i0];
  const double t1 = f0_of_xx0*t0;
  const double t3 = (f0_of_xx0*f0_of_xx0);
  const double hDD11 = in[14 * Ntot + idx];
  const double t10 = hDD11*t3 + t3;
  const double t12 = (f0_of_xx0*f0_of_xx0*f0_of_xx0*f0_of_xx0);
  const double hDD12 = in[15 * Ntot + idx];
  const double t13 = (hDD12*hDD12)*t0*t12;
  const double t4 = t0*t3;
  const double hDD02 = in[13 * Ntot + idx];
  const double t11 = (hDD02*hDD02)*t4;
  const double hDD22 = in[16 * Ntot + idx];
  const double t7 = hDD22*t4 + t4;
  const double hDD01 = in[12 * Ntot + idx];
  const double t8 = (hDD01*hDD01)*t3;
  const double hDD00 = in[11 * Ntot + idx];
  const double t9 = hDD00 + 1.0;
  const double t14 = (1.0 / (2.0*hDD01*hDD02*hDD12*t0*t12 - t10*t11 + t10*t7*t9 - t13*t9 - t7*t8));
  const double t15 = t14*(t10*t7 - t13);
  const double t16 = (Rational_1_2)*t15;
  const double f1_of_xx1__D1 = rfm1[p.Nx1 + i1];
  const double t17 = f1_of_xx1*f1_of_xx1__D1;
  const double t18 = 2.0*t3;
  const double t19 = t17*t18;
  const double hDD_dD221 = p.invdxx1 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1 * s1)] - in[16 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2 * s1)] - in[16 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t20 = hDD22*t19 + hDD_dD221*t4 + t19;
  const double t21 = -t20;
  const double t22 = (f0_of_xx0*f0_of_xx0*f0_of_xx0)*hDD12;
  const double t23 = -f0_of_xx0*hDD01*t7 + hDD02*t0*t22;
  const double t24 = (Rational_1_2)*t14;
  const double t25 = t23*t24;
  const double t26 = t14*(t10*t9 - t8);
  const double t27 = 2.0*f0_of_xx0;
  const double hDD_dD110 = p.invdxx0 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1)] - in[14 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2)] - in[14 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t28 = hDD11*t27 + hDD_dD110*t3 + t27;
  const double hDD_dD011 = p.invdxx1 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1 * s1)] - in[12 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2 * s1)] - in[12 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t29 = 2.0*f0_of_xx0*hDD_dD011 - t28;
  const double t30 = 2.0*f1_of_xx1;
  const double hDD_dD121 = p.invdxx1 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1 * s1)] - in[15 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2 * s1)] - in[15 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t31 = f1_of_xx1__D1*hDD12*t18 + hDD_dD121*t3*t30;
  const double t32 = f0_of_xx0*f1_of_xx1;
  const double t33 = f1_of_xx1*hDD01*t22 - hDD02*t10*t32;
  const double t34 = t24*t33;
  const double hDD_dD111 = p.invdxx1 * ((2.0 / 3.0) * (in[14 * Ntot + idx + (1 * s1)] - in[14 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[14 * Ntot + idx + (2 * s1)] - in[14 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t35 = hDD_dD111*t3;
  const double t36 = t14*(-t11 + t7*t9);
  const double t37 = f1_of_xx1*t27;
  const double hDD_dD020 = p.invdxx0 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1)] - in[13 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2)] - in[13 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t38 = hDD02*t30 + hDD_dD020*t37;
  const double hDD_dD001 = p.invdxx1 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1 * s1)] - in[11 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2 * s1)] - in[11 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double hDD_dD010 = p.invdxx0 * ((2.0 / 3.0) * (in[12 * Ntot + idx + (1)] - in[12 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[12 * Ntot + idx + (2)] - in[12 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t39 = 2.0*hDD01 - hDD_dD001 + hDD_dD010*t27;
  const double t40 = f1_of_xx1*t3;
  const double hDD_dD120 = p.invdxx0 * ((2.0 / 3.0) * (in[15 * Ntot + idx + (1)] - in[15 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[15 * Ntot + idx + (2)] - in[15 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t41 = hDD12*t37 + hDD_dD120*t40;
  const double hDD_dD021 = p.invdxx1 * ((2.0 / 3.0) * (in[13 * Ntot + idx + (1 * s1)] - in[13 * Ntot + idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[13 * Ntot + idx + (2 * s1)] - in[13 * Ntot + idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t42 = -f0_of_xx0*f1_of_xx1*hDD_dD021 - f0_of_xx0*f1_of_xx1__D1*hDD02 + t41;
  const double t43 = -t42;
  const double t44 = hDD01*hDD02*t40 - hDD12*t40*t9;
  const double t45 = 2.0*t14;
  const double t46 = t44*t45;
  const double t47 = t33*t45;
  const double t48 = f0_of_xx0*f1_of_xx1__D1*hDD02 + hDD_dD021*t32 + t41;
  const double t49 = t23*t45;
  const double t2 = 2.0*t1;
  const double hDD_dD220 = p.invdxx0 * ((2.0 / 3.0) * (in[16 * Ntot + idx + (1)] - in[16 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[16 * Ntot + idx + (2)] - in[16 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double t5 = hDD22*t2 + hDD_dD220*t4 + t2;
  const double t6 = -t5;
  const double hDD_dD000 = p.invdxx0 * ((2.0 / 3.0) * (in[11 * Ntot + idx + (1)] - in[11 * Ntot + idx + (-1)]) + (-1.0 / 12.0) * (in[11 * Ntot + idx + (2)] - in[11 * Ntot + idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  gfs[17 * Ntot + idx] = t15*(hDD_dD000*t16 + t25*t39 + t34*t38) + t26*(t1 + t16*t6 + t21*t25) + t36*(f0_of_xx0 + t16*t29 + t25*t35 + t31*t34) + t46*(t16*t43 + t20*t34) + t47*(t25*t42 + t34*t5) + t49*(hDD_dD001*t16 + t25*t28 + t34*t48);
  const double t50 = (Rational_1_2)*t36;
  const double t51 = t24*t44;
  const double t52 = -1.0/f0_of_xx0;
  gfs[18 * Ntot + idx] = f0_of_xx0*(t15*(hDD_dD000*t25 + t38*t51 + t39*t50) + t26*(t17 + t21*t50 + t25*t6) + t36*(t25*t29 + t31*t51 + t35*t50) + t46*(t20*t51 + t25*t43) + t47*(t42*t50 + t5*t51) + t49*(hDD_dD001*t25 + t28*t50 + t48*t51 + t52));
  const double t53 = (Rational_1_2)*t26;
  gfs[19 * Ntot + idx] = t32*(t15*(hDD_dD000*t34 + t38*t53 + t39*t51) + t26*(t21*t51 + t34*t6) + t36*(t29*t34 + t31*t53 + t35*t51) + t46*(t20*t53 + t34*t43 - f1_of_xx1__D1/f1_of_xx1) + t47*(t42*t51 + t5*t53 + t52) + t49*(hDD_dD001*t34 + t28*t51 + t48*t53));
}
#undef Rational_1_2
#undef Rational_2_3

template <bool KEEP, typename K>
static hipError_t rk_det_launch_Spherical_sym2_KO0_fd4(hipStream_t s, K *kin, const double *y_n, double *y_run, double *out,
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
    hipLaunchKernelGGL((bssn_rk_det_Spherical_sym2_KO0_fd4<NP_, IN_, NT_, KEEP>), g, dim3(nt), 0, s, kin, y_n, y_run, out, rfm0, rfm1, p,   \
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
extern "C" hipError_t launch_bssn_rk_det_Spherical_sym2_KO0_fd4(hipStream_t s, const double *kin, const double *y_n, double *y_run,
    double *out, const double *rfm0, const double *rfm1, bhah_kparams p) {
  return rk_det_launch_Spherical_sym2_KO0_fd4<false>(s, kin, y_n, y_run, out, rfm0, rfm1, p, nullptr, nullptr);
}
// The RK pass with the inner boundary condition folded in.
extern "C" hipError_t launch_bssn_rk_det_inner_Spherical_sym2_KO0_fd4(hipStream_t s, const double *kin, const double *y_n,
    double *y_run, double *out, const double *rfm0, const double *rfm1, bhah_kparams p, const int *map,
    const int *pairs) {
  return rk_det_launch_Spherical_sym2_KO0_fd4<false>(s, kin, y_n, y_run, out, rfm0, rfm1, p, reinterpret_cast<const int2 *>(map),
                                    reinterpret_cast<const int2 *>(pairs));
}

// Host-side launchers (one translation unit per variant; no relocatable device code needed).
extern "C" hipError_t launch_bssn_constraints_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, const double *in,
    const double *aux, double *diag, const double *rfm0, const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_constraints_Spherical_sym2_KO0_fd4, g, b, 0, s, in, aux, diag, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_bssn_detgamma_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, double *gfs, const double *rfm0,
    const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_detgamma_Spherical_sym2_KO0_fd4, g, b, 0, s, gfs, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_bssn_initial_lambda_Spherical_sym2_KO0_fd4(dim3 g, dim3 b, hipStream_t s, double *gfs, const double *rfm0,
    const double *rfm1, bhah_kparams p) {
  hipLaunchKernelGGL(bssn_initial_lambda_Spherical_sym2_KO0_fd4, g, b, 0, s, gfs, rfm0, rfm1, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_bssn_ens_rk_det_Spherical_sym2_KO0_fd4(dim3 g, hipStream_t s, const bhah_member *mem,
    const bhah_item *items, int nitems, int k_sel, int out_sel, int substep, int np) {
  if (np == 2)
    hipLaunchKernelGGL(bssn_ens_rk_det_Spherical_sym2_KO0_fd4<2>, g, dim3(256), 0, s, mem, items, nitems, k_sel, out_sel, substep);
  else
    hipLaunchKernelGGL(bssn_ens_rk_det_Spherical_sym2_KO0_fd4<1>, g, dim3(256), 0, s, mem, items, nitems, k_sel, out_sel, substep);
  return hipGetLastError();
}

extern "C" hipError_t launch_bssn_rk_det_taped_Spherical_sym2_KO0_fd4(hipStream_t s, double *k, const double *y_n, double *y_run,
    double *out, const double *rfm0, const double *rfm1, bhah_kparams p, const int *map, const int *pairs) {
  return rk_det_launch_Spherical_sym2_KO0_fd4<true>(s, k, y_n, y_run, out, rfm0, rfm1, p, reinterpret_cast<const int2 *>(map),
                                   reinterpret_cast<const int2 *>(pairs));
}
