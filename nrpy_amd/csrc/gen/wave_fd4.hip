// Generated by nrpy_amd/codegen/hip_gen.py -- do not edit.
#include <hip/hip_runtime.h>
#include <math.h>

#include "../bhah_device_types.h"
// ---- scalar wave kernels, Cartesian, fd_order=4

extern "C" __global__ void __launch_bounds__(256)
wave_rhs_fd4(const double *__restrict__ in, double *__restrict__ rhs, const bhah_kparams p) {
  const int i0 = p.NG + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int i1 = p.NG + (int)(blockIdx.y * blockDim.y + threadIdx.y);
  const int i2 = p.NG + (int)blockIdx.z;
  if (i0 >= p.Nx0 - p.NG || i1 >= p.Nx1 - p.NG) return;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;

  const double vv = in[1 * Ntot + idx];
  rhs[0 * Ntot + idx] = vv;
  const double wavespeed = p.wavespeed;
  const double t0 = (wavespeed*wavespeed);
  const double uu_dDD00 = p.invdxx0 * p.invdxx0 * ((-5.0 / 2.0) * in[idx] + (4.0 / 3.0) * (in[idx + (1)] + in[idx + (-1)]) + (-1.0 / 12.0) * (in[idx + (2)] + in[idx + (-2)]));
  __builtin_amdgcn_sched_barrier(0);
  const double uu_dDD11 = p.invdxx1 * p.invdxx1 * ((-5.0 / 2.0) * in[idx] + (4.0 / 3.0) * (in[idx + (1 * s1)] + in[idx + (-1 * s1)]) + (-1.0 / 12.0) * (in[idx + (2 * s1)] + in[idx + (-2 * s1)]));
  __builtin_amdgcn_sched_barrier(0);
  const double uu_dDD22 = p.invdxx2 * p.invdxx2 * ((-5.0 / 2.0) * in[idx] + (4.0 / 3.0) * (in[idx + (1 * s2)] + in[idx + (-1 * s2)]) + (-1.0 / 12.0) * (in[idx + (2 * s2)] + in[idx + (-2 * s2)]));
  __builtin_amdgcn_sched_barrier(0);
  rhs[1 * Ntot + idx] = t0*uu_dDD00 + t0*uu_dDD11 + t0*uu_dDD22;
}

// rhs_eval and the RK4 substep update in one pass at interior points.  Ghost values enter only
// through the five-point lines of uu, and in a stage past the first they are the quadratic
// extrapolation of the line's own interior points (the boundary condition of every stage), so
// with GHOSTS false each thread forms them from the values it holds and the stage's ghost zones
// need not be filled: one boundary launch a step instead of one a stage.  The arithmetic is
// the boundary kernel's, so the state is the same bit for bit.
namespace wave_fd4 {
// 3 f1 - 3 f2 + f3, as the boundary kernel forms it
__device__ __forceinline__ double extrapolate(double f1, double f2, double f3) {
#pragma clang fp contract(off)
  return +3.0 * f1 - 3.0 * f2 + 1.0 * f3;
}
// The second-derivative sum along one direction; u: the centre value; lo, hi: interior points
// below and above (at least three interior points in every direction, checked by the host).
template <bool GHOSTS>
__device__ __forceinline__ double line(const double *__restrict__ f, long idx, long s, double u, int lo, int hi) {
  double a1 = f[idx + s], a2 = f[idx + 2 * s], b1 = f[idx - s], b2 = f[idx - 2 * s];
  if (!GHOSTS) {
    if (hi == 0) {
      a1 = extrapolate(u, b1, b2);
      a2 = extrapolate(a1, u, b1);
    } else if (hi == 1) {
      a2 = extrapolate(a1, u, b1);
    }
    if (lo == 0) {
      b1 = extrapolate(u, a1, a2);
      b2 = extrapolate(b1, u, a1);
    } else if (lo == 1) {
      b2 = extrapolate(b1, u, a1);
    }
  }
  return (-5.0 / 2.0) * u + (4.0 / 3.0) * (a1 + b1) + (-1.0 / 12.0) * (a2 + b2);
}
}  // namespace wave_fd4
template <bool GHOSTS>
__global__ void __launch_bounds__(256)
wave_rhs_rk_fd4(const double *__restrict__ in, const double *y_n, double *__restrict__ y_run,
                  double *out, const bhah_kparams p) {
  using namespace wave_fd4;
  // Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2):
  // renumber them so XCD k sweeps the k-th contiguous eighth of the tiles and
  // stencil neighbours share an L2.
  unsigned bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  {
    const unsigned gx = gridDim.x, gy = gridDim.y, n = gx * gy * gridDim.z;
    const unsigned h = bx + gx * (by + gy * bz), x = h & 7u, r = n & 7u;
    const unsigned l = x * (n >> 3) + (x < r ? x : r) + (h >> 3);
    bx = l % gx;
    by = (l / gx) % gy;
    bz = l / (gx * gy);
  }
  const int i0 = p.NG + (int)(bx * blockDim.x + threadIdx.x);
  const int i1 = p.NG + (int)(by * blockDim.y + threadIdx.y);
  const int i2 = p.NG + (int)bz;
  if (i0 >= p.Nx0 - p.NG || i1 >= p.Nx1 - p.NG) return;
  const long s1 = p.s1, s2 = p.s2, Ntot = p.Ntot;
  const long idx = i0 + s1 * i1 + s2 * i2;

  constexpr int NGF = 2;
  double kk[NGF], ctr[NGF];
  const double u = in[idx], c2 = p.wavespeed * p.wavespeed;
  kk[0] = in[Ntot + idx];
  const double uu_dDD00 = p.invdxx0 * p.invdxx0 * line<GHOSTS>(in, idx, 1, u, i0 - 2, p.Nx0 - 3 - i0);
  const double uu_dDD11 = p.invdxx1 * p.invdxx1 * line<GHOSTS>(in, idx, s1, u, i1 - 2, p.Nx1 - 3 - i1);
  const double uu_dDD22 = p.invdxx2 * p.invdxx2 * line<GHOSTS>(in, idx, s2, u, i2 - 2, p.Nx2 - 3 - i2);
  kk[1] = c2 * uu_dDD00 + c2 * uu_dDD11 + c2 * uu_dDD22;
  ctr[0] = u;
  ctr[1] = kk[0];

  // RK4 substep update (register_all_MoL_step_forward_in_time.c:4-103), in registers.
  const double dt = p.dt;
  double nxt[NGF];
  if (p.substep == 1) {
#pragma unroll
    for (int g = 0; g < NGF; g++) {
      const double k = kk[g];
      y_run[g * Ntot + idx] = (1.0 / 6.0) * dt * k;
      nxt[g] = (1.0 / 2.0) * dt * k + ctr[g];
    }
  } else if (p.substep == 4) {
#pragma unroll
    for (int g = 0; g < NGF; g++) {
      const double k = kk[g];
      nxt[g] = (1.0 / 6.0) * dt * k + y_n[g * Ntot + idx] + y_run[g * Ntot + idx];
    }
  } else {
    const double a = (p.substep == 2) ? (1.0 / 2.0) : 1.0;
#pragma unroll
    for (int g = 0; g < NGF; g++) {
      const double k = kk[g];
      y_run[g * Ntot + idx] = (1.0 / 3.0) * dt * k + y_run[g * Ntot + idx];
      nxt[g] = a * dt * k + y_n[g * Ntot + idx];
    }
  }

#pragma unroll
  for (int g = 0; g < NGF; g++) out[g * Ntot + idx] = nxt[g];
}


extern "C" hipError_t launch_wave_rhs_fd4(dim3 g, dim3 b, hipStream_t s, const double *in, double *rhs, bhah_kparams p) {
  hipLaunchKernelGGL(wave_rhs_fd4, g, b, 0, s, in, rhs, p);
  return hipGetLastError();
}
extern "C" hipError_t launch_wave_rhs_rk_fd4(dim3 g, dim3 b, hipStream_t s, const double *in, const double *y_n,
    double *y_run, double *out, bhah_kparams p, int ghosts) {
  if (ghosts) hipLaunchKernelGGL(wave_rhs_rk_fd4<true>, g, b, 0, s, in, y_n, y_run, out, p);
  else hipLaunchKernelGGL(wave_rhs_rk_fd4<false>, g, b, 0, s, in, y_n, y_run, out, p);
  return hipGetLastError();
}
