// 3-D stiffness on general hexahedra (mesh databases with irregular
// elements): the weak-form internal force of
// compute_stiffness_interaction.tpp:143-259 extended to (xi, eta, gamma)
// with the full per-point derivative matrix (xix ... gammaz) and jacobian of
// the 3-D database (src/io/mesh/impl/fortran/dim3/mesh.cpp:208-265):
//   du_c/dx_r = sum_s (du_c/dxi_s) dxi_s/dx_r           (gradient.hpp:81-103)
//   sigma = lambda tr(eps) I + 2 mu eps                  (isotropic, kappa + 4/3 mu)
//   F_cs = J sum_r sigma_cr dxi_s/dx_r                   (point/stress.hpp:118-139)
//   r_c = -sum_s w w sum_l F_cs(l) hprime_wgll           (divergence.hpp:86-98)
// One thread owns an (i, j) column of an element and its 5 points along k;
// the xi and eta integrands go through LDS, the gamma ones stay in registers.
// 5 elements per 128-thread workgroup.
//
// ATOMIC adds the element forces to the acceleration with float atomics.  The
// default scatter stores them (forces_3d_general_kernel, all elements in one
// launch, with the source and Stacey terms beside them) and sums every point's
// contributions in one pass that also applies the mass, the corrector and the
// next predictor (update_3d_general_kernel): source terms, then the elements in
// color order, then the Stacey terms, the order in which one launch per color
// added them, so the results keep their bits.  On 10,296 elements (half of them
// irregular) the eight color launches took 110 us a step, each too small to
// fill the device; now 21 us for the forces and 21 us for the update.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace sfx {

namespace {

constexpr int EG = 5;

inline unsigned groups(long long n, int per) { return static_cast<unsigned>((n + per - 1) / per); }

// The element forces of workgroup `block`.  STORE: into re (element, component,
// point); else added to f.a with atomics.  geo_of: row of geo of each element,
// or -1 for a regular one (derivatives 0 but xix = etay = gammaz = xr, jacobian
// jr).  kmu: one (kappa, mu) pair per element, or null.
template <bool STORE>
__device__ __forceinline__ void general_forces(int block, int nspec, const int *__restrict__ gather,
                                               const int *__restrict__ geo_of, const float *__restrict__ geo,
                                               float xr, float jr, const float *__restrict__ kappa_,
                                               const float *__restrict__ mu_, const float *__restrict__ kmu,
                                               const GllConst &q, const Fields &f, float *__restrict__ re) {
  __shared__ float su[EG][3][125];
  __shared__ float sF0[EG][3][125];  // F(c, xi)
  __shared__ float sF1[EG][3][125];  // F(c, eta)

  const int t = threadIdx.x;
  const int el = t / 25;
  const int col = t - el * 25;
  const int j = col / 5, i = col - (col / 5) * 5;
  const int e = block * EG + el;
  const bool active = (el < EG) && (e < nspec);
  const size_t base = static_cast<size_t>(e) * 125 + col;
  const int np = f.nglob_pad;

  int g[5];
  float u[5][3];
  const float *ge = nullptr;
  if (active) {
#pragma unroll
    for (int k = 0; k < 5; k++) g[k] = gather[base + k * 25];
    const int gi = geo_of[e];
    if (gi >= 0) ge = geo + static_cast<size_t>(gi) * 1250 + col;
#pragma unroll
    for (int k = 0; k < 5; k++)
#pragma unroll
      for (int c = 0; c < 3; c++) u[k][c] = f.u[c * np + g[k]];
#pragma unroll
    for (int k = 0; k < 5; k++)
#pragma unroll
      for (int c = 0; c < 3; c++) su[el][c][k * 25 + col] = u[k][c];
  }
  __syncthreads();

  float F2[5][3];  // F(c, gamma), in registers
  if (active) {
#pragma unroll
    for (int k = 0; k < 5; k++) {
      float d9[9], J;
      if (ge) {
#pragma unroll
        for (int d = 0; d < 9; d++) d9[d] = ge[d * 125 + k * 25];
        J = ge[9 * 125 + k * 25];
      } else {
#pragma unroll
        for (int d = 0; d < 9; d++) d9[d] = d % 4 ? 0.0f : xr;
        J = jr;
      }
      float dr[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};  // dr[c][s] = du_c / dxi_s
#pragma unroll
      for (int l = 0; l < 5; l++) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          dr[c][0] += q.hp[i][l] * su[el][c][k * 25 + j * 5 + l];
          dr[c][1] += q.hp[j][l] * su[el][c][k * 25 + l * 5 + i];
          dr[c][2] += q.hp[k][l] * u[l][c];
        }
      }
      float du[3][3];  // du[c][r] = du_c / dx_r
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) du[c][r] = dr[c][0] * d9[0 + r] + dr[c][1] * d9[3 + r] + dr[c][2] * d9[6 + r];
      const float kappa = kmu ? kmu[2 * static_cast<size_t>(e)] : kappa_[base + k * 25];
      const float mu = kmu ? kmu[2 * static_cast<size_t>(e) + 1] : mu_[base + k * 25];
      const float lp2m = kappa + (4.0f / 3.0f) * mu;
      const float lambda = lp2m - 2.0f * mu;
      const float tr = du[0][0] + du[1][1] + du[2][2];
      float s[3][3];
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int r = 0; r < 3; r++) s[c][r] = mu * (du[c][r] + du[r][c]) + (c == r ? lambda * tr : 0.0f);
      const int p = k * 25 + col;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        sF0[el][c][p] = J * (s[c][0] * d9[0] + s[c][1] * d9[1] + s[c][2] * d9[2]);
        sF1[el][c][p] = J * (s[c][0] * d9[3] + s[c][1] * d9[4] + s[c][2] * d9[5]);
        F2[k][c] = J * (s[c][0] * d9[6] + s[c][1] * d9[7] + s[c][2] * d9[8]);
      }
    }
  }
  __syncthreads();
  if (!active) return;
  const float wi = q.w[i], wj = q.w[j];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    float r0[3] = {0, 0, 0}, r1[3] = {0, 0, 0}, r2[3] = {0, 0, 0};
#pragma unroll
    for (int l = 0; l < 5; l++) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        r0[c] += sF0[el][c][k * 25 + j * 5 + l] * q.hpw[i][l];
        r1[c] += sF1[el][c][k * 25 + l * 5 + i] * q.hpw[j][l];
        r2[c] += F2[l][c] * q.hpw[k][l];
      }
    }
    const float wjk = wj * q.w[k], wik = wi * q.w[k], wij = wi * wj;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float r = -(wjk * r0[c] + wik * r1[c] + wij * r2[c]);
      if constexpr (STORE)
        re[static_cast<size_t>(e) * 375 + c * 125 + k * 25 + col] = r;
      else
        unsafeAtomicAdd(&f.a[c * np + g[k]], r);
    }
  }
}

__global__ __launch_bounds__(128) void stiffness_3d_general_kernel(int nspec, const int *__restrict__ gather,
                                                                   General3D m, GllConst q, Fields f) {
  general_forces<false>(blockIdx.x, nspec, gather, m.geo_of, m.geo, m.xr, m.jr, m.kappa, m.mu, m.kmu, q, f, nullptr);
}

// Element forces, then one workgroup per source (its 125 terms), then the
// Stacey entries 125 to a workgroup, each in its block of 375 floats of re.
__global__ __launch_bounds__(128) void forces_3d_general_kernel(int nspec, int nblocks, const int *__restrict__ gather,
                                                                General3D m, GllConst q, Fields f, int nsrc, int istep,
                                                                const float *__restrict__ array,
                                                                const float *__restrict__ stf, int nbnd,
                                                                const int *__restrict__ bgather,
                                                                const float *__restrict__ normal,
                                                                const float *__restrict__ weight,
                                                                const float *__restrict__ rho_vp,
                                                                const float *__restrict__ rho_vs,
                                                                float *__restrict__ re) {
  const int b = blockIdx.x, t = threadIdx.x;
  if (b < nblocks) {
    general_forces<true>(b, nspec, gather, m.geo_of, m.geo, m.xr, m.jr, m.kappa, m.mu, m.kmu, q, f, re);
    return;
  }
  if (t >= 125) return;
  if (b < nblocks + nsrc) {
    const int s = b - nblocks;
    const float sv = stf[static_cast<size_t>(istep) * nsrc + s];
#pragma unroll
    for (int c = 0; c < 3; c++)
      re[(static_cast<size_t>(nspec) + s) * 375 + c * 125 + t] = sv * array[(static_cast<size_t>(s) * 3 + c) * 125 + t];
    return;
  }
  // stacey.tpp:36-72, the operations of stacey_kernel<3>
  const int blk = b - nblocks - nsrc;
  const int k = blk * 125 + t;
  if (k >= nbnd) return;
  const int g = bgather[k], np = f.nglob_pad;
  float n[3], v[3];
  float vn = 0.0f, nn = 0.0f;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    n[d] = normal[k * 3 + d];
    v[d] = f.v[d * np + g];
    vn += v[d] * n[d];
    nn += n[d] * n[d];
  }
  const float j1 = sqrtf(nn);
  const float w = weight[k], rvp = rho_vp[k], rvs = rho_vs[k];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const float fac = ((vn * n[d] / (j1 * j1)) * (rvp - rvs)) + v[d] * rvs;
    re[(static_cast<size_t>(nspec) + nsrc + blk) * 375 + d * 125 + t] = -1.0f * fac * j1 * w;
  }
}

// Adds to s a point's contributions [k0, k1) of ent (offsets of their first
// component), in order; the first four entries' loads are issued together
// (indices clamped to the last one).
__device__ __forceinline__ void point_force(const uint32_t *__restrict__ ent, const float *__restrict__ re, int k0, int k1,
                                            float s[3]) {
  if (k1 <= k0) return;
  uint32_t o[4];
  float r[4][3];
#pragma unroll
  for (int j = 0; j < 4; j++) o[j] = ent[k0 + j < k1 ? k0 + j : k1 - 1];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int c = 0; c < 3; c++) r[j][c] = re[static_cast<size_t>(o[j]) + c * 125];
#pragma unroll
  for (int j = 0; j < 4; j++)
    if (k0 + j < k1)
#pragma unroll
      for (int c = 0; c < 3; c++) s[c] += r[j][c];
  for (int k = k0 + 4; k < k1; k++)
#pragma unroll
    for (int c = 0; c < 3; c++) s[c] += re[static_cast<size_t>(ent[k]) + c * 125];
}

// One thread per point: a = M^-1 f; divide: a is stored; else corrector and
// the next predictor on u, v.  add: the sum starts from the stored a.
__global__ __launch_bounds__(256) void update_3d_general_kernel(int nglob, const int *__restrict__ off,
                                                                const uint32_t *__restrict__ ent,
                                                                const float *__restrict__ re, Fields f,
                                                                NewmarkConst nc, int divide, int add) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= nglob) return;
  float m[3], u[3], v[3], s[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const size_t o = c * static_cast<size_t>(f.nglob_pad) + g;
    m[c] = f.minv[o];
    u[c] = f.u[o];
    v[c] = f.v[o];
    s[c] = add ? f.a[o] : 0.0f;
  }
  point_force(ent, re, off[g], off[g + 1], s);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const size_t o = c * static_cast<size_t>(f.nglob_pad) + g;
    const float ac = s[c] * m[c];
    if (divide) {
      f.a[o] = ac;
      continue;
    }
    const float v1 = v[c] + nc.dto2 * ac;
    f.u[o] = u[c] + (nc.dt * v1 + nc.dt2o2 * ac);
    f.v[o] = v1 + nc.dto2 * ac;
    if (add) f.a[o] = 0.0f;
  }
}

// One workgroup per receiver: the samples seismogram_kernel<3> takes, the
// acceleration summed from its contributions.
__global__ __launch_bounds__(128) void seismogram_3d_general_kernel(int nrec, int ntypes,
                                                                    const int *__restrict__ types, int isig,
                                                                    const int *__restrict__ ispec,
                                                                    const int *__restrict__ gather,
                                                                    const float *__restrict__ h, Fields f, float dto2,
                                                                    float *__restrict__ seismo,
                                                                    const int *__restrict__ off,
                                                                    const uint32_t *__restrict__ ent,
                                                                    const float *__restrict__ re, int need_a,
                                                                    int add) {
  __shared__ float red[4][3][2];
  const int r = blockIdx.x, p = threadIdx.x;
  const int g = p < 125 ? gather[static_cast<size_t>(ispec[r]) * 125 + p] : 0;
  const float hw = p < 125 ? h[static_cast<size_t>(r) * 125 + p] : 0.0f;
  float u[3] = {0, 0, 0}, v[3] = {0, 0, 0}, a[3] = {0, 0, 0};
  if (p < 125) {
    float m[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const size_t o = c * static_cast<size_t>(f.nglob_pad) + g;
      u[c] = f.u[o];
      v[c] = f.v[o];
      m[c] = f.minv[o];
      if (add) a[c] = f.a[o];
    }
    if (need_a) {
      point_force(ent, re, off[g], off[g + 1], a);
#pragma unroll
      for (int c = 0; c < 3; c++) a[c] = a[c] * m[c];
    }
  }
  for (int it = 0; it < ntypes; it++) {
    const int type = types[it];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float x = type == 0 ? u[c] : type == 1 ? v[c] + dto2 * a[c] : a[c];
      float s = hw * x;
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) s += __shfl_down(s, d, 64);
      if ((p & 63) == 0) red[it][c][p >> 6] = s;
    }
  }
  __syncthreads();
  if (p < 3)
    for (int it = 0; it < ntypes; it++)
      seismo[((static_cast<size_t>(isig) * ntypes + it) * nrec + r) * 3 + p] = red[it][p][0] + red[it][p][1];
}

}  // namespace

void launch_stiffness_3d_general(hipStream_t s, int nspec, const int *gather, const General3D &m, const GllConst &q,
                                 Fields f) {
  if (nspec > 0)
    hipLaunchKernelGGL(stiffness_3d_general_kernel, dim3(groups(nspec, EG)), dim3(128), 0, s, nspec, gather, m, q, f);
}

void launch_forces_3d_general(hipStream_t s, int nspec, const int *gather, const General3D &m, const GllConst &q,
                              Fields f, int nsrc, int istep, const float *array, const float *stf, int nbnd,
                              const int *bgather, const float *normal, const float *weight, const float *rho_vp,
                              const float *rho_vs, float *re) {
  const unsigned nb = groups(nspec, EG);
  hipLaunchKernelGGL(forces_3d_general_kernel, dim3(nb + nsrc + groups(nbnd, 125)), dim3(128), 0, s, nspec,
                     static_cast<int>(nb), gather, m, q, f, nsrc, istep, array, stf, nbnd, bgather, normal, weight,
                     rho_vp, rho_vs, re);
}

void launch_update_3d_general(hipStream_t s, int nglob, const int *off, const uint32_t *ent, const float *re, Fields f,
                              NewmarkConst nc, int divide, int add) {
  if (nglob > 0)
    hipLaunchKernelGGL(update_3d_general_kernel, dim3(groups(nglob, 256)), dim3(256), 0, s, nglob, off, ent, re, f, nc,
                       divide, add);
}

void launch_seismograms_3d_general(hipStream_t s, int nrec, int ntypes, const int *types, int isig, const int *ispec,
                                   const int *gather, const float *h, Fields f, float dto2, float *seismo,
                                   const int *off, const uint32_t *ent, const float *re, int need_a, int add) {
  if (nrec > 0 && ntypes > 0)
    hipLaunchKernelGGL(seismogram_3d_general_kernel, dim3(nrec), dim3(128), 0, s, nrec, ntypes, types, isig, ispec,
                       gather, h, f, dto2, seismo, off, ent, re, need_a, add);
}

}  // namespace sfx
