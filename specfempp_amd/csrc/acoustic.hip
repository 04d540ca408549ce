// 2-D acoustic medium and elastic-acoustic coupling kernels (gfx950, wave64).
//
// Reference kernels these replace:
//   acoustic stiffness   compute_stiffness_interaction.tpp:143-259 with the
//                        acoustic stress rho^-1 grad chi
//                        (include/medium/dim2/acoustic/isotropic/stress.hpp),
//                        the acoustic Stacey term (stacey.tpp:172-213) and the
//                        free surface (boundary_conditions/dirichlet: the
//                        point's contribution is set to zero)
//   acoustic sources     compute_source_interaction.tpp:80-95 with
//                        include/medium/dim2/acoustic/isotropic/source.hpp
//                        (stf * lagrange / kappa)
//   coupling             include/coupled_interface/coupled_interface.tpp and
//                        interface_kernels.hpp:18-54 (acoustic side: factor
//                        n . u; elastic side: factor n chi_dot_dot)
//   seismograms          compute_seismogram.tpp:103-135 with
//                        include/medium/dim2/acoustic/isotropic/wavefield.hpp
//                        (grad chi / rho; pressure -chi_dot_dot)
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace sfx {

namespace {

constexpr int EA = 5;  // acoustic elements per 128-thread workgroup

inline unsigned blocks_of(long long n, int per) { return static_cast<unsigned>((n + per - 1) / per); }

template <bool ATOMIC> __device__ __forceinline__ void add_to(float *p, float v) {
  if constexpr (ATOMIC)
    unsafeAtomicAdd(p, v);
  else
    *p += v;
}

// One thread per GLL point of EA elements.  chi and the integrand F are
// staged in LDS; the derivative matrices' rows are held in registers.
template <bool ATOMIC>
__global__ __launch_bounds__(128) void acoustic_stiffness_2d_kernel(
    int first, int count, const int *__restrict__ gather, const float *__restrict__ xix_,
    const float *__restrict__ xiz_, const float *__restrict__ gammax_, const float *__restrict__ gammaz_,
    const float *__restrict__ jac_, const float *__restrict__ rho_inv_, const float *__restrict__ stacey_,
    const int *__restrict__ dirichlet_, GllConst q, Fields f) {
  __shared__ float sc[EA][25];
  __shared__ float sF[EA][2][25];
  const int t = threadIdx.x;
  const int el = t / 25;
  const int p = t - el * 25;
  const int iz = p / 5, ix = p - (p / 5) * 5;
  const int el_idx = blockIdx.x * EA + el;
  const bool active = (el < EA) && (el_idx < count);
  const size_t idx = static_cast<size_t>(first + el_idx) * 25 + p;
  int g = 0;
  if (active) {
    g = gather[idx];
    sc[el][p] = f.u[g];
  }
  __syncthreads();
  if (active) {
    float dxi = 0.0f, dga = 0.0f;
#pragma unroll
    for (int l = 0; l < 5; l++) {
      dxi += q.hp[ix][l] * sc[el][iz * 5 + l];
      dga += q.hp[iz][l] * sc[el][l * 5 + ix];
    }
    const float xix = xix_[idx], xiz = xiz_[idx], gammax = gammax_[idx], gammaz = gammaz_[idx], J = jac_[idx];
    const float ri = rho_inv_[idx];
    const float du0 = fmaf(xix, dxi, gammax * dga);
    const float du1 = fmaf(xiz, dxi, gammaz * dga);
    const float T0 = ri * du0, T1 = ri * du1;
    // core/specfem/point/stress.hpp:118-139 for one component
    sF[el][0][p] = J * fmaf(T0, xix, T1 * xiz);
    sF[el][1][p] = J * fmaf(T0, gammax, T1 * gammaz);
  }
  __syncthreads();
  if (!active) return;
  // include/algorithms/divergence.hpp:86-98
  float t1 = 0.0f, t2 = 0.0f;
#pragma unroll
  for (int l = 0; l < 5; l++) {
    t1 += sF[el][0][iz * 5 + l] * q.hpw[ix][l];
    t2 += sF[el][1][l * 5 + ix] * q.hpw[iz][l];
  }
  float r = -fmaf(q.w[iz], t1, q.w[ix] * t2);
  const float c = stacey_[idx];
  if (c != 0.0f) r = fmaf(-c, f.v[g], r);
  if (dirichlet_[idx]) r = 0.0f;
  add_to<ATOMIC>(&f.a[g], r);
}

// a[self] += factor (nx u_x[other] + nz u_z[other]) into the acoustic field
// from the elastic displacement (to_elastic = 0), or
// a_x[self] += factor nx chi_dot_dot[other], a_z[self] += factor nz
// chi_dot_dot[other] into the elastic field (to_elastic = 1).
__global__ __launch_bounds__(256) void coupling_2d_kernel(int n, const int *__restrict__ self,
                                                          const int *__restrict__ other,
                                                          const float *__restrict__ coef, Fields dst, Fields src,
                                                          int to_elastic) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int s = self[i], o = other[i];
  const float factor = coef[3 * i], nx = coef[3 * i + 1], nz = coef[3 * i + 2];
  if (to_elastic) {
    const float chi_dd = src.a[o];
    unsafeAtomicAdd(&dst.a[s], factor * nx * chi_dd);
    unsafeAtomicAdd(&dst.a[dst.nglob_pad + s], factor * nz * chi_dd);
  } else {
    unsafeAtomicAdd(&dst.a[s], factor * fmaf(nx, src.u[o], nz * src.u[src.nglob_pad + o]));
  }
}

// One workgroup per acoustic source (in application order), one thread per
// element point.
__global__ __launch_bounds__(64) void acoustic_sources_kernel(int norder, int nsrc, int istep,
                                                              const int *__restrict__ order,
                                                              const int *__restrict__ ispec,
                                                              const int *__restrict__ gather,
                                                              const float *__restrict__ array,
                                                              const float *__restrict__ stf,
                                                              const float *__restrict__ kappa, Fields f) {
  const int p = threadIdx.x, k = blockIdx.x;
  if (p >= 25 || k >= norder) return;
  const int s = order[k];
  const float sv = stf[static_cast<size_t>(istep) * nsrc + s];
  const size_t idx = static_cast<size_t>(ispec[s]) * 25 + p;
  unsafeAtomicAdd(&f.a[gather[idx]], sv * array[static_cast<size_t>(s) * 50 + p] / kappa[idx]);
}

// Receiver r by one workgroup of 64 threads: the element's potential (or its time
// derivatives) in LDS, the gradient times 1/rho at every point, Lagrange
// weights, wave reduction.  Pressure is -chi_dot_dot.
__device__ __forceinline__ void acoustic_seismogram(int r, int nrec, int ntypes, const int *__restrict__ types, int isig,
                                                    const int *__restrict__ ispec, const int *__restrict__ gather,
                                                    const float *__restrict__ h, const float *__restrict__ xix_,
                                                    const float *__restrict__ xiz_, const float *__restrict__ gammax_,
                                                    const float *__restrict__ gammaz_,
                                                    const float *__restrict__ rho_inv_, const GllConst &q, Fields f,
                                                    float *__restrict__ seismo, float *sc) {
  const int p = threadIdx.x;
  const int iz = p / 5, ix = p - (p / 5) * 5;
  const size_t idx = static_cast<size_t>(ispec[r]) * 25 + (p < 25 ? p : 0);
  const int g = p < 25 ? gather[idx] : 0;
  const float hw = p < 25 ? h[static_cast<size_t>(r) * 25 + p] : 0.0f;
  for (int it = 0; it < ntypes; it++) {
    const int type = types[it];
    const float *fld = type == 0 ? f.u : (type == 1 ? f.v : f.a);
    __syncthreads();
    if (p < 25) sc[p] = fld[g];
    __syncthreads();
    float v0 = 0.0f, v1 = 0.0f;
    if (p < 25) {
      if (type == 3) {
        v0 = -sc[p];
      } else {
        float dxi = 0.0f, dga = 0.0f;
#pragma unroll
        for (int l = 0; l < 5; l++) {
          dxi += q.hp[ix][l] * sc[iz * 5 + l];
          dga += q.hp[iz][l] * sc[l * 5 + ix];
        }
        const float ri = rho_inv_[idx];
        v0 = ri * fmaf(xix_[idx], dxi, gammax_[idx] * dga);
        v1 = ri * fmaf(xiz_[idx], dxi, gammaz_[idx] * dga);
      }
      v0 *= hw;
      v1 *= hw;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      v0 += __shfl_down(v0, off, 64);
      v1 += __shfl_down(v1, off, 64);
    }
    if (p == 0) {
      float *o = seismo + ((static_cast<size_t>(isig) * ntypes + it) * nrec + r) * 2;
      o[0] = v0;
      o[1] = type == 3 ? 0.0f : v1;
    }
  }
}

__global__ __launch_bounds__(64) void acoustic_seismogram_kernel(
    const int *__restrict__ list, int nrec, int ntypes, const int *__restrict__ types, int isig,
    const int *__restrict__ ispec, const int *__restrict__ gather, const float *__restrict__ h,
    const float *__restrict__ xix, const float *__restrict__ xiz, const float *__restrict__ gammax,
    const float *__restrict__ gammaz, const float *__restrict__ rho_inv, GllConst q, Fields f,
    float *__restrict__ seismo) {
  __shared__ float sc[25];
  acoustic_seismogram(list[blockIdx.x], nrec, ntypes, types, isig, ispec, gather, h, xix, xiz, gammax, gammaz, rho_inv,
                      q, f, seismo, sc);
}

// ---------------------------------------------------------------------------
// Coupled steps without color launches.
//
// A step took about 20 launches (a launch per color and medium, sources,
// interface, Stacey, seismograms, updates), and its time was theirs: at 120x80
// elements the kernels ran 2 to 4 us each, as long as it takes to submit one.
// Here all forces are stored in one launch (both media read only the
// predicted fields), the acoustic points are summed in a second, the elastic
// ones, which need chi_dot_dot at the interface, in a third, with one more on
// sampled steps.  120x80 elements, 40 receivers on every step: 71 -> 17.3 us a
// step (forces 4.7, acoustic points 3.5, samples 3.9, update 4.9 us, each a
// launch's latency and two dependent loads; the floor by bytes is below 4 us).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(128) void coupled_forces_kernel(CoupledStep m, GllConst q, int istep, Fields el,
                                                             Fields ac, int b_ac, int b_src, int b_src_ac, int b_bnd,
                                                             int b_cpl) {
#pragma clang fp contract(off)
  // multiply-adds are written out as the separate launches' kernels contract
  // them, so that steps taken through the seams give the same bits
  __shared__ float su[EA][2][25];
  __shared__ float sF[EA][4][25];
  const int t = threadIdx.x, b = blockIdx.x;
  const int ei = t / 25, p = t - ei * 25;
  const int iz = p / 5, ix = p - (p / 5) * 5;
  if (b < b_ac) {  // elastic elements: the arithmetic of stiffness_2d_kernel
    const int np = el.nglob_pad;
    const bool active = ei < EA && b * EA + ei < m.nel;
    const int e = b * EA + ei < m.nel ? b * EA + ei : m.nel - 1;
    const size_t idx = static_cast<size_t>(e) * 25 + p;
    const int g = m.gather[idx];
    const float u0 = el.u[g], u1 = el.u[np + g];
    const float xix = m.pg.xix[idx], xiz = m.pg.xiz[idx], gammax = m.pg.gammax[idx], gammaz = m.pg.gammaz[idx];
    const float J = m.jac[idx], kappa = m.pg.kappa[idx], mu = m.pg.mu[idx];
    float hpx[5], hpz[5], hwx[5], hwz[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      hpx[l] = q.hp[ix][l];
      hpz[l] = q.hp[iz][l];
      hwx[l] = q.hpw[ix][l];
      hwz[l] = q.hpw[iz][l];
    }
    const float wx = q.w[ix], wz = q.w[iz];
    if (active) {
      su[ei][0][p] = u0;
      su[ei][1][p] = u1;
    }
    __syncthreads();
    if (active) {
      float dxi[2] = {0.0f, 0.0f}, dga[2] = {0.0f, 0.0f};
#pragma unroll
      for (int l = 0; l < 5; l++) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
          dxi[c] = fmaf(hpx[l], su[ei][c][iz * 5 + l], dxi[c]);
          dga[c] = fmaf(hpz[l], su[ei][c][l * 5 + ix], dga[c]);
        }
      }
      float du[2][2];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        du[c][0] = fmaf(xix, dxi[c], gammax * dga[c]);
        du[c][1] = fmaf(xiz, dxi[c], gammaz * dga[c]);
      }
      const float lp2m = fmaf(4.0f / 3.0f, mu, kappa);
      const float lambda = lp2m - 2.0f * mu;
      const float sxx = fmaf(lp2m, du[0][0], lambda * du[1][1]);
      const float szz = fmaf(lp2m, du[1][1], lambda * du[0][0]);
      const float sxz = mu * (du[0][1] + du[1][0]);
      sF[ei][0][p] = J * fmaf(sxx, xix, sxz * xiz);
      sF[ei][1][p] = J * fmaf(sxx, gammax, sxz * gammaz);
      sF[ei][2][p] = J * fmaf(sxz, xix, szz * xiz);
      sF[ei][3][p] = J * fmaf(sxz, gammax, szz * gammaz);
    }
    __syncthreads();
    if (!active) return;
    float t1[2] = {0.0f, 0.0f}, t2[2] = {0.0f, 0.0f};
#pragma unroll
    for (int l = 0; l < 5; l++) {
#pragma unroll
      for (int c = 0; c < 2; c++) {
        t1[c] = fmaf(sF[ei][2 * c][iz * 5 + l], hwx[l], t1[c]);
        t2[c] = fmaf(sF[ei][2 * c + 1][l * 5 + ix], hwz[l], t2[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < 2; c++) m.re[static_cast<size_t>(e) * 50 + c * 25 + p] = -fmaf(wz, t1[c], wx * t2[c]);
    return;
  }
  if (b < b_src) {  // acoustic elements: the arithmetic of acoustic_stiffness_2d_kernel
    const int i = (b - b_ac) * EA + ei;
    const bool active = ei < EA && i < m.nac;
    const int e = i < m.nac ? i : m.nac - 1;
    const size_t idx = static_cast<size_t>(m.nel + e) * 25 + p;
    const int g = m.gather[idx];
    const float chi = ac.u[g], v = ac.v[g], c = m.ac_stacey[idx];
    const float xix = m.pg.xix[idx], xiz = m.pg.xiz[idx], gammax = m.pg.gammax[idx], gammaz = m.pg.gammaz[idx];
    const float J = m.jac[idx], ri = m.rho_inv[idx];
    const int free_surface = m.ac_dirichlet[idx];
    if (active) su[ei][0][p] = chi;
    __syncthreads();
    if (active) {
      float dxi = 0.0f, dga = 0.0f;
#pragma unroll
      for (int l = 0; l < 5; l++) {
        dxi = fmaf(q.hp[ix][l], su[ei][0][iz * 5 + l], dxi);
        dga = fmaf(q.hp[iz][l], su[ei][0][l * 5 + ix], dga);
      }
      const float du0 = fmaf(xix, dxi, gammax * dga);
      const float du1 = fmaf(xiz, dxi, gammaz * dga);
      const float T0 = ri * du0, T1 = ri * du1;
      sF[ei][0][p] = J * fmaf(T0, xix, T1 * xiz);
      sF[ei][1][p] = J * fmaf(T0, gammax, T1 * gammaz);
    }
    __syncthreads();
    if (!active) return;
    float t1 = 0.0f, t2 = 0.0f;
#pragma unroll
    for (int l = 0; l < 5; l++) {
      t1 = fmaf(sF[ei][0][iz * 5 + l], q.hpw[ix][l], t1);
      t2 = fmaf(sF[ei][1][l * 5 + ix], q.hpw[iz][l], t2);
    }
    float r = -fmaf(q.w[iz], t1, q.w[ix] * t2);
    if (c != 0.0f) r = fmaf(-c, v, r);
    if (free_surface) r = 0.0f;
    m.re[m.at_ac + static_cast<size_t>(e) * 25 + p] = r;
    return;
  }
  if (b < b_bnd) {  // a source
    if (t >= 25) return;
    const bool elastic = b < b_src_ac;
    const int k = b - (elastic ? b_src : b_src_ac);
    const int s = elastic ? m.order_el[k] : m.order_ac[k];
    const float sv = m.stf[static_cast<size_t>(istep) * m.nsrc + s];
    const float *array = m.src_array + static_cast<size_t>(s) * 50 + t;
    if (elastic) {
#pragma unroll
      for (int c = 0; c < 2; c++) m.re[m.at_src_el + static_cast<size_t>(k) * 50 + c * 25 + t] = sv * array[c * 25];
    } else {
      m.re[m.at_src_ac + static_cast<size_t>(k) * 25 + t] =
          sv * array[0] / m.pg.kappa[static_cast<size_t>(m.src_ispec[s]) * 25 + t];
    }
    return;
  }
  if (b < b_cpl) {  // Stacey entries: the arithmetic of stacey_kernel<2>
    const int k = (b - b_bnd) * 128 + t;
    if (k >= m.nbnd) return;
    const int g = m.bnd_gather[k];
    const int np = el.nglob_pad;
    float n[2], v[2];
#pragma unroll
    for (int d = 0; d < 2; d++) {
      n[d] = m.bnd_normal[k * 2 + d];
      v[d] = el.v[d * np + g];
    }
    const float vn = fmaf(v[1], n[1], v[0] * n[0]), nn = fmaf(n[0], n[0], n[1] * n[1]);
    const float j1 = sqrtf(nn);
    const float w = m.bnd_weight[k], rvp = m.bnd_rvp[k], rvs = m.bnd_rvs[k];
#pragma unroll
    for (int d = 0; d < 2; d++) {
      const float fac = fmaf(rvs, v[d], (vn * n[d] / (j1 * j1)) * (rvp - rvs));
      m.re[m.at_bnd + static_cast<size_t>(k / 25) * 50 + d * 25 + k % 25] = -1.0f * fac * j1 * w;
    }
    return;
  }
  const int i = (b - b_cpl) * 128 + t;  // interface entries of the acoustic side
  if (i >= m.ncpl_ac) return;
  const int o = m.ac_other[i];
  const float factor = m.ac_coef[3 * i], nx = m.ac_coef[3 * i + 1], nz = m.ac_coef[3 * i + 2];
  m.re[m.at_cpl + static_cast<size_t>(i)] = factor * fmaf(nx, el.u[o], nz * el.u[el.nglob_pad + o]);
}

// s (the point's stored acceleration) + the contributions of its record e, in
// order.  The loads of the four inline ones are issued together, absent ones
// re-reading the first value of re.
template <int NC>
__device__ __forceinline__ void add_contributions(const CoupledStep &m, uint4 e, float s[NC]) {
#pragma clang fp contract(off)
  auto term = [&](uint32_t o) {  // elastic side of interface entry o
    const int k = static_cast<int>(o & CONTRIB_INDEX);
    const float factor = m.el_coef[3 * k], chi_dd = m.dd[m.el_other[k]];
#pragma unroll
    for (int c = 0; c < NC; c++) s[c] += factor * m.el_coef[3 * k + 1 + c] * chi_dd;
  };
  if (e.x >= CONTRIB_LIST) {
    const int row = static_cast<int>(e.x & CONTRIB_INDEX);
    for (int k = m.list_off[row]; k < m.list_off[row + 1]; k++) {
      const uint32_t o = m.list[k];
      if (NC == 2 && o >= CONTRIB_TERM) {
        term(o);
        continue;
      }
#pragma unroll
      for (int c = 0; c < NC; c++) s[c] += m.re[static_cast<size_t>(o) + c * 25];
    }
    return;
  }
  const uint32_t o[4] = {e.x, e.y, e.z, e.w};
  float r[4][NC];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int c = 0; c < NC; c++) r[j][c] = m.re[o[j] < CONTRIB_NONE ? static_cast<size_t>(o[j]) + c * 25 : 0];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (o[j] < CONTRIB_NONE) {
#pragma unroll
      for (int c = 0; c < NC; c++) s[c] += r[j][c];
    } else if (NC == 2 && o[j] >= CONTRIB_TERM) {
      term(o[j]);
    }
  }
}

// One thread per acoustic point: mass division and corrector.  chi_dot_dot goes
// to dd, the stored acceleration is cleared as the predictor leaves it.
__global__ __launch_bounds__(256) void coupled_acoustic_kernel(CoupledStep m, Fields f, NewmarkConst nc) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= m.nglob_ac) return;
  const float minv = f.minv[g], v = f.v[g];
  float s[1] = {f.a[g]};
  add_contributions<1>(m, m.ent_ac[g], s);
  const float a = s[0] * minv;
  m.dd[g] = a;
  f.a[g] = 0.0f;
  f.v[g] = fmaf(nc.dto2, a, v);
}

// Elastic points: mass division, corrector and next predictor; acoustic points:
// next predictor.
__global__ __launch_bounds__(256) void coupled_update_kernel(CoupledStep m, Fields el, Fields ac, NewmarkConst nc,
                                                             int b_ac) {
#pragma clang fp contract(off)
  if (static_cast<int>(blockIdx.x) >= b_ac) {
    const int g = (blockIdx.x - b_ac) * 256 + threadIdx.x;
    if (g >= m.nglob_ac) return;
    const float a = m.dd[g], v = ac.v[g];
    ac.u[g] = ac.u[g] + fmaf(nc.dt2o2, a, nc.dt * v);
    ac.v[g] = fmaf(nc.dto2, a, v);
    return;
  }
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= m.nglob_el) return;
  const int np = el.nglob_pad;
  float minv[2], u[2], v[2], s[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const size_t o = c * static_cast<size_t>(np) + g;
    minv[c] = el.minv[o];
    u[c] = el.u[o];
    v[c] = el.v[o];
    s[c] = el.a[o];
  }
  add_contributions<2>(m, m.ent_el[g], s);
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const size_t o = c * static_cast<size_t>(np) + g;
    const float a = s[c] * minv[c];
    const float v1 = fmaf(nc.dto2, a, v[c]);
    el.u[o] = u[c] + fmaf(nc.dt2o2, a, nc.dt * v1);
    el.v[o] = fmaf(nc.dto2, a, v1);
    el.a[o] = 0.0f;
  }
}

// One workgroup per receiver: the state after the corrector.  Elastic
// accelerations are summed from their contributions; acoustic receivers read dd.
__global__ __launch_bounds__(64) void coupled_seismogram_kernel(CoupledStep m, GllConst q, int isig, Fields el,
                                                                Fields ac, float dto2) {
  __shared__ float su[2][25];
  if (static_cast<int>(blockIdx.x) >= m.nrec_el) {
    acoustic_seismogram(m.rec_ac[blockIdx.x - m.nrec_el], m.nrec, m.ntypes, m.types, isig, m.rec_ispec, m.gather,
                        m.rec_h, m.pg.xix, m.pg.xiz, m.pg.gammax, m.pg.gammaz, m.rho_inv, q,
                        Fields{ac.u, ac.v, m.dd, ac.minv, ac.nglob_pad}, m.seismo, su[0]);
    return;
  }
  const int r = m.rec_el[blockIdx.x], p = threadIdx.x, np = el.nglob_pad, e = m.rec_ispec[r];
  float u[2] = {0, 0}, v[2] = {0, 0}, a[2] = {0, 0}, hw = 0.0f;
  if (p < 25) {
    const int g = m.gather[static_cast<size_t>(e) * 25 + p];
    hw = m.rec_h[static_cast<size_t>(r) * 25 + p];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      u[c] = el.u[c * np + g];
      v[c] = el.v[c * np + g];
      a[c] = el.a[c * np + g];
    }
    add_contributions<2>(m, m.ent_el[g], a);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      a[c] = a[c] * el.minv[c * np + g];
      su[c][p] = u[c];
    }
  }
  __syncthreads();
  for (int it = 0; it < m.ntypes; it++) {
    const int type = m.types[it];
    float x[2];
    if (type == 3) {
      x[0] = p < 25 ? pressure_2d(m.pg, q, su, e, p) : 0.0f;
      x[1] = 0.0f;
    } else {
#pragma unroll
      for (int c = 0; c < 2; c++) x[c] = type == 0 ? u[c] : type == 1 ? fmaf(dto2, a[c], v[c]) : a[c];
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
      float s = hw * x[c];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
      if (p == 0) m.seismo[((static_cast<size_t>(isig) * m.ntypes + it) * m.nrec + r) * 2 + c] = s;
    }
  }
}

}  // namespace

void launch_acoustic_stiffness_2d(hipStream_t s, int first, int count, bool atomic, const int *gather,
                                  const float *xix, const float *xiz, const float *gammax, const float *gammaz,
                                  const float *jac, const float *rho_inv, const float *stacey, const int *dirichlet,
                                  const GllConst &q, Fields f) {
  if (count <= 0) return;
  if (atomic)
    hipLaunchKernelGGL(acoustic_stiffness_2d_kernel<true>, dim3(blocks_of(count, EA)), dim3(128), 0, s, first, count,
                       gather, xix, xiz, gammax, gammaz, jac, rho_inv, stacey, dirichlet, q, f);
  else
    hipLaunchKernelGGL(acoustic_stiffness_2d_kernel<false>, dim3(blocks_of(count, EA)), dim3(128), 0, s, first,
                       count, gather, xix, xiz, gammax, gammaz, jac, rho_inv, stacey, dirichlet, q, f);
}

void launch_coupling_2d(hipStream_t s, int n, const int *self, const int *other, const float *coef, Fields dst,
                        Fields src, int to_elastic) {
  if (n <= 0) return;
  hipLaunchKernelGGL(coupling_2d_kernel, dim3(blocks_of(n, 256)), dim3(256), 0, s, n, self, other, coef, dst, src,
                     to_elastic);
}

void launch_acoustic_sources(hipStream_t s, int norder, int nsrc, int istep, const int *order, const int *ispec,
                             const int *gather, const float *array, const float *stf, const float *kappa, Fields f) {
  if (norder <= 0) return;
  hipLaunchKernelGGL(acoustic_sources_kernel, dim3(norder), dim3(64), 0, s, norder, nsrc, istep, order, ispec, gather,
                     array, stf, kappa, f);
}

void launch_acoustic_seismograms(hipStream_t s, int nlist, const int *list, int nrec, int ntypes, const int *types,
                                 int isig, const int *ispec, const int *gather, const float *h, const float *xix,
                                 const float *xiz, const float *gammax, const float *gammaz, const float *rho_inv,
                                 const GllConst &q, Fields f, float *seismo) {
  if (nlist <= 0 || ntypes <= 0) return;
  hipLaunchKernelGGL(acoustic_seismogram_kernel, dim3(nlist), dim3(64), 0, s, list, nrec, ntypes, types, isig, ispec,
                     gather, h, xix, xiz, gammax, gammaz, rho_inv, q, f, seismo);
}

void launch_coupled_forces(hipStream_t s, const CoupledStep &m, const GllConst &q, int istep, Fields el, Fields ac) {
  const unsigned b_ac = blocks_of(m.nel, EA), b_src = b_ac + blocks_of(m.nac, EA), b_src_ac = b_src + m.nsrc_el,
                 b_bnd = b_src_ac + m.nsrc_ac, b_cpl = b_bnd + blocks_of(m.nbnd, 128),
                 n = b_cpl + blocks_of(m.ncpl_ac, 128);
  hipLaunchKernelGGL(coupled_forces_kernel, dim3(n), dim3(128), 0, s, m, q, istep, el, ac, static_cast<int>(b_ac),
                     static_cast<int>(b_src), static_cast<int>(b_src_ac), static_cast<int>(b_bnd),
                     static_cast<int>(b_cpl));
}

void launch_coupled_acoustic(hipStream_t s, const CoupledStep &m, Fields ac, NewmarkConst nc) {
  hipLaunchKernelGGL(coupled_acoustic_kernel, dim3(blocks_of(m.nglob_ac, 256)), dim3(256), 0, s, m, ac, nc);
}

void launch_coupled_seismograms(hipStream_t s, const CoupledStep &m, const GllConst &q, int isig, Fields el, Fields ac,
                                float dto2) {
  if (m.nrec_el + m.nrec_ac <= 0 || m.ntypes <= 0) return;
  hipLaunchKernelGGL(coupled_seismogram_kernel, dim3(m.nrec_el + m.nrec_ac), dim3(64), 0, s, m, q, isig, el, ac, dto2);
}

void launch_coupled_update(hipStream_t s, const CoupledStep &m, Fields el, Fields ac, NewmarkConst nc) {
  const unsigned b_ac = blocks_of(m.nglob_el, 256);
  hipLaunchKernelGGL(coupled_update_kernel, dim3(b_ac + blocks_of(m.nglob_ac, 256)), dim3(256), 0, s, m, el, ac, nc,
                     static_cast<int>(b_ac));
}

}  // namespace sfx
