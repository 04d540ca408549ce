// 2-D patch kernels (gfx950, wave64): one workgroup advances one patch of
// elements by a time step (see patch2d.hpp).
//
// Reference kernels these replace (include/kokkos_kernels/impl/):
//   compute_stiffness_interaction.tpp:143-259, its Stacey branch
//   (boundary_conditions/stacey/stacey.tpp:36-72), compute_source_interaction
//   .tpp:80-95, compute_seismogram.tpp:103-135, divide_mass_matrix.tpp:42-49
//   and newmark.tpp:11-116 in one launch.
//
// Measured on MI355X against the kernels these replaced (element forces to
// memory, then one pass per point: two launches and 130 bytes per point
// moved; or nine launches per step with element colors), per step:
//   80 x 80 quads          8.4 us   (colored: 32 us, bound by its launches)
//   177 x 131, moved      11.5 us   (two-pass: 36 us)
//   1000 x 900, random   247 us     (two-pass: 424 us)
// At the large size a launch moves 44 bytes per point (2.6 TB/s) and keeps the
// vector units busy for 150 of its 247 us (1,100 instructions per wavefront;
// without fused multiply-adds in the exact form): it is bound by the latency
// of its phases at five wavefronts per SIMD.  Workgroups of four wavefronts
// matter: with five (64 elements) only 2.3 of 4 workgroups were resident per
// CU and the same step took 318 us.
#include "division.hpp"
#include "lattice.hpp"
#include "patch2d.hpp"

namespace sfx {

namespace {

// a * b + c: with EXACT the product is rounded before the sum, else one fused
// multiply-add.
template <bool EXACT> __device__ __forceinline__ float mad(float a, float b, float c) {
  if constexpr (EXACT) {
#pragma clang fp contract(off)
    return a * b + c;
  } else {
    return fmaf(a, b, c);
  }
}

// a[i] with a uniform base and a 32-bit byte offset (i < 2^30)
__device__ __forceinline__ float at(const float *a, unsigned i) {
  return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(a) + (i * 4u));
}
__device__ __forceinline__ int at(const uint16_t *a, unsigned i) {
  return *reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(a) + (i * 2u));
}
__device__ __forceinline__ void put(float *a, unsigned i, float v) {
  *reinterpret_cast<float *>(reinterpret_cast<char *>(a) + (i * 4u)) = v;
}

// The row constants of the four-node form: x and z derivatives in xi.
template <int GEOM>
__device__ __forceinline__ void row_geometry(const Geom2D &gm, int row, const float *c, float &xxi, float &zxi) {
#pragma clang fp contract(off)
  xxi = 0.0f;
  zxi = 0.0f;
  if constexpr (GEOM == GEOM2D_CTRL4) {
    const float *d = gm.dsh + row * 40;
    xxi = d[0] * c[0];
    zxi = d[0] * c[1];
#pragma unroll
    for (int n = 1; n < 4; n++) {
      xxi += d[n] * c[2 * n];
      zxi += d[n] * c[2 * n + 1];
    }
  }
}

// Geometry of local point p = row * 5 + i of element e (plan order); the
// control-node forms repeat the host's float operations in the host's order
// (no contraction, correctly rounded division).  c: the element's control
// nodes, or its record.
template <int GEOM>
__device__ __forceinline__ void patch_geometry(const Geom2D &gm, int e, int row, int i, const float *c, float xxi,
                                               float zxi, float &xix, float &xiz, float &gammax, float &gammaz,
                                               float &J) {
#pragma clang fp contract(off)
  const int p = row * 5 + i;
  if constexpr (GEOM == GEOM2D_POINT) {
    const size_t idx = static_cast<size_t>(e) * 25 + p;
    xix = gm.xix[idx];
    xiz = gm.xiz[idx];
    gammax = gm.gammax[idx];
    gammaz = gm.gammaz[idx];
    J = gm.jac[idx];
  } else if constexpr (GEOM == GEOM2D_RECORD) {
    xix = c[0];
    xiz = c[1];
    gammax = c[2];
    gammaz = c[3];
    J = c[4];
  } else {
    float xgamma = 0.0f, zgamma = 0.0f;
    if constexpr (GEOM == GEOM2D_CTRL4) {
      const float *d = gm.dsh + i * 8 + 4;
      xgamma = d[0] * c[0];
      zgamma = d[0] * c[1];
#pragma unroll
      for (int n = 1; n < 4; n++) {
        xgamma += d[n] * c[2 * n];
        zgamma += d[n] * c[2 * n + 1];
      }
    } else {
      constexpr int NG = GEOM;
      const float *d = gm.dsh + p * (2 * NG);
      xxi = 0.0f;
      zxi = 0.0f;
#pragma unroll
      for (int n = 0; n < NG; n++) {
        xxi += d[n] * c[2 * n];
        zxi += d[n] * c[2 * n + 1];
        xgamma += d[NG + n] * c[2 * n];
        zgamma += d[NG + n] * c[2 * n + 1];
      }
    }
    J = xxi * zgamma - xgamma * zxi;
    const float y = reciprocal(J);
    xix = quotient(zgamma, J, y);
    gammax = quotient(-zxi, J, y);
    xiz = quotient(-xgamma, J, y);
    gammaz = quotient(xxi, J, y);
  }
}

template <int PE> constexpr int patch_threads() { return (PE * 5 + 63) / 64 * 64; }

// Sum of an interior point's contributions in order, the first one (table
// entry ea) given: its local index l tells how many there are (the points are
// sorted by that number).
__device__ __forceinline__ float2 interior_force(const PatchHead &h, const uint16_t *__restrict__ tab,
                                                 const float *st, int l, int ea, int eb) {
#pragma clang fp contract(off)
  const float2 *f = reinterpret_cast<const float2 *>(st);
  float2 s = f[ea];
  if (l >= h.n1) {
    const float2 r = f[eb];
    s.x += r.x;
    s.y += r.y;
    const int m = l - h.n1 - h.n2;
    if (m >= 0)
      for (int k = tab[h.off3 + m]; k < tab[h.off3 + m + 1]; k++) {
        const float2 q = f[tab[h.ent3 + k]];
        s.x += q.x;
        s.y += q.y;
      }
  }
  return s;
}

template <bool EXACT> struct Newmark {
  float dt, dto2, dt2o2;
  // corrector of this step and predictor of the next: v1 is the corrected
  // velocity (divide_mass_matrix.tpp:42-49, newmark.tpp:11-116)
  __device__ __forceinline__ void operator()(float a, float &u, float &v, float &v1) const {
    v1 = mad<EXACT>(dto2, a, v);
    if constexpr (EXACT) {
#pragma clang fp contract(off)
      u = u + (dt * v1 + dt2o2 * a);
      v = v1 + dto2 * a;
    } else {
      u = u + fmaf(dt2o2, a, dt * v1);  // as the colored path's update contracts it
      v = fmaf(dto2, a, v1);
    }
  }
};

// Sum of n contributions from k0 on, in order, after a0 and a1; the first four
// are loaded together (indices clamped to the last one).
__device__ __forceinline__ void boundary_force(const float2 *__restrict__ rb, int k0, int n, float s[2],
                                               float a0 = 0.0f, float a1 = 0.0f) {
#pragma clang fp contract(off)
  float2 r[4];
#pragma unroll
  for (int j = 0; j < 4; j++) r[j] = rb[k0 + (j < n ? j : n - 1)];
  s[0] = a0;
  s[1] = a1;
#pragma unroll
  for (int j = 0; j < 4; j++)
    if (j < n) {
      s[0] += r[j].x;
      s[1] += r[j].y;
    }
  for (int j = 4; j < n; j++) {
    const float2 q = rb[k0 + j];
    s[0] += q.x;
    s[1] += q.y;
  }
}

// Where the boundary state of a launch lies.
struct BoundaryState {
  const float *u0, *u1, *v0, *v1;
};
__device__ __forceinline__ BoundaryState boundary_state(const PatchTables &T, const PatchState &S, int rd) {
  const size_t nb = T.nbnd;
  if (rd) return {S.ub, S.ub + nb, S.ub + 2 * nb, S.ub + 3 * nb};
  return {S.u + T.nint, S.u + T.np + static_cast<size_t>(T.nint), S.v + T.nint, S.v + T.np + static_cast<size_t>(T.nint)};
}

// Samples of step `step` at one receiver, by one wavefront (compute_seismogram
// .tpp:103-135): u, corrected v and a at its element's points, from the
// snapshot the last launch took of interior points and, for boundary points,
// from the state and contributions that launch left in buffers rd.  sign: of
// the time step; top: sample index of step 0 when the steps run backwards, or -1.
template <int GEOM, bool EPROP, bool EXACT>
__device__ __forceinline__ void sample_receiver(int r, bool store, int step, int top, float sign, int rd,
                                                const PatchTables &T, const PatchState &S, const GllConst &q) {
  const int lane = threadIdx.x & 63;
  const int p = lane < 25 ? lane : 0;
  const int4 rc = T.rec[r];
  const int rp = T.rp_of[r * 25 + p];
  const PatchSim sim = T.sim[rc.z];
  const float hw = lane < 25 ? T.rec_h[static_cast<size_t>(rc.x) * 25 + p] : 0.0f;
  store = store && step >= 0 && step < sim.nstep && step % sim.nsb == 0 && lane == 0;
  const int isig = top >= 0 ? top - step / sim.nsb : step / sim.nsb;
  float x[6];
  if (rp >= 0) {
    const float *smp = T.snap + 6 * (static_cast<size_t>(rd) * T.nrow + rp);
#pragma unroll
    for (int i = 0; i < 6; i++) x[i] = smp[i];
  } else {
#pragma clang fp contract(off)
    const int b = -1 - rp;
    const BoundaryState bs = boundary_state(T, S, rd);
    const float u[2] = {bs.u0[b], bs.u1[b]}, v[2] = {bs.v0[b], bs.v1[b]};
    float s[2];
    const int k0 = T.boff[b];
    boundary_force(S.rb[rd], k0, T.boff[b + 1] - k0, s);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const float a = s[c] * T.minv[c * static_cast<size_t>(T.np) + T.nint + b];
      x[c] = u[c];
      x[2 + c] = mad<EXACT>(sign * sim.dto2, a, v[c]);
      x[4 + c] = a;
    }
  }
  for (int it = 0; it < T.ntypes; it++) {
    const int type = T.types[it];
    float val[2];
    if (type == 3) {
      // pressure (include/medium/dim2/elastic/isotropic/wavefield.hpp:49-85)
      const int iz = p / 5, ix = p - iz * 5;
      float dxi[2] = {0.0f, 0.0f}, dga[2] = {0.0f, 0.0f};
#pragma unroll
      for (int l = 0; l < 5; l++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          dxi[c] += q.hp[ix][l] * __shfl(x[c], iz * 5 + l, 64);
          dga[c] += q.hp[iz][l] * __shfl(x[c], l * 5 + ix, 64);
        }
      const size_t e = rc.w;
      constexpr int NC = GEOM == GEOM2D_POINT ? 1 : GEOM == GEOM2D_RECORD ? 8 : 2 * GEOM;
      const float *cc = GEOM == GEOM2D_POINT ? nullptr : (GEOM == GEOM2D_RECORD ? T.geom.record : T.geom.ctrl) + e * NC;
      float xxi, zxi, xix, xiz, gammax, gammaz, J;
      row_geometry<GEOM>(T.geom, iz, cc, xxi, zxi);
      patch_geometry<GEOM>(T.geom, rc.w, iz, ix, cc, xxi, zxi, xix, xiz, gammax, gammaz, J);
      const float du00 = xix * dxi[0] + gammax * dga[0];
      const float du11 = xiz * dxi[1] + gammaz * dga[1];
      const float kap = EPROP ? T.kmu[2 * e] : T.kappa[e * 25 + p];
      const float mu = EPROP ? T.kmu[2 * e + 1] : T.mu[e * 25 + p];
      const float lp2m = kap + (4.0f / 3.0f) * mu;
      const float lambda = lp2m - 2.0f * mu;
      const double fac = static_cast<double>(lambda) + (2.0 / 3.0) * static_cast<double>(mu);
      val[0] = hw * static_cast<float>(-1.0 * (fac * static_cast<double>(du00 + du11)));
      val[1] = 0.0f;
    } else {
#pragma unroll
      for (int c = 0; c < 2; c++) val[c] = hw * (type == 0 ? x[c] : type == 1 ? x[2 + c] : x[4 + c]);
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
      float s = lane < 25 ? val[c] : 0.0f;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
      // + 0: the sum over a second, empty wavefront
      if (store)
        T.seismo[sim.seis + ((static_cast<long long>(isig) * T.ntypes + it) * sim.nrec + rc.y) * 2 + c] = s + 0.0f;
    }
  }
}

// A time step of one patch.  Thread t holds row t % 5 (five points along xi)
// of element t / 5: the xi contractions stay in registers, the gamma ones read
// the element's other rows from LDS.  Workgroups past the patches sample the
// receivers, one wavefront each.
// Five wavefronts per SIMD (96 registers): 269 us at 1000 x 900 with four.
// RECORD (contracted form): the Stacey elements' forces are kept for the adjoint
// run; in a form of its own, as its branches cost the plain step 1 us in 8.
template <int PE, int GEOM, bool EPROP, bool EXACT, bool RECORD>
__global__ __launch_bounds__(patch_threads<PE>()) __attribute__((amdgpu_waves_per_eu(5))) void patch_step_kernel(int npatch, int nrec, PatchTables T,
                                                                        PatchState S, GllConst q, PatchLaunch L) {
  constexpr int NT = patch_threads<PE>();
  constexpr int NP = PatchCap<PE>::points, NB = PatchCap<PE>::boundary;
  constexpr int NI = (NP + NT - 1) / NT;       // interior points per thread
  static_assert(NB <= NT, "one boundary point per thread");
  __shared__ float su[2][NP];                  // displacement of the patch's points
  __shared__ float sv[2][NB];                  // velocity of its boundary points
  // displacement by element, then the element forces; F(c, gamma), then
  // (contracted form) the Stacey terms
  __shared__ __align__(16) float se[PE * 100];
  float *const sF = se + PE * 50;

  const int t = threadIdx.x;
  const int n = (L.base ? *L.base : 0) + L.step;
  if (L.next && blockIdx.x == 0 && t == 0) *L.next = n + 1;
  if (static_cast<int>(blockIdx.x) >= npatch) {
    const int r = (blockIdx.x - npatch) * (NT / 64) + (t >> 6);  // wavefronts past the last receiver repeat it
    sample_receiver<GEOM, EPROP, EXACT>(r < nrec ? r : nrec - 1, r < nrec, n - 1, -1, 1.0f, L.rd, T, S, q);
    return;
  }
  const PatchHead h = T.head[xcd_block(blockIdx.x, npatch)];
  if (n >= h.nstep) return;
  const Newmark<EXACT> newmark{h.dt, h.dto2, h.dt2o2};
  const size_t np = T.np;
  const uint16_t *__restrict__ tab = T.tab;

  // All loads that depend on the patch alone are issued here, without
  // branches: idle lanes repeat the last element (and store its values again),
  // point or entry.
  const int le = t / 5, row = t - le * 5;
  const int lc = le < h.nel ? le : h.nel - 1;
  const int e = h.el0 + lc;
  PatchPoint bp{0, 0, 1, 0};
  if (h.nb > 0) bp = T.bpt[h.b0 + (t < h.nb ? t : h.nb - 1)];
  // the patch's interior points and elements: uniform bases
  float *const u0p = S.u + h.pt0, *const u1p = S.u + np + h.pt0;
  float *const v0p = S.v + h.pt0, *const v1p = S.v + np + h.pt0;
  const float *const m0p = T.minv + h.pt0, *const m1p = T.minv + np + h.pt0;
  float ui[NI][2];
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int l = t + k * NT;
    const unsigned g = l < h.nint ? l : h.nint - 1;
    ui[k][0] = at(u0p, g);
    ui[k][1] = at(u1p, g);
  }
  const uint4 rw = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(tab + h.lidx) + (lc * 5 + row) * 16u);
  constexpr int NC = GEOM == GEOM2D_POINT ? 1 : GEOM == GEOM2D_RECORD ? 8 : 2 * GEOM;
  float ctrl[NC];
  if constexpr (GEOM != GEOM2D_POINT) {
    const float *c = (GEOM == GEOM2D_RECORD ? T.geom.record : T.geom.ctrl) + static_cast<size_t>(h.el0) * NC;
#pragma unroll
    for (int i = 0; i < NC; i++) ctrl[i] = at(c, lc * NC + i);
  }
  float ke = 0.0f, me = 0.0f;
  if constexpr (EPROP) {
    const float *km = T.kmu + 2 * static_cast<size_t>(h.el0);
    ke = at(km, 2 * lc);
    me = at(km, 2 * lc + 1);
  }
  // boundary points first receive the contributions of the last step
  if (h.nb > 0) {
#pragma clang fp contract(off)
    const int b = bp.b & 0x7fffffff;
    const size_t o = T.nint + static_cast<size_t>(b);
    const BoundaryState bs = boundary_state(T, S, L.rd);
    float u[2] = {bs.u0[b], bs.u1[b]}, v[2] = {bs.v0[b], bs.v1[b]};
    if (L.pending) {
      const float m[2] = {T.minv[o], T.minv[np + o]};
      float s[2];
      boundary_force(S.rb[L.rd], bp.k0, bp.n, s);
#pragma unroll
      for (int c = 0; c < 2; c++) {
        float v1;
        newmark(s[c] * m[c], u[c], v[c], v1);
      }
    }
    if (t < h.nb) {
      su[0][h.nint + t] = u[0];
      su[1][h.nint + t] = u[1];
      sv[0][t] = v[0];
      sv[1][t] = v[1];
      if (bp.b < 0 && L.advance) {  // the owner passes the state on
        const BoundaryState to = boundary_state(T, S, L.rd ^ 1);
        const_cast<float *>(to.u0)[b] = u[0];
        const_cast<float *>(to.u1)[b] = u[1];
        const_cast<float *>(to.v0)[b] = v[0];
        const_cast<float *>(to.v1)[b] = v[1];
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NI; k++)
    if (t + k * NT < h.nint) {
      su[0][t + k * NT] = ui[k][0];
      su[1][t + k * NT] = ui[k][1];
    }
  __syncthreads();

  // the row's displacement in registers and, by element, in LDS
  const unsigned li[5] = {rw.x & 0xffffu, rw.x >> 16, rw.y & 0xffffu, rw.y >> 16, rw.z & 0xffffu};
  float u[2][5];
#pragma unroll
  for (int i = 0; i < 5; i++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      u[c][i] = su[c][li[i]];
      se[lc * 50 + c * 25 + row * 5 + i] = u[c][i];
    }
  float hrow[5], hwrow[5];
#pragma unroll
  for (int l = 0; l < 5; l++) {
    hrow[l] = q.hp[row][l];
    hwrow[l] = q.hpw[row][l];
  }
  float xxi, zxi;
  row_geometry<GEOM>(T.geom, row, ctrl, xxi, zxi);
  __syncthreads();
  float F[2][5];  // F(c, xi) of the row
#pragma unroll
  for (int i = 0; i < 5; i++) {
    float dxi[2], dga[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      dxi[c] = q.hp[i][0] * u[c][0];
      dga[c] = hrow[0] * se[lc * 50 + c * 25 + i];
#pragma unroll
      for (int l = 1; l < 5; l++) {
        dxi[c] = mad<EXACT>(q.hp[i][l], u[c][l], dxi[c]);
        dga[c] = mad<EXACT>(hrow[l], se[lc * 50 + c * 25 + l * 5 + i], dga[c]);
      }
    }
    const int p = row * 5 + i;
    float xix, xiz, gammax, gammaz, J;
    patch_geometry<GEOM>(T.geom, e, row, i, ctrl, xxi, zxi, xix, xiz, gammax, gammaz, J);
    float kappa = ke, mu = me;
    if constexpr (!EPROP) {
      kappa = T.kappa[static_cast<size_t>(e) * 25 + p];
      mu = T.mu[static_cast<size_t>(e) * 25 + p];
    }
    {
#pragma clang fp contract(off)
      float du[2][2];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        du[c][0] = mad<EXACT>(xix, dxi[c], gammax * dga[c]);
        du[c][1] = mad<EXACT>(xiz, dxi[c], gammaz * dga[c]);
      }
      // include/medium/dim2/elastic/isotropic/stress.hpp:25-48 with
      // lambda + 2 mu = kappa + 4/3 mu
      const float lp2m = mad<EXACT>(4.0f / 3.0f, mu, kappa);
      const float lambda = lp2m - 2.0f * mu;
      const float sxx = mad<EXACT>(lp2m, du[0][0], lambda * du[1][1]);
      const float szz = mad<EXACT>(lp2m, du[1][1], lambda * du[0][0]);
      const float sxz = mu * (du[0][1] + du[1][0]);
      // core/specfem/point/stress.hpp:129-136
      F[0][i] = J * mad<EXACT>(sxx, xix, sxz * xiz);
      F[1][i] = J * mad<EXACT>(sxz, xix, szz * xiz);
      sF[lc * 25 + p] = J * mad<EXACT>(sxx, gammax, sxz * gammaz);
      sF[PE * 25 + lc * 25 + p] = J * mad<EXACT>(sxz, gammax, szz * gammaz);
    }
    // one point after the other: interleaving all five would need more
    // registers than five wavefronts per SIMD have
    __builtin_amdgcn_sched_barrier(0);
  }
  // what the update reads, requested now: the velocity, M^-1 (its components
  // are equal where no Stacey term enters) and the first contributions
  float vi[NI][2], mi[NI][2];
  int ea[NI], eb[NI];
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int l = t + k * NT;
    const int ll = l < h.nint ? l : h.nint - 1;
    vi[k][0] = at(v0p, ll);
    vi[k][1] = at(v1p, ll);
    mi[k][0] = at(m0p, ll);
    mi[k][1] = mi[k][0];
    if (h.nseg > 0) mi[k][1] = at(m1p, ll);
    ea[k] = at(tab + h.enta, ll);
    eb[k] = at(tab + h.entb, ll >= h.n1 && h.n1 < h.nint ? ll - h.n1 : 0);
  }
  __syncthreads();
  // include/algorithms/divergence.hpp:86-98; the forces overwrite the
  // displacement in se (all reads of it are before the barrier)
  const float wrow = q.w[row];
#pragma unroll
  for (int i = 0; i < 5; i++) {
    float r[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma clang fp contract(off)
      float t1 = F[c][0] * q.hpw[i][0], t2 = sF[c * PE * 25 + lc * 25 + i] * hwrow[0];
#pragma unroll
      for (int l = 1; l < 5; l++) {
        t1 = mad<EXACT>(F[c][l], q.hpw[i][l], t1);
        t2 = mad<EXACT>(sF[c * PE * 25 + lc * 25 + l * 5 + i], hwrow[l], t2);
      }
      r[c] = -mad<EXACT>(wrow, t1, q.w[i] * t2);
    }
    *reinterpret_cast<float2 *>(&se[lc * 50 + 2 * (row * 5 + i)]) = make_float2(r[0], r[1]);
    if constexpr (RECORD)
      if (T.rec_row[e] >= 0)
        *reinterpret_cast<float2 *>(L.rec + n * L.rec_stride + (static_cast<size_t>(T.rec_row[e]) * 25 + row * 5 + i) * 2) =
            make_float2(r[0], r[1]);
  }
  __syncthreads();

  if (h.nseg > 0) {
    // Stacey traction with the predicted velocity (stacey.tpp:36-72), the
    // entries of an element point summed in order; EXACT adds them to the
    // element's force, as the oracle does, otherwise they are contributions of
    // their own, summed last
    for (int sg = h.seg0 + t; sg < h.seg0 + h.nseg; sg += NT) {
#pragma clang fp contract(off)
      const int l = T.seg_loc[sg], sp = T.seg_pt[sg];
      const int k0 = T.seg_off[sg], k1 = T.seg_off[sg + 1];
      float v[2];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        if (l < h.nint)
          v[c] = S.v[c * np + h.pt0 + l];
        else
          v[c] = sv[c][l - h.nint];
      }
      float s[2] = {0.0f, 0.0f};
      for (int k = k0; k < k1; k++) {
        const float nv[2] = {T.bnormal[2 * k], T.bnormal[2 * k + 1]};
        const float w = T.bweight[k], rvp = T.brvp[k], rvs = T.brvs[k];
        const float vn = mad<EXACT>(v[1], nv[1], v[0] * nv[0]);
        const float nn = mad<EXACT>(nv[0], nv[0], nv[1] * nv[1]);
        const float j1 = sqrtf(nn);
#pragma unroll
        for (int d = 0; d < 2; d++) {
          const float fac = mad<EXACT>(rvs, v[d], (vn * nv[d] / (j1 * j1)) * (rvp - rvs));
          s[d] += -1.0f * fac * j1 * w;
        }
      }
      if constexpr (EXACT) {
        se[2 * sp] += s[0];
        se[2 * sp + 1] += s[1];
      } else {
        reinterpret_cast<float2 *>(sF)[sg - h.seg0] = make_float2(s[0], s[1]);
        if constexpr (RECORD)  // a Stacey element's record holds its force with the traction
          *reinterpret_cast<float2 *>(L.rec + n * L.rec_stride +
                                      (static_cast<size_t>(T.rec_row[h.el0 + sp / 25]) * 25 + sp % 25) * 2) =
              make_float2(se[2 * sp] + s[0], se[2 * sp + 1] + s[1]);
      }
    }
    __syncthreads();
  }
  if (h.nsrc > 0) {
    // sources: 25 threads per element that holds some, each adding all of them
    // at its point in application order
    for (int k = t / 25; k < h.nsrc; k += NT / 25) {
      const int4 se4 = T.src_el[h.src0 + k];
      const int p = t % 25;
      if (t / 25 == NT / 25) break;
      // EXACT adds them to the force one by one, as the oracle does; otherwise
      // their sum is a contribution of its own
      float2 *const f = reinterpret_cast<float2 *>(se) + (EXACT ? se4.x : PE + k) * 25 + (EXACT ? 0 : h.nseg) + p;
      float o[2] = {EXACT ? f->x : 0.0f, EXACT ? f->y : 0.0f};
      for (int i = se4.y; i < se4.z; i++) {
#pragma clang fp contract(off)
        const int id = T.src_id[i];
        const float amp = T.stf[n * T.stf_step + id * T.stf_src];
#pragma unroll
        for (int c = 0; c < 2; c++) o[c] += amp * T.src_array[(static_cast<size_t>(id) * 2 + c) * 25 + p];
      }
      *f = make_float2(o[0], o[1]);
    }
    __syncthreads();
  }

  // contributions of the boundary points, for the next launch
  {
    float2 *out = S.rb[L.rd ^ 1];
    const float2 *f = reinterpret_cast<const float2 *>(se);
    for (int k = t; k < h.nbent; k += NT) out[T.bslot[h.be0 + k]] = f[tab[h.bent + k]];
  }
  const bool snapshot = h.rm0 >= 0 && L.advance && n % h.nsb == 0;
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int l = t + k * NT;
    if (l >= h.nint) continue;
    const float2 s = interior_force(h, tab, se, l, ea[k], eb[k]);
    const float a0 = s.x * mi[k][0], a1 = s.y * mi[k][1];
    if (L.advance) {
      float u0 = su[0][l], u1 = su[1][l], v0 = vi[k][0], v1 = vi[k][1], w0, w1;
      newmark(a0, u0, v0, w0);
      newmark(a1, u1, v1, w1);
      put(u0p, l, u0);
      put(u1p, l, u1);
      put(v0p, l, v0);
      put(v1p, l, v1);
      if (snapshot) {  // of a receiver's element point, before it was advanced
        const int rowi = T.rmap[h.rm0 + l];
        if (rowi >= 0) {
          float *o = T.snap + 6 * (static_cast<size_t>(L.rd ^ 1) * T.nrow + rowi);
          o[0] = su[0][l];
          o[1] = su[1][l];
          o[2] = w0;
          o[3] = w1;
          o[4] = a0;
          o[5] = a1;
        }
      }
    }
    if (!L.advance || L.store_a) {
      float *const a0p = S.a + h.pt0, *const a1p = S.a + np + h.pt0;
      // a force held in the stored a joins here, out of the way of fused steps
      const bool add = !EXACT && L.add_a;
      put(a0p, l, add ? (s.x + at(a0p, l)) * mi[k][0] : a0);
      put(a1p, l, add ? (s.y + at(a1p, l)) * mi[k][1] : a1);
    }
  }
}

// One step of the combined adjoint + backward loop (time_marching.tpp:160-215)
// of one patch: the adjoint field (A, forward in time, adjoint sources, Stacey)
// and then the backward field (B, -dt, forward sources, the recorded force at
// Stacey elements, compute_stiffness_interaction.tpp:119-136) go through the
// phases of patch_step_kernel one after the other in the same LDS; the adjoint
// gradients and accelerations stay in registers for the Frechet kernels'
// products (frechet_derivative.hpp:58-118): Kmu, Kkappa per element point, R
// (of the rho kernel) per point.
template <int PE, int GEOM, bool EPROP>
__global__ __launch_bounds__(patch_threads<PE>()) __attribute__((amdgpu_waves_per_eu(4))) void patch_pair_kernel(
    int npatch, int nrec, PatchTables T, PatchState A, PatchState B, GllConst q, PatchPairLaunch L, PatchPairTables P) {
  constexpr int NT = patch_threads<PE>();
  constexpr int NP = PatchCap<PE>::points, NB = PatchCap<PE>::boundary;
  constexpr int NI = (NP + NT - 1) / NT;
  __shared__ float su[2][NP];
  __shared__ float sv[2][NB];
  __shared__ __align__(16) float se[PE * 100];
  float *const sF = se + PE * 50;
  float2 *const f2 = reinterpret_cast<float2 *>(se);
  float2 *const fx = reinterpret_cast<float2 *>(sF);  // Stacey and source contributions

  const int t = threadIdx.x;
  if (static_cast<int>(blockIdx.x) >= npatch) {
    const int r = (blockIdx.x - npatch) * (NT / 64) + (t >> 6);
    sample_receiver<GEOM, EPROP, false>(r < nrec ? r : nrec - 1, r < nrec, L.step + 1, L.top, -1.0f, L.rd, T, B, q);
    return;
  }
  const int patch = xcd_block(blockIdx.x, npatch);
  const PatchHead h = T.head[patch];
  const size_t np = T.np;
  const uint16_t *__restrict__ tab = T.tab;
  const int le = t / 5, row = t - le * 5;
  const int lc = le < h.nel ? le : h.nel - 1;
  const int e = h.el0 + lc;
  const int rrow = T.rec_row[e];
  const size_t krow = static_cast<size_t>(P.kslot[e]) * 25 + row * 5;
  PatchPoint bp{0, 0, 1, 0};
  if (h.nb > 0) bp = T.bpt[h.b0 + (t < h.nb ? t : h.nb - 1)];
  const uint4 rw = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(tab + h.lidx) + (lc * 5 + row) * 16u);
  const unsigned li[5] = {rw.x & 0xffffu, rw.x >> 16, rw.y & 0xffffu, rw.y >> 16, rw.z & 0xffffu};
  constexpr int NC = GEOM == GEOM2D_POINT ? 1 : GEOM == GEOM2D_RECORD ? 8 : 2 * GEOM;
  float ctrl[NC];
  if constexpr (GEOM != GEOM2D_POINT) {
    const float *c = (GEOM == GEOM2D_RECORD ? T.geom.record : T.geom.ctrl) + static_cast<size_t>(h.el0) * NC;
#pragma unroll
    for (int i = 0; i < NC; i++) ctrl[i] = at(c, lc * NC + i);
  }
  float ke = 0.0f, me = 0.0f;
  if constexpr (EPROP) {
    const float *km = T.kmu + 2 * static_cast<size_t>(h.el0);
    ke = at(km, 2 * lc);
    me = at(km, 2 * lc + 1);
  }
  float hrow[5], hwrow[5];
#pragma unroll
  for (int l = 0; l < 5; l++) {
    hrow[l] = q.hp[row][l];
    hwrow[l] = q.hpw[row][l];
  }
  const float wrow = q.w[row];
  float xxi, zxi;
  row_geometry<GEOM>(T.geom, row, ctrl, xxi, zxi);

  float dua[5][4];          // adjoint gradients of the row
  float aa[NI][2], ab[2];   // adjoint acceleration: interior, boundary point
#pragma unroll
  for (int fi = 0; fi < 2; fi++) {
    const PatchState &S = fi ? B : A;
    const Newmark<false> newmark{fi ? -h.dt : h.dt, fi ? -h.dto2 : h.dto2, h.dt2o2};
    float *const u0p = S.u + h.pt0, *const u1p = S.u + np + h.pt0;
    float *const v0p = S.v + h.pt0, *const v1p = S.v + np + h.pt0;
    const float *const m0p = T.minv + h.pt0, *const m1p = T.minv + np + h.pt0;
    float ui[NI][2];
#pragma unroll
    for (int k = 0; k < NI; k++) {
      const int l = t + k * NT;
      const unsigned g = l < h.nint ? l : h.nint - 1;
      ui[k][0] = at(u0p, g);
      ui[k][1] = at(u1p, g);
    }
    if (h.nb > 0) {
      const int b = bp.b & 0x7fffffff;
      const size_t o = T.nint + static_cast<size_t>(b);
      const BoundaryState bs = boundary_state(T, S, L.rd);
      float u[2] = {bs.u0[b], bs.u1[b]}, v[2] = {bs.v0[b], bs.v1[b]};
      if (L.pending) {
        const float m[2] = {T.minv[o], T.minv[np + o]};
        float s[2];
        boundary_force(S.rb[L.rd], bp.k0, bp.n, s);
        if (fi == 0) {
          ab[0] = s[0] * m[0];
          ab[1] = s[1] * m[1];
        } else if (t < h.nb && bp.b < 0) {
          P.R[o] += h.dt * fmaf(ab[1], u[1], ab[0] * u[0]);
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {
          float v1;
          newmark(s[c] * m[c], u[c], v[c], v1);
        }
      }
      if (t < h.nb) {
        su[0][h.nint + t] = u[0];
        su[1][h.nint + t] = u[1];
        sv[0][t] = v[0];
        sv[1][t] = v[1];
        if (bp.b < 0) {
          const BoundaryState to = boundary_state(T, S, L.rd ^ 1);
          const_cast<float *>(to.u0)[b] = u[0];
          const_cast<float *>(to.u1)[b] = u[1];
          const_cast<float *>(to.v0)[b] = v[0];
          const_cast<float *>(to.v1)[b] = v[1];
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NI; k++)
      if (t + k * NT < h.nint) {
        su[0][t + k * NT] = ui[k][0];
        su[1][t + k * NT] = ui[k][1];
      }
    __syncthreads();
    float u[2][5];
#pragma unroll
    for (int i = 0; i < 5; i++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        u[c][i] = su[c][li[i]];
        se[lc * 50 + c * 25 + row * 5 + i] = u[c][i];
      }
    __syncthreads();
    float F[2][5];
#pragma unroll
    for (int i = 0; i < 5; i++) {
      float dxi[2], dga[2];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        dxi[c] = q.hp[i][0] * u[c][0];
        dga[c] = hrow[0] * se[lc * 50 + c * 25 + i];
#pragma unroll
        for (int l = 1; l < 5; l++) {
          dxi[c] = fmaf(q.hp[i][l], u[c][l], dxi[c]);
          dga[c] = fmaf(hrow[l], se[lc * 50 + c * 25 + l * 5 + i], dga[c]);
        }
      }
      const int p = row * 5 + i;
      float xix, xiz, gammax, gammaz, J;
      patch_geometry<GEOM>(T.geom, e, row, i, ctrl, xxi, zxi, xix, xiz, gammax, gammaz, J);
      float kappa = ke, mu = me;
      if constexpr (!EPROP) {
        kappa = T.kappa[static_cast<size_t>(e) * 25 + p];
        mu = T.mu[static_cast<size_t>(e) * 25 + p];
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
      F[0][i] = J * fmaf(sxx, xix, sxz * xiz);
      F[1][i] = J * fmaf(sxz, xix, szz * xiz);
      sF[lc * 25 + p] = J * fmaf(sxx, gammax, sxz * gammaz);
      sF[PE * 25 + lc * 25 + p] = J * fmaf(sxz, gammax, szz * gammaz);
      if (fi == 0) {
        dua[i][0] = du[0][0];
        dua[i][1] = du[0][1];
        dua[i][2] = du[1][0];
        dua[i][3] = du[1][1];
      } else if (le < h.nel) {
        // the strain kernels, as stiffness_pair_2d_kernel forms them
        const float kap2 = lp2m - mu;
        const float asxz = 0.5f * (dua[i][2] + dua[i][1]), bsxz = 0.5f * (du[1][0] + du[0][1]);
        const float kk = (dua[i][0] + dua[i][3]) * (du[0][0] + du[1][1]);
        const float km = dua[i][0] * du[0][0] + dua[i][3] * du[1][1] + 2.0f * asxz * bsxz - (1.0f / 3.0f) * kk;
        P.Kkappa[krow + i] += -1.0f * kap2 * h.dt * kk;
        P.Kmu[krow + i] += -2.0f * mu * h.dt * km;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    float vi[NI][2], mi[NI][2], ri[NI];
    int ea[NI], eb[NI];
#pragma unroll
    for (int k = 0; k < NI; k++) {
      const int l = t + k * NT;
      const int ll = l < h.nint ? l : h.nint - 1;
      vi[k][0] = at(v0p, ll);
      vi[k][1] = at(v1p, ll);
      mi[k][0] = at(m0p, ll);
      mi[k][1] = mi[k][0];
      if (h.nseg > 0) mi[k][1] = at(m1p, ll);
      ri[k] = fi ? at(P.R + h.pt0, ll) : 0.0f;
      ea[k] = at(tab + h.enta, ll);
      eb[k] = at(tab + h.entb, ll >= h.n1 && h.n1 < h.nint ? ll - h.n1 : 0);
    }
    float2 rr[5];
#pragma unroll
    for (int i = 0; i < 5; i++) rr[i] = make_float2(0.0f, 0.0f);
    if (fi && rrow >= 0)
#pragma unroll
      for (int i = 0; i < 5; i++)
        rr[i] = *reinterpret_cast<const float2 *>(L.rec + (static_cast<size_t>(rrow) * 25 + row * 5 + i) * 2);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 5; i++) {
      float r[2];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        float t1 = F[c][0] * q.hpw[i][0], t2 = sF[c * PE * 25 + lc * 25 + i] * hwrow[0];
#pragma unroll
        for (int l = 1; l < 5; l++) {
          t1 = fmaf(F[c][l], q.hpw[i][l], t1);
          t2 = fmaf(sF[c * PE * 25 + lc * 25 + l * 5 + i], hwrow[l], t2);
        }
        r[c] = -fmaf(wrow, t1, q.w[i] * t2);
      }
      f2[lc * 25 + row * 5 + i] = fi && rrow >= 0 ? rr[i] : make_float2(r[0], r[1]);
    }
    __syncthreads();
    // the Stacey and source contributions of this field; the other field's
    // are zero
    for (int sg = t; sg < h.nseg; sg += NT) {
      float s[2] = {0.0f, 0.0f};
      if (fi == 0) {
        const int l = T.seg_loc[h.seg0 + sg];
        float v[2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
          if (l < h.nint)
            v[c] = S.v[c * np + h.pt0 + l];
          else
            v[c] = sv[c][l - h.nint];
        }
        for (int k = T.seg_off[h.seg0 + sg]; k < T.seg_off[h.seg0 + sg + 1]; k++) {
          const float nv[2] = {T.bnormal[2 * k], T.bnormal[2 * k + 1]};
          const float w = T.bweight[k], rvp = T.brvp[k], rvs = T.brvs[k];
          const float vn = fmaf(v[1], nv[1], v[0] * nv[0]);
          const float nn = fmaf(nv[0], nv[0], nv[1] * nv[1]);
          const float j1 = sqrtf(nn);
#pragma unroll
          for (int d = 0; d < 2; d++) {
            const float fac = fmaf(rvs, v[d], (vn * nv[d] / (j1 * j1)) * (rvp - rvs));
            s[d] += -1.0f * fac * j1 * w;
          }
        }
      }
      fx[sg] = make_float2(s[0], s[1]);
    }
    for (int k = t / 25; k < h.nsrc && t < NT / 25 * 25; k += NT / 25) {
      const int p = t % 25;
      float o[2] = {0.0f, 0.0f};
      if (fi == 1) {
        const int4 s4 = T.src_el[h.src0 + k];
        for (int i = s4.y; i < s4.z; i++) {
          const int id = T.src_id[i];
          const float amp = T.stf[L.step * T.stf_step + id * T.stf_src];
#pragma unroll
          for (int c = 0; c < 2; c++) o[c] += amp * T.src_array[(static_cast<size_t>(id) * 2 + c) * 25 + p];
        }
      }
      fx[h.nseg + k * 25 + p] = make_float2(o[0], o[1]);
    }
    if (fi == 0) {
      // adjoint sources join their element's force
      const int2 as = P.adj_head[patch];
      for (int k = as.x + t / 25; k < as.y && t < NT / 25 * 25; k += NT / 25) {
        const int p = t % 25;
        const int4 s4 = P.adj_el[k];
        float o[2] = {0.0f, 0.0f};
        for (int i = s4.y; i < s4.z; i++) {
          const int id = P.adj_id[i];
          const float amp = P.adj_stf[L.step * P.adj_step + id];
#pragma unroll
          for (int c = 0; c < 2; c++) o[c] += amp * P.adj_array[(static_cast<size_t>(id) * 2 + c) * 25 + p];
        }
        const float2 x = f2[s4.x * 25 + p];
        f2[s4.x * 25 + p] = make_float2(o[0] + x.x, o[1] + x.y);
      }
    }
    __syncthreads();
    {
      float2 *out = S.rb[L.rd ^ 1];
      for (int k = t; k < h.nbent; k += NT) out[T.bslot[h.be0 + k]] = f2[tab[h.bent + k]];
    }
    const bool snapshot = fi && h.rm0 >= 0 && L.step % h.nsb == 0;
#pragma unroll
    for (int k = 0; k < NI; k++) {
      const int l = t + k * NT;
      if (l >= h.nint) continue;
      const float2 s = interior_force(h, tab, se, l, ea[k], eb[k]);
      const float a0 = s.x * mi[k][0], a1 = s.y * mi[k][1];
      float x0 = su[0][l], x1 = su[1][l], v0 = vi[k][0], v1 = vi[k][1], w0, w1;
      if (fi == 0) {
        aa[k][0] = a0;
        aa[k][1] = a1;
      } else {
        put(P.R + h.pt0, l, ri[k] + h.dt * fmaf(aa[k][1], x1, aa[k][0] * x0));
      }
      newmark(a0, x0, v0, w0);
      newmark(a1, x1, v1, w1);
      put(u0p, l, x0);
      put(u1p, l, x1);
      put(v0p, l, v0);
      put(v1p, l, v1);
      if (snapshot) {
        const int rowi = T.rmap[h.rm0 + l];
        if (rowi >= 0) {
          float *o = T.snap + 6 * (static_cast<size_t>(L.rd ^ 1) * T.nrow + rowi);
          o[0] = su[0][l];
          o[1] = su[1][l];
          o[2] = w0;
          o[3] = w1;
          o[4] = a0;
          o[5] = a1;
        }
      }
    }
    __syncthreads();
  }
}

// The boundary points of both fields after the last of a run of such steps.
__global__ __launch_bounds__(256) void patch_pair_boundary_kernel(PatchTables T, PatchState A, PatchState B,
                                                                  NewmarkConst nc, int rd, float *__restrict__ R) {
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= T.nbnd) return;
  const int k0 = T.boff[b], n = T.boff[b + 1] - k0;
  float aa[2];
#pragma unroll
  for (int fi = 0; fi < 2; fi++) {
    const PatchState &S = fi ? B : A;
    const Newmark<false> nm{fi ? -nc.dt : nc.dt, fi ? -nc.dto2 : nc.dto2, nc.dt2o2};
    float s[2], rho = 0.0f;
    boundary_force(S.rb[rd], k0, n, s);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const size_t o = c * static_cast<size_t>(T.np) + T.nint + b;
      const float a = s[c] * T.minv[o];
      float u = rd ? S.ub[c * static_cast<size_t>(T.nbnd) + b] : S.u[o];
      float v = rd ? S.ub[(2 + c) * static_cast<size_t>(T.nbnd) + b] : S.v[o], v1;
      if (fi)
        rho = fmaf(aa[c], u, rho);
      else
        aa[c] = a;
      nm(a, u, v, v1);
      S.u[o] = u;
      S.v[o] = v;
    }
    if (fi) R[T.nint + b] += nc.dt * rho;
  }
}

// One thread per boundary point: see launch_patch_boundary.
template <bool EXACT>
__global__ __launch_bounds__(256) void patch_boundary_kernel(PatchTables T, PatchState S, Newmark<EXACT> nm, int rd,
                                                             int advance, int store_a, int add_a) {
#pragma clang fp contract(off)
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= T.nbnd) return;
  float s[2];
  const int k0 = T.boff[b];
  const float *const stored = S.a + T.nint + b;
  boundary_force(S.rb[rd], k0, T.boff[b + 1] - k0, s, add_a ? stored[0] : 0.0f, add_a ? stored[T.np] : 0.0f);
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const size_t o = c * static_cast<size_t>(T.np) + T.nint + b;
    const float a = s[c] * T.minv[o];
    if (advance) {
      float u = rd ? S.ub[c * static_cast<size_t>(T.nbnd) + b] : S.u[o];
      float v = rd ? S.ub[(2 + c) * static_cast<size_t>(T.nbnd) + b] : S.v[o], v1;
      nm(a, u, v, v1);
      S.u[o] = u;
      S.v[o] = v;
    }
    if (!advance || store_a) S.a[o] = a;
  }
}

__global__ __launch_bounds__(256) void take_kernel(int n, const int *__restrict__ index,
                                                   const float *__restrict__ src, float *__restrict__ dst) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[index[i]];
}
__global__ __launch_bounds__(256) void put_kernel(int n, const int *__restrict__ index,
                                                  const float *__restrict__ src, float *__restrict__ dst) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[index[i]] = src[i];
}

template <int PE, int GEOM, bool EPROP>
void launch_step(hipStream_t s, int npatch, int nrec, bool exact, const PatchTables &t, const PatchState &st, const GllConst &q,
                 const PatchLaunch &l) {
  constexpr int NT = patch_threads<PE>();
  const dim3 grid(npatch + (nrec + NT / 64 - 1) / (NT / 64)), block(NT);
  if (exact)
    hipLaunchKernelGGL((patch_step_kernel<PE, GEOM, EPROP, true, false>), grid, block, 0, s, npatch, nrec, t, st, q, l);
  else if (l.rec)
    hipLaunchKernelGGL((patch_step_kernel<PE, GEOM, EPROP, false, true>), grid, block, 0, s, npatch, nrec, t, st, q, l);
  else
    hipLaunchKernelGGL((patch_step_kernel<PE, GEOM, EPROP, false, false>), grid, block, 0, s, npatch, nrec, t, st, q, l);
}

template <int PE, int GEOM>
void launch_step_prop(hipStream_t s, int npatch, int nrec, bool exact, const PatchTables &t, const PatchState &st,
                      const GllConst &q, const PatchLaunch &l) {
  if (t.kmu)
    launch_step<PE, GEOM, true>(s, npatch, nrec, exact, t, st, q, l);
  else
    launch_step<PE, GEOM, false>(s, npatch, nrec, exact, t, st, q, l);
}

template <int PE>
void launch_step_geom(hipStream_t s, int npatch, int nrec, bool exact, const PatchTables &t, const PatchState &st,
                      const GllConst &q, const PatchLaunch &l) {
  switch (t.geom.mode) {
    case GEOM2D_RECORD: return launch_step_prop<PE, GEOM2D_RECORD>(s, npatch, nrec, exact, t, st, q, l);
    case GEOM2D_CTRL4: return launch_step_prop<PE, GEOM2D_CTRL4>(s, npatch, nrec, exact, t, st, q, l);
    case GEOM2D_CTRL9: return launch_step_prop<PE, GEOM2D_CTRL9>(s, npatch, nrec, exact, t, st, q, l);
    case GEOM2D_POINT: return launch_step_prop<PE, GEOM2D_POINT>(s, npatch, nrec, exact, t, st, q, l);
    default: throw std::invalid_argument("patch step: unknown geometry form");
  }
}

template <int PE, int GEOM>
void launch_pair_prop(hipStream_t s, int npatch, int nrec, const PatchTables &t, const PatchState &a,
                      const PatchState &b, const GllConst &q, const PatchPairLaunch &l, const PatchPairTables &p) {
  constexpr int NT = patch_threads<PE>();
  const dim3 grid(npatch + (nrec + NT / 64 - 1) / (NT / 64)), block(NT);
  if (t.kmu)
    hipLaunchKernelGGL((patch_pair_kernel<PE, GEOM, true>), grid, block, 0, s, npatch, nrec, t, a, b, q, l, p);
  else
    hipLaunchKernelGGL((patch_pair_kernel<PE, GEOM, false>), grid, block, 0, s, npatch, nrec, t, a, b, q, l, p);
}
template <int PE>
void launch_pair_geom(hipStream_t s, int npatch, int nrec, const PatchTables &t, const PatchState &a,
                      const PatchState &b, const GllConst &q, const PatchPairLaunch &l, const PatchPairTables &p) {
  switch (t.geom.mode) {
    case GEOM2D_RECORD: return launch_pair_prop<PE, GEOM2D_RECORD>(s, npatch, nrec, t, a, b, q, l, p);
    case GEOM2D_CTRL4: return launch_pair_prop<PE, GEOM2D_CTRL4>(s, npatch, nrec, t, a, b, q, l, p);
    case GEOM2D_CTRL9: return launch_pair_prop<PE, GEOM2D_CTRL9>(s, npatch, nrec, t, a, b, q, l, p);
    case GEOM2D_POINT: return launch_pair_prop<PE, GEOM2D_POINT>(s, npatch, nrec, t, a, b, q, l, p);
    default: throw std::invalid_argument("patch pair: unknown geometry form");
  }
}

}  // namespace

void launch_patch_step(hipStream_t s, int pe, int npatch, int nrec, bool exact, const PatchTables &t,
                       const PatchState &st, const GllConst &q, const PatchLaunch &l) {
  if (!l.pending || t.ntypes <= 0) nrec = 0;
  if (npatch + nrec <= 0) return;
  if (pe == PATCH_LARGE)
    launch_step_geom<PATCH_LARGE>(s, npatch, nrec, exact, t, st, q, l);
  else
    launch_step_geom<PATCH_SMALL>(s, npatch, nrec, exact, t, st, q, l);
}

void launch_patch_boundary(hipStream_t s, bool exact, const PatchTables &t, const PatchState &st, NewmarkConst nc,
                           int rd, int advance, int store_a, int add_a) {
  if (t.nbnd <= 0) return;
  const dim3 grid((t.nbnd + 255) / 256);
  if (exact)
    hipLaunchKernelGGL(patch_boundary_kernel<true>, grid, dim3(256), 0, s, t, st,
                       (Newmark<true>{nc.dt, nc.dto2, nc.dt2o2}), rd, advance, store_a, add_a);
  else
    hipLaunchKernelGGL(patch_boundary_kernel<false>, grid, dim3(256), 0, s, t, st,
                       (Newmark<false>{nc.dt, nc.dto2, nc.dt2o2}), rd, advance, store_a, add_a);
}

void launch_patch_pair(hipStream_t s, int pe, int npatch, int nrec, const PatchTables &t, const PatchState &adj,
                       const PatchState &bwd, const GllConst &q, const PatchPairLaunch &l, const PatchPairTables &p) {
  if (!l.pending || t.ntypes <= 0) nrec = 0;
  if (npatch + nrec <= 0) return;
  if (pe == PATCH_LARGE)
    launch_pair_geom<PATCH_LARGE>(s, npatch, nrec, t, adj, bwd, q, l, p);
  else
    launch_pair_geom<PATCH_SMALL>(s, npatch, nrec, t, adj, bwd, q, l, p);
}

void launch_patch_pair_boundary(hipStream_t s, const PatchTables &t, const PatchState &adj, const PatchState &bwd,
                                NewmarkConst nc, int rd, float *R) {
  if (t.nbnd > 0)
    hipLaunchKernelGGL(patch_pair_boundary_kernel, dim3((t.nbnd + 255) / 256), dim3(256), 0, s, t, adj, bwd, nc, rd, R);
}

void launch_take(hipStream_t s, int n, const int *index, const float *src, float *dst) {
  if (n > 0) hipLaunchKernelGGL(take_kernel, dim3((n + 255) / 256), dim3(256), 0, s, n, index, src, dst);
}
void launch_put(hipStream_t s, int n, const int *index, const float *src, float *dst) {
  if (n > 0) hipLaunchKernelGGL(put_kernel, dim3((n + 255) / 256), dim3(256), 0, s, n, index, src, dst);
}

}  // namespace sfx
