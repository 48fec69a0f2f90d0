// LES layer of the 2nd-order channel step: the eddy viscosity of the WALE and
// MTS models (src/CFD_2nd/m_LESModels.f90) and the partially implicit LES
// scheme that uses it (the *_PIMP_LES routines of m_TSchemePIMP_inc.f90):
// right-hand sides with the variable-viscosity stress divergence, y-implicit
// Crank-Nicolson solves whose coefficients vary along every line, and the
// pressure update with the eddy viscosity.
//
// Layout as everywhere in the library: element (i, jj, k) at
// i + nx (jj + (ny+3) k); x and z wrap by index, the wall ghost planes
// jj = 0 and jj = ny+1 are stored.  nut is such a field.  Expressions keep
// the reference's operation order (compiled without contraction), so the
// fields agree with a strict-IEEE build of the reference to rounding of the
// library power function in WALE only.
#include "c3d_internal.h"

#include <type_traits>

namespace c3d {

namespace {

constexpr int LBX = 64, LBY = 4, LKCH = 8;

__device__ __forceinline__ int wm(int i, int n) { return i == 0 ? n - 1 : i - 1; }
__device__ __forceinline__ int wp(int i, int n) { return i == n - 1 ? 0 : i + 1; }

// 1-D grid of 64 x 4 (i, j) tiles times runs of LKCH z planes
#define LES_CELL()                                                            \
  const int cgx_ = (g.nx + LBX - 1) / LBX, cgy_ = (g.ny + LBY - 1) / LBY;     \
  const int lb_ = xcd_remap(blockIdx.x, gridDim.x);                           \
  const int i = (lb_ % cgx_) * LBX + threadIdx.x;                             \
  const int jc = ((lb_ / cgx_) % cgy_) * LBY + threadIdx.y + 1;               \
  const int kz0 = (lb_ / (cgx_ * cgy_)) * LKCH;                               \
  const int kz1 = min(g.nz, kz0 + LKCH)

// f(a, b, c) of a field at x index a, stored y row b, z index c; the caller
// names nx and nyh
#define A(f, a, b, c) \
  f[(long long)(a) + (long long)nx * ((long long)(b) + (long long)nyh * (long long)(c))]

inline int les_blocks(const Geom& g) {
  return ((g.nx + LBX - 1) / LBX) * ((g.ny + LBY - 1) / LBY) * ((g.nz + LKCH - 1) / LKCH);
}

}  // namespace

template <typename T>
struct LesCoef {
  T rdx, rdz, rdx2, rdz2, xnu, twoxnu;
  T pmGamma, pmTheta, pmAlpha, pmBetaT, gx, gy, gz;
  T fc[9];    // test-filter weights, fc[4] already minus one
  int bcym, bcyp;
};

template <typename T>
static LesCoef<T> make_les_coef(const c3d_ctx* c) {
  LesCoef<T> q;
  q.rdx = (T)c->rdx; q.rdz = (T)c->rdz; q.rdx2 = (T)c->rdx2; q.rdz2 = (T)c->rdz2;
  q.xnu = (T)c->p.xnu;
  q.twoxnu = (T)(2.0 * c->p.xnu);
  q.pmGamma = (T)c->pmGamma; q.pmTheta = (T)c->pmTheta; q.pmAlpha = (T)c->pmAlpha;
  q.pmBetaT = (T)c->pmBetaT;
  q.gx = (T)c->p.gravity[0]; q.gy = (T)c->p.gravity[1]; q.gz = (T)c->p.gravity[2];
  for (int s = 0; s < 9; ++s) q.fc[s] = (T)c->les_fcoe[s];
  q.fc[4] = (T)(c->les_fcoe[4] - 1.0);
  q.bcym = c->p.bc[2];
  q.bcyp = c->p.bc[3];
  return q;
}

template <typename T>
static const LesMet<T>& lesmet(const c3d_ctx* c);
template <>
const LesMet<double>& lesmet<double>(const c3d_ctx* c) { return c->lmd; }
template <>
const LesMet<float>& lesmet<float>(const c3d_ctx* c) { return c->lmf; }
template <typename T>
static const Metrics<T>& met(const c3d_ctx* c);
template <>
const Metrics<double>& met<double>(const c3d_ctx* c) { return c->md; }
template <>
const Metrics<float>& met<float>(const c3d_ctx* c) { return c->mf; }

// the ghost rows of SetBC_and_UpdateHalo_SGS (m_LESModels.f90:375-428),
// written by the threads of the first and last interior rows
template <typename T>
__device__ __forceinline__ void nut_ghosts(const Geom& g, const LesCoef<T>& q, T* nut, int i,
                                           int jc, int k, T v) {
  if (jc == 1) nut[fidx(g, i, 0, k)] = q.bcym == C3D_BC_NOSLIP ? q.twoxnu - v : v;
  if (jc == g.ny) nut[fidx(g, i, g.ny + 1, k)] = q.bcyp == C3D_BC_NOSLIP ? q.twoxnu - v : v;
}

// ---------------------------------------------------------------------------
// Clc_SGS_WALE (m_LESModels.f90:72-135); Clc_SGS_MTS (:145-258) with
// ClcVelStrainRate (:328-370).
//
// A workgroup owns 64 x 4 cells and marches a run of z planes.  Each plane of
// u, v, w over the tile plus its halo (one cell, two above in x for the test
// filter) passes once through LDS, two buffers in turn, requested a plane ahead;
// the values at the planes a cell still needs stay in registers, so a plane
// costs 19 LDS reads a thread.  The uz plane staged is one further up for MTS
// (LZ = 2), whose residual on the face k+1 reaches k+2; that residual is the next
// cell's at k, and the one quantity kept.  The squared residuals the reference
// stores in Ktemp are formed by each cell for its other faces (same operands,
// same operations).  Bound: FP64 arithmetic, some 280 vector instructions a cell
// (vector units active 67 % of the time), beside 4 words per cell of HBM.
// With every operand fetched on its own (MTS: over 90 loads a cell, both
// residuals of each component from memory) MTS took 0.724 ms at 384x192x288,
// WALE 0.026 ms at 96x96x72; now 0.284 (2.4 TB/s) and 0.018 ms.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T filt_res(const T* F, const T* a, const T* b, const T* c) {
  return F[0] * a[0] + F[1] * a[1] + F[2] * a[2] + F[3] * b[0] + F[4] * b[1] + F[5] * b[2] +
         F[6] * c[0] + F[7] * c[1] + F[8] * c[2];
}

template <typename T, bool MTS>
__global__ __launch_bounds__(LBX* LBY, 2) void k_sgs(Geom g, Metrics<T> m, LesMet<T> lm,
                                                     LesCoef<T> q, const T* __restrict__ ux,
                                                     const T* __restrict__ uy,
                                                     const T* __restrict__ uz,
                                                     T* __restrict__ nut, int kchunk) {
  constexpr int LZ = MTS ? 2 : 1;
  constexpr int LW = LBX + (MTS ? 3 : 2), LP = LW * (LBY + 2);
  constexpr int NT = LBX * LBY, NS = (LP + NT - 1) / NT;
  __shared__ T sb[2][3][LP];
  const int tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int tid = tx + LBX * ty;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int gxb = (nx + LBX - 1) / LBX, gyb = (ny + LBY - 1) / LBY;
  const int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int i0 = (lb % gxb) * LBX, j0 = ((lb / gxb) % gyb) * LBY + 1;
  const int k0 = (lb / (gxb * gyb)) * kchunk, k1 = min(nz, k0 + kchunk);
  // staging slots as in the right-hand sides below
  unsigned so[NS];
  bool sl[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int e = tid + NT * s;
    const int jj = e / LW, ii = e - jj * LW;
    int i = i0 - 1 + ii;
    i = i < 0 ? nx - 1 : (i >= nx ? i % nx : i);
    sl[s] = e < LP;
    so[s] = sl[s] ? (unsigned)(min(j0 - 1 + jj, ny + 1) * nx + i) * (unsigned)sizeof(T) : 0u;
  }
  T st[3][NS];
  // ux, uy of plane k+1 and uz of plane k+LZ, periodic
  auto fetch = [&](int k) {
    const int ka = (k + 1 + 2 * nz) % nz, kb = (k + LZ + 2 * nz) % nz;
    const T* const f[3] = {ux + g.plane * ka, uy + g.plane * ka, uz + g.plane * kb};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int s = 0; s < NS; ++s) st[a][s] = *(const T*)((const char*)f[a] + so[s]);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (sl[s]) {
#pragma unroll
        for (int a = 0; a < 3; ++a) sb[buf][a][tid + NT * s] = st[a][s];
      }
  };
  const int jc = j0 + ty, jrow = min(jc, ny), jp = jrow + 1;
  const int e = (ty + 1) * LW + tx + 1;
  const int i = i0 + tx;
  const bool live = i < nx && jc <= ny;
  const T caj = m.rdyp[jrow];
  const T cac1 = m.rdyc[jrow];
  const T cac2 = m.rdyc[jp];
  const T cac12 = cac1 - cac2;
  const T rdx = q.rdx, rdz = q.rdz, oneEighth = T(0.125);
  const T rdelta = MTS ? lm.rdelta[jrow] : T(0);
  T CwDelta2 = MTS ? T(0) : T(0.325) * lm.delta[jrow];
  CwDelta2 = CwDelta2 * CwDelta2;
  // [plane][x]: x = i-1, i, i+1, i+2.  ux and uy: planes k-1, k, k+1; ux on the
  // rows beside: k, k+1; uz: k, k+1, k+LZ
  T u[3][4], um[2][2], up[2][2], v[3][3], vp[3][3], w[LZ + 1][3], wm[LZ + 1], wp_[LZ + 1];
  auto take = [&](int buf) {  // shift by a plane and append the staged one
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int x = 0; x < 4; ++x) u[p][x] = u[p + 1][x];
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        v[p][x] = v[p + 1][x];
        vp[p][x] = vp[p + 1][x];
      }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      um[0][x] = um[1][x];
      up[0][x] = up[1][x];
    }
#pragma unroll
    for (int p = 0; p < LZ; ++p) {
#pragma unroll
      for (int x = 0; x < 3; ++x) w[p][x] = w[p + 1][x];
      wm[p] = wm[p + 1];
      wp_[p] = wp_[p + 1];
    }
    const T* U = sb[buf][0] + e;
    const T* V = sb[buf][1] + e;
    const T* W = sb[buf][2] + e;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      u[2][x] = U[x - 1];
      v[2][x] = V[x - 1];
      vp[2][x] = V[LW + x - 1];
      w[LZ][x] = W[x - 1];
    }
    if (MTS) u[2][3] = U[2];
    um[1][0] = U[-LW]; um[1][1] = U[1 - LW];
    up[1][0] = U[LW]; up[1][1] = U[1 + LW];
    wm[LZ] = W[-LW];
    wp_[LZ] = W[LW];
  };
  // the planes below the run
  for (int k = k0 - LZ - 1; k < k0; ++k) {
    fetch(k);
    stage(k & 1);
    __syncthreads();
    take(k & 1);
  }
  T rz0 = T(0);
  if (MTS) rz0 = filt_res(q.fc, w[0], w[1], w[LZ]);
  fetch(k0);
  stage(k0 & 1);
  __syncthreads();
  for (int k = k0; k < k1; ++k) {
    fetch(k + 1);
    take(k & 1);
    const T dudx = (u[1][2] - u[1][1]) * rdx;
    const T dvdy = (vp[1][1] - v[1][1]) * caj;
    const T dwdz = (w[1][1] - w[0][1]) * rdz;
    T nv;
    if (MTS) {
      const T st4 = oneEighth * ((vp[1][2] - vp[1][0] + v[1][2] - v[1][0]) * rdx +
                                 (up[0][1] + up[0][0]) * cac2 + (u[1][2] + u[1][1]) * cac12 -
                                 (um[0][1] + um[0][0]) * cac1);
      const T st5 = oneEighth * ((u[2][2] + u[2][1] - u[0][2] - u[0][1]) * rdz +
                                 (w[1][2] - w[1][0] + w[0][2] - w[0][0]) * rdx);
      const T st6 = oneEighth * ((vp[2][1] + v[2][1] - vp[0][1] - v[0][1]) * rdz +
                                 (wp_[1] + wp_[0]) * cac2 + (w[1][1] + w[0][1]) * cac12 -
                                 (wm[1] + wm[0]) * cac1);
      const T strain = sqrt(T(2) * (dudx * dudx + dvdy * dvdy + dwdz * dwdz) +
                            T(4) * (st4 * st4 + st5 * st5 + st6 * st6));
      // Kes: ux residual on the faces i and i+1, uy on the nodes jc and jc+1,
      // uz on the faces k and k+1 (:159-230)
      const T* F = q.fc;
      const T rx0 = filt_res(F, u[0], u[1], u[2]);
      const T rx1 = filt_res(F, u[0] + 1, u[1] + 1, u[2] + 1);
      T Kes = T(0.5) * (rx0 * rx0 + rx1 * rx1);
      const T ry0 = filt_res(F, v[0], v[1], v[2]), ry1 = filt_res(F, vp[0], vp[1], vp[2]);
      Kes = Kes + T(0.5) * (ry0 * ry0 + ry1 * ry1);
      const T rz1 = filt_res(F, w[0], w[1], w[LZ]);
      Kes = Kes + T(0.5) * (rz0 * rz0 + rz1 * rz1);
      rz0 = rz1;
      T Ts = sqrt(Kes) * rdelta + strain / T(10);
      if (Ts < T(1.00E-10))
        Ts = T(0);
      else
        Ts = T(1) / Ts;
      nv = T(0.05) * Kes * Ts + q.xnu;
    } else {
      const T dudy = ((up[0][1] + up[0][0]) * cac2 + (u[1][2] + u[1][1]) * cac12 -
                      (um[0][1] + um[0][0]) * cac1) * T(0.25);
      const T dudz = (u[2][2] + u[2][1] - u[0][2] - u[0][1]) * rdz * T(0.25);
      const T dvdx = (vp[1][2] - vp[1][0] + v[1][2] - v[1][0]) * rdx * T(0.25);
      const T dvdz = (vp[2][1] + v[2][1] - vp[0][1] - v[0][1]) * rdz * T(0.25);
      const T dwdx = (w[1][2] - w[1][0] + w[0][2] - w[0][0]) * rdx * T(0.25);
      const T dwdy = ((wp_[1] + wp_[0]) * cac2 + (w[1][1] + w[0][1]) * cac12 -
                      (wm[1] + wm[0]) * cac1) * T(0.25);
      const T S11 = dudx;
      const T S12 = (dudy + dvdx) * T(0.5);
      const T S13 = (dudz + dwdx) * T(0.5);
      const T S22 = dvdy;
      const T S23 = (dvdz + dwdy) * T(0.5);
      const T S33 = dwdz;
      const T SijSij = S11 * S11 + S22 * S22 + S33 * S33 + T(2) * (S12 * S12 + S13 * S13 + S23 * S23);
  
      T Sd11 = dudx * dudx + dudy * dvdx + dudz * dwdx;
      const T Sd12 = (dudx * dudy + dudy * dvdy + dudz * dwdy + dvdx * dudx + dvdy * dvdx + dvdz * dwdx) * T(0.5);
      const T Sd13 = (dudx * dudz + dudy * dvdz + dudz * dwdz + dwdx * dudx + dwdy * dvdx + dwdz * dwdx) * T(0.5);
      T Sd22 = dvdx * dudy + dvdy * dvdy + dvdz * dwdy;
      const T Sd23 = (dvdx * dudz + dvdy * dvdz + dvdz * dwdz + dwdx * dudy + dwdy * dvdy + dwdz * dwdy) * T(0.5);
      T Sd33 = dwdx * dudz + dwdy * dvdz + dwdz * dwdz;
      const T SdTrace = (Sd11 + Sd22 + Sd33) / T(3);
      Sd11 = Sd11 - SdTrace;
      Sd22 = Sd22 - SdTrace;
      Sd33 = Sd33 - SdTrace;
      const T SdijSdij =
          Sd11 * Sd11 + Sd22 * Sd22 + Sd33 * Sd33 + T(2) * (Sd12 * Sd12 + Sd13 * Sd13 + Sd23 * Sd23);
      // the reference's powers (**1.5, **2.5, **1.25) of these non-negative
      // sums through square roots: x^1.5 = x sqrt(x), x^2.5 = x^2 sqrt(x),
      // x^1.25 = x sqrt(sqrt(x)), a few ulp from pow at a fraction of its cost
      const T sdh = sqrt(SdijSdij), sh = sqrt(SijSij);
      nv = CwDelta2 * (SdijSdij * sdh) /
               (SijSij * SijSij * sh + SdijSdij * sqrt(sdh)) + q.xnu;
    }
    stage((k + 1) & 1);
    if (live) {
      nut[fidx(g, i, jc, k)] = nv;
      nut_ghosts(g, q, nut, i, jc, k, nv);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// clcRhsX_PIMP_LES (m_TSchemePIMP_inc.f90:80-156), clcRhsY_PIMP_LES
// (:214-272), clcRhsZ_PIMP_LES (:330-387).  MASK bit 0/1/2 selects x/y/z;
// the x component writes the per-block partial of the bulk integral.
//
// The form of the full-implicit right-hand sides: a workgroup owns a tile of
// 64 x 4 cells and marches a run of z planes; each plane of u, v, w, p, nut
// over the tile plus a one-cell halo is loaded once into LDS (three rotating
// plane buffers, plane k+2 in flight in registers while plane k is computed,
// one barrier per plane), neighbours are LDS reads, values at k-1 roll through
// registers, histories are requested before the prefetch and results stored
// after the staging.  Bound: HBM, 14 words per cell.  Fetching each operand on
// its own, over 150 loads per cell with an address computed for each, took
// 0.886 ms at 384x192x288 and 0.032 ms at 96x96x72 (FP64); this takes 0.495 ms
// (4.8 TB/s) and 0.025 ms.  With the rows of a wavefront in registers, x
// neighbours by DPP and the neighbour rows from the caches instead of LDS it
// took 0.608 ms: those rows, 9 of 26 loads, mostly came from L2.
// ---------------------------------------------------------------------------
template <typename T, int MASK, bool NTS>
__global__ __launch_bounds__(LBX* LBY, 2) void k_rhs_les(Geom g, Metrics<T> m, LesCoef<T> q,
                                                         const T* __restrict__ ux,
                                                         const T* __restrict__ uy,
                                                         const T* __restrict__ uz,
                                                         const T* __restrict__ pr,
                                                         const T* __restrict__ nut,
                                                         T* __restrict__ rx, T* __restrict__ ry,
                                                         T* __restrict__ rz, T* __restrict__ hx,
                                                         T* __restrict__ hy, T* __restrict__ hz,
                                                         double* __restrict__ partials,
                                                         DevScalars* sc, int kchunk) {
  constexpr int LW = LBX + 2, LP = LW * (LBY + 2);             // one field's tile plane
  constexpr int NT = LBX * LBY, NS = (LP + NT - 1) / NT;       // staging slots per thread
  __shared__ T sb[3][5][LP];
  __shared__ long long shf[LBY][4];
  const int tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int tid = tx + LBX * ty;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int gxb = (nx + LBX - 1) / LBX, gyb = (ny + LBY - 1) / LBY;
  const int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int i0 = (lb % gxb) * LBX, j0 = ((lb / gxb) % gyb) * LBY + 1;
  const int k0 = (lb / (gxb * gyb)) * kchunk, k1 = min(nz, k0 + kchunk);
  // staging slot s: tile element e = tid + NT s at halo row e / LW, column
  // e % LW (periodic); rows past the top ghost repeat it and are never read
  unsigned so[NS];
  bool sl[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int e = tid + NT * s;
    const int jj = e / LW, ii = e - jj * LW;
    int i = i0 - 1 + ii;
    i = i < 0 ? nx - 1 : (i >= nx ? i % nx : i);
    sl[s] = e < LP;
    so[s] = sl[s] ? (unsigned)(min(j0 - 1 + jj, ny + 1) * nx + i) * (unsigned)sizeof(T) : 0u;
  }
  const T* const fld[5] = {ux, uy, uz, pr, nut};
  T st[5][NS];
  auto fetch = [&](int k) {
#pragma unroll
    for (int f = 0; f < 5; ++f)
#pragma unroll
      for (int s = 0; s < NS; ++s)
        st[f][s] = *(const T*)((const char*)(fld[f] + g.plane * k) + so[s]);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (sl[s]) {
#pragma unroll
        for (int f = 0; f < 5; ++f) sb[buf][f][tid + NT * s] = st[f][s];
      }
  };
  const int jc = j0 + ty, jrow = min(jc, ny);
  const int e = (ty + 1) * LW + tx + 1;
  const bool live = i0 + tx < nx && jc <= ny;
  const T rdx = q.rdx, rdz = q.rdz;
  const T qdx1 = T(0.25) * rdx, qdx3 = T(0.25) * rdz;
  const T rdyp = m.rdyp[jrow], sucaj = T(0.25) * m.rdyp[jrow];
  const T sucac = m.rdyc[jrow], qsucac = T(0.25) * sucac;
  const T ap2c = m.ap2c[jrow], am2c = m.am2c[jrow], ap2p = m.ap2p[jrow], am2p = m.am2p[jrow];
  const T am1c = q.rdx2, ap1c = q.rdx2, am3c = q.rdz2, ap3c = q.rdz2;
  const T s1coe = m.s1coe[jrow];
  const T twoBT = T(2) * q.pmBetaT;
  long long s1[4] = {0, 0, 0, 0};
  // values at k-1, rolled
  T u[3], v[3], w[3], t[3], tm[3], t_xm[3], t_xp[3], vp[2], tp[2], p[2], u_xp;
  fetch(k0 == 0 ? nz - 1 : k0 - 1);
  stage(0);
  fetch(k0);
  stage(1);
  fetch(wp(k0, nz));
  stage(2);
  __syncthreads();
  u[1] = sb[0][0][e]; v[1] = sb[0][1][e]; w[1] = sb[0][2][e]; p[1] = sb[0][3][e];
  t[1] = sb[0][4][e]; t_xm[1] = sb[0][4][e - 1]; t_xp[1] = sb[0][4][e + 1];
  tm[1] = sb[0][4][e - LW]; tp[1] = sb[0][4][e + LW];
  vp[1] = sb[0][1][e + LW]; u_xp = sb[0][0][e + 1];
  __syncthreads();
  int bm = 0, bc = 1, bp = 2;
  const unsigned oi = (unsigned)(jrow * nx + min(i0 + tx, nx - 1)) * (unsigned)sizeof(T);
  for (int k = k0; k < k1; ++k) {
    auto at = [&](const T* f) { return (const char*)(f + g.plane * k) + oi; };
    T hxo, hyo, hzo;
    if (MASK & 1) hxo = C3D_LD_ONCE((const T*)at(hx));
    if (MASK & 2) hyo = C3D_LD_ONCE((const T*)at(hy));
    if (MASK & 4) hzo = C3D_LD_ONCE((const T*)at(hz));
    const int k2 = min(k + 2, k1);
    fetch(k2 >= nz ? k2 - nz : k2);
    const T* U = sb[bc][0] + e; const T* V = sb[bc][1] + e; const T* W = sb[bc][2] + e;
    const T* P = sb[bc][3] + e; const T* N = sb[bc][4] + e;
    const T* W1 = sb[bp][2] + e; const T* N1 = sb[bp][4] + e;
    const T ukm_xp = u_xp;
    u[0] = u[1]; v[0] = v[1]; w[0] = w[1]; t[0] = t[1]; tm[0] = tm[1];
    t_xm[0] = t_xm[1]; t_xp[0] = t_xp[1]; vp[0] = vp[1]; tp[0] = tp[1]; p[0] = p[1];
    u[1] = U[0]; v[1] = V[0]; w[1] = W[0]; p[1] = P[0]; t[1] = N[0];
    u[2] = sb[bp][0][e]; v[2] = sb[bp][1][e]; w[2] = W1[0]; t[2] = N1[0];
    tm[1] = N[-LW]; tm[2] = N1[-LW]; tp[1] = N[LW];
    t_xm[1] = N[-1]; t_xp[1] = N[1]; t_xm[2] = N1[-1];
    vp[1] = V[LW];
    u_xp = U[1];
    const T u_xm = U[-1], u_yp = U[LW], u_ym = U[-LW], um_xp = U[1 - LW];
    const T v_xm = V[-1], v_xp = V[1], v_ym = V[-LW], vp_xm = V[LW - 1];
    const T w_xm = W[-1], w_xp = W[1], w_yp = W[LW], w1_xm = W1[-1];
    const T wm[2] = {W[-LW], W1[-LW]};
    const T tm_xm = N[-LW - 1], tm_xp = N[-LW + 1], tp_xm = N[LW - 1];
    const T p_xm = P[-1], p_ym = P[-LW];
    T ox, oy, oz, cx, cy, cz;
    if (MASK & 1) {
      const T h11 = ((u_xp + u[1]) * (u_xp + u[1]) -
                     (u[1] + u_xm) * (u[1] + u_xm)) * qdx1;
      const T h12 = ((vp[1] + vp_xm) * (u_yp + u[1]) -
                     (v[1] + v_xm) * (u[1] + u_ym)) * sucaj;
      const T h13 = ((w[2] + w1_xm) * (u[2] + u[1]) -
                     (w[1] + w_xm) * (u[1] + u[0])) * qdx3;
      const T visa = T(0.25) * (t[1] + t_xm[1] + tm[1] + tm_xm);
      const T visb = T(0.25) * (t[1] + t_xm[1] + tp[1] + tp_xm);
      const T visc = T(0.25) * (t[1] + t_xm[1] + t[0] + t_xm[0]);
      const T visd = T(0.25) * (t[1] + t_xm[1] + t[2] + t_xm[2]);
      const T sgs1 = q.rdx2 * (t[1] * (u_xp - u[1]) -
                               t_xm[1] * (u[1] - u_xm));
      const T sgs2 = rdx * rdyp *
                     (visb * (vp[1] - vp_xm) - visa * (v[1] - v_xm));
      const T sgs3 = rdx * rdz *
                     (visd * (w[2] - w1_xm) - visc * (w[1] - w_xm));
      const T d11q1 = sgs1;
      const T d22q1 = ap2c * visb * (u_yp - u[1]) -
                      am2c * visa * (u[1] - u_ym);
      const T d33q1 = ap3c * visd * (u[2] - u[1]) -
                      am3c * visc * (u[1] - u[0]);
      const T dcq13 = d11q1 + d33q1;
      const T gradp1 = (p[1] - p_xm) * rdx;
      if (live) fix_add(s1, (double)(u[1] * s1coe));
      const T convEd1 = -h11 - h12 - h13 + sgs1 + sgs2 + sgs3 + dcq13 + q.gx;
      ox = (q.pmGamma * convEd1 + q.pmTheta * hxo - q.pmAlpha * gradp1 + twoBT * d22q1);
      cx = convEd1;
    }
    if (MASK & 2) {
      const T h21 = ((u_xp + um_xp) * (v_xp + v[1]) -
                     (u[1] + u_ym) * (v[1] + v_xm)) * qdx1;
      const T h22 = ((vp[1] + v[1]) * (vp[1] + v[1]) -
                     (v[1] + v_ym) * (v[1] + v_ym)) * qsucac;
      const T h23 = ((w[2] + wm[1]) * (v[2] + v[1]) -
                     (w[1] + wm[0]) * (v[1] + v[0])) * qdx3;
      const T visa = T(0.25) * (t[1] + t_xm[1] + tm[1] + tm_xm);
      const T visb = T(0.25) * (t[1] + t_xp[1] + tm[1] + tm_xp);
      const T visc = T(0.25) * (t[1] + tm[1] + t[0] + tm[0]);
      const T visd = T(0.25) * (t[1] + tm[1] + t[2] + tm[2]);
      const T sgs1 = rdx * sucac *
                     (visb * (u_xp - um_xp) - visa * (u[1] - u_ym));
      const T sgs2 = ap2p * t[1] * (vp[1] - v[1]) -
                     am2p * tm[1] * (v[1] - v_ym);
      const T sgs3 = rdz * sucac *
                     (visd * (w[2] - wm[1]) - visc * (w[1] - wm[0]));
      const T d11q2 = ap1c * visb * (v_xp - v[1]) -
                      am1c * visa * (v[1] - v_xm);
      const T d22q2 = sgs2;
      const T d33q2 = ap3c * visd * (v[2] - v[1]) -
                      am3c * visc * (v[1] - v[0]);
      const T dcq13 = d11q2 + d33q2;
      const T gradp2 = (p[1] - p_ym) * sucac;
      const T convEd2 = -h21 - h22 - h23 + sgs1 + sgs2 + sgs3 + dcq13 + q.gy;
      oy = (q.pmGamma * convEd2 + q.pmTheta * hyo - q.pmAlpha * gradp2 + twoBT * d22q2);
      cy = convEd2;
    }
    if (MASK & 4) {
      const T h31 = ((u_xp + ukm_xp) * (w_xp + w[1]) -
                     (u[1] + u[0]) * (w[1] + w_xm)) * qdx1;
      const T h32 = ((vp[1] + vp[0]) * (w_yp + w[1]) -
                     (v[1] + v[0]) * (w[1] + wm[0])) * sucaj;
      const T h33 = ((w[2] + w[1]) * (w[2] + w[1]) -
                     (w[1] + w[0]) * (w[1] + w[0])) * qdx3;
      const T visa = T(0.25) * (t[0] + t_xm[0] + t[1] + t_xm[1]);
      const T visb = T(0.25) * (t[0] + t_xp[0] + t[1] + t_xp[1]);
      const T visc = T(0.25) * (t[0] + tm[0] + tm[1] + t[1]);
      const T visd = T(0.25) * (t[0] + tp[0] + tp[1] + t[1]);
      const T sgs1 = rdx * rdz *
                     (visb * (u_xp - ukm_xp) - visa * (u[1] - u[0]));
      const T sgs2 = rdz * rdyp *
                     (visd * (vp[1] - vp[0]) - visc * (v[1] - v[0]));
      const T sgs3 = q.rdz2 * (t[1] * (w[2] - w[1]) -
                               t[0] * (w[1] - w[0]));
      const T d11q3 = ap1c * visb * (w_xp - w[1]) -
                      am1c * visa * (w[1] - w_xm);
      const T d22q3 = ap2c * visd * (w_yp - w[1]) -
                      am2c * visc * (w[1] - wm[0]);
      const T d33q3 = sgs3;
      const T dcq13 = d11q3 + d33q3;
      const T gradp3 = (p[1] - p[0]) * rdz;
      const T convEd3 = -h31 - h32 - h33 + sgs1 + sgs2 + sgs3 + dcq13 + q.gz;
      oz = (q.pmGamma * convEd3 + q.pmTheta * hzo - q.pmAlpha * gradp3 + twoBT * d22q3);
      cz = convEd3;
    }
    stage(bm);
    if (live) {
      auto sto = [&](T* f, T val) { C3D_ST_ONCE(val, (T*)at(f)); };
      if (MASK & 1) { sto(rx, ox); sto(hx, cx); }
      if (MASK & 2) { sto(ry, oy); sto(hy, cy); }
      if (MASK & 4) { sto(rz, oz); sto(hz, cz); }
    }
    __syncthreads();
    const int b = bm;
    bm = bc; bc = bp; bp = b;
  }
  if (MASK & 1) {
    // reproducible block sum of the four limbs (order independent)
#pragma unroll
    for (int l = 0; l < 4; ++l)
      for (int o = 32; o > 0; o >>= 1) s1[l] += __shfl_down(s1[l], o, 64);
    const int tid = threadIdx.x + LBX * threadIdx.y;
    if ((tid & 63) == 0)
      for (int l = 0; l < 4; ++l) shf[tid >> 6][l] = s1[l];
    __syncthreads();
    if (tid == 0) {
      long long a[4] = {0, 0, 0, 0};
      for (int l = 0; l < 4; ++l)
        for (int w = 0; w < LBY; ++w) a[l] += shf[w][l];
      if (MASK == 7) {  // the fused substep's integral
        bulk_add(sc, a);
      } else {
        long long* pf = (long long*)partials + 4LL * blockIdx.x;
        for (int l = 0; l < 4; ++l) pf[l] = a[l];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// clcU1Hat_PIMP_LES (:466-499), clcU2Hat_PIMP_LES (:626-662),
// clcU3Hat_PIMP_LES (:776-809): per (i, k) line, InverseTridiagonal
// (m_Tools.f90:218-245) with the coefficients of each row built from nut.
// ADDD adds dd to RhsX as it is loaded (the constant-flow-rate shift of clcRhsX,
// :146-151).
//
// The line is cut into segments of LC rows, as in the full-implicit sweep:
// the forward pass keeps only each segment's last value and pivot (two words
// per segment and line, in the scratch field), the backward pass forms a
// segment's rows again from there (the same operations on the same operands,
// so the same values), substitutes and updates u.  A segment's right-hand
// side and nut rows are requested one segment ahead of the recurrence, in
// unconditional loads (rows past the last are read from it and not used).
// Traffic: the right-hand side and nut twice, u once, u written (7 words per
// component before: the forward values and factors of every row went to memory
// and back).  The metric rows are restrict arguments, so they come through
// scalar loads: as vector loads among the prefetches, waiting for one would
// wait for the prefetch before it.  The two quotients by a row's pivot share its reciprocal.
// Storing sweeps that loaded row by row were bound by HBM on large grids and
// by the loads' latency on small ones: the three took 0.896 ms at 384x192x288 and
// 0.072 ms at 96x96x72 (FP64), these take 0.490 and 0.030 ms.
// Lines are dealt flat over (i, k); the three components of a line's tile are
// neighbouring workgroups on one XCD and share its nut rows in L2.
// ---------------------------------------------------------------------------
constexpr int LC = 8;

template <typename T, int COMP, bool ADDD, bool NTS>
__device__ __forceinline__ void les_y_line(const Geom& g, const T* __restrict__ am,
                                           const T* __restrict__ ap, T bt,
                                           const T* __restrict__ nut,
                                           const T* __restrict__ rhs, T* __restrict__ ck,
                                           T* __restrict__ u, const T* __restrict__ duy,
                                           T dd, long long line) {
  const int nx = g.nx, ny = g.ny;
  const int i = (int)(line % nx), k = (int)(line / nx);
  const long long base = i + g.plane * k, nl = (long long)nx * g.nz;
  const T* pr = rhs + base;
  const T* pa = nut + base;
  // the face neighbour of nut: one cell down in x (ux) or z (uz)
  const T* pb = nut + (COMP == 0 ? wm(i, nx) + g.plane * k : i + g.plane * wm(k, g.nz));
  T* pu = u + base;
  T* pc = ck + line;
  const T wallv = COMP == 1 ? duy[line] : T(0);
  const int nseg = (ny + LC - 1) / LC, top = nseg - 1;
  struct Seg {
    T r[LC], a[LC + 2], b[LC + 2];  // right-hand side; nut rows one below to one above
  };
  // Only the top segment has rows past the last (read from it, not used); the
  // others run without the row clamp and guard, which is a branch of its own
  // around every row.
  using Gd = std::true_type;
  using Un = std::false_type;
  auto load = [&](Seg& y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
    const int lo = s * LC + 1;
#pragma unroll
    for (int q = 0; q < LC; ++q) y.r[q] = pr[(long long)nx * (G ? min(lo + q, ny) : lo + q)];
#pragma unroll
    for (int q = 0; q < LC + 2; ++q) {
      const long long o = (long long)nx * (G ? min(lo - 1 + q, ny + 1) : lo - 1 + q);
      y.a[q] = pa[o];
      if (COMP != 1) y.b[q] = pb[o];
    }
  };
  // the matrix row's coefficients: rt1 below, rt2 above
  auto coef = [&](const Seg& y, int q, int j, T& rt1, T& rt2) {
    if (COMP == 0) {
      const T c = y.a[q + 1] + y.b[q + 1];
      rt1 = bt * (T(0.25) * (c + y.a[q] + y.b[q])) * am[j];
      rt2 = bt * (T(0.25) * (c + y.a[q + 2] + y.b[q + 2])) * ap[j];
    } else if (COMP == 1) {
      rt1 = bt * y.a[q] * am[j];
      rt2 = bt * y.a[q + 1] * ap[j];
    } else {
      rt1 = bt * (T(0.25) * (y.b[q + 1] + y.b[q] + y.a[q + 1] + y.a[q])) * am[j];
      rt2 = bt * (T(0.25) * (y.b[q + 1] + y.b[q + 2] + y.a[q + 1] + y.a[q + 2])) * ap[j];
    }
  };
  T f = T(0), vecm = T(1), rv = T(1), cprev = T(0);  // rv: 1/vecm
  T ar[LC];
  // forward through segment s from (f, vecm, rv, cprev): values into y.r,
  // factors into ar.  Row 1 has nothing below: f = 0, vecm = 1 and cprev = 0
  // give its pivot b and value r/b.
  auto fwd = [&](Seg& y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
    const int lo = s * LC + 1;
#pragma unroll
    for (int q = 0; q < LC; ++q) {
      const int j = lo + q;
      if (!G || j <= ny) {
        T rt1, rt2, fj = ADDD ? y.r[q] + dd : y.r[q];
        coef(y, q, j, rt1, rt2);
        if (COMP == 1 && q == 0 && s == 0) {  // the wall row
          rt1 = rt2 = T(0);
          fj = wallv;
        }
        const T a = -rt1, b = rt1 + rt2 + T(1);
        ar[q] = quot(cprev, vecm, rv);
        vecm = b - a * ar[q];
        rv = quot_recip(vecm);
        f = quot(fj - a * f, vecm, rv);
        cprev = -rt2;
        y.r[q] = f;
      }
    }
  };
  auto save = [&](int s) {
    pc[nl * (2 * s)] = f;
    pc[nl * (2 * s + 1)] = vecm;
  };
  T x = T(0), arn = T(0);  // the solution and factor of the row above
  // through segment s: u's words are requested before the next segment's, so
  // waiting for them leaves that prefetch in flight
  T uv[LC];
  auto loadu = [&](int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
    const int lo = s * LC + 1;
#pragma unroll
    for (int q = 0; q < LC; ++q)
      uv[q] = C3D_LD_ONCE(&pu[(long long)nx * (G ? min(lo + q, ny) : lo + q)]);
  };
  auto back = [&](const Seg& y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
    const int lo = s * LC + 1;
#pragma unroll
    for (int q = LC - 1; q >= 0; --q) {
      const int j = lo + q;
      if (!G || j <= ny) {
        if (!G || j < ny) x = y.r[q] - (q + 1 < LC ? ar[q + 1] : arn) * x;
        C3D_ST_ONCE(uv[q] + x, &pu[(long long)nx * j]);
      }
    }
    arn = ar[0];
  };
  Seg ya, yb;
  int s = 0;
  if (top == 0) load(ya, 0, Gd{});
  else load(ya, 0, Un{});
  for (; s + 2 < top; s += 2) {
    load(yb, s + 1, Un{});
    __builtin_amdgcn_sched_barrier(0);
    fwd(ya, s, Un{});
    save(s);
    load(ya, s + 2, Un{});
    __builtin_amdgcn_sched_barrier(0);
    fwd(yb, s + 1, Un{});
    save(s + 1);
  }
  if (s + 2 == top) {
    load(yb, s + 1, Un{});
    __builtin_amdgcn_sched_barrier(0);
    fwd(ya, s, Un{});
    save(s);
    load(ya, top, Gd{});
    __builtin_amdgcn_sched_barrier(0);
    fwd(yb, s + 1, Un{});
    save(s + 1);
  } else if (s + 1 == top) {
    load(yb, top, Gd{});
    __builtin_amdgcn_sched_barrier(0);
    fwd(ya, s, Un{});
    save(s);
    ya = yb;
  }
  fwd(ya, top, Gd{});
  x = f;
  loadu(top, Gd{});
  if (top > 0) load(yb, top - 1, Un{});
  __builtin_amdgcn_sched_barrier(0);
  back(ya, top, Gd{});
  for (s = top - 1; s >= 0; --s) {
    ya = yb;
    loadu(s, Un{});
    f = T(0);
    vecm = rv = T(1);
    cprev = T(0);
    if (s > 0) {
      f = pc[nl * (2 * s - 2)];
      vecm = pc[nl * (2 * s - 1)];
      load(yb, s - 1, Un{});
    }
    __builtin_amdgcn_sched_barrier(0);
    if (s > 0) {
      rv = quot_recip(vecm);
      // the row below the segment's first: its upper coefficient
      const int j = s * LC;
      T rt2;
      if (COMP == 0)
        rt2 = bt * (T(0.25) * (ya.a[0] + ya.b[0] + ya.a[1] + ya.b[1])) * ap[j];
      else if (COMP == 1)
        rt2 = bt * ya.a[0] * ap[j];
      else
        rt2 = bt * (T(0.25) * (ya.b[0] + ya.b[1] + ya.a[0] + ya.a[1])) * ap[j];
      cprev = -rt2;
    }
    fwd(ya, s, Un{});
    back(ya, s, Un{});
  }
}

template <typename T, int COMP, bool ADDD, bool NTS>
__global__ __launch_bounds__(64) void k_les_y(Geom g, const T* __restrict__ am,
                                              const T* __restrict__ ap, T bt,
                                              const T* __restrict__ nut,
                                              const T* __restrict__ rhs, T* __restrict__ ck,
                                              T* __restrict__ u, const T* __restrict__ duy,
                                              const DevScalars* __restrict__ sc) {
  const long long line = (long long)blockIdx.x * 64 + threadIdx.x;
  if (line >= (long long)g.nx * g.nz) return;
  les_y_line<T, COMP, ADDD, NTS>(g, am, ap, bt, nut, rhs, ck, u, duy,
                                       ADDD ? (T)sc->dpmdxns : T(0), line);
}

// The three component solves of one LES substep in one launch, component
// fastest, each with its own velocity, right-hand side and checkpoint scratch.
// The solves are independent (each reads only nut and its own arrays).
template <typename T>
struct LesY3 {
  T* u[3];
  const T* rhs[3];
  T* ck[3];
  const T* duy;
};

template <typename T, bool ADDD, bool NTS>
__global__ __launch_bounds__(64) void k_les_y3(Geom g, const T* __restrict__ amc,
                                               const T* __restrict__ apc,
                                               const T* __restrict__ amp,
                                               const T* __restrict__ app, T bt,
                                               const T* __restrict__ nut, LesY3<T> a, Bulk bk,
                                               DevScalars* sc) {
  const int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int comp = lb % 3;
  const long long line = (long long)(lb / 3) * 64 + threadIdx.x;
  if (line >= (long long)g.nx * g.nz) return;
  if (comp == 0)
    les_y_line<T, 0, ADDD, NTS>(g, amc, apc, bt, nut, a.rhs[0], a.ck[0], a.u[0], nullptr,
                                ADDD ? (T)bulk_shift(bk, sc, line == 0) : T(0), line);
  else if (comp == 1)
    les_y_line<T, 1, false, NTS>(g, amp, app, bt, nut, a.rhs[1], a.ck[1], a.u[1], a.duy, T(0),
                                 line);
  else
    les_y_line<T, 2, false, NTS>(g, amc, apc, bt, nut, a.rhs[2], a.ck[2], a.u[2], nullptr, T(0),
                                 line);
}

// ---------------------------------------------------------------------------
// PressureUpdate_PIMP_LES (:878-904): p += (1 - pmBetaT d/dy nut d/dy) phi.
// phi's wall ghosts must hold the Neumann copies (SetBC_and_UpdateHalo_pr).
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(LBX* LBY) void k_prupd_les(Geom g, Metrics<T> m, T bt,
                                                        const T* __restrict__ nut,
                                                        const T* __restrict__ phi,
                                                        T* __restrict__ pr) {
  LES_CELL();
  if (i >= g.nx || jc > g.ny) return;
  const int nx = g.nx, nyh = g.nyh;
  const int jm = jc - 1, jp = jc + 1;
  const T metr1 = m.rdyp[jc] * m.rdyc[jc];
  const T metr2 = m.rdyp[jc] * m.rdyc[jp];
  for (int k = kz0; k < kz1; ++k) {
    const T visd = T(0.5) * (A(nut, i, jp, k) + A(nut, i, jc, k));
    const T visc = T(0.5) * (A(nut, i, jc, k) + A(nut, i, jm, k));
    const T pmBetap = -(bt * metr2 * visd);
    const T pmBetam = -(bt * metr1 * visc);
    const T pmBetac = -(pmBetap + pmBetam) + T(1);
    const long long c = fidx(g, i, jc, k);
    pr[c] = pr[c] + pmBetap * A(phi, i, jp, k) + pmBetac * phi[c] + pmBetam * A(phi, i, jm, k);
  }
}

// ---------------------------------------------------------------------------
// The end of an LES substep in one pass: SetBC_and_UpdateHalo_pr of phi,
// FluidVelUpdate (m_TScheme.f90:281-306), PressureUpdate_PIMP_LES, and the wall
// ghosts of SetBC_and_UpdateHalo and SetBC_and_UpdateHalo_pr.  Rows 1, 2 and ny
// write the ghosts of u and p from their new values, and phi's from phi.  A thread walks a run of z planes of its
// column and requests plane k+1 before it stores plane k (one counter covers
// both).  As five launches, phi was read twice and each launch cost about 5 us:
// 0.235 + 0.143 + 0.016 ms at 384x192x288, now 0.354 ms; 5 launches fewer a
// substep at 96x96x72.
// ---------------------------------------------------------------------------
constexpr int PLKCH = 16;  // longest z run

template <typename T, bool NTS>
__global__ __launch_bounds__(LBX* LBY) void k_proj_les(Geom g, Metrics<T> m, T rdxE, T rdzE,
                                                       T alpha, T bt, WallBC wb, int kchunk,
                                                       const T* __restrict__ nut,
                                                       T* __restrict__ phi,
                                                       T* __restrict__ ux, T* __restrict__ uy,
                                                       T* __restrict__ uz, T* __restrict__ pr) {
  const int gxb = (g.nx + LBX - 1) / LBX, gyb = (g.ny + LBY - 1) / LBY;
  const int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int i = (lb % gxb) * LBX + threadIdx.x;
  const int jc = ((lb / gxb) % gyb) * LBY + threadIdx.y + 1;
  if (i >= g.nx || jc > g.ny) return;
  const int k0 = (lb / (gxb * gyb)) * kchunk, k1 = min(g.nz, k0 + kchunk);
  const int im = wm(i, g.nx);
  const T sucac = m.rdyc[jc] * alpha;
  const T metr1 = m.rdyp[jc] * m.rdyc[jc], metr2 = m.rdyp[jc] * m.rdyc[jc + 1];
  const long long row = (long long)g.nx * jc;
  struct Plane {
    T ph, phx, phm, php, tm, t, tp, u, v, w, p;
  };
  auto fetch = [&](int k, Plane& a) {
    const long long c = row + g.plane * k + i;
    a.ph = phi[c];
    a.phx = phi[c - i + im];
    a.phm = phi[c - g.nx];
    a.php = phi[c + g.nx];
    a.tm = nut[c - g.nx];
    a.t = nut[c];
    a.tp = nut[c + g.nx];
    a.u = C3D_LD_ONCE(&ux[c]);
    a.v = C3D_LD_ONCE(&uy[c]);
    a.w = C3D_LD_ONCE(&uz[c]);
    a.p = C3D_LD_ONCE(&pr[c]);
  };
  auto update = [&](int k, const Plane& a, T phz, auto wallv) {
    constexpr bool WALL = decltype(wallv)::value;
    __builtin_amdgcn_sched_barrier(0);  // this plane's stores stay behind the next one's loads
    const long long c = row + g.plane * k + i;
    const T ph = a.ph;
    const T phm = WALL && jc == 1 ? ph : a.phm, php = WALL && jc == g.ny ? ph : a.php;
    const T un = a.u - (ph - a.phx) * rdxE;
    T vn = a.v - (ph - phm) * sucac;
    const T wn = a.w - (ph - phz) * rdzE;
    if (WALL) vn = walls_vel(g, wb, jc, c, un, vn, wn, ux, uy, uz);
    const T visd = T(0.5) * (a.tp + a.t);
    const T visc = T(0.5) * (a.t + a.tm);
    const T bp = -(bt * metr2 * visd);
    const T bm = -(bt * metr1 * visc);
    const T bc = -(bp + bm) + T(1);
    const T pn = a.p + bp * php + bc * ph + bm * phm;
    // phi's ghosts too: the thread that writes one is the only one that reads it
    if (WALL && jc == 1) {
      pr[c - g.nx] = pn;
      phi[c - g.nx] = ph;
    }
    if (WALL && jc == g.ny) {
      pr[c + g.nx] = pn;
      phi[c + g.nx] = ph;
    }
    C3D_ST_ONCE(un, &ux[c]);
    C3D_ST_ONCE(vn, &uy[c]);
    C3D_ST_ONCE(wn, &uz[c]);
    C3D_ST_ONCE(pn, &pr[c]);
  };
  auto march = [&](auto wallv) {
    T phz = phi[row + g.plane * wm(k0, g.nz) + i];
    Plane a, b;
    fetch(k0, a);
    int k = k0;
    for (; k + 2 < k1; k += 2) {
      fetch(k + 1, b);
      update(k, a, phz, wallv);
      phz = a.ph;
      fetch(k + 2, a);
      update(k + 1, b, phz, wallv);
      phz = b.ph;
    }
    if (k + 1 < k1) {
      fetch(k + 1, b);
      update(k, a, phz, wallv);
      update(k + 1, b, a.ph, wallv);
    } else {
      update(k, a, phz, wallv);
    }
  };
  // a wavefront is one row: those that write no ghost run without the tests
  if (jc <= 2 || jc == g.ny) march(std::true_type{});
  else march(std::false_type{});
}
#undef A

// ===========================================================================
// launchers
// ===========================================================================
template <typename T>
static int sgs_t(c3d_ctx* c, const void* ux, const void* uy, const void* uz, void* nut) {
  const Geom& g = c->g;
  const LesCoef<T> q = make_les_coef<T>(c);
  const int tiles = ((g.nx + LBX - 1) / LBX) * ((g.ny + LBY - 1) / LBY);
  const int kc = march_kchunk((long long)tiles * LBY, g.nz, c->les_type == 2 ? 2 : 3);
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(tiles * ((g.nz + kc - 1) / kc)), dim3(LBX, LBY), 0, c->stream, g,
                       met<T>(c), lesmet<T>(c), q, (const T*)ux, (const T*)uy, (const T*)uz,
                       (T*)nut, kc);
  };
  if (c->les_type == 2) launch(k_sgs<T, false>);
  else launch(k_sgs<T, true>);
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

int launch_sgs(c3d_ctx* c, const void* ux, const void* uy, const void* uz, void* nut) {
  hipEvent_t ev;
  prof_begin(c, ST_SGS, &ev);
  int rc = c->les_closure ? closure_nut(c->les_closure, c, ux, uy, uz, nut)
           : c->prec == C3D_FP64 ? sgs_t<double>(c, ux, uy, uz, nut)
                                 : sgs_t<float>(c, ux, uy, uz, nut);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  prof_end(c, ST_SGS, ev, 4.0 * N * c->esize);
  return C3D_OK;
}

static int rhs_les_kchunk(const Geom& g) {
  const int gx = (g.nx + LBX - 1) / LBX, gy = (g.ny + LBY - 1) / LBY;
  return march_kchunk((long long)gx * gy * LBY, g.nz, 2);
}
static int rhs_les_blocks(const Geom& g) {
  const int kc = rhs_les_kchunk(g);
  return ((g.nx + LBX - 1) / LBX) * ((g.ny + LBY - 1) / LBY) * ((g.nz + kc - 1) / kc);
}

template <typename T>
static int rhs_les_t(c3d_ctx* c, int mask, const void* ux, const void* uy, const void* uz,
                     const void* pr, void* rx, void* ry, void* rz, void* hx, void* hy, void* hz) {
  const Geom& g = c->g;
  const LesCoef<T> q = make_les_coef<T>(c);
  const T* nut = (const T*)c->state[C3D_NUT];
  const int kc = rhs_les_kchunk(g), nb = rhs_les_blocks(g);
  if ((mask & 1) && 4 * nb > c->max_partials) {
    set_error("rhs_les: partial buffer too small");
    return C3D_ERR_ARG;
  }
  auto launch = [&](auto mc, auto ntc) {
    hipLaunchKernelGGL((k_rhs_les<T, decltype(mc)::value, decltype(ntc)::value>), dim3(nb),
                       dim3(LBX, LBY), 0, c->stream, g, met<T>(c), q, (const T*)ux, (const T*)uy,
                       (const T*)uz, (const T*)pr, nut, (T*)rx, (T*)ry, (T*)rz, (T*)hx, (T*)hy,
                       (T*)hz, c->d_partials, c->d_sc, kc);
  };
#define RL(M)                                                                       \
  if (g.nt) launch(std::integral_constant<int, M>{}, std::true_type{});             \
  else launch(std::integral_constant<int, M>{}, std::false_type{})
  switch (mask) {
    case 1: RL(1); break;
    case 2: RL(2); break;
    case 4: RL(4); break;
    case 7: RL(7); break;
    default: set_error("rhs_les: bad component mask"); return C3D_ERR_ARG;
  }
#undef RL
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

int launch_rhs_les(c3d_ctx* c, int mask, const void* ux, const void* uy, const void* uz,
                   const void* pr, void* rx, void* ry, void* rz, void* hx, void* hy, void* hz,
                   int want_bulk) {
  hipEvent_t ev;
  const int st = mask == 7 ? ST_RHS : ST_RHS1;
  prof_begin(c, st, &ev);
  int rc = c->prec == C3D_FP64 ? rhs_les_t<double>(c, mask, ux, uy, uz, pr, rx, ry, rz, hx, hy, hz)
                               : rhs_les_t<float>(c, mask, ux, uy, uz, pr, rx, ry, rz, hx, hy, hz);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  const int ncomp = (mask & 1) + ((mask >> 1) & 1) + ((mask >> 2) & 1);
  prof_end(c, st, ev, (ncomp == 3 ? 14.0 : 7.0) * N * c->esize);
  if (want_bulk && mask == 1 && c->p.is_ux_const)
    return launch_bulk_finalize(c, rhs_les_blocks(c->g), c->cur_ns == 1);
  return C3D_OK;
}

template <typename T>
static int les_y_t(c3d_ctx* c, int comp, void* u, const void* rhs, const void* duy, int addd) {
  const Geom& g = c->g;
  const dim3 grid((unsigned)(((long long)g.nx * g.nz + 63) / 64)), blk(64);
  const T bt = (T)c->pmBetaT;
  const T* nut = (const T*)c->state[C3D_NUT];
  auto launch = [&](auto cc, auto dc, auto ntc) {
    hipLaunchKernelGGL(
        (k_les_y<T, decltype(cc)::value, decltype(dc)::value, decltype(ntc)::value>), grid, blk, 0,
        c->stream, g, comp == 1 ? met<T>(c).am2p : lesmet<T>(c).am2ccn,
        comp == 1 ? met<T>(c).ap2p : lesmet<T>(c).ap2ccn, bt, nut, (const T*)rhs, (T*)c->tmpA,
        (T*)u, (const T*)duy, (const DevScalars*)c->d_sc);
  };
  using Yes = std::true_type;
  using No = std::false_type;
  auto by_nt = [&](auto cc, auto dc) {
    if (g.nt) launch(cc, dc, Yes{});
    else launch(cc, dc, No{});
  };
  if (comp == 0 && addd) by_nt(std::integral_constant<int, 0>{}, Yes{});
  else if (comp == 0) by_nt(std::integral_constant<int, 0>{}, No{});
  else if (comp == 1) by_nt(std::integral_constant<int, 1>{}, No{});
  else by_nt(std::integral_constant<int, 2>{}, No{});
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

int launch_les_y(c3d_ctx* c, int comp, void* u, void* rhs, const void* duy_ym, int add_dpmdxns) {
  if (comp == 1 && !duy_ym) {
    set_error("clcU2Hat: duy_ym is required");
    return C3D_ERR_ARG;
  }
  hipEvent_t ev;
  prof_begin(c, ST_ADI_Y, &ev);
  int rc = c->prec == C3D_FP64 ? les_y_t<double>(c, comp, u, rhs, duy_ym, add_dpmdxns)
                               : les_y_t<float>(c, comp, u, rhs, duy_ym, add_dpmdxns);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  prof_end(c, ST_ADI_Y, ev, 4.0 * N * c->esize);
  return C3D_OK;
}

template <typename T>
static int les_y3_t(c3d_ctx* c, void* const u[3], void* const rhs[3], const void* duy, int addd) {
  const Geom& g = c->g;
  LesY3<T> a;
  void* const ck[3] = {c->tmpA, c->les_arr[0], c->les_arr[1]};
  for (int d = 0; d < 3; ++d) {
    a.u[d] = (T*)u[d];
    a.rhs[d] = (const T*)rhs[d];
    a.ck[d] = (T*)ck[d];
  }
  a.duy = (const T*)duy;
  const dim3 grid((unsigned)(3 * (((long long)g.nx * g.nz + 63) / 64))), blk(64);
  const T bt = (T)c->pmBetaT;
  const T* nut = (const T*)c->state[C3D_NUT];
  auto launch = [&](auto dc, auto ntc) {
    hipLaunchKernelGGL((k_les_y3<T, decltype(dc)::value, decltype(ntc)::value>), grid, blk, 0,
                       c->stream, g, lesmet<T>(c).am2ccn, lesmet<T>(c).ap2ccn, met<T>(c).am2p,
                       met<T>(c).ap2p, bt, nut, a, make_bulk(c), c->d_sc);
  };
  if (addd) {
    if (g.nt) launch(std::true_type{}, std::true_type{});
    else launch(std::true_type{}, std::false_type{});
  } else {
    if (g.nt) launch(std::false_type{}, std::true_type{});
    else launch(std::false_type{}, std::false_type{});
  }
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

int launch_les_y3(c3d_ctx* c, void* const u[3], void* const rhs[3], const void* duy_ym,
                  int add_dpmdxns) {
  if (!duy_ym || !c->les_arr[0] || !c->les_arr[1]) {
    set_error("LES y-solves: duy_ym and the LES scratch fields are required");
    return C3D_ERR_ARG;
  }
  hipEvent_t ev;
  prof_begin(c, ST_ADI_Y, &ev);
  int rc = c->prec == C3D_FP64 ? les_y3_t<double>(c, u, rhs, duy_ym, add_dpmdxns)
                               : les_y3_t<float>(c, u, rhs, duy_ym, add_dpmdxns);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  prof_end(c, ST_ADI_Y, ev, 12.0 * N * c->esize);
  return C3D_OK;
}

template <typename T>
static int proj_les_t(c3d_ctx* c, void* phi, void* ux, void* uy, void* uz, void* pr) {
  const Geom& g = c->g;
  // down to two planes a run until every CU has four workgroups (the rule of the
  // second-order projection)
  const int tiles = ((g.nx + LBX - 1) / LBX) * ((g.ny + LBY - 1) / LBY);
  int kc = PLKCH;
  while (kc > 2 && tiles * ((g.nz + kc - 1) / kc) < 1024) kc /= 2;
  const dim3 grid(tiles * ((g.nz + kc - 1) / kc)), blk(LBX, LBY);
  auto launch = [&](auto ntc) {
    hipLaunchKernelGGL((k_proj_les<T, decltype(ntc)::value>), grid, blk, 0, c->stream, g, met<T>(c),
                       (T)(c->rdx * c->pmAlpha), (T)(c->rdz * c->pmAlpha), (T)c->pmAlpha,
                       (T)c->pmBetaT, make_wallbc(c), kc, (const T*)c->state[C3D_NUT], (T*)phi,
                       (T*)ux, (T*)uy, (T*)uz, (T*)pr);
  };
  if (g.nt) launch(std::true_type{});
  else launch(std::false_type{});
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

int launch_proj_les(c3d_ctx* c, void* phi, void* ux, void* uy, void* uz, void* pr) {
  hipEvent_t ev;
  prof_begin(c, ST_PROJ, &ev);
  int rc = c->prec == C3D_FP64 ? proj_les_t<double>(c, phi, ux, uy, uz, pr)
                               : proj_les_t<float>(c, phi, ux, uy, uz, pr);
  if (rc) return rc;
  prof_end(c, ST_PROJ, ev, 10.0 * (double)c->g.nx * c->g.ny * c->g.nz * c->esize);
  return C3D_OK;
}

int launch_prupd_les(c3d_ctx* c, void* pr, const void* phi) {
  const Geom& g = c->g;
  hipEvent_t ev;
  prof_begin(c, ST_PRUPD, &ev);
  if (c->prec == C3D_FP64)
    hipLaunchKernelGGL(k_prupd_les<double>, dim3(les_blocks(g)), dim3(LBX, LBY), 0, c->stream, g,
                       c->md, (double)c->pmBetaT, (const double*)c->state[C3D_NUT],
                       (const double*)phi, (double*)pr);
  else
    hipLaunchKernelGGL(k_prupd_les<float>, dim3(les_blocks(g)), dim3(LBX, LBY), 0, c->stream, g,
                       c->mf, (float)c->pmBetaT, (const float*)c->state[C3D_NUT],
                       (const float*)phi, (float*)pr);
  C3D_HIP(hipGetLastError());
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  prof_end(c, ST_PRUPD, ev, 4.0 * N * c->esize);
  return C3D_OK;
}

}  // namespace c3d
