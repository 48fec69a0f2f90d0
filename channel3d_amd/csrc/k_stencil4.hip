// Kernels of the 4th-order channel step (src/CFD_4th): the fused right-hand
// sides clcRhsXYZ, the pressure source, the projection with the
// Helmholtz-corrected pressure update, the wall ghosts and the 4th-order
// divergence check.
//
// x and z use 4th-order staggered differences (1,-27,27,-1)/24,
// interpolations (-1,9,9,-1)/16 and second differences (-1,16,-30,16,-1)/12
// (m_MeshAndMetries.f90:87-91); y stays 2nd order.  The reference builds six
// interpolated helper fields (uxhx ... uzhz, m_TScheme.f90:203-233) and
// exchanges their halos before the right-hand sides; here each helper value
// is recomputed where it is used, from the same four neighbours in the same
// order, so nothing extra is written to or read back from HBM.  Periodic x
// and z neighbours wrap by index (offsets up to 3).  Expressions keep the
// reference's evaluation order; the file is compiled without contraction.
#include "c3d_internal.h"

namespace c3d {

constexpr int B4X = 64, B4Y = 4, K4CH = 4;

__device__ __forceinline__ int wr(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// read-only view of a field with periodic x/z wrap
template <typename T>
struct View {
  const T* __restrict__ p;
  int nx, nz;
  long long plane;
  __device__ __forceinline__ T operator()(int i, int jj, int k) const {
    return p[(long long)wr(i, nx) + (long long)nx * jj + plane * (long long)wr(k, nz)];
  }
};


// 1-D grid of 64 x 4 (i, j) tiles times z runs, XCD-remapped, x fastest
#define CELL4_BLOCK(KCH)                                                      \
  const int cgx_ = (g.nx + B4X - 1) / B4X, cgy_ = (g.ny + B4Y - 1) / B4Y;     \
  const int clb_ = xcd_remap(blockIdx.x, gridDim.x);                          \
  const int cbx = clb_ % cgx_, cby = (clb_ / cgx_) % cgy_, cbz = clb_ / (cgx_ * cgy_); \
  const int i = cbx * B4X + threadIdx.x;                                      \
  const int jc = cby * B4Y + threadIdx.y + 1;                                 \
  const int k0 = cbz * (KCH), k1 = min(g.nz, k0 + (KCH))

__device__ __forceinline__ void block_fix4(long long* v, long long (*sh)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q)
    for (int o = 32; o > 0; o >>= 1) v[q] += __shfl_down(v[q], o, 64);
  const int tid = threadIdx.x + blockDim.x * threadIdx.y;
  const int lane = tid & 63, w = tid >> 6;
  if (lane == 0)
    for (int q = 0; q < 4; ++q) sh[w][q] = v[q];
  __syncthreads();
  if (tid == 0) {
    const int nw = (blockDim.x * blockDim.y + 63) / 64;
    for (int q = 0; q < 4; ++q) {
      long long a = 0;
      for (int u = 0; u < nw; ++u) a += sh[u][q];
      v[q] = a;
    }
  }
}

__device__ __forceinline__ double block_max4(double v, double* sh) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
  const int tid = threadIdx.x + blockDim.x * threadIdx.y;
  const int lane = tid & 63, w = tid >> 6;
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0;
  if (tid == 0) {
    const int nw = (blockDim.x * blockDim.y + 63) / 64;
    for (int q = 0; q < nw; ++q) r = fmax(r, sh[q]);
  }
  return r;
}

// ---------------------------------------------------------------------------
// clcRhsXYZ (m_TScheme.f90:189-438, the branch without scalar or particle
// coupling).  RhsX (:243-290), RhsY (:293-330), RhsZ (:333-370); with
// want_flow the block partial of s3tot = sum (d11+d33+d22) dyp (:271) is
// accumulated as reproducible fixed-point limbs (2: into the fused substep's
// slots).
//
// A wavefront owns 64 x cells of one row and marches a run of z planes.
//  - z: every value along the own column (u, v, w, p, uy one row up, and the
//    z- and x-interpolated factors of the z fluxes) enters once, when its
//    plane arrives, and rolls through registers.
//  - x: each plane's rows go through LDS with three cells on either side; lane
//    n < 6 also carries one of those six edge columns.  A row belongs to its
//    wavefront alone and a wavefront's LDS accesses complete in order, so
//    nothing waits at a workgroup barrier.
//  - y: the neighbour rows are read directly; the wavefront one row over has
//    just read them, so they come from L1.
// The next plane's words are requested before this plane is computed, and this
// plane's results are stored after that, so waiting for the one never waits
// for the other.  26 memory operations per wavefront and plane where every
// operand fetched on its own took about 110, each with its own periodic index:
// bound by the FP64 pipeline (about 450 operations per cell, uncontracted)
// and HBM (13 words).  192x128x160 FP64: 0.288 ms so, 0.125 ms now (3.3 TB/s
// of its 13 words).
// ---------------------------------------------------------------------------
constexpr int R4E = 3;                 // edge columns on either side
constexpr int R4L = 64 + 2 * R4E + 2;  // an LDS row, with a slot for idle lanes

template <typename T>
__global__ __launch_bounds__(B4X* B4Y, 2) void k_rhs4(Geom g, Metrics<T> m, Coef4<T> cf,
                                                   const double* __restrict__ dyp,
                                                   const T* __restrict__ ux, const T* __restrict__ uy,
                                                   const T* __restrict__ uz, const T* __restrict__ pr,
                                                   T* __restrict__ rx, T* __restrict__ ry,
                                                   T* __restrict__ rz, T* __restrict__ hx,
                                                   T* __restrict__ hy, T* __restrict__ hz,
                                                   double* __restrict__ partials,
                                                   DevScalars* sc, int want_flow,
                                                   int kchunk) {
  __shared__ long long shf[8][4];
  enum { RU, RV, RW, RP, RVP, RUM, RIZ, RW2, NROW };
  __shared__ T rows[B4Y][NROW][R4L];
  const int gxb = (g.nx + B4X - 1) / B4X, gyb = (g.ny + B4Y - 1) / B4Y;
  const int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int i0 = (lb % gxb) * B4X;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int jc = ((lb / gxb) % gyb) * B4Y + wv + 1;
  const int k0 = (lb / (gxb * gyb)) * kchunk, k1 = min(g.nz, k0 + kchunk);
  const int lane = threadIdx.x;
  const int nx = g.nx, nz = g.nz;
  long long s3[4] = {0, 0, 0, 0};
  if (jc <= g.ny) {
    const int last = min(B4X, nx - i0) - 1;
    const bool live = lane <= last;
    const int i = min(i0 + lane, nx - 1);
    // edge column of lanes 0..5 and its place in a row; idle lanes repeat
    // lane 0's column into the spare slot
    const int ie = lane < 3 || lane >= 6 ? wr(i0 - 3 + (lane < 3 ? lane : 0), nx)
                                         : wr(i0 + last + 1 + lane - 3, nx);
    const int pe = lane < 3 ? lane : lane < 6 ? last + 1 + lane : R4L - 1;
    const int e = R4E + lane;
    T(*const row)[R4L] = rows[wv];
    const int jm = jc - 1, jp = jc + 1, nyp = g.ny + 1;
    const T sucaj = m.rdyp[jc], sucac = m.rdyc[jc];
    const T qsucac = T(0.25) * sucac;
    const T IY1 = m.yint[jc], IY2 = T(1) - IY1;
    const T IY3 = m.yint[jp], IY4 = T(1) - IY3;
    const T am2c = m.am2c[jc], ac2c = m.ac2c[jc], ap2c = m.ap2c[jc];
    const T am2p = m.am2p[jc], ac2p = m.ac2p[jc], ap2p = m.ap2p[jc];
    const double dy = dyp[jc];
    const T ucrf = cf.ucrf;
    // word at byte `at` of row j, plane k (periodic): a scalar row address
    // plus a 32-bit lane offset
    auto ld = [&](const T* f, int j, int k, unsigned at) {
      return *(const T*)((const char*)(f + ((long long)nx * j + g.plane * wr(k, nz))) + at);
    };
    const unsigned oi = i * (unsigned)sizeof(T), oe = ie * (unsigned)sizeof(T);
    // 4-point interpolation (-1, 9, 9, -1)/16, difference (1, -27, 27, -1)/24
    // and second difference (-1, 16, -30, 16, -1)/12 of neighbouring values.
    // The weights are symmetric to the bit, so one of each pair is kept: a
    // product with the negated weight, subtracted, rounds the same.
    auto i4 = [](T a, T b, T c, T d) {
      return T(-0.0625) * a + T(0.5625) * b + T(0.5625) * c + T(-0.0625) * d;
    };
    const T dx1 = cf.dx1, dx3 = cf.dx3, dz1 = cf.dz1, dz3 = cf.dz3;
    auto d5x = [&](T a, T b, T c, T d, T f) {
      return cf.dxx1 * a + cf.dxx2 * b + cf.dxx3 * c + cf.dxx2 * d + cf.dxx1 * f;
    };
    auto d5z = [&](const T* c) {
      return cf.dzz1 * c[0] + cf.dzz2 * c[1] + cf.dzz3 * c[2] + cf.dzz2 * c[3] + cf.dzz1 * c[4];
    };
    auto put = [&](int r, T own, T edge) {
      row[r][e] = own;
      row[r][pe] = edge;  // after the own cells: a partial tile's right edge wins
    };
    auto fence = [&]() {
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_wave_barrier();
    };
    // x interpolation ("B") of the row in r at the own cell
    auto ixb_of = [&](int r) { return i4(row[r][e - 2], row[r][e - 1], row[r][e], row[r][e + 1]); };

    // the words of one plane's step: u, v, w at k+3; uz one row down at k+2;
    // p, uy one row up and the edge of ux at k+1; the rest at k
    struct Next {
      T u3, v3, w3, wm2, ew2, p1, vp1, eu1;
      T um, up, vm, wp, pm, ev, ep, evp, eum, hx, hy, hz;
    };
    auto fetch = [&](int k, Next& n) {
      const int kc = wr(k, nz);
      n.hx = ld(hx, jc, kc, oi);
      n.hy = ld(hy, jc, kc, oi);
      n.hz = ld(hz, jc, kc, oi);
      n.u3 = ld(ux, jc, k + 3, oi);
      n.v3 = ld(uy, jc, k + 3, oi);
      n.w3 = ld(uz, jc, k + 3, oi);
      n.wm2 = ld(uz, jm, k + 2, oi);
      n.ew2 = ld(uz, jc, k + 2, oe);
      n.p1 = ld(pr, jc, k + 1, oi);
      n.vp1 = ld(uy, jp, k + 1, oi);
      n.eu1 = ld(ux, jc, k + 1, oe);
      n.um = ld(ux, jm, kc, oi);
      n.up = ld(ux, jp, kc, oi);
      n.vm = ld(uy, jm, kc, oi);
      n.wp = ld(uz, jp, kc, oi);
      n.pm = ld(pr, jm, kc, oi);
      n.ev = ld(uy, jc, kc, oe);
      n.ep = ld(pr, jc, kc, oe);
      n.evp = ld(uy, jp, kc, oe);
      n.eum = ld(ux, jm, kc, oe);
    };

    // rolled columns; index 0 is the oldest plane named beside each
    T u[6], v[6], w[6];             // k-2 .. k+3
    T zu[4], zv[4], xw[4], yw[4];   // izb(ux), izb(uy), ixb(uz), uz at the xz edge: k-1 .. k+2
    T za[4];                        // iza(uz): k-2 .. k+1
    T p[4], vp[4], eu[4];           // k-2 .. k+1
    T wm[3], ew[3];                 // k .. k+2
    {
      T a[6], b[6], c[6];           // planes k0-3 .. k0+2
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        a[q] = ld(ux, jc, k0 - 3 + q, oi);
        b[q] = ld(uy, jc, k0 - 3 + q, oi);
        c[q] = ld(uz, jc, k0 - 3 + q, oi);
      }
      T wl[3], el[3];               // planes k0-1 .. k0+1
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        wl[q] = ld(uz, jm, k0 - 1 + q, oi);
        el[q] = ld(uz, jc, k0 - 1 + q, oe);
        p[q + 1] = ld(pr, jc, k0 - 2 + q, oi);
        vp[q + 1] = ld(uy, jp, k0 - 2 + q, oi);
        eu[q + 1] = ld(ux, jc, k0 - 2 + q, oe);
      }
      // every column holds its values one slot up: the first step shifts
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        u[q + 1] = a[q + 1];
        v[q + 1] = b[q + 1];
        w[q + 1] = c[q + 1];
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        zu[q + 1] = i4(a[q], a[q + 1], a[q + 2], a[q + 3]);
        zv[q + 1] = i4(b[q], b[q + 1], b[q + 2], b[q + 3]);
        za[q + 1] = i4(c[q], c[q + 1], c[q + 2], c[q + 3]);
        yw[q + 1] = IY1 * wl[q] + IY2 * c[q + 2];
        put(RW2, c[q + 2], el[q]);
        fence();
        xw[q + 1] = ixb_of(RW2);
        fence();
      }
      wm[1] = wl[1];
      wm[2] = wl[2];
      ew[1] = el[1];
      ew[2] = el[2];
    }

    Next n;
    fetch(k0, n);
    for (int k = k0; k < k1; ++k) {
      // the arriving planes
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        u[q] = u[q + 1];
        v[q] = v[q + 1];
        w[q] = w[q + 1];
      }
      u[5] = n.u3;
      v[5] = n.v3;
      w[5] = n.w3;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        zu[q] = zu[q + 1];
        zv[q] = zv[q + 1];
        xw[q] = xw[q + 1];
        yw[q] = yw[q + 1];
        za[q] = za[q + 1];
        p[q] = p[q + 1];
        vp[q] = vp[q + 1];
        eu[q] = eu[q + 1];
      }
      p[3] = n.p1;
      vp[3] = n.vp1;
      eu[3] = n.eu1;
      wm[0] = wm[1]; wm[1] = wm[2]; wm[2] = n.wm2;
      ew[0] = ew[1]; ew[1] = ew[2]; ew[2] = n.ew2;
      zu[3] = i4(u[2], u[3], u[4], u[5]);
      zv[3] = i4(v[2], v[3], v[4], v[5]);
      za[3] = i4(w[2], w[3], w[4], w[5]);
      yw[3] = IY1 * wm[2] + IY2 * w[4];
      const T uc = u[2], vc = v[2], wc = w[2], pc = p[2];
      put(RU, uc, eu[2]);
      put(RV, vc, n.ev);
      put(RW, wc, ew[0]);
      put(RP, pc, n.ep);
      put(RVP, vp[2], n.evp);
      put(RUM, n.um, n.eum);
      put(RIZ, zu[1], i4(eu[0], eu[1], eu[2], eu[3]));
      put(RW2, w[4], ew[2]);
      const T um = n.um, up = n.up, vm = n.vm, wp = n.wp, pm = n.pm;
      const T hxo = n.hx, hyo = n.hy, hzo = n.hz;
      fence();
      // past the run's last plane this reads (periodic) planes it drops
      fetch(k + 1, n);
      fence();
      const T* U = row[RU] + e;
      const T* V = row[RV] + e;
      const T* W = row[RW] + e;
      const T* P = row[RP] + e;
      const T* UM = row[RUM] + e;
      const T* IZ = row[RIZ] + e;
      xw[3] = ixb_of(RW2);
      auto sto = [&](T* f, T val) {
        if (live) *(T*)((char*)(f + ((long long)nx * jc + g.plane * k)) + oi) = val;
      };
      // The three components one after the other: moved together, their LDS
      // operands do not fit the registers.
      // ---- RhsX ----
      {
        const T u3m = U[-3], u2m = U[-2], u1m = U[-1], u1p = U[1], u2p = U[2], u3p = U[3];
        const T vxc = ixb_of(RV);
        const T uxhyc = IY1 * um + IY2 * uc;
        const T uxhyp = IY3 * uc + IY4 * up;
        const T as = i4(u3m, u2m, u1m, uc), am = i4(u2m, u1m, uc, u1p);
        const T ac = i4(u1m, uc, u1p, u2p), ap = i4(uc, u1p, u2p, u3p);
        const T h11 = dx1 * as * (as + ucrf) - dx3 * am * (am + ucrf) + dx3 * ac * (ac + ucrf) -
                      dx1 * ap * (ap + ucrf);
        const T uyhx_p = (jp == nyp) ? T(0) : ixb_of(RVP);
        const T h12 = (uyhx_p * uxhyp - vxc * uxhyc) * sucaj;
        const T h13 = dz1 * zu[0] * xw[0] - dz3 * zu[1] * xw[1] + dz3 * zu[2] * xw[2] -
                      dz1 * zu[3] * xw[3];
        const T d11 = d5x(u2m, u1m, uc, u1p, u2p);
        const T d22 = ap2c * up + ac2c * uc + am2c * um;
        const T d33 = d5z(u);
        const T dcq13 = d11 + d33;
        if (want_flow && live) fix_add(s3, (double)(dcq13 + d22) * dy);
        const T conv = -h11 - h12 - h13 + cf.xnu * dcq13 + cf.gx;
        const T gradp = dx1 * P[-2] - dx3 * P[-1] + dx3 * pc - dx1 * P[1];
        sto(rx, cf.pmGamma * conv + cf.pmTheta * hxo - cf.pmAlpha * gradp + T(2) * cf.pmBeta * d22);
        sto(hx, conv);
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- RhsY ----
      {
        const T v3m = V[-3], v2m = V[-2], v1m = V[-1], v1p = V[1], v2p = V[2], v3p = V[3];
        const T vxc = i4(v2m, v1m, vc, v1p);
        const T uxhym = IY1 * UM[-1] + IY2 * U[-1] + ucrf;
        const T uxhyc = IY1 * um + IY2 * uc + ucrf;
        const T uxhyp = IY1 * UM[1] + IY2 * U[1] + ucrf;
        const T uxhyu = IY1 * UM[2] + IY2 * U[2] + ucrf;
        const T h21 = dx1 * i4(v3m, v2m, v1m, vc) * uxhym - dx3 * vxc * uxhyc +
                      dx3 * i4(v1m, vc, v1p, v2p) * uxhyp - dx1 * i4(vc, v1p, v2p, v3p) * uxhyu;
        const T vpc = vp[2];
        const T h22 = ((vpc + vc) * (vpc + vc) - (vc + vm) * (vc + vm)) * qsucac;
        const T h23 = dz1 * zv[0] * yw[0] - dz3 * zv[1] * yw[1] + dz3 * zv[2] * yw[2] -
                      dz1 * zv[3] * yw[3];
        const T d11 = d5x(v2m, v1m, vc, v1p, v2p);
        const T d22 = ap2p * vpc + ac2p * vc + am2p * vm;
        const T d33 = d5z(v);
        const T dcq13 = d11 + d33;
        const T conv = -h21 - h22 - h23 + cf.xnu * dcq13 + cf.gy;
        const T gradp = (pc - pm) * sucac;
        sto(ry, cf.pmGamma * conv + cf.pmTheta * hyo - cf.pmAlpha * gradp + T(2) * cf.pmBeta * d22);
        sto(hy, conv);
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- RhsZ ----
      {
        const T zvp = (jp == nyp) ? T(0) : i4(vp[0], vp[1], vp[2], vp[3]);
        const T w3m = W[-3], w2m = W[-2], w1m = W[-1], w1p = W[1], w2p = W[2], w3p = W[3];
        const T uzhyc = IY1 * wm[0] + IY2 * wc;
        const T uzhyp = IY3 * wc + IY4 * wp;
        const T h31 = dx1 * i4(w3m, w2m, w1m, wc) * (IZ[-1] + ucrf) -
                      dx3 * xw[1] * (zu[1] + ucrf) +
                      dx3 * i4(w1m, wc, w1p, w2p) * (IZ[1] + ucrf) -
                      dx1 * i4(wc, w1p, w2p, w3p) * (IZ[2] + ucrf);
        const T h32 = (zvp * uzhyp - zv[1] * uzhyc) * sucaj;
        const T h33 = dz1 * za[0] * za[0] - dz3 * za[1] * za[1] + dz3 * za[2] * za[2] -
                      dz1 * za[3] * za[3];
        const T d11 = d5x(w2m, w1m, wc, w1p, w2p);
        const T d22 = ap2c * wp + ac2c * wc + am2c * wm[0];
        const T d33 = d5z(w);
        const T dcq13 = d11 + d33;
        const T conv = -h31 - h32 - h33 + cf.xnu * dcq13 + cf.gz;
        const T gradp = dz1 * p[0] - dz3 * p[1] + dz3 * pc - dz1 * p[3];
        sto(rz, cf.pmGamma * conv + cf.pmTheta * hzo - cf.pmAlpha * gradp + T(2) * cf.pmBeta * d22);
        sto(hz, conv);
      }
      fence();
    }
  }
  if (want_flow) {
    block_fix4(s3, shf);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
      if (want_flow == 2) {
        bulk_add(sc, s3);
      } else {
        long long* pf = (long long*)partials + 4LL * blockIdx.x;
        for (int q = 0; q < 4; ++q) pf[q] = s3[q];
      }
    }
  }
}

// constant flow rate of the 4th-order code (m_TScheme.f90:392-407):
// dpmdxns = xnu * s3tot1 / (nxc*nzc) / yly, dp1ns = pmAlpha * dpmdxns,
// PrGradAver += dpmdxns * pmAlphaC (reset by PMcoeUpdate at ns=1).
// One workgroup, fixed summation order.
__global__ void k_flow4_finalize(const double* __restrict__ partials, int n, DevScalars* sc,
                                 double xnu, double nxnz, double yly, double alpha, double alphaC,
                                 int reset_aver) {
  __shared__ long long sh[4][1024];
  const int t = threadIdx.x;
  const long long* pf = (const long long*)partials;
  long long a[4] = {0, 0, 0, 0};
  for (int q = t; q < n; q += blockDim.x)
    for (int l = 0; l < 4; ++l) a[l] += pf[4LL * q + l];
  for (int l = 0; l < 4; ++l) sh[l][t] = a[l];
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (t < w)
      for (int l = 0; l < 4; ++l) sh[l][t] += sh[l][t + w];
    __syncthreads();
  }
  if (t == 0) {
    const long long tot[4] = {sh[0][0], sh[1][0], sh[2][0], sh[3][0]};
    const double s3tot1 = fix_value(tot);
    const double dpmdxns = xnu * s3tot1 / nxnz / yly;
    sc->dpmdxns = dpmdxns;
    sc->PrGradNow = dpmdxns;
    sc->dp1ns = alpha * dpmdxns;
    const double aver = reset_aver ? 0.0 : sc->PrGradAver;
    sc->PrGradAver = aver + dpmdxns * alphaC;
  }
}

template <typename T>
__global__ void k_sub_dp1ns(Geom g, T* __restrict__ f, const DevScalars* sc) {
  CELL4_BLOCK(K4CH);
  if (i >= g.nx || jc > g.ny) return;
  const T d = (T)sc->dp1ns;
  for (int k = k0; k < k1; ++k) {
    const long long c = fidx(g, i, jc, k);
    f[c] = f[c] - d;
  }
}

// ---------------------------------------------------------------------------
// clcPrSrc (m_TScheme.f90:114-143) and CheckDivergence (m_Tools.f90:54-81):
// div = Dx4 ux + (uy(j+1)-uy(j)) rdyp + Dz4 uz; WRITE stores prsrc = div/pmAlpha
// ---------------------------------------------------------------------------
// MAXTO: the workgroups raise the slots of `word` instead of writing partials.  WALLS: uy on
// the walls is vym / vyp whatever its rows hold (the substep's
// SetBC_and_UpdateHaloForPrSrc).
template <typename T, bool WRITE, bool MAXTO, bool WALLS>
__global__ __launch_bounds__(B4X* B4Y) void k_div4(Geom g, Metrics<T> m, Coef4<T> cf, T sudtal,
                                                   T vym, T vyp, DevScalars* sc, int word,
                                                   const T* __restrict__ ux_, const T* __restrict__ uy_,
                                                   const T* __restrict__ uz_, T* __restrict__ prsrc,
                                                   double* __restrict__ partials) {
  __shared__ double sh[8];
  CELL4_BLOCK(4 * K4CH);
  double dm = 0.0;
  if (i < g.nx && jc <= g.ny) {
    const View<T> ux{ux_, g.nx, g.nz, g.plane}, uy{uy_, g.nx, g.nz, g.plane};
    const View<T> uz{uz_, g.nx, g.nz, g.plane};
    const T sucaj = m.rdyp[jc];
    for (int k = k0; k < k1; ++k) {
      const T dudx = cf.dx1 * ux(i - 1, jc, k) + cf.dx2 * ux(i, jc, k) + cf.dx3 * ux(i + 1, jc, k) +
                     cf.dx4 * ux(i + 2, jc, k);
      T v0 = uy(i, jc, k), v1 = uy(i, jc + 1, k);
      if (WALLS) {
        v0 = jc == 1 ? vym : v0;
        v1 = jc == g.ny ? vyp : v1;
      }
      const T dvdy = (v1 - v0) * sucaj;
      const T dwdz = cf.dz1 * uz(i, jc, k - 1) + cf.dz2 * uz(i, jc, k) + cf.dz3 * uz(i, jc, k + 1) +
                     cf.dz4 * uz(i, jc, k + 2);
      const T rdiv = dudx + dvdy + dwdz;
      dm = fmax(dm, (double)fabs(rdiv));
      if (WRITE) prsrc[fidx(g, i, jc, k)] = sudtal * rdiv;
    }
  }
  const double r = block_max4(dm, sh);
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    if (MAXTO) raise_max(sc, word, r);
    else partials[blockIdx.x] = r;
  }
}

__global__ void k_max4_finalize(const double* __restrict__ partials, int n, double* out,
                                DevScalars* sc, int word) {
  __shared__ double sh[1024];
  const int t = threadIdx.x;
  double s = 0.0;
  for (int q = t; q < n; q += blockDim.x) s = fmax(s, partials[q]);
  sh[t] = s;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (t < w) sh[t] = fmax(sh[t], sh[t + w]);
    __syncthreads();
  }
  if (t == 0) {
    *out = sh[0];
    drop_max(sc, word);
  }
}

// ---------------------------------------------------------------------------
// FluidVelUpdate (m_TScheme.f90:148-173) and PressureUpdate (:590-610):
// u -= pmAlpha * grad4(phi);  p += (1 - pmBeta Lyy) phi.  With GHOST the
// Neumann ghosts of SetBC_and_UpdateHalo_pr (phi(0)=phi(1),
// phi(nyp)=phi(nyc)) are applied on the fly.
// ---------------------------------------------------------------------------
// WALLS: the ghosts that SetBC_and_UpdateHalo (4th, m_BC_and_Halo.f90:51-96) and
// SetBC_and_UpdateHalo_pr would set, written by rows 1 and ny from their new
// values instead of by two more launches.
struct WallBC4 {
  int channel;                       // 1: FT_CH, 0: FT_HC
  double uxm, uzm, uxp, uyp, uzp;    // wall values (ym / yp)
};

template <typename T, bool VEL, bool PRS, bool GHOST, bool WALLS = false>
__global__ __launch_bounds__(B4X* B4Y) void k_proj4(Geom g, Metrics<T> m, Coef4<T> cf, T alpha,
                                                    T beta, WallBC4 wb,
                                                    const T* __restrict__ phi_,
                                                    T* __restrict__ ux, T* __restrict__ uy,
                                                    T* __restrict__ uz, T* __restrict__ pr) {
  CELL4_BLOCK(K4CH);
  if (i >= g.nx || jc > g.ny) return;
  const View<T> ph{phi_, g.nx, g.nz, g.plane};
  const T sucac = m.rdyc[jc];
  const T pmBetap = -beta * m.ap2Pr[jc];
  const T pmBetac = -beta * m.ac2Pr[jc] + T(1);
  const T pmBetam = -beta * m.am2Pr[jc];
  for (int k = k0; k < k1; ++k) {
    const long long c = fidx(g, i, jc, k);
    const T pc = ph(i, jc, k);
    const T pm = (GHOST && jc == 1) ? pc : ph(i, jc - 1, k);
    if (VEL) {
      const T dpdx = cf.dx1 * ph(i - 2, jc, k) + cf.dx2 * ph(i - 1, jc, k) + cf.dx3 * pc +
                     cf.dx4 * ph(i + 1, jc, k);
      const T dpdy = (pc - pm) * sucac;
      const T dpdz = cf.dz1 * ph(i, jc, k - 2) + cf.dz2 * ph(i, jc, k - 1) + cf.dz3 * pc +
                     cf.dz4 * ph(i, jc, k + 1);
      const T un = ux[c] - alpha * dpdx, wn = uz[c] - alpha * dpdz;
      T vn = uy[c] - alpha * dpdy;
      if (WALLS && jc == g.ny) {
        const long long t = c + g.nx;
        ux[t] = wb.channel ? (T)wb.uxp * T(2) - un : un;
        uy[t] = wb.channel ? (T)wb.uyp : T(0);
        uz[t] = wb.channel ? (T)wb.uzp * T(2) - wn : wn;
      }
      if (WALLS && jc == 1) {
        ux[c - g.nx] = (T)wb.uxm * T(2) - un;
        vn = T(0);  // uy_ym of the 4th-order code
        uz[c - g.nx] = (T)wb.uzm * T(2) - wn;
      }
      ux[c] = un;
      uy[c] = vn;
      uz[c] = wn;
    }
    if (PRS) {
      const T pp = (GHOST && jc == g.ny) ? pc : ph(i, jc + 1, k);
      const T pn = pr[c] + pmBetap * pp + pmBetac * pc + pmBetam * pm;
      if (WALLS && jc == 1) pr[c - g.nx] = pn;
      if (WALLS && jc == g.ny) pr[c + g.nx] = pn;
      pr[c] = pn;
    }
  }
}

// ---------------------------------------------------------------------------
// Wall ghosts of the 4th-order code, m_BC_and_Halo.f90 (4th): full=1
// SetBC_and_UpdateHalo (:51-96), full=0 SetBC_and_UpdateHaloForPrSrc
// (:101-134).  Channel (no-slip top) or half channel (free-slip top).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_bc4_vel(Geom g, WallBC4 b, T* __restrict__ ux, T* __restrict__ uy,
                          T* __restrict__ uz, const T* __restrict__ uy_ym, int full) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  if (i >= g.nx || k >= g.nz) return;
  const int ny = g.ny, nyp = ny + 1;
  const T v_ym = uy_ym[i + (long long)g.nx * k];
  if (!full) {
    uy[fidx(g, i, nyp, k)] = b.channel ? (T)b.uyp : T(0);
    uy[fidx(g, i, 1, k)] = v_ym;
    return;
  }
  if (b.channel) {
    ux[fidx(g, i, nyp, k)] = (T)b.uxp * T(2) - ux[fidx(g, i, ny, k)];
    uy[fidx(g, i, nyp, k)] = (T)b.uyp;
    uz[fidx(g, i, nyp, k)] = (T)b.uzp * T(2) - uz[fidx(g, i, ny, k)];
  } else {
    ux[fidx(g, i, nyp, k)] = ux[fidx(g, i, ny, k)];
    uy[fidx(g, i, nyp, k)] = T(0);
    uz[fidx(g, i, nyp, k)] = uz[fidx(g, i, ny, k)];
  }
  ux[fidx(g, i, 0, k)] = (T)b.uxm * T(2) - ux[fidx(g, i, 1, k)];
  uy[fidx(g, i, 1, k)] = v_ym;
  uz[fidx(g, i, 0, k)] = (T)b.uzm * T(2) - uz[fidx(g, i, 1, k)];
}

// ===========================================================================
// launchers
// ===========================================================================
template <typename T>
Coef4<T> make_coef4(const c3d_ctx* c) {
  Coef4<T> f;
  f.dx1 = (T)c->dxc[0]; f.dx2 = (T)c->dxc[1]; f.dx3 = (T)c->dxc[2]; f.dx4 = (T)c->dxc[3];
  f.dz1 = (T)c->dzc[0]; f.dz2 = (T)c->dzc[1]; f.dz3 = (T)c->dzc[2]; f.dz4 = (T)c->dzc[3];
  f.dxx1 = (T)c->dxxc[0]; f.dxx2 = (T)c->dxxc[1]; f.dxx3 = (T)c->dxxc[2];
  f.dxx4 = (T)c->dxxc[3]; f.dxx5 = (T)c->dxxc[4];
  f.dzz1 = (T)c->dzzc[0]; f.dzz2 = (T)c->dzzc[1]; f.dzz3 = (T)c->dzzc[2];
  f.dzz4 = (T)c->dzzc[3]; f.dzz5 = (T)c->dzzc[4];
  f.ic1 = (T)c->icoe[0]; f.ic2 = (T)c->icoe[1]; f.ic3 = (T)c->icoe[2]; f.ic4 = (T)c->icoe[3];
  f.ucrf = (T)c->p.u_crf;
  f.xnu = (T)c->p.xnu;
  f.gx = (T)c->p.gravity[0]; f.gy = (T)c->p.gravity[1]; f.gz = (T)c->p.gravity[2];
  f.pmGamma = (T)c->pmGamma; f.pmTheta = (T)c->pmTheta;
  f.pmAlpha = (T)c->pmAlpha; f.pmBeta = (T)c->pmBeta;
  return f;
}
template Coef4<double> make_coef4<double>(const c3d_ctx*);
template Coef4<float> make_coef4<float>(const c3d_ctx*);

template <typename T>
static const Metrics<T>& mets4(const c3d_ctx* c);
template <>
const Metrics<double>& mets4<double>(const c3d_ctx* c) { return c->md; }
template <>
const Metrics<float>& mets4<float>(const c3d_ctx* c) { return c->mf; }

static inline int nblocks4(const Geom& g, int kch) {
  return ((g.nx + B4X - 1) / B4X) * ((g.ny + B4Y - 1) / B4Y) * ((g.nz + kch - 1) / kch);
}

template <typename T>
static int rhs4_t(c3d_ctx* c, const void* ux, const void* uy, const void* uz, const void* pr,
                  void* rx, void* ry, void* rz, void* hx, void* hy, void* hz, int want_flow) {
  const Geom& g = c->g;
  const int kc = march_kchunk((long long)((g.nx + B4X - 1) / B4X) * ((g.ny + B4Y - 1) / B4Y * B4Y),
                              g.nz, 4);
  const int nb = nblocks4(g, kc);
  if (want_flow == 1 && 4 * nb > c->max_partials) {
    set_error("rhs4: partial buffer too small");
    return C3D_ERR_ARG;
  }
  hipLaunchKernelGGL((k_rhs4<T>), dim3(nb), dim3(B4X, B4Y), 0, c->stream, g, mets4<T>(c),
                     make_coef4<T>(c), (const double*)c->d_dyp, (const T*)ux, (const T*)uy,
                     (const T*)uz, (const T*)pr, (T*)rx, (T*)ry, (T*)rz, (T*)hx, (T*)hy, (T*)hz,
                     c->d_partials, c->d_sc, want_flow, kc);
  C3D_HIP(hipGetLastError());
  if (want_flow == 1) {
    hipLaunchKernelGGL(k_flow4_finalize, dim3(1), dim3(1024), 0, c->stream, c->d_partials, nb,
                       c->d_sc, c->p.xnu, (double)(g.nx * g.nz), c->p.yly, c->pmAlpha, c->pmAlphaC,
                       c->cur_ns == 1);
    C3D_HIP(hipGetLastError());
  }
  return C3D_OK;
}

int launch_rhs4(c3d_ctx* c, const void* ux, const void* uy, const void* uz, const void* pr,
                void* rx, void* ry, void* rz, void* hx, void* hy, void* hz, int want_flow) {
  hipEvent_t ev;
  prof_begin(c, ST_RHS, &ev);
  int rc = c->prec == C3D_FP64 ? rhs4_t<double>(c, ux, uy, uz, pr, rx, ry, rz, hx, hy, hz, want_flow)
                               : rhs4_t<float>(c, ux, uy, uz, pr, rx, ry, rz, hx, hy, hz, want_flow);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  prof_end(c, ST_RHS, ev, 13.0 * N * c->esize);
  return C3D_OK;
}

int launch_sub_dp1ns(c3d_ctx* c, void* rx) {
  const Geom& g = c->g;
  const dim3 grid(nblocks4(g, K4CH));
  if (c->prec == C3D_FP64)
    hipLaunchKernelGGL(k_sub_dp1ns<double>, grid, dim3(B4X, B4Y), 0, c->stream, g, (double*)rx,
                       (const DevScalars*)c->d_sc);
  else
    hipLaunchKernelGGL(k_sub_dp1ns<float>, grid, dim3(B4X, B4Y), 0, c->stream, g, (float*)rx,
                       (const DevScalars*)c->d_sc);
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

// word: the slots that max |div| goes to (raise), or whose plain field it goes to
template <typename T, bool WRITE, bool WALLS>
static int div4_t(c3d_ctx* c, const void* ux, const void* uy, const void* uz, void* prsrc,
                  T sudtal, int word, bool raise) {
  const Geom& g = c->g;
  const int nb = nblocks4(g, 4 * K4CH);
  if (!raise && nb > c->max_partials) {
    set_error("div4: partial buffer too small");
    return C3D_ERR_ARG;
  }
  const T vyp = (T)(c->p.bc[3] == C3D_BC_NOSLIP ? c->p.uybc[3] : 0.0);
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(nb), dim3(B4X, B4Y), 0, c->stream, g, mets4<T>(c),
                       make_coef4<T>(c), sudtal, T(0), vyp, c->d_sc, word, (const T*)ux, (const T*)uy,
                       (const T*)uz, (T*)prsrc, c->d_partials);
  };
  if (raise) {
    launch(k_div4<T, WRITE, true, WALLS>);
    C3D_HIP(hipGetLastError());
    return C3D_OK;
  }
  launch(k_div4<T, WRITE, false, WALLS>);
  C3D_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_max4_finalize, dim3(1), dim3(1024), 0, c->stream, c->d_partials, nb,
                     word == RED_DIV1 ? &c->d_sc->divmax1 : &c->d_sc->divmax2, c->d_sc, word);
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

int launch_prsrc4(c3d_ctx* c, const void* ux, const void* uy, const void* uz, void* prsrc,
                  double alpha_override, bool walls) {
  hipEvent_t ev;
  prof_begin(c, ST_PRSRC, &ev);
  const double alpha = alpha_override > 0.0 ? alpha_override : c->pmAlpha;
  const int out = RED_DIV1;
  int rc;
  if (c->prec == C3D_FP64)
    rc = walls ? div4_t<double, true, true>(c, ux, uy, uz, prsrc, 1.0 / alpha, out, true)
               : div4_t<double, true, false>(c, ux, uy, uz, prsrc, 1.0 / alpha, out, false);
  else
    rc = walls ? div4_t<float, true, true>(c, ux, uy, uz, prsrc, (float)(1.0 / alpha), out, true)
               : div4_t<float, true, false>(c, ux, uy, uz, prsrc, (float)(1.0 / alpha), out, false);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  prof_end(c, ST_PRSRC, ev, 4.0 * N * c->esize);
  return C3D_OK;
}

int launch_div4(c3d_ctx* c, const void* ux, const void* uy, const void* uz, bool closing) {
  hipEvent_t ev;
  prof_begin(c, ST_DIAG, &ev);
  const int out = RED_DIV2;
  int rc = c->prec == C3D_FP64
               ? div4_t<double, false, false>(c, ux, uy, uz, nullptr, 0.0, out, closing)
               : div4_t<float, false, false>(c, ux, uy, uz, nullptr, 0.f, out, closing);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  prof_end(c, ST_DIAG, ev, 3.0 * N * c->esize);
  return C3D_OK;
}

static WallBC4 make_wallbc4(const c3d_ctx* c) {
  WallBC4 b;
  b.channel = c->p.bc[3] == C3D_BC_NOSLIP ? 1 : 0;
  b.uxm = c->p.uxbc[2];
  b.uzm = c->p.uzbc[2];
  b.uxp = c->p.uxbc[3];
  b.uyp = c->p.uybc[3];
  b.uzp = c->p.uzbc[3];
  return b;
}

template <typename T>
static int proj4_t(c3d_ctx* c, const void* phi, void* ux, void* uy, void* uz, void* pr, int vel,
                   int prs, int ghost, bool walls) {
  const Geom& g = c->g;
  const WallBC4 wb = make_wallbc4(c);
  const dim3 grid(nblocks4(g, K4CH)), blk(B4X, B4Y);
  const T alpha = (T)c->pmAlpha, beta = (T)c->pmBeta;
  const Coef4<T> cf = make_coef4<T>(c);
#define PROJ4(V, P, G)                                                                          \
  hipLaunchKernelGGL((k_proj4<T, V, P, G>), grid, blk, 0, c->stream, g, mets4<T>(c), cf, alpha, \
                     beta, wb, (const T*)phi, (T*)ux, (T*)uy, (T*)uz, (T*)pr)
  if (walls) {
    hipLaunchKernelGGL((k_proj4<T, true, true, true, true>), grid, blk, 0, c->stream, g,
                       mets4<T>(c), cf, alpha, beta, wb, (const T*)phi, (T*)ux, (T*)uy, (T*)uz,
                       (T*)pr);
  } else if (vel && prs) {
    if (ghost) PROJ4(true, true, true); else PROJ4(true, true, false);
  } else if (vel) {
    if (ghost) PROJ4(true, false, true); else PROJ4(true, false, false);
  } else {
    if (ghost) PROJ4(false, true, true); else PROJ4(false, true, false);
  }
#undef PROJ4
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

static int proj4(c3d_ctx* c, const void* phi, void* ux, void* uy, void* uz, void* pr, int do_vel,
                 int do_pr, int ghost_from_interior, bool walls) {
  if (!do_vel && !do_pr) return C3D_OK;
  const int st = (do_vel && do_pr) ? ST_PROJ : do_vel ? ST_VELUPD : ST_PRUPD;
  hipEvent_t ev;
  prof_begin(c, st, &ev);
  int rc = c->prec == C3D_FP64
               ? proj4_t<double>(c, phi, ux, uy, uz, pr, do_vel, do_pr, ghost_from_interior, walls)
               : proj4_t<float>(c, phi, ux, uy, uz, pr, do_vel, do_pr, ghost_from_interior, walls);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz;
  const double words = (do_vel && do_pr) ? 9.0 : do_vel ? 7.0 : 3.0;
  prof_end(c, st, ev, words * N * c->esize);
  return C3D_OK;
}

int launch_proj4(c3d_ctx* c, const void* phi, void* ux, void* uy, void* uz, void* pr, int do_vel,
                 int do_pr, int ghost_from_interior) {
  return proj4(c, phi, ux, uy, uz, pr, do_vel, do_pr, ghost_from_interior, false);
}

int launch_proj4_walls(c3d_ctx* c, const void* phi, void* ux, void* uy, void* uz, void* pr) {
  return proj4(c, phi, ux, uy, uz, pr, 1, 1, 1, true);
}

int launch_bc4_vel(c3d_ctx* c, void* ux, void* uy, void* uz, const void* uy_ym, int full) {
  const Geom& g = c->g;
  const WallBC4 b = make_wallbc4(c);
  hipEvent_t ev;
  prof_begin(c, ST_BC, &ev);
  const dim3 grid((g.nx + 255) / 256, g.nz), blk(256);
  if (c->prec == C3D_FP64)
    hipLaunchKernelGGL(k_bc4_vel<double>, grid, blk, 0, c->stream, g, b, (double*)ux, (double*)uy,
                       (double*)uz, (const double*)uy_ym, full);
  else
    hipLaunchKernelGGL(k_bc4_vel<float>, grid, blk, 0, c->stream, g, b, (float*)ux, (float*)uy,
                       (float*)uz, (const float*)uy_ym, full);
  C3D_HIP(hipGetLastError());
  prof_end(c, ST_BC, ev, 0.0);
  return C3D_OK;
}

}  // namespace c3d
