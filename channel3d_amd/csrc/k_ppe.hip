// Wall-normal tridiagonal solves of the pressure Poisson equation in
// (kx, kz) space and the PPE driver, clcPPE_x1 (m_Poisson.f90:567-688).
//
// For every (kx, kz) the reference solves, with InverseTridiagonal
// (m_Tools.f90:218-245), a = am2Pr(j), c = ap2Pr(j),
// b = ac2Pr(j) + WaveNumX + WaveNumZ; the (0,0) mode has its first row
// replaced by phi = 0 (the gauge, :627-648).  The complex half spectrum
// stores the real and imaginary parts of a mode side by side; both share
// the coefficients (as the reference's half-complex storage does), so one
// thread runs the elimination once for the two right-hand sides.  Threads
// own consecutive kx, so every access of a sweep is coalesced.
#include "c3d_internal.h"

#include <type_traits>

namespace c3d {

template <typename T>
struct CT2;
template <>
struct CT2<double> { using t = double2; };
template <>
struct CT2<float> { using t = float2; };

// Lines (kx, kz) are numbered kx + (nk+1) kz and dealt to consecutive
// threads, so only the last workgroup has idle threads.  nk+1 is one more
// than a power of two or a multiple of 64 on most grids: with 64 threads per
// kz row, a row's last wavefront held one live thread (512x256x512: 320
// threads for 257 lines).  The two-lane sweep of 192x128x160 (97 lines a row)
// took 0.051 ms instead of 0.064 for it.
struct Line {
  int kx, kz;
};
__device__ __forceinline__ Line line_of(const Geom& g, long long l) {
  Line r;
  r.kz = (int)(l / (g.nk + 1));
  r.kx = (int)(l - (long long)(g.nk + 1) * r.kz);
  return r;
}

// The rows of the wall-normal operator and the wavenumber terms, as restrict
// arguments of their own: a sweep's row coefficients are the same for every
// lane, and the compiler loads them through the scalar unit only where no
// store can alias them.  As vector loads (from a struct of pointers) they
// queue behind the prefetched segment, and waiting for one drains it.
#define PprRows(T)                                                                      \
  const T *__restrict__ am, const T *__restrict__ ac, const T *__restrict__ ap,         \
      const T *__restrict__ wx, const T *__restrict__ wz
#define PPR_OF(m) (m).am2Pr, (m).ac2Pr, (m).ap2Pr, (m).wavex, (m).wavez

template <typename T>
__device__ __forceinline__ void k_tridiag_body(const Geom& g, PprRows(T),
                                               typename CT2<T>::t* __restrict__ spec,
                                               T* __restrict__ sarr, Line ln) {
  using T2 = typename CT2<T>::t;
  const int kx = ln.kx, kz = ln.kz;
  if (kz >= g.nz) return;
  const int ny = g.ny;
  const long long P = g.P;
  const long long base = kx + P * (long long)ny * kz;
  const T lx = wx[kx], lz = wz[kz];
  const bool pin = (kx == 0 && kz == 0);
  // row j = 1
  T vecm = pin ? T(1) : (ac[1] + lx) + lz;
  T rv = quot_recip(vecm);
  T cprev = pin ? T(0) : ap[1];
  // register rings keep the next PD rows of each sweep in flight; the main
  // loops carry no conditionals so the loads stay outstanding across steps
  constexpr int PD = 8;
  T2 buf[PD];
#pragma unroll
  for (int q = 0; q < PD; ++q) buf[q] = spec[base + P * min(1 + q, ny - 1)];
  T2 f = spec[base];
  if (pin) {
    f.x = 0;
    f.y = 0;
  }
  f.x = quot(f.x, vecm, rv);
  f.y = quot(f.y, vecm, rv);
  spec[base] = f;
  auto fwd = [&](int j0, T2 fj) {
    const int jr = j0 + 1;
    const T arr = quot(cprev, vecm, rv);
    const T a = am[jr];
    vecm = ((ac[jr] + lx) + lz) - a * arr;
    rv = quot_recip(vecm);
    f.x = quot(fj.x - a * f.x, vecm, rv);
    f.y = quot(fj.y - a * f.y, vecm, rv);
    sarr[base + P * j0] = arr;
    cprev = ap[jr];
  };
  int jb = 1;
  for (; jb + 2 * PD <= ny - 1; jb += PD) {
#pragma unroll
    for (int q = 0; q < PD; ++q) {
      const int j0 = jb + q;
      const T2 fj = buf[q];
      buf[q] = spec[base + P * (j0 + PD)];
      fwd(j0, fj);
      spec[base + P * j0] = f;
    }
  }
#pragma unroll
  for (int q = 0; q < PD; ++q) {
    const int j0 = jb + q;
    if (j0 < ny) {
      fwd(j0, buf[q]);
      spec[base + P * j0] = f;
    }
  }
  for (int j0 = jb + PD; j0 < ny; ++j0) {
    fwd(j0, spec[base + P * j0]);
    spec[base + P * j0] = f;
  }
  T2 fb[PD];
  T ab[PD];
#pragma unroll
  for (int q = 0; q < PD; ++q) {
    const int jn = max(ny - 2 - q, 0);
    fb[q] = spec[base + P * jn];
    ab[q] = sarr[base + P * (jn + 1)];
  }
  jb = ny - 2;
  for (; jb - 2 * PD + 1 >= 0; jb -= PD) {
#pragma unroll
    for (int q = 0; q < PD; ++q) {
      const int j0 = jb - q;
      const T2 fj = fb[q];
      const T arr1 = ab[q];
      fb[q] = spec[base + P * (j0 - PD)];
      ab[q] = sarr[base + P * (j0 - PD + 1)];
      f.x = fj.x - arr1 * f.x;
      f.y = fj.y - arr1 * f.y;
      spec[base + P * j0] = f;
    }
  }
#pragma unroll
  for (int q = 0; q < PD; ++q) {
    const int j0 = jb - q;
    if (j0 >= 0) {
      f.x = fb[q].x - ab[q] * f.x;
      f.y = fb[q].y - ab[q] * f.y;
      spec[base + P * j0] = f;
    }
  }
  for (int j0 = jb - PD; j0 >= 0; --j0) {
    const T arr1 = sarr[base + P * (j0 + 1)];
    const T2 fj = spec[base + P * j0];
    f.x = fj.x - arr1 * f.x;
    f.y = fj.y - arr1 * f.y;
    spec[base + P * j0] = f;
  }
}

// ---------------------------------------------------------------------------
// The same elimination without storing the factors and the forward pass.
// The line is cut into segments of C rows.  The forward pass keeps, per
// segment end, the running value f and pivot vecm (three reals per line and
// segment, in the spectral scratch array).  The backward pass walks the
// segments from the top: it reruns the segment's forward recurrence from
// its checkpoint -- the same operations on the same operands, hence the same
// pivots, factors and values -- then substitutes backward and stores the
// solution.  The top segment's values are still in registers.  Traffic per
// complex element: read, read again, write (48 B in FP64) instead of 80 B;
// results equal k_tridiag's bit for bit.
// ---------------------------------------------------------------------------
template <typename T, int C, bool NTS = false>
__device__ __forceinline__ void k_tridiag_ck_body(const Geom& g, PprRows(T),
                                                  typename CT2<T>::t* __restrict__ spec,
                                                  T* __restrict__ ckp, Line ln) {
  using T2 = typename CT2<T>::t;
  const int kx = ln.kx, kz = ln.kz;
  if (kz >= g.nz) return;
  const int ny = g.ny;
  const int nseg = (ny + C - 1) / C;
  const long long P = g.P;
  const long long base = kx + P * (long long)ny * kz;
  const long long cs = P * (long long)g.nz;             // checkpoint plane stride
  T* ck = ckp + kx + P * (long long)kz;
  const T lx = wx[kx], lz = wz[kz];
  const bool pin = (kx == 0 && kz == 0);
  using Gd = std::true_type;   // the top segment: rows past the last one
  using Un = std::false_type;  // the others, without the row guard
  T2 y[C];
  T ar[C];
  T vecm = T(1), rv = T(1), cprev = T(0);  // rv: 1/vecm
  T2 f;
  f.x = 0;
  f.y = 0;
  auto load = [&](int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
#pragma unroll
    for (int q = 0; q < C; ++q)
      if (!G || s * C + q < ny) y[q] = spec[base + P * (s * C + q)];
  };
  // one segment's forward recurrence from (f, vecm, rv, cprev).  Row 1 has
  // nothing below: f = 0, vecm = 1 and cprev = 0 give its pivot and value.
  auto run = [&](int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j0 = s * C + q;
      if (!G || j0 < ny) {
        const int jr = j0 + 1;
        const T arr = quot(cprev, vecm, rv);
        const T a = am[jr];
        T2 fj = y[q];
        T cj = ap[jr];
        vecm = ((ac[jr] + lx) + lz) - a * arr;
        if (q == 0 && s == 0 && pin) {  // the gauge row
          vecm = T(1);
          fj.x = fj.y = cj = T(0);
        }
        rv = quot_recip(vecm);
        f.x = quot(fj.x - a * f.x, vecm, rv);
        f.y = quot(fj.y - a * f.y, vecm, rv);
        cprev = cj;
        ar[q] = arr;
        y[q] = f;
      }
    }
  };
  // backward through segment s (forward values in y)
  T2 x;
  T arnext = T(0);
  auto back = [&](int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
#pragma unroll
    for (int q = C - 1; q >= 0; --q) {
      const int j0 = s * C + q;
      if (!G || j0 < ny) {
        if (!G || j0 < ny - 1) {
          const T a1 = q + 1 < C ? ar[q + 1] : arnext;
          x.x = y[q].x - a1 * x.x;
          x.y = y[q].y - a1 * x.y;
        }
        C3D_ST_ONCE(x.x, &spec[base + P * j0].x);  // written once
        C3D_ST_ONCE(x.y, &spec[base + P * j0].y);
      }
    }
    arnext = ar[0];
  };
  const int top = nseg - 1;
  for (int s = 0; s < top; ++s) {
    load(s, Un{});
    run(s, Un{});
    ck[cs * (3 * s + 0)] = f.x;
    ck[cs * (3 * s + 1)] = f.y;
    ck[cs * (3 * s + 2)] = vecm;
  }
  load(top, Gd{});
  run(top, Gd{});
  x = f;
  back(top, Gd{});
  for (int s = top - 1; s >= 0; --s) {
    f.x = f.y = T(0);
    vecm = rv = T(1);
    cprev = T(0);
    if (s > 0) {
      f.x = ck[cs * (3 * (s - 1) + 0)];
      f.y = ck[cs * (3 * (s - 1) + 1)];
      vecm = ck[cs * (3 * (s - 1) + 2)];
      cprev = ap[s * C];
    }
    load(s, Un{});
    __builtin_amdgcn_sched_barrier(0);
    if (s > 0) rv = quot_recip(vecm);
    run(s, Un{});
    back(s, Un{});
  }
}

// The same elimination with the real and imaginary parts of a wavenumber
// pair on two neighbouring lanes (lane 2n the real part, 2n+1 the
// imaginary part), both computing the shared pivots -- the same operations,
// so the same values -- and with each segment's right-hand side loaded one
// segment ahead.  Half the registers per lane of k_tridiag_ck_body: twice the
// wavefronts on grids with few lines, room for the prefetch and for longer
// segments on large ones.  The three quotients by a pivot share its
// reciprocal.  Before (vector loads of the row coefficients, a guard around
// every row, divisions; one lane on large grids) and now, FP64: four
// 512x256x512 fields 1.640 -> 1.241 ms, 768x384x576 0.986 -> 0.903 ms,
// 192x128x160 0.051 -> 0.040 ms, 96x96x72 0.031 -> 0.025 ms, 64^3 0.023 ->
// 0.017 ms.
// Only the top segment has rows past ny, so only its loads and stores carry
// the row guard (a guarded access is a branch of its own, and the compiler
// then waits for every outstanding load, the prefetched segment included).
template <typename T, int C, bool NTS = false>
__device__ __forceinline__ void k_tridiag_ck2_body(const Geom& g, PprRows(T),
                                                   typename CT2<T>::t* __restrict__ spec,
                                                   T* __restrict__ ckp, Line ln) {
  const int part = threadIdx.x & 1;  // 0: real, 1: imaginary part
  const int kx = ln.kx, kz = ln.kz;
  if (kz >= g.nz) return;
  const int ny = g.ny;
  const int nseg = (ny + C - 1) / C, top = nseg - 1;
  const long long P = g.P;
  // this lane's component of row j: sp[P2 * j]
  T* sp = (T*)spec + 2 * (kx + P * (long long)ny * kz) + part;
  const long long P2 = 2 * P;
  const long long cs = P * (long long)g.nz;  // checkpoint plane stride
  T* ck = ckp + kx + P * (long long)kz;
  const T lx = wx[kx], lz = wz[kz];
  const bool pin = (kx == 0 && kz == 0);
  using Gd = std::true_type;
  using Un = std::false_type;
  auto load = [&](T* y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
    const int lo = s * C;
#pragma unroll
    for (int q = 0; q < C; ++q)
      if (!G || lo + q < ny) y[q] = sp[P2 * (lo + q)];
  };
  T ar[C];
  T vecm = T(1), rv = T(1), cprev = T(0), f = T(0);  // rv: 1/vecm
  // one segment's forward recurrence from (f, vecm, rv, cprev).  Row 1 has
  // nothing below: f = 0, vecm = 1 and cprev = 0 give its pivot and value.
  auto run = [&](T* y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
    const int lo = s * C;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j0 = lo + q;
      if (!G || j0 < ny) {
        const int jr = j0 + 1;
        const T arr = quot(cprev, vecm, rv);
        const T a = am[jr];
        T fj = y[q], cj = ap[jr];
        vecm = ((ac[jr] + lx) + lz) - a * arr;
        if (q == 0 && s == 0 && pin) {  // the gauge row
          vecm = T(1);
          fj = cj = T(0);
        }
        rv = quot_recip(vecm);
        f = quot(fj - a * f, vecm, rv);
        cprev = cj;
        ar[q] = arr;
        y[q] = f;
      }
    }
  };
  auto save = [&](int s) {  // checkpoint at the end of segment s
    ck[cs * (3 * s + part)] = f;
    ck[cs * (3 * s + 2)] = vecm;  // both lanes hold the same pivot
  };
  T x = T(0), arnext = T(0);
  // backward substitution through segment s (forward values in y)
  auto back = [&](const T* y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
    const int lo = s * C;
#pragma unroll
    for (int q = C - 1; q >= 0; --q) {
      const int j0 = lo + q;
      if (!G || j0 < ny) {
        if (!G || j0 < ny - 1) {
          const T a1 = q + 1 < C ? ar[q + 1] : arnext;
          x = y[q] - a1 * x;
        }
        C3D_ST_ONCE(x, &sp[P2 * j0]);  // written once
      }
    }
    arnext = ar[0];
  };
  T ya[C], yb[C];
  // forward: the segments below the top in pairs, each load a segment ahead
  if (top == 0) {
    load(ya, 0, Gd{});
    run(ya, 0, Gd{});
  } else {
    load(ya, 0, Un{});
    int s = 0;
    for (; s + 2 < top; s += 2) {
      load(yb, s + 1, Un{});
      __builtin_amdgcn_sched_barrier(0);
      run(ya, s, Un{});
      save(s);
      load(ya, s + 2, Un{});
      __builtin_amdgcn_sched_barrier(0);
      run(yb, s + 1, Un{});
      save(s + 1);
    }
    if (s + 1 < top) {
      load(yb, s + 1, Un{});
      __builtin_amdgcn_sched_barrier(0);
      run(ya, s, Un{});
      save(s);
      load(ya, top, Gd{});
      __builtin_amdgcn_sched_barrier(0);
      run(yb, s + 1, Un{});
      save(s + 1);
      run(ya, top, Gd{});
    } else {
      load(yb, top, Gd{});
      __builtin_amdgcn_sched_barrier(0);
      run(ya, s, Un{});
      save(s);
      run(yb, top, Gd{});
#pragma unroll
      for (int q = 0; q < C; ++q) ya[q] = yb[q];
    }
  }
  // backward; ya and ar hold the top segment
  x = f;
  if (top > 0) load(yb, top - 1, Un{});
  __builtin_amdgcn_sched_barrier(0);
  back(ya, top, Gd{});
  for (int s = top - 1; s >= 0; --s) {
    // yb holds segment s as stored; its checkpoint is requested before the
    // segment below, which goes into ya
    f = T(0);
    vecm = rv = T(1);
    cprev = T(0);
    if (s > 0) {
      f = ck[cs * (3 * (s - 1) + part)];
      vecm = ck[cs * (3 * (s - 1) + 2)];
      load(ya, s - 1, Un{});
      __builtin_amdgcn_sched_barrier(0);
      rv = quot_recip(vecm);
      cprev = ap[s * C];
    }
    run(yb, s, Un{});
    back(yb, s, Un{});
#pragma unroll
    for (int q = 0; q < C; ++q) yb[q] = ya[q];
  }
}

template <typename T, int C, bool NTS = false>
__global__ __launch_bounds__(256) void k_tridiag_ck2(Geom g, PprRows(T),
                                                     typename CT2<T>::t* __restrict__ spec,
                                                     T* __restrict__ ckp, long long bsp,
                                                     long long bck) {
  k_tridiag_ck2_body<T, C, NTS>(g, am, ac, ap, wx, wz, spec + bsp * blockIdx.y, ckp + bck * blockIdx.y,
                                line_of(g, ((long long)blockIdx.x * blockDim.x + threadIdx.x) >> 1));
}

// The two-lane sweep with a line's forward values and factors kept in LDS (96
// reals per row of a wavefront's 32 pairs) instead of checkpoints: the backward
// pass substitutes at once where it otherwise runs each segment's elimination a
// second time.  The same operations on the same operands, so the same values.
// For grids with one or two wavefronts per CU: there the serial chain, not
// traffic, is the time (64^3 19.4 -> 14.8 us, 96x96x72 24.9 -> 19.0, 150x101x108
// 28.8 -> 22.6).  With more lines than that a second round of workgroups costs as
// much as the first, and the checkpointed form holds more wavefronts.  PER:
// workgroups that share a CU's LDS.
template <typename T, int PER>
constexpr int tri_lds_rows() {
  return 159744 / (96 * PER * (int)sizeof(T));
}

template <typename T, int PER, bool NTS>
__global__ __launch_bounds__(64) void k_tridiag_lds(Geom g, PprRows(T),
                                                    typename CT2<T>::t* __restrict__ spec,
                                                    long long bsp) {
  constexpr int C = 16;
  __shared__ T sf[tri_lds_rows<T, PER>() * 64];  // forward values of a lane
  __shared__ T sa[tri_lds_rows<T, PER>() * 32];  // factors, one for a pair's two lanes
  const int lane = threadIdx.x, part = lane & 1, pair = lane >> 1;
  const Line ln = line_of(g, ((long long)blockIdx.x * 64 + lane) >> 1);
  const int kx = ln.kx, kz = ln.kz;
  if (kz >= g.nz) return;  // no barrier below: a lane reads what it wrote
  const int ny = g.ny, top = (ny + C - 1) / C - 1;
  const long long P2 = 2LL * g.P;
  T* sp = (T*)(spec + bsp * blockIdx.y) + 2 * (kx + (long long)g.P * ny * kz) + part;
  const T lx = wx[kx], lz = wz[kz];
  const bool pin = (kx == 0 && kz == 0);
  using Gd = std::true_type;  // the top segment: rows past the last one
  using Un = std::false_type;
  auto load = [&](T* y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
#pragma unroll
    for (int q = 0; q < C; ++q)
      if (!G || s * C + q < ny) y[q] = sp[P2 * (s * C + q)];
  };
  // Row 1 has nothing below: f = 0, vecm = 1 and cprev = 0 give its pivot and value
  T vecm = T(1), rv = T(1), cprev = T(0), f = T(0);
  auto run = [&](const T* y, int s, auto gv) {
    constexpr bool G = decltype(gv)::value;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int j0 = s * C + q;
      if (!G || j0 < ny) {
        const int jr = j0 + 1;
        const T arr = quot(cprev, vecm, rv);
        const T a = am[jr];
        T fj = y[q], cj = ap[jr];
        vecm = ((ac[jr] + lx) + lz) - a * arr;
        if (q == 0 && s == 0 && pin) {  // the gauge row
          vecm = T(1);
          fj = cj = T(0);
        }
        rv = quot_recip(vecm);
        f = quot(fj - a * f, vecm, rv);
        cprev = cj;
        sf[j0 * 64 + lane] = f;
        sa[j0 * 32 + pair] = arr;
      }
    }
  };
  T ya[C], yb[C];
  if (top == 0) {
    load(ya, 0, Gd{});
    run(ya, 0, Gd{});
  } else {
    load(ya, 0, Un{});
    int s = 0;
    for (; s + 2 < top; s += 2) {  // each load a segment ahead
      load(yb, s + 1, Un{});
      __builtin_amdgcn_sched_barrier(0);
      run(ya, s, Un{});
      load(ya, s + 2, Un{});
      __builtin_amdgcn_sched_barrier(0);
      run(yb, s + 1, Un{});
    }
    if (s + 1 < top) {
      load(yb, s + 1, Un{});
      __builtin_amdgcn_sched_barrier(0);
      run(ya, s, Un{});
      load(ya, top, Gd{});
      __builtin_amdgcn_sched_barrier(0);
      run(yb, s + 1, Un{});
      run(ya, top, Gd{});
    } else {
      load(yb, top, Gd{});
      __builtin_amdgcn_sched_barrier(0);
      run(ya, s, Un{});
      run(yb, top, Gd{});
    }
  }
  T x = f;
  C3D_ST_ONCE(x, &sp[P2 * (ny - 1)]);
#pragma unroll 16
  for (int j0 = ny - 2; j0 >= 0; --j0) {
    x = sf[j0 * 64 + lane] - sa[(j0 + 1) * 32 + pair] * x;
    C3D_ST_ONCE(x, &sp[P2 * j0]);
  }
}

// The one-lane form, which C3D_TRIDIAG_LANES=1 selects to compare with.  At
// least 4 waves per SIMD: the FP64 body fits 128 VGPRs without spilling.
// Batches: blockIdx.y selects the field; its spectrum starts bsp complex
// elements, its checkpoints bck reals after the first field's.
template <typename T, int C, bool NTS = false>
__global__ __launch_bounds__(256, 4) void k_tridiag_ck(Geom g, PprRows(T),
                                                    typename CT2<T>::t* __restrict__ spec,
                                                    T* __restrict__ ckp, long long bsp,
                                                    long long bck) {
  k_tridiag_ck_body<T, C, NTS>(g, am, ac, ap, wx, wz, spec + bsp * blockIdx.y, ckp + bck * blockIdx.y,
                               line_of(g, (long long)blockIdx.x * 256 + threadIdx.x));
}

template <typename T>
__global__ __launch_bounds__(256) void k_tridiag_b(Geom g, PprRows(T),
                                                   typename CT2<T>::t* __restrict__ spec,
                                                   T* __restrict__ sarr, long long bsp,
                                                   long long bck) {
  k_tridiag_body<T>(g, am, ac, ap, wx, wz, spec + bsp * blockIdx.y, sarr + bck * blockIdx.y,
                    line_of(g, (long long)blockIdx.x * 256 + threadIdx.x));
}

// Rows per segment of the two-lane sweep on large grids.  A segment costs three
// checkpoint words per line, written and read (9 % of the traffic at 16 FP64
// rows), its rows the registers.  FP64 (256-thread workgroups) 16 / 20 / 24 / 32
// rows: 1.361 / 1.295 / 1.241 / 1.487 ms for four 512x256x512 fields and 1.004
// / 0.904 / 0.903 / 0.946 ms at 768x384x576; the one-lane form takes 1.58 and
// 1.08 ms on the same box.  FP32 16 / 24 / 32 / 48 rows: 0.402 / 0.387 / 0.368 /
// 0.398 ms for two 512x256x512 fields.
template <typename T>
constexpr int tri_rows() {
  return sizeof(T) == 8 ? 24 : 32;
}

template <typename T>
static int tridiag_t(c3d_ctx* c, void* spec, void* ck, const Batch& b) {
  const Geom& g = c->g;
  const long long nl = (long long)(g.nk + 1) * g.nz;  // lines of one field
  const Metrics<T>& m = *(const Metrics<T>*)(c->prec == C3D_FP64 ? (const void*)&c->md
                                                                  : (const void*)&c->mf);
  constexpr int CSEG = 16;
  auto launch = [&](auto kern, int threads, int lanes) {
    const dim3 grid((unsigned)((nl * lanes + threads - 1) / threads), b.n), blk(threads);
    hipLaunchKernelGGL(kern, grid, blk, 0, c->stream, g, PPR_OF(m), (typename CT2<T>::t*)spec,
                       (T*)ck, b.spec, b.ck);
  };
  auto launch_lds = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)((nl * 2 + 63) / 64), b.n), dim3(64), 0, c->stream, g,
                       PPR_OF(m), (typename CT2<T>::t*)spec, b.spec);
  };
  // checkpoints: 3 reals per line and segment, in the spectral scratch
  const long long need = 3LL * ((g.ny + CSEG - 1) / CSEG) * g.P * g.nz;
  if (c->ymode == YS_STORE || need > (long long)g.P * g.ny * g.nz) {
    launch(k_tridiag_b<T>, 256, 1);
  } else if (c->tri_lanes == 1) {
    if (g.nt) launch(k_tridiag_ck<T, CSEG, true>, 256, 1);
    else launch(k_tridiag_ck<T, CSEG, false>, 256, 1);
  } else if (c->tri_lanes == 0 && nl * b.n * 2 <= 512LL * 64 && g.ny <= tri_lds_rows<T, 2>()) {
    if (g.nt) launch_lds(k_tridiag_lds<T, 2, true>);
    else launch_lds(k_tridiag_lds<T, 2, false>);
  } else if (c->tri_lanes == 0 && nl * b.n * 2 <= 256LL * 64 && g.ny <= tri_lds_rows<T, 1>()) {
    if (g.nt) launch_lds(k_tridiag_lds<T, 1, true>);
    else launch_lds(k_tridiag_lds<T, 1, false>);
  } else if (nl * b.n * 2 <= 1024LL * 64) {
    // at most a wavefront per SIMD, or lines too long for LDS: the serial chains
    // bound the sweep, and single-wave workgroups of 16-row segments spread them
    // over the most CUs (192x128x160: 0.040 ms against 0.043)
    if (g.nt) launch(k_tridiag_ck2<T, CSEG, true>, 64, 2);
    else launch(k_tridiag_ck2<T, CSEG, false>, 64, 2);
  } else {
    // memory bound (384x192x288: 0.103 ms against 0.114 in FP64, 0.065 against
    // 0.073 in FP32)
    if (g.nt) launch(k_tridiag_ck2<T, tri_rows<T>(), true>, 256, 2);
    else launch(k_tridiag_ck2<T, tri_rows<T>(), false>, 256, 2);
  }
  C3D_HIP(hipGetLastError());
  return C3D_OK;
}

// ck: the checkpoint (or factor) scratch, nspec reals per field
int launch_tridiag(c3d_ctx* c, void* spec, void* ck, const Batch& b) {
  hipEvent_t ev;
  prof_begin(c, ST_TRIDIAG, &ev);
  int rc = c->prec == C3D_FP64 ? tridiag_t<double>(c, spec, ck, b) : tridiag_t<float>(c, spec, ck, b);
  if (rc) return rc;
  const double N = (double)c->g.nx * c->g.ny * c->g.nz * b.n;
  prof_end(c, ST_TRIDIAG, ev, 2.0 * N * c->esize);
  return C3D_OK;
}

// ===========================================================================
// Mixed-precision solve: FP32 transforms and y solves, FP64 residual of the
// discrete operator, FP32 correction solves added to the FP64 solution.
// ===========================================================================

// The (0,0) mode in FP64: the Neumann y operator with the gauge row is the
// ill-conditioned system of the solve (its FP32 error would bound what the
// refinement can reach).  w holds 3 ny doubles, then the gauge value at
// w[3 ny]: the first row is phi(0,0,1) = w[3 ny] (0 in the first solve, as the
// reference pins it; in a correction solve, minus the current solution's
// value, so the refined solution keeps the reference's gauge -- without it
// the FP32 rounding of the first solve's plane mean at j = 1 would survive
// every sweep as a constant offset).
//
// One workgroup: its threads move the line through LDS, MCH rows at a time,
// and lanes 0 and 1 run the recurrence of the real and the imaginary part from
// there; the pivots and factors of the line (fac: vecm[ny], arr[ny]) do not
// depend on the data and come from the host, formed with the same operations.
// As one thread's loop over global memory (two dependent loads and three
// divisions per row) this line bounded the
// kernel: 0.60 ms for two 512x256x512 fields, 0.48 ms from LDS, where the
// other lines' one-lane sweep bounds it (0.37 ms with the two-lane sweep).
constexpr int MCH = 256;

template <typename T2>
__device__ void mean_mode_fp64(const Geom& g, const Metrics<double>& m,
                               const double* __restrict__ fac, T2* spec, double* w) {
  __shared__ double sv[2][MCH], sa[MCH], sd[MCH];
  const int ny = g.ny, t = threadIdx.x;
  const long long P = g.P;
  double f = 0.0;
  for (int c0 = 0; c0 < ny; c0 += MCH) {
    const int n = min(MCH, ny - c0);
    __syncthreads();
    if (t < n) {
      const T2 v = spec[P * (c0 + t)];
      sv[0][t] = c0 + t == 0 ? w[3 * ny] : (double)v.x;  // row 0: the gauge row
      sv[1][t] = c0 + t == 0 ? 0.0 : (double)v.y;
      sa[t] = c0 + t == 0 ? 0.0 : m.am2Pr[c0 + t + 1];
      sd[t] = fac[c0 + t];
    }
    __syncthreads();
    if (t < 2) {
      int r = 0;
      if (c0 == 0) {
        f = sv[t][0];
        r = 1;
      }
#pragma unroll 8
      for (; r < n; ++r) {
        f = (sv[t][r] - sa[r] * f) / sd[r];
        sv[t][r] = f;
      }
    }
    __syncthreads();
    if (t < n) {
      w[c0 + t] = sv[0][t];
      w[ny + c0 + t] = sv[1][t];
    }
  }
  // backward: x_j = w_j - arr_{j+1} x_{j+1}, the last row's f is x
  for (int c0 = (ny - 1) / MCH * MCH; c0 >= 0; c0 -= MCH) {
    const int n = min(MCH, ny - c0);
    __syncthreads();
    if (t < n) {
      sv[0][t] = w[c0 + t];
      sv[1][t] = w[ny + c0 + t];
      sa[t] = c0 + t + 1 < ny ? fac[ny + c0 + t + 1] : 0.0;
    }
    __syncthreads();
    if (t < 2) {
      int r = n - 1;
      if (c0 + r == ny - 1) --r;  // already f
#pragma unroll 8
      for (; r >= 0; --r) {
        f = sv[t][r] - sa[r] * f;
        sv[t][r] = f;
      }
    }
    __syncthreads();
    if (t < n) {
      T2 o;
      o.x = sv[0][t];
      o.y = sv[1][t];
      spec[P * (c0 + t)] = o;
    }
  }
}

// Workgroup 0 of a field solves the (0,0) mode, the others every other line
// by the checkpointed elimination.
template <typename T, int C>
__global__ __launch_bounds__(256) void k_tridiag_mixed(Geom g, PprRows(T), Metrics<double> md,
                                                       const double* __restrict__ fac,
                                                       typename CT2<T>::t* __restrict__ spec,
                                                       T* __restrict__ ckp, double* w,
                                                       long long bsp, long long bck,
                                                       long long bw) {
  spec += bsp * blockIdx.y;
  if (blockIdx.x == 0) {
    mean_mode_fp64(g, md, fac, spec, w + bw * blockIdx.y);
    return;
  }
  const long long l = ((long long)(blockIdx.x - 1) * 256 + threadIdx.x) >> 1;
  if (l == 0) return;
  k_tridiag_ck2_body<T, C>(g, am, ac, ap, wx, wz, spec, ckp + bck * blockIdx.y, line_of(g, l));
}

// r = f - L phi in FP64, L the discrete operator the spectral solve inverts:
// 3-point x and z second differences and the Neumann y operator am2Pr/ac2Pr/
// ap2Pr (whose wall entries are zero, so wall ghosts are never read)
//
// A wavefront owns 64 x cells of PR rows and marches a chunk of kchunk z
// planes: phi is loaded once per plane (its rows, one row on either side, and
// the two x cells beside them), the planes below and above are the lane's own
// registers, the x neighbours come from the lanes beside it by DPP, and plane
// k+2 is requested before plane k is computed.  Bound: HBM, 20 B per cell.
// The form it replaced (one plane per workgroup, seven phi loads per cell,
// workgroups of one plane spread over the XCDs, so each L2 fetched every plane
// three times) took 0.984 ms for two 512x256x512 fields, this one 0.556 ms
// (4.8 TB/s; a plain copy reaches 4.8-6.0 TB/s).
//
// The wavefronts holding the plane j = 1 also write the sum of phi over
// their 64 x-points to part[k * gxb + x tile] (the gauge).
// blockIdx.x = the tile (x fastest, then y, z chunk, field), XCD-remapped;
// batches: fields bf reals apart, partial sums bpart doubles apart.
constexpr int PR = 4;

template <typename TR, bool NTS>
__global__ __launch_bounds__(256) void k_ppe_resid(Geom g, Metrics<double> m, double rdx2,
                                                   double rdz2, const double* __restrict__ f,
                                                   const double* __restrict__ phi,
                                                   TR* __restrict__ r, double* __restrict__ part,
                                                   long long bf, long long bpart, int kchunk) {
  const int gxb = (g.nx + 63) / 64, gyb = (g.ny + 4 * PR - 1) / (4 * PR);
  const int nch = (g.nz + kchunk - 1) / kchunk;
  int lb = xcd_remap(blockIdx.x, gridDim.x);
  const int bx = lb % gxb, i0 = bx * 64;
  lb /= gxb;
  const int j0 = ((lb % gyb) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.y)) * PR + 1;
  lb /= gyb;
  const int k0 = (lb % nch) * kchunk, q = lb / nch;
  if (j0 > g.ny) return;
  const int k1 = min(g.nz, k0 + kchunk);
  f += bf * q;
  phi += bf * q;
  r += bf * q;
  part += bpart * q;
  const int lane = threadIdx.x, last = min(63, g.nx - 1 - i0);
  const int i = min(i0 + lane, g.nx - 1);
  const bool live = lane <= last;
  const int ie = lane == last ? (i0 + last == g.nx - 1 ? 0 : i0 + last + 1)
                              : (i0 == 0 ? g.nx - 1 : i0 - 1);
  const int nx = g.nx, ny = g.ny;
  struct Plane {  // rows j0-1 .. j0+PR (past the top ghost: the ghost again)
    double c[PR + 2], e[PR], f[PR];
  };
  auto fetch = [&](int k, Plane& a) {
    const double* p = phi + g.plane * k;
    const double* pf = f + g.plane * k;
#pragma unroll
    for (int t = 0; t < PR + 2; ++t) a.c[t] = p[(long long)nx * min(j0 - 1 + t, ny + 1) + i];
#pragma unroll
    for (int t = 0; t < PR; ++t) {
      const long long row = (long long)nx * min(j0 + t, ny);
      a.e[t] = p[row + ie];
      a.f[t] = C3D_LD_ONCE(&pf[row + i]);  // read once
    }
  };
  auto step = [&](int k, const double* dn, const Plane& a, const Plane& up) {
    if (j0 == 1) {
      double v = live ? a.c[1] : 0.0;
      for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
      if (lane == 0) part[(long long)k * gxb + bx] = v;
    }
#pragma unroll
    for (int t = 0; t < PR; ++t) {
      const int j = j0 + t;
      if (j <= ny) {
        const double pc = a.c[t + 1];
        const double xm = row_prev(pc, a.e[t]), xp = row_next(pc, a.e[t], lane, last);
        double lap = (xp - 2.0 * pc + xm) * rdx2 + (up.c[t + 1] - 2.0 * pc + dn[t]) * rdz2 +
                     m.ac2Pr[j] * pc;
        if (j > 1) lap += m.am2Pr[j] * a.c[t];
        if (j < ny) lap += m.ap2Pr[j] * a.c[t + 2];
        if (live) r[(long long)nx * j + g.plane * k + i] = (TR)(a.f[t] - lap);
      }
    }
  };
  // past the chunk's last plane (k1) the prefetch repeats it
  auto wrapk = [&](int k) { return min(k, k1) == g.nz ? 0 : min(k, k1); };
  double dn[PR];
  {
    const double* p = phi + g.plane * (k0 == 0 ? g.nz - 1 : k0 - 1);
#pragma unroll
    for (int t = 0; t < PR; ++t) dn[t] = p[(long long)nx * min(j0 + t, ny) + i];
  }
  auto roll = [&](const Plane& a) {
#pragma unroll
    for (int t = 0; t < PR; ++t) dn[t] = a.c[t + 1];
  };
  Plane a, b, c;
  fetch(k0, a);
  fetch(wrapk(k0 + 1), b);
  for (int k = k0; k < k1; k += 3) {
    fetch(wrapk(k + 2), c);
    step(k, dn, a, b);
    roll(a);
    if (k + 1 < k1) {
      fetch(wrapk(k + 3), a);
      step(k + 1, dn, b, c);
      roll(b);
    }
    if (k + 2 < k1) {
      fetch(wrapk(k + 4), b);
      step(k + 2, dn, c, a);
      roll(c);
    }
  }
}

// w[3 ny] = -(sum of the partials, in index order): the gauge value of the
// next correction solve; 0 resets it to the reference's pin.  One workgroup
// per field of a batch (w and part bw doubles apart).
__global__ void k_gauge(const double* __restrict__ part, int n, double* w, int ny, int reset,
                        long long bw) {
  __shared__ double sh[256];
  const int t = threadIdx.x;
  part += bw * blockIdx.x;
  w += bw * blockIdx.x;
  double a = 0.0;
  for (int q = t; q < n; q += 256) a += part[q];
  sh[t] = a;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) sh[t] += sh[t + h];
    __syncthreads();
  }
  if (t == 0) w[3 * ny] = reset ? 0.0 : -sh[0];
}

// The mixed-precision solve of a batch of sources (one field: the default
// batch on the context's own scratch).  spec: FP32 spectra (b.spec32 apart),
// ck: FP32 checkpoints, w: (0,0)-mode work and gauge partials (b.mean apart),
// resid: FP32 residual fields (b.field apart).
static int ppe_mixed(c3d_ctx* c, const void* prsrc, void* phi, int sweeps, void* spec, void* ck,
                     double* w, float* resid, const Batch& b) {
  int rc = ensure_mixed_tables(c);
  if (rc) return rc;
  const Geom& g = c->g;
  auto solve32 = [&]() -> int {
    int r;
    if ((r = launch_fft32(c, FFT32_Z_FWD, nullptr, spec, nullptr, 0, b))) return r;
    hipEvent_t ev;
    prof_begin(c, ST_TRIDIAG, &ev);
    const long long nl = (long long)(g.nk + 1) * g.nz;
    const dim3 grid((unsigned)(1 + (2 * nl + 255) / 256), b.n), blk(256);
    hipLaunchKernelGGL((k_tridiag_mixed<float, tri_rows<float>()>), grid, blk, 0, c->stream,
                       g, PPR_OF(c->mf), c->md, c->d_meanfac, (float2*)spec, (float*)ck, w,
                       b.spec32, b.ck, b.mean);
    C3D_HIP(hipGetLastError());
    prof_end(c, ST_TRIDIAG, ev, 2.0 * (double)g.nx * g.ny * g.nz * b.n * 4);
    return launch_fft32(c, FFT32_Z_INV, nullptr, spec, nullptr, 0, b);
  };
  double* gpart = w + 3 * ((size_t)g.ny + 1);
  const int ngp = ((g.nx + 63) / 64) * g.nz;
  hipLaunchKernelGGL(k_gauge, dim3(b.n), dim3(256), 0, c->stream, gpart, 0, w, g.ny, 1, b.mean);
  C3D_HIP(hipGetLastError());
  if ((rc = launch_fft32(c, FFT32_X_FWD_F64, prsrc, spec, nullptr, 0, b))) return rc;
  if ((rc = solve32())) return rc;
  if ((rc = launch_fft32(c, FFT32_X_INV_SET, nullptr, spec, (double*)phi, c->normfft, b)))
    return rc;
  for (int s = 0; s < sweeps; ++s) {
    hipEvent_t ev;
    prof_begin(c, ST_RESID, &ev);
    const int tiles = ((g.nx + 63) / 64) * ((g.ny + 4 * PR - 1) / (4 * PR));
    const int kch = resid_kchunk(g, tiles, b.n);
    const dim3 grid(tiles * ((g.nz + kch - 1) / kch) * b.n), blk(64, 4);
    if (g.nt)
      hipLaunchKernelGGL((k_ppe_resid<float, true>), grid, blk, 0, c->stream, g, c->md, c->rdx2,
                         c->rdz2, (const double*)prsrc, (const double*)phi, resid, gpart, b.field,
                         b.mean, kch);
    else
      hipLaunchKernelGGL((k_ppe_resid<float, false>), grid, blk, 0, c->stream, g, c->md, c->rdx2,
                         c->rdz2, (const double*)prsrc, (const double*)phi, resid, gpart, b.field,
                         b.mean, kch);
    C3D_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_gauge, dim3(b.n), dim3(256), 0, c->stream, gpart, ngp, w, g.ny, 0,
                       b.mean);
    C3D_HIP(hipGetLastError());
    prof_end(c, ST_RESID, ev, (double)g.nx * g.ny * g.nz * b.n * (8 + 8 + 4));
    if ((rc = launch_fft32(c, FFT32_X_FWD_F32, resid, spec, nullptr, 0, b))) return rc;
    if ((rc = solve32())) return rc;
    if ((rc = launch_fft32(c, FFT32_X_INV_ADD, nullptr, spec, (double*)phi, c->normfft, b)))
      return rc;
  }
  return C3D_OK;
}

static int run_ppe_mixed(c3d_ctx* c, void* prsrc, void* phi, int sweeps) {
  int rc = ensure_mixed_tables(c);
  if (!rc) rc = ensure_resid32(c);
  if (rc) return rc;
  // the FP64 spectral array holds the FP32 spectrum
  return ppe_mixed(c, prsrc, phi, sweeps, c->spec, c->sarr, c->d_mean64, c->resid32, Batch());
}

// clcPPE_x1: forward x, forward z, y solves, inverse z, inverse x * normfft.
// prsrc is read only (the reference overwrites it with unscaled phi; callers
// of this library never read it back).
int run_ppe(c3d_ctx* c, void* prsrc, void* phi) {
  int rc;
  if (c->ppe_sweeps >= 0) return run_ppe_mixed(c, prsrc, phi, c->ppe_sweeps);
  if ((rc = launch_fft_x_fwd(c, prsrc, c->spec))) return rc;
  return run_ppe_from_spectrum(c, phi);
}

int run_ppe_from_spectrum(c3d_ctx* c, void* phi) {
  int rc;
  if ((rc = launch_fft_z(c, c->spec, 0))) return rc;
  if ((rc = launch_tridiag(c, c->spec, c->sarr))) return rc;
  if ((rc = launch_fft_z(c, c->spec, 1))) return rc;
  return launch_fft_x_inv(c, c->spec, phi, c->normfft);
}

// A batch of pressure solves: every pass one launch over the whole batch.
// sweeps < 0: the FP64 solve (the kernels of the single solve, so each
// field's result equals c3d_ppe's bit for bit); sweeps >= 0: the
// mixed-precision solve with that many refinement sweeps.
int ppe_batch_ws(c3d_ctx* c, int nb, const void* prsrc, void* phi, int sweeps,
                 const BatchWork& ws) {
  int rc;
  const Geom& g = c->g;
  Batch b;
  b.n = nb;
  b.field = g.nfield;
  b.spec = g.nspec;
  b.spec32 = g.nspec;      // FP32 spectra packed in the FP64 batch array
  b.ck = g.nspec;
  b.mean = batch_mean_len(g);
  if (sweeps >= 0)
    return ppe_mixed(c, prsrc, phi, sweeps, ws.spec, ws.ck, ws.mean, ws.resid, b);
  if ((rc = launch_fft_x_fwd(c, prsrc, ws.spec, b))) return rc;
  if ((rc = launch_fft_z(c, ws.spec, 0, b))) return rc;
  if ((rc = launch_tridiag(c, ws.spec, ws.ck, b))) return rc;
  if ((rc = launch_fft_z(c, ws.spec, 1, b))) return rc;
  return launch_fft_x_inv(c, ws.spec, phi, c->normfft, b);
}

int run_ppe_batch(c3d_ctx* c, int nb, const void* prsrc, void* phi, int sweeps) {
  int rc;
  if ((rc = ensure_batch(c, nb, sweeps >= 0))) return rc;
  BatchWork ws;
  ws.spec = c->bspec;
  ws.ck = c->bsarr;
  ws.mean = c->bmean;
  ws.resid = (float*)c->bres;
  return ppe_batch_ws(c, nb, prsrc, phi, sweeps, ws);
}

}  // namespace c3d
