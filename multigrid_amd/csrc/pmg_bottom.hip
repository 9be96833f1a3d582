// pmg_bottom.hip -- the two coarsest levels of a V-cycle (pmgc/mgcsd.cc:
// 325-473 between entering and leaving the second coarsest level).
//
// A level of a few thousand points gives the chip a microsecond of work per
// sweep, and every launch costs three to five: as separate launches the
// level takes two per sweep, one each for the residual, the restriction, the
// product of the damping factor and the prolongation.  Here one workgroup
// does the level's way down (k_bottom_down) and another its way up
// (k_bottom_up), with the iterate in LDS and workgroup barriers for kernel
// boundaries; the operator streams from the L2 once per sweep with the
// two-element loads of g27_couplings, issued before the barrier their values
// do not depend on.  It also leaves the other compute units to other
// requests.  What bounds it: the instructions of the few wavefronts of a
// class (37 loads, 18 LDS reads, two 27-term sums each), 1.1 us per class at
// 13^3.  Measured (MI355X, two sweeps each way, down + up): 13^3 14.2 + 16.1
// us in FP32 and 14.9 + 17.8 in FP64 against about 45 as 14 launches in a
// graph (97^3 mixed request 2888 -> 2775 us, 16 mixed requests of 65^3 to
// 161^3 35.3 -> 34.7 ms); 17^3 22.9 + 24.7 in FP32, even with the launches
// alone and ahead of them under load, but 28.7 + 33.3 in FP64 and 45 + 52 at
// 21^3 against 48 and 60: so the limits of BOT_MAXN.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <type_traits>

#include "pmg_device.h"
#include "pmg_internal.h"

namespace pmg {

namespace {

// Largest level, in points (the measurements above).
template <class T>
constexpr int BOT_MAXN = sizeof(T) == 4 ? 17 * 17 * 17 : 13 * 13 * 13;
constexpr int BOT_PAD = 8;
// FP32 16 wavefronts of at most 128 registers, FP64 8 of at most 256.
template <class T>
constexpr int BOT_NT = sizeof(T) == 4 ? 1024 : 512;

template <class T>
struct Bot {
  GBottom<T> a;
  int nu, np;  // sweeps; pairs per row
};

// The pairs of the rows of a level, wavefront by wavefront: a wavefront takes
// 64 / np whole rows, lane (r, m) pair m of its row r.
struct BotLane {
  int wave, r, m, rpw;
  bool live;
  __device__ BotLane(int np) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    rpw = 64 / np;
    r = lane / np, m = lane % np;
    live = r < rpw;
  }
};

// The four values from X[p - 1 + d] on of a pair at p.
template <class T>
__device__ __forceinline__ void lds4(const T *X, int p, T (&v)[4]) {
#pragma unroll
  for (int q = 0; q < 4; q++) v[q] = X[p - 1 + q];
}
template <class T, bool PL>
__device__ __forceinline__ void lds_rows(const T *X, int p, int sy, int sz,
                                         G27X<T> &r, T (&own)[4]) {
  lds4(X, p, own);
  lds4(X, p + sy, r.xN);
  lds4(X, p - sy, r.xS);
  if constexpr (PL) {
    lds4(X, p + sz, r.xu[0]);
    lds4(X, p + sy + sz, r.xu[1]);
    lds4(X, p - sy + sz, r.xu[2]);
    lds4(X, p - sz, r.xd[0]);
    lds4(X, p + sy - sz, r.xd[1]);
    lds4(X, p - sy - sz, r.xd[2]);
  } else {
#pragma unroll
    for (int q = 0; q < 12; q++)
      r.xu[q / 4][q % 4] = r.xd[q / 4][q % 4] = (T)0;
  }
}

// Calls f(p, first) for the pairs of the rows (j, k) = (j0 + sj a, k0 + sk b),
// a < nj, b < nk, p their index; every wavefront passes one workgroup
// barrier, after `load` of its first task and before `work` of it.
template <class T, class LoadF, class WorkF>
__device__ __forceinline__ void bot_rows(const BotLane &L, int shift, int nx,
                                         int ny, int j0, int sj, int nj, int k0,
                                         int sk, int nk, LoadF load,
                                         WorkF work) {
  constexpr int NW = BOT_NT<T> / 64;
  const int rows = nj * nk, tasks = (rows + L.rpw - 1) / L.rpw;
  bool waited = false;
  int w = L.wave + shift;
  if (w >= NW) w -= NW;
  for (int t = w; t < tasks; t += NW) {
    const int row = t * L.rpw + L.r;
    const bool ok = L.live && row < rows;
    const int q = ok ? row : 0;
    const int j = j0 + sj * (q % nj), k = k0 + sk * (q / nj);
    const int i = 2 + 2 * (ok ? L.m : 0);
    const int p = ((k - 1) * ny + (j - 1)) * nx + i - 1;
    load(p);
    if (!waited) {
      __syncthreads();
      waited = true;
    }
    work(p, ok, i + 1 <= nx - 1);
  }
  if (!waited) __syncthreads();
}

// One 8-colour sweep (Vgsrb27x, gsd.cc:160-211) on X in LDS: the four row
// classes with a barrier before each, the two colours of a row between
// adjacent lanes, as gs27_row.  zero: X is zero (the couplings to planes that
// are still zero in the first two classes are not read).
template <class T, int ADJ, bool PL>
__device__ __forceinline__ void bot_class(const GBottom<T> &a,
                                          const BotLane &L, int np, int cls,
                                          int shift, T *X) {
  const int nx = a.d.nx, ny = a.d.ny, nz = a.d.nz;
  const int sy = nx, sz = nx * ny;
  const size_t n = (size_t)sz * nz;
  const int pz = cls >> 1, py = cls & 1;
  G27C<T> c;
  T f[2];
  bot_rows<T>(
      L, shift, nx, ny, 2 + py, 2, count_parity(ny, py), 2 + pz, 2,
      count_parity(nz, pz),
      [&](int p) {
        const unsigned off = (unsigned)p * (unsigned)sizeof(T);
        g27_couplings<PL>(a.ac, a.cc, n, sy, sz, off, c);
        ldn(lane_at(a.f, 0, off), f);
      },
      [&](int p, bool ok, bool both) {
        G27X<T> x;
        T own[4];
        lds_rows<T, PL>(X, p, sy, sz, x, own);
        const G27Part<T> g0 = g27_part<T, 0>(c, x, false),
                         g1 = g27_part<T, 1>(c, x, false);
        auto fin = [&](const G27Part<T> &g, T rhs, T xw, T xe) -> T {
          return (rhs + ((g27_plane(g, xw, xe) + g.u) + g.dd)) / g.dg;
        };
        T n0 = own[1], n1 = own[2];
        if (ADJ == 0) {
          n0 = fin(g0, f[0], own[0], own[2]);
          const T e = __shfl_down(n0, 1, 64);
          const T v = fin(g1, f[1], n0, L.m + 1 < np ? e : own[3]);
          n1 = both ? v : n1;
        } else {
          const T v = fin(g1, f[1], own[1], own[3]);
          n1 = both ? v : n1;
          const T w = __shfl_up(n1, 1, 64);
          n0 = fin(g0, f[0], L.m > 0 ? w : own[0], n1);
        }
        if (ok) {
          X[p] = n0;
          if (both) X[p + 1] = n1;
        }
      });
}
template <class T, int ADJ>
__device__ __forceinline__ void bot_sweeps(const GBottom<T> &a,
                                           const BotLane &L, int np, int nu,
                                           bool zero, T *X) {
  constexpr int HALF = BOT_NT<T> / 128;
#pragma unroll 1
  for (int it = 0; it < nu; it++) {
#pragma unroll 1
    for (int ph = 0; ph < 4; ph++) {
      const int cls = ADJ ? 3 - ph : ph;
      // alternate halves of the wavefronts start with the rows of
      // successive classes: a half that is idle in one class loads for the
      // next meanwhile
      if (zero && it == 0 && ph < 2)
        bot_class<T, ADJ, false>(a, L, np, cls, (ph & 1) * HALF, X);
      else
        bot_class<T, ADJ, true>(a, L, np, cls, (ph & 1) * HALF, X);
    }
  }
}

template <class T>
__global__ __launch_bounds__(BOT_NT<T>) void k_bottom_down(
    const GTab<Bot<T>> tab) {
  __shared__ T X[BOT_MAXN<T> + BOT_PAD], R[BOT_MAXN<T> + BOT_PAD];
  const Bot<T> &b = tab.a[blockIdx.x];
  const GBottom<T> &a = b.a;
  const int nx = a.d.nx, ny = a.d.ny, nz = a.d.nz;
  const int sy = nx, sz = nx * ny, n = sz * nz, tid = threadIdx.x;
  const BotLane L(b.np);
  for (int p = tid; p < n + BOT_PAD; p += BOT_NT<T>) X[p] = (T)0;
  bot_sweeps<T, 0>(a, L, b.np, b.nu, true, X);
  {  // residual (matvecd.cc:460-528)
    G27C<T> c;
    T f[2];
    bot_rows<T>(
        L, 0, nx, ny, 2, 1, ny - 2, 2, 1, nz - 2,
        [&](int p) {
          const unsigned off = (unsigned)p * (unsigned)sizeof(T);
          g27_couplings<true>(a.ac, a.cc, (size_t)n, sy, sz, off, c);
          ldn(lane_at(a.f, 0, off), f);
        },
        [&](int p, bool ok, bool both) {
          G27X<T> x;
          T own[4];
          lds_rows<T, true>(X, p, sy, sz, x, own);
          const G27Part<T> g0 = g27_part<T, 0>(c, x, false),
                           g1 = g27_part<T, 1>(c, x, false);
          if (!ok) return;
          R[p] = (((f[0] + g27_plane(g0, own[0], own[2])) + g0.u) + g0.dd) -
                 g0.dg * own[1];
          if (both)
            R[p + 1] =
                (((f[1] + g27_plane(g1, own[1], own[3])) + g1.u) + g1.dd) -
                g1.dg * own[2];
        });
  }
  // the iterate for the way up (its boundary entries stay zero)
  for (int p = tid; p < n; p += BOT_NT<T>) a.x[p] = X[p];
  __syncthreads();
  // restriction (matvecd.cc:755-795)
  const int cx = a.dc.nx, cy = a.dc.ny, cz = a.dc.nz;
  const int ni = cx - 2, nj = cy - 2, nint = ni * nj * (cz - 2);
  const size_t nc = (size_t)cx * cy * cz;
  for (int q = tid; q < nint; q += BOT_NT<T>) {
    // separate multiplies and adds, as restrict_body: the same bits
#pragma clang fp contract(off)
    const int ii = 2 + q % ni, jj = 2 + (q / ni) % nj, kk = 2 + q / (ni * nj);
    const size_t pC = ix(cx, cy, ii, jj, kk);
    const int f = (int)ix(nx, ny, 2 * ii - 1, 2 * jj - 1, 2 * kk - 1);
    const int off[9] = {0,       sy,      -sy,    1,      -1,
                        1 + sy, -1 + sy, 1 - sy, -1 - sy};
    const int zo[3] = {0, sz, -sz};
    T w[27], t[3];
#pragma unroll
    for (int m = 0; m < 27; m++) w[m] = a.pc[(size_t)m * nc + pC];
#pragma unroll
    for (int z = 0; z < 3; z++) {
      T acc = w[9 * z] * R[f + zo[z]];
#pragma unroll
      for (int m = 1; m < 9; m++) acc += w[9 * z + m] * R[f + zo[z] + off[m]];
      t[z] = acc;
    }
    a.fc[pC] = t[0] + t[1] + t[2];
  }
}

template <class T, int ADJ>
__global__ __launch_bounds__(BOT_NT<T>) void k_bottom_up(
    const GTab<Bot<T>> tab) {
  __shared__ T X[BOT_MAXN<T> + BOT_PAD];
  __shared__ double red[2][BOT_NT<T> / 64];
  const Bot<T> &b = tab.a[blockIdx.x];
  const GBottom<T> &a = b.a;
  const int nx = a.d.nx, ny = a.d.ny, nz = a.d.nz;
  const int sy = nx, sz = nx * ny, n = sz * nz, tid = threadIdx.x;
  const BotLane L(b.np);
  const T damp = (T)*a.damp;
  for (int p = tid; p < n; p += BOT_NT<T>) X[p] = a.x[p];
  if (tid < BOT_PAD) X[n + tid] = (T)0;
  __syncthreads();
  {  // x += damp P xc on the interior (matvecd.cc:878-960, mgcsd.cc:458):
     // one coarse cell per thread, its 8 fine points
    const int cx = a.dc.nx, cy = a.dc.ny;
    const int ni = cx - 1, nj = cy - 1, ncell = ni * nj * (a.dc.nz - 1);
    const size_t nc = (size_t)cx * cy * a.dc.nz;
    for (int q = tid; q < ncell; q += BOT_NT<T>) {
      const int ii = 1 + q % ni, jj = 1 + (q / ni) % nj, kk = 1 + q / (ni * nj);
      const size_t c0 = ix(cx, cy, ii, jj, kk);
      T v[8];
      // fine point (di, dj, dk) of the cell: the corners e <= d that can
      // reach it, in the order x, y, z of the reference's sums; P plane of
      // the offset from the corner's fine point.  Multiply-adds written out
      // as interp_body's are, the first product on top of the second
#pragma unroll
      for (int d = 0; d < 8; d++) {
        const int dx = d & 1, dy = (d >> 1) & 1, dz = d >> 2;
        T acc = (T)0, w0 = (T)0, x0 = (T)0;
        int m = 0;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int ex = e & 1, ey = (e >> 1) & 1, ez = e >> 2;
          if (ex > dx || ey > dy || ez > dz) continue;
          const int ox = dx ? (ex ? -1 : 1) : 0, oy = dy ? (ey ? -1 : 1) : 0,
                    oz = dz ? (ez ? -1 : 1) : 0;
          const size_t pe = c0 + ex + (size_t)ey * cx + (size_t)ez * cx * cy;
          const T x = a.xc[pe];
          const T w = d ? a.pc[(size_t)pplane(ox, oy, oz) * nc + pe] : (T)1;
          if (m == 0)
            w0 = w, x0 = x;
          else
            acc = m == 1 ? fma(w0, x0, w * x) : fma(w, x, acc);
          m++;
        }
        if (d == 0) acc = x0;
        v[d] = acc;
      }
      const int i = 2 * ii - 1, j = 2 * jj - 1, k = 2 * kk - 1;
#pragma unroll
      for (int d = 0; d < 8; d++) {
        const int fi = i + (d & 1), fj = j + ((d >> 1) & 1), fk = k + (d >> 2);
        if (fi >= 2 && fj >= 2 && fk >= 2) {
          T &x = X[(int)ix(nx, ny, fi, fj, fk)];
          x = fma(damp, v[d], x);
        }
      }
    }
  }
  bot_sweeps<T, ADJ>(a, L, b.np, b.nu, false, X);
  // the result, and the damping factor of its prolongation (mgcsd.cc:
  // 429-452): (x . f) / (x . A x), 0 when the denominator is 0
  double a0 = 0.0, a1 = 0.0;
  {
    G27C<T> c;
    T f[2];
    bot_rows<T>(
        L, 0, nx, ny, 2, 1, ny - 2, 2, 1, nz - 2,
        [&](int p) {
          const unsigned off = (unsigned)p * (unsigned)sizeof(T);
          g27_couplings<true>(a.ac, a.cc, (size_t)n, sy, sz, off, c);
          ldn(lane_at(a.f, 0, off), f);
        },
        [&](int p, bool ok, bool both) {
          G27X<T> x;
          T own[4];
          lds_rows<T, true>(X, p, sy, sz, x, own);
          const G27Part<T> g0 = g27_part<T, 0>(c, x, false),
                           g1 = g27_part<T, 1>(c, x, false);
          const T y0 = ((-g27_plane(g0, own[0], own[2]) + -g0.u) + -g0.dd) +
                       g0.dg * own[1];
          const T y1 = ((-g27_plane(g1, own[1], own[3]) + -g1.u) + -g1.dd) +
                       g1.dg * own[2];
          if (!ok) return;
          a0 += (double)own[1] * (double)f[0];
          a1 += (double)own[1] * (double)y0;
          a.x[p] = own[1];
          if (both) {
            a0 += (double)own[2] * (double)f[1];
            a1 += (double)own[2] * (double)y1;
            a.x[p + 1] = own[2];
          }
        });
  }
  a0 = wave_sum(a0), a1 = wave_sum(a1);
  if ((tid & 63) == 0) red[0][tid >> 6] = a0, red[1][tid >> 6] = a1;
  __syncthreads();
  if (tid < 64) {
    constexpr int NW = BOT_NT<T> / 64;
    a0 = wave_sum(tid < NW ? red[0][tid] : 0.0);
    a1 = wave_sum(tid < NW ? red[1][tid] : 0.0);
    if (tid == 0) *a.damp = a1 != 0.0 ? a0 / a1 : 0.0;
  }
}

}  // namespace

// The coarsest level's CG has a damping factor to hand over, the level is
// small enough, and its rows fit a wavefront.
template <class T>
bool bottom_fits(const Dim &d, int numdia, const Dim &dc, int numdiac) {
  return numdia == 27 && cg_rows_fits(dc, numdiac) && d.nx >= 5 &&
         d.ny >= 5 && d.nz >= 5 && d.nx == 2 * dc.nx - 1 &&
         d.ny == 2 * dc.ny - 1 && d.nz == 2 * dc.nz - 1 &&
         d.n() <= (size_t)BOT_MAXN<T> && (d.nx - 1) / 2 <= 64;
}

// One workgroup per problem, in launches of at most GMAX.
template <class T, class LaunchF>
static void bottom_launch(const GBottom<T> *j, int n, int nu, LaunchF launch) {
  for (int q0 = 0; q0 < n; q0 += GMAX) {
    GTab<Bot<T>> t{};
    const int m = std::min(GMAX, n - q0);
    for (int q = 0; q < m; q++)
      t.a[q] = Bot<T>{j[q0 + q], nu, (j[q0 + q].d.nx - 1) / 2};
    launch(t, m);
  }
  if (hipGetLastError() != hipSuccess)
    fprintf(stderr, "pmg: launch of the bottom levels failed\n");
}
template <class T>
void bottom_down(const GBottom<T> *j, int n, int nu, hipStream_t s) {
  bottom_launch<T>(j, n, nu, [&](const GTab<Bot<T>> &t, int m) {
    k_bottom_down<T><<<m, BOT_NT<T>, 0, s>>>(t);
  });
}
template <class T>
void bottom_up(const GBottom<T> *j, int n, int nu, int iadjoint,
               hipStream_t s) {
  bottom_launch<T>(j, n, nu, [&](const GTab<Bot<T>> &t, int m) {
    if (iadjoint)
      k_bottom_up<T, 1><<<m, BOT_NT<T>, 0, s>>>(t);
    else
      k_bottom_up<T, 0><<<m, BOT_NT<T>, 0, s>>>(t);
  });
}
template bool bottom_fits<float>(const Dim &, int, const Dim &, int);
template bool bottom_fits<double>(const Dim &, int, const Dim &, int);
template void bottom_down<float>(const GBottom<float> *, int, int, hipStream_t);
template void bottom_down<double>(const GBottom<double> *, int, int,
                                  hipStream_t);
template void bottom_up<float>(const GBottom<float> *, int, int, int,
                               hipStream_t);
template void bottom_up<double>(const GBottom<double> *, int, int, int,
                                hipStream_t);

}  // namespace pmg
