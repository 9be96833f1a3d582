// pmg_device.h -- device code shared by the kernel files: indexing, wavefront
// sums, vector loads and the pair form of the 27-point operator; and the
// argument tables of the grouped launches.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <type_traits>
#include <vector>

#include "pmg_internal.h"

namespace pmg {

__host__ __device__ inline size_t ix(int nx, int ny, int i, int j, int k) {
  return ((size_t)(k - 1) * (size_t)ny + (size_t)(j - 1)) * (size_t)nx +
         (size_t)(i - 1);
}

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// P plane of the offset (dx, dy, dz) (pmgc/matvecd.cc:809-816)
__host__ __device__ constexpr int pplane(int dx, int dy, int dz) {
  return 9 * (dz == 0 ? 0 : (dz == 1 ? 1 : 2)) +
         (dy == -1 ? (dx == -1 ? 8 : (dx == 0 ? 2 : 7))
                   : (dy == 0 ? (dx == -1 ? 4 : (dx == 0 ? 0 : 3))
                              : (dx == -1 ? 6 : (dx == 0 ? 1 : 5))));
}

// One DPP lane move of a double (both 32-bit halves with the same control);
// lanes without a source, or in rows outside ROWMASK, read 0.
template <int CTRL, int ROWMASK>
__device__ inline double dpp_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL,
                                             ROWMASK, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL,
                                             ROWMASK, 0xF, true);
  return __hiloint2double(hi, lo);
}

// Sum over the 64 lanes of a wavefront, returned in every lane.  Row
// prefix sums by row_shr 1, 2, 4, 8 leave each 16-lane row's total in its
// lane 15; row_bcast15 and row_bcast31 fold the four rows into lane 63,
// which is then read out.  All moves stay in the VALU (no LDS round trips
// as with lane shuffles), and the order of additions is fixed.
__device__ inline double wave_sum(double v) {
  v += dpp_f64<0x111, 0xF>(v);  // row_shr:1
  v += dpp_f64<0x112, 0xF>(v);  // row_shr:2
  v += dpp_f64<0x114, 0xF>(v);  // row_shr:4
  v += dpp_f64<0x118, 0xF>(v);  // row_shr:8
  v += dpp_f64<0x142, 0xA>(v);  // row_bcast:15 into rows 1, 3
  v += dpp_f64<0x143, 0xC>(v);  // row_bcast:31 into rows 2, 3
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
  return __hiloint2double(hi, lo);
}

// All lanes take part in the DPP moves below (no lane without a source).
template <int CTRL>
__device__ __forceinline__ double dpp_all(double v) {
  return dpp_f64<CTRL, 0xF>(v);
}
// v plus the values of the lane 16 (32) away in its pair of rows (halves).
__device__ __forceinline__ double add_rows16(double v) {
  const auto lo = __builtin_amdgcn_permlane16_swap(
      __double2loint(v), __double2loint(v), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(
      __double2hiint(v), __double2hiint(v), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ __forceinline__ double add_rows32(double v) {
  const auto lo = __builtin_amdgcn_permlane32_swap(
      __double2loint(v), __double2loint(v), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(
      __double2hiint(v), __double2hiint(v), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
// Sums of four values over the wavefront for little more than the price of
// one: two exchanges hand each lane of a quad the quad's sum of one of the
// values, and five additions then run on one register.  Lane l returns the
// wavefront's sum of a[l % 4].
__device__ __forceinline__ double wave_sum4(const double (&a)[4]) {
  const bool odd = threadIdx.x & 1, two = threadIdx.x & 2;
  const double b0 = (odd ? a[1] : a[0]) + dpp_all<0xB1>(odd ? a[0] : a[1]);
  const double b1 = (odd ? a[3] : a[2]) + dpp_all<0xB1>(odd ? a[2] : a[3]);
  double c = (two ? b1 : b0) + dpp_all<0x4E>(two ? b0 : b1);
  c += dpp_all<0x124>(c);  // row_ror:4, row_ror:8: the row's four quads
  c += dpp_all<0x128>(c);
  return add_rows32(add_rows16(c));
}

// Two or four consecutive elements by one load each (two for four doubles),
// aligned to the element only.
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void ldn(const float *p, float (&v)[2]) {
  const f32x2u t = *(const f32x2u *)p;
  v[0] = t.x, v[1] = t.y;
}
__device__ __forceinline__ void ldn(const double *p, double (&v)[2]) {
  const f64x2u t = *(const f64x2u *)p;
  v[0] = t.x, v[1] = t.y;
}
__device__ __forceinline__ void ldn(const float *p, float (&v)[4]) {
  const f32x4u t = *(const f32x4u *)p;
  v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w;
}
__device__ __forceinline__ void ldn(const double *p, double (&v)[4]) {
  const f64x2u t = *(const f64x2u *)p, u = *(const f64x2u *)(p + 2);
  v[0] = t.x, v[1] = t.y, v[2] = u.x, v[3] = u.y;
}
__device__ __forceinline__ void stn(float *p, const float (&v)[4]) {
  f32x4u t;
  t.x = v[0], t.y = v[1], t.z = v[2], t.w = v[3];
  *(f32x4u *)p = t;
}
__device__ __forceinline__ void stn(double *p, const double (&v)[4]) {
  f64x2u t, u;
  t.x = v[0], t.y = v[1], u.x = v[2], u.y = v[3];
  *(f64x2u *)p = t;
  *(f64x2u *)(p + 2) = u;
}
// Element di of a row whose first element is base, for the lane `off` bytes
// into the row: the base is the same for the whole wavefront (a scalar
// address) and the lane part stays one 32-bit offset for every array.
template <class T>
__device__ __forceinline__ const T *lane_at(const T *base, int di,
                                            unsigned off) {
  return (const T *)((const char *)(base + di) + off);
}

// The operands of a pair of i-adjacent points (i0, i0 + 1) of a 27-point
// level (gsd.cc:160-211, matvecd.cc:137-170), as loaded.  Every coupling
// comes for both points with one two-element load and every neighbouring row
// of x with one four-element load (i0 - 1 .. i0 + 2): 37 loads of a pair
// against 106 scalar ones.  The kernels on 27-point levels were bound by the
// rate at which a compute unit takes vector memory instructions, not by
// bytes (MI355X, the sweeps per paired launch, scalar loads -> these: 145^3
// FP32 56 -> 44 us, 81^3 FP32 11.2 -> 8.4, FP64 16.5 -> 12.2, 33^3 and 17^3
// FP64 8.2 -> 5.8 us; the same sums in the same order).  The four-element
// loads of the last pair of the grid's last row reach one element past the
// end of x, whose value no sum uses; interp_body's reach two past the end of
// xc, and its pair loads one past the end of pc.  Every array these kernels
// are given has room for that (allocations are padded).
template <class T>
struct G27C {          // couplings, the right-hand side, the diagonal's parts
  T cN[2], cS[2];      // oN(p), oN(p - sy)
  T cE[2], cW;         // oE(p) of both points, oE(p - 1) of the first
  T c[4][2];           // oNE(p), oNW(p), oNW(p + 1 - sy), oNE(p - 1 - sy)
  T cu[9][2], cd[9][2];
  T oC[2], cc[2];
};
template <class T>
struct G27X {
  T xN[4], xS[4];        // x of rows j + 1, j - 1 in the own plane
  T xu[3][4], xd[3][4];  // rows j, j + 1, j - 1 of the planes above, below
};
// A = ac + base, cc: the arrays at an index `base` that is the same for the
// whole wavefront (a row or a plane); the pair's first point lies off bytes
// further.  PL: the planes above and below are wanted (else they count as
// zero and are not loaded).
template <bool PL, class T>
__device__ __forceinline__ void g27_couplings(const T *__restrict__ A,
                                              const T *__restrict__ cc,
                                              size_t n, long long sy,
                                              long long sz, unsigned off,
                                              G27C<T> &r) {
  auto at = [&](int pl, long long d) {
    return lane_at(A + (long long)pl * (long long)n + d, 0, off);
  };
  ldn(at(2, 0), r.cN);
  ldn(at(2, -sy), r.cS);
  ldn(at(1, 0), r.cE);
  r.cW = *at(1, -1);
  ldn(at(4, 0), r.c[0]);
  ldn(at(5, 0), r.c[1]);
  ldn(at(5, 1 - sy), r.c[2]);
  ldn(at(4, -1 - sy), r.c[3]);
  // planes uC, uN, uS, uE, uW, uNE, uNW, uSE, uSW of the plane above
  constexpr int pu[9] = {3, 8, 9, 6, 7, 10, 11, 12, 13};
  // the plane below couples through the mirrored plane of the neighbour
  constexpr int pd[9] = {3, 9, 8, 7, 6, 13, 12, 11, 10};
  const long long du[9] = {0,       sy,      -sy,    1,      -1,
                           1 + sy, -1 + sy, 1 - sy, -1 - sy};
  if constexpr (PL) {
#pragma unroll
    for (int m = 0; m < 9; m++) {
      ldn(at(pu[m], 0), r.cu[m]);
      ldn(at(pd[m], du[m] - sz), r.cd[m]);
    }
  } else {
#pragma unroll
    for (int m = 0; m < 9; m++)
      r.cu[m][0] = r.cu[m][1] = r.cd[m][0] = r.cd[m][1] = (T)0;
  }
  ldn(at(0, 0), r.oC);
  ldn(lane_at(cc, 0, off), r.cc);
}
// The neighbour rows from three arrays by their offset (dy, dz): xN (dy odd,
// dz = 0), xU (dy = 0, dz odd), xNU (dy and dz odd), each at the base.
template <bool PL, class T>
__device__ __forceinline__ void g27_rows(const T *xN, const T *xU,
                                         const T *xNU, long long sy,
                                         long long sz, unsigned off,
                                         G27X<T> &r) {
  ldn(lane_at(xN + sy, -1, off), r.xN);
  ldn(lane_at(xN - sy, -1, off), r.xS);
  if constexpr (PL) {
    ldn(lane_at(xU + sz, -1, off), r.xu[0]);
    ldn(lane_at(xNU + sy + sz, -1, off), r.xu[1]);
    ldn(lane_at(xNU - sy + sz, -1, off), r.xu[2]);
    ldn(lane_at(xU - sz, -1, off), r.xd[0]);
    ldn(lane_at(xNU + sy - sz, -1, off), r.xd[1]);
    ldn(lane_at(xNU - sy - sz, -1, off), r.xd[2]);
  } else {
#pragma unroll
    for (int m = 0; m < 12; m++) r.xu[m / 4][m % 4] = r.xd[m / 4][m % 4] = (T)0;
  }
}

// The terms of one point that do not involve the two in-row neighbours,
// summed in the reference's order as far as they go.  The multiply-adds are
// written out: of a sum of two products the compiler may round either one
// first, and its choice differed between the colours of a sweep (1 of 14
// points an ulp off after two FP32 sweeps).  The coarsest CG of a mixed
// cycle stops after up to 25 iterations at 1e-2, where its iterates have
// grown such an ulp into a different iteration count now and then, which
// moves a potential by up to 1.4e-9 of its norm.
template <class T>
struct G27Part {
  T a;             // oN(p) x(p+sy) + oN(p-sy) x(p-sy): the first two terms
  T cE, cW;
  T c[4], xv[4];   // the four in-plane terms after the in-row ones
  T u, dd, dg;     // upper and lower plane sums, oC + cc
};
// Point s (0, 1) of the pair; zN: the rows j +- 1 of the own plane count as
// zero.
template <class T, int s>
__device__ __forceinline__ G27Part<T> g27_part(const G27C<T> &r,
                                               const G27X<T> &x, bool zN) {
  auto Z = [](T v, bool z) -> T { return z ? (T)0 : v; };
  G27Part<T> g;
  g.a = fma(r.cN[s], Z(x.xN[s + 1], zN), r.cS[s] * Z(x.xS[s + 1], zN));
  g.cE = r.cE[s];
  g.cW = s ? r.cE[0] : r.cW;
  const T xv[4] = {x.xN[s + 2], x.xN[s], x.xS[s + 2], x.xS[s]};
#pragma unroll
  for (int m = 0; m < 4; m++) g.c[m] = r.c[m][s], g.xv[m] = Z(xv[m], zN);
  // terms C, N, S, E, W, NE, NW, SE, SW: the row of the plane and the place
  // in it
  constexpr int tr[9] = {0, 1, 2, 0, 0, 1, 1, 2, 2};
  constexpr int te[9] = {1, 1, 1, 2, 0, 2, 0, 2, 0};
  T u = fma(r.cu[0][s], x.xu[0][s + 1], r.cu[1][s] * x.xu[1][s + 1]);
  T dd = fma(r.cd[0][s], x.xd[0][s + 1], r.cd[1][s] * x.xd[1][s + 1]);
#pragma unroll
  for (int m = 2; m < 9; m++) {
    u = fma(r.cu[m][s], x.xu[tr[m]][s + te[m]], u);
    dd = fma(r.cd[m][s], x.xd[tr[m]][s + te[m]], dd);
  }
  g.u = u;
  g.dd = dd;
  g.dg = r.oC[s] + r.cc[s];
  return g;
}
// The in-plane sum from the part and the in-row neighbours xw, xe.
template <class T>
__device__ __forceinline__ T g27_plane(const G27Part<T> &g, T xw, T xe) {
  T o = fma(g.cW, xw, fma(g.cE, xe, g.a));
#pragma unroll
  for (int m = 0; m < 4; m++) o = fma(g.c[m], g.xv[m], o);
  return o;
}

__host__ __device__ inline int count_parity(int n, int par) {  // #{v in [2, n-1] : v%2 == par}
  const int first = 2 + par;
  return first > n - 1 ? 0 : (n - 1 - first) / 2 + 1;
}

template <class A>
struct GTab {
  A a[GMAX];
};

// Launch f(tab, count) for each run of at most GMAX consecutive entries of
// the problems whose key equals key (entries built by mk(q) into the tab).
template <class A, class KeyF, class MkF, class LaunchF>
static void g_split(int n, KeyF key, MkF mk, LaunchF launch) {
  std::vector<char> done(n, 0);
  for (int q0 = 0; q0 < n; q0++) {
    if (done[q0]) continue;
    const auto k0 = key(q0);
    GTab<A> t{};
    int m = 0;
    for (int q = q0; q < n; q++) {
      if (done[q] || !(key(q) == k0)) continue;
      done[q] = 1;
      t.a[m++] = mk(q);
      if (m == GMAX) {
        launch(t, m, k0);
        m = 0;
      }
    }
    if (m) launch(t, m, k0);
  }
}

}  // namespace pmg
