// lmh_hex27.h -- tensor-product (sum-factorised) evaluation on HEX27 elements
// with the 3x3x3 Gauss rule, shared by the HEX27 element kernels.
//
// The shapes are products of 1D quadratic Lagrange shapes and the points a
// product of 1D Gauss points, so the map and the reference gradients at all 27
// points follow from three contractions of length 3 instead of 27-node sums.
// Nine lanes work on one element (seven elements per wavefront, 63 of 64 lanes
// busy): lane l = (q1, q2) = (l % 3, l / 3) owns the three points q3 = 0..2 of
// its column.  It contracts directions 1 and 2 from the element's nodal values
// in LDS, then direction 3 in registers: 108 multiply-adds per nodal field and
// column (36 per point) instead of 81 per point, all of them on busy lanes.
#pragma once

#include "lmh_internal.h"

namespace lmh {

// 1D quadratic shapes in libMesh's order of a direction's positions: 0 = the
// -1 end, 1 = the +1 end, 2 = the middle; Gauss points -g, 0, g.
constexpr double kG3 = 0.77459666924148337703585307995648;
__host__ __device__ constexpr double h27_x(int q) { return q == 0 ? -kG3 : (q == 1 ? 0.0 : kG3); }
__host__ __device__ constexpr double h27_p(int q, int i) {
  return i == 0 ? 0.5 * h27_x(q) * (h27_x(q) - 1.0)
                : (i == 1 ? 0.5 * h27_x(q) * (h27_x(q) + 1.0) : 1.0 - h27_x(q) * h27_x(q));
}
__host__ __device__ constexpr double h27_d(int q, int i) {
  return i == 0 ? h27_x(q) - 0.5 : (i == 1 ? h27_x(q) + 0.5 : -2.0 * h27_x(q));
}
__host__ __device__ constexpr double h27_w(int q) { return q == 1 ? 8.0 / 9.0 : 5.0 / 9.0; }

constexpr int kH27PerWave = 7;

// lattice position i1 + 3 i2 + 9 i3 of each local node (positions per
// direction as above), and its inverse
__device__ const uint8_t kH27Lat[27] = {0,  1,  4,  3,  9,  10, 13, 12, 2,  7,  5,  6,  18, 19,
                                        22, 21, 11, 16, 14, 15, 8,  20, 25, 23, 24, 17, 26};
__device__ const uint8_t kH27Node[27] = {0,  1,  8,  3,  2,  10, 11, 9,  20, 4,  5,  16, 7, 6,
                                         18, 19, 17, 25, 12, 13, 21, 15, 14, 23, 24, 22, 26};

// value of a 1D table at a lane-dependent point
template <typename F>
__device__ inline double h27_pick(int q, F f) {
  return q == 0 ? f(0) : (q == 1 ? f(1) : f(2));
}

// One wavefront per workgroup: LDS written by some lanes, read by others.
__device__ inline void h27_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct H27Lane {
  int el, l;               // element slot of the wavefront, (q1, q2) column
  double p1[3], d1[3];     // 1D shapes / derivatives at the lane's q1
  double p2[3], d2[3];     // at the lane's q2
  double w12;              // weight of (q1, q2)
  __device__ explicit H27Lane(int lane) {
    el = lane / 9;
    l = lane - 9 * el;
    const int q1 = l % 3, q2 = l / 3;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      p1[i] = h27_pick(q1, [&](int q) { return h27_p(q, i); });
      d1[i] = h27_pick(q1, [&](int q) { return h27_d(q, i); });
      p2[i] = h27_pick(q2, [&](int q) { return h27_p(q, i); });
      d2[i] = h27_pick(q2, [&](int q) { return h27_d(q, i); });
    }
    w12 = h27_pick(q1, [](int q) { return h27_w(q); }) * h27_pick(q2, [](int q) { return h27_w(q); });
  }
};

// Reference gradients of NF nodal fields at the lane's three points:
// g[q3][f][r] = sum_a F_a dphi_a/dxi_r, fields in lattice order in LDS
// (F[lat * ST + f]); with NV > 0 also the values v[q3][f] of the first NV.
template <int NF, int NV, int ST = NF>
__device__ inline void h27_refgrad(const double *F, const H27Lane &L, double (&g)[3][NF][3],
                                   double (&v)[3][NV > 0 ? NV : 1]) {
#pragma unroll
  for (int q = 0; q < 3; ++q) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int r = 0; r < 3; ++r) g[q][f][r] = 0.0;
#pragma unroll
    for (int f = 0; f < NV; ++f) v[q][f] = 0.0;
  }
#pragma unroll
  for (int i3 = 0; i3 < 3; ++i3) {
    double a0[NF], a1[NF], a2[NF];  // (phi', phi), (phi, phi'), (phi, phi) in directions 1, 2
#pragma unroll
    for (int f = 0; f < NF; ++f) a0[f] = a1[f] = a2[f] = 0.0;
#pragma unroll
    for (int i2 = 0; i2 < 3; ++i2)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const double *x = F + (9 * i3 + 3 * i2) * ST + f;
        const double p = L.p1[0] * x[0] + L.p1[1] * x[ST] + L.p1[2] * x[2 * ST];
        const double d = L.d1[0] * x[0] + L.d1[1] * x[ST] + L.d1[2] * x[2 * ST];
        a0[f] += L.p2[i2] * d;
        a1[f] += L.d2[i2] * p;
        a2[f] += L.p2[i2] * p;
      }
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        if (h27_p(q, i3) != 0.0) {  // compile-time zeros of the middle point
          g[q][f][0] += h27_p(q, i3) * a0[f];
          g[q][f][1] += h27_p(q, i3) * a1[f];
          if (f < NV) v[q][f] += h27_p(q, i3) * a2[f];
        }
        if (h27_d(q, i3) != 0.0) g[q][f][2] += h27_d(q, i3) * a2[f];
      }
    __builtin_amdgcn_sched_barrier(0);  // one plane's nodes in registers at a time
  }
}

// Cofactor rows c[r] of the map J[r][c] = dx_c/dxi_r (J^{-1} has columns
// c[r] / det: dxi_r/dx = c[r] / det) and det J.
__device__ inline double cofactors(const double (&J)[3][3], double (&c)[3][3]) {
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double *a = J[(r + 1) % 3], *b = J[(r + 2) % 3];
    c[r][0] = a[1] * b[2] - a[2] * b[1];
    c[r][1] = a[2] * b[0] - a[0] * b[2];
    c[r][2] = a[0] * b[1] - a[1] * b[0];
  }
  return J[0][0] * c[0][0] + J[0][1] * c[0][1] + J[0][2] * c[0][2];
}

// M = s C C^T, C the cofactor rows: put(m, value) for the components 11, 12, 13,
// 22, 23, 33.  s is on one factor, not on the product: C C^T alone leaves the range
// of FP64 for elements smaller than 1e-77 or larger than 1e77, M at 1e-102 and 1e102.
template <typename P>
__device__ inline void cofactor_metric(const double (&c)[3][3], double s, P &&put) {
  int m = 0;
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double a = s * c[r][0], b = s * c[r][1], d = s * c[r][2];
#pragma unroll
    for (int k = r; k < 3; ++k, ++m) put(m, a * c[k][0] + b * c[k][1] + d * c[k][2]);
  }
}

// M[q3] = w / det C C^T (components as above) and
// det at the lane's three points, from the coordinates' reference gradients; w(q3)
// is the point's factor.  The gradients need not outlive it.
template <typename W>
__device__ inline void h27_metric(const double (&g)[3][3][3], W &&w, double (&M)[3][6], double (&det)[3], int *err) {
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double J[3][3], c[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int k = 0; k < 3; ++k) J[r][k] = g[q][k][r];
    det[q] = cofactors(J, c);
    if (!(det[q] > 0.0)) raise_flag(err);
    cofactor_metric(c, w(q) / det[q], [&](int m, double v) { M[q][m] = v; });
  }
}
// M v for such a point
__device__ inline void h27_apply(const double (&M)[6], const double (&v)[3], double (&y)[3]) {
  y[0] = M[0] * v[0] + M[1] * v[1] + M[2] * v[2];
  y[1] = M[1] * v[0] + M[3] * v[1] + M[4] * v[2];
  y[2] = M[2] * v[0] + M[4] * v[1] + M[5] * v[2];
}

}  // namespace lmh
