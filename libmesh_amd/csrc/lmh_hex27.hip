// lmh_hex27.hip -- HEX27 element kernels on the tensor-product evaluation of
// lmh_hex27.h: residual of the Poisson physics, QoI derivative and adjoint
// gradient, none of which needs an element matrix.
//
// What bounds them: the element data are small (27 nodes, a few fields), so the
// kernels are FP64-instruction and LDS-read bound.  With one element per
// wavefront and a lane per point, 27 of 64 lanes worked and every point summed
// 27 nodes against a 17 KB table in LDS (three workgroups per CU).  Here seven
// elements share a wavefront, each lane forms three points by sum factorisation
// and no table is read.  Residual and adjoint form the metric (six values a
// point) from the coordinates first and only then the other fields' gradients,
// and form their lane constants anew in every group: 168 registers and three
// wavefronts per SIMD instead of 242 and two (residual) or more than 256 and one
// (adjoint); four spill (45 and 38 us).  64,000 elements (40^3), before -> now:
// residual element stage 555 (element matrices, then K_e u_e) -> 33.8 us, QoI 290 ->
// 20.9 us, adjoint gradient 326 -> 30.5 us; the three calls with their gathers and
// host waits 1290 -> 159 us.
#include <algorithm>

#include "lmh_hex27.h"

namespace lmh {

// Nodal data of the wavefront's seven elements.
struct H27Slots {
  int el[3], lat[3];
  bool live[3];
  __device__ explicit H27Slots(int lane) {
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const int k = lane + 64 * m;
      live[m] = k < 27 * kH27PerWave;
      const int kk = live[m] ? k : 0;
      el[m] = kk / 27;
      lat[m] = kH27Lat[kk - 27 * el[m]];
    }
  }
  // entries t = e0 * 27 + lane + 64 m of an n_elem x 27 table (clamped to the last)
  __device__ inline void ids(const int32_t *__restrict__ tab, int64_t e0, int64_t total, int lane,
                             int32_t (&id)[3]) const {
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const int64_t t = e0 * 27 + lane + 64 * m;
      id[m] = tab[t < total ? t : total - 1];
    }
  }
};

// The wavefront's node coordinates x to LDS, relative to their element's centre
// node, and the centres to s_c (four values per element).  J is a difference of
// nodal coordinates: formed from absolute ones it loses the digits that the
// element's place takes.  64^3 matrices against 80-bit arithmetic, largest error of
// an entry over the largest entry, mean of 24 elements: absolute 3.7e-15 (sums over
// a table 3.1e-15), relative 2.0e-16.  The matrix kernel takes 453 -> 466 us for
// 64^3 with f = 1, 74 -> 70 for 31 x 29 x 37 with the sine; 40^3 residual 32.2 ->
// 33.8, QoI 21.4 -> 20.9, adjoint 30.3 -> 30.5, every load issued before the first
// use (one after the other: residual 34.9, adjoint 33.2).
template <int NF, int ST>
__device__ inline void h27_store_nodes(const H27Slots &sl, const double (&x)[3][3], double *s_f, double *s_c) {
#pragma unroll
  for (int m = 0; m < 3; ++m)
    if (sl.live[m] && sl.lat[m] == 26) {
#pragma unroll
      for (int c = 0; c < 3; ++c) s_c[sl.el[m] * 4 + c] = x[m][c];
    }
  h27_sync();
  double r[3][3];  // idle slots' too: no branch between the reads
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int c = 0; c < 3; ++c) r[m][c] = x[m][c] - s_c[sl.el[m] * 4 + c];
#pragma unroll
  for (int m = 0; m < 3; ++m)
    if (sl.live[m]) {
      double *d = s_f + sl.el[m] * ST + sl.lat[m] * NF;
#pragma unroll
      for (int c = 0; c < 3; ++c) d[c] = r[m][c];
    }
}

// Element vectors R_e = K_e u_e - F_e without K_e: at each point the reference
// flux M grad u (M = JxW kappa G G^T) and f JxW, contracted with the test
// functions direction 3 first (in registers), then directions 1 and 2 through
// LDS, lane l owning the test functions (i1, i2) = (l % 3, l / 3).
template <int FK>
__global__ __launch_bounds__(64, 3) void k_hex27_residual(const double *__restrict__ xyz,
                                                          const int32_t *__restrict__ conn,
                                                          const int32_t *__restrict__ edofs,
                                                          const double *__restrict__ kappa, const double *__restrict__ u,
                                                          int64_t ne, double *__restrict__ Fe, int *__restrict__ err) {
  constexpr int NF = 4, ST = 27 * NF + 1;  // odd stride: the elements' broadcasts fall in different banks
  __shared__ double s_f[kH27PerWave * ST];
  __shared__ double s_h[kH27PerWave * 81];
  __shared__ __attribute__((aligned(16))) double s_c[kH27PerWave * 4];
  const int lane = threadIdx.x;
  const int64_t total = ne * 27, groups = (ne + kH27PerWave - 1) / kH27PerWave;
  for (int64_t gr = blockIdx.x; gr < groups; gr += gridDim.x) {
    int lg = lane;
    asm volatile("" : "+v"(lg));  // lane constants formed again for every group, not held
    const H27Slots sl(lg);
    int32_t nd[3], dof[3];
    sl.ids(conn, gr * kH27PerWave, total, lane, nd);
    sl.ids(edofs, gr * kH27PerWave, total, lane, dof);
    const H27Lane L(lg);
    const int64_t e0 = gr * kH27PerWave, e = e0 + L.el;
    double x[3][3], um[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
#pragma unroll
      for (int c = 0; c < 3; ++c) x[m][c] = xyz[3 * (int64_t)nd[m] + c];
      um[m] = u[dof[m]];
    }
    h27_store_nodes<NF, ST>(sl, x, s_f, s_c);
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (sl.live[m]) s_f[sl.el[m] * ST + sl.lat[m] * NF + 3] = um[m];
    const bool on = L.el < kH27PerWave && e < ne;
    h27_sync();
    if (on) {
      const double kap = kappa ? kappa[e] : 1.0;
      double M[3][6], det[3], pos[3][FK ? 3 : 1], none[3][1];
      {
        double g[3][3][3];
        h27_refgrad<3, FK ? 3 : 0, NF>(s_f + L.el * ST, L, g, pos);
        h27_metric(g, [&](int q) { return kap * (L.w12 * h27_w(q)); }, M, det, err);
      }
      __builtin_amdgcn_sched_barrier(0);
      double g[3][1][3];
      h27_refgrad<1, 0, NF>(s_f + L.el * ST + 3, L, g, none);
      double h[3][3];
#pragma unroll
      for (int i = 0; i < 3; ++i) h[i][0] = h[i][1] = h[i][2] = 0.0;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double fl[3];
        h27_apply(M[q], g[q][0], fl);
        double fj = det[q] * (L.w12 * h27_w(q));
        if constexpr (FK != 0) {
          const double *c = s_c + L.el * 4;
          fj *= forcing(FK, c[0] + pos[q][0], c[1] + pos[q][1], c[2] + pos[q][2]);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          h[i][0] += h27_p(q, i) * fl[0];
          h[i][1] += h27_p(q, i) * fl[1];
          h[i][2] += h27_d(q, i) * fl[2] - h27_p(q, i) * fj;
        }
      }
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) s_h[L.el * 81 + (3 * i + k) * 9 + L.l] = h[i][k];
    }
    h27_sync();
    if (on) {
      double pt[3], dt[3], pt2[3], dt2[3];  // the lane's test functions at the 1D points
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        pt[q] = h27_pick(L.l % 3, [&](int i) { return h27_p(q, i); });
        dt[q] = h27_pick(L.l % 3, [&](int i) { return h27_d(q, i); });
        pt2[q] = h27_pick(L.l / 3, [&](int i) { return h27_p(q, i); });
        dt2[q] = h27_pick(L.l / 3, [&](int i) { return h27_d(q, i); });
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const double *H = s_h + L.el * 81 + 27 * i;
        double s = 0.0;
#pragma unroll
        for (int q2 = 0; q2 < 3; ++q2) {
          double a = 0.0, b = 0.0;
#pragma unroll
          for (int q1 = 0; q1 < 3; ++q1) {
            const int q = 3 * q2 + q1;
            a += dt[q1] * H[q] + pt[q1] * H[18 + q];
            b += pt[q1] * H[9 + q];
          }
          s += pt2[q2] * a + dt2[q2] * b;
        }
        Fe[e * 27 + kH27Node[9 * i + L.l]] = s;
      }
    }
    h27_sync();
  }
}

// Q_i = sum over the points inside [lo, hi]^3 of JxW phi_i.
__global__ __launch_bounds__(64) void k_hex27_qoi(const double *__restrict__ xyz, const int32_t *__restrict__ conn,
                                                  int64_t ne, double lo, double hi, double *__restrict__ Q,
                                                  int *__restrict__ err) {
  constexpr int NF = 3, ST = 27 * NF;
  __shared__ double s_f[kH27PerWave * ST];
  __shared__ double s_h[kH27PerWave * 27];
  __shared__ __attribute__((aligned(16))) double s_c[kH27PerWave * 4];
  const int lane = threadIdx.x;
  const H27Slots sl(lane);
  const H27Lane L(lane);
  double pt[3], pt2[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    pt[q] = h27_pick(L.l % 3, [&](int i) { return h27_p(q, i); });
    pt2[q] = h27_pick(L.l / 3, [&](int i) { return h27_p(q, i); });
  }
  const int64_t total = ne * 27, groups = (ne + kH27PerWave - 1) / kH27PerWave;
  int32_t nd[3];
  sl.ids(conn, (int64_t)blockIdx.x * kH27PerWave, total, lane, nd);
  for (int64_t gr = blockIdx.x; gr < groups; gr += gridDim.x) {
    const int64_t e = gr * kH27PerWave + L.el;
    double x[3][3];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int c = 0; c < 3; ++c) x[m][c] = xyz[3 * (int64_t)nd[m] + c];
    h27_store_nodes<NF, ST>(sl, x, s_f, s_c);
    sl.ids(conn, (gr + gridDim.x) * kH27PerWave, total, lane, nd);
    const bool on = L.el < kH27PerWave && e < ne;
    h27_sync();
    if (on) {
      double g[3][NF][3], pos[3][3], h[3] = {0.0, 0.0, 0.0};
      h27_refgrad<NF, 3>(s_f + L.el * ST, L, g, pos);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double J[3][3], c[3][3];
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
          for (int k = 0; k < 3; ++k) J[r][k] = g[q][k][r];
        const double det = cofactors(J, c);
        if (!(det > 0.0)) raise_flag(err);
        const double *o = s_c + L.el * 4;
        const double x = o[0] + pos[q][0], y = o[1] + pos[q][1], z = o[2] + pos[q][2];
        const bool in = x >= lo && x <= hi && y >= lo && y <= hi && z >= lo && z <= hi;
        const double jc = in ? det * (L.w12 * h27_w(q)) : 0.0;
#pragma unroll
        for (int i = 0; i < 3; ++i) h[i] += h27_p(q, i) * jc;
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) s_h[L.el * 27 + 9 * i + L.l] = h[i];
    }
    h27_sync();
    if (on) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const double *H = s_h + L.el * 27 + 9 * i;
        double s = 0.0;
#pragma unroll
        for (int q2 = 0; q2 < 3; ++q2)
          s += pt2[q2] * (pt[0] * H[3 * q2] + pt[1] * H[3 * q2 + 1] + pt[2] * H[3 * q2 + 2]);
        Q[e * 27 + kH27Node[9 * i + L.l]] = s;
      }
    }
    h27_sync();
  }
}

// dJ/dkappa_e = -sum_q JxW grad(lambda).grad(u), nodal values masked to the
// free DoFs (see k_adjoint_kappa).
__global__ __launch_bounds__(64, 3) void k_hex27_adjoint(const double *__restrict__ xyz,
                                                         const int32_t *__restrict__ conn,
                                                         const int32_t *__restrict__ edofs,
                                                         const uint8_t *__restrict__ cons, const double *__restrict__ u,
                                                         const double *__restrict__ lam, int64_t ne,
                                                         double *__restrict__ grad, int *__restrict__ err) {
  constexpr int NF = 5, ST = 27 * NF;
  __shared__ double s_f[kH27PerWave * ST];
  __shared__ __attribute__((aligned(16))) double s_c[kH27PerWave * 4];
  const int lane = threadIdx.x;
  const int64_t total = ne * 27, groups = (ne + kH27PerWave - 1) / kH27PerWave;
  for (int64_t gr = blockIdx.x; gr < groups; gr += gridDim.x) {
    int lg = lane;
    asm volatile("" : "+v"(lg));  // lane constants formed again for every group, not held
    const H27Slots sl(lg);
    int32_t nd[3], dof[3];
    sl.ids(conn, gr * kH27PerWave, total, lane, nd);
    sl.ids(edofs, gr * kH27PerWave, total, lane, dof);
    const H27Lane L(lg);
    const int64_t e = gr * kH27PerWave + L.el;
    // all loads issued before any is looked at
    double x[3][3], um[3], lm[3];
    int cv[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
#pragma unroll
      for (int c = 0; c < 3; ++c) x[m][c] = xyz[3 * (int64_t)nd[m] + c];
      cv[m] = cons[dof[m]];
      um[m] = u[dof[m]];
      lm[m] = lam[dof[m]];
    }
    h27_store_nodes<NF, ST>(sl, x, s_f, s_c);
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (sl.live[m]) {
        double *d = s_f + sl.el[m] * ST + sl.lat[m] * NF;
        d[3] = cv[m] ? 0.0 : um[m];
        d[4] = cv[m] ? 0.0 : lm[m];
      }
    const bool on = L.el < kH27PerWave && e < ne;
    h27_sync();
    double s = 0.0;
    if (on) {
      double M[3][6], det[3], none[3][1];
      {
        double g[3][3][3];
        h27_refgrad<3, 0, NF>(s_f + L.el * ST, L, g, none);
        h27_metric(g, [&](int q) { return L.w12 * h27_w(q); }, M, det, err);
      }
      __builtin_amdgcn_sched_barrier(0);
      double g[3][2][3];
      h27_refgrad<2, 0, NF>(s_f + L.el * ST + 3, L, g, none);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double y[3];
        h27_apply(M[q], g[q][0], y);
        s += y[0] * g[q][1][0] + y[1] * g[q][1][1] + y[2] * g[q][1][2];
      }
    }
    // sum of the element's nine columns in a fixed order
    s += __shfl(s, lane + 3) + __shfl(s, lane + 6);
    const double s1 = __shfl(s, lane + 1), s2 = __shfl(s, lane + 2);
    if (on && L.l == 0) grad[e] = -(s + s1 + s2);
    h27_sync();
  }
}

// ---------------------------------------------------------------------------
// Element matrices of the Poisson operator by sum factorisation, one wavefront
// per workgroup, up to seven elements of geometry at a time.
//
//   K_ij = sum_{r,s} sum_q a_r(q,i) M_rs(q) a_s(q,j),  M = JxW kappa G G^T,
//
// with a_r the product of 1D shapes whose direction-r factor is the derivative.
// Per element, 54 of 64 lanes: lane t = 9 c + k, c one of the six unordered
// pairs i3 <= j3 (K is symmetric), k first a column (q1, q2), then a pair
// (i2, j2):
//   S (8 arrays) = direction 3 contracted, lane (q1, q2) x (i3, j3)
//   T (4 x 3, by the kind of direction 1's factors: dd, dp, pd, pp)
//                = direction 2 contracted, lane (i2, j2) x (i3, j3), S through LDS
//   K = direction 1 contracted in registers, nine entries (i1, j1) per lane,
// each written with its mirror to an LDS tile that leaves as 16-byte stores.
// 195 multiply-adds per lane instead of the 84 16x16x4 matrix instructions
// (86,000 multiply-adds with their padding) of the table contraction this
// replaces, which also formed its operands from nine LDS reads per k-step.
// FP64 throughout; the FP32 operator is the FP64 entry rounded once.
// Bound by LDS reads and their latency: S is read array by array, a column set in
// five 16-byte reads (nine 8-byte reads of all arrays held at once took 250
// registers, two wavefronts per SIMD: FP64 633, FP32 600 us), and what a phase
// needs is formed in it, not kept across (lane constants and the next group's
// indices in registers spilled 116 bytes a lane: 580 and 480 us; 28 bytes are
// left).  262,144 elements: FP64 1545 -> 543 us, FP32 1258 -> 448 us.  The next
// element's S ahead of this one's T: 256 registers and 350 bytes of spills, 913 us.
// ---------------------------------------------------------------------------
// Elements whose geometry a wavefront forms together and wavefronts per CU that
// fit (168 registers, LDS).  FP64: 7 and 9; six elements let twelve in, whose
// stores then get in each other's way (64^3 724 us against 577).  FP32: 6 and 12
// (64^3 473 us; 491 with 7 and 10).
template <typename CT>
struct H27Group {
  static constexpr int per = sizeof(CT) == 8 ? 7 : 6, waves = sizeof(CT) == 8 ? 9 : 12,
                       grid = sizeof(CT) == 8 ? 20 : 12;  // workgroups per CU
};
template <typename CT, int FK>
__global__ __launch_bounds__(64, 3) void k_hex27_poisson(const double *__restrict__ xyz,
                                                         const int32_t *__restrict__ conn,
                                                         const int32_t *__restrict__ edofs,
                                                         const uint8_t *__restrict__ cons,
                                                         const double *__restrict__ kappa, int constrain, int per,
                                                         int64_t ne, CT *__restrict__ Ke, double *__restrict__ Fe,
                                                         int *__restrict__ err) {
  constexpr int NF = 3, ST = 27 * NF;
  // node coordinates of the group; then, per element, S and the matrix tile
  __shared__ __attribute__((aligned(16))) double s_buf[sizeof(CT) == 8 ? 730 : kH27PerWave * ST];
  __shared__ double s_m[H27Group<CT>::per * 162];  // M[el][6 components][q3][q1q2]
  __shared__ __attribute__((aligned(16))) double s_c[kH27PerWave * 4];
  double *s_h = s_buf;  // over the coordinates: a wavefront's lanes have all read them by then
  const int lane = threadIdx.x;
  // the matrix lanes: pair (i3, j3) of c, pair (i2, j2) of k
  const int t54 = lane < 54 ? lane : 0, cc = t54 / 9, kk = t54 - 9 * cc;
  const int i3 = cc < 3 ? cc : (cc == 5 ? 1 : 0), j3 = cc < 3 ? cc : (cc == 3 ? 1 : 2);
  const int i2 = kk % 3, j2 = kk / 3;
  const int64_t total = ne * 27, groups = (ne + per - 1) / per;
  for (int64_t gr = blockIdx.x; gr < groups; gr += gridDim.x) {
    // lane constants of this phase: formed again for every group (the opaque
    // lane index keeps the compiler from holding both phases' in registers)
    int lg = lane;
    asm volatile("" : "+v"(lg));
    const H27Slots sl(lg);
    int32_t nd[3], dof[3];
    sl.ids(conn, gr * per, total, lane, nd);
    sl.ids(edofs, gr * per, total, lane, dof);
    const H27Lane L(lg);
    const int64_t e0 = gr * per;
    const int cnt = (int)(ne - e0 < per ? ne - e0 : per);
    unsigned long long bits[3];  // constrained flags, bit 27 el + node of the group
    double x[3][3];
    int cv[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) cv[m] = cons[dof[m]];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int c = 0; c < 3; ++c) x[m][c] = xyz[3 * (int64_t)nd[m] + c];
    // loaded with the rest, not one after the other where they are used
    asm volatile("" : "+v"(cv[0]), "+v"(cv[1]), "+v"(cv[2]));
    h27_store_nodes<NF, ST>(sl, x, s_buf, s_c);
#pragma unroll
    for (int m = 0; m < 3; ++m) bits[m] = constrain ? __ballot(cv[m] != 0 && sl.live[m]) : 0ull;
    auto mask_of = [&](int el) -> unsigned {  // 27 flags of element el, by local node
      const int b = 27 * el, w = b >> 6, o = b & 63;
      unsigned long long v = bits[0];
      if (w == 1) v = bits[1];
      if (w == 2) v = bits[2];
      v >>= o;
      if (o > 37) v |= (w == 0 ? bits[1] : bits[2]) << (64 - o);
      return (unsigned)v & 0x7ffffffu;
    };
    const bool on = L.el < cnt;
    h27_sync();
    if (on) {
      const double kap = kappa ? kappa[e0 + L.el] : 1.0;
      double g[3][NF][3], pos[3][FK ? 3 : 1], h[3] = {0.0, 0.0, 0.0};
      h27_refgrad<NF, FK ? 3 : 0>(s_buf + L.el * ST, L, g, pos);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double J[3][3], c[3][3];
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
          for (int k = 0; k < 3; ++k) J[r][k] = g[q][k][r];
        const double det = cofactors(J, c);
        if (!(det > 0.0)) raise_flag(err);
        const double w = L.w12 * h27_w(q);
        double *M = s_m + L.el * 162 + 9 * q + L.l;  // components 11, 12, 13, 22, 23, 33
        cofactor_metric(c, kap * w / det, [&](int m, double v) { M[27 * m] = v; });
        double fj = det * w;
        if constexpr (FK != 0) {
          const double *o = s_c + L.el * 4;
          fj *= forcing(FK, o[0] + pos[q][0], o[1] + pos[q][1], o[2] + pos[q][2]);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) h[i] += h27_p(q, i) * fj;
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) s_h[L.el * 27 + 9 * i + L.l] = h[i];
    }
    h27_sync();
    if (on) {
      const unsigned cm = mask_of(L.el);
      double pt[3], pt2[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        pt[q] = h27_pick(L.l % 3, [&](int i) { return h27_p(q, i); });
        pt2[q] = h27_pick(L.l / 3, [&](int i) { return h27_p(q, i); });
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const double *H = s_h + L.el * 27 + 9 * i;
        double s = 0.0;
#pragma unroll
        for (int q2 = 0; q2 < 3; ++q2)
          s += pt2[q2] * (pt[0] * H[3 * q2] + pt[1] * H[3 * q2 + 1] + pt[2] * H[3 * q2 + 2]);
        const int a = kH27Node[9 * i + L.l];
        Fe[(e0 + L.el) * 27 + a] = (cm >> a) & 1u ? 0.0 : s;
      }
    }
    int a3 = i3, b3 = j3, a2 = i2, b2 = j2;
    asm volatile("" : "+v"(a3), "+v"(b3), "+v"(a2), "+v"(b2));
    int ni[3], nj[3];  // local nodes of the lane's rows (i1, i2, i3) and columns (j1, j2, j3)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      ni[i] = kH27Node[9 * a3 + 3 * a2 + i];
      nj[i] = kH27Node[9 * b3 + 3 * b2 + i];
    }
    double pi3[3], di3[3], pj3[3], dj3[3], pi2[3], di2[3], pj2[3], dj2[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      pi3[q] = h27_pick(a3, [&](int i) { return h27_p(q, i); });
      di3[q] = h27_pick(a3, [&](int i) { return h27_d(q, i); });
      pj3[q] = h27_pick(b3, [&](int i) { return h27_p(q, i); });
      dj3[q] = h27_pick(b3, [&](int i) { return h27_d(q, i); });
      pi2[q] = h27_pick(a2, [&](int i) { return h27_p(q, i); });
      di2[q] = h27_pick(a2, [&](int i) { return h27_d(q, i); });
      pj2[q] = h27_pick(b2, [&](int i) { return h27_p(q, i); });
      dj2[q] = h27_pick(b2, [&](int i) { return h27_d(q, i); });
    }
    for (int el = 0; el < cnt; ++el) {
      const unsigned cm = __builtin_amdgcn_readfirstlane(mask_of(el));
      if (lane < 54) {
        const double *M = s_m + el * 162 + kk;  // kk: the column (q1, q2)
        double S[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const double m11 = M[9 * q], m12 = M[27 + 9 * q], m13 = M[54 + 9 * q], m22 = M[81 + 9 * q],
                       m23 = M[108 + 9 * q], m33 = M[135 + 9 * q];
          const double pp = pi3[q] * pj3[q], pd = pi3[q] * dj3[q], dp = di3[q] * pj3[q], dd = di3[q] * dj3[q];
          S[0] += pp * m11;
          S[1] += pp * m12;
          S[2] += pp * m22;
          S[3] += pd * m13;
          S[4] += dp * m13;
          S[5] += pd * m23;
          S[6] += dp * m23;
          S[7] += dd * m33;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) s_buf[60 * k + 10 * cc + kk] = S[k];
      }
      h27_sync();
      double K[3][3];
      if (lane < 54) {
        // an array's nine columns (and a pad) in five 16-byte reads, array by array
        typedef double d2 __attribute__((ext_vector_type(2)));
        double T[3][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};  // [q1][dd, dp, pd, pp]
        auto array = [&](int k, auto &&add) {
          double S[10];
#pragma unroll
          for (int u = 0; u < 5; ++u) {
            const d2 w = *(const d2 *)(s_buf + 60 * k + 10 * cc + 2 * u);
            S[2 * u] = w[0];
            S[2 * u + 1] = w[1];
          }
#pragma unroll
          for (int q2 = 0; q2 < 3; ++q2)
#pragma unroll
            for (int q1 = 0; q1 < 3; ++q1) add(T[q1], q2, S[3 * q2 + q1]);
        };
        array(0, [&](double(&t)[4], int q, double s) { t[0] += pi2[q] * pj2[q] * s; });
        array(1, [&](double(&t)[4], int q, double s) {
          t[1] += pi2[q] * dj2[q] * s;
          t[2] += di2[q] * pj2[q] * s;
        });
        array(2, [&](double(&t)[4], int q, double s) { t[3] += di2[q] * dj2[q] * s; });
        array(3, [&](double(&t)[4], int q, double s) { t[1] += pi2[q] * pj2[q] * s; });
        array(4, [&](double(&t)[4], int q, double s) { t[2] += pi2[q] * pj2[q] * s; });
        array(5, [&](double(&t)[4], int q, double s) { t[3] += di2[q] * pj2[q] * s; });
        array(6, [&](double(&t)[4], int q, double s) { t[3] += pi2[q] * dj2[q] * s; });
        array(7, [&](double(&t)[4], int q, double s) { t[3] += pi2[q] * pj2[q] * s; });
        double K0[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
        for (int q1 = 0; q1 < 3; ++q1) {
          const double tdd = T[q1][0], tdp = T[q1][1], tpd = T[q1][2], tpp = T[q1][3];
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            const double u = h27_d(q1, j) * tdd + h27_p(q1, j) * tdp, v = h27_d(q1, j) * tpd + h27_p(q1, j) * tpp;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
              if (h27_d(q1, i) != 0.0) K0[i][j] += h27_d(q1, i) * u;
              if (h27_p(q1, i) != 0.0) K0[i][j] += h27_p(q1, i) * v;
            }
          }
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) K[i][j] = K0[i][j];
      }
      h27_sync();  // S is read
      CT *tile = (CT *)s_buf;
      if (lane < 54) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            double v = K[i][j];
            if (((cm >> ni[i]) | (cm >> nj[j])) & 1u) v = ni[i] == nj[j] ? 1.0 : 0.0;
            tile[ni[i] * 27 + nj[j]] = (CT)v;
            if (cc >= 3) tile[nj[j] * 27 + ni[i]] = (CT)v;
          }
      }
      h27_sync();
      CT *out = Ke + (e0 + el) * 729;
      constexpr int V = 16 / sizeof(CT), NV = 729 / V;  // 16-byte pieces, and the last entry
      typedef CT vt __attribute__((ext_vector_type(V)));
      typedef vt vtu __attribute__((aligned(sizeof(CT))));
#pragma unroll
      for (int k = 0; k < (NV + 63) / 64; ++k)
        if (64 * k + 63 < NV || 64 * k + lane < NV)
          *(vtu *)(out + V * (64 * k + lane)) = *(const vt *)(tile + V * (64 * k + lane));
      if (lane == 0) out[728] = tile[728];
      h27_sync();
    }
  }
}

static int h27_grid(lmh_context *ctx, int64_t ne) {
  return grid_for((ne + kH27PerWave - 1) / kH27PerWave, 1, ctx->cu_count * 32);
}

template <typename CT>
int hex27_poisson(lmh_context *ctx, const lmh_mesh *m, const lmh_dofmap *dm, const double *kappa, int f_kind,
                  int constrain, CT *Ke, double *Fe) {
  const int64_t ne = m->n_elem;
  if (ne == 0) return LMH_OK;
  // as many elements share the geometry lanes as one round of wavefronts takes (Q2
  // 20^3: 36 us with whole groups in two rounds, 30 in one)
  const int64_t waves = (int64_t)ctx->cu_count * H27Group<CT>::waves;
  const int per = (int)std::min<int64_t>(H27Group<CT>::per, (ne + waves - 1) / waves);
  const int g = grid_for((ne + per - 1) / per, 1, ctx->cu_count * H27Group<CT>::grid);
  const char *name = sizeof(CT) == 8 ? "element_hex27_fp64" : "element_hex27_fp32";
  if (f_kind == 0)
    LMH_LAUNCH(ctx, name, (k_hex27_poisson<CT, 0>), dim3(g), dim3(64), 0, m->xyz, m->conn, dm->edofs,
               dm->cons, kappa, constrain, per, ne, Ke, Fe, ctx->g_flag);
  else
    LMH_LAUNCH(ctx, name, (k_hex27_poisson<CT, 1>), dim3(g), dim3(64), 0, m->xyz, m->conn, dm->edofs,
               dm->cons, kappa, constrain, per, ne, Ke, Fe, ctx->g_flag);
  return check_launch("k_hex27_poisson");
}
template int hex27_poisson<double>(lmh_context *, const lmh_mesh *, const lmh_dofmap *, const double *, int, int,
                                   double *, double *);
template int hex27_poisson<float>(lmh_context *, const lmh_mesh *, const lmh_dofmap *, const double *, int, int,
                                  float *, double *);

int hex27_residual(lmh_context *ctx, const lmh_mesh *m, const lmh_dofmap *dm, const double *kappa, int f_kind,
                   const double *u, double *Fe) {
  if (m->n_elem == 0) return LMH_OK;
  const int g = h27_grid(ctx, m->n_elem);
  if (f_kind == 0)
    LMH_LAUNCH(ctx, "element_residual", k_hex27_residual<0>, dim3(g), dim3(64), 0, m->xyz, m->conn, dm->edofs, kappa,
               u, m->n_elem, Fe, ctx->g_flag);
  else
    LMH_LAUNCH(ctx, "element_residual", k_hex27_residual<1>, dim3(g), dim3(64), 0, m->xyz, m->conn, dm->edofs, kappa,
               u, m->n_elem, Fe, ctx->g_flag);
  return check_launch("k_hex27_residual");
}

int hex27_qoi(lmh_context *ctx, const lmh_mesh *m, double lo, double hi, double *Q) {
  if (m->n_elem == 0) return LMH_OK;
  LMH_LAUNCH(ctx, "qoi_box", k_hex27_qoi, dim3(h27_grid(ctx, m->n_elem)), dim3(64), 0, m->xyz, m->conn, m->n_elem, lo,
             hi, Q, ctx->g_flag);
  return check_launch("k_hex27_qoi");
}

int hex27_adjoint(lmh_context *ctx, const lmh_mesh *m, const lmh_dofmap *dm, const double *u, const double *lam,
                  double *grad) {
  if (m->n_elem == 0) return LMH_OK;
  LMH_LAUNCH(ctx, "adjoint_kappa", k_hex27_adjoint, dim3(h27_grid(ctx, m->n_elem)), dim3(64), 0, m->xyz, m->conn,
             dm->edofs, dm->cons, u, lam, m->n_elem, grad, ctx->g_flag);
  return check_launch("k_hex27_adjoint");
}

}  // namespace lmh
