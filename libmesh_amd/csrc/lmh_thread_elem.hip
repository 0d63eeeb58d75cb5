// lmh_thread_elem.hip -- element kernels with one element per thread, for the
// elements whose nodal data fit a thread's registers: TET4, TET10, HEX8, with
// any quadrature rule.
//
// A wavefront per element leaves most lanes idle on these types (10 to 14 of
// 64 on TET10, 4 or 5 on TET4) and reads the reference tables from LDS for
// every product.  With a thread per element every lane works, the points are
// walked in step, and the tables are wave-uniform: they are read through the
// scalar cache into scalar registers, which the FP64 multiply-adds take as an
// operand.
#include <algorithm>

#include "lmh_internal.h"

namespace lmh {

constexpr int kTB = 64;  // threads per workgroup

template <int N>
__device__ inline void te_coords(const double *__restrict__ xyz, const int32_t *__restrict__ conn, int64_t e,
                                 double (&X)[N][3]) {
  int32_t nd[N];
#pragma unroll
  for (int a = 0; a < N; ++a) nd[a] = conn[e * N + a];
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int c = 0; c < 3; ++c) X[a][c] = xyz[3 * (int64_t)nd[a] + c];
}

// Cofactor rows c[r] of J[r][k] = sum_a X_a[k] dref_a[r] (dxi_r/dx = c[r] / det)
// and det J; dref: 3 N wave-uniform values.
template <int N>
__device__ inline double te_map(const double (&X)[N][3], const double *__restrict__ dref, double (&c)[3][3]) {
  double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int k = 0; k < 3; ++k) J[r][k] += X[a][k] * dref[3 * a + r];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const double *a = J[(r + 1) % 3], *b = J[(r + 2) % 3];
    c[r][0] = a[1] * b[2] - a[2] * b[1];
    c[r][1] = a[2] * b[0] - a[0] * b[2];
    c[r][2] = a[0] * b[1] - a[1] * b[0];
  }
  return J[0][0] * c[0][0] + J[0][1] * c[0][1] + J[0][2] * c[0][2];
}

template <int N>
__device__ inline void te_point(const double (&X)[N][3], const double *__restrict__ phi, double (&x)[3]) {
  x[0] = x[1] = x[2] = 0.0;
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] += X[a][k] * phi[a];
}

// TET4's map and shape derivatives are the same at every point: what does not
// depend on the point is formed at the first, with the weights' sum (1,536,000
// elements: matrices 105 -> 79 us with the sine forcing, FP32 with f = 1 70 -> 50).
template <int N>
__device__ inline double te_weight(const double *__restrict__ pts, int nq) {
  if (N != 4) return 0.0;
  double w = 0.0;
  for (int q = 0; q < nq; ++q) w += pts[(int64_t)q * (1 + 4 * N)];
  return w;
}

// Residual vectors R_e = K_e u_e - F_e from the flux at each point.
template <int N, int FK>
__global__ __launch_bounds__(kTB) void k_thread_residual(const double *__restrict__ pts, int nq,
                                                         const double *__restrict__ xyz,
                                                         const int32_t *__restrict__ conn,
                                                         const int32_t *__restrict__ edofs,
                                                         const double *__restrict__ kappa, const double *__restrict__ u,
                                                         int64_t ne, double *__restrict__ Fe, int *__restrict__ err) {
  const int64_t e = blockIdx.x * (int64_t)kTB + threadIdx.x;
  if (e >= ne) return;
  double X[N][3], U[N], R[N];
  te_coords<N>(xyz, conn, e, X);
#pragma unroll
  for (int a = 0; a < N; ++a) {
    U[a] = u[edofs[e * N + a]];
    R[a] = 0.0;
  }
  const double kap = kappa ? kappa[e] : 1.0;
  const double wsum = te_weight<N>(pts, nq);
  double det = 0.0;
  bool bad = false;
  for (int q = 0; q < nq; ++q) {
    const double *P = pts + (int64_t)q * (1 + 4 * N), *phi = P + 1, *d = P + 1 + N;
    if (N != 4 || q == 0) {
      double c[3][3], g[3] = {0, 0, 0}, v[3], fl[3];
      det = te_map<N>(X, d, c);
      bad |= !(det > 0.0);
#pragma unroll
      for (int a = 0; a < N; ++a)
#pragma unroll
        for (int r = 0; r < 3; ++r) g[r] += U[a] * d[3 * a + r];
      // on one factor, not on the product: c c^T alone leaves the range of FP64 for
      // elements smaller than 1e-77 or larger than 1e77
      const double s = kap * (N == 4 ? wsum : P[0]) / det;
#pragma unroll
      for (int r = 0; r < 3; ++r) g[r] *= s;
#pragma unroll
      for (int k = 0; k < 3; ++k) v[k] = g[0] * c[0][k] + g[1] * c[1][k] + g[2] * c[2][k];
#pragma unroll
      for (int r = 0; r < 3; ++r) fl[r] = c[r][0] * v[0] + c[r][1] * v[1] + c[r][2] * v[2];
#pragma unroll
      for (int a = 0; a < N; ++a) R[a] += fl[0] * d[3 * a] + fl[1] * d[3 * a + 1] + fl[2] * d[3 * a + 2];
    }
    double fj = det * P[0];
    if constexpr (FK != 0) {
      double x[3];
      te_point<N>(X, phi, x);
      fj *= forcing(FK, x[0], x[1], x[2]);
    }
#pragma unroll
    for (int a = 0; a < N; ++a) R[a] -= fj * phi[a];
  }
  if (bad) raise_flag(err);
#pragma unroll
  for (int a = 0; a < N; ++a) Fe[e * N + a] = R[a];
}

// Q_i = sum over the points inside [lo, hi]^3 of JxW phi_i.
template <int N>
__global__ __launch_bounds__(kTB) void k_thread_qoi(const double *__restrict__ pts, int nq,
                                                    const double *__restrict__ xyz, const int32_t *__restrict__ conn,
                                                    int64_t ne, double lo, double hi, double *__restrict__ Q,
                                                    int *__restrict__ err) {
  const int64_t e = blockIdx.x * (int64_t)kTB + threadIdx.x;
  if (e >= ne) return;
  double X[N][3], R[N];
  te_coords<N>(xyz, conn, e, X);
#pragma unroll
  for (int a = 0; a < N; ++a) R[a] = 0.0;
  double det = 0.0;
  bool bad = false;
  for (int q = 0; q < nq; ++q) {
    const double *P = pts + (int64_t)q * (1 + 4 * N), *phi = P + 1, *d = P + 1 + N;
    double c[3][3], x[3];
    if (N != 4 || q == 0) det = te_map<N>(X, d, c);
    bad |= !(det > 0.0);
    te_point<N>(X, phi, x);
    const bool in =
        x[0] >= lo && x[0] <= hi && x[1] >= lo && x[1] <= hi && x[2] >= lo && x[2] <= hi;
    const double jc = in ? det * P[0] : 0.0;
#pragma unroll
    for (int a = 0; a < N; ++a) R[a] += jc * phi[a];
  }
  if (bad) raise_flag(err);
#pragma unroll
  for (int a = 0; a < N; ++a) Q[e * N + a] = R[a];
}

// dJ/dkappa_e = -sum_q JxW grad(lambda).grad(u), values masked to the free DoFs.
template <int N>
__global__ __launch_bounds__(kTB) void k_thread_adjoint(const double *__restrict__ pts, int nq,
                                                        const double *__restrict__ xyz,
                                                        const int32_t *__restrict__ conn,
                                                        const int32_t *__restrict__ edofs,
                                                        const uint8_t *__restrict__ cons, const double *__restrict__ u,
                                                        const double *__restrict__ lam, int64_t ne,
                                                        double *__restrict__ grad, int *__restrict__ err) {
  const int64_t e = blockIdx.x * (int64_t)kTB + threadIdx.x;
  if (e >= ne) return;
  double X[N][3], U[N], W[N];
  te_coords<N>(xyz, conn, e, X);
#pragma unroll
  for (int a = 0; a < N; ++a) {
    const int32_t dof = edofs[e * N + a];
    const bool cn = cons[dof] != 0;
    U[a] = cn ? 0.0 : u[dof];
    W[a] = cn ? 0.0 : lam[dof];
  }
  double s = 0.0;
  bool bad = false;
  const double wsum = te_weight<N>(pts, nq);
  for (int q = 0; q < (N == 4 ? 1 : nq); ++q) {
    const double *P = pts + (int64_t)q * (1 + 4 * N), *d = P + 1 + N;
    double c[3][3], gu[3] = {0, 0, 0}, gl[3] = {0, 0, 0};
    const double det = te_map<N>(X, d, c);
    bad |= !(det > 0.0);
#pragma unroll
    for (int a = 0; a < N; ++a)
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        gu[r] += U[a] * d[3 * a + r];
        gl[r] += W[a] * d[3 * a + r];
      }
    const double f = (N == 4 ? wsum : P[0]) / det;
#pragma unroll
    for (int r = 0; r < 3; ++r) gu[r] *= f;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      s += (gu[0] * c[0][k] + gu[1] * c[1][k] + gu[2] * c[2][k]) *
           (gl[0] * c[0][k] + gl[1] * c[1][k] + gl[2] * c[2][k]);
  }
  if (bad) raise_flag(err);
  grad[e] = -s;
}

// Constrained (if `constrain`) element matrix and vector of the Poisson
// operator, FP64 arithmetic, stored as CT.  The upper triangle accumulates in
// registers (K is symmetric: M_q is); rows are written out in blocks of R rows
// through LDS, so the workgroup's 64 matrices leave as coalesced runs instead
// of one 8-byte store per lane and matrix.  Bound by the FP64 multiply-adds at
// two wavefronts per SIMD (230 to 250 registers: the triangle and the nodes).
// One element per wavefront before: TET10 122,000 elements 1646 -> 63 us, TET4
// 1,536,000 elements 6096 -> 79 us, HEX8 512,000 352 -> 97 us (FP32 3921 -> 84).
template <int N, int R, typename CT, int FK>
__global__ __launch_bounds__(kTB) __attribute__((amdgpu_waves_per_eu(2))) void k_thread_poisson(
    const double *__restrict__ pts, int nq, const double *__restrict__ xyz, const int32_t *__restrict__ conn,
    const int32_t *__restrict__ edofs, const uint8_t *__restrict__ cons, const double *__restrict__ kappa,
    int constrain, int64_t ne, CT *__restrict__ Ke, double *__restrict__ Fe, int *__restrict__ err) {
  static_assert(N % R == 0, "whole blocks of rows");
  constexpr int W = R * N, ST = W + 1;  // odd stride: the lanes' slots fall in different banks
  __shared__ CT tile[kTB * ST];
  const int lane = threadIdx.x;
  const int64_t e0 = blockIdx.x * (int64_t)kTB;
  const bool live = e0 + lane < ne;
  const int64_t e = live ? e0 + lane : ne - 1;
  double X[N][3], K[N * (N + 1) / 2], F[N];
  te_coords<N>(xyz, conn, e, X);
  unsigned cm = 0;
  if (constrain)
#pragma unroll
    for (int a = 0; a < N; ++a) cm |= (cons[edofs[e * N + a]] != 0 ? 1u : 0u) << a;
  const double kap = kappa ? kappa[e] : 1.0;
#pragma unroll
  for (int k = 0; k < N * (N + 1) / 2; ++k) K[k] = 0.0;
#pragma unroll
  for (int a = 0; a < N; ++a) F[a] = 0.0;
  const double wsum = te_weight<N>(pts, nq);
  double det = 0.0;
  bool bad = false;
  for (int q = 0; q < nq; ++q) {
    const double *P = pts + (int64_t)q * (1 + 4 * N), *phi = P + 1, *d = P + 1 + N;
    if (N != 4 || q == 0) {
      double c[3][3], M[3][3];
      det = te_map<N>(X, d, c);
      bad |= !(det > 0.0);
      const double s = kap * (N == 4 ? wsum : P[0]) / det;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const double a = s * c[r][0], b = s * c[r][1], f = s * c[r][2];
#pragma unroll
        for (int t = r; t < 3; ++t) M[r][t] = M[t][r] = a * c[t][0] + b * c[t][1] + f * c[t][2];
      }
      int k = 0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        double v[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) v[t] = M[0][t] * d[3 * i] + M[1][t] * d[3 * i + 1] + M[2][t] * d[3 * i + 2];
#pragma unroll
        for (int j = i; j < N; ++j, ++k) K[k] += v[0] * d[3 * j] + v[1] * d[3 * j + 1] + v[2] * d[3 * j + 2];
      }
    }
    double fj = det * P[0];
    if constexpr (FK != 0) {
      double x[3];
      te_point<N>(X, phi, x);
      fj *= forcing(FK, x[0], x[1], x[2]);
    }
#pragma unroll
    for (int a = 0; a < N; ++a) F[a] += fj * phi[a];
  }
  if (bad && live) raise_flag(err);
  const int64_t left = (ne - e0 < kTB ? ne - e0 : kTB) * W;  // entries of this block of rows
#pragma unroll
  for (int i0 = 0; i0 < N; i0 += R) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int i = i0 + r, lo = i < j ? i : j, hi = i < j ? j : i;
        double v = K[lo * N - lo * (lo - 1) / 2 + (hi - lo)];
        if (((cm >> i) | (cm >> j)) & 1u) v = i == j ? 1.0 : 0.0;
        tile[lane * ST + r * N + j] = (CT)v;
      }
    __syncthreads();
    for (int t = lane; t < left; t += kTB) {
      const int el = t / W, o = t - el * W;
      Ke[(e0 + el) * (N * N) + i0 * N + o] = tile[el * ST + o];
    }
    __syncthreads();
  }
  if (live)
#pragma unroll
    for (int a = 0; a < N; ++a) Fe[e * N + a] = (cm >> a) & 1u ? 0.0 : F[a];
}

static dim3 te_grid(int64_t ne) { return dim3((unsigned)((ne + kTB - 1) / kTB)); }

template <int N>
static int residual_n(lmh_context *ctx, const FETable *t, const lmh_mesh *m, const lmh_dofmap *dm,
                      const double *kappa, int f_kind, const double *u, double *Fe) {
  if (f_kind == 0)
    LMH_LAUNCH(ctx, "element_residual", (k_thread_residual<N, 0>), te_grid(m->n_elem), dim3(kTB), 0, t->d_points(),
               t->nq, m->xyz, m->conn, dm->edofs, kappa, u, m->n_elem, Fe, ctx->g_flag);
  else
    LMH_LAUNCH(ctx, "element_residual", (k_thread_residual<N, 1>), te_grid(m->n_elem), dim3(kTB), 0, t->d_points(),
               t->nq, m->xyz, m->conn, dm->edofs, kappa, u, m->n_elem, Fe, ctx->g_flag);
  return check_launch("k_thread_residual");
}

int thread_residual(lmh_context *ctx, const FETable *t, const lmh_mesh *m, const lmh_dofmap *dm, const double *kappa,
                    int f_kind, const double *u, double *Fe) {
  if (m->n_elem == 0) return LMH_OK;
  switch (t->n) {
    case 4: return residual_n<4>(ctx, t, m, dm, kappa, f_kind, u, Fe);
    case 8: return residual_n<8>(ctx, t, m, dm, kappa, f_kind, u, Fe);
    case 10: return residual_n<10>(ctx, t, m, dm, kappa, f_kind, u, Fe);
  }
  return set_error(LMH_ERR_UNSUPPORTED, "no thread kernel for %d nodes", t->n);
}

int thread_qoi(lmh_context *ctx, const FETable *t, const lmh_mesh *m, double lo, double hi, double *Q) {
  if (m->n_elem == 0) return LMH_OK;
#define TE_QOI(N)                                                                                                   \
  LMH_LAUNCH(ctx, "qoi_box", k_thread_qoi<N>, te_grid(m->n_elem), dim3(kTB), 0, t->d_points(), t->nq, m->xyz, m->conn, \
             m->n_elem, lo, hi, Q, ctx->g_flag)
  switch (t->n) {
    case 4: TE_QOI(4); break;
    case 8: TE_QOI(8); break;
    case 10: TE_QOI(10); break;
    default: return set_error(LMH_ERR_UNSUPPORTED, "no thread kernel for %d nodes", t->n);
  }
#undef TE_QOI
  return check_launch("k_thread_qoi");
}

int thread_adjoint(lmh_context *ctx, const FETable *t, const lmh_mesh *m, const lmh_dofmap *dm, const double *u,
                   const double *lam, double *grad) {
  if (m->n_elem == 0) return LMH_OK;
#define TE_ADJ(N)                                                                                                     \
  LMH_LAUNCH(ctx, "adjoint_kappa", k_thread_adjoint<N>, te_grid(m->n_elem), dim3(kTB), 0, t->d_points(), t->nq, m->xyz, \
             m->conn, dm->edofs, dm->cons, u, lam, m->n_elem, grad, ctx->g_flag)
  switch (t->n) {
    case 4: TE_ADJ(4); break;
    case 8: TE_ADJ(8); break;
    case 10: TE_ADJ(10); break;
    default: return set_error(LMH_ERR_UNSUPPORTED, "no thread kernel for %d nodes", t->n);
  }
#undef TE_ADJ
  return check_launch("k_thread_adjoint");
}

template <int N, int R, typename CT>
static int poisson_n(lmh_context *ctx, const FETable *t, const lmh_mesh *m, const lmh_dofmap *dm, const double *kappa,
                     int f_kind, int constrain, CT *Ke, double *Fe) {
  if (f_kind == 0)
    LMH_LAUNCH(ctx, "element_thread", (k_thread_poisson<N, R, CT, 0>), te_grid(m->n_elem), dim3(kTB), 0,
               t->d_points(), t->nq, m->xyz, m->conn, dm->edofs, dm->cons, kappa, constrain, m->n_elem, Ke, Fe,
               ctx->g_flag);
  else
    LMH_LAUNCH(ctx, "element_thread", (k_thread_poisson<N, R, CT, 1>), te_grid(m->n_elem), dim3(kTB), 0,
               t->d_points(), t->nq, m->xyz, m->conn, dm->edofs, dm->cons, kappa, constrain, m->n_elem, Ke, Fe,
               ctx->g_flag);
  return check_launch("k_thread_poisson");
}

template <typename CT>
int thread_poisson(lmh_context *ctx, const FETable *t, const lmh_mesh *m, const lmh_dofmap *dm, const double *kappa,
                   int f_kind, int constrain, CT *Ke, double *Fe) {
  if (m->n_elem == 0) return LMH_OK;
  switch (t->n) {
    case 4: return poisson_n<4, 4, CT>(ctx, t, m, dm, kappa, f_kind, constrain, Ke, Fe);
    case 8: return poisson_n<8, 2, CT>(ctx, t, m, dm, kappa, f_kind, constrain, Ke, Fe);
    case 10: return poisson_n<10, 2, CT>(ctx, t, m, dm, kappa, f_kind, constrain, Ke, Fe);
  }
  return set_error(LMH_ERR_UNSUPPORTED, "no thread kernel for %d nodes", t->n);
}
template int thread_poisson<double>(lmh_context *, const FETable *, const lmh_mesh *, const lmh_dofmap *,
                                    const double *, int, int, double *, double *);
template int thread_poisson<float>(lmh_context *, const FETable *, const lmh_mesh *, const lmh_dofmap *,
                                   const double *, int, int, float *, double *);

}  // namespace lmh
