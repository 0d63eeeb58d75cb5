// lmh_scatter.hip -- element matrices and vectors into CSR values and the
// right-hand side, gather form on tiles of rows (element DoF counts up to 32).
//
// A wavefront owns a tile of consecutive rows (up to kTileSlots stored entries
// and 64 rows) and sums it in LDS.  The tile's incidences (element, local row)
// are taken in rounds -- the first of every row, then the second, ... -- so
// that the lane groups of one step (GS lanes per incidence, 64 / GS
// incidences) always work on different rows: no two lanes of a step add to one
// entry, and the entries of a row sum in ascending element order, the order of
// the reference's element loop (LDS operations of a wavefront execute in
// order).  The incidence sequence, with gaps where a round's end would repeat a
// row within a step, and the slot offsets in the order the lanes read them are
// built once with the matrix.
//
// What bounds it: vector memory instructions, then the bytes.  One row per
// half wavefront took about 20 loads and stores per row (offsets, incidences
// and right-hand-side entries one at a time, row pointers twice); a tile of
// eight Q2 rows takes about 32.  Before -> now: 64^3 Q2 FP64 1377 -> 635 us (3.0
// GB moved), FP32 1053 -> 409 us, TET10 122,000 elements 134 -> 54 us, TET4
// 1,536,000 elements 519 -> 137 us, HEX8 512,000 elements 312 -> 115 us.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "lmh_internal.h"

namespace lmh {

constexpr int kTileSlots = 512, kTileRows = 64, kTileSteps = 16;  // steps whose loads are in flight together

// Walks the incidence sequence of a tile, one wavefront with a row per lane:
// put(step slot, incidence, row) in the lane of every entry, gap(slot) for every
// gap; returns the padded length, whole groups of kTileQuad steps.  In round k the
// rows that have a k-th incidence follow each other; where one of them is already
// in the step that the last round left open, the rest begin the next step.
constexpr int kTileQuad = 4;  // steps whose offsets a lane reads at once
template <typename F, typename H>
__device__ inline int tile_walk(const int32_t *__restrict__ inc_ptr, int32_t r0, int nr, int pi, F &&put, H &&gap) {
  const int lane = threadIdx.x & 63;
  const uint64_t below = (1ull << lane) - 1;
  const int32_t b = lane < nr ? inc_ptr[r0 + lane] : 0, cnt = lane < nr ? inc_ptr[r0 + lane + 1] - b : 0;
  int pos = 0;
  uint64_t open = 0;  // rows of the step that pos is in
  for (int k = 0;; ++k) {
    const bool on = cnt > k;
    const uint64_t m = __ballot(on);
    if (!m) break;
    const int n = __popcll(m), rank = __popcll(m & below), left = pos % pi ? pi - pos % pi : pi;
    const uint64_t clash = __ballot(on && rank < left && (open >> lane & 1));
    int mine = pos + rank, next = pos + n;
    if (clash) {
      const int c = __popcll(m & ((clash & -clash) - 1)), step = (pos / pi + 1) * pi;
      if (rank >= c) mine = step + rank - c;
      next = step + n - c;
      if (pos + c + lane < step) gap(pos + c + lane);
    }
    if (on) put(mine, b + k, lane);
    const uint64_t same = __ballot(on && mine / pi == next / pi);
    open = next % pi == 0 ? 0 : pos / pi == next / pi ? open | same : same;
    pos = next;
  }
  const int q = pi * kTileQuad, len = (pos + q - 1) / q * q;
  if (pos + lane < len) gap(pos + lane);  // q <= 64
  return len;
}

__global__ __launch_bounds__(256) void k_tile_count(const int32_t *__restrict__ inc_ptr,
                                                    const int32_t *__restrict__ tr, int64_t nt, int pi,
                                                    int32_t *__restrict__ len) {
  for (int64_t t = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6); t < nt; t += (int64_t)gridDim.x * 4) {
    const int l = tile_walk(
        inc_ptr, tr[t], tr[t + 1] - tr[t], pi, [](int, int32_t, int) {}, [](int) {});
    if ((threadIdx.x & 63) == 0) len[t] = l;
  }
}

// seq: {incidence (element * dpe + local row) or -1, entry base | row << 16}, within the tile
__device__ inline void tile_fill(const int32_t *__restrict__ inc_ptr, const int32_t *__restrict__ inc,
                                 const int32_t *__restrict__ rp, int32_t r0, int32_t nr, int32_t s0, int pi,
                                 int2 *seq, int4 *__restrict__ tile) {
  const int32_t b0 = rp[r0];
  const int len = tile_walk(
      inc_ptr, r0, nr, pi,
      [&](int pos, int32_t k, int r) { seq[s0 + pos] = make_int2(inc[k], (rp[r0 + r] - b0) | (r << 16)); },
      [&](int pos) { seq[s0 + pos] = make_int2(-1, 0); });
  if ((threadIdx.x & 63) == 0) *tile = make_int4(r0, nr, s0, len / pi);
}

__global__ __launch_bounds__(256) void k_tile_fill(const int32_t *__restrict__ inc_ptr,
                                                   const int32_t *__restrict__ inc, const int32_t *__restrict__ rp,
                                                   const int32_t *__restrict__ tr, const int32_t *__restrict__ start,
                                                   int64_t nt, int pi, int2 *__restrict__ seq,
                                                   int4 *__restrict__ tile) {
  for (int64_t t = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6); t < nt; t += (int64_t)gridDim.x * 4)
    tile_fill(inc_ptr, inc, rp, tr[t], tr[t + 1] - tr[t], start[t], pi, seq, tile + t);
}

// Offset j of sequence entry s: lane (g, j) of step I reads its kTileQuad
// consecutive steps' offsets at once, at ((I / quad) * 64 + lane) * quad + I % quad.
template <typename OT>
__device__ inline void tile_offset(const int2 *seq, int64_t s, int j, int dpe, int gs, int pi,
                                   const uint16_t *__restrict__ off, OT *__restrict__ map) {
  const int64_t I = s / pi;
  const int lane = (int)(s - I * pi) * gs + j;
  const int32_t ei = seq[s].x;
  map[((I / kTileQuad) * 64 + lane) * kTileQuad + I % kTileQuad] =
      ei >= 0 && j < dpe ? (OT)off[(int64_t)ei * dpe + j] : (OT)0;
}

template <typename OT>
__global__ __launch_bounds__(256) void k_tile_map(const int2 *__restrict__ seq, int64_t total, int dpe, int gs,
                                                  const uint16_t *__restrict__ off, OT *__restrict__ map) {
  const int pi = 64 / gs;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total * gs;
       t += (int64_t)gridDim.x * blockDim.x)
    tile_offset(seq, t / gs, (int)(t % gs), dpe, gs, pi, off, map);
}

// The whole plan of a small matrix in one launch: a wavefront per tile, whose place
// in the sequence comes from a counter (which tile comes first makes no difference).
template <typename OT>
__global__ __launch_bounds__(256) void k_tile_plan(const int32_t *__restrict__ inc_ptr,
                                                   const int32_t *__restrict__ inc, const int32_t *__restrict__ rp,
                                                   const int32_t *__restrict__ tr, int64_t nt, int dpe, int gs,
                                                   const uint16_t *__restrict__ off, int32_t *__restrict__ count,
                                                   int2 *seq, int4 *__restrict__ tile, OT *__restrict__ map) {
  const int64_t t = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6);
  if (t >= nt) return;
  const int lane = threadIdx.x & 63, pi = 64 / gs;
  const int32_t r0 = tr[t], nr = tr[t + 1] - r0;
  const int len = tile_walk(
      inc_ptr, r0, nr, pi, [](int, int32_t, int) {}, [](int) {});
  int32_t s0 = 0;
  if (lane == 0) s0 = atomicAdd(count, len);
  s0 = __shfl(s0, 0);
  tile_fill(inc_ptr, inc, rp, r0, nr, s0, pi, seq, tile + t);
  __threadfence_block();  // the lanes read each other's entries
  for (int u = lane; u < len * gs; u += 64) tile_offset(seq, s0 + u / gs, u % gs, dpe, gs, pi, off, map);
}

// FP64: the LDS adder (no value returns to the wavefront, so a step does not
// wait for the one before); no two lanes of a step share an entry, so its
// result does not depend on lane order.  FP32: read, add, write; the FP32 LDS
// adder is slow here (64^3 Q2 1177 us against 409).
__device__ inline void lds_add(double *p, double v) { unsafeAtomicAdd(p, v); }
__device__ inline void lds_add(float *p, float v) { *p += v; }

// GS: lanes per incidence (the power of two >= dpe); OT: offset type.
template <typename T, int GS, typename OT>
__global__ __launch_bounds__(64) void k_scatter_tiles(const int4 *__restrict__ tiles, int64_t nt,
                                                      const int2 *__restrict__ seq, const OT *__restrict__ map,
                                                      int dpe, const int32_t *__restrict__ rp,
                                                      const T *__restrict__ Ke, const double *__restrict__ Fe,
                                                      T *__restrict__ vals, double *__restrict__ rhs) {
  constexpr int PI = 64 / GS, Q = kTileQuad;
  typedef OT oq __attribute__((ext_vector_type(Q)));
  extern __shared__ __align__(16) unsigned char smraw[];
  double *facc = (double *)smraw;  // kTileRows right-hand-side entries
  T *acc = (T *)(facc + kTileRows);
  const int lane = threadIdx.x, g = lane / GS, j = lane % GS;
  int64_t t, hi, step;
  xcd_walk(nt, t, hi, step);
  for (; t < hi; t += step) {  // one tile with the launch's grid
    const int4 tl = tiles[t];
    const int32_t r0 = tl.x, nr = tl.y, s0 = tl.z, M = tl.w;
    const int32_t b0 = rp[r0], len = rp[r0 + nr] - b0;
    for (int k = lane; k < len; k += 64) acc[k] = (T)0;
    facc[lane] = 0.0;
    const oq *mp = (const oq *)map + (int64_t)(s0 / PI / Q) * 64 + lane;
    // U steps whose loads are in flight together
    auto chunk = [&](int m0, auto uc) {
      constexpr int U = decltype(uc)::value;
      const int mc = M - m0 < U ? M - m0 : U;  // a multiple of Q
      // the steps' sequence entries, one per lane (U * PI of them, in turns of 64)
      int2 sv[(U * PI + 63) / 64];
      double fv[(U * PI + 63) / 64];
#pragma unroll
      for (int c = 0; c < (U * PI + 63) / 64; ++c) {
        const int idx = 64 * c + lane;
        sv[c] = seq[s0 + m0 * PI + (idx < mc * PI ? idx : 0)];
        if (idx >= mc * PI) sv[c].x = -1;
        fv[c] = rhs && sv[c].x >= 0 ? Fe[sv[c].x] : 0.0;
      }
      oq ov[U / Q];
#pragma unroll
      for (int q = 0; q < U / Q; ++q) ov[q] = mp[(int64_t)(m0 / Q + (q * Q < mc ? q : 0)) * 64];
      T v[U];
      int32_t ei[U], rb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int src = u * PI + g;
        ei[u] = __shfl(sv[(u * PI) / 64].x, src & 63);
        rb[u] = __shfl(sv[(u * PI) / 64].y, src & 63);
        const bool on = ei[u] >= 0 && j < dpe;
        v[u] = Ke[on ? (int64_t)ei[u] * dpe + j : 0];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int src = u * PI + g;
        const double f = __shfl(fv[(u * PI) / 64], src & 63);
        if (ei[u] >= 0) {
          if (j < dpe) lds_add(&acc[(rb[u] & 0xffff) + ov[u / Q][u % Q]], v[u]);
          if (j == 0) lds_add(&facc[rb[u] >> 16], f);
        }
        // a step's additions precede the next step's (one wavefront: in order)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
    };
    for (int m0 = 0; m0 < M; m0 += kTileSteps)
      if (M - m0 > kTileSteps / 2)
        chunk(m0, std::integral_constant<int, kTileSteps>{});
      else
        chunk(m0, std::integral_constant<int, kTileSteps / 2>{});
    for (int k = lane; k < len; k += 64) vals[b0 + k] = acc[k];
    if (rhs && lane < nr) rhs[r0 + lane] = facc[lane];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

static int group_lanes(int dpe) { return dpe <= 4 ? 4 : dpe <= 8 ? 8 : dpe <= 16 ? 16 : 32; }

// Small matrices: the plan in one launch and one allocation, whose sequence is sized
// for the worst case (every incidence alone in its step) instead of counted first
// and waited for.  Matrix creation, without a plan / counted first / this way: Q1
// 8^3 383, 467, 390 us, Q2 4^3 385, 468, 394, TET10 3^3 462, 559, 468.  Up to 2 MB, of
// which a Q1 matrix uses a fifth, or 8 MB where the matrix's values take as much (Q2,
// whose plan fills half of it).
static bool plan_worst_case(size_t bytes, size_t values) {
  return bytes <= (2 << 20) || (bytes <= (8 << 20) && bytes <= values);
}

// Below this many rows a tetrahedral matrix has no tiles.  Its rows have up to 24
// incidences and a few entries, so a tile's steps are a long chain with most of
// their lane groups idle; two rows to a wavefront (k_scatter_rows) end sooner while
// the GPU holds all of them.  A scatter among others, rows / tiles: TET4 1,315 rows
// 8.2 / 10.4 us, 5,631 11.1 / 11.2, 9,541 16.5 / 13.4; three variables 2,373 rows 8.5 /
// 9.9, 6,093 12.3 / 11.7; TET10 4,881 rows 9.4 / 9.8, 8,245 10.9 / 10.2; three variables
// 3,459 9.3 / 10.3, 7,755 12.5 / 11.2.  Hexahedra (at most 8 incidences) 3.9 / 3.6 at
// the smallest sizes.
constexpr int64_t kTetTileRows = 5500;

// Tiles of the matrix's rows; h_rp: its row pointers.  Patterns the tiles do
// not take (more than 32 element DoFs, a row beyond 4096 entries, small tetrahedral
// ones) and matrices without room for the plan keep the row kernels.  `rows` holds what a
// copy on the stream may still read: for the caller to keep until it has waited.
int matrix_build_tiles(lmh_matrix *A, const std::vector<int32_t> &h_rp, std::vector<int32_t> &rows) {
  const lmh_dofmap *dm = A->dm;
  lmh_context *ctx = A->ctx;
  if (!dm || dm->dpe > 32 || A->max_row > 4096 || A->rows == 0) return LMH_OK;
  const bool tet = dm->mesh->type == LMH_TET4 || dm->mesh->type == LMH_TET10;
  if (tet && A->rows < kTetTileRows) return LMH_OK;
  const int gs = group_lanes(dm->dpe), pi = 64 / gs;
  // small matrices: fewer entries per tile, so that every CU has several
  const int64_t want = A->nnz / ((int64_t)ctx->cu_count * 8);
  const int cap = (int)std::min<int64_t>(kTileSlots, std::max<int64_t>(64, want));
  rows.assign(1, 0);
  for (int64_t r = 0; r < A->rows; ++r) {
    const int32_t f = rows.back();
    if (r > f && (h_rp[r + 1] - h_rp[f] > cap || r - f >= kTileRows)) rows.push_back((int32_t)r);
  }
  rows.push_back((int32_t)A->rows);
  const int64_t nt = (int64_t)rows.size() - 1;
  rows.push_back(0);  // k_tile_plan's counter
  const bool wide = A->max_row > 256;
  // tiles, sequence, offsets and `more` bytes in one allocation
  auto allocate = [&](int64_t total, size_t more) {
    auto line = [](size_t bytes) { return (bytes + 255) & ~(size_t)255; };  // a wavefront's reads start on a line
    const size_t seq = line(sizeof(int4) * nt), map = seq + line(sizeof(int2) * total),
                 end = map + line((wide ? 2 : 1) * (size_t)total * gs);
    if (hipMalloc((void **)&A->st_tile, end + more) != hipSuccess) {
      (void)hipGetLastError();
      A->st_tile = nullptr;
      return (unsigned char *)nullptr;
    }
    unsigned char *m = (unsigned char *)A->st_tile;
    A->st_seq = (int2 *)(m + seq);
    A->st_map = m + map;
    return m + end;
  };
  const int64_t most = dm->mesh->n_elem * dm->dpe * pi + nt * (int64_t)(pi * kTileQuad);
  if (plan_worst_case((size_t)most * (8 + gs * (wide ? 2 : 1)), sizeof(double) * (size_t)A->nnz)) {
    int32_t *dtr = (int32_t *)allocate(most, sizeof(int32_t) * rows.size());
    if (!dtr) return LMH_OK;
    LMH_HIP(hipMemcpyAsync(dtr, rows.data(), sizeof(int32_t) * rows.size(), hipMemcpyHostToDevice, ctx->stream));
    const dim3 g((unsigned)((nt + 3) / 4));
    if (wide)
      LMH_LAUNCH(ctx, "tile_plan", k_tile_plan<uint16_t>, g, dim3(256), 0, dm->inc_ptr, dm->inc, A->rp,
                 (const int32_t *)dtr, nt, dm->dpe, gs, A->off, dtr + nt + 1, A->st_seq, A->st_tile,
                 (uint16_t *)A->st_map);
    else
      LMH_LAUNCH(ctx, "tile_plan", k_tile_plan<uint8_t>, g, dim3(256), 0, dm->inc_ptr, dm->inc, A->rp,
                 (const int32_t *)dtr, nt, dm->dpe, gs, A->off, dtr + nt + 1, A->st_seq, A->st_tile,
                 (uint8_t *)A->st_map);
    LMH_TRY(check_launch("k_tile_plan"));
  } else {
    int32_t *tmp = nullptr;  // tile rows, lengths, starts: nt + 1 each
    if (hipMallocAsync((void **)&tmp, sizeof(int32_t) * 3 * (nt + 1), ctx->stream) != hipSuccess) {
      (void)hipGetLastError();
      return LMH_OK;
    }
    int32_t *dtr = tmp, *len = tmp + nt + 1, *start = len + nt + 1;
    auto plan = [&]() -> int {
      LMH_HIP(hipMemcpyAsync(dtr, rows.data(), sizeof(int32_t) * (nt + 1), hipMemcpyHostToDevice, ctx->stream));
      LMH_HIP(hipMemsetAsync(len, 0, sizeof(int32_t) * (nt + 1), ctx->stream));
      const int g = grid_for(nt, 4, 16384);
      LMH_LAUNCH(ctx, "tile_plan", k_tile_count, dim3(g), dim3(256), 0, dm->inc_ptr, (const int32_t *)dtr, nt, pi,
                 len);
      LMH_TRY(check_launch("k_tile_count"));
      int64_t total = 0;
      const int rc = exclusive_scan_i32(ctx, len, start, nt, &total);
      if (rc == LMH_ERR_UNSUPPORTED) return LMH_OK;  // a sequence beyond 32-bit places
      LMH_TRY(rc);
      if (!allocate(total, 0)) return LMH_OK;
      LMH_LAUNCH(ctx, "tile_plan", k_tile_fill, dim3(g), dim3(256), 0, dm->inc_ptr, dm->inc, A->rp,
                 (const int32_t *)dtr, (const int32_t *)start, nt, pi, A->st_seq, A->st_tile);
      LMH_TRY(check_launch("k_tile_fill"));
      if (total == 0) return LMH_OK;
      const int gm = grid_for(total * gs, 256, 16384);
      if (wide)
        LMH_LAUNCH(ctx, "tile_plan", k_tile_map<uint16_t>, dim3(gm), dim3(256), 0, A->st_seq, total, dm->dpe, gs,
                   A->off, (uint16_t *)A->st_map);
      else
        LMH_LAUNCH(ctx, "tile_plan", k_tile_map<uint8_t>, dim3(gm), dim3(256), 0, A->st_seq, total, dm->dpe, gs,
                   A->off, (uint8_t *)A->st_map);
      return check_launch("k_tile_map");
    };
    const int rc = plan();
    (void)hipFreeAsync(tmp, ctx->stream);
    LMH_TRY(rc);
    if (!A->st_tile) return LMH_OK;
  }
  A->st_wide = wide;
  A->st_slots = std::max(cap, A->max_row);
  A->n_stile = nt;
  return LMH_OK;
}

template <typename T, int GS>
static void launch_tiles(lmh_matrix *A, const T *Ke, const double *Fe, T *vals, double *rhs) {
  lmh_context *ctx = A->ctx;
  const char *name = sizeof(T) == 8 ? "scatter_gather_fp64" : "scatter_gather_fp32";
  // a workgroup per tile: the hardware's dispatch balances tiles of uneven
  // length (64^3 Q2 FP64 635 us; 680 us with 128 workgroups per CU, 723 with 32)
  const dim3 g((unsigned)((A->n_stile + NXCD - 1) / NXCD * NXCD));
  const size_t shm = sizeof(double) * kTileRows + sizeof(T) * (size_t)A->st_slots;
  if (A->st_wide)
    LMH_LAUNCH(ctx, name, (k_scatter_tiles<T, GS, uint16_t>), g, dim3(64), shm, A->st_tile, A->n_stile, A->st_seq,
               (const uint16_t *)A->st_map, A->dm->dpe, A->rp, Ke, Fe, vals, rhs);
  else
    LMH_LAUNCH(ctx, name, (k_scatter_tiles<T, GS, uint8_t>), g, dim3(64), shm, A->st_tile, A->n_stile, A->st_seq,
               (const uint8_t *)A->st_map, A->dm->dpe, A->rp, Ke, Fe, vals, rhs);
}

template <typename T>
int scatter_tiles(lmh_matrix *A, const T *Ke, const double *Fe, T *vals, double *rhs) {
  switch (group_lanes(A->dm->dpe)) {
    case 4: launch_tiles<T, 4>(A, Ke, Fe, vals, rhs); break;
    case 8: launch_tiles<T, 8>(A, Ke, Fe, vals, rhs); break;
    case 16: launch_tiles<T, 16>(A, Ke, Fe, vals, rhs); break;
    default: launch_tiles<T, 32>(A, Ke, Fe, vals, rhs); break;
  }
  return check_launch("k_scatter_tiles");
}
template int scatter_tiles<double>(lmh_matrix *, const double *, const double *, double *, double *);
template int scatter_tiles<float>(lmh_matrix *, const float *, const double *, float *, double *);

}  // namespace lmh
