// Sparse operations on the assembled CSR (rows = test dofs, sorted columns):
// the product y = K x, dof constraints (Dirichlet by simplification) and a
// Jacobi-preconditioned conjugate gradient solve.
//
// SpMV: G lanes of a wavefront share one row; each lane walks the row with
// stride G, then the G partial sums are combined by shuffles.  G is picked
// from the mean row length so that short rows (P1) do not leave most lanes
// idle.
//
// CG: an iteration is four launches (product, p.q, update with r.z and r.r,
// direction); every scalar of the recurrence lives in device memory and
// comes from fixed-order reductions, and so does the stopping test, so the
// host launches iterations in batches and looks once per batch; the result
// does not depend on scheduling or on the batch, nor on which of the products'
// kernels runs: all of them sum a row in k_spmv's order.
#include <hip/hip_runtime.h>

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "gfx_internal.h"

namespace gfx {
namespace {

constexpr int kSpmvThreads = 256;
constexpr int kRedThreads = 256;   // threads of a reduction block
constexpr int kRedBlocks = 1024;   // most partial sums of a dot product
constexpr int kMaxProdBlocks = 2048;  // most blocks of a CG product (8 a CU)

template <int G, bool ACC>
__global__ __launch_bounds__(kSpmvThreads) void k_spmv(int64_t n, const int64_t *__restrict__ indptr,
                                                        const int32_t *__restrict__ indices,
                                                        const double *__restrict__ vals,
                                                        const double *__restrict__ x,
                                                        double *__restrict__ y) {
  const int64_t row = ((int64_t)blockIdx.x * kSpmvThreads + threadIdx.x) / G;
  const int lane = threadIdx.x % G;
  double s = 0.0;
  if (row < n) {
    const int64_t b = indptr[row], e = indptr[row + 1];
    for (int64_t k = b + lane; k < e; k += G) s += vals[k] * x[indices[k]];
  }
  for (int off = G / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, G);
  if (row < n && lane == 0) y[row] = ACC ? y[row] + s : s;
}

template <int G>
hipError_t spmv_g(hipStream_t s, int64_t n, const int64_t *indptr, const int32_t *indices,
                  const double *vals, const double *x, double *y, bool acc) {
  const int64_t threads = n * G;
  const unsigned grid = (unsigned)((threads + kSpmvThreads - 1) / kSpmvThreads);
  if (acc) k_spmv<G, true><<<grid, kSpmvThreads, 0, s>>>(n, indptr, indices, vals, x, y);
  else k_spmv<G, false><<<grid, kSpmvThreads, 0, s>>>(n, indptr, indices, vals, x, y);
  return hipGetLastError();
}

// ------------------------------------------- adding into another matrix
// The plan's CSR (rows = test dofs) added into a caller matrix whose pattern
// holds it.  CSR target: one thread per row walks both sorted rows (the
// target's row is a superset).  CSC target (GetFEM's col_matrix orientation:
// column = trial dof, sorted rows = test dofs): each entry (r, c) is found by
// a binary search in the target's column c.  An entry the target lacks sets
// bit 8 of the error flag (the value is dropped).
__global__ void k_add_into_csr(int64_t n, const int64_t *__restrict__ ip, const int32_t *__restrict__ ix,
                               const double *__restrict__ v, const int64_t *__restrict__ tip,
                               const int32_t *__restrict__ tix, double *__restrict__ tv, int *__restrict__ err) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= n) return;
  int64_t t = tip[row];
  const int64_t te = tip[row + 1];
  for (int64_t k = ip[row]; k < ip[row + 1]; ++k) {
    const int32_t c = ix[k];
    while (t < te && tix[t] < c) ++t;
    if (t < te && tix[t] == c) tv[t] += v[k];
    else atomicOr(err, 8);
  }
}

__global__ void k_add_into_csc(int64_t n, const int64_t *__restrict__ ip, const int32_t *__restrict__ ix,
                               const double *__restrict__ v, const int64_t *__restrict__ tcp,
                               const int32_t *__restrict__ tri, double *__restrict__ tv, int *__restrict__ err) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= n) return;
  for (int64_t k = ip[row]; k < ip[row + 1]; ++k) {
    const int32_t c = ix[k];
    int64_t lo = tcp[c], hi = tcp[c + 1];
    while (lo < hi) {
      const int64_t mid = (lo + hi) / 2;
      if (tri[mid] < row) lo = mid + 1;
      else hi = mid;
    }
    if (lo < tcp[c + 1] && tri[lo] == row) tv[lo] += v[k];
    else atomicOr(err, 8);
  }
}

// union of two CSR patterns with the same rows: per-row merge counts, then
// the merged columns and, for every entry of either input, its position in
// the union
__global__ void k_union_count(int64_t n, const int64_t *__restrict__ ipa, const int32_t *__restrict__ ixa,
                              const int64_t *__restrict__ ipb, const int32_t *__restrict__ ixb,
                              int64_t *__restrict__ cnt) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= n) return;
  int64_t a = ipa[row], ae = ipa[row + 1], b = ipb[row], be = ipb[row + 1], m = 0;
  while (a < ae || b < be) {
    const int32_t ca = a < ae ? ixa[a] : INT32_MAX, cb = b < be ? ixb[b] : INT32_MAX;
    a += ca <= cb;
    b += cb <= ca;
    ++m;
  }
  cnt[row] = m;
}

__global__ void k_union_fill(int64_t n, const int64_t *__restrict__ ipa, const int32_t *__restrict__ ixa,
                             const int64_t *__restrict__ ipb, const int32_t *__restrict__ ixb,
                             const int64_t *__restrict__ ipu, int32_t *__restrict__ ixu,
                             int64_t *__restrict__ mapa, int64_t *__restrict__ mapb) {
  const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= n) return;
  int64_t a = ipa[row], ae = ipa[row + 1], b = ipb[row], be = ipb[row + 1], u = ipu[row];
  while (a < ae || b < be) {
    const int32_t ca = a < ae ? ixa[a] : INT32_MAX, cb = b < be ? ixb[b] : INT32_MAX;
    const int32_t c = ca < cb ? ca : cb;
    ixu[u] = c;
    if (ca == c) mapa[a++] = u;
    if (cb == c) mapb[b++] = u;
    ++u;
  }
}

// out[map[k]] += v[k] (map injective: no two entries share a target)
__global__ void k_scatter_add(int64_t nnz, const int64_t *__restrict__ map, const double *__restrict__ v,
                              double *__restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nnz) out[map[k]] += v[k];
}

// dst[k] = src[map[k]] (composition of position maps)
__global__ void k_gather_i64(int64_t n, const int64_t *__restrict__ map, const int64_t *__restrict__ src,
                             int64_t *__restrict__ dst) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) dst[k] = src[map[k]];
}

// ---------------------------------------------- transposition (CSC export)
// the entries' rows and positions, before their stable sort by column; a
// group of 8 lanes per row
__global__ void k_csc_entries(int64_t n, const int64_t *__restrict__ ip, int32_t *__restrict__ row,
                              uint32_t *__restrict__ pos) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, r = t / 8;
  if (r >= n) return;
  const int64_t e = ip[r + 1];
  for (int64_t k = ip[r] + t % 8; k < e; k += 8) {
    row[k] = (int32_t)r;
    pos[k] = (uint32_t)k;
  }
}

// the sorted entries' rows and values, and the column pointers: an entry opens
// the columns after the previous entry's up to its own
__global__ void k_csc_fill(int64_t n, int64_t nnz, const int32_t *__restrict__ col, const uint32_t *__restrict__ pos,
                           const int32_t *__restrict__ row, const double *__restrict__ v, int64_t *__restrict__ cp,
                           uint32_t *__restrict__ rows, double *__restrict__ vals) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const uint32_t p = pos[k];
  rows[k] = (uint32_t)row[p];
  if (vals) vals[k] = v[p];
  for (int64_t c = k ? (int64_t)col[k - 1] + 1 : 0; c <= col[k]; ++c) cp[c] = k;
  if (k == nnz - 1)
    for (int64_t c = (int64_t)col[k] + 1; c <= n; ++c) cp[c] = nnz;
}

__global__ void k_fill_f64(int64_t n, double *__restrict__ p, double v) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = v;
}

// ---------------------------------------------------------------- CG
// The recurrence's scalars after an iteration; two of them, the launches of
// an iteration reading one and writing the other.  done: the loop has ended
// (the launches that follow in the batch do nothing but hand the state on).
struct CgScal {
  double rz, rr, bb, pq;
  int it, done;
};

// Lane exchanges of doubles: data-parallel moves within rows of 16 lanes, swaps
// across them (a move costs a few cycles, a shuffle through the LDS unit some fifty).
struct Dbl2 {
  double a, b;
};
__device__ __forceinline__ uint32_t lo32(double v) { return (uint32_t)__builtin_bit_cast(uint64_t, v); }
__device__ __forceinline__ uint32_t hi32(double v) { return (uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32); }
__device__ __forceinline__ double dbl(uint32_t lo, uint32_t hi) {
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// {a's lower 32 lanes, b's lower}, {a's upper, b's upper}
__device__ __forceinline__ Dbl2 swap32(double a, double b) {
  const auto l = __builtin_amdgcn_permlane32_swap(lo32(a), lo32(b), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(hi32(a), hi32(b), false, false);
  return {dbl(l[0], h[0]), dbl(l[1], h[1])};
}
// by rows of 16 lanes: {a0 b0 a2 b2}, {a1 b1 a3 b3}
__device__ __forceinline__ Dbl2 swap16(double a, double b) {
  const auto l = __builtin_amdgcn_permlane16_swap(lo32(a), lo32(b), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi32(a), hi32(b), false, false);
  return {dbl(l[0], h[0]), dbl(l[1], h[1])};
}
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  return v + dbl(__builtin_amdgcn_update_dpp(0, (int)lo32(v), CTRL, 0xf, 0xf, true),
                 __builtin_amdgcn_update_dpp(0, (int)hi32(v), CTRL, 0xf, 0xf, true));
}
// sum over each G lanes (16, 32 or 64), every lane gets its group's: the tree
// of lane ^ G/2, ..., lane ^ 1
template <int G>
__device__ __forceinline__ double group_sum(double v) {
  if constexpr (G == 64) {
    const Dbl2 r = swap32(v, v);
    v = r.a + r.b;
  }
  if constexpr (G >= 32) {
    const Dbl2 r = swap16(v, v);
    v = r.a + r.b;
  }
  v = dpp_add<0x128>(v);  // row_ror 8
  v = dpp_add<0x124>(v);  // row_ror 4: the same as lane ^ 4, the sums repeat every 8 lanes
  v = dpp_add<0x4e>(v);   // quad_perm 2 3 0 1
  return dpp_add<0xb1>(v);  // quad_perm 1 0 3 2
}

// sum over the block, every thread gets it: thread t and t + 128, then t + 64,
// t + 32, ..., t + 1
__device__ __forceinline__ double block_sum(double v, double *sh) {
  __syncthreads();  // the last use of sh
  sh[threadIdx.x] = v;
  __syncthreads();
  const int l = threadIdx.x & 63;
  return group_sum<64>((sh[l] + sh[l + 128]) + (sh[l + 64] + sh[l + 192]));
}

// the sum of a launch's n partials, in a fixed order, by every block that needs it
__device__ __forceinline__ double partials_sum(const double *__restrict__ part, int n, double *sh) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += kRedThreads) s += part[i];
  return block_sum(s, sh);
}

// inverse diagonal (0 where the diagonal is absent or zero: that dof is left alone)
__global__ void k_inv_diag(int64_t n, const int64_t *__restrict__ indptr,
                           const int32_t *__restrict__ indices, const double *__restrict__ vals,
                           double *__restrict__ dinv) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t lo = indptr[i], hi = indptr[i + 1];
  double d = 0.0;
  while (lo < hi) {  // sorted columns: binary search for column i
    const int64_t mid = (lo + hi) / 2;
    const int32_t c = indices[mid];
    if (c == i) { d = vals[mid]; break; }
    if (c < i) lo = mid + 1;
    else hi = mid;
  }
  dinv[i] = d != 0.0 ? 1.0 / d : 0.0;
}

// 3x3 block Jacobi for vector fields (dof = 3 node + component): the inverse
// of each node's diagonal block; a singular block (e.g. rows cleared by a
// Dirichlet simplification) falls back to the inverse diagonal of that node
__global__ void k_inv_block3(int64_t nn, const int64_t *__restrict__ indptr,
                             const int32_t *__restrict__ indices, const double *__restrict__ vals,
                             const uint16_t *__restrict__ nslots, double *__restrict__ minv) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= nn) return;
  double M[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  auto first = [&](int64_t row) {  // first entry with a column >= 3u (sorted columns)
    int64_t lo = indptr[row], hi = indptr[row + 1];
    while (lo < hi) {
      const int64_t mid = (lo + hi) / 2;
      if (indices[mid] < 3 * u) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  if (nslots && (nslots[u] & 0x8000)) {  // a full node: the three rows have the same columns
    const int64_t len = 3 * (nslots[u] & 0x7fff), lo = first(3 * u);
    if (lo < indptr[3 * u + 1] && indices[lo] == 3 * u)
      for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) M[a][b] = vals[lo + a * len + b];
  } else {
    for (int a = 0; a < 3; ++a) {
      const int64_t row = 3 * u + a;
      for (int64_t k = first(row); k < indptr[row + 1] && indices[k] < 3 * u + 3; ++k) M[a][indices[k] - 3 * u] = vals[k];
    }
  }
  const double c00 = M[1][1] * M[2][2] - M[1][2] * M[2][1], c01 = M[1][2] * M[2][0] - M[1][0] * M[2][2],
               c02 = M[1][0] * M[2][1] - M[1][1] * M[2][0];
  const double det = M[0][0] * c00 + M[0][1] * c01 + M[0][2] * c02;
  double *o = minv + 9 * u;
  const double scale = fabs(M[0][0]) + fabs(M[1][1]) + fabs(M[2][2]);
  if (det != 0.0 && fabs(det) > 1e-300 && fabs(det) > 1e-14 * scale * scale * scale) {
    const double id = 1.0 / det;
    o[0] = c00 * id; o[1] = (M[0][2] * M[2][1] - M[0][1] * M[2][2]) * id;
    o[2] = (M[0][1] * M[1][2] - M[0][2] * M[1][1]) * id;
    o[3] = c01 * id; o[4] = (M[0][0] * M[2][2] - M[0][2] * M[2][0]) * id;
    o[5] = (M[0][2] * M[1][0] - M[0][0] * M[1][2]) * id;
    o[6] = c02 * id; o[7] = (M[0][1] * M[2][0] - M[0][0] * M[2][1]) * id;
    o[8] = (M[0][0] * M[1][1] - M[0][1] * M[1][0]) * id;
  } else {
    for (int t = 0; t < 9; ++t) o[t] = 0.0;
    for (int a = 0; a < 3; ++a) o[4 * a] = M[a][a] != 0.0 ? 1.0 / M[a][a] : 0.0;
  }
}

// z = M^-1 r on one unit: a dof (QB = 1, inverse diagonal) or a node's three
// dofs (QB = 3, inverse 3x3 block)
template <int QB>
__device__ __forceinline__ void precond(const double *__restrict__ minv, int64_t u, const double (&r)[QB],
                                        double (&z)[QB]) {
  if constexpr (QB == 1) {
    z[0] = minv[u] * r[0];
  } else {
    const double *M = minv + 9 * u;
    for (int a = 0; a < 3; ++a) z[a] = M[3 * a] * r[0] + M[3 * a + 1] * r[1] + M[3 * a + 2] * r[2];
  }
}

// r = b - r (r holds K x on entry), z = M^-1 r, p = z; partials of r.z, r.r, b.b
template <int QB>
__global__ __launch_bounds__(kRedThreads) void k_cg_start(int64_t nu, const double *__restrict__ b,
                                                          const double *__restrict__ minv,
                                                          double *__restrict__ r, double *__restrict__ z,
                                                          double *__restrict__ p, double *__restrict__ part) {
  __shared__ double sh[kRedThreads];
  double rz = 0, rr = 0, bb = 0;
  for (int64_t u = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; u < nu; u += (int64_t)gridDim.x * kRedThreads) {
    double ri[QB], zi[QB];
    for (int a = 0; a < QB; ++a) ri[a] = b[QB * u + a] - r[QB * u + a];
    precond<QB>(minv, u, ri, zi);
    for (int a = 0; a < QB; ++a) {
      const int64_t i = QB * u + a;
      r[i] = ri[a]; z[i] = zi[a]; p[i] = zi[a];
      rz += ri[a] * zi[a]; rr += ri[a] * ri[a]; bb += b[i] * b[i];
    }
  }
  rz = block_sum(rz, sh); rr = block_sum(rr, sh); bb = block_sum(bb, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = rz; part[gridDim.x + blockIdx.x] = rr; part[2 * gridDim.x + blockIdx.x] = bb;
  }
}

// whether the loop stops at |r|^2 = rr: gmm::cg's test on |r| / |b|
__device__ __forceinline__ bool cg_stops(double rr, double bb, double rtol) { return !(sqrt(rr) / sqrt(bb) > rtol); }

__global__ __launch_bounds__(kRedThreads) void k_cg_first(const double *__restrict__ part, int n, double rtol,
                                                          CgScal *__restrict__ sc) {
  __shared__ double sh[kRedThreads];
  const double rz = partials_sum(part, n, sh), rr = partials_sum(part + n, n, sh);
  const double bb = partials_sum(part + 2 * n, n, sh);
  if (threadIdx.x == 0) *sc = CgScal{rz, rr, bb, 0.0, 0, bb == 0.0 || cg_stops(rr, bb, rtol)};
}

// Node lists of the full nodes (every component pair of every neighbour
// stored): their three rows hold the same columns, whole triples in order, so
// one int per neighbour node stands for nine column indices.  The list of the
// node whose values start at b0 starts at b0 / 9, which leaves each its room.
__global__ void k_cg_nodes(int64_t nn, const uint16_t *__restrict__ nslots, const int64_t *__restrict__ indptr,
                           const int32_t *__restrict__ indices, int32_t *__restrict__ nodes) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, u = t / 8;
  if (u >= nn || !(nslots[u] & 0x8000)) return;
  const int64_t b0 = indptr[3 * u];
  const int ns = nslots[u] & 0x7fff;
  for (int s = (int)(t % 8); s < ns; s += 8) nodes[b0 / 9 + s] = indices[b0 + 3 * s] / 3;
}

// q = K p (sc null: no iteration, the product of the start).
// The blocks of an XCD sweep one eighth of the units, so that the x that
// neighbouring rows share stays in its L2.
// A row per G lanes (scalar fields, workspace matrices and short rows).
template <int G>
__global__ __launch_bounds__(kRedThreads, 8) void k_cg_spmv(int64_t n, int64_t chunk,
                                                            const int64_t *__restrict__ indptr,
                                                            const int32_t *__restrict__ indices,
                                                            const double *__restrict__ vals,
                                                            const double *__restrict__ p, double *__restrict__ q,
                                                            const CgScal *__restrict__ sc) {
  if (sc && sc->done) return;
  constexpr int kPer = kRedThreads / G;
  const int lane = threadIdx.x % G;
  const int64_t first = (int64_t)(blockIdx.x & 7) * chunk, last = min(n, first + chunk);
  const int64_t step = (int64_t)(gridDim.x >> 3) * kPer;
  for (int64_t u = first + (int64_t)(blockIdx.x >> 3) * kPer + threadIdx.x / G; u < last; u += step) {
    double s = 0.0;
    const int64_t e = indptr[u + 1];
    for (int64_t k = indptr[u] + lane; k < e; k += G) s += vals[k] * p[indices[k]];
    for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
    if (lane == 0) q[u] = s;
  }
}

// A node's three rows per wavefront (3x3 block Jacobi's fields); a column's x
// serves all three.  Bound by HBM: 8 bytes an entry and, in full nodes, 4/9
// for its index.  A full node's columns go in tiles of 64; the next tile's
// node ids and values are issued between this tile's x and its sums, so that
// a tile costs one memory latency, not three (the loads of a wavefront return
// in order: issued before the x they would have to arrive first).  The node's
// start and slot count are the same for every lane and come by scalar loads,
// a node ahead.
// G: lanes of a row's sum, k_spmv's (16 or 32).  A row's sum there is G chains
// and a tree, and 40 unconverged iterations turn another order's last bits into
// differences of up to 1e-9 (seen over random right-hand sides), so the tile's
// 64 products are dealt to the same G chains: lane swaps put a row's tile, G
// columns after G columns, on the row's own G lanes (two rows share a register
// at 32, all three at 16).
// Every other product goes through the matrix backwards (`back`), so that it
// begins with what the last one left in the memory-side cache (256 MB): a matrix
// of about that size, swept one way, would find none of it.
// Measured at P2 elasticity, 24^3 x 6 (367,000 rows, 28.7 M entries, 242 MB): 68 us
// (one way 72; the same with 64 chains a row) against 111 us for a row per 32
// lanes (12 bytes an entry, two latencies a row); 82 us with the values loaded
// non-temporally (rows share cache lines: they were fetched twice), 95-146 us
// with a node per 16 or 32 lanes, 115 us at half the wavefronts.
template <int G>
__global__ __launch_bounds__(kRedThreads, 8) void k_cg_spmv3(int64_t nn, int64_t chunk,
                                                             const int64_t *__restrict__ indptr,
                                                             const int32_t *__restrict__ indices,
                                                             const double *__restrict__ vals,
                                                             const uint16_t *__restrict__ nslots,
                                                             const int32_t *__restrict__ nodes,
                                                             const double *__restrict__ p, double *__restrict__ q,
                                                             const CgScal *__restrict__ sc, bool back) {
  if (sc && sc->done) return;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t first = (int64_t)(blockIdx.x & 7) * chunk, last = min(nn, first + chunk);
  int64_t step = (int64_t)(gridDim.x >> 3) * (kRedThreads / 64);
  struct Node {
    int64_t b0;      // its first value
    int r1, r2, r3;  // rows 1 and 2 and the end, from there
    int len;         // columns of the longest row
    bool full;
  };
  auto node = [&](int64_t v) {
    const int64_t b0 = indptr[3 * v];
    Node d{b0, (int)(indptr[3 * v + 1] - b0), (int)(indptr[3 * v + 2] - b0), (int)(indptr[3 * v + 3] - b0), 0,
           (nslots[v] & 0x8000) != 0};
    d.len = max(d.r1, max(d.r2 - d.r1, d.r3 - d.r2));
    return d;
  };
  // a tile's columns and values; indices past a row's end are clamped to the
  // node's last entry and their products left out of the sums
  int c0 = 0, c1 = 0, c2 = 0;
  double v0 = 0.0, v1 = 0.0, v2 = 0.0;
  auto load = [&](const Node &d, int k0) {
    const int k = k0 + lane;
    const unsigned i0 = min(k, d.r3 - 1), i1 = min(d.r1 + k, d.r3 - 1), i2 = min(d.r2 + k, d.r3 - 1);
    if (d.full) {
      c0 = (nodes + d.b0 / 9)[(unsigned)min(k, d.len - 1) / 3];
    } else {
      const int32_t *ix = indices + d.b0;
      c0 = ix[i0];
      c1 = ix[i1];
      c2 = ix[i2];
    }
    const double *v = vals + d.b0;
    v0 = v[i0];
    v1 = v[i1];
    v2 = v[i2];
  };
  int64_t u = first + (int64_t)(blockIdx.x >> 3) * (kRedThreads / 64) + w;
  if (back && u < last) {  // the same nodes, last to first
    u += (last - 1 - u) / step * step;
    step = -step;
  }
  Node cur{};
  if (u < last) {
    cur = node(u);
    if (cur.len) load(cur, 0);
  }
  for (; u >= first && u < last; u += step) {
    const Node nxt = node(max(first, min(u + step, last - 1)));
    const int l0 = cur.r1, l1 = cur.r2 - cur.r1, l2 = cur.r3 - cur.r2;  // the rows' lengths
    double s = 0.0, s2 = 0.0;
    if (!cur.len && nxt.len) load(nxt, 0);
    for (int k0 = 0; k0 < cur.len; k0 += 64) {
      const int k = k0 + lane;
      double x0, x1, x2;
      if (cur.full) {
        x0 = x1 = x2 = p[3 * (int64_t)c0 + (unsigned)min(k, cur.len - 1) % 3];
      } else {
        x0 = p[c0];
        x1 = p[c1];
        x2 = p[c2];
      }
      const double a0 = v0, a1 = v1, a2 = v2;
      if (k0 + 64 < cur.len) load(cur, k0 + 64);
      else if (nxt.len) load(nxt, 0);
      const int kg = k0 + lane % G;
      if constexpr (G == 32) {  // s: row 0 in the lower lanes, row 1 in the upper; s2: row 2 in both
        const Dbl2 a = swap32(a0, a1), x = swap32(x0, x1), b = swap32(a2, a2), y = swap32(x2, x2);
        const int l01 = lane < 32 ? l0 : l1;
        if (kg < l01) s = fma(a.a, x.a, s);
        if (kg < l2) s2 = fma(b.a, y.a, s2);
        if (kg + 32 < l01) s = fma(a.b, x.b, s);
        if (kg + 32 < l2) s2 = fma(b.b, y.b, s2);
      } else {  // s: rows 0, 1 and 2 in the first three 16 lanes
        const Dbl2 a01 = swap16(a0, a1), a22 = swap16(a2, a2), x01 = swap16(x0, x1), x22 = swap16(x2, x2);
        const Dbl2 a = swap32(a01.a, a22.a), x = swap32(x01.a, x22.a);
        const Dbl2 b = swap32(a01.b, a22.b), y = swap32(x01.b, x22.b);
        const int l = lane < 16 ? l0 : (lane < 32 ? l1 : l2);
        if (kg < l) s = fma(a.a, x.a, s);
        if (kg + 16 < l) s = fma(b.a, y.a, s);
        if (kg + 32 < l) s = fma(a.b, x.b, s);
        if (kg + 48 < l) s = fma(b.b, y.b, s);
      }
    }
    s = group_sum<G>(s);
    if constexpr (G == 32) {
      s2 = group_sum<G>(s2);
      if (lane == 0 || lane == 32) q[3 * u + (lane >> 5)] = s;
      if (lane == 1) q[3 * u + 2] = s2;
    } else {
      if (lane % 16 == 0 && lane < 48) q[3 * u + (lane >> 4)] = s;
    }
    cur = nxt;
  }
}

// partials of p.q, apart from the product, whose blocks hold the rows in another
// order than the one the sum is taken in: 4.8 us at 367,000 rows, q still in the
// caches; in the product (another order of the sum) it came free
__global__ __launch_bounds__(kRedThreads) void k_cg_dot(int64_t n, const double *__restrict__ p,
                                                        const double *__restrict__ q,
                                                        const CgScal *__restrict__ sc,
                                                        double *__restrict__ part) {
  __shared__ double sh[kRedThreads];
  if (sc->done) return;
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kRedThreads)
    s += p[i] * q[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// alpha = r.z / p.q; x += alpha p, r -= alpha q, z = M^-1 r; partials of r.z and r.r
template <int QB>
__global__ __launch_bounds__(kRedThreads) void k_cg_update(int64_t nu, CgScal *__restrict__ sc,
                                                           const double *__restrict__ ppart, int np,
                                                           const double *__restrict__ p,
                                                           const double *__restrict__ q,
                                                           const double *__restrict__ minv,
                                                           double *__restrict__ x, double *__restrict__ r,
                                                           double *__restrict__ z, double *__restrict__ part) {
  __shared__ double sh[kRedThreads];
  if (sc->done) return;
  const double pq = partials_sum(ppart, np, sh), alpha = pq != 0.0 ? sc->rz / pq : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) sc->pq = pq;  // for the next launch; none of this one reads it
  double rz = 0, rr = 0;
  for (int64_t u = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; u < nu; u += (int64_t)gridDim.x * kRedThreads) {
    double ri[QB], zi[QB];
    for (int a = 0; a < QB; ++a) {
      const int64_t i = QB * u + a;
      x[i] += alpha * p[i];
      ri[a] = r[i] - alpha * q[i];
    }
    precond<QB>(minv, u, ri, zi);
    for (int a = 0; a < QB; ++a) {
      const int64_t i = QB * u + a;
      r[i] = ri[a]; z[i] = zi[a];
      rz += ri[a] * zi[a]; rr += ri[a] * ri[a];
    }
  }
  rz = block_sum(rz, sh); rr = block_sum(rr, sh);
  if (threadIdx.x == 0) { part[blockIdx.x] = rz; part[gridDim.x + blockIdx.x] = rr; }
}

// beta = (r.z) / (r.z before); p = z + beta p; the next iteration's scalars
__global__ __launch_bounds__(kRedThreads) void k_cg_direction(int64_t n, const CgScal *__restrict__ sc,
                                                              const double *__restrict__ part, int np, double rtol,
                                                              const double *__restrict__ z, double *__restrict__ p,
                                                              CgScal *__restrict__ next) {
  __shared__ double sh[kRedThreads];
  if (sc->done) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *next = *sc;
    return;
  }
  const double rz = partials_sum(part, np, sh), rr = partials_sum(part + np, np, sh);
  const double beta = sc->rz != 0.0 ? rz / sc->rz : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0)  // p.q <= 0: K not positive definite along p
    *next = CgScal{rz, rr, sc->bb, sc->pq, sc->it + 1, sc->pq <= 0.0 || cg_stops(rr, sc->bb, rtol)};
  for (int64_t i = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kRedThreads)
    p[i] = z[i] + beta * p[i];
}

unsigned nb256(int64_t n) { return (unsigned)((n + 255) / 256); }

// ---------------------------------------------------------- dof constraints
// fixed[i] = 1 for a constrained dof, go[i] its prescribed value.  One
// thread per row; the row's entries are read before any is cleared, so the
// symmetric linear right-hand side correction uses the assembled K.
__global__ void k_dof_constraints(int64_t n, const int64_t *__restrict__ indptr,
                                  const int32_t *__restrict__ indices, double *__restrict__ vals,
                                  const uint8_t *__restrict__ fixed, const double *__restrict__ go,
                                  const double *__restrict__ pr, double *__restrict__ rhs, int flags,
                                  int *__restrict__ err) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const bool mat = flags & GFX_BUILD_MATRIX, vec = (flags & GFX_BUILD_RHS) && rhs;
  const bool lin = flags & GFX_MODEL_LINEAR, sym = flags & GFX_MODEL_SYMMETRIC;
  const int64_t b = indptr[i], e = indptr[i + 1];
  if (fixed[i]) {
    if (vec) rhs[i] = lin ? go[i] : go[i] - (pr ? pr[i] : 0.0);
    if (mat) {
      bool diag = false;
      for (int64_t k = b; k < e; ++k) {
        const bool d = indices[k] == i;
        vals[k] = d ? 1.0 : 0.0;
        diag |= d;
      }
      if (!diag) atomicOr(err, 4);
    }
    return;
  }
  if (vec && lin && sym) {  // rhs -= K(:, fixed) go
    double s = 0.0;
    for (int64_t k = b; k < e; ++k)
      if (fixed[indices[k]]) s += vals[k] * go[indices[k]];
    rhs[i] -= s;
  }
  if (mat && sym)
    for (int64_t k = b; k < e; ++k)
      if (fixed[indices[k]]) vals[k] = 0.0;
}

}  // namespace

hipError_t launch_dof_constraints(hipStream_t s, int64_t n, const int64_t *indptr, const int32_t *indices,
                                  double *vals, const uint8_t *fixed, const double *go, const double *pr,
                                  double *rhs, int flags, int *err) {
  if (n == 0) return hipSuccess;
  k_dof_constraints<<<nb256(n), 256, 0, s>>>(n, indptr, indices, vals, fixed, go, pr, rhs, flags, err);
  return hipGetLastError();
}

hipError_t launch_spmv(hipStream_t s, int64_t n, int64_t nnz, const int64_t *indptr,
                       const int32_t *indices, const double *vals, const double *x, double *y, bool acc) {
  if (n == 0) return hipSuccess;
  const double mean = (double)nnz / (double)n;
  if (mean <= 12) return spmv_g<4>(s, n, indptr, indices, vals, x, y, acc);
  if (mean <= 24) return spmv_g<8>(s, n, indptr, indices, vals, x, y, acc);
  if (mean <= 64) return spmv_g<16>(s, n, indptr, indices, vals, x, y, acc);
  return spmv_g<32>(s, n, indptr, indices, vals, x, y, acc);
}

hipError_t launch_add_into(hipStream_t s, bool csc, int64_t n, const int64_t *ip, const int32_t *ix,
                           const double *v, const int64_t *tp, const int32_t *ti, double *tv, int *err) {
  if (n == 0) return hipSuccess;
  if (csc) k_add_into_csc<<<nb256(n), 256, 0, s>>>(n, ip, ix, v, tp, ti, tv, err);
  else k_add_into_csr<<<nb256(n), 256, 0, s>>>(n, ip, ix, v, tp, ti, tv, err);
  return hipGetLastError();
}

hipError_t launch_union_count(hipStream_t s, int64_t n, const int64_t *ipa, const int32_t *ixa,
                              const int64_t *ipb, const int32_t *ixb, int64_t *cnt) {
  if (n == 0) return hipSuccess;
  k_union_count<<<nb256(n), 256, 0, s>>>(n, ipa, ixa, ipb, ixb, cnt);
  return hipGetLastError();
}

hipError_t launch_union_fill(hipStream_t s, int64_t n, const int64_t *ipa, const int32_t *ixa,
                             const int64_t *ipb, const int32_t *ixb, const int64_t *ipu, int32_t *ixu,
                             int64_t *mapa, int64_t *mapb) {
  if (n == 0) return hipSuccess;
  k_union_fill<<<nb256(n), 256, 0, s>>>(n, ipa, ixa, ipb, ixb, ipu, ixu, mapa, mapb);
  return hipGetLastError();
}

hipError_t launch_scatter_add(hipStream_t s, int64_t nnz, const int64_t *map, const double *v, double *out) {
  if (nnz == 0) return hipSuccess;
  k_scatter_add<<<nb256(nnz), 256, 0, s>>>(nnz, map, v, out);
  return hipGetLastError();
}

hipError_t launch_gather_i64(hipStream_t s, int64_t n, const int64_t *map, const int64_t *src, int64_t *dst) {
  if (n == 0) return hipSuccess;
  k_gather_i64<<<nb256(n), 256, 0, s>>>(n, map, src, dst);
  return hipGetLastError();
}

hipError_t launch_fill_f64(hipStream_t s, int64_t n, double *p, double v) {
  if (n == 0) return hipSuccess;
  k_fill_f64<<<nb256(n), 256, 0, s>>>(n, p, v);
  return hipGetLastError();
}

size_t csc_sort_bytes(int64_t nnz, int bits) {
  size_t bytes = 0;
  if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const int32_t *)nullptr, (int32_t *)nullptr,
                                         (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)nnz, 0, bits) !=
      hipSuccess)
    return 0;
  return bytes;
}

hipError_t csr_to_csc(hipStream_t s, int64_t n, int64_t nnz, int bits, const int64_t *ip, const int32_t *ix,
                      const double *v, void *tmp, size_t tmp_bytes, int32_t *row, uint32_t *pos, int32_t *col,
                      uint32_t *pos2, int64_t *cp, uint32_t *rows, double *vals) {
  k_csc_entries<<<nb256(8 * n), 256, 0, s>>>(n, ip, row, pos);
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, ix, col, pos, pos2, (int)nnz, 0, bits, s);
  if (e != hipSuccess) return e;
  k_csc_fill<<<nb256(nnz), 256, 0, s>>>(n, nnz, col, pos2, row, v, cp, rows, vals);
  return hipGetLastError();
}

// preconditioner storage (3 n: room for the 3x3 blocks) + r, z, p, q +
// partials + scalars, then the full nodes' lists (an int per 9 entries)
static size_t cg_vector_doubles(int64_t n) {
  return 7 * (size_t)n + 4 * kRedBlocks + 2 * sizeof(CgScal) / sizeof(double);
}
size_t cg_workspace_doubles(int64_t n, int64_t nnz) { return cg_vector_doubles(n) + (size_t)nnz / 18 + 2; }

// ------------------------------------------------------------------ GMRES
namespace {

constexpr int kGmBlocks = 256;  // partial sums per dot product (fixed order)
constexpr int kGmRows = 8;      // basis vectors per block of the multi-dot

// a row without diagonal (or a zero one) is left unscaled
__global__ void k_gm_fix_dinv(int64_t n, double *__restrict__ dinv) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && dinv[i] == 0.0) dinv[i] = 1.0;
}

// y = dinv x
__global__ void k_gm_scale_diag(int64_t n, const double *__restrict__ dinv, const double *x, double *y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = dinv[i] * x[i];
}

// w = b - w
__global__ void k_gm_sub(int64_t n, const double *__restrict__ b, double *__restrict__ w) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) w[i] = b[i] - w[i];
}

// partials of V_k . w for the basis vectors k0 .. k0 + kGmRows - 1 (k < nk)
__global__ __launch_bounds__(kRedThreads) void k_gm_multidot(int64_t n, int nk, const double *__restrict__ V,
                                                             const double *__restrict__ w,
                                                             double *__restrict__ part) {
  __shared__ double sh[kRedThreads];
  const int k0 = blockIdx.y * kGmRows;
  double acc[kGmRows];
  for (int r = 0; r < kGmRows; ++r) acc[r] = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; i < n; i += (int64_t)kGmBlocks * kRedThreads) {
    const double wi = w[i];
    for (int r = 0; r < kGmRows; ++r)
      if (k0 + r < nk) acc[r] += V[(int64_t)(k0 + r) * n + i] * wi;
  }
  for (int r = 0; r < kGmRows; ++r) {
    const double t = block_sum(acc[r], sh);  // uniform: every thread takes part
    if (threadIdx.x == 0 && k0 + r < nk) part[(int64_t)(k0 + r) * kGmBlocks + blockIdx.x] = t;
  }
}

// h_k (+)= sum of the partials of k, in a fixed order
__global__ __launch_bounds__(kRedThreads) void k_gm_sum(int nk, const double *__restrict__ part,
                                                        double *__restrict__ h, int accumulate) {
  __shared__ double sh[kRedThreads];
  const int k = blockIdx.x;
  double s = 0.0;
  for (int i = threadIdx.x; i < kGmBlocks; i += kRedThreads) s += part[(int64_t)k * kGmBlocks + i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0 && k < nk) h[k] = accumulate ? h[k] + s : s;
}

// w -= sum_k h_k V_k
__global__ void k_gm_project(int64_t n, int nk, const double *__restrict__ V, const double *__restrict__ h,
                             double *__restrict__ w) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double t = w[i];
  for (int k = 0; k < nk; ++k) t -= h[k] * V[(int64_t)k * n + i];
  w[i] = t;
}

// out = w * (1 / a)  with a = *anorm (0 leaves zeros)
__global__ void k_gm_normalize(int64_t n, const double *__restrict__ anorm, const double *__restrict__ w,
                               double *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const double a = *anorm;
  if (i < n) out[i] = a != 0.0 ? w[i] * (1.0 / a) : 0.0;
}

// x += sum_k y_k V_k
__global__ void k_gm_combine(int64_t n, int nk, const double *__restrict__ V, const double *__restrict__ y,
                             double *__restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double t = x[i];
  for (int k = 0; k < nk; ++k) t += y[k] * V[(int64_t)k * n + i];
  x[i] = t;
}

// ||w||^2 partials then the norm into *out
__global__ __launch_bounds__(kRedThreads) void k_gm_norm(int64_t n, const double *__restrict__ w,
                                                         double *__restrict__ part) {
  __shared__ double sh[kRedThreads];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kRedThreads + threadIdx.x; i < n; i += (int64_t)kGmBlocks * kRedThreads)
    s += w[i] * w[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
__global__ __launch_bounds__(kRedThreads) void k_gm_norm_final(const double *__restrict__ part,
                                                               double *__restrict__ out) {
  __shared__ double sh[kRedThreads];
  double s = 0.0;
  for (int i = threadIdx.x; i < kGmBlocks; i += kRedThreads) s += part[i];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) *out = sqrt(s);
}

// Givens rotation zeroing b in (a, b), as gmm::Givens_rotation
void givens(double a, double b, double &c, double &s) {
  if (b == 0.0) { c = 1.0; s = 0.0; return; }
  if (std::fabs(b) > std::fabs(a)) {
    const double t = a / b;
    s = 1.0 / std::sqrt(1.0 + t * t);
    c = s * t;
  } else {
    const double t = b / a;
    c = 1.0 / std::sqrt(1.0 + t * t);
    s = c * t;
  }
}
void rotate(double &x, double &y, double c, double s) {
  const double t = c * x + s * y;
  y = c * y - s * x;
  x = t;
}

}  // namespace

size_t gmres_workspace_doubles(int64_t n, int m) {
  return (size_t)(m + 1) * (size_t)n + 3 * (size_t)n + (size_t)(m + 2) * kGmBlocks + 2 * (size_t)(m + 2) + 8;
}

// gmm::gmres (src/gmm/gmm_solver_gmres.h:85-157): restarted, left
// preconditioned (gmm::ilu_precond, or the inverse diagonal), the stopping test on the
// preconditioned residual relative to ||M b||, a restart that makes no
// progress ten times in a row ends the solve.  The basis is orthogonalised by
// classical Gram-Schmidt applied twice (two batched passes per step, where
// gmm runs modified Gram-Schmidt one vector at a time): the same subspace,
// with the same orthogonality to working precision.  The Hessenberg matrix,
// its Givens rotations and the triangular solve live on the host.
hipError_t gmres_solve(hipStream_t s, int64_t n, int64_t nnz, const int64_t *indptr, const int32_t *indices,
                       const double *vals, const double *b, double *x, double rtol, int maxit, int m,
                       double *work, const IluData *ilu, int *iters, double *rel_res) {
  *iters = 0;
  *rel_res = 0.0;
  if (n == 0) return hipSuccess;
  if (m < 1) return hipErrorInvalidValue;
  double *V = work, *dinv = V + (size_t)(m + 1) * n, *w = dinv + n, *u = w + n;
  double *part = u + n, *hd = part + (size_t)(m + 2) * kGmBlocks, *yd = hd + (m + 2);
  double *anorm = yd + (m + 2);
  hipError_t e;
  const unsigned nb = nb256(n);
  auto norm = [&](const double *v, double &out) -> hipError_t {
    k_gm_norm<<<kGmBlocks, kRedThreads, 0, s>>>(n, v, part);
    k_gm_norm_final<<<1, kRedThreads, 0, s>>>(part, anorm);
    hipError_t er = hipMemcpyAsync(&out, anorm, 8, hipMemcpyDeviceToHost, s);
    if (er == hipSuccess) er = hipStreamSynchronize(s);
    return er;
  };
  k_inv_diag<<<nb, 256, 0, s>>>(n, indptr, indices, vals, dinv);
  k_gm_fix_dinv<<<nb, 256, 0, s>>>(n, dinv);
  // out = M^-1 in (in == out allowed): the ILU solves or the inverse diagonal
  auto prec = [&](const double *in, double *out) -> hipError_t {
    if (ilu) return ilu_apply(s, *ilu, indptr, indices, in, out);
    k_gm_scale_diag<<<nb, 256, 0, s>>>(n, dinv, in, out);
    return hipGetLastError();
  };
  // ||M b||
  if ((e = prec(b, w)) != hipSuccess) return e;
  double bn = 0.0;
  if ((e = norm(w, bn)) != hipSuccess) return e;
  if (bn == 0.0) {
    if ((e = hipMemsetAsync(x, 0, 8 * (size_t)n, s)) != hipSuccess) return e;
    return hipStreamSynchronize(s);
  }
  auto residual = [&](double &beta) -> hipError_t {  // w = M (b - A x), beta = ||w||
    hipError_t er = launch_spmv(s, n, nnz, indptr, indices, vals, x, w, false);
    if (er != hipSuccess) return er;
    k_gm_sub<<<nb, 256, 0, s>>>(n, b, w);
    if ((er = prec(w, w)) != hipSuccess) return er;
    return norm(w, beta);
  };
  double beta = 0.0;
  if ((e = residual(beta)) != hipSuccess) return e;
  double beta_old = beta;
  int blocked = 0, it = 0;
  std::vector<double> H((size_t)(m + 1) * m), cr(m + 1), sr(m + 1), g(m + 1), h(m + 2);
  while (beta / bn > rtol && it < maxit) {
    k_gm_normalize<<<nb, 256, 0, s>>>(n, anorm, w, V);  // anorm holds beta
    std::fill(g.begin(), g.end(), 0.0);
    g[0] = beta;
    int i = 0;
    do {
      // u = M A V_i, orthogonalised against V_0..V_i twice
      if ((e = launch_spmv(s, n, nnz, indptr, indices, vals, V + (size_t)i * n, u, false)) != hipSuccess) return e;
      if ((e = prec(u, u)) != hipSuccess) return e;
      const int nk = i + 1;
      const dim3 grid(kGmBlocks, (unsigned)((nk + kGmRows - 1) / kGmRows));
      for (int pass = 0; pass < 2; ++pass) {
        k_gm_multidot<<<grid, kRedThreads, 0, s>>>(n, nk, V, u, part);
        k_gm_sum<<<nk, kRedThreads, 0, s>>>(nk, part, pass == 0 ? hd : yd, 0);
        k_gm_project<<<nb, 256, 0, s>>>(n, nk, V, pass == 0 ? hd : yd, u);
      }
      if ((e = hipGetLastError()) != hipSuccess) return e;
      double a = 0.0;
      if ((e = norm(u, a)) != hipSuccess) return e;
      if ((e = hipMemcpy(h.data(), hd, 8 * (size_t)nk, hipMemcpyDeviceToHost)) != hipSuccess) return e;
      std::vector<double> h2((size_t)nk);
      if ((e = hipMemcpy(h2.data(), yd, 8 * (size_t)nk, hipMemcpyDeviceToHost)) != hipSuccess) return e;
      double *col = &H[(size_t)i * (m + 1)];  // column i of H (column-major)
      for (int k = 0; k < nk; ++k) col[k] = h[k] + h2[k];
      col[i + 1] = a;
      k_gm_normalize<<<nb, 256, 0, s>>>(n, anorm, u, V + (size_t)(i + 1) * n);
      for (int k = 0; k < i; ++k) rotate(col[k], col[k + 1], cr[k], sr[k]);
      givens(col[i], col[i + 1], cr[i], sr[i]);
      rotate(col[i], col[i + 1], cr[i], sr[i]);
      rotate(g[i], g[i + 1], cr[i], sr[i]);
      ++i;
      ++it;
    } while (std::fabs(g[i]) / bn > rtol && i < m && it < maxit);
    // y = H(0:i, 0:i)^{-1} g, x += V y
    std::vector<double> y(g.begin(), g.begin() + i);
    for (int r = i - 1; r >= 0; --r) {
      for (int c = r + 1; c < i; ++c) y[r] -= H[(size_t)c * (m + 1) + r] * y[c];
      y[r] /= H[(size_t)r * (m + 1) + r];
    }
    if ((e = hipMemcpyAsync(yd, y.data(), 8 * (size_t)i, hipMemcpyHostToDevice, s)) != hipSuccess) return e;
    k_gm_combine<<<nb, 256, 0, s>>>(n, i, V, yd, x);
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;  // y is read before it changes
    beta_old = std::min(beta, beta_old);
    if ((e = residual(beta)) != hipSuccess) return e;
    if (i < m - 1 || beta_old <= beta) ++blocked;
    else blocked = 0;
    if (blocked > 10) break;
  }
  *iters = it;
  *rel_res = beta / bn;
  return hipSuccess;
}


// the blocks of a product whose blocks do `per` units at a time, and the units of an XCD
static int cg_prod_blocks(int64_t nu, int per, int64_t &chunk) {
  chunk = (nu + 7) / 8;
  return (int)std::min<int64_t>(8 * std::max<int64_t>(1, (chunk + per - 1) / per), kMaxProdBlocks);
}

static hipError_t cg_product(hipStream_t s, int64_t n, int64_t nnz, const int64_t *indptr, const int32_t *indices,
                             const double *vals, const uint16_t *nslots, const int32_t *nodes, const double *p,
                             double *q, const CgScal *sc, bool back) {
  int64_t chunk;
  const double mean = (double)nnz / (double)n;  // the bounds of launch_spmv
  // a wavefront per node where a tile of its row has at least 24 of 64 columns
  // (one cube of P1 elements has less); 16 or 32 lanes a sum, as launch_spmv
  if (nslots && mean > 24) {
    const int nblocks = cg_prod_blocks(n / 3, kRedThreads / 64, chunk);
    auto k = mean > 64 ? k_cg_spmv3<32> : k_cg_spmv3<16>;
    k<<<(unsigned)nblocks, kRedThreads, 0, s>>>(n / 3, chunk, indptr, indices, vals, nslots, nodes, p, q, sc, back);
    return hipGetLastError();
  }
  auto run = [&](auto g) {
    constexpr int G = decltype(g)::value;
    const int nblocks = cg_prod_blocks(n, kRedThreads / G, chunk);
    k_cg_spmv<G><<<(unsigned)nblocks, kRedThreads, 0, s>>>(n, chunk, indptr, indices, vals, p, q, sc);
  };
  if (mean <= 12) run(std::integral_constant<int, 4>{});
  else if (mean <= 24) run(std::integral_constant<int, 8>{});
  else if (mean <= 64) run(std::integral_constant<int, 16>{});
  else run(std::integral_constant<int, 32>{});
  return hipGetLastError();
}

// One iteration's launches; cur and next: the scalars before and after it.
template <int QB>
static hipError_t cg_iterations(hipStream_t s, int64_t n, int64_t nnz, const int64_t *indptr, const int32_t *indices,
                                const double *vals, const uint16_t *nslots, const int32_t *nodes, const double *b,
                                double *x, double rtol, int maxit, double *work, CgScal *h) {
  double *minv = work, *r = work + 3 * n, *z = work + 4 * n, *p = work + 5 * n, *q = work + 6 * n;
  double *part = work + 7 * n, *ppart = part + 3 * kRedBlocks;
  CgScal *sc = reinterpret_cast<CgScal *>(ppart + kRedBlocks);
  const int64_t nu = n / QB;
  const int nb = (int)std::min<int64_t>(kRedBlocks, (nu + kRedThreads - 1) / kRedThreads);
  const int nd = (int)std::min<int64_t>(kRedBlocks, (n + kRedThreads - 1) / kRedThreads);
  hipError_t e;
  k_cg_start<QB><<<nb, kRedThreads, 0, s>>>(nu, b, minv, r, z, p, part);
  k_cg_first<<<1, kRedThreads, 0, s>>>(part, nb, rtol, sc);
  // batches: the host waits once for each; a batch is at most as long as all
  // before it, so that the launches after the end are never the most of them
  int it = 0, batch = 4;
  do {
    const int end = std::min(maxit, it + batch);
    for (; it < end; ++it) {
      CgScal *cur = sc + (it & 1), *next = sc + (~it & 1);
      if ((e = cg_product(s, n, nnz, indptr, indices, vals, nslots, nodes, p, q, cur, it & 1)) != hipSuccess) return e;
      k_cg_dot<<<nd, kRedThreads, 0, s>>>(n, p, q, cur, ppart);
      k_cg_update<QB><<<nb, kRedThreads, 0, s>>>(nu, cur, ppart, nd, p, q, minv, x, r, z, part);
      k_cg_direction<<<nd, kRedThreads, 0, s>>>(n, cur, part, nb, rtol, z, p, next);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(h, sc + (it & 1), sizeof *h, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
    batch = std::min(std::max(batch, it), 32);
  } while (!h->done && it < maxit);
  return hipSuccess;
}

hipError_t cg_solve(hipStream_t s, int64_t n, int64_t nnz, const int64_t *indptr, const int32_t *indices,
                    const double *vals, const uint16_t *nslots, const double *b, double *x, double rtol, int maxit,
                    int qb, double *work, int *iters, double *rel_res) {
  *iters = 0;
  *rel_res = 0.0;
  if (n == 0) return hipSuccess;
  if (qb != 1 && (qb != 3 || n % 3 != 0)) return hipErrorInvalidValue;
  double *minv = work, *r = work + 3 * n;
  int32_t *nodes = reinterpret_cast<int32_t *>(work + cg_vector_doubles(n));
  const int64_t nu = n / qb;
  hipError_t e;
  if (qb == 3) k_inv_block3<<<nb256(nu), 256, 0, s>>>(nu, indptr, indices, vals, nslots, minv);
  else k_inv_diag<<<nb256(n), 256, 0, s>>>(n, indptr, indices, vals, minv);
  if (qb != 3) nslots = nullptr;
  if (nslots) k_cg_nodes<<<nb256(8 * nu), 256, 0, s>>>(nu, nslots, indptr, indices, nodes);
  if ((e = cg_product(s, n, nnz, indptr, indices, vals, nslots, nodes, x, r, nullptr, false)) != hipSuccess) return e;
  CgScal h{};
  e = qb == 3 ? cg_iterations<3>(s, n, nnz, indptr, indices, vals, nslots, nodes, b, x, rtol, maxit, work, &h)
              : cg_iterations<1>(s, n, nnz, indptr, indices, vals, nslots, nodes, b, x, rtol, maxit, work, &h);
  if (e != hipSuccess) return e;
  if (h.bb == 0.0) {  // b = 0: x = 0 is the solution
    if ((e = hipMemsetAsync(x, 0, 8 * (size_t)n, s)) != hipSuccess) return e;
    return hipStreamSynchronize(s);
  }
  *iters = h.it;
  *rel_res = sqrt(h.rr) / sqrt(h.bb);
  return hipSuccess;
}

}  // namespace gfx
