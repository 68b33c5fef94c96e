// The order-2 polynomial route of the workspace: tangent matrices of the
// integrands the matrix kernels do not cover (several fem variables, blocks
// between two mesh_fems, data fields, polynomial nonlinearities), as
// ga_workspace::assembly(2) (src/getfem_generic_assembly_workspace.cc:791-936)
// runs them with the two-mesh_fem matrix instruction
// ga_instruction_matrix_assembly_mf_mf
// (src/getfem_generic_assembly_compile_and_exec.cc:5074-5189) and
// add_elem_matrix (:4853-4936).
//
// k_poly_mat   one wavefront per element and block: the element matrix
//              sum_q w_q |J| of the bilinear form that the program's outputs
//              give in the two fields' base functions, in registers; then the
//              element's threshold 1e-14 max|elem| (a zero element adds
//              nothing): entries at or below it are written as 0, so that
//              what is stored and not zero is what add_elem_matrix inserts.
// k_poly_ref   the same for affine elements and outputs without fem fields,
//              through the reference tensor.
// The matrix.  Which entries of which elements meet in a matrix entry depends
// on the dof tables alone, so it is worked out once per set of expressions
// (poly_structure): every candidate (block, element, entry) sorted by (row,
// column), stably, so that the candidates of an entry stay in the order in
// which add_elem_matrix adds them.  An assembly then sums each entry's
// candidates in that order (k_poly_runs) straight into the CSR of the last
// assembly, and sees on the way whether the entries that have any candidate
// are still the stored ones; only where they are not are the CSR's rows and
// columns made anew (poly_pattern).
// Beyond 2^31 candidates, or the workspace's own limit, the kept entries are
// sorted at every assembly instead (k_poly_emit, poly_to_csr).
#include <hip/hip_runtime.h>

#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "gfx_internal.h"

namespace gfx {
namespace {

constexpr int kPm = 64;  // one wavefront
constexpr int kPoly1d = 256;

__device__ __forceinline__ double pm_wave_max(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ int pm_wave_sum(int v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Bound by FP64 issue and the LDS.  A lane owns tiles of one column (j, b)
// and the rows of kPmNodes test nodes, NP tiles in all, with their sums in
// registers.  Per point the products of the outputs with the trial field's
// base functions, U[(a, p)][(j, b)] = sum_r O[(a, p), (b, r)] psi_j[r], are
// formed once in LDS and then serve every test node: 5 products an entry and
// point instead of 21 with a load each.  The test function's slots [P0, P1)
// are those in use (its value, its gradient or both); so are r's.  Outputs
// without a fem field are the same at every point and evaluated once.
// A point's sum over p is formed before w_q |J| takes it into the entry, as
// the reference does: adding the products one by one rounded the entry three
// or four times a point, and its error against exact sums grew by 10 % (P2) to
// 60 % (P3).
// Measured, (1 + p^2) Grad_u:Grad_Test_u - p^2 Div_Test_u + p^3 Test_p with u P2
// vector and p P1 on 15^3 x 6 = 20,250 elements: the three blocks 1.60 ms, a
// whole assembly 1.73 ms against 6.26 ms with an LDS load a product and the
// sums in LDS.
constexpr int kPmNodes = 5;

template <int QT, int NP, int P0, int P1>
__global__ __launch_bounds__(kPm) void k_poly_mat(PolyMatArgs a) {
  extern __shared__ double lds_pm[];
  const ScalarField &ft = a.f[a.vt], &fs = a.f[a.vs];
  const int qs = fs.qdim, ndt = ft.nd, nds = fs.nd, nc = nds * qs, ne = ndt * QT * nc, w4 = 4 * qs;
  double *T = lds_pm;                  // symbols
  double *O = T + a.nsym;              // outputs
  double *bt = O + a.nout;             // [node][4]: phi, real gradient
  double *bs = bt + 4 * ndt;
  double *U = bs + 4 * nds;            // [(a, p)][column]
  double *V = U + 4 * QT * nc;         // the fields' nodal values, [field][node][component]
  const int64_t e = blockIdx.x;
  const int t = threadIdx.x;
  // geometry, the same on every lane: once for an affine tetrahedron, at
  // every point for a hexahedron (a degenerate point leaves the element,
  // uniformly)
  const int32_t *cv = a.cvx + (int64_t)a.nv * e;
  double B[9], aJ = 0.0;
  bool ok = poly_geometry(a.pts, cv, a.nv, a.gN, B, aJ);
  for (int q = 1; ok && a.gN && q < a.nq; ++q) {  // every hexahedron point checked first
    double Bq[9], aq;
    ok = poly_geometry(a.pts, cv, a.nv, a.gN + (int64_t)q * a.nv * 3, Bq, aq);
  }
  double *dst = a.elem + e * ne;
  if (!ok) {
    if (t == 0) atomicOr(a.err, 1);
    for (int x = t; x < ne; x += kPm) dst[x] = 0.0;
    return;
  }
  for (int c = t; c < a.nconst; c += kPm) T[a.const_off + c] = a.consts[c];
  if (a.varying) {
    double *v = V;
    for (int fi = 0; fi < a.nf; ++fi) {
      const ScalarField &f = a.f[fi];
      const int n = f.nd * f.qdim;
      for (int x = t; x < n; x += kPm) {
        const int i = x / f.qdim;
        v[x] = f.U[(int64_t)f.dofs[e * f.nd + i] + (x - i * f.qdim)];
      }
      v += n;
    }
  }
  __syncthreads();
  auto outputs = [&]() {  // one lane per output, its monomials in a fixed order
    for (int o = t; o < a.nout; o += kPm) {
      double s = 0.0;
      for (int m = a.mptr[o]; m < a.mptr[o + 1]; ++m) {
        double v = a.mcoef[m];
        for (int x = a.moff[m]; x < a.moff[m + 1]; ++x) v *= T[a.msym[x]];
        s += v;
      }
      O[o] = s;
    }
  };
  if (!a.varying) outputs();
  // this lane's tiles: column, first test node
  const int groups = (ndt + kPmNodes - 1) / kPmNodes;
  int col[NP], row0[NP];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    const int x = t + k * kPm;
    const bool in = x < groups * nc;
    col[k] = in ? x % nc : 0;
    row0[k] = in ? x / nc * kPmNodes : ndt;  // ndt: no tile
  }
  double acc[NP][kPmNodes][QT];
#pragma unroll
  for (int k = 0; k < NP; ++k)
#pragma unroll
    for (int i = 0; i < kPmNodes; ++i)
#pragma unroll
      for (int c = 0; c < QT; ++c) acc[k][i][c] = 0.0;
  for (int q = 0; q < a.nq; ++q) {
    if (a.gN && q > 0) poly_geometry(a.pts, cv, a.nv, a.gN + (int64_t)q * a.nv * 3, B, aJ);
    // base functions of the two fields at the point
    for (int x = t; x < ndt + nds; x += kPm) {
      const bool test = x < ndt;
      const ScalarField &f = test ? ft : fs;
      const int i = test ? x : x - ndt;
      const double *h = f.gref + ((int64_t)q * f.nd + i) * 3;
      double *o = (test ? bt : bs) + 4 * i;
      o[0] = f.phi[q * f.nd + i];
      for (int b = 0; b < 3; ++b) o[1 + b] = B[3 * b] * h[0] + B[3 * b + 1] * h[1] + B[3 * b + 2] * h[2];
    }
    if (a.varying) {
      // symbol table: lane -> (field, component)
      int kc = t;
      const double *v0 = V;
      for (int fi = 0; fi < a.nf; ++fi) {
        const ScalarField &f = a.f[fi];
        if (kc >= 0 && kc < f.qdim) {
          double v = 0.0, r0 = 0.0, r1 = 0.0, r2 = 0.0;
          for (int i = 0; i < f.nd; ++i) {
            const double u = v0[i * f.qdim + kc];
            const double *g = f.gref + ((int64_t)q * f.nd + i) * 3;
            v += f.phi[q * f.nd + i] * u;
            r0 += g[0] * u; r1 += g[1] * u; r2 += g[2] * u;
          }
          T[f.off + kc] = v;
          for (int b = 0; b < 3; ++b)
            T[f.off + f.qdim + 3 * kc + b] = B[3 * b] * r0 + B[3 * b + 1] * r1 + B[3 * b + 2] * r2;
        }
        kc -= f.qdim;
        v0 += f.nd * f.qdim;
      }
      __syncthreads();
      outputs();
    }
    __syncthreads();
    const double wJ = a.qw[q] * aJ;
    for (int x = t; x < 4 * QT * nc; x += kPm) {
      const int ap = x / nc, c = x - ap * nc, p = ap / QT, ca = ap - p * QT;  // U row p QT + ca
      if (p < P0 || p >= P1) continue;
      const int j = c / qs, cb = c - j * qs;
      const double *Or = O + (p == 0 ? ca : QT + 3 * ca + p - 1) * w4, *b = bs + 4 * j;
      double s = a.rmask & 1 ? Or[cb] * b[0] : 0.0;
      if (a.rmask & 14) {
        s += Or[qs + 3 * cb] * b[1];
        s += Or[qs + 3 * cb + 1] * b[2];
        s += Or[qs + 3 * cb + 2] * b[3];
      }
      U[x] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      double u[P1 - P0][QT];
#pragma unroll
      for (int p = P0; p < P1; ++p)
#pragma unroll
        for (int c = 0; c < QT; ++c) u[p - P0][c] = U[(p * QT + c) * nc + col[k]];
#pragma unroll
      for (int i = 0; i < kPmNodes; ++i) {
        const double *b = bt + 4 * min(row0[k] + i, ndt - 1);
#pragma unroll
        for (int c = 0; c < QT; ++c) {
          double s = b[P0] * u[0][c];
#pragma unroll
          for (int p = P0 + 1; p < P1; ++p) s += b[p] * u[p - P0][c];
          acc[k][i][c] += wJ * s;
        }
      }
    }
    __syncthreads();
  }
  double mx = 0.0;
#pragma unroll
  for (int k = 0; k < NP; ++k)
#pragma unroll
    for (int i = 0; i < kPmNodes; ++i)
      if (row0[k] + i < ndt)
#pragma unroll
        for (int c = 0; c < QT; ++c) mx = fmax(mx, fabs(acc[k][i][c]));
  mx = pm_wave_max(mx);
  const double th = mx > 0.0 ? 1e-14 * mx : INFINITY;
#pragma unroll
  for (int k = 0; k < NP; ++k)
#pragma unroll
    for (int i = 0; i < kPmNodes; ++i)
      if (row0[k] + i < ndt)
#pragma unroll
        for (int c = 0; c < QT; ++c) {
          const double v = acc[k][i][c];
          dst[((row0[k] + i) * QT + c) * nc + col[k]] = fabs(v) > th ? v : 0.0;
        }
}

// Affine elements whose outputs read no fem field: the point sum goes through
// the reference tensor of a pair of base functions,
//   E[(i, a), (j, b)] = |J| sum_{p, r} O[(a, p), (b, r)] (B' R_ij B'^T)_{p r},
//   R_ij[p][r] = sum_q w_q phi_i^p psi_j^r  (p, r: value, reference gradient),
// B' = 1 for the value and B for the gradient: 54 + 81 products a pair of vector
// base functions instead of 45 and a share of U at each of the points.
// A lane keeps its pair (i, j), and with it R_ij in registers, for all the
// elements that its workgroup passes over, `epb` side by side; a chunk's
// geometry is formed first, a lane an element.  Bound by FP64 issue and the
// latency of the start.  R comes from the host, where it is summed in long
// double: formed here, by every workgroup in FP64, its roundings were most of
// the matrix's error.
// Measured, u P2 vector + p P1 on 15^3 x 6 = 20,250 elements: the four blocks
// 0.109 ms (58 us for the 30 x 30 one), 0.154 ms with R formed by every
// workgroup; through the points (k_poly_mat) 0.59 ms.
// An entry within a factor kPrNear of its element's threshold sets bit 16 of
// the error flag: whether the reference stores it is decided by the roundings
// of the sum over the points, and the caller has the matrices formed that way.
constexpr double kPrNear = 4.0;
constexpr int kPrIters = 8;      // passes of a workgroup where the elements are enough to fill the card
constexpr int kPrMaxChunk = 512; // elements of a workgroup

template <int QT, int QS>
__global__ __launch_bounds__(512) void k_poly_ref(PolyMatArgs a, int epb, int iters) {
  extern __shared__ double lds_pr[];
  const ScalarField &ft = a.f[a.vt], &fs = a.f[a.vs];
  const int ndt = ft.nd, nds = fs.nd, pairs = ndt * nds, nc = nds * QS, ne = ndt * QT * nc, chunk = epb * iters;
  constexpr int w4 = 4 * QS;
  double *T = lds_pr;                                            // symbols
  double *O = T + a.nsym;                                        // outputs
  double *geo = O + a.nout;                                      // [element][10]: B, |J|
  unsigned long long *smax = reinterpret_cast<unsigned long long *>(geo + 10 * chunk);  // max |entry|, as its bits
  const int t = threadIdx.x, lane = t & 63;
  const int64_t e0 = (int64_t)blockIdx.x * chunk;
  for (int c = t; c < a.nconst; c += blockDim.x) T[a.const_off + c] = a.consts[c];
  for (int x = t; x < chunk; x += blockDim.x) {
    double B[9], aJ;
    smax[x] = 0;
    if (e0 + x < a.n_cv) {
      if (!poly_geometry(a.pts, a.cvx + (int64_t)a.nv * (e0 + x), a.nv, nullptr, B, aJ)) {  // its entries are 0
        atomicOr(a.err, 1);
        aJ = 0.0;
        for (int c = 0; c < 9; ++c) B[c] = 0.0;
      }
      for (int c = 0; c < 9; ++c) geo[10 * x + c] = B[c];
      geo[10 * x + 9] = aJ;
    }
  }
  const int slot = t / pairs, pr = t - slot * pairs, i = pr / nds, j = pr - i * nds;
  const bool on = slot < epb;
  const bool t0 = a.pmask & 1, t1 = a.pmask & 14, s0 = a.rmask & 1, s1 = a.rmask & 14;  // slots in use
  double R[4][4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int r = 0; r < 4; ++r) R[p][r] = on ? a.R[(4 * p + r) * pairs + pr] : 0.0;
  __syncthreads();
  for (int o = t; o < a.nout; o += blockDim.x) {  // its monomials in a fixed order
    double s = 0.0;
    for (int m = a.mptr[o]; m < a.mptr[o + 1]; ++m) {
      double v = a.mcoef[m];
      for (int x = a.moff[m]; x < a.moff[m + 1]; ++x) v *= T[a.msym[x]];
      s += v;
    }
    O[o] = s;
  }
  __syncthreads();
  for (int it = 0; it < iters; ++it) {
    const int x = it * epb + slot;
    const int64_t e = e0 + x;
    const bool live = on && e < a.n_cv;
    double v[QT][QS];
#pragma unroll
    for (int c = 0; c < QT; ++c)
#pragma unroll
      for (int b = 0; b < QS; ++b) v[c][b] = 0.0;
    double mx = 0.0;
    if (live) {
      double B[9];
#pragma unroll
      for (int c = 0; c < 9; ++c) B[c] = geo[10 * x + c];
      const double aJ = geo[10 * x + 9];
      // adds O[.][p][.][r] S, with S the (p, r) entry of |J| B' R B'^T
      auto add = [&](int p, int r, double S) {
#pragma unroll
        for (int c = 0; c < QT; ++c)
#pragma unroll
          for (int b = 0; b < QS; ++b)
            v[c][b] += O[(p == 0 ? c : QT + 3 * c + p - 1) * w4 + (r == 0 ? b : QS + 3 * b + r - 1)] * S;
      };
      if (t0 && s0) add(0, 0, aJ * R[0][0]);
      if (t0 && s1) {
#pragma unroll
        for (int r = 0; r < 3; ++r)
          add(0, 1 + r, aJ * (R[0][1] * B[3 * r] + R[0][2] * B[3 * r + 1] + R[0][3] * B[3 * r + 2]));
      }
      if (t1 && s0) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          add(1 + p, 0, aJ * (B[3 * p] * R[1][0] + B[3 * p + 1] * R[2][0] + B[3 * p + 2] * R[3][0]));
      }
      if (t1 && s1) {
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          double W[3];
#pragma unroll
          for (int c = 0; c < 3; ++c)
            W[c] = aJ * (R[1 + c][1] * B[3 * r] + R[1 + c][2] * B[3 * r + 1] + R[1 + c][3] * B[3 * r + 2]);
#pragma unroll
          for (int p = 0; p < 3; ++p) add(1 + p, 1 + r, B[3 * p] * W[0] + B[3 * p + 1] * W[1] + B[3 * p + 2] * W[2]);
        }
      }
#pragma unroll
      for (int c = 0; c < QT; ++c)
#pragma unroll
        for (int b = 0; b < QS; ++b) mx = fmax(mx, fabs(v[c][b]));
    }
    // the elements that meet in this wavefront, one after the other
    const int k1 = min((t | 63) / pairs, epb - 1);
    for (int k = (t & ~63) / pairs; k <= k1; ++k) {
      const double m = pm_wave_max(slot == k ? mx : 0.0);
      if (lane == 0) atomicMax(&smax[it * epb + k], (unsigned long long)__double_as_longlong(m));
    }
    __syncthreads();
    if (live) {
      const double m = __longlong_as_double((long long)smax[x]);
      const double th = m > 0.0 ? 1e-14 * m : INFINITY, lo = th / kPrNear, hi = th * kPrNear;
      double *dst = a.elem + e * ne + (int64_t)i * QT * nc + j * QS;
      bool near = false;
#pragma unroll
      for (int c = 0; c < QT; ++c)
#pragma unroll
        for (int b = 0; b < QS; ++b) {
          const double x = fabs(v[c][b]);
          near |= x > lo && x <= hi;
          dst[c * nc + b] = x > th ? v[c][b] : 0.0;
        }
      if (near) atomicOr(a.err, 16);
    }
  }
}

// ------------------------------------------------------------ structure
// (row, column) key and position in the element matrices of every candidate
// of a block
__global__ __launch_bounds__(kPoly1d) void k_poly_keys(PolyEmitArgs a, int64_t base) {
  const int nc = a.nds * a.qs, ne = a.ndt * a.qt * nc;
  const int64_t x = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (x >= a.n_cv * ne) return;
  const int64_t e = x / ne;
  const int y = (int)(x - e * ne), r = y / nc, c = y - r * nc, i = r / a.qt, j = c / a.qs;
  const int64_t row = a.first_t + a.dt[e * a.ndt + i] + (r - i * a.qt);
  const int64_t col = a.first_s + a.ds[e * a.nds + j] + (c - j * a.qs);
  a.keys[x] = (uint64_t)(row * a.ncols + col);
  a.pos[x] = (uint32_t)(base + x);
}

// entry u's first candidate, row and column
__global__ __launch_bounds__(kPoly1d) void k_poly_entries(int64_t n, const uint64_t *__restrict__ key,
                                                          const int64_t *__restrict__ head,
                                                          const int64_t *__restrict__ pos, int64_t ncols,
                                                          uint32_t *__restrict__ start, int32_t *__restrict__ row,
                                                          int32_t *__restrict__ col) {
  const int64_t k = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (k >= n) return;
  if (head[k]) {
    start[pos[k]] = (uint32_t)k;
    row[pos[k]] = (int32_t)(key[k] / (uint64_t)ncols);
    col[pos[k]] = (int32_t)(key[k] % (uint64_t)ncols);
  }
  if (k == n - 1) start[pos[k] + head[k]] = (uint32_t)n;
}

// Every entry: its candidates summed in order, the zeros (entries that their
// element does not insert) left out.  WRITE: whether it has any other, into
// `stored` as 1 or 0.  Otherwise the sum into the CSR's values at the entry's
// place, and bit 4 of the error flag where an entry that is not stored has a
// candidate or one that is has none.
// Bound by the latency and traffic of the candidates' values, three an entry
// (P2): neighbouring entries of a row read the same element rows.  kRun of them
// are loaded together, since most entries have no more and wait once then.
// Measured at 23.4 M candidates of 7.5 M entries: 0.122 ms (two together 0.131,
// eight 0.137, one after the other 0.188), where emitting, sorting and summing
// the kept entries took 1.75 ms.
constexpr int kRun = 4;  // candidates loaded together

template <bool WRITE>
__global__ __launch_bounds__(kPoly1d) void k_poly_runs(int64_t n, const uint32_t *__restrict__ start,
                                                       const uint32_t *__restrict__ src,
                                                       const double *__restrict__ elem, int64_t *__restrict__ stored,
                                                       const uint32_t *__restrict__ place, double *__restrict__ v,
                                                       int *__restrict__ err) {
  const int64_t u = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (u >= n) return;
  const uint32_t k0 = start[u], e = start[u + 1];
  uint32_t p = kPolyNone;
  if constexpr (!WRITE) p = place[u];
  double s = 0.0;
  bool any = false;
  for (uint32_t k = k0; k < e; k += kRun) {
    uint32_t at[kRun];
    double x[kRun];
#pragma unroll
    for (int i = 0; i < kRun; ++i) at[i] = src[min(k + i, e - 1)];
#pragma unroll
    for (int i = 0; i < kRun; ++i) x[i] = elem[at[i]];
#pragma unroll
    for (int i = 0; i < kRun; ++i) {
      any |= k + i < e && x[i] != 0.0;
      s += k + i < e ? x[i] : 0.0;
    }
  }
  if constexpr (WRITE) {
    stored[u] = any;
  } else {
    if (any != (p != kPolyNone)) atomicOr(err, 4);
    if (p != kPolyNone) v[p] = s;
  }
}

// places of the stored entries (pos: the exclusive scan of `stored`), their
// columns and the row pointers; row pointers of the rows up to an entry's own
// are opened by it
__global__ __launch_bounds__(kPoly1d) void k_poly_places(int64_t n, const int64_t *__restrict__ stored,
                                                         const int64_t *__restrict__ pos,
                                                         const int32_t *__restrict__ row,
                                                         const int32_t *__restrict__ col, int64_t nrows,
                                                         uint32_t *__restrict__ place, int64_t *__restrict__ ip,
                                                         int32_t *__restrict__ ix) {
  const int64_t u = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (u >= n) return;
  place[u] = stored[u] ? (uint32_t)pos[u] : kPolyNone;
  if (stored[u]) ix[pos[u]] = col[u];
  const int64_t r = row[u], rp = u == 0 ? -1 : row[u - 1];
  for (int64_t rr = rp + 1; rr <= r; ++rr) ip[rr] = pos[u];
  if (u == n - 1)
    for (int64_t rr = r + 1; rr <= nrows; ++rr) ip[rr] = pos[u] + stored[u];
}

// ------------------------------------------------- without the structure
__global__ __launch_bounds__(kPm) void k_poly_count(int64_t n_cv, int ne, const double *__restrict__ elem,
                                                    int64_t *__restrict__ cnt) {
  const int64_t e = blockIdx.x;
  int n = 0;
  for (int x = threadIdx.x; x < ne; x += kPm) n += elem[e * ne + x] != 0.0;
  n = pm_wave_sum(n);
  if (threadIdx.x == 0) cnt[e] = n;
}

__global__ __launch_bounds__(kPm) void k_poly_emit(PolyEmitArgs a) {
  const int64_t e = blockIdx.x;
  const int t = threadIdx.x;
  const int nc = a.nds * a.qs, ne = a.ndt * a.qt * nc;
  const double *E = a.elem + e * ne;
  int64_t pos = a.off[e];
  for (int x0 = 0; x0 < ne; x0 += kPm) {
    const int x = x0 + t;
    const double v = x < ne ? E[x] : 0.0;
    const bool keep = v != 0.0;
    const uint64_t bal = __ballot(keep);
    if (keep) {
      const int r = x / nc, c = x - r * nc;
      const int i = r / a.qt, j = c / a.qs;
      const int64_t row = a.first_t + a.dt[e * a.ndt + i] + (r - i * a.qt);
      const int64_t col = a.first_s + a.ds[e * a.nds + j] + (c - j * a.qs);
      const int64_t p = pos + __popcll(bal & ((1ull << t) - 1ull));
      a.keys[p] = (uint64_t)(row * a.ncols + col);
      a.vals[p] = v;
    }
    pos += __popcll(bal);
  }
}

// head[k] = 1 where a run of equal keys starts
__global__ void k_poly_head(int64_t n, const uint64_t *__restrict__ key, int64_t *__restrict__ head) {
  const int64_t k = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (k < n) head[k] = (k == 0 || key[k] != key[k - 1]) ? 1 : 0;
}

// run u starts at start[u]; its column; the run count
__global__ void k_poly_starts(int64_t n, const uint64_t *__restrict__ key, const int64_t *__restrict__ head,
                              const int64_t *__restrict__ pos, int64_t ncols, int64_t *__restrict__ start,
                              int32_t *__restrict__ ix, int64_t *__restrict__ nnz) {
  const int64_t k = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (k >= n) return;
  if (head[k]) {
    start[pos[k]] = k;
    ix[pos[k]] = (int32_t)(key[k] % (uint64_t)ncols);
  }
  if (k == n - 1) {
    const int64_t u = pos[k] + head[k];
    start[u] = n;
    *nnz = u;
  }
}

// each value summed over its run in order (the element order)
__global__ void k_poly_sum(int64_t n, const int64_t *__restrict__ start, const int64_t *__restrict__ nnz,
                           const double *__restrict__ vals, double *__restrict__ v) {
  const int64_t u = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (u >= n || u >= *nnz) return;
  const int64_t b = start[u], e = start[u + 1];
  double s = vals[b];
  for (int64_t k = b + 1; k < e; ++k) s += vals[k];
  v[u] = s;
}

// row pointers: run u opens the rows after the previous run's row up to its own
__global__ void k_poly_indptr(int64_t n, const uint64_t *__restrict__ key, const int64_t *__restrict__ start,
                              const int64_t *__restrict__ nnz, int64_t nrows, int64_t ncols,
                              int64_t *__restrict__ ip) {
  const int64_t u = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  const int64_t m = *nnz;
  if (u >= n || u >= m) return;
  const int64_t r = (int64_t)(key[start[u]] / (uint64_t)ncols);
  const int64_t rp = u == 0 ? -1 : (int64_t)(key[start[u - 1]] / (uint64_t)ncols);
  for (int64_t rr = rp + 1; rr <= r; ++rr) ip[rr] = u;
  if (u == m - 1)
    for (int64_t rr = r + 1; rr <= nrows; ++rr) ip[rr] = m;
}

__global__ void k_poly_zero_ip(int64_t n, int64_t *__restrict__ ip, int64_t *__restrict__ nnz) {
  const int64_t k = (int64_t)blockIdx.x * kPoly1d + threadIdx.x;
  if (k < n) ip[k] = 0;
  if (k == 0) *nnz = 0;
}

unsigned pm_blocks(int64_t n) { return (unsigned)((n + kPoly1d - 1) / kPoly1d); }

}  // namespace

template <int QT, int P0, int P1>
static hipError_t launch_poly_mat_p(hipStream_t s, const PolyMatArgs &a, size_t lds) {
  const int nc = a.f[a.vs].nd * a.f[a.vs].qdim, tiles = (a.f[a.vt].nd + kPmNodes - 1) / kPmNodes * nc;
  const unsigned grid = (unsigned)a.n_cv;
  if (tiles <= kPm) k_poly_mat<QT, 1, P0, P1><<<grid, kPm, lds, s>>>(a);
  else if (tiles <= 2 * kPm) k_poly_mat<QT, 2, P0, P1><<<grid, kPm, lds, s>>>(a);
  else if (tiles <= 4 * kPm) k_poly_mat<QT, 4, P0, P1><<<grid, kPm, lds, s>>>(a);
  else if (tiles <= 8 * kPm) k_poly_mat<QT, 8, P0, P1><<<grid, kPm, lds, s>>>(a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

template <int QT>
static hipError_t launch_poly_mat_q(hipStream_t s, const PolyMatArgs &a, size_t lds) {
  if (!(a.pmask & 14)) return launch_poly_mat_p<QT, 0, 1>(s, a, lds);
  return a.pmask & 1 ? launch_poly_mat_p<QT, 0, 4>(s, a, lds) : launch_poly_mat_p<QT, 1, 4>(s, a, lds);
}

template <int QT, int QS>
static hipError_t launch_poly_ref(hipStream_t s, const PolyMatArgs &a) {
  const int pairs = a.f[a.vt].nd * a.f[a.vs].nd;
  const int threads = pairs <= 256 ? 256 : 512;
  const int epb = threads / pairs;
  int64_t iters = a.n_cv / ((int64_t)epb * 1024);  // four workgroups a CU before any takes a second pass
  iters = std::min<int64_t>({std::max<int64_t>(iters, 1), kPrIters, kPrMaxChunk / epb});
  const int chunk = epb * (int)iters;
  const size_t lds = 8 * (size_t)(a.nsym + a.nout + 11 * chunk);
  if (lds > 64 * 1024) return hipErrorInvalidValue;
  k_poly_ref<QT, QS><<<(unsigned)((a.n_cv + chunk - 1) / chunk), threads, lds, s>>>(a, epb, (int)iters);
  return hipGetLastError();
}

hipError_t launch_poly_mat(hipStream_t s, const PolyMatArgs &a) {
  if (a.n_cv == 0) return hipSuccess;
  if (a.nf < 1 || a.nf > kScalarMaxFields || a.vt < 0 || a.vt >= a.nf || a.vs < 0 || a.vs >= a.nf ||
      a.nout > kPolyMaxOut || a.f[a.vt].nd > kPolyMaxNd || a.f[a.vs].nd > kPolyMaxNd ||
      (int64_t)a.f[a.vt].nd * a.f[a.vt].qdim * a.f[a.vs].nd * a.f[a.vs].qdim > kPolyMaxEntries)
    return hipErrorInvalidValue;
  int lanes = 0, vals = 0;
  for (int i = 0; i < a.nf; ++i) {
    lanes += a.f[i].qdim;
    vals += a.f[i].nd * a.f[i].qdim;
  }
  if (lanes > kPm) return hipErrorInvalidValue;
  const int qt = a.f[a.vt].qdim, nc = a.f[a.vs].nd * a.f[a.vs].qdim;
  const size_t lds = 8 * (size_t)(a.nsym + a.nout + 4 * (a.f[a.vt].nd + a.f[a.vs].nd) + 4 * qt * nc +
                                  (a.varying ? vals : 0));
  if (lds > 64 * 1024) return hipErrorInvalidValue;
  // tetrahedra and a program without fem fields: one reference tensor a pair
  // serves every element (a field's values or a hexahedron's points make the
  // integrand another one in each)
  if (a.R && a.f[a.vt].nd * a.f[a.vs].nd <= 512) {
    const int qs = a.f[a.vs].qdim;
#define GFX_REF(QT, QS) \
  if (qt == QT && qs == QS) return launch_poly_ref<QT, QS>(s, a)
    GFX_REF(1, 1);
    GFX_REF(1, 2);
    GFX_REF(1, 3);
    GFX_REF(2, 1);
    GFX_REF(2, 2);
    GFX_REF(2, 3);
    GFX_REF(3, 1);
    GFX_REF(3, 2);
    GFX_REF(3, 3);
#undef GFX_REF
  }
  if (qt == 1) return launch_poly_mat_q<1>(s, a, lds);
  if (qt == 2) return launch_poly_mat_q<2>(s, a, lds);
  if (qt == 3) return launch_poly_mat_q<3>(s, a, lds);
  return hipErrorInvalidValue;
}

hipError_t launch_poly_emit(hipStream_t s, const PolyEmitArgs &a) {
  if (a.n_cv == 0) return hipSuccess;
  k_poly_emit<<<(unsigned)a.n_cv, kPm, 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_poly_count(hipStream_t s, int64_t n_cv, int ne, const double *elem, int64_t *cnt) {
  if (n_cv == 0) return hipSuccess;
  k_poly_count<<<(unsigned)n_cv, kPm, 0, s>>>(n_cv, ne, elem, cnt);
  return hipGetLastError();
}

hipError_t launch_poly_keys(hipStream_t s, const PolyEmitArgs &a, int64_t base) {
  const int64_t n = a.n_cv * a.ndt * a.qt * a.nds * a.qs;
  if (n == 0) return hipSuccess;
  k_poly_keys<<<pm_blocks(n), kPoly1d, 0, s>>>(a, base);
  return hipGetLastError();
}

size_t poly_structure_bytes(int64_t n, int end_bit) {
  size_t bytes = 0;
  if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint64_t *)nullptr, (uint64_t *)nullptr,
                                         (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)n, 0, end_bit) !=
      hipSuccess)
    return 0;
  return bytes;
}

hipError_t poly_sort_candidates(hipStream_t s, void *tmp, size_t tmp_bytes, const uint64_t *keys, uint64_t *keys2,
                                const uint32_t *pos, uint32_t *src, int64_t n, int end_bit, int64_t *head,
                                int64_t *scan, int64_t *work) {
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, keys, keys2, pos, src, (int)n, 0, end_bit, s);
  if (e != hipSuccess) return e;
  k_poly_head<<<pm_blocks(n), kPoly1d, 0, s>>>(n, keys2, head);
  return scan_exclusive_i64(s, head, scan, n, work);
}

hipError_t launch_poly_entries(hipStream_t s, int64_t n, const uint64_t *keys, const int64_t *head,
                               const int64_t *scan, int64_t ncols, uint32_t *start, int32_t *row, int32_t *col) {
  k_poly_entries<<<pm_blocks(n), kPoly1d, 0, s>>>(n, keys, head, scan, ncols, start, row, col);
  return hipGetLastError();
}

hipError_t launch_poly_runs(hipStream_t s, int64_t n, const uint32_t *start, const uint32_t *src, const double *elem,
                            const uint32_t *place, double *v, int *err) {
  if (n == 0) return hipSuccess;
  k_poly_runs<false><<<pm_blocks(n), kPoly1d, 0, s>>>(n, start, src, elem, nullptr, place, v, err);
  return hipGetLastError();
}

hipError_t poly_pattern(hipStream_t s, int64_t n, const uint32_t *start, const uint32_t *src, const double *elem,
                        const int32_t *row, const int32_t *col, int64_t nrows, int64_t *work, uint32_t *place,
                        int64_t *ip, int32_t *ix) {
  int64_t *stored = work, *pos = work + n, *tmp = work + 2 * n + 1;
  k_poly_runs<true><<<pm_blocks(n), kPoly1d, 0, s>>>(n, start, src, elem, stored, nullptr, nullptr, nullptr);
  hipError_t e = scan_exclusive_i64(s, stored, pos, n, tmp);
  if (e != hipSuccess) return e;
  k_poly_places<<<pm_blocks(n), kPoly1d, 0, s>>>(n, stored, pos, row, col, nrows, place, ip, ix);
  return hipGetLastError();
}

hipError_t launch_poly_empty(hipStream_t s, int64_t nrows, int64_t *ip, int64_t *d_nnz) {
  k_poly_zero_ip<<<pm_blocks(nrows + 1), kPoly1d, 0, s>>>(nrows + 1, ip, d_nnz);
  return hipGetLastError();
}

size_t poly_sort_bytes(int64_t n, int end_bit) {
  size_t bytes = 0;
  if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint64_t *)nullptr, (uint64_t *)nullptr,
                                         (const double *)nullptr, (double *)nullptr, (int)n, 0, end_bit) !=
      hipSuccess)
    return 0;
  return bytes;
}

hipError_t poly_to_csr(hipStream_t s, void *tmp, size_t tmp_bytes, uint64_t *keys, double *vals, uint64_t *keys2,
                       double *vals2, int64_t n, int end_bit, int64_t nrows, int64_t ncols, int64_t *work,
                       int64_t *ip, int32_t *ix, double *v, int64_t *d_nnz) {
  if (n == 0) {
    k_poly_zero_ip<<<pm_blocks(nrows + 1), kPoly1d, 0, s>>>(nrows + 1, ip, d_nnz);
    return hipGetLastError();
  }
  hipError_t e = hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, keys, keys2, vals, vals2, (int)n, 0,
                                                    end_bit, s);
  if (e != hipSuccess) return e;
  int64_t *head = work, *pos = work + n, *start = work + 2 * n, *stmp = work + 3 * n + 1;
  k_poly_head<<<pm_blocks(n), kPoly1d, 0, s>>>(n, keys2, head);
  if ((e = scan_exclusive_i64(s, head, pos, n, stmp)) != hipSuccess) return e;
  k_poly_starts<<<pm_blocks(n), kPoly1d, 0, s>>>(n, keys2, head, pos, ncols, start, ix, d_nnz);
  k_poly_sum<<<pm_blocks(n), kPoly1d, 0, s>>>(n, start, d_nnz, vals2, v);
  k_poly_indptr<<<pm_blocks(n), kPoly1d, 0, s>>>(n, keys2, start, d_nnz, nrows, ncols, ip);
  return hipGetLastError();
}

}  // namespace gfx
