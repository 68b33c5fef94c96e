// The order-0 / order-1 route of the workspace: potentials and their
// derivatives (ga_workspace::assembly(0 | 1),
// src/getfem_generic_assembly_workspace.cc:791-936, with the potential and
// vector assembly instructions of
// src/getfem_generic_assembly_compile_and_exec.cc:4669-4735) for integrands
// the compile stage turned into polynomial programs.
//
// k_scalar_elem: G lanes per element (affine tetrahedra, or Q1 hexahedra with
// the geometry at every point), a lane per integration point.
// The lane fills its row of a symbol table in LDS (values and gradients of the
// fem fields the program reads, from the element's nodal values in LDS, then
// the fixed-size constants), evaluates the program's monomials into its output
// coefficients and weights them; then the lanes take the results: order 0, the
// potential's element value (one lane adds the points in order); order 1, the
// element vector of the differentiated variable, a lane per dof,
//   elem[i, a] = sum_q w_q |J| (c_a phi_i + sum_b c_(q + 3a + b) (B grad phi_i)_b),
// with the B of a point taken to the coefficients' side and the sum over the
// points compensated (the coefficients' own roundings cost up to 6 % of the
// vector's error on hexahedra, which the sum's more than make good).
// The program is the same for every thread (uniform loads).  Element vectors
// go to a buffer and are summed per dof over the node's incidences (no
// atomics); element values are summed by a fixed-order two-stage reduction,
// so both results are deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "gfx_internal.h"

namespace gfx {
namespace {

constexpr int kScThreads = 64;  // one wavefront
constexpr int kScRedThreads = 256;
constexpr int kScRedBlocks = 256;

// Bound by latency (dependent loads and FP64 chains), so the points go side by
// side: with a lane per element, 20,250 elements were 317 wavefronts for the
// whole chip, each with 15 points one after another.  Measured there (u P2
// vector + p P1): 44 us a variable (58 us with a node's base function loaded
// again for each component), 222 us with a lane per element.
template <int G>
__global__ __launch_bounds__(kScThreads) void k_scalar_elem(ScalarArgs a, int nsym, int nvals) {
  extern __shared__ double lds_sc[];
  constexpr int kPer = kScThreads / G;
  const int t = threadIdx.x, g = t / G, l = t % G;
  double *T = lds_sc + t;                           // symbols, T[s * kScThreads]
  double *O = T + nsym * kScThreads;                // outputs, then (order 1) the weighted coefficients
  double *V = lds_sc + (nsym + max(a.nout, 12)) * kScThreads + g * nvals;  // nodal values, [field][node][component]
  const int64_t e0 = (int64_t)blockIdx.x * kPer + g;
  const bool live = e0 < a.n_cv;
  const int64_t e = live ? e0 : a.n_cv - 1;  // past the last element: computed, not written
  {
    double *v = V;
    for (int fi = 0; fi < a.nf; ++fi) {
      const ScalarField &f = a.f[fi];
      const int n = f.nd * f.qdim;
      for (int x = l; x < n; x += G) {
        const int i = x / f.qdim;
        v[x] = f.U[(int64_t)f.dofs[e * f.nd + i] + (x - i * f.qdim)];
      }
      v += n;
    }
  }
  for (int c = 0; c < a.nconst; ++c) T[(a.const_off + c) * kScThreads] = a.consts[c];
  const int32_t *cv = a.cvx + (int64_t)a.nv * e;
  const ScalarField &vf = a.f[a.vf];
  const int Q = vf.qdim, nl = a.order == 1 ? vf.nd * Q : 0;
  double acc = 0.0;
  __syncthreads();
  for (int q0 = 0; q0 < a.nq; q0 += G) {
    const int q = min(q0 + l, a.nq - 1), nq = min(G, a.nq - q0);  // the points of this round
    double B[9], aJ = 0.0;
    const bool ok = poly_geometry(a.pts, cv, a.nv, a.gN ? a.gN + (int64_t)q * a.nv * 3 : nullptr, B, aJ);
    if (!ok && live) atomicOr(a.err, 1);
    const double wJ = ok ? a.qw[q] * aJ : 0.0;
    const double *v0 = V;
    for (int fi = 0; fi < a.nf; ++fi) {
      const ScalarField &f = a.f[fi];
      const double *phi = f.phi + q * f.nd, *gr = f.gref + (int64_t)q * f.nd * 3;
      const auto field = [&](auto qd) {  // a node's base function and gradient serve the components together
        constexpr int QD = decltype(qd)::value;
        double v[QD], r0[QD], r1[QD], r2[QD];
#pragma unroll
        for (int c = 0; c < QD; ++c) v[c] = r0[c] = r1[c] = r2[c] = 0.0;
#pragma unroll 2
        for (int i = 0; i < f.nd; ++i) {
          const double h = phi[i], g0 = gr[3 * i], g1 = gr[3 * i + 1], g2 = gr[3 * i + 2];
#pragma unroll
          for (int c = 0; c < QD; ++c) {
            const double u = v0[i * QD + c];
            v[c] += h * u;
            r0[c] += g0 * u; r1[c] += g1 * u; r2[c] += g2 * u;
          }
        }
#pragma unroll
        for (int c = 0; c < QD; ++c) {
          T[(f.off + c) * kScThreads] = v[c];
          for (int b = 0; b < 3; ++b)
            T[(f.off + QD + 3 * c + b) * kScThreads] = B[3 * b] * r0[c] + B[3 * b + 1] * r1[c] + B[3 * b + 2] * r2[c];
        }
      };
      if (f.qdim == 1) field(std::integral_constant<int, 1>{});
      else if (f.qdim == 2) field(std::integral_constant<int, 2>{});
      else field(std::integral_constant<int, 3>{});  // (a mesh_fem has at most three)
      v0 += f.nd * f.qdim;
    }
    for (int o = 0; o < a.nout; ++o) O[o * kScThreads] = 0.0;
    for (int m = 0; m < a.nm; ++m) {
      double v = a.mcoef[m];
      for (int s = a.moff[m]; s < a.moff[m + 1]; ++s) v *= T[a.msym[s] * kScThreads];
      O[a.mout[m] * kScThreads] += v;
    }
    if (a.order == 0) {
      O[0] = wJ * O[0];
      __syncthreads();
      if (l == 0)
        for (int k = 0; k < nq; ++k) acc += O[k];
    } else {
      // w_q |J| times the value's and (against the reference gradients) the gradient's coefficients
      double cw[3][4];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (c >= Q) break;
        const double *oc = O + (Q + 3 * c) * kScThreads;
        const double o0 = oc[0], o1 = oc[kScThreads], o2 = oc[2 * kScThreads];
        cw[c][0] = wJ * O[c * kScThreads];
#pragma unroll
        for (int d = 0; d < 3; ++d) cw[c][1 + d] = wJ * (o0 * B[d] + o1 * B[3 + d] + o2 * B[6 + d]);
      }
#pragma unroll
      for (int c = 0; c < 3; ++c)
        if (c < Q)
#pragma unroll
          for (int d = 0; d < 4; ++d) O[(4 * c + d) * kScThreads] = cw[c][d];
      __syncthreads();
      double *el = a.elem + e * nl;
      for (int x = l; x < nl; x += G) {
        const int i = x / Q, c = x - i * Q;
        const double *w = lds_sc + (nsym + 4 * c) * kScThreads + g * G;  // point k: w[k]
        double s = q0 && live ? el[x] : 0.0, lost = 0.0;  // (what the sum's roundings take is added at the end)
        for (int k = 0; k < nq; ++k) {
          const int p = (q0 + k) * vf.nd + i;
          const double *h = vf.gref + (int64_t)p * 3;
          const double v = w[k] * vf.phi[p] + w[kScThreads + k] * h[0] + w[2 * kScThreads + k] * h[1] +
                           w[3 * kScThreads + k] * h[2];
          const double y = s + v, r = y - s;
          lost += (s - (y - r)) + (v - r);
          s = y;
        }
        if (live) el[x] = s + lost;
      }
    }
    __syncthreads();
  }
  if (a.order == 0 && l == 0 && live) a.elem[e] = acc;
}

__device__ __forceinline__ double sc_block_sum(double v, double *sh) {
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int off = kScRedThreads / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  return sh[0];
}

// partial sums of x over a fixed grid (each block a fixed stride of x), then
// one block sums the partials: the order never depends on scheduling
__global__ __launch_bounds__(kScRedThreads) void k_sc_partial(int64_t n, const double *__restrict__ x,
                                                              double *__restrict__ part) {
  __shared__ double sh[kScRedThreads];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kScRedThreads + threadIdx.x; i < n;
       i += (int64_t)kScRedBlocks * kScRedThreads)
    s += x[i];
  s = sc_block_sum(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(kScRedThreads) void k_sc_final(const double *__restrict__ part,
                                                            double *__restrict__ out) {
  __shared__ double sh[kScRedThreads];
  double s = 0.0;
  for (int i = threadIdx.x; i < kScRedBlocks; i += kScRedThreads) s += part[i];
  s = sc_block_sum(s, sh);
  if (threadIdx.x == 0) *out = s;
}

}  // namespace

int64_t scalar_partials() { return kScRedBlocks; }

hipError_t launch_scalar_elem(hipStream_t s, const ScalarArgs &a) {
  if (a.n_cv == 0) return hipSuccess;
  if (a.nf < 1 || a.nf > kScalarMaxFields || a.nout > kScalarMaxOut || a.vf < 0 || a.vf >= a.nf ||
      a.f[a.vf].qdim > 3)
    return hipErrorInvalidValue;
  int nvals = 0;
  for (int i = 0; i < a.nf; ++i) nvals += a.f[i].nd * a.f[i].qdim;
  const int nsym = a.const_off + a.nconst;
  auto lds = [&](int g) {
    return 8 * ((size_t)(nsym + std::max(a.nout, 12)) * kScThreads + (size_t)(kScThreads / g) * nvals);
  };
  auto grid = [&](int g) { return (unsigned)((a.n_cv + kScThreads / g - 1) / (kScThreads / g)); };
  // as many lanes as the rule has points, and the elements of a wavefront
  // must fit its LDS
  if (a.nq <= 1 && lds(1) <= 48 * 1024) k_scalar_elem<1><<<grid(1), kScThreads, lds(1), s>>>(a, nsym, nvals);
  else if (a.nq <= 4 && lds(4) <= 48 * 1024) k_scalar_elem<4><<<grid(4), kScThreads, lds(4), s>>>(a, nsym, nvals);
  else if (a.nq <= 16 && lds(16) <= 64 * 1024) k_scalar_elem<16><<<grid(16), kScThreads, lds(16), s>>>(a, nsym, nvals);
  else if (a.nq <= 32 && lds(32) <= 64 * 1024) k_scalar_elem<32><<<grid(32), kScThreads, lds(32), s>>>(a, nsym, nvals);
  else if (lds(64) <= 64 * 1024) k_scalar_elem<64><<<grid(64), kScThreads, lds(64), s>>>(a, nsym, nvals);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_scalar_sum(hipStream_t s, int64_t n, const double *x, double *part, double *out) {
  k_sc_partial<<<kScRedBlocks, kScRedThreads, 0, s>>>(n, x, part);
  k_sc_final<<<1, kScRedThreads, 0, s>>>(part, out);
  return hipGetLastError();
}

}  // namespace gfx
