// Element-batched assembly (non-affine elements / nonlinear material):
// a workgroup computes a whole element matrix, the matrices go to an HBM
// buffer (row-major, rows = Test_u), and a node-patch gather adds the rows
// each node owns into its CSR rows, with GetFEM's per-element insertion
// threshold (compile_and_exec.cc:5441-5453).  Used for the compressible
// Neo-Hookean (Bonet) tangent and residual on Q2 hexahedra:
//   GWFL ((Id+Grad_u)*(Compressible_Neo_Hookean_Bonet_PK2(Grad_u,[lambda;mu]))):Grad_Test_u
//   (src/getfem_nonlinear_elasticity.cc:2319-2320), law :612-696, derivative
//   wrapper :1799-1827.
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "gfx_internal.h"

namespace gfx {

namespace {

constexpr int kEbThreads = 256;
constexpr int kNd = 27, kNl = 81, kNv = 8;

// The Neo-Hookean element computations are two kernels.
// k_nh_points, a wavefront per two elements (lane = point, then node):
//   K_q = G grad(N)(q), J_q, B_q = K_q^{-T}, wJ_q = |J_q| w_q     (trilinear map)
//   H_q = sum_i U_i (x) grad(phi_i)(q) B_q^T;  F_q = I + H_q
//   S_q = mu (I - C^-1) + lambda/2 ln(I3) C^-1                    (Bonet law)
//   re[(i,a)] = sum_q wJ_q (F_q S_q B_q grad(phi_i)(q))_a
// and, for a tangent, the kNhPd values per point that k_nh_tangent needs.
// k_nh_tangent, a workgroup per element, the tangent K[(i,a),(j,b)] =
// sum_q g[q][i][c] D_q[(a,c),(b,n)] g[q][j][n] with D_q[(a,c),(b,n)] = wJ_q
// (delta_ab S[n][c] + F[a][k] A[k c m n] F[b][m]) (the GWFL derivative of the
// residual, A = dS/dE) in the spatial form (h = F^{-T} g): per node pair and
// point, two outer products of spatial gradients and a dot product, as
// products on the matrix cores in FP64 (FP64 form) or FP32 (FP32 form), upper
// tiles only (nh_phase_b).
constexpr int kNq = 27;
constexpr int kKeepWords = (kNl * kNl + 31) / 32;  // keep-bit words per element (206)
// k_nh_points' values per point, each kNq consecutive doubles of the element's
// run: A = F^{-T} B row-major (h = A grad(phi)), alpha = wJ lambda, beta =
// wJ (mu - lambda ln J), and the node term's symmetric kernel M (00, 01, 02,
// 11, 12, 22)
constexpr int kNhPd = 17;

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

// maximum over a wavefront in its lane 63: VALU lane moves, no trip through
// the LDS (a lane without a source keeps its own value)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_max(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return fmax(v, __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}
__device__ __forceinline__ double wave_max(double v) {
  v = dpp_max<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: lane 15 of each row has the row's maximum
  v = dpp_max<0x112, 0xf>(v);
  v = dpp_max<0x114, 0xf>(v);
  v = dpp_max<0x118, 0xf>(v);
  v = dpp_max<0x142, 0xa>(v);     // row_bcast 15 into rows 1 and 3
  return dpp_max<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
}

// Lane layout of the 16x16x4 matrix-core products (v_mfma_f64_16x16x4_f64,
// v_mfma_f32_16x16x4_f32): A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k
// (both instructions); D[i][j] in lane j + 16 (i / 4), element i % 4 for the
// FP32 one, but in lane j + 16 (i % 4), element i / 4 for the FP64 one
// (BdbMfma<T>::row gives the row of lane group g and element r).
template <typename T>
struct BdbMfma;
template <>
struct BdbMfma<double> {
  typedef __attribute__((__vector_size__(4 * sizeof(double)))) double v4;
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int r) { return 4 * r + g; }
};
template <>
struct BdbMfma<float> {
  typedef f32x4 v4;
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
};

// Phase B in the spatial form (see k_nh_tangent) on the matrix cores, in T
// (FP64: v_mfma_f64_16x16x4_f64; FP32: v_mfma_f32_16x16x4_f32, exact
// products and FP32 sums).  With H_c[i][q] = h_qic (node i, point q), the
// (a, b) component block of K over the node pairs is
//   K_ab = H_a diag(alpha) H_b^T + H_b diag(beta) H_a^T + delta_ab K3,
//   K3 = sum_c H_c M_c^T,  M_c[j][q] = (M_q h_qj)_c,
// so both outer-product terms of a block go into one accumulator and no
// value moves between lanes; for a = b they are one product, with alpha + beta.  A tile is a 16 x 16 node tile (I, J) in
// {0, 1}^2 (27 nodes and 5 zero pads) of one component pair (a, b); the k
// axis is the 27 points and one zero (7 steps of 4).  hC (point q's row of
// kNhRow values: [c][32 nodes], zero pads) holds h as the fragments read it:
// one LDS read per value; the row's 16 spare values keep the four points of a
// fragment in different banks.
// K is symmetric: with P = 2 a + I and Q = 2 b + J only the 21 tiles P <= Q
// are formed (the others are their transposes), and of K3 the node tiles
// (0, 0), (0, 1), (1, 1).  Wavefront w < 3 forms K3 tile w beside the three
// tiles (a, a) of the same node tiles, to which it is added, from the same
// fragments, and two of the twelve tiles with a < b; wavefront 3 forms the
// other six (70, 70, 70, 84 products).  Each tile is stored from its
// accumulators: 16-value runs of its own rows, 4-value runs of its
// transpose's, which the L2 joins (plain stores: as non-temporal ones the
// short runs took twice the time).
constexpr int kNhQ = 28, kNhN = 32, kNhRow = 3 * kNhN + 16;

// tile N (0..20): wavefront N / 5 (N < 15) takes N % 5 = 0..2 as the (a, a)
// tiles of its K3 node tile and 3..4 as with-a<b tiles 2 (N / 5) + (N % 5 - 3);
// N >= 15 are the with-a<b tiles 6..11 of wavefront 3.  With-a<b tile n:
// (a, b) = (0,1), (0,2), (1,2) for n / 4 = 0, 1, 2, (I, J) = (n % 4 / 2, n % 2).
template <int N>
struct NhTile {
  static constexpr bool diag = N < 15 && N % 5 < 3;  // an (a, a) tile: K3 added
  static constexpr int w = N < 15 ? N / 5 : 3;
  static constexpr int n = N < 15 ? 2 * w + (N % 5 - 3) : 6 + (N - 15);  // with-a<b index (when !diag)
  static constexpr int a = diag ? N % 5 : (n / 4 == 2 ? 1 : 0);
  static constexpr int b = diag ? N % 5 : (n / 4 == 0 ? 1 : 2);
  static constexpr int I = diag ? w / 2 : n % 4 / 2;
  static constexpr int J = diag ? (w + 1) / 2 : n % 2;
  static constexpr int P = 2 * a + I, Q = 2 * b + J;
  static_assert(P <= Q, "upper tiles only");
};
static_assert(NhTile<0>::P == 0 && NhTile<0>::Q == 0 && NhTile<5>::P == 0 && NhTile<5>::Q == 1 &&
              NhTile<14>::a == 0 && NhTile<14>::b == 2 && NhTile<14>::I == 0 && NhTile<14>::J == 1 &&
              NhTile<20>::a == 1 && NhTile<20>::b == 2 && NhTile<20>::I == 1 && NhTile<20>::J == 1,
              "tile table");

// one k-step of tile N: f[c][I] = h at this lane's point, component c, node 16 I + lr
template <typename T, int N>
__device__ __forceinline__ void nh_w_mma(typename BdbMfma<T>::v4 &acc, T al, T be, const T (&f)[3][2]) {
  typedef NhTile<N> D;
  if constexpr (D::diag) {  // both terms are the same product
    acc = BdbMfma<T>::mma((al + be) * f[D::a][D::I], f[D::a][D::J], acc);
  } else {
    acc = BdbMfma<T>::mma(al * f[D::a][D::I], f[D::b][D::J], acc);
    acc = BdbMfma<T>::mma(be * f[D::b][D::I], f[D::a][D::J], acc);
  }
}
template <typename T, int T0, int... U>
__device__ __forceinline__ void nh_w_step(std::integer_sequence<int, U...>, typename BdbMfma<T>::v4 (&acc)[6], T al,
                                          T be, const T (&f)[3][2]) {
  (nh_w_mma<T, T0 + U>(acc[U], al, be, f), ...);
}

// the products of tiles T0 .. T0 + NT - 1 (accumulators acc[0 .. NT - 1]) and,
// for the wavefronts that have diagonal tiles, of their K3 node tile:
// K3[i][j] = sum_q h_qi^T M_q h_qj, k = (c, q): A = h_qic, B = (M_q h_qj)_c
template <typename T, int T0, int NT>
__device__ __forceinline__ void nh_w_tiles(int lr, int lg, const T *hC, const double *pd,
                                           typename BdbMfma<T>::v4 (&acc)[6], typename BdbMfma<T>::v4 &k3) {
  constexpr int w = T0 / 5, I3 = w / 2, J3 = (w + 1) / 2;
#pragma unroll
  for (int u = 0; u < 6; ++u) acc[u] = typename BdbMfma<T>::v4{T(0), T(0), T(0), T(0)};
  k3 = typename BdbMfma<T>::v4{T(0), T(0), T(0), T(0)};
#pragma unroll 1  // (in full it takes 104 registers, a wavefront less per SIMD, for nothing)
  for (int st = 0; st < kNhQ / 4; ++st) {
    T f[3][2];
    const int q = 4 * st + lg;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int I = 0; I < 2; ++I) f[c][I] = hC[q * kNhRow + c * kNhN + 16 * I + lr];
    const double *pq = pd + min(q, kNq - 1);  // (hC is zero at q = 27)
    const T al = (T)pq[9 * kNq], be = (T)pq[10 * kNq];
    nh_w_step<T, T0>(std::make_integer_sequence<int, NT>{}, acc, al, be, f);
    if constexpr (w < 3) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        // row c of the symmetric M: its entries (c, 0), (c, 1), (c, 2)
        const T m = (T)pq[(11 + c) * kNq] * f[0][J3] + (T)pq[(11 + (c == 0 ? 1 : 2 + c)) * kNq] * f[1][J3] +
                    (T)pq[(11 + (c == 0 ? 2 : 3 + c)) * kNq] * f[2][J3];
        k3 = BdbMfma<T>::mma(f[c][I3], m, k3);
      }
    }
  }
}

// tile N's entries into E (node-blocked: entry ((3 i + a) 3 + b) 27 + j for
// K[(i,a),(j,b)]), K3 added to (a, a) tiles, the transpose written for P < Q
template <typename T, int N>
__device__ __forceinline__ void nh_w_store1(int lr, int lg, const typename BdbMfma<T>::v4 &acc,
                                            const typename BdbMfma<T>::v4 &k3, T *E) {
  typedef NhTile<N> D;
  const int j = 16 * D::J + lr;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int i = 16 * D::I + BdbMfma<T>::row(lg, x);
    const T v = D::diag ? acc[x] + k3[x] : acc[x];
    if (i < kNd && j < kNd) {
      E[((3 * i + D::a) * 3 + D::b) * kNd + j] = v;
      if (D::P != D::Q) E[((3 * j + D::b) * 3 + D::a) * kNd + i] = v;
    }
  }
}
// the keep bits (row-major over (3 i + a, 3 j + b)) of the same entries
template <typename T, int N>
__device__ __forceinline__ void nh_w_bits1(int lr, int lg, double th, const typename BdbMfma<T>::v4 &acc,
                                           const typename BdbMfma<T>::v4 &k3, uint32_t *skeep) {
  typedef NhTile<N> D;
  const int j = 16 * D::J + lr;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int i = 16 * D::I + BdbMfma<T>::row(lg, x);
    const T v = D::diag ? acc[x] + k3[x] : acc[x];
    if (i < kNd && j < kNd && (double)fabs(v) > th) {
      const int d = (3 * i + D::a) * kNl + 3 * j + D::b, m = (3 * j + D::b) * kNl + 3 * i + D::a;
      atomicOr(&skeep[d >> 5], 1u << (d & 31));
      if (D::P != D::Q) atomicOr(&skeep[m >> 5], 1u << (m & 31));
    }
  }
}
template <typename T, int T0, int... U>
__device__ __forceinline__ void nh_w_store(std::integer_sequence<int, U...>, int lr, int lg,
                                           const typename BdbMfma<T>::v4 (&acc)[6],
                                           const typename BdbMfma<T>::v4 &k3, T *E) {
  (nh_w_store1<T, T0 + U>(lr, lg, acc[U], k3, E), ...);
}
template <typename T, int T0, int... U>
__device__ __forceinline__ void nh_w_bits(std::integer_sequence<int, U...>, int lr, int lg, double th,
                                          const typename BdbMfma<T>::v4 (&acc)[6],
                                          const typename BdbMfma<T>::v4 &k3, uint32_t *skeep) {
  (nh_w_bits1<T, T0 + U>(lr, lg, th, acc[U], k3, skeep), ...);
}

// this lane's largest |entry| of tiles T0 .. T0 + NT - 1 (K3 added to the
// (a, a) tiles; the zero pads add nothing)
template <typename T, int N>
__device__ __forceinline__ double nh_w_max1(const typename BdbMfma<T>::v4 &acc, const typename BdbMfma<T>::v4 &k3) {
  double m = 0.0;
#pragma unroll
  for (int x = 0; x < 4; ++x) m = fmax(m, (double)fabs(NhTile<N>::diag ? acc[x] + k3[x] : acc[x]));
  return m;
}
template <typename T, int T0, int... U>
__device__ __forceinline__ double nh_w_max_seq(std::integer_sequence<int, U...>,
                                               const typename BdbMfma<T>::v4 (&acc)[6],
                                               const typename BdbMfma<T>::v4 &k3) {
  double m = 0.0;
  ((m = fmax(m, nh_w_max1<T, T0 + U>(acc[U], k3))), ...);
  return m;
}
template <typename T, int T0, int NT>
__device__ __forceinline__ double nh_w_max(const typename BdbMfma<T>::v4 (&acc)[6],
                                           const typename BdbMfma<T>::v4 &k3) {
  return nh_w_max_seq<T, T0>(std::make_integer_sequence<int, NT>{}, acc, k3);
}

// this lane's smallest |entry| of tiles T0 .. T0 + NT - 1 (zero pads aside), 0
// where one is not a number: every entry is kept where it is above the threshold
template <typename T, int N>
__device__ __forceinline__ double nh_w_min1(int lr, int lg, const typename BdbMfma<T>::v4 &acc,
                                            const typename BdbMfma<T>::v4 &k3) {
  typedef NhTile<N> D;
  double m = INFINITY;
  bool nan = false;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const bool in = 16 * D::I + BdbMfma<T>::row(lg, x) < kNd && 16 * D::J + lr < kNd;
    const double v = (double)fabs(D::diag ? acc[x] + k3[x] : acc[x]);
    m = fmin(m, in ? v : INFINITY);
    nan |= v != v;
  }
  return nan ? 0.0 : m;
}
template <typename T, int T0, int... U>
__device__ __forceinline__ double nh_w_min_seq(std::integer_sequence<int, U...>, int lr, int lg,
                                               const typename BdbMfma<T>::v4 (&acc)[6],
                                               const typename BdbMfma<T>::v4 &k3) {
  double m = INFINITY;
  ((m = fmin(m, nh_w_min1<T, T0 + U>(lr, lg, acc[U], k3))), ...);
  return m;
}
template <typename T, int T0, int NT>
__device__ __forceinline__ double nh_w_min(int lr, int lg, const typename BdbMfma<T>::v4 (&acc)[6],
                                           const typename BdbMfma<T>::v4 &k3) {
  return nh_w_min_seq<T, T0>(std::make_integer_sequence<int, NT>{}, lr, lg, acc, k3);
}

// One wavefront's part, tiles T0 .. T0 + NT - 1.  KEEP: 0 no keep bits; 1 they
// are compared with the stored ones (bit 32 of the error flag when any
// differs); 2 they are written.
template <typename T, int KEEP, int T0, int NT>
__device__ __forceinline__ void nh_phase_b(int t, int64_t e, const double *pd, const T *hC, uint32_t *skeep,
                                           double *red, int was_full, const EbArgs &a) {
  typedef typename BdbMfma<T>::v4 v4;
  constexpr int w = T0 / 5, kWaves = kEbThreads / 64;
  constexpr auto tiles = std::make_integer_sequence<int, NT>{};
  const int l = t % 64, lr = l % 16, lg = l / 16;
  v4 acc[6], k3;
  nh_w_tiles<T, T0, NT>(lr, lg, hC, pd, acc, k3);
  // threshold 1e-14 max|K| (all-zero element skipped), from the accumulators,
  // and (negated) the smallest |entry|, one barrier for both
  const double mx = wave_max(nh_w_max<T, T0, NT>(acc, k3));
  double mn = 0.0;
  if constexpr (KEEP != 0) mn = wave_max(-nh_w_min<T, T0, NT>(lr, lg, acc, k3));
  if (l == 63) {
    red[w] = mx;
    if (KEEP != 0) red[kWaves + w] = mn;
  }
  if (KEEP != 0)  // (where they are needed; before the barrier that their use is behind)
    for (int x = t; x < kKeepWords; x += kEbThreads) skeep[x] = 0u;
  __syncthreads();
  double mxe = red[0];
  for (int v = 1; v < kWaves; ++v) mxe = fmax(mxe, red[v]);
  const double th = mxe > 0.0 ? 1e-14 * mxe : INFINITY;
  if (t == 0) a.thr[e] = th;
  nh_w_store<T, T0>(tiles, lr, lg, acc, k3, reinterpret_cast<T *>(a.E) + e * kNl * kNl);
  if constexpr (KEEP != 0) {
    // An element that keeps every entry (nearly all do) has words of ones: they
    // are not formed.  full[e] says that of the stored words.
    double mne = red[kWaves];
    for (int v = 1; v < kWaves; ++v) mne = fmax(mne, red[kWaves + v]);
    const bool full = -mne > th;  // (uniform)
    if (KEEP == 1 && t == 0 && was_full != (full ? 1 : 0)) atomicOr(a.err, 32);
    if (KEEP == 2 && t == 0) a.full[e] = full ? 1 : 0;
    if (KEEP == 1 && full) return;
    if (!full) {
      nh_w_bits<T, T0>(tiles, lr, lg, th, acc, k3, skeep);
      __syncthreads();
    }
    bool same = true;
    for (int x = t; x < kKeepWords; x += kEbThreads) {
      const uint32_t bits = !full ? skeep[x] : (x == kKeepWords - 1 ? (1u << (kNl * kNl % 32)) - 1u : 0xffffffffu);
      if constexpr (KEEP == 2) a.keep[e * kKeepWords + x] = bits;
      else same &= a.keep[e * kKeepWords + x] == bits;
    }
    if (!same) atomicOr(a.err, 32);
  }
}

// Points and residual.  Bound by FP64 issue and the LDS.  A half wavefront
// per element, 27 of its 32 lanes at work: the sums over nodes and over points
// are tensor products, done one direction at a time (72 products a lane each
// way instead of 243), so lane (x, y, z) is in turn a point or a node along
// each direction and the partial sums pass through the element's own LDS
// block; only the wavefront's own lanes read it, so no workgroup barrier is
// needed.  Measured in kernel traces: 41 us at 31^3 elements (the tangent kernel,
// which a residual took before, 835), 49 with the points' values, 172 with them
// at 48^3 = 110,592.
constexpr int kNhHalf = 32;

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool TANGENT>
__global__ __launch_bounds__(kEbThreads) void k_nh_points(EbArgs a) {
  __shared__ double T1[2][3][3];                                  // l_m(x_q), dl_m(x_q): [.][m][q]
  __shared__ double bufA[kEbThreads / kNhHalf][9][kNhHalf];       // partial sums, component-major
  __shared__ double bufB[kEbThreads / kNhHalf][9][kNhHalf];
  if (threadIdx.x < 18) T1[threadIdx.x / 9][threadIdx.x % 9 / 3][threadIdx.x % 3] = a.t1d[threadIdx.x];
  __syncthreads();
  const int slot = threadIdx.x / kNhHalf, l = threadIdx.x % kNhHalf;
  const bool on = l < kNq;
  const int t = on ? l : 0, tx = t % 3, ty = t / 3 % 3, tz = t / 9;
  const int64_t e0 = (int64_t)blockIdx.x * (kEbThreads / kNhHalf) + slot;
  const bool live = e0 < a.n_cv;
  const int64_t e = live ? e0 : a.n_cv - 1;  // past the last element: computed, not written
  double (&A)[9][kNhHalf] = bufA[slot];
  double (&Bf)[9][kNhHalf] = bufB[slot];
  {  // the nodes' displacements, and the vertices behind them
    const double *u = a.U + a.dofs[kNd * e + t];
    const double *x = a.pts + 3 * (int64_t)a.cvx[kNv * e + l % kNv];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      A[c][l] = u[c];
      A[3 + c][l] = x[c];
    }
  }
  wave_lds_fence();
  // K = sum_v X_v (x) grad N_v at this lane's point (vertex dx + 2 dy + 4 dz)
  double k[9];  // column-major K(r,c)
  {
    const double x1 = a.xq[tx], y1 = a.xq[ty], z1 = a.xq[tz], x0 = 1.0 - x1, y0 = 1.0 - y1, z0 = 1.0 - z1;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const double *X = A[3 + r];
      k[r] = y0 * z0 * (X[1] - X[0]) + y1 * z0 * (X[3] - X[2]) + y0 * z1 * (X[5] - X[4]) + y1 * z1 * (X[7] - X[6]);
      k[r + 3] = x0 * z0 * (X[2] - X[0]) + x1 * z0 * (X[3] - X[1]) + x0 * z1 * (X[6] - X[4]) + x1 * z1 * (X[7] - X[5]);
      k[r + 6] = x0 * y0 * (X[4] - X[0]) + x1 * y0 * (X[5] - X[1]) + x0 * y1 * (X[6] - X[2]) + x1 * y1 * (X[7] - X[3]);
    }
  }
  const double lam = a.ca ? a.ca[e] : a.ca_c, mu = a.cb ? a.cb[e] : a.cb_c;
  // H = sum_i U_i (x) grad(phi_i), one direction at a time:
  // x: lane (point x, node y, node z) -> value and d/dx
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double v = 0.0, d = 0.0;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const double u = A[c][m + 3 * ty + 9 * tz];
      v += T1[0][m][tx] * u;
      d += T1[1][m][tx] * u;
    }
    Bf[2 * c][l] = v;
    Bf[2 * c + 1][l] = d;
  }
  wave_lds_fence();
  // y: lane (point x, point y, node z) -> d/dx, d/dy, value
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double dx = 0.0, dy = 0.0, v = 0.0;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const double w = Bf[2 * c][tx + 3 * m + 9 * tz];
      dx += T1[0][m][ty] * Bf[2 * c + 1][tx + 3 * m + 9 * tz];
      dy += T1[1][m][ty] * w;
      v += T1[0][m][ty] * w;
    }
    A[3 * c][l] = dx;
    A[3 * c + 1][l] = dy;
    A[3 * c + 2][l] = v;
  }
  wave_lds_fence();
  // z: lane = point
  double Hr[9];  // row-major d u_c / d xi_d
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double dx = 0.0, dy = 0.0, dz = 0.0;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const int o = tx + 3 * ty + 9 * m;
      dx += T1[0][m][tz] * A[3 * c][o];
      dy += T1[0][m][tz] * A[3 * c + 1][o];
      dz += T1[1][m][tz] * A[3 * c + 2][o];
    }
    Hr[3 * c] = dx; Hr[3 * c + 1] = dy; Hr[3 * c + 2] = dz;
  }
  double B[9], F[9], wJ;
  {
    const double a0 = k[4] * k[8] - k[5] * k[7];
    const double a1 = k[5] * k[6] - k[3] * k[8];
    const double a2 = k[3] * k[7] - k[4] * k[6];
    const double J = k[0] * a0 + k[1] * a1 + k[2] * a2;
    if (J == 0.0 && live && on) atomicOr(a.err, 1);
    const double rJ = 1.0 / J;  // B row-major B(r,c)
    B[0] = a0 * rJ; B[3] = a1 * rJ; B[6] = a2 * rJ;
    B[1] = (k[2] * k[7] - k[1] * k[8]) * rJ;
    B[4] = (k[0] * k[8] - k[2] * k[6]) * rJ;
    B[7] = (k[1] * k[6] - k[0] * k[7]) * rJ;
    B[2] = (k[1] * k[5] - k[2] * k[4]) * rJ;
    B[5] = (k[2] * k[3] - k[0] * k[5]) * rJ;
    B[8] = (k[0] * k[4] - k[1] * k[3]) * rJ;
    wJ = fabs(J) * a.qw[t];
  }
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c)
      F[3 * r + c] = Hr[3 * r] * B[3 * c] + Hr[3 * r + 1] * B[3 * c + 1] + Hr[3 * r + 2] * B[3 * c + 2] + (r == c ? 1.0 : 0.0);
  // the law
  const double f0 = F[4] * F[8] - F[5] * F[7], f1 = F[5] * F[6] - F[3] * F[8], f2 = F[3] * F[7] - F[4] * F[6];
  const double detF = F[0] * f0 + F[1] * f1 + F[2] * f2;
  double S[9], ln3;
  {
    double C[9], Ci[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) C[3 * i + j] = F[i] * F[j] + F[3 + i] * F[3 + j] + F[6 + i] * F[6 + j];
    const double c0 = C[4] * C[8] - C[5] * C[7];
    const double c1 = C[5] * C[6] - C[3] * C[8];
    const double c2 = C[3] * C[7] - C[4] * C[6];
    const double I3 = C[0] * c0 + C[1] * c1 + C[2] * c2;
    const double rI3 = 1.0 / I3;
    Ci[0] = c0 * rI3; Ci[3] = c1 * rI3; Ci[6] = c2 * rI3;
    Ci[1] = (C[2] * C[7] - C[1] * C[8]) * rI3;
    Ci[4] = (C[0] * C[8] - C[2] * C[6]) * rI3;
    Ci[7] = (C[1] * C[6] - C[0] * C[7]) * rI3;
    Ci[2] = (C[1] * C[5] - C[2] * C[4]) * rI3;
    Ci[5] = (C[2] * C[3] - C[0] * C[5]) * rI3;
    Ci[8] = (C[0] * C[4] - C[1] * C[3]) * rI3;
    ln3 = log(I3);
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      S[i] = mu * ((i % 4 == 0 ? 1.0 : 0.0) - Ci[i]) + 0.5 * lam * ln3 * Ci[i];
      if (detF <= 0.0) S[i] += 1e200 * C[i];  // the law's penalty on inverted points
    }
  }
  // Q = wJ F S B (first Piola stress against the reference gradients), component-major
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    double P[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) P[c] = wJ * (F[3 * r] * S[c] + F[3 * r + 1] * S[3 + c] + F[3 * r + 2] * S[6 + c]);
#pragma unroll
    for (int d = 0; d < 3; ++d) Bf[3 * r + d][l] = P[0] * B[d] + P[1] * B[3 + d] + P[2] * B[6 + d];
  }
  if (TANGENT && live && on) {
    double *pd = a.pd + e * (kNhPd * kNq) + t;
    const double rF = 1.0 / detF;
    double Fi[9];  // F^{-1}, row-major
    Fi[0] = f0 * rF; Fi[3] = f1 * rF; Fi[6] = f2 * rF;
    Fi[1] = (F[2] * F[7] - F[1] * F[8]) * rF;
    Fi[4] = (F[0] * F[8] - F[2] * F[6]) * rF;
    Fi[7] = (F[1] * F[6] - F[0] * F[7]) * rF;
    Fi[2] = (F[1] * F[5] - F[2] * F[4]) * rF;
    Fi[5] = (F[2] * F[3] - F[0] * F[5]) * rF;
    Fi[8] = (F[0] * F[4] - F[1] * F[3]) * rF;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int d = 0; d < 3; ++d) pd[(3 * c + d) * kNq] = Fi[c] * B[d] + Fi[3 + c] * B[3 + d] + Fi[6 + c] * B[6 + d];
    pd[9 * kNq] = wJ * lam;
    pd[10 * kNq] = wJ * (mu - 0.5 * lam * ln3);
    // the node term's kernel in the spatial gradients: with g = F^T h,
    // gamma g_i . g_j + pen (F g_i) . (F g_j) = h_i^T M h_j, M = gamma b + pen b^2,
    // b = F F^T (symmetric), gamma = wJ mu, pen = 1e200 wJ where det F <= 0
    const double ga = wJ * mu, pen = detF <= 0.0 ? wJ * 1e200 : 0.0;
    double b[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) b[3 * r + c] = F[3 * r] * F[3 * c] + F[3 * r + 1] * F[3 * c + 1] + F[3 * r + 2] * F[3 * c + 2];
    int o = 11;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = r; c < 3; ++c, ++o) {
        double m = ga * b[3 * r + c];
        if (pen != 0.0) m += pen * (b[3 * r] * b[c] + b[3 * r + 1] * b[3 + c] + b[3 * r + 2] * b[6 + c]);
        pd[o * kNq] = m;
      }
  }
  wave_lds_fence();
  // re = sum_q Q_q grad(phi_i)(q), the directions the other way round:
  // z: lane (point x, point y, node z)
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double r0 = 0.0, r1 = 0.0, r2 = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int o = tx + 3 * ty + 9 * q;
      r0 += T1[0][tz][q] * Bf[3 * c][o];
      r1 += T1[0][tz][q] * Bf[3 * c + 1][o];
      r2 += T1[1][tz][q] * Bf[3 * c + 2][o];
    }
    A[3 * c][l] = r0;
    A[3 * c + 1][l] = r1;
    A[3 * c + 2][l] = r2;
  }
  wave_lds_fence();
  // y: lane (point x, node y, node z)
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double r0 = 0.0, r1 = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int o = tx + 3 * q + 9 * tz;
      r0 += T1[0][ty][q] * A[3 * c][o];
      r1 += T1[1][ty][q] * A[3 * c + 1][o] + T1[0][ty][q] * A[3 * c + 2][o];
    }
    Bf[2 * c][l] = r0;
    Bf[2 * c + 1][l] = r1;
  }
  wave_lds_fence();
  // x: lane = node
  double *re = a.res + e * kNl + 3 * t;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double r = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int o = q + 3 * ty + 9 * tz;
      r += T1[1][tx][q] * Bf[2 * c][o] + T1[0][tx][q] * Bf[2 * c + 1][o];
    }
    if (live && on) re[c] = r;
  }
}

// The tangent in the spatial form.  With h_qi = F_q^{-T} g_qi (spatial
// gradients), the push-forward of this law's material tangent is
// J c = lambda 1 x 1 + (mu - lambda ln J)(two symmetric identities), and
// F^{-1} b F^{-T} = I folds the stress term into mu g_qi . g_qj, so the
// (i, j) block of D's contraction is, per point,
//   wJ_q [lambda h_qi (x) h_qj + (mu - lambda ln J_q) h_qj (x) h_qi
//         + (mu g_qi . g_qj + pen_q (F g_qi) . (F g_qj)) I]
// (pen_q = 1e200 where det F <= 0: the derivative of the penalty term 1e200 C
// that the law adds to S there).  Same matrix as the material form
// D[(a,c),(b,n)] = wJ (delta_ab S_nc + F_ak A_kcmn F_bm) up to roundoff,
// without forming D or D g (nh_phase_b).  h = A grad(phi) from the points'
// values, which k_nh_points leaves in memory (3.7 KB an element): its serial
// phases (27 of 256 threads at work) used to take as long here as the products.
// Bound by no single unit: the matrix cores are 49 % busy, the VALU 24 %, the
// stores of E (5.8 GB) run at 3 TB/s; a workgroup is 2 us at the points' values
// and gradients (issued together, before anything waits), 4 us at the products
// and 4 us at the maximum and the stores, five workgroups a CU taking turns.
// Measured at 48^3 = 110,592 elements with the keep check: 1.93 ms.  2.64 ms
// with the gradients loaded after the points' values, a barrier each for the
// maximum and for the keep check, K3 in a pass of its own, two products for
// a = b and E staged in the LDS (four more barriers); 3.21 ms with the serial
// phases inside and the keep words always formed.  Workgroups that stay for
// many elements and fetch the next one's values ahead took 2.2 ms.
template <typename Real, int KEEP>
__global__ __launch_bounds__(kEbThreads, 5) void k_nh_tangent(EbArgs a) {
  __shared__ double pd[kNhPd * kNq];
  __shared__ Real hC[kNhQ * kNhRow];  // the spatial gradients in the fragments' layout
  __shared__ double red[2 * (kEbThreads / 64)];
  __shared__ uint32_t skeep[KEEP ? kKeepWords : 1];  // the element's keep bits, where not all are set
  const int64_t e = blockIdx.x;
  const int t = threadIdx.x;
  const double *src = a.pd + e * (kNhPd * kNq);
  constexpr int kPd = (kNhPd * kNq + kEbThreads - 1) / kEbThreads;
  double pv[kPd];
#pragma unroll
  for (int r = 0; r < kPd; ++r) pv[r] = src[min(t + r * kEbThreads, kNhPd * kNq - 1)];
  const int was_full = KEEP == 1 && t == 0 ? a.full[e] : 0;
  // hC[q][c][i] = h_qic in Real (zero for q = 27 and nodes i >= 27): thread
  // (i, q mod 8) takes every eighth point; its gradients are on the way while
  // the points' values are
  static_assert(kNhN * 8 == kEbThreads, "a thread per (node, point mod 8)");
  constexpr int kHq = (kNhQ + 7) / 8;
  const int i = t % kNhN, q0 = t / kNhN;
  double g[kHq][3];
#pragma unroll
  for (int r = 0; r < kHq; ++r) {
    const double *gp = a.gref + (min(q0 + 8 * r, kNq - 1) * kNd + min(i, kNd - 1)) * 3;
#pragma unroll
    for (int c = 0; c < 3; ++c) g[r][c] = gp[c];
  }
#pragma unroll
  for (int r = 0; r < kPd; ++r)
    if (t + r * kEbThreads < kNhPd * kNq) pd[t + r * kEbThreads] = pv[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kHq; ++r) {
    const int q = q0 + 8 * r, qc = min(q, kNq - 1);
    const bool in = q < kNq && i < kNd;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double h = pd[3 * c * kNq + qc] * g[r][0] + pd[(3 * c + 1) * kNq + qc] * g[r][1] +
                       pd[(3 * c + 2) * kNq + qc] * g[r][2];
      if (q < kNhQ) hC[q * kNhRow + c * kNhN + i] = in ? (Real)h : Real(0);
    }
  }
  __syncthreads();
  // the wavefront index as a scalar: the branches on it are uniform (each
  // branch meets the same barriers)
  const int w = __builtin_amdgcn_readfirstlane(t / 64);
  if (w == 0) nh_phase_b<Real, KEEP, 0, 5>(t, e, pd, hC, skeep, red, was_full, a);
  else if (w == 1) nh_phase_b<Real, KEEP, 5, 5>(t, e, pd, hC, skeep, red, was_full, a);
  else if (w == 2) nh_phase_b<Real, KEEP, 10, 5>(t, e, pd, hC, skeep, red, was_full, a);
  else nh_phase_b<Real, KEEP, 15, 6>(t, e, pd, hC, skeep, red, was_full, a);
}

// node-patch gather of the rows of buffered element matrices: the Q rows of
// an incidence are one contiguous run of Q*NL values (FP64 or FP32); the runs
// of all the node's incidences are streamed by the whole workgroup at once
// (independent loads, LDS atomics), then the node's CSR rows are written once.
// TH threads per workgroup: 256 for the Q2 hexahedra (one node, long runs;
// four wavefronts owning two, two, two and three (row component, column
// component) pairs), 64 for the affine tets' packed wave groups (short
// runs, more groups in flight); wavefront w writes rows w, w + TH/64, ... of
// each node.
constexpr int kGatherThreadsQ2 = 256;

// npw (1..4) small patches of one bin share a workgroup: their incidence
// lists are concatenated and streamed together; patch k's accumulator starts
// at the prefix sum of Q*Q*ns over the patches before it.
constexpr int kGatherNpw = 4;

template <int ND, int Q, typename TE, int TH, int MI = 64>
__global__ __launch_bounds__(TH) void k_gather_emat(PatchArgs a, const TE *__restrict__ E,
                                                    const double *__restrict__ thr) {
  extern __shared__ double acc[];  // the npw accumulators, acc_cap doubles in all
  constexpr int kMaxInc = MI;      // incidences per workgroup (checked by the launcher)
  __shared__ int64_t sbase[kMaxInc];   // element-matrix run of each incidence
  __shared__ double sthr[kMaxInc];
  __shared__ uint16_t sslot[kMaxInc * ND];
  __shared__ int sacc[kMaxInc];        // accumulator offset and slot count of each incidence's patch
  __shared__ int sns[kMaxInc];
  constexpr int NL = ND * Q, RUN = Q * NL;
  const int64_t wg = blockIdx.x;
  const int npw = a.npw;
  const int64_t pos0 = ((wg & 7) * (int64_t)a.xcd_chunk + (wg >> 3)) * npw;
  if (pos0 >= a.n_nodes) return;
  const int t = threadIdx.x;
  PatchDesc dsc[kGatherNpw];
  int pre[kGatherNpw + 1];
  pre[0] = 0;
#pragma unroll
  for (int k = 0; k < kGatherNpw; ++k) {
    dsc[k] = PatchDesc{0, 0, 0u};
    if (k < npw && pos0 + k < a.n_nodes) dsc[k] = a.desc[pos0 + k];
    pre[k + 1] = pre[k] + (int)(dsc[k].ninc_ns & 0xffffu);
  }
  const int total_inc = pre[kGatherNpw];
  if (total_inc > kMaxInc) return;  // excluded by the launcher
  // staging, flattened over the workgroup's incidences (patch k of combined
  // incidence c: the number of patch starts at or below c): the incidence
  // words and slot maps are loaded together, then the thresholds
  auto patch_of = [&](int c) { return (int)(c >= pre[1]) + (int)(c >= pre[2]) + (int)(c >= pre[3]); };
  int gi0[kGatherNpw], gns[kGatherNpw], pre4[kGatherNpw], aoff[kGatherNpw];
  int apre = 0;  // accumulator of patch k at the prefix sum of Q*Q*ns
#pragma unroll
  for (int k = 0; k < kGatherNpw; ++k) {
    gi0[k] = dsc[k].i0;
    gns[k] = (int)(dsc[k].ninc_ns >> 16) & 0x7fff;
    pre4[k] = pre[k];
    aoff[k] = apre;
    apre += Q * Q * gns[k];
  }
  auto sel = [](const int (&v)[kGatherNpw], int k) {  // by value: no indexed array
    return k == 0 ? v[0] : (k == 1 ? v[1] : (k == 2 ? v[2] : v[3]));
  };
  // presence words of the patches that are not full (patch k's at the prefix
  // sum wpre[k]), staged in LDS behind the accumulators with the other staged
  // data, so that the write-out makes no global loads
  int wpre[kGatherNpw];
  int wtot = 0;
#pragma unroll
  for (int k = 0; k < kGatherNpw; ++k) {
    wpre[k] = wtot;
    wtot += (dsc[k].ninc_ns >> 31) ? 0 : (Q * Q * gns[k] + 31) / 32;
  }
  uint32_t *swords = reinterpret_cast<uint32_t *>(acc + a.lds_acc);
  uint32_t inc = 0;
  if (t < total_inc) {
    const int k = patch_of(t);
    inc = a.inc[sel(gi0, k) + (t - sel(pre4, k))];
  }
  for (int x = t; x < total_inc * ND; x += TH) {
    const int c = x / ND, k = patch_of(c);
    sslot[x] = a.slot[((int64_t)sel(gi0, k) + (c - sel(pre4, k))) * ND + (x - c * ND)];
  }
  for (int x = t; x < wtot; x += TH) {
    const int k = (int)(x >= wpre[1]) + (int)(x >= wpre[2]) + (int)(x >= wpre[3]);
    swords[x] = a.mask[(int64_t)sel(gi0, k) * a.mwpi + (x - sel(wpre, k))];
  }
  for (int x = t; x < apre; x += TH) acc[x] = 0.0;
  if (t < total_inc) {
    const int k = patch_of(t);
    const int64_t e = inc >> 5;
    sbase[t] = e * (int64_t)NL * NL + (int64_t)(inc & 31) * RUN;
    sthr[t] = thr[e];
    sacc[t] = sel(aoff, k);
    sns[t] = sel(gns, k);
  }
  __syncthreads();
  // the stream: incidence by incidence (uniform across the workgroup), each
  // thread owning the offsets t, t + TH, ... of the incidence's run, whose
  // (row, node, component) split is fixed; kI incidences' loads are issued
  // before any is used (offsets past the run load entry 0 and are dropped).
  // One wavefront (affine tets, runs of 90 or 180, 12-24 incidences per
  // group) loads kI incidences with clamped indices; 256 threads (Q2
  // hexahedra, runs of 243, often fewer incidences than kI) skip the loads
  // past the group's last incidence.
  // Which entries (row component x, column node j, column component y) of
  // a run a thread owns.  One wavefront (E row-major, run offset
  // x NL + j Q + y): t, t + 64, ...  Several wavefronts (E node-blocked, run
  // offset (x Q + y) ND + j, the Neo-Hookean element kernel's layout): each
  // owns whole (x, y) pairs, each ND consecutive values: 64 / ND pairs for
  // all but the last wavefront, which owns the rest in NV passes.  Every
  // accumulator entry (x, slot, y) is then added to by one wavefront only,
  // in incidence order, and no two lanes of one ds_add_f64 share an entry
  // (the nodes of an incidence have distinct slots): the sums do not depend
  // on timing.
  constexpr bool kPairs = TH > 64;
  constexpr int kW = TH / 64, kPpw = 64 / ND, kLast = Q * Q - kPpw * (kW - 1);
  static_assert(!kPairs || (kLast > 0 && kLast * ND <= 2 * 64), "the last wavefront's pairs fit two passes");
  constexpr int NV = kPairs ? (kLast * ND + 63) / 64 : (RUN + TH - 1) / TH;
  constexpr int kI = TH == 64 ? (NV >= 16 ? 1 : 16 / NV) : 8;
  int ov[NV], xv[NV], jv[NV], yv[NV];
  bool okv[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (kPairs) {  // E node-blocked: pair p's ND values are consecutive
      const int w = t / 64, L = t % 64 + 64 * v;  // this wavefront's value index
      const int p = kPpw * w + L / ND;
      okv[v] = w < kW - 1 ? L < kPpw * ND : L < kLast * ND;
      xv[v] = okv[v] ? p / Q : 0;
      yv[v] = okv[v] ? p % Q : 0;
      jv[v] = okv[v] ? L % ND : 0;
      ov[v] = okv[v] ? p * ND + jv[v] : 0;
    } else {
      const int o = t + v * TH;
      okv[v] = o < RUN;
      ov[v] = okv[v] ? o : 0;
      xv[v] = ov[v] / NL;
      const int c = ov[v] - xv[v] * NL;
      jv[v] = c / Q;
      yv[v] = c - jv[v] * Q;
    }
  }
  for (int c0 = 0; c0 < total_inc; c0 += kI) {
    TE val[kI][NV];
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      if (TH == 64 || c0 + i < total_inc) {  // uniform
        const int64_t base = sbase[min(c0 + i, total_inc - 1)];
#pragma unroll
        for (int v = 0; v < NV; ++v) val[i][v] = __builtin_nontemporal_load(E + base + ov[v]);  // read once
      }
    }
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      const int k = c0 + i;
      if (k >= total_inc) break;
      const double th = sthr[k];
      const int ns = sns[k], ak = sacc[k];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const double x = (double)val[i][v];
        if (okv[v] && fabs(x) > th) atomicAdd(&acc[ak + (xv[v] * ns + sslot[k * ND + jv[v]]) * Q + yv[v]], x);
      }
    }
  }
  __syncthreads();
  // values are streamed past the caches (written once, never re-read here)
  const int w = t / 64, lane = t % 64;
#pragma unroll
  for (int k = 0; k < kGatherNpw; ++k) {
    if (k >= npw || pos0 + k >= a.n_nodes) break;
    const int nsraw = (int)(dsc[k].ninc_ns >> 16), ns = nsraw & 0x7fff;
    const double *ak = acc + aoff[k];
    if (nsraw & 0x8000) {  // all rows full: the node's Q rows are one contiguous run of the CSR
      double *dst = a.vals + dsc[k].rowbase;
      for (int d = t; d < Q * ns * Q; d += TH) __builtin_nontemporal_store(ak[d], dst + d);
      continue;
    }
    // wavefront x writes row x from the presence bits; the node's rows are
    // consecutive CSR rows, so row x starts after the present entries of
    // rows 0..x-1 (bits [0, x*ns*Q) of the node's presence words)
    const uint32_t *m = swords + wpre[k];
    for (int x = w; x < Q; x += TH / 64) {
      const int off = x * ns * Q, len = ns * Q;
      int cnt = 0;
      for (int b0 = 0; b0 < off; b0 += 64 * 32) {
        const int b = b0 + 32 * lane;  // this lane's word of the prefix
        if (b < off) {
          const uint32_t word = m[b >> 5];
          cnt += __popc(off - b >= 32 ? word : (word & ((1u << (off - b)) - 1u)));
        }
      }
      for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
      int64_t base = dsc[k].rowbase + cnt;
      // kOut chunks of 64 per round: presence words and values are read with
      // clamped indices before any ballot, so their latencies overlap
      constexpr int kOut = 8;
      for (int c0 = 0; c0 < len; c0 += kOut * 64) {
        uint32_t word[kOut];
        double val[kOut];
#pragma unroll
        for (int u = 0; u < kOut; ++u) {
          const int dc = off + min(c0 + u * 64 + lane, len - 1);
          word[u] = m[dc >> 5];
          val[u] = ak[dc];
        }
#pragma unroll
        for (int u = 0; u < kOut; ++u) {
          const int d = c0 + u * 64 + lane;
          const bool pr = (d < len) & (bool)((word[u] >> ((off + d) & 31)) & 1u);
          const uint64_t bal = __ballot(pr);
          if (pr) __builtin_nontemporal_store(val[u], a.vals + base + __popcll(bal & ((1ull << lane) - 1ull)));
          base += __popcll(bal);
        }
      }
    }
  }
}

// Element-batched isotropic elasticity on the matrix cores (affine tets, the
// bf16 split form): E = sum_q w_q |J| B_q^T D B_q with B_q the 6 x NL Voigt
// strain-displacement matrix at point q (engineering shears; rows xx, yy, zz,
// yz, xz, xy) and D the isotropic Voigt matrix (lambda + 2 mu on the normal
// diagonal, lambda off it, mu on the shears).  D = S S with the symmetric root
// S = sqrt(2 mu) I + c 1 1^T on the normal block, c = (sqrt(2 mu + 3 lambda)
// - sqrt(2 mu)) / 3, and sqrt(mu) on the shears (D positive definite: mu > 0,
// 3 lambda + 2 mu > 0).  With F_q = sqrt(|w_q| |J|) S B_q,
// E = sum_q sign(w_q) F_q^T F_q: one product E[m][n] = sum_k A[m][k] C[k][n]
// with A[m][k] = F[k][m], C[k][n] = sign F[k][n] and k = 8 q + s (s < 6; 6, 7
// zero), so one 32-wide k-step is 4 points.  E is symmetric: one wavefront
// computes one element's upper NT x NT tiles (16 x 16) and mirrors them.
// MFMA 16x16x32 bf16 lane layout: A[i][k] in lane i + 16 (k / 8), element
// k % 8; C[k][j] in lane j + 16 (k / 8), element k % 8; D[i][j] in lane
// j + 16 (i / 4), element i % 4.  So the A fragment of row tile a and the C
// fragment of column tile a are the same registers (up to the sign of w_q):
// the 8 rows of F at one point (q = 4 step + lane / 16) for the dof
// 16 a + lane % 16, built from the reference gradient of its shape function
// (the same for every element: staged in LDS once per workgroup) and the
// element's inverse Jacobian, then split into bf16 hi + lo; the products
// hi hi, hi lo and lo hi are accumulated in FP32 (lo lo is below 2^-16 of
// the leading term).  The workgroup's four wavefronts sweep the elements with
// a grid stride, the next element's record loaded while the current one is
// computed.  E is written row-major in FP32 (rows = test dofs (i, a)) through
// the wavefront's LDS block as whole 16-byte pieces.
__device__ __forceinline__ void split2(float x, __bf16 &hi, __bf16 &lo) {
  hi = (__bf16)x;
  lo = (__bf16)(x - (float)hi);
}

typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;

__device__ __forceinline__ bf16x8 bf16_xor(const bf16x8 &x, uint32_t m) {
  u32x4 u = __builtin_bit_cast(u32x4, x);
  u ^= m;
  return __builtin_bit_cast(bf16x8, u);
}

// rows of F at the point of the staged reference gradient h (h.w = the signed
// sqrt(|w_q|)) for dof m (m >= NL: padding, zero); on / off / sh: sqrt(|J|)
// times the normal-diagonal, normal-off-diagonal and shear factors of S
template <int NL>
__device__ __forceinline__ void bdb_factor(const float4 *hp, int m, const float (&Bm)[9], float on, float off,
                                           float sh, bf16x8 &hi, bf16x8 &lo) {
  const float4 h = hp[m < NL ? m / 3 : 0];
  const float gx = Bm[0] * h.x + Bm[1] * h.y + Bm[2] * h.z;
  const float gy = Bm[3] * h.x + Bm[4] * h.y + Bm[5] * h.z;
  const float gz = Bm[6] * h.x + Bm[7] * h.y + Bm[8] * h.z;
  const int ax = m % 3;
  const float r = m < NL ? fabsf(h.w) : 0.f;  // padding rows are zero
  const float ga = r * (ax == 0 ? gx : (ax == 1 ? gy : gz)), vn = on * ga, vo = off * ga;
  const float rs = sh * r;
  float v[8];
  v[0] = ax == 0 ? vn : vo;
  v[1] = ax == 1 ? vn : vo;
  v[2] = ax == 2 ? vn : vo;
  v[3] = rs * (ax == 1 ? gz : (ax == 2 ? gy : 0.f));  // yz
  v[4] = rs * (ax == 0 ? gz : (ax == 2 ? gx : 0.f));  // xz
  v[5] = rs * (ax == 0 ? gy : (ax == 1 ? gx : 0.f));  // xy
  v[6] = v[7] = 0.f;
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    __bf16 a, b;
    split2(v[x], a, b);
    hi[x] = a;
    lo[x] = b;
  }
}

constexpr int kBdbMaxGroups = 8192;

// the k-steps of one element: fragments of the NT dof tiles at 4 points, then
// the upper tiles' three bf16 products; NEG: C = sign(w_q) F (one XOR)
template <int ND, bool NEG>
__device__ __forceinline__ void bdb_steps(const float4 *hs, int steps, int qq, int lr, const float (&Bm)[9],
                                          float on, float off, float sh,
                                          f32x4 (&acc)[((3 * ND + 15) / 16) * ((3 * ND + 15) / 16 + 1) / 2]) {
  constexpr int NL = 3 * ND, NT = (NL + 15) / 16;
  for (int k = 0; k < steps; ++k) {
    const float4 *hp = hs + (4 * k + qq) * ND;
    bf16x8 fh[NT], fl[NT];
#pragma unroll
    for (int a = 0; a < NT; ++a) bdb_factor<NL>(hp, 16 * a + lr, Bm, on, off, sh, fh[a], fl[a]);
    const uint32_t sgn = NEG && hp[0].w < 0.f ? 0x80008000u : 0u;
    int p = 0;
#pragma unroll
    for (int b = 0; b < NT; ++b) {
      const bf16x8 ch = NEG ? bf16_xor(fh[b], sgn) : fh[b];
      const bf16x8 cl = NEG ? bf16_xor(fl[b], sgn) : fl[b];
#pragma unroll
      for (int a = 0; a <= b; ++a, ++p) {
        acc[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fl[a], ch, acc[p], 0, 0, 0);
        acc[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fh[a], cl, acc[p], 0, 0, 0);
        acc[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fh[a], ch, acc[p], 0, 0, 0);
      }
    }
  }
}

// rows of the element matrix staged at once: half of them when that half is a
// whole number of 16-byte pieces (P3: 30 x 60 floats), else all (P2)
__host__ __device__ constexpr int bdb_stage_rows(int nl) { return (nl / 2) * nl % 4 == 0 && nl % 2 == 0 ? nl / 2 : nl; }

template <int ND>
__global__ __launch_bounds__(256) void k_elast_bdb_mfma(int64_t n_cv, int nq, const double *__restrict__ rec,
                                                        const double *__restrict__ gref,
                                                        const double *__restrict__ qw, float *__restrict__ E) {
  constexpr int NL = 3 * ND, NT = (NL + 15) / 16, NP = NT * (NT + 1) / 2;
  constexpr int RC = bdb_stage_rows(NL), KC = NL / RC;
  static_assert(NL * NL % 4 == 0, "element matrices are whole float4 runs");
  extern __shared__ float4 hs[];  // [4 * steps][ND]: (reference gradient of phi_i at point q,
                                  // signed sqrt(|w_q|)), then one RC x NL float block per wavefront
  const int t = threadIdx.x, w = t / 64, l = t % 64;
  const int steps = (nq + 3) / 4;
  float *es = reinterpret_cast<float *>(hs + 4 * steps * ND) + w * RC * NL;
  int neg = 0;
  for (int x = t; x < 4 * steps * ND; x += 256) {
    const int q = x / ND;
    float4 h{0.f, 0.f, 0.f, 0.f};
    if (q < nq) {
      const double *g = gref + (int64_t)x * 3;  // [q][i][3]
      const double wq = qw[q];
      h = float4{(float)g[0], (float)g[1], (float)g[2], (float)copysign(sqrt(fabs(wq)), wq)};
      neg |= wq < 0.0;
    }
    hs[x] = h;
  }
  const bool any_neg = __syncthreads_or(neg);  // a rule with negative weights
  const int lr = l % 16, qq = l / 16;
  const int64_t stride = 4 * (int64_t)gridDim.x;
  int64_t e = 4 * (int64_t)blockIdx.x + __builtin_amdgcn_readfirstlane(w);  // uniform: scalar record loads
  if (e >= n_cv) return;  // no barrier follows
  double nx[11];  // the record of the element in flight: B row-major, |J| lambda, |J| mu
#pragma unroll
  for (int x = 0; x < 9; ++x) nx[x] = rec[kRecStride * e + x];
#pragma unroll
  for (int x = 0; x < 2; ++x) nx[9 + x] = rec[kRecStride * e + 12 + x];
  for (; e < n_cv; e += stride) {
    float Bm[9];
#pragma unroll
    for (int x = 0; x < 9; ++x) Bm[x] = (float)nx[x];
    // S's factors in FP32 (the products are rounded to bf16 pairs anyway); the
    // record's coefficients carry |J|, and S(|J| lambda, |J| mu) = sqrt(|J|) S(lambda, mu)
    const float lam = (float)nx[9], mu = (float)nx[10];
    // c = (sqrt(2 mu + 3 lambda) - sqrt(2 mu)) / 3 without the cancellation
    const float s2m = sqrtf(2.f * mu), c = lam / (sqrtf(2.f * mu + 3.f * lam) + s2m);
    const float on = s2m + c, off = c, sh = sqrtf(mu);
    const int64_t en = min(e + stride, n_cv - 1);
#pragma unroll
    for (int x = 0; x < 9; ++x) nx[x] = rec[kRecStride * en + x];
#pragma unroll
    for (int x = 0; x < 2; ++x) nx[9 + x] = rec[kRecStride * en + 12 + x];
    f32x4 acc[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) acc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (any_neg)  // uniform: only rules with a negative weight pay for the signs
      bdb_steps<ND, true>(hs, steps, qq, lr, Bm, on, off, sh, acc);
    else
      bdb_steps<ND, false>(hs, steps, qq, lr, Bm, on, off, sh, acc);
    // KC row chunks of RC rows, each staged whole and written as 16-byte pieces
#pragma unroll
    for (int h = 0; h < KC; ++h) {
      int p = 0;
#pragma unroll
      for (int b = 0; b < NT; ++b)
#pragma unroll
        for (int a = 0; a <= b; ++a, ++p) {
          const int col = 16 * b + lr;
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const int row = 16 * a + 4 * qq + x;
            if (row < NL && col < NL) {
              if (row / RC == h) es[(row - RC * h) * NL + col] = acc[p][x];
              if (a != b && col / RC == h) es[(col - RC * h) * NL + row] = acc[p][x];
            }
          }
        }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const f32x4 *es4 = reinterpret_cast<const f32x4 *>(es);
      f32x4 *E4 = reinterpret_cast<f32x4 *>(E + e * NL * NL + RC * h * NL);
      for (int x = l; x < RC * NL / 4; x += 64) __builtin_nontemporal_store(es4[x], E4 + x);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // reads done before the next writes
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
}

// V[node*Q + x] = sum over incidences (e, i) of res[(e*nd + i)*Q + x]; one
// thread per dof, so that the Q threads of a node read consecutive values (one
// thread per node read them Q times apart, one after another)
template <int Q>
__global__ __launch_bounds__(256) void k_gather_vec(int64_t n_dof, int nd, const int32_t *__restrict__ inc_ptr,
                                                    const uint32_t *__restrict__ inc,
                                                    const double *__restrict__ res,
                                                    double *__restrict__ V) {
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n_dof) return;
  const int64_t n = d / Q;
  const int x = (int)(d - n * Q), k1 = inc_ptr[n + 1];
  double s = 0.0;
  for (int k = inc_ptr[n]; k < k1; ++k) {
    const uint32_t c = inc[k];
    s += res[((int64_t)(c >> 5) * nd + (c & 31)) * Q + x];
  }
  V[d] = s;
}

}  // namespace

int64_t nh_point_doubles(int64_t n_cv) { return n_cv * kNhPd * kNq; }

hipError_t launch_nh_points(hipStream_t s, const EbArgs &a) {
  if (a.n_cv == 0) return hipSuccess;
  if (a.nq != kNq) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)((a.n_cv + kEbThreads / kNhHalf - 1) / (kEbThreads / kNhHalf));
  if (a.pd) k_nh_points<true><<<grid, kEbThreads, 0, s>>>(a);
  else k_nh_points<false><<<grid, kEbThreads, 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_nh_tangent(hipStream_t s, const EbArgs &a, int precision, int keep) {
  if (a.n_cv == 0) return hipSuccess;
  if (a.nq != kNq || !a.pd || (keep && (precision != GFX_PREC_FP64 || a.kwords != kKeepWords)))
    return hipErrorInvalidValue;  // keep bits come from the FP64 pass
  const unsigned grid = (unsigned)a.n_cv;
  if (precision == GFX_PREC_FP32) k_nh_tangent<float, 0><<<grid, kEbThreads, 0, s>>>(a);
  else if (keep == kNhKeepCheck) k_nh_tangent<double, 1><<<grid, kEbThreads, 0, s>>>(a);
  else if (keep == kNhKeepWrite) k_nh_tangent<double, 2><<<grid, kEbThreads, 0, s>>>(a);
  else k_nh_tangent<double, 0><<<grid, kEbThreads, 0, s>>>(a);
  return hipGetLastError();
}

// Element-batched isotropic elasticity on the FP64 and FP32 matrix cores
// (v_mfma_f64_16x16x4_f64, v_mfma_f32_16x16x4_f32): the symmetric root
// factorization of the bf16 form above, E = sum_q sign(w_q) F_q^T F_q with
// F_q = sqrt(|w_q| |J|) S B_q, computed in T.  The k axis is the 6 Voigt rows
// of every point back to back (k = 6 q + s, no padding rows), 4 k per MFMA.
// Lane layout of the 16x16x4 products: A[i][k] in lane i + 16 k, C[k][j] in
// lane j + 16 k (both instructions); D[i][j] in lane j + 16 (i / 4), element
// i % 4 for v_mfma_f32_16x16x4_f32, but in lane j + 16 (i % 4), element i / 4
// for v_mfma_f64_16x16x4_f64 (BdbMfma<T>::row gives the row of a lane group g
// and element r).  So a lane holds one F value per dof tile and k-step, and
// the A fragment of row tile a is the C fragment of column tile a up to
// sign(w_q).  One wavefront per element (grid stride), only the upper tiles
// computed.  E (row-major, T) is stored from the accumulators: tile (a, b) as
// 16-value runs of its rows, its mirror (b, a) as 4-value runs per lane.
// F[s][m] of one point: Voigt row s (xx, yy, zz, yz, xz, xy) of S B_q for
// dof m = 3 i + ax, from the staged (reference gradient of phi_i, signed
// sqrt(|w_q|)) h; on / off / sh: the normal-diagonal, normal-off-diagonal and
// shear factors of S (with |J| folded in)
template <typename T>
__device__ __forceinline__ T bdb_fvalue(const T (&h)[4], int s, int ax, const T (&Bm)[9], T on, T off, T sh) {
  const T gx = Bm[0] * h[0] + Bm[1] * h[1] + Bm[2] * h[2];
  const T gy = Bm[3] * h[0] + Bm[4] * h[1] + Bm[5] * h[2];
  const T gz = Bm[6] * h[0] + Bm[7] * h[1] + Bm[8] * h[2];
  const T r = h[3] < T(0) ? -h[3] : h[3];
  T v;
  if (s < 3) {
    v = (s == ax ? on : off) * (ax == 0 ? gx : (ax == 1 ? gy : gz));
  } else {
    // shear rows: yz (s 3) couples y and z, xz (4) x and z, xy (5) x and y
    const int p = s == 3 ? 1 : 0, q = s == 5 ? 1 : 2;
    const T gp = p == 0 ? gx : gy, gq = q == 1 ? gy : gz;
    v = ax == p ? sh * gq : (ax == q ? sh * gp : T(0));
  }
  return r * v;
}

template <int ND, typename T>
__global__ __launch_bounds__(256) void k_elast_bdb_mfma_hp(int64_t n_cv, int nq, const double *__restrict__ rec,
                                                           const double *__restrict__ gref,
                                                           const double *__restrict__ qw, T *__restrict__ E) {
  typedef typename BdbMfma<T>::v4 v4;
  constexpr int NL = 3 * ND, NT = (NL + 15) / 16, NP = NT * (NT + 1) / 2;
  extern __shared__ double hs_raw[];  // [nq][ND][4] in T: reference gradient, signed sqrt(|w_q|)
  T *hs = reinterpret_cast<T *>(hs_raw);
  const int t = threadIdx.x, w = t / 64, l = t % 64;
  int neg = 0;
  for (int x = t; x < nq * ND; x += 256) {
    const double *g = gref + (int64_t)x * 3;  // [q][i][3]
    const double wq = qw[x / ND];
    hs[4 * x] = (T)g[0];
    hs[4 * x + 1] = (T)g[1];
    hs[4 * x + 2] = (T)g[2];
    hs[4 * x + 3] = (T)copysign(sqrt(fabs(wq)), wq);
    neg |= wq < 0.0;
  }
  const bool any_neg = __syncthreads_or(neg);
  const int lr = l % 16, lg = l / 16;
  const int K = 6 * nq, steps = (K + 3) / 4;
  const int64_t stride = 4 * (int64_t)gridDim.x;
  for (int64_t e = 4 * (int64_t)blockIdx.x + __builtin_amdgcn_readfirstlane(w); e < n_cv; e += stride) {
    const double *re = rec + kRecStride * e;  // uniform: scalar loads
    T Bm[9];
#pragma unroll
    for (int x = 0; x < 9; ++x) Bm[x] = (T)re[x];
    // S(|J| lambda, |J| mu) = sqrt(|J|) S(lambda, mu)
    const T lam = (T)re[12], mu = (T)re[13];
    const T s2m = sqrt(T(2) * mu), c = lam / (sqrt(T(2) * mu + T(3) * lam) + s2m);
    const T on = s2m + c, off = c, sh = sqrt(mu);
    v4 acc[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) acc[p] = v4{T(0), T(0), T(0), T(0)};
    int q = lg / 6, sv = lg % 6;  // this lane's k = 4 step + lg as (point, Voigt row)
    for (int st = 0; st < steps; ++st) {
      const bool kin = q < nq;
      T f[NT];
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        const int m = 16 * a + lr;
        T h[4] = {T(0), T(0), T(0), T(0)};
        if (kin && m < NL) {
          const T *hp = hs + 4 * (q * ND + m / 3);  // q < nq, m / 3 < ND here
          h[0] = hp[0]; h[1] = hp[1]; h[2] = hp[2]; h[3] = hp[3];
        }
        f[a] = bdb_fvalue<T>(h, sv, m % 3, Bm, on, off, sh);
      }
      const T sg = any_neg && hs[4 * (min(q, nq - 1) * ND) + 3] < T(0) ? T(-1) : T(1);
      int p = 0;
#pragma unroll
      for (int b = 0; b < NT; ++b) {
        const T cb = sg * f[b];
#pragma unroll
        for (int a = 0; a <= b; ++a, ++p) acc[p] = BdbMfma<T>::mma(f[a], cb, acc[p]);
      }
      sv += 4;
      if (sv >= 6) { sv -= 6; ++q; }
    }
    T *Ee = E + e * (int64_t)(NL * NL);
    int p = 0;
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int a = 0; a <= b; ++a, ++p) {
        const int col = 16 * b + lr;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * a + BdbMfma<T>::row(lg, r);
          if (row < NL && col < NL) {
            __builtin_nontemporal_store(acc[p][r], Ee + row * NL + col);
            if (a != b) __builtin_nontemporal_store(acc[p][r], Ee + col * NL + row);
          }
        }
      }
  }
}

hipError_t launch_elast_bdb_mfma(hipStream_t s, int64_t n_cv, int nd, int nq, const double *rec,
                                 const double *gref, const double *qw, float *E) {
  if (n_cv == 0) return hipSuccess;
  // one float4 per (point, node), then the staged rows of one element matrix per wavefront
  const size_t lds = 16 * (size_t)(4 * ((nq + 3) / 4)) * nd + 4 * 4 * (size_t)(bdb_stage_rows(3 * nd) * 3 * nd);
  if (nq < 1 || lds > 64 * 1024) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)std::min<int64_t>((n_cv + 3) / 4, kBdbMaxGroups);  // 4 wavefronts each
  if (nd == 10) k_elast_bdb_mfma<10><<<grid, 256, lds, s>>>(n_cv, nq, rec, gref, qw, E);
  else if (nd == 20) k_elast_bdb_mfma<20><<<grid, 256, lds, s>>>(n_cv, nq, rec, gref, qw, E);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

// the FP64 (E64) or FP32 (E32) matrix-core form; the other pointer is null
hipError_t launch_elast_bdb_mfma_hp(hipStream_t s, int64_t n_cv, int nd, int nq, const double *rec,
                                    const double *gref, const double *qw, double *E64, float *E32) {
  if (n_cv == 0) return hipSuccess;
  const size_t lds = (size_t)nq * nd * 4 * (E64 ? sizeof(double) : sizeof(float));
  if (lds > 64 * 1024) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)std::min<int64_t>((n_cv + 3) / 4, kBdbMaxGroups);  // 4 wavefronts each
  if (E64) {
    if (nd == 10) k_elast_bdb_mfma_hp<10, double><<<grid, 256, lds, s>>>(n_cv, nq, rec, gref, qw, E64);
    else if (nd == 20) k_elast_bdb_mfma_hp<20, double><<<grid, 256, lds, s>>>(n_cv, nq, rec, gref, qw, E64);
    else return hipErrorInvalidValue;
  } else {
    if (nd == 10) k_elast_bdb_mfma_hp<10, float><<<grid, 256, lds, s>>>(n_cv, nq, rec, gref, qw, E32);
    else if (nd == 20) k_elast_bdb_mfma_hp<20, float><<<grid, 256, lds, s>>>(n_cv, nq, rec, gref, qw, E32);
    else return hipErrorInvalidValue;
  }
  return hipGetLastError();
}


hipError_t launch_gather_emat(hipStream_t s, const PatchArgs &a0, const void *E, bool e_fp32, const double *thr,
                              int acc_cap, int group_inc) {
  // acc_cap: the largest sum of Q*Q*nslots over the patches of one workgroup
  // (doubles of LDS); group_inc: the largest number of incidences of one workgroup
  if (a0.n_nodes == 0) return hipSuccess;
  PatchArgs a = a0;
  if (a.npw < 1 || a.npw > kGatherNpw) return hipErrorInvalidValue;
  const int64_t groups = (a.n_nodes + a.npw - 1) / a.npw;
  a.xcd_chunk = (int)((groups + 7) / 8);
  const unsigned grid = (unsigned)(8 * (int64_t)a.xcd_chunk);
  // accumulators, then the presence words: at most ceil(Q*Q*ns/32) per patch,
  // so acc_cap/32 + kGatherNpw in all
  if (acc_cap < 0 || 8 * (size_t)acc_cap > 48 * 1024 || group_inc > 64) return hipErrorInvalidValue;
  a.lds_acc = acc_cap;
  const size_t lds = (size_t)acc_cap * sizeof(double) + 4 * (size_t)(acc_cap / 32 + kGatherNpw);
  const double *E64 = static_cast<const double *>(E);
  const float *E32 = static_cast<const float *>(E);
  if (a.nd == 27 && a.qdim == 3) {
    if (e_fp32) k_gather_emat<27, 3, float, kGatherThreadsQ2><<<grid, kGatherThreadsQ2, lds, s>>>(a, E32, thr);
    else k_gather_emat<27, 3, double, kGatherThreadsQ2><<<grid, kGatherThreadsQ2, lds, s>>>(a, E64, thr);
  } else if (a.nd == 10 && a.qdim == 3 && !e_fp32) {  // element-batched affine P2, FP64 matrix cores
    if (group_inc <= 32) k_gather_emat<10, 3, double, 64, 32><<<grid, 64, lds, s>>>(a, E64, thr);
    else k_gather_emat<10, 3, double, 64><<<grid, 64, lds, s>>>(a, E64, thr);
  } else if (a.nd == 20 && a.qdim == 3 && !e_fp32) {  // element-batched affine P3, FP64 matrix cores
    if (group_inc <= 32) k_gather_emat<20, 3, double, 64, 32><<<grid, 64, lds, s>>>(a, E64, thr);
    else k_gather_emat<20, 3, double, 64><<<grid, 64, lds, s>>>(a, E64, thr);
  } else if (a.nd == 10 && a.qdim == 3 && e_fp32) {  // element-batched affine P2 (bf16 split form)
    // groups of at most 32 incidences (the packed waves): half the static
    // LDS per group, so more groups fit on a CU
    if (group_inc <= 32) k_gather_emat<10, 3, float, 64, 32><<<grid, 64, lds, s>>>(a, E32, thr);
    else k_gather_emat<10, 3, float, 64><<<grid, 64, lds, s>>>(a, E32, thr);
  } else if (a.nd == 20 && a.qdim == 3 && e_fp32) {  // element-batched affine P3
    if (group_inc <= 32) k_gather_emat<20, 3, float, 64, 32><<<grid, 64, lds, s>>>(a, E32, thr);
    else k_gather_emat<20, 3, float, 64><<<grid, 64, lds, s>>>(a, E32, thr);
  }
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_gather_vec(hipStream_t s, int64_t n_nodes, int nd, int Q, const int32_t *inc_ptr,
                             const uint32_t *inc, const double *res, double *V) {
  if (n_nodes == 0) return hipSuccess;
  const int64_t n = n_nodes * Q;
  const unsigned grid = (unsigned)((n + 255) / 256);
  if (Q == 3) k_gather_vec<3><<<grid, 256, 0, s>>>(n, nd, inc_ptr, inc, res, V);
  else if (Q == 2) k_gather_vec<2><<<grid, 256, 0, s>>>(n, nd, inc_ptr, inc, res, V);
  else if (Q == 1) k_gather_vec<1><<<grid, 256, 0, s>>>(n, nd, inc_ptr, inc, res, V);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace gfx
