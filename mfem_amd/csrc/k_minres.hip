// Indefinite (KKT) Newton system and MINRES ("minres-indefinite-block").
//
// Unknowns [dx (3 nfree); ds (ns x nT); lambda (ns x nT)], ns = 6 on
// tetrahedra and 3 on triangles, the element parts stored structure-of-arrays
// (component i of element e at i * nT + e) so that they alias the mixed
// variable's ds and lambda arrays. On triangles the z rows of dx hold only
// the mass, which never couples to the rest, and stay exactly zero.
//
//   K = [[PMP, 0, Gx], [0, Hloc, C], [Gx^T, C, 0]]
//   Gx = -PJW diag(dSdF), C = vol Sym, Hloc = vol Hpsi (Hpsi = h^2 Hessian)
//
// is applied matrix-free as BlockMatrix::scaleAndAddTo does (reference
// src/linear_solvers/block_matrix.h:74-125 with Displacement::product_hessian,
// displacement.h:59-63, and MixedStretch::product_*, mixed_stretch.cpp:373-434).
// In this build's notation dsdF is ds/dF (6 x 9) and dSdF = dsdF^T Sym, so the
// lambda rows read -vol Sym dsdF Jloc dx + vol Sym ds and the x rows gather
// -vol Jloc^T dsdF^T Sym lambda per tet.
//
// The preconditioner is diag(Chebyshev(PMP), Hloc^-1, S_e^-1), S_e the element
// blocks of the Schur complement Gx^T Mlump^-1 Gx + C Hloc^-1 C, and MINRES
// follows Eigen 3.4's preconditioned Lanczos/Givens recurrence
// (unsupported/Eigen/src/IterativeSolvers/MINRES.h). One iteration is
//   k_mr_tet, k_mr_vertex   p/x update of the previous iteration; v_new = K w - beta v_old
//   k_mr_prec               alpha = v_new . w; v_new -= alpha v; w_new = P v_new (element
//                           blocks, first Chebyshev step of the mass block)
//   k_mr_cheb x 3           Chebyshev steps of the mass block
//   k_mr_fin_beta           beta_new, Givens rotation, stopping test
// with every scalar in one MinresCtrl block on the device. Lanczos vectors are
// stored unnormalised: v_k = V_k / beta_k, w_k = W_k / beta_k. Every sum is a
// per-workgroup partial reduced in index order by a one-workgroup kernel, or by
// every workgroup of the kernel that needs it (alpha, where the partials are few).
//
// At 23k tets no kernel has work for the chip (184 workgroups of elements, 24 of
// vertices at 256 each) and each is a chain of memory latencies, so the splits
// below are made for many short chains. An iteration takes 42 us, 76 us before (launches included):
// element product 23.7 -> 12.5 us (the update's loads no longer wait for its
// stores, in workgroups of their own), vertex product 15.2 -> 7.6 us and a Chebyshev
// step 6.6 -> 4.8 us (a lane to a component, 16 gathers in flight, 64 vertices a
// workgroup), preconditioner 9.2 + 3.9 + 4.5 us -> 6.5 us in one launch. Sums keep
// the order of one lane to a vertex and 256 vertices a workgroup: 500 iterations
// amplify a last place to 1e-4 and, on some states, to the leading digits.
#include <hip/hip_runtime.h>
#include "device_math.h"
#include "kernels.h"
#include "reduce.h"

namespace mfemhip {

namespace {

constexpr int kTetBS = 128;
constexpr int kVtxBS = 256;
constexpr int kFinBS = 1024;
constexpr int kLanes = 4;   // lanes of a vertex, one to a component (the fourth idles)
constexpr int kSub = kVtxBS / kWave;  // workgroups of a vertex partial, see vertex_partial
constexpr int kGather = 16;  // indices / values in flight per lane and gather batch
constexpr int kUpdate = 4;   // entries of the p/x update per lane

// Per-dimension element shape: corners, entries of s (Voigt, off-diagonals
// weighted 2 by Sym), consistent-mass divisor (rho vol / 20 on a tet, / 12 on
// a triangle), packed index of a symmetric ns x ns matrix (i <= j).
template <int DIM>
struct Elem {
  static constexpr int NC = DIM + 1, NS = DIM == 3 ? 6 : 3, NF = DIM * DIM;
  static constexpr double kMassDiv = DIM == 3 ? 20.0 : 12.0;
  __device__ static double symw(int i) { return i < DIM ? 1.0 : 2.0; }
  __device__ static int sym(int i, int j) {
    if (i > j) { const int t = i; i = j; j = t; }
    return DIM == 3 ? sym6(i, j) : sym3(i, j);
  }
};

// XCD-contiguous work split: workgroup b runs on XCD b % 8 (round-robin
// dispatch), and XCD x owns items [n x / 8, n (x + 1) / 8), so that the
// vertices and tets one XCD touches, and the lines their gathers read, stay
// in that XCD's L2. Returns n for lanes past the end of their range.
__device__ __forceinline__ int xcd_index(int n) {
  const int xcd = blockIdx.x & 7, lb = blockIdx.x >> 3;
  const long long start = (long long)n * xcd / 8, end = (long long)n * (xcd + 1) / 8;
  const long long i = start + (long long)lb * blockDim.x + threadIdx.x;
  return i < end ? (int)i : n;
}

// The same split with kLanes consecutive lanes to an item.
__device__ __forceinline__ int xcd_row(int n) {
  const int xcd = blockIdx.x & 7, lb = blockIdx.x >> 3;
  const long long start = (long long)n * xcd / 8, end = (long long)n * (xcd + 1) / 8;
  const long long i = start + (long long)lb * (blockDim.x / kLanes) + threadIdx.x / kLanes;
  return i < end ? (int)i : n;
}

// y + the component r of a row's mass blocks times scale * src, in row order:
// indices, then values, in flight together
__device__ __forceinline__ double mass_gather(const int* __restrict__ col,
                                              const double* __restrict__ mass, int b, int b1, int r,
                                              const double* __restrict__ src, double scale) {
  double y = 0;
  for (; b < b1; b += kGather) {
    int j[kGather];
    double mm[kGather], w[kGather];
#pragma unroll
    for (int u = 0; u < kGather; ++u) {
      j[u] = b + u < b1 ? col[b + u] : -1;
      mm[u] = b + u < b1 ? mass[b + u] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kGather; ++u)
      if (j[u] >= 0) w[u] = src[3 * j[u] + r];
#pragma unroll
    for (int u = 0; u < kGather; ++u)
      if (j[u] >= 0) y += mm[u] * (w[u] * scale);
  }
  return y;
}

// The component r of the sum of the element contributions at a vertex, in order
__device__ __forceinline__ double element_gather(const int* __restrict__ inc, int p, int p1, int r,
                                                 const double* __restrict__ fe) {
  double z = 0;
  for (; p < p1; p += kGather) {
    int ek[kGather];
    double f[kGather];
#pragma unroll
    for (int u = 0; u < kGather; ++u) ek[u] = p + u < p1 ? inc[p + u] : -1;
#pragma unroll
    for (int u = 0; u < kGather; ++u)
      if (ek[u] >= 0) f[u] = fe[(size_t)(ek[u] >> 2) * 12 + 3 * (ek[u] & 3) + r];
#pragma unroll
    for (int u = 0; u < kGather; ++u)
      if (ek[u] >= 0) z += f[u];
  }
  return z;
}

// a . b over the components, which the first three lanes of the vertex hold
__device__ __forceinline__ double dot3(double a, double b) {
  const int l0 = (int)(threadIdx.x & (kWave - kLanes));
  double d = 0;
#pragma unroll
  for (int r = 0; r < 3; ++r) d += __shfl(a, l0 + r) * __shfl(b, l0 + r);
  return d;
}

// Partial of a workgroup's 64 vertices (acc: the vertex's value in each of its
// lanes). The kSub workgroups of 256 consecutive vertices lie side by side in
// parts, and vertex_part adds them up: the order of one 256-lane workgroup.
__device__ __forceinline__ void vertex_partial(double acc, double* parts) {
  __shared__ double sm[kWave];
  if ((threadIdx.x & (kLanes - 1)) == 0) sm[threadIdx.x / kLanes] = acc;
  __syncthreads();
  if (threadIdx.x >= kWave) return;
  const double v = wave_sum(sm[threadIdx.x]);
  const int xcd = blockIdx.x & 7, lb = blockIdx.x >> 3;
  if (threadIdx.x == 0) parts[kSub * (8 * (lb / kSub) + xcd) + lb % kSub] = v;
}
// Partial i of ntet element workgroups followed by the vertex ones.
__device__ __forceinline__ double mr_part(const double* __restrict__ parts, int ntet, int i) {
  if (i < ntet) return parts[i];
  const double* v = parts + ntet + kSub * (size_t)(i - ntet);
  double r = v[0];
#pragma unroll
  for (int k = 1; k < kSub; ++k) r += v[k];
  return r;
}

inline int blocks_for(int n, int bs) {
  if (n <= 0) return 0;
  const int per_xcd = (n + 7) / 8;
  return 8 * ((per_xcd + bs - 1) / bs);
}

// Sum of ntet + nvtx partials in index order (strided by lane, then the block tree).
__device__ __forceinline__ double fin_sum(const double* parts, int ntet, int nvtx, double* sm) {
  double acc = 0;
  for (int i = threadIdx.x; i < ntet + nvtx; i += kFinBS) acc += mr_part(parts, ntet, i);
  return block_reduce_all<kFinBS, 0>(acc, sm);
}
// The same sum of at most kFinBS partials, to the last bit, by kTetBS threads.
constexpr int kFoldParts = kFinBS;
__device__ __forceinline__ double fold_sum(const double* parts, int ntet, int nvtx, double* sm) {
  constexpr int kChunks = kFinBS / kTetBS;  // of kWave partials, per wave
  const int n = ntet + nvtx, wid = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  double v[kChunks];
#pragma unroll
  for (int k = 0; k < kChunks; ++k) {
    const int i = (wid + k * (kTetBS / kWave)) * kWave + lane;
    v[k] = i < n ? mr_part(parts, ntet, i) : 0.0;
  }
#pragma unroll
  for (int k = 0; k < kChunks; ++k)
    if (k * kTetBS < n) {
      v[k] = wave_sum(v[k]);
      if (lane == 0) sm[wid + k * (kTetBS / kWave)] = v[k];
    }
  __syncthreads();
  double r = sm[0];
  for (int w = 1; w * kWave < n; ++w) r += sm[w];
  return r;
}

// ---------------------------------------------------------------- setup
// S_e = Sym (vol^2 B Lambda B^T + vol Hpsi^-1) Sym with B = dsdF Jloc and
// Lambda = 1 / Mlump on free corners (0 on pinned ones), inverted by Cholesky
// into Sinv (packed symmetric, stride nT). A block that is not positive
// definite becomes NaN, which the MINRES scalars report.
template <typename Real, int DIM>
__global__ __launch_bounds__(kTetBS) void k_kkt_setup(TetMeshDev m, const Real* __restrict__ dsdF,
                                                      const Real* __restrict__ Hinv,
                                                      const double* __restrict__ mlump_inv,
                                                      double* __restrict__ Sinv) {
  using E = Elem<DIM>;
  constexpr int NC = E::NC, NS = E::NS;
  const int e = xcd_index(m.nT);
  if (e >= m.nT) return;
  const int nT = m.nT;
  const double vol = m.vol[e];
  const int4 t = m.T[e];
  const int v[4] = {t.x, t.y, t.z, t.w};
  double lam[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int f = m.free_map[v[k]];
    lam[k] = f >= 0 ? mlump_inv[f] : 0.0;
  }
  // G(c, c') = sum_k Lambda_k dX(k, c) dX(k, c')
  double dx[3 * NC];
#pragma unroll
  for (int k = 0; k < NC; ++k)
#pragma unroll
    for (int c = 0; c < DIM; ++c) dx[3 * k + c] = m.dX[(3 * k + c) * nT + e];
  double G[DIM * DIM];
#pragma unroll
  for (int c = 0; c < DIM; ++c)
#pragma unroll
    for (int c2 = 0; c2 < DIM; ++c2) {
      double a = 0;
#pragma unroll
      for (int k = 0; k < NC; ++k) a += lam[k] * dx[3 * k + c] * dx[3 * k + c2];
      G[c + DIM * c2] = a;
    }
  // B Lambda B^T = dsdF (I (x) G) dsdF^T, one row r of F at a time
  double A[NS * NS];
#pragma unroll
  for (int i = 0; i < NS * NS; ++i) A[i] = 0.0;
#pragma unroll 1
  for (int r = 0; r < DIM; ++r) {
    double J[NS * DIM];  // J[i + NS c] = dsdF(i, r + DIM c)
#pragma unroll
    for (int c = 0; c < DIM; ++c)
#pragma unroll
      for (int i = 0; i < NS; ++i) J[i + NS * c] = (double)dsdF[(i + NS * (r + DIM * c)) * nT + e];
    double T[NS * DIM];  // T = J G
#pragma unroll
    for (int c = 0; c < DIM; ++c)
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        double a = 0;
#pragma unroll
        for (int c2 = 0; c2 < DIM; ++c2) a += J[i + NS * c2] * G[c2 + DIM * c];
        T[i + NS * c] = a;
      }
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        double a = 0;
#pragma unroll
        for (int c = 0; c < DIM; ++c) a += T[i + NS * c] * J[j + NS * c];
        A[i + NS * j] += a;
      }
  }
#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const double h = (double)Hinv[E::sym(i, j) * nT + e];
      A[i + NS * j] = E::symw(i) * (vol * vol * A[i + NS * j] + vol * h) * E::symw(j);
    }
  // Cholesky A = L L^T (lower, in place), then Sinv = L^-T L^-1
  bool ok = true;
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    double d = A[j + NS * j];
#pragma unroll
    for (int k = 0; k < j; ++k) d -= A[j + NS * k] * A[j + NS * k];
    ok = ok && d > 0.0;
    d = sqrt(fmax(d, 0.0));
    A[j + NS * j] = d;
    const double id = 1.0 / d;
#pragma unroll
    for (int i = j + 1; i < NS; ++i) {
      double s = A[i + NS * j];
#pragma unroll
      for (int k = 0; k < j; ++k) s -= A[i + NS * k] * A[j + NS * k];
      A[i + NS * j] = s * id;
    }
  }
  double Li[NS * NS];  // L^-1 (lower)
#pragma unroll
  for (int i = 0; i < NS * NS; ++i) Li[i] = 0.0;
#pragma unroll
  for (int c = 0; c < NS; ++c) {
    Li[c + NS * c] = 1.0 / A[c + NS * c];
#pragma unroll
    for (int i = c + 1; i < NS; ++i) {
      double s = 0;
#pragma unroll
      for (int k = c; k < i; ++k) s -= A[i + NS * k] * Li[k + NS * c];
      Li[i + NS * c] = s / A[i + NS * i];
    }
  }
#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int j = i; j < NS; ++j) {
      double s = 0;
#pragma unroll
      for (int k = j; k < NS; ++k) s += Li[k + NS * i] * Li[k + NS * j];
      Sinv[E::sym(i, j) * nT + e] = ok ? s : NAN;
    }
}

// ---------------------------------------------------------------- rhs
// b = [-PM (x_full - x_tilde - h^2 g); -vol g; vol Sym (S - s)]
// (linear_system.h:67-86): the inertia part per tet into fe (gathered per
// free vertex by k_kkt_rhs_vtx), the element parts straight into b.
template <int DIM>
__global__ __launch_bounds__(kTetBS) void k_kkt_rhs_tet(TetMeshDev m, const double* __restrict__ x,
                                                        Inertia in, const double* __restrict__ g,
                                                        const double* __restrict__ S,
                                                        const double* __restrict__ s,
                                                        double* __restrict__ fe, KktVec b,
                                                        double* __restrict__ parts) {
  __shared__ double sm[kTetBS / kWave];
  const int e = xcd_index(m.nT);
  double acc = 0.0;
  if (e < m.nT) {
    using E = Elem<DIM>;
    constexpr int NC = E::NC;
    const int nT = m.nT;
    const double vol = m.vol[e];
    const int4 t = m.T[e];
    const int v[4] = {t.x, t.y, t.z, t.w};
    double d[3 * NC], dsum[3] = {0, 0, 0};
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const double dd = x[3 * v[k] + r] - in.x_tilde[3 * v[k] + r] - in.h2g[r];
        d[3 * k + r] = dd;
        dsum[r] += dd;
      }
    const double mc = m.density * vol / E::kMassDiv;
    double* fo = fe + (size_t)e * 12;
#pragma unroll
    for (int j = 0; j < 3 * NC; ++j) fo[j] = -mc * (d[j] + dsum[j % 3]);
#pragma unroll
    for (int i = 0; i < E::NS; ++i) {
      const double bs = -vol * g[i * nT + e];
      const double bl = vol * E::symw(i) * (S[i * nT + e] - s[i * nT + e]);
      b.s[i * nT + e] = bs;
      b.l[i * nT + e] = bl;
      acc += bs * bs + bl * bl;
    }
  }
  block_partial<kTetBS, 0>(acc, parts, sm);
}

__global__ __launch_bounds__(kVtxBS) void k_kkt_rhs_vtx(int nfree, const int* __restrict__ inc_ptr,
                                                        const int* __restrict__ inc,
                                                        const double* __restrict__ fe, KktVec b,
                                                        double* __restrict__ parts) {
  const int i = xcd_row(nfree), lane = threadIdx.x & (kLanes - 1), r = min(lane, 2);
  double acc = 0.0;
  if (i < nfree) {
    const double a = element_gather(inc, inc_ptr[i], inc_ptr[i + 1], r, fe);
    if (lane < 3) b.x[3 * i + r] = a;
    acc = dot3(a, a);
  }
  vertex_partial(acc, parts);
}

// ---------------------------------------------------------------- iteration
struct MrVecs {
  KktVec wc;  // W_k (scale beta_k)
  KktVec vo;  // in: V_{k-1} (scale beta_{k-1}); out: V_{k+1} before alpha
  KktVec wo;  // W_{k-1} (scale beta_{k-1})
  KktVec pa;  // p_{k-2}
  KktVec pb;  // p_{k-3}
  KktVec pn;  // out: p_{k-1} (the slot of p_{k-4})
  KktVec x;   // solution
};

// Update of the previous iteration, p_{k-1} = (w_{k-1} - r2 p_{k-2} -
// r3 p_{k-3}) / r1 and x += beta_one c eta p_{k-1}, by the workgroups of k_mr_tet
// past those of the product (block = 0, 1, ... of them): the s part, the lambda
// part, the x part. A streaming pass whose loads are all in flight before the
// first store; inside the product it was a chain of 24 of them.
inline __host__ __device__ int update_blocks(long n) {
  return (int)((n + kUpdate * kTetBS - 1) / (kUpdate * kTetBS));
}
__device__ __forceinline__ void mr_update(const MinresCtrl& c, int block, long ne, long nx,
                                          const MrVecs& V) {
  const int be = update_blocks(ne);
  const int part = block < be ? 0 : block < 2 * be ? 1 : 2;
  const double* wo = part == 0 ? V.wo.s : part == 1 ? V.wo.l : V.wo.x;
  const double* pa = part == 0 ? V.pa.s : part == 1 ? V.pa.l : V.pa.x;
  const double* pb = part == 0 ? V.pb.s : part == 1 ? V.pb.l : V.pb.x;
  double* pn = part == 0 ? V.pn.s : part == 1 ? V.pn.l : V.pn.x;
  double* x = part == 0 ? V.x.s : part == 1 ? V.x.l : V.x.x;
  const long n = part == 2 ? nx : ne;
  const long i0 = (long)(block - part * be) * kUpdate * kTetBS + threadIdx.x;
  double w[kUpdate], a[kUpdate], b[kUpdate], xv[kUpdate];
#pragma unroll
  for (int u = 0; u < kUpdate; ++u) {
    const long i = i0 + u * kTetBS;
    if (i < n) {
      w[u] = wo[i];
      a[u] = pa[i];
      b[u] = pb[i];
      xv[u] = x[i];
    }
  }
#pragma unroll
  for (int u = 0; u < kUpdate; ++u) {
    const long i = i0 + u * kTetBS;
    if (i < n) {
      const double p = (w[u] / c.beta_prev - c.r2 * a[u] - c.r3 * b[u]) / c.r1;
      pn[i] = p;
      x[i] = xv[u] + c.coef * p;
    }
  }
}

template <typename Real, int DIM>
__global__ __launch_bounds__(kTetBS) void k_mr_tet(TetMeshDev m, const MinresCtrl* __restrict__ ctrl,
                                                   const Real* __restrict__ dsdF,
                                                   const Real* __restrict__ Hpsi, MrVecs V,
                                                   double* __restrict__ fe,
                                                   double* __restrict__ parts, int nproduct) {
  using E = Elem<DIM>;
  constexpr int NC = E::NC, NS = E::NS, NF = E::NF;
  constexpr int kFePitch = 13;  // x-row contributions staged per tet (odd pitch: LDS banks)
  __shared__ double sm[kTetBS / kWave];
  __shared__ double fe_stage[kTetBS * kFePitch];
  const MinresCtrl c = *ctrl;
  const int nT = m.nT;
  if ((int)blockIdx.x >= nproduct) {
    if (c.pending) mr_update(c, (int)blockIdx.x - nproduct, (long)NS * nT, 3L * m.nfree, V);
    return;
  }
  const int e = xcd_index(m.nT);
  if (c.done) return;
  double acc = 0.0;
  if (e < nT) {
    const double vol = m.vol[e];
    const double ib = 1.0 / c.beta;
    const double ratio = c.beta / c.beta_prev;
    double ws[NS], wl[NS], vo_s[NS], vo_l[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      ws[i] = V.wc.s[i * nT + e] * ib;
      wl[i] = V.wc.l[i * nT + e] * ib;
      vo_s[i] = V.vo.s[i * nT + e];
      vo_l[i] = V.vo.l[i * nT + e];
    }
    // Jloc w_x over the free corners
    const int4 t = m.T[e];
    const int v[4] = {t.x, t.y, t.z, t.w};
    double Fw[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i) Fw[i] = 0.0;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int f = m.free_map[v[k]];
      double wk[DIM];
#pragma unroll
      for (int r = 0; r < DIM; ++r) wk[r] = f >= 0 ? V.wc.x[3 * f + r] * ib : 0.0;
#pragma unroll
      for (int cc = 0; cc < DIM; ++cc) {
        const double d = m.dX[(3 * k + cc) * nT + e];
#pragma unroll
        for (int r = 0; r < DIM; ++r) Fw[r + DIM * cc] += wk[r] * d;
      }
    }
    // u = dsdF Fw and tv = dsdF^T (Sym w_l), one pass over dsdF
    double u[NS], tv[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i) tv[i] = 0.0;
#pragma unroll
    for (int i = 0; i < NS; ++i) u[i] = 0.0;
#pragma unroll
    for (int mm = 0; mm < NF; ++mm)
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const double js = (double)dsdF[(i + NS * mm) * nT + e];
        u[i] += js * Fw[mm];
        tv[mm] += js * E::symw(i) * wl[i];
      }
    // x rows of this element: -vol Jloc^T tv (the z rows of a triangle: 0),
    // staged in LDS and written below as contiguous runs
    double* fo = fe_stage + threadIdx.x * kFePitch;
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        double a = 0;
        if (r < DIM)
#pragma unroll
          for (int cc = 0; cc < DIM; ++cc) a += m.dX[(3 * k + cc) * nT + e] * tv[r + DIM * cc];
        fo[3 * k + r] = -vol * a;
      }
    // s rows: Hloc w_s + vol Sym w_l ; lambda rows: vol Sym (w_s - u)
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      double a = 0;
#pragma unroll
      for (int j = 0; j < NS; ++j) a += (double)Hpsi[E::sym(i, j) * nT + e] * ws[j];
      const double ys = vol * a + vol * E::symw(i) * wl[i];
      const double yl = vol * E::symw(i) * (ws[i] - u[i]);
      const long is = (long)i * nT + e;
      // v_new = K w - beta v_old, v_old = V_{k-1} / beta_{k-1}
      const double vs = ys - ratio * vo_s[i];
      const double vl = yl - ratio * vo_l[i];
      V.vo.s[is] = vs;
      V.vo.l[is] = vl;
      acc += fma(vs, ws[i], vl * wl[i]);
    }
  }
  // the staged x-row contributions of this wave's live tets, which are a
  // contiguous prefix of the wave (xcd_index hands out consecutive items)
  {
    const int lane = threadIdx.x & (kWave - 1);
    const int nlive = __popcll(__ballot(e < nT));
    const int e0 = __shfl(e, 0);
    const double* ws = fe_stage + (threadIdx.x - lane) * kFePitch;
    __syncthreads();
    for (int idx = lane; idx < nlive * 3 * NC; idx += kWave) {
      const int t = idx / (3 * NC), j = idx - t * (3 * NC);
      fe[(size_t)(e0 + t) * 12 + j] = ws[t * kFePitch + j];
    }
  }
  block_partial<kTetBS, 0>(acc, parts, sm);
}

__global__ __launch_bounds__(kVtxBS) void k_mr_vertex(int nfree, const int* __restrict__ rowptr,
                                                      const int* __restrict__ col,
                                                      const double* __restrict__ mass,
                                                      const int* __restrict__ inc_ptr,
                                                      const int* __restrict__ inc,
                                                      const double* __restrict__ fe,
                                                      const MinresCtrl* __restrict__ ctrl, MrVecs V,
                                                      double* __restrict__ parts) {
  const MinresCtrl c = *ctrl;
  if (c.done) return;
  const int i = xcd_row(nfree), lane = threadIdx.x & (kLanes - 1), r = min(lane, 2);
  double acc = 0.0;
  if (i < nfree) {
    const double ib = 1.0 / c.beta;
    const double ratio = c.beta / c.beta_prev;
    const long ir = 3L * i + r;
    const double vo = V.vo.x[ir], wi = V.wc.x[ir];
    const double y = mass_gather(col, mass, rowptr[i], rowptr[i + 1], r, V.wc.x, ib);
    const double z = element_gather(inc, inc_ptr[i], inc_ptr[i + 1], r, fe);
    const double vn = (y + z) - ratio * vo;
    if (lane < 3) V.vo.x[ir] = vn;
    acc = dot3(vn, wi * ib);
  }
  vertex_partial(acc, parts);
}

// alpha = v_new . w; the pending update has been applied by now.
__global__ __launch_bounds__(kFinBS) void k_mr_fin_alpha(MinresCtrl* ctrl, const double* parts,
                                                         int ntet, int nvtx) {
  __shared__ double sm[kFinBS / kWave];
  const bool done = ctrl->done;
  __syncthreads();
  if (threadIdx.x == 0) ctrl->pending = 0;
  if (done) return;
  const double a = fin_sum(parts, ntet, nvtx, sm);
  if (threadIdx.x == 0) ctrl->alpha = a;
}

// v_new -= alpha v_k (init: alpha = 0, v_k absent) and w_new = P v_new: by the
// first nelem workgroups on the element parts, Hloc^-1 = Hpsi^-1 / vol on s and
// S_e^-1 on lambda; by the others on the x part, with the first Chebyshev step of
// the mass block, r = v_new, d = D^-1 r / theta, z = d. With nvtx > 0 every
// workgroup sums alpha from parts_a itself while its loads are in flight
// (k_mr_fin_alpha and its launch took 6 us an iteration), and the first stores it.
template <typename Real, int DIM>
__global__ __launch_bounds__(kTetBS) void k_mr_prec(TetMeshDev m, MinresCtrl* ctrl, int init,
                                                    int nelem, int nvtx,
                                                    const double* __restrict__ parts_a,
                                                    const Real* __restrict__ Hinv,
                                                    const double* __restrict__ Sinv,
                                                    const double* __restrict__ dinv, double theta,
                                                    KktVec vn, KktVec vc, KktVec wn,
                                                    double* __restrict__ cr,
                                                    double* __restrict__ cd,
                                                    double* __restrict__ parts) {
  using E = Elem<DIM>;
  constexpr int NS = E::NS, NH = NS * (NS + 1) / 2;
  __shared__ double sm[kFinBS / kWave];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  if (!init && ctrl->done) {
    if (nvtx > 0 && first) ctrl->pending = 0;
    return;
  }
  const double beta = ctrl->beta;
  auto combine = [&] {  // alpha / beta; every thread comes here
    if (init) return 0.0;
    if (nvtx == 0) return ctrl->alpha / beta;
    const double alpha = fold_sum(parts_a, nelem, nvtx, sm);
    if (first) {
      ctrl->alpha = alpha;
      ctrl->pending = 0;  // the update of the previous iteration has been applied
    }
    return alpha / beta;
  };
  if ((int)blockIdx.x >= nelem) {
    const long n = 3L * m.nfree;
    const long ir = (long)((int)blockIdx.x - nelem) * kTetBS + threadIdx.x;
    double v = 0, c = 0, di = 0;
    if (ir < n) {
      v = vn.x[ir];
      if (!init) c = vc.x[ir];
      di = dinv[ir / 3];
    }
    const double ab = combine();
    if (ir >= n) return;
    if (!init) {
      v -= ab * c;
      vn.x[ir] = v;
    }
    const double d = di * v / theta;
    cr[ir] = v;
    cd[ir] = d;
    wn.x[ir] = d;
    return;
  }
  const int e = xcd_index(m.nT);
  const int nT = m.nT;
  double vs[NS], vl[NS], cs[NS], cl[NS], hi[NH], si[NH], vol = 1.0;
  if (e < nT) {
    vol = m.vol[e];
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const long is = (long)i * nT + e;
      vs[i] = vn.s[is];
      vl[i] = vn.l[is];
      cs[i] = init ? 0.0 : vc.s[is];
      cl[i] = init ? 0.0 : vc.l[is];
    }
#pragma unroll
    for (int k = 0; k < NH; ++k) {
      hi[k] = (double)Hinv[k * nT + e];
      si[k] = Sinv[k * nT + e];
    }
  }
  const double ab = combine();
  double acc = 0.0;
  if (e < nT) {
    if (!init)
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const long is = (long)i * nT + e;
        vs[i] -= ab * cs[i];
        vl[i] -= ab * cl[i];
        vn.s[is] = vs[i];
        vn.l[is] = vl[i];
      }
    const double iv = 1.0 / vol;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      double a = 0, b = 0;
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const int k = E::sym(i, j);
        a += hi[k] * vs[j];
        b += si[k] * vl[j];
      }
      const long is = (long)i * nT + e;
      const double zs = a * iv;
      wn.s[is] = zs;
      wn.l[is] = b;
      acc += vs[i] * zs + vl[i] * b;
    }
  }
  block_partial<kTetBS, 0>(acc, parts, sm);
}

// One Chebyshev step: r -= PMP d_in; d_out = c1 d_in + c2 D^-1 r; z += d_out.
// The last step also writes the partials of v_new . z.
__global__ __launch_bounds__(kVtxBS) void k_mr_cheb(int nfree, const int* __restrict__ rowptr,
                                                    const int* __restrict__ col,
                                                    const double* __restrict__ mass,
                                                    const double* __restrict__ dinv,
                                                    const MinresCtrl* __restrict__ ctrl, double c1,
                                                    double c2, const double* __restrict__ d_in,
                                                    double* __restrict__ d_out,
                                                    double* __restrict__ cr, KktVec vn, KktVec wn,
                                                    int last, int init,
                                                    double* __restrict__ parts) {
  if (!init && ctrl->done) return;
  const int i = xcd_row(nfree), lane = threadIdx.x & (kLanes - 1), r = min(lane, 2);
  double acc = 0.0;
  if (i < nfree) {
    const long ir = 3L * i + r;
    const double di = dinv[i], ri = cr[ir], dr = d_in[ir], zr = wn.x[ir], vr = vn.x[ir];
    const double y = mass_gather(col, mass, rowptr[i], rowptr[i + 1], r, d_in, 1.0);
    const double rr = ri - y;
    const double d = fma(c2 * di, rr, c1 * dr);
    const double z = zr + d;
    if (lane < 3) {
      cr[ir] = rr;
      d_out[ir] = d;
      wn.x[ir] = z;
    }
    if (last) acc = dot3(vr, z);
  }
  if (last) vertex_partial(acc, parts);
}

// beta_new, the Givens rotation and the stopping test of one iteration.
__global__ __launch_bounds__(kFinBS) void k_mr_fin_beta(MinresCtrl* ctrl, const double* parts,
                                                        int ntet, int nvtx) {
  __shared__ double sm[kFinBS / kWave];
  if (ctrl->done) return;
  const double b2 = fin_sum(parts, ntet, nvtx, sm);
  if (threadIdx.x != 0) return;
  MinresCtrl c = *ctrl;
  if (!(b2 >= 0.0)) {  // preconditioner not positive definite (or NaN)
    c.fail = 1;
    c.done = 1;
    *ctrl = c;
    return;
  }
  const double bn = sqrt(b2);
  const double beta = c.beta, alpha = c.alpha;
  const double r2 = c.s * alpha + c.c * c.c_old * beta;
  const double r3 = c.s_old * beta;
  const double r1_hat = c.c * alpha - c.c_old * c.s * beta;
  const double r1 = sqrt(r1_hat * r1_hat + bn * bn);
  c.c_old = c.c;
  c.s_old = c.s;
  c.c = r1_hat / r1;
  c.s = bn / r1;
  c.r1 = r1;
  c.r2 = r2;
  c.r3 = r3;
  c.coef = c.beta_one * c.c * c.eta;
  c.pending = 1;
  c.res2 *= c.s * c.s;
  if (c.res2 < c.threshold2) {
    c.done = 1;
  } else {
    c.eta = -c.s * c.eta;
    c.iter += 1;
    if (c.iter >= c.max_iters) c.done = 1;
  }
  c.beta_prev = beta;
  c.beta = bn;
  *ctrl = c;
}

// Control block for a bare product (beta = 1, nothing pending, not stopped).
__global__ void k_mr_ctrl_unit(MinresCtrl* ctrl) {
  MinresCtrl c{};
  c.beta = c.beta_prev = c.beta_one = c.r1 = 1.0;
  *ctrl = c;
}

// Scalars after the right-hand side and its preconditioned image.
__global__ __launch_bounds__(kFinBS) void k_mr_fin_init(MinresCtrl* ctrl, const double* parts_b,
                                                        const double* parts_w, int ntet, int nvtx,
                                                        double tol, int max_iters) {
  __shared__ double sm[kFinBS / kWave];
  const double rhs2 = fin_sum(parts_b, ntet, nvtx, sm);
  const double b2 = fin_sum(parts_w, ntet, nvtx, sm);
  if (threadIdx.x != 0) return;
  MinresCtrl c{};
  c.rhs2 = rhs2;
  c.threshold2 = tol * tol * rhs2;
  c.res2 = rhs2;
  c.max_iters = max_iters;
  c.c = c.c_old = 1.0;
  c.s = c.s_old = 0.0;
  c.eta = 1.0;
  c.beta_prev = 1.0;
  c.r1 = 1.0;
  if (rhs2 == 0.0 || max_iters <= 0) {
    c.done = 1;
    c.beta = c.beta_one = 1.0;
  } else if (!(b2 >= 0.0)) {
    c.done = 1;
    c.fail = 1;
    c.beta = c.beta_one = 1.0;
  } else {
    c.beta = c.beta_one = sqrt(b2);
  }
  *ctrl = c;
}

}  // namespace

int kkt_tet_blocks(int nT) { return blocks_for(nT, kTetBS); }
int kkt_vertex_blocks(int nfree) { return kSub * blocks_for(nfree, kVtxBS); }

template <typename Real>
void launch_kkt_setup(const KktSystem<Real>& S, hipStream_t st) {
  if (S.m.nT == 0) return;
  if (S.m.dim == 2)
    hipLaunchKernelGGL((k_kkt_setup<Real, 2>), dim3(kkt_tet_blocks(S.m.nT)), dim3(kTetBS), 0, st,
                       S.m, S.dsdF, S.Hinv, S.mlump_inv, S.Sinv);
  else
    hipLaunchKernelGGL((k_kkt_setup<Real, 3>), dim3(kkt_tet_blocks(S.m.nT)), dim3(kTetBS), 0, st,
                       S.m, S.dsdF, S.Hinv, S.mlump_inv, S.Sinv);
}

// Chebyshev constants for the mass block over [1/2, 5/2]: theta 1.5,
// delta 1, sigma = theta / delta; rho_0 = 1 / sigma, rho_j = 1 / (2 sigma -
// rho_{j-1}); step j uses c1 = rho_j rho_{j-1}, c2 = 2 rho_j / delta.
namespace {
constexpr double kChebTheta = 1.5, kChebDelta = 1.0;

template <typename Real>
void launch_precondition(const KktSystem<Real>& S, int init, KktVec vn, KktVec vc, KktVec wn,
                         hipStream_t st) {
  const int nbT = kkt_tet_blocks(S.m.nT), nbV = kkt_vertex_blocks(S.m.nfree);
  const int nvtx = nbV / kSub;
  const bool fold = !init && nvtx > 0 && nbT + nvtx <= kFoldParts;
  if (!init && !fold)
    hipLaunchKernelGGL(k_mr_fin_alpha, dim3(1), dim3(kFinBS), 0, st, S.ctrl, S.parts[0], nbT,
                       nvtx);
  const dim3 grid(nbT + (int)((3L * S.m.nfree + kTetBS - 1) / kTetBS));
  if (grid.x == 0) return;
  auto kernel = S.m.dim == 2 ? k_mr_prec<Real, 2> : k_mr_prec<Real, 3>;
  hipLaunchKernelGGL(kernel, grid, dim3(kTetBS), 0, st, S.m, S.ctrl, init, nbT, fold ? nvtx : 0, S.parts[0],
                     S.Hinv, S.Sinv, S.mdinv, kChebTheta, vn, vc, wn, S.cheb_r, S.cheb_d[0],
                     S.parts[1]);
  if (nbV == 0) return;
  const double sigma = kChebTheta / kChebDelta;
  double rho = 1.0 / sigma;
  for (int j = 1; j < kMassChebSteps; ++j) {
    const double rho1 = 1.0 / (2.0 * sigma - rho);
    const int last = j == kMassChebSteps - 1;
    hipLaunchKernelGGL(k_mr_cheb, dim3(nbV), dim3(kVtxBS), 0, st, S.m.nfree, S.rowptr, S.col,
                       S.mass, S.mdinv, S.ctrl, rho1 * rho, 2.0 * rho1 / kChebDelta,
                       S.cheb_d[(j - 1) & 1], S.cheb_d[j & 1], S.cheb_r, vn, wn, last, init,
                       S.parts[1] + nbT);
    rho = rho1;
  }
}

// The element part of v_new = K w - beta v_old, with the pending p/x update.
template <typename Real>
void launch_element_product(const KktSystem<Real>& S, const MrVecs& V, bool update,
                            hipStream_t st) {
  const int nbT = kkt_tet_blocks(S.m.nT), ns = S.m.dim == 2 ? 3 : 6;
  int grid = nbT;
  if (update) grid += 2 * update_blocks((long)ns * S.m.nT) + update_blocks(3L * S.m.nfree);
  if (grid == 0) return;
  auto kernel = S.m.dim == 2 ? k_mr_tet<Real, 2> : k_mr_tet<Real, 3>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kTetBS), 0, st, S.m, S.ctrl, S.dsdF, S.Hpsi, V, S.fe,
                     S.parts[0], nbT);
}
}  // namespace

template <typename Real>
void launch_minres_init(const KktSystem<Real>& S, const double* x_full, const Inertia& in,
                        const double* g, const double* Smat, const double* s, KktVec b, KktVec w,
                        double tol, int max_iters, hipStream_t st) {
  const int nbT = kkt_tet_blocks(S.m.nT), nbV = kkt_vertex_blocks(S.m.nfree);
  if (nbT > 0)
    if (S.m.dim == 2)
      hipLaunchKernelGGL((k_kkt_rhs_tet<2>), dim3(nbT), dim3(kTetBS), 0, st, S.m, x_full, in, g,
                         Smat, s, S.fe, b, S.parts[0]);
    else
      hipLaunchKernelGGL((k_kkt_rhs_tet<3>), dim3(nbT), dim3(kTetBS), 0, st, S.m, x_full, in, g,
                         Smat, s, S.fe, b, S.parts[0]);
  if (nbV > 0)
    hipLaunchKernelGGL(k_kkt_rhs_vtx, dim3(nbV), dim3(kVtxBS), 0, st, S.m.nfree, S.inc_ptr,
                       S.inc, S.fe, b, S.parts[0] + nbT);
  launch_precondition(S, 1, b, b, w, st);
  hipLaunchKernelGGL(k_mr_fin_init, dim3(1), dim3(kFinBS), 0, st, S.ctrl, S.parts[0],
                     S.parts[1], nbT, nbV / kSub, tol, max_iters);
}

template <typename Real>
void launch_minres_iteration(const KktSystem<Real>& S, const MinresBuffers& B, long k,
                             hipStream_t st, hipEvent_t* tet_ev) {
  const int nbT = kkt_tet_blocks(S.m.nT), nbV = kkt_vertex_blocks(S.m.nfree);
  auto mod3 = [](long j) { return (int)(((j % 3) + 3) % 3); };
  MrVecs V;
  V.wc = B.w[k & 1];
  V.wo = B.w[(k + 1) & 1];
  V.vo = B.v[(k + 1) & 1];
  V.pa = B.p[mod3(k - 2)];
  V.pb = B.p[mod3(k - 3)];
  V.pn = B.p[mod3(k - 1)];  // p_{k-1} replaces p_{k-4}
  V.x = B.x;
  if (tet_ev) (void)hipEventRecord(tet_ev[0], st);
  launch_element_product(S, V, true, st);
  if (tet_ev) (void)hipEventRecord(tet_ev[1], st);
  if (nbV > 0)
    hipLaunchKernelGGL(k_mr_vertex, dim3(nbV), dim3(kVtxBS), 0, st, S.m.nfree, S.rowptr, S.col,
                       S.mass, S.inc_ptr, S.inc, S.fe, S.ctrl, V, S.parts[0] + nbT);
  // v_new (in V_{k-1}'s buffer) -= alpha v_k; w_new into W_{k-1}'s buffer
  launch_precondition(S, 0, B.v[(k + 1) & 1], B.v[k & 1], B.w[(k + 1) & 1], st);
  hipLaunchKernelGGL(k_mr_fin_beta, dim3(1), dim3(kFinBS), 0, st, S.ctrl, S.parts[1], nbT,
                     nbV / kSub);
}

template <typename Real>
void launch_kkt_apply(const KktSystem<Real>& S, int which, KktVec in, KktVec out, KktVec scratch,
                      hipStream_t st) {
  const int nbT = kkt_tet_blocks(S.m.nT), nbV = kkt_vertex_blocks(S.m.nfree);
  if (which == 1) {  // out = P in
    launch_kkt_setup(S, st);
    launch_precondition(S, 1, in, in, out, st);
    return;
  }
  // out = K in - 1 * 0: the product kernels with beta = 1 and v_old = 0
  hipLaunchKernelGGL(k_mr_ctrl_unit, dim3(1), dim3(1), 0, st, S.ctrl);
  (void)hipMemsetAsync(out.x, 0, 3 * (size_t)S.m.nfree * sizeof(double), st);
  (void)hipMemsetAsync(out.s, 0, 6 * (size_t)S.m.nT * sizeof(double), st);
  (void)hipMemsetAsync(out.l, 0, 6 * (size_t)S.m.nT * sizeof(double), st);
  MrVecs V;
  V.wc = in;
  V.wo = in;
  V.vo = out;
  V.pa = V.pb = V.pn = V.x = scratch;
  launch_element_product(S, V, false, st);
  if (nbV > 0)
    hipLaunchKernelGGL(k_mr_vertex, dim3(nbV), dim3(kVtxBS), 0, st, S.m.nfree, S.rowptr, S.col,
                       S.mass, S.inc_ptr, S.inc, S.fe, S.ctrl, V, S.parts[0] + nbT);
}

#define MFEM_MINRES_INST(Real)                                                                  \
  template void launch_kkt_setup<Real>(const KktSystem<Real>&, hipStream_t);                    \
  template void launch_minres_init<Real>(const KktSystem<Real>&, const double*, const Inertia&, \
                                         const double*, const double*, const double*, KktVec,    \
                                         KktVec, double, int, hipStream_t);                      \
  template void launch_minres_iteration<Real>(const KktSystem<Real>&, const MinresBuffers&, long, \
                                              hipStream_t, hipEvent_t*);                         \
  template void launch_kkt_apply<Real>(const KktSystem<Real>&, int, KktVec, KktVec, KktVec,      \
                                       hipStream_t);
MFEM_MINRES_INST(float)
MFEM_MINRES_INST(double)

}  // namespace mfemhip
