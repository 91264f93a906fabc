// Batched small-matrix kernels of the orthogonalizer and the formers (FP64).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "small.hpp"

namespace mcnla {

namespace {

constexpr int kSmallThreads = 256;
constexpr int kLds = kMaxL * (kMaxL + 1);

// LDS of one eigen-problem.
struct EigLds {
  double a[kLds];
  double v[kLds];
  double cs[2 * kMaxL];  // lds_jacobi's rotations; lds_psd_eig's d and nrm
  int pq[2 * kMaxL];
  double red[2 * (kEigThreads / kWave)];
  int ord[kMaxL];
};

// Eigen-decomposition of the symmetric n x n matrix in sh.a (both triangles): w (descending) and
// V as batched_syev gives them.  A matrix that is positive definite at working precision goes
// through its Cholesky factor, any other one (the symmetric former's, a rank-deficient or
// non-finite Gram matrix) through the two-sided Jacobi.  The matrix is first scaled by a power of
// two to a largest diagonal entry in [1/2, 1).
__device__ void eig_sorted(int n, bool definite, EigLds& sh, double* w, double* V) {
  const int ld = lds_ld(n), tid = threadIdx.x;
  double* d = sh.cs;
  double* nrm = sh.cs + kMaxL;
  double mx = 0.0;
  for (int i = 0; i < n; ++i) mx = fmax(mx, sh.a[i * ld + i]);
  int e = 0;
  if (definite && mx > 0.0 && isfinite(mx)) {
    (void)frexp(mx, &e);
    __syncthreads();
    for (int q = tid; q < n * n; q += kEigThreads) {
      double* x = &sh.a[(q / n) * ld + q % n];
      *x = ldexp(*x, -e);
    }
    __syncthreads();
    if (lds_psd_eig(n, sh.a, sh.v, d, nrm, sh.pq)) {
      lds_psd_eig_sorted(n, sh.v, sh.a, nrm, sh.ord, ldexp(1.0, e), w, V);
      return;
    }
    __syncthreads();
    for (int q = tid; q < n * n; q += kEigThreads) {  // the matrix again, unscaled
      const int i = q / n, j = q % n;
      if (i >= j) {
        const double x = ldexp(i == j ? d[i] : sh.a[j * ld + i], e);
        sh.a[i * ld + j] = x;
      }
    }
    __syncthreads();
    for (int q = tid; q < n * n; q += kEigThreads) {
      const int i = q / n, j = q % n;
      if (i < j) sh.a[i * ld + j] = sh.a[j * ld + i];
    }
  }
  __syncthreads();
  lds_jacobi(n, sh.a, sh.v, true, sh.cs, sh.pq, sh.red);
  lds_eig_sorted(n, sh.a, sh.v, w, V, sh.ord);
}

// One workgroup per matrix: W[b] -> (w[b] descending, V[b]).
__global__ __launch_bounds__(kEigThreads) void batched_syev_kernel(const double* __restrict__ W,
                                                                  double* __restrict__ w,
                                                                  double* __restrict__ V, int n) {
  __shared__ EigLds sh;
  const int64_t b = blockIdx.x;
  const double* Wb = W + b * n * n;
  const int ld = lds_ld(n);
  for (int e = threadIdx.x; e < n * n; e += kEigThreads) {
    const int i = e / n, j = e % n;
    // symmetrize from the lower triangle (i >= j)
    sh.a[i * ld + j] = (i >= j) ? Wb[i * n + j] : Wb[j * n + i];
  }
  __syncthreads();
  eig_sorted(n, true, sh, w + b * n, V + b * n * n);
}

// T_i = V_i diag(1/sqrt(w_i)) into rows [i*l, (i+1)*l) of the Nl x l stack.
__global__ void orth_transforms_kernel(const double* __restrict__ w, const double* __restrict__ V,
                                       double* __restrict__ T, int64_t N, int l, int* bad) {
  const int64_t total = N * l * l;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = e / (l * l);
    const int r = (e / l) % l, c = e % l;
    const double ev = w[b * l + c];
    if (r == 0) {
      // an eigenvalue at or below l eps of the block's largest is zero at working precision:
      // the sketch does not have full column rank (or holds NaN / Inf)
      double wmax = 0.0;
      for (int q = 0; q < l; ++q) wmax = fmax(wmax, w[b * l + q]);
      if (!(ev > l * 0x1p-52 * wmax)) atomicAdd(bad, 1);
    }
    T[e] = V[e] / sqrt(ev);
  }
}

__global__ void gram_diag_blocks_kernel(const double* __restrict__ G, int64_t ldg,
                                        double* __restrict__ W, int64_t N, int l) {
  const int64_t total = N * l * l;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = e / (l * l);
    const int r = (e / l) % l, c = e % l;
    W[e] = G[(b * l + r) * ldg + b * l + c];
  }
}

// Bs = blockdiag(T)' G blockdiag(T), block (I, J) = T_I' G_IJ T_J for I >= J: one workgroup per
// block pair, G_IJ, T_I, T_J and H = G_IJ T_J in LDS (dynamic, 4 NP (NP + 1) doubles, l <= NP,
// zero-padded) and both products on f64 MFMA tiles.  Bs is symmetric in exact arithmetic; the
// entries with global row >= column are computed and written to both halves, so that it is exactly
// symmetric (its rows can then stand in for its columns).  Bound by one workgroup's chain of loads,
// products and stores per CU at l = 64 (33 KB a matrix): all loads are in flight together, and the
// block goes through LDS so that it and its mirror image are written in whole rows (the mirror entry
// by entry, 64 KB apart, and the loads one round after another took 1015 us at l = 64, N = 128, 396
// now, and 92 at l = 60, N = 32, 33 now).
constexpr int kCongThreads = 512;

template <int NP>
__global__ __launch_bounds__(kCongThreads) void congruence_kernel(const double* __restrict__ G,
                                                                 const double* __restrict__ T,
                                                                 double* __restrict__ Bs, int64_t N,
                                                                 int l) {
  extern __shared__ double smem[];
  constexpr int LD = NP + 1, NB = NP * LD, NT = NP / 16, NW = kCongThreads / kWave;
  constexpr int E = (NP * NP + kCongThreads - 1) / kCongThreads;
  double* sG = smem;  // then the result
  double* sTi = sG + NB;
  double* sTj = sTi + NB;
  double* sH = sTj + NB;
  const int64_t nl = N * l;
  // block pair p -> (I, J), I >= J, p = I (I + 1) / 2 + J
  const int64_t p = blockIdx.y * static_cast<int64_t>(gridDim.x) + blockIdx.x;
  if (p >= N * (N + 1) / 2) return;
  int64_t I = static_cast<int64_t>((sqrt(8.0 * static_cast<double>(p) + 1.0) - 1.0) / 2.0);
  while (I * (I + 1) / 2 > p) --I;
  while ((I + 1) * (I + 2) / 2 <= p) ++I;
  const int64_t J = p - I * (I + 1) / 2;
  const int tid = threadIdx.x;
  const double* g = G + I * l * nl + J * l;
  const double* ti = T + I * l * l;
  const double* tj = T + J * l * l;
  double v[3][E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = tid + u * kCongThreads, a = e / NP, b = e % NP;
    const bool in = a < l && b < l;
    v[0][u] = in ? g[a * nl + b] : 0.0;
    v[1][u] = in ? ti[a * l + b] : 0.0;
    v[2][u] = in ? tj[a * l + b] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = tid + u * kCongThreads, a = e / NP, b = e % NP;
    if (a >= NP) break;
    sG[a * LD + b] = v[0][u];
    sTi[a * LD + b] = v[1][u];
    sTj[a * LD + b] = v[2][u];
  }
  __syncthreads();
  const int wave = tid / kWave, lane = tid % kWave;
  for (int t = wave; t < NT * NT; t += NW) {  // H = G_IJ T_J
    const int i0 = (t / NT) * 16, j0 = (t % NT) * 16;
    const d4 acc = lds_mfma_tile<false, false>(NP, LD, sG, sTj, i0, j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) sH[(i0 + lane / 16 + 4 * r) * LD + j0 + lane % 16] = acc[r];
  }
  __syncthreads();
  for (int t = wave; t < NT * NT; t += NW) {  // T_I' H
    const int i0 = (t / NT) * 16, j0 = (t % NT) * 16;
    const d4 acc = lds_mfma_tile<true, false>(NP, LD, sTi, sH, i0, j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) sG[(i0 + lane / 16 + 4 * r) * LD + j0 + lane % 16] = acc[r];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = tid + u * kCongThreads, a = e / NP, b = e % NP;
    if (a >= l || b >= l) continue;
    Bs[(I * l + a) * nl + J * l + b] = sG[I == J && a < b ? b * LD + a : a * LD + b];
    if (I != J) Bs[(J * l + a) * nl + I * l + b] = sG[b * LD + a];
  }
}

// T_i = L_i^{-T} from the Cholesky factorization W_i = L_i L_i' (one workgroup per block), so
// that Y_i T_i has orthonormal columns when W_i = Y_i' Y_i.  L_0 is also written to L0 (lower
// triangle, zeros above).  A pivot that is not above l eps of W_i's largest diagonal entry flags
// *bad.
//
// One elimination makes both: step k subtracts a_ik / d_k times row k from the rows below it, in
// the trailing lower triangle of A (D = diag(d) in the end, L = A D^-1/2) and in X, which starts
// as I and ends as D^1/2 L^-1.  1024 threads own an entry of every 16th column each; one barrier
// per step, 0.5 us (12.8 us at l = 20, 25 at l = 40; factorization, division and a substitution by
// one thread per column, three barriers a step, took 25 and 65).
__global__ __launch_bounds__(kEigThreads) void cholesky_transforms_kernel(
    const double* __restrict__ W, double* __restrict__ T, double* __restrict__ L0, int l,
    int* bad) {
  __shared__ double a[kLds];
  __shared__ double x[kLds];
  __shared__ double rs[kMaxL];  // 1 / sqrt(d)
  const int ld = lds_ld(l);
  const int64_t b = blockIdx.x;
  const double* Wb = W + b * l * l;
  const int tid = threadIdx.x;
  for (int e = tid; e < l * l; e += kEigThreads) {
    const int i = e / l, j = e % l;
    a[i * ld + j] = (i >= j) ? Wb[i * l + j] : 0.0;
    x[i * ld + j] = i == j ? 1.0 : 0.0;
  }
  __syncthreads();
  // A pivot at or below l eps of the largest diagonal entry is zero at working precision: the
  // sketch does not have full column rank (or W holds NaN / Inf, which fails the test too).
  double wmax = 0.0;
  for (int i = 0; i < l; ++i) wmax = fmax(wmax, a[i * ld + i]);
  const double floor_piv = l * 0x1p-52 * wmax;
  __syncthreads();
  bool fail = false;
  const int r = tid >> 4, c0 = tid & 15;
  for (int k = 0; k < l; ++k) {
    const double akk = a[k * ld + k], d = (akk > 0.0) ? akk : 1.0;
    fail = fail || !(akk > floor_piv);
    if (tid == 0) rs[k] = 1.0 / sqrt(d);
    if (r > k && r < l) {
      const double f = a[r * ld + k] / d;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = c0 + 16 * j;
        if (c <= k)
          x[r * ld + c] -= f * x[k * ld + c];
        else if (c <= r)
          a[r * ld + c] -= f * a[c * ld + k];
      }
    }
    __syncthreads();
  }
  double* Tb = T + b * l * l;
  for (int e = tid; e < l * l; e += kEigThreads) {
    const int i = e / l, j = e % l;
    Tb[e] = i <= j ? x[j * ld + i] * rs[j] : 0.0;  // T = X'
    if (b == 0 && L0 != nullptr) L0[e] = (i >= j) ? a[i * ld + j] * rs[j] : 0.0;
  }
  if (fail && tid == 0) atomicAdd(bad, 1);
}

// out (m x n, row-major FP64, ld n) = A (FP32 or FP64, row- or column-major, lda), through
// 32 x 32 LDS tiles so that reads and writes are both coalesced.
template <typename TS, bool COLMAJOR>
__global__ __launch_bounds__(256) void to_rowmajor_f64_kernel(const TS* __restrict__ A, int64_t lda,
                                                             int64_t m, int64_t n,
                                                             double* __restrict__ out) {
  __shared__ double tile[32][33];
  const int64_t r0 = static_cast<int64_t>(blockIdx.y) * 32, c0 = static_cast<int64_t>(blockIdx.x) * 32;
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (COLMAJOR) {  // column c0 + ty + 8q, rows r0 + tx contiguous
      const int64_t r = r0 + tx, c = c0 + ty + 8 * q;
      tile[tx][ty + 8 * q] = (r < m && c < n) ? static_cast<double>(A[r + c * lda]) : 0.0;
    } else {
      const int64_t r = r0 + ty + 8 * q, c = c0 + tx;
      tile[ty + 8 * q][tx] = (r < m && c < n) ? static_cast<double>(A[r * lda + c]) : 0.0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t r = r0 + ty + 8 * q, c = c0 + tx;
    if (r < m && c < n) out[r * n + c] = tile[ty + 8 * q][tx];
  }
}

// Q_i = Y_i T_i in place: a workgroup takes kBdRows rows of one sketch, 64 at a time, through LDS
// (T_i once) and f64 MFMA tiles.  Memory-bound: Y read and written once (20000 x 512 in 32 us, 5.1
// TB/s; a thread per row and sketch, its row strided over the wave, took 957 us).
constexpr int kBdRows = 256;

template <typename T, int NP>
__global__ __launch_bounds__(256) void apply_blockdiag_kernel(T* __restrict__ Y, int64_t m,
                                                              int64_t N, int l,
                                                              const double* __restrict__ Tst) {
  constexpr int LA = NP + 2, LB = NP + 16, NT = NP / 16;  // fragments on distinct banks
  __shared__ double sy[64 * LA];
  __shared__ double st[NP * LB];
  const int64_t blk = blockIdx.y * static_cast<int64_t>(gridDim.x) + blockIdx.x;
  const int64_t b = blk % N, nl = N * l, first = blk / N * kBdRows;
  if (first >= m) return;
  const int64_t r1 = first + kBdRows < m ? first + kBdRows : m;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, c = lane & 15,
            kq = lane >> 4;
  for (int e = tid; e < NP * NP; e += 256) {
    const int i = e / NP, j = e % NP;
    st[i * LB + j] = i < l && j < l ? Tst[b * l * l + i * l + j] : 0.0;
  }
  for (int64_t r0 = first; r0 < r1; r0 += 64) {
    constexpr int E = 64 * NP / 256;
    double v[E];
#pragma unroll
    for (int u = 0; u < E; ++u) {
      const int e = tid + u * 256, i = e / NP, j = e % NP;
      v[u] = r0 + i < r1 && j < l ? static_cast<double>(Y[(r0 + i) * nl + b * l + j]) : 0.0;
    }
    __syncthreads();  // the previous rows are done with sy (and T_i is in place)
#pragma unroll
    for (int u = 0; u < E; ++u) sy[(tid + u * 256) / NP * LA + (tid + u * 256) % NP] = v[u];
    __syncthreads();
    d4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int k = 0; k < NP; k += 4) {
      const double y = sy[(wave * 16 + c) * LA + k + kq];
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(y, st[(k + kq) * LB + 16 * j + c], acc[j], 0,
                                                      0, 0);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t i = r0 + wave * 16 + kq + 4 * r;
        if (i < r1 && 16 * j + c < l) Y[i * nl + b * l + 16 * j + c] = static_cast<T>(acc[j][r]);
      }
  }
}

// Former: eig of Wg (l x l) -> eigw (descending), eigv; Wk = eigv[:, :k]; S = sqrt(eigw[:k]).
// symmetric (Wg = Qbar' A Qbar of a symmetric A): the k largest eigenpairs in ascending order,
// S = the eigenvalues themselves (row_block_symmetric_former.hpp:65-66,127-130).
// One l x l problem on one workgroup.
__global__ __launch_bounds__(kEigThreads) void former_small_kernel(const double* __restrict__ Wg,
                                                                  int l, int k, bool symmetric,
                                                                  double* __restrict__ eigw,
                                                                  double* __restrict__ eigv,
                                                                  double* __restrict__ Wk,
                                                                  double* __restrict__ S) {
  __shared__ EigLds sh;
  const int ld = lds_ld(l);
  for (int e = threadIdx.x; e < l * l; e += kEigThreads) {
    const int i = e / l, j = e % l;
    sh.a[i * ld + j] = 0.5 * (Wg[i * l + j] + Wg[j * l + i]);
  }
  __syncthreads();
  eig_sorted(l, !symmetric, sh, eigw, eigv);
  for (int e = threadIdx.x; e < l * k; e += blockDim.x) {
    const int i = e / k, j = e % k;
    Wk[e] = eigv[i * l + (symmetric ? k - 1 - j : j)];
  }
  for (int j = threadIdx.x; j < k; j += blockDim.x)
    S[j] = symmetric ? eigw[k - 1 - j] : sqrt(fmax(eigw[j], 0.0));
}

__global__ void scale_columns_kernel(double* __restrict__ X, int64_t rows, int k,
                                     const double* __restrict__ S, bool inverse) {
  const int64_t total = rows * k;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const double s = S[e % k];
    X[e] = inverse ? X[e] / s : X[e] * s;
  }
}

// out[j] = ||X[:, j]||_2 for a row-major rows x k matrix; one workgroup per column.
__global__ void column_norms_kernel(const double* __restrict__ X, int64_t rows, int k,
                                    double* __restrict__ out) {
  __shared__ double red[kSmallThreads / kWave];
  const int j = blockIdx.x;
  double acc = 0.0;
  for (int64_t r = threadIdx.x; r < rows; r += blockDim.x) {
    const double x = X[r * k + j];
    acc += x * x;
  }
  acc = wave_sum(acc);
  if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) s += red[w];
    out[j] = sqrt(s);
  }
}

unsigned grid_for(int64_t total, int threads = 256, int64_t cap = 16384) {
  int64_t b = ceil_div(total, threads);
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return static_cast<unsigned>(b);
}

}  // namespace

void batched_syev(const double* W, double* w, double* V, int64_t batch, int n, hipStream_t st) {
  MCNLA_REQUIRE(n >= 1 && n <= kMaxL, MCNLA_ERR_INVALID, "eigen problem larger than 64");
  if (batch <= 0) return;
  hipLaunchKernelGGL(batched_syev_kernel, dim3(static_cast<unsigned>(batch)), dim3(kEigThreads),
                     0, st, W, w, V, n);
  MCNLA_LAUNCHED();
}

void orth_transforms(const double* w, const double* V, double* Tst, int64_t N, int l, int* bad,
                     hipStream_t st) {
  hipLaunchKernelGGL(orth_transforms_kernel, dim3(grid_for(N * l * l)), dim3(256), 0, st, w, V, Tst,
                     N, l, bad);
  MCNLA_LAUNCHED();
}

void gram_diag_blocks(const double* G, int64_t ldg, double* W, int64_t N, int l, hipStream_t st) {
  hipLaunchKernelGGL(gram_diag_blocks_kernel, dim3(grid_for(N * l * l)), dim3(256), 0, st, G, ldg,
                     W, N, l);
  MCNLA_LAUNCHED();
}

void congruence_blockdiag(const double* G, const double* Tst, double* Bs, int64_t N, int l,
                          hipStream_t st) {
  MCNLA_REQUIRE(l >= 1 && l <= kMaxL, MCNLA_ERR_INVALID, "l > 64");
  const int64_t pairs = N * (N + 1) / 2;
  if (pairs == 0) return;
  const int np = pad16(l);
  const size_t lds = static_cast<size_t>(4) * np * (np + 1) * sizeof(double);
  const int64_t gx = std::min<int64_t>(pairs, 1 << 22);  // a dimension holds fewer than 2^32 threads
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(ceil_div(pairs, gx)));
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kCongThreads), lds, st, G, Tst, Bs, N, l);
  };
  if (np == 16) go(congruence_kernel<16>);
  else if (np == 32) go(congruence_kernel<32>);
  else if (np == 48) go(congruence_kernel<48>);
  else go(congruence_kernel<64>);
  MCNLA_LAUNCHED();
}

void to_rowmajor_f64(const void* A, int64_t lda, bool a_f32, bool colmajor, int64_t m, int64_t n,
                     double* out, hipStream_t st) {
  if (m == 0 || n == 0) return;
  MCNLA_REQUIRE(ceil_div(m, 32) < 65536, MCNLA_ERR_INVALID, "too many rows for the converter");
  const dim3 grid(static_cast<unsigned>(ceil_div(n, 32)), static_cast<unsigned>(ceil_div(m, 32)));
  if (a_f32) {
    if (colmajor)
      hipLaunchKernelGGL((to_rowmajor_f64_kernel<float, true>), grid, dim3(256), 0, st,
                         static_cast<const float*>(A), lda, m, n, out);
    else
      hipLaunchKernelGGL((to_rowmajor_f64_kernel<float, false>), grid, dim3(256), 0, st,
                         static_cast<const float*>(A), lda, m, n, out);
  } else {
    if (colmajor)
      hipLaunchKernelGGL((to_rowmajor_f64_kernel<double, true>), grid, dim3(256), 0, st,
                         static_cast<const double*>(A), lda, m, n, out);
    else
      hipLaunchKernelGGL((to_rowmajor_f64_kernel<double, false>), grid, dim3(256), 0, st,
                         static_cast<const double*>(A), lda, m, n, out);
  }
  MCNLA_LAUNCHED();
}

void cholesky_transforms(const double* W, int64_t N, int l, double* Tst, double* L0, int* bad,
                         hipStream_t st) {
  MCNLA_REQUIRE(l >= 1 && l <= kMaxL, MCNLA_ERR_INVALID, "l > 64");
  if (N <= 0) return;
  hipLaunchKernelGGL(cholesky_transforms_kernel, dim3(static_cast<unsigned>(N)), dim3(kEigThreads),
                     0, st, W, Tst, L0, l, bad);
  MCNLA_LAUNCHED();
}

void apply_blockdiag(void* Y, bool y_f32, int64_t m, int64_t N, int l, const double* Tst,
                     hipStream_t st) {
  MCNLA_REQUIRE(l <= kMaxL, MCNLA_ERR_INVALID, "l > 64");
  if (m <= 0 || N <= 0) return;
  const int64_t blocks = ceil_div(m, kBdRows) * N, gx = std::min<int64_t>(blocks, 1 << 22);
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(ceil_div(blocks, gx)));
  auto launch = [&](auto* y) {
    using T = std::remove_pointer_t<decltype(y)>;
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, y, m, N, l, Tst);
    };
    if (l <= 16) go(apply_blockdiag_kernel<T, 16>);
    else if (l <= 32) go(apply_blockdiag_kernel<T, 32>);
    else if (l <= 48) go(apply_blockdiag_kernel<T, 48>);
    else go(apply_blockdiag_kernel<T, 64>);
  };
  if (y_f32) launch(static_cast<float*>(Y));
  else launch(static_cast<double*>(Y));
  MCNLA_LAUNCHED();
}

void former_small(const double* Wg, int l, int k, double* eigw, double* eigv, double* Wk,
                  double* S, hipStream_t st, bool symmetric) {
  MCNLA_REQUIRE(l >= 1 && l <= kMaxL && k >= 1 && k <= l, MCNLA_ERR_INVALID, "former sizes");
  hipLaunchKernelGGL(former_small_kernel, dim3(1), dim3(kEigThreads), 0, st, Wg, l, k, symmetric,
                     eigw, eigv, Wk, S);
  MCNLA_LAUNCHED();
}

void scale_columns(double* X, int64_t rows, int k, const double* S, bool inverse,
                   hipStream_t st) {
  hipLaunchKernelGGL(scale_columns_kernel, dim3(grid_for(rows * k)), dim3(256), 0, st, X, rows, k,
                     S, inverse);
  MCNLA_LAUNCHED();
}

void column_norms(const double* X, int64_t rows, int k, double* out, hipStream_t st) {
  hipLaunchKernelGGL(column_norms_kernel, dim3(static_cast<unsigned>(k)), dim3(kSmallThreads), 0,
                     st, X, rows, k, out);
  MCNLA_LAUNCHED();
}

}  // namespace mcnla
