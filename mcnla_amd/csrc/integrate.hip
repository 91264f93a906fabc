// Integrators on the Gram matrix Bs = Qs' Qs (Nl x Nl), FP64.
//
// Both KN and Wen-Yin only touch Qs through products Qs'(Qs X) = Bs X, so once Bs is formed
// every iteration works on Nl x l and l x l matrices that stay in L2 (the reference's Gramian
// forms, row_block_gramian_kolmogorov_nagumo_integrator.hpp:106-226 and
// row_block_gramian_wen_yin_integrator.hpp:114-328).  The basis is carried as coefficients:
// Qc = Q0 F~ + Qs E~, so Qbar = Qs * M with M = E~ + [F~; 0].
//
// Every iteration t is a fixed sequence of kernels gated by st->converged_at: a kernel of
// iteration t does nothing once convergence was detected at an earlier iteration, so the host can
// enqueue a chunk of iterations and synchronize once per chunk.  Iteration t reads the buffers of
// parity t&1 and writes parity (t+1)&1.
#include "common.hpp"
#include "kernels.hpp"
#include "small.hpp"

#include <algorithm>
#include <climits>
#include <vector>

namespace mcnla {

struct IntegratorState {
  int converged_at;  // iteration index that met the stopping test, INT_MAX while running
  int nan_seen;      // a non-finite value appeared in the l x l step
  double res;        // last residual (KN: ||s - 1||_2, WY: mu)
  double taug, zeta, phi, mu;  // Wen-Yin scalars
};
static_assert(sizeof(IntegratorState) <= 256, "the state's slot in the workspace");

namespace {

constexpr int kThreads = 256;
constexpr int kRows = 32;   // Nl rows per workgroup in the WY step-size pass
constexpr int kURows = 32;  // Nl rows per workgroup in the WY update
constexpr int kPRows = 64;  // Nl rows per workgroup in the partial dot products

__device__ __forceinline__ bool skip(const IntegratorState* st, int t) {
  return st->converged_at < t;
}

// Per-block partial products over kPRows rows of the Nl x l matrices B and Bg:
// P[blk][0] = B_blk' B_blk, P[blk][1] = B_blk' Bg_blk, P[blk][2] = Bg_blk' Bg_blk (nparts 3).
__global__ __launch_bounds__(kThreads) void gram_partials_kernel(int t, const IntegratorState* st,
                                                                int64_t nl, int l,
                                                                const double* __restrict__ B,
                                                                const double* __restrict__ Bg,
                                                                double* __restrict__ P,
                                                                int nparts) {
  if (skip(st, t)) return;
  __shared__ double sB[kPRows][kMaxL + 1];
  __shared__ double sG[kPRows][kMaxL + 1];
  const int64_t r0 = blockIdx.x * (int64_t)kPRows;
  for (int e = threadIdx.x; e < kPRows * l; e += kThreads) {
    const int rr = e / l, j = e % l;
    const int64_t r = r0 + rr;
    sB[rr][j] = (r < nl) ? B[r * l + j] : 0.0;
    sG[rr][j] = (r < nl) ? Bg[r * l + j] : 0.0;
  }
  __syncthreads();
  // the nparts l x l products over the block's rows on f64 MFMA tiles (16 x 16, k = row)
  double* Pb = P + blockIdx.x * (int64_t)nparts * l * l;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int nt1 = pad16(l) / 16, tiles = nt1 * nt1;
  for (int tile = wave; tile < nparts * tiles; tile += kThreads / kWave) {
    const int part = tile / tiles, i0 = ((tile % tiles) / nt1) * 16, j0 = (tile % nt1) * 16;
    const double(*X)[kMaxL + 1] = (part == 2) ? sG : sB;
    const double(*Y)[kMaxL + 1] = (part == 0) ? sB : sG;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int k0 = 0; k0 < kPRows; k0 += 4) {
      const int k = k0 + lane / 16;
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(X[k][i0 + lane % 16], Y[k][j0 + lane % 16], acc,
                                                 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + lane / 16 + 4 * r, j = j0 + lane % 16;
      if (i < l && j < l) Pb[part * l * l + i * l + j] = acc[r];
    }
  }
}

// sum_blk P[blk][q] in block order (deterministic).  The loads of 16 blocks are issued before
// any is added, so a thread waits for one memory round trip per 16 blocks, not per block.
__device__ __forceinline__ double sum_partials(const double* __restrict__ P, int64_t nblk,
                                               int64_t count, int64_t q) {
  double total = 0.0;
  for (int64_t b0 = 0; b0 < nblk; b0 += 16) {
    double v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = (b0 + j < nblk) ? P[(b0 + j) * count + q] : 0.0;
#pragma unroll
    for (int j = 0; j < 16; ++j) total += v[j];
  }
  return total;
}

// Two such sums at once (32 loads in flight); q1 < 0 skips the second.
__device__ __forceinline__ void sum_partials2(const double* __restrict__ P, int64_t nblk,
                                              int64_t count, int64_t q0, int64_t q1, double& s0,
                                              double& s1) {
  s0 = 0.0;
  s1 = 0.0;
  for (int64_t b0 = 0; b0 < nblk; b0 += 16) {
    double v[16], w[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      v[j] = (b0 + j < nblk) ? P[(b0 + j) * count + q0] : 0.0;
      w[j] = (b0 + j < nblk && q1 >= 0) ? P[(b0 + j) * count + q1] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      s0 += v[j];
      s1 += w[j];
    }
  }
}

__global__ void reduce_partials_kernel(int t, const IntegratorState* st,
                                       const double* __restrict__ P, int64_t nblk, int count,
                                       double scale, double* __restrict__ out) {
  if (skip(st, t)) return;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= count) return;
  out[q] = scale * sum_partials(P, nblk, count, q);
}

// A KN partial holds the lower triangles of Bc'Bc and of Bc'Bg + Bg'Bc over some rows, one after
// the other, row by row: l (l + 1) doubles.
__device__ __forceinline__ int tri(int i, int j) {
  return i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i;
}

// The KN l x l step (row_block_kolmogorov_nagumo_integrator.hpp:146-201): Dc = Bc'Bc/N and
// Dgc = sym(Bc'Bgc)/N from the partials P (nblk of them, as above), Z = Dgc - Dc^2,
// eig(Z), s = sqrt(1/2 + sqrt(1/4 - lambda)), C = V diag(s) V', Cinv = V diag(1/s) V',
// F = C - Dc Cinv, convergence when !(||s - 1||_2 >= tol).
//
// C and Cinv are matrix functions of Z, so they are computed here without the eigenvectors:
// X = (I - 4Z)^{1/2} and then C = ((I + X)/2)^{1/2}, Cinv = C^{-1} by two coupled Newton-Schulz
// iterations on MFMA tiles in LDS (both converge quadratically because Z is positive
// semidefinite with lambda <= 1/4), and ||s - 1||_2 = ||C - I||_F.  Should an iteration not
// converge (lambda at or above 1/4, non-finite input) the step falls back to a Jacobi
// eigen-decomposition and the formulas above, which also reproduce the reference's NaN there.
// The series form of the step, for x = 4Z of small norm (all but the first few iterations: rho =
// ||x||_F falls below 0.13 within five of 20 to 80 iterations on the workloads measured).  With
// s = sqrt(1/2 + sqrt(1/4 - z)) = sqrt((1 + sqrt(1 - x)) / 2), the powers s^-r are
// sum_k a_k x^k with a_0 = 1, a_{k+1} / a_k = (2k + r)(2k + r + 1) / (4 (k + 1)(k + r + 1)) (the
// r-th power of the Catalan generating function): C is r = -1/2 and Cinv r = 1/2.  Both are
// evaluated to degree 4b - 1 (Paterson-Stockmeyer with x, x^2, x^3, x^4), b the smallest whose
// truncation is below 1.5e-17.
constexpr int kSeriesMaxB = 10;
struct SeriesTable {
  double c[4 * kSeriesMaxB] = {}, ci[4 * kSeriesMaxB] = {};
  constexpr SeriesTable() {
    for (int which = 0; which < 2; ++which) {
      const double r = which == 0 ? -0.5 : 0.5;
      double a = 1.0;
      for (int k = 0; k < 4 * kSeriesMaxB; ++k) {
        (which == 0 ? c : ci)[k] = a;
        a *= (2 * k + r) * (2 * k + r + 1) / (4 * (k + 1) * (k + r + 1));
      }
    }
  }
};
__constant__ const SeriesTable kSeries;
// rho up to which degree 4b - 1 suffices, b = 2, 3, ... (the tail sum a_k rho^k, k >= 4b, of Cinv
// is 1.5e-17 there).
__device__ __forceinline__ int series_blocks(double rho) {
  constexpr double limit[kSeriesMaxB - 1] = {0.01435, 0.06178, 0.12669, 0.19394, 0.25695,
                                             0.31369, 0.36401, 0.40845, 0.44771};
  int b = 2;
  for (; b <= kSeriesMaxB; ++b)
    if (rho <= limit[b - 2]) return b;
  return 0;  // also for a NaN
}

constexpr int kStepThreads = 512;
constexpr int kStepWaves = kStepThreads / kWave;

// Leading dimension of the np x np LDS matrices of the series step: rows and column walks of the
// 16 x 16 x 4 fragments on distinct banks (at np = 64, where four matrices would not fit, pairs).
template <int NP>
__host__ __device__ constexpr int series_ld() {
  return NP == 16 ? 18 : NP == 64 ? 66 : 50;
}
constexpr int kStepBuf = kMaxL * series_ld<kMaxL>();  // doubles per buffer
static_assert(kMaxL * (kMaxL + 1) <= kStepBuf, "the other forms' buffers fit");

// One 16 x 16 tile of A B + acc for symmetric A, B in LDS (both read along rows).
template <int NP>
__device__ __forceinline__ d4 sym_tile(const double* A, const double* B, int i0, int j0, d4 acc) {
  constexpr int LD = series_ld<NP>();
  const int lane = threadIdx.x & (kWave - 1), c = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int k = 0; k < NP; k += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[(k + kq) * LD + i0 + c], B[(k + kq) * LD + j0 + c],
                                               acc, 0, 0, 0);
  return acc;
}

// Writes a tile of the lower triangle and its mirror image.
template <int NP>
__device__ __forceinline__ void put_sym(double* X, int i0, int j0, const d4& v) {
  constexpr int LD = series_ld<NP>();
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = i0 + (lane >> 4) + 4 * r, j = j0 + (lane & 15);
    X[i * LD + j] = v[r];
    if (i0 != j0) X[j * LD + i] = v[r];
  }
}

// The lower-triangle tile q (0, 1, ... row by row): its origin.
__device__ __forceinline__ void lower_tile(int q, int& i0, int& j0) {
  const int ti = q >= 6 ? 3 : q >= 3 ? 2 : q >= 1 ? 1 : 0;
  i0 = ti * 16;
  j0 = (q - ti * (ti + 1) / 2) * 16;
}

// All forms of the step run on kStepThreads threads (the whole workgroup) with four buffers of
// kStepBuf doubles in smem, and leave Cinv in the second and F in the third (leading dimension
// series_ld<NP>(); F is zero past l).  They return ||C - I||_F (NaN or infinite when Z is not).

// The eigen-decomposition form.
template <int NP>
__device__ double kn_step_eigen(int l, double invN, const double* __restrict__ P, int64_t nblk,
                                double* smem) {
  __shared__ double s[kMaxL];
  __shared__ double cs[2 * kMaxL];
  __shared__ int pq[2 * kMaxL];
  __shared__ double red[8];
  constexpr int LD = series_ld<NP>(), EP = (NP * NP + kStepThreads - 1) / kStepThreads;
  double* z = smem;
  double* v = smem + kStepBuf;
  double* a = smem + 2 * kStepBuf;
  double* dc = smem + 3 * kStepBuf;
  const int ld = lds_ld(l), ll = l * l, half = l * (l + 1) / 2;
  for (int e = threadIdx.x; e < ll; e += kStepThreads) {  // Dc into dc, Dgc into a
    const int i = e / l, j = e % l, q = tri(i, j);
    dc[i * ld + j] = invN * sum_partials(P, nblk, 2 * half, q);
    a[i * ld + j] = 0.5 * invN * sum_partials(P, nblk, 2 * half, half + q);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < ll; e += kStepThreads) {  // Z = Dgc - Dc Dc'
    const int i = e / l, j = e % l;
    double x = a[i * ld + j];
    for (int q = 0; q < l; ++q) x -= dc[i * ld + q] * dc[j * ld + q];
    z[i * ld + j] = x;
  }
  __syncthreads();
  lds_jacobi(l, z, v, true, cs, pq, red);
  for (int i = threadIdx.x; i < l; i += kStepThreads)
    s[i] = sqrt(0.5 + sqrt(0.25 - z[i * ld + i]));
  __syncthreads();
  for (int e = threadIdx.x; e < ll; e += kStepThreads) {  // Cinv into `a`
    const int i = e / l, j = e % l;
    double ci = 0.0;
    for (int q = 0; q < l; ++q) ci += v[i * ld + q] * v[j * ld + q] / s[q];
    a[i * ld + j] = ci;
  }
  __syncthreads();
  double f[EP], ci[EP];  // F = C - Dc Cinv, C on the fly
#pragma unroll
  for (int u = 0; u < EP; ++u) {
    const int e = threadIdx.x + u * kStepThreads, i = e / NP, j = e % NP;
    f[u] = 0.0;
    ci[u] = 0.0;
    if (i < l && j < l) {
      double c = 0.0, dci = 0.0;
      for (int q = 0; q < l; ++q) {
        c += v[i * ld + q] * v[j * ld + q] * s[q];
        dci += dc[i * ld + q] * a[q * ld + j];
      }
      f[u] = c - dci;
      ci[u] = a[i * ld + j];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < EP; ++u) {
    const int e = threadIdx.x + u * kStepThreads, i = e / NP, j = e % NP;
    if (i >= NP) break;
    smem[kStepBuf + i * LD + j] = ci[u];
    smem[2 * kStepBuf + i * LD + j] = f[u];
  }
  __syncthreads();
  double r = 0.0;
  for (int q = 0; q < l; ++q) r += (s[q] - 1.0) * (s[q] - 1.0);
  return sqrt(r);
}

// The Newton-Schulz form: X = (I - 4Z)^{1/2}, C = ((I + X)/2)^{1/2}, Cinv = C^{-1}.
template <int NP>
__device__ double kn_step_ns(int l, double invN, const double* __restrict__ P, int64_t nblk,
                             double* smem, double* red) {
  constexpr int LD = series_ld<NP>(), NT1 = NP / 16;
  double* sY = smem;
  double* sW = smem + kStepBuf;
  double* sT = smem + 2 * kStepBuf;
  double* sDc = smem + 3 * kStepBuf;
  const int half = l * (l + 1) / 2;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid & (kWave - 1);
  // Dc into sDc, Dgc into sT, both zero-padded
  for (int e = tid; e < NP * NP; e += kStepThreads) {
    const int i = e / NP, j = e % NP, q = tri(i, j);
    double dc = 0.0, dgc = 0.0;
    if (i < l && j < l) sum_partials2(P, nblk, 2 * half, q, half + q, dc, dgc);
    sDc[i * LD + j] = invN * dc;
    sT[i * LD + j] = 0.5 * invN * dgc;
  }
  __syncthreads();
  // Y = I - 4Z with Z = Dgc - Dc Dc'
  for (int tile = wave; tile < NT1 * NT1; tile += kStepWaves) {
    const int i0 = (tile / NT1) * 16, j0 = (tile % NT1) * 16;
    const d4 acc = lds_mfma_tile<false, true>(NP, LD, sDc, sDc, i0, j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + (lane >> 4) + 4 * r, j = j0 + (lane & 15);
      sY[i * LD + j] = ((i == j) ? 1.0 : 0.0) - 4.0 * (sT[i * LD + j] - acc[r]);
    }
  }
  __syncthreads();
  int ok = lds_ns_sqrt<kStepWaves>(NP, LD, sY, sW, sT, red, 60);
  if (ok > 0) {
    for (int e = tid; e < NP * NP; e += kStepThreads) {
      const int i = e / NP, j = e % NP;
      sY[i * LD + j] = 0.5 * (((i == j) ? 1.0 : 0.0) + sY[i * LD + j]);
    }
    __syncthreads();
    ok = lds_ns_sqrt<kStepWaves>(NP, LD, sY, sW, sT, red, 60);
  }
  if (ok <= 0) {  // rare: eigen-decomposition instead
    __syncthreads();
    return kn_step_eigen<NP>(l, invN, P, nblk, smem);
  }
  // C = sY, Cinv = sW; F = C - Dc Cinv; ||C - I||_F (the padding of C is the identity)
  double rs = 0.0;
  for (int tile = wave; tile < NT1 * NT1; tile += kStepWaves) {
    const int i0 = (tile / NT1) * 16, j0 = (tile % NT1) * 16;
    const d4 acc = lds_mfma_tile<false, false>(NP, LD, sDc, sW, i0, j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + (lane >> 4) + 4 * r, j = j0 + (lane & 15);
      const double c = sY[i * LD + j];
      sT[i * LD + j] = i < l && j < l ? c - acc[r] : 0.0;
      const double d = c - ((i == j) ? 1.0 : 0.0);
      rs += d * d;
    }
  }
  rs = wave_sum(rs);
  __syncthreads();  // red is reused
  if (lane == 0) red[wave] = rs;
  __syncthreads();
  double tot = 0.0;
  for (int w = 0; w < kStepWaves; ++w) tot += red[w];
  return sqrt(tot);
}

// Returns false (uniformly, with nothing written) when x is too large for the series.  Waves own
// lower-triangle tiles of the results: all matrices are symmetric polynomials of Z (and Dc), so
// only those tiles are computed, six MFMA chains of NP / 4 where the square-root iterations take
// eighteen; every barrier is one of about 5 + 2b.
template <int NP>
__device__ bool kn_step_series(int l, double invN, const double* __restrict__ P, int64_t nblk,
                               double* smem, double* red, double* res) {
  constexpr int LD = series_ld<NP>(), NT1 = NP / 16, NTL = NT1 * (NT1 + 1) / 2;
  constexpr int Q1 = (NTL + kStepWaves - 1) / kStepWaves;      // tiles per wave
  constexpr int Q2 = (2 * NTL + kStepWaves - 1) / kStepWaves;  // tiles of C and Cinv per wave
  double* bX = smem;                  // x, then the polynomial of C
  double* bX2 = smem + kStepBuf;      // x^2, then the polynomial of Cinv
  double* bX4 = smem + 2 * kStepBuf;  // Dgc, then x^4
  double* bDc = smem + 3 * kStepBuf;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid & (kWave - 1);
  const int half = l * (l + 1) / 2;
  const d4 zero = {0.0, 0.0, 0.0, 0.0};
  // Dc into bDc, Dgc into bX4: job q < NTL is the tile q of Dc, the rest those of Dgc; the loads of
  // all of a wave's jobs and of four partials are in flight together
  {
    d4 sum[Q2];
    int off[Q2][4];
    bool in[Q2][4];
#pragma unroll
    for (int q = 0; q < Q2; ++q) {
      const int job = wave + q * kStepWaves;
      int i0, j0;
      lower_tile(job < NTL ? job : job - NTL, i0, j0);
      sum[q] = zero;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + (lane >> 4) + 4 * r, j = j0 + (lane & 15);
        in[q][r] = job < 2 * NTL && i < l && j < l;
        off[q][r] = in[q][r] ? (job < NTL ? 0 : half) + tri(i, j) : 0;
      }
    }
    constexpr int UB = Q2 == 1 ? 16 : Q2 == 2 ? 8 : 4;
    for (int64_t b = 0; b < nblk; b += UB) {
      double v[UB][Q2][4];
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        const double* Pb = P + (b + u < nblk ? b + u : b) * 2 * half;
#pragma unroll
        for (int q = 0; q < Q2; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) v[u][q][r] = Pb[off[q][r]];
      }
#pragma unroll
      for (int u = 0; u < UB; ++u)
        if (b + u < nblk) {
#pragma unroll
          for (int q = 0; q < Q2; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[q][r] += v[u][q][r];
        }
    }
#pragma unroll
    for (int q = 0; q < Q2; ++q) {
      const int job = wave + q * kStepWaves;
      if (job >= 2 * NTL) continue;
      int i0, j0;
      lower_tile(job < NTL ? job : job - NTL, i0, j0);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sum[q][r] = in[q][r] ? (job < NTL ? invN : 0.5 * invN) * sum[q][r] : 0.0;
      put_sym<NP>(job < NTL ? bDc : bX4, i0, j0, sum[q]);
    }
  }
  __syncthreads();
  // x = 4 (Dgc - Dc^2) and rho^2 = ||x||_F^2
  double ss = 0.0;
#pragma unroll
  for (int q = 0; q < Q1; ++q) {
    const int tile = wave + q * kStepWaves;
    if (tile >= NTL) continue;
    int i0, j0;
    lower_tile(tile, i0, j0);
    const d4 d = sym_tile<NP>(bDc, bDc, i0, j0, zero);
    d4 x;
    double s4 = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      x[r] = 4.0 * (bX4[(i0 + (lane >> 4) + 4 * r) * LD + j0 + (lane & 15)] - d[r]);
      s4 += x[r] * x[r];
    }
    ss += i0 != j0 ? 2.0 * s4 : s4;
    put_sym<NP>(bX, i0, j0, x);
  }
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  double rho2 = 0.0;
#pragma unroll
  for (int w = 0; w < kStepWaves; ++w) rho2 += red[w];
  const int nb = series_blocks(sqrt(rho2));
  if (nb == 0) {
    __syncthreads();  // the buffers are reused
    return false;
  }
#pragma unroll
  for (int q = 0; q < Q1; ++q) {  // x^2
    const int tile = wave + q * kStepWaves;
    if (tile >= NTL) continue;
    int i0, j0;
    lower_tile(tile, i0, j0);
    put_sym<NP>(bX2, i0, j0, sym_tile<NP>(bX, bX, i0, j0, zero));
  }
  __syncthreads();
  // x^4 into LDS; every owner of a tile of C (jobs 0 .. NTL - 1) or Cinv (the rest) keeps the
  // tile of x, x^2 and x^3
  d4 x1[Q2], x2[Q2], x3[Q2];
#pragma unroll
  for (int q = 0; q < Q2; ++q) {
    const int job = wave + q * kStepWaves;
    if (job >= 2 * NTL) continue;
    int i0, j0;
    lower_tile(job < NTL ? job : job - NTL, i0, j0);
    if (job < NTL) put_sym<NP>(bX4, i0, j0, sym_tile<NP>(bX2, bX2, i0, j0, zero));
    x3[q] = sym_tile<NP>(bX, bX2, i0, j0, zero);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + (lane >> 4) + 4 * r, j = j0 + (lane & 15);
      x1[q][r] = bX[i * LD + j];
      x2[q][r] = bX2[i * LD + j];
    }
  }
  __syncthreads();
  for (int b = nb - 1; b >= 0; --b) {  // P := P x^4 + a_4b I + ... + a_4b+3 x^3
    d4 acc[Q2];
#pragma unroll
    for (int q = 0; q < Q2; ++q) {
      const int job = wave + q * kStepWaves;
      if (job >= 2 * NTL) continue;
      const bool inv = job >= NTL;
      int i0, j0;
      lower_tile(inv ? job - NTL : job, i0, j0);
      const double* a = (inv ? kSeries.ci : kSeries.c) + 4 * b;
      const double a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + (lane >> 4) + 4 * r, j = j0 + (lane & 15);
        acc[q][r] = fma(a3, x3[q][r], fma(a2, x2[q][r], fma(a1, x1[q][r], i == j ? a0 : 0.0)));
      }
      if (b != nb - 1) acc[q] = sym_tile<NP>(inv ? bX2 : bX, bX4, i0, j0, acc[q]);
    }
    if (b != nb - 1) __syncthreads();
#pragma unroll
    for (int q = 0; q < Q2; ++q) {
      const int job = wave + q * kStepWaves;
      if (job >= 2 * NTL) continue;
      int i0, j0;
      lower_tile(job < NTL ? job : job - NTL, i0, j0);
      put_sym<NP>(job < NTL ? bX : bX2, i0, j0, acc[q]);
    }
    __syncthreads();
  }
  // F = C - Dc Cinv over x^4, ||C - I||_F
  double rs = 0.0;
  for (int tile = wave; tile < NT1 * NT1; tile += kStepWaves) {
    const int i0 = (tile / NT1) * 16, j0 = (tile % NT1) * 16;
    const d4 acc = sym_tile<NP>(bDc, bX2, i0, j0, zero);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + (lane >> 4) + 4 * r, j = j0 + (lane & 15);
      const double c = bX[i * LD + j];
      bX4[i * LD + j] = i < l && j < l ? c - acc[r] : 0.0;
      const double d = c - ((i == j) ? 1.0 : 0.0);
      rs += d * d;  // the padding of C is the identity
    }
  }
  rs = wave_sum(rs);
  if (lane == 0) red[wave] = rs;
  __syncthreads();
  double tot = 0.0;
  for (int w = 0; w < kStepWaves; ++w) tot += red[w];
  *res = sqrt(tot);
  return true;
}

// A KN iteration is two or three launches:
//   1. product: workgroup b owns rows [R b, R b + R) of the Nl x l matrices and forms Bg = Bs Bc / N
//      on them: its 8 waves take an eighth of K each, both operands straight from L2 into MFMA
//      registers, and sum their tiles through LDS in wave order; then its partial
//      [Bc'Bc, Bc'Bg + Bg'Bc] -> P[b] (f64 MFMA, lower triangles);
//   2. from nine workgroups on, kn_sum sums the partials element by element, in block order;
//   3. update: every workgroup runs the l x l step for itself and updates its rows of B and E.
// All sums are in a fixed order.  Repeating the step (6 us at l = 32, 17 us at l = 64) in every
// workgroup costs no time; doing it once, in the last workgroup of the product to finish, cost a
// ticket and a device-scope fence (4 us, twice with two levels of partials), one CU summing all
// partials (45 GB/s: 8 us at Nl = 2048 and l = 32, 25 us at Nl = 8192 and l = 64) and F and Cinv
// through memory.

// Rows per workgroup of the product: 16, so that the chip fills, while that makes at most 256
// workgroups, then 32 (twice the use of each line of Bc).
int step_rows(int64_t nl) { return nl <= 4096 ? 16 : 32; }

// Partials that the update sums itself.
constexpr int64_t kDirectPartials = 8;

// sums[e] = sum_b P[b][e]: 64 elements per workgroup, a quarter of the blocks per wave.
__device__ __forceinline__ void kn_sum_body(const double* __restrict__ P, int64_t nblk, int count,
                                            double* __restrict__ sums, int64_t blk) {
  __shared__ double part[kThreads];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int64_t e = blk * kWave + lane;
  const int64_t per = (nblk + 3) / 4, b0 = wave * per < nblk ? wave * per : nblk;
  const int64_t n = b0 + per < nblk ? per : nblk - b0;
  part[threadIdx.x] = e < count ? sum_partials(P + b0 * count, n, count, e) : 0.0;
  __syncthreads();
  if (wave == 0 && e < count)
    sums[e] = ((part[lane] + part[64 + lane]) + part[128 + lane]) + part[192 + lane];
}

// The tile of Bs Bc of one wave: RB rows from r0 by NP columns over k in [k0, k1), in stages of
// 16 k.  In a stage, lane group kq takes k = 4 kq .. 4 kq + 3 (the
// same in both operands), so that a lane's four entries of Bs are 32 contiguous bytes and a row's
// 16 are one line (VEC: 16-byte loads; Bs 16-byte aligned and nl even).  Columns past l and rows
// past nl repeat valid ones (their results are not used); k past k1 enters as zero.
template <int NP, int RB, bool VEC>
__device__ __forceinline__ void kn_product(const double* __restrict__ Bs,
                                           const double* __restrict__ B, int nl, int l, int r0,
                                           int k0, int k1, d4 (&acc)[RB / 16][NP / 16]) {
  constexpr int NT = NP / 16, RT = RB / 16;
  const int lane = threadIdx.x & (kWave - 1), c = lane & 15, kq = lane >> 4;
  const double* row[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = r0 + 16 * i + c;
    row[i] = Bs + static_cast<int64_t>(r < nl ? r : nl - 1) * nl;
  }
  int col[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) col[j] = j * 16 + c < l ? j * 16 + c : l - 1;
  // D stages of 16 k in registers: a stage's loads are issued D - 1 stages ahead (past the last
  // whole stage they repeat it), with no branch in the loop that would make the compiler wait
  constexpr int D = RT * NT <= 3 ? 4 : 3;
  double a[D][RT][4], b[D][4][NT];
  auto load = [&](int k, double (&x)[RT][4], double (&y)[4][NT]) {
    const int kk = k + 4 * kq;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      if constexpr (VEC) {
        const double2 p = *reinterpret_cast<const double2*>(row[i] + kk);
        const double2 q = *reinterpret_cast<const double2*>(row[i] + kk + 2);
        x[i][0] = p.x;
        x[i][1] = p.y;
        x[i][2] = q.x;
        x[i][3] = q.y;
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) x[i][u] = row[i][kk + u];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j) y[u][j] = B[static_cast<int64_t>(kk + u) * l + col[j]];
  };
  auto mul = [&](const double (&x)[RT][4], const double (&y)[4][NT]) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][u], y[u][j], acc[i][j], 0, 0, 0);
  };
  const int n = (k1 - k0) / 16;  // whole stages
  if (n > 0) {
#pragma unroll
    for (int s = 0; s < D - 1; ++s) load(k0 + 16 * (s < n ? s : n - 1), a[s], b[s]);
    int s0 = 0;
    for (; s0 + D <= n; s0 += D) {
#pragma unroll
      for (int s = 0; s < D; ++s) {
        const int ahead = s0 + s + D - 1;
        load(k0 + 16 * (ahead < n ? ahead : n - 1), a[(s + D - 1) % D], b[(s + D - 1) % D]);
        mul(a[s], b[s]);
      }
    }
#pragma unroll
    for (int s = 0; s < D - 1; ++s)
      if (s0 + s < n) mul(a[s], b[s]);
  }
  if (k0 + 16 * n < k1) {  // the last, partial stage
    const int kk = k0 + 16 * n + 4 * kq;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool in = kk + u < k1;
      const int kc = in ? kk + u : k0;
#pragma unroll
      for (int i = 0; i < RT; ++i) a[0][i][u] = in ? row[i][kc] : 0.0;
#pragma unroll
      for (int j = 0; j < NT; ++j) b[0][u][j] = B[static_cast<int64_t>(kc) * l + col[j]];
    }
    mul(a[0], b[0]);
  }
}

// A wave's product tile, written to LDS (leading dimension NP + 2).
template <int NP, int RB>
__device__ __forceinline__ void kn_product_tile(const double* __restrict__ Bs,
                                                const double* __restrict__ B, int nl, int l,
                                                bool vec, int r0, int k0, int k1, double* out) {
  constexpr int NT = NP / 16, RT = RB / 16;
  const int lane = threadIdx.x & (kWave - 1);
  d4 acc[RT][NT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  if (vec)
    kn_product<NP, RB, true>(Bs, B, nl, l, r0, k0, k1, acc);
  else
    kn_product<NP, RB, false>(Bs, B, nl, l, r0, k0, k1, acc);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        out[(16 * i + (lane >> 4) + 4 * r) * (NP + 2) + 16 * j + (lane & 15)] = acc[i][j][r];
}

// Workgroup `blk` of the product (kStepThreads threads), `rows` (16 or 32) rows each; l <= NP.
template <int NP>
__device__ __forceinline__ void kn_product_body(int t, const IntegratorState* st, int nl, int l,
                                                int rows, bool vec, double invN,
                                                const double* __restrict__ Bs,
                                                const double* __restrict__ B,
                                                double* __restrict__ Bg, double* __restrict__ P,
                                                int64_t blk) {
  if (skip(st, t)) return;
  constexpr int NT = NP / 16, LT = NP + 2;
  __shared__ double smem[kStepWaves * 32 * LT];
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int r0 = static_cast<int>(blk) * rows;
  const int per = (nl + 16 * kStepWaves - 1) / (16 * kStepWaves) * 16;  // k per wave
  const int k0 = wave * per < nl ? wave * per : nl, k1 = k0 + per < nl ? k0 + per : nl;
  const int tile = rows * LT;
  if (rows == 16)
    kn_product_tile<NP, 16>(Bs, B, nl, l, vec, r0, k0, k1, smem + wave * tile);
  else
    kn_product_tile<NP, 32>(Bs, B, nl, l, vec, r0, k0, k1, smem + wave * tile);
  __syncthreads();
  // the rows of Bg (summed in wave order, written out) and of B, then side by side in LDS
  constexpr int EP = 32 * NP / kStepThreads;  // elements per thread, at most
  double gv[EP], bv[EP];
#pragma unroll
  for (int u = 0; u < EP; ++u) {
    const int e = tid + u * kStepThreads, rr = e / NP, j = e % NP;
    const bool in = rr < rows && r0 + rr < nl && j < l;
    const int64_t o = static_cast<int64_t>(r0 + rr) * l + j;
    bv[u] = in ? B[o] : 0.0;
    double g = 0.0;
    if (rr < rows) {
#pragma unroll
      for (int w = 0; w < kStepWaves; ++w) g += smem[w * tile + rr * LT + j];
    }
    gv[u] = in ? invN * g : 0.0;
    if (in) Bg[o] = gv[u];
  }
  __syncthreads();
  constexpr int ldr = NP + 16;  // rows k, k + 1 half the banks apart
  double* sB = smem;
  double* sG = smem + 32 * ldr;
#pragma unroll
  for (int u = 0; u < EP; ++u) {
    const int e = tid + u * kStepThreads, rr = e / NP, j = e % NP;
    if (rr >= rows) break;
    sB[rr * ldr + j] = bv[u];
    sG[rr * ldr + j] = gv[u];
  }
  __syncthreads();
  const int half = l * (l + 1) / 2;
  double* Pb = P + blk * (2 * half);
  // lower-triangle tiles of B'B and B'G + G'B over the block's rows; the two-product jobs first
  constexpr int NTL = NT * (NT + 1) / 2;
  for (int job = wave; job < 2 * NTL; job += kStepWaves) {
    const bool cross = job < NTL;
    int i0, j0;
    lower_tile(cross ? job : job - NTL, i0, j0);
    const int ci = i0 + lane % 16, cj = j0 + lane % 16;
    d4 p = {0.0, 0.0, 0.0, 0.0};
    if (cross) {
#pragma unroll 4
      for (int q = 0; q < rows; q += 4) {
        const int k = (q + lane / 16) * ldr;
        p = __builtin_amdgcn_mfma_f64_16x16x4f64(sB[k + ci], sG[k + cj], p, 0, 0, 0);
        p = __builtin_amdgcn_mfma_f64_16x16x4f64(sG[k + ci], sB[k + cj], p, 0, 0, 0);
      }
    } else {
#pragma unroll 4
      for (int q = 0; q < rows; q += 4) {
        const int k = (q + lane / 16) * ldr;
        p = __builtin_amdgcn_mfma_f64_16x16x4f64(sB[k + ci], sB[k + cj], p, 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + lane / 16 + 4 * r;
      if (i < l && cj <= i) Pb[(cross ? half : 0) + i * (i + 1) / 2 + cj] = p[r];
    }
  }
}

// The l x l step and B+ = Bc F + Bg Cinv, E+ = Ec F + invN Bc Cinv on kUpdRows rows per workgroup
// (f64 MFMA tiles; the rows are loaded before the step and go to LDS after it); the last workgroup
// makes FF+ = FFc F.  Every element is one chain of MFMAs over k, whatever the grid.
constexpr int kUpdRows = 32;

// Workgroups of the update: the row blocks and one for FF+.
int64_t kn_update_blocks(int64_t nl) { return ceil_div(nl, kUpdRows) + 1; }

template <int NP>
__device__ __forceinline__ void kn_update_body(
    int t, IntegratorState* st, int64_t nl, int l, double invN, double tol,
    const double* __restrict__ P, int64_t nblk, const double* __restrict__ Bc,
    const double* __restrict__ Bg, double* __restrict__ Bp, const double* __restrict__ Ec,
    double* __restrict__ Ep, const double* __restrict__ FFc, double* __restrict__ FFp, int64_t blk,
    int64_t nblocks) {
  if (skip(st, t)) return;
  constexpr int LD = series_ld<NP>(), NT = NP / 16, ER = kUpdRows * NP / kStepThreads;
  static_assert(2 * kUpdRows * LD <= kStepBuf, "two row blocks fit a step buffer");
  __shared__ double smem[4 * kStepBuf];
  __shared__ double red[kStepWaves];
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, c = lane & 15,
            kq = lane >> 4;
  const bool ff = blk == nblocks - 1;
  const int64_t r0 = blk * kUpdRows;
  double v[3][ER];
#pragma unroll
  for (int u = 0; u < ER; ++u) {
    const int e = tid + u * kStepThreads, r = e / NP, j = e % NP;
    const bool in = !ff && r0 + r < nl && j < l;
    const int64_t o = in ? (r0 + r) * l + j : 0;
    v[0][u] = in ? Bc[o] : 0.0;
    v[1][u] = in ? Bg[o] : 0.0;
    v[2][u] = in ? Ec[o] : 0.0;
  }
  double res;
  if (!kn_step_series<NP>(l, invN, P, nblk, smem, red, &res))
    res = kn_step_ns<NP>(l, invN, P, nblk, smem, red);
  if (blk == 0 && tid == 0) {
    st->res = res;
    if (!isfinite(res)) st->nan_seen = 1;
    if (!(res >= tol)) st->converged_at = t;
  }
  double* sBc = smem;  // over C
  double* sBg = smem + kUpdRows * LD;
  const double* sC = smem + kStepBuf;
  const double* sF = smem + 2 * kStepBuf;
  double* sEc = smem + 3 * kStepBuf;  // over Dc
  __syncthreads();
  if (ff) {
    for (int e = tid; e < NP * NP; e += kStepThreads) {
      const int i = e / NP, j = e % NP;
      sEc[i * LD + j] = i < l && j < l ? FFc[i * l + j] : 0.0;
    }
  } else {
#pragma unroll
    for (int u = 0; u < ER; ++u) {
      const int e = tid + u * kStepThreads, r = e / NP, j = e % NP;
      sBc[r * LD + j] = v[0][u];
      sBg[r * LD + j] = v[1][u];
      sEc[r * LD + j] = v[2][u];
    }
  }
  __syncthreads();
  const int tiles = (ff ? NT : kUpdRows / 16) * NT;
  const int64_t rows = ff ? l : (nl - r0 < kUpdRows ? nl - r0 : kUpdRows);
  for (int job = wave; job < (ff ? tiles : 2 * tiles); job += kStepWaves) {
    const bool eside = job < tiles;
    const int tile = eside ? job : job - tiles, i0 = (tile / NT) * 16, j0 = (tile % NT) * 16;
    const double* x = (eside ? sEc : sBc) + (i0 + c) * LD;  // times F
    const double* y = (eside ? sBc : sBg) + (i0 + c) * LD;  // times Cinv
    d4 p = {0.0, 0.0, 0.0, 0.0}, q = p;
#pragma unroll
    for (int k0 = 0; k0 < NP; k0 += 4) {
      const int k = k0 + kq;
      p = __builtin_amdgcn_mfma_f64_16x16x4f64(x[k], sF[k * LD + j0 + c], p, 0, 0, 0);
      if (!ff) q = __builtin_amdgcn_mfma_f64_16x16x4f64(y[k], sC[k * LD + j0 + c], q, 0, 0, 0);
    }
    double* out = ff ? FFp : eside ? Ep : Bp;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + kq + 4 * r, j = j0 + c;
      if (i < rows && j < l)
        out[(ff ? i : r0 + i) * l + j] = eside ? p[r] + invN * q[r] : p[r] + q[r];
    }
  }
}

// ---------------------------------------------------------------------------------------------
// KN iterations of several solves per launch.  A group's launch runs workgroup x of member y
// (blockIdx.y) on that member's own buffers, shapes, state and iteration index, with the
// workgroup -> rows/tiles map the member would have alone, so a member's arithmetic (and result,
// bit for bit) does not depend on the group it runs in or on when it joined.  A solve alone is a
// group of one.  The member table is a
// by-value kernel argument (read through the kernel-argument segment), so a launch needs no
// device memory of its own and can be recorded into a HIP graph as is.

struct KnMember {
  const double* Bs;   // Nl x Nl
  double* B[2];
  double* Bg;
  double* E[2];
  double* FF[2];
  double* P;          // partials of the product's workgroups
  double* sums;       // their sums (P itself when the update sums them)
  IntegratorState* st;
  int64_t nl, nblk, nsum, upd_blocks;  // nsum: partials left at `sums`
  double invN, tol;
  int l, rows, vec;   // rows per product workgroup; Bs takes 16-byte loads
  int t;              // the member's iteration index in this launch
};

struct KnGroup {
  int count;
  KnMember m[kMaxKnGroup];
};
static_assert(sizeof(KnGroup) <= 4096, "the member table fits the kernel arguments");

// The product and the update are launched once per class of l present (NP = l rounded up to 32, 48
// or 64).
template <int NP>
__global__ __launch_bounds__(kStepThreads) void kn_product_group_kernel(KnGroup g) {
  const KnMember& m = g.m[blockIdx.y];
  if (blockIdx.x >= m.nblk) return;
  kn_product_body<NP>(m.t, m.st, static_cast<int>(m.nl), m.l, m.rows, m.vec != 0, m.invN, m.Bs,
                      m.B[m.t & 1], m.Bg, m.P, blockIdx.x);
}

__global__ __launch_bounds__(kThreads) void kn_sum_group_kernel(KnGroup g) {
  const KnMember& m = g.m[blockIdx.y];
  const int count = m.l * (m.l + 1);
  if (m.nsum == m.nblk || static_cast<int64_t>(blockIdx.x) * kWave >= count || skip(m.st, m.t))
    return;
  kn_sum_body(m.P, m.nblk, count, m.sums, blockIdx.x);
}

template <int NP>
__global__ __launch_bounds__(kStepThreads) void kn_update_group_kernel(KnGroup g) {
  const KnMember& m = g.m[blockIdx.y];
  const int t = m.t;
  if (blockIdx.x >= m.upd_blocks) return;
  const int c = t & 1, p = c ^ 1;
  kn_update_body<NP>(t, m.st, m.nl, m.l, m.invN, m.tol, m.sums, m.nsum, m.B[c], m.Bg, m.B[p],
                     m.E[c], m.E[p], m.FF[c], m.FF[p], blockIdx.x, m.upd_blocks);
}

// out[2i] = converged_at, out[2i + 1] = nan_seen of member i (one read-back for the group).
__global__ void kn_flags_kernel(KnGroup g, int* out) {
  const int i = threadIdx.x;
  if (i >= g.count) return;
  out[2 * i] = g.m[i].st->converged_at;
  out[2 * i + 1] = g.m[i].st->nan_seen;
}

// ---------------------------------------------------------------------------------------------
// Wen-Yin (row_block_gramian_wen_yin_integrator.hpp:162-317).  The line search needs
// ||Bc Fc + Bg Fgc||_F^2 per trial step; with Dc = Bc'Bc/N, Dgc = Bc'Bg/N and Hgg = Bg'Bg/N it is
// N * (tr(Fc'Dc Fc) + 2 tr(Fc'Dgc Fgc) + tr(Fgc'Hgg Fgc)), so every trial is l x l work.

struct WyConst {
  static constexpr double tau0 = 1.0, taumax = 1e14, taumin = 1e-14, beta = 0.5, sigma = 1e-4,
                          eta = 0.85;
  static constexpr int taumaxiter = 20;
};

// The l x l Wen-Yin kernels run on one workgroup of 16 waves.  An l x l matrix (l <= 64, padded
// with zeros to np = pad16(l)) is cut into (np/16)^2 tiles of 16 x 16: wave w owns tile
// (w / nt1, w % nt1), nt1 = np/16, and lane ln its entries (i0 + ln/16 + 4r, j0 + ln%16),
// r = 0..3 -- the layout of a v_mfma_f64_16x16x4f64 result, so a product lands in the registers
// of the entries it defines.  Four np x (np + 1) LDS buffers.
constexpr int kWyWaves = 16;
constexpr int kWyThreads = kWyWaves * kWave;

size_t wy_lds_bytes(int l) {
  const size_t np = pad16(l);
  return 4 * np * (np + 1) * sizeof(double) + 2 * kMaxL * sizeof(int) + kWyWaves * sizeof(double);
}

struct WyTile {
  int i0, j0, oj, ib;  // tile origin, owned column, first owned row
  bool act;            // the wave owns a tile
  __device__ WyTile(int np) {
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, nt1 = np / 16;
    act = wave < nt1 * nt1;
    i0 = act ? (wave / nt1) * 16 : 0;
    j0 = act ? (wave % nt1) * 16 : 0;
    oj = j0 + (lane & 15);
    ib = i0 + (lane >> 4);
  }
  __device__ int row(int r) const { return ib + 4 * r; }
};

// Gauss-Jordan inverse with partial pivoting of the l x l matrix in X (LDS, leading dimension
// ld): the inverse LAPACK getrf+getri computes (getrfi.hpp:117-124).  Rows are never swapped:
// step k eliminates column k with the unused row p_k of largest |x_ik| (first on ties) and keeps
// the new column of the inverse in place of column k, so on return M[p_k][q] with p_q = j holds
// inv[k][j] (piv[k] = p_k) -- the same operations as with explicit row and column interchanges.
// Each step reads one buffer and writes the other, so it needs one barrier; wave 0 also forms
// the next pivot column and picks the next pivot.  Every thread must call this; returns the
// buffer that holds M.
__device__ double* wy_gj_inverse(int l, int ld, double* X, double* Y, int* piv, const WyTile& w) {
  const int lane = threadIdx.x % kWave;
  const bool wave0 = threadIdx.x < kWave;
  bool used = false;  // wave 0: row `lane` was a pivot
  // pick the pivot of column k among the unused rows; y = |column k| of this lane's row
  auto choose = [&](double y, int k) {
    const bool cand = lane < l && !used;
    double key = cand ? fabs(y) : -1.0;
    if (cand && key != key) key = -0.5;  // NaN only when no finite candidate is left
    int idx = cand ? lane : kWave;
    for (int off = 32; off > 0; off >>= 1) {
      const double ok = __shfl_xor(key, off, kWave);
      const int oi = __shfl_xor(idx, off, kWave);
      if (ok > key || (ok == key && oi < idx)) {
        key = ok;
        idx = oi;
      }
    }
    if (lane == idx) used = true;
    if (lane == 0) piv[k] = idx;
  };
  if (wave0) choose(lane < l ? X[lane * ld] : 0.0, 0);
  __syncthreads();
  for (int k = 0; k < l; ++k) {
    const int p = piv[k];
    const double pv = 1.0 / X[p * ld + k];
    if (w.act && w.oj < l) {
      const int j = w.oj;
      const double rk = (j == k) ? pv : X[p * ld + j] * pv;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = w.row(r);
        if (i >= l) continue;
        if (i == p) {
          Y[i * ld + j] = rk;
        } else {
          const double f = X[i * ld + k];
          Y[i * ld + j] = (j == k) ? -f * rk : X[i * ld + j] - f * rk;
        }
      }
    }
    if (wave0 && k + 1 < l) {
      double y = 0.0;
      if (lane < l) {
        const double rk1 = X[p * ld + k + 1] * pv;
        y = (lane == p) ? rk1 : X[lane * ld + k + 1] - X[lane * ld + k] * rk1;
      }
      choose(y, k + 1);
    }
    __syncthreads();
    double* z = X;
    X = Y;
    Y = z;
  }
  return X;
}

// Line search + phi/zeta update (row_block_gramian_wen_yin_integrator.hpp:181-222).  D3 = [Dc;
// Dgc; Hgg] of parity c.  Writes Fc, Fgc.
//
// The reference inverts C = [[Dc/2 - I/tau, I/2], [-Dgc/2, -Dc/2 - I/tau]] (2l x 2l) for every
// trial tau and takes Fgc = X12 Dc - X11, Fc = X22 Dc - X21 + I from X = C^{-1}, i.e.
// [Fgc; Fc - I] = C^{-1} [-I; Dc].  Eliminating the second block row of that solve gives
//   Fgc = (4/tau) (K + (4/tau^2) I)^{-1},  Fc = -I - (Dc - s I) Fgc,  K = Dgc - Dc^2, s = 2/tau,
// one l x l inverse per trial.  Its test value (1/2N) ||Bc Fc + Bg Fgc||_F^2 with Dc = Bc'Bc/N,
// Dgc = Bc'Bg/N, Hgg = Bg'Bg/N is, with F = Fgc,
//   phit = 1/2 [tr(Dc) - 2 tr((K + s Dc) F) + tr(F' X(s) F)],  X(s) = X0 + s X1 + s^2 Dc,
//   X0 = Dc^3 - Dc Dgc - (Dc Dgc)' + Hgg,  X1 = Dgc + Dgc' - 2 Dc^2,
// so a trial costs one inverse and one product.  K, X0 and X1 stay in registers (owned entries).
__global__ __launch_bounds__(kWyThreads) void wy_search_kernel(int t, IntegratorState* st, int l,
                                                              const double* __restrict__ D3,
                                                              double* __restrict__ Fc,
                                                              double* __restrict__ Fgc) {
  if (skip(st, t)) return;
  extern __shared__ double dyn[];
  __shared__ double phit_s, trdc_s;
  __shared__ int accept_s;
  const int np = pad16(l), ld = np + 1, nb = np * ld;
  double* B0 = dyn;  // Dc
  double* B1 = B0 + nb;
  double* B2 = B1 + nb;
  double* B3 = B2 + nb;
  int* piv = reinterpret_cast<int*>(B3 + nb);
  int* pinv = piv + kMaxL;
  double* red = reinterpret_cast<double*>(pinv + kMaxL);
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const WyTile w(np);
  const int oj = w.oj;
  const double* Dc = D3;
  const double* Dgc = D3 + l * l;
  const double* Hgg = D3 + 2 * l * l;
  for (int e = tid; e < np * np; e += kWyThreads) {
    const int i = e / np, j = e % np;
    const bool in = i < l && j < l;
    B0[i * ld + j] = in ? Dc[i * l + j] : 0.0;
    B1[i * ld + j] = in ? Dgc[i * l + j] : 0.0;
  }
  __syncthreads();
  if (w.act) {  // Dc^2 into B2
    const d4 a = lds_mfma_tile<false, false>(np, ld, B0, B0, w.i0, w.j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) B2[w.row(r) * ld + oj] = a[r];
  }
  __syncthreads();
  double K[4] = {0, 0, 0, 0}, X0[4] = {0, 0, 0, 0}, X1[4] = {0, 0, 0, 0};
  if (w.act) {
    const d4 c3 = lds_mfma_tile<false, false>(np, ld, B0, B2, w.i0, w.j0);  // Dc^3
    const d4 cg = lds_mfma_tile<false, false>(np, ld, B0, B1, w.i0, w.j0);  // Dc Dgc
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = w.row(r);
      const double g = B1[i * ld + oj], d2 = B2[i * ld + oj];
      K[r] = g - d2;
      X1[r] = g + B1[oj * ld + i] - 2.0 * d2;
      X0[r] = c3[r];
      B3[i * ld + oj] = cg[r];
    }
  }
  if (wave == 0) {
    const double d = wave_sum(lane < l ? B0[lane * ld + lane] : 0.0);
    if (lane == 0) trdc_s = d;
  }
  __syncthreads();
  if (w.act) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = w.row(r);
      const double h = (i < l && oj < l) ? Hgg[i * l + oj] : 0.0;
      X0[r] = X0[r] - B3[i * ld + oj] - B3[oj * ld + i] + h;
    }
  }
  __syncthreads();  // B1..B3 are free from here
  const double phi = st->phi, mu = st->mu, trdc = trdc_s;
  double tau = st->taug, phit = phi, s = 2.0 / tau;
  double* Fb = B2;
  for (int ti = 0; ti < WyConst::taumaxiter; ++ti, tau *= WyConst::beta) {
    const double c = 4.0 / (tau * tau);
    s = 2.0 / tau;
    if (w.act) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = w.row(r);
        B1[i * ld + oj] = K[r] + (i == oj ? c : 0.0);
      }
    }
    __syncthreads();
    const double* R = wy_gj_inverse(l, ld, B1, B2, piv, w);
    Fb = (R == B1) ? B2 : B1;
    if (tid < l) pinv[piv[tid]] = tid;
    __syncthreads();
    if (w.act) {  // F = (4/tau) a^{-1} (gathered from the pivoted form), Xs = X0 + s X1 + s^2 Dc
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = w.row(r);
        Fb[i * ld + oj] = (i < l && oj < l) ? (4.0 / tau) * R[piv[i] * ld + pinv[oj]] : 0.0;
        B3[i * ld + oj] = X0[r] + s * X1[r] + s * s * B0[i * ld + oj];
      }
    }
    __syncthreads();
    double part = 0.0;
    if (w.act) {
      const d4 xf = lds_mfma_tile<false, false>(np, ld, B3, Fb, w.i0, w.j0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = w.row(r);
        part += Fb[i * ld + oj] * xf[r] - 2.0 * (K[r] + s * B0[i * ld + oj]) * Fb[oj * ld + i];
      }
    }
    part = wave_sum(part);
    if (lane == 0) red[wave] = part;
    __syncthreads();
    if (tid == 0) {
      double sum = trdc;
      for (int q = 0; q < kWyWaves; ++q) sum += red[q];
      phit_s = 0.5 * sum;
      accept_s = (phit_s >= phi + tau * WyConst::sigma * mu) ? 1 : 0;
    }
    __syncthreads();
    phit = phit_s;
    if (accept_s) break;
  }
  if (w.act) {  // Fgc = F, Fc = s F - Dc F - I
    const d4 df = lds_mfma_tile<false, false>(np, ld, B0, Fb, w.i0, w.j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = w.row(r);
      if (i < l && oj < l) {
        const double f = Fb[i * ld + oj];
        Fgc[i * l + oj] = f;
        Fc[i * l + oj] = s * f - df[r] - (i == oj ? 1.0 : 0.0);
      }
    }
  }
  if (tid == 0) {
    const double zeta = st->zeta;
    st->phi = (WyConst::eta * zeta * phi + phit) / (WyConst::eta * zeta + 1.0);
    st->zeta = WyConst::eta * zeta + 1.0;
  }
}

// B+ = Bc Fc + Bg Fgc; U1 = Bc Fgc / N; BsU1 = Bg Fgc (= Bs U1); E+ = U1 + Ec Fc; FF+ = FFc Fc.
__global__ __launch_bounds__(kThreads) void wy_update_kernel(
    int t, const IntegratorState* st, int64_t nl, int l, double invN,
    const double* __restrict__ Bc, const double* __restrict__ Bg, double* __restrict__ Bp,
    double* __restrict__ U1, double* __restrict__ BsU1, const double* __restrict__ Ec,
    double* __restrict__ Ep, const double* __restrict__ FFc, double* __restrict__ FFp,
    const double* __restrict__ Fc, const double* __restrict__ Fgc) {
  if (skip(st, t)) return;
  // Workgroup b updates rows [kURows b, kURows b + kURows): their rows of Bc, Bg, Ec are staged
  // in LDS (coalesced), lane j of wave w computes column j of rows w, w + 4, ... (F and G are
  // read once per k for all of them); each sum runs over k in order.  The first
  // ceil(l^2 / kThreads) workgroups also form FF+ = FFc F, one entry per thread.
  __shared__ double sF[kMaxL * kMaxL];
  __shared__ double sG[kMaxL * kMaxL];
  __shared__ double sR[3][kURows][kMaxL];
  constexpr int RW = kURows / (kThreads / kWave);  // rows per wave
  const int tid = threadIdx.x;
  for (int e = tid; e < l * l; e += kThreads) {
    sF[e] = Fc[e];
    sG[e] = Fgc[e];
  }
  const int64_t r0 = blockIdx.x * static_cast<int64_t>(kURows);
  for (int e = tid; e < kURows * l; e += kThreads) {
    const int rr = e / l, j = e % l;
    const int64_t r = r0 + rr;
    const bool ok = r < nl;
    sR[0][rr][j] = ok ? Bc[r * l + j] : 0.0;
    sR[1][rr][j] = ok ? Bg[r * l + j] : 0.0;
    sR[2][rr][j] = ok ? Ec[r * l + j] : 0.0;
  }
  __syncthreads();
  const int j = tid % kWave, w = tid / kWave;
  if (j < l && r0 < nl) {
    double bcf[RW], bgg[RW], bcg[RW], ecf[RW];
#pragma unroll
    for (int u = 0; u < RW; ++u) bcf[u] = bgg[u] = bcg[u] = ecf[u] = 0.0;
    for (int q = 0; q < l; ++q) {
      const double f = sF[q * l + j], g = sG[q * l + j];
#pragma unroll
      for (int u = 0; u < RW; ++u) {
        const int rr = w + 4 * u;
        const double bc = sR[0][rr][q], bg = sR[1][rr][q], ec = sR[2][rr][q];
        bcf[u] += bc * f;
        bgg[u] += bg * g;
        bcg[u] += bc * g;
        ecf[u] += ec * f;
      }
    }
#pragma unroll
    for (int u = 0; u < RW; ++u) {
      const int64_t r = r0 + w + 4 * u;
      if (r < nl) {
        const int64_t e = r * l + j;
        Bp[e] = bcf[u] + bgg[u];
        U1[e] = invN * bcg[u];
        BsU1[e] = bgg[u];
        Ep[e] = invN * bcg[u] + ecf[u];
      }
    }
  }
  // FF+: this workgroup's entries [kThreads b, kThreads (b + 1)) lie in rows
  // [kThreads b / l, ...] of FFc: at most kThreads / l + 1 rows, staged like the others
  const int64_t fe0 = blockIdx.x * static_cast<int64_t>(kThreads);
  if (fe0 < static_cast<int64_t>(l) * l) {
    __syncthreads();  // sR is reused
    const int i0 = static_cast<int>(fe0 / l);
    const int nr = std::min(l - i0, kThreads / l + 1);
    double* sFF = &sR[0][0][0];
    for (int e = tid; e < nr * l; e += kThreads) sFF[e] = FFc[i0 * l + e];
    __syncthreads();
    const int64_t fe = fe0 + tid;
    if (fe < static_cast<int64_t>(l) * l) {
      const int i = static_cast<int>(fe / l), jj = static_cast<int>(fe % l);
      double acc = 0.0;
      for (int q = 0; q < l; ++q) acc += sFF[(i - i0) * l + q] * sF[q * l + jj];
      FFp[fe] = acc;
    }
  }
}

// mu = sum |diag(Dg+)| - ||D+||_F^2; stop when mu < tol^2 (row_block_gramian_wen_yin_integrator.hpp:247-255).
__global__ void wy_check_kernel(int t, IntegratorState* st, int l, double tol,
                                const double* __restrict__ D3p) {
  if (skip(st, t)) return;
  __shared__ double red[kThreads / kWave];
  const double* Dp = D3p;
  const double* Dgp = D3p + l * l;
  double part = 0.0;
  for (int e = threadIdx.x; e < l * l; e += blockDim.x) {
    const int i = e / l, j = e % l;
    part -= Dp[e] * Dp[e];
    if (i == j) part += fabs(Dgp[e]);
  }
  part = wave_sum(part);
  if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = part;
  __syncthreads();
  if (threadIdx.x == 0) {
    double mu = 0.0;
    for (int w = 0; w < (int)(blockDim.x / kWave); ++w) mu += red[w];
    st->mu = mu;
    st->res = mu;
    if (!isfinite(mu)) st->nan_seen = 1;
    if (mu < tol * tol) st->converged_at = t;
  }
}

// Nl-row pass for the step-size terms (row_block_gramian_wen_yin_integrator.hpp:260-312):
// U2 = (B+ - Bc)/N - U1 D+, BsU = Bs U1 (odd) or Bs U2 = (Bg+ - Bgc) - BsU1 D+ (even);
// per-block partials [Bc'U1, Bc'U2, Bc'Mc (l x l each), U1.BsU, U2.BsU], where
// Mc = E~c + [F~c; 0] are the coefficients of Qc = Qs Mc, so Bc'Mc = Qc'Qc.
__global__ __launch_bounds__(kThreads) void wy_terms_kernel(
    int t, const IntegratorState* st, int64_t nl, int l, double invN, int odd,
    const double* __restrict__ Bc, const double* __restrict__ Bp, const double* __restrict__ Bgc,
    const double* __restrict__ Bgp, const double* __restrict__ U1,
    const double* __restrict__ BsU1, const double* __restrict__ Dp,
    const double* __restrict__ Ec, const double* __restrict__ FFc, double* __restrict__ P) {
  if (skip(st, t) || st->converged_at == t) return;
  __shared__ double sD[kMaxL * kMaxL];
  __shared__ double sBc[kRows][kMaxL + 1];  // rows padded: the MFMA fragment reads below
  __shared__ double sU1[kRows][kMaxL + 1];  // take two k-rows per 32 lanes
  __shared__ double sU2[kRows][kMaxL + 1];
  __shared__ double sBsU[kRows][kMaxL];
  __shared__ double sM[kRows][kMaxL + 1];
  __shared__ double sBsU1[kRows][kMaxL];
  __shared__ double red[2][kThreads / kWave];
  for (int e = threadIdx.x; e < l * l; e += kThreads) sD[e] = Dp[e];
  const int64_t r0 = blockIdx.x * (int64_t)kRows;
  // the block's rows of U1 and BsU1 go to LDS first (coalesced): the products with D+ below
  // read them along the row
  for (int e = threadIdx.x; e < kRows * l; e += kThreads) {
    const int rr = e / l, j = e % l;
    const int64_t r = r0 + rr;
    sU1[rr][j] = (r < nl) ? U1[r * l + j] : 0.0;
    sBsU1[rr][j] = (r < nl) ? BsU1[r * l + j] : 0.0;
  }
  // columns l .. pad16(l) of the MFMA operands are zero (those tiles' outputs are not stored)
  for (int e = threadIdx.x; e < kRows * (kMaxL - l); e += kThreads) {
    const int rr = e / (kMaxL - l), j = l + e % (kMaxL - l);
    sBc[rr][j] = 0.0;
    sU1[rr][j] = 0.0;
    sU2[rr][j] = 0.0;
    sM[rr][j] = 0.0;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kRows * l; e += kThreads) {
    const int rr = e / l, j = e % l;
    const int64_t r = r0 + rr;
    double bc = 0, u2 = 0, bsu = 0, mc = 0;
    if (r < nl) {
      const int64_t o = r * l;
      bc = Bc[o + j];
      mc = Ec[o + j] + (r < l ? FFc[o + j] : 0.0);
      double u1d = 0.0, bsu1d = 0.0;
      for (int q = 0; q < l; ++q) {
        u1d += sU1[rr][q] * sD[q * l + j];
        bsu1d += sBsU1[rr][q] * sD[q * l + j];
      }
      u2 = invN * (Bp[o + j] - bc) - u1d;
      bsu = odd ? sBsU1[rr][j] : (Bgp[o + j] - Bgc[o + j]) - bsu1d;
    }
    sBc[rr][j] = bc;
    sU2[rr][j] = u2;
    sBsU[rr][j] = bsu;
    sM[rr][j] = mc;
  }
  __syncthreads();
  const int count = 3 * l * l + 2;
  double* Pb = P + blockIdx.x * (int64_t)count;
  {  // Bc'U1, Bc'U2, Bc'Mc over the block's rows on f64 MFMA tiles (16 x 16, k = row)
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int nt1 = pad16(l) / 16, tiles = nt1 * nt1;
    for (int tile = wave; tile < 3 * tiles; tile += kThreads / kWave) {
      const int part = tile / tiles, i0 = ((tile % tiles) / nt1) * 16, j0 = (tile % nt1) * 16;
      const double(*Y)[kMaxL + 1] = part == 0 ? sU1 : (part == 1 ? sU2 : sM);
      d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
      for (int k0 = 0; k0 < kRows; k0 += 4) {
        const int k = k0 + lane / 16;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sBc[k][i0 + lane % 16], Y[k][j0 + lane % 16],
                                                   acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + lane / 16 + 4 * r, j = j0 + lane % 16;
        if (i < l && j < l) Pb[part * l * l + i * l + j] = acc[r];
      }
    }
  }
  double d1 = 0.0, d2 = 0.0;
  for (int e = threadIdx.x; e < kRows * l; e += kThreads) {
    const int rr = e / l, j = e % l;
    d1 += sU1[rr][j] * sBsU[rr][j];
    d2 += sU2[rr][j] * sBsU[rr][j];
  }
  d1 = wave_sum(d1);
  d2 = wave_sum(d2);
  if (threadIdx.x % kWave == 0) {
    red[0][threadIdx.x / kWave] = d1;
    red[1][threadIdx.x / kWave] = d2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s1 = 0, s2 = 0;
    for (int w = 0; w < kThreads / kWave; ++w) {
      s1 += red[0][w];
      s2 += red[1][w];
    }
    Pb[3 * l * l] = s1;
    Pb[3 * l * l + 1] = s2;
  }
}

// t1, t2 and the Barzilai-Borwein step (row_block_gramian_wen_yin_integrator.hpp:260-316), with
// T = [Bc'U1; Bc'U2; Qc'Qc; U1.BsU; U2.BsU] (reduced, unscaled).  The quadratic terms in Phi use
// the actual Qc'Qc where the reference's Gramian form assumes the identity: ||dQ||^2 =
// ||Qc Phi1 + Qs U1||^2 then equals the row-block form's explicit sum of squares, and the step
// size no longer amplifies the drift of Qc'Qc from I (with the identity, a 1e-15 perturbation of
// the input moves the result by ~1e-5 at the CPU-runnable workload).
__global__ __launch_bounds__(kWyThreads) void wy_tau_kernel(int t, IntegratorState* st, int l,
                                                           int odd, const double* __restrict__ Dc,
                                                           const double* __restrict__ Dp,
                                                           const double* __restrict__ Fc,
                                                           const double* __restrict__ T) {
  if (skip(st, t) || st->converged_at == t) return;
  extern __shared__ double dyn[];
  __shared__ double red7[7][kWyWaves];
  const int np = pad16(l), ld = np + 1, nb = np * ld;
  double* sF = dyn;        // Fc
  double* sD = sF + nb;    // D+
  double* sQ = sD + nb;    // Qc'Qc
  double* sP2 = sQ + nb;   // Phi2 = Dc - Fc D+
  const double* BtU1 = T;
  const double* BtU2 = T + l * l;
  const double* QQ = T + 2 * l * l;
  const double u1bsu = T[3 * l * l], u2bsu = T[3 * l * l + 1];
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const WyTile w(np);
  const int oj = w.oj;
  for (int e = tid; e < np * np; e += kWyThreads) {
    const int i = e / np, j = e % np;
    const bool in = i < l && j < l;
    sF[i * ld + j] = in ? Fc[i * l + j] : 0.0;
    sD[i * ld + j] = in ? Dp[i * l + j] : 0.0;
    sQ[i * ld + j] = in ? QQ[i * l + j] : 0.0;
  }
  __syncthreads();
  if (w.act) {
    const d4 fd = lds_mfma_tile<false, false>(np, ld, sF, sD, w.i0, w.j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = w.row(r);
      sP2[i * ld + oj] = ((i < l && oj < l) ? Dc[i * l + oj] : 0.0) - fd[r];
    }
  }
  __syncthreads();
  // <X, QQ Y> = sum_ij X_ij (QQ Y)_ij with Phi1 = Fc - I, so QQ Phi1 = QQ Fc - QQ
  double v[7] = {0, 0, 0, 0, 0, 0, 0};  // p11, p1bu1, p12, p1bu2, p2bu1, p22, p2bu2
  if (w.act) {
    const d4 q1 = lds_mfma_tile<false, false>(np, ld, sQ, sF, w.i0, w.j0);
    const d4 q2 = lds_mfma_tile<false, false>(np, ld, sQ, sP2, w.i0, w.j0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = w.row(r);
      if (i < l && oj < l) {
        const double ph1 = sF[i * ld + oj] - (i == oj ? 1.0 : 0.0), ph2 = sP2[i * ld + oj];
        const double qp1 = q1[r] - sQ[i * ld + oj];
        const double bu1 = BtU1[i * l + oj], bu2 = BtU2[i * l + oj];
        v[0] += ph1 * qp1;
        v[1] += ph1 * bu1;
        v[2] += ph1 * q2[r];
        v[3] += ph1 * bu2;
        v[4] += ph2 * bu1;
        v[5] += ph2 * q2[r];
        v[6] += ph2 * bu2;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const double x = wave_sum(v[k]);
    if (lane == 0) red7[k][wave] = x;
  }
  __syncthreads();
  if (tid == 0) {
    double s[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int k = 0; k < 7; ++k)
      for (int q = 0; q < kWyWaves; ++q) s[k] += red7[k][q];
    double t1, t2;
    if (odd) {
      t1 = s[0] + 2.0 * s[1] + u1bsu;
      t2 = s[2] + s[3] + s[4] + u2bsu;
    } else {
      t1 = s[2] + s[3] + s[4] + u1bsu;
      t2 = s[5] + 2.0 * s[6] + u2bsu;
    }
    double tg = fabs(t1 / t2);
    if (tg < WyConst::taumin) tg = WyConst::taumin;
    if (tg > WyConst::taumax) tg = WyConst::taumax;
    st->taug = tg;
  }
}

// ---------------------------------------------------------------------------------------------
__global__ void init_state_kernel(IntegratorState* st) {
  st->converged_at = INT_MAX;
  st->nan_seen = 0;
  st->res = 0.0;
  st->taug = WyConst::tau0;
  st->zeta = 1.0;
  st->phi = 0.0;
  st->mu = 0.0;
}

// B0 = first l columns of Bs; E0 = 0; FF0 = I.
__global__ void init_coef_kernel(const double* __restrict__ Bs, int64_t nl, int l,
                                 double* __restrict__ B0, double* __restrict__ E0,
                                 double* __restrict__ FF0) {
  const int64_t total = nl * l;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e / l;
    const int j = e % l;
    B0[e] = Bs[r * nl + j];
    E0[e] = 0.0;
    if (e < (int64_t)l * l) FF0[e] = ((e / l) == (e % l)) ? 1.0 : 0.0;
  }
}

// WY initial scalars: phi = ||Bc||^2 / 2N = tr(Dc)/2, mu = sum|diag(Dgc)| - ||Dc||^2.
// One wave.
__global__ void wy_init_scalars_kernel(IntegratorState* st, int l, const double* __restrict__ D3) {
  const double* Dc = D3;
  const double* Dgc = D3 + l * l;
  const int lane = threadIdx.x;
  double tr = 0.0, dg = 0.0, sq = 0.0;
  for (int i = lane; i < l; i += kWave) {
    tr += Dc[i * l + i];
    dg += fabs(Dgc[i * l + i]);
  }
  for (int e = lane; e < l * l; e += kWave) sq += Dc[e] * Dc[e];
  tr = wave_sum(tr);
  dg = wave_sum(dg);
  sq = wave_sum(sq);
  if (lane == 0) {
    st->phi = 0.5 * tr;
    st->mu = dg - sq;
  }
}

// Final re-orthonormalization of the basis Qbar = Qs M: Gm = M' Bs M = N * sum_blk P[blk][1]
// (P from gram_partials_kernel over M and Bs M / N), W = Gm^{-1/2} by the Newton-Schulz square
// root; Qbar W is the orthonormal basis nearest to Qbar (Loewdin).  The iterations keep Qbar
// orthonormal only to the rounding they accumulate (as the reference's own updates do); this
// step removes it.  W = I when Gm is not positive definite.
// (16 waves: one 16 x 16 tile of each product per wave at l = 64.)
__global__ __launch_bounds__(kWyThreads) void polish_kernel(int l, double N,
                                                           const double* __restrict__ P,
                                                           int64_t nblk, double* __restrict__ Wout) {
  __shared__ double sY[kMaxL * (kMaxL + 1)];
  __shared__ double sW[kMaxL * (kMaxL + 1)];
  __shared__ double sT[kMaxL * (kMaxL + 1)];
  __shared__ double red[kWyWaves];
  const int np = pad16(l), ld = np + 1, ll = l * l;
  for (int e = threadIdx.x; e < np * np; e += kWyThreads) {
    const int i = e / np, j = e % np;
    sT[i * ld + j] = (i < l && j < l) ? N * sum_partials(P, nblk, 2 * ll, ll + i * l + j)
                                      : ((i == j) ? 1.0 : 0.0);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < np * np; e += kWyThreads) {
    const int i = e / np, j = e % np;
    sY[i * ld + j] = 0.5 * (sT[i * ld + j] + sT[j * ld + i]);
  }
  __syncthreads();
  const int ok = lds_ns_sqrt<kWyWaves>(np, ld, sY, sW, sT, red, 60);
  for (int e = threadIdx.x; e < ll; e += kWyThreads) {
    const int i = e / l, j = e % l;
    Wout[e] = ok > 0 ? sW[i * ld + j] : ((i == j) ? 1.0 : 0.0);
  }
}

// out = X W for X Nl x l and W l x l (row-major).
__global__ __launch_bounds__(kThreads) void right_mul_kernel(int64_t nl, int l,
                                                            const double* __restrict__ X,
                                                            const double* __restrict__ W,
                                                            double* __restrict__ out) {
  __shared__ double sW[kMaxL * kMaxL];
  for (int e = threadIdx.x; e < l * l; e += kThreads) sW[e] = W[e];
  __syncthreads();
  const int64_t total = nl * l;
  for (int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * kThreads) {
    const int64_t r = e / l;
    const int j = e % l;
    const double* x = X + r * l;
    double acc = 0.0;
    for (int q = 0; q < l; ++q) acc += x[q] * sW[q * l + j];
    out[e] = acc;
  }
}

// M = E + [FF; 0]  (Nl x l).
__global__ void coef_kernel(const double* __restrict__ E, const double* __restrict__ FF,
                            int64_t nl, int l, double* __restrict__ M) {
  const int64_t total = nl * l;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    M[e] = E[e] + (e < (int64_t)l * l ? FF[e] : 0.0);
  }
}

// Workgroups of wy_update_kernel: the row blocks, and at least those FF+ = FFc F needs.
unsigned wy_update_blocks(int64_t nl, int l) {
  const int64_t b = std::max(ceil_div(nl, kURows), ceil_div(static_cast<int64_t>(l) * l, kThreads));
  return static_cast<unsigned>(b);
}

unsigned grid_elems(int64_t total) {
  int64_t b = ceil_div(total, kThreads);
  if (b > 4096) b = 4096;
  if (b < 1) b = 1;
  return static_cast<unsigned>(b);
}

struct Layout {
  int64_t nl;
  int l;
  int64_t nblk_p;  // blocks of gram_partials_kernel
  int64_t nblk_t;  // blocks of wy_terms_kernel
  int64_t splits;  // split-K factor of the Bs products
  double* B[2];
  double* Bg[2];
  double* E[2];
  double* FF[2];
  double* D3[2];   // [Dc; Dgc; Hgg] per parity
  double* F;       // KN F / WY Fc
  double* C;       // KN Cinv / WY Fgc
  double* U1;
  double* BsU1;
  double* P;       // partial dot products
  double* Pbg;     // split-K partials of the Bs products
  double* T;       // reduced WY terms, 3 l^2 + 2
  int* flags;      // a KN group's read-back of [converged_at, nan_seen] per member
  IntegratorState* st;
  size_t bytes;
};

Layout layout(char* base, int64_t N, int l) {
  Layout L{};
  L.nl = N * l;
  L.l = l;
  L.nblk_p = ceil_div(L.nl, kPRows);
  L.nblk_t = ceil_div(L.nl, kRows);
  {  // about 256 workgroups (512 for large Nl, where each split stays long), >= 128 k per split
    const int64_t tiles = ceil_div(L.nl, 128);
    int64_t sp = ceil_div(L.nl > 2048 ? 512 : 256, tiles);
    const int64_t cap = ceil_div(L.nl, 128);
    L.splits = sp < cap ? sp : cap;
    if (L.splits < 1) L.splits = 1;
  }
  const size_t nll = static_cast<size_t>(L.nl) * l, ll = static_cast<size_t>(l) * l;
  size_t off = 0;
  auto take = [&](size_t elems) {
    double* p = reinterpret_cast<double*>(base ? base + off : nullptr);
    off += ((elems * sizeof(double) + 255) / 256) * 256;
    return p;
  };
  for (int i = 0; i < 2; ++i) {
    L.B[i] = take(nll);
    L.Bg[i] = take(nll);
    L.E[i] = take(nll);
    L.FF[i] = take(ll);
    L.D3[i] = take(3 * ll);
  }
  L.F = take(ll);
  L.C = take(ll);
  L.U1 = take(nll);
  L.BsU1 = take(nll);
  const size_t pp = static_cast<size_t>(L.nblk_p) * 3 * ll;
  const size_t pt = static_cast<size_t>(L.nblk_t) * (3 * ll + 2);
  // (a KN iteration's (ceil(nl / 16) + 1) l (l + 1) doubles of partials and their sums fit pt)
  L.P = take(pp > pt ? pp : pt);
  L.Pbg = take(static_cast<size_t>(L.splits + 1) * nll);
  L.T = take(3 * ll + 2);
  L.flags = reinterpret_cast<int*>(take(kMaxKnGroup));  // 2 kMaxKnGroup ints
  L.st = reinterpret_cast<IntegratorState*>(base ? base + off : nullptr);
  off += 256;
  L.bytes = off;
  return L;
}

}  // namespace

size_t integrator_workspace_bytes(int64_t N, int l) { return layout(nullptr, N, l).bytes; }

IterationGraphs::~IterationGraphs() {
  for (auto& e : execs) (void)hipGraphExecDestroy(e.second);
  if (cap) (void)hipStreamDestroy(cap);
}

namespace {

// Bout = Bs * Bin / N (Bout null: only the split-K partials into L.Pbg), gated on t, through the
// GEMM dispatch (the Wen-Yin iterations and the final polish).
void bs_product(const GramIntegrator& g, const Layout& L, const double* Bin, double* Bout, int t,
                hipStream_t st) {
  const int64_t nl = L.nl;
  GemmF64Args p;
  p.M = nl;
  p.N = g.l;
  p.K = nl;
  p.A = g.Bs;
  p.lda = nl;
  p.a_mcontig = false;
  p.B = Bin;
  p.ldb = g.l;
  p.C = Bout;
  p.ldc = g.l;
  p.alpha = 1.0 / static_cast<double>(g.N);
  p.shape = g.l <= 32 ? GemmShape::kTallN32 : GemmShape::kTallN64;
  p.splits = L.splits;
  p.kchunk = ceil_div(ceil_div(nl, L.splits), 16) * 16;
  p.partial = L.Pbg;
  p.gate = &L.st->converged_at;
  p.gate_t = t;
  if (g.l > 32 && nl % 2 == 0) {
    // 256 x 64 DMA tiles of Bs read as M-contiguous (Bs is stored exactly symmetric, so its
    // rows stand in for its columns): 157 us for the 8192 x 8192 Bs at l = 64, against 175 us
    // streamed and 196 us register-staged
    p.a_mcontig = true;
    p.b_ncontig = true;
    p.shape = GemmShape::kSquare;
  } else {
    // Bs streamed into LDS by DMA (tall_stream_kernel; the register-staged kernel where its
    // operand conditions fail)
    p.kernel = 1;
  }
  gemm_f64(p, st);
}

void check_integrator(const GramIntegrator& g, const Layout& L) {
  MCNLA_REQUIRE(g.l >= 1 && g.l <= kMaxL, MCNLA_ERR_INVALID, "integrator needs 1 <= l <= 64");
  MCNLA_REQUIRE(g.N >= 1, MCNLA_ERR_INVALID, "integrator needs N >= 1");
  MCNLA_REQUIRE(g.ws_bytes >= L.bytes, MCNLA_ERR_INVALID, "integrator workspace too small");
}

// State reset, B0 = Bs(:, 0:l), E0 = 0, FF0 = I.
void init_iteration(const GramIntegrator& g, const Layout& L, hipStream_t st) {
  hipLaunchKernelGGL(init_state_kernel, dim3(1), dim3(1), 0, st, L.st);
  MCNLA_LAUNCHED();
  hipLaunchKernelGGL(init_coef_kernel, dim3(grid_elems(L.nl * g.l)), dim3(kThreads), 0, st, g.Bs,
                     L.nl, g.l, L.B[0], L.E[0], L.FF[0]);
  MCNLA_LAUNCHED();
}

// The coefficients after `iters` iterations, re-orthonormalized: coef = M W with
// M = E + [FF; 0] and W = (M' Bs M)^{-1/2}.
void finish_iteration(const GramIntegrator& g, const Layout& L, int64_t iters, double* coef,
                      hipStream_t st) {
  const int64_t nl = L.nl;
  const int l = g.l;
  const int fin = static_cast<int>(iters & 1);
  hipLaunchKernelGGL(coef_kernel, dim3(grid_elems(nl * l)), dim3(kThreads), 0, st, L.E[fin],
                     L.FF[fin], nl, l, L.U1);
  MCNLA_LAUNCHED();
  bs_product(g, L, L.U1, L.BsU1, -1, st);
  hipLaunchKernelGGL(gram_partials_kernel, dim3(static_cast<unsigned>(L.nblk_p)), dim3(kThreads),
                     0, st, -1, L.st, nl, l, L.U1, L.BsU1, L.P, 2);
  MCNLA_LAUNCHED();
  hipLaunchKernelGGL(polish_kernel, dim3(1), dim3(kWyThreads), 0, st, l, static_cast<double>(g.N),
                     L.P, L.nblk_p, L.F);
  MCNLA_LAUNCHED();
  hipLaunchKernelGGL(right_mul_kernel, dim3(grid_elems(nl * l)), dim3(kThreads), 0, st, nl, l, L.U1,
                     L.F, coef);
  MCNLA_LAUNCHED();
}

KnMember kn_member(const GramIntegrator& g, const Layout& L) {
  KnMember m{};
  const int64_t nl = L.nl;
  m.Bs = g.Bs;
  m.B[0] = L.B[0];
  m.B[1] = L.B[1];
  m.Bg = L.Bg[0];
  m.E[0] = L.E[0];
  m.E[1] = L.E[1];
  m.FF[0] = L.FF[0];
  m.FF[1] = L.FF[1];
  m.P = L.P;
  m.st = L.st;
  m.nl = nl;
  m.l = g.l;
  m.rows = step_rows(nl);
  m.nblk = ceil_div(nl, m.rows);
  const bool direct = m.nblk <= kDirectPartials;
  m.nsum = direct ? m.nblk : 1;
  m.sums = direct ? L.P : L.P + m.nblk * g.l * (g.l + 1);
  m.vec = (reinterpret_cast<uintptr_t>(g.Bs) % 16 == 0 && nl % 2 == 0) ? 1 : 0;
  m.upd_blocks = kn_update_blocks(nl);
  m.invN = 1.0 / static_cast<double>(g.N);
  m.tol = g.tol;
  return m;
}

// One KN iteration of the members in `act` (member i at its iteration act.m[i].t): the products (a
// launch per class of l present), the sums of their partials, then the l x l steps and updates.
void launch_kn_iteration(const KnGroup& act, hipStream_t st) {
  KnGroup cls[3];
  int64_t bp[3] = {0, 0, 0}, bu[3] = {0, 0, 0}, bs = 0;
  for (auto& c : cls) c.count = 0;
  for (int i = 0; i < act.count; ++i) {
    const KnMember& m = act.m[i];
    const int c = m.l <= 32 ? 0 : m.l <= 48 ? 1 : 2;
    cls[c].m[cls[c].count++] = m;
    bp[c] = std::max(bp[c], m.nblk);
    bu[c] = std::max(bu[c], m.upd_blocks);
    if (m.nsum != m.nblk)
      bs = std::max<int64_t>(bs, ceil_div(static_cast<int64_t>(m.l) * (m.l + 1), kWave));
    MCNLA_REQUIRE(m.nl < (1LL << 31), MCNLA_ERR_INVALID, "integrator grid too large");
  }
  auto launch = [&](auto kernel, const KnGroup& g, int64_t blocks, int threads) {
    if (g.count == 0 || blocks == 0) return;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks), g.count), dim3(threads), 0, st,
                       g);
    MCNLA_LAUNCHED();
  };
  launch(kn_product_group_kernel<32>, cls[0], bp[0], kStepThreads);
  launch(kn_product_group_kernel<48>, cls[1], bp[1], kStepThreads);
  launch(kn_product_group_kernel<64>, cls[2], bp[2], kStepThreads);
  launch(kn_sum_group_kernel, act, bs, kThreads);
  launch(kn_update_group_kernel<32>, cls[0], bu[0], kStepThreads);
  launch(kn_update_group_kernel<48>, cls[1], bu[1], kStepThreads);
  launch(kn_update_group_kernel<64>, cls[2], bu[2], kStepThreads);
}

// The KN loop of a group.  `graphs` (a group of one only) records each chunk once and replays it.
void run_kn(const GramIntegrator* gs, double* const* coefs, int count, hipStream_t st,
            IterationGraphs* graphs, int64_t* iterations, bool* converged, bool* numeric_ok) {
  MCNLA_REQUIRE(count >= 1 && count <= kMaxKnGroup, MCNLA_ERR_INVALID,
                "a KN group holds 1 to 16 solves");
  MCNLA_REQUIRE(graphs == nullptr || count == 1, MCNLA_ERR_INVALID,
                "iteration graphs are recorded for a single solve only");
  std::vector<Layout> Ls(count);
  KnGroup all;
  all.count = count;
  for (int i = 0; i < count; ++i) {
    MCNLA_REQUIRE(!gs[i].wen_yin, MCNLA_ERR_INVALID, "a KN group holds KN integrations only");
    Ls[i] = layout(gs[i].ws, gs[i].N, gs[i].l);
    check_integrator(gs[i], Ls[i]);
    all.m[i] = kn_member(gs[i], Ls[i]);
  }
  for (int i = 0; i < count; ++i) init_iteration(gs[i], Ls[i], st);

  std::vector<int> conv_at(count, INT_MAX), nan_seen(count, 0), flags(2 * count);
  int64_t t = 0;
  int64_t chunk = 8;
  hipStream_t ls = st;  // where the iteration launches go: a capture stream while recording
  for (;;) {
    int64_t tmax = 0;  // the furthest iteration any unconverged member may still run
    for (int i = 0; i < count; ++i)
      if (conv_at[i] == INT_MAX) tmax = std::max(tmax, gs[i].maxiter);
    if (t >= tmax) break;
    const int64_t tend = (t + chunk < tmax) ? t + chunk : tmax;
    hipGraphExec_t exec = graphs ? graphs->find(t, tend) : nullptr;
    const bool recording = exec == nullptr && graphs != nullptr;
    if (recording) {
      if (!graphs->cap) MCNLA_HIP(hipStreamCreateWithFlags(&graphs->cap, hipStreamNonBlocking));
      ls = graphs->cap;
      MCNLA_HIP(hipStreamBeginCapture(ls, hipStreamCaptureModeThreadLocal));
    }
    const int64_t t0 = t;
    if (exec != nullptr) {
      t = tend;
    } else try {
      for (; t < tend; ++t) {
        KnGroup act;  // members not known to have converged and below their maxiter
        act.count = 0;
        for (int i = 0; i < count; ++i)
          if (conv_at[i] == INT_MAX && t < gs[i].maxiter) {
            act.m[act.count] = all.m[i];
            act.m[act.count++].t = static_cast<int>(t);
          }
        launch_kn_iteration(act, ls);
      }
    } catch (...) {
      if (recording) {  // leave the capture stream usable
        hipGraph_t partial = nullptr;
        (void)hipStreamEndCapture(ls, &partial);
        if (partial) (void)hipGraphDestroy(partial);
      }
      throw;
    }
    if (recording) {
      hipGraph_t graph = nullptr;
      MCNLA_HIP(hipStreamEndCapture(ls, &graph));
      ls = st;
      hipGraphExec_t made = nullptr;
      const hipError_t e = hipGraphInstantiate(&made, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      MCNLA_HIP(e);
      graphs->execs.push_back({{t0, tend}, made});
      exec = made;
    }
    if (exec != nullptr) MCNLA_HIP(hipGraphLaunch(exec, st));
    hipLaunchKernelGGL(kn_flags_kernel, dim3(1), dim3(kWave), 0, st, all, Ls[0].flags);
    MCNLA_LAUNCHED();
    MCNLA_HIP(hipMemcpyAsync(flags.data(), Ls[0].flags, 2 * count * sizeof(int),
                             hipMemcpyDeviceToHost, st));
    MCNLA_HIP(hipStreamSynchronize(st));
    bool running = false;
    for (int i = 0; i < count; ++i) {
      conv_at[i] = flags[2 * i];
      nan_seen[i] = flags[2 * i + 1];
      if (conv_at[i] == INT_MAX && t < gs[i].maxiter) running = true;
    }
    if (!running) break;
    if (chunk < 32) chunk *= 2;
  }
  for (int i = 0; i < count; ++i) {
    const int64_t iters =
        (conv_at[i] != INT_MAX) ? static_cast<int64_t>(conv_at[i]) + 1 : gs[i].maxiter;
    finish_iteration(gs[i], Ls[i], iters, coefs[i], st);
    if (iterations) iterations[i] = iters;
    if (converged) converged[i] = conv_at[i] != INT_MAX;
    if (numeric_ok) numeric_ok[i] = nan_seen[i] == 0;
  }
}

}  // namespace

void integrate_gram_group(const GramIntegrator* gs, double* const* coefs, int count,
                          hipStream_t st, int64_t* iterations, bool* converged, bool* numeric_ok) {
  run_kn(gs, coefs, count, st, nullptr, iterations, converged, numeric_ok);
}

struct KnBatch::Impl {
  struct Slot {
    bool used = false;
    GramIntegrator g;
    Layout L;
    KnMember m;
    int64_t t = 0;
    int conv_at = INT_MAX;
    int nan_seen = 0;
  };
  int* flags = nullptr;
  Slot slot[kMaxKnGroup];
  int host[2 * kMaxKnGroup];
  bool live(const Slot& x) const {
    return x.used && x.conv_at == INT_MAX && x.t < x.g.maxiter;
  }
};

KnBatch::KnBatch(int* flags) : impl_(new Impl) { impl_->flags = flags; }
KnBatch::~KnBatch() { delete impl_; }

int KnBatch::free_slots() const {
  int n = 0;
  for (const auto& x : impl_->slot) n += x.used ? 0 : 1;
  return n;
}

int KnBatch::add(const GramIntegrator& g, hipStream_t st) {
  MCNLA_REQUIRE(!g.wen_yin, MCNLA_ERR_INVALID, "a KN batch holds KN integrations only");
  for (int i = 0; i < kMaxKnGroup; ++i) {
    Impl::Slot& x = impl_->slot[i];
    if (x.used) continue;
    x.g = g;
    x.L = layout(g.ws, g.N, g.l);
    check_integrator(g, x.L);
    x.m = kn_member(g, x.L);
    x.t = 0;
    x.conv_at = INT_MAX;
    x.nan_seen = 0;
    init_iteration(g, x.L, st);
    x.used = true;
    return i;
  }
  throw Error{MCNLA_ERR_STATE, "KN batch is full"};
}

void KnBatch::advance(int iters, hipStream_t st) {
  for (int k = 0; k < iters; ++k) {
    KnGroup act;
    act.count = 0;
    for (auto& x : impl_->slot)
      if (impl_->live(x)) {
        act.m[act.count] = x.m;
        act.m[act.count++].t = static_cast<int>(x.t);
        ++x.t;
      }
    if (act.count == 0) break;
    launch_kn_iteration(act, st);
  }
  KnGroup used;
  used.count = 0;
  int who[kMaxKnGroup];
  for (int i = 0; i < kMaxKnGroup; ++i)
    if (impl_->slot[i].used) {
      who[used.count] = i;
      used.m[used.count++] = impl_->slot[i].m;
    }
  if (used.count == 0) return;
  hipLaunchKernelGGL(kn_flags_kernel, dim3(1), dim3(kWave), 0, st, used, impl_->flags);
  MCNLA_LAUNCHED();
  MCNLA_HIP(hipMemcpyAsync(impl_->host, impl_->flags, 2 * used.count * sizeof(int),
                           hipMemcpyDeviceToHost, st));
  MCNLA_HIP(hipStreamSynchronize(st));
  for (int j = 0; j < used.count; ++j) {
    Impl::Slot& x = impl_->slot[who[j]];
    x.conv_at = impl_->host[2 * j];
    x.nan_seen = impl_->host[2 * j + 1];
  }
}

bool KnBatch::running(int slot) const { return impl_->live(impl_->slot[slot]); }

int64_t KnBatch::iterations(int slot) const {
  const Impl::Slot& x = impl_->slot[slot];
  return x.conv_at != INT_MAX ? static_cast<int64_t>(x.conv_at) + 1 : x.t;
}

bool KnBatch::converged(int slot) const { return impl_->slot[slot].conv_at != INT_MAX; }

bool KnBatch::numeric_ok(int slot) const { return impl_->slot[slot].nan_seen == 0; }

void KnBatch::finish(int slot, double* coef, hipStream_t st) {
  Impl::Slot& x = impl_->slot[slot];
  MCNLA_REQUIRE(x.used && !impl_->live(x), MCNLA_ERR_STATE, "KN batch member still running");
  finish_iteration(x.g, x.L, iterations(slot), coef, st);
  x.used = false;
}

void KnBatch::drop(int slot) { impl_->slot[slot].used = false; }

int64_t integrate_gram(const GramIntegrator& g, double* coef, hipStream_t st, bool* converged,
                       bool* numeric_ok) {
  if (!g.wen_yin) {
    int64_t iters = 0;
    bool conv = false, ok = true;
    run_kn(&g, &coef, 1, st, g.graphs, &iters, &conv, &ok);
    if (converged) *converged = conv;
    if (numeric_ok) *numeric_ok = ok;
    return iters;
  }
  Layout L = layout(g.ws, g.N, g.l);
  check_integrator(g, L);
  const int l = g.l;
  const int64_t nl = L.nl;
  const double invN = 1.0 / static_cast<double>(g.N);
  const int ll = l * l;
  const unsigned gp = static_cast<unsigned>(L.nblk_p);
  hipStream_t ls = st;  // where the iteration launches go: a capture stream while recording

  init_iteration(g, L, st);
  const size_t wy_lds = wy_lds_bytes(l);
  for (const void* f : {reinterpret_cast<const void*>(wy_search_kernel),
                        reinterpret_cast<const void*>(wy_tau_kernel)})
    MCNLA_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(wy_lds)));
  // Bg0 = Bs B0 / N and [Dc; Dgc; Hgg] of parity 0.
  bs_product(g, L, L.B[0], L.Bg[0], -1, st);
  hipLaunchKernelGGL(gram_partials_kernel, dim3(gp), dim3(kThreads), 0, st, -1, L.st, nl, l,
                     L.B[0], L.Bg[0], L.P, 3);
  MCNLA_LAUNCHED();
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(ceil_div(3 * ll, kThreads)), dim3(kThreads), 0,
                     st, -1, L.st, L.P, L.nblk_p, 3 * ll, invN, L.D3[0]);
  MCNLA_LAUNCHED();
  hipLaunchKernelGGL(wy_init_scalars_kernel, dim3(1), dim3(64), 0, st, L.st, l, L.D3[0]);
  MCNLA_LAUNCHED();

  int64_t t = 0;
  int64_t chunk = 8;
  int host_conv = INT_MAX;
  int nan_seen = 0;
  while (t < g.maxiter) {
    const int64_t tend = (t + chunk < g.maxiter) ? t + chunk : g.maxiter;
    hipGraphExec_t exec = g.graphs ? g.graphs->find(t, tend) : nullptr;
    if (exec == nullptr && g.graphs) {  // record this chunk once
      if (!g.graphs->cap) MCNLA_HIP(hipStreamCreateWithFlags(&g.graphs->cap, hipStreamNonBlocking));
      ls = g.graphs->cap;
      MCNLA_HIP(hipStreamBeginCapture(ls, hipStreamCaptureModeThreadLocal));
    }
    const int64_t t0 = t;
    const bool recording = exec == nullptr && g.graphs != nullptr;
    if (exec != nullptr) {
      t = tend;
    } else try {
      for (; t < tend; ++t) {
        const int c = static_cast<int>(t & 1), p = c ^ 1;
        const int ti = static_cast<int>(t);
        const int odd = p;  // the reference toggles is_odd before using it: odd = !(t & 1)
        hipLaunchKernelGGL(wy_search_kernel, dim3(1), dim3(kWyThreads), wy_lds, ls, ti, L.st, l,
                           L.D3[c], L.F, L.C);
        MCNLA_LAUNCHED();
        hipLaunchKernelGGL(wy_update_kernel, dim3(wy_update_blocks(nl, l)), dim3(kThreads), 0, ls, ti,
                           L.st, nl, l, invN, L.B[c], L.Bg[c], L.B[p], L.U1, L.BsU1, L.E[c],
                           L.E[p], L.FF[c], L.FF[p], L.F, L.C);
        MCNLA_LAUNCHED();
        bs_product(g, L, L.B[p], L.Bg[p], ti, ls);
        hipLaunchKernelGGL(gram_partials_kernel, dim3(gp), dim3(kThreads), 0, ls, ti, L.st, nl, l,
                           L.B[p], L.Bg[p], L.P, 3);
        MCNLA_LAUNCHED();
        hipLaunchKernelGGL(reduce_partials_kernel, dim3(ceil_div(3 * ll, kThreads)), dim3(kThreads),
                           0, ls, ti, L.st, L.P, L.nblk_p, 3 * ll, invN, L.D3[p]);
        MCNLA_LAUNCHED();
        hipLaunchKernelGGL(wy_check_kernel, dim3(1), dim3(kThreads), 0, ls, ti, L.st, l, g.tol,
                           L.D3[p]);
        MCNLA_LAUNCHED();
        hipLaunchKernelGGL(wy_terms_kernel, dim3(static_cast<unsigned>(L.nblk_t)), dim3(kThreads), 0,
                           ls, ti, L.st, nl, l, invN, odd, L.B[c], L.B[p], L.Bg[c], L.Bg[p], L.U1,
                           L.BsU1, L.D3[p], L.E[c], L.FF[c], L.P);
        MCNLA_LAUNCHED();
        hipLaunchKernelGGL(reduce_partials_kernel, dim3(ceil_div(3 * ll + 2, kThreads)),
                           dim3(kThreads), 0, ls, ti, L.st, L.P, L.nblk_t, 3 * ll + 2, 1.0, L.T);
        MCNLA_LAUNCHED();
        hipLaunchKernelGGL(wy_tau_kernel, dim3(1), dim3(kWyThreads), wy_lds, ls, ti, L.st, l, odd,
                           L.D3[c], L.D3[p], L.F, L.T);
        MCNLA_LAUNCHED();
      }
    } catch (...) {
      if (recording) {  // leave the capture stream usable
        hipGraph_t partial = nullptr;
        (void)hipStreamEndCapture(ls, &partial);
        if (partial) (void)hipGraphDestroy(partial);
        ls = st;
      }
      throw;
    }
    if (recording) {
      hipGraph_t graph = nullptr;
      MCNLA_HIP(hipStreamEndCapture(ls, &graph));
      ls = st;
      hipGraphExec_t made = nullptr;
      const hipError_t e = hipGraphInstantiate(&made, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      MCNLA_HIP(e);
      g.graphs->execs.push_back({{t0, tend}, made});
      exec = made;
    }
    if (exec != nullptr) MCNLA_HIP(hipGraphLaunch(exec, st));
    int fl[2] = {INT_MAX, 0};
    MCNLA_HIP(hipMemcpyAsync(fl, &L.st->converged_at, sizeof(fl), hipMemcpyDeviceToHost, st));
    MCNLA_HIP(hipStreamSynchronize(st));
    host_conv = fl[0];
    nan_seen = fl[1];
    if (host_conv != INT_MAX) break;
    if (chunk < 32) chunk *= 2;
  }
  const int64_t iters = (host_conv != INT_MAX) ? static_cast<int64_t>(host_conv) + 1 : g.maxiter;
  finish_iteration(g, L, iters, coef, st);
  if (converged) *converged = (host_conv != INT_MAX);
  if (numeric_ok) *numeric_ok = (nan_seen == 0);
  return iters;
}

}  // namespace mcnla
