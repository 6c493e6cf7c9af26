// Block preconditioned CG for k right-hand sides that share one operator: CG.solve with an
// (ndof, k) right-hand side (pymoto/solvers/iterative.py:259-403, Ji & Li's breakdown-free block
// CG).  Per iteration, with P, Q, R, Z, W the k-column blocks:
//   Q = A P;  alpha = (P^T Q)^-1 P^T R;  X += P alpha;
//   R = B - A X every `restart` iterations (including the first), else R -= Q alpha;
//   stop when max_j ||r_j|| / ||b_j|| <= tol;
//   Z = M R (one V-cycle per column);  beta = -(P^T Q)^-1 Q^T Z;  P = orth(Z + P beta).
// orth() is the reference's modified Gram-Schmidt (iterative.py:259-292) on the vectors: column i of
// the result is v_i minus its projections on the kept columns before it, dropped when its squared norm
// falls below 1e-15 of ||v_i||^2 (normalised to unit length in the initial orth, as the reference
// does).  Dropped columns are kept as zero vectors with their rows and columns masked out of the
// k x k algebra, which is the same arithmetic as compacting them.
//
// Everything runs on the device, in as few passes over the blocks as the dependences allow: P^T Q and
// P^T R in one, X and R with the squared norms of R in one, W = Z + P beta with the first Gram-Schmidt
// products in one, then one pass per further column.  The partial sums of a pass are added, in a fixed
// order, by the kernel that needs them (every block of it), the small dense algebra by one block.  So an
// iteration is two fixed launch sequences (before and after the convergence test) that are captured once
// as HIP graphs and replayed; the host polls pinned memory for the stopping test, as the
// single-right-hand-side runtime does.
// Four columns of 1,635,075 entries: 0.21 ms per iteration outside the products and the preconditioner
// (products, algebra and Gram-Schmidt as a launch per dot product, update and row of a product: 0.52 ms).
#include <cmath>
#include <new>
#include <type_traits>

#include "mg_impl.h"

namespace pmt {

constexpr int kMaxRhs = 8;

template <typename T>
struct VecSetT {
  const T* v[kMaxRhs];
};
using VecSet = VecSetT<double>;
struct OutSet {
  double* v[kMaxRhs];
};

// small device state, in doubles
struct Small {
  enum {
    PQINV = 0,  // (P^T Q)^-1 on the active set
    ALPHA = PQINV + kMaxRhs * kMaxRhs,
    BETA = ALPHA + kMaxRhs * kMaxRhs,
    ACTIVE = BETA + kMaxRhs * kMaxRhs,
    BNORM = ACTIVE + kMaxRhs,
    TVAL = BNORM + kMaxRhs,
    MGS_B0 = TVAL + kMaxRhs,  // ||v_i||^2 before orthogonalisation
    TMAX = MGS_B0 + kMaxRhs,  // max of TVAL
    SEQ = TMAX + 1,           // number of the last convergence test published to the host
    SIZE = SEQ + 7
  };
};

// Blocks of the kernels that sum over the vectors: two per CU; 12 loads per thread keep enough in flight, and
// the kernels that add the partial sums read few of them.  Partial sum of entry e: partial[e * nb + block].
constexpr int kSumBlocks = 512;

struct BlockCG {
  long long n = 0;
  int kcap = 0;
  double* mem = nullptr;  // X, B, P, Q, R, Z, W blocks of kcap columns + a zero column
  double* X = nullptr;
  double* B = nullptr;
  double* P = nullptr;
  double* Q = nullptr;
  double* R = nullptr;
  double* Z = nullptr;
  double* zero = nullptr;
  double* sm = nullptr;       // Small::SIZE doubles
  double* partial = nullptr;  // kSumBlocks * 2 * kMaxRhs^2
  double* host = nullptr;     // pinned: [max relative residual, test number], then TVAL
  double seq = 0.0;           // convergence tests launched so far (the number the next wait polls for)
  // captured iterations: [0] operator + alpha + restart residual, [1] same with recurrence, [2] beta + orth
  hipGraphExec_t exec[3] = {nullptr, nullptr, nullptr};
  int graph_k = 0, graph_epoch = -1;
  // vectors of the V-cycle of kcap columns in the precision `vec_prec` (64 or 32), null if they did not fit
  void* vec = nullptr;
  int vec_prec = 0;
  float* z32 = nullptr;
  // captured work runs on a stream of the handle (the caller's may be the legacy default stream,
  // which cannot be captured), ordered after and before the caller's stream with two events
  hipStream_t cs = nullptr;
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
};

// ------------------------------------------------------------------------------------------------
// kernels
// ------------------------------------------------------------------------------------------------

// v[e] summed over the 64 lanes for N entries at once: each exchange halves the entries a lane still holds
// (N + 6 shuffles instead of 6 N); lane l ends with entry l / (64 / N)
template <int N>
__device__ __forceinline__ double wave_sums(double (&v)[N]) {
  const int lane = threadIdx.x & 63;
  int off = 32;
#pragma unroll
  for (int h = N / 2; h >= 1; h >>= 1) {
    const bool up = (lane & off) != 0;
#pragma unroll
    for (int e = 0; e < h; ++e) {
      const double send = up ? v[e] : v[e + h], keep = up ? v[e + h] : v[e];
      v[e] = keep + __shfl_xor(send, off, 64);
    }
    off >>= 1;
  }
  for (; off >= 1; off >>= 1) v[0] += __shfl_xor(v[0], off, 64);
  return v[0];
}

// the block's sums (256 threads) of N entries to partial[e * nb + block]
template <int N>
__device__ __forceinline__ void block_sums(double (&v)[N], double* __restrict__ partial) {
  __shared__ double red[4][N];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double t = wave_sums<N>(v);
  if (lane % (64 / N) == 0) red[wave][lane / (64 / N)] = t;
  __syncthreads();
  if (threadIdx.x < N)
    partial[(long long)threadIdx.x * gridDim.x + blockIdx.x] =
        ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
}

// S[e] = sum over the nb blocks of partial[e * nb + block], e < E, by a block of NT threads in a fixed order
template <int E, int NT>
__device__ __forceinline__ void sum_entries(const double* __restrict__ partial, int nb, double* S) {
  constexpr int G = NT / E < 64 ? NT / E : 64;  // lanes per entry
  const int e = threadIdx.x / G, g = threadIdx.x % G;
  if (e < E) {
    double acc = 0.0;
#pragma unroll 8
    for (int b = g; b < nb; b += G) acc += partial[(long long)e * nb + b];
#pragma unroll
    for (int off = G / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (g == 0) S[e] = acc;
  }
  __syncthreads();
}

// partial sums of A^T B1 (entry a * K + b) and, NB == 2, of A^T B2 (entry K * K + a * K + b)
template <int K, int NB, typename T>
__global__ void __launch_bounds__(256)
gram_kernel(long long n, VecSet A, VecSetT<T> B1, VecSetT<T> B2, double* __restrict__ partial) {
  double acc[NB * K * K];
#pragma unroll
  for (int e = 0; e < NB * K * K; ++e) acc[e] = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    double va[K], vb[NB][K];  // (T float: the preconditioner's result, widened)
#pragma unroll
    for (int a = 0; a < K; ++a) va[a] = A.v[a][i];
#pragma unroll
    for (int b = 0; b < K; ++b) vb[0][b] = B1.v[b][i];
    if (NB == 2)
#pragma unroll
      for (int b = 0; b < K; ++b) vb[NB - 1][b] = B2.v[b][i];
#pragma unroll
    for (int m = 0; m < NB; ++m)
#pragma unroll
      for (int a = 0; a < K; ++a)
#pragma unroll
        for (int b = 0; b < K; ++b) acc[(m * K + a) * K + b] = fma(va[a], vb[m][b], acc[(m * K + a) * K + b]);
  }
  block_sums<NB * K * K>(acc, partial);
}

// partial sums of r_j . r_j
template <int K>
__global__ void __launch_bounds__(256) norms_kernel(long long n, VecSet R, double* __restrict__ partial) {
  double acc[K];
#pragma unroll
  for (int j = 0; j < K; ++j) acc[j] = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const double v = R.v[j][i];
      acc[j] = fma(v, v, acc[j]);
    }
  block_sums<K>(acc, partial);
}

// X += P alpha and, RES, R -= Q alpha with the partial sums of r_j . r_j
template <int K, bool RES>
__global__ void __launch_bounds__(256)
update_kernel(long long n, int k, VecSet P, VecSet Q, const double* __restrict__ alpha, VecSet X, OutSet Xo, VecSet R,
              OutSet Ro, double* __restrict__ partial) {
  __shared__ double c[K * kMaxRhs];
  for (int t = threadIdx.x; t < K * kMaxRhs; t += 256) c[t] = alpha[t];
  __syncthreads();
  double acc[K];
#pragma unroll
  for (int j = 0; j < K; ++j) acc[j] = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    double p[K], q[K], x[K], r[K];
#pragma unroll
    for (int a = 0; a < K; ++a) {
      p[a] = P.v[a][i];
      x[a] = X.v[a][i];
      if (RES) q[a] = Q.v[a][i];
      if (RES) r[a] = R.v[a][i];
    }
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (j >= k) break;
#pragma unroll
      for (int a = 0; a < K; ++a) x[j] = fma(p[a], c[a * kMaxRhs + j], x[j]);
      Xo.v[j][i] = x[j];
      if (RES) {
#pragma unroll
        for (int a = 0; a < K; ++a) r[j] = fma(q[a], -c[a * kMaxRhs + j], r[j]);
        Ro.v[j][i] = r[j];
        acc[j] = fma(r[j], r[j], acc[j]);
      }
    }
  }
  if (RES) block_sums<K>(acc, partial);
}

// alpha = (P^T Q)^-1 P^T R from the partial sums of both products (entries 0.. and K * K..), one block.  The
// inverse of the active principal submatrix by Gauss-Jordan with row pivoting, a thread per entry of the
// K x 2K tableau; an inactive (dropped) column has zero products and stands as a unit row and column, which
// leaves the arithmetic of the others unchanged.  Its rows and columns of the inverse are zero.  The columns from
// k to K are never active: ACTIVE is written for the k columns of a solve only and may hold an earlier, wider one's.
template <int K>
__global__ void __launch_bounds__(1024) bcg_alpha_kernel(int k, const double* __restrict__ partial, int nb, double* sm) {
  __shared__ double S[2 * K * K];
  __shared__ double a[K][2 * K];
  __shared__ double inv[K][K];
  const int tid = threadIdx.x, r = tid / (2 * K), c = tid % (2 * K);
  const bool own = r < K;
  auto active = [&](int j) { return j < k && sm[Small::ACTIVE + j] != 0.0; };
  sum_entries<2 * K * K, 1024>(partial, nb, S);
  if (own) a[r][c] = c >= K ? (c - K == r ? 1.0 : 0.0) : active(r) && active(c) ? S[r * K + c] : r == c ? 1.0 : 0.0;
  __syncthreads();
  for (int d = 0; d < K; ++d) {
    double v = 0.0;
    if (own) {
      int piv = d;
      for (int t = d + 1; t < K; ++t)
        if (fabs(a[t][d]) > fabs(a[piv][d])) piv = t;
      const double top = a[piv][c] * (1.0 / a[piv][d]);  // row d after the swap and the scaling
      const int src = r == piv ? d : r;                  // where row r's entries are before the swap
      const double f = a[src][d];
      v = r == d ? top : f != 0.0 ? a[src][c] - f * top : a[src][c];
    }
    __syncthreads();
    if (own) a[r][c] = v;
    __syncthreads();
  }
  if (own && c < K) inv[r][c] = active(r) && active(c) ? a[r][K + c] : 0.0;
  __syncthreads();
  if (tid < kMaxRhs * kMaxRhs) {
    const int i = tid / kMaxRhs, j = tid % kMaxRhs;
    double s = 0.0;
    if (i < K && j < K)
      for (int m = 0; m < K; ++m) s += inv[i][m] * S[K * K + m * K + j];
    sm[Small::PQINV + tid] = i < K && j < K ? inv[i][j] : 0.0;
    sm[Small::ALPHA + tid] = s;
  }
}

// beta = -(P^T Q)^-1 Q^T Z from the partial sums of Q^T Z
template <int K>
__global__ void __launch_bounds__(1024) bcg_beta_kernel(const double* __restrict__ partial, int nb, double* sm) {
  __shared__ double S[K * K];
  sum_entries<K * K, 1024>(partial, nb, S);
  const int tid = threadIdx.x, i = tid / kMaxRhs, j = tid % kMaxRhs;
  if (tid >= kMaxRhs * kMaxRhs) return;
  double s = 0.0;
  if (i < K && j < K)
    for (int m = 0; m < K; ++m) s += sm[Small::PQINV + i * kMaxRhs + m] * S[m * K + j];
  sm[Small::BETA + tid] = -s;
}

// value and number to pinned host memory, in the order publish_wait relies on
__device__ inline void publish(double v, double seq, double* host) {
  volatile double* h = host;
  h[0] = v;
  __threadfence_system();
  h[1] = seq;
  __threadfence_system();
}

// per-column relative residuals from the partial sums of r_j . r_j (entries 0..); the first call (init) also
// sets ||b_j|| from those of b_j . b_j (entries K..).  The largest goes to the host with the test's number.
template <int K>
__global__ void __launch_bounds__(512)
bcg_check_kernel(int k, int init, const double* __restrict__ partial, int nb, double* sm, double* host) {
  __shared__ double S[2 * K];
  if (init)
    sum_entries<2 * K, 512>(partial, nb, S);
  else
    sum_entries<K, 512>(partial, nb, S);
  if (threadIdx.x != 0) return;
  double* bn = sm + Small::BNORM;
  // a non-finite column (NaN/inf in b, x0 or the iterates) makes the maximum NaN, which the host turns into
  // an error; a zero column counts as converged
  double mx = 0.0;
  for (int j = 0; j < k; ++j) {
    const double b = init ? sqrt(S[K + j]) : bn[j];
    if (init) bn[j] = b;
    const double t = b == 0.0 ? 0.0 : sqrt(S[j]) / b;
    sm[Small::TVAL + j] = t;
    mx = (t != t || mx != mx) ? t + mx : fmax(mx, t);
  }
  const double seq = sm[Small::SEQ] + 1.0;
  sm[Small::TMAX] = mx;
  sm[Small::SEQ] = seq;
  publish(mx, seq, host);
}

// Modified Gram-Schmidt on the vectors, as orth() does (iterative.py:259-292): column i starts as
// v_i and loses its projection on every kept column j < i in turn; it is dropped (zeroed, ACTIVE = 0)
// when its squared norm falls below 1e-15 of ||v_i||^2, and scaled to unit length when normalising.
// (Orthogonalising through the Gram matrix V^T V instead squares the condition number of V, which the
// block recurrence does not tolerate near convergence.)
// Pass J takes column J - 1, final but for its scale, from all columns after it and sums the products of
// column J with them for the next pass: the projections of a column come in the same order as column by
// column, in one pass over the columns left instead of one per pair.

// w_j = z_j (+ sum_a p_a beta[a][j]) to column j of P; sums w_j . w_j (entries 0..) and w_0 . w_j (entries K..)
template <int K, bool COMBINE, typename T>
__global__ void __launch_bounds__(256)
orth_first_kernel(long long n, int k, VecSet P, VecSetT<T> Z, const double* __restrict__ beta, OutSet out,
                  double* __restrict__ partial) {
  __shared__ double c[K * kMaxRhs];
  if (COMBINE)
    for (int t = threadIdx.x; t < K * kMaxRhs; t += 256) c[t] = beta[t];
  __syncthreads();
  double acc[2 * K];
#pragma unroll
  for (int j = 0; j < 2 * K; ++j) acc[j] = 0.0;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    double p[K], w[K];
#pragma unroll
    for (int a = 0; a < K; ++a) {
      if (COMBINE) p[a] = P.v[a][i];
      w[a] = Z.v[a][i];
    }
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (j >= k) break;
      if (COMBINE)
#pragma unroll
        for (int a = 0; a < K; ++a) w[j] = fma(p[a], c[a * kMaxRhs + j], w[j]);
      out.v[j][i] = w[j];
      acc[j] = fma(w[j], w[j], acc[j]);
      acc[K + j] = fma(w[0], w[j], acc[K + j]);
    }
  }
  block_sums<2 * K>(acc, partial);
}

// the scale of column j (0: dropped) and the projection coefficients coef[i] of the columns after it, from the
// sums t[i] = w_j . w_i; every block computes them, block 0 records the column's state
template <int K>
__device__ __forceinline__ void orth_column(const double* t, double b0, int j, int normalize, double* sm, double* coef,
                                            double* scale) {
  const int i = threadIdx.x;
  if (i < K) {
    const double b1 = t[j];
    const bool keep = b0 > 0.0 && b1 / b0 >= 1e-15;
    const double sc = keep ? (normalize ? 1.0 / sqrt(b1) : 1.0) : 0.0;
    coef[i] = keep ? (normalize ? sc * t[i] : t[i] / b1) : 0.0;
    if (i == 0) *scale = sc;
    if (i == 0 && blockIdx.x == 0) sm[Small::ACTIVE + j] = keep ? 1.0 : 0.0;
  }
  __syncthreads();
}

template <int K, int J>
__global__ void __launch_bounds__(256)
orth_pass_kernel(long long n, int k, int normalize, const double* __restrict__ pin, VecSet P, OutSet out, double* sm,
                 double* __restrict__ partial) {
  __shared__ double S[2 * K], coef[K], scale;
  if (J == 1)
    sum_entries<2 * K, 256>(pin, gridDim.x, S);
  else
    sum_entries<K, 256>(pin, gridDim.x, S);
  if (J == 1 && blockIdx.x == 0 && threadIdx.x < K) sm[Small::MGS_B0 + threadIdx.x] = S[threadIdx.x];
  orth_column<K>(J == 1 ? S + K : S, J == 1 ? S[0] : sm[Small::MGS_B0 + J - 1], J - 1, normalize, sm, coef, &scale);
  const double sc = scale;
  double acc[K];
#pragma unroll
  for (int i = 0; i < K; ++i) acc[i] = 0.0;
  for (long long r = (long long)blockIdx.x * 256 + threadIdx.x; r < n; r += (long long)gridDim.x * 256) {
    double w[K];
#pragma unroll
    for (int i = J - 1; i < K; ++i) w[i] = P.v[i][r];
    const double pj = sc * w[J - 1];
    if (sc != 1.0) out.v[J - 1][r] = pj;
#pragma unroll
    for (int i = J; i < K; ++i) {
      if (i >= k) break;
      w[i] = fma(-coef[i], pj, w[i]);
      out.v[i][r] = w[i];
      acc[i] = fma(w[J], w[i], acc[i]);
    }
  }
  block_sums<K>(acc, partial);
}

// the last column's scale (the only column's: FIRST)
template <int K, bool FIRST>
__global__ void __launch_bounds__(256)
orth_last_kernel(long long n, int j, int normalize, const double* __restrict__ pin, double* __restrict__ p, double* sm) {
  __shared__ double S[2 * K], coef[K], scale;
  if (FIRST)
    sum_entries<2 * K, 256>(pin, gridDim.x, S);
  else
    sum_entries<K, 256>(pin, gridDim.x, S);
  orth_column<K>(FIRST ? S + K : S, FIRST ? S[0] : sm[Small::MGS_B0 + j], j, normalize, sm, coef, &scale);
  const double sc = scale;
  if (sc == 1.0) return;
  for (long long r = (long long)blockIdx.x * 256 + threadIdx.x; r < n; r += (long long)gridDim.x * 256) p[r] *= sc;
}

// ------------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------------

template <typename T>
static VecSetT<T> vset(const T* base, long long n, int k, const double* zero) {
  VecSetT<T> s;
  for (int j = 0; j < kMaxRhs; ++j) s.v[j] = j < k ? base + (long long)j * n : (const T*)zero;
  return s;
}
static OutSet oset(double* base, long long n, int k) {  // nullptr: not written
  OutSet s;
  for (int j = 0; j < kMaxRhs; ++j) s.v[j] = j < k ? base + (long long)j * n : nullptr;
  return s;
}

static int kround(int k) { return k <= 1 ? 1 : k <= 2 ? 2 : k <= 4 ? 4 : 8; }

static unsigned sum_blocks(long long n) {
  const long long b = (n + 255) / 256;
  return (unsigned)(b < kSumBlocks ? b : kSumBlocks);
}

// f(std::integral_constant<int, K>) for the smallest instantiated K >= k
template <typename F>
static void with_k(int k, F&& f) {
  switch (kround(k)) {
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    default: f(std::integral_constant<int, 8>()); break;
  }
}

// partial sums of the squared column norms, entries slot * K ...
static int launch_norms(BlockCG* w, int k, const double* R, int slot, hipStream_t s) {
  const unsigned nb = sum_blocks(w->n);
  const VecSet r = vset(R, w->n, k, w->zero);
  with_k(k, [&](auto kk) {
    constexpr int K = decltype(kk)::value;
    norms_kernel<K><<<nb, 256, 0, s>>>(w->n, r, w->partial + (long long)slot * K * nb);
  });
  return check_launch("norms_kernel");
}

static int launch_check(BlockCG* w, int k, bool init, hipStream_t s) {
  const int nb = (int)sum_blocks(w->n);
  with_k(k, [&](auto kk) {
    bcg_check_kernel<decltype(kk)::value><<<1, 512, 0, s>>>(k, init ? 1 : 0, w->partial, nb, w->sm, w->host);
  });
  return check_launch("bcg_check_kernel");
}

static double* col(double* base, long long n, int j) { return base + (long long)j * n; }

// passes J .. k - 1 of the Gram-Schmidt, the partial sums alternating between the two halves of the buffer
template <int K, int J>
static void orth_passes(BlockCG* w, int k, int normalize, const VecSet& p, const OutSet& po, hipStream_t s) {
  if constexpr (J < K) {
    if (J >= k) return;
    const unsigned nb = sum_blocks(w->n);
    double* half = w->partial + (long long)kSumBlocks * kMaxRhs * kMaxRhs;
    orth_pass_kernel<K, J><<<nb, 256, 0, s>>>(w->n, k, normalize, J % 2 ? w->partial : half, p, po, w->sm,
                                              J % 2 ? half : w->partial);
    orth_passes<K, J + 1>(w, k, normalize, p, po, s);
  }
}

// is M R left in z32, in FP32, instead of Z?
static bool z_is_f32(const pmt_mg* mg, const BlockCG* w, int k) { return k > 1 && w->vec && mg->prec != 64; }

// P = orth(Z), or orth(Z + P beta) (iterative.py:259-292)
template <typename T>
static int orth_into_P(BlockCG* w, int k, bool initial, const T* Z, hipStream_t s) {
  const long long n = w->n;
  const unsigned nb = sum_blocks(n);
  const VecSet p = vset(w->P, n, k, w->zero);
  const VecSetT<T> z = vset(Z, n, k, w->zero);
  const OutSet po = oset(w->P, n, k);
  const double* beta = w->sm + Small::BETA;
  const int nz = initial ? 1 : 0;
  with_k(k, [&](auto kk) {
    constexpr int K = decltype(kk)::value;
    if (initial)
      orth_first_kernel<K, false, T><<<nb, 256, 0, s>>>(n, k, p, z, beta, po, w->partial);
    else
      orth_first_kernel<K, true, T><<<nb, 256, 0, s>>>(n, k, p, z, beta, po, w->partial);
    orth_passes<K, 1>(w, k, nz, p, po, s);
    double* half = w->partial + (long long)kSumBlocks * kMaxRhs * kMaxRhs;
    const double* last = k % 2 ? w->partial : half;  // where pass k - 1 left its sums
    if (k == 1)
      orth_last_kernel<K, true><<<nb, 256, 0, s>>>(n, 0, nz, last, w->P, w->sm);
    else
      orth_last_kernel<K, false><<<nb, 256, 0, s>>>(n, k - 1, nz, last, col(w->P, n, k - 1), w->sm);
  });
  return check_launch("orth kernels");
}

// Z = M R, in reduced precision left in z32: one V-cycle of all columns (the launches of a V-cycle are mostly short: k columns at once cost little
// more than one, and share the coefficients of the stored levels); column by column without its vectors
static int precondition_columns(pmt_mg* mg, BlockCG* w, int k, hipStream_t s) {
  if (k > 1 && w->vec) return mg_precondition_columns(mg, w->R, w->Z, w->z32, s, k);
  for (int j = 0; j < k; ++j) PMT_TRY(mg_precondition(mg, col(w->R, w->n, j), col(w->Z, w->n, j), s));
  return PMT_OK;
}

// iteration part 1: Q = A P, alpha, X += P alpha, R update, convergence test
static int iter_part1(pmt_mg* mg, BlockCG* w, int k, bool restart_now, hipStream_t s) {
  const long long n = w->n;
  const unsigned nb = sum_blocks(n);
  const VecSet p = vset(w->P, n, k, w->zero), q = vset(w->Q, n, k, w->zero), r = vset(w->R, n, k, w->zero),
               x = vset(w->X, n, k, w->zero);
  const OutSet xo = oset(w->X, n, k), ro = oset(w->R, n, k);
  const double* alpha = w->sm + Small::ALPHA;
  PMT_TRY(mg_level_apply(mg, 0, MODE_APPLY, w->P, nullptr, w->Q, s, k));
  with_k(k, [&](auto kk) {
    constexpr int K = decltype(kk)::value;
    if constexpr (K < 8) {
      gram_kernel<K, 2, double><<<nb, 256, 0, s>>>(n, p, q, r, w->partial);
    } else {  // 128 sums per thread would not stay in registers
      gram_kernel<K, 1, double><<<nb, 256, 0, s>>>(n, p, q, q, w->partial);
      gram_kernel<K, 1, double><<<nb, 256, 0, s>>>(n, p, r, r, w->partial + (long long)K * K * nb);
    }
    bcg_alpha_kernel<K><<<1, 1024, 0, s>>>(k, w->partial, (int)nb, w->sm);
    if (restart_now)
      update_kernel<K, false><<<nb, 256, 0, s>>>(n, k, p, q, alpha, x, xo, r, ro, w->partial);
    else
      update_kernel<K, true><<<nb, 256, 0, s>>>(n, k, p, q, alpha, x, xo, r, ro, w->partial);
  });
  PMT_TRY(check_launch("block CG update"));
  if (restart_now) {
    PMT_TRY(mg_level_apply(mg, 0, MODE_RESIDUAL, w->X, w->B, w->R, s, k));
    PMT_TRY(launch_norms(w, k, w->R, 0, s));
  }
  return launch_check(w, k, false, s);
}

// beta and P = orth(Z + P beta)
template <typename T>
static int next_directions(BlockCG* w, int k, const T* Z, hipStream_t s) {
  const long long n = w->n;
  const unsigned nb = sum_blocks(n);
  const VecSet q = vset(w->Q, n, k, w->zero);
  const VecSetT<T> z = vset(Z, n, k, w->zero);
  with_k(k, [&](auto kk) {
    constexpr int K = decltype(kk)::value;
    gram_kernel<K, 1, T><<<nb, 256, 0, s>>>(n, q, z, z, w->partial);
    bcg_beta_kernel<K><<<1, 1024, 0, s>>>(w->partial, (int)nb, w->sm);
  });
  PMT_TRY(check_launch("block CG beta"));
  return orth_into_P<T>(w, k, false, Z, s);
}

// iteration part 2: Z = M R, beta, P = orth(Z + P beta)
static int iter_part2(pmt_mg* mg, BlockCG* w, int k, hipStream_t s) {
  PMT_TRY(precondition_columns(mg, w, k, s));
  return z_is_f32(mg, w, k) ? next_directions<float>(w, k, w->z32, s) : next_directions<double>(w, k, w->Z, s);
}

static void drop_graphs(BlockCG* w) {
  for (auto& e : w->exec) {
    if (e) (void)hipGraphExecDestroy(e);
    e = nullptr;
  }
  w->graph_k = 0;
  w->graph_epoch = -1;
}

// the levels' vectors for a V-cycle of kcap columns, in one allocation: u, t, b, r per level (FP32: and the
// result of the fine level).  Without the memory for them the columns go one by one.  Four loads on
// 128x64x64: a V-cycle of 4 columns 0.42 ms (one by one 4 x 0.21 ms).
template <typename T>
static void level_columns(pmt_mg* mg, BlockCG* w) {
  long long total = 0;
  T* base = nullptr;
  auto carve = [&] {
    T* p = base;
    auto take = [&](T** v, long long n) {
      if (base) *v = p;
      p += n * w->kcap;
      total += n * w->kcap;
    };
    for (int l = 0; l < mg->nlev; ++l) {
      Level& L = mg->L[l];
      LevelCols<T>& c = L.cols<T>();
      if (l > 0) take(&c.u, L.ndof);
      if (l > 0 || sizeof(T) == 4) take(&c.b, L.ndof);
      if (l < mg->nlev - 1) take(&c.t, L.ndof);
      if (l < mg->nlev - 1) take(&c.r, L.ndof);
    }
    if (sizeof(T) == 4) take((T**)&w->z32, w->n);
  };
  carve();
  if (hipMalloc(&w->vec, (size_t)total * sizeof(T)) != hipSuccess) {
    (void)hipGetLastError();
    w->vec = nullptr;
    return;
  }
  base = (T*)w->vec;
  carve();
}

static void ensure_columns(pmt_mg* mg, BlockCG* w) {
  const int prec = mg->prec == 64 ? 64 : 32;
  if (w->vec_prec == prec) return;
  if (w->vec) (void)hipFree(w->vec);
  w->vec = nullptr;
  w->vec_prec = prec;
  drop_graphs(w);
  if (prec == 64)
    level_columns<double>(mg, w);
  else
    level_columns<float>(mg, w);
}

static void free_workspace(BlockCG* w) {
  drop_graphs(w);
  if (w->vec) (void)hipFree(w->vec);
  if (w->mem) (void)hipFree(w->mem);
  if (w->host) (void)hipHostFree(w->host);
  if (w->ev_in) (void)hipEventDestroy(w->ev_in);
  if (w->ev_out) (void)hipEventDestroy(w->ev_out);
  if (w->cs) (void)hipStreamDestroy(w->cs);
  delete w;
}

static int ensure_workspace(pmt_mg* mg, int k, hipStream_t s) {
  BlockCG* w = mg->bcg;
  const long long n = mg->L[0].ndof;
  if (w && w->kcap >= k && w->n == n) return PMT_OK;
  const int kc = kround(k);
  if (w) {
    PMT_HIP(hipStreamSynchronize(s));
    mg_forget_stream(mg, w->cs);
    free_workspace(w);
    mg->bcg = nullptr;
  }
  w = new (std::nothrow) BlockCG();
  if (!w) return arg_error("block CG: out of host memory");
  w->n = n;
  w->kcap = kc;
  const long long doubles = 6LL * kc * n + n + Small::SIZE + 2LL * kSumBlocks * kMaxRhs * kMaxRhs;
  hipError_t e = hipMalloc((void**)&w->mem, (size_t)doubles * sizeof(double));
  if (e != hipSuccess) {
    delete w;
    return hip_status(e, "block CG workspace");
  }
  double* p = w->mem;
  w->X = p;
  p += (long long)kc * n;
  w->B = p;
  p += (long long)kc * n;
  w->P = p;
  p += (long long)kc * n;
  w->Q = p;
  p += (long long)kc * n;
  w->R = p;
  p += (long long)kc * n;
  w->Z = p;
  p += (long long)kc * n;
  w->zero = p;
  p += n;
  w->sm = p;
  p += Small::SIZE;
  w->partial = p;
  e = hipHostMalloc((void**)&w->host, 16 * sizeof(double), hipHostMallocCoherent);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&w->cs, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&w->ev_in, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&w->ev_out, hipEventDisableTiming);
  if (e != hipSuccess) {
    free_workspace(w);
    return hip_status(e, "block CG stream/events");
  }
  w->host[0] = 0.0;
  w->host[1] = -1.0;  // no test number yet
  mg->bcg = w;
  // zero column and zeroed blocks (a fill kernel, not a memset: the buffers are captured later)
  return launch_fill(6LL * kc * n + n + Small::SIZE, 0.0, w->mem, s);
}

template <typename F>
static int capture(hipGraphExec_t* exec, hipStream_t s, F&& body) {
  hipGraph_t graph = nullptr;
  PMT_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  const int rc = body();
  const hipError_t e = hipStreamEndCapture(s, &graph);
  if (rc != PMT_OK) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  PMT_HIP(e);
  const hipError_t ei = hipGraphInstantiate(exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  return hip_status(ei, "hipGraphInstantiate");
}

// the largest relative residual of the last convergence test (launched with launch_check)
static int read_max(BlockCG* w, hipStream_t s, double* mx) {
  return publish_wait(w->host, w->seq, w->sm + Small::TMAX, w->host + 2, mx, s);
}

void block_cg_release(pmt_mg* mg) {
  if (!mg->bcg) return;
  mg_forget_stream(mg, mg->bcg->cs);
  free_workspace(mg->bcg);
  mg->bcg = nullptr;
}

void block_cg_invalidate(pmt_mg* mg) {
  if (mg->bcg) drop_graphs(mg->bcg);
}

}  // namespace pmt

using namespace pmt;

extern "C" {

int pmt_block_pcg_solve(pmt_mg* mg, int k, const double* B, double* X, int x0_is_zero, double tol, int maxit,
                        int restart, int use_graph, int* iters, double* relres, double* history, void* stream) {
  if (!mg || !B || !X || k < 1 || k > kMaxRhs || maxit < 0 || restart < 1)
    return arg_error("pmt_block_pcg_solve: bad argument (1 <= k <= 8 right-hand sides)");
  if (!mg->ready) {
    set_error("pmt_block_pcg_solve: call pmt_mg_update first");
    return PMT_ERR_STATE;
  }
  hipStream_t caller = (hipStream_t)stream;
  PMT_TRY(ensure_workspace(mg, k, caller));
  BlockCG* w = mg->bcg;
  if (k > 1) ensure_columns(mg, w);
  // all work on the handle's stream, after what the caller queued before this call
  hipStream_t s = w->cs;
  PMT_HIP(hipEventRecord(w->ev_in, caller));
  PMT_HIP(hipStreamWaitEvent(s, w->ev_in, 0));
  PMT_TRY(mg_join(mg, s));  // the coarsest inverse of the last update, before anything is captured on s
  const long long n = w->n;
  const size_t bytes = (size_t)k * n * sizeof(double);
  PMT_HIP(hipMemcpyAsync(w->B, B, bytes, hipMemcpyDeviceToDevice, s));
  if (x0_is_zero) {
    PMT_TRY(launch_fill((long long)k * n, 0.0, w->X, s));
    PMT_HIP(hipMemcpyAsync(w->R, B, bytes, hipMemcpyDeviceToDevice, s));
  } else {
    PMT_HIP(hipMemcpyAsync(w->X, X, bytes, hipMemcpyDeviceToDevice, s));
    PMT_TRY(mg_level_apply(mg, 0, MODE_RESIDUAL, w->X, w->B, w->R, s, k));
  }
  // numbers of this solve's convergence tests: past any that an earlier, failed solve may still publish
  w->seq += 2.0;
  PMT_TRY(launch_fill(1, w->seq, w->sm + Small::SEQ, s));
  PMT_TRY(launch_norms(w, k, w->R, 0, s));
  PMT_TRY(launch_norms(w, k, w->B, 1, s));
  PMT_TRY(launch_check(w, k, true, s));
  double mx = 0.0;
  w->seq += 1.0;
  PMT_TRY(read_max(w, s, &mx));
  bool done = mx <= tol;
  if (history) history[0] = mx;
  auto non_finite = [&](int at) -> int {
    PMT_HIP(hipEventRecord(w->ev_out, s));
    PMT_HIP(hipStreamWaitEvent(caller, w->ev_out, 0));
    if (iters) *iters = at;
    if (relres)
      for (int j = 0; j < k; ++j) relres[j] = mx;
    set_error("pmt_block_pcg_solve: non-finite residual at iteration " + std::to_string(at) +
              " (non-finite right-hand side, start vector or operator)");
    return PMT_ERR_NUMERIC;
  };
  if (!std::isfinite(mx)) return non_finite(0);
  int it = 0;
  if (!done) {
    // P = orth(Z, normalize=True), Z = M R
    PMT_TRY(precondition_columns(mg, w, k, s));
    if (z_is_f32(mg, w, k))
      PMT_TRY(orth_into_P<float>(w, k, true, w->z32, s));
    else
      PMT_TRY(orth_into_P<double>(w, k, true, w->Z, s));
    const bool graphs = use_graph != 0;
    if (graphs && (w->graph_k != k || w->graph_epoch != tuning_epoch())) {
      drop_graphs(w);
      PMT_TRY(capture(&w->exec[0], s, [&] { return iter_part1(mg, w, k, true, s); }));
      PMT_TRY(capture(&w->exec[1], s, [&] { return iter_part1(mg, w, k, false, s); }));
      PMT_TRY(capture(&w->exec[2], s, [&] { return iter_part2(mg, w, k, s); }));
      w->graph_k = k;
      w->graph_epoch = tuning_epoch();
    }
    for (it = 0; it < maxit; ++it) {
      const bool rs = it % restart == 0;
      if (graphs)
        PMT_HIP(hipGraphLaunch(w->exec[rs ? 0 : 1], s));
      else
        PMT_TRY(iter_part1(mg, w, k, rs, s));
      w->seq += 1.0;
      PMT_TRY(read_max(w, s, &mx));
      done = mx <= tol;
      if (history) history[it + 1] = mx;
      if (!std::isfinite(mx)) return non_finite(it + 1);
      if (done) break;
      if (graphs)
        PMT_HIP(hipGraphLaunch(w->exec[2], s));
      else
        PMT_TRY(iter_part2(mg, w, k, s));
    }
    if (it < maxit) ++it;
  }
  PMT_HIP(hipMemcpyAsync(X, w->X, bytes, hipMemcpyDeviceToDevice, s));
  PMT_HIP(hipMemcpyAsync(w->host + 2, w->sm + Small::TVAL, (size_t)k * sizeof(double), hipMemcpyDeviceToHost, s));
  PMT_HIP(hipEventRecord(w->ev_out, s));
  PMT_HIP(hipStreamWaitEvent(caller, w->ev_out, 0));
  PMT_HIP(hipStreamSynchronize(s));
  if (relres)
    for (int j = 0; j < k; ++j) relres[j] = w->host[2 + j];
  if (iters) *iters = it;
  return PMT_OK;
}

}  // extern "C"
