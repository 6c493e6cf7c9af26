// Element-wise and reduction kernels: SIMP power law, axpby, deterministic dot products,
// Dirichlet split for the linear-dependency-aware solve, and the fused CG vector updates.
//
// Reductions use a fixed grid of kReduceBlocks blocks with grid-stride loops, per-block
// partials in a caller workspace, and a single-block second stage summing the partials in a
// fixed order, so every dot product is bit-reproducible run to run.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "launch.h"

namespace pmt {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

int hip_status(hipError_t err, const char* where) {
  if (err == hipSuccess) return PMT_OK;
  set_error(std::string(where) + ": " + hipGetErrorString(err));
  return PMT_ERR_HIP;
}

int check_launch(const char* where) { return hip_status(hipGetLastError(), where); }

// x^p: repeated products for a small whole exponent (ip >= 0; SIMP's p = 3 and its derivative's 2, within
// an ulp or two of pow and a fraction of its cost), else pow
__device__ inline double powlaw_pow(double x, double p, int ip) {
  if (ip < 0) return pow(x, p);
  double r = 1.0;
  for (int k = 0; k < ip; ++k) r *= x;
  return r;
}

// ip for powlaw_pow: p itself when it is a whole number in [0, 8], else -1
static int powlaw_int_exponent(double p) { return (p >= 0.0 && p <= 8.0 && p == std::floor(p)) ? (int)p : -1; }

__global__ void powlaw_fwd_kernel(long long n, double a, double b, double p, int ip, const double* __restrict__ x,
                                  double* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = a + b * powlaw_pow(x[i], p, ip);
}

// Heaviside projection (ex_compliance_robust.py:139, a MathExpression of the reference):
//   y = (tanh(beta*eta) + tanh(beta*(x - eta))) / (tanh(beta*eta) + tanh(beta*(1 - eta)))
// dx = dy * beta * (1 - tanh^2(beta*(x - eta))) / den; optional dbeta_i = dy_i * dy_i/dbeta.
__global__ void heaviside_fwd_kernel(long long n, double beta, double eta, const double* __restrict__ x,
                                     double* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double te = tanh(beta * eta);
  const double den = te + tanh(beta * (1.0 - eta));
  y[i] = (te + tanh(beta * (x[i] - eta))) / den;
}

__global__ void heaviside_bwd_kernel(long long n, double beta, double eta, const double* __restrict__ x,
                                     const double* __restrict__ dy, double* __restrict__ dx, int accumulate,
                                     double* __restrict__ dbeta) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double te = tanh(beta * eta), t1 = tanh(beta * (1.0 - eta)), tx = tanh(beta * (x[i] - eta));
  const double den = te + t1, num = te + tx;
  const double g = dy[i] * beta * (1.0 - tx * tx) / den;
  dx[i] = accumulate ? dx[i] + g : g;
  if (dbeta) {
    const double dnum = eta * (1.0 - te * te) + (x[i] - eta) * (1.0 - tx * tx);
    const double dden = eta * (1.0 - te * te) + (1.0 - eta) * (1.0 - t1 * t1);
    dbeta[i] = dy[i] * (dnum / den - num * dden / (den * den));
  }
}

// OC update for one bisection value lmid (pymoto/common/optimizers.py:420-433):
//   xnew = clip(x * sqrt(-min(dg, 0) / lmid), max(xmin, x - move), min(xmax, x + move))
// and per-block partial sums of xnew (for the volume test).
__global__ void oc_update_kernel(long long n, const double* __restrict__ x, const double* __restrict__ dg,
                                 double xmin, double xmax, double move, double lmid, double* __restrict__ xnew,
                                 double* __restrict__ partial);

__global__ void powlaw_bwd_kernel(long long n, double c, double q, int iq, const double* __restrict__ x,
                                  const double* __restrict__ dy, double* __restrict__ dx, int accumulate) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const double v = dy[i] * (c * powlaw_pow(x[i], q, iq));
    dx[i] = accumulate ? dx[i] + v : v;
  }
}

__global__ void axpby_kernel(long long n, double a, const double* __restrict__ x, double b, double* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (x ? a * x[i] : 0.0) + (b == 0.0 ? 0.0 : b * y[i]);
}

__device__ inline double block_sum(double v) {
  __shared__ double sh[kReduceThreads / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) {
    for (int w = 0; w < kReduceThreads / 64; ++w) r += sh[w];
  }
  __syncthreads();
  return r;  // valid in thread 0
}

// stage 1: NOUT dot products sharing the grid-stride loop; partial[o*kReduceBlocks + block]
template <int NOUT>
__global__ void __launch_bounds__(kReduceThreads)
dot_stage1(long long n, const double* __restrict__ a0, const double* __restrict__ b0, const double* __restrict__ a1,
           const double* __restrict__ b1, double* __restrict__ partial) {
  double s0 = 0.0, s1 = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    s0 = fma(a0[i], b0[i], s0);
    if (NOUT > 1) s1 = fma(a1[i], b1[i], s1);
  }
  double r0 = block_sum(s0);
  if (threadIdx.x == 0) partial[blockIdx.x] = r0;
  if (NOUT > 1) {
    double r1 = block_sum(s1);
    if (threadIdx.x == 0) partial[kReduceBlocks + blockIdx.x] = r1;
  }
}

// stage 2: out[o] = sum of partials (fixed order), one block
template <int NOUT>
__global__ void __launch_bounds__(kReduceThreads) dot_stage2(const double* __restrict__ partial, double* __restrict__ out) {
  for (int o = 0; o < NOUT; ++o) {
    double s = 0.0;
    for (int b = threadIdx.x; b < kReduceBlocks; b += blockDim.x) s += partial[o * kReduceBlocks + b];
    double r = block_sum(s);
    if (threadIdx.x == 0) out[o] = r;
  }
}

// out[0] = sum of nparts partials (fixed order, one block of 1024 threads, each thread's strided loads
// issued eight at a time); host (optional): also hands the sum to the host through pinned memory (the
// protocol of publish_kernel: value, system-scope fence, sequence number)
constexpr int kStage2Threads = 1024;
__global__ void __launch_bounds__(kStage2Threads) parts_stage2(const double* __restrict__ partial, long long nparts,
                                                               double* __restrict__ out, double seq, double* host) {
  double s = 0.0;
  long long b = threadIdx.x;
  for (; b + 7LL * kStage2Threads < nparts; b += 8LL * kStage2Threads) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = partial[b + (long long)k * kStage2Threads];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += v[k];
  }
  for (; b < nparts; b += kStage2Threads) s += partial[b];
  __shared__ double sh[kStage2Threads / 64];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = 0.0;
    for (int w = 0; w < kStage2Threads / 64; ++w) r += sh[w];
    out[0] = r;
    if (host) {
      volatile double* h = host;
      h[0] = r;
      __threadfence_system();
      h[1] = seq;
      __threadfence_system();
    }
  }
}

__global__ void oc_update_kernel(long long n, const double* __restrict__ x, const double* __restrict__ dg,
                                 double xmin, double xmax, double move, double lmid, double* __restrict__ xnew,
                                 double* __restrict__ partial) {
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const double xi = x[i];
    const double lb = fmax(xmin, xi - move), ub = fmin(xmax, xi + move);
    const double v = fmin(fmax(xi * sqrt(-fmin(dg[i], 0.0) / lmid), lb), ub);
    xnew[i] = v;
    s += v;
  }
  const double t = block_sum(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// The whole OC bisection on the device (pmt_oc_step).  A pass evaluates the 2^kOcLv - 1 multipliers that the next
// kOcLv bisection steps can ask for (the nodes of the bisection tree under [l1, l2]) in one sweep over x and
// dg; the next pass starts with summing the partials and walking the kOcLv decisions (every block for itself,
// block 0 leaves the new interval in the other of two states), so the host reads nothing between the steps and
// nothing is launched between the passes.  Every sum is formed as oc_update_kernel and dot_stage2 form it
// (the same blocks, strides and tree), so the decisions and the design are those of the step-by-step
// bisection, bit for bit.
// x sqrt(s / l) falls with l: above s (x / lb)^2 the entry is lb, below s (x / ub)^2 it is ub; outside a
// 1e-12 margin of the two (the computed value is good to 4e-16) the root is not evaluated.
// 30 steps of 524,288 elements: 152 us (163 us with a launch for the decisions after each pass, 734 us with a launch
// pair and a host read per step).  More steps per pass save launches, but every multiplier costs every element a
// root: 4 steps took 193 instead of 166 us, 5 took 255.  (Letting the pass's last block choose, behind a ticket, saves the second launch
// but costs every block a release fence: 27 instead of 8.8 us per pass.)
struct OcState {
  double l1, l2, last, maxdg;  // last: the multiplier of the last step
};
constexpr int kOcLv = 3, kOcNodes = (1 << kOcLv) - 1;
constexpr int kOcState = 8;    // doubles that hold a state
constexpr int kOcThreads = 1024;  // of a pass: kOcGroups blocks of oc_update_kernel in one, so that few blocks sum
constexpr int kOcGroups = kOcThreads / kReduceThreads;

__global__ void oc_init_kernel(double l1, double l2, OcState* st) { *st = OcState{l1, l2, 0.0, 0.0}; }

// the multiplier of tree node h >= 1: its bits below the leading one are the decisions (1: l1 = mid)
__device__ inline double oc_node(int h, double a, double b) {
  for (int bit = 30 - __clz(h); bit >= 0; --bit) {
    const double m = 0.5 * (a + b);
    if ((h >> bit) & 1)
      a = m;
    else
      b = m;
  }
  return 0.5 * (a + b);
}

// the decisions of a pass (prev: its state before, partial: its sums) by a block of kOcThreads, into `out` of every
// thread: a wave per sum, in dot_stage2's order (4 waves of strided sums, their trees, then wave after wave); nb
// blocks wrote partials, the others have no entries
__device__ inline void oc_choose(int nb, double tol, double target, int first, const OcState* __restrict__ prev,
                                 const double* __restrict__ partial, OcState& out) {
  constexpr int M = kOcNodes, NW = kReduceThreads / 64, NK = kReduceBlocks / kReduceThreads;
  static_assert(M < kOcThreads / 64, "a wave per sum");
  __shared__ double sums[M + 1];
  out = *prev;
  if (!(out.l2 - out.l1 > tol) && !first) return;
  const int lane = threadIdx.x & 63, c = threadIdx.x >> 6;
  if (c < M) {
    double p[NW][NK];
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const int b = w * 64 + lane + k * kReduceThreads;
        p[w][k] = b < nb ? partial[c * kReduceBlocks + b] : 0.0;
      }
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      double t = 0.0;
#pragma unroll
      for (int k = 0; k < NK; ++k) t += p[w][k];
      for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
      r += t;
    }
    if (lane == 0) sums[c] = r;
  }
  if (first && c == M) {
    double m = -INFINITY;
    for (int b = lane; b < nb; b += 64) {
      const double o = partial[M * kReduceBlocks + b];
      m = (o > m || o != o) ? o : m;
    }
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_down(m, off, 64);
      m = (o > m || o != o) ? o : m;
    }
    if (lane == 0) sums[M] = m;
  }
  __syncthreads();
  int h = 1;
  for (int step = 0; step < kOcLv && out.l2 - out.l1 > tol; ++step) {
    out.last = 0.5 * (out.l1 + out.l2);
    if (sums[h - 1] - target > 0.0) {
      out.l1 = out.last;
      h = 2 * h + 1;
    } else {
      out.l2 = out.last;
      h = 2 * h;
    }
  }
  if (first) out.maxdg = sums[M];
}

// pass p: the decisions of pass p - 1 (p > 0; states and partials alternate between two sets), then the sums of its
// own multipliers.  A group of 256 threads forms one block's partials of oc_update_kernel.
__global__ void __launch_bounds__(kOcThreads)
oc_pass_kernel(long long n, int nb, const double* __restrict__ x, const double* __restrict__ dg, double xmin,
               double xmax, double move, double tol, double target, int pass, const OcState* __restrict__ prev,
               const double* __restrict__ pin, OcState* __restrict__ st, double* __restrict__ partial) {
  constexpr int M = kOcNodes;
  __shared__ double lm[M], wsum[kOcThreads / 64][M];
  __shared__ double red[kOcThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool first = pass == 0;
  OcState now;
  if (first) {
    now = *prev;
  } else {
    oc_choose(nb, tol, target, pass == 1, prev, pin, now);
    if (blockIdx.x == 0 && tid == 0) *st = now;
  }
  const double l1 = now.l1, l2 = now.l2;
  if (!(l2 - l1 > tol) && !first) return;
  if (tid < M) lm[tid] = oc_node(tid + 1, l1, l2);
  __syncthreads();
  const int group = tid / kReduceThreads, block = (int)blockIdx.x * kOcGroups + group, gt = tid % kReduceThreads;
  double s[M];
#pragma unroll
  for (int c = 0; c < M; ++c) s[c] = 0.0;
  double mx = -INFINITY;
  for (long long i = (long long)block * kReduceThreads + gt; i < n; i += (long long)kReduceBlocks * kReduceThreads) {
    const double xi = x[i], di = dg[i];
    const double lb = fmax(xmin, xi - move), ub = fmin(xmax, xi + move), g = -fmin(di, 0.0);
    mx = (di > mx || di != di) ? di : mx;
    // outside these the clip decides (needs positive x, bounds and multipliers; else every value is evaluated)
    const bool sure = xi > 0.0 && lb > 0.0 && ub >= lb && g > 0.0 && l1 >= 0.0;
    const double rl = xi / lb, ru = xi / ub;
    const double hi = sure ? g * rl * rl * (1.0 + 1e-12) : INFINITY, lo = sure ? g * ru * ru * (1.0 - 1e-12) : -INFINITY;
#pragma unroll
    for (int c = 0; c < M; ++c) {
      double v = lm[c] > hi ? lb : ub;
      if (!(lm[c] > hi || lm[c] < lo)) v = fmin(fmax(xi * sqrt(g / lm[c]), lb), ub);
      s[c] += v;
    }
  }
  // block_sum of every entry, with one barrier for all
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int c = 0; c < M; ++c) s[c] += __shfl_down(s[c], off, 64);
  if (lane == 0) {
#pragma unroll
    for (int c = 0; c < M; ++c) wsum[wave][c] = s[c];
  }
  if (first) {
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_down(mx, off, 64);
      mx = (o > mx || o != o) ? o : mx;
    }
    if (lane == 0) red[wave] = mx;
  }
  __syncthreads();
  if (block >= nb) return;
  const int w0 = group * (kReduceThreads / 64);
  if (gt < M) {
    double r = 0.0;
    for (int w = 0; w < kReduceThreads / 64; ++w) r += wsum[w0 + w][gt];
    partial[gt * kReduceBlocks + block] = r;
  }
  if (first && gt == M) {
    double m = red[w0];
    for (int w = 1; w < kReduceThreads / 64; ++w) m = (red[w0 + w] > m || red[w0 + w] != red[w0 + w]) ? red[w0 + w] : m;
    partial[M * kReduceBlocks + block] = m;
  }
}

// the decisions of the last pass
__global__ void __launch_bounds__(kOcThreads)
oc_last_kernel(int nb, double tol, double target, int first, const OcState* __restrict__ prev,
               const double* __restrict__ partial, OcState* st) {
  OcState now;
  oc_choose(nb, tol, target, first, prev, partial, now);
  __syncthreads();
  if (threadIdx.x == 0) *st = now;
}

// the design of the last step's multiplier
__global__ void oc_write_kernel(long long n, const double* __restrict__ x, const double* __restrict__ dg, double xmin,
                                double xmax, double move, const OcState* __restrict__ st, double* __restrict__ xnew) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double xi = x[i];
  const double lb = fmax(xmin, xi - move), ub = fmin(xmax, xi + move);
  xnew[i] = fmin(fmax(xi * sqrt(-fmin(dg[i], 0.0) / st->last), lb), ub);
}

int launch_dot(long long n, const double* x, const double* y, double* out, double* work, hipStream_t s) {
  dot_stage1<1><<<kReduceBlocks, kReduceThreads, 0, s>>>(n, x, y, nullptr, nullptr, work);
  PMT_TRY(check_launch("dot_stage1"));
  dot_stage2<1><<<1, kReduceThreads, 0, s>>>(work, out);
  return check_launch("dot_stage2");
}

int launch_dot2(long long n, const double* a0, const double* b0, const double* a1, const double* b1, double* out,
                double* work, hipStream_t s) {
  dot_stage1<2><<<kReduceBlocks, kReduceThreads, 0, s>>>(n, a0, b0, a1, b1, work);
  PMT_TRY(check_launch("dot_stage1<2>"));
  dot_stage2<2><<<1, kReduceThreads, 0, s>>>(work, out);
  return check_launch("dot_stage2<2>");
}

// CG: r -= alpha q, partial ||r||^2 (x += alpha p comes later, with the p update); alpha = sc[1]/sc[0] read on
// device; r32 (optional): the new r rounded to FP32, the input of a
// reduced-precision preconditioner; u1 (optional): omega * D^-1 * r, the preconditioner's first sweep from zero
// in its precision (the expression of jacobi0_kernel).  One pass over the vectors: a block
// owns kXrPer * 256 consecutive entries (strided by 256 per step, so every step is coalesced and the
// steps' loads are independent) and writes its sum of r^2 to partial[block]; the fixed-order second
// stage is parts_stage2.  At 12.8M dofs: 71 us (4 per thread) for the 461 MB of the mixed-precision
// update, where the fixed 1024-block grid-stride loop of the dots took 84 us.
constexpr int kXrPer = 4;
constexpr long long kMaxParts = 2048;

long long cg_xr_parts(long long n) { return (n + 256LL * kXrPer - 1) / (256LL * kXrPer); }

// The sums of NOUT sets of np <= kMaxParts partials (set o at partial + o * np), in a fixed order, in every thread
// of a block of 256: a kernel that needs them adds them itself, all loads in flight, instead of waiting for a
// launch that does (3 to 4 us each on the chain of a small problem's iteration; 1 us here).  An iteration on
// 96x48x48 (FP64) so took 15 us less of 180; on 256x128x128 (760 partials, 12,530 blocks that add them) the same.
template <int NOUT>
__device__ inline void block_parts(const double* __restrict__ partial, int np, double (&out)[NOUT]) {
  constexpr int PER = (int)(kMaxParts / kReduceThreads);
  __shared__ double sh[NOUT][kReduceThreads / 64];
  double v[NOUT][PER];
#pragma unroll
  for (int o = 0; o < NOUT; ++o)
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int b = threadIdx.x + k * kReduceThreads;
      v[o][k] = b < np ? partial[o * np + b] : 0.0;
    }
#pragma unroll
  for (int o = 0; o < NOUT; ++o) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < PER; ++k) t += v[o][k];
    for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    if ((threadIdx.x & 63) == 0) sh[o][threadIdx.x >> 6] = t;
  }
  __syncthreads();
#pragma unroll
  for (int o = 0; o < NOUT; ++o) {
    out[o] = 0.0;
    for (int w = 0; w < kReduceThreads / 64; ++w) out[o] += sh[o][w];
  }
}

// dots (np > 0): the partials of p.q and p.r, added here; block 0 leaves the sums in sc[0], sc[1]
template <bool PARTS, typename U>
__global__ void __launch_bounds__(kReduceThreads)
cg_xr_update(long long n, double* __restrict__ sc, const double* __restrict__ dots, int np,
             const double* __restrict__ q, double* __restrict__ r, double* __restrict__ partial,
             float* __restrict__ r32, const U* __restrict__ dinv, U omega, U* __restrict__ u1) {
  const long long base = (long long)blockIdx.x * (256 * kXrPer) + threadIdx.x;
  double qv[kXrPer], rv[kXrPer];
  U dv[kXrPer];
  if constexpr (PARTS) {  // the entries' loads are in flight during the sums
#pragma unroll
    for (int k = 0; k < kXrPer; ++k) {
      const long long i = base + 256LL * k < n ? base + 256LL * k : n - 1;
      qv[k] = q[i];
      rv[k] = r[i];
      dv[k] = u1 ? dinv[i] : (U)0;
    }
  }
  double alpha;
  if constexpr (PARTS) {
    double pq[2];
    block_parts<2>(dots, np, pq);
    alpha = pq[1] / pq[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      sc[0] = pq[0];
      sc[1] = pq[1];
    }
  } else {
    alpha = sc[1] / sc[0];
  }
  double s = 0.0;
  auto step = [&](int k) {
    const long long i = base + 256LL * k;
    const double v = PARTS ? fma(-alpha, qv[k], rv[k]) : fma(-alpha, q[i], r[i]);
    r[i] = v;
    const U rf = (U)v;
    if (r32) r32[i] = (float)v;
    if (u1) u1[i] = omega * (PARTS ? dv[k] : dinv[i]) * rf;
    s = fma(v, v, s);
  };
  if (base + 256LL * (kXrPer - 1) < n) {  // every block but the last: no bounds test between the steps
#pragma unroll
    for (int k = 0; k < kXrPer; ++k) step(k);
  } else {
#pragma unroll
    for (int k = 0; k < kXrPer; ++k)
      if (base + 256LL * k < n) step(k);
  }
  double t = block_sum(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// alpha = r.b / b.b from their partials (dot_stage1's; the sums and bits of dot_stage2): r -= alpha b and, with y,
// y += sign alpha x
__global__ void __launch_bounds__(kReduceThreads)
lda_project_kernel(long long n, const double* __restrict__ partial, const double* __restrict__ b,
                   const double* __restrict__ x, double sign, double* __restrict__ r, double* __restrict__ y) {
  double bv[kXrPer], xv[kXrPer], rv[kXrPer], yv[kXrPer], rb[2];
  const long long base = (long long)blockIdx.x * (256 * kXrPer) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kXrPer; ++k) {  // in flight during the sums
    const long long i = base + 256LL * k < n ? base + 256LL * k : n - 1;
    bv[k] = b[i];
    rv[k] = r[i];
    xv[k] = y ? x[i] : 0.0;
    yv[k] = y ? y[i] : 0.0;
  }
  block_parts<2>(partial, kReduceBlocks, rb);
  const double alpha = rb[0] / rb[1], ya = sign * alpha;
#pragma unroll
  for (int k = 0; k < kXrPer; ++k) {
    const long long i = base + 256LL * k;
    if (i >= n) return;
    r[i] = fma(-alpha, bv[k], rv[k]);
    if (y) y[i] = fma(ya, xv[k], yv[k]);
  }
}

// partials of a0.b0 (entry 0..) and a1.b1 (entry np..), blocks as dot_flat
__global__ void __launch_bounds__(kReduceThreads)
dot2_flat(long long n, const double* __restrict__ a0, const double* __restrict__ b0, const double* __restrict__ a1,
          const double* __restrict__ b1, double* __restrict__ partial) {
  double s0 = 0.0, s1 = 0.0;
  const long long base = (long long)blockIdx.x * (256 * kXrPer) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kXrPer; ++k) {
    const long long i = base + 256LL * k;
    if (i < n) {
      s0 = fma(a0[i], b0[i], s0);
      s1 = fma(a1[i], b1[i], s1);
    }
  }
  const double t0 = block_sum(s0), t1 = block_sum(s1);
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = t0;
    partial[gridDim.x + blockIdx.x] = t1;
  }
}

// x.y in one flat pass (the cg_xr_update blocking: kXrPer * 256 entries per block, partial[block]); its
// second stage is parts_stage2.  For the dots of the CG loop, whose bits need not match pmt_dot's.
template <typename Y>
__global__ void __launch_bounds__(kReduceThreads)
dot_flat(long long n, const double* __restrict__ x, const Y* __restrict__ y, double* __restrict__ partial) {
  double s = 0.0;
  const long long base = (long long)blockIdx.x * (256 * kXrPer) + threadIdx.x;
  if (base + 256LL * (kXrPer - 1) < n) {
#pragma unroll
    for (int k = 0; k < kXrPer; ++k) s = fma(x[base + 256LL * k], (double)y[base + 256LL * k], s);
  } else {
    for (int k = 0; k < kXrPer; ++k)
      if (base + 256LL * k < n) s = fma(x[base + 256LL * k], (double)y[base + 256LL * k], s);
  }
  const double t = block_sum(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// CG restart branch: x += alpha p only
__global__ void cg_x_update(long long n, const double* __restrict__ sc, const double* __restrict__ p,
                            double* __restrict__ x) {
  const double alpha = sc[1] / sc[0];
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = fma(alpha, p[i], x[i]);
}

// CG: p = z + beta p with beta = -sc[3]/sc[0]   (iterative.py:394-395); z FP64 or the FP32 output of a
// reduced-precision preconditioner (widened exactly).  x (optional): first the x update the iteration's
// cg_xr_update left out, x += alpha p with alpha = sc[1]/sc[0] and the old p - the same
// expression, so the iterates are bitwise those of the undeferred update, for one read of p fewer
template <typename Z, bool WITHX>
__global__ void cg_p_update(long long n, const double* __restrict__ sc, const Z* __restrict__ z,
                            double* __restrict__ p, double* __restrict__ x) {
  const double beta = -sc[3] / sc[0];
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const double pv = p[i];
    if (WITHX) x[i] = fma(sc[1] / sc[0], pv, x[i]);
    p[i] = fma(beta, pv, (double)z[i]);
  }
}

// the same with q.z from its np partials (few blocks of kXrPer entries per thread: each adds them)
template <typename Z, bool WITHX>
__global__ void __launch_bounds__(kReduceThreads)
cg_p_update_parts(long long n, const double* __restrict__ sc, const double* __restrict__ parts, int np,
                  const Z* __restrict__ z, double* __restrict__ p, double* __restrict__ x) {
  double qz[1], pv[kXrPer], zv[kXrPer], xv[kXrPer];
  const double pq = sc[0], alpha = WITHX ? sc[1] / pq : 0.0;
  const long long base = (long long)blockIdx.x * (256 * kXrPer) + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kXrPer; ++k) {
    const long long i = base + 256LL * k < n ? base + 256LL * k : n - 1;  // loads in flight during the sum
    pv[k] = p[i];
    zv[k] = (double)z[i];
    xv[k] = WITHX ? x[i] : 0.0;
  }
  block_parts<1>(parts, np, qz);
  const double beta = -qz[0] / pq;
#pragma unroll
  for (int k = 0; k < kXrPer; ++k) {
    const long long i = base + 256LL * k;
    if (i >= n) return;
    if (WITHX) x[i] = fma(alpha, pv[k], xv[k]);
    p[i] = fma(beta, pv[k], zv[k]);
  }
}

// p = z / sqrt(sc[k])  (orth(z, normalize=True) for one column, iterative.py:286-290)
__global__ void scale_rsqrt(long long n, const double* __restrict__ sc, int k, const double* __restrict__ z,
                            double* __restrict__ p) {
  const double inv = 1.0 / sqrt(sc[k]);
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = z[i] * inv;
}

__global__ void bc_split_kernel(long long nnodes, int D, const uint8_t* __restrict__ bcm, double bcdiag,
                                const double* __restrict__ rhs, double* __restrict__ rl, double* __restrict__ sol) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nnodes * D) return;
  const long long n = q / D;
  const int d = (int)(q - n * D);
  const bool fixed = bcm && ((bcm[n] >> d) & 1u);
  const double v = rhs[q];
  rl[q] = fixed ? 0.0 : v;
  sol[q] = fixed ? v / bcdiag : 0.0;
}

__global__ void axpy_free_kernel(long long nnodes, int D, const uint8_t* __restrict__ bcm, double a,
                                 const double* __restrict__ x, double* __restrict__ y) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nnodes * D) return;
  const long long n = q / D;
  const int d = (int)(q - n * D);
  const bool fixed = bcm && ((bcm[n] >> d) & 1u);
  if (!fixed) y[q] = fma(a, x[q], y[q]);
}

__global__ void fill_kernel(long long n, double v, double* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = v;
}

int launch_axpby(long long n, double a, const double* x, double b, double* y, hipStream_t s) {
  if (n <= 0) return PMT_OK;
  axpby_kernel<<<blocks_for(n, 256), 256, 0, s>>>(n, a, x, b, y);
  return check_launch("axpby_kernel");
}

bool cg_sums_inline(long long np) { return np <= kMaxParts; }

template <typename U>
int launch_cg_xr_update(long long n, double* sc, const double* dots, long long np, const double* q, double* r,
                        double* work, double* out_rr, hipStream_t s, float* r32, const U* dinv, double omega, U* u1,
                        double* host, double seq) {
  if (n <= 0) return PMT_OK;
  const long long parts = cg_xr_parts(n);
  if (dots)
    cg_xr_update<true, U><<<(unsigned)parts, kReduceThreads, 0, s>>>(n, sc, dots, (int)np, q, r, work, r32, dinv,
                                                                    (U)omega, u1);
  else
    cg_xr_update<false, U><<<(unsigned)parts, kReduceThreads, 0, s>>>(n, sc, nullptr, 0, q, r, work, r32, dinv,
                                                                     (U)omega, u1);
  PMT_TRY(check_launch("cg_xr_update"));
  parts_stage2<<<1, kStage2Threads, 0, s>>>(work, parts, out_rr, seq, host);
  return check_launch("parts_stage2");
}
template int launch_cg_xr_update<double>(long long, double*, const double*, long long, const double*, double*, double*,
                                         double*, hipStream_t, float*, const double*, double, double*, double*, double);
template int launch_cg_xr_update<float>(long long, double*, const double*, long long, const double*, double*, double*,
                                        double*, hipStream_t, float*, const float*, double, float*, double*, double);

int launch_dot2_flat(long long n, const double* a0, const double* b0, const double* a1, const double* b1,
                     double* work, hipStream_t s) {
  if (n <= 0) return PMT_OK;
  dot2_flat<<<(unsigned)cg_xr_parts(n), kReduceThreads, 0, s>>>(n, a0, b0, a1, b1, work);
  return check_launch("dot2_flat");
}

double publish_sequence() {
  static std::atomic<long long> seq{0};
  return (double)seq.fetch_add(1, std::memory_order_relaxed) + 1.0;
}

int publish_wait(const double* host, double seq, const double* dev, double* pinned, double* v, hipStream_t s) {
  const volatile double* h = host;
  const auto t0 = std::chrono::steady_clock::now();
  for (;;) {
    if (h[1] == seq) {
      *v = h[0];
      return PMT_OK;
    }
    if (std::chrono::steady_clock::now() - t0 > std::chrono::seconds(1)) {
      PMT_HIP(hipMemcpyAsync(pinned, dev, sizeof(double), hipMemcpyDeviceToHost, s));
      PMT_HIP(hipStreamSynchronize(s));
      *v = *pinned;
      return PMT_OK;
    }
  }
}

// v -> host-visible memory (pinned): host[0] = value, then (after a system-scope fence) host[1] = seq, so a
// host thread that polls host[1] for the sequence number it expects reads a complete value in host[0]
// without a stream synchronisation, whatever the value is (NaN included)
__global__ void publish_kernel(const double* __restrict__ v, double seq, double* host) {
  if (threadIdx.x == 0) {
    volatile double* h = host;
    h[0] = v[0];
    __threadfence_system();
    h[1] = seq;
    __threadfence_system();
  }
}

int launch_publish(const double* v, double seq, double* host, hipStream_t s) {
  publish_kernel<<<1, 64, 0, s>>>(v, seq, host);
  return check_launch("publish_kernel");
}

template <typename Y>
int launch_dot_flat(long long n, const double* x, const Y* y, double* out, double* work, hipStream_t s) {
  if (n <= 0) return PMT_OK;
  const long long parts = cg_xr_parts(n);
  dot_flat<Y><<<(unsigned)parts, kReduceThreads, 0, s>>>(n, x, y, work);
  PMT_TRY(check_launch("dot_flat"));
  parts_stage2<<<1, kStage2Threads, 0, s>>>(work, parts, out, 0.0, nullptr);
  return check_launch("parts_stage2");
}
template int launch_dot_flat<double>(long long, const double*, const double*, double*, double*, hipStream_t);
template int launch_dot_flat<float>(long long, const double*, const float*, double*, double*, hipStream_t);

int launch_cg_x_update(long long n, const double* sc, const double* p, double* x, hipStream_t s) {
  cg_x_update<<<blocks_for(n, 256), 256, 0, s>>>(n, sc, p, x);
  return check_launch("cg_x_update");
}

template <typename Z>
int launch_cg_beta_update(long long n, double* sc, const double* q, const Z* z, double* p, double* work, double* x,
                          hipStream_t s) {
  if (n <= 0) return PMT_OK;
  const long long parts = cg_xr_parts(n);
  if (!cg_sums_inline(parts)) {
    PMT_TRY(launch_dot_flat(n, q, z, sc + 3, work, s));
    if (x)
      cg_p_update<Z, true><<<blocks_for(n, 256), 256, 0, s>>>(n, sc, z, p, x);
    else
      cg_p_update<Z, false><<<blocks_for(n, 256), 256, 0, s>>>(n, sc, z, p, nullptr);
    return check_launch("cg_p_update");
  }
  dot_flat<Z><<<(unsigned)parts, kReduceThreads, 0, s>>>(n, q, z, work);
  PMT_TRY(check_launch("dot_flat"));
  if (x)
    cg_p_update_parts<Z, true><<<(unsigned)parts, kReduceThreads, 0, s>>>(n, sc, work, (int)parts, z, p, x);
  else
    cg_p_update_parts<Z, false><<<(unsigned)parts, kReduceThreads, 0, s>>>(n, sc, work, (int)parts, z, p, nullptr);
  return check_launch("cg_p_update_parts");
}
template int launch_cg_beta_update<double>(long long, double*, const double*, const double*, double*, double*, double*,
                                           hipStream_t);
template int launch_cg_beta_update<float>(long long, double*, const double*, const float*, double*, double*, double*,
                                          hipStream_t);

int launch_scale_rsqrt(long long n, const double* sc, int k, const double* z, double* p, hipStream_t s) {
  scale_rsqrt<<<blocks_for(n, 256), 256, 0, s>>>(n, sc, k, z, p);
  return check_launch("scale_rsqrt");
}

__global__ void to_double_kernel(long long n, const float* __restrict__ x, double* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (double)x[i];
}

int launch_to_double(long long n, const float* x, double* y, hipStream_t s) {
  if (n <= 0) return PMT_OK;
  to_double_kernel<<<blocks_for(n, 256), 256, 0, s>>>(n, x, y);
  return check_launch("to_double_kernel");
}

__global__ void jacobi_apply_kernel(long long n, double w, const double* __restrict__ diag,
                                    const double* __restrict__ r, double* __restrict__ z) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) z[i] = w * r[i] / diag[i];
}

// ---------------------------------------------------------------------------------------------
// Dot products of k column pairs without a caller workspace: the per-block partial sums live in a
// file-scope device array (one copy per GPU, kept until the process ends).  Same grid, loop and
// summation order per column as dot_stage1<1> / dot_stage2<1>, so each column's result is bit-identical
// to pmt_dot's.  Every partial is written before it is read, so nothing needs clearing between calls.
constexpr int kNoAllocMaxCols = 8;
static __device__ __align__(256) double scratch[kNoAllocMaxCols * kReduceBlocks];  // 64 KiB
constexpr int kMaxDevices = 64;
static double* g_scratch_ptr[kMaxDevices];  // device address of `scratch`, per device
static std::mutex g_scratch_mu;

// Device address of this device's `scratch`, looked up once per device with that device current.
// In host code the array's name is only a host-side stand-in; kernels get this pointer.
static int scratch_for_current_device(double** out) {
  int dev = 0;
  PMT_TRY(hip_status(hipGetDevice(&dev), "hipGetDevice"));
  if (dev < 0 || dev >= kMaxDevices) return arg_error("pmt_dot_noalloc: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    PMT_TRY(hip_status(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)"));
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return PMT_OK;
}

__global__ void __launch_bounds__(kReduceThreads)
dot_cols_stage1(long long n, const double* __restrict__ x, const double* __restrict__ y,
                double* __restrict__ partial) {
  const long long off = (long long)blockIdx.y * n;
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    s = fma(x[off + i], y[off + i], s);
  const double r = block_sum(s);
  if (threadIdx.x == 0) partial[blockIdx.y * kReduceBlocks + blockIdx.x] = r;
}

__global__ void __launch_bounds__(kReduceThreads)
dot_cols_stage2(const double* __restrict__ partial, double* __restrict__ out) {
  const double* p = partial + (long long)blockIdx.x * kReduceBlocks;
  double s = 0.0;
  for (int b = threadIdx.x; b < kReduceBlocks; b += blockDim.x) s += p[b];
  const double r = block_sum(s);
  if (threadIdx.x == 0) out[blockIdx.x] = r;
}

// ---------------------------------------------------------------------------------------------
// Deflation of the preconditioned residual by a coarse space W (A-orthogonal projection):
// z <- z - W Einv (AW)^T z with Einv = (W^T A W)^-1, all in FP64.  Stage 1: per-block partial sums of the
// m dots AW_j . z (fixed grid, deterministic); stage 2: one block sums them in a fixed order and forms
// c = Einv d; then every entry of z loses sum_j W_j c_j.
__global__ void __launch_bounds__(kReduceThreads)
cs_dots_stage1(long long n, const double* __restrict__ AW, const double* __restrict__ z, double* __restrict__ partial) {
  const double* w = AW + (long long)blockIdx.y * n;
  double s = 0.0;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    s = fma(w[i], z[i], s);
  const double t = block_sum(s);
  if (threadIdx.x == 0) partial[blockIdx.y * kReduceBlocks + blockIdx.x] = t;
}

__global__ void __launch_bounds__(kReduceThreads)
cs_coef_kernel(int m, const double* __restrict__ partial, SmallMat Einv, double* __restrict__ c) {
  __shared__ double d[4];
  for (int j = 0; j < m; ++j) {
    double s = 0.0;
    for (int b = threadIdx.x; b < kReduceBlocks; b += blockDim.x) s += partial[j * kReduceBlocks + b];
    const double t = block_sum(s);
    if (threadIdx.x == 0) d[j] = t;
  }
  __syncthreads();
  if (threadIdx.x < m) {
    double v = 0.0;
    for (int k = 0; k < m; ++k) v = fma(Einv.e[threadIdx.x * m + k], d[k], v);
    c[threadIdx.x] = v;
  }
}

__global__ void cs_sub_kernel(long long n, int m, const double* __restrict__ W, const double* __restrict__ c,
                              double* __restrict__ z) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v = 0.0;
  for (int j = 0; j < m; ++j) v = fma(W[(long long)j * n + i], c[j], v);
  z[i] -= v;
}

int launch_coarse_correct(long long n, int m, const double* W, const double* AW, const SmallMat& Einv, double* buf,
                          double* z, hipStream_t s) {
  if (m <= 0) return PMT_OK;
  double* c = buf;
  double* partial = buf + 4;
  cs_dots_stage1<<<dim3(kReduceBlocks, m), kReduceThreads, 0, s>>>(n, AW, z, partial);
  PMT_TRY(check_launch("cs_dots_stage1"));
  cs_coef_kernel<<<1, kReduceThreads, 0, s>>>(m, partial, Einv, c);
  PMT_TRY(check_launch("cs_coef_kernel"));
  cs_sub_kernel<<<blocks_for(n, 256), 256, 0, s>>>(n, m, W, c, z);
  return check_launch("cs_sub_kernel");
}

int launch_fill(long long n, double v, double* y, hipStream_t s) {
  if (n <= 0) return PMT_OK;
  fill_kernel<<<blocks_for(n, 256), 256, 0, s>>>(n, v, y);
  return check_launch("fill_kernel");
}

}  // namespace pmt

using namespace pmt;

extern "C" {

const char* pmt_last_error(void) { return g_last_error.c_str(); }

int pmt_abi_version(void) { return 1; }

int pmt_reduce_work_size(void) { return 2 * kReduceBlocks; }

int pmt_powlaw_fwd(long long n, double a, double b, double p, const double* x, double* y, void* stream) {
  if (n < 0 || (n > 0 && (!x || !y))) return arg_error("pmt_powlaw_fwd: bad argument");
  if (n == 0) return PMT_OK;
  powlaw_fwd_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, a, b, p, powlaw_int_exponent(p), x, y);
  return check_launch("powlaw_fwd_kernel");
}

int pmt_powlaw_bwd(long long n, double c, double q, const double* x, const double* dy, double* dx, int accumulate,
                   void* stream) {
  if (n < 0 || (n > 0 && (!x || !dy || !dx))) return arg_error("pmt_powlaw_bwd: bad argument");
  if (n == 0) return PMT_OK;
  powlaw_bwd_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, c, q, powlaw_int_exponent(q), x, dy, dx,
                                                                         accumulate);
  return check_launch("powlaw_bwd_kernel");
}

int pmt_heaviside_fwd(long long n, double beta, double eta, const double* x, double* y, void* stream) {
  if (n < 0 || (n > 0 && (!x || !y))) return arg_error("pmt_heaviside_fwd: bad argument");
  if (n == 0) return PMT_OK;
  heaviside_fwd_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, beta, eta, x, y);
  return check_launch("heaviside_fwd_kernel");
}

int pmt_heaviside_bwd(long long n, double beta, double eta, const double* x, const double* dy, double* dx,
                      int accumulate, double* dbeta, void* stream) {
  if (n < 0 || (n > 0 && (!x || !dy || !dx))) return arg_error("pmt_heaviside_bwd: bad argument");
  if (n == 0) return PMT_OK;
  heaviside_bwd_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, beta, eta, x, dy, dx, accumulate,
                                                                           dbeta);
  return check_launch("heaviside_bwd_kernel");
}

int pmt_oc_work_size(void) { return 2 * kOcState + 2 * (kOcNodes + 1) * kReduceBlocks; }

int pmt_oc_step(long long n, const double* x, const double* dg, double xmin, double xmax, double move, double l1,
                double l2, double tol, double target, double* xnew, double* work, void* stream) {
  if (n <= 0 || !x || !dg || !xnew || !work || !(l1 >= 0.0) || !std::isfinite(l1) || !std::isfinite(l2) ||
      std::isnan(tol))
    return arg_error("pmt_oc_step: bad argument (finite interval with 0 <= l1)");
  hipStream_t s = (hipStream_t)stream;
  OcState* st[2] = {(OcState*)work, (OcState*)(work + kOcState)};
  double* partial[2] = {work + 2 * kOcState, work + 2 * kOcState + (kOcNodes + 1) * kReduceBlocks};
  static_assert(sizeof(OcState) <= kOcState * sizeof(double), "OC state");
  oc_init_kernel<<<1, 1, 0, s>>>(l1, l2, st[0]);
  PMT_TRY(check_launch("oc_init_kernel"));
  int steps = 0;
  for (double w = l2 - l1; w > tol && steps < 1100; w *= 0.5) ++steps;
  const int nb = (int)std::min<long long>(kReduceBlocks, (n + kReduceThreads - 1) / kReduceThreads);
  const int passes = std::max(1, (steps + 1 + kOcLv - 1) / kOcLv);  // one step to spare for the rounding of the halvings
  for (int p = 0; p < passes; ++p) {  // pass p leaves its state in st[p % 2] (pass 0: finds it there)
    oc_pass_kernel<<<(nb + kOcGroups - 1) / kOcGroups, kOcThreads, 0, s>>>(
        n, nb, x, dg, xmin, xmax, move, tol, target, p, st[p > 0 ? (p - 1) % 2 : 0], partial[(p + 1) % 2], st[p % 2],
        partial[p % 2]);
    PMT_TRY(check_launch("oc_pass_kernel"));
  }
  oc_last_kernel<<<1, kOcThreads, 0, s>>>(nb, tol, target, passes == 1, st[(passes - 1) % 2], partial[(passes - 1) % 2],
                                          st[0]);
  PMT_TRY(check_launch("oc_last_kernel"));
  oc_write_kernel<<<blocks_for(n, 256), 256, 0, s>>>(n, x, dg, xmin, xmax, move, st[0], xnew);
  return check_launch("oc_write_kernel");
}

int pmt_oc_update(long long n, const double* x, const double* dg, double xmin, double xmax, double move,
                  double lmid, double* xnew, double* sum_out, double* work, void* stream) {
  if (n <= 0 || !x || !dg || !xnew || !sum_out || !work || !(lmid > 0.0))
    return arg_error("pmt_oc_update: bad argument");
  hipStream_t s = (hipStream_t)stream;
  oc_update_kernel<<<kReduceBlocks, kReduceThreads, 0, s>>>(n, x, dg, xmin, xmax, move, lmid, xnew, work);
  PMT_TRY(check_launch("oc_update_kernel"));
  dot_stage2<1><<<1, kReduceThreads, 0, s>>>(work, sum_out);
  return check_launch("dot_stage2");
}

int pmt_axpby(long long n, double a, const double* x, double b, double* y, void* stream) {
  if (n < 0 || (n > 0 && !y)) return arg_error("pmt_axpby: bad argument");
  return launch_axpby(n, a, x, b, y, (hipStream_t)stream);
}

int pmt_lda_project(long long n, const double* b, const double* x, double sign, double* r, double* y, double* work,
                    void* stream) {
  if (n < 0 || !work || (n > 0 && (!b || !r || (y && !x)))) return arg_error("pmt_lda_project: bad argument");
  if (n == 0) return PMT_OK;
  hipStream_t s = (hipStream_t)stream;
  dot_stage1<2><<<kReduceBlocks, kReduceThreads, 0, s>>>(n, r, b, b, b, work);
  PMT_TRY(check_launch("dot_stage1<2>"));
  lda_project_kernel<<<(unsigned)cg_xr_parts(n), kReduceThreads, 0, s>>>(n, work, b, x, sign, r, y);
  return check_launch("lda_project_kernel");
}

int pmt_dot(long long n, const double* x, const double* y, double* out, double* work, void* stream) {
  if (n < 0 || !x || !y || !out || !work) return arg_error("pmt_dot: bad argument");
  return launch_dot(n, x, y, out, work, (hipStream_t)stream);
}

int pmt_jacobi_apply(long long n, double w, const double* diag, const double* r, double* z, void* stream) {
  if (n < 0 || (n > 0 && (!diag || !r || !z))) return arg_error("pmt_jacobi_apply: bad argument");
  if (n == 0) return PMT_OK;
  jacobi_apply_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, w, diag, r, z);
  return check_launch("jacobi_apply_kernel");
}

int pmt_dot_noalloc(int k, long long n, const double* x, const double* y, double* out, void* stream) {
  if (k < 1 || n < 0 || !x || !y || !out) return arg_error("pmt_dot_noalloc: bad argument");
  if (k > kNoAllocMaxCols)
    return arg_error(("pmt_dot_noalloc: k = " + std::to_string(k) + " column pairs exceed the maximum of " +
                      std::to_string(kNoAllocMaxCols) + " (the static scratch holds 8 x 1024 partial sums)").c_str());
  double* partial = nullptr;
  PMT_TRY(scratch_for_current_device(&partial));
  hipStream_t s = (hipStream_t)stream;
  dot_cols_stage1<<<dim3(kReduceBlocks, k), kReduceThreads, 0, s>>>(n, x, y, partial);
  PMT_TRY(check_launch("dot_cols_stage1"));
  dot_cols_stage2<<<k, kReduceThreads, 0, s>>>(partial, out);
  return check_launch("dot_cols_stage2");
}

int pmt_bc_split_ndof(int nelx, int nely, int nelz, int ndof, const uint8_t* bcmask, double bcdiag,
                      const double* rhs, double* rhs_loc, double* sol, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || ndof < 1 || ndof > 8 || !rhs || !rhs_loc || !sol)
    return arg_error("pmt_bc_split: bad argument");
  GridDims g = make_grid(nelx, nely, nelz);
  bc_split_kernel<<<blocks_for(g.nnodes * ndof, 256), 256, 0, (hipStream_t)stream>>>(g.nnodes, ndof, bcmask, bcdiag,
                                                                                     rhs, rhs_loc, sol);
  return check_launch("bc_split_kernel");
}

int pmt_bc_split(int nelx, int nely, int nelz, const uint8_t* bcmask, double bcdiag, const double* rhs,
                 double* rhs_loc, double* sol, void* stream) {
  return pmt_bc_split_ndof(nelx, nely, nelz, nelz > 0 ? 3 : 2, bcmask, bcdiag, rhs, rhs_loc, sol, stream);
}

int pmt_axpy_free_ndof(int nelx, int nely, int nelz, int ndof, const uint8_t* bcmask, double a, const double* x,
                       double* y, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || ndof < 1 || ndof > 8 || !x || !y) return arg_error("pmt_axpy_free: bad argument");
  GridDims g = make_grid(nelx, nely, nelz);
  axpy_free_kernel<<<blocks_for(g.nnodes * ndof, 256), 256, 0, (hipStream_t)stream>>>(g.nnodes, ndof, bcmask, a, x,
                                                                                      y);
  return check_launch("axpy_free_kernel");
}

int pmt_axpy_free(int nelx, int nely, int nelz, const uint8_t* bcmask, double a, const double* x, double* y,
                  void* stream) {
  return pmt_axpy_free_ndof(nelx, nely, nelz, nelz > 0 ? 3 : 2, bcmask, a, x, y, stream);
}

}  // extern "C"
