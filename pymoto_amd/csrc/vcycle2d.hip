// Q4 levels of the multigrid V-cycle with all smoothing sweeps of a visit in one launch.
//
// A 2D level is small (9,922 unknowns for the 120x40 beam): one launch per sweep, residual and transfer, 49 per
// CG iteration, cost far more than their work (3 us each against 0.1 us of arithmetic).  A block takes a square
// of nodes with a halo of one node per sweep, keeps its operator rows in registers (the 9 blocks of a node's
// row: formed from the 4 densities around it on the fine grid, read from the half stencil on the others) and
// the iterate in LDS, and runs the sweeps between barriers; the nodes of the halo are computed again by every
// block that needs them, one ring fewer per sweep.
//   down: first sweep from zero, the other sweeps, the residual and its restriction;
//   up:   prolongation of the correction, the sweeps.
// Blocks are up to 32 x 32 threads, one node each: with the default 5 sweeps 22 x 22 nodes (up) and 10 x 10
// coarse nodes (down) per block, so half of the arithmetic is the halo's - cheaper than a launch at small
// sizes; at large ones the operator rows are read once instead of once per sweep, which pays for a middle range
// of sweep counts (v2_ok).
// 120x40, 5 sweeps, 4 grids: 37 us per cycle in 7 launches (18 x 18 threads on the fine grid); about 150 us in 37
// launches of one sweep or transfer each.
#include "mg_impl.h"

namespace pmt {

namespace {

constexpr int kV2W = 32;  // threads per block side, at most
// LDS: two buffers of (W + 2)^2 values, a ring of zeros around the threads' nodes

template <typename T>
struct alignas(2 * sizeof(T)) V2 {
  T x, y;
};

template <typename T>
struct V2Op {
  const T* H;  // half stencil (levels >= 1), or null: the fine grid
  const T* dinv;
  const T* xe;
  const double* K0;
  const uint8_t* bcm;
  T bcdiag;
};

// the operator row of node (i, j): A[o][d][d2] towards the neighbour o = (dy + 1) * 3 + dx + 1; 0 outside the grid
template <typename T, bool FINE>
__device__ inline void v2_row(const V2Op<T>& op, const GridDims& g, int i, int j, T (&A)[9][2][2]) {
  const bool in = i >= 0 && i < g.nx && j >= 0 && j < g.ny;
  const int n = j * g.nx + i;
  if constexpr (FINE) {
    T x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ei = i - 1 + (e & 1), ej = j - 1 + (e >> 1);
      x[e] = (in && ei >= 0 && ei < g.ex && ej >= 0 && ej < g.ey) ? op.xe[ej * g.ex + ei] : (T)0;
    }
    const unsigned mk = in ? op.bcm[n] : 0u;
#pragma unroll
    for (int o = 0; o < 9; ++o) {
      const int dx = o % 3 - 1, dy = o / 3 - 1;
      const bool nb = in && i + dx >= 0 && i + dx < g.nx && j + dy >= 0 && j + dy < g.ny;
      const unsigned mm = nb ? op.bcm[n + dy * g.nx + dx] : 0u;
      T a[2][2] = {};
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // the elements (i - 1 + ex, j - 1 + ey) that hold both nodes
        const int ex = e & 1, ey = e >> 1, bx = dx + 1 - ex, by = dy + 1 - ey;
        if (bx < 0 || bx > 1 || by < 0 || by > 1) continue;
        const int ln = (1 - ex) + 2 * (1 - ey), lm = bx + 2 * by;
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
          for (int d2 = 0; d2 < 2; ++d2) a[d][d2] = fma((T)op.K0[(2 * ln + d) * 8 + 2 * lm + d2], x[e], a[d][d2]);
      }
      // Dirichlet rows and columns vanish, bcdiag on their diagonal
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int d2 = 0; d2 < 2; ++d2) {
          const bool cut = ((mk >> d) & 1u) || ((mm >> d2) & 1u);
          A[o][d][d2] = cut ? ((o == 4 && d == d2) ? op.bcdiag : (T)0) : a[d][d2];
        }
    }
  } else {
    const long long nn = g.nnodes;
#pragma unroll
    for (int o = 0; o < 9; ++o) {
      const int dx = o % 3 - 1, dy = o / 3 - 1;
      const bool nb = in && i + dx >= 0 && i + dx < g.nx && j + dy >= 0 && j + dy < g.ny;
      // centre and forward blocks at n, a backward one the transpose of the neighbour's forward block
      const int at = o >= 4 ? n : n + dy * g.nx + dx;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int d2 = 0; d2 < 2; ++d2) {
          const int c = o >= 4 ? ((o - 4) * 2 + d) * 2 + d2 : ((4 - o) * 2 + d2) * 2 + d;
          A[o][d][d2] = nb ? op.H[c * nn + at] : (T)0;
        }
    }
  }
}

// A u at the thread's node from the iterate in LDS
template <typename T>
__device__ inline V2<T> v2_apply(const T (&A)[9][2][2], const V2<T>* u, int c, int row) {
  V2<T> r = {(T)0, (T)0};
#pragma unroll
  for (int o = 0; o < 9; ++o) {
    const V2<T> v = u[c + (o / 3 - 1) * row + o % 3 - 1];
    r.x = fma(A[o][0][0], v.x, r.x);
    r.x = fma(A[o][0][1], v.y, r.x);
    r.y = fma(A[o][1][0], v.x, r.y);
    r.y = fma(A[o][1][1], v.y, r.y);
  }
  return r;
}

// sweeps k0 .. n-1 from the iterate u (register and LDS buffer `cur`): u + a_k D^-1 (b - A u) + b_k (u - u_prev)
template <typename T>
__device__ inline void v2_sweeps(const T (&A)[9][2][2], const Sweeps2& sw, int k0, V2<T> dv, V2<T> bv, V2<T>& u,
                                 V2<T> up, V2<T>* buf, int& cur, int c, int row) {
  for (int k = k0; k < sw.n; ++k) {
    const V2<T> au = v2_apply<T>(A, buf + cur, c, row);
    const T a = (T)sw.a[k], be = (T)sw.b[k];
    const V2<T> un = {u.x + a * dv.x * (bv.x - au.x) + be * (u.x - up.x),
                      u.y + a * dv.y * (bv.y - au.y) + be * (u.y - up.y)};
    up = u;
    u = un;
    cur = row * row - cur;
    buf[cur + c] = u;
    __syncthreads();
  }
}

template <typename T, bool FINE>
__global__ void __launch_bounds__(kV2W * kV2W)
v2_down_kernel(GridDims gf, GridDims gc, V2Op<T> op, Sweeps2 sw, int ct, const T* __restrict__ b, T* __restrict__ uo,
               T* __restrict__ bc) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  V2<T>* buf = (V2<T>*)lds;
  const int tx = threadIdx.x, ty = threadIdx.y, row = blockDim.x + 2, c = (ty + 1) * row + tx + 1;
  const int I0 = blockIdx.x * ct, J0 = blockIdx.y * ct;
  const int i = 2 * I0 - 1 - sw.n + tx, j = 2 * J0 - 1 - sw.n + ty;
  const bool in = i >= 0 && i < gf.nx && j >= 0 && j < gf.ny;
  const long long n = (long long)j * gf.nx + i;
  b += 2 * (long long)blockIdx.z * gf.nnodes;  // column
  uo += 2 * (long long)blockIdx.z * gf.nnodes;
  bc += 2 * (long long)blockIdx.z * gc.nnodes;
  for (int q = ty * blockDim.x + tx; q < 2 * row * row; q += blockDim.x * blockDim.x) buf[q] = {(T)0, (T)0};
  T A[9][2][2];
  v2_row<T, FINE>(op, gf, i, j, A);
  const V2<T> zero = {(T)0, (T)0};
  const V2<T> bv = in ? *(const V2<T>*)(b + 2 * n) : zero, dv = in ? *(const V2<T>*)(op.dinv + 2 * n) : zero;
  const T a0 = (T)sw.a[0];
  V2<T> u = {a0 * dv.x * bv.x, a0 * dv.y * bv.y};
  int cur = 0;
  __syncthreads();
  buf[c] = u;
  __syncthreads();
  v2_sweeps<T>(A, sw, 1, dv, bv, u, zero, buf, cur, c, row);
  if (in && i >= 2 * I0 && i < 2 * (I0 + ct) && j >= 2 * J0 && j < 2 * (J0 + ct)) *(V2<T>*)(uo + 2 * n) = u;
  const V2<T> au = v2_apply<T>(A, buf + cur, c, row);
  cur = row * row - cur;
  buf[cur + c] = in ? V2<T>{bv.x - au.x, bv.y - au.y} : zero;
  __syncthreads();
  // fine node (2 I, 2 J): the coarse right-hand side from the 3 x 3 residuals around it
  if ((i & 1) || (j & 1)) return;
  const int I = i >> 1, J = j >> 1;
  if (I < I0 || I >= I0 + ct || I >= gc.nx || J < J0 || J >= J0 + ct || J >= gc.ny) return;
  V2<T> s = zero;
#pragma unroll
  for (int o = 0; o < 9; ++o) {
    const T w = (T)((o % 3 == 1 ? 1.0 : 0.5) * (o / 3 == 1 ? 1.0 : 0.5));
    const V2<T> r = buf[cur + c + (o / 3 - 1) * row + o % 3 - 1];
    s.x = fma(w, r.x, s.x);
    s.y = fma(w, r.y, s.y);
  }
  *(V2<T>*)(bc + 2 * ((long long)J * gc.nx + I)) = s;
}

template <typename T, bool FINE>
__global__ void __launch_bounds__(kV2W * kV2W)
v2_up_kernel(GridDims gf, GridDims gc, V2Op<T> op, Sweeps2 sw, int t, const T* __restrict__ b, const T* __restrict__ ui,
             const T* __restrict__ ec, T* __restrict__ uo) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  V2<T>* buf = (V2<T>*)lds;
  const int tx = threadIdx.x, ty = threadIdx.y, row = blockDim.x + 2, c = (ty + 1) * row + tx + 1;
  const int i = blockIdx.x * t - sw.n + tx, j = blockIdx.y * t - sw.n + ty;
  const bool in = i >= 0 && i < gf.nx && j >= 0 && j < gf.ny;
  const long long n = (long long)j * gf.nx + i;
  b += 2 * (long long)blockIdx.z * gf.nnodes;  // column
  ui += 2 * (long long)blockIdx.z * gf.nnodes;
  uo += 2 * (long long)blockIdx.z * gf.nnodes;
  ec += 2 * (long long)blockIdx.z * gc.nnodes;
  for (int q = ty * blockDim.x + tx; q < 2 * row * row; q += blockDim.x * blockDim.x) buf[q] = {(T)0, (T)0};
  T A[9][2][2];
  v2_row<T, FINE>(op, gf, i, j, A);
  const V2<T> zero = {(T)0, (T)0};
  const V2<T> bv = in ? *(const V2<T>*)(b + 2 * n) : zero, dv = in ? *(const V2<T>*)(op.dinv + 2 * n) : zero;
  V2<T> u = zero;
  if (in) {
    u = *(const V2<T>*)(ui + 2 * n);
    // bilinear interpolation: along an axis of even fine index the second corner repeats the first with weight 0
    const int oi = i & 1, oj = j & 1;
    const T wx[2] = {(T)(oi ? 0.5 : 1.0), (T)(oi ? 0.5 : 0.0)}, wy[2] = {(T)(oj ? 0.5 : 1.0), (T)(oj ? 0.5 : 0.0)};
    V2<T> e = zero;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const T w = wx[q & 1] * wy[q >> 1];
      const V2<T> v = *(const V2<T>*)(ec + 2 * ((long long)((j >> 1) + (q >> 1) * oj) * gc.nx + (i >> 1) + (q & 1) * oi));
      e.x = fma(w, v.x, e.x);
      e.y = fma(w, v.y, e.y);
    }
    u.x += e.x;
    u.y += e.y;
  }
  int cur = 0;
  __syncthreads();
  buf[c] = u;
  __syncthreads();
  v2_sweeps<T>(A, sw, 0, dv, bv, u, zero, buf, cur, c, row);
  if (in && tx >= sw.n && tx < sw.n + t && ty >= sw.n && ty < sw.n + t) *(V2<T>*)(uo + 2 * n) = u;
}

template <typename T>
V2Op<T> v2_op(const pmt_mg* mg, const Level& L, const LevelBuf<T>& B, bool fine, const T* xe) {
  return V2Op<T>{fine ? nullptr : B.H, B.dinv, xe, mg->K0, mg->bcm, (T)mg->bcdiag};
}

}  // namespace

// Up to how many thousand nodes (0: any number) a level's visit of 1 to 10 sweeps goes in two launches, on the fine
// grid and on the others, in FP64 and FP32.  Small levels save the launches and win with every sweep count.  On a
// grid that fills the chip the halo counts: a launch per sweep computes a node once per sweep, a block here
// (32 / (32 - 2 n))^2 times, which the operator rows kept in registers pay for in the middle of the range only, and
// least where a launch per sweep forms them from the densities or reads half the bytes.  Microseconds saved by the two
// launches, at 148,000 / 263,000 / 1,051,000 nodes (fine) and 37,000 / 263,000 / 1,051,000 (stencil):
//   sweeps                  1              2               5                8                10
//   FP64 fine          4/ -1/ -21     11/  6/  -8     20/ 13/  10     18/ -8/ -106    -13/-85/ -423
//   FP32 fine          2/ -4/ -28     10/  1/ -19     18/  9/  -9     17/ -7/ -107     -6/-65/ -381
//   FP64 stencil       3/-11/ -33      9/  4/  15     22/ 44/ 137     40/ 52/   97     23/  5/ -194
//   FP32 stencil       3/-11/ -34      8/ -4/ -10     27/ 13/  40     37/  4/   -4     31/-35/ -214
// (a V-cycle of a 1024x1024 grid with 5 sweeps takes 318 us in FP64).  In FP64 2 to 6 sweeps of the fine grid lose up to
// 49 us between 0.6 and 2.4 million nodes and gain 29 to 159 us at 4.2 million or with 4 and more columns.  The fine
// operator takes one column per launch, the stencils all columns of a block, so there the limit is one of all columns' nodes.
bool v2_ok(const pmt_mg* mg, int l, bool fp32, int cols) {
  static const int limit[2][2][kV2MaxSweeps] = {
      {{150, 0, 0, 0, 0, 0, 265, 150, 150, 70}, {100, 0, 0, 0, 0, 0, 0, 0, 0, 265}},
      {{150, 265, 265, 265, 265, 265, 265, 150, 150, 70}, {70, 150, 0, 0, 0, 0, 0, 0, 150, 100}}};
  const Level& L = mg->L[l];
  if (mg->dim != 2 || L.steps < 1 || L.steps > kV2MaxSweeps) return false;
  const int most = limit[fp32 ? 1 : 0][l > 0 ? 1 : 0][L.steps - 1];
  return most == 0 || L.g.nnodes * (l > 0 ? cols : 1) <= 1000LL * most;
}

// Threads per block side for a grid of nx x ny outputs, `out(w)` of them per side: the fewest wavefronts per
// compute unit.  A sweep is bound by the LDS reads of a block's wavefronts, so while the blocks do not fill
// the chip small ones are faster, although most of their nodes are halo; beyond, large ones compute less.
template <typename F>
int v2_side(int nx, int ny, int cols, F out) {
  int best = kV2W;
  long long cost = 0;
  for (int w = kV2W; w >= 12; w -= 2) {
    const int t = out(w);
    if (t < 1) break;
    const long long blocks = (long long)cols * ((nx + t - 1) / t) * ((ny + t - 1) / t);
    const long long c = (blocks + device_cu_count() - 1) / device_cu_count() * ((w * w + 63) / 64);
    if (w == kV2W || c < cost) {
      cost = c;
      best = w;
    }
  }
  return best;
}

template <typename T>
size_t v2_lds(int w) {
  return 2 * sizeof(V2<T>) * (w + 2) * (w + 2);
}

template <typename T>
int launch_v2_down(pmt_mg* mg, int l, const T* xe, const Sweeps2& sw, const T* b, T* u, T* bc, hipStream_t s,
                   int cols) {
  Level& L = mg->L[l];
  const GridDims& gc = mg->L[l + 1].g;
  auto coarse = [&](int w) { return (w - 2 - 2 * sw.n) / 2; };  // 2 ct + 1 residuals per side and the halo
  const int w = v2_side(gc.nx, gc.ny, cols, coarse), ct = coarse(w);
  const dim3 grid((gc.nx + ct - 1) / ct, (gc.ny + ct - 1) / ct, cols), block(w, w);
  const V2Op<T> op = v2_op<T>(mg, L, L.buf<T>(), l == 0, xe);
  if (l == 0)
    v2_down_kernel<T, true><<<grid, block, v2_lds<T>(w), s>>>(L.g, gc, op, sw, ct, b, u, bc);
  else
    v2_down_kernel<T, false><<<grid, block, v2_lds<T>(w), s>>>(L.g, gc, op, sw, ct, b, u, bc);
  return check_launch("v2_down_kernel");
}

template <typename T>
int launch_v2_up(pmt_mg* mg, int l, const T* xe, const Sweeps2& sw, const T* b, const T* ui, const T* ec, T* uo,
                 hipStream_t s, int cols) {
  Level& L = mg->L[l];
  auto nodes = [&](int w) { return w - 2 * sw.n; };
  const int w = v2_side(L.g.nx, L.g.ny, cols, nodes), t = nodes(w);
  const dim3 grid((L.g.nx + t - 1) / t, (L.g.ny + t - 1) / t, cols), block(w, w);
  const V2Op<T> op = v2_op<T>(mg, L, L.buf<T>(), l == 0, xe);
  if (l == 0)
    v2_up_kernel<T, true><<<grid, block, v2_lds<T>(w), s>>>(L.g, mg->L[l + 1].g, op, sw, t, b, ui, ec, uo);
  else
    v2_up_kernel<T, false><<<grid, block, v2_lds<T>(w), s>>>(L.g, mg->L[l + 1].g, op, sw, t, b, ui, ec, uo);
  return check_launch("v2_up_kernel");
}

#define PMT_V2_INST(T)                                                                                              \
  template int launch_v2_down<T>(pmt_mg*, int, const T*, const Sweeps2&, const T*, T*, T*, hipStream_t, int);        \
  template int launch_v2_up<T>(pmt_mg*, int, const T*, const Sweeps2&, const T*, const T*, const T*, T*,             \
                               hipStream_t, int);
PMT_V2_INST(double)
PMT_V2_INST(float)
#undef PMT_V2_INST

}  // namespace pmt
