// Scalar (one unknown per node) finite-element operators for AssemblePoisson (thermal conduction,
// electric permittivity; pymoto/modules/assembly.py:523-560) and a geometric-multigrid PCG for them.
//
// Operator: K(x) = sum_e x_e P0 with P0 the (2^D x 2^D) element matrix, Dirichlet rows and columns
// zeroed and bcdiag on their diagonal (AssembleGeneral, assembly.py:209-230,245-296), applied matrix
// free and node-centric: thread n gathers the 2^D elements around node n and the 3^D neighbour values
// (no scatter, no atomics, fixed summation order).
//
// Multigrid: every level has its operator as a node stencil S[c][node] (3^D coefficients, c =
// (dz+1)*9 + (dy+1)*3 + dx+1, coefficient-major so a wave reads consecutive nodes of one coefficient);
// level 0 from the elements (and applied from them where the element matrix allows), level l+1 as the
// Galerkin product R^T S_l R with the trilinear (bilinear) transfer of GeometricMultigrid.setup_interpolation
// (pymoto/solvers/iterative.py:178-220, weights 1, 1/2, 1/4, 1/8), which keeps the reference's Dirichlet
// diagonal inside the coarse operators
// (iterative.py:173).  V-cycle: damped-Jacobi pre-smoothing whose first sweep starts from zero, residual,
// restriction, inner level, prolongation, post-smoothing (iterative.py:222-256); the coarsest grid is
// solved with an explicit FP64 inverse (blocked Gauss-Jordan of coarse.hip).  The CG loop follows
// CG.solve for one right-hand side (iterative.py:340-403).
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>
#include <vector>

#include "launch.h"

namespace pmt {

namespace {

constexpr int kScalarMaxLevels = 12;

template <int DIM>
struct SCfg {
  static constexpr int NN = 1 << DIM;           // nodes per element
  static constexpr int NS = DIM == 3 ? 27 : 9;  // stencil coefficients per node
};

__device__ inline void node_ijk(const GridDims& g, long long n, int& i, int& j, int& k) {
  i = (int)(n % g.nx);
  const long long t = n / g.nx;
  j = (int)(t % g.ny);
  k = (int)(t / g.ny);
}

// ---------------------------------------------------------------------------------------------
// fine operator from the elements
// MODE 0: y = K u ; MODE 1: y = b - K u
template <int DIM, int MODE>
__global__ void __launch_bounds__(256)
scalar_apply_kernel(GridDims g, const double* __restrict__ P0, const double* __restrict__ xe,
                    const uint8_t* __restrict__ bcm, double bcdiag, const double* __restrict__ u,
                    const double* __restrict__ b, double* __restrict__ y) {
  constexpr int NN = SCfg<DIM>::NN;
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= g.nnodes) return;
  int i, j, k;
  node_ijk(g, n, i, j, k);
  double acc = 0.0;
  if (bcm && (bcm[n] & 1u)) {
    acc = bcdiag * u[n];
  } else {
    // elements (ei, ej, ek) = (i - 1 + ox, ...), local index of node n inside it a = (1-ox) + 2(1-oy) + 4(1-oz)
#pragma unroll
    for (int oz = 0; oz < (DIM == 3 ? 2 : 1); ++oz)
#pragma unroll
      for (int oy = 0; oy < 2; ++oy)
#pragma unroll
        for (int ox = 0; ox < 2; ++ox) {
          const int ei = i - 1 + ox, ej = j - 1 + oy, ek = DIM == 3 ? k - 1 + oz : 0;
          if (ei < 0 || ei >= g.ex || ej < 0 || ej >= g.ey || ek < 0 || ek >= g.ez) continue;
          const int a = (1 - ox) + 2 * (1 - oy) + (DIM == 3 ? 4 * (1 - oz) : 0);
          const double xv = xe[((long long)ek * g.ey + ej) * g.ex + ei];
          double s = 0.0;
#pragma unroll
          for (int c = 0; c < NN; ++c) {
            const long long m = ((long long)(ek + ((c >> 2) & 1)) * g.ny + (ej + ((c >> 1) & 1))) * g.nx + (ei + (c & 1));
            const double um = (bcm && (bcm[m] & 1u)) ? 0.0 : u[m];
            s = fma(P0[a * NN + c], um, s);
          }
          acc = fma(xv, s, acc);
        }
  }
  y[n] = MODE == 0 ? acc : b[n] - acc;
}

// diag(K)
template <int DIM>
__global__ void scalar_diag_kernel(GridDims g, const double* __restrict__ P0, const double* __restrict__ xe,
                                   const uint8_t* __restrict__ bcm, double bcdiag, double* __restrict__ d) {
  constexpr int NN = SCfg<DIM>::NN;
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= g.nnodes) return;
  int i, j, k;
  node_ijk(g, n, i, j, k);
  if (bcm && (bcm[n] & 1u)) {
    d[n] = bcdiag;
    return;
  }
  double acc = 0.0;
  for (int oz = 0; oz < (DIM == 3 ? 2 : 1); ++oz)
    for (int oy = 0; oy < 2; ++oy)
      for (int ox = 0; ox < 2; ++ox) {
        const int ei = i - 1 + ox, ej = j - 1 + oy, ek = DIM == 3 ? k - 1 + oz : 0;
        if (ei < 0 || ei >= g.ex || ej < 0 || ej >= g.ey || ek < 0 || ek >= g.ez) continue;
        const int a = (1 - ox) + 2 * (1 - oy) + (DIM == 3 ? 4 * (1 - oz) : 0);
        acc = fma(xe[((long long)ek * g.ey + ej) * g.ex + ei], P0[a * NN + a], acc);
      }
  d[n] = acc;
}

// dx_e (+)= alpha * u_e^T P0 v_e, Dirichlet entries of u and v zeroed (assembly.py:298-315)
template <int DIM>
__global__ void __launch_bounds__(256)
scalar_sens_kernel(GridDims g, const double* __restrict__ P0, const uint8_t* __restrict__ bcm,
                   const double* __restrict__ u, const double* __restrict__ v, double alpha,
                   double* __restrict__ dx, int accumulate) {
  constexpr int NN = SCfg<DIM>::NN;
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= g.nel) return;
  const int ei = (int)(e % g.ex);
  const long long t = e / g.ex;
  const int ej = (int)(t % g.ey);
  const int ek = (int)(t / g.ey);
  double ue[NN], ve[NN];
#pragma unroll
  for (int a = 0; a < NN; ++a) {
    const long long m = ((long long)(ek + ((a >> 2) & 1)) * g.ny + (ej + ((a >> 1) & 1))) * g.nx + (ei + (a & 1));
    const bool fixed = bcm && (bcm[m] & 1u);
    ue[a] = fixed ? 0.0 : u[m];
    ve[a] = fixed ? 0.0 : v[m];
  }
  double s = 0.0;
#pragma unroll
  for (int a = 0; a < NN; ++a) {
    double r = 0.0;
#pragma unroll
    for (int c = 0; c < NN; ++c) r = fma(P0[a * NN + c], ve[c], r);
    s = fma(ue[a], r, s);
  }
  dx[e] = accumulate ? fma(alpha, s, dx[e]) : alpha * s;
}

// ---------------------------------------------------------------------------------------------
// stencils

// level-0 stencil from the elements: S[c][n] = sum over elements e around n of x_e P0[a(n,e)][b] for the
// neighbour m = corner b of e at offset c; Dirichlet rows: bcdiag on the centre only; Dirichlet columns 0
template <int DIM>
__global__ void scalar_stencil_fine_kernel(GridDims g, const double* __restrict__ P0, const double* __restrict__ xe,
                                           const uint8_t* __restrict__ bcm, double bcdiag, double* __restrict__ S) {
  constexpr int NN = SCfg<DIM>::NN, NS = SCfg<DIM>::NS;
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= g.nnodes) return;
  int i, j, k;
  node_ijk(g, n, i, j, k);
  double st[NS];
#pragma unroll
  for (int c = 0; c < NS; ++c) st[c] = 0.0;
  if (bcm && (bcm[n] & 1u)) {
    st[NS / 2] = bcdiag;
  } else {
#pragma unroll
    for (int oz = 0; oz < (DIM == 3 ? 2 : 1); ++oz)
#pragma unroll
      for (int oy = 0; oy < 2; ++oy)
#pragma unroll
        for (int ox = 0; ox < 2; ++ox) {
          const int ei = i - 1 + ox, ej = j - 1 + oy, ek = DIM == 3 ? k - 1 + oz : 0;
          if (ei < 0 || ei >= g.ex || ej < 0 || ej >= g.ey || ek < 0 || ek >= g.ez) continue;
          const int a = (1 - ox) + 2 * (1 - oy) + (DIM == 3 ? 4 * (1 - oz) : 0);
          const double xv = xe[((long long)ek * g.ey + ej) * g.ex + ei];
#pragma unroll
          for (int b = 0; b < NN; ++b) {
            const int bx = b & 1, by = (b >> 1) & 1, bz = DIM == 3 ? (b >> 2) & 1 : 0;
            const long long m = ((long long)(ek + bz) * g.ny + (ej + by)) * g.nx + (ei + bx);
            if (bcm && (bcm[m] & 1u)) continue;
            // offset of m from n per axis: (e + corner) - node = corner - (1 - o)
            const int dx = bx - (1 - ox), dy = by - (1 - oy), dz = DIM == 3 ? bz - (1 - oz) : 0;
            const int c = DIM == 3 ? (dz + 1) * 9 + (dy + 1) * 3 + (dx + 1) : (dy + 1) * 3 + (dx + 1);
            st[c] = fma(xv, P0[a * NN + b], st[c]);
          }
        }
  }
#pragma unroll
  for (int c = 0; c < NS; ++c) S[(long long)c * g.nnodes + n] = st[c];
}

// Galerkin coarse stencil Sc = R^T Sf R, one axis at a time: the transfer is a product of 1-D ones (weights 1 at
// the fine image 2 I, 1/2 beside it), so coarsening x, then y, then z gives the same sums in 13 multiply-adds per
// axis and pair of the other offsets instead of 13^3 for all.  Along the axis, with i = 2 I + di, j = 2 (I + c') +
// dj and weights w(di) w(dj): Sc[c'][I] = sum over the pairs with |j - i| <= 1 (7 for c' = 0, 3 for c' = +-1) of
// w w S[j - i][i].  A stencil entry that points outside the grid is 0 by construction.  One thread per coarse
// node; in: n x m x q nodes (x, y, z), out: the same with the axis halved.
// 80x80x48: 66 us for the three axes of the first level (1.6 ms as one kernel of nested pair loops).
// The three passes take a slab of coarse planes (rows in 2D) at a time, so that what lies between them stays
// small (kSlab): S and T are the slab's part of arrays whose coefficients lie ss and ts apart, nl planes of the last
// axis; the last axis itself is halved from its plane `first` (the image of the slab's first coarse plane) on to cl.
template <int DIM, int AXIS>
__global__ void __launch_bounds__(256)
scalar_coarsen_kernel(int nx, int ny, int nl, int first, int cl, const double* __restrict__ S, long long ss,
                      double* __restrict__ T, long long ts) {
  constexpr int NS = SCfg<DIM>::NS, ST = AXIS == 0 ? 1 : AXIS == 1 ? 3 : 9;  // stride of the axis offset in c
  constexpr bool LAST = AXIS == DIM - 1;
  if (DIM == 2) ny = nl;
  const int nz = DIM == 3 ? nl : 1;
  const int cx = AXIS == 0 ? (nx + 1) / 2 : nx, cy = AXIS == 1 ? (LAST ? cl : (ny + 1) / 2) : ny, cz = AXIS == 2 ? cl : nz;
  const long long N = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (N >= (long long)cx * cy * cz) return;
  const int I = (int)(N % cx), J = (int)((N / cx) % cy), K = (int)(N / ((long long)cx * cy));
  const int pos = 2 * (AXIS == 0 ? I : AXIS == 1 ? J : K) + (LAST ? first : 0), len = AXIS == 0 ? nx : AXIS == 1 ? ny : nz;
  const long long at = ((long long)(AXIS == 2 ? pos : K) * ny + (AXIS == 1 ? pos : J)) * nx + (AXIS == 0 ? pos : I);
  const long long step = AXIS == 0 ? 1 : AXIS == 1 ? nx : (long long)nx * ny;
  const bool in[3] = {pos > 0, true, pos + 1 < len};
#pragma unroll
  for (int o = 0; o < NS / 3; ++o) {  // the offsets along the other axes
    const int c0 = AXIS == 0 ? 3 * o : AXIS == 1 ? (o / 3) * 9 + o % 3 : o;
    double v[3][3];  // [di + 1][j - i + 1]
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int f = 0; f < 3; ++f) v[d][f] = in[d] ? S[(c0 + f * ST) * ss + at + (d - 1) * step] : 0.0;
#pragma unroll
    for (int cp = -1; cp <= 1; ++cp) {
      double acc = 0.0;
#pragma unroll
      for (int di = -1; di <= 1; ++di)
#pragma unroll
        for (int dj = -1; dj <= 1; ++dj) {
          const int f = 2 * cp + dj - di;
          if (f < -1 || f > 1) continue;
          acc = fma((di ? 0.5 : 1.0) * (dj ? 0.5 : 1.0), v[di + 1][f + 1], acc);
        }
      T[(c0 + (cp + 1) * ST) * ts + N] = acc;
    }
  }
}

// One operator pass on a level.
//   y = A v (kApply), b - A v (kResidual) or v + w D^-1 (b - A v) (kSweep) with the iterate
//   v = u (kPlain), w D^-1 b (kFirst: the first sweep from zero is formed on the way, so it and the second are one
//   pass) or u + R e (kCorrected: the prolongation likewise); kApply with r: also the block's parts of v.y and v.r.
// The operator: the stencil S of the level, or (ELEM, the fine grid when P0[a][b] depends on a ^ b only, as every
// box element of an isotropic material has it) the densities around the node.  Then the row is p[0] times the
// sum of the node's densities at the centre, p[a] times the sum of those of the elements shared with the neighbour
// elsewhere: 9 products per element layer and node plane, and the 27 coefficients (69 MB at 80x80x48, read by
// each of 5 passes per V-cycle) are not read at all.
// A block of 32 x 8 threads takes NZ node planes; v with a ring of one node around them (zero outside the grid
// and, with ELEM, on Dirichlet nodes) is staged in LDS at once, every load in flight together: the grids are
// small, so a block's time is its chain of memory latencies (walking the planes with a prefetch of one took
// 12 us for a fine sweep at 80x80x48 and 9 us at 20x20x12).  NZ falls with the grid until the blocks fill the
// chip (level_planes).
// 9 us for a fine sweep and 4-5 us for one of the levels below at 80x80x48; with the prolongation 18 us.
enum { kApply = 0, kResidual = 1, kSweep = 2 };
enum { kPlain = 0, kFirst = 1, kCorrected = 2 };

struct LevelArgs {
  const double* S;     // stencil
  const double* xe;    // ELEM: densities, the 8 values of P0, mask and its diagonal
  double p[8];
  const uint8_t* bcm;
  double bcdiag;
  const double *dinv, *u, *b, *e, *r;
  double omega;
  double* y;
  double* parts;       // kApply: [v.y of each block][v.r of each block]
  int cnx, cny;        // kCorrected: nodes of the coarse grid of e
};

template <int DIM, bool ELEM, int SRC, int MODE, int NZ>
__global__ void __launch_bounds__(256)
scalar_level_kernel(GridDims g, int tiles_x, int tiles_y, LevelArgs A) {
  constexpr int TX = 32, TY = 8, LX = TX + 2, LP = LX * (TY + 2), NS = SCfg<DIM>::NS;
  constexpr int NP = DIM == 3 ? NZ + 2 : 1, PER = (NP * LP + 255) / 256;  // staged planes, cells per thread
  __shared__ double lds[NP * LP];
  const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
  const int tile = blockIdx.x % (tiles_x * tiles_y), chunk = blockIdx.x / (tiles_x * tiles_y);
  const int i0 = (tile % tiles_x) * TX, j0 = (tile / tiles_x) * TY;
  const int k0 = chunk * NZ;
  const int i = i0 + tx, j = j0 + ty;
  const bool own = i < g.nx && j < g.ny;
  const int nxy = g.nx * g.ny;
  // the iterate at node (ii, jj, kk) of the grid
  auto value = [&](int ii, int jj, int kk) -> double {
    const int n = kk * nxy + jj * g.nx + ii;
    if (SRC == kFirst) return A.omega * A.dinv[n] * A.b[n];
    double v = A.u[n];
    if (SRC == kCorrected) {
      const int oi = ii & 1, oj = jj & 1, ok = DIM == 3 ? kk & 1 : 0;
      double s = 0.0;
#pragma unroll
      for (int c = 0; c < (1 << DIM); ++c) {  // the second corner of an even index repeats the first, weight 0
        const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
        const double w = (oi ? 0.5 : 1.0 - cx) * (oj ? 0.5 : 1.0 - cy) * (ok ? 0.5 : 1.0 - cz);
        s = fma(w, A.e[(((kk >> 1) + cz * ok) * A.cny + (jj >> 1) + cy * oj) * A.cnx + (ii >> 1) + cx * oi], s);
      }
      v += s;
    }
    return v;
  };
  auto masked = [&](int n) { return ELEM && A.bcm && (A.bcm[n] & 1u); };
  {
    double v[PER];
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      const int q = tid + 256 * t, pl = q / LP, cell = q % LP;
      const int ii = i0 - 1 + cell % LX, jj = j0 - 1 + cell / LX, kk = DIM == 3 ? k0 - 1 + pl : 0;
      // no branch around a load (the loads of all cells are to be in flight together): a cell outside reads the
      // nearest node and drops it
      const int ci = min(max(ii, 0), g.nx - 1), cj = min(max(jj, 0), g.ny - 1), ck = min(max(kk, 0), g.nz - 1);
      const unsigned m = ELEM && A.bcm ? A.bcm[ck * nxy + cj * g.nx + ci] & 1u : 0u;
      const double f = value(ci, cj, ck);
      v[t] = (ii == ci && jj == cj && kk == ck && !m) ? f : 0.0;
    }
#pragma unroll
    for (int t = 0; t < PER; ++t)
      if (tid + 256 * t < NP * LP) lds[tid + 256 * t] = v[t];
  }
  const int c = (ty + 1) * LX + tx + 1;
  // the 3 x 3 values around the node in staged plane pl
  auto window = [&](int pl, double (&w)[9]) {
#pragma unroll
    for (int o = 0; o < 9; ++o) w[o] = lds[pl * LP + c + (o / 3 - 1) * LX + o % 3 - 1];
  };
  // ELEM: the 4 densities of element layer kk around node (i, j)
  auto layer = [&](int kk, double (&x)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ei = i - 1 + (e & 1), ej = j - 1 + (e >> 1);
      const int ci = min(max(ei, 0), g.ex - 1), cj = min(max(ej, 0), g.ey - 1), ck = min(max(kk, 0), g.ez - 1);
      const double f = A.xe[((long long)ck * g.ey + cj) * g.ex + ci];
      x[e] = (ei == ci && ej == cj && kk == ck) ? f : 0.0;
    }
  };
  // the sums of x v over a plane by class: centre, x neighbours, y neighbours, diagonal
  auto classes = [](const double (&x)[4], const double (&v)[9], double (&s)[4]) {
    s[0] = (x[0] + x[1] + x[2] + x[3]) * v[4];
    s[1] = fma(x[0] + x[2], v[3], (x[1] + x[3]) * v[5]);
    s[2] = fma(x[0] + x[1], v[1], (x[2] + x[3]) * v[7]);
    s[3] = fma(x[0], v[0], fma(x[1], v[2], fma(x[2], v[6], x[3] * v[8])));
  };
  double sum_y = 0.0, sum_r = 0.0;
  auto finish = [&](int kk, double av, double centre) {
    if (!own || kk >= g.nz) return;
    const int n = kk * nxy + j * g.nx + i;
    if (masked(n)) {
      centre = value(i, j, kk);
      av = A.bcdiag * centre;
    }
    if (MODE == kApply) {
      A.y[n] = av;
      if (A.r) {
        sum_y = fma(centre, av, sum_y);
        sum_r = fma(centre, A.r[n], sum_r);
      }
    } else if (MODE == kResidual) {
      A.y[n] = A.b[n] - av;
    } else {
      A.y[n] = centre + A.omega * A.dinv[n] * (A.b[n] - av);
    }
  };
  if constexpr (DIM == 2) {
    __syncthreads();
    double w[9], av = 0.0;
    window(0, w);
    if constexpr (ELEM) {
      double x[4], s[4];
      layer(0, x);
      classes(x, w, s);
#pragma unroll
      for (int a = 0; a < 4; ++a) av = fma(A.p[a], s[a], av);
    } else if (own) {
#pragma unroll
      for (int o = 0; o < 9; ++o) av = fma(A.S[(long long)o * g.nnodes + j * g.nx + i], w[o], av);
    }
    finish(0, av, w[4]);
  } else if constexpr (ELEM) {
    // element layer kk joins planes kk and kk + 1: each gets p[0..3] of its own plane and p[4..7] of the other
    double x[NZ + 1][4];
#pragma unroll
    for (int l = 0; l <= NZ; ++l) layer(k0 - 1 + l, x[l]);
    __syncthreads();
    double lo[9], hi[9], s[4], t[4], acc = 0.0;
    window(0, lo);
#pragma unroll
    for (int l = 0; l <= NZ; ++l) {
      window(l + 1, hi);
      classes(x[l], lo, s);
      classes(x[l], hi, t);
      double up = 0.0;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        acc = fma(A.p[a], s[a], fma(A.p[4 + a], t[a], acc));
        up = fma(A.p[a], t[a], fma(A.p[4 + a], s[a], up));
      }
      if (l > 0) finish(k0 - 1 + l, acc, lo[4]);
      acc = up;
#pragma unroll
      for (int o = 0; o < 9; ++o) lo[o] = hi[o];
    }
  } else {
    double w[3][9], cf[2][NS];
    auto coefficients = [&](int kk, double (&d)[NS]) {
#pragma unroll
      for (int o = 0; o < NS; ++o)
        d[o] = A.S[(long long)o * g.nnodes + min(kk, g.nz - 1) * nxy + min(j, g.ny - 1) * g.nx + min(i, g.nx - 1)];
    };
    coefficients(k0, cf[0]);
    __syncthreads();
    window(0, w[0]);
    window(1, w[1]);
#pragma unroll
    for (int l = 0; l < NZ; ++l) {
      if (l + 1 < NZ) coefficients(k0 + l + 1, cf[(l + 1) & 1]);
      window(l + 2, w[2]);
      double av = 0.0;
#pragma unroll
      for (int o = 0; o < NS; ++o) av = fma(cf[l & 1][o], w[o / 9][o % 9], av);
      finish(k0 + l, av, w[1][4]);
#pragma unroll
      for (int o = 0; o < 9; ++o) {
        w[0][o] = w[1][o];
        w[1][o] = w[2][o];
      }
    }
  }
  if (MODE != kApply || !A.r) return;
  __shared__ double red[2][4];
  for (int off = 32; off > 0; off >>= 1) {
    sum_y += __shfl_down(sum_y, off, 64);
    sum_r += __shfl_down(sum_r, off, 64);
  }
  if ((tid & 63) == 0) {
    red[0][tid >> 6] = sum_y;
    red[1][tid >> 6] = sum_r;
  }
  __syncthreads();
  if (tid < 2) A.parts[tid * gridDim.x + blockIdx.x] = ((red[tid][0] + red[tid][1]) + red[tid][2]) + red[tid][3];
}

// out[h] = sum of the parts of half h, in a fixed order (one block)
__global__ void __launch_bounds__(512) scalar_sum2_kernel(int nparts, const double* __restrict__ parts,
                                                          double* __restrict__ out) {
  const int h = threadIdx.x >> 8, t = threadIdx.x & 255;
  double s = 0.0;
  for (int b = t; b < nparts; b += 256) s += parts[h * nparts + b];
  __shared__ double red[8];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (t == 0) out[h] = ((red[4 * h] + red[4 * h + 1]) + red[4 * h + 2]) + red[4 * h + 3];
}

// D^-1 from the centre coefficients
__global__ void scalar_dinv_kernel(long long n, const double* __restrict__ centre, double* __restrict__ dinv) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dinv[i] = 1.0 / centre[i];
}

template <int DIM>
__global__ void scalar_restrict_kernel(GridDims gf, GridDims gc, const double* __restrict__ rf,
                                       double* __restrict__ rc) {
  const long long N = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (N >= gc.nnodes) return;
  int I, J, K;
  node_ijk(gc, N, I, J, K);
  // every load issued at once: outside the grid the centre is read with weight 0
  double acc = 0.0;
  const long long centre = ((long long)(DIM == 3 ? 2 * K : 0) * gf.ny + 2 * J) * gf.nx + 2 * I;
#pragma unroll
  for (int c = 0; c < SCfg<DIM>::NS; ++c) {
    const int dx = c % 3 - 1, dy = (c / 3) % 3 - 1, dz = DIM == 3 ? c / 9 - 1 : 0;
    const int fi = 2 * I + dx, fj = 2 * J + dy, fk = 2 * K + dz;
    const bool in = fi >= 0 && fi < gf.nx && fj >= 0 && fj < gf.ny && fk >= 0 && fk < gf.nz;
    const double w = in ? (dx ? 0.5 : 1.0) * (dy ? 0.5 : 1.0) * (dz ? 0.5 : 1.0) : 0.0;
    acc = fma(w, rf[in ? centre + dx + (long long)gf.nx * (dy + (long long)gf.ny * dz) : centre], acc);
  }
  rc[N] = acc;
}

// dense coarsest matrix from its stencil
template <int DIM>
__global__ void scalar_dense_kernel(GridDims g, const double* __restrict__ S, double* __restrict__ A) {
  constexpr int NS = SCfg<DIM>::NS;
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= g.nnodes) return;
  int i, j, k;
  node_ijk(g, n, i, j, k);
  for (int c = 0; c < NS; ++c) {
    const int dx = c % 3 - 1, dy = (c / 3) % 3 - 1, dz = DIM == 3 ? c / 9 - 1 : 0;
    const int ii = i + dx, jj = j + dy, kk = k + dz;
    if (ii < 0 || ii >= g.nx || jj < 0 || jj >= g.ny || kk < 0 || kk >= g.nz) continue;
    A[n * g.nnodes + ((long long)kk * g.ny + jj) * g.nx + ii] = S[(long long)c * g.nnodes + n];
  }
}

__global__ void scalar_fill_kernel(long long n, double v, double* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = v;
}

int launch_scalar_fine(int mode, const GridDims& g, const double* P0, const double* xe, const uint8_t* bcm,
                       double bcdiag, const double* u, const double* b, double* y, hipStream_t s) {
  const unsigned blocks = blocks_for(g.nnodes, 256);
  if (g.dim == 3) {
    if (mode == 0)
      scalar_apply_kernel<3, 0><<<blocks, 256, 0, s>>>(g, P0, xe, bcm, bcdiag, u, b, y);
    else
      scalar_apply_kernel<3, 1><<<blocks, 256, 0, s>>>(g, P0, xe, bcm, bcdiag, u, b, y);
  } else {
    if (mode == 0)
      scalar_apply_kernel<2, 0><<<blocks, 256, 0, s>>>(g, P0, xe, bcm, bcdiag, u, b, y);
    else
      scalar_apply_kernel<2, 1><<<blocks, 256, 0, s>>>(g, P0, xe, bcm, bcdiag, u, b, y);
  }
  return check_launch("scalar_apply_kernel");
}

}  // namespace
}  // namespace pmt

using namespace pmt;

// ---------------------------------------------------------------------------------------------
// scalar multigrid handle
struct pmt_smg {
  int dim = 3;
  int nlev = 0;
  GridDims g[kScalarMaxLevels];
  double omega[kScalarMaxLevels] = {};
  int steps[kScalarMaxLevels] = {};
  double* S[kScalarMaxLevels] = {};  // stencils (levels 0..nlev-1)
  double* dinv[kScalarMaxLevels] = {};  // inverse diagonals (levels above the coarsest)
  double* u[kScalarMaxLevels] = {};  // corrections (levels >= 1)
  double* b[kScalarMaxLevels] = {};  // right-hand sides (levels >= 1)
  double* t[kScalarMaxLevels] = {};  // work: iterate, residual
  double* W[2] = {};                 // a slab's stencils coarsened along x, along x and y
  long long wlen[2] = {};            // doubles of W
  bool sym = false;                  // P0 is symmetric
  bool elem = false;                 // P0[a][b] depends on a ^ b only: the fine grid is applied from the densities
  double pe[8] = {};                 // then P0[0][a]
  double* parts = nullptr;           // block parts of the dots fused with the fine operator
  double* host = nullptr;            // pinned [value, sequence number] of the stopping test, [.., 4 scalars]
  double* P0 = nullptr;              // element matrix (device)
  double* Ainv = nullptr;            // coarsest inverse
  double* gjw = nullptr;             // workspace of its inversion
  const double* xe = nullptr;
  const uint8_t* bcm = nullptr;
  double bcdiag = 0.0;
  bool ready = false;
  // CG vectors and scalars
  double *r = nullptr, *z = nullptr, *p = nullptr, *q = nullptr, *sc = nullptr, *work = nullptr;
  long long bytes = 0;
  std::vector<void*> allocs;
};

namespace {

int smg_alloc(pmt_smg* h, double** p, long long count) {
  void* q = nullptr;
  PMT_HIP(hipMalloc(&q, (size_t)(count > 0 ? count : 1) * sizeof(double)));
  h->allocs.push_back(q);
  h->bytes += count * (long long)sizeof(double);
  *p = static_cast<double*>(q);
  return PMT_OK;
}

// Coarse planes of a slab whose 2 m + 1 fine planes, a and b doubles each after the first and second axis, fit
// into wa and wb doubles; at least one.  64 MB after the first axis: one slab up to about 0.6 million nodes, and the
// work arrays add 0.1 GB to a hierarchy instead of 0.75 of its fine stencil (162 bytes per node beside 310).  128^3: an
// update in four slabs 7.76 ms, in one 7.73.
constexpr long long kSlab = 1LL << 23;
int slab_planes(long long a, long long b, int ncl, long long wa, long long wb) {
  long long fine = wa / a;
  if (b > 0) fine = std::min(fine, wb / b);
  return fine >= 2LL * ncl - 1 ? ncl : (int)std::max(1LL, (fine - 1) / 2);
}

// node planes per block: 4, and 2 or 1 while the blocks do not give every CU two
int level_planes(const GridDims& g) {
  const long long blocks = (long long)((g.nx + 31) / 32) * ((g.ny + 7) / 8) * g.nz, want = 2LL * device_cu_count();
  return blocks >= 4 * want ? 4 : blocks >= 2 * want ? 2 : 1;
}
int level_blocks(const GridDims& g) {
  const int nz = level_planes(g);
  return (g.nx + 31) / 32 * ((g.ny + 7) / 8) * ((g.nz + nz - 1) / nz);
}

template <int SRC, int MODE>
int smg_level(pmt_smg* h, int l, LevelArgs a, hipStream_t s) {
  const GridDims& g = h->g[l];
  const int tx = (g.nx + 31) / 32, ty = (g.ny + 7) / 8, blocks = level_blocks(g), planes = level_planes(g);
  a.dinv = h->dinv[l];
  a.omega = h->omega[l];
  const bool elem = l == 0 && h->elem;
  if (elem) {
    a.xe = h->xe;
    a.bcm = h->bcm;
    a.bcdiag = h->bcdiag;
    for (int q = 0; q < 8; ++q) a.p[q] = h->pe[q];
  } else {
    a.S = h->S[l];
  }
  auto run = [&](auto kernel) { kernel<<<blocks, 256, 0, s>>>(g, tx, ty, a); };
  auto pick = [&](auto nz) {
    constexpr int NZ = decltype(nz)::value;
    elem ? run(scalar_level_kernel<3, true, SRC, MODE, NZ>) : run(scalar_level_kernel<3, false, SRC, MODE, NZ>);
  };
  if (h->dim == 2)
    elem ? run(scalar_level_kernel<2, true, SRC, MODE, 1>) : run(scalar_level_kernel<2, false, SRC, MODE, 1>);
  else if (planes == 4)
    pick(std::integral_constant<int, 4>{});
  else if (planes == 2)
    pick(std::integral_constant<int, 2>{});
  else
    pick(std::integral_constant<int, 1>{});
  return check_launch("scalar_level_kernel");
}

// S[l + 1] = R^T S[l] R by slabs of the last axis, as many coarse planes (2D: rows) at a time as W takes: m of them
// need the 2 m + 1 fine planes around their images
template <int DIM>
int smg_coarsen(pmt_smg* h, int l, hipStream_t s) {
  constexpr int NS = SCfg<DIM>::NS;
  const GridDims &gf = h->g[l], &gc = h->g[l + 1];
  const int nl = DIM == 3 ? gf.nz : gf.ny, ncl = DIM == 3 ? gc.nz : gc.ny;
  const long long fp = DIM == 3 ? (long long)gf.nx * gf.ny : gf.nx;  // nodes of a plane: fine, after x, after x and y
  const long long xp = DIM == 3 ? (long long)gc.nx * gf.ny : gc.nx, cp = DIM == 3 ? (long long)gc.nx * gc.ny : gc.nx;
  const int m = slab_planes(NS * xp, DIM == 3 ? NS * cp : 0, ncl, h->wlen[0], h->wlen[1]);
  for (int c0 = 0; c0 < ncl; c0 += m) {
    const int cl = std::min(m, ncl - c0), f0 = std::max(2 * c0 - 1, 0), f1 = std::min(2 * (c0 + cl - 1) + 2, nl);
    const int n = f1 - f0, first = 2 * c0 - f0;
    const double* S = h->S[l] + f0 * fp;
    double* T = h->S[l + 1] + c0 * cp;
    scalar_coarsen_kernel<DIM, 0><<<blocks_for(n * xp, 256), 256, 0, s>>>(gf.nx, gf.ny, n, 0, 0, S, gf.nnodes, h->W[0],
                                                                        n * xp);
    if constexpr (DIM == 3) {
      scalar_coarsen_kernel<3, 1><<<blocks_for(n * cp, 256), 256, 0, s>>>(gc.nx, gf.ny, n, 0, 0, h->W[0], n * xp, h->W[1],
                                                                        n * cp);
      scalar_coarsen_kernel<3, 2><<<blocks_for(cl * cp, 256), 256, 0, s>>>(gc.nx, gc.ny, n, first, cl, h->W[1], n * cp, T,
                                                                         gc.nnodes);
    } else {
      scalar_coarsen_kernel<2, 1><<<blocks_for(cl * cp, 256), 256, 0, s>>>(gc.nx, 0, n, first, cl, h->W[0], n * xp, T,
                                                                         gc.nnodes);
    }
    PMT_TRY(check_launch("scalar_coarsen_kernel"));
  }
  return PMT_OK;
}

int smg_apply(pmt_smg* h, int l, const double* u, double* y, hipStream_t s, const double* r = nullptr) {
  LevelArgs a{};
  a.u = u;
  a.y = y;
  a.r = r;
  a.parts = h->parts;
  return smg_level<kPlain, kApply>(h, l, a, s);
}

int smg_residual(pmt_smg* h, int l, const double* u, const double* b, double* y, hipStream_t s) {
  LevelArgs a{};
  a.u = u;
  a.b = b;
  a.y = y;
  return smg_level<kPlain, kResidual>(h, l, a, s);
}

// z = V-cycle(r) on level l (output written to z; rhs r; both length nnodes of level l)
int smg_vcycle(pmt_smg* h, int l, const double* r, double* z, hipStream_t s) {
  const GridDims& g = h->g[l];
  if (l == h->nlev - 1) return launch_gemv<double>(g.nnodes, h->Ainv, r, z, s);
  const int steps = h->steps[l];
  // pre-smoothing from zero (iterative.py:232-233); the first two sweeps are one pass.  The passes alternate between
  // t and z, from the one that has the last of the `steps` post-sweeps write z
  double *cur = steps == 1 ? h->t[l] : z, *oth = steps == 1 ? z : h->t[l];
  LevelArgs a{};
  a.b = r;
  if (steps == 1) {
    PMT_TRY(launch_jacobi0<double>(g.nnodes, h->dinv[l], r, h->omega[l], cur, s));
  } else {
    a.y = cur;
    PMT_TRY((smg_level<kFirst, kSweep>(h, l, a, s)));
  }
  for (int k = 2; k < steps; ++k) {
    a.u = cur;
    a.y = oth;
    PMT_TRY((smg_level<kPlain, kSweep>(h, l, a, s)));
    std::swap(cur, oth);
  }
  // residual, restriction, inner level
  PMT_TRY(smg_residual(h, l, cur, r, oth, s));
  const GridDims& gc = h->g[l + 1];
  const unsigned cblocks = blocks_for(gc.nnodes, 256);
  if (h->dim == 3)
    scalar_restrict_kernel<3><<<cblocks, 256, 0, s>>>(g, gc, oth, h->b[l + 1]);
  else
    scalar_restrict_kernel<2><<<cblocks, 256, 0, s>>>(g, gc, oth, h->b[l + 1]);
  PMT_TRY(check_launch("scalar_restrict_kernel"));
  PMT_TRY(smg_vcycle(h, l + 1, h->b[l + 1], h->u[l + 1], s));
  // post-smoothing, the prolongation within its first sweep
  for (int k = 0; k < steps; ++k) {
    a.u = cur;
    a.y = oth;
    if (k == 0) {
      a.e = h->u[l + 1];
      a.cnx = gc.nx;
      a.cny = gc.ny;
      PMT_TRY((smg_level<kCorrected, kSweep>(h, l, a, s)));
    } else {
      PMT_TRY((smg_level<kPlain, kSweep>(h, l, a, s)));
    }
    std::swap(cur, oth);
  }
  return cur == z ? PMT_OK : arg_error("smg_vcycle: internal buffer parity error");
}

}  // namespace

extern "C" {

int pmt_scalar_apply(int nelx, int nely, int nelz, const double* P0, const double* xe, const uint8_t* bcmask,
                     double bcdiag, const double* u, double* y, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || !P0 || !xe || !u || !y) return arg_error("pmt_scalar_apply: bad argument");
  return launch_scalar_fine(0, make_grid(nelx, nely, nelz), P0, xe, bcmask, bcdiag, u, nullptr, y,
                            (hipStream_t)stream);
}

int pmt_scalar_residual(int nelx, int nely, int nelz, const double* P0, const double* xe, const uint8_t* bcmask,
                        double bcdiag, const double* b, const double* u, double* r, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || !P0 || !xe || !b || !u || !r) return arg_error("pmt_scalar_residual: bad argument");
  return launch_scalar_fine(1, make_grid(nelx, nely, nelz), P0, xe, bcmask, bcdiag, u, b, r, (hipStream_t)stream);
}

int pmt_scalar_diagonal(int nelx, int nely, int nelz, const double* P0, const double* xe, const uint8_t* bcmask,
                        double bcdiag, double* diag, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || !P0 || !xe || !diag) return arg_error("pmt_scalar_diagonal: bad argument");
  GridDims g = make_grid(nelx, nely, nelz);
  hipStream_t s = (hipStream_t)stream;
  if (g.dim == 3)
    scalar_diag_kernel<3><<<blocks_for(g.nnodes, 256), 256, 0, s>>>(g, P0, xe, bcmask, bcdiag, diag);
  else
    scalar_diag_kernel<2><<<blocks_for(g.nnodes, 256), 256, 0, s>>>(g, P0, xe, bcmask, bcdiag, diag);
  return check_launch("scalar_diag_kernel");
}

int pmt_scalar_sens_contract(int nelx, int nely, int nelz, const double* P0, const uint8_t* bcmask, const double* u,
                             const double* v, double alpha, double* dx, int accumulate, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || !P0 || !u || !v || !dx) return arg_error("pmt_scalar_sens_contract: bad argument");
  GridDims g = make_grid(nelx, nely, nelz);
  hipStream_t s = (hipStream_t)stream;
  if (g.dim == 3)
    scalar_sens_kernel<3><<<blocks_for(g.nel, 256), 256, 0, s>>>(g, P0, bcmask, u, v, alpha, dx, accumulate);
  else
    scalar_sens_kernel<2><<<blocks_for(g.nel, 256), 256, 0, s>>>(g, P0, bcmask, u, v, alpha, dx, accumulate);
  return check_launch("scalar_sens_kernel");
}

int pmt_smg_create(int nelx, int nely, int nelz, int nlevels, const double* omega, const int* steps,
                   const double* P0_host, pmt_smg** out) {
  if (!out || !P0_host || !grid_ok(nelx, nely, nelz) || nlevels < 2 || nlevels > kScalarMaxLevels || !omega ||
      !steps)
    return arg_error("pmt_smg_create: bad argument");
  *out = nullptr;
  pmt_smg* h = new pmt_smg();
  h->dim = nelz > 0 ? 3 : 2;
  h->nlev = nlevels;
  int ex = nelx, ey = nely, ez = nelz;
  for (int l = 0; l < nlevels; ++l) {
    if (l > 0) {
      if (ex % 2 || ey % 2 || (h->dim == 3 && ez % 2)) {
        delete h;
        return arg_error("pmt_smg_create: every level above the coarsest needs even element counts");
      }
      ex /= 2;
      ey /= 2;
      ez = h->dim == 3 ? ez / 2 : 0;
    }
    h->g[l] = make_grid(ex, ey, ez);
    if (l < nlevels - 1) {
      h->omega[l] = omega[l];
      h->steps[l] = steps[l] < 1 ? 1 : steps[l];
    }
  }
  const int NN = 1 << h->dim, NS = h->dim == 3 ? 27 : 9;
  const long long nc = h->g[nlevels - 1].nnodes;
  int rc = PMT_OK;
  auto A = [&](double** p, long long n) {
    if (rc == PMT_OK) rc = smg_alloc(h, p, n);
  };
  A(&h->P0, NN * NN);
  for (int l = 0; l < nlevels; ++l) {
    A(&h->S[l], NS * h->g[l].nnodes);
    if (l < nlevels - 1) {
      A(&h->dinv[l], h->g[l].nnodes);
      A(&h->t[l], h->g[l].nnodes);
    }
    if (l > 0) {
      A(&h->u[l], h->g[l].nnodes);
      A(&h->b[l], h->g[l].nnodes);
    }
  }
  A(&h->Ainv, nc * nc);
  A(&h->gjw, gj_work_size(nc));
  const GridDims& g0 = h->g[0];
  const long long n0 = g0.nnodes;
  {
    const GridDims& g1 = h->g[1];
    const long long a = NS * (h->dim == 3 ? (long long)g1.nx * g0.ny : g1.nx);  // doubles of a fine plane after x
    const long long b = h->dim == 3 ? (long long)NS * g1.nx * g1.ny : 0;        // after x and y
    const int ncl = h->dim == 3 ? g1.nz : g1.ny;
    const int m = slab_planes(a, 0, ncl, kSlab, 0), fine = m == ncl ? 2 * ncl - 1 : 2 * m + 1;
    h->wlen[0] = a * fine;
    h->wlen[1] = b * fine;
    A(&h->W[0], h->wlen[0]);
    if (h->dim == 3) A(&h->W[1], h->wlen[1]);
  }
  A(&h->parts, 2LL * level_blocks(g0));
  // whether P0[a][b] depends on a ^ b only (to rounding): an isotropic box element
  double big = 0.0;
  for (int q = 0; q < NN * NN; ++q) big = std::max(big, std::fabs(P0_host[q]));
  h->elem = big > 0.0 && n0 < (1LL << 31);
  for (int a = 0; a < NN; ++a)
    for (int b = 0; b < NN; ++b)
      if (!(std::fabs(P0_host[a * NN + b] - P0_host[a ^ b]) <= 1e-14 * big)) h->elem = false;
  h->sym = symmetric_matrix(NN, P0_host);
  for (int a = 0; a < NN; ++a) h->pe[a] = P0_host[a];
  A(&h->r, n0);
  A(&h->z, n0);
  A(&h->p, n0);
  A(&h->q, n0);
  A(&h->sc, 8);
  A(&h->work, std::max<long long>(2 * kReduceBlocks, cg_xr_parts(n0)));
  if (rc == PMT_OK) rc = hip_status(hipHostMalloc((void**)&h->host, 8 * sizeof(double), hipHostMallocCoherent),
                                    "hipHostMalloc");
  if (rc == PMT_OK) h->host[1] = -1.0;  // no sequence number
  if (rc == PMT_OK) rc = hip_status(hipMemcpy(h->P0, P0_host, NN * NN * sizeof(double), hipMemcpyHostToDevice),
                                    "pmt_smg_create: copy P0");
  if (rc != PMT_OK) {
    pmt_smg_destroy(h);
    return rc;
  }
  *out = h;
  return PMT_OK;
}

int pmt_smg_destroy(pmt_smg* h) {
  if (!h) return PMT_OK;
  (void)hipDeviceSynchronize();
  for (void* p : h->allocs) (void)hipFree(p);
  if (h->host) (void)hipHostFree(h->host);
  delete h;
  return PMT_OK;
}

long long pmt_smg_level_nodes(pmt_smg* h, int level) {
  if (!h || level < 0 || level >= h->nlev) return arg_error("pmt_smg_level_nodes: bad argument");
  return h->g[level].nnodes;
}

int pmt_smg_update(pmt_smg* h, const double* xe, const uint8_t* bcmask, double bcdiag, void* stream) {
  if (!h || !xe) return arg_error("pmt_smg_update: bad argument");
  hipStream_t s = (hipStream_t)stream;
  h->xe = xe;
  h->bcm = bcmask;
  h->bcdiag = bcdiag;
  const GridDims& g0 = h->g[0];
  if (h->dim == 3)
    scalar_stencil_fine_kernel<3><<<blocks_for(g0.nnodes, 128), 128, 0, s>>>(g0, h->P0, xe, bcmask, bcdiag, h->S[0]);
  else
    scalar_stencil_fine_kernel<2><<<blocks_for(g0.nnodes, 128), 128, 0, s>>>(g0, h->P0, xe, bcmask, bcdiag, h->S[0]);
  PMT_TRY(check_launch("scalar_stencil_fine_kernel"));
  for (int l = 0; l + 1 < h->nlev; ++l) {
    const GridDims& gf = h->g[l];
    const GridDims& gc = h->g[l + 1];
    scalar_dinv_kernel<<<blocks_for(gf.nnodes, 256), 256, 0, s>>>(
        gf.nnodes, h->S[l] + (h->dim == 3 ? 13 : 4) * gf.nnodes, h->dinv[l]);
    PMT_TRY(check_launch("scalar_dinv_kernel"));
    PMT_TRY(h->dim == 3 ? smg_coarsen<3>(h, l, s) : smg_coarsen<2>(h, l, s));
  }
  const int L = h->nlev - 1;
  const long long nc = h->g[L].nnodes;
  scalar_fill_kernel<<<blocks_for(nc * nc, 256), 256, 0, s>>>(nc * nc, 0.0, h->Ainv);
  PMT_TRY(check_launch("scalar_fill_kernel"));
  if (h->dim == 3)
    scalar_dense_kernel<3><<<blocks_for(nc, 128), 128, 0, s>>>(h->g[L], h->S[L], h->Ainv);
  else
    scalar_dense_kernel<2><<<blocks_for(nc, 128), 128, 0, s>>>(h->g[L], h->S[L], h->Ainv);
  PMT_TRY(check_launch("scalar_dense_kernel"));
  PMT_TRY(gj_invert(nc, h->sym, h->Ainv, h->gjw, s));
  h->ready = true;
  return PMT_OK;
}

int pmt_smg_vcycle(pmt_smg* h, const double* r, double* z, void* stream) {
  if (!h || !r || !z) return arg_error("pmt_smg_vcycle: bad argument");
  if (!h->ready) {
    set_error("pmt_smg_vcycle: call pmt_smg_update first");
    return PMT_ERR_STATE;
  }
  return smg_vcycle(h, 0, r, z, (hipStream_t)stream);
}

int pmt_smg_level_apply(pmt_smg* h, int level, const double* u, double* y, void* stream) {
  if (!h || level < 0 || level >= h->nlev || !u || !y) return arg_error("pmt_smg_level_apply: bad argument");
  if (!h->ready) {
    set_error("pmt_smg_level_apply: call pmt_smg_update first");
    return PMT_ERR_STATE;
  }
  return smg_apply(h, level, u, y, (hipStream_t)stream);
}

int pmt_smg_pcg_solve(pmt_smg* h, const double* b, double* x, int x0_is_zero, double tol, int maxit, int restart,
                      int* iters, double* relres, double* history, void* stream) {
  if (!h || !b || !x || maxit < 0 || restart < 1) return arg_error("pmt_smg_pcg_solve: bad argument");
  if (!h->ready) {
    set_error("pmt_smg_pcg_solve: call pmt_smg_update first");
    return PMT_ERR_STATE;
  }
  hipStream_t s = (hipStream_t)stream;
  const long long n = h->g[0].nnodes;
  double* sc = h->sc;  // 0 p.q  1 p.r  2 r.r  3 q.z  4 b.b  5 r.r or z.z
  if (iters) *iters = 0;
  if (relres) *relres = 0.0;
  if (x0_is_zero) PMT_TRY(launch_fill(n, 0.0, x, s));
  // r = b - A x ; bn = |b| ; |r|
  PMT_TRY(smg_residual(h, 0, x, b, h->r, s));
  PMT_TRY(launch_dot2(n, b, b, h->r, h->r, sc + 4, h->work, s));
  PMT_HIP(hipMemcpyAsync(h->host + 4, sc + 4, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
  PMT_HIP(hipStreamSynchronize(s));
  const double bn = std::sqrt(h->host[4]);
  if (!std::isfinite(h->host[4]) || !std::isfinite(h->host[5])) {
    set_error("pmt_smg_pcg_solve: non-finite right-hand side or start vector");
    return PMT_ERR_NUMERIC;
  }
  if (bn == 0.0) return launch_fill(n, 0.0, x, s);  // b = 0: x = 0 (CG.solve returns x0 only when it already meets tol)
  double tval = std::sqrt(h->host[5]) / bn;
  if (history) history[0] = tval;
  if (tval <= tol) {
    if (relres) *relres = tval;
    return PMT_OK;
  }
  // z = M r ; p = orth(z) = z / |z| (CG.solve works on (n, 1) blocks and orth normalises the first
  // direction, iterative.py:259-292, 360-362)
  PMT_TRY(smg_vcycle(h, 0, h->r, h->z, s));
  PMT_TRY(launch_dot(n, h->z, h->z, sc + 5, h->work, s));
  PMT_TRY(launch_scale_rsqrt(n, sc, 5, h->z, h->p, s));
  const int nparts = level_blocks(h->g[0]);
  int it = 0;
  double tprev = 0.0;
  bool x_pending = false;  // x lacks this iteration's alpha p (added by the p update or after the loop)
  for (it = 0; it < maxit; ++it) {
    PMT_TRY(smg_apply(h, 0, h->p, h->q, s, h->r));
    const bool inline_sums = it % restart != 0 && cg_sums_inline(nparts);  // the r update adds the partials
    if (!inline_sums) {
      scalar_sum2_kernel<<<1, 512, 0, s>>>(nparts, h->parts, sc);
      PMT_TRY(check_launch("scalar_sum2_kernel"));
    }
    const double seq = publish_sequence();
    if (it % restart == 0) {
      PMT_TRY(launch_cg_x_update(n, sc, h->p, x, s));
      PMT_TRY(smg_residual(h, 0, x, b, h->r, s));
      PMT_TRY(launch_dot(n, h->r, h->r, sc + 2, h->work, s));
      PMT_TRY(launch_publish(sc + 2, seq, h->host, s));
    } else {
      PMT_TRY(launch_cg_xr_update<double>(n, sc, inline_sums ? h->parts : nullptr, nparts, h->q, h->r,
                                          h->work, sc + 2, s, nullptr, nullptr, 0.0, nullptr, h->host, seq));
      x_pending = true;
    }
    // z = M r, beta = -(q.z) / (p.q), p = z + beta p
    auto next_direction = [&]() -> int {
      PMT_TRY(smg_vcycle(h, 0, h->r, h->z, s));
      PMT_TRY(launch_cg_beta_update(n, sc, h->q, h->z, h->p, h->work, x_pending ? x : nullptr, s));
      x_pending = false;
      return PMT_OK;
    };
    // enqueued before the host waits for r.r when the residual's rate says this iteration will not stop (the
    // iterates are the same either way)
    const bool ahead = tval * (tprev > 0.0 ? tval / tprev : 0.3) > 2.0 * tol;
    if (ahead) PMT_TRY(next_direction());
    double rr = 0.0;
    PMT_TRY(publish_wait(h->host, seq, sc + 2, h->host + 4, &rr, s));
    tprev = tval;
    if (!std::isfinite(rr)) {
      PMT_HIP(hipStreamSynchronize(s));  // nothing enqueued ahead is left running on the caller's buffers
      set_error(("pmt_smg_pcg_solve: non-finite residual at iteration " + std::to_string(it + 1)).c_str());
      if (iters) *iters = it + 1;
      return PMT_ERR_NUMERIC;
    }
    tval = std::sqrt(rr) / bn;
    if (history) history[it + 1] = tval;
    if (tval <= tol) break;
    if (!ahead) PMT_TRY(next_direction());
  }
  if (x_pending) PMT_TRY(launch_cg_x_update(n, sc, h->p, x, s));
  if (iters) *iters = it < maxit ? it + 1 : maxit;
  if (relres) *relres = tval;
  return PMT_OK;
}

}  // extern "C"
