// Coarse-grid operators of the geometric multigrid (pymoto/solvers/iterative.py:168-176).
//
// Galerkin R^T A R element by element: every fine element c lies in one coarse element E and
// the trilinear prolongation restricted to c only reads E's nodes, u_c = P_c u_E with
// P_c = p_c (x) I_D, p_c[a][A] = prod_dims w(f, A_bit), f = child_bit + a_bit in {0,1,2},
// w(0,0) = w(2,1) = 1, w(1,*) = 1/2, else 0.  Hence R^T A R = assemble_E sum_c P_c^T A_c P_c.
// On the fine level A_c = x_c M_c K0 M_c + D_c with M_c the Dirichlet mask and D_c the bcdiag
// diagonal of Dirichlet dofs shared equally by the mult(node) elements around each node, so
// that the element sum reproduces A = P K P + bcdiag I_bc of the reference assembly
// (assembly.py:209-230, 267-272).  On coarser levels A_c is the stored element matrix of the
// child.  The coarse element matrices are then summed per node into a 3^D block stencil.
//
// Coarsest level: dense matrix from the stencil, explicit inverse by blocked Gauss-Jordan
// (no pivoting; the Galerkin operator is SPD), applied as a dense GEMV in every V-cycle -
// the direct solve of auto_determine_solver (iterative.py:174-176).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "launch.h"

namespace pmt {

// One block per coarse element; thread t = (A, B) node pair owns the D x D block (A, B) of K_E.
// FINE: A_c built from x_c, K0, the Dirichlet mask and bcdiag/mult; else read from Kf.
// Does coarse element (CI, CJ, CK) contain a Dirichlet node among its 3^D fine nodes?
template <int DIM>
__device__ inline bool touches_bc(const GridDims& gf, const uint8_t* __restrict__ bcm, int CI, int CJ, int CK) {
  for (int q = 0; q < (DIM == 3 ? 27 : 9); ++q) {
    const int i = 2 * CI + q % 3, j = 2 * CJ + (q / 3) % 3, k = DIM == 3 ? 2 * CK + q / 9 : 0;
    if (bcm[((long long)k * gf.ny + j) * gf.nx + i]) return true;
  }
  return false;
}

// Fine -> first coarse level (hex8).  A child without Dirichlet nodes contributes x_c G_c with
// G_c = P_c^T K0 P_c fixed (P_c^T (x_c K0) P_c); the children with Dirichlet nodes contribute the masked
// P_c^T (x_c M K0 M + D_c) P_c, collected per flagged coarse element as a correction dK in a compact
// list (the order of the list is irrelevant: each entry only touches its own element's correction).
//  1. galerkin_bc_flags_kernel: per coarse element the bit set of children with a Dirichlet node, the
//     list of flagged elements and the element -> list position map (-1: not flagged);
//  2. galerkin_fine_bc_kernel: dK of the listed elements (one wave per element, lane = (A, B)).
__global__ void galerkin_bc_flags_kernel(GridDims gf, GridDims gc, const uint8_t* __restrict__ bcm,
                                         uint8_t* __restrict__ cflag, int* __restrict__ list, int* __restrict__ count,
                                         int* __restrict__ map) {
  const long long E = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (E >= gc.nel) return;
  const int CI = (int)(E % gc.ex);
  const long long tt = E / gc.ex;
  const int CJ = (int)(tt % gc.ey), CK = (int)(tt / gc.ey);
  unsigned m27 = 0;  // bit q: fine node (q%3, q/3%3, q/9) of the element is Dirichlet
  for (int q = 0; q < 27; ++q) {
    const int i = 2 * CI + q % 3, j = 2 * CJ + (q / 3) % 3, k = 2 * CK + q / 9;
    if (bcm[((long long)k * gf.ny + j) * gf.nx + i]) m27 |= 1u << q;
  }
  unsigned flags = 0;
  for (int c = 0; c < 8; ++c)
    for (int a = 0; a < 8; ++a) {
      const int q = ((c >> 2) + (a >> 2)) * 9 + (((c >> 1) & 1) + ((a >> 1) & 1)) * 3 + (c & 1) + (a & 1);
      if ((m27 >> q) & 1u) flags |= 1u << c;
    }
  cflag[E] = (uint8_t)flags;
  int idx = -1;
  if (flags) {
    idx = atomicAdd(count, 1);
    list[idx] = (int)E;
  }
  map[E] = idx;
}

__global__ void zero_int_kernel(int* p) { *p = 0; }

void zero_int(int* p, hipStream_t s) { zero_int_kernel<<<1, 1, 0, s>>>(p); }

// dK of a listed element: block (A, B) of the sum over its flagged children of P_c^T (x_c M K0 M + D_c) P_c.
// One 64-lane block per listed element, lane = (A, B) 3x3 block; per child in two passes through LDS:
// T[a][B] = sum_b w(c, b, B) K_c[a][b] (lane a = A), then dK[A][B] += sum_a w(c, a, A) T[a][B] - no
// divergent loops (the first form, with data-dependent skips over zero weights, took 200 us per update at
// 256x128x128).
__global__ void __launch_bounds__(64)
galerkin_fine_bc_kernel(GridDims gf, GridDims gc, const double* __restrict__ K0, const double* __restrict__ xe,
                        const uint8_t* __restrict__ bcm, double bcdiag, const uint8_t* __restrict__ cflag,
                        const int* __restrict__ list, double* __restrict__ dK) {
  constexpr int NE = 24;
  __shared__ double sK0[NE * NE];
  __shared__ double sT[8][8][9];  // [a][B][d * 3 + d2]
  const int lane = threadIdx.x, A = lane >> 3, B = lane & 7;
  for (int q = lane; q < NE * NE; q += 64) sK0[q] = K0[q];
  const long long w = blockIdx.x;
  const long long E = list[w];
  const int CI = (int)(E % gc.ex);
  const long long tt = E / gc.ex;
  const int CJ = (int)(tt % gc.ey), CK = (int)(tt / gc.ey);
  const unsigned flags = cflag[E];
  double acc[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) acc[q] = 0.0;
  __syncthreads();
  for (int c = 0; c < 8; ++c) {
    if (!((flags >> c) & 1u)) continue;  // uniform over the block
    const int fi = 2 * CI + (c & 1), fj = 2 * CJ + ((c >> 1) & 1), fk = 2 * CK + ((c >> 2) & 1);
    const double xv = xe[((long long)fk * gf.ey + fj) * gf.ex + fi];
    unsigned mk[8];
#pragma unroll
    for (int b = 0; b < 8; ++b)
      mk[b] = bcm[((long long)(fk + ((b >> 2) & 1)) * gf.ny + fj + ((b >> 1) & 1)) * gf.nx + fi + (b & 1)];
    // row corner a = A of the child: its Dirichlet mask and the number of elements sharing its node
    const int ai = fi + (A & 1), aj = fj + ((A >> 1) & 1), ak = fk + ((A >> 2) & 1);
    const unsigned ma = mk[A];
    const double dsplit =
        bcdiag / (double)(((ai > 0) + (ai < gf.nx - 1)) * ((aj > 0) + (aj < gf.ny - 1)) * ((ak > 0) + (ak < gf.nz - 1)));
    double t[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) t[q] = 0.0;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const double wb = pweight<3>(c, b, B);
      const unsigned mb = mk[b];
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int d2 = 0; d2 < 3; ++d2) {
          const bool fa = (ma >> d) & 1u, fb = (mb >> d2) & 1u;
          double v = (fa || fb) ? 0.0 : xv * sK0[(A * 3 + d) * NE + b * 3 + d2];
          if (A == b && d == d2 && fa) v += dsplit;
          t[d * 3 + d2] = fma(wb, v, t[d * 3 + d2]);
        }
    }
    __syncthreads();  // the previous child's reads of sT are done
#pragma unroll
    for (int q = 0; q < 9; ++q) sT[A][B][q] = t[q];
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      const double wa = pweight<3>(c, a, A);
#pragma unroll
      for (int q = 0; q < 9; ++q) acc[q] = fma(wa, sT[a][B][q], acc[q]);
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int d2 = 0; d2 < 3; ++d2) dK[w * NE * NE + (A * 3 + d) * NE + B * 3 + d2] = acc[d * 3 + d2];
}

template <int DIM, bool FINE>
__global__ void __launch_bounds__(64)
galerkin_kernel(GridDims gf, GridDims gc, const double* __restrict__ K0, const double* __restrict__ xe,
                const uint8_t* __restrict__ bcm, double bcdiag, const double* __restrict__ Kf,
                double* __restrict__ Kc, int bc_only) {
  constexpr int NN = 1 << DIM;
  constexpr int NE = NN * DIM;
  __shared__ double sA[NE * NE];
  __shared__ double sT[NE * NE];
  __shared__ double sK0[FINE ? NE * NE : 1];
  const long long E = blockIdx.x;
  const int tid = threadIdx.x;  // NN*NN threads
  const int CI = (int)(E % gc.ex);
  const long long tt = E / gc.ex;
  const int CJ = (int)(tt % gc.ey);
  const int CK = (int)(tt / gc.ey);
  if (FINE && bc_only && !(bcm && touches_bc<DIM>(gf, bcm, CI, CJ, CK))) return;  // whole block leaves
  if (FINE) {
    for (int q = tid; q < NE * NE; q += NN * NN) sK0[q] = K0[q];
  }
  const int tA = tid / NN, tB = tid % NN;
  double acc[DIM][DIM];
#pragma unroll
  for (int d = 0; d < DIM; ++d)
#pragma unroll
    for (int d2 = 0; d2 < DIM; ++d2) acc[d][d2] = 0.0;

  for (int c = 0; c < NN; ++c) {
    const int fi = 2 * CI + (c & 1), fj = 2 * CJ + ((c >> 1) & 1), fk = DIM == 3 ? 2 * CK + ((c >> 2) & 1) : 0;
    const long long fe = ((long long)fk * gf.ey + fj) * gf.ex + fi;
    __syncthreads();  // previous child's sA/sT fully consumed (and sK0 loaded)
    if (FINE) {
      const double xc = xe[fe];
      for (int q = tid; q < NE * NE; q += NN * NN) {
        const int r = q / NE, s = q % NE;
        const int a = r / DIM, d = r % DIM, b = s / DIM, d2 = s % DIM;
        const int ai = fi + (a & 1), aj = fj + ((a >> 1) & 1), ak = DIM == 3 ? fk + ((a >> 2) & 1) : 0;
        const int bi = fi + (b & 1), bj = fj + ((b >> 1) & 1), bk = DIM == 3 ? fk + ((b >> 2) & 1) : 0;
        const long long na = ((long long)ak * gf.ny + aj) * gf.nx + ai;
        const long long nb = ((long long)bk * gf.ny + bj) * gf.nx + bi;
        const bool fa = bcm && ((bcm[na] >> d) & 1u);
        const bool fb = bcm && ((bcm[nb] >> d2) & 1u);
        double v = (fa || fb) ? 0.0 : xc * sK0[q];
        if (r == s && fa) {
          const int mult = ((ai > 0) + (ai < gf.nx - 1)) * ((aj > 0) + (aj < gf.ny - 1)) *
                           (DIM == 3 ? ((ak > 0) + (ak < gf.nz - 1)) : 1);
          v += bcdiag / (double)mult;
        }
        sA[q] = v;
      }
    } else {
      for (int q = tid; q < NE * NE; q += NN * NN) sA[q] = Kf[fe * NE * NE + q];
    }
    __syncthreads();
    // T = A_c P_c : thread (a = tA, B = tB) computes rows a*D+d, cols B*D+d2
    {
      const int a = tA, B = tB;
      double t[DIM][DIM];
#pragma unroll
      for (int d = 0; d < DIM; ++d)
#pragma unroll
        for (int d2 = 0; d2 < DIM; ++d2) t[d][d2] = 0.0;
      for (int b = 0; b < NN; ++b) {
        const double w = pweight<DIM>(c, b, B);
        if (w == 0.0) continue;
#pragma unroll
        for (int d = 0; d < DIM; ++d)
#pragma unroll
          for (int d2 = 0; d2 < DIM; ++d2) t[d][d2] = fma(w, sA[(a * DIM + d) * NE + b * DIM + d2], t[d][d2]);
      }
#pragma unroll
      for (int d = 0; d < DIM; ++d)
#pragma unroll
        for (int d2 = 0; d2 < DIM; ++d2) sT[(a * DIM + d) * NE + B * DIM + d2] = t[d][d2];
    }
    __syncthreads();
    // K_E(A, B) += sum_a p_c[a][A] T(a, B)
    for (int a = 0; a < NN; ++a) {
      const double w = pweight<DIM>(c, a, tA);
      if (w == 0.0) continue;
#pragma unroll
      for (int d = 0; d < DIM; ++d)
#pragma unroll
        for (int d2 = 0; d2 < DIM; ++d2) acc[d][d2] = fma(w, sT[(a * DIM + d) * NE + tB * DIM + d2], acc[d][d2]);
    }
  }
#pragma unroll
  for (int d = 0; d < DIM; ++d)
#pragma unroll
    for (int d2 = 0; d2 < DIM; ++d2) Kc[E * NE * NE + (tA * DIM + d) * NE + tB * DIM + d2] = acc[d][d2];
}

// Level-1 stencil straight from the fine densities (hex8): S[o](n) = sum over the coarse elements E
// holding n and n+o of K_E(loc n, loc n+o), K_E = sum over unflagged children of x_c G_c plus the
// correction dK of flagged elements.  Thread = coarse node; the 64 child densities of its 8 elements
// are held in registers, the offset/element/child loops are unrolled so every G entry is a
// compile-time offset (scalar loads).  KIND 0: full stencil (out.S); 1: half stencil and D^-1; 2: D^-1
// only (the level's operator is applied without a stencil).
template <int KIND>
__global__ void __launch_bounds__(256)
stencil_from_fine_kernel(GridDims gf, GridDims gc, const double* __restrict__ G, const double* __restrict__ xe,
                         const uint8_t* __restrict__ cflag, const int* __restrict__ map, const double* __restrict__ dK,
                         StencilOut out) {
  constexpr int NE = 24;
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= gc.nnodes) return;
  const int i = (int)(n % gc.nx);
  const long long t = n / gc.nx;
  const int j = (int)(t % gc.ny);
  const int k = (int)(t / gc.ny);
  const long long nn = gc.nnodes;
  double xv[8][8];
  unsigned fl[8];
  long long Eix[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int ei = i - 1 + (e & 1), ej = j - 1 + ((e >> 1) & 1), ek = k - 1 + ((e >> 2) & 1);
    const bool ok = ei >= 0 && ei < gc.ex && ej >= 0 && ej < gc.ey && ek >= 0 && ek < gc.ez;
    const long long E = ok ? ((long long)ek * gc.ey + ej) * gc.ex + ei : 0;
    Eix[e] = E;
    fl[e] = ok ? cflag[E] : 0u;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      double v = 0.0;
      if (ok) v = xe[((long long)(2 * ek + ((c >> 2) & 1)) * gf.ey + (2 * ej + ((c >> 1) & 1))) * gf.ex + 2 * ei + (c & 1)];
      xv[e][c] = ((fl[e] >> c) & 1u) ? 0.0 : v;  // flagged children come from dK below
    }
  }
  int o = 0;
#pragma unroll
  for (int dz = -1; dz <= 1; ++dz)
#pragma unroll
    for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
      for (int dx = -1; dx <= 1; ++dx, ++o) {
        if (KIND == 1 && o < 13) continue;  // backward blocks: the neighbours' forward blocks transposed
        if (KIND == 2 && o != 13) continue;
        double blk[3][3];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int d2 = 0; d2 < 3; ++d2) blk[d][d2] = 0.0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int ex = e & 1, ey = (e >> 1) & 1, ez = (e >> 2) & 1;
          const int bx = dx + 1 - ex, by = dy + 1 - ey, bz = dz + 1 - ez;
          if (bx < 0 || bx > 1 || by < 0 || by > 1 || bz < 0 || bz > 1) continue;  // compile time
          const int A = (1 - ex) + 2 * (1 - ey) + 4 * (1 - ez), B = bx + 2 * by + 4 * bz;
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const double* g = G + c * NE * NE + (A * 3) * NE + B * 3;
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
              for (int d2 = 0; d2 < 3; ++d2) blk[d][d2] = fma(xv[e][c], g[d * NE + d2], blk[d][d2]);
          }
          if (fl[e]) {
            const double* K = dK + (long long)map[Eix[e]] * NE * NE + (A * 3) * NE + B * 3;
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
              for (int d2 = 0; d2 < 3; ++d2) blk[d][d2] += K[d * NE + d2];
          }
        }
        if (KIND == 2) {
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const double v = 1.0 / blk[d][d];
            out.dinv[n * 3 + d] = v;
            if (out.dinv32) out.dinv32[n * 3 + d] = (float)v;
          }
        } else {
          emit_block<KIND == 1>(out, o, blk, n, nn);
        }
      }
}

// Per-node block stencil S[(o*D+d)*D+d2][n] = sum over elements E holding n and n+o of K_E(loc n, loc n+o)
template <int DIM>
__global__ void stencil_from_elements_kernel(GridDims g, const double* __restrict__ Ke, double* __restrict__ S) {
  constexpr int NN = 1 << DIM;
  constexpr int NE = NN * DIM;
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= g.nnodes) return;
  const int i = (int)(n % g.nx);
  const long long t = n / g.nx;
  const int j = (int)(t % g.ny);
  const int k = (int)(t / g.ny);
  const long long nn = g.nnodes;
  constexpr int ZLO = DIM == 3 ? -1 : 0, ZHI = DIM == 3 ? 1 : 0;
  int o = 0;
  for (int dz = ZLO; dz <= ZHI; ++dz)
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx, ++o) {
        double blk[DIM][DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d)
#pragma unroll
          for (int d2 = 0; d2 < DIM; ++d2) blk[d][d2] = 0.0;
        for (int e = 0; e < NN; ++e) {
          const int ex = e & 1, ey = (e >> 1) & 1, ez = DIM == 3 ? (e >> 2) & 1 : 1;
          const int bx = dx + 1 - ex, by = dy + 1 - ey, bz = DIM == 3 ? dz + 1 - ez : 0;
          if (bx < 0 || bx > 1 || by < 0 || by > 1 || bz < 0 || bz > 1) continue;
          const int ei = i - 1 + ex, ej = j - 1 + ey, ek = DIM == 3 ? k - 1 + ez : 0;
          if (ei < 0 || ei >= g.ex || ej < 0 || ej >= g.ey || ek < 0 || ek >= g.ez) continue;
          const long long E = ((long long)ek * g.ey + ej) * g.ex + ei;
          const int locn = (1 - ex) + 2 * (1 - ey) + (DIM == 3 ? 4 * (1 - ez) : 0);
          const int locm = bx + 2 * by + 4 * bz;
          const double* KE = Ke + E * NE * NE;
#pragma unroll
          for (int d = 0; d < DIM; ++d)
#pragma unroll
            for (int d2 = 0; d2 < DIM; ++d2) blk[d][d2] += KE[(locn * DIM + d) * NE + locm * DIM + d2];
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d)
#pragma unroll
          for (int d2 = 0; d2 < DIM; ++d2) S[((long long)(o * DIM + d) * DIM + d2) * nn + n] = blk[d][d2];
      }
}

// dense row-major A (n x n, n = nnodes*D) from the stencil; A must be zero-filled first
template <int DIM>
__global__ void dense_from_stencil_kernel(GridDims g, const double* __restrict__ S, double* __restrict__ A) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= g.nnodes) return;
  const int i = (int)(n % g.nx);
  const long long t = n / g.nx;
  const int j = (int)(t % g.ny);
  const int k = (int)(t / g.ny);
  const long long N = g.nnodes * DIM;
  constexpr int ZLO = DIM == 3 ? -1 : 0, ZHI = DIM == 3 ? 1 : 0;
  int o = 0;
  for (int dz = ZLO; dz <= ZHI; ++dz)
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx, ++o) {
        const int ii = i + dx, jj = j + dy, kk = k + dz;
        if (ii < 0 || ii >= g.nx || jj < 0 || jj >= g.ny || kk < 0 || kk >= g.nz) continue;
        const long long m = ((long long)kk * g.ny + jj) * g.nx + ii;
        for (int d = 0; d < DIM; ++d)
          for (int d2 = 0; d2 < DIM; ++d2)
            A[(n * DIM + d) * N + m * DIM + d2] = S[((long long)(o * DIM + d) * DIM + d2) * g.nnodes + n];
      }
}

// ---------------- blocked Gauss-Jordan inversion (in place), block size GJB ----------------
// Panel k: with P = A[K][K]^-1, the old row panel R = A[K][:] and column panel C = A[:][K],
//   A[K][K] = P, A[K][j] = P R_j, A[i][K] = -C_i P, A[i][j] -= C_i (P R_j)   (no pivoting: the operator is SPD)
// One launch per panel, a block per 64 x 64 tile: the panels are read from copies that the previous launch's
// blocks of that row and column wrote beside the matrix, so the tiles are updated in place; P R_j is formed
// again by every block of a column (the same work as the update, on compute units that would wait
// otherwise).  Of a symmetric matrix only the tiles on and above the diagonal are kept: its processed and its
// remaining part stay symmetric and the entries between them change sign when mirrored, so the row panel is the
// column panel transposed, negated for the processed columns; the last panel's launch writes the other half.
// The block of the next diagonal tile inverts it at the end of its update, so its chain of
// pivots runs beside the other tiles of the launch.
// 21 us per panel at n = 847 (14 panels) and bound by that chain; four launches per panel (diagonal inverse, column
// copy, row panel, update) took 76 us.  From n = 1900 on the tiles bound it: 12.9 ms at n = 6069 (24 ms for all
// tiles, 49 ms in four launches per panel).
constexpr int GJB = 64;
constexpr int GJL = GJB + 2;  // LDS row stride: the 16 rows x 2 entries of a half wave's operand read lie in 64 banks
typedef double gj_d4 __attribute__((ext_vector_type(4)));

// 1 / x to an ulp (a correctly rounded division is a longer dependent chain)
__device__ inline double gj_rcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// In-place inverse of a 64 x 64 tile held by 4 waves in the matrix-core result layout (a wave per 32 x 32
// quadrant: entry r of m[a][b] is row 32 (wave / 2) + 16 a + 4 r + lane / 16, column 32 (wave % 2) + 16 b +
// lane % 16): block Gauss-Jordan with 4 x 4 pivot blocks Q, 16 steps with one barrier each.  The pivot rows R
// and columns C go through LDS (sh: two buffers); every thread solves for the row of Q^-1 that it needs; the
// rest is m -= C (Q^-1 R), one matrix operation per 16 x 16 tile.  The pivot rows are one register (r = s % 4) of
// all lanes of a tile row and become Q^-1 R; in the pivot columns m counts as 0 and R as the identity.
// 12 us, a chain of dependent FP64 operations.  (With the whole of Q inverted by every thread, for (C Q^-1) R,
// 15 us; 4 x 4 entries per thread and the rank-4 update without the matrix cores 22 us; one pivot per step, the
// whole tile moving through LDS, 40 us.)
constexpr int kGjShared = 2 * (256 + 256 + 16);  // doubles
__device__ inline void gj_invert_tile(gj_d4 (&m)[2][2], double* sh, int tid) {
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lq = lane >> 4;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const double unit[4] = {lq == 0 ? 1.0 : 0.0, lq == 1 ? 1.0 : 0.0, lq == 2 ? 1.0 : 0.0, lq == 3 ? 1.0 : 0.0};
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    double* rows = sh + (s & 1) * kGjShared / 2;  // R [4][64], the identity in the pivot columns
    double* cols = rows + 256;                    // C [64][4]
    double* pivot = cols + 256;                   // Q [4][4]
    const int ta = (s / 4) % 2;                   // tile of the pivot in its quadrant
    const bool own_r = wr == (s / 8) * 32, own_c = wc == (s / 8) * 32;
    const bool piv = own_c && l16 / 4 == s % 4;   // (of tile column ta)
    if (own_r) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const double v = m[ta][b][s % 4], e = l16 % 4 == lq ? 1.0 : 0.0;
        rows[lq * 64 + wc + 16 * b + l16] = b == ta && piv ? e : v;
        if (b == ta && piv) pivot[lq * 4 + l16 % 4] = v;
      }
    }
    if (piv) {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) cols[(wr + 16 * a + 4 * r + lq) * 4 + l16 % 4] = m[a][ta][r];
    }
    __syncthreads();
    double q[4][4], c[2], rr[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) q[i][j] = pivot[i * 4 + j];
#pragma unroll
    for (int a = 0; a < 2; ++a) c[a] = cols[(wr + 16 * a + l16) * 4 + lq];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int k = 0; k < 4; ++k) rr[b][k] = rows[k * 64 + wc + 16 * b + l16];
    const double keep = piv ? 0.0 : 1.0;
#pragma unroll
    for (int a = 0; a < 2; ++a) m[a][ta] *= keep;
    // this lane's row y of Q^-1: y Q = e, Q = L U with the unit diagonal in L, y U first, along with the elimination
    double y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = unit[j];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const double inv = gj_rcp(q[p][p]);
      y[p] *= inv;
#pragma unroll
      for (int j = p + 1; j < 4; ++j) y[j] = fma(-y[p], q[p][j], y[j]);
#pragma unroll
      for (int i = p + 1; i < 4; ++i) {
        q[i][p] *= inv;
#pragma unroll
        for (int j = p + 1; j < 4; ++j) q[i][j] = fma(-q[i][p], q[p][j], q[i][j]);
      }
    }
#pragma unroll
    for (int p = 3; p > 0; --p)
#pragma unroll
      for (int j = 0; j < p; ++j) y[j] = fma(-y[p], q[p][j], y[j]);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      double w = y[0] * rr[b][0];  // row lq of Q^-1 R
#pragma unroll
      for (int k = 1; k < 4; ++k) w = fma(y[k], rr[b][k], w);
#pragma unroll
      for (int a = 0; a < 2; ++a) m[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(-c[a], w, m[a][b], 0, 0, 0);
      if (own_r) m[ta][b][s % 4] = w;
    }
  }
}

// the inverse of a tile in that layout, its entries beyond kk x kk replaced by the identity, into P (zero
// beyond kk x kk: the panel products read full tiles)
__device__ inline void gj_invert_into(gj_d4 (&m)[2][2], double* sh, int kk, int tid, double* __restrict__ P) {
  const int lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
  auto each = [&](auto f) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          f(a, b, r, (wave >> 1) * 32 + 16 * a + 4 * r + lq, (wave & 1) * 32 + 16 * b + l16);
  };
  each([&](int a, int b, int r, int row, int col) {
    if (row >= kk || col >= kk) m[a][b][r] = row == col ? 1.0 : 0.0;
  });
  gj_invert_tile(m, sh, tid);
  each([&](int a, int b, int r, int row, int col) {
    P[row * GJB + col] = (row < kk && col < kk) ? m[a][b][r] : 0.0;
  });
}

// Panel copies and inverse of the first diagonal tile: block 0 inverts, block 1 + t copies tile t of the row
// panel, block 1 + nb + t tile t of the column panel.  C[i][c] = A[i][k0 + c], R[r][j] = A[k0 + r][j].
__global__ void __launch_bounds__(256, 2) gj_first_kernel(long long n, int nb, const double* __restrict__ A,
                                                       double* __restrict__ P, double* __restrict__ C,
                                                       double* __restrict__ R) {
  __shared__ double sh[kGjShared];
  const int tid = threadIdx.x, kk = (int)(n < GJB ? n : GJB);
  if (blockIdx.x == 0) {
    gj_d4 m[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = (tid >> 7) * 32 + 16 * a + 4 * r + ((tid & 63) >> 4);
          const int col = ((tid >> 6) & 1) * 32 + 16 * b + (tid & 15);
          m[a][b][r] = (row < kk && col < kk) ? A[row * n + col] : 0.0;
        }
    gj_invert_into(m, sh, kk, tid, P);
    return;
  }
  const bool col = (int)blockIdx.x > nb;
  const long long o0 = (long long)((blockIdx.x - 1) % nb) * GJB;
  for (int q = tid; q < GJB * GJB; q += 256) {
    const int r = q / GJB, c = q % GJB;
    const long long i = col ? o0 + r : r, j = col ? c : o0 + c;
    const double v = (i < n && j < n) ? A[i * n + j] : 0.0;
    if (col && i < n) C[i * GJB + c] = v;
    if (!col && j < n) R[r * n + j] = v;
  }
}

// index of the first tile of row bi among the tiles on and above the diagonal
__device__ inline int gj_row_start(int bi, int nb) { return bi * nb - bi * (bi - 1) / 2; }

template <bool SYM>
__global__ void __launch_bounds__(256, 2)
gj_step_kernel(long long n, int nb, int k, double* __restrict__ A, const double* __restrict__ P, double* __restrict__ Pn,
               const double* __restrict__ C, double* __restrict__ Cn, const double* __restrict__ R,
               double* __restrict__ Rn) {
  __shared__ double sA[GJB * GJL];
  __shared__ double sB[GJB * GJL];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  // the next diagonal tile, with the inversion after its update, goes first
  int t = blockIdx.x;
  if (k + 1 < nb) {
    const int next = SYM ? gj_row_start(k + 1, nb) : (k + 1) * nb + k + 1;
    t = t == 0 ? next : t == next ? 0 : t;
  }
  int bi = t / nb, bj = t % nb;
  if (SYM) {  // the largest row that starts at or before t
    bi = (int)((2 * nb + 1 - sqrtf((float)((2 * nb + 1) * (2 * nb + 1) - 8 * t))) * 0.5f);
    bi = max(0, min(bi, nb - 1));
    while (bi > 0 && gj_row_start(bi, nb) > t) --bi;
    while (bi + 1 < nb && gj_row_start(bi + 1, nb) <= t) ++bi;
    bj = bi + t - gj_row_start(bi, nb);
  }
  const bool row_k = bi == k, col_k = bj == k;
  const long long i0 = (long long)bi * GJB, j0 = (long long)bj * GJB;
  // 64 x 64 tile of a row-major array, zero beyond rows x cols: all 16 loads of a thread in flight at once
  constexpr int PER = GJB * GJB / 256;
  auto fetch = [&](double (&d)[PER], const double* src, long long ld, long long rows, long long cols) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int r = (tid + 256 * u) / GJB, c = tid % GJB;
      d[u] = (r < rows && c < cols) ? src[r * ld + c] : 0.0;
    }
  };
  auto put = [&](double* dst, const double (&d)[PER]) {
#pragma unroll
    for (int u = 0; u < PER; ++u) dst[(tid + 256 * u) / GJB * GJL + tid % GJB] = d[u];
  };
  gj_d4 acc[2][2];
  // acc = sA sB, a wave per 32 x 32 quadrant (A: row l16, entry lq; B: entry lq, column l16; transposed: sB holds B^T)
  auto product = [&](auto transposed) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = gj_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int k4 = 0; k4 < GJB; k4 += 4) {
      double x[2], y[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) x[a] = sA[(wr + 16 * a + l16) * GJL + k4 + lq];
#pragma unroll
      for (int b = 0; b < 2; ++b)
        y[b] = transposed ? sB[(wc + 16 * b + l16) * GJL + k4 + lq] : sB[(k4 + lq) * GJL + wc + 16 * b + l16];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[a], y[b], acc[a][b], 0, 0, 0);
    }
  };
  double tp[PER], tr[PER], tc[PER];
  fetch(tp, P, GJB, GJB, GJB);
  if (!col_k) {
    if (SYM)
      fetch(tr, C + j0 * GJB, GJB, n - j0, GJB);
    else
      fetch(tr, R + j0, n, GJB, n - j0);
  }
  // entry r of acc[a][b]: row wr + 16 a + 4 r + lq, column wc + 16 b + l16
  gj_d4 v[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long long i = i0 + wr + 16 * a + 4 * r + lq, j = j0 + wc + 16 * b + l16;
        v[a][b][r] = (!row_k && !col_k && i < n && j < n) ? A[i * n + j] : 0.0;
      }
  if (!row_k) fetch(tc, C + i0 * GJB, GJB, n - i0, GJB);
  if (!col_k) {
    put(sA, tp);
    put(sB, tr);
    __syncthreads();
    product(std::integral_constant<bool, SYM>());  // P R_j (SYM: up to the sign)
    __syncthreads();
  }
  if (!row_k) {
    put(sA, tc);
    if (col_k) {
      put(sB, tp);
    } else {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) sB[(wr + 16 * a + 4 * r + lq) * GJL + wc + 16 * b + l16] = acc[a][b][r];
    }
    __syncthreads();
    product(std::false_type());
    const double sign = SYM && bj < k ? 1.0 : -1.0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) v[a][b] += sign * acc[a][b];
  } else {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[a][b][r] = col_k ? P[(wr + 16 * a + 4 * r + lq) * GJB + wc + 16 * b + l16] : acc[a][b][r];
  }
  const bool next_row = bi == k + 1, next_col = bj == k + 1;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int lr = wr + 16 * a + 4 * r + lq, lc = wc + 16 * b + l16;
        const long long i = i0 + lr, j = j0 + lc;
        if (i < n && j < n) A[i * n + j] = v[a][b][r];
        if (SYM) {
          if (next_col && i < n) Cn[i * GJB + lc] = v[a][b][r];
          if (next_row && !next_col && j < n) Cn[j * GJB + lr] = v[a][b][r];
          if (k + 1 == nb && bi != bj && i < n && j < n) A[j * n + i] = v[a][b][r];
        } else {
          if (next_row && j < n) Rn[lr * n + j] = v[a][b][r];
          if (next_col && i < n) Cn[i * GJB + lc] = v[a][b][r];
        }
      }
  if (!(next_row && next_col)) return;
  __syncthreads();  // sB was read by the last product
  gj_invert_into(v, sB, (int)(n - i0 < GJB ? n - i0 : GJB), tid, Pn);
}

// y = A x, one 64-lane wave per row, FP64 sums; IO double, or float (the FP64 coarsest inverse applied to an FP32
// right-hand side: the widening, the product and the rounding in one).  Each lane has 8 entries of its row in
// flight.  1911 unknowns: 7.1 us (12.3 us with the loads left to the loop), 847: 3.7 (6.6).
// Up to NC of the `cols` columns x, y per block share a row's entries.
template <typename T, typename IO, int NC>
__global__ void __launch_bounds__(256) gemv_kernel(long long n, int cols, const T* __restrict__ A,
                                                   const IO* __restrict__ x, IO* __restrict__ y) {
  const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= n) return;
  const int col0 = (int)blockIdx.y * NC;
  const T* a = A + row * n;
  const IO* xc[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) xc[k] = x + n * min(col0 + k, cols - 1);
  T s[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) s[k] = 0;
  long long c = lane;
  for (; c + 7 * 64 < n; c += 8 * 64) {
    T v[8];
    IO w[NC][8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[u] = a[c + 64 * u];
#pragma unroll
      for (int k = 0; k < NC; ++k) w[k][u] = xc[k][c + 64 * u];
    }
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int u = 0; u < 8; ++u) s[k] = fma(v[u], (T)w[k][u], s[k]);
  }
  T v[7];
  IO w[NC][7];
#pragma unroll
  for (int u = 0; u < 7; ++u) {
    const bool in = c + 64 * u < n;
    v[u] = in ? a[c + 64 * u] : (T)0;
#pragma unroll
    for (int k = 0; k < NC; ++k) w[k][u] = in ? xc[k][c + 64 * u] : (IO)0;
  }
#pragma unroll
  for (int k = 0; k < NC; ++k) {
#pragma unroll
    for (int u = 0; u < 7; ++u)
      if (c + 64 * u < n) s[k] = fma(v[u], (T)w[k][u], s[k]);
    for (int off = 32; off > 0; off >>= 1) s[k] += __shfl_down(s[k], off, 64);
    if (lane == 0 && col0 + k < cols) y[n * (col0 + k) + row] = (IO)s[k];
  }
}

template <typename T, typename IO>
static void launch_gemv_t(long long n, const T* A, const IO* x, IO* y, int cols, hipStream_t s) {
  if (cols == 1)
    gemv_kernel<T, IO, 1><<<blocks_for(n, 4), 256, 0, s>>>(n, cols, A, x, y);
  else
    gemv_kernel<T, IO, 4><<<dim3(blocks_for(n, 4), (cols + 3) / 4), 256, 0, s>>>(n, cols, A, x, y);
}

// y = (float) x
__global__ void to_float_kernel(long long n, const double* __restrict__ x, float* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (float)x[i];
}

void galerkin_child_matrices(int dim, const double* K0, double* G) {
  const int NN = 1 << dim, NE = NN * dim;
  for (int c = 0; c < NN; ++c) {
    double* g = G + (long long)c * NE * NE;
    for (int q = 0; q < NE * NE; ++q) g[q] = 0.0;
    // G_c[A d][B d2] = sum_{a, b} p_c[a][A] K0[a d][b d2] p_c[b][B]
    for (int A = 0; A < NN; ++A)
      for (int B = 0; B < NN; ++B)
        for (int a = 0; a < NN; ++a) {
          const double wa = dim == 3 ? pweight<3>(c, a, A) : pweight<2>(c, a, A);
          if (wa == 0.0) continue;
          for (int b = 0; b < NN; ++b) {
            const double wb = dim == 3 ? pweight<3>(c, b, B) : pweight<2>(c, b, B);
            if (wb == 0.0) continue;
            for (int d = 0; d < dim; ++d)
              for (int d2 = 0; d2 < dim; ++d2)
                g[(A * dim + d) * NE + B * dim + d2] += wa * wb * K0[(a * dim + d) * NE + b * dim + d2];
          }
        }
  }
}

int launch_galerkin_fine(const GridDims& gf, const double* K0, const double* xe, const uint8_t* bcm, double bcdiag,
                         double* Kc, hipStream_t s) {
  GridDims gc = make_grid(gf.ex / 2, gf.ey / 2, gf.dim == 3 ? gf.ez / 2 : 0);
  if (gf.dim == 3)
    galerkin_kernel<3, true><<<(unsigned)gc.nel, 64, 0, s>>>(gf, gc, K0, xe, bcm, bcdiag, nullptr, Kc, 0);
  else
    galerkin_kernel<2, true><<<(unsigned)gc.nel, 16, 0, s>>>(gf, gc, K0, xe, bcm, bcdiag, nullptr, Kc, 0);
  return check_launch("galerkin_kernel<fine>");
}

int launch_level1_flags(const GridDims& gf, const uint8_t* bcm, uint8_t* cflag, int* list, int* map, hipStream_t s) {
  GridDims gc = make_grid(gf.ex / 2, gf.ey / 2, gf.ez / 2);
  int* count = list + gc.nel;
  zero_int(count, s);
  galerkin_bc_flags_kernel<<<blocks_for(gc.nel, 256), 256, 0, s>>>(gf, gc, bcm, cflag, list, count, map);
  return check_launch("galerkin_bc_flags_kernel");
}

int launch_level1_dk(const GridDims& gf, const double* K0, const double* xe, const uint8_t* bcm, double bcdiag,
                     const uint8_t* cflag, const int* list, int nlist, double* dK, hipStream_t s) {
  if (nlist <= 0) return PMT_OK;
  GridDims gc = make_grid(gf.ex / 2, gf.ey / 2, gf.ez / 2);
  galerkin_fine_bc_kernel<<<(unsigned)nlist, 64, 0, s>>>(gf, gc, K0, xe, bcm, bcdiag, cflag, list, dK);
  return check_launch("galerkin_fine_bc_kernel");
}

int launch_galerkin_coarse(const GridDims& gf, const double* Kf, double* Kc, hipStream_t s) {
  GridDims gc = make_grid(gf.ex / 2, gf.ey / 2, gf.dim == 3 ? gf.ez / 2 : 0);
  if (gf.dim == 3)
    galerkin_kernel<3, false><<<(unsigned)gc.nel, 64, 0, s>>>(gf, gc, nullptr, nullptr, nullptr, 0.0, Kf, Kc, 0);
  else
    galerkin_kernel<2, false><<<(unsigned)gc.nel, 16, 0, s>>>(gf, gc, nullptr, nullptr, nullptr, 0.0, Kf, Kc, 0);
  return check_launch("galerkin_kernel<coarse>");
}

int launch_stencil_from_fine(const GridDims& gf, const double* G, const double* xe, const uint8_t* cflag,
                             const int* map, const double* dK, const StencilOut& out, hipStream_t s) {
  GridDims gc = make_grid(gf.ex / 2, gf.ey / 2, gf.ez / 2);
  if (out.S)
    stencil_from_fine_kernel<0><<<blocks_for(gc.nnodes, 256), 256, 0, s>>>(gf, gc, G, xe, cflag, map, dK, out);
  else if (out.H)
    stencil_from_fine_kernel<1><<<blocks_for(gc.nnodes, 256), 256, 0, s>>>(gf, gc, G, xe, cflag, map, dK, out);
  else
    stencil_from_fine_kernel<2><<<blocks_for(gc.nnodes, 256), 256, 0, s>>>(gf, gc, G, xe, cflag, map, dK, out);
  return check_launch("stencil_from_fine_kernel");
}

int launch_stencil_from_elements(const GridDims& g, const double* Ke, double* S, hipStream_t s) {
  dim3 grid(blocks_for(g.nnodes, 128));
  if (g.dim == 3)
    stencil_from_elements_kernel<3><<<grid, 128, 0, s>>>(g, Ke, S);
  else
    stencil_from_elements_kernel<2><<<grid, 128, 0, s>>>(g, Ke, S);
  return check_launch("stencil_from_elements_kernel");
}

int launch_dense_from_stencil(const GridDims& g, const double* S, double* A, hipStream_t s) {
  const long long N = g.nnodes * g.dim;
  PMT_TRY(launch_fill(N * N, 0.0, A, s));
  dim3 grid(blocks_for(g.nnodes, 128));
  if (g.dim == 3)
    dense_from_stencil_kernel<3><<<grid, 128, 0, s>>>(g, S, A);
  else
    dense_from_stencil_kernel<2><<<grid, 128, 0, s>>>(g, S, A);
  return check_launch("dense_from_stencil_kernel");
}

bool symmetric_matrix(int m, const double* K0) {
  double scale = 0.0, skew = 0.0;
  for (int i = 0; i < m; ++i)
    for (int j = 0; j < m; ++j) {
      scale = std::max(scale, std::fabs(K0[i * m + j]));
      skew = std::max(skew, std::fabs(K0[i * m + j] - K0[j * m + i]));
    }
  return skew <= 1e-14 * scale;
}

int gj_invert(long long n, bool symmetric, double* A, double* ws, hipStream_t s) {
  const int nb = (int)((n + GJB - 1) / GJB);
  double *P[2], *C[2], *R[2];
  for (int h = 0; h < 2; ++h) {  // this panel's and the next one's
    P[h] = ws + h * GJB * GJB;
    C[h] = ws + 2 * GJB * GJB + h * n * GJB;
    R[h] = ws + 2 * GJB * GJB + (2 + h) * n * GJB;
  }
  gj_first_kernel<<<1 + 2 * nb, 256, 0, s>>>(n, nb, A, P[0], C[0], R[0]);
  PMT_TRY(check_launch("gj_first_kernel"));
  for (int k = 0; k < nb; ++k) {
    const int h = k & 1;
    if (symmetric)
      gj_step_kernel<true><<<nb * (nb + 1) / 2, 256, 0, s>>>(n, nb, k, A, P[h], P[1 - h], C[h], C[1 - h], nullptr,
                                                             nullptr);
    else
      gj_step_kernel<false><<<nb * nb, 256, 0, s>>>(n, nb, k, A, P[h], P[1 - h], C[h], C[1 - h], R[h], R[1 - h]);
    PMT_TRY(check_launch("gj_step_kernel"));
  }
  return PMT_OK;
}

template <typename T>
int launch_gemv(long long n, const T* A, const T* x, T* y, hipStream_t s, int cols) {
  launch_gemv_t<T, T>(n, A, x, y, cols, s);
  return check_launch("gemv_kernel");
}
template int launch_gemv<double>(long long, const double*, const double*, double*, hipStream_t, int);
template int launch_gemv<float>(long long, const float*, const float*, float*, hipStream_t, int);

int launch_gemv_f32io(long long n, const double* A, const float* x, float* y, hipStream_t s, int cols) {
  launch_gemv_t<double, float>(n, A, x, y, cols, s);
  return check_launch("gemv_kernel<double, float>");
}

// y = (float) x and u1 = w * dinv * y: an FP32 V-cycle's right-hand side and its first fine sweep from zero
// (the expression of jacobi0_kernel)
__global__ void to_float_first_kernel(long long n, const double* __restrict__ x, float* __restrict__ y,
                                      const float* __restrict__ dinv, float w, float* __restrict__ u1) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const long long c = blockIdx.y * n + i;
    const float v = (float)x[c];
    y[c] = v;
    u1[c] = w * dinv[i] * v;
  }
}

int launch_to_float_first(long long n, const double* x, float* y, const float* dinv, float w, float* u1,
                          hipStream_t s, int cols) {
  if (n <= 0) return PMT_OK;
  to_float_first_kernel<<<dim3(blocks_for(n, 256), cols), 256, 0, s>>>(n, x, y, dinv, w, u1);
  return check_launch("to_float_first_kernel");
}

int launch_to_float(long long n, const double* x, float* y, hipStream_t s) {
  if (n <= 0) return PMT_OK;
  to_float_kernel<<<blocks_for(n, 256), 256, 0, s>>>(n, x, y);
  return check_launch("to_float_kernel");
}

}  // namespace pmt
