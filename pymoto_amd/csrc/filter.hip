// FilterConv forward and adjoint (pymoto/modules/filter.py:8-220).
//
// The reference pads an element-index array axis by axis with numpy padding modes and then
// convolves.  Padding an index array along one axis applies the same 1-D index map to every
// line, so the padded field is xpad[a,b,c] = x[mx[a], my[b], mz[c]] with one small map per axis
// (built on the host at setup); constant-padded cells carry map = -1 and a value, with the later
// axis winning at corners as the reference's override order does.  Forward: one thread per element
// gathers the kx*ky*kz window ('valid' convolution).  Adjoint: one thread per element visits the
// padded cells that map onto it (per-axis inverse lists; interior elements have exactly one) and
// evaluates the 'full' correlation there - a gather, so no atomics and a deterministic sum.
#include <algorithm>
#include <type_traits>

#include "launch.h"

namespace pmt {

__global__ void __launch_bounds__(256)
filter_fwd_kernel(int nx, int ny, int nz, int kx, int ky, int kz, const double* __restrict__ w,
                  const int32_t* __restrict__ map, const double* __restrict__ cval, const double* __restrict__ x,
                  double* __restrict__ y) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nel = (long long)nx * ny * nz;
  if (e >= nel) return;
  const int i = (int)(e % nx);
  const long long t = e / nx;
  const int j = (int)(t % ny);
  const int k = (int)(t / ny);
  const int Lx = nx + kx - 1, Ly = ny + ky - 1;
  const int32_t* mx = map;
  const int32_t* my = map + Lx;
  const int32_t* mz = map + Lx + Ly;
  const double* cx = cval;
  const double* cy = cval + Lx;
  const double* cz = cval + Lx + Ly;
  double acc = 0.0;
  for (int r = 0; r < kz; ++r) {
    const int c = k + kz - 1 - r;
    const int mc = mz[c];
    for (int q = 0; q < ky; ++q) {
      const int b = j + ky - 1 - q;
      const int mb = my[b];
      for (int p = 0; p < kx; ++p) {
        const int a = i + kx - 1 - p;
        const int ma = mx[a];
        double v;
        if (mc < 0)
          v = cz[c];
        else if (mb < 0)
          v = cy[b];
        else if (ma < 0)
          v = cx[a];
        else
          v = x[((long long)mc * ny + mb) * nx + ma];
        acc = fma(w[((long long)p * ky + q) * kz + r], v, acc);
      }
    }
  }
  y[e] = acc;
}

__global__ void __launch_bounds__(256)
filter_bwd_kernel(int nx, int ny, int nz, int kx, int ky, int kz, const double* __restrict__ w,
                  const int32_t* __restrict__ inv_ptr, const int32_t* __restrict__ inv_idx,
                  const double* __restrict__ dy, double* __restrict__ dx) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nel = (long long)nx * ny * nz;
  if (e >= nel) return;
  const int i = (int)(e % nx);
  const long long t = e / nx;
  const int j = (int)(t % ny);
  const int k = (int)(t / ny);
  const int32_t* px = inv_ptr;
  const int32_t* py = inv_ptr + (nx + 1);
  const int32_t* pz = inv_ptr + (nx + 1) + (ny + 1);
  double acc = 0.0;
  for (int ic = pz[k]; ic < pz[k + 1]; ++ic) {
    const int c = inv_idx[ic];
    for (int ib = py[j]; ib < py[j + 1]; ++ib) {
      const int b = inv_idx[ib];
      for (int ia = px[i]; ia < px[i + 1]; ++ia) {
        const int a = inv_idx[ia];
        double cell = 0.0;  // correlate 'full' at padded cell (a, b, c)
        for (int r = 0; r < kz; ++r) {
          const int cc = c - (kz - 1) + r;
          if (cc < 0 || cc >= nz) continue;
          for (int q = 0; q < ky; ++q) {
            const int bb = b - (ky - 1) + q;
            if (bb < 0 || bb >= ny) continue;
            for (int p = 0; p < kx; ++p) {
              const int aa = a - (kx - 1) + p;
              if (aa < 0 || aa >= nx) continue;
              cell = fma(w[((long long)p * ky + q) * kz + r], dy[((long long)cc * ny + bb) * nx + aa], cell);
            }
          }
        }
        acc += cell;
      }
    }
  }
  dx[e] = acc;
}

// The same two kernels with the kernel extents fixed at compile time (KXY x KXY x KZ, the shapes that
// FilterConv builds from a radius): the per-axis maps are read once per element and the KXY^2 KZ taps
// are unrolled, so every load of a thread is independent and in flight at once (the general kernels
// chain them through their loops).  Same summation order as the general kernels.
template <int KXY, int KZ>
__global__ void __launch_bounds__(256)
filter_fwd_fixed_kernel(int nx, int ny, int nz, const double* __restrict__ w, const int32_t* __restrict__ map,
                        const double* __restrict__ cval, const double* __restrict__ x, double* __restrict__ y) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nel = (long long)nx * ny * nz;
  if (e >= nel) return;
  const int i = (int)(e % nx);
  const long long t = e / nx;
  const int j = (int)(t % ny);
  const int k = (int)(t / ny);
  const int Lx = nx + KXY - 1, Ly = ny + KXY - 1;
  int ma[KXY], mb[KXY], mc[KZ];
#pragma unroll
  for (int p = 0; p < KXY; ++p) ma[p] = map[i + KXY - 1 - p];
#pragma unroll
  for (int q = 0; q < KXY; ++q) mb[q] = map[Lx + j + KXY - 1 - q];
#pragma unroll
  for (int r = 0; r < KZ; ++r) mc[r] = map[Lx + Ly + k + KZ - 1 - r];
  double acc = 0.0;
#pragma unroll
  for (int r = 0; r < KZ; ++r)
#pragma unroll
    for (int q = 0; q < KXY; ++q)
#pragma unroll
      for (int p = 0; p < KXY; ++p) {
        double v;
        if (mc[r] < 0)
          v = cval[Lx + Ly + k + KZ - 1 - r];
        else if (mb[q] < 0)
          v = cval[Lx + j + KXY - 1 - q];
        else if (ma[p] < 0)
          v = cval[i + KXY - 1 - p];
        else
          v = x[((long long)mc[r] * ny + mb[q]) * nx + ma[p]];
        acc = fma(w[(p * KXY + q) * KZ + r], v, acc);
      }
  y[e] = acc;
}

// The element's padded cells are exactly its own position shifted by the half widths (the element is at
// least (K-1)/2 from every mirrored, replicated or wrapped face, or the padding is constant).
__device__ inline bool filter_single_cell(const int32_t* __restrict__ inv_ptr, const int32_t* __restrict__ inv_idx,
                                          int nx, int ny, int hx, int hz, int i, int j, int k) {
  const int32_t* px = inv_ptr;
  const int32_t* py = inv_ptr + (nx + 1);
  const int32_t* pz = inv_ptr + (nx + 1) + (ny + 1);
  return px[i + 1] - px[i] == 1 && inv_idx[px[i]] == i + hx && py[j + 1] - py[j] == 1 &&
         inv_idx[py[j]] == j + hx && pz[k + 1] - pz[k] == 1 && inv_idx[pz[k]] == k + hz;
}

// The 'full' correlation of dy at padded cell (a, b, c), the taps in the order r, q, p.  The loads of a
// plane of taps are issued together, with the address of a tap outside the grid clamped to 0 (a branch
// around each load would wait for every one of them in turn).
template <int KXY, int KZ>
__device__ inline double filter_bwd_cell(int nx, int ny, int nz, const double* __restrict__ w,
                                         const double* __restrict__ dy, int a, int b, int c) {
  double acc = 0.0;
#pragma unroll(KXY <= 3 ? KZ : 1)
  for (int r = 0; r < KZ; ++r) {
    const int cc = c - (KZ - 1) + r;
    double v[KXY][KXY];
    bool in[KXY][KXY];
#pragma unroll
    for (int q = 0; q < KXY; ++q) {
      const int bb = b - (KXY - 1) + q;
      const bool row = cc >= 0 && cc < nz && bb >= 0 && bb < ny;
      const long long base = row ? ((long long)cc * ny + bb) * nx : 0;
#pragma unroll
      for (int p = 0; p < KXY; ++p) {
        const int aa = a - (KXY - 1) + p;
        in[q][p] = row && aa >= 0 && aa < nx;
        v[q][p] = dy[in[q][p] ? base + aa : 0];
      }
    }
#pragma unroll
    for (int q = 0; q < KXY; ++q)
#pragma unroll
      for (int p = 0; p < KXY; ++p) {
        const double t = fma(w[(p * KXY + q) * KZ + r], v[q][p], acc);
        acc = in[q][p] ? t : acc;
      }
  }
  return acc;
}

// dx_e of element (i, j, k) by its inverse lists: the sum, in list order, of the correlation at every
// padded cell that maps onto it
template <int KXY, int KZ>
__device__ inline double filter_bwd_gather(int nx, int ny, int nz, const double* __restrict__ w,
                                           const int32_t* __restrict__ inv_ptr, const int32_t* __restrict__ inv_idx,
                                           const double* __restrict__ dy, int i, int j, int k) {
  const int32_t* px = inv_ptr;
  const int32_t* py = inv_ptr + (nx + 1);
  const int32_t* pz = inv_ptr + (nx + 1) + (ny + 1);
  double acc = 0.0;
  for (int ic = pz[k]; ic < pz[k + 1]; ++ic)
    for (int ib = py[j]; ib < py[j + 1]; ++ib)
      for (int ia = px[i]; ia < px[i + 1]; ++ia)
        acc += filter_bwd_cell<KXY, KZ>(nx, ny, nz, w, dy, inv_idx[ia], inv_idx[ib], inv_idx[ic]);
  return acc;
}

template <int KXY, int KZ>
__global__ void __launch_bounds__(256)
filter_bwd_fixed_kernel(int nx, int ny, int nz, const double* __restrict__ w, const int32_t* __restrict__ inv_ptr,
                        const int32_t* __restrict__ inv_idx, const double* __restrict__ dy, double* __restrict__ dx) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nel = (long long)nx * ny * nz;
  if (e >= nel) return;
  const int i = (int)(e % nx);
  const long long t = e / nx;
  const int j = (int)(t % ny);
  const int k = (int)(t / ny);
  dx[e] = filter_bwd_gather<KXY, KZ>(nx, ny, nz, w, inv_ptr, inv_idx, dy, i, j, k);
}

// Cell t of the shell of half widths hx (x and y) and hz of an nx x ny x nz box, in three disjoint slab sets
// - x slabs (all j, k), y slabs (interior i), z slabs (interior i, j).  False past the last.
__device__ inline bool shell_cell(long long t, int nx, int ny, int nz, int hx, int hz, int& i, int& j, int& k) {
  const int wx = min(nx, 2 * hx), wy = min(ny, 2 * hx), wz = min(nz, 2 * hz);
  const long long cx = (long long)wx * ny * nz, cy = (long long)(nx - wx) * wy * nz;
  const long long cz = (long long)(nx - wx) * (ny - wy) * wz;
  // slab index a of width wa on an axis of extent n: the first half-width, then the last
  auto side = [](int a, int wa, int n, int h) { return (a < h || wa == n) ? a : n - wa + a; };
  if (t < cx) {
    i = side((int)(t % wx), wx, nx, hx);
    t /= wx;
    j = (int)(t % ny);
    k = (int)(t / ny);
  } else if ((t -= cx) < cy) {
    i = wx / 2 + (int)(t % (nx - wx));
    t /= (nx - wx);
    j = side((int)(t % wy), wy, ny, hx);
    k = (int)(t / wy);
  } else if ((t -= cy) < cz) {
    i = wx / 2 + (int)(t % (nx - wx));
    t /= (nx - wx);
    j = wy / 2 + (int)(t % (ny - wy));
    k = side((int)(t / (ny - wy)), wz, nz, hz);
  } else {
    return false;
  }
  return true;
}

inline long long shell_cells(long long nx, long long ny, long long nz, int hx, int hz) {
  const long long wx = std::min(nx, 2LL * hx), wy = std::min(ny, 2LL * hx), wz = std::min(nz, 2LL * hz);
  return wx * ny * nz + (nx - wx) * wy * nz + (nx - wx) * (ny - wy) * wz;
}

// The elements with more than one padded cell (mirrored, replicated or wrapped cells map there) lie within
// the half widths of a face with every padding mode.  With a workspace g of the padded extents the box
// kernel evaluates the correlation once per padded cell and filter_bwd_fold_kernel adds up each such
// element's cells, eight loads at a time: an element in a corner has 8 (symmetric) to 64 (edge, 7^3) of
// them, and walking those with all their taps in one thread bounded the whole adjoint (21.6 us of 49 at
// 256x128x128 with 3^3; 461 us at 75x51x33 with 7^3).  Without a workspace the list walk stays
// (filter_bwd_shell_kernel).
__global__ void __launch_bounds__(256)
filter_bwd_fold_kernel(int nx, int ny, int nz, int kxy, int kz, const int32_t* __restrict__ inv_ptr,
                       const int32_t* __restrict__ inv_idx, const double* __restrict__ g, double* __restrict__ dx) {
  const int hx = (kxy - 1) / 2, hz = (kz - 1) / 2;
  int i, j, k;
  if (!shell_cell((long long)blockIdx.x * blockDim.x + threadIdx.x, nx, ny, nz, hx, hz, i, j, k)) return;
  if (filter_single_cell(inv_ptr, inv_idx, nx, ny, hx, hz, i, j, k)) return;
  const int32_t* px = inv_ptr + i;
  const int32_t* py = inv_ptr + (nx + 1) + j;
  const int32_t* pz = inv_ptr + (nx + 1) + (ny + 1) + k;
  const int pa = px[0], pb = py[0], pc = pz[0];
  const int na = px[1] - pa, nb = py[1] - pb, nc = pz[1] - pc, cells = na * nb * nc;
  const long long lx = nx + kxy - 1, ly = ny + kxy - 1;
  double acc = 0.0;
  // counted up instead of divided out of t: 75x51x33 with 7^3 8.9 us (two divisions per cell: 13.5), 256x128x128 with
  // 3^3 5.8 (7.2)
  int a = 0, b = 0, c = 0;
  for (int t = 0; t < cells; t += 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[u] = g[(inv_idx[pc + min(c, nc - 1)] * ly + inv_idx[pb + b]) * lx + inv_idx[pa + a]];
      ++a;
      b += a == na;
      a = a == na ? 0 : a;
      c += b == nb;
      b = b == nb ? 0 : b;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = t + u < cells ? acc + v[u] : acc;
  }
  dx[((long long)k * ny + j) * nx + i] = acc;
}

template <int KXY, int KZ>
__global__ void __launch_bounds__(256)
filter_bwd_shell_kernel(int nx, int ny, int nz, const double* __restrict__ w, const int32_t* __restrict__ inv_ptr,
                        const int32_t* __restrict__ inv_idx, const double* __restrict__ dy, double* __restrict__ dx) {
  int i, j, k;
  constexpr int HX = (KXY - 1) / 2, HZ = (KZ - 1) / 2;
  if (!shell_cell((long long)blockIdx.x * blockDim.x + threadIdx.x, nx, ny, nz, HX, HZ, i, j, k)) return;
  if (filter_single_cell(inv_ptr, inv_idx, nx, ny, HX, HZ, i, j, k)) return;
  dx[((long long)k * ny + j) * nx + i] = filter_bwd_gather<KXY, KZ>(nx, ny, nz, w, inv_ptr, inv_idx, dy, i, j, k);
}

int g_filter_tiled = 1;  // PMT_TUNE_FILTER: 1 boxes in LDS (default), 0 per-element gathers

// Box kernels (KXY x KXY x kz): the whole window of a box of outputs in LDS at once.  256 threads as
// 32 x nty x ntz, a thread the column of OY outputs above its row; per z tap the OY rows it needs slide by
// one per y tap, so a value is read from LDS once per z tap for OY outputs.  The weights of a z tap lie one
// per lane and are broadcast through scalar registers (v_readlane; as scalar loads, KXY^2 strided ones per z
// tap, each wait also drained the LDS reads).  The taps are summed in the order of the gather kernels (r,
// then q, then p): the same bits.  FWD: outputs are elements, the box holds their padded cells, resolved
// through the maps.  Adjoint: outputs are the padded cells, the box holds dy (zero outside the grid); the
// cell of an element without other cells is its result, every other one goes to the workspace g (if given)
// for filter_bwd_fold_kernel.
// Forward / adjoint with its fold: 22.9 / 34.2 us at 256x128x128 with 3^3, 14.8 / 23.3 us at 75x51x33 with 7^3 (with a
// branch around each load of the box 23.2 / 35.3 and 15.2 / 24.1).  A ring of LDS planes streamed in z took 26.3 / 47.6 and 62.9 / 151 us
// (5^3 held 450 registers, one wave per SIMD), the per-element gathers 69 / 165 us for 7^3 (which the adjoint
// without a workspace still takes).
template <int KXY, int OY, bool FWD>
__global__ void __launch_bounds__(256)
filter_box_kernel(int nx, int ny, int nz, int kz, int nty, int tiles_x, int tiles_y, unsigned m_ly,
                   const double* __restrict__ w, const int32_t* __restrict__ m0, const int32_t* __restrict__ m1,
                   const double* __restrict__ cval, const double* __restrict__ in, double* __restrict__ out,
                   double* __restrict__ g) {
  constexpr int HX = (KXY - 1) / 2, LX = 32 + KXY - 1, NW = (KXY * KXY + 63) / 64;
  extern __shared__ double box[];
  const int ntz = 8 / nty, hz = (kz - 1) / 2, ly = OY * nty + KXY - 1, lz = ntz + kz - 1;
  const int tid = threadIdx.x, lane = tid & 63, tx = tid & 31, ty = (tid >> 5) % nty, tz = (tid >> 5) / nty;
  const int tile = blockIdx.x % (tiles_x * tiles_y);
  const int i0 = (tile % tiles_x) * 32, j0 = (tile / tiles_x) * OY * nty, k0 = (blockIdx.x / (tiles_x * tiles_y)) * ntz;
  const int plx = nx + KXY - 1, ply = ny + KXY - 1, plz = nz + kz - 1;
  const int nbox = LX * ly * lz;
  // source index of the box's columns, rows and planes: >= 0 inside, -1 constant padding, -2 nothing (0)
  int* sx = (int*)(box + nbox);
  int* sy = sx + LX;
  int* sz = sy + ly;
  // adjoint: whether the element at an output column, row or plane has only its own cell on that axis
  int* one = sz + lz;
  if (!FWD)
    for (int t = tid; t < 32 + OY * nty + ntz; t += 256) {
      const int ax = t < 32 ? 0 : t < 32 + OY * nty ? 1 : 2;
      const int e = ax == 0 ? i0 + t - HX : ax == 1 ? j0 + t - 32 - HX : k0 + t - 32 - OY * nty - hz;
      const int n = ax == 0 ? nx : ax == 1 ? ny : nz, h = ax == 2 ? hz : HX;
      const int32_t* ptr = m0 + (ax == 0 ? 0 : ax == 1 ? nx + 1 : nx + ny + 2);
      one[t] = e >= 0 && e < n && ptr[e + 1] - ptr[e] == 1 && m1[ptr[e]] == e + h;
    }
  for (int t = tid; t < LX + ly + lz; t += 256) {
    const int ax = t < LX ? 0 : t < LX + ly ? 1 : 2;
    const int q = ax == 0 ? t : ax == 1 ? t - LX : t - LX - ly;
    const int at = (ax == 0 ? i0 : ax == 1 ? j0 : k0) + q, n = ax == 0 ? nx : ax == 1 ? ny : nz;
    const int kk = ax == 2 ? kz : KXY;
    int v;
    if (FWD) {
      v = at < n + kk - 1 ? m0[(ax == 0 ? 0 : ax == 1 ? plx : plx + ply) + at] : -2;
      if (v < -1) v = at < n + kk - 1 ? -1 : -2;
    } else {
      v = at - (kk - 1);
      if (v < 0 || v >= n) v = -2;
    }
    sx[t] = v;
  }
  __syncthreads();
  // 8 values per thread and step: their loads are in flight together, without a branch around any (a cell outside
  // everything reads in[0])
  for (int q0 = tid; q0 < nbox; q0 += 256 * 8) {
    double v[8];
    unsigned keep = 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int q = min(q0 + 256 * u, nbox - 1);
      const int a = q % LX, t = q / LX, c = (int)(((unsigned)t * m_ly) >> 20), b = t - c * ly;
      const int ma = sx[a], mb = sy[b], mc = sz[c];
      const bool inside = (ma | mb | mc) >= 0, fixed = FWD && !inside && ma != -2 && mb != -2 && mc != -2;
      const double* src = fixed ? cval : in;
      const int at = inside ? (mc * ny + mb) * nx + ma
                            : fixed ? (mc < 0 ? plx + ply + k0 + c : mb < 0 ? plx + j0 + b : i0 + a) : 0;
      v[u] = src[at];
      keep |= (inside || fixed ? 1u : 0u) << u;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (q0 + 256 * u < nbox) box[q0 + 256 * u] = (keep >> u) & 1u ? v[u] : 0.0;
  }
  __syncthreads();
  double acc[OY];
#pragma unroll
  for (int o = 0; o < OY; ++o) acc[o] = 0.0;
  double wl[NW], wn[NW];  // weights of this z tap and the next: lane l holds tap (p, q) = (l / KXY, l % KXY)
  auto weights = [&](int r, double (&d)[NW]) {
#pragma unroll
    for (int h = 0; h < NW; ++h) d[h] = 64 * h + lane < KXY * KXY ? w[(64 * h + lane) * kz + r] : 0.0;
  };
  weights(0, wl);
  for (int r = 0; r < kz; ++r) {
    weights(r + 1 < kz ? r + 1 : r, wn);
    const double* pl = box + ((FWD ? tz + kz - 1 - r : tz + r) * ly + ty * OY) * LX + tx;
    double win[OY][KXY];  // row y of the column's window in slot y % OY
    auto load = [&](int y) {
#pragma unroll
      for (int p = 0; p < KXY; ++p) win[y % OY][p] = pl[y * LX + p];
    };
#pragma unroll
    for (int o = 0; o < OY; ++o) load(FWD ? KXY - 1 + o : o);
#pragma unroll
    for (int q = 0; q < KXY; ++q) {
      if (q > 0) load(FWD ? KXY - 1 - q : q + OY - 1);
#pragma unroll
      for (int p = 0; p < KXY; ++p) {
        const int l = p * KXY + q;
        const long long bits = __double_as_longlong(wl[l / 64]);
        const unsigned lo = __builtin_amdgcn_readlane((int)bits, l % 64);
        const unsigned hi = __builtin_amdgcn_readlane((int)(bits >> 32), l % 64);
        const double wt = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
#pragma unroll
        for (int o = 0; o < OY; ++o)
          acc[o] = fma(wt, FWD ? win[(o + KXY - 1 - q) % OY][KXY - 1 - p] : win[(o + q) % OY][p], acc[o]);
      }
    }
#pragma unroll
    for (int h = 0; h < NW; ++h) wl[h] = wn[h];
  }
  const int a = i0 + tx, c = k0 + tz;
  if (a >= (FWD ? nx : plx) || c >= (FWD ? nz : plz)) return;
#pragma unroll
  for (int o = 0; o < OY; ++o) {
    const int b = j0 + ty * OY + o;
    if (b >= (FWD ? ny : ply)) break;
    if (FWD) {
      out[(c * ny + b) * nx + a] = acc[o];
      continue;
    }
    if (one[tx] & one[32 + ty * OY + o] & one[32 + OY * nty + tz])
      out[((c - hz) * ny + b - HX) * nx + a - HX] = acc[o];
    else if (g)
      g[((long long)c * ply + b) * plx + a] = acc[o];
  }
}

struct FilterBox {
  int oy, nty, ly;
  size_t lds;
};

// The box over an lx x ly x lz range of outputs: 32 x 8 x 4 (one plane: 32 x 32) with 4 outputs per thread;
// half as high with 2 while those boxes are too few to give every CU two.  (Twice as high with 8, less halo
// per output: 24.5 instead of 21.4 us for 3^3 forward at 256x128x128.)
inline FilterBox filter_box(int kxy, int kz, long long lx, long long ly, long long lz) {
  FilterBox b;
  b.nty = kz == 1 ? 8 : 2;
  const long long boxes = (lx + 31) / 32 * ((ly + 4 * b.nty - 1) / (4 * b.nty)) * ((lz + 8 / b.nty - 1) / (8 / b.nty));
  b.oy = boxes < 2LL * device_cu_count() ? 2 : 4;
  b.ly = b.oy * b.nty + kxy - 1;
  const int x = 32 + kxy - 1, z = 8 / b.nty + kz - 1;
  b.lds = sizeof(double) * x * b.ly * z + sizeof(int) * (x + b.ly + z + 32 + b.oy * b.nty + 8 / b.nty);
  return b;
}

// whether the box kernels take these extents: equal ones of 3 to 15 in x and y (their weights of a z tap lie one per
// lane), any in z whose box fits: boxes above 64 KB of LDS (3D from 11^3, 3 x 3 x 21 with 4 outputs per thread, 3 x 3 x 37
// with 2) stay with the gather kernels, and so does the adjoint of the kernels above 5 without a workspace
inline bool filter_box_ok(bool fwd, int nx, int ny, int nz, int kx, int ky, int kz, const double* work) {
  if (kx != ky || kx < 3 || kx > 15) return false;
  if (!fwd && !work && !(kx <= 5 && (kz == kx || kz == 1))) return false;
  return (fwd ? filter_box(kx, kz, nx, ny, nz) : filter_box(kx, kz, nx + kx - 1, ny + kx - 1, nz + kz - 1)).lds <= 65536;
}

template <int KXY>
void launch_filter_box_k(bool fwd, int nx, int ny, int nz, int kz, const double* w, const int32_t* m0,
                          const int32_t* m1, const double* cv, const double* in, double* out, double* work,
                          hipStream_t s) {
  const int lx = fwd ? nx : nx + KXY - 1, ly = fwd ? ny : ny + KXY - 1, lz = fwd ? nz : nz + kz - 1;
  const FilterBox b = filter_box(KXY, kz, lx, ly, lz);
  const int ntz = 8 / b.nty, tiles_x = (lx + 31) / 32, tiles_y = (ly + b.oy * b.nty - 1) / (b.oy * b.nty);
  const unsigned blocks = (unsigned)(tiles_x * tiles_y * ((lz + ntz - 1) / ntz));
  // t / ly for t < ly lz as t m_ly >> 20: exact while t ly < 2^20, and 64 KB of LDS in rows of 34 doubles and more hold
  // ly lz <= 240 of them, with ly <= 46
  const unsigned m_ly = (1u << 20) / b.ly + 1;
  auto run = [&](auto kernel) {
    kernel<<<blocks, 256, b.lds, s>>>(nx, ny, nz, kz, b.nty, tiles_x, tiles_y, m_ly, w, m0, m1, cv, in, out, work);
  };
  auto pick = [&](auto is_fwd) {
    constexpr bool F = decltype(is_fwd)::value;
    if (b.oy == 4) return run(filter_box_kernel<KXY, 4, F>);
    run(filter_box_kernel<KXY, 2, F>);
  };
  if (fwd) return pick(std::true_type{});
  pick(std::false_type{});
  const unsigned shell = blocks_for(shell_cells(nx, ny, nz, (KXY - 1) / 2, (kz - 1) / 2), 256);
  if (work) {
    filter_bwd_fold_kernel<<<shell, 256, 0, s>>>(nx, ny, nz, KXY, kz, m0, m1, work, out);
  } else if constexpr (KXY <= 5) {
    if (kz == 1)
      filter_bwd_shell_kernel<KXY, 1><<<shell, 256, 0, s>>>(nx, ny, nz, w, m0, m1, in, out);
    else
      filter_bwd_shell_kernel<KXY, KXY><<<shell, 256, 0, s>>>(nx, ny, nz, w, m0, m1, in, out);
  }
}

void launch_filter_box(bool fwd, int nx, int ny, int nz, int kxy, int kz, const double* w, const int32_t* m0,
                        const int32_t* m1, const double* cv, const double* in, double* out, double* work,
                        hipStream_t s) {
  switch (kxy) {
    case 3: return launch_filter_box_k<3>(fwd, nx, ny, nz, kz, w, m0, m1, cv, in, out, work, s);
    case 5: return launch_filter_box_k<5>(fwd, nx, ny, nz, kz, w, m0, m1, cv, in, out, work, s);
    case 7: return launch_filter_box_k<7>(fwd, nx, ny, nz, kz, w, m0, m1, cv, in, out, work, s);
    case 9: return launch_filter_box_k<9>(fwd, nx, ny, nz, kz, w, m0, m1, cv, in, out, work, s);
    case 11: return launch_filter_box_k<11>(fwd, nx, ny, nz, kz, w, m0, m1, cv, in, out, work, s);
    case 13: return launch_filter_box_k<13>(fwd, nx, ny, nz, kz, w, m0, m1, cv, in, out, work, s);
    default: return launch_filter_box_k<15>(fwd, nx, ny, nz, kz, w, m0, m1, cv, in, out, work, s);
  }
}

// the box kernels index with 32-bit element numbers
inline bool filter_32bit_ok(long long nel) { return g_filter_tiled && nel < (1LL << 31); }

// DensityFilter (pymoto/modules/filter.py:223-378): y_i = so_i * sum_j H_ij (si_j * x_j) over the
// clipped window |j - i|_inf <= int(radius) with H_ij = max(0, radius - |i - j|) in element units.
// Forward: si = 1, so = 1/s; adjoint: si = 1/s, so = 1 (H symmetric); s = H 1 with si = so = 1.
__global__ void density_filter_kernel(int nx, int ny, int nz, double radius, int dxy, int dz,
                                      const double* __restrict__ x, const double* __restrict__ si,
                                      const double* __restrict__ so, double* __restrict__ y) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)nx * ny * nz) return;
  const int i = (int)(e % nx), j = (int)((e / nx) % ny), k = (int)(e / ((long long)nx * ny));
  double acc = 0.0;
  for (int kk = max(k - dz, 0); kk <= min(k + dz, nz - 1); ++kk)
    for (int jj = max(j - dxy, 0); jj <= min(j + dxy, ny - 1); ++jj)
      for (int ii = max(i - dxy, 0); ii <= min(i + dxy, nx - 1); ++ii) {
        const double di = ii - i, dj = jj - j, dk = kk - k;
        const double w = radius - sqrt(di * di + dj * dj + dk * dk);
        if (w <= 0.0) continue;
        const long long m = ((long long)kk * ny + jj) * nx + ii;
        acc = fma(w, si ? si[m] * x[m] : x[m], acc);
      }
  y[e] = so ? acc * so[e] : acc;
}

}  // namespace pmt

using namespace pmt;

extern "C" {

int pmt_filter_fwd(int nelx, int nely, int nelz, int kx, int ky, int kz, const double* w, const int32_t* map,
                   const double* cval, const double* x, double* y, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || kx < 1 || ky < 1 || kz < 1 || !(kx & 1) || !(ky & 1) || !(kz & 1) || !w ||
      !map || !cval || !x || !y)
    return arg_error("pmt_filter_fwd: bad argument");
  const int nz = nelz > 0 ? nelz : 1;
  if (nelz == 0 && kz != 1) return arg_error("pmt_filter_fwd: 2D grid needs kz == 1");
  const long long nel = (long long)nelx * nely * nz;
  const unsigned nb = blocks_for(nel, 256);
  hipStream_t s = (hipStream_t)stream;
  if (filter_32bit_ok(nel) && filter_box_ok(true, nelx, nely, nz, kx, ky, kz, nullptr)) {
    launch_filter_box(true, nelx, nely, nz, kx, kz, w, map, nullptr, cval, x, y, nullptr, s);
    return check_launch("filter_box_kernel");
  }
  if (kx == 3 && ky == 3 && kz == 3)
    filter_fwd_fixed_kernel<3, 3><<<nb, 256, 0, s>>>(nelx, nely, nz, w, map, cval, x, y);
  else if (kx == 3 && ky == 3 && kz == 1)
    filter_fwd_fixed_kernel<3, 1><<<nb, 256, 0, s>>>(nelx, nely, nz, w, map, cval, x, y);
  else if (kx == 5 && ky == 5 && kz == 5)
    filter_fwd_fixed_kernel<5, 5><<<nb, 256, 0, s>>>(nelx, nely, nz, w, map, cval, x, y);
  else if (kx == 5 && ky == 5 && kz == 1)
    filter_fwd_fixed_kernel<5, 1><<<nb, 256, 0, s>>>(nelx, nely, nz, w, map, cval, x, y);
  else
    filter_fwd_kernel<<<nb, 256, 0, s>>>(nelx, nely, nz, kx, ky, kz, w, map, cval, x, y);
  return check_launch("filter_fwd_kernel");
}

int pmt_density_filter(int nelx, int nely, int nelz, double radius, const double* x, const double* scale_in,
                       const double* scale_out, double* y, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || !(radius > 0.0) || radius > 15.0 || !x || !y)
    return arg_error("pmt_density_filter: bad argument (0 < radius <= 15)");
  const int nz = nelz > 0 ? nelz : 1;
  const long long nel = (long long)nelx * nely * nz;
  density_filter_kernel<<<blocks_for(nel, 256), 256, 0, (hipStream_t)stream>>>(nelx, nely, nz, radius, (int)radius,
                                                                              nelz > 0 ? (int)radius : 0, x,
                                                                              scale_in, scale_out, y);
  return check_launch("density_filter_kernel");
}

int pmt_filter_bwd(int nelx, int nely, int nelz, int kx, int ky, int kz, const double* w, const int32_t* inv_ptr,
                   const int32_t* inv_idx, const double* dy, double* dx, void* stream) {
  return pmt_filter_bwd_work(nelx, nely, nelz, kx, ky, kz, w, inv_ptr, inv_idx, dy, dx, nullptr, stream);
}

long long pmt_filter_work_size(int nelx, int nely, int nelz, int kx, int ky, int kz) {
  if (!grid_ok(nelx, nely, nelz) || kx < 1 || ky < 1 || kz < 1) return arg_error("pmt_filter_work_size: bad argument");
  return ((long long)nelx + kx - 1) * ((long long)nely + ky - 1) * ((long long)(nelz > 0 ? nelz : 1) + kz - 1);
}

int pmt_filter_bwd_work(int nelx, int nely, int nelz, int kx, int ky, int kz, const double* w, const int32_t* inv_ptr,
                        const int32_t* inv_idx, const double* dy, double* dx, double* work, void* stream) {
  if (!grid_ok(nelx, nely, nelz) || kx < 1 || ky < 1 || kz < 1 || !(kx & 1) || !(ky & 1) || !(kz & 1) || !w ||
      !inv_ptr || !inv_idx || !dy || !dx)
    return arg_error("pmt_filter_bwd: bad argument");
  const int nz = nelz > 0 ? nelz : 1;
  if (nelz == 0 && kz != 1) return arg_error("pmt_filter_bwd: 2D grid needs kz == 1");
  const long long nel = (long long)nelx * nely * nz;
  const unsigned nb = blocks_for(nel, 256);
  hipStream_t s = (hipStream_t)stream;
  if (filter_32bit_ok(nel) && filter_box_ok(false, nelx, nely, nz, kx, ky, kz, work)) {
    launch_filter_box(false, nelx, nely, nz, kx, kz, w, inv_ptr, inv_idx, nullptr, dy, dx, work, s);
    return check_launch("filter_box_kernel");
  }
  if (kx == 3 && ky == 3 && kz == 3)
    filter_bwd_fixed_kernel<3, 3><<<nb, 256, 0, s>>>(nelx, nely, nz, w, inv_ptr, inv_idx, dy, dx);
  else if (kx == 3 && ky == 3 && kz == 1)
    filter_bwd_fixed_kernel<3, 1><<<nb, 256, 0, s>>>(nelx, nely, nz, w, inv_ptr, inv_idx, dy, dx);
  else if (kx == 5 && ky == 5 && kz == 5)
    filter_bwd_fixed_kernel<5, 5><<<nb, 256, 0, s>>>(nelx, nely, nz, w, inv_ptr, inv_idx, dy, dx);
  else if (kx == 5 && ky == 5 && kz == 1)
    filter_bwd_fixed_kernel<5, 1><<<nb, 256, 0, s>>>(nelx, nely, nz, w, inv_ptr, inv_idx, dy, dx);
  else
    filter_bwd_kernel<<<nb, 256, 0, s>>>(nelx, nely, nz, kx, ky, kz, w, inv_ptr, inv_idx, dy, dx);
  return check_launch("filter_bwd_kernel");
}

}  // extern "C"
