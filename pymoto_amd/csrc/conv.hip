// Kernels of the learned warm start: a 3D convolutional encoder-decoder on the element grid with
// BF16 activations and weights and FP32 accumulation (forward, backward to the input, backward to
// the weights), plus the pooling, upsampling, masking and optimiser kernels around them.
//
// Layout: activations channels-last, X[voxel][c] with voxel = (z*ny + y)*nx + x (the element order
// of pymoto/common/domain.py:200-251) and c contiguous, BF16; weights W[tap][cout][cin] BF16 with
// tap = (dz+1)*9 + (dy+1)*3 + (dx+1); zero padding outside the grid.
//
// Convolution as an implicit GEMM on the matrix cores (v_mfma_f32_16x16x32_bf16): the reduction runs over
// k = tap*cin + ci in chunks of 32, from a box of voxels staged in LDS.  The backward pass to the input is
// the same kernel on the flipped, transposed weights.  The weight gradient is a per-tap GEMM over voxels
// (M = cout, N = cin, K = voxels) from channel-major boxes in LDS, accumulated per block and reduced over
// blocks in a fixed order (deterministic).
#include <algorithm>

#include "launch.h"

namespace pmt {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

__device__ inline unsigned short f2bf(float f) {  // round to nearest even (finite inputs)
  const unsigned u = __float_as_uint(f);
  return (unsigned short)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
__device__ inline float bf2f(unsigned short h) { return __uint_as_float(((unsigned)h) << 16); }

struct Vox {
  int nx, ny, nz;
  long long n;
};

// n / d by multiplication (m = mdiv_magic(d), 0 for d = 1): exact while n * d < 2^32
__device__ inline unsigned mdiv(unsigned n, unsigned m) { return m ? __umulhi(n, m) : n; }

// A block's box of 2^(lx+ly+lz) output voxels and the voxels around it that it stages in LDS.
struct ConvTile {
  int lx, ly, lz;     // log2 extents
  int ntx, nty;       // boxes per grid row / column
  long long ntiles;
  unsigned m_row, m_plane;  // mdiv of the staged row length and rows per plane
};

// Y[v][co] = act(bias[co] + sum_{tap, ci} W[tap][co][ci] * X[v + off(tap)][ci])
//
// The 27 taps read every voxel's channels 27 times: from LDS, where a block keeps the box of 16 MT WM
// output voxels it computes plus one voxel around it (zeros outside the grid; with 32 or 64 channels a
// voxel is padded by 16 bytes so the 16 voxels of a wave's read fall in different banks).  A wave owns 16
// output channels and MT groups of 16 voxels, and keeps all its weights (27 CIN x 16) in registers while
// the block walks its boxes.  The weights are the A operand, so a lane ends with 4 consecutive channels of
// one voxel and stores 8 bytes.  The k order (tap, channel in chunks of 32) is that of the sums' definition
// above for every box shape, so the result does not depend on the box.
// 20 us for 16 -> 16 channels at 128x64x64 (40 us when the taps were read from global memory, one wave per
// 16 voxels and all channels, weights re-read from L2), bound by the staging's latency; 14 us for 64 -> 64 at
// 32x16x16 (33 us before), bound by the 221 KB of weights that each of its 256 blocks reads from L2.
template <int CIN, int COUT, int MT, bool RELU>
__global__ void __launch_bounds__(256, CIN >= 64 ? 1 : 2)
conv3d_fwd_kernel(Vox g, ConvTile tl, const unsigned short* __restrict__ X, const unsigned short* __restrict__ W,
                  const float* __restrict__ bias, unsigned short* __restrict__ Y) {
  constexpr int KCH = (27 * CIN + 31) / 32;
  constexpr int WN = COUT / 16;                        // waves over the output channels
  constexpr int VS = CIN * 2 + (CIN >= 32 ? 16 : 0);  // bytes of a staged voxel
  constexpr int CPV = CIN / 8;                         // 16-byte parts of a voxel
  extern __shared__ __attribute__((aligned(16))) char xs[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kq = lane >> 4;
  const int wn = wave % WN, wm = wave / WN;
  const int rowv = (1 << tl.lx) + 2, rows = (1 << tl.ly) + 2, planes = (1 << tl.lz) + 2;
  const int row_b = rowv * VS, plane_b = rows * row_b;
  bf16x8 w[KCH];
#pragma unroll
  for (int q = 0; q < KCH; ++q) {
    const int k0 = 32 * q + 8 * kq;
    u4v r = {0u, 0u, 0u, 0u};
    if (k0 < 27 * CIN) r = *(const u4v*)(W + ((long long)(k0 / CIN) * COUT + 16 * wn + (lane & 15)) * CIN + k0 % CIN);
    w[q] = __builtin_bit_cast(bf16x8, r);
  }
  float bv[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) bv[r] = bias ? bias[16 * wn + 4 * kq + r] : 0.0f;
  int vx[MT], vy[MT], vz[MT], base[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = (wm * MT + mt) * 16 + (lane & 15);
    vx[mt] = m & ((1 << tl.lx) - 1);
    vy[mt] = (m >> tl.lx) & ((1 << tl.ly) - 1);
    vz[mt] = m >> (tl.lx + tl.ly);
    base[mt] = vz[mt] * plane_b + vy[mt] * row_b + vx[mt] * VS;
  }
  const int parts = planes * rows * rowv * CPV;
  for (long long t = blockIdx.x; t < tl.ntiles; t += gridDim.x) {
    const int tx = (int)(t % tl.ntx), ty = (int)((t / tl.ntx) % tl.nty), tz = (int)(t / ((long long)tl.ntx * tl.nty));
    const int x0 = tx << tl.lx, y0 = ty << tl.ly, z0 = tz << tl.lz;
    __syncthreads();
    for (int i = threadIdx.x; i < parts; i += 256) {
      const unsigned hv = i / CPV, part = i % CPV;
      const unsigned row = mdiv(hv, tl.m_row), hz = mdiv(row, tl.m_plane);
      const int xx = x0 + (int)(hv - row * rowv) - 1, yy = y0 + (int)(row - hz * rows) - 1, zz = z0 + (int)hz - 1;
      u4v v = {0u, 0u, 0u, 0u};
      if (xx >= 0 && xx < g.nx && yy >= 0 && yy < g.ny && zz >= 0 && zz < g.nz)
        v = *(const u4v*)(X + (((long long)zz * g.ny + yy) * g.nx + xx) * CIN + part * 8);
      *(u4v*)(xs + hv * VS + part * 16) = v;
    }
    __syncthreads();
    f4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < KCH; ++q) {
      // the lane's tap: the same for the whole wave with >= 32 channels, else one of the chunk's 2 or 4
      int off = 0;
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int k0 = 32 * q + 8 * h, tap = k0 / CIN;
        if (h > 0 && tap == (32 * q + 8 * (h - 1)) / CIN) continue;
        const int o = tap < 27 ? (tap / 9) * plane_b + ((tap / 3) % 3) * row_b + (tap % 3) * VS : 0;
        off = kq >= h ? o : off;
      }
      off += ((32 * q + 8 * kq) % CIN) * 2;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        u4v r = *(const u4v*)(xs + base[mt] + off);
        if (32 * (q + 1) > 27 * CIN && 32 * q + 8 * kq >= 27 * CIN) r = u4v{0u, 0u, 0u, 0u};  // past the last tap
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[q], __builtin_bit_cast(bf16x8, r), acc[mt], 0, 0, 0);
      }
    }
    // D[row = 4*(lane/16) + r][col = lane%16]: channel 16*wn + row, voxel col
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int x = x0 + vx[mt], y = y0 + vy[mt], z = z0 + vz[mt];
      if (x >= g.nx || y >= g.ny || z >= g.nz) continue;
      unsigned short o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[mt][r] + bv[r];
        if (RELU) v = v > 0.0f ? v : 0.0f;
        o[r] = f2bf(v);
      }
      const uint2 pk = {o[0] | ((unsigned)o[1] << 16), o[2] | ((unsigned)o[3] << 16)};
      *(uint2*)(Y + (((long long)z * g.ny + y) * g.nx + x) * COUT + 16 * wn + 4 * kq) = pk;
    }
  }
}

// Wt[tap][ci][co] = W[26 - tap][co][ci]: the backward pass to the input is a forward convolution of
// the output gradient with these weights
__global__ void conv3d_flip_kernel(int cin, int cout, const unsigned short* __restrict__ W,
                                   unsigned short* __restrict__ Wt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = 27 * cin * cout;
  if (i >= n) return;
  const int tap = i / (cin * cout), rem = i % (cin * cout), ci = rem / cout, co = rem % cout;
  Wt[i] = W[((26 - tap) * cout + co) * cin + ci];
}

// The box of 8 XG x TY x TZ voxels that a weight-gradient block stages at a time.
struct WgradTile {
  int xg, ty, tz;
  int ntx, nty;
  long long ntiles;
  int cs, csg;              // 2-byte entries per staged channel of X and of G
  unsigned m_xrow, m_xrows;  // mdiv of (4 xg + 2) pairs per staged X row, of its rows per plane
  unsigned m_grow, m_grows;  // the same of 4 xg, ty for G
  unsigned m_xg, m_ty;       // of xg, ty (groups of 8 voxels)
};

// How the 4 waves of a weight-gradient block share dW: over the 16-channel tiles of ci, then of co, then
// (small layers) over the voxels.  A block of a layer with more than 4 tiles takes the 9 taps of one z offset.
template <int CIN, int COUT>
struct WgradCfg {
  static constexpr int NI = COUT / 16, NJ = (CIN + 15) / 16;
  static constexpr int CW = NJ;                                // waves over ci
  static constexpr int OW = NI < 4 / CW ? NI : 4 / CW;         // waves over co
  static constexpr int KS = 4 / (CW * OW);                     // waves over the voxels
  static constexpr int TW = NI / OW;                           // co tiles per wave
  static constexpr int NDZ = NI * NJ <= 4 ? 3 : 1;             // z offsets per block
  static constexpr int ROW = 27 * CIN * COUT + COUT;           // a block's partial sums: dW, then dbias
};

// Partial dW[tap][co][ci] of one block = sum over its voxels of G[v][co] * X[v + off(tap)][ci], and the
// partial sum of G (the bias gradient).  grid (blocks, 3 / NDZ).
//
// The contraction runs over voxels, so both operands need 8 consecutive voxels of one channel: the block
// transposes its box to channel-major rows in LDS once (pairs of voxels, 4-byte writes) and all taps read
// it from there; the three x offsets of a row share one 16-byte read and the two words beside it, shifted
// by one voxel in registers.  RAGGED (the box does not divide the grid): a voxel outside the grid has
// G = 0, and its X operand is masked to 0 as well, so a non-finite X next to the edge stays out of the
// offsets that do not use it.
// 27 us for 16 -> 16 channels at 128x64x64, 18 us for 64 -> 64 at 32x16x16, the bias sum included.  Loading
// both operands voxel by voxel from global memory (2 bytes a load, once per tap) took 514 and 38 us, one
// block per channel for the bias sum another 541 and 13 us.
template <int CIN, int COUT, bool RAGGED>
__global__ void __launch_bounds__(256, 2)
conv3d_wgrad_kernel(Vox g, WgradTile tl, const unsigned short* __restrict__ X, const unsigned short* __restrict__ G,
                    float* __restrict__ partial) {
  using C = WgradCfg<CIN, COUT>;
  constexpr int NDZ = C::NDZ, TW = C::TW, KS = C::KS, NT = 9 * NDZ;
  extern __shared__ __attribute__((aligned(16))) unsigned short ls[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kq = lane >> 4, ch = lane & 15;
  const int wj = wave % C::CW, wi = (wave / C::CW) % C::OW, ks = wave / (C::CW * C::OW);
  const int dz0 = NDZ == 3 ? -1 : (int)blockIdx.y - 1;  // first z offset of this block
  const int xr = 8 * tl.xg + 16, xrows = tl.ty + 2, xplanes = tl.tz + NDZ - 1;
  unsigned short* Xs = ls;
  unsigned short* Gs = ls + C::NJ * 16 * tl.cs;
  f4 acc[NT][TW], accb[TW];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < TW; ++b) acc[a][b] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int b = 0; b < TW; ++b) accb[b] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  const bool with_bias = wj == 0 && (NDZ == 3 || blockIdx.y == 0);
  const bf16x8 ones = __builtin_bit_cast(bf16x8, u4v{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});
  const int ngroups = tl.xg * tl.ty * tl.tz;  // a multiple of 4
  // two voxels (x, x + 1) of 8 channels into 8 channel rows
  auto put = [](unsigned short* row, int cstride, u4v a, u4v b) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      *(unsigned*)(row + (2 * c) * cstride) = __builtin_amdgcn_perm(b[c], a[c], 0x05040100u);
      *(unsigned*)(row + (2 * c + 1) * cstride) = __builtin_amdgcn_perm(b[c], a[c], 0x07060302u);
    }
  };
  auto fetch = [&](const unsigned short* base, int c, int x, int y, int z, int part) {
    u4v v = {0u, 0u, 0u, 0u};
    if (x >= 0 && x < g.nx && y >= 0 && y < g.ny && z >= 0 && z < g.nz)
      v = *(const u4v*)(base + (((long long)z * g.ny + y) * g.nx + x) * c + part * 8);
    return v;
  };
  if (CIN == 8)  // the tile's upper 8 rows do not exist
    for (int i = threadIdx.x; i < 8 * tl.cs / 2; i += 256) *(unsigned*)(Xs + 8 * tl.cs + 2 * i) = 0u;
  for (long long t = blockIdx.x; t < tl.ntiles; t += gridDim.x) {
    const int tx = (int)(t % tl.ntx), ty = (int)((t / tl.ntx) % tl.nty), tz = (int)(t / ((long long)tl.ntx * tl.nty));
    const int x0 = tx * 8 * tl.xg, y0 = ty * tl.ty, z0 = tz * tl.tz;
    __syncthreads();
    const int pairs = 4 * tl.xg + 2;  // staged x: -2 .. 8 xg + 1
    for (int i = threadIdx.x; i < xplanes * xrows * pairs * (CIN / 8); i += 256) {
      const unsigned part = i % (CIN / 8), q = i / (CIN / 8);
      const unsigned row = mdiv(q, tl.m_xrow), pl = mdiv(row, tl.m_xrows);
      const int px = 2 * (int)(q - row * pairs) - 2;
      const int x = x0 + px, y = y0 + (int)(row - pl * xrows) - 1, z = z0 + (int)pl + dz0;
      put(Xs + part * 8 * tl.cs + row * xr + 8 + px, tl.cs, fetch(X, CIN, x, y, z, part), fetch(X, CIN, x + 1, y, z, part));
    }
    for (int i = threadIdx.x; i < tl.tz * tl.ty * 4 * tl.xg * (COUT / 8); i += 256) {
      const unsigned part = i % (COUT / 8), q = i / (COUT / 8);
      const unsigned row = mdiv(q, tl.m_grow), pl = mdiv(row, tl.m_grows);
      const int px = 2 * (int)(q - row * 4 * tl.xg);
      const int x = x0 + px, y = y0 + (int)(row - pl * tl.ty), z = z0 + (int)pl;
      put(Gs + part * 8 * tl.csg + row * 8 * tl.xg + px, tl.csg, fetch(G, COUT, x, y, z, part),
          fetch(G, COUT, x + 1, y, z, part));
    }
    __syncthreads();
    for (int c = ks; c < ngroups / 4; c += KS) {
      const unsigned grp = 4 * c + kq;  // this lane's 8 voxels
      const unsigned row = mdiv(grp, tl.m_xg), pl = mdiv(row, tl.m_ty);
      const int gx = (int)(grp - row * tl.xg), gy = (int)(row - pl * tl.ty);
      u4v mask = {~0u, ~0u, ~0u, ~0u};
      if (RAGGED) {
        const int left = (y0 + gy < g.ny && z0 + (int)pl < g.nz) ? g.nx - (x0 + 8 * gx) : 0;  // voxels inside
#pragma unroll
        for (int k = 0; k < 4; ++k) mask[k] = (left > 2 * k ? 0xffffu : 0u) | (left > 2 * k + 1 ? 0xffff0000u : 0u);
      }
      bf16x8 A[TW];
#pragma unroll
      for (int b = 0; b < TW; ++b) {
        A[b] = *(const bf16x8*)(Gs + (16 * (wi * TW + b) + ch) * tl.csg + row * 8 * tl.xg + 8 * gx);
        if (with_bias) accb[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[b], ones, accb[b], 0, 0, 0);
      }
      const unsigned short* xp = Xs + (16 * wj + ch) * tl.cs + (pl * xrows + gy) * xr + 8 + 8 * gx;
#pragma unroll
      for (int dz = 0; dz < NDZ; ++dz)
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
          const unsigned short* xq = xp + (dz * xrows + dy) * xr;
          const u4v m = *(const u4v*)xq;
          const unsigned lo = *(const unsigned*)(xq - 2), hi = *(const unsigned*)(xq + 8);
          const unsigned s0 = __builtin_amdgcn_alignbyte(m[0], lo, 2), s1 = __builtin_amdgcn_alignbyte(m[1], m[0], 2),
                         s2 = __builtin_amdgcn_alignbyte(m[2], m[1], 2), s3 = __builtin_amdgcn_alignbyte(m[3], m[2], 2),
                         s4 = __builtin_amdgcn_alignbyte(hi, m[3], 2);
          const u4v sh[3] = {u4v{s0, s1, s2, s3}, m, u4v{s1, s2, s3, s4}};
#pragma unroll
          for (int dx = 0; dx < 3; ++dx) {
            const bf16x8 B = __builtin_bit_cast(bf16x8, RAGGED ? sh[dx] & mask : sh[dx]);
            const int tap = (dz * 3 + dy) * 3 + dx;
#pragma unroll
            for (int b = 0; b < TW; ++b)
              acc[tap][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[b], B, acc[tap][b], 0, 0, 0);
          }
        }
    }
  }
  // waves that share a tile: sum them through LDS in a fixed order, one wave after the other
  if (KS > 1) {
    float* red = (float*)ls + (wave % (C::CW * C::OW)) * (NT + 1) * 256;
    for (int k = 1; k < KS; ++k) {
      __syncthreads();
      if (ks == k) {
#pragma unroll
        for (int a = 0; a <= NT; ++a) *(f4*)(red + a * 256 + lane * 4) = a < NT ? acc[a < NT ? a : 0][0] : accb[0];
      }
      __syncthreads();
      if (ks == 0) {
#pragma unroll
        for (int a = 0; a < NT; ++a) acc[a][0] += *(const f4*)(red + a * 256 + lane * 4);
        accb[0] += *(const f4*)(red + NT * 256 + lane * 4);
      }
    }
    if (ks) return;
  }
  // D[row = 4*(lane/16) + r][col = lane%16] -> co = 16 * tile + row, ci = 16 wj + col
  float* out = partial + (long long)blockIdx.x * C::ROW;
#pragma unroll
  for (int b = 0; b < TW; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int co = 16 * (wi * TW + b) + 4 * kq + r, ci = 16 * wj + ch;
#pragma unroll
      for (int a = 0; a < NT; ++a)
        if (CIN >= 16 || ch < CIN) out[((long long)((dz0 + 1) * 9 + a) * COUT + co) * CIN + ci] = acc[a][b][r];
      if (with_bias && ch == 0) out[27 * CIN * COUT + co] = accb[b][r];
    }
}

// dW[i] = sum_b partial[b][i] and, behind it, dbias (fixed order): a block owns 16 quadruples of entries, 16
// threads each, so the loads of one entry are 16 ways parallel (the 512 partials of the 16 x 16 layers in 4
// batches of 8 loads; one thread per entry took 16 us)
__global__ void __launch_bounds__(256) conv3d_wgrad_reduce(int nblocks, int row, int m, const float* __restrict__ partial,
                                                           float* __restrict__ dW, float* __restrict__ dbias) {
  const int col = threadIdx.x & 15, slice = threadIdx.x >> 4;
  const int i = 4 * (blockIdx.x * 16 + col);
  f4 s = {0.0f, 0.0f, 0.0f, 0.0f};
  if (i < row) {
#pragma unroll 8
    for (int b = slice; b < nblocks; b += 16) s += *(const f4*)(partial + (long long)b * row + i);
  }
  __shared__ f4 red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 8; w > 0; w >>= 1) {
    if (slice < w) red[threadIdx.x] += red[threadIdx.x + 16 * w];
    __syncthreads();
  }
  if (slice || i >= row) return;
  for (int k = 0; k < 4; ++k) {
    if (i < m)
      dW[i + k] = red[col][k];
    else if (dbias)
      dbias[i - m + k] = red[col][k];
  }
}

// G *= (Y > 0)  (ReLU backward from the layer output)
__global__ void relu_mask_kernel(long long n, const unsigned short* __restrict__ Y, unsigned short* __restrict__ G) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && !(bf2f(Y[i]) > 0.0f)) G[i] = 0;
}

// 2x2x2 average pooling (fine grid nx, ny, nz even) and its adjoint
__global__ void pool2_kernel(Vox f, int c, const unsigned short* __restrict__ X, unsigned short* __restrict__ Y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int cx = f.nx / 2, cy = f.ny / 2, cz = f.nz / 2;
  const long long n = (long long)cx * cy * cz * c;
  if (i >= n) return;
  const int ch = (int)(i % c);
  const long long v = i / c;
  const int x = (int)(v % cx), y = (int)((v / cx) % cy), z = (int)(v / ((long long)cx * cy));
  float s = 0.0f;
  for (int d = 0; d < 8; ++d) {
    const long long m = ((long long)(2 * z + (d >> 2)) * f.ny + (2 * y + ((d >> 1) & 1))) * f.nx + 2 * x + (d & 1);
    s += bf2f(X[m * c + ch]);
  }
  Y[i] = f2bf(0.125f * s);
}

__global__ void pool2_bwd_kernel(Vox f, int c, const unsigned short* __restrict__ dY, unsigned short* __restrict__ dX) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= f.n * c) return;
  const int ch = (int)(i % c);
  const long long v = i / c;
  const int x = (int)(v % f.nx), y = (int)((v / f.nx) % f.ny), z = (int)(v / ((long long)f.nx * f.ny));
  const long long p = ((long long)(z / 2) * (f.ny / 2) + y / 2) * (f.nx / 2) + x / 2;
  dX[i] = f2bf(0.125f * bf2f(dY[p * c + ch]));
}

// Y[fine] = X[parent] + S[fine] (nearest upsampling plus skip connection); the adjoint to X sums the
// 8 children (the adjoint to S is the identity)
__global__ void up2_add_kernel(Vox f, int c, const unsigned short* __restrict__ X, const unsigned short* __restrict__ S,
                               unsigned short* __restrict__ Y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= f.n * c) return;
  const int ch = (int)(i % c);
  const long long v = i / c;
  const int x = (int)(v % f.nx), y = (int)((v / f.nx) % f.ny), z = (int)(v / ((long long)f.nx * f.ny));
  const long long p = ((long long)(z / 2) * (f.ny / 2) + y / 2) * (f.nx / 2) + x / 2;
  Y[i] = f2bf(bf2f(X[p * c + ch]) + bf2f(S[i]));
}

__global__ void up2_bwd_kernel(Vox f, int c, const unsigned short* __restrict__ dY, unsigned short* __restrict__ dX) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int cx = f.nx / 2, cy = f.ny / 2, cz = f.nz / 2;
  if (i >= (long long)cx * cy * cz * c) return;
  const int ch = (int)(i % c);
  const long long v = i / c;
  const int x = (int)(v % cx), y = (int)((v / cx) % cy), z = (int)(v / ((long long)cx * cy));
  float s = 0.0f;
  for (int d = 0; d < 8; ++d) {
    const long long m = ((long long)(2 * z + (d >> 2)) * f.ny + (2 * y + ((d >> 1) & 1))) * f.nx + 2 * x + (d & 1);
    s += bf2f(dY[m * c + ch]);
  }
  dX[i] = f2bf(s);
}

// Nodal displacement from the first 3 channels of the element output: the mean over the elements
// around each node; and its adjoint (hex8, dof = node*3 + d)
__global__ void elem_to_node_kernel(Vox e, int c, const unsigned short* __restrict__ Xe, float* __restrict__ u) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nx = e.nx + 1, ny = e.ny + 1, nz = e.nz + 1;
  if (q >= (long long)nx * ny * nz * 3) return;
  const int d = (int)(q % 3);
  const long long n = q / 3;
  const int i = (int)(n % nx), j = (int)((n / nx) % ny), k = (int)(n / ((long long)nx * ny));
  float s = 0.0f;
  int cnt = 0;
  for (int a = 0; a < 8; ++a) {
    const int ei = i - (a & 1), ej = j - ((a >> 1) & 1), ek = k - ((a >> 2) & 1);
    if (ei < 0 || ei >= e.nx || ej < 0 || ej >= e.ny || ek < 0 || ek >= e.nz) continue;
    s += bf2f(Xe[(((long long)ek * e.ny + ej) * e.nx + ei) * c + d]);
    ++cnt;
  }
  u[q] = s / (float)cnt;
}

__global__ void elem_to_node_bwd_kernel(Vox e, int c, const float* __restrict__ du, unsigned short* __restrict__ dXe) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= e.n * c) return;
  const int ch = (int)(q % c);
  const long long v = q / c;
  if (ch >= 3) {
    dXe[q] = 0;
    return;
  }
  const int nx = e.nx + 1, ny = e.ny + 1, nz = e.nz + 1;
  const int ei = (int)(v % e.nx), ej = (int)((v / e.nx) % e.ny), ek = (int)(v / ((long long)e.nx * e.ny));
  float s = 0.0f;
  for (int a = 0; a < 8; ++a) {
    const int i = ei + (a & 1), j = ej + ((a >> 1) & 1), k = ek + ((a >> 2) & 1);
    const int cnt = (i > 0 && i < nx - 1 ? 2 : 1) * (j > 0 && j < ny - 1 ? 2 : 1) * (k > 0 && k < nz - 1 ? 2 : 1);
    s += du[(((long long)k * ny + j) * nx + i) * 3 + ch] / (float)cnt;
  }
  dXe[q] = f2bf(s);
}

// Adam step on FP32 master weights, with the BF16 copy refreshed (t is the 1-based step)
__global__ void adam_kernel(long long n, float lr, float b1, float b2, float eps, int t, const float* __restrict__ grad,
                            float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                            unsigned short* __restrict__ wb) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gr = grad[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gr;
  const float vi = b2 * v[i] + (1.0f - b2) * gr * gr;
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / (1.0f - powf(b1, (float)t)), vh = vi / (1.0f - powf(b2, (float)t));
  const float wi = w[i] - lr * mh / (sqrtf(vh) + eps);
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
}

__global__ void add_bf16_kernel(long long n, const unsigned short* __restrict__ a, const unsigned short* __restrict__ b,
                                unsigned short* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(bf2f(a[i]) + bf2f(b[i]));
}

__global__ void f32_to_bf16_kernel(long long n, const float* __restrict__ x, unsigned short* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

__global__ void bf16_to_f32_kernel(long long n, const unsigned short* __restrict__ x, float* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = bf2f(x[i]);
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
static Vox vox(int nx, int ny, int nz) {
  Vox g;
  g.nx = nx;
  g.ny = ny;
  g.nz = nz;
  g.n = (long long)nx * ny * nz;
  return g;
}

static bool conv_shape_ok(int nx, int ny, int nz, int cin, int cout) {
  const bool c_ok = (cin == 8 || cin == 16 || cin == 32 || cin == 64) && (cout == 16 || cout == 32 || cout == 64);
  return c_ok && nx > 0 && ny > 0 && nz > 0 && ((long long)nx * ny * nz) % 16 == 0;
}

#define PMT_CONV_CASES(F) \
  F(8, 16) F(16, 16) F(16, 32) F(16, 64) F(32, 16) F(32, 32) F(32, 64) F(64, 16) F(64, 32) F(64, 64)

static unsigned mdiv_magic(unsigned d) { return d == 1 ? 0u : (unsigned)(0x100000000ull / d + 1); }

// The box shape for 16 * MT * WM output voxels: the fewest staged and computed voxels over the whole grid
// (a staged voxel costs about half a computed one: one read and one LDS write against 27 LDS reads and
// matrix operations shared by the channels).
static ConvTile conv_tile(const Vox& g, int log2v, int voxel_bytes, size_t* lds) {
  ConvTile best{};
  double cost = -1.0;
  for (int lx = 0; lx <= 5; ++lx)
    for (int ly = 0; ly + lx <= log2v; ++ly) {
      const int lz = log2v - lx - ly;
      if (lz > 5) continue;
      const long long nt = (long long)((g.nx + (1 << lx) - 1) >> lx) * ((g.ny + (1 << ly) - 1) >> ly) *
                           ((g.nz + (1 << lz) - 1) >> lz);
      const int hv = ((1 << lx) + 2) * ((1 << ly) + 2) * ((1 << lz) + 2);
      if (hv * voxel_bytes > 65536) continue;
      const double c = (double)nt * ((1 << log2v) + 0.5 * hv);
      if (cost < 0.0 || c < cost) {
        cost = c;
        best.lx = lx;
        best.ly = ly;
        best.lz = lz;
        best.ntx = (g.nx + (1 << lx) - 1) >> lx;
        best.nty = (g.ny + (1 << ly) - 1) >> ly;
        best.ntiles = nt;
        best.m_row = mdiv_magic((1 << lx) + 2);
        best.m_plane = mdiv_magic((1 << ly) + 2);
        *lds = (size_t)hv * voxel_bytes;
      }
    }
  return best;
}

template <int CI, int CO, int MT>
static int conv_fwd_mt(const Vox& g, const unsigned short* X, const unsigned short* W, const float* bias, int relu,
                       unsigned short* Y, hipStream_t s) {
  constexpr int voxels = 16 * MT * 4 / (CO / 16), log2v = __builtin_ctz(voxels);
  size_t lds = 0;
  const ConvTile tl = conv_tile(g, log2v, CI * 2 + (CI >= 32 ? 16 : 0), &lds);
  // one wave of resident blocks: 64 input channels hold 216 weight registers per lane (1 block per CU)
  const long long cap = (long long)device_cu_count() * (CI >= 64 ? 1 : CI >= 32 ? 2 : 4);
  const unsigned grid = (unsigned)std::min(tl.ntiles, cap);
  if (relu)
    conv3d_fwd_kernel<CI, CO, MT, true><<<grid, 256, lds, s>>>(g, tl, X, W, bias, Y);
  else
    conv3d_fwd_kernel<CI, CO, MT, false><<<grid, 256, lds, s>>>(g, tl, X, W, bias, Y);
  return check_launch("conv3d_fwd_kernel");
}

// 2 groups of 16 voxels per wave while the boxes are too few to give every CU two, else 4 (a larger box
// stages fewer voxels per output); 64 -> 16 channels always 2 (its box of 4 exceeds 64 KB of LDS)
static int conv_fwd(const Vox& g, int cin, int cout, const unsigned short* X, const unsigned short* W,
                    const float* bias, int relu, unsigned short* Y, hipStream_t s) {
  const bool small = g.n / (16 * 4 * 4 / (cout / 16)) < 2LL * device_cu_count();
#define F(CI, CO)                                                                          \
  if (cin == CI && cout == CO)                                                             \
    return small ? conv_fwd_mt<CI, CO, 2>(g, X, W, bias, relu, Y, s)                       \
                 : conv_fwd_mt<CI, CO, (CI == 64 && CO == 16) ? 2 : 4>(g, X, W, bias, relu, Y, s);
  PMT_CONV_CASES(F)
#undef F
  return arg_error("conv3d: unsupported channel counts");
}

// Blocks of a weight gradient: enough to fill the chip, few enough that writing and summing their partial
// sums (27 cin cout floats each) stays cheap: about 14 MB in all.
static int wgrad_blocks(int cin, int cout) { return std::min(512, std::max(64, 512 * 256 / (cin * cout))); }

template <int CI, int CO>
static int conv_wgrad(const Vox& g, const unsigned short* X, const unsigned short* G, float* dW, float* dbias,
                      float* work, hipStream_t s) {
  using C = WgradCfg<CI, CO>;
  WgradTile best{};
  size_t lds = 0;
  double cost = -1.0;
  auto odd8 = [](int v) { return ((v + 7) / 8 | 1) * 8; };  // 8 x odd entries: channel rows fall in different banks
  for (int xg = 1; xg <= 4; xg *= 2)
    for (int ty = 1; ty <= 8; ty *= 2)
      for (int tz = 1; tz <= 4; tz *= 2) {
        if (xg * ty * tz % 4) continue;
        const int xrows = (ty + 2) * (tz + C::NDZ - 1);
        const int cs = odd8(xrows * (8 * xg + 16)), csg = odd8(ty * tz * 8 * xg);
        size_t b = 2ull * (C::NJ * 16 * cs + CO * csg);
        if (C::KS > 1) b = std::max(b, (size_t)C::CW * C::OW * (9 * C::NDZ + 1) * 1024);
        if (b > 65536) continue;
        const int ntx = (g.nx + 8 * xg - 1) / (8 * xg), nty = (g.ny + ty - 1) / ty, ntz = (g.nz + tz - 1) / tz;
        const long long nt = (long long)ntx * nty * ntz;
        // staged 8-channel pairs of voxels, and the groups of 8 voxels (27 taps each, shared by the waves)
        const double c = (double)nt * (xrows * (4 * xg + 2) * (CI / 8) + ty * tz * 4 * xg * (CO / 8) +
                                       12.0 * xg * ty * tz * C::TW / C::KS + 128.0);
        if (cost < 0.0 || c < cost) {
          cost = c;
          lds = b;
          best = WgradTile{xg, ty, tz, ntx, nty, nt, cs, csg, mdiv_magic(4 * xg + 2), mdiv_magic(ty + 2),
                           mdiv_magic(4 * xg), mdiv_magic(ty), mdiv_magic(xg), mdiv_magic(ty)};
        }
      }
  const int nb = (int)std::min<long long>(best.ntiles, wgrad_blocks(CI, CO));
  const dim3 grid(nb, 3 / C::NDZ);
  if (g.nx % (8 * best.xg) || g.ny % best.ty || g.nz % best.tz)
    conv3d_wgrad_kernel<CI, CO, true><<<grid, 256, lds, s>>>(g, best, X, G, work);
  else
    conv3d_wgrad_kernel<CI, CO, false><<<grid, 256, lds, s>>>(g, best, X, G, work);
  PMT_TRY(check_launch("conv3d_wgrad_kernel"));
  conv3d_wgrad_reduce<<<blocks_for(C::ROW / 4, 16), 256, 0, s>>>(nb, C::ROW, 27 * CI * CO, work, dW, dbias);
  return check_launch("conv3d_wgrad_reduce");
}

}  // namespace pmt

using namespace pmt;

extern "C" {

int pmt_conv3d_fwd(int nx, int ny, int nz, int cin, int cout, const void* X, const void* W, const float* bias,
                   int relu, void* Y, void* stream) {
  if (!conv_shape_ok(nx, ny, nz, cin, cout) || !X || !W || !Y)
    return arg_error("pmt_conv3d_fwd: bad argument (cin in 8/16/32/64, cout in 16/32/64, voxels % 16 == 0)");
  return conv_fwd(vox(nx, ny, nz), cin, cout, (const unsigned short*)X, (const unsigned short*)W, bias, relu,
                  (unsigned short*)Y, (hipStream_t)stream);
}

int pmt_conv3d_bwd_data(int nx, int ny, int nz, int cin, int cout, const void* dY, const void* W, void* Wt, void* dX,
                        void* stream) {
  if (!conv_shape_ok(nx, ny, nz, cout, cin) || cin < 16 || !dY || !W || !Wt || !dX)
    return arg_error("pmt_conv3d_bwd_data: bad argument (cin in 16/32/64, cout in 16/32/64, voxels % 16 == 0)");
  hipStream_t s = (hipStream_t)stream;
  const int n = 27 * cin * cout;
  conv3d_flip_kernel<<<blocks_for(n, 256), 256, 0, s>>>(cin, cout, (const unsigned short*)W, (unsigned short*)Wt);
  PMT_TRY(check_launch("conv3d_flip_kernel"));
  return conv_fwd(vox(nx, ny, nz), cout, cin, (const unsigned short*)dY, (const unsigned short*)Wt, nullptr, 0,
                  (unsigned short*)dX, s);
}

int pmt_conv3d_wgrad_work_size(int cin, int cout) { return wgrad_blocks(cin, cout) * (27 * cin * cout + cout); }

int pmt_conv3d_bwd_weight(int nx, int ny, int nz, int cin, int cout, const void* X, const void* dY, float* dW,
                          float* dbias, float* work, void* stream) {
  if (!conv_shape_ok(nx, ny, nz, cin, cout) || !X || !dY || !dW || !work)
    return arg_error("pmt_conv3d_bwd_weight: bad argument");
  hipStream_t s = (hipStream_t)stream;
  const Vox g = vox(nx, ny, nz);
#define F(CI, CO)                \
  if (cin == CI && cout == CO) \
    return conv_wgrad<CI, CO>(g, (const unsigned short*)X, (const unsigned short*)dY, dW, dbias, work, s);
  PMT_CONV_CASES(F)
#undef F
  return arg_error("pmt_conv3d_bwd_weight: unsupported channel counts");
}

int pmt_relu_mask_bf16(long long n, const void* Y, void* G, void* stream) {
  if (n < 0 || (n > 0 && (!Y || !G))) return arg_error("pmt_relu_mask_bf16: bad argument");
  if (n == 0) return PMT_OK;
  relu_mask_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, (const unsigned short*)Y,
                                                                        (unsigned short*)G);
  return check_launch("relu_mask_kernel");
}

int pmt_pool2_bf16(int nx, int ny, int nz, int c, const void* X, void* Y, void* stream) {
  if (nx % 2 || ny % 2 || nz % 2 || c <= 0 || !X || !Y) return arg_error("pmt_pool2_bf16: bad argument");
  const long long n = (long long)(nx / 2) * (ny / 2) * (nz / 2) * c;
  pool2_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(vox(nx, ny, nz), c, (const unsigned short*)X,
                                                                    (unsigned short*)Y);
  return check_launch("pool2_kernel");
}

int pmt_pool2_bwd_bf16(int nx, int ny, int nz, int c, const void* dY, void* dX, void* stream) {
  if (nx % 2 || ny % 2 || nz % 2 || c <= 0 || !dY || !dX) return arg_error("pmt_pool2_bwd_bf16: bad argument");
  const Vox f = vox(nx, ny, nz);
  pool2_bwd_kernel<<<blocks_for(f.n * c, 256), 256, 0, (hipStream_t)stream>>>(f, c, (const unsigned short*)dY,
                                                                              (unsigned short*)dX);
  return check_launch("pool2_bwd_kernel");
}

int pmt_up2_add_bf16(int nx, int ny, int nz, int c, const void* X, const void* S, void* Y, void* stream) {
  if (nx % 2 || ny % 2 || nz % 2 || c <= 0 || !X || !S || !Y) return arg_error("pmt_up2_add_bf16: bad argument");
  const Vox f = vox(nx, ny, nz);
  up2_add_kernel<<<blocks_for(f.n * c, 256), 256, 0, (hipStream_t)stream>>>(f, c, (const unsigned short*)X,
                                                                            (const unsigned short*)S,
                                                                            (unsigned short*)Y);
  return check_launch("up2_add_kernel");
}

int pmt_up2_bwd_bf16(int nx, int ny, int nz, int c, const void* dY, void* dX, void* stream) {
  if (nx % 2 || ny % 2 || nz % 2 || c <= 0 || !dY || !dX) return arg_error("pmt_up2_bwd_bf16: bad argument");
  const long long n = (long long)(nx / 2) * (ny / 2) * (nz / 2) * c;
  up2_bwd_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(vox(nx, ny, nz), c, (const unsigned short*)dY,
                                                                      (unsigned short*)dX);
  return check_launch("up2_bwd_kernel");
}

int pmt_elem_to_node(int nelx, int nely, int nelz, int c, const void* Xe, float* u, void* stream) {
  if (nelx <= 0 || nely <= 0 || nelz <= 0 || c < 3 || !Xe || !u) return arg_error("pmt_elem_to_node: bad argument");
  const long long n = (long long)(nelx + 1) * (nely + 1) * (nelz + 1) * 3;
  elem_to_node_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(vox(nelx, nely, nelz), c,
                                                                          (const unsigned short*)Xe, u);
  return check_launch("elem_to_node_kernel");
}

int pmt_elem_to_node_bwd(int nelx, int nely, int nelz, int c, const float* du, void* dXe, void* stream) {
  if (nelx <= 0 || nely <= 0 || nelz <= 0 || c < 3 || !du || !dXe)
    return arg_error("pmt_elem_to_node_bwd: bad argument");
  const Vox e = vox(nelx, nely, nelz);
  elem_to_node_bwd_kernel<<<blocks_for(e.n * c, 256), 256, 0, (hipStream_t)stream>>>(e, c, du, (unsigned short*)dXe);
  return check_launch("elem_to_node_bwd_kernel");
}

int pmt_adam_step(long long n, float lr, float b1, float b2, float eps, int t, const float* grad, float* w, float* m,
                  float* v, void* wb, void* stream) {
  if (n < 0 || t < 1 || (n > 0 && (!grad || !w || !m || !v))) return arg_error("pmt_adam_step: bad argument");
  if (n == 0) return PMT_OK;
  adam_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, lr, b1, b2, eps, t, grad, w, m, v,
                                                                  (unsigned short*)wb);
  return check_launch("adam_kernel");
}

int pmt_add_bf16(long long n, const void* a, const void* b, void* y, void* stream) {
  if (n < 0 || (n > 0 && (!a || !b || !y))) return arg_error("pmt_add_bf16: bad argument");
  if (n == 0) return PMT_OK;
  add_bf16_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, (const unsigned short*)a,
                                                                       (const unsigned short*)b, (unsigned short*)y);
  return check_launch("add_bf16_kernel");
}

int pmt_f32_to_bf16(long long n, const float* x, void* y, void* stream) {
  if (n < 0 || (n > 0 && (!x || !y))) return arg_error("pmt_f32_to_bf16: bad argument");
  if (n == 0) return PMT_OK;
  f32_to_bf16_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, x, (unsigned short*)y);
  return check_launch("f32_to_bf16_kernel");
}

int pmt_bf16_to_f32(long long n, const void* x, float* y, void* stream) {
  if (n < 0 || (n > 0 && (!x || !y))) return arg_error("pmt_bf16_to_f32: bad argument");
  if (n == 0) return PMT_OK;
  bf16_to_f32_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(n, (const unsigned short*)x, y);
  return check_launch("bf16_to_f32_kernel");
}

}  // extern "C"
