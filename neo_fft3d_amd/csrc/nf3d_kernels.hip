// gfx950 kernels of the denoiser other than the per-shape tile kernels
// (nf3d_tile.h, compiled per block shape from nf3d_shape.hip): the pattern
// estimator and the shape dispatcher.
#include "nf3d_fft.h"
#include "nf3d_internal.h"

namespace nf3d {

// ----------------------------------------------------------------- pattern
// Blocks of the pattern search (src/helper.cpp:60-63): two blocks of border.
__device__ __forceinline__ bool pattern_candidate(int nox, int noy, int bx, int by) {
  return by >= 2 && by < noy - 2 && bx >= 2 && bx < nox - 2;
}

// |X - g G|^2 times the pattern window, one coefficient (src/helper.cpp:66-75).
__device__ __forceinline__ float pattern_term(float2 c, float2 g, float gcur, float pw) {
#pragma clang fp contract(off)
  const float c0 = c.x - gcur * g.x, c1 = c.y - gcur * g.y;
  const float psd = c0 * c0 + c1 * c1;
  return psd * pw;
}

// Sum of the windowed, degrid-corrected power of each candidate block, in
// the reference's sequential float order (src/helper.cpp:57-89).  A wavefront
// per block: its 64 lanes read the spectrum, the gridsample and the pattern
// window row by row of 64 coefficients (coalesced, the next PS_ROWS rows in
// flight) and leave the terms in LDS; every lane then adds them in order, 16
// bytes a read.  Bound by that serial chain of bh * (bw/2+1) adds, which the
// blocks' wavefronts (two to three per SIMD at 1080p) run side by side; with
// a lane per block instead, every load was a line of its own and the few
// wavefronts waited for each: 137 us on a 1920x1080 plane's 2,232 blocks of
// 48x48, now 11.9 us.
constexpr int PS_CHUNK = 512;             // terms of a block in LDS at a time
constexpr int PS_ROWS = PS_CHUNK / 64;
__global__ void __launch_bounds__(64) k_pattern_sums(PatternJob J) {
#pragma clang fp contract(off)
  __shared__ __align__(16) float term[PS_CHUNK];
  const int b = blockIdx.x, l = threadIdx.x;
  const int by = b / J.nox, bx = b - by * J.nox;
  if (!pattern_candidate(J.nox, J.noy, bx, by)) {
    if (l == 0) J.sums[b] = 3.0e38f;
    return;
  }
  const int n = J.bh * J.outwidth;
  const float2* blk = J.spec + (size_t)b * n;
  const float gcur = J.degrid * blk[0].x / J.grid[0].x;
  float2 c[PS_ROWS], g[PS_ROWS];
  float w[PS_ROWS];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < PS_ROWS; u++) {
      const int k = min(k0 + u * 64 + l, n - 1);
      c[u] = blk[k];
      g[u] = J.grid[k];
      w[u] = J.pwin[k];
    }
  };
  load(0);
  float s = 0.0f;
  for (int k0 = 0; k0 < n; k0 += PS_CHUNK) {
#pragma unroll
    for (int u = 0; u < PS_ROWS; u++) term[u * 64 + l] = pattern_term(c[u], g[u], gcur, w[u]);
    __syncthreads();
    if (k0 + PS_CHUNK < n) load(k0 + PS_CHUNK);
    const int m = min(PS_CHUNK, n - k0);
    int k = 0;
#pragma unroll 4
    for (; k + 8 <= m; k += 8) {  // (every lane adds: the same sum)
      const float4 a = *reinterpret_cast<const float4*>(term + k), d = *reinterpret_cast<const float4*>(term + k + 4);
      s += a.x;
      s += a.y;
      s += a.z;
      s += a.w;
      s += d.x;
      s += d.y;
      s += d.z;
      s += d.w;
    }
    for (; k < m; k++) s += term[k];
    __syncthreads();
  }
  if (l == 0) J.sums[b] = s;
}

// The first strict minimum below 1e15 of n candidates in block order, `at(k,
// value, index)`: the smallest value, the lowest index of equal ones
// (src/helper.cpp:82-88).  256 lanes take the candidates in turn and meet in
// LDS (one lane alone waited for every load: k_pattern_set took 124 us on
// 1,856 sums, now 6.7 us).  Returns the index, 0x7fffffff for none, the value
// in rv[0].
constexpr int NO_BLOCK = 0x7fffffff;
template <class At>
__device__ __forceinline__ int first_minimum(int n, At at, float* rv, int* ri) {
  const int t = threadIdx.x;
  float best = 1e15f;
  int where = NO_BLOCK;
  for (int k = t; k < n; k += 256) {
    float s;
    int i;
    at(k, s, i);
    if (s < best) {
      best = s;
      where = i;
    }
  }
  __syncthreads();  // (a second search: the first one's result is read)
  rv[t] = best;
  ri[t] = where;
  __syncthreads();
  int h = 1;
  while (h < min(n, 256)) h <<= 1;  // lanes past n hold no block
  for (h >>= 1; h > 0; h >>= 1) {
    if (t < h && (rv[t + h] < rv[t] || (rv[t + h] == rv[t] && ri[t + h] < ri[t]))) {
      rv[t] = rv[t + h];
      ri[t] = ri[t + h];
    }
    __syncthreads();
  }
  return ri[0];
}

// ... over the sums of the search range's blocks in [x0, x1) x [y0, y1): the
// block's index by * nox + bx.
__device__ __forceinline__ int pattern_search(const PatternJob& J, int x0, int x1, int y0, int y1, float* rv, int* ri) {
  x0 = max(x0, 2);
  y0 = max(y0, 2);
  x1 = min(x1, J.nox - 2);
  y1 = min(y1, J.noy - 2);
  const int w = max(x1 - x0, 0), n = w * max(y1 - y0, 0);
  return first_minimum(
      n,
      [&](int k, float& s, int& i) {
        const int y = k / w;
        i = (y0 + y) * J.nox + x0 + (k - y * w);
        s = J.sums[i];
      },
      rv, ri);
}

// The search of each block row, for regions that take the whole plane's block.
__global__ void __launch_bounds__(256) k_pattern_rows(PatternJob J) {
  __shared__ float rv[256];
  __shared__ int ri[256];
  const int y = blockIdx.x, i = pattern_search(J, 0, J.nox, y, y + 1, rv, ri);
  if (threadIdx.x == 0) {
    J.row_min[y] = rv[0];
    J.row_at[y] = i;
  }
}

// The searched block, or the given one, and its pattern (src/helper.cpp:
// 82-88, 111-130).  One workgroup.
__global__ void __launch_bounds__(256) k_pattern_set(PatternJob J) {
#pragma clang fp contract(off)
  __shared__ float rv[256];
  __shared__ int ri[256];
  int px = J.px, py = J.py;
  if (px == 0 && py == 0) {
    const int i = pattern_search(J, 0, J.nox, 0, J.noy, rv, ri);
    if (i != NO_BLOCK) {
      py = i / J.nox;
      px = i - py * J.nox;
    }
  }
  if (threadIdx.x == 0) {
    J.choice[0] = px;
    J.choice[1] = py;
  }
  const float2* blk = J.spec + ((size_t)py * J.nox + px) * J.bh * J.outwidth;
  const float gcur = J.degrid * blk[0].x / J.grid[0].x;
  for (int k = threadIdx.x; k < J.bh * J.outwidth; k += blockDim.x)
    J.pattern2d[k] = pattern_term(blk[k], J.grid[k], gcur, J.pwin[k]);
}

// Spatially varying noise pattern (no reference counterpart; it generalises
// FindPatternBlock / SetPattern, src/helper.cpp:46-132, to regions): the
// block grid is cut into regions of rx x ry blocks, and each region takes the
// pattern of its own first strict minimum of the same sums over the blocks
// of the reference's search range (blocks 2..nox-3, 2..noy-3) that lie in
// it -- or, for a region with none of them, the block chosen for the whole
// plane: J.choice, written by k_pattern_set; null: the first minimum of the
// block rows' (J.row_min, written by k_pattern_rows), or without them
// searched here, see launch_pattern_regions.  The pattern goes to every
// block of the region: out2d = |X - g G|^2 pwin, out3d = out2d * mult3d
// (out3d null: out2d alone).  blockIdx.x: the region, blockIdx.y: 256 of the
// coefficients (1080p at 48x48 in regions of 4 x 4 has 144 regions, fewer
// than there are CUs).
__global__ void __launch_bounds__(256) k_pattern_regions(PatternJob J, int rx, int ry, float* out2d, float* out3d,
                                                         float mult3d) {
#pragma clang fp contract(off)
  __shared__ float rv[256];
  __shared__ int ri[256];
  const int nqx = (J.nox + rx - 1) / rx;
  const int qy = blockIdx.x / nqx, qx = blockIdx.x - qy * nqx;
  const int x0 = qx * rx, x1 = min(J.nox, x0 + rx), y0 = qy * ry, y1 = min(J.noy, y0 + ry);
  int c = pattern_search(J, x0, x1, y0, y1, rv, ri);
  if (c == NO_BLOCK) {  // (uniform)
    if (J.choice)
      c = J.choice[1] * J.nox + J.choice[0];
    else if (J.row_min)
      c = first_minimum(J.noy, [&](int k, float& v, int& i) { v = J.row_min[k]; i = J.row_at[k]; }, rv, ri);
    else
      c = pattern_search(J, 0, J.nox, 0, J.noy, rv, ri);
    if (c == NO_BLOCK) c = 0;
  }
  const int n = J.bh * J.outwidth;
  const int k = blockIdx.y * 256 + threadIdx.x;
  if (k >= n) return;
  const float2* blk = J.spec + (size_t)c * n;
  const float gcur = J.degrid * blk[0].x / J.grid[0].x;
  const float v = pattern_term(blk[k], J.grid[k], gcur, J.pwin[k]);
  const float v3 = v * mult3d;
  for (int by = y0; by < y1; by++)
    for (int bx = x0; bx < x1; bx++) {
      const size_t o = ((size_t)by * J.nox + bx) * n + k;
      out2d[o] = v;
      if (out3d) out3d[o] = v3;
    }
}

// ---------------------------------------------------------------- dispatch
// Block shapes compiled for k_tile (one translation unit each).
#define NF3D_SHAPES(X) X(8, 8) X(16, 16) X(24, 24) X(32, 32) X(48, 48) X(64, 64) X(32, 16) X(16, 32)

#define X(W, H)                                                                                          \
  hipError_t launch_tile_##W##x##H(int mode, int bt, int onchip, int mf, const TileLaunch& l, hipStream_t s); \
  hipError_t launch_run_##W##x##H(int mode, int bt, int shp, int mf, const RunBatch& l, hipStream_t s); \
  hipError_t launch_seam_run_##W##x##H(int mf, const RunBatch& l, hipStream_t s);
NF3D_SHAPES(X)
#undef X

bool block_shape_supported(int bw, int bh) {
#define X(W, H) if (bw == W && bh == H) return true;
  NF3D_SHAPES(X)
#undef X
  return false;
}

int tile_blocks_per_wg(int bw, int bh) {
  // TShape<BW,BH,128>::BPW: 128 lanes / max(bw/2+1, bh/2)
  int cols = bw / 2 + 1, pairs = bh / 2;
  return 128 / (cols > pairs ? cols : pairs);
}

int run_blocks_per_wg(int bw, int bh, int mf) {
  // RunShape<BW,BH,MF>::BPW
  return mf && bw == 48 && bh == 48 ? 4 : tile_blocks_per_wg(bw, bh);
}

bool mfma_dft_supported(int bw, int bh) { return bw == bh && (bw == 32 || bw == 48 || bw == 64); }

hipError_t launch_tile(int mode, int bt, int onchip, int mf, int bw, int bh, const TileLaunch& l, hipStream_t s) {
  if (mf && !mfma_dft_supported(bw, bh)) return hipErrorInvalidValue;
#define X(W, H) if (bw == W && bh == H) return launch_tile_##W##x##H(mode, bt, onchip, mf, l, s);
  NF3D_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_run(int mode, int bt, int shp, int mf, int bw, int bh, const RunBatch& l, hipStream_t s) {
  if (mf && !mfma_dft_supported(bw, bh)) return hipErrorInvalidValue;
#define X(W, H) if (bw == W && bh == H) return launch_run_##W##x##H(mode, bt, shp, mf, l, s);
  NF3D_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_seam_run(int mf, int bw, int bh, const RunBatch& l, hipStream_t s) {
#define X(W, H) if (bw == W && bh == H) return launch_seam_run_##W##x##H(mf, l, s);
  NF3D_SHAPES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_pattern(const PatternJob& J, hipStream_t s) {
  int nb = J.nox * J.noy;
  hipLaunchKernelGGL(k_pattern_sums, dim3(nb), dim3(64), 0, s, J);
  if (J.choice) hipLaunchKernelGGL(k_pattern_set, dim3(1), dim3(256), 0, s, J);
  return hipGetLastError();
}

// Blocks of a plane past which regions without a block of the search range
// take the plane's from the block rows' minima instead of each searching the
// plane: the rows' launch costs 2 us, a search one more for every 3,000 blocks
// and all the border regions' searches together the caches' rate.  Whole call,
// search and rows: 2,310 blocks 22 and 23 us, 3,726 72 and 73 (in regions of one
// block 90 and 87), 8,349 59 and 57, 32,776 76 and 59, 519,901 of 8x8 in regions
// of one block (5,992 of them on the border) 2,516 and 660.
constexpr int REGION_SCAN = 4096;
hipError_t launch_pattern_regions(const PatternJob& J, int rx, int ry, float* out2d, float* out3d, float mult3d,
                                  hipStream_t s) {
  if (rx < 1 || ry < 1) return hipErrorInvalidValue;
  const int nqx = (J.nox + rx - 1) / rx, nqy = (J.noy + ry - 1) / ry, nq = nqx * nqy;
  const int nk = (J.bh * J.outwidth + 255) / 256;
  PatternJob P = J;
  if (!J.choice && J.row_min) {
    // regions without a block of the search range, those of the plane's
    // border: region columns (rows) with one have a block in [2, n - 2)
    auto searched = [](int n, int r) { return n > 4 ? (n - 3) / r - 2 / r + 1 : 0; };
    if (J.nox * J.noy > REGION_SCAN && searched(J.nox, rx) * searched(J.noy, ry) < nq)
      hipLaunchKernelGGL(k_pattern_rows, dim3(J.noy), dim3(256), 0, s, J);
    else
      P.row_min = nullptr;
  }
  hipLaunchKernelGGL(k_pattern_regions, dim3(nq, nk), dim3(256), 0, s, P, rx, ry, out2d, out3d, mult3d);
  return hipGetLastError();
}

}  // namespace nf3d
