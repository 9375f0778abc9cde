// Frame-loop kernel of the denoiser: k_run<BW,BH,NT,MODE,BT,SHP,MF>.
//
// A workgroup owns one tile (up to BPW horizontally adjacent blocks of one
// block row, the tile of k_tile) and filters it for a run of consecutive
// frames, so one launch covers many frames and no workgroup waits for the
// others between frames.  Per frame the phases are those of k_tile (gather,
// row r2c, column FFT, spectral pass, column inverse, row c2r, overlap-add);
// what changes is where the data waits are:
//   - the spectral pass runs down each column in chunks of rows: the ring
//     spectra / Kalman state of chunk k+DR (DR up to 3) and the table rows of
//     chunk k+1 are loaded while chunk k is computed; the first chunks are
//     loaded before the forward column FFT;
//   - the gains are specialised at compile time on the sharpen / dehalo case
//     (SHP) and degrid is branch-free (a zero fraction when it is off).
// Wiener 3D: the newest frame of each window (frame m + (BT-1)/2) is
// transformed on chip and stored to ring slot (frame % BT); the BT-1 older
// spectra are the ones the same lanes stored in earlier iterations (or the
// launches before), so the loop needs no synchronisation beyond the
// workgroup.  Kalman state likewise stays with its tile.  Seam partials go to
// a per-frame seam buffer that k_seam_run finishes after the launch.  With MF
// the row and column transforms are the matrix-core DFT products of
// nf3d_mfma.h (32x32, 48x48 and 64x64 blocks).
#pragma once
#include "nf3d_tile.h"

namespace nf3d {

__device__ __forceinline__ const RunBatch& kernarg_batch(const RunBatch& arg) {
#if defined(__HIP_DEVICE_COMPILE__)
  (void)arg;
  return *(const RunBatch*)__builtin_amdgcn_kernarg_segment_ptr();
#else
  return arg;
#endif
}

// The same record through an offset the compiler cannot see through (zero at
// run time): loads of launch fields inside a loop stay in the loop instead of
// being hoisted into registers that live across it.
__device__ __forceinline__ const RunBatch& kernarg_batch_opaque(const RunBatch& arg) {
#if defined(__HIP_DEVICE_COMPILE__)
  (void)arg;
  int zero = 0;
  asm volatile("" : "+s"(zero));
  return *(const RunBatch*)((const char*)__builtin_amdgcn_kernarg_segment_ptr() + zero);
#else
  return arg;
#endif
}

// The job of a workgroup: the last one whose first workgroup it is past.
__device__ __forceinline__ int batch_job(const RunBatch& B, int wg) {
  int jb = 0;
  for (int k = 1; k < B.njobs; k++)
    if (wg >= B.job[k].wg_begin) jb = k;
  return jb;
}

// Wavefront of a lane index, as a scalar value.
__device__ __forceinline__ int wave_of(int t) { return __builtin_amdgcn_readfirstlane(t >> 6); }

// A workgroup's tile: a lane pair per spectral column and per row pair of
// each block, so that BPW blocks fill the 256 lanes.  The matrix-core form of
// 48x48 blocks takes four, one per wavefront: a fifth costs its transforms a
// second round in which three wavefronts wait (tiles are only a split of the
// work: every pixel's sums keep their order).
template <int BW, int BH, bool MF>
struct RunShape : TShape<BW, BH, 128, (MF && BW == 48 && BH == 48) ? 4 : 0> {};

// ------------------------------------------- gather / overlap-add by column
// Lane (block b, column j) reads block b's column j of every row straight
// from the plane (reflect-101 addressing), kept as bits so that no use waits
// on a load before the windowing.  Lanes past the tile's blocks load its last
// block's.
template <int BW, int BH>
__device__ __forceinline__ void gather_load(const PlaneJob& J, uint32_t (&raw)[BH], const uint8_t* src,
                                            const int* rowoff, int bx0, int nblk, int stepx, int t) {
  const int tb = t / BW, b = min(tb, nblk - 1), j = t - tb * BW;
  const int sx = reflect101((bx0 + b) * stepx + j - J.mirw, J.Wc) + J.lc;
  // 32-bit byte offsets from the uniform plane base: one add per sample
  // (rows are < 2^31 bytes from the base: checked by the host)
  auto load = [&](auto* as) {
    using T = typename std::remove_pointer<decltype(as)>::type;
    const int sxb = sx * (int)sizeof(T);
    static_for<0, BH>([&](auto ii) {
      raw[ii] = *reinterpret_cast<const T*>(src + (unsigned)(rowoff[decltype(ii)::value] + sxb));
    });
  };
  if (J.pix == 1) load((uint8_t*)nullptr);  // (uniform)
  else if (J.pix == 2) load((uint16_t*)nullptr);
  else load((uint32_t*)nullptr);
}

// The loaded samples, windowed, into the block's row pairs.  The window
// product is (p * wx) * wy for every sample: the value of the
// region-by-region order of gather_tile (wx or wy is exactly 1 outside its
// bands) except in the bands at the plane's top and bottom edge, where that
// order multiplies by wy first, or by wx * wy at the corners; one rounding
// apart (the parity bar is against the FP64 product).  EDGE: that order there
// too (the matrix-core form keeps it; only tiles of the first and last block
// row pay for the selection).
template <int BW, int BH, int SA, int LA, bool EDGE>
__device__ __forceinline__ void gather_window(const PlaneJob& J, float2* stage, const uint32_t (&raw)[BH],
                                              const float* winx, const float* winy, int by, int bx0, int nblk, int t) {
  const int b = t / BW, j = t - b * BW;
  if (b >= nblk) return;  // lanes past the tile's blocks
  const float wx = winx[j];
  float* d = reinterpret_cast<float*>(&stage[b * LA + j]);
  auto window = [&](auto value) {  // (value: the sample less the centring)
    if constexpr (EDGE) {
      const int top = by == 0 ? J.oh : 0, bot = by == J.noy - 1 ? BH - J.oh : BH;  // uniform
      const int bx = bx0 + b;
      const bool xedge = (bx == 0 && j < J.ow) || (bx == J.nox - 1 && j >= BW - J.ow);
      static_for<0, BH>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        const float px = value(raw[i]), wy = winy[i];
        const bool yedge = i < top || i >= bot;
        const float f0 = yedge ? (xedge ? wx * wy : wy) : wx;
        const float f1 = yedge ? (xedge ? 1.0f : wx) : wy;
        d[(i >> 1) * SA * 2 + (i & 1)] = (px * f0) * f1;
      });
    } else {
      static_for<0, BH>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        const float px = value(raw[i]);
        d[(i >> 1) * SA * 2 + (i & 1)] = (px * wx) * winy[i];
      });
    }
  };
  const float base = J.base;
  if (J.pix == 4) window([](uint32_t r) { return __uint_as_float(r); });  // (uniform; float planes are not centred)
  else if (base == 0.0f) window([](uint32_t r) { return (float)r; });
  else window([=](uint32_t r) { return (float)r - base; });
}

// n / d for 0 <= n < 2^22 and 1 <= d <= 64 (inv = 1/d rounded): the float
// quotient is within one of the exact one, and one correction each way
// makes it exact.
__device__ __forceinline__ int div_small(int n, int d, float inv) {
  int q = (int)((float)n * inv);
  const int r = n - q * d;
  q += r >= d ? 1 : 0;
  q -= r < 0 ? 1 : 0;
  return q;
}

// Overlap-add of the tile rows [r0, r1) (uniform) in NQ tile columns per lane,
// xl + 64 q, in the reference's float order (src/buffer.cpp:381-560): the
// columns' block(s), synthesis weights and offsets are worked out once; then
// the rows of the upper band, of this block row alone and of the lower band
// each in a loop without a condition per row, the LDS reads of RC rows in
// every column together.  A loop's last rows may repeat its last row (the same
// value to the same place).  wsyn: [left x (BW) | right x (BW) | top y (BH) |
// bottom y (BH)], the y windows times norm; rowdst: element offset of each
// tile row in a seam plane (x) and in the destination (y).  Both in LDS: a
// global load here would wait (vmcnt counts stores too) for every store
// issued before it.
template <int PIX, int BW, int BH, int LSYN, int SYNW, int NQ>
__device__ __forceinline__ void overlap_rows(const PlaneJob& J, uint8_t* dst, float* seam, const float* syn,
                                             const float* wsyn, const int2* rowdst, int by, int bx0, int nblk, int RW,
                                             int stepx, int stepy, int xl, int r0, int r1) {
  constexpr int XL = 0, XR = BW, YL = 2 * BW, YR = 2 * BW + BH, RC = 4;
  using T = typename std::conditional<PIX == 1, uint8_t, typename std::conditional<PIX == 2, uint16_t, float>::type>::type;
  const float rounder = PIX == 4 ? 0.0f : 0.5f;
  const float fbase = (float)J.obase, norm = J.norm;
  const int ow = J.ow, oh = J.oh, maxval = J.maxval;
  const int P = (int)J.seam_plane;
  T* dpl = reinterpret_cast<T*>(dst + (long long)J.tc * J.dst_pitch + (long long)J.lc * sizeof(T));
  const float inv = 1.0f / (float)stepx;
  // x class: 0 exclusive column, 1 band inside the tile, 2 band shared with
  // the left tile (this tile holds its right block), 3 band shared with the
  // right tile (this tile holds its left block), 4 outside the plane
  int cls[NQ], la[NQ], lb[NQ], x[NQ];
  float wa[NQ], wb[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int xq = xl + 64 * q, xt = min(xq, RW - 1);
    x[q] = bx0 * stepx + xq - J.mirw;
    const int bl = min(div_small(xt, stepx, inv), nblk - 1), j = xt - bl * stepx;
    const bool right = j >= stepx;            // past the last block's body
    const bool left = !right && j < ow;
    const bool inner = left && bl >= 1;
    lb[q] = bl * LSYN + j;
    la[q] = inner ? lb[q] - LSYN + stepx : lb[q];
    wa[q] = right ? wsyn[XR + min(j - stepx, BW - 1)] : inner ? wsyn[XR + j] : 0.0f;
    wb[q] = right ? 0.0f : left ? wsyn[XL + j] : 1.0f;
    cls[q] = right ? 3 : left ? (inner ? 1 : 2) : 0;
    if (xq >= RW || x[q] < 0 || x[q] >= J.Wc) cls[q] = 4;
  }
  // the tile rows inside the plane
  const int y0 = max(r0, J.mirh - by * stepy), y1 = min(r1, J.Hc + J.mirh - by * stepy);
  auto rows = [&](int a, int b, auto&& body) {
#pragma unroll 1
    for (int i = a; i < b; i += RC) {
      int ii[RC];
      float h[NQ][RC];
#pragma unroll
      for (int u = 0; u < RC; u++) ii[u] = min(i + u, b - 1);
#pragma unroll
      for (int q = 0; q < NQ; q++)
#pragma unroll
        for (int u = 0; u < RC; u++) h[q][u] = syn[la[q] + ii[u] * SYNW] * wa[q] + syn[lb[q] + ii[u] * SYNW] * wb[q];
      body(ii, h);
    }
  };
  // rows of two block rows: the seam buffer gets this one's part.  Row seam:
  // slot 0 = upper block row's part, slot 1 = lower's (times its window).
  // Corner: A upper-left, B upper-right, C lower-left, D lower-right.
  auto band = [&](int a, int b, int yw, bool top) {
    rows(a, b, [&](const int (&ii)[RC], const float (&h)[NQ][RC]) {
      int o[RC];
      float w[RC];
#pragma unroll
      for (int u = 0; u < RC; u++) {
        o[u] = rowdst[ii[u]].x;
        w[u] = wsyn[yw + ii[u]];
      }
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        if (cls[q] == 4) continue;
        const int slot = top ? (cls[q] <= 1 ? 1 : cls[q] == 3 ? 2 : 3) : (cls[q] == 2 ? 1 : 0);
        const int so = slot * P + x[q];
#pragma unroll
        for (int u = 0; u < RC; u++) seam[(unsigned)(o[u] + so)] = cls[q] <= 1 ? h[q][u] * w[u] : h[q][u];
      }
    });
  };
  band(y0, min(y1, oh), YL, true);
  // rows of this block row only: pixels, or, in the columns shared with the
  // neighbouring tiles, parts (slot 0 = left block's, slot 1 = right's)
  rows(max(y0, oh), min(y1, stepy), [&](const int (&ii)[RC], const float (&h)[NQ][RC]) {
    int2 o[RC];
#pragma unroll
    for (int u = 0; u < RC; u++) o[u] = rowdst[ii[u]];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      if (cls[q] <= 1) {
#pragma unroll
        for (int u = 0; u < RC; u++) {
          const float v = h[q][u] * norm + rounder + fbase;
          T px;
          if constexpr (PIX == 4) {
            const float p = v < 0.0f ? 0.0f : v;
            px = p > 1.0f ? 1.0f : p;
          } else {
            int qi = (int)v;
            qi = qi < 0 ? 0 : qi;
            px = (T)(qi > maxval ? maxval : qi);
          }
          dpl[(unsigned)(o[u].y + x[q])] = px;
        }
      } else if (cls[q] <= 3) {
        const int so = (cls[q] == 3 ? 0 : P) + x[q];
#pragma unroll
        for (int u = 0; u < RC; u++) seam[(unsigned)(o[u].x + so)] = h[q][u];
      }
    }
  });
  band(max(y0, stepy), y1, YR - stepy, false);
}

// Overlap-add of the tile.  From 32 rows on, the four wavefronts take a
// quarter of the rows each, every lane the columns 64 apart (a tile is some
// 170 columns wide: one lane per column for all rows leaves the last
// wavefront without work); with fewer rows, setting up several columns a lane
// costs more than it spreads.  In thousands of cycles a 48x48 frame: 25 (one
// lane a column, conditions and LDS reads row by row), 17 (row loops), 12 (all
// columns together); UHD bt=5 64/16, 10 frames: 3280 -> 3000 us.
template <int PIX, int BW, int BH, int BPW, int LSYN, int SYNW, int QM>
__device__ __forceinline__ void overlap_cols(const PlaneJob& J, uint8_t* dst, float* seam, const float* syn,
                                             const float* wsyn, const int2* rowdst, int by, int bx0, int nblk, int RW,
                                             int stepx, int stepy, int t) {
  if constexpr (BH >= 32) {
    const int r0 = wave_of(t) * (BH / 4);
    constexpr int NQ = (BPW * BW + 63) / 64;  // without overlap; one less is the usual case
    if constexpr (QM < NQ) {  // (fewer registers)
#pragma unroll 1
      for (int x0 = 0; x0 < RW; x0 += 64 * QM)
        overlap_rows<PIX, BW, BH, LSYN, SYNW, QM>(J, dst, seam, syn, wsyn, rowdst, by, bx0, nblk, RW, stepx, stepy,
                                                  x0 + (t & 63), r0, r0 + BH / 4);
    } else if (RW <= (NQ - 1) * 64)
      overlap_rows<PIX, BW, BH, LSYN, SYNW, NQ - 1>(J, dst, seam, syn, wsyn, rowdst, by, bx0, nblk, RW, stepx, stepy,
                                                    t & 63, r0, r0 + BH / 4);
    else
      overlap_rows<PIX, BW, BH, LSYN, SYNW, NQ>(J, dst, seam, syn, wsyn, rowdst, by, bx0, nblk, RW, stepx, stepy,
                                                t & 63, r0, r0 + BH / 4);
  } else {
    overlap_rows<PIX, BW, BH, LSYN, SYNW, 1>(J, dst, seam, syn, wsyn, rowdst, by, bx0, nblk, RW, stepx, stepy, t, 0,
                                             BH);
  }
}

// ------------------------------------------------------------ spectral pass
// Sharpen / dehalo factor of one element (src/code_impl/Sharpen.cpp:102-105);
// for SHP_GENERAL the sharpen factor is exactly 1 when sharpen == 0, so the
// product equals the reference's dehalo-only factor.
template <int SHP>
__device__ __forceinline__ float shp_factor(const SpecParams& J, float psd, float wsh, float wdh) {
  if constexpr (SHP == SHP_SHARPEN) return sharpen_factor(J, psd, wsh);
  else return sharpen_factor(J, psd, wsh) * dehalo_factor(J, psd, wdh);
}

// Sharpen pass of one element (src/code_impl/Sharpen.cpp:13-133); degrid
// fraction zero when degrid is off.
template <int SHP>
__device__ __forceinline__ float2 sharpen_s(const SpecParams& J, float2 x, const Tab& T, float gf) {
  const float g0 = gf * T.g.x, g1 = gf * T.g.y;
  const float cr = x.x - g0, ci = x.y - g1;
  const float psd = power(cr, ci);
  const float f = shp_factor<SHP>(J, psd, T.wsh, T.wdh);
  return make_float2(fmaf_(cr, f, g0), fmaf_(ci, f, g1));
}

// Apply2D (src/code_impl/Apply.cpp:13-65) with the sharpen factor folded in
// when no pattern is used.
template <int SHP>
__device__ __forceinline__ float2 apply2d_s(const SpecParams& J, float2 x, const Tab& T, float gf) {
  const float g0 = gf * T.g.x, g1 = gf * T.g.y;
  const float cr = x.x - g0, ci = x.y - g1;
  const float psd = power(cr, ci);
  float f = fmaf_(-T.sig, __builtin_amdgcn_rcpf(psd), 1.0f);
  f = __builtin_fmaxf(f, J.lowlimit);  // f is never NaN (psd >= 1e-15)
  if constexpr (SHP != SHP_NONE) {
    if (!J.use_pattern) f *= shp_factor<SHP>(J, psd, T.wsh, T.wdh);
  }
  return make_float2(fmaf_(cr, f, g0), fmaf_(ci, f, g1));
}

// One chunk of CH rows of a lane's column: the ring spectra / Kalman state
// (HBM, loaded several chunks ahead) and the table values (cache-resident,
// one chunk ahead).
template <int MODE, int NQ, int CH>
struct RingBuf {
  float2 v[NQ > 0 ? NQ : 1][CH];
  KalState ks[MODE == MODE_KALMAN ? CH : 1];
};
template <int SHP, int CH>
struct TabBuf {
  float2 g[CH];
  float sig[CH];
  float wsh[SHP != SHP_NONE ? CH : 1];
  float wdh[SHP == SHP_GENERAL ? CH : 1];
};

// ------------------------------------------------------------- split FFTs
// A transform of N points is split over a pair of lanes l and l + 32 of a
// wavefront (h = 0, 1): two transforms of N/2 points, of the even values on
// lane l and of the odd ones on lane l + 32, and one radix-2 step.  The swap
// below gives each lane both operands of half of that step's butterflies, so
// no lane computes a butterfly's half that the other lane also computes (with
// a full exchange, both lanes twiddled and half of the results were thrown
// away: 10 instructions a value instead of 6).

// Exchanges a of the upper 32 lanes with b of the lower 32.
__device__ __forceinline__ void half_swap(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void half_swap(float2& a, float2& b) {
  half_swap(a.x, b.x);
  half_swap(a.y, b.y);
}
// The other lane's value of the pair.
__device__ __forceinline__ float2 half_other(float2 v, int h) {
  float2 a = v, b = v;
  half_swap(a, b);  // a: the lower lanes' value, b: the upper lanes'
  return h ? a : b;
}

// Forward radix-2 step: in, c[k] = E[k] (lane 0) / O[k] (lane 1), k < N/2; out,
// X[k] = E[k] + w^k O[k] and X[k + N/2] = E[k] - w^k O[k], w = exp(-2 pi i / N):
// lane h holds X[h N/4 + i] in c[i] and X[N/2 + h N/4 + i] in c[N/4 + i],
// i < N/4.  (w^(k + N/4) = -i w^k: the same product, turned, on lane 1.)
template <int N>
__device__ __forceinline__ void split_combine_fwd(float2 (&c)[N / 2], int h) {
  static_for<0, N / 4>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    float2 e = c[k], o = c[k + N / 4];
    half_swap(e, o);
    if constexpr (k != 0) {
      constexpr float wr = (float)ct::cos2pi(k, N), wi = (float)(-ct::sin2pi(k, N));
      o = cmul(o, wr, wi);
    }
    o = h ? make_float2(o.y, -o.x) : o;
    c[k] = cadd(e, o);
    c[k + N / 4] = csub(e, o);
  });
}

// Inverse of the above (unnormalised, FFTW c2r convention), X in lane h as
// split_combine_fwd leaves it: the even values come from the N/2-point
// inverse transform of X[k] + X[k + N/2], the odd ones from that of
// w^-k (X[k] - X[k + N/2]); lane h ends with the inputs of its half.
template <int N>
__device__ __forceinline__ void split_combine_inv(float2 (&c)[N / 2], int h) {
  static_for<0, N / 4>([&](auto kk) {
    constexpr int k = decltype(kk)::value;
    float2 s = cadd(c[k], c[k + N / 4]), d = csub(c[k], c[k + N / 4]);
    if constexpr (k != 0) {
      constexpr float wr = (float)ct::cos2pi(k, N), wi = (float)ct::sin2pi(k, N);
      d = cmul(d, wr, wi);
    }
    d = h ? make_float2(-d.y, d.x) : d;
    half_swap(s, d);
    c[k] = s;
    c[k + N / 4] = d;
  });
}

// ------------------------------------------------------------------ kernel
// Register arrays (row and column transforms, chunk buffers) are computed by
// every lane, idle lanes on a duplicate of a valid column (indices clamped to
// the tile), and only stores are predicated: a register written under a lane
// mask keeps its old value in the other lanes, which would hold it live around
// the frame loop.
//
// Each spectral column has a lane pair, which runs the spectral pass over half
// of the column's rows each.
//
// FFT form: gather and overlap-add by column; the row transforms use the first
// BPW * BH/2 * 2 lanes (the other wavefronts skip them); a lane pair splits a
// row pair's or a column's transform in two half-length transforms
// (split_combine_*).
//
// MF: the 2D transforms as DFT-matrix products on the matrix cores (32x32,
// 48x48 and 64x64 blocks, nf3d_mfma.h), a wavefront per block in turn, in
// place of the row and column FFTs.  With two lanes a column and rolled tile
// loops it takes 128 / 155 / 188 registers (32 / 48 / 64, bt = 3), so two to
// four wavefronts share a SIMD: 48/16 on 3840x2160 4:2:0, 8 frames, 3480 us
// at one wavefront per SIMD with 424 registers, 1800 us with that change alone,
// 1600 now.
//
// Waves per SIMD the register budget is cut for (LDS allows three workgroups
// per CU at 48x48): three, or two for the variants whose spectral pass holds
// more per element (four or five frames, the dehalo factor, the Kalman state
// with a sharpen pass, 64-row columns), which would otherwise spill.
template <int BH, int MODE, int BT, int SHP, bool RES>
constexpr int run_waves_per_simd() {
  if constexpr (BH >= 64 || (MODE == MODE_W3D && (BT >= 4 || SHP == SHP_GENERAL)) ||
                (MODE == MODE_KALMAN && (SHP != SHP_NONE || (RES && BH > 32))))
    return 2;
  else return 3;
}

//
// RES (Kalman): a lane keeps its elements' state in registers from the first
// frame of a launch to its last (12 bytes an element: 48 registers at 32x32,
// 72 at 48x48) instead of reading and writing it for every frame: UHD 4:2:0
// 10-bit, 11 frames a launch, 8x8 1289 -> 760 us, 16x16 1569 -> 975, 24x24
// 1530 -> 1080, 32x32 1452 -> 1140, 48x48 1477 -> 1350.  At 64x64 96 more do
// not fit (344 bytes of scratch a lane: 1649 -> 2437).
template <int BW, int BH, int NT, int MODE, int BT, int SHP, bool MF = false, bool RES = false>
__global__ void __launch_bounds__(NT, (run_waves_per_simd<BH, MODE, BT, SHP, RES>())) k_run(RunBatch B_arg) {
  const RunBatch& B0 = kernarg_batch(B_arg);
  const int jb = batch_job(B0, blockIdx.x);
  const RunLaunch& L0 = B0.job[jb];
  using S = RunShape<BW, BH, MF>;
  static_assert(NT == 256, "a lane pair per spectral column of BPW blocks");
  constexpr int CR = BH / 2;  // spectral rows per column lane
  constexpr int COLS = S::COLS, PAIRS = S::PAIRS, BPW = S::BPW, SR = S::SR, LSPEC = S::LSPEC;
  constexpr int SYNW = S::SYNW, LSYN = S::LSYN, SA = S::SA, LA = S::LA;
  constexpr int FROM = MODE == MODE_W3D ? -(BT / 2) : 0;
  constexpr int TO = MODE == MODE_W3D ? (BT - 1) / 2 : 0;
  constexpr int NQ = MODE == MODE_W3D ? BT - 1 : 0;  // ring frames per element
  constexpr int CH = (MODE == MODE_W3D) ? 4 : 2;  // rows per chunk (two chunks of loads in flight)
  constexpr int NCH = CR / CH;
  static_assert(CR % CH == 0 && BH % 8 == 0 && BW % 4 == 0, "block shape");
  // MODE_FWD: the forward transforms only, frame m0 + i stored to ring slot
  // (m0 + i) % BT -- the Wiener-3D window frames a range starts with, so
  // every spectrum in the ring comes from this kernel's arithmetic
  // chunks of ring rows in flight ahead of the one being computed
  // (a register budget of 168 for three wavefronts per SIMD)
  constexpr int DR = MODE == MODE_W3D && NQ <= 2 ? 2 : 1;
  using RBuf = RingBuf<MODE, NQ, CH>;
  using TBuf = TabBuf<SHP, CH>;
  __shared__ __align__(16) unsigned char smem[S::BYTES];
  __shared__ float s_gf[BPW], s_gfs[BPW];
  __shared__ __align__(16) float winx[BW];
  __shared__ __align__(16) float winy[BH];
  __shared__ __align__(16) float wsyn[2 * BW + 2 * BH];  // synthesis windows: left, right, top, bottom bands
  // byte offset of the source row of each tile row (< 2^31: checked by the host)
  __shared__ __align__(16) int rowoff[BH];
  // element offsets of each tile row in a seam plane and in the destination
  __shared__ __align__(16) int2 rowdst[BH];
  float2* spec = reinterpret_cast<float2*>(smem);
  float2* stage = reinterpret_cast<float2*>(smem);
  float* syn = reinterpret_cast<float*>(smem);

  // ---- tile and frames of this workgroup
  const int g = blockIdx.x - L0.wg_begin;
  const int chunk = g / L0.ntiles;
  const int tile = g - chunk * L0.ntiles;
  const int i0 = chunk * L0.fpw;
  const int i1 = min(L0.nframes, i0 + L0.fpw);
  const int by = tile / L0.J.ntx;
  const int bx0 = (tile - by * L0.J.ntx) * BPW;
  const int nblk = min(BPW, L0.J.nox - bx0);
  const int stepx = BW - L0.J.ow, stepy = BH - L0.J.oh;
  const int RW = (nblk - 1) * stepx + BW;
  {
    const PlaneJob& J = L0.J;
    const int t = threadIdx.x;
    for (int i = t; i < BW; i += NT) winx[i] = J.wanx[i];
    for (int i = t; i < BH; i += NT) {
      // (the FFT form's row transforms take halved samples: exact)
      winy[i] = MF ? J.wany[i] : 0.5f * J.wany[i];
      rowoff[i] = (int)((long long)(cover_to_src_row(J, by * stepy + i) + J.tc) * J.src_pitch);
      const int yo = interior_to_out_row(J, by * stepy + i - J.mirh);  // (used inside the plane only)
      rowdst[i] = make_int2(yo * J.Wc, yo * (int)(J.dst_pitch / (long long)J.pix));
    }
    for (int i = t; i < J.ow; i += NT) {
      wsyn[i] = J.wsynxl[i];
      wsyn[BW + i] = J.wsynxr[i];
    }
    for (int i = t; i < J.oh; i += NT) {
      wsyn[2 * BW + i] = J.wsynyl[i] * J.norm;
      wsyn[2 * BW + BH + i] = J.wsynyr[i] * J.norm;
    }
  }
  __syncthreads();

  // Wiener 3D loads a frame's samples ahead, to be in flight during the
  // overlap-add of the frame before (48x48: 7.9 of 69 thousand cycles of a
  // frame were that wait; 1080p 64 frames 2416 -> 2372 us).  The other modes
  // have the registers for more wavefronts instead, which hide it as well
  // (Kalman), or one frame a workgroup (2D).
  constexpr bool AHEAD = MODE == MODE_W3D;
  uint32_t raw[BH];
  if constexpr (AHEAD) gather_load<BW, BH>(L0.J, raw, L0.src[i0], rowoff, bx0, nblk, stepx, (int)threadIdx.x);
  // the lane's Kalman state (RES; lanes past the tile's columns hold a copy of
  // one of them, and store nothing)
  static_assert(!RES || MODE == MODE_KALMAN, "the resident state is the Kalman mode's");
  KalState kst[RES ? CR : 1];
  auto state_at = [&](auto ii) {
    constexpr int i = decltype(ii)::value;
    const int t = threadIdx.x, cl = (t >> 6) * 32 + (t & 31), hh = (t >> 5) & 1;
    const int cbr = cl / COLS, cc = cl - cbr * COLS, cb = min(cbr, nblk - 1);
    return ((size_t)(by * L0.J.nox + bx0) + cb) * (BH * COLS) +
           (size_t)(hh * (CR / 2) + i + (i >= CR / 2 ? CR / 2 : 0)) * COLS + cc;
  };
  if constexpr (RES)
    static_for<0, CR>([&](auto i) { kst[i] = KalState{L0.J.kal_last[state_at(i)], L0.J.kal_sum[state_at(i)]}; });
#pragma unroll 1
  for (int fi = i0; fi < i1; fi++) {
    // The lane index, the launch record and the LDS tables are reached
    // through values the compiler cannot see through, so lane addresses and
    // launch fields are recomputed inside the loop instead of hundreds of
    // loop-invariant values being kept live across it.
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    int zo = 0;
    asm volatile("" : "+s"(zo));
    const RunLaunch& L = kernarg_batch_opaque(B_arg).job[jb];
    const PlaneJob& J = L.J;
    const float* wx = winx + zo;
    const float* wy = winy + zo;
    const int* ro = rowoff + zo;
    const int m = L.m0 + fi;
    // column lanes: a pair (l, l + 32) per column, half hh: rows hh * CR/2 + i
    // and BH/2 + hh * CR/2 + i, i < CR/2, of the spectrum after the forward
    // transform (value j of the lane: row hh * CR/2 + col_row(j))
    const int cl = (t >> 6) * 32 + (t & 31), hh = (t >> 5) & 1;
    const int cbr = cl / COLS, cc = cl - cbr * COLS;
    const bool col_on = cbr < nblk;
    const int cb = col_on ? cbr : nblk - 1;
    // row lanes: a pair per row pair
    const int rbr = cl / PAIRS, rp = cl - rbr * PAIRS;
    const bool row_on = rbr < nblk;
    const int rb = row_on ? rbr : nblk - 1;
    // wavefronts with no row pair of the tile skip the row transforms
    const bool row_wave = wave_of(t) * 32 < BPW * PAIRS;
    const size_t tile_spec0 = (size_t)(by * J.nox + bx0) * (BH * COLS);
    // element (hh * CR/2, cc) of this lane's column: its first spectral row
    const size_t colo = tile_spec0 + (size_t)cb * (BH * COLS) + (size_t)(hh * (CR / 2)) * COLS + cc;
    // the pattern: one for the plane, or this block's (learned PSD)
    const float* pat = J.use_pattern ? (MODE == MODE_W3D ? J.pattern3d : J.pattern2d) +
                                           (J.pattern_per_block ? colo - cc : (size_t)(hh * (CR / 2)) * COLS)
                                     : nullptr;
    const float grid0 = J.grid[0].x;
    const SpecParams SP(J);

    // ---- 1. windowed pixels into per-block row pairs
    if constexpr (!AHEAD) gather_load<BW, BH>(J, raw, L.src[fi], ro, bx0, nblk, stepx, t);
    if (MF && (by == 0 || by == J.noy - 1)) gather_window<BW, BH, SA, LA, MF>(J, stage, raw, wx, wy, by, bx0, nblk, t);
    else gather_window<BW, BH, SA, LA, false>(J, stage, raw, wx, wy, by, bx0, nblk, t);
    __syncthreads();
    if constexpr (MF) {
      // ---- 2-3. 2D r2c on the matrix cores, in rounds of one block per
      // wavefront, highest blocks first.  Spectral block b overlaps only the
      // gather stage of blocks b and b+1 (static_assert below), so a round
      // writes over stages its own round or earlier rounds have read, and one
      // barrier per round (operands loaded by every wavefront) is enough.
      static_assert(BW == BH && (BW == 32 || BW == 48 || BW == 64), "matrix-core DFT: 32x32, 48x48 or 64x64 blocks");
      static_assert(LSPEC >= LA && 2 * LA - LSPEC >= (BPW - 1) * (LSPEC - LA), "spectra overlap stages b, b+1 only");
      constexpr int NW = NT / 64, MB = (BPW + NW - 1) / NW;
      const int wave = wave_of(t), lane = t & 63;
      const DftTile* T = static_cast<const DftTile*>(J.dft_tab);
      const float sx = J.dft_sx;
#pragma unroll 1
      for (int q = 0; q < MB; q++) {
        // (a wavefront past the tile's blocks loads block 0's place and does
        // not use it: operands loaded under a branch would keep their old
        // values alive around the loops)
        const int b = nblk - 1 - (q * NW + wave), bl = max(b, 0);  // uniform in the wavefront
        const DftIn<BW> din = dft_fwd_load<BW>(
            [&](int r, int c) {
              return reinterpret_cast<const float*>(stage)[2 * (bl * LA + (r >> 1) * SA + c) + (r & 1)];
            },
            sx, lane);
        __syncthreads();  // the round's stages read
        if (b >= 0)
          dft_fwd_compute<BW, true>(din, sx, T, lane, [&](int r, int k, float2 zz) { spec[b * LSPEC + r * SR + k] = zz; });
      }
    } else if (!row_wave) {
      __syncthreads();  // gather stage dead; spectral layout from here
    } else {
      // ---- 2. row r2c, a lane pair per two real rows packed as one complex
      // row (samples halved by the window): its BW-point transform Z split
      // over the pair, then the rows' spectra (Z[k] + conj Z[BW-k]) and
      // (Z[k] - conj Z[BW-k]) / i.  With Q = BW/4, lane 0 holds Z[i] and
      // Z[2Q + i], lane 1 Z[Q + i] and Z[3Q + i] (P[i] and R[i]); two values
      // i = j, j + Q/2 of both are swapped so that lane 0 has all four of j
      // and lane 1 all four of j + Q/2, each the columns i and Q + i.
      constexpr int HW = BW / 2, Q = BW / 4;
      float2 z[HW];
      static_for<0, HW>([&](auto j) { z[j] = stage[rb * LA + rp * SA + 2 * decltype(j)::value + hh]; });
      __syncthreads();  // gather stage dead; spectral layout from here
      fft<HW, -1>(z);
      split_combine_fwd<BW>(z, hh);
      float2* row = spec + rb * LSPEC + 2 * rp * SR;
      auto put = [&](float2* d, float2 a, float2 b) {  // columns from Z[k] and Z[BW - k]
        d[0] = make_float2(a.x + b.x, a.y - b.y);
        d[SR] = make_float2(a.y + b.y, b.x - a.x);
      };
      // (every lane exchanges; lanes without a row pair of the tile store nothing)
      static_for<1, Q / 2>([&](auto jj) {
        constexpr int j = decltype(jj)::value;
        half_swap(z[j], z[j + Q / 2]);              // lane 0: P[j] of both lanes; lane 1: P[j + Q/2] of both
        half_swap(z[HW - j], z[HW - j - Q / 2]);    // ... R[Q - j], R[Q - j - Q/2]
      });
      const float2 other = half_other(z[Q + Q / 2], hh);
      if (row_on) {
        static_for<1, Q / 2>([&](auto jj) {
          constexpr int j = decltype(jj)::value;
          float2* d = row + hh * (Q / 2) + j;
          put(d, z[j], z[HW - j - Q / 2]);
          put(d + Q, z[j + Q / 2], z[HW - j]);
        });
        put(row + Q / 2 + hh * Q, z[Q / 2], other);       // i = Q/2: P[i] with the other lane's R[Q - i]
        put(row + hh * Q, z[0], hh ? z[Q] : z[0]);        // column 0 / Q
        if (hh == 0) put(row + HW, z[Q], z[Q]);           // column BW/2
      }
    }
    __syncthreads();

    // row (past hh * CR/2) of the lane's value j in the spectrum ...
    auto col_row = [](auto j) { return decltype(j)::value + (decltype(j)::value >= CR / 2 ? CR / 2 : 0); };
    // ... and the LDS row it is read from and goes back to: that row, or (FFT
    // form) the transforms' inputs and outputs, even rows on lane 0, odd on lane 1
    auto lds_row = [=](auto j) {
      return MF ? hh * (CR / 2) + decltype(j)::value + (decltype(j)::value >= CR / 2 ? CR / 2 : 0)
                : 2 * decltype(j)::value + hh;
    };
    if constexpr (MODE == MODE_FWD) {
      // ---- 3. forward column transforms to the ring, then the next frame
      float2 fc[CR];
      static_for<0, CR>([&](auto j) { fc[j] = spec[cb * LSPEC + lds_row(j) * SR + cc]; });
      __syncthreads();  // spectra read: the next frame's gather may write the stage
      if constexpr (!MF) {
        fft<CR, -1>(fc);
        split_combine_fwd<BH>(fc, hh);
      }
      if (col_on) {
        float2* out = L.ring + (size_t)(m % BT) * L.spec_elems + colo;
        static_for<0, CR>([&](auto i) { out[col_row(i) * COLS] = fc[i]; });
      }
      continue;
    }
    // ---- 3. column lanes: chunk 0 in flight during the forward column FFT
    const float2* rq[NQ > 0 ? NQ : 1];
    static_for<0, NQ>([&](auto qq) {
      constexpr int q = decltype(qq)::value;
      rq[q] = L.ring + (size_t)((m + FROM + q) % BT) * L.spec_elems;
    });
    auto load_ring = [&](auto kc, RBuf& b) {
      constexpr int k = decltype(kc)::value;
      static_for<0, CH>([&](auto uu) {
        constexpr int u = decltype(uu)::value, i = k * CH + u;
        const size_t o = colo + (size_t)col_row(std::integral_constant<int, i>{}) * COLS;
        static_for<0, NQ>([&](auto qq) { b.v[decltype(qq)::value][u] = rq[decltype(qq)::value][o]; });
        if constexpr (MODE == MODE_KALMAN && !RES) b.ks[u] = KalState{J.kal_last[o], J.kal_sum[o]};
      });
    };
    const int tab0 = hh * (CR / 2) * COLS + cc;  // table element of the lane's first row
    auto load_tab = [&](auto kc, TBuf& b) {
      constexpr int k = decltype(kc)::value;
      static_for<0, CH>([&](auto uu) {
        constexpr int u = decltype(uu)::value, i = k * CH + u;
        const int kk = col_row(std::integral_constant<int, i>{}) * COLS + tab0;
        b.g[u] = J.grid[kk];
        if constexpr (SHP != SHP_NONE) b.wsh[u] = J.wsharpen[kk];
        if constexpr (SHP == SHP_GENERAL) b.wdh[u] = J.wdehalo[kk];
      });
      if (pat) {
        static_for<0, CH>([&](auto uu) {
          constexpr int i = k * CH + decltype(uu)::value;
          b.sig[decltype(uu)::value] = pat[col_row(std::integral_constant<int, i>{}) * COLS + cc];
        });
      } else {
        static_for<0, CH>([&](auto uu) { b.sig[decltype(uu)::value] = J.sigma2; });
      }
    };
    auto tab = [&](const TBuf& b, auto uu) {
      constexpr int u = decltype(uu)::value;
      Tab T;
      T.g = b.g[u];
      T.sig = b.sig[u];
      T.wsh = 0.0f;
      T.wdh = 0.0f;
      if constexpr (SHP != SHP_NONE) T.wsh = b.wsh[u];
      if constexpr (SHP == SHP_GENERAL) T.wdh = b.wdh[u];
      return T;
    };
    RBuf rbuf[DR + 1];
    TBuf tbuf[2];
    float2 col[CR];
    static_for<0, (DR < NCH ? DR : NCH)>([&](auto kc) { load_ring(kc, rbuf[decltype(kc)::value]); });
    load_tab(std::integral_constant<int, 0>{}, tbuf[0]);
    static_for<0, CR>([&](auto j) { col[j] = spec[cb * LSPEC + lds_row(j) * SR + cc]; });
    if constexpr (!MF) {
      fft<CR, -1>(col);
      split_combine_fwd<BH>(col, hh);
    }
    if constexpr (MODE == MODE_W3D) {
      if (col_on) {
        float2* out = L.ring + (size_t)((m + TO) % BT) * L.spec_elems + colo;
        static_for<0, CR>([&](auto i) { out[col_row(i) * COLS] = col[i]; });
      }
    }
    // ---- 4a. per-block degrid fractions from the input DC and from the
    // filtered DC (code_impl_C.h:64); lane 0 of each block computes both
    if (col_on && cc == 0 && hh == 0) {
      const Tab T0 = tab(tbuf[0], std::integral_constant<int, 0>{});
      float gf = 0.0f, dcf;
      if constexpr (MODE == MODE_W3D) {
        float2 w[5];
#pragma unroll
        for (int q = 0; q < 5; q++) w[q] = make_float2(0.0f, 0.0f);
        static_for<0, NQ>([&](auto qq) { w[decltype(qq)::value] = rbuf[0].v[decltype(qq)::value][0]; });
        w[NQ] = col[0];
        gf = J.use_degrid ? J.degrid * w[BT / 2].x / grid0 : 0.0f;
        dcf = apply3d_elem<BT>(SP, w, T0, gf).x;
      } else if constexpr (MODE == MODE_W2D) {
        gf = J.use_degrid ? J.degrid * col[0].x / grid0 : 0.0f;
        dcf = apply2d_s<SHP>(SP, col[0], T0, gf).x;
      } else if constexpr (MODE == MODE_KALMAN) {
        KalState st;
        if constexpr (RES) st = kst[0];
        else st = rbuf[0].ks[0];
        dcf = kalman_elem(SP, col[0], T0, st).x;
      } else {
        dcf = col[0].x;
      }
      s_gf[cb] = gf;
      s_gfs[cb] = J.use_degrid ? J.degrid * dcf / grid0 : 0.0f;
    }
    __syncthreads();
    // ---- 4b. spectral pass down the column, chunk k+1 loading under chunk k
    {
      const float gf = s_gf[cb], gfs = s_gfs[cb];
      static_for<0, NCH>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if constexpr (k + DR < NCH) load_ring(std::integral_constant<int, k + DR>{}, rbuf[(k + DR) % (DR + 1)]);
        if constexpr (k + 1 < NCH) load_tab(std::integral_constant<int, k + 1>{}, tbuf[(k + 1) & 1]);
        const RBuf& b = rbuf[k % (DR + 1)];
        const TBuf& tb = tbuf[k & 1];
        static_for<0, CH>([&](auto uu) {
          constexpr int u = decltype(uu)::value, i = k * CH + u;
          const Tab T = tab(tb, uu);
          float2 r;
          if constexpr (MODE == MODE_W3D) {
            float2 w[5];
#pragma unroll
            for (int q = 0; q < 5; q++) w[q] = make_float2(0.0f, 0.0f);
            static_for<0, NQ>([&](auto qq) { w[decltype(qq)::value] = b.v[decltype(qq)::value][u]; });
            w[NQ] = col[i];
            r = apply3d_elem<BT>(SP, w, T, gf);
            if constexpr (SHP != SHP_NONE) r = sharpen_s<SHP>(SP, r, T, gfs);
          } else if constexpr (MODE == MODE_W2D) {
            r = apply2d_s<SHP>(SP, col[i], T, gf);
            if constexpr (SHP != SHP_NONE) {
              const float2 rs = sharpen_s<SHP>(SP, r, T, gfs);
              r = SP.use_pattern ? rs : r;
            }
          } else if constexpr (MODE == MODE_KALMAN) {
            KalState st;
            if constexpr (RES) st = kst[i];
            else st = b.ks[u];
            r = kalman_elem(SP, col[i], T, st);
            if constexpr (RES) {
              kst[i] = st;
            } else if (col_on) {
              const size_t o = colo + (size_t)col_row(std::integral_constant<int, i>{}) * COLS;
              J.kal_last[o] = st.last;
              J.kal_sum[o] = st.sum;
            }
            if constexpr (SHP != SHP_NONE) r = sharpen_s<SHP>(SP, r, T, gfs);
          } else {
            r = sharpen_s<SHP>(SP, col[i], T, gfs);
          }
          col[i] = r;
        });
        // chunk k's results are pinned here (an empty asm that clobbers
        // memory): the compiler neither sinks the gains below the later
        // chunks' loads nor hoists those loads above them, so at most two
        // chunks of loads are in registers at once
        static_for<0, CH>([&](auto uu) {
          float2& cv = col[k * CH + decltype(uu)::value];
          float a = cv.x, b = cv.y;
          asm volatile("" : "+v"(a), "+v"(b) : : "memory");
          cv.x = a;
          cv.y = b;
        });
      });
    }
    // ---- 5. column inverse FFT, back to LDS for the row c2r
    if constexpr (!MF) {
      split_combine_inv<BH>(col, hh);
      fft<CR, +1>(col);
    }
    if (col_on) {
      static_for<0, CR>([&](auto j) { spec[cb * LSPEC + lds_row(j) * SR + cc] = col[j]; });
    }
    __syncthreads();
    if constexpr (MF) {
      // ---- 5-6. 2D c2r on the matrix cores (DC and Nyquist imaginary parts
      // dropped by the tables), in rounds of one block per wavefront, lowest
      // blocks first: synthesised block b overlaps only the spectra of blocks
      // b-1 and b (static_assert below)
      static_assert(LSYN <= 2 * LSPEC && 2 * LSPEC - LSYN <= 2 * LSPEC / (BPW > 1 ? BPW - 1 : 1),
                    "synthesised rows overlap spectra b-1, b only");
      constexpr int NW = NT / 64, MB = (BPW + NW - 1) / NW;
      const int wave = wave_of(t), lane = t & 63;
      const DftTile* T = static_cast<const DftTile*>(J.dft_tab);
      const float sz = J.dft_sz;
#pragma unroll 1
      for (int q = 0; q < MB; q++) {
        const int b = q * NW + wave, bl = min(b, nblk - 1);  // uniform in the wavefront
        const DftSpec<BW> dsp = dft_inv_load<BW>([&](int r, int k) { return spec[bl * LSPEC + r * SR + k]; }, sz, lane);
        __syncthreads();  // the round's spectra read
        if (b < nblk)
          dft_inv_compute<BW, true>(dsp, sz, T, lane, [&](int r, int c0, f4 x) {
            float* d = syn + b * LSYN + r * SYNW + c0;
            d[0] = x[0];
            d[1] = x[1];
            d[2] = x[2];
            d[3] = x[3];
          });
      }
    } else if (!row_wave) {
      __syncthreads();  // spectral layout dead; synthesised rows next
    } else {
      // ---- 6. row c2r, a lane pair per two rows: lane h builds Z[k] and
      // Z[k + BW/2], k = h BW/4 + i, of the packed spectrum from columns k and
      // BW/2 - k of both rows (DC and Nyquist imaginary parts dropped) and the
      // pair reduces them to its half-length inverse transforms' inputs; lane
      // h ends with output columns 2j + h.
      constexpr int HW = BW / 2, Q = BW / 4;
      const float2* lo = spec + rb * LSPEC + 2 * rp * SR + hh * Q;         // column k = lo[i]
      const float2* hi = spec + rb * LSPEC + 2 * rp * SR + HW - hh * Q;    // column BW/2 - k = hi[-i]
      float2 z[HW];
      static_for<0, Q>([&](auto ii) {
        constexpr int i = decltype(ii)::value;
        float2 a = lo[i], b = lo[SR + i], c = hi[-i], d = hi[SR - i];
        if constexpr (i == 0) {  // lane 0: columns 0 and BW/2
          a.y = hh ? a.y : 0.0f;
          b.y = hh ? b.y : 0.0f;
          c.y = hh ? c.y : 0.0f;
          d.y = hh ? d.y : 0.0f;
        }
        z[i] = make_float2(a.x - b.y, a.y + b.x);
        z[Q + i] = make_float2(c.x + d.y, d.x - c.y);
      });
      split_combine_inv<BW>(z, hh);
      __syncthreads();  // spectral layout dead; synthesised rows next
      fft<HW, +1>(z);
      if (row_on) {
        float* d0 = syn + rb * LSYN + 2 * rp * SYNW + hh;
        static_for<0, HW>([&](auto j) {
          d0[2 * decltype(j)::value] = z[j].x;
          d0[SYNW + 2 * decltype(j)::value] = z[j].y;
        });
      }
    }
    __syncthreads();
    if constexpr (AHEAD) {
      // (after the last frame nothing: an undefined value would stay alive)
      if (fi + 1 < i1) gather_load<BW, BH>(J, raw, L.src[fi + 1], ro, bx0, nblk, stepx, t);
      else static_for<0, BH>([&](auto i) { raw[i] = 0; });
    }
    // ---- 7. overlap-add inside the tile; seam partials to this frame's seam buffer
    uint8_t* dst = L.dst[fi];
    float* seam = J.seam + (size_t)fi * 4 * (size_t)J.seam_plane;
    const float* ws = wsyn + zo;
    const int2* rd = rowdst + zo;
    if (J.pix == 1) overlap_cols<1, BW, BH, BPW, LSYN, SYNW, RES ? 2 : 4>(J, dst, seam, syn, ws, rd, by, bx0, nblk, RW, stepx, stepy, t);
    else if (J.pix == 2) overlap_cols<2, BW, BH, BPW, LSYN, SYNW, RES ? 2 : 4>(J, dst, seam, syn, ws, rd, by, bx0, nblk, RW, stepx, stepy, t);
    else overlap_cols<4, BW, BH, BPW, LSYN, SYNW, RES ? 2 : 4>(J, dst, seam, syn, ws, rd, by, bx0, nblk, RW, stepx, stepy, t);
    __syncthreads();  // syn read; the next frame's gather writes the stage
  }
  if constexpr (RES) {
    const int t = threadIdx.x, cl = (t >> 6) * 32 + (t & 31);
    if (cl / COLS < nblk)
      static_for<0, CR>([&](auto i) {
        L0.J.kal_last[state_at(i)] = kst[i].last;
        L0.J.kal_sum[state_at(i)] = kst[i].sum;
      });
  }
}

// One finished sample (src/buffer.cpp:406: store_px's rounding and clamping)
// of an integer format.
__device__ __forceinline__ unsigned seam_int(float v, int maxval) {
  int q = (int)v;
  q = q < 0 ? 0 : q;
  return (unsigned)(q > maxval ? maxval : q);
}

// Four consecutive floats at any float's address (one 16-byte load).
struct __attribute__((packed, aligned(4))) FloatQuad {
  float x, y, z, w;
};

// Seam pixels of every frame of a k_run launch, finished from the partial
// sums in the reference's float order (src/buffer.cpp:445-477); two wavefronts
// per output row and frame, two rows a workgroup.  Rows inside a horizontal
// band finish the whole row, four pixels a lane (16-byte loads of each
// partial, one store), SU such groups of each lane in flight, the corner
// partials where a vertical seam crosses; a row's last group may repeat pixels
// of the one before (the same values).  Other rows finish only the columns of
// the vertical seams between tiles.  Memory-bound: 8 bytes in and a sample out
// per band pixel, 4 TB/s on UHD planes.  With a workgroup per row, eight
// single pixels of each lane in flight whatever the row's width, narrow planes
// issued mostly repeated loads: 720x576 4:2:2, 13 frames 27.7 us, now 17.5.
constexpr int SEAM_ROWS = 2, SEAM_LANES = 128;
template <int BW, int BH, int BPW>
__global__ void __launch_bounds__(SEAM_LANES * SEAM_ROWS) k_seam_run(RunBatch B_arg) {
  const RunLaunch& L = kernarg_batch(B_arg).job[blockIdx.z];
  const PlaneJob& J = L.J;
  const int yo = blockIdx.x * SEAM_ROWS + wave_of(threadIdx.x) / (SEAM_LANES / 64);  // uniform in the wavefront
  const int fi = blockIdx.y, lane = threadIdx.x & (SEAM_LANES - 1);
  if (yo >= J.Hc || fi >= L.nframes) return;
  const float* sm = J.seam + (size_t)fi * 4 * (size_t)J.seam_plane;
  uint8_t* dst = L.dst[fi];
  const int stepx = BW - J.ow, stepy = BH - J.oh;
  int ry = yo;
  if (J.interlaced) ry = (yo & 1) == 0 ? (yo >> 1) : (J.Hc >> 1) + ((J.Hc - 1 - yo) >> 1);
  const int cy = ry + J.mirh, r = cy / stepy, i = cy - r * stepy;
  const int pix = J.pix, maxval = J.maxval, Wc = J.Wc, mirw = J.mirw, ow = J.ow;
  const float rounder = pix == 4 ? 0.0f : 0.5f;
  const float fbase = (float)J.obase;
  const size_t P = (size_t)J.seam_plane;
  const float* row = sm + (size_t)yo * Wc;
  const float inv = 1.0f / (float)stepx;
  constexpr int SU = 4;
  if (i < J.oh && r >= 1) {
    const float wyr = J.wsynyr[i] * J.norm, wyl = J.wsynyl[i] * J.norm;
    auto finish = [&](bool cor, float A, float B, float C, float D) {
      return cor ? (A + B) * wyr + (C + D) * wyl + rounder + fbase : A + B + rounder + fbase;
    };
    const int n4 = (Wc + 3) >> 2;  // (planes are at least five pixels wide: half a block's reflection fits)
    uint8_t* out = dst + (long long)(yo + J.tc) * J.dst_pitch + (long long)J.lc * pix;
    for (int g0 = 0; g0 < n4; g0 += SEAM_LANES * SU) {
      FloatQuad up[SU], lo[SU], cA[SU], cB[SU];
      int own[SU], next[SU];  // pixels of the group in a corner: from its first block, from the next one
#pragma unroll
      for (int u = 0; u < SU; u++) {
        if (g0 + SEAM_LANES * u >= n4) break;  // (uniform)
        const int x = min(4 * (g0 + SEAM_LANES * u + lane), Wc - 4);
        const int cx = x + mirw, c = div_small(cx, stepx, inv), j = cx - c * stepx, m = c % BPW;
        up[u] = *reinterpret_cast<const FloatQuad*>(row + x);
        lo[u] = *reinterpret_cast<const FloatQuad*>(row + P + x);
        // columns j, j + 1, ... of block column c (a seam's if c is a tile's
        // first), then columns 0, 1, ... of the next (stepx >= 4)
        own[u] = m == 0 && c >= 1 ? min(max(ow - j, 0), 4) : 0;
        next[u] = m == BPW - 1 ? min(max(j + 4 - stepx, 0), ow) : 0;
        if (own[u] + next[u] > 0) {
          cA[u] = *reinterpret_cast<const FloatQuad*>(row + 2 * P + x);
          cB[u] = *reinterpret_cast<const FloatQuad*>(row + 3 * P + x);
        } else {
          cA[u] = cB[u] = FloatQuad{0.0f, 0.0f, 0.0f, 0.0f};
        }
        if (next[u] > 0) own[u] = stepx - j;  // first pixel of the next block
      }
#pragma unroll
      for (int u = 0; u < SU; u++) {
        if (g0 + SEAM_LANES * u >= n4) break;
        const int g = g0 + SEAM_LANES * u + lane;
        if (g >= n4) continue;
        auto cor = [&](int e) { return next[u] > 0 ? e >= own[u] && e < own[u] + next[u] : e < own[u]; };
        const float v0 = finish(cor(0), up[u].x, lo[u].x, cA[u].x, cB[u].x);
        const float v1 = finish(cor(1), up[u].y, lo[u].y, cA[u].y, cB[u].y);
        const float v2 = finish(cor(2), up[u].z, lo[u].z, cA[u].z, cB[u].z);
        const float v3 = finish(cor(3), up[u].w, lo[u].w, cA[u].w, cB[u].w);
        uint8_t* o = out + (size_t)min(4 * g, Wc - 4) * pix;
        if (pix == 1) {
          const unsigned q = seam_int(v0, maxval) | seam_int(v1, maxval) << 8 | seam_int(v2, maxval) << 16 |
                             seam_int(v3, maxval) << 24;
          __builtin_memcpy(o, &q, 4);  // (any alignment)
        } else if (pix == 2) {
          const uint2 q = make_uint2(seam_int(v0, maxval) | seam_int(v1, maxval) << 16,
                                     seam_int(v2, maxval) | seam_int(v3, maxval) << 16);
          __builtin_memcpy(o, &q, 8);
        } else {
          auto unit = [](float v) {
            const float f = v < 0.0f ? 0.0f : v;
            return f > 1.0f ? 1.0f : f;
          };
          const float4 q = make_float4(unit(v0), unit(v1), unit(v2), unit(v3));
          __builtin_memcpy(o, &q, 16);
        }
      }
    }
  } else {
    const int nseam = (J.nox - 1) / BPW;  // tile boundaries at block columns BPW, 2*BPW, ...
    const float inv_ow = 1.0f / (float)max(ow, 1);
    for (int k = lane; k < nseam * ow; k += SEAM_LANES) {
      const int q = div_small(k, ow, inv_ow);
      const int x = (q + 1) * BPW * stepx + (k - q * ow) - mirw;
      if (x >= 0 && x < Wc) {
        const float v = (row[x] + row[P + x]) * J.norm + rounder + fbase;
        store_px(J, dst, yo, x, v);
      }
    }
  }
}

template <int BW, int BH, bool MF>
hipError_t launch_run_modes(int mode, int bt, int shp, const RunBatch& L, hipStream_t s) {
  constexpr int NT = 256;
  dim3 grid(L.total_wg), block(NT);
#define NF3D_RUN(M, B, H) hipLaunchKernelGGL((k_run<BW, BH, NT, M, B, H, MF>), grid, block, 0, s, L)
#define NF3D_RUN_RES(H) \
  hipLaunchKernelGGL((k_run<BW, BH, NT, MODE_KALMAN, 0, H, false, true>), grid, block, 0, s, L)
#define NF3D_RUN_SHP(M, B)                                   \
  switch (shp) {                                             \
    case SHP_NONE: NF3D_RUN(M, B, SHP_NONE); break;          \
    case SHP_SHARPEN: NF3D_RUN(M, B, SHP_SHARPEN); break;    \
    case SHP_GENERAL: NF3D_RUN(M, B, SHP_GENERAL); break;    \
    default: return hipErrorInvalidValue;                    \
  }
  switch (mode) {
    case MODE_FWD:
      switch (bt) {
        case 2: NF3D_RUN(MODE_FWD, 2, SHP_NONE); break;
        case 3: NF3D_RUN(MODE_FWD, 3, SHP_NONE); break;
        case 4: NF3D_RUN(MODE_FWD, 4, SHP_NONE); break;
        case 5: NF3D_RUN(MODE_FWD, 5, SHP_NONE); break;
        default: return hipErrorInvalidValue;
      }
      break;
    case MODE_W2D: NF3D_RUN_SHP(MODE_W2D, 0); break;
    case MODE_KALMAN:
      // the state stays in registers where a launch has the frames to make up
      // for loading it all at once at the start (one frame: 32x32 177 -> 184
      // us) and, at 48x48, for two instead of three wavefronts a SIMD (one
      // frame: 193 -> 213 us)
      if constexpr (!MF && BH <= 48) {
        if (L.max_frames >= (BH <= 32 ? 2 : 4)) {
          switch (shp) {
            case SHP_NONE: NF3D_RUN_RES(SHP_NONE); break;
            case SHP_SHARPEN: NF3D_RUN_RES(SHP_SHARPEN); break;
            case SHP_GENERAL: NF3D_RUN_RES(SHP_GENERAL); break;
            default: return hipErrorInvalidValue;
          }
          break;
        }
      }
      NF3D_RUN_SHP(MODE_KALMAN, 0);
      break;
    case MODE_SHARPEN:
      if (shp == SHP_SHARPEN) NF3D_RUN(MODE_SHARPEN, 0, SHP_SHARPEN);
      else if (shp == SHP_GENERAL) NF3D_RUN(MODE_SHARPEN, 0, SHP_GENERAL);
      else return hipErrorInvalidValue;
      break;
    case MODE_W3D:
      switch (bt) {
        case 2: NF3D_RUN_SHP(MODE_W3D, 2); break;
        case 3: NF3D_RUN_SHP(MODE_W3D, 3); break;
        case 4: NF3D_RUN_SHP(MODE_W3D, 4); break;
        case 5: NF3D_RUN_SHP(MODE_W3D, 5); break;
        default: return hipErrorInvalidValue;
      }
      break;
    default: return hipErrorInvalidValue;
  }
#undef NF3D_RUN_SHP
#undef NF3D_RUN_RES
#undef NF3D_RUN
  return hipGetLastError();
}

// mf: the matrix-core DFT form (32x32, 48x48 and 64x64 blocks).
template <int BW, int BH>
hipError_t launch_run_shape(int mode, int bt, int shp, int mf, const RunBatch& L, hipStream_t s) {
  if (L.njobs < 1 || L.njobs > RUN_MAX_JOBS) return hipErrorInvalidValue;
  int wg = 0;
  for (int k = 0; k < L.njobs; k++) {
    const RunLaunch& R = L.job[k];
    if (R.nframes < 1 || R.nframes > RUN_MAX_FRAMES || R.fpw < 1 || R.wg_begin != wg) return hipErrorInvalidValue;
    if (mf && !R.J.dft_tab) return hipErrorInvalidValue;
    wg += R.ntiles * ((R.nframes + R.fpw - 1) / R.fpw);
  }
  if (wg != L.total_wg) return hipErrorInvalidValue;
  if (mf) {
    if constexpr (BW == BH && (BW == 32 || BW == 48 || BW == 64)) return launch_run_modes<BW, BH, true>(mode, bt, shp, L, s);
    else return hipErrorInvalidValue;
  }
  return launch_run_modes<BW, BH, false>(mode, bt, shp, L, s);
}

template <int BW, int BH>
hipError_t launch_seam_run_shape(int mf, const RunBatch& L, hipStream_t s) {
  if (L.njobs < 1 || L.njobs > RUN_MAX_JOBS || L.max_frames < 1 || L.max_frames > RUN_MAX_FRAMES) return hipErrorInvalidValue;
  dim3 sgrid((L.max_hc + SEAM_ROWS - 1) / SEAM_ROWS, L.max_frames, L.njobs);
  constexpr int BPW = RunShape<BW, BH, false>::BPW, BPW_MF = RunShape<BW, BH, true>::BPW;
  if constexpr (BPW_MF != BPW) {
    if (mf) {
      hipLaunchKernelGGL((k_seam_run<BW, BH, BPW_MF>), sgrid, dim3(256), 0, s, L);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((k_seam_run<BW, BH, BPW>), sgrid, dim3(256), 0, s, L);
  return hipGetLastError();
}

}  // namespace nf3d
