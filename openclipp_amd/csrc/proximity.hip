// proximity.hip -- direct (VALU) template matching for every type and channel count.
//
// Semantics (reference cl-files/ImageProximity.cl:44-466):
//   D(x,y) = sum_{v<th} sum_{u<tw} g(s(x+u-tw/2, y+v-th/2), t(u,v)),  s = 0 outside the image,
//   g = (s-t)^2 (SqrDistance), |s-t| (AbsDistance), s*t (CrossCorr);
//   the Norm ops divide by sqrt(sum s^2 * sum t^2) over the same zero-padded window.
//
// Kernels:
//   prox_tile_f32  REAL = float sources (F32, U32, S32).  Each workgroup owns a 64-row x
//                  (4*R)-column output tile; the source tile plus halo is staged in LDS
//                  (zero padded, converted to float), one band of template rows at a time.
//                  A thread owns R horizontally adjacent outputs of one row (lanes = rows,
//                  waves = column groups), keeps a sliding window of R+U-1 source values in
//                  registers and takes template values as wave-uniform scalar loads, so every
//                  LDS float feeds up to U FMAs and every template float R FMAs.  Each output
//                  accumulates in the reference order (template row outer, column inner) with
//                  one fused multiply-add per tap, which is the reference's order under
//                  OpenCL's default FP contraction.
//   prox_sad8      AbsDistance of 8-bit sources: the same tiling on dwords of four bytes.
//   prox_tile_int  8- and 16-bit integer sources (what neither prox_sad8 nor the int8 matrix cores
//                  of mfma_i8.hip take): the same tiling with exact integer sums (int32 where the
//                  bound allows, int64 otherwise), rounded once to float.
//   prox_direct    one output per thread, reference order, any type (F64 sources and
//                  templates too wide for the LDS tile).
// Norm denominators: FP64 window sums of squares, of F32 sources from the staged tile where it holds them
// (prox_norm_from_tile), else from the sum-of-squares integral of the source (exclusive, (W+1) x (H+1)
// layout) by four corners; and the FP64 sum of squares of the template.
#include <algorithm>

#include "device_common.h"

namespace ocip {

namespace {

constexpr int kTileRows = 64;      // output rows per workgroup (one per lane)
constexpr int kWaves = 4;          // waves per workgroup, side by side in x
constexpr int kTileStatic = 32;    // the float tile kernels' static LDS (tile_f32's sums of t^2)
constexpr int kLdsBudget = 64 * 1024 - kTileStatic;   // dynamic LDS that needs no attribute

// ------------------------------------------------------------------------- template staging
// The staged template and its sums, by one workgroup (the sums have one fixed order and no
// second launch).  Bound by memory latency: up to kPrepWide threads, K elements per thread in
// flight (one for templates of that many elements or fewer, which start sooner), (row, column)
// stepped along with the element index instead of divided out.  64x64: 9.0 -> 5.0 us, 256x256:
// 122 -> 35 us against 256 threads with one element in flight.
constexpr int kPrepWide = 1024;

template <int TYPE, int KIND, int K>
__global__ __launch_bounds__(kPrepWide) void template_prep(const char *tpl, int tw, int th,
                                                           int tstep, int nch, int ch, int pitch,
                                                           void *out, double *sums,
                                                           unsigned *peak)
{
   __shared__ double red[2][kPrepWide / 64];
   __shared__ unsigned redp[kPrepWide / 64];
   double s2 = 0, s1 = 0;
   unsigned top = 0;
   const int n = pitch * th, B = blockDim.x;
   const int dv = B / pitch, du = B - dv * pitch;
   int v = threadIdx.x / pitch, u = threadIdx.x - v * pitch;
   for (int i0 = threadIdx.x; i0 < n; i0 += K * B) {
      double val[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
         val[k] = i0 + k * B < n && u < tw ? (double)ld<TYPE>(tpl + (size_t)v * tstep, u * nch + ch)
                                           : 0.0;
         u += du;
         v += dv;
         if (u >= pitch) {
            u -= pitch;
            ++v;
         }
      }
#pragma unroll
      for (int k = 0; k < K; ++k) {
         const int i = i0 + k * B;
         if (i < n) {
            if (KIND == 0) static_cast<float *>(out)[i] = (float)val[k];
            else if (KIND == 1) static_cast<double *>(out)[i] = val[k];
            else static_cast<int32_t *>(out)[i] = (int32_t)val[k];
         }
         const double q = val[k] * val[k];
         s2 += q;
         s1 += val[k];
         top = max(top, (unsigned)__double2hiint(q) & 0x7fffffffu);
      }
   }
   s2 = wave_sum(s2);
   s1 = wave_sum(s1);
   const int wave = threadIdx.x >> 6, waves = B >> 6;
   if (peak) {
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) top = max(top, (unsigned)__shfl_xor((int)top, d, 64));
   }
   if ((threadIdx.x & 63) == 0) { red[0][wave] = s2; red[1][wave] = s1; redp[wave] = top; }
   __syncthreads();
   if (threadIdx.x < 2) {
      double t = red[threadIdx.x][0];
      for (int w = 1; w < waves; ++w) t += red[threadIdx.x][w];
      sums[threadIdx.x] = t;
   }
   if (threadIdx.x == 2 && peak) {
      for (int w = 0; w < waves; ++w) top = max(top, redp[w]);
      *peak = top;
   }
}


// ------------------------------------------------------------------------- per-tap maths
template <int OP> __device__ __forceinline__ float tap(float acc, float s, float t)
{
   if (OP == kSSD || OP == kSSDNorm) { float d = s - t; return __builtin_fmaf(d, d, acc); }
   if (OP == kSAD) return acc + __builtin_fabsf(s - t);
   return __builtin_fmaf(s, t, acc);
}

// U template columns starting at LDS column `col` (row pointer `lrow`) for R outputs.
// ALIGNED: col - SHIFT is a multiple of 4 floats, so the window is read with 16-byte LDS
// loads from there (SHIFT values before col read and not used).
template <int OP, int R, int U, bool ALIGNED, int SHIFT = 0>
__device__ __forceinline__ void chunk_f32(float (&acc)[R], const float *lrow, int col,
                                          const float *__restrict__ trow)
{
   constexpr int N = R + U - 1;
   float s[(N + SHIFT + 3) / 4 * 4];
   if (ALIGNED) {
#pragma unroll
      for (int i = 0; i < (N + SHIFT + 3) / 4; ++i) {
         float4 q = *reinterpret_cast<const float4 *>(lrow + col - SHIFT + 4 * i);
         s[4 * i] = q.x; s[4 * i + 1] = q.y; s[4 * i + 2] = q.z; s[4 * i + 3] = q.w;
      }
   } else {
#pragma unroll
      for (int i = 0; i < N; ++i) s[i + SHIFT] = lrow[col + i];
   }
   float t[U];
#pragma unroll
   for (int k = 0; k < U; ++k) t[k] = trow[k];
#pragma unroll
   for (int k = 0; k < U; ++k)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] = tap<OP>(acc[r], s[r + k + SHIFT], t[k]);
}

template <int TYPE>
__device__ __forceinline__ void stage_tile_f32(float *lds, int ldsw, int nrows, int ncols,
                                               const char *src, int W, int H, int sstep,
                                               int nch, int ch, int sx0, int sy0)
{
   // eight elements per thread in flight; element i = r ldsw + c, (r, c) stepped along with i
   // (256 elements a step) instead of divided out for each element
   const int n = nrows * ldsw;
   const int dq = 256 / ldsw, dr = 256 - dq * ldsw;
   int r = threadIdx.x / ldsw, c = threadIdx.x - r * ldsw;
   for (int i0 = threadIdx.x; i0 < n; i0 += 256 * 8) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
         const int i = i0 + 256 * k;
         const int sx = sx0 + c, sy = sy0 + r;
         v[k] = (i < n && c < ncols && sx >= 0 && sx < W && sy >= 0 && sy < H)
                    ? (float)ld<TYPE>(src + (size_t)sy * sstep, sx * nch + ch) : 0.f;
         c += dr;
         r += dq;
         if (c >= ldsw) {
            c -= ldsw;
            ++r;
         }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k)
         if (i0 + 256 * k < n) lds[i0 + 256 * k] = v[k];
   }
}

// stage_tile_f32 for 1-channel F32 images: groups of four columns, one 16-byte load each (at any
// alignment) where the group lies wholly inside the image, eight groups per thread in flight;
// the same values in the columns that the taps read (up to ncols + 2).
__device__ __forceinline__ void stage_tile_f32_v4(float *lds, int ldsw, int nrows, int ncols,
                                                  const char *src, int W, int H, int sstep,
                                                  int sx0, int sy0)
{
   const int gpr = (ncols + 6) / 4, n4 = nrows * gpr;   // columns 0 .. ncols + 2, within the pitch
   // group i = r gpr + g, (r, g) stepped along with i (256 groups a step) instead of divided out
   const int dq = 256 / gpr, dr = 256 - dq * gpr;
   int r = threadIdx.x / gpr, g = threadIdx.x - r * gpr;
   for (int i0 = threadIdx.x; i0 < n4; i0 += 256 * 8) {
      float4 v[8];
      int at[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
         const int i = i0 + 256 * k;
         const int c = 4 * g;
         at[k] = r * ldsw + c;
         const int sx = sx0 + c, sy = sy0 + r;
         const bool rowin = i < n4 && sy >= 0 && sy < H;
         const float *srow = reinterpret_cast<const float *>(src + (size_t)(rowin ? sy : 0) * sstep);
         if (rowin && c + 4 <= ncols && sx >= 0 && sx + 4 <= W) {
            const f32x4_u q = *reinterpret_cast<const f32x4_u *>(srow + sx);
            v[k] = make_float4(q[0], q[1], q[2], q[3]);
         } else {
            float e[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
               e[j] = (rowin && c + j < ncols && sx + j >= 0 && sx + j < W) ? srow[sx + j] : 0.f;
            v[k] = make_float4(e[0], e[1], e[2], e[3]);
         }
         g += dr;
         r += dq;
         if (g >= gpr) {
            g -= gpr;
            ++r;
         }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
         const int i = i0 + 256 * k;
         if (i >= n4) break;
         *reinterpret_cast<float4 *>(lds + at[k]) = v[k];
      }
   }
}

// Window sums of s^2 of a tile's outputs from the staged tile (F32 values of rows y0 - cy ..
// y0 - cy + kTileRows + th - 2, columns x0 - cx .. x0 - cx + kWaves R + tw - 2, zero outside
// the image), in FP64, for the Norm ops when the whole template fits one band.  Two passes
// through LDS past the staged tile (tile_sqsum_lds bytes):
//   h(rho, q)  = sum over u < tw of s(q + u, rho)^2    (rho < kTileRows + th - 1, q < kWaves R)
//   SS(y, q)   = sum over v < th of h(y + v, q)         (y < kTileRows)
// each as the difference of two running sums (lead - lag) of exact FP64 squares along its
// row or column, started at the tile (a window of zeros gives exactly 0).  Returns SS of the
// lane's row y = lane and columns colbase .. colbase + R - 1.  Every thread of the workgroup
// takes part (two barriers).
__host__ __device__ constexpr size_t tile_sqsum_offset(int rows, int ldsw)
{
   return ((size_t)rows * ldsw * sizeof(float) + 15) / 16 * 16;
}
size_t tile_sqsum_lds(int R, int th)
{
   return (size_t)(kTileRows + th - 1 + kTileRows) * kWaves * R * sizeof(double);
}

template <int R>
__device__ __forceinline__ void tile_sqsums(float *lds, int ldsw, int tw, int th, int lane,
                                            int colbase, double (&ss)[R])
{
   constexpr int C4 = kWaves * R;
   const int nrows = kTileRows + th - 1;
   double *hb = reinterpret_cast<double *>(reinterpret_cast<char *>(lds) +
                                           tile_sqsum_offset(nrows, ldsw));
   double *sb = hb + (size_t)nrows * C4;
   // h: one task per staged row and R-column group
   for (int t = threadIdx.x; t < nrows * kWaves; t += 256) {
      const int rho = t / kWaves, q0 = (t - rho * kWaves) * R;
      const float *row = lds + (size_t)rho * ldsw + q0;
      double lead = 0.0, lag = 0.0;
      for (int u = 0; u < tw; ++u) lead = fma((double)row[u], (double)row[u], lead);
      double *hrow = hb + (size_t)rho * C4 + q0;
      hrow[0] = lead;
#pragma unroll
      for (int r = 1; r < R; ++r) {
         lead = fma((double)row[tw + r - 1], (double)row[tw + r - 1], lead);
         lag = fma((double)row[r - 1], (double)row[r - 1], lag);
         hrow[r] = lead - lag;
      }
   }
   __syncthreads();
   // SS: 256 threads = C4 columns x (256 / C4) groups of consecutive output rows
   {
      constexpr int kGroups = 256 / C4, kRows = kTileRows / kGroups;
      static_assert(256 % C4 == 0 && kTileRows % kGroups == 0, "row groups");
      const int q = threadIdx.x % C4, y0 = (threadIdx.x / C4) * kRows;
      double lead = 0.0, lag = 0.0;
      for (int v = 0; v < th; ++v) lead += hb[(size_t)(y0 + v) * C4 + q];
      sb[(size_t)y0 * C4 + q] = lead;
      for (int y = y0 + 1; y < y0 + kRows; ++y) {
         lead += hb[(size_t)(y + th - 1) * C4 + q];
         lag += hb[(size_t)(y - 1) * C4 + q];
         sb[(size_t)y * C4 + q] = lead - lag;
      }
   }
   __syncthreads();
#pragma unroll
   for (int r = 0; r < R; ++r) ss[r] = sb[(size_t)lane * C4 + colbase + r];
}

// One output tile (x0, y0).  Starts with a barrier, so consecutive calls may reuse the LDS.  1-channel F32
// images are staged by stage_tile_f32_v4; with 8 outputs per thread (V4) in an instance of their own,
// since its loads in flight take twice the registers of the other staging (several channels ran 6 to 20
// percent slower with both: 34 -> 74 registers).
template <int OP, int TYPE, int R, bool V4>
__device__ __forceinline__ void tile_f32(float *lds, const char *src, int W, int H, int sstep,
                                         int nch, int ch, const float *__restrict__ tp, int tpitch,
                                         int tw, int th, const double *__restrict__ tsums,
                                         const double *__restrict__ integ, char *dst, int dstep,
                                         int vb, int ldsw, int cx, int cy, int x0, int y0)
{
   constexpr int U = 8;
   const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
   const int ncols = kWaves * R + tw - 1;
   const int nfull = tw / U, rem = tw - nfull * U;
   const int colbase = wave * R;

   float acc[R];
#pragma unroll
   for (int r = 0; r < R; ++r) acc[r] = 0.f;
   const bool v4 = V4 || (TYPE == SImage::F32 && R == 16 && nch == 1);
   // sum t^2 where the host passes none: each workgroup its own from the template (in place), the
   // loads under the staging's
   __shared__ double red[4];
   static_assert(sizeof red == kTileStatic, "static LDS");
   if ((OP == kSSDNorm || OP == kCCNorm) && !tsums) {
      double t2 = 0.0;
      const int n = tw * th;
      for (int i = threadIdx.x; i < n; i += 256) {
         const int v = i / tw;
         const double t = (double)tp[(size_t)v * tpitch + (i - v * tw)];
         t2 = fma(t, t, t2);
      }
      t2 = wave_sum(t2);
      if (lane == 0) red[wave] = t2;
   }

   for (int v0 = 0; v0 < th; v0 += vb) {
      const int nv = min(vb, th - v0);
      __syncthreads();
      if (v4)
         stage_tile_f32_v4(lds, ldsw, kTileRows + nv - 1, ncols, src, W, H, sstep, x0 - cx,
                           y0 - cy + v0);
      else
         stage_tile_f32<TYPE>(lds, ldsw, kTileRows + nv - 1, ncols, src, W, H, sstep, nch, ch,
                              x0 - cx, y0 - cy + v0);
      __syncthreads();
      for (int v = 0; v < nv; ++v) {
         const float *lrow = lds + (size_t)(lane + v) * ldsw;
         const float *trow = tp + (size_t)(v0 + v) * tpitch;
         int u0 = 0;
         for (int c = 0; c < nfull; ++c, u0 += U)
            chunk_f32<OP, R, U, true>(acc, lrow, colbase + u0, trow + u0);
         if (rem & 4) { chunk_f32<OP, R, 4, true>(acc, lrow, colbase + u0, trow + u0); u0 += 4; }
         // the 2- and 1-column chunks from 16-byte reads of a 16-byte aligned column (4-byte
         // LDS reads of consecutive rows would meet in the same banks), the 1-column chunk after
         // a 2-column one from two columns before its own: the reads end at most at column
         // ncols + 2, inside the row pitch
         if (rem & 2) { chunk_f32<OP, R, 2, true>(acc, lrow, colbase + u0, trow + u0); u0 += 2; }
         if (rem & 1) {
            if (rem & 2) chunk_f32<OP, R, 1, true, 2>(acc, lrow, colbase + u0, trow + u0);
            else chunk_f32<OP, R, 1, true>(acc, lrow, colbase + u0, trow + u0);
         }
      }
   }

   const int oy = y0 + lane;
   if (OP == kSSDNorm || OP == kCCNorm) {
      const double tt = tsums ? tsums[0] : red[0] + red[1] + red[2] + red[3];
      double ss[R];
      if (integ) {
         // all integral corners of the R outputs first, then the divisions
#pragma unroll
         for (int r = 0; r < R; ++r) ss[r] = window_sqsum(integ, W, H, x0 + colbase + r, oy, tw, th);
      } else {
         // the whole template was staged in one band (the host passes no integral only
         // then): the window sums of s^2 from the staged tile, in FP64
         tile_sqsums<R>(lds, ldsw, tw, th, lane, colbase, ss);
      }
      if (oy >= H) return;
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] = (float)((double)acc[r] * rsqrt64(ss[r] * tt));
   }
   if (oy >= H) return;
   float *drow = reinterpret_cast<float *>(dst + (size_t)oy * dstep);
   if (nch == 1 && x0 + colbase + R <= W) {
#pragma unroll
      for (int r = 0; r < R; r += 4)
         *reinterpret_cast<f32x4_u *>(drow + x0 + colbase + r) =
             f32x4_u{acc[r], acc[r + 1], acc[r + 2], acc[r + 3]};
      return;
   }
#pragma unroll
   for (int r = 0; r < R; ++r) {
      const int ox = x0 + colbase + r;
      if (ox < W) drow[ox * nch + ch] = acc[r];
   }
}

template <int OP, int TYPE, int R, bool V4>
__global__ __launch_bounds__(256) void prox_tile_f32(const char *src, int W, int H, int sstep,
                                                      int nch, int ch,
                                                      const float *__restrict__ tp, int tpitch,
                                                      int tw, int th,
                                                      const double *__restrict__ tsums,
                                                      const double *__restrict__ integ,
                                                      char *dst, int dstep, int vb, int ldsw,
                                                      int cx, int cy)
{
   extern __shared__ float lds[];
   // one-dimensional grid in XCD-aware tile order
   const int tiles_x = (W + kWaves * R - 1) / (kWaves * R);
   const int tile = xcd_tile(blockIdx.x, gridDim.x);
   tile_f32<OP, TYPE, R, V4>(lds, src, W, H, sstep, nch, ch, tp, tpitch, tw, th, tsums, integ, dst,
                         dstep, vb, ldsw, cx, cy, (tile % tiles_x) * (kWaves * R),
                         (tile / tiles_x) * kTileRows);
}

// CrossCorr_Norm of the tiles that the split-FP16 kernel flagged (SplitFlags): a workgroup walks
// every gridDim.x-th tile and computes those that a flagged tile of that kernel overlaps.  With
// no tile flagged it ends at once (4.6 us at 4096^2).  All flagged, 4096^2/64x64 (a NaN in the source) takes
// 2140 us in all, 2285 with 768 workgroups instead of up to 2048, 2066 by prox_tile_f32.
template <int R>
__global__ __launch_bounds__(256) void prox_tile_f32_flagged(const char *src, int W, int H,
                                                              int sstep,
                                                              const float *__restrict__ tp,
                                                              int tpitch, int tw, int th,
                                                              const double *__restrict__ tsums,
                                                              const double *__restrict__ integ,
                                                              char *dst, int dstep, int vb,
                                                              int ldsw, SplitFlags f)
{
   extern __shared__ float lds[];
   if (*f.any == 0u) return;
   const int tiles_x = (W + kWaves * R - 1) / (kWaves * R);
   const int tiles = tiles_x * ((H + kTileRows - 1) / kTileRows);
   for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
      const int x0 = (t % tiles_x) * (kWaves * R), y0 = (t / tiles_x) * kTileRows;
      const int bx1 = min(x0 + kWaves * R, W) - 1, by1 = min(y0 + kTileRows, H) - 1;
      bool any = false;
      for (int by = y0 / f.tile_h; by <= by1 / f.tile_h; ++by)
         for (int bx = x0 / f.tile_w; bx <= bx1 / f.tile_w; ++bx)
            any |= f.flags[by * f.tiles_x + bx] != 0u;
      if (any)
         tile_f32<kCCNorm, SImage::F32, R, R == 8>(lds, src, W, H, sstep, 1, 0, tp, tpitch, tw, th, tsums,
                                           integ, dst, dstep, vb, ldsw, tw / 2, th / 2, x0, y0);
   }
}

// ------------------------------------------------------------------------- exact integers
template <int TYPE>
__device__ __forceinline__ void stage_tile_int(int32_t *lds, int ldsw, int nrows, int ncols,
                                               const char *src, int W, int H, int sstep,
                                               int nch, int ch, int sx0, int sy0)
{
   const int n = nrows * ldsw;
   // element i = r ldsw + c, (r, c) stepped along with i (256 elements a step) instead of
   // divided out for each element
   const int dq = 256 / ldsw, dr = 256 - dq * ldsw;
   int r = threadIdx.x / ldsw, c = threadIdx.x - r * ldsw;
   for (int i0 = threadIdx.x; i0 < n; i0 += 256 * 8) {
      int32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
         const int i = i0 + 256 * k;
         const int sx = sx0 + c, sy = sy0 + r;
         v[k] = (i < n && c < ncols && sx >= 0 && sx < W && sy >= 0 && sy < H)
                    ? (int32_t)ld<TYPE>(src + (size_t)sy * sstep, sx * nch + ch) : 0;
         c += dr;
         r += dq;
         if (c >= ldsw) {
            c -= ldsw;
            ++r;
         }
      }
#pragma unroll
      for (int k = 0; k < 8; ++k)
         if (i0 + 256 * k < n) lds[i0 + 256 * k] = v[k];
   }
}

// One tap.  int32 sums come from 8-bit sources, whose values and differences fit the 24-bit
// multiplies (v_mad_i32_i24), and for SAD from 16-bit sources too; SAD takes v_sad_u16 (the
// absolute differences of both 16-bit halves plus c; its operands are kept in 0..65535, see
// sad_key, so the high halves are zero).
template <int OP, class ACC> __device__ __forceinline__ ACC itap(ACC acc, int32_t s, int32_t t)
{
   if constexpr (sizeof(ACC) == 4) {
      if (OP == kSSD || OP == kSSDNorm) { int32_t d = s - t; return acc + __mul24(d, d); }
      if (OP == kSAD) return (ACC)__builtin_amdgcn_sad_u16((uint32_t)s, (uint32_t)t, (uint32_t)acc);
      return acc + __mul24(s, t);
   } else {
      if (OP == kSSD || OP == kSSDNorm) { int32_t d = s - t; return acc + (ACC)d * (ACC)d; }
      if (OP == kSAD) { int32_t d = s - t; return acc + (ACC)(d < 0 ? -d : d); }
      return acc + (ACC)s * (ACC)t;
   }
}

// Operand of itap: for SAD with int32 sums on a signed source, the value + 128 (8-bit) or
// + 32768 (16-bit), which maps it in order onto 0..255 or 0..65535 (a sign-extended
// negative value would put 0xffff in v_sad_u16's high half); any other value unchanged.
template <int OP, int TYPE, class ACC> __device__ __forceinline__ int32_t sad_key(int32_t v)
{
   if (OP != kSAD || sizeof(ACC) != 4) return v;
   return TYPE == SImage::S8 ? v + 128 : TYPE == SImage::S16 ? v + 32768 : v;
}

constexpr int kIntU = 8;   // template columns per unrolled chunk of prox_tile_int

// Four 8-bit values (low bytes of a..d) in one dword, a in the low byte.
__device__ __forceinline__ uint32_t pack4(int32_t a, int32_t b, int32_t c, int32_t d)
{
   const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0C0C0400u);
   const uint32_t hi = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x0C0C0400u);
   return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// Four taps at once on packed bytes: v_dot4_u32_u8 / v_dot4_i32_i8.
template <int TYPE> __device__ __forceinline__ int32_t itap4(int32_t acc, uint32_t s, uint32_t t)
{
   if (TYPE == SImage::S8) return __builtin_amdgcn_sdot4((int32_t)s, (int32_t)t, acc, false);
   return (int32_t)__builtin_amdgcn_udot4(s, t, (uint32_t)acc, false);
}

// With int32 sums (8-bit sources) SqrDistance and SqrDistance_Norm take the cross term only,
// one multiply-add per tap, and finish as sum s^2 - 2 sum s*t + sum t^2: the window's sum of
// squares from the FP64 integral (an exact integer below 2^53), sum t^2 from tsums[0].
template <int OP, class ACC> constexpr bool ssd_via_cc()
{
   return (OP == kSSD || OP == kSSDNorm) && sizeof(ACC) == 4;
}

template <int OP, int TYPE, int R, class ACC>
__global__ __launch_bounds__(256) void prox_tile_int(const char *src, int W, int H, int sstep,
                                                      int nch, int ch,
                                                      const int32_t *__restrict__ tp, int tpitch,
                                                      int tw, int th,
                                                      const double *__restrict__ tsums,
                                                      const double *__restrict__ integ,
                                                      char *dst, int dstep, int vb, int ldsw)
{
   extern __shared__ int32_t ldsi[];
   constexpr bool kViaCC = ssd_via_cc<OP, ACC>();
   constexpr int TOP = kViaCC ? kCC : OP;   // the op of each tap
   // 8-bit sources with int32 sums: four taps per instruction on packed bytes
   constexpr bool kPacked = sizeof(ACC) == 4 && (TYPE == SImage::U8 || TYPE == SImage::S8) &&
                            (TOP == kCC || TOP == kCCNorm);
   const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
   const int x0 = blockIdx.x * (kWaves * R), y0 = blockIdx.y * kTileRows;
   const int cx = tw / 2, cy = th / 2;
   const int ncols = kWaves * R + tw - 1;
   const int colbase = wave * R;

   ACC acc[R];
#pragma unroll
   for (int r = 0; r < R; ++r) acc[r] = 0;

   for (int v0 = 0; v0 < th; v0 += vb) {
      const int nv = min(vb, th - v0);
      __syncthreads();
      stage_tile_int<TYPE>(ldsi, ldsw, kTileRows + nv - 1, ncols, src, W,
                           H, sstep, nch, ch, x0 - cx, y0 - cy + v0);
      __syncthreads();
      for (int v = 0; v < nv; ++v) {
         const int32_t *lrow = ldsi + (size_t)(lane + v) * ldsw + colbase;
         const int32_t *trow = tp + (size_t)(v0 + v) * tpitch;
         // the template row in chunks of kIntU columns: kIntU template values and the
         // R + kIntU - 1 window values they meet, then R x kIntU taps (exact integer sums,
         // so the order is free); LDS columns used: colbase .. colbase + R + tw - 2 (the
         // 16-byte reads below take up to one more, inside the row pitch)
         int u0 = 0;
         if constexpr (kPacked) {
            // the window as bytes: aligned dwords q[m] = sw[4m .. 4m+3], the dword starting
            // at byte j = 4m + a by v_alignbyte_b32 of q[m+1]:q[m].  sw is read as 16-byte
            // LDS loads (lrow + u0 is 16-byte aligned: ldsw, colbase and u0 are multiples of
            // 4); the last of them takes one column past the R + kIntU - 1 used, at most
            // column ncols, inside the row pitch (ldsw >= ncols + 4), and its value is
            // never used.
            constexpr int NQ = (R + kIntU - 1 + 3) / 4;
            for (; u0 + kIntU <= tw; u0 += kIntU) {
               int32_t sw[4 * NQ];
               const int4 *w4 = reinterpret_cast<const int4 *>(lrow + u0);
#pragma unroll
               for (int m = 0; m < NQ; ++m) {
                  const int4 v4 = w4[m];
                  sw[4 * m] = v4.x; sw[4 * m + 1] = v4.y; sw[4 * m + 2] = v4.z; sw[4 * m + 3] = v4.w;
               }
               uint32_t q[NQ], tq[kIntU / 4];
#pragma unroll
               for (int m = 0; m < NQ; ++m) q[m] = pack4(sw[4 * m], sw[4 * m + 1], sw[4 * m + 2], sw[4 * m + 3]);
#pragma unroll
               for (int g = 0; g < kIntU / 4; ++g)
                  tq[g] = pack4(trow[u0 + 4 * g], trow[u0 + 4 * g + 1], trow[u0 + 4 * g + 2],
                                trow[u0 + 4 * g + 3]);
#pragma unroll
               for (int g = 0; g < kIntU / 4; ++g)
#pragma unroll
                  for (int r = 0; r < R; ++r) {
                     const int j = r + 4 * g;
                     const uint32_t pj = (j & 3) == 0 ? q[j >> 2]
                                         : __builtin_amdgcn_alignbyte(q[(j >> 2) + 1], q[j >> 2], j & 3);
                     acc[r] = itap4<TYPE>(acc[r], pj, tq[g]);
                  }
            }
         }
         for (; u0 + kIntU <= tw; u0 += kIntU) {
            // the same 16-byte window reads as above
            constexpr int NQ = (R + kIntU - 1 + 3) / 4;
            int32_t t[kIntU], sw[4 * NQ];
#pragma unroll
            for (int k = 0; k < kIntU; ++k) t[k] = sad_key<TOP, TYPE, ACC>(trow[u0 + k]);
            const int4 *w4 = reinterpret_cast<const int4 *>(lrow + u0);
#pragma unroll
            for (int m = 0; m < NQ; ++m) {
               const int4 v4 = w4[m];
               sw[4 * m] = v4.x; sw[4 * m + 1] = v4.y; sw[4 * m + 2] = v4.z; sw[4 * m + 3] = v4.w;
            }
#pragma unroll
            for (int j = 0; j < R + kIntU - 1; ++j) sw[j] = sad_key<TOP, TYPE, ACC>(sw[j]);
#pragma unroll
            for (int k = 0; k < kIntU; ++k)
#pragma unroll
               for (int r = 0; r < R; ++r) acc[r] = itap<TOP, ACC>(acc[r], sw[r + k], t[k]);
         }
         if (u0 < tw) {
            // the last tw % kIntU taps (1 to kIntU - 1) from 16-byte reads of the aligned column
            // u0 too (4-byte LDS reads of consecutive rows would meet in the same banks); the
            // reads end at most at column colbase + R + tw + 1 <= ncols + 2, inside the row
            // pitch
            const int rem = tw - u0;
            constexpr int NQ = (R + kIntU - 1 + 3) / 4;
            int32_t t[kIntU - 1], sw[4 * NQ];
            const int4 *w4 = reinterpret_cast<const int4 *>(lrow + u0);
#pragma unroll
            for (int m = 0; m < NQ; ++m) {
               int4 v4 = make_int4(0, 0, 0, 0);
               if (4 * m < R + rem - 1) v4 = w4[m];
               sw[4 * m] = v4.x; sw[4 * m + 1] = v4.y; sw[4 * m + 2] = v4.z; sw[4 * m + 3] = v4.w;
            }
#pragma unroll
            for (int j = 0; j < R + kIntU - 2; ++j) sw[j] = sad_key<TOP, TYPE, ACC>(sw[j]);
#pragma unroll
            for (int k = 0; k < kIntU - 1; ++k) t[k] = k < rem ? sad_key<TOP, TYPE, ACC>(trow[u0 + k]) : 0;
#pragma unroll
            for (int k = 0; k < kIntU - 1; ++k) {
               if (k >= rem) break;
#pragma unroll
               for (int r = 0; r < R; ++r) acc[r] = itap<TOP, ACC>(acc[r], sw[r + k], t[k]);
            }
         }
      }
   }

   const int oy = y0 + lane;
   if (oy >= H) return;
   float *drow = reinterpret_cast<float *>(dst + (size_t)oy * dstep);
   float val[R];
   if constexpr (kViaCC || OP == kSSDNorm || OP == kCCNorm) {
      // the sums are integers, exact in FP64 below 2^53 (always, for 8-bit sources).
      // Four outputs at a time, each group
      // stored before the next group's integral corners are loaded (the scheduling
      // barriers keep them apart): all sixteen outputs' corners at once would hold about
      // 100 more VGPRs and cost a wave per SIMD
      const double tt = tsums[0];
#pragma unroll
      for (int g = 0; g < R; g += 4) {
         double ss[4];
#pragma unroll
         for (int r = 0; r < 4; ++r)
            ss[r] = window_sqsum(integ, W, H, x0 + colbase + g + r, oy, tw, th);
#pragma unroll
         for (int r = 0; r < 4; ++r) {
            const double c = (double)acc[g + r];
            const double d = kViaCC ? ss[r] - 2.0 * c + tt : c;
            const float v = OP == kSSD ? (float)d : (float)(d * rsqrt64(ss[r] * tt));
            const int ox = x0 + colbase + g + r;
            if (ox < W) drow[ox * nch + ch] = v;
         }
         __builtin_amdgcn_sched_barrier(0);
      }
      return;
   } else {
#pragma unroll
      for (int r = 0; r < R; ++r) val[r] = (float)acc[r];
   }
#pragma unroll
   for (int r = 0; r < R; ++r) {
      const int ox = x0 + colbase + r;
      if (ox < W) drow[ox * nch + ch] = val[r];
   }
}

// ------------------------------------------------------------------------- 8-bit AbsDistance
// Exact int32 sums, four v_sad_u8 per 16 taps and output.  The staged tile holds, for each column c,
// the dword P(c) of the keyed bytes (sad_key) of columns c, c + 4, c + 8, c + 12, so that the
// taps u0 .. u0 + 15 of the output at window column x are |P(x + u0 + k) - Q(u0 + k)|, k < 4, bytewise,
// with Q the template's bytes in the same order (sad8_template): no realignment by bytes.  A
// group of four columns' P is the 4 x 4 byte transpose of 16 source bytes, so the tile is staged
// from one 16-byte load (at any alignment) and eight byte permutes per group, straight into LDS.
// Bound by VALU issue (sads) and the window reads.  1919x1079/31x23 46.7 -> 32.5 us, 4096^2/32x32
// 260 -> 160 us against staging as int32, two LDS passes of repacking and a second template
// launch.  8 outputs per thread at every size: 16 ran 4096^2/32x32 in 157 us, but 640x480/48x48 in
// 54 instead of 38, 2500x2001/61x64 in 306 instead of 267.
constexpr int kSad8R = 8;
constexpr int sad8_blocks(int tw) { return (tw + 15) / 16; }
// columns of P that a tile's outputs read, in whole groups
constexpr int sad8_cols(int tw) { return kWaves * kSad8R + 16 * (sad8_blocks(tw) - 1) + 4; }

__device__ __forceinline__ void transpose4x4(const uint32_t (&q)[4], uint32_t (&p)[4])
{
   const uint32_t t0 = __builtin_amdgcn_perm(q[1], q[0], 0x05010400u);   // 0 4 1 5
   const uint32_t t1 = __builtin_amdgcn_perm(q[1], q[0], 0x07030602u);   // 2 6 3 7
   const uint32_t t2 = __builtin_amdgcn_perm(q[3], q[2], 0x05010400u);   // 8 12 9 13
   const uint32_t t3 = __builtin_amdgcn_perm(q[3], q[2], 0x07030602u);   // 10 14 11 15
   p[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
   p[1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
   p[2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
   p[3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
}

// Q of a template: four dwords per row and block of 16 columns, zero bytes past the row; channel
// blockIdx.y of nch.  One thread per (row, block).
template <int TYPE>
__global__ __launch_bounds__(256) void sad8_template(const unsigned char *tpl, int tw, int th,
                                                     int tstep, int nch, uint32_t *out)
{
   const int nb = sad8_blocks(tw);
   const int i = blockIdx.x * 256 + threadIdx.x, ch = blockIdx.y;
   if (i >= nb * th) return;
   const int v = i / nb, b = i - v * nb;
   const unsigned char *row = tpl + (size_t)v * tstep;
   uint32_t q[4] = {0, 0, 0, 0}, p[4];
#pragma unroll
   for (int k = 0; k < 16; ++k) {
      const int u = 16 * b + k;
      const uint32_t t = u < tw ? row[u * nch + ch] ^ (TYPE == SImage::S8 ? 0x80u : 0u) : 0u;
      q[k / 4] |= t << (8 * (k % 4));
   }
   transpose4x4(q, p);
#pragma unroll
   for (int k = 0; k < 4; ++k) out[((size_t)ch * th * nb + i) * 4 + k] = p[k];
}

// Channel blockIdx.y: its plane plane8 bytes after the one before, its Q likewise.
template <int TYPE>
__global__ __launch_bounds__(256) void prox_sad8(const unsigned char *src, int W, int H, int sstep,
                                                 size_t plane8, const uint32_t *__restrict__ tq,
                                                 int tw, int th, char *dst, int dstep, int nch,
                                                 int vb, int ldsw)
{
   extern __shared__ uint32_t ldsp[];
   constexpr int R = kSad8R;
   constexpr uint32_t kKey = TYPE == SImage::S8 ? 0x80808080u : 0u;
   const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ch = blockIdx.y;
   const int tiles_x = (W + kWaves * R - 1) / (kWaves * R);
   const int tile = xcd_tile(blockIdx.x, gridDim.x);
   const int x0 = (tile % tiles_x) * (kWaves * R), y0 = (tile / tiles_x) * kTileRows;
   const int nb = sad8_blocks(tw), gpr = sad8_cols(tw) / 4;
   const int colbase = wave * R, sx0 = x0 - tw / 2;
   src += ch * plane8;
   tq += (size_t)ch * th * nb * 4;

   uint32_t acc[R];
#pragma unroll
   for (int r = 0; r < R; ++r) acc[r] = 0;
   for (int v0 = 0; v0 < th; v0 += vb) {
      const int nv = min(vb, th - v0), sy0 = y0 - th / 2 + v0;
      const int items = (kTileRows + nv - 1) * gpr;
      __syncthreads();
      {
         // group i = r gpr + g, (r, g) stepped along with i; eight groups in flight
         constexpr int K = 8;
         const int dq = 256 / gpr, dr = 256 - dq * gpr;
         int r = threadIdx.x / gpr, g = threadIdx.x - r * gpr;
         for (int i0 = threadIdx.x; i0 < items; i0 += 256 * K) {
            uint32_t q[K][4];
            int at[K];
#pragma unroll
            for (int k = 0; k < K; ++k) {
               const int sx = sx0 + 4 * g, sy = sy0 + r;
               at[k] = r * ldsw + 4 * g;
               const bool rowin = i0 + 256 * k < items && sy >= 0 && sy < H;
               const unsigned char *row = src + (size_t)(rowin ? sy : 0) * sstep;
               if (rowin && sx >= 0 && sx + 16 <= W) {
                  const u32x4_b b = *reinterpret_cast<const u32x4_b *>(row + sx);
#pragma unroll
                  for (int j = 0; j < 4; ++j) q[k][j] = b[j];
               } else {
#pragma unroll
                  for (int j = 0; j < 4; ++j) q[k][j] = 0;
                  if (rowin && sx + 16 > 0 && sx < W) {
#pragma unroll
                     for (int j = 0; j < 16; ++j) {
                        const int x = sx + j;
                        if (x >= 0 && x < W) q[k][j / 4] |= (uint32_t)row[x] << (8 * (j % 4));
                     }
                  }
               }
               g += dr;
               r += dq;
               if (g >= gpr) {
                  g -= gpr;
                  ++r;
               }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
               if (i0 + 256 * k >= items) break;
               uint32_t p[4];
#pragma unroll
               for (int j = 0; j < 4; ++j) q[k][j] ^= kKey;
               transpose4x4(q[k], p);
               *reinterpret_cast<uint4 *>(ldsp + at[k]) = make_uint4(p[0], p[1], p[2], p[3]);
            }
         }
      }
      __syncthreads();
      for (int v = 0; v < nv; ++v) {
         const uint32_t *lrow = ldsp + (size_t)(lane + v) * ldsw + colbase;
         const uint32_t *trow = tq + (size_t)(v0 + v) * nb * 4;
         auto window = [&](int u0, uint32_t (&pw)[R + 4]) {
            // (an empty asm with a memory clobber: each step reads its window afresh as 16-byte
            // loads, rather than the compiler carrying one dword over from the step before
            // and reading the rest as conflicting 4-byte loads)
            asm volatile("" ::: "memory");
            const uint4 *w4 = reinterpret_cast<const uint4 *>(lrow + u0);
#pragma unroll
            for (int m = 0; m < (R + 4) / 4; ++m) {
               const uint4 a = w4[m];
               pw[4 * m] = a.x; pw[4 * m + 1] = a.y; pw[4 * m + 2] = a.z; pw[4 * m + 3] = a.w;
            }
         };
         int u0 = 0;
         for (; u0 + 16 <= tw; u0 += 16) {
            uint32_t pw[R + 4], t[4];
            window(u0, pw);
#pragma unroll
            for (int k = 0; k < 4; ++k) t[k] = trow[u0 / 4 + k];
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
               for (int k = 0; k < 4; ++k) acc[r] = __builtin_amdgcn_sad_u8(pw[r + k], t[k], acc[r]);
         }
         if (u0 < tw) {
            // a last block of 1 to 15 taps: dword k has the bytes j of the taps u0 + k + 4 j < tw,
            // the others masked out of P (they are zero in Q)
            const int rem = tw - u0;
            uint32_t pw[R + 4];
            window(u0, pw);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
               const int nbytes = (rem - k + 3) >> 2;
               const uint32_t t = trow[u0 / 4 + k];
               if (nbytes >= 4) {
#pragma unroll
                  for (int r = 0; r < R; ++r) acc[r] = __builtin_amdgcn_sad_u8(pw[r + k], t, acc[r]);
               } else if (nbytes > 0) {
                  const uint32_t mk = (1u << (8 * nbytes)) - 1u;
#pragma unroll
                  for (int r = 0; r < R; ++r)
                     acc[r] = __builtin_amdgcn_sad_u8(pw[r + k] & mk, t, acc[r]);
               }
            }
         }
      }
   }
   const int oy = y0 + lane;
   if (oy >= H) return;
   float *drow = reinterpret_cast<float *>(dst + (size_t)oy * dstep);
   const int ox = x0 + colbase;
   if (nch == 1 && ox + R <= W) {
#pragma unroll
      for (int r = 0; r < R; r += 4)
         *reinterpret_cast<f32x4_u *>(drow + ox + r) =
             f32x4_u{(float)acc[r], (float)acc[r + 1], (float)acc[r + 2], (float)acc[r + 3]};
      return;
   }
#pragma unroll
   for (int r = 0; r < R; ++r)
      if (ox + r < W) drow[(ox + r) * nch + ch] = (float)acc[r];
}

// ------------------------------------------------------------------------- direct
template <int OP, int TYPE, class REALT, class STAGED>
__global__ __launch_bounds__(256) void prox_direct(const char *src, int W, int H, int sstep,
                                                    int nch, int ch,
                                                    const STAGED *__restrict__ tp, int tpitch,
                                                    int tw, int th,
                                                    const double *__restrict__ tsums,
                                                    const double *__restrict__ integ,
                                                    char *dst, int dstep)
{
   const int x = blockIdx.x * 16 + (threadIdx.x & 15);
   const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
   if (x >= W || y >= H) return;
   const int left = -(tw / 2), top = -(th / 2);
   REALT sum = 0;
   for (int h = 0; h < th; ++h) {
      const int py = y + h + top;
      const bool rowin = py >= 0 && py < H;
      const char *srow = src + (size_t)(rowin ? py : 0) * sstep;
      for (int w = 0; w < tw; ++w) {
         const int px = x + w + left;
         const REALT t = (REALT)tp[(size_t)h * tpitch + w];
         REALT s = 0;
         if (rowin && px >= 0 && px < W) s = (REALT)ld<TYPE>(srow, px * nch + ch);
         if (OP == kSSD || OP == kSSDNorm) { REALT d = s - t; sum = fma(d, d, sum); }
         else if (OP == kSAD) sum += fabs(s - t);
         else sum = fma(s, t, sum);
      }
   }
   REALT val = sum;
   if (OP == kSSDNorm || OP == kCCNorm)
      val = (REALT)((double)sum / sqrt(window_sqsum(integ, W, H, x, y, tw, th) * tsums[0]));
   reinterpret_cast<REALT *>(dst + (size_t)y * dstep)[x * nch + ch] = val;
}

int lds_pitch(int ncols)
{
   // multiple of 4 floats (16-byte loads) and = 4 mod 32 so that lanes reading the same
   // column of consecutive rows start on different banks
   int p = (ncols + 4 + 3) / 4 * 4;
   while (p % 32 != 4) p += 4;
   return p;
}

}  // namespace

void launch_template_prep(hipStream_t s, const View &t, int channel, int pitch, int kind,
                          void *out, double *sums, unsigned *peak)
{
   KernelTimer kt(s, "template_prep");
   const long long n = (long long)pitch * t.height;
   const int threads = n >= kPrepWide ? kPrepWide : n <= 64 ? 64 : (int)((n + 63) / 64 * 64);
   OCIP_TYPE_SWITCH(t.type, TT, {
      const char *p = static_cast<const char *>(t.ptr);
      auto go = [&](auto kernel) {
         kernel<<<1, threads, 0, s>>>(p, t.width, t.height, t.step, t.channels, channel, pitch, out,
                                      sums, peak);
      };
      if (n <= kPrepWide) {
         if (kind == 0) go(template_prep<TT, 0, 1>);
         else if (kind == 1) go(template_prep<TT, 1, 1>);
         else go(template_prep<TT, 2, 1>);
      } else {
         if (kind == 0) go(template_prep<TT, 0, 8>);
         else if (kind == 1) go(template_prep<TT, 1, 8>);
         else go(template_prep<TT, 2, 8>);
      }
   });
   launch_check("template_prep");
}

// Output columns per lane of the tiled kernels: 8, twice the workgroups and less staged at once, or
// 16, fewer LDS reads per tap.  8 below 2 Mpx, whose workgroups of 16 do not fill the GPU (640x480/48x48
// SqrDistance 172 us with 16, 104 with 8), 16 above where it is the faster one (us with 16, with 8):
//   templates 96 columns wide, whose halo is a third of a tile of 16 and half of one of 8 (CrossCorr F32
//   x 4 1920x1080/20x100 600, 668), or tall and a few columns wide (CrossCorr 2048x1024/150x4 U8 168, 235,
//   U16 140, 193, F32 x 4 433, 534);
//   AbsDistance of 16-bit unsigned images from 200 taps on (1920x1080/64x64 300, 419; 16x16 36, 40);
//   SqrDistance(_Norm) and AbsDistance with 1024 taps where the tiles of 16 are about two workgroups
//   per CU, all resident, and those of 8 a third and a fourth (1920x1080/64x64 F32 348, 375; 4000x2000
//   the other way round: 1180, 1120);
//   up to 1024 taps from 4 Mpx on (F32 CrossCorr 4096^2: 8x8 57, 64; 64x64 1994, 1951).
// The F32 Norm ops, whose window sums come from tiles of 8 but from an integral with 16, take 16 up to
// 1024 taps only where the integral is the smaller part (SqrDistance_Norm 4096^2: 8x8 282, 189; 16x16
// 297, 323; 2048^2/16x16 103, 81), and not in images of less than 2048 columns: the tiles' sums round
// relative to the tile's energy, the integral's to all of the image above and left, and one NaN there
// reaches the rest of the image (SqrDistance_Norm 2000x4200/16x16 217, 192; 2000x4400/24x24 322, 323).
static int tile_r(int op, const View &S, const View &T)
{
   const long long px = (long long)S.width * S.height, taps = (long long)T.width * T.height;
   const bool norm = S.type == SImage::F32 && (op == kSSDNorm || op == kCCNorm);
   if (px < 2000000) return 8;
   if (T.width >= 96 || (T.height >= 100 && T.width < 8)) return 16;   // (no tile holds their window sums)
   if (op == kSAD && S.type == SImage::U16 && taps >= 200 && T.width >= 8) return 16;
   if (taps >= 1024) {
      const long long tiles = (long long)((S.width + 63) / 64) * ((S.height + kTileRows - 1) / kTileRows);
      return (op == kSSD || op == kSSDNorm || op == kSAD) && tiles > 384 && tiles <= 512 ? 16 : 8;
   }
   if (px < (norm ? 8 : 4) * (1 << 20)) return 8;
   if (norm && (taps < 200 || S.width < 2048)) return 8;
   return 16;
}

bool prox_norm_from_tile(int op, const View &S, const View &T)
{
   if ((op != kSSDNorm && op != kCCNorm) || S.type != SImage::F32 || T.width <= 0 || T.height <= 0)
      return false;
   const int R = tile_r(op, S, T);
   const int ldsw = lds_pitch(kWaves * R + T.width - 1);
   const int rows_fit = kLdsBudget / (ldsw * 4) - (kTileRows - 1);
   if (rows_fit < T.height) return false;   // one band
   return tile_sqsum_offset(kTileRows + T.height - 1, ldsw) + tile_sqsum_lds(R, T.height) <=
          (size_t)kLdsBudget;
}

// The tile of prox_sad8 in LDS: pitch and template rows per band (0: it does not fit)
static void sad8_tile(int tw, int th, int &ldsw, int &vb)
{
   ldsw = sad8_cols(tw);
   while (ldsw % 32 != 4) ldsw += 4;   // 16-byte reads of consecutive rows on different banks
   vb = std::max(0, std::min(th, kLdsBudget / (ldsw * 4) - (kTileRows - 1)));
}

bool sad8_ok(int op, const View &S, const View &T)
{
   if (op != kSAD || (S.type != SImage::U8 && S.type != SImage::S8)) return false;
   if (S.channels != 1 && S.channels != 2 && S.channels != 4) return false;
   if (T.width <= 0 || T.height <= 0 || (long long)T.width * T.height * 65025LL >= (1LL << 31))
      return false;   // int32 sums
   int ldsw, vb;
   sad8_tile(T.width, T.height, ldsw, vb);
   return vb >= 1;
}

static size_t sad8_template_bytes(const View &T)
{
   return ((size_t)T.channels * T.height * sad8_blocks(T.width) * 16 + 255) / 256 * 256;
}

size_t sad8_work_bytes(const View &S, const View &T)
{
   return sad8_template_bytes(T) + planes8_bytes(S);
}

void launch_sad8(hipStream_t s, const View &image, const View &T, void *dst, int dstep, void *work)
{
   const int tw = T.width, th = T.height, nch = image.channels, R = kSad8R;
   uint32_t *tq = static_cast<uint32_t *>(work);
   View S = image;
   size_t plane8 = 0;
   if (nch > 1) S = launch_planes8(s, image, static_cast<char *>(work) + sad8_template_bytes(T), &plane8);
   int ldsw, vb;
   sad8_tile(tw, th, ldsw, vb);
   const unsigned tiles = ((S.width + kWaves * R - 1) / (kWaves * R)) * ((S.height + kTileRows - 1) / kTileRows);
   const size_t lds = (size_t)(kTileRows + vb - 1) * ldsw * 4;
   const int items = sad8_blocks(tw) * th;
   auto go = [&](auto prep, auto kernel) {
      {
         KernelTimer kt(s, "template_prep");
         prep<<<dim3((items + 255) / 256, nch), 256, 0, s>>>(
             static_cast<const unsigned char *>(T.ptr), tw, th, T.step, nch, tq);
         launch_check("sad8_template");
      }
      KernelTimer kt(s, "prox_sad8");
      kernel<<<dim3(tiles, nch), 256, lds, s>>>(static_cast<const unsigned char *>(S.ptr), S.width,
                                                S.height, S.step, plane8, tq, tw, th,
                                                static_cast<char *>(dst), dstep, nch, vb, ldsw);
      launch_check("prox_sad8");
   };
   if (S.type == SImage::U8) go(sad8_template<SImage::U8>, prox_sad8<SImage::U8>);
   else go(sad8_template<SImage::S8>, prox_sad8<SImage::S8>);
}

void launch_proximity_flagged(hipStream_t s, const View &S, const View &T, void *dst, int dstep,
                              const void *tstage, int tpitch, const double *tsums,
                              const double *integ, const SplitFlags &f)
{
   const int W = S.width, H = S.height, tw = T.width, th = T.height;
   const int R = tile_r(kCCNorm, S, T);   // (8 where the tiles have the window sums)
   const int ldsw = lds_pitch(kWaves * R + tw - 1);
   const int vb = min(th, kLdsBudget / (ldsw * 4) - (kTileRows - 1));   // >= 1: split_ncc_ok
   const size_t lds = integ ? (size_t)(kTileRows + vb - 1) * ldsw * 4
                            : tile_sqsum_offset(kTileRows + vb - 1, ldsw) + tile_sqsum_lds(R, th);
   if (!integ && !prox_norm_from_tile(kCCNorm, S, T)) fail(CL_INVALID_VALUE, "integral required");
   const int tiles = ((W + kWaves * R - 1) / (kWaves * R)) * ((H + kTileRows - 1) / kTileRows);
   KernelTimer kt(s, "prox_flagged");
   auto go = [&](auto kernel) {
      kernel<<<min(tiles, 2048), 256, lds, s>>>(
          static_cast<const char *>(S.ptr), W, H, S.step, static_cast<const float *>(tstage), tpitch,
          tw, th, tsums, integ, static_cast<char *>(dst), dstep, vb, ldsw, f);
   };
   if (R == 16) go(prox_tile_f32_flagged<16>); else go(prox_tile_f32_flagged<8>);
   launch_check("prox_flagged");
}

// The tile kernel reads an F32 template's rows as scalar loads wherever they lie, and for the Norm
// ops each workgroup sums t^2 by itself, up to kTileTaps taps (four a thread); past that, or with
// the denominators from the integral, template_prep's launch costs less than the sums.
// (SqrDistance_Norm 1024^2/16x16 30.6 -> 22.2 us with the vector staging and stores.)
bool prox_template_in_place(int op, const View &S, const View &T, bool have_integral)
{
   constexpr int kTileTaps = 1024;
   if (S.type != SImage::F32 || S.channels != 1 || T.width <= 0 || T.height <= 0) return false;
   const int ncols = kWaves * tile_r(op, S, T) + T.width - 1;
   if (kLdsBudget / (lds_pitch(ncols) * 4) - (kTileRows - 1) < 1) return false;   // prox_direct
   const bool norm = op == kSSDNorm || op == kCCNorm;
   return !norm || (!have_integral && T.width * T.height <= kTileTaps);
}

template <int OP>
static void launch_op(hipStream_t s, const View &S, const View &T, void *dst, int dstep,
                      const void *tstage, int tpitch, const double *tsums, const double *integ,
                      int ch)
{
   const int W = S.width, H = S.height, tw = T.width, th = T.height;
   const char *src = static_cast<const char *>(S.ptr);
   const bool small_int = S.type == SImage::U8 || S.type == SImage::S8 ||
                          S.type == SImage::U16 || S.type == SImage::S16;
   const int R = tile_r(OP, S, T);
   const int ncols = kWaves * R + tw - 1;
   // int32 accumulation is exact when taps * max|term| < 2^31: 8-bit sources up to 33025
   // taps, and AbsDistance on 16-bit sources up to 32768 taps; the other 16-bit cases
   // accumulate in int64.
   const bool bits8 = S.type == SImage::U8 || S.type == SImage::S8;
   const long long taps = (long long)tw * th;
   const bool fits32 = bits8 ? taps * 65025LL < (1LL << 31)
                             : OP == kSAD && taps * 65535LL < (1LL << 31);
   const int ldsw = lds_pitch(ncols);
   const int rows_fit = kLdsBudget / (ldsw * 4) - (kTileRows - 1);
   const bool tiled = S.type != SImage::F64 && rows_fit >= 1 && th > 0 && tw > 0;

   if (!tiled) {
      KernelTimer kt(s, "prox_direct");
      dim3 grid((W + 15) / 16, (H + 15) / 16);
      if (S.type == SImage::F64) {
         prox_direct<OP, SImage::F64, double, double><<<grid, 256, 0, s>>>(
             src, W, H, S.step, S.channels, ch, static_cast<const double *>(tstage), tpitch, tw,
             th, tsums, integ, static_cast<char *>(dst), dstep);
      } else if (small_int) {
         OCIP_TYPE_SWITCH(S.type, TT, {
            prox_direct<OP, TT, float, int32_t><<<grid, 256, 0, s>>>(
                src, W, H, S.step, S.channels, ch, static_cast<const int32_t *>(tstage), tpitch,
                tw, th, tsums, integ, static_cast<char *>(dst), dstep);
         });
      } else {
         OCIP_TYPE_SWITCH(S.type, TT, {
            prox_direct<OP, TT, float, float><<<grid, 256, 0, s>>>(
                src, W, H, S.step, S.channels, ch, static_cast<const float *>(tstage), tpitch,
                tw, th, tsums, integ, static_cast<char *>(dst), dstep);
         });
      }
      launch_check("prox_direct");
      return;
   }

   const int vb = min(th, rows_fit);
   size_t lds = (size_t)(kTileRows + vb - 1) * ldsw * 4;
   dim3 grid((W + kWaves * R - 1) / (kWaves * R), (H + kTileRows - 1) / kTileRows);
   // Norm ops on F32 sources with no integral: window sums from the staged tile
   if ((OP == kSSDNorm || OP == kCCNorm) && !integ) {
      if (!prox_norm_from_tile(OP, S, T)) fail(CL_INVALID_VALUE, "integral required");
      lds = tile_sqsum_offset(kTileRows + vb - 1, ldsw) + tile_sqsum_lds(R, th);
   }

#define OCIP_TILE_F32(TT_, R_, V4_)                                                            \
   prox_tile_f32<OP, TT_, R_, V4_><<<grid.x * grid.y, 256, lds, s>>>(                          \
       src, W, H, S.step, S.channels, ch, static_cast<const float *>(tstage), tpitch, tw, th, \
       tsums, integ, static_cast<char *>(dst), dstep, vb, ldsw, tw / 2, th / 2)
#define OCIP_TILE_INT(TT_, R_, ACC_)                                                             \
   prox_tile_int<OP, TT_, R_, ACC_><<<grid, 256, lds, s>>>(                                     \
       src, W, H, S.step, S.channels, ch, static_cast<const int32_t *>(tstage), tpitch, tw, th, \
       tsums, integ, static_cast<char *>(dst), dstep, vb, ldsw)

   if (small_int) {
      KernelTimer kt(s, "prox_tile_int");
      OCIP_TYPE_SWITCH(S.type, TT, {
         if (fits32) {
            if (R == 16) OCIP_TILE_INT(TT, 16, int32_t); else OCIP_TILE_INT(TT, 8, int32_t);
         } else {
            if (R == 16) OCIP_TILE_INT(TT, 16, long long); else OCIP_TILE_INT(TT, 8, long long);
         }
      });
      launch_check("prox_tile_int");
   } else {
      KernelTimer kt(s, "prox_tile_f32");
      switch (S.type) {
      case SImage::F32:
         if (R == 16) OCIP_TILE_F32(SImage::F32, 16, false);
         else if (S.channels == 1) OCIP_TILE_F32(SImage::F32, 8, true);
         else OCIP_TILE_F32(SImage::F32, 8, false);
         break;
      case SImage::U32:
         if (R == 16) OCIP_TILE_F32(SImage::U32, 16, false); else OCIP_TILE_F32(SImage::U32, 8, false);
         break;
      case SImage::S32:
         if (R == 16) OCIP_TILE_F32(SImage::S32, 16, false); else OCIP_TILE_F32(SImage::S32, 8, false);
         break;
      default: fail(CL_IMAGE_FORMAT_NOT_SUPPORTED, "type");
      }
      launch_check("prox_tile_f32");
   }
#undef OCIP_TILE_F32
#undef OCIP_TILE_INT
}

void launch_proximity(hipStream_t s, int op, const View &S, const View &T, void *dst, int dstep,
                      const void *tstage, int tpitch, const double *tsums, const double *integ,
                      int ch)
{
   switch (op) {
   case kSSD: launch_op<kSSD>(s, S, T, dst, dstep, tstage, tpitch, tsums, integ, ch); break;
   case kSSDNorm: launch_op<kSSDNorm>(s, S, T, dst, dstep, tstage, tpitch, tsums, integ, ch); break;
   case kSAD: launch_op<kSAD>(s, S, T, dst, dstep, tstage, tpitch, tsums, integ, ch); break;
   case kCC: launch_op<kCC>(s, S, T, dst, dstep, tstage, tpitch, tsums, integ, ch); break;
   case kCCNorm: launch_op<kCCNorm>(s, S, T, dst, dstep, tstage, tpitch, tsums, integ, ch); break;
   default: fail(CL_INVALID_VALUE, "op");
   }
}

}  // namespace ocip
