// integral.hip -- inclusive 2-D prefix sum / sum of squares in FP64.
//
// Semantics: reference Integral.cl / Integral.cpp (I(x,y) = sum over j<=y, i<=x of f(S[j][i]),
// same size as the source, f = identity or square; include/OpenCLIPP.h:639-645).  The
// reference sums in the Dest precision through a 5-launch, 64x8 block scan with serial
// junction loops (Integral.cl:39-460).  Here every sum is formed in FP64 (exact for 8/16-bit
// integer sources, whose partial sums stay below 2^53) and rounded once to the Dest type.
//
// Design: the image is cut into tiles of 32 rows x 256 columns, one wavefront per tile
// (4 columns per lane), so every scan is a wavefront shuffle scan with no barrier.  Three
// launches, with the source read twice and the output written once:
//   1. aggregates: per tile, its column sums, its row sums and its total;
//   2. carries   : exclusive scans of the column sums over tile rows, of the row sums over
//                  tile columns, and the 2-D exclusive scan of the tile totals;
//   3. final     : per tile, the in-tile 2-D scan (a running column sum per lane and one
//                  wavefront scan per row) plus the three carries.
// HBM traffic: 2 x source + 1 x output (+ small aggregates).
#include <type_traits>

#include "device_common.h"

namespace ocip {

namespace {

constexpr int kThreads = 64;            // one wavefront per tile: no barriers
constexpr int kVec = 4;                 // columns per lane
constexpr int kCW = kThreads * kVec;    // tile width (256)
constexpr int kRH = 32;                 // tile height
constexpr int kRowUnroll = 8;           // rows whose loads are issued together

struct IntegralAux {
   // layout inside the aux buffer (doubles):
   //   colsum  [RB][W]     column sums per tile row, then exclusive-scanned over tile rows
   //   rowsum  [H][CB]     row sums per tile column, then exclusive-scanned over tile columns
   //   tiletot [RB][CB]    tile totals, then 2-D exclusive-scanned (corner carries)
   //   tilepeak [RB][CB]   (unsigned) high word of the tile's largest f
   double *colsum, *rowsum, *tiletot;
   unsigned *tilepeak;
   int CB, RB;
};

__host__ __device__ inline int cdiv(int a, int b) { return (a + b - 1) / b; }

IntegralAux aux_layout(void *base, int W, int H)
{
   IntegralAux a;
   a.CB = cdiv(W, kCW);
   a.RB = cdiv(H, kRH);
   double *p = static_cast<double *>(base);
   a.colsum = p;
   a.rowsum = a.colsum + (size_t)a.RB * W;
   a.tiletot = a.rowsum + (size_t)H * a.CB;
   a.tilepeak = reinterpret_cast<unsigned *>(a.tiletot + (size_t)a.RB * a.CB);
   return a;
}

// Four elements read or written at once, at the element's own alignment (see f32x4_u).  (A vector
// type: from a struct's array the selection of `values` was compiled into an indexed copy in scratch
// memory; SqrIntegral of F64 3001x2003 into F32 49.6 -> 32.5 us.)
template <class T> struct Vec4 {
   typedef T type __attribute__((ext_vector_type(4), aligned(alignof(T))));
};

// The lane's 4 elements of a row as loaded, unconditionally, so that many rows can be in flight in
// ragged tiles too: rows from y1 on read the row before, columns from W on the last ones inside
// (VEC: 1-channel rows of at least 4 elements, one vector load at column min(x0, W - 4)).
template <int TYPE, bool VEC>
__device__ __forceinline__ typename Vec4<typename ElemT<TYPE>::type>::type
load_raw(const char *src, int step, int y, int y1, int x0, int W, int nch, int ch)
{
   typedef typename ElemT<TYPE>::type T;
   typedef typename Vec4<T>::type V;
   const char *row = src + (size_t)min(y, y1 - 1) * step;
   if (VEC) return *reinterpret_cast<const V *>(row + (size_t)min(x0, W - 4) * sizeof(T));
   V q;
#pragma unroll
   for (int j = 0; j < kVec; ++j) q[j] = ld<TYPE>(row, min(x0 + j, W - 1) * nch + ch);
   return q;
}

// f(s) for the lane's 4 columns of row y from load_raw's elements, 0 outside [0, y1) x [0, W).
// WHOLE: the tile lies inside the image.
template <class T, bool WHOLE, bool SQR, bool VEC, class A>
__device__ __forceinline__ void values(typename Vec4<T>::type q, int y, int y1, int x0, int W, A (&v)[kVec])
{
   const int d = VEC && !WHOLE ? x0 - min(x0, W - 4) : 0;   // the vector starts d columns early
#pragma unroll
   for (int j = 0; j < kVec; ++j) {
      T e = q[j];
      if (!WHOLE) {
#pragma unroll
         for (int k = j + 1; k < kVec; ++k)
            if (d == k - j) e = q[k];
         if (y >= y1 || x0 + j >= W) e = (T)0;
      }
      const A f = (A)e;
      v[j] = SQR ? f * f : f;
   }
}

// body(whole) with whole = std::true_type for tiles wholly inside the image, false_type for others
template <class F> __device__ __forceinline__ void by_tile(int cb, int rb, int W, int H, F &&body)
{
   if ((cb + 1) * kCW <= W && (rb + 1) * kRH <= H) body(std::true_type());
   else body(std::false_type());
}

// 1. per-tile aggregates: column sums, row sums, tile total (and the tile's peak where the
// caller wants the image's: f >= 0 then).  Bound by memory latency: kAggRows rows of raw elements
// are in flight per lane and converted afterwards, 8-bit images are summed in int32 (a tile's
// column holds at most 32 x 255^2), and two lanes share each row's sum (U8 4096^2: 16 -> 7 us,
// F32: 17 -> 15 us; rows of odd pitch took one load per element before: 3001x2003 F32 66 -> 29 us for
// all three launches).
constexpr int kAggRows = 16;

template <int TYPE, bool SQR, bool VEC, bool PEAK>
__global__ __launch_bounds__(kThreads) void integral_aggregate(const char *src, int W, int H,
                                                                int step, int nch, int ch,
                                                                IntegralAux aux)
{
   constexpr bool kInt = TYPE == SImage::U8 || TYPE == SImage::S8;
   typedef typename std::conditional<kInt, int, double>::type A;
   // each lane's partial row sums, rows x lanes (odd pitch: the walks along the rows spread
   // over the banks); lanes r and r + 32 then sum the halves of row r in lane order
   __shared__ A part[kRH][kThreads + 1];
   static_assert(kRH % kAggRows == 0 && 2 * kRH == kThreads, "rows of the tile");
   const int cb = blockIdx.x, rb = blockIdx.y;
   const int x0 = cb * kCW + threadIdx.x * kVec;
   const int y0 = rb * kRH, y1 = min(y0 + kRH, H);
   A col[kVec] = {0, 0, 0, 0};
   unsigned peak = 0;
   by_tile(cb, rb, W, H, [&](auto whole) {
      for (int y = y0; y < y1; y += kAggRows) {
         typename Vec4<typename ElemT<TYPE>::type>::type q[kAggRows];
#pragma unroll
         for (int r = 0; r < kAggRows; ++r)
            q[r] = load_raw<TYPE, VEC>(src, step, y + r, y1, x0, W, nch, ch);
#pragma unroll
         for (int r = 0; r < kAggRows; ++r) {
            A v[kVec], rs = 0;
            values<typename ElemT<TYPE>::type, decltype(whole)::value, SQR, VEC>(q[r], y + r, y1, x0, W, v);
#pragma unroll
            for (int j = 0; j < kVec; ++j) {
               col[j] += v[j];
               rs += v[j];
               if (PEAK) peak = max(peak, (unsigned)__double2hiint((double)v[j]) & 0x7fffffffu);
            }
            part[y - y0 + r][threadIdx.x] = rs;   // rows past y1 hold 0 and are not summed
         }
      }
   });
#pragma unroll
   for (int j = 0; j < kVec; ++j)
      if (x0 + j < W) aux.colsum[(size_t)rb * W + x0 + j] = (double)col[j];
   __syncthreads();
   const int r = threadIdx.x & 31, l0 = threadIdx.x & 32;
   A rs = 0;
   if (r < y1 - y0)
#pragma unroll 8
      for (int l = 0; l < 32; ++l) rs += part[r][l0 + l];
   rs += __shfl_xor(rs, 32, 64);
   if (r < y1 - y0 && l0 == 0) aux.rowsum[(size_t)(y0 + r) * aux.CB + cb] = (double)rs;
   const double tot = wave_sum(l0 == 0 ? (double)rs : 0.0);
   if (threadIdx.x == 0) aux.tiletot[(size_t)rb * aux.CB + cb] = tot;
   if (PEAK) {
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) peak = max(peak, (unsigned)__shfl_xor((int)peak, d, 64));
      if (threadIdx.x == 0) aux.tilepeak[(size_t)rb * aux.CB + cb] = peak;
   }
}

// exclusive scan in place of n values at p[0], p[stride], ...
__device__ __forceinline__ void exclusive_scan_strided(double *p, int n, size_t stride)
{
   // 32 loads in flight: the scans are chains of round trips (128 tile rows at 4096 rows)
   constexpr int B = 32;
   double acc = 0;
   for (int k = 0; k < n; k += B) {
      double v[B];
#pragma unroll
      for (int i = 0; i < B; ++i) v[i] = k + i < n ? p[(size_t)(k + i) * stride] : 0.0;
#pragma unroll
      for (int i = 0; i < B; ++i) {
         if (k + i < n) p[(size_t)(k + i) * stride] = acc;
         acc += v[i];
      }
   }
}

// Exclusive scans down n rows (W elements apart) of COLS adjacent columns, in place, by one
// workgroup of 256 threads: 256 / COLS groups of rows, one per thread of a column, whose sums
// go through LDS; up to K rows of a group stay in registers between the two passes, more are read
// again.  One round trip to memory where a thread per column took n / 32: the carries of 4096^2
// (128 tile rows) 10.0 -> 6.0 us.
template <int COLS, int K>
__device__ __forceinline__ void scan_columns(double *base, int n, size_t W, int x, int xend)
{
   constexpr int GROUPS = 256 / COLS;
   __shared__ double total[GROUPS][COLS];
   const int c = threadIdx.x % COLS, g = threadIdx.x / COLS;
   const int per = cdiv(n, GROUPS), k0 = min(g * per, n), k1 = min(k0 + per, n);
   double *p = base + min(x + c, xend - 1);
   double v[K], sum = 0.0;
   for (int k = k0; k < k1; k += K) {
#pragma unroll
      for (int i = 0; i < K; ++i) v[i] = k + i < k1 ? p[(size_t)(k + i) * W] : 0.0;
#pragma unroll
      for (int i = 0; i < K; ++i) sum += v[i];
   }
   __syncthreads();   // (an earlier call's totals are read)
   total[g][c] = sum;
   __syncthreads();
   double acc = 0.0;
   for (int w = 0; w < g; ++w) acc += total[w][c];
   for (int k = k0; k < k1; k += K) {
      if (per > K) {
#pragma unroll
         for (int i = 0; i < K; ++i) v[i] = k + i < k1 ? p[(size_t)(k + i) * W] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < K; ++i) {
         if (k + i < k1 && x + c < xend) p[(size_t)(k + i) * W] = acc;
         acc += v[i];
      }
   }
}

// 2. carries.  blockIdx.y = 0: column sums over tile rows, 64 columns a block;
//              blockIdx.y = 1: row sums over tile columns, one thread per row;
//              blockIdx.y = 2: 2-D exclusive scan of the tile totals (block 0);
//              blockIdx.y = 3: the largest tile peak into *peak (block 0, where wanted).
__global__ __launch_bounds__(256) void integral_carries(int W, int H, IntegralAux aux,
                                                        unsigned *peak)
{
   if (blockIdx.y == 3) {
      if (blockIdx.x) return;
      __shared__ unsigned red[4];
      unsigned m = 0;
      for (int k = threadIdx.x; k < aux.RB * aux.CB; k += 256) m = max(m, aux.tilepeak[k]);
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, d, 64));
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
      __syncthreads();
      if (threadIdx.x == 0) *peak = max(max(red[0], red[1]), max(red[2], red[3]));
      return;
   }
   const int i = blockIdx.x * 256 + threadIdx.x;
   if (blockIdx.y == 0) {
      if (blockIdx.x * 64 < W) scan_columns<64, 32>(aux.colsum, aux.RB, W, blockIdx.x * 64, W);
   } else if (blockIdx.y == 1) {
      if (i < H) exclusive_scan_strided(aux.rowsum + (size_t)i * aux.CB, aux.CB, 1);
   } else if (blockIdx.x == 0) {
      // along each tile row, then down each tile column:
      // corner[rb][cb] = sum over rb' < rb, cb' < cb of the tile totals
      for (int rb = threadIdx.x; rb < aux.RB; rb += 256)
         exclusive_scan_strided(aux.tiletot + (size_t)rb * aux.CB, aux.CB, 1);
      __syncthreads();
      for (int cb = 0; cb < aux.CB; cb += 16)
         scan_columns<16, 8>(aux.tiletot, aux.RB, aux.CB, cb, aux.CB);
   }
}

// 4 output values of a row at column x0 (j = 0..3)
template <class T>
__device__ __forceinline__ void store4(T *o, int x0, int W, const double (&val)[kVec])
{
   if (x0 + kVec <= W) {
      typename Vec4<T>::type q;
#pragma unroll
      for (int j = 0; j < kVec; ++j) q[j] = (T)val[j];
      *reinterpret_cast<typename Vec4<T>::type *>(o + x0) = q;
      return;
   }
#pragma unroll
   for (int j = 0; j < kVec; ++j)
      if (x0 + j < W) o[x0 + j] = (T)val[j];
}

// 3. final pass.  OUT: 0 = F32 inclusive, 1 = F64 inclusive (both with the caller's pitch),
// 2 = the internal exclusive layout.
template <int TYPE, bool SQR, bool VEC, int OUT>
__global__ __launch_bounds__(kThreads) void integral_final(const char *src, int W, int H,
                                                            int step, int nch, int ch,
                                                            IntegralAux aux, char *out,
                                                            int ostep)
{
   const int cb = blockIdx.x, rb = blockIdx.y;
   const int x0 = cb * kCW + threadIdx.x * kVec;
   const int y0 = rb * kRH, y1 = min(y0 + kRH, H);

   // carry from the tiles above: prefix over this tile's columns of the column carries
   double px[kVec];
   {
      double loc = 0;
#pragma unroll
      for (int j = 0; j < kVec; ++j) {
         const int x = x0 + j;
         loc += x < W ? aux.colsum[(size_t)rb * W + x] : 0.0;
         px[j] = loc;
      }
      const double excl = wave_inclusive_scan(loc) - loc;
#pragma unroll
      for (int j = 0; j < kVec; ++j) px[j] += excl;
   }
   const double corner = aux.tiletot[(size_t)rb * aux.CB + cb];
   const size_t P = excl_pitch(W);

   if (OUT == 2) {
      // row 0 and column 0 of the exclusive layout are 0
      double *o = reinterpret_cast<double *>(out) + kExclOffset;
      if (rb == 0) {
#pragma unroll
         for (int j = 0; j < kVec; ++j)
            if (x0 + j < W) o[x0 + j + 1] = 0.0;
         if (cb == 0 && threadIdx.x == 0) o[0] = 0.0;
      }
      if (cb == 0)
         for (int y = y0 + threadIdx.x; y < y1; y += kThreads) o[(size_t)(y + 1) * P] = 0.0;
   }

   double colrun[kVec] = {0, 0, 0, 0};
   double py = 0;
   by_tile(cb, rb, W, H, [&](auto whole) {
      for (int y = y0; y < y1; y += kRowUnroll) {
         typename Vec4<typename ElemT<TYPE>::type>::type q[kRowUnroll];
         double v[kRowUnroll][kVec];
         double rc[kRowUnroll];
#pragma unroll
         for (int r = 0; r < kRowUnroll; ++r) {
            q[r] = load_raw<TYPE, VEC>(src, step, y + r, y1, x0, W, nch, ch);
            rc[r] = aux.rowsum[(size_t)min(y + r, y1 - 1) * aux.CB + cb];   // (unused from y1 on)
         }
#pragma unroll
         for (int r = 0; r < kRowUnroll; ++r)
            values<typename ElemT<TYPE>::type, decltype(whole)::value, SQR, VEC>(q[r], y + r, y1, x0, W, v[r]);
         // the lane's prefixes of the batch's rows, then their wavefront scans together
         double p[kRowUnroll][kVec], inc[kRowUnroll];
#pragma unroll
         for (int r = 0; r < kRowUnroll; ++r) {
            double loc = 0;
#pragma unroll
            for (int j = 0; j < kVec; ++j) {
               colrun[j] += v[r][j];
               loc += colrun[j];
               p[r][j] = loc;
            }
            inc[r] = loc;
         }
         wave_incl_scan_f64<kRowUnroll>(inc);
#pragma unroll
         for (int r = 0; r < kRowUnroll; ++r) {
            py += rc[r];
            const double base = corner + py + (inc[r] - p[r][kVec - 1]);
            const int yy = y + r;
            if (yy >= y1) continue;
            double val[kVec];
#pragma unroll
            for (int j = 0; j < kVec; ++j) val[j] = base + p[r][j] + px[j];
            if (OUT == 0)
               store4<float>(reinterpret_cast<float *>(out + (size_t)yy * ostep), x0, W, val);
            else if (OUT == 1)
               store4<double>(reinterpret_cast<double *>(out + (size_t)yy * ostep), x0, W, val);
            else
               store4<double>(reinterpret_cast<double *>(out) + (size_t)(yy + 1) * P +
                                        kExclOffset + 1, x0, W, val);
         }
      }
   });
}

}  // namespace

size_t integral_aux_bytes(int W, int H)
{
   size_t CB = cdiv(W, kCW), RB = cdiv(H, kRH);
   return (RB * W + (size_t)H * CB + RB * CB) * sizeof(double) + RB * CB * sizeof(unsigned);
}

template <int TT, bool VEC>
static void launch_integral_t(hipStream_t s, const char *src, const View &v, int channel,
                              bool sqr, void *out, int ostep, int mode, IntegralAux aux,
                              unsigned *peak)
{
   const int W = v.width, H = v.height;
   dim3 grid(aux.CB, aux.RB);
   KernelTimer kt(s, "integral");
   auto aggregate = [&](auto kernel) {
      kernel<<<grid, kThreads, 0, s>>>(src, W, H, v.step, v.channels, channel, aux);
   };
   if (peak) {
      if constexpr (TT == SImage::F32) aggregate(integral_aggregate<TT, true, VEC, true>);
      else fail(CL_INVALID_VALUE, "the peak of F32 images only");
   } else if (sqr) {
      aggregate(integral_aggregate<TT, true, VEC, false>);
   } else {
      aggregate(integral_aggregate<TT, false, VEC, false>);
   }
   launch_check("integral_aggregate");
   integral_carries<<<dim3(max(cdiv(W, 64), cdiv(H, 256)), peak ? 4 : 3), 256, 0, s>>>(W, H, aux, peak);
   launch_check("integral_carries");
   char *o = static_cast<char *>(out);
#define OCIP_FINAL(SQ, M) \
   integral_final<TT, SQ, VEC, M><<<grid, kThreads, 0, s>>>(src, W, H, v.step, v.channels, channel, aux, o, ostep)
#define OCIP_FINAL_M(SQ)                                                    \
   if (mode == 2) OCIP_FINAL(SQ, 2);                                        \
   else if (mode == 1) OCIP_FINAL(SQ, 1); else OCIP_FINAL(SQ, 0);
   if (sqr) { OCIP_FINAL_M(true) } else { OCIP_FINAL_M(false) }
#undef OCIP_FINAL_M
#undef OCIP_FINAL
   launch_check("integral_final");
}

void launch_integral(hipStream_t s, const View &v, int channel, bool sqr, void *out, int ostep,
                     int out_type, void *auxp, unsigned *peak)
{
   IntegralAux aux = aux_layout(auxp, v.width, v.height);
   const char *src = static_cast<const char *>(v.ptr);
   const int mode = out_type == SImage::F32 ? 0 : (out_type == SImage::F64 ? 1 : 2);
   const bool vec = v.channels == 1 && v.width >= 4;
   OCIP_TYPE_SWITCH(v.type, TT, {
      if (vec) launch_integral_t<TT, true>(s, src, v, channel, sqr, out, ostep, mode, aux, peak);
      else launch_integral_t<TT, false>(s, src, v, channel, sqr, out, ostep, mode, aux, peak);
   });
}

}  // namespace ocip
