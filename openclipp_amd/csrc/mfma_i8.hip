// mfma_i8.hip -- CrossCorr, CrossCorr_Norm, SqrDistance and SqrDistance_Norm of 8- and 16-bit integer
// images on int8 matrix cores, exact whole-number sums throughout.
//
// v_mfma_i32_32x32x32_i8 takes 32 source columns per instruction (a BF16 product takes 16) and adds
// into int32, so sums are exact without flushes.  Values v of source and template become signed bytes
// of v - K,
//   S8   v                                                                         K = 0
//   U8   v - 128                                                                   K = 128
//   S16  v - 128   = 256 h + l, h the high byte, l the low byte - 128              K = 128
//   U16  v - 32896 = 256 h + l, h the high byte - 128, l the low byte - 128        K = 32896
// (pixels outside the image: 0 - K), products of 16-bit types one int32 sum per place, put together
// in FP64 (exact below 2^53).  With s, t now the values less K, n taps, and window sums S1 of s, SS of
// s^2 (window_sums), T1 and TT those of the template:
//   SqrDistance = SS - 2 sum s t + TT   (a difference keeps when both lose K),
//   CrossCorr = sum s t + K S1 + K T1 + K^2 n,
//   and the true sums of squares SS + 2 K S1 + K^2 n, TT + 2 K T1 + K^2 n for the Norm ops.
//
// The contraction is the row-pair one of mfma_kernels.h (crosscorr_mfma_pair) with chunks of 32 source
// columns: MFMA column n = 16 dy + dx, output row Y0 - 1 + 32 w + m + dy,
//   B_kc[k][n] = t(32 kc + k - dx, 2 s + 1 - dy), KC = ceil((tw + 15) / 32),
// 127 output rows by 16 NT columns per workgroup, the whole template's source rows staged at once.
// Lane l of a fragment holds row or column l % 32 and k = 16 (l / 32) + i, i < 16; A and B share
// that order, so any order of the instruction's own gives the same sums.
#include <algorithm>

#include "mfma_kernels.h"

namespace ocip {

namespace {

using mfma::kPairRows;
using mfma::kTileRows;

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef const i32x4 __attribute__((address_space(1))) *gfrag_i8;

constexpr bool is16(int type) { return type == SImage::U16 || type == SImage::S16; }
// digits of a value; its offset K
__host__ __device__ constexpr int i8_digits(int type) { return type == SImage::U16 || type == SImage::S16 ? 2 : 1; }

__host__ __device__ constexpr int i8_key(int type)
{
   return type == SImage::U16 ? 32896 : type == SImage::S8 ? 0 : 128;
}

__host__ __device__ constexpr int i8_chunks(int tw) { return (tw + 15 + 31) / 32; }
__host__ __device__ constexpr int i8_steps(int th) { return (th + 1) / 2; }
// n-tiles of 16 columns per wavefront.  8-bit: two, against four SqrDistance 4096^2/32x32 50 -> 47.6 us,
// colour CrossCorr_Norm 1280x960/24x24 42 -> 33 (twice the wavefronts per SIMD), one 60 and 33.5.
// 16-bit: one, against two CrossCorr_Norm 2048x1536/31x31 60 -> 51 us (48x48 of 4000x3000 233 -> 248).
// (kernel times without the window sums)
__host__ __device__ constexpr int i8_nt(int digits) { return digits == 1 ? 2 : 1; }
__host__ __device__ constexpr int i8_lcols(int digits, int KC) { return 16 * (i8_nt(digits) - 1) + 32 * KC; }

// pitch of the row sums of window_sums over C columns: an odd multiple of 16 bytes (16-byte stores of
// 8 consecutive rows on distinct banks)
__host__ __device__ constexpr int hsum_pitch(int C, int bytes) { return C + 16 / bytes; }

// B fragments (the digits, lowest first) of channel blockIdx.y, one (row pair, chunk) per wavefront;
// the last block the sums of the template less K: sums[2 ch] = TT, sums[2 ch + 1] = T1.
template <int TYPE>
__global__ __launch_bounds__(256) void i8_prep(const char *tpl, int tw, int th, int tstep, int nch,
                                               i32x4 *frag, double *sums)
{
   constexpr int K = i8_key(TYPE), ND = i8_digits(TYPE);
   __shared__ double red[2][4];
   const int ch = blockIdx.y, KC = i8_chunks(tw), S = i8_steps(th);
   if (blockIdx.x == gridDim.x - 1) {
      double s2 = 0.0, s1 = 0.0;
      const int n = tw * th;
      for (int i0 = threadIdx.x; i0 < n; i0 += 256 * 8) {
         int t[8];
#pragma unroll
         for (int k = 0; k < 8; ++k) {
            const int i = min(i0 + 256 * k, n - 1), v = i / tw, u = i - v * tw;
            t[k] = (int)ld<TYPE>(tpl + (size_t)v * tstep, u * nch + ch);
         }
#pragma unroll
         for (int k = 0; k < 8; ++k) {
            const double q = i0 + 256 * k < n ? (double)(t[k] - K) : 0.0;
            s2 += q * q;
            s1 += q;
         }
      }
      s2 = wave_sum(s2);
      s1 = wave_sum(s1);
      if ((threadIdx.x & 63) == 0) {
         red[0][threadIdx.x >> 6] = s2;
         red[1][threadIdx.x >> 6] = s1;
      }
      __syncthreads();
      if (threadIdx.x < 2)
         sums[2 * ch + threadIdx.x] = red[threadIdx.x][0] + red[threadIdx.x][1] + red[threadIdx.x][2] +
                                      red[threadIdx.x][3];
      return;
   }
   const int f = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
   if (f >= S * KC) return;
   const int s = f / KC, kc = f - s * KC;
   const int n = lane & 31, dy = n >> 4, dx = n & 15, kb = 16 * (lane >> 5);
   const int v = 2 * s + 1 - dy;
   const char *row = tpl + (size_t)(v < th ? v : 0) * tstep;
   uint32_t q[ND][4];
#pragma unroll
   for (int p = 0; p < ND; ++p)
#pragma unroll
      for (int i = 0; i < 4; ++i) q[p][i] = 0;
#pragma unroll
   for (int i = 0; i < 16; ++i) {
      const int u = 32 * kc + kb + i - dx;
      int t = (int)ld<TYPE>(row, min(max(u, 0), tw - 1) * nch + ch);   // (in range: all 16 in flight)
      t = v < th && u >= 0 && u < tw ? t - K : 0;
#pragma unroll
      for (int p = 0; p < ND; ++p) {
         const int digit = (int)(int8_t)t;
         q[p][i / 4] |= ((uint32_t)digit & 0xffu) << (8 * (i % 4));
         t = (t - digit) >> 8;
      }
   }
   i32x4 *out = frag + ((size_t)(ch * S * KC + f) * ND) * 64 + lane;
#pragma unroll
   for (int p = 0; p < ND; ++p)
      out[64 * p] = i32x4{(int)q[p][0], (int)q[p][1], (int)q[p][2], (int)q[p][3]};
}

struct I8Args {
   const unsigned char *src;
   int W, H, sstep;
   int tw, th;
   const i32x4 *frag;
   const double *sums;          // i8_prep
   float *dst;
   int dstep, op;
   size_t plane8;               // bytes from one channel's source to the next
   int nch;                     // channels, interleaved in the map
};

// Source rows [row0, row0 + nrows) x columns [col0, col0 + 16 groups) as signed bytes, 16 columns
// per item, at byte pitch ldsp (plane h at `plane` bytes past plane l).
template <int TYPE, int GROUPS>
__device__ __forceinline__ void stage_i8(const I8Args &a, const unsigned char *src, unsigned char *lds,
                                         int ldsp, int plane, int row0, int col0, int nrows)
{
   constexpr bool B16 = is16(TYPE);
   constexpr int DW = B16 ? 8 : 4;   // dwords of 16 elements
   constexpr int K = 4;              // items in flight
   constexpr uint32_t kFlip = 0x80808080u;
   const int total = nrows * GROUPS;
   for (int it0 = threadIdx.x; it0 < total; it0 += 256 * K) {
      uint32_t q[K][DW];
#pragma unroll
      for (int k = 0; k < K; ++k) {
         const int it = it0 + 256 * k, r = it / GROUPS, g = it - r * GROUPS;
         const int sy = row0 + r, sx = col0 + 16 * g;
         const bool rowin = it < total && sy >= 0 && sy < a.H;
         const unsigned char *row = src + (size_t)(rowin ? sy : 0) * a.sstep;
         if (rowin && sx >= 0 && sx + 16 <= a.W) {
#pragma unroll
            for (int j = 0; j < DW / 4; ++j) {
               const u32x4_b b = *reinterpret_cast<const u32x4_b *>(row + sx * (B16 ? 2 : 1) + 16 * j);
#pragma unroll
               for (int e = 0; e < 4; ++e) q[k][4 * j + e] = b[e];
            }
         } else {
#pragma unroll
            for (int j = 0; j < DW; ++j) q[k][j] = 0;
            if (rowin && sx + 16 > 0 && sx < a.W) {
#pragma unroll
               for (int j = 0; j < 16; ++j) {
                  const int x = sx + j;
                  if (x < 0 || x >= a.W) continue;
                  if (B16) q[k][j / 2] |= (uint32_t)reinterpret_cast<const uint16_t *>(row)[x] << (16 * (j % 2));
                  else q[k][j / 4] |= (uint32_t)row[x] << (8 * (j % 4));
               }
            }
         }
      }
#pragma unroll
      for (int k = 0; k < K; ++k) {
         const int it = it0 + 256 * k, r = it / GROUPS, g = it - r * GROUPS;
         if (it >= total) break;
         uint4 *at = reinterpret_cast<uint4 *>(lds + (size_t)r * ldsp + 16 * g);
         if constexpr (B16) {
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
               lo[j] = __builtin_amdgcn_perm(q[k][2 * j + 1], q[k][2 * j], 0x06040200u) ^ kFlip;
               hi[j] = __builtin_amdgcn_perm(q[k][2 * j + 1], q[k][2 * j], 0x07050301u);
               if (TYPE == SImage::U16) hi[j] ^= kFlip;
            }
            *at = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            *reinterpret_cast<uint4 *>(lds + plane + (size_t)r * ldsp + 16 * g) =
                make_uint4(hi[0], hi[1], hi[2], hi[3]);
         } else {
            if (TYPE == SImage::U8) {
#pragma unroll
               for (int j = 0; j < 4; ++j) q[k][j] ^= kFlip;
            }
            *at = make_uint4(q[k][0], q[k][1], q[k][2], q[k][3]);
         }
      }
   }
}

// Window sums of s^2 (SQ) or of s, s less K, from the staged rows: of output column `col` of C, rows
// row0 .. row0 + 128 C / 256 - 1, exact integers.  First the sums over tw columns for every staged
// row and output column (hs), thread = row, running along it; then over th rows, thread = output
// column and a run of rows.  Differences of running sums (squares are only ever added: sums that
// took some off were compiled into byte dot products that added them).  The sums of squares add 12 us
// to the 49 of SqrDistance U8 4096^2/32x32 and save the 23 us of a kernel that wrote them to memory; for
// 16-bit types 4 to 51 (2048x1536/31x31) and the integral's 25.
template <int TYPE, int C, bool SQ, class Sum>
__device__ __forceinline__ void window_sums(const unsigned char *lds, int ldsp, int plane, int nrows,
                                            Sum *hs, int tw, int th, int col, int row0,
                                            Sum (&ss)[kTileRows * C / 256])
{
   constexpr bool B16 = is16(TYPE);
   constexpr int HP = hsum_pitch(C, sizeof(Sum)), kRun = kTileRows * C / 256;
   // four elements
   struct Px { uint32_t l, h; };
   auto dword = [&](const unsigned char *row, int k) {
      Px q;
      q.l = reinterpret_cast<const uint32_t *>(row)[k];
      q.h = B16 ? reinterpret_cast<const uint32_t *>(row + plane)[k] : 0u;
      return q;
   };
   auto add = [&](Sum acc, const Px &q, int e) -> Sum {
      int v = (int)(q.l << (24 - 8 * e)) >> 24;
      if (B16) v += (int)(q.h << (24 - 8 * e)) >> 24 << 8;
      if constexpr (!SQ) return acc + v;
      else if constexpr (B16) return acc + (uint64_t)((uint32_t)abs(v) * (uint32_t)abs(v));
      else return acc + __mul24(v, v);
   };
   for (int r = threadIdx.x; r < nrows; r += 256) {
      const unsigned char *row = lds + (size_t)r * ldsp;
      Sum lead = 0, lag = 0;
      int k = 0;
      for (; 4 * k + 4 <= tw; ++k) {
         const Px q = dword(row, k);
#pragma unroll
         for (int e = 0; e < 4; ++e) lead = add(lead, q, e);
      }
      Px q = dword(row, k);   // (the bytes past the row's last are never used)
#pragma unroll
      for (int e = 0; e < 3; ++e)
         if (e < (tw & 3)) lead = add(lead, q, e);
      Sum *out = hs + (size_t)r * HP;
#pragma unroll
      for (int j = 0; j < C / 4; ++j) {
         // elements tw + 4 j .. of the row enter, elements 4 j .. leave
         const Px n = dword(row, k + j + 1), o = dword(row, j);
         const Px in = {__builtin_amdgcn_alignbyte(n.l, q.l, tw & 3), __builtin_amdgcn_alignbyte(n.h, q.h, tw & 3)};
         q = n;
         Sum w[4];
#pragma unroll
         for (int e = 0; e < 4; ++e) {
            w[e] = lead - lag;
            lead = add(lead, in, e);
            lag = add(lag, o, e);
         }
         int4 *at = reinterpret_cast<int4 *>(out + 4 * j);
         if constexpr (sizeof(Sum) == 8) {
            at[0] = make_int4((int)w[0], (int)(w[0] >> 32), (int)w[1], (int)(w[1] >> 32));
            at[1] = make_int4((int)w[2], (int)(w[2] >> 32), (int)w[3], (int)(w[3] >> 32));
         } else {
            at[0] = make_int4(w[0], w[1], w[2], w[3]);
         }
      }
   }
   __syncthreads();
   const Sum *h = hs + (size_t)row0 * HP + col;
   Sum lead = 0, lag = 0;
   for (int i = 0; i < th - 1; ++i) lead += h[i * HP];
#pragma unroll
   for (int i = 0; i < kRun; ++i) {
      lead += h[(th - 1 + i) * HP];
      ss[i] = lead - lag;
      lag += h[i * HP];
   }
}

__device__ __forceinline__ i32x16 mma_i8(i32x4 a, i32x4 b, i32x16 c)
{
   return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// Bound by latency (staging, window sums, products and epilogue, three or four workgroups per CU over one
// another) above the map's bytes (SqrDistance U8 4096^2/32x32: 55 us in all, 84 MB = 16 us at the copy
// rate, 14 us of MFMA issue) and, for large 16-bit templates, the MFMAs.  Whole calls, against BF16
// products flushed into int32 every few rows and the window sums from a kernel of their own:
// SqrDistance U8 4096^2/32x32 98 -> 55 us, CrossCorr 68 -> 53, /64x64 148 -> 108; against the tile
// kernel's int64 sums and the integral: CrossCorr_Norm U16 2048x1536/31x31 154 -> 46 us.  With the
// template's values whole (a digit more, 256 times 0 or 1) instead of less K and window sums of s:
// CrossCorr U8 66 us (64x64 168), CrossCorr_Norm U16 51.  More wavefronts per SIMD by bounds on the
// registers (3, 4): no faster, spills at 4.
template <int TYPE, int KC>
__global__ __launch_bounds__(256, is16(TYPE) && KC > 2 ? 1 : 2)
void crosscorr_i8(I8Args a, int ldsp, int tiles_x, int tiles)
{
   constexpr bool B16 = is16(TYPE);
   constexpr int ND = i8_digits(TYPE), NL = 2 * ND - 1, K = i8_key(TYPE);   // digits, int32 sums
   constexpr int NT = i8_nt(ND), C = 16 * NT, NA = NT + 2 * KC - 2;
   typedef typename std::conditional<B16, double, int>::type V;   // a half row's cross term
   constexpr int TP = C + (B16 ? 2 : 4);                          // pitch of the paired tile
   extern __shared__ uint4 lds_v[];
   unsigned char *lds = reinterpret_cast<unsigned char *>(lds_v);
   // a tile's channels one after the other on one XCD, whose L2 puts their interleaved stores together
   // (each channel's map in a plane of its own and a kernel to join them: colour CrossCorr_Norm
   // 1280x960/24x24 50 us instead of 38.5, SqrDistance 4096^2/32x32 338 instead of 225)
   const int tc = xcd_tile(blockIdx.x, tiles * a.nch), t = tc / a.nch, ch = tc - t * a.nch;
   const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
   const int x0 = (t % tiles_x) * C, Y0 = (t / tiles_x) * kPairRows;
   const int S = i8_steps(a.th), nrows = kTileRows - 2 + 2 * S, plane = nrows * ldsp;
   const unsigned char *src = a.src + ch * a.plane8;
   char *dst = reinterpret_cast<char *>(a.dst + ch);
   const gfrag_i8 fr = (gfrag_i8)(a.frag + (size_t)ch * S * KC * ND * 64 + lane);
   const double tt = a.sums[2 * ch], t1 = a.sums[2 * ch + 1];

   // LDS row r = source row Y0 - cy + r; wave w reads rows 32 w + m + 2 s
   stage_i8<TYPE, i8_lcols(ND, KC) / 16>(a, src, lds, ldsp, plane, Y0 - a.th / 2, x0 - a.tw / 2, nrows);
   __syncthreads();
   // the op's window sums, in registers until the epilogue: thread = output column `col`, kRun rows
   // from `row0` on
   constexpr int kRun = kTileRows * C / 256;
   const int col = threadIdx.x % C, row0 = threadIdx.x / C * kRun;
   typedef typename std::conditional<B16, uint64_t, int>::type Sum;
   Sum ss[kRun];
   int s1[kRun];
   unsigned char *hs = lds + ND * plane;
   if (a.op != kCC)
      window_sums<TYPE, C, true>(lds, ldsp, plane, nrows, reinterpret_cast<Sum *>(hs), a.tw, a.th, col, row0, ss);
   if (K && a.op != kSSD) {
      __syncthreads();
      window_sums<TYPE, C, false>(lds, ldsp, plane, nrows, reinterpret_cast<int *>(hs), a.tw, a.th, col, row0, s1);
   }

   i32x16 acc[NL][NT];
#pragma unroll
   for (int l = 0; l < NL; ++l)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int i = 0; i < 16; ++i) acc[l][j][i] = 0;
   // (a wave whose output rows all lie below the image has nothing to multiply)
   if (Y0 - 1 + 32 * wave < a.H) {
      i32x4 b[2][KC][ND];
      auto fetch = [&](int s, i32x4 (&q)[KC][ND]) {
#pragma unroll
         for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int p = 0; p < ND; ++p) q[kc][p] = fr[(size_t)((s * KC + kc) * ND + p) * 64];
      };
      const unsigned char *arow = lds + (size_t)(wave * 32 + (lane & 31)) * ldsp + 16 * (lane >> 5);
      auto step = [&](int s, const i32x4 (&q)[KC][ND]) {
         i32x4 x[ND][NA];
#pragma unroll
         for (int c = 0; c < NA; ++c)
#pragma unroll
            for (int p = 0; p < ND; ++p)
               x[p][c] = *reinterpret_cast<const i32x4 *>(arow + p * plane + (size_t)(2 * s) * ldsp + 16 * c);
#pragma unroll
         for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int k = 0; k < ND * ND; ++k) {
               // digit of s, digit of t: (l, l), (h, l), (h, h), (l, h)
               constexpr int kA[4] = {0, 1, 1, 0}, kB[4] = {0, 0, 1, 1};
#pragma unroll
               for (int j = 0; j < NT; ++j)
                  acc[kA[k] + kB[k]][j] = mma_i8(x[kA[k]][j + 2 * kc], q[kc][kB[k]], acc[kA[k] + kB[k]][j]);
            }
      };
      fetch(0, b[0]);
      int s = 0;
      for (; s + 1 < S; s += 2) {
         // keep each prefetch ahead of the MFMAs of the step before it
         fetch(s + 1, b[1]);
         __builtin_amdgcn_sched_barrier(0);
         step(s, b[0]);
         fetch(min(s + 2, S - 1), b[0]);
         __builtin_amdgcn_sched_barrier(0);
         step(s + 1, b[1]);
      }
      if (s < S) step(s, b[0]);
   }

   // Pair the halves in LDS: tile row r = 32 w + m + dy holds output row Y0 - 1 + r; C fragment: lane
   // holds column n = lane % 32, rows m = 8 (i / 4) + 4 (lane / 32) + i % 4.
   V *tile = reinterpret_cast<V *>(lds);
   const int n = lane & 31, dy = n >> 4, dx = n & 15;
   const int rb = 32 * wave + 4 * (lane >> 5) + dy;
   auto half = [&](int j, int i) -> V {
      V v = (V)acc[NL - 1][j][i];
#pragma unroll
      for (int l = NL - 2; l >= 0; --l) v = v * (V)256 + (V)acc[l][j][i];
      return v;
   };
   __syncthreads();
   if (dy) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int i = 0; i < 16; ++i) tile[(rb + 8 * (i / 4) + (i % 4)) * TP + 16 * j + dx] = half(j, i);
   }
   __syncthreads();
   if (!dy) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int i = 0; i < 16; ++i) tile[(rb + 8 * (i / 4) + (i % 4)) * TP + 16 * j + dx] += half(j, i);
   }
   __syncthreads();
   // (whole numbers throughout, below 2^31 or 2^53)
   const V n1 = (V)(a.tw * a.th), vtt = (V)tt, kt = K * (V)t1 + K * n1 * K;
   const double ttrue = tt + 2.0 * K * t1 + (double)K * K * (double)(a.tw * a.th);
   const int x = x0 + col;
   if (x >= a.W) return;
#pragma unroll
   for (int i = 0; i < kRun; ++i) {
      const int r = row0 + i, y = Y0 + r;
      if (r >= kPairRows || y >= a.H) continue;
      const V cross = tile[(r + 1) * TP + col];
      V d;
      if (a.op == kSSD || a.op == kSSDNorm) d = (V)ss[i] - 2 * cross + vtt;
      else d = cross + (K ? K * (V)s1[i] : (V)0) + kt;
      float v = (float)d;
      if (a.op == kSSDNorm || a.op == kCCNorm) {
         const V sst = (V)ss[i] + (K ? 2 * K * (V)s1[i] + K * n1 * K : (V)0);
         v = (float)((double)d * rsqrt64((double)sst * ttrue));
      }
      reinterpret_cast<float *>(dst + (size_t)y * a.dstep)[x * a.nch] = v;
   }
}

template <int TYPE>
void launch_i8(hipStream_t s, I8Args a, const View &S, const View &T)
{
   constexpr int ND = i8_digits(TYPE), NT = i8_nt(ND);
   constexpr bool B16 = is16(TYPE);
   a.src = static_cast<const unsigned char *>(S.ptr);
   a.W = S.width; a.H = S.height; a.sstep = S.step;
   a.tw = T.width; a.th = T.height;
   a.nch = T.channels;
   const int KC = i8_chunks(a.tw), steps = i8_steps(a.th), nch = T.channels;
   {
      KernelTimer kt(s, "template_prep");
      i8_prep<TYPE><<<dim3((steps * KC + 3) / 4 + 1, nch), 256, 0, s>>>(
          static_cast<const char *>(T.ptr), a.tw, a.th, T.step, nch, const_cast<i32x4 *>(a.frag),
          const_cast<double *>(a.sums));
      launch_check("i8_prep");
   }
   // an odd multiple of 16 bytes: the A reads of 8 consecutive rows on distinct banks
   int ldsp = i8_lcols(ND, KC);
   if (ldsp % 32 == 0) ldsp += 16;
   const int nrows = kTileRows - 2 + 2 * steps;
   const int sum = B16 && a.op != kCC ? 8 : 4;
   const size_t sums = (size_t)(nrows + 1) * hsum_pitch(16 * NT, sum) * sum;
   const size_t staging = (size_t)ND * nrows * ldsp + (a.op == kCC && i8_key(TYPE) == 0 ? 0 : sums);
   const size_t pairing = (size_t)(kTileRows + 1) * (16 * NT + (B16 ? 2 : 4)) * (B16 ? 8 : 4);
   const size_t lds = std::max(staging, pairing);
   const int tiles_x = (a.W + 16 * NT - 1) / (16 * NT), tiles_y = (a.H + kPairRows - 1) / kPairRows;
   KernelTimer kt(s, "crosscorr_mfma_int");
   auto go = [&](auto kernel) {
      if (lds > 64 * 1024)
         hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                   "lds attribute");
      kernel<<<tiles_x * tiles_y * nch, 256, lds, s>>>(a, ldsp, tiles_x, tiles_x * tiles_y);
   };
   switch (KC) {
   case 1: go(crosscorr_i8<TYPE, 1>); break;
   case 2: go(crosscorr_i8<TYPE, 2>); break;
   case 3: go(crosscorr_i8<TYPE, 3>); break;
   case 4: go(crosscorr_i8<TYPE, 4>); break;
   default: fail(CL_INVALID_VALUE, "template width");
   }
   launch_check("crosscorr_i8");
}

// ------------------------------------------------------------------------- planes
// Interleaved 8-bit channels into planes of their own (row pitch plane8_step, plane pitch H rows),
// zeros between the width and the pitch: the kernels after it take every channel of an image in one
// launch, as 1-channel images with wide loads.  Four pixels per thread.  Bound by HBM: 2 W H NCH
// bytes.
int plane8_step(int W) { return (W + 15) / 16 * 16; }

template <int NCH>
__global__ __launch_bounds__(256) void split_planes8(const unsigned char *__restrict__ src, int W,
                                                     int H, int sstep,
                                                     unsigned char *__restrict__ dst, int dstep)
{
   const int k = blockIdx.x * 256 + threadIdx.x, groups = dstep / 4;
   const int y = k / groups, x = 4 * (k - y * groups);
   if (y >= H) return;
   const unsigned char *row = src + (size_t)y * sstep;
   uint32_t q[NCH];   // the 4 NCH bytes of the thread's pixels
   if (x + 4 <= W) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) q[i] = reinterpret_cast<const u32_b *>(row + x * NCH)[i];
   } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i) q[i] = 0;
#pragma unroll
      for (int i = 0; i < 4 * NCH; ++i)
         if (x + i / NCH < W) q[i / 4] |= (uint32_t)row[x * NCH + i] << (8 * (i % 4));
   }
#pragma unroll
   for (int c = 0; c < NCH; ++c) {
      uint32_t v = 0;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
         const int i = p * NCH + c;
         v |= (q[i / 4] >> (8 * (i % 4)) & 0xffu) << (8 * p);
      }
      *reinterpret_cast<uint32_t *>(dst + ((size_t)c * H + y) * dstep + x) = v;
   }
}

static unsigned plane_blocks(int H, int step) { return (unsigned)(((long long)H * (step / 4) + 255) / 256); }

}  // namespace

size_t planes8_bytes(const View &S)
{
   return S.channels > 1 ? (size_t)S.channels * S.height * plane8_step(S.width) : 0;
}

View launch_planes8(hipStream_t s, const View &image, void *planes, size_t *plane8)
{
   KernelTimer kt(s, "split_planes8");
   View S = image;
   S.ptr = planes;
   S.step = plane8_step(image.width);
   S.channels = 1;
   *plane8 = (size_t)S.height * S.step;
   auto go = [&](auto kernel) {
      kernel<<<plane_blocks(S.height, S.step), 256, 0, s>>>(
          static_cast<const unsigned char *>(image.ptr), S.width, S.height, image.step,
          static_cast<unsigned char *>(planes), S.step);
   };
   if (image.channels == 2) go(split_planes8<2>); else go(split_planes8<4>);
   launch_check("split_planes8");
   return S;
}

bool int_mfma_ok(int op, const View &S, const View &T)
{
   const char *e = getenv("OCIP_INT_MFMA");
   if ((e && e[0] == '0') || op == kSAD) return false;
   if ((S.type != SImage::U8 && S.type != SImage::S8) || T.type != S.type) return false;
   if (S.channels != 1 && S.channels != 2 && S.channels != 4) return false;
   const int tw = T.width, th = T.height;
   if (tw <= 0 || th <= 0 || i8_chunks(tw) > 4 || th > 128) return false;
   // the whole sum in int32
   return (long long)tw * th * (S.type == SImage::U8 ? 255 * 255 : 128 * 128) < (1LL << 31);
}

// Sums (two per channel), then the fragments of every channel (two digits at most).
constexpr size_t kSumsBytes = 256;

size_t i8_work_bytes(const View &T)
{
   const size_t n = 2 * (size_t)T.channels * i8_steps(T.height) * i8_chunks(T.width) * 64 * sizeof(i32x4);
   return kSumsBytes + (n + 255) / 256 * 256;
}

size_t int_mfma_work_bytes(const View &S, const View &T)
{
   return i8_work_bytes(T) + planes8_bytes(S);
}

static I8Args work_args(int op, void *work)
{
   I8Args a{};
   a.sums = static_cast<const double *>(work);
   a.frag = reinterpret_cast<const i32x4 *>(static_cast<const char *>(work) + kSumsBytes);
   a.op = op;
   return a;
}

void launch_int_mfma(hipStream_t s, int op, const View &image, const View &T, float *dst, int dstep,
                     void *work)
{
   const int nch = image.channels;
   // S: the image or (several channels) its first plane, the others plane8 bytes apart
   View S = image;
   I8Args a = work_args(op, work);
   a.dst = dst;
   a.dstep = dstep;
   if (nch > 1) S = launch_planes8(s, image, static_cast<char *>(work) + i8_work_bytes(T), &a.plane8);
   if (T.type == SImage::S8) launch_i8<SImage::S8>(s, a, S, T);
   else launch_i8<SImage::U8>(s, a, S, T);
}

// Every size up to the widest template of four chunks: against the tile kernel, CrossCorr 160x120/2x2
// 9.9 -> 9.0 us, 640x480/3x3 11.2 -> 10.5, 4096^2/8x8 120 -> 75, /64x64 2428 -> 358; SqrDistance
// 160x120/4x4 11.3 -> 9.4, 2048x1536/31x31 192 -> 49.  (The height keeps the staged rows and their
// sums within the LDS and the products within int32.)
bool int16_mfma_ok(int op, const View &S, const View &T)
{
   const char *e = getenv("OCIP_INT_MFMA");
   if ((e && e[0] == '0') || op == kSAD) return false;
   if (!is16(S.type) || T.type != S.type || S.channels != 1) return false;
   return T.width > 0 && T.height > 0 && i8_chunks(T.width) <= 4 && T.height <= 128;
}

void launch_int16_mfma(hipStream_t s, int op, const View &S, const View &T, float *dst, int dstep, void *work)
{
   I8Args a = work_args(op, work);
   a.dst = dst;
   a.dstep = dstep;
   if (S.type == SImage::U16) launch_i8<SImage::U16>(s, a, S, T);
   else launch_i8<SImage::S16>(s, a, S, T);
}

}  // namespace ocip
