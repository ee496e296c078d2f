// fft.hip -- template matching through 2-D FFTs (the reference's large-template path).
//
// Reference: ImageProximityFFT::{CrossCorr, CrossCorr_Norm, SqrDistance, SqrDistance_Norm}
// (C++/programs/ImageProximityFFT.cpp:115-267) and its kernels
// (cl-files/ImageProximityFFT.cl:55-212): the source is placed at (tw/2, th/2) in a zero image
// of Wb x Hb (W + tw/2, H + th/2 rounded up to a length whose only prime factors are 2, 3
// and 5, ImageProximityFFT.cpp:48-56, FFT.cpp:85-103), the template at (0, 0) in another; the
// correlation is the inverse FFT of FFT(source) * conj(FFT(template)) / (Wb Hb)
// (mulAndScaleSpectrums), cropped to W x H; the Norm ops divide by sqrt(SS TT) with SS the
// window sum of s^2 from the square integral (AreaSqSum) and TT = SumSqr(template).  The
// circular correlation equals the zero-padded one because every wrapped index lands in the
// zero border.
//
// This build computes in FP64 complex arithmetic (the reference uses clFFT in single
// precision and an F32 integral) with its own mixed-radix (2, 3, 4, 5, 8, 9) Stockham FFT in LDS.
// Every image is real, so only the spectrum columns kx <= Wb / 2 are formed and rows travel in
// pairs, two real rows a, b as one complex row a + i b:
//   pass 1 (fft_rows_pair): one workgroup per pair of rows of the source or the template, FFT
//          along x, the two half spectra separated by Hermitian symmetry
//          (A = (Z(k) + conj Z(-k)) / 2, B = (Z(k) - conj Z(-k)) / 2i), written transposed;
//          rows outside the images are never formed;
//   pass 2 (fft_cols): one workgroup per spectrum column kx: FFT along y of the template's column
//          T, then of the source's S, the product conj(S conj T) / (Wb Hb), FFT along y again (an
//          inverse transform of conjugated data), rows y < H written transposed;
//   pass 3 (fft_rows_epi): one workgroup per pair of output rows: their half spectra completed
//          (Q(-k) = conj Q(k)) and packed as Q_a + i Q_b, FFT along x, real and imaginary part the
//          two correlation rows, the epilogue of the op, stored as float.
// Against one complex transform of source + i template over the whole padded image: half the rows
// in passes 1 and 3, three column transforms instead of four, half the intermediate bytes.
#include <algorithm>
#include <cmath>
#include <vector>

#include "device_common.h"

namespace ocip {

namespace {

constexpr int kFftMaxStages = 24;
// one row of complex doubles in the 160 KiB of LDS (less room for static LDS)
constexpr int kFftMaxLen = (160 * 1024 - 256) / 16;
constexpr int kFftThreads = 1024;
// Workgroups of the proximity passes for transforms of up to kFftSmallLen points: 8 wavefronts, two
// on each SIMD, with 128 registers and half a CU's LDS (lengths up to about 4600 with their
// twiddles), so that two workgroups share a CU and one computes while the other waits at a
// barrier or for memory.  4320 points: 278 + 110 + 118 us for the three passes at 4096^2/256x256 (before
// map_at) against 350 + 131 + 162 us with 10 wavefronts (640 threads, one round for a radix-8 stage), whose
// 3 + 3 + 2 + 2 on the SIMDs leaves no room for a second workgroup.  Longer transforms take
// kFftThreads, one workgroup per CU.
constexpr int kFftSmallThreads = 512, kFftSmallLen = kFftMaxLen / 2;

struct FftPlan {
   int n, nstages, twsize;
   int radix[kFftMaxStages];
   int span[kFftMaxStages];   // product of the radices of the earlier stages
   int twoff[kFftMaxStages];  // offset of the stage's twiddles exp(-2 pi i k / (span radix))
};

// q = x / d and r = x mod d for 0 <= x < 2^24, 0 < d, from a float reciprocal corrected by
// one step (the float quotient is within one of the true one)
__device__ __forceinline__ int div_small(int x, int d, float rcp, int &r)
{
   int q = (int)((float)x * rcp);
   r = x - q * d;
   if (r < 0) {
      --q;
      r += d;
   } else if (r >= d) {
      ++q;
      r -= d;
   }
   return q;
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b)
{
   return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
// -i z and +i z
__device__ __forceinline__ double2 mul_mi(double2 z) { return make_double2(z.y, -z.x); }
__device__ __forceinline__ double2 mul_pi(double2 z) { return make_double2(-z.y, z.x); }
__device__ __forceinline__ double2 cscale(double2 z, double s) { return make_double2(z.x * s, z.y * s); }

// Forward DFTs of length R (sign -1) in place.
template <int R> __device__ __forceinline__ void dft(double2 (&u)[R]);

template <> __device__ __forceinline__ void dft<2>(double2 (&u)[2])
{
   const double2 a = u[0], b = u[1];
   u[0] = cadd(a, b);
   u[1] = csub(a, b);
}

template <> __device__ __forceinline__ void dft<3>(double2 (&u)[3])
{
   const double s = 0.86602540378443864676;  // sin(2 pi / 3)
   const double2 a = u[0], t1 = cadd(u[1], u[2]), d = csub(u[1], u[2]);
   const double2 t2 = make_double2(a.x - 0.5 * t1.x, a.y - 0.5 * t1.y);
   const double2 t3 = cscale(mul_mi(d), s);
   u[0] = cadd(a, t1);
   u[1] = cadd(t2, t3);
   u[2] = csub(t2, t3);
}

template <> __device__ __forceinline__ void dft<4>(double2 (&u)[4])
{
   const double2 t0 = cadd(u[0], u[2]), t1 = csub(u[0], u[2]);
   const double2 t2 = cadd(u[1], u[3]), t3 = mul_mi(csub(u[1], u[3]));
   u[0] = cadd(t0, t2);
   u[2] = csub(t0, t2);
   u[1] = cadd(t1, t3);
   u[3] = csub(t1, t3);
}

template <> __device__ __forceinline__ void dft<5>(double2 (&u)[5])
{
   const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;  // cos(2pi/5), cos(4pi/5)
   const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;   // sin(2pi/5), sin(4pi/5)
   const double2 a = u[0];
   const double2 t1 = cadd(u[1], u[4]), t2 = cadd(u[2], u[3]);
   const double2 t3 = csub(u[1], u[4]), t4 = csub(u[2], u[3]);
   const double2 m1 = make_double2(a.x + c1 * t1.x + c2 * t2.x, a.y + c1 * t1.y + c2 * t2.y);
   const double2 m2 = make_double2(a.x + c2 * t1.x + c1 * t2.x, a.y + c2 * t1.y + c1 * t2.y);
   const double2 n1 = make_double2(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y);
   const double2 n2 = make_double2(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y);
   u[0] = make_double2(a.x + t1.x + t2.x, a.y + t1.y + t2.y);
   u[1] = cadd(m1, mul_mi(n1));
   u[4] = cadd(m1, mul_pi(n1));
   u[2] = cadd(m2, mul_mi(n2));
   u[3] = cadd(m2, mul_pi(n2));
}

// 8 points: DFT4 of the even and of the odd inputs, the odd ones times w8^k = exp(-2 pi i k/8)
template <> __device__ __forceinline__ void dft<8>(double2 (&u)[8])
{
   const double r = 0.70710678118654752440;  // 1 / sqrt(2)
   double2 e[4] = {u[0], u[2], u[4], u[6]}, o[4] = {u[1], u[3], u[5], u[7]};
   dft<4>(e);
   dft<4>(o);
   const double2 t[4] = {o[0], make_double2(r * (o[1].x + o[1].y), r * (o[1].y - o[1].x)),
                         mul_mi(o[2]), make_double2(r * (o[3].y - o[3].x), -r * (o[3].x + o[3].y))};
#pragma unroll
   for (int k = 0; k < 4; ++k) {
      u[k] = cadd(e[k], t[k]);
      u[k + 4] = csub(e[k], t[k]);
   }
}

// 9 points: DFT3 over m of x[3m + p] for p = 0, 1, 2, twiddles w9^(p k1), DFT3 over p:
// X[k1 + 3 k2]
template <> __device__ __forceinline__ void dft<9>(double2 (&u)[9])
{
   // w9^1, w9^2, w9^4 with w9 = exp(-2 pi i / 9)
   const double2 w1 = make_double2(0.76604444311897803520, -0.64278760968653932632);
   const double2 w2 = make_double2(0.17364817766693034885, -0.98480775301220805936);
   const double2 w4 = make_double2(-0.93969262078590838405, -0.34202014332566873304);
   double2 a[3][3];
#pragma unroll
   for (int p = 0; p < 3; ++p) {
      double2 v[3] = {u[p], u[p + 3], u[p + 6]};
      dft<3>(v);
      a[p][0] = v[0];
      a[p][1] = v[1];
      a[p][2] = v[2];
   }
   a[1][1] = cmul(a[1][1], w1);
   a[1][2] = cmul(a[1][2], w2);
   a[2][1] = cmul(a[2][1], w2);
   a[2][2] = cmul(a[2][2], w4);
#pragma unroll
   for (int k1 = 0; k1 < 3; ++k1) {
      double2 v[3] = {a[0][k1], a[1][k1], a[2][k1]};
      dft<3>(v);
      u[k1] = v[0];
      u[k1 + 3] = v[1];
      u[k1 + 6] = v[2];
   }
}

// Workgroup barrier that orders LDS only (a full __syncthreads also waits for the
// workgroup's outstanding global loads and stores, which the FFT stages do not need).
__device__ __forceinline__ void lds_barrier()
{
   __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
   __builtin_amdgcn_s_barrier();
   __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One Stockham stage of radix R over nseq sequences of length n stored back to back in LDS:
// butterfly b (k = b mod span) takes x[b + j n/R], multiplies input j by w^(j k),
// w = exp(-2 pi i / (span R)), and writes DFT output j to x[(b - k) R + k + j span].  All
// inputs are read into registers before any output is written (one buffer).
template <int R, int THREADS, int MAXN>
__device__ __forceinline__ void fft_stage(double2 *x, int n, int nseq, int span,
                                          const double2 *__restrict__ tw)
{
   constexpr int MAXB = (MAXN / R + THREADS - 1) / THREADS;
   const int m = n / R, total = m * nseq;
   const float rm = 1.0f / (float)m, rs = 1.0f / (float)span;
   double2 u[MAXB][R];
#pragma unroll
   for (int q = 0; q < MAXB; ++q) {
      const int g = threadIdx.x + q * THREADS;
      if (g < total) {
         int b, k;
         const int seq = nseq == 1 ? (b = g, 0) : div_small(g, m, rm, b);
         div_small(b, span, rs, k);
         const double2 *xs = x + seq * n;
#pragma unroll
         for (int j = 0; j < R; ++j) u[q][j] = xs[b + j * m];
         if (k) {
            const double2 w = tw[k];
            double2 wj = w;
#pragma unroll
            for (int j = 1; j < R; ++j) {
               u[q][j] = cmul(u[q][j], wj);
               if (j + 1 < R) wj = cmul(wj, w);
            }
         }
         dft<R>(u[q]);
      }
   }
   lds_barrier();
#pragma unroll
   for (int q = 0; q < MAXB; ++q) {
      const int g = threadIdx.x + q * THREADS;
      if (g < total) {
         int b, k;
         const int seq = nseq == 1 ? (b = g, 0) : div_small(g, m, rm, b);
         div_small(b, span, rs, k);
         double2 *xs = x + seq * n + (b - k) * R + k;
#pragma unroll
         for (int j = 0; j < R; ++j) xs[j * span] = u[q][j];
      }
   }
   lds_barrier();
}

// Forward FFT (unnormalised) of nseq sequences of length P.n in LDS, natural order in and out;
// tw: the plan's twiddles, in LDS.
// LARGE: the plan may hold radix-8 and radix-9 stages.  THREADS threads, at most MAXN points in all.
template <bool LARGE = false, int THREADS = kFftThreads, int MAXN = kFftMaxLen>
__device__ __forceinline__ void lds_fft(double2 *x, int nseq, const FftPlan *__restrict__ P, const double2 *tw)
{
   const int n = P->n, ns = P->nstages;
   for (int s = 0; s < ns; ++s) {
      const double2 *t = tw + P->twoff[s];
      const int span = P->span[s];
      switch (P->radix[s]) {
      case 2: fft_stage<2, THREADS, MAXN>(x, n, nseq, span, t); break;
      case 3: fft_stage<3, THREADS, MAXN>(x, n, nseq, span, t); break;
      case 4: fft_stage<4, THREADS, MAXN>(x, n, nseq, span, t); break;
      case 8:
         if constexpr (LARGE) fft_stage<8, THREADS, MAXN>(x, n, nseq, span, t);
         break;
      case 9:
         if constexpr (LARGE) fft_stage<9, THREADS, MAXN>(x, n, nseq, span, t);
         break;
      default: fft_stage<5, THREADS, MAXN>(x, n, nseq, span, t); break;
      }
   }
}


// Pitch of the transposed half spectra of h rows: whole 128-byte lines, and one more so that the
// columns of a power-of-two height do not meet in the same cache sets and channels (pass 1 at 4096^2: 161 -> 156 us).
__host__ __device__ constexpr int spectrum_pitch(int h) { return (h + 7) / 8 * 8 + 8; }

// Passes 1 and 2 take their work in XCD-aware order (xcd_tile): the workgroups of one XCD take
// consecutive row pairs or columns, so the transposed stores of neighbours fill the same lines
// of that XCD's L2.
template <bool SMALL> struct FftShape {
   static constexpr int threads = SMALL ? kFftSmallThreads : kFftThreads;
   static constexpr int maxn = SMALL ? kFftSmallLen : kFftMaxLen;
};
// (both shapes come to four wavefronts per SIMD)
#define OCIP_FFT_BOUNDS(SMALL) \
   __launch_bounds__(FftShape<SMALL>::threads) \
       __attribute__((amdgpu_waves_per_eu(4, 4)))

// Pass 1: rows 2 j, 2 j + 1 of the source (j < (H + 1) / 2, at x = tw/2 of the padded row) or,
// after those, of the template (at x = 0), zero elsewhere, FFT along x, both half spectra stored
// transposed: outs[kx * spectrum_pitch(H) + y], outt likewise (32 bytes a column).  The
// template's pairs also leave their FP64 sum of t^2 in tpart.
template <bool SMALL>
__global__ OCIP_FFT_BOUNDS(SMALL) void fft_rows_pair(const char *__restrict__ S, int W, int H,
                                                     int sstep, const char *__restrict__ T, int tw,
                                                     int th, int tstep,
                                                     const FftPlan *__restrict__ pw,
                                                     const double2 *__restrict__ tww,
                                                     double2 *__restrict__ outs,
                                                     double2 *__restrict__ outt,
                                                     double *__restrict__ tpart)
{
   constexpr int THREADS = FftShape<SMALL>::threads;
   extern __shared__ double2 fbuf[];
   const int Wb = pw->n;
   double2 *ltw = fbuf + Wb;
   for (int i = threadIdx.x; i < pw->twsize; i += THREADS) ltw[i] = tww[i];
   const int pairs = (H + 1) / 2, g = xcd_tile(blockIdx.x, gridDim.x);
   const bool tpl = g >= pairs;
   const int y = 2 * (tpl ? g - pairs : g);
   const int w = tpl ? tw : W, h = tpl ? th : H, x0 = tpl ? 0 : tw / 2;
   const char *base = (tpl ? T : S) + (size_t)y * (tpl ? tstep : sstep);
   const float *ra = reinterpret_cast<const float *>(base);
   const bool two = y + 1 < h;   // (a row alone is read twice and counted once)
   const float *rb = two ? reinterpret_cast<const float *>(base + (tpl ? tstep : sstep)) : ra;
   // E elements a thread in flight (unconditional loads, from column 0 outside the row)
   constexpr int E = 4;
   double t2 = 0.0;
#pragma unroll 1
   for (int xb = threadIdx.x; xb < Wb; xb += E * THREADS) {
      float va[E], vb[E];
#pragma unroll
      for (int i = 0; i < E; ++i) {
         const int sx = xb + i * THREADS - x0;
         const int c = sx >= 0 && sx < w ? sx : 0;
         va[i] = ra[c];
         vb[i] = rb[c];
      }
#pragma unroll
      for (int i = 0; i < E; ++i) {
         const int x = xb + i * THREADS, sx = x - x0;
         const bool in = sx >= 0 && sx < w;
         const double a = in ? (double)va[i] : 0.0, b = in && two ? (double)vb[i] : 0.0;
         if (x < Wb) fbuf[x] = make_double2(a, b);
         t2 += a * a + b * b;
      }
   }
   lds_barrier();
   lds_fft<true, THREADS, FftShape<SMALL>::maxn>(fbuf, 1, pw, ltw);
   const int hp = spectrum_pitch(h);
   double2 *out = (tpl ? outt : outs) + y;
   for (int k = threadIdx.x; k <= Wb / 2; k += THREADS) {
      const double2 z = fbuf[k], zc = cconj(fbuf[k == 0 ? 0 : Wb - k]);
      double2 *o = out + (size_t)k * hp;
      o[0] = cscale(cadd(z, zc), 0.5);
      o[1] = cscale(mul_mi(csub(z, zc)), 0.5);
   }
   if (tpl) {
      // the twiddles are not read any more: their LDS takes the waves' sums
      double *red = reinterpret_cast<double *>(fbuf + Wb);
      t2 = wave_sum(t2);
      lds_barrier();
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t2;
      lds_barrier();
      if (threadIdx.x == 0) {
         t2 = 0.0;
         for (int i = 0; i < THREADS / 64; ++i) t2 += red[i];
         tpart[g - pairs] = t2;
      }
   }
}

// Where the map's half spectra between passes 2 and 3 hold row y, column kx: blocks of kMapRows rows, a
// column's values of a block side by side.  Pass 2 stores a column, so a row apart each would be 16 bytes of
// a line, which left L2 before its neighbours' columns filled it (338 MB written for 142 at 4320 points);
// pass 3 reads two rows at a time.  Passes 2 + 3 at 4096^2/256x256: 273 + 116 us with rows apart,
// 265 + 120 with blocks of 2, 249 + 125 of 4, 251 + 152 of 8.
constexpr int kMapRows = 4;
__host__ __device__ constexpr size_t map_at(int y, int kx, int half)
{
   return ((size_t)(y / kMapRows) * half + kx) * kMapRows + y % kMapRows;
}

// Pass 2: spectrum column kx <= Wb / 2: FFT along y of the template's column (at y = 0) and of the
// source's (at y = th/2), the conjugated product, FFT along y again; rows y < H stored
// transposed (map_at).  One column in LDS at a time, the template's spectrum in
// registers meanwhile.
template <bool SMALL>
__global__ OCIP_FFT_BOUNDS(SMALL) void fft_cols(const double2 *__restrict__ ins,
                                                const double2 *__restrict__ inT, int half, int H,
                                                int th, const FftPlan *__restrict__ ph,
                                                const double2 *__restrict__ twh, double scale,
                                                double2 *__restrict__ out)
{
   constexpr int THREADS = FftShape<SMALL>::threads, MAXN = FftShape<SMALL>::maxn;
   constexpr int PER = (kFftSmallLen + THREADS - 1) / THREADS;   // Hb <= kFftSmallLen (fft_sizes)
   extern __shared__ double2 fbuf[];
   const int Hb = ph->n, kx = xcd_tile(blockIdx.x, gridDim.x), cy = th / 2;
   double2 *ltw = fbuf + Hb;
   for (int i = threadIdx.x; i < ph->twsize; i += THREADS) ltw[i] = twh[i];
   const double2 *tc = inT + (size_t)kx * spectrum_pitch(th);
   const double2 *sc = ins + (size_t)kx * spectrum_pitch(H);
   const double2 zero = make_double2(0.0, 0.0);
   for (int y = threadIdx.x; y < Hb; y += THREADS) fbuf[y] = y < th ? tc[y] : zero;
   lds_barrier();
   lds_fft<true, THREADS, MAXN>(fbuf, 1, ph, ltw);
   double2 t[PER];
#pragma unroll
   for (int i = 0; i < PER; ++i) {
      const int y = threadIdx.x + i * THREADS;
      if (y < Hb) {
         t[i] = fbuf[y];
         fbuf[y] = y >= cy && y < H + cy ? sc[y - cy] : zero;   // (its own entry)
      }
   }
   lds_barrier();
   lds_fft<true, THREADS, MAXN>(fbuf, 1, ph, ltw);
#pragma unroll
   for (int i = 0; i < PER; ++i) {
      const int y = threadIdx.x + i * THREADS;
      if (y < Hb) fbuf[y] = cconj(cscale(cmul(fbuf[y], cconj(t[i])), scale));
   }
   lds_barrier();
   lds_fft<true, THREADS, MAXN>(fbuf, 1, ph, ltw);
   for (int y = threadIdx.x; y < H; y += THREADS) out[map_at(y, kx, half)] = fbuf[y];
}

// Pass 3: output rows 2 j and 2 j + 1: FFT along x of Q_a + i Q_b = the two correlation rows, the
// op's epilogue (ImageProximityFFT.cl:86-147, in FP64 with SS from the FP64 integral and
// TT = the sum of the ntpart sums of tpart).
template <bool SMALL>
__global__ OCIP_FFT_BOUNDS(SMALL) void fft_rows_epi(const double2 *__restrict__ in, int half, int W,
                                                    int H, const FftPlan *__restrict__ pw,
                                                    const double2 *__restrict__ tww, int op, int tw,
                                                    int th, const double *__restrict__ integ,
                                                    const double *__restrict__ tpart, int ntpart,
                                                    char *__restrict__ dst, int dstep)
{
   constexpr int THREADS = FftShape<SMALL>::threads;
   extern __shared__ double2 fbuf[];
   const int Wb = pw->n, y = 2 * blockIdx.x;
   const bool two = y + 1 < H;
   double2 *ltw = fbuf + Wb;
   for (int i = threadIdx.x; i < pw->twsize; i += THREADS) ltw[i] = tww[i];
   const double2 *qa = in + map_at(y, 0, half), *qb = two ? qa + 1 : qa;   // (y even: one block)
   {
      constexpr int PER = (FftShape<SMALL>::maxn / 2 + THREADS) / THREADS;
      double2 a[PER], b[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
         const int k = min((int)threadIdx.x + i * THREADS, half - 1);
         a[i] = qa[(size_t)k * kMapRows];
         b[i] = qb[(size_t)k * kMapRows];
      }
#pragma unroll
      for (int i = 0; i < PER; ++i) {
         const int k = threadIdx.x + i * THREADS;
         if (k >= half) break;
         fbuf[k] = cadd(a[i], mul_pi(b[i]));
         if (k > 0 && k < Wb - k) fbuf[Wb - k] = cadd(cconj(a[i]), mul_pi(cconj(b[i])));
      }
   }
   lds_barrier();
   lds_fft<true, THREADS, FftShape<SMALL>::maxn>(fbuf, 1, pw, ltw);
   double tt = 0.0;
   if (op != kCC) {
      // every wavefront sums the parts alike
      for (int i = threadIdx.x & 63; i < ntpart; i += 64) tt += tpart[i];
      tt = wave_sum(tt);
   }
   float *da = reinterpret_cast<float *>(dst + (size_t)y * dstep);
   float *db = reinterpret_cast<float *>(dst + (size_t)(two ? y + 1 : y) * dstep);
   if (op == kCC) {
      for (int x = threadIdx.x; x < W; x += THREADS) {
         const double2 c = fbuf[x];
         da[x] = (float)c.x;
         if (two) db[x] = (float)c.y;
      }
      return;
   }
   // E columns' window sums at a time: all their integral corners in flight
   constexpr int E = 2;
   for (int x0 = threadIdx.x; x0 < W; x0 += E * THREADS) {
      double ss[E][2];
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const int x = min(x0 + e * THREADS, W - 1);
         ss[e][0] = window_sqsum(integ, W, H, x, y, tw, th);
         ss[e][1] = window_sqsum(integ, W, H, x, y + 1, tw, th);
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
         const int x = x0 + e * THREADS;
         if (x >= W) break;
         const double2 c = fbuf[x];
         const double cc[2] = {c.x, c.y};
         float v[2];
#pragma unroll
         for (int r = 0; r < 2; ++r) {
            const double d = op == kCCNorm ? cc[r] : ss[e][r] - 2.0 * cc[r] + tt;
            v[r] = (float)(op == kSSD ? d : d * rsqrt64(ss[e][r] * tt));
         }
         da[x] = v[0];
         if (two) db[x] = v[1];
      }
   }
}

// ---- the generic 2-D FFT (reference FFT::Forward / Inverse, C++/programs/FFT.cpp:140-283):
// real W x H image <-> Hermitian half spectrum (W/2 + 1) x H, complex values interleaved
// (re, im) in F32 or F64, unnormalised both ways (clfftSetPlanScale(..., 1)).  Computed in FP64;
// work holds (W/2 + 1) x H complex doubles, one row per spectrum column kx.

// Forward, pass 1: row y of the real image, FFT along x, columns kx <= W/2 stored transposed.
template <class T>
__global__ __launch_bounds__(kFftThreads) void fft_r2c_rows(const char *__restrict__ src, int sstep,
                                                            int H, const FftPlan *__restrict__ pw,
                                                            const double2 *__restrict__ tww,
                                                            double2 *__restrict__ work)
{
   extern __shared__ double2 fbuf[];
   const int W = pw->n, y = xcd_tile(blockIdx.x, gridDim.x);
   double2 *ltw = fbuf + W;
   for (int i = threadIdx.x; i < pw->twsize; i += kFftThreads) ltw[i] = tww[i];
   const T *row = reinterpret_cast<const T *>(src + (size_t)y * sstep);
   for (int x = threadIdx.x; x < W; x += kFftThreads) fbuf[x] = make_double2((double)row[x], 0.0);
   lds_barrier();
   lds_fft<true>(fbuf, 1, pw, ltw);
   for (int kx = threadIdx.x; kx <= W / 2; kx += kFftThreads) work[(size_t)kx * H + y] = fbuf[kx];
}

// Forward, pass 2: spectrum column kx, FFT along y, stored as row ky, column kx of dst.
template <class T>
__global__ __launch_bounds__(kFftThreads) void fft_r2c_cols(const double2 *__restrict__ work,
                                                            const FftPlan *__restrict__ ph,
                                                            const double2 *__restrict__ twh,
                                                            char *__restrict__ dst, int dstep)
{
   extern __shared__ double2 fbuf[];
   const int H = ph->n, kx = xcd_tile(blockIdx.x, gridDim.x);
   double2 *ltw = fbuf + H;
   for (int i = threadIdx.x; i < ph->twsize; i += kFftThreads) ltw[i] = twh[i];
   for (int y = threadIdx.x; y < H; y += kFftThreads) fbuf[y] = work[(size_t)kx * H + y];
   lds_barrier();
   lds_fft(fbuf, 1, ph, ltw);
   for (int ky = threadIdx.x; ky < H; ky += kFftThreads) {
      T *d = reinterpret_cast<T *>(dst + (size_t)ky * dstep) + 2 * kx;
      d[0] = (T)fbuf[ky].x;
      d[1] = (T)fbuf[ky].y;
   }
}

// Inverse, pass 1: column kx of the half spectrum, inverse FFT along y as the FFT of the
// conjugate; the conjugated result stored as row kx of work.
template <class T>
__global__ __launch_bounds__(kFftThreads) void fft_c2r_cols(const char *__restrict__ src, int sstep,
                                                            const FftPlan *__restrict__ ph,
                                                            const double2 *__restrict__ twh,
                                                            double2 *__restrict__ work)
{
   extern __shared__ double2 fbuf[];
   const int H = ph->n, kx = xcd_tile(blockIdx.x, gridDim.x);
   double2 *ltw = fbuf + H;
   for (int i = threadIdx.x; i < ph->twsize; i += kFftThreads) ltw[i] = twh[i];
   for (int ky = threadIdx.x; ky < H; ky += kFftThreads) {
      const T *v = reinterpret_cast<const T *>(src + (size_t)ky * sstep) + 2 * kx;
      fbuf[ky] = make_double2((double)v[0], -(double)v[1]);
   }
   lds_barrier();
   lds_fft(fbuf, 1, ph, ltw);
   for (int y = threadIdx.x; y < H; y += kFftThreads) work[(size_t)kx * H + y] = fbuf[y];
}

// Inverse, pass 2: row y: the conjugated row spectrum completed by Hermitian symmetry
// (Z(W - kx) = conj Z(kx)), FFT along x, real part stored.
template <class T>
__global__ __launch_bounds__(kFftThreads) void fft_c2r_rows(const double2 *__restrict__ work, int H,
                                                            const FftPlan *__restrict__ pw,
                                                            const double2 *__restrict__ tww,
                                                            char *__restrict__ dst, int dstep)
{
   extern __shared__ double2 fbuf[];
   const int W = pw->n, y = blockIdx.x;
   double2 *ltw = fbuf + W;
   for (int i = threadIdx.x; i < pw->twsize; i += kFftThreads) ltw[i] = tww[i];
   for (int kx = threadIdx.x; kx < W; kx += kFftThreads)
      fbuf[kx] = kx <= W / 2 ? work[(size_t)kx * H + y] : cconj(work[(size_t)(W - kx) * H + y]);
   lds_barrier();
   lds_fft<true>(fbuf, 1, pw, ltw);
   T *row = reinterpret_cast<T *>(dst + (size_t)y * dstep);
   for (int x = threadIdx.x; x < W; x += kFftThreads) row[x] = (T)fbuf[x].x;
}


// Stages for a 2^a 3^b 5^c length, larger radices last (the twiddle table of a stage has span
// entries, so this keeps the table small): LARGE (row plans), radix 8 and 9 where they fit
// (fewer passes through LDS) and 4 / 2 and 3 for what is left; otherwise radices 2 to 5.
// Twiddles appended to `table`, offsets relative to the plan's first entry.
void make_plan(int n, FftPlan &p, std::vector<double2> &table, bool large)
{
   p.n = n;
   p.nstages = 0;
   const int base = (int)table.size();
   int rest = n, span = 1;
   auto add = [&](int r) {
      if (p.nstages >= kFftMaxStages) fail(CL_INVALID_IMAGE_SIZE, "FFT length");
      p.radix[p.nstages] = r;
      p.span[p.nstages] = span;
      p.twoff[p.nstages] = (int)table.size() - base;
      for (int k = 0; k < span; ++k) {
         const long double a = -2.0L * 3.14159265358979323846264338327950288L * k / ((long double)span * r);
         table.push_back(make_double2((double)cosl(a), (double)sinl(a)));
      }
      span *= r;
      rest /= r;
      ++p.nstages;
   };
   int twos = 0, m = n;
   while (m % 2 == 0) {
      m /= 2;
      ++twos;
   }
   if (!large) {
      if (twos % 2) add(2);
      while (rest % 3 == 0) add(3);
      while (rest % 4 == 0) add(4);
      while (rest % 5 == 0) add(5);
      if (rest != 1) fail(CL_INVALID_IMAGE_SIZE, "FFT length with a prime factor above 5");
      p.twsize = (int)table.size() - base;
      return;
   }
   int threes = 0;
   for (int q = m; q % 3 == 0; q /= 3) ++threes;
   // radix 8 and 9 where they fit (fewer LDS passes), 4 / 2 and 3 for the rest
   if (twos % 3 == 1 && twos >= 4) {
      add(4);
      add(4);
      twos -= 4;
   } else if (twos % 3 == 1) {
      add(2);
      twos -= 1;
   } else if (twos % 3 == 2) {
      add(4);
      twos -= 2;
   }
   const int nines = threes / 2;
   for (int k = threes - 2 * nines; k > 0; --k) add(3);
   while (rest % 5 == 0) add(5);
   for (; twos > 0; twos -= 3) add(8);
   for (int k = nines; k > 0; --k) add(9);
   if (rest != 1) fail(CL_INVALID_IMAGE_SIZE, "FFT length with a prime factor above 5");
   p.twsize = (int)table.size() - base;
}

// LDS of a pass: data plus the plan's twiddles, in complex doubles (at least the waves' sums of
// fft_rows_pair); pair_lds: two columns (the path's limit on the padded height)
size_t row_lds(const FftPlan &p) { return (size_t)(p.n + std::max(p.twsize, 8)) * sizeof(double2); }
size_t pair_lds(const FftPlan &p) { return (size_t)(2 * p.n + p.twsize) * sizeof(double2); }

}  // namespace

// FFT.cpp:85-103 IsSupportedLength (multiples of 5 accepted: not an NVIDIA platform)
bool fft_supported_length(int n)
{
   if (n < 1) return false;
   for (int f : {2, 3, 5})
      while (n % f == 0) n /= f;
   return n == 1;
}

// ImageProximityFFT.cpp:48-56
int fft_padded_length(int n)
{
   while (!fft_supported_length(n)) ++n;
   return n;
}

struct FftState {
   int Wb = 0, Hb = 0, hbase = 0;   // hbase: first twiddle of the height plan
   FftPlan pw{}, ph{};
   DevBuf twid, plans, a, b, t, tpart;   // plans: pw and ph, read by the kernels
   ~FftState()
   {
      twid.release();
      plans.release();
      a.release();
      b.release();
      t.release();
      tpart.release();
   }
};

FftState *fft_state_create() { return new FftState(); }
void fft_state_destroy(FftState *s) { delete s; }

cl_int fft_sizes(int W, int H, int tw, int th, int *Wb, int *Hb)
{
   *Wb = fft_padded_length(W + tw / 2);
   *Hb = fft_padded_length(H + th / 2);
   // The reference stops at 2^24 padded points (a clFFT limit, FFT.cpp:170-171); here the
   // limit is LDS: one row of the padded width, or two columns of the padded height, of
   // complex doubles plus the plan's twiddles per workgroup.
   if (*Wb > kFftMaxLen || 2 * *Hb > kFftMaxLen) return CL_INVALID_IMAGE_SIZE;
   std::vector<double2> table;
   FftPlan pw, ph;
   make_plan(*Wb, pw, table, true);
   make_plan(*Hb, ph, table, false);
   if (row_lds(pw) > (size_t)kFftMaxLen * sizeof(double2) ||
       pair_lds(ph) > (size_t)kFftMaxLen * sizeof(double2))
      return CL_INVALID_IMAGE_SIZE;
   return CL_SUCCESS;
}

// Sizes the state's plans and buffers for a W x H source and tw x th template.
void fft_prepare(hipStream_t s, FftState *st, int W, int H, int tw, int th)
{
   int Wb, Hb;
   if (fft_sizes(W, H, tw, th, &Wb, &Hb) != CL_SUCCESS) fail(CL_INVALID_IMAGE_SIZE, "image too big for the FFT path");
   if (st->Wb == Wb && st->Hb == Hb) return;
   std::vector<double2> table;  // the width plan's twiddles, then the height plan's
   make_plan(Wb, st->pw, table, true);
   st->hbase = (int)table.size();
   make_plan(Hb, st->ph, table, true);
   st->twid.ensure(table.size() * sizeof(double2));
   hip_check(hipMemcpyAsync(st->twid.ptr, table.data(), table.size() * sizeof(double2),
                            hipMemcpyHostToDevice, s), "twiddles");
   const FftPlan both[2] = {st->pw, st->ph};
   st->plans.ensure(sizeof(both));
   hip_check(hipMemcpyAsync(st->plans.ptr, both, sizeof(both), hipMemcpyHostToDevice, s), "plans");
   hip_check(hipStreamSynchronize(s), "twiddles");
   // half spectra of the source's and the template's rows (transposed) and of the map's rows, for
   // any image and template of this padded size
   const size_t half = Wb / 2 + 1;
   st->a.ensure(half * spectrum_pitch(Hb) * sizeof(double2));
   st->b.ensure(half * ((Hb + kMapRows - 1) / kMapRows * kMapRows) * sizeof(double2));
   st->t.ensure(half * spectrum_pitch(Hb) * sizeof(double2));
   st->tpart.ensure((size_t)((Hb + 1) / 2) * sizeof(double));
   st->Wb = Wb;
   st->Hb = Hb;
   static bool lds_set = false;
   if (!lds_set) {
      for (const void *k : {reinterpret_cast<const void *>(fft_rows_pair<true>),
                            reinterpret_cast<const void *>(fft_rows_pair<false>),
                            reinterpret_cast<const void *>(fft_cols<true>),
                            reinterpret_cast<const void *>(fft_rows_epi<true>),
                            reinterpret_cast<const void *>(fft_rows_epi<false>)})
         hip_check(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kFftMaxLen * (int)sizeof(double2)),
                   "lds attribute");
      lds_set = true;
   }
}

void launch_proximity_fft(hipStream_t s, FftState *st, int op, const View &S, const View &T,
                          const double *integ, void *dst, int dstep)
{
   fft_prepare(s, st, S.width, S.height, T.width, T.height);
   const int Wb = st->Wb, Hb = st->Hb, half = Wb / 2 + 1;
   const double2 *tww = static_cast<const double2 *>(st->twid.ptr), *twh = tww + st->hbase;
   double2 *a = static_cast<double2 *>(st->a.ptr), *b = static_cast<double2 *>(st->b.ptr);
   double2 *t = static_cast<double2 *>(st->t.ptr);
   double *tpart = static_cast<double *>(st->tpart.ptr);
   const FftPlan *plans = static_cast<const FftPlan *>(st->plans.ptr);
   const int spairs = (S.height + 1) / 2, tpairs = (T.height + 1) / 2;
   const bool small = Wb <= kFftSmallLen;
   const int threads = small ? kFftSmallThreads : kFftThreads;
   {
      KernelTimer kt(s, "fft_rows_pair");
      auto go = [&](auto kernel) {
         kernel<<<spairs + tpairs, threads, row_lds(st->pw), s>>>(
             static_cast<const char *>(S.ptr), S.width, S.height, S.step,
             static_cast<const char *>(T.ptr), T.width, T.height, T.step, plans, tww, a, t, tpart);
      };
      if (small) go(fft_rows_pair<true>); else go(fft_rows_pair<false>);
      launch_check("fft_rows_pair");
   }
   {
      KernelTimer kt(s, "fft_cols");
      fft_cols<true><<<half, kFftSmallThreads, row_lds(st->ph), s>>>(
          a, t, half, S.height, T.height, plans + 1, twh, 1.0 / ((double)Wb * Hb), b);
      launch_check("fft_cols");
   }
   {
      KernelTimer kt(s, "fft_rows_epi");
      auto go = [&](auto kernel) {
         kernel<<<spairs, threads, row_lds(st->pw), s>>>(
             b, half, S.width, S.height, plans, tww, op, T.width, T.height, integ, tpart, tpairs,
             static_cast<char *>(dst), dstep);
      };
      if (small) go(fft_rows_epi<true>); else go(fft_rows_epi<false>);
      launch_check("fft_rows_epi");
   }
}

// ---- generic FFT entry points -------------------------------------------------------------

cl_int fft_plain_sizes(int W, int H)
{
   if (!fft_supported_length(W) || !fft_supported_length(H)) return CL_INVALID_IMAGE_SIZE;
   std::vector<double2> table;
   FftPlan pw, ph;
   make_plan(W, pw, table, true);
   make_plan(H, ph, table, false);
   if (row_lds(pw) > (size_t)kFftMaxLen * sizeof(double2) ||
       row_lds(ph) > (size_t)kFftMaxLen * sizeof(double2))
      return CL_INVALID_IMAGE_SIZE;
   return CL_SUCCESS;
}

// Plans for exactly W x H (no padding) and a (W/2 + 1) x H work buffer.
static void fft_prepare_plain(hipStream_t s, FftState *st, int W, int H)
{
   if (fft_plain_sizes(W, H) != CL_SUCCESS) fail(CL_INVALID_IMAGE_SIZE, "FFT size");
   if (st->Wb == W && st->Hb == H) return;
   std::vector<double2> table;
   make_plan(W, st->pw, table, true);
   st->hbase = (int)table.size();
   make_plan(H, st->ph, table, false);
   st->twid.ensure(table.size() * sizeof(double2));
   hip_check(hipMemcpyAsync(st->twid.ptr, table.data(), table.size() * sizeof(double2),
                            hipMemcpyHostToDevice, s), "twiddles");
   const FftPlan both[2] = {st->pw, st->ph};
   st->plans.ensure(sizeof(both));
   hip_check(hipMemcpyAsync(st->plans.ptr, both, sizeof(both), hipMemcpyHostToDevice, s), "plans");
   hip_check(hipStreamSynchronize(s), "twiddles");
   st->a.ensure((size_t)(W / 2 + 1) * H * sizeof(double2));
   st->Wb = W;
   st->Hb = H;
   static bool lds_set = false;
   if (!lds_set) {
      for (const void *k : {reinterpret_cast<const void *>(fft_r2c_rows<float>),
                            reinterpret_cast<const void *>(fft_r2c_rows<double>),
                            reinterpret_cast<const void *>(fft_r2c_cols<float>),
                            reinterpret_cast<const void *>(fft_r2c_cols<double>),
                            reinterpret_cast<const void *>(fft_c2r_cols<float>),
                            reinterpret_cast<const void *>(fft_c2r_cols<double>),
                            reinterpret_cast<const void *>(fft_c2r_rows<float>),
                            reinterpret_cast<const void *>(fft_c2r_rows<double>)})
         hip_check(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       kFftMaxLen * (int)sizeof(double2)),
                   "lds attribute");
      lds_set = true;
   }
}

void fft_plain_prepare(hipStream_t s, FftState *st, int W, int H) { fft_prepare_plain(s, st, W, H); }

template <class T>
static void fft_forward_t(hipStream_t s, FftState *st, const View &real, const View &cplx)
{
   const int W = real.width, H = real.height;
   const double2 *tww = static_cast<const double2 *>(st->twid.ptr), *twh = tww + st->hbase;
   const FftPlan *plans = static_cast<const FftPlan *>(st->plans.ptr);
   double2 *work = static_cast<double2 *>(st->a.ptr);
   KernelTimer kt(s, "fft_r2c");
   fft_r2c_rows<T><<<H, kFftThreads, row_lds(st->pw), s>>>(static_cast<const char *>(real.ptr),
                                                           real.step, H, plans, tww, work);
   launch_check("fft_r2c_rows");
   fft_r2c_cols<T><<<W / 2 + 1, kFftThreads, row_lds(st->ph), s>>>(
       work, plans + 1, twh, const_cast<char *>(static_cast<const char *>(cplx.ptr)), cplx.step);
   launch_check("fft_r2c_cols");
}

template <class T>
static void fft_inverse_t(hipStream_t s, FftState *st, const View &cplx, const View &real)
{
   const int W = real.width, H = real.height;
   const double2 *tww = static_cast<const double2 *>(st->twid.ptr), *twh = tww + st->hbase;
   const FftPlan *plans = static_cast<const FftPlan *>(st->plans.ptr);
   double2 *work = static_cast<double2 *>(st->a.ptr);
   KernelTimer kt(s, "fft_c2r");
   fft_c2r_cols<T><<<W / 2 + 1, kFftThreads, row_lds(st->ph), s>>>(
       static_cast<const char *>(cplx.ptr), cplx.step, plans + 1, twh, work);
   launch_check("fft_c2r_cols");
   fft_c2r_rows<T><<<H, kFftThreads, row_lds(st->pw), s>>>(
       work, H, plans, tww, const_cast<char *>(static_cast<const char *>(real.ptr)), real.step);
   launch_check("fft_c2r_rows");
}

void launch_fft(hipStream_t s, FftState *st, bool forward, const View &real, const View &cplx)
{
   fft_prepare_plain(s, st, real.width, real.height);
   const bool f64 = real.type == SImage::F64;
   if (forward) {
      if (f64) fft_forward_t<double>(s, st, real, cplx);
      else fft_forward_t<float>(s, st, real, cplx);
   } else {
      if (f64) fft_inverse_t<double>(s, st, cplx, real);
      else fft_inverse_t<float>(s, st, cplx, real);
   }
}

}  // namespace ocip
