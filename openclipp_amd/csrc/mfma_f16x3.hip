// CrossCorr_Norm of F32 images on split-FP16 MFMA: instances of the row-pair kernel.
#include "mfma_kernels.h"

namespace ocip {
namespace mfma {

namespace {

// Fragments of a split-FP16 template, one per wavefront of the first fblocks workgroups (the sum of
// squares and the peaks come from template_prep), and *any cleared; then one wavefront per tile:
// whether one of 64 outputs of it, 8 columns and 16 rows apart, has a window that the split or the
// integral may not hold (the line of pair_tile's doubt).
__global__ __launch_bounds__(256) void split_prep(BatchDesc d, TileArgs a, int fblocks, int tiles_x, int tiles)
{
   if (blockIdx.x == 0 && threadIdx.x == 0) *a.any = 0u;
   const SplitRange sr = split_range(a.peaks, d.tw * d.th);
   if (!sr.ok) return;
   const int lane = threadIdx.x & 63;
   if ((int)blockIdx.x < fblocks) {
      const int f = blockIdx.x * 4 + (threadIdx.x >> 6);
      if (f < pair_frag_steps(d.th, 1) * d.KC)
         build_pair_fragment<kF16x3>(d.tptr, d.tstep, d.tw, d.th, d.KC, 1, f, lane, d.frag0, d.frag1,
                                     pow2f(sr.kt));
      return;
   }
   const int t = (blockIdx.x - fblocks) * 4 + (threadIdx.x >> 6);
   if (t >= tiles) return;
   const int x = t % tiles_x * (16 * kSplitNT) + 8 * (lane & 7), y = t / tiles_x * kPairRows + 16 * (lane >> 3);
   bool doubt = false;
   if (x < a.W && y < a.H) {
      const double last = a.integ[(size_t)min(y - a.th / 2 + a.th, a.H) * excl_pitch(a.W) + kExclOffset +
                                  min(x - a.tw / 2 + a.tw, a.W)];
      const double ss = window_sqsum(a.integ, a.W, a.H, x, y, a.tw, a.th);
      doubt = !(ss >= sr.least_ss) || !(ss >= a.ill * last);
   }
   doubt = __any(doubt);
   if (lane == 0) a.flags[t] = (unsigned)doubt;
}

template <int KC, bool LOLO> void pair(hipStream_t s, const SingleLaunch &L)
{
   auto k = crosscorr_mfma_pair<kF16x3, KC, kSplitNT, kModeNCC, LOLO>;
   // set for every call: the attribute belongs to the device that is current
   hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax),
             "lds attribute");
   const int tiles = L.grid.x * L.grid.y;
   k<<<tiles, 256, L.lds, s>>>(L.a, L.ldsp, (int)L.grid.x, tiles, L.z);
}

}  // namespace

template <bool LOLO> static void pairs(hipStream_t s, const SingleLaunch &L)
{
   switch (L.KC) {
   case 1: pair<1, LOLO>(s, L); break;
   case 2: pair<2, LOLO>(s, L); break;
   case 3: pair<3, LOLO>(s, L); break;
   case 4: pair<4, LOLO>(s, L); break;
   case 5: pair<5, LOLO>(s, L); break;
   case 6: pair<6, LOLO>(s, L); break;
   case 7: pair<7, LOLO>(s, L); break;
   default: fail(CL_INVALID_VALUE, "template width");
   }
}

// lo lo (pair_mfma_f16x3) is taken below kLoLoTaps taps.  It matters where all of a window's lo are alike:
// constant images of 1 + 2^-11 are off by 7e-8 with it (8x8 to 24x24) and 2.4e-7 without, FP32 sums by
// 1.2e-7 to 2e-7.  With more taps the roundings of FP32 sums have long outgrown its 2^-22 (constant images
// at 32x32, root mean square 5.4e-6 against 3.2e-7; noise 3.7e-7 against 8.4e-8), and a fourth product
// costs 19 percent of 4096^2/64x64 (556 -> 663 us) against 4 of 4000x2000/31x31 (157 -> 164).
constexpr int kLoLoTaps = 1024;

void launch_split_pair(hipStream_t s, const SingleLaunch &L)
{
   if (L.a.tw * L.a.th < kLoLoTaps) pairs<true>(s, L); else pairs<false>(s, L);
   launch_check("crosscorr_mfma_split");
}

void launch_split_prep(hipStream_t s, const BatchDesc &d, const TileArgs &a, int tiles_x, int tiles)
{
   const int nfrag = pair_frag_steps(d.th, 1) * d.KC, fblocks = (nfrag + 3) / 4;
   split_prep<<<fblocks + (tiles + 3) / 4, 256, 0, s>>>(d, a, fblocks, tiles_x, tiles);
   launch_check("split_prep");
}

}  // namespace mfma
}  // namespace ocip
