// CrossCorr_Norm of F32 images on split-FP16 MFMA: instances of the row-pair kernel.
#include "mfma_kernels.h"

namespace ocip {
namespace mfma {

namespace {

// Fragments of a split-FP16 template, one per wavefront (the sum of squares and the peaks come
// from template_prep), and *any cleared.
__global__ __launch_bounds__(256) void split_prep(BatchDesc d, const unsigned *__restrict__ peaks,
                                                   unsigned *any)
{
   if (blockIdx.x == 0 && threadIdx.x == 0) *any = 0u;
   const SplitRange sr = split_range(peaks, d.tw * d.th);
   const int nfrag = pair_frag_steps(d.th, 1) * d.KC;
   const int f = blockIdx.x * 4 + (threadIdx.x >> 6);
   if (f < nfrag && sr.ok)
      build_pair_fragment<kF16x3>(d.tptr, d.tstep, d.tw, d.th, d.KC, 1, f, threadIdx.x & 63,
                                  d.frag0, d.frag1, pow2f(sr.kt));
}

template <int KC> void pair(hipStream_t s, const SingleLaunch &L)
{
   auto k = crosscorr_mfma_pair<kF16x3, KC, 4, kModeNCC>;
   // set for every call: the attribute belongs to the device that is current
   hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax),
             "lds attribute");
   const int tiles = L.grid.x * L.grid.y;
   k<<<tiles, 256, L.lds, s>>>(L.a, L.ldsp, (int)L.grid.x, tiles, L.z);
}

}  // namespace

void launch_split_pair(hipStream_t s, const SingleLaunch &L)
{
   switch (L.KC) {
   case 1: pair<1>(s, L); break;
   case 2: pair<2>(s, L); break;
   case 3: pair<3>(s, L); break;
   case 4: pair<4>(s, L); break;
   case 5: pair<5>(s, L); break;
   case 6: pair<6>(s, L); break;
   case 7: pair<7>(s, L); break;
   default: fail(CL_INVALID_VALUE, "template width");
   }
   launch_check("crosscorr_mfma_split");
}

void launch_split_prep(hipStream_t s, const BatchDesc &d, const unsigned *peaks, unsigned *any)
{
   const int nfrag = pair_frag_steps(d.th, 1) * d.KC;
   split_prep<<<(nfrag + 3) / 4, 256, 0, s>>>(d, peaks, any);
   launch_check("split_prep");
}

}  // namespace mfma
}  // namespace ocip
