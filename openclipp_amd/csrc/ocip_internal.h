// Internal declarations shared by the C-ABI layer (capi.cpp) and the HIP kernels.
//
// Object model (reference equivalents in brackets):
//   Context  [COpenCL, C++/OpenCL.cpp:48-69]  one GPU + one in-order HIP stream, plus the
//            device workspaces the proximity ops reuse between calls.
//   Image    [Image/Buffer, C++/Image.cpp:147-165, C++/Buffer.cpp:100-194]  Height*Step
//            bytes of device memory, the caller's host pointer (not copied), an in-device flag.
//   Program  [Integral / Statistics programs, include/c++/Programs/Integral.h:32-61]
//            scratch buffers owned by an ocipProgram handle.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include <string>
#include <vector>

#include "OpenCLIPP.h"

#ifndef CL_INVALID_BUFFER_SIZE
#define CL_INVALID_BUFFER_SIZE -61
#endif

namespace ocip {

// An error raised anywhere below the C ABI; the ABI layer returns `code`.
struct Error {
   cl_int code;
   const char *what;
};

[[noreturn]] inline void fail(cl_int code, const char *what) { throw Error{code, what}; }

// Failing HIP call: the error is mapped to an OpenCL code; with OCIP_VERBOSE set in the
// environment the HIP error text is printed to stderr.
void report_hip_error(hipError_t e, const char *what);
inline void hip_check(hipError_t e, const char *what)
{
   if (e != hipSuccess) {
      report_hip_error(e, what);
      fail(e == hipErrorOutOfMemory ? CL_MEM_OBJECT_ALLOCATION_FAILURE : CL_OUT_OF_RESOURCES, what);
   }
}

// Growable device buffer (contents are not preserved by `ensure`).
struct DevBuf {
   void *ptr = nullptr;
   size_t bytes = 0;
   void ensure(size_t n);
   void release();
   template <class T> T *as() const { return static_cast<T *>(ptr); }
};

struct Context;
struct BatchCache;

enum : uint32_t { kImageMagic = 0x474d494fu /*OIMG*/, kContextMagic = 0x5854434fu /*OCTX*/,
                  kProgramMagic = 0x4752504fu /*OPRG*/ };

// desc describes the device image the kernels see.  A 3-channel (colour) image is held on
// the device as 4 channels with the fourth set to 255 (reference ColorImage,
// C++/Image.cpp:243-275): host_desc keeps the caller's 3-channel layout, `stage` a device copy
// of it, and transfers convert between the two.
struct Image {
   uint32_t magic = kImageMagic;
   Context *ctx = nullptr;
   SImage desc{};
   SImage host_desc{};
   void *host = nullptr;
   void *dev = nullptr;
   void *stage = nullptr;   // colour images only
   size_t bytes = 0;        // bytes of the host image (Height * host Step)
   bool in_device = false;
};

// Colour conversions between the 3-channel host layout and the 4-channel device layout.
void launch_copy3to4(hipStream_t s, int type, const void *src, int sstep, void *dst, int dstep,
                     int width, int height);
void launch_copy4to3(hipStream_t s, int type, const void *src, int sstep, void *dst, int dstep,
                     int width, int height);

enum ProgramKind { kProgIntegral = 1, kProgStatistics = 2, kProgProximityFFT = 3, kProgFFT = 4 };

struct FftState;
FftState *fft_state_create();
void fft_state_destroy(FftState *s);

struct Program {
   uint32_t magic = kProgramMagic;
   Context *ctx = nullptr;
   int kind = 0;
   DevBuf scratch;
   FftState *fft = nullptr;   // kProgProximityFFT, kProgFFT: plans, twiddles, work buffers
};

// Per-template data the proximity kernels read: the template as F32 (or F64 / int32)
// with zero-padded rows, plus FP64 sum of squares.
struct TemplateBuf {
   DevBuf data;      // th rows x pitch elements
   DevBuf sums;      // [0] = sum t^2 (double), [1] = sum t (double)
};

constexpr size_t kHostOutBytes = 16 * 1024;

struct Context {
   uint32_t magic = kContextMagic;
   int device = 0;
   hipStream_t stream = nullptr;
   std::string name;
   int num_cus = 0;
   TemplateBuf tmpl;      // template staging for the single-template ops
   DevBuf integ;          // FP64 exclusive sum-of-squares integral, (W+1) x (H+1)
   DevBuf integ_aux;      // integral scan aggregates
   DevBuf stats;          // reduction partials for MinIndx / MaxIndx, MFMA fragments
   DevBuf work;           // gradient workspace
   void *host_out = nullptr;   // kHostOutBytes of pinned memory that reductions leave results in
   BatchCache *batch = nullptr;  // recorded batch graphs (mfma.hip)
};

// Kernel timing: construct before a launch, destroy after it.  Records a HIP event pair on
// `s` when timing is enabled (ocipEnableKernelTiming), nothing otherwise.
// While suspended (stream capture), no timing events are recorded.
void timing_suspend(bool suspend);
struct KernelTimer {
   KernelTimer(hipStream_t s, const char *name);
   ~KernelTimer();
   hipStream_t stream;
   const char *name;
   void *start = nullptr;
};

// ---------------------------------------------------------------------------------------
// Element types (SImage::EDataType)
inline int elem_size(int t)
{
   switch (t) {
   case SImage::U8: case SImage::S8: return 1;
   case SImage::U16: case SImage::S16: return 2;
   case SImage::U32: case SImage::S32: case SImage::F32: return 4;
   case SImage::F64: return 8;
   default: return 0;
   }
}
inline bool is_float(int t) { return t == SImage::F32 || t == SImage::F64; }
inline bool is_unsigned(int t) { return t == SImage::U8 || t == SImage::U16 || t == SImage::U32; }

// Proximity operations
enum ProxOp { kSSD = 0, kSSDNorm = 1, kSAD = 2, kCC = 3, kCCNorm = 4 };

// A device image view handed to kernel launchers.
struct View {
   const void *ptr;
   int width, height, step;   // step in bytes
   int channels, type;
};

// Internal exclusive FP64 integral (window sums for the Norm ops and gradients): H+1 rows of
// excl_pitch(W) doubles; entry (j, i) = sum over rows < j and columns < i (0 <= i <= W)
// sits at j * pitch + i + kExclOffset, so that entries 1..W of a row start on a 32-byte
// boundary and a row is written with full 32-byte stores.
constexpr int kExclOffset = 3;
__host__ __device__ inline size_t excl_pitch(int W) { return ((size_t)W + kExclOffset + 1 + 3) / 4 * 4; }
inline size_t excl_bytes(int W, int H) { return excl_pitch(W) * ((size_t)H + 1) * sizeof(double); }

// ---------------------------------------------------------------------------------------
// Kernel launchers (defined in the .hip files).  All enqueue on `s` and return immediately.

// Integral of f(src) with f = identity or square, FP64 sums.
//   out_type F32/F64 with inclusive same-size layout (public API), or
//   out_type = -1: the internal exclusive layout above (out_step ignored).
size_t integral_aux_bytes(int width, int height);
// peak (sqr of F32 images, may be null): receives the high word of the largest f.
void launch_integral(hipStream_t s, const View &src, int channel, bool sqr, void *out,
                     int out_step, int out_type, void *aux, unsigned *peak = nullptr);

// Template staging: converts the template to the kernels' compute type with a row pitch of
// `pitch` elements (zero padding), and writes FP64 sum(t^2), sum(t) to sums[0..1].
// kind 0: float, 1: double, 2: int32.  peak (may be null): receives the high word of the largest
// t^2 in FP64.
void launch_template_prep(hipStream_t s, const View &tpl, int channel, int pitch, int kind,
                          void *out, double *sums, unsigned *peak = nullptr);

// Plain (VALU) proximity for any type/channel count.  `integ` is the exclusive FP64
// sum-of-squares integral of the source for the Norm ops (null for the others).
void launch_proximity(hipStream_t s, int op, const View &src, const View &tpl, void *dst,
                      int dst_step, const void *tstage, int tpitch, const double *tsums,
                      const double *integ, int channel);
// 1-channel F32 templates that launch_proximity reads in place (tstage = the image, tpitch its
// pitch in floats, tsums null): no staging launch.
bool prox_template_in_place(int op, const View &src, const View &tpl, bool have_integral);
// The plain Norm ops on F32 sources whose template fits one LDS band form the window sums
// of s^2 inside the tile kernel (launch_proximity with no integral)
bool prox_norm_from_tile(int op, const View &src, const View &tpl);

// CrossCorr_Norm of F32 1-channel images on split-FP16 MFMA (as accurate as the FP32 sums of
// launch_proximity, mfma_kernels.h): split_ncc_ok tells whether the path takes the call.  peaks
// (launch_integral's of the source, launch_template_prep's of the template, in this order)
// and integ come first; the tiles that the split cannot hold, or (tile_sums: prox_norm_from_tile
// holds for the call) whose sums of squares the integral cannot, are then computed by
// launch_proximity_flagged (tile_sums: integ null), from the flags (one per tile_w x tile_h
// outputs, tiles_x a row) that launch_split_ncc left in `work`.
struct SplitFlags {
   const unsigned *any, *flags;   // any: 0 where no tile is flagged
   int tiles_x, tile_w, tile_h;
};
bool split_ncc_ok(int op, const View &src, const View &T);
size_t split_ncc_work_bytes(const View &src, const View &T);
SplitFlags launch_split_ncc(hipStream_t s, const View &src, const View &T, const double *tsums,
                            const double *integ, bool tile_sums, const unsigned *peaks, float *dst,
                            int dst_step, void *work);
void launch_proximity_flagged(hipStream_t s, const View &src, const View &T, void *dst,
                              int dst_step, const void *tstage, int tpitch, const double *tsums,
                              const double *integ, const SplitFlags &f);

// MFMA cross-correlation (F32 1-channel source and template), precision 1..3.
// The template's fragments and sum of squares (tsums[0]) are built from T in the call.
// may_tune = false: no autotuning (no timing events); the variant tuned earlier for this
// shape, else a fixed default.
void launch_crosscorr_mfma(hipStream_t s, int precision, bool norm, const View &src,
                           const View &T, double *tsums, const double *integ, float *dst,
                           int dst_step, void *work, bool may_tune = true);
// The single-template MFMA Norm path forms its denominators from the source image; only
// templates wider than 513 columns read the FP64 sum-of-squares integral instead.
// Split-BF16 CrossCorr maps (no Norm) of n sources of one size (row pitches sstep[]) with one
// template; up to 16 sources per launch.  The template, its fragments (crosscorr_split_frag_bytes;
// the layout that the kernel variant reads is prepared by the first launch that takes it) and
// sums (sum t^2 to sums[0]):
constexpr int kSplitImages = 16;   // sources per launch of launch_crosscorr_split
size_t crosscorr_split_frag_bytes(int tw, int th);
struct SplitTemplate {
   View T;
   void *frags;
   double *sums;
   bool ready[2] = {false, false};   // the layouts of crosscorr_mfma and crosscorr_mfma_pair
};
void launch_crosscorr_split(hipStream_t s, int n, const float *const *src, const int *sstep,
                            float *const *dst, int dstep, int W, int H, SplitTemplate &t);
bool crosscorr_mfma_needs_integral(int tw);
size_t crosscorr_mfma_work_bytes(int precision, int width, int height, int tw, int th);

// Scratch of the entry point that allocates nothing (noalloc.hip): a device array of
// kNoAllocScratchBytes per GPU.  noalloc_scratch_init takes its address on `device` (which
// must be current) once; noalloc_scratch returns that address.
constexpr size_t kNoAllocScratchBytes = (size_t)8 << 20;
constexpr size_t kNoAllocSumsBytes = 256;   // template sums ahead of the fragments
void noalloc_scratch_init(int device);
void *noalloc_scratch(int device);

// The interleaved channels (2 or 4) of an 8-bit image as 1-channel planes in `planes`
// (planes8_bytes): the view of the first, the others *plane8 bytes apart.
size_t planes8_bytes(const View &image);
View launch_planes8(hipStream_t s, const View &image, void *planes, size_t *plane8);

// AbsDistance of 8-bit images (every channel in one launch), exact int32 sums.
bool sad8_ok(int op, const View &src, const View &T);
size_t sad8_work_bytes(const View &src, const View &T);
void launch_sad8(hipStream_t s, const View &src, const View &T, void *dst, int dst_step, void *work);

// Exact integer sums on int8 MFMA, bit for bit prox_tile_int's maps (OCIP_INT_MFMA=0 turns both
// off); the _ok functions tell whether they take the call.  8-bit images, CrossCorr,
// CrossCorr_Norm, SqrDistance and SqrDistance_Norm, every channel in one launch:
bool int_mfma_ok(int op, const View &src, const View &T);
size_t int_mfma_work_bytes(const View &src, const View &T);
void launch_int_mfma(hipStream_t s, int op, const View &src, const View &T, float *dst, int dst_step,
                     void *work);
// the same of 16-bit 1-channel images:
bool int16_mfma_ok(int op, const View &src, const View &T);
size_t i8_work_bytes(const View &T);
void launch_int16_mfma(hipStream_t s, int op, const View &src, const View &T, float *dst, int dst_step,
                       void *work);

// Batched MFMA CrossCorr_Norm (ssd = false) or SqrDistance_Norm (ssd = true) of F32 1-channel
// templates against one F32 1-channel source, recorded into a HIP graph on first use and
// replayed for identical arguments.  The cache belongs to the context.
BatchCache *batch_cache_create();
void batch_cache_destroy(BatchCache *c);
void run_batch_mfma(hipStream_t s, BatchCache *cache, int num_cus, int precision, bool ssd,
                    const View &S, const std::vector<View> &T, const std::vector<float *> &dst,
                    const std::vector<int> &dstep);

// Gradients (backward.hip) of L = sum_i [sum G1_i CrossCorr_Norm(S_i, t) + sum G2_i
// SqrDistance(S_i, t)] over n same-size F32 1-channel images: G1 / G2 null leaves that op out;
// dS[i] / dT may be null.  dT is the sum over the batch.
size_t backward_work_bytes(int n, int W, int H, int tw, int th, int tpitch);
void launch_backward_batch(hipStream_t s, int n, const View *S, const View *G1, const View *G2,
                           const float *tstage, int tpitch, int tw, int th, const double *tsums,
                           void *work, void *aux, char *const *dS, const int *dsstep, char *dT,
                           int dtstep);

// Proximity through 2-D FFTs (FP64): op kSSD, kSSDNorm, kCC or kCCNorm on an F32 1-channel
// source and template into an F32 dest.  integ: the exclusive FP64 sum-of-squares integral
// (all ops but kCC).  fft_sizes gives the padded transform size or
// CL_INVALID_IMAGE_SIZE when the image is too big for the path.
cl_int fft_sizes(int W, int H, int tw, int th, int *Wb, int *Hb);
void fft_prepare(hipStream_t s, FftState *st, int W, int H, int tw, int th);
void launch_proximity_fft(hipStream_t s, FftState *st, int op, const View &S, const View &T,
                          const double *integ, void *dst, int dstep);

// Generic 2-D FFT (F32 or F64): forward real W x H -> half spectrum (W/2 + 1) x H of
// interleaved complex values, inverse back, unnormalised.  fft_plain_sizes: CL_SUCCESS or
// CL_INVALID_IMAGE_SIZE (a length with a prime factor above 5, or beyond LDS).
cl_int fft_plain_sizes(int W, int H);
void fft_plain_prepare(hipStream_t s, FftState *st, int W, int H);
void launch_fft(hipStream_t s, FftState *st, bool forward, const View &real, const View &cplx);

// Per-channel sum (sqr = false) or sum of squares of an image into result[0..channels),
// blocking.  partials: sum_partials_bytes of device scratch; host_out: the context's.
size_t sum_partials_bytes(int width, int height);
void launch_sum(hipStream_t s, bool sqr, const View &src, void *partials, void *host_out,
                double *result);
// Min / max of a 1-channel image and the pixel holding it, in the reference's reduction order
// (its tie-breaks and float partials), blocking.
size_t minmax_partials_bytes(int width, int height);
void launch_minmax(hipStream_t s, bool want_max, const View &src, void *partials, void *host_out,
                   double *host_result, int *ix, int *iy);

}  // namespace ocip
