// rtm_slab_launch.hpp -- host side of the full-row FP32 step (rtm_slab.hpp).
#pragma once
#include "rtm_internal.hpp"

namespace rtmhip {
namespace slab {

constexpr int kSlabTaper = 1024;  // longest taper table held in LDS

// y tiles, x chunks and their length; nyt 0: the kernel does not serve the step
struct SlabGrid {
    int nyt, nxc, xchunk;
};

// Launches for even and odd row lengths: nzw waves of 128 z per row, `form`
// the fusion (form_of).
enum Form { kPlain, kOut, kOutUpper, kImage, kImageOutUpper };
hipError_t launch_even(int nzw, Form form, const float *P, float *PP, const float *V,
                       const Coefs &cf, const Grid &g, const SlabGrid &sg, const ImageFuse &fz,
                       const TaperFuse &tf, int *flag, hipStream_t s);
hipError_t launch_odd(int nzw, Form form, const float *P, float *PP, const float *V,
                      const Coefs &cf, const Grid &g, const SlabGrid &sg, const ImageFuse &fz,
                      const TaperFuse &tf, int *flag, hipStream_t s);

// y waves per block and rows per wave: 12 waves (3 per SIMD at up to 168
// registers) whatever the row length.
constexpr int kRows = 3;
constexpr int y_waves(int nzw) { return 12 / nzw; }

}  // namespace slab

// The step (radius 4, FP32) that the full-row kernel serves: no taper, taper3D
// or the upper taper on the output, imaging without a taper or with the upper
// taper on the output.  arrays: how many of the grid's size the loop touches from
// one such step to the next (P, PP and V alone: 3).  launch_slab takes the plan
// of the same step.
slab::SlabGrid slab_plan(int radius, const Grid &g, const ImageFuse *fuse, const TaperFuse *taper,
                         int arrays = 3);
hipError_t launch_slab(const slab::SlabGrid &plan, const float *P, float *PP, const float *V,
                       const Coefs &cf, const Grid &g, const ImageFuse *fuse,
                       const TaperFuse *taper, int *flag, hipStream_t s);

}  // namespace rtmhip
