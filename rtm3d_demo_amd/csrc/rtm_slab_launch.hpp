// rtm_slab_launch.hpp -- host side of the full-row FP32 step (rtm_slab.hpp).
#pragma once
#include "rtm_internal.hpp"

namespace rtmhip {
namespace slab {

constexpr int kSlabTaper = 1024;  // longest taper table held in LDS

struct SlabGrid {
    int nyt, nxc, xchunk;
};

// Work of a step on the cells around the updated ones, done in the same pass:
// save / restore (at most one) point to the step's layer [nx][ny][4] of the
// upper-border history (blen b, even, >= 8), zframe: see k_slab.  Covers the
// rows that the step updates; the x and y frame is the caller's.
struct SlabShell {
    float *save;
    const float *restore;
    int b;
    int zframe;
};

// Launches for even and odd row lengths: nzw waves of 128 z per row, `form`
// the fusion (form_of).
enum Form { kPlain, kPlainRestore, kOut, kOutUpper, kOutUpperSave, kImage, kImageOutUpper };
hipError_t launch_even(int nzw, Form form, const float *P, float *PP, const float *V,
                       const Coefs &cf, const Grid &g, const SlabGrid &sg, const ImageFuse &fz,
                       const TaperFuse &tf, const SlabShell &sh, int *flag, hipStream_t s);
hipError_t launch_odd(int nzw, Form form, const float *P, float *PP, const float *V,
                      const Coefs &cf, const Grid &g, const SlabGrid &sg, const ImageFuse &fz,
                      const TaperFuse &tf, const SlabShell &sh, int *flag, hipStream_t s);

// y waves per block and rows per wave: 12 waves (3 per SIMD at up to 168
// registers) whatever the row length.
constexpr int kRows = 3;
constexpr int y_waves(int nzw) { return 12 / nzw; }

}  // namespace slab

// The step (radius 4, FP32) that the full-row kernel serves: no taper, taper3D
// or the upper taper on the output, imaging without a taper or with the upper
// taper on the output.
bool slab_fits(int radius, const Grid &g, const ImageFuse *fuse, const TaperFuse *taper);
hipError_t launch_slab(const float *P, float *PP, const float *V, const Coefs &cf, const Grid &g,
                       const ImageFuse *fuse, const TaperFuse *taper, int *flag, hipStream_t s,
                       const slab::SlabShell *shell = nullptr);

}  // namespace rtmhip
