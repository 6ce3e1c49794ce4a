// rtm_slab_odd.hip -- the full-row FP32 step for odd row lengths.
#include "rtm_slab.hpp"

namespace rtmhip {
namespace slab {
namespace {

template <int NZW, bool IMG, int TAPER>
hipError_t run(const float *P, float *PP, const float *V, const Coefs &cf, const Grid &g,
               const SlabGrid &sg, const ImageFuse &fz, const TaperFuse &tf, int *flag,
               hipStream_t s)
{
    constexpr int NYW = y_waves(NZW);
    hipLaunchKernelGGL((k_slab<NZW, NYW, kRows, IMG, TAPER, true>),
                       dim3((unsigned)(sg.nyt * sg.nxc)), dim3(64 * NZW, NYW), 0, s, P, PP, V, cf,
                       g, sg, fz, tf, flag);
    return hipGetLastError();
}

template <int NZW, typename... A>
hipError_t by_form(Form form, A &&...a)
{
    switch (form) {
    case kPlain: return run<NZW, false, 0>(a...);
    case kOut: return run<NZW, false, 3>(a...);
    case kOutUpper: return run<NZW, false, 4>(a...);
    case kImage: return run<NZW, true, 0>(a...);
    default: return run<NZW, true, 4>(a...);
    }
}

}  // namespace

hipError_t launch_odd(int nzw, Form form, const float *P, float *PP, const float *V,
                       const Coefs &cf, const Grid &g, const SlabGrid &sg, const ImageFuse &fz,
                       const TaperFuse &tf, int *flag, hipStream_t s)
{
    switch (nzw) {
    case 2: return by_form<2>(form, P, PP, V, cf, g, sg, fz, tf, flag, s);
    case 3: return by_form<3>(form, P, PP, V, cf, g, sg, fz, tf, flag, s);
    case 4: return by_form<4>(form, P, PP, V, cf, g, sg, fz, tf, flag, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace slab
}  // namespace rtmhip
