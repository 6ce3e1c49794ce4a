// rtm_slab.hip -- dispatch of the full-row FP32 step.
#include "rtm_slab_launch.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>

namespace rtmhip {
namespace {

int compute_units()
{
    static std::atomic<int> known{0};
    int n = known.load();
    if (n > 0) return n;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        n = 256;
    known.store(n);
    return n;
}

// One block of 12 waves fills a CU, so a launch runs in whole rounds of one
// block per CU: the x chunk count whose rounds take the fewest plane steps.  A
// chunk of n planes costs n steps and about 6 more to fill the x ring (2R + 1
// planes of loads, no arithmetic).
struct March {
    int chunk;
    long long steps;  // plane steps, one after the other
};
March choose_march(int nyt, int nxi)
{
    const int cus = compute_units();
    long long best = -1;
    int best_chunk = nxi;
    for (int n = 1; n <= 64 && n <= nxi; ++n) {
        const int chunk = (nxi + n - 1) / n;
        const long long blocks = (long long)nyt * ((nxi + chunk - 1) / chunk);
        const long long cost = (blocks + cus - 1) / cus * (chunk + 6);
        if (best < 0 || cost < best) {
            best = cost;
            best_chunk = chunk;
        }
    }
    return March{best_chunk, best};
}

int y_tiles(const Grid &g)
{
    const int rows = slab::y_waves((g.nz + 127) / 128) * slab::kRows;
    return (g.ny - 8 + rows - 1) / rows;
}

}  // namespace

slab::SlabGrid slab_plan(int radius, const Grid &g, const ImageFuse *fuse, const TaperFuse *taper)
{
    using namespace slab;
    const SlabGrid none{0, 0, 0};
    if (radius != 4 || g.nx <= 8 || g.ny <= 8 || g.nz <= 128 || g.nz > 512) return none;
    if (g.sy != g.nz || g.sx != (long long)g.ny * g.nz) return none;
    // 32-bit byte offsets inside a plane
    if (g.sx * 4 >= (1LL << 31)) return none;
    if (taper && taper->b > 0) {
        if (taper->b > kSlabTaper || (taper->all != 2 && taper->all != 3)) return none;
        if (taper->all == 2 && (fuse || taper->b < 4 || 2 * taper->b >= g.nx ||
                                2 * taper->b >= g.ny || 2 * taper->b >= g.nz))
            return none;
        if (taper->all == 3 && (taper->hold < 0 || taper->hold > taper->b)) return none;
    }
    // A plane step takes 2.2-2.5 us (3.9-4.6 with imaging) whatever the row
    // length; the waves of rtm_stencil.hip take 2.6-3.4 us (4.6-6.7) per
    // million cells, more where rows fill their tiles badly -- where part of
    // this kernel's lanes idle too.  The lines lie between the sizes measured
    // on either side, us, this kernel / the best waves or rows (steps per
    // million filled cells).  Plain: 302 x 278 x 256 59.6 / 64.1 (1.12), 240^3
    // 42.8 / 45.1 (1.331), but 640 x 300 x 140 117 / 102 (1.348), 192^3
    // 24.8 / 23.6 (1.71).  Imaging: 640 x 300 x 140 189 / 201 (1.348), but 200 x
    // 180 x 300 72 / 67 (1.47); odd rows 301 x 277 x 259 153 / 169 (1.255), but
    // 400 x 260 x 161 125 / 120 (1.326).
    const double fill = std::sqrt((double)((g.nz + 127) / 128 * 128) / g.nz);
    const double line = (!fuse ? 1.335e-6 : (g.nz & 1) ? 1.32e-6 : 1.4e-6) * fill;
    const int nyt = y_tiles(g);
    const March m = choose_march(nyt, g.nx - 8);
    if ((double)m.steps >= line * (double)g.nx * g.ny * g.nz) return none;
    return SlabGrid{nyt, (g.nx - 8 + m.chunk - 1) / m.chunk, m.chunk};
}

hipError_t launch_slab(const slab::SlabGrid &plan, const float *P, float *PP, const float *V,
                       const Coefs &cf, const Grid &g, const ImageFuse *fuse,
                       const TaperFuse *taper, int *flag, hipStream_t s)
{
    using namespace slab;
    if (plan.nyt <= 0) return hipErrorInvalidValue;
    ImageFuse fz{};
    TaperFuse tf{};
    if (fuse) {
        fz = *fuse;
        fz.rdx = std::max(1, fz.rdx);
        fz.rdy = std::max(1, fz.rdy);
    }
    const bool tap = taper && taper->b > 0;
    if (tap) tf = *taper;
    const Form form = fuse ? (tap ? kImageOutUpper : kImage)
                           : (!tap ? kPlain : (tf.all == 2 ? kOut : kOutUpper));
    const int nzw = (g.nz + 127) / 128;
    return (g.nz & 1) ? launch_odd(nzw, form, P, PP, V, cf, g, plan, fz, tf, flag, s)
                      : launch_even(nzw, form, P, PP, V, cf, g, plan, fz, tf, flag, s);
}

}  // namespace rtmhip
