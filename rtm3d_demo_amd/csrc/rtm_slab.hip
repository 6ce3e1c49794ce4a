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

bool slab_fits(int radius, const Grid &g, const ImageFuse *fuse, const TaperFuse *taper)
{
    using namespace slab;
    if (radius != 4 || g.nx <= 8 || g.ny <= 8 || g.nz <= 128 || g.nz > 512) return false;
    if (g.sy != g.nz || g.sx != (long long)g.ny * g.nz) return false;
    // 32-bit byte offsets inside a plane
    if (g.sx * 4 >= (1LL << 31)) return false;
    if (taper && taper->b > 0) {
        if (taper->b > kSlabTaper || (taper->all != 2 && taper->all != 3)) return false;
        if (taper->all == 2 && (fuse || taper->b < 4 || 2 * taper->b >= g.nx ||
                                2 * taper->b >= g.ny || 2 * taper->b >= g.nz))
            return false;
        if (taper->all == 3 && (taper->hold < 0 || taper->hold > taper->b)) return false;
    }
    // A plane step takes 2.7-3.0 us (4.6-5.1 with imaging) whatever the row
    // length; the waves of rtm_stencil.hip take 3.1-3.4 us (6.0-6.7) per
    // million cells, more where rows fill their tiles badly -- where part of
    // this kernel's lanes idle too.  Measured, us, this kernel / the best
    // waves or rows (plain; imaging): 592 x 592 x 336 374 / 403; 627 / 713,
    // 336^3 125 / 134; 225 / 249, 302 x 278 x 256 64 / 65; 111 / 143,
    // 880 x 880 x 480 1142 / 1260; 1917 / 2419.  Outside the rule: 192^3
    // 29 / 24; 50 / 41, 300 x 300 x 272 91 / 85, 640 x 300 x 140 131 / 100,
    // 301 x 277 x 259 75 / 74; 186 / 164.
    const double fill = std::sqrt((double)((g.nz + 127) / 128 * 128) / g.nz);
    const double line = (fuse && !(g.nz & 1) ? 1.35e-6 : 1.2e-6) * fill;
    return (double)choose_march(y_tiles(g), g.nx - 8).steps <
           line * (double)g.nx * g.ny * g.nz;
}

hipError_t launch_slab(const float *P, float *PP, const float *V, const Coefs &cf, const Grid &g,
                       const ImageFuse *fuse, const TaperFuse *taper, int *flag, hipStream_t s,
                       const slab::SlabShell *shell)
{
    using namespace slab;
    if (!slab_fits(4, g, fuse, taper)) return hipErrorInvalidValue;
    ImageFuse fz{};
    TaperFuse tf{};
    if (fuse) {
        fz = *fuse;
        fz.rdx = std::max(1, fz.rdx);
        fz.rdy = std::max(1, fz.rdy);
    }
    const bool tap = taper && taper->b > 0;
    if (tap) tf = *taper;
    SlabShell sh{};
    if (shell) sh = *shell;
    Form form = fuse ? (tap ? kImageOutUpper : kImage)
                     : (!tap ? kPlain : (tf.all == 2 ? kOut : kOutUpper));
    if (sh.save || sh.restore) {
        if (sh.b < 8 || (sh.b & 1)) return hipErrorInvalidValue;
        if (sh.save && form == kOutUpper) form = kOutUpperSave;
        else if (sh.restore && form == kPlain) form = kPlainRestore;
        else return hipErrorInvalidValue;
    }
    const int nzw = (g.nz + 127) / 128;
    SlabGrid sg;
    sg.nyt = y_tiles(g);
    sg.xchunk = choose_march(sg.nyt, g.nx - 8).chunk;
    sg.nxc = (g.nx - 8 + sg.xchunk - 1) / sg.xchunk;
    return (g.nz & 1) ? launch_odd(nzw, form, P, PP, V, cf, g, sg, fz, tf, sh, flag, s)
                      : launch_even(nzw, form, P, PP, V, cf, g, sg, fz, tf, sh, flag, s);
}

}  // namespace rtmhip
