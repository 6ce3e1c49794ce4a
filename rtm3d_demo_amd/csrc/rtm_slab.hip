// rtm_slab.hip -- dispatch of the full-row FP32 step.
#include "rtm_slab_launch.hpp"

#include <algorithm>
#include <atomic>

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

slab::SlabGrid slab_plan(int radius, const Grid &g, const ImageFuse *fuse, const TaperFuse *taper,
                         int arrays)
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
    // A plane step of every block takes 2.3-2.7 us (plain), 2.5-2.8 (upper taper
    // on the output), 2.7-2.9 (taper3D on the output) or 3.8-5 (imaging), what
    // its lanes do not fill included; the waves take 3.0-3.3 us per million
    // cells while the loop's arrays stay in the Infinity Cache (256 MB; the line
    // is at 360), 3.4-3.9 beyond, and full rows or waves with imaging 5.5-7.  So
    // the kernel serves a step below a number of plane steps per million cells,
    // us on either side of it, this kernel / the best other (plane steps per
    // million cells):
    //   plain: 302 x 278 x 256 61.9 / 64.6 (1.12), but 240 x 200 x 400 67.7 / 58.5
    //     (1.46), 350 x 350 x 160 78.3 / 62.3 (1.68); odd rows, whose stores are
    //     cacheable, 400 x 260 x 161 53.3 / 56.1 (1.67); past the cache 448 x 448 x
    //     300 199 / 222 (1.33), but 592 x 592 x 161 217 / 213 (1.60); between the
    //     receiver steps of a backward loop, 6 arrays, both steps together 250 x
    //     250 x 300 168 / 174 (1.44);
    //   upper taper: 330 x 330 x 256 78.4 / 90.5 (1.04), but 280 x 280 x 256 64.7 /
    //     61.8 (1.15); odd 301 x 277 x 259 69.3 / 73.3 (1.53), 400 x 260 x 161 57.9 /
    //     58.0 (1.67); past the cache 448 x 448 x 300 207 / 222 (1.33), but 592 x
    //     592 x 161 232 / 215;
    //   taper3D: 330 x 330 x 256 81.9 / 91.5, but 302 x 278 x 256 67.6 / 64.9; odd
    //     301 x 277 x 255 56.5 / 65.3 (1.13), but 301 x 277 x 259 74.9 / 71.0; past the
    //     cache 528 x 528 x 400 396 / 418 (1.22), but 336 x 336 x 400 170 / 168 (1.35);
    //     beside the frequency accumulators, both fields and those together, 301 x
    //     277 x 259 413 / 424, 240 x 200 x 300 234 / 239 (1.46);
    //   imaging: 300 x 300 x 180 89.5 / 97.1 (1.60), 592 x 592 x 161 345 / 362 (1.60),
    //     but 640 x 300 x 140 195 / 184 (1.82), 592 x 592 x 150 341 / 336 (1.71).
    const double cells = 1e-6 * g.nx * g.ny * g.nz;
    const bool cached = cells * arrays < 90.0, odd = g.nz & 1;
    double line;
    if (fuse) line = 1.65;
    else if (!taper || taper->b <= 0) line = !cached ? 1.5 : odd ? 1.7 : 1.2;
    else if (taper->all == 3) line = !cached ? 1.45 : odd ? 1.6 : 1.13;
    else line = arrays > 6 ? 1.55 : !cached ? 1.3 : odd ? 1.35 : 1.08;
    const int nyt = y_tiles(g);
    const March m = choose_march(nyt, g.nx - 8);
    if ((double)m.steps >= line * cells) return none;
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
