// rtm_dct.hip -- transform coding of source-wavefield snapshots (no reference
// counterpart: the reference keeps the source field by HBC reconstruction or
// as exact snapshots).
//
// The extended grid is cut into 8 x 8 x 32 bricks (x, y, z; z fastest, the
// z origin at 0, so a brick's z lines are 128-byte rows); a brick's cells
// outside the imaging range z in [z0, z1) (or past the grid) enter as 0.
// Each brick goes through the orthonormal 3D DCT-II (separable: 32-point
// along z, 8-point along y and x).  One threshold per snapshot keeps the
// largest coefficients of the whole snapshot within a budget of K: the
// threshold is a power of two, the lowest whose kept count fits (from
// exponent histograms of the coefficients), so between about K/2 and K
// coefficients survive.  A kept coefficient is one 32-bit entry: its index
// in the brick (11 bits) and its value divided by the brick's largest
// magnitude, in FP16; a brick table holds each brick's first entry, entry
// count and scale.  Decoding scatters a brick's entries into a zero brick,
// runs the inverse transform and either writes the cells or applies the
// imaging condition img += w * (v * PR) directly.
//
// A brick is handled by one block of 256 threads in LDS; blocks loop over
// bricks and add their exponent histograms to one 256-bin histogram.  The
// DCT-II's rows are even or odd about their middle, so its inverse computes a
// line's two halves from the same products: 25 operations per cell against 48
// for a learned basis.  (The forward transform keeps the plain sums: which
// coefficients a threshold keeps, and how they round to FP16, should not
// depend on a regrouping.)
#include "rtm_internal.hpp"

#include <algorithm>

namespace rtmhip {
namespace {

constexpr int kDctThreads = 256;
constexpr int kLine = 33;                   // padded z line in LDS
constexpr int kTile = 8 * 8 * kLine;        // one brick in LDS
constexpr int kCells = 8 * 8 * 32;          // 2048 cells / coefficients per brick

// The default basis, orthonormal DCT-II matrices D[u][i] = s(u) cos(pi (2i +
// 1) u / 2n), s(0) = sqrt(1/n), s(u > 0) = sqrt(2/n), evaluated at compile
// time (cosine by range reduction and its Taylor series in double).  The
// transforms read the basis through a pointer with wave-uniform indices, so
// its entries come through scalar loads.
constexpr double kPi = 3.14159265358979323846;
constexpr double ccos(double x)
{
    const double two_pi = 2.0 * kPi;
    x -= (double)(long long)(x / two_pi) * two_pi;
    if (x > kPi) x -= two_pi;
    double term = 1.0, sum = 1.0;
    for (int k = 1; k < 40; ++k) {
        term *= -x * x / (double)((2 * k - 1) * (2 * k));
        sum += term;
    }
    return sum;
}
constexpr BrickBasis make_dct_basis()
{
    BrickBasis t{};
    for (int u = 0; u < 32; ++u)
        for (int i = 0; i < 32; ++i)
            t.z[u][i] = (float)((u ? 0.25 : 0.17677669529663688) *
                                ccos(kPi * (double)((2 * i + 1) * u) / 64.0));
    for (int u = 0; u < 8; ++u)
        for (int i = 0; i < 8; ++i) {
            t.x[u][i] = (float)((u ? 0.5 : 0.35355339059327379) *
                                ccos(kPi * (double)((2 * i + 1) * u) / 16.0));
            t.y[u][i] = t.x[u][i];
        }
    return t;
}
__constant__ BrickBasis kDct = make_dct_basis();

// Basis entries: the caller's (L, read through B with wave-uniform indices,
// so they come through scalar loads) or the compile-time DCT-II table, whose
// entries at constant indices the compiler folds into the instructions.
template <bool L>
__device__ __forceinline__ float bz(const BrickBasis *__restrict__ B, int u, int i)
{
    if constexpr (L) return B->z[u][i];
    else return kDct.z[u][i];
}
template <bool L>
__device__ __forceinline__ float bx(const BrickBasis *__restrict__ B, int u, int i)
{
    if constexpr (L) return B->x[u][i];
    else return kDct.x[u][i];
}
template <bool L>
__device__ __forceinline__ float by(const BrickBasis *__restrict__ B, int u, int i)
{
    if constexpr (L) return B->y[u][i];
    else return kDct.y[u][i];
}

__global__ void k_put_basis(BrickBasis *__restrict__ dst)
{
    const int *src = reinterpret_cast<const int *>(&kDct);
    int *d = reinterpret_cast<int *>(dst);
    for (int i = threadIdx.x; i < (int)(sizeof(BrickBasis) / 4); i += blockDim.x) d[i] = src[i];
}

__device__ __forceinline__ void brick_coords(long long br, const DctLayout &L, int &x0, int &y0,
                                             int &z0)
{
    const int bz = (int)(br % L.nbz);
    const long long r = br / L.nbz;
    const int by = (int)(r % L.nby);
    const int bx = (int)(r / L.nby);
    x0 = 8 * bx;
    y0 = 8 * by;
    z0 = 32 * bz;
}

// One 8-point line through the basis, forward and inverse.
template <typename M>
__device__ __forceinline__ void line8_forward(const float (&in)[8], float (&o)[8], M &&basis)
{
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        float a = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) a = __builtin_fmaf(basis(u, i), in[i], a);
        o[u] = a;
    }
}
template <bool L, typename M>
__device__ __forceinline__ void line8_inverse(const float (&in)[8], float (&o)[8], M &&basis)
{
    if constexpr (L) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float a = 0.0f;
#pragma unroll
            for (int u = 0; u < 8; ++u) a = __builtin_fmaf(basis(u, i), in[u], a);
            o[i] = a;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float e = 0.0f, d = 0.0f;
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
                e = __builtin_fmaf(basis(u, i), in[u], e);
                d = __builtin_fmaf(basis(u + 1, i), in[u + 1], d);
            }
            o[i] = e + d;
            o[7 - i] = e - d;
        }
    }
}

// Forward transform of the brick in t (layout [x][y][z], z padded to 33);
// leaves coefficient (u, v, w) at t[(u*8 + v)*33 + w], except that the x
// pass's outputs stay in the thread's out (x index u = 0..7 at y = tid>>5,
// z = tid&31).  z pass: wave q computes outputs 8q .. 8q+7 of the 64 lines
// (lane = line), so every matrix index is wave-uniform.
template <bool L>
__device__ __forceinline__ void dct3_forward(float *t, const BrickBasis *__restrict__ B,
                                             float (&out)[8])
{
    const int tid = threadIdx.x;
    {   // z
        const int l = tid & 63;
        const int q = __builtin_amdgcn_readfirstlane(tid >> 6);
        float in[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) in[k] = t[l * kLine + k];
        float o[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            float a = 0.0f;
#pragma unroll
            for (int k = 0; k < 32; ++k) a = __builtin_fmaf(bz<L>(B, 8 * q + r, k), in[k], a);
            o[r] = a;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r) t[l * kLine + 8 * q + r] = o[r];
        __syncthreads();
    }
    {   // y: line (i, k)
        const int i = tid >> 5, k = tid & 31;
        float in[8], o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) in[j] = t[(i * 8 + j) * kLine + k];
        line8_forward(in, o, [&](int u, int j) { return by<L>(B, u, j); });
        // the thread's own line: no other thread reads or writes it
#pragma unroll
        for (int u = 0; u < 8; ++u) t[(i * 8 + u) * kLine + k] = o[u];
        __syncthreads();
    }
    {   // x: line (j, k)
        const int j = tid >> 5, k = tid & 31;
        float in[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) in[i] = t[(i * 8 + j) * kLine + k];
        line8_forward(in, out, [&](int u, int i) { return bx<L>(B, u, i); });
    }
}

// Inverse transform (coefficients in t as dct3_forward leaves them).  z pass
// first, by waves of 8 outputs as forward; the x pass's outputs stay in the
// thread's out: out[i] is the cell (i, tid >> 5, tid & 31).
template <bool L>
__device__ __forceinline__ void dct3_inverse(float *t, const BrickBasis *__restrict__ B,
                                             float (&out)[8])
{
    const int tid = threadIdx.x;
    {   // z
        const int l = tid & 63;
        const int q = __builtin_amdgcn_readfirstlane(tid >> 6);
        float in[32];
#pragma unroll
        for (int w = 0; w < 32; ++w) in[w] = t[l * kLine + w];
        float o[8];
        if constexpr (L) {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                float a = 0.0f;
#pragma unroll
                for (int w = 0; w < 32; ++w) a = __builtin_fmaf(bz<L>(B, w, 8 * q + r), in[w], a);
                o[r] = a;
            }
        } else {
            // cells 4q + r and their mirror images
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float e = 0.0f, d = 0.0f;
#pragma unroll
                for (int w = 0; w < 32; w += 2) {
                    e = __builtin_fmaf(bz<L>(B, w, 4 * q + r), in[w], e);
                    d = __builtin_fmaf(bz<L>(B, w + 1, 4 * q + r), in[w + 1], d);
                }
                o[r] = e + d;
                o[4 + r] = e - d;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int z = L ? 8 * q + r : (r < 4 ? 4 * q + r : 31 - 4 * q - (r - 4));
            t[l * kLine + z] = o[r];
        }
        __syncthreads();
    }
    {   // y
        const int i = tid >> 5, k = tid & 31;
        float in[8], o[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) in[u] = t[(i * 8 + u) * kLine + k];
        line8_inverse<L>(in, o, [&](int u, int j) { return by<L>(B, u, j); });
#pragma unroll
        for (int j = 0; j < 8; ++j) t[(i * 8 + j) * kLine + k] = o[j];
        __syncthreads();
    }
    {   // x
        const int j = tid >> 5, k = tid & 31;
        float in[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) in[u] = t[(u * 8 + j) * kLine + k];
        line8_inverse<L>(in, out, [&](int u, int i) { return bx<L>(B, u, i); });
    }
}

// Cell e (0..2047) of a brick: x = e >> 8, y = (e >> 5) & 7, z = e & 31
// (the coefficient index uses the same order).
__device__ __forceinline__ int tile_index(int e) { return (e >> 5) * kLine + (e & 31); }

// Transform of every brick: coefficients to coef[brick][2048] (index
// (u*8 + v)*32 + w), the brick's largest magnitude to table[brick][2]; the
// exponent histogram of the non-zero magnitudes is accumulated in LDS per
// block and added to hist[256] (zeroed beforehand).
//
// A block keeps kHistCopies histograms, one per group of lanes: the
// coefficients of a brick crowd a few exponents, and one histogram serialised
// the 64 lanes of a wave on them (2048 LDS cycles a brick).  528 x 528 x 400,
// 446 MB in and 464 out: 0.339 ms with one histogram and the brick's rows read
// lane by lane through LDS, 0.228 now (4.0 TB/s).
constexpr int kHistCopies = 16;
template <typename T>
__global__ void __launch_bounds__(kDctThreads)
    k_dct_encode(const T *__restrict__ F, Grid g, int z0, int z1, DctLayout L,
                 const BrickBasis *__restrict__ B, float *__restrict__ coef,
                 unsigned *__restrict__ hist, unsigned *__restrict__ table)
{
    __shared__ float t[kTile];
    __shared__ unsigned h[256 * kHistCopies];
    __shared__ unsigned wmax[kDctThreads / 64];
    const int tid = threadIdx.x;
    for (int i = tid; i < 256 * kHistCopies; i += kDctThreads) h[i] = 0;
    const unsigned copy = tid & (kHistCopies - 1);
    const bool learned = B->learned != 0;
    // this thread's column of cells: (y, z) fixed, x = 0 .. 7
    const int j = tid >> 5, k = tid & 31;
    for (long long br = blockIdx.x; br < L.nbr; br += gridDim.x) {
        int bx0, by0, bz0;
        brick_coords(br, L, bx0, by0, bz0);
        const bool in = by0 + j < g.ny && bz0 + k >= z0 && bz0 + k < z1;
        const T *f = F + ((long long)bx0 * g.sx + (long long)min(by0 + j, g.ny - 1) * g.sy +
                          min(max(bz0 + k, z0), z1 - 1));
        float v[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] = wld(f[(long long)min(m, g.nx - 1 - bx0) * g.sx]);
        __syncthreads();  // the previous brick's x pass has read t
#pragma unroll
        for (int m = 0; m < 8; ++m)
            t[(m * 8 + j) * kLine + k] = in && bx0 + m < g.nx ? v[m] : 0.0f;
        __syncthreads();
        float out[8];
        if (learned)
            dct3_forward<true>(t, B, out);
        else
            dct3_forward<false>(t, B, out);
        float *cb = coef + br * kCells;
        unsigned mx = 0;  // as bits: a NaN counts as the largest
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            cb[(u * 8 + j) * 32 + k] = out[u];
            const unsigned bits = __builtin_bit_cast(unsigned, out[u]) & 0x7fffffffu;
            mx = max(mx, bits);
            if (bits) atomicAdd(&h[(bits >> 23) * kHistCopies + copy], 1u);
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) mx = max(mx, (unsigned)__shfl_xor(mx, d, 64));
        if ((tid & 63) == 0) wmax[tid >> 6] = mx;
        __syncthreads();
        if (tid == 0)
            table[br * 3 + 2] = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    }
    __syncthreads();
    unsigned n = 0;
    for (int c = 0; c < kHistCopies; ++c) n += h[tid * kHistCopies + c];
    if (n) atomicAdd(&hist[tid], n);
}

__global__ void k_dct_clear(unsigned *__restrict__ hist) { hist[threadIdx.x] = 0; }

// Threshold of one snapshot: meta[0] = the lowest power-of-two magnitude
// (as float bits) whose kept count (|c| >= it) is at most K, meta[1] = that
// count, meta[2] = 0 (the entry counter of the packing pass).
__global__ void __launch_bounds__(kDctThreads)
    k_dct_select(const unsigned *__restrict__ hist, long long K, unsigned *__restrict__ meta)
{
    __shared__ unsigned long long tot[256];
    tot[threadIdx.x] = hist[threadIdx.x];
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long cum = 0;
        unsigned thr = 0x7f800000u;  // nothing kept below infinity if bin 255 overflows
        int e = 255;
        for (; e >= 0; --e) {
            if (cum + tot[e] > (unsigned long long)K) break;
            cum += tot[e];
        }
        // bins above e are kept; bin 0 (subnormal magnitudes) starts at bits 1
        thr = e < 0 ? 1u : ((unsigned)(e + 1) << 23);
        meta[0] = thr;
        meta[1] = (unsigned)cum;
        meta[2] = 0;
    }
}

// Packing: the coefficients with |c| >= threshold, per brick in index order,
// appended to the entry pool, and the brick table {first entry, count, scale}
// (the scale is there from the encoding pass).
//
// A block takes kPackBricks consecutive bricks at a time, all their
// coefficients in registers, and reserves their entries with one atomic: one
// counter for all bricks of the chip serialised them (one atomic per brick:
// 0.56 ms for the 56,628 bricks of a 528 x 528 x 400 grid, 9 times the time
// of reading the coefficients).  A brick whose scale is below the threshold is
// not read.  528 x 528 x 400: 0.562 ms, now 0.139.
//
// Eight bricks to a block, but two for up to kPackFew bricks, which eight to a
// block would leave most of the chip without (us, two / eight: 64 bricks 4.3 /
// 9.5, 288 5.6 / 10.9, 684 10.2 / 11.0, 2880 24.9 / 15.5).
constexpr long long kPackFew = 768;
template <int kPackBricks>
__global__ void __launch_bounds__(kDctThreads)
    k_dct_pack(const float *__restrict__ coef, DctLayout L, unsigned *__restrict__ meta,
               unsigned *__restrict__ entries, unsigned *__restrict__ table)
{
    constexpr int NW = kDctThreads / 64;
    __shared__ unsigned wsum[NW][kPackBricks];
    __shared__ unsigned sbase;
    const unsigned thr = meta[0];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const long long groups = (L.nbr + kPackBricks - 1) / kPackBricks;
    for (long long gr = blockIdx.x; gr < groups; gr += gridDim.x) {
        const long long b0 = gr * kPackBricks;
        float scale[kPackBricks];
        float4 c[kPackBricks][2];  // this thread: 8 consecutive coefficients of each
#pragma unroll
        for (int q = 0; q < kPackBricks; ++q) {
            scale[q] = b0 + q < L.nbr ? __builtin_bit_cast(float, table[(b0 + q) * 3 + 2]) : 0.0f;
            c[q][0] = c[q][1] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (b0 + q < L.nbr && __builtin_bit_cast(unsigned, scale[q]) >= thr) {
                const float4 *p =
                    reinterpret_cast<const float4 *>(coef + (b0 + q) * kCells + 8 * tid);
                c[q][0] = p[0];
                c[q][1] = p[1];
            }
        }
        // kept coefficients of each brick: this thread's bits, and the counts'
        // prefix over the block (index order = thread order), two bricks to a
        // word (a brick has at most 2048)
        unsigned keep[kPackBricks], incl[kPackBricks / 2], own[kPackBricks / 2];
#pragma unroll
        for (int q = 0; q < kPackBricks; ++q) {
            const float *v = reinterpret_cast<const float *>(c[q]);
            unsigned kq = 0;
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const unsigned bits = __builtin_bit_cast(unsigned, v[m]) & 0x7fffffffu;
                if (bits >= thr && bits) kq |= 1u << m;
            }
            keep[q] = kq;
            const unsigned n = __popc(kq);
            if (q & 1) own[q / 2] |= n << 16;
            else own[q / 2] = n;
        }
#pragma unroll
        for (int p = 0; p < kPackBricks / 2; ++p) {
            unsigned s = own[p];
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const unsigned o = __shfl_up(s, d, 64);
                if (lane >= d) s += o;
            }
            incl[p] = s;
            if (lane == 63) {
                wsum[wv][2 * p] = s & 0xffffu;
                wsum[wv][2 * p + 1] = s >> 16;
            }
        }
        __syncthreads();
        if (tid == 0) {
            unsigned total = 0;
#pragma unroll
            for (int q = 0; q < kPackBricks; ++q)
#pragma unroll
                for (int w = 0; w < NW; ++w) total += wsum[w][q];
            sbase = total ? atomicAdd(&meta[2], total) : 0u;
        }
        __syncthreads();
        unsigned base = sbase;
#pragma unroll
        for (int q = 0; q < kPackBricks; ++q) {
            unsigned before = 0, total = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                if (w < wv) before += wsum[w][q];
                total += wsum[w][q];
            }
            if (tid == 0 && b0 + q < L.nbr) {
                table[(b0 + q) * 3 + 0] = total ? base : 0u;
                table[(b0 + q) * 3 + 1] = total;
            }
            const unsigned mine = (incl[q / 2] - own[q / 2]) >> (q & 1 ? 16 : 0) & 0xffffu;
            unsigned pos = base + before + mine;
            const float *v = reinterpret_cast<const float *>(c[q]);
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                if ((keep[q] >> m) & 1u) {
                    // a division, not a product with 1/scale: the reciprocal
                    // of a subnormal scale overflows (FP32 fields reach
                    // subnormal magnitudes far from the source), the quotient
                    // stays <= 1
                    const _Float16 hv = (_Float16)(v[m] / scale[q]);
                    entries[pos++] = (unsigned)(8 * tid + m) |
                                     ((unsigned)__builtin_bit_cast(unsigned short, hv) << 16);
                }
            }
            base += total;
        }
        __syncthreads();  // wsum / sbase reused by the next group
    }
}

// Decoding: each brick rebuilt from its entries; IMG: img += w * (v * PR) on the
// imaging range, else out = v there (FP32, the grid's layout).  The z lines
// first, while most coefficients are zero rows; a DCT's lines are folded into
// their even and odd halves (half the products), a caller's basis is not; a
// brick without entries is not transformed.  528 x 528 x 400, imaging (1.3 GB of
// img and PR): 0.382 ms, now 0.272.
template <typename T, bool IMG>
__global__ void __launch_bounds__(kDctThreads)
    k_dct_decode(const unsigned *__restrict__ entries, const unsigned *__restrict__ table,
                 DctLayout L, const BrickBasis *__restrict__ B, Grid g, int z0, int z1,
                 const T *__restrict__ PR, float *__restrict__ img, float w,
                 float *__restrict__ out)
{
    __shared__ float t[kTile];
    const int tid = threadIdx.x;
    const bool learned = B->learned != 0;
    // this thread's column of cells: (y, z) fixed, x = 0 .. 7
    const int j = tid >> 5, k = tid & 31;
    for (long long br = blockIdx.x; br < L.nbr; br += gridDim.x) {
        const unsigned base = table[br * 3 + 0], n = table[br * 3 + 1];
        const float scale = __builtin_bit_cast(float, table[br * 3 + 2]);
        // the imaging operands, loaded (at clamped places) before the inverse
        // transform so that their latency overlaps it; PR as raw bits in
        // 32-bit registers, widened after the transform
        int bx0, by0, bz0;
        brick_coords(br, L, bx0, by0, bz0);
        const bool in = by0 + j < g.ny && bz0 + k >= z0 && bz0 + k < z1;
        const long long o = (long long)bx0 * g.sx +
                            (long long)min(by0 + j, g.ny - 1) * g.sy +
                            min(max(bz0 + k, z0), z1 - 1);
        unsigned pr[8];
        float im[8];
        if (IMG) {
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const long long om = o + (long long)min(m, g.nx - 1 - bx0) * g.sx;
                if constexpr (sizeof(T) == 2)
                    pr[m] = reinterpret_cast<const unsigned short *>(PR)[om];
                else
                    pr[m] = reinterpret_cast<const unsigned *>(PR)[om];
                im[m] = img[om];
            }
        }
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (n) {  // the same for the block
            __syncthreads();  // the previous brick's x pass has read t
            for (int e = tid; e < kTile; e += kDctThreads) t[e] = 0.0f;
            __syncthreads();
            for (unsigned e = tid; e < n; e += kDctThreads) {
                const unsigned u = entries[base + e];
                const float c = (float)__builtin_bit_cast(_Float16, (unsigned short)(u >> 16));
                t[tile_index((int)(u & 0x7ffu))] = c * scale;
            }
            __syncthreads();
            if (learned)
                dct3_inverse<true>(t, B, v);
            else
                dct3_inverse<false>(t, B, v);
        }
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            if (!in || bx0 + m >= g.nx) continue;
            if (IMG) {
                float prv;
                if constexpr (sizeof(T) == 2)
                    prv = wld(__builtin_bit_cast(T, (unsigned short)pr[m]));
                else
                    prv = __builtin_bit_cast(float, pr[m]);
                const float p = v[m] * prv;
                img[o + (long long)m * g.sx] = im[m] + w * p;
            } else {
                out[o + (long long)m * g.sx] = v[m];
            }
        }
    }
}

// blocks per launch: each loops over bricks (up to 16 per CU on 256 CUs)
inline unsigned dct_blocks(long long nbr) { return (unsigned)std::min<long long>(nbr, 4096); }

}  // namespace

hipError_t dct_default_basis(BrickBasis *dst, hipStream_t s)
{
    hipLaunchKernelGGL(k_put_basis, dim3(1), dim3(256), 0, s, dst);
    return hipGetLastError();
}

DctLayout dct_layout(const Grid &g)
{
    DctLayout L{};
    L.nbx = (g.nx + 7) / 8;
    L.nby = (g.ny + 7) / 8;
    L.nbz = (g.nz + 31) / 32;
    L.nbr = (long long)L.nbx * L.nby * L.nbz;
    L.nblk = (int)dct_blocks(L.nbr);
    return L;
}

template <typename T>
hipError_t launch_dct_encode(const T *F, const Grid &g, int z0, int z1, const DctLayout &L,
                             const BrickBasis *B, long long K, float *coef, unsigned *hist,
                             unsigned *meta, unsigned *entries, unsigned *table, hipStream_t s)
{
    if (L.nbr <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dct_clear, dim3(1), dim3(256), 0, s, hist);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_dct_encode<T>, dim3(L.nblk), dim3(kDctThreads), 0, s, F, g, z0, z1, L, B,
                       coef, hist, table);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_dct_select, dim3(1), dim3(kDctThreads), 0, s, hist, K, meta);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(L.nbr <= kPackFew ? k_dct_pack<2> : k_dct_pack<8>, dim3(L.nblk),
                       dim3(kDctThreads), 0, s, coef, L, meta, entries, table);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_dct_decode(const unsigned *entries, const unsigned *table, const DctLayout &L,
                             const BrickBasis *B, const Grid &g, int z0, int z1, const T *PR,
                             float *img, float w, float *out, hipStream_t s)
{
    if (L.nbr <= 0) return hipSuccess;
    if (PR)
        hipLaunchKernelGGL((k_dct_decode<T, true>), dim3(L.nblk), dim3(kDctThreads), 0, s,
                           entries, table, L, B, g, z0, z1, PR, img, w, out);
    else
        hipLaunchKernelGGL((k_dct_decode<T, false>), dim3(L.nblk), dim3(kDctThreads), 0, s,
                           entries, table, L, B, g, z0, z1, PR, img, w, out);
    return hipGetLastError();
}

#define RTM_INSTANTIATE_DCT(T)                                                                 \
    template hipError_t launch_dct_encode<T>(const T *, const Grid &, int, int,                \
                                             const DctLayout &, const BrickBasis *, long long,   \
                                             float *, unsigned *, unsigned *, unsigned *,        \
                                             unsigned *, hipStream_t);                           \
    template hipError_t launch_dct_decode<T>(const unsigned *, const unsigned *,               \
                                             const DctLayout &, const BrickBasis *,              \
                                             const Grid &, int, int, const T *, float *, float,  \
                                             float *, hipStream_t);
RTM_INSTANTIATE_DCT(float)
RTM_INSTANTIATE_DCT(_Float16)
RTM_INSTANTIATE_DCT(__bf16)

}  // namespace rtmhip
