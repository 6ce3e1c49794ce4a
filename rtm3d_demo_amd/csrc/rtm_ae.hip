// rtm_ae.hip -- kernels of the snapshot autoencoder (learned compression of
// source-wavefield snapshots; no reference counterpart).
//
// A snapshot region is cut into 32^3 bricks, each normalised by its largest
// magnitude and stored as FP16 in "AE order": element e of a brick is cell
// (8 ax + 2 mx + lx, 8 ay + 2 my + ly, 8 az + 2 mz + lz) with
//   e = ((a * 64 + m) * 8 + l),  a = (ax*4+ay)*4+az,  m = (mx*4+my)*4+mz,
//   l = (lx*2+ly)*2+lz.
// In this order every layer of the network is a plain row-major GEMM over
// non-overlapping patches:
//   L1  2^3 patches, 1 -> 8 channels, tanh    [4096 rows x 8]  * [8 x 8]
//   L2  4^3 patches, 8 -> 32 channels (code)   [64 rows x 512]  * [512 x 32]
//   L3  transposed L2, 32 -> 8, tanh           [64 rows x 32]   * [32 x 512]
//   L4  transposed L1, 8 -> 1                  [4096 rows x 8]  * [8 x 8]
// so one brick of 32768 FP16 values (64 KB) becomes 2048 FP16 codes (4 KB)
// plus its scale.  The products run on the matrix cores (FP16 operands, FP32
// accumulation): inference as one launch per direction with every layer in
// registers, a training step as one launch for the gradient (each block's
// partial sums in a slab of its own) and one that adds the slabs and updates.
#include "rtm_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace rtmhip {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
// accesses to the caller's brick and code arrays (any 2-byte alignment)
typedef half8_t half8_any __attribute__((aligned(2)));
typedef half4_t half4_any __attribute__((aligned(2)));

constexpr int kGemmThreads = 256;  // 4 waves; 64 x 64 tile of C, 32 x 32 per wave
constexpr int kBrick = 32768;

__device__ __forceinline__ float load_elem(const void *p, long long i, int is_half)
{
    return is_half ? (float)static_cast<const _Float16 *>(p)[i] : static_cast<const float *>(p)[i];
}

// C(m, n) (+)= sum_k A(m, k) B(k, n), A(m, k) = A[m*sam + k*sak] and
// B(k, n) = B[k*sbk + n*sbn] (either FP32 or FP16 in memory, FP16 operands).
// Epilogue: + bias[n], tanh (act 1); or atomic accumulation of a split-K
// partial (accumulate != 0; blockIdx.z selects the K range).
//
// gfx950's MFMA 16x16x32 (FP16 in, FP32 accumulate): lane l supplies row
// l % 16 of A and column l % 16 of B with eight k values each, k-slot group
// l / 16; A and B use the same k assignment, so the sum over k is the same
// whichever k each slot of the instruction stands for.  D(i, j) of a tile is
// lane j + 16 * (i / 4), item i % 4.  Both operands sit in LDS k-contiguous
// (B transposed), so each lane reads its eight values as one 16-byte load.
__global__ void __launch_bounds__(kGemmThreads) k_gemm(AeGemm p)
{
    constexpr int KT = 32, KP = KT + 8;  // k per tile; padded LDS row (80 B)
    __shared__ __align__(16) _Float16 As[64][KP];
    __shared__ __align__(16) _Float16 Bt[64][KP];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const long long m0 = (long long)blockIdx.x * 64;
    const int n0 = blockIdx.y * 64;
    const long long kb = (long long)blockIdx.z * p.kchunk;
    const long long ke = min((long long)p.K, kb + p.kchunk);
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    float4_t acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (long long k0 = kb; k0 < ke; k0 += KT) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int idx = tid * 8 + q;  // 0 .. 2047
            {
                const int mm = idx >> 5, kk = idx & 31;
                const long long m = m0 + mm, k = k0 + kk;
                float v = 0.f;
                if (m < p.M && k < ke) v = load_elem(p.A, m * p.sam + k * p.sak, p.a_half);
                As[mm][kk] = (_Float16)v;
            }
            {
                const int kk = idx >> 6, nn = idx & 63;
                const long long k = k0 + kk;
                const int n = n0 + nn;
                float v = 0.f;
                if (n < p.N && k < ke) v = load_elem(p.B, k * p.sbk + (long long)n * p.sbn, p.b_half);
                Bt[nn][kk] = (_Float16)v;
            }
        }
        __syncthreads();
        const int r = lane & 15, kq = (lane >> 4) * 8;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const half8_t a = *reinterpret_cast<const half8_t *>(&As[wm + 16 * i + r][kq]);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const half8_t b = *reinterpret_cast<const half8_t *>(&Bt[wn + 16 * j + r][kq]);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc[i][j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const long long m = m0 + wm + 16 * i + 4 * (lane >> 4) + v;
                const int n = n0 + wn + 16 * j + (lane & 15);
                if (m >= p.M || n >= p.N) continue;
                float r = acc[i][j][v];
                float *c = p.C + m * p.ldc + n;
                if (p.accumulate) {
                    atomicAdd(c, r);
                } else {
                    if (p.bias) r += p.bias[n];
                    if (p.act == 1) r = tanhf(r);
                    *c = r;
                }
            }
}

// One block per brick: scale = max |v| over the brick's in-grid cells, then
// the FP16 values v * (1 / scale) (zero outside the grid, and the whole
// brick zero with scale 0 when max |v| is zero or subnormal).
//
// Bound by memory (4 B read and 2 B written per cell).  A lane owns patches
// of 2 x 2 x 2 cells, the 16 lanes (az, mz) of a row covering its 32 z: a
// load instruction reads 4 whole 128-byte rows, a store 4 runs of 256 bytes
// of the brick, and the field is read once -- the cells wait in registers
// for the brick's scale.  VEC: the z pairs are 8-byte aligned and whole.  Salt snapshot
// (592 x 592 x 256, 2888 bricks): 0.176 ms, 3.1 TB/s (0.374 ms in brick order,
// two reads of the field).
constexpr int kCutThreads = 512;

// Block h of n as the position of its work in memory order: XCD h % 8 takes a
// contiguous run, so the 128-byte lines that two z neighbours share (the
// region starts at z = blen, in general inside a line) stay in one L2.
__device__ __forceinline__ unsigned xcd_run(unsigned h, unsigned n)
{
    const unsigned q = n >> 3, r = n & 7, k = h & 7;
    return k * q + min(k, r) + (h >> 3);
}

template <bool VEC>
__global__ void __launch_bounds__(kCutThreads)
    k_bricks(const float *__restrict__ F, Grid g, AeRegion r, _Float16 *__restrict__ out,
             float *__restrict__ scales)
{
    constexpr int NW = kCutThreads / 64, NP = 64 / NW;  // waves, patches per lane
    __shared__ float red[NW];
    const int b = (int)xcd_run(blockIdx.x, gridDim.x);
    const int bz = b % r.nbz, by = (b / r.nbz) % r.nby, bx = b / (r.nbz * r.nby);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int mz = lane & 3, my = (lane >> 2) & 3, az = lane >> 4;
    const int z0 = r.z0 + 32 * bz + 8 * az + 2 * mz;
    float v[NP][2][2][2];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const int p = k * NW + wv;  // (ax, mx, ay) of this patch
        const int x0 = r.x0 + 32 * bx + 2 * (p >> 2);
        const int y0 = r.y0 + 32 * by + 8 * (p & 3) + 2 * my;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                // every lane loads (at a clamped place) and selects after: a
                // branch around the load would wait for it
                const int x = min(x0 + i, r.x1 - 1), y = min(y0 + j, r.y1 - 1);
                const float *f = F + (long long)x * g.sx + (long long)y * g.sy;
                if (VEC) {
                    const float2 u =
                        *reinterpret_cast<const float2 *>(f + min(z0, r.z1 - 2));
                    v[k][i][j][0] = u.x;
                    v[k][i][j][1] = u.y;
                } else {
                    v[k][i][j][0] = f[min(z0, r.z1 - 1)];
                    v[k][i][j][1] = f[min(z0 + 1, r.z1 - 1)];
                }
            }
    }
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const int p = k * NW + wv;
        const int x0 = r.x0 + 32 * bx + 2 * (p >> 2);
        const int y0 = r.y0 + 32 * by + 8 * (p & 3) + 2 * my;
#pragma unroll
        for (int l = 0; l < 8; ++l)
            if (x0 + (l >> 2) >= r.x1 || y0 + ((l >> 1) & 1) >= r.y1 || z0 + (l & 1) >= r.z1)
                v[k][l >> 2][(l >> 1) & 1][l & 1] = 0.f;
    }
    float mx = 0.f;
#pragma unroll
    for (int k = 0; k < NP; ++k)
#pragma unroll
        for (int l = 0; l < 8; ++l) mx = fmaxf(mx, fabsf(v[k][l >> 2][(l >> 1) & 1][l & 1]));
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
    if (lane == 0) red[wv] = mx;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NW; ++k) mx = fmaxf(mx, red[k]);
    // a brick whose largest magnitude is below the smallest normal float
    // (1/s would overflow) is stored as zero
    const float s = mx >= 1.17549435e-38f ? mx : 0.f;
    if (threadIdx.x == 0) scales[b] = s;
    const float inv = s > 0.f ? 1.0f / s : 0.f;
    _Float16 *o = out + (long long)b * kBrick + az * 512 + my * 32 + mz * 8;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const int p = k * NW + wv;
        const int a = (p >> 4) * 16 + (p & 3) * 4, m = (p >> 2) & 3;
        half8_t h;
#pragma unroll
        for (int l = 0; l < 8; ++l) {
            const float c = v[k][l >> 2][(l >> 1) & 1][l & 1];
            // the FP32 product rounded, then narrowed; +0 in a zero brick
            h[l] = wst<_Float16>(s > 0.f ? c * inv : 0.f);
        }
        *reinterpret_cast<half8_any *>(o + a * 512 + m * 128) = h;
    }
}

// Fused inference.  A chunk is 16 consecutive rows a of the middle layers (a
// quarter of a brick: one ax, all ay and az), handled by one wave with
// nothing shared between waves but the weights.  Both GEMMs of a direction
// run transposed (weights as the A operand, rows a as the columns of B), so
// the first product's result -- lane j + 16 g holds rows 4 g + v of column j
// of a 16 x 16 tile -- is the second product's B operand as it stands: the
// second product's weights take the k order {4 g + v, 16 + 4 g + v} instead of the
// natural one, and no value crosses lanes.  The 8 x 8 layers take four
// patches at a time as one 32 x 32 block-diagonal product (K = 32 filled); where
// an infinity or a NaN meets the zeros off its diagonal, one patch at a time
// (patch_product), so that no patch hears of another's.
// Rounding is the separate layers': FP16 operands, FP32 sums, bias and tanh
// in FP32, FP16 again for the next layer.
//
// Bound by the bricks' bytes (encode: 189 MB read) and the field's (decode: 357
// MB written) with tanhf's instructions close behind; a shorter rational tanh
// was no faster (encode 0.076, decode 0.137 ms).  Salt snapshot, 2888 bricks:
// encode 0.083 ms, decode 0.109 ms; as separate GEMM launches with FP32
// intermediates in memory and brick order on the field's side 1.3 and 1.8 ms.
constexpr int kAeThreads = 512;
constexpr int kAeFrag = 16 * 2 * 64 * 8;  // the 512 x 32 weights as MFMA fragments
constexpr long long kOffW1 = 0, kOffB1 = 64, kOffW2 = 72, kOffB2 = kOffW2 + 512 * 32,
                    kOffW3 = kOffB2 + 32, kOffB3 = kOffW3 + 32 * 512, kOffW4 = kOffB3 + 512,
                    kOffB4 = kOffW4 + 64;

// Lane and slot of element k (0..31) in the order {4 g + v, 16 + 4 g + v}.
__device__ __forceinline__ int frag_pos(int i, int k)
{
    return (i + 16 * ((k >> 2) & 3)) * 8 + (k & 3) + 4 * (k >> 4);
}

// A tile of the block-diagonal product of four patches, one patch's operand at
// a time, the others' zeroed: kp(s) is the patch of slot s, op(v) that of
// result item v.
template <typename K, typename O>
__device__ __forceinline__ float4_t patch_product(const half8_t &a, const half8_t &b, K &&kp,
                                                  O &&op)
{
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    float4_t d = zero;
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
        half8_t m;
#pragma unroll
        for (int s = 0; s < 8; ++s) m[s] = kp(s) == p ? b[s] : (_Float16)0.f;
        const float4_t dp = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, m, zero, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) d[v] = op(v) == p ? dp[v] : d[v];
    }
    return d;
}

__global__ void __launch_bounds__(kAeThreads)
    k_ae_encode(const _Float16 *__restrict__ X, const float *__restrict__ w, long long chunks,
                _Float16 *__restrict__ codes)
{
    __shared__ __align__(16) _Float16 w2[kAeFrag];  // [q][t][lane][slot]
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    for (int e = tid; e < 512 * 32; e += kAeThreads) {
        const int k = e >> 5, n = e & 31;
        w2[((k >> 5) * 2 + (n >> 4)) * 512 + frag_pos(n & 15, k & 31)] =
            (_Float16)w[kOffW2 + e];
    }
    half8_t w1[2];  // row o = 16 t + j: patch o / 8, channel o % 8; k = 8 g + s: patch g
    float b1[4], b2[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int o = 16 * t + j;
#pragma unroll
        for (int s = 0; s < 8; ++s)
            w1[t][s] = (o >> 3) == g ? (_Float16)w[kOffW1 + s * 8 + (o & 7)] : (_Float16)0.f;
#pragma unroll
        for (int v = 0; v < 4; ++v) b2[t][v] = w[kOffB2 + 16 * t + 4 * g + v];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) b1[v] = w[kOffB1 + ((4 * g + v) & 7)];
    __syncthreads();
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    const long long c = (long long)xcd_run(blockIdx.x, gridDim.x) * (kAeThreads / 64) + (tid >> 6);
    if (c >= chunks) return;
    {
        const _Float16 *x = X + (c * 16 + j) * 512 + g * 8;
        float4_t acc[2];
        auto layers = [&]<bool apart>(std::bool_constant<apart>) {
        acc[0] = acc[1] = zero;
#pragma unroll(apart ? 1 : 16)
        for (int q = 0; q < 16; ++q) {
            const half8_t xb = *reinterpret_cast<const half8_any *>(x + q * 32);
            half8_t h;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float4_t d =
                    apart ? patch_product(w1[t], xb, [&](int) { return g; },
                                          [&](int) { return 2 * t + (g >> 1); })
                          : __builtin_amdgcn_mfma_f32_16x16x32_f16(w1[t], xb, zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) h[4 * t + v] = wst<_Float16>(tanhf(d[v] + b1[v]));
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    *reinterpret_cast<const half8_t *>(&w2[((q * 2 + t) * 64 + lane) * 8]), h,
                    acc[t], 0, 0, 0);
        }
        };
        layers(std::false_type{});
        // a NaN anywhere in a row makes all its codes NaN
        if (__any(acc[0][0] != acc[0][0])) layers(std::true_type{});
        _Float16 *z = codes + (c * 16 + j) * 32 + 4 * g;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            half4_t o;
#pragma unroll
            for (int v = 0; v < 4; ++v) o[v] = wst<_Float16>(acc[t][v] + b2[t][v]);
            *reinterpret_cast<half4_any *>(z + 16 * t) = o;
        }
    }
}

// Codes -> the region's cells of F (value times its brick's scale).  The
// last layer's 32 outputs of four patches (2 x 2 x 8 cells) are assigned to
// the rows of its two tiles so that lane (j, g) holds the run z = 4 h .. 4 h
// + 3 with (lx, h) = (g / 2, g % 2), ly = t: one 16-byte store per tile
// (VEC: the runs are 16-byte aligned), (az, h) filling 128-byte rows.
template <bool VEC>
__global__ void __launch_bounds__(kAeThreads)
    k_ae_decode(const _Float16 *__restrict__ codes, const float *__restrict__ w, long long chunks,
                const float *__restrict__ scales, Grid gr, AeRegion r, float *__restrict__ F)
{
    __shared__ __align__(16) _Float16 w3[kAeFrag];  // [q][t][lane][slot]
    __shared__ __align__(16) float b3[512];
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    for (int e = tid; e < 32 * 512; e += kAeThreads) {
        const int k = e >> 9, n = e & 511;
        w3[((n >> 4) * 64 + (n & 15) + 16 * (k >> 3)) * 8 + (k & 7)] = (_Float16)w[kOffW3 + e];
    }
    for (int e = tid; e < 512; e += kAeThreads) b3[e] = w[kOffB3 + e];
    half8_t w4[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        // row j of tile t: lx = j / 8, z = j % 8 (patch z / 2), ly = t
        const int z = j & 7, l = (j >> 3) * 4 + t * 2 + (z & 1);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int k = (s & 3) + 4 * g + 16 * (s >> 2);  // patch k / 8, channel k % 8
            w4[t][s] = (k >> 3) == (z >> 1) ? (_Float16)w[kOffW4 + (k & 7) * 8 + l]
                                            : (_Float16)0.f;
        }
    }
    float b4[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 2; ++v) b4[t][v] = w[kOffB4 + (g >> 1) * 4 + t * 2 + v];
    __syncthreads();
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    const long long c = (long long)xcd_run(blockIdx.x, gridDim.x) * (kAeThreads / 64) + (tid >> 6);
    if (c >= chunks) return;
    {
        const half8_t zb = *reinterpret_cast<const half8_any *>(codes + (c * 16 + j) * 32 + g * 8);
        const int b = (int)(c >> 2), ax = (int)(c & 3);
        const float scale = scales[b];
        const int bz = b % r.nbz, by = (b / r.nbz) % r.nby, bx = b / (r.nbz * r.nby);
        const int x0 = r.x0 + 32 * bx + 8 * ax + (g >> 1);
        const int y0 = r.y0 + 32 * by + 8 * (j >> 2);
        const int z0 = r.z0 + 32 * bz + 8 * (j & 3) + 4 * (g & 1);
        float4_t nans = zero;  // 0, or NaN in a column with a NaN
        const half8_t none = {};
        auto layers = [&]<bool apart>(std::bool_constant<apart>) {
#pragma unroll(apart ? 1 : 16)
        for (int q = 0; q < 16; ++q) {
            half8_t h;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    *reinterpret_cast<const half8_t *>(&w3[((q * 2 + t) * 64 + lane) * 8]), zb,
                    zero, 0, 0, 0);
                const float4_t bb =
                    *reinterpret_cast<const float4_t *>(&b3[q * 32 + 16 * t + 4 * g]);
#pragma unroll
                for (int v = 0; v < 4; ++v) h[4 * t + v] = wst<_Float16>(tanhf(d[v] + bb[v]));
            }
            if (!apart)
                nans = __builtin_amdgcn_mfma_f32_16x16x32_f16(none, h, nans, 0, 0, 0);
            const int x = x0 + 2 * (q >> 2), y = y0 + 2 * (q & 3);
            float *p = F + (long long)x * gr.sx + (long long)y * gr.sy + z0;
#pragma unroll
            for (int t = 0; t < 2; ++t, p += gr.sy) {
                const float4_t d =
                    apart ? patch_product(
                                w4[t], h, [&](int s) { return (g >> 1) + 2 * (s >> 2); },
                                [&](int v) { return 2 * (g & 1) + (v >> 1); })
                          : __builtin_amdgcn_mfma_f32_16x16x32_f16(w4[t], h, zero, 0, 0, 0);
                float4_t o;
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = (d[v] + b4[t][v & 1]) * scale;
                if (x < r.x1 && y + t < r.y1) {
                    if (VEC && z0 + 4 <= r.z1) {
                        *reinterpret_cast<float4_t *>(p) = o;
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            if (z0 + v < r.z1) p[v] = o[v];
                    }
                }
            }
        }
        };
        layers(std::false_type{});
        if (__any(nans[0] != nans[0])) layers(std::true_type{});
    }
}

// Gradient of 0.5 * sum (Y - X)^2, forward and backward of one batch in one
// launch.  A tile is 16 rows a of the middle layers, as in k_ae_encode; the
// block's 8 waves take 64 of the 512 elements of a row each (q = 2 w, 2 w + 1),
// so everything between the two sums over all elements (z and dz, through LDS)
// stays in a wave: lane j + 16 g holds row j, elements 32 q + 16 t + 4 g + v.
// The products over elements run transposed as there; the products over rows
// (weight gradients) read their FP16 operands from LDS row-transposed, 16 rows
// to one 16x16x16 product, and accumulate in registers over the block's tiles;
// for the 8 x 8 layers the diagonal blocks of a 16 x 16 product are two
// patches.  A block writes its partial gradient and squared error to a slab of
// its own, k_ae_update adds the slabs.  Rounding as in separate GEMM launches:
// FP16 operands, FP32 sums, FP32 between layers.
//
// Bound by the slabs (134 KB per block written and read back) and by latency:
// one tile per block at 64 bricks (256 blocks).  One step on 64 bricks: 0.040 ms
// and 0.007 of k_ae_update; as 11 GEMM launches of 0.035 ms with every layer in
// memory, column sums and elementwise passes 0.50 ms.
constexpr int kSlabFloats = (int)kOffB4 + 8 + 16;  // parameters, then the loss; padded
constexpr int kLossAt = (int)kOffB4 + 8;
constexpr int kTrainBlocks = 256;  // one per CU: slabs stay few
constexpr int kRowPad = 20;        // LDS row of 16 row values (halves)

__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__global__ void __launch_bounds__(kAeThreads)
    k_ae_gradient(const _Float16 *__restrict__ X, const int *__restrict__ idx, int tiles,
                  const float *__restrict__ w, float *__restrict__ slabs)
{
    constexpr int NW = kAeThreads / 64;
    static_assert(NW == 8);
    __shared__ float zred[NW][8][64], dzred[NW][8][64];
    __shared__ __align__(16) _Float16 tr[NW][32 + 64 + 64][kRowPad];
    const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    _Float16(*tc)[kRowPad] = tr[wv], (*ta)[kRowPad] = tr[wv] + 32, (*tb)[kRowPad] = tr[wv] + 96;
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    // element (slot s of lane group g) in the k order of a product's result
    auto kel = [&](int s) { return (s & 3) + 4 * g + 16 * (s >> 2); };
    auto half8 = [](const float(&v)[2][4]) {
        half8_t h;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) h[4 * t + i] = wst<_Float16>(v[t][i]);
        return h;
    };
    // both tiles of a block-diagonal product (kp as in patch_product)
    auto diagonal = [&](const half8_t(&a)[2], const half8_t &b, float4_t(&d)[2], auto kp) {
        float s = 0.f;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b, zero, 0, 0, 0);
            s += d[t][0] + d[t][1] + d[t][2] + d[t][3];
        }
        if (__any(s != s)) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
                d[t] = patch_product(a[t], b, kp, [&](int) { return 2 * t + (g >> 1); });
        }
    };
    auto natural = [&](int) { return g; };                       // k = 8 g + s
    auto result = [&](int s) { return (g >> 1) + 2 * (s >> 2); };  // k = kel(s)
    // 32 elements of the lane's row into LDS, element-major
    auto put = [&](_Float16(*dst)[kRowPad], const half8_t &h) {
#pragma unroll
        for (int s = 0; s < 8; ++s) dst[kel(s)][j] = h[s];
    };
    // operand of a product over the 16 rows: elements i0 + j, rows 4 g + s
    auto get = [&](const _Float16(*src)[kRowPad], int i0) {
        return *reinterpret_cast<const half4_t *>(&src[i0 + j][4 * g]);
    };
    float4_t gw2[4][2], gw3[2][4], gw1 = zero, gw4 = zero;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) gw2[i][t] = gw3[t][i] = zero;
    float gb1[4] = {}, gb4[4] = {}, gb2[2][4] = {}, gb3[2][2][4] = {}, loss = 0.f;

    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        // the weights are read anew for each tile (L2): the accumulators leave
        // no registers to keep them
        int again = 0;
        asm volatile("" : "+s"(again));
        const float *wt = w + again;
        const long long brick = idx ? idx[tile >> 2] : tile >> 2;
        const _Float16 *x = X + brick * kBrick + ((tile & 3) * 16 + j) * 512 + wv * 64;
        // ---- forward ----
        float h1[2][2][4], z[2][4];
        half8_t xd[2];  // x in the products' result order
        {
            float4_t acc[2] = {zero, zero};
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const half8_t xb = *reinterpret_cast<const half8_any *>(x + q * 32 + g * 8);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const half4_t u =
                        *reinterpret_cast<const half4_any *>(x + q * 32 + 16 * t + 4 * g);
#pragma unroll
                    for (int v = 0; v < 4; ++v) xd[q][4 * t + v] = u[v];
                }
                half8_t a1[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int o = 16 * t + j;  // row: patch o / 8, channel o % 8
#pragma unroll
                    for (int s = 0; s < 8; ++s)
                        a1[t][s] = (o >> 3) == g ? (_Float16)wt[kOffW1 + s * 8 + (o & 7)]
                                                 : (_Float16)0.f;
                }
                float4_t d[2];
                diagonal(a1, xb, d, natural);
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        h1[q][t][v] = tanhf(d[t][v] + wt[kOffB1 + ((4 * g + v) & 7)]);
                const half8_t h = half8(h1[q]);
                const float *w2 = wt + kOffW2 + (wv * 64 + q * 32) * 32 + j;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    half8_t a;
#pragma unroll
                    for (int s = 0; s < 8; ++s) a[s] = (_Float16)w2[kel(s) * 32 + 16 * t];
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, h, acc[t], 0, 0, 0);
                }
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) zred[wv][4 * t + v][lane] = acc[t][v];
            __syncthreads();
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float sum = 0.f;
#pragma unroll
                    for (int k = 0; k < NW; ++k) sum += zred[k][4 * t + v][lane];
                    z[t][v] = sum + wt[kOffB2 + 16 * t + 4 * g + v];
                }
        }
        const half8_t zh = half8(z);
        wave_lds_fence();  // the previous tile's reads of tc, ta, tb
        put(tc, zh);
        float d3[2][2][4];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            float h3[2][4], dy[2][4];
            const float *w3 = wt + kOffW3 + wv * 64 + q * 32 + j;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                half8_t a;
#pragma unroll
                for (int s = 0; s < 8; ++s) a[s] = (_Float16)w3[kel(s) * 512 + 16 * t];
                const float4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, zh, zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    h3[t][v] = tanhf(d[v] + wt[kOffB3 + wv * 64 + q * 32 + 16 * t + 4 * g + v]);
            }
            const half8_t h3h = half8(h3);
            half8_t a4[2];
            float4_t d4[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int o = 16 * t + j;
#pragma unroll
                for (int s = 0; s < 8; ++s)
                    a4[t][s] = (o >> 3) == (kel(s) >> 3)
                                   ? (_Float16)wt[kOffW4 + (kel(s) & 7) * 8 + (o & 7)]
                                   : (_Float16)0.f;
            }
            diagonal(a4, h3h, d4, result);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    dy[t][v] = d4[t][v] + wt[kOffB4 + ((4 * g + v) & 7)] - (float)xd[q][4 * t + v];
                    loss += dy[t][v] * dy[t][v];
                    gb4[v] += dy[t][v];
                }
            }
            // ---- backward ----
            const half8_t dyh = half8(dy);
            put(ta + 32 * q, h3h);
            put(tb + 32 * q, dyh);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int o = 16 * t + j;
#pragma unroll
                for (int s = 0; s < 8; ++s)
                    a4[t][s] = (o >> 3) == (kel(s) >> 3)
                                   ? (_Float16)wt[kOffW4 + (o & 7) * 8 + (kel(s) & 7)]
                                   : (_Float16)0.f;
            }
            diagonal(a4, dyh, d4, result);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    d3[q][t][v] = d4[t][v] * (1.0f - h3[t][v] * h3[t][v]);
                    gb3[q][t][v] += d3[q][t][v];
                }
            }
        }
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < 4; ++i)
            gw4 = __builtin_amdgcn_mfma_f32_16x16x16f16(get(ta, 16 * i), get(tb, 16 * i), gw4, 0,
                                                        0, 0);
        wave_lds_fence();
        float dz[2][4];
        {
            float4_t acc[2] = {zero, zero};
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const half8_t d3h = half8(d3[q]);
                put(ta + 32 * q, d3h);
                put(tb + 32 * q, half8(h1[q]));
                const float *w3 = wt + kOffW3 + j * 512 + wv * 64 + q * 32 + 4 * g;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    half8_t a;
#pragma unroll
                    for (int s = 0; s < 8; ++s)
                        a[s] = (_Float16)w3[16 * t * 512 + 16 * (s >> 2) + (s & 3)];
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, d3h, acc[t], 0, 0, 0);
                }
            }
            wave_lds_fence();
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    gw3[t][i] = __builtin_amdgcn_mfma_f32_16x16x16f16(
                        get(tc, 16 * t), get(ta, 16 * i), gw3[t][i], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) dzred[wv][4 * t + v][lane] = acc[t][v];
            __syncthreads();
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float sum = 0.f;
#pragma unroll
                    for (int k = 0; k < NW; ++k) sum += dzred[k][4 * t + v][lane];
                    dz[t][v] = sum;
                    gb2[t][v] += sum;
                }
        }
        const half8_t dzh = half8(dz);
        put(tc, dzh);
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                gw2[i][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(
                    get(tb, 16 * i), get(tc, 16 * t), gw2[i][t], 0, 0, 0);
        wave_lds_fence();
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            float d1[2][4];
            const float *w2 = wt + kOffW2 + (wv * 64 + q * 32 + j) * 32 + 4 * g;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                half8_t a;
#pragma unroll
                for (int s = 0; s < 8; ++s)
                    a[s] = (_Float16)w2[16 * t * 32 + 16 * (s >> 2) + (s & 3)];
                const float4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, dzh, zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    d1[t][v] = d[v] * (1.0f - h1[q][t][v] * h1[q][t][v]);
                    gb1[v] += d1[t][v];
                }
            }
            put(ta + 32 * q, xd[q]);
            put(tb + 32 * q, half8(d1));
        }
        wave_lds_fence();
#pragma unroll
        for (int i = 0; i < 4; ++i)
            gw1 = __builtin_amdgcn_mfma_f32_16x16x16f16(get(ta, 16 * i), get(tb, 16 * i), gw1, 0,
                                                        0, 0);
    }

    // ---- the block's slab ----
    float *out = slabs + (long long)blockIdx.x * kSlabFloats;
    // result (i, j) of a 16 x 16 product: lane j + 16 (i / 4), item i % 4
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                out[kOffW2 + (wv * 64 + 16 * i + 4 * g + v) * 32 + 16 * t + j] = gw2[i][t][v];
                out[kOffW3 + (16 * t + 4 * g + v) * 512 + wv * 64 + 16 * i + j] = gw3[t][i][v];
            }
    // sums over the 16 rows (lanes j)
    auto rows = [&](float v) {
#pragma unroll
        for (int d = 8; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
        return v;
    };
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float b = rows(gb3[q][t][v]);
                if (j == 0) out[kOffB3 + wv * 64 + q * 32 + 16 * t + 4 * g + v] = b;
            }
    if (wv == 0) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float b = rows(gb2[t][v]);
                if (j == 0) out[kOffB2 + 16 * t + 4 * g + v] = b;
            }
    }
    // over the waves: the 8 x 8 layers (two diagonal blocks each), their
    // biases (lane groups g and g + 2 hold the same channels) and the loss
    __syncthreads();
    float(*red)[8][64] = zred;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        red[wv][v][lane] = gw1[v];
        red[wv][4 + v][lane] = gw4[v];
    }
    float(*redb)[8][64] = dzred;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        redb[wv][v][lane] = rows(gb1[v]);
        redb[wv][4 + v][lane] = rows(gb4[v]);
    }
    __syncthreads();
    // 64 + 64 weights, 8 + 8 biases
    if (tid < 144) {
        const bool second = tid >= 128 ? tid >= 136 : tid >= 64;  // layer 4
        float sum = 0.f;
        if (tid < 128) {
            const int c = (tid & 63) >> 3, o = tid & 7;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const int i = 8 * p + c, l = 8 * p + o + 16 * (i >> 2);
                for (int k = 0; k < NW; ++k) sum += red[k][(second ? 4 : 0) + (i & 3)][l];
            }
            out[(second ? kOffW4 : kOffW1) + c * 8 + o] = sum;
        } else {
            const int o = tid & 7;
#pragma unroll
            for (int p = 0; p < 2; ++p)
                for (int k = 0; k < NW; ++k)
                    sum += redb[k][(second ? 4 : 0) + (o & 3)][16 * (2 * p + (o >> 2))];
            out[(second ? kOffB4 : kOffB1) + o] = sum;
        }
    }
    loss = rows(loss);
#pragma unroll
    for (int d = 16; d < 64; d <<= 1) loss += __shfl_xor(loss, d, 64);
    __syncthreads();
    if (lane == 0) red[0][0][wv] = loss;
    __syncthreads();
    if (tid == 0) {
        float sum = 0.f;
        for (int k = 0; k < NW; ++k) sum += red[0][0][k];
        out[kLossAt] = sum;
    }
}

// The gradient and the loss as sums of the slabs, in their order, then with w
// one step of Adam (Kingma & Ba 2015), bias correction folded into the step
// size.  A block takes 64 parameters, 4 threads each.
__global__ void __launch_bounds__(256)
    k_ae_update(const float *__restrict__ slabs, int nslabs, float *__restrict__ grad,
                float *__restrict__ loss, float *__restrict__ w, float *__restrict__ m,
                float *__restrict__ v, float lr_t, float b1, float b2, float eps)
{
    __shared__ float red[4][64];
    const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    float sum = 0.f;
    if (i <= kLossAt) {
#pragma unroll 8
        for (int k = part; k < nslabs; k += 4) sum += slabs[(long long)k * kSlabFloats + i];
    }
    red[part][lane] = sum;
    __syncthreads();
    if (part != 0 || i > kLossAt) return;
    const float gi = red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane];
    if (i == kLossAt) {
        *loss = gi;
        return;
    }
    grad[i] = gi;
    if (!w) return;
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] = w[i] - lr_t * mi / (sqrtf(vi) + eps);
}

// The region's z runs of n cells (n a power of two) are aligned in F.
inline bool runs_aligned(const float *F, const Grid &g, const AeRegion &r, int n)
{
    return ((uintptr_t)F & (4 * n - 1)) == 0 && (g.sx & (n - 1)) == 0 && (g.sy & (n - 1)) == 0 &&
           (r.z0 & (n - 1)) == 0;
}

}  // namespace

hipError_t launch_ae_gemm(const AeGemm &p, hipStream_t s)
{
    if (p.M <= 0 || p.N <= 0 || p.K <= 0) return hipSuccess;
    AeGemm q = p;
    long long splits = 1;
    if (q.accumulate) {
        if (q.kchunk <= 0) {
            // split K so that the launch has about 1024 blocks, 256..65536 per split
            const long long tiles = ((q.M + 63) / 64) * ((q.N + 63) / 64);
            const long long want = std::max(1LL, 1024 / std::max(1LL, tiles));
            q.kchunk = (int)std::min(65536LL, std::max(256LL, (q.K + want - 1) / want));
        }
        q.kchunk = (q.kchunk + 31) / 32 * 32;
        splits = (q.K + q.kchunk - 1) / q.kchunk;
    } else {
        q.kchunk = (int)((q.K + 31) / 32 * 32);
    }
    const long long gm = (q.M + 63) / 64, gn = (q.N + 63) / 64;
    if (gm > 0x7fffffffLL || gn > 65535 || splits > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gemm, dim3((unsigned)gm, (unsigned)gn, (unsigned)splits),
                       dim3(kGemmThreads), 0, s, q);
    return hipGetLastError();
}

size_t ae_gradient_floats(int n)
{
    return (size_t)std::min(4 * n, kTrainBlocks) * kSlabFloats;
}

hipError_t launch_ae_gradient(const void *bricks, const int *idx, int n, const float *w,
                              float *slabs, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ae_gradient, dim3((unsigned)std::min(4 * n, kTrainBlocks)),
                       dim3(kAeThreads), 0, s, static_cast<const _Float16 *>(bricks), idx, 4 * n,
                       w, slabs);
    return hipGetLastError();
}

hipError_t launch_ae_update(const float *slabs, int n, float *grad, float *loss, float *w,
                            float *m, float *v, float lr_t, float b1, float b2, float eps,
                            hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ae_update, dim3((unsigned)(kLossAt / 64 + 1)), dim3(256), 0, s, slabs,
                       std::min(4 * n, kTrainBlocks), grad, loss, w, m, v, lr_t, b1, b2, eps);
    return hipGetLastError();
}

hipError_t launch_bricks(const float *F, const Grid &g, const AeRegion &r, void *out,
                         float *scales, hipStream_t s)
{
    const long long nb = (long long)r.nbx * r.nby * r.nbz;
    if (nb <= 0) return hipSuccess;
    if (nb > 0x7fffffffLL) return hipErrorInvalidValue;
    const bool pairs = runs_aligned(F, g, r, 2) && (r.z1 & 1) == 0;
    hipLaunchKernelGGL(pairs ? k_bricks<true> : k_bricks<false>, dim3((unsigned)nb),
                       dim3(kCutThreads), 0, s, F, g, r, static_cast<_Float16 *>(out), scales);
    return hipGetLastError();
}

// One chunk per wave, four chunks per brick.
inline unsigned ae_blocks(long long n)
{
    constexpr int waves = kAeThreads / 64;
    return (unsigned)((4 * n + waves - 1) / waves);
}

hipError_t launch_ae_encode(const void *bricks, const float *w, long long n, void *codes,
                            hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_ae_encode, dim3(ae_blocks(n)), dim3(kAeThreads), 0, s,
                       static_cast<const _Float16 *>(bricks), w, 4 * n,
                       static_cast<_Float16 *>(codes));
    return hipGetLastError();
}

hipError_t launch_ae_decode(const void *codes, const float *w, long long n, const float *scales,
                            const Grid &g, const AeRegion &r, float *F, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(runs_aligned(F, g, r, 4) ? k_ae_decode<true> : k_ae_decode<false>,
                       dim3(ae_blocks(n)), dim3(kAeThreads), 0, s,
                       static_cast<const _Float16 *>(codes), w, 4 * n, scales, g, r, F);
    return hipGetLastError();
}

}  // namespace rtmhip
