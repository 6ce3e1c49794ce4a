// rtm_slab.hpp -- the FP32 order-8 step on full-row blocks, two z cells per
// lane.  Included by the translation units that instantiate it (even and odd
// row lengths).  Arithmetic, fusions and rounding are those of the kernels in
// rtm_stencil.hip (rtm-3d/src/platform/host/RTMCPUPlatform.cpp:325-395,
// :513-540, :566-657, :710-920), so results are bit-identical to them but for
// the sign of a zero after an underflow.
//
// What bounds it: the bytes that miss the XCD's L2.  A wave that marches its
// own 4-row tile (k_stencil_wave2) re-reads its 8 halo rows from beyond L2,
// because their owner loaded them R planes earlier, as the lead of its x ring,
// and the XCD's 4 MB hold about two planes of the tiles it works on: 22.0
// bytes per cell against the 16 of P, PP, V in and PP out.  Here
//   * a block holds whole rows (NZW waves of 128 z each) of NYW x RY rows, so
//     no z halo exists, and its rows' y neighbours come from LDS;
//   * the 2R halo rows around the block are loaded together with the ring's
//     lead plane, at the time when the neighbouring blocks load them as their
//     own, and wait R planes in registers: they hit L2;
//   * PP, V, the imaging operands and the stores are non-temporal, so they do
//     not push P out of L2;
//   * the next plane is staged into LDS during this plane's arithmetic (its
//     centre rows have been in the ring for R planes): one barrier per plane,
//     with nothing to wait for behind it.
// That is 17.2 bytes per cell (FETCH_SIZE + WRITE_SIZE).  Salt grid, 592 x 592
// x 336, ms, against the best wave or row shape: plain 0.355 (0.417), upper
// taper on the output 0.353 (0.431), taper3D on the output 0.368 (0.474),
// imaging with the upper taper 0.622 (0.714); 5.0 TB/s of algorithmic
// bytes for the plain step.  With branches around the loads and stores (see
// bounded_view) the first three were 0.373, 0.381 and 0.404.  Halos loaded a
// plane ahead instead of with the lead: 18.8 bytes per cell, 4 % slower;
// cacheable streams: plain 2 %, imaging 6 % slower.  The x ring's 60 registers
// and the 20 of the waiting halo rows set 3 rows per wave (4 rows spill),
// 12 waves per CU.  It is then bound by the 5 to 6 TB/s beyond L2 and nearly as
// much by the VALU (55 % of its issue slots; imaging 37 %).
#pragma once
#include "rtm_internal.hpp"
#include "rtm_slab_launch.hpp"

#include <type_traits>
#include <utility>

#pragma clang fp contract(off)

namespace rtmhip {
namespace slab {

constexpr int R = 4;
constexpr int kNonTemporal = 2;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Raw buffer view of one plane: descriptor in scalar registers, so an access
// is descriptor + scalar row offset + the lane's 32-bit z offset.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_view(const void *p)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, -1, 0x00020000);
}

// The same with the plane's size: a store whose lane offset is kDropped is out
// of range and discarded by the memory unit.  So a plane's step has no branch
// around a load or a store, and its wait counts are exact: with branches the
// compiler must assume at every join that the later loads were not issued, and
// waits for all of them where only PP and V are needed (plain step, salt grid:
// 0.373 ms with branches, 0.348 without).
constexpr unsigned kDropped = 0x7ffffff0u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t bounded_view(void *p, long long cells)
{
    return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)(cells * 4), 0x00020000);
}

// One z pair (8 bytes at 4-byte alignment).
template <int POLICY = 0>
__device__ __forceinline__ void ld_pair(__amdgpu_buffer_rsrc_t rs, unsigned soff, unsigned voff,
                                        float (&v)[2])
{
    const u32x2 u = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)voff, (int)soff, POLICY);
    // elements copied out first: a bit cast of u.y reads element 0 here
    const unsigned lo = u.x, hi = u.y;
    v[0] = __builtin_bit_cast(float, lo);
    v[1] = __builtin_bit_cast(float, hi);
}
template <int POLICY>
__device__ __forceinline__ void st_pair(__amdgpu_buffer_rsrc_t rs, unsigned soff, unsigned voff,
                                        float a, float b)
{
    u32x2 u;
    u.x = __builtin_bit_cast(unsigned, a);
    u.y = __builtin_bit_cast(unsigned, b);
    __builtin_amdgcn_raw_buffer_store_b64(u, rs, (int)voff, (int)soff, POLICY);
}
template <int POLICY>
__device__ __forceinline__ void st_one(__amdgpu_buffer_rsrc_t rs, unsigned soff, unsigned voff,
                                       float a)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, a), rs, (int)voff,
                                          (int)soff, POLICY);
}

__device__ __forceinline__ float uniform(float v)
{
    return __builtin_bit_cast(float,
                              __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// Block-wide barrier ordering LDS only: loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// IMG: img += ps * pp on z in [z0, z1) off the receiver cells.  TAPER 0 none;
// 3 taper3D on the output; 4 the upper taper on the output (cells z < b -
// hold), the centre PP tapered once.  ODD: odd nz (the last pair of a row is
// half outside; pairs may be updated by halves).
//
// The frame taper and the upper-border history stay out of this kernel: its
// first z wave would do them for the whole block, and the others wait at the
// barrier (saving the layer and tapering the z frame here: 0.383 -> 0.437 ms,
// more than the pass of their own takes).
template <int NZW, int NYW, int RY, bool IMG, int TAPER, bool ODD>
__global__ void __launch_bounds__(64 * NZW *NYW, 1)
    k_slab(const float *__restrict__ P, float *__restrict__ PP, const float *__restrict__ V,
           const Coefs cf, const Grid g, const SlabGrid sg, const ImageFuse fz,
           const TaperFuse tf, int *__restrict__ flag)
{
    constexpr int TY = NYW * RY;
    constexpr int LW = 128 * NZW + 2 * R;  // LDS row: z in [-R, 128 NZW + R)
    constexpr int LH = TY + 2 * R;
    constexpr int NH = (2 * R + NYW - 1) / NYW;  // halo rows per wave
    constexpr int NR = 2 * R + 2;
    // cache policy of the streamed operands (rows of odd length share their
    // last cache line with the next row: 301 x 277 x 255 60 us, non-temporal 73)
    constexpr int POL = ODD ? 0 : kNonTemporal;
    constexpr bool OUT = TAPER == 3, OUTU = TAPER == 4;
    __shared__ __align__(16) float tile[2][LH][LW];
    __shared__ float tab[TAPER ? kSlabTaper : 1];  // taper table g[b]
    const float *__restrict__ PS = static_cast<const float *>(fz.ps);

    int by, bx;
    {
        const int n = sg.nyt * sg.nxc, h = blockIdx.x;
        const int q = n >> 3, r = n & 7, k = h & 7, j = h >> 3;
        const int t = k * q + min(k, r) + j;
        by = t % sg.nyt;
        bx = t / sg.nyt;
    }
    const int zl = threadIdx.x;
    const int yw = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int wz0 = (__builtin_amdgcn_readfirstlane(threadIdx.x) & ~63) * 2;  // wave's first z
    const int z = 2 * zl;
    const int y0 = R + by * TY;
    const int xb = R + bx * sg.xchunk;
    const int xe = min(xb + sg.xchunk, g.nx - R);
    const unsigned zc = (unsigned)min(z, g.nz - 2);
    const unsigned zoff = zc * 4u;
    // the lane at z = nz - 1 (odd nz) loads the pair before and shifts it
    const bool zlast = ODD && z == g.nz - 1;
    // nz, z and R even: a pair is updated whole or not at all
    const bool zcomp = (z >= R) && (z < g.nz - R);
    const bool zcomp1 = ODD ? (z >= R) && (z + 1 < g.nz - R) : zcomp;

    if (TAPER) {
        const int tid = threadIdx.y * (64 * NZW) + threadIdx.x;
        for (int i = tid; i < tf.b; i += 64 * NZW * NYW) tab[i] = tf.t[i];
        __syncthreads();
    }
    auto lat = [&](int i, int n) -> float {
        const int j = i < tf.b ? tf.b - 1 - i : (i >= n - tf.b ? i - (n - tf.b) : -1);
        return j >= 0 ? tab[max(j, 0)] : 1.0f;
    };
    const bool wtap = TAPER && (OUT || wz0 < tf.b);
    bool ztap[2];
    float fzl[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int za = min(z + a, g.nz - 1);
        ztap[a] = wtap && (OUT ? (za < tf.b || za >= g.nz - tf.b) : (z + a < tf.b));
        fzl[a] = 1.0f;
        if (ztap[a]) fzl[a] = OUT ? lat(za, g.nz) : tab[tf.b - 1 - (z + a)];
    }
    // lanes that store: every pair with an updated cell (an odd row's last one
    // writes its other cell back unchanged), with OUT also the z frame's; an
    // odd row's last cell alone
    const bool wpair = OUT ? z + 1 < g.nz : zcomp;
    const bool wone = ODD && OUT && z + 1 == g.nz;
    // the image: pairs with an imaged cell, the imaged cells, the receivers'
    const bool ipair = IMG && zcomp && z + 1 >= fz.z0 && z < fz.z1;
    const bool icell[2] = {IMG && z >= fz.z0 && z < fz.z1,
                           IMG && zcomp1 && z + 1 >= fz.z0 && z + 1 < fz.z1};
    const bool rcell[2] = {IMG && z == fz.rz, IMG && z + 1 == fz.rz};
    // cells whose stored value carries the upper taper
    const bool ucell[2] = {OUTU && ztap[0] && z < tf.b - tf.hold,
                           OUTU && ztap[1] && z + 1 < tf.b - tf.hold};

    unsigned rowb[RY];
    unsigned ymask = 0, rmask = 0;
    float fyr[RY];
#pragma unroll
    for (int r = 0; r < RY; ++r) {
        const int y = y0 + yw * RY + r;
        const int yc = min(y, g.ny - 1);
        rowb[r] = (unsigned)yc * (unsigned)g.sy * 4u;
        if (y < g.ny - R) ymask |= 1u << r;
        if (IMG) {
            const int dy = y - fz.ry0;
            if (dy >= 0 && (dy % fz.rdy) == 0 && (dy / fz.rdy) < fz.rny) rmask |= 1u << r;
        }
        fyr[r] = 1.0f;
        if (wtap) fyr[r] = uniform(lat(yc, g.ny));
    }
    // halo rows h = yw, yw + NYW, ... of the 2R around the block's rows
    unsigned hrow[NH];
    int hl[NH];
#pragma unroll
    for (int i = 0; i < NH; ++i) {
        const int h = yw + i * NYW;
        const int y = min(h < R ? y0 - R + h : y0 + TY + (h - R), g.ny - 1);
        hl[i] = h < R ? h : TY + h;
        hrow[i] = (unsigned)y * (unsigned)g.sy * 4u;
    }

    float q[NR][RY][2];
    // Halo planes in flight (divides NR).  Imaging with the taper has no
    // registers for more than 2 (spilling 5: 0.624 ms, 2: 0.605)
    constexpr int NHR = IMG && OUTU ? 2 : R + 1;
    static_assert(NR % NHR == 0);
    float hv[NHR][NH][2];

    auto plane_fx = [&](int x) -> float { return wtap ? uniform(lat(x, g.nx)) : 1.0f; };
    auto tap = [&](float v, int a, float fx, float fy) -> float {
        v *= ztap[a] ? fy : 1.0f;
        v *= ztap[a] ? fx : 1.0f;
        v *= fzl[a];
        return v;
    };
    // taper3D at a value: ((v*fy)*fx)*fz on the z border, (v*fx)*fy off it
    auto tapo = [&](float v, int a, float fx, float fy) -> float {
        if (ztap[a]) {
            v *= fy;
            v *= fx;
            v *= fzl[a];
        } else {
            v *= fx;
            v *= fy;
        }
        return v;
    };
    auto ld_row = [&](__amdgpu_buffer_rsrc_t rs, unsigned row, float(&v)[2]) {
        ld_pair(rs, row, zoff, v);
        if (ODD) v[0] = zlast ? v[1] : v[0];
    };
    auto load_ring = [&](int x, float(&dst)[RY][2]) {
        const auto rs = plane_view(P + (size_t)x * (size_t)g.sx);
#pragma unroll
        for (int r = 0; r < RY; ++r) ld_row(rs, rowb[r], dst[r]);
    };
    auto load_halo = [&](int x, float(&h)[NH][2]) {
        const auto rs = plane_view(P + (size_t)x * (size_t)g.sx);
#pragma unroll
        for (int i = 0; i < NH; ++i) ld_row(rs, hrow[i], h[i]);
    };
    // A plane of the block in LDS: this wave's rows (their ring slot) and its
    // share of the halo rows.
    auto stage = [&](int buf, const float(&rows)[RY][2], const float(&h)[NH][2]) {
        float(*tl)[LW] = tile[buf];
#pragma unroll
        for (int r = 0; r < RY; ++r)
            *reinterpret_cast<float2 *>(&tl[R + yw * RY + r][R + z]) =
                make_float2(rows[r][0], rows[r][1]);
#pragma unroll
        for (int i = 0; i < NH; ++i)
            if ((i + 1) * NYW <= 2 * R || yw + i * NYW < 2 * R)
                *reinterpret_cast<float2 *>(&tl[hl[i]][R + z]) = make_float2(h[i][0], h[i][1]);
    };

#pragma unroll
    for (int s = 0; s <= 2 * R; ++s) load_ring(xb - R + s, q[s]);
#pragma unroll
    for (int s = 0; s < NHR; ++s) load_halo(xb + s, hv[s]);
    stage(0, q[R], hv[0]);
    lds_barrier();

    bool bad0 = false, bad1 = false;
    int x = xb;
    auto step = [&]<int K>(std::integral_constant<int, K>) -> bool {
        if (x >= xe) return false;
        constexpr int cur = K & 1;
        constexpr int ctr = (K + R) % NR;
        const size_t pl = (size_t)x * (size_t)g.sx;
        const auto rpp = bounded_view(PP + pl, g.sx);
        const auto rv = plane_view(V + pl);
        const auto rps = plane_view(IMG ? PS + pl : PP);
        const auto rimg = bounded_view(IMG ? fz.img + pl : PP, g.sx);
        float(*tl)[LW] = tile[cur];
        // this plane's PP, V (and imaging operands), used after the Laplacians
        float c_pp[RY][2], c_v[RY][2], c_ps[RY][2], c_img[RY][2];
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            ld_pair<POL>(rpp, rowb[r], zoff, c_pp[r]);
            ld_pair<POL>(rv, rowb[r], zoff, c_v[r]);
            if (ODD && OUT) c_pp[r][0] = zlast ? c_pp[r][1] : c_pp[r][0];
        }
        if (IMG) {
#pragma unroll
            for (int r = 0; r < RY; ++r) {
                ld_pair<POL>(rps, rowb[r], zoff, c_ps[r]);
                ld_pair<POL>(rimg, rowb[r], zoff, c_img[r]);
            }
        }
        load_ring(min(x + 1 + R, g.nx - 1), q[(K + 2 * R + 1) % NR]);
        stage(cur ^ 1, q[(ctr + 1) % NR], hv[(K + 1) % NHR]);
        load_halo(min(x + NHR, g.nx - 1), hv[K % NHR]);
        bool rcvx = false;
        if (IMG) {
            const int dx = x - fz.rx0;
            rcvx = dx >= 0 && (dx % fz.rdx) == 0 && (dx / fz.rdx) < fz.rnx;
        }
        float fxc = 1.0f;
        if (TAPER) fxc = plane_fx(x);
        float yn[2 * R][2];  // rows above and below this wave's
#pragma unroll
        for (int h = 0; h < 2 * R; ++h) {
            const float2 u = *reinterpret_cast<const float2 *>(
                &tl[yw * RY + (h < R ? h : RY + h)][R + z]);
            yn[h][0] = u.x;
            yn[h][1] = u.y;
        }
        float lapl[RY][2];
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            float w[2 * R + 2];  // cells z - R .. z + R + 1
            const float2 *t2 = reinterpret_cast<const float2 *>(&tl[R + yw * RY + r][z]);
#pragma unroll
            for (int k = 0; k <= R; ++k) {
                const float2 u = t2[k];
                w[2 * k] = u.x;
                w[2 * k + 1] = u.y;
            }
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const float p = q[ctr][r][a];
                float ax, ay, az;
#pragma unroll
                for (int io = 0; io <= 2 * R; ++io) {
                    const int ry = r + io - R;
                    const float vx = q[(K + io) % NR][r][a];
                    const float vy = ry < 0 ? yn[ry + R][a]
                                            : (ry >= RY ? yn[R + ry - RY][a] : q[ctr][ry][a]);
                    const float vz = (io == R) ? p : w[io + a];
                    if (io == 0) {
                        // 0 + v*c in one instruction (the same number; only
                        // a negative product that underflows gives -0 here)
                        ax = __builtin_fmaf(vx, cf.c[0][io], 0.f);
                        ay = __builtin_fmaf(vy, cf.c[1][io], 0.f);
                        az = __builtin_fmaf(vz, cf.c[2][io], 0.f);
                    } else {
                        ax += vx * cf.c[0][io];
                        ay += vy * cf.c[1][io];
                        az += vz * cf.c[2][io];
                    }
                }
                lapl[r][a] = ax + ay + az;
                // pinned: otherwise it sinks into finish's two branches
                asm volatile("" : "+v"(lapl[r][a]));
            }
        }
        // the upper taper's arithmetic only in the waves that it reaches
        auto finish = [&]<bool taped>(std::bool_constant<taped>) {
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            float npp[2], o[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                float pp = c_pp[r][a];
                if (OUT) {
                    if (tf.pp_taps > 0) pp = tapo(pp, a, fxc, fyr[r]);
                } else if (taped) {
                    pp = tap(pp, a, fxc, fyr[r]);
                }
                npp[a] = 2.f * q[ctr][r][a] - pp + c_v[r][a] * lapl[r][a];
                o[a] = npp[a];
                // (z frame: not updated; PP tapered once more as the next
                // step's P)
                if (OUT) o[a] = tapo((a ? zcomp1 : zcomp) ? npp[a] : pp, a, fxc, fyr[r]);
                if (taped) o[a] = ucell[a] ? tap(npp[a], a, fxc, fyr[r]) : o[a];
            }
            const bool row = (ymask >> r) & 1u;
            if (ODD && !OUT) o[1] = zcomp1 ? o[1] : c_pp[r][1];
            st_pair<POL>(rpp, rowb[r], row && wpair ? zoff : kDropped, o[0], o[1]);
            if (ODD && OUT) st_one<POL>(rpp, rowb[r], row && wone ? zoff + 4u : kDropped, o[0]);
            bad0 |= row && npp[0] != npp[0];
            bad1 |= row && npp[1] != npp[1];
            if (IMG) {
                // cells of a pair outside [z0, z1) or under a receiver keep
                // their value
                const bool rc = rcvx && ((rmask >> r) & 1u);
                float iv[2];
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    const bool on = icell[a] && !(rc && rcell[a]);
                    iv[a] = on ? c_img[r][a] + c_ps[r][a] * npp[a] : c_img[r][a];
                }
                st_pair<POL>(rimg, rowb[r], row && ipair ? zoff : kDropped, iv[0], iv[1]);
            }
        }
        };
        if (OUTU && wtap) finish(std::true_type{});
        else finish(std::false_type{});
        lds_barrier();
        ++x;
        return true;
    };
    while (x < xe) {
        [&]<int... Ks>(std::integer_sequence<int, Ks...>) {
            (step(std::integral_constant<int, Ks>{}) && ...);
        }(std::make_integer_sequence<int, NR>{});
    }
    if ((zcomp && bad0) || (zcomp1 && bad1)) atomicOr(flag, 1);
}

}  // namespace slab
}  // namespace rtmhip
