// device_common.hpp — device-side building blocks shared by every gfx950 kernel of the
// SPH step: smoothing kernels, cell hashing, wave reductions.
//
// Arithmetic contract (matches the FP32 oracle): every value is float, evaluated in the
// reference's expression order, with FMA contraction disabled (-ffp-contract=off) and
// correctly rounded division and square root. Cell coordinates are computed in double.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"

namespace mps {
namespace dev {

constexpr uint32_t kEmpty = 0xFFFFFFFFu;
constexpr int kBlock = 256;  // 4 wave64s per workgroup for particle-parallel kernels

// Place of entry k of slot i in the fluid neighbour lists and in every array stored per entry of
// them (N slots): the entries 4g .. 4g+3 of a slot lie side by side, groups of all slots after one
// another, so a lane can load or store four entries at once (16 bytes of slots) and a wave still
// touches contiguous memory.
__device__ __forceinline__ size_t ell(uint32_t k, uint32_t i, uint32_t N) { return (size_t(k >> 2) * N + i) * 4u + (k & 3u); }

// --------------------------------------------------------------------- float3 helpers
struct f3 {
    float x, y, z;
};
__device__ __forceinline__ f3 mk(float4 a) { return {a.x, a.y, a.z}; }
__device__ __forceinline__ f3 operator-(f3 a, f3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ f3 operator+(f3 a, f3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ f3 operator*(float s, f3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ f3 operator*(f3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
// glm order: (x*x + y*y) + z*z
__device__ __forceinline__ float dot3(f3 a, f3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ __forceinline__ float len3(f3 a) { return __builtin_sqrtf(dot3(a, a)); }

// --------------------------------------------------------------------- smoothing kernels
// Constants of MPSSPHKernel.cuh:9-15 rounded to float.
constexpr float kW = static_cast<float>(1.5666814710608447114749495456982);
constexpr float kG = static_cast<float>(14.323944878270580219199538703526);
constexpr float kCubicW = static_cast<float>(2.5464790894703253723021402139602);
constexpr float kCubicG = static_cast<float>(15.278874536821952233812841283761);
constexpr float kSTW = static_cast<float>(7.2756545413437867780061148970292);
constexpr float kSTG = static_cast<float>(21.826963624031360334018344691088);
constexpr float kEps = static_cast<float>(1.0e-20);
constexpr float kFltEps = 1.19209290e-7f;  // FLT_EPSILON

// W(d, 1/h): poly6 (CUBIC=false) or cubic spline (MPSSPHKernel.cuh:28-45)
template <bool CUBIC>
__device__ __forceinline__ float Wk(float dist, float invh) {
    const float ratio = dist * invh;
    if (ratio >= 1.0f) return 0.0f;
    if (CUBIC) {
        if (ratio >= 0.5f) {
            const float temp = (1.0f - ratio) * invh;
            return kCubicW * 2.0f * temp * temp * temp;
        }
        return kCubicW * invh * invh * invh * ((6.0f * ratio - 6.0f) * ratio * ratio + 1.0f);
    }
    const float tmp = (1.0f - ratio * ratio) * invh;
    return kW * tmp * tmp * tmp;
}
// G(d, 1/h) with grad W_ij = G * x_ij: spiky or cubic (MPSSPHKernel.cuh:46-65)
template <bool CUBIC>
__device__ __forceinline__ float Gk(float dist, float invh) {
    const float ratio = dist * invh;
    if (ratio < kEps || ratio >= 1.0f) return 0.0f;
    const float invh2 = invh * invh;
    if (CUBIC) {
        if (ratio > 0.5f) {
            const float temp = (1.0f - ratio) * invh2;
            return -kCubicG / dist * temp * temp;
        }
        return kCubicG / dist * invh2 * invh2 * (3.0f * ratio - 2.0f) * ratio;
    }
    const float tmp = (1.0f - ratio) * invh2;
    return -kG / dist * tmp * tmp;
}
// Pair factor of the viscosity operator, G(d) / ((d^2 + h2) (d + FLT_EPSILON))
// (MPSSPHNonPressureUtil.cuh:617-618), regrouped to one division: the 1/d inside G joins the
// denominators, Phi = (G d) / ((d (d^2 + h2)) (d + FLT_EPSILON)). The oracle evaluates the
// same expression in the same order (its Phik).
template <bool CUBIC>
__device__ __forceinline__ float Phik(float dist, float invh, float h2) {
    const float ratio = dist * invh;
    if (ratio < kEps || ratio >= 1.0f) return 0.0f;
    const float invh2 = invh * invh;
    float num;
    if (CUBIC) {
        if (ratio > 0.5f) {
            const float temp = (1.0f - ratio) * invh2;
            num = -kCubicG * temp * temp;
        } else {
            num = kCubicG * invh2 * invh2 * (3.0f * ratio - 2.0f) * ratio;
        }
    } else {
        const float tmp = (1.0f - ratio) * invh2;
        num = -kG * tmp * tmp;
    }
    return num / ((dist * (dist * dist + h2)) * (dist + kFltEps));
}
// surface-tension kernels (MPSSPHKernel.cuh:67-84)
__device__ __forceinline__ float STWk(float dist, float invh) {
    float ratio = dist * invh;
    ratio = ratio < 0.5f ? 0.5f : ratio;
    if (ratio >= 1.0f) return 0.0f;
    const float temp = (1.0f - ratio) * invh;
    return kSTW * temp * temp * temp;
}
__device__ __forceinline__ float STGk(float dist, float invh) {
    const float ratio = dist * invh;
    if (ratio <= 0.5f || ratio >= 1.0f) return 0.0f;
    const float temp = (1.0f - ratio) * invh * invh;
    return -kSTG / dist * temp * temp;
}

// --------------------------------------------------------------------- hashing
struct HashGeom {
    uint32_t hx, hy, hz;  // powers of two
    double inv_cell;      // 1.0 / double(cell)
};
struct i3 {
    int x, y, z;
};
// trunc(x * (1/cell)) + H/2, product in double (MPSSpatialHash.cuh:9-19)
__device__ __forceinline__ i3 grid_pos(float x, float y, float z, const HashGeom& g) {
    return {static_cast<int>(static_cast<double>(x) * g.inv_cell) + static_cast<int>(g.hx >> 1),
            static_cast<int>(static_cast<double>(y) * g.inv_cell) + static_cast<int>(g.hy >> 1),
            static_cast<int>(static_cast<double>(z) * g.inv_cell) + static_cast<int>(g.hz >> 1)};
}
// linear cell index with per-axis wrap (MPSSpatialHash.cuh:21-27)
__device__ __forceinline__ uint32_t grid_index(int x, int y, int z, const HashGeom& g) {
    return ((static_cast<uint32_t>(z) & (g.hz - 1u)) * g.hy + (static_cast<uint32_t>(y) & (g.hy - 1u))) * g.hx +
           (static_cast<uint32_t>(x) & (g.hx - 1u));
}
__device__ __forceinline__ uint32_t split_by3(uint32_t x) {
    if (x == 1024u) x--;
    x = (x | x << 16u) & 0x030000FFu;
    x = (x | x << 8u) & 0x0300F00Fu;
    x = (x | x << 4u) & 0x030C30C3u;
    x = (x | x << 2u) & 0x09249249u;
    return x;
}
// Workgroups of a launch go to the 8 XCDs round-robin (workgroup b runs on XCD b % 8), and
// each XCD has its own L2. Renumbering so that XCD x runs one contiguous range of logical
// workgroups keeps the particles a workgroup gathers, which are near it in slot order, in
// the L2 that already holds them. A bijection on [0, n) for every n.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t n) {
    constexpr uint32_t X = 8u;
    const uint32_t per = n / X, rem = n % X, x = b % X;
    return x * per + min(x, rem) + b / X;
}

// Morton key; adds H/2 on top of grid_pos's H/2 (MPSSpatialHash.cuh:29-45)
__device__ __forceinline__ uint32_t grid_zindex(i3 p, const HashGeom& g) {
    const uint32_t x = static_cast<uint32_t>(p.x + static_cast<int>(g.hx >> 1u)) & (g.hx - 1u);
    const uint32_t y = static_cast<uint32_t>(p.y + static_cast<int>(g.hy >> 1u)) & (g.hy - 1u);
    const uint32_t z = static_cast<uint32_t>(p.z + static_cast<int>(g.hz >> 1u)) & (g.hz - 1u);
    return split_by3(x) | (split_by3(y) << 1u) | (split_by3(z) << 2u);
}

// Whether a launch that was enqueued ahead of its predecessor's end has to do nothing.
__device__ __forceinline__ bool shut(const launch::Gate& g) {
    return (g.rec && g.rec->done == kSkipped) || (g.running && *g.running != 0u);
}

// --------------------------------------------------------------------- quads of lanes
// A quad of lanes shares one slot: each lane forms a term, and every lane adds the four terms to its
// copy of the sum in the order of the lanes. No lane of the quad may be masked off.
template <int L>
__device__ __forceinline__ float quad_lane(float v) {  // the value of lane L of the quad, by DPP
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), L * 0x55, 0xF, 0xF, true));
}
__device__ __forceinline__ float add_quad(float s, float t) {
    return (((s + quad_lane<0>(t)) + quad_lane<1>(t)) + quad_lane<2>(t)) + quad_lane<3>(t);
}
__device__ __forceinline__ f3 add_quad(f3 s, f3 t) { return {add_quad(s.x, t.x), add_quad(s.y, t.y), add_quad(s.z, t.z)}; }

// two terms per lane: t0 + u0 + t1 + u1 + ...
__device__ __forceinline__ float add_quad(float s, float t, float u) {
    s = (s + quad_lane<0>(t)) + quad_lane<0>(u);
    s = (s + quad_lane<1>(t)) + quad_lane<1>(u);
    s = (s + quad_lane<2>(t)) + quad_lane<2>(u);
    return (s + quad_lane<3>(t)) + quad_lane<3>(u);
}
__device__ __forceinline__ f3 add_quad(f3 s, f3 t, f3 u) {
    return {add_quad(s.x, t.x, u.x), add_quad(s.y, t.y, u.y), add_quad(s.z, t.z, u.z)};
}
__device__ __forceinline__ float sub_quad(float s, float t) {
    return (((s - quad_lane<0>(t)) - quad_lane<1>(t)) - quad_lane<2>(t)) - quad_lane<3>(t);
}
__device__ __forceinline__ f3 sub_quad(f3 s, f3 t) { return {sub_quad(s.x, t.x), sub_quad(s.y, t.y), sub_quad(s.z, t.z)}; }
template <int Q, class T>
__device__ __forceinline__ T add_lanes(T s, T t) {
    if constexpr (Q == 4) return add_quad(s, t);
    else return s + t;
}
template <int Q, class T>
__device__ __forceinline__ T sub_lanes(T s, T t) {
    if constexpr (Q == 4) return sub_quad(s, t);
    else return s - t;
}
// --------------------------------------------------------------------- wave/block reductions
// Sum of a double over the wave in every lane, in the order of the butterfly v += v[lane ^ off],
// off = 32, 16, 8, 4, 2, 1. The first two steps swap half waves and rows of 16 lanes; after them
// (and after each further step) the values repeat every `off` lanes of a row, where rotating by
// `off` reads what lane ^ off holds. No step goes through LDS, as a shuffle does (the sums sit at
// the end of the latency chain of every solver launch).
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum_d(double v) {
    {
        const uint32_t lo = __double2loint(v), hi = __double2hiint(v);
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        v = __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
    }
    {
        const uint32_t lo = __double2loint(v), hi = __double2hiint(v);
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        v = __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
    }
    v += dpp_d<0x128>(v);  // row_ror:8
    v += dpp_d<0x124>(v);
    v += dpp_d<0x122>(v);
    v += dpp_d<0x121>(v);
    return v;
}
// Sum of a double over a workgroup of NW waves in a fixed order (the butterfly within a wave, then
// the waves in order), valid in every thread. `lds` holds NW values and may be written again only
// after a further barrier.
template <int NW>
__device__ __forceinline__ double block_total(double v, double* lds) {
    v = wave_sum_d(v);
    if ((threadIdx.x & 63u) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double t[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) t[w] = lds[w];
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < NW; w++) s += t[w];
    return s;
}
// The same over a workgroup of kBlock threads; `lds` may be used again at once.
__device__ __forceinline__ double block_sum_d(double v, double* lds /*[kBlock/64]*/) {
    const double s = block_total<kBlock / 64>(v, lds);
    __syncthreads();
    return s;
}

// Statistics of the block halos by one workgroup of 1024 threads (no same-address atomics from every
// workgroup of the build): stats[0] = largest halo staged, stats[1] = blocks not staged, stats[2] =
// blocks with a halo or not staged, stats[3] = blocks whose halo is staged but deeper than
// kHaloShallow.
__device__ __forceinline__ void fold_halo_stats(const uint32_t* __restrict__ hn, uint32_t nblk, uint32_t* __restrict__ stats) {
    __shared__ uint32_t wm[1024 / 64], ws[1024 / 64], wb[1024 / 64], wd[1024 / 64];
    uint32_t mx = 0u, sp = 0u, bl = 0u, dp = 0u;
    for (uint32_t b = threadIdx.x; b < nblk; b += blockDim.x) {
        const uint32_t h = hn[b];
        if (h > kHaloCap) sp++;
        else mx = max(mx, h);
        if (h) bl++;
        if (h > kHaloShallow && h <= kHaloCap) dp++;
    }
    for (int off = 32; off > 0; off >>= 1) {
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, off, 64));
        sp += (uint32_t)__shfl_xor((int)sp, off, 64);
        bl += (uint32_t)__shfl_xor((int)bl, off, 64);
        dp += (uint32_t)__shfl_xor((int)dp, off, 64);
    }
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0) {
        wm[wave] = mx;
        ws[wave] = sp;
        wb[wave] = bl;
        wd[wave] = dp;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < blockDim.x / 64; w++) {
            mx = max(mx, wm[w]);
            sp += ws[w];
            bl += wb[w];
            dp += wd[w];
        }
        stats[0] = mx;
        stats[1] = sp;
        stats[2] = bl;
        stats[3] = dp;
    }
}

}  // namespace dev
}  // namespace mps
