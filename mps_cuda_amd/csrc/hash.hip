// hash.hip — spatial hash and neighbour search for gfx950.
//
// Replaces SpatialHash::UpdateHash / ZSort / BuildNeighorhood (MPSSpatialHash.cu:53-218,
// MPSSpatialHash.cuh:83-271). Design:
//   * cell keys computed in double exactly like GetGridPos (trunc(x*(1/cell)) + H/2);
//   * a stable LSD radix sort written here (digits of up to 11 bits, wave64 ballot ranking), so ties
//     keep ascending particle id — the order the reference's neighbour lists depend on;
//   * cell start/end tables cleared incrementally (only cells occupied last step), plus a
//     copy of the positions in key order so the 27-cell scan reads contiguous memory;
//   * one search pass per particle (no count/scan/fill double scan): fluid neighbours go to ELL
//     storage in groups of four entries per slot (ell(), device_common.hpp), the wall neighbours
//     to column-major ELL storage nbr[k*N + i], the boundary-boundary list to rows of K slots (it is read once, when the walls move),
//     the per-particle count to cnt[i]; overflow past the capacity is counted and reported
//     so the host can grow the capacity and search again;
//   * the fluid search stages a workgroup's candidates in LDS, row by row, so that each
//     particle walks its 27 cells as 9 contiguous runs (k_neighbors_fluid).
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace mps {
namespace dev {

// ===================================================================== radix sort
// Stable LSD radix sort of (key, value) pairs. Two ways by size:
//   * up to kSortOne items, one workgroup keeps them in registers and trades them through LDS
//     between the passes: one launch for all passes;
//   * beyond, tiles of kSortTile items, a histogram and a scatter per pass. Up to kSortSelf tiles
//     every scatter workgroup sums the histograms of the tiles before its own (and of all, for the
//     digits' totals) by itself; with more tiles a scan in between does it once.
// In a tile every wave owns a contiguous strip and counts its digits in its own LDS counters, so
// ranking needs no barrier: equal digits of a round are ranked by ballots, rounds by the counter.
// What bounds it: launches and their latency up to some 100 k items (15 launches of 3-5 us with
// 8-bit digits, a scan of three launches and a barrier per round: 250 particles 65 -> 9.5 us, 33 k
// 74 -> 23), then the scattered 4-byte stores (1 M: 95 -> 45 us).
constexpr int kSortThreads = 256;
constexpr int kSortRounds = 8;
constexpr int kSortTile = kSortThreads * kSortRounds;
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kOneThreads = 1024;
constexpr int kOneWaves = kOneThreads / 64;
constexpr int kOneRounds = 8;
constexpr uint32_t kSortOne = kOneThreads * kOneRounds;
constexpr uint32_t kSortSelf = 32;
constexpr int kOneDigit = 8;

// Inclusive scan of one value per thread over W waves (every thread calls it; ws: W + 1 words).
template <int W>
__device__ __forceinline__ uint32_t block_incl_scan(uint32_t v, uint32_t* ws) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(v, off, 64);
        if (lane >= off) v += t;
    }
    if (lane == 63) ws[w] = v;
    __syncthreads();
    uint32_t before = 0u;
#pragma unroll
    for (int q = 0; q < W; q++) before += q < w ? ws[q] : 0u;
    __syncthreads();
    return v + before;
}
// Rank of this lane's digit among the wave's items so far; cnt: the wave's own 2^D counters.
template <int D>
__device__ __forceinline__ uint32_t wave_rank(uint32_t d, bool valid, uint32_t* cnt) {
    const uint64_t lt = (1ull << (threadIdx.x & 63)) - 1ull;
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < D; b++) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    const uint32_t before = __popcll(m & lt);
    const uint32_t base = cnt[d];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (valid && before == 0u) cnt[d] = base + __popcll(m);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return base + before;
}

__global__ void __launch_bounds__(kOneThreads) k_radix_one(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                         uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n,
                                                         int bits) {
    constexpr uint32_t kDigits = 1u << kOneDigit;
    __shared__ uint32_t cnt[kOneWaves][kDigits];
    __shared__ uint32_t ws[kOneWaves];
    __shared__ uint2 item[kSortOne];
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const uint32_t rounds = (n + kOneThreads - 1u) / kOneThreads;
    const uint32_t first = w * 64u * rounds + lane;
    uint2 it[kOneRounds];
#pragma unroll
    for (uint32_t r = 0; r < kOneRounds; r++) {
        const uint32_t i = first + 64u * r;
        const bool valid = r < rounds && i < n;
        it[r] = valid ? make_uint2(kin[i], vin[i]) : make_uint2(0u, 0u);
    }
    for (int shift = 0; shift < bits; shift += kOneDigit) {
        for (uint32_t c = t; c < kOneWaves * kDigits; c += kOneThreads) cnt[0][c] = 0u;
        __syncthreads();
        uint32_t rank[kOneRounds];
#pragma unroll
        for (uint32_t r = 0; r < kOneRounds; r++)
            if (r < rounds) rank[r] = wave_rank<kOneDigit>((it[r].x >> shift) & (kDigits - 1u), first + 64u * r < n, cnt[w]);
        __syncthreads();
        // a digit's counters become the position of each wave's first item of it
        uint32_t tot = 0u;
        if (t < kDigits)
            for (int q = 0; q < kOneWaves; q++) {
                const uint32_t c = cnt[q][t];
                cnt[q][t] = tot;
                tot += c;
            }
        const uint32_t before = block_incl_scan<kOneWaves>(tot, ws) - tot;
        if (t < kDigits)
            for (int q = 0; q < kOneWaves; q++) cnt[q][t] += before;
        __syncthreads();
        const bool last = shift + kOneDigit >= bits;
#pragma unroll
        for (uint32_t r = 0; r < kOneRounds; r++)
            if (r < rounds && first + 64u * r < n) {
                const uint32_t at = cnt[w][(it[r].x >> shift) & (kDigits - 1u)] + rank[r];
                if (last) {
                    kout[at] = it[r].x;
                    vout[at] = it[r].y;
                } else {
                    item[at] = it[r];
                }
            }
        if (last) break;
        __syncthreads();
#pragma unroll
        for (uint32_t r = 0; r < kOneRounds; r++)
            if (r < rounds && first + 64u * r < n) it[r] = item[first + 64u * r];
    }
}

// hist[tile][digit]
template <int D>
__global__ void __launch_bounds__(kSortThreads) k_radix_hist(const uint32_t* __restrict__ keys, uint32_t n, int shift,
                                                           uint32_t* __restrict__ hist) {
    constexpr uint32_t kDigits = 1u << D;
    __shared__ uint32_t h[kDigits];
    for (uint32_t d = threadIdx.x; d < kDigits; d += kSortThreads) h[d] = 0u;
    __syncthreads();
    const uint32_t base = blockIdx.x * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortRounds; r++) {
        const uint32_t i = base + r * kSortThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & (kDigits - 1u)], 1u);
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < kDigits; d += kSortThreads) hist[size_t(blockIdx.x) * kDigits + d] = h[d];
}

// Exclusive scan of the histograms over the tiles, in place, and the digits' totals: 16 digits
// (a 64-byte line of every tile) per workgroup, a run of tiles per thread.
constexpr uint32_t kScanDigits = 16;
constexpr uint32_t kScanRuns = 64;
__global__ void __launch_bounds__(kScanDigits* kScanRuns) k_radix_scan(uint32_t* __restrict__ hist, uint32_t digits,
                                                                        uint32_t tiles, uint32_t* __restrict__ total) {
    __shared__ uint32_t run[kScanRuns][kScanDigits];
    const uint32_t d = blockIdx.x * kScanDigits + threadIdx.x % kScanDigits, r = threadIdx.x / kScanDigits;
    const uint32_t per = (tiles + kScanRuns - 1u) / kScanRuns;
    const uint32_t t0 = min(r * per, tiles), t1 = min(t0 + per, tiles);
    uint32_t sum = 0u;
#pragma unroll 8
    for (uint32_t t = t0; t < t1; t++) sum += hist[size_t(t) * digits + d];
    run[r][threadIdx.x % kScanDigits] = sum;
    __syncthreads();
    uint32_t before = 0u, all = 0u;
#pragma unroll 8
    for (uint32_t q = 0; q < kScanRuns; q++) {
        const uint32_t v = run[q][threadIdx.x % kScanDigits];
        before += q < r ? v : 0u;
        all += v;
    }
    if (r == 0u) total[d] = all;
#pragma unroll 8
    for (uint32_t t = t0; t < t1; t++) {
        const uint32_t v = hist[size_t(t) * digits + d];
        hist[size_t(t) * digits + d] = before;
        before += v;
    }
}

// SELF: hist holds the tiles' counts; otherwise their exclusive scan, with the totals beside it.
template <int D, bool SELF>
__global__ void __launch_bounds__(kSortThreads) k_radix_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                              uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n,
                                                              int shift, const uint32_t* __restrict__ hist, uint32_t tiles,
                                                              const uint32_t* __restrict__ total) {
    constexpr uint32_t kDigits = 1u << D;
    constexpr uint32_t kPer = (kDigits + kSortThreads - 1u) / kSortThreads;  // digits per thread, neighbours
    __shared__ uint32_t cnt[kSortWaves][kDigits];
    __shared__ uint32_t ws[kSortWaves];
    const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const uint32_t first = blockIdx.x * kSortTile + w * (64u * kSortRounds) + lane;
    uint32_t key[kSortRounds], val[kSortRounds], rank[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; r++) {
        const uint32_t i = first + 64u * r;
        key[r] = i < n ? kin[i] : 0u;
        val[r] = i < n ? vin[i] : 0u;
    }
    const uint32_t d0 = t * kPer;
    uint32_t before[kPer], tot[kPer], sum = 0u;
#pragma unroll
    for (uint32_t q = 0; q < kPer; q++) before[q] = tot[q] = 0u;
    if (d0 < kDigits) {
        if constexpr (SELF) {
#pragma unroll 8
            for (uint32_t b = 0; b < tiles; b++)
#pragma unroll
                for (uint32_t q = 0; q < kPer; q++) {
                    const uint32_t h = hist[size_t(b) * kDigits + d0 + q];
                    before[q] += b < blockIdx.x ? h : 0u;
                    tot[q] += h;
                }
        } else {
#pragma unroll
            for (uint32_t q = 0; q < kPer; q++) {
                before[q] = hist[size_t(blockIdx.x) * kDigits + d0 + q];
                tot[q] = total[d0 + q];
            }
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < kPer; q++) {
        before[q] += sum;
        sum += tot[q];
    }
    for (uint32_t c = t; c < kSortWaves * kDigits; c += kSortThreads) cnt[0][c] = 0u;
    const uint32_t base = block_incl_scan<kSortWaves>(sum, ws) - sum;  // (its barriers follow the clearing)
#pragma unroll
    for (int r = 0; r < kSortRounds; r++)
        rank[r] = wave_rank<D>((key[r] >> shift) & (kDigits - 1u), first + 64u * r < n, cnt[w]);
    __syncthreads();
    if (d0 < kDigits) {
#pragma unroll
        for (uint32_t q = 0; q < kPer; q++) {
            uint32_t at = base + before[q];
#pragma unroll
            for (int v = 0; v < kSortWaves; v++) {
                const uint32_t c = cnt[v][d0 + q];
                cnt[v][d0 + q] = at;
                at += c;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; r++)
        if (first + 64u * r < n) {
            const uint32_t at = cnt[w][(key[r] >> shift) & (kDigits - 1u)] + rank[r];
            kout[at] = key[r];
            vout[at] = val[r];
        }
}

// ===================================================================== hashing
// Keys of a set held in id order. With several scenes the scene index sits above the cell
// bits (scene << shift), so a sort keeps every scene contiguous; `scene` is null for one.
__global__ void __launch_bounds__(kBlock) k_cell_keys(const float4* __restrict__ pos, uint32_t n, HashGeom g, int morton,
                                                    const uint32_t* __restrict__ scene, int shift,
                                                    uint32_t* __restrict__ key, uint32_t* __restrict__ id) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = pos[i];
    const i3 c = grid_pos(p.x, p.y, p.z, g);
    const uint32_t k = morton ? grid_zindex(c, g) : grid_index(c.x, c.y, c.z, g);
    key[i] = scene ? (scene[i] << shift) | k : k;
    id[i] = i;
}

// Keys of particles held in slot order, written at their reference index: keyref[perm[s]]
// (scene index above the cell bits). Padding slots between scenes (perm = kEmpty) are skipped.
__global__ void __launch_bounds__(kBlock) k_cell_keys_slots(const float4* __restrict__ pos, const uint32_t* __restrict__ perm,
                                                          uint32_t n, HashGeom g, int morton, const uint32_t* __restrict__ blk_scene,
                                                          int shift, uint32_t* __restrict__ keyref, uint32_t* __restrict__ iota) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    iota[s] = s;
    const uint32_t ref = perm[s];
    if (ref == kEmpty) return;
    const float4 p = pos[s];
    const i3 c = grid_pos(p.x, p.y, p.z, g);
    const uint32_t k = morton ? grid_zindex(c, g) : grid_index(c.x, c.y, c.z, g);
    keyref[ref] = (blk_scene[blockIdx.x] << shift) | k;
}
// Morton code of the (wrapped) cell of each slot, written at the slot's reference index;
// sorting by it keeps each cell contiguous and blocks of slots spatially compact.
__device__ __forceinline__ uint32_t cell_morton(i3 c, const HashGeom& g) {
    const uint32_t x = static_cast<uint32_t>(c.x) & (g.hx - 1u);
    const uint32_t y = static_cast<uint32_t>(c.y) & (g.hy - 1u);
    const uint32_t z = static_cast<uint32_t>(c.z) & (g.hz - 1u);
    return split_by3(x) | (split_by3(y) << 1u) | (split_by3(z) << 2u);
}
// First launch of the fluid hash: empties the cell table of the last one and writes the new keys.
__global__ void __launch_bounds__(kBlock) k_fluid_keys(const float4* __restrict__ pos, const uint32_t* __restrict__ perm, uint32_t n,
                                                     HashGeom g, const uint32_t* __restrict__ blk_scene, int shift,
                                                     uint32_t* __restrict__ keyref, uint32_t* __restrict__ iota,
                                                     const uint32_t* __restrict__ mkey, const uint32_t* __restrict__ lkey,
                                                     uint32_t n_old, uint32_t* __restrict__ start, uint32_t* __restrict__ end) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n_old) {
        const uint32_t m = mkey[s];
        if (m != kEmpty && (s == 0 || mkey[s - 1] != m)) start[lkey[s]] = end[lkey[s]] = kEmpty;
    }
    if (s >= n) return;
    iota[s] = s;
    const uint32_t ref = perm[s];
    if (ref == kEmpty) return;
    const float4 p = pos[s];
    keyref[ref] = (blk_scene[blockIdx.x] << shift) | cell_morton(grid_pos(p.x, p.y, p.z, g), g);
}
// Last launch of the fluid hash: sorted position q (key[q], reference id id[q]) -> slot
// q + delta[scene], where scene s's sorted range [cum_s, cum_s + count_s) lands on its slots
// [begin_s, end_s). A thread takes its particle's whole state from the old slot (src) to the new
// one, relabels it (perm, inv; no other thread reads or writes this particle's inv) and enters the
// bounds of its run in the cell table, which is indexed by scene * C + the reference's linear cell
// key (lkey keeps that index for clearing and for exporting the hash). Padding slots keep
// kEmpty in perm, src and mkey. One pass for what were twelve launches (the labels, a gather per array,
// the inverse, the table), each of which read src again: 250 particles 45 -> 5 us, 33 k 53 -> 12; 1 M
// 81 -> 44, 4 TB/s of the 176 bytes per particle, whose loads follow inv in groups of a cell.
__global__ void __launch_bounds__(kBlock) k_fluid_reorder(const uint32_t* __restrict__ key, const uint32_t* __restrict__ id,
                                                        uint32_t nref, HashGeom g, int shift, uint32_t C,
                                                        const uint32_t* __restrict__ delta, uint32_t* __restrict__ inv,
                                                        uint32_t* __restrict__ perm, uint32_t* __restrict__ src,
                                                        uint32_t* __restrict__ mkey, uint32_t* __restrict__ lkey,
                                                        uint32_t* __restrict__ hash_perm, uint32_t* __restrict__ start,
                                                        uint32_t* __restrict__ end, launch::FluidMove mv) {
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nref) return;
    const uint32_t k = key[q], ref = id[q];
    const uint32_t o = inv[ref];
    const uint32_t slot = q + delta[k >> shift];
    float4 a[4];
    float b[5];
#pragma unroll
    for (int v = 0; v < 4; v++) a[v] = mv.from4[v][o];
#pragma unroll
    for (int v = 0; v < 5; v++) b[v] = mv.from1[v][o];
    perm[slot] = ref;
    inv[ref] = slot;
    src[slot] = o;
    mkey[slot] = k;
    hash_perm[q] = ref;
#pragma unroll
    for (int v = 0; v < 4; v++) mv.to4[v][slot] = a[v];
#pragma unroll
    for (int v = 0; v < 5; v++) mv.to1[v][slot] = b[v];
    const i3 c = grid_pos(a[0].x, a[0].y, a[0].z, g);
    const uint32_t t = (k >> shift) * C + grid_index(c.x, c.y, c.z, g);
    lkey[slot] = t;
    if (q == 0 || key[q - 1] != k) start[t] = slot;
    if (q == nref - 1 || key[q + 1] != k) end[t] = slot + 1;
}
// inv[perm[s]] = s (padding slots skipped)
__global__ void __launch_bounds__(kBlock) k_invert(const uint32_t* __restrict__ perm, uint32_t n, uint32_t* __restrict__ inv) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && perm[s] != kEmpty) inv[perm[s]] = s;
}
// perm[s] = map[perm[s]]  (relabel reference ids after a Z-sort)
__global__ void __launch_bounds__(kBlock) k_relabel(uint32_t* __restrict__ perm, const uint32_t* __restrict__ map, uint32_t n) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && perm[s] != kEmpty) perm[s] = map[perm[s]];
}
__global__ void __launch_bounds__(kBlock) k_fill_u32(uint32_t* __restrict__ p, size_t n, uint32_t v) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Reset only the cells that the previous sorted keys occupied.
__global__ void __launch_bounds__(kBlock) k_clear_cells(const uint32_t* __restrict__ key, uint32_t n, uint32_t* __restrict__ start,
                                                      uint32_t* __restrict__ end) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t k = key[s];
    if (s == 0 || key[s - 1] != k) {
        start[k] = kEmpty;
        end[k] = kEmpty;
    }
}

// ReorderHash_kernel (MPSSpatialHash.cuh:115-145) + positions in key order.
__global__ void __launch_bounds__(kBlock) k_cell_table(const uint32_t* __restrict__ key, const uint32_t* __restrict__ id, uint32_t n,
                                                     uint32_t* __restrict__ start, uint32_t* __restrict__ end,
                                                     const float4* __restrict__ pos, float4* __restrict__ spos) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t k = key[s];
    if (s == 0 || key[s - 1] != k) {
        start[k] = s;
        if (s > 0) end[key[s - 1]] = s;
    }
    if (s == n - 1) end[k] = n;
    if (spos) spos[s] = pos[id[s]];
}

// 27-cell scan (Research, MPSSpatialHash.cuh:47-80): z outer, y, x inner; slots in key order.
// Neighbour when |x_i - x_j| < (4 r_i + 4 r_j) * 0.5, self excluded when SELF.
// The 27 (start, end) pairs are loaded up front, so their latencies overlap instead of
// adding up cell after cell; candidates are read two at a time for the same reason. Lists
// are written in the layout LAYOUT.
// Neighbour test of the reference: |x_i - x_j| < (h_i + h_j) / 2 with h = 4 r.
// sqrt is monotone and correctly rounded: far from the cut-off the squared distance decides;
// near it the exact test of the reference runs.
__device__ __forceinline__ bool within(const float4& xi, float ri, const float4& q) {
    const float ddx = xi.x - q.x, ddy = xi.y - q.y, ddz = xi.z - q.z;
    const float dd = (ddx * ddx + ddy * ddy) + ddz * ddz;
    const float rj = q.w * 4.0f;
    const float thr = (ri + rj) * 0.5f;
    const float t2 = thr * thr;
    if (dd < t2 * 0.9999f) return true;
    if (dd > t2 * 1.0001f) return false;
    return __builtin_sqrtf(dd) < thr;
}

// The neighbour test of one radius against squared distances: sqrt(dd) < thr exactly when
// dd < cut_of(thr). The square root is monotone and correctly rounded, so the distances that pass are
// those below one float, the smallest x with sqrt(x) >= thr; it lies within 2 ulp of the rounded
// thr * thr (sqrt(x) rounds up to thr from (thr - ulp/2)^2 on), and the search for it starts above.
__device__ __forceinline__ float cut_of(float thr) {
    float x = thr * thr;
    x = __uint_as_float(__float_as_uint(x) + (x < 3.0e38f ? 2u : 0u));
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const float y = __uint_as_float(__float_as_uint(x) - (x > 0.0f ? 1u : 0u));
        if (__builtin_sqrtf(y) >= thr) x = y;
    }
    return x;
}
// m = 2 m + (dd < cut): the hits of a run collect from its first copy in the top bit down. A NaN
// distance is no hit.
__device__ __forceinline__ void push_hit(uint32_t& m, float dd, float cut) {
    asm("v_cmp_lt_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(dd), "v"(cut) : "vcc");
}

// Where a search puts its lists: rows of K slots (out[i*K + k]), columns (out[k*stride + i]) or
// groups of four entries (ell()).
enum ListLayout { kRows, kCols, kGroups };
template <int LAYOUT>
__device__ __forceinline__ size_t list_at(uint32_t k, uint32_t i, uint32_t K, uint32_t stride) {
    if constexpr (LAYOUT == kRows) return size_t(i) * K + k;
    else if constexpr (LAYOUT == kCols) return size_t(k) * stride + i;
    else return ell(k, i, stride);
}

template <bool SELF, int LAYOUT>
__device__ __forceinline__ uint32_t search_cells(float4 xi, uint32_t i, const HashGeom& g, const uint32_t* __restrict__ start,
                                                 const uint32_t* __restrict__ end, const uint32_t* __restrict__ ids,
                                                 const float4* __restrict__ spos, uint32_t* __restrict__ out, uint32_t K,
                                                 uint32_t stride) {
    const i3 p = grid_pos(xi.x, xi.y, xi.z, g);
    const float ri = xi.w * 4.0f;
    uint32_t k = 0u;
    auto test = [&](float4 q, uint32_t s) {
        if (within(xi, ri, q)) {
            const uint32_t j = ids ? ids[s] : s;
            if (!(SELF && j == i)) {
                if (k < K) out[list_at<LAYOUT>(k, i, K, stride)] = j;
                k++;
            }
        }
    };
    // the 27 cells in the reference order; the loop stays rolled (an unrolled walk does not fit
    // the instruction cache)
#pragma unroll 1
    for (int t = 0; t < 27; t++) {
        const uint32_t c = grid_index(p.x + (t % 3) - 1, p.y + (t / 3) % 3 - 1, p.z + t / 9 - 1, g);
        uint32_t s = start[c];
        const uint32_t e = end[c];
        // an empty cell has start = end = 0xFFFFFFFF: only e - s (never s + 1) is formed,
        // and only once s < e is known
        if (s < e) {
            for (; e - s >= 2u; s += 2) {
                const float4 q0 = spos[s], q1 = spos[s + 1];
                test(q0, s);
                test(q1, s + 1);
            }
            if (s < e) test(spos[s], s);
        }
    }
    return k;
}

// Per-workgroup (largest count, sum of counts) of up to two lists, written to st[blk] and
// st[n + blk]; k_count_fold reduces them (no same-address atomics from every wave).
template <int L, uint32_t NW = kBlock / 64>
__device__ __forceinline__ void block_counts(const uint32_t (&c)[L], uint2* __restrict__ st, uint32_t n, uint32_t blk) {
    __shared__ uint32_t wm[L][NW], ws[L][NW];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
    for (int l = 0; l < L; l++) {
        uint32_t mx = c[l], sm = c[l];
        for (int off = 32; off > 0; off >>= 1) {
            mx = max(mx, (uint32_t)__shfl_xor((int)mx, off, 64));
            sm += (uint32_t)__shfl_xor((int)sm, off, 64);
        }
        if (lane == 0) {
            wm[l][wave] = mx;
            ws[l][wave] = sm;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int l = 0; l < L; l++) {
            uint32_t mx = 0u, sm = 0u;
            for (uint32_t w = 0; w < NW; w++) {
                mx = max(mx, wm[l][w]);
                sm += ws[l][w];
            }
            st[size_t(l) * n + blk] = make_uint2(mx, sm);
        }
    }
}

// The counts of a search over its workgroups' records: workgroup l of the launch folds list l into
// maxc[l] and nnz[l]. The fluid search's launch has a third workgroup, which counts its halos (hn):
// stats[0] = largest staged, [1] = not staged, [2] = blocks with neighbours, [3] = staged but deeper
// than kHaloShallow (blocks left to k_halo_build are counted after it).
constexpr int kCountFoldThreads = 1024;
__global__ void __launch_bounds__(kCountFoldThreads) k_count_fold(const uint2* __restrict__ st, uint32_t n, uint32_t* maxc,
                                                                unsigned long long* nnz, const uint32_t* __restrict__ hn,
                                                                uint32_t* __restrict__ stats) {
    if (blockIdx.x == 2u) {
        fold_halo_stats(hn, n, stats);
        return;
    }
    __shared__ uint32_t wm[kCountFoldThreads / 64];
    __shared__ unsigned long long ws[kCountFoldThreads / 64];
    uint32_t mx = 0u;
    unsigned long long sm = 0ull;
    st += size_t(blockIdx.x) * n;
    constexpr uint32_t R = 4;  // records of a thread in flight
    for (uint32_t k0 = threadIdx.x; k0 < n; k0 += R * blockDim.x) {
        uint2 v[R];
#pragma unroll
        for (uint32_t q = 0; q < R; q++) {
            const uint32_t k = k0 + q * blockDim.x;
            v[q] = k < n ? st[k] : make_uint2(0u, 0u);
        }
#pragma unroll
        for (uint32_t q = 0; q < R; q++) {
            mx = max(mx, v[q].x);
            sm += v[q].y;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, off, 64));
        sm += __shfl_xor(sm, off, 64);
    }
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0) {
        wm[wave] = mx;
        ws[wave] = sm;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < blockDim.x / 64; w++) {
            mx = max(mx, wm[w]);
            sm += ws[w];
        }
        maxc[blockIdx.x] = mx;
        nnz[blockIdx.x] = sm;
    }
}

// Scene s's cells are entries [s*C, (s+1)*C) of both tables.
//
// A workgroup owns 256 consecutive fluid slots (sorted by cell, so each cell's particles are
// one run). The first particle of each run registers the 9 (y, z) rows of its 27 cells in an
// LDS hash of the block's rows (a row keyed by its wrapped y, z), widening the row's x range to
// cover x-1..x+1. Each row's cells are then numbered in x order over that range, each cell's
// bounds are read once, and all fluid (then wall) particles of those cells are staged in LDS
// in that order, each with its slot (a wall particle: its id) in place of the radius. So the
// three cells x-1, x, x+1 of any row of a particle are one contiguous run of staged copies, and
// every particle walks its 27 cells in the reference order as 9 row runs: first a hit mask per
// run, then the hits of all runs as list entries. The staged copies that are anybody's hit are the
// block's halo (halo.hip): their slots in ascending order, and every list entry as a position
// among them, are written by the same kernel, which has the lists and the copies at hand.
//
// Q = 4 shares a slot among a quad of lanes, which take the runs 0..8 in turn.
//
// Staged fluid particles of several radii: a run's mask is made with the cut-off of the widest pair
// that the block can hold, then the radii of its hits are read and each is tested with its own.
// (1M particles of two radii, hash, search and density: 2110 us with such blocks left to the tables of a
// second pass, 985 with one lane per slot over the tables in the only pass, now 653.)
//
// A block may have more rows, cells or candidates than the LDS holds, or a run of more copies than a
// hit mask has bits. The first pass over many blocks (LAST false) leaves such a block alone
// (n = kHaloLeft); a second one, with room for more and a quad per slot, takes it, and searches the
// global tables for a set that does not fit even there. The first pass does so itself where waiting
// would not help: walls of several radii, more candidates than the second pass holds, cells far wider
// than the support (kWideCell; 257k particles, cells of two supports 581 us against 778, of three 1599
// against 1994), and, where many blocks have too many rows or cells (scattered particles, a hash that
// wraps the scene around), whatever does not fit (1M scattered particles, one to a cell: 944 us for hash,
// search and density with a second pass, 568 without). The halo of a block whose fluid was searched in
// the tables is left to k_halo_build. The lists are the same whichever way.
//
// Bound by its vector instructions and LDS latency: of the ~50 us that a workgroup takes (1M
// particles, four workgroups per CU) the distance tests are 13, writing the lists 9, the halo 15,
// registering rows and staging 14. Search and halos together, before (a search of its own and
// k_halo_build) -> now: 250 particles 97 -> 48 us, 33k 207 -> 57, 45k near rest density 365 -> 75, 257k
// 179 -> 110, 525k near rest density 630 -> 343, 1M 433 -> 330.
template <uint32_t HASH_BITS, uint32_t ROWS, uint32_t CELLS, uint32_t CAND, uint32_t WORDS>
struct SearchCaps {
    static constexpr uint32_t kHashBits = HASH_BITS, kRowHash = 1u << HASH_BITS;
    static constexpr uint32_t kRows = ROWS, kCells = CELLS, kCand = CAND;
    static constexpr uint32_t kWords = WORDS, kRun = 32u * WORDS;  // a run's hit mask
};
// Near rest density a block has 1500-2700 candidates; particles in thin sheets give up to 200 rows
// and 850 cells; a cell at the origin is two cells wide (coordinates are truncated towards 0), so
// there a run can hold over 100 copies.
using SearchStd = SearchCaps<7, 96, 384, 1920, 3>;     // 39 KB: four workgroups per CU
using SearchDense = SearchCaps<7, 96, 384, 2752, 3>;   // 52 KB: three (525k near rest density: 437 -> 343 us)
using SearchWide = SearchCaps<9, 224, 1024, 3328, 8>;  // 78 KB: two
constexpr uint32_t kWideCell = 32;                   // a cell with more fluid is a wide one (one support wide: up to 20)
constexpr uint32_t kSrchPad = 4;                     // a group of four read at the end of a run stays in the array
constexpr uint32_t kNoRow = 0xFFFFFFFFu;
// Bits of a block's `mixed` beside 1 and 2 (fluid, walls of several radii): k_halo_build has to do its
// halo; it has a wide cell; the first pass leaves it to the second.
constexpr uint32_t kNoHalo = 4u, kWideCells = 8u, kLeave = 16u;
constexpr uint32_t kHit = 0x80000000u;  // marks a staged fluid copy that is in a list (slots are below 2^31)

// Inclusive scan of a 64-bit value over the workgroup's NW waves; `ws` holds NW wave totals
// (synchronise before reusing it). `total` receives the block's sum.
template <uint32_t NW>
__device__ __forceinline__ unsigned long long block_scan_u64(unsigned long long v, unsigned long long* ws,
                                                             unsigned long long& total) {
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    for (uint32_t off = 1; off < 64u; off <<= 1) {
        const uint32_t lo = __shfl_up(static_cast<uint32_t>(v), off, 64);
        const uint32_t hi = __shfl_up(static_cast<uint32_t>(v >> 32), off, 64);
        if (lane >= off) v += (static_cast<unsigned long long>(hi) << 32) | lo;
    }
    if (lane == 63u) ws[w] = v;
    __syncthreads();
    total = 0ull;
    for (uint32_t q = 0; q < NW; q++) {
        if (q < w) v += ws[q];
        total += ws[q];
    }
    return v;
}

template <int L>
__device__ __forceinline__ uint32_t quad_u32(uint32_t v) {  // the value of lane L of the quad
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), L * 0x55, 0xF, 0xF, true));
}
__device__ __forceinline__ uint32_t quad_sum(uint32_t v) { return quad_u32<0>(v) + quad_u32<1>(v) + quad_u32<2>(v) + quad_u32<3>(v); }
// Sum over the quad's lanes before lane l (every lane reads every other: no lane may be masked off).
__device__ __forceinline__ uint32_t quad_before(uint32_t v, uint32_t l) {
    const uint32_t a = quad_u32<0>(v), b = quad_u32<1>(v), c = quad_u32<2>(v);
    return (l > 0u ? a : 0u) + (l > 1u ? b : 0u) + (l > 2u ? c : 0u);
}

// search_cells by a quad of lanes: every lane takes a candidate of each four (two fours in flight), and
// the hits of a four enter the list in candidate order. The count is valid in every lane.
template <bool SELF, int LAYOUT>
__device__ __forceinline__ uint32_t search_cells_quad(float4 xi, uint32_t i, uint32_t l, const HashGeom& g,
                                                      const uint32_t* __restrict__ start, const uint32_t* __restrict__ end,
                                                      const uint32_t* __restrict__ ids, const float4* __restrict__ spos,
                                                      uint32_t* __restrict__ out, uint32_t K, uint32_t stride) {
    const i3 p = grid_pos(xi.x, xi.y, xi.z, g);
    const float ri = xi.w * 4.0f;
    uint32_t k = 0u;
#pragma unroll 1
    for (int t = 0; t < 27; t++) {
        const uint32_t c = grid_index(p.x + (t % 3) - 1, p.y + (t / 3) % 3 - 1, p.z + t / 9 - 1, g);
        const uint32_t s0 = start[c], e = end[c];
        const uint32_t n = s0 < e ? e - s0 : 0u;  // (the same in the four lanes, as are all counts)
        for (uint32_t o = 0; o < n; o += 8u) {
            float4 q[2];
#pragma unroll
            for (uint32_t h = 0; h < 2u; h++) q[h] = spos[s0 + min(o + 4u * h + l, n - 1u)];
#pragma unroll
            for (uint32_t h = 0; h < 2u; h++) {
                const uint32_t at = o + 4u * h + l;
                bool hit = at < n && within(xi, ri, q[h]);
                uint32_t j = s0 + at;
                if (hit && ids) j = ids[j];
                if (SELF && j == i) hit = false;
                const uint32_t one = hit ? 1u : 0u;
                const uint32_t pl = k + quad_before(one, l);
                if (hit && pl < K) out[list_at<LAYOUT>(pl, i, K, stride)] = j;
                k += quad_sum(one);
            }
        }
    }
    return k;
}

// The hits of one slot among its 9 row runs; with Q = 4 a lane holds the runs l, l + 4 and 8 (l = 0).
template <int Q, uint32_t WORDS>
struct RowHits {
    static constexpr uint32_t kRuns = Q == 1 ? 9 : 3;
    uint32_t lo[kRuns];             // first staged copy of each run
    uint32_t m[kRuns][WORDS];       // its hits, one bit per copy
    uint32_t at[kRuns];             // list position of its first hit
    uint32_t count;                 // hits of all runs

    // run(r) gives the [lo, hi) of run r; `self` is the slot's own staged copy (any other value:
    // none); a copy is a hit when its squared distance is below `cut` and, with `sift` set, the copy
    // passes drop() too. False if a run is too long for its mask (for the whole quad).
    template <class Run, class Drop>
    __device__ __forceinline__ bool test(const float4* cand, uint32_t l, const float4& xi, float cut, uint32_t self, Run&& run,
                                         bool sift, Drop&& drop) {
        uint32_t over = 0u, n[kRuns];
#pragma unroll
        for (uint32_t q = 0; q < kRuns; q++) {
            const uint32_t r = Q == 1 ? q : l + 4u * q;
            uint32_t a = 0u, b = 0u;
            if (r < 9u) run(r, a, b);
            lo[q] = a;
            over |= b - a > 32u * WORDS ? 1u : 0u;
            n[q] = 0u;
#pragma unroll
            for (uint32_t w = 0; w < WORDS; w++) {
                uint32_t mm = 0u;
                const uint32_t c0 = a + 32u * w;
                if (c0 < b) {
                    const uint32_t len = min(b - c0, 32u);
                    uint32_t k = 0;
                    for (; k < len; k += 4u) {
                        float4 v[4];
#pragma unroll
                        for (uint32_t e = 0; e < 4u; e++) v[e] = cand[c0 + k + e];  // <= hi + 2 < array size
#pragma unroll
                        for (uint32_t e = 0; e < 4u; e++) {
                            const float dx = xi.x - v[e].x, dy = xi.y - v[e].y, dz = xi.z - v[e].z;
                            push_hit(mm, (dx * dx + dy * dy) + dz * dz, cut);
                        }
                    }
                    mm = __brev(mm) >> (32u - k);                // bit e: copy c0 + e
                    mm &= len < 32u ? (1u << len) - 1u : ~0u;  // the group of four read past hi
                    const uint32_t d = self - c0;
                    if (d < 32u) mm &= ~(1u << d);
                    if (sift) mm = sifted(mm, c0, drop);
                }
                m[q][w] = mm;
                n[q] += __popc(mm);
            }
        }
        if constexpr (Q == 1) {
            count = 0u;
#pragma unroll
            for (uint32_t q = 0; q < kRuns; q++) {
                at[q] = count;
                count += n[q];
            }
            return !over;
        } else {
            const uint32_t t0 = quad_sum(n[0]), t1 = quad_sum(n[1]);
            at[0] = quad_before(n[0], l);
            at[1] = t0 + quad_before(n[1], l);
            at[2] = t0 + t1;
            count = t0 + t1 + quad_sum(n[2]);
            return quad_sum(over) == 0u;
        }
    }
    // The bits e of mm whose copy c0 + e is kept: drop(copies) takes four at a time (a copy again where
    // fewer are left) and gives the set of those to drop.
    template <class Drop>
    static __device__ __forceinline__ uint32_t sifted(uint32_t mm, uint32_t c0, Drop&& drop) {
        for (uint32_t left = mm; left;) {
            uint32_t b[4], t[4];
#pragma unroll
            for (uint32_t e = 0; e < 4u; e++) {
                b[e] = left & (0u - left);  // the lowest bit
                left ^= b[e];
                t[e] = c0 + (b[e] ? static_cast<uint32_t>(__builtin_ctz(b[e])) : 0u);
            }
            const uint32_t out = drop(t);
#pragma unroll
            for (uint32_t e = 0; e < 4u; e++) mm &= (out >> e) & 1u ? ~b[e] : ~0u;
        }
        return mm;
    }
    // use(list position, staged copy) for every hit, in list order within a run
    template <class Use>
    __device__ __forceinline__ void each(Use&& use) const {
#pragma unroll
        for (uint32_t q = 0; q < kRuns; q++) {
            uint32_t k = at[q];
#pragma unroll
            for (uint32_t w = 0; w < WORDS; w++) {
                uint32_t b = m[q][w];
                while (b) {
                    const uint32_t t = lo[q] + 32u * w + static_cast<uint32_t>(__builtin_ctz(b));
                    b &= b - 1u;
                    use(k, t);
                    k++;
                }
            }
        }
    }
};

//
// mode: of the first pass which blocks it leaves (SearchLeave); of the last 1 if it takes only those.
template <int Q, class Caps, bool LAST>
__global__ void __launch_bounds__(Q * kBlock) k_neighbors_fluid(const float4* __restrict__ pos, Scenes sc, uint32_t C, HashGeom g,
                                                          HashView fl, HashView bd, uint32_t* __restrict__ nff, uint32_t Kff,
                                                          uint32_t* __restrict__ cff, uint32_t* __restrict__ nfb, uint32_t Kfb,
                                                          uint32_t* __restrict__ cfb, uint2* __restrict__ bstat,
                                                          launch::HaloOut ho, int mode, NbrCounters* __restrict__ ctr) {
    constexpr uint32_t kThreads = Q * kBlock, kWaves = kThreads / 64u;
    constexpr uint32_t kRowHash = Caps::kRowHash, kRows = Caps::kRows, kCells = Caps::kCells, kCand = Caps::kCand;
    constexpr uint32_t kCellsPer = (kCells + kThreads - 1u) / kThreads;  // cells per thread
    static_assert(kRows <= kThreads && kRows <= 255u + 1u && kRows < kRowHash, "one row per thread");
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    if (LAST && mode && ho.n[blk] != kHaloLeft) return;  // the first pass did this block
    const uint32_t tid = threadIdx.x;
    const uint32_t i = blk * kBlock + tid / Q;
    const uint32_t l = tid % Q;
    const uint32_t N = sc.N;
    const uint32_t sid = sc.blk_scene[blk];
    const uint32_t end = sc.P[sid].end;
    const bool live = i < end;
    const size_t base = size_t(sid) * C;
    const uint32_t* fstart = fl.start + base;
    const uint32_t* fend = fl.end + base;
    const uint32_t* bstart = bd.start + base;
    const uint32_t* bend = bd.end + base;
    __shared__ uint32_t rkey[kRowHash];      // row hash: wrapped key of the row's cell x = 0
    __shared__ int rxlo[kRowHash], rxhi[kRowHash];  // the row's x range (unwrapped)
    __shared__ uint16_t rbase[kRowHash];     // the row's first cell
    __shared__ uint16_t rslot[kRows];        // hash slot of each row, in registration order
    static_assert(kCells % 8u == 0u, "the halo pass reads eight cells at a time");
    __shared__ __align__(16) uint32_t ecell[kCells], efs[kCells], ebs[kCells];
    __shared__ uint16_t efo[kCells + 1], ebo[kCells + 1];
    __shared__ float4 cand[kCand + kSrchPad];
    __shared__ unsigned long long ws[kWaves];
    __shared__ uint32_t nrow, mixed, first[2];  // first: first cell with fluid, with walls
    __shared__ uint32_t widest;  // largest |radius| of the fluid copies that differ from the first, as bits
    auto row_hash = [](uint32_t c) -> uint32_t { return (c * 2654435761u) >> (32u - Caps::kHashBits); };
    for (uint32_t t = tid; t < kRowHash; t += kThreads) {
        rkey[t] = kNoRow;
        rxlo[t] = 0x7FFFFFFF;
        rxhi[t] = -0x7FFFFFFF - 1;
    }
    if (tid == 0) {
        widest = 0u;
        nrow = 0u;
        mixed = 0u;
        first[0] = first[1] = kNoRow;
    }
    const float4 xi = live ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const i3 p = grid_pos(xi.x, xi.y, xi.z, g);
    bool leader = live;
    if (live && tid >= Q) {
        const float4 xp = pos[i - 1];
        const i3 pp = grid_pos(xp.x, xp.y, xp.z, g);
        leader = pp.x != p.x || pp.y != p.y || pp.z != p.z;
    }
    __syncthreads();
    // 1. rows (inserts stop once the block is known to be over the cap, so the table never
    //    fills; every probe loop is bounded anyway)
    if (leader) {
        for (uint32_t r = l; r < 9u; r += Q) {
            if (*(volatile uint32_t*)&nrow > kRows) break;
            const uint32_t k = grid_index(0, p.y + int(r % 3u) - 1, p.z + int(r / 3u) - 1, g);
            uint32_t h = row_hash(k);
            for (uint32_t probe = 0; probe < kRowHash; probe++) {
                if (probe > 7u && *(volatile uint32_t*)&nrow > kRows) break;  // (a probe of a full table is long)
                const uint32_t prev = atomicCAS(&rkey[h], kNoRow, k);
                if (prev == kNoRow) {
                    const uint32_t e = atomicAdd(&nrow, 1u);
                    if (e < kRows) rslot[e] = static_cast<uint16_t>(h);
                }
                if (prev == kNoRow || prev == k) {
                    atomicMin(&rxlo[h], p.x - 1);
                    atomicMax(&rxhi[h], p.x + 1);
                    break;
                }
                h = (h + 1u) & (kRowHash - 1u);
            }
        }
    }
    __syncthreads();
    const uint32_t nr = nrow;
    // (in a grid one cell wide a run holds the particle's own cell three times, but `self` is one copy of it)
    bool staged = nr <= kRows && g.hx > 1u;
    // whether what cannot be walked in LDS searches the global tables here, and is not left to a second pass
    bool tables = LAST || mode == launch::kLeaveNone || (mode != launch::kLeaveAll && !staged);
    uint32_t nc = 0u;
    // 2. number each row's cells over its x range (rows in registration order)
    if (staged) {
        const uint32_t h = tid < nr ? rslot[tid] : 0u;
        const uint32_t len = tid < nr ? static_cast<uint32_t>(min(static_cast<long long>(rxhi[h]) - rxlo[h] + 1,
                                                                 static_cast<long long>(kCells) + 1)) : 0u;
        unsigned long long tot;
        const uint32_t b0 = static_cast<uint32_t>(block_scan_u64<kWaves>(len, ws, tot)) - len;
        nc = static_cast<uint32_t>(tot);
        staged = nc <= kCells;
        tables |= mode != launch::kLeaveAll && !staged;
        if (staged && tid < nr) {
            rbase[h] = static_cast<uint16_t>(b0);
            if (len > g.hx) atomicOr(&mixed, kNoHalo);  // the row wraps around: a cell is staged twice (see 6.)
            const uint32_t k0 = rkey[h];
            for (uint32_t q = 0; q < len; q++) ecell[b0 + q] = k0 + (static_cast<uint32_t>(rxlo[h] + static_cast<int>(q)) & (g.hx - 1u));
        }
        __syncthreads();
    }
    if (!LAST && !staged && tid == 0) atomicAdd(&ctr->spread, 1u);
    // 3. bounds of each cell (read once) and offsets of its staged copies: fluid from 0, walls
    //    after all fluid
    uint32_t tf = 0u, tb = 0u;
    if (staged) {
        uint32_t fc[kCellsPer], bc[kCellsPer], fsum = 0u, bsum = 0u;
#pragma unroll
        for (uint32_t q = 0; q < kCellsPer; q++) {
            const uint32_t e = kCellsPer * tid + q;
            fc[q] = bc[q] = 0u;
            if (e < nc) {
                const uint32_t c = ecell[e];
                const uint32_t s0 = fstart[c], s1 = fend[c];
                efs[e] = s0;
                fc[q] = s0 < s1 ? s1 - s0 : 0u;  // an empty cell has start = end = 0xFFFFFFFF
                if (bd.n) {
                    const uint32_t b0 = bstart[c], b1 = bend[c];
                    ebs[e] = b0;
                    bc[q] = b0 < b1 ? b1 - b0 : 0u;
                }
            }
            fsum += fc[q];
            bsum += bc[q];
            if (!LAST && fc[q] > kWideCell) atomicOr(&mixed, kWideCells);
        }
        const unsigned long long mine = (static_cast<unsigned long long>(bsum) << 32) | fsum;
        unsigned long long tot;
        const unsigned long long ex = block_scan_u64<kWaves>(mine, ws, tot) - mine;
        tf = static_cast<uint32_t>(tot & 0xFFFFFFFFull);
        tb = static_cast<uint32_t>(tot >> 32);
        staged = static_cast<unsigned long long>(tf) + tb <= kCand;
        tables |= static_cast<unsigned long long>(tf) + tb > SearchWide::kCand || (mixed & kWideCells);
        if (!LAST && tid == 0 && !tables && static_cast<unsigned long long>(tf) + tb > SearchStd::kCand) atomicAdd(&ctr->crowded, 1u);
        uint32_t fo = static_cast<uint32_t>(ex & 0xFFFFFFFFull), bo = static_cast<uint32_t>(ex >> 32);
        if (staged) {
            // each copy's w first holds its cell (read back by the staging pass)
#pragma unroll
            for (uint32_t q = 0; q < kCellsPer; q++) {
                const uint32_t e = kCellsPer * tid + q;
                if (e < nc) {
                    efo[e] = static_cast<uint16_t>(fo);
                    ebo[e] = static_cast<uint16_t>(tf + bo);
                    for (uint32_t k = 0; k < fc[q]; k++) cand[fo + k].w = __uint_as_float(e);
                    for (uint32_t k = 0; k < bc[q]; k++) cand[tf + bo + k].w = __uint_as_float(e);
                    if (fc[q]) atomicMin(&first[0], e);
                    if (bc[q]) atomicMin(&first[1], e);
                }
                fo += fc[q];
                bo += bc[q];
            }
            if (tid == 0) {
                efo[nc] = static_cast<uint16_t>(tf);
                ebo[nc] = static_cast<uint16_t>(tf + tb);
            }
        }
        __syncthreads();
    }
    // 4. stage the candidates with their ids (copy t of cell e is particle efs[e] + t - efo[e]),
    //    kStage loads of a thread in flight. `mixed` records whether some fluid (bit 0) or wall (bit 1)
    //    candidate has another radius than the first staged candidate of its set.
    float rf = 0.0f, rw = 0.0f;  // the first fluid's radius, the walls' common one
    if (staged) {
        constexpr uint32_t kStage = 4;
        uint32_t mx = 0u;
        float rmax = 0.0f;
        auto stage = [&](uint32_t t_lo, uint32_t t_hi, const uint32_t* es, const uint16_t* eo, const float4* from, const uint32_t* id,
                         float r0, uint32_t bit) {
            for (uint32_t t0 = t_lo + tid; t0 < t_hi; t0 += kStage * kThreads) {
                float4 v[kStage];
                uint32_t s[kStage];
#pragma unroll
                for (uint32_t q = 0; q < kStage; q++) {
                    const uint32_t t = t0 + q * kThreads;
                    if (t < t_hi) {
                        const uint32_t e = __float_as_uint(cand[t].w);
                        s[q] = es[e] + (t - eo[e]);
                        v[q] = from[s[q]];
                        if (id) s[q] = id[s[q]];
                    }
                }
#pragma unroll
                for (uint32_t q = 0; q < kStage; q++) {
                    const uint32_t t = t0 + q * kThreads;
                    if (t < t_hi) {
                        cand[t] = make_float4(v[q].x, v[q].y, v[q].z, __uint_as_float(s[q]));
                        mx |= v[q].w != r0 ? bit : 0u;
                        rmax = fmaxf(rmax, fabsf(v[q].w));  // (a NaN is nobody's neighbour)
                    }
                }
            }
        };
        if (tf) {
            rf = pos[efs[first[0]]].w;
            stage(0u, tf, efs, efo, pos, nullptr, rf, 1u);
            if (mx) atomicMax(&widest, __float_as_uint(rmax));
        }
        if (tb) {
            rw = bd.spos[ebs[first[1]]].w;
            stage(tf, tf + tb, ebs, ebo, bd.spos, bd.id, rw, 2u);
        }
        if (mx) atomicOr(&mixed, mx);
        __syncthreads();
    }
    // 5. the search proper: 9 rows (z, then y offsets), each the run of cells x-1, x, x+1
    uint32_t a = 0u, b = 0u;
    const uint32_t mix = staged ? mixed : 3u;
    const float ri = xi.w * 4.0f;
    // the particle's cell x + dx in row (y, z)
    auto cell_of = [&](int dx, int y, int z) -> uint32_t {
        const uint32_t k = grid_index(0, y, z, g);
        uint32_t h = row_hash(k);
#pragma unroll 1
        for (uint32_t probe = 0; probe < kRowHash && rkey[h] != k; probe++) h = (h + 1u) & (kRowHash - 1u);
        return rkey[h] == k ? rbase[h] + static_cast<uint32_t>(p.x + dx - rxlo[h]) : kNoRow;
    };
    auto run_of = [&](const uint16_t* eo, uint32_t r, uint32_t& lo, uint32_t& hi) {
        const uint32_t e = cell_of(-1, p.y + int(r % 3u) - 1, p.z + int(r / 3u) - 1);
        if (e == kNoRow) return;  // not reached: every row of a run was registered
        lo = eo[e];
        hi = eo[e + 3u];
    };
    // a fluid copy of another radius is a neighbour by the pair's own cut-off: its radius is read for the
    // hits of the widest pair only
    auto drop = [&](const uint32_t (&t)[4]) -> uint32_t {
        float4 q[4];
        float r[4];
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) q[e] = cand[t[e]];
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) r[e] = pos[__float_as_uint(q[e].w) & ~kHit].w;
        uint32_t out = 0u;
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) out |= within(xi, ri, make_float4(q[e].x, q[e].y, q[e].z, r[e])) ? 0u : 1u << e;
        return out;
    };
    RowHits<Q, Caps::kWords> hits;
    bool have = false;  // `hits` are this slot's fluid neighbours
    if (live) {
        if (staged) {
            const uint32_t eh = cell_of(0, p.y, p.z);
            const uint32_t self = eh == kNoRow ? kNoRow : efo[eh] + (i - efs[eh]);
            const bool sift = mix & 1u;
            const float rj = fmaxf(fabsf(rf), __uint_as_float(widest)) * 4.0f;
            have = hits.test(cand, l, xi, cut_of(sift ? (fabsf(ri) + rj) * 0.5f : (ri + ri) * 0.5f), self,
                             [&](uint32_t r, uint32_t& lo, uint32_t& hi) { run_of(efo, r, lo, hi); }, sift, drop);
        }
        if (have) {
            a = hits.count;
            hits.each([&](uint32_t k, uint32_t t) {
                const uint32_t s = __float_as_uint(cand[t].w) & ~kHit;
                cand[t].w = __uint_as_float(s | kHit);
                if (k < Kff) nff[ell(k, i, N)] = s;
            });
        } else if (tables) {
            if constexpr (Q == 1) a = search_cells<true, kGroups>(xi, i, g, fstart, fend, fl.id, fl.spos, nff, Kff, N);
            else a = search_cells_quad<true, kGroups>(xi, i, l, g, fstart, fend, fl.id, fl.spos, nff, Kff, N);
            atomicOr(&mixed, kNoHalo);
        } else {
            atomicOr(&mixed, kLeave);
        }
        if (bd.n) {
            if (staged && tb == 0u) {
                b = 0u;  // no wall particle in any cell of the block
            } else {
                RowHits<Q, Caps::kWords> wh;
                if (!(mix & 2u) && wh.test(cand, l, xi, cut_of((ri + rw * 4.0f) * 0.5f), kNoRow,
                                           [&](uint32_t r, uint32_t& lo, uint32_t& hi) { run_of(ebo, r, lo, hi); }, false,
                                           [](const uint32_t (&)[4]) -> uint32_t { return 0u; })) {
                    b = wh.count;
                    wh.each([&](uint32_t k, uint32_t t) {
                        if (k < Kfb) nfb[size_t(k) * N + i] = __float_as_uint(cand[t].w);
                    });
                } else if (tables || (staged && (mix & 2u))) {  // (no form stages walls of several radii)
                    if constexpr (Q == 1) b = search_cells<false, kCols>(xi, i, g, bstart, bend, bd.id, bd.spos, nfb, Kfb, N);
                    else b = search_cells_quad<false, kCols>(xi, i, l, g, bstart, bend, bd.id, bd.spos, nfb, Kfb, N);
                } else {
                    atomicOr(&mixed, kLeave);
                }
            }
        }
    }
    if (l == 0u && i < N) {
        cff[i] = a;
        cfb[i] = b;
    }
    // 6. the block's halo: the marked copies, cells in order of their first slot (cells are disjoint
    //    slot ranges, so that is ascending slot order; a block with a cell staged twice is left out)
    __syncthreads();
    const bool leave = (!staged && !tables) || (mixed & kLeave);
    if (leave || !staged || (mixed & kNoHalo)) {
        if (tid == 0) {
            ho.n[blk] = leave ? kHaloLeft : kHaloTodo;
            atomicAdd(leave ? &ctr->left : &ctr->todo, 1u);
        }
    } else {
        // marked copies of each cell (in ecell, no longer needed), then their sum over the cells with
        // smaller slots
        uint32_t mine = 0u;
#pragma unroll
        for (uint32_t q = 0; q < kCellsPer; q++) {
            const uint32_t e = kCellsPer * tid + q;
            if (e < nc) {
                uint32_t n = 0u;
                for (uint32_t t = efo[e]; t < efo[e + 1u]; t++) n += __float_as_uint(cand[t].w) >> 31;
                ecell[e] = n;
                if (efo[e + 1u] == efo[e]) efs[e] = 0xFFFFFFFFu;
                mine += n;
            } else if (e < kCells) {
                ecell[e] = 0u;
            }
        }
        unsigned long long tot;
        block_scan_u64<kWaves>(mine, ws, tot);  // (ends with every ecell written)
        const uint32_t H = static_cast<uint32_t>(tot);
        const bool fits = H <= ho.limit;
        if (tid == 0) ho.n[blk] = fits ? H : kHaloCap + 1u;
        if (fits) {
            uint32_t* out = ho.idx + size_t(blk) * kHaloCap;
            uint32_t from[kCellsPer];
#pragma unroll
            for (uint32_t q = 0; q < kCellsPer; q++) from[q] = 0u;
            const uint32_t e0 = kCellsPer * tid;
            if (e0 < nc) {
                uint32_t s[kCellsPer];
#pragma unroll
                for (uint32_t q = 0; q < kCellsPer; q++) s[q] = e0 + q < nc ? efs[e0 + q] : 0u;
                // four cells per read, two reads ahead (cells past nc count nothing)
                for (uint32_t e = 0; e < nc; e += 8u) {
                    uint4 se[2], n[2];
#pragma unroll
                    for (uint32_t h = 0; h < 2u; h++) {
                        se[h] = reinterpret_cast<const uint4*>(efs)[e / 4u + h];
                        n[h] = reinterpret_cast<const uint4*>(ecell)[e / 4u + h];
                    }
#pragma unroll
                    for (uint32_t h = 0; h < 2u; h++)
#pragma unroll
                        for (uint32_t q = 0; q < kCellsPer; q++)
                            from[q] += (se[h].x < s[q] ? n[h].x : 0u) + (se[h].y < s[q] ? n[h].y : 0u) +
                                       (se[h].z < s[q] ? n[h].z : 0u) + (se[h].w < s[q] ? n[h].w : 0u);
                }
            }
            __syncthreads();  // every position base is known before the copies' slots give way to positions
#pragma unroll
            for (uint32_t q = 0; q < kCellsPer; q++) {
                const uint32_t e = e0 + q;
                if (e < nc) {
                    uint32_t at = from[q];
                    for (uint32_t t = efo[e]; t < efo[e + 1u]; t++) {
                        const uint32_t w = __float_as_uint(cand[t].w);
                        if (w & kHit) {
                            out[at] = w & ~kHit;
                            cand[t].w = __uint_as_float(at);
                            at++;
                        }
                    }
                }
            }
            __syncthreads();
            if (have)
                hits.each([&](uint32_t k, uint32_t t) {
                    if (k < Kff) ho.nb16[ell(k, i, N)] = static_cast<uint16_t>(__float_as_uint(cand[t].w));
                });
        }
    }
    const uint32_t cnt[2] = {l == 0u ? a : 0u, l == 0u ? b : 0u};
    block_counts<2, kWaves>(cnt, bstat, gridDim.x, blk);
}

__global__ void __launch_bounds__(kBlock) k_neighbors_boundary(const float4* __restrict__ pos, uint32_t B,
                                                             const uint32_t* __restrict__ scene, uint32_t C, HashGeom g,
                                                             HashView bd, uint32_t* __restrict__ nbb, uint32_t Kbb,
                                                             uint32_t* __restrict__ cbb, uint2* __restrict__ bstat) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t a = 0u;
    if (i < B) {
        const size_t base = scene ? size_t(scene[i]) * C : 0;
        a = search_cells<true, kRows>(pos[i], i, g, bd.start + base, bd.end + base, bd.id, bd.spos, nbb, Kbb, B);
        cbb[i] = a;
    }
    const uint32_t cnt[1] = {a};
    block_counts<1>(cnt, bstat, gridDim.x, blockIdx.x);
}

// Ref lists of coupled fluid objects (SpatialHash::BuildNeighorhood(obj, ref, refHash),
// MPSSpatialHash.cu:184-218, .cuh:180-271): for each fluid slot, the particles of every other
// scene within (h_i + h_j)/2, scene after scene in ascending order, each scene's part in the
// 27-cell order of that scene's own table (the walk of the wall lists, on another table).
__global__ void __launch_bounds__(kBlock) k_neighbors_ref(const float4* __restrict__ pos, Scenes sc, uint32_t C, HashGeom g,
                                                        HashView fl, uint32_t* __restrict__ nfr, uint32_t Kfr,
                                                        uint32_t* __restrict__ cfr, uint2* __restrict__ bstat) {
    const uint32_t blk = blockIdx.x;
    const uint32_t i = blk * kBlock + threadIdx.x;
    const uint32_t N = sc.N;
    const uint32_t sid = sc.blk_scene[blk];
    uint32_t k = 0u;
    if (i < sc.P[sid].end) {
        const float4 xi = pos[i];
        for (uint32_t t = 0; t < sc.S; t++) {
            if (t == sid) continue;
            const uint32_t at = k < Kfr ? k : Kfr;  // entries past the capacity are counted, not written
            k += search_cells<false, kCols>(xi, i, g, fl.start + size_t(t) * C, fl.end + size_t(t) * C, nullptr, fl.spos,
                                           nfr + size_t(at) * N, Kfr - at, N);
        }
    }
    if (i < N) cfr[i] = k;
    const uint32_t cnt[1] = {k};
    block_counts<1>(cnt, bstat, gridDim.x, blk);
}

// Z-sort payload permutation (MPSSpatialHash.cu:101-140): out[s] = in[perm[s]].
__global__ void __launch_bounds__(kBlock) k_gather_f4(const uint32_t* __restrict__ perm, uint32_t n, const float4* __restrict__ in,
                                                    float4* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && perm[s] != kEmpty) out[s] = in[perm[s]];
}
__global__ void __launch_bounds__(kBlock) k_gather_u32(const uint32_t* __restrict__ perm, uint32_t n, const uint32_t* __restrict__ in,
                                                     uint32_t* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && perm[s] != kEmpty) out[s] = in[perm[s]];
}
__global__ void __launch_bounds__(kBlock) k_gather_f2(const uint32_t* __restrict__ perm, uint32_t n, const float2* __restrict__ in,
                                                    float2* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && perm[s] != kEmpty) out[s] = in[perm[s]];
}
__global__ void __launch_bounds__(kBlock) k_gather_f1(const uint32_t* __restrict__ perm, uint32_t n, const float* __restrict__ in,
                                                    float* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n && perm[s] != kEmpty) out[s] = in[perm[s]];
}

}  // namespace dev

// ===================================================================== host launchers
namespace launch {
using namespace dev;

static inline unsigned nb(size_t n, unsigned b = kBlock) { return unsigned((n + b - 1) / b); }

// Fewest passes of at most 11 bits: a 64^3 grid takes two passes of 9 bits, a 128^3 grid two of 11
// (with at most 8 bits, three each: 1 M particles 45 against 60 us, 257 k 34 against 49, 33 k 23
// against 28).
constexpr int kMaxDigit = 11;

size_t radix_temp_words(uint32_t n) {
    return (size_t((n + kSortTile - 1) / kSortTile) + 1) << kMaxDigit;
}

int radix_sort(uint32_t*& keys, uint32_t*& vals, uint32_t*& keys_alt, uint32_t*& vals_alt, uint32_t* temp, uint32_t n,
               int key_bits, hipStream_t s) {
    if (n == 0 || key_bits <= 0) return 0;
    if (n <= kSortOne) {
        launch_k(k_radix_one, 1, kOneThreads, 0, s, keys, vals, keys_alt, vals_alt, n, key_bits);
        std::swap(keys, keys_alt);
        std::swap(vals, vals_alt);
        return 0;
    }
    const uint32_t tiles = (n + kSortTile - 1) / kSortTile;
    const int passes = (key_bits + kMaxDigit - 1) / kMaxDigit;
    const int digit = std::max((key_bits + passes - 1) / passes, 4);  // 16 digits per scanning workgroup
    uint32_t* total = temp + (size_t(tiles) << digit);
    auto pass = [&](auto d, int shift) {
        constexpr int D = decltype(d)::value;
        launch_k(k_radix_hist<D>, tiles, kSortThreads, 0, s, keys, n, shift, temp);
        if (tiles <= kSortSelf) {
            launch_k(k_radix_scatter<D, true>, tiles, kSortThreads, 0, s, keys, vals, keys_alt, vals_alt, n, shift, temp, tiles,
                     total);
        } else {
            launch_k(k_radix_scan, (1u << D) / kScanDigits, kScanDigits * kScanRuns, 0, s, temp, 1u << D, tiles, total);
            launch_k(k_radix_scatter<D, false>, tiles, kSortThreads, 0, s, keys, vals, keys_alt, vals_alt, n, shift, temp, tiles,
                     total);
        }
    };
    for (int shift = 0; shift < key_bits; shift += digit) {
        switch (digit) {
            case 11: pass(std::integral_constant<int, 11>{}, shift); break;
            case 10: pass(std::integral_constant<int, 10>{}, shift); break;
            case 9: pass(std::integral_constant<int, 9>{}, shift); break;
            case 8: pass(std::integral_constant<int, 8>{}, shift); break;
            case 7: pass(std::integral_constant<int, 7>{}, shift); break;
            case 6: pass(std::integral_constant<int, 6>{}, shift); break;
            case 5: pass(std::integral_constant<int, 5>{}, shift); break;
            default: pass(std::integral_constant<int, 4>{}, shift); break;
        }
        std::swap(keys, keys_alt);
        std::swap(vals, vals_alt);
    }
    return 0;
}

void cell_keys(const float4* pos, uint32_t n, const HashGeom& g, int morton, const uint32_t* scene, int shift, uint32_t* key,
               uint32_t* id, hipStream_t s) {
    if (n) launch_k(k_cell_keys, nb(n), kBlock, 0, s, pos, n, g, morton, scene, shift, key, id);
}
void cell_keys_slots(const float4* pos, const uint32_t* perm, uint32_t n, const HashGeom& g, int morton,
                     const uint32_t* blk_scene, int shift, uint32_t* keyref, uint32_t* iota, hipStream_t s) {
    if (n) launch_k(k_cell_keys_slots, nb(n), kBlock, 0, s, pos, perm, n, g, morton, blk_scene, shift, keyref, iota);
}
void fluid_keys(const float4* pos, const uint32_t* perm, uint32_t n, const HashGeom& g, const uint32_t* blk_scene, int shift,
                uint32_t* keyref, uint32_t* iota, const uint32_t* mkey, const uint32_t* lkey, uint32_t n_old, uint32_t* start,
                uint32_t* end, hipStream_t s) {
    const uint32_t m = std::max(n, n_old);
    if (m) launch_k(k_fluid_keys, nb(m), kBlock, 0, s, pos, perm, n, g, blk_scene, shift, keyref, iota, mkey, lkey, n_old,
                    start, end);
}
void fluid_reorder(const uint32_t* key, const uint32_t* id, uint32_t nref, const HashGeom& g, int shift, uint32_t C,
                   const uint32_t* delta, uint32_t* inv, uint32_t* perm, uint32_t* src, uint32_t* mkey, uint32_t* lkey,
                   uint32_t* hash_perm, uint32_t* start, uint32_t* end, const FluidMove& mv, hipStream_t s) {
    if (nref) launch_k(k_fluid_reorder, nb(nref), kBlock, 0, s, key, id, nref, g, shift, C, delta, inv, perm, src, mkey, lkey,
                       hash_perm, start, end, mv);
}
void invert(const uint32_t* perm, uint32_t n, uint32_t* inv, hipStream_t s) {
    if (n) launch_k(k_invert, nb(n), kBlock, 0, s, perm, n, inv);
}
void relabel(uint32_t* perm, const uint32_t* map, uint32_t n, hipStream_t s) {
    if (n) launch_k(k_relabel, nb(n), kBlock, 0, s, perm, map, n);
}
void fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t s) {
    if (n) launch_k(k_fill_u32, unsigned((n + kBlock - 1) / kBlock), kBlock, 0, s, p, n, v);
}
void clear_cells(const uint32_t* key, uint32_t n, uint32_t* start, uint32_t* end, hipStream_t s) {
    if (n) launch_k(k_clear_cells, nb(n), kBlock, 0, s, key, n, start, end);
}
void cell_table(const uint32_t* key, const uint32_t* id, uint32_t n, uint32_t* start, uint32_t* end, const float4* pos,
                float4* spos, hipStream_t s) {
    if (n) launch_k(k_cell_table, nb(n), kBlock, 0, s, key, id, n, start, end, pos, spos);
}
void neighbors_fluid(const float4* pos, const Scenes& sc, uint32_t C, const HashGeom& g, const HashView& fl, const HashView& bd,
                     uint32_t* nff, uint32_t Kff, uint32_t* cff, uint32_t* nfb, uint32_t Kfb, uint32_t* cfb, uint2* bstat,
                     HaloOut ho, SearchPasses passes, SearchLeave leave, int dense, NbrCounters* ctr, hipStream_t s) {
    if (!sc.N) return;
    const uint32_t g_ = nb(sc.N);
    ho.limit = ho.limit == 0u || ho.limit > kHaloCap ? kHaloCap : ho.limit;
#define MPS_SEARCH(Q, CAPS, LAST, MODE)                                                                                       \
    launch_k(k_neighbors_fluid<Q, CAPS, LAST>, g_, Q * kBlock, 0, s, pos, sc, C, g, fl, bd, nff, Kff, cff, nfb, Kfb, cfb, bstat, \
             ho, MODE, ctr)
    // Up to two workgroups per CU one pass of the quad form (its blocks have the chip to themselves:
    // 128 workgroups 206 -> 72 us with the halos); beyond, the one-lane form and, where the last
    // search left blocks (or this one did: passes = kSearchLeft), the quad form over those.
    if (g_ <= kSearchOnePass) {
        MPS_SEARCH(4, SearchWide, true, 0);
    } else {
        if (passes != kSearchLeft) {
            if (dense) MPS_SEARCH(1, SearchDense, false, leave);
            else MPS_SEARCH(1, SearchStd, false, leave);
        }
        if (passes != kSearchFirst) MPS_SEARCH(4, SearchWide, true, 1);
    }
#undef MPS_SEARCH
    // (max_ff, max_fb) and (nnz_ff, nnz_fb) are neighbours in the record
    launch_k(k_count_fold, 3, kCountFoldThreads, 0, s, bstat, g_, &ctr->max_ff, &ctr->nnz_ff, ho.n, ho.stats);
}
void neighbors_ref(const float4* pos, const Scenes& sc, uint32_t C, const HashGeom& g, const HashView& fl, uint32_t* nfr,
                   uint32_t Kfr, uint32_t* cfr, uint2* bstat, NbrCounters* ctr, hipStream_t s) {
    if (!sc.N) return;
    const uint32_t g_ = nb(sc.N);
    launch_k(k_neighbors_ref, g_, kBlock, 0, s, pos, sc, C, g, fl, nfr, Kfr, cfr, bstat);
    launch_k(k_count_fold, 1, kCountFoldThreads, 0, s, bstat, g_, &ctr->max_fr, &ctr->nnz_fr, nullptr, nullptr);
}
void neighbors_boundary(const float4* pos, uint32_t B, const uint32_t* scene, uint32_t C, const HashGeom& g, const HashView& bd,
                        uint32_t* nbb, uint32_t Kbb, uint32_t* cbb, uint2* bstat, NbrCounters* ctr, hipStream_t s) {
    if (!B) return;
    const uint32_t g_ = nb(B);
    launch_k(k_neighbors_boundary, g_, kBlock, 0, s, pos, B, scene, C, g, bd, nbb, Kbb, cbb, bstat);
    launch_k(k_count_fold, 1, kCountFoldThreads, 0, s, bstat, g_, &ctr->max_bb, &ctr->nnz_bb, nullptr, nullptr);
}
void gather_f4(const uint32_t* perm, uint32_t n, const float4* in, float4* out, hipStream_t s) {
    if (n) launch_k(k_gather_f4, nb(n), kBlock, 0, s, perm, n, in, out);
}
void gather_u32(const uint32_t* perm, uint32_t n, const uint32_t* in, uint32_t* out, hipStream_t s) {
    if (n) launch_k(k_gather_u32, nb(n), kBlock, 0, s, perm, n, in, out);
}
void gather_f2(const uint32_t* perm, uint32_t n, const float2* in, float2* out, hipStream_t s) {
    if (n) launch_k(k_gather_f2, nb(n), kBlock, 0, s, perm, n, in, out);
}
void gather_f1(const uint32_t* perm, uint32_t n, const float* in, float* out, hipStream_t s) {
    if (n) launch_k(k_gather_f1, nb(n), kBlock, 0, s, perm, n, in, out);
}

}  // namespace launch
}  // namespace mps
