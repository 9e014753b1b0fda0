// sph.hip — DFSPH / implicit viscosity / advection kernels for gfx950.
//
// One thread (or, in small grids, four lanes) per particle walks its ELL neighbour lists (fluid
// then boundary), accumulating in registers in the reference's order, so a per-particle
// result equals (0 + fluid sum) + boundary sum exactly as the reference's two kernels and
// AtomicAdd produce it. Passes that the reference splits into several kernels over the
// same neighbour list are fused (density + alpha + gravity; delta + stiffness + error
// reduction; pressure force + velocity update; ST + XSPH + viscosity + final A.p).
//
// Quantities that stay fixed while a solver iterates are computed once per step or per
// solve and kept per neighbour slot: the kernel gradient factor G_ij (written by the alpha
// pass, read by every DF/CD iteration) and the two scalar coefficients of the implicit
// viscosity/surface-tension operator (written by the CG set-up pass), so an iteration
// streams 4-8 bytes per pair instead of re-evaluating square roots and divisions.
//
// Convergence sums: each workgroup reduces its T-rounded terms in double and writes one
// partial; the workgroups that need the sum, or in large grids a one-workgroup fold kernel, add the
// partials in index order (deterministic, no FP64 atomics) and update a SolverDev record on the device. Kernels of later iterations
// read SolverDev::done first (those that fold: SolverDev::it) and exit at once, so the host can
// enqueue several iterations before it looks at the result.
#include "device_common.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace mps {
namespace dev {

__device__ __forceinline__ uint32_t nbr_ff(const Nbr& nb, uint32_t k, uint32_t i, uint32_t N) {
    return nb.ff[ell(k, i, N)];
}
__device__ __forceinline__ uint32_t nbr_fb(const Nbr& nb, uint32_t k, uint32_t i, uint32_t N) {
    return nb.fb[size_t(k) * N + i];
}

// Walks the wall list of slot i in list order, kWallBatch entries at a time: the batch's
// indices are loaded together, then gather(j, entry) fetches each entry's wall record, and only
// then does use(true, entry, record) consume them in order. A batch costs about one dependent
// memory latency instead of two per entry. With a quad per slot (Q = 4) lane part l handles the
// batch's entry l, and use(false, ...) is called in the lanes past the list's end, whose term has
// to be +0.
constexpr uint32_t kWallBatch = 4;
template <int Q, class Gather, class Use>
__device__ __forceinline__ void walk_walls(const Nbr& nb, uint32_t i, uint32_t l, uint32_t N, uint32_t cb, Gather&& gather, Use&& use) {
    using Rec = decltype(gather(0u, size_t(0)));
    for (uint32_t k0 = 0; k0 < cb; k0 += kWallBatch) {
        if constexpr (Q == 4) {
            const bool in = k0 + l < cb;
            const uint32_t k = in ? k0 + l : k0;
            const size_t entry = size_t(k) * N + i;
            const Rec w = gather(nbr_fb(nb, k, i, N), entry);
            use(in, entry, w);
        } else {
            uint32_t j[kWallBatch];
#pragma unroll
            for (uint32_t q = 0; q < kWallBatch; q++) j[q] = k0 + q < cb ? nbr_fb(nb, k0 + q, i, N) : 0u;
            Rec w[kWallBatch];
#pragma unroll
            for (uint32_t q = 0; q < kWallBatch; q++)
                if (k0 + q < cb) w[q] = gather(j[q], size_t(k0 + q) * N + i);
#pragma unroll
            for (uint32_t q = 0; q < kWallBatch; q++)
                if (k0 + q < cb) use(true, size_t(k0 + q) * N + i, w[q]);
        }
    }
}

// Block-reduce `v` (double) in a fixed order and publish the workgroup's partial.
// COH: device-coherent store (agent scope), for the persistent solver's barrier without fences.
template <bool COH = false>
__device__ __forceinline__ void block_partial(double v, double* __restrict__ partials, uint32_t blk) {
    __shared__ double lds[kBlock / 64];
    const double bs = block_total<kBlock / 64>(v, lds);
    if (threadIdx.x == 0) {
        if constexpr (COH) __hip_atomic_store(partials + blk, bs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else partials[blk] = bs;
    }
}
// Loads and stores of the CG vectors that other workgroups read within one launch of the
// persistent solver: device-coherent (agent scope) when COH, so that no cache write-back or
// invalidation is needed at its barriers; plain otherwise.
template <bool COH>
__device__ __forceinline__ f3 ld3c(const f3* p) {
    if constexpr (COH) {
        const float* q = reinterpret_cast<const float*>(p);
        return {__hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                __hip_atomic_load(q + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)};
    } else {
        return *p;
    }
}
template <bool COH>
__device__ __forceinline__ void st3c(f3* p, f3 v) {
    if constexpr (COH) {
        float* q = reinterpret_cast<float*>(p);
        __hip_atomic_store(q, v.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(q + 1, v.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(q + 2, v.z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *p = v;
    }
}
__device__ __forceinline__ void block_partial(double v, double* __restrict__ partials) {
    block_partial(v, partials, blockIdx.x);
}
// Sum of partials[0..n) in index-strided order, valid in every thread of a workgroup of
// kFoldThreads (call it again only after a further barrier).
constexpr int kFoldThreads = 1024;
__device__ __forceinline__ double fold(const double* __restrict__ partials, uint32_t n) {
    __shared__ double lds[kFoldThreads / 64];
    double s = 0.0;
    constexpr uint32_t R = 8;  // loads in flight per thread; the adds keep the index order
    for (uint32_t k0 = threadIdx.x; k0 < n; k0 += R * blockDim.x) {
        double v[R];
#pragma unroll
        for (uint32_t q = 0; q < R; q++) {
            const uint32_t k = k0 + q * blockDim.x;
            v[q] = k < n ? partials[k] : 0.0;
        }
#pragma unroll
        for (uint32_t q = 0; q < R; q++)
            if (k0 + q * blockDim.x < n) s += v[q];
    }
    return block_total<kFoldThreads / 64>(s, lds);
}

// The fold of the kFoldThreads-thread fold kernels, computed by one kBlock-thread workgroup in
// exactly their order: thread t plays their threads t + kBlock v (v < kFoldThreads / kBlock);
// each sums its strided partials left to right, each of their waves is reduced by the same
// butterfly (the played threads of one of their waves all sit in one wave here, in the same
// lanes), and every thread adds the wave totals in wave order. Valid in every thread; call it
// again only after a further barrier.
template <bool COH>
__device__ __forceinline__ double fold_as_fold_kernel(const double* __restrict__ partials, uint32_t n) {
    constexpr uint32_t V = kFoldThreads / kBlock;
    constexpr uint32_t kWaves = kFoldThreads / 64;
    constexpr uint32_t R = 4;  // strides of kFoldThreads loaded per batch: R * V loads in flight
    __shared__ double wsum[kWaves];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    auto ld = [&](uint32_t k) -> double {
        if constexpr (COH) return __hip_atomic_load(partials + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else return partials[k];
    };
    double s[V];
#pragma unroll
    for (uint32_t v = 0; v < V; v++) s[v] = 0.0;
    for (uint32_t m0 = 0; m0 * kFoldThreads < n; m0 += R) {
        double t[R][V];
#pragma unroll
        for (uint32_t r = 0; r < R; r++)
#pragma unroll
            for (uint32_t v = 0; v < V; v++) {
                const uint32_t k = threadIdx.x + v * kBlock + (m0 + r) * kFoldThreads;
                t[r][v] = k < n ? ld(k) : 0.0;
            }
#pragma unroll
        for (uint32_t r = 0; r < R; r++)
#pragma unroll
            for (uint32_t v = 0; v < V; v++)
                if (threadIdx.x + v * kBlock + (m0 + r) * kFoldThreads < n) s[v] += t[r][v];
    }
#pragma unroll
    for (uint32_t v = 0; v < V; v++) {
        const double x = wave_sum_d(s[v]);
        if (lane == 0) wsum[wave + v * (kBlock / 64)] = x;
    }
    __syncthreads();
    double w[kWaves];
#pragma unroll
    for (uint32_t q = 0; q < kWaves; q++) w[q] = wsum[q];
    double t = 0.0;
#pragma unroll
    for (uint32_t q = 0; q < kWaves; q++) t += w[q];
    return t;
}

// The same sum in a workgroup of Q * kBlock threads, valid in every thread (Q = 4: the fold kernels'
// own thread count).
template <int Q>
__device__ __forceinline__ double fold_everywhere(const double* __restrict__ partials, uint32_t n) {
    if constexpr (Q == 1) {
        return fold_as_fold_kernel<false>(partials, n);
    } else {
        static_assert(Q * kBlock == kFoldThreads, "the quad forms have the fold kernels' size");
        return fold(partials, n);
    }
}

// ---- walks of the fluid lists
// The fluid lists, and everything stored per list entry, keep the four entries 4g .. 4g+3 of a
// slot side by side (ell(), device_common.hpp). With one lane per slot (Q = 1) a lane loads a group
// of four at once: 8 bytes of halo positions, 16 of G_ij, 16 each of a_ij and b_ij. Against one
// entry per load (columns, two entries in flight) a walk waits for a quarter of the round trips and
// issues a quarter of the loads and addresses: A.p 25 -> 15 us at 45k particles (66 neighbours each),
// 85 -> 70 us at 525k (61), 76 -> 73 us at 1M (31; there the stream itself is the bound, and the
// unused entries of the last groups cost 10 % more bytes: 482 -> 530 MB). With a quad per slot
// (Q = 4) lane part l of the quad takes entry 4g + l of every group, and the group's four terms
// are added to the running sum one after the other, in list order, by every lane of the quad
// (add_quad): a sum has the same bits in both forms. An entry past the end of the list
// contributes +0 there; the sums start at +0 (or a positive term), and x + 0 = x, x - 0 = x for
// every value that such a sum can take.
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// block_partial of a workgroup with a quad per slot (`v` counts in lane part 0): the slots'
// values are put back one per lane and reduced by the first wave in block_total's order, so the
// partial has the same bits.
template <int Q, bool COH = false>
__device__ __forceinline__ void slot_partial(double v, double* __restrict__ partials, uint32_t blk) {
    if constexpr (Q == 1) {
        block_partial<COH>(v, partials, blk);
    } else {
        static_assert(!COH, "the persistent solver runs one lane per slot");
        __shared__ double pv[kBlock];
        if (threadIdx.x % Q == 0) pv[threadIdx.x / Q] = v;
        __syncthreads();
        if (threadIdx.x < 64) {
            double w[kBlock / 64], s = 0.0;
#pragma unroll
            for (int q = 0; q < kBlock / 64; q++) w[q] = wave_sum_d(pv[64 * q + threadIdx.x]);
#pragma unroll
            for (int q = 0; q < kBlock / 64; q++) s += w[q];
            if (threadIdx.x == 0) partials[blk] = s;
        }
    }
}

// The neighbours named by one group (Q = 1) or by this lane's entry of it (Q = 4): positions in
// the block's halo (STAGED) or slots.
template <int Q, bool STAGED>
struct GroupIdx;
template <>
struct GroupIdx<1, true> {
    uint2 w;
    __device__ __forceinline__ void load(const Nbr&, const Halo& hl, size_t group, uint32_t) {
        w = reinterpret_cast<const uint2*>(hl.nb16)[group];
    }
    __device__ __forceinline__ uint32_t at(int e) const { return e < 2 ? (e ? w.x >> 16 : w.x & 0xFFFFu) : (e == 3 ? w.y >> 16 : w.y & 0xFFFFu); }
};
template <>
struct GroupIdx<1, false> {
    v4u w;
    __device__ __forceinline__ void load(const Nbr& nb, const Halo&, size_t group, uint32_t) {
        w = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(nb.ff) + group);
    }
    __device__ __forceinline__ uint32_t at(int e) const { return w[e]; }
};
template <bool STAGED>
struct GroupIdx<4, STAGED> {
    uint32_t w;
    __device__ __forceinline__ void load(const Nbr& nb, const Halo& hl, size_t group, uint32_t l) {
        if constexpr (STAGED) w = hl.nb16[4 * group + l];
        else w = __builtin_nontemporal_load(nb.ff + 4 * group + l);
    }
    __device__ __forceinline__ uint32_t at(int) const { return w; }
};
// The arrays of values per list entry that a walk streams, with non-temporal loads where they are over the
// caches (GroupVal). (The
// coefficients a_ij and b_ij are two arrays and not pairs, so that each of a lane's 16-byte loads
// belongs to a contiguous kilobyte of the wave: with pairs, two loads touch every line, and the
// line is fetched twice.)
struct Streams {
    const float *a = nullptr, *b = nullptr, *aT = nullptr, *bT = nullptr;
};
// KEEP: without the hint, for arrays that a solve streams again and again and that stay in a cache from
// one launch to the next. The grids with a quad per slot always do (their 2 MB per XCD in its L2: A.p at
// 45k particles, 66 neighbours each, 14.8 -> 12.1 us); with one lane per slot A.p does while its stream
// fits the 256 MB memory-side cache (Halo::keep; at spacing 0.6 of rest: 257k 22.7 -> 21.2 us, 405k 35.1 ->
// 30.8, 512k 39.3 -> 36.7, 636k and 197 MB 50.0 -> 48.2, 804k and 250 MB 63.4 -> 68.0, 1M 71 -> 82).
template <int Q, bool KEEP = false>
struct GroupVal {
    typename std::conditional<Q == 1, v4f, float>::type v;
    __device__ __forceinline__ void load(const float* p, size_t group, uint32_t l) {
        if constexpr (Q != 1) v = p[4 * group + l];
        else if constexpr (KEEP) v = reinterpret_cast<const v4f*>(p)[group];
        else v = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(p) + group);
    }
    __device__ __forceinline__ void load(const Streams& s, size_t group, uint32_t l) { load(s.a, group, l); }
    __device__ __forceinline__ float at(int e) const {
        if constexpr (Q == 1) return v[e];
        else return v;
    }
};
template <int Q, bool KEEP>
struct GroupAB {
    GroupVal<Q, KEEP> a, b;
    __device__ __forceinline__ void load(const Streams& s, size_t group, uint32_t l) {
        a.load(s.a, group, l);
        b.load(s.b, group, l);
    }
};
template <int Q, bool KEEP>
struct GroupABT {
    GroupVal<Q, KEEP> a, b, aT, bT;
    __device__ __forceinline__ void load(const Streams& s, size_t group, uint32_t l) {
        a.load(s.a, group, l);
        b.load(s.b, group, l);
        aT.load(s.aT, group, l);
        bT.load(s.bT, group, l);
    }
};
struct NoVal {
    __device__ __forceinline__ void load(const Streams&, size_t, uint32_t) {}
};

// Groups requested before the halo staging, and halo records that a thread stages per pass. A.p
// at 1M particles (31 neighbours each), one run: 1 group and 2 records 73.3 us, 2 and 2 74.7,
// 1 and 4 75.8, 2 and 4 77.0 (with 4 records the evaluation and the density are 1-3 us faster).
constexpr int kPreApply = 1, kPreEval = 1, kPrePressure = 1;  // one lane per slot
constexpr int kPreQuad = 8;                                   // a quad per slot
template <int Q>
constexpr uint32_t kHaloLoads = Q == 1 ? 4 : 2;
constexpr uint32_t kHaloLoadsApply = 2;

// A walk over the c entries of one slot: whole groups in order, one being loaded ahead of the one
// in use, then the rest (c % 4). begin() requests the first PRE groups and the rest, so that these
// loads run beside the halo staging between begin() and run(). full(group number, indices, values)
// and rest(group number, indices, values, c % 4) consume them.
template <int Q, bool STAGED, class Val, int PRE>
struct Walk {
    using Idx = GroupIdx<Q, STAGED>;
    Idx ip[PRE], ir;
    Val vp[PRE], vr;
    const Nbr& nb;
    const Halo& hl;
    const Streams val;  // the arrays that Val reads
    uint32_t i, l, N, gf, nr;
    __device__ __forceinline__ Walk(const Nbr& nb, const Halo& hl, const Streams& val, uint32_t i, uint32_t l, uint32_t N, uint32_t c)
        : nb(nb), hl(hl), val(val), i(i), l(l), N(N), gf(c >> 2), nr(c & 3u) {
#pragma unroll
        for (uint32_t g = 0; g < PRE; g++)
            if (g < gf) get(g, ip[g], vp[g]);
        if (nr) get(gf, ir, vr);
    }
    __device__ __forceinline__ void get(uint32_t g, Idx& x, Val& v) const {
        const size_t group = size_t(g) * N + i;
        x.load(nb, hl, group, l);
        v.load(val, group, l);
    }
    template <class Full, class Rest>
    __device__ __forceinline__ void run(Full&& full, Rest&& rest) {
        Idx xn;
        Val vn;
        if (PRE < gf) get(PRE, xn, vn);
#pragma unroll
        for (uint32_t g = 0; g < PRE; g++)
            if (g < gf) full(g, ip[g], vp[g]);
        for (uint32_t g = PRE; g < gf; g++) {
            const Idx x = xn;
            const Val v = vn;
            if (g + 1 < gf) get(g + 1, xn, vn);
            full(g, x, v);
        }
        if (nr) rest(gf, ir, vr, nr);
    }
};

// What every halo-staged kernel requests first: these loads depend on the workgroup's number
// alone, so the kernel waits for two memory latencies (these, then what they lead to) and not for
// one per lookup. The first halo slots are read before the halo's size is known (a row always has
// kHaloCap words); padding slots have a list length of 0.
template <int Q, uint32_t R>
struct BlockHead {
    static constexpr uint32_t kThreads = Q * kBlock;
    uint32_t i, l, c, H;
    const uint32_t* hs;
    uint32_t sh[R];
    __device__ __forceinline__ BlockHead(uint32_t blk, uint32_t N, const uint32_t* cff, const Halo& hl) {
        i = blk * kBlock + threadIdx.x / Q;
        l = threadIdx.x % Q;
        c = i < N ? cff[i] : 0u;
        H = hl.n[blk];
        hs = hl.idx + size_t(blk) * kHaloCap;
#pragma unroll
        for (uint32_t q = 0; q < R; q++) {
            const uint32_t t = threadIdx.x + q * kThreads;
            sh[q] = t < kHaloCap ? hs[t] : 0u;
        }
    }
    // store(t, load(s)) for every halo record t < H (s = its slot): R records per thread and
    // pass, all their loads before the first LDS store (past the halo's end a thread loads slot 0
    // and stores nothing).
    template <class Load, class Store>
    __device__ __forceinline__ void stage(Load&& load, Store&& store) const {
        using Rec = decltype(load(0u));
        for (uint32_t t0 = threadIdx.x; t0 < H; t0 += R * kThreads) {
            Rec rec[R];
#pragma unroll
            for (uint32_t q = 0; q < R; q++) {
                const uint32_t t = t0 + q * kThreads;
                rec[q] = load(t < H ? (t0 == threadIdx.x ? sh[q] : hs[t]) : 0u);
            }
#pragma unroll
            for (uint32_t q = 0; q < R; q++) {
                const uint32_t t = t0 + q * kThreads;
                if (t < H) store(t, rec[q]);
            }
        }
    }
};

// LDS staging depth (records per workgroup, <= kHaloCap) of each halo-staged kernel: with wide
// records the depth decides how many workgroups share a CU's 160 KiB. A block with a deeper halo
// gathers from global memory instead, with the same results. A.p and the DF/CD evaluation
// (24-byte records) stage kHaloShallow = 1264 records (30.3 KB, five workgroups per CU) or, when
// the host sees enough deeper halos (Halo::deep), kHaloCap = 1536 (36.9 KB, four): near rest
// density a block's halo holds ~1400 slots, and gathering them costs the evaluation 198 us
// instead of 54 (525k particles at 0.95 of the rest density). The CG setup (36-byte records)
// stages 1104 (39.7 KB, four per CU) or, with deep halos, runs its quad form at kHaloCap (54 KB:
// 260 -> 160 us there). The quad forms of all three stage kHaloCap.
constexpr uint32_t kStageEval = kHaloShallow;
constexpr uint32_t kStageSetup = 1104;
constexpr uint32_t kStageAp = kHaloShallow;
constexpr uint32_t kStageDensity = kHaloShallow, kStageST = kHaloShallow, kStagePApply = kHaloShallow;
static_assert(kStageEval <= kHaloCap && kStageSetup <= kHaloCap && kStageAp <= kHaloCap && kStageDensity <= kHaloCap &&
                  kStageST <= kHaloCap && kStagePApply <= kHaloCap,
              "staging depths");

// ----------------------------------------------------------------- boundary volume
// ComputeBoundaryParticleVolume_kernel (MPSSPHBaseUtil.cuh:10-41): S_b = W(0) + sum W_bk.
// S_b depends only on boundary positions, so it is computed when they change.
template <bool CUBIC>
__global__ void __launch_bounds__(kBlock) k_boundary_sum(const float4* __restrict__ bpos, uint32_t B, const uint32_t* __restrict__ nbb,
                                                       uint32_t Kbb, const uint32_t* __restrict__ cbb, float* __restrict__ S) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B) return;
    const float4 xi4 = bpos[i];
    const f3 xi = mk(xi4);
    const float hi = xi4.w * 4.0f;
    const float invHi = 1.0f / hi;
    float vol = Wk<CUBIC>(0.0f, invHi);
    const uint32_t c = cbb[i];
    for (uint32_t k = 0; k < c; k++) {
        const uint32_t j = nbb[size_t(i) * Kbb + k];
        vol += Wk<CUBIC>(len3(xi - mk(bpos[j])), invHi);
    }
    S[i] = vol;
}
// ComputeBoundaryParticleVolumeFinal_kernel (:78-86) on top of the AtomicAdd into the
// never-cleared volume (Q1): V <- 1/(V + S).
__global__ void __launch_bounds__(kBlock) k_boundary_volume(const float* __restrict__ S, float* __restrict__ vol, uint32_t B, int faithful) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B) return;
    float v = faithful ? vol[i] : 0.0f;
    v += S[i];
    vol[i] = 1.0f / v;
}

// Several wall objects (a wall particle's object in obj[]): sums kept per object, walls of the
// own object first (ComputeBoundaryParticleVolume_kernel self + ref, MPSSPHBaseUtil.cuh:10-76).
// Per-object accumulators stay in registers: updates and reads select the element with
// unrolled compares instead of a dynamic index.
template <class T, class F>
__device__ __forceinline__ void at_obj(T (&a)[kMaxWallObjects], uint32_t o, F&& f) {
#pragma unroll
    for (uint32_t q = 0; q < kMaxWallObjects; q++)
        if (q == o) f(a[q]);
}
template <bool CUBIC>
__global__ void __launch_bounds__(kBlock) k_boundary_sum_obj(const float4* __restrict__ bpos, uint32_t B,
                                                           const uint32_t* __restrict__ nbb, uint32_t Kbb,
                                                           const uint32_t* __restrict__ cbb, const uint32_t* __restrict__ obj,
                                                           float4* __restrict__ S4) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B) return;
    const float4 xi4 = bpos[i];
    const f3 xi = mk(xi4);
    const float invHi = 1.0f / (xi4.w * 4.0f);
    float v[kMaxWallObjects] = {0.f, 0.f, 0.f, 0.f};
    at_obj(v, obj[i], [&](float& a) { a = Wk<CUBIC>(0.0f, invHi); });
    const uint32_t c = cbb[i];
    for (uint32_t k = 0; k < c; k++) {
        const uint32_t j = nbb[size_t(i) * Kbb + k];
        const float w = Wk<CUBIC>(len3(xi - mk(bpos[j])), invHi);
        at_obj(v, obj[j], [&](float& a) { a += w; });
    }
    S4[i] = make_float4(v[0], v[1], v[2], v[3]);
}
__global__ void __launch_bounds__(kBlock) k_boundary_volume_obj(const float4* __restrict__ S4, const uint32_t* __restrict__ obj,
                                                              uint32_t nobj, float* __restrict__ vol, uint32_t B, int faithful) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B) return;
    const float4 s4 = S4[i];
    const float s[kMaxWallObjects] = {s4.x, s4.y, s4.z, s4.w};
    const uint32_t own = obj[i];
    float v = faithful ? vol[i] : 0.0f;
    at_obj(s, own, [&](const float& a) { v += a; });
#pragma unroll
    for (uint32_t q = 0; q < kMaxWallObjects; q++)
        if (q < nobj && q != own) v += s[q];
    vol[i] = 1.0f / v;
}

// ----------------------------------------------------------------- density, alpha, gravity
// ComputeDensity_kernel ff/fb + Final + DensityColorTest (MPSSPHBaseUtil.cuh:88-221),
// ComputeDFSPHFactor_kernel ff/fb + Final (MPSSPHDFSPHUtil.cuh:10-137),
// ApplyGravity + UpdateVelocity (MPSAdvectUtil.cuh:8-34).
// Also stores G_ij per neighbour slot (pG_ff, pG_fb) when kDoPairs is set.
template <bool CUBIC, bool REF, bool BOBJ, int Q>
__global__ void __launch_bounds__(Q * kBlock) k_density_alpha(int flags, Scenes sc, Nbr nb, Halo hl, const float4* __restrict__ pos,
                                                        float4* __restrict__ vel, const float4* __restrict__ bpos,
                                                        const float* __restrict__ bvol, float* __restrict__ rho,
                                                        float* __restrict__ alpha, float4* __restrict__ color,
                                                        float* __restrict__ pG_ff, float* __restrict__ pG_fb) {
    static_assert(Q == 1 || !(REF || BOBJ), "coupled scenes and wall objects run one lane per slot");
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t N = sc.N;
    const bool dens = flags & launch::kDoDensity, alph = flags & launch::kDoAlpha;
    const bool pairs = flags & launch::kDoPairs;
    const bool walk = dens || alph || pairs;
    // the block's halo positions in LDS (see k_cg_apply)
    __shared__ float4 la[kStageDensity];
    BlockHead<Q, kHaloLoads<Q>> hd(blk, N, nb.cff, hl);
    const uint32_t i = hd.i, l = hd.l, c = walk ? hd.c : 0u;
    const uint32_t cb = walk && i < N ? nb.cfb[i] : 0u;
    const float4 xi4 = i < N ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t sid = sc.blk_scene[blk];
    const StepParams P = sc.P[sid];
    const bool live = i < P.end;
    const f3 xi = mk(xi4);
    const float hi = xi4.w * 4.0f;
    const float invHi = 1.0f / hi;
    float sf = dens ? P.V * Wk<CUBIC>(0.0f, invHi) : 0.0f;
    f3 gf{0.f, 0.f, 0.f};
    float s = 0.0f;
    // terms of one pair; W, G, grad and its square
    struct Term {
        float w, G, s2;
        f3 g;
    };
    auto term = [&](f3 xj) -> Term {
        Term t{0.f, 0.f, 0.f, {0.f, 0.f, 0.f}};
        const f3 xij = xi - xj;
        const float dist = len3(xij);
        if (dens) t.w = P.V * Wk<CUBIC>(dist, invHi);
        if (alph || pairs) {
            t.G = Gk<CUBIC>(dist, invHi);
            t.g = (P.V * t.G) * xij;
            t.s2 = dot3(t.g, t.g);
        }
        return t;
    };
    auto walk_fluid = [&](auto staged) {
        constexpr bool STAGED = decltype(staged)::value;
        Walk<Q, STAGED, NoVal, 1> wk(nb, hl, Streams{}, i, l, N, live ? c : 0u);
        if constexpr (STAGED) {
            hd.stage([&](uint32_t j) { return pos[j]; }, [&](uint32_t t, const float4& x) { la[t] = x; });
            __syncthreads();
        }
        auto at = [&](uint32_t j) { return mk(STAGED ? la[j] : pos[j]); };
        wk.run(
            [&](uint32_t g, const auto& x, const NoVal&) {
                const size_t group = size_t(g) * N + i;
                if constexpr (Q == 1) {
                    f3 xj[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) xj[e] = at(x.at(e));
                    v4f G;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const Term t = term(xj[e]);
                        sf += t.w;
                        gf = gf + t.g;
                        s += t.s2;
                        G[e] = t.G;
                    }
                    if (pairs) reinterpret_cast<v4f*>(pG_ff)[group] = G;
                } else {
                    const Term t = term(at(x.at(0)));
                    sf = add_quad(sf, t.w);
                    gf = add_quad(gf, t.g);
                    s = add_quad(s, t.s2);
                    if (pairs) pG_ff[4 * group + l] = t.G;
                }
            },
            [&](uint32_t g, const auto& x, const NoVal&, uint32_t n) {
                const size_t group = size_t(g) * N + i;
                if constexpr (Q == 1) {
#pragma unroll
                    for (int e = 0; e < 3; e++) {
                        if (e < int(n)) {
                            const Term t = term(at(x.at(e)));
                            sf += t.w;
                            gf = gf + t.g;
                            s += t.s2;
                            if (pairs) pG_ff[4 * group + e] = t.G;
                        }
                    }
                } else {
                    Term t{0.f, 0.f, 0.f, {0.f, 0.f, 0.f}};
                    if (l < n) {
                        t = term(at(x.at(0)));
                        if (pairs) pG_ff[4 * group + l] = t.G;
                    }
                    sf = add_quad(sf, t.w);
                    gf = add_quad(gf, t.g);
                    s = add_quad(s, t.s2);
                }
            });
    };
    if (walk) {
        if (hd.H <= kStageDensity) walk_fluid(std::true_type{});
        else walk_fluid(std::false_type{});
    }
    if (!live) return;
    if (walk) {
        float sb = 0.0f;
        f3 gb{0.f, 0.f, 0.f};
        float sbo[kMaxWallObjects] = {0.f, 0.f, 0.f, 0.f};  // per wall object (BOBJ)
        f3 gbo[kMaxWallObjects] = {};
        struct WallRec {
            float4 x;
            float vb;
            uint32_t o;
        };
        walk_walls<Q>(nb, i, l, N, cb,
                   [&](uint32_t j, size_t) { return WallRec{bpos[j], bvol[j], BOBJ ? nb.fbo[j] : 0u}; },
                   [&](bool in, size_t slot, const WallRec& w) {
            const f3 xij = xi - mk(w.x);
            const float dist = len3(xij);
            const float vb = w.vb;
            float wk = 0.0f, G = 0.0f;
            f3 gg{0.f, 0.f, 0.f};
            if (in) {
                if (dens) wk = vb * Wk<CUBIC>(dist, invHi);
                if (alph || pairs) {
                    G = Gk<CUBIC>(dist, invHi);
                    gg = (vb * G) * xij;
                    if (pairs) pG_fb[slot] = G;
                }
            }
            if constexpr (BOBJ) {
                at_obj(sbo, w.o, [&](float& a) { a += wk; });
                at_obj(gbo, w.o, [&](f3& a) { a = a + gg; });
            } else {
                sb = add_lanes<Q>(sb, wk);
                gb = add_lanes<Q>(gb, gg);
            }
        });
        // ((own + each ref object's sum, in scene order) + walls), as the reference's Sub
        // kernels accumulate them one after the other
        float d = 0.0f;
        d += sf;
        f3 g{0.f, 0.f, 0.f};
        g = g + gf;
        float a = 0.0f;
        a += s;
        if constexpr (REF) {  // ComputeDensity / ComputeDFSPHFactor ref (MPSSPHBaseUtil.cuh:122-156, MPSSPHDFSPHUtil.cuh:49-88)
            if (dens || alph) {
                const uint32_t cr = nb.cfr[i];
                uint32_t cur = kEmpty;
                float Vt = 0.0f, sr = 0.0f, ssr = 0.0f;
                f3 gr{0.f, 0.f, 0.f};
                for (uint32_t k = 0; k < cr; k++) {
                    const uint32_t j = nb.fr[size_t(k) * N + i];
                    const uint32_t t = sc.blk_scene[j / kBlock];
                    if (t != cur) {
                        if (cur != kEmpty) {
                            d += sr;
                            g = g + gr;
                            a += ssr;
                        }
                        cur = t;
                        Vt = sc.P[t].V;
                        sr = 0.0f;
                        ssr = 0.0f;
                        gr = f3{0.f, 0.f, 0.f};
                    }
                    const f3 xij = xi - mk(pos[j]);
                    const float dist = len3(xij);
                    if (dens) sr += Vt * Wk<CUBIC>(dist, invHi);
                    if (alph) {
                        const f3 grad = (Vt * Gk<CUBIC>(dist, invHi)) * xij;
                        gr = gr + grad;
                        ssr += dot3(grad, grad);
                    }
                }
                if (cur != kEmpty) {
                    d += sr;
                    g = g + gr;
                    a += ssr;
                }
            }
        }
        if (dens) {
            if constexpr (BOBJ) {
#pragma unroll
                for (uint32_t q = 0; q < kMaxWallObjects; q++)
                    if (q < nb.nbo) d += sbo[q];
            } else {
                d += sb;
            }
            const float r = d * P.rho0;
            if (l == 0) rho[i] = r;
            const float ratio = r / P.rho0;
            const float blue = fminf(fmaxf(1.0f - ratio, 0.0f), 1.0f);
            const float green = fminf(fmaxf(ratio < 1.0f ? ratio : 1.0f - (ratio - 1.0f), 0.0f), 1.0f);
            const float red = fminf(fmaxf(ratio - 1.0f, 0.0f), 1.0f);
            if (l == 0) color[i] = make_float4(red, green, blue, 1.0f);
        }
        if (alph) {
            if constexpr (BOBJ) {
#pragma unroll
                for (uint32_t q = 0; q < kMaxWallObjects; q++)
                    if (q < nb.nbo) g = g + gbo[q];
            } else {
                g = g + gb;
            }
            a += dot3(g, g);
            if (l == 0) alpha[i] = a > kEps ? 1.0f / a : 0.0f;
        }
    }
    if (l == 0 && (flags & launch::kDoGravity)) {
        float4 v4 = vel[i];
        const float m = v4.w;
        const f3 F = f3{0.f, 0.f, 0.f} + f3{P.gx, P.gy, P.gz} * m;
        if (m > 1.0e-10f) {
            const float c = P.dt / m;
            v4.x = v4.x + c * F.x;
            v4.y = v4.y + c * F.y;
            v4.z = v4.z + c * F.z;
            vel[i] = v4;
        }
    }
}

// ----------------------------------------------------------------- pressure solves
// The start of a loop: its record, by all threads of a workgroup. skip: the loop before it has not ended.
__device__ __forceinline__ void reset_record(SolverDev* st, bool skip) {
    if (threadIdx.x == 0) {
        st->done = skip ? kSkipped : 0u;
        st->l = 1u;
        st->counter = 0u;
        st->it = 0u;
        st->rr = 0.0;
        st->pAp = 0.0;
        st->thr = 0.0;
        st->alpha = 0.0f;
        st->beta = 0.0f;
    }
    for (uint32_t k = threadIdx.x; k < MPS_MAX_ITER_LOG; k += blockDim.x) st->log[k] = 0.0;
}
// The same by a launch over the fluid's workgroups that runs before the loop: each scene's first
// workgroup resets the scene's record (a launch of its own took 2.5 us and a gap, four a step).
__device__ __forceinline__ void reset_records(const launch::LoopStart& ls, const Scenes& sc, uint32_t blk, uint32_t sid) {
    if (!ls.rec || blk != sc.P[sid].blk0) return;
    reset_record(ls.rec + sid, shut(ls.gate));
    if (blk == 0u && threadIdx.x == 0) *ls.active = sc.S;
}

// ComputeDensityDelta_kernel ff/fb (MPSSPHDFSPHUtil.cuh:139-257) fused with
// ComputeDFStiffness_kernel / ComputeCDStiffness_kernel (:259-340); G_ij comes from the
// alpha pass. Each workgroup publishes its sum of positive errors for k_fold_pressure.
// The records of the block's halo (x_j, v_j) are staged in LDS (see k_cg_apply); the pairs
// are summed in list order on both paths.
template <bool DF, bool REF, bool CUBIC, bool BOBJ, int Q, bool DEEP>
__global__ void __launch_bounds__(Q * kBlock) k_pressure_eval(Scenes sc, Nbr nb, Halo hl, const float4* __restrict__ pos,
                                                        const float4* __restrict__ vel, const float4* __restrict__ bpos,
                                                        const float* __restrict__ bvol, const float4* __restrict__ bvel,
                                                        const float* __restrict__ rho, const float* __restrict__ alpha,
                                                        const float* __restrict__ pG_ff, const float* __restrict__ pG_fb,
                                                        float* __restrict__ kappa, float* __restrict__ delta,
                                                        SolverDev* st, double* __restrict__ partials) {
    static_assert(Q == 1 || !(REF || BOBJ), "coupled scenes and wall objects run one lane per slot");
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t N = sc.N;
    constexpr uint32_t kDepth = DEEP ? kHaloCap : kStageEval;
    __shared__ float4 la[kDepth];
    __shared__ float2 lb[kDepth];
    BlockHead<Q, kHaloLoads<Q>> hd(blk, N, nb.cff, hl);
    const uint32_t i = hd.i, l = hd.l;
    const bool in = i < N;
    const uint32_t cb = in ? nb.cfb[i] : 0u;
    const float4 xi4 = in ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const f3 vi = in ? mk(vel[i]) : f3{0.f, 0.f, 0.f};
    const float rhoi = in ? rho[i] : 0.0f, alphai = in ? alpha[i] : 0.0f;
    const uint32_t sid = sc.blk_scene[blk];
    const bool done = st[sid].done != 0u;  // this scene's loop has finished
    const StepParams P = sc.P[sid];
    if (blk == P.blk0 && threadIdx.x == 0) st[sid].it = done ? 0u : st[sid].l;  // for an apply that folds
    if (done) return;
    const bool live = i < P.end;
    const f3 xi = mk(xi4);
    float df = 0.0f;
    using Val = GroupVal<Q>;
    auto walk_fluid = [&](auto staged) {
        constexpr bool STAGED = decltype(staged)::value;
        Walk<Q, STAGED, Val, Q == 1 ? kPreEval : kPreQuad> wk(nb, hl, Streams{pG_ff}, i, l, N, hd.c);
        struct Rec {
            f3 x, v;
        };
        if constexpr (STAGED) {
            hd.stage([&](uint32_t j) { return Rec{mk(pos[j]), mk(vel[j])}; },
                     [&](uint32_t t, const Rec& r) {
                         la[t] = make_float4(r.x.x, r.x.y, r.x.z, r.v.x);
                         lb[t] = make_float2(r.v.y, r.v.z);
                     });
            __syncthreads();
        }
        auto at = [&](uint32_t j) -> Rec {
            if constexpr (STAGED) {
                const float4 a = la[j];
                const float2 b = lb[j];
                return {mk(a), {a.w, b.x, b.y}};
            } else {
                return {mk(pos[j]), mk(vel[j])};
            }
        };
        auto term = [&](float G, const Rec& r) { return P.V * G * dot3(xi - r.x, vi - r.v); };
        wk.run(
            [&](uint32_t, const auto& x, const Val& G) {
                if constexpr (Q == 1) {
                    Rec r[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) r[e] = at(x.at(e));
#pragma unroll
                    for (int e = 0; e < 4; e++) df += term(G.at(e), r[e]);
                } else {
                    df = add_quad(df, term(G.at(0), at(x.at(0))));
                }
            },
            [&](uint32_t, const auto& x, const Val& G, uint32_t n) {
                if constexpr (Q == 1) {
#pragma unroll
                    for (int e = 0; e < 3; e++)
                        if (e < int(n)) df += term(G.at(e), at(x.at(e)));
                } else {
                    df = add_quad(df, l < n ? term(G.at(0), at(x.at(0))) : 0.0f);
                }
            });
    };
    if (hd.H <= kDepth) walk_fluid(std::true_type{});
    else walk_fluid(std::false_type{});
    double epos = 0.0;
    if (live) {
        float db = 0.0f;
        float dbo[kMaxWallObjects] = {0.f, 0.f, 0.f, 0.f};
        struct WallRec {
            float4 x, v;
            float vb, G;
            uint32_t o;
        };
        walk_walls<Q>(nb, i, l, N, cb,
                   [&](uint32_t j, size_t slot) {
                       return WallRec{bpos[j], bvel[j], bvol[j], pG_fb[slot], BOBJ ? nb.fbo[j] : 0u};
                   },
                   [&](bool in, size_t, const WallRec& w) {
            const f3 xij = xi - mk(w.x);
            const f3 vij = vi - mk(w.v);
            const float t = in ? w.vb * w.G * dot3(xij, vij) : 0.0f;
            if constexpr (BOBJ) at_obj(dbo, w.o, [&](float& a) { a += t; });
            else db = add_lanes<Q>(db, t);
        });
        float d = 0.0f;
        d += df;
        if constexpr (REF) {  // ComputeDensityDelta ref (MPSSPHDFSPHUtil.cuh:177-216): one sum per ref object
            const float invHi = 1.0f / (xi4.w * 4.0f);
            const uint32_t cr = nb.cfr[i];
            uint32_t cur = kEmpty;
            float Vt = 0.0f, dr = 0.0f;
            for (uint32_t k = 0; k < cr; k++) {
                const uint32_t j = nb.fr[size_t(k) * N + i];
                const uint32_t t = sc.blk_scene[j / kBlock];
                if (t != cur) {
                    if (cur != kEmpty) d += dr;
                    cur = t;
                    Vt = sc.P[t].V;
                    dr = 0.0f;
                }
                const f3 xij = xi - mk(pos[j]);
                const f3 vij = vi - mk(vel[j]);
                dr += Vt * Gk<CUBIC>(len3(xij), invHi) * dot3(xij, vij);
            }
            if (cur != kEmpty) d += dr;
        }
        if constexpr (BOBJ) {
#pragma unroll
            for (uint32_t q = 0; q < kMaxWallObjects; q++)
                if (q < nb.nbo) d += dbo[q];
        } else {
            d += db;
        }
        float e;
        if (DF) {
            const float a = d * P.dt;
            const float b = rhoi / P.rho0 + P.dt * d - 0.8f;
            e = a < b ? a : b;
        } else {
            e = rhoi / P.rho0 + P.dt * d - 1.0f;
        }
        if (e > 0.0f) {
            epos = double(e);
            e *= alphai / (P.dt * P.dt);
        } else {
            e = 0.0f;
        }
        if (l == 0) {
            delta[i] = d;
            kappa[i] = e;
        }
    }
    slot_partial<Q>(epos, partials, blk);
}

// Mean positive error and the loop decision of the DF/CD drivers
// (MPSSPHDFSPHUtil.cu:331-333,417-419): break when E < tol and l > lmin. `s` is the scene's sum of
// errors in iteration `it`; a scene that finishes leaves the count of active scenes.
__device__ __forceinline__ void record_pressure(SolverDev* sd, double E, bool ok, uint32_t it, uint32_t* active) {
    if (it - 1 < MPS_MAX_ITER_LOG) sd->log[it - 1] = E;
    if (ok) {
        sd->done = 1u;
        sd->l = it;
        atomicSub(active, 1u);
    } else {
        sd->l = it + 1;
    }
}
// Workgroup s folds scene s's partials. The iteration number is the record's l (1 after the reset,
// it + 1 after iteration it), so the launches of a chunk do not depend on where the chunk starts.
__global__ void __launch_bounds__(kFoldThreads) k_fold_pressure(Scenes sc, const double* __restrict__ partials,
                                                        SolverDev* st, uint32_t* active, double tol, uint32_t lmin) {
    const uint32_t sid = blockIdx.x;
    SolverDev* sd = st + sid;
    if (sd->done) return;
    const uint32_t it = sd->l;
    const StepParams P = sc.P[sid];
    const double s = fold(partials + P.blk0, P.nblk);
    if (threadIdx.x == 0) {
        const double E = s / double(P.count);
        record_pressure(sd, E, E < tol && it > lmin, it, active);
    }
}

// Coupled fluid objects run one pressure loop: a single workgroup folds every scene's errors
// and the loop ends at the first iteration where every scene has E < tol and l > lmin (all
// scenes then finish together, with the same l).
__global__ void __launch_bounds__(kFoldThreads) k_fold_pressure_joint(Scenes sc, const double* __restrict__ partials,
                                                              SolverDev* st, uint32_t* active, double tol, uint32_t lmin) {
    if (st[0].done) return;
    const uint32_t it = st[0].l;
    __shared__ uint32_t all_ok;
    if (threadIdx.x == 0) all_ok = 1u;
    __syncthreads();
    for (uint32_t sid = 0; sid < sc.S; sid++) {
        const StepParams P = sc.P[sid];
        const double s = fold(partials + P.blk0, P.nblk);
        if (threadIdx.x == 0) {
            const double E = P.count ? s / double(P.count) : 0.0;
            if (it - 1 < MPS_MAX_ITER_LOG) st[sid].log[it - 1] = E;
            if (!(E < tol && it > lmin)) all_ok = 0u;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const bool ok = all_ok != 0u;
        for (uint32_t sid = 0; sid < sc.S; sid++) {
            if (ok) st[sid].done = 1u;
            st[sid].l = ok ? it : it + 1;
        }
        if (ok) *active = 0u;
    }
}

// ApplyDFSPH_kernel ff/fb + ApplyDFSPHFinal_kernel (MPSSPHDFSPHUtil.cuh:342-468) + UpdateVelocity.
// The halo's (x_j, kappa_j) are staged in LDS (see k_cg_apply).
// FOLD: every workgroup folds its scene's errors itself, in the fold kernels' order, and takes the
// loop decision of k_fold_pressure; the scene's first workgroup records it (`done`, `l`). That may
// happen while the waves of another workgroup are still to start, so nobody looks at what it writes:
// whether the loop runs at all is read from `it`, which the evaluation wrote and this launch does
// not, and is therefore the same for every wave that goes through the fold's barriers. One launch
// less per iteration (4 us and its gap) for ~1 us in the apply.
template <bool REF, bool CUBIC, bool BOBJ, int Q, bool FOLD>
__global__ void __launch_bounds__(Q * kBlock) k_pressure_apply(Scenes sc, Nbr nb, Halo hl, const float4* __restrict__ pos,
                                                         float4* __restrict__ vel, const float4* __restrict__ bpos,
                                                         const float* __restrict__ bvol, const float* __restrict__ pG_ff,
                                                         const float* __restrict__ pG_fb, const float* __restrict__ kappa,
                                                         SolverDev* st, launch::FoldPressure fp) {
    static_assert(Q == 1 || !(REF || BOBJ), "coupled scenes and wall objects run one lane per slot");
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t N = sc.N;
    __shared__ float4 la[kStagePApply];
    BlockHead<Q, kHaloLoads<Q>> hd(blk, N, nb.cff, hl);
    const uint32_t i = hd.i, l = hd.l;
    const bool in = i < N;
    const uint32_t cb = in ? nb.cfb[i] : 0u;
    const float4 xi4 = in ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 vi4 = in ? vel[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float pi = in ? kappa[i] : 0.0f;
    const uint32_t sid = sc.blk_scene[blk];
    const StepParams P = sc.P[sid];
    if constexpr (FOLD) {
        const uint32_t it = st[sid].it;
        if (it == 0u) return;
        const double E = fold_everywhere<Q>(fp.partials + P.blk0, P.nblk) / double(P.count);
        const bool ok = E < fp.tol && it > fp.lmin;
        if (blk == P.blk0 && threadIdx.x == 0) record_pressure(st + sid, E, ok, it, fp.active);
        if (ok) return;
    } else {
        if (st[sid].done) return;
    }
    const bool live = i < P.end;
    const f3 xi = mk(xi4);
    f3 ff{0.f, 0.f, 0.f};
    using Val = GroupVal<Q>;
    auto walk_fluid = [&](auto staged) {
        constexpr bool STAGED = decltype(staged)::value;
        Walk<Q, STAGED, Val, Q == 1 ? kPrePressure : kPreQuad> wk(nb, hl, Streams{pG_ff}, i, l, N, hd.c);
        auto rec = [&](uint32_t j) {
            const float4 x = pos[j];
            return make_float4(x.x, x.y, x.z, kappa[j]);
        };
        if constexpr (STAGED) {
            hd.stage(rec, [&](uint32_t t, const float4& r) { la[t] = r; });
            __syncthreads();
        }
        auto at = [&](uint32_t j) -> float4 {
            if constexpr (STAGED) return la[j];
            else return rec(j);
        };
        auto term = [&](float G, const float4& a) { return 0.5f * P.V * (pi + a.w) * G * (xi - mk(a)); };
        wk.run(
            [&](uint32_t, const auto& x, const Val& G) {
                if constexpr (Q == 1) {
                    float4 r[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) r[e] = at(x.at(e));
#pragma unroll
                    for (int e = 0; e < 4; e++) ff = ff - term(G.at(e), r[e]);
                } else {
                    ff = sub_quad(ff, term(G.at(0), at(x.at(0))));
                }
            },
            [&](uint32_t, const auto& x, const Val& G, uint32_t n) {
                if constexpr (Q == 1) {
#pragma unroll
                    for (int e = 0; e < 3; e++)
                        if (e < int(n)) ff = ff - term(G.at(e), at(x.at(e)));
                } else {
                    f3 t{0.f, 0.f, 0.f};
                    if (l < n) t = term(G.at(0), at(x.at(0)));
                    ff = sub_quad(ff, t);
                }
            });
    };
    if (hd.H <= kStagePApply) walk_fluid(std::true_type{});
    else walk_fluid(std::false_type{});
    if (!live) return;
    f3 fb{0.f, 0.f, 0.f};
    f3 fbo[kMaxWallObjects] = {};
    struct WallRec {
        float4 x;
        float vb, G;
        uint32_t o;
    };
    walk_walls<Q>(nb, i, l, N, cb,
               [&](uint32_t j, size_t slot) { return WallRec{bpos[j], bvol[j], pG_fb[slot], BOBJ ? nb.fbo[j] : 0u}; },
               [&](bool in, size_t, const WallRec& w) {
        const f3 xij = xi - mk(w.x);
        f3 fij{0.f, 0.f, 0.f};
        if (in) fij = 0.5f * w.vb * pi * w.G * xij;
        if constexpr (BOBJ) at_obj(fbo, w.o, [&](f3& a) { a = a - fij; });
        else fb = sub_lanes<Q>(fb, fij);
    });
    f3 F{0.f, 0.f, 0.f};
    F = F + ff;
    if constexpr (REF) {  // ApplyDFSPH ref (MPSSPHDFSPHUtil.cuh:379-418): one sum per ref object
        const float invHi = 1.0f / (xi4.w * 4.0f);
        const uint32_t cr = nb.cfr[i];
        uint32_t cur = kEmpty;
        float Vt = 0.0f;
        f3 fr{0.f, 0.f, 0.f};
        for (uint32_t k = 0; k < cr; k++) {
            const uint32_t j = nb.fr[size_t(k) * N + i];
            const uint32_t t = sc.blk_scene[j / kBlock];
            if (t != cur) {
                if (cur != kEmpty) F = F + fr;
                cur = t;
                Vt = sc.P[t].V;
                fr = f3{0.f, 0.f, 0.f};
            }
            const f3 xij = xi - mk(pos[j]);
            fr = fr - 0.5f * Vt * (pi + kappa[j]) * Gk<CUBIC>(len3(xij), invHi) * xij;
        }
        if (cur != kEmpty) F = F + fr;
    }
    if constexpr (BOBJ) {
#pragma unroll
        for (uint32_t q = 0; q < kMaxWallObjects; q++)
            if (q < nb.nbo) F = F + fbo[q];
    } else {
        F = F + fb;
    }
    float4 v4 = vi4;
    const float m = v4.w;
    F = m * F;
    if (l == 0 && m > 1.0e-10f) {
        const float cdt = P.dt / m;
        v4.x = v4.x + cdt * F.x;
        v4.y = v4.y + cdt * F.y;
        v4.z = v4.z + cdt * F.z;
        vel[i] = v4;
    }
}

// ----------------------------------------------------------------- viscosity + surface tension CG
// ComputeSurfaceTensionFactor_kernel (MPSSPHNonPressureUtil.cuh:425-465) with the stored
// G_ij; also x0 = v (the copy into pPredictVel, MPSSPHNonPressureUtil.cu:144-147).
template <int Q>
__global__ void __launch_bounds__(Q * kBlock) k_st_factor(Scenes sc, Nbr nb, Halo hl, const float4* __restrict__ pos,
                                                    const float4* __restrict__ vel, const float* __restrict__ pG_ff,
                                                    float* __restrict__ fst, float4* __restrict__ cgx, launch::LoopStart ls) {
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t N = sc.N;
    // the block's halo (x_j, v_j, m_j) in LDS (see k_cg_apply)
    __shared__ float4 la[kStageST], lb[kStageST];
    BlockHead<Q, kHaloLoads<Q>> hd(blk, N, nb.cff, hl);
    const uint32_t i = hd.i, l = hd.l;
    const bool in = i < N;
    const float4 xi4 = in ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 vi4 = in ? vel[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t sid = sc.blk_scene[blk];
    reset_records(ls, sc, blk, sid);
    const bool live = i < sc.P[sid].end;
    const f3 xi = mk(xi4), vi = mk(vi4);
    float d = 0.0f;
    using Val = GroupVal<Q>;
    auto walk_fluid = [&](auto staged) {
        constexpr bool STAGED = decltype(staged)::value;
        Walk<Q, STAGED, Val, 1> wk(nb, hl, Streams{pG_ff}, i, l, N, hd.c);
        struct Rec {
            float4 x, v;
        };
        if constexpr (STAGED) {
            hd.stage([&](uint32_t j) { return Rec{pos[j], vel[j]}; },
                     [&](uint32_t t, const Rec& r) {
                         la[t] = make_float4(r.x.x, r.x.y, r.x.z, r.v.x);
                         lb[t] = make_float4(r.v.y, r.v.z, r.v.w, 0.0f);
                     });
            __syncthreads();
        }
        auto at = [&](uint32_t j) -> Rec {
            if constexpr (STAGED) {
                const float4 e = la[j], g = lb[j];
                return {e, make_float4(e.w, g.x, g.y, g.z)};
            } else {
                return {pos[j], vel[j]};
            }
        };
        auto term = [&](float G, const Rec& r) { return r.v.w * dot3(vi - mk(r.v), G * (xi - mk(r.x))); };
        wk.run(
            [&](uint32_t, const auto& x, const Val& G) {
                if constexpr (Q == 1) {
                    Rec r[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) r[e] = at(x.at(e));
#pragma unroll
                    for (int e = 0; e < 4; e++) d += term(G.at(e), r[e]);
                } else {
                    d = add_quad(d, term(G.at(0), at(x.at(0))));
                }
            },
            [&](uint32_t, const auto& x, const Val& G, uint32_t n) {
                if constexpr (Q == 1) {
#pragma unroll
                    for (int e = 0; e < 3; e++)
                        if (e < int(n)) d += term(G.at(e), at(x.at(e)));
                } else {
                    d = add_quad(d, l < n ? term(G.at(0), at(x.at(0))) : 0.0f);
                }
            });
    };
    if (hd.H <= kStageST) walk_fluid(std::true_type{});
    else walk_fluid(std::false_type{});
    if (live && l == 0) {
        fst[i] = d;
        cgx[i] = make_float4(vi4.x, vi4.y, vi4.z, 0.0f);
    }
}

// g_ij of the surface-tension operator (MPSSPHNonPressureUtil.cuh:503-512,563-572)
__device__ __forceinline__ float st_g(const StepParams& P, f3 vij, f3 xij, float dist, float invHi, float mi, float mj,
                                      float di, float dj, float fi, float fj, float& mij) {
    mij = 0.5f * (mi + mj);
    const float invDij = 2.0f / (di + dj);
    const float stW = STWk(dist, invHi);
    const f3 stG = STGk(dist, invHi) * xij;
    return (stW + P.dt * (dot3(vij, stG) - (fi + fj) * invDij * 0.5f * stW)) * invDij;
}

// Once per solve: right-hand side (ComputeSurfaceTensionCGb_kernel, :467-521) and the pair
// coefficients of the implicit operator (ST :523-585, viscosity :587-635, final :637-648):
//   a_ij = dt (cs_i m_ij g_ij + cx (m_j/rho_j) W_ij),   b_ij = -dt cv_i c_ij,
//   c_ij = (0.5(m_i+m_j) (1/rho_j)) Phi(d_ij)   (the reference's (0.5(m_i+m_j)/rho_j) /
//          (d^2 + 0.01 h_i^2) G_ij / (d + FLT_EPSILON) regrouped, see Phik),
//   cs_i = dt sigma/m_i, cx = XSPH/dt, cv_i = 10 rho0 mu/rho_i.
// Writes a_ij (ca), b_ij (cb, unless null), and 1/rho_i per slot (irho, unless null) for the A.p
// that recomputes b_ij.
// T: also the coefficients (a_ji, b_ji) of the pair seen from the neighbour, which the adjoint's
// transposed operator streams: the same expressions with the ends exchanged. (The lists are
// symmetric; what the neighbour's own entry holds has the same bits, since every factor that depends
// on the pair is even in x_ij.)
template <bool CUBIC, int Q, bool T>
__global__ void __launch_bounds__(Q * kBlock) k_cg_setup(Scenes sc, Nbr nb, Halo hl, const float4* __restrict__ pos,
                                                   const float4* __restrict__ vel, const float* __restrict__ rho,
                                                   const float* __restrict__ fst, float* __restrict__ ca, float* __restrict__ cb, float* __restrict__ caT,
                                                   float* __restrict__ cbT, float4* __restrict__ cgb, float* __restrict__ irho) {
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t N = sc.N;
    // the block's halo (x_j, v_j, m_j, rho_j, f_j) in LDS (see k_cg_apply)
    constexpr uint32_t kDepth = Q == 1 ? kStageSetup : kHaloCap;
    __shared__ float4 la[kDepth], lb[kDepth];
    __shared__ typename std::conditional<T, float2, float>::type lc[kDepth];  // f_j; T: (f_j, r_j)
    BlockHead<Q, kHaloLoads<Q>> hd(blk, N, nb.cff, hl);
    const uint32_t i = hd.i, l = hd.l;
    const bool in = i < N;
    const float4 xi4 = in ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 vi4 = in ? vel[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float di = in ? rho[i] : 0.0f, fi = in ? fst[i] : 0.0f;
    const uint32_t sid = sc.blk_scene[blk];
    const StepParams P = sc.P[sid];
    const bool live = i < P.end;
    const f3 xi = mk(xi4), vi = mk(vi4);
    const float mi = vi4.w;
    const float hi = xi4.w * 4.0f;
    const float invHi = 1.0f / hi;
    const float onePercentHSq = 0.01f * hi * hi;
    const float cs = P.dt * P.sigma / mi;
    const float cx = P.xsph / P.dt;
    const float cv = 10.0f * P.rho0 * P.mu / di;
    f3 bi{0.f, 0.f, 0.f};
    struct Rec {
        float4 x, v;
        float rho, f;
    };
    struct Term {
        float a, b, aT, bT;
        f3 s;
    };
    auto term = [&](const Rec& r) -> Term {
        const float mj = r.v.w, dj = r.rho;
        const f3 xij = xi - mk(r.x);
        const float dist = len3(xij);
        float mij;
        const float gij = st_g(P, vi - mk(r.v), xij, dist, invHi, mi, mj, di, dj, fi, r.f, mij);
        const float sij = mij * gij;
        const float wij = mj / dj * Wk<CUBIC>(dist, invHi);
        Term t;
        t.a = P.dt * (cs * sij + cx * wij);
        t.b = t.aT = t.bT = 0.0f;
        if (T || cb) {
            const float irhoj = 1.0f / dj;
            const float cij = 0.5f * (mi + mj) * irhoj * Phik<CUBIC>(dist, invHi, onePercentHSq);
            t.b = -P.dt * cv * cij;
        }
        t.s = sij * xij;
        if constexpr (T) {
            const float hj = r.x.w * 4.0f, invHj = 1.0f / hj;
            float mji;
            const float gji = st_g(P, vi - mk(r.v), xij, dist, invHj, mj, mi, dj, di, r.f, fi, mji);
            const float sji = mji * gji;
            const float wji = mi / di * Wk<CUBIC>(dist, invHj);
            t.aT = P.dt * (P.dt * P.sigma / mj * sji + cx * wji);
            const float cvj = 10.0f * P.rho0 * P.mu / dj;
            const float cji = 0.5f * (mj + mi) * (1.0f / di) * Phik<CUBIC>(dist, invHj, 0.01f * hj * hj);
            t.bT = -P.dt * cvj * cji;
        }
        return t;
    };
    auto walk_fluid = [&](auto staged) {
        constexpr bool STAGED = decltype(staged)::value;
        Walk<Q, STAGED, NoVal, 1> wk(nb, hl, Streams{}, i, l, N, hd.c);
        if constexpr (STAGED) {
            hd.stage([&](uint32_t j) { return Rec{pos[j], vel[j], rho[j], fst[j]}; },
                     [&](uint32_t t, const Rec& r) {
                         la[t] = make_float4(r.x.x, r.x.y, r.x.z, r.v.x);
                         lb[t] = make_float4(r.v.y, r.v.z, r.v.w, r.rho);
                         if constexpr (T) lc[t] = make_float2(r.f, r.x.w);
                         else lc[t] = r.f;
                     });
            __syncthreads();
        }
        auto at = [&](uint32_t j) -> Rec {
            if constexpr (STAGED) {
                const float4 e = la[j], g = lb[j];
                const auto f = lc[j];
                if constexpr (T) return {make_float4(e.x, e.y, e.z, f.y), make_float4(e.w, g.x, g.y, g.z), g.w, f.x};
                else return {e, make_float4(e.w, g.x, g.y, g.z), g.w, f};
            } else {
                return {pos[j], vel[j], rho[j], fst[j]};
            }
        };
        // one entry's coefficients at its place in the list
        auto put = [&](size_t entry, const Term& t) {
            ca[entry] = t.a;
            if (T || cb) cb[entry] = t.b;
            if constexpr (T) {
                caT[entry] = t.aT;
                cbT[entry] = t.bT;
            }
        };
        wk.run(
            [&](uint32_t g, const auto& x, const NoVal&) {
                const size_t group = size_t(g) * N + i;
                if constexpr (Q == 1) {
                    Term t[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        t[e] = term(at(x.at(e)));
                        bi = bi - t[e].s;
                    }
                    reinterpret_cast<v4f*>(ca)[group] = v4f{t[0].a, t[1].a, t[2].a, t[3].a};
                    if (T || cb) reinterpret_cast<v4f*>(cb)[group] = v4f{t[0].b, t[1].b, t[2].b, t[3].b};
                    if constexpr (T) {
                        reinterpret_cast<v4f*>(caT)[group] = v4f{t[0].aT, t[1].aT, t[2].aT, t[3].aT};
                        reinterpret_cast<v4f*>(cbT)[group] = v4f{t[0].bT, t[1].bT, t[2].bT, t[3].bT};
                    }
                } else {
                    const Term t = term(at(x.at(0)));
                    put(4 * group + l, t);
                    bi = sub_quad(bi, t.s);
                }
            },
            [&](uint32_t g, const auto& x, const NoVal&, uint32_t n) {
                const size_t group = size_t(g) * N + i;
                if constexpr (Q == 1) {
#pragma unroll 1
                    for (int e = 0; e < int(n); e++) {
                        const Term t = term(at(x.at(e)));
                        put(4 * group + e, t);
                        bi = bi - t.s;
                    }
                } else {
                    Term t{0.f, 0.f, 0.f, 0.f, {0.f, 0.f, 0.f}};
                    if (l < n) {
                        t = term(at(x.at(0)));
                        put(4 * group + l, t);
                    }
                    bi = sub_quad(bi, t.s);
                }
            });
    };
    if (hd.H <= kDepth) walk_fluid(std::true_type{});
    else walk_fluid(std::false_type{});
    if (!live || l != 0) return;
    if (irho) irho[i] = 1.0f / di;
    const f3 b = (P.dt * P.sigma / mi) * bi + vi;
    cgb[i] = make_float4(b.x, b.y, b.z, 0.0f);
}

// (A p)_i = (1+f) p_i + sum_j [ a_ij p_ij + (b_ij (p_ij . x_ij)) x_ij ].
// a_ij is written once per solve by k_cg_setup and streamed here with non-temporal loads. b_ij
// is either streamed with it (RECOMP false: 8 bytes per pair) or recomputed here from the
// geometry (RECOMP true: 4 bytes per pair streamed, one square root and one division per pair:
// b_ij = (-dt cv_i) ((0.5 (m_i + m_j) (1/rho_j)) Phi(d_ij)), the expression k_cg_setup
// evaluates). The block's halo records (x_j, p_j: 24 bytes; with m_j and 1/rho_j when b_ij is
// recomputed: 32 bytes) are staged in LDS first, with coalesced loads of the sorted halo list,
// and each pair reads its neighbour there through the 16-bit list; a block whose halo is over
// the limit gathers from global memory. Both paths visit the same pairs in the same order, so
// the result depends on neither the path nor RECOMP.
// The search direction of UpdateCGDirection_kernel (MPSCGKernel.cuh:123-133),
// p = r + beta p_prev, is formed here for every record read (own and halo) instead of in a
// pass of its own; the block writes its own p for the update kernel (pout, while pprev is
// read: the host alternates the two buffers). beta = 0 in the first iteration, where
// pprev = r, so p = r.
// The CG vectors are packed 12-byte triples (f3).
// MODE 0: A x0 with f = 0 (x0 in x0) fused with InitCGResidual_kernel (MPSCGKernel.cuh:5-19):
//         r = b - A x0, pout = r, x = x0, partial sums of r.r.
// MODE 1: A p with f (r in rr), partial sums of p.Ap (MPSCGKernel.cuh:21-67).
// One workgroup's share of A.p: block `blk`. head() gives its scene, whether that scene's loop has
// finished, and the search-direction factor; it is called once the loads that need none of these
// are on their way.
// TRANS: the adjoint's A_f^T p, (1+f) p_i + sum_j [ (a_ij p_i - a_ji p_j) + (b_ij (p_i.x_ij) -
// b_ji (p_j.x_ij)) x_ij ], with the neighbour's coefficients streamed beside the own ones; its MODE 0
// starts a solve from a guess x0 (r = b - A_f^T x0, f included; partial sums of r.r and, gridDim.x
// further, of b.b). At 64k particles (256 workgroups, 28 neighbours each) an iteration of the
// transposed solve took five launches and 44 us with one entry per load and its records gathered from
// L2 (24 us of it A^T.p); staged, in groups, with the direction and the folds inside: two and 17 us.
// PCOH: the partial sum is stored device-coherently (a workgroup of the same launch folds it).
struct CgHead {
    uint32_t sid;
    bool done;
    float beta;
};
template <int MODE, bool RECOMP, bool CUBIC, bool COH = false, bool PCOH = COH, uint32_t DEPTH = kStageAp, int Q = 1, bool TRANS = false, bool KEEP = false, class Head>
__device__ __forceinline__ void cg_apply_block(uint32_t blk, Head&& head, const Scenes& sc, const Nbr& nb,
                                               const Halo& hl, const Streams& coef,
                                               const float4* __restrict__ pos, const float4* __restrict__ vel,
                                               const float* __restrict__ rho, const float* __restrict__ irho,
                                               const float4* __restrict__ x0, const f3* __restrict__ rr,
                                               const f3* __restrict__ pprev, f3* __restrict__ pout, f3* __restrict__ Ap,
                                               const float4* __restrict__ b, f3* __restrict__ r, f3* __restrict__ x,
                                               double* __restrict__ partials) {
    const uint32_t N = sc.N;
    using LB = typename std::conditional<RECOMP, float4, float2>::type;
    __shared__ float4 la[DEPTH];
    __shared__ LB lb[DEPTH];
    BlockHead<Q, kHaloLoadsApply> hd(blk, N, nb.cff, hl);
    const uint32_t i = hd.i, l = hd.l;
    const CgHead ch = head();
    if (ch.done) return;
    const float bta = ch.beta;
    const StepParams P = sc.P[ch.sid];
    const bool live = i < P.end;
    // the vector the operator is applied to, at slot j
    auto vec = [&](uint32_t j) -> f3 {
        if (MODE == 0) return mk(x0[j]);
        const f3 a = ld3c<COH>(rr + j), q = ld3c<COH>(pprev + j);
        return {a.x + bta * q.x, a.y + bta * q.y, a.z + bta * q.z};
    };
    // b_ij's per-particle factors, as k_cg_setup forms them (RECOMP)
    float mi = 0.0f, ncv = 0.0f, invHi = 0.0f, h2 = 0.0f;
    f3 xi{0.f, 0.f, 0.f}, pi{0.f, 0.f, 0.f}, acc{0.f, 0.f, 0.f};
    // one halo record: (x_j, p_j) and, for RECOMP, (m_j, 1/rho_j)
    struct Rec {
        f3 x, p;
        float m, irho;
    };
    auto term = [&](float a, float bb, const Rec& q) -> f3 {
        const f3 xij = xi - q.x;
        const f3 pij = pi - q.p;
        if constexpr (RECOMP) {
            const float dist = len3(xij);
            const float cij = 0.5f * (mi + q.m) * q.irho * Phik<CUBIC>(dist, invHi, h2);
            const float bij = ncv * cij;
            return a * pij + (bij * dot3(pij, xij)) * xij;
        } else {
            return a * pij + (bb * dot3(pij, xij)) * xij;
        }
    };
    using Val = typename std::conditional<TRANS, GroupABT<Q, KEEP>,
                                          typename std::conditional<RECOMP, GroupVal<Q>, GroupAB<Q, KEEP>>::type>::type;
    auto walk_fluid = [&](auto staged) {
        constexpr bool STAGED = decltype(staged)::value;
        // the first groups are loaded before the halo staging: their stream overlaps the
        // staging's gathers instead of following them
        Walk<Q, STAGED, Val, Q == 1 ? kPreApply : kPreQuad> wk(nb, hl, coef, i, l, N, hd.c);
        auto rec = [&](uint32_t j) -> Rec {
            const float4 xj = pos[j];
            if constexpr (RECOMP) return {mk(xj), vec(j), vel[j].w, irho[j]};
            else return {mk(xj), vec(j), 0.0f, 0.0f};
        };
        if (live) {
            const float4 xi4 = pos[i];
            xi = mk(xi4);
            pi = vec(i);
            if constexpr (RECOMP) {
                mi = vel[i].w;
                const float cv = 10.0f * P.rho0 * P.mu / rho[i];
                ncv = -P.dt * cv;
                const float hi = xi4.w * 4.0f;
                invHi = 1.0f / hi;
                h2 = 0.01f * hi * hi;
            }
        }
        if constexpr (STAGED) {
            hd.stage(rec, [&](uint32_t t, const Rec& q) {
                la[t] = make_float4(q.x.x, q.x.y, q.x.z, q.p.x);
                if constexpr (RECOMP) lb[t] = make_float4(q.p.y, q.p.z, q.m, q.irho);
                else lb[t] = make_float2(q.p.y, q.p.z);
            });
            __syncthreads();
        }
        auto at = [&](uint32_t j) -> Rec {
            if constexpr (STAGED) {
                const float4 a = la[j];
                const LB e = lb[j];
                if constexpr (RECOMP) return {mk(a), {a.w, e.x, e.y}, e.z, e.w};
                else return {mk(a), {a.w, e.x, e.y}, 0.0f, 0.0f};
            } else {
                return rec(j);
            }
        };
        // the terms of one entry, added to the sum one after the other (one term, or two if TRANS)
        struct Terms {
            f3 a, b;
        };
        auto entry = [&](const Val& v, int e, const Rec& q) -> Terms {
            if constexpr (TRANS) {
                const f3 xij = xi - q.x;
                return {v.a.at(e) * pi - v.aT.at(e) * q.p, (v.b.at(e) * dot3(pi, xij) - v.bT.at(e) * dot3(q.p, xij)) * xij};
            } else if constexpr (RECOMP) {
                return {term(v.at(e), 0.0f, q), {}};
            } else {
                return {term(v.a.at(e), v.b.at(e), q), {}};
            }
        };
        auto add = [&](const Terms& t) {
            if constexpr (Q == 1) {
                acc = acc + t.a;
                if constexpr (TRANS) acc = acc + t.b;
            } else if constexpr (TRANS) {
                acc = add_quad(acc, t.a, t.b);
            } else {
                acc = add_quad(acc, t.a);
            }
        };
        wk.run(
            [&](uint32_t, const auto& jx, const Val& v) {
                if constexpr (Q == 1) {
                    Rec q[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) q[e] = at(jx.at(e));
#pragma unroll
                    for (int e = 0; e < 4; e++) add(entry(v, e, q[e]));
                } else {
                    add(entry(v, 0, at(jx.at(0))));
                }
            },
            [&](uint32_t, const auto& jx, const Val& v, uint32_t n) {
                if constexpr (Q == 1) {
#pragma unroll
                    for (int e = 0; e < 3; e++)
                        if (e < int(n)) add(entry(v, e, at(jx.at(e))));
                } else {
                    Terms t{};
                    if (l < n) t = entry(v, 0, at(jx.at(0)));
                    add(t);
                }
            });
    };
    if (hd.H <= DEPTH) walk_fluid(std::true_type{});  // the same for the whole block
    else walk_fluid(std::false_type{});               // halo over the limit: gather from global memory
    double part = 0.0, part_b = 0.0;
    if (live && l == 0) {
        const float f = MODE == 0 && !TRANS ? 0.0f : P.cg_factor;
        const f3 o = pi * (1.0f + f) + acc;
        if (MODE == 0) {
            const float4 bi = b[i];
            const f3 ri{bi.x - o.x, bi.y - o.y, bi.z - o.z};
            r[i] = ri;
            pout[i] = ri;
            x[i] = pi;
            part = double(ri.x * ri.x) + double(ri.y * ri.y) + double(ri.z * ri.z);
            if constexpr (TRANS) part_b = double(bi.x * bi.x) + double(bi.y * bi.y) + double(bi.z * bi.z);
        } else {
            st3c<COH>(pout + i, pi);
            Ap[i] = o;
            part = double(pi.x * o.x) + double(pi.y * o.y) + double(pi.z * o.z);
        }
    }
    slot_partial<Q, PCOH>(part, partials, blk);
    if constexpr (TRANS && MODE == 0) {
        __syncthreads();
        slot_partial<Q>(part_b, partials + gridDim.x, blk);
    }
}

// What k_fold_cg<2> records of iteration `it`: `s` is the new r.r, `prev` the one before.
__device__ __forceinline__ void record_cg(SolverDev* st, double s, double prev, bool done, uint32_t* active) {
    const uint32_t it = st->l;
    st->beta = float(s / prev);
    st->rr = s;
    if (it < MPS_MAX_ITER_LOG) st->log[it] = s;
    st->l = it + 1;
    if (done) {
        st->done = 1u;
        atomicSub(active, 1u);
    }
}
__device__ __forceinline__ bool cg_done(double s, double thr, double tol) { return s < thr || (tol < 0.0 && s == 0.0); }

// FOLD (MODE 1): every workgroup first folds its scene's r.r of the last update itself, in the fold
// kernels' order, forms beta and takes the convergence test of k_fold_cg<2>; the scene's first
// workgroup records them, possibly before the waves of another workgroup start. Before the fold
// every wave therefore reads only words of the record that this launch does not write: `thr`, and
// `it` (0: the loop has ended) and `rr_prev`, which the update keeps.
template <int MODE, bool RECOMP, bool CUBIC, bool DEEP = false, int Q = 1, bool FOLD = false, bool TRANS = false, bool KEEP = false>
__global__ void __launch_bounds__(Q * kBlock) k_cg_apply(Scenes sc, Nbr nb, Halo hl, Streams coef, const float4* __restrict__ pos,
                                                   const float4* __restrict__ vel, const float* __restrict__ rho,
                                                   const float* __restrict__ irho, const float4* __restrict__ x0,
                                                   const f3* __restrict__ rr, const f3* __restrict__ pprev,
                                                   f3* __restrict__ pout, f3* __restrict__ Ap,
                                                   const float4* __restrict__ b, f3* __restrict__ r, f3* __restrict__ x,
                                                   SolverDev* st, double* __restrict__ partials, launch::FoldCg fc) {
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    auto head = [&]() -> CgHead {
        const uint32_t sid = sc.blk_scene[blk];
        if (MODE == 0) return {sid, false, 0.0f};
        if constexpr (FOLD) {
            if (st[sid].it == 0u) return {sid, true, 0.0f};
            const uint32_t blk0 = sc.P[sid].blk0;
            const double prev = st[sid].rr_prev, thr = st[sid].thr;
            const double s = fold_everywhere<Q>(fc.partials + blk0, sc.P[sid].nblk);
            const bool done = cg_done(s, thr, fc.tol);
            if (blk == blk0 && threadIdx.x == 0) record_cg(st + sid, s, prev, done, fc.active);
            return {sid, done, float(s / prev)};
        }
        return {sid, st[sid].done != 0u, st[sid].beta};
    };
    cg_apply_block<MODE, RECOMP, CUBIC, false, false, DEEP ? kHaloCap : kStageAp, Q, TRANS, KEEP>(
        blk, head, sc, nb, hl, coef, pos, vel, rho, irho, x0, rr, pprev, pout, Ap, b, r, x, partials);
}

// Scalars of CGSolver (MPSSolver.cuh:31-65). MODE 0: r.r of the initial residual and the
// first convergence test; 1: alpha = r.r / p.Ap; 2: r.r of the new residual, beta, test.
// Workgroup s folds scene s's partials.
// MODE 2 takes the iteration number from the record's l (it, when iteration it is folded).
template <int MODE>
__global__ void __launch_bounds__(kFoldThreads) k_fold_cg(Scenes sc, const double* __restrict__ partials, SolverDev* stv,
                                                  uint32_t* active, double tol) {
    const uint32_t sid = blockIdx.x;
    SolverDev* st = stv + sid;
    if (st->done) return;
    const StepParams P = sc.P[sid];
    const double s = fold(partials + P.blk0, P.nblk);
    if (threadIdx.x != 0) return;
    if (MODE == 0) {
        st->rr = s;
        st->log[0] = s;
        st->l = 1u;
        st->thr = tol < 0.0 ? -tol * s : tol;  // a negative tolerance is relative to r0.r0
        if (s < st->thr || (tol < 0.0 && s == 0.0)) {
            st->done = 1u;
            atomicSub(active, 1u);
        }
    } else if (MODE == 1) {
        st->pAp = s;
        st->alpha = float(st->rr / s);
    } else {
        record_cg(st, s, st->rr, cg_done(s, st->thr, tol), active);
    }
}

// UpdateCGResidual_kernel + the r.r half of ComputeCGBetaParam_kernel (MPSCGKernel.cuh:69-121), on
// packed triples.
template <bool COH = false, bool PCOH = COH>
__device__ __forceinline__ void cg_update3_block(uint32_t blk, uint32_t end, float a, f3* __restrict__ x,
                                                 f3* __restrict__ r, const f3* __restrict__ p, const f3* __restrict__ Ap,
                                                 double* __restrict__ partials) {
    const uint32_t i = blk * blockDim.x + threadIdx.x;
    double part = 0.0;
    if (i < end) {
        const f3 pi = ld3c<COH>(p + i), api = Ap[i];
        f3 xi = x[i], ri = ld3c<COH>(r + i);
        xi.x = xi.x + a * pi.x;
        xi.y = xi.y + a * pi.y;
        xi.z = xi.z + a * pi.z;
        ri.x = ri.x - a * api.x;
        ri.y = ri.y - a * api.y;
        ri.z = ri.z - a * api.z;
        x[i] = xi;
        st3c<COH>(r + i, ri);
        part = double(ri.x * ri.x) + double(ri.y * ri.y) + double(ri.z * ri.z);
    }
    block_partial<PCOH>(part, partials, blk);
}
// FOLD: every workgroup first folds its scene's p.Ap itself and forms alpha (k_fold_cg<1>); the
// scene's first workgroup records it and keeps what the next A.p reads before its own fold: the r.r
// as rr_prev, and the iteration, or 0 once the loop has ended, as `it`. No workgroup of this launch
// reads either, and none writes `done`.
template <bool FOLD>
__global__ void __launch_bounds__(kBlock) k_cg_update3(Scenes sc, f3* __restrict__ x, f3* __restrict__ r,
                                                     const f3* __restrict__ p, const f3* __restrict__ Ap,
                                                     SolverDev* st, const double* __restrict__ pAp,
                                                     double* __restrict__ partials) {
    const uint32_t sid = sc.blk_scene[blockIdx.x];
    const bool done = st[sid].done != 0u;
    const bool first = FOLD && blockIdx.x == sc.P[sid].blk0 && threadIdx.x == 0;  // keeps the record
    if (first) st[sid].it = done ? 0u : st[sid].l;
    if (done) return;
    float alpha;
    if constexpr (FOLD) {
        const uint32_t blk0 = sc.P[sid].blk0;
        const double rr = st[sid].rr;
        const double s = fold_as_fold_kernel<false>(pAp + blk0, sc.P[sid].nblk);
        alpha = float(rr / s);
        if (first) {
            st[sid].pAp = s;
            st[sid].alpha = alpha;
            st[sid].rr_prev = rr;
        }
    } else {
        alpha = st[sid].alpha;
    }
    cg_update3_block(blockIdx.x, sc.P[sid].end, alpha, x, r, p, Ap, partials);
}

// ----------------------------------------------------------------- persistent CG
// Grid-wide barrier of a co-resident grid (cooperative launch). The wait is bounded: after
// `spin` polls, or when another workgroup gave up, it sets gs->gave_up and returns false, and
// the caller leaves the kernel; every workgroup's wait then ends within `spin` polls.
// COH false: agent-scope fences publish the workgroup's writes before it arrives and make the
// others' visible after the barrier (each workgroup writes back and invalidates its L2).
// COH true: the data that crosses workgroups is written and read device-coherently (ld3c,
// st3c, coherent partials), so each wave only waits until its own stores are performed before
// the workgroup arrives, and the barrier orders nothing else.
template <bool COH>
__device__ __forceinline__ bool grid_barrier(GridSync* gs, uint32_t nwg, uint32_t spin) {
    __shared__ uint32_t ok_s;
    if constexpr (COH) __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t ok = 1u;
        const uint32_t g = __hip_atomic_load(&gs->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (!COH) __threadfence();
        // arrivals are counted per group of kGridGroup workgroups, and the last of each group
        // counts the group: 16 + nwg/16 serialized atomics instead of nwg
        const uint32_t grp = blockIdx.x / kGridGroup;
        const uint32_t gsize = min(kGridGroup, nwg - grp * kGridGroup);
        const uint32_t ngrp = (nwg + kGridGroup - 1u) / kGridGroup;
        bool last = false;
        if (__hip_atomic_fetch_add(&gs->group[grp], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == gsize) {
            __hip_atomic_store(&gs->group[grp], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if constexpr (COH) __builtin_amdgcn_s_waitcnt(0);
            if (__hip_atomic_fetch_add(&gs->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == ngrp) {
                last = true;
                __hip_atomic_store(&gs->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if constexpr (COH) {
                    __builtin_amdgcn_s_waitcnt(0);
                    __hip_atomic_fetch_add(&gs->gen, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
                    __hip_atomic_fetch_add(&gs->gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        if (!last) {
            uint32_t polls = 0;
            while (__hip_atomic_load(&gs->gen, COH ? __ATOMIC_RELAXED : __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) == g) {
                if (__hip_atomic_load(&gs->gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u || ++polls > spin) {
                    ok = 0u;
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
        }
        if (!ok) __hip_atomic_store(&gs->gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (!COH) __threadfence();
        ok_s = ok && __hip_atomic_load(&gs->gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u;
    }
    __syncthreads();
    return ok_s != 0u;
}

// The CG iterations of CGSolver (MPSSolver.cuh:31-65) in one launch of a co-resident grid (one
// workgroup per 256-slot block of every scene), for iterations 1..cap after the initial
// residual (k_cg_apply<0> + k_fold_cg<0> ran before). Per iteration: A.p with the direction
// update (cg_apply_block) -> barrier -> every workgroup folds p.Ap itself (the fold kernels'
// order, so alpha has the same bits) -> x, r update (cg_update3_block) -> barrier -> r.r fold,
// beta and the test. The scene's first workgroup keeps the solver record as the fold kernels
// do. A scene that converged sits out; the loop ends for everyone when no scene is running
// (the running count is read right after the first barrier, where no workgroup changes it) or
// after iteration cap. Partial sums alternate between two buffers, so a fold never reads a
// buffer that the next phase writes. Results are those of the chunked launches bit for bit.
template <bool RECOMP, bool CUBIC, bool COH>
__global__ void __launch_bounds__(kBlock) k_cg_persistent(Scenes sc, Nbr nb, Halo hl, Streams coef, const float4* __restrict__ pos,
                                                        const float4* __restrict__ vel, const float* __restrict__ rho,
                                                        const float* __restrict__ irho, f3* __restrict__ r,
                                                        f3* __restrict__ pbuf0, f3* __restrict__ pbuf1, f3* __restrict__ Ap,
                                                        f3* __restrict__ x, SolverDev* stv, uint32_t* active,
                                                        double* __restrict__ partA, double* __restrict__ partB,
                                                        GridSync* gs, uint32_t cap, double tol, uint32_t spin) {
    const uint32_t nwg = gridDim.x;
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t sid = sc.blk_scene[blk];
    const StepParams P = sc.P[sid];
    SolverDev* st = stv + sid;
    const bool writer = blk == P.blk0 && threadIdx.x == 0;
    __shared__ uint32_t running_s;
    bool done = st->done != 0u;
    double rr = st->rr;
    const double thr = st->thr;
    float beta = st->beta;
    for (uint32_t k = 1; k <= cap; k++) {
        f3* pprev = (k & 1u) ? pbuf0 : pbuf1;  // p of iteration k - 1 (p_0 = r in pbuf0)
        f3* pout = (k & 1u) ? pbuf1 : pbuf0;
        if (!done)
            cg_apply_block<1, RECOMP, CUBIC, COH>(blk, [&]() -> CgHead { return {sid, false, beta}; }, sc, nb, hl, coef, pos, vel, rho, irho, nullptr, r, pprev,
                                                  pout, Ap, nullptr, nullptr, nullptr, partA);
        if (!grid_barrier<COH>(gs, nwg, spin)) return;
        if (threadIdx.x == 0) running_s = __hip_atomic_load(active, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (running_s == 0u) return;
        float alpha = 0.0f;
        if (!done) {
            const double pAp = fold_as_fold_kernel<COH>(partA + P.blk0, P.nblk);
            alpha = float(rr / pAp);
            if (writer) {
                st->pAp = pAp;
                st->alpha = alpha;
            }
            cg_update3_block<COH>(blk, P.end, alpha, x, r, pout, Ap, partB);
        }
        if (!grid_barrier<COH>(gs, nwg, spin)) return;
        if (!done) {
            const double s = fold_as_fold_kernel<COH>(partB + P.blk0, P.nblk);
            beta = float(s / rr);
            rr = s;
            done = s < thr || (tol < 0.0 && s == 0.0);
            if (writer) {
                st->beta = beta;
                st->rr = s;
                if (k < MPS_MAX_ITER_LOG) st->log[k] = s;
                st->l = k + 1u;
                if (done) {
                    st->done = 1u;
                    atomicSub(active, 1u);
                }
            }
        }
    }
}

// ----------------------------------------------------------------- folds in the last workgroup
// The chunked CG without fold launches: each workgroup stores its partial device-coherently,
// waits until the store is performed and counts itself; the scene's last workgroup to arrive
// then sees every partial, folds them in the fold kernels' order (fold_as_fold_kernel, so the
// scalars have the same bits) and updates the record as k_fold_cg<MODE> would, for the next
// launch. Nothing waits for anything: the other workgroups simply end. Arrivals are counted in
// two levels, as same-address atomics serialize: groups of kArriveGroup consecutive workgroups
// of the scene count in arrive[blk0 + group], and the last of each group counts the group in
// the solver record's counter. Every counter is back at zero when the launch ends.
constexpr uint32_t kArriveGroup = 64;
template <int MODE>
__device__ __forceinline__ void fold_in_last_workgroup(const Scenes& sc, uint32_t sid, uint32_t blk,
                                                       const double* __restrict__ partials, SolverDev* stv, uint32_t* active,
                                                       double tol, uint32_t* arrive) {
    __shared__ uint32_t last_s;
    const StepParams P = sc.P[sid];
    SolverDev* st = stv + sid;
    __builtin_amdgcn_s_waitcnt(0);  // the partial (thread 0's coherent store) is performed
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t grp = (blk - P.blk0) / kArriveGroup;
        const uint32_t gsize = min(kArriveGroup, P.nblk - grp * kArriveGroup);
        const uint32_t ngrp = (P.nblk + kArriveGroup - 1u) / kArriveGroup;
        uint32_t* gc = arrive + P.blk0 + grp;
        bool last = false;
        if (__hip_atomic_fetch_add(gc, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == gsize) {
            __hip_atomic_store(gc, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last = __hip_atomic_fetch_add(&st->counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == ngrp;
        }
        last_s = last;
    }
    __syncthreads();
    if (!last_s) return;
    const double s = fold_as_fold_kernel<true>(partials + P.blk0, P.nblk);
    if (threadIdx.x != 0) return;
    __hip_atomic_store(&st->counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (MODE == 1) {
        st->pAp = s;
        st->alpha = float(st->rr / s);
    } else {
        record_cg(st, s, st->rr, cg_done(s, st->thr, tol), active);
    }
}
// k_cg_apply<1> + k_fold_cg<1> in one launch
template <bool RECOMP, bool CUBIC>
__global__ void __launch_bounds__(kBlock) k_cg_apply_fold(Scenes sc, Nbr nb, Halo hl, Streams coef, const float4* __restrict__ pos,
                                                        const float4* __restrict__ vel, const float* __restrict__ rho,
                                                        const float* __restrict__ irho, const f3* __restrict__ rr,
                                                        const f3* __restrict__ pprev, f3* __restrict__ pout,
                                                        f3* __restrict__ Ap, SolverDev* st, double* __restrict__ partials,
                                                        uint32_t* arrive) {
    const uint32_t blk = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t sid = sc.blk_scene[blk];
    if (st[sid].done) return;
    cg_apply_block<1, RECOMP, CUBIC, false, true>(blk, [&]() -> CgHead { return {sid, false, st[sid].beta}; }, sc, nb, hl, coef, pos, vel, rho, irho, nullptr, rr,
                                                  pprev, pout, Ap, nullptr, nullptr, nullptr, partials);
    fold_in_last_workgroup<1>(sc, sid, blk, partials, st, nullptr, 0.0, arrive);
}
// k_cg_update3 + k_fold_cg<2> in one launch
__global__ void __launch_bounds__(kBlock) k_cg_update3_fold(Scenes sc, f3* __restrict__ x, f3* __restrict__ r,
                                                          const f3* __restrict__ p, const f3* __restrict__ Ap, SolverDev* st,
                                                          double* __restrict__ partials, uint32_t* active, double tol,
                                                          uint32_t* arrive) {
    const uint32_t sid = sc.blk_scene[blockIdx.x];
    if (st[sid].done) return;
    cg_update3_block<false, true>(blockIdx.x, sc.P[sid].end, st[sid].alpha, x, r, p, Ap, partials);
    fold_in_last_workgroup<2>(sc, sid, blockIdx.x, partials, st, active, tol, arrive);
}

__global__ void __launch_bounds__(kBlock) k_copy_vel_out3(Scenes sc, const f3* __restrict__ x, float4* __restrict__ vel,
                                                        launch::Gate gate, launch::LoopStart ls) {
    const uint32_t sid = sc.blk_scene[blockIdx.x];
    reset_records(ls, sc, blockIdx.x, sid);
    if (shut(gate)) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= sc.P[sid].end) return;
    const f3 xi = x[i];
    float4 v = vel[i];
    v.x = xi.x;
    v.y = xi.y;
    v.z = xi.z;
    vel[i] = v;
}
__global__ void __launch_bounds__(kBlock) k_copy_vel_out(Scenes sc, const float4* __restrict__ x, float4* __restrict__ vel) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= sc.P[sc.blk_scene[blockIdx.x]].end) return;
    const float4 xi = x[i];
    float4 v = vel[i];
    v.x = xi.x;
    v.y = xi.y;
    v.z = xi.z;
    vel[i] = v;
}

// ----------------------------------------------------------------- Jacobi viscosity
// ComputeJacobiViscosity kernels (MPSSPHNonPressureUtil.cuh:90-194, commented out in the
// reference): per particle a 3x3 block with A_ij = V G/((d^2+0.01h^2)(d+eps)) x_ij x_ij^T.
template <bool CUBIC>
__global__ void __launch_bounds__(kBlock) k_jacobi_candidate(Scenes sc, Nbr nb, const float4* __restrict__ pos,
                                                           const float4* __restrict__ vel, const float* __restrict__ rho,
                                                           const float4* __restrict__ u, float4* __restrict__ out) {
    const uint32_t sid = sc.blk_scene[blockIdx.x];
    const StepParams P = sc.P[sid];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t N = P.N;
    if (i >= P.end) return;
    const float4 xi4 = pos[i];
    const f3 xi = mk(xi4);
    const float h = xi4.w * 4.0f;
    const float invH = 1.0f / h;
    const float onePercentHSq = 0.01f * h * h;
    float A[3][3] = {{0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}, {0.f, 0.f, 0.f}};
    f3 Avj{0.f, 0.f, 0.f};
    const uint32_t c = nb.cff[i];
    for (uint32_t k = 0; k < c; k++) {
        const uint32_t j = nbr_ff(nb, k, i, N);
        const f3 xij = xi - mk(pos[j]);
        const float dist = len3(xij);
        if (dist < h) {
            const f3 uj = mk(u[j]);
            const float cc = P.V * Gk<CUBIC>(dist, invH) / ((dist * dist + onePercentHSq) * (dist + kFltEps));
            const float M[3][3] = {{cc * (xij.x * xij.x), cc * (xij.y * xij.x), cc * (xij.z * xij.x)},
                                   {cc * (xij.x * xij.y), cc * (xij.y * xij.y), cc * (xij.z * xij.y)},
                                   {cc * (xij.x * xij.z), cc * (xij.y * xij.z), cc * (xij.z * xij.z)}};
            const f3 uM{dot3(uj, f3{M[0][0], M[0][1], M[0][2]}), dot3(uj, f3{M[1][0], M[1][1], M[1][2]}),
                        dot3(uj, f3{M[2][0], M[2][1], M[2][2]})};
            Avj = Avj - uM;
#pragma unroll
            for (int a = 0; a < 3; a++)
#pragma unroll
                for (int bq = 0; bq < 3; bq++) A[a][bq] = A[a][bq] - M[a][bq];
        }
    }
    const float al = P.dt * 10.0f * P.mu / rho[i];
    Avj = Avj * al;
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int bq = 0; bq < 3; bq++) A[a][bq] = A[a][bq] * al + (a == bq ? 1.0f : 0.0f);
    const float oneOverDet = 1.0f / (+A[0][0] * (A[1][1] * A[2][2] - A[2][1] * A[1][2]) -
                                     A[1][0] * (A[0][1] * A[2][2] - A[2][1] * A[0][2]) +
                                     A[2][0] * (A[0][1] * A[1][2] - A[1][1] * A[0][2]));
    float I[3][3];
    I[0][0] = +(A[1][1] * A[2][2] - A[2][1] * A[1][2]) * oneOverDet;
    I[1][0] = -(A[1][0] * A[2][2] - A[2][0] * A[1][2]) * oneOverDet;
    I[2][0] = +(A[1][0] * A[2][1] - A[2][0] * A[1][1]) * oneOverDet;
    I[0][1] = -(A[0][1] * A[2][2] - A[2][1] * A[0][2]) * oneOverDet;
    I[1][1] = +(A[0][0] * A[2][2] - A[2][0] * A[0][2]) * oneOverDet;
    I[2][1] = -(A[0][0] * A[2][1] - A[2][0] * A[0][1]) * oneOverDet;
    I[0][2] = +(A[0][1] * A[1][2] - A[1][1] * A[0][2]) * oneOverDet;
    I[1][2] = -(A[0][0] * A[1][2] - A[1][0] * A[0][2]) * oneOverDet;
    I[2][2] = +(A[0][0] * A[1][1] - A[1][0] * A[0][1]) * oneOverDet;
    if (isinf(I[0][0]) || isnan(I[0][0])) {
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int bq = 0; bq < 3; bq++) I[a][bq] = 0.0f;
    }
    const f3 rhs = mk(vel[i]) + Avj;
    out[i] = make_float4(dot3(rhs, f3{I[0][0], I[0][1], I[0][2]}), dot3(rhs, f3{I[1][0], I[1][1], I[1][2]}),
                         dot3(rhs, f3{I[2][0], I[2][1], I[2][2]}), 0.0f);
}

__global__ void __launch_bounds__(kBlock) k_jacobi_relax(uint32_t N, const float4* __restrict__ cand, const float4* __restrict__ cur,
                                                       const float4* __restrict__ prev, float ur, float w0, float w1, float w2,
                                                       float4* __restrict__ o0, float4* __restrict__ o1, float4* __restrict__ o2) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const f3 nw = mk(cand[i]), c = mk(cur[i]), pv = mk(prev[i]);
    const f3 t = ur * (nw - c) + c - pv;
    const f3 a = w0 * t + pv, b = w1 * t + pv, d = w2 * t + pv;
    o0[i] = make_float4(a.x, a.y, a.z, 0.f);
    o1[i] = make_float4(b.x, b.y, b.z, 0.f);
    o2[i] = make_float4(d.x, d.y, d.z, 0.f);
}

// ComputeJacobiError_0/1_kernel (MPSSPHNonPressureUtil.cuh:195-333): per-block partial sums
// of |u_i - a_i sum_j (x_ij.(u_i-u_j)) grad_ij - v0_i| for up to three candidates.
template <bool CUBIC>
__global__ void __launch_bounds__(kBlock) k_jacobi_error(Scenes sc, Nbr nb, const float4* __restrict__ pos,
                                                       const float4* __restrict__ vel, const float* __restrict__ rho,
                                                       const float4* __restrict__ u0, const float4* __restrict__ u1,
                                                       const float4* __restrict__ u2, int ncand, double* __restrict__ partials) {
    __shared__ double lds[kBlock / 64];
    const uint32_t sid = sc.blk_scene[blockIdx.x];
    const StepParams P = sc.P[sid];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t N = P.N;
    const float4* U[3] = {u0, u1, u2};
    for (int q = 0; q < ncand; q++) {
        double e = 0.0;
        if (i < P.end) {
            const float4 xi4 = pos[i];
            const f3 xi = mk(xi4);
            const float h = xi4.w * 4.0f;
            const float invH = 1.0f / h;
            const float onePercentHSq = 0.01f * h * h;
            const f3 ui = mk(U[q][i]);
            f3 Av{0.f, 0.f, 0.f};
            const uint32_t c = nb.cff[i];
            for (uint32_t k = 0; k < c; k++) {
                const uint32_t j = nbr_ff(nb, k, i, N);
                const f3 xij = xi - mk(pos[j]);
                const float dist = len3(xij);
                if (dist < h) {
                    const f3 grad = P.V * Gk<CUBIC>(dist, invH) / ((dist * dist + onePercentHSq) * (dist + kFltEps)) * xij;
                    Av = Av + dot3(xij, ui - mk(U[q][j])) * grad;
                }
            }
            Av = Av * (P.dt * 10.0f * P.mu / rho[i]);
            e = double(len3(ui - Av - mk(vel[i])));
        }
        const double bs = block_sum_d(e, lds);
        if (threadIdx.x == 0) partials[size_t(q) * gridDim.x + blockIdx.x] = bs;
    }
}
__global__ void __launch_bounds__(kBlock) k_fold_partials(const double* __restrict__ partials, uint32_t nblk, int ncand,
                                                        double* __restrict__ out) {
    __shared__ double lds[kBlock / 64];
    for (int q = 0; q < ncand; q++) {
        double s = 0.0;
        for (uint32_t k = threadIdx.x; k < nblk; k += blockDim.x) s += partials[size_t(q) * nblk + k];
        s = block_sum_d(s, lds);
        if (threadIdx.x == 0) out[q] = s;
    }
}

// ----------------------------------------------------------------- advection
// BoundaryCollision_kernel + UpdatePosition_kernel (MPSAdvectUtil.cuh:36-77)
__global__ void __launch_bounds__(kBlock) k_advect(Scenes sc, float4* __restrict__ pos, float4* __restrict__ vel,
                                                 uint32_t* __restrict__ nonfinite, launch::Gate gate) {
    if (shut(gate)) return;
    const uint32_t sid = sc.blk_scene[blockIdx.x];
    const StepParams P = sc.P[sid];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.end) return;
    float4 x4 = pos[i];
    float4 v4 = vel[i];
    float v[3] = {v4.x, v4.y, v4.z};
    const float x[3] = {x4.x, x4.y, x4.z};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float pk = x[k] + v[k] * P.dt;
        if (pk < P.bmin[k] && v[k] < 0.0f) v[k] = (fabsf(v[k]) < 1.0e-4f) ? 0.0f : -v[k] * 0.4f;
        else if (pk > P.bmax[k] && v[k] > 0.0f) v[k] = (fabsf(v[k]) < 1.0e-4f) ? 0.0f : -v[k] * 0.4f;
    }
    v4.x = v[0];
    v4.y = v[1];
    v4.z = v[2];
    x4.x = x[0] + P.dt * v[0];
    x4.y = x[1] + P.dt * v[1];
    x4.z = x[2] + P.dt * v[2];
    vel[i] = v4;
    pos[i] = x4;
    const bool bad = !isfinite(x4.x) || !isfinite(x4.y) || !isfinite(x4.z) || !isfinite(v4.x) || !isfinite(v4.y) ||
                     !isfinite(v4.z);
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(nonfinite, 1u);
}

// One workgroup per scene: st[blockIdx.x] starts a new loop; *active = S.
__global__ void k_solver_reset(SolverDev* stv, uint32_t S, uint32_t* active) {
    reset_record(stv + blockIdx.x, false);
    if (blockIdx.x == 0 && threadIdx.x == 0) *active = S;
}
// The start of a step: the first loop's records, the step's flags, the search's counters.
__global__ void k_step_begin(SolverDev* stv, uint32_t S, uint32_t* active, uint32_t* flags, uint32_t nf, uint32_t* ctr, uint32_t nc) {
    reset_record(stv + blockIdx.x, false);
    if (blockIdx.x) return;
    if (threadIdx.x == 0) *active = S;
    if (threadIdx.x < nf) flags[threadIdx.x] = 0u;
    if (threadIdx.x < nc) ctr[threadIdx.x] = 0u;
}
// Plain streaming copy (16-byte vectors), used only to calibrate byte counters.
__global__ void __launch_bounds__(kBlock) k_calib_copy(const float4* __restrict__ a, float4* __restrict__ b, size_t n) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) b[i] = a[i];
}
// STREAM-style copy for measuring what the memory system gives a copy: one 16-byte vector per
// thread (no grid-stride loop), non-temporal loads and stores. Measured on MI355X: 6.7 TB/s
// against 4.8 TB/s for the grid-stride k_calib_copy above, which stays as the byte-counter
// reference (its loads and stores are ordinary ones, counted like the kernels' own).
typedef float v4f __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(kBlock) k_stream_copy(const float4* __restrict__ a, float4* __restrict__ b, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        __builtin_nontemporal_store(__builtin_nontemporal_load(reinterpret_cast<const v4f*>(a) + i), reinterpret_cast<v4f*>(b) + i);
}
__global__ void k_zero_words(uint32_t* __restrict__ p, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}
// Fluid arrays between slot order and the host's order (element `ref` of w floats): w floats at
// `off` of each slot's `stride`, for elements [first, first + n / w). The staged side is read or
// written contiguously. What bounds an upload or a read is the copy over the host's link and the
// host's page faults: packing, permuting and three staging vectors on the host took 7 ms an upload and
// 5 ms a read of 1 M velocities (now below 2 each; uploading and querying 300 k particles 2.0 -> 0.83 ms).
template <bool OUT>
__global__ void __launch_bounds__(kBlock) k_array_move(uint32_t n, uint32_t first, uint32_t w, uint32_t stride, uint32_t off,
                                                     const uint32_t* __restrict__ inv, float* __restrict__ slots,
                                                     float* __restrict__ staged) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const uint32_t e = t / w;
    float& a = slots[size_t(inv[first + e]) * stride + off + (t - e * w)];
    if (OUT) staged[t] = a;
    else a = staged[t];
}
// New fluid particles [first, first + n) from staged positions, radii and, where given,
// velocities and masses; slot = id = position in the upload.
__global__ void __launch_bounds__(kBlock) k_fluid_upload(uint32_t n, uint32_t first, const float* __restrict__ xyz,
                                                       const float* __restrict__ rad, const float* __restrict__ vxyz,
                                                       const float* __restrict__ mass, float one_mass, float4* __restrict__ pos,
                                                       float4* __restrict__ vel, float4* __restrict__ color,
                                                       uint32_t* __restrict__ perm, uint32_t* __restrict__ inv) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const uint32_t i = first + t;
    pos[i] = make_float4(xyz[3 * size_t(t)], xyz[3 * size_t(t) + 1], xyz[3 * size_t(t) + 2], rad[t]);
    float4 v = make_float4(0.f, 0.f, 0.f, mass ? mass[t] : one_mass);
    if (vxyz) {
        v.x = vxyz[3 * size_t(t)];
        v.y = vxyz[3 * size_t(t) + 1];
        v.z = vxyz[3 * size_t(t) + 2];
    }
    vel[i] = v;
    color[i] = make_float4(0.f, 0.f, 1.f, 1.f);
    perm[i] = i;
    inv[i] = i;
}
// The fluid of a batch of scenes from their staged arrays: slot s of scene q is its particle s - begin;
// the slots from a scene's end to its last workgroup's are padding (perm kEmpty). Packing the records
// on the host and copying 56 bytes per particle took 12 scenes of 370 k particles 2.0 ms.
__global__ void __launch_bounds__(kBlock) k_batch_upload(uint32_t N, const float* __restrict__ staged,
                                                       const launch::SceneSource* __restrict__ src,
                                                       const uint32_t* __restrict__ blk_scene, float4* __restrict__ pos,
                                                       float4* __restrict__ vel, float4* __restrict__ color,
                                                       uint32_t* __restrict__ perm, uint32_t* __restrict__ inv) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= N) return;
    const launch::SceneSource q = src[blk_scene[blockIdx.x]];
    const uint32_t i = s - q.begin;
    float4 p = make_float4(0.f, 0.f, 0.f, 0.f), v = p;
    uint32_t ref = kEmpty;
    if (i < q.nf) {
        const float* a = staged + q.pos + 3 * size_t(i);
        p = make_float4(a[0], a[1], a[2], staged[q.rad + i]);
        if (q.vel != launch::kNoArray) {
            const float* u = staged + q.vel + 3 * size_t(i);
            v = make_float4(u[0], u[1], u[2], 0.f);
        }
        v.w = q.mass != launch::kNoArray ? staged[q.mass + i] : q.one_mass;
        ref = q.ref0 + i;
        inv[ref] = s;
    }
    pos[s] = p;
    vel[s] = v;
    color[s] = make_float4(0.f, 0.f, 1.f, 1.f);
    perm[s] = ref;
}
// Their walls: wall b belongs to the last scene whose walls start at or before b.
__global__ void __launch_bounds__(kBlock) k_batch_upload_walls(uint32_t B, uint32_t S, const float* __restrict__ staged,
                                                             const launch::SceneSource* __restrict__ src, float4* __restrict__ bpos,
                                                             float4* __restrict__ bvel, uint32_t* __restrict__ bscene,
                                                             float4* __restrict__ bcolor, float* __restrict__ bvol,
                                                             uint32_t* __restrict__ bface, float2* __restrict__ bbcc,
                                                             uint32_t* __restrict__ cbb) {
    const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
    if (b >= B) return;
    uint32_t lo = 0, hi = S;  // src[lo].b0 <= b < src[hi].b0
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) / 2u;
        if (src[mid].b0 <= b) lo = mid;
        else hi = mid;
    }
    const launch::SceneSource q = src[lo];
    const uint32_t i = b - q.b0;
    const float* a = staged + q.bpos + 3 * size_t(i);
    bpos[b] = make_float4(a[0], a[1], a[2], staged[q.brad + i]);
    bvel[b] = make_float4(0.f, 0.f, 0.f, q.bmass != launch::kNoArray ? staged[q.bmass + i] : 0.f);
    bscene[b] = lo;
    bcolor[b] = make_float4(0.f, 0.f, 0.f, 0.f);
    bvol[b] = 0.f;
    bface[b] = cbb[b] = 0u;
    bbcc[b] = make_float2(0.f, 0.f);
}
// Derived state of a new fluid: zero; mkey and src kEmpty.
__global__ void __launch_bounds__(kBlock) k_fluid_reset(uint32_t n, float* __restrict__ rho, float* __restrict__ alpha,
                                                      float* __restrict__ kappa, float* __restrict__ delta,
                                                      float* __restrict__ fst, float4* __restrict__ cgb,
                                                      uint32_t* __restrict__ cff, uint32_t* __restrict__ cfb,
                                                      uint32_t* __restrict__ mkey, uint32_t* __restrict__ src) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rho[i] = alpha[i] = kappa[i] = delta[i] = fst[i] = 0.f;
    cgb[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    cff[i] = cfb[i] = 0u;
    mkey[i] = src[i] = kEmpty;
}

// Render feed: positions and radii de-interleaved for the host (replaces the GL buffers
// SPHRenderer binds as SSBOs, MPSSPHRenderer.cpp:22-29).
__global__ void __launch_bounds__(kBlock) k_pack_readback(uint32_t n, const float4* __restrict__ pos, const float4* __restrict__ color,
                                                        const uint32_t* __restrict__ perm, float* __restrict__ xyz,
                                                        float* __restrict__ rad, float* __restrict__ rgba) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t i = perm[s];  // reference index of slot s
    if (i == kEmpty) return;     // padding between scenes
    const float4 p = pos[s];
    if (xyz) {
        xyz[3 * size_t(i)] = p.x;
        xyz[3 * size_t(i) + 1] = p.y;
        xyz[3 * size_t(i) + 2] = p.z;
    }
    if (rad) rad[i] = p.w;
    if (rgba) reinterpret_cast<float4*>(rgba)[i] = color[s];
}

// The same for a renderer that reads double positions and radii (SPHRenderer's shader,
// src/shader/particleShader.vert:3-4): the float values widened exactly.
__global__ void __launch_bounds__(kBlock) k_pack_readback_f64(uint32_t n, const float4* __restrict__ pos,
                                                            const float4* __restrict__ color, const uint32_t* __restrict__ perm,
                                                            double* __restrict__ xyz, double* __restrict__ rad,
                                                            float* __restrict__ rgba) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t i = perm[s];
    if (i == kEmpty) return;
    const float4 p = pos[s];
    if (xyz) {
        xyz[3 * size_t(i)] = double(p.x);
        xyz[3 * size_t(i) + 1] = double(p.y);
        xyz[3 * size_t(i) + 2] = double(p.z);
    }
    if (rad) rad[i] = double(p.w);
    if (rgba) reinterpret_cast<float4*>(rgba)[i] = color[s];
}

}  // namespace dev

// ===================================================================== host launchers
namespace launch {
using namespace dev;
static inline unsigned nb_(size_t n) { return unsigned((n + kBlock - 1) / kBlock); }
// Which form of a list walk a launch takes. With few workgroups the chip is idle and a walk is a
// chain of latencies, which a quad per slot cuts to a quarter; with many, the one-lane form moves
// more bytes per instruction. Measured (us, quad / one lane), dam break: 128 workgroups: A.p 7.5 /
// 8.3, evaluation 8.2 / 11.5, CG setup 16 / 23, density 15 / 26; 349: A.p 17 / 12.5, evaluation
// 11.6 / 14.6, setup 28 / 36, density 25 / 31; 649: A.p 26 / 17, evaluation 18.5 / 17.0. So A.p, the
// pressure apply and the ST factor take a quad up to one workgroup per CU, the evaluation, the
// density and the CG setup up to two.
constexpr unsigned kQuadOnePerCu = 256, kQuadTwoPerCu = 512;
static inline bool quad(const Scenes& sc, unsigned most) { return nb_(sc.N) <= most; }

void boundary_sum(int cubic, const float4* bpos, uint32_t B, const uint32_t* nbb, uint32_t Kbb, const uint32_t* cbb, float* S,
                  hipStream_t s) {
    if (!B) return;
    if (cubic) launch_k(k_boundary_sum<true>, nb_(B), kBlock, 0, s, bpos, B, nbb, Kbb, cbb, S);
    else launch_k(k_boundary_sum<false>, nb_(B), kBlock, 0, s, bpos, B, nbb, Kbb, cbb, S);
}
void boundary_sum_obj(int cubic, const float4* bpos, uint32_t B, const uint32_t* nbb, uint32_t Kbb, const uint32_t* cbb,
                      const uint32_t* obj, float4* S4, hipStream_t s) {
    if (!B) return;
    launch_k(cubic ? k_boundary_sum_obj<true> : k_boundary_sum_obj<false>, nb_(B), kBlock, 0, s, bpos, B, nbb, Kbb, cbb, obj, S4);
}
void boundary_volume_obj(const float4* S4, const uint32_t* obj, uint32_t nobj, float* vol, uint32_t B, int faithful,
                         hipStream_t s) {
    if (B) launch_k(k_boundary_volume_obj, nb_(B), kBlock, 0, s, S4, obj, nobj, vol, B, faithful);
}
void boundary_volume(const float* S, float* vol, uint32_t B, int faithful, hipStream_t s) {
    if (B) launch_k(k_boundary_volume, nb_(B), kBlock, 0, s, S, vol, B, faithful);
}
void density_alpha(int cubic, int flags, const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos, float4* vel,
                   const float4* bpos, const float* bvol, float* rho, float* alpha, float4* color, float* pG_ff,
                   float* pG_fb, hipStream_t s) {
    if (!sc.N) return;
    using K = decltype(&k_density_alpha<false, false, false, 1>);
    static constexpr K tab[8] = {k_density_alpha<false, false, false, 1>, k_density_alpha<false, false, true, 1>,
                                 k_density_alpha<false, true, false, 1>,  k_density_alpha<false, true, true, 1>,
                                 k_density_alpha<true, false, false, 1>,  k_density_alpha<true, false, true, 1>,
                                 k_density_alpha<true, true, false, 1>,   k_density_alpha<true, true, true, 1>};
    const K k = tab[(cubic ? 4 : 0) | (nb.fr ? 2 : 0) | (nb.fbo ? 1 : 0)];
    if (!nb.fr && !nb.fbo && quad(sc, kQuadTwoPerCu)) {
        launch_k(cubic ? k_density_alpha<true, false, false, 4> : k_density_alpha<false, false, false, 4>, nb_(sc.N), 4 * kBlock, 0, s,
                 flags, sc, nb, hl, pos, vel, bpos, bvol, rho, alpha, color, pG_ff, pG_fb);
        return;
    }
    launch_k(k, nb_(sc.N), kBlock, 0, s, flags, sc, nb, hl, pos, vel, bpos, bvol, rho, alpha, color, pG_ff, pG_fb);
}
void pressure_eval(int cubic, int df, const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos, const float4* vel,
                   const float4* bpos, const float* bvol, const float4* bvel, const float* rho, const float* alpha,
                   const float* pG_ff, const float* pG_fb, float* kappa, float* delta, SolverDev* st, double* partials,
                   hipStream_t s) {
    if (!sc.N) return;
    const unsigned g = nb_(sc.N);
    // the ref sums evaluate G_ij themselves (the stored G covers the own and wall lists only);
    // `cubic` matters for the ref instances only
    using K = decltype(&k_pressure_eval<true, false, false, false, 1, false>);
    static constexpr K tab[16] = {
        k_pressure_eval<false, false, false, false, 1, false>, k_pressure_eval<false, false, false, true, 1, false>,
        k_pressure_eval<false, false, false, false, 1, false>, k_pressure_eval<false, false, false, true, 1, false>,
        k_pressure_eval<false, true, false, false, 1, false>,  k_pressure_eval<false, true, false, true, 1, false>,
        k_pressure_eval<false, true, true, false, 1, false>,   k_pressure_eval<false, true, true, true, 1, false>,
        k_pressure_eval<true, false, false, false, 1, false>,  k_pressure_eval<true, false, false, true, 1, false>,
        k_pressure_eval<true, false, false, false, 1, false>,  k_pressure_eval<true, false, false, true, 1, false>,
        k_pressure_eval<true, true, false, false, 1, false>,   k_pressure_eval<true, true, false, true, 1, false>,
        k_pressure_eval<true, true, true, false, 1, false>,    k_pressure_eval<true, true, true, true, 1, false>};
    const K k = tab[(df ? 8 : 0) | (nb.fr ? 4 : 0) | (cubic ? 2 : 0) | (nb.fbo ? 1 : 0)];
    if (!nb.fr && !nb.fbo && quad(sc, kQuadTwoPerCu)) {
        launch_k(df ? k_pressure_eval<true, false, false, false, 4, true> : k_pressure_eval<false, false, false, false, 4, true>, g, 4 * kBlock, 0, s,
                 sc, nb, hl, pos, vel, bpos, bvol, bvel, rho, alpha, pG_ff, pG_fb, kappa, delta, st, partials);
        return;
    }
    if (!nb.fr && !nb.fbo && hl.deep) {
        launch_k(df ? k_pressure_eval<true, false, false, false, 1, true> : k_pressure_eval<false, false, false, false, 1, true>, g, kBlock, 0, s,
                 sc, nb, hl, pos, vel, bpos, bvol, bvel, rho, alpha, pG_ff, pG_fb, kappa, delta, st, partials);
        return;
    }
    launch_k(k, g, kBlock, 0, s, sc, nb, hl, pos, vel, bpos, bvol, bvel, rho, alpha, pG_ff, pG_fb, kappa, delta, st, partials);
}
void fold_pressure(const Scenes& sc, const double* partials, SolverDev* st, uint32_t* active, double tol, uint32_t lmin,
                   int joint, hipStream_t s) {
    if (!sc.N) return;
    if (joint) launch_k(k_fold_pressure_joint, 1, kFoldThreads, 0, s, sc, partials, st, active, tol, lmin);
    else launch_k(k_fold_pressure, sc.S, kFoldThreads, 0, s, sc, partials, st, active, tol, lmin);
}
void pressure_apply(int cubic, const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos, float4* vel, const float4* bpos,
                    const float* bvol, const float* pG_ff, const float* pG_fb, const float* kappa, SolverDev* st,
                    const FoldPressure* fold, hipStream_t s) {
    if (!sc.N) return;
    using K = decltype(&k_pressure_apply<false, false, false, 1, false>);
    static constexpr K tab[8] = {k_pressure_apply<false, false, false, 1, false>, k_pressure_apply<false, false, true, 1, false>,
                                 k_pressure_apply<false, false, false, 1, false>, k_pressure_apply<false, false, true, 1, false>,
                                 k_pressure_apply<true, false, false, 1, false>,  k_pressure_apply<true, false, true, 1, false>,
                                 k_pressure_apply<true, true, false, 1, false>,   k_pressure_apply<true, true, true, 1, false>};
    const K k = tab[(nb.fr ? 4 : 0) | (cubic ? 2 : 0) | (nb.fbo ? 1 : 0)];
    if (!nb.fr && !nb.fbo && quad(sc, kQuadOnePerCu)) {
        launch_k(fold ? k_pressure_apply<false, false, false, 4, true> : k_pressure_apply<false, false, false, 4, false>, nb_(sc.N),
                 4 * kBlock, 0, s, sc, nb, hl, pos, vel, bpos, bvol, pG_ff, pG_fb, kappa, st, fold ? *fold : FoldPressure{});
        return;
    }
    if (fold && !nb.fr)
        launch_k(nb.fbo ? k_pressure_apply<false, false, true, 1, true> : k_pressure_apply<false, false, false, 1, true>, nb_(sc.N),
                 kBlock, 0, s, sc, nb, hl, pos, vel, bpos, bvol, pG_ff, pG_fb, kappa, st, *fold);
    else
        launch_k(k, nb_(sc.N), kBlock, 0, s, sc, nb, hl, pos, vel, bpos, bvol, pG_ff, pG_fb, kappa, st, FoldPressure{});
}
void st_factor(const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos, const float4* vel, const float* pG_ff, float* fst,
               float4* cgx, const LoopStart& ls, hipStream_t s) {
    if (!sc.N) return;
    if (quad(sc, kQuadOnePerCu)) launch_k(k_st_factor<4>, nb_(sc.N), 4 * kBlock, 0, s, sc, nb, hl, pos, vel, pG_ff, fst, cgx, ls);
    else launch_k(k_st_factor<1>, nb_(sc.N), kBlock, 0, s, sc, nb, hl, pos, vel, pG_ff, fst, cgx, ls);
}
void cg_setup(int cubic, const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos, const float4* vel, const float* rho,
              const float* fst, float* ca, float* cb, float* caT, float* cbT, float4* cgb, float* irho, hipStream_t s) {
    if (!sc.N) return;
    const bool q = hl.deep || quad(sc, kQuadTwoPerCu);
    using K = decltype(&k_cg_setup<true, 1, false>);
    static constexpr K tab[8] = {k_cg_setup<false, 1, false>, k_cg_setup<false, 1, true>, k_cg_setup<false, 4, false>,
                                 k_cg_setup<false, 4, true>,  k_cg_setup<true, 1, false>, k_cg_setup<true, 1, true>,
                                 k_cg_setup<true, 4, false>,  k_cg_setup<true, 4, true>};
    launch_k(tab[(cubic ? 4 : 0) | (q ? 2 : 0) | (caT ? 1 : 0)], nb_(sc.N), q ? 4 * kBlock : kBlock, 0, s, sc, nb, hl, pos, vel, rho,
             fst, ca, cb, caT, cbT, cgb, irho);
}
void cg_apply(int mode, const CgOperator& op, const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos,
              const float4* x0, const f3* rr, const f3* pprev, f3* pout, f3* Ap, const float4* b, f3* r, f3* x,
              SolverDev* st, double* partials, const FoldCg* fold, hipStream_t s) {
    if (!sc.N) return;
    const unsigned g = nb_(sc.N);
    const bool q = !op.recompute && quad(sc, kQuadOnePerCu);
    const unsigned threads = q ? 4 * kBlock : kBlock;
    const Streams coef{op.ca, op.cb, op.caT, op.cbT};
#define MPS_CG_APPLY(M, R, C, ...)                                                                                   \
    launch_k(k_cg_apply<M, R, C, ##__VA_ARGS__>, g, threads, 0, s, sc, nb, hl, coef, pos, op.vel, op.rho, op.irho, \
             x0, rr, pprev, pout, Ap, b, r, x, st, partials, fold ? *fold : FoldCg{})
    if (op.caT) {  // transposed (deep staging: its registers allow four workgroups per CU anyway)
        if (q) {
            if (mode == 0) MPS_CG_APPLY(0, false, true, true, 4, false, true);
            else if (fold) MPS_CG_APPLY(1, false, true, true, 4, true, true);
            else MPS_CG_APPLY(1, false, true, true, 4, false, true);
        } else {
            if (mode == 0) MPS_CG_APPLY(0, false, true, true, 1, false, true);
            else if (fold && hl.keep) MPS_CG_APPLY(1, false, true, true, 1, true, true, true);
            else if (fold) MPS_CG_APPLY(1, false, true, true, 1, true, true);
            else if (hl.keep) MPS_CG_APPLY(1, false, true, true, 1, false, true, true);
            else MPS_CG_APPLY(1, false, true, true, 1, false, true);
        }
    } else if (q) {
        if (mode == 0) MPS_CG_APPLY(0, false, true, true, 4);
        else if (fold) MPS_CG_APPLY(1, false, true, true, 4, true);
        else MPS_CG_APPLY(1, false, true, true, 4);
    } else if (!op.recompute && op.deep) {
        if (mode == 0) MPS_CG_APPLY(0, false, true, true);
        else if (fold && hl.keep) MPS_CG_APPLY(1, false, true, true, 1, true, false, true);
        else if (fold) MPS_CG_APPLY(1, false, true, true, 1, true);
        else if (hl.keep) MPS_CG_APPLY(1, false, true, true, 1, false, false, true);
        else MPS_CG_APPLY(1, false, true, true);
    } else if (!op.recompute) {
        if (mode == 0) MPS_CG_APPLY(0, false, true);
        else if (fold && hl.keep) MPS_CG_APPLY(1, false, true, false, 1, true, false, true);
        else if (fold) MPS_CG_APPLY(1, false, true, false, 1, true);
        else if (hl.keep) MPS_CG_APPLY(1, false, true, false, 1, false, false, true);
        else MPS_CG_APPLY(1, false, true);
    } else if (op.cubic) {
        if (mode == 0) MPS_CG_APPLY(0, true, true);
        else MPS_CG_APPLY(1, true, true);
    } else {
        if (mode == 0) MPS_CG_APPLY(0, true, false);
        else MPS_CG_APPLY(1, true, false);
    }
#undef MPS_CG_APPLY
}
void cg_apply_fold(const CgOperator& op, const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos, const f3* rr,
                   const f3* pprev, f3* pout, f3* Ap, SolverDev* st, double* partials, uint32_t* arrive, hipStream_t s) {
    if (!sc.N) return;
    const unsigned g = nb_(sc.N);
    const Streams coef{op.ca, op.cb};
#define MPS_CG_APPLY_FOLD(R, C)                                                                                    \
    launch_k(k_cg_apply_fold<R, C>, g, kBlock, 0, s, sc, nb, hl, coef, pos, op.vel, op.rho, op.irho, rr, pprev, \
             pout, Ap, st, partials, arrive)
    if (!op.recompute) MPS_CG_APPLY_FOLD(false, true);
    else if (op.cubic) MPS_CG_APPLY_FOLD(true, true);
    else MPS_CG_APPLY_FOLD(true, false);
#undef MPS_CG_APPLY_FOLD
}
void cg_update3_fold(const Scenes& sc, f3* x, f3* r, const f3* p, const f3* Ap, SolverDev* st, double* partials,
                     uint32_t* active, double tol, uint32_t* arrive, hipStream_t s) {
    if (sc.N) launch_k(k_cg_update3_fold, nb_(sc.N), kBlock, 0, s, sc, x, r, p, Ap, st, partials, active, tol, arrive);
}
static const void* persistent_fn(const CgOperator& op, int coherent) {
    if (coherent) {
        if (!op.recompute) return reinterpret_cast<const void*>(k_cg_persistent<false, true, true>);
        return op.cubic ? reinterpret_cast<const void*>(k_cg_persistent<true, true, true>)
                        : reinterpret_cast<const void*>(k_cg_persistent<true, false, true>);
    }
    if (!op.recompute) return reinterpret_cast<const void*>(k_cg_persistent<false, true, false>);
    return op.cubic ? reinterpret_cast<const void*>(k_cg_persistent<true, true, false>)
                    : reinterpret_cast<const void*>(k_cg_persistent<true, false, false>);
}
uint32_t cg_persistent_capacity(const CgOperator& op, int coherent) {
    int dev = 0, per_cu = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, persistent_fn(op, coherent), kBlock, 0) != hipSuccess) return 0;
    return uint32_t(per_cu) * uint32_t(prop.multiProcessorCount);
}
void cg_persistent(const CgOperator& op, int coherent, const Scenes& sc, const Nbr& nb, const Halo& hl, const float4* pos,
                   f3* r, f3* pbuf0, f3* pbuf1, f3* Ap, f3* x, SolverDev* st, uint32_t* active, double* partA,
                   double* partB, GridSync* gs, uint32_t cap, double tol, uint32_t spin, hipStream_t s) {
    if (!sc.N) return;
    const uint32_t nblk = nb_(sc.N);
    Streams coef{op.ca, op.cb};
    void* args[] = {const_cast<Scenes*>(&sc), const_cast<Nbr*>(&nb), const_cast<Halo*>(&hl), &coef,
                    const_cast<float4**>(&pos), const_cast<float4**>(&op.vel),
                    const_cast<float**>(&op.rho), const_cast<float**>(&op.irho), &r, &pbuf0, &pbuf1, &Ap, &x, &st, &active,
                    &partA, &partB, &gs, &cap, &tol, &spin};
    const hipError_t rc = hipLaunchCooperativeKernel(persistent_fn(op, coherent), dim3(nblk), dim3(kBlock), args, 0, s);
    if (rc != hipSuccess) throw LaunchError{rc};
}
void fold_cg(int mode, const Scenes& sc, const double* partials, SolverDev* st, uint32_t* active, double tol, hipStream_t s) {
    if (!sc.N) return;
    if (mode == 0) launch_k(k_fold_cg<0>, sc.S, kFoldThreads, 0, s, sc, partials, st, active, tol);
    else if (mode == 1) launch_k(k_fold_cg<1>, sc.S, kFoldThreads, 0, s, sc, partials, st, active, tol);
    else launch_k(k_fold_cg<2>, sc.S, kFoldThreads, 0, s, sc, partials, st, active, tol);
}
void cg_update3(const Scenes& sc, f3* x, f3* r, const f3* p, const f3* Ap, SolverDev* st, const double* pAp, double* partials,
                hipStream_t s) {
    if (sc.N) launch_k(pAp ? k_cg_update3<true> : k_cg_update3<false>, nb_(sc.N), kBlock, 0, s, sc, x, r, p, Ap, st, pAp, partials);
}
// Every consumer workgroup reads all partial sums of its scene, so the work grows with the square of
// the workgroups. Whole passes (fold launches -> folds in the consumers): 128 workgroups 15.5 ->
// 14.1 ms, 1006 24.5 -> 22.8, 2051 33.8 -> 34.3, 3907 65.7 -> 68.4 (there A.p 73.0 -> 79.8 us and
// the update 11.4 -> 15.5, against two fold launches of 4.0). The line is on the whole grid's
// workgroups: in a batch each folds its own scene's sums only, but each pays the round trip (64 scenes,
// 17.5 k workgroups, scenes of up to 1024: 22.3 ms per step with fold launches, 22.7 without).
bool fold_in_consumer(uint32_t blocks) { return blocks <= 1536; }
void copy_vel_out3(const Scenes& sc, const f3* x, float4* vel, const Gate& gate, const LoopStart& ls, hipStream_t s) {
    if (sc.N) launch_k(k_copy_vel_out3, nb_(sc.N), kBlock, 0, s, sc, x, vel, gate, ls);
}
void copy_vel_out(const Scenes& sc, const float4* x, float4* vel, hipStream_t s) {
    if (sc.N) launch_k(k_copy_vel_out, nb_(sc.N), kBlock, 0, s, sc, x, vel);
}
void jacobi_candidate(int cubic, const Scenes& sc, const Nbr& nb, const float4* pos, const float4* vel,
                      const float* rho, const float4* u, float4* out, hipStream_t s) {
    if (!sc.N) return;
    if (cubic) launch_k(k_jacobi_candidate<true>, nb_(sc.N), kBlock, 0, s, sc, nb, pos, vel, rho, u, out);
    else launch_k(k_jacobi_candidate<false>, nb_(sc.N), kBlock, 0, s, sc, nb, pos, vel, rho, u, out);
}
void jacobi_relax(uint32_t N, const float4* cand, const float4* cur, const float4* prev, float ur, const float* w3,
                  float4* o0, float4* o1, float4* o2, hipStream_t s) {
    if (N) launch_k(k_jacobi_relax, nb_(N), kBlock, 0, s, N, cand, cur, prev, ur, w3[0], w3[1], w3[2], o0, o1, o2);
}
void jacobi_error(int cubic, const Scenes& sc, const Nbr& nb, const float4* pos, const float4* vel,
                  const float* rho, const float4* u0, const float4* u1, const float4* u2, int ncand, double* partials,
                  double* err3, hipStream_t s) {
    if (!sc.N) return;
    const unsigned g = nb_(sc.N);
    if (cubic) launch_k(k_jacobi_error<true>, g, kBlock, 0, s, sc, nb, pos, vel, rho, u0, u1, u2, ncand, partials);
    else launch_k(k_jacobi_error<false>, g, kBlock, 0, s, sc, nb, pos, vel, rho, u0, u1, u2, ncand, partials);
    launch_k(k_fold_partials, 1, kBlock, 0, s, partials, g, ncand, err3);
}
void advect(const Scenes& sc, float4* pos, float4* vel, uint32_t* nonfinite, const Gate& gate, hipStream_t s) {
    if (sc.N) launch_k(k_advect, nb_(sc.N), kBlock, 0, s, sc, pos, vel, nonfinite, gate);
}
void step_begin(SolverDev* st, uint32_t S, uint32_t* active, uint32_t* flags, uint32_t nf, NbrCounters* ctr, hipStream_t s) {
    static_assert(sizeof(NbrCounters) / 4 <= kBlock, "one word per thread");
    launch_k(k_step_begin, S, kBlock, 0, s, st, S, active, flags, nf, reinterpret_cast<uint32_t*>(ctr), sizeof(NbrCounters) / 4);
}
void solver_reset(SolverDev* st, uint32_t S, uint32_t* active, hipStream_t s) {
    if (S) launch_k(k_solver_reset, S, kBlock, 0, s, st, S, active);
}
void calib_copy(const float4* a, float4* b, size_t n, hipStream_t s) {
    if (n) launch_k(k_calib_copy, 4096, kBlock, 0, s, a, b, n);
}
void stream_copy(const float4* a, float4* b, size_t n, hipStream_t s) {
    if (n) launch_k(k_stream_copy, unsigned((n + kBlock - 1) / kBlock), kBlock, 0, s, a, b, n);
}
void zero_words(uint32_t* p, size_t n, hipStream_t s) {
    if (n) launch_k(k_zero_words, unsigned((n + kBlock - 1) / kBlock), kBlock, 0, s, p, n);
}
void array_move(bool out, uint32_t n, uint32_t first, uint32_t w, uint32_t stride, uint32_t off, const uint32_t* inv, float* slots,
                float* staged, hipStream_t s) {
    if (!n) return;
    if (out) launch_k(k_array_move<true>, nb_(size_t(n) * w), kBlock, 0, s, n * w, first, w, stride, off, inv, slots, staged);
    else launch_k(k_array_move<false>, nb_(size_t(n) * w), kBlock, 0, s, n * w, first, w, stride, off, inv, slots, staged);
}
void fluid_upload(uint32_t n, uint32_t first, const float* xyz, const float* rad, const float* vxyz, const float* mass,
                  float one_mass, float4* pos, float4* vel, float4* color, uint32_t* perm, uint32_t* inv, hipStream_t s) {
    if (n) launch_k(k_fluid_upload, nb_(n), kBlock, 0, s, n, first, xyz, rad, vxyz, mass, one_mass, pos, vel, color, perm, inv);
}
void batch_upload(uint32_t N, const float* staged, const SceneSource* src, const uint32_t* blk_scene, float4* pos, float4* vel,
                  float4* color, uint32_t* perm, uint32_t* inv, hipStream_t s) {
    if (N) launch_k(k_batch_upload, nb_(N), kBlock, 0, s, N, staged, src, blk_scene, pos, vel, color, perm, inv);
}
void batch_upload_walls(uint32_t B, uint32_t S, const float* staged, const SceneSource* src, float4* bpos, float4* bvel,
                        uint32_t* bscene, float4* bcolor, float* bvol, uint32_t* bface, float2* bbcc, uint32_t* cbb, hipStream_t s) {
    if (B) launch_k(k_batch_upload_walls, nb_(B), kBlock, 0, s, B, S, staged, src, bpos, bvel, bscene, bcolor, bvol, bface, bbcc, cbb);
}
void fluid_reset(uint32_t n, float* rho, float* alpha, float* kappa, float* delta, float* fst, float4* cgb, uint32_t* cff,
                 uint32_t* cfb, uint32_t* mkey, uint32_t* src, hipStream_t s) {
    if (n) launch_k(k_fluid_reset, nb_(n), kBlock, 0, s, n, rho, alpha, kappa, delta, fst, cgb, cff, cfb, mkey, src);
}
void pack_readback(uint32_t n, const float4* pos, const float4* color, const uint32_t* perm, float* xyz, float* rad,
                   float* rgba, hipStream_t s) {
    if (n) launch_k(k_pack_readback, nb_(n), kBlock, 0, s, n, pos, color, perm, xyz, rad, rgba);
}
void pack_readback_f64(uint32_t n, const float4* pos, const float4* color, const uint32_t* perm, double* xyz, double* rad,
                       float* rgba, hipStream_t s) {
    if (n) launch_k(k_pack_readback_f64, nb_(n), kBlock, 0, s, n, pos, color, perm, xyz, rad, rgba);
}

}  // namespace launch
}  // namespace mps
