// One very large world on the whole device: the same step as the per-world
// kernel (Step(AabbTreeWorld&, const StepConf&), AabbTreeWorld.cpp:2144-2219,
// doToi == false) but every phase spread over the GPU, with two changes of
// method:
//
// * Broadphase: every moved proxy's fat AABB against every proxy's, a thread
//   per proxy and the moved ones in tiles (k_pairs_find).  It answers the same
//   queries as the reference's DynamicTree (FindContacts,
//   AabbTreeWorld.cpp:709-751): for every moved proxy, all proxies of other
//   bodies whose fat AABBs overlap it.  The pair sets are identical; new
//   contacts are appended in proxy order, those of one proxy in Morton order,
//   instead of key order.  The linear BVH below (Morton codes, a
//   workgroup-wide LSD radix sort, Karras' radix-tree construction, bottom-up
//   bounds refit, escape indices for a stackless traversal) serves the pair
//   finder as a call of its own, whose proxies have no bound in number.
// * Solver: graph-coloured Gauss-Seidel.  Touching contacts are coloured so no
//   two contacts of a colour share a dynamic body; each colour is solved in
//   parallel, colours in sequence, with the reference's per-constraint
//   arithmetic (warm start, SolveVelocityConstraint with the block solver,
//   SolvePositionConstraint).  All awake dynamic bodies form one system (no
//   island split, no sleeping).  Results are not the reference's bits (the
//   sweep order differs); they are judged by penetration, momentum and
//   stacking behaviour.
//
// Order-sensitive bookkeeping (stable contact compaction, the touching list,
// the colour order, the order of new contacts) computes places from counts and
// ranks, never from the order in which workgroups arrive, so every run is
// deterministic.
#include <mutex>

#include "../../include/playrho_amd.h"
#include "big_world.hpp"
#include "step_device.hpp"

namespace prxd {

using prx::BigState;

constexpr int kBlock = prx::kBigBlock;  // threads of the single-workgroup kernels
constexpr int kGrid = 256;              // threads per workgroup of the grid-wide kernels
constexpr int kSweepBlocks = 64;        // workgroups of a colour sweep launch (16,384 threads)
constexpr int kSmallBlock = 1024;       // threads of the one-workgroup solve and sweeps
// The most bodies of a world that one workgroup solves (k_big_solve_small); its
// state would fit LDS up to 4096.  A step by one workgroup and by the grid's
// launches, boxes of settled drops: 1000 bodies 451 and 534 us, 1500: 530 and
// 579, 2000: 608 and 603, 2500: 676 and 616, 4000: 935 and 667.  While few have
// landed the one workgroup stays ahead (4000 bodies: 338 and 463 us at step 20,
// 605 and 637 at 140, 957 and 742 at 230); the settled state decides, since that
// is where a world spends its time.
constexpr int kSmallBodies = 2048;
constexpr int kBigToiPasses = 2;  // time-of-impact passes per step against static shapes
// Bound on tree depth for the parent walks (a Karras tree over 30-bit codes
// with index tie-breaks is at most 30 + 32 deep).
constexpr int kMaxDepth = 96;

__device__ __forceinline__ WorldCtx big_ctx(const DeviceState& d) {
    const WorldHeader& H = d.hdr[0];
    WorldCtx x;
    x.w = 0;
    x.bo = 0;
    x.nb = H.nbodies;
    x.po = 0;
    x.np = H.nproxies;
    x.co = 0;
    x.cap = H.contact_cap;
    x.jo = 0;
    x.nj = 0;
    x.eo = 0;
    x.ecap = 0;
    x.lane = int(threadIdx.x) & (kWave - 1);
    return x;
}

// Exclusive prefix sum over the workgroup (kBlock threads); lds holds
// kBlock / 64 + 1 ints.  Returns the thread's prefix; total receives the sum.
__device__ __forceinline__ int block_exclusive_scan(int v, int* lds, int& total) {
    const int lane = int(threadIdx.x) & (kWave - 1), wave = int(threadIdx.x) >> 6;
    const int incl = wave_incl_scan(v, lane);
    if (lane == kWave - 1) lds[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int w = 0; w < kBlock / kWave; ++w) {
            const int t = lds[w];
            lds[w] = run;
            run += t;
        }
        lds[kBlock / kWave] = run;
    }
    __syncthreads();
    const int r = lds[wave] + incl - v;
    total = lds[kBlock / kWave];
    __syncthreads();
    return r;
}

__device__ __forceinline__ float block_reduce_max(float v, float* lds) {
    for (int o = 32; o > 0; o >>= 1) v = fmax_std(v, __shfl_xor(v, o));
    const int lane = int(threadIdx.x) & (kWave - 1), wave = int(threadIdx.x) >> 6;
    if (lane == 0) lds[wave] = v;
    __syncthreads();
    float r = lds[0];
    for (int w = 1; w < kBlock / kWave; ++w) r = fmax_std(r, lds[w]);
    __syncthreads();
    return r;
}

__device__ __forceinline__ float block_reduce_min(float v, float* lds) {
    for (int o = 32; o > 0; o >>= 1) v = fmin_std(v, __shfl_xor(v, o));
    const int lane = int(threadIdx.x) & (kWave - 1), wave = int(threadIdx.x) >> 6;
    if (lane == 0) lds[wave] = v;
    __syncthreads();
    float r = lds[0];
    for (int w = 1; w < kBlock / kWave; ++w) r = fmin_std(r, lds[w]);
    __syncthreads();
    return r;
}

// ---------------------------------------------------------------------------
// Pre-phase.

// Sum of sums[0..n) over the workgroup (kGrid threads); lds holds kGrid / 64 ints.
__device__ __forceinline__ int block_sum_of(const int* sums, int n, int* lds) {
    int v = 0;
    for (int j = int(threadIdx.x); j < n; j += kGrid) v += sums[j];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    const int lane = int(threadIdx.x) & (kWave - 1), wave = int(threadIdx.x) >> 6;
    __syncthreads();
    if (lane == 0) lds[wave] = v;
    __syncthreads();
    int r = 0;
#pragma unroll
    for (int w = 0; w < kGrid / kWave; ++w) r += lds[w];
    return r;
}

// Rank of a flagged thread among the workgroup's flagged threads (kGrid
// threads, lds as above); total receives their count.
__device__ __forceinline__ int block_rank(bool flag, int* lds, int& total) {
    const unsigned long long m = __ballot(flag);
    const int lane = int(threadIdx.x) & (kWave - 1), wave = int(threadIdx.x) >> 6;
    __syncthreads();
    if (lane == 0) lds[wave] = __popcll(m);
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < kGrid / kWave; ++w) {
        before += (w < wave) ? lds[w] : 0;
        total += lds[w];
    }
    return before + __popcll(m & lanes_below(lane));
}

// Order-preserving integer images of floats, for atomic minima and maxima.
__device__ __forceinline__ int sep_key(float f) {
    const int bits = __float_as_int(f);
    return bits >= 0 ? bits : (bits ^ 0x7fffffff);
}
__device__ __forceinline__ float sep_of_key(int key) { return __int_as_float(key >= 0 ? key : (key ^ 0x7fffffff)); }

__device__ __forceinline__ int* find_state(const BigState& g, int slot) { return g.find + slot * prx::kFindWords; }

__device__ __forceinline__ std::uint32_t hash_slot(std::uint64_t key, int mask) {
    const std::uint64_t h = key * 0x9e3779b97f4a7c15ull;
    return std::uint32_t(h >> 32) & std::uint32_t(mask);
}

// Entries of the set of existing contact keys carry the step they were
// inserted in, so an entry of an earlier step reads as free and the set needs
// no clearing: (step << 32) | proxy of the lower key << 16 | the other proxy.
__device__ __forceinline__ unsigned long long hash_entry(const BigState& g, int pa, int pb) {
    return (static_cast<unsigned long long>(unsigned(g.counters[prx::kBigStep])) << 32) | (unsigned(pa) << 16) |
           unsigned(pb);
}
__device__ __forceinline__ void hash_insert(const BigState& g, int pa, int pb) {
    const unsigned long long want = hash_entry(g, pa, pb);
    std::uint32_t h = hash_slot(want & 0xffffffffull, g.hashMask);
    auto* table = reinterpret_cast<unsigned long long*>(g.hash);
    for (int probe = 0; probe <= g.hashMask; ++probe) {
        unsigned long long seen = __hip_atomic_load(table + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while ((seen >> 32) != (want >> 32)) {
            const unsigned long long prev = atomicCAS(table + h, seen, want);
            if (prev == seen) return;
            seen = prev;
        }
        if (seen == want) return;
        h = (h + 1u) & std::uint32_t(g.hashMask);
    }
}
__device__ __forceinline__ bool hash_has(const BigState& g, int pa, int pb) {
    const unsigned long long want = hash_entry(g, pa, pb);
    std::uint32_t h = hash_slot(want & 0xffffffffull, g.hashMask);
    for (int probe = 0; probe <= g.hashMask; ++probe) {
        const unsigned long long v = g.hash[h];
        if (v == want) return true;
        if ((v >> 32) != (want >> 32)) return false;
        h = (h + 1u) & std::uint32_t(g.hashMask);
    }
    return false;
}

// DestroyContacts (AabbTreeWorld.cpp:2290-2331) removes the contacts whose
// fat AABBs no longer overlap by a stable compaction in three grid-wide
// launches: k_big_mark counts the kept contacts of each workgroup's range,
// k_big_gather places each kept record behind the kept ones before it (into
// scratch, since its slot may hold a record not read yet) and k_big_contacts
// copies them back.  Contacts before the first destroyed one stay where they
// are and are not copied; in a settled world few or none move.  One 1024-thread
// workgroup walking the list took 222 us a step at 73,000 contacts; the marks
// take 8 us and the gathering, with the key set's insertion, 15.
__device__ __forceinline__ bool still_overlaps(const DeviceState& d, int i) {
    const int2 pr = d.c_prox[i];
    return overlap(d.paabb[pr.x], d.paabb[pr.y]);
}

// CreateProxies (AabbTreeWorld.cpp:557-579; a pending proxy has no contact),
// the first third of DestroyContacts, and the step's counters cleared.
__global__ __launch_bounds__(kGrid) void k_big_mark(DeviceState d, BigState g, StepParams c) {
    __shared__ int s_cnt[kGrid / kWave];
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i == 0) {
        for (int k = 0; k < prx::kStats; ++k) d.hdr[0].stats[k] = 0u;
        d.hdr[0].stats[prx::kStRegMinSeparation] = 0x7f800000u;
        d.hdr[0].stats[prx::kStToiMinSeparation] = 0x7f800000u;
        g.counters[prx::kBigStep] += 1;
    }
    if (i < prx::kFindSlots * prx::kFindWords) {
        const int w = i % prx::kFindWords;
        g.find[i] = (w == prx::kFindLoX || w == prx::kFindLoY)   ? sep_key(__builtin_inff())
                    : (w == prx::kFindHiX || w == prx::kFindHiY) ? sep_key(-__builtin_inff())
                                                                 : 0;
    }
    if (i < d.hdr[0].nproxies && (d.pflags[i] & prx::kProxyPending)) {
        const int gb = d.pbody[i];
        d.paabb[i] = proxy_aabb(shape_proxy(d, d.pshape[i]), body_xf0(d, gb), body_xf1(d, gb), c, true);
        d.pflags[i] = prx::kProxyMoved;
    }
    const int nc = d.hdr[0].ncontacts;
    if (int(blockIdx.x) * kGrid >= nc) return;
    bool keep = false;
    if (i < nc) {
        keep = still_overlaps(d, i);
        if (!keep) {
            atomicMin(&g.counters[prx::kBigFirstGone], i);
            const std::uint32_t mh = d.m_hdr[i].x;
            if (((mh >> 8) & 0xffu) > 0 && !(d.c_flags[i] & prx::kSensor)) {
                const int2 bd = d.c_body[i];
                body_set_awake(d, bd.x);
                body_set_awake(d, bd.y);
            }
        }
    }
    int tot = 0;
    (void)block_rank(keep, s_cnt, tot);
    if (threadIdx.x == 0) g.blockSum[blockIdx.x] = tot;
}

constexpr int kMoveStride = 7;  // float4 of a contact record in the compaction's scratch (s_vc2)
static_assert(kMoveStride <= prx::kQuadVc, "s_vc2 holds kQuadVc float4 a contact slot");

__global__ __launch_bounds__(kGrid) void k_big_gather(DeviceState d, BigState g) {
    __shared__ int s_cnt[kGrid / kWave];
    const int nc = d.hdr[0].ncontacts;
    const int blk = int(blockIdx.x);
    if (blk * kGrid >= nc && blk > 0) return;
    const int i = blk * kGrid + int(threadIdx.x);
    const bool keep = i < nc && still_overlaps(d, i);
    const int before = block_sum_of(g.blockSum, blk, s_cnt);
    int tot = 0;
    const int dst = before + block_rank(keep, s_cnt, tot);
    if ((blk + 1) * kGrid >= nc && threadIdx.x == 0) {
        g.counters[prx::kBigKept] = before + tot;
        d.hdr[0].stats[prx::kStPreDestroyed] = std::uint32_t(nc - before - tot);
    }
    if (!keep) return;
    const int2 pr = d.c_prox[i];
    hash_insert(g, pr.x, pr.y);
    if (dst == i) return;
    const int2 bd = d.c_body[i], sh = d.c_shape[i];
    float4* o = d.s_vc2 + std::size_t(dst) * kMoveStride;
    o[0] = float4{__int_as_float(pr.x), __int_as_float(pr.y), __int_as_float(bd.x), __int_as_float(bd.y)};
    o[1] = float4{__int_as_float(sh.x), __int_as_float(sh.y), __uint_as_float(d.c_id[i]), __uint_as_float(d.c_flags[i])};
    o[2] = d.c_mat[i];
    const uint4 mh = d.m_hdr[i];
    o[3] = float4{__uint_as_float(mh.x), __uint_as_float(mh.y), __uint_as_float(mh.z), __uint_as_float(mh.w)};
    o[4] = d.m_geo[i];
    o[5] = d.m_p0[i];
    o[6] = d.m_p1[i];
}

// UpdateContacts (AabbTreeWorld.cpp:2333-2421): narrowphase of the contacts
// flagged or with a body whose position changed (:1546-1551), one thread per
// contact; the same threads list the moved proxies and reduce the bounds of
// the AABB centres for the pair search that follows (slot: which of the
// step's searches; slot 0 first completes the compaction of k_big_gather).
__global__ __launch_bounds__(kGrid) void k_big_contacts(DeviceState d, BigState g, StepParams c, int slot) {
    __shared__ int s_cnt[kGrid / kWave];
    __shared__ int s_base;
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    const int nc = slot == 0 ? g.counters[prx::kBigKept] : d.hdr[0].ncontacts;
    const int np = d.hdr[0].nproxies;
    int* const fs = find_state(g, slot);
    if (slot == 0 && i == 0) d.hdr[0].ncontacts = nc;
    if (int(blockIdx.x) * kGrid < np) {
        const bool moved = i < np && (d.pflags[i] & prx::kProxyMoved) != 0;
        int tot = 0;
        const int r = block_rank(moved, s_cnt, tot);
        if (threadIdx.x == 0) s_base = tot ? atomicAdd(&fs[prx::kFindMoved], tot) : 0;
        __syncthreads();
        if (moved) g.moved[s_base + r] = i;
        float lox = __builtin_inff(), loy = __builtin_inff(), hix = -__builtin_inff(), hiy = -__builtin_inff();
        if (i < np) {
            const float4 a = d.paabb[i];
            const float cx = (a.x + a.z) * 0.5f, cy = (a.y + a.w) * 0.5f;
            lox = fmin_std(lox, cx);
            loy = fmin_std(loy, cy);
            hix = fmax_std(hix, cx);
            hiy = fmax_std(hiy, cy);
        }
        for (int o = 32; o > 0; o >>= 1) {
            lox = fmin_std(lox, __shfl_xor(lox, o));
            loy = fmin_std(loy, __shfl_xor(loy, o));
            hix = fmax_std(hix, __shfl_xor(hix, o));
            hiy = fmax_std(hiy, __shfl_xor(hiy, o));
        }
        if ((threadIdx.x & (kWave - 1)) == 0) {
            atomicMin(&fs[prx::kFindLoX], sep_key(lox));
            atomicMin(&fs[prx::kFindLoY], sep_key(loy));
            atomicMax(&fs[prx::kFindHiX], sep_key(hix));
            atomicMax(&fs[prx::kFindHiY], sep_key(hiy));
        }
    }
    if (i >= nc) return;
    if (slot == 0 && i >= g.counters[prx::kBigFirstGone]) {
        const float4* o = d.s_vc2 + std::size_t(i) * kMoveStride;
        const float4 a = o[0], b = o[1], h = o[3];
        d.c_prox[i] = int2{__float_as_int(a.x), __float_as_int(a.y)};
        d.c_body[i] = int2{__float_as_int(a.z), __float_as_int(a.w)};
        d.c_shape[i] = int2{__float_as_int(b.x), __float_as_int(b.y)};
        d.c_id[i] = __float_as_uint(b.z);
        d.c_flags[i] = __float_as_uint(b.w);
        d.c_mat[i] = o[2];
        d.m_hdr[i] = uint4{__float_as_uint(h.x), __float_as_uint(h.y), __float_as_uint(h.z), __float_as_uint(h.w)};
        d.m_geo[i] = o[4];
        d.m_p0[i] = o[5];
        d.m_p1[i] = o[6];
    }
    bool update = (d.c_flags[i] & prx::kNeedsUpdating) != 0;
    if (slot != 0) {
        const int2 bd = d.c_body[i];
        update = update || ((d.bflags[bd.x] | d.bflags[bd.y]) & 0x100u) != 0;
    }
    if (update) {
        update_contact(d, 0, i, c);
        if (slot == 0) {
            const unsigned long long m = __ballot(1);
            if (__popcll(m & lanes_below(int(threadIdx.x) & (kWave - 1))) == 0)
                atomicAdd(&d.hdr[0].stats[prx::kStPreUpdated], std::uint32_t(__popcll(m)));
        }
    }
}

// Grid position of a proxy's AABB centre in the bounds of all centres, as a
// 30-bit Morton code.
__device__ __forceinline__ std::uint32_t spread15(std::uint32_t v) {
    v &= 0x7fffu;
    v = (v | (v << 8)) & 0x00ff00ffu;
    v = (v | (v << 4)) & 0x0f0f0f0fu;
    v = (v | (v << 2)) & 0x33333333u;
    v = (v | (v << 1)) & 0x55555555u;
    return v;
}
__device__ __forceinline__ std::uint32_t morton_code(float4 b, float4 a) {
    const float cx = (a.x + a.z) * 0.5f, cy = (a.y + a.w) * 0.5f;
    const float sx = (b.z > b.x) ? 32767.0f / (b.z - b.x) : 0.0f;
    const float sy = (b.w > b.y) ? 32767.0f / (b.w - b.y) : 0.0f;
    const float fx = fmin_std(fmax_std((cx - b.x) * sx, 0.0f), 32767.0f);
    const float fy = fmin_std(fmax_std((cy - b.y) * sy, 0.0f), 32767.0f);
    return (spread15(std::uint32_t(fx)) << 1) | spread15(std::uint32_t(fy));
}

// FindContacts (AabbTreeWorld.cpp:709-751): every proxy r against every moved
// proxy p, with the AddContacts filters (AabbTreeWorld.cpp:2424-2470: existing
// key, neither body accelerable, shape filters) applied to the overlapping
// pairs.  A pair of two moved proxies counts once, for the lower index.  The
// pairs left are listed as (p, Morton code of r, r), the order in which
// k_pairs_create appends them.
//
// A thread holds one proxy r; the moved ones pass in tiles of 64 through LDS.
// The test is four comparisons, so 20,000 proxies against all of themselves
// cost less than the tree that the search once built for each call (sort
// 169 us and refit 133 us in one workgroup's and one climb's latency at 20,000
// proxies, whatever had moved): 5 us with nothing moved, 25 on average over a
// settled world's searches and 0.11 ms with all moved.
constexpr int kMovedTile = 64;
constexpr int kMovedSplit = 16;  // grid.y: tiles in flight per proxy
__global__ __launch_bounds__(kGrid) void k_pairs_find(DeviceState d, BigState g, int slot) {
    __shared__ float4 s_box[kMovedTile];
    __shared__ int s_p[kMovedTile];
    int* const fs = find_state(g, slot);
    const int r = int(blockIdx.x * blockDim.x + threadIdx.x);
    // Position-changed marks and the first destroyed contact have been read
    // by k_big_contacts.
    if (slot == 0 && r == 0 && blockIdx.y == 0) g.counters[prx::kBigFirstGone] = 0x7fffffff;
    if (blockIdx.y == 0 && r < d.hdr[0].nbodies) d.bflags[r] &= ~0x100u;
    const int moved = fs[prx::kFindMoved];
    const int np = d.hdr[0].nproxies;
    if (int(blockIdx.y) * kMovedTile >= moved || int(blockIdx.x) * kGrid >= np) return;
    const bool valid = r < np;
    const float4 box = valid ? d.paabb[r] : float4{0, 0, 0, 0};
    const bool movedR = valid && (d.pflags[r] & prx::kProxyMoved) != 0;
    const int bodyR = valid ? d.pbody[r] : -1;
    const float4 bounds{sep_of_key(fs[prx::kFindLoX]), sep_of_key(fs[prx::kFindLoY]), sep_of_key(fs[prx::kFindHiX]),
                        sep_of_key(fs[prx::kFindHiY])};
    int hits = 0;
    for (int base = int(blockIdx.y) * kMovedTile; base < moved; base += int(gridDim.y) * kMovedTile) {
        const int n = min(kMovedTile, moved - base);
        __syncthreads();
        if (int(threadIdx.x) < n) {
            const int p = g.moved[base + int(threadIdx.x)];
            s_p[threadIdx.x] = p;
            s_box[threadIdx.x] = d.paabb[p];
        }
        __syncthreads();
        for (int k = 0; k < n; ++k) {
            if (!(valid && overlap(box, s_box[k]))) continue;
            const int p = s_p[k];
            if (r == p || (movedR && p > r)) continue;
            const int bodyP = d.pbody[p];
            if (bodyP == bodyR) continue;
            ++hits;
            const int pa = min(p, r), pb = max(p, r);
            if (hash_has(g, pa, pb)) continue;
            if (!((d.bflags[bodyP] | d.bflags[bodyR]) & prx::kAccelerable)) continue;
            if (!should_collide(d, d.pshape[pa], d.pshape[pb])) continue;
            const int at = atomicAdd(&fs[prx::kFindFresh], 1);
            if (at < g.pairCap)
                g.fresh[at] = (static_cast<unsigned long long>(unsigned(p)) << 46) |
                              (static_cast<unsigned long long>(morton_code(bounds, box)) << 16) | unsigned(r);
        }
    }
    for (int o = 32; o > 0; o >>= 1) hits += __shfl_xor(hits, o);
    if ((threadIdx.x & (kWave - 1)) == 0 && hits) {
        const int before = atomicAdd(&fs[prx::kFindHits], hits);
        if (before + hits > g.pairCap) atomicOr(reinterpret_cast<unsigned*>(&d.hdr[0].status), prx::kStatusScratchOverflow);
    }
}

// Contact creation (AabbTreeWorld.cpp:2470-2547) for the listed pairs, bodies
// woken, and the new contacts' narrowphase.  A pair's place behind the
// existing contacts is its rank: the number of listed pairs with a smaller
// key, counted through LDS tiles.  The workgroup that ends last publishes the
// new contact count (all have read the old one by then).
__global__ __launch_bounds__(kGrid) void k_pairs_create(DeviceState d, BigState g, StepParams c, int slot, int statSlot) {
    __shared__ unsigned long long s_key[kGrid];
    WorldHeader& H = d.hdr[0];
    int* const fs = find_state(g, slot);
    const int n = min(fs[prx::kFindFresh], g.pairCap);
    const int moved = fs[prx::kFindMoved];
    const int nc0 = H.ncontacts, cap = H.contact_cap;
    for (int k = int(blockIdx.x * blockDim.x + threadIdx.x); k < moved; k += int(gridDim.x * blockDim.x))
        d.pflags[g.moved[k]] &= ~prx::kProxyMoved;
    for (int base = int(blockIdx.x) * kGrid; base < n; base += int(gridDim.x) * kGrid) {
        const int j = base + int(threadIdx.x);
        const unsigned long long key = j < n ? g.fresh[j] : ~0ull;
        int rank = 0;
        for (int t = 0; t < n; t += kGrid) {
            __syncthreads();
            s_key[threadIdx.x] = t + int(threadIdx.x) < n ? g.fresh[t + int(threadIdx.x)] : ~0ull;
            __syncthreads();
            const int cnt = min(kGrid, n - t);
            for (int q = 0; q < cnt; ++q) rank += s_key[q] < key ? 1 : 0;
        }
        const int idx = nc0 + rank;
        if (j >= n || idx >= cap) continue;
        const int p = int(key >> 46), r = int(key & 0xffffull);
        const int pa = min(p, r), pb = max(p, r);
        const int ba = d.pbody[pa], bb = d.pbody[pb];
        const int sa = d.pshape[pa], sb = d.pshape[pb];
        const std::uint32_t fa = d.bflags[ba], fb = d.bflags[bb];
        const int4 sia = d.shape_i[sa], sib = d.shape_i[sb];
        const float4 sfa = d.shape_f[sa], sfb = d.shape_f[sb];
        std::uint32_t flags = prx::kCEnabled | prx::kNeedsUpdating;
        if ((fa | fb) & prx::kImpenetrable) flags |= prx::kCImpenetrable;
        const bool sensor = sia.z != 0 || sib.z != 0;
        if (sensor) flags |= prx::kSensor;
        d.c_prox[idx] = int2{pa, pb};
        d.c_body[idx] = int2{ba, bb};
        d.c_shape[idx] = int2{sa, sb};
        d.c_id[idx] = std::uint32_t(idx);
        d.c_flags[idx] = flags;
        d.c_mat[idx] = float4{__builtin_sqrtf(sfa.y * sfb.y), (sfa.z > sfb.z) ? sfa.z : sfb.z, 0.0f, 0.0f};
        d.m_hdr[idx] = uint4{0u, kDefaultCf, kDefaultCf, 0u};
        d.m_geo[idx] = float4{0, 0, 0, 0};
        d.m_p0[idx] = float4{0, 0, 0, 0};
        d.m_p1[idx] = float4{0, 0, 0, 0};
        if (!sensor) {
            if (fa & prx::kSpeedable) atomicOr(&d.bflags[ba], prx::kAwake);
            if (fb & prx::kSpeedable) atomicOr(&d.bflags[bb], prx::kAwake);
        }
        hash_insert(g, pa, pb);
        update_contact(d, 0, idx, c);
    }
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(&fs[prx::kFindDone], 1) == int(gridDim.x) - 1) {
        int nadd = n;
        if (nc0 + nadd > cap) {
            atomicOr(reinterpret_cast<unsigned*>(&H.status), prx::kStatusContactOverflow);
            nadd = cap - nc0;
        }
        H.ncontacts = nc0 + nadd;
        H.stats[statSlot] += std::uint32_t(nadd);
    }
}

// ---------------------------------------------------------------------------
// Linear BVH over the proxies' fat AABBs.

// Bounds of the AABB centres (one workgroup).
__global__ __launch_bounds__(kBlock) void k_lbvh_bounds(DeviceState d, BigState g) {
    __shared__ float s_red[kBlock / kWave];
    const int np = d.hdr[0].nproxies;
    float lox = __builtin_inff(), loy = __builtin_inff(), hix = -__builtin_inff(), hiy = -__builtin_inff();
    for (int p = int(threadIdx.x); p < np; p += kBlock) {
        const float4 a = d.paabb[p];
        const float cx = (a.x + a.z) * 0.5f, cy = (a.y + a.w) * 0.5f;
        lox = fmin_std(lox, cx);
        loy = fmin_std(loy, cy);
        hix = fmax_std(hix, cx);
        hiy = fmax_std(hiy, cy);
    }
    lox = block_reduce_min(lox, s_red);
    loy = block_reduce_min(loy, s_red);
    hix = block_reduce_max(hix, s_red);
    hiy = block_reduce_max(hiy, s_red);
    if (threadIdx.x == 0) g.bounds[0] = float4{lox, loy, hix, hiy};
}

// 30-bit Morton code of each proxy's AABB centre.
__global__ void k_lbvh_morton(DeviceState d, BigState g) {
    const int p = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (p >= d.hdr[0].nproxies) return;
    g.morton[p] = morton_code(g.bounds[0], d.paabb[p]);
    g.order[p] = p;
}

// Stable LSD radix sort of (key, value) pairs by the low `bits` bits of the
// key, one workgroup, 8-bit digits, ping-ponging with the second buffers;
// an even number of passes leaves the result in the first buffers.  Ranks
// within a tile come from per-wave digit matching (8 ballots) plus per-wave
// digit counts in LDS.
__device__ __forceinline__ void block_radix_sort(std::uint32_t* k0, int* v0, std::uint32_t* k1, int* v1, int n,
                                                 int passes) {
    __shared__ int s_base[256];
    __shared__ int s_tile[256];
    __shared__ int s_wave[kBlock / kWave][256];
    const int lane = int(threadIdx.x) & (kWave - 1), wave = int(threadIdx.x) >> 6;
    for (int pass = 0; pass < passes; ++pass) {
        const int shift = 8 * pass;
        std::uint32_t* ks = (pass & 1) ? k1 : k0;
        int* vs = (pass & 1) ? v1 : v0;
        std::uint32_t* kd = (pass & 1) ? k0 : k1;
        int* vd = (pass & 1) ? v0 : v1;
        for (int t = int(threadIdx.x); t < 256; t += kBlock) s_base[t] = 0;
        for (int t = int(threadIdx.x); t < 256 * (kBlock / kWave); t += kBlock) (&s_wave[0][0])[t] = 0;
        __syncthreads();
        for (int i = int(threadIdx.x); i < n; i += kBlock) atomicAdd(&s_base[(ks[i] >> shift) & 0xffu], 1);
        __syncthreads();
        if (threadIdx.x == 0) {
            int run = 0;
            for (int t = 0; t < 256; ++t) {
                const int c = s_base[t];
                s_base[t] = run;
                run += c;
            }
        }
        __syncthreads();
        for (int base = 0; base < n; base += kBlock) {
            const int i = base + int(threadIdx.x);
            const bool valid = i < n;
            std::uint32_t key = 0;
            int val = 0;
            int dig = 0;
            if (valid) {
                key = ks[i];
                val = vs[i];
                dig = int((key >> shift) & 0xffu);
            }
            unsigned long long peers = __ballot(valid);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const bool bit = (dig >> b) & 1;
                const unsigned long long m = __ballot(bit);
                peers &= bit ? m : ~m;
            }
            const int rank = __popcll(peers & lanes_below(lane));
            if (valid && rank == 0) s_wave[wave][dig] = __popcll(peers);
            __syncthreads();
            for (int t = int(threadIdx.x); t < 256; t += kBlock) {
                int run = 0;
                for (int w = 0; w < kBlock / kWave; ++w) {
                    const int c = s_wave[w][t];
                    s_wave[w][t] = run;
                    run += c;
                }
                s_tile[t] = run;
            }
            __syncthreads();
            if (valid) {
                const int dst = s_base[dig] + s_wave[wave][dig] + rank;
                kd[dst] = key;
                vd[dst] = val;
            }
            __syncthreads();
            for (int t = int(threadIdx.x); t < 256; t += kBlock) {
                s_base[t] += s_tile[t];
                for (int w = 0; w < kBlock / kWave; ++w) s_wave[w][t] = 0;
            }
            __syncthreads();
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_lbvh_sort(DeviceState d, BigState g) {
    block_radix_sort(g.morton, g.order, g.morton2, g.order2, d.hdr[0].nproxies, 4);
}

__device__ __forceinline__ int lbvh_delta(const std::uint32_t* code, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    const std::uint32_t a = code[i], b = code[j];
    if (a == b) return 32 + __clz(std::uint32_t(i) ^ std::uint32_t(j));
    return __clz(a ^ b);
}

// Karras' radix-tree construction: internal node i (0 is the root) covers a
// key range with one end at i; children are internal nodes or leaves.  Node
// ids: internal 0..n-2, leaf k at n-1+k.
__global__ void k_lbvh_build(DeviceState d, BigState g) {
    const int n = d.hdr[0].nproxies;
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i == 0) g.parent[0] = -1;
    if (i >= n - 1) return;
    const std::uint32_t* code = g.morton;
    const int dr = lbvh_delta(code, n, i, i + 1), dl = lbvh_delta(code, n, i, i - 1);
    const int dir = (dr - dl) > 0 ? 1 : -1;
    const int dmin = lbvh_delta(code, n, i, i - dir);
    int lmax = 2;
    while (lbvh_delta(code, n, i, i + lmax * dir) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1) {
        if (lbvh_delta(code, n, i, i + (l + t) * dir) > dmin) l += t;
    }
    const int j = i + l * dir;
    const int dnode = lbvh_delta(code, n, i, j);
    int s = 0;
    int t = l;
    do {
        t = (t + 1) >> 1;
        if (lbvh_delta(code, n, i, i + (s + t) * dir) > dnode) s += t;
    } while (t > 1);
    const int gamma = i + s * dir + (dir < 0 ? -1 : 0);
    const int lo = min(i, j), hi = max(i, j);
    const int left = (lo == gamma) ? (n - 1 + gamma) : gamma;
    const int right = (hi == gamma + 1) ? (n - 1 + gamma + 1) : (gamma + 1);
    g.left[i] = left;
    g.right[i] = right;
    g.parent[left] = i;
    g.parent[right] = i;
    g.visit[i] = 0;
}

// Bottom-up bounds: each leaf climbs; the second child to arrive at a node
// writes the node's union and continues.
__global__ void k_lbvh_refit(DeviceState d, BigState g) {
    const int n = d.hdr[0].nproxies;
    const int k = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (k >= n) return;
    const int leaf = n - 1 + k;
    g.naabb[leaf] = d.paabb[g.order[k]];
    if (n == 1) return;
    __threadfence();
    int cur = g.parent[leaf];
    for (int depth = 0; cur >= 0; ++depth) {
        if (depth > kMaxDepth) {
            d.hdr[0].status |= prx::kStatusScratchOverflow;
            return;
        }
        if (atomicAdd(&g.visit[cur], 1) == 0) return;
        __threadfence();
        const volatile float4* nb = g.naabb;
        const int l = g.left[cur], r = g.right[cur];
        const float4 a = float4{nb[l].x, nb[l].y, nb[l].z, nb[l].w};
        const float4 b = float4{nb[r].x, nb[r].y, nb[r].z, nb[r].w};
        g.naabb[cur] = float4{fmin_std(a.x, b.x), fmin_std(a.y, b.y), fmax_std(a.z, b.z), fmax_std(a.w, b.w)};
        __threadfence();
        cur = g.parent[cur];
    }
}

// Escape index of every node: the next node of a depth-first pre-order walk
// once the node's subtree is done (-1 past the end).
__global__ void k_lbvh_escape(DeviceState d, BigState g) {
    const int n = d.hdr[0].nproxies;
    const int node = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (node >= 2 * n - 1) return;
    int cur = node, esc = -1;
    for (int depth = 0; cur != 0 && depth <= kMaxDepth; ++depth) {
        const int p = g.parent[cur];
        if (g.left[p] == cur) {
            esc = g.right[p];
            break;
        }
        cur = p;
    }
    g.escape[node] = esc;
}

// FindContacts for one moved proxy p (AabbTreeWorld.cpp:709-751): proxies of
// other bodies whose fat AABB overlaps p's.  A pair of two moved proxies is
// emitted by the lower index only, so every key appears once.  Pass 0
// counts, pass 1 writes at the proxy's offset.
template <int kPass>
__global__ void k_lbvh_pairs(DeviceState d, BigState g) {
    const int n = d.hdr[0].nproxies;
    const int p = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (p >= n) return;
    int count = 0;
    if (d.pflags[p] & prx::kProxyMoved) {
        const float4 q = d.paabb[p];
        const int bodyP = d.pbody[p];
        int at = 0;
        if constexpr (kPass == 1) at = g.pcount[p];
        const int end = (kPass == 1) ? min(g.pcount[p + 1], g.pairCap) : 0;
        int node = 0;
        for (int visits = 0; node >= 0 && visits < 4 * n; ++visits) {
            if (overlap(g.naabb[node], q)) {
                if (node >= n - 1) {
                    const int r = g.order[node - (n - 1)];
                    if (r != p && d.pbody[r] != bodyP && (!(d.pflags[r] & prx::kProxyMoved) || p < r)) {
                        if constexpr (kPass == 0) {
                            ++count;
                        } else {
                            if (at < end) g.pairs[at] = int2{min(p, r), max(p, r)};
                            ++at;
                        }
                    }
                    node = g.escape[node];
                } else {
                    node = g.left[node];
                }
            } else {
                node = g.escape[node];
            }
        }
    }
    if constexpr (kPass == 0) g.pcount[p] = count;
}

// Exclusive scan of the per-proxy pair counts (one workgroup); pcount[n] is
// the total (clamped to the pair capacity, with the overflow status set).
__global__ __launch_bounds__(kBlock) void k_lbvh_scan(DeviceState d, BigState g) {
    __shared__ int s_scan[kBlock / kWave + 1];
    const int n = d.hdr[0].nproxies;
    int carry = 0;
    for (int base = 0; base < n; base += kBlock) {
        const int i = base + int(threadIdx.x);
        const int v = (i < n) ? g.pcount[i] : 0;
        int tot = 0;
        const int r = block_exclusive_scan(v, s_scan, tot);
        if (i < n) g.pcount[i] = carry + r;
        carry += tot;
    }
    if (threadIdx.x == 0) {
        g.pcount[n] = carry;
        g.counters[prx::kBigPairs] = min(carry, g.pairCap);
        if (carry > g.pairCap) d.hdr[0].status |= prx::kStatusScratchOverflow;
    }
}

// ---------------------------------------------------------------------------
// Solve.

__device__ __forceinline__ bool moves(const DeviceState& d, int b) {
    return (d.bflags[b] & prx::kAccelerable) != 0;
}

// Touching, enabled, non-sensor.
__device__ __forceinline__ bool solved_contact(const DeviceState& d, int i) {
    const std::uint32_t f = d.c_flags[i];
    return (f & prx::kCEnabled) && (f & prx::kTouching) && !(f & prx::kSensor);
}

// Body constraints (GetBodyConstraints, AabbTreeWorld.cpp:276-287): every
// dynamic body takes part and is kept awake; others keep their pose.  Also
// the touching contacts of each workgroup's range counted, and the
// colouring's initial state: no colour used at any body, a new claim epoch.
__global__ __launch_bounds__(kGrid) void k_big_bodies(DeviceState d, BigState g, StepParams c) {
    __shared__ int s_cnt[kGrid / kWave];
    const int b = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (b == 0) {
        g.counters[prx::kBigColors] = 0;
        g.counters[prx::kBigLeft] = 0;
        g.counters[prx::kBigEpoch] += 1;
        g.counters[prx::kBigWork] = 0;
    }
    if (b < prx::kBigSweepSlots) g.sweep[b] = (b < prx::kBigPosSlot) ? 0 : 0x7f800000;  // 0.0f; key of +inf
    if (b < d.hdr[0].nbodies) {
        const std::uint32_t f = d.bflags[b];
        const float4 p1 = d.pos1[b];
        g.used[b] = 0ull;
        if ((f & prx::kSpeedable) && (f & prx::kEnabled)) {
            d.bflags[b] = f | prx::kAwake;
            d.pos0[b] = p1;
            d.s_bc_pos[b] = p1;
            d.s_bc_vel[b] = integrated_velocity(d, b, c);
        } else {
            d.s_bc_pos[b] = p1;
            d.s_bc_vel[b] = float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    const int nc = d.hdr[0].ncontacts;
    if (int(blockIdx.x) * kGrid >= nc) return;
    int tot = 0;
    (void)block_rank(b < nc && solved_contact(d, b), s_cnt, tot);
    if (threadIdx.x == 0) g.blockSum[blockIdx.x] = tot;
}

// Graph colouring by rounds of speculative first-fit (two grid-wide launches
// per round).  A colour is a set of touching contacts in which no dynamic
// body appears twice: every uncoloured contact proposes the lowest colour
// free at both its dynamic bodies; at each (body, colour) the lowest list
// position wins; contacts that won all their claims take the colour.  Static
// and kinematic bodies are never changed by a contact solve, so they do not
// constrain the colouring.  A round starts only if the previous one left
// contacts uncoloured.
__device__ __forceinline__ unsigned long long claim_key(const BigState& g, int round, int e) {
    const unsigned epoch = unsigned(g.counters[prx::kBigEpoch]) * 64u + unsigned(round);
    return (static_cast<unsigned long long>(~epoch) << 32) | static_cast<unsigned>(e);
}

// The touching contacts in contact order (k_big_bodies counted them), and the
// first round's proposals: no colour is used yet, so every contact proposes
// colour 0.
__global__ __launch_bounds__(kGrid) void k_big_touch_list(DeviceState d, BigState g) {
    __shared__ int s_cnt[kGrid / kWave];
    const int nc = d.hdr[0].ncontacts;
    const int blk = int(blockIdx.x), i = blk * kGrid + int(threadIdx.x);
    if (blk * kGrid >= nc && blk > 0) return;
    const bool t = i < nc && solved_contact(d, i);
    const int before = block_sum_of(g.blockSum, nc > 0 ? blk : 0, s_cnt);
    int tot = 0;
    const int e = before + block_rank(t, s_cnt, tot);
    if ((blk + 1) * kGrid >= nc && threadIdx.x == 0) {
        const int m = before + tot;
        g.counters[prx::kBigTouching] = m;
        g.counters[prx::kBigRounds] = m > 0 ? 1 : 0;
        g.counters[prx::kBigLeft + 1] = m;  // read by round 0 as "left after the previous round"
    }
    if (!t) return;
    g.list[e] = i;
    g.color[e] = -1;
    g.tent[e] = 0;
    const int2 bd = d.c_body[i];
    const unsigned long long key = claim_key(g, 0, e);
    if (moves(d, bd.x)) atomicMin(&g.claim[bd.x * prx::kBigMaxColors], key);
    if (moves(d, bd.y)) atomicMin(&g.claim[bd.y * prx::kBigMaxColors], key);
}

// Claims and used masks are changed by atomics; a round that runs in the same
// launch as the one before (kSame) reads them with agent-scope loads.
template <bool kSame>
__device__ __forceinline__ unsigned long long seen64(const void* p) {
    if constexpr (kSame)
        return __hip_atomic_load(static_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else return *static_cast<const unsigned long long*>(p);
}

template <bool kSame>
__device__ __forceinline__ void col_propose(const DeviceState& d, const BigState& g, int round, int e) {
    const int2 bd = d.c_body[g.list[e]];
    const bool ma = moves(d, bd.x), mb = moves(d, bd.y);
    std::uint64_t mask = 0ull;
    if (ma) mask |= seen64<kSame>(g.used + bd.x);
    if (mb) mask |= seen64<kSame>(g.used + bd.y);
    const unsigned long long freeCols = ~mask & ((1ull << prx::kBigMaxColors) - 1ull);
    const int col = freeCols ? (__ffsll(freeCols) - 1) : -1;
    g.tent[e] = col;
    if (col < 0) return;
    const unsigned long long key = claim_key(g, round, e);
    if (ma) atomicMin(&g.claim[bd.x * prx::kBigMaxColors + col], key);
    if (mb) atomicMin(&g.claim[bd.y * prx::kBigMaxColors + col], key);
}

// Whether contact e won its claims (and took its colour); ncol grows to the
// colours in use.
template <bool kSame>
__device__ __forceinline__ bool col_commit(const DeviceState& d, const BigState& g, int round, int e, int& ncol) {
    const int col = g.tent[e];
    if (col < 0) return false;
    const int2 bd = d.c_body[g.list[e]];
    const bool ma = moves(d, bd.x), mb = moves(d, bd.y);
    const unsigned long long key = claim_key(g, round, e);
    if (ma && seen64<kSame>(&g.claim[bd.x * prx::kBigMaxColors + col]) != key) return false;
    if (mb && seen64<kSame>(&g.claim[bd.y * prx::kBigMaxColors + col]) != key) return false;
    g.color[e] = col;
    const unsigned long long bit = 1ull << col;
    if (ma) atomicOr(reinterpret_cast<unsigned long long*>(g.used + bd.x), bit);
    if (mb) atomicOr(reinterpret_cast<unsigned long long*>(g.used + bd.y), bit);
    ncol = (col + 1 > ncol) ? col + 1 : ncol;
    return true;
}

__global__ __launch_bounds__(kGrid) void k_col_propose(DeviceState d, BigState g, int round) {
    // The count this round's commit accumulates starts at zero, also when the
    // colouring is already complete, so that "done" carries to later rounds.
    const bool done = g.counters[prx::kBigLeft + ((round + 1) & 1)] == 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        g.counters[prx::kBigLeft + (round & 1)] = 0;
        if (!done) g.counters[prx::kBigRounds] = round + 1;
    }
    if (done) return;
    const int m = g.counters[prx::kBigTouching];
    for (int e = int(blockIdx.x * blockDim.x + threadIdx.x); e < m; e += int(gridDim.x * blockDim.x))
        if (g.color[e] < 0) col_propose<false>(d, g, round, e);
}

// keepWork: the contacts left go to the work list (list2) of k_col_rest.
__global__ __launch_bounds__(kGrid) void k_col_commit(DeviceState d, BigState g, int round, int keepWork) {
    if (g.counters[prx::kBigLeft + ((round + 1) & 1)] == 0) return;
    const int m = g.counters[prx::kBigTouching];
    int left = 0, ncol = 0;
    for (int e = int(blockIdx.x * blockDim.x + threadIdx.x); e < m; e += int(gridDim.x * blockDim.x)) {
        if (g.color[e] >= 0 || col_commit<false>(d, g, round, e, ncol)) continue;
        ++left;
        if (keepWork) g.list2[atomicAdd(&g.counters[prx::kBigWork], 1)] = e;
    }
    // One atomic per wavefront.
    for (int off = kWave / 2; off > 0; off >>= 1) {
        left += __shfl_xor(left, off);
        const int o = __shfl_xor(ncol, off);
        ncol = (o > ncol) ? o : ncol;
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        if (left) atomicAdd(&g.counters[prx::kBigLeft + (round & 1)], left);
        if (ncol) atomicMax(&g.counters[prx::kBigColors], ncol);
    }
}

// The rounds from `first` on, by one workgroup over the contacts the grid's
// rounds left: a round here costs two workgroup barriers instead of two
// launches.  The lowest list position wins a claim, so a round colours a tenth
// to a half of what is left: of 49,000 touching contacts 22,000 are left after
// 4 rounds and 1,000 after 8, of which the rest take 6 to 8 rounds more.  With
// 4 grid rounds this kernel took 340 us; with 8 it takes 130 over the 600 steps
// of a drop and 230 over the last 100.  A round that colours nothing is the
// last: the lowest position with a free colour always wins, so what is left
// touches a body that has contacts of every colour, and is solved serially.
constexpr int kGridRounds = 8;
__global__ __launch_bounds__(kBlock) void k_col_rest(DeviceState d, BigState g, int first) {
    __shared__ int s_left, s_ncol;
    const int n = g.counters[prx::kBigWork];
    if (n == 0) return;
    int round = first, before = n;
    for (; round < prx::kBigColorRounds; ++round) {
        if (threadIdx.x == 0) s_left = s_ncol = 0;
        for (int k = int(threadIdx.x); k < n; k += kBlock) {
            const int e = g.list2[k];
            if (g.color[e] < 0) col_propose<true>(d, g, round, e);
        }
        __threadfence();
        __syncthreads();
        int left = 0, ncol = 0;
        for (int k = int(threadIdx.x); k < n; k += kBlock) {
            const int e = g.list2[k];
            if (g.color[e] < 0 && !col_commit<true>(d, g, round, e, ncol)) ++left;
        }
        if (left) atomicAdd(&s_left, left);
        if (ncol) atomicMax(&s_ncol, ncol);
        __threadfence();
        __syncthreads();
        const int rest = s_left;
        if (threadIdx.x == 0 && s_ncol > g.counters[prx::kBigColors]) g.counters[prx::kBigColors] = s_ncol;
        __syncthreads();
        if (rest == 0 || rest == before) {  // all coloured, or none left has a colour free
            ++round;
            break;
        }
        before = rest;
    }
    if (threadIdx.x == 0) g.counters[prx::kBigRounds] = round;
}

// The colour order: within a colour the contacts with two manifold points come
// first, so that a wavefront's updates take one path of the velocity solve
// (block or sequential) and of the position solve; the order within a colour
// does not change a result.  Two buckets per colour, then the serial bucket
// (list order).  A box of settled drops, a step with the last launch of a sweep
// taking colours of 256, 512, 1024, 2048, 4096 and 8192 contacts in all: 5000
// bodies 670, 659, 675, 679, 750, 911 us; 10,000: 806, 800, 800, 853, 900, 1085;
// 50,000: 1538, 1540, 1539, 1595, 1608, 1914.
constexpr int kColourBuckets = 2 * prx::kBigMaxColors;
constexpr int kBuckets = kColourBuckets + 1;
__device__ __forceinline__ int colour_bucket(const DeviceState& d, const BigState& g, int e) {
    const int col = g.color[e];
    if (col < 0) return kColourBuckets;
    return 2 * col + (((d.m_hdr[g.list[e]].x >> 8) & 0xffu) == 2u ? 0 : 1);
}
constexpr int kTailContacts = 512;

// Bucket counts of each workgroup's range of the touching list.
__global__ __launch_bounds__(kGrid) void k_big_buckets(DeviceState d, BigState g) {
    __shared__ int s_cnt[kBuckets];
    const int m = g.counters[prx::kBigTouching];
    const int blk = int(blockIdx.x), e = blk * kGrid + int(threadIdx.x);
    if (blk * kGrid >= m) return;
    if (threadIdx.x < kBuckets) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    if (e < m) atomicAdd(&s_cnt[colour_bucket(d, g, e)], 1);
    __syncthreads();
    if (threadIdx.x < kBuckets) g.blockHist[blk * kBuckets + int(threadIdx.x)] = s_cnt[threadIdx.x];
}

// The wave's lanes holding the same bucket.
__device__ __forceinline__ unsigned long long bucket_peers(bool valid, int bucket) {
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
        const bool bit = (bucket >> b) & 1;
        const unsigned long long mm = __ballot(bit);
        peers &= bit ? mm : ~mm;
    }
    return peers;
}

// The velocity and position constraint record of contact gi at place e of
// the colour order (GetPositionConstraints / GetVelocityConstraints,
// AabbTreeWorld.cpp:289-357).
template <bool kLds>
__device__ __forceinline__ void big_record(const DeviceState& d, const StepParams& c, const Bodies<kLds>& bs, int gi, int e) {
    const int2 bd = d.c_body[gi];
    const int2 ss = d.c_shape[gi];
    const float rA = d.shape_f[ss.x].x, rB = d.shape_f[ss.y].x;
    const BodyC A = load_bodyc(d, bd.x), B = load_bodyc(d, bd.y);
    const float4 pA = bs.pos(bd.x), pB = bs.pos(bd.y);
    const Xf xfA = get_xf(pA.x, pA.y, pA.z, A.lc);
    const Xf xfB = get_xf(pB.x, pB.y, pB.z, B.lc);
    const Manifold mf = load_manifold(d, gi);
    const WM wm = world_manifold(mf, xfA, rA, xfB, rB);
    const float4 mt = d.c_mat[gi];
    const Vc vc = make_vc(wm, mt.x, mt.y, mt.z, bd.x, bd.y, A, pA, bs.vel(bd.x), B, pB, bs.vel(bd.y), c);
    store_vc(d.s_vc + std::size_t(e) * prx::kVcStride, vc, A, B);
    store_pc(d.s_pc + std::size_t(e) * prx::kPcStride, mf, bd.x, bd.y, rA + rB, A, B);
}

// The stable colour order of the touching list (list order within a colour)
// and the constraint records in that order.  A contact's place is its
// colour's start, the colour's contacts in earlier workgroups' ranges, and
// its rank among its own range's.
__global__ __launch_bounds__(kGrid) void k_big_records(DeviceState d, BigState g, StepParams c) {
    __shared__ int s_total[kBuckets], s_before[kBuckets], s_start[kBuckets + 1];
    __shared__ int s_wave[kGrid / kWave][kBuckets];
    const int m = g.counters[prx::kBigTouching];
    const int blk = int(blockIdx.x), e = blk * kGrid + int(threadIdx.x);
    if (blk * kGrid >= m && blk > 0) return;
    const int lane = int(threadIdx.x) & (kWave - 1), wave = int(threadIdx.x) >> 6;
    if (threadIdx.x < kBuckets) s_total[threadIdx.x] = s_before[threadIdx.x] = 0;
    for (int k = int(threadIdx.x); k < (kGrid / kWave) * kBuckets; k += kGrid) (&s_wave[0][0])[k] = 0;
    __syncthreads();
    const int words = ((m + kGrid - 1) / kGrid) * kBuckets;
    for (int k = int(threadIdx.x); k < words; k += kGrid) {
        const int col = k % kBuckets, cnt = g.blockHist[k];
        if (!cnt) continue;
        atomicAdd(&s_total[col], cnt);
        if (k / kBuckets < blk) atomicAdd(&s_before[col], cnt);
    }
    const bool valid = e < m;
    const int col = valid ? colour_bucket(d, g, e) : 0;
    const unsigned long long peers = bucket_peers(valid, col);
    const int rank = __popcll(peers & lanes_below(lane));
    if (valid && rank == 0) s_wave[wave][col] = __popcll(peers);
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int k = 0; k < kBuckets; ++k) {
            s_start[k] = run;
            run += s_total[k];
        }
        s_start[kBuckets] = run;
    }
    __syncthreads();
    if (blk == 0) {
        // colorStart: the colours' starts, the serial bucket's, the end.
        if (threadIdx.x <= prx::kBigMaxColors) g.colorStart[threadIdx.x] = s_start[2 * threadIdx.x];
        if (threadIdx.x == 0) {
            g.colorStart[prx::kBigMaxColors + 1] = m;
            // The sweeps' last launch takes every colour from the first whose
            // successors hold few contacts in all (k_big_sweep).
            int k = prx::kBigMaxColors;
            while (k > 0 && m - s_start[2 * (k - 1)] <= kTailContacts) --k;
            g.counters[prx::kBigTail] = k;
        }
    }
    if (!valid) return;
    int at = s_start[col] + s_before[col] + rank;
    for (int w = 0; w < wave; ++w) at += s_wave[w][col];
    const int gi = g.list[e];
    g.list2[at] = gi;
    const Bodies<false> bs{d.s_bc_pos, d.s_bc_vel, d.hdr[0].nbodies};
    big_record(d, c, bs, gi, at);
}

// A sweep over the colours in order: colours 0 to kGridColours - 1 by a launch
// each, the whole grid striding over the colour (no dynamic body appears twice
// in it), and the rest by one workgroup's launch with a barrier between
// colours.  First-fit colouring leaves the contacts in the first few colours,
// so that launch starts at the first colour whose successors hold at most
// kTailContacts contacts in all, and the grid's launches of later colours
// return at once.  A launch for each of the 16 colours and the serial bucket
// spent 2.5 us on every empty one.  4, 6, 7, 8 and 10 launches, a step of 10,000
// settled bodies: 895, 781, 798, 818 and 909 us, of 50,000: 2490, 1587, 1540,
// 1558 and 1651 (4 and 10 measured with kTailContacts at 2048).
constexpr int kGridColours = 7;

// The sweeps' work on a constraint: its record (float4 kRec of them, read
// ahead by the one-workgroup sweeps) and the update, with the body state in bs.
struct WarmSweep {
    static constexpr bool kMin = false;
    static constexpr int kRec = prx::kVcStride;
    static __device__ __forceinline__ const float4* rec(const DeviceState& d, int e) {
        return d.s_vc + std::size_t(e) * prx::kVcStride;
    }
    template <bool kLds>
    static __device__ __forceinline__ float one(const DeviceState&, const StepParams&, const Bodies<kLds>& bs,
                                                const float4 (&r)[kRec], int) {
        BodyC A, B;
        const Vc vc = load_vc(r, A, B);
        warm_start_one(vc, A, B, bs);  // WarmStartVelocities, AabbTreeWorld.cpp:264-274
        return 0.0f;
    }
};
struct VelocitySweep {
    static constexpr bool kMin = false;
    static constexpr int kRec = prx::kVcStride;
    static __device__ __forceinline__ const float4* rec(const DeviceState& d, int e) {
        return d.s_vc + std::size_t(e) * prx::kVcStride;
    }
    template <bool kLds>
    static __device__ __forceinline__ float one(const DeviceState& d, const StepParams&, const Bodies<kLds>& bs,
                                                const float4 (&r)[kRec], int e) {
        float4* out = d.s_vc + std::size_t(e) * prx::kVcStride;
        BodyC A, B;
        Vc vc = load_vc(r, A, B);
        const float mi = solve_velocity_one(vc, A, B, bs);  // SolveVelocityConstraintsViaGS
        out[4] = float4{vc.p[0].ni, vc.p[0].ti, vc.p[0].nm, vc.p[0].tm};
        out[7] = float4{vc.p[1].ni, vc.p[1].ti, vc.p[1].nm, vc.p[1].tm};
        return mi;
    }
};
struct PositionSweep {
    static constexpr bool kMin = true;
    static constexpr int kRec = prx::kPcStride;
    static __device__ __forceinline__ const float4* rec(const DeviceState& d, int e) {
        return d.s_pc + std::size_t(e) * prx::kPcStride;
    }
    template <bool kLds>
    static __device__ __forceinline__ float one(const DeviceState&, const StepParams& c, const Bodies<kLds>& bs,
                                                const float4 (&r)[kRec], int) {
        const Pc pc = load_pc(r);
        float4 pa = bs.pos(pc.bA);
        float4 pb = bs.pos(pc.bB);
        const float sep = solve_pc(pc.m, pc.totalRadius, pc.A, pc.B, pa, pb, c);  // SolvePositionConstraintsViaGS
        bs.set_pos(pc.bA, pa);
        bs.set_pos(pc.bB, pb);
        return sep;
    }
};
template <class Sweep>
__device__ __forceinline__ void sweep_load(const DeviceState& d, int e, float4 (&r)[Sweep::kRec]) {
    const float4* src = Sweep::rec(d, e);
#pragma unroll
    for (int f = 0; f < Sweep::kRec; ++f) r[f] = src[f];
}

// Velocity iteration `it` stops the sweeps if an earlier iteration's largest
// impulse change was at most regMinMomentum (the early exit of
// SolveRegIslandViaGS, AabbTreeWorld.cpp:1610-1616).
__device__ __forceinline__ bool velocity_done(const BigState& g, const StepParams& c, int it) {
    for (int j = 0; j < it; ++j)
        if (__int_as_float(g.sweep[prx::kBigVelSlot + j]) <= c.regMinMomentum) return true;
    return false;
}

// Position iteration `it` stops if an earlier one reached regMinSeparation
// (AabbTreeWorld.cpp:1627-1642).  Slots hold order-preserving keys of floats.
__device__ __forceinline__ bool position_done(const BigState& g, const StepParams& c, int it) {
    for (int j = 0; j < it; ++j)
        if (sep_of_key(g.sweep[prx::kBigPosSlot + j]) >= c.regMinSeparation) return true;
    return false;
}

// Whether iteration `it` of a sweep runs, its neutral extreme, and the
// wave's extreme over its constraints added to the iteration's slot.
template <class Sweep>
__device__ __forceinline__ bool sweep_runs(const BigState& g, const StepParams& c, int it) {
    if constexpr (Sweep::kMin) return !position_done(g, c, it);
    else return !velocity_done(g, c, it);
}
template <class Sweep>
__device__ __forceinline__ float sweep_more(float a, float b) {
    if constexpr (Sweep::kMin) return fmin_std(a, b);
    else return fmax_std(a, b);
}
template <class Sweep>
__device__ __forceinline__ void sweep_report(const BigState& g, int it, float v) {
    for (int off = kWave / 2; off > 0; off >>= 1) v = sweep_more<Sweep>(v, __shfl_xor(v, off));
    if ((threadIdx.x & (kWave - 1)) != 0) return;
    if constexpr (Sweep::kMin) {
        if (v < __builtin_inff()) atomicMin(&g.sweep[prx::kBigPosSlot + it], sep_key(v));
    } else {
        if (v > 0.0f) atomicMax(&g.sweep[prx::kBigVelSlot + it], __float_as_int(v));
    }
}

// Iteration `it` over colour k < kGridColours.
template <class Sweep>
__global__ __launch_bounds__(kGrid) void k_big_sweep(DeviceState d, BigState g, StepParams c, int it, int k) {
    if (k >= g.counters[prx::kBigTail] || !sweep_runs<Sweep>(g, c, it)) return;
    const Bodies<false> bs{d.s_bc_pos, d.s_bc_vel, d.hdr[0].nbodies};
    float v = Sweep::kMin ? __builtin_inff() : 0.0f;
    const int e1 = g.colorStart[k + 1];
    for (int e = g.colorStart[k] + int(blockIdx.x * blockDim.x + threadIdx.x); e < e1; e += int(gridDim.x * blockDim.x))
    {
        float4 rec[Sweep::kRec];
        sweep_load<Sweep>(d, e, rec);
        v = sweep_more<Sweep>(v, Sweep::one(d, c, bs, rec, e));
    }
    sweep_report<Sweep>(g, it, v);
}

// A sweep by one workgroup over colours [k0, k1), a barrier between colours,
// then the serial bucket in list order by one thread; returns the thread's
// extreme.  start: the colours' first places and, at kBigMaxColors and after
// it, the serial bucket's and the end.  A constraint always falls to the same
// thread, which reads the next one's record (of this colour or the next)
// while it solves the present one.
template <class Sweep, bool kLds>
__device__ __forceinline__ float sweep_colours(const DeviceState& d, const StepParams& c, const Bodies<kLds>& bs,
                                               const int* start, int k0, int k1) {
    float v = Sweep::kMin ? __builtin_inff() : 0.0f;
    const int tid = int(threadIdx.x);
    float4 cur[Sweep::kRec], next[Sweep::kRec];
    if (k0 < k1 && start[k0] + tid < start[k0 + 1]) sweep_load<Sweep>(d, start[k0] + tid, cur);
    for (int k = k0; k < k1; ++k) {
        const int e1 = start[k + 1];
        const int ahead = (k + 1 < k1 && e1 + tid < start[k + 2]) ? e1 + tid : -1;
        int e = start[k] + tid;
        if (e >= e1 && ahead >= 0) sweep_load<Sweep>(d, ahead, cur);
        while (e < e1) {
            const int after = e + kSmallBlock < e1 ? e + kSmallBlock : ahead;
            if (after >= 0) sweep_load<Sweep>(d, after, next);
            v = sweep_more<Sweep>(v, Sweep::one(d, c, bs, cur, e));
#pragma unroll
            for (int f = 0; f < Sweep::kRec; ++f) cur[f] = next[f];
            e += kSmallBlock;
        }
        __syncthreads();
    }
    if (tid == 0)
        for (int e = start[prx::kBigMaxColors]; e < start[prx::kBigMaxColors + 1]; ++e) {
            sweep_load<Sweep>(d, e, cur);
            v = sweep_more<Sweep>(v, Sweep::one(d, c, bs, cur, e));
        }
    return v;
}

// Iteration `it` over the other colours (one workgroup) and, in list order,
// the serial bucket.
template <class Sweep>
__global__ __launch_bounds__(kSmallBlock) void k_big_sweep_rest(DeviceState d, BigState g, StepParams c, int it) {
    if (!sweep_runs<Sweep>(g, c, it)) return;
    const Bodies<false> bs{d.s_bc_pos, d.s_bc_vel, d.hdr[0].nbodies};
    __shared__ int s_start[prx::kBigMaxColors + 2];
    if (threadIdx.x < prx::kBigMaxColors + 2) s_start[threadIdx.x] = g.colorStart[threadIdx.x];
    __syncthreads();
    const int first = min(g.counters[prx::kBigTail], kGridColours);
    sweep_report<Sweep>(g, it, sweep_colours<Sweep>(d, c, bs, s_start, first, g.counters[prx::kBigColors]));
}

// IntegratePositions (AabbTreeWorld.cpp:176-188).
template <bool kLds>
__device__ __forceinline__ void big_integrate(const DeviceState& d, const StepParams& c, const Bodies<kLds>& bs, int b) {
    const std::uint32_t fb = d.bflags[b];
    if (!((fb & prx::kSpeedable) && (fb & prx::kEnabled))) return;
    float4 p = bs.pos(b);
    const float4 v = bs.vel(b);
    p.x = p.x + c.dt * v.x;
    p.y = p.y + c.dt * v.y;
    p.z = p.z + c.dt * v.z;
    bs.set_pos(b, p);
}
__global__ __launch_bounds__(kGrid) void k_big_integrate(DeviceState d, StepParams c) {
    const int nb = d.hdr[0].nbodies;
    const int b = int(blockIdx.x * blockDim.x + threadIdx.x);
    const Bodies<false> bs{d.s_bc_pos, d.s_bc_vel, nb};
    if (b < nb) big_integrate(d, c, bs, b);
}

// The colouring's rounds from round 0's commit on, the colour order, the
// records and all the sweeps of a world of at most kSmallBodies bodies, by one
// workgroup with the body state in LDS (32 bytes a body): between colours
// there is a workgroup barrier where the grid's form has a launch.  Same
// colours, order and arithmetic as the grid's form.
__global__ __launch_bounds__(kSmallBlock) void k_big_solve_small(DeviceState d, BigState g, StepParams c) {
    __shared__ int s_cnt[kBuckets], s_start[prx::kBigMaxColors + 2];
    __shared__ int s_wave[kSmallBlock / kWave][kBuckets];
    __shared__ int s_left, s_ncol;
    __shared__ int s_ext;
    const int tid = int(threadIdx.x), lane = tid & (kWave - 1), wave = tid >> 6;
    const int m = g.counters[prx::kBigTouching];
    const int nb = d.hdr[0].nbodies;
    const Bodies<true> bs{nullptr, nullptr, nb};
    for (int b = tid; b < nb; b += kSmallBlock) {
        bs.set_pos(b, d.s_bc_pos[b]);
        bs.set_vel(b, d.s_bc_vel[b]);
    }
    // Colours.
    int colors = 0, before = m;
    for (int round = 0; round < prx::kBigColorRounds; ++round) {
        if (tid == 0) {
            s_left = 0;
            s_ncol = colors;
        }
        if (round > 0)
            for (int e = tid; e < m; e += kSmallBlock)
                if (g.color[e] < 0) col_propose<true>(d, g, round, e);
        __threadfence();
        __syncthreads();
        int left = 0, ncol = 0;
        for (int e = tid; e < m; e += kSmallBlock)
            if (g.color[e] < 0 && !col_commit<true>(d, g, round, e, ncol)) ++left;
        if (left) atomicAdd(&s_left, left);
        if (ncol) atomicMax(&s_ncol, ncol);
        __threadfence();
        __syncthreads();
        const int rest = s_left;
        colors = s_ncol;
        if (tid == 0) g.counters[prx::kBigRounds] = round + 1;
        __syncthreads();
        if (rest == 0 || rest == before) break;
        before = rest;
    }
    // Colour order.
    if (tid < kBuckets) s_cnt[tid] = 0;
    __syncthreads();
    for (int e = tid; e < m; e += kSmallBlock) atomicAdd(&s_cnt[colour_bucket(d, g, e)], 1);
    __syncthreads();
    if (tid == 0) {
        int run = 0;
        for (int k = 0; k < kBuckets; ++k) {
            const int n = s_cnt[k];
            s_cnt[k] = run;
            if ((k & 1) == 0) s_start[k >> 1] = run;
            run += n;
        }
        s_start[prx::kBigMaxColors + 1] = run;
        g.counters[prx::kBigColors] = colors;
    }
    __syncthreads();
    for (int base = 0; base < m; base += kSmallBlock) {
        for (int k = tid; k < (kSmallBlock / kWave) * kBuckets; k += kSmallBlock) (&s_wave[0][0])[k] = 0;
        __syncthreads();
        const int e = base + tid;
        const bool valid = e < m;
        const int col = valid ? colour_bucket(d, g, e) : 0;
        const unsigned long long peers = bucket_peers(valid, col);
        const int rank = __popcll(peers & lanes_below(lane));
        if (valid && rank == 0) s_wave[wave][col] = __popcll(peers);
        __syncthreads();
        if (valid) {
            int at = s_cnt[col] + rank;
            for (int w = 0; w < wave; ++w) at += s_wave[w][col];
            const int gi = g.list[e];
            g.list2[at] = gi;
            big_record(d, c, bs, gi, at);
        }
        __syncthreads();
        if (tid < kBuckets)
            for (int w = 0; w < kSmallBlock / kWave; ++w) s_cnt[tid] += s_wave[w][tid];
        __syncthreads();
    }
    // One sweep; returns its extreme.
    auto sweep = [&](auto kind) {
        using Sweep = decltype(kind);
        float v = sweep_colours<Sweep>(d, c, bs, s_start, 0, colors);
        for (int off = kWave / 2; off > 0; off >>= 1) v = sweep_more<Sweep>(v, __shfl_xor(v, off));
        if (tid == 0) s_ext = Sweep::kMin ? 0x7f800000 : 0;
        __syncthreads();
        if (lane == 0) {
            if constexpr (Sweep::kMin) {
                if (v < __builtin_inff()) atomicMin(&s_ext, sep_key(v));
            } else {
                if (v > 0.0f) atomicMax(&s_ext, __float_as_int(v));
            }
        }
        __syncthreads();
        const int ext = s_ext;
        __syncthreads();
        return ext;
    };
    if (c.warmStart) sweep(WarmSweep{});
    for (int it = 0; it < int(c.velIters); ++it) {
        const int x = sweep(VelocitySweep{});
        if (tid == 0) g.sweep[prx::kBigVelSlot + it] = x;
        if (__int_as_float(x) <= c.regMinMomentum) break;
    }
    for (int b = tid; b < nb; b += kSmallBlock) big_integrate(d, c, bs, b);
    __syncthreads();
    for (int it = 0; it < int(c.posIters); ++it) {
        const int x = sweep(PositionSweep{});
        if (tid == 0) g.sweep[prx::kBigPosSlot + it] = x;
        if (sep_of_key(x) >= c.regMinSeparation) break;
    }
    for (int b = tid; b < nb; b += kSmallBlock) {
        d.s_bc_pos[b] = bs.pos(b);
        d.s_bc_vel[b] = bs.vel(b);
    }
}

// AssignImpulses (AabbTreeWorld.cpp:208-227), the body writeback
// (AabbTreeWorld.cpp:1652-1664) and the body's proxies synchronised
// (AabbTreeWorld.cpp:1532-1544, 2564-2585); records the smallest separation
// of the last position iteration run.
__global__ __launch_bounds__(kGrid) void k_big_finish(DeviceState d, BigState g, StepParams c) {
    const int m = g.counters[prx::kBigTouching];
    const int nb = d.hdr[0].nbodies;
    const int tid = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (tid == 0) {
        float last = __builtin_inff();
        for (int j = 0; j < int(c.posIters); ++j) {
            if (position_done(g, c, j)) break;
            last = sep_of_key(g.sweep[prx::kBigPosSlot + j]);
        }
        g.metrics[prx::kBigMinSeparation] = last;
    }
    if (tid < m) {
        const int gi = g.list2[tid];
        const float4* rec = d.s_vc + std::size_t(tid) * prx::kVcStride;
        const std::uint32_t n = __float_as_uint(rec[1].w);
        float4 m0 = d.m_p0[gi];
        m0.z = rec[4].x;
        m0.w = rec[4].y;
        d.m_p0[gi] = m0;
        if (n > 1) {
            float4 m1 = d.m_p1[gi];
            m1.z = rec[7].x;
            m1.w = rec[7].y;
            d.m_p1[gi] = m1;
        }
    }
    if (tid >= nb) return;
    const std::uint32_t f = d.bflags[tid];
    g.toiLeft[tid] = 1.0f;  // the part of the step a body has left before its first time-of-impact event
    if (!((f & prx::kSpeedable) && (f & prx::kEnabled))) return;
    const Bodies<false> bs{d.s_bc_pos, d.s_bc_vel, nb};
    const float4 bv = bs.vel(tid);
    const float4 bp = bs.pos(tid);
    const float4 p1 = d.pos1[tid];
    if (!(p1.x == bp.x && p1.y == bp.y) || p1.z != bp.z) {
        d.pos1[tid] = float4{bp.x, bp.y, bp.z, 0.0f};
        const float4 l = d.lcinv[tid];
        const Xf xf = get_xf(bp.x, bp.y, bp.z, V2{l.x, l.y});
        d.xf[tid] = float4{xf.p.x, xf.p.y, xf.q.x, xf.q.y};
        d.bflags[tid] = f | 0x100u;
    }
    float4 v = d.vel[tid];
    v.x = bv.x;
    v.y = bv.y;
    v.z = bv.z;
    d.vel[tid] = v;
    const WorldCtx x = big_ctx(d);
    const std::uint32_t moved = synchronize_body(d, x, tid, c);
    if (moved) atomicAdd(&d.hdr[0].stats[prx::kStRegProxiesMoved], moved);
}

// Coloured mode with doToi: continuous collision of dynamic bodies against
// static shapes, after the regular phase.  Every enabled non-sensor contact
// between an awake dynamic body and a static body gets its time of impact
// over the step's sweep (GetToiViaSat, TimeOfImpact.cpp:35-251, as in the
// per-world TOI phase); each body keeps its earliest (ties: the lower contact
// index).  That body is advanced to its pose at the time of impact (Body::
// Advance, Body.hpp:1004-1009), the contact's velocity constraint is built
// and solved there against the static body with the TOI velocity iterations
// (VelocityConstraint, SolveVelocityConstraint with restitution and friction,
// as SolveToiViaGS does for the contact, AabbTreeWorld.cpp:1991-2057) after
// its position iterations at the TOI resolution rate, and the body is
// integrated over the rest of the step with the new velocity.  Its
// proxies and contacts are then synchronised and updated.  A second pass
// checks the sweep from the solved pose to the new end pose.  This is a
// reduced form of the reference's TOI phase: at most two events per body and
// step, the island is the body and the static body of its earliest contact,
// and contacts between dynamic bodies get no time of impact.
__global__ void k_big_toi_static(DeviceState d, BigState g, StepParams c) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= d.hdr[0].ncontacts) return;
    const std::uint32_t f = d.c_flags[i];
    if (!(f & prx::kCEnabled) || (f & prx::kSensor)) return;
    const int2 bd = d.c_body[i];
    const std::uint32_t fa = d.bflags[bd.x], fb = d.bflags[bd.y];
    const bool aDyn = (fa & prx::kAccelerable) && !(fb & prx::kSpeedable);
    const bool bDyn = (fb & prx::kAccelerable) && !(fa & prx::kSpeedable);
    if (!aDyn && !bDyn) return;
    const int dyn = aDyn ? bd.x : bd.y;
    if (!(d.bflags[dyn] & prx::kAwake)) return;
    const SweepD sA = normalized(sweep_of(d, bd.x));
    const SweepD sB = normalized(sweep_of(d, bd.y));
    const int2 sh = d.c_shape[i];
    const ToiRes r = toi_via_sat(shape_proxy(d, sh.x), sA, shape_proxy(d, sh.y), sB, c);
    if (r.time >= 0.0f && r.time < 1.0f)
        atomicMin(&g.toiKey[dyn], (static_cast<unsigned long long>(__float_as_uint(r.time)) << 32) |
                                      static_cast<unsigned long long>(std::uint32_t(i)));
}

__global__ void k_big_toi_apply(DeviceState d, BigState g, StepParams c) {
    const int b = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (b >= d.hdr[0].nbodies) return;
    const unsigned long long key = g.toiKey[b];
    if (key == ~0ull) return;
    g.toiKey[b] = ~0ull;
    const float t = __uint_as_float(std::uint32_t(key >> 32));  // a fraction of the sweep's time
    const int i = int(std::uint32_t(key & 0xffffffffull));
    const int2 bd = d.c_body[i];
    const int2 ss = d.c_shape[i];
    const int o = (bd.x == b) ? bd.y : bd.x;  // the static body
    float4 p = lerp_pos(d.pos0[b], d.pos1[b], t);
    const BodyC Bd = load_bodyc(d, b), Bo = load_bodyc(d, o);
    const float4 po = d.pos1[o];
    const Xf xfD = get_xf(p.x, p.y, p.z, Bd.lc);
    const Xf xfO = get_xf(po.x, po.y, po.z, Bo.lc);
    const bool dynIsA = (bd.x == b);
    const Xf& xfA = dynIsA ? xfD : xfO;
    const Xf& xfB = dynIsA ? xfO : xfD;
    Manifold m = collide_shapes(shape_proxy(d, ss.x), xfA, shape_proxy(d, ss.y), xfB, c.linearSlop, c.maxCirclesRatio);
    float4 v = d.vel[b];
    if (m.n > 0) {
        const float rA = d.shape_f[ss.x].x, rB = d.shape_f[ss.y].x;
        const BodyC& A = dynIsA ? Bd : Bo;
        const BodyC& B = dynIsA ? Bo : Bd;
        // Position iterations at the TOI resolution rate until the TOI minimum
        // separation (the TOI island's position solve, SolveToiViaGS).
        StepParams ps = c;
        ps.regResolutionRate = c.toiResolutionRate;
        float4 qo = po;
        for (std::uint32_t it = 0; it < c.toiPosIters; ++it) {
            float4& qa = dynIsA ? p : qo;
            float4& qb = dynIsA ? qo : p;
            const float sep = solve_pc(m, rA + rB, A, B, qa, qb, ps);
            if (sep >= c.toiMinSeparation) break;
        }
        // Velocity constraint at the solved pose, no warm start, TOI iterations.
        const float4 pA = dynIsA ? p : po, pB = dynIsA ? po : p;
        const Xf xA = get_xf(pA.x, pA.y, pA.z, A.lc), xB = get_xf(pB.x, pB.y, pB.z, B.lc);
        const WM wm = world_manifold(m, xA, rA, xB, rB);
        const float4 mt = d.c_mat[i];
        const float4 vo{0.0f, 0.0f, 0.0f, 0.0f};
        float4 vA = dynIsA ? v : vo, vB = dynIsA ? vo : v;
        StepParams vconf = c;
        vconf.warmStart = 0u;
        Vc vc = make_vc(wm, mt.x, mt.y, mt.z, bd.x, bd.y, A, pA, vA, B, pB, vB, vconf);
        for (std::uint32_t it = 0; it < c.toiVelIters; ++it) {
            float inc = solve_dir(vc, true, A, B, vA, vB);
            if (vc.n == 1 || (vc.K00 == 0.0f && vc.K11 == 0.0f && vc.K01 == 0.0f))
                inc = fmax_std(inc, solve_dir(vc, false, A, B, vA, vB));
            else
                inc = fmax_std(inc, block_solve(vc, A, B, vA, vB));
            if (inc <= c.toiMinMomentum) break;
        }
        const float4 vn = dynIsA ? vA : vB;
        v.x = vn.x;
        v.y = vn.y;
        v.z = vn.z;
        d.vel[b] = v;
    }
    // The rest of the step with the new velocity; the sweep from the solved
    // pose to the new end pose is what a further pass of this step checks.
    const float left = g.toiLeft[b] * (1.0f - t);
    g.toiLeft[b] = left;
    const float h = left * c.dt;
    d.pos0[b] = p;
    p.x = p.x + h * v.x;
    p.y = p.y + h * v.y;
    p.z = p.z + h * v.z;
    d.pos1[b] = p;
    const Xf xf = get_xf(p.x, p.y, p.z, Bd.lc);
    d.xf[b] = float4{xf.p.x, xf.p.y, xf.q.x, xf.q.y};
    d.bflags[b] |= 0x100u;  // contacts to update
    const WorldCtx x = big_ctx(d);
    const std::uint32_t moved = synchronize_body(d, x, b, c);
    atomicAdd(&d.hdr[0].stats[prx::kStToiIslandsSolved], 1u);
    if (moved) atomicAdd(&d.hdr[0].stats[prx::kStToiProxiesMoved], moved);
}

// Smallest separation over touching contacts at the current poses (a
// diagnostic; separation below zero is penetration).
__global__ void k_big_metrics(DeviceState d, BigState g) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= d.hdr[0].ncontacts) return;
    const std::uint32_t f = d.c_flags[i];
    if (!(f & prx::kTouching) || (f & prx::kSensor)) return;
    const int2 bd = d.c_body[i];
    const int2 ss = d.c_shape[i];
    const float4 xa = d.xf[bd.x], xb = d.xf[bd.y];
    const Xf xfA{V2{xa.x, xa.y}, V2{xa.z, xa.w}}, xfB{V2{xb.x, xb.y}, V2{xb.z, xb.w}};
    const Manifold mf = load_manifold(d, i);
    const float tr = d.shape_f[ss.x].x + d.shape_f[ss.y].x;
    float s = __builtin_inff();
#pragma unroll
    for (std::uint32_t k = 0; k < 2; ++k)
        if (k < mf.n) s = fmin_std(s, get_psm(mf, k, xfA, xfB).sep - tr);
    if (s < __builtin_inff()) {
        // Order-preserving integer image of the float for atomicMin.
        const int bits = __float_as_int(s);
        const int key = bits >= 0 ? bits : (bits ^ 0x7fffffff);
        atomicMin(reinterpret_cast<int*>(g.counters + prx::kBigMinSepBits), key);
    }
}

}  // namespace prxd

// ---------------------------------------------------------------------------
// Host-side launch sequences (compiled in this translation unit).

namespace {

unsigned Blocks(int n, int t) { return unsigned((n + t - 1) / t > 0 ? (n + t - 1) / t : 1); }

// UpdateContacts, then FindContacts + AddContacts (slot: which of the step's
// searches; statSlot: the stats word counting the added contacts) with the new
// contacts' narrowphase.
void UpdateAndFind(const prx::DeviceState& d, const prx::BigState& g, const prx::StepParams& c, int slot, int statSlot,
                   hipStream_t s) {
    using namespace prxd;
    hipLaunchKernelGGL(k_big_contacts, dim3(Blocks(g.cap, kGrid)), dim3(kGrid), 0, s, d, g, c, slot);
    hipLaunchKernelGGL(k_pairs_find, dim3(Blocks(g.P > g.B ? g.P : g.B, kGrid), kMovedSplit), dim3(kGrid), 0, s, d, g, slot);
    hipLaunchKernelGGL(k_pairs_create, dim3(256), dim3(kGrid), 0, s, d, g, c, slot, statSlot);
}

template <class Sweep>
void SweepLaunches(const prx::DeviceState& d, const prx::BigState& g, const prx::StepParams& c, int it, hipStream_t s) {
    using namespace prxd;
    for (int k = 0; k < kGridColours; ++k)
        hipLaunchKernelGGL(k_big_sweep<Sweep>, dim3(kSweepBlocks), dim3(kGrid), 0, s, d, g, c, it, k);
    hipLaunchKernelGGL(k_big_sweep_rest<Sweep>, dim3(1), dim3(kSmallBlock), 0, s, d, g, c, it);
}

}  // namespace

// One step of the large world (P proxies, B bodies, contact capacity cap; a
// contact has two proxies and the capacity is above P and B).
extern "C" hipError_t prx_big_launch_step(const prx::DeviceState* dp, const prx::BigState* gp,
                                          const prx::StepParams* c, hipStream_t s) {
    using namespace prxd;
    const prx::DeviceState& d = *dp;
    const prx::BigState& g = *gp;
    const int B = g.B, cap = g.cap;
    const dim3 perContact(Blocks(cap, kGrid)), block(kGrid);
    hipLaunchKernelGGL(k_big_mark, perContact, block, 0, s, d, g, *c);
    hipLaunchKernelGGL(k_big_gather, perContact, block, 0, s, d, g);
    UpdateAndFind(d, g, *c, 0, prx::kStPreAdded, s);
    if (c->dt != 0.0f) {
        hipLaunchKernelGGL(k_big_bodies, perContact, block, 0, s, d, g, *c);
        hipLaunchKernelGGL(k_big_touch_list, perContact, block, 0, s, d, g);
        if (B <= kSmallBodies) {
            hipLaunchKernelGGL(k_big_solve_small, dim3(1), dim3(kSmallBlock), std::size_t(B) * 32, s, d, g, *c);
        } else {
            const unsigned colBlocks = Blocks(cap, kGrid) < 1024u ? Blocks(cap, kGrid) : 1024u;
            for (int r = 0; r < kGridRounds; ++r) {
                if (r > 0) hipLaunchKernelGGL(k_col_propose, dim3(colBlocks), block, 0, s, d, g, r);
                hipLaunchKernelGGL(k_col_commit, dim3(colBlocks), block, 0, s, d, g, r, r == kGridRounds - 1 ? 1 : 0);
            }
            hipLaunchKernelGGL(k_col_rest, dim3(1), dim3(kBlock), 0, s, d, g, kGridRounds);
            hipLaunchKernelGGL(k_big_buckets, perContact, block, 0, s, d, g);
            hipLaunchKernelGGL(k_big_records, perContact, block, 0, s, d, g, *c);
            if (c->warmStart) SweepLaunches<WarmSweep>(d, g, *c, 0, s);
            for (int it = 0; it < int(c->velIters); ++it) SweepLaunches<VelocitySweep>(d, g, *c, it, s);
            hipLaunchKernelGGL(k_big_integrate, dim3(Blocks(B, kGrid)), block, 0, s, d, *c);
            for (int it = 0; it < int(c->posIters); ++it) SweepLaunches<PositionSweep>(d, g, *c, it, s);
        }
        hipLaunchKernelGGL(k_big_finish, perContact, block, 0, s, d, g, *c);
        UpdateAndFind(d, g, *c, 1, prx::kStRegAdded, s);
        if (c->doToi) {
            // Two passes: a body's second event in a step (another static
            // shape reached while moving on) is found from the sweep the
            // first left.
            for (int pass = 0; pass < kBigToiPasses; ++pass) {
                hipLaunchKernelGGL(k_big_toi_static, perContact, block, 0, s, d, g, *c);
                hipLaunchKernelGGL(k_big_toi_apply, dim3(Blocks(B, kGrid)), block, 0, s, d, g, *c);
                UpdateAndFind(d, g, *c, 2 + pass, prx::kStToiAdded, s);
            }
        }
    }
    return hipGetLastError();
}

// Allows the small worlds' solve its LDS (more than the default limit).
extern "C" hipError_t prx_big_prepare(int nbodies) {
    if (nbodies > prxd::kSmallBodies) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(prxd::k_big_solve_small),
                               hipFuncAttributeMaxDynamicSharedMemorySize, prxd::kSmallBodies * 32);
}

// Pair finding only (for tests of the LBVH against brute force): proxies'
// fat AABBs, bodies and moved flags must be set in d.
extern "C" hipError_t prx_big_launch_pairs(const prx::DeviceState* dp, const prx::BigState* gp, hipStream_t s) {
    using namespace prxd;
    const prx::DeviceState& d = *dp;
    const prx::BigState& g = *gp;
    const int P = g.P;
    hipLaunchKernelGGL(k_lbvh_bounds, dim3(1), dim3(kBlock), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_morton, dim3(Blocks(P, kGrid)), dim3(kGrid), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_sort, dim3(1), dim3(kBlock), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_build, dim3(Blocks(P, kGrid)), dim3(kGrid), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_refit, dim3(Blocks(P, kGrid)), dim3(kGrid), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_escape, dim3(Blocks(2 * P, kGrid)), dim3(kGrid), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_pairs<0>, dim3(Blocks(P, kGrid)), dim3(kGrid), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_scan, dim3(1), dim3(kBlock), 0, s, d, g);
    hipLaunchKernelGGL(k_lbvh_pairs<1>, dim3(Blocks(P, kGrid)), dim3(kGrid), 0, s, d, g);
    return hipGetLastError();
}

extern "C" hipError_t prx_big_launch_metrics(const prx::DeviceState* dp, const prx::BigState* gp, hipStream_t s) {
    using namespace prxd;
    hipLaunchKernelGGL(k_big_metrics, dim3(Blocks(gp->cap, kGrid)), dim3(kGrid), 0, s, *dp, *gp);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Pair finding without allocation.  The LBVH's working arrays for up to
// kNoAllocMaxProxies proxies live in one file-scope device array; the caller
// passes device buffers for the inputs and outputs and a stream.  Each device
// holds its own copy of the array, whose address is looked up once per
// device (hipGetSymbolAddress) and used for every kernel argument.

namespace {

constexpr int kNoAllocMaxProxies = 1 << 16;

constexpr std::size_t Align256(std::size_t n) { return (n + 255) & ~std::size_t(255); }

// Byte offsets of the working arrays inside the scratch array (sized for
// kNoAllocMaxProxies; a call with fewer proxies uses the front of each).
struct NoAllocLayout {
    static constexpr std::size_t N = std::size_t(kNoAllocMaxProxies);
    static constexpr std::size_t hdr = 0;
    static constexpr std::size_t paabb = Align256(hdr + sizeof(prx::WorldHeader));
    static constexpr std::size_t pflags = Align256(paabb + 16 * N);
    static constexpr std::size_t morton = Align256(pflags + 4 * N);
    static constexpr std::size_t morton2 = Align256(morton + 4 * N);
    static constexpr std::size_t order = Align256(morton2 + 4 * N);
    static constexpr std::size_t order2 = Align256(order + 4 * N);
    static constexpr std::size_t left = Align256(order2 + 4 * N);
    static constexpr std::size_t right = Align256(left + 4 * N);
    static constexpr std::size_t parent = Align256(right + 4 * N);
    static constexpr std::size_t escape = Align256(parent + 8 * N);
    static constexpr std::size_t visit = Align256(escape + 8 * N);
    static constexpr std::size_t naabb = Align256(visit + 4 * N);
    static constexpr std::size_t bounds = Align256(naabb + 32 * N);
    static constexpr std::size_t pcount = Align256(bounds + 16);
    static constexpr std::size_t counters = Align256(pcount + 4 * (N + 1));
    static constexpr std::size_t bytes = Align256(counters + 4 * prx::kBigCounters);
};

}  // namespace

// About 6.6 MB per device, held until the process ends.
static __device__ __align__(256) unsigned char scratch[NoAllocLayout::bytes];

namespace prxd {

// Inputs into the LBVH's proxy arrays: fat AABBs (4 floats each, any 4-byte
// alignment), moved flags; the header carries the proxy count and a cleared
// status (a fill by kernel, so the call can be captured in a graph).
__global__ void k_noalloc_prep(DeviceState d, const float* aabbs, const std::uint8_t* moved, int n) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i == 0) {
        d.hdr[0].nproxies = n;
        d.hdr[0].status = 0;
    }
    if (i >= n) return;
    d.paabb[i] = float4{aabbs[4 * i], aabbs[4 * i + 1], aabbs[4 * i + 2], aabbs[4 * i + 3]};
    d.pflags[i] = moved[i] ? prx::kProxyMoved : 0u;
}

// The pair count for the caller: the number found (above cap: only cap were
// written), or -1 when the tree walk exceeded its depth bound.
__global__ void k_noalloc_count(DeviceState d, BigState g, int* count) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const int total = g.pcount[g.P];
    const bool depth = (d.hdr[0].status & prx::kStatusScratchOverflow) != 0 && total <= g.pairCap;
    *count = depth ? -1 : total;
}

}  // namespace prxd

namespace {

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mutex;
unsigned char* g_noalloc_ptr[kNoAllocMaxDevices] = {};

// The current device's copy of the scratch array, looked up on the first
// call on that device.
hipError_t NoAllocScratch(unsigned char** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_noalloc_mutex);
    if (!g_noalloc_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_noalloc_ptr[dev] = static_cast<unsigned char*>(p);
    }
    *out = g_noalloc_ptr[dev];
    return hipSuccess;
}

}  // namespace

// Returns a PRX_* status; *err names the failure.
extern "C" int prx_lbvh_pairs_noalloc_impl(const float* aabbs, const std::int32_t* bodies, const std::uint8_t* moved,
                                           int n, std::int32_t* pairs, int cap, int* count, void* stream,
                                           const char** err) {
    using namespace prxd;
    if (!aabbs || !bodies || !moved || n <= 0 || !count || cap < 0 || (cap > 0 && !pairs)) {
        *err = "bad argument";
        return PRX_E_INVALID_ARGUMENT;
    }
    if (n > kNoAllocMaxProxies) {
        *err = "more proxies than the allocation-free pair finder holds (65536)";
        return PRX_E_LENGTH;
    }
    if ((reinterpret_cast<std::uintptr_t>(pairs) & 7u) || (reinterpret_cast<std::uintptr_t>(bodies) & 3u) ||
        (reinterpret_cast<std::uintptr_t>(aabbs) & 3u) || (reinterpret_cast<std::uintptr_t>(count) & 3u)) {
        *err = "misaligned buffer (pairs need 8-byte, the others 4-byte alignment)";
        return PRX_E_INVALID_ARGUMENT;
    }
    unsigned char* base = nullptr;
    if (NoAllocScratch(&base) != hipSuccess) {
        *err = "device scratch lookup failed";
        return PRX_E_DEVICE;
    }
    using L = NoAllocLayout;
    prx::DeviceState d{};
    d.nworlds = 1;
    d.hdr = reinterpret_cast<prx::WorldHeader*>(base + L::hdr);
    d.paabb = reinterpret_cast<float4*>(base + L::paabb);
    d.pflags = reinterpret_cast<std::uint32_t*>(base + L::pflags);
    d.pbody = const_cast<int*>(reinterpret_cast<const int*>(bodies));
    prx::BigState g{};
    g.P = n;
    g.B = 1;
    g.cap = 1;
    g.pairCap = cap;
    g.morton = reinterpret_cast<std::uint32_t*>(base + L::morton);
    g.morton2 = reinterpret_cast<std::uint32_t*>(base + L::morton2);
    g.order = reinterpret_cast<int*>(base + L::order);
    g.order2 = reinterpret_cast<int*>(base + L::order2);
    g.left = reinterpret_cast<int*>(base + L::left);
    g.right = reinterpret_cast<int*>(base + L::right);
    g.parent = reinterpret_cast<int*>(base + L::parent);
    g.escape = reinterpret_cast<int*>(base + L::escape);
    g.visit = reinterpret_cast<int*>(base + L::visit);
    g.naabb = reinterpret_cast<float4*>(base + L::naabb);
    g.bounds = reinterpret_cast<float4*>(base + L::bounds);
    g.pcount = reinterpret_cast<int*>(base + L::pcount);
    g.counters = reinterpret_cast<int*>(base + L::counters);
    g.pairs = reinterpret_cast<int2*>(pairs);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_noalloc_prep, dim3(Blocks(n, kGrid)), dim3(kGrid), 0, s, d, aabbs, moved, n);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = prx_big_launch_pairs(&d, &g, s);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_noalloc_count, dim3(1), dim3(64), 0, s, d, g, count);
        e = hipGetLastError();
    }
    if (e != hipSuccess) {
        *err = hipGetErrorString(e);
        return PRX_E_DEVICE;
    }
    return PRX_OK;
}
